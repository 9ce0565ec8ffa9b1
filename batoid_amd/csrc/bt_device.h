// bt_device.h -- per-ray FP64 device functions of the trace hot path.
//
// Surface sag / normal / time-to-intersect, media n(lambda) and obscuration
// programs, evaluated on descriptors that live in device memory.  All
// threads of a launch read the same descriptor, so its fields are
// wave-uniform (scalar loads); only the per-ray arithmetic is vector work.
//
// Operation order follows the reference expression by expression and the
// library is compiled with -ffp-contract=off, so with IEEE-correct FP64
// division and square root the results are bit-identical to the reference's
// CPU build (which has no FMA on baseline x86-64).  Citations are to
// jmeyers314/batoid.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "../../include/batoid_amd.h"
#include "bt_mlp.h"

#define BT_DEV __device__ __forceinline__

namespace bt {

// Descriptors and coefficient tables are read through the constant address
// space (no launch that reads them writes them, and every lane of a wave reads
// one address: scalar loads), tables gathered per lane through the global
// one.  The compiler infers this from generic pointers in small kernels only;
// a plan kernel left with flat loads took twice the time.
#define BT_CONSTANT __attribute__((address_space(4)))
#define BT_GLOBAL __attribute__((address_space(1)))
using SurfPtr = const BT_CONSTANT bt_surface*;
using MediumPtr = const BT_CONSTANT bt_medium*;
using ObscPtr = const BT_CONSTANT bt_obsc*;
using StepPtr = const BT_CONSTANT bt_step*;
using CoefPtr = const BT_CONSTANT double*;
using TrimPtr = const BT_CONSTANT int*;
using StreamPtr = const BT_CONSTANT bt_poly_stream*;
using TablePtr = const BT_GLOBAL double*;

// ---------------------------------------------------------------------------
// Square roots, reciprocal roots and quotients, correctly rounded, without
// range handling where it cannot change a bit.
//
// The compiler's IEEE sqrt scales x < 2^-767 by 2^256 before the v_rsq_f64
// estimate, refines it (g = x r, h = r/2; one coupled Goldschmidt step; two
// Newton corrections from the residual d = x - g*g), unscales, and selects x
// itself for +-0 and +inf.  Its IEEE division rescales operands of extreme
// exponent (v_div_scale), refines v_rcp_f64 by two Newton steps, applies one
// Markstein correction q + (n - d q) r, and patches special operands
// (v_div_fixup).  Where no operand, quotient or remainder comes near the
// ends of the exponent range all of that range handling is the identity, and
// the *_plain functions below run the refinement alone.  They also share it:
//  * the h that the root's iteration leaves is 1/(2 sqrt(x)) to ~2^-47, so
//    one Newton step gives the reciprocal of a root (2 instructions instead
//    of v_rcp_f64 and 4), and quotients by one denominator (x/r and y/r, the
//    velocity by an index) share one reciprocal: a quotient is then 3
//    instructions instead of 11 (v_rcp_f64 alone takes four issue slots);
//  * from a reciprocal y of d in [1, 2) to 1/2 + e ulp, q = n y and then
//    q + (n - d q) y is n/d correctly rounded (the division's own last step)
//    for every n if d^2 (1 + 2 e) < 4: a quotient in [1, 2) is no closer than
//    2^-105 / d to the midpoint of two doubles, and the error of y moves the
//    sum by 2^-107 d (1 + 2 e) at most (in [1/2, 1) both are half as large).
//    A Newton step from 2^-47 has e < 2^-41, which leaves the d within 2^11
//    ulps below 2.  There every second 1/d lies a hair above a midpoint, and
//    the step, whose error is to the lower side, may round it down:
//    recip_root and recip_nearest see to these.
// Every function of the trace exists in two forms.  The plain form (kPlain
// true) runs these alone and notes in a Range what could have left their
// range; a wave votes once on its lanes' Ranges, and only if one left it is
// the work done again, by the whole wave, in the full form, whose roots and
// divisions are the compiler's sequences.  The full form (overflow, rays that
// leave an asphere's domain) stays out of the plain form's registers.
//
// A Range is two running extremes in vector registers, an instruction or two
// per value noted: the compares and scalar masks of a test at each root cost
// the plan kernel of the analytic surfaces 11 % (1.93 against 1.73 ms for
// 1e7 rays through twelve interfaces).  What is noted:
//  * arguments of roots (a zero, a negative one, one below 2^-767, an
//    overflow, a NaN) and denominators;
//  * the exponents of a ray's x and y at each surface and of its final
//    velocity: nothing nonzero below 2^-383.  So x*x + y*y, whose root is
//    taken without a note of its own, is 0 (see off_axis) or at least 2^-766,
//    and no remainder n - d q of a quotient underflows.  (A difference of two doubles is 0 or at least an ulp of
//    theirs, so tiny values come only from tiny values; where a Newton
//    iterate alone is tiny, its slopes are lost beside the other terms.)
// ---------------------------------------------------------------------------
struct Range {
    uint32_t high = 0;           // largest high word noted
    int32_t low = 0;             // smallest exponent noted

    // w >= 1 expected: an overflow, a NaN or a negative w is out of range
    __device__ __forceinline__ void above(double w)
    {
        high = max(high, (uint32_t)__double2hiint(w));
    }
    // as above, and what is below 2^-767 too: its high word wraps round
    __device__ __forceinline__ void positive(double w)
    {
        high = max(high, (uint32_t)__double2hiint(w) - ((1023u - 767u) << 20));
    }
    __device__ __forceinline__ void not_tiny(double a, double b)
    {
        low = min(min(low, __builtin_amdgcn_frexp_exp(a)), __builtin_amdgcn_frexp_exp(b));
    }
    __device__ __forceinline__ void leave() { high = ~0u; }
    // roots' arguments from 2^-767 to 2^857, slopes' below 2^601
    __device__ __forceinline__ bool left() const { return high >= ((1023u + 601u) << 20); }
    // that, and nothing nonzero below 2^-383
    __device__ __forceinline__ bool plain() const { return !left() & (low >= -382); }
};


BT_DEV bool sqrt_in_plain_range(double x)
{
    return x >= 0x1p-767 && x <= 0x1.fffffffffffffp+1023;
}

// sqrt(x); h becomes 1/(2 sqrt(x)) to ~2^-47.
BT_DEV double sqrt_plain(double x, double& h)
{
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r;
    h = r * 0.5;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    return __builtin_fma(d, h, g);
}

// 1/d to within an ulp, from y0 = 1/d to ~2^-40 or better.
BT_DEV double recip_refine(double d, double y0)
{
    return __builtin_fma(y0, __builtin_fma(-d, y0, 1.0), y0);
}

// y with its last bit set.
BT_DEV double odd(double y)
{
    return __longlong_as_double(__double_as_longlong(y) | 1);
}

// 1/g for quotients by g = sqrt_plain(x, h).  Next below a power of two h is
// right to 2^-53, and g of all ones is the one whose reciprocal the step from
// an even 2h rounds down (from 2h = 1/g rounded down it stays there).
BT_DEV double recip_root(double g, double h) { return recip_refine(g, odd(h + h)); }

// 1/d for quotients by any d, from y0 = 1/d to ~2^-46: a second step, whose
// multiplier's last bit carries the one case (d of all ones) that it leaves on
// a midpoint over it.
BT_DEV double recip_nearest(double d, double y0)
{
    const double y = recip_refine(d, y0);
    return __builtin_fma(__builtin_fma(-d, y, 1.0), odd(y), y);
}

// 1/d to within an ulp.  With div_plain the steps are the compiler's division's,
// and so are the results.
BT_DEV double recip_plain(double d)
{
    return recip_refine(d, recip_refine(d, __builtin_amdgcn_rcp(d)));
}

// n/d from y = 1/d to within an ulp.
BT_DEV double div_plain(double n, double d, double y)
{
    const double q = n * y;
    return __builtin_fma(__builtin_fma(-d, q, n), y, q);
}

// As div_plain, with the quotient's sign right for n = +-0 too.
BT_DEV double div_plain_signed(double n, double d, double y)
{
    return __builtin_amdgcn_div_fixup(div_plain(n, d, y), d, n);
}

// 2^-200 <= |d| < 2^201, on the exponent bits (a scalar test where d is
// wave-uniform).
BT_DEV bool plain_exponent(double d)
{
    return (((uint32_t)__double2hiint(d) >> 20) & 0x7ffu) - (1023u - 200u) <= 400u;
}

// 1/sqrt(x), two roundings; g becomes sqrt(x).  (Not from h: next to 1 -- the
// root of a unit velocity's square -- g is often 1 - 2^-53, whose reciprocal
// rounds up from a hair above a midpoint, which the refinement of 2h misses.)
BT_DEV double rsqrt_plain(double x, double& g)
{
    double h;
    g = sqrt_plain(x, h);
    const double y = recip_plain(g);
    return __builtin_fma(__builtin_fma(-g, y, 1.0), y, y);
}

BT_DEV double cr_sqrt(double x)
{
    double h;
    if (__all(sqrt_in_plain_range(x))) return sqrt_plain(x, h);
    return __builtin_sqrt(x);
}

BT_DEV double cr_rsqrt(double x)                    // 1/sqrt(x): two roundings
{
    double root;
    if (__all(sqrt_in_plain_range(x))) return rsqrt_plain(x, root);
    return 1.0 / __builtin_sqrt(x);
}

// sqrt(x) and 1/sqrt(x) (two roundings) in either form; `root` becomes
// sqrt(x), the reciprocal of the result to an ulp, or 0 in the full form.
template <bool kPlain>
BT_DEV double root_of(double x, Range& rg)
{
    if constexpr (kPlain) {
        double h;
        rg.positive(x);
        return sqrt_plain(x, h);
    } else {
        return cr_sqrt(x);
    }
}

template <bool kPlain>
BT_DEV double recip_root_of(double x, double& root, Range& rg)
{
    if constexpr (kPlain) {
        rg.positive(x);
        return rsqrt_plain(x, root);
    } else {
        root = 0.0;
        return cr_rsqrt(x);
    }
}

// ---------------------------------------------------------------------------
// Bicubic table (src/table.cpp:42-158)
// ---------------------------------------------------------------------------
BT_DEV double spline1(double x, double v0, double v1, double d0, double d1)
{
    double a = 2*(v0-v1) + d0 + d1;
    double b = 3*(v1-v0) - 2*d0 - d1;
    double c = d0;
    double d = v0;
    return d + x*(c + x*(b + x*a));
}

BT_DEV double grad1(double x, double v0, double v1, double d0, double d1)
{
    double a = 2*(v0-v1) + d0 + d1;
    double b = 3*(v1-v0) - 2*d0 - d1;
    double c = d0;
    return c + x*(2*b + x*3*a);
}

// int(std::floor(u)) as baseline x86-64 evaluates it: NaN and values outside
// the int range become INT_MIN and fail the cell range test.  (The GPU's own
// conversion would map NaN to 0, a valid cell.)
BT_DEV int cell_index(double u)
{
    double f = floor(u);
    if (!(f >= -2147483648.0 && f < 2147483648.0)) return (int)0x80000000;
    return (int)f;
}

BT_DEV bool table_cell(SurfPtr s, double x, double y, int& ix, int& iy)
{
    ix = cell_index((x - s->p[0])/s->p[2]);
    iy = cell_index((y - s->p[1])/s->p[3]);
    return !(ix >= s->n1-1 || ix < 0 || iy >= s->n2-1 || iy < 0);
}

BT_DEV double table_eval(SurfPtr s, double x, double y)
{
    int ix, iy;
    if (!table_cell(s, x, y, ix, iy))
        return s->flags ? __builtin_nan("") : 0.0;
    const double dx = s->p[2], dy = s->p[3];
    const TablePtr z = (TablePtr)s->a0;
    const TablePtr zx = (TablePtr)s->a1;
    const TablePtr zy = (TablePtr)s->a2;
    const TablePtr zxy = (TablePtr)s->a3;
    double xgrid = s->p[0] + ix*dx;
    double ygrid = s->p[1] + iy*dy;
    double xfrac = (x - xgrid)/dx;
    double yfrac = (y - ygrid)/dy;
    const int64_t k0 = (int64_t)s->n1*iy + ix, k1 = k0 + s->n1;
    double val0 = spline1(xfrac, z[k0], z[k0+1], zx[k0]*dx, zx[k0+1]*dx);
    double val1 = spline1(xfrac, z[k1], z[k1+1], zx[k1]*dx, zx[k1+1]*dx);
    double der0 = spline1(xfrac, zy[k0], zy[k0+1], zxy[k0]*dx, zxy[k0+1]*dx);
    double der1 = spline1(xfrac, zy[k1], zy[k1+1], zxy[k1]*dx, zxy[k1+1]*dx);
    return spline1(yfrac, val0, val1, der0*dy, der1*dy);
}

BT_DEV void table_grad(SurfPtr s, double x, double y,
                       double& dzdx, double& dzdy)
{
    int ix, iy;
    if (!table_cell(s, x, y, ix, iy)) {
        double v = s->flags ? __builtin_nan("") : 0.0;
        dzdx = v; dzdy = v;
        return;
    }
    const double dx = s->p[2], dy = s->p[3];
    const TablePtr z = (TablePtr)s->a0;
    const TablePtr zx = (TablePtr)s->a1;
    const TablePtr zy = (TablePtr)s->a2;
    const TablePtr zxy = (TablePtr)s->a3;
    double xgrid = s->p[0] + ix*dx;
    double ygrid = s->p[1] + iy*dy;
    double xfrac = (x - xgrid)/dx;
    double yfrac = (y - ygrid)/dy;
    const int64_t k0 = (int64_t)s->n1*iy + ix, k1 = k0 + s->n1;
    // the 16 table values of the cell, each read once
    const double z00 = z[k0], z01 = z[k0+1], z10 = z[k1], z11 = z[k1+1];
    const double x00 = zx[k0], x01 = zx[k0+1], x10 = zx[k1], x11 = zx[k1+1];
    const double y00 = zy[k0], y01 = zy[k0+1], y10 = zy[k1], y11 = zy[k1+1];
    const double c00 = zxy[k0], c01 = zxy[k0+1], c10 = zxy[k1], c11 = zxy[k1+1];

    double val0 = grad1(xfrac, z00, z01, x00*dx, x01*dx);
    double val1 = grad1(xfrac, z10, z11, x10*dx, x11*dx);
    double der0 = grad1(xfrac, y00, y01, c00*dx, c01*dx);
    double der1 = grad1(xfrac, y10, y11, c10*dx, c11*dx);
    dzdx = spline1(yfrac, val0, val1, der0*dy, der1*dy)/dx;

    val0 = grad1(yfrac, z00, z10, y00*dy, y10*dy);
    val1 = grad1(yfrac, z01, z11, y01*dy, y11*dy);
    der0 = grad1(yfrac, x00, x10, c00*dy, c10*dy);
    der1 = grad1(yfrac, x01, x11, c01*dy, c11*dy);
    dzdy = spline1(xfrac, val0, val1, der0*dx, der1*dx)/dy;
}

// ---------------------------------------------------------------------------
// 2-D Horner (src/polynomialSurface.cpp:50-66)
// ---------------------------------------------------------------------------
// A table's steps as one stream of quads (bt_poly_stream): rows from the last
// down, each row's coefficients from its last down, with +0.0 in front to a
// multiple of four; bit k of `row_ends` says that a row ends with quad k, and
// its highest bit is the last quad's.  The argument below makes the steps over
// the +0.0 in front exact.  A quad is one 32-byte scalar load, issued while the
// quad before it is used (the stream has one quad more than its steps); two
// quads per pass, so that no register is copied.  The loop over single
// coefficients waits for a load and runs eight scalar instructions for its two
// of FP64, which left the Sum kernels' SIMDs idle a third to two thirds of the
// time.  Plan kernels with it, with one quad per pass and with two, same card
// and clocks: 704, 587, 573 us (1e6 rays, three perturbed mirrors), 1071, 934,
// 916 (3e6, conic start), 461, 311, 303 (3e5, freeform), 764, 635, 623 (the
// batched trace of 1.1e6).  The two gradients' streams side by side in one loop,
// or all three tables' as one stream, were 3 to 9 % slower on the freeform
// (scalar registers spill; more scalar work per quad).
BT_DEV double horner2d_stream(double x, double y, CoefPtr c, uint64_t row_ends)
{
    double r = 0.0, h = 0.0;
    auto quad = [&](double k0, double k1, double k2, double k3) {
        h *= y; h += k0;
        h *= y; h += k1;
        h *= y; h += k2;
        h *= y; h += k3;
        if (row_ends & 1) {
            asm volatile("");                    // a branch, not six selects
            r *= x;
            r += h;
            h = 0.0;
        }
        row_ends >>= 1;
    };
    double c0 = c[0], c1 = c[1], c2 = c[2], c3 = c[3];
    __builtin_amdgcn_s_waitcnt(0xc07f);          // lgkmcnt(0): else each pass waits up front
    for (;;) {
        const double d0 = c[4], d1 = c[5], d2 = c[6], d3 = c[7];
        __builtin_amdgcn_sched_barrier(0);
        quad(c0, c1, c2, c3);
        if (!row_ends) break;
        c0 = c[8]; c1 = c[9]; c2 = c[10]; c3 = c[11];
        c += 8;
        __builtin_amdgcn_sched_barrier(0);
        quad(d0, d1, d2, d3);
        if (!row_ends) break;
    }
    return r;
}

// horner2d over trimmed bounds.  `trim` holds the last row with a
// coefficient other than +0.0 (-1 if none), then each row's length up to
// its last such coefficient; without it the loops run over all of the table.
// The full loop starts each row (and the outer sum) from 0.0 and, over a run
// of +0.0 coefficients with a finite argument, stays exactly +0.0:
// (+-0)*y + (+0) == +0.  Starting after such a run from 0.0 therefore gives
// the same bits, and rows of only +0.0 add exactly +0.0 where the full loop
// does.  A wave with any non-finite argument (0*inf is NaN inside the skipped
// steps) runs the full loop.
BT_DEV double horner2d(double x, double y, CoefPtr c, int nx, int ny, TrimPtr trim)
{
    double r = 0.0;
    for (int i = trim ? trim[0] : ny-1; i >= 0; i--) {
        const CoefPtr row = c + (int64_t)i*nx;
        double h = 0.0;
        for (int j = (trim ? trim[1 + i] : nx) - 1; j >= 0; j--) { h *= y; h += row[j]; }
        r *= x;
        r += h;
    }
    return r;
}

// Table `which` (0: coefficients, 1, 2: x and y gradients) of a POLYNOMIAL
// record at (u, v) from its origin; `finite`: all of the wave's u and v are.
// The record's optional a3: trim tables of the three, in that order, then
// (flag BT_POLY_STREAMS) their streams' bt_poly_stream and the streams.
BT_DEV double poly_table(SurfPtr s, int which, double u, double v, bool finite)
{
    const int n2 = s->n2;
    TrimPtr trim = (TrimPtr)reinterpret_cast<const int*>(s->a3);
    if (!finite) trim = nullptr;
    if (trim) {
        if (s->flags & BT_POLY_STREAMS) {
            const TrimPtr head = trim + ((1 + 3*n2 + 15) & ~15);
            const StreamPtr st = (StreamPtr)head + which;
            const uint64_t row_ends = st->row_ends;
            if (row_ends)
                return horner2d_stream(u, v, (CoefPtr)(head + 16) + st->first, row_ends);
        }
        if (which > 0) trim += 1 + n2 + (which - 1)*n2;
    }
    const CoefPtr c = (CoefPtr)(which == 0 ? s->a0 : which == 1 ? s->a1 : s->a2);
    return horner2d(u, v, c, s->n1 - (which > 0), n2 - (which > 0), trim);
}

// A value that is the same in every lane, in scalar registers.
BT_DEV double wave_value(double v)
{
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Sag and / or normal of a Bicubic at one point (bicubic.cpp:19-40), sharing
// the cell and its 16 table values; each result is bit-identical to
// table_eval's and table_grad's.  `inv`: 1/nz to an ulp, or 0.  With the
// record's optional reciprocals of the grid steps the four (sag) or six
// (normal) divisions by dx and dy, ten at a point of a Newton iteration, are
// three or four instructions each.
template <bool kPlain, bool kSag, bool kNormal>
BT_DEV void table_point(SurfPtr s, double x, double y, double& sag, double& nx,
                        double& ny, double& nz, double& inv, Range& rg)
{
    if constexpr (!kPlain) {
        if constexpr (kSag) sag = table_eval(s, x, y);
        if constexpr (kNormal) {
            double dzdx, dzdy;
            table_grad(s, x, y, dzdx, dzdy);
            inv = 0.0;
            if (__builtin_isnan(dzdx)) {
                nx = __builtin_nan(""); ny = nx; nz = nx;
            } else {
                nz = cr_rsqrt(1 + dzdx*dzdx + dzdy*dzdy);
                nx = -dzdx*nz;
                ny = -dzdy*nz;
            }
        }
    } else {
        if (s->n1 < 2 || s->n2 < 2) {                // no cell to read
            rg.leave();
            if constexpr (kSag) sag = 0.0;
            if constexpr (kNormal) { nx = 0.0; ny = 0.0; nz = 1.0; inv = 1.0; }
            return;
        }
        const double dx = s->p[2], dy = s->p[3];
        const double x0 = s->p[0], y0 = s->p[1];
        if (!plain_exponent(dx) || !plain_exponent(dy)) rg.leave();
        // not given (0), or not 1/dx and 1/dy to less than 2^-53, which the
        // correctly rounded ones are and the quotients need.  (Three perturbed
        // mirrors, 434,328 rays: 0.331 ms without them, 0.329 with; 0.69 when
        // the wave was sent to the full form, 0.47 with that form alone.  Kept in
        // vector registers the two cost records that give them 3 %.)
        double rx = s->p[4], ry = s->p[5];
        if (!(fabs(__builtin_fma(-dx, rx, 1.0)) < 0x1p-53)
            || !(fabs(__builtin_fma(-dy, ry, 1.0)) < 0x1p-53)) {
            rx = wave_value(recip_nearest(dx, recip_plain(dx)));
            ry = wave_value(recip_nearest(dy, recip_plain(dy)));
        }
        const double ux = x - x0, uy = y - y0;
        const double fx = floor(div_plain(ux, dx, rx)), fy = floor(div_plain(uy, dy, ry));
        const bool inside = (fx >= 0.0) & (fx < (double)(s->n1 - 1)) & (fy >= 0.0)
                            & (fy < (double)(s->n2 - 1));
        const TablePtr z = (TablePtr)s->a0;
        const TablePtr zx = (TablePtr)s->a1;
        const TablePtr zy = (TablePtr)s->a2;
        const TablePtr zxy = (TablePtr)s->a3;
        // a lane outside the table reads its first cell
        const int64_t k0 = inside ? (int64_t)s->n1*(int)fy + (int)fx : 0, k1 = k0 + s->n1;
        const double z00 = z[k0], z01 = z[k0+1], z10 = z[k1], z11 = z[k1+1];
        const double x00 = zx[k0], x01 = zx[k0+1], x10 = zx[k1], x11 = zx[k1+1];
        const double y00 = zy[k0], y01 = zy[k0+1], y10 = zy[k1], y11 = zy[k1+1];
        const double c00 = zxy[k0], c01 = zxy[k0+1], c10 = zxy[k1], c11 = zxy[k1+1];
        const double xn = x - (x0 + fx*dx), yn = y - (y0 + fy*dy);
        const double xfrac = div_plain_signed(xn, dx, rx);
        const double yfrac = div_plain_signed(yn, dy, ry);
        double ts = 0.0, dzdx = 0.0, dzdy = 0.0;
        if constexpr (kSag) {
            double val0 = spline1(xfrac, z00, z01, x00*dx, x01*dx);
            double val1 = spline1(xfrac, z10, z11, x10*dx, x11*dx);
            double der0 = spline1(xfrac, y00, y01, c00*dx, c01*dx);
            double der1 = spline1(xfrac, y10, y11, c10*dx, c11*dx);
            ts = spline1(yfrac, val0, val1, der0*dy, der1*dy);
        }
        if constexpr (kNormal) {
            double val0 = grad1(xfrac, z00, z01, x00*dx, x01*dx);
            double val1 = grad1(xfrac, z10, z11, x10*dx, x11*dx);
            double der0 = grad1(xfrac, y00, y01, c00*dx, c01*dx);
            double der1 = grad1(xfrac, y10, y11, c10*dx, c11*dx);
            const double gx = spline1(yfrac, val0, val1, der0*dy, der1*dy);
            val0 = grad1(yfrac, z00, z10, y00*dy, y10*dy);
            val1 = grad1(yfrac, z01, z11, y01*dy, y11*dy);
            der0 = grad1(yfrac, x00, x10, c00*dy, c10*dy);
            der1 = grad1(yfrac, x01, x11, c01*dy, c11*dy);
            const double gy = spline1(xfrac, val0, val1, der0*dx, der1*dx);
            dzdx = div_plain_signed(gx, dx, rx);
            dzdy = div_plain_signed(gy, dy, ry);
            rg.not_tiny(gx, gy);
        }
        if (!__all(inside)) {                        // outside: NaN or 0 (table.cpp:60-66)
            const double v = s->flags ? __builtin_nan("") : 0.0;
            ts = inside ? ts : v;
            dzdx = inside ? dzdx : v;
            dzdy = inside ? dzdy : v;
        }
        if constexpr (kSag) sag = ts;
        if constexpr (kNormal) {
            const double w = 1 + dzdx*dzdx + dzdy*dzdy;
            rg.above(__builtin_fmax(w, 1.0));        // NaN slopes (outside): a NaN normal
            nz = rsqrt_plain(w, inv);
            nx = -dzdx*nz;
            ny = -dzdy*nz;
        }
    }
}

// ---------------------------------------------------------------------------
// Quadric family (src/quadric.cpp, src/asphere.cpp)
// ---------------------------------------------------------------------------
// result + sum of an Asphere's n even terms c[i] r2^(i+1) (asphere.cpp:37-46),
// or its slope's dc[i] r r2^i (asphere.cpp:53-59): term starts at the first
// power and grows by r2.  (All coefficients in one 64-byte scalar load
// instead of a load per term: the same time on the analytic kernel, 4 % more
// on the Sum kernels, whose scalar registers are short.)
BT_DEV double even_terms(CoefPtr c, int n, double result, double term, double r2)
{
    // n anew for each evaluation: a test of it shared by two Newton loops is
    // kept as a mask of the lanes active in the first, which may have none in
    // common with those of the second, and then no terms reads as some
    asm volatile("" : "+s"(n));
    for (int i = 0; i < n; i++) {
        result += c[i]*term;
        term *= r2;
    }
    return result;
}

// x*x + y*y for the plain form's root.  A ray at the vertex (0) goes on with
// 2^-767, whose slopes are lost beside 1: the normal is (+-0, +-0, 1), and
// arrival_normal gives the zeros their sign, which nothing before depends on.
// The chief ray of every centred field meets the vertices; while its wave ran
// the full form after the plain one, 49 rays through twelve interfaces took 68
// us, 38 in the full form alone, 34 now (with three perturbed mirrors 181, 122,
// 81).  Others pay 1 % (a NaN is taken for 2^-767, too, but no ray gets here
// with one before a root of its discriminant or sag was noted).
BT_DEV double off_axis(double r2) { return __builtin_fmax(r2, 0x1p-767); }

// Sag and / or normal of a Quadric (kAsphere false) or an Asphere (true) at
// one point: quadric.cpp:18-39, asphere.cpp:37-62.  `inv`: 1/nz to an ulp,
// or 0.  Bound by FP64 issue: the normal's three divisions start from the
// roots' own h here (the reciprocal of its third root does not: rsqrt_plain).
template <bool kPlain, bool kAsphere, bool kSag, bool kNormal>
BT_DEV void conic_point(SurfPtr s, double x, double y, double& sag, double& nx,
                        double& ny, double& nz, double& inv, Range& rg)
{
    const double R = s->p[0], cp1R2 = s->p[8];
    const double r2 = x*x + y*y;
    if constexpr (kPlain) {
        if (!plain_exponent(R)) rg.leave();
        if constexpr (kSag) {
            const double v = 1.-r2*cp1R2;
            rg.positive(v);
            double h;
            const double d = R*(1.+sqrt_plain(v, h));
            sag = div_plain(r2, d, recip_plain(d));
            if constexpr (kAsphere) sag = even_terms((CoefPtr)s->a0, s->n1, sag, r2, r2);
        }
        if constexpr (kNormal) {
            double hr, hu;
            const double r = sqrt_plain(off_axis(r2), hr);
            const double u = 1-r*r*cp1R2;
            const double d = R*sqrt_plain(u, hu);
            const double y0 = (hu + hu) * (R*s->p[3]);   // 1/sqrt(u) * (R * 1/R/R)
            double dzdr = div_plain(r, d, recip_nearest(d, y0));
            if constexpr (kAsphere) dzdr = even_terms((CoefPtr)s->a1, s->n1, dzdr, r, r*r);
            const double w = 1+dzdr*dzdr;
            rg.above(w);                                 // a NaN for u = 0
            nz = rsqrt_plain(w, inv);
            const double yr = recip_root(r, hr);
            nx = -div_plain_signed(x, r, yr)*dzdr*nz;
            ny = -div_plain_signed(y, r, yr)*dzdr*nz;
        }
    } else {
        if constexpr (kSag) {
            sag = R != 0 ? r2/(R*(1.+cr_sqrt(1.-r2*cp1R2))) : 0.0;
            if constexpr (kAsphere) sag = even_terms((CoefPtr)s->a0, s->n1, sag, r2, r2);
        }
        if constexpr (kNormal) {
            const double r = cr_sqrt(r2);
            inv = 0.0;
            if (r == 0.0) {
                nx = 0.0; ny = 0.0; nz = 1.0;
            } else {
                double dzdr = R != 0.0 ? r/(R*cr_sqrt(1-r*r*cp1R2)) : 0.0;
                if constexpr (kAsphere)
                    dzdr = even_terms((CoefPtr)s->a1, s->n1, dzdr, r, r*r);
                nz = cr_rsqrt(1+dzdr*dzdr);
                nx = -x/r*dzdr*nz;
                ny = -y/r*dzdr*nz;
            }
        }
    }
}

// Normal of a Sphere (sphere.cpp:23-35, 66-69).
template <bool kPlain>
BT_DEV void sphere_normal(SurfPtr s, double x, double y, double& nx, double& ny,
                          double& nz, double& inv, Range& rg)
{
    const double Rinv = s->p[2];
    const double rsqr = x*x + y*y;
    if constexpr (kPlain) {
        double hr, hu;
        const double r = sqrt_plain(off_axis(rsqr), hr);
        const double rat = r*Rinv;
        const double u = 1-rat*rat;
        const double su = sqrt_plain(u, hu);
        const double dzdr = div_plain(rat, su, recip_root(su, hu));
        const double w = 1+dzdr*dzdr;
        if (!plain_exponent(Rinv)) rg.leave();
        rg.above(w);                                     // a NaN for u = 0
        nz = rsqrt_plain(w, inv);
        const double yr = recip_root(r, hr);
        nx = -div_plain_signed(x, r, yr)*dzdr*nz;
        ny = -div_plain_signed(y, r, yr)*dzdr*nz;
    } else {
        inv = 0.0;
        if (s->p[0] == 0.0 || rsqr == 0.0) {
            nx = 0.0; ny = 0.0; nz = 1.0;
        } else {
            const double r = cr_sqrt(rsqr);
            const double rat = r*Rinv;
            const double dzdr = rat/cr_sqrt(1-rat*rat);
            nz = cr_rsqrt(1+dzdr*dzdr);
            nx = -x/r*dzdr*nz;
            ny = -y/r*dzdr*nz;
        }
    }
}

BT_DEV bool finite_wave(double u, double v)
{
    return __all(__builtin_isfinite(u) && __builtin_isfinite(v));
}

BT_DEV double poly_sag(SurfPtr s, double x, double y)
{                                                    // polynomialSurface.cpp:35-37
    const double u = x-s->p[0], v = y-s->p[1];
    return poly_table(s, 0, u, v, finite_wave(u, v));
}

// polynomialSurface.cpp:35-48
template <bool kPlain, bool kSag>
BT_DEV void poly_point(SurfPtr s, double x, double y, double& sag, double& nx, double& ny,
                       double& nz, double& inv, Range& rg)
{
    const double u = x-s->p[0], v = y-s->p[1];
    const bool finite = finite_wave(u, v);
    if constexpr (kSag) sag = poly_table(s, 0, u, v, finite);
    double gx = -poly_table(s, 1, u, v, finite);
    double gy = -poly_table(s, 2, u, v, finite);
    nz = recip_root_of<kPlain>(gx*gx + gy*gy + 1, inv, rg);
    nx = gx*nz;
    ny = gy*nz;
}

// ---------------------------------------------------------------------------
// Surface kinds a kernel is compiled for.
//  * kKindsAll: every kind, Sums of any children (a switch over the kind of
//    each child inside the Sum's loop);
//  * kKindsAnalytic: Plane, Sphere, Paraboloid, Quadric, Asphere and Tilted,
//    no Sums -- the Bicubic, polynomial and Sum code paths are left out,
//    which lets a plan kernel for such optics keep far fewer registers;
//  * kKindsSumAPB: those analytic leaves plus Sums of exactly (Asphere,
//    Polynomial, Bicubic), in that order (a perturbed conic mirror: figure,
//    low-order Zernike error, measured high-frequency map).  The Sum's three
//    children are evaluated by their own functions with no kind switch, so
//    each Newton step carries only the registers those three need;
//  * kKindsFlatSums: every kind, Sums whose children are all leaves (the
//    evaluation of nested Sums is left out: it costs the one-level Sum path
//    registers).
// kKindsAll also evaluates Sums of Sums, to kMaxSumDepth levels below a Sum.
// Under a restricted set any other kind (or Sum layout) evaluates to NaN and
// so fails.
// ---------------------------------------------------------------------------
constexpr int kKindsAll = 0;
constexpr int kKindsAnalytic = 1;
constexpr int kKindsSumAPB = 2;
constexpr int kKindsFlatSums = 3;

// Kind sets whose interactions run plain first.  kKindsAll, whose nested Sums
// are inlined to three levels, keeps the full form alone: two forms of it
// would double the largest kernels for the rarest optics.
template <int K>
constexpr bool kVoted = K != kKindsAll;

// The kind set of leaves (records that are not Sums) under set K.
constexpr int leaf_set(int K)
{
    return (K == kKindsAll || K == kKindsFlatSums) ? kKindsAll : kKindsAnalytic;
}

// A Sum record laid out as kKindsSumAPB requires (records s+1..s+3 follow it).
BT_DEV bool sum_is_apb(SurfPtr s)
{
    return s->nchild == 3 && s[1].kind == BT_ASPHERE && s[2].kind == BT_POLYNOMIAL &&
           s[3].kind == BT_BICUBIC;
}

// ---------------------------------------------------------------------------
// Leaf surfaces: sag and normal.  `inv` beside a normal is 1/nz to an ulp in
// the plain form: a Sum's slopes nx/nz and ny/nz start from it.
// ---------------------------------------------------------------------------
template <int K, bool kPlain>
BT_DEV double leaf_sag(SurfPtr s, double x, double y, Range& rg)
{
    double sag, nx, ny, nz, inv;
    switch (s->kind) {
    case BT_PLANE:                                   // plane.cpp:15-17
        return 0.0;
    case BT_SPHERE:                                  // sphere.cpp:17-21
        if (s->p[0] != 0)
            return s->p[0]*(1-root_of<kPlain>(1-(x*x + y*y)*s->p[3], rg));
        return 0.0;
    case BT_PARABOLOID:                              // paraboloid.cpp:17-23
        if (s->p[0] != 0) {
            double r2 = x*x + y*y;
            return r2*s->p[2];
        }
        return 0.0;
    case BT_QUADRIC:                                 // quadric.cpp:18-25
        conic_point<kPlain, false, true, false>(s, x, y, sag, nx, ny, nz, inv, rg);
        return sag;
    case BT_ASPHERE:                                 // asphere.cpp:37-46
        conic_point<kPlain, true, true, false>(s, x, y, sag, nx, ny, nz, inv, rg);
        return sag;
    case BT_TILTED:                                  // tilted.cpp:16-18
        return x*s->p[0] + y*s->p[1];
    case BT_BICUBIC:                                 // bicubic.cpp:19-21
        if constexpr (K == kKindsAll) {
            table_point<kPlain, true, false>(s, x, y, sag, nx, ny, nz, inv, rg);
            return sag;
        }
        break;
    case BT_POLYNOMIAL:                              // polynomialSurface.cpp:35-37
        if constexpr (K == kKindsAll) return poly_sag(s, x, y);
        break;
    }
    return __builtin_nan("");
}

template <int K, bool kPlain>
BT_DEV void leaf_normal(SurfPtr s, double x, double y,
                        double& nx, double& ny, double& nz, double& inv, Range& rg)
{
    double sag;
    inv = 0.0;
    switch (s->kind) {
    case BT_PLANE:                                   // plane.cpp:19-23
        nx = 0.0; ny = 0.0; nz = 1.0; inv = 1.0;
        return;
    case BT_SPHERE:                                  // sphere.cpp:23-35, 66-69
        sphere_normal<kPlain>(s, x, y, nx, ny, nz, inv, rg);
        return;
    case BT_PARABOLOID: {                            // paraboloid.cpp:25-37
        if (s->p[0] == 0) {
            nx = 0.0; ny = 0.0; nz = 1.0; inv = 1.0;
        } else {
            const double Rinv = s->p[1];
            nz = recip_root_of<kPlain>(1+(x*x+y*y)*Rinv*Rinv, inv, rg);
            nx = -x*Rinv*nz;
            ny = -y*Rinv*nz;
        }
        return;
    }
    case BT_QUADRIC:                                 // quadric.cpp:27-39
        conic_point<kPlain, false, false, true>(s, x, y, sag, nx, ny, nz, inv, rg);
        return;
    case BT_ASPHERE:                                 // asphere.cpp:48-62
        conic_point<kPlain, true, false, true>(s, x, y, sag, nx, ny, nz, inv, rg);
        return;
    case BT_TILTED: {                                // tilted.cpp:20-27
        const double tx = s->p[0], ty = s->p[1];
        nx = -tx;
        ny = -ty;
        nz = root_of<kPlain>(1 - tx*tx - ty*ty, rg);
        if constexpr (kPlain) inv = recip_plain(nz);
        return;
    }
    case BT_BICUBIC:                                 // bicubic.cpp:23-40
        if constexpr (K == kKindsAll) {
            table_point<kPlain, false, true>(s, x, y, sag, nx, ny, nz, inv, rg);
            return;
        }
        break;
    case BT_POLYNOMIAL:                              // polynomialSurface.cpp:39-48
        if constexpr (K == kKindsAll) {
            poly_point<kPlain, false>(s, x, y, sag, nx, ny, nz, inv, rg);
            return;
        }
        break;
    }
    nx = __builtin_nan(""); ny = nx; nz = nx;
}

// Sag and / or normal at one point (the reference evaluates them separately;
// the results here are bit-identical, with shared work evaluated once).
template <int K, bool kPlain, bool kSag, bool kNormal>
BT_DEV void leaf_point(SurfPtr s, double x, double y, double& sag,
                       double& nx, double& ny, double& nz, double& inv, Range& rg)
{
    if constexpr (kSag && kNormal) {
        if (s->kind == BT_ASPHERE) {
            conic_point<kPlain, true, true, true>(s, x, y, sag, nx, ny, nz, inv, rg);
            return;
        }
        if constexpr (K == kKindsAll) {
            if (s->kind == BT_BICUBIC) {
                table_point<kPlain, true, true>(s, x, y, sag, nx, ny, nz, inv, rg);
                return;
            }
            if (s->kind == BT_POLYNOMIAL) {
                poly_point<kPlain, true>(s, x, y, sag, nx, ny, nz, inv, rg);
                return;
            }
        }
    }
    if constexpr (kSag) sag = leaf_sag<K, kPlain>(s, x, y, rg);
    if constexpr (kNormal) leaf_normal<K, kPlain>(s, x, y, nx, ny, nz, inv, rg);
}

// sx += nx/nz, sy += ny/nz; plain: from inv = 1/nz to an ulp, whose step is
// right but for an nz of all ones, which no rounded reciprocal of a root is
// (between 1 and 1 + 2^-52 there is no double); a Tilted's inv is right there.
template <bool kPlain>
BT_DEV void add_slope(double& sx, double& sy, double nx, double ny, double nz, double inv)
{
    if constexpr (kPlain) {
        const double y = recip_refine(nz, inv);
        sx += div_plain(nx, nz, y);                  // the sign of a zero term is lost in
        sy += div_plain(ny, nz, y);                  // sums that start from +0
    } else {
        sx += nx/nz;
        sy += ny/nz;
    }
}

template <bool kPlain>
BT_DEV void sum_normal_from_slopes(double sx, double sy, double& nx, double& ny, double& nz,
                                   Range& rg)
{
    const double w = sx*sx + sy*sy + 1;
    if constexpr (kPlain) {
        double root;
        rg.above(__builtin_fmax(w, 1.0));            // a child's NaN slopes: a NaN normal
        nz = rsqrt_plain(w, root);
    } else {
        nz = cr_rsqrt(w);
    }
    nx = sx*nz;
    ny = sy*nz;
}

// Sums of any kinds (kKindsAll).  A Sum record is followed by its children,
// each a leaf record or a Sum with its own subtree; a Sum's n1 counts the
// records below it, so the next sibling starts 1 + n1 records on.  Children
// that are Sums are evaluated by the same rules (sum.cpp:23-45 calls the
// child's own sag / normal), to kMaxSumDepth levels of nesting below a Sum
// (the host refuses deeper trees; a deeper child evaluates to NaN).
constexpr int kMaxSumDepth = 3;

BT_DEV SurfPtr next_child(SurfPtr c)
{
    return c + (c->kind == BT_SUM ? 1 + c->n1 : 1);
}

template <int D, bool kPlain, bool kSag, bool kNormal>
BT_DEV void sum_point_all(SurfPtr s, double x, double y, double& sag,
                          double& nx, double& ny, double& nz, Range& rg)
{                                                    // sum.cpp:23-45
    double result = 0.0, sx = 0.0, sy = 0.0, ts, tnx, tny, tnz, inv;
    SurfPtr c = s + 1;
    const int nc = s->nchild;
    for (int i = 0; i < nc; i++, c = next_child(c)) {
        if (c->kind != BT_SUM) {
            leaf_point<kKindsAll, kPlain, kSag, kNormal>(c, x, y, ts, tnx, tny, tnz, inv, rg);
        } else {
            inv = 0.0;
            if constexpr (D > 0)
                sum_point_all<D - 1, kPlain, kSag, kNormal>(c, x, y, ts, tnx, tny, tnz, rg);
            else { ts = __builtin_nan(""); tnx = ts; tny = ts; tnz = ts; }
        }
        if constexpr (kSag) result += ts;
        if constexpr (kNormal) add_slope<kPlain>(sx, sy, tnx, tny, tnz, inv);
    }
    if constexpr (kSag) sag = result;
    if constexpr (kNormal) sum_normal_from_slopes<kPlain>(sx, sy, nx, ny, nz, rg);
}

// A Sum whose layout sum_is_apb has accepted.
template <bool kPlain, bool kSag, bool kNormal>
BT_DEV void apb_point(SurfPtr s, double x, double y, double& sag,
                      double& nx, double& ny, double& nz, Range& rg)
{
    double result = 0.0, sx = 0.0, sy = 0.0, ts, tnx, tny, tnz, inv;
    conic_point<kPlain, true, kSag, kNormal>(s + 1, x, y, ts, tnx, tny, tnz, inv, rg);
    if constexpr (kSag) result += ts;
    if constexpr (kNormal) add_slope<kPlain>(sx, sy, tnx, tny, tnz, inv);
    if constexpr (kNormal) {
        poly_point<kPlain, kSag>(s + 2, x, y, ts, tnx, tny, tnz, inv, rg);
        if constexpr (kSag) result += ts;
        add_slope<kPlain>(sx, sy, tnx, tny, tnz, inv);
    }
    if constexpr (kSag && !kNormal) result += poly_sag(s + 2, x, y);
    table_point<kPlain, kSag, kNormal>(s + 3, x, y, ts, tnx, tny, tnz, inv, rg);
    if constexpr (kSag) sag = result + ts;
    if constexpr (kNormal) {
        add_slope<kPlain>(sx, sy, tnx, tny, tnz, inv);
        sum_normal_from_slopes<kPlain>(sx, sy, nx, ny, nz, rg);
    }
}

// Sum records are followed by their children (sum.cpp:23-45).  The Sum's
// sag is 0 + child sags in child order, its normal from the sum of the
// children's slopes (-n_x/n_z, -n_y/n_z) in child order, so the unrolled
// kKindsSumAPB form is the same operations as the loops.
template <int K, bool kPlain, bool kSag, bool kNormal>
BT_DEV void surf_point(SurfPtr s, double x, double y, double& sag,
                       double& nx, double& ny, double& nz, Range& rg)
{
    constexpr int L = leaf_set(K);
    double inv;
    if (K == kKindsAnalytic || s->kind != BT_SUM) {
        leaf_point<L, kPlain, kSag, kNormal>(s, x, y, sag, nx, ny, nz, inv, rg);
        return;
    }
    if constexpr (K == kKindsSumAPB) {
        if (sum_is_apb(s)) {
            apb_point<kPlain, kSag, kNormal>(s, x, y, sag, nx, ny, nz, rg);
        } else {
            const double nan = __builtin_nan("");
            if constexpr (kSag) sag = nan;
            if constexpr (kNormal) { nx = nan; ny = nan; nz = nan; }
        }
    } else if constexpr (K == kKindsFlatSums) {
        double result = 0.0, sx = 0.0, sy = 0.0, ts, tnx, tny, tnz;
        const int nc = s->nchild;
        for (int i = 0; i < nc; i++) {
            leaf_point<L, kPlain, kSag, kNormal>(s + 1 + i, x, y, ts, tnx, tny, tnz, inv, rg);
            if constexpr (kSag) result += ts;
            if constexpr (kNormal) add_slope<kPlain>(sx, sy, tnx, tny, tnz, inv);
        }
        if constexpr (kSag) sag = result;
        if constexpr (kNormal) sum_normal_from_slopes<kPlain>(sx, sy, nx, ny, nz, rg);
    } else if constexpr (K == kKindsAll) {
        sum_point_all<kMaxSumDepth, kPlain, kSag, kNormal>(s, x, y, sag, nx, ny, nz, rg);
    }
}

// Sag alone and normal alone, for callers without an interaction's vote.
template <int K = kKindsAll>
BT_DEV double surf_sag(SurfPtr s, double x, double y)
{
    double sag, nx, ny, nz;
    Range rg;
    surf_point<K, false, true, false>(s, x, y, sag, nx, ny, nz, rg);
    return sag;
}

template <int K = kKindsAll>
BT_DEV void surf_normal(SurfPtr s, double x, double y,
                        double& nx, double& ny, double& nz)
{
    double sag;
    Range rg;
    surf_point<K, false, false, true>(s, x, y, sag, nx, ny, nz, rg);
}

// Surface evaluators for the Newton loops.  SurfEval<K> dispatches on the
// record's kind at every evaluation; where the caller already knows the kind
// (an Asphere leaf, a Sum laid out as kKindsSumAPB requires) the loop is
// instantiated with that kind's functions directly, so it carries no switch
// over the other kinds.  Every evaluator computes exactly what surf_point
// computes for that record.  kGrid: the record may hold a Bicubic, whose sag
// is NaN off its grid.
template <int K>
struct SurfEval {
    static constexpr bool kGrid = K != kKindsAnalytic;
    template <bool kPlain, bool kSag, bool kNormal>
    static BT_DEV void point(SurfPtr s, double x, double y, double& sag,
                             double& nx, double& ny, double& nz, Range& rg)
    {
        surf_point<K, kPlain, kSag, kNormal>(s, x, y, sag, nx, ny, nz, rg);
    }
};

// A record known to be a leaf (not a Sum).
template <int K>
struct LeafEval {
    static constexpr bool kGrid = K == kKindsAll;
    template <bool kPlain, bool kSag, bool kNormal>
    static BT_DEV void point(SurfPtr s, double x, double y, double& sag,
                             double& nx, double& ny, double& nz, Range& rg)
    {
        double inv;
        leaf_point<K, kPlain, kSag, kNormal>(s, x, y, sag, nx, ny, nz, inv, rg);
    }
};

struct AsphereEval {                                 // asphere.cpp:37-62
    static constexpr bool kGrid = false;
    template <bool kPlain, bool kSag, bool kNormal>
    static BT_DEV void point(SurfPtr s, double x, double y, double& sag,
                             double& nx, double& ny, double& nz, Range& rg)
    {
        double inv;
        conic_point<kPlain, true, kSag, kNormal>(s, x, y, sag, nx, ny, nz, inv, rg);
    }
};

struct SumAPBEval {                                  // sum.cpp:23-45
    static constexpr bool kGrid = true;
    template <bool kPlain, bool kSag, bool kNormal>
    static BT_DEV void point(SurfPtr s, double x, double y, double& sag,
                             double& nx, double& ny, double& nz, Range& rg)
    {
        apb_point<kPlain, kSag, kNormal>(s, x, y, sag, nx, ny, nz, rg);
    }
};

// Record `s` with every test of its fields made anew.  A wave-uniform test (the
// kind, a count, an optional table) that two Newton loops share can be kept as a
// mask of the lanes active in the first one's last iteration, which may have
// none in common with those of the second; true then reads as false, and a table
// that is not there is read (the count of an Asphere's terms was shared like
// that: see even_terms).  So a Sum's first child is iterated by a pointer of its
// own, and so is what follows a loop on the same record.  Inside one loop lanes
// only leave, so that a mask holds all that come after.  (Shorter lives of
// scalar registers, too: 614 -> 599 us for 1e6 rays, three perturbed mirrors;
// 313 either way for the freeform.)
BT_DEV SurfPtr anew(SurfPtr s)
{
    asm volatile("" : "+s"(s));
    return s;
}

BT_DEV bool same_bits(double a, double b)
{
    return __double_as_longlong(a) == __double_as_longlong(b);
}

// Tangent-plane Newton with exactly `niter` iterations (surface.cpp:22-49).
//
// Each iteration is a pure function of dt (the ray origin and direction are
// fixed): dt -> rP(dt), sag(rP), normal(rP) -> dt'.  So once an iterate
// repeats bit for bit -- a fixed point dt' == dt, or a two-cycle between
// neighbouring doubles dt'' == dt -- every remaining iterate is known, and the
// loop stops with exactly the state (dt, rP, sag) that running all `niter`
// iterations would leave.  Results are bit-identical to the full loop.
//
struct NormalMemo {              // the normal at the ray's point at dt
    double dt, nx, ny, nz;
    bool ok;
};

// The plain form evaluates sag and normal together at each iterate (roots'
// arguments, table cells and coefficient loads shared) and leaves the final
// point's normal for the reflection or refraction there.  The full form
// evaluates them apart, which needs fewer registers; its memo is the last
// normal evaluated, used where it belongs to the final point.
template <class Ev, bool kPlain>
BT_DEV bool newton(SurfPtr s, double x, double y, double z,
                   double vx, double vy, double vz, double& dt, int niter, Range& rg,
                   NormalMemo* memo = nullptr)
{
    double nx, ny, nz, sz, rPz, unused;
    double pdt = 0.0;            // the iterate before the current one (iter >= 1)
    if constexpr (kPlain) {
        bool last = niter <= 0;  // nothing is iterated from the current point
        for (int iter = 0;; iter++) {
            const double rPx = x+vx*dt;
            const double rPy = y+vy*dt;
            rPz = z+vz*dt;
            Ev::template point<true, true, true>(s, rPx, rPy, sz, nx, ny, nz, rg);
            if (last) break;
            double dtn = (rPx-x)*nx + (rPy-y)*ny + (sz-z)*nz;
            dtn /= (nx*vx + ny*vy + nz*vz);
            if (same_bits(dtn, dt)) break;        // fixed point: state unchanged
            // off a Bicubic's grid: every later iterate is NaN, and the ray
            // fails
            if (Ev::kGrid && !(dtn == dtn)) { sz = dtn; break; }
            // two-cycle: iterates alternate between the next point and this
            // one; the remaining niter-1-iter iterations end on the next
            // point if that count is even, else here
            const bool cycle = iter >= 1 && same_bits(dtn, pdt);
            if (cycle && ((niter - 1 - iter) & 1)) break;
            last = cycle || iter + 1 >= niter;
            pdt = dt;
            dt = dtn;
        }
        if (memo) *memo = NormalMemo{dt, nx, ny, nz, true};
    } else {
        double rPx = x+vx*dt;
        double rPy = y+vy*dt;
        rPz = z+vz*dt;
        Ev::template point<false, true, false>(s, rPx, rPy, sz, unused, unused, unused, rg);
        for (int iter = 0; iter < niter; iter++) {
            Ev::template point<false, false, true>(s, rPx, rPy, unused, nx, ny, nz, rg);
            if (memo) *memo = NormalMemo{dt, nx, ny, nz, true};
            double dtn = (rPx-x)*nx + (rPy-y)*ny + (sz-z)*nz;
            dtn /= (nx*vx + ny*vy + nz*vz);
            if (same_bits(dtn, dt)) break;
            const double odt = dt, oz = rPz, osz = sz;
            dt = dtn;
            rPx = x+vx*dt;
            rPy = y+vy*dt;
            rPz = z+vz*dt;
            Ev::template point<false, true, false>(s, rPx, rPy, sz, unused, unused, unused, rg);
            if (iter >= 1 && same_bits(dt, pdt)) {
                if ((niter - 1 - iter) & 1) { dt = odt; rPz = oz; sz = osz; }
                break;
            }
            pdt = odt;
        }
    }
    return fabs(sz-rPz) < 1e-12;
}

// std::max(a, b) = (a < b) ? b : a; std::min(a, b) = (b < a) ? b : a.
BT_DEV double pick_root(double vzR, double dt1, double dt2)
{
    if (vzR < 0) return (dt1 < dt2) ? dt2 : dt1;
    return (dt2 < dt1) ? dt2 : dt1;
}

template <bool kPlain>
BT_DEV bool quadric_tti(SurfPtr s, double x, double y, double z,
                        double vx, double vy, double vz, double& dt, Range& rg)
{                                                    // quadric.cpp:41-70
    double z0term = z-s->p[6];
    double vrr0 = vx*x + vy*y;
    double a = vz*vz + (vx*vx+vy*vy)*s->p[5];
    double b = 2*(vz*z0term + vrr0*s->p[5]);
    double c = z0term*z0term - s->p[7] + (x*x + y*y)*s->p[5];
    double discriminant = b*b - 4*a*c;
    if (discriminant < 0)
        return false;
    const double root = root_of<kPlain>(discriminant, rg);
    double dt1;
    if (b > 0)
        dt1 = (-b - root) / (2*a);
    else
        dt1 = 2*c / (-b + root);
    double dt2 = c / (a*dt1);
    double z1 = z + vz*dt1;
    double z2 = z + vz*dt2;
    dt = (fabs(z1) < fabs(z2)) ? dt1 : dt2;
    return true;
}

template <int K, bool kPlain>
BT_DEV bool leaf_tti(SurfPtr s, double x, double y, double z,
                     double vx, double vy, double vz, double& dt, int niter, Range& rg,
                     NormalMemo* memo = nullptr)
{
    switch (s->kind) {
    case BT_PLANE:                                   // plane.cpp:25-31
        if (vz == 0) return false;
        dt = -z/vz;
        return true;
    case BT_SPHERE: {                                // sphere.cpp:37-64
        const double R = s->p[0];
        double vr2 = vx*vx + vy*vy;
        double vz2 = vz*vz;
        double vrr0 = vx*x + vy*y;
        double r02 = x*x + y*y;
        double z0term = z-R;
        double a = vz2 + vr2;
        double b = 2*vz*z0term + 2*vrr0;
        double c = z0term*z0term - s->p[1] + r02;
        double discriminant = b*b - 4*a*c;
        if (discriminant < 0) return false;
        const double root = root_of<kPlain>(discriminant, rg);
        double dt1;
        if (b > 0)
            dt1 = (-b - root) / (2*a);
        else
            dt1 = 2*c / (-b + root);
        double dt2 = c / (a*dt1);
        dt = pick_root(vz*R, dt1, dt2);
        return true;
    }
    case BT_PARABOLOID: {                            // paraboloid.cpp:39-71
        double a = (vx*vx + vy*vy)*s->p[2];
        double b = (x*vx + y*vy)*s->p[1] - vz;
        double c = (x*x + y*y)*s->p[2] - z;
        if (a == 0) {
            dt = -c/b;
            return true;
        }
        double discriminant = b*b - 4*a*c;
        if (discriminant < 0) return false;
        const double root = root_of<kPlain>(discriminant, rg);
        double dt1;
        if (b > 0)
            dt1 = (-b - root) / (2*a);
        else
            dt1 = 2*c / (-b + root);
        double dt2 = c / (a*dt1);
        dt = pick_root(vz*s->p[0], dt1, dt2);
        return true;
    }
    case BT_QUADRIC:
        return quadric_tti<kPlain>(s, x, y, z, vx, vy, vz, dt, rg);
    case BT_ASPHERE:                                 // asphere.cpp:75-85
        if (!quadric_tti<kPlain>(s, x, y, z, vx, vy, vz, dt, rg)) return false;
        return newton<AsphereEval, kPlain>(s, x, y, z, vx, vy, vz, dt, niter, rg, memo);
    case BT_TILTED: {                                // tilted.cpp:29-37
        double num = z - x*s->p[0] - y*s->p[1];
        double den = vx*s->p[0] + vy*s->p[1] - vz;
        if (den == 0) return false;
        dt = num/den;
        return true;
    }
    case BT_BICUBIC:
    case BT_POLYNOMIAL:                              // surface.cpp:22-49
        if constexpr (K == kKindsAll)
            return newton<LeafEval<K>, kPlain>(s, x, y, z, vx, vy, vz, dt, niter, rg, memo);
        break;
    }
    return false;
}

// sum.cpp:47-56: the first child's intersection (itself a Sum's, to the
// nesting depth kKindsAll allows) seeds Newton on the Sum.
template <int D, bool kPlain>
BT_DEV bool sum_tti_all(SurfPtr s, double x, double y, double z,
                        double vx, double vy, double vz, double& dt, int niter, Range& rg,
                        NormalMemo* memo)
{
    const SurfPtr c = anew(s + 1);
    bool hit = false;
    if (c->kind != BT_SUM) {
        hit = leaf_tti<kKindsAll, kPlain>(c, x, y, z, vx, vy, vz, dt, niter, rg);
    } else {
        if constexpr (D > 0)
            hit = sum_tti_all<D - 1, kPlain>(c, x, y, z, vx, vy, vz, dt, niter, rg, nullptr);
    }
    if (!hit) return false;
    return newton<SurfEval<kKindsAll>, kPlain>(s, x, y, z, vx, vy, vz, dt, niter, rg, memo);
}

template <int K, bool kPlain>
BT_DEV bool surf_tti(SurfPtr s, double x, double y, double z,
                     double vx, double vy, double vz, double& dt, int niter, Range& rg,
                     NormalMemo* memo = nullptr)
{
    constexpr int L = leaf_set(K);
    if (K == kKindsAnalytic || s->kind != BT_SUM)
        return leaf_tti<L, kPlain>(s, x, y, z, vx, vy, vz, dt, niter, rg, memo);
    if constexpr (K == kKindsSumAPB) {
        if (!sum_is_apb(s)) return false;
        if (!leaf_tti<L, kPlain>(anew(s + 1), x, y, z, vx, vy, vz, dt, niter, rg)) return false;
        return newton<SumAPBEval, kPlain>(s, x, y, z, vx, vy, vz, dt, niter, rg, memo);
    } else if constexpr (K == kKindsFlatSums) {
        if (!leaf_tti<L, kPlain>(anew(s + 1), x, y, z, vx, vy, vz, dt, niter, rg)) return false;
        return newton<SurfEval<K>, kPlain>(s, x, y, z, vx, vy, vz, dt, niter, rg, memo);
    } else {
        return sum_tti_all<kMaxSumDepth, kPlain>(s, x, y, z, vx, vy, vz, dt, niter, rg, memo);
    }
}

// The surface's analytic base start: the root of a Sum's first child or of an
// Asphere's conic (the starts of sum.cpp:53 and asphere.cpp:82, without the
// Newton refinement that follows them); surfaces without one start at 0.
template <int K, bool kPlain>
BT_DEV bool conic_start(SurfPtr s, double x, double y, double z, double vx,
                        double vy, double vz, double& dt, Range& rg)
{
    SurfPtr c = s;
    if (K != kKindsAnalytic)
        while (c->kind == BT_SUM) c = c + 1;     // the first leaf of nested Sums
    dt = 0.0;
    switch (c->kind) {
    case BT_ASPHERE:
    case BT_QUADRIC:
        return quadric_tti<kPlain>(c, x, y, z, vx, vy, vz, dt, rg);
    case BT_PLANE:
    case BT_SPHERE:
    case BT_PARABOLOID:
    case BT_TILTED:
        return leaf_tti<leaf_set(K), kPlain>(c, x, y, z, vx, vy, vz, dt, 0, rg);
    default:
        return true;
    }
}


BT_DEV bool newton_surface(SurfPtr s)
{
    return s->kind == BT_SUM || s->kind == BT_ASPHERE || s->kind == BT_BICUBIC ||
           s->kind == BT_POLYNOMIAL;
}

constexpr double kFastTol = 1e-14;   // sag gap accepted by the fast starts [m]

// Newton on the full surface from `dt` until |sag - z| <= kFastTol, with at
// most `max_iter` updates (the reference's niter: a fast start never takes
// more iterations than the reference would, so a ray whose reference
// iteration from the same start has not converged by then is handed back to
// the reference path, which decides it).  At 1e-13 m the residual position
// errors, carried through a three-mirror optic, reach ~1e-14 in the final
// direction cosines; 1e-14 m keeps them an order of magnitude below that.
template <class Ev, bool kPlain>
BT_DEV bool newton_fast(SurfPtr s, double x, double y, double z,
                        double vx, double vy, double vz, double& dt, NormalMemo* memo,
                        int max_iter, Range& rg)
{
    double rPx = x+vx*dt, rPy = y+vy*dt, rPz = z+vz*dt;
    double sz, nx, ny, nz;
    Ev::template point<kPlain, true, true>(s, rPx, rPy, sz, nx, ny, nz, rg);
    for (int it = 0; it < max_iter; it++) {
        if (fabs(sz-rPz) <= kFastTol) break;
        double d = (rPx-x)*nx + (rPy-y)*ny + (sz-z)*nz;
        dt = d / (nx*vx + ny*vy + nz*vz);
        if (Ev::kGrid && !(dt == dt)) return false;
        rPx = x+vx*dt;
        rPy = y+vy*dt;
        rPz = z+vz*dt;
        Ev::template point<kPlain, true, true>(s, rPx, rPy, sz, nx, ny, nz, rg);
    }
    if (!(fabs(sz-rPz) <= kFastTol)) return false;
    *memo = NormalMemo{dt, nx, ny, nz, true};
    return true;
}

// One Newton update of `dt` on an Asphere alone (its sag and normal at the
// ray's point at `dt`); `dt` is kept where the update is not finite.
template <bool kPlain>
BT_DEV void asphere_update(SurfPtr c, double x, double y, double z, double vx,
                           double vy, double vz, double& dt, Range& rg)
{
    const double rPx = x+vx*dt, rPy = y+vy*dt;
    double sz, nx, ny, nz;
    AsphereEval::point<kPlain, true, true>(c, rPx, rPy, sz, nx, ny, nz, rg);
    const double d = (rPx-x)*nx + (rPy-y)*ny + (sz-z)*nz;
    const double t = d / (nx*vx + ny*vy + nz*vz);
    if (t == t) dt = t;
}

// Intersection with a fast start, then Newton on the full surface to the
// fast tolerance.  Starts:
// * BT_START_CONIC on a Sum whose first child is an Asphere: that Asphere's
//   conic root moved by one Newton update on the Asphere (the Sum's other
//   terms then hold the whole remaining gap, so the Sum's own, costlier,
//   iteration takes one update where the conic root needs up to two);
// * BT_START_CONIC on another Sum: the reference's own start, its first
//   child's root (sum.cpp:53), so the fast iteration runs the reference's
//   iterates;
// * otherwise the base conic's root (the ray origin where the surface has
//   no conic base) plus `correction` (the network's prediction for
//   BT_START_MLP, 0 for BT_START_CONIC).
// The reference path decides every ray the fast start does not settle.
template <int K, bool kPlain>
BT_DEV bool fast_tti(SurfPtr s, double x, double y, double z, double vx,
                     double vy, double vz, double& dt, int niter, double correction,
                     Range& rg, NormalMemo* memo)
{
    if (newton_surface(s)) {
        double d0 = 0.0;
        bool start;
        if (K != kKindsAnalytic && correction == 0.0 && s->kind == BT_SUM) {
            SurfPtr c = s + 1;
            if (c->kind == BT_ASPHERE) {
                start = quadric_tti<kPlain>(c, x, y, z, vx, vy, vz, d0, rg);
                if (start) asphere_update<kPlain>(c, x, y, z, vx, vy, vz, d0, rg);
            } else if constexpr (K != kKindsSumAPB) {
                start = surf_tti<K, kPlain>(anew(c), x, y, z, vx, vy, vz, d0, niter, rg);
            } else {
                start = false;                  // not a Sum(Asphere, Polynomial, Bicubic)
            }
        } else {
            start = conic_start<K, kPlain>(s, x, y, z, vx, vy, vz, d0, rg);
            d0 += correction;
        }
        bool conv = false;
        if (start && d0 == d0) {
            if (s->kind == BT_ASPHERE)
                conv = newton_fast<AsphereEval, kPlain>(s, x, y, z, vx, vy, vz, d0, memo, niter, rg);
            else if constexpr (K == kKindsSumAPB)
                conv = sum_is_apb(s) &&
                       newton_fast<SumAPBEval, kPlain>(s, x, y, z, vx, vy, vz, d0, memo, niter,
                                                       rg);
            else
                conv = newton_fast<SurfEval<K>, kPlain>(s, x, y, z, vx, vy, vz, d0, memo, niter, rg);
        }
        if (conv) {
            dt = d0;
            return true;
        }
    }
    dt = 0.0;
    return surf_tti<K, kPlain>(anew(s), x, y, z, vx, vy, vz, dt, niter, rg, memo);
}

// ---------------------------------------------------------------------------
// Media (src/medium.cpp)
// ---------------------------------------------------------------------------
BT_DEV double medium_n(MediumPtr m, double w)
{
    switch (m->kind) {
    case BT_MED_CONST:                               // medium.cpp:30-32
        return m->p[0];
    case BT_MED_TABLE: {                             // medium.cpp:89-105
        const TablePtr args = (TablePtr)m->a0;
        const TablePtr vals = (TablePtr)m->a1;
        const int size = m->n;
        if (w < args[0]) return __builtin_nan("");
        if (w > args[size-1]) return __builtin_nan("");
        int u;
        for (u = 1; u < size; u++)
            if (w < args[u]) break;
        double out = (w - args[u-1]);
        out *= (vals[u] - vals[u-1]);
        out /= (args[u] - args[u-1]);
        out += vals[u-1];
        return out;
    }
    case BT_MED_SELLMEIER: {                         // medium.cpp:145-149
        const CoefPtr p = m->p;
        double x = w*w*1e12;
        return cr_sqrt(1.0 + p[0]*x/(x-p[3]) + p[1]*x/(x-p[4]) + p[2]*x/(x-p[5]));
    }
    case BT_MED_SUMITA: {                            // medium.cpp:186-191
        const CoefPtr A = m->p;
        double x = w*w*1e12;
        double y = 1./x;
        return cr_sqrt(A[0] + A[1]*x + y*(A[2] + y*(A[3] + y*(A[4] + y*A[5]))));
    }
    case BT_MED_AIR: {                               // medium.cpp:237-245
        const double P = m->p[0], T = m->p[1], W = m->p[2];
        double s2 = 1e-12 / (w*w);
        double n_minus_one = (64.328 + (29498.1 / (146.0 - s2))
                              + (255.4 / (41.0 - s2))) * 1.e-6;
        n_minus_one *= P * (1.0 + (1.049 - 0.0157 * T) * 1.e-6 * P)
                       / (720.883 * (1.0 + 0.003661 * T));
        n_minus_one -= (0.0624 - 0.000680 * s2)/(1.0 + 0.003661 * T) * W * 1.e-6;
        return 1+n_minus_one;
    }
    }
    return __builtin_nan("");
}

// ---------------------------------------------------------------------------
// hypot as the reference gets it from x86-64 libm (glibc >= 2.35): the
// corrected square root of C. F. Borges, "An improved algorithm for
// hypot(a, b)" (2019), in its form without fused multiply-add, with
// power-of-two rescaling far from 1.  Bit-identical to libm's hypot,
// including the ~0.4 % of arguments where that is not the correctly
// rounded value -- which decides flags of rays that land exactly on a
// circular obscuration edge (a hexapolar ring at the pupil radius).
// Needs -ffp-contract=off (no fusing of the products below).
// ---------------------------------------------------------------------------
BT_DEV double hypot_kernel(double ax, double ay)    // ax >= ay >= 0
{
    double h = cr_sqrt(ax*ax + ay*ay);
    double t1, t2;
    if (h <= 2.0*ay) {
        double delta = h - ay;
        t1 = ax*(2.0*delta - ax);
        t2 = (delta - 2.0*(ax - ay))*delta;
    } else {
        double delta = h - ax;
        t1 = 2.0*delta*(ax - 2.0*ay);
        t2 = (4.0*delta - ay)*ay + delta*delta;
    }
    h -= (t1 + t2)/(2.0*h);
    return h;
}

BT_DEV double ref_hypot(double x, double y)
{
    if (!__builtin_isfinite(x) || !__builtin_isfinite(y)) {
        if (__builtin_isinf(x) || __builtin_isinf(y)) return __builtin_inf();
        return x + y;
    }
    x = fabs(x);
    y = fabs(y);
    const double ax = x < y ? y : x;
    const double ay = x < y ? x : y;
    constexpr double kScale = 0x1p-600, kEps = 0x1p-54;
    if (ax > 0x1p+511) {
        if (ay <= ax*kEps) return ax + ay;
        return hypot_kernel(ax*kScale, ay*kScale)/kScale;
    }
    if (ay < 0x1p-511) {
        if (ax >= ay/kEps) return ax + ay;
        return hypot_kernel(ax/kScale, ay/kScale)*kScale;
    }
    if (ay <= ax*kEps) return ax + ay;
    return hypot_kernel(ax, ay);
}

// The comparison hypot(x, y) < r decided from s = x*x + y*y without the
// square root: -1 when hypot(x, y) < r for certain, +1 when > r, 0 when s
// lies within 2^-43 (~1.1e-13) of r*r (or outside the range where that
// bound holds: NaN, inf, r outside {0} and (2^-465, 2^465), s >= 2^930),
// where only libm's value decides.  s carries at most ~2^-51 relative error
// and libm's hypot is within 1 ulp of the true value, far inside the 2^-43
// margin, so a decided comparison agrees with libm's.  The bounds are powers
// of two so that each compare takes its constant as an instruction literal
// instead of holding it in registers across the interface loop.
BT_DEV int cmp_hypot(double x, double y, double r)
{
    const double s = x*x + y*y;
    if (r == 0.0) return (s > 0.0 && s < 0x1p930) ? 1 : 0;   // an annulus from 0
    if (!(r > 0x1p-465 && r < 0x1p465)) return 0;
    if (!(s < 0x1p930)) return 0;
    const double r2 = r*r;
    const double d = s - r2;
    const double m = r2*0x1p-43;
    if (d > m) return 1;
    if (d < -m) return -1;
    return 0;
}

// ---------------------------------------------------------------------------
// Obscuration programs (src/obscuration.cpp); the stack is a bit mask.
// ---------------------------------------------------------------------------
BT_DEV bool polygon_contains(ObscPtr o, double x, double y)
{                                                    // obscuration.cpp:201-225
    const CoefPtr xp = (CoefPtr)o->a0;
    const CoefPtr yp = (CoefPtr)o->a1;
    const int size = o->n;
    double x1 = xp[0];
    double y1 = yp[0];
    double xinters = 0.0;
    bool inside = false;
    for (int i = 1; i <= size; i++) {
        const int k = (i == size) ? 0 : i;
        double x2 = xp[k];
        double y2 = yp[k];
        double ymin = (y2 < y1) ? y2 : y1;
        double ymax = (y1 < y2) ? y2 : y1;
        double xmax = (x1 < x2) ? x2 : x1;
        if (y > ymin && y <= ymax && x <= xmax) {
            if (y1 != y2)
                xinters = (y-y1)*(x2-x1)/(y2-y1)+x1;
            if (x1 == x2 || x <= xinters)
                inside = !inside;
        }
        x1 = x2;
        y1 = y2;
    }
    return inside;
}

BT_DEV bool obsc_contains(ObscPtr prog, int len, double x, double y)
{
    uint32_t stack = 0;   // bit k = stack slot k
    int sp = 0;
    for (int k = 0; k < len; k++) {
        ObscPtr o = prog + k;
        const CoefPtr p = o->p;
        bool v;
        switch (o->op) {
        case BT_OB_CIRCLE: {                         // obscuration.cpp:32-34
            const double dx = x-p[1], dy = y-p[2];
            const int c = cmp_hypot(dx, dy, p[0]);
            v = c ? (c < 0) : (ref_hypot(dx, dy) < p[0]);
            break;
        }
        case BT_OB_ANNULUS: {                        // obscuration.cpp:80-83
            const double dx = x-p[2], dy = y-p[3];
            const int ci = cmp_hypot(dx, dy, p[0]), co = cmp_hypot(dx, dy, p[1]);
            if (ci && co) {
                v = (ci > 0) && (co < 0);
            } else {
                const double h = ref_hypot(dx, dy);
                v = (p[0] <= h) && (h < p[1]);
            }
            break;
        }
        case BT_OB_RECTANGLE: {                      // obscuration.cpp:117-121
            double xp = (x-p[2])*p[4] + (y-p[3])*p[5];
            double yp = -(x-p[2])*p[5] + (y-p[3])*p[4];
            v = (xp > -p[0]/2 && xp < p[0]/2 && yp > -p[1]/2 && yp < p[1]/2);
            break;
        }
        case BT_OB_RAY: {                            // obscuration.cpp:155-159
            double xp = (x-p[1])*p[3] + (y-p[2])*p[4];
            double yp = -(x-p[1])*p[4] + (y-p[2])*p[3];
            v = (xp > 0.0 && yp > -p[0]/2 && yp < p[0]/2);
            break;
        }
        case BT_OB_POLYGON:
            v = polygon_contains(o, x, y);
            break;
        case BT_OB_NEGATION:                         // obscuration.cpp:320-322
            stack ^= (1u << (sp-1));
            continue;
        case BT_OB_UNION:                            // obscuration.cpp:364-370
        case BT_OB_INTERSECTION: {                   // obscuration.cpp:415-421
            const int m = o->n;
            const uint32_t mask = ((m >= 32) ? 0xffffffffu : ((1u << m) - 1u)) << (sp - m);
            const uint32_t bits = stack & mask;
            v = (o->op == BT_OB_UNION) ? (bits != 0) : (bits == mask);
            stack &= ~mask;
            sp -= m;
            break;
        }
        default:
            v = false;
        }
        stack = (stack & ~(1u << sp)) | ((uint32_t)v << sp);
        sp++;
    }
    return sp > 0 && ((stack >> (sp-1)) & 1u);
}

// ---------------------------------------------------------------------------
// One Interface: transform, intersect, interact, obscure
// (src/batoid.cpp:221-505 and optic.py:419-422)
// ---------------------------------------------------------------------------
struct Ray {
    double x, y, z, vx, vy, vz, t, w;
    bool vig, fail;
};

// What a refraction and the reflected part of a split share at a surface of
// normal n (batoid.cpp:453-470, 620-640): the incoming index n1 = 1/|v|, the
// unit velocity nv, and the normal turned against it with alpha = nv.n <= 0.
struct Incidence {
    double n1, root, nvx, nvy, nvz, nx, ny, nz, alpha;
};

template <bool kPlain>
BT_DEV Incidence incidence(double nx, double ny, double nz, double vx, double vy, double vz,
                           Range& rg)
{
    Incidence c;
    double n1 = vx*vx;
    n1 += vy*vy;
    n1 += vz*vz;
    c.n1 = recip_root_of<kPlain>(n1, c.root, rg);
    c.nvx = vx*c.n1;
    c.nvy = vy*c.n1;
    c.nvz = vz*c.n1;
    double alpha = c.nvx*nx;
    alpha += c.nvy*ny;
    alpha += c.nvz*nz;
    if (alpha > 0.) {
        nx *= -1; ny *= -1; nz *= -1;
        alpha *= -1;
    }
    c.nx = nx; c.ny = ny; c.nz = nz;
    c.alpha = alpha;
    return c;
}

// The velocity refracted into a medium of index n2 (batoid.cpp:474-496);
// true for total internal reflection (NaN velocity).  Into a medium of index
// exactly 1 (vacuum, or air given as a constant 1) the reference's divisions
// by n2 return their numerators bit for bit (x/1 == x in IEEE arithmetic,
// signed zeros, infinities and NaNs included), so that case runs without
// them; into any other the plain form's four quotients share one reciprocal.
template <bool kPlain>
BT_DEV bool refract_velocity(const Incidence& c, double n2, double& vx, double& vy, double& vz,
                             Range& rg)
{
    const bool unit = __all(n2 == 1.0);
    double eta = c.n1, inv = 0.0;
    if (!unit) {
        if constexpr (kPlain) {
            rg.positive(n2);
            inv = recip_plain(n2);
            eta = div_plain(c.n1, n2, inv);
        } else {
            eta /= n2;
        }
    }
    const double sinsqr = eta*eta*(1-c.alpha*c.alpha);
    if (sinsqr > 1.0) {
        vx = __builtin_nan(""); vy = vx; vz = vx;
        return true;
    }
    const double nfactor = eta*c.alpha + root_of<kPlain>(1-sinsqr, rg);
    vx = eta*c.nvx - nfactor*c.nx;
    vy = eta*c.nvy - nfactor*c.ny;
    vz = eta*c.nvz - nfactor*c.nz;
    if (!unit) {
        if constexpr (kPlain) {
            vx = div_plain_signed(vx, n2, inv);
            vy = div_plain_signed(vy, n2, inv);
            vz = div_plain_signed(vz, n2, inv);
        } else {
            vx /= n2;
            vy /= n2;
            vz /= n2;
        }
    }
    return false;
}

// The velocity v - 2 alpha n / n1 of the reflected part of a split
// (batoid.cpp:642-645), in place.
template <bool kPlain>
BT_DEV void split_reflect(const Incidence& c, double& vx, double& vy, double& vz, Range& rg)
{
    const double ax = 2*c.alpha*c.nx, ay = 2*c.alpha*c.ny, az = 2*c.alpha*c.nz;
    if constexpr (kPlain) {
        const double inv = recip_refine(c.n1, c.root);   // as in add_slope
        vx = vx - div_plain_signed(ax, c.n1, inv);
        vy = vy - div_plain_signed(ay, c.n1, inv);
        vz = vz - div_plain_signed(az, c.n1, inv);
    } else {
        vx = vx - ax/c.n1;
        vy = vy - ay/c.n1;
        vz = vz - az/c.n1;
    }
}

// A ray in an Interface's frame, advanced to its surface.
struct Arrival {
    double x, y, z, vx, vy, vz, t, dt;
    NormalMemo memo;
};

// A rotation by nothing: the unit matrix, zeros of either sign (tested on the
// scalar unit).  Its products are exact, so 12 FMAs give the bits of the 18
// products and 12 sums, signed zeros and NaNs included.  Only in the kernels
// of analytic surfaces, which issue bounds: 1780 -> 1745 us for 1e7 rays
// through twelve Interfaces; the freeform kernel was 2 % slower with it.
template <class Frame>
BT_DEV bool unrotated(Frame m)
{
    auto bits = [](double v) { return __builtin_bit_cast(uint64_t, v); };
    const uint64_t off = bits(m[1]) | bits(m[2]) | bits(m[3]) | bits(m[5]) | bits(m[6]) | bits(m[7]);
    const uint64_t dia = (bits(m[0]) ^ bits(1.0)) | (bits(m[4]) ^ bits(1.0)) | (bits(m[8]) ^ bits(1.0));
    return ((off << 1) | dia) == 0;
}

// Frame change and intersection; false where the ray misses the surface.
template <int K, bool kPlain, class Frame>
BT_DEV bool arrive(Frame dr, Frame drot,
                   SurfPtr surf, const Ray& r, int niter, int start,
                   double correction, Arrival& a, Range& rg)
{
    double dx = r.x-dr[0];
    double dy = r.y-dr[1];
    double dz = r.z-dr[2];
    if (K == kKindsAnalytic && unrotated(drot)) {
        a.x = __builtin_fma(dz, drot[6], __builtin_fma(dy, drot[3], dx));
        a.y = __builtin_fma(dz, drot[7], __builtin_fma(dx, drot[1], dy));
        a.z = __builtin_fma(dy, drot[5], __builtin_fma(dx, drot[2], dz));
        a.vx = __builtin_fma(r.vz, drot[6], __builtin_fma(r.vy, drot[3], r.vx));
        a.vy = __builtin_fma(r.vz, drot[7], __builtin_fma(r.vx, drot[1], r.vy));
        a.vz = __builtin_fma(r.vy, drot[5], __builtin_fma(r.vx, drot[2], r.vz));
    } else {
        a.x = dx*drot[0] + dy*drot[3] + dz*drot[6];
        a.y = dx*drot[1] + dy*drot[4] + dz*drot[7];
        a.z = dx*drot[2] + dy*drot[5] + dz*drot[8];
        a.vx = r.vx*drot[0] + r.vy*drot[3] + r.vz*drot[6];
        a.vy = r.vx*drot[1] + r.vy*drot[4] + r.vz*drot[7];
        a.vz = r.vx*drot[2] + r.vy*drot[5] + r.vz*drot[8];
    }
    a.t = r.t;
    a.dt = 0.0;
    a.memo.ok = false;
    const bool hit =
        (start == BT_START_REFERENCE)
            ? surf_tti<K, kPlain>(surf, a.x, a.y, a.z, a.vx, a.vy, a.vz, a.dt, niter, rg,
                                  &a.memo)
            : fast_tti<K, kPlain>(surf, a.x, a.y, a.z, a.vx, a.vy, a.vz, a.dt, niter,
                                  correction, rg, &a.memo);
    if (!hit) return false;
    a.x += a.vx * a.dt;
    a.y += a.vy * a.dt;
    a.z += a.vz * a.dt;
    a.t += a.dt;
    if constexpr (kPlain) rg.not_tiny(a.x, a.y);
    return true;
}

// The normal at the intersection, reusing Newton's when it was evaluated at
// this very point.
template <int K, bool kPlain>
BT_DEV void arrival_normal(SurfPtr surf, const Arrival& a, double& nx, double& ny,
                           double& nz, Range& rg)
{
    if (a.memo.ok && same_bits(a.memo.dt, a.dt)) {
        nx = a.memo.nx; ny = a.memo.ny; nz = a.memo.nz;
    } else {
        double sag;
        if constexpr (!kPlain) surf = anew(surf);    // after Newton only in the full form
        surf_point<K, kPlain, false, true>(surf, a.x, a.y, sag, nx, ny, nz, rg);
    }
    if constexpr (kPlain) {                          // quadric.cpp:29, asphere.cpp:50
        const bool vertex = (a.x == 0.0) & (a.y == 0.0);
        if (__builtin_expect(__any(vertex), 0)) {
            const int kind = surf->kind;
            if (kind == BT_SPHERE || kind == BT_QUADRIC || kind == BT_ASPHERE) {
                nx = vertex ? 0.0 : nx;
                ny = vertex ? 0.0 : ny;
            }
        }
    }
}

// One interaction in the plain or the full form, on a ray that has not
// failed; returns true when the ray's kinematic state was (re)written.
template <int K, bool kPlain, class Frame>
BT_DEV bool interact(int action, Frame dr, Frame drot, SurfPtr surf, double n2,
                     Ray& r, int niter, int start, double correction, Range& rg)
{
    Arrival a;
    if (!arrive<K, kPlain>(dr, drot, surf, r, niter, start, correction, a, rg)) {
        r.fail = true;
        r.vig = true;
        return false;          // left in the previous frame
    }
    double nx, ny, nz;
    if (action == BT_ACT_REFLECT) {                  // batoid.cpp:340-353
        arrival_normal<K, kPlain>(surf, a, nx, ny, nz, rg);
        double alpha = a.vx*nx;
        alpha += a.vy*ny;
        alpha += a.vz*nz;
        a.vx -= 2*alpha*nx;
        a.vy -= 2*alpha*ny;
        a.vz -= 2*alpha*nz;
    } else if (action == BT_ACT_REFRACT) {           // batoid.cpp:453-496
        arrival_normal<K, kPlain>(surf, a, nx, ny, nz, rg);
        const Incidence c = incidence<kPlain>(nx, ny, nz, a.vx, a.vy, a.vz, rg);
        if (refract_velocity<kPlain>(c, n2, a.vx, a.vy, a.vz, rg)) {
            r.fail = true;                           // total internal reflection
            r.vig = true;
        }
    }
    r.x = a.x; r.y = a.y; r.z = a.z;
    r.vx = a.vx; r.vy = a.vy; r.vz = a.vz;
    r.t = a.t;
    return true;
}

// A ray that has not failed split at a surface (batoid.cpp:582-672): `r`
// becomes the refracted part, `q` the reflected one; false where the ray
// misses, with both parts failed and left in the previous frame.
template <int K, bool kPlain, class Frame>
BT_DEV bool split_parts(Frame dr, Frame drot,
                        SurfPtr surf, double n2, Ray& r, Ray& q, int niter, Range& rg)
{
    Arrival a;
    if (!arrive<K, kPlain>(dr, drot, surf, r, niter, BT_START_REFERENCE, 0.0, a, rg)) {
        r.fail = true;
        r.vig = true;
        q = r;
        return false;
    }
    double nx, ny, nz;
    arrival_normal<K, kPlain>(surf, a, nx, ny, nz, rg);
    const Incidence c = incidence<kPlain>(nx, ny, nz, a.vx, a.vy, a.vz, rg);
    r.x = a.x; r.y = a.y; r.z = a.z;
    r.t = a.t;
    q = r;
    q.vx = a.vx; q.vy = a.vy; q.vz = a.vz;
    split_reflect<kPlain>(c, q.vx, q.vy, q.vz, rg);
    if (refract_velocity<kPlain>(c, n2, r.vx, r.vy, r.vz, rg)) {
        r.fail = true;
        r.vig = true;
    }
    return true;
}

// split_parts with the wave's vote.
template <int K, class Frame>
BT_DEV bool split_ray(Frame dr, Frame drot,
                      SurfPtr surf, double n2, Ray& r, Ray& q, int niter)
{
    Range rg;
    if constexpr (!kVoted<K>)
        return split_parts<K, false>(dr, drot, surf, n2, r, q, niter, rg);
    Ray p = r;
    bool hit = split_parts<K, true>(dr, drot, surf, n2, p, q, niter, rg);
    rg.not_tiny(p.vx, p.vy);
    rg.not_tiny(p.vz, q.vz);
    rg.not_tiny(q.vx, q.vy);
    if (__all(rg.plain()))
        r = p;
    else
        hit = split_parts<K, false>(dr, drot, surf, n2, r, q, niter, rg);
    return hit;
}

// Returns true when the ray's kinematic state was (re)written.  `n2` is the
// outgoing medium's index at the ray's wavelength (used by REFRACT only); the
// reference evaluates it after the intersection (batoid.cpp:474), but it is
// a pure function of the wavelength, so callers may evaluate it once per ray
// and medium and reuse it across Interfaces.
template <int K, class Frame>
BT_DEV bool apply_interaction(int action, Frame dr, Frame drot,
                              SurfPtr surf, double n2,
                              Ray& r, int niter, int start = BT_START_REFERENCE,
                              double correction = 0.0)
{
    if (r.fail) return false;
    Range rg;
    if constexpr (!kVoted<K>)
        return interact<K, false>(action, dr, drot, surf, n2, r, niter, start, correction, rg);
    Ray p = r;
    bool moved = interact<K, true>(action, dr, drot, surf, n2, p, niter, start, correction, rg);
    rg.not_tiny(p.vx, p.vy);
    rg.not_tiny(p.vz, p.vz);
    if (__all(rg.plain()))
        r = p;
    else
        moved = interact<K, false>(action, dr, drot, surf, n2, r, niter, start, correction, rg);
    return moved;
}

}  // namespace bt
