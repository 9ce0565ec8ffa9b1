// bt_plan.h -- the fused plan kernel (bt_trace_plan): every Interface of an
// optic applied while a ray stays in registers.  One source file per kind set
// instantiates it (bt_plan_*.hip), so that the sets compile side by side.
#pragma once

#include "bt_device.h"
#include "bt_common.h"

namespace bt {

// The network's input at an MLP step: the ray's point on the surface's base
// conic and its direction, in the step's local frame (the frame change is
// apply_interaction's).
template <int K>
__device__ __forceinline__ void mlp_features(StepPtr st, SurfPtr surf, const Ray& r,
                                             const MlpPacked* P, float (&f)[kMlpIn])
{
    const CoefPtr dr = st->dr;
    const CoefPtr m = st->drot;
    double dx = r.x-dr[0], dy = r.y-dr[1], dz = r.z-dr[2];
    double x = dx*m[0] + dy*m[3] + dz*m[6];
    double y = dx*m[1] + dy*m[4] + dz*m[7];
    double z = dx*m[2] + dy*m[5] + dz*m[8];
    double vx = r.vx*m[0] + r.vy*m[3] + r.vz*m[6];
    double vy = r.vx*m[1] + r.vy*m[4] + r.vz*m[7];
    double vz = r.vx*m[2] + r.vy*m[5] + r.vz*m[8];
    double dtc = 0.0;
    Range rg;
    if (r.fail || !conic_start<K, false>(surf, x, y, z, vx, vy, vz, dtc, rg)) {
        // keep this lane's share of the wave's evaluation finite
        for (int k = 0; k < kMlpIn; k++) f[k] = P->norm[k];
        return;
    }
    f[0] = (float)(x + vx*dtc);
    f[1] = (float)(y + vy*dtc);
    f[2] = (float)(z + vz*dtc);
    f[3] = (float)vx;
    f[4] = (float)vy;
    f[5] = (float)vz;
}

// Waves per SIMD: the analytic-kinds kernels of modes 0 and 1 are held to
// six (77 and 79 VGPRs), the Sum(Asphere, Polynomial, Bicubic) kernels to
// four (128 VGPRs; mode 0 spills 16 words outside its Newton loops), the
// others of mode 0 to four and of modes 1 and 2 to three (left alone the
// compiler would settle for two).  Mode 0 at three, four and five waves: 621,
// 573, 655 us (1e6 rays, three perturbed mirrors), 320, 304, 372 (3e5,
// freeform); the conic start on the first, 3e6 rays: 1002, 918, 1305.
template <int Mode, int K>
constexpr int plan_waves_per_simd()
{
    if (K == kKindsAnalytic && Mode < 2) return 6;
    if (K == kKindsSumAPB) return Mode == 2 ? 3 : 4;
    return Mode == 0 ? 4 : 3;     // kKindsAll, kKindsFlatSums
}

// Networks a plan kernel keeps in LDS (45 KB per workgroup).
constexpr int kMlpLds = 4;

// Ray i of `in` through every step of the plan while it stays in registers, in
// the plain form (what may have left its range noted in `rg`) or the full one.
// A ray's wavelength never changes, so the index of the plan's (first)
// dispersive medium is evaluated once per ray up front.
//
// Mode 0: reference starts only.  Mode 1: CONIC starts honoured (an MLP step
// runs as CONIC).  Mode 2: MLP starts too; MLP inference is a wave-wide MFMA
// product, so in this variant every lane of a wave stays in the step loop
// (lanes past the end work on a copy of the last ray and store nothing).
template <int Mode, int K, bool kPlain>
__device__ __forceinline__ void trace_steps(bt_plan plan, bt_rays in, int64_t i,
                                            int niter, int need_w, const MlpPacked* nets,
                                            Ray& r, Range& rg)
{
    constexpr bool Fast = Mode > 0;
    constexpr bool Mlp = Mode > 1;
    const StepPtr steps = (StepPtr)plan.steps;
    const SurfPtr surfaces = (SurfPtr)plan.surfaces;
    const MediumPtr media = (MediumPtr)plan.media;
    const ObscPtr obscs = (ObscPtr)plan.obscs;
    r.fail = in.failed[i] != 0;
    r.vig = in.vignetted[i] != 0;
    r.x = in.x[i]; r.y = in.y[i]; r.z = in.z[i];
    r.vx = in.vx[i]; r.vy = in.vy[i]; r.vz = in.vz[i];
    r.t = in.t[i];
    // Refractive indices: a constant medium's is its record's (a scalar
    // load); the plan's first dispersive medium is evaluated once per ray and
    // kept; any other dispersive medium is evaluated at its refraction, with
    // the wavelength read again from memory (it is not held in registers).
    const int nmed = plan.nmedia;
    int cm = -1;                               // the cached medium (wave-uniform)
    for (int m = 0; m < nmed; m++)
        if (media[m].kind != BT_MED_CONST) { cm = m; break; }
    double ncm = 0.0;
    if (need_w && cm >= 0 && !r.fail) ncm = medium_n(media + cm, in.wavelength[i]);
    const int nstep = plan.nstep;
    int mslot = 0;                             // next LDS network (wave-uniform)
    for (int k = 0; k < nstep; k++) {
        if (!Mlp && r.fail && r.vig) break;    // nothing below can change this ray
        const StepPtr st = steps + k;
        const SurfPtr surf = surfaces + st->surface;
        const int action = st->action;
        double n2 = 0.0;
        if (action == BT_ACT_REFRACT && !r.fail) {
            const int mi = st->medium;
            const MediumPtr med = media + mi;
            n2 = (med->kind == BT_MED_CONST) ? med->p[0]           // medium.cpp:30-32
                 : (mi == cm) ? ncm : medium_n(med, in.wavelength[i]);
        }
        double correction = 0.0;
        int start = Fast ? st->start : BT_START_REFERENCE;
        if (start == BT_START_MLP && (!Mlp || !st->mlp || mslot >= kMlpLds))
            start = BT_START_CONIC;
        if (Mlp && start == BT_START_MLP) {     // uniform: whole wave
            const MlpPacked* P = nets + mslot;
            mslot++;
            float f[kMlpIn];
            mlp_features<K>(st, surf, r, P, f);
            correction = (double)mlp_predict_wave(P, f);
        }
        if (!r.fail)
            interact<K, kPlain>(action, st->dr, st->drot, surf, n2, r, niter, start,
                                correction, rg);
        const int olen = st->obsc_len;
        if (olen > 0 && !r.vig)
            r.vig = obsc_contains(obscs + st->obsc, olen, r.x, r.y);
        if constexpr (kPlain && K == kKindsAnalytic)
            if (__any(rg.left())) break;        // the full form decides
    }
}

// Kernels whose waves run the plan in the plain form, vote once at its end,
// and read their rays again for the full form if a lane left the plain range
// (an overflow, a ray beyond an asphere's domain): the full form shares no
// live register with the plain loop.  (A vote at each step kept the ray twice
// and cost a wave of occupancy: 1.96 against 1.78 ms for 1e7 rays of the
// analytic kernel.)  A wave of the analytic kernel stops at the step where a root
// left the range: a 512 x 512 beam 1.6 times as wide as the pupil of a
// 20-interface corrector, 29 % of which fails, takes 152 to 172 us, 203 to 208
// with the whole plan in both forms, 138 in the full form alone; others pay
// 0.4 % (2 % for the Sums, whose failing rays mostly leave the Bicubic's grid,
// which is no cause for the full form).  Kernel times before and after, at the same clocks:
// 2.01 -> 1.78 ms (analytic, 1e7 rays x 12; 1.84 with quotients right for every
// denominator and vertices in the plain form), 0.86 -> 0.70 ms (three perturbed
// mirrors, 1e6), 1.18 -> 1.08 (the same, conic start, 3e6), 0.49 -> 0.46
// (freeform, 3e5), 41 -> 35 us (162 rays).  Bound by FP64 issue.  The
// nested-Sum and learned-start kernels hold the full form alone: theirs is as
// large as two of the others.
template <int Mode, int K>
constexpr bool plan_voted() { return K != kKindsAll && Mode < 2; }

template <int Mode, int K>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(plan_waves_per_simd<Mode, K>())))
void k_plan(
    bt_plan plan, bt_rays in, bt_rays out, int niter, int need_w)
{
    constexpr bool Mlp = Mode > 1;
    // Mode 2: the networks of the plan's first kMlpLds MLP steps, copied to
    // LDS once per workgroup (a wave-wide inference then reads its weight
    // fragments from LDS, not from L2); later MLP steps run as CONIC.
    const MlpPacked* nets = nullptr;
    if constexpr (Mlp) {
        __shared__ MlpPacked lds_nets[kMlpLds];
        int slot = 0;
        for (int k = 0; k < plan.nstep && slot < kMlpLds; k++) {
            const bt_step* st = plan.steps + k;
            if (st->start != BT_START_MLP || !st->mlp) continue;
            const uint4* src = static_cast<const uint4*>(st->mlp);
            uint4* dst = reinterpret_cast<uint4*>(lds_nets + slot);
            for (int q = threadIdx.x; q < (int)(sizeof(MlpPacked) / 16); q += kBlock)
                dst[q] = src[q];
            slot++;
        }
        __syncthreads();
        nets = lds_nets;
    }
    const int64_t i0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (!Mlp && i0 >= in.n) return;
    const bool live = i0 < in.n;
    int64_t i = live ? i0 : in.n - 1;
    Ray r;
    Range rg;
    if constexpr (plan_voted<Mode, K>()) {
        trace_steps<Mode, K, true>(plan, in, i, niter, need_w, nets, r, rg);
        rg.not_tiny(r.vx, r.vy);
        rg.not_tiny(r.vz, r.vz);
        if (__builtin_expect(!__all(rg.plain()), 0)) {
            asm("" : "+v"(i));                  // nothing is kept from the plain pass
            trace_steps<Mode, K, false>(plan, in, i, niter, need_w, nets, r, rg);
        }
    } else {
        trace_steps<Mode, K, false>(plan, in, i, niter, need_w, nets, r, rg);
    }
    if (Mlp && !live) return;
    out.x[i] = r.x; out.y[i] = r.y; out.z[i] = r.z;
    out.vx[i] = r.vx; out.vy[i] = r.vy; out.vz[i] = r.vz;
    out.t[i] = r.t;
    out.vignetted[i] = r.vig;
    out.failed[i] = r.fail;
    if (out.wavelength != in.wavelength) out.wavelength[i] = in.wavelength[i];
    if (out.flux != in.flux) out.flux[i] = in.flux[i];
}

template <int K>
inline void launch_plan_kinds(int mode, dim3 grid, hipStream_t st, const bt_plan& plan,
                              const bt_rays& in, const bt_rays& out, int niter, int need_w)
{
    if (mode == 0)
        hipLaunchKernelGGL((k_plan<0, K>), grid, dim3(kBlock), 0, st, plan, in, out, niter, need_w);
    else if (mode == 1)
        hipLaunchKernelGGL((k_plan<1, K>), grid, dim3(kBlock), 0, st, plan, in, out, niter, need_w);
    else
        hipLaunchKernelGGL((k_plan<2, K>), grid, dim3(kBlock), 0, st, plan, in, out, niter, need_w);
}

}  // namespace bt
