// bt_split.hip -- ghost splitting: rSplit and the ray selection of traceSplit.
//
// bt_rsplit splits every ray that reaches a surface into its refracted and
// reflected parts in one pass (src/batoid.cpp:509-674): lane i intersects
// ray i with the reference's Newton iteration, then writes the reflected
// ray to the split buffer and the refracted ray back in place, with the
// coating's flux fractions.  The arithmetic is the reference's, operation by
// operation.
//
// traceSplit (batoid/optic.py:1244-1282) keeps, after every Interface, only
// the rays that are unvignetted and above a flux threshold.  Here that
// filter is an order-preserving stream compaction: per-block counts from
// wave ballots, one exclusive scan over the blocks, then a scatter that
// recomputes each ray's rank from the same ballots.
#include <hip/hip_runtime.h>
#include <string>

#include "bt_device.h"
#include "bt_common.h"

namespace bt {

// One ray of rSplit; returns false for a ray traceSplit's filter had
// already dropped (live mode), which is left untouched.  `lr` / `ls`: the
// refracted and split parts pass traceSplit's filter afterwards.
template <int K>
__device__ __forceinline__ void rsplit_ray(
    int64_t i, const Xform& xf, const bt_surface* __restrict__ surf,
    const bt_medium* __restrict__ m2, double reflect, double transmit,
    const bt_obsc* __restrict__ obsc, int olen, const bt_rays& rv, const bt_rays& sp,
    int niter, int live, double min_flux, bool& lr, bool& ls)
{                                                    // batoid.cpp:582-672
    lr = ls = false;
    // traceSplit's filter (optic.py:1262) has already dropped this ray: it
    // stays as it is, and its split part is only marked dropped too
    if (live && (rv.vignetted[i] != 0 || !(rv.flux[i] >= min_flux))) {
        if (sp.vignetted) sp.vignetted[i] = 1;
        return;
    }
    Ray r;
    r.x = rv.x[i]; r.y = rv.y[i]; r.z = rv.z[i];
    r.vx = rv.vx[i]; r.vy = rv.vy[i]; r.vz = rv.vz[i];
    r.t = rv.t[i];
    const double w = rv.wavelength[i], f = rv.flux[i];
    r.vig = rv.vignetted[i] != 0;
    r.fail = rv.failed[i] != 0;
    const bool fail0 = r.fail;
    Ray q = r;                       // the split ray starts as a copy (trace.py:125)
    double rf = f, sf = f;
    bool hit = false;
    if (!fail0) {
        hit = split_ray<K>(xf.dr, xf.drot, (SurfPtr)surf, medium_n((MediumPtr)m2, w), r, q, niter);
        if (hit) {
            rf = f*transmit;
            sf = f*reflect;
            rv.x[i] = r.x; rv.y[i] = r.y; rv.z[i] = r.z;
            rv.vx[i] = r.vx; rv.vy[i] = r.vy; rv.vz[i] = r.vz;
            rv.t[i] = r.t;
            rv.flux[i] = rf;
        }
        if (r.fail) {
            rv.failed[i] = 1;
            rv.vignetted[i] = 1;
        }
    }
    // the Interface's obscuration on both parts (optic.py:491-494), every
    // ray included, as batoid.cpp:151-172
    if (olen > 0) {
        if (!r.vig && obsc_contains((ObscPtr)obsc, olen, r.x, r.y)) {
            rv.vignetted[i] = 1;
            r.vig = true;
        }
        if (!q.vig) q.vig = obsc_contains((ObscPtr)obsc, olen, q.x, q.y);
    }
    lr = !r.vig && rf >= min_flux;
    ls = !q.vig && sf >= min_flux;
    if (!sp.flux) return;                           // no split part asked for
    sp.flux[i] = sf;
    sp.vignetted[i] = q.vig;
    sp.failed[i] = q.fail;
    // live mode: a split ray the filter drops (vignetted, or its flux below
    // min_flux -- every one once the ray's flux times the reflectivity is)
    // is never copied out or traced further, and every later pass reads
    // only its flux and flags
    if (live && !ls) return;
    sp.x[i] = q.x; sp.y[i] = q.y; sp.z[i] = q.z;
    sp.vx[i] = q.vx; sp.vy[i] = q.vy; sp.vz[i] = q.vz;
    sp.t[i] = q.t;
    sp.wavelength[i] = w;
}

// `counts` (live mode, may be null): the numbers of refracted and split
// rays that pass traceSplit's filter, added up by wave ballots into
// kCountSlots partial sums each (the wave's block picks the slot), so that
// no one address takes every wave's atomic.
constexpr int kCountSlots = 64;

template <int K>
__global__ __launch_bounds__(kBlock) void k_rsplit(
    Xform xf, const bt_surface* __restrict__ surf, const bt_medium* __restrict__ m2,
    double reflect, double transmit, const bt_obsc* __restrict__ obsc, int olen, bt_rays rv,
    bt_rays sp, int niter, int live, double min_flux, unsigned long long* __restrict__ counts)
{
    const int64_t i = (int64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    bool lr = false, ls = false;
    if (i < rv.n)
        rsplit_ray<K>(i, xf, surf, m2, reflect, transmit, obsc, olen, rv, sp, niter, live,
                      min_flux, lr, ls);
    if (counts) {
        const uint64_t mr = __ballot(lr), ms = __ballot(ls);
        if ((threadIdx.x & 63) == 0) {
            const int slot = (int)(blockIdx.x % kCountSlots);
            if (mr) atomicAdd(counts + slot, (unsigned long long)__popcll(mr));
            if (ms) atomicAdd(counts + kCountSlots + slot, (unsigned long long)__popcll(ms));
        }
    }
}

// ---------------------------------------------------------------------------
// A ray set carried through consecutive Interfaces in one pass (bt_split_chains)
//
// Between two reflections a traceSplit set meets every Interface on its way
// out.  One launch per Interface reads and writes the whole set each time
// (132 B a ray and Interface, and a launch); here the ray stays in registers
// over the chain, each split's reflected part goes to its own buffer as it
// arises, and a ray that the filter drops is only marked dropped in the
// buffers that follow.  Bytes: the set once in and once out, each reflected
// ray that is kept once.  Bound by FP64 issue then, as the plan kernel.
// traceSplit of 998,388 rays, 44 paths: see batoid_amd/split_chain.py.
// ---------------------------------------------------------------------------
using ChainStepPtr = const BT_CONSTANT bt_chain_step*;
using ChainPtr = const BT_CONSTANT bt_chain*;
using SetPtr = const BT_CONSTANT bt_rays*;

__device__ __forceinline__ bt_rays read_set(SetPtr p)
{
    bt_rays r;
    r.x = p->x; r.y = p->y; r.z = p->z;
    r.vx = p->vx; r.vy = p->vy; r.vz = p->vz;
    r.t = p->t; r.wavelength = p->wavelength; r.flux = p->flux;
    r.vignetted = p->vignetted; r.failed = p->failed;
    r.n = p->n;
    return r;
}

struct ChainRay {
    Ray r;
    double flux;
    bool drop;                       // by the filter, or never kept
};

template <int K, bool kPlain>
__device__ __forceinline__ void chain_ray(ChainStepPtr steps, int nstep, bt_rays in, int64_t i,
                                          double min_flux, int first_live, int niter,
                                          ChainRay& c, Range& rg)
{
    Ray& r = c.r;
    r.vig = in.vignetted[i] != 0;
    c.flux = in.flux[i];
    c.drop = first_live && (r.vig || !(c.flux >= min_flux));
    r.fail = false;
    if (!c.drop) {
        r.fail = in.failed[i] != 0;
        r.x = in.x[i]; r.y = in.y[i]; r.z = in.z[i];
        r.vx = in.vx[i]; r.vy = in.vy[i]; r.vz = in.vz[i];
        r.t = in.t[i];
    }
    MediumPtr cached = nullptr;      // the dispersive medium `index` belongs to
    double index = 0.0;
    for (int k = 0; k < nstep; k++) {
        const ChainStepPtr st = steps + k;
        const SurfPtr surf = (SurfPtr)st->surface;
        const MediumPtr m2 = (MediumPtr)st->medium;
        const int action = st->action, olen = st->obsc_len;
        const bool dispersive = action == BT_ACT_SPLIT && m2->kind != BT_MED_CONST;
        const bool fresh = dispersive && m2 != cached;
        if (dispersive) cached = m2;
        double* const sflux = st->split.flux;
        if (!c.drop) {
            if (action == BT_ACT_SPLIT) {
                Ray q = r;           // the split ray starts as a copy (trace.py:125)
                double sf = c.flux;
                if (fresh) index = medium_n(m2, in.wavelength[i]);
                if (!r.fail && split_parts<K, kPlain>(st->dr, st->drot, surf,
                                                      dispersive ? index : m2->p[0], r, q,
                                                      niter, rg)) {
                    sf = c.flux*st->reflectivity;
                    c.flux *= st->transmissivity;
                }
                if (olen > 0 && !q.vig) q.vig = obsc_contains((ObscPtr)st->obsc, olen, q.x, q.y);
                if (sflux) {
                    sflux[i] = sf;
                    st->split.vignetted[i] = q.vig;
                    st->split.failed[i] = q.fail;
                    if (!q.vig && sf >= min_flux) {  // else no later pass reads it
                        st->split.x[i] = q.x; st->split.y[i] = q.y; st->split.z[i] = q.z;
                        st->split.vx[i] = q.vx; st->split.vy[i] = q.vy; st->split.vz[i] = q.vz;
                        st->split.t[i] = q.t;
                        st->split.wavelength[i] = in.wavelength[i];
                        if constexpr (kPlain) {
                            rg.not_tiny(q.vx, q.vy);
                            rg.not_tiny(q.vz, q.vz);
                        }
                    }
                }
            } else if (!r.fail) {
                interact<K, kPlain>(action, st->dr, st->drot, surf, 0.0, r, niter,
                                    BT_START_REFERENCE, 0.0, rg);
            }
            if (olen > 0 && !r.vig) r.vig = obsc_contains((ObscPtr)st->obsc, olen, r.x, r.y);
            c.drop = r.vig || !(c.flux >= min_flux);
        } else if (sflux) {
            st->split.vignetted[i] = 1;
        }
    }
}

// Chain blockIdx.y over its rays: the sets that one turn back after another
// leaves independent run in one launch (36 sets of 1e6 rays fill the chip for
// 4 ms; one by one each ended on a nearly empty last round of waves).
template <int K>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(K == kKindsAnalytic ? 6 : 3)))
void k_split_chains(ChainPtr chains, double min_flux, int niter)
{
    const ChainPtr chain = chains + blockIdx.y;
    const bt_rays rays = read_set(&chain->rays);
    const ChainStepPtr steps = (ChainStepPtr)chain->steps;
    const int nstep = chain->nstep, flags = chain->flags;
    const int first_live = (flags & BT_CHAIN_FILTERED) != 0;
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= rays.n) return;
    ChainRay c;
    Range rg;
    if constexpr (kVoted<K>) {
        chain_ray<K, true>(steps, nstep, rays, i, min_flux, first_live, niter, c, rg);
        if (!c.drop) {
            rg.not_tiny(c.r.vx, c.r.vy);
            rg.not_tiny(c.r.vz, c.r.vz);
        }
        if (__builtin_expect(!__all(rg.plain()), 0)) {
            asm("" : "+v"(i));                  // nothing is kept from the plain pass
            chain_ray<K, false>(steps, nstep, rays, i, min_flux, first_live, niter, c, rg);
        }
    } else {
        chain_ray<K, false>(steps, nstep, rays, i, min_flux, first_live, niter, c, rg);
    }
    if (flags & BT_CHAIN_NO_OUTPUT) return;
    const bool keep = (flags & BT_CHAIN_KEEP) != 0;
    if (keep && (rays.vignetted[i] != 0 || !(rays.flux[i] >= min_flux))) return;
    rays.flux[i] = c.flux;
    rays.vignetted[i] = c.r.vig;
    rays.failed[i] = c.r.fail;
    if (first_live && c.drop && !keep) return;  // no later pass reads the rest
    rays.x[i] = c.r.x; rays.y[i] = c.r.y; rays.z[i] = c.r.z;
    rays.vx[i] = c.r.vx; rays.vy[i] = c.r.vy; rays.vz[i] = c.r.vz;
    rays.t[i] = c.r.t;
}

// ---------------------------------------------------------------------------
// Order-preserving selection: block b covers rays [256 b, 256 b + 256).
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool selected(const bt_rays& in, int64_t i, double min_flux)
{                                                    // optic.py:1262
    return i < in.n && in.vignetted[i] == 0 && in.flux[i] >= min_flux;
}

// Rank of this lane among the block's selected rays, and the block total.
__device__ __forceinline__ int block_rank(bool keep, int& total)
{
    __shared__ int wave_count[kBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t m = __ballot(keep);
    if (lane == 0) wave_count[wave] = __popcll(m);
    __syncthreads();
    int base = 0;
    total = 0;
    for (int k = 0; k < kBlock / 64; k++) {
        if (k < wave) base += wave_count[k];
        total += wave_count[k];
    }
    return base + __popcll(m & ((1ull << lane) - 1ull));
}

// The same over blockIdx.y = 0 .. sets of n rays each, with the per-set
// workspaces side by side: one launch where traceSplit's leaving sets took
// one each.
__global__ __launch_bounds__(kBlock) void k_select_count_many(SetPtr sets, double min_flux,
                                                              int64_t stride,
                                                              int64_t* __restrict__ counts)
{
    const bt_rays in = read_set(sets + blockIdx.y);
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    int total;
    block_rank(selected(in, i, min_flux), total);
    if (threadIdx.x == 0) counts[blockIdx.y * stride + blockIdx.x] = total;
}

__global__ __launch_bounds__(kBlock) void k_select_count(bt_rays in, double min_flux,
                                                         int64_t* __restrict__ counts)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    int total;
    block_rank(selected(in, i, min_flux), total);
    if (threadIdx.x == 0) counts[blockIdx.x] = total;
}

// Exclusive scan of the block counts by one workgroup, in chunks of
// kBlock * kScanPer counts taken in order: each thread sums kScanPer
// consecutive counts, the thread sums are scanned within each wave by
// shuffles and across the four waves through LDS (two barriers per chunk).
constexpr int kScanPer = 4;

__global__ __launch_bounds__(kBlock) void k_select_scan(const int64_t* __restrict__ counts,
                                                        int64_t nblocks,
                                                        int64_t* __restrict__ offsets,
                                                        int64_t* __restrict__ total,
                                                        int64_t stride)
{
    counts += blockIdx.x * stride;              // one workgroup per set
    offsets += blockIdx.x * stride;
    total += blockIdx.x;
    __shared__ int64_t wave_sum[kBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int64_t carry = 0;
    for (int64_t base = 0; base < nblocks; base += (int64_t)kBlock * kScanPer) {
        const int64_t b0 = base + (int64_t)threadIdx.x * kScanPer;
        int64_t c[kScanPer];
        int64_t sum = 0;
        for (int k = 0; k < kScanPer; k++) {
            c[k] = b0 + k < nblocks ? counts[b0 + k] : 0;
            sum += c[k];
        }
        int64_t incl = sum;                          // inclusive scan within the wave
        for (int d = 1; d < 64; d <<= 1) {
            const int64_t v = __shfl_up(incl, d, 64);
            if (lane >= d) incl += v;
        }
        if (lane == 63) wave_sum[wave] = incl;
        __syncthreads();
        int64_t before = carry, chunk = 0;
        for (int w = 0; w < kBlock / 64; w++) {
            if (w < wave) before += wave_sum[w];
            chunk += wave_sum[w];
        }
        __syncthreads();                             // wave_sum is rewritten next chunk
        int64_t run = before + incl - sum;
        for (int k = 0; k < kScanPer; k++) {
            if (b0 + k < nblocks) offsets[b0 + k] = run;
            run += c[k];
        }
        carry += chunk;
    }
    if (threadIdx.x == 0) *total = carry;
}

__device__ __forceinline__ void scatter_ray(const bt_rays& in, double min_flux,
                                            const int64_t* __restrict__ offsets,
                                            const bt_rays& out)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const bool keep = selected(in, i, min_flux);
    int total;
    const int rank = block_rank(keep, total);
    if (!keep) return;
    const int64_t o = offsets[blockIdx.x] + rank;
    if (o >= out.n) return;                          // out smaller than the count
    out.x[o] = in.x[i]; out.y[o] = in.y[i]; out.z[o] = in.z[i];
    out.vx[o] = in.vx[i]; out.vy[o] = in.vy[i]; out.vz[o] = in.vz[i];
    out.t[o] = in.t[i];
    out.wavelength[o] = in.wavelength[i];
    out.flux[o] = in.flux[i];
    out.vignetted[o] = in.vignetted[i];
    out.failed[o] = in.failed[i];
}

__global__ __launch_bounds__(kBlock) void k_select_scatter(bt_rays in, double min_flux,
                                                           const int64_t* __restrict__ offsets,
                                                           bt_rays out)
{
    scatter_ray(in, min_flux, offsets, out);
}

__global__ __launch_bounds__(kBlock) void k_select_scatter_many(
    SetPtr sets, double min_flux, const int64_t* __restrict__ offsets, int64_t stride, SetPtr outs)
{
    const bt_rays in = read_set(sets + blockIdx.y), out = read_set(outs + blockIdx.y);
    if (out.n == 0) return;
    scatter_ray(in, min_flux, offsets + blockIdx.y * stride, out);
}

int64_t select_blocks(int64_t n) { return (n + kBlock - 1) / kBlock; }

}  // namespace bt

using namespace bt;

extern "C" {

namespace {
int rsplit_launch(const bt_surface* surface, const double* dr, const double* drot,
                  const bt_medium* m2, const bt_coating* coating, const bt_obsc* obsc,
                  int obsc_len, bt_rays rays, bt_rays split, int niter, int live,
                  double min_flux, int kinds, int64_t* counts, void* stream, const char* name)
{
    const std::string n(name);
    if (!surface || !dr || !drot || !m2 || !coating)
        return fail(BT_E_NULL, n + ": null argument");
    if (obsc_len < 0 || (obsc_len > 0 && !obsc))
        return fail(BT_E_SIZE, n + ": bad obscuration program");
    if (niter < 0) return fail(BT_E_SIZE, n + ": negative niter");
    // live mode may ask for no split part: every split column NULL, n = 0
    const bool no_split = live && split.n == 0 && !split.x && !split.y && !split.z &&
                          !split.vx && !split.vy && !split.vz && !split.t &&
                          !split.wavelength && !split.flux && !split.vignetted && !split.failed;
    if (rays.n < 0 || (!no_split && split.n < rays.n))
        return fail(BT_E_SIZE, n + ": split holds fewer rays");
    if (rays.n == 0) return 0;
    if (!rays_ok(rays) || (!no_split && !rays_ok(split)))
        return fail(BT_E_NULL, n + ": incomplete ray columns");
    if (rays.n > (int64_t)0x7fffffff * kBlock)
        return fail(BT_E_SIZE, n + ": too many rays");
    auto* c = reinterpret_cast<unsigned long long*>(counts);
    if (kinds & BT_PLAN_ANALYTIC)
        hipLaunchKernelGGL(k_rsplit<kKindsAnalytic>, dim3(grid_for(rays.n)), dim3(kBlock), 0,
                           as_stream(stream), make_xform(dr, drot), surface, m2,
                           coating->reflectivity, coating->transmissivity, obsc, obsc_len, rays,
                           split, niter, live, min_flux, c);
    else
        hipLaunchKernelGGL(k_rsplit<kKindsAll>, dim3(grid_for(rays.n)), dim3(kBlock), 0,
                           as_stream(stream), make_xform(dr, drot), surface, m2,
                           coating->reflectivity, coating->transmissivity, obsc, obsc_len, rays,
                           split, niter, live, min_flux, c);
    return check_launch(name);
}
}  // namespace

int bt_rsplit(const bt_surface* surface, const double* dr, const double* drot,
              const bt_medium* m2, const bt_coating* coating, const bt_obsc* obsc,
              int obsc_len, bt_rays rays, bt_rays split, int niter, void* stream)
{
    return rsplit_launch(surface, dr, drot, m2, coating, obsc, obsc_len, rays, split, niter, 0,
                         0.0, 0, nullptr, stream, "bt_rsplit");
}

int bt_rsplit_live(const bt_surface* surface, const double* dr, const double* drot,
                   const bt_medium* m2, const bt_coating* coating, const bt_obsc* obsc,
                   int obsc_len, bt_rays rays, bt_rays split, double min_flux, int niter,
                   int kinds, int64_t* counts, void* stream)
{
    return rsplit_launch(surface, dr, drot, m2, coating, obsc, obsc_len, rays, split, niter, 1,
                         min_flux, kinds, counts, stream, "bt_rsplit_live");
}

int bt_split_chains(const bt_chain* chains, int nchain, int64_t n, double min_flux, int niter,
                    int kinds, void* stream)
{
    if (nchain < 0 || nchain > 65535 || n < 0 || niter < 0)
        return fail(BT_E_SIZE, "bt_split_chains: bad count");
    if (n > (int64_t)0x7fffffff * kBlock) return fail(BT_E_SIZE, "bt_split_chains: too many rays");
    if (nchain == 0 || n == 0) return 0;
    if (!chains) return fail(BT_E_NULL, "bt_split_chains: null chains");
    const auto kernel = (kinds & BT_PLAN_ANALYTIC)    ? k_split_chains<kKindsAnalytic>
                        : (kinds & BT_PLAN_FLAT_SUMS) ? k_split_chains<kKindsFlatSums>
                                                      : k_split_chains<kKindsAll>;
    hipLaunchKernelGGL(kernel, dim3(grid_for(n), (unsigned)nchain), dim3(kBlock), 0,
                       as_stream(stream), (ChainPtr)chains, min_flux, niter);
    return check_launch("bt_split_chains");
}

int64_t bt_select_workspace_bytes(int64_t n)
{
    if (n < 0) return -1;
    return 2 * (select_blocks(n) + 1) * (int64_t)sizeof(int64_t);
}

int bt_select_count(bt_rays in, double min_flux, int64_t* count, void* workspace,
                    int64_t workspace_bytes, void* stream)
{
    if ((in.n > 0 && !rays_ok(in)) || in.n < 0 || !count || !workspace)
        return fail(BT_E_NULL, "bt_select_count: null argument");
    if (workspace_bytes < bt_select_workspace_bytes(in.n))
        return fail(BT_E_SIZE, "bt_select_count: workspace too small");
    const int64_t nb = select_blocks(in.n);
    int64_t* counts = static_cast<int64_t*>(workspace);
    int64_t* offsets = counts + nb + 1;
    hipStream_t s = as_stream(stream);
    if (nb > 0) {
        if (nb > 0x7fffffff) return fail(BT_E_SIZE, "bt_select_count: too many rays");
        hipLaunchKernelGGL(k_select_count, dim3((unsigned)nb), dim3(kBlock), 0, s, in,
                           min_flux, counts);
        const int rc = check_launch("bt_select_count");
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_select_scan, dim3(1), dim3(kBlock), 0, s, (const int64_t*)counts, nb,
                       offsets, count, (int64_t)0);
    return check_launch("bt_select_count");
}

int bt_select_scatter(bt_rays in, double min_flux, bt_rays out, const void* workspace,
                      int64_t workspace_bytes, void* stream)
{
    if ((in.n > 0 && !rays_ok(in)) || in.n < 0 || !workspace ||
        (out.n > 0 && !rays_ok(out)))
        return fail(BT_E_NULL, "bt_select_scatter: null argument");
    if (workspace_bytes < bt_select_workspace_bytes(in.n))
        return fail(BT_E_SIZE, "bt_select_scatter: workspace too small");
    const int64_t nb = select_blocks(in.n);
    if (nb == 0 || out.n == 0) return 0;
    const int64_t* offsets = static_cast<const int64_t*>(workspace) + nb + 1;
    hipLaunchKernelGGL(k_select_scatter, dim3((unsigned)nb), dim3(kBlock), 0,
                       as_stream(stream), in, min_flux, offsets, out);
    return check_launch("bt_select_scatter");
}

int bt_select_count_many(const bt_rays* in, int nset, int64_t n, double min_flux, int64_t* count,
                         void* workspace, int64_t workspace_bytes, void* stream)
{
    if (nset < 0 || nset > 65535 || n < 0) return fail(BT_E_SIZE, "bt_select_count_many: bad count");
    if (nset == 0) return 0;
    if (!in || !count || !workspace) return fail(BT_E_NULL, "bt_select_count_many: null argument");
    if (workspace_bytes / nset < bt_select_workspace_bytes(n))
        return fail(BT_E_SIZE, "bt_select_count_many: workspace too small");
    const int64_t nb = select_blocks(n), stride = 2 * (nb + 1);
    if (nb > 0x7fffffff) return fail(BT_E_SIZE, "bt_select_count_many: too many rays");
    int64_t* counts = static_cast<int64_t*>(workspace);
    hipStream_t s = as_stream(stream);
    if (nb > 0) {
        hipLaunchKernelGGL(k_select_count_many, dim3((unsigned)nb, (unsigned)nset), dim3(kBlock),
                           0, s, (SetPtr)in, min_flux, stride, counts);
        const int rc = check_launch("bt_select_count_many");
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_select_scan, dim3((unsigned)nset), dim3(kBlock), 0, s,
                       (const int64_t*)counts, nb, counts + nb + 1, count, stride);
    return check_launch("bt_select_count_many");
}

int bt_select_scatter_many(const bt_rays* in, const bt_rays* out, int nset, int64_t n,
                           double min_flux, const void* workspace, int64_t workspace_bytes,
                           void* stream)
{
    if (nset < 0 || nset > 65535 || n < 0)
        return fail(BT_E_SIZE, "bt_select_scatter_many: bad count");
    const int64_t nb = select_blocks(n), stride = 2 * (nb + 1);
    if (nset == 0 || nb == 0) return 0;
    if (!in || !out || !workspace) return fail(BT_E_NULL, "bt_select_scatter_many: null argument");
    if (workspace_bytes / nset < bt_select_workspace_bytes(n))
        return fail(BT_E_SIZE, "bt_select_scatter_many: workspace too small");
    if (nb > 0x7fffffff) return fail(BT_E_SIZE, "bt_select_scatter_many: too many rays");
    const int64_t* offsets = static_cast<const int64_t*>(workspace) + nb + 1;
    hipLaunchKernelGGL(k_select_scatter_many, dim3((unsigned)nb, (unsigned)nset), dim3(kBlock),
                       0, as_stream(stream), (SetPtr)in, min_flux, offsets, stride, (SetPtr)out);
    return check_launch("bt_select_scatter_many");
}

}  // extern "C"
