// sieve_pm1s.hip -- the all-ones Glynn sieve on the FP64 matrix cores with symmetric powers:
// the terms of _hafnian.py:443-462 (plain) and :546-569 (even loop) when rpt is all ones,
// complex matrices (and real ones, one real MFMA per block product), half-products
// formulation, with 60% of the block products of sieve_pm1m.hip at n_pad = 40, each complex one
// from three real MFMAs.
//
// With A = Ax symmetric, X the swap of the two halves and D_d = diag(d) (d = +-1 repeating over
// the halves, so X D_d = D_d X and (X D_d)^2 = I), the term matrix is B = A X D_d and
//     C_a = B^a X D_d = A (X D_d A)^(a-1)   is symmetric, and so is V_a = D_d C_a D_d.
// Each wave keeps V_a in LDS and forms the products
//     R_(a+1) = V_a (X A) = D_d C_(a+1),   V_(a+1)[i][j] = R_(a+1)[i][j] d_j,
// on the matrix cores for the upper block groups only (T (T + 1) / 2 of the T^2 groups of
// sieve_pm1m.hip), with X A staged once per workgroup and no sign in the products: the lane
// stores R d_j at (i, j) and, by symmetry, at (j, i).  The power traces are
//     tr(B^(a+b)) = sum_(i,k) C_a[i][k] V_b[swap k][swap i] = sum_(i,k) d_i R_a[i][k] V_b[swap k][swap i],
// a summand symmetric in (i, k): the upper groups off the diagonal count twice and the row sign
// d_i scales each row group's partial sum once.  The loop vectors z_a = B^a D follow the chain
// z_a = A (X D_d z_(a-1)), and the loop dots use y_a = X D_d z_a as in sieve_pm1m.hip.  The
// montrealer (0/1 factors: D_d^2 is not I) stays on sieve_pm1m.hip.  Each wave keeps the power
// traces and loop scalars of its last few terms in LDS and forms their coefficients together,
// one term per lane.
//
// Lane map and MFMA layout as sieve_pm1m.hip: x = lane & 3, br = bit 2, bc = bit 3,
// y = lane >> 4; group (p, q) holds R[8p + 4br + y][8q + 4bc + x].  The signs d of the lane's
// rows and columns live in one mask register and flip the sign bit of the values they scale;
// where a complex product takes four MFMAs, its -Im(a) Im(b) term uses the matrix core's negate
// modifier on B.
#include <algorithm>

#include "pm1s_body.h"
#include "wh_launch.h"

// The real plain instance at T = 3 (n = 17..24) fits 128 registers and, without the loop
// vectors and slots, 33 KB of LDS per 4-wave workgroup: four waves per SIMD instead of three.
template <int T, bool LOOP, bool RE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu((RE && T == 3 && !LOOP) ? 4 : 1)))
wh_sieve_pm1s(const wh_job_dev* __restrict__ jobs, int njobs, const cplx* __restrict__ pool,
              double4* __restrict__ partials, int64_t block_offset) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    const int64_t b = blockIdx.x + block_offset;
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].chunk_base <= b) lo = mid; else hi = mid - 1;
    }
    pm1s_body<T, LOOP, RE>(jobs[lo], pool, partials, b, wh_smem, blockDim.x / WH_WAVE);
}

// ---- Persistent form for a whole batch: the chunks of the symmetric-kernel groups with tile
// sides 4..6 (the per-class launches' blocks, the same chunking and the same per-chunk work,
// so every partial is bit-identical) are items of one queue, largest class first; each
// workgroup of the grid (as many as stay resident) takes items from an atomic counter until the
// queue is empty.  The last workgroup to finish (a second counter) folds every job of the batch
// in wh_fold's order.  A one-thread kernel clears the two counters first (a kernel,
// not a memset, so the pair can sit in a captured graph).  Other kernel classes of the batch
// run before them on the same stream.
struct MixedItems {
    int ngroups;
    int njobs;  // jobs folded at the end (the whole batch)
    wh_mixed_group g[WH_MIXED_MAX_GROUPS];
};

template <int T, bool LOOP>
__device__ __noinline__ void mixed_item(const wh_job_dev* __restrict__ jobs, int lo, int hi, const cplx* __restrict__ pool,
                                        double4* __restrict__ partials, int64_t b, unsigned char* smem, int nw) {
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].chunk_base <= b) lo = mid; else hi = mid - 1;
    }
    pm1s_body<T, LOOP>(jobs[lo], pool, partials, b, smem, nw);
}

__global__ void __launch_bounds__(256)
wh_sieve_pm1s_persistent(const wh_job_dev* __restrict__ jobs, const cplx* __restrict__ pool,
                         double4* __restrict__ partials, unsigned* __restrict__ counters, double2* __restrict__ out,
                         MixedItems items) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    __shared__ int s_item;
    __shared__ int s_last;
    int total = 0;
    for (int k = 0; k < items.ngroups; ++k) total += (int)(items.g[k].block_end - items.g[k].block_begin);
    for (;;) {
        if (threadIdx.x == 0) s_item = (int)atomicAdd(&counters[0], 1u);
        __syncthreads();  // also: the previous item's last LDS reads are done
        int i = s_item;
        __syncthreads();
        if (i >= total) break;
        int k = 0;
        while (i >= (int)(items.g[k].block_end - items.g[k].block_begin)) {
            i -= (int)(items.g[k].block_end - items.g[k].block_begin);
            ++k;
        }
        const wh_mixed_group& G = items.g[k];
        const int64_t b = G.block_begin + i;
        const int lo = G.job_begin, hi = G.job_end - 1;
#define WH_MIXED_CASE(TT)                                                                   \
    case TT:                                                                                \
        if (G.loop) mixed_item<TT, true>(jobs, lo, hi, pool, partials, b, wh_smem, G.nw);  \
        else mixed_item<TT, false>(jobs, lo, hi, pool, partials, b, wh_smem, G.nw);        \
        break;
        switch (G.T) {
            WH_MIXED_CASE(1)
            WH_MIXED_CASE(2)
            WH_MIXED_CASE(3)
            WH_MIXED_CASE(4)
            WH_MIXED_CASE(5)
            WH_MIXED_CASE(6)
            default: break;
        }
#undef WH_MIXED_CASE
    }
    // the partials this workgroup wrote are visible device-wide before it counts itself done
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) s_last = atomicAdd(&counters[1], 1u) == gridDim.x - 1;
    __syncthreads();
    if (!s_last) return;
    __threadfence();
    for (int q = threadIdx.x / WH_WAVE; q < items.njobs; q += blockDim.x / WH_WAVE)
        wh_fold_job(jobs[q], partials, out, threadIdx.x % WH_WAVE);
}

__global__ void wh_clear_counters(unsigned* __restrict__ counters) { counters[threadIdx.x] = 0u; }

size_t wh_pm1s_lds_bytes(int T, int nw, bool real, bool loop) {
    size_t NP = 8 * (size_t)T, S = NP + WH_PM1S_PAD;
    size_t PTN = 4 * (size_t)T + 4, NB = T >= 6 ? 1 : T == 5 ? 7 : 8;
    size_t mat = (NP * S * (real ? sizeof(double) : sizeof(cplx)) + 31) / 32 * 32;
    size_t dvn = loop ? NP : 0, sl = loop ? 2 * PTN : PTN;
    size_t small = (NB * sl + 2 * dvn) * sizeof(cplx);
    return (1 + nw) * mat + dvn * sizeof(cplx) + nw * small + nw * sizeof(double4) + 32;
}

// the dynamic-LDS limit set on each instance (shared by its launches and occupancy queries, so
// that a query for a smaller workgroup never lowers what a launch relies on)
template <int T, bool LOOP, bool RE>
static wh_lds_limit& lds_limit_s() {
    static wh_lds_limit lim;
    return lim;
}

template <int T, bool LOOP, bool RE>
static hipError_t launch_s(const wh_job_dev* jobs, int njobs, const void* pool, void* partials, int64_t nblocks,
                           int64_t block_offset, int nw, hipStream_t stream) {
    size_t lds = wh_pm1s_lds_bytes(T, nw, RE, LOOP);
    hipError_t err = wh_raise_lds_limit((const void*)wh_sieve_pm1s<T, LOOP, RE>, lds, lds_limit_s<T, LOOP, RE>());
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((wh_sieve_pm1s<T, LOOP, RE>), dim3((unsigned)nblocks), dim3(nw * WH_WAVE), lds, stream,
                       jobs, njobs, (const cplx*)pool, (double4*)partials, block_offset);
    return hipGetLastError();
}

hipError_t wh_launch_pm1s_persistent(const wh_mixed_group* groups, int ngroups, const wh_job_dev* jobs, int njobs,
                                     const void* pool, void* partials, unsigned* counters, void* out, int nwg,
                                     hipStream_t stream) {
    if (ngroups < 1 || ngroups > WH_MIXED_MAX_GROUPS || nwg < 1) return hipErrorInvalidValue;
    MixedItems items;
    items.ngroups = ngroups;
    items.njobs = njobs;
    size_t lds = 0;
    for (int k = 0; k < ngroups; ++k) {
        items.g[k] = groups[k];
        if (groups[k].T < 1 || groups[k].T > 6 || groups[k].nw < 1 || groups[k].nw > 4) return hipErrorInvalidValue;
        lds = std::max(lds, wh_pm1s_lds_bytes(groups[k].T, groups[k].nw, false, true));
    }
    static wh_lds_limit lim;
    hipError_t err = wh_raise_lds_limit((const void*)wh_sieve_pm1s_persistent, lds, lim);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(wh_clear_counters, dim3(1), dim3(2), 0, stream, counters);
    hipLaunchKernelGGL(wh_sieve_pm1s_persistent, dim3((unsigned)nwg), dim3(256), lds, stream, jobs,
                       (const cplx*)pool, (double4*)partials, counters, (double2*)out, items);
    return hipGetLastError();
}

template <int T, bool LOOP, bool RE>
static int resident_s(int nw) {
    int blocks = 0;
    const size_t lds = wh_pm1s_lds_bytes(T, nw, RE, LOOP);
    if (lds > 160 * 1024) return 0;  // the CU's LDS: no workgroup of this size fits
    // a failed query leaves no error behind for the caller's next HIP call to report
    if (wh_raise_lds_limit((const void*)wh_sieve_pm1s<T, LOOP, RE>, lds, lds_limit_s<T, LOOP, RE>()) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, (const void*)wh_sieve_pm1s<T, LOOP, RE>, nw * WH_WAVE,
                                                     lds) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return blocks;
}

int wh_pm1s_resident(int T, int nw, bool real, bool loop) {
    if (nw < 1 || nw > 4) return 0;
#define WH_PM1S_RES(TT)                                                                        \
    case TT:                                                                                   \
        return loop ? resident_s<TT, true, false>(nw) : resident_s<TT, false, false>(nw);
#define WH_PM1S_RES_R(TT)                                                                      \
    case TT:                                                                                   \
        if (real) return loop ? resident_s<TT, true, true>(nw) : resident_s<TT, false, true>(nw); \
        return loop ? resident_s<TT, true, false>(nw) : resident_s<TT, false, false>(nw);
    switch (T) {
        WH_PM1S_RES_R(1)
        WH_PM1S_RES_R(2)
        WH_PM1S_RES_R(3)
        WH_PM1S_RES_R(4)
        WH_PM1S_RES_R(5)
        WH_PM1S_RES(6)
        WH_PM1S_RES(7)
        WH_PM1S_RES(8)
        default: return 0;
    }
#undef WH_PM1S_RES
#undef WH_PM1S_RES_R
}

hipError_t wh_launch_pm1s(int T, bool loop, bool real, const wh_job_dev* jobs, int njobs, const void* pool,
                          void* partials, int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream) {
#define WH_PM1S_ARGS jobs, njobs, pool, partials, nblocks, block_offset, nw, stream
#define WH_PM1S_CASE(TT)                                                              \
    case TT:                                                                          \
        return loop ? launch_s<TT, true, false>(WH_PM1S_ARGS) : launch_s<TT, false, false>(WH_PM1S_ARGS);
#define WH_PM1S_CASE_R(TT)                                                            \
    case TT:                                                                          \
        if (real) return loop ? launch_s<TT, true, true>(WH_PM1S_ARGS) : launch_s<TT, false, true>(WH_PM1S_ARGS); \
        return loop ? launch_s<TT, true, false>(WH_PM1S_ARGS) : launch_s<TT, false, false>(WH_PM1S_ARGS);
    switch (T) {
        WH_PM1S_CASE_R(1)
        WH_PM1S_CASE_R(2)
        WH_PM1S_CASE_R(3)
        WH_PM1S_CASE_R(4)
        WH_PM1S_CASE_R(5)
        WH_PM1S_CASE(6)
        WH_PM1S_CASE(7)
        WH_PM1S_CASE(8)
        default: return hipErrorInvalidValue;
    }
#undef WH_PM1S_CASE
#undef WH_PM1S_CASE_R
#undef WH_PM1S_ARGS
}
