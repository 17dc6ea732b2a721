// montrealer.hip -- the montrealer and the loop montrealer of one matrix (thewalrus/_montrealer.py
// :37-101) as sums over walks.
//
// The reference sums tr(Sigma_S^n) over the subsets S of the n modes with alternating signs, 2^n
// terms of n products; what survives the signs are the closed walks of n steps that visit every mode
// once (on either of its two copies), each counted 2n times over its starting points and directions,
// and for the loop part the open walks conj(zeta) .. zeta that do.  Those are summed here directly,
// by subset: with F[S][v, c] the weight of all walks over the modes of S that end on copy c of v,
//     F[S][v, c] = sum_(u in S \ v, c') F[S \ v][u, c'] Sigma[(u, c'), (v, c)],
// which takes 2^n n^2 multiply-adds and cancels nothing (the alternating sum loses a digit every
// two or three modes).  Three sums: closed walks from either copy of mode 0 over the other modes
// (halved: rotations and directions), and open walks over all modes.  Each is met in the middle: F
// grows from the start over subsets of up to ceil(r / 2) of its r modes, its mirror image G (walks
// onward to the end) over up to floor(r / 2), and
//     sum_(|S| = ceil(r/2)) sum_(w not in S) (F[S] Sigma)[w, c] G[rest][w, c].
// A layer holds the subsets of one size by rank (combinatorial number system), s x 2 values each,
// so only two layers of F and G are kept.
//
// Bound: launches and their latency up to n = 16 (a layer is a few microseconds of gathers from L2),
// memory traffic above.  The subset sum on the matrix cores (sieve_pm1m.hip, which plans and batches
// of montrealer requests still run) took 847 us of kernel at n = 14 and 3.3 ms at n = 16.
#include <algorithm>

#include "wh_device.h"
#include "wh_launch.h"

namespace {

constexpr int kMaxModes = 24;
constexpr int kThreads = 256;
constexpr int kFinalBlocks = 256;   // partial sums per task
constexpr int kWholeModes = 8;      // up to here one workgroup, every layer in LDS
constexpr int kWholeThreads = 1024;
constexpr int kFewValues = 1100;    // layers up to this many values share the first launch

struct RankTable {
    uint32_t c[kMaxModes + 1][kMaxModes + 2];  // C(p, k)
    constexpr RankTable() : c() {
        for (int p = 0; p <= kMaxModes; ++p) {
            c[p][0] = 1;
            for (int k = 1; k <= kMaxModes + 1; ++k) c[p][k] = p == 0 ? 0 : c[p - 1][k - 1] + c[p - 1][k];
        }
    }
};
static __constant__ RankTable kRank = RankTable();

// the table in LDS (a lane's lookups are a dependent chain: 64 cycles each there, several times that
// through the caches)
struct RankLds {
    const uint32_t* c;
    __device__ __forceinline__ uint32_t operator()(int p, int k) const { return c[p * (kMaxModes + 2) + k]; }
};
constexpr int kRankWords = (kMaxModes + 1) * (kMaxModes + 2);
__device__ __forceinline__ RankLds load_rank(uint32_t* lds) {
    for (int e = threadIdx.x; e < kRankWords; e += blockDim.x) lds[e] = (&kRank.c[0][0])[e];
    return RankLds{lds};
}

// the subset of size k with this rank, as a mask over r modes
__device__ __forceinline__ uint32_t unrank(const RankLds& C, uint32_t rank, int k, int r) {
    uint32_t mask = 0;
    for (int p = r - 1; k > 0 && p >= 0; --p) {
        const uint32_t c = C(p, k);
        if (c <= rank) {
            mask |= 1u << p;
            rank -= c;
            --k;
        }
    }
    return mask;
}
__device__ __forceinline__ uint32_t rank_of(const RankLds& C, uint32_t mask) {
    uint32_t rank = 0;
    for (int k = 1; mask; ++k, mask &= mask - 1) rank += C(__ffs((int)mask) - 1, k);
    return rank;
}

}  // namespace

// One walk sum: r modes (modes base .. base + r - 1 of the matrix), a = ceil(r / 2), b = r - a.
struct wh_mtl_task {
    int r, base, a, b;
};
struct wh_mtl_args {
    int n, ntask;
    wh_mtl_task t[3];
    const double2* sigma;  // 2n x 2n
    const double2* ends;   // per task: start [r][2], then end [r][2] (task stride 4 n)
    int64_t stride;        // complex elements of one layer buffer; buffers [task][dir][parity]
};

// f(u, x0, x1) for every mode u of the subset and its two stored values at src, in order; the loads
// of four modes are issued together (one at a time, each is a round trip to L2)
template <class F>
__device__ __forceinline__ void for_ends(uint32_t mask, int count, const cplx* src, F f) {
    for (int i = 0; i < count; i += 4) {
        cplx x[8];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (i + q < count) {
                x[2 * q] = src[2 * (i + q)];
                x[2 * q + 1] = src[2 * (i + q) + 1];
            }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (i + q < count) {
                f(__ffs((int)mask) - 1, x[2 * q], x[2 * q + 1]);
                mask &= mask - 1;
            }
    }
}

// value idx = (rank, j) of layer s from the layer below: the kept mode p_j of the rank's subset as
// the end point.  K(u, c', v, c): the step's weight.
template <class Step>
__device__ __forceinline__ void mtl_value(const RankLds& C, const cplx* below, cplx* out, int64_t idx, int s, int r, Step K) {
    const uint32_t rank = (uint32_t)(idx / s);
    const int j = (int)(idx - (int64_t)rank * s);
    uint32_t mask = unrank(C, rank, s, r);
    uint32_t m = mask;
    for (int i = 0; i < j; ++i) m &= m - 1;
    const int v = __ffs((int)m) - 1;
    uint32_t rest = mask & ~(1u << v);
    const cplx* src = below + (int64_t)rank_of(C, rest) * (s - 1) * 2;
    cplx o0 = cmk(0.0, 0.0), o1 = cmk(0.0, 0.0);
    for_ends(rest, s - 1, src, [&](int u, cplx x0, cplx x1) {
        cmac(o0, x0, K(u, 0, v, 0));
        cmac(o0, x1, K(u, 1, v, 0));
        cmac(o1, x0, K(u, 0, v, 1));
        cmac(o1, x1, K(u, 1, v, 1));
    });
    out[2 * idx] = o0;
    out[2 * idx + 1] = o1;
}

// Sigma blocks by mode pair in LDS: sg[((u n + v) 2 + c') 2 + c] = Sigma[(u, c'), (v, c)]
__device__ __forceinline__ void mtl_load_sigma(cplx* sg, const double2* sigma, int n) {
    for (int e = threadIdx.x; e < 4 * n * n; e += blockDim.x) {
        const int c = e & 1, cp = (e >> 1) & 1, uv = e >> 2, u = uv / n, v = uv - u * n;
        const double2 x = sigma[(int64_t)(u + cp * n) * 2 * n + v + c * n];
        sg[e] = cmk(x.x, x.y);
    }
}

// value idx of layer s of (task, direction) from buffer to buffer
__device__ __forceinline__ void mtl_step(const RankLds& C, const cplx* sg, int n, const wh_mtl_task& T, int dir,
                                         const cplx* below, cplx* out, int64_t idx, int s) {
    const int base = T.base;
    if (dir == 0)
        mtl_value(C, below, out, idx, s, T.r, [&](int u, int cp, int v, int c) {
            return sg[(((u + base) * n + v + base) * 2 + cp) * 2 + c];
        });
    else  // onward walks: the step leads from v to u
        mtl_value(C, below, out, idx, s, T.r, [&](int u, int cp, int v, int c) {
            return sg[(((v + base) * n + u + base) * 2 + c) * 2 + cp];
        });
}

// Layers s0..s1 of every task, both directions: grid.y = task x 2 + direction.  One layer takes as
// many workgroups as it has values; the first few (s1 > s0) are small and run in one workgroup per
// (task, direction), a barrier between layers instead of a launch.
__global__ void __launch_bounds__(1024)
wh_mtl_layer(wh_mtl_args A, cplx* work, int s0, int s1) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    __shared__ uint32_t s_rank[kRankWords];
    cplx* sg = reinterpret_cast<cplx*>(wh_smem);
    const int task = blockIdx.y >> 1, dir = blockIdx.y & 1;
    const wh_mtl_task T = A.t[task];
    const int last = min(s1, dir ? T.b : T.a);
    if (s0 > last ) return;
    const RankLds C = load_rank(s_rank);
    mtl_load_sigma(sg, A.sigma, A.n);
    __syncthreads();
    for (int s = s0; s <= last; ++s) {
        const int64_t count = (int64_t)C(T.r, s) * s;
        const cplx* below = s == 2 ? reinterpret_cast<const cplx*>(A.ends) + (int64_t)task * 4 * A.n + dir * 2 * T.r
                                   : work + ((task * 2 + dir) * 2 + ((s - 1) & 1)) * A.stride;
        cplx* out = work + ((task * 2 + dir) * 2 + (s & 1)) * A.stride;
        for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < count;
             idx += (int64_t)gridDim.x * blockDim.x)
            mtl_step(C, sg, A.n, T, dir, below, out, idx, s);
        __syncthreads();  // (with several layers the grid is one workgroup wide)
    }
}

// item idx of the meeting sum: subset S of size a by rank, and its k-th mode outside (b > 0) or its
// k-th mode (b = 0: the end weights themselves)
__device__ __forceinline__ cplx mtl_meet(const RankLds& C, const wh_mtl_task& T, int n, const cplx* sg, const cplx* F, const cplx* G,
                                         const cplx* end, int64_t idx) {
    const int per = T.b > 0 ? T.b : T.a;
    const uint32_t rank = (uint32_t)(idx / per);
    const int k = (int)(idx - (int64_t)rank * per);
    const uint32_t mask = unrank(C, rank, T.a, T.r);
    const cplx* src = F + (int64_t)rank * T.a * 2;
    cplx o = cmk(0.0, 0.0);
    if (T.b == 0) {
        uint32_t m = mask;
        for (int i = 0; i < k; ++i) m &= m - 1;
        const int v = __ffs((int)m) - 1;
        cmac(o, src[2 * k], end[2 * v]);
        cmac(o, src[2 * k + 1], end[2 * v + 1]);
        return o;
    }
    const uint32_t out = ~mask & ((1u << T.r) - 1u);
    uint32_t m = out;
    for (int i = 0; i < k; ++i) m &= m - 1;
    const int w = __ffs((int)m) - 1;
    cplx h0 = cmk(0.0, 0.0), h1 = cmk(0.0, 0.0);
    for_ends(mask, T.a, src, [&](int u, cplx x0, cplx x1) {
        const cplx* q = sg + ((u + T.base) * n + w + T.base) * 4;
        cmac(h0, x0, q[0]);
        cmac(h0, x1, q[2]);
        cmac(h1, x0, q[1]);
        cmac(h1, x1, q[3]);
    });
    const cplx* g = G + ((int64_t)rank_of(C, out) * T.b + k) * 2;
    cmac(o, h0, g[0]);
    cmac(o, h1, g[1]);
    return o;
}

// sum of the block's lanes' compensated sums on thread 0 (fixed order)
__device__ __forceinline__ csum block_csum(csum acc, double4* s_w) {
    for (int m = 1; m < WH_WAVE; m <<= 1) {
        const double r = __shfl_xor(acc.sr, m, WH_WAVE), rc = __shfl_xor(acc.cr, m, WH_WAVE);
        const double i = __shfl_xor(acc.si, m, WH_WAVE), ic = __shfl_xor(acc.ci, m, WH_WAVE);
        acc.add_pair(r, rc, i, ic);
    }
    if (threadIdx.x % WH_WAVE == 0) s_w[threadIdx.x / WH_WAVE] = make_double4(acc.sr, acc.cr, acc.si, acc.ci);
    __syncthreads();
    csum s;
    s.zero();
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x / WH_WAVE); ++w) s.add_pair(s_w[w].x, s_w[w].y, s_w[w].z, s_w[w].w);
    __syncthreads();
    return s;
}

__global__ void __launch_bounds__(kThreads)
wh_mtl_meet(wh_mtl_args A, const cplx* __restrict__ work, double4* __restrict__ partials) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    __shared__ double4 s_w[kThreads / WH_WAVE];
    __shared__ uint32_t s_rank[kRankWords];
    cplx* sg = reinterpret_cast<cplx*>(wh_smem);
    const int task = blockIdx.y;
    const wh_mtl_task T = A.t[task];
    const RankLds C = load_rank(s_rank);
    mtl_load_sigma(sg, A.sigma, A.n);
    __syncthreads();
    const cplx* ends = reinterpret_cast<const cplx*>(A.ends) + (int64_t)task * 4 * A.n;
    const cplx* F = T.a == 1 ? ends : work + ((task * 2 + 0) * 2 + (T.a & 1)) * A.stride;
    const cplx* G = T.b == 1 ? ends + 2 * T.r : work + ((task * 2 + 1) * 2 + (T.b & 1)) * A.stride;
    const int64_t count = (int64_t)C(T.r, T.a) * (T.b > 0 ? T.b : T.a);
    csum acc;
    acc.zero();
    for (int64_t idx = (int64_t)blockIdx.x * kThreads + threadIdx.x; idx < count; idx += (int64_t)gridDim.x * kThreads)
        acc.add(mtl_meet(C, T, A.n, sg, F, G, ends + 2 * T.r, idx));
    const csum s = block_csum(acc, s_w);
    if (threadIdx.x == 0) partials[(int64_t)task * kFinalBlocks + blockIdx.x] = make_double4(s.sr, s.cr, s.si, s.ci);
}

// the tasks' sums, halved and added; out and flag are pinned host memory
__global__ void __launch_bounds__(WH_WAVE)
wh_mtl_fold(const double4* __restrict__ partials, int ntask, int blocks, double2* __restrict__ out,
            uint64_t* __restrict__ flag, uint64_t seq) {
    csum s;
    s.zero();
    for (int t = 0; t < ntask; ++t) {
        const csum a = wave_fold(partials + (int64_t)t * kFinalBlocks, blocks, 1, threadIdx.x);
        s.add_pair(a.sr, a.cr, a.si, a.ci);
    }
    if (threadIdx.x == 0) {
        *out = make_double2(0.5 * (s.sr + s.cr), 0.5 * (s.si + s.ci));
        wh_call_done(flag, seq);
    }
}

// n <= kWholeModes: one workgroup, inputs from pinned memory, every layer in LDS
__global__ void __launch_bounds__(kWholeThreads)
wh_mtl_whole(wh_mtl_args A, double2* __restrict__ result, uint64_t* __restrict__ flag, uint64_t seq) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    __shared__ double4 s_w[kWholeThreads / WH_WAVE];
    __shared__ uint32_t s_rank[kRankWords];
    const RankLds C = load_rank(s_rank);
    cplx* sg = reinterpret_cast<cplx*>(wh_smem);
    cplx* ends = sg + 4 * A.n * A.n;
    cplx* work = ends + 4 * A.n * A.ntask;
    const int n = A.n;
    mtl_load_sigma(sg, A.sigma, n);
    for (int e = threadIdx.x; e < 4 * n * A.ntask; e += blockDim.x) {
        const double2 x = A.ends[e];
        ends[e] = cmk(x.x, x.y);
    }
    __syncthreads();
    int top = 0;
    for (int t = 0; t < A.ntask; ++t) top = max(top, A.t[t].a);
    const int groups = A.ntask * 2, per = kWholeThreads / WH_WAVE / groups * WH_WAVE;  // threads per (task, dir)
    const int grp = threadIdx.x / per, lane = threadIdx.x % per;
    for (int s = 2; s <= top; ++s) {
        if (grp < groups) {
            const int task = grp >> 1, dir = grp & 1;
            const wh_mtl_task T = A.t[task];
            if (s <= (dir ? T.b : T.a)) {
                const int count = (int)C(T.r, s) * s;
                const cplx* below = s == 2 ? ends + task * 4 * n + dir * 2 * T.r
                                           : work + (grp * 2 + ((s - 1) & 1)) * (int)A.stride;
                cplx* out = work + (grp * 2 + (s & 1)) * (int)A.stride;
                for (int idx = lane; idx < count; idx += per) mtl_step(C, sg, n, T, dir, below, out, idx, s);
            }
        }
        __syncthreads();
    }
    csum sum;
    sum.zero();
    for (int t = 0; t < A.ntask; ++t) {
        const wh_mtl_task T = A.t[t];
        const cplx* e = ends + t * 4 * n;
        const cplx* F = T.a == 1 ? e : work + ((t * 2 + 0) * 2 + (T.a & 1)) * (int)A.stride;
        const cplx* G = T.b == 1 ? e + 2 * T.r : work + ((t * 2 + 1) * 2 + (T.b & 1)) * (int)A.stride;
        const int count = (int)C(T.r, T.a) * (T.b > 0 ? T.b : T.a);
        csum acc;
        acc.zero();
        for (int idx = threadIdx.x; idx < count; idx += blockDim.x)
            acc.add(mtl_meet(C, T, n, sg, F, G, e + 2 * T.r, idx));
        const csum s = block_csum(acc, s_w);
        sum.add_pair(s.sr, s.cr, s.si, s.ci);
    }
    if (threadIdx.x == 0) {
        *result = make_double2(0.5 * (sum.sr + sum.cr), 0.5 * (sum.si + sum.ci));
        wh_call_done(flag, seq);
    }
}

namespace {

int64_t choose(int n, int k) { return RankTable().c[n][k]; }

wh_mtl_args mtl_args(int n, bool loop) {
    wh_mtl_args A = {};
    A.n = n;
    A.ntask = (n > 1 ? 2 : 0) + (loop ? 1 : 0);
    for (int t = 0; t < A.ntask; ++t) {
        const bool open = loop && t == A.ntask - 1;
        wh_mtl_task& T = A.t[t];
        T.r = open ? n : n - 1;
        T.base = open ? 0 : 1;
        T.a = (T.r + 1) / 2;
        T.b = T.r - T.a;
        for (int s = 2; s <= T.a; ++s) A.stride = std::max(A.stride, choose(T.r, s) * s * 2);
    }
    return A;
}

}  // namespace

int wh_mtl_whole_modes() { return kWholeModes; }
size_t wh_mtl_ends_elems(int n, bool loop) { return (size_t)mtl_args(n, loop).ntask * 4 * n; }
size_t wh_mtl_work_bytes(int n, bool loop) {
    const wh_mtl_args A = mtl_args(n, loop);
    return (size_t)std::max<int64_t>(A.stride, 1) * A.ntask * 4 * sizeof(cplx) +
           (size_t)A.ntask * kFinalBlocks * sizeof(double4);
}

// Per task (closed walks from copy 0 and 1 of mode 0 when n > 1, then open walks): the weights of a
// first and of a last step by mode and copy.
void wh_mtl_ends(int n, const double* sigma, const double* zeta, double* ends) {
    const wh_mtl_args A = mtl_args(n, zeta != nullptr);
    for (int t = 0; t < A.ntask; ++t) {
        const wh_mtl_task& T = A.t[t];
        double* st = ends + (size_t)t * 8 * n;
        double* en = st + 4 * (size_t)T.r;
        for (int v = 0; v < T.r; ++v)
            for (int c = 0; c < 2; ++c) {
                const size_t e = (size_t)v + T.base + (size_t)c * n;
                for (int q = 0; q < 2; ++q) {
                    if (T.base == 0) {
                        st[(v * 2 + c) * 2 + q] = q ? -zeta[2 * e + 1] : zeta[2 * e];
                        en[(v * 2 + c) * 2 + q] = zeta[2 * e + q];
                    } else {
                        const size_t z = (size_t)t * n;  // copy t of mode 0
                        st[(v * 2 + c) * 2 + q] = sigma[(z * 2 * n + e) * 2 + q];
                        en[(v * 2 + c) * 2 + q] = sigma[(e * 2 * n + z) * 2 + q];
                    }
                }
            }
    }
}

// The walk sums of one matrix: sigma and ends in pinned (n <= kWholeModes) or device memory, work of
// wh_mtl_work_bytes on the device.
hipError_t wh_launch_montrealer(int n, bool loop, const void* sigma, const void* ends, void* work, void* out,
                                uint64_t* flag, uint64_t seq, hipStream_t stream) {
    if (n < 2 || n > kMaxModes) return hipErrorInvalidValue;
    wh_mtl_args A = mtl_args(n, loop);
    A.sigma = (const double2*)sigma;
    A.ends = (const double2*)ends;
    if (n <= kWholeModes) {
        const size_t lds = ((size_t)4 * n * n + 4 * n * A.ntask + (size_t)A.stride * A.ntask * 4) * sizeof(cplx);
        static wh_lds_limit lim;
        hipError_t e = wh_raise_lds_limit((const void*)wh_mtl_whole, lds, lim);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(wh_mtl_whole, dim3(1), dim3(kWholeThreads), lds, stream, A, (double2*)out, flag, seq);
        return hipGetLastError();
    }
    cplx* layers = (cplx*)work;
    double4* partials = (double4*)(layers + A.stride * A.ntask * 4);
    const size_t lds = (size_t)4 * n * n * sizeof(cplx);
    int top = 0;
    int64_t items = 1;
    for (int t = 0; t < A.ntask; ++t) {
        top = std::max(top, A.t[t].a);
        items = std::max(items, choose(A.t[t].r, A.t[t].a) * std::max(A.t[t].b, 1));
    }
    auto largest = [&](int s) {
        int64_t count = 0;
        for (int t = 0; t < A.ntask; ++t) count = std::max(count, choose(A.t[t].r, s) * s);
        return count;
    };
    int s = 2;
    while (s < top && largest(s + 1) <= kFewValues) ++s;  // layers 2..s in one launch
    hipLaunchKernelGGL(wh_mtl_layer, dim3(1, (unsigned)A.ntask * 2), dim3(1024), lds, stream, A, layers, 2, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    for (++s; s <= top; ++s) {
        hipLaunchKernelGGL(wh_mtl_layer, dim3((unsigned)((largest(s) + kThreads - 1) / kThreads), (unsigned)A.ntask * 2),
                           dim3(kThreads), lds, stream, A, layers, s, s);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    const int blocks = (int)std::min<int64_t>(kFinalBlocks, (items + kThreads - 1) / kThreads);
    hipLaunchKernelGGL(wh_mtl_meet, dim3((unsigned)blocks, (unsigned)A.ntask), dim3(kThreads), lds, stream, A, layers,
                       partials);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(wh_mtl_fold, dim3(1), dim3(WH_WAVE), 0, stream, partials, A.ntask, blocks, (double2*)out, flag,
                       seq);
    return hipGetLastError();
}
