// hermite.hip -- the multidimensional Hermite recursion behind hafnian_batched: the loop
// hafnians of reduction(A, k) for every k below the cutoffs, as one tensor G
// (thewalrus/_hermite_multidimensional.py:173-216, recursion :251-303).
//
// G[idx] = y_i G[idx - e_i] - sum_(l >= i, ki_l > 0) w(ki_l) R_il G[idx - e_i - e_l], where i is
// the first nonzero position of idx and ki = idx - e_i (w(k) = k, or sqrt(k) with a final
// division by sqrt(idx_i) for the renormalised form).  An entry depends only on entries with
// the same zero prefix and a smaller value at position i, so the tensor fills in steps
// (i, v): i from n-1 down to 0, v = 1..cut_i - 1.  Step (i, v) is the contiguous slice
// [v stride_i, (v + 1) stride_i) of the row-major tensor -- every entry of it in parallel, with
// coalesced reads of the slices v - 1 and v - 2.  Steps whose slice is small run inside one
// workgroup (barrier between steps; the innermost positions' whole subtensor in LDS, where a step
// takes 0.3 us against 1.3 us through the caches); the large ones are one launch each.  HBM-bound:
// per entry one write and 1 + (n - i) reads of 16 bytes.  A tensor goes to the host by a kernel that
// writes pinned memory chunk by chunk, each chunk with its flag (wh_copy_out).
#include <algorithm>
#include <cstring>

#include "wh_device.h"

#define WH_HERM_MAXN 32

struct wh_herm_args {
    int n;
    int renorm;
    int cut[WH_HERM_MAXN];
    int64_t stride[WH_HERM_MAXN];
};

// One entry of slice (i, v): s indexes the suffix (positions i+1..n-1).  U: the index type (32-bit
// divisions take a third of the time of 64-bit ones and serve every tensor below 2^32 entries).
template <class U>
__device__ __forceinline__ void herm_entry(const wh_herm_args& a, const cplx* __restrict__ R,
                                           const cplx* __restrict__ y, const double* __restrict__ sq, cplx* G, int i,
                                           int v, U s) {
    const U lin = (U)v * (U)a.stride[i] + s;
    const U ki = lin - (U)a.stride[i];
    cplx u = cmul(y[i], G[ki]);
    const int n = a.n;
    // l = i: ki_i = v - 1
    if (v > 1) {
        double w = a.renorm ? sq[v - 1] : (double)(v - 1);
        u = csub(u, cmul(cmulr(R[i * n + i], w), G[ki - (U)a.stride[i]]));
    }
    for (int l = i + 1; l < n; ++l) {
        int kl = (int)((s / (U)a.stride[l]) % (U)a.cut[l]);
        if (kl > 0) {
            double w = a.renorm ? sq[kl] : (double)kl;
            u = csub(u, cmul(cmulr(R[i * n + l], w), G[ki - (U)a.stride[l]]));
        }
    }
    G[lin] = a.renorm ? cdivr(u, sq[v]) : u;
}

// Steps (i, v) for i = n-1 down to i_stop (exclusive), every v, in one workgroup; positions past
// i_lds in LDS (their subtensor of lds_count entries), then written out.
extern "C" __global__ void __launch_bounds__(1024)
wh_hermite_small(wh_herm_args a, const cplx* __restrict__ R, const cplx* __restrict__ y,
                 const double* __restrict__ sq, const cplx* __restrict__ C, cplx* G, int i_stop, int i_lds,
                 int lds_count) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    cplx* sub = reinterpret_cast<cplx*>(wh_smem);
    if (threadIdx.x == 0) {
        sub[0] = C[0];
        if (lds_count == 0) G[0] = C[0];
    }
    __syncthreads();
    int i = a.n - 1;
    for (; i > i_lds; --i)
        for (int v = 1; v < a.cut[i]; ++v) {
            for (uint32_t s = threadIdx.x; s < (uint32_t)a.stride[i]; s += blockDim.x)
                herm_entry<uint32_t>(a, R, y, sq, sub, i, v, s);
            __syncthreads();
        }
    for (int e = threadIdx.x; e < lds_count; e += blockDim.x) G[e] = sub[e];
    __syncthreads();
    for (; i > i_stop; --i)
        for (int v = 1; v < a.cut[i]; ++v) {
            for (int64_t s = threadIdx.x; s < a.stride[i]; s += blockDim.x)
                herm_entry<uint64_t>(a, R, y, sq, G, i, v, (uint64_t)s);
            __syncthreads();
        }
}

// One step (i, v) over its whole slice (grid-stride).
template <class U>
__global__ void __launch_bounds__(256)
wh_hermite_step(wh_herm_args a, const cplx* __restrict__ R, const cplx* __restrict__ y,
                const double* __restrict__ sq, cplx* G, int i, int v) {
    const U step = (U)gridDim.x * blockDim.x, end = (U)a.stride[i];
    for (U s = (U)blockIdx.x * blockDim.x + threadIdx.x; s < end; s += step) herm_entry<U>(a, R, y, sq, G, i, v, s);
}

// Device memory to pinned memory in chunks of chunk_elems (16 B each), in order: each workgroup
// copies its share of a chunk and then sets its flag of that chunk to seq.
constexpr int kCopyBlocks = 64;
__global__ void __launch_bounds__(256)
wh_copy_out(const double2* __restrict__ src, double2* __restrict__ dst, int64_t count, int64_t chunk_elems,
            uint64_t* __restrict__ flags, uint64_t seq) {
    for (int64_t c = 0, at = 0; at < count; ++c, at += chunk_elems) {
        const int64_t end = min(count, at + chunk_elems);
        for (int64_t e = at + (int64_t)blockIdx.x * 256 + threadIdx.x; e < end; e += (int64_t)kCopyBlocks * 256)
            dst[e] = src[e];
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0) wh_call_done(&flags[c * kCopyBlocks + blockIdx.x], seq);
    }
}

#include "wh_launch.h"

int wh_copy_out_flags() { return kCopyBlocks; }
hipError_t wh_launch_copy_out(const void* src, void* pinned, int64_t count, int64_t chunk_elems, uint64_t* flags,
                              uint64_t seq, hipStream_t stream) {
    if (count < 1 || chunk_elems < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(wh_copy_out, dim3(kCopyBlocks), dim3(256), 0, stream, (const double2*)src, (double2*)pinned,
                       count, chunk_elems, flags, seq);
    return hipGetLastError();
}

// Enqueues the whole recursion; every entry of G is written here (C: the value at index 0).
// Positions whose slice (stride) is at most small_max run in the single-workgroup kernel.
hipError_t wh_launch_hermite(int n, const int* cut, int renorm, const void* R, const void* y, const double* sq,
                             const void* C, void* G, hipStream_t stream) {
    wh_herm_args a;
    memset(&a, 0, sizeof a);
    a.n = n;
    a.renorm = renorm;
    int64_t total = 1;
    for (int l = n - 1; l >= 0; --l) {
        a.cut[l] = cut[l];
        a.stride[l] = total;
        total *= cut[l];
    }
    const int64_t small_max = 8192;
    int i_stop = n - 1;  // positions > i_stop go to the small kernel
    while (i_stop >= 0 && a.stride[i_stop] <= small_max) --i_stop;
    const int64_t lds_max = 6144;  // entries: 96 KB
    int i_lds = n - 1;  // positions > i_lds in LDS
    while (i_lds > i_stop && a.stride[i_lds] * a.cut[i_lds] <= lds_max) --i_lds;
    const int64_t lds_count = i_lds < n - 1 ? a.stride[i_lds + 1] * a.cut[i_lds + 1] : 0;
    const size_t lds = (size_t)std::max<int64_t>(lds_count, 1) * sizeof(cplx);
    static wh_lds_limit lim;
    hipError_t e = wh_raise_lds_limit((const void*)wh_hermite_small, lds, lim);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(wh_hermite_small, dim3(1), dim3(1024), lds, stream, a, (const cplx*)R, (const cplx*)y, sq,
                       (const cplx*)C, (cplx*)G, i_stop, i_lds, (int)lds_count);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    for (int i = i_stop; i >= 0; --i) {
        int64_t blocks = (a.stride[i] + 255) / 256;
        if (blocks > (1 << 20)) blocks = 1 << 20;  // grid-stride beyond 2^28 work-items
        for (int v = 1; v < a.cut[i]; ++v) {
            if (total + blocks * 256 < ((int64_t)1 << 32))
                hipLaunchKernelGGL(wh_hermite_step<uint32_t>, dim3((unsigned)blocks), dim3(256), 0, stream, a,
                                   (const cplx*)R, (const cplx*)y, sq, (cplx*)G, i, v);
            else
                hipLaunchKernelGGL(wh_hermite_step<uint64_t>, dim3((unsigned)blocks), dim3(256), 0, stream, a,
                                   (const cplx*)R, (const cplx*)y, sq, (cplx*)G, i, v);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}
