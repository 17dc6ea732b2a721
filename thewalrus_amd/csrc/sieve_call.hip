// sieve_call.hip -- the all-ones symmetric-power sieve (sieve_pm1s.hip) for one request per launch:
// the drop-in's synchronous call up to n = 24 (tile sides 1 to 3), whose few thousand terms leave
// most of the chip idle in the batch form (four terms in a row per wave: an n = 20 call had 32
// workgroups of 36 us on 256 CUs).  One term per wave (wh_call): the same bits.  From n = 26 on a
// call's chunks fill the chip and the batch form stays.
#include "pm1s_body.h"
#include "wh_launch.h"

// WHOLE: the request is one chunk of at most 8 terms (n <= 8): one workgroup of nsplit x nw waves,
// which fetches the staged inputs (pinned host memory) into LDS in one PCIe round trip and folds.
template <int T, bool LOOP, bool RE, bool WHOLE>
__global__ void __launch_bounds__(WHOLE ? 512 : 256)
wh_sieve_call(const wh_job_dev* __restrict__ job, const cplx* __restrict__ pool, wh_call C) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    const int nw = blockDim.x / WH_WAVE;
    const int wave = threadIdx.x / WH_WAVE;
    if constexpr (WHOLE) {
        __shared__ double4 s_terms[8];
        double2* in = reinterpret_cast<double2*>(wh_smem + C.in_off);
        for (int i = threadIdx.x; i < C.in_bytes / 16; i += blockDim.x) in[i] = reinterpret_cast<const double2*>(job)[i];
        __syncthreads();
        const wh_job_dev& J = *reinterpret_cast<const wh_job_dev*>(in);
        const cplx* P = reinterpret_cast<const cplx*>(in) +
                        (reinterpret_cast<const unsigned char*>(pool) - reinterpret_cast<const unsigned char*>(job)) / 16;
        pm1s_body<T, LOOP, RE, true>(J, P, nullptr, 0, wh_smem, nw, wave, s_terms);
        __syncthreads();
        if (wave == 0) wh_call_fold(J, C, s_terms, threadIdx.x);
    } else {
        pm1s_body<T, LOOP, RE, true>(*job, pool, nullptr, blockIdx.x / C.nsplit, wh_smem, nw,
                                     blockIdx.x % C.nsplit * nw + wave, C.terms + (int64_t)blockIdx.x * nw);
    }
}

// Folds a call's terms: one thread per chunk, then one wave over the chunks (wh_call_fold's order).
constexpr int kFoldCallThreads = 512;
__global__ void __launch_bounds__(kFoldCallThreads)
wh_fold_call(const wh_job_dev* __restrict__ job, wh_call C) {
    __shared__ double4 s_chunk[kFoldCallThreads];
    const wh_job_dev& J = *job;
    for (int c = threadIdx.x; c < J.nchunks; c += kFoldCallThreads) s_chunk[c] = wh_call_chunk(C, C.terms, c);
    __syncthreads();
    if (threadIdx.x >= WH_WAVE) return;
    const csum acc = wave_fold_with(J.nchunks, threadIdx.x, [&](int64_t c) { return s_chunk[c]; });
    const double2 v = wh_job_value(J, acc);
    if (threadIdx.x == 0) {
        *C.out = v;
        wh_call_done(C.flag, C.seq);
    }
}
int wh_fold_call_chunks() { return kFoldCallThreads; }

hipError_t wh_launch_fold_call(const wh_job_dev* job, int nchunks, const wh_call& C, hipStream_t stream) {
    if (nchunks < 1 || nchunks > kFoldCallThreads) return hipErrorInvalidValue;
    const int threads = (nchunks + WH_WAVE - 1) / WH_WAVE * WH_WAVE;
    hipLaunchKernelGGL(wh_fold_call, dim3(1), dim3(threads), 0, stream, job, C);
    return hipGetLastError();
}

// A call's inputs from the pinned staging block (read over PCIe) to device memory.  A kernel, not
// a copy: the copy's completion is a signal the next kernel's queue waits for, 7 to 10 us after
// a 2 us transfer, where two kernels of one stream follow each other at once.
__global__ void __launch_bounds__(256)
wh_stage_in(const double2* __restrict__ src, double2* __restrict__ dst, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < count) dst[i] = src[i];
}

hipError_t wh_launch_stage_in(const void* pinned, void* dst, size_t bytes, hipStream_t stream) {
    const int64_t count = (int64_t)((bytes + 15) / 16);
    if (count < 1) return hipSuccess;
    if (count > (int64_t)256 * 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(wh_stage_in, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream,
                       (const double2*)pinned, (double2*)dst, count);
    return hipGetLastError();
}

int wh_pm1s_call_terms(int T) { return T == 1 ? GeoS<1>::NB : T == 2 ? GeoS<2>::NB : T == 3 ? GeoS<3>::NB : 0; }

template <int T, bool LOOP, bool RE, bool WHOLE>
static hipError_t launch_call(const wh_job_dev* job, const void* pool, int64_t nblocks, int nw, wh_call C,
                              hipStream_t stream) {
    size_t lds = (wh_pm1s_lds_bytes(T, nw, RE, LOOP) + 15) / 16 * 16;
    C.in_off = (int)lds;
    if (WHOLE) lds += C.in_bytes;
    static wh_lds_limit lim;
    hipError_t err = wh_raise_lds_limit((const void*)wh_sieve_call<T, LOOP, RE, WHOLE>, lds, lim);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((wh_sieve_call<T, LOOP, RE, WHOLE>), dim3((unsigned)nblocks), dim3(nw * WH_WAVE), lds, stream,
                       job, (const cplx*)pool, C);
    return hipGetLastError();
}

hipError_t wh_launch_pm1s_call(int T, bool loop, bool real, const wh_job_dev* job, const void* pool, int64_t nblocks,
                               bool whole, const wh_call& C, hipStream_t stream) {
    const int nw = whole ? C.nw * C.nsplit : C.nw;
    if (C.nw < 1 || C.nsplit < 1 || nw > (whole ? 8 : 4) || (whole && (T != 1 || nblocks != 1)))
        return hipErrorInvalidValue;
    if (whole) {
        if (real)
            return loop ? launch_call<1, true, true, true>(job, pool, 1, nw, C, stream)
                        : launch_call<1, false, true, true>(job, pool, 1, nw, C, stream);
        return loop ? launch_call<1, true, false, true>(job, pool, 1, nw, C, stream)
                    : launch_call<1, false, false, true>(job, pool, 1, nw, C, stream);
    }
#define WH_CALL_ARGS job, pool, nblocks, nw, C, stream
#define WH_CALL_CASE(TT)                                                                                \
    case TT:                                                                                            \
        if (real)                                                                                       \
            return loop ? launch_call<TT, true, true, false>(WH_CALL_ARGS)                              \
                        : launch_call<TT, false, true, false>(WH_CALL_ARGS);                            \
        return loop ? launch_call<TT, true, false, false>(WH_CALL_ARGS)                                 \
                    : launch_call<TT, false, false, false>(WH_CALL_ARGS);
    switch (T) {
        WH_CALL_CASE(1)
        WH_CALL_CASE(2)
        WH_CALL_CASE(3)
        default: return hipErrorInvalidValue;
    }
#undef WH_CALL_CASE
#undef WH_CALL_ARGS
}
