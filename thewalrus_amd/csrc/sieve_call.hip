// sieve_call.hip -- the all-ones symmetric-power sieve (sieve_pm1s.hip) for one request per launch:
// the drop-in's synchronous call up to n = 24 (tile sides 1 to 3), whose few thousand terms leave
// most of the chip idle in the batch form (four terms in a row per wave: an n = 20 call had 32
// workgroups of 36 us on 256 CUs).  One term per wave (wh_call): the same bits.  From n = 26 on a
// call's chunks fill the chip and the batch form stays.
#include "pm1s_body.h"
#include "wh_launch.h"

template <int T, bool LOOP, bool RE>
__global__ void __launch_bounds__(512)
wh_sieve_call(const wh_job_dev* __restrict__ job, const cplx* __restrict__ pool, wh_call C) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    const int nw = blockDim.x / WH_WAVE;
    const int wave = threadIdx.x / WH_WAVE;
    const wh_job_dev& J = *job;
    __shared__ double4 s_terms[8];
    // block -> (chunk, part), or the one block's waves -> (part, wave): the wave's offset in its chunk
    const bool whole = nw > C.nw;
    const int part = whole ? wave / C.nw : blockIdx.x % C.nsplit;
    pm1s_body<T, LOOP, RE, true>(J, pool, nullptr, whole ? 0 : blockIdx.x / C.nsplit, wh_smem, nw,
                                 part * C.nw + wave % C.nw, whole ? s_terms : C.terms + (int64_t)blockIdx.x * nw);
    if (whole) {
        __syncthreads();
        if (wave == 0) wh_call_fold(J, C, s_terms, threadIdx.x);
    }
}

// Folds a call's terms: one wave.
__global__ void __launch_bounds__(WH_WAVE)
wh_fold_call(const wh_job_dev* __restrict__ job, wh_call C) {
    wh_call_fold(*job, C, C.terms, threadIdx.x);
}

hipError_t wh_launch_fold_call(const wh_job_dev* job, const wh_call& C, hipStream_t stream) {
    hipLaunchKernelGGL(wh_fold_call, dim3(1), dim3(WH_WAVE), 0, stream, job, C);
    return hipGetLastError();
}

int wh_pm1s_call_terms(int T) { return T == 1 ? GeoS<1>::NB : T == 2 ? GeoS<2>::NB : T == 3 ? GeoS<3>::NB : 0; }

template <int T, bool LOOP, bool RE>
static hipError_t launch_call(const wh_job_dev* job, const void* pool, int64_t nblocks, int nw, const wh_call& C,
                              hipStream_t stream) {
    const size_t lds = wh_pm1s_lds_bytes(T, nw, RE, LOOP);
    static wh_lds_limit lim;
    hipError_t err = wh_raise_lds_limit((const void*)wh_sieve_call<T, LOOP, RE>, lds, lim);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((wh_sieve_call<T, LOOP, RE>), dim3((unsigned)nblocks), dim3(nw * WH_WAVE), lds, stream, job,
                       (const cplx*)pool, C);
    return hipGetLastError();
}

hipError_t wh_launch_pm1s_call(int T, bool loop, bool real, const wh_job_dev* job, const void* pool, int64_t nblocks,
                               int nw, const wh_call& C, hipStream_t stream) {
    if (nw < 1 || nw > 8 || C.nw < 1 || C.nsplit < 1) return hipErrorInvalidValue;
#define WH_CALL_ARGS job, pool, nblocks, nw, C, stream
#define WH_CALL_CASE(TT)                                                                                       \
    case TT:                                                                                                   \
        if (real) return loop ? launch_call<TT, true, true>(WH_CALL_ARGS) : launch_call<TT, false, true>(WH_CALL_ARGS); \
        return loop ? launch_call<TT, true, false>(WH_CALL_ARGS) : launch_call<TT, false, false>(WH_CALL_ARGS);
    switch (T) {
        WH_CALL_CASE(1)
        WH_CALL_CASE(2)
        WH_CALL_CASE(3)
        default: return hipErrorInvalidValue;
    }
#undef WH_CALL_CASE
#undef WH_CALL_ARGS
}
