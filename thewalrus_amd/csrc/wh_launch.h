// wh_launch.h -- host-side launchers exported by the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

// A kernel's dynamic-LDS limit, raised only when a launch needs more than the kernel was last
// given on the current device: hipFuncSetAttribute costs about as much as the launch itself, and
// the limit never has to shrink.  One instance per kernel (a function-local static).
struct wh_lds_limit {
    std::atomic<size_t> bytes[64];  // per device; zero in static storage
    std::mutex mu;
};
inline hipError_t wh_raise_lds_limit(const void* fn, size_t lds, wh_lds_limit& lim) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (lim.bytes[dev].load(std::memory_order_acquire) >= lds) return hipSuccess;
    std::lock_guard<std::mutex> g(lim.mu);
    if (lim.bytes[dev].load(std::memory_order_relaxed) >= lds) return hipSuccess;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e == hipSuccess) lim.bytes[dev].store(lds, std::memory_order_release);
    return e;
}

struct wh_job_dev;
struct wh_lhb_job;
struct wh_call;

size_t wh_generic_lds_bytes(int MM, int NQ);
hipError_t wh_launch_generic(const wh_job_dev* jobs, int njobs, const void* pool, void* partials,
                             int64_t nblocks, int64_t block_offset, int MM, int NQ, hipStream_t stream);
size_t wh_pm1_lds_bytes(int T, bool real, int nw);
hipError_t wh_launch_pm1(int T, bool half, bool real, bool loop, const wh_job_dev* jobs, int njobs,
                         const void* pool, void* partials, int64_t nblocks, int64_t block_offset,
                         int nw, hipStream_t stream);
size_t wh_pm1m_lds_bytes(int T, int nw);
hipError_t wh_launch_pm1m(int T, bool loop, bool mtl, const wh_job_dev* jobs, int njobs, const void* pool,
                          void* partials, int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream);
size_t wh_pm1s_lds_bytes(int T, int nw, bool real, bool loop);
// Workgroups of nw waves that one CU holds for that instance (registers, LDS, wave slots), from
// the runtime's occupancy calculator on the current device; 0 when it cannot say.
int wh_pm1s_resident(int T, int nw, bool real, bool loop);
struct wh_mixed_group;
hipError_t wh_launch_pm1s_persistent(const wh_mixed_group* groups, int ngroups, const wh_job_dev* jobs, int njobs,
                                     const void* pool, void* partials, unsigned* counters, void* out, int nwg,
                                     hipStream_t stream);
hipError_t wh_launch_pm1s(int T, bool loop, bool real, const wh_job_dev* jobs, int njobs, const void* pool,
                          void* partials, int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream);
size_t wh_rep_lds_bytes(int T, bool real, bool loop, int nw, int H);
size_t wh_rep4_lds_bytes(bool real, bool loop, int nw, int H);
hipError_t wh_launch_rep4(int H, bool real, bool loop, const wh_job_dev* jobs, int njobs, const void* pool,
                          void* partials, int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream);
hipError_t wh_launch_rep(int T, int H, bool real, bool loop, const wh_job_dev* jobs, int njobs, const void* pool,
                         void* partials, int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream);
size_t wh_sym_lds_bytes(int T, int nw, bool loop, int H);
hipError_t wh_launch_sym(int T, bool loop, int H, const wh_job_dev* jobs, int njobs, const void* pool, void* partials,
                         int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream);
// Single-call forms (wh_call): the most terms per wave a chunk may have (0: no such form for that
// tile side), the launches over nblocks = chunks x nsplit workgroups of C.nw waves (then the fold),
// or (whole, T = 1) one workgroup of C.nsplit x C.nw waves (at most 8) that reads the staged inputs
// (job first, C.in_bytes) from pinned memory and folds.
int wh_pm1s_call_terms(int T);
hipError_t wh_launch_pm1s_call(int T, bool loop, bool real, const wh_job_dev* job, const void* pool, int64_t nblocks,
                               bool whole, const wh_call& C, hipStream_t stream);
int wh_sym_call_terms(int T);
hipError_t wh_launch_sym_call(int T, bool loop, int H, const wh_job_dev* job, const void* pool, void* partials,
                              int64_t nblocks, const wh_call& C, hipStream_t stream);
int wh_fold_call_chunks();  // the most chunks the fold takes
hipError_t wh_launch_fold_call(const wh_job_dev* job, int nchunks, const wh_call& C, hipStream_t stream);
// Copies `bytes` (rounded up to 16) from pinned host memory to device memory with a kernel.
hipError_t wh_launch_stage_in(const void* pinned, void* dst, size_t bytes, hipStream_t stream);
hipError_t wh_launch_fold(const wh_job_dev* jobs, int njobs, const void* partials, void* out,
                          hipStream_t stream);
size_t wh_lhb_lds_bytes(int T, int nw, int nmax, int nf);
int wh_lhb_waves(int T, int nmax, int nf);
hipError_t wh_launch_lhb(const wh_lhb_job* job, const void* pool, void* partials, int64_t nblocks, int T, bool full,
                         int nw, int nmax, int nf, int nout, void* out, uint64_t* flag, uint64_t seq,
                         hipStream_t stream);
// Montrealer of one matrix by walk sums (2 <= n <= 24): the staged inputs are Sigma (2n x 2n) and
// wh_mtl_ends_elems values written by wh_mtl_ends (in pinned memory for n up to
// wh_mtl_whole_modes, else in device memory); out and flag are pinned host memory.
int wh_mtl_whole_modes();
size_t wh_mtl_ends_elems(int n, bool loop);
size_t wh_mtl_work_bytes(int n, bool loop);
void wh_mtl_ends(int n, const double* sigma, const double* zeta, double* ends);
hipError_t wh_launch_montrealer(int n, bool loop, const void* sigma, const void* ends, void* work, void* out,
                                uint64_t* flag, uint64_t seq, hipStream_t stream);
hipError_t wh_launch_hermite(int n, const int* cut, int renorm, const void* R, const void* y, const double* sq,
                             const void* C, void* G, hipStream_t stream);
// Copies count 16-byte elements to pinned memory in chunks, in order; a chunk is there once its
// wh_copy_out_flags() flags (pinned, [chunk][flag]) read seq.
int wh_copy_out_flags();
hipError_t wh_launch_copy_out(const void* src, void* pinned, int64_t count, int64_t chunk_elems, uint64_t* flags,
                              uint64_t seq, hipStream_t stream);
