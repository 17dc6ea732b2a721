// sieve_rep4.hip -- repeated rows with 2E <= 12 (2E <= 10 for odd N; h = ceil(N / 2) <= 16), four terms
// per wave, with symmetric powers on the FP64 matrix cores (tile side 3 of the repeated-row class):
// the terms of _hafnian.py:443-462 (plain) and :546-569 (loop).
//
// v_mfma_f64_4x4x4f64 forms four independent 4 x 4 x 4 block products, block b on the lanes with
// (lane >> 2) & 3 == b: with x = lane & 3 and y = lane >> 4, a lane supplies A[x][y] and B[y][x] of
// its block and receives D[y][x].  Term g of the wave takes block g, so one instruction advances
// the four terms, and a term's 12 x 12 matrices pad to 3 x 3 blocks where one term on a whole wave
// (sieve_sym.hip) pads to 16.  The powers are sieve_sym.hip's: B = A G with G = X Delta,
// C_a = A (G A)^(a-1) symmetric, W_a = C_a Delta in LDS, C_(a+1) = W_a (X A) for the 6 upper blocks
// (each complex block product three real MFMAs, 54 per power for four terms, or four in plain requests,
// where it lowers the error), traces
// tr(B^(a+b)) = sum_i delta_i sum_k C_a[i][k] W_b[s i][s k], z_a = W_a (X D), loop scalars
// sum_e delta_e z_a[s e] z_b[e].  Lane (x, y) of a term holds C[4 bi + y][4 bj + x], bi <= bj.  The
// coefficient series takes one 16-lane row per term (series_steps).
//
// A matrix that is not symmetric takes its full powers (sym_device.h), one term on the whole wave.
//
// Bound: FP64 issue: on 1024 requests of 8 modes and 32 photons (1.26 ms) the matrix cores are busy 26% of
// the time and the other vector instructions take 43%.  The registers
// leave three waves per SIMD, the LDS of two-wave workgroups with loops (31.7 KB) ten per CU; LDS bank
// conflicts take 24% of the CUs' busy cycles.  With full powers and separate row and column loop vectors
// (81 MFMAs and about 560 vector instructions per power of four terms, 244 registers) the same requests
// took 1.9 ms.  Four values stay spilled in the complex loop instance (X D is read from LDS for that: with
// it in registers 18).  One term per wave on the vector kernel padded to 8
// takes 1.4 to 1.6 times as long for 2E <= 8, on sieve_sym.hip padded to 16 2.4 times for 2E in 9..12.
#include "sym_device.h"
#include "wh_launch.h"

namespace {

constexpr int kR4N = 12;  // padded side
constexpr int kR4S = 13;  // LDS row stride (elements)
__host__ __device__ constexpr int r4_ptn(int H) { return H + 3; }  // p_1 .. p_(h+1), v likewise

// entry i of a matrix or vector in LDS: complex, or for the real instance its real part only
template <bool RE>
__device__ __forceinline__ cplx eget(const cplx* m, int i) {
    if constexpr (RE) return cmk(reinterpret_cast<const double*>(m)[i], 0.0);
    else return m[i];
}
template <bool RE>
__device__ __forceinline__ void eput(cplx* m, int i, cplx v) {
    if constexpr (RE) reinterpret_cast<double*>(m)[i] = v.re;
    else m[i] = v;
}

// Eight sums over each term's 16 lanes (lane bits 0, 1, 4, 5) at once: lane l returns the sum of
// v[((l >> 1) & 1) | (((l >> 4) & 3) << 1)] (halving stages over lane bits 5, 4, 1, then 0).
__device__ __forceinline__ double term16_sum8(const double (&v)[8], int lane) {
    double s1[4], s2[2];
#pragma unroll
    for (int k = 0; k < 4; ++k) s1[k] = dswap32(v[k], v[k + 4]);  // value k + 4 bit5
#pragma unroll
    for (int k = 0; k < 2; ++k) s2[k] = dswap16(s1[k], s1[k + 2]);  // value k + 2 bit4 + 4 bit5
    const bool b1 = (lane >> 1) & 1;
    const double keep = b1 ? s2[1] : s2[0], send = b1 ? s2[0] : s2[1];
    const double s3 = keep + dpp_d<WH_DPP_XOR2>(send);  // value bit1 + 2 bit4 + 4 bit5
    return s3 + dpp_d<WH_DPP_XOR1>(s3);
}
// over lane bits 0, 1 (the lanes of a term with the same y: one row)
__device__ __forceinline__ double xrow_sum(double v) {
    v += dpp_d<WH_DPP_XOR1>(v);
    return v + dpp_d<WH_DPP_XOR2>(v);
}

// LDS (bytes, every part a multiple of 16): X A, X D, D | per wave: four W, z of two powers of four
// terms, four term slots (p, v), prefactors | waves' sums, binomials
__host__ __device__ constexpr size_t r4_even(size_t e) { return (e + 1) / 2 * 2; }
__host__ __device__ constexpr size_t r4_head(size_t esz) { return r4_even((size_t)kR4N * kR4S + 2 * kR4N) * esz; }
__host__ __device__ constexpr size_t r4_wave(size_t esz, bool loop, int H) {
    return (r4_even((size_t)4 * kR4N * kR4S) + (loop ? 4 * 2 * kR4N : 0)) * esz +
           (size_t)4 * r4_ptn(H) * (loop ? 2 : 1) * sizeof(cplx) + 4 * sizeof(double);
}
__host__ __device__ constexpr size_t r4_lds(size_t esz, bool loop, int nw, int H) {
    return r4_head(esz) + nw * r4_wave(esz, loop, H) + nw * sizeof(double4) +
           r4_even((size_t)(kR4N / 2) * (H + 1)) * sizeof(double);
}

// The chunk [t0, t1) of a matrix that is not exactly symmetric: false if its triangles were replaced by
// their mean, else the wave's sum of terms by the full powers (sym_device.h), one term on the whole wave,
// is in wres.
template <bool RE, bool LOOP, int H>
__device__ __forceinline__ bool rep4_full(const wh_job_dev& J, const cplx* pool, int64_t t0, int64_t t1, int nw) {
    extern __shared__ __align__(32) unsigned char wh_smem[];
    constexpr int N = kR4N, S = kR4S, PTN = r4_ptn(H);
    constexpr size_t esz = RE ? sizeof(double) : sizeof(cplx);
    const int wave = threadIdx.x / WH_WAVE, lane = threadIdx.x % WH_WAVE;
    const bool odd = (J.flags & WH_F_ODD) != 0, glynn = (J.flags & WH_F_GLYNN) != 0;
    const int ne0 = J.E, ne = ne0 + (odd ? 1 : 0), h0 = J.N / 2;
    auto at = [&](size_t bytes) { return reinterpret_cast<cplx*>(wh_smem + bytes); };
    cplx* XA = at(0);
    auto entry = [&](int i, int j) {  // A[i][j] by request index
        return swp(i < ne0 ? i : i - ne0 + ne, ne) * S + (j < ne0 ? j : j - ne0 + ne);
    };
    auto get = [&](int i, int j) { return eget<RE>(XA, entry(i, j)); };
    double* scale = reinterpret_cast<double*>(at(r4_head(esz)));  // (the first wave's W)
    if (!(J.flags & WH_F_NONSYM) && !settle_symmetry(2 * ne0, odd ? kSymTolOdd : kSymTolEven, scale, get,
                                                     [&](int i, int j, cplx v) { eput<RE>(XA, entry(i, j), v); }))
        return false;
    // P | z | delta over the wave's W, p | v | o | e over its slots
    const size_t w0 = r4_head(esz) + wave * r4_wave(esz, LOOP, H);
    cplx* P = at(w0);
    cplx* z = P + N * S;
    double* dl = reinterpret_cast<double*>(z + N);
    cplx* p = at(w0 + (r4_even((size_t)4 * N * S) + (LOOP ? 4 * 2 * N : 0)) * esz);
    cplx* out[2] = {p + PTN, p + 2 * PTN};
    cplx* e = p + (LOOP ? 3 : 1) * PTN;
    double4* wres = reinterpret_cast<double4*>(wh_smem + r4_head(esz) + nw * r4_wave(esz, LOOP, H));
    const double* btab = reinterpret_cast<const double*>(wres + nw);
    const cplx* V = odd ? pool + J.v_off : nullptr;
    const cplx* Dg = LOOP ? pool + J.d_off : nullptr;
    const int el = lane < ne0 ? J.e[lane] : 0;
    uint32_t w = 1;
    for (int l = lane + 1; l < ne0; ++l) w *= (uint32_t)(J.e[l] + 1);
    csum acc;
    acc.zero();
    for (int64_t t = t0 + wave; t < t1; t += nw) {
        const int k = lane < ne0 ? (int)(((uint32_t)t / w) % (uint32_t)(el + 1)) : 0;
        const int delta = glynn ? 2 * k - el : k;
        double bin = lane < ne0 ? btab[lane * (H + 1) + k] : 1.0;
        for (int m = 1; m < 8; m <<= 1) bin *= __shfl_xor(bin, m, WH_WAVE);  // ne0 <= 6: lanes 0..7
        bin = __shfl(bin, 0, WH_WAVE);
        const int par = __popcll(__ballot(k & 1)) & 1;
        double prefac = ((h0 - par) & 1) ? -bin : bin;
        if (!odd && glynn && __shfl(delta, 0, WH_WAVE) == 0) prefac *= 0.5;
        wave_lds_sync();
        if (lane < ne0) dl[lane] = (double)delta;
        wave_lds_sync();
        if constexpr (LOOP)
            full_scalars<2>(get, [&](int j) { return Dg[j]; },
                            [&](int l, int j) { return l == 0 ? Dg[j] : odd ? V[j] : cmk(0.0, 0.0); }, ne0, h0, dl, P, S,
                            z, p, out, lane);
        else
            full_scalars<0>(get, 0, 0, ne0, h0, dl, P, S, nullptr, p, {nullptr}, lane);
        const cplx f = full_coeff<LOOP>(odd ? J.N : h0, odd, cmk(J.oddloop_re, J.oddloop_im), p, out[0], out[1], e, lane);
        acc.add(cmulr(f, prefac));
    }
    if (lane == 0) wres[wave] = make_double4(acc.sr, acc.cr, acc.si, acc.ci);
    return true;
}
// The complex instances call it: inlined, the main loop's schedule came out 1.2 times as long (512
// requests of 8 modes and 32 photons 609 -> 736 us with 9 to 12 spilled registers, plain ones 504 -> 596
// with none).  The real ones have room for it, and as a call it would cost the plain one its fourth
// wave per SIMD (235 -> 254 us).
template <bool RE, bool LOOP, int H>
__device__ __noinline__ bool rep4_full_call(const wh_job_dev& J, const cplx* pool, int64_t t0, int64_t t1, int nw) {
    return rep4_full<RE, LOOP, H>(J, pool, t0, t1, nw);
}

}  // namespace

#ifndef WH_REP4_WAVES_PER_EU
#define WH_REP4_WAVES_PER_EU 3
#endif
template <bool RE, bool LOOP, int H>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WH_REP4_WAVES_PER_EU)))
wh_sieve_rep4(const wh_job_dev* __restrict__ jobs, int njobs, const cplx* __restrict__ pool,
              double4* __restrict__ partials, int64_t block_offset) {
    extern __shared__ __align__(32) unsigned char wh_smem[];
    constexpr int N = kR4N, S = kR4S, PTN = r4_ptn(H);
    constexpr size_t esz = RE ? sizeof(double) : sizeof(cplx);
    const int64_t b = blockIdx.x + block_offset;
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].chunk_base <= b) lo = mid; else hi = mid - 1;
    }
    const wh_job_dev& J = jobs[lo];
    const int nw = blockDim.x / WH_WAVE;
    const int wave = threadIdx.x / WH_WAVE;
    const int lane = threadIdx.x % WH_WAVE;
    const int grp = (lane >> 2) & 3;  // the term (MFMA block) of the lane
    const int x = lane & 3, y = lane >> 4;
    const int gl = x + 4 * y;         // the lane's index within its term
    const int gbase = 4 * grp;        // the term's lane with gl = 0
    const bool odd = (J.flags & WH_F_ODD) != 0;  // the unpaired mode as one more edge, as in sieve_sym.hip
    const int ne0 = J.E, ne = ne0 + (odd ? 1 : 0), n = 2 * ne, h = (J.N + 1) / 2;
    const bool glynn = (J.flags & WH_F_GLYNN) != 0;

    // element pointers are cplx*, indexed through eget / eput (doubles for the real instance)
    auto at = [&](size_t bytes) { return reinterpret_cast<cplx*>(wh_smem + bytes); };
    cplx* XA = at(0);
    cplx* XD = at((size_t)N * S * esz);
    cplx* Dv = at(((size_t)N * S + N) * esz);
    const size_t w0 = r4_head(esz) + wave * r4_wave(esz, LOOP, H);
    cplx* W = at(w0 + (size_t)grp * N * S * esz);  // this term's W_a
    cplx* Z = at(w0 + (r4_even((size_t)4 * N * S) + (LOOP ? grp * 2 * N : 0)) * esz);
    cplx* slots = at(w0 + (r4_even((size_t)4 * N * S) + (LOOP ? 4 * 2 * N : 0)) * esz);
    constexpr int SL = LOOP ? 2 * PTN : PTN;
    double* pf = reinterpret_cast<double*>(slots + 4 * SL);
    double4* wres = reinterpret_cast<double4*>(wh_smem + r4_head(esz) + nw * r4_wave(esz, LOOP, H));
    double* btab = reinterpret_cast<double*>(wres + nw);
    // the partner of index c in the other half (identity on the padding)
    auto sw = [&](int c) { return c < ne ? c + ne : c < n ? c - ne : c; };

    const cplx* A = pool + J.a_off;
    const cplx* V = odd ? pool + J.v_off : nullptr;
    const cplx* Dg = LOOP ? pool + J.d_off : nullptr;
    const int n0 = 2 * ne0;
    bool rough = (J.flags & WH_F_NONSYM) != 0;  // not exactly symmetric, or not finite
    for (int e = threadIdx.x; e < N * N; e += blockDim.x) {
        const int r = e / N, c = e - r * N;
        cplx v = cmk(0.0, 0.0);
        if (r < n && c < n) {
            const int rs = sw(r);
            const int ro = rs < ne ? rs : rs - ne, co = c < ne ? c : c - ne;     // edges
            const int ri = rs < ne ? ro : ro + ne0, ci = c < ne ? co : co + ne0;  // request indices
            if (ro < ne0 && co < ne0) {
                v = A[ri * n0 + ci];
                rough = rough || !twins(v, A[ci * n0 + ri]);
            } else if (ro < ne0 && c == ne - 1) {
                v = V[ri];
                rough = rough || !finite_c(v);
            } else if (co < ne0 && rs == ne - 1) {
                v = V[ci];
            }
        }
        eput<RE>(XA, r * S + c, v);
    }
    if (LOOP) {
        auto weight = [&](int e) {
            const int eo = e < ne ? e : e - ne;
            if (eo < ne0) return Dg[e < ne ? eo : eo + ne0];
            return e < ne ? cmk(J.oddloop_re, J.oddloop_im) : cmk(0.0, 0.0);
        };
        for (int e = threadIdx.x; e < N; e += blockDim.x) {
            eput<RE>(XD, e, e < n ? weight(sw(e)) : cmk(0.0, 0.0));
            const cplx d = e < n ? weight(e) : cmk(0.0, 0.0);
            rough = rough || !finite_c(d);
            eput<RE>(Dv, e, d);
        }
    }
    for (int e = threadIdx.x; e < ne0 * (H + 1); e += blockDim.x) {
        const int i = e / (H + 1), k = e - i * (H + 1), ei = J.e[i];
        btab[e] = k <= ei ? binom_t(ei, k) : 0.0;
    }

    const int64_t t0 = (b - J.chunk_base) * J.chunk_terms;
    int64_t t1 = t0 + J.chunk_terms;
    if (t1 > J.steps) t1 = J.steps;
    csum acc;
    acc.zero();

    bool full = __syncthreads_or(rough);
    if (full) {
        if constexpr (RE) full = rep4_full<RE, LOOP, H>(J, pool, t0, t1, nw);
        else full = rep4_full_call<RE, LOOP, H>(J, pool, t0, t1, nw);
    }
    // lane gl < ne0 of each term owns digit gl: its base and the weight of the digits after it
    const int my_e = gl < ne0 ? J.e[gl] : 0;
    uint32_t my_w = 1;
    for (int l = gl + 1; l < ne0; ++l) my_w *= (uint32_t)(J.e[l] + 1);
    // the lane of the term holding the digit of index c's edge (index 0 for the padding)
    auto dlane = [&](int c) {
        const int d = c < ne ? c : c < n ? c - ne : 0;
        return gbase + (d & 3) + 16 * (d >> 2);
    };
    const int gs = gl < n ? sw(gl) : 0, ge = gl < n ? gl : 0;

    for (int64_t t = t0 + 4 * wave; t < t1 && !full; t += 4 * nw) {
        const bool valid = t + grp < t1;
        const uint32_t tu = (uint32_t)(valid ? t + grp : t);
        const int k = gl < ne0 ? (int)((tu / my_w) % (uint32_t)(my_e + 1)) : 0;
        const int delta = gl < ne0 ? (glynn ? 2 * k - my_e : k) : odd && gl == ne0 ? -1 : 0;
        int ksum = k;
        double bin = gl < ne0 ? btab[gl * (H + 1) + k] : 1.0;
        // over the term's 16 lanes (lane bits 0, 1, 4, 5): every lane receives the total
#pragma unroll
        for (int m = 1; m <= 32; m = m == 2 ? 16 : 2 * m) {
            ksum += __shfl_xor(ksum, m, WH_WAVE);
            bin *= __shfl_xor(bin, m, WH_WAVE);  // exact: a product of integers below 2^53
        }
        const int delta0 = __shfl(delta, gbase, WH_WAVE);
        double prefac = (((h - ksum) & 1) ? -1.0 : 1.0) * bin;
        if (!odd && glynn && delta0 == 0) prefac *= 0.5;
        if (!valid) prefac = 0.0;
        double dc[3], dr[3];  // delta of the lane's columns 4 c + x and rows 4 c + y (0 on the padding)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int dj = __shfl(delta, dlane(4 * c + x), WH_WAVE), di = __shfl(delta, dlane(4 * c + y), WH_WAVE);
            dc[c] = 4 * c + x < n ? (double)dj : 0.0;
            dr[c] = 4 * c + y < n ? (double)di : 0.0;
        }
        const int dg = __shfl(delta, dlane(gl), WH_WAVE);
        const double dl = gl < n ? (double)dg : 0.0;

        cplx* pt = slots + grp * SL;
        cplx* lv = pt + PTN;
        cplx C[6];  // upper blocks (0,0) (0,1) (0,2) (1,1) (1,2) (2,2)
        {
            int g = 0;
#pragma unroll
            for (int bi = 0; bi < 3; ++bi)
#pragma unroll
                for (int bj = bi; bj < 3; ++bj) C[g++] = eget<RE>(XA, sw(4 * bi + y) * S + 4 * bj + x);
        }
        auto store = [&]() {
            int g = 0;
#pragma unroll
            for (int bi = 0; bi < 3; ++bi)
#pragma unroll
                for (int bj = bi; bj < 3; ++bj, ++g) {
                    eput<RE>(W, (4 * bi + y) * S + 4 * bj + x, cmulr(C[g], dc[bj]));
                    if (bi < bj) eput<RE>(W, (4 * bj + x) * S + 4 * bi + y, cmulr(C[g], dr[bi]));
                }
        };
        auto trace = [&]() {  // lane part of sum_i delta_i sum_k C[i][k] W[s i][s k]
            cplx s = cmk(0.0, 0.0);
            int g = 0;
#pragma unroll
            for (int bi = 0; bi < 3; ++bi) {
                const int rs = sw(4 * bi + y) * S;
                cplx sd = cmk(0.0, 0.0), so = cmk(0.0, 0.0);
#pragma unroll
                for (int bj = bi; bj < 3; ++bj, ++g) {
                    const cplx w = eget<RE>(W, rs + sw(4 * bj + x));
                    if (bi == bj) cmac(sd, C[g], w);
                    else cmac(so, C[g], w);
                }
                s.re = fma(dr[bi], fma(2.0, so.re, sd.re), s.re);
                if (!RE) s.im = fma(dr[bi], fma(2.0, so.im, sd.im), s.im);
            }
            return s;
        };
        wave_lds_sync();  // the previous term's reads of W, z and the slots are done
        store();
        // p_1 = sum_e delta_e A[e][s e]
        cplx to = cmk(0.0, 0.0), f = cmk(0.0, 0.0), zp = cmk(0.0, 0.0);
        if (gl < n) to = cmulr(eget<RE>(XA, gs * S + gs), dl);
        if (LOOP) {  // f = delta_e z_(a-1)[s e], zp = z_(a-1)[e] of the lane's index, from z_0 = D
            f = cmulr(eget<RE>(Dv, gs), dl);
            zp = eget<RE>(Dv, ge);
        }
        if (LOOP && !RE && odd && gl == 0) lv[1] = cneg(Dv[ne - 1]);  // u_1
        wave_lds_sync();
        const int Ah = (h + 1) / 2;
#pragma unroll 1
        for (int a = 1;; ++a) {
            cplx te = trace();
            cplx v0 = cmk(0.0, 0.0), v1 = cmk(0.0, 0.0);
            if (LOOP) {
                // z_a = W_a (X D): upper entries from the registers, lower ones from LDS
                cplx* zc = RE ? reinterpret_cast<cplx*>(reinterpret_cast<double*>(Z) + (a & 1) * N) : Z + (a & 1) * N;
                cplx xd[3];  // X D at the lane's columns
#pragma unroll
                for (int c = 0; c < 3; ++c) xd[c] = eget<RE>(XD, 4 * c + x);
                int g = 0;
#pragma unroll
                for (int bi = 0; bi < 3; ++bi) {
                    cplx s = cmk(0.0, 0.0);
#pragma unroll
                    for (int bj = 0; bj < 3; ++bj) {
                        if (bj < bi) cmac(s, eget<RE>(W, (4 * bi + y) * S + 4 * bj + x), xd[bj]);
                        else cmac(s, cmulr(C[g++], dc[bj]), xd[bj]);
                    }
                    s.re = xrow_sum(s.re);
                    if (!RE) s.im = xrow_sum(s.im);
                    eput<RE>(zc, 4 * bi + y, s);  // the same value from the row's lanes
                }
                wave_lds_sync();
                const cplx zn = eget<RE>(zc, ge);
                v0 = cmul(f, zp);  // v_(2a-1)
                v1 = cmul(f, zn);  // v_(2a)
                if (!RE && odd) {  // b_(2a-1), b_(2a), u_(2a), u_(2a+1)
                    const double k0 = a - 0.5, k1 = a;
                    to = cmk(fma(k0, v0.re, 0.5 * to.re), fma(k0, v0.im, 0.5 * to.im));
                    te = cmk(fma(k1, v1.re, 0.5 * te.re), fma(k1, v1.im, 0.5 * te.im));
                    const cplx yd = cmulr(eget<RE>(W, gs * S + ne - 1), dl);
                    v0 = cmul(yd, zp);
                    v1 = cmul(yd, zn);
                }
                f = cmulr(eget<RE>(zc, gs), dl);
                zp = zn;
            }
            const double v8[8] = {to.re, RE ? 0.0 : to.im, te.re, RE ? 0.0 : te.im,
                                  v0.re, RE ? 0.0 : v0.im, v1.re, RE ? 0.0 : v1.im};
            const double sum8 = term16_sum8(v8, lane);
            const int kv = ((lane >> 1) & 1) | (((lane >> 4) & 3) << 1);
            if ((lane & 1) == 0 && (LOOP || kv < 4)) {
                cplx* dst = (kv < 4 ? pt : lv + (!RE && odd ? 1 : 0)) + 2 * a - 1 + ((kv >> 1) & 1);
                (kv & 1 ? dst->im : dst->re) = sum8;
            }
            if (a >= Ah) break;
            // C_(a+1) = W_a (X A) on the matrix cores, the four terms at once
            double X[6], Y[6], Zm[6];
#pragma unroll
            for (int g = 0; g < 6; ++g) X[g] = Y[g] = Zm[g] = 0.0;
#pragma unroll
            for (int kc = 0; kc < 3; ++kc) {
                cplx av[3], bv[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    av[c] = eget<RE>(W, (4 * c + x) * S + 4 * kc + y);
                    bv[c] = eget<RE>(XA, (4 * kc + y) * S + 4 * c + x);
                }
                int g = 0;
#pragma unroll
                for (int bi = 0; bi < 3; ++bi)
#pragma unroll
                    for (int bj = bi; bj < 3; ++bj, ++g) {
                        X[g] = mfma4(av[bi].re, bv[bj].re, X[g]);
                        if (!RE && !LOOP) {
                            X[g] = mfma4_nb(av[bi].im, bv[bj].im, X[g]);
                            Zm[g] = mfma4(av[bi].re, bv[bj].im, Zm[g]);
                            Zm[g] = mfma4(av[bi].im, bv[bj].re, Zm[g]);
                        } else if (!RE) {
                            Y[g] = mfma4(av[bi].im, bv[bj].im, Y[g]);
                            Zm[g] = mfma4(av[bi].re + av[bi].im, bv[bj].re + bv[bj].im, Zm[g]);
                        }
                    }
            }
#pragma unroll
            for (int g = 0; g < 6; ++g)
                C[g] = RE ? cmk(X[g], 0.0) : !LOOP ? cmk(X[g], Zm[g]) : cmk(X[g] - Y[g], Zm[g] - (X[g] + Y[g]));
            to = trace();  // C_(a+1) with W_a: p_(2a+1)
            wave_lds_sync();
            store();
            wave_lds_sync();
        }
        if (gl == 0) pf[grp] = prefac;
        wave_lds_sync();
        {  // the four terms' coefficients, one 16-lane row each
            const int m = (lane & 15) + 1, j = lane >> 4;
            const cplx* sl = slots + j * SL;
            cplx bb = cmk(0.0, 0.0);
            if (m <= h) {
                const bool sums = LOOP && !(!RE && odd);  // (odd N: b itself)
                const double half = LOOP && !sums ? 1.0 : 0.5;
                bb.re = half * sl[m].re;
                if (!RE) bb.im = half * sl[m].im;
                if (sums) {
                    bb.re = fma(0.5 * m, sl[PTN + m].re, bb.re);
                    if (!RE) bb.im = fma(0.5 * m, sl[PTN + m].im, bb.im);
                }
            }
            const bool whole = LOOP && !RE && odd;
            cplx s;
            if (LOOP && !whole) s = series_row<RE, false>(bb, h);
            else s = series_row<RE, true>(bb, h);
            if (whole) s = odd_row<16>(s, sl + PTN, h, lane);
            const double p = pf[j];
            if (m == h && p != 0.0) acc.add(cmulr(s, whole ? p : p * kInv.v[h]));
        }
    }

    // lane h - 1 of each 16-lane row holds its row's sum: the rows, then the waves, in order
    csum s;
    s.zero();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int src = 16 * j + h - 1;
        const double r = __shfl(acc.sr, src, WH_WAVE), rc = __shfl(acc.cr, src, WH_WAVE);
        const double i = __shfl(acc.si, src, WH_WAVE), ic = __shfl(acc.ci, src, WH_WAVE);
        s.add_pair(r, rc, i, ic);
    }
    if (lane == 0 && !full) wres[wave] = make_double4(s.sr, s.cr, s.si, s.ci);
    __syncthreads();
    if (threadIdx.x == 0) {
        csum sm;
        sm.zero();
        for (int w = 0; w < nw; ++w) {
            const double4 pq = wres[w];
            sm.add_pair(pq.x, pq.y, pq.z, pq.w);
        }
        partials[b] = make_double4(sm.sr, sm.cr, sm.si, sm.ci);
    }
}

size_t wh_rep4_lds_bytes(bool real, bool loop, int nw, int H) {
    return r4_lds(real ? sizeof(double) : sizeof(cplx), loop, nw, H);
}

template <bool RE, bool LOOP, int H>
static hipError_t launch_rep4(const wh_job_dev* jobs, int njobs, const void* pool, void* partials, int64_t nblocks,
                              int64_t block_offset, int nw, hipStream_t stream) {
    const size_t lds = wh_rep4_lds_bytes(RE, LOOP, nw, H);
    static wh_lds_limit lim;
    hipError_t err = wh_raise_lds_limit((const void*)wh_sieve_rep4<RE, LOOP, H>, lds, lim);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((wh_sieve_rep4<RE, LOOP, H>), dim3((unsigned)nblocks), dim3(nw * WH_WAVE), lds, stream, jobs,
                       njobs, (const cplx*)pool, (double4*)partials, block_offset);
    return hipGetLastError();
}

hipError_t wh_launch_rep4(int H, bool real, bool loop, const wh_job_dev* jobs, int njobs, const void* pool,
                          void* partials, int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream) {
#define WH_REP4_ARGS jobs, njobs, pool, partials, nblocks, block_offset, nw, stream
#define WH_REP4_CASE(HH)                                                                                          \
    case HH:                                                                                                      \
        if (real) return loop ? launch_rep4<true, true, HH>(WH_REP4_ARGS) : launch_rep4<true, false, HH>(WH_REP4_ARGS); \
        return loop ? launch_rep4<false, true, HH>(WH_REP4_ARGS) : launch_rep4<false, false, HH>(WH_REP4_ARGS);
    switch (H) {
        WH_REP4_CASE(8)
        WH_REP4_CASE(16)
        default: return hipErrorInvalidValue;
    }
#undef WH_REP4_CASE
#undef WH_REP4_ARGS
}
