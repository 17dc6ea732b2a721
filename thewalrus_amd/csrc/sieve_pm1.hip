// sieve_pm1.hip -- the Glynn sieve for even N with every repetition equal to one: the terms of
// the plain hafnian (_hafnian.py:443-462) and the even loop hafnian (:546-569) when rpt is all
// ones.  Every digit is then 0/1, every delta is +-1, no row is ever dropped (m = n), and
//     AX_S = M diag(d),   M = Ax X  (the same for all 2^(h-1) terms of a matrix),
// with d_c = delta_(c mod h).  A workgroup keeps M in LDS once; each wave walks terms and
// forms B^(a+1) = (B^a M) diag(d) with a register-tiled product: the wave is an 8 x 8 grid of
// lanes, each owning a T x T tile of the n_pad x n_pad power (n_pad = 8T, zero padded).
//
// Template parameters: T (tile side), REAL (matrix and loop weights real: the same products
// in real arithmetic, which is what complex arithmetic computes when every imaginary part is
// zero), LOOP (add the loop terms of f_loop, _hafnian.py:233-234).
#include "wh_device.h"
#include "wh_launch.h"

namespace {

template <bool REAL> struct Elem;
template <> struct Elem<true> {
    using T = double;
};
template <> struct Elem<false> {
    using T = cplx;
};

__device__ __forceinline__ void emac(double& acc, double a, double b) { acc = fma(a, b, acc); }
__device__ __forceinline__ void emac(cplx& acc, cplx a, cplx b) { cmac(acc, a, b); }
__device__ __forceinline__ double escale(double x, double s) { return x * s; }
__device__ __forceinline__ cplx escale(cplx x, double s) { return cmulr(x, s); }
__device__ __forceinline__ void ezero(double& x) { x = 0.0; }
__device__ __forceinline__ void ezero(cplx& x) { x = cmk(0.0, 0.0); }
__device__ __forceinline__ cplx etoc(double x) { return cmk(x, 0.0); }
__device__ __forceinline__ cplx etoc(cplx x) { return x; }
__device__ __forceinline__ double eload(const cplx* p, int64_t i, double*) { return p[i].re; }
__device__ __forceinline__ cplx eload(const cplx* p, int64_t i, cplx*) { return p[i]; }
__device__ __forceinline__ double eone(double*) { return 1.0; }
__device__ __forceinline__ cplx eone(cplx*) { return cmk(1.0, 0.0); }
__device__ __forceinline__ double ezero_v(double*) { return 0.0; }
__device__ __forceinline__ cplx ezero_v(cplx*) { return cmk(0.0, 0.0); }
__device__ __forceinline__ double eget(cplx z, double*) { return z.re; }
__device__ __forceinline__ cplx eget(cplx z, cplx*) { return z; }
__device__ __forceinline__ double emul(double a, double b) { return a * b; }
__device__ __forceinline__ cplx emul(cplx a, cplx b) { return cmul(a, b); }
__device__ __forceinline__ double eadd(double a, double b) { return a + b; }
__device__ __forceinline__ cplx eadd(cplx a, cplx b) { return cadd(a, b); }
__device__ __forceinline__ double ediv(double a, double d) { return a / d; }
__device__ __forceinline__ cplx ediv(cplx a, double d) { return cdivr(a, d); }

// factor of column c of the current term: delta_(c mod h) = +1 if digit set, else `unset`
// (-1 for the Glynn sieve, 0 for the montrealer's subset inclusion-exclusion)
__device__ __forceinline__ double col_sign(uint64_t t, int c, int h, double unset) {
    int i = c < h ? c : c - h;
    if (i >= h) return 1.0;  // zero padding
    return ((t >> (h - 1 - i)) & 1ull) ? 1.0 : unset;
}


// ---- tile helpers: lane (ti, tj) owns rows I0..I0+T-1, columns J0..J0+T-1 of the power.
// LDS matrices are (8T) x (8T) with row stride 8T + 1 elements: the eight row tiles a
// product step reads then start on distinct LDS banks.
#ifndef WH_PM1_PAD
#define WH_PM1_PAD 1
#endif
#ifndef WH_PM1_KUNROLL
#define WH_PM1_KUNROLL 2
#endif
#ifndef WH_PM1_PIPELINE
#define WH_PM1_PIPELINE 1
#endif
// Reciprocals 1/k (k <= WH_EMAX) for the exponential recurrence of the term coefficient.
__constant__ double kInvJ[WH_EMAX + 1] = {
    0.0,        1.0,        1.0 / 2,  1.0 / 3,  1.0 / 4,  1.0 / 5,  1.0 / 6,  1.0 / 7,  1.0 / 8,
    1.0 / 9,    1.0 / 10,   1.0 / 11, 1.0 / 12, 1.0 / 13, 1.0 / 14, 1.0 / 15, 1.0 / 16, 1.0 / 17,
    1.0 / 18,   1.0 / 19,   1.0 / 20, 1.0 / 21, 1.0 / 22, 1.0 / 23, 1.0 / 24, 1.0 / 25, 1.0 / 26,
    1.0 / 27,   1.0 / 28,   1.0 / 29, 1.0 / 30, 1.0 / 31, 1.0 / 32};

// [eta^h] exp(sum_i a_i eta^i) for h <= H: e_0 = 1, e_k = (1/k) sum_(i=1..k) b_i e_(k-i) with
// b_i = i a_i = p_i / 2 (+ i v_i / 2 with loops); fixed trip counts keep e[] in registers.
template <class E, int H, bool LOOP>
__device__ __forceinline__ E coeff_top_e(const cplx* pt, const cplx* lv, int h) {
    E b[H + 1], e[H + 1];
#pragma unroll
    for (int i = 1; i <= H; ++i) {
        E v = escale(eget(pt[i], (E*)nullptr), 0.5);
        if (LOOP) v = eadd(v, escale(eget(lv[i], (E*)nullptr), 0.5 * i));
        b[i] = i <= h ? v : ezero_v((E*)nullptr);
    }
    e[0] = eone((E*)nullptr);
    E res = e[0];
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        E s0 = ezero_v((E*)nullptr), s1 = ezero_v((E*)nullptr);
#pragma unroll
        for (int i = 1; i <= k; i += 2) emac(s0, b[i], e[k - i]);
#pragma unroll
        for (int i = 2; i <= k; i += 2) emac(s1, b[i], e[k - i]);
        e[k] = escale(eadd(s0, s1), kInvJ[k]);
        if (k == h) res = e[k];
    }
    return res;
}

// The same coefficient with b_i kept in the term's slot (written over p_i) instead of registers:
// about half the registers of coeff_top_e, for the repeated-row kernel's H = 16.
template <class E, int H, bool LOOP>
__device__ __forceinline__ E coeff_top_lds(cplx* pt, const cplx* lv, int h) {
#pragma unroll
    for (int i = 1; i <= H; ++i) {
        E v = escale(eget(pt[i], (E*)nullptr), 0.5);
        if (LOOP) v = eadd(v, escale(eget(lv[i], (E*)nullptr), 0.5 * i));
        pt[i] = etoc(i <= h ? v : ezero_v((E*)nullptr));
    }
    E e[H + 1];
    e[0] = eone((E*)nullptr);
    E res = e[0];
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        E s0 = ezero_v((E*)nullptr), s1 = ezero_v((E*)nullptr);
#pragma unroll
        for (int i = 1; i <= k; i += 2) emac(s0, eget(pt[i], (E*)nullptr), e[k - i]);
#pragma unroll
        for (int i = 2; i <= k; i += 2) emac(s1, eget(pt[i], (E*)nullptr), e[k - i]);
        e[k] = escale(eadd(s0, s1), kInvJ[k]);
        if (k == h) res = e[k];
    }
    return res;
}

template <int T> struct Lds {
    static constexpr int S = 8 * T + WH_PM1_PAD;
};

// Per wave, NB term slots of p_0 .. p_(4T+1) and v_0 .. v_(4T+1) (h <= 4T; a spare last entry):
// the coefficients of up to NB terms are formed together, one term per lane.  NB fits the LDS
// beside the powers (complex T = 5 at 4 waves, T = 6 at 3 waves).
__host__ __device__ constexpr int pm1_ptn(int T) { return 4 * T + 4; }
__host__ __device__ constexpr int pm1_nb(int T, bool real) { return real ? 8 : T == 6 ? 2 : T == 5 ? 7 : 8; }

template <int T, class E>
__device__ __forceinline__ void tile_store(E* Pw, const E (&acc)[T][T], int I0, int J0) {
    wave_lds_sync();  // the other lanes' reads of the previous power are done
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
        for (int c = 0; c < T; ++c) Pw[(I0 + r) * Lds<T>::S + J0 + c] = acc[r][c];
    wave_lds_sync();  // the whole power is stored before any lane reads it
}

// acc = (Pw Ms) diag(sign_J): one step of the power sequence, k summed in order.  The
// operands of step k + 1 are loaded while step k's multiply-adds run (register double
// buffer), so LDS latency is hidden even with one wave per SIMD.
template <int T, class E>
__device__ __forceinline__ void tile_load_k(const E* Pw, const E* Ms, int I0, int J0, int k, E (&av)[T],
                                            E (&bv)[T]) {
    constexpr int S = Lds<T>::S;
#pragma unroll
    for (int r = 0; r < T; ++r) av[r] = Pw[(I0 + r) * S + k];
#pragma unroll
    for (int c = 0; c < T; ++c) bv[c] = Ms[k * S + J0 + c];
}

template <int T, class E>
__device__ __forceinline__ void tile_mac_k(E (&nacc)[T][T], const E (&av)[T], const E (&bv)[T]) {
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
        for (int c = 0; c < T; ++c) emac(nacc[r][c], av[r], bv[c]);
}

template <int T, class E>
__device__ __forceinline__ void tile_product(const E* Pw, const E* Ms, E (&acc)[T][T], int I0, int J0,
                                             int n, const double (&sgnJ)[T]) {
    E nacc[T][T];
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
        for (int c = 0; c < T; ++c) ezero(nacc[r][c]);
#if WH_PM1_PIPELINE
    E a0[T], b0[T], a1[T], b1[T];
    tile_load_k<T>(Pw, Ms, I0, J0, 0, a0, b0);
    int k = 0;
    for (; k + 2 <= n; k += 2) {
        tile_load_k<T>(Pw, Ms, I0, J0, k + 1, a1, b1);
        tile_mac_k<T>(nacc, a0, b0);
        // unconditional prefetch (the last one re-reads row k, unused) keeps the operand
        // registers free of branch merges
        const int kn = k + 2 < n ? k + 2 : k;
        tile_load_k<T>(Pw, Ms, I0, J0, kn, a0, b0);
        tile_mac_k<T>(nacc, a1, b1);
    }
    if (k < n) tile_mac_k<T>(nacc, a0, b0);
    // keep later LDS reads (transposed tiles) from being hoisted into the loop's live range
    asm volatile("" ::: "memory");
#else
#pragma unroll WH_PM1_KUNROLL
    for (int k = 0; k < n; ++k) {
        E av[T], bv[T];
        tile_load_k<T>(Pw, Ms, I0, J0, k, av, bv);
        tile_mac_k<T>(nacc, av, bv);
    }
#endif
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
        for (int c = 0; c < T; ++c) acc[r][c] = escale(nacc[r][c], sgnJ[c]);
}

template <int T, class E>
__device__ __forceinline__ E tile_trace(const E (&acc)[T][T], bool diag) {
    E tr;
    ezero(tr);
    if (diag) {
#pragma unroll
        for (int r = 0; r < T; ++r) tr = eadd(tr, acc[r][r]);
    }
    return tr;
}

// lane part of <acc, X^T> = sum_(i in I, j in J) acc[i][j] X[j][i], X in LDS
template <int T, class E>
__device__ __forceinline__ E tile_tdot(const E* X, const E (&acc)[T][T], int I0, int J0) {
    E s;
    ezero(s);
#pragma unroll
    for (int c = 0; c < T; ++c)
#pragma unroll
        for (int r = 0; r < T; ++r) emac(s, acc[r][c], X[(J0 + c) * Lds<T>::S + I0 + r]);
    return s;
}

// lane part of XD_d B D
template <int T, class E>
__device__ __forceinline__ E tile_bilinear(const E (&acc)[T][T], const E (&xdI)[T], const E (&dJ)[T]) {
    E bl;
    ezero(bl);
#pragma unroll
    for (int r = 0; r < T; ++r) {
        E rowsum;
        ezero(rowsum);
#pragma unroll
        for (int c = 0; c < T; ++c) emac(rowsum, acc[r][c], dJ[c]);
        emac(bl, xdI[r], rowsum);
    }
    return bl;
}

__device__ __forceinline__ double shfl_e(double v, int src) { return __shfl(v, src, WH_WAVE); }
__device__ __forceinline__ cplx shfl_e(cplx v, int src) {
    return cmk(__shfl(v.re, src, WH_WAVE), __shfl(v.im, src, WH_WAVE));
}
__device__ __forceinline__ double group8_e(double v) { return group8_sum(v); }
__device__ __forceinline__ cplx group8_e(cplx v) { return cmk(group8_sum(v.re), group8_sum(v.im)); }
__device__ __forceinline__ double stride8_e(double v) { return stride8_sum(v); }
__device__ __forceinline__ cplx stride8_e(cplx v) { return cmk(stride8_sum(v.re), stride8_sum(v.im)); }

// (B D)[I0 + r]: rows summed over the 8 column tiles of the lane's row group
template <int T, class E>
__device__ __forceinline__ void tile_zvec(const E (&acc)[T][T], const E (&dJ)[T], E (&z)[T]) {
#pragma unroll
    for (int r = 0; r < T; ++r) {
        ezero(z[r]);
#pragma unroll
        for (int c = 0; c < T; ++c) emac(z[r], acc[r][c], dJ[c]);
        z[r] = group8_e(z[r]);
    }
}

// (XD_d B)[J0 + c]: columns summed over the 8 row tiles of the lane's column group
template <int T, class E>
__device__ __forceinline__ void tile_yvec(const E (&acc)[T][T], const E (&xdI)[T], E (&y)[T]) {
#pragma unroll
    for (int c = 0; c < T; ++c) {
        ezero(y[c]);
#pragma unroll
        for (int r = 0; r < T; ++r) emac(y[c], xdI[r], acc[r][c]);
        y[c] = stride8_e(y[c]);
    }
}

template <int T, bool REAL, bool LOOP, bool HALF>
__device__ __forceinline__ void pm1_body(const wh_job_dev& J, const cplx* __restrict__ pool,
                                         double4* __restrict__ partials, int64_t b,
                                         unsigned char* smem) {
    using E = typename Elem<REAL>::T;
    constexpr int NP = 8 * T;  // padded side
    constexpr int S = Lds<T>::S;  // LDS row stride (elements)
    const int nw = blockDim.x / WH_WAVE;
    const int wave = threadIdx.x / WH_WAVE;
    const int lane = threadIdx.x % WH_WAVE;
    const int ti = lane >> 3, tj = lane & 7;
    const int n = 2 * J.E;
    const int h = J.E;
    // montrealer terms (_montrealer.py:37-101): 0/1 column factors, p_h and v_h only
    const bool mtl = (J.flags & WH_F_MTL) != 0;
    const double unset = mtl ? 0.0 : -1.0;

    // ---- LDS carve
    E* Ms = reinterpret_cast<E*>(smem);
    E* Pw = Ms + NP * S + wave * NP * S;
    E* vecs = Ms + (1 + nw) * NP * S;           // XD0[NP], D[NP] (loop)
    E* XD0 = vecs;
    E* Dv = vecs + NP;
    constexpr int PTN = pm1_ptn(T);
    constexpr int NB = pm1_nb(T, REAL);
    cplx* slots = reinterpret_cast<cplx*>(vecs + 2 * NP) + wave * (NB * 2 * PTN);
    double4* wres = reinterpret_cast<double4*>(reinterpret_cast<cplx*>(vecs + 2 * NP) + nw * (NB * 2 * PTN));

    // ---- stage M = Ax X (column c of M is column (c + h) mod n of Ax), zero padded
    const cplx* A = pool + J.a_off;
    for (int e = threadIdx.x; e < NP * NP; e += blockDim.x) {
        int r = e / NP, c = e - r * NP;
        E v;
        ezero(v);
        if (r < n && c < n) {
            int src = c < h ? c + h : c - h;
            v = eload(A, (int64_t)r * n + src, (E*)nullptr);
        }
        Ms[r * S + c] = v;
    }
    if (LOOP) {
        const cplx* Dg = pool + J.d_off;
        for (int e = threadIdx.x; e < NP; e += blockDim.x) {
            E xd, dd;
            ezero(xd);
            ezero(dd);
            if (e < n) {
                if (mtl) {  // the caller stages conj(X zeta) and X zeta
                    xd = eload(pool + J.v_off, e, (E*)nullptr);
                    dd = eload(Dg, e, (E*)nullptr);
                } else {
                    int src = e < h ? e + h : e - h;  // (X D)[e]
                    xd = eload(Dg, src, (E*)nullptr);
                    dd = eload(Dg, e, (E*)nullptr);
                }
            }
            XD0[e] = xd;
            Dv[e] = dd;
        }
    }
    __syncthreads();

    const int64_t t0 = (b - J.chunk_base) * J.chunk_terms;
    int64_t t1 = t0 + J.chunk_terms;
    if (t1 > J.steps) t1 = J.steps;
    const int I0 = ti * T, J0 = tj * T;

    csum acc_sum;
    acc_sum.zero();

    int slot = 0;
    int64_t t_batch = t0 + wave;  // the batch's first term
    for (int64_t t = t0 + wave; t < t1; t += nw) {
        const uint64_t tu = (uint64_t)t;
        cplx* pt = slots + slot * 2 * PTN;  // p[0..h]
        cplx* lv = pt + PTN;                // loop scalars v[1..h]
        double sgnJ[T];
#pragma unroll
        for (int c = 0; c < T; ++c) sgnJ[c] = col_sign(tu, J0 + c, h, unset);
        const double prefac = mtl ? (((__popcll(tu) + 1) & 1) ? -1.0 : 1.0)
                                  : (((h - __popcll(tu)) & 1) ? -1.0 : 1.0);

        // P_1 = M diag(d)
        E acc[T][T];
#pragma unroll
        for (int r = 0; r < T; ++r)
#pragma unroll
            for (int c = 0; c < T; ++c) acc[r][c] = escale(Ms[(I0 + r) * S + J0 + c], sgnJ[c]);

        // loop: per-lane row weights XD_d[I] and column weights D[J], read from LDS where
        // used so they do not occupy registers across the products
        auto load_xd = [&](E (&xdI)[T]) {
#pragma unroll
            for (int r = 0; r < T; ++r) xdI[r] = escale(XD0[I0 + r], col_sign(tu, I0 + r, h, unset));
        };
        auto load_d = [&](E (&dJ)[T]) {
#pragma unroll
            for (int c = 0; c < T; ++c) dJ[c] = Dv[J0 + c];
        };

        if constexpr (!HALF) {
            // the reference's order: B^(a+1) = B^a B for a < h, p_a = tr(B^a)
            for (int a = 1; a <= h; ++a) {
                E tr = tile_trace<T>(acc, ti == tj);
                E bl;
                ezero(bl);
                if (LOOP && a <= h - 1) {
                    E xdI[T], dJ[T];
                    load_xd(xdI);
                    load_d(dJ);
                    bl = tile_bilinear<T>(acc, xdI, dJ);
                }
                cplx trc = wave_csum(etoc(tr));
                cplx blc = LOOP ? wave_csum(etoc(bl)) : cmk(0.0, 0.0);
                if (lane == 0) {
                    pt[a] = trc;
                    if (LOOP && a <= h - 1) lv[a + 1] = blc;
                }
                if (a == h) break;
                tile_store<T>(Pw, acc, I0, J0);
                tile_product<T>(Pw, Ms, acc, I0, J0, n, sgnJ);
            }
        } else {
            // powers up to B^A, A = ceil(h/2); tr(B^(2a)) = <B^a, (B^a)^T> and
            // tr(B^(2a+1)) = <B^(a+1), (B^a)^T>.  Loop scalars v_k = XD B^(k-1) D from
            // y_a = XD B^a (column tiles) and z_a = B^a D (row tiles):
            // v_(2a) = y_a . z_(a-1), v_(2a+1) = y_a . z_a, dotted on the diagonal lanes, where
            // the lane's column and row tiles cover the same indices.
            const int A = (h + 1) / 2;
            E zprev[T];
            if (LOOP) {
#pragma unroll
                for (int r = 0; r < T; ++r) zprev[r] = Dv[I0 + r];  // z_0 = D
            }
            tile_store<T>(Pw, acc, I0, J0);
            for (int a = 1; a <= A; ++a) {
                E qo, qe;
                if (a == 1) {
                    qo = tile_trace<T>(acc, ti == tj);   // tr(B)
                    qe = tile_tdot<T>(Pw, acc, I0, J0);  // <B, B^T>
                } else {
                    tile_product<T>(Pw, Ms, acc, I0, J0, n, sgnJ);  // acc = B^a
                    qo = tile_tdot<T>(Pw, acc, I0, J0);            // Pw holds B^(a-1)
                    tile_store<T>(Pw, acc, I0, J0);
                    qe = tile_tdot<T>(Pw, acc, I0, J0);
                }
                // the power's results, summed over the wave eight at once: p_ko, p_ke, v_2a, v_(2a+1)
                E de, dodd;
                ezero(de);
                ezero(dodd);
                E znew[T];
                if (LOOP) {
                    E y[T], xdI[T], dJ[T];
                    load_xd(xdI);
                    load_d(dJ);
                    tile_yvec<T>(acc, xdI, y);
                    tile_zvec<T>(acc, dJ, znew);
                    if (ti == tj) {
#pragma unroll
                        for (int c = 0; c < T; ++c) {
                            emac(de, y[c], zprev[c]);
                            emac(dodd, y[c], znew[c]);
                        }
                    }
                }
                const cplx qoc = etoc(qo), qec = etoc(qe), dec = etoc(de), doc = etoc(dodd);
                const double v8[8] = {qoc.re, qoc.im, qec.re, qec.im, dec.re, dec.im, doc.re, doc.im};
                const double sum8 = wave_sum8(v8, lane);
                const int ko = a == 1 ? 1 : 2 * a - 1, ke = a == 1 ? 2 : 2 * a;
                if ((lane & 7) == 0) {  // lane 8k holds the sum of v8[k]
                    const int k = lane >> 3;
                    double* dst = nullptr;
                    if (k < 2) dst = &pt[ko].re;
                    else if (k < 4) dst = &pt[ke].re;  // ke <= h + 1 < PTN
                    else if (LOOP && k < 6 && 2 * a <= h) dst = &lv[2 * a].re;
                    else if (LOOP && k >= 6 && 2 * a + 1 <= h) dst = &lv[2 * a + 1].re;
                    if (dst) dst[k & 1] = sum8;
                }
                if (LOOP) {
#pragma unroll
                    for (int r = 0; r < T; ++r) zprev[r] = znew[r];
                }
            }
        }
        if (LOOP) {
            // v_1 = XD_d . D
            E part;
            ezero(part);
            for (int e = lane; e < n; e += WH_WAVE) emac(part, escale(XD0[e], col_sign(tu, e, h, unset)), Dv[e]);
            cplx v1 = wave_csum(etoc(part));
            if (lane == 0) lv[1] = v1;
        }
        wave_lds_sync();  // pt and lv as lane 0 stored them

        if (mtl) {
            // montrealer term: sign (p_h / 2h + v_h / 2), v_h = conj(zeta_S) Sigma_S^(h-1) zeta_S
            if (lane == h) {
                E f = ediv(eget(pt[h], (E*)nullptr), (double)(2 * h));
                if (LOOP) f = eadd(f, ediv(eget(lv[h], (E*)nullptr), 2.0));
                acc_sum.add(cmulr(etoc(f), prefac));
            }
            continue;
        }
        // coefficient of eta^h in exp(sum_i a_i eta^i), a_i = p_i / 2i (+ v_i / 2): the
        // reference builds it factor by factor (_hafnian.py:200-208, :232-241); here lane j runs
        // the power-series exponential e_k = (1/k) sum_(i<=k) (i a_i) e_(k-i) in registers for
        // the j-th term of a batch of up to NB terms
        ++slot;
        if (slot == NB || t + nw >= t1) {
            wave_lds_sync();  // pt and lv of every slot as lane 0 stored them
            if (lane < slot) {
                const cplx* ptj = slots + lane * 2 * PTN;
                const uint64_t tj = (uint64_t)(t_batch + (int64_t)lane * nw);
                const double pj = ((h - __popcll(tj)) & 1) ? -1.0 : 1.0;
                const E top = coeff_top_e<E, 4 * T, LOOP>(ptj, ptj + PTN, h);
                acc_sum.add(cmulr(etoc(top), pj));
            }
            wave_lds_sync();  // the slots are free again
            slot = 0;
            t_batch = t + nw;
        }
    }

    // fold the lanes' partial sums in lane order (montrealer: lane h holds them all), then the
    // waves of this workgroup in wave order
    if (mtl) {
        if (lane == h) wres[wave] = make_double4(acc_sum.sr, acc_sum.cr, acc_sum.si, acc_sum.ci);
    } else {
        double4* lsum = reinterpret_cast<double4*>(slots);
        if (lane < NB) lsum[lane] = make_double4(acc_sum.sr, acc_sum.cr, acc_sum.si, acc_sum.ci);
        wave_lds_sync();
        if (lane == 0) {
            csum s;
            s.zero();
            for (int j = 0; j < NB; ++j) {
                double4 pq = lsum[j];
                s.add_pair(pq.x, pq.y, pq.z, pq.w);
            }
            wres[wave] = make_double4(s.sr, s.cr, s.si, s.ci);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        csum s;
        s.zero();
        for (int w = 0; w < nw; ++w) {
            double4 p = wres[w];
            s.add_pair(p.x, p.y, p.z, p.w);
        }
        partials[b] = make_double4(s.sr, s.cr, s.si, s.ci);
    }
}

// ---- Repeated rows: any edge multiplicities, even N, Glynn or inclusion-exclusion, on the same
// register-tiled products.  Term t has mixed-radix digits k_i (digit 0 most significant, base
// e_i + 1, _hafnian.py:162-180) and delta_i = 2 k_i - e_i (Glynn) or k_i.  The reference keeps
// the rows and columns of Ax X with delta_i != 0 and scales the columns by delta (AX_S,
// :288-312); here every term works on the padded B = M diag(d), M = Ax X, d_c = delta_(c mod E).
// A column with delta = 0 is zero, so under a permutation B is block triangular with AX_S as
// its kept block, and tr(B^k) = tr(AX_S^k); the loop weights XD_d = (X D) diag(d) vanish on the
// same indices, so XD_d B^(k-1) D = XD_S AX_S^(k-1) D_S.  The powers run to B^ceil(h/2) with
// h = N/2 as in the all-ones kernel (direct powers where the reference extends the traces by
// the characteristic polynomial, charpoly.py:321-326), and the term is
// (-1)^(h - sum k) prod C(e_i, k_i) (1/2 for Glynn when delta_0 = 0) [eta^h] exp(sum a_i eta^i)
// (_hafnian.py:444-460, :546-569).  Every job of a launch has 2E <= 8T, h <= H and fewer than
// 2^31 terms (the host checks).
__host__ __device__ constexpr int rep_nb() { return 8; }
__host__ __device__ constexpr int rep_ptn(int H) { return H + 4; }

template <int T, bool REAL, bool LOOP, int H>
__device__ __forceinline__ void rep_body(const wh_job_dev& J, const cplx* __restrict__ pool,
                                         double4* __restrict__ partials, int64_t b, unsigned char* smem) {
    using E = typename Elem<REAL>::T;
    constexpr int NP = 8 * T;
    constexpr int S = Lds<T>::S;
    constexpr int PTN = rep_ptn(H);
    constexpr int NB = rep_nb();
    const int nw = blockDim.x / WH_WAVE;
    const int wave = threadIdx.x / WH_WAVE;
    const int lane = threadIdx.x % WH_WAVE;
    const int ti = lane >> 3, tj = lane & 7;
    const int ne = J.E;
    const int n = 2 * ne;
    const int h = J.N / 2;
    const bool glynn = (J.flags & WH_F_GLYNN) != 0;

    // ---- LDS carve: M, one power per wave, XD0 / D, per-wave term slots, per-wave results,
    // the binomial table C(e_i, k) (row i, k = 0..H)
    E* Ms = reinterpret_cast<E*>(smem);
    E* Pw = Ms + NP * S + wave * NP * S;
    E* vecs = Ms + (1 + nw) * NP * S;
    E* XD0 = vecs;
    E* Dv = vecs + NP;
    cplx* slots = reinterpret_cast<cplx*>(vecs + 2 * NP) + wave * (NB * 2 * PTN);
    double4* wres = reinterpret_cast<double4*>(reinterpret_cast<cplx*>(vecs + 2 * NP) + nw * (NB * 2 * PTN));
    double* btab = reinterpret_cast<double*>(wres + nw);

    const cplx* A = pool + J.a_off;
    for (int e = threadIdx.x; e < NP * NP; e += blockDim.x) {
        int r = e / NP, c = e - r * NP;
        E v;
        ezero(v);
        if (r < n && c < n) {
            int src = c < ne ? c + ne : c - ne;
            v = eload(A, (int64_t)r * n + src, (E*)nullptr);
        }
        Ms[r * S + c] = v;
    }
    if (LOOP) {
        const cplx* Dg = pool + J.d_off;
        for (int e = threadIdx.x; e < NP; e += blockDim.x) {
            E xd, dd;
            ezero(xd);
            ezero(dd);
            if (e < n) {
                int src = e < ne ? e + ne : e - ne;  // (X D)[e]
                xd = eload(Dg, src, (E*)nullptr);
                dd = eload(Dg, e, (E*)nullptr);
            }
            XD0[e] = xd;
            Dv[e] = dd;
        }
    }
    for (int e = threadIdx.x; e < ne * (H + 1); e += blockDim.x) {
        int i = e / (H + 1), k = e - i * (H + 1);
        btab[e] = binom_d(J.e[i], k);
    }
    __syncthreads();

    const int64_t t0 = (b - J.chunk_base) * J.chunk_terms;
    int64_t t1 = t0 + J.chunk_terms;
    if (t1 > J.steps) t1 = J.steps;
    const int I0 = ti * T, J0 = tj * T;
    // lane i < ne owns digit i: its base and the weight of the digits after it
    const int my_e = lane < ne ? J.e[lane] : 0;
    uint32_t my_w = 1;
    for (int l = lane + 1; l < ne; ++l) my_w *= (uint32_t)(J.e[l] + 1);
    // the edge index of column (and row) c, for c < n: c mod ne
    int srcJ[T], srcI[T];
#pragma unroll
    for (int c = 0; c < T; ++c) {
        int col = J0 + c, row = I0 + c;
        srcJ[c] = col < ne ? col : col < n ? col - ne : 0;
        srcI[c] = row < ne ? row : row < n ? row - ne : 0;
    }
    const int src_l = lane < ne ? lane : lane < n ? lane - ne : 0;

    csum acc_sum;
    acc_sum.zero();

    int slot = 0;
    for (int64_t t = t0 + wave; t < t1; t += nw) {
        const uint32_t tu = (uint32_t)t;
        // _hafnian.py:444-459: digits, sign, binomial product, delta
        const int k = lane < ne ? (int)((tu / my_w) % (uint32_t)(my_e + 1)) : 0;
        const int delta = lane < ne ? (glynn ? 2 * k - my_e : k) : 0;
        int ksum = k;
        double bin = lane < ne ? btab[lane * (H + 1) + k] : 1.0;
#pragma unroll
        for (int msk = 1; msk < 8; msk <<= 1) {  // ne <= 8: lanes 0..7 hold every digit
            ksum += __shfl_xor(ksum, msk, 8);
            bin *= __shfl_xor(bin, msk, 8);  // exact: a product of integers below 2^53
        }
        ksum = __shfl(ksum, 0, WH_WAVE);
        bin = __shfl(bin, 0, WH_WAVE);
        const int delta0 = __shfl(delta, 0, WH_WAVE);
        double prefac = (((h - ksum) & 1) ? -1.0 : 1.0) * bin;
        if (glynn && delta0 == 0) prefac *= 0.5;
        double sgnJ[T], sgnI[T];
#pragma unroll
        for (int c = 0; c < T; ++c) {
            const double dj = (double)__shfl(delta, srcJ[c], WH_WAVE);
            const double di = (double)__shfl(delta, srcI[c], WH_WAVE);
            sgnJ[c] = J0 + c < n ? dj : 0.0;
            sgnI[c] = I0 + c < n ? di : 0.0;
        }
        const double dl = (double)__shfl(delta, src_l, WH_WAVE);

        cplx* pt = slots + slot * 2 * PTN;  // pt[0] = (prefactor, 0); p[1..h]
        cplx* lv = pt + PTN;                // loop scalars v[1..h]
        E acc[T][T];
#pragma unroll
        for (int r = 0; r < T; ++r)
#pragma unroll
            for (int c = 0; c < T; ++c) acc[r][c] = escale(Ms[(I0 + r) * S + J0 + c], sgnJ[c]);
        auto load_xd = [&](E (&xdI)[T]) {
#pragma unroll
            for (int r = 0; r < T; ++r) xdI[r] = escale(XD0[I0 + r], sgnI[r]);
        };
        auto load_d = [&](E (&dJ)[T]) {
#pragma unroll
            for (int c = 0; c < T; ++c) dJ[c] = Dv[J0 + c];
        };
        // powers up to B^A, A = ceil(h/2): tr(B^(2a)) = <B^a, (B^a)^T>, tr(B^(2a+1)) =
        // <B^(a+1), (B^a)^T>; loop scalars v_(2a) = y_a . z_(a-1), v_(2a+1) = y_a . z_a with
        // y_a = XD_d B^a and z_a = B^a D (as in the all-ones kernel)
        const int Ah = (h + 1) / 2;
        E zprev[T];
        if (LOOP) {
#pragma unroll
            for (int r = 0; r < T; ++r) zprev[r] = Dv[I0 + r];
        }
        tile_store<T>(Pw, acc, I0, J0);
        for (int a = 1; a <= Ah; ++a) {
            E qo, qe;
            if (a == 1) {
                qo = tile_trace<T>(acc, ti == tj);
                qe = tile_tdot<T>(Pw, acc, I0, J0);
            } else {
                tile_product<T>(Pw, Ms, acc, I0, J0, n, sgnJ);
                qo = tile_tdot<T>(Pw, acc, I0, J0);
                tile_store<T>(Pw, acc, I0, J0);
                qe = tile_tdot<T>(Pw, acc, I0, J0);
            }
            // the power's results, summed over the wave eight at once: p_ko, p_ke, v_2a, v_(2a+1)
            E de, dodd;
            ezero(de);
            ezero(dodd);
            E znew[T];
            if (LOOP) {
                E y[T], xdI[T], dJ[T];
                load_xd(xdI);
                load_d(dJ);
                tile_yvec<T>(acc, xdI, y);
                tile_zvec<T>(acc, dJ, znew);
                if (ti == tj) {
#pragma unroll
                    for (int c = 0; c < T; ++c) {
                        emac(de, y[c], zprev[c]);
                        emac(dodd, y[c], znew[c]);
                    }
                }
            }
            const cplx qoc = etoc(qo), qec = etoc(qe), dec = etoc(de), doc = etoc(dodd);
            const double v8[8] = {qoc.re, qoc.im, qec.re, qec.im, dec.re, dec.im, doc.re, doc.im};
            const double sum8 = wave_sum8(v8, lane);
            const int ko = a == 1 ? 1 : 2 * a - 1, ke = a == 1 ? 2 : 2 * a;
            if ((lane & 7) == 0) {  // lane 8k holds the sum of v8[k]
                const int k = lane >> 3;
                double* dst = nullptr;
                if (k < 2) dst = &pt[ko].re;
                else if (k < 4) dst = &pt[ke].re;  // ke <= h + 1 < PTN
                else if (LOOP && k < 6 && 2 * a <= h) dst = &lv[2 * a].re;
                else if (LOOP && k >= 6 && 2 * a + 1 <= h) dst = &lv[2 * a + 1].re;
                if (dst) dst[k & 1] = sum8;
            }
            if (LOOP) {
#pragma unroll
                for (int r = 0; r < T; ++r) zprev[r] = znew[r];
            }
        }
        if (LOOP) {
            // v_1 = XD_d . D (n <= 64: lane e holds index e)
            E part;
            ezero(part);
            if (lane < n) emac(part, escale(XD0[lane], dl), Dv[lane]);
            cplx v1 = wave_csum(etoc(part));
            if (lane == 0) lv[1] = v1;
        }
        if (lane == 0) pt[0] = cmk(prefac, 0.0);
        wave_lds_sync();  // pt and lv as lane 0 stored them

        // the coefficients of up to NB terms together, lane j for the batch's j-th term
        ++slot;
        if (slot == NB || t + nw >= t1) {
            wave_lds_sync();
            if (lane < slot) {
                cplx* ptj = slots + lane * 2 * PTN;
                const E top = coeff_top_lds<E, H, LOOP>(ptj, ptj + PTN, h);
                acc_sum.add(cmulr(etoc(top), ptj[0].re));
            }
            wave_lds_sync();  // the slots are free again
            slot = 0;
        }
    }

    double4* lsum = reinterpret_cast<double4*>(slots);
    if (lane < NB) lsum[lane] = make_double4(acc_sum.sr, acc_sum.cr, acc_sum.si, acc_sum.ci);
    wave_lds_sync();
    if (lane == 0) {
        csum s;
        s.zero();
        for (int j = 0; j < NB; ++j) {
            double4 pq = lsum[j];
            s.add_pair(pq.x, pq.y, pq.z, pq.w);
        }
        wres[wave] = make_double4(s.sr, s.cr, s.si, s.ci);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        csum s;
        s.zero();
        for (int w = 0; w < nw; ++w) {
            double4 p = wres[w];
            s.add_pair(p.x, p.y, p.z, p.w);
        }
        partials[b] = make_double4(s.sr, s.cr, s.si, s.ci);
    }
}

}  // namespace

template <int T, bool REAL, bool LOOP, bool HALF>
__global__ void __launch_bounds__(256)
wh_sieve_pm1(const wh_job_dev* __restrict__ jobs, int njobs, const cplx* __restrict__ pool,
             double4* __restrict__ partials, int64_t block_offset) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    const int64_t b = blockIdx.x + block_offset;
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].chunk_base <= b) lo = mid; else hi = mid - 1;
    }
    pm1_body<T, REAL, LOOP, HALF>(jobs[lo], pool, partials, b, wh_smem);
}

size_t wh_pm1_lds_bytes(int T, bool real, int nw) {
    size_t esz = real ? sizeof(double) : sizeof(cplx);
    size_t NP = 8 * (size_t)T, S = NP + WH_PM1_PAD;
    size_t mat = (NP * S * esz + 31) / 32 * 32;  // keeps the later regions 32-byte aligned
    return (1 + nw) * mat + 2 * NP * esz + nw * (size_t)(pm1_nb(T, real) * 2 * pm1_ptn(T)) * sizeof(cplx) +
           nw * sizeof(double4) + 32;
}

template <int T, bool REAL, bool LOOP, bool HALF>
static hipError_t launch_t(const wh_job_dev* jobs, int njobs, const void* pool, void* partials,
                           int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream) {
    size_t lds = wh_pm1_lds_bytes(T, REAL, nw);
    static wh_lds_limit lim;
    hipError_t err = wh_raise_lds_limit((const void*)wh_sieve_pm1<T, REAL, LOOP, HALF>, lds, lim);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((wh_sieve_pm1<T, REAL, LOOP, HALF>), dim3((unsigned)nblocks), dim3(nw * WH_WAVE), lds,
                       stream, jobs, njobs, (const cplx*)pool, (double4*)partials, block_offset);
    return hipGetLastError();
}

template <int T, bool HALF>
static hipError_t launch_rl(bool real, bool loop, const wh_job_dev* jobs, int njobs, const void* pool,
                            void* partials, int64_t nblocks, int64_t off, int nw, hipStream_t s) {
    if (real) {
        if (loop) return launch_t<T, true, true, HALF>(jobs, njobs, pool, partials, nblocks, off, nw, s);
        return launch_t<T, true, false, HALF>(jobs, njobs, pool, partials, nblocks, off, nw, s);
    }
    if (loop) return launch_t<T, false, true, HALF>(jobs, njobs, pool, partials, nblocks, off, nw, s);
    return launch_t<T, false, false, HALF>(jobs, njobs, pool, partials, nblocks, off, nw, s);
}

template <int T>
static hipError_t launch_h(bool half, bool real, bool loop, const wh_job_dev* jobs, int njobs,
                           const void* pool, void* partials, int64_t nblocks, int64_t off, int nw,
                           hipStream_t s) {
    if (half) return launch_rl<T, true>(real, loop, jobs, njobs, pool, partials, nblocks, off, nw, s);
    return launch_rl<T, false>(real, loop, jobs, njobs, pool, partials, nblocks, off, nw, s);
}

hipError_t wh_launch_pm1(int T, bool half, bool real, bool loop, const wh_job_dev* jobs, int njobs,
                         const void* pool, void* partials, int64_t nblocks, int64_t block_offset,
                         int nw, hipStream_t stream) {
    switch (T) {
        case 1: return launch_h<1>(half, real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
        case 2: return launch_h<2>(half, real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
        case 3: return launch_h<3>(half, real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
        case 4: return launch_h<4>(half, real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
        case 5: return launch_h<5>(half, real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
        case 6: return launch_h<6>(half, real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
        default: return hipErrorInvalidValue;
    }
}


// Four waves per SIMD: the complex H = 16 instances then keep part of the coefficient state in
// scratch (about 190 bytes per lane) instead of running two or three waves per SIMD.
#ifndef WH_REP_WAVES_PER_EU
#define WH_REP_WAVES_PER_EU 4
#endif
template <int T, bool REAL, bool LOOP, int H>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WH_REP_WAVES_PER_EU)))
wh_sieve_rep(const wh_job_dev* __restrict__ jobs, int njobs, const cplx* __restrict__ pool,
             double4* __restrict__ partials, int64_t block_offset) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    const int64_t b = blockIdx.x + block_offset;
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].chunk_base <= b) lo = mid; else hi = mid - 1;
    }
    rep_body<T, REAL, LOOP, H>(jobs[lo], pool, partials, b, wh_smem);
}

// Tile side 3 of the repeated-row class is the four-terms-per-wave kernel (sieve_rep4.hip, 2E <= 12).
size_t wh_rep_lds_bytes(int T, bool real, bool loop, int nw, int H) {
    if (T == 3) return wh_rep4_lds_bytes(real, loop, nw, H);
    size_t esz = real ? sizeof(double) : sizeof(cplx);
    size_t NP = 8 * (size_t)T, S = NP + WH_PM1_PAD;
    return (1 + nw) * NP * S * esz + 2 * NP * esz + nw * (size_t)(rep_nb() * 2 * rep_ptn(H)) * sizeof(cplx) +
           nw * sizeof(double4) + (size_t)NP / 2 * (H + 1) * sizeof(double) + 32;
}

template <int T, bool REAL, bool LOOP, int H>
static hipError_t launch_rep_t(const wh_job_dev* jobs, int njobs, const void* pool, void* partials,
                               int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream) {
    size_t lds = wh_rep_lds_bytes(T, REAL, LOOP, nw, H);
    static wh_lds_limit lim;
    hipError_t err = wh_raise_lds_limit((const void*)wh_sieve_rep<T, REAL, LOOP, H>, lds, lim);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((wh_sieve_rep<T, REAL, LOOP, H>), dim3((unsigned)nblocks), dim3(nw * WH_WAVE), lds,
                       stream, jobs, njobs, (const cplx*)pool, (double4*)partials, block_offset);
    return hipGetLastError();
}

template <int T, int H>
static hipError_t launch_rep_rl(bool real, bool loop, const wh_job_dev* jobs, int njobs, const void* pool,
                                void* partials, int64_t nblocks, int64_t off, int nw, hipStream_t s) {
    if (real) {
        if (loop) return launch_rep_t<T, true, true, H>(jobs, njobs, pool, partials, nblocks, off, nw, s);
        return launch_rep_t<T, true, false, H>(jobs, njobs, pool, partials, nblocks, off, nw, s);
    }
    if (loop) return launch_rep_t<T, false, true, H>(jobs, njobs, pool, partials, nblocks, off, nw, s);
    return launch_rep_t<T, false, false, H>(jobs, njobs, pool, partials, nblocks, off, nw, s);
}

hipError_t wh_launch_rep(int T, int H, bool real, bool loop, const wh_job_dev* jobs, int njobs, const void* pool,
                         void* partials, int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream) {
    if (T == 1 && H == 8) return launch_rep_rl<1, 8>(real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
    if (T == 1 && H == 16) return launch_rep_rl<1, 16>(real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
    if (T == 2 && H == 8) return launch_rep_rl<2, 8>(real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
    if (T == 2 && H == 16) return launch_rep_rl<2, 16>(real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
    if (T == 3) return wh_launch_rep4(H, real, loop, jobs, njobs, pool, partials, nblocks, block_offset, nw, stream);
    return hipErrorInvalidValue;
}
