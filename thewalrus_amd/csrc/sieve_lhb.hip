// sieve_lhb.hip -- batched loop hafnian: one sieve over the fixed modes' edges and the batched
// mode's edge gives the loop hafnian for every photon number 0..N_cutoff of the batched mode
// at once (the core of Gaussian boson sampling's chain rule).  Restates
// _calc_loop_hafnian_batch_even (thewalrus/loop_hafnian_batch.py:52-123) and
// _calc_loop_hafnian_batch_odd (:128-208) per term, and with nD diagonals sharing the matrix
// _calc_loop_hafnian_batch_gamma_even / _odd (loop_hafnian_batch_gamma.py:53-129, :132-219).
//
// A wave takes a term's power traces p_k from symmetric powers on the matrix cores (sieve_sym.hip's
// formulation, sym_device.h), up to A = ceil(n_max / 4), and the odd scalars from w_a = B^a V =
// W_a (X V), V the batched mode's row (and the odd mode's row, V0, for the odd variant's terms with
// k0 = k1 = 0, _hafnian.py:360-380):
//     XD_d B^(a+b) D = sum_e delta_e z_a[s e] z_b[e],   oddVX B^(a+b) D = sum_e delta_e w_a[s e] z_b[e].
// Then the coefficient series f_loop(n_max), f_loop_odd(n_max) and f_loop_odd(n_fixed) run side by
// side, one order per lane (right-looking exponential recurrence), and lane q adds output q's term.
//
// Precision: with tens of photons the signed terms cancel by 10^5 to 10^7, and it is the loop
// scalars of the wide terms (delta up to the batch's 6 and more, weights of order 1) and the series'
// own cancellation that reach the result: with either in plain double the sampler's step of 16
// modes, 22 + 12 photons loses to 2e-9 on some inputs (5e-12 typical).  So z_a = A (G z_(a-1)),
// their dots and the series run in two-word arithmetic (error-free products and sums, a low word
// beside each value): 3e-10 at worst and 1.5e-12 typical over the same inputs, where the
// double-only general kernel this one replaced had 5e-10 and 5e-12; the traces, whose rounding
// weighs 20 times less, stay in double.
//
// FULL: a matrix that is not symmetric (sym_device.h; V stands on the left of the odd scalars, so an
// asymmetry counts in the first order) takes its traces from the full powers and every loop scalar from
// the chain z_a, in two words too.
//
// Split: a workgroup takes one chunk of terms for one diagonal, one term per wave at a time; chunks
// of one term per wave up to 1024 workgroups.  A term's powers are repeated per diagonal, at every
// chunk count: against the one-wave LDS kernel, which shared them from 1024 chunks on, ten diagonals
// of 19, 22 and 26 clicks took 1.06 -> 0.36, 1.93 -> 0.69 and 15.5 -> 4.2 ms, nine of 28 photons with 12
// more 15.9 -> 2.9 ms.  What bounds it is the serial chain of a term (ceil(n_max / 4) products, then
// n_max recurrence steps) at 2 waves per SIMD: in a sampler's step of 16 modes the matrix cores are busy 8%
// and the other vector instructions 49% of 97 us.  The two-word vectors do not all fit the registers: 16,
// 57 and 144 values are spilled on tile sides 2, 3 and 6 (none on the others).
#include <algorithm>

#include "sym_device.h"
#include "wh_launch.h"

namespace {

// ---- two-word arithmetic (sym_device.h: acc2)
// (s, c) += (ah + al)(bh + bl)
__device__ __forceinline__ void mac22(double& s, double& c, double ah, double al, double bh, double bl) {
#pragma clang fp contract(off)
    const double p = ah * bh;
    acc2(s, c, p, fma(al, bh, fma(ah, bl, fma(ah, bh, -p))));
}
__device__ __forceinline__ void norm2(double& s, double& c) {
#pragma clang fp contract(off)
    const double t = s + c, bb = t - s;
    c = (s - (t - bb)) + (c - bb);
    s = t;
}
struct cplx2 {
    cplx h, l;
};
__device__ __forceinline__ void cnorm2(cplx2& a) {
    norm2(a.h.re, a.l.re);
    norm2(a.h.im, a.l.im);
}
__device__ __forceinline__ void cmac2(cplx2& s, cplx a, cplx2 b) {  // s += a b
    mac2(s.h.re, s.l.re, a.re, b.h.re, b.l.re);
    mac2(s.h.re, s.l.re, -a.im, b.h.im, b.l.im);
    mac2(s.h.im, s.l.im, a.re, b.h.im, b.l.im);
    mac2(s.h.im, s.l.im, a.im, b.h.re, b.l.re);
}
__device__ __forceinline__ void cmac22(cplx2& s, cplx2 a, cplx2 b) {
    mac22(s.h.re, s.l.re, a.h.re, a.l.re, b.h.re, b.l.re);
    mac22(s.h.re, s.l.re, -a.h.im, -a.l.im, b.h.im, b.l.im);
    mac22(s.h.im, s.l.im, a.h.re, a.l.re, b.h.im, b.l.im);
    mac22(s.h.im, s.l.im, a.h.im, a.l.im, b.h.re, b.l.re);
}
__device__ __forceinline__ cplx2 czero2() {
    cplx2 z;
    z.h = z.l = cmk(0.0, 0.0);
    return z;
}
__device__ __forceinline__ cplx2 cscale2(cplx2 a, double d) {  // d (a.h + a.l)
    cplx2 r = czero2();
    mac2(r.h.re, r.l.re, d, a.h.re, a.l.re);
    mac2(r.h.im, r.l.im, d, a.h.im, a.l.im);
    return r;
}
template <int CTRL>
__device__ __forceinline__ void dpp_add2(cplx2& s) {
    const double r = dpp_d<CTRL>(s.h.re), rc = dpp_d<CTRL>(s.l.re), i = dpp_d<CTRL>(s.h.im), ic = dpp_d<CTRL>(s.l.im);
    acc2(s.h.re, s.l.re, r, rc);
    acc2(s.h.im, s.l.im, i, ic);
}
__device__ __forceinline__ cplx2 shfl2(cplx2 s, int src) {
    cplx2 r;
    r.h = cmk(__shfl(s.h.re, src, WH_WAVE), __shfl(s.h.im, src, WH_WAVE));
    r.l = cmk(__shfl(s.l.re, src, WH_WAVE), __shfl(s.l.im, src, WH_WAVE));
    return r;
}
// Orders of one coefficient series, as offsets into the wave's LDS: b_1.. in two words (index 0
// unused) and e_0.. rounded.  (Offsets, not pointers: a lane picks its series, and a selected
// pointer would be accessed as flat memory.)
struct SeriesLds {
    int bh, bl, e;
};

__host__ __device__ constexpr size_t lhb_wave_cplx(int T, int nmax, int nf) {
    const size_t NP = 8 * (size_t)T, S = NP + 2, PN = (size_t)nmax / 2 + 4, A = ((size_t)nmax / 2 + 1) / 2;
    // W | z_0 .. z_A in two words | G z | w, w0 of two powers | p, v (two words), o, o0 | the three
    // series (b in two words, e) | delta; at least the wave's 128 output sums at the end
    const size_t all = NP * S + 2 * (A + 1) * NP + 2 * NP + 4 * NP + 5 * PN +
                       3 * ((size_t)nmax + 1 + nmax / 2 + 1 + nf + 1) + NP / 2;
    return all < 256 ? 256 : all;
}

// exp series of the lane's task by the right-looking recurrence: the task's orders 1..len live on
// lanes base .. base + len - 1, s = sum_(i < k) b_(m-i) e_i in two words; steps run to the longest
// task.  e_k itself is passed on rounded (its rounding weighs 10 times less than the sum's).
__device__ __forceinline__ void series_lanes(cplx* w, const SeriesLds& t, int base, int len, int maxlen, int lane) {
    const int m = lane - base + 1;
    const bool on = m >= 1 && m <= len;
    cplx2 s = czero2();
    if (on) {
        s.h = w[t.bh + m];
        s.l = w[t.bl + m];
    }
#pragma unroll 1
    for (int k = 1; k < maxlen; ++k) {
        const cplx ek = cmulr(cadd(s.h, s.l), kInv.v[k]);
        const int src = (base + k - 1) & 63;
        const cplx e = cmk(__shfl(ek.re, src, WH_WAVE), __shfl(ek.im, src, WH_WAVE));
        if (on && m > k) {
            cplx2 b;
            b.h = w[t.bh + m - k];
            b.l = w[t.bl + m - k];
            cmac2(s, e, b);
        }
    }
    if (on) w[t.e + m] = cmulr(cadd(s.h, s.l), kInv.v[m]);
}

// the same by rows for series of more than 64 orders: e_k = (1 / k) sum_i b_i e_(k-i), the lanes
// sharing the sum
__device__ __forceinline__ void series_rows(cplx* w, const SeriesLds& t, int len, int lane) {
#pragma unroll 1
    for (int k = 1; k <= len; ++k) {
        cplx2 s = czero2();
        for (int i = lane + 1; i <= k; i += WH_WAVE) {
            cplx2 b;
            b.h = w[t.bh + i];
            b.l = w[t.bl + i];
            cmac2(s, w[t.e + k - i], b);
        }
        for (int x = 1; x < WH_WAVE; x <<= 1) {
            const cplx2 o = shfl2(s, lane ^ x);
            acc2(s.h.re, s.l.re, o.h.re, o.l.re);
            acc2(s.h.im, s.l.im, o.h.im, o.l.im);
        }
        if (lane == 0) w[t.e + k] = cmulr(cadd(s.h, s.l), kInv.v[k]);
        wave_lds_sync();
    }
}

}  // namespace

// partials[J.part_off + chunk * nD * L + kd * L + q] = (sum_re, err_re, sum_im, err_im) of
// output q of diagonal kd.  Block chunk_base + chunk * nD + kd takes the chunk's terms for
// diagonal kd.
template <int T, bool FULL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(T <= 3 ? 2 : 1)))
wh_sieve_lhb(const wh_lhb_job* __restrict__ job, const cplx* __restrict__ pool,
             double4* __restrict__ partials, int max_n, int max_nf) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    constexpr int NP = GeoG<T>::NP;
    constexpr int S = GeoG<T>::S;
    constexpr int NG = GeoG<T>::NG;
    const int64_t b = blockIdx.x;
    const wh_lhb_job& J = *job;
    const int nw = blockDim.x / WH_WAVE;
    const int wave = threadIdx.x / WH_WAVE;
    const int lane = threadIdx.x % WH_WAVE;
    LaneMapG L;
    L.x = lane & 3;
    L.br = (lane >> 2) & 1;
    L.bc = (lane >> 3) & 1;
    L.y = lane >> 4;
    const int E = J.E, n = 2 * E, nL = J.L;
    const int nf = J.n_fixed, nmax = J.n_max;
    const bool oddv = (J.flags & WH_LHB_ODD) != 0;
    const bool glynn = (J.flags & WH_LHB_GLYNN) != 0;
    const int he = nmax / 2;  // f_loop(n_max) order
    const int Ahalf = (he + 1) / 2;
    const int64_t chunk = (b - J.chunk_base) / J.nD;
    const int kd = (int)((b - J.chunk_base) % J.nD);
    const int64_t t0 = chunk * J.chunk_terms;
    int64_t t1 = t0 + J.chunk_terms;
    if (t1 > J.steps) t1 = J.steps;

    // ---- LDS carve (wh_lhb_lds_bytes)
    const size_t wsz = lhb_wave_cplx(T, max_n, max_nf);
    const size_t PN = (size_t)max_n / 2 + 4;
    cplx* XA = reinterpret_cast<cplx*>(wh_smem);
    cplx* Dv = XA + NP * S;
    cplx* Wv = Dv + NP + wave * wsz;
    const int ZA = (max_n / 2 + 1) / 2 + 1;  // rows z_0 .. z_A
    cplx* zh = Wv + NP * S;
    cplx* zl = zh + ZA * NP;
    cplx* th = zl + ZA * NP;  // G z_(a-1)
    cplx* tl = th + NP;
    cplx* Wb = tl + NP;       // w of two powers, then w0
    cplx* pt = Wb + 4 * NP;
    cplx* lv = pt + PN;
    cplx* lvl = lv + PN;
    cplx* ov = lvl + PN;
    cplx* ov0 = ov + PN;
    SeriesLds fo, fe, f0;
    fo.bh = (int)(ov0 - Wv + PN);
    fo.bl = fo.bh + max_n + 1;
    fo.e = fo.bl + max_n + 1;
    fe.bh = fo.e + max_n + 1;
    fe.bl = fe.bh + max_n / 2 + 1;
    fe.e = fe.bl + max_n / 2 + 1;
    f0.bh = fe.e + max_n / 2 + 1;
    f0.bl = f0.bh + max_nf + 1;
    f0.e = f0.bl + max_nf + 1;
    double* dl = reinterpret_cast<double*>(Wv + f0.e + max_nf + 1);
    double* btab = reinterpret_cast<double*>(Dv + NP + nw * wsz);

    // ---- stage X A (row r holds row swap(r) of A), zero padded, and the diagonal
    const cplx* A = pool + J.a_off;
    for (int e = threadIdx.x; e < NP * NP; e += blockDim.x) {
        const int r = e / NP, c = e - r * NP;
        cplx v = cmk(0.0, 0.0);
        if (r < n && c < n) v = A[(int64_t)swp(r, E) * n + c];
        XA[r * S + c] = v;
    }
    for (int e = threadIdx.x; e < NP; e += blockDim.x)
        Dv[e] = e < n ? pool[J.d_off + (int64_t)kd * n + e] : cmk(0.0, 0.0);
    const int my_e = lane < E ? J.e[lane] : 0;
    int64_t my_w = 1;  // product of (e_l + 1) over l > lane
    int my_row = 0;
    for (int l = 0; l < E; ++l) {
        const int el = __builtin_amdgcn_readlane(my_e, l);
        if (l > lane) my_w *= (int64_t)(el + 1);
        if (l < lane && l >= 1) my_row += el + 1;
    }
    if (wave == 0 && lane >= 1 && lane < E)  // edges 1.. (the batched edge has its own factor)
        for (int k = 0; k <= my_e; ++k) btab[my_row + k] = binom_t(my_e, k);
    __syncthreads();

    const Bop<T> B[1] = {};  // X A stays in LDS: the registers go to the two-word vectors
    cplx xo[T];  // X V at the lane's columns (V = row 0 of A = row E of X A)
#pragma unroll
    for (int q = 0; q < T; ++q) xo[q] = XA[E * S + swp(L.cd(q), E)];
    // z rows: PARTS lanes share a row
    constexpr int PARTS = T == 1 ? 8 : T == 2 ? 4 : T <= 4 ? 2 : 1;
    const int zrow = lane / PARTS, zpart = lane % PARTS;
    const int nk = (n + 3) / 4;
    const bool wide = nmax > WH_WAVE;
    const bool small = J.steps < ((int64_t)1 << 31);
    const int es = lane < n ? swp(lane, E) : 0, ee = lane < n ? lane : 0;
    const cplx D0 = Dv[0], D1 = Dv[1];

    csum acc0, acc1;  // outputs lane and lane + 64
    acc0.zero();
    acc1.zero();

    for (int64_t t = t0 + wave; t < t1; t += nw) {
        // loop_hafnian_batch.py:86-97: digits, binomial product over edges 1.., delta
        int k = 0;
        if (lane < E) {
            if (small) k = (int)(((uint32_t)t / (uint32_t)my_w) % (uint32_t)(my_e + 1));
            else k = (int)((t / my_w) % (int64_t)(my_e + 1));
        }
        const int delta = glynn ? 2 * k - my_e : k;
        wave_lds_sync();
        if (lane < NP) dl[lane] = 0.0;
        wave_lds_sync();
        if (lane < E) dl[lane] = dl[lane + E] = (double)delta;
        double bin = lane >= 1 && lane < E ? btab[my_row + k] : 1.0;
        // exact: products of small integers (E <= 24: lanes 0..31)
        bin *= dpp_d<WH_DPP_XOR1>(bin);
        bin *= dpp_d<WH_DPP_XOR2>(bin);
        bin *= dpp_d<WH_DPP_HALF_MIRROR>(bin);
        bin *= dpp_d<WH_DPP_MIRROR>(bin);
        bin *= __shfl_xor(bin, 16, WH_WAVE);
        bin = __shfl(bin, 0, WH_WAVE);
        const int par = __popcll(__ballot(k & 1)) & 1;  // parity of sum k
        const int k0 = __shfl(k, 0, WH_WAVE);
        const int k1 = __shfl(k, 1, WH_WAVE);
        const bool odd0 = oddv && k0 == 0 && k1 == 0;
        wave_lds_sync();
        double dr[T], dc[T];
#pragma unroll
        for (int p = 0; p < T; ++p) {
            dr[p] = dl[L.rd(p)];
            dc[p] = dl[L.cd(p)];
        }
        const double de = lane < n ? dl[lane] : 0.0;

        // C_1 = A; W_1 = A Delta; z_0 = D, w_0 = V, w0_0 = V0
        double cR[NG], cI[NG];
        {
            int g = 0;
#pragma unroll
            for (int p = 0; p < T; ++p)
#pragma unroll
                for (int q = p; q < T; ++q, ++g) {
                    const cplx m = XA[swp(L.rd(p), E) * S + L.cd(q)];
                    cR[g] = m.re;
                    cI[g] = m.im;
                }
        }
        cplx to = cmk(0.0, 0.0);
        if (lane < n) to = cmulr(XA[es * S + es], de);
        if constexpr (!FULL) sym_store<T>(Wv, cR, cI, dr, dc, L);
        if (lane < NP) {
            Wb[lane] = XA[E * S + lane];
            if (odd0) Wb[2 * NP + lane] = XA[(E + 1) * S + lane];
            cplx2 z;
            z.h = Dv[lane];
            z.l = cmk(0.0, 0.0);
            zh[lane] = z.h;
            zl[lane] = z.l;
            z = FULL && de == 0.0 ? czero2() : cscale2(z, de);
            const int at = swp(lane, E);  // (G z)[s e] = delta_e z[e]
            th[at] = z.h;
            tl[at] = z.l;
        }
        wave_lds_sync();
        // z_a = A (G z_(a-1)), a = 1..A, in two words; with more than 64 photons on to a = h, the odd
        // scalars oddVX B^(a-1) D = V . G z_(a-1) from it too (there their rounding outweighs the
        // traces').  FULL: every scalar, v_a = D . G z_(a-1) among them, over the edges with delta != 0
#pragma unroll 1
        for (int a = 1; a <= (wide || FULL ? he : Ahalf); ++a) {
            if (wide || FULL) {
                cplx2 t = czero2(), o = czero2(), o0 = czero2(), v = czero2();
                if (lane < n && !(FULL && dl[lane] == 0.0)) {
                    t.h = th[lane];
                    t.l = tl[lane];
                    if constexpr (FULL) cmac2(v, Dv[lane], t);
                    cmac2(o, XA[E * S + lane], t);
                    if (odd0) cmac2(o0, XA[(E + 1) * S + lane], t);
                }
#pragma unroll 1
                for (int x = 1; x < WH_WAVE; x <<= 1) {
                    t = shfl2(o, lane ^ x);
                    acc2(o.h.re, o.l.re, t.h.re, t.l.re);
                    acc2(o.h.im, o.l.im, t.h.im, t.l.im);
                    t = shfl2(o0, lane ^ x);
                    acc2(o0.h.re, o0.l.re, t.h.re, t.l.re);
                    acc2(o0.h.im, o0.l.im, t.h.im, t.l.im);
                    if constexpr (FULL) {
                        t = shfl2(v, lane ^ x);
                        acc2(v.h.re, v.l.re, t.h.re, t.l.re);
                        acc2(v.h.im, v.l.im, t.h.im, t.l.im);
                    }
                }
                if constexpr (FULL) cnorm2(v);
                if (lane == 0) {
                    ov[a] = cadd(o.h, o.l);
                    ov0[a] = cadd(o0.h, o0.l);
                    if constexpr (FULL) {
                        lv[a] = v.h;
                        lvl[a] = v.l;
                    }
                }
            }
            cplx2 s = czero2();
            if (zrow < NP) {
                const cplx* Ar = XA + swp(zrow, E) * S;
#pragma unroll 2
                for (int j = zpart; j < n; j += PARTS) {
                    if (FULL && dl[j] == 0.0) continue;
                    cplx2 t;
                    t.h = th[j];
                    t.l = tl[j];
                    cmac2(s, Ar[j], t);
                }
            }
            if constexpr (PARTS >= 2) dpp_add2<WH_DPP_XOR1>(s);
            if constexpr (PARTS >= 4) dpp_add2<WH_DPP_XOR2>(s);
            if constexpr (PARTS >= 8) dpp_add2<WH_DPP_HALF_MIRROR>(s);
            cnorm2(s);
            wave_lds_sync();
            if (zpart == 0 && zrow < NP) {
                if (!FULL && a <= Ahalf) {
                    zh[a * NP + zrow] = s.h;
                    zl[a * NP + zrow] = s.l;
                }
                s = FULL && dl[zrow] == 0.0 ? czero2() : cscale2(s, dl[zrow]);
                const int at = swp(zrow, E);
                th[at] = s.h;
                tl[at] = s.l;
            }
            wave_lds_sync();
        }
        // v_k = sum_e delta_e z_a[s e] z_b[e], a = (k - 1) / 2, b = k / 2: lanes k and k + 32 take
        // every other edge
#pragma unroll 1
        for (int kb = 0; kb < he && !FULL; kb += 32) {
            const int kk = kb + (lane & 31) + 1;
            cplx2 s = czero2();
            if (kk <= he) {
                const cplx *ah = zh + (kk - 1) / 2 * NP, *al = zl + (kk - 1) / 2 * NP;
                const cplx *bh = zh + kk / 2 * NP, *bl = zl + kk / 2 * NP;
#pragma unroll 1
                for (int e = lane >> 5; e < E; e += 2) {
                    cplx2 x = czero2(), a0, a1, b0, b1;
                    a0.h = ah[e]; a0.l = al[e]; a1.h = ah[e + E]; a1.l = al[e + E];
                    b0.h = bh[e]; b0.l = bl[e]; b1.h = bh[e + E]; b1.l = bl[e + E];
                    cmac22(x, a1, b0);
                    cmac22(x, a0, b1);
                    const double d = dl[e];
                    mac2(s.h.re, s.l.re, d, x.h.re, x.l.re);
                    mac2(s.h.im, s.l.im, d, x.h.im, x.l.im);
                }
            }
            const cplx2 o = shfl2(s, lane ^ 32);
            acc2(s.h.re, s.l.re, o.h.re, o.l.re);
            acc2(s.h.im, s.l.im, o.h.im, o.l.im);
            cnorm2(s);
            if (lane < 32 && kk <= he) {
                lv[kk] = s.h;
                lvl[kk] = s.l;
            }
        }
        wave_lds_sync();
        if constexpr (FULL)
            full_scalars<0>([&](int i, int j) { return XA[swp(i, E) * S + j]; }, 0, 0, E, he, dl, Wv, S, nullptr, pt,
                            {nullptr}, lane);
#pragma unroll 1
        for (int a = 1; a <= Ahalf && !FULL; ++a) {
            if (a > 1) {
                sym_product<T, false>(Wv, XA, B, cR, cI, L, nk);
                to = sym_trace<T>(Wv, cR, cI, dr, L, E);  // C_a with W_(a-1): p_(2a-1)
                wave_lds_sync();
                sym_store<T>(Wv, cR, cI, dr, dc, L);
                wave_lds_sync();
            }
            const cplx te = sym_trace<T>(Wv, cR, cI, dr, L, E);  // p_(2a)
            cplx* wp = Wb + ((a - 1) & 1) * NP;
            cplx* wc = Wb + (a & 1) * NP;
            if (a < Ahalf && !wide) {
                sym_matvec<T>(Wv, xo, wc, L);
                if (odd0) {
                    cplx x0[T];
#pragma unroll
                    for (int q = 0; q < T; ++q) x0[q] = XA[(E + 1) * S + swp(L.cd(q), E)];
                    sym_matvec<T>(Wv, x0, wc + 2 * NP, L);
                }
            }
            // orders 2a - 1 (the previous vectors) and 2a
            const cplx zpe = cmulr(zh[(a - 1) * NP + ee], de), zce = cmulr(zh[a * NP + ee], de);
            const cplx os = wp[es];
            const cplx o0 = cmul(zpe, os), o1 = cmul(zce, os);
            const double va[8] = {to.re, to.im, te.re, te.im, o0.re, o0.im, o1.re, o1.im};
            const double sa = wave_sum8(va, lane);  // lane 8k: value k
            const int kv = lane >> 3, at = 2 * a - 1 + ((kv >> 1) & 1);
            if ((lane & 7) == 0 && (kv < 4 || !wide)) {
                cplx* d1 = (kv < 4 ? pt : ov) + at;
                (kv & 1 ? d1->im : d1->re) = sa;
            }
            if (odd0 && !wide) {
                const cplx os0 = wp[2 * NP + es];
                const cplx q0 = cmul(zpe, os0), q1 = cmul(zce, os0);
                const double vb[8] = {q0.re, q0.im, q1.re, q1.im, 0.0, 0.0, 0.0, 0.0};
                const double sb = wave_sum8(vb, lane);
                if ((lane & 7) == 0 && kv < 4) (kv & 1 ? ov0[at].im : ov0[at].re) = sb;
            }
        }
        wave_lds_sync();
        // b_i = i a_i of the three series (_hafnian.py:212-241 f_loop; :246-285 f_loop_odd, in
        // x = sqrt(eta): the self-edge at order 1, the even orders of f_loop, the odd row's scalars)
#pragma unroll 1
        for (int i = lane + 1; i <= nmax; i += WH_WAVE) {
            const int j = i >> 1;
            cplx2 bo = czero2(), b0 = czero2();
            if ((i & 1) == 0) {  // p_j + j v_j
                bo.h = pt[j];
                mac2(bo.h.re, bo.l.re, (double)j, lv[j].re, lvl[j].re);
                mac2(bo.h.im, bo.l.im, (double)j, lv[j].im, lvl[j].im);
                cnorm2(bo);
                b0 = bo;
                Wv[fe.bh + j] = cmulr(bo.h, 0.5);
                Wv[fe.bl + j] = cmulr(bo.l, 0.5);
            } else if (i == 1) {
                bo.h = D0;
                b0.h = D1;
            } else {
                bo.h = ov[j];
                bo = cscale2(bo, (double)i);
                if (odd0) {
                    b0.h = ov0[j];
                    b0 = cscale2(b0, (double)i);
                }
            }
            Wv[fo.bh + i] = bo.h;
            Wv[fo.bl + i] = bo.l;
            if (odd0 && i <= nf) {
                Wv[f0.bh + i] = b0.h;
                Wv[f0.bl + i] = b0.l;
            }
        }
        wave_lds_sync();
        const int nf0 = odd0 ? nf : 0;
        if (lane == 0) Wv[fo.e] = Wv[fe.e] = Wv[f0.e] = cmk(1.0, 0.0);
        wave_lds_sync();
        if (nmax + he + nf0 <= WH_WAVE) {
            const bool in_o = lane < nmax, in_e = !in_o && lane < nmax + he;
            SeriesLds mine;
            mine.bh = in_o ? fo.bh : in_e ? fe.bh : f0.bh;
            mine.bl = in_o ? fo.bl : in_e ? fe.bl : f0.bl;
            mine.e = in_o ? fo.e : in_e ? fe.e : f0.e;
            series_lanes(Wv, mine, in_o ? 0 : in_e ? nmax : nmax + he, in_o ? nmax : in_e ? he : nf0, nmax, lane);
        } else if (nmax <= WH_WAVE) {
            series_lanes(Wv, fo, 0, nmax, nmax, lane);
            series_lanes(Wv, fe, 0, he, he, lane);
            if (odd0) series_lanes(Wv, f0, 0, nf, nf, lane);
        } else {
            series_rows(Wv, fo, nmax, lane);
            series_rows(Wv, fe, he, lane);
            if (odd0) series_rows(Wv, f0, nf, lane);
        }
        wave_lds_sync();

        // loop_hafnian_batch.py:108-121 (even) and :183-202 (odd): output q on lane q mod 64
        const int start = 2 * k0 + (oddv ? 1 : 0);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int q = lane + r * WH_WAVE;
            if (q >= nL) continue;
            cplx v = cmk(0.0, 0.0);
            bool any = false;
            if (q >= start) {
                const int N = nf + q;
                const double pm = (((N / 2 - par) & 1) != 0) ? -1.0 : 1.0;
                const int half = oddv ? (q - 1) / 2 : q / 2;
                const double nb = binom_t(half, k0) * bin;
                const bool use_even = oddv ? (N % 2 == 0) : (q % 2 == 0);
                v = cmulr(Wv[use_even ? fe.e + N / 2 : fo.e + N], nb * pm);
                any = true;
            }
            if (q == 0 && odd0) {
                const double pm = (((nf / 2 - par) & 1) != 0) ? -1.0 : 1.0;
                v = cmulr(Wv[f0.e + nf], bin * pm);  // start >= 1 here: the only contribution
                any = true;
            }
            if (any) {
                if (r == 0) acc0.add(v); else acc1.add(v);
            }
        }
        wave_lds_sync();
    }
    // the waves of this workgroup in wave order
    double4* mine = reinterpret_cast<double4*>(Wv);
    if (lane < nL) mine[lane] = make_double4(acc0.sr, acc0.cr, acc0.si, acc0.ci);
    if (lane + WH_WAVE < nL) mine[lane + WH_WAVE] = make_double4(acc1.sr, acc1.cr, acc1.si, acc1.ci);
    __syncthreads();
    double4* out = partials + J.part_off + (chunk * J.nD + kd) * nL;
    for (int q = threadIdx.x; q < nL; q += blockDim.x) {
        csum s;
        s.zero();
        for (int w = 0; w < nw; ++w) {
            const double4 pq = reinterpret_cast<const double4*>(Dv + NP + w * wsz)[q];
            s.add_pair(pq.x, pq.y, pq.z, pq.w);
        }
        out[q] = make_double4(s.sr, s.cr, s.si, s.ci);
    }
}

// Folds each output's chunk partials (wave_fold's order) and applies 0.5^((n_fixed + q) // 2) for
// Glynn (loop_hafnian_batch.py:119-122, :204-207).  One workgroup, a wave per output in turn; out and
// flag are pinned host memory.
constexpr int kFoldLhbWaves = 16;
extern "C" __global__ void __launch_bounds__(kFoldLhbWaves * WH_WAVE)
wh_fold_lhb(const wh_lhb_job* __restrict__ job, const double4* __restrict__ partials, double2* __restrict__ out,
            uint64_t* __restrict__ flag, uint64_t seq) {
    const wh_lhb_job& J = *job;
    const int nout = J.nD * J.L;
    const int lane = threadIdx.x % WH_WAVE;
    for (int o = threadIdx.x / WH_WAVE; o < nout; o += blockDim.x / WH_WAVE) {
        const csum acc = wave_fold(partials + J.part_off + o, J.nchunks, nout, lane);
        double re = acc.sr + acc.cr, im = acc.si + acc.ci;
        if (J.flags & WH_LHB_GLYNN) {
            const double sc = ldexp(1.0, -((J.n_fixed + o % J.L) / 2));
            re *= sc;
            im *= sc;
        }
        if (lane == 0) out[J.out_off + o] = make_double2(re, im);
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) wh_call_done(flag, seq);
}

size_t wh_lhb_lds_bytes(int T, int nw, int nmax, int nf) {
    const size_t NP = 8 * (size_t)T, S = NP + 2;
    return (NP * S + NP + nw * lhb_wave_cplx(T, nmax, nf)) * sizeof(cplx) +
           kSymBinom * sizeof(double);
}

// Waves per workgroup: the most per CU under the LDS (8 by the registers up to T = 3, 4 above).
int wh_lhb_waves(int T, int nmax, int nf) {
    int best = 1, best_w = 0;
    for (int nw = 1; nw <= 4; ++nw) {
        int per_cu = (int)(160 * 1024 / wh_lhb_lds_bytes(T, nw, nmax, nf)) * nw;
        if (per_cu > (T <= 3 ? 8 : 4)) per_cu = T <= 3 ? 8 : 4;
        if (per_cu >= best_w && per_cu > 0) { best_w = per_cu; best = nw; }
    }
    return best;
}

template <int T, bool FULL>
static hipError_t launch_lhb(const wh_lhb_job* job, const void* pool, void* partials, int64_t nblocks,
                             int nw, int nmax, int nf, hipStream_t stream) {
    const size_t lds = wh_lhb_lds_bytes(T, nw, nmax, nf);
    static wh_lds_limit lim;
    hipError_t err = wh_raise_lds_limit((const void*)wh_sieve_lhb<T, FULL>, lds, lim);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((wh_sieve_lhb<T, FULL>), dim3((unsigned)nblocks), dim3(nw * WH_WAVE), lds, stream, job,
                       (const cplx*)pool, (double4*)partials, nmax, nf);
    return hipGetLastError();
}

// One job: its chunks x diagonals workgroups, then the fold of its nout outputs into pinned host memory.
// full: the matrix is not symmetric.
hipError_t wh_launch_lhb(const wh_lhb_job* job, const void* pool, void* partials, int64_t nblocks, int T, bool full,
                         int nw, int nmax, int nf, int nout, void* out, uint64_t* flag, uint64_t seq,
                         hipStream_t stream) {
    if (nw < 1 || nw > 4 || nmax < 0 || nmax > WH_NMAX || nf < 0 || nf > nmax) return hipErrorInvalidValue;
    hipError_t err;
#define WH_LHB_CASE(TT)                                                                     \
    case TT:                                                                                \
        err = full ? launch_lhb<TT, true>(job, pool, partials, nblocks, nw, nmax, nf, stream)   \
                   : launch_lhb<TT, false>(job, pool, partials, nblocks, nw, nmax, nf, stream); \
        break;
    switch (T) {
        WH_LHB_CASE(1)
        WH_LHB_CASE(2)
        WH_LHB_CASE(3)
        WH_LHB_CASE(4)
        WH_LHB_CASE(5)
        WH_LHB_CASE(6)
        default: return hipErrorInvalidValue;
    }
#undef WH_LHB_CASE
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(wh_fold_lhb, dim3(1), dim3(std::min(nout, kFoldLhbWaves) * WH_WAVE), 0, stream, job,
                       (const double4*)partials, (double2*)out, flag, seq);
    return hipGetLastError();
}
