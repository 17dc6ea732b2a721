// sym_device.h -- symmetric powers of the term matrix for any column factors on the FP64 matrix
// cores: the per-wave building blocks shared by sieve_sym.hip (single requests) and sieve_lhb.hip
// (batched loop hafnians).  Notation as in sieve_sym.hip: B = A G with G = X Delta,
// C_a = A (G A)^(a-1) symmetric, W_a = C_a Delta in the wave's LDS.
//
// Those powers hold for a symmetric matrix only, which the entry points do not require: hafnian
// accepts a relative asymmetry of 1e-5, the others check nothing.  The start of a workgroup (for the
// batched loop hafnian: the host) compares the entries and takes a matrix that is not symmetric
// through its full powers (full_scalars), so that a term is the reference's for every matrix.
#pragma once
#include "wh_device.h"

namespace {

// 1 / k for the coefficient recurrences
struct InvTable {
    double v[WH_NMAX + 2];
    constexpr InvTable() : v() {
        for (int k = 1; k < WH_NMAX + 2; ++k) v[k] = 1.0 / k;
    }
};
static __constant__ InvTable kInv = InvTable();

// C(n, k) for every edge multiplicity (n <= WH_NMAX / 2), by Pascal in 64 bits (C(64, 32) < 2^61),
// rounded once; binom_d's remainders cost a workgroup's start several microseconds
constexpr int kBinomSide = WH_NMAX / 2 + 1;
struct BinomTable {
    double v[kBinomSide][kBinomSide];
    constexpr BinomTable() : v() {
        uint64_t row[kBinomSide] = {};
        row[0] = 1;
        for (int n = 0; n < kBinomSide; ++n) {
            if (n > 0)
                for (int k = n; k >= 1; --k) row[k] += row[k - 1];
            for (int k = 0; k < kBinomSide; ++k) v[n][k] = (double)row[k];
        }
    }
};
static __constant__ BinomTable kBinom = BinomTable();
__device__ __forceinline__ double binom_t(int n, int k) { return kBinom.v[n][k]; }

// ---- two-word arithmetic: a value is hi + lo, an accumulator a sum s with its collected error c.
// (contraction off: a product that feeds an error-free sum must be the rounded one)
__device__ __forceinline__ void acc2(double& s, double& c, double p, double e) {
#pragma clang fp contract(off)
    const double t = s + p, bb = t - s;
    c += ((s - (t - bb)) + (p - bb)) + e;
    s = t;
}
// (s, c) += a (bh + bl)
__device__ __forceinline__ void mac2(double& s, double& c, double a, double bh, double bl) {
#pragma clang fp contract(off)
    const double p = a * bh;
    acc2(s, c, p, fma(a, bl, fma(a, bh, -p)));
}
// (s, c) += a b, four instructions: the error of a product smaller than s is kept whole, of a larger one
// to its own rounding
__device__ __forceinline__ void macp(double& s, double& c, double a, double b) {
    const double t = fma(a, b, s);
    c += fma(a, b, s - t);
    s = t;
}
template <bool RE>
__device__ __forceinline__ void cmacp(cplx& s, cplx& c, cplx a, cplx b) {
    macp(s.re, c.re, a.re, b.re);
    if constexpr (!RE) {
        macp(s.re, c.re, -a.im, b.im);
        macp(s.im, c.im, a.re, b.im);
        macp(s.im, c.im, a.im, b.re);
    }
}
// Lane map of the 4x4x4 instruction as in sieve_pm1s.hip: group (p, q) holds
// C[8p + 4br + y][8q + 4bc + x].
template <int T> struct GeoG {
    static constexpr int NP = 8 * T;
    static constexpr int S = NP + 2;  // LDS row stride: as sieve_pm1s.hip
    static constexpr int NG = T * (T + 1) / 2;
};
constexpr int kSymBinom = WH_NMAX / 2 + WH_EMAX + 4;  // binomials C(e_i, k) of all edges

struct LaneMapG {
    int x, y, br, bc;
    __device__ int rd(int p) const { return 8 * p + 4 * br + y; }
    __device__ int cd(int q) const { return 8 * q + 4 * bc + x; }
};

// X A operands of one k chunk
template <int T> struct Bop {
    cplx b[T];
};

// C_new = W (X A), upper groups, k chunks [0, nk); complex products from three real ones (as
// sieve_pm1s.hip: Re = X - Y, Im = Z - X - Y with X = sum Re a Re b, Y = sum Im a Im b,
// Z = sum (Re a + Im a)(Re b + Im b)).
// BREG: X A's operands (2T x T complex per lane) stay in registers over a workgroup's terms.
// FOUR: complex products from four real ones (plain terms: without loop scalars the powers' rounding is
// most of a term's; inclusion-exclusion on 16 modes 0.88 of the error, 250 against 234 us).
template <int T, bool BREG, bool FOUR = false>
__device__ __forceinline__ void sym_product(const cplx* W, const cplx* XA, const Bop<T> (&B)[BREG ? 2 * T : 1],
                                            double (&cR)[GeoG<T>::NG], double (&cI)[GeoG<T>::NG], const LaneMapG& L,
                                            int nk) {
    constexpr int S = GeoG<T>::S;
    constexpr int NG = GeoG<T>::NG;
    double cY[FOUR ? 1 : NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        cR[g] = cI[g] = 0.0;
        if constexpr (!FOUR) cY[g] = 0.0;
    }
    const int ia = (4 * L.br + L.x) * S + L.y;
    const int ib = L.y * S + 4 * L.bc + L.x;
    auto chunk = [&](int kc) {
        cplx av[T], bq[T];
#pragma unroll
        for (int p = 0; p < T; ++p) av[p] = W[ia + 8 * p * S + 4 * kc];
#pragma unroll
        for (int q = 0; q < T; ++q) {
            if constexpr (BREG) bq[q] = B[kc].b[q];
            else bq[q] = XA[ib + 4 * kc * S + 8 * q];
        }
        int g = 0;
#pragma unroll
        for (int p = 0; p < T; ++p)
#pragma unroll
            for (int q = p; q < T; ++q, ++g) {
                cR[g] = mfma4(av[p].re, bq[q].re, cR[g]);
                if constexpr (FOUR) {
                    cR[g] = mfma4_nb(av[p].im, bq[q].im, cR[g]);
                    cI[g] = mfma4(av[p].re, bq[q].im, cI[g]);
                    cI[g] = mfma4(av[p].im, bq[q].re, cI[g]);
                } else {
                    cY[g] = mfma4(av[p].im, bq[q].im, cY[g]);
                    cI[g] = mfma4(av[p].re + av[p].im, bq[q].re + bq[q].im, cI[g]);
                }
            }
    };
    if constexpr (T <= 4) {  // (operands in registers need constant chunk indices)
#pragma unroll
        for (int kc = 0; kc < 2 * T; ++kc) {
            if (kc >= nk) break;
            chunk(kc);
        }
    } else {
#pragma unroll 2
        for (int kc = 0; kc < nk; ++kc) chunk(kc);
    }
    if constexpr (!FOUR) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const double x = cR[g], y = cY[g];
            cR[g] = x - y;
            cI[g] = cI[g] - (x + y);
        }
    }
}

// lane part of tr(B^(a+b)) = sum_i delta_i sum_k C_a[i][k] W_b[s i][s k]
template <int T>
__device__ __forceinline__ cplx sym_trace(const cplx* W, const double (&cR)[GeoG<T>::NG],
                                          const double (&cI)[GeoG<T>::NG], const double (&dr)[T], const LaneMapG& L,
                                          int E) {
    constexpr int S = GeoG<T>::S;
    cplx s = cmk(0.0, 0.0);
    int g = 0;
#pragma unroll
    for (int p = 0; p < T; ++p) {
        const int rs = swp(L.rd(p), E) * S;
        cplx sd = cmk(0.0, 0.0), so = cmk(0.0, 0.0);
#pragma unroll
        for (int q = p; q < T; ++q, ++g) {
            const cplx w = W[rs + swp(L.cd(q), E)];
            if (q == p) cmac(sd, cmk(cR[g], cI[g]), w);
            else cmac(so, cmk(cR[g], cI[g]), w);
        }
        s.re = fma(dr[p], fma(2.0, so.re, sd.re), s.re);
        s.im = fma(dr[p], fma(2.0, so.im, sd.im), s.im);
    }
    return s;
}

template <int T>
__device__ __forceinline__ void sym_store(cplx* W, const double (&cR)[GeoG<T>::NG], const double (&cI)[GeoG<T>::NG],
                                          const double (&dr)[T], const double (&dc)[T], const LaneMapG& L) {
    constexpr int S = GeoG<T>::S;
    int g = 0;
#pragma unroll
    for (int p = 0; p < T; ++p)
#pragma unroll
        for (int q = p; q < T; ++q, ++g) {
            const cplx c = cmk(cR[g], cI[g]);
            W[L.rd(p) * S + L.cd(q)] = cmulr(c, dc[q]);
            if (p < q) W[L.cd(q) * S + L.rd(p)] = cmulr(c, dr[p]);
        }
}

// z = W xd by rows (xd the lane's columns of X D); every lane of a row stores the same sum
template <int T>
__device__ __forceinline__ void sym_matvec(const cplx* W, const cplx (&xd)[T], cplx* z, const LaneMapG& L) {
    constexpr int S = GeoG<T>::S;
#pragma unroll
    for (int p = 0; p < T; ++p) {
        cplx s = cmk(0.0, 0.0);
#pragma unroll
        for (int q = 0; q < T; ++q) cmac(s, W[L.rd(p) * S + L.cd(q)], xd[q]);
        s.re += dpp_d<WH_DPP_XOR1>(s.re);
        s.im += dpp_d<WH_DPP_XOR1>(s.im);
        s.re += dpp_d<WH_DPP_XOR2>(s.re);
        s.im += dpp_d<WH_DPP_XOR2>(s.im);
        s.re += dpp_d<WH_DPP_ROR8>(s.re);
        s.im += dpp_d<WH_DPP_ROR8>(s.im);
        z[L.rd(p)] = s;
    }
}

// ---- Matrices that are not exactly symmetric.
// With A = S + N, N antisymmetric, transposition turns every trace tr((A G)^k) and every scalar
// D^T (G A)^k G D into that of S - N: an even-N term is an even function of N, and its symmetric part
// stands for it up to N^2.  A scalar with another vector on its left (odd N, batched loop hafnians)
// is not: there N counts in the first order.  So the matrix is replaced by (A + A^T) / 2 where
// |N_ij| <= tol m_i m_j / max m, m_i the largest entry of row and column i (alike for A and for any
// diagonal scaling of it), and goes through its full powers where it is not, or where an entry is not
// finite (a dropped row may hold anything).
// The tolerances stand in wh_device.h.
__device__ __forceinline__ bool finite_c(cplx v) { return fabs(v.re) + fabs(v.im) < INFINITY; }
// a_ij and a_ji are one finite number
__device__ __forceinline__ bool twins(cplx a, cplx b) { return a.re == b.re && a.im == b.im && finite_c(a); }

// The whole workgroup, for a staged matrix of side n that is not exactly symmetric and finite: true if
// it needs its full powers; else its two triangles are replaced by their mean.  get(i, j) and
// put(i, j, v): the staged entries; scale: n doubles of LDS nobody reads before the next barrier.
template <class Get, class Put>
__device__ __forceinline__ bool settle_symmetry(int n, double tol, double* scale, Get get, Put put) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        double m = 0.0;
        for (int j = 0; j < n; ++j) {
            const cplx a = get(i, j), b = get(j, i);
            if (!finite_c(a) || !finite_c(b)) m = INFINITY;
            m = fmax(m, fmax(fmax(fabs(a.re), fabs(a.im)), fmax(fabs(b.re), fabs(b.im))));
        }
        scale[i] = m;
    }
    __syncthreads();
    double top = 0.0;
    for (int i = 0; i < n; ++i) top = fmax(top, scale[i]);
    bool far = !(top < INFINITY);
    for (int e = threadIdx.x; e < n * n && !far; e += blockDim.x) {
        const int i = e / n, j = e - i * n;
        const cplx d = csub(get(i, j), get(j, i));
        const double s = fmax(fabs(d.re), fabs(d.im));
        if (s != 0.0 && !(0.5 * s / scale[i] <= tol * (scale[j] / top))) far = true;
    }
    if (__syncthreads_or(far)) return true;
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
        const int i = e / n, j = e - i * n;
        if (i >= j) continue;  // (one thread per pair)
        const cplx a = get(i, j), b = get(j, i);
        const cplx m = cmk(0.5 * a.re + 0.5 * b.re, 0.5 * a.im + 0.5 * b.im);
        put(i, j, m);
        put(j, i, m);
    }
    __syncthreads();
    return false;
}

// A term's scalars from the full powers of B = A G, as the reference forms them (charpoly.py:302-327,
// _hafnian.py:212-285): p[k] = tr(B^k) and, with vectors, out[l][k] = (X left_l)_d B^(k-1) D for
// k = 1..h, by one wave.  A(i, j), D(j), left(l, j): the matrix and the vectors, by request index;
// E edges, delta of edge e at dl[e]; rows and columns with delta = 0 take part in nothing, whatever they
// hold.  P: n x n complex of LDS with row stride S; z: n complex.  One lane per entry of a few rows at
// a time, in place row by row; both operands from LDS, as in sieve_generic.hip.
template <int NL, class GetA, class GetD, class GetL>
__device__ __forceinline__ void full_scalars(GetA A, GetD D, GetL left, int E, int h, const double* dl, cplx* P, int S,
                                             cplx* z, cplx* p, cplx* const (&out)[NL > 0 ? NL : 1], int lane) {
    const int n = 2 * E;
    auto edge = [&](int c) { return c < E ? c : c - E; };
    const double my_d = lane < n ? dl[edge(lane)] : 0.0;
    const int rows = WH_WAVE / n, row = lane / n, col = lane - row * n;  // (lanes past rows n idle)
    const bool on = row < rows;
    const int cs = swp(col, E);
    const double cd = on ? dl[edge(col)] : 0.0;
    cplx zl = cmk(0.0, 0.0);
    cplx lv[NL > 0 ? NL : 1];
    if constexpr (NL > 0) {
        if (my_d != 0.0) {
            zl = D(lane);
#pragma unroll
            for (int l = 0; l < NL; ++l) lv[l] = cmulr(left(l, swp(lane, E)), my_d);
        }
    }
    for (int i = row; i < n && on; i += rows) {
        cplx v = cmk(0.0, 0.0);
        if (cd != 0.0 && dl[edge(i)] != 0.0) v = cmulr(A(i, cs), cd);
        P[i * S + col] = v;
    }
    wave_lds_sync();
#pragma unroll 1
    for (int k = 1;; ++k) {
        const cplx tr = wave_csum(lane < n ? P[lane * S + lane] : cmk(0.0, 0.0));
        if (lane == 0) p[k] = tr;
        if constexpr (NL > 0) {
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                const cplx s = wave_csum(my_d != 0.0 ? cmul(lv[l], zl) : cmk(0.0, 0.0));
                if (lane == 0) out[l][k] = s;
            }
        }
        if (k >= h) break;
        if constexpr (NL > 0) {
            if (lane < n) z[lane] = cmulr(zl, my_d);
            wave_lds_sync();
            zl = cmk(0.0, 0.0);
            if (my_d != 0.0)
                for (int c = 0; c < n; ++c)
                    if (dl[edge(c)] != 0.0) cmac(zl, A(lane, swp(c, E)), z[c]);
            wave_lds_sync();
        }
#pragma unroll 1
        for (int i0 = 0; i0 < n; i0 += rows) {
            const int i = i0 + row;
            const bool here = on && i < n;
            cplx s = cmk(0.0, 0.0);
            if (here)
                for (int q = 0; q < n; ++q)
                    if (dl[edge(q)] != 0.0) cmac(s, P[i * S + q], A(q, cs));
            wave_lds_sync();
            if (here) P[i * S + col] = cd != 0.0 ? cmulr(s, cd) : cmk(0.0, 0.0);
            wave_lds_sync();
        }
    }
    wave_lds_sync();
}

// Coefficient `top` of a term's series from its full scalars: f and f_loop (_hafnian.py:184-241), or for
// odd N f_loop_odd (:246-285, orders in sqrt(eta)); e: top + 1 complex of LDS.  e_k = (1 / k) sum_i b_i
// e_(k-i), the lanes sharing the sum; every lane returns the value.
template <bool LOOP>
__device__ __forceinline__ cplx full_coeff(int top, bool odd, cplx oddloop, const cplx* p, const cplx* v,
                                           const cplx* o, cplx* e, int lane) {
    if (lane == 0) e[0] = cmk(1.0, 0.0);
    wave_lds_sync();
    cplx r = cmk(1.0, 0.0);
#pragma unroll 1
    for (int k = 1; k <= top; ++k) {
        cplx s = cmk(0.0, 0.0);
        for (int i = lane + 1; i <= k; i += WH_WAVE) {
            cplx b;  // i a_i
            if (!odd) {
                b = cmulr(p[i], 0.5);
                if (LOOP) b = cadd(b, cmulr(v[i], 0.5 * i));
            } else if (i == 1) {
                b = oddloop;
            } else if ((i & 1) == 0) {
                b = cadd(p[i / 2], cmulr(v[i / 2], 0.5 * i));
            } else {
                b = cmulr(o[(i - 1) / 2], (double)i);
            }
            cmac(s, b, e[k - i]);
        }
        r = cmulr(wave_csum(s), kInv.v[k]);
        if (lane == 0) e[k] = r;
        wave_lds_sync();
    }
    return r;
}

#define WH_DPP_ROW_SHR1 0x111     // lane i of a 16-lane row takes lane i - 1 (0 for lane 0)
#define WH_DPP_ROW_NEWBCAST 0x150 // + l: every lane of a row takes the row's lane l

// The exponential recurrence of a term over a 16-lane row: lane m - 1 brings b_m = m a_m (0 past
// m = h <= 16) and receives s_m = sum_(i < m) b_(m-i) e_i, e_m = s_m / m.  In step K lane K - 1's
// e_K joins the later orders.  TWO keeps s in two words (s, c): plain and odd-N terms, where its rounding
// was the largest part (inclusion-exclusion on 10 and 16 modes: 0.8 of the error with one word, for 2%
// of the time); with even-N loops it is not, and one word is 4% faster.
template <bool RE, bool TWO, int K>
__device__ __forceinline__ void series_steps(cplx& s, cplx& c, cplx& b, int h) {
    if constexpr (K < 16) {
        if (K < h) {  // uniform over the wave
            b.re = dpp_d<WH_DPP_ROW_SHR1>(b.re);  // lane m - 1 now holds b_(m-K), 0 for m <= K
            if (!RE) b.im = dpp_d<WH_DPP_ROW_SHR1>(b.im);
            const double re = TWO ? s.re + c.re : s.re, im = TWO ? s.im + c.im : s.im;
            const cplx e = cmk(dpp_d<WH_DPP_ROW_NEWBCAST + K - 1>(re) * (1.0 / K),
                               RE ? 0.0 : dpp_d<WH_DPP_ROW_NEWBCAST + K - 1>(im) * (1.0 / K));
            if constexpr (TWO) cmacp<RE>(s, c, b, e);
            else if constexpr (RE) s.re = fma(b.re, e.re, s.re);
            else cmac(s, b, e);
            series_steps<RE, TWO, K + 1>(s, c, b, h);
        }
    }
}
template <bool RE, bool TWO>
__device__ __forceinline__ cplx series_row(cplx b, int h) {
    cplx s = b, c = cmk(0.0, 0.0);
    series_steps<RE, TWO, 1>(s, c, b, h);
    return TWO ? cadd(s, c) : s;
}

// Odd N (sieve_sym.hip): sum_(k <= h) u_k e_(h-k) from the lanes' s_m of LANES (16 or 64) lanes, on every
// one of them.
template <int LANES>
__device__ __forceinline__ cplx odd_row(cplx s, const cplx* u, int h, int lane) {
    const int m = (lane & (LANES - 1)) + 1;
    cplx t = cmk(0.0, 0.0), c = t;
    if (m < h) cmacp<false>(t, c, u[h - m], cmulr(s, kInv.v[m]));
    else if (m == h) t = u[h];
    auto add = [&](double r, double rc, double i, double ic) {
        acc2(t.re, c.re, r, rc);
        acc2(t.im, c.im, i, ic);
    };
    add(dpp_d<WH_DPP_XOR1>(t.re), dpp_d<WH_DPP_XOR1>(c.re), dpp_d<WH_DPP_XOR1>(t.im), dpp_d<WH_DPP_XOR1>(c.im));
    add(dpp_d<WH_DPP_XOR2>(t.re), dpp_d<WH_DPP_XOR2>(c.re), dpp_d<WH_DPP_XOR2>(t.im), dpp_d<WH_DPP_XOR2>(c.im));
    add(dpp_d<WH_DPP_HALF_MIRROR>(t.re), dpp_d<WH_DPP_HALF_MIRROR>(c.re), dpp_d<WH_DPP_HALF_MIRROR>(t.im),
        dpp_d<WH_DPP_HALF_MIRROR>(c.im));
    add(dpp_d<WH_DPP_MIRROR>(t.re), dpp_d<WH_DPP_MIRROR>(c.re), dpp_d<WH_DPP_MIRROR>(t.im), dpp_d<WH_DPP_MIRROR>(c.im));
    for (int x = 16; x < LANES; x <<= 1)
        add(__shfl_xor(t.re, x, WH_WAVE), __shfl_xor(c.re, x, WH_WAVE), __shfl_xor(t.im, x, WH_WAVE),
            __shfl_xor(c.im, x, WH_WAVE));
    return cadd(t, c);
}

}  // namespace
