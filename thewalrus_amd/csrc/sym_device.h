// sym_device.h -- symmetric powers of the term matrix for any column factors on the FP64 matrix
// cores: the per-wave building blocks shared by sieve_sym.hip (single requests) and sieve_lhb.hip
// (batched loop hafnians).  Notation as in sieve_sym.hip: B = A G with G = X Delta,
// C_a = A (G A)^(a-1) symmetric, W_a = C_a Delta in the wave's LDS.
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

__device__ __forceinline__ double mfma4(double a, double b, double c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
// c + a (-b): for the f64 instructions the last operand holds the negate bits (A, B, C)
__device__ __forceinline__ double mfma4_nb(double a, double b, double c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 2);
}
// the partner of index c in the other half of 2E indices (identity on the padding)
__device__ __forceinline__ int swp(int c, int E) { return c < E ? c + E : (c < 2 * E ? c - E : c); }

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
template <int T, bool BREG>
__device__ __forceinline__ void sym_product(const cplx* W, const cplx* XA, const Bop<T> (&B)[BREG ? 2 * T : 1],
                                            double (&cR)[GeoG<T>::NG], double (&cI)[GeoG<T>::NG], const LaneMapG& L,
                                            int nk) {
    constexpr int S = GeoG<T>::S;
    constexpr int NG = GeoG<T>::NG;
    double cY[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) cR[g] = cI[g] = cY[g] = 0.0;
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
#ifdef WH_SYM_4M
                cR[g] = mfma4_nb(av[p].im, bq[q].im, cR[g]);
                cI[g] = mfma4(av[p].re, bq[q].im, cI[g]);
                cI[g] = mfma4(av[p].im, bq[q].re, cI[g]);
#else
                cY[g] = mfma4(av[p].im, bq[q].im, cY[g]);
                cI[g] = mfma4(av[p].re + av[p].im, bq[q].re + bq[q].im, cI[g]);
#endif
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
#ifndef WH_SYM_4M
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const double x = cR[g], y = cY[g];
        cR[g] = x - y;
        cI[g] = cI[g] - (x + y);
    }
#endif
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

#define WH_DPP_ROW_SHR1 0x111     // lane i of a 16-lane row takes lane i - 1 (0 for lane 0)
#define WH_DPP_ROW_NEWBCAST 0x150 // + l: every lane of a row takes the row's lane l

// One step of the exponential recurrence over 16-lane rows: lane m - 1 holds s_m =
// sum_(i < K) b_(m-i) e_i so far; e_K = s_K / K from lane K - 1 joins the later orders.
template <int K>
__device__ __forceinline__ void series_step(cplx& s, cplx& b) {
    b.re = dpp_d<WH_DPP_ROW_SHR1>(b.re);  // lane m - 1 now holds b_(m-K), 0 for m <= K
    b.im = dpp_d<WH_DPP_ROW_SHR1>(b.im);
    const cplx e = cmulr(cmk(dpp_d<WH_DPP_ROW_NEWBCAST + K - 1>(s.re), dpp_d<WH_DPP_ROW_NEWBCAST + K - 1>(s.im)),
                         1.0 / K);
    cmac(s, b, e);
}
template <int K>
__device__ __forceinline__ void series_steps(cplx& s, cplx& b, int h) {
    if constexpr (K < 16) {
        if (K < h) {  // uniform over the wave
            series_step<K>(s, b);
            series_steps<K + 1>(s, b, h);
        }
    }
}

}  // namespace
