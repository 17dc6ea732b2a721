// sieve_sym.hip -- the power-trace sieve for any edge multiplicities on the FP64 matrix cores with
// symmetric powers: repeated rows past the repeated-row kernel's limits, inclusion-exclusion, and
// odd-N loop hafnians (Glynn); the terms of _hafnian.py:443-462 (plain) and :546-569 (loop).
//
// With A = Ax symmetric, X the swap of the two halves and Delta = diag(delta) (delta repeats over
// the halves, so G = X Delta = Delta X is symmetric), the term matrix on every row is B = A G (a
// column with delta = 0 is zero, so the dropped rows of the reference change no trace and no loop
// scalar) and
//     C_a = A (G A)^(a-1)   is symmetric,  B^a = C_a G.
// A wave keeps W_a = C_a Delta in LDS and forms C_(a+1) = W_a (X A) on the matrix cores, upper
// 8 x 8 block groups only, X A staged once per workgroup; it stores C delta_j at (i, j) and
// C delta_i at (j, i).  Powers run to A = ceil(h / 2); with s the half swap
//     tr(B^(a+b)) = sum_i delta_i sum_k C_a[i][k] W_b[s i][s k]     (symmetric in i, k: the groups
//                                                                    off the diagonal count twice)
//     z_a = B^a D = W_a (X D),  XD_d B^(a+b) D = sum_e delta_e z_a[s e] z_b[e].
// The coefficient of eta^h of exp(sum (p_k / 2k + v_k / 2) eta^k) follows from the exponential
// recurrence, four terms of a wave at a time (16 lanes each, one order per lane).
//
// Odd N: the unpaired mode becomes one more edge, with a partner that couples to nothing and
// carries a loop of weight s (lhaf of the two is the product lhaf x s), delta = -1 (multiplicity 1,
// and Glynn's sum is even in delta, so one sign of that edge is the whole sum): the same 2h + 1
// photon sum over the same terms, as an even-N request of h + 1.  The value is what s multiplies
// once, and only that is formed: with y_a = B^a e_partner, which is W_a's column of the unpaired mode,
//     u_(a+b+1) = sum_e delta_e y_a[s e] z_b[e],
// z from D without the partner's loop, the coefficient is sum_k u_k e_(h-k), e the series of the rest.
// (With s = 1 as a number the terms also carry powers of s that cancel in their sum only: 1.2 to 1.5
// times the error.)  p_k and v_k are then summed as one value, b_k = p_k / 2 + k v_k / 2.
//
// A matrix that is not symmetric (sym_device.h) takes the full powers of B and, for odd N, the
// reference's own series in sqrt(eta), one term at a time (the edge above would pass V's walks through
// A in both directions): n h (n + 1) multiply-adds from LDS per term, the general kernel's cost.
//
// Bound: FP64 issue (matrix cores and the epilogue's vector FP64 share the pipe) at 2-4 waves per
// SIMD (one for sides above 32), which hide the serial steps of a power (product, trace, store, sums).
// A 23-mode call (2048 waves, two per SIMD, one term each) is its terms' chain: matrix cores busy 16%,
// the other vector instructions 21% of 41 us.
// It replaced the one-wave LDS kernel (sieve_generic.hip: every complex multiply-add read two
// 16-byte operands from LDS, h - 1 full products per term) for these requests.
#include "sym_device.h"
#include "wh_launch.h"

namespace {

constexpr int kSymBatch = 4;  // terms whose coefficients are formed together (16 lanes each)

// One wave's LDS (complex entries): W, z rows of two powers, term slots (p_1.., v_1..), then
// doubles: delta by index and the slots' prefactors.
__host__ __device__ constexpr size_t sym_wave_cplx(int T, bool loop, int H) {
    const size_t NP = 8 * (size_t)T, S = NP + 2, PN = (size_t)H + 2;
    return NP * S + (loop ? 2 * NP : 0) + kSymBatch * PN * (loop ? 2 : 1) + NP / 2 + kSymBatch / 2;
}

// b_m = m a_m of a term's coefficient series exp(sum_i (p_i / 2i + v_i / 2) eta^i), the term's p and v
// at sl and sl + PN (odd N: b itself at sl)
template <bool LOOP>
__device__ __forceinline__ cplx series_coeff(const cplx* sl, int PN, int h, int m, bool odd) {
    cplx b = cmk(0.0, 0.0);
    if (m <= h) {
        b = cmulr(sl[m], odd ? 1.0 : 0.5);
        if (LOOP && !odd) {
            const cplx v = sl[PN + m];
            b.re = fma(0.5 * m, v.re, b.re);
            b.im = fma(0.5 * m, v.im, b.im);
        }
    }
    return b;
}

}  // namespace

// jobs[]: sorted by chunk_base; block b finds its job by binary search.  partials[b] =
// (sum_re, err_re, sum_im, err_im) of the chunk's signed terms.  H: the largest h the launch's
// slots hold.
// CALL: the single-call form (wh_call; one job, chunks of at most kSymBatch terms per wave).
template <int T, bool LOOP, bool CALL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CALL && T < 3 ? 2 : T == 1 ? 4 : T <= 3 ? 3 : T == 4 ? 2 : 1)))
wh_sieve_sym(const wh_job_dev* __restrict__ jobs, int njobs, const cplx* __restrict__ pool,
             double4* __restrict__ partials, int64_t block_offset, int H, wh_call C) {
    extern __shared__ __align__(16) unsigned char wh_smem[];
    constexpr int NP = GeoG<T>::NP;
    constexpr int S = GeoG<T>::S;
    constexpr int NG = GeoG<T>::NG;
    const int64_t b = CALL ? blockIdx.x / C.nsplit : blockIdx.x + block_offset;  // CALL: (chunk, part)
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].chunk_base <= b) lo = mid; else hi = mid - 1;
    }
    const wh_job_dev& J = jobs[lo];
    const int nw = blockDim.x / WH_WAVE;
    const int wave = threadIdx.x / WH_WAVE;
    const int lane = threadIdx.x % WH_WAVE;
    LaneMapG L;
    L.x = lane & 3;
    L.br = (lane >> 2) & 1;
    L.bc = (lane >> 3) & 1;
    L.y = lane >> 4;
    const bool odd = (J.flags & WH_F_ODD) != 0;
    const bool glynn = (J.flags & WH_F_GLYNN) != 0;
    const int E0 = J.E;                  // the request's edges
    const int E = E0 + (odd ? 1 : 0);    // and the unpaired mode's
    const int n = 2 * E;
    const int h = (J.N + 1) / 2;
    const int Ahalf = (h + 1) / 2;
    const int PN = H + 2;

    // ---- LDS carve (wh_sym_lds_bytes)
    cplx* XA = reinterpret_cast<cplx*>(wh_smem);
    cplx* Dv = XA + NP * S;
    cplx* Wv = Dv + (LOOP ? NP : 0) + (size_t)wave * sym_wave_cplx(T, LOOP, H);
    cplx* Zb = Wv + NP * S;                       // z rows of two powers
    cplx* slots = Zb + (LOOP ? 2 * NP : 0);
    const int SL = LOOP ? 2 * PN : PN;
    double* dl = reinterpret_cast<double*>(slots + kSymBatch * SL);  // delta by index
    double* pf = dl + NP;                                            // prefactors by slot
    double* btab = reinterpret_cast<double*>(Dv + (LOOP ? NP : 0) + (size_t)nw * sym_wave_cplx(T, LOOP, H));
    double4* wres = reinterpret_cast<double4*>(btab + kSymBinom);

    // ---- stage X A (row r holds row swap(r) of A), zero padded; for odd N the unpaired mode is
    // index E - 1 and its partner 2E - 1
    const cplx* A = pool + J.a_off;
    const cplx* V = odd ? pool + J.v_off : nullptr;
    const cplx* Dg = LOOP ? pool + J.d_off : nullptr;
    const int n0 = 2 * E0;
    bool rough = (J.flags & WH_F_NONSYM) != 0;  // not exactly symmetric, or not finite
    {
        for (int e = threadIdx.x; e < NP * NP; e += blockDim.x) {
            const int r = e / NP, c = e - r * NP;
            cplx v = cmk(0.0, 0.0);
            if (r < n && c < n) {
                const int rs = swp(r, E);
                const int ro = rs < E ? rs : rs - E, co = c < E ? c : c - E;  // edges
                const int ri = rs < E ? ro : ro + E0, ci = c < E ? co : co + E0;  // request indices
                if (ro < E0 && co < E0) {
                    v = A[ri * n0 + ci];
                    rough = rough || !twins(v, A[ci * n0 + ri]);
                } else if (ro < E0 && c == E - 1) {
                    v = V[ri];
                    rough = rough || !finite_c(v);
                } else if (co < E0 && rs == E - 1) {
                    v = V[ci];
                }
            }
            XA[r * S + c] = v;
        }
        if (LOOP) {
            for (int e = threadIdx.x; e < NP; e += blockDim.x) {
                cplx v = cmk(0.0, 0.0);
                if (e < n) {
                    const int eo = e < E ? e : e - E;
                    if (eo < E0) {
                        v = Dg[e < E ? eo : eo + E0];
                        rough = rough || !finite_c(v);
                    } else {
                        v = e < E ? cmk(J.oddloop_re, J.oddloop_im) : cmk(0.0, 0.0);
                    }
                }
                Dv[e] = v;
            }
        }
    }
    // lane i < E0 owns digit i: its radix, weight and binomial row
    const int my_e = lane < E0 ? J.e[lane] : 0;
    int64_t my_w = 1;
    int my_row = 0;
    bool ones = true;
    for (int l = 0; l < E0; ++l) {
        const int el = __builtin_amdgcn_readlane(my_e, l);
        if (l > lane) my_w *= (int64_t)(el + 1);
        if (l < lane) my_row += el + 1;
        ones = ones && el <= 1;
    }
    if (!ones && wave == 0 && lane < E0)
        for (int k = 0; k <= my_e; ++k) btab[my_row + k] = binom_t(my_e, k);

    int64_t t0 = (b - J.chunk_base) * J.chunk_terms;
    int64_t t1 = t0 + J.chunk_terms;
    if (t1 > J.steps) t1 = J.steps;
    if (CALL) {
        t0 += (int64_t)(blockIdx.x % C.nsplit) * nw;
        if (t1 > t0 + nw) t1 = t0 + nw;
    }
    const bool small = J.steps < ((int64_t)1 << 31);
    csum acc;
    acc.zero();

    // term t: its delta by index into the wave's LDS; returns its signed binomial product
    auto term_factors = [&](int64_t t) {
        // _hafnian.py:444-459: digits, binomial product, sign, delta
        int k = 0;
        if (lane < E0) {
            if (small) k = (int)(((uint32_t)t / (uint32_t)my_w) % (uint32_t)(my_e + 1));
            else k = (int)((t / my_w) % (int64_t)(my_e + 1));
        }
        const int delta = glynn ? 2 * k - my_e : k;
        wave_lds_sync();  // the previous term's reads of dl are done
        if (lane < NP) dl[lane] = 0.0;
        wave_lds_sync();
        if (lane < E0) dl[lane] = dl[lane + E] = (double)delta;
        if (odd && lane == E0) dl[lane] = dl[lane + E] = -1.0;
        double bin = !ones && lane < E0 ? btab[my_row + k] : 1.0;
        if (!ones) {  // exact: products of small integers
            bin *= dpp_d<WH_DPP_XOR1>(bin);
            bin *= dpp_d<WH_DPP_XOR2>(bin);
            bin *= dpp_d<WH_DPP_HALF_MIRROR>(bin);
            bin *= dpp_d<WH_DPP_MIRROR>(bin);
            bin *= __shfl_xor(bin, 16, WH_WAVE);  // E0 <= 32: lanes 0..31
        }
        const int par = __popcll(__ballot(k & 1)) & 1;
        double prefac = ((h - par) & 1) ? -bin : bin;
        if (!odd && glynn && __shfl(delta, 0, WH_WAVE) == 0) prefac *= 0.5;
        return prefac;
    };

    if (__syncthreads_or(rough)) {
        auto get = [&](int i, int j) {  // A[i][j] by request index
            const int ie = i < E0 ? i : i - E0 + E, je = j < E0 ? j : j - E0 + E;
            return XA[swp(ie, E) * S + je];
        };
        auto put = [&](int i, int j, cplx v) {
            const int ie = i < E0 ? i : i - E0 + E, je = j < E0 ? j : j - E0 + E;
            XA[swp(ie, E) * S + je] = v;
        };
        double* scale = reinterpret_cast<double*>(Dv + (LOOP ? NP : 0));  // (the first wave's W)
        if ((J.flags & WH_F_NONSYM) || settle_symmetry(n0, odd ? kSymTolOdd : kSymTolEven, scale, get, put)) {
            // p | v | o | e over the wave's slots
            cplx* p = slots;
            cplx* e = slots + (LOOP ? 3 : 1) * PN;
            cplx* out[2] = {slots + PN, slots + 2 * PN};
            const int h0 = J.N / 2;
            for (int64_t t = t0 + wave; t < t1; t += nw) {
                // (h0, not the h with one more edge; the binomials' product is on lanes 0..31 only)
                const double prefac = __shfl(term_factors(t), 0, WH_WAVE) * (odd ? -1.0 : 1.0);
                wave_lds_sync();
                if constexpr (LOOP)
                    full_scalars<2>(get, [&](int j) { return Dg[j]; },
                                    [&](int l, int j) { return l == 0 ? Dg[j] : odd ? V[j] : cmk(0.0, 0.0); }, E0, h0, dl,
                                    Wv, S, Zb, p, out, lane);
                else
                    full_scalars<0>(get, 0, 0, E0, h0, dl, Wv, S, nullptr, p, {nullptr}, lane);
                const cplx f = full_coeff<LOOP>(odd ? J.N : h0, odd, cmk(J.oddloop_re, J.oddloop_im), p, out[0], out[1],
                                                e, lane);
                if (lane == h - 1) acc.add(cmulr(f, prefac));
                wave_lds_sync();
            }
            t1 = t0;  // no term is left
        }
    }

    constexpr bool BREG = T <= 2;  // (where they fit beside the accumulators)
    Bop<T> B[BREG ? 2 * T : 1];
    if constexpr (BREG) {
#pragma unroll
        for (int kc = 0; kc < 2 * T; ++kc)
#pragma unroll
            for (int q = 0; q < T; ++q) B[kc].b[q] = XA[(L.y + 4 * kc) * S + 4 * L.bc + L.x + 8 * q];
    }
    cplx xd[T];
    if (LOOP) {
#pragma unroll
        for (int q = 0; q < T; ++q) xd[q] = Dv[swp(L.cd(q), E)];
    }
    const int nk = (n + 3) / 4;  // k chunks that are not all padding

    int slot = 0;
    for (int64_t t = t0 + wave; t < t1; t += nw) {
        cplx* pt = slots + slot * SL;
        cplx* lv = pt + PN;
        const double prefac = term_factors(t);
        if (lane == 0) pf[slot] = prefac;
        wave_lds_sync();
        double dr[T], dc[T];
#pragma unroll
        for (int p = 0; p < T; ++p) {
            dr[p] = dl[L.rd(p)];
            dc[p] = dl[L.cd(p)];
        }
        const double de = lane < n ? dl[lane < NP ? lane : 0] : 0.0;
        const int es = lane < n ? swp(lane, E) : 0, ee = lane < n ? lane : 0;

        // C_1 = A; W_1 = A Delta
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
        // p_1 = sum_e delta_e A[e][s e]
        cplx to = cmk(0.0, 0.0);
        if (lane < n) to = cmulr(XA[es * S + es], de);
        sym_store<T>(Wv, cR, cI, dr, dc, L);
        if (LOOP) {
            for (int e = lane; e < NP; e += WH_WAVE) Zb[e] = Dv[e];  // z_0 = D
        }
        if (LOOP && odd && lane == 0) lv[1] = cneg(Dv[E - 1]);  // u_1
        wave_lds_sync();
#pragma unroll 1
        for (int a = 1;; ++a) {
            // W_a in LDS, C_a in registers, to = the lane's part of p_(2a-1)
            cplx te = sym_trace<T>(Wv, cR, cI, dr, L, E);
            cplx v0 = cmk(0.0, 0.0), v1 = cmk(0.0, 0.0);
            if (LOOP) {
                cplx* zp = Zb + ((a - 1) & 1) * NP;
                cplx* zc = Zb + (a & 1) * NP;
                sym_matvec<T>(Wv, xd, zc, L);
                wave_lds_sync();
                const cplx f = cmulr(zp[ee], de);
                v0 = cmul(f, zp[es]);  // v_(2a-1)
                v1 = cmul(f, zc[es]);  // v_(2a)
                if (odd) {  // b_(2a-1), b_(2a), u_(2a), u_(2a+1)
                    const double k0 = a - 0.5, k1 = a;
                    to = cmk(fma(k0, v0.re, 0.5 * to.re), fma(k0, v0.im, 0.5 * to.im));
                    te = cmk(fma(k1, v1.re, 0.5 * te.re), fma(k1, v1.im, 0.5 * te.im));
                    const cplx y = cmulr(Wv[es * S + E - 1], de);
                    v0 = cmul(y, zp[ee]);
                    v1 = cmul(y, zc[ee]);
                }
            }
            const double v[8] = {to.re, to.im, te.re, te.im, v0.re, v0.im, v1.re, v1.im};
            const double s = wave_sum8(v, lane);  // lane 8k: value k
            if ((lane & 7) == 0 && (LOOP || lane < 32)) {
                const int kv = lane >> 3;
                cplx* dst = (kv < 4 ? pt : lv + (odd ? 1 : 0)) + 2 * a - 1 + ((kv >> 1) & 1);
                (kv & 1 ? dst->im : dst->re) = s;
            }
            if (a >= Ahalf) break;
            sym_product<T, BREG, !LOOP>(Wv, XA, B, cR, cI, L, nk);
            to = sym_trace<T>(Wv, cR, cI, dr, L, E);  // C_(a+1) with W_a: p_(2a+1)
            wave_lds_sync();
            sym_store<T>(Wv, cR, cI, dr, dc, L);
            wave_lds_sync();
        }
        ++slot;
        if (slot == kSymBatch || t + nw >= t1) {
            wave_lds_sync();
            if (h <= 16) {
                const int m = (lane & 15) + 1, j = lane >> 4;
                const int js = j < slot ? j : 0;
                const cplx* sl = slots + js * SL;
                const cplx bb = series_coeff<LOOP>(sl, PN, h, m, odd);
                cplx s;
                if (LOOP && !odd) s = series_row<false, false>(bb, h);
                else s = series_row<false, true>(bb, h);
                if (LOOP && odd) s = odd_row<16>(s, sl + PN, h, lane);
                if (m == h && j < slot) acc.add(cmulr(s, odd ? pf[j] : pf[j] * kInv.v[h]));
            } else {
                // one term at a time over the wave, lane m - 1 holding s_m (h <= 64)
                for (int j = 0; j < slot; ++j) {
                    const int m = lane + 1;
                    const cplx* sl = slots + j * SL;
                    const cplx b0 = series_coeff<LOOP>(sl, PN, h, m, odd);
                    cplx s = b0, c = cmk(0.0, 0.0);
                    // (two words, as series_steps, and e in two words too: long series cancel more)
                    const bool two = !(LOOP && !odd);
                    for (int kk = 1; kk < h; ++kk) {
                        const cplx eh = cmulr(cmk(__shfl(s.re, kk - 1, WH_WAVE), __shfl(s.im, kk - 1, WH_WAVE)),
                                              kInv.v[kk]);
                        const int src = lane - kk < 0 ? 0 : lane - kk;
                        cplx bs = cmk(__shfl(b0.re, src, WH_WAVE), __shfl(b0.im, src, WH_WAVE));
                        if (lane < kk) bs = cmk(0.0, 0.0);
                        if (!two) {
                            cmac(s, bs, eh);
                            continue;
                        }
                        const cplx el = cmulr(cmk(__shfl(c.re, kk - 1, WH_WAVE), __shfl(c.im, kk - 1, WH_WAVE)),
                                              kInv.v[kk]);
                        mac2(s.re, c.re, bs.re, eh.re, el.re);
                        mac2(s.re, c.re, -bs.im, eh.im, el.im);
                        mac2(s.im, c.im, bs.re, eh.im, el.im);
                        mac2(s.im, c.im, bs.im, eh.re, el.re);
                    }
                    s = cadd(s, c);
                    if (LOOP && odd) s = odd_row<64>(s, sl + PN, h, lane);
                    if (m == h) acc.add(cmulr(s, odd ? pf[j] : pf[j] * kInv.v[h]));
                }
            }
            wave_lds_sync();  // the slots are free again
            slot = 0;
        }
    }

    if constexpr (CALL) {  // the wave's one term (row 0)
        if (lane == h - 1) C.terms[(int64_t)blockIdx.x * nw + wave] = make_double4(acc.sr, acc.cr, acc.si, acc.ci);
        return;
    }
    // the lanes that kept sums (one per 16-lane row, or lane h - 1), then the waves, in order
    if (h <= 16) {
        csum s;
        s.zero();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int src = 16 * j + h - 1;
            const double r = __shfl(acc.sr, src, WH_WAVE), rc = __shfl(acc.cr, src, WH_WAVE);
            const double i = __shfl(acc.si, src, WH_WAVE), ic = __shfl(acc.ci, src, WH_WAVE);
            s.add_pair(r, rc, i, ic);
        }
        if (lane == 0) wres[wave] = make_double4(s.sr, s.cr, s.si, s.ci);
    } else if (lane == h - 1) {
        wres[wave] = make_double4(acc.sr, acc.cr, acc.si, acc.ci);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        csum s;
        s.zero();
        for (int w = 0; w < nw; ++w) {
            const double4 pq = wres[w];
            s.add_pair(pq.x, pq.y, pq.z, pq.w);
        }
        partials[b] = make_double4(s.sr, s.cr, s.si, s.ci);
    }
}

size_t wh_sym_lds_bytes(int T, int nw, bool loop, int H) {
    const size_t NP = 8 * (size_t)T, S = NP + 2;
    return (NP * S + (loop ? NP : 0) + nw * sym_wave_cplx(T, loop, H)) * sizeof(cplx) + kSymBinom * sizeof(double) +
           nw * sizeof(double4);
}

template <int T, bool LOOP, bool CALL>
static hipError_t launch_sym(const wh_job_dev* jobs, int njobs, const void* pool, void* partials, int64_t nblocks,
                             int64_t block_offset, int nw, int H, const wh_call& C, hipStream_t stream) {
    const size_t lds = wh_sym_lds_bytes(T, nw, LOOP, H);
    static wh_lds_limit lim;
    hipError_t err = wh_raise_lds_limit((const void*)wh_sieve_sym<T, LOOP, CALL>, lds, lim);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((wh_sieve_sym<T, LOOP, CALL>), dim3((unsigned)nblocks), dim3(nw * WH_WAVE), lds, stream, jobs,
                       njobs, (const cplx*)pool, (double4*)partials, block_offset, H, C);
    return hipGetLastError();
}

hipError_t wh_launch_sym(int T, bool loop, int H, const wh_job_dev* jobs, int njobs, const void* pool, void* partials,
                         int64_t nblocks, int64_t block_offset, int nw, hipStream_t stream) {
    if (H < 1 || H > WH_NMAX / 2 || nw < 1 || nw > 4) return hipErrorInvalidValue;
    const wh_call C = {};
#define WH_SYM_CASE(TT)                                                                                               \
    case TT:                                                                                                          \
        return loop ? launch_sym<TT, true, false>(jobs, njobs, pool, partials, nblocks, block_offset, nw, H, C, stream) \
                    : launch_sym<TT, false, false>(jobs, njobs, pool, partials, nblocks, block_offset, nw, H, C, stream);
    switch (T) {
        WH_SYM_CASE(1)
        WH_SYM_CASE(2)
        WH_SYM_CASE(3)
        WH_SYM_CASE(4)
        WH_SYM_CASE(5)
        WH_SYM_CASE(6)
        default: return hipErrorInvalidValue;
    }
#undef WH_SYM_CASE
}

int wh_sym_call_terms(int T) { return T <= 3 ? kSymBatch : 0; }

hipError_t wh_launch_sym_call(int T, bool loop, int H, const wh_job_dev* job, const void* pool, void* partials,
                              int64_t nblocks, const wh_call& C, hipStream_t stream) {
    const int nw = C.nw;
    if (H < 1 || H > WH_NMAX / 2 || nw < 1 || nw > 4 || C.nsplit < 1) return hipErrorInvalidValue;
#define WH_SYM_CASE(TT)                                                                                  \
    case TT:                                                                                             \
        return loop ? launch_sym<TT, true, true>(job, 1, pool, partials, nblocks, 0, nw, H, C, stream)   \
                    : launch_sym<TT, false, true>(job, 1, pool, partials, nblocks, 0, nw, H, C, stream);
    switch (T) {
        WH_SYM_CASE(1)
        WH_SYM_CASE(2)
        WH_SYM_CASE(3)
        default: return hipErrorInvalidValue;
    }
#undef WH_SYM_CASE
}
