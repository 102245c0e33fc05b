// fj_fquad.h -- the fused F kernel of the classes with an f shell
// (fj_floop.h: the formulas; fj_fitem.h: items, screen, digestion) with the
// class a template parameter, the sums over primitives in the matrix cores'
// accumulators and one digestion per ket. With i over the bra's primitive
// pairs and j over the ket's,
//
//   V_j[q][ab] = sum_i sum_p [p + q]_ij E^{ab}_p(i)         16 x 16 tiles over p
//   x[cd][ab] += sum_q (-1)^|q| E^{cd}_q(j) V_j[q][ab]      16 x 16 tiles over q
//
// V's accumulators are the second product's B operand as they stand (element
// v of a lane is row l / 16 + 4 v, the row that step v of the product wants
// from it), so V never leaves the registers, and x is formed once per j, not
// once per primitive quartet. The E products are formed from the axis tables
// in LDS as they are needed; [p + q] is gathered from the tower.
//
// A workgroup of four wavefronts takes a work item's kets one after another.
// Each wavefront holds one ab tile: up to 16 bra functions it works alone (its
// own E tables and towers; the four take different j, or different i where a
// ket has fewer j), up to 32 two share a tower and up to 64 four, and the 100
// of (ff| go to two workgroups. (With two ab tiles to a wavefront their
// accumulators leave room for one workgroup on a CU: (ff|ff) 2.77 ms against
// 1.81, (df|ff) 2.02 against 1.06.) At the end of a ket x goes through LDS 16
// bra functions at a time, lanes over (ab, c), (ab, d) and cd, each summing
// over the other ket function, so a lane adds into an F block once per sum,
// not per element.
//
// Padding reads a valid element: rows and columns of it are dropped, the
// summed index is multiplied by zero (bit 30 of a table entry).
//
// Bound, for the d and f pairs, by the matrix cores and the FP64 instructions
// that form their operands ((ff|ff): 7.4 VALU instructions a step, the cores busy
// 27% of the time), for the low classes by the latency of a workgroup (Boys
// function, tower levels, digestion) and by new code for every launch. Measured
// on MI355X, 4 atoms s,s,p,d,f, 4 streams, 18,274 quartets (1.3 million
// primitive quartets with an f): the build 38.0 -> 9.7 ms; another of 4 atoms
// with longer contractions, one stream, 36.6 -> 9.0 ms; one atom 2.1 -> 1.9 ms.
//
// The includer provides fj_device.h (the device one, or the CPU emulation).
#pragma once
#include "fj_fitem.h"

namespace {

constexpr int FQ_THREADS = 256;

constexpr int fq_cart(int l) { return (l + 1) * (l + 2) / 2; }
constexpr int fq_herm(int n) { return (n + 1) * (n + 2) * (n + 3) / 6; }   // |t| <= n
constexpr int fq_up(int n, int d) { return (n + d - 1) / d; }
constexpr int fq_max(int a, int b) { return a > b ? a : b; }

template <int LA, int LB, int LC, int LD>
struct Fq {
    static constexpr int NA = fq_cart(LA), NB = fq_cart(LB), NC = fq_cart(LC), ND = fq_cart(LD);
    static constexpr int NAB = NA * NB, NCD = NC * ND, LAB = LA + LB, LCD = LC + LD, L = LAB + LCD;
    static constexpr int NP = fq_herm(LAB), NQ = fq_herm(LCD), NR = fq_herm(L);
    // tiles of q, ab and cd; wavefronts that share a tower, one ab tile each;
    // workgroups that share a ket, four ab tiles each
    static constexpr int MV = fq_up(NQ, 16), MN = fq_up(NAB, 16), MX = fq_up(NCD, 16);
    static constexpr int WT = MN == 1 ? 1 : MN == 2 ? 2 : 4, G = 4 / WT, Z = fq_up(MN, 4);
    static constexpr int KP = fq_up(NP, 4), KQ = fq_up(NQ, 4);
    // bra primitives of a step: their Boys functions and tower levels overlap
    static constexpr int IB = WT == 1 ? (NR <= 56 ? 8 : NR <= 165 ? 4 : 2) : 4;
    static constexpr int TB = (LA + 1) * (LB + 1) * (LAB + 1), TK = (LC + 1) * (LD + 1) * (LCD + 1);
    static constexpr int XS = NCD | 1;
    static constexpr int BLK = NAB + NCD + NA * NC + NA * ND + NB * NC + NB * ND;
    // Steps of V unrolled where a bra has many (4 atoms 13.7 -> 12.4 ms); for
    // the low classes, whose launches are short, new code costs more than it
    // gives (2 atoms, one stream, 8.0 -> 8.5 ms with every class unrolled).
    static constexpr int UNROLL = KP >= 9 ? 2 : 1;
    // table widths
    static constexpr int PW = 16 * WT * Z, QW = 16 * MV, CW = 16 * MX;
    struct Lds {
        double eb[G][IB * 3 * TB];
        double ek[G][3 * TK];
        double r[fq_max(G * 2 * IB * NR, 16 * XS)];   // towers; 16 bra functions of x
        double seed[G][IB * (L + 4)];                 // [0]^(m), PQ
        double w[BLK], f[BLK];
        int tw[NR];
    };
    // pb (p, ab) and pc (q, cd): offsets of the three E, 10 bits each, and the
    // padding's zero; ad: the index of p + q; tw: the tower's steps.
    struct Tab {
        int pb[4 * KP * PW], pc[4 * KQ * CW], tw[NR];
        short ad[4 * KP * QW];
    };
    struct Herm {
        int c[NR][3];
        constexpr Herm() : c() {
            int k = 0;
            for (int n = 0; k < NR; ++n)
                for (int x = n; x >= 0; --x)
                    for (int y = n - x; y >= 0; --y, ++k) {
                        c[k][0] = x;
                        c[k][1] = y;
                        c[k][2] = n - x - y;
                    }
        }
        static constexpr int at(int x, int y, int z) {
            return (x + y + z) * (x + y + z + 1) * (x + y + z + 2) / 6 + (y + z) * (y + z + 1) / 2 + z;
        }
    };
    static constexpr int entry(const Herm& h, int l1, int l2, int ij, int t) {
        const int n2 = fq_cart(l2), a = fq_herm(l1) - fq_cart(l1) + ij / n2, b = fq_herm(l2) - fq_cart(l2) + ij % n2;
        int v = 0;
        for (int k = 0; k < 3; ++k)
            v |= ((h.c[a][k] * (l2 + 1) + h.c[b][k]) * (l1 + l2 + 1) + h.c[t][k]) << (10 * k);
        return v;
    }
    static constexpr Tab make() {
        const Herm h;
        Tab T = {};
        for (int p = 0; p < 4 * KP; ++p) {
            const int t = p < NP ? p : NP - 1;
            for (int ab = 0; ab < PW; ++ab)
                T.pb[p * PW + ab] = entry(h, LA, LB, ab < NAB ? ab : NAB - 1, t) | (p < NP ? 0 : 1 << 30);
            for (int q = 0; q < QW; ++q) {
                const int *x = h.c[t], *y = h.c[q < NQ ? q : NQ - 1];
                T.ad[p * QW + q] = (short)Herm::at(x[0] + y[0], x[1] + y[1], x[2] + y[2]);
            }
        }
        for (int q = 0; q < 4 * KQ; ++q) {
            const int t = q < NQ ? q : NQ - 1;
            for (int cd = 0; cd < CW; ++cd)
                T.pc[q * CW + cd] = entry(h, LC, LD, cd < NCD ? cd : NCD - 1, t) | (q < NQ ? 0 : 1 << 30);
        }
        for (int j = 1; j < NR; ++j) {
            const int d = h.c[j][0] ? 0 : h.c[j][1] ? 1 : 2, e = h.c[j][d] - 1;
            const int i1 = Herm::at(h.c[j][0] - (d == 0), h.c[j][1] - (d == 1), h.c[j][2] - (d == 2));
            const int i2 = e > 0 ? Herm::at(h.c[j][0] - 2 * (d == 0), h.c[j][1] - 2 * (d == 1), h.c[j][2] - 2 * (d == 2)) : 0;
            T.tw[j] = i1 | (i2 << 10) | (d << 20) | (e << 22);
        }
        return T;
    }
};

template <int LA, int LB, int LC, int LD>
__device__ const typename Fq<LA, LB, LC, LD>::Tab fq_tab = Fq<LA, LB, LC, LD>::make();

// One axis's E^{ij}_t, row i: raised in i from E^{00}_0 = f, then along j.
// ODD: with the sign (-1)^t.
template <int L1, int L2, bool ODD>
__device__ __forceinline__ void fq_rows(double* __restrict__ e_, int i, double zeta, double pa, double pb, double f) {
    constexpr int T = L1 + L2;
    const double h = 0.5 / zeta;
    double e[T + 2];
#pragma unroll
    for (int t = 0; t <= T + 1; ++t) e[t] = t == 0 ? f : 0.0;
#pragma unroll
    for (int r = 0; r < L1 + L2; ++r) {
        const bool up = r < L1;
        const double x = up ? pa : pb;
        double below = 0.0;
        if (!up) {
#pragma unroll
            for (int t = 0; t <= T; ++t) e_[(i * (L2 + 1) + (r - L1)) * (T + 1) + t] = ODD && t % 2 ? -e[t] : e[t];
        }
#pragma unroll
        for (int t = 0; t <= T; ++t) {
            const double v = x * e[t] + (double)(t + 1) * e[t + 1] + h * below;
            below = e[t];
            e[t] = up && r >= i ? e[t] : v;
        }
    }
#pragma unroll
    for (int t = 0; t <= T; ++t) e_[(i * (L2 + 1) + L2) * (T + 1) + t] = ODD && t % 2 ? -e[t] : e[t];
}

// The E product of a pb or pc entry; PAD: the table has padding.
template <int T, bool PAD>
__device__ __forceinline__ double fq_value(const double* __restrict__ e, int o) {
    const double v = e[o & 1023] * e[T + ((o >> 10) & 1023)] * e[2 * T + (PAD ? (o >> 20) & 1023 : o >> 20)];
    return PAD && (o & (1 << 30)) ? 0.0 : v;
}

}  // namespace

// Work items as fj_floop_k's. Every __syncthreads sits in control flow uniform
// over the workgroup; the matrix cores' steps and fj_wave_sync in control flow
// uniform over the wavefront.
template <int LA, int LB, int LC, int LD>
__global__ void __launch_bounds__(FQ_THREADS, 2) fj_fquad_k(int span, FjFArgs a) {
    typedef Fq<LA, LB, LC, LD> Q;
    constexpr int NA = Q::NA, NB = Q::NB, NC = Q::NC, ND = Q::ND, NAB = Q::NAB, NCD = Q::NCD, L = Q::L;
    constexpr int NP = Q::NP, NQ = Q::NQ, NR = Q::NR, MV = Q::MV, MN = Q::MN, MX = Q::MX, KP = Q::KP;
    constexpr int WT = Q::WT, G = Q::G, GL = 64 * WT, IB = Q::IB, TB = Q::TB, TK = Q::TK, XS = Q::XS;
    __shared__ typename Q::Lds S;
    const typename Q::Tab& T = fq_tab<LA, LB, LC, LD>;
    FjFlItem it;
    if (!fj_fl_item(a, span, it)) return;   // uniform
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, l4 = lane >> 4;
    const int grp = wave / WT, wt = wave % WT, gl = wt * 64 + lane;
    const int tile0 = 4 * (int)blockIdx.z;   // the workgroup's first ab tile
    double* const R0 = S.r + grp * 2 * IB * NR;
    double* const R1 = R0 + IB * NR;
    double* const seed = S.seed[grp];
    double* const eb = S.eb[grp];
    double* const ek = S.ek[grp];
    double* const xs = S.r;
    // the lanes that share a tower meet
    auto meet = [] {
        if constexpr (WT == 1) fj_wave_sync();
        else __syncthreads();
    };
    for (int r = tid; r < NR; r += FQ_THREADS) S.tw[r] = T.tw[r];
    FjFlBlocks blk;
    {
        const int n[6] = {NAB, NCD, NA * NC, NA * ND, NB * NC, NB * ND};
        int at = 0;
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            blk.w[i] = S.w + at;
            blk.f[i] = S.f + at;
            at += n[i];
        }
    }
    const int bra = it.bra, kab = it.kab;
    const int sa = a.bra.sh[2 * bra], sb = a.bra.sh[2 * bra + 1];
    const int oa = a.bra.ao[2 * bra], ob = a.bra.ao[2 * bra + 1];
    const double Gb = a.bra.G[bra];
    const double* __restrict__ bp = a.bra.prim + 8 * (size_t)it.kb0;
    __syncthreads();

    for (int kk = it.k0; kk < it.k1; ++kk) {
        FjFlKet q;
        if (!fj_fl_ket(a, it, kk, sa, sb, Gb, q)) continue;   // uniform
        const int kcd = q.kcd;
        const double* __restrict__ kp = a.ket.prim + 8 * (size_t)q.kc0;
        fj_fl_load(blk, it.S.D, it.S.n_ao, oa, ob, q.oc, q.od, NA, NB, NC, ND, q.s_j, q.s_k, tid, FQ_THREADS);
        fj_v4d x[MX];
#pragma unroll
        for (int m = 0; m < MX; ++m) x[m] = fj_v4d{0.0, 0.0, 0.0, 0.0};
        // groups over j, and over i where there are fewer j than groups
        const int WJ = min(G, kcd), WI = G / WJ, gj = grp % WJ, gi = grp / WJ;
        for (int jb = 0; jb < kcd; jb += WJ) {
            const int j = jb + gj;
            const bool jv = j < kcd && gi < WI;
            const double* __restrict__ rk = kp + 8 * (jv ? j : 0);
            const double qz = rk[6], Qx = rk[0], Qy = rk[1], Qz = rk[2];
            if (gl < 3 * (LC + 1)) {
                const int k = gl / (LC + 1);
                const double cd = LD ? a.ket.sep[3 * q.k + k] : 0.0;
                fq_rows<LC, LD, true>(ek + k * TK, gl - k * (LC + 1), qz, rk[3 + k], rk[3 + k] + cd, k == 0 ? rk[7] : 1.0);
            }
            fj_v4d V[MV];
#pragma unroll
            for (int m = 0; m < MV; ++m) V[m] = fj_v4d{0.0, 0.0, 0.0, 0.0};
            for (int i0 = 0; i0 < kab; i0 += WI * IB) {
                const int ib = i0 + gi * IB, nb = jv ? max(min(kab - ib, IB), 0) : 0;   // uniform over the group
                for (int r = gl; r < nb * 3 * (LA + 1); r += GL) {
                    const int bk = r / (LA + 1), b = bk / 3, k = bk - 3 * b;
                    const double* __restrict__ rb = bp + 8 * (ib + b);
                    const double sep = LB ? a.bra.sep[3 * bra + k] : 0.0;
                    fq_rows<LA, LB, false>(eb + bk * TB, r - bk * (LA + 1), rb[6], rb[3 + k], rb[3 + k] + sep, k == 0 ? rb[7] : 1.0);
                }
                if (wt == WT - 1 && lane < nb) {
                    const double* __restrict__ rb = bp + 8 * (ib + lane);
                    const double p = rb[6], PQx = rb[0] - Qx, PQy = rb[1] - Qy, PQz = rb[2] - Qz;
                    const double rho = p * qz / (p + qz);
                    double* const w = seed + lane * (L + 4);
                    double Fm[L + 1];
                    fj_boys<L>(rho * (PQx * PQx + PQy * PQy + PQz * PQz), Fm);
                    double wm = FJ_TWO_OVER_SQRT_PI * sqrt(rho);
#pragma unroll
                    for (int m = 0; m <= L; ++m) {
                        w[m] = wm * Fm[m];
                        wm *= -2.0 * rho;
                    }
                    w[L + 1] = PQx;
                    w[L + 2] = PQy;
                    w[L + 3] = PQz;
                    ((L & 1) ? R1 : R0)[lane * NR] = w[L];
                }
                meet();
#pragma unroll
                for (int m = L - 1; m >= 0; --m) {
                    double* __restrict__ cur = (m & 1) ? R1 : R0;
                    const double* __restrict__ prv = (m & 1) ? R0 : R1;
                    const int n_m = fq_herm(L - m);
                    for (int r = gl; r < nb * n_m; r += GL) {
                        const int b = r / n_m, h = r - b * n_m;
                        const double* __restrict__ w = seed + b * (L + 4);
                        double v;
                        if (h == 0) {
                            v = w[m];
                        } else {
                            const int t = S.tw[h], c1 = t >> 22;
                            v = w[L + 1 + ((t >> 20) & 3)] * prv[b * NR + (t & 1023)];
                            if (c1 > 0) v += (double)c1 * prv[b * NR + ((t >> 10) & 1023)];
                        }
                        cur[b * NR + h] = v;
                    }
                    meet();
                }
                if constexpr (NP == 1) {   // one p: four i a step
                    for (int s = 0; s < nb; s += 4) {
                        const int b = min(s + l4, nb - 1);
                        const double e = eb[b * 3] * eb[b * 3 + 1] * eb[b * 3 + 2], bv = s + l4 < nb ? e : 0.0;
#pragma unroll
                        for (int m = 0; m < MV; ++m)
                            V[m] = fj_mfma_f64_16x16x4(R0[b * NR + min(16 * m + l16, NQ - 1)], bv, V[m]);
                    }
                } else {
                    for (int b = 0; b < nb; ++b) {
                        const double* __restrict__ R = R0 + b * NR;
                        const double* __restrict__ e = eb + b * 3 * TB;
#pragma unroll Q::UNROLL
                        for (int ks = 0; ks < KP; ++ks) {
                            const int p = 4 * ks + l4;
                            const short* __restrict__ ad = T.ad + p * Q::QW + l16;
                            const double bv = fq_value<TB, NP % 4 != 0>(e, T.pb[p * Q::PW + 16 * (tile0 + wt) + l16]);
#pragma unroll
                            for (int m = 0; m < MV; ++m) V[m] = fj_mfma_f64_16x16x4(R[ad[16 * m]], bv, V[m]);
                        }
                    }
                }
                meet();   // before the next tables
            }
            if (jv) {
#pragma unroll
                for (int m = 0; m < MV; ++m)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        if (16 * m + 4 * v >= NQ) continue;   // steps past every q
                        const int* __restrict__ pc = T.pc + (16 * m + 4 * v + l4) * Q::CW + l16;
#pragma unroll
                        for (int c = 0; c < MX; ++c) x[c] = fj_mfma_f64_16x16x4(fq_value<TK, NQ % 4 != 0>(ek, pc[16 * c]), V[m][v], x[c]);
                    }
            }
            meet();   // before the next j's tables
        }
        // the six blocks, 16 bra functions at a time
        __syncthreads();   // the towers are free, w is loaded
        for (int o = 0; o < WT; ++o) {
            const int ab0 = 16 * (tile0 + o), nr = min(16, NAB - ab0);
            if (nr <= 0) break;
            for (int g = 0; g < WJ * WI; ++g) {   // the groups' sums in turn
                if (grp == g && wt == o) {
#pragma unroll
                    for (int c = 0; c < MX; ++c)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const int cd = 16 * c + l4 + 4 * v;
                            if (cd < NCD) xs[l16 * XS + cd] = g ? xs[l16 * XS + cd] + x[c][v] : x[c][v];
                        }
                }
                __syncthreads();
            }
            for (int r = tid; r < nr * (NC + ND) + NCD; r += FQ_THREADS) {
                if (r < nr * NC) {
                    const int i = r / NC, c = r - i * NC, ab = ab0 + i, ia = ab / NB, jb = ab - ia * NB;
                    const double* __restrict__ xr = xs + i * XS + c * ND;
                    double sj = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
                    for (int d = 0; d < ND; ++d) {
                        sj += xr[d] * blk.w[1][c * ND + d];
                        s1 += xr[d] * blk.w[5][jb * ND + d];
                        s2 += xr[d] * blk.w[3][ia * ND + d];
                    }
                    atomicAdd(&blk.f[0][ab], sj);
                    atomicAdd(&blk.f[2][ia * NC + c], s1);
                    atomicAdd(&blk.f[4][jb * NC + c], s2);
                } else if (r < nr * (NC + ND)) {
                    const int k = r - nr * NC, i = k / ND, d = k - i * ND, ab = ab0 + i, ia = ab / NB, jb = ab - ia * NB;
                    const double* __restrict__ xr = xs + i * XS + d;
                    double s1 = 0.0, s2 = 0.0;
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        s1 += xr[c * ND] * blk.w[4][jb * NC + c];
                        s2 += xr[c * ND] * blk.w[2][ia * NC + c];
                    }
                    atomicAdd(&blk.f[3][ia * ND + d], s1);
                    atomicAdd(&blk.f[5][jb * ND + d], s2);
                } else {
                    const int cd = r - nr * (NC + ND);
                    double s = 0.0;
                    for (int i = 0; i < nr; ++i) s += xs[i * XS + cd] * blk.w[0][ab0 + i];
                    blk.f[1][cd] += s;   // one lane per cd
                }
            }
            __syncthreads();
        }
        // the ket's six blocks into F (the caller closes F + F^T)
        fj_fl_flush(blk, it.S.F, it.S.n_ao, oa, ob, q.oc, q.od, NA, NB, NC, ND, tid, FQ_THREADS);
        __syncthreads();   // before the next ket rewrites the blocks
    }
}
