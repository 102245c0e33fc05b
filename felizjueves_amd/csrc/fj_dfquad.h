// fj_dfquad.h -- the density-fitting integrals (fj_dfloop.h: the formulas, the
// cells, the records) with the class a template parameter and the bra's
// transform on the FP64 matrix cores, for aux shells through g:
//
//   out[ab][(cell, c)] = sum_i sum_p E^{ab}_p(i) T_i[p][(cell, c)]
//   T_i[p][(cell, c)]  = s_k sum_q (-1)^|q| [p + q]_ik E^c_q(k)   (summed over k)
//
// i over the bra's primitive pairs, k over the cell's aux primitives. A
// workgroup of four wavefronts takes CW consecutive cells (and, of those, runs
// with one bra); its wavefronts take different i and work alone until they add
// up their sums. Per i: the bra's E in the wavefront's LDS; per k the cells'
// Hermite towers (levels ordered by the wavefront alone) and T, a lane's
// column fixed (at most four terms an element: the single-centre E^c_q is
// zero unless c - q is even in every direction, and a power of 1 / 2 alpha
// times a whole number); then 16 x 16 tiles of out with p as the summed
// index, kept in the accumulators over i. Tile padding reads valid elements
// and is dropped (rows, columns) or multiplied by a zero A operand (p).
//
// Bound by latency (the Boys seeds and tower levels of a few cells per
// wavefront, which issues VALU instructions in 14 to 21% of its cycles; the
// matrix cores are busy at most 10%) and, for the low classes, by the launch
// itself. Measured on
// MI355X, 9 atoms s,s,p,d with 1,260 aux functions s..g, every class alone, in
// the loop form and here: (mn|P) 33.0 -> 2.6 ms ((dd|g) 9.74 -> 0.21 ms, 45 pairs
// x 36 shells; (ss|s) 0.068 -> 0.038), the metric 0.49 -> 0.36 ms. With the
// wavefronts of a workgroup on different cells of one bra instead of different
// i (101 to 770 workgroups of long lanes) (mn|P) took 10.0 ms.
//
// The includer provides fj_device.h (the device one, or the CPU emulation)
// and fj_dfloop.h.
#pragma once

namespace {

constexpr int DQ_THREADS = 256;
constexpr int DQ_WAVES = 4;
constexpr int DQ_LMAX_AUX = 4;

constexpr int dq_cart(int l) { return (l + 1) * (l + 2) / 2; }
constexpr int dq_herm(int n) { return (n + 1) * (n + 2) * (n + 3) / 6; }
constexpr int dq_up(int n, int d) { return (n + d - 1) / d; }
constexpr int dq_max(int a, int b) { return a > b ? a : b; }

template <int LA, int LB, int LC>
struct Dq {
    static constexpr int NB = dq_cart(LB), NAB = dq_cart(LA) * NB, NC = dq_cart(LC);
    static constexpr int LAB = LA + LB, LT = LAB + LC;
    static constexpr int NT = dq_herm(LAB), NQ = dq_herm(LC), NR = dq_herm(LT);
    // cells of a workgroup: columns (cell, c) filling one or two 16-wide tiles
    static constexpr int CW = LC == 0 ? 8 : LC <= 2 ? 5 : LC == 3 ? 3 : 2;
    static constexpr int N = CW * NC, NTL = dq_up(N, 16), MX = dq_up(NAB, 16), KX = dq_up(NT, 4);
    static constexpr int TB = (LA + 1) * (LB + 1) * (LAB + 1);   // one axis's E
    static constexpr int TERMS = LC >= 4 ? 4 : LC >= 2 ? 2 : 1;
    static constexpr int TS = N | 1;              // row stride of T
    static constexpr bool PAB = NAB * NT <= 2100; // pab in LDS, else ((df|, (ff|) from memory
    static constexpr int UNROLL = KX <= 9 ? KX : 1;   // (the f pairs' steps unrolled spill 1.2 KB a lane)
    struct Lds {
        double eb[DQ_WAVES][3 * TB];
        double r[DQ_WAVES][2 * CW * NR];
        double t[DQ_WAVES][dq_max(NT * TS, 16 * NTL * 4 * MX)];   // at the end, one wavefront's sums
        double seed[DQ_WAVES][CW * (LT + 7)];     // [0]^(m), PQ, s_k (-1)^lc (1/2a)^(lc - m)
        int pab[PAB ? NAB * NT : 1];              // (ab, p): offsets of its three E, 10 bits each
        int tw[NR];                               // the tower's steps
        short add[NT * NQ];                       // the index of p + q
        int b0[CW], b1[CW];                       // the cells' bra records
    };
    // The class's index tables: pab, tw and add, and each component's terms:
    // q, the power m = (lc - |q|) / 2 of 2 alpha, the whole number.
    struct Tab {
        int pab[NAB * NT], tw[NR];
        short add[NT * NQ];
        int n[NC], q[NC][TERMS], m[NC][TERMS];
        double f[NC][TERMS];
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
    // E^i_t of a single centre over (1 / 2 alpha)^((i + t) / 2)
    static constexpr int e1(int i, int t) {
        return t < 0 || t > i ? 0 : i == 0 ? 1 : e1(i - 1, t - 1) + (t + 1) * e1(i - 1, t + 1);
    }
    static constexpr Tab make() {
        const Herm h;
        Tab T = {};
        const int a0 = dq_herm(LA) - dq_cart(LA), b0 = dq_herm(LB) - dq_cart(LB), c0 = NQ - NC;
        for (int r = 0; r < NAB * NT; ++r)
            for (int k = 0; k < 3; ++k)
                T.pab[r] |= ((h.c[a0 + r / NT / NB][k] * (LB + 1) + h.c[b0 + r / NT % NB][k]) * (LAB + 1) + h.c[r % NT][k])
                            << (10 * k);
        for (int j = 1; j < NR; ++j) {
            const int d = h.c[j][0] ? 0 : h.c[j][1] ? 1 : 2, e = h.c[j][d] - 1;
            const int i1 = Herm::at(h.c[j][0] - (d == 0), h.c[j][1] - (d == 1), h.c[j][2] - (d == 2));
            const int i2 = e > 0 ? Herm::at(h.c[j][0] - 2 * (d == 0), h.c[j][1] - 2 * (d == 1), h.c[j][2] - 2 * (d == 2)) : 0;
            T.tw[j] = i1 | (i2 << 10) | (d << 20) | (e << 22);
        }
        for (int r = 0; r < NT * NQ; ++r) {
            const int *p = h.c[r / NQ], *q = h.c[r % NQ];
            T.add[r] = (short)Herm::at(p[0] + q[0], p[1] + q[1], p[2] + q[2]);
        }
        for (int c = 0; c < NC; ++c)
            for (int q = 0; q < NQ; ++q) {
                const int *x = h.c[c0 + c], *y = h.c[q];
                if ((x[0] - y[0]) % 2 || (x[1] - y[1]) % 2 || (x[2] - y[2]) % 2) continue;
                const int f = e1(x[0], y[0]) * e1(x[1], y[1]) * e1(x[2], y[2]);
                if (f == 0) continue;
                T.q[c][T.n[c]] = q;
                T.m[c][T.n[c]] = (LC - y[0] - y[1] - y[2]) / 2;
                T.f[c][T.n[c]++] = f;
            }
        return T;
    }
};

template <int LA, int LB, int LC>
__device__ const typename Dq<LA, LB, LC>::Tab dq_tab = Dq<LA, LB, LC>::make();

// One axis's E^{ij}_t, row i: raised in i from E^{00}_0 = f, then along j.
template <int L1, int L2>
__device__ __forceinline__ void dq_rows(double* __restrict__ e_, int i, double zeta, double pa, double pb, double f) {
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
            for (int t = 0; t <= T; ++t) e_[(i * (L2 + 1) + (r - L1)) * (T + 1) + t] = e[t];
        }
#pragma unroll
        for (int t = 0; t <= T; ++t) {
            const double v = x * e[t] + (double)(t + 1) * e[t + 1] + h * below;
            below = e[t];
            e[t] = up && r >= i ? e[t] : v;
        }
    }
#pragma unroll
    for (int t = 0; t <= T; ++t) e_[(i * (L2 + 1) + L2) * (T + 1) + t] = e[t];
}

}  // namespace

// Cells blockIdx.x CW .. + CW - 1. Every __syncthreads sits in control
// flow uniform over the workgroup; the matrix cores' steps and fj_wave_sync in
// control flow uniform over the wavefront.
template <int LA, int LB, int LC>
__global__ void __launch_bounds__(DQ_THREADS, (LA + LB >= 5 ? 1 : 2)) fj_dfquad_k(FjDfArgs g) {
    typedef Dq<LA, LB, LC> Q;
    constexpr int NAB = Q::NAB, NC = Q::NC, NB = Q::NB, NT = Q::NT, NR = Q::NR, LT = Q::LT, CW = Q::CW, N = Q::N;
    constexpr int NTL = Q::NTL, MX = Q::MX, KX = Q::KX, TB = Q::TB, TS = Q::TS, SS = LT + 7;
    __shared__ typename Q::Lds S;
    const typename Q::Tab& T = dq_tab<LA, LB, LC>;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, l4 = lane >> 4;
    double* const R0 = S.r[wave];
    double* const R1 = S.r[wave] + CW * NR;
    double* const seed = S.seed[wave];
    double* const eb = S.eb[wave];
    double* const tt = S.t[wave];
    if constexpr (Q::PAB)
        for (int r = tid; r < NAB * NT; r += DQ_THREADS) S.pab[r] = T.pab[r];
    const int* const pab = Q::PAB ? S.pab : T.pab;
    for (int r = tid; r < NR; r += DQ_THREADS) S.tw[r] = T.tw[r];
    for (int r = tid; r < NT * Q::NQ; r += DQ_THREADS) S.add[r] = T.add[r];
    const int c0 = (int)blockIdx.x * CW, nc = min(CW, g.n_cell - c0);
    if (tid < nc) {
        S.b0[tid] = g.b_rec0[c0 + tid];
        S.b1[tid] = g.b_rec1[c0 + tid];
    }
    // this lane's column of T and its terms
    constexpr int NP = 16 * NTL;
    static_assert(NP <= 64 && 64 % NP == 0, "columns of T");
    const int col0 = lane % NP, cell0 = min(col0, N - 1) / NC, comp0 = min(col0, N - 1) % NC;
    int tq[Q::TERMS], tm[Q::TERMS];
    double tf[Q::TERMS];
#pragma unroll
    for (int t = 0; t < Q::TERMS; ++t) {   // (a missing term is zero times the first q's integral)
        tq[t] = T.q[comp0][t];
        tm[t] = T.m[comp0][t];
        tf[t] = T.f[comp0][t];
    }
    __syncthreads();
    for (int r0 = 0; r0 < nc;) {
        // a run of cells with one bra
        const int i0 = S.b0[r0], i1 = S.b1[r0], f0 = c0 + r0;
        int r1 = r0 + 1;
        while (r1 < nc && S.b0[r1] == i0 && S.b1[r1] == i1) ++r1;
        const int mine = r1 - r0;
        fj_v4d acc[MX][NTL];
#pragma unroll
        for (int m = 0; m < MX; ++m)
#pragma unroll
            for (int n = 0; n < NTL; ++n) acc[m][n] = fj_v4d{0.0, 0.0, 0.0, 0.0};
        // the most aux primitives of the run's cells, and one of them
        int nk = 0, some = 0;
        for (int c = 0; c < mine; ++c) {
            const int k0 = g.k_rec0[f0 + c], n = g.k_rec1[f0 + c] - k0;
            if (n > nk) {
                nk = n;
                some = k0;
            }
        }
        for (int i = nk ? i0 + wave : i1; i < i1; i += DQ_WAVES) {   // uniform over the wavefront
            const double p = g.zeta[i], Px = g.P[3 * i], Py = g.P[3 * i + 1], Pz = g.P[3 * i + 2];
            if (lane < 3 * (LA + 1)) {
                const int k = lane / (LA + 1);
                const double pa = g.XPA ? g.XPA[3 * i + k] : 0.0, pb = g.XPB ? g.XPB[3 * i + k] : 0.0;
                dq_rows<LA, LB>(eb + k * TB, lane - k * (LA + 1), p, pa, pb, exp(p * pa * pb) * (k == 0 ? g.s_bra[i] : 1.0));
            }
            for (int k = 0; k < nk; ++k) {
                if (lane < CW) {   // a cell past the run's, or out of primitives: zeros
                    const int cell = f0 + min(lane, mine - 1), k0 = g.k_rec0[cell];
                    const bool in = lane < mine && k0 + k < g.k_rec1[cell];
                    const int kk = in ? k0 + k : some;
                    const double a = g.alpha[kk], rho = p * a / (p + a);
                    const double x = Px - g.A[3 * kk], y = Py - g.A[3 * kk + 1], z = Pz - g.A[3 * kk + 2];
                    double* const w = seed + lane * SS;
                    double Fm[LT + 1];
                    fj_boys<LT>(rho * (x * x + y * y + z * z), Fm);
                    double wm = in ? FJ_TWO_OVER_SQRT_PI * sqrt(rho) : 0.0;
#pragma unroll
                    for (int m = 0; m <= LT; ++m) {
                        w[m] = wm * Fm[m];
                        wm *= -2.0 * rho;
                    }
                    w[LT + 1] = x;
                    w[LT + 2] = y;
                    w[LT + 3] = z;
                    // s (-1)^|q| (1/2a)^(lc - m), |q| = lc - 2 m: one sign for every m
                    const double h = -0.5 / a;
                    double f = g.s_aux[kk];
#pragma unroll
                    for (int m = 0; m < LC; ++m) f *= h;
                    w[LT + 4] = f;
                    w[LT + 5] = f * (2.0 * a);
                    w[LT + 6] = f * (2.0 * a) * (2.0 * a);
                    ((LT & 1) ? R1 : R0)[lane * NR] = w[LT];
                }
                fj_wave_sync();
#pragma unroll
                for (int m = LT - 1; m >= 0; --m) {
                    double* __restrict__ cur = (m & 1) ? R1 : R0;
                    const double* __restrict__ prv = (m & 1) ? R0 : R1;
                    const int n_m = dq_herm(LT - m);
                    for (int r = lane; r < CW * n_m; r += 64) {
                        const int c = r / n_m, j = r - c * n_m;
                        const double* __restrict__ w = seed + c * SS;
                        double v;
                        if (j == 0) {
                            v = w[m];
                        } else {
                            const int t = S.tw[j], c1 = t >> 22;
                            v = w[LT + 1 + ((t >> 20) & 3)] * prv[c * NR + (t & 1023)];
                            if (c1 > 0) v += (double)c1 * prv[c * NR + ((t >> 10) & 1023)];
                        }
                        cur[c * NR + j] = v;
                    }
                    fj_wave_sync();
                }
                // T: a lane's column, rows p in turn, added over the aux primitives
                double cf[Q::TERMS];
#pragma unroll
                for (int t = 0; t < Q::TERMS; ++t) cf[t] = tf[t] * seed[cell0 * SS + LT + 4 + tm[t]];
                const double* __restrict__ R = R0 + cell0 * NR;
                for (int pp = lane / NP; pp < NT; pp += 64 / NP) {
                    double v = 0.0;
#pragma unroll
                    for (int t = 0; t < Q::TERMS; ++t) v += cf[t] * R[S.add[pp * Q::NQ + tq[t]]];
                    if (col0 < N) tt[pp * TS + col0] = k ? tt[pp * TS + col0] + v : v;
                }
                fj_wave_sync();
            }
            // out += E T
#pragma unroll Q::UNROLL
            for (int ks = 0; ks < KX; ++ks) {
                const int pp = 4 * ks + l4, pc = min(pp, NT - 1);
                double bv[NTL];
#pragma unroll
                for (int n = 0; n < NTL; ++n) bv[n] = tt[pc * TS + min(16 * n + l16, N - 1)];
#pragma unroll
                for (int m = 0; m < MX; ++m) {
                    const int o = pab[min(16 * m + l16, NAB - 1) * NT + pc];
                    const double v = eb[o & 1023] * eb[TB + ((o >> 10) & 1023)] * eb[2 * TB + (o >> 20)];
                    const double av = pp < NT ? v : 0.0;
#pragma unroll
                    for (int n = 0; n < NTL; ++n) acc[m][n] = fj_mfma_f64_16x16x4(av, bv[n], acc[m][n]);
                }
            }
            fj_wave_sync();   // before the next tables
        }
        // the wavefronts' sums, in turn into the first's (a wavefront past the
        // bra's primitives has none)
        double* const sum = &S.t[0][0];
        for (int w = 1; w < min(DQ_WAVES, i1 - i0); ++w) {   // uniform over the workgroup
            __syncthreads();
            if (wave == w) {
#pragma unroll
                for (int x = 0; x < MX * NTL * 4; ++x) sum[x * 64 + lane] = acc[x / 4 / NTL][x / 4 % NTL][x % 4];
            }
            __syncthreads();
            if (wave == 0) {
#pragma unroll
                for (int x = 0; x < MX * NTL * 4; ++x) acc[x / 4 / NTL][x / 4 % NTL][x % 4] += sum[x * 64 + lane];
            }
        }
        __syncthreads();   // before a next run's T
        if (wave != 0) {
            r0 = r1;
            continue;
        }
        // the scatter, mirrored; a diagonal cell writes its lower triangle
#pragma unroll
        for (int n = 0; n < NTL; ++n) {
            const int col = 16 * n + l16, c = col / NC, cc = col - c * NC;
            if (col >= N || c >= mine) continue;   // (no barrier below)
            const int cell = f0 + c, oa = g.off_a[cell], oc = g.off_c[cell];
            const size_t nx = (size_t)g.n_aux;
#pragma unroll
            for (int m = 0; m < MX; ++m)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int ab = 16 * m + l4 + 4 * v, a = ab / NB, b = ab - a * NB;
                    if (ab >= NAB) continue;
                    const double x = acc[m][n][v];
                    if (g.mode == 0) {
                        const int ob = g.off_b[cell];
                        if (oa == ob && a < b) continue;
                        const size_t na = (size_t)g.n_ao;
                        g.out[((oa + a) * na + ob + b) * nx + oc + cc] = x;
                        g.out[((ob + b) * na + oa + a) * nx + oc + cc] = x;
                    } else {
                        if (oa == oc && a < cc) continue;
                        g.out[(oa + a) * nx + oc + cc] = x;
                        g.out[(oc + cc) * nx + oa + a] = x;
                    }
                }
        }
        r0 = r1;
    }
}
