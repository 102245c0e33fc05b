// fj_gfquad.h -- the fused two-electron gradient (fj_gfloop.h: the weights,
// the stream, the formulas) with the class a template parameter and every
// contraction over primitives and Hermite indices on the FP64 matrix cores.
//
// A workgroup of four wavefronts takes a quartet (or a range of its primitive
// quartets). With i over the bra's primitive pairs and j over the ket's,
//
//   Wk_j[ab][u] = (-1)^|u| sum_cd w E^{cd}_u(j)       once per j and wavefront
//   Wb_i[cd][t] = sum_ab w E^{ab}_t(i)                once per i and pass over j
//   Y_ij[ab][t] = sum_u Wk_j[ab][u] [t + u]_ij        gA, gB += sum dE^{ab}_t(i) Y_ij
//   X_j[cd][u] += sum_i sum_t Wb_i[cd][t] [t + u]_ij  gC, gD once per j
//
// (all four centres: taking one of them from the others would put into it the
// residue 2 zeta (rounding of P) that the records' P leaves in their sum, 1e-10
// of the 8-atom gradient). The weights' transforms are shared by a quartet's
// primitives and X is summed over i in the accumulators, where the loop form
// forms all of it per primitive quartet: at (dd|dd) about 300 thousand
// operations per primitive quartet are left, nearly all in the two products
// with [t + u]. A pass is four j (one per wavefront). A quartet cut into
// pieces (few quartets) is cut into ranges of j first, then of i.
//
// Wavefronts take different j (or, for one or two j, different i); the i are
// taken IB at a time: their E tables and Wb by the workgroup, then each
// wavefront, IBW of them at a time, their Hermite towers in its own LDS
// (levels ordered by the wavefront alone), X and Y. [t + u] is gathered from
// the tower as the matrix cores' B operand, at offsets that are the same in
// every step and stay packed in registers; columns are (i, t) pairs, so the
// low classes fill the 16 x 16 tiles with several i. The padding of a tile
// reads a valid element and its result is dropped (rows and columns) or is
// multiplied by a zero A operand (the summed index).
//
// Measured on MI355X, every class of the s,s,p,d 8-atom gradient alone (29.8
// million primitive quartets): 666 ms in the loop form, 54 ms here, and 22.3
// -> 3.0 ms for the three-atom one; e.g. (dd|dd) 32.2 -> 4.8 ms, (sp|dd) 75.8
// -> 2.8 ms, (ss|sp) 4.8 -> 1.1 ms. The matrix cores are busy 11 to 27% of the
// time of the classes with a d shell in the ket; to each matrix step come 8 to
// 44 VALU instructions of the towers and the last stage (9 at (dd|dd)), and the
// wavefronts wait in 14 to 28% of their cycles.
//
// The includer provides fj_device.h (the device one, or the CPU emulation)
// and fj_gfloop.h.
#pragma once

namespace {

constexpr int GQ_THREADS = 256;
constexpr int GQ_WAVES = 4;

constexpr int gq_cart(int l) { return (l + 1) * (l + 2) / 2; }
constexpr int gq_herm(int n) { return (n + 1) * (n + 2) * (n + 3) / 6; }   // |t| <= n
constexpr int gq_up(int n, int d) { return (n + d - 1) / d; }

template <int LA, int LB, int LC, int LD>
struct Gq {
    static constexpr int NB = gq_cart(LB), ND = gq_cart(LD);
    static constexpr int NAB = gq_cart(LA) * NB, NCD = gq_cart(LC) * ND;
    static constexpr int LAB = LA + LB, LCD = LC + LD, LT = LAB + LCD + 1;   // the tower's order
    static constexpr int NT = gq_herm(LAB), NT1 = gq_herm(LAB + 1);
    static constexpr int NU = gq_herm(LCD), NU1 = gq_herm(LCD + 1), NR = gq_herm(LT);
    // bra primitives of a wavefront's step -- its columns (i, t) fill 16-wide
    // tiles (4 per i: 4, 8 or 16 i; 10: 3 or 6; 20: 3; 35 and 56: one i),
    // fewer where the towers are large -- and of a batch
    static constexpr int IBW = NT1 == 4 ? (NR <= 20 ? 16 : NR <= 56 ? 8 : 4)
                                        : NT1 == 10 ? (NR <= 56 ? 6 : 3) : NT1 == 20 ? 3 : 1;
    // Where a batch of four steps keeps a second workgroup off the CU, two,
    // and pcd read from memory ((sd|dd) 5.42 -> 4.88 ms, (pd|dd) 7.64 -> 7.15
    // ms of the 8-atom gradient; the others lose by it: (sp|dd) 2.63 -> 2.96 ms,
    // (dd|dd), one workgroup either way, 4.49 -> 4.69 ms).
    static constexpr bool TIGHT = LCD == 4 && (LAB == 2 || LAB == 3), PCD = !TIGHT;
    static constexpr int SB = TIGHT ? 2 : 4, IB = SB * IBW;
    // tiles and steps of Y = Wk [t + u] (rows ab, columns (i, t), over u), of
    // X += Wb [t + u] (rows cd, columns u, over (i, t)), of Wb and of Wk
    static constexpr int MY = gq_up(NAB, 16), NY = gq_up(IBW * NT1, 16), KY = gq_up(NU, 4);
    static constexpr int MX = gq_up(NCD, 16), NX = gq_up(NU1, 16), KX = gq_up(IBW * NT, 4);
    static constexpr int KWB = gq_up(NAB, 4);
    static constexpr int NWK = gq_up(NU, 16), KWK = gq_up(NCD, 4);
    // one axis's table (value and its derivatives by the two centres), [i][j][t]
    static constexpr int TB = (LA + 1) * (LB + 1) * (LAB + 2), TK = (LC + 1) * (LD + 1) * (LCD + 2);
    static constexpr int WS = NCD | 1;          // row strides of w, Wb and a wavefront's Wk rows
    static constexpr int WBS = NCD | 1;
    // raw E rows [i][j][t] of one axis, i <= l1 + 1, j <= l2 + 1
    static constexpr int EB = (LA + 2) * (LB + 2) * (LAB + 3), EK = (LC + 2) * (LD + 2) * (LCD + 3);
    static constexpr int gq_max(int a, int b) { return a > b ? a : b; }
    static constexpr int SCR = gq_max(gq_max(2 * IBW * NR, NU * 17), gq_max(3 * EK, 8 * NU1));
    static constexpr int WB = gq_max(IB * NT * WBS, IB * 3 * EB);
    struct Lds {
        double w[NAB * WS];
        double wb[WB];                // a batch's Wb; before it, the raw E of its tables
        double eb[IB * 3 * TB * 3];
        double ek[GQ_WAVES * 3 * TK * 3];
        double scr[GQ_WAVES][SCR];    // towers; raw E of the ket, 16 columns of Wk, 8 rows of X
        double seed[GQ_WAVES][IBW * (LT + 4)];   // [0]^(m), PQ
        double red[GQ_WAVES][12];
        int pab[NAB * NT1];   // (ab, t): offsets of its three table entries, 10 bits each
        int pcd[PCD ? NCD * NU1 : 1];
        int tw[NR];           // the tower's steps
    };
    // The class's index tables: pab, pcd and tw as in Lds, and each lane's
    // tower offsets in the B operands, two to a word: Y's step (ks, n) reads
    // [t + u] of column n = (i, t) and row u, X's of row (i, t) and column u.
    struct Tab {
        int pab[NAB * NT1], pcd[NCD * NU1], tw[NR];
        signed char sign[NU1];   // (-1)^|u|
        int iy[gq_up(KY * NY, 2)][64], ix[gq_up(KX * NX, 2)][64];
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
        constexpr int add(int t, int u) const {   // the index of t + u
            return at(c[t][0] + c[u][0], c[t][1] + c[u][1], c[t][2] + c[u][2]);
        }
    };
    static constexpr int entry(const Herm& h, int l1, int l2, int r, int t) {
        const int n2 = gq_cart(l2), a = gq_herm(l1) - gq_cart(l1) + r / n2, b = gq_herm(l2) - gq_cart(l2) + r % n2;
        int v = 0;
        for (int k = 0; k < 3; ++k)
            v |= ((h.c[a][k] * (l2 + 1) + h.c[b][k]) * (l1 + l2 + 2) + h.c[t][k]) << (10 * k);
        return v;
    }
    static constexpr Tab make() {
        const Herm h;
        Tab T = {};
        for (int r = 0; r < NAB * NT1; ++r) T.pab[r] = entry(h, LA, LB, r / NT1, r % NT1);
        for (int r = 0; r < NCD * NU1; ++r) T.pcd[r] = entry(h, LC, LD, r / NU1, r % NU1);
        for (int u = 0; u < NU1; ++u) T.sign[u] = (h.c[u][0] + h.c[u][1] + h.c[u][2]) % 2 ? -1 : 1;
        for (int j = 1; j < NR; ++j) {
            const int d = h.c[j][0] ? 0 : h.c[j][1] ? 1 : 2, e = h.c[j][d] - 1;
            const int i1 = Herm::at(h.c[j][0] - (d == 0), h.c[j][1] - (d == 1), h.c[j][2] - (d == 2));
            const int i2 = e > 0 ? Herm::at(h.c[j][0] - 2 * (d == 0), h.c[j][1] - 2 * (d == 1), h.c[j][2] - 2 * (d == 2)) : 0;
            T.tw[j] = i1 | (i2 << 10) | (d << 20) | (e << 22);
        }
        for (int l = 0; l < 64; ++l) {
            for (int s = 0; s < KY * NY; ++s) {
                const int u = 4 * (s / NY) + l / 16, n = 16 * (s % NY) + l % 16;
                const int cu = u < NU ? u : NU - 1, cn = n < IBW * NT1 ? n : IBW * NT1 - 1;
                T.iy[s / 2][l] |= ((cn / NT1) * NR + h.add(cn % NT1, cu)) << (16 * (s % 2));
            }
            for (int s = 0; s < KX * NX; ++s) {
                const int k = 4 * (s / NX) + l / 16, u = 16 * (s % NX) + l % 16;
                const int ck = k < IBW * NT ? k : IBW * NT - 1, cu = u < NU1 ? u : NU1 - 1;
                T.ix[s / 2][l] |= ((ck / NT) * NR + h.add(ck % NT, cu)) << (16 * (s % 2));
            }
        }
        return T;
    }
};

template <int LA, int LB, int LC, int LD>
__device__ const typename Gq<LA, LB, LC, LD>::Tab gq_tab = Gq<LA, LB, LC, LD>::make();

// The E of one axis of a primitive pair (its centres at pa, pb from the
// product centre) times f, in two passes with a barrier of the caller's
// between them, so that no lane holds a table. First the raw rows
// [i][j][t], j <= l2 + 1, of one i <= l1 + 1: raised in i from E^{00}, then in
// j along the row.
template <int L1, int L2>
__device__ __forceinline__ void gq_rows(double* __restrict__ raw, int i, double zeta, double pa, double pb, double f) {
    constexpr int J = L2 + 1, T = L1 + 1 + J;
    const double h = 0.5 / zeta;
    double e[T + 2];
#pragma unroll
    for (int t = 0; t <= T + 1; ++t) e[t] = t == 0 ? f : 0.0;
#pragma unroll
    for (int r = 0; r < L1 + 1 + J; ++r) {
        const bool up = r < L1 + 1;   // the raises in i, done in the first i of them
        const double x = up ? pa : pb;
        double below = 0.0;
        if (!up) {
#pragma unroll
            for (int t = 0; t <= T; ++t) raw[(i * (J + 1) + (r - L1 - 1)) * (T + 1) + t] = e[t];
        }
#pragma unroll
        for (int t = 0; t <= T; ++t) {
            const double v = x * e[t] + (double)(t + 1) * e[t + 1] + h * below;
            below = e[t];
            e[t] = up && r >= i ? e[t] : v;
        }
    }
#pragma unroll
    for (int t = 0; t <= T; ++t) raw[(i * (J + 1) + J) * (T + 1) + t] = e[t];
}

// Then entry r of the table [i <= l1][j <= l2][t <= l1 + l2 + 1], three values:
// E, and its derivatives by the first centre, 2 xa E^{i+1,j} - i E^{i-1,j}
// (x2a = 2 xa), and by the second.
template <int L1, int L2>
__device__ __forceinline__ void gq_entry(double* __restrict__ out, const double* __restrict__ raw, int r, double x2a,
                                         double x2b) {
    constexpr int J = L2 + 1, T1 = L1 + 2 + J, S = (J + 1) * T1;   // row strides of raw
    const int t = r % (L1 + L2 + 2), ij = r / (L1 + L2 + 2), i = ij / (L2 + 1), j = ij - i * (L2 + 1);
    const double* __restrict__ e = raw + i * S + j * T1 + t;
    out[r * 3] = e[0];
    out[r * 3 + 1] = x2a * e[S] - (i ? (double)i * e[-S] : 0.0);
    out[r * 3 + 2] = x2b * e[T1] - (j ? (double)j * e[-T1] : 0.0);
}

template <int T>
__device__ __forceinline__ double gq_value(const double* __restrict__ e, int p) {
    return e[(p & 1023) * 3] * e[(T + ((p >> 10) & 1023)) * 3] * e[(2 * T + (p >> 20)) * 3];
}

}  // namespace

// Work items blockIdx.x, + gridDim.x, ... of n_items (see fj_gf_item). Every
// __syncthreads sits in control flow uniform over the workgroup; the matrix
// cores' steps and fj_wave_sync in control flow uniform over the wavefront.
template <int LA, int LB, int LC, int LD>
__global__ void __launch_bounds__(GQ_THREADS, (LA + LB + LC + LD == 8 ? 1 : 2)) fj_gfquad_k(FjGfArgs g0, const FjGfJob* jobs, int n_jobs,
                                                          long long n_items) {
    typedef Gq<LA, LB, LC, LD> Q;
    constexpr int NAB = Q::NAB, NCD = Q::NCD, NT = Q::NT, NT1 = Q::NT1, NU = Q::NU, NU1 = Q::NU1, NR = Q::NR;
    constexpr int IBW = Q::IBW, IB = Q::IB, LT = Q::LT, WS = Q::WS, WBS = Q::WBS, TB = Q::TB, TK = Q::TK;
    constexpr int MY = Q::MY, NY = Q::NY, KY = Q::KY, MX = Q::MX, NX = Q::NX, KX = Q::KX;
    __shared__ typename Q::Lds S;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, l4 = lane >> 4;
    double* const R0 = S.scr[wave];
    double* const R1 = S.scr[wave] + IBW * NR;
    double* const seed = S.seed[wave];
    double* const ek = S.ek + wave * 3 * TK * 3;

    const typename Q::Tab& T = gq_tab<LA, LB, LC, LD>;
    for (int r = tid; r < NAB * NT1; r += GQ_THREADS) S.pab[r] = T.pab[r];
    if constexpr (Q::PCD)
        for (int r = tid; r < NCD * NU1; r += GQ_THREADS) S.pcd[r] = T.pcd[r];
    const int* const pcd = Q::PCD ? S.pcd : T.pcd;
    for (int r = tid; r < NR; r += GQ_THREADS) S.tw[r] = T.tw[r];
    int iy[gq_up(KY * NY, 2)], ix[gq_up(KX * NX, 2)];   // this lane's tower offsets
#pragma unroll
    for (int s = 0; s < gq_up(KY * NY, 2); ++s) iy[s] = T.iy[s][lane];
#pragma unroll
    for (int s = 0; s < gq_up(KX * NX, 2); ++s) ix[s] = T.ix[s][lane];

    for (long long q0 = (long long)blockIdx.x; q0 < n_items; q0 += (long long)gridDim.x) {
        FjGfArgs g = g0;
        int pq0, pq1, bra, ket;
        const double deg = fj_gf_item(g, jobs, n_jobs, q0, pq0, pq1, bra, ket);
        // piece c of the quartet's n: a range of columns j and one of rows i
        const int k_cd = g.k_cd, n = (g.k_ab * k_cd + g.chunk - 1) / g.chunk, c = pq0 / g.chunk;
        const int n4 = (k_cd + 3) / 4, pj = min(n, n4), pi = min(n / pj, g.k_ab), cj = c % pj, ci = c / pj;
        if (ci >= pi) continue;   // uniform; the pieces before have it all
        const int j0 = 4 * (int)((long long)cj * n4 / pj), j1 = min(k_cd, 4 * (int)((long long)(cj + 1) * n4 / pj));
        const int i_lo = (int)((long long)ci * g.k_ab / pi), i_hi = (int)((long long)(ci + 1) * g.k_ab / pi) - 1;
        __syncthreads();   // the previous item's readers of w are done
        {
            const size_t n = (size_t)g.n_ao;
            const int oa = g.bra_ao[2 * bra], ob = g.bra_ao[2 * bra + 1];
            const int oc = g.ket_ao[2 * ket], od = g.ket_ao[2 * ket + 1];
            const double* __restrict__ D = g.D;
            for (int r = tid; r < NAB * NCD; r += GQ_THREADS) {
                const int ab = r / NCD, cd = r - ab * NCD;
                const int a = oa + ab / Q::NB, b = ob + ab % Q::NB, c = oc + cd / Q::ND, d = od + cd % Q::ND;
                S.w[ab * WS + cd] = deg * (4.0 * D[a * n + b] * D[c * n + d] - D[a * n + c] * D[b * n + d] -
                                           D[a * n + d] * D[b * n + c]);
            }
        }
        const double* __restrict__ AB = g.AB + 3 * bra;
        const double* __restrict__ CD = g.CD + 3 * ket;
        const double* __restrict__ bp = g.bra_prim + (size_t)bra * g.k_ab * GF_REC;
        const double* __restrict__ kp = g.ket_prim + (size_t)ket * k_cd * GF_REC;
        double gA[3] = {0.0, 0.0, 0.0}, gB[3] = {0.0, 0.0, 0.0};
        double gC[3] = {0.0, 0.0, 0.0}, gD[3] = {0.0, 0.0, 0.0};
        // wavefronts over j, and over i where there are fewer than three j
        const int WJ = min(4, j1 - j0 == 3 ? 4 : j1 - j0), WI = GQ_WAVES / WJ, wj = wave % WJ, wi = wave / WJ;
        __syncthreads();

        for (int jb = j0; jb < j1; jb += WJ) {
            const int j = jb + wj;
            const bool jv = j < j1;
            const double* __restrict__ rk = kp + (jv ? j : j0) * GF_REC;
            const double qz = rk[6], Qx = rk[0], Qy = rk[1], Qz = rk[2];
            // the ket's axis tables (U in the x axis), then Wk as A operands
            if (lane < 3 * (LC + 2)) {
                const int k = lane / (LC + 2);
                gq_rows<LC, LD>(R0 + k * Q::EK, lane - k * (LC + 2), qz, rk[3 + k], rk[3 + k] + CD[k],
                                   k == 0 ? rk[7] : 1.0);
            }
            fj_wave_sync();
            for (int r = lane; r < 3 * TK; r += 64) {
                const int k = r / TK;
                gq_entry<LC, LD>(ek + k * TK * 3, R0 + k * Q::EK, r - k * TK, 2.0 * rk[8], 2.0 * rk[9]);
            }
            fj_wave_sync();
            double wk[MY][KY];
#pragma unroll
            for (int m = 0; m < MY; ++m) {
                fj_v4d acc[Q::NWK];
#pragma unroll
                for (int n = 0; n < Q::NWK; ++n) acc[n] = fj_v4d{0.0, 0.0, 0.0, 0.0};
                const int ab = min(16 * m + l16, NAB - 1);
                for (int ks = 0; ks < Q::KWK; ++ks) {
                    const int cd = 4 * ks + l4, cc = min(cd, NCD - 1);
                    const double av = cd < NCD ? S.w[ab * WS + cc] : 0.0;
#pragma unroll
                    for (int n = 0; n < Q::NWK; ++n) {
                        const int u = min(16 * n + l16, NU - 1);
                        acc[n] = fj_mfma_f64_16x16x4(av, gq_value<TK>(ek, pcd[cc * NU1 + u]), acc[n]);
                    }
                }
#pragma unroll
                for (int n = 0; n < Q::NWK; ++n) {
                    const int u = 16 * n + l16;
                    const bool odd = T.sign[min(u, NU - 1)] < 0;
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (u < NU) S.scr[wave][u * 17 + l4 + 4 * v] = odd ? -acc[n][v] : acc[n][v];
                }
                fj_wave_sync();
#pragma unroll
                for (int ks = 0; ks < KY; ++ks) {
                    const int u = 4 * ks + l4;
                    wk[m][ks] = u < NU ? S.scr[wave][min(u, NU - 1) * 17 + l16] : 0.0;
                }
                fj_wave_sync();
            }
            fj_v4d xa[MX][NX];
#pragma unroll
            for (int m = 0; m < MX; ++m)
#pragma unroll
                for (int n = 0; n < NX; ++n) xa[m][n] = fj_v4d{0.0, 0.0, 0.0, 0.0};

            for (int ib = i_lo; ib <= i_hi; ib += IB) {
                const int nr = min(IB, i_hi - ib + 1);   // the batch's rows
                __syncthreads();   // the previous batch's readers of eb and wb are done
                for (int r = tid; r < nr * 3 * (LA + 2); r += GQ_THREADS) {
                    const int bk = r / (LA + 2), b = bk / 3, k = bk - 3 * b;
                    const double* __restrict__ rb = bp + (ib + b) * GF_REC;
                    gq_rows<LA, LB>(S.wb + bk * Q::EB, r - bk * (LA + 2), rb[6], rb[3 + k], rb[3 + k] + AB[k],
                                       k == 0 ? rb[7] : 1.0);
                }
                __syncthreads();
                for (int r = tid; r < nr * 3 * TB; r += GQ_THREADS) {
                    const int bk = r / TB, i = ib + bk / 3;
                    gq_entry<LA, LB>(S.eb + bk * TB * 3, S.wb + bk * Q::EB, r - bk * TB, 2.0 * bp[i * GF_REC + 8],
                                     2.0 * bp[i * GF_REC + 9]);
                }
                __syncthreads();
                // Wb of the batch: rows cd, columns (i, t), over ab
                for (int n = wave; 16 * n < nr * NT; n += GQ_WAVES) {
                    const int col = min(16 * n + l16, nr * NT - 1), b = col / NT, t = col - b * NT;
                    const double* __restrict__ e = S.eb + b * 3 * TB * 3;
                    fj_v4d acc[MX];
#pragma unroll
                    for (int m = 0; m < MX; ++m) acc[m] = fj_v4d{0.0, 0.0, 0.0, 0.0};
                    for (int ks = 0; ks < Q::KWB; ++ks) {
                        const int ab = 4 * ks + l4, aa = min(ab, NAB - 1);
                        const double bv = gq_value<TB>(e, S.pab[aa * NT1 + t]);
#pragma unroll
                        for (int m = 0; m < MX; ++m) {
                            const double av = ab < NAB ? S.w[aa * WS + min(16 * m + l16, NCD - 1)] : 0.0;
                            acc[m] = fj_mfma_f64_16x16x4(av, bv, acc[m]);
                        }
                    }
#pragma unroll
                    for (int m = 0; m < MX; ++m)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const int cd = 16 * m + l4 + 4 * v;
                            if (16 * n + l16 < nr * NT && cd < NCD) S.wb[col * WBS + cd] = acc[m][v];
                        }
                }
                __syncthreads();
                for (int s = wi; s < Q::SB; s += WI) {
                    const int i0 = ib + s * IBW;
                    if (!jv || i0 > i_hi) break;   // uniform over the wavefront
                    const int last = min(IBW - 1, i_hi - i0);   // the step's last row with tables
                    // seeds (zero past the last row), then the towers' levels
                    if (lane < IBW) {
                        const int i = i0 + min(lane, last);
                        const bool in = lane <= last;
                        const double* __restrict__ rb = bp + i * GF_REC;
                        const double p = rb[6], x = rb[0] - Qx, y = rb[1] - Qy, z = rb[2] - Qz;
                        const double rho = p * qz / (p + qz);
                        double* const w = seed + lane * (LT + 4);
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
                        ((LT & 1) ? R1 : R0)[lane * NR] = w[LT];
                    }
                    fj_wave_sync();
#pragma unroll
                    for (int m = LT - 1; m >= 0; --m) {
                        double* __restrict__ cur = (m & 1) ? R1 : R0;
                        const double* __restrict__ prv = (m & 1) ? R0 : R1;
                        const int n_m = gq_herm(LT - m);
                        for (int r = lane; r < IBW * n_m; r += 64) {
                            const int b = IBW == 1 ? 0 : r / n_m, h = r - b * n_m;
                            const double* __restrict__ w = seed + b * (LT + 4);
                            double v;
                            if (h == 0) {
                                v = w[m];
                            } else {
                                const int t = S.tw[h], c1 = t >> 22;
                                v = w[LT + 1 + ((t >> 20) & 3)] * prv[b * NR + (t & 1023)];
                                if (c1 > 0) v += (double)c1 * prv[b * NR + ((t >> 10) & 1023)];
                            }
                            cur[b * NR + h] = v;
                        }
                        fj_wave_sync();
                    }
                    // X += Wb [t + u]
                    {
                        const double* __restrict__ wb = S.wb + s * IBW * NT * WBS;
#pragma unroll
                        for (int ks = 0; ks < KX; ++ks) {
                            const int k = 4 * ks + l4;
                            double av[MX];
#pragma unroll
                            for (int m = 0; m < MX; ++m) {
                                const double t = wb[min(k, (last + 1) * NT - 1) * WBS + min(16 * m + l16, NCD - 1)];
                                av[m] = k < IBW * NT ? t : 0.0;
                            }
#pragma unroll
                            for (int n = 0; n < NX; ++n) {
                                const int c = ks * NX + n;
                                const double bv = R0[(c & 1) ? ix[c / 2] >> 16 : ix[c / 2] & 0xffff];
#pragma unroll
                                for (int m = 0; m < MX; ++m) xa[m][n] = fj_mfma_f64_16x16x4(av[m], bv, xa[m][n]);
                            }
                        }
                    }
                    // Y, 16 columns at a time, and the bra's centres (the
                    // empty statements keep the next tiles' loads from moving
                    // up and spilling)
#pragma unroll
                    for (int n = 0; n < NY; ++n) {
                        if (16 * n >= (last + 1) * NT1) break;   // uniform
                        __asm__ volatile("" ::: "memory");
                        fj_v4d y[MY];
#pragma unroll
                        for (int m = 0; m < MY; ++m) y[m] = fj_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                        for (int ks = 0; ks < KY; ++ks) {
                            const int c = ks * NY + n;
                            const double bv = R0[(c & 1) ? iy[c / 2] >> 16 : iy[c / 2] & 0xffff];
#pragma unroll
                            for (int m = 0; m < MY; ++m) y[m] = fj_mfma_f64_16x16x4(wk[m][ks], bv, y[m]);
                        }
                        const int col = 16 * n + l16, b = min(col, IBW * NT1 - 1) / NT1, t = min(col, IBW * NT1 - 1) % NT1;
                        const double* __restrict__ e = S.eb + (s * IBW + min(b, last)) * 3 * TB * 3;
#pragma unroll
                        for (int m = 0; m < MY; ++m) {
                            __asm__ volatile("" ::: "memory");
#pragma unroll
                            for (int v = 0; v < 4; ++v) {
                                const int ab = 16 * m + l4 + 4 * v;
                                if (16 * m + 4 * v >= NAB) continue;   // rows past every lane's
                                const int p = S.pab[min(ab, NAB - 1) * NT1 + t];
                                const double* __restrict__ ex = e + (p & 1023) * 3;
                                const double* __restrict__ ey = e + (TB + ((p >> 10) & 1023)) * 3;
                                const double* __restrict__ ez = e + (2 * TB + (p >> 20)) * 3;
                                const double c = ab < NAB && col < IBW * NT1 ? y[m][v] : 0.0;
                                const double yz = c * (ey[0] * ez[0]), xz = c * (ex[0] * ez[0]), xy = c * (ex[0] * ey[0]);
                                gA[0] += ex[1] * yz;
                                gA[1] += ey[1] * xz;
                                gA[2] += ez[1] * xy;
                                gB[0] += ex[2] * yz;
                                gB[1] += ey[2] * xz;
                                gB[2] += ez[2] * xy;
                            }
                        }
                    }
                    fj_wave_sync();   // before the next towers
                }
            }
            // the ket's centres, from this j's X: 8 rows cd at a time through
            // LDS, lanes over (cd, u) (the tiles' own lanes would hold every
            // table value at once)
            if (jv) {
#pragma unroll
                for (int h = 0; h < 2 * MX; ++h) {
                    if (8 * h >= NCD) continue;
#pragma unroll
                    for (int n = 0; n < NX; ++n)
#pragma unroll
                        for (int v = 0; v < 2; ++v)
                            if (16 * n + l16 < NU1)
                                S.scr[wave][(l4 + 4 * v) * NU1 + 16 * n + l16] = xa[h / 2][n][2 * (h % 2) + v];
                    fj_wave_sync();
                    const int cd0 = 8 * h, n_el = min(8, NCD - cd0) * NU1;
#pragma unroll 1
                    for (int r = lane; r < n_el; r += 64) {
                        const int p = pcd[cd0 * NU1 + r], u = r % NU1;
                        const double* __restrict__ ex = ek + (p & 1023) * 3;
                        const double* __restrict__ ey = ek + (TK + ((p >> 10) & 1023)) * 3;
                        const double* __restrict__ ez = ek + (2 * TK + (p >> 20)) * 3;
                        const double c = T.sign[u] < 0 ? -S.scr[wave][r] : S.scr[wave][r];
                        const double yz = ey[0] * ez[0], xz = ex[0] * ez[0], xy = ex[0] * ey[0];
                        gC[0] += c * ex[1] * yz;
                        gC[1] += c * ey[1] * xz;
                        gC[2] += c * ez[1] * xy;
                        gD[0] += c * ex[2] * yz;
                        gD[1] += c * ey[2] * xz;
                        gD[2] += c * ez[2] * xy;
                    }
                    fj_wave_sync();
                }
            }
            fj_wave_sync();   // before the next j's tables
        }

        // the twelve sums over the workgroup, then into G
        const double v[12] = {gA[0], gA[1], gA[2], gB[0], gB[1], gB[2], gC[0], gC[1], gC[2], gD[0], gD[1], gD[2]};
#pragma unroll
        for (int c = 0; c < 12; ++c) {
            const double s = fj_wave_sum(v[c]);
            if (lane == 0) S.red[wave][c] = s;
        }
        __syncthreads();
        if (tid < 12) {
            const int pos = tid / 3, k = tid - 3 * pos;
            double s = 0.0;
            for (int w = 0; w < GQ_WAVES; ++w) s += S.red[w][tid];
            const int atom = pos == 0 ? g.bra_at[2 * bra] : pos == 1 ? g.bra_at[2 * bra + 1]
                           : pos == 2 ? g.ket_at[2 * ket] : g.ket_at[2 * ket + 1];
            atomicAdd(g.G + 3 * atom + k, s);
        }
    }
}
