// fj_coop.h -- the quartet-cooperative form of the generated HGP F kernels
// (gen/c_<class>.hip): what does not depend on the class's recurrences.
//
// The per-lane form (gen/f_<class>.hip) gives a lane a contracted quartet, or
// a chunk of its primitive quartets, and the whole of its HRR and digestion.
// A build of few quartets then either runs long lanes on an idle chip, or
// splits the primitives and pays an HRR and some hundred F atomics, onto the
// same addresses, per chunk. Here a wavefront takes up to NQ kets of a bra
// pair, deals their primitive quartets evenly to its lanes, sums the lanes'
// boundaries per quartet in LDS, and then transforms and digests each quartet
// once, lanes over components:
//   A  lanes over primitive quartets: the class's VRR groups, each group's
//      targets summed over the lanes of a quartet (CH targets at a time: a
//      lane's values to LDS, then CH x 64 / CH lanes sum CH lanes' values each
//      and add into the quartet's boundary, one LDS atomic per quartet met);
//   B  lanes over (quartet, f): the bra HRR of one column, in place;
//   C  lanes over (quartet, ab): the ket HRR of one row, into X (the largest
//      classes' X in slices of a);
//   D  lanes over the elements of the six F blocks: one sum over X each and
//      one global atomic (F_ab: once per workgroup).
// A workgroup is four wavefronts of one item: they share the bra's records and
// deal the item's kets in turn, or, where those are fewer, its primitives. A
// boundary is summed by one wavefront alone, so in a fixed order: the HRR
// cancels, and would amplify the rounding of a changing one (2.7e-12 between
// two builds of the three-atom system with four wavefronts adding into it).
#pragma once

#define FJ_COOP_THREADS 256
#define FJ_COOP_WAVES 4
#define FJ_COOP_ROW 65     // stride of one target's row of 64 lanes

// The kets of a wavefront's current batch, compacted to the live ones.
template <int NQ>
struct FjCoopKets {
    int k[NQ];      // ket pair
    int p0[NQ];     // its first primitive record
    int n[NQ];      // primitive quartets
    int lane0[NQ];  // first lane (over the parts) and lanes
    int lanes[NQ];
    int live[NQ];   // before compaction: primitive records, 0 for a dead ket
    int pk[NQ], pp[NQ];
};

// Adds CNT <= CH targets' values of the wavefront's lanes (red[i][lane]) to
// the boundaries of the lanes' quartets: lane (i, sub) sums target i over the
// CH lanes from CH sub, whose quartets are q0, q0 + 1, ... with a step after
// each lane set in mask.
template <int CNT, int CH>
__device__ __forceinline__ void fj_coop_reduce(const double* __restrict__ red, int lane, unsigned mask,
                                               int q0, int nq, double* __restrict__ bnd, int reg,
                                               int pos) {
    const int i = lane & (CH - 1);
    if (i < CNT && q0 < nq) {
        const double* __restrict__ row = red + i * FJ_COOP_ROW + (lane & ~(CH - 1));
        double* __restrict__ dst = bnd + q0 * reg + pos + i;
        if (mask == 0) {   // one quartet: four independent chains
            double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
            for (int l = 0; l < CH; l += 4) {
                s0 += row[l];
                s1 += row[l + 1];
                s2 += row[l + 2];
                s3 += row[l + 3];
            }
            unsafeAtomicAdd(dst, (s0 + s1) + (s2 + s3));
        } else {
            double s = 0.0;
            int q = q0;
#pragma unroll
            for (int l = 0; l < CH; ++l) {
                s += row[l];
                if ((mask >> l) & 1) {
                    unsafeAtomicAdd(dst, s);
                    s = 0.0;
                    dst += reg;
                    ++q;
                }
            }
            if (q < nq) unsafeAtomicAdd(dst, s);
        }
    }
}

// The six F blocks of a quartet as one list of elements: ab, cd, ac, ad, bc,
// bd, each row-major.
template <int NA, int NB, int NC, int ND>
struct FjCoopBlocks {
    static constexpr int CD = NA * NB, AC = CD + NC * ND, AD = AC + NA * NC, BC = AD + NA * ND,
                         BD = BC + NB * NC, N = BD + NB * ND;
    // block of element o: its two shells (0..3 = a..d) and components
    __device__ static __forceinline__ void of(int o, int& s0, int& s1, int& i, int& j) {
        int r, n;
        if (o < CD) { s0 = 0; s1 = 1; r = o; n = NB; }
        else if (o < AC) { s0 = 2; s1 = 3; r = o - CD; n = ND; }
        else if (o < AD) { s0 = 0; s1 = 2; r = o - AC; n = NC; }
        else if (o < BC) { s0 = 0; s1 = 3; r = o - AD; n = ND; }
        else if (o < BD) { s0 = 1; s1 = 2; r = o - BC; n = NC; }
        else { s0 = 1; s1 = 3; r = o - BD; n = ND; }
        i = r / n;
        j = r - i * n;
    }
    // F element (i, j) of shells s0, s1: the sum of its quartet's integrals
    // X[ab][cd] (row stride XS; rows of a in [a0, a1) only, the first at X)
    // with the weighted density block w (same element order) it meets.
    template <int XS>
    __device__ static __forceinline__ double sum(const double* __restrict__ X, const double* __restrict__ w,
                                                 int s0, int s1, int i, int j, int a0, int a1) {
        int x, su, sv, nu, nv, b;   // sum over (u, v): w[b + u nv + v] X[x + u su + v sv]
        if (s0 == 0) {
            if (i < a0 || i >= a1) return 0.0;
            const int r = (i - a0) * NB * XS;
            if (s1 == 1) { x = r + j * XS; su = ND; sv = 1; nu = NC; nv = ND; b = CD; }
            else if (s1 == 2) { x = r + j * ND; su = XS; sv = 1; nu = NB; nv = ND; b = BD; }
            else { x = r + j; su = XS; sv = ND; nu = NB; nv = NC; b = BC; }
        } else {
            nu = a1 - a0;
            su = NB * XS;
            if (s0 == 2) { x = i * ND + j; sv = XS; nv = NB; b = 0; }
            else if (s1 == 2) { x = i * XS + j * ND; sv = 1; nv = ND; b = AD; }
            else { x = i * XS + j; sv = ND; nv = NC; b = AC; }
            b += a0 * nv;
        }
        double t = 0.0;
        for (int u = 0; u < nu; ++u)
            for (int v = 0; v < nv; ++v) t += w[b + u * nv + v] * X[x + u * su + v * sv];
        return t;
    }
};

// The live kets of the n <= NQ list entries first, first + step, ... of one
// bra pair, the lanes each gets over `parts` wavefronts, and their number.
// Every lane of the wavefront calls it.
template <int NQ>
__device__ __forceinline__ int fj_coop_kets(const FjFArgs& a, const FjSys& S, FjCoopKets<NQ>& K, int bra,
                                            int kab, int first, int step, int n, int parts) {
    const int lane = (int)threadIdx.x & 63;
    if (lane < n) {
        const int v = a.ket_list[first + step * lane];
        const int k = v & 0x1ffff, lo = (v >> 17) & 0x7f, cnt = (v >> 24) & 0x7f;
        int p0, kcd;
        fj_side_range(a.ket, k, p0, kcd);
        const int sa = a.bra.sh[2 * bra], sb = a.bra.sh[2 * bra + 1];
        const int sc = a.ket.sh[2 * k], sd = a.ket.sh[2 * k + 1];
        const double* __restrict__ Dsh = S.Dsh;
        const int ns = S.n_sh;
        double dmax = 2.0 * Dsh[sa * ns + sb];
        dmax = fmax(dmax, 2.0 * Dsh[sc * ns + sd]);
        dmax = fmax(dmax, 0.5 * Dsh[sa * ns + sc]);
        dmax = fmax(dmax, 0.5 * Dsh[sa * ns + sd]);
        dmax = fmax(dmax, 0.5 * Dsh[sb * ns + sc]);
        dmax = fmax(dmax, 0.5 * Dsh[sb * ns + sd]);
        const bool live = k >= a.diag * bra && kcd > lo && !(a.bra.G[bra] * (a.ket.G[k] * dmax) < a.tau);
        K.pk[lane] = k;
        K.pp[lane] = p0 + lo;
        K.live[lane] = live ? (cnt ? min(kcd - lo, cnt) : kcd - lo) : 0;
    }
    fj_wave_sync();
    int nq = 0, N = 0, rank = 0;
    for (int i = 0; i < n; ++i) {
        if (i == lane) rank = nq;
        const int kcd = K.live[i];
        nq += kcd > 0;
        N += kab * kcd;
    }
    // the fewest passes t over the lanes that give every quartet whole lanes
    const int LN = 64 * parts;
    int t = max(1, (N + LN - 1) / LN);
    for (;; ++t) {   // ends: at t = N every quartet takes one lane, and n <= 64
        int s = 0;
        for (int i = 0; i < n; ++i) s += (kab * K.live[i] + t - 1) / t;
        if (s <= LN) break;
    }
    if (lane < n && K.live[lane] > 0) {
        int l0 = 0;
        for (int i = 0; i < lane; ++i) l0 += (kab * K.live[i] + t - 1) / t;
        K.k[rank] = K.pk[lane];
        K.p0[rank] = K.pp[lane];
        K.n[rank] = kab * K.live[lane];
        K.lane0[rank] = l0;
        K.lanes[rank] = (kab * K.live[lane] + t - 1) / t;
    }
    fj_wave_sync();
    return nq;
}
