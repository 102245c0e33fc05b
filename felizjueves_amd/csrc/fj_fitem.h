// fj_fitem.h -- what the fused F kernels of the classes with an f shell share
// (fj_floop.h, fj_fquad.h): the work item, its kets with the screen and the
// degeneracy, and a quartet's six density and F blocks in LDS.
//
// The includer provides fj_device.h.
#pragma once

// The workgroup's share of a launch: the bra pair, its kets [k0, k1), the
// system and the bra's primitive-pair range [kb0, kb0 + kab). The work item
// is (bra pair, first ket, system | bra chunk, ket end), or (x, y * span,
// the single system, n_ket) without a work list; an item covers at most
// `span` kets and, with a work list, workgroup (x, y) takes the y-th of
// gridDim.y equal slices of item x's kets. False (uniformly) when there is
// nothing to do.
struct FjFlItem {
    int bra, k0, k1, kmin, kb0, kab;
    FjSys S;
};

__device__ __forceinline__ bool fj_fl_item(const FjFArgs& a, int span, FjFlItem& it) {
    int kb_lo = 0, kb_n = 0;
    if (a.work) {
        const int4 w = a.work[blockIdx.x];
        const int end = min(w.w, w.y + span), sub = (span + (int)gridDim.y - 1) / (int)gridDim.y;
        it.bra = w.x;
        it.k0 = w.y + (int)blockIdx.y * sub;
        it.k1 = min(end, it.k0 + sub);
        it.S = a.sys[w.z & 0xffff];
        kb_lo = (w.z >> 16) & 0xff;
        kb_n = (w.z >> 24) & 0xff;
    } else {
        it.bra = (int)blockIdx.x;
        it.k0 = (int)blockIdx.y * span;
        it.S = a.one;
        it.k1 = min(a.ket.n, it.k0 + span);
    }
    it.kmin = a.diag * it.bra;
    if (it.k0 >= it.k1 || (!a.ket_list && it.k0 + span <= it.kmin)) return false;
    fj_side_range(a.bra, it.bra, it.kb0, it.kab);
    if (it.kab > FJ_MAX_PRIM_PAIRS || kb_lo >= it.kab) return false;
    it.kb0 += kb_lo;
    it.kab = kb_n ? min(it.kab - kb_lo, kb_n) : it.kab - kb_lo;
    return true;
}

// One ket of the item: its pair index, primitive-pair range [kc0, kc0 +
// kcd), shells, AO offsets and the J / K digestion scales of the quartet's
// degeneracy. False (uniformly) when it is below the diagonal, screened out
// (G_ab G_cd times the largest density block it digests into, under tau)
// or empty.
struct FjFlKet {
    int k, kc0, kcd, sc, sd, oc, od;
    double s_j, s_k;
};

__device__ __forceinline__ bool fj_fl_ket(const FjFArgs& a, const FjFlItem& it, int kk, int sa, int sb,
                                          double Gb, FjFlKet& q) {
    int kc_lo = 0, kc_n = 0;
    q.k = kk;
    if (a.ket_list) {
        const int v = a.ket_list[kk];
        q.k = v & 0x1ffff;
        kc_lo = (v >> 17) & 0x7f;
        kc_n = (v >> 24) & 0x7f;
    }
    const int k = q.k;
    if (k < it.kmin) return false;
    q.sc = a.ket.sh[2 * k];
    q.sd = a.ket.sh[2 * k + 1];
    const int ns = it.S.n_sh;
    const double* __restrict__ Dsh = it.S.Dsh;
    double dmax = 2.0 * Dsh[sa * ns + sb];
    dmax = fmax(dmax, 2.0 * Dsh[q.sc * ns + q.sd]);
    dmax = fmax(dmax, 0.5 * Dsh[sa * ns + q.sc]);
    dmax = fmax(dmax, 0.5 * Dsh[sa * ns + q.sd]);
    dmax = fmax(dmax, 0.5 * Dsh[sb * ns + q.sc]);
    dmax = fmax(dmax, 0.5 * Dsh[sb * ns + q.sd]);
    if (Gb * (a.ket.G[k] * dmax) < a.tau) return false;
    fj_side_range(a.ket, k, q.kc0, q.kcd);
    if (q.kcd > FJ_MAX_PRIM_PAIRS || q.kcd <= kc_lo) return false;
    q.kc0 += kc_lo;
    q.kcd = kc_n ? min(q.kcd - kc_lo, kc_n) : q.kcd - kc_lo;
    double deg = 1.0;
    if (sa == sb) deg *= 0.5;
    if (q.sc == q.sd) deg *= 0.5;
    if (a.diag && k == it.bra) deg *= 0.5;
    q.s_j = 2.0 * deg;
    q.s_k = -0.5 * deg;
    q.oc = a.ket.ao[2 * k];
    q.od = a.ket.ao[2 * k + 1];
    return true;
}

// The six blocks of a quartet in LDS, in the order ab, cd, ac, ad, bc, bd:
// w the weighted density blocks (J scale on ab and cd, K scale on the
// others), f the F accumulators. fj_fl_load fills w and zeroes f;
// fj_fl_flush adds f into F with one global atomic per nonzero element.
struct FjFlBlocks {
    double* w[6];
    double* f[6];
};

__device__ __forceinline__ void fj_fl_load(const FjFlBlocks& B, const double* __restrict__ D, int n_ao,
                                           int oa, int ob, int oc, int od, int na, int nb, int nc,
                                           int nd, double s_j, double s_k, int lane, int nthr) {
    const int r0[6] = {oa, oc, oa, oa, ob, ob}, c0[6] = {ob, od, oc, od, oc, od};
    const int nr[6] = {na, nc, na, na, nb, nb}, ncol[6] = {nb, nd, nc, nd, nc, nd};
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        const double sc = i < 2 ? s_j : s_k;
        for (int j = lane; j < nr[i] * ncol[i]; j += nthr) {
            B.w[i][j] = sc * D[(size_t)(r0[i] + j / ncol[i]) * n_ao + c0[i] + j % ncol[i]];
            B.f[i][j] = 0.0;
        }
    }
}

__device__ __forceinline__ void fj_fl_flush(const FjFlBlocks& B, double* F, int n_ao, int oa, int ob,
                                            int oc, int od, int na, int nb, int nc, int nd, int lane,
                                            int nthr) {
    const int r0[6] = {oa, oc, oa, oa, ob, ob}, c0[6] = {ob, od, oc, od, oc, od};
    const int nr[6] = {na, nc, na, na, nb, nb}, ncol[6] = {nb, nd, nc, nd, nc, nd};
#pragma unroll
    for (int i = 0; i < 6; ++i)
        for (int j = lane; j < nr[i] * ncol[i]; j += nthr)
            if (B.f[i][j] != 0.0)
                unsafeAtomicAdd(F + (size_t)(r0[i] + j / ncol[i]) * n_ao + c0[i] + j % ncol[i], B.f[i][j]);
}
