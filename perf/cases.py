"""The workloads this framework is measured on: two-electron builds over
seeded synthetic molecules, each through the entry points a program calls.

A case names a molecule (its atoms, largest shell and the recipe number that
fixes its contraction depths and exponents) and how it is built. A seed
moves every atom a little and draws a new closed-shell density, as the steps
of a geometry optimisation do. The tables, plans and captured graphs that
such a program keeps over its SCF iterations are made in `prepare`; `run` is
one build.

`exact` evaluates the same integrals by the textbook McMurchie-Davidson
expansion (Helgaker, Joergensen, Olsen, "Molecular Electronic-Structure
Theory", chapter 9) with plain torch in 64 bits.
"""

import math
from functools import lru_cache
from pathlib import Path

import numpy as np
import torch

import felizjueves_amd
from felizjueves_amd import df, gradient, hjk, jk, native, pairs, systems
from felizjueves_amd.basis import Basis, Shell, primitive_norm
from felizjueves_amd.fock import FockBuilder
from felizjueves_amd.hgp import cost
from felizjueves_amd.selector import LearnedSelector

TAU = 1e-12
JITTER = 0.02   # bohr: how far a seed moves an atom


def listed():
    return [
        # an SCF iteration of a small molecule: launches and latency, one graph replay
        dict(name="fock-3-graph", kind="fock", atoms=3, lmax=2, recipe=1, streams=1, graph=True, mixed=False),
        # the builder as a first program calls it: eager, one stream, the default plan
        dict(name="fock-9-eager", kind="fock", atoms=9, lmax=2, recipe=9, streams=1, graph=False, mixed=False),
        # an SCF iteration at the headline size: 40 atoms, four streams, one graph
        dict(name="fock-40-graph", kind="fock", atoms=40, lmax=2, recipe=2, streams=4, graph=True, mixed=False),
        # mixed precision with the learned selector choosing tiers per build
        dict(name="fock-17-mixed", kind="fock", atoms=17, lmax=2, recipe=5, streams=4, graph=True, mixed=True),
        # a batch of molecules in one builder (a data-generation run)
        dict(name="fock-batch-5", kind="batch", atoms=7, molecules=5, lmax=2, recipe=11, streams=4),
        # shells through f (a triple-zeta basis)
        dict(name="fock-4-f", kind="fock", atoms=4, lmax=3, recipe=7, streams=4, graph=False, mixed=False),
        # J and K by themselves on the Hermite engines (J alone for pure functionals, K for hybrids)
        dict(name="coulomb-10", kind="coulomb", atoms=10, lmax=2, recipe=2, mixed=False),
        dict(name="exchange-5", kind="exchange", atoms=5, lmax=2, recipe=6, mixed=False),
        # the split J build of a small molecule, staged and captured once per geometry
        dict(name="split-j-3", kind="split", atoms=3, lmax=2, recipe=1, screen="j"),
        # nuclear gradients: one small molecule (molecular dynamics) and a larger one
        dict(name="gradient-3", kind="gradient", atoms=3, lmax=2, recipe=1),
        dict(name="gradient-8", kind="gradient", atoms=8, lmax=2, recipe=3),
        # the density-fitting tensors: metric and three-center integrals, aux shells s..g
        dict(name="fitting-9", kind="fitting", atoms=9, lmax=2, recipe=4, aux=4),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo - 0.4), math.log(hi + 0.4)))))

    recipe = rng.randrange(100, 1_000_000)
    kind = rng.choice(["fock", "fock", "fock-f", "batch", "coulomb", "exchange", "split", "gradient", "gradient", "fitting"])
    if kind == "fock":
        return dict(kind="fock", atoms=size(2, 30), lmax=rng.choice([1, 2, 2, 2]), recipe=recipe, streams=rng.choice([1, 2, 4]),
                    graph=rng.random() < 0.6, mixed=rng.random() < 0.3)
    if kind == "fock-f":
        return dict(kind="fock", atoms=size(1, 4), lmax=3, recipe=recipe, streams=rng.choice([1, 4]), graph=False, mixed=False)
    if kind == "batch":
        return dict(kind="batch", atoms=size(3, 8), molecules=rng.randint(2, 6), lmax=2, recipe=recipe, streams=rng.choice([1, 4]))
    if kind == "coulomb":
        return dict(kind="coulomb", atoms=size(2, 10), lmax=rng.choice([1, 2, 2]), recipe=recipe, mixed=rng.random() < 0.3)
    if kind == "exchange":
        return dict(kind="exchange", atoms=size(2, 5), lmax=rng.choice([1, 2, 2]), recipe=recipe, mixed=rng.random() < 0.3)
    if kind == "split":
        return dict(kind="split", atoms=size(1, 3), lmax=rng.choice([1, 2, 2]), recipe=recipe, screen=rng.choice(["j", "k"]))
    if kind == "gradient":
        return dict(kind="gradient", atoms=size(2, 7), lmax=rng.choice([1, 2, 2]), recipe=recipe)
    return dict(kind="fitting", atoms=size(1, 9), lmax=rng.choice([1, 2, 3]), recipe=recipe, aux=rng.randint(2, 4))


# ---------------------------------------------------------------------------
# Molecules


def _recipe(atoms, lmax, recipe):
    """Coordinates (bohr) and shells per atom of a molecule at rest."""
    rng = np.random.default_rng(recipe)
    coords = systems.chain_geometry(rng, atoms) if atoms < 4 else systems.cluster_geometry(rng, atoms)
    ls = tuple(l for l in (0, 0, 1, 2, 3) if l <= lmax)  # noqa: E741
    return coords, [systems.atom_shells(rng, c, ls) for c in coords]


def _molecule(case, seed, member=0):
    """(basis, density, coordinates) of the case's molecule for this seed."""
    coords, shells = _recipe(case["atoms"] + member % 3, case["lmax"], case["recipe"] + 1000 * member)
    rng = np.random.default_rng([seed, member, case["recipe"]])
    coords = coords + rng.uniform(-JITTER, JITTER, size=coords.shape)
    basis = Basis([Shell(s.l, tuple(float(x) for x in c), s.exponents, s.coefficients) for c, sh in zip(coords, shells) for s in sh])
    return basis, systems.closed_shell_density(rng, basis.n_ao, max(2, 5 * len(coords) // 2)), coords


def _members(case, seed):
    return [_molecule(case, seed, m) for m in range(case["molecules"])]


def _aux(case, coords):
    """Even-tempered single-primitive aux shells s..g, `aux` per atom and momentum."""
    l, c, e = [], [], []  # noqa: E741
    for at in coords:
        for m in range(5):
            for k in range(case["aux"]):
                l.append(m)
                c.append(at)
                e.append(0.3 * 2.5**k)
    return df.AuxBasis(l, c, [1] * len(l), e, [primitive_norm(m, x) for m, x in zip(l, e)])


@lru_cache(maxsize=1)
def _selector():
    return LearnedSelector.load(Path(felizjueves_amd.__file__).parent / "tuned" / "selector")


# ---------------------------------------------------------------------------
# The calls


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        mols = _members(case, seed)
        fb = FockBuilder.batch([(b, D) for b, D, _ in mols], tau=TAU)
        fb.to_device()
        return dict(kind=kind, builder=fb, D=[native.to_dev(D) for _, D, _ in mols], streams=case["streams"])
    basis, D, coords = _molecule(case, seed)
    D_dev = native.to_dev(D)
    if kind == "fock":
        fb = FockBuilder(basis, D, tau=TAU, mixed=case["mixed"], selector=_selector() if case["mixed"] else None)
        fb.to_device()
        if case["graph"]:
            fb.capture(D_dev, n_streams=case["streams"])
        return dict(kind="replay" if case["graph"] else "fock", builder=fb, D=D_dev, streams=case["streams"])
    if kind == "coulomb":
        return dict(kind=kind, chain=jk.CoulombChain(basis, tau=TAU, mixed=case["mixed"]), D=D_dev)
    if kind == "exchange":
        return dict(kind=kind, engine=jk.ExchangeBuild(basis, tau=TAU, mixed=case["mixed"]), D=D_dev)
    if kind == "split":
        build = hjk.HJKBuild(basis, D, tau=TAU, screen=case["screen"])
        build.capture(hjk.STREAMS)
        return dict(kind=kind, build=build)
    if kind == "gradient":
        stream = gradient.gf_launches(basis, gradient.shell_atoms(basis, coords))
        return dict(kind=kind, runner=gradient.GpuGfRunner(stream, len(coords), basis.n_ao), D=D_dev)
    aux = _aux(case, coords)
    fit = df.DfIntegrals(aux, basis)
    return dict(kind=kind, fit=fit, metric=torch.empty((aux.n_aux,) * 2, dtype=torch.float64, device=native.device()),
                eri3=torch.empty((basis.n_ao, basis.n_ao, aux.n_aux), dtype=torch.float64, device=native.device()))


def run(state):
    kind = state["kind"]
    if kind == "replay":
        return state["builder"].replay()
    if kind in ("fock", "batch"):
        return state["builder"].build(state["D"], n_streams=state["streams"])
    if kind == "coulomb":
        return state["chain"].run(state["D"])
    if kind == "exchange":
        return state["engine"].run(state["D"], n_streams=4)
    if kind == "split":
        return state["build"].replay()
    if kind == "gradient":
        return state["runner"].run(state["D"], n_streams=4)
    return dict(metric=state["fit"].metric(state["metric"]), eri3=state["fit"].eri3(state["eri3"], n_streams=4))


# ---------------------------------------------------------------------------
# What a pass cannot do without


def _classes(basis, D, screened):
    """Per pair class (la <= lb): (G, primitive pairs) of its unique shell
    pairs; `screened` drops what the pair bounds prune."""
    out = {}
    if screened:
        for p in pairs.kept_pairs(basis, D, TAU, 1)[0]:
            out.setdefault((p.la, p.lb), []).append((p.G, p.degree))
    else:
        for a in range(basis.n_sh):
            for b in range(a, basis.n_sh):
                c = tuple(sorted((int(basis.shell_l[a]), int(basis.shell_l[b]))))
                out.setdefault(c, []).append((math.inf, int(basis.shell_nprim[a] * basis.shell_nprim[b])))
    return {c: np.array(v, dtype=np.float64) for c, v in out.items()}


def _quartets(classes):
    """(class, contracted quartets, primitive quartets) over the unique quartets with G_ab G_cd >= TAU."""
    cs = sorted(classes)
    for i, x in enumerate(cs):
        for y in cs[i:]:
            bra, ket = classes[x], classes[y][np.argsort(-classes[y][:, 0])]
            n = np.searchsorted(-ket[:, 0], -TAU / bra[:, 0], side="right")
            deg = np.concatenate([[0.0], np.cumsum(ket[:, 1])])
            half = 0.5 if x == y else 1.0
            yield (*x, *y), half * float(n.sum()), half * float((bra[:, 1] * deg[n]).sum())


def _herm(n):
    return (n + 1) * (n + 2) * (n + 3) // 6


def _cart(n):
    return (n + 1) * (n + 2) // 2


@lru_cache(maxsize=None)
def _tower(n):
    """Two operations per entry of the Hermite recurrence through order n."""
    return 2 * sum(_herm(n - m) for m in range(n + 1))


def work(case):
    kind = case["kind"]
    mols = _members(case, 0) if kind == "batch" else [_molecule(case, 0)]
    size = flops = 0.0
    for basis, D, coords in mols:
        n = basis.n_ao
        cl = _classes(basis, D, kind not in ("gradient", "fitting", "coulomb"))
        records = 8 * 8 * sum(float(v[:, 1].sum()) for v in cl.values())
        size += 16 * n * n + records   # the density, the result, the primitive-pair records
        if kind == "fitting":
            aux = _aux(case, coords)
            size += 8 * (aux.n_aux**2 + n * n * aux.n_aux) - 16 * n * n
            shells = np.bincount(aux.shell_l, minlength=5)
            for (la, lb), v in cl.items():
                for lp in range(5):
                    # the tower, and the bra transform of the aux components' Hermite integrals
                    per = _tower(la + lb + lp) + 2 * _herm(la + lb) * _cart(lp) * (1 + _cart(la) * _cart(lb))
                    flops += per * float(v[:, 1].sum()) * shells[lp]
            continue
        for cls, quartets, prims in _quartets(cl):
            la, lb, lc, ld = cls
            c = cost(cls)
            if kind == "coulomb":
                flops += prims * (_tower(sum(cls)) + 4 * _herm(la + lb) * _herm(lc + ld))
            elif kind == "gradient":
                # one weight transform and one contraction with the Hermite integrals per side
                nab, ncd = _cart(la) * _cart(lb), _cart(lc) * _cart(ld)
                flops += prims * (_tower(sum(cls) + 1) + 2 * _herm(lc + ld) * nab * _herm(la + lb + 1) + 2 * _herm(la + lb) * ncd)
            else:
                flops += prims * c.per_prim + quartets * c.per_quartet
    return {"bytes": float(size), "flops": float(flops)}


def tolerance(case):
    if case["kind"] in ("coulomb", "exchange") and case["mixed"]:
        return {"rel": 1e-6, "max": 1e-4}    # the Hermite towers in 32 bits
    if case["kind"] == "fock" and case["mixed"]:
        return {"rel": 1e-10, "max": 1e-8}   # the selected quartets in 32 bits, under their error budget
    # 64-bit sums in another order, or by another recurrence: 2e-14 to 2e-13
    # from `exact`, and cancelling recurrences lose up to ten times that
    return {"rel": 2e-12, "max": 1e-10}


# ---------------------------------------------------------------------------
# The same integrals in plain torch


@lru_cache(maxsize=None)
def _herms(n):
    return tuple((x, y, m - x - y) for m in range(n + 1) for x in range(m, -1, -1) for y in range(m - x, -1, -1))


def _carts(l):  # noqa: E741
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Side:
    """Primitive pairs of one class: centre P, exponent p, factor (with the
    contraction coefficients), their contracted pair, and the expansion
    E[n, rows, Hermite] of every Cartesian product (or, with `derivative`, of
    its three derivatives with respect to the first centre)."""

    def __init__(self, la, lb, A, B, al, be, co, pair, derivative=False):
        t = lambda v: torch.as_tensor(np.asarray(v, dtype=np.float64), device=_device())  # noqa: E731
        A, B, al, be = t(A), t(B), t(al), t(be)
        self.l, self.pair = la + lb + int(derivative), torch.as_tensor(np.asarray(pair), device=_device())
        self.n_pair = int(self.pair.max()) + 1
        self.p = al + be
        self.P = (al[:, None] * A + be[:, None] * B) / self.p[:, None]
        up = int(derivative)
        axes = [self._axis(la + up, lb, self.P[:, k] - A[:, k], self.P[:, k] - B[:, k],
                           torch.exp(-al * be / self.p * (A[:, k] - B[:, k]) ** 2)) for k in range(3)]

        def row(a, b):
            return torch.stack([axes[0][a[0], b[0]][x] * axes[1][a[1], b[1]][y] * axes[2][a[2], b[2]][z] for x, y, z in _herms(self.l)], 1)

        rows = []
        for k in range(3) if derivative else (None,):
            for a in _carts(la):
                for b in _carts(lb):
                    if k is None:
                        rows.append(row(a, b))
                        continue
                    r = 2 * al[:, None] * row(tuple(v + (i == k) for i, v in enumerate(a)), b)
                    if a[k]:
                        r = r - a[k] * row(tuple(v - (i == k) for i, v in enumerate(a)), b)
                    rows.append(r)
        self.E = torch.stack(rows, 1) * t(co)[:, None, None]

    def _axis(self, la, lb, pa, pb, e0):
        top, zero = self.l + 1, torch.zeros_like(e0)
        E = {(0, 0): [e0] + [zero] * top}
        for i in range(la + 1):
            for j in range(lb + 1):
                if (i, j) == (0, 0):
                    continue
                prev, x = (E[i - 1, j], pa) if i else (E[i, j - 1], pb)
                E[i, j] = [x * prev[t] + (prev[t - 1] / (2 * self.p) if t else 0) + ((t + 1) * prev[t + 1] if t < top else 0) for t in range(top + 1)]
        return E


def _boys(top, T):
    T = T.clamp(min=1e-13)
    m = top + 0.5
    F = [None] * top + [torch.special.gammainc(torch.full_like(T, m), T) * math.gamma(m) / (2 * T**m)]
    e = torch.exp(-T)
    for k in range(top, 0, -1):
        F[k - 1] = (2 * T * F[k] + e) / (2 * k - 1)
    return F


def _block(bra, ket):
    """(rows of bra | rows of ket) contracted: [bra pairs, bra rows, ket pairs, ket rows]."""
    top = bra.l + ket.l
    herm = _herms(top)
    at = {h: i for i, h in enumerate(herm)}
    hb, hk = _herms(bra.l), _herms(ket.l)
    index = torch.tensor([[at[tuple(x + y for x, y in zip(t, u))] for u in hk] for t in hb], device=_device())
    sign = torch.tensor([(-1.0) ** sum(u) for u in hk], dtype=torch.float64, device=_device())
    Ek = (ket.E * sign).transpose(1, 2).contiguous()
    nb, nk, rb, rk = len(bra.p), len(ket.p), bra.E.shape[1], ket.E.shape[1]
    out = torch.zeros((bra.n_pair, rb, ket.n_pair, rk), dtype=torch.float64, device=_device())
    step = max(1, int(1.5e8 // (nk * len(hb) * (len(hk) + rk))))
    for i in range(0, nb, step):
        P, p, n = bra.P[i:i + step], bra.p[i:i + step], min(step, nb - i)
        R = P[:, None] - ket.P[None]
        a = p[:, None] * ket.p / (p[:, None] + ket.p)
        F = _boys(top, a * (R * R).sum(-1))
        pre = 2 * math.pi**2.5 / (p[:, None] * ket.p * torch.sqrt(p[:, None] + ket.p))
        F = [f * pre * (-2 * a) ** m for m, f in enumerate(F)]
        tower = {(0, 0, 0): F}
        for h in herm[1:]:
            k = next(d for d in range(3) if h[d])
            one = tuple(v - (d == k) for d, v in enumerate(h))
            two = tuple(v - 2 * (d == k) for d, v in enumerate(h))
            more = top - sum(h) + 1
            tower[h] = [R[..., k] * tower[one][m + 1] + ((h[k] - 1) * tower[two][m + 1] if h[k] > 1 else 0) for m in range(more)]
        H = torch.stack([tower[h][0] for h in herm], 0)[index.reshape(-1)].view(len(hb), len(hk), n, nk)
        del tower
        x = torch.bmm(H.permute(3, 2, 0, 1).reshape(nk, n * len(hb), len(hk)).contiguous(), Ek)        # [ket, (bra, t), row]
        x = torch.zeros((ket.n_pair, n * len(hb), rk), dtype=torch.float64, device=_device()).index_add_(0, ket.pair, x)
        x = x.view(ket.n_pair, n, len(hb), rk).permute(1, 2, 0, 3).reshape(n, len(hb), -1).contiguous()
        x = torch.bmm(bra.E[i:i + step].contiguous(), x)                                               # [bra, row, (pair, row)]
        out.view(bra.n_pair, -1).index_add_(0, bra.pair[i:i + step], x.view(n, -1))
    return out


def _sides(basis, ordered=False, derivative=False):
    """{(la, lb): (side, [(a, b)])} of the unique (or every ordered) shell pair."""
    by = {}
    for a in range(basis.n_sh):
        for b in range(basis.n_sh) if ordered else range(a, basis.n_sh):
            s, t = basis.shells[a], basis.shells[b]
            by.setdefault((s.l, t.l), []).append((a, b))
    out = {}
    for (la, lb), prs in by.items():
        cols = [[], [], [], [], [], []]
        for k, (a, b) in enumerate(prs):
            s, t = basis.shells[a], basis.shells[b]
            for x, cx in zip(s.exponents, s.coefficients):
                for y, cy in zip(t.exponents, t.coefficients):
                    for c, v in zip(cols, (s.centre, t.centre, x, y, cx * cy, k)):
                        c.append(v)
        out[la, lb] = (_Side(la, lb, *cols, derivative=derivative), prs)
    return out


def _functions(basis, l1, l2, prs):
    """First and second function of every row of a class's pairs, [pairs, rows]."""
    ao = np.asarray(basis.shell_ao)
    a, b = np.array([p for p, _ in prs]), np.array([q for _, q in prs])
    i = ao[a][:, None, None] + np.arange(_cart(l1))[None, :, None] + 0 * np.arange(_cart(l2))
    j = ao[b][:, None, None] + 0 * np.arange(_cart(l1))[None, :, None] + np.arange(_cart(l2))
    return tuple(torch.as_tensor(v.reshape(len(prs), -1), device=_device()) for v in (i, j))


def _eri(basis):
    n = basis.n_ao
    out = torch.zeros((n * n, n * n), dtype=torch.float64, device=_device())
    sides = _sides(basis)
    names = list(sides)
    for x, cx in enumerate(names):
        bra, pb = sides[cx]
        i, j = (v.reshape(-1) for v in _functions(basis, *cx, pb))
        for cy in names[x:]:
            ket, pk = sides[cy]
            k, l = (v.reshape(-1) for v in _functions(basis, *cy, pk))  # noqa: E741
            v = _block(bra, ket).view(len(i), len(k))
            for r in (i * n + j, j * n + i):
                for c in (k * n + l, l * n + k):
                    out[r[:, None], c[None]] = v
                    out[c[:, None], r[None]] = v.t().contiguous()
    return out


def _jk(basis, D):
    n = basis.n_ao
    V = _eri(basis)
    D = torch.as_tensor(D, device=_device())
    J = (V @ D.reshape(-1)).view(n, n)
    K = (V.view(n, n, n, n).transpose(1, 2).reshape(n * n, n * n) @ D.reshape(-1)).view(n, n)
    return J, K


def _gradient(basis, D, coords):
    D = torch.as_tensor(D, device=_device())
    atom = np.repeat(np.arange(len(coords)), basis.n_sh // len(coords))
    G = torch.zeros((len(coords), 3), dtype=torch.float64, device=_device())
    kets = _sides(basis)
    for cx, (bra, pb) in _sides(basis, ordered=True, derivative=True).items():
        i, j = _functions(basis, *cx, pb)
        at = torch.as_tensor(atom[[a for a, _ in pb]], device=_device())
        for cy, (ket, pk) in kets.items():
            k, l = _functions(basis, *cy, pk)  # noqa: E741
            twice = torch.as_tensor(np.array([1.0 if c == d else 2.0 for c, d in pk]), device=_device())
            v = _block(bra, ket).view(len(pb), 3, i.shape[1], len(pk), k.shape[1])
            I, J, K, L = i[:, :, None, None], j[:, :, None, None], k[None, None], l[None, None]
            w = D[I, J] * D[K, L] - 0.25 * (D[I, K] * D[J, L] + D[I, L] * D[J, K])
            w = 2.0 * w * twice[None, None, :, None]
            G.index_add_(0, at, (v * w[:, None]).sum((2, 3, 4)))
    return G


def _fitting(basis, case, coords):
    aux = _aux(case, coords)
    sides = {}
    for m in range(5):
        s = np.nonzero(np.asarray(aux.shell_l) == m)[0]
        A = np.asarray(aux.shell_centre)[s]
        side = _Side(m, 0, A, A, aux.exps[s], 0 * aux.exps[s], aux.coefs[s], np.arange(len(s)))
        at = torch.as_tensor((np.asarray(aux.shell_ao)[s][:, None] + np.arange(_cart(m))).reshape(-1), device=_device())
        sides[m] = (side, at)
    metric = torch.zeros((aux.n_aux,) * 2, dtype=torch.float64, device=_device())
    eri3 = torch.zeros((basis.n_ao, basis.n_ao, aux.n_aux), dtype=torch.float64, device=_device())
    for ket, c in sides.values():
        for bra, r in sides.values():
            metric[r[:, None], c[None]] = _block(bra, ket).view(len(r), len(c))
        for cx, (bra, pb) in _sides(basis).items():
            i, j = (v.reshape(-1) for v in _functions(basis, *cx, pb))
            v = _block(bra, ket).view(len(i), len(c))
            eri3[i[:, None], j[:, None], c[None]] = v
            eri3[j[:, None], i[:, None], c[None]] = v
    return dict(metric=metric, eri3=eri3)


def exact(case, seed):
    kind = case["kind"]
    most = {"gradient": 8, "fitting": 9}.get(kind, 4 if case["lmax"] > 2 else 10)
    if case["atoms"] > most:
        return None
    if kind == "batch":
        out = []
        for basis, D, _ in _members(case, seed):
            J, K = _jk(basis, D)
            out.append(J - 0.5 * K)
        return out
    basis, D, coords = _molecule(case, seed)
    if kind == "gradient":
        return _gradient(basis, D, coords)
    if kind == "fitting":
        return _fitting(basis, case, coords)
    J, K = _jk(basis, D)
    if kind == "coulomb" or case.get("screen") == "j":
        return J
    return K if kind in ("exchange", "split") else J - 0.5 * K
