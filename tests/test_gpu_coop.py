"""GPU: the quartet-cooperative F launches against the per-lane ones of the
same plans: every class through d in both pair orders, few quartets (lanes
shared over several workgroups) and many, a density the plan was not made
with, batches, both tiers, and graph replays. Both forms run the same
recurrences in FP64 and differ in the order of their sums: 1e-13 of max|G| is
ten times what the cancelling HRR makes of that (measured 1.3e-14)."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def _pair(systems, **kw):
    from felizjueves_amd.fock import FockBuilder
    return [FockBuilder.batch(systems, tau=1e-12, coop=c, **kw) for c in (False, True)]


def _close(A, B, rel=1e-13):
    a, b = A.cpu().numpy(), B.cpu().numpy()
    err, big = np.abs(a - b).max(), np.abs(a).max()
    print(f"max|dG|={err:.2e} max|G|={big:.2e}", flush=True)
    assert big > 0 and err <= rel * max(1.0, big)


@pytest.mark.parametrize("n_atoms", [1, 2, 3, 7])
def test_cooperative_equals_per_lane(n_atoms):
    _need_gpu()
    from felizjueves_amd import native
    from felizjueves_amd.systems import closed_shell_density, config1, config2
    s = config1() if n_atoms == 3 else config2(seed=31, n_atoms=n_atoms)
    lane, coop = _pair([(s.basis, s.D)])
    rng = np.random.default_rng(8)
    for D in (s.D, closed_shell_density(rng, s.basis.n_ao, 3)):
        Dd = native.to_dev(D)
        _close(lane.build([Dd])[0], coop.build([Dd])[0])
    assert all(L.coop is None for L in lane.launches)
    assert all(L.coop is not None for L in coop.launches)
    if n_atoms == 3:
        assert max(L.coop.parts for L in coop.launches) > 1
        assert len(coop.launches) == 45   # every class pair


def test_cooperative_batch_and_streams():
    _need_gpu()
    from felizjueves_amd import native
    from felizjueves_amd.systems import config1, config2
    sy = [config1(), config2(seed=4, n_atoms=4), config2(seed=9, n_atoms=6)]
    lane, coop = _pair([(s.basis, s.D) for s in sy])
    Dd = [native.to_dev(s.D) for s in sy]
    for a, b in zip(lane.build(Dd), coop.build(Dd, n_streams=4)):
        _close(a, b)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("form", ["lane", "tuned", "some"])
def test_per_lane_launches_on_streams_and_in_a_graph(form, mixed):
    """Per-lane launches, classes with a workspace among them, alone and
    beside cooperative ones (the shipped 40-atom configuration; a few class
    pairs named) on four streams, eager and replayed, for two densities,
    against the oracle at the bars of either tier."""
    _need_gpu()
    from felizjueves_amd import autotune, native
    from felizjueves_amd.fock import FockBuilder
    from felizjueves_amd.systems import closed_shell_density, config2
    from test_builder_oracle import oracle_build
    s = config2(seed=2, n_atoms=10)
    named = {(2, 2, 2, 2): 128, (0, 2, 2, 2): 64, (1, 1, 1, 2): 256, (0, 0, 0, 0): 64}
    kw = {"lane": dict(coop=False), "some": dict(threads=named, lane_flops={c: 3e5 for c in named}),
          "tuned": autotune.builder_kwargs(autotune.load(autotune.Path(autotune.__file__).parent / "tuned" /
                                                         "c2_40atom.json"))}[form]
    fb = FockBuilder(s.basis, s.D, tau=1e-12, mixed=mixed, **kw)
    Dd = native.to_dev(s.D)
    fb.capture(Dd, n_streams=4)
    lane = [L for L in fb.launches if L.coop is None]
    assert any(native.workspace_bytes(L.cls, L.threads, len(L.work)) for L in lane)
    assert (len(lane) == len(fb.launches)) == (form == "lane")
    bar = 1e-8 if mixed else 1e-10
    for D in (s.D, closed_shell_density(np.random.default_rng(3), s.basis.n_ao, 20)):
        Dd.copy_(native.to_dev(D))
        Go = oracle_build(FockBuilder(s.basis, D, tau=1e-12), D)
        worst = 0.0
        for _ in range(3):
            worst = max(worst, np.abs(fb.replay().cpu().numpy() - Go).max())
            worst = max(worst, np.abs(fb.build(Dd, n_streams=4).cpu().numpy() - Go).max())
        print(form, mixed, "max|dG|", worst, "per-lane", len(lane), "of", len(fb.launches), flush=True)
        assert worst <= bar


def test_cooperative_tiers_and_replays():
    """A mixed build in either form: both choose tiers for the plan's items,
    and the cooperative one keeps in FP64 the quartets that lie in items of
    both tiers; they agree to the FP32 tier's error (2e-11 on this system's
    size); replays equal the eager build."""
    _need_gpu()
    from felizjueves_amd import native
    from felizjueves_amd.systems import closed_shell_density, config2
    s = config2(seed=2, n_atoms=10)
    lane, coop = _pair([(s.basis, s.D)], mixed=True)
    Dd = native.to_dev(s.D)
    Gl = lane.build([Dd])[0]
    coop.capture([Dd], n_streams=4)
    rng = np.random.default_rng(3)
    for k in range(3):
        Gc = coop.replay()[0]
        assert np.abs((Gc - Gl).cpu().numpy()).max() <= 1e-10
        assert 0 < coop.fp32_share() <= lane.fp32_share()
        Dd.copy_(native.to_dev(closed_shell_density(rng, s.basis.n_ao, 20 + k)))
        Gl = lane.build([Dd])[0]


@pytest.mark.parametrize("lane_flops", [None, 3e4])
def test_split_quartets_run_in_fp32_only_where_every_chunk_may(lane_flops):
    """The network judges a planned item by that item's features, so the items
    of a split quartet may get different tiers: after a build, a cooperative
    item is in FP32 where all the planned items under it are, and nowhere
    else; also for tiers set at random, which no launch's items share."""
    _need_gpu()
    from pathlib import Path
    from felizjueves_amd import native
    from felizjueves_amd.fock import MIXED, FockBuilder
    from felizjueves_amd.selector import LearnedSelector
    from felizjueves_amd.systems import config2
    sel = LearnedSelector.load(Path(__file__).resolve().parent.parent / "felizjueves_amd" / "tuned" / "selector")
    s = config2(seed=2, n_atoms=10)
    fb = FockBuilder(s.basis, s.D, tau=1e-12, mixed=True, selector=sel, lane_flops=lane_flops, coop=True)
    G64 = FockBuilder(s.basis, s.D, tau=1e-12).build(native.to_dev(s.D)).cpu().numpy()
    G = fb.build(native.to_dev(s.D), n_streams=4).cpu().numpy()
    assert np.abs(G - G64).max() <= 1e-8 and fb.fp32_share() > 0
    rng = np.random.default_rng(1)
    raised = 0
    for tiers in (None, 0.5, 0.9):
        if tiers is not None:
            flat = fb._cover[2]
            flat.copy_(native.to_dev((rng.random(flat.numel()) < tiers).astype(np.int32)))
            native.tier_cover(*fb._cover)
        for L in fb.launches:
            assert L.precision == MIXED and L.coop is not None
            t, got = L.tier_dev.cpu().numpy(), L.coop.tier.cpu().numpy()
            off, under = L.coop.cover
            want = np.array([t[under[a:b]].min() for a, b in zip(off, off[1:])])
            assert np.array_equal(got, want)
            raised += int((t[L.coop.parent] > got).sum())
    assert raised > 0


def test_cooperative_entry_refuses():
    _need_gpu()
    from felizjueves_amd import native
    from felizjueves_amd.systems import config1
    s = config1()
    _, fb = _pair([(s.basis, s.D)])
    fb.to_device()
    L = fb.launches[0]
    sys = fb._sys([native.to_dev(s.D)])
    d = L.coop.dev
    for parts, kets in ((0, d[1]), (65, d[1]), (1, None)):
        with pytest.raises(native.FjError):
            native.call_fc(L.cls, parts, L.bra.side, L.ket.side, d[0], 1, kets, d[2], None, sys, L.diag, fb.tau)
    assert native.coop_batch((0, 0, 3, 3)) == 0 and native.coop_batch((0, 0, 0, 0)) > 0


@pytest.mark.parametrize("screen", ["j", "k"])
@pytest.mark.parametrize("tau,n_streams", [(0.0, 1), (1e-12, 4)])
def test_split_build_without_a_plan(screen, tau, n_streams):
    """hjk.HJKBuild on the Coulomb or exchange blocks alone, eager and three
    graph replays with eager builds between them, against the oracle's sweep
    of every ordered quartet (at tau, at most 2e4 quartets below tau / 2 each
    are dropped, of either sign: 7e-11 together)."""
    _need_gpu()
    from felizjueves_amd import hjk
    from felizjueves_amd.systems import config1
    from oracle import oracle as O
    s = config1()
    ref = O.fock_ordered(s.basis, s.D)[screen == "k"]
    b = hjk.HJKBuild(s.basis, s.D, tau=tau, screen=screen)
    got = [b.run(n_streams).cpu().numpy()]
    b.capture(n_streams)
    for _ in range(3):
        got.append(b.replay().cpu().numpy())
        got.append(b.run(n_streams).cpu().numpy())
    for X in got:
        assert np.abs(X - ref).max() <= 1e-12 * max(1.0, np.abs(ref).max()) + 100 * tau
        assert np.abs(X - X.T).max() == 0.0   # closed
    print(screen, tau, "max|X - sweep|", max(np.abs(X - ref).max() for X in got), flush=True)
    assert b.quartets_computed > 0 and b.flops > 0
    with pytest.raises(RuntimeError):   # a width the split kernels refuse is refused still
        hjk.HJKBuild(s.basis, s.D, tau=tau, screen=screen, threads=100).run()
