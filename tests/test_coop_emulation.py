"""The quartet-cooperative F kernels on the CPU: a class's generated kernel
run unchanged against the emulated device header (tests/emu) under
AddressSanitizer, over the builder's work list of a two-atom s,s,p,d system
(pairs in both orders), against the oracle's launch of the same tables; and
the work list against the plan it is made from."""

import os
import shutil
import subprocess

import numpy as np
import pytest

from felizjueves_amd import fock, gen_hip
from felizjueves_amd import pairs as P
from oracle import oracle as O
from test_builder_oracle import builder_tables_host
from test_kernel_emulation import EMU, ROOT


def _builder(**kw):
    from felizjueves_amd.basis import Basis
    from felizjueves_amd.systems import atom_shells, closed_shell_density
    rng = np.random.default_rng(5)
    shells = atom_shells(rng, (0.0, 0.0, 0.0)) + atom_shells(rng, (0.9, -1.1, 1.2))
    basis = Basis(shells)
    D = closed_shell_density(rng, basis.n_ao, 6)
    return fock.FockBuilder(basis, D, tau=1e-12, planner="python", **kw), D


# one class with each boundary: no HRR, one side's, both; Boys columns from
# the global table and in LDS; one and several VRR groups; lanes shared over
# two workgroups; batches of two kets (a batch edge within an item); a batch
# of every ket of the class; and (batch None) the plan's own items, which hold
# chunks of the bra's and of the kets' primitives
CASES = [((0, 0, 0, 0), 1, 32), ((0, 1, 0, 1), 2, 2), ((1, 0, 1, 1), 1, 3), ((0, 2, 1, 2), 1, 2), ((0, 1, 2, 2), 2, 32),
         ((0, 1, 1, 1), 2, None)]


def run_work_list(fb, D, L, work, kets, parent, parts, tmp_path, flags):
    """F of launch L's class from the emulated kernel over a work list, and
    from the oracle's launch of the same tables."""
    b = fb.basis
    host = builder_tables_host(fb)
    Dsh = P.density_blocks(b, D)
    exe = tmp_path / "emu"
    r = subprocess.run(["g++", "-std=c++20", "-O1", "-g0", "-fsanitize=address", f"-I{ROOT / 'include'}", f"-I{tmp_path}",
                        *flags, str(EMU / "coop_emu.cpp"), "-o", str(exe), "-lpthread"], cwd=tmp_path,
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    with open(tmp_path / "case.bin", "wb") as f:
        np.array([L.bra.n, L.ket.n, len(work), parts, b.n_sh, b.n_ao, L.diag], dtype=np.int32).tofile(f)
        np.array([fb.tau]).tofile(f)

        def put(x, dt):
            x = np.ascontiguousarray(x, dtype=dt).ravel()
            np.array([x.size], dtype=np.int64).tofile(f)
            x.tofile(f)
        for c in (L.cls[:2], L.cls[2:]):
            t = host[c]
            for k, dt in (("prim", "f8"), ("off", "i4"), ("sep", "f8"), ("G", "f8"), ("sh", "i4"), ("ao", "i4")):
                put(t[k], dt)
        for x, dt in ((work, "i4"), (kets, "i4"), (parent, "i4"), (np.zeros(len(L.work)), "i4"), (Dsh, "f8"), (D, "f8")):
            put(x, dt)
    r = subprocess.run([str(exe), str(tmp_path / "case.bin"), str(tmp_path / "F.bin")], cwd=tmp_path,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"), capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    F = np.fromfile(tmp_path / "F.bin").reshape(b.n_ao, b.n_ao)
    Fo = np.zeros_like(F)
    O.fx_launch(L.cls, host[L.cls[:2]], host[L.cls[2:]], L.diag, b.n_sh, b.n_ao, fb.tau, Dsh, D, Fo, pre=True)
    assert np.abs(Fo).max() > 0
    return F, Fo


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
@pytest.mark.parametrize("cls,parts,batch", CASES)
def test_cooperative_kernel_on_cpu_vs_oracle(cls, parts, batch, tmp_path):
    fb, D = _builder(**(dict(lane_flops=1e3) if batch is None else {}))
    L = [x for x in fb.launches if x.cls == cls][0]
    # items of up to 64 kets, so that the kernel takes several batches per item
    if batch is None:
        work, kets, parent = L.work, L.ket_list, np.arange(len(L.work))
        assert (work[:, 2] >> 16).any() and (kets >> 17).any()
    else:
        work, kets, parent = fock.coop_items(L.work, L.ket_list, 64 if batch == 2 else batch)
    name = "".join(map(str, cls))
    gen_hip.generate([], tmp_path / "gen")
    gen_hip.generate_coop([cls], tmp_path / "gen")
    if batch == 2:
        h = tmp_path / "gen" / f"c_{name}.h"
        n = gen_hip.coop_shape(cls)["nq"]
        t = h.read_text()
        assert f"min({n}, (w.w - first" in t and f"first += step * {n})" in t
        h.write_text(t.replace(f"min({n}, (w.w - first", "min(2, (w.w - first").replace(f"first += step * {n})", "first += step * 2)"))
    shutil.copy(EMU / "fj_device_emu.h", tmp_path / "fj_device.h")
    shutil.copy(ROOT / "felizjueves_amd" / "csrc" / "fj_coop.h", tmp_path / "fj_coop.h")
    F, Fo = run_work_list(fb, D, L, work, kets, parent, parts, tmp_path,
                          [f'-DCLS_HEADER="gen/c_{name}.h"', f"-DKERNEL=fj_c_{name}_k"])
    # the same recurrences, summed over primitives in another order
    assert np.abs(F - Fo).max() <= 1e-12 * max(1.0, np.abs(Fo).max())


@pytest.mark.parametrize("kw", [dict(), dict(lane_flops=1e3), dict(lane_flops=1e30), dict(mixed=True)])
@pytest.mark.parametrize("batch", [1, 3, 32])
def test_cooperative_items_are_the_plan(kw, batch):
    """Every quartet of a plan once, whole, in an item of its bra and parent."""
    fb, _ = _builder(**kw)
    for L in fb.launches:
        work, kets, parent = fock.coop_items(L.work, L.ket_list, batch)
        planned = set()
        for b, k0, z, k1 in L.work:
            planned |= {(int(b), int(e) & 0x1ffff) for e in L.ket_list[k0:k1]}
        got = []
        for (b, k0, z, k1), p in zip(work, parent):
            assert 0 < k1 - k0 <= batch and L.work[p][0] == b and z == L.work[p][2] & 0xffff
            got += [(int(b), int(k)) for k in kets[k0:k1]]
        assert len(got) == len(set(got)) and set(got) == planned


@pytest.mark.parametrize("kw", [dict(), dict(lane_flops=1e3), dict(lane_flops=3e4), dict(lane_flops=1e30)])
def test_cooperative_items_know_every_planned_item_under_them(kw):
    """A quartet's chunks may lie in several planned items, each with a tier
    of its own: the item that takes the quartet whole names all of them."""
    fb, _ = _builder(mixed=True, **kw)
    several = 0
    for L in fb.launches:
        items = fock.coop_items(L.work, L.ket_list, 3)
        off, under = fock.coop_cover(L.work, L.ket_list, items)
        holds: dict = {}   # (bra, ket) -> planned items with a chunk of it
        for p, (b, k0, z, k1) in enumerate(L.work):
            for e in L.ket_list[k0:k1]:
                holds.setdefault((int(b), int(e) & 0x1ffff), set()).add(p)
        work, kets, parent = items
        assert len(off) == len(work) + 1 and off[-1] == len(under)
        for i, (b, k0, z, k1) in enumerate(work):
            want = set().union(*(holds[int(b), int(k)] for k in kets[k0:k1]))
            assert set(under[off[i]:off[i + 1]].tolist()) == want and parent[i] in want
            several += len(want) > 1
    assert (several > 0) == (kw != dict(lane_flops=1e30))


def test_the_form_of_a_launch(monkeypatch):
    """A launch past its class pair's PER_LANE_QUARTETS keeps the per-lane form
    by default; coop says otherwise, and a class pair without a line, or a
    shaped one, has no such choice."""
    monkeypatch.setattr(fock.native, "coop_batch", lambda cls: 4)
    monkeypatch.setattr(fock.native, "to_dev", lambda x: x)
    fb, _ = _builder()
    lines = 0
    for L in fb.launches:
        line = fock.PER_LANE_QUARTETS.get(L.cls)
        for n, per_lane in ((1, False), (10 ** 9, line is not None)) + (((line - 1, False), (line, True)) if line else ()):
            L.n_quartets = n
            for coop, want in ((None, per_lane), (True, False), (False, True), ({L.cls}, False), (set(), per_lane)):
                fb.coop = coop
                assert (fb._coop(L) is None) == want, (L.cls, n, coop)
        lines += line is not None
        fb.coop, fb.class_threads = None, {L.cls: 64}
        L.n_quartets = 1
        assert fb._coop(L) is None
        fb.class_threads = {}
    assert lines == len(fock.PER_LANE_QUARTETS)


def test_the_tuner_chooses_between_the_forms(monkeypatch):
    """A class pair over COOP_MARGIN faster cooperatively than in its best
    per-lane shape is tuned to that form, any other to its shape, and the
    configuration builds so whatever the default rule says."""
    from felizjueves_amd import autotune
    monkeypatch.setattr(fock.native, "coop_batch", lambda cls: 4)
    monkeypatch.setattr(fock.native, "to_dev", lambda x: x)
    monkeypatch.setattr(fock, "PER_LANE_QUARTETS", {(0, 0, 0, 0): 1})
    fb, D = _builder()

    def launch_times(fb, D_devs, reps=3):   # (pp|dd) cooperatively 1% faster than the best shape, the rest 20%
        for L in fb.launches:
            L.coop = fb._coop(L)
        return {L.cls: (0.99 if L.cls == (1, 1, 2, 2) else 0.8) if L.coop is not None
                else 1.0 + abs(L.threads - 128) / 64 for L in fb.launches}
    monkeypatch.setattr(autotune, "launch_times", launch_times)
    monkeypatch.setattr(autotune, "build_time", lambda fb, D_devs, n, steps=10: float(n))
    cfg = autotune.tune([(fb.basis, D)], planner="python")
    assert cfg["threads"] == {"1122": 128} and set(cfg["lane_flops"]) == {"1122"} and cfg["n_streams"] == 1
    assert cfg["cooperative_ms"]["1122"] == [1.0, 0.99] and cfg["cooperative_ms"]["0000"] == [1.0, 0.8]
    assert len(cfg["coop"]) == len(fb.launches) - 1
    tuned = fock.FockBuilder(fb.basis, D, planner="python", **autotune.builder_kwargs(cfg))
    assert {L.cls for L in tuned.launches if tuned._coop(L) is None} == {(1, 1, 2, 2)}
    cfg.pop("coop")   # an older configuration: the default rule
    old = fock.FockBuilder(fb.basis, D, planner="python", **autotune.builder_kwargs(cfg))
    assert {L.cls for L in old.launches if old._coop(L) is None} == {(1, 1, 2, 2), (0, 0, 0, 0)}
