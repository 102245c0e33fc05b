"""The matrix-core F kernel (csrc/fj_fquad.h) on the CPU against the emulated
device header, under AddressSanitizer: classes of every split of the bra over
the wavefronts (one, two and four to a tower; one p), with more bra
primitives than a step takes, and over builder work lists with chunks of the
bra's and the kets' primitives and each item's kets in slices, against the
oracle."""

import shutil
import subprocess

import numpy as np
import pytest

from felizjueves_amd import fock, gen_hip, pairs as P
from felizjueves_amd.basis import Basis
from felizjueves_amd.hgp import builder_classes
from oracle import oracle as O
from test_coop_emulation import run_work_list
from test_kloop_emulation import CSRC, EMU, ROOT, _run, _shell

CLASSES = {
    "alone": [(0, 0, 0, 3), (0, 0, 3, 3), (0, 1, 2, 3), (0, 3, 0, 3), (0, 3, 2, 2), (1, 2, 1, 3), (1, 3, 2, 3)],
    "shared": [(2, 2, 2, 3), (2, 3, 3, 3), (3, 3, 3, 3)],
}


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
@pytest.mark.parametrize("kind", list(CLASSES))
def test_matrix_core_fock_on_cpu_vs_oracle(kind, tmp_path):
    classes = CLASSES[kind]
    built = {c for cs in gen_hip.fq_units([c for c in builder_classes(3) if max(c) == 3]).values() for c in cs}
    assert set(classes) <= built
    A, B = (0.0, 0.0, 0.0), (0.7, -1.1, 1.3)
    basis = Basis([_shell(0, A, (3.1, 0.9, 0.3), (0.3, 0.5, 0.4)), _shell(3, A, (0.7,), (1.0,)),
                   _shell(1, B, (1.9, 0.6), (0.4, 0.7)), _shell(2, B, (0.9,), (1.0,))])
    D = np.random.default_rng(5).normal(size=(basis.n_ao,) * 2)
    D = 0.1 * (D + D.T)
    plan = P.f_launches(basis, D, tau=0.0, n=1)
    Dsh = P.density_blocks(basis, D)
    launches = [L for L in plan.launches if L.cls in classes]
    assert {L.cls for L in launches} == set(classes)
    (tmp_path / "gen").mkdir()
    shutil.copy(EMU / "fj_device_emu.h", tmp_path / "fj_device.h")
    shutil.copy(CSRC / "gen" / "fj_boys_table.h", tmp_path / "gen" / "fj_boys_table.h")
    names = " ".join("FJ_FQ_CLASS({}, {}, {}, {})".format(*c) for c in classes)
    r = subprocess.run(["g++", "-std=c++20", "-O1", "-g0", "-fsanitize=address", f"-I{ROOT / 'include'}", f"-I{tmp_path}",
                        f'-DFQUAD_HEADER="{CSRC / "fj_fquad.h"}"', f"-DCLASSES={names}", str(EMU / "fquad_emu.cpp"),
                        "-o", str(tmp_path / "emu"), "-lpthread"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    Fo = np.zeros((basis.n_ao,) * 2)
    with open(tmp_path / "case.bin", "wb") as f:
        np.array([len(launches), basis.n_ao], dtype=np.int32).tofile(f)
        for L in launches:
            a = P.launch_args(basis, plan, L, D, Dsh)
            O.f_launch(L.cls, a, Fo)
            np.array([*L.cls, a["n_bra"], a["n_ket"], a["k_ab"], a["k_cd"], a["n_sh"], a["n_ao"], a["diag"]],
                     dtype=np.int32).tofile(f)
            np.array([a["tau"]], dtype=np.float64).tofile(f)
            for key, dt in (("bra_prim", float), ("AB", float), ("G_ab", float), ("bra_sh", np.int32), ("bra_ao", np.int32),
                            ("ket_prim", float), ("CD", float), ("G_cd", float), ("ket_sh", np.int32),
                            ("ket_ao", np.int32), ("Dsh", float), ("D", float)):
                if (key == "AB" and not L.cls[1]) or (key == "CD" and not L.cls[3]):
                    continue
                x = np.ascontiguousarray(a[key], dtype=dt).ravel()
                np.array([x.size], dtype=np.int64).tofile(f)
                x.tofile(f)
    F = _run(tmp_path / "emu", tmp_path, "F.bin").reshape(Fo.shape)
    # both expand in the same Hermite integrals: rounding, as the loop form's test
    assert np.abs(F - Fo).max() <= 1e-12 * max(1.0, np.abs(Fo).max())


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
@pytest.mark.parametrize("cls,lane_flops,slices", [((0, 1, 1, 3), 2e3, 3), ((0, 0, 2, 3), 2e3, 1), ((1, 2, 1, 3), 1e30, 2),
                                                   ((2, 2, 2, 3), 1e30, 1)])
def test_matrix_core_fock_over_work_lists(cls, lane_flops, slices, tmp_path):
    """As the builder launches it: `span` 64 kets to an item, its kets over
    `slices` workgroups."""
    A, B = (0.0, 0.0, 0.0), (0.7, -1.1, 1.3)
    basis = Basis([_shell(0, A, (3.1, 0.9, 0.3), (0.3, 0.5, 0.4)), _shell(3, A, (0.7, 0.4), (0.6, 0.5)),
                   _shell(1, B, (1.9, 0.6), (0.4, 0.7)), _shell(2, B, (0.9, 0.5), (0.6, 0.5)),
                   _shell(0, B, (0.8, 0.2), (0.5, 0.6))])
    D = np.random.default_rng(5).normal(size=(basis.n_ao,) * 2)
    D = 0.1 * (D + D.T)
    fb = fock.FockBuilder(basis, D, tau=1e-12, planner="python", lane_flops=lane_flops)
    L = [x for x in fb.launches if x.cls == cls][0]
    if lane_flops < 1e30:
        assert (L.work[:, 2] >> 16).any() and (L.ket_list >> 17).any()
    shutil.copy(EMU / "fj_device_emu.h", tmp_path / "fj_device.h")
    (tmp_path / "gen").mkdir()
    shutil.copy(CSRC / "gen" / "fj_boys_table.h", tmp_path / "gen" / "fj_boys_table.h")
    t = ", ".join(map(str, cls))
    F, Fo = run_work_list(fb, D, L, L.work, L.ket_list, np.arange(len(L.work)), slices, tmp_path,
                          [f'-DCLS_HEADER="{CSRC / "fj_fquad.h"}"', f"-DCALL=fj_fquad_k<{t}>(64, a)",
                           f"-DGRID_Z=Fq<{t}>::Z"])
    assert np.abs(F - Fo).max() <= 1e-12 * max(1.0, np.abs(Fo).max())
