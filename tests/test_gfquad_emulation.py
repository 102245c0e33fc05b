"""The matrix-core gradient kernel (csrc/fj_gfquad.h) on the CPU against the
emulated device header, under AddressSanitizer: every launch of a two-atom
s, d / p stream (every class), quartets in pieces that cut
through their rows of primitives, and deeper contractions, whose bra rows
take several batches and whose ket primitives several passes, against the
oracle."""

import os
import shutil
import subprocess

import numpy as np
import pytest

from felizjueves_amd import gen_hip
from felizjueves_amd import gradient as GR
from oracle import oracle as O
from felizjueves_amd.basis import Basis
from felizjueves_amd.systems import closed_shell_density
from test_gradient import CSRC, EMU, ROOT, _shell, _w

QUAD = CSRC / "fj_gfquad.h"


def _build(td, classes):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    (td / "gen").mkdir()
    shutil.copy(EMU / "fj_device_emu.h", td / "fj_device.h")
    shutil.copy(CSRC / "gen" / "fj_boys_table.h", td / "gen" / "fj_boys_table.h")
    cases = " ".join(f"FJ_GQ_CLASS({a}, {b}, {c}, {d})" for a, b, c, d in classes)
    r = subprocess.run(["g++", "-std=c++20", "-O1", "-g0", "-fsanitize=address", f"-I{ROOT / 'include'}", f"-I{td}",
                        f'-DGFLOOP_HEADER="{CSRC / "fj_gfloop.h"}"', f'-DGFQUAD_HEADER="{QUAD}"', f"-DCLASSES={cases}",
                        str(EMU / "gfquad_emu.cpp"), "-o", str(td / "emu"), "-lpthread"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return td / "emu"


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return _build(tmp_path_factory.mktemp("gfquad"), gen_hip.gf_classes())


def _system():
    # every class once, one, two or four primitive pairs a side: so many columns
    # j for the wavefronts, and one batch of i, not full
    A, B = (0.1, -0.2, 0.3), (-0.7, 0.8, 0.4)
    basis = Basis([_shell(0, A, (2.1, 0.4), (0.4, 0.7)), _shell(2, A, (0.9,), (1.0,)), _shell(1, B, (1.7, 0.6), (0.3, 0.5))])
    return basis, [0, 0, 1], closed_shell_density(np.random.default_rng(3), basis.n_ao, 3)


def _gradient(exe, td, basis, at, D, pieces):
    st = GR.gf_launches(basis, at)
    with open(td / "case.bin", "wb") as f:
        np.array([len(st.launches), 2, basis.n_ao], dtype=np.int32).tofile(f)
        _w(f, D, np.float64)
        for L in st.launches:
            b, k = st.sides[L.bra], st.sides[L.ket]
            chunk = -(-b.degree * k.degree // pieces)
            np.array([*L.cls, b.n, k.n, b.degree, k.degree, 2, basis.n_ao, L.diag, chunk], dtype=np.int32).tofile(f)
            for s in (b, k):
                _w(f, s.prim, np.float64)
                _w(f, s.sep, np.float64)
                _w(f, s.sh, np.int32)
                _w(f, s.ao, np.int32)
                _w(f, s.at, np.int32)
    r = subprocess.run([str(exe), str(td / "case.bin"), str(td / "G.bin")], cwd=td,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"), capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-3000:]
    G = np.fromfile(td / "G.bin").reshape(2, 3)
    Go = O.grad_ordered(basis, at, 2, D)
    err = np.abs(G - Go).max()
    print("error", err, "scale", np.abs(Go).max(), flush=True)
    # sums of a few thousand terms of the gradient's size in another order
    assert err <= 1e-12 * np.abs(Go).max()
    return st


def test_matrix_core_gradient_on_cpu_vs_oracle(exe, tmp_path):
    basis, at, D = _system()
    # a quartet in three pieces, not whole rows: items share a bra primitive
    st = _gradient(exe, tmp_path, basis, at, D, 3)
    assert {L.cls for L in st.launches} == set(gen_hip.gf_classes())


# (l, primitives) of a shell on either atom; bra batches of the classes: 64
# rows at (ss|ss), 12 at (pp|pp), 4 at (dd|dd), 6 at (sd|dd)
DEEP = {"s": ((0, 9), (0, 1)), "p": ((1, 5), (1, 1)), "d": ((2, 3), (2, 1)), "sd": ((0, 4), (2, 2))}


@pytest.fixture(scope="module")
def deep_exe(tmp_path_factory):
    return _build(tmp_path_factory.mktemp("gfdeep"), [(0, 0, 0, 0), (1, 1, 1, 1), (2, 2, 2, 2), (0, 0, 0, 2), (0, 0, 2, 2),
                                                      (0, 2, 0, 2), (0, 2, 2, 2)])


@pytest.mark.parametrize("name,pieces", [("s", 1), ("s", 9), ("p", 1), ("p", 20), ("d", 1), ("d", 5), ("sd", 1), ("sd", 3)])
def test_matrix_core_gradient_of_deep_contractions(name, pieces, deep_exe, tmp_path):
    """Several batches of a bra's rows (the tables and weights in LDS
    rewritten) and several passes over the ket's primitives, the last of them
    with idle wavefronts (5, 9, 25 and 81 primitives by fours, 3 alone); whole
    quartets, and pieces that cut the ket's primitives alone and the bra's
    rows too, some of them left empty."""
    (l0, n0), (l1, n1) = DEEP[name]
    e = lambda n, x: tuple(x * 1.7 ** -np.arange(n))   # noqa: E731
    c = lambda n: tuple(0.6 - 0.05 * np.arange(n))   # noqa: E731
    basis = Basis([_shell(l0, (0.1, -0.2, 0.3), e(n0, 3.0), c(n0)), _shell(l1, (-0.7, 0.8, 0.4), e(n1, 0.9), c(n1))])
    D = closed_shell_density(np.random.default_rng(3), basis.n_ao, min(3, basis.n_ao - 1))
    _gradient(deep_exe, tmp_path, basis, [0, 1], D, pieces)


@pytest.mark.parametrize("cls", [(0, 0, 0, 0), (0, 1, 0, 2), (1, 1, 2, 2), (2, 2, 2, 2)])
@pytest.mark.parametrize("k_ab,k_cd,pieces", [(36, 36, 37), (1, 36, 37), (36, 1, 37), (5, 9, 4), (7, 5, 12), (3, 9, 9), (4, 4, 1),
                                              (81, 2, 2048)])
def test_pieces_cut_the_ket_before_the_rows(cls, k_ab, k_cd, pieces):
    """The pieces that a chunk makes in the kernel are ranges of whole passes
    over the ket first, then of at least two steps' rows (but for a last
    remainder's share)."""
    n = -(-k_ab * k_cd // GR.quad_chunk(cls, k_ab, k_cd, pieces))   # as fj_gfquad.h has it
    pj = min(n, -(-k_cd // 4))
    pi = min(n // pj, k_ab)
    rows = 2 * GR.quad_rows(cls) * (4 if k_cd == 1 else 2 if k_cd == 2 else 1)
    assert pj == min(pieces, -(-k_cd // 4)) and pj * pi <= n
    assert pj * pi <= pieces + pj - 1 and pi <= -(-k_ab // rows)
    assert pj * pi >= min(pieces, pj * -(-k_ab // rows)) or pi == n // pj
