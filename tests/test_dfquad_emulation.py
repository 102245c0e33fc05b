"""The matrix-core density-fitting kernel (csrc/fj_dfquad.h) on the CPU
against the emulated device header, under AddressSanitizer: a metric and a
three-center call with contracted and single aux shells s..g and AO shells
through f, against the oracle."""

import os
import shutil
import subprocess

import numpy as np
import pytest

from felizjueves_amd import df, gen_hip
from felizjueves_amd.basis import Basis, primitive_norm
from oracle import oracle as O
from test_gradient import CSRC, EMU, ROOT, _shell, _w


def _case():
    A, B = (0.1, -0.2, 0.3), (-0.7, 0.8, 0.4)
    basis = Basis([_shell(0, A, (2.1, 0.4), (0.4, 0.7)), _shell(2, A, (0.9,), (1.0,)), _shell(1, B, (1.7, 0.6, 0.3), (0.3, 0.5, 0.2)),
                   _shell(3, B, (0.8,), (1.0,))])
    # per momentum: more shells than a wavefront's cells, of one, two and three primitives
    l, c, n, e, k = [], [], [], [], []  # noqa: E741
    for m, sizes in enumerate(((1, 2, 1), (2, 1), (1, 1), (2,), (1, 3))):
        for j, s in enumerate(sizes):
            l.append(m)
            c.append(A if j % 2 else B)
            n.append(s)
            x = 0.5 + 0.4 * np.arange(s) + 0.3 * j
            e += list(x)
            k += [w * primitive_norm(m, a) for w, a in zip((0.7, 0.4, 0.2), x)]
    return basis, df.AuxBasis(l, c, n, e, k)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
@pytest.mark.parametrize("kind", ["metric", "eri3"])
def test_matrix_core_fitting_on_cpu_vs_oracle(kind, tmp_path):
    basis, aux = _case()
    A, alpha, s_aux, _, _ = aux.records()
    if kind == "metric":
        classes = df.metric_classes(aux)
        z3 = np.zeros((len(alpha), 3))
        bra = {"zeta_ab": alpha, "P": A, "XPA": z3, "XPB": z3, "s_ab": s_aux}
        keys = ("p_rec0", "p_rec1", "q_rec0", "q_rec1", "off_p", "off_p", "off_q")
        three = [(p, 0, q) for p, q in classes]
    else:
        classes, bra = df.eri3_classes(basis, aux)
        keys = ("ab_rec0", "ab_rec1", "p_rec0", "p_rec1", "off_a", "off_b", "off_p")
        three = list(classes)
    built = {c for unit in gen_hip.dq_classes().values() for c in unit}
    assert set(three) <= built
    (tmp_path / "gen").mkdir()
    shutil.copy(EMU / "fj_device_emu.h", tmp_path / "fj_device.h")
    shutil.copy(CSRC / "gen" / "fj_boys_table.h", tmp_path / "gen" / "fj_boys_table.h")
    names = " ".join(f"FJ_DQ_CLASS({a}, {b}, {c})" for a, b, c in three)
    r = subprocess.run(["g++", "-std=c++20", "-O1", "-g0", "-fsanitize=address", f"-I{ROOT / 'include'}", f"-I{tmp_path}",
                        f'-DDFLOOP_HEADER="{CSRC / "fj_dfloop.h"}"', f'-DDFQUAD_HEADER="{CSRC / "fj_dfquad.h"}"',
                        f"-DCLASSES={names}", str(EMU / "dfquad_emu.cpp"), "-o", str(tmp_path / "emu"), "-lpthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    n_ao = 0 if kind == "metric" else basis.n_ao
    with open(tmp_path / "case.bin", "wb") as f:
        np.array([kind == "metric", n_ao, aux.n_aux, len(classes)], dtype=np.int32).tofile(f)
        for k in ("zeta_ab", "P", "XPA", "XPB", "s_ab"):
            _w(f, bra[k], np.float64)
        for x in (A, alpha, s_aux):
            _w(f, x, np.float64)
        for l3, dc in zip(three, classes.values()):
            np.array([*l3, dc.n, 1], dtype=np.int32).tofile(f)
            for k in keys:
                _w(f, dc.arrays[k], np.int32)
    r = subprocess.run([str(tmp_path / "emu"), str(tmp_path / "case.bin"), str(tmp_path / "out.bin")], cwd=tmp_path,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"), capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    X = np.fromfile(tmp_path / "out.bin")
    Xo = O.df_metric(aux) if kind == "metric" else O.df_eri3(basis, aux)
    err = np.abs(X - Xo.ravel()).max() / np.abs(Xo).max()
    print(kind, "error", err, flush=True)
    assert err < 1e-13   # a few hundred terms in another order
