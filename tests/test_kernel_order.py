"""Kernels whose waves share LDS, run from their source on the CPU
(tests/emu) with each wave in turn as far ahead of the others as the barriers
let it be: the results must not depend on which one."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = next((c for c in ("/opt/rocm/llvm/bin/clang++", shutil.which("clang++")) if c and os.path.exists(c)), None)
ORDERS = [(0, 1, 2, 3), (3, 2, 1, 0), (1, 0, 3, 2), (2, 3, 0, 1)]


def build(tmp_path_factory, name):
    if CLANG is None:
        pytest.skip("no clang++")
    so = str(tmp_path_factory.mktemp("emu") / (name + ".so"))
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-O1", "-w", "-shared", "-fPIC", "-I", os.path.join(HERE, "emu"),
                    os.path.join(HERE, "emu", name + ".cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.fixture(scope="module")
def leaf(tmp_path_factory):
    return build(tmp_path_factory, "emu_leaf")


def inverses(leaf, L, uplo, order, unit=False):
    """(inverse blocks, flags) of the kernel for the triangle of L."""
    n, dt = L.shape[0], L.dtype
    blocks = (n + 63) // 64
    A = np.asfortranarray(L)
    W = np.full((blocks, 64, 64), np.nan, dt)
    F = np.full(blocks, -1, np.int32)
    fn = leaf.emu_trtri64_f64 if dt == np.float64 else leaf.emu_trtri64_f32
    i64 = ctypes.c_int64
    assert fn(i64(n), ptr(A), i64(1), i64(n), int(uplo == "L"), int(unit), ptr(W), ptr(F),
              (ctypes.c_int * 4)(*order)) == 0
    return W.transpose(0, 2, 1), F


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("big", [0, 1, 2, 3])
def test_inverse_and_flag_do_not_depend_on_the_wave_ahead(leaf, dt, uplo, big):
    """A 64-block whose rows of one 16-row sub-block are 1000 times the others:
    kappa_1 = 1000 or more, so it is flagged for refinement, whichever wave is
    ahead; the norm of the inverse alone would not flag it.  The second block
    is well-conditioned and is not flagged.  Inverses within rounding of
    numpy's (substitution in blocks: 64 eps kappa, relative to the largest)."""
    rng = np.random.default_rng(big)
    n = 100
    L = np.tril(rng.uniform(-1, 1, (n, n)) / n, -1) + np.eye(n)
    r0 = 16 * big if uplo == "L" else 48 - 16 * big
    L[r0:r0 + 16] *= 1000.0
    A = (L if uplo == "L" else L.T).astype(dt)
    runs = [inverses(leaf, A, uplo, o) for o in ORDERS]
    for W, F in runs:
        assert list(F) == [1, 0]
        assert np.array_equal(W, runs[0][0])
    for b, o in ((0, 0), (1, 64)):
        D = A[o:o + 64, o:o + 64].astype(np.float64)
        nb = D.shape[0]
        ref = np.linalg.inv(D)
        kappa = np.abs(D).sum(0).max() * np.abs(ref).sum(0).max()
        assert np.max(np.abs(runs[0][0][b][:nb, :nb] - ref)) <= 64 * np.finfo(dt).eps * kappa * np.max(np.abs(ref))
