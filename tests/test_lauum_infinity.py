"""Where an infinity of the factor goes in U*U^T / L^T*L (lauum's product
kernels, run from their source on the CPU): an element of the product is
touched only by the entries that its sum holds."""
import ctypes

import numpy as np
import pytest

from test_kernel_order import build, ptr


@pytest.fixture(scope="module")
def lauum(tmp_path_factory):
    return build(tmp_path_factory, "emu_lauum")


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("large", [0, 1])
@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("at", [(100, 50), (70, 64), (139, 3), (40, 40)])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_only_the_sums_that_hold_it(lauum, dt, large, uplo, at, value):
    n = 140
    rng = np.random.default_rng(5)
    L = np.tril(rng.standard_normal((n, n))).astype(dt)
    L[at] = value
    A = np.array(L if uplo == "L" else L.T, order="F", copy=True)
    fn = lauum.emu_lauum_f64 if dt == np.float64 else lauum.emu_lauum_f32
    assert fn(int(uplo == "L"), large, ctypes.c_int64(n), ptr(A), ctypes.c_int64(n)) == 0
    got = A if uplo == "L" else A.T
    D = L.astype(np.float64)
    with np.errstate(invalid="ignore"):
        for i in range(n):
            for j in range(i + 1):
                ref = np.sum(D[i:, i] * D[i:, j])
                bound = (n + 2) * np.finfo(dt).eps * np.sum(np.abs(D[i:, i] * D[i:, j]))
                if np.isfinite(ref):
                    assert abs(got[i, j] - ref) <= bound, (i, j)
                else:
                    assert np.array_equal(got[i, j], dt(ref), equal_nan=True), (i, j)
