"""The tiled GEMM (csrc/kernels_tile.hip) at the edges of its tiles, K slices, K splits and tile sizes, against float64 NumPy."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
P3, F16 = 3, 2  # operand codes of mlh_selftest_gemm: fp32 as three bf16 planes, IEEE half


def selftest(pkg, code, a, b, r=None, swiglu=False):
    m, k = a.shape
    n = b.shape[0]
    c = np.full((m, n // 2 if swiglu else n), np.nan, dtype=np.float32)
    rc = pkg.dev.mlh_selftest_gemm(code | (0x100 if swiglu else 0), m, n, k, a.ctypes.data, b.ctypes.data,
                                   r.ctypes.data if r is not None else None, c.ctypes.data, 0, ctypes.byref(ctypes.c_double()))
    assert rc == 0
    return c


@pytest.mark.parametrize("m,n,k", [(1, 1, 32), (64, 64, 32), (65, 63, 64), (16, 768, 2048), (63, 129, 96), (130, 70, 1056), (300, 768, 768),
                                   (1900, 2100, 64), (2049, 1025, 96)])
def test_planes(pkg, m, n, k):
    """fp32 through the planes: one K slice up to a split K, 64 x 64 tiles and (many tiles) 128 x 128; the error must be
    that of fp32 sums, also where the magnitudes of a row span thirty powers of two."""
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k), dtype=np.float32) * np.exp2(rng.integers(-15, 15, (m, 1))).astype(np.float32)
    b = rng.standard_normal((n, k), dtype=np.float32)
    r = rng.standard_normal((m, n), dtype=np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64).T
    bound = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T  # |a||b|
    assert np.max(np.abs(selftest(pkg, P3, a, b) - want) / bound) <= 2e-7 * np.sqrt(k)
    assert np.max(np.abs(selftest(pkg, P3, a, b, r) - (want + r)) / (bound + np.abs(r))) <= 2e-7 * np.sqrt(k)


@pytest.mark.parametrize("code", [P3, F16])
@pytest.mark.parametrize("m,n,k", [(65, 64, 64), (129, 130, 128), (70, 62, 4096), (1500, 3000, 128)])
def test_swiglu_and_half(pkg, code, m, n, k):
    rng = np.random.default_rng(m + 3 * n + k)
    a = rng.standard_normal((m, k)).astype(np.float16).astype(np.float32)
    b = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float16).astype(np.float32)
    p = a.astype(np.float64) @ b.astype(np.float64).T
    assert np.max(np.abs(selftest(pkg, code, a, b) - p)) <= 4e-6 * np.sqrt(k) * np.max(np.abs(p)) + 1e-5
    want = p[:, 0::2] / (1 + np.exp(-p[:, 0::2])) * p[:, 1::2]
    tol = 2e-5 if code == P3 else 2.0 ** -11
    assert np.max(np.abs(selftest(pkg, code, a, b, swiglu=True) - want)) <= tol * np.max(np.abs(want)) + 2e-6 * np.sqrt(k)
