"""Least squares at the edges of its blocks: antenna counts around the 16-antenna blocks of the normal
matrix and of the solve, pilot counts around a step, a wave's and a workgroup's share, and the general
real matrix around the solve's block sizes.

Tolerance: the normal equations and the solve run in FP64 on exact products (the general matrix sums at
most 64 KB of rows in FP32 first, each sum off by at most 16384 / (n + 1) * 2^-24 of its magnitude),
so the weights, rounded to FP32, are within the rounding and the FP64 (FP32) error times the condition
number cond(A)^2 of A^T A.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def embed(x):
    a = np.concatenate([x.real, x.imag]).T.astype(np.float64)
    b = np.concatenate([x.imag, -x.real]).T.astype(np.float64)
    return a, b


def c64(rng, *shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


@pytest.mark.parametrize("N", [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64])
@pytest.mark.parametrize("T", [200, 1031])
def test_antenna_blocks(require_gpu, N, T):
    run(N, T)


@pytest.mark.parametrize("N,T", [(1, 1), (1, 2), (3, 7), (3, 8), (3, 9), (3, 31), (3, 33), (3, 127), (3, 129), (5, 255), (3, 16384),
                                 (3, 16385), (4, 16417), (2, 40003)])
def test_pilot_shares(require_gpu, N, T):
    run(N, T)


def run(N, T):
    from libapsm_amd import LlsNomaDetector
    rng = np.random.default_rng(N * 100003 + T)
    x = c64(rng, N, T)
    y = (c64(rng, 1, N) @ x)[0] + 0.1 * c64(rng, T)
    y = y.astype(np.complex64)
    lls = LlsNomaDetector(N)
    lls.train(x, y)
    w = np.asarray(lls.getWeightMat(), np.float64).reshape(-1)[:2 * N]
    a, b = embed(x)
    A, t = np.concatenate([a, b]), np.concatenate([y.real, y.imag]).astype(np.float64)
    ref, _, _, sv = np.linalg.lstsq(A, t, rcond=None)
    cond2 = (sv[0] / sv[-1]) ** 2
    tol = (2.0 ** -24 + 100 * N * 2.0 ** -52 * cond2) * np.linalg.norm(ref)
    e = np.abs(w - ref).max()
    print(f"N {N} T {T}: {e:.2e} of {tol:.2e}", flush=True)
    assert e <= tol


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 32, 33, 64, 65, 100, 127, 128])
def test_general_matrix(require_gpu, n):
    from libapsm_amd import LlsNomaDetector
    from libapsm_amd._lib import DeviceArray
    rng = np.random.default_rng(n)
    m = 5 * n + 40
    A = rng.standard_normal((m, n)).astype(np.float32)
    y = rng.standard_normal(m).astype(np.float32)
    dA, dy = DeviceArray(np.ascontiguousarray(A.T)), DeviceArray(y)
    lls = LlsNomaDetector(64)
    lls.trainLowLevel(dA.ptr, dy.ptr, n, 1, m)
    w = np.asarray(lls.getWeightMat(), np.float64).reshape(-1)[:n]
    ref, _, _, sv = np.linalg.lstsq(A.astype(np.float64), y.astype(np.float64), rcond=None)
    rows = min(m, 16384 // (n + 1))
    tol = (2.0 ** -24 + rows * 2.0 ** -24 * (sv[0] / sv[-1]) ** 2) * max(np.linalg.norm(ref), np.linalg.norm(y) / sv[-1])
    e = np.abs(w - ref).max()
    print(f"n {n}: {e:.2e} of {tol:.2e}", flush=True)
    assert e <= tol
