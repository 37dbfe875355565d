"""Least squares where antennas depend on each other: the estimates stay at the noise, with weights that
FP32 carries, and an empty antenna, or pilots too few for more than one antenna, are reported.

Tolerance: the residual may exceed that of the best fit without the dependent antenna, rounded to FP32, by
the FP32 rounding of the estimate's terms, 2 N 2^-24 sum |w||x| (at most N + 4 roundings a term).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def c64(rng, *shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


def problem(kind, N, T, seed):
    rng = np.random.default_rng(seed)
    x, noise = c64(rng, N, T), c64(rng, T)
    if kind == "equal":
        x[1] = x[0]
    elif kind == "sum":
        x[1] = x[0] * np.complex64(0.5 + 0.25j) + x[2]
    return x, (x[0] + 0.3 * x[-1] + 0.05 * noise).astype(np.complex64)


@pytest.mark.parametrize("kind,N,T", [("equal", 2, 50), ("equal", 8, 685), ("equal", 17, 300), ("equal", 64, 1000), ("sum", 4, 200),
                                      ("sum", 8, 685), ("sum", 40, 500)])
def test_dependent_antenna_keeps_the_estimates(require_gpu, kind, N, T):
    from libapsm_amd import LlsNomaDetector
    for seed in range(12):
        x, y = problem(kind, N, T, seed)
        lls = LlsNomaDetector(N)
        lls.train(x, y)
        w = np.asarray(lls.getWeightMat(), np.float64).reshape(-1)[:2 * N]
        e = np.sqrt(np.mean(np.abs(lls.detect(x) - y) ** 2))
        A = np.delete(x, 1, axis=0).astype(np.complex128).T
        best = np.sqrt(np.mean(np.abs(A @ np.linalg.lstsq(A, y.astype(np.complex128), rcond=None)[0] - y) ** 2))
        terms = (np.abs(w[:N]) + np.abs(w[N:])) @ np.abs(x).max(axis=1)
        tol = best + 2 * N * 2.0 ** -24 * terms
        print(f"{kind} N {N} T {T} seed {seed}: residual {e:.6f} of {tol:.6f}, weights to {np.abs(w).max():.3g}", flush=True)
        assert e <= tol and tol < 1.1 * best


@pytest.mark.parametrize("N,T", [(8, 4), (16, 10), (64, 40)])
def test_too_few_pilots_are_reported(require_gpu, N, T):
    from libapsm_amd import ApsmError, LlsNomaDetector
    for seed in range(5):
        x, y = problem("", N, T, seed)
        with pytest.raises(ApsmError):
            LlsNomaDetector(N).train(x, y)


@pytest.mark.parametrize("N", [1, 3, 17, 64])
def test_empty_antenna_is_reported(require_gpu, N):
    from libapsm_amd import ApsmError, LlsNomaDetector
    x, y = problem("", N, 10 * N + 20, N)
    x[N // 2] = 0
    with pytest.raises(ApsmError):
        LlsNomaDetector(N).train(x, y)
