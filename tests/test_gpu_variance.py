"""The variance heuristic around its 64-pilot tiles, and at magnitudes whose squares leave the float
range (the kernel then falls back to hypotf).

Tolerance: a distance is a sum of N magnitudes of 1 ulp (2^-23) each, summed and rooted in FP32: the
root's relative error is below (N / 2 + 2) * 2^-24; the variance is its square, rounded twice.
"""
import numpy as np
import pytest

from helpers import small_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,T,scale", [(1, 3, 1.0), (3, 63, 1.0), (4, 64, 1.0), (5, 65, 1.0), (16, 129, 1.0), (64, 200, 1.0),
                                       (4, 130, 1e-13), (7, 70, 3e-10), (8, 100, 1e16), (2, 66, 1e-5)])
def test_tiles_and_magnitudes(require_gpu, oracle, N, T, scale):
    from libapsm_amd import ApsmNomaDetectorFactory
    d = small_problem(N=N, U=3, T=T, M=10, seed=T)
    rx = (d["rx_train"] * np.float32(scale)).astype(np.complex64)
    det = ApsmNomaDetectorFactory.build(dict(otype="APSM", windowSize=1, dictionarySize=T, gaussianKernelVariance=0.0), N)
    det.train(rx, d["tx_train"][0])
    got, ref = det.getTrainingState()["variance"], oracle.variance_heuristic(rx)
    tol = (N + 8) * 2.0 ** -24
    print(f"N {N} T {T} scale {scale:g}: gpu {got:.9g} oracle {ref:.9g} off {abs(got / ref - 1):.2e} of {tol:.2e}", flush=True)
    assert got == pytest.approx(ref, rel=tol)
