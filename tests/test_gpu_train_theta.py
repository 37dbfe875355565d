"""The linear part theta = sum_j c_j x_j of a trained detector against the same sum in 64 bits over the detector's
own coefficients and pilots (the dictionary holds all of them), so that only the sum's rounding counts:
every lane layout of the window sequencer, several blocks each, the largest block of every layout among them.

Tolerance, per component: a rounding at the size of v is off by 2^-25 |v| / sqrt(3) rms at most. theta itself is
rounded once a block and a few times (at most 12) at the end, a block's rows are added in runs of m = ceil(512 N /
threads) whose partial sums are of sqrt(m) terms at most, and the end's in runs and a tree of 8: six times
the rms of (blocks + 12) |theta|^2 + (m + 8) sum (c x)^2.
"""
import numpy as np
import pytest

from helpers import small_problem
from test_gpu_detect_tiles import rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 4, 8])
@pytest.mark.parametrize("w", [1, 20, 40, 64, 80, 112, 113, 126, 160])
def test_theta_is_the_sum_over_the_coefficients(require_gpu, N, w):
    from libapsm_amd import ApsmNomaDetectorFactory
    T, users = 4000, 3
    d = small_problem(N=N, U=users, T=T, M=10, seed=w + N, mod="QAM16")
    det = ApsmNomaDetectorFactory.build(dict(otype="APSM", windowSize=w, dictionarySize=T, eB=0.001, gaussianKernelVariance=0.1), N, users)
    det.train(d["rx_train"], d["tx_train"][:users])
    st = det.getTrainingState()
    X, c = rows(d["rx_train"]), st["coeffs"].astype(np.float64)
    assert c.shape == (users, X.shape[0])
    ref = c @ X
    m = -(-512 * N // 320)
    var = (T / 300 + 12) * ref ** 2 + (m + 8) * (c ** 2 @ X ** 2)
    tol = 6 * 2.0 ** -25 / np.sqrt(3) * np.sqrt(var)
    e = np.abs(st["theta"].astype(np.float64) - ref)
    k = np.unravel_index(np.argmax(e / tol), e.shape)
    print(f"w {w} N {N}: {e[k]:.2e} of {tol[k]:.2e}", flush=True)
    assert (e <= tol).all()
