"""The window sequencer against the oracle in its largest blocks: every lane layout with a dictionary that lets a
block run to the layout's limit, with and without rows leaving the dictionary, and across calls.

Tolerance: over its life in the window a row's f is rounded w times at its own size, and a few times (16) at
its start and per block; each rounding is off by 2^-25 |f| / sqrt(3) rms. An error of f goes into the
coefficients, and through the sums over rows into estimates, with a gain of a few (4 taken). Six times the
rms of that.
"""
import numpy as np
import pytest

from helpers import small_problem, to_ri

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,dict_size,T,cuts", [(20, 900, 1100, []), (40, 700, 1500, [600]), (64, 620, 700, []), (80, 600, 1400, [3, 900]),
                                                (112, 560, 1300, []), (113, 470, 1100, []), (113, 1100, 1100, [400]), (126, 480, 1200, [477]),
                                                (126, 1200, 1200, []), (160, 500, 1200, []), (160, 1300, 1300, [324, 325])])
def test_largest_blocks(require_gpu, oracle, w, dict_size, T, cuts):
    from libapsm_amd import ApsmNomaDetectorFactory
    N, users = 6, 2
    d = small_problem(N=N, U=3, T=T, M=200, seed=w + T)
    cfg = dict(windowSize=w, dictionarySize=dict_size, eB=0.005, gaussianKernelVariance=0.1)
    det = ApsmNomaDetectorFactory.build(dict(cfg, otype="APSM"), N, users)
    for a, b in zip([0] + cuts, cuts + [T]):
        det.train(d["rx_train"][:, a:b], d["tx_train"][:users, a:b])
    est, st = np.atleast_2d(det.detect(d["rx_data"])), det.getTrainingState()
    for u in range(users):
        o = oracle.Apsm(cfg, N)
        o.train(d["rx_train"], d["tx_train"][u], incremental=True)
        ref, so = o.detect(d["rx_data"]), o.state()
        size = max(np.abs(ref).max(), np.abs(to_ri(d["tx_train"][u])).max())
        tol = 6 * 4 * 2.0 ** -25 / np.sqrt(3) * np.sqrt(w + 16 * (2 + T / 324)) * size
        e, c = np.abs(to_ri(est[u]) - ref).max(), np.abs(st["coeffs"][u] - so["coeffs"]).max()
        print(f"w {w} dict {dict_size} T {T} cuts {cuts} user {u}: soft {e:.2e} coeffs {c:.2e} of {tol:.2e}", flush=True)
        assert e <= tol and c <= tol
