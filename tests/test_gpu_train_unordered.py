"""Targets that are not a number: a pilot whose symbol is unknown projects nothing (the threshold compares
unordered), and the rows around it train as if it had been met. Every lane layout of the window sequencer,
both parts or one, within a block, at its ends and across calls.

Tolerance: as the window sequencer's tests, sums of at most 1e3 terms below one in FP32, 6e-5.
"""
import numpy as np
import pytest

from helpers import small_problem, to_ri

pytestmark = pytest.mark.gpu

ATOL = 1e-4


@pytest.mark.parametrize("w,cuts,users", [(1, [], 1), (8, [], 1), (20, [70], 2), (40, [], 1), (64, [], 3), (80, [33], 1), (112, [], 1),
                                          (113, [], 1), (160, [100, 300], 2)])
def test_unknown_targets_project_nothing(require_gpu, oracle, w, cuts, users):
    from libapsm_amd import ApsmNomaDetectorFactory
    T, N = 2 * w + 240, 4
    d = small_problem(N=N, U=3, T=T, M=65, seed=w)
    tx = d["tx_train"][:users].copy()
    nan = np.float32("nan")
    for u in range(users):
        for k in (0, w // 2, w, w + 1, T // 2 + 3 * u, T - 1):
            tx[u, k] = complex(nan, nan) if k % 2 == 0 else complex(tx[u, k].real, nan) if k % 3 == 0 else complex(nan, tx[u, k].imag)
    cfg = dict(windowSize=w, dictionarySize=w + 150, eB=0.01, gaussianKernelVariance=0.1)
    det = ApsmNomaDetectorFactory.build(dict(cfg, otype="APSM"), N, users)
    for a, b in zip([0] + cuts, cuts + [T]):
        det.train(d["rx_train"][:, a:b], tx[:, a:b])
    est = np.atleast_2d(det.detect(d["rx_data"]))
    st = det.getTrainingState()
    for u in range(users):
        o = oracle.Apsm(cfg, N)
        o.train(d["rx_train"], tx[u], incremental=True)
        so = o.state()
        assert np.isfinite(so["coeffs"]).all()
        e = np.abs(to_ri(est[u]) - o.detect(d["rx_data"])).max()
        c = np.abs(st["coeffs"][u] - so["coeffs"]).max()
        print(f"w {w} cuts {cuts} user {u}: soft {e:.2e} coeffs {c:.2e}", flush=True)
        assert e <= ATOL and c <= ATOL
