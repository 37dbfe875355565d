"""The window sequencer (sampleStep 2) at the edges of its layouts: windows at and around every
lane layout's limit, dictionaries down to the window itself (blocks of one step, rows leaving the
dictionary at every step), short streams that never fill the window, and streams cut into calls.

Tolerance: a row's f is a sum of at most 2 (dictionary + window) terms below one in FP32, each
rounded at 2^-24, so about 1e3 * 2^-24 = 6e-5; the projections contract earlier errors.
"""
import numpy as np
import pytest

from helpers import small_problem, to_ri

pytestmark = pytest.mark.gpu

ATOL = 1e-4


def run(oracle, N, T, cfg, cuts, users=1, seed=0):
    from libapsm_amd import ApsmNomaDetectorFactory
    d = small_problem(N=N, U=3, T=T, M=65, seed=seed)
    det = ApsmNomaDetectorFactory.build(dict(cfg, otype="APSM"), N, users)
    edges = [0] + cuts + [T]
    for a, b in zip(edges, edges[1:]):
        det.train(d["rx_train"][:, a:b], d["tx_train"][:users, a:b])
    est = np.atleast_2d(det.detect(d["rx_data"]))
    st = det.getTrainingState()
    for u in range(users):
        o = oracle.Apsm(cfg, N)
        o.train(d["rx_train"], d["tx_train"][u], incremental=True)
        so = o.state()
        e = np.abs(to_ri(est[u]) - o.detect(d["rx_data"])).max()
        c = np.abs(st["coeffs"][u] - so["coeffs"]).max()
        print(f"w {cfg['windowSize']} dict {cfg['dictionarySize']} T {T} cuts {cuts} user {u}: soft {e:.2e} coeffs {c:.2e}", flush=True)
        assert e <= ATOL and c <= ATOL


@pytest.mark.parametrize("w", [1, 3, 4, 19, 20, 21, 40, 41, 64, 65, 80, 81, 112, 113, 159, 160])
def test_window_layouts(require_gpu, oracle, w):
    cfg = dict(windowSize=w, dictionarySize=2 * w + 40, eB=0.01, gaussianKernelVariance=0.1)
    run(oracle, 4, 5 * w + 90, cfg, [], seed=w)


@pytest.mark.parametrize("w,dict_size", [(1, 1), (2, 2), (7, 8), (20, 20), (21, 22), (40, 40), (80, 83), (160, 160)])
def test_dictionary_near_the_window(require_gpu, oracle, w, dict_size):
    cfg = dict(windowSize=w, dictionarySize=dict_size, eB=0.001, gaussianKernelVariance=0.2)
    run(oracle, 3, dict_size + 70, cfg, [], seed=w + 1)


@pytest.mark.parametrize("w,T,cuts", [(20, 1, []), (20, 19, []), (40, 90, [1, 2, 39, 41]), (64, 700, [30, 66, 600]),
                                      (160, 900, [100, 161, 500, 501]), (10, 1100, [1])])
def test_short_and_cut_streams(require_gpu, oracle, w, T, cuts):
    cfg = dict(windowSize=w, dictionarySize=max(w, T // 2), eB=0.01, gaussianKernelVariance=0.1)
    run(oracle, 5, T, cfg, cuts, users=2, seed=T)


@pytest.mark.parametrize("N,T,cuts,users", [(1, 129, [64], 1), (16, 200, [63, 65, 130], 3), (21, 300, [128, 257], 2), (64, 260, [1, 65, 193], 1),
                                            (33, 400, [70, 320], 5)])
def test_calls_around_the_staging_tiles(require_gpu, oracle, N, T, cuts, users):
    """Pilots are staged 64 to a workgroup and kept rows copied 2048 floats to a workgroup."""
    cfg = dict(windowSize=8, dictionarySize=100, eB=0.01, gaussianKernelVariance=0.5)
    from libapsm_amd import ApsmNomaDetectorFactory
    d = small_problem(N=N, U=max(users, 3), T=T, M=65, seed=T)
    det = ApsmNomaDetectorFactory.build(dict(cfg, otype="APSM"), N, users)
    for a, b in zip([0] + cuts, cuts + [T]):
        det.train(d["rx_train"][:, a:b], d["tx_train"][:users, a:b])
    est = np.atleast_2d(det.detect(d["rx_data"]))
    st = det.getTrainingState()
    for u in range(users):
        o = oracle.Apsm(cfg, N)
        o.train(d["rx_train"], d["tx_train"][u], incremental=True)
        e = np.abs(to_ri(est[u]) - o.detect(d["rx_data"])).max()
        c = np.abs(st["coeffs"][u] - o.state()["coeffs"]).max()
        print(f"N {N} T {T} cuts {cuts} user {u}: soft {e:.2e} coeffs {c:.2e}", flush=True)
        assert e <= ATOL and c <= ATOL
