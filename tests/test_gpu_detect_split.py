"""A recording detected in one call and in pieces gives the same bits: short FP32 calls share a dictionary's
entries out over waves, long ones take them in one wave, and both add the same sums in the same order.
Dictionaries below, at and around the 32-entry blocks, four parts and whole tiles.
"""
import numpy as np
import pytest

from helpers import small_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp32", "bf16"])
@pytest.mark.parametrize("N,users,G", [(3, 1, 1), (8, 1, 32), (8, 2, 33), (4, 1, 64), (16, 3, 95), (16, 10, 97), (7, 12, 128), (21, 1, 129),
                                       (30, 5, 160), (32, 16, 200), (32, 1, 257), (64, 1, 33), (64, 4, 65), (43, 10, 130), (64, 16, 300),
                                       (8, 1, 1000)])
def test_pieces_give_the_bits_of_the_whole(require_gpu, mode, N, users, G):
    from libapsm_amd import ApsmNomaDetectorFactory
    M, cuts = 16384 + 3000, [1, 40, 5000, 19000]
    d = small_problem(N=N, U=max(users, 3), T=G, M=M, seed=N + G)
    cfg = dict(otype="APSM", windowSize=min(G, 16), dictionarySize=G, eB=0.01, gaussianKernelVariance=0.5, detectPrecision=mode)
    det = ApsmNomaDetectorFactory.build(cfg, N, users)
    det.train(d["rx_train"], d["tx_train"][:users] if users > 1 else d["tx_train"][0])
    whole = np.atleast_2d(det.detect(d["rx_data"])).copy()
    pieces = [np.atleast_2d(det.detect(np.ascontiguousarray(d["rx_data"][:, a:b]))).copy() for a, b in zip([0] + cuts, cuts + [M])]
    print(f"{mode} N {N} users {users} G {G}", flush=True)
    np.testing.assert_array_equal(np.concatenate(pieces, axis=1), whole)
