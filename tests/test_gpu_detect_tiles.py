"""The matrix-core detect at the edges of its tiles: dictionaries around one and two 32-entry blocks and
one and two tiles, antenna counts with and without gaps in the rows, samples around a wave's and a
workgroup's share, one user and padded user groups.

The reference evaluates f = wL theta.x + wG sum_j c_j exp(-g |x - z_j|^2) in 64 bits from the handle's
own state. Tolerance, per output: an FP32 sum of n terms is off by at most n * 2^-24 times the sum of
their magnitudes, so the linear part by (2N + 4) * 2^-24 * sum |theta||x|, and an exponent by
d = (2N + 8) * 2^-24 * g (|x| + |z|)^2 (16-bit inputs add 2 g |x||z| times twice their half ulp), which
takes a term c_j K_j off by c_j K_j (e^d - 1); the sum over G entries and the exponential's own error
add (2G + 8) * 2^-24 * sum |c_j| K_j.
"""
import numpy as np
import pytest

from helpers import small_problem

pytestmark = pytest.mark.gpu

HALF_ULP = {"fp32-matrix": 0.0, "bf16": 2.0 ** -9, "fp16": 2.0 ** -11}


def rows(x):
    a = np.concatenate([x.real, x.imag]).T.astype(np.float64)
    b = np.concatenate([x.imag, -x.real]).T.astype(np.float64)
    return np.stack([a, b], axis=1).reshape(-1, a.shape[1])


def check(mode, N, G, M, users):
    from libapsm_amd import ApsmNomaDetectorFactory
    d = small_problem(N=N, U=max(users, 3), T=G, M=M, seed=N + G + M)
    cfg = dict(otype="APSM", windowSize=min(G, 16), dictionarySize=G, eB=0.01, gaussianKernelVariance=0.5, detectPrecision=mode)
    det = ApsmNomaDetectorFactory.build(cfg, N, users)
    det.train(d["rx_train"], d["tx_train"][:users] if users > 1 else d["tx_train"][0])
    est = np.atleast_2d(det.detect(d["rx_data"]))
    st = det.getTrainingState()
    X, Z = rows(d["rx_data"]), rows(d["rx_train"])
    c, theta = st["coeffs"].astype(np.float64), st["theta"].astype(np.float64)
    assert c.shape == (users, Z.shape[0])
    g = 0.5 / st["variance"]
    xn, zn = np.linalg.norm(X, axis=1)[:, None], np.linalg.norm(Z, axis=1)[None, :]
    K = np.exp(-g * np.maximum(xn ** 2 + zn ** 2 - 2 * X @ Z.T, 0))
    f = 0.5 * X @ theta.T + 0.5 * K @ c.T
    eps = 2.0 ** -24
    off = (2 * N + 8) * eps * g * (xn + zn) ** 2 + 4 * g * HALF_ULP[mode] * xn * zn
    tol = 0.5 * (2 * N + 4) * eps * np.abs(X) @ np.abs(theta).T \
        + 0.5 * (K * (np.expm1(off) + (2 * G + 8) * eps)) @ np.abs(c).T + eps
    for u in range(users):
        got = np.stack([est[u].real, est[u].imag], axis=1).reshape(-1)
        e = np.abs(got - f[:, u])
        print(f"{mode} N {N} G {G} M {M} user {u} of {users}: {e.max():.2e} of {tol[np.argmax(e / tol[:, u]), u]:.2e}", flush=True)
        assert (e <= tol[:, u]).all()


@pytest.mark.parametrize("mode", list(HALF_ULP))
@pytest.mark.parametrize("N", [2, 4, 7, 8, 13, 16, 30, 32, 43, 64])
@pytest.mark.parametrize("G", [1, 32, 33, 64, 97, 130])
def test_tile_edges(require_gpu, mode, N, G):
    check(mode, N, G, 129, 1)


@pytest.mark.parametrize("M", [1, 31, 33, 128, 257])
@pytest.mark.parametrize("N,users", [(5, 2), (8, 3), (16, 5), (32, 8), (64, 10), (21, 16), (8, 9), (16, 13)])
def test_samples_and_user_groups(require_gpu, M, N, users):
    check("fp32-matrix", N, 70, M, users)


@pytest.mark.parametrize("M", [16384, 16385])
@pytest.mark.parametrize("N,G,users", [(3, 1, 1), (8, 33, 3), (16, 97, 1), (32, 130, 2), (64, 65, 1), (13, 200, 10)])
def test_around_the_parts_rule(require_gpu, M, N, G, users):
    """The last call whose dictionary entries are shared out over waves, and the first that is not."""
    check("fp32-matrix", N, G, M, users)


def test_batch_by_parts_equals_single_handles(require_gpu):
    """Calls by parts: a batch keeps the parts' sums apart in one wave (up to 4 users) or shares them out."""
    from libapsm_amd import ApsmBatch, ApsmNomaDetectorFactory
    shapes = [(2, 1, 40, 70), (8, 1, 200, 300), (16, 3, 150, 64), (30, 9, 260, 129), (32, 4, 33, 31), (64, 2, 100, 257), (64, 12, 70, 65),
              (16, 1, 90, 17000)]
    data = [small_problem(N=N, U=max(U, 3), T=T, M=M, seed=N + U) for N, U, T, M in shapes]
    cfgs = [dict(windowSize=10, dictionarySize=T, eB=0.01, gaussianKernelVariance=0.5) for _, _, T, _ in shapes]
    b = ApsmBatch(cfgs, [s[0] for s in shapes], [s[1] for s in shapes])
    b.plan([d["rx_train"] for d in data], [d["tx_train"][:s[1]] for d, s in zip(data, shapes)], [d["rx_data"] for d in data])
    b.synchronize()
    for i, ((N, U, T, M), d, cfg) in enumerate(zip(shapes, data, cfgs)):
        print(f"instance {i}: N {N} users {U} T {T} M {M}", flush=True)
        det = ApsmNomaDetectorFactory.build(dict(cfg, otype="APSM"), N, U)
        det.train(d["rx_train"], d["tx_train"][:U] if U > 1 else d["tx_train"][0])
        np.testing.assert_array_equal(np.atleast_2d(b.estimates(i)), np.atleast_2d(det.detect(d["rx_data"])).astype(np.complex64))
