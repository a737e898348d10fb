"""Truncated pivoted QR at the edges of its blocks of 16 deferred reflectors: ranks below, at
and past a block, tiles of one row or column, tall, wide and ragged ones, columns that are
equal or lose their norm to the pivots (their norms are formed anew), and zero."""
import numpy as np
import pytest

from oracle import frank_oracle as fo

pytestmark = pytest.mark.gpu


def _matrix(rng, m, n, k, kind):
    q = lambda r: np.linalg.qr(rng.standard_normal((r, min(r, k))))[0]
    U, V = q(m), q(n)
    k = min(U.shape[1], V.shape[1])
    decay = {"flat": 0.02, "steep": 1.0, "equal": 0.1}[kind]
    A = (U[:, :k] * 10.0 ** (-decay * np.arange(k))) @ V[:, :k].T
    if kind == "equal" and n > 3:
        A[:, n // 2:] = A[:, : n - n // 2] * (1 + 1e-9)
    return A


@pytest.mark.parametrize("kind", ["flat", "steep", "equal"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 7, 1), (9, 1, 1), (15, 40, 15), (64, 64, 16), (130, 65, 17),
                                   (33, 200, 32), (512, 512, 40), (300, 512, 33), (512, 100, 48)])
def test_rank_and_factors(torch_gpu, kind, m, n, k):
    print(f"geqp3 {kind} {m} x {n} rank {k}", flush=True)
    torch = torch_gpu
    from frank_amd import dense
    A = _matrix(np.random.default_rng(m + n), m, n, k, kind)
    eps = 1e-8
    Q, R = dense.truncated_geqp3(torch.from_numpy(A).cuda(), eps)
    Qr, Rr = fo.truncated_geqp3(A, eps)
    Q, R = Q.cpu().numpy(), R.cpu().numpy()
    r, u = Q.shape[1], np.finfo(float).eps
    # the stopping rule compares column norms that carry an error of sqrt(u) (the downdating's limit), so
    # the rank may differ by one where a pivot is that close to the threshold
    assert abs(r - Qr.shape[1]) <= 1
    # a remainder of n columns, none above eps ||A||; r reflectors of rounding
    assert np.linalg.norm(A - Q @ R) <= (eps * np.sqrt(n) * 1.01 + 8 * r * u) * np.linalg.norm(A)
    assert np.abs(Q.T @ Q - np.eye(r)).max() <= 16 * max(r, 8) * u


def test_fixed_number_of_pivots_past_a_block(torch_gpu):
    """The ID's prefix of k steps: the oracle's pivots, for well separated norms."""
    torch = torch_gpu
    from frank_amd import dense
    rng = np.random.default_rng(5)
    A = np.linalg.qr(rng.standard_normal((90, 90)))[0] * (1.2 ** -rng.permutation(90))
    for k in (1, 15, 16, 17, 40):
        V, cols = dense.one_sided_id(torch.from_numpy(A).cuda(), k)
        Vr, colsr = fo.one_sided_id(A, k)
        assert cols == [int(c) for c in colsr]
        np.testing.assert_allclose(V.cpu().numpy(), Vr, rtol=0, atol=1e-12)
