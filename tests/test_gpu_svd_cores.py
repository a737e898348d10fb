"""Cores of the batched low-rank addition at the edges of the Jacobi SVD kernel's
variants (16, 32, 64 and 128 columns; FP64 above 64 keeps one array in LDS), with the
spectra that take its different ways: full numerical rank, a tail the pivoted QR drops,
numerically rank-deficient cores kept at a larger fixed rank, and zero."""
import numpy as np
import pytest

from oracle import frank_oracle as fo

pytestmark = pytest.mark.gpu


def _pair(rng, m, n, k1, k2, decay, common):
    """Two factored matrices (orthonormal bases, singular values 10^(-decay i)); with
    common bases the sum has numerical rank max(k1, k2)."""
    q = lambda rows, k: np.linalg.qr(rng.standard_normal((rows, k)))[0]
    s = lambda k: np.diag(10.0 ** (-decay * np.arange(k)))
    if common:
        k = max(k1, k2)
        U, V = q(m, k), q(n, k)
        U2, V2 = U, V
    else:
        U, V, U2, V2 = q(m, k1), q(n, k1), q(m, k2), q(n, k2)
    return (U[:, :k1], s(k1), V[:, :k1].T), (U2[:, :k2], s(k2), V2[:, :k2].T)


def _add(torch, fa, pairs, cap, eps, dtype):
    As, Bs = [], []
    for (U, S, V), B in pairs:
        m, k = U.shape
        slot = lambda r, c, x: torch.nn.functional.pad(torch.from_numpy(np.ascontiguousarray(x)),
                                                       (0, c - x.shape[1], 0, r - x.shape[0])).to("cuda", dtype)
        As.append((slot(m, cap, U), slot(cap, cap, S), slot(cap, V.shape[1], V), k))
        Bs.append(tuple(torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dtype) for x in B))
    ranks = fa.lr_add_batched(As, Bs, eps=eps, lra="rounded_addition", cap=cap)
    return [tuple(x.double().cpu().numpy() for x in (a[0][:, :r], a[1][:r, :r], a[2][:r])) for a, r in zip(As, ranks)]


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("k1,k2", [(1, 1), (2, 1), (8, 8), (9, 8), (16, 15), (16, 16), (17, 16), (31, 32), (32, 32),
                                   (33, 32), (64, 63), (64, 64)])
@pytest.mark.parametrize("decay", [0.05, 0.2])
def test_core_sizes(torch_gpu, fa, dtype, k1, k2, decay):
    print(f"cores {dtype} {k1}+{k2} decay {decay}", flush=True)
    torch = torch_gpu
    rng = np.random.default_rng(100 * k1 + k2)
    u = np.finfo(dtype).eps
    eps = 1e-9 if dtype == "float64" else 1e-5
    pairs = [_pair(rng, 200, 150, k1, k2, decay, c) for c in (False, True)]
    for (A, B), (U, S, V) in zip(pairs, _add(torch, fa, pairs, 128, eps, getattr(torch, dtype))):
        D = (A[0] @ A[1]) @ A[2] + (B[0] @ B[1]) @ B[2]
        sv = np.linalg.svd(D, compute_uv=False)
        K = k1 + k2
        r = U.shape[1]
        # the truncation rule keeps sqrt(K - r) sigma_r <= eps ||sigma||; the tail is at most that, and
        # rounding (QR of both panels, the core's products and rotations) some K u on top
        err = np.linalg.norm(D - (U @ S) @ V)
        assert err <= (1.01 * eps + 8 * K * u) * np.linalg.norm(sv)
        assert np.linalg.norm(sv[r:]) <= (eps + 8 * K * u) * np.linalg.norm(sv)
        assert np.abs(np.diag(S) - sv[:r]).max() <= 8 * K * u * sv[0]
        # right vectors: pairwise orthogonal to the rotation threshold 8 max(K, 8) u
        assert np.abs(V @ V.T - np.eye(r)).max() <= 16 * max(K, 8) * u
        # above 64 columns FP64 forms u_i = M v_i / sigma_i: the same times sigma_1 / sigma_r
        lim = 16 * max(K, 8) * u * (sv[0] / sv[r - 1] if dtype == "float64" and K > 64 else 1.0)
        assert np.abs(U.T @ U - np.eye(r)).max() <= lim
        # the oracle's rank, where the decision is not within rounding of the threshold
        want = fo.find_svd_truncation_rank(sv[:min(K, len(sv))], eps)
        if dtype == "float64":
            assert r == want


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("k1,k2", [(2, 2), (8, 8), (12, 20), (24, 24), (30, 34)])
def test_fixed_rank_above_the_numerical_rank(torch_gpu, fa, dtype, k1, k2):
    """eps = 0 keeps rank k1 although the sum's numerical rank is far smaller: the missing
    vectors of both bases are completed to orthonormal sets.  Also the zero core."""
    print(f"fixed rank {dtype} {k1}+{k2}", flush=True)
    torch = torch_gpu
    rng = np.random.default_rng(k1)
    u = np.finfo(dtype).eps
    A, B = _pair(rng, 160, 130, k1, k2, 4.0, True)  # numerical rank at most 5
    Z = (A[0], 0 * A[1], A[2]), (B[0], 0 * B[1], B[2])
    for (P, Q), (U, S, V) in zip([(A, B), Z], _add(torch, fa, [(A, B), Z], 64, 0.0, getattr(torch, dtype))):
        D = (P[0] @ P[1]) @ P[2] + (Q[0] @ Q[1]) @ Q[2]
        K = k1 + k2
        assert U.shape[1] == k1
        assert np.linalg.norm(D - (U @ S) @ V) <= 8 * K * u * np.linalg.norm(D)
        assert np.abs(V @ V.T - np.eye(k1)).max() <= 16 * max(K, 8) * u
        assert np.abs(U.T @ U - np.eye(k1)).max() <= 16 * max(K, 8) * u


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("k", [4, 8, 16, 32, 64])
@pytest.mark.parametrize("kind", ["overflow", "inf", "nan"])
def test_core_that_is_not_finite(torch_gpu, fa, dtype, k, kind):
    """A core that overflows (bases of a large norm), or operands with an infinity or a NaN, give a tile
    that is not finite either, and not zeros; the other additions of the batch are not touched."""
    print(f"not finite {dtype} K={2 * k} {kind}", flush=True)
    torch = torch_gpu
    rng = np.random.default_rng(k)
    u = np.finfo(dtype).eps
    A, B = _pair(rng, 150, 140, k, k, 0.1, False)
    bad = [x.copy() for x in A]
    if kind == "overflow":
        big = 1e30 if dtype == "float32" else 1e200
        bad[1] = big * bad[1]
        bad[2] = big * bad[2]
    else:
        bad[0][3, 1] = np.inf if kind == "inf" else np.nan
    for eps in (1e-5, 0.0):
        X, Y, Z = _add(torch, fa, [(A, B), (tuple(bad), B), (A, B)], 128, eps, getattr(torch, dtype))
        assert not np.isfinite((Y[0] @ Y[1]) @ Y[2]).any()
        for x, z in zip(X, Z):
            assert np.array_equal(x, z)
        D = (A[0] @ A[1]) @ A[2] + (B[0] @ B[1]) @ B[2]
        sv = np.linalg.svd(D, compute_uv=False)
        tail = np.linalg.norm(sv[X[0].shape[1]:])
        assert np.linalg.norm(D - (X[0] @ X[1]) @ X[2]) <= tail * (1 + 1e-5) + 16 * k * u * np.linalg.norm(sv)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_sweep_counters_with_zero_cores(torch_gpu, fa, dtype):
    """Zero cores and cores of one column count as problems of no sweeps."""
    torch = torch_gpu
    rng = np.random.default_rng(1)
    dt = getattr(torch, dtype)
    ctx = fa.Context()
    for k, scale, most in ((8, 0.0, 0), (32, 0.0, 0), (8, 1.0, 60)):
        pairs = [_pair(rng, 90, 80, k, k, 0.1, False) for _ in range(5)]
        As, Bs = [], []
        for (U, S, V), B in pairs:
            slots = [torch.zeros(s, dtype=dt, device="cuda") for s in ((90, 64), (64, 64), (64, 80))]
            for t, x in zip(slots, (U, scale * S, V)):
                t[:x.shape[0], :x.shape[1]] = torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt)
            As.append((*slots, k))
            Bs.append(tuple(torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt) for x in (B[0], scale * B[1], B[2])))
        ctx.counters(reset=True)
        fa.lr_add_batched(As, Bs, eps=0.0, lra="rounded_addition", cap=64, ctx=ctx)
        c = ctx.counters()
        assert c["svd_problems"] == 5
        assert (0 if scale == 0.0 else 5) <= c["svd_sweeps"] <= 5 * most
        assert 0 <= c["svd_max_sweeps"] <= most


@pytest.mark.parametrize("k", [4, 8, 16, 32])
@pytest.mark.parametrize("low", [1e-30, 1e-85, 1e-120])
def test_blocks_of_very_different_norm(torch_gpu, fa, k, low):
    """A tile and `low` times another on other rows and columns, at an eps below that ratio: nothing mixes
    them, so the small one is kept, and as accurately as the large one."""
    print(f"blocks K={2 * k} {low:g}", flush=True)
    rng = np.random.default_rng(k)
    u = np.finfo(float).eps
    parts, tiles = [], []
    for rows, cols, scale in ((slice(0, 80), slice(0, 70), 1.0), (slice(80, 150), slice(70, 130), low)):
        # (bases that are not orthonormal: the cores then need rotations)
        X, Y = rng.standard_normal((rows.stop - rows.start, k)), rng.standard_normal((k, cols.stop - cols.start))
        U, V = np.zeros((150, k)), np.zeros((k, 130))
        U[rows], V[:, cols] = X, Y
        parts.append((U, scale * np.eye(k), V))
        tiles.append((rows, cols, scale, X @ Y))
    ((U, S, V),) = _add(torch_gpu, fa, [tuple(parts)], 128, 1e-3 * low, torch_gpu.float64)
    for rows, cols, scale, D in tiles:
        assert np.linalg.norm((U[rows] @ (S / scale)) @ V[:, cols] - D) <= 8 * 2 * k * u * np.linalg.norm(D)
