"""QR and basis update of the batched low-rank addition at the edges of the blocked FP64
kernels' tiles (16 rows, 16 columns), of their variants (64, 128, 256 rows; 16, 32, 64, 128
columns; past them, and in FP32, the unblocked kernels), for tiles smaller than the columns
added, both layouts of the bases, and both additions (rounded; fast, which projects first)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [  # (m, n) of the items of one batch, ranks k1, k2
    ([(1, 1), (1, 5), (16, 3)], 1, 1),
    ([(15, 17), (16, 16), (31, 33)], 7, 8),
    ([(17, 40), (64, 63), (48, 20)], 9, 7),
    ([(64, 64), (61, 18)], 16, 16),
    ([(65, 66), (128, 20), (127, 33)], 17, 15),
    ([(129, 128), (256, 40), (255, 100)], 8, 8),
    ([(256, 200), (130, 256)], 17, 16),
    ([(257, 300), (512, 64), (511, 60)], 5, 6),
    ([(512, 512), (300, 498)], 16, 15),
    ([(512, 400), (512, 100)], 24, 33),
    ([(64, 64), (50, 49)], 40, 24),  # more columns than rows
    ([(64, 64), (48, 64)], 48, 48),
    ([(128, 128), (100, 70)], 64, 64),
    ([(256, 256), (140, 250)], 60, 60),
    ([(512, 512), (400, 300)], 64, 64),
]


def _lowrank(rng, m, n, k):
    q = lambda rows: np.linalg.qr(rng.standard_normal((rows, k)))[0]
    return q(m), np.diag(2.0 ** (-np.arange(k) / 4.0)), q(n).T


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("lra", ["rounded_addition", "fast_rounded_addition"])
@pytest.mark.parametrize("case", range(len(SIZES)))
def test_tile_edges(torch_gpu, fa, dtype, lra, case):
    shapes, k1, k2 = SIZES[case]
    print(f"{dtype} {lra} {shapes} {k1}+{k2}", flush=True)
    torch = torch_gpu
    rng = np.random.default_rng(case)
    u = np.finfo(dtype).eps
    # the fast addition is the one of a fixed rank (eps = 0): the rank kept is k1
    eps = 0.0 if lra.startswith("fast") else (1e-9 if dtype == "float64" else 1e-5)
    dt = getattr(torch, dtype)
    cap = 128
    As, Bs, Ds = [], [], []
    for i, (m, n) in enumerate(shapes):
        ka, kb = min(k1, m, n), min(k2, m, n)
        A, B = _lowrank(rng, m, n, ka), _lowrank(rng, m, n, kb)
        Ds.append((A[0] @ A[1]) @ A[2] + (B[0] @ B[1]) @ B[2])

        def slot(r, c, x):
            return torch.nn.functional.pad(torch.from_numpy(np.ascontiguousarray(x)),
                                           (0, c - x.shape[1], 0, r - x.shape[0])).to("cuda", dt)
        As.append((slot(m, cap, A[0]), slot(cap, cap, A[1]), slot(cap, n, A[2]), ka))
        Bs.append(tuple(torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt) for x in B))
    ranks = fa.lr_add_batched(As, Bs, eps=eps, lra=lra, cap=cap)
    for (U, S, V, k), r, D, B in zip(As, ranks, Ds, Bs):
        U, S, V = (x.double().cpu().numpy() for x in (U[:, :r], S[:r, :r], V[:r]))
        K = k + B[0].shape[1]
        sv = np.linalg.svd(D, compute_uv=False)
        if eps == 0.0:
            assert r == k
        # the best error of the rank kept, plus rounding: K reflectors a side and the core's rotations,
        # each a few u of the norm (the truncated part's second-order share is inside eps)
        tail = np.linalg.norm(sv[r:])
        assert np.linalg.norm(D - (U @ S) @ V) <= (1.01 * eps + 8 * K * u) * np.linalg.norm(sv) + tail * (1 + 1e-6)
        assert tail <= (eps + 8 * K * u) * np.linalg.norm(sv) or eps == 0.0
        # products of K reflectors times vectors orthogonal to the rotation threshold 8 max(K, 8) u
        assert np.abs(V @ V.T - np.eye(r)).max() <= 16 * max(K, 8) * u
        # above 64 columns FP64 forms u_i = M v_i / sigma_i: the same times sigma_1 / sigma_r
        lim = 16 * max(K, 8) * u * (sv[0] / sv[r - 1] if dtype == "float64" and K > 64 else 1.0)
        assert np.abs(U.T @ U - np.eye(r)).max() <= lim


@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_both_routes_of_a_tall_narrow_batch(torch_gpu, fa, dtype):
    """129 to 256 rows and at most 32 columns: up to 128 additions in FP64 take the blocked kernels, more
    (and FP32 always) the unblocked ones; the same additions give the same sums either way."""
    torch = torch_gpu
    rng = np.random.default_rng(3)
    u, dt, k, cap = np.finfo(dtype).eps, getattr(torch, dtype), 9, 32
    ops = [(_lowrank(rng, 200, 150, k), _lowrank(rng, 200, 150, k)) for _ in range(129)]

    def run(items):
        up = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt)
        As = []
        for A, _ in items:
            U, S, V = (torch.zeros(s, dtype=dt, device="cuda") for s in ((200, cap), (cap, cap), (cap, 150)))
            U[:, :k], S[:k, :k], V[:k] = up(A[0]), up(A[1]), up(A[2])
            As.append((U, S, V, k))
        ranks = fa.lr_add_batched(As, [tuple(up(x) for x in B) for _, B in items], eps=0.0, lra="rounded_addition",
                                  cap=cap)
        assert list(ranks) == [k] * len(items)
        return [((a[0][:, :k] @ a[1][:k, :k]) @ a[2][:k]).double().cpu().numpy() for a in As]
    for (A, B), X, Z in zip(ops, run(ops[:128]), run(ops)):
        D = (A[0] @ A[1]) @ A[2] + (B[0] @ B[1]) @ B[2]
        sv = np.linalg.svd(D, compute_uv=False)
        # each is the best rank-k approximation to 8 K u of the norm (K = 2 k reflectors and rotations);
        # they may differ by more where sigma_k and sigma_k+1 are close, so both go against D
        for Y in (X, Z):
            assert np.linalg.norm(D - Y) <= np.linalg.norm(sv[k:]) + 8 * 2 * k * u * np.linalg.norm(sv)
