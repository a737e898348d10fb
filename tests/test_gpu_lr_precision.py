"""Rounding of the batched low-rank additions, beside the truncation: the mean error of
the sums over a batch, against a product in extended precision, at the level that the
arithmetic gives (and not only within the bounds of a single addition)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _operands(rng, m, n, k1, k2, decay):
    q = lambda r, k: np.linalg.qr(rng.standard_normal((r, k)))[0]
    s = lambda k: np.diag(10.0 ** (-decay * np.arange(k)))
    return (q(m, k1), s(k1), q(n, k1).T), (q(m, k2), s(k2), q(n, k2).T)


def _add(torch, fa, ops, dtype, eps, lra, cap=128):
    """(U, S, V) of every sum, and the sums of the operands as the GPU got them, in long double."""
    dt = getattr(torch, dtype)
    up = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt)
    wide = lambda x: x.double().cpu().numpy().astype(np.longdouble)
    As, Bs, Ds = [], [], []
    for A, B in ops:
        A, B = tuple(up(x) for x in A), tuple(up(x) for x in B)
        k = A[1].shape[0]
        slots = [torch.zeros(s, dtype=dt, device="cuda") for s in ((A[0].shape[0], cap), (cap, cap), (cap, A[2].shape[1]))]
        for t, x in zip(slots, A):
            t[:x.shape[0], :x.shape[1]] = x
        As.append((*slots, k))
        Bs.append(B)
        Ds.append(sum(wide(U) @ (wide(S) @ wide(V)) for U, S, V in (A, B)))
    ranks = fa.lr_add_batched(As, Bs, eps=eps, lra=lra, cap=cap)
    return [tuple(wide(x) for x in (a[0][:, :r], a[1][:r, :r], a[2][:r])) for a, r in zip(As, ranks)], Ds


def _norm(x):
    return float(np.linalg.norm(x.astype(np.float64)))


@pytest.mark.parametrize("m", [64, 128, 256])
def test_fp32_sums(torch_gpu, fa, m):
    """Singular values 10^(-i/2): the error is a few roundings (u = 2^-24) of the leading ones.  Mean over
    48 additions, a reflector at a time: 2.1e-7 of the norm at m = 64 (3.5 u), less above; with the
    reflectors in compact WY form 2.9, 2.6 and 2.5e-7 at m = 64, 128, 256 (4.9, 4.4, 4.3 u)."""
    rng = np.random.default_rng(m)
    out, Ds = _add(torch_gpu, fa, [_operands(rng, m, m, 16, 16, 0.5) for _ in range(48)], "float32", 1e-6,
                   "rounded_addition")
    tails = [np.linalg.svd(D.astype(np.float64), compute_uv=False)[U.shape[1]:] for (U, _, _), D in zip(out, Ds)]
    err = [(_norm(D - U @ (S @ V)) - np.linalg.norm(t)) / _norm(D) for (U, S, V), D, t in zip(out, Ds, tails)]
    print(f"fp32 sums m={m}: mean error {np.mean(err):.3e}", flush=True)
    assert np.mean(err) <= 4.0 * 2.0 ** -24


@pytest.mark.parametrize("m,limit", [(64, 1.95e-7), (512, 1.7e-7)])
def test_fp32_cores(torch_gpu, fa, m, limit):
    """The same mean with the squared column norms of the core's QR in FP64: 1.81e-7 at m = 64 and 1.59e-7
    at m = 512; with them in FP32 2.09 and 1.80e-7.  The limits lie between."""
    rng = np.random.default_rng(m)
    out, Ds = _add(torch_gpu, fa, [_operands(rng, m, m, 16, 16, 0.5) for _ in range(48)], "float32", 1e-6,
                   "rounded_addition")
    tails = [np.linalg.svd(D.astype(np.float64), compute_uv=False)[U.shape[1]:] for (U, _, _), D in zip(out, Ds)]
    err = [(_norm(D - U @ (S @ V)) - np.linalg.norm(t)) / _norm(D) for (U, S, V), D, t in zip(out, Ds, tails)]
    print(f"fp32 cores m={m}: mean error {np.mean(err):.3e}", flush=True)
    assert np.mean(err) <= limit


@pytest.mark.parametrize("eps", [1e-2, 1e-4, 1e-6, 1e-8])
@pytest.mark.parametrize("k", [6, 8, 16, 32, 64])
@pytest.mark.parametrize("decay", [0.1, 0.5])
def test_parts_of_a_truncated_sum(torch_gpu, fa, k, eps, decay):
    """The singular values and bases that a truncation keeps are those of the whole sum, to rounding, and
    not only the product U S V within eps."""
    rng = np.random.default_rng(k)
    u = np.finfo(np.float64).eps
    out, Ds = _add(torch_gpu, fa, [_operands(rng, 200, 150, k, k, decay) for _ in range(8)], "float64", eps,
                   "rounded_addition")
    for (U, S, V), D in zip(out, Ds):
        r, K = U.shape[1], 2 * k
        sv = np.linalg.svd(D.astype(np.float64), compute_uv=False)
        # each side (K reflectors, the core's rotations; numpy's own) to a few sqrt(K) u of the norm
        assert np.abs(np.diag(S).astype(np.float64) - sv[:r]).max() <= 8 * np.sqrt(K) * u * np.linalg.norm(sv)
        # vectors orthogonal to the rotation threshold tol = 8 max(K, 8) u; above 64 columns u_i = M v_i / sigma_i,
        # in which the larger ones stand with sigma_j (v_j^T v_i) / sigma_i
        tol = 8 * max(K, 8) * u
        assert np.abs((V @ V.T).astype(np.float64) - np.eye(r)).max() <= 2 * tol
        assert np.abs((U.T @ U).astype(np.float64) - np.eye(r)).max() <= 2 * tol * (sv[0] / sv[r - 1] if K > 64 else 1)


def test_left_vectors_of_large_cores(torch_gpu, fa):
    """Above 64 columns, sigma_r = 1e-8 of the norm: u_i = M v_i / sigma_i are as orthogonal as the v_i leave
    them.  Mean of 48 additions: 9.0e-6 with every column of the core rotated to 8 K u; 1.7e-5 with the
    columns below u ||M||_F left out, 2.8e-5 below 1e-11 ||M||_F; a few 1e-6 with the rotations to 2 K u."""
    rng = np.random.default_rng(7)
    out, _ = _add(torch_gpu, fa, [_operands(rng, 200, 150, 64, 64, 0.5) for _ in range(48)], "float64", 1e-8,
                  "rounded_addition")
    err = [np.abs((U.T @ U).astype(np.float64) - np.eye(U.shape[1])).max() for U, _, _ in out]
    print(f"left vectors: {np.mean(err):.3e}", flush=True)
    assert np.mean(err) <= 9e-6


@pytest.mark.parametrize("m,n,k1,k2", [(64, 60, 5, 3), (64, 64, 16, 9), (128, 100, 17, 16), (256, 200, 16, 16),
                                       (256, 256, 40, 24)])
def test_projection_leaves_nothing_of_the_basis(torch_gpu, fa, m, n, k1, k2):
    """The fast addition projects X's bases on C's.  Where X lies within 1e-7 of them and that remainder
    decides what is kept, the new basis is still orthonormal to rounding."""
    rng = np.random.default_rng(m + k1)
    u = np.finfo(np.float64).eps
    ops = []
    for _ in range(4):
        A = _operands(rng, m, n, k1, k1, 0.0)[0]
        k = min(k1, k2)
        near = lambda W: np.linalg.qr(W[:, rng.permutation(k1)[:k]] + 1e-7 * rng.standard_normal((W.shape[0], k)))[0]
        U, V = near(A[0]), near(A[2].T)
        # X = U V^T at 1e14: what it has outside C's bases, 1e-7 of each, weighs as much as C itself
        ops.append(((A[0], A[1], A[2]), (U, 1e14 * np.eye(k), V.T)))
    out, _ = _add(torch_gpu, fa, ops, "float64", 0.0, "fast_rounded_addition")
    for U, S, V in out:
        K = k1 + k2
        assert np.abs((U.T @ U).astype(np.float64) - np.eye(U.shape[1])).max() <= 16 * max(K, 8) * u
        assert np.abs((V @ V.T).astype(np.float64) - np.eye(U.shape[1])).max() <= 16 * max(K, 8) * u


@pytest.mark.parametrize("lra,eps", [("rounded_addition", 0.0), ("rounded_addition", 1e-10), ("fast_rounded_addition", 0.0)])
@pytest.mark.parametrize("k", [4, 8, 12, 16])
def test_right_vectors_of_small_cores(torch_gpu, fa, k, lra, eps):
    """Up to 32 columns in FP64 the right vectors come from reflectors and rotations alone: orthogonal to
    a few roundings a reflector, 2 K u, below the rotation threshold of 8 max(K, 8) u (the left ones')."""
    rng = np.random.default_rng(k)
    u = np.finfo(np.float64).eps
    out, Ds = _add(torch_gpu, fa, [_operands(rng, 128, 100, k, k, d) for d in (0.1, 0.3, 0.5) for _ in range(8)],
                   "float64", eps, lra)
    K = 2 * k
    for (U, S, V), D in zip(out, Ds):
        r = U.shape[1]
        assert np.abs((V @ V.T).astype(np.float64) - np.eye(r)).max() <= 2 * K * u
        assert np.abs((U.T @ U).astype(np.float64) - np.eye(r)).max() <= 16 * max(K, 8) * u
        tail = np.linalg.norm(np.linalg.svd(D.astype(np.float64), compute_uv=False)[r:])
        assert _norm(D - U @ (S @ V)) <= tail * (1 + 1e-6) + 8 * K * u * _norm(D)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("m,k", [(64, 12), (128, 8), (256, 16), (256, 24), (256, 40), (400, 16)])
def test_chain_of_fast_additions(torch_gpu, fa, dtype, m, k):
    """Twelve additions from the space that C spans, as a fixed-rank block LU makes them: each sum has the rank
    that is kept, so what is left is the rounding of twelve additions.  It does not grow with the loss of
    orthogonality that each passes on to the next (one projection in blocks of 16 left errors of 1e-3 in FP32
    and bases 1e-7 from orthonormal in FP64)."""
    torch = torch_gpu
    rng = np.random.default_rng(5)
    u, dt, cap, steps = np.finfo(dtype).eps, getattr(torch, dtype), 128, 12
    up = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt)
    wide = lambda x: x.double().cpu().numpy().astype(np.longdouble)
    q = lambda r, c: np.linalg.qr(rng.standard_normal((r, c)))[0]
    s = np.diag(10.0 ** (-0.2 * np.arange(k)))
    spaces = [(q(m, k), q(m, k)) for _ in range(4)]
    As, Ds, size = [], [], []
    for a, b in spaces:
        U, S, V = (torch.zeros(x, dtype=dt, device="cuda") for x in ((m, cap), (cap, cap), (cap, m)))
        U[:, :k], S[:k, :k], V[:k] = up(a), up(s), up(b.T)
        As.append((U, S, V, k))
        Ds.append(wide(U[:, :k]) @ (wide(S[:k, :k]) @ wide(V[:k])))
    for _ in range(steps):
        Bs = [(up(a @ q(k, k)), up(s), up((b @ q(k, k)).T)) for a, b in spaces]
        Ds = [D + wide(U) @ (wide(S) @ wide(V)) for D, (U, S, V) in zip(Ds, Bs)]
        assert list(fa.lr_add_batched(As, Bs, eps=0.0, lra="fast_rounded_addition", cap=cap)) == [k] * len(As)
    # rounding of each addition (some sqrt(K) u of the norms of its operands, K = 2 k), and the operands' own,
    # which lie in C's space to u only; above 64 columns FP64 forms u_i = M v_i / sigma_i, and U S V is off by
    # what the v_i are from orthogonal, the rotation threshold 2 K u
    lim = 4 * np.sqrt(2 * k) * u + (2 * 2 * k * u if dtype == "float64" and 2 * k > 64 else 0.0)
    for (U, S, V, _), D in zip(As, Ds):
        err = _norm(D - wide(U[:, :k]) @ (wide(S[:k, :k]) @ wide(V[:k]))) / _norm(D)
        print(f"chain {dtype} m={m} k={k}: {err:.2e}", flush=True)
        assert err <= steps * lim
        # FP64 up to 256 rows projects twice: the bases stay at the rotation threshold 8 max(K, 8) u, left and right
        if dtype == "float64" and m <= 256 and 2 * k <= 64:
            for W in (wide(U[:, :k]), wide(V[:k]).T):
                assert np.abs((W.T @ W).astype(np.float64) - np.eye(k)).max() <= 4 * 8 * max(2 * k, 8) * u
