"""Batched low-rank additions of operands of any norm: the truncation is relative to the
tile, so a tile of norm 1e-16 is recompressed as accurately as one of norm 1, whatever
its rows (each variant of the blocked QR, and the unblocked one above 256 rows)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the scale sits in S, in U or in V of both operands
SCALES = {"float32": [1e-10, 1e-12, 1e-14, 1e-16, 1e-19, 1e-26, 1e10, 1e20],
          "float64": [1e-16, 1e-100, 1e-149, 1e-157, 1e-200, 1e100, 1e160]}


def _pair(rng, m, n, k1, k2):
    q = lambda r, k: np.linalg.qr(rng.standard_normal((r, k)))[0]
    s = lambda k: np.diag(10.0 ** (-np.arange(k) / 4.0))
    return (q(m, k1), s(k1), q(n, k1).T), (q(m, k2), s(k2), q(n, k2).T)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("where", ["s", "u", "v"])
@pytest.mark.parametrize("m,n,k1,k2", [(64, 48, 8, 7), (64, 64, 20, 12), (128, 100, 32, 32), (128, 128, 60, 50), (200, 256, 9, 6),
                                       (256, 256, 30, 34), (256, 180, 64, 64), (300, 280, 16, 16), (512, 500, 60, 60)])
def test_accuracy_does_not_depend_on_the_norm(torch_gpu, fa, dtype, where, m, n, k1, k2):
    torch = torch_gpu
    u, dt, cap = np.finfo(dtype).eps, getattr(torch, dtype), 128
    eps = 1e-6 if dtype == "float32" else 1e-10
    rng = np.random.default_rng(m + k1)
    for scale in SCALES[dtype]:
        print(f"scale {dtype} {where} {m}x{n} {k1}+{k2} {scale:g}", flush=True)
        up = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt)
        ops = [_pair(rng, m, n, k1, k2) for _ in range(3)]
        As, Bs = [], []
        for A, B in ops:
            # (scaled after rounding to the type, so that the operands are the same at every scale)
            A, B = ([up(x) * (scale if "usv"[i] == where else 1.0) for i, x in enumerate(F)] for F in (A, B))
            slots = [torch.zeros(s, dtype=dt, device="cuda") for s in ((m, cap), (cap, cap), (cap, n))]
            for t, x in zip(slots, A):
                t[:x.shape[0], :x.shape[1]] = x
            As.append((*slots, k1))
            Bs.append(tuple(B))
        ins = [[x.double().cpu().numpy() for x in (a[0][:, :k1], a[1][:k1, :k1], a[2][:k1], *b)]
               for a, b in zip(As, Bs)]
        ranks = fa.lr_add_batched(As, Bs, eps=eps, lra="rounded_addition", cap=cap)
        for (U, S, V, _), (Ua, Sa, Va, Ub, Sb, Vb), r in zip(As, ins, ranks):
            # in the operands' own units: numpy's sums then neither under- nor overflow
            Ua, Sa, Va, Ub, Sb, Vb = (x / (scale if i % 3 == "usv".index(where) else 1.0)
                                      for i, x in enumerate((Ua, Sa, Va, Ub, Sb, Vb)))
            D = (Ua @ Sa) @ Va + (Ub @ Sb) @ Vb
            U, S, V = (x.double().cpu().numpy() for x in (U[:, :r], S[:r, :r], V[:r]))
            sv = np.linalg.svd(D, compute_uv=False)
            K = k1 + k2
            # the truncation (eps) and K reflectors and rotations of rounding, relative to the sum's own norm
            assert np.linalg.norm(D - (U @ (S / scale)) @ V) <= (1.01 * eps + 8 * K * u) * np.linalg.norm(sv)
            assert np.abs(np.diag(S) / scale - sv[:r]).max() <= 8 * K * u * sv[0]
            assert np.linalg.norm(sv[r:]) <= (eps + 8 * K * u) * np.linalg.norm(sv)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_columns_of_different_norms_and_zero_columns(torch_gpu, fa, dtype):
    """A panel whose columns differ by many orders of magnitude, with zero columns among them: the
    largest decide the result, and none of the others turns it into NaN."""
    torch = torch_gpu
    rng = np.random.default_rng(2)
    u, dt, k, cap = np.finfo(dtype).eps, getattr(torch, dtype), 12, 32
    up = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt)
    for m, n in ((60, 64), (120, 128), (250, 200), (400, 300)):
        A, B = _pair(rng, m, n, k, k)
        A, B = (A[0], np.diag(10.0 ** (-3.0 * np.arange(k))), A[2]), (B[0], np.diag([1.0, 0, 1e-30, 0, 1e-9] + [0.0] * 7), B[2])
        U, S, V = (torch.zeros(s, dtype=dt, device="cuda") for s in ((m, cap), (cap, cap), (cap, n)))
        U[:, :k], S[:k, :k], V[:k] = up(A[0]), up(A[1]), up(A[2])
        (r,) = fa.lr_add_batched([(U, S, V, k)], [tuple(up(x) for x in B)], eps=1e-5, lra="rounded_addition", cap=cap)
        D = (A[0] @ A[1]) @ A[2] + (B[0] @ B[1]) @ B[2]
        U, S, V = (x.double().cpu().numpy() for x in (U[:, :r], S[:r, :r], V[:r]))
        assert np.linalg.norm(D - (U @ S) @ V) <= (1.01e-5 + 16 * k * u) * np.linalg.norm(D)


@pytest.mark.parametrize("dtype,scale", [("float32", 2.0 ** -132), ("float64", 2.0 ** -1030)])
@pytest.mark.parametrize("k", [6, 12, 24, 40])
def test_denormal_tiles(torch_gpu, fa, dtype, scale, k):
    """A tile of denormal numbers is recompressed to their spacing."""
    torch = torch_gpu
    rng = np.random.default_rng(k)
    u, dt, cap, m, n = np.finfo(dtype).eps, getattr(torch, dtype), 128, 120, 100
    spacing = float(np.finfo(dtype).smallest_subnormal) / scale  # in the operands' own units
    up = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt)
    A, B = _pair(rng, m, n, k, k)
    A, B = (A[0], np.eye(k), A[2]), (B[0], np.eye(k), B[2])
    U, S, V = (torch.zeros(s, dtype=dt, device="cuda") for s in ((m, cap), (cap, cap), (cap, n)))
    U[:, :k], S[:k, :k], V[:k] = up(A[0]), up(scale * A[1]), up(A[2])
    (r,) = fa.lr_add_batched([(U, S, V, k)], [(up(B[0]), up(scale * B[1]), up(B[2]))], eps=1e-3,
                             lra="rounded_addition", cap=cap)
    D = A[0] @ A[2] + B[0] @ B[2]
    U, S, V = (x.double().cpu().numpy() for x in (U[:, :r], S[:r, :r], V[:r]))
    K = 2 * k
    # both panels' entries and the core's are rounded to the spacing (m K, K^2 of them, taken through K products)
    lim = (1.01e-3 + 8 * K * u) * np.linalg.norm(D) + spacing * K * np.sqrt(m * n)
    assert np.linalg.norm(D - (U @ (S / scale)) @ V) <= lim
