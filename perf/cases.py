"""The performance cases: what a program that uses this framework has it do.

Every case goes through the public Python surface of ``frank_amd`` (or, for the
large batch of additions, through the C entry point ``frk_slr_add_batched`` with
pointer arrays built once, as ``bench.py`` calls it).  A case is a dict of plain
values with a ``kind``:

  lu        restore a compressed matrix into its working copy, BLR-LU in place
            (the factorization overwrites its input), one block solve
  refine    the same, with the solve refined in FP64 against the exact kernel
            matrix; FP64 tiles at eps 1e-10 or FP32 tiles at eps 1e-6
  kept      solves with factors kept from before: A x = b and A^T y = b
  qr        restore, tiled Householder BLR-QR in place, Q formed by applying its
            reflectors to the identity in BLR form, Q and R fetched
  add       batched low-rank additions (rounded, or fast at fixed rank)
  adjoint   differentiable solve of a gaussian kernel system, forward + backward
            (builds, factors and solves; the backward reuses the factors)
  build     compression of a kernel matrix to BLR form, one product with it
  tilelu    batched dense tile LU without pivoting

Low-rank factors are unique only up to rotations of close singular vectors, so an
addition's result is returned as the sums it represents, expanded.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import frank_amd as fa
from frank_amd import _lib as L
from frank_amd.autograd import blr_solve
from frank_amd.inputs import morton_sort, mt19937_uniform, uniform_points


def listed():
    return [
        # the reference's own test sizes: a small matrix where launches and waits are everything
        dict(name="lu_small", kind="lu", n=512, nb=8, eps=1e-8, rank=0, admis=0, nrhs=1),
        # BLR-LU at fixed rank with the fast addition (16 x 16 tiles of 256), one right-hand side
        dict(name="lu_fixed_rank", kind="lu", n=4096, nb=16, eps=0.0, rank=16, admis=0, nrhs=1),
        # an uneven grid (13 tiles of 320) with dense neighbours of the diagonal
        # (strong admissibility): every Dense / LowRank product of the Schur updates
        dict(name="lu_dense_band", kind="lu", n=4160, nb=13, eps=1e-6, rank=0, admis=1, nrhs=3),
        # the benchmark's headline: FP32 tiles and recompression, FP64 diagonal, FP64 refinement
        dict(name="refine_mixed_32768", kind="refine", n=32768, nb=64, precision="f32", nrhs=8),
        # the same system on the plain FP64 path
        dict(name="refine_f64_32768", kind="refine", n=32768, nb=64, precision="f64", nrhs=8),
        # a program that factors once and solves with many right-hand sides, both directions
        dict(name="kept_solves_16384", kind="kept", n=16384, nb=32, eps=1e-8, nrhs=8),
        # tiled BLR-QR of a 2-D problem with ranks capped at 64 (tiles of 256)
        dict(name="qr_2d_1536", kind="qr", n=1536, nb=6, eps=1e-8),
        # recompression of a large uneven batch in FP32 (the batched-addition benchmark's pairs)
        dict(name="add_f32_batch", kind="add", batch=2048, m=0, n=0, k1=0, k2=0, dtype="f32", eps=1e-6, lra="rounded"),
        # a few FP64 additions: the latency of one call
        dict(name="add_f64_few", kind="add", batch=8, m=300, n=200, k1=12, k2=9, dtype="f64", eps=1e-10,
             lra="rounded"),
        # one differentiable gaussian-kernel system with 64-point tiles and ranks near the tile size
        dict(name="adjoint_2048", kind="adjoint", n=2048, nb=32, ell=0.15),
        # construction and one product with the compressed matrix (time to the first matvec)
        dict(name="build_matvec_16384", kind="build", n=16384, nb=32, dim=1, eps=1e-8, nrhs=4),
        # batched dense LU of mid-sized diagonal tiles
        dict(name="tilelu_32x256", kind="tilelu", batch=32, n=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind, then sizes spread over its range (odd ones included)."""
    kind = rng.choice(["lu", "lu", "refine", "kept", "qr", "add", "add", "adjoint", "build", "tilelu"])
    if kind == "lu":
        b = 64 * _log_int(rng, 1, 8)
        nb = _log_int(rng, 2, 20)
        n = b * nb
        if rng.random() < 0.3:
            rank = rng.choice([8, 12, 16])
            return dict(kind="lu", n=n, nb=nb, eps=0.0, rank=rank, admis=0, nrhs=rng.choice([1, 2, 5, 8]))
        return dict(kind="lu", n=n, nb=nb, eps=rng.choice([1e-6, 1e-8, 1e-10]), rank=0, admis=rng.choice([0, 0, 1, 2]),
                    nrhs=rng.choice([1, 2, 5, 8, 16]))
    if kind == "refine":
        nb = _log_int(rng, 8, 64)
        return dict(kind="refine", n=64 * rng.randrange(4, 9) * nb, nb=nb, precision=rng.choice(["f32", "f64"]),
                    nrhs=rng.choice([1, 3, 8, 16]))
    if kind == "kept":
        nb = _log_int(rng, 4, 32)
        return dict(kind="kept", n=64 * rng.randrange(2, 9) * nb, nb=nb, eps=rng.choice([1e-6, 1e-8, 1e-10]),
                    nrhs=rng.choice([1, 2, 4, 7, 8, 16]))
    if kind == "qr":
        nb = rng.randrange(2, 7)
        return dict(kind="qr", n=nb * _log_int(rng, 80, 256), nb=nb, eps=rng.choice([1e-6, 1e-8]))
    if kind == "add":
        if rng.random() < 0.4:
            return dict(kind="add", batch=_log_int(rng, 32, 2048), m=0, n=0, k1=0, k2=0, dtype="f32", eps=1e-6,
                        lra="rounded")
        fixed = rng.random() < 0.3
        return dict(kind="add", batch=_log_int(rng, 1, 256), m=_log_int(rng, 96, 512), n=_log_int(rng, 96, 512),
                    k1=rng.randrange(2, 17 if fixed else 33), k2=rng.randrange(2, 33), dtype="f64",
                    eps=0.0 if fixed else rng.choice([1e-6, 1e-8, 1e-10]), lra="fast" if fixed else "rounded")
    if kind == "adjoint":
        nb = _log_int(rng, 4, 32)
        return dict(kind="adjoint", n=64 * nb, nb=nb, ell=round(rng.uniform(0.05, 0.3), 3))
    if kind == "build":
        b = rng.choice([128, 256, 400, 512])
        nb = _log_int(rng, 3, 32)
        return dict(kind="build", n=b * nb - rng.randrange(0, nb), nb=nb, dim=1, eps=rng.choice([1e-6, 1e-8, 1e-10]),
                    nrhs=rng.choice([1, 2, 4, 8]))
    return dict(kind="tilelu", batch=_log_int(rng, 2, 64), n=_log_int(rng, 17, 512))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _points(case, seed):
    n = case["n"]
    if case["kind"] == "qr":
        p, _ = morton_sort(uniform_points(n, 2, seed=seed), 6)
    elif case["kind"] == "adjoint":
        p, _ = morton_sort(uniform_points(n, 3, seed=seed), 4)
    else:
        p = np.sort(mt19937_uniform(seed, n))[None, :]
    return [np.ascontiguousarray(q) for q in p]


def _rhs(n, nrhs, seed):
    return torch.from_numpy(np.random.default_rng(seed + 1).standard_normal((n, nrhs))).cuda()


_SHIFT = {"lu": 1e-2, "refine": 1e-2, "kept": 1e-2, "qr": 0.0, "build": 1e-2, "tilelu": 1e-2}
_SIZES, _RANKS = [64, 128, 256, 512], [8, 16, 32, 64]


def _add_groups(case):
    """Additions grouped by tile size: [(m, n, [(k1, k2), ...])].  m = 0: the uneven
    batch (m, n from {64..512}, ranks from {8..64}, drawn uniformly; the case alone
    fixes them, so that every seed's outputs have the same shapes)."""
    if case["m"]:
        return [(case["m"], case["n"], [(case["k1"], case["k2"])] * case["batch"])]
    g = np.random.default_rng(case["batch"])
    by = {}
    for _ in range(case["batch"]):
        mn = (int(g.choice(_SIZES)), int(g.choice(_SIZES)))
        by.setdefault(mn, []).append((int(g.choice(_RANKS)), int(g.choice(_RANKS))))
    return [(m, n, by[(m, n)]) for m, n in sorted(by)]


def _add_inputs(case, seed):
    """Per size group, on the GPU: the A slots (U m x cap, S cap x cap, V cap x n, unused
    columns zero) in one slab each, the B factors in one slab per rank k2.  Factors are
    N(0, 1) (orthonormal bases for the fixed-rank addition, as its operands always have),
    singular values 10^(-i/4)."""
    dt = torch.float32 if case["dtype"] == "f32" else torch.float64
    cap = 64 if case["m"] else 128
    out = []
    for gi, (m, n, ks) in enumerate(_add_groups(case)):
        gen = torch.Generator(device="cuda").manual_seed(seed * 1000 + gi)

        def basis(c, rows, width):
            x = torch.randn((c, rows, width), generator=gen, device="cuda", dtype=dt)
            return torch.linalg.qr(x).Q.contiguous() if case["eps"] == 0.0 else x

        def factors(ranks, width):
            kept = torch.tensor(ranks, device="cuda")[:, None] > torch.arange(width, device="cuda")[None, :]
            U = basis(len(ranks), m, width) * kept[:, None, :]
            V = basis(len(ranks), n, width).transpose(1, 2) * kept[:, :, None]
            s = 10.0 ** (-torch.arange(width, device="cuda", dtype=torch.float64) / 4.0)
            return U, torch.diag_embed((s * kept).to(dt)), V.contiguous()

        ks = sorted(ks, key=lambda k: k[1])
        B = []
        for k2 in sorted({k[1] for k in ks}):
            B.append(factors([k2] * sum(k[1] == k2 for k in ks), k2))
        out.append(dict(m=m, n=n, ks=ks, A=factors([k[0] for k in ks], cap), B=B))
    return out, cap


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def _matrix(case, seed, eps=None, rank=0, admis=0, ctx=None):
    return fa.BlrMatrix.from_kernel(_points(case, seed), case["nb"], eps=case["eps"] if eps is None else eps,
                                    rank=rank, admis=float(admis), shift=_SHIFT[case["kind"]],
                                    kcap=rank if rank else 64, ctx=ctx)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "lu":
        A = _matrix(case, seed, rank=case["rank"], admis=case["admis"])
        A.set_lra("fast_rounded_addition" if case["rank"] else "rounded_addition")
        return dict(kind=kind, A=A, F=A.clone(), b=_rhs(case["n"], case["nrhs"], seed))
    if kind == "refine":
        f32 = case["precision"] == "f32"
        A = _matrix(case, seed, eps=1e-6 if f32 else 1e-10)
        if f32:
            A = A.convert("f32")
        A.set_lra("rounded_addition")
        b = _rhs(case["n"], case["nrhs"], seed)
        return dict(kind=kind, A=A, F=A.clone(), b=b)
    if kind == "kept":
        F = _matrix(case, seed)
        F.set_lra("rounded_addition")
        F.getrf()
        return dict(kind=kind, F=F, b=_rhs(case["n"], case["nrhs"], seed))
    if kind == "qr":
        ctx = fa.Context()
        ctx.set_rank_cap(True)
        A = _matrix(case, seed, ctx=ctx)
        A.set_lra("rounded_addition")
        Q = fa.BlrMatrix.from_kernel(_points(case, seed), case["nb"], eps=case["eps"], kcap=64, kernel="identity",
                                     ctx=ctx)
        Q.set_lra("rounded_addition")
        return dict(kind=kind, A=A, F=A.clone(), I=Q, Q=Q.clone())
    if kind == "add":
        groups, cap = _add_inputs(case, seed)
        st = dict(kind=kind, cap=cap, eps=case["eps"], groups=groups)
        st["work"] = [tuple(x.clone() for x in g["A"]) for g in groups]
        st["k1"] = [k1 for g in groups for (k1, _) in g["ks"]]
        if case["dtype"] == "f64":
            st["lra"] = "fast_rounded_addition" if case["lra"] == "fast" else "rounded_addition"
            return st
        # the C entry's host arrays, laid out once as a program that owns its slots does
        import ctypes as C
        batch = len(st["k1"])

        def ptrs(slabs):
            return (C.c_void_p * batch)(*[x.data_ptr() + t * x.stride(0) * x.element_size()
                                          for x in slabs for t in range(x.shape[0])])

        st["ptrs"] = [ptrs([w[q] for w in st["work"]]) for q in range(3)]
        st["ptrs"] += [ptrs([f[q] for g in groups for f in g["B"]]) for q in range(3)]
        reps = [len(g["ks"]) for g in groups]
        st["m"] = np.repeat([g["m"] for g in groups], reps).astype(np.int32)
        st["n"] = np.repeat([g["n"] for g in groups], reps).astype(np.int32)
        st["kb"] = np.array([k2 for g in groups for (_, k2) in g["ks"]], dtype=np.int32)
        torch.cuda.synchronize()
        return st
    if kind == "adjoint":
        return dict(kind=kind, pts=np.vstack(_points(case, seed)), b=_rhs(case["n"], 1, seed), nb=case["nb"],
                    ell=case["ell"])
    if kind == "build":
        return dict(kind=kind, case=dict(case), seed=seed, pts=_points(case, seed), x=_rhs(case["n"], case["nrhs"], seed))
    a = _tiles(case, seed)
    return dict(kind=kind, a=a, w=torch.empty_like(a))


def _tiles(case, seed):
    """Diagonal tiles of the 1-D kernel matrix (what the tile LU factors in BLR-LU)."""
    x = torch.from_numpy(np.sort(mt19937_uniform(seed, case["n"] * case["batch"]))).cuda().reshape(case["batch"], -1)
    a = 1.0 / ((x[:, :, None] - x[:, None, :]).abs() + 1e-3)
    return a + 1e-2 * torch.eye(case["n"], dtype=a.dtype, device=a.device)


def run(state):
    kind = state["kind"]
    if kind == "lu":
        F = state["F"].copy_from(state["A"]).getrf()
        return F.solve(state["b"].clone())
    if kind == "refine":
        F = state["F"].copy_from(state["A"]).getrf()
        x = torch.empty_like(state["b"])
        F.refine(state["b"], x, tol=1e-10, max_iter=60)
        return x
    if kind == "kept":
        F = state["F"]
        return [F.solve(state["b"].clone()), F.solve(state["b"].clone(), trans=True)]
    if kind == "qr":
        F = state["F"].copy_from(state["A"])
        Q = F.apply_q(F.qr(), state["Q"].copy_from(state["I"]))
        return dict(r=np.triu(F.dense()), q=Q.dense())
    if kind == "add":
        for g, w in zip(state["groups"], state["work"]):
            for dst, src in zip(w, g["A"]):
                dst.copy_(src)
        if "ptrs" not in state:
            As = [(w[0][t], w[1][t], w[2][t], k1) for g, w in zip(state["groups"], state["work"])
                  for t, (k1, _) in enumerate(g["ks"])]
            Bs = [tuple(x[t] for x in f) for g in state["groups"] for f in g["B"] for t in range(f[0].shape[0])]
            ranks = fa.lr_add_batched(As, Bs, eps=state["eps"], lra=state["lra"], cap=state["cap"])
        else:
            ranks = np.array(state["k1"], dtype=np.int32)
            torch.cuda.current_stream().synchronize()
            Ua, Sa, Va, Ub, Sb, Vb = state["ptrs"]
            L.check(fa.lib().frk_slr_add_batched(fa.default_context().h, L.LRA_ROUNDED, len(ranks),
                                                 state["m"].ctypes.data, state["n"].ctypes.data, state["eps"],
                                                 state["cap"], Ua, Sa, Va, ranks.ctypes.data, Ub, Sb, Vb,
                                                 state["kb"].ctypes.data))
        # the sums: each addition's kept columns expanded
        out, o = [], 0
        rk = torch.as_tensor(np.asarray(ranks, dtype=np.int64)).cuda()
        for U, S, V in state["work"]:
            r = rk[o:o + U.shape[0], None]
            o += U.shape[0]
            on = torch.arange(S.shape[1], device=S.device)[None, :] < r
            out.append((U * on[:, None, :]) @ (torch.where(on[:, None, :] & on[:, :, None], S, 0) @ (V * on[:, :, None])))
        return out
    if kind == "adjoint":
        b = state["b"].clone().requires_grad_(True)
        ell = torch.tensor(state["ell"], dtype=torch.float64, requires_grad=True)
        u = blr_solve(b, ell, state["pts"], state["nb"], eps=1e-12, shift=1e-4, kcap=64)
        (0.5 * (u * u).sum()).backward()
        return dict(u=u.detach(), db=b.grad, dell=ell.grad)
    if kind == "build":
        c = state["case"]
        A = fa.BlrMatrix.from_kernel(state["pts"], c["nb"], eps=c["eps"], shift=_SHIFT["build"], kcap=64)
        return A.matvec(state["x"], torch.zeros_like(state["x"]))
    w = state["w"].copy_(state["a"])
    fa.getrf_nopiv_batched(list(w))
    return w


# ---------------------------------------------------------------------------
# what a pass cannot do without, and the answers in 64 bits
# ---------------------------------------------------------------------------
def _mean_rank(case):
    """Typical rank of an off-diagonal tile of these kernels at the case's accuracy."""
    if case.get("rank"):
        return case["rank"]
    eps = case.get("eps") or (1e-6 if case.get("precision") == "f32" else 1e-10)
    return 3.0 - 0.3 * math.log10(eps) if case["kind"] != "qr" else 40.0


def work(case):
    kind = case["kind"]
    n = case["n"]
    if kind == "add":
        # both bases and cores in, the sum of the kept rank out; QR of both panels, small
        # SVD, both bases rebuilt
        by = fl = 0.0
        s = 4.0 if case["dtype"] == "f32" else 8.0
        for m, nn, ks in _add_groups(case):
            for k1, k2 in ks:
                K = k1 + k2
                by += s * ((m + nn) * (K + k1) + k1 * k1 + k2 * k2 + k1)
                fl += 4.0 * (m + nn) * K * K + 24.0 * K ** 3 + 2.0 * (m + nn) * K * k1
        return dict(bytes=by, flops=fl)
    if kind == "tilelu":
        return dict(bytes=16.0 * case["batch"] * n * n, flops=case["batch"] * 2.0 / 3.0 * n ** 3)
    nb = case["nb"]
    b = n / nb
    if kind == "adjoint":
        # tiles of nearly full rank: the factors written and read by two solves, the dense
        # LU, two solves, the matrix and one matrix-free product with dA/d ell
        return dict(bytes=8.0 * (3.0 * n * n + 7.0 * n), flops=2.0 / 3.0 * n ** 3 + 4.0 * n * n + 20.0 * n * n)
    r = _mean_rank(case)
    s = 4.0 if case.get("precision") == "f32" else 8.0
    off = nb * (nb - 1.0)
    lr = off * r * (2.0 * b + r)
    dense = n * b * (1.0 + 2.0 * case.get("admis", 0))
    nrhs = case.get("nrhs", 0)
    if kind == "build":
        # points in, vectors in and out; a rank-r factorization needs r columns and rows of every tile
        return dict(bytes=8.0 * (n + 2.0 * n * nrhs), flops=off * 4.0 * r * r * b + 6.0 * off * r * b +
                    2.0 * (lr + dense) * nrhs)
    if kind == "kept":
        return dict(bytes=2.0 * 8.0 * (lr + dense + 2.0 * n * nrhs), flops=2.0 * 2.0 * (lr + dense) * nrhs)
    steps3 = nb * (nb - 1.0) * (2.0 * nb - 1.0) / 6.0
    if kind == "qr":
        # the factorization, then the same reflectors applied to the identity
        return dict(bytes=8.0 * 4.0 * (lr + dense), flops=2.0 * steps3 * 16.0 * b * r * r + nb * 4.0 / 3.0 * b ** 3)
    # LU: diagonal factors, panel solves, one recompressed rank-2r sum per tile and step
    fl = nb * 2.0 / 3.0 * b ** 3 + off * 2.0 * r * b * b + steps3 * (16.0 * b * r * r)
    by = s * 2.0 * (lr + dense) + 8.0 * 2.0 * n * nrhs
    fl += 2.0 * (lr + dense) * nrhs
    if kind == "refine":
        fl += 2.0 * n * n * nrhs + 4.0 * n * n
    return dict(bytes=by, flops=fl)


def tolerance(case):
    """About four times the largest error against exact() seen over these ranges.  What
    decides it is the compression: another correct implementation keeps another basis or
    another rank where a singular value lies at the threshold, and its results then differ
    by what the truncation leaves out (eps, or the fixed rank's remainder) times the
    sensitivity of the operation."""
    kind, eps = case["kind"], case.get("eps")
    if kind == "lu":
        return dict(rel=40.0 * eps if eps else {8: 1e-5, 12: 3e-8, 16: 1e-10}[case["rank"]])
    if kind == "refine":
        return dict(rel=6e-4 if case["precision"] == "f32" else 2e-8)
    if kind == "kept":
        return dict(rel=40.0 * eps)
    if kind == "qr":
        return dict(rel=2e-5 if eps == 1e-8 else 2e-6)
    if kind == "add":
        return dict(rel=2.5e-6 if case["dtype"] == "f32" else 2.0 * eps if eps else 1e-12)
    if kind == "adjoint":
        return dict(rel=3e-7)
    if kind == "build":
        return dict(rel=8.0 * eps)
    return dict(rel=4e-14)


def _dense_kernel(pts, shift, kernel="laplace", ell=0.0):
    p = torch.from_numpy(np.vstack(pts)).cuda()
    n = p.shape[1]
    if kernel == "laplace" and p.shape[0] == 1:
        a = (p[0][:, None] - p[0][None, :]).abs_().add_(1e-3).reciprocal_()
    else:
        d2 = sum((q[:, None] - q[None, :]) ** 2 for q in p)
        a = 1.0 / (d2.sqrt() + 1e-3) if kernel == "laplace" else torch.exp(-d2 / (2.0 * ell ** 2))
    a.diagonal().add_(shift)
    return a


def exact(case, seed):
    kind = case["kind"]
    if kind in ("lu", "refine", "kept"):
        # the exact kernel matrix: symmetric positive definite
        a = _dense_kernel(_points(case, seed), _SHIFT[kind])
        x = torch.linalg.solve(a, _rhs(case["n"], case["nrhs"], seed))
        return [x, x.clone()] if kind == "kept" else x
    if kind == "build":
        return _dense_kernel(_points(case, seed), _SHIFT[kind]) @ _rhs(case["n"], case["nrhs"], seed)
    if kind == "adjoint":
        pts, ell = _points(case, seed), case["ell"]
        a = _dense_kernel(pts, 1e-4, "gaussian", ell)
        u = torch.linalg.solve(a, _rhs(case["n"], 1, seed))
        lam = torch.linalg.solve(a, u)
        p = torch.from_numpy(np.vstack(pts)).cuda()
        d2 = sum((q[:, None] - q[None, :]) ** 2 for q in p)
        a.diagonal().sub_(1e-4)
        return dict(u=u, db=lam, dell=-(lam * ((a * d2 / ell ** 3) @ u)).sum().cpu())
    if kind == "tilelu":
        a = _tiles(case, seed)
        for k in range(case["n"] - 1):
            a[:, k + 1:, k] /= a[:, k, k, None]
            a[:, k + 1:, k + 1:] -= a[:, k + 1:, k, None] * a[:, k, None, k + 1:]
        return a
    if kind == "add":
        out = []
        for g in _add_inputs(case, seed)[0]:
            U, S, V = (x.double() for x in g["A"])
            B = ([x.double() for x in f] for f in g["B"])
            s = U @ (S @ V) + torch.cat([u @ (c @ v) for u, c, v in B])
            if case["eps"] == 0.0:  # fixed rank: the best approximation of that rank
                u, sv, v = torch.linalg.svd(s, full_matrices=False)
                k = g["ks"][0][0]
                s = (u[:, :, :k] * sv[:, None, :k]) @ v[:, :k]
            out.append(s)
        return out
    # qr: the tiled flat-tree Householder QR on the dense matrix
    n, nb = case["n"], case["nb"]
    b = n // nb
    at = [slice(b * i, b * (i + 1)) for i in range(nb)]
    w = np.concatenate([_dense_kernel(_points(case, seed), 0.0).cpu().numpy(), np.eye(n)], axis=1)
    for k in range(nb):
        for i in range(k, nb):
            rows = np.r_[at[k]] if i == k else np.r_[at[k], at[i]]
            a = w[rows, at[k]]
            if i > k:
                a[:b] = np.triu(a[:b])
            q, _ = np.linalg.qr(a, mode="complete")
            w[rows, at[k]] = a
            w[rows, at[k].start:] = q.T @ w[rows, at[k].start:]
    return dict(r=np.triu(w[:, :n]), q=w[:, n:].T.copy())
