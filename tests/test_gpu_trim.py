"""Device memory that a context keeps between calls is given back on request."""
import ctypes

import numpy as np
import pytest

from frank_amd import _lib as L


def test_null_context_is_an_argument_error():
    assert L.lib().frk_ctx_trim(ctypes.c_void_p(None)) == L.FRK_ERR_ARG


@pytest.mark.gpu
def test_build_buffer_is_given_back(torch_gpu, fa):
    torch = torch_gpu
    from frank_amd.inputs import sorted_uniform_points
    ctx = fa.Context()
    free = lambda: (ctx.synchronize(), torch.cuda.synchronize(), torch.cuda.mem_get_info()[0])[2]
    build = lambda: fa.BlrMatrix.from_kernel([sorted_uniform_points(8192)], 16, eps=1e-8, shift=1e-2, kcap=64, ctx=ctx)
    A = build()
    held = free()
    ctx.trim()
    tiles = 16 * 15 * 512 * 512 * 8  # the uncompressed tiles of the build
    assert free() >= held + tiles
    ctx.trim()  # nothing left: allowed
    # the matrix is whole, and everything runs on a context without buffers
    xs = torch.from_numpy(np.random.default_rng(0).standard_normal((8192, 2))).cuda()
    y, z, w = (torch.zeros_like(xs) for _ in range(3))
    A.matvec(xs, y)
    ctx.trim()
    B = build()
    assert np.array_equal(A.ranks(), B.ranks())
    B.matvec(xs, z)
    assert torch.equal(y, z)
    A.set_lra("rounded_addition")
    ctx.trim()
    A.getrf()
    ctx.trim()
    A.solve(y)
    assert torch.linalg.norm(y - xs) <= 1e-6 * torch.linalg.norm(xs)
    B.matvec(xs, w)
    assert torch.equal(w, z)
