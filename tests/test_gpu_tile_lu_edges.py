"""The one-launch tile LU where its last 64 x 64 block is ragged: the padding of that
block must be the identity whatever wave stores last (a zero left on the padded diagonal
turns the block's inverses into NaN)."""
import numpy as np
import pytest

from oracle import frank_oracle as fo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 17, 63, 66, 127, 191, 250, 319, 383, 385, 447, 511])
def test_ragged_last_block(torch_gpu, fa, n):
    torch = torch_gpu
    print(f"tile LU n={n}", flush=True)
    a = fo.laplacend([fo.get_sorted_random_vector(2 * n)], 0, n, 0, n) + 10.0 * np.eye(n)
    ref_l, ref_u = fo.getrf_nopiv(a)
    for _ in range(3):
        t = torch.from_numpy(a.copy()).cuda()
        assert list(fa.getrf_nopiv_batched([t])) == [0]
        lu = t.cpu().numpy()
        np.testing.assert_allclose(np.tril(lu, -1) + np.eye(n), ref_l, rtol=0, atol=1e-12)
        np.testing.assert_allclose(np.triu(lu), ref_u, rtol=0, atol=1e-12 * np.abs(ref_u).max())


@pytest.mark.parametrize("n,nb", [(5003, 13), (1000, 3), (999, 8)])
def test_blr_lu_with_ragged_tiles(torch_gpu, fa, n, nb):
    """A block LU whose tiles are not whole multiples of 64 solves to the compression accuracy."""
    torch = torch_gpu
    from frank_amd.inputs import sorted_uniform_points
    print(f"BLR-LU n={n} nb={nb}", flush=True)
    eps = 1e-8
    A = fa.BlrMatrix.from_kernel([sorted_uniform_points(n)], nb, eps=eps, shift=1e-2, kcap=64)
    xs = torch.from_numpy(fo.random_uniform(n, 1)).cuda()
    b = torch.zeros_like(xs)
    A.matvec(xs, b)
    A.set_lra("rounded_addition")
    A.getrf()
    A.solve(b)
    assert torch.linalg.norm(b - xs) <= eps * torch.linalg.norm(xs)
