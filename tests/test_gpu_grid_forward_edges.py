"""GPU: the forward gather in all its variants -- one, two and three active
dims, one and four coils per thread (with a chunk that does not fill), three,
four and eight taps per dim, periodic grids of even and odd dims, samples over
the edges of k-space, and the staged tiles of a 3-D plan (even and odd first dim:
with and without) -- against the oracle, FP32 sums of both sides: 1e-5 as for
every operator."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def d16(*d):
    return list(d) + [1] * (16 - len(d))


def relerr(a, ref):
    a = np.asarray(a, np.complex128).ravel()
    ref = np.asarray(ref, np.complex128).ravel()
    return float(np.linalg.norm(a - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("dims", [(50, 1, 1), (1, 24, 1), (33, 28, 1), (20, 1, 14), (12, 10, 16), (11, 12, 9)])
@pytest.mark.parametrize("C", [1, 4, 7])
@pytest.mark.parametrize("width,periodic", [(6.0, False), (6.0, True), (7.5, False), (10.0, False)])
@pytest.mark.parametrize("M", [1, 65, 3000])
def test_grid_forward_edges(dims, C, width, periodic, M):
    import bart_amd as ba
    rng = np.random.default_rng(M + C + dims[0])
    traj = np.zeros((M, 3), np.complex64)
    for d in range(3):
        if dims[d] > 1:
            traj[:, d] = (rng.random(M) - 0.5) * dims[d] * 1.05
    img = (rng.standard_normal((C,) + dims[::-1]) + 1j * rng.standard_normal((C,) + dims[::-1])).astype(np.complex64)
    w = (0.5 + rng.random(M)).astype(np.complex64)
    conf = ba.NufftConf.defaults(toeplitz=False, width=width, periodic=periodic)
    op = ba.nufft_create2(d16(1, M, 1, C), d16(*dims, C), d16(3, M), ba.traj_array(traj), weights=w, conf=conf)
    ref = O.Nufft(dims, traj, C, weights=w, toeplitz=False, width=width, periodic=periodic)
    x = torch.from_numpy(img.reshape(-1)).cuda()
    y = op.forward(x)
    assert relerr(y.cpu(), ref.forward(img)) < 1e-5
    assert torch.equal(y, op.forward(x))
    op.free()
