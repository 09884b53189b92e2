"""GPU: the adjoint gridding at the edges of its work split -- one, two and
three active dims, every coil-chunk width (4, 8, 16) with a chunk that does
not fill, four and eight taps per dim, tiles cut by the grid, periodic grids of
even and odd dims, among them some smaller than the kernel's reach and some with
fewer points than taps, batches of visits that do not fill and tiles
split over several work items -- against the oracle, FP32 sums of both sides:
1e-5 as for every operator."""
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


@pytest.mark.parametrize("dims", [(50, 1, 1), (33, 28, 1), (10, 12, 9), (18, 16, 1), (8, 6, 4), (5, 3, 2), (2, 1, 1)])
@pytest.mark.parametrize("C", [1, 7, 17])
@pytest.mark.parametrize("width,periodic", [(6.0, False), (6.0, True), (10.0, False), (10.0, True)])
@pytest.mark.parametrize("M", [1, 300, 9000])
def test_grid_adjoint_edges(dims, C, width, periodic, M):
    import bart_amd as ba
    rng = np.random.default_rng(M + C + dims[0])
    traj = np.zeros((M, 3), np.complex64)
    for d in range(3):
        if dims[d] > 1:
            # most samples near the centre (tiles of thousands of visits),
            # some over the edges of k-space
            k = rng.standard_normal(M) * dims[d] / 12
            far = rng.random(M) < 0.3
            k[far] = (rng.random(far.sum()) - 0.5) * dims[d] * 1.05
            traj[:, d] = k
    ksp = (rng.standard_normal((C, M)) + 1j * rng.standard_normal((C, M))).astype(np.complex64)
    w = (0.5 + rng.random(M)).astype(np.complex64)
    conf = ba.NufftConf.defaults(toeplitz=False, width=width, periodic=periodic)
    op = ba.nufft_create2(d16(1, M, 1, C), d16(*dims, C), d16(3, M), ba.traj_array(traj), weights=w, conf=conf)
    ref = O.Nufft(dims, traj, C, weights=w, toeplitz=False, width=width, periodic=periodic)
    y = torch.from_numpy(ksp.reshape(-1)).cuda()
    a = op.adjoint(y)
    assert relerr(a.cpu(), ref.adjoint(ksp)) < 1e-5
    assert torch.equal(a, op.adjoint(y))
    op.free()


# samples many periods away (coordinates of 1/64: exact in FP32) are those of the
# first period, at the ends of the grid too
@pytest.mark.parametrize("dims", [(32, 1, 1), (20, 33, 1), (12, 10, 9)])
@pytest.mark.parametrize("periods", [5, 9, -11])
def test_grid_periods_away(dims, periods):
    import bart_amd as ba
    C, M = 3, 2000
    rng = np.random.default_rng(7)
    traj = np.zeros((M, 3), np.complex64)
    for d in range(3):
        if dims[d] > 1:
            traj[:, d] = np.round((rng.random(M) - 0.5) * dims[d] * 64) / 64
    far = traj + np.array([n * periods if n > 1 else 0 for n in dims])
    ksp = (rng.standard_normal((C, M)) + 1j * rng.standard_normal((C, M))).astype(np.complex64)
    y = torch.from_numpy(ksp.reshape(-1)).cuda()
    conf = ba.NufftConf.defaults(toeplitz=False, periodic=True)
    out = []
    for t in (traj, far):
        op = ba.nufft_create2(d16(1, M, 1, C), d16(*dims, C), d16(3, M), ba.traj_array(t.astype(np.complex64)), conf=conf)
        a = op.adjoint(y)
        out.append((a.cpu(), op.forward(a).cpu()))
        op.free()
    assert relerr(out[1][0], out[0][0]) < 1e-6
    assert relerr(out[1][1], out[0][1]) < 1e-6
