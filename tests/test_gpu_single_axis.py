"""GPU: plans with one active axis give the same numbers whichever axis that
is -- forward, adjoint, the PSF and the Toeplitz normal operator, at the
lengths whose FFT (of n or, for the PSF, of 2 n points) has a kernel of its own
and at others -- and agree with the oracle to 1e-5, as every operator."""
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


@pytest.mark.parametrize("n", [8, 16, 32, 33, 40, 64, 96, 128, 160, 192, 256, 320, 384])
def test_single_axis(n):
    import bart_amd as ba
    rng = np.random.default_rng(n)
    M, C = 500, 2
    k = (rng.random(M) - 0.5) * n * 0.98
    img = (rng.standard_normal((C, n)) + 1j * rng.standard_normal((C, n))).astype(np.complex64)
    first = None
    for axis in range(3):
        dims = tuple(n if d == axis else 1 for d in range(3))
        traj = np.zeros((M, 3), np.complex64)
        traj[:, axis] = k
        op = ba.nufft_create2(d16(1, M, 1, C), d16(*dims, C), d16(3, M), ba.traj_array(traj),
                              conf=ba.NufftConf.defaults(toeplitz=True))
        ref = O.Nufft(dims, traj, C, toeplitz=True)
        x = torch.from_numpy(img.reshape(-1)).cuda()
        y = op.forward(x)
        cim = img.reshape((C,) + dims[::-1])
        assert relerr(y.cpu(), ref.forward(cim)) < 1e-5
        assert relerr(op.normal(x).cpu(), ref.normal(cim)) < 1e-5
        out = [y.cpu().numpy(), op.adjoint(y).cpu().numpy(), np.asarray(op.get_psf()).ravel(),
               op.normal(x).cpu().numpy()]
        op.free()
        if first is None:
            first = out
        for a, b in zip(out, first):
            assert np.array_equal(a, b)
