"""GPU: the FFT passes over sub-grid pairs at the lengths where their plan
changes -- one, two and three radices, every odd radix, the lengths with a
kernel of their own, column groups that do not fill, coil groups of more than one coil, and lengths without a pair
kernel (over 1024, or no three radices of at most 16) -- against the oracle:
forward, adjoint and the Toeplitz normal operator with coil maps, and over 4096
points without them.  FP32
transforms of both sides: 1e-5, as for every operator."""
import numpy as np
import pytest

import oracle as O
from bart_amd import inputs as I

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def d16(*d):
    return list(d) + [1] * (16 - len(d))


def relerr(a, ref):
    a = np.asarray(a, np.complex128).ravel()
    ref = np.asarray(ref, np.complex128).ravel()
    return float(np.linalg.norm(a - ref) / np.linalg.norm(ref))


CASES = [
    ((2, 16, 1), 3),        # one radix each
    ((13, 14, 1), 2),
    ((18, 22, 1), 2),       # two radices; 18 columns: a group of 16 and two more
    ((169, 26, 1), 3),      # 13 x 13, 2 x 13
    ((210, 36, 1), 2),      # 14 x 15, 6 x 6
    ((121, 1, 1), 2),       # one-dimensional
    ((44, 1, 60), 2),       # active axes x and z
    ((1, 50, 1), 2),        # first active axis is y
    ((320, 24, 1), 5),      # three radices along x
    ((24, 384, 1), 5),      # three radices along y
    ((286, 20, 1), 2),      # 2 x 11 x 13: 143 lanes
    ((512, 520, 1), 16),    # partial images of two coils
    ((30, 28, 33), 3),      # 3-D, unequal
    ((12, 18, 320), 2),     # 3-D, three radices along the last axis
    ((625, 12, 1), 2),      # 5^4: no three radices
    ((12, 1040, 1), 2),     # over 1024
    ((1040, 1, 1), 2),
    ((625, 12, 1), 6),      # coil groups of two
    ((9, 1250, 1), 1),      # columns that do not fill a block of four
    ((10, 7, 1040), 2),     # 3-D, over 1024 along the last axis
    ((6, 1040, 5), 2),      # ... and along one in between
    ((1, 18, 1), 48),       # one-dimensional: groups of 16 coils
    ((24, 1, 1), 7),
    ((1, 1, 2048), 4),
    # 32, 64, 128 and 256 (a kernel of their own): rows and columns, rows that do
    # not fill a wave or a work-group, ragged column groups, one and four waves
    ((32, 33, 1), 2),
    ((64, 3, 1), 1),
    ((128, 18, 1), 3),
    ((256, 7, 1), 2),
    ((18, 64, 1), 2),
    ((33, 32, 1), 2),
    ((1, 32, 1), 2),
    ((5, 128, 1), 2),
    ((22, 256, 1), 2),
    ((1, 64, 1), 3),
    ((256, 128, 1), 17),
    ((64, 10, 128), 5),
    ((6, 128, 64), 2),
    ((32, 32, 32), 3),
]


@pytest.mark.parametrize("dims,C", CASES)
def test_pair_lengths(dims, C):
    import bart_amd as ba
    rng = np.random.default_rng(dims[0] * 7 + dims[1] * 3 + dims[2] + C)
    R, S = 40, 25
    traj = np.zeros((R * S, 3), np.complex64)
    for d in range(3):
        if dims[d] > 1:
            traj[:, d] = (rng.random(R * S) - 0.5) * dims[d] * 0.98
    shape = (C, dims[2], dims[1], dims[0])

    def crandn(s):
        return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)

    maps = crandn(shape)
    maps /= np.sqrt(np.sum(np.abs(maps) ** 2, 0, keepdims=True))
    img, ksp = crandn(shape[1:]), crandn((C, R * S))
    ref = O.Nufft(dims, traj, C, toeplitz=True)
    op, nu = ba.sense_nc_init(d16(*dims, C), d16(*dims, C), maps, d16(1, R, S, C), d16(3, R, S), ba.traj_array(traj),
                              nufft_op=True)
    x = torch.from_numpy(img.reshape(-1)).cuda()
    y = torch.from_numpy(ksp.reshape(-1)).cuda()
    assert relerr(op.forward(x).cpu(), ref.sense_forward(maps, img)) < 1e-5
    assert relerr(op.adjoint(y).cpu(), ref.sense_adjoint(maps, ksp)) < 1e-5
    assert relerr(op.normal(x).cpu(), ref.sense_normal(maps, img)) < 1e-5
    assert relerr(nu.adjoint(y).cpu(), ref.adjoint(ksp)) < 1e-5
    cim = torch.from_numpy((maps * img).reshape(-1)).cuda()
    assert relerr(nu.normal(cim).cpu(), ref.normal(maps * img)) < 1e-5
    nu.free()
    op.free()


# over 4096 points a block holds one member of a pair
def test_single_members():
    import bart_amd as ba
    dims, C, M = (3, 4400, 1), 2, 500
    rng = np.random.default_rng(1)
    traj = np.zeros((M, 3), np.complex64)
    for d in range(2):
        traj[:, d] = (rng.random(M) - 0.5) * dims[d] * 0.98

    def crandn(*s):
        return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)

    img, ksp = crandn(C, 1, dims[1], dims[0]), crandn(C, M)
    ref = O.Nufft(dims, traj, C, toeplitz=False)
    op = ba.nufft_create2(d16(1, M, 1, C), d16(*dims, C), d16(3, M), ba.traj_array(traj),
                          conf=ba.NufftConf.defaults(toeplitz=False))
    assert relerr(op.forward(torch.from_numpy(img.reshape(-1)).cuda()).cpu(), ref.forward(img)) < 1e-5
    assert relerr(op.adjoint(torch.from_numpy(ksp.reshape(-1)).cuda()).cpu(), ref.adjoint(ksp)) < 1e-5
    op.free()


# ... and so the normal operator of a given PSF, against its definition in 64
# bits (12 points: the definition itself, on the pair kernels)
@pytest.mark.parametrize("n", [12, 4400])
def test_single_members_normal(n):
    import bart_amd as ba
    dims, C = (3, n, 1), 2
    rng = np.random.default_rng(n)

    def crandn(*s):
        return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)

    img, psf = crandn(C, n, 3), crandn(4, n, 3)
    conf = ba.NufftConf.defaults(toeplitz=True)
    op = ba.nufft_create_normal(d16(*dims, C), list(dims) + [1] * 13 + [4], psf.reshape(-1), conf=conf)
    y = op.normal(torch.from_numpy(img.reshape(-1)).cuda()).cpu()
    op.free()

    def phase(m, b):
        j = np.arange(m)
        c = m // 2
        fm = np.exp(2j * np.pi * (j - c / 2) * c / m)
        shift = -0.5 * b + m / 2 - m // 2
        return np.exp(2j * np.pi * shift / m * (j - m / 2)) * fm

    ref = 0
    for s in range(4):
        l = phase(n, s >> 1)[:, None] * phase(3, s & 1)[None, :]
        ref = ref + np.conj(l) * np.fft.ifft2(psf[s] * np.fft.fft2(l * img.astype(np.complex128)))
    assert relerr(y, ref) < 1e-5


def test_first_axis_limit():
    """The entry points take 2^d transforms of the first axis up to 8192 points."""
    import bart_amd as ba
    traj = np.zeros((8, 3), np.complex64)
    op = ba.nufft_create2(d16(1, 8, 1, 1), d16(2560, 4, 1, 1), d16(3, 8, 1), ba.traj_array(traj),
                          conf=ba.NufftConf.defaults(toeplitz=False))
    with pytest.raises(ba.BartError, match="exceeds LDS budget"):
        op.forward(torch.zeros(2560 * 4, dtype=torch.complex64, device="cuda"))


# more partial images of the sum over coils than one sum takes: 64 of several
# coils each, and a number of coils without a divisor that gives 64 (67, 130)
@pytest.mark.parametrize("dims,C", [((12, 10, 1), 128), ((14, 1, 1), 130), ((32, 6, 1), 67), ((16, 12, 1), 96)])
def test_many_coils(dims, C):
    test_pair_lengths(dims, C)
