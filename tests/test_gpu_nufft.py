"""GPU parity: the HIP library through its C ABI against the CPU oracle (a C
restatement of BART's NUFFT path) on identical seeded inputs.

Tolerances: relative L2 <= 1e-5 for single operator applications (the
north-star bar against BART), looser where FP32 error compounds over many CG
iterations (stated per test).
"""
import numpy as np
import pytest

import bart_amd as ba
import oracle as O
from bart_amd import inputs as I
from conftest import crandn, relerr

pytestmark = pytest.mark.gpu


def dims16(*d):
    return list(d) + [1] * (16 - len(d))


def make_nufft(img, C, traj, R, S, weights=None, **conf):
    X, Y, Z = img
    c = ba.NufftConf.defaults(**conf)
    return ba.nufft_create2(dims16(1, R, S, C), dims16(X, Y, Z, C), dims16(3, R, S), ba.traj_array(traj),
                            dims16(1, R, S) if weights is not None else None, weights, c)


# --------------------------------------------------------------------------
# FFT
# --------------------------------------------------------------------------

@pytest.mark.parametrize("n", [2, 8, 12, 30, 64, 128, 192, 256, 320, 384, 512, 640, 768, 56, 286, 1024])
def test_fft_1d_matches_numpy(n):
    x = crandn((5, n), n)
    y = ba.fft([n, 1, 1, 5], 1, x)
    ref = np.fft.fft(x.astype(np.complex128), axis=1)
    assert relerr(y.reshape(5, n), ref) < 2e-6
    z = ba.ifft([n, 1, 1, 5], 1, x)
    refi = np.fft.ifft(x.astype(np.complex128), axis=1) * n
    assert relerr(z.reshape(5, n), refi) < 2e-6


@pytest.mark.parametrize("shape,flags", [((16, 24, 1), 3), ((64, 64, 1), 3), ((256, 256, 1), 3),
                                         ((12, 10, 8), 7), ((32, 32, 32), 7), ((40, 1, 20), 5),
                                         ((16, 24, 8), 2), ((16, 24, 8), 4),
                                         ((64, 64, 8), 7), ((96, 96, 4), 7), ((128, 128, 6), 7)])
def test_fft_nd_matches_numpy(shape, flags):
    # square x-y slices of 3-d arrays go through the LDS slice passes
    X, Y, Z = shape
    x = crandn((3, Z, Y, X), X + Y + Z)
    y = ba.fft([X, Y, Z, 3], flags, x).reshape(3, Z, Y, X)
    axes = tuple(3 - a for a in range(3) if flags & (1 << a))
    ref = np.fft.fftn(x.astype(np.complex128), axes=axes)
    assert relerr(y, ref) < 3e-6
    z = ba.ifft([X, Y, Z, 3], flags, x).reshape(3, Z, Y, X)
    refi = np.fft.ifftn(x.astype(np.complex128), axes=axes) * np.prod([shape[a] for a in range(3) if flags & (1 << a)])
    assert relerr(z, refi) < 3e-6


# --------------------------------------------------------------------------
# NUFFT forward / adjoint
# --------------------------------------------------------------------------

CASES_2D = [
    dict(n=64, C=3, R=128, S=21, periodic=False),
    dict(n=64, C=1, R=128, S=33, periodic=True),
    dict(n=96, C=4, R=192, S=17, periodic=False),
]


@pytest.mark.parametrize("case", CASES_2D)
def test_nufft_2d_forward_adjoint(case):
    n, C, R, S = case["n"], case["C"], case["R"], case["S"]
    traj = I.radial_traj(R, S)
    cim = crandn((C, 1, n, n), 1)
    ksp = crandn((C, R * S), 2)
    ref = O.Nufft((n, n, 1), traj, C, toeplitz=False, periodic=case["periodic"])
    op = make_nufft((n, n, 1), C, traj, R, S, toeplitz=False, periodic=case["periodic"])
    k = op.forward(cim).reshape(C, R * S)
    assert relerr(k, ref.forward(cim)) < 1e-5
    x = op.adjoint(ksp).reshape(C, 1, n, n)
    assert relerr(x, ref.adjoint(ksp)) < 1e-5


def test_nufft_2d_weights():
    n, C, R, S = 64, 2, 128, 15
    traj = I.radial_traj(R, S)
    w = (0.5 + np.random.default_rng(3).random(R * S)).astype(np.complex64)
    cim = crandn((C, 1, n, n), 4)
    ksp = crandn((C, R * S), 5)
    ref = O.Nufft((n, n, 1), traj, C, weights=w, toeplitz=False)
    op = make_nufft((n, n, 1), C, traj, R, S, weights=w, toeplitz=False)
    assert relerr(op.forward(cim).reshape(C, -1), ref.forward(cim)) < 1e-5
    assert relerr(op.adjoint(ksp).reshape(C, 1, n, n), ref.adjoint(ksp)) < 1e-5


def test_nufft_3d_forward_adjoint():
    n, C = 24, 2
    traj = I.phyllotaxis_kooshball(spokes=64, readout=48)
    R, S = 48, 64
    cim = crandn((C, n, n, n), 6)
    ksp = crandn((C, R * S), 7)
    ref = O.Nufft((n, n, n), traj, C, toeplitz=False)
    op = make_nufft((n, n, n), C, traj, R, S, toeplitz=False)
    assert relerr(op.forward(cim).reshape(C, -1), ref.forward(cim)) < 1e-5
    assert relerr(op.adjoint(ksp).reshape(C, n, n, n), ref.adjoint(ksp)) < 1e-5


@pytest.mark.parametrize("dims,C,weighted", [((20, 12, 10), 6, True), ((15, 12, 10), 3, False),
                                              ((32, 32, 32), 5, False), ((48, 40, 36), 4, True)])
def test_nufft_3d_forward_home_tiles(monkeypatch, dims, C, weighted):
    # forward gather from home tiles staged in LDS (3-D, even x size) against
    # the per-sample gather from the grid: the same terms in the same order,
    # so the same bits; a partial coil chunk (C not a multiple of 4), grid
    # edges inside a tile and samples beyond the grid (readout longer than
    # the y and z sizes); odd x size: per-sample gather only
    X, Y, Z = dims
    R, S = 2 * X, 150
    traj = I.phyllotaxis_kooshball(spokes=S, readout=R)
    w = (0.5 + np.random.default_rng(8).random(R * S)).astype(np.complex64) if weighted else None
    cim = crandn((C, Z, Y, X), 70 + X)
    a = make_nufft(dims, C, traj, R, S, weights=w, toeplitz=False)
    monkeypatch.setenv("BART_AMD_FWD_TILES", "off")
    b = make_nufft(dims, C, traj, R, S, weights=w, toeplitz=False)
    fa, fb = a.forward(cim), b.forward(cim)
    assert np.array_equal(fa, fb)
    ref = O.Nufft(dims, traj, C, weights=w, toeplitz=False)
    assert relerr(fa.reshape(C, -1), ref.forward(cim)) < 1e-5


@pytest.mark.parametrize("n,C,S", [(32, 3, 200), (64, 1, 300)])
def test_nufft_3d_slice_path(n, C, S):
    # x-y slices transformed in LDS (square slices up to 128 x 128); the dense
    # centre tiles are split over several work-groups in the tile kernel
    R = 2 * n
    traj = I.phyllotaxis_kooshball(spokes=S, readout=R)
    cim = crandn((C, n, n, n), 60 + n)
    ksp = crandn((C, R * S), 61 + n)
    ref = O.Nufft((n, n, n), traj, C, toeplitz=False)
    op = make_nufft((n, n, n), C, traj, R, S, toeplitz=False)
    assert relerr(op.forward(cim).reshape(C, -1), ref.forward(cim)) < 1e-5
    assert relerr(op.adjoint(ksp).reshape(C, n, n, n), ref.adjoint(ksp)) < 1e-5


def test_nufft_3d_32_points():
    # 32^3: every axis on the kernels of that length
    n, C, R, S = 32, 2, 64, 60
    traj = I.phyllotaxis_kooshball(spokes=S, readout=R)
    cim = crandn((C, n, n, n), 66)
    ksp = crandn((C, R * S), 67)
    op = make_nufft((n, n, n), C, traj, R, S, toeplitz=False)
    ref = O.Nufft((n, n, n), traj, C, toeplitz=False)
    assert relerr(op.forward(cim).reshape(C, -1), ref.forward(cim).reshape(C, -1)) < 1e-5
    assert relerr(op.adjoint(ksp).reshape(C, -1), ref.adjoint(ksp).reshape(C, -1)) < 1e-5
    op.free()


def test_nufft_2d_dense_adjoint():
    # 2-D radial with a centre dense enough to split tiles (> 2048 visits)
    n, C, R, S = 64, 2, 128, 201
    traj = I.radial_traj(R, S)
    ksp = crandn((C, R * S), 64)
    ref = O.Nufft((n, n, 1), traj, C, toeplitz=False)
    op = make_nufft((n, n, 1), C, traj, R, S, toeplitz=False)
    assert relerr(op.adjoint(ksp).reshape(C, 1, n, n), ref.adjoint(ksp)) < 1e-5


def test_nufft_2d_adjoint_many_work_items():
    # 448^2: 784 tiles x 2 coil chunks (20 coils = 16 + 4), more work items
    # than the persistent work-groups of the adjoint gridding, so that each
    # work-group runs several items in a row; repeated calls are bitwise equal
    n, C, R, S = 448, 20, 896, 41
    traj = I.radial_traj(R, S)
    ksp = crandn((C, R * S), 65)
    ref = O.Nufft((n, n, 1), traj, C, toeplitz=False)
    op = make_nufft((n, n, 1), C, traj, R, S, toeplitz=False)
    a = op.adjoint(ksp)
    assert relerr(a.reshape(C, 1, n, n), ref.adjoint(ksp)) < 1e-5
    assert np.array_equal(a, op.adjoint(ksp))


def test_nufft_nonsquare_and_1d():
    traj = I.radial_traj(64, 9)
    traj[:, 1] *= 0.5
    op = make_nufft((64, 32, 1), 2, traj, 64, 9, toeplitz=False)
    ref = O.Nufft((64, 32, 1), traj, 2, toeplitz=False)
    cim = crandn((2, 1, 32, 64), 8)
    assert relerr(op.forward(cim).reshape(2, -1), ref.forward(cim)) < 1e-5
    t1 = np.zeros((40, 3), np.complex64)
    t1[:, 0] = np.linspace(-15.5, 15.5, 40)
    op1 = make_nufft((32, 1, 1), 1, t1, 40, 1, toeplitz=False)
    ref1 = O.Nufft((32, 1, 1), t1, 1, toeplitz=False)
    x = crandn((1, 1, 1, 32), 9)
    assert relerr(op1.forward(x).reshape(1, -1), ref1.forward(x)) < 1e-5


def test_nufft_cartesian_is_unitary_centred_dft():
    # tests/nufft.mk:28-36: Cartesian trajectory, periodic -> fftuc (nrmse 5e-5)
    n = 64
    traj = I.cartesian_traj(n, n)
    img = I.ellipse_phantom(n, seed=11)
    op = make_nufft((n, n, 1), 1, traj, n * n, 1, toeplitz=False, periodic=True)
    k = op.forward(img).reshape(n, n)
    F = np.fft.fftshift(np.fft.fft2(np.fft.ifftshift(img[0].astype(np.complex128)))) / n
    assert relerr(k, F) < 5e-5


def test_nufft_vs_fp64_nudft():
    # tests/nufft.mk:41-49: NUFFT vs NUDFT on a radial trajectory (nrmse 2e-5)
    n, R, S = 64, 128, 12
    traj = I.radial_traj(R, S)
    img = I.ellipse_phantom(n, seed=12)
    op = make_nufft((n, n, 1), 1, traj, R, S, toeplitz=False, periodic=True)
    k = op.forward(img).reshape(1, -1)
    ref = O.nudft_forward((n, n, 1), traj, img)
    assert relerr(k, ref) < 2e-5
    a = op.adjoint(k.astype(np.complex64)).reshape(1, 1, n, n)
    refa = O.nudft_adjoint((n, n, 1), traj, k)
    assert relerr(a, refa) < 2e-5


@pytest.mark.parametrize("img,C", [((32, 32, 1), 1), ((32, 32, 1), 2), ((12, 10, 8), 2)])
def test_nudft_matches_fp64(img, C):
    # nufft -s (noncart/nudft.c): BART scales by 1/sqrt(size of the coil-image
    # array), i.e. 1/sqrt(N C); the FP64 reference scales by 1/sqrt(N)
    X, Y, Z = img
    R, S = 2 * X, 9
    traj = I.radial_traj(R, S) if Z == 1 else I.phyllotaxis_kooshball(spokes=S, readout=R)
    op = ba.nudft_create(dims16(1, R, S, C), dims16(X, Y, Z, C), dims16(3, R, S), ba.traj_array(traj))
    x = crandn((C, Z, Y, X), 90)
    k = op.forward(x).reshape(C, -1)
    assert relerr(k, O.nudft_forward(img, traj, x) / np.sqrt(C)) < 1e-5
    y = crandn((C, R * S), 91)
    a = op.adjoint(y).reshape(C, Z, Y, X)
    assert relerr(a, O.nudft_adjoint(img, traj, y) / np.sqrt(C)) < 1e-5
    # normal operator = adjoint(forward(x))
    nrm = op.normal(x).reshape(C, Z, Y, X)
    assert relerr(nrm, op.adjoint(op.forward(x)).reshape(C, Z, Y, X)) < 1e-6


def test_nufft_adjoint_dot_test():
    # utests/test_nufft.c:108-121 / tests/nufft.mk:90-104
    n, C, R, S = 128, 2, 256, 64
    traj = I.radial_traj(R, S)
    op = make_nufft((n, n, 1), C, traj, R, S, toeplitz=False)
    x = crandn((C, 1, n, n), 13)
    y = crandn((C, R * S), 14)
    Ax = op.forward(x)
    Ahy = op.adjoint(y)
    s1 = np.vdot(y.ravel().astype(np.complex128), Ax.astype(np.complex128))
    s2 = np.vdot(Ahy.astype(np.complex128), x.ravel().astype(np.complex128))
    assert abs(s1 - s2) / abs(s1) < 1e-5


# --------------------------------------------------------------------------
# PSF and Toeplitz normal operator
# --------------------------------------------------------------------------

@pytest.mark.parametrize("img,R,S,C,weighted", [((64, 64, 1), 128, 21, 2, False), ((48, 48, 1), 96, 13, 3, True),
                                                ((20, 20, 20), 40, 48, 2, False),
                                                ((32, 32, 32), 64, 150, 2, True),
                                                # z lengths with the pair z-pass (sub-grids s, s + 4
                                                # share one x-y transform)
                                                ((32, 32, 64), 64, 120, 2, True),
                                                ((64, 64, 64), 128, 100, 2, False)])
def test_psf_and_toeplitz_normal(img, R, S, C, weighted):
    X, Y, Z = img
    traj = I.radial_traj(R, S) if Z == 1 else I.phyllotaxis_kooshball(spokes=S, readout=R)
    w = (0.5 + np.random.default_rng(4).random(R * S)).astype(np.complex64) if weighted else None
    ref = O.Nufft(img, traj, C, weights=w, toeplitz=True)
    op = make_nufft(img, C, traj, R, S, weights=w, toeplitz=True)
    psf = op.get_psf().reshape(ref.psf().shape)
    assert relerr(psf, ref.psf()) < 1e-5
    x = crandn((C, Z, Y, X), 15)
    y = op.normal(x).reshape(C, Z, Y, X)
    assert relerr(y, ref.normal(x)) < 1e-5


@pytest.mark.parametrize("Z", [64, 128, 256, 512])
def test_nufft_3d_z_lengths(Z):
    # forward, adjoint and the Toeplitz normal operator at the power-of-two
    # lengths of the last axis: three with kernels of their own, and three
    # radices (512)
    img, R, S, C = (32, 32, Z), 64, 90, 2
    X, Y, Z = img
    traj = I.phyllotaxis_kooshball(spokes=S, readout=R)
    w = (0.5 + np.random.default_rng(5).random(R * S)).astype(np.complex64)
    op = make_nufft(img, C, traj, R, S, weights=w, toeplitz=False)
    ref = O.Nufft(img, traj, C, weights=w, toeplitz=False)
    cim = crandn((C, Z, Y, X), 18)
    ksp = crandn((C, R * S), 19)
    assert relerr(op.forward(cim).reshape(C, -1), ref.forward(cim)) < 1e-5
    assert relerr(op.adjoint(ksp).reshape(C, Z, Y, X), ref.adjoint(ksp)) < 1e-5
    op.free()
    t = make_nufft(img, C, traj, R, S, weights=w, toeplitz=True)
    reft = O.Nufft(img, traj, C, weights=w, toeplitz=True)
    assert relerr(t.normal(cim).reshape(C, Z, Y, X), reft.normal(cim)) < 1e-5
    t.free()


def test_toeplitz_3d_64_points():
    # 64^3, three coils: split, turn and merge of every axis at that length
    img, R, S, C = (64, 64, 64), 128, 80, 3
    traj = I.phyllotaxis_kooshball(spokes=S, readout=R)
    op = make_nufft(img, C, traj, R, S, toeplitz=True)
    ref = O.Nufft(img, traj, C, toeplitz=True)
    x = crandn((C, 64, 64, 64), 17)
    assert relerr(op.normal(x).reshape(C, 64, 64, 64), ref.normal(x)) < 1e-5
    op.free()


def test_psf_update_roundtrip():
    n, R, S = 32, 64, 11
    traj = I.radial_traj(R, S)
    op = make_nufft((n, n, 1), 1, traj, R, S, toeplitz=True)
    psf = op.get_psf()
    x = crandn((1, 1, n, n), 16)
    y0 = op.normal(x)
    op.update_psf(2.0 * psf)
    y1 = op.normal(x)
    assert relerr(y1, 2.0 * y0) < 1e-6


# --------------------------------------------------------------------------
# SENSE model (sense_nc_init) and CG
# --------------------------------------------------------------------------

def make_sense(n, C, R, S, Z=1, seed=0, lam_weights=None):
    if Z == 1:
        traj = I.radial_traj(R, S)
        img = I.ellipse_phantom(n, seed=seed)
    else:
        traj = I.phyllotaxis_kooshball(spokes=S, readout=R)
        img = I.ellipsoid_phantom(n, nell=6, seed=seed)
    maps = I.gaussian_coils((Z, n, n), C, seed=seed)
    max_dims = dims16(n, n, Z, C)
    op = ba.sense_nc_init(max_dims, dims16(n, n, Z, C), maps, dims16(1, R, S, C), dims16(3, R, S),
                          ba.traj_array(traj))
    ref = O.Nufft((n, n, Z), traj, C, toeplitz=True)
    return op, ref, maps, img, traj


def test_sense_forward_adjoint_normal():
    n, C, R, S = 64, 4, 128, 31
    op, ref, maps, img, traj = make_sense(n, C, R, S, seed=21)
    k = op.forward(img).reshape(C, -1)
    kr = ref.sense_forward(maps, img)
    assert relerr(k, kr) < 1e-5
    y = crandn((C, R * S), 22)
    a = op.adjoint(y).reshape(1, n, n)
    assert relerr(a, ref.sense_adjoint(maps, y)) < 1e-5
    x = crandn((1, n, n), 23)
    nn = op.normal(x).reshape(1, n, n)
    assert relerr(nn, ref.sense_normal(maps, x)) < 1e-5


@pytest.mark.parametrize("n,C", [(32, 4), (32, 6), (64, 3)])
def test_sense_3d_square(n, C):
    # square 3-D plans on the kernels of 32 and 64 points, with the coil sum of
    # S^H over coil groups
    R, S = 2 * n, 120
    op, ref, maps, img, traj = make_sense(n, C, R, S, Z=n, seed=25)
    k = op.forward(img).reshape(C, -1)
    assert relerr(k, ref.sense_forward(maps, img)) < 1e-5
    y = crandn((C, R * S), 26)
    assert relerr(op.adjoint(y).reshape(n, n, n), ref.sense_adjoint(maps, y)) < 1e-5
    x = crandn((n, n, n), 27)
    assert relerr(op.normal(x).reshape(n, n, n), ref.sense_normal(maps, x)) < 1e-5


def test_cgsense_matches_oracle():
    # pics -S -w 1 -r 0.01 -i 30 -t: CG on (A^H A + lambda I) x = A^H y
    n, C, R, S = 64, 4, 128, 41
    op, ref, maps, img, traj = make_sense(n, C, R, S, seed=31)
    y = I.add_noise(ref.sense_forward(maps, img), 1e-3, seed=31)
    b = ref.sense_adjoint(maps, y)
    bg = op.adjoint(y).reshape(1, n, n)
    assert relerr(bg, b) < 1e-5
    lam = 0.01
    # The oracle's adjoint gridding adds with OpenMP atomics (as BART's CPU
    # gridding, noncart/grid.c:482-485), so its sums vary in the last bits
    # from run to run, and FP32 CG amplifies that with the iteration count
    # and the GPU and CPU operators round differently: on this problem the
    # error vs the oracle grows about tenfold every two iterations (measured
    # over four runs: 4 it 7e-7, 6 it 5e-6 .. 1e-5, 8 it 6e-5 .. 1.2e-4,
    # 30 it 2e-5 .. 2e-4).  The solution is compared after 6 iterations; the
    # 30-iteration one by the residual it reaches.
    xr6, _, _, _ = ref.cgsense(maps, b, lam, 6, 0.0)
    x6, _, _ = ba.lsqr_conjgrad(op, b, 6, lam, 0.0)
    err6 = relerr(x6.reshape(1, n, n), xr6)
    xr, itr, trr, _ = ref.cgsense(maps, b, lam, 30, 0.0)
    x, st, tr = ba.lsqr_conjgrad(op, b, 30, lam, 0.0)
    assert st.iterations == itr == 30

    def resid(v):
        v = v.reshape(1, n, n).astype(np.complex64)
        r = b.astype(np.complex128) - ref.sense_normal(maps, v) - lam * v
        return np.linalg.norm(r) / np.linalg.norm(b)

    print(f"cg-sense: 6 it rel err vs oracle {err6:.2e}; 30 it residual {resid(x):.2e} (oracle {resid(xr):.2e}),"
          f" rel err {relerr(x.reshape(1, n, n), xr):.2e}")
    assert err6 < 1e-4
    # measured: GPU 2.19e-4 (deterministic); oracle 1.453e-4 .. 1.471e-4 over
    # 1 and 8 threads -- FP32 CG residuals after 30 iterations of this
    # ill-conditioned problem agree in order, not in digits
    assert resid(x) < 2.0 * resid(xr)
    # the recursively updated residual norms of FP32 CG follow each other
    # closely only for the first iterations of an ill-conditioned problem
    assert np.max(np.abs(tr[:6] / trr[:6] - 1)) < 1e-4
    # deterministic: a second solve gives bitwise the same result
    x2, st2, tr2 = ba.lsqr_conjgrad(op, b, 30, lam, 0.0)
    assert np.array_equal(x2, x) and np.array_equal(tr2, tr)


def test_cgsense_tolerance_and_warm_start():
    n, C, R, S = 64, 4, 128, 41
    op, ref, maps, img, traj = make_sense(n, C, R, S, seed=32)
    y = ref.sense_forward(maps, img)
    b = op.adjoint(y).reshape(1, n, n)
    x, st, tr = ba.lsqr_conjgrad(op, b, 100, 0.01, 1e-4)
    assert st.status == 2 and st.iterations < 100
    assert st.resid <= 1e-4 * st.bnorm * 1.0001
    # warm start from the solution converges immediately (pics -W)
    x2, st2, _ = ba.lsqr_conjgrad(op, b, 100, 0.01, 1e-4, x0=x.reshape(1, n, n))
    assert st2.iterations <= 2
    # 0 iterations return the warm start unchanged (tests/pics.mk:184-190)
    x3, st3, _ = ba.lsqr_conjgrad(op, b, 0, 0.01, 0.0, x0=x.reshape(1, n, n))
    assert np.array_equal(x3.reshape(-1), x.reshape(-1))
    # fallback: a bad warm start is replaced by zero
    bad = (1e3 * crandn((1, n, n), 33)).astype(np.complex64)
    x4, st4, _ = ba.lsqr_conjgrad(op, b, 100, 0.01, 1e-4, x0=bad, fallback=True)
    assert st4.fell_back and st4.status == 2
    assert np.array_equal(x4.reshape(-1), x.reshape(-1))


def test_cg_monitor_errors_of_the_iterates():
    # pics -T (iter/monitor.c): err[k] = ||truth - x_k|| / ||truth|| for the
    # iterate x_k that iteration k starts from (x_0 = 0: error 1); x_k is
    # the result of a solve stopped after k iterations; the monitor changes
    # no bit of the solve
    n, C, R, S = 64, 4, 128, 41
    op, ref, maps, img, traj = make_sense(n, C, R, S, seed=34)
    b = op.adjoint(ref.sense_forward(maps, img)).reshape(1, n, n)
    x_plain, st_plain, tr_plain = ba.lsqr_conjgrad(op, b, 12, 0.01, 0.0)
    mon = ba.CgMonitor(op, img, 12)
    x, st, tr = ba.lsqr_conjgrad(op, b, 12, 0.01, 0.0)
    err = mon.errors(st.iterations)
    assert np.array_equal(x, x_plain) and np.array_equal(tr, tr_plain)
    assert abs(err[0] - 1.0) < 1e-6
    for k in (1, 2, 5, 11):
        xk, _, _ = ba.lsqr_conjgrad(op, b, k, 0.01, 0.0)
        assert abs(err[k] / relerr(xk.reshape(1, n, n), img) - 1) < 1e-5
    assert err[11] < err[1]
    mon.close()
    x2, _, _ = ba.lsqr_conjgrad(op, b, 12, 0.01, 0.0)
    assert np.array_equal(x2, x_plain)


def test_device_pointers_with_torch():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("torch's bundled HIP runtime was initialised after this library's")
    n, C, R, S = 64, 2, 128, 21
    traj = I.radial_traj(R, S)
    op = make_nufft((n, n, 1), C, traj, R, S, toeplitz=True)
    ref = O.Nufft((n, n, 1), traj, C, toeplitz=True)
    x = crandn((C, 1, n, n), 41)
    xd = torch.from_numpy(x.reshape(-1)).to("cuda")
    k = op.forward(xd)
    assert k.is_cuda
    assert relerr(k.cpu().numpy().reshape(C, -1), ref.forward(x)) < 1e-5
    nn = op.normal(xd)
    assert relerr(nn.cpu().numpy().reshape(x.shape), ref.normal(x)) < 1e-5


def test_errors_are_reported():
    with pytest.raises(ba.BartError):
        ba.nufft_create2(dims16(1, 10, 1, 2), dims16(16, 16, 1, 3), dims16(3, 10, 1),
                         np.zeros(30, np.complex64))
    # the non-decomposed grid (nufft -1) and compressed PSF storage are not built
    with pytest.raises(ba.BartError):
        ba.nufft_create2(dims16(1, 10, 1, 1), dims16(16, 16, 1, 1), dims16(3, 10, 1),
                         np.zeros(30, np.complex64), conf=ba.NufftConf.defaults(decomp=False))
    with pytest.raises(ba.BartError):
        ba.nufft_create2(dims16(1, 10, 1, 1), dims16(16, 16, 1, 1), dims16(3, 10, 1),
                         np.zeros(30, np.complex64), conf=ba.NufftConf.defaults(compress_psf=True))
    # batch dims with and without trajectories of their own are not mixed
    with pytest.raises(ba.BartError):
        ba.nufft_create2(dims16(1, 10, 1, 1, 1, 2, 2), dims16(16, 16, 1, 1, 1, 2, 2), dims16(3, 10, 1, 1, 1, 2),
                         np.zeros(60, np.complex64))


@pytest.mark.parametrize("img,C,mode", [((64, 64, 1), 8, "lowmem"), ((64, 64, 1), 6, "zero_overhead"),
                                        ((32, 32, 32), 4, "lowmem"), ((64, 64, 64), 3, "zero_overhead")])
def test_low_memory_modes(img, C, mode):
    # --lowmem / --zero-mem (noncart/nufft.c:1629-2003): the plan holds a
    # chunk of coils (stack S c N <= C N, or S N) and is applied chunk by
    # chunk; NUFFT, SENSE and CG agree with the default mode to BART's
    # tolerance for these modes (tests/nufft.mk:366-400, nrmse 1e-6), and
    # the NUFFT of each coil is unchanged bit for bit
    X, Y, Z = img
    n = X
    if Z == 1:
        R, S = 2 * n, 33
        traj = I.radial_traj(R, S)
    else:
        R, S = 2 * n, 60
        traj = I.phyllotaxis_kooshball(spokes=S, readout=R)
    M = R * S
    kw = {mode: True}
    op0 = make_nufft(img, C, traj, R, S, toeplitz=True)
    op1 = make_nufft(img, C, traj, R, S, toeplitz=True, **kw)
    x = crandn((C, Z, Y, X), 61)
    y = crandn((C, M), 62)
    assert np.array_equal(op1.forward(x), op0.forward(x))
    assert relerr(op1.adjoint(y), op0.adjoint(y)) < 1e-6
    assert relerr(op1.normal(x), op0.normal(x)) < 1e-6
    maps = I.gaussian_coils((Z, Y, X), C, seed=63)
    conf0 = ba.NufftConf.defaults()
    conf1 = ba.NufftConf.defaults(**kw)
    s0 = ba.sense_nc_init(dims16(X, Y, Z, C), dims16(X, Y, Z, C), maps, dims16(1, R, S, C), dims16(3, R, S),
                          ba.traj_array(traj), conf=conf0)
    s1 = ba.sense_nc_init(dims16(X, Y, Z, C), dims16(X, Y, Z, C), maps, dims16(1, R, S, C), dims16(3, R, S),
                          ba.traj_array(traj), conf=conf1)
    im = crandn((Z, Y, X), 64)
    assert np.array_equal(s1.forward(im), s0.forward(im))
    b0, b1 = s0.adjoint(y), s1.adjoint(y)
    assert relerr(b1, b0) < 1e-6
    assert relerr(s1.normal(im), s0.normal(im)) < 1e-6
    x0, st0, tr0 = ba.lsqr_conjgrad(s0, b0, 5, 0.01, 0.0)
    x1, st1, tr1 = ba.lsqr_conjgrad(s1, b0, 5, 0.01, 0.0)
    assert st1.iterations == 5 and relerr(x1, x0) < 1e-5
    ref = O.Nufft(img, traj, C, toeplitz=True)
    assert relerr(s1.normal(im).reshape(Z, Y, X), ref.sense_normal(maps, im)) < 1e-5
    for o in (op0, op1, s0, s1):
        o.free()


@pytest.mark.parametrize("img,C", [((64, 64, 1), 2), ((32, 32, 32), 2)])
def test_strang_preconditioner_and_preconditioned_cg(img, C):
    # nufft_precond_create (noncart/precond.c:46-164) against the oracle's
    # complex128 restatement; lsqr with the preconditioner (iter/lsqr.c:126-142):
    # CG on P (A^H A + lambda I) x = P b, against complex128 CG on the
    # oracle's operator and preconditioner
    X, Y, Z = img
    n = X
    if Z == 1:
        R, S = 2 * n, 41
        traj = I.radial_traj(R, S)
    else:
        R, S = 2 * n, 80
        traj = I.phyllotaxis_kooshball(spokes=S, readout=R)
    op = make_nufft(img, C, traj, R, S, toeplitz=True)
    ref = O.Nufft(img, traj, C, toeplitz=True)
    pre = ba.Precond(op)
    _, apply_o = O.precond_strang(ref)
    x = crandn((C, Z, Y, X), 81)
    assert relerr(pre.apply(x).reshape(C, Z, Y, X), apply_o(x)) < 1e-5
    y = crandn((C, R * S), 82)
    b = op.adjoint(y).reshape(C, Z, Y, X)
    lam = 0.01
    xg, st, trg = ba.lsqr_conjgrad_precond(op, pre, b, 5, lam, 0.0)
    pn = lambda v: apply_o(ref.normal_fp64(v) + lam * np.asarray(v, np.complex128).reshape(C, Z, Y, X))
    x64, tr64 = O.cg_fp64(pn, apply_o(b), 0.0, 5)
    assert st.iterations == 5
    assert float(np.max(np.abs(trg / tr64 - 1))) < 1e-4
    assert relerr(xg.reshape(x64.shape), x64) < 1e-4
    pre.free()
    op.free()


def test_real_psf():
    # --nufft-conf real-psf (noncart/nufft.c:1128-1137): the PSF keeps its
    # real part; the Toeplitz operator multiplies by it (against the oracle
    # with the same real PSF)
    n, C, R, S = 64, 2, 128, 41
    traj = I.radial_traj(R, S)
    op0 = make_nufft((n, n, 1), C, traj, R, S, toeplitz=True)
    op1 = make_nufft((n, n, 1), C, traj, R, S, toeplitz=True, real=True)
    p0, p1 = op0.get_psf(), op1.get_psf()
    assert np.all(p1.imag == 0) and np.array_equal(p1.real, p0.real)
    ref = O.Nufft((n, n, 1), traj, C, toeplitz=True)
    ref.set_psf(ref.psf().real.astype(np.complex64))
    x = crandn((C, 1, n, n), 91)
    assert relerr(op1.normal(x).reshape(C, 1, n, n), ref.normal(x)) < 1e-5
    op0.free()
    op1.free()
