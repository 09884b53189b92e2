"""The work that users of this library have it do, as measurable cases.

Non-Cartesian MRI reconstruction: the NUFFT and its adjoint (with and without
coil maps), CG-SENSE solves (single, batched over slices, 2-D and 3-D), the
subspace operators and the layers of the warm-start network.  `listed` holds
named cases from the smallest call to the largest, `draw` gives more of the
same ranges.  `prepare` makes what a program holds before the call (operator
handle and data on the GPU), `run` is one pass through the public entry
points, `exact` the same outputs from plain torch in 64 bits.
"""
import math

import numpy as np
import torch

import bart_amd as ba

DEV = "cuda"


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------

def _nufft(name, direction, nx, ny, nz, coils, spokes, readout, traj="radial", maps=False, weights=False):
    c = dict(kind="nufft", direction=direction, nx=nx, ny=ny, nz=nz, coils=coils, spokes=spokes, readout=readout,
             traj=traj, maps=maps, weights=weights)
    return dict(name=name, **c) if name else c


def _cg(name, nx, ny, nz, coils, spokes, readout, iters, traj="radial"):
    c = dict(kind="cg", nx=nx, ny=ny, nz=nz, coils=coils, spokes=spokes, readout=readout, traj=traj,
             iters=iters, lam=0.01)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one frame of a real-time series or a coil-compressed scout: the
        # smallest call, where latency and launches count
        _nufft("fwd_2d_64_c4", "forward", 64, 64, 1, 4, 31, 128),
        # density-compensated gridding reconstruction of a 2-D radial scan
        # with coil maps
        _nufft("adj_2d_256_c8", "adjoint", 256, 256, 1, 8, 201, 512, maps=True, weights=True),
        # the forward model of a 2-D variable-density spiral, 32 coils
        _nufft("fwd_2d_spiral_320_c32", "forward", 320, 320, 1, 32, 24, 4096, traj="spiral"),
        # a rectangular field of view with sizes off the powers of two, an odd
        # coil and spoke count and an odd readout
        _nufft("adj_2d_210x176_c7", "adjoint", 210, 176, 1, 7, 89, 419),
        # 3-D kooshball: both directions of the NUFFT, the largest single call
        _nufft("adj_3d_128_c16", "adjoint", 128, 128, 128, 16, 8192, 256, traj="koosh"),
        _nufft("fwd_3d_128_c16", "forward", 128, 128, 128, 16, 8192, 256, traj="koosh"),
        # CG-SENSE of one 2-D radial slice, 30 iterations (the default count).
        # The solves weight the samples by their density, as reconstructions
        # of radial data do: unweighted, the thousandfold density of the
        # k-space centre makes CG carry single-precision roundings up to 1 %
        _cg("cg_2d_256_c8", 256, 256, 1, 8, 201, 512, 30),
        # CG-SENSE of a 3-D volume with unequal sides, few iterations
        _cg("cg_3d_96x80x60_c6", 96, 80, 60, 6, 1500, 192, 8, traj="koosh"),
        # CG-SENSE of the 3-D kooshball: the largest solve
        _cg("cg_3d_128_c16", 128, 128, 128, 16, 8192, 256, 20, traj="koosh"),
        # slices of a study, uneven in size, coils and spokes, solved together
        dict(name="cg_batch_24_slices", kind="batch", slices=24, nmin=128, nmax=384, cmin=8, cmax=32, spokesmin=21,
             spokesmax=201, iters=30, lam=0.01, geometry=4),
        # subspace reconstruction of a dynamic scan: adjoint and normal
        # operator on the coefficient images
        dict(name="basis_256_c8_t64_k4", kind="basis", n=256, coils=8, frames=64, spokes=4, readout=512, rank=4),
        # one layer of the warm-start network in training, forward and both
        # gradients
        dict(name="conv_48_256_b8", kind="conv", batch=8, cin=48, cout=48, height=256, width=256),
    ]


def _smooth(n):
    """The nearest size at or below n whose prime factors the FFT takes."""
    while True:
        m = n
        for p in (2, 3, 5, 7, 11, 13):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n -= 1


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size2(rng):
    """A 2-D matrix: half of them square powers-of-two-ish sizes as scanners
    reconstruct them, half any supported size and rectangular."""
    if rng.random() < 0.5:
        n = rng.choice([64, 128, 192, 256, 320, 384])
        return n, n
    n = _smooth(_logint(rng, 40, 400))
    return n, _smooth(max(24, int(n * rng.uniform(0.6, 1.0))))


def _size3(rng):
    if rng.random() < 0.4:
        n = rng.choice([32, 64, 96, 128])
        return n, n, n
    n = _smooth(_logint(rng, 24, 120))
    return tuple(_smooth(max(20, int(n * rng.uniform(0.6, 1.0)))) for _ in range(3))


def _draw_nufft(rng):
    if rng.random() < 0.6:
        nx, ny = _size2(rng)
        nm = max(nx, ny)
        traj = rng.choice(["radial", "radial", "spiral"])
        spokes = _logint(rng, 8, 40) if traj == "spiral" else _logint(rng, 13, 401)
        readout = _logint(rng, 1000, 4096) if traj == "spiral" else int(nm * rng.uniform(1.2, 2.0))
        return _nufft("", rng.choice(["forward", "adjoint"]), nx, ny, 1, _logint(rng, 1, 32), spokes, readout,
                      traj=traj, maps=rng.random() < 0.5, weights=rng.random() < 0.3)
    nx, ny, nz = _size3(rng)
    nm = max(nx, ny, nz)
    return _nufft("", rng.choice(["forward", "adjoint"]), nx, ny, nz, _logint(rng, 1, 16), _logint(rng, 200, min(6000, max(300, nm * nm // 2))),
                  int(nm * rng.uniform(1.2, 2.0)), traj="koosh", maps=rng.random() < 0.5,
                  weights=rng.random() < 0.3)


def _draw_cg(rng):
    # small images are solved in few iterations: beyond convergence CG only
    # amplifies roundings
    if rng.random() < 0.6:
        nx, ny = _size2(rng)
        n = max(nx, ny)
        return _cg("", nx, ny, 1, _logint(rng, 2, 32), _logint(rng, 21, max(40, min(301, n))),
                   int(n * rng.uniform(1.4, 2.0)), rng.randint(4, max(5, min(30, n // 10))))
    nx, ny, nz = _size3(rng)
    n = max(nx, ny, nz)
    return _cg("", nx, ny, nz, _logint(rng, 2, 12), _logint(rng, 300, min(5000, max(400, n * n // 2))),
               int(n * rng.uniform(1.4, 2.0)), rng.randint(3, 6), traj="koosh")


def draw(rng):
    u = rng.random()
    if u < 0.4:
        return _draw_nufft(rng)
    if u < 0.7:
        return _draw_cg(rng)
    if u < 0.8:
        nmin = rng.choice([64, 96, 128, 192])
        return dict(kind="batch", slices=rng.randint(2, 24), nmin=nmin, nmax=rng.choice([256, 320, 384]),
                    cmin=rng.randint(2, 8), cmax=rng.randint(8, 24), spokesmin=21, spokesmax=rng.randint(60, 128),
                    iters=rng.randint(5, max(6, nmin // 10)), lam=0.01, geometry=rng.randint(0, 1 << 20))
    if u < 0.9:
        n = _smooth(_logint(rng, 48, 300))
        return dict(kind="basis", n=n, coils=rng.randint(2, 12), frames=rng.randint(8, 64), spokes=rng.randint(1, 5),
                    readout=int(n * rng.uniform(1.4, 2.0)), rank=rng.randint(2, 6))
    # widths in multiples of 8, as the weight gradient takes them
    return dict(kind="conv", batch=rng.randint(1, 8), cin=rng.choice([2, 16, 32, 48, 48]),
                cout=rng.choice([2, 16, 32, 48, 48]), height=_logint(rng, 24, 256),
                width=8 * rng.randint(3, 32))


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

def _rng(seed, salt=0):
    return np.random.default_rng((int(seed) & 0xFFFFFFFF) * 1000003 + salt)


def _trajectory(kind, dims, spokes, readout, seed):
    """[M, 3] float32 coordinates; golden-angle radial, variable-density
    spiral or 3-D kooshball, turned by an angle of the seed and stretched to
    the field of view of each dim."""
    r = _rng(seed, 1)
    turn = r.uniform(0.0, 2.0 * np.pi)
    if kind == "spiral":
        t = (np.arange(readout) + 0.5) / readout
        rad = 0.5 / 8.0 * np.expm1(math.log(9.0) * t)
        turns = max(dims) / (2.0 * spokes) * 1.5
        th = 2.0 * np.pi * (turns * t[None, :] + np.arange(spokes)[:, None] / spokes) + turn
        k = np.stack([rad * np.cos(th), rad * np.sin(th), np.zeros_like(th)], -1) * (1.0 - 2.0 / max(dims))
    else:
        read = (np.arange(readout) + 0.5 - readout / 2.0) / readout
        j = np.arange(spokes)
        if kind == "koosh":
            phi = 2.0 * np.pi * j / (((1.0 + math.sqrt(5.0)) / 2.0) ** 2) + turn
            theta = 0.5 * np.pi * np.sqrt(j / spokes)
            d = np.stack([np.sin(theta) * np.cos(phi), np.sin(theta) * np.sin(phi), np.cos(theta)], -1)
        else:
            a = j * np.pi * (math.sqrt(5.0) - 1.0) / 2.0 + turn
            d = np.stack([np.sin(a), np.cos(a), np.zeros_like(a)], -1)
        k = read[None, :, None] * d[:, None, :]
    return np.ascontiguousarray(k.reshape(-1, 3) * np.asarray(dims, np.float64)[None, :]).astype(np.float32)


def _grid(dims):
    """Pixel coordinates of the field of view [-1, 1]^d, [z, y, x] each."""
    ax = [(torch.arange(n, device=DEV, dtype=torch.float32) - n // 2) * (2.0 / n) if n > 1
          else torch.zeros(1, device=DEV) for n in dims]
    return ax[0].view(1, 1, -1), ax[1].view(1, -1, 1), ax[2].view(-1, 1, 1)


def _image(dims, seed):
    """Ellipses (ellipsoids) of random intensity times a smooth phase."""
    r = _rng(seed, 2)
    x, y, z = _grid(dims)
    img = torch.zeros(dims[2], dims[1], dims[0], device=DEV)
    for _ in range(10):
        c = r.uniform(-0.5, 0.5, 3)
        a = r.uniform(0.08, 0.45, 3)
        inside = ((x - c[0]) / a[0]) ** 2 + ((y - c[1]) / a[1]) ** 2
        if dims[2] > 1:
            inside = inside + ((z - c[2]) / a[2]) ** 2
        img += float(r.uniform(0.1, 1.0)) * (inside <= 1.0)
    p = r.uniform(-1.5, 1.5, 4)
    ph = p[0] * x + p[1] * y + p[2] * z + p[3] * (x * x - y * y)
    return torch.polar(img, ph.expand_as(img).contiguous()).contiguous()


def _coil_centres(C, nd):
    if nd == 2:
        a = 2.0 * np.pi * np.arange(C) / C
        return np.stack([0.6 * np.cos(a), 0.6 * np.sin(a), np.zeros(C)], -1)
    h = -1.0 + (2.0 * np.arange(C) + 1.0) / C
    a = 2.0 * np.pi * np.arange(C) / ((1.0 + math.sqrt(5.0)) / 2.0)
    s = np.sqrt(np.maximum(0.0, 1.0 - h * h))
    return 0.6 * np.stack([s * np.cos(a), s * np.sin(a), h], -1)


def _coil_values(C, nd, seed, x, y, z):
    """Gaussian coil sensitivities with a smooth phase, root sum of squares 1."""
    r = _rng(seed, 3)
    cen = _coil_centres(C, nd)
    m = []
    for c in range(C):
        q = r.uniform(-1.0, 1.0, 2)
        q2 = r.uniform(0.0, 2.0 * np.pi)
        d2 = (x - cen[c, 0]) ** 2 + (y - cen[c, 1]) ** 2 + (z - cen[c, 2]) ** 2
        mag = torch.exp(-d2 / (2.0 * 0.7 ** 2))
        m.append(torch.polar(mag, (q[0] * x + q[1] * y + q2).expand_as(mag).contiguous()))
    m = torch.stack(m)
    return m / m.abs().square().sum(0, keepdim=True).sqrt()


def _maps(dims, C, seed):
    x, y, z = _grid(dims)
    return _coil_values(C, 2 if dims[2] == 1 else 3, seed, x, y, z).to(torch.complex64).contiguous()


def _kspace(traj, dims, C, seed, frames=1):
    """k-space [C, M] (or [frames, C, M / frames]) of a sum of Gaussian blobs
    seen by the coils, with noise: the decay of real data, from the closed
    form (no operator is involved)."""
    r = _rng(seed, 4)
    nd = 2 if dims[2] == 1 else 3
    J = 6
    pos = torch.from_numpy(r.uniform(-0.6, 0.6, (J, 3))).float().to(DEV)
    if nd == 2:
        pos[:, 2] = 0.0
    amp = r.uniform(0.3, 1.0, J) * np.exp(1j * r.uniform(0, 2 * np.pi, J))
    sig = torch.from_numpy(r.uniform(0.03, 0.2, J)).float().to(DEV)
    sens = _coil_values(C, nd, seed, pos[:, 0].contiguous(), pos[:, 1].contiguous(), pos[:, 2].contiguous())
    a = (sens * torch.from_numpy(amp).to(DEV).to(torch.complex64)[None]).contiguous()  # [C, J]
    k = torch.from_numpy(traj).to(DEV)
    M = k.shape[0]
    y = torch.zeros(C, M, dtype=torch.complex64, device=DEV)
    scale = math.sqrt(float(np.prod(dims)))
    for j in range(J):
        # blob exp(-|x|^2 / 2 sig^2) in field-of-view units [-1, 1]
        ph = torch.zeros(M, device=DEV)
        q2 = torch.zeros(M, device=DEV)
        for d in range(nd):
            ph += k[:, d] * (pos[j, d] * 0.5)
            q2 += (k[:, d] * (math.pi * sig[j])) ** 2
        ph = (ph - ph.floor()) * (-2.0 * math.pi)
        e = torch.polar(torch.exp(-0.5 * q2) * (scale * float(sig[j]) ** nd), ph)
        y += a[:, j, None] * e[None]
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) + 17)
    s = 1e-3 * float(y.abs().max()) / math.sqrt(2.0)
    y += s * torch.randn(C, M, dtype=torch.complex64, device=DEV, generator=g)
    if frames > 1:
        y = y.view(C, frames, M // frames).transpose(0, 1)
    return y.contiguous()


def _weights(traj, dims):
    """Square root of the density compensation of radial samples (a ramp in
    2-D, its square in 3-D), as reconstructions weight them."""
    q = 2.0 * np.sqrt(np.sum((traj / np.asarray(dims, np.float32)[None, :]) ** 2, -1)) + 1.0 / max(dims)
    return (np.sqrt(q) if dims[2] == 1 else q).astype(np.complex64)


def _d16(*d):
    return list(d) + [1] * (16 - len(d))


def _sense_op(dims, C, spokes, readout, traj, maps, weights):
    return ba.sense_nc_init(_d16(*dims, C), _d16(*dims, C), maps, _d16(1, readout, spokes, C),
                            _d16(3, readout, spokes), ba.traj_array(traj), weights=weights)


def _slices(case):
    """The slices of a batch case: square matrices of the sizes that scanners
    reconstruct, uneven coils and spokes.  The geometry is the case's own,
    the contents are the seed's."""
    r = _rng(case["geometry"], 5)
    sizes = [n for n in (64, 96, 128, 160, 192, 256, 320, 384) if case["nmin"] <= n <= case["nmax"]]
    out = []
    for _ in range(case["slices"]):
        n = int(r.choice(sizes))
        out.append((n, int(r.integers(case["cmin"], case["cmax"] + 1)),
                    int(r.integers(case["spokesmin"], case["spokesmax"] + 1))))
    return out


def _basis(case, seed):
    r = _rng(seed, 6)
    T, K = case["frames"], case["rank"]
    t = np.arange(T) / T
    decay = np.exp(-np.outer(t, r.uniform(0.2, 6.0, 3 * K))) * np.exp(1j * np.outer(t, r.uniform(-1, 1, 3 * K)))
    q, _ = np.linalg.qr(decay)
    return np.ascontiguousarray(q[:, :K]).astype(np.complex64)  # [T, K]


def _conv_inputs(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    B, ci, co, H, W = (case[k] for k in ("batch", "cin", "cout", "height", "width"))
    x = torch.relu(torch.randn(B, ci, H, W, device=DEV, generator=g)) * 0.2
    w = torch.randn(co, ci, 3, 3, device=DEV, generator=g) * math.sqrt(2.0 / (9 * ci))
    b = torch.randn(co, device=DEV, generator=g) * 0.01
    dy = torch.randn(B, co, H, W, device=DEV, generator=g) * 1e-3
    return x, w, b, dy


def _dims(case):
    return (case["nx"], case["ny"], case["nz"])


# --------------------------------------------------------------------------
# prepare, run
# --------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "conv":
        x, w, b, dy = _conv_inputs(case, seed)
        return dict(kind=kind, x=x, w=w, b=b, dy=dy)

    if kind == "batch":
        ops, ys = [], []
        for i, (n, C, spokes) in enumerate(_slices(case)):
            dims = (n, n, 1)
            s = int(seed) * 64 + i
            traj = _trajectory("radial", dims, spokes, 2 * n, s)
            ops.append(_sense_op(dims, C, spokes, 2 * n, traj, _maps(dims, C, s), _weights(traj, dims)))
            ys.append(_kspace(traj, dims, C, s).view(-1))
        return dict(kind=kind, ops=ops, ys=ys, iters=case["iters"], lam=case["lam"])

    if kind == "basis":
        n, C, T, K = case["n"], case["coils"], case["frames"], case["rank"]
        dims = (n, n, 1)
        Mf = case["spokes"] * case["readout"]
        traj = _trajectory("radial", dims, T * case["spokes"], case["readout"], seed)
        bas = np.ascontiguousarray(_basis(case, seed).T)
        op = ba.sense_nc_init(_d16(n, n, 1, C, 1, 1, K), _d16(n, n, 1, C), _maps(dims, C, seed),
                              _d16(1, Mf, 1, C, 1, T), _d16(3, Mf, 1, 1, 1, T),
                              np.ascontiguousarray(traj.reshape(T, Mf, 3).astype(np.complex64)),
                              basis_dims=_d16(1, 1, 1, 1, 1, T, K), basis=bas)
        return dict(kind=kind, op=op, y=_kspace(traj, dims, C, seed, frames=T).view(-1))

    dims = _dims(case)
    C, spokes, R = case["coils"], case["spokes"], case["readout"]
    traj = _trajectory(case["traj"], dims, spokes, R, seed)

    if kind == "cg":
        op = _sense_op(dims, C, spokes, R, traj, _maps(dims, C, seed), _weights(traj, dims))
        return dict(kind=kind, op=op, y=_kspace(traj, dims, C, seed).view(-1), iters=case["iters"], lam=case["lam"])

    w = _weights(traj, dims) if case["weights"] else None
    maps = _maps(dims, C, seed) if case["maps"] else None
    conf = ba.NufftConf.defaults(toeplitz=False)
    if maps is not None:
        op = ba.sense_nc_init(_d16(*dims, C), _d16(*dims, C), maps, _d16(1, R, spokes, C), _d16(3, R, spokes),
                              ba.traj_array(traj), conf=conf, weights=w)
    else:
        op = ba.nufft_create2(_d16(1, R, spokes, C), _d16(*dims, C), _d16(3, R, spokes), ba.traj_array(traj),
                              weights=w, conf=conf)
    if case["direction"] == "forward":
        img = _image(dims, seed)
        src = img if maps is not None else (img[None] * _maps(dims, C, seed)).contiguous()
    else:
        src = _kspace(traj, dims, C, seed)
    return dict(kind=kind, op=op, direction=case["direction"], src=src.view(-1))


def run(state):
    kind = state["kind"]
    if kind == "nufft":
        op = state["op"]
        return op.forward(state["src"]) if state["direction"] == "forward" else op.adjoint(state["src"])
    if kind == "cg":
        b = state["op"].adjoint(state["y"])
        x, _, _ = ba.lsqr_conjgrad(state["op"], b, state["iters"], state["lam"], 0.0)
        return dict(adjoint=b, x=x)
    if kind == "batch":
        bs = [op.adjoint(y) for op, y in zip(state["ops"], state["ys"])]
        xs, _, _ = ba.lsqr_conjgrad_batch(state["ops"], bs, state["iters"], state["lam"], 0.0)
        return dict(adjoint=bs, x=xs)
    if kind == "basis":
        b = state["op"].adjoint(state["y"])
        return dict(adjoint=b, normal=state["op"].normal(b))
    y = ba.conv3x3(state["x"], state["w"], state["b"], relu=True)
    dx = ba.conv3x3_bwd_data(state["dy"], state["w"])
    dw, db = ba.conv3x3_bwd_weights(state["x"], state["dy"])
    return dict(y=y, dx=dx, dw=dw, db=db)


# --------------------------------------------------------------------------
# work, tolerance
# --------------------------------------------------------------------------

def _shape_work(dims, C, M, maps, weights):
    N = dims[0] * dims[1] * dims[2]
    d = sum(1 for n in dims if n > 1)
    b = 8 * C * M + 4 * d * M + (8 * M if weights else 0) + (8 * C * N + 8 * N if maps else 8 * C * N)
    S = 1 << d
    f = S * C * 5.0 * N * math.log2(N) + 4.0 * C * M * 6 ** d
    return b, f


def _cg_work(dims, C, M, iters):
    N = dims[0] * dims[1] * dims[2]
    S = 1 << sum(1 for n in dims if n > 1)
    b, f = _shape_work(dims, C, M, True, True)
    return b + iters * 8 * N * (9 + C + S), f + iters * (2 * S * C * 5.0 * N * math.log2(N) + 30.0 * S * C * N)


def work(case):
    kind = case["kind"]
    if kind == "conv":
        B, ci, co, H, W = (case[k] for k in ("batch", "cin", "cout", "height", "width"))
        px = B * H * W
        return dict(bytes=4 * (px * 2 * (ci + co) + 3 * 9 * ci * co), flops=3 * 2.0 * 9 * ci * co * px)
    if kind == "batch":
        t = [_cg_work((n, n, 1), C, 2 * n * sp, case["iters"]) for n, C, sp in _slices(case)]
        return dict(bytes=sum(b for b, _ in t), flops=sum(f for _, f in t))
    if kind == "basis":
        n, C, K = case["n"], case["coils"], case["rank"]
        N, M = n * n, case["frames"] * case["spokes"] * case["readout"]
        fft = 4 * C * K * 5.0 * N * math.log2(N)
        b = 8 * C * M + 8 * M + 2 * 8 * C * N + 3 * 8 * K * N + 8 * K * K * 4 * N
        return dict(bytes=b, flops=3 * fft + 8.0 * C * K * M + 4.0 * C * K * M * 36 + 8.0 * 4 * C * K * K * N)
    dims, C = _dims(case), case["coils"]
    M = case["spokes"] * case["readout"]
    if kind == "cg":
        b, f = _cg_work(dims, C, M, case["iters"])
    else:
        b, f = _shape_work(dims, C, M, case["maps"], case["weights"])
    return dict(bytes=b, flops=f)


def tolerance(case):
    kind = case["kind"]
    if kind == "nufft":
        # 32-bit sums over up to tens of thousands of samples per grid point;
        # measured against 64 bits: up to 8e-7, largest difference 3e-6
        return dict(rel=4e-6, max=4e-5)
    if kind == "basis":
        # measured: 7e-7, largest 2e-6
        return dict(rel=4e-6, max=4e-5)
    if kind == "conv":
        # bf16 operands as the entry points state, 32-bit sums over up to
        # half a million pixels; measured: 1e-6, largest 2.5e-6
        return dict(rel=4e-6, max=2e-5)
    # CG carries a rounding of one iteration through all that follow;
    # measured: up to 2e-5, largest 1.9e-4
    return dict(rel=1e-4, max=1e-3)


# --------------------------------------------------------------------------
# The same outputs in 64 bits: the decomposed 2x oversampled Kaiser-Bessel
# NUFFT (width 6, 1001-entry table with linear interpolation, sample
# positions rounded to float32), DFTs as matrices per axis
# --------------------------------------------------------------------------

_C128 = torch.complex128
_BETA = float(np.float32(math.pi * math.sqrt((6.0 / 2.0 * 1.5) ** 2 - 0.8)))


def _kb_table():
    x = np.arange(1001) / 999.0 / 2.0
    t = np.zeros(1001)
    m = x < 0.5
    t[m] = np.i0(_BETA * np.sqrt(1.0 - (2.0 * x[m]) ** 2)) / np.i0(_BETA)
    return torch.from_numpy(t.astype(np.float32).astype(np.float64)).to(DEV)


def _taps(k, n, table, periodic):
    """Indices [M, 8] into the 2 n points (sub-grid s at s n) and weights."""
    M = k.shape[0]
    if n == 1:
        return torch.zeros(M, 1, dtype=torch.long, device=DEV), torch.ones(M, 1, dtype=torch.float64, device=DEV)
    idx, wts = [], []
    for s in range(2):
        shift = float(np.float32(-0.5 * s + (n / 2.0 - n // 2)))
        pos = ((k.double() + shift).float() + np.float32(n // 2)).double()
        lo, hi = torch.ceil(pos - 1.5), torch.floor(pos + 1.5)
        for j in range(4):
            g = lo + j
            ok = g <= hi
            x = 2.0 * (g - pos).abs() / 3.0 * 999.0
            i = x.floor().clamp(0, 999).long()
            f = x - i
            w = (1.0 - f) * table[i] + f * table[(i + 1).clamp(max=1000)]
            gi = g.long()
            if periodic:
                gi = gi % n
            else:
                ok = ok & (gi >= 0) & (gi < n)
                gi = gi.clamp(0, n - 1)
            idx.append(gi + s * n)
            wts.append(torch.where(ok, w, torch.zeros_like(w)))
    return torch.stack(idx, 1), torch.stack(wts, 1)


def _fftmod(n):
    j = torch.arange(n, dtype=torch.float64, device=DEV)
    c = n // 2
    return torch.exp(2j * math.pi * ((j - c / 2.0) * c / n))


def _lin(n, s):
    """Linear phase of sub-grid s with fftmod and the unitary scale."""
    j = torch.arange(n, dtype=torch.float64, device=DEV)
    grad = 2.0 * math.pi * (-0.5 * s + (n / 2.0 - n // 2)) / n
    return torch.exp(1j * grad * (j - n / 2.0)) * _fftmod(n) / math.sqrt(n)


def _rolloff(n):
    i = torch.arange(n, dtype=torch.float64, device=DEV)
    x = ((i - n // 2) / (2 * n)).float().double()
    a = _BETA ** 2 - (math.pi * x * 6.0) ** 2
    q = a.abs().sqrt()
    f = torch.where(a > 0, torch.sinh(q) / q, torch.sin(q) / q) / float(np.i0(_BETA))
    return 1.0 / f / 6.0


def _axis_matrix(n):
    """[2 n, n]: image axis -> the points of both sub-grids."""
    if n == 1:
        return torch.ones(1, 1, dtype=_C128, device=DEV)
    j = torch.arange(n, device=DEV)
    dft = torch.exp(-2j * math.pi * ((j[:, None] * j[None, :]) % n).double() / n)
    rows = [_fftmod(n)[:, None] * dft * (_lin(n, s) * _rolloff(n))[None, :] for s in range(2)]
    return torch.cat(rows, 0).contiguous()


def _along(a, m, axis):
    """m applied along `axis` of a (2-D products of contiguous operands)."""
    a = a.movedim(axis, 0)
    shape = a.shape
    out = torch.mm(m, a.reshape(shape[0], -1).contiguous())
    return out.view(m.shape[0], *shape[1:]).movedim(0, axis)


class _Nufft64:
    def __init__(self, dims, traj, weights=None, periodic=False):
        self.dims = dims
        k = torch.from_numpy(traj).to(DEV)
        table = _kb_table()
        self.t = [_taps(k[:, d].contiguous(), dims[d], table, periodic) for d in range(3)]
        self.e = [_axis_matrix(n) for n in dims]
        self.g = [m.shape[0] for m in self.e]
        self.M = k.shape[0]
        self.w = None if weights is None else torch.from_numpy(np.ascontiguousarray(weights)).to(DEV).to(_C128)

    def _each(self):
        (i0, w0), (i1, w1), (i2, w2) = self.t
        for z in range(i2.shape[1]):
            for y in range(i1.shape[1]):
                wzy = w2[:, z] * w1[:, y]
                row = (i2[:, z] * self.g[1] + i1[:, y]) * self.g[0]
                for x in range(i0.shape[1]):
                    yield row + i0[:, x], wzy * w0[:, x]

    def forward(self, cim):
        """[C, z, y, x] -> [C, M]"""
        a = cim.to(_C128)
        for d in range(3):
            a = _along(a, self.e[d], 3 - d)
        C = a.shape[0]
        a = torch.view_as_real(a.reshape(C, -1).t().contiguous()).view(-1, 2 * C)
        out = torch.zeros(self.M, 2 * C, dtype=torch.float64, device=DEV)
        for i, w in self._each():
            out += a.index_select(0, i) * w[:, None]
        out = torch.view_as_complex(out.view(self.M, C, 2)).t()
        return out * self.w[None] if self.w is not None else out

    def adjoint(self, ksp):
        """[C, M] (complex, or real where the values are) -> [C, z, y, x]"""
        C = ksp.shape[0]
        if ksp.is_complex():
            v = ksp.to(_C128)
            if self.w is not None:
                v = v * self.w.conj()[None]
            v = torch.view_as_real(v.t().contiguous()).view(self.M, 2 * C)
        else:
            v = ksp.double().t().contiguous()
        a = torch.zeros(self.g[0] * self.g[1] * self.g[2], v.shape[1], dtype=torch.float64, device=DEV)
        for i, w in self._each():
            a.index_add_(0, i, v * w[:, None])
        a = torch.view_as_complex(a.view(-1, C, 2)) if ksp.is_complex() else a.to(_C128)
        a = a.t().reshape(C, self.g[2], self.g[1], self.g[0])
        for d in range(3):
            a = _along(a, self.e[d].conj().t().contiguous(), 3 - d)
        return a


class _Toeplitz64:
    """The Toeplitz normal operator: psf [P, S, z, y, x] of P k-space weightings."""

    def __init__(self, dims, traj, vals):
        self.dims = dims
        n2 = tuple(2 * n if n > 1 else 1 for n in dims)
        psf = _Nufft64(n2, traj * np.float32(2.0), periodic=True).adjoint(vals)
        for d in range(3):
            if n2[d] > 1:
                shape = [1, 1, 1, 1]
                shape[3 - d] = n2[d]
                fm = _fftmod(n2[d]).view(shape)
                psf = torch.fft.fft(psf * fm, dim=3 - d) * fm / math.sqrt(n2[d])
        self.lin, self.psf = [], []
        act = [d for d in range(3) if dims[d] > 1]
        self.axes = [3 - d for d in act]
        for s in range(1 << len(act)):
            bit = {d: (s >> b) & 1 for b, d in enumerate(act)}
            p, l = psf, torch.ones(1, 1, 1, 1, dtype=_C128, device=DEV)
            for d in act:
                p = p.index_select(3 - d, torch.arange(bit[d], n2[d], 2, device=DEV))
                shape = [1, 1, 1, 1]
                shape[3 - d] = dims[d]
                l = l * _lin(dims[d], bit[d]).view(shape)
            self.psf.append(p)
            self.lin.append(l)

    def normal(self, x, mix=None):
        """x [C, z, y, x]; mix: the product of the PSF and the transform"""
        N = x.shape[1] * x.shape[2] * x.shape[3]
        out = torch.zeros_like(x)
        for p, l in zip(self.psf, self.lin):
            f = torch.fft.fftn(x * l, dim=self.axes)
            f = f * p if mix is None else mix(p, f)
            out += torch.fft.ifftn(f, dim=self.axes) * (N * l.conj())
        return out


def _cg64(normal, b, iters, lam):
    x, r, p = torch.zeros_like(b), b.clone(), b.clone()
    rs = float(torch.linalg.vector_norm(r)) ** 2
    for _ in range(iters):
        ap = normal(p) + lam * p
        alpha = rs / float(torch.sum(p.conj() * ap).real)
        x += alpha * p
        r -= alpha * ap
        new = float(torch.linalg.vector_norm(r)) ** 2
        p = r + (new / rs) * p
        rs = new
    return x


def _cg_case64(dims, C, spokes, readout, kind, seed, iters, lam):
    traj = _trajectory(kind, dims, spokes, readout, seed)
    w = _weights(traj, dims)
    maps = _maps(dims, C, seed).to(_C128)
    b = (_Nufft64(dims, traj, w).adjoint(_kspace(traj, dims, C, seed)) * maps.conj()).sum(0)
    vals = torch.from_numpy(w).to(DEV).to(_C128).abs().square()[None]
    t = _Toeplitz64(dims, traj, vals)
    x = _cg64(lambda p: (t.normal(p[None] * maps) * maps.conj()).sum(0), b, iters, lam)
    return b.reshape(-1), x.reshape(-1)


def _conv64(x, w):
    """zero-padded 3 x 3 cross-correlation as nine matrix products"""
    B, ci, H, W = x.shape
    xp = torch.nn.functional.pad(x, (1, 1, 1, 1))
    out = torch.zeros(w.shape[0], B * H * W, dtype=torch.float64, device=DEV)
    for u in range(3):
        for v in range(3):
            s = xp[:, :, u:u + H, v:v + W].transpose(0, 1).reshape(ci, -1).contiguous()
            out += torch.mm(w[:, :, u, v].contiguous(), s)
    return out.view(-1, B, H, W).transpose(0, 1).contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind == "conv":
        x, w, b, dy = _conv_inputs(case, seed)
        xr, wr, dr = (t.to(torch.bfloat16).double() for t in (x, w, dy))
        y = torch.relu(_conv64(xr, wr) + b.double()[None, :, None, None])
        dx = _conv64(dr, wr.flip(2, 3).transpose(0, 1).contiguous())
        B, ci, H, W = x.shape
        xp = torch.nn.functional.pad(xr, (1, 1, 1, 1))
        dt = dr.transpose(0, 1).reshape(w.shape[0], -1).contiguous()
        dw = torch.zeros(w.shape, dtype=torch.float64, device=DEV)
        for u in range(3):
            for v in range(3):
                s = xp[:, :, u:u + H, v:v + W].permute(0, 2, 3, 1).reshape(-1, ci).contiguous()
                dw[:, :, u, v] = torch.mm(dt, s)
        return dict(y=y, dx=dx, dw=dw, db=dy.double().sum((0, 2, 3)))

    if kind == "batch":
        out = [_cg_case64((n, n, 1), C, spokes, 2 * n, "radial", int(seed) * 64 + i, case["iters"], case["lam"])
               for i, (n, C, spokes) in enumerate(_slices(case))]
        return dict(adjoint=[b for b, _ in out], x=[x for _, x in out])

    if kind == "basis":
        n, C, T, K = case["n"], case["coils"], case["frames"], case["rank"]
        dims = (n, n, 1)
        traj = _trajectory("radial", dims, T * case["spokes"], case["readout"], seed)
        Mf = case["spokes"] * case["readout"]
        bas = torch.from_numpy(_basis(case, seed)).to(DEV).to(_C128)
        per = bas.repeat_interleave(Mf, 0).t().contiguous()  # [K, M]
        maps = _maps(dims, C, seed).to(_C128)
        y = _kspace(traj, dims, C, seed, frames=T).transpose(0, 1).reshape(C, -1).to(_C128)
        nu = _Nufft64(dims, traj)
        b = torch.stack([(nu.adjoint(y * per[k].conj()[None]) * maps.conj()).sum(0) for k in range(K)])
        vals = torch.stack([per[k].conj() * per[l] for k in range(K) for l in range(K)])
        t = _Toeplitz64(dims, traj, vals)

        def mix(p, f):
            p = p.view(K, K, *p.shape[1:])
            f = f.view(C, K, *f.shape[1:])
            return torch.stack([sum(p[k, l][None] * f[:, l] for l in range(K)) for k in range(K)],
                               1).reshape(C * K, *p.shape[2:])

        z = t.normal((maps[:, None] * b[None]).reshape(C * K, 1, n, n), mix).view(C, K, 1, n, n)
        return dict(adjoint=b.reshape(-1), normal=(z * maps.conj()[:, None]).sum(0).reshape(-1))

    dims = _dims(case)
    C, spokes, R = case["coils"], case["spokes"], case["readout"]
    if kind == "cg":
        b, x = _cg_case64(dims, C, spokes, R, case["traj"], seed, case["iters"], case["lam"])
        return dict(adjoint=b, x=x)
    traj = _trajectory(case["traj"], dims, spokes, R, seed)
    nu = _Nufft64(dims, traj, _weights(traj, dims) if case["weights"] else None)
    if case["direction"] == "forward":
        img, maps = _image(dims, seed), _maps(dims, C, seed)
        cim = img.to(_C128)[None] * maps if case["maps"] else img[None] * maps
        return nu.forward(cim).reshape(-1)
    out = nu.adjoint(_kspace(traj, dims, C, seed))
    if case["maps"]:
        out = (out * _maps(dims, C, seed).to(_C128).conj()).sum(0)
    return out.reshape(-1)
