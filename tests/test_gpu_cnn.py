"""GPU: the warm-start network's 3x3 convolution layers (matrix cores,
bfloat16 operands, FP32 accumulation) against the FP64 oracle
(oracle/cnn.py).

The oracle is evaluated on the operands rounded to bfloat16 exactly as the
kernels round them, so the only difference left is FP32 accumulation order:
relative L2 <= 1e-5.  Against the unrounded operands the bfloat16 rounding
(8-bit mantissa) shows as a relative error of a few 1e-3, printed."""
import numpy as np
import pytest

import bart_amd as ba
from oracle import cnn as R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda")


def relerr(a, ref):
    a = np.asarray(a, np.float64)
    return float(np.linalg.norm(a - ref) / np.linalg.norm(ref))


SHAPES = [(2, 2, 48, 6, 64), (1, 48, 48, 5, 128), (2, 48, 2, 4, 64), (1, 3, 5, 3, 100), (1, 48, 48, 3, 256)]


@pytest.mark.parametrize("B,Cin,Cout,H,W", SHAPES)
def test_conv3x3_forward(B, Cin, Cout, H, W):
    rng = np.random.default_rng(Cin * 100 + Cout)
    x = rng.standard_normal((B, Cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((Cout, Cin, 3, 3)) / np.sqrt(9 * Cin)).astype(np.float32)
    bias = rng.standard_normal(Cout).astype(np.float32)
    res = rng.standard_normal((B, Cout, H, W)).astype(np.float32)
    y = ba.conv3x3(dev(x), dev(w), dev(bias)).cpu().numpy()
    ref = R.conv3x3(R.bf16(x), R.bf16(w), bias)
    print(f"forward vs bf16-operand oracle {relerr(y, ref):.1e}, vs fp64 {relerr(y, R.conv3x3(x, w, bias)):.1e}")
    assert relerr(y, ref) < 1e-5
    yr = ba.conv3x3(dev(x), dev(w), dev(bias), relu=True).cpu().numpy()
    assert relerr(yr, np.maximum(ref, 0)) < 1e-5
    ys = ba.conv3x3(dev(x), dev(w), None, res=dev(res)).cpu().numpy()
    assert relerr(ys, R.conv3x3(R.bf16(x), R.bf16(w)) + res) < 1e-5


@pytest.mark.parametrize("B,Cin,Cout,H,W", SHAPES)
def test_conv3x3_backward_data(B, Cin, Cout, H, W):
    rng = np.random.default_rng(7 + Cin)
    w = (rng.standard_normal((Cout, Cin, 3, 3)) / np.sqrt(9 * Cin)).astype(np.float32)
    dy = rng.standard_normal((B, Cout, H, W)).astype(np.float32)
    dx = ba.conv3x3_bwd_data(dev(dy), dev(w)).cpu().numpy()
    ref = R.conv3x3_bwd_data(R.bf16(dy), R.bf16(w))
    assert relerr(dx, ref) < 1e-5


@pytest.mark.parametrize("B,Cin,Cout,H,W", [s for s in SHAPES if s[4] % 8 == 0] + [(3, 48, 48, 17, 64)])
def test_conv3x3_backward_weights(B, Cin, Cout, H, W):
    rng = np.random.default_rng(11 + Cout)
    x = rng.standard_normal((B, Cin, H, W)).astype(np.float32)
    dy = rng.standard_normal((B, Cout, H, W)).astype(np.float32)
    dw, db = ba.conv3x3_bwd_weights(dev(x), dev(dy))
    rdw, rdb = R.conv3x3_bwd_weights(R.bf16(x), R.bf16(dy))
    assert relerr(dw.cpu().numpy(), rdw) < 1e-5
    # the bias gradient sums dy in FP32 without rounding it
    assert relerr(db.cpu().numpy(), R.conv3x3_bwd_weights(x, dy)[1]) < 1e-5


# edges of the launch: strips of 256 pixels, 16-pixel and 32-pixel tiles,
# channel groups of 8 and 16 (and the two groups of output-channel tiles), one
# row, more rows than a work-group takes, pointers off 16 bytes.  FP32 sums of
# at most 9 * 64 products (forward) or B H W products (gradients).
EDGES = [(1, 1, 1, 1, 8), (1, 64, 64, 3, 257), (2, 33, 17, 9, 24), (1, 17, 64, 2, 40), (1, 56, 48, 5, 16),
         (3, 40, 33, 300, 8), (1, 9, 49, 2, 515),
         # strips of equal width, and halves of a strip for few rows; the weight
         # gradient's largest LDS layout and all its tiles
         (1, 48, 48, 2, 320), (1, 2, 48, 5, 320), (2, 16, 16, 700, 272), (1, 56, 64, 3, 256)]


@pytest.mark.parametrize("B,Cin,Cout,H,W", EDGES)
@pytest.mark.parametrize("offset", [0, 1])
def test_conv3x3_edges(B, Cin, Cout, H, W, offset):
    rng = np.random.default_rng(B + 3 * Cin + 5 * Cout + 7 * W)
    x = rng.standard_normal((B, Cin, H, W)).astype(np.float32)
    dy = rng.standard_normal((B, Cout, H, W)).astype(np.float32)
    w = (rng.standard_normal((Cout, Cin, 3, 3)) / np.sqrt(9 * Cin)).astype(np.float32)

    def shifted(a):
        flat = torch.zeros(a.size + offset, dtype=torch.float32, device="cuda")
        flat[offset:] = dev(a).reshape(-1)
        return flat[offset:].view(a.shape)

    y = ba.conv3x3(shifted(x), dev(w)).cpu().numpy()
    assert relerr(y, R.conv3x3(R.bf16(x), R.bf16(w))) < 1e-5
    dx = ba.conv3x3_bwd_data(shifted(dy), dev(w)).cpu().numpy()
    assert relerr(dx, R.conv3x3_bwd_data(R.bf16(dy), R.bf16(w))) < 1e-5
    if W % 8 or W > 256 or (Cout + 31) // 32 * ((9 * Cin + 31) // 32) > 32:
        return
    dw, db = ba.conv3x3_bwd_weights(shifted(x), shifted(dy))
    assert relerr(dw.cpu().numpy(), R.conv3x3_bwd_weights(R.bf16(x), R.bf16(dy))[0]) < 1e-5
    assert relerr(db.cpu().numpy(), R.conv3x3_bwd_weights(x, dy)[1]) < 1e-5


def test_conv3x3_rejects_bad_shapes():
    x = torch.zeros((1, 65, 4, 64), device="cuda")
    w = torch.zeros((8, 65, 3, 3), device="cuda")
    with pytest.raises(ba.BartError, match="channels"):
        ba.conv3x3(x, w)
    x = torch.zeros((1, 4, 4, 100), device="cuda")
    dy = torch.zeros((1, 4, 4, 100), device="cuda")
    with pytest.raises(ba.BartError, match="multiple of 8"):
        ba.conv3x3_bwd_weights(x, dy)


# A row is padded to 32 pixels for the matrix cores: the last pixel has no left
# tap in the image and must not reach that tap's gradient through the padding.
@pytest.mark.parametrize("W", [8, 24, 32, 40])
def test_conv3x3_backward_weights_nonfinite_last_pixel(W):
    rng = np.random.default_rng(W)
    x = rng.standard_normal((2, 17, 5, W)).astype(np.float32)
    dy = rng.standard_normal((2, 3, 5, W)).astype(np.float32)
    x[1, 4, 2, W - 1] = np.inf
    dw = ba.conv3x3_bwd_weights(dev(x), dev(dy))[0].cpu().numpy()
    x[1, 4, 2, W - 1] = 0
    ref = R.conv3x3_bwd_weights(R.bf16(x), R.bf16(dy))[0]
    assert not np.any(np.isfinite(dw[:, 4, :, 1:]))
    dw[:, 4, :, 1:] = ref[:, 4, :, 1:]
    assert relerr(dw, ref) < 1e-5
