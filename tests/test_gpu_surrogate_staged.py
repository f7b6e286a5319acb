"""The staged convolution kernels at the edges of their dispatch: every
block shape (few and many blocks), ragged image sizes, channel counts that
end inside a block, float32 and bf16 results, the ReLU mask on load, and
operands that are not 16-byte aligned, which take the general kernel.

Tolerance: the FP32 accumulation bound K * 2^-23 * sum |products| of
test_gpu_surrogate_ops, against float64 convolutions of the same bf16
operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -23


def _conv64(x, w):
    return torch.nn.functional.conv2d(x.double().cpu().permute(0, 3, 1, 2), w.double().cpu().permute(0, 3, 1, 2),
                                      padding=1).permute(0, 2, 3, 1)


def _operands(N, H, W, Cin, Cout, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + N * H + W + 7 * Cin + Cout)
    x = torch.randn(N, H, W, Cin, device="cuda", generator=g).to(torch.bfloat16)
    w = (0.2 * torch.randn(Cout, 3, 3, Cin, device="cuda", generator=g)).to(torch.bfloat16)
    return x, w, torch.randn(Cout, device="cuda", generator=g), g


# (N, H, W, Cin, Cout): each block shape of the dispatch, sizes that end
# inside a block in every direction
SHAPES = [(9, 121, 250, 32, 8), (9, 121, 250, 96, 24), (5, 121, 250, 64, 96), (5, 121, 250, 32, 96),
          (9, 121, 125, 64, 72), (9, 121, 125, 64, 64), (5, 61, 125, 64, 40), (3, 61, 125, 32, 32),
          (1, 61, 125, 32, 64), (1, 33, 17, 128, 136), (1, 1, 1, 32, 8), (2, 3, 40, 256, 16), (1, 70, 1, 64, 32),
          (3, 50, 70, 8, 40), (2, 9, 33, 16, 8), (1, 17, 31, 24, 64), (2, 8, 32, 40, 32), (1, 25, 65, 48, 24),
          (1, 7, 100, 56, 32), (1, 20, 20, 72, 40)]


@pytest.mark.parametrize("shape", SHAPES)
def test_staged_convolution(shape):
    from fingering_dynamics_amd import surrogate_ops as so
    x, w, b, _ = _operands(*shape)
    ref = _conv64(x, w) + b.double().cpu()
    bound = 9 * shape[3] * EPS * (_conv64(x.abs(), w.abs()) + b.double().cpu().abs()) + 1e-30
    y = so.conv3x3(x, w, b, out_dtype=torch.float32).double().cpu()
    assert torch.all((y - ref).abs() <= bound)
    r = so.conv3x3(x, w, b, relu=True).double().cpu()
    assert torch.all((r - ref.clamp(min=0)).abs() <= 2.0 ** -8 * ref.abs() + bound)
    n = so.conv3x3(x, w, out_dtype=torch.float32).double().cpu()   # no bias
    assert torch.all((n - (ref - b.double().cpu())).abs() <= bound)


@pytest.mark.parametrize("shape", SHAPES)
def test_staged_convolution_masks_on_load(shape):
    from fingering_dynamics_amd import surrogate_ops as so
    x, w, _, g = _operands(*shape)
    m = torch.randn(x.shape, device="cuda", generator=g).relu().to(torch.bfloat16)
    m.view(-1)[0] = -0.0                                           # negative zero is masked
    pre = torch.where(m > 0, x, torch.zeros_like(x))
    got = so.conv3x3_bwd_data(x, w, out_dtype=torch.float32, relu_y=m)
    bound = 2 * 9 * shape[3] * EPS * _conv64(pre.abs(), w.abs()) + 1e-30   # either may take another block shape
    assert torch.all((got.double().cpu() - so.conv3x3_bwd_data(pre, w, out_dtype=torch.float32).double().cpu()).abs()
                     <= bound)


@pytest.mark.parametrize("shape", SHAPES)
def test_unaligned_operands_take_the_general_kernel(shape):
    """A contiguous x two bytes off a 16-byte boundary: the same values, up
    to the order of the FP32 sums (the same order when the channels make
    one chunk)."""
    from fingering_dynamics_amd import surrogate_ops as so
    x, w, b, _ = _operands(*shape)
    buf = torch.empty(x.numel() + 1, dtype=torch.bfloat16, device="cuda")
    off = buf[1:].view(x.shape).copy_(x)
    assert off.data_ptr() % 16 != 0
    y, z = [so.conv3x3(t, w, b, out_dtype=torch.float32) for t in (x, off)]
    if shape[3] <= 56:
        assert torch.equal(y, z)
    bound = 2 * 9 * shape[3] * EPS * (_conv64(x.abs(), w.abs()) + b.double().cpu().abs()) + 1e-30
    assert torch.all((y - z).double().cpu().abs() <= bound)


def test_infinite_pixels_reach_their_neighbours_only():
    """An infinite pixel at the image's corner: infinite or NaN outputs at
    the 2 x 2 pixels its taps reach, finite ones elsewhere (padding and the
    zero-filled part of a K step multiply nothing infinite)."""
    from fingering_dynamics_amd import surrogate_ops as so
    for Cin in (8, 24, 32, 40, 64):
        x, w, b, _ = _operands(1, 19, 45, Cin, 32)
        x[0, 0, 0, :] = float("inf")
        bad = ~torch.isfinite(so.conv3x3(x, w, b, out_dtype=torch.float32)).all(dim=3)[0]
        assert bool(bad[:2, :2].all()) and int(bad.sum()) == 4


# weight gradient: every channel-block kind, strips that end inside the image
# and at its edge, one row and column, runs of rows that do not divide the
# height, fewer work items than wave groups and several per group
WSHAPES = [(1, 1, 1, 8, 8), (1, 1, 40, 32, 32), (2, 37, 33, 8, 32), (3, 12, 64, 16, 72), (2, 19, 31, 32, 16),
           (1, 50, 65, 96, 8), (2, 33, 96, 32, 32), (4, 61, 70, 32, 64), (2, 9, 33, 64, 32), (3, 21, 45, 128, 24),
           (2, 20, 32, 64, 64), (5, 35, 61, 72, 136), (1, 130, 32, 64, 64), (40, 16, 32, 128, 128),
           (9, 100, 128, 24, 40), (2, 40, 6, 96, 48)]


def _wgrad64(x, dy):
    xa, da = [t.double().cpu().permute(0, 3, 1, 2) for t in (x, dy)]
    Cout, Cin = da.shape[1], xa.shape[1]
    return torch.nn.grad.conv2d_weight(xa, (Cout, Cin, 3, 3), da, padding=1).permute(0, 2, 3, 1), da.sum((0, 2, 3))


@pytest.mark.parametrize("shape", WSHAPES)
def test_weight_gradient(shape):
    """dw and dbias, with and without the ReLU mask, from a scratch full of
    NaN (nothing is read that was not written), the same on every call."""
    from fingering_dynamics_amd import surrogate_ops as so
    N, H, W, Cin, Cout = shape
    x, _, _, g = _operands(N, H, W, Cin, Cout)
    dy = torch.randn(N, H, W, Cout, device="cuda", generator=g).to(torch.bfloat16)
    y = torch.randn(N, H, W, Cout, device="cuda", generator=g).to(torch.bfloat16)
    n = int(so.load().fds_bwd_weight_scratch(N, H, W, Cin, Cout))
    scratch = torch.full((n,), float("nan"), device="cuda")
    for mask in (None, y):
        d = dy if mask is None else torch.where(mask > 0, dy, torch.zeros_like(dy))
        dw, db = so.conv3x3_bwd_weight(x, dy, scratch=scratch, relu_y=mask)
        rw, rb = _wgrad64(x, d)
        bw, bb = _wgrad64(x.abs(), d.abs())
        P = N * H * W
        assert torch.all((dw.double().cpu() - rw).abs() <= 2 * P * EPS * bw + 1e-30)
        assert torch.all((db.double().cpu() - rb).abs() <= 2 * P * EPS * bb + 1e-30)
        again, _ = so.conv3x3_bwd_weight(x, dy, with_bias=False, relu_y=mask)
        assert torch.equal(dw, again)


@pytest.mark.parametrize("shape", [(2, 37, 33, 8, 32), (4, 61, 70, 32, 64), (3, 21, 45, 128, 24), (5, 35, 61, 72, 136)])
def test_weight_gradient_of_unaligned_operands(shape):
    """x two bytes off a 16-byte boundary takes the general kernel."""
    from fingering_dynamics_amd import surrogate_ops as so
    N, H, W, Cin, Cout = shape
    x, _, _, g = _operands(N, H, W, Cin, Cout)
    dy = torch.randn(N, H, W, Cout, device="cuda", generator=g).to(torch.bfloat16)
    buf = torch.empty(x.numel() + 1, dtype=torch.bfloat16, device="cuda")
    off = buf[1:].view(x.shape).copy_(x)
    (dw, db), (dw2, db2) = so.conv3x3_bwd_weight(x, dy), so.conv3x3_bwd_weight(off, dy)
    bw, bb = _wgrad64(x.abs(), dy.abs())
    P = N * H * W
    assert torch.all((dw - dw2).double().cpu().abs() <= 4 * P * EPS * bw + 1e-30)
    assert torch.all((db - db2).double().cpu().abs() <= 4 * P * EPS * bb + 1e-30)


@pytest.mark.parametrize("H,W", [(5, 40), (37, 64), (40, 33)])
def test_infinite_pixel_in_the_weight_gradient(H, W):
    """An infinite x on the image's edge (channel 3) meets dy only where a
    tap takes it to a pixel of the image: its products are infinite there
    and absent elsewhere, never infinity times a padded zero."""
    from fingering_dynamics_amd import surrogate_ops as so
    for Cin, Cout in ((32, 32), (64, 64), (8, 32), (32, 8)):
        for h, w in ((0, 0), (0, W - 1), (H - 1, W - 1), (H - 1, 0), (H // 2, W - 1), (H - 1, W // 2)):
            x = torch.ones(1, H, W, Cin, device="cuda", dtype=torch.bfloat16)
            x[0, h, w, 3] = float("inf")
            dw, _ = so.conv3x3_bwd_weight(x, torch.ones(1, H, W, Cout, device="cuda", dtype=torch.bfloat16))
            for dh in range(3):
                for dv in range(3):
                    inside = 0 <= h - dh + 1 < H and 0 <= w - dv + 1 < W
                    t = dw[:, dh, dv]
                    assert bool(torch.isinf(t[:, 3]).all() if inside else torch.isfinite(t[:, 3]).all())
                    assert bool(torch.isfinite(t[:, :3]).all()) and bool(torch.isfinite(t[:, 4:]).all())
