"""Weight gradients on both sides of the line between the two kernels: layers
large enough for conv_wgrad, of every channel-block kind, with strips and runs
of rows that end inside the image, and small ones on the general kernel, whose
pixel slices end within a step, at one and beyond one.

Tolerance: the FP32 accumulation bound 2 P 2^-23 * sum |products| against
float64 convolutions of the same bf16 operands."""
import pytest
import torch

from tests.test_gpu_surrogate_staged import EPS, _operands, _wgrad64

pytestmark = pytest.mark.gpu

LARGE = [(9, 100, 70, 96, 8), (14, 90, 97, 8, 32), (10, 61, 93, 72, 136), (24, 61, 67, 24, 40), (24, 61, 67, 64, 24),
         (16, 99, 99, 32, 32), (12, 70, 41, 32, 16), (33, 32, 65, 16, 40), (70, 25, 64, 96, 48), (60, 41, 33, 64, 72)]
SMALL = [(1, 7, 9, 16, 40), (1, 8, 8, 64, 64), (1, 5, 13, 72, 8), (2, 8, 16, 32, 32), (1, 16, 32, 24, 96),
         (3, 9, 19, 64, 136), (64, 2, 2, 40, 64), (50, 31, 1, 8, 16), (2, 300, 3, 64, 32), (64, 16, 8, 64, 72)]


@pytest.mark.parametrize("shape", LARGE + SMALL)
def test_weight_gradient(shape):
    from fingering_dynamics_amd import surrogate_ops as so
    N, H, W, Cin, Cout = shape
    x, _, _, g = _operands(N, H, W, Cin, Cout)
    dy, y = [torch.randn(N, H, W, Cout, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2)]
    scratch = torch.full((int(so.load().fds_bwd_weight_scratch(N, H, W, Cin, Cout)),), float("nan"), device="cuda")
    P = N * H * W
    for mask in (None, y):
        d = dy if mask is None else torch.where(mask > 0, dy, torch.zeros_like(dy))
        dw, db = so.conv3x3_bwd_weight(x, dy, scratch=scratch, relu_y=mask)
        rw, rb = _wgrad64(x, d)
        bw, bb = _wgrad64(x.abs(), d.abs())
        assert torch.all((dw.double().cpu() - rw).abs() <= 2 * P * EPS * bw + 1e-30)
        assert torch.all((db.double().cpu() - rb).abs() <= 2 * P * EPS * bb + 1e-30)
        assert torch.equal(dw, so.conv3x3_bwd_weight(x, dy, with_bias=False, relu_y=mask)[0])


@pytest.mark.parametrize("N,H,W", [(48, 40, 33), (30, 37, 64), (24, 45, 70)])
def test_infinite_pixel(N, H, W):
    """As the test of the same name in test_gpu_surrogate_staged, in one image
    of a batch that conv_wgrad takes."""
    from fingering_dynamics_amd import surrogate_ops as so
    for Cin, Cout in ((32, 32), (64, 64), (8, 32), (32, 8)):
        for n, h, w in ((0, 0, 0), (N - 1, 0, W - 1), (N // 2, H - 1, W - 1), (N - 1, H - 1, 0), (1, H // 2, W - 1)):
            x = torch.ones(N, H, W, Cin, device="cuda", dtype=torch.bfloat16)
            x[n, h, w, 3] = float("inf")
            dw, _ = so.conv3x3_bwd_weight(x, torch.ones(N, H, W, Cout, device="cuda", dtype=torch.bfloat16))
            for dh in range(3):
                for dv in range(3):
                    inside = 0 <= h - dh + 1 < H and 0 <= w - dv + 1 < W
                    t = dw[:, dh, dv]
                    assert bool(torch.isinf(t[:, 3]).all() if inside else torch.isfinite(t[:, 3]).all())
                    assert bool(torch.isfinite(t[:, :3]).all()) and bool(torch.isfinite(t[:, 4:]).all())


def test_small_layers_take_no_longer_than_on_the_general_kernel():
    """The line between the kernels: 67 x 201 x 2 pixels of 96 -> 96 channels
    took 159 us on conv_wgrad and 79 on the general kernel, which an x two
    bytes off a 16-byte boundary takes."""
    from fingering_dynamics_amd import surrogate_ops as so
    N, H, W, Cin, Cout = 67, 201, 2, 96, 96
    x, _, _, g = _operands(N, H, W, Cin, Cout)
    dy = torch.randn(N, H, W, Cout, device="cuda", generator=g).to(torch.bfloat16)
    off = torch.empty(x.numel() + 1, dtype=torch.bfloat16, device="cuda")[1:].view(x.shape).copy_(x)

    def us(t):
        best = 1e9
        for _ in range(5):
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record()
            for _ in range(10):
                so.conv3x3_bwd_weight(t, dy)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        return best
    us(x), us(off)
    assert us(x) < 1.3 * us(off)
