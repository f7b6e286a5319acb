"""Convolutions of narrow images (up to eight columns) on both sides of the line
between the staged kernels, which compute 32 columns, and the general one.

Tolerance: the FP32 accumulation bound K 2^-23 * sum |products| against
float64 convolutions of the same bf16 operands."""
import pytest
import torch

from tests.test_gpu_surrogate_staged import EPS, _conv64, _operands

pytestmark = pytest.mark.gpu

SHAPES = [(67, 201, 2, 48, 96), (64, 256, 1, 64, 64), (3, 999, 3, 40, 200), (40, 250, 4, 16, 40), (64, 64, 2, 48, 96),
          (9, 33, 8, 64, 64), (200, 30, 5, 8, 8), (100, 50, 1, 32, 192), (33, 100, 7, 96, 24)]


@pytest.mark.parametrize("shape", SHAPES)
def test_narrow_images(shape):
    from fingering_dynamics_amd import surrogate_ops as so
    x, w, b, g = _operands(*shape)
    ref, mag = _conv64(x, w) + b.double().cpu(), _conv64(x.abs(), w.abs()) + b.double().cpu().abs()
    bound = 9 * shape[3] * EPS * mag + 1e-30
    y = so.conv3x3(x, w, b, out_dtype=torch.float32).double().cpu()
    assert torch.all((y - ref).abs() <= bound)
    r = so.conv3x3(x, w, b, relu=True).double().cpu()
    assert torch.all((r - ref.clamp(min=0)).abs() <= 2.0 ** -8 * ref.abs() + bound)
    m = torch.randn(x.shape, device="cuda", generator=g).relu().to(torch.bfloat16)
    pre = torch.where(m > 0, x, torch.zeros_like(x))
    d = so.conv3x3_bwd_data(x, w, out_dtype=torch.float32, relu_y=m).double().cpu()
    assert torch.all((d - _conv64(pre, w)).abs() <= bound)


def test_narrow_images_take_no_longer_than_on_the_general_kernel():
    """48 -> 96 channels on 67 x 201 x 2 pixels: 51 us staged, 25 on the general
    kernel, which an x two bytes off a 16-byte boundary takes."""
    from fingering_dynamics_amd import surrogate_ops as so
    x, w, b, _ = _operands(67, 201, 2, 48, 96)
    off = torch.empty(x.numel() + 1, dtype=torch.bfloat16, device="cuda")[1:].view(x.shape).copy_(x)

    def us(t):
        best = 1e9
        for _ in range(5):
            a, c = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record()
            for _ in range(20):
                so.conv3x3(t, w, b)
            c.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(c) * 50)
        return best
    us(x), us(off)
    assert us(x) < 1.3 * us(off)
