"""Reads and restarts that go straight between the caller's device arrays and
the state: against the host paths, bit for bit, at widths that are no
multiple of the row pitch, with some outputs left out, with outputs that
overlap, and at every stage a handle can be in."""
import ctypes

import numpy as np
import pytest
import torch

from tests.helpers import circle_domain, rect_domain

pytestmark = pytest.mark.gpu


def _solver(H, W, kind):
    from fingering_dynamics_amd.lbm import Compute
    from fingering_dynamics_amd.params import LbmParams
    if kind == "walled":
        mask, bits, _ = rect_domain(H, W, max(1, W // 25), size=3, seed=W, x_min=12)
        return Compute(mask, bits, LbmParams.walled(H, W, M=10.0, psi_wall=-0.5, gamma=1.0027))
    mask, bits, _ = circle_domain(H, W, 3, 5, 0.9, seed=5, x_lo=12)
    return Compute(mask, bits, LbmParams.periodic(H, W, M=5.0, psi_wall=0.0, n_inv_cols=10))


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("H,W,kind", [(34, 64, "periodic"), (40, 131, "periodic"), (33, 70, "walled")])
def test_device_fields_at_every_stage(H, W, kind):
    cm = _solver(H, W, kind)
    f, g = None, None

    def check():
        host = [a.copy() for a in cm.fields()]
        dev = cm.fields_device()
        torch.cuda.synchronize()
        for a, b in zip(host, dev.cpu().numpy()):
            assert np.array_equal(a, b)
        one = torch.full((2, H, W), 7.0, device="cuda")
        torch.cuda.synchronize()
        assert cm._lib.fd_fields_device(cm._h, None, _ptr(one[1]), None, None) == 0
        torch.cuda.synchronize()
        assert np.array_equal(one[1].cpu().numpy(), host[1]) and bool((one[0] == 7.0).all())
        # two outputs in one array: the later one stands, as with copies in turn
        assert cm._lib.fd_fields_device(cm._h, _ptr(one[0]), _ptr(one[0]), None, None) == 0
        torch.cuda.synchronize()
        assert np.array_equal(one[0].cpu().numpy(), host[1])

    check()                                     # N = 0 of fd_init
    cm.step(3)
    check()                                     # a running state
    f, g = cm.populations()
    cm.set_populations(f, g)
    check()                                     # handed-over populations
    cm.step(2)
    fields = [torch.as_tensor(a).cuda() for a in cm.fields()]
    torch.cuda.synchronize()
    cm.init_fields_device(*fields)
    check()                                     # N = 0 of a restart
    cm.close()


@pytest.mark.parametrize("H,W,kind", [(34, 64, "periodic"), (40, 131, "periodic"), (33, 70, "walled")])
def test_restart_from_device_fields_equals_host_restart(H, W, kind):
    a, b = _solver(H, W, kind), _solver(H, W, kind)
    a.step(5)
    fields = [v.copy() for v in a.fields()]
    dev = [torch.as_tensor(v).cuda() for v in fields]
    torch.cuda.synchronize()
    a.init_fields_device(*dev)
    b.init_fields(*fields)
    a.synchronize()
    for t in dev:
        t.fill_(float("nan"))                   # the handle keeps what the reads of N = 0 need
    torch.cuda.synchronize()
    assert a.mass() == b.mass() and a.watchdog() == b.watchdog()
    for x, y in zip(a.fields() + a.populations(), b.fields() + b.populations()):
        assert np.array_equal(x, y)
    a.step(7)
    b.step(7)
    for x, y in zip(a.fields() + a.populations(), b.fields() + b.populations()):
        assert np.array_equal(x, y)
    assert a.mass() == b.mass()
    a.close()
    b.close()
