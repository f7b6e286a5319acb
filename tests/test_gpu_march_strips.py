"""The three-iteration march's strips against one launch per iteration, bit
for bit: widths where an inner strip (all of whose lanes are columns 1 ...
W-2) first exists, ends at the last column allowed and is followed by one or
two edge strips; chunks of any height; walls, periodic x, obstacles that are
kept out of memory and leaky ones that stream on."""
import numpy as np
import pytest

from fingering_dynamics_amd.params import (LbmParams, OUTLET_PRESSURE, PROFILE_CONST, X_PERIODIC)
from tests.helpers import circle_domain, rect_domain

pytestmark = pytest.mark.gpu


def _domain(kind, H, W):
    if kind == "circles":
        mask, bits, _ = circle_domain(H, W, 3, 5, 0.9, seed=W, x_lo=12)
        return mask, bits, LbmParams.periodic(H, W, M=10.0, psi_wall=-0.2, n_inv_cols=10, profile=PROFILE_CONST,
                                              outlet=OUTLET_PRESSURE, psi_visc_bound=1.0)
    mask, bits, _ = rect_domain(H, W, max(2, H * W // 500), size=4, seed=W, x_min=14)
    if kind == "x_periodic":
        return mask, bits, LbmParams.periodic(H, W, M=5.0, psi_wall=0.0, x_bc=X_PERIODIC, gx=1e-6, profile=PROFILE_CONST)
    if kind == "rects":
        return mask, bits, LbmParams.periodic(H, W, M=5.0, psi_wall=0.0, n_inv_cols=10, profile=PROFILE_CONST)
    return mask, bits, LbmParams.walled(H, W, shipped_walls=False, M=20.0, psi_wall=-0.5, gamma=1.0027)


@pytest.mark.parametrize("kind", ["rects", "circles", "walled", "x_periodic"])
@pytest.mark.parametrize("H,W,waves,rows", [(23, 104, 1, 5), (23, 105, 1, 7), (40, 106, 2, 40), (31, 152, 1, 1),
                                            (31, 153, 2, 3), (64, 154, 1, 16), (64, 193, 1, 22), (50, 320, 2, 9),
                                            (97, 333, 1, 80)])
def test_strips_equal_one_iteration_per_launch(kind, H, W, waves, rows):
    from fingering_dynamics_amd.lbm import Compute
    mask, bits, params = _domain(kind, H, W)
    psi0 = np.full((H, W), -1.0)
    psi0[:, :max(2, W // 5)] = 1.0
    psi0 += 0.01 * np.random.default_rng(H * W).standard_normal((H, W))
    a, b = Compute(mask, bits, params, psi0=psi0), Compute(mask, bits, params, psi0=psi0)
    a.set_fusion(3, waves, rows)
    b.set_fusion(1)
    for n in (3, 12, 13):
        a.step(n)
        b.step(n)
        for x, y in zip(a.fields() + a.populations(), b.fields() + b.populations()):
            assert np.array_equal(x, y, equal_nan=True)
    a.close()
    b.close()


@pytest.mark.parametrize("depth", [2, 3])
@pytest.mark.parametrize("H,W,rows", [(2048, 1500, 90), (1023, 2050, 31)])
def test_a_full_device_equals_one_iteration_per_launch(depth, H, W, rows):
    """Several waves on every SIMD: a store's data registers are read late, so a kernel that writes them too soon
    after it issued the store (the link masks of the next phase) stores other values here and not on small grids."""
    from fingering_dynamics_amd.lbm import Compute
    mask, bits, _ = rect_domain(H, W, 150, size=8, seed=W, x_min=14)
    params = LbmParams.periodic(H, W, M=5.0, psi_wall=0.0, n_inv_cols=10, profile=PROFILE_CONST)
    psi0 = np.full((H, W), -1.0)
    psi0[:, :W // 5] = 1.0
    a, b = Compute(mask, bits, params, psi0=psi0), Compute(mask, bits, params, psi0=psi0)
    a.set_fusion(depth, 1, rows)
    b.set_fusion(1)
    for _ in range(3):
        a.step(2 * depth)
        b.step(2 * depth)
        for x, y in zip(a.populations(), b.populations()):
            assert np.array_equal(x, y, equal_nan=True)
    a.close()
    b.close()
