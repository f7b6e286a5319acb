"""Tiles held in LDS (several iterations per launch on small domains) against
one launch per iteration, bit for bit: every tile shape, sizes that end
inside a tile, domains smaller than a tile's margin (rows and columns that
wrap several times), every boundary, leaky solids, iteration counts that
leave remainders, states handed over between the kernels, graph replay."""
import numpy as np
import pytest

from fingering_dynamics_amd.params import (LbmParams, OUTLET_PRESSURE, PROFILE_CONST, X_PERIODIC, Y_WALLS)
from tests.helpers import circle_domain, rect_domain

pytestmark = pytest.mark.gpu


def _domain(kind, H, W):
    n = max(1, H * W // 700)
    if kind == "open":      # no obstacle: sizes too small for one
        mask, bits = np.ones((H, W), dtype=bool), np.zeros((H, W), dtype=np.uint8)
        return mask, bits, LbmParams.periodic(H, W, M=5.0, psi_wall=0.3, n_inv_cols=2, profile=PROFILE_CONST)
    if kind == "open_x":
        mask, bits = np.ones((H, W), dtype=bool), np.zeros((H, W), dtype=np.uint8)
        return mask, bits, LbmParams.periodic(H, W, M=2.0, psi_wall=-0.3, x_bc=X_PERIODIC, y_bc=Y_WALLS, wall_lo=0,
                                              wall_hi=H - 1, profile=PROFILE_CONST, u0=0.0)
    if kind == "circles":   # complete links are not used here: leaky solids
        mask, bits, _ = circle_domain(H, W, 3, 5, 0.88, seed=5, x_lo=12)
        return mask, bits, LbmParams.periodic(H, W, M=10.0, psi_wall=-0.2, n_inv_cols=10, profile=PROFILE_CONST,
                                              outlet=OUTLET_PRESSURE, psi_visc_bound=1.0)
    mask, bits, _ = rect_domain(H, W, min(n, 60), size=4, seed=7, x_min=14)
    if kind == "gauss":
        return mask, bits, LbmParams.periodic(H, W, M=5.0, psi_wall=0.0, n_inv_cols=10)
    if kind == "x_periodic":
        return mask, bits, LbmParams.periodic(H, W, M=5.0, psi_wall=0.0, x_bc=X_PERIODIC, gx=1e-6)
    return mask, bits, LbmParams.walled(H, W, M=20.0, psi_wall=-0.5, gamma=1.0027,
                                        shipped_walls=kind == "walled_shipped")


def _solver(kind, H, W, tiles):
    from fingering_dynamics_amd.lbm import Compute
    mask, bits, params = _domain(kind, H, W)
    rng = np.random.default_rng(H * W)
    psi0 = np.full((H, W), -1.0)
    psi0[:, :max(2, W // 5)] = 1.0
    psi0 += 0.01 * rng.standard_normal((H, W))
    cm = Compute(mask, bits, params, psi0=psi0)
    if tiles:
        assert cm.auto_launch()
    else:
        cm.set_fusion(1)
    return cm


def _same(a, b):
    for x, y in zip(a.fields() + a.populations(), b.fields() + b.populations()):
        assert np.array_equal(x, y, equal_nan=True)
    assert a.mass() == b.mass() or np.isnan(a.mass()[0])


# by size: 8 x 8 tiles up to 24 x 13; each with a height and width that end
# inside a tile
CASES = [("open", 3, 3), ("open", 4, 5), ("open", 9, 37), ("open_x", 3, 4), ("open_x", 11, 30), ("gauss", 48, 97),
         ("circles", 60, 131), ("walled_edge", 40, 150), ("walled_shipped", 41, 99), ("x_periodic", 30, 70),
         ("gauss", 100, 401), ("walled_shipped", 99, 400), ("circles", 151, 601), ("walled_edge", 163, 515),
         ("walled_shipped", 151, 601), ("x_periodic", 150, 450), ("gauss", 300, 599), ("walled_edge", 299, 560),
         ("circles", 330, 703), ("walled_shipped", 399, 801), ("x_periodic", 330, 700)]


@pytest.mark.parametrize("kind,H,W", CASES)
def test_tiles_equal_one_iteration_per_launch(kind, H, W):
    a, b = _solver(kind, H, W, True), _solver(kind, H, W, False)
    for n in (1, 2, 3, 7, 12, 13):
        a.step(n)
        b.step(n)
        _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("kind,H,W", [("gauss", 100, 401), ("walled_shipped", 151, 601), ("circles", 300, 599)])
def test_tiles_between_other_kernels_and_states(kind, H, W):
    """Switching between tiles, the marching kernels and graph replay, and
    stepping from handed-over populations, restarts and restored states."""
    a, b = _solver(kind, H, W, True), _solver(kind, H, W, False)

    def go(n):
        a.step(n)
        b.step(n)

    go(5)
    a.set_fusion(2)
    go(6)
    assert a.auto_launch()
    a.use_graph(True)
    for n in (40, 3, 33):
        go(n)
        _same(a, b)
    a.use_graph(False)
    f, g = a.populations()
    for c in (a, b):
        c.set_populations(f, g)
    go(9)
    _same(a, b)
    state = a.save_state()
    go(4)
    a.load_state(state)
    b.load_state(state)
    go(5)
    _same(a, b)
    fields = [v.copy() for v in a.fields()]
    for c in (a, b):
        c.init_fields(*fields)
    go(11)
    _same(a, b)
    times = a.autotune(candidates=((2, 1, 2), (1, 1, 1)), steps=6)
    assert (0, 0, 0) in times
    b.step(a.t - b.t)
    _same(a, b)
    a.close()
    b.close()


def test_large_domains_march():
    from fingering_dynamics_amd.lbm import Compute
    H, W = 1000, 1000
    cm = Compute(np.ones((H, W), dtype=bool), np.zeros((H, W), dtype=np.uint8),
                 LbmParams.periodic(H, W, M=5.0, psi_wall=0.0))
    assert not cm.auto_launch()
    cm.close()


@pytest.mark.parametrize("sizes", [[(40, 90)], [(64, 200), (33, 131), (128, 70)]])
@pytest.mark.parametrize("n", [2, 3, 5, 8, 14])
def test_ensemble_remainders(sizes, n):
    """A batched remainder of two iterations runs the two-iteration kernel."""
    from fingering_dynamics_amd.ensemble import Ensemble
    a = [_solver("walled_edge", H, W, True) for H, W in sizes]
    b = [_solver("walled_edge", H, W, False) for H, W in sizes]
    ens = Ensemble(a)
    assert ens.depth == 3
    for _ in range(2):
        ens.step(n)
        for c in b:
            c.step(n)
    ens.step_sequential(n)
    for x, y in zip(a, b):
        y.step(n)
        _same(x, y)
    ens.close()
    for c in a + b:
        c.close()
