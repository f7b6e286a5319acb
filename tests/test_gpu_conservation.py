"""Density and phase of a closed box on the GPU: nothing leaves it, so the
sums over its nodes stay what they were."""
import numpy as np
import pytest

from fingering_dynamics_amd.lbm import Compute
from fingering_dynamics_amd.params import LbmParams, X_PERIODIC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1.0, 5.0, 20.0])
def test_closed_droplet_keeps_its_density(M):
    # a collision's bias in a node's sum of f is below 2^-27 (that of its
    # rounded constants below 2^-28, tests/test_node_precision.py, and as much
    # again because most nodes hold nearly the same values)
    H = W = 64
    n = 2000
    y, x = np.mgrid[0:H, 0:W]
    psi = np.tanh((16 - np.hypot(y - 32, x - 32)) / 1.4)
    cm = Compute(np.ones((H, W), bool), np.zeros((H, W), np.uint8),
                 LbmParams.periodic(H, W, M=M, psi_wall=0.0, x_bc=X_PERIODIC))
    cm.init(psi)
    cm.step(1)
    rho0 = cm.mass()[0]
    cm.step(n)
    rho1, _, bad = cm.mass()
    cm.close()
    assert bad == 0
    assert abs(rho1 / rho0 - 1) < n * 2.0 ** -27
