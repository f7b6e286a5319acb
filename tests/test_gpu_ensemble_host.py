"""What an ensemble's step costs the host: the launch shape is chosen when the
table is built, not for every launch."""
import time

import numpy as np
import pytest

from fingering_dynamics_amd.lbm import Compute
from fingering_dynamics_amd.params import LbmParams

pytestmark = pytest.mark.gpu


def test_sequential_steps_take_no_longer_with_the_default_shape():
    # 512 domains: choosing the height is a scan over 90 heights and all of
    # them, some 130 us, where a launch takes about 10
    from fingering_dynamics_amd.ensemble import Ensemble
    H, W = 64, 256
    mask, bits = np.ones((H, W), bool), np.zeros((H, W), np.uint8)
    params = LbmParams.periodic(H, W, M=5.0, psi_wall=0.0)
    cms = [Compute(mask, bits, params) for _ in range(512)]
    ens = Ensemble(cms)

    def host_seconds(n):
        best = 1e9
        ens.step_sequential(2 * n)                  # builds the table
        for _ in range(3):
            ens.synchronize()
            t0 = time.perf_counter()
            ens.step_sequential(n)                  # one launch per domain, asynchronous
            best = min(best, time.perf_counter() - t0)
        return best

    depth, wx, rows = ens.fusion
    default = [host_seconds(n) for n in (3, 2)]     # three iterations a launch, a remainder of two
    ens.set_fusion(2, wx, rows)
    ens.set_fusion(3, wx, rows)
    chosen = [host_seconds(n) for n in (3, 2)]
    ens.close()
    for c in cms:
        c.close()
    for d, c in zip(default, chosen):
        assert d < 3 * c + 2e-3, (default, chosen)
