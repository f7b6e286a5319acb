"""Graph replay of the marching kernels (Compute.use_graph(True)): every call
below replays the captured pair of launches, and each follows a change of the
depth, of the launch shape at one depth, of the parity or of the state, so that
a pair captured for another configuration would show.  Compared bit for bit
with eager launches of one iteration, with reads between the replays."""
import pytest

from tests.test_gpu_tiles import _same, _solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,H,W", [("gauss", 48, 97), ("walled_edge", 163, 515), ("circles", 151, 601),
                                      ("x_periodic", 150, 450)])
def test_replays_of_the_marching_kernels(kind, H, W):
    a, b = _solver(kind, H, W, True), _solver(kind, H, W, False)
    a.use_graph(True)
    # 4 x depth iterations and more in a call are replayed; the odd counts
    # leave remainders and flip the buffers' parity
    for depth, wx, rows, steps in ((3, 1, 7, (12, 19)), (3, 1, 24, (14, 30)), (3, 2, 24, (25,)), (2, 1, 5, (8, 13)),
                                   (2, 4, 16, (21, 10)), (1, 0, 0, (4, 9)), (3, 1, 7, (37,)), (2, 1, 5, (17, 17))):
        a.set_fusion(depth, wx, rows)
        if depth == 1:
            a.set_tile(2, 3)
        for n in steps:
            a.step(n)
            b.step(n)
            _same(a, b)
    a.set_fusion(1)
    a.set_tile(1, 9)                      # depth 1, another shape
    for n in (8, 15):
        a.step(n)
        b.step(n)
        _same(a, b)
    assert a.auto_launch()                # tiles, then the march again
    for depth in (None, 3):
        if depth:
            a.set_fusion(depth)
        a.step(50)
        b.step(50)
        _same(a, b)
    blob = b.save_state()                 # another state in the same buffers
    for c in (a, b):
        c.step(5)
        c.load_state(blob)
        c.step(23)
    _same(a, b)
    a.close()
    b.close()
