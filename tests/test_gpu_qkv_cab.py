"""On small planes a HAB's qkv linear and its CAB's first conv share one launch (the
conv's blocks, rounded up to a multiple of 8, at most half of 256 CUs): one tile, a
number of tiles that is no multiple of 8, and the planes on both sides of the line."""
import numpy as np
import pytest

from conftest import OP_TOL, make_weights

pytestmark = pytest.mark.gpu


# conv tiles: hat-s 16 x 16 pixels, hat 8 x 16
@pytest.mark.parametrize("net,h,w", [("hat-s", 16, 16), ("hat-s", 48, 80), ("hat-s", 128, 256), ("hat-s", 144, 240),
                                     ("hat", 16, 16), ("hat", 48, 80), ("hat", 128, 128), ("hat", 128, 144)])
def test_hab_on_both_sides(weights_dir, net, h, w):
    import hat_amd as hl
    import oracle
    path = make_weights(weights_dir, net, 4, 3, [2])
    be = hl.Backend(hl.Weights(path))
    x = np.random.default_rng(31).standard_normal((h * w, 144 if net == "hat-s" else 180)).astype(np.float32)
    got, _ = be.hab(0, 1, h, w, x)
    be.close()
    want = oracle.OracleModel(path).hab(x, h, w, 0, 1)
    assert np.abs(got - want).max() < OP_TOL
