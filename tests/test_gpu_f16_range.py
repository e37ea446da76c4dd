"""The split-f16 attention needs q, k and v inside f16's range. The host bounds them
from the weights and the input's largest value, folds balancing powers of two into
the weights, and runs the FP32 kernels where no power of two fits. One token of an
outlier value moves that bound without touching the other windows, which must come
out as always: within OP_TOL of the oracle, on either side of the rule."""
import numpy as np
import pytest

from conftest import OP_TOL

pytestmark = pytest.mark.gpu


# bound of q (times scale log2 e) times bound of k: about 3e2, 2e6 (f16, scaled) and
# 2e12, past the 2^30 that two balanced f16 operands can hold (FP32 kernels)
@pytest.mark.parametrize("c", [144, 180])
@pytest.mark.parametrize("outlier", [3.0, 300.0, 3e5])
def test_swmsa_outlier_leaves_other_windows(c, outlier):
    import hat_amd as hl
    import oracle
    rng = np.random.default_rng(11)
    hp, wp, heads = 32, 48, 6

    def n(std, *s):
        return (rng.standard_normal(s) * std).astype(np.float32)
    x = n(1.0, hp * wp, c)
    x[0, 5] = outlier
    w = (n(0.07, 3 * c, c), n(0.1, 3 * c), n(0.07, c, c), n(0.1, c), n(0.5, 961, heads))
    got, _, _ = hl.op_swmsa(x, hp, wp, c, heads, 0, *w)
    want = oracle.swmsa_op(x, hp, wp, c, heads, 0, *w)
    assert np.isfinite(got).all()
    rest = np.ones((hp, wp), bool)
    rest[:16, :16] = False
    d = np.abs(got - want)[rest.ravel()]
    assert d.max() < OP_TOL, f"worst |diff| {d.max():.3e}"


@pytest.mark.parametrize("scale", [1e-6, 1e5])
def test_swmsa_value_scale(scale):
    """v's own power of two: values far from 1 come out as precisely."""
    import hat_amd as hl
    import oracle
    rng = np.random.default_rng(12)
    hp, wp, c, heads = 16, 32, 144, 6

    def n(std, *s):
        return (rng.standard_normal(s) * std).astype(np.float32)
    x = n(1.0, hp * wp, c)
    qkv_w, qkv_b = n(0.07, 3 * c, c), n(0.1, 3 * c)
    qkv_w[2 * c:] *= np.float32(scale)
    qkv_b[2 * c:] *= np.float32(scale)
    w = (qkv_w, qkv_b, n(0.07, c, c), np.zeros(c, np.float32), n(0.5, 961, heads))
    got, _, _ = hl.op_swmsa(x, hp, wp, c, heads, 8, *w)
    want = oracle.swmsa_op(x, hp, wp, c, heads, 8, *w)
    assert np.abs(got - want).max() < OP_TOL * scale
