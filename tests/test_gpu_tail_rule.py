"""The block tails take 64-token blocks while those are at most one a CU (256), else
128-token ones. Windows whose neighbourhood is the same on a plane of either side
of that line come out alike: each side is within OP_TOL of the oracle, so they
differ by at most twice that."""
import numpy as np
import pytest

from conftest import OP_TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c", [144, 180])
def test_ocab_same_on_both_sides(c):
    import hat_amd as hl
    rng = np.random.default_rng(21)
    heads, mlp = 6, 2

    def n(std, *s):
        return (rng.standard_normal(s) * std).astype(np.float32)
    big = n(1.0, 128, 144, c)
    shapes = [(c,), (c,), (3 * c, c), (3 * c,), (c, c), (c,), (1521, heads), (c,), (c,),
              (mlp * c, c), (mlp * c,), (c, mlp * c), (c,)]
    ws = [n(0.05, *s) for s in shapes]
    ws[0] += 1.0
    ws[7] += 1.0
    # the last two windows of a row on the small plane see its edge: 96 columns are shared
    got_l = hl.op_ocab(big.reshape(-1, c), 128, 144, c, heads, mlp, ws)[0].reshape(128, 144, c)
    got_s = hl.op_ocab(np.ascontiguousarray(big[:, :128]).reshape(-1, c), 128, 128, c, heads, mlp, ws)[0].reshape(128, 128, c)
    assert np.isfinite(got_l).all() and np.isfinite(got_s).all()
    d = np.abs(got_l[:, :96] - got_s[:, :96]).max()
    assert d < 2 * OP_TOL, f"worst |diff| {d:.3e}"
