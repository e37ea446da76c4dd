"""The window attention's softmax over the score distributions that choose its form: a
wave takes probabilities straight from the scores where its first 32 keys lie near 0,
the online maximum where they do not, and does the item again where the first keys
promised what the later ones do not keep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HEADS = 6
# A score of size S carries the roundings of q, k, their split (2^-22 each) and the sum,
# about 2^-21 S together, in the oracle as here: at S = 25 1.2e-5 of a probability, on
# attention outputs of up to 3, and the 2e-5 of the ops on top.
TOL = 6e-5


def _weights(c, case, seed):
    rng = np.random.default_rng(seed)

    def n(std, *s):
        return (rng.standard_normal(s) * std).astype(np.float32)
    qkv_w, qkv_b, proj_w, proj_b = n(0.07, 3 * c, c), n(0.1, 3 * c), n(0.07, c, c), n(0.1, c)
    tables = [n(0.5, rows, HEADS) for rows in (961, 1521)]
    d = c // HEADS
    if case == "per head":  # q . k from flat to several units
        for i, f in enumerate([0.05, 0.5, 1.0, 2.0, 3.0, 4.0]):
            qkv_w[i * d:(i + 1) * d] *= np.float32(f)
    for t in tables:
        if case == "low":
            t -= np.float32(3.0)
        elif case == "high":
            t += np.float32(9.0)
        elif case == "wide table":
            t *= np.float32(8.0)
        elif case == "spikes":  # flat but for a few offsets, most of them seen by later keys only
            t[::97] += np.float32(20.0)
        elif case == "heads apart":
            t += np.array([0, -3, 6, -12, 12, 1], np.float32)
    return qkv_w, qkv_b, proj_w, proj_b, tables


CASES = ["near zero", "per head", "low", "high", "wide table", "spikes", "heads apart"]


@pytest.mark.parametrize("c", [144, 180])
@pytest.mark.parametrize("case", CASES)
def test_swmsa(c, case):
    import hat_amd as hl
    import oracle
    h, w = 32, 48
    qkv_w, qkv_b, proj_w, proj_b, (table, _) = _weights(c, case, 51)
    x = np.random.default_rng(52).standard_normal((h * w, c), dtype=np.float32)
    for shift in (0, 8):
        print(f"swmsa {c} {case} shift {shift}", flush=True)
        args = (x, h, w, c, HEADS, shift, qkv_w, qkv_b, proj_w, proj_b, table)
        got = hl.op_swmsa(*args)[0]
        assert np.isfinite(got).all()
        assert np.abs(got - oracle.swmsa_op(*args)).max() < TOL


@pytest.mark.parametrize("c", [144, 180])
@pytest.mark.parametrize("case", CASES)
def test_ocab(c, case):
    import hat_amd as hl
    import oracle
    h, w = 48, 48  # every kind of window: corner, edge and inside
    qkv_w, qkv_b, proj_w, proj_b, (_, table) = _weights(c, case, 53)
    rng = np.random.default_rng(54)
    x = rng.standard_normal((h * w, c), dtype=np.float32)
    one, zero = np.ones(c, np.float32), np.zeros(c, np.float32)
    mlp = [(rng.standard_normal(s) * 0.02).astype(np.float32) for s in [(2 * c, c), (2 * c,), (c, 2 * c), (c,)]]
    ws = [one, zero, qkv_w, qkv_b, proj_w, proj_b, table, one, zero, *mlp]
    print(f"ocab {c} {case}", flush=True)
    got = hl.op_ocab(x, h, w, c, HEADS, 2, ws)[0]
    assert np.isfinite(got).all()
    assert np.abs(got - oracle.ocab_op(x, h, w, c, HEADS, 2, ws)).max() < TOL
