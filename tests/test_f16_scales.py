"""The powers of two that bring operands into f16's range, where the values are far
from 1 or the attention's q and k admit none (the FP32 attention then runs before the
split-f16 tail)."""
import ctypes as C

import numpy as np
import pytest

from checkpoint_edit import edited
from conftest import FWD_MEAN_TOL, FWD_TOL, OP_TOL, make_weights

HEADS = 6


class _QkvScale(C.Structure):
    _fields_ = [("q", C.c_float), ("k", C.c_float), ("v", C.c_float), ("ok", C.c_bool)]


def _qkv_scale(bq, bk, bv, head_dim):
    import hat_amd as hl
    f = hl.lib()._ZN3hat9qkv_scaleEdddi  # hat::qkv_scale(double, double, double, int)
    f.restype, f.argtypes = _QkvScale, [C.c_double, C.c_double, C.c_double, C.c_int]
    return f(bq, bk, bv, head_dim)


@pytest.mark.parametrize("bq,bk,ok", [(10.0, 10.0, True), (1e6, 1e6, False), (1e30, 1e-30, False),
                                      (float("inf"), 1.0, False)])
@pytest.mark.parametrize("bv", [1e-6, 1.0, 1e5])
def test_v_is_scaled_whatever_becomes_of_q_and_k(bq, bk, ok, bv):
    """v feeds the split tail whichever attention runs."""
    s = _qkv_scale(bq, bk, bv, 24)
    assert s.ok == ok and (ok or s.q == s.k == 1.0)
    assert 2.0 ** 14 <= bv * s.v <= 2.0 ** 15


def _no_pair(q_w, q_b, k_w, k_b):
    """q and k bounded past 2^30 together, scores unchanged: two dims of the first head
    with 1e6 on one side and zeros on the other."""
    q_b[0], k_w[0], k_b[0] = 1e6, 0.0, 0.0
    k_b[1], q_w[1], q_b[1] = 1e6, 0.0, 0.0


@pytest.mark.gpu
@pytest.mark.parametrize("c", [144, 180])
@pytest.mark.parametrize("vs", [1e-6, 1.0, 1e7])
def test_ocab_behind_the_fp32_attention(c, vs):
    import hat_amd as hl
    import oracle
    rng = np.random.default_rng(41)

    def n(std, *s):
        return (rng.standard_normal(s) * std).astype(np.float32)
    h, w = 32, 48
    x = n(1.0, h * w, c)
    ws = [n(0.05, *s) for s in [(c,), (c,), (3 * c, c), (3 * c,), (c, c), (c,), (1521, HEADS), (c,), (c,),
                                (2 * c, c), (2 * c,), (c, 2 * c), (c,)]]
    ws[0] += 1.0
    ws[7] += 1.0
    _no_pair(ws[2][:c], ws[3][:c], ws[2][c:2 * c], ws[3][c:2 * c])
    # v times vs, the projection over vs: the block's output stays
    ws[2][2 * c:] *= np.float32(vs)
    ws[3][2 * c:] *= np.float32(vs)
    ws[4] /= np.float32(vs)
    print(f"ocab {c} channels, v times {vs}", flush=True)
    got = hl.op_ocab(x, h, w, c, HEADS, 2, ws)[0]
    assert np.isfinite(got).all()
    assert np.abs(got - oracle.ocab_op(x, h, w, c, HEADS, 2, ws)).max() < OP_TOL


@pytest.mark.gpu
@pytest.mark.parametrize("net", ["hat-s", "hat"])
@pytest.mark.parametrize("vs", [1e-6, 1.0, 1e7])
def test_hab_behind_the_fp32_attention(weights_dir, net, vs):
    """The same in a HAB, whose FP32 attention also computes the channel gate."""
    import hat_amd as hl
    import oracle
    c = 144 if net == "hat-s" else 180

    def edit(meta, t):
        for b in (0, 1):
            p = f"layers.0.residual_group.blocks.{b}.attn."
            qw, qb = t[p + "qkv.weight"], t[p + "qkv.bias"]
            _no_pair(qw[:c], qb[:c], qw[c:2 * c], qb[c:2 * c])
            qw[2 * c:] *= np.float32(vs)
            qb[2 * c:] *= np.float32(vs)
            t[p + "proj.weight"] *= np.float32(4.0 / vs)
    path = edited(make_weights(weights_dir, net, 4, 7, [2]), weights_dir / f"{net}_nopair_{vs}.safetensors", edit)
    be, om = hl.Backend(hl.Weights(path)), oracle.OracleModel(path)
    x = np.random.default_rng(42).standard_normal((32 * 48, c), dtype=np.float32)
    for block in (0, 1):
        print(f"hab {net} block {block}, v times {vs}", flush=True)
        got = be.hab(0, block, 32, 48, x)[0]
        assert np.isfinite(got).all()
        assert np.abs(got - om.hab(x, 32, 48, 0, block)).max() < OP_TOL
    be.close()


@pytest.mark.gpu
@pytest.mark.parametrize("c", [144, 180])
@pytest.mark.parametrize("outlier", [5.0, 100.0])
def test_swmsa_small_tokens_beside_an_outlier(c, outlier):
    """Tokens of 1e-3 and one of an everyday size: the other windows come out as
    precisely as always, relative to their own size. Their q, k and v differ from the
    oracle's by rounding alone: 2^-22 of an operand from the split, the sum of 180
    terms, and the same again for P V and the projection, below 2e-6 of the largest."""
    import hat_amd as hl
    import oracle
    rng = np.random.default_rng(43)

    def n(std, *s):
        return (rng.standard_normal(s) * std).astype(np.float32)
    h, w = 32, 48
    x = n(1e-3, h * w, c)
    x[0, 5] = outlier
    ws = (n(0.07, 3 * c, c), np.zeros(3 * c, np.float32), n(0.07, c, c), np.zeros(c, np.float32), n(0.5, 961, HEADS))
    print(f"swmsa {c} channels, one value of {outlier}", flush=True)
    got = hl.op_swmsa(x, h, w, c, HEADS, 0, *ws)[0]
    want = oracle.swmsa_op(x, h, w, c, HEADS, 0, *ws)
    rest = np.ones((h, w), bool)
    rest[:16, :16] = False
    d = np.abs(got - want)[rest.ravel()].max() / np.abs(want[rest.ravel()]).max()
    assert d < 2e-6, f"worst |diff| over the largest: {d:.3e}"


@pytest.mark.gpu
@pytest.mark.parametrize("c", [144, 180])
@pytest.mark.parametrize("dead", ["attention", "mlp"])
def test_ocab_with_a_dead_branch(c, dead):
    """A branch whose weights have all but vanished adds nothing to a block input of any
    size: its scales, which the input shares in the sums, stay clear of overflow."""
    import hat_amd as hl
    import oracle
    rng = np.random.default_rng(44)

    def n(std, *s):
        return (rng.standard_normal(s) * std).astype(np.float32)
    h, w = 16, 32
    x = n(1000.0, h * w, c)
    ws = [n(0.05, *s) for s in [(c,), (c,), (3 * c, c), (3 * c,), (c, c), (c,), (1521, HEADS), (c,), (c,),
                                (2 * c, c), (2 * c,), (c, 2 * c), (c,)]]
    ws[0] += 1.0
    ws[7] += 1.0
    for i in (2, 3, 4) if dead == "attention" else (9, 10, 11):
        ws[i] *= np.float32(1e-18)
    print(f"ocab {c} channels, dead {dead}", flush=True)
    got = hl.op_ocab(x, h, w, c, HEADS, 2, ws)[0]
    assert np.isfinite(got).all()
    assert np.abs(got - oracle.ocab_op(x, h, w, c, HEADS, 2, ws)).max() < 1000 * OP_TOL


def _planes_times(s):
    """An edit that takes the trunk's and the head's planes to s times their size and
    the image back: every branch that adds to them, conv_first and the head's biases
    times s, conv_last over s."""
    def edit(meta, t):
        f = np.float32(s)
        for k in t:
            branch = k.endswith((".proj.weight", ".proj.bias", ".fc2.weight", ".fc2.bias", ".cab.2.weight", ".cab.2.bias"))
            norm = k.startswith("patch_embed.norm.")
            trunk = k.startswith(("conv_first.", "conv_after_body."))
            bias = k.endswith(".bias") and (k.startswith(("conv_before_upsample.", "upsample."))
                                            or k.startswith("layers.") and k.endswith(".conv.bias"))
            if branch or norm or trunk or bias:
                t[k] *= f
        t["conv_last.weight"] /= f
    return edit


@pytest.mark.gpu
@pytest.mark.parametrize("net", ["hat-s", "hat"])
@pytest.mark.parametrize("s", [1e-5, 1e5])
def test_planes_far_from_one(weights_dir, net, s):
    """The Winograd convs find their inputs' range on the device."""
    import hat_amd as hl
    import oracle
    path = edited(make_weights(weights_dir, net, 4, 7, [2, 2]), weights_dir / f"{net}_times_{s}.safetensors", _planes_times(s))
    be, om = hl.Backend(hl.Weights(path)), oracle.OracleModel(path)
    for h, w in [(32, 48), (70, 100)]:
        img = np.random.default_rng(45).random((3, h, w), dtype=np.float32)
        print(f"forward {net} {h}x{w}, planes times {s}", flush=True)
        d = np.abs(be.forward(h, w, img) - om.forward(h, w, img))
        assert d.max() < FWD_TOL and d.mean() < FWD_MEAN_TOL
    be.close()


@pytest.mark.gpu
@pytest.mark.parametrize("net,scale", [("hat-s", 4), ("hat", 2)])
def test_no_range_is_kept_from_the_pass_before(weights_dir, net, scale):
    """After an image of 1e6, one of the usual size comes out as on a new backend,
    bit for bit."""
    import hat_amd as hl
    W = hl.Weights(make_weights(weights_dir, net, scale, 7, [2, 2]))
    img = np.random.default_rng(46).random((3, 40, 56), dtype=np.float32)
    be = hl.Backend(W)
    want = be.forward(40, 56, img)
    be.close()
    be = hl.Backend(W)
    assert np.isfinite(be.forward(40, 56, img * np.float32(1e6))).all()
    assert np.array_equal(be.forward(40, 56, img), want)
    be.close()


@pytest.mark.gpu
@pytest.mark.parametrize("cab", [1e-6, 1e3, 1e8])
def test_folded_conv2_beside_the_projection(weights_dir, cab):
    """The folded conv2 and the projection share the tail's accumulators: conv2's
    weights far below the projection's, and far above, where the projection's are
    scaled down to make room."""
    import hat_amd as hl
    import oracle

    def edit(meta, t):
        for k in t:
            if k.endswith(".cab.2.weight"):
                t[k] *= np.float32(cab)
    path = edited(make_weights(weights_dir, "hat-s", 4, 7, [2]), weights_dir / f"cab_{cab}.safetensors", edit)
    be, om = hl.Backend(hl.Weights(path)), oracle.OracleModel(path)
    x = np.random.default_rng(47).standard_normal((32 * 48, 144), dtype=np.float32)
    for block in (0, 1):
        print(f"hab block {block}, conv2 times {cab}", flush=True)
        want = om.hab(x, 32, 48, 0, block)
        assert np.abs(be.hab(0, block, 32, 48, x)[0] - want).max() < OP_TOL * max(1.0, np.abs(want).max())
    be.close()
