"""A block's linears are uploaded as the kernels that run the block read them: at 144
channels a CAB that is not 6 wide keeps conv2 as a conv, and its block runs the
projection and the MLP as FP32 linears."""
import numpy as np
import pytest

from checkpoint_edit import compress_ratio, edited
from conftest import FWD_TOL, OP_TOL, make_weights


# 144 channels: 24 gives the folded CAB, 3 a CAB of 48; 180: 3 the usual 60
CASES = [("hat-s", 24), ("hat-s", 3), ("hat-s", 36), ("hat", 3), ("hat", 30)]


def _checkpoint(weights_dir, net, ratio):
    src = make_weights(weights_dir, net, 2, 5, [2])
    return edited(src, weights_dir / f"{net}_ratio{ratio}.safetensors", compress_ratio(ratio))


@pytest.mark.parametrize("net,ratio", CASES)
def test_every_linear_a_block_reads_is_uploaded(weights_dir, net, ratio):
    """The pass that counts the upload's bytes walks every tensor as the upload
    does and refuses a network whose blocks would read weights that it leaves out."""
    import hat_amd as hl
    assert hl.Weights(_checkpoint(weights_dir, net, ratio)).gpu_plan(32, 32)["weights"] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("net,ratio", CASES)
def test_cab_widths_match_the_oracle(weights_dir, net, ratio):
    import hat_amd as hl
    import oracle
    path = _checkpoint(weights_dir, net, ratio)
    W = hl.Weights(path)
    be, om = hl.Backend(W), oracle.OracleModel(path)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((32 * 48, W.embed), dtype=np.float32)
    img = rng.random((3, 20, 40), dtype=np.float32)
    for block in (0, 1):
        print(f"hab {net} compress ratio {ratio} block {block}", flush=True)
        assert np.abs(be.hab(0, block, 32, 48, x)[0] - om.hab(x, 32, 48, 0, block)).max() < OP_TOL
    assert np.abs(be.forward(20, 40, img) - om.forward(20, 40, img)).max() < FWD_TOL
    be.close()
