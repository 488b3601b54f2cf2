"""Float 3x3 convolutions on three-plane bf16 splits (conv3_split_kernel; beyond 256 x 256 channels Winograd), over channel counts that end inside a 64-channel
chunk and inside a column tile, and over the batches where the tile changes: against the oracle, and every row equal to
the same row in another batch; magnitudes far from one, where the planes' exponents range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trunk,mid,act,scale", [
    (192, 192, "ACTIVATION_MISH", 1.0), (128, 72, "ACTIVATION_RELU", 1.0), (40, 264, "ACTIVATION_MISH", 1.0), (256, 264, "ACTIVATION_MISH", 1.0),
    (64, 64, "ACTIVATION_RELU", 1e12), (64, 64, "ACTIVATION_RELU", 1e-12)])
def test_float_convolutions_match_oracle_in_every_tile(kgx, synth, oracle, trunk, mid, act, scale):
    arch = synth.Arch(f"t-split{mid}", 14, trunk, [("res", mid), ("gpool", trunk, 64), ("res", mid)], mid_c=mid, gpool_c=64,
                      act=act, mid_bn_gain=scale)
    mb = synth.write_model(arch, 3)
    n = 34
    sp, gl, _ = synth.make_inputs(n, 4, board_sizes=[19, 13, 9, 19, 7])
    net = kgx.Net(mb)
    h = kgx.Handle(net, n, "f32")
    print(f"f32 split convolutions: {trunk}/{mid}, {act}, scale {scale}", flush=True)
    full = h.forward(sp, gl)
    r = [0, 3, n - 1]
    ref = oracle.Model(mb).forward(sp[r], gl[r])
    # The float tier's bound: 1e-4 of the largest output.
    assert np.isfinite(full).all() and np.abs(full[r] - ref).max() <= 1e-4 * np.abs(ref).max()
    for k in (1, 5, 8, 9, 16, 17, 22, 33):
        assert np.array_equal(h.forward(sp[:k], gl[:k]), full[:k]), k
    h.close()
