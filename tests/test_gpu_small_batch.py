"""The launches that 16-bit handles take at few pixels (conv_small_kernel: 64, 128 or 192 pixels x 16 channels per
workgroup): every row equals, bit for bit, the same row in a batch that takes the large tiles, at the batches
where the tile changes; and two rows against the oracle."""
import numpy as np
import pytest

from test_gpu_parity import check, emulated

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f16", "bf16"])
@pytest.mark.parametrize("trunk,mid,act,batches", [
    (192, 192, "ACTIVATION_MISH", (1, 3, 4, 7, 8, 11, 12)),  # tiles change after 3, 7 and 11 rows
    (128, 128, "ACTIVATION_RELU", (1, 5, 6, 11, 12, 17, 18)),  # after 5, 11 and 17; the run-time activation
    (64, 72, "ACTIVATION_MISH", (1, 9, 10, 19, 20, 29, 30)),  # 72 outputs: a ragged last column tile
])
def test_rows_equal_the_large_tiles(kgx, synth, oracle, prec, trunk, mid, act, batches):
    print(f"small launches: {prec}, {trunk}/{mid} channels, {act}", flush=True)
    arch = synth.Arch(f"t-small{mid}", 14, trunk, [("res", mid), ("gpool", trunk, 32), ("res", mid)], mid_c=mid,
                      gpool_c=32, act=act)
    mb = synth.write_model(arch, 5)
    n = batches[-1]
    sp, gl, _ = synth.make_inputs(n, 9, board_sizes=[19, 13, 19, 9, 7])
    net = kgx.Net(mb)
    h = kgx.Handle(net, n, prec)
    full = h.forward(sp, gl)
    for k in batches[:-1]:
        assert np.array_equal(h.forward(sp[:k], gl[:k]), full[:k]), k
    h.close()
    r = [0, n - 1]
    check(full[r], oracle.Model(mb).forward(sp[r], gl[r]), net.P, net.S, prec, "small launches",
          emulated(oracle, mb, prec, sp[r], gl[r]))


@pytest.mark.parametrize("prec", ["f16", "bf16"])
@pytest.mark.parametrize("act", ["ACTIVATION_MISH", "ACTIVATION_RELU"])
def test_junction_rows_equal_the_48_pixel_tiles(kgx, synth, prec, act):
    """Junctions, the stem and the head junction on 16-pixel (up to 11 rows), 32-pixel (up to 22) and 48-pixel tiles."""
    print(f"small junctions: {prec}, {act}", flush=True)
    arch = synth.Arch("t-smalljunction", 14, 384, [("nbt", 192, [("res", 192)]), ("nbt", 192, [("gpool", 192, 64)])] * 2,
                      mid_c=192, gpool_c=64, act=act)
    n = 23
    sp, gl, _ = synth.make_inputs(n, 13, board_sizes=[19, 13, 9])
    h = kgx.Handle(kgx.Net(synth.write_model(arch, 8)), n, prec)
    full = h.forward(sp, gl)
    for k in (1, 2, 11, 12, 22):
        assert np.array_equal(h.forward(sp[:k], gl[:k]), full[:k]), k
    h.close()
