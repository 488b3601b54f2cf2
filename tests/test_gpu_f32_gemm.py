"""Float GEMMs on three-plane bf16 splits (gemm_split_kernel, gemm_split_lds_kernel) through the blocks that use them: projections whose K is
fewer steps than there are wave pairs, columns that end inside a 64-column tile, every epilogue (q|k|v with rotation,
gated and mish hidden layers, residual adds, 1x1 convolutions with emissions), over the three row tiles: against the oracle,
and every row equal to the same row in another batch. Widths that do not fit keep the float matrix unit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trunk,blocks", [
    (96, [("attn", 2, 1, 32, 32, "fixed"), ("ffn", 80, True), ("attn", 5, 5, 32, 32, "none"), ("ffn", 160, False)]),
    (64, [("attn", 1, 1, 64, 64, "learnable"), ("ffn", 1024, True), ("ffn", 256, False)]),
    (160, [("attn", 3, 3, 64, 64, "fixed"), ("ffn", 208, True), ("ffn", 160, False)]),
    (72, [("attn", 3, 1, 16, 16, "fixed"), ("ffn", 100, False)]),
    (128, [("nbt", 96, [("res", 96)]), ("nbt", 40, [("res", 40)])])])
def test_float_gemms_match_oracle_in_every_tile(kgx, synth, oracle, trunk, blocks):
    arch = synth.Arch(f"t-gemm{trunk}", 15, trunk, blocks, p1_c=16, g1_c=16, v1_c=16, v2_c=24)
    mb = synth.write_model(arch, 6)
    n = 90
    sp, gl, _ = synth.make_inputs(n, 5, board_sizes=[19, 13, 9, 2])
    net = kgx.Net(mb)
    h = kgx.Handle(net, n, "f32")
    print(f"f32 split GEMMs: {trunk}, {blocks}", flush=True)
    full = h.forward(sp, gl)
    r = [0, 2, n - 1]
    ref = oracle.Model(mb).forward(sp[r], gl[r])
    # The float tier's bound: 1e-4 of the largest output.
    assert np.isfinite(full).all() and np.abs(full[r] - ref).max() <= 1e-4 * np.abs(ref).max()
    for k in (1, 3, 10, 40, 89):
        assert np.array_equal(h.forward(sp[:k], gl[:k]), full[:k]), k
    h.close()
