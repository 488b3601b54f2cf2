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


def _set_weights(mb, old, new):
    """The model bytes with one weight array replaced (the arrays are written as raw float blocks)."""
    assert mb.count(old.tobytes()) == 1 and old.shape == new.shape
    return mb.replace(old.tobytes(), np.ascontiguousarray(new, np.float32).tobytes())


def _one_channel_net(synth):
    """A mish feed-forward block (256 -> 1024 -> 256) behind a trunk that is zero but for channel 0: with it, every token's
    normalized row is 16 ln[0] in channel 0, so a hidden value is set by one weight."""
    arch = synth.Arch("t-onechannel", 15, 256, [("ffn", 1024, False)], p1_c=16, g1_c=16, v1_c=16, v2_c=24,
                      act="ACTIVATION_RELU")
    mb, t = synth.write_model_tree(arch, 11)
    mb = _set_weights(mb, t["stem"].transpose(2, 3, 1, 0), np.zeros_like(t["stem"].transpose(2, 3, 1, 0)))
    g = np.zeros_like(t["stem_mm"])
    g[0, 0] = 1.0
    mb = _set_weights(mb, t["stem_mm"], g)
    n = 90
    sp, gl, _ = synth.make_inputs(n, 3)
    gl[:] = 0.0
    gl[:, 0] = 1000.0
    return mb, t, t["blocks"][0], sp, gl


BATCHES = (1, 10, 90)  # the 256-column product over 1024 inputs takes 32-, 96- and 128-row tiles


def test_float_gemm_keeps_the_top_of_the_range(kgx, synth, oracle):
    """Finite operands from 3.3962e38 up, which round to infinity as bf16 values, as an activation and as a weight."""
    mb, t, b, sp, gl = _one_channel_net(synth)
    top = np.float32(3.4e38)
    l1, l2 = b["l1"].copy(), b["l2"].copy()
    l1[0, 5] = top / (np.float32(16.0) * b["ln"]["w"][0])  # hidden feature 5 near the largest float
    l2[5] *= np.float32(1e-30)
    l1[0, 7] = 1e-30
    l2[7] = np.where(l2[7] < 0, -top, top)
    mb = _set_weights(_set_weights(mb, b["l1"], l1), b["l2"], l2)
    ref = oracle.Model(mb).forward(sp[:1], gl[:1])
    assert np.abs(ref).max() > 1e6
    net = kgx.Net(mb)
    h = kgx.Handle(net, len(sp), "f32")
    for n in BATCHES:
        print(f"top of the float range: {n} rows", flush=True)
        out = h.forward(sp[:n], gl[:n])
        # The float tier's bound: 1e-4 of the largest output.
        assert np.isfinite(out).all() and np.abs(out[0] - ref[0]).max() <= 1e-4 * np.abs(ref).max(), n
    h.close()


def test_float_gemm_keeps_infinities(kgx, synth, monkeypatch):
    """A hidden value that overflows to infinity reaches the trunk as the infinity of its weight's sign, as on the float matrix
    unit (KGX_CONV=wino4): positive in channel 0 alone, so that every ownership output is +inf through positive weights."""
    mb, t, b, sp, gl = _one_channel_net(synth)
    l1, l2 = b["l1"].copy(), b["l2"].copy()
    l1[0, 5] = 1e38
    l2[5] = -np.abs(l2[5]) - np.float32(1e-3)
    l2[5, 0] = 0.5
    own = t["heads"]["own"].transpose(2, 3, 1, 0)
    mb = _set_weights(_set_weights(mb, b["l1"], l1), b["l2"], l2)
    mb = _set_weights(mb, own, np.abs(own) + np.float32(1e-3))
    net = kgx.Net(mb)
    h = kgx.Handle(net, len(sp), "f32")
    monkeypatch.setenv("KGX_CONV", "wino4")
    unit = kgx.Handle(net, len(sp), "f32")
    for n in BATCHES:
        print(f"infinite operands: {n} rows", flush=True)
        out, ref = h.forward(sp[:n], gl[:n]), unit.forward(sp[:n], gl[:n])
        assert np.isposinf(ref[:, -361:]).all() and np.array_equal(out, ref, equal_nan=True), n
    h.close()
    unit.close()
