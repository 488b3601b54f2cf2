"""Attention of float handles (attn_f32_kernel): every head dim, shared key/value heads, learnable and no rotation, on
ragged boards, against the oracle; and rows that do not depend on the batch across the two query-block widths (up to 24
(row, head) pairs take 16 queries per workgroup, more take 32)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,dim,rope", [(4, 4, 64, "fixed"), (4, 2, 32, "learnable"), (6, 1, 16, "none"),
                                               (5, 5, 64, "none")])
def test_float_attention_matches_oracle_at_both_widths(kgx, synth, oracle, heads, kv, dim, rope):
    arch = synth.Arch(f"t-attn{dim}", 15, 64, [("attn", heads, kv, dim, dim, rope), ("ffn", 96, True),
                                              ("attn", heads, kv, dim, dim, rope)],
                      p1_c=16, g1_c=16, v1_c=16, v2_c=24, qk_gain=2.0)
    mb = synth.write_model(arch, 17)
    n = 20 // heads + 2  # the whole batch takes the wide blocks, up to 24 // heads rows the narrow ones
    sp, gl, _ = synth.make_inputs(n, 23, board_sizes=[19, 9, 13, 2])
    net = kgx.Net(mb)
    h = kgx.Handle(net, n, "f32")
    print(f"f32 attention {heads}/{kv} heads of {dim}, {n} rows", flush=True)
    out = h.forward(sp, gl)
    ref = oracle.Model(mb).forward(sp, gl)
    # The float tier's bound: 1e-4 of the largest output.
    assert np.abs(out - ref).max() <= 1e-4 * np.abs(ref).max()
    for k in (1, 20 // heads, 20 // heads + 1):
        assert np.array_equal(h.forward(sp[:k], gl[:k]), out[:k]), k
    h.close()


def test_float_attention_scores_far_below_zero(kgx, synth, oracle):
    """Scores of -1e33 and less (keys opposite to every query): the largest one still takes the softmax, and the key slots
    past the board's last point none of it. Tokens of two kinds, the last point's kind not the one its like attend to."""
    arch = synth.Arch("t-negscores", 15, 64, [("attn", 1, 1, 64, 64, "none")], stem_k=1, p1_c=16, g1_c=16, v1_c=16, v2_c=24)
    mb, t = synth.write_model_tree(arch, 12)
    b = t["blocks"][0]

    def put(old, new):
        nonlocal mb
        assert mb.count(old.tobytes()) == 1
        mb = mb.replace(old.tobytes(), np.ascontiguousarray(new, np.float32).tobytes())

    stem = np.zeros_like(t["stem"].transpose(2, 3, 1, 0))  # [1, 1, planes, channels]
    stem[0, 0, 0, 0] = stem[0, 0, 1, 1] = 1.0
    put(t["stem"].transpose(2, 3, 1, 0), stem)
    put(t["stem_mm"], np.zeros_like(t["stem_mm"]))
    put(b["q"], np.eye(64, dtype=np.float32) * np.float32(1e16))
    put(b["k"], np.eye(64, dtype=np.float32) * np.float32(-1e16))
    n = 25  # both query-block widths
    sp, gl, _ = synth.make_inputs(n, 3)
    sp = sp.reshape(n, 22, 361).copy()
    sp[:, 1] = 0.0
    sp[:, 1, :100] = 1.0
    sp = sp.reshape(n, 22, 19, 19)
    ref = oracle.Model(mb).forward(sp[:2], gl[:2])
    net = kgx.Net(mb)
    h = kgx.Handle(net, n, "f32")
    for k in (2, n):
        print(f"f32 attention, scores far below zero: {k} rows", flush=True)
        out = h.forward(sp[:k], gl[:k])
        # The float tier's bound: 1e-4 of the largest output.
        assert np.abs(out[:2] - ref).max() <= 1e-4 * np.abs(ref).max(), k
    h.close()
