"""Attention of float handles (attn_f32_kernel): every head dim, shared key/value heads, learnable and no rotation, on
ragged boards, against the oracle; and rows that do not depend on the batch across the two query-block widths (up to 20
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
    n = 20 // heads + 2  # the whole batch takes the wide blocks, up to 20 // heads rows the narrow ones
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
