"""Float handles keep 24-bit operands: their 3x3 convolutions and GEMMs take float products as six products of bf16 planes, and
the loss of any one of them (about 17 bits instead of 24) stays far inside the float tier's 1e-4. Here the relative
2-norm error of shallow nets is held to about four times what the device shows, and an emulation of the same nets shows
that each product's loss exceeds that."""

import numpy as np
import pytest
import torch

import torch_ref

# name -> (version, trunk, blocks, bound): the device measures 3.4e-7 (conv), 3.4e-7 (nbt), 4.2e-7 (swiglu) and 2.3e-7 (mish).
NETS = {
    "conv": (14, 128, [("res", 128), ("res", 72)], 1.4e-6),
    "nbt": (14, 128, [("nbt", 64, [("res", 64)])], 1.4e-6),
    "swiglu": (15, 256, [("ffn", 512, True)] * 2, 1.7e-6),
    "mish": (15, 256, [("ffn", 1024, False)] * 3, 0.9e-6),
}
PRODUCTS = [(2, 0), (1, 1), (1, 0), (0, 2), (0, 1), (0, 0)]  # (plane of the activation, plane of the weight)


def _net(synth, name):
    version, trunk, blocks, bound = NETS[name]
    # (A 1x1 stem and ReLU: the Winograd stem and the fast exponential would add errors of their own.)
    arch = synth.Arch(f"t-acc-{name}", version, trunk, blocks, mid_c=64, p1_c=16, g1_c=16, v1_c=16, v2_c=24, stem_k=1,
                      act="ACTIVATION_RELU")
    return synth.write_model_tree(arch, 5), bound


class _PlaneProducts(torch_ref.Ref):
    """The float64 network with its blocks' products of activations and weights taken over bf16 planes of both."""

    def __init__(self, tree, products):
        super().__init__(tree)
        self.products, self.on = products, False

    def product(self, f, x, w):
        def planes(v):
            out, rest = [], v.to(torch.float32)
            for _ in range(3):
                h = rest.to(torch.bfloat16).to(torch.float32)
                out.append(h.to(torch.float64))
                rest = rest - h
            return out

        a, b = planes(x), planes(w)
        return sum(f(a[i], b[j]) for i, j in self.products)

    def conv(self, x, w):
        if not self.on:
            return super().conv(x, w)
        return self.product(lambda a, b: torch.nn.functional.conv2d(a, b, padding=w.shape[-1] // 2), x, torch_ref._t(w))

    def stack(self, x, blocks):
        matmul, on = torch.matmul, self.on
        torch.matmul = lambda a, b: self.product(matmul, a, b) if b.dim() == 2 else matmul(a, b)
        self.on = True
        try:
            return super().stack(x, blocks)
        finally:
            torch.matmul, self.on = matmul, on


def _error(out, ref):
    return float(np.linalg.norm(out - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("name", sorted(NETS))
def test_bound_excludes_the_loss_of_any_plane_product(synth, name):
    (_, tree), bound = _net(synth, name)
    sp, gl, _ = synth.make_inputs(2, 6, board_sizes=[19, 13])
    ref = torch_ref.Ref(tree).forward(sp, gl)
    assert _error(_PlaneProducts(tree, PRODUCTS).forward(sp, gl), ref) <= bound / 8
    for lost in PRODUCTS:
        kept = [p for p in PRODUCTS if p != lost]
        assert _error(_PlaneProducts(tree, kept).forward(sp, gl), ref) > 1.3 * bound, lost


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(NETS))
def test_float_products_keep_24_bits(kgx, synth, oracle, name):
    (mb, _), bound = _net(synth, name)
    n, rows = 90, [0, 1, 2, 45, 89]
    sp, gl, _ = synth.make_inputs(n, 6, board_sizes=[19, 13, 9])
    ref = oracle.Model(mb).forward(sp[rows], gl[rows]).astype(np.float64)
    h = kgx.Handle(kgx.Net(mb), n, "f32")
    print(f"float accuracy: {name}", flush=True)
    for k in (n, 3):
        here = [i for i, r in enumerate(rows) if r < k]
        e = _error(h.forward(sp[:k], gl[:k])[[rows[i] for i in here]], ref[here])
        print(f"{name}, {k} rows: relative error {e:.2e}", flush=True)
        assert e <= bound, k
    h.close()
