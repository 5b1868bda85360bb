"""A token whose activations hold a NaN or an infinity: its own result is undefined, its neighbours' are those of a batch without
it, whatever the gating and whichever launches route the batch."""
import numpy as np
import pytest
import torch

import synth
from gpu_util import banks_on_device, dev

pytestmark = pytest.mark.gpu

GATINGS = {"softmax": (1, False, True), "softmax_biased": (1, True, True), "softmax_raw": (1, False, False), "sigmoid": (2, False, True), "sigmoid_biased": (2, True, True),
           "selected_softmax": (3, False, True), "sqrt_softplus": (4, False, True)}


@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q4_K"])
@pytest.mark.parametrize("n", [5, 800])
@pytest.mark.parametrize("gating", sorted(GATINGS))
def test_neighbours_of_a_token_without_numbers(oracle, gating, n, fmt):
    import tqllm_amd as tq
    mode, biased, norm = GATINGS[gating]
    cfg = dict(hidden=512, ff=256, experts=33, topk=4, shared_ff=256, wtype=getattr(oracle, fmt), rtype="bf16", xtype="bf16")
    gate, up, down = banks_on_device(cfg, synth.make_banks(cfg, seed=3, distinct=5))
    inp = synth.make_inputs(cfg, n, seed=n)
    bias = torch.rand(33, device="cuda") * 0.1 if biased else None
    layer = tq.MoeLayer(dev(inp["router"]), dev(inp["shared_gate"]), gate, up, down, 4, shared_ff=256, gating=mode, probs_bias=bias, norm_weights=norm)
    x = dev(inp["x"])
    others = torch.arange(n, device="cuda") != 2
    want = layer.forward(x)
    for at, value in (([7], float("nan")), ([3, 200], float("inf")), (slice(None), float("nan"))):
        y = x.clone()
        y[2, at] = value
        out, ids, w, _ = layer.forward(y, return_routing=True)
        ids = ids.cpu().numpy()
        assert ids.min() >= 0 and ids.max() < 33 and all(len(set(row)) == 4 for row in ids.tolist())
        assert torch.equal(out[others], want[others]) and torch.isfinite(want).all()


@pytest.mark.parametrize("fmt,n", [("IQ4_XS", 60), ("Q6_K", 60), ("Q6_K", 250), ("IQ3_S", 60), ("IQ3_S", 250), ("IQ3_S", 800), ("NVFP4G", 60)])
def test_neighbours_in_items_of_all_sizes(oracle, fmt, n):
    """The token without numbers takes or leaves a row of its neighbours' experts: their items' row tiles change, their bits do not."""
    test_neighbours_of_a_token_without_numbers(oracle, "softmax", n, fmt)
