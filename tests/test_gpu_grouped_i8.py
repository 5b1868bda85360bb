"""The int8 grouped products of the layer on rows in quantiser order (IQ4_XS), at the row counts where items and row tiles begin and
end: the same integer sums and the same roundings as the entry points on gathered rows, so the same bits."""
import numpy as np
import pytest
import torch

import synth
from gpu_util import banks_on_device, dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    import tqllm_amd
    return tqllm_amd


def on_gathered_rows(tq, layer, x, ids, w, logits, blocks, shared_ff):
    """The layer's output from the modular entry points."""
    n, k = ids.shape
    experts = layer.gate.experts - (1 if shared_ff else 0)
    ext = tq.moe_extend_ids(ids, experts) if shared_ff else ids
    slots = ext.shape[1]
    lists = tq.moe_dispatch(ext, layer.gate.experts)[:3]
    shared_w = torch.sigmoid(logits[:, experts]).contiguous() if shared_ff else None
    if blocks:
        act = tq.expert_gemm_gateup_i8_blocks(layer.gate, layer.up, *tq.group_rows_i8_blocks(x, lists, n * slots, slots), lists, n, slots, k, shared_ff)
        y = tq.expert_gemm_i8_blocks(layer.down, *tq.group_rows_i8_blocks(act, lists, n * slots, 1), lists, n, slots, k, shared_ff)
    else:
        act = tq.expert_gemm_gateup_i8(layer.gate, layer.up, *tq.group_rows_i8(x, lists, n * slots, slots), lists, n, slots, k, shared_ff)
        y = tq.expert_gemm_i8(layer.down, *tq.group_rows_i8(act, lists, n * slots, 1), lists, n, slots, k, shared_ff)
    return tq.moe_combine_strided(y.view(n, slots, -1), slots, w, shared_w)


@pytest.mark.parametrize("blocks", [1, 2])
@pytest.mark.parametrize("n,hidden,ff,shared_ff", [(64, 256, 256, 0), (65, 512, 256, 256), (96, 256, 768, 256), (127, 1280, 512, 512), (128, 256, 512, 256), (129, 768, 1280, 0),
                                                  (161, 2048, 256, 256), (700, 768, 512, 0), (1030, 256, 512, 512)])
@pytest.mark.parametrize("experts", [7, 60])
def test_layer_equals_the_products_on_gathered_rows(tq, oracle, blocks, n, hidden, ff, shared_ff, experts):
    """Seven experts (items of 64 rows): two of them and the shared one hold exactly n rows up to 161 tokens. Sixty (items of 32)."""
    cfg = dict(hidden=hidden, ff=ff, experts=experts, topk=2, shared_ff=shared_ff, wtype=oracle.IQ4_XS, rtype="f32", xtype="f32")
    banks = banks_on_device(cfg, synth.make_banks(cfg, seed=n + hidden, distinct=3))
    inp = synth.make_inputs(cfg, n, seed=n)
    x, router = (np.array(inp[k][1], dtype=np.float32) for k in ("x", "router"))
    if n < 700 and experts == 7:
        x[:, 0] = 4.0
        router[:, 0] = [0, 3, 0, 0, 4, 0, 0]
    x[3] = 0.0                                   # a row without a scale
    x = torch.from_numpy(x).cuda()
    layer = tq.MoeLayer(torch.from_numpy(router).cuda(), dev(inp["shared_gate"]) if shared_ff else None, *banks, 2, shared_ff=shared_ff, act_blocks=blocks)
    assert layer.path(n) == "grouped_i8"
    out, ids, w, logits = layer.forward(x, return_routing=True)
    want = on_gathered_rows(tq, layer, x, ids, w, logits, blocks == 1, shared_ff)
    if shared_ff:        # (the shared expert's weight is the device's sigmoid on one side, torch's on the other)
        assert synth.errors(out.cpu().numpy(), want.cpu().numpy())[1] < 1e-6
    else:
        assert torch.equal(out, want)


@pytest.mark.parametrize("experts", [7, 60])
def test_largest_sums_of_a_scale_per_32(tq, oracle, experts):
    """A sub-block's integer sum at its bounds, 32 * 127 * 127 with either sign (every weight the table's first value, rows of one value):
    the sums reach fp32 by another way than on the gathered rows, and with the same bits."""
    n = 130
    cfg = dict(hidden=512, ff=256, experts=experts, topk=2, shared_ff=0, wtype=oracle.IQ4_XS, rtype="f32", xtype="f32")
    raws = [np.array(raw).reshape(-1, 136) for raw in synth.make_banks(cfg, seed=9, distinct=3)]
    for raw in raws[:2]:
        raw[:, 8:] = 0
    banks = banks_on_device(cfg, [raw.reshape(-1) for raw in raws])
    inp = synth.make_inputs(cfg, n, seed=n)
    x = torch.ones((n, 512), device="cuda")
    x[1::2] = -0.25
    x[2::3] *= torch.linspace(0.0, 1.0, 512, device="cuda")
    layer = tq.MoeLayer(dev(inp["router"]), None, *banks, 2, act_blocks=1)
    assert layer.path(n) == "grouped_i8"
    out, ids, w, logits = layer.forward(x, return_routing=True)
    assert torch.isfinite(out).all() and torch.equal(out, on_gathered_rows(tq, layer, x, ids, w, logits, True, 0))
