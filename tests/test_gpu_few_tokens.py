"""One to a few tokens: the launches that route for themselves and combine, against the oracle, at the edges of their ranges
(one unit a block, experts at a power of two of the lanes, a shared expert narrower than the routed ones, the last batches that
take them and the first that do not, by tokens, by the weights read and by the units of a token; half and whole tiles of the down blocks)."""
import numpy as np
import pytest
import torch

import synth
from gpu_util import banks_on_device, clear_tokens, dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    import tqllm_amd
    return tqllm_amd


@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q4_K", "Q6_K", "IQ3_S", "NVFP4G"])
@pytest.mark.parametrize("n,hidden,ff,experts,topk,shared_ff", [(1, 256, 256, 4, 1, 0), (2, 512, 768, 64, 6, 256), (5, 2304, 512, 128, 8, 512), (6, 1280, 512, 129, 10, 256),
                                                               (7, 512, 256, 65, 3, 0), (8, 512, 256, 65, 3, 0), (1, 512, 1536, 513, 16, 512), (2, 2816, 256, 9, 2, 256),
                                                               (5, 2560, 1280, 33, 8, 256), (1, 512, 2816, 8, 5, 0), (1, 512, 2816, 8, 6, 0),
                                                               (1, 4096, 256, 5, 2, 0), (1, 4352, 256, 5, 2, 256),
                                                               (12, 512, 256, 65, 3, 256), (13, 512, 256, 65, 3, 256), (9, 1024, 512, 300, 8, 0), (6, 2048, 768, 40, 10, 768)])
def test_layer_of_few_tokens(tq, oracle, fmt, n, hidden, ff, experts, topk, shared_ff):
    cfg = dict(hidden=hidden, ff=ff, experts=experts, topk=topk, shared_ff=shared_ff, wtype=getattr(oracle, fmt), rtype="bf16", xtype="bf16")
    raws = synth.make_banks(cfg, seed=n + hidden, distinct=min(experts + 1, 8))
    gate, up, down = banks_on_device(cfg, raws)
    inp = synth.make_inputs(cfg, n, seed=n)
    layer = tq.MoeLayer(dev(inp["router"]), dev(inp["shared_gate"]) if shared_ff else None, gate, up, down, topk, shared_ff=shared_ff, weight_scale=2.5)
    assert layer.path(n) == "decode"
    x = dev(inp["x"])
    out, ids, w, logits = (t.cpu().numpy() for t in layer.forward(x, return_routing=True))
    want, want_ids, want_w = oracle.layer_forward(inp["x"][1], logits, *raws, cfg["wtype"], hidden, ff, experts, topk, shared_ff=shared_ff, act_mode=0, threads=16, scale=2.5)
    clear = clear_tokens(oracle, logits, experts, topk, ids, want_ids)
    assert np.array_equal(ids[clear], want_ids[clear]) and np.abs(w[clear] - want_w[clear]).max() < 3e-6
    assert synth.errors(out[clear], want[clear])[1] < 1e-3
    res = torch.randn_like(x)
    got = layer.forward(x, residual=res)
    assert torch.equal(got, (torch.from_numpy(out).cuda().bfloat16().float() + res.float()).bfloat16())


@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q4_K"])
def test_down_rows_wider_than_the_decode_products_take(tq, oracle, fmt):
    """8448 columns: batches of up to six tokens have the launches of few tokens whatever they read, the next is refused."""
    cfg = dict(hidden=256, ff=8448, experts=8, topk=2, shared_ff=0, wtype=getattr(oracle, fmt), rtype="bf16", xtype="bf16")
    raws = synth.make_banks(cfg, seed=5, distinct=2)
    inp = synth.make_inputs(cfg, 7, seed=6)
    layer = tq.MoeLayer(dev(inp["router"]), None, *banks_on_device(cfg, raws), 2)
    x = dev(inp["x"])
    for n in (1, 6):
        out, ids, _, logits = (t.cpu().numpy() for t in layer.forward(x[:n], return_routing=True))
        want, want_ids, _ = oracle.layer_forward(inp["x"][1][:n], logits, *raws, cfg["wtype"], 256, 8448, 8, 2, act_mode=0, threads=16)
        assert np.array_equal(ids, want_ids) and synth.errors(out, want)[1] < 1e-3
    with pytest.raises(tq.TqmoeError, match="too wide"):
        layer.forward(x)


def test_batches_that_outgrow_the_workspace(tq, oracle):
    """A layer's workspace grows with the batches it is given, with and without residual rows, and its results are those of a new layer."""
    cfg = dict(hidden=512, ff=256, experts=8, topk=2, shared_ff=0, wtype=oracle.IQ4_XS, rtype="bf16", xtype="bf16")
    banks = banks_on_device(cfg, synth.make_banks(cfg, seed=3))
    inp = synth.make_inputs(cfg, 300, seed=4)
    make = lambda: tq.MoeLayer(dev(inp["router"]), None, *banks, 2)
    layer, x = make(), dev(inp["x"])
    for n, residual in ((1, None), (40, None), (300, x), (2, x), (200, None)):
        res = residual[:n].contiguous() if residual is not None else None
        assert torch.equal(layer.forward(x[:n], residual=res), make().forward(x[:n], residual=res))
    assert layer._ws.numel() == layer.workspace(300).numel()


@pytest.mark.parametrize("experts", [65, 300])
@pytest.mark.parametrize("spread", [70, 100, 4000])
def test_logits_far_apart(tq, oracle, experts, spread):
    """Logits whose exponentials are all there, partly in the subnormal range, and zero for all but a few experts (which then
    follow by index): every block of the first launch selects what the launch writes down as the routing."""
    cfg = dict(hidden=256, ff=256, experts=experts, topk=8, shared_ff=0, wtype=oracle.IQ4_XS, rtype="f32", xtype="f32")
    raws = synth.make_banks(cfg, seed=spread, distinct=5)
    inp = synth.make_inputs(cfg, 2, seed=7)
    x, router = (np.array(inp[k][1], dtype=np.float32) for k in ("x", "router"))
    x[:, 0] = [1.0, 0.5]
    router[:] = 0.0
    router[:, 0] = -np.random.default_rng(spread).permutation(experts) * (spread / experts)
    layer = tq.MoeLayer(torch.from_numpy(router).cuda(), None, *banks_on_device(cfg, raws), 8)
    out, ids, w, logits = (t.cpu().numpy() for t in layer.forward(torch.from_numpy(x).cuda(), return_routing=True))
    want, want_ids, want_w = oracle.layer_forward(x, logits, *raws, cfg["wtype"], 256, 256, experts, 8, act_mode=0, threads=4)
    assert np.array_equal(ids, want_ids) and np.abs(w - want_w).max() < 3e-6
    assert synth.errors(out, want)[1] < 1e-3
