"""A token's result is the same bits whatever the other tokens of its batch are: they decide how many rows its experts' products
have, and with that the size and place of its items, and nothing else."""
import pytest
import torch

import synth
from gpu_util import banks_on_device, dev

pytestmark = pytest.mark.gpu



def layer_and_rows(oracle, fmt, n, experts, act_blocks, hidden=512, ff=256):
    import tqllm_amd as tq
    cfg = dict(hidden=hidden, ff=ff, experts=experts, topk=4, shared_ff=256, wtype=getattr(oracle, fmt), rtype="bf16", xtype="bf16")
    banks = banks_on_device(cfg, synth.make_banks(cfg, seed=61, distinct=5))
    inp = synth.make_inputs(cfg, n, seed=62)
    return tq.MoeLayer(dev(inp["router"]), dev(inp["shared_gate"]), *banks, 4, shared_ff=256, act_blocks=act_blocks), dev(inp["x"])


def check(layer, x, crowded):
    """The batch as it is, and with other tokens: all of them near the first kept one, so that its four experts have a row of
    every token, then all of them its opposite, so that they have few."""
    n = x.shape[0]
    kept = torch.tensor([0, 1, n // 2], device="cuda")       # tokens that stay
    others = torch.ones(n, dtype=torch.bool, device="cuda")
    others[kept] = False
    want, ids, _, _ = layer.forward(x, return_routing=True)
    noise = 0.05 * torch.randn(x.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(5))
    for sign in (1, -1):
        y = torch.where(others[:, None], (sign * x[:1].float() + noise).to(x.dtype), x)
        out, ids2, _, _ = layer.forward(y, return_routing=True)
        assert torch.equal(ids2[kept], ids[kept])
        rows = [(ids2 == e).any(dim=1).sum().item() for e in ids[0].tolist()]
        assert min(rows) > 0.5 * n if sign == 1 else max(rows) < crowded, rows
        assert torch.equal(out[kept], want[kept]), [synth.errors(out[t].cpu().numpy(), want[t].cpu().numpy())[1] for t in kept.tolist()]


@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q4_K", "Q6_K", "IQ3_S", "NVFP4G", "Q5_K", "IQ2_S"])
@pytest.mark.parametrize("n,path", [(8, "decode"), (16, "decode"), (31, "decode"), (60, "grouped"), (250, "grouped"), (800, "grouped")])
def test_result_does_not_depend_on_the_other_tokens(oracle, fmt, n, path):
    """The decode products, and the grouped ones with 5, 37 and 118 rows an expert on average: items of all sizes, with one row tile
    in one batch and several in the other."""
    layer, x = layer_and_rows(oracle, fmt, n, 60 if path == "decode" else 33, 0)
    assert layer.path(n).startswith(path)
    check(layer, x, max(4, 0.3 * n))


@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q4_K", "IQ3_S"])
@pytest.mark.parametrize("n", [70, 400])
@pytest.mark.parametrize("act_blocks", [1, 2])
def test_int8_result_does_not_depend_on_the_other_tokens(oracle, fmt, n, act_blocks):
    layer, x = layer_and_rows(oracle, fmt, n, 33, act_blocks)
    assert layer.path(n) == "grouped_i8"
    check(layer, x, 0.3 * n)


@pytest.mark.parametrize("copies", [51, 52])
def test_plan_of_more_chunks_than_compute_units(oracle, copies):
    """Five assignments of each token: 255 chunks of 1024, whose items a block of its own plans, and 260, where the first chunk's does. All
    copies of a token are the same bits, and those of a batch of one copy but for the sum's order, which the rows an expert decide: halves
    of 2^-11 in the activations, two products behind each other."""
    layer, x = layer_and_rows(oracle, "Q4_K", 1024, 33, 0)
    out = layer.forward(x.repeat(copies, 1)).view(copies, 1024, -1)
    assert torch.equal(out, out[:1].expand_as(out))
    assert synth.errors(out[0].cpu().numpy(), layer.forward(x).cpu().numpy())[1] < 2 * 2.0 ** -11
