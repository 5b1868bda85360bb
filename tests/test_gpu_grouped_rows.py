"""The grouped products on prepared rows inside the layer, at the row counts where items and row tiles begin and end: fp16
(IQ4_XS, Q4_K, Q6_K, IQ3_S) against the fp32 oracle, NVFP4G against the oracle of its E4M3 operands."""
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
@pytest.mark.parametrize("n,hidden,ff,shared_ff", [(32, 256, 256, 0), (33, 512, 256, 256), (64, 256, 512, 256), (65, 1280, 256, 0), (128, 256, 768, 512),
                                                  (129, 512, 512, 512), (700, 768, 512, 0)])
def test_layer_on_prepared_rows(tq, oracle, fmt, n, hidden, ff, shared_ff):
    """Two of the seven experts take every token (their lists hold exactly n rows), and the shared one where there is one; the
    largest batch is routed freely."""
    cfg = dict(hidden=hidden, ff=ff, experts=7, topk=2, shared_ff=shared_ff, wtype=getattr(oracle, fmt), rtype="f32", xtype="f32")
    raws = synth.make_banks(cfg, seed=n + hidden)
    gate, up, down = banks_on_device(cfg, raws)
    inp = synth.make_inputs(cfg, n, seed=n)
    x, router = (np.array(inp[k][1], dtype=np.float32) for k in ("x", "router"))
    if n < 700:
        x[:, 0] = 4.0
        router[:, 0] = [0, 3, 0, 0, 4, 0, 0]
    layer = tq.MoeLayer(torch.from_numpy(router).cuda(), dev(inp["shared_gate"]) if shared_ff else None, gate, up, down, 2, shared_ff=shared_ff)
    fp8 = fmt == "NVFP4G"
    assert layer.path(n) == ("grouped_fp8" if fp8 else "grouped_f16")
    out, ids, w, logits = (t.cpu().numpy() for t in layer.forward(torch.from_numpy(x).cuda(), return_routing=True))
    want, want_ids, _ = oracle.layer_forward(x, logits, *raws, cfg["wtype"], hidden, ff, 7, 2, shared_ff=shared_ff, act_mode=2 if fp8 else 0, threads=16)
    clear = clear_tokens(oracle, logits, 7, 2, ids, want_ids)
    assert n == 700 or (np.bincount(ids.reshape(-1), minlength=7) == [0, n, 0, 0, n, 0, 0]).all()
    mx, rel = synth.errors(out[clear], want[clear])
    top = float(np.abs(want[clear]).max())     # E4M3's coarse steps amplify last-bit differences of the act rows
    assert mx < 1e-2 * (max(1.0, top) if fp8 else 1.0) and rel < (3e-3 if fp8 else 1e-3), (mx, rel)


@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q4_K", "Q6_K", "IQ3_S"])
@pytest.mark.parametrize("n,hidden,ff,shared_ff", [(86, 256, 256, 0), (97, 512, 256, 0), (90, 512, 512, 256), (128, 256, 768, 0), (129, 1280, 256, 0)])
def test_layer_on_items_of_64_rows(tq, oracle, fmt, n, hidden, ff, shared_ff):
    """24.5 to 37 rows an expert on average: items of one and two row tiles, the last ones of 22, 33, 26, 64 and one row."""
    test_layer_on_prepared_rows(tq, oracle, fmt, n, hidden, ff, shared_ff)


def one_row_tile_error(tq, oracle, fmt, shared_ff, n=32):
    """Error of a layer whose products are items of n rows and fewer, against float64 on the decoded weights."""
    cfg = dict(hidden=512, ff=512, experts=7, topk=2, shared_ff=shared_ff, wtype=getattr(oracle, fmt), rtype="f32", xtype="f32")
    raws = synth.make_banks(cfg, seed=51)
    inp = synth.make_inputs(cfg, n, seed=52)
    layer = tq.MoeLayer(dev(inp["router"]), dev(inp["shared_gate"]), *banks_on_device(cfg, raws), 2, shared_ff=shared_ff)
    assert layer.path(n) == "grouped_f16"
    out, ids, w, logits = (t.cpu().numpy() for t in layer.forward(dev(inp["x"]), return_routing=True))
    g, u, d = (oracle.dequantize(cfg["wtype"], raw, 8 * 512 * 512).reshape(8, 512, 512).astype(np.float64) for raw in raws)
    x = inp["x"][1].astype(np.float64)

    def expert(e, lim):
        a, b = x @ g[e, :lim].T, x @ u[e, :lim].T
        return a / (1 + np.exp(-a)) * b @ d[e, :, :lim].T

    rows = np.stack([expert(e, 512) for e in range(7)], axis=1)[np.arange(n)[:, None], ids]
    want = (rows * w[:, :, None]).sum(axis=1) + expert(7, shared_ff) / (1 + np.exp(-logits[:, 7:].astype(np.float64)))
    return synth.errors(out, want)[1]


@pytest.mark.parametrize("shared_ff", [128, 384, 512])
def test_iq3_s_items_of_one_row_tile(tq, oracle, shared_ff):
    """One row tile's sums take IQ3_S's super-block factor themselves, every fourth stage and after the last: lists of a few
    rows, the shared expert's of 32, its down product ending inside a super-block. Against float64 on the decoded weights: the
    operands of each product are rounded to fp16 (2^-12 of a term at most, the sums' errors average), the weights are not."""
    assert one_row_tile_error(tq, oracle, "IQ3_S", shared_ff) < 2.0 ** -11


@pytest.mark.parametrize("shared_ff", [128, 384, 512])
@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q6_K"])
def test_items_of_one_row_tile(tq, oracle, fmt, shared_ff):
    """The same with values times integer scales past fp16's eleven bits: rounded once (2^-12 of a term at most), as the input is."""
    assert one_row_tile_error(tq, oracle, fmt, shared_ff) < 2.0 ** -11


@pytest.mark.parametrize("shared_ff", [128, 512])
@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q6_K"])
def test_items_of_two_row_tiles(tq, oracle, fmt, shared_ff):
    """Items of up to 64 rows keep the factor outside too: the same bound."""
    assert one_row_tile_error(tq, oracle, fmt, shared_ff, n=100) < 2.0 ** -11


@pytest.mark.parametrize("fmt,n,shared_ff", [("Q4_K", 2048, 128), ("Q4_K", 2047, 256), ("Q6_K", 2048, 256), ("IQ3_S", 2048, 128)])
def test_down_rows_past_the_range_of_halves(tq, oracle, fmt, n, shared_ff):
    """Results past 65504, the largest half, before the weighted sum: down rows are fp32 but where the int8 products, whose rows
    are halves, would have taken the batch (Q4_K, 2048 tokens, whole super-blocks everywhere). Against float64 on the decoded weights."""
    cfg = dict(hidden=256, ff=256, experts=7, topk=2, shared_ff=shared_ff, wtype=getattr(oracle, fmt), rtype="f32", xtype="f32")
    raws = synth.make_banks(cfg, seed=11, sigma=0.5)
    inp = synth.make_inputs(cfg, n, seed=12)
    x = np.ascontiguousarray(inp["x"][1] * 6)
    layer = tq.MoeLayer(dev(inp["router"]), dev(inp["shared_gate"]), *banks_on_device(cfg, raws), 2, shared_ff=shared_ff)
    assert layer.path(n) == "grouped_f16"
    out, ids, w, logits = (t.cpu().numpy() for t in layer.forward(torch.from_numpy(x).cuda(), return_routing=True))
    g, u, d = (oracle.dequantize(cfg["wtype"], raw, 8 * 256 * 256).reshape(8, 256, 256).astype(np.float64) for raw in raws)

    def expert(e, rows, lim):
        a, b = rows @ g[e, :lim].T, rows @ u[e, :lim].T
        return a / (1 + np.exp(-np.clip(a, -700, 700))) * b @ d[e, :, :lim].T

    rows = np.stack([expert(e, x.astype(np.float64), 256) for e in range(7)], axis=1)[np.arange(n)[:, None], ids]
    want = (rows * w[:, :, None]).sum(axis=1) + expert(7, x.astype(np.float64), shared_ff) / (1 + np.exp(-logits[:, 7:].astype(np.float64)))
    assert np.abs(rows).max() > 65504 and np.isfinite(out).all()
    assert synth.errors(out, want)[1] < 1e-3


def test_rows_past_the_shared_expert_are_zero_whatever_the_bank_holds(tq, oracle):
    """The shared expert has 256 of the bank's 512 rows; the others are infinite in the gate bank and NaN in the up bank."""
    cfg = dict(hidden=256, ff=512, experts=3, topk=1, shared_ff=256, wtype=oracle.NVFP4G, rtype="f32", xtype="f32")
    raws = synth.make_banks(cfg, seed=21)
    inp = synth.make_inputs(cfg, 70, seed=22)
    x = dev(inp["x"])
    for raw, value in zip(raws[:2], (np.inf, np.nan)):
        elems, nbytes = oracle.BLOCK[cfg["wtype"]]
        raw.reshape(4, 512, 256 // elems, nbytes)[3, 256:, :, 0:4] = np.frombuffer(np.float32(value).tobytes(), np.uint8)
    gate, up, down = banks_on_device(cfg, raws)
    ids = tq.moe_extend_ids(torch.randint(0, 3, (70, 1), dtype=torch.int32, device="cuda"), 3)
    lists = tq.moe_dispatch(ids, 4)[:3]
    act = tq.expert_gemm_gateup_fp8(gate, up, *tq.gather_rows_i8(*tq.quant_rows_fp8(x), lists, 140, 2), lists, 70, 2, 1, 256).view(70, 2, 512)
    assert not act[:, 1, 256:].any() and torch.isfinite(act).all() and act[:, 1, :256].any()


@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q4_K", "NVFP4G"])
def test_layer_on_operands_that_are_not_aligned(tq, oracle, fmt):
    """Bank planes eight bytes, input rows one element and the workspace three bytes past a multiple of 16: the router's and the
    products' transfers to LDS need that multiple, and the kernels that load into registers take over."""
    cfg = dict(hidden=512, ff=256, experts=60, topk=4, shared_ff=0, wtype=getattr(oracle, fmt), rtype="bf16", xtype="bf16")
    raws = synth.make_banks(cfg, seed=31, distinct=4)
    banks = banks_on_device(cfg, raws)
    n = 3100                                     # 49 x 1 blocks of the router's kernel for large batches
    inp = synth.make_inputs(cfg, n, seed=32)
    x, router = dev(inp["x"]), dev(inp["router"])
    want, ids, _, logits = tq.MoeLayer(router, None, *banks, 4, act_blocks=2 if fmt == "IQ4_XS" else 0).forward(x, return_routing=True)

    def moved(t, elements):
        raw = torch.empty(t.numel() + 64, dtype=t.dtype, device="cuda")
        out = raw[elements:elements + t.numel()].view(t.shape)
        out.copy_(t)
        return out

    for b in banks:
        b.codes, b.aux = moved(b.codes.view(torch.uint8), 8), moved(b.aux.view(torch.uint8), 8)
    layer = tq.MoeLayer(moved(router, 1), None, *banks, 4, act_blocks=2 if fmt == "IQ4_XS" else 0)
    layer._ws = moved(layer.workspace(n), 3)
    out, ids2, _, logits2 = layer.forward(moved(x, 1), return_routing=True)
    assert torch.equal(logits, logits2) and torch.equal(ids, ids2)
    if fmt == "NVFP4G":      # the fp16 products in place of the fp8 ones: within their bar of fp32 activations
        assert layer.path(n) == "grouped_f16"
        out, want = out[:64], torch.from_numpy(oracle.layer_forward(inp["x"][1][:64], logits.cpu().numpy()[:64], *raws, cfg["wtype"], 512, 256, 60, 4, act_mode=0, threads=16)[0])
    assert synth.errors(out.cpu().numpy(), want.cpu().numpy())[1] < 1e-3


def test_fp8_products_refuse_operands_that_are_not_aligned(tq, oracle):
    cfg = dict(hidden=256, ff=256, experts=3, topk=1, shared_ff=0, wtype=oracle.NVFP4G, rtype="f32", xtype="f32")
    gate, up, down = banks_on_device(cfg, synth.make_banks(cfg, seed=41))
    lists = tq.moe_dispatch(torch.zeros((64, 1), dtype=torch.int32, device="cuda"), 3)[:3]
    q, s = tq.gather_rows_i8(*tq.quant_rows_fp8(torch.randn((64, 256), device="cuda")), lists, 64, 1)
    assert tq.expert_gemm_fp8(down, q, s, lists, 64, 1, 1).shape[0] == 64
    with pytest.raises(tq.TqmoeError, match="16 bytes"):
        tq.expert_gemm_fp8(down, torch.empty(q.numel() + 16, dtype=q.dtype, device="cuda")[8:8 + q.numel()].view(q.shape), s, lists, 64, 1, 1)
