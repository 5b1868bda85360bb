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
