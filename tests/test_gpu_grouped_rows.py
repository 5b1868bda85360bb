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
