"""Performance cases of the MoE layer, from one decoded token to an 8192-token prefill.

A case is one block of a model's forward pass: the whole layer (router, top-k, routed and shared experts, combine) called
through MoeLayer.forward on inputs that lie on the GPU, for one batch of tokens. `layers` > 1 stands for a decode step
through that many layers of a model, each with banks of its own, so that a small batch's weights come from HBM as they do
in a model and not from the last-level cache. With `residual` the call has the steps either side: add_rmsnorm in front, the
residual added to the result.

Keys of a case: gate (format of the gate and up banks), down (of the down bank), hidden, ff, experts, topk, shared (an
always-on shared expert of the same ff), tokens, layers, dtype (of the router and the activations), skew (Zipf(1.1) expert
popularity in place of balanced routing), gating, act_blocks (MoeLayer's), residual.
"""
import math

import numpy as np
import torch

import tqllm_amd as tq
from tqllm_amd.api import BLOCK

FORMATS = {"iq4_xs": tq.IQ4_XS, "q4_k": tq.Q4_K, "iq3_s": tq.IQ3_S, "nvfp4": tq.NVFP4G, "q6_k": tq.Q6_K}
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
GATINGS = {"softmax": tq.GATE_SOFTMAX, "sigmoid": tq.GATE_SIGMOID}
ZIPF_S = 1.1
MOST_FLOPS = 2.1e12          # of a drawn case: no more than the largest listed one
MOST_BANK_BYTES = 2.3e9      # of a drawn case's layer


def _case(**kw):
    c = dict(gate="iq4_xs", down="iq4_xs", hidden=2048, ff=512, experts=512, topk=10, shared=True, tokens=1, layers=1, dtype="bf16", skew=False,
             gating="softmax", act_blocks=0, residual=False)
    c.update(kw)
    return c


def listed():
    q4k = dict(gate="q4_k", down="q4_k", ff=768, experts=64, topk=8, shared=False, dtype="f32")
    iq3s = dict(gate="iq3_s", down="iq3_s", ff=768, experts=256, topk=8, shared=False)
    return [
        # one user's chat: a token at a time through eight layers of the 512-expert model
        _case(name="iq4_xs_t1", layers=8),
        # several users' tokens in one decode step, or a short speculative draft
        _case(name="iq4_xs_t16", tokens=16),
        # the tail of a prompt, or a prompt shorter than a chunk; popular experts, a ragged count of tokens
        _case(name="iq4_xs_t333_skewed", tokens=333, skew=True),
        # a full prefill chunk with the expert popularity that real text shows: the headline workload
        _case(name="iq4_xs_t4096_skewed", tokens=4096, skew=True),
        # prefill with a scale per 32 activations (the setting for models with outlier activations), balanced routing
        _case(name="iq4_xs_t1501_act_blocks", tokens=1501, act_blocks=1),
        # a smaller K-quant model with fp32 activations, one token and four layers
        _case(name="q4_k_t1", layers=4, **q4k),
        # the same, a long prompt
        _case(name="q4_k_t4096", tokens=4096, **q4k),
        # the usual K-quant mixture (down kept wider) of a model with sigmoid routing, a few users' tokens, an odd number of
        # experts; with the norm in front and the residual behind
        _case(name="q4_k_q6_k_t23_block", gate="q4_k", down="q6_k", ff=768, experts=125, topk=6, tokens=23, gating="sigmoid", residual=True),
        # a lattice format: a large decode batch of a busy server, and a short prompt
        _case(name="iq3_s_t64", tokens=64, **iq3s),
        _case(name="iq3_s_t512", tokens=512, **iq3s),
        # fp4 experts of a large model: a small batch, and the largest prefill chunk
        _case(name="nvfp4_t7", gate="nvfp4", down="nvfp4", hidden=3072, ff=1536, experts=256, topk=8, tokens=7),
        _case(name="nvfp4_t8192", gate="nvfp4", down="nvfp4", hidden=3072, ff=1536, experts=256, topk=8, tokens=8192),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    gate, down = rng.choice([("iq4_xs", "iq4_xs"), ("iq4_xs", "iq4_xs"), ("q4_k", "q4_k"), ("q4_k", "q6_k"), ("iq3_s", "iq3_s"), ("nvfp4", "nvfp4")])
    while True:
        c = _case(gate=gate, down=down, hidden=256 * rng.randint(4, 12), ff=256 * rng.randint(2, 6), experts=_log_int(rng, 60, 512), topk=rng.randint(4, 10),
                  shared=rng.random() < 0.5, tokens=_log_int(rng, 1, 8192), dtype="f32" if rng.random() < 0.2 else "bf16",
                  gating="sigmoid" if rng.random() < 0.25 else "softmax")
        c["residual"] = c["dtype"] == "bf16" and rng.random() < 0.3
        c["skew"] = c["tokens"] >= 64 and not c["residual"] and c["gating"] == "softmax" and rng.random() < 0.5
        c["act_blocks"] = 1 if c["tokens"] >= 256 and gate == down and gate != "nvfp4" and rng.random() < 0.2 else 0
        if work(c)["flops"] <= MOST_FLOPS and _bank_bytes(c) * _banks(c) <= MOST_BANK_BYTES:
            return c


def _banks(c):
    return c["experts"] + (1 if c["shared"] else 0)


def _bank_bytes(c):
    """Bytes of one expert's three matrices."""
    def per_weight(f):
        elems, nbytes = BLOCK[FORMATS[f]]
        return nbytes / elems
    return c["hidden"] * c["ff"] * (2 * per_weight(c["gate"]) + per_weight(c["down"]))


def _popularity(c):
    p = 1.0 / np.arange(1, c["experts"] + 1) ** ZIPF_S
    return p / p.sum()


def _distinct(c):
    """Expected number of routed experts that get a token."""
    e, k, t = c["experts"], c["topk"], c["tokens"]
    if not c["skew"]:
        return e * (1.0 - (1.0 - k / e) ** t)
    logits = np.random.default_rng(0).standard_normal((t, e), dtype=np.float32) + np.log(_popularity(c)).astype(np.float32)
    return len(np.unique(np.argpartition(-logits, k - 1, axis=1)[:, :k]))


def work(case):
    c = case
    size = 4 if c["dtype"] == "f32" else 2
    slots = c["topk"] + (1 if c["shared"] else 0)
    bank = (_distinct(c) + (1 if c["shared"] else 0)) * _bank_bytes(c)
    router = _banks(c) * c["hidden"] * size
    rows = c["tokens"] * c["hidden"]
    out = rows * (2 if c["residual"] else 4)
    extra = rows * 2 if c["residual"] else 0            # the residual rows, next to the normed ones
    flops = c["tokens"] * (slots * 6.0 * c["ff"] * c["hidden"] + 2.0 * _banks(c) * c["hidden"])
    return {"bytes": c["layers"] * (bank + router + rows * size + out + extra), "flops": c["layers"] * flops}


def tolerance(case):
    """The grouped products take 8-bit or fp16 operands: a requantised activation that falls on the other side of a rounding
    step, or a token whose last expert changes between two logits a rounding apart, is what two correct implementations
    differ by. The decode products take activations of fifteen bits, and sum in fp32."""
    few = case["tokens"] * (case["topk"] + 1) <= 3 * case["experts"] and case["tokens"] <= 64
    return {"rel": 3e-4, "max": 0.02} if few and not case["residual"] else {"rel": 1e-2, "max": 0.4}


def _blocks(fmt, rows, cols, gen):
    """GGUF blocks of [rows][cols]: random valid codes and sub-scales, block scales that give weights of about 0.02."""
    elems, nbytes = BLOCK[FORMATS[fmt]]
    n = rows * cols // elems
    raw = torch.empty((n, nbytes), dtype=torch.uint8, device="cuda")
    raw.view(-1)[: n * nbytes // 8 * 8].view(torch.int64).random_(-2 ** 63, None, generator=gen)

    def uniform(shape, lo, hi):
        return torch.rand(shape, device="cuda", generator=gen) * (hi - lo) + lo

    def halves(at, lo, hi, signed=False):
        d = uniform((n,), lo, hi)
        if signed:
            d = torch.where(torch.rand(n, device="cuda", generator=gen) < 0.5, -d, d)
        raw[:, at:at + 2] = d.to(torch.float16).view(torch.uint8).reshape(n, 2)

    if fmt == "iq4_xs":
        halves(0, 4e-5, 8e-5, signed=True)
    elif fmt == "iq3_s":
        halves(0, 1.5e-4, 3e-4, signed=True)
    elif fmt == "q4_k":
        halves(0, 1e-4, 2e-4)
        halves(2, 1e-4, 2e-4)
    elif fmt == "q6_k":
        halves(208, 1.5e-5, 3e-5, signed=True)
    elif fmt == "nvfp4":
        raw[:, 0:4] = uniform((rows,), 5e-4, 2.5e-3).repeat_interleave(cols // elems).view(torch.uint8).reshape(n, 4)
        raw[:, 4:12] = torch.randint(0x28, 0x58, (n, 8), dtype=torch.uint8, device="cuda", generator=gen)   # E4M3 0.125 .. 16
    return raw.reshape(-1)


def _layer(c, gen):
    h, f, e, banks = c["hidden"], c["ff"], c["experts"], _banks(c)
    dtype = DTYPES[c["dtype"]]
    trio = [tq.ExpertBank(FORMATS[fmt], _blocks(fmt, banks * rows, cols, gen), banks, rows, cols)
            for fmt, rows, cols in ((c["gate"], f, h), (c["gate"], f, h), (c["down"], h, f))]
    router = torch.randn((e, h), device="cuda", generator=gen) * h ** -0.5
    x = torch.randn((c["tokens"], h), device="cuda", generator=gen)
    if c["skew"]:      # the last activation of every token is 1 and carries the logarithm of the experts' popularity
        p = torch.from_numpy(np.log(_popularity(c)).astype(np.float32)).cuda()
        router[:, -1] = p[torch.randperm(e, device="cuda", generator=gen)]
        x[:, -1] = 1.0
    shared_gate = (torch.randn((h,), device="cuda", generator=gen) * 0.02).to(dtype) if c["shared"] else None
    bias = torch.rand((e,), device="cuda", generator=gen) * 0.1 if c["gating"] == "sigmoid" else None
    layer = tq.MoeLayer(router.to(dtype), shared_gate, *trio, c["topk"], shared_ff=f if c["shared"] else 0, gating=GATINGS[c["gating"]], probs_bias=bias,
                        act_blocks=c["act_blocks"])
    norm = 1.0 + 0.1 * torch.randn((h,), device="cuda", generator=gen) if c["residual"] else None
    return layer, x.to(dtype), norm


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return [_layer(case, gen) for _ in range(case["layers"])]


def run(state):
    outs = []
    for layer, x, norm in state:
        if norm is None:
            outs.append(layer.forward(x))
        else:
            outs.append(layer.forward(tq.add_rmsnorm(x, None, norm, 1e-6), residual=x))
    return outs
