"""GPU parity of the decode products of the tile-major formats where their split can go wrong: a row cut over waves into
equal and unequal shares (eleven super-blocks over eight, four and two waves), ragged last tiles (the row-wise kernels take them), batches that stage their input rows and that walk several (two, four)
row tiles a wave, more input rows of one expert than a block serves. Against float64 on the decoded weights."""
import numpy as np
import pytest
import torch

import synth
from gpu_util import dev

pytestmark = pytest.mark.gpu

FORMATS = {"iq4_xs": 23, "q4_k": 12, "q6_k": 14, "iq3_s": 21, "nvfp4": 323}
SHAPES = [(64, 1280, 1, 3), (96, 1536, 2, 3), (32, 1792, 1, 2), (40, 512, 5, 3), (33, 768, 14, 3), (1024, 512, 40, 4), (160, 2304, 13, 1),
          (64, 2816, 1, 3), (64, 2816, 6, 3), (320, 2816, 18, 4), (1024, 2816, 17, 4), (2048, 1792, 30, 2), (2048, 512, 80, 4), (2048, 256, 160, 3)]


@pytest.mark.parametrize("fmt", sorted(FORMATS))
@pytest.mark.parametrize("rows,cols,n,experts", SHAPES)
def test_decode_products(oracle, fmt, rows, cols, n, experts):
    import tqllm_amd as tq
    wtype = FORMATS[fmt]
    if fmt == "iq4_xs" and rows % 32:
        pytest.skip("IQ4_XS experts have whole tiles")
    rng = np.random.default_rng(rows + cols + n)
    k = min(2, experts)
    raw = oracle.quantize(wtype, (rng.standard_normal((experts * rows, cols)) * 0.02).astype(np.float32))
    bank = tq.ExpertBank(wtype, raw, experts, rows, cols)
    dec = oracle.dequantize(wtype, raw, experts * rows * cols).reshape(experts, rows, cols).astype(np.float64)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    xe = rng.standard_normal((n * k, cols)).astype(np.float32)
    ids = np.stack([rng.permutation(experts)[:k] for _ in range(n)]).astype(np.int32)
    two = tq.expert_matvec2(bank, bank, tq.quant_act(dev(x)), dev(ids))
    one = tq.expert_matvec(bank, tq.quant_act(dev(xe)), dev(ids), per_expert_input=True)
    torch.cuda.synchronize()
    assert torch.equal(two[0], two[1])
    for got, rows_in in ((two[0], np.repeat(x, k, axis=0)), (one, xe)):
        want = np.stack([dec[e] @ rows_in[a].astype(np.float64) for a, e in enumerate(ids.reshape(-1))])
        mx, rel = synth.errors(got.cpu().numpy(), want)
        assert rel < 2e-4 and mx < 1e-3, (mx, rel)


@pytest.mark.parametrize("fmt", sorted(FORMATS))
@pytest.mark.parametrize("assignments", [64, 65, 192, 193, 512, 513, 1024, 1025, 2048])
def test_rows_of_a_block_are_found_past_the_first_ids(oracle, fmt, assignments):
    """A block finds its expert's rows in 192 ids at once, or 512 at a time: an expert with four rows on both sides of id 512, one whose first row
    comes behind it, one with many, ids that are skipped, the last id of the most one launch takes."""
    import tqllm_amd as tq
    wtype, rows, cols, experts = FORMATS[fmt], 64, 256, 9
    rng = np.random.default_rng(assignments)
    raw = oracle.quantize(wtype, (rng.standard_normal((experts * rows, cols)) * 0.02).astype(np.float32))
    bank = tq.ExpertBank(wtype, raw, experts, rows, cols)
    dec = oracle.dequantize(wtype, raw, experts * rows * cols).reshape(experts, rows, cols).astype(np.float64)
    ids = rng.integers(0, 6, assignments).astype(np.int32)
    ids[rng.random(assignments) < 0.05] = -1
    ids[[i for i in (63, 505, 511, 512, 513, 1023, 1024) if i < assignments]] = 6       # its blocks: 63 .. 512, 513 .. 1024
    ids[[i for i in (514, 600, 1030) if i < assignments]] = 7
    ids[-1] = 8
    x = rng.standard_normal((assignments, cols)).astype(np.float32)
    image, dev_ids, live = tq.quant_act(dev(x)), dev(ids[:, None]), ids >= 0
    want = np.stack([dec[e] @ x[a].astype(np.float64) for a, e in enumerate(ids) if e >= 0])
    for got in (*tq.expert_matvec2(bank, bank, image, dev_ids), tq.expert_matvec(bank, image, dev_ids)):
        mx, rel = synth.errors(got.cpu().numpy().reshape(assignments, rows)[live], want)
        assert rel < 2e-4 and mx < 1e-3, (mx, rel)
