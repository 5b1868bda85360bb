"""Host-side checks that need no GPU: the C-ABI library loads and exports every entry point include/tqmoe.h declares, the
pure-host entry points (sizes, layouts) answer, bad arguments and a missing device are reported through the error
record (there is no CPU path to fall back to), the C++ adapter header compiles, and the product never touches the oracle."""
import ctypes as C
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "tqmoe.h")


@pytest.fixture(scope="module")
def tq():
    import tqllm_amd
    return tqllm_amd


def declared_functions():
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    return sorted(set(re.findall(r"\b(tqmoe_[a-z0-9_]+)\s*\(", text)))


def test_every_declared_entry_point_is_exported(tq):
    names = declared_functions()
    assert len(names) >= 24 and "tqmoe_layer_forward" in names and "tqmoe_expert_gemm_i8" in names
    lib = tq.lib()
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing
    assert tq.abi_version() == 2      # with the tile-major planes of Q4_K, Q6_K, IQ3_S and NVFP4G banks


def test_host_only_entry_points(tq):
    lib = tq.lib()
    code, aux = C.c_size_t(), C.c_size_t()
    err = tq.api._err()
    # IQ4_XS: 16 B of codes per 32 weights, 8 B per 256; rows in tiles of 32
    assert lib.tqmoe_bank_layout(tq.IQ4_XS, 64, 2048, C.byref(code), C.byref(aux), C.byref(err)) == 0
    assert (code.value, aux.value) == (64 * 2048 // 2, 64 * 2048 // 256 * 8)
    assert lib.tqmoe_bank_layout(tq.IQ3_S, 10, 512, C.byref(code), C.byref(aux), C.byref(err)) == 0
    assert (code.value, aux.value) == (10 * 16 * 12, 10 * 2 * 16)
    assert lib.tqmoe_bank_layout(tq.NVFP4G, 10, 256, C.byref(code), C.byref(aux), C.byref(err)) == 0
    assert code.value == 10 * 128 and aux.value == 160 + 40
    assert lib.tqmoe_bank_layout(tq.Q4_K, 10, 100, C.byref(code), C.byref(aux), C.byref(err)) == -1   # cols not a multiple of 256
    assert b"tqmoe_bank_layout" in err.message
    assert lib.tqmoe_bank_layout(7, 10, 256, C.byref(code), C.byref(aux), C.byref(err)) == -2         # unknown format
    assert lib.tqmoe_act_image_bytes(3, 2048) == 3 * 64 * 72
    assert lib.tqmoe_act_image_bytes(3, 100) == 0
    assert lib.tqmoe_dispatch_workspace_bytes(512, 4096, 10) > 0


def test_bank_format_ids_and_layouts_agree(tq):
    """Every bank format of the header's enum has the same GGUF type id in the Python mirror and in the oracle, the same GGUF
    block size in both, and a device layout whose code and aux sizes follow the header's description."""
    import oracle
    text = open(HEADER).read()
    ids = {m.group(1): int(m.group(2)) for m in re.finditer(r"TQMOE_((?:I?Q\d\w*)|NVFP4G)\s*=\s*(\d+)", text)}
    assert len(ids) == 16 and ids["IQ4_XS"] == 23 and ids["NVFP4G"] == 323
    # bytes per 32 weights of the code plane, and of the aux plane per 256 weights (NVFP4G: per 16 weights a byte, plus 4 per row)
    code_per_sub = {"IQ4_XS": 16, "Q4_K": 16, "Q5_K": 16, "IQ4_NL": 16, "Q4_0": 16, "NVFP4G": 16, "IQ3_S": 12, "IQ3_XXS": 12, "IQ2_S": 12,
                    "IQ2_XS": 12, "Q3_K": 12, "IQ2_XXS": 8, "Q2_K": 8, "IQ1_S": 8, "Q6_K": 24, "Q8_0": 32}
    aux_per_256 = {"IQ4_XS": 8, "Q5_K": 48, "Q6_K": 32, "Q3_K": 32, "Q2_K": 32}
    lib = tq.lib()
    for name, tid in ids.items():
        assert getattr(tq, name) == tid and getattr(oracle, name) == tid, name
        assert tq.api.BLOCK[tid] == oracle.BLOCK[tid], name
        code, aux = C.c_size_t(), C.c_size_t()
        err = tq.api._err()
        rows, cols = 64, 1024
        assert lib.tqmoe_bank_layout(tid, rows, cols, C.byref(code), C.byref(aux), C.byref(err)) == 0, name
        assert code.value == rows * cols // 32 * code_per_sub[name], name
        want_aux = rows * cols // 16 + rows * 4 if name == "NVFP4G" else rows * cols // 256 * aux_per_256.get(name, 16)
        assert aux.value == want_aux, name


def test_errors_are_reported_not_swallowed(tq):
    lib = tq.lib()
    err = tq.api._err()
    # bad shape: reported before any device work
    assert lib.tqmoe_topk(None, None, None, None, 8, 2, 1, 1.0, None, C.byref(err)) == -1
    assert err.code == -1 and err.message
    # err may be NULL
    assert lib.tqmoe_topk(None, None, None, None, 8, 2, 1, 1.0, None, None) == -1
    # a short error struct is left alone
    short = tq.api._Error(8, 0, b"")
    assert lib.tqmoe_topk(None, None, None, None, 8, 2, 1, 1.0, None, C.byref(short)) == -1 and short.code == 0


def test_no_device_is_an_error_not_a_fallback(tq):
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    lib = tq.lib()
    err = tq.api._err()
    buf = (C.c_float * 64)()
    ids = (C.c_int32 * 4)()
    rc = lib.tqmoe_topk(buf, ids, buf, None, 8, 2, 1, 1.0, None, C.byref(err))
    assert rc == -3 and b"no CPU path" in err.message


def fake_layer(tq, hidden, ff, experts, topk, shared, fmt, down=None):
    """A descriptor whose pointers are never read: for the answers that come before any device work."""
    bank = lambda f, rows, cols: tq.api._Bank(C.sizeof(tq.api._Bank), f, experts + int(shared), rows, cols, 4096, 4096)
    return tq.api._Layer(C.sizeof(tq.api._Layer), hidden, ff, experts, topk, int(shared), ff if shared else 0, 1.0, 4096, 4096, tq.BF16, bank(fmt, ff, hidden),
                         bank(fmt, ff, hidden), bank(down or fmt, hidden, ff), 1, 0, None, 0, 0.0, 0)


@pytest.mark.parametrize("fmt", ["IQ4_XS", "Q4_K", "Q5_K", "NVFP4G", "IQ2_S"])
def test_grouped_products_refuse_more_than_4096_experts(tq, fmt):
    """4096 routed experts and a shared one are 4097 lists, one more than the dispatch takes: the layer refuses the batches that
    need the lists before anything is enqueued, and takes the small ones (which here end at the missing workspace)."""
    lib, err = tq.lib(), tq.api._err()
    run = lambda d, n: lib.tqmoe_layer_forward(C.byref(d), 4096, tq.BF16, n, 4096, tq.F32, None, None, None, None, 0, None, C.byref(err))
    over, most = (fake_layer(tq, 512, 256, experts, 8, True, getattr(tq, fmt)) for experts in (4096, 4095))
    assert run(over, 2000) == -1 and b"4096 experts" in err.message
    assert run(over, 4) == -4 and run(most, 2000) == -4


@pytest.mark.parametrize("hidden,ff,experts,topk,shared", [(2048, 512, 512, 10, True), (1024, 768, 64, 1, False), (2048, 768, 33, 1, False), (256, 2048, 512, 4, False),
                                                           (4096, 768, 128, 1, True), (3072, 256, 4095, 2, False)])
def test_workspace_of_the_largest_batch_is_enough_for_every_smaller_one(tq, hidden, ff, experts, topk, shared):
    """An engine asks for the workspace once, for its largest batch; other products and items take over at lines below it."""
    bytes_for = tq.lib().tqmoe_layer_workspace_bytes
    for fmt, down in (("IQ4_XS", None), ("Q4_K", "Q6_K"), ("Q6_K", None), ("IQ3_S", None), ("NVFP4G", None), ("NVFP4G", "Q6_K"), ("Q5_K", None), ("IQ2_S", None)):
        for act_blocks in (0, 1, 2):
            d = fake_layer(tq, hidden, ff, experts, topk, shared, getattr(tq, fmt), getattr(tq, down) if down else None)
            d.act_blocks = act_blocks
            sizes = [bytes_for(C.byref(d), n) for n in list(range(1, 4200)) + [8192, 50000]]
            assert sizes[0] > 0 and sizes == sorted(sizes), (fmt, down, act_blocks)


def test_planes_that_are_not_aligned_take_the_general_products(tq):
    """The fp8 products move 16-byte pieces to LDS: a layer whose planes start elsewhere runs on the fp16 products."""
    d = fake_layer(tq, 512, 256, 16, 4, False, tq.NVFP4G)
    assert tq.lib().tqmoe_layer_path(C.byref(d), 500) == 3
    for bank in (d.gate, d.up, d.down):
        for plane in ("codes", "aux"):
            setattr(bank, plane, 4104)
            assert tq.lib().tqmoe_layer_path(C.byref(d), 500) == 2
            setattr(bank, plane, 4096)


def test_adapter_header_compiles(tmp_path):
    src = tmp_path / "use.cpp"
    src.write_text('#include "tqmoe_adapter.hpp"\n'
                   "int main() { tqmoe_error e = tqmoe_hip::fresh(); (void)e; return tqmoe_hip::ExpertFormat::has_expert_matvec() ? 0 : 1; }\n")
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-fsyntax-only", "-I", os.path.join(ROOT, "include"), str(src)])
    # the override mixin against a base class that restates the reference's expert virtuals (tests/adapter_check.cpp): a
    # signature that does not match the base fails to compile there; the GPU test runs the program
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-fsyntax-only", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                           "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "adapter_check.cpp")])
    # the C header alone is plain C
    csrc = tmp_path / "use.c"
    csrc.write_text('#include "tqmoe.h"\nint main(void) { return (int)sizeof(tqmoe_layer) == 0; }\n')
    subprocess.check_call(["gcc", "-std=c99", "-Wall", "-Wextra", "-Werror", "-fsyntax-only", "-I", os.path.join(ROOT, "include"), str(csrc)])


def test_product_does_not_use_the_oracle():
    pkg = os.path.join(ROOT, "tqllm_amd")
    for base, _, files in os.walk(pkg):
        if os.path.basename(base) == "build":
            continue
        for f in files:
            if f.endswith((".py", ".hip", ".cuh", ".h", ".hpp")):
                text = open(os.path.join(base, f), errors="replace").read()
                assert "oracle" not in text.lower(), os.path.join(base, f)
