"""CPU checks of the drop-in boundary: the library loads and exports every symbol the header declares, the
ctypes table covers the header, the Python functions keep the reference's signatures, and argument checks
fire before any launch."""
import inspect
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header_symbols():
    text = open(os.path.join(ROOT, "include", "mi355_fp8.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mi355_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from lightllm_amd import _lib

    lib = _lib.lib()
    names = _header_symbols()
    assert len(names) >= 11
    for n in names:
        assert hasattr(lib, n), f"{n} declared in the header but not exported"
    assert sorted(_lib.SIGNATURES) == names, "ctypes table and header disagree"


def test_error_strings():
    from lightllm_amd import _lib

    lib = _lib.lib()
    assert lib.mi355_error_string(0) == b"ok"
    for code in range(-6, 0):
        assert lib.mi355_error_string(code) not in (b"ok", b"unknown error code")
    assert lib.mi355_error_string(-99) == b"unknown error code"


def test_pure_host_entry_points():
    from lightllm_amd import _lib

    lib = _lib.lib()
    # rows of the schedule table: min(pairs, ceil((pairs + E*(bm-1))/bm))   (reference test_moe_align2)
    assert lib.mi355_moe_align2_rows(100, 4, 16) == 10
    assert lib.mi355_moe_align2_rows(8, 10, 16) == 8
    assert lib.mi355_grouped_block_m(32768, 256, 4096, 7168) == 256
    assert lib.mi355_grouped_block_m(32768, 256, 4096, 7168 + 128) == 256   # any K/128 takes the 256-row blocks
    assert lib.mi355_grouped_block_m(64, 256, 4096, 7168) == 16
    # 12..64 rows per expert: the two-queue launch of 256-row blocks where it has more tiles than compute units
    # (256 assumed without a device), the row-sized tiles otherwise
    assert lib.mi355_grouped_block_m(8192, 256, 4096, 7168) == 256
    assert lib.mi355_grouped_block_m(2048, 256, 4096, 7168) == 16
    assert lib.mi355_grouped_block_m(16 * 24, 16, 4096, 7168) == 32
    assert lib.mi355_grouped_block_m(16 * 50, 16, 4096, 8192) == 64
    assert lib.mi355_grouped_block_m(64 * 50, 64, 1024, 7168) == 64
    assert lib.mi355_grouped_block_m(64 * 50, 64, 2816, 2048) == 128
    # 8 experts: 64-row blocks from 9 rows per expert; few tiles or a small launch with a short K: 128-row blocks
    assert lib.mi355_grouped_block_m(8 * 24, 8, 4096, 7168) == 64
    assert lib.mi355_grouped_block_m(8 * 50, 8, 4096, 14336) == 128
    assert lib.mi355_grouped_block_m(128 * 64, 128, 2048, 768) == 128
    assert lib.mi355_grouped_block_m(128 * 300, 128, 2048, 768) == 256
    # an expert's N under 4096: the two-queue launch from 25 rows per expert
    assert lib.mi355_grouped_block_m(128 * 16, 128, 3072, 4096) == 16
    assert lib.mi355_grouped_block_m(128 * 32, 128, 3072, 4096) == 256
    assert lib.mi355_block_fp8_gemm_workspace_bytes(4096, 4096, 4096, 0) == 65536  # large M: tile counters only
    assert lib.mi355_block_fp8_gemm_workspace_bytes(32, 4096, 14336, 0) > 65536   # the stream shares K
    assert lib.mi355_block_fp8_gemm_workspace_bytes(8, 4096, 14336, 0) == 0        # one share per unit, whole K


def test_preconditions_are_checked_before_launch():
    """Null pointers and bad shapes are rejected on the host; nothing reaches the (absent) GPU."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    assert lib.mi355_group_quant_fp8(None, 0, None, None, 4, 100, 128, 1e-10, 1, 1, None) == -2   # K % 128
    assert lib.mi355_group_quant_fp8(None, 0, None, None, 4, 256, 0, 1e-10, 4, 1, None) == -1     # group <= 0
    assert lib.mi355_group_quant_fp8(None, 0, None, None, 4, 256, 96, 1e-10, 4, 1, None) == -2    # K % group
    assert lib.mi355_group_quant_fp8(None, 0, None, None, 4, 256, 128, 1e-10, 2, 1, None) == -1   # null
    assert lib.mi355_group_quant_fp8(None, 0, None, None, 0, 256, 128, 1e-10, 2, 1, None) == 0    # empty
    # other block sizes: only the plain kernel (AUTO or GENERIC) takes them
    assert lib.mi355_block_fp8_gemm(None, None, None, None, None, 4, 4, 128, 128, 1, 128, 4, 1, 1, 1, 1, 64, 128,
                                    None, 0, 2, None) == -6
    assert lib.mi355_block_fp8_gemm(None, None, None, None, None, 4, 4, 128, 128, 1, 128, 4, 1, 1, 1, 1, 64, 128,
                                    None, 0, 0, None) == -1
    assert lib.mi355_block_fp8_gemm(None, None, None, None, None, 4, 4, 128, 128, 1, 128, 4, 1, 1, 1, 1, 0, 128,
                                    None, 0, 0, None) == -1
    assert lib.mi355_block_fp8_gemm(None, None, None, None, None, 4, 4, 128, 128, 1, 128, 4, 1, 1, 1, 1, 128, 128,
                                    None, 0, 0, None) == -1
    assert lib.mi355_block_fp8_gemm(None, None, None, None, None, 0, 4, 128, 128, 1, 128, 4, 1, 1, 1, 1, 128, 128,
                                    None, 0, 0, None) == 0
    assert lib.mi355_block_weight_quant_fp8(None, 7, None, None, 4, 4, 128, None) == -1
    assert lib.mi355_moe_align2(None, 0, 16, 4, None, None) == -1


def test_grouped_block_m_holds_under_uneven_routing():
    """The row blocks around the lines between the weight streams and the launches whose time does not depend on how the
    rows are spread: rows per expert -> block, per (experts, N, K)."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    expect = {
        (256, 4096, 7168): {8: 16, 12: 16, 13: 256, 16: 256, 20: 256}, (256, 7168, 2048): {11: 16, 12: 256, 16: 256},
        (128, 4096, 7168): {16: 16, 17: 256}, (128, 7168, 2048): {11: 16, 12: 256},
        (32, 4096, 7168): {16: 16, 20: 32, 21: 256}, (64, 7168, 2048): {15: 16, 16: 256}, (32, 7168, 2048): {16: 16, 17: 256},
        (128, 4096, 1536): {11: 16, 12: 256}, (128, 3072, 4096): {16: 16, 24: 32, 25: 256},
        (8, 28672, 4096): {12: 16, 20: 32, 21: 64}, (8, 4096, 14336): {12: 16, 13: 64, 20: 64}, (8, 2048, 4096): {20: 32, 21: 64},
        (8, 7168, 1024): {8: 16, 9: 64}, (128, 1536, 2048): {8: 16, 9: 32, 24: 32, 25: 256}, (128, 2048, 768): {9: 16, 16: 16},
    }
    got = {s: {a: lib.mi355_grouped_block_m(a * s[0], *s) for a in e} for s, e in expect.items()}
    assert got == expect, {s: (got[s], expect[s]) for s in expect if got[s] != expect[s]}


def test_grouped_block_m_of_launches_too_small_for_the_weight_streams():
    """Where the 64-column tiles of the streams are too few, or a step costs two row blocks and nothing pays for it, the
    rows go to ring tiles, in blocks of the average size and with the lines those have."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    expect = {
        (16, 1024, 3072): {8: 16, 12: 16, 16: 16, 20: 32}, (32, 1536, 2048): {9: 16, 16: 16, 17: 32},
        (64, 4096, 5120): {16: 16, 17: 256}, (64, 2048, 2048): {9: 32, 16: 32, 20: 32},
        (16, 1536, 4096): {16: 16, 24: 32},
    }
    got = {s: {a: lib.mi355_grouped_block_m(a * s[0], *s) for a in e} for s, e in expect.items()}
    assert got == expect, {s: (got[s], expect[s]) for s in expect if got[s] != expect[s]}


def test_grouped_gemm_takes_schedules_of_up_to_2_31_tiles():
    """The limit is the launch's own tile count, in 128-column tiles for every block size: a schedule whose 64-column
    tiles would pass 2^31 is refused by the weight streams alone, and runs as ring tiles (the addresses are made up)."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    a = 1 << 40

    def call(block_m, rows, n, k):
        return lib.mi355_grouped_block_fp8_gemm(a, a, a, a, a, a, a, a, rows, block_m, 1024, 1024, 8, 1, n, k, 0, a, None, 0, None)

    for block_m in (16, 32, 64, 128, 256):
        for k in (1024, 2048):
            assert call(block_m, 1 << 20, 1 << 18, k) == -6, (block_m, k)   # 2^31 tiles of 128 columns
            if not torch.cuda.is_available():   # past the check: the launch itself is what fails here
                assert call(block_m, 700000, 1 << 18, k) == -5, (block_m, k)


def test_linear_that_quantizes_in_its_stream_refuses_an_output_over_its_activations():
    """Without room for quantized activations every workgroup reads x while others store C: an overlap of the two is
    refused before any launch (no memory is touched; the addresses are made up)."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    x, w, ws, room = 1 << 40, 1 << 41, 1 << 42, 1 << 43

    def call(c, m, n, k, ldc):
        return lib.mi355_block_fp8_linear(x, 0, w, ws, c, m, n, k, k, k // 128, 1, ldc, None, None, room, 1 << 30, 0, None)

    for m, n, k, ldc in [(1, 4096, 4096, 4096), (4, 4096, 4096, 4096), (8, 2048, 4096, 2048), (4, 2112, 7168, 4096)]:
        assert lib.mi355_block_fp8_linear_fused(m, n, k, 0) == 1
        x_bytes, c_bytes = 2 * m * k, 2 * ((m - 1) * ldc + n)
        for c in (x, x + 64, x + x_bytes - 16, x - c_bytes + 16):
            assert call(c, m, n, k, ldc) == -1, (m, n, k, c - x)
        if not torch.cuda.is_available():   # past the check: the launch itself is what fails here
            for c in (x + x_bytes, x - c_bytes):
                assert call(c, m, n, k, ldc) == -5, (m, n, k, c - x)


REFERENCE_SIGNATURES = {
    # (module, function): signature string of the reference's function of the same name
    ("lightllm_amd.quantization.fp8act_quant_kernel", "per_token_group_quant_fp8"):
        "(x, group_size, eps=1e-10, dtype=torch.float8_e4m3fn, column_major_scales=False, scale_tma_aligned=False, alloc_func=torch.empty)",
    ("lightllm_amd.quantization.fp8act_quant_kernel", "lightllm_per_token_group_quant_fp8"):
        "(x, group_size, x_q, x_s, eps=1e-10, dtype=torch.float8_e4m3fn)",
    ("lightllm_amd.quantization.fp8w8a8_block_gemm_kernel", "w8a8_block_fp8_matmul"):
        "(A, B, Ascale, Bscale, C, block_size, dtype=torch.bfloat16, run_config=None)",
    ("lightllm_amd.quantization.fp8w8a8_block_quant_kernel", "weight_quant"): "(x, block_size=128)",
    ("lightllm_amd.quantization.fp8w8a8_block_quant_kernel", "mm_weight_quant"): "(x, block_size=128)",
    ("lightllm_amd.fused_moe.grouped_fused_moe", "moe_align_fused"):
        "(expert_to_token_index, expert_to_weight, expert_token_num, topk_ids, topk_weights)",
    ("lightllm_amd.fused_moe.grouped_fused_moe", "moe_align2"): "(token_num_mul_topk_num, exports_token_num, block_m)",
    ("lightllm_amd.fused_moe.grouped_fused_moe", "grouped_matmul"):
        "(token_num_mul_topk_num, token_inputs, token_input_scale, expert_to_token_num, expert_to_token_index, "
        "expert_to_weights, expert_weights, expert_to_weights_scale, topk_num, out, mul_routed_weight, use_fp8_w8a8, "
        "alloc_tensor_func=torch.empty, reused_mblock_infos=None, run_config=None, bias=None)",
    ("lightllm_amd.fused_moe.grouped_fused_moe", "fused_experts_impl"):
        "(hidden_states, w1, w2, topk_weights, topk_ids, inplace=False, use_fp8_w8a8=False, use_int8_w8a16=False, "
        "w1_bias=None, w2_bias=None, w1_scale=None, w2_scale=None, a1_scale=None, a2_scale=None, "
        "alloc_tensor_func=torch.empty, run_config=None, layout=blocked, limit=None, alpha=None)",
    ("lightllm_amd.fused_moe.grouped_fused_moe", "inplace_fused_experts_impl"):
        "(hidden_states, w1, w2, topk_weights, topk_ids, use_fp8_w8a8=False, use_int8_w8a16=False, w1_bias=None, "
        "w2_bias=None, w1_scale=None, w2_scale=None, a1_scale=None, a2_scale=None, layout=blocked, alpha=None, limit=None)",
    ("lightllm_amd.fused_moe.grouped_fused_moe", "outplace_fused_experts_impl"):
        "(hidden_states, w1, w2, topk_weights, topk_ids, use_fp8_w8a8=False, use_int8_w8a16=False, w1_bias=None, "
        "w2_bias=None, w1_scale=None, w2_scale=None, a1_scale=None, a2_scale=None, layout=blocked, alpha=None, limit=None)",
    ("lightllm_amd.fused_moe.grouped_fused_moe", "fused_experts"):
        "(hidden_states, w1, w2, topk_weights, topk_ids, inplace=False, use_fp8_w8a8=False, use_int8_w8a16=False, "
        "w1_scale=None, w2_scale=None, a1_scale=None, a2_scale=None, w1_bias=None, w2_bias=None, layout=blocked, "
        "alpha=None, limit=None)",
}


def _sig_string(fn):
    parts = []
    for p in inspect.signature(fn).parameters.values():
        if p.default is inspect._empty:
            parts.append(p.name)
        else:
            d = p.default
            if d is torch.empty:
                d = "torch.empty"
            elif isinstance(d, torch.dtype):
                d = str(d)
            parts.append(f"{p.name}={d}")
    return "(" + ", ".join(parts) + ")"


@pytest.mark.parametrize("key", sorted(REFERENCE_SIGNATURES))
def test_python_signatures_match_the_reference(key):
    import importlib

    mod, name = key
    fn = getattr(importlib.import_module(mod), name)
    assert _sig_string(fn) == REFERENCE_SIGNATURES[key]


def test_quantization_method_surface():
    """The plug-in object exposes what LightLLM's MMWeightTpl calls (quantize_method.py:25-149, w8a8.py:418-533)."""
    from lightllm_amd.quantization import QUANTMETHODS, QuantizationMethod, WeightPack

    cls = type(QUANTMETHODS.get("fp8w8a8-b128"))
    assert issubclass(cls, QuantizationMethod)
    assert type(QUANTMETHODS.get("fp8w8a8-b128-triton", platform="cuda")) is cls
    assert QUANTMETHODS.get("fp8w8a8-b128") is not QUANTMETHODS.get("fp8w8a8-b128")   # a fresh object per lookup
    with pytest.raises(ValueError):
        QUANTMETHODS.get("no-such-method")
    with pytest.raises(ValueError):
        QUANTMETHODS.get("fp8w8a8-b128", platform="musa")
    apply_sig = list(inspect.signature(cls.apply).parameters)
    assert apply_sig == ["self", "input_tensor", "weight_pack", "out", "workspace", "use_custom_tensor_mananger", "bias"]
    for meth in ("quantize", "create_weight", "create_moe_weight", "load_weight", "load_weight_scale",
                 "load_weight_zero_point", "_create_weight", "_split_weight_pack", "_check_weight_need_quanted"):
        assert callable(getattr(cls, meth))
    m = cls()
    assert m.block_size == 128 and m.weight_scale_suffix == "weight_scale_inv" and m.has_weight_scale
    assert m.method_name.startswith("fp8w8a8-b128")
    pack = WeightPack(weight=torch.zeros((2, 4, 4)), weight_scale=torch.ones((2, 1, 1)))
    assert pack.load_ok == [False, False, True]
    sub = pack.get_expert(1)
    assert sub.weight.shape == (4, 4) and sub.weight_scale.shape == (1, 1) and sub.weight_zero_point is None
    # fused weights are split as views along dim -2, scales in units of 128 rows
    big = WeightPack(weight=torch.zeros((384, 256)), weight_scale=torch.zeros((3, 2)))
    parts = m._split_weight_pack(big, [256, 128], -2, [2, 1], -2)
    assert [p.weight.shape[0] for p in parts] == [256, 128] and [p.weight_scale.shape[0] for p in parts] == [2, 1]
    assert parts[1].weight.data_ptr() == big.weight[256:].data_ptr()


def test_operators_refuse_cpu_tensors():
    """No CPU fallback: the operators raise instead of computing on the host."""
    from lightllm_amd._lib import Mi355Error
    from lightllm_amd.quantization import per_token_group_quant_fp8

    with pytest.raises(Mi355Error):
        per_token_group_quant_fp8(torch.zeros((2, 128), dtype=torch.bfloat16), 128)


def test_shape_table_choices_on_256_compute_units():
    """The shape -> kernel table for the model linears it was measured on, planned for 256 compute units with
    room for every workspace.  A change of a rule that moves one of these shapes shows here."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    T256, T128, SKINNY, GENERIC, T256x128, STREAMK, XSHARE, ROWS, CU, ROWSM = 1, 2, 3, 4, 5, 8, 9, 10, 11, 12
    expect = {
        (4096, 36864, 7168): T256, (4096, 2112, 7168): T256, (2048, 24576, 1536): T256, (256, 36864, 7168): T256,
        (512, 36864, 7168): T256,                       # launched as a full round plus a second launch for the rest
        (1, 28672, 4096): SKINNY, (8, 4096, 14336): CU, (16, 14336, 4096): CU, (1, 7168, 8192): SKINNY, (64, 4096, 14336): SKINNY, (8, 36864, 7168): SKINNY,
        (64, 128256, 4096): XSHARE, (64, 8192, 8192): SKINNY, (64, 16384, 7168): SKINNY,   # 512 / 256 workgroups
        (64, 14336, 4096): ROWS, (48, 10240, 8192): ROWS, (64, 6144, 4096): SKINNY,
        (16, 7168, 18432): CU, (32, 18432, 7168): ROWS, (32, 28672, 4096): SKINNY, (8, 7168, 18432): CU,
        (16, 36864, 4096): ROWS, (24, 36864, 7168): ROWS, (64, 28672, 4096): ROWS, (100, 7168, 18432): ROWS, (128, 24576, 1536): ROWS,
        (128, 2112, 7168): ROWS, (200, 4096, 14336): ROWS, (384, 4096, 14336): ROWS,
        (192, 36864, 7168): ROWS, (176, 28672, 4096): ROWS, (224, 28672, 4096): T128,   # narrower workgroups up to 208 rows
        (300, 28672, 4096): T256, (512, 4096, 4096): ROWSM, (2048, 4096, 4096): ROWSM, (1024, 1024, 4096): ROWSM,
        (3072, 4096, 4096): T256, (1024, 6144, 4096): T128, (1024, 4096, 8192): STREAMK,   # more than 8 row blocks, a wider N, a longer K
        (300, 36864, 7168): T256,                       # likewise: a full round and the rest
        (512, 7168, 18432): STREAMK, (2048, 4096, 14336): STREAMK, (1024, 7168, 18432): STREAMK,
        (2048, 2112, 7168): ROWSM, (512, 4096, 14336): STREAMK,     # the panel split
        (240, 7168, 18432): STREAMK, (352, 7168, 18432): STREAMK, (300, 7168, 18432): ROWS,
        (768, 2112, 7168): ROWSM, (768, 2112, 8192): T256x128, (600, 5120, 6144): T256x128, (512, 5120, 5120): ROWSM, (1024, 2112, 7168): ROWSM, (512, 4096, 7168): STREAMK,
        (384, 16384, 4096): T128, (512, 16384, 7168): STREAMK, (300, 10240, 8192): ROWS, (384, 10240, 4096): T128,
        (512, 1536, 7168): T128, (4096, 7168, 256): T128, (1024, 512, 7168): T128, (256, 4096, 4096): T128,
        (16, 256, 100): GENERIC,
    }
    got = {shape: lib.mi355_block_fp8_gemm_plan(*shape, 1 << 32, 256) for shape in expect}
    assert got == expect, {k: (got[k], expect[k]) for k in expect if got[k] != expect[k]}


def test_shape_table_at_17_to_64_rows():
    """Large weights on either side of the lines between the three weight streams (planned for 256 compute units): each shape
    was timed on both kernels and runs on the one that is ahead."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    SKINNY, XSHARE, ROWS = 3, 9, 10
    expect = {
        # one round of wide tiles against a third or a second, nearly empty one of 64-row tiles
        (46, 20992, 8576): ROWS, (47, 55680, 10240): ROWS, (46, 50069, 2688): ROWS, (51, 18816, 2688): ROWS, (33, 21312, 11264): ROWS,
        (39, 18096, 8192): ROWS, (22, 51200, 20480): ROWS, (30, 36864, 7168): ROWS,
        (40, 15360, 5120): SKINNY, (41, 19168, 2176): SKINNY, (33, 8192, 8192): SKINNY, (56, 12288, 4096): SKINNY, (24, 45504, 4096): SKINNY,
        (60, 16000, 4992): SKINNY, (48, 28672, 4096): SKINNY, (20, 40960, 4096): SKINNY,
        # the same under few K steps, whatever the weights' size
        (40, 30208, 512): ROWS, (19, 48128, 256): ROWS, (62, 36583, 384): ROWS, (46, 26624, 128): ROWS, (34, 79616, 256): XSHARE, (30, 12000, 512): SKINNY,
        # more than five rounds of 64-row tiles; turned starts
        (40, 116480, 1280): XSHARE, (46, 86144, 12672): XSHARE, (38, 66176, 7424): SKINNY, (43, 105664, 4096): SKINNY,
    }
    got = {shape: lib.mi355_block_fp8_gemm_plan(*shape, 1 << 32, 256) for shape in expect}
    assert got == expect, {k: (got[k], expect[k]) for k in expect if got[k] != expect[k]}


def test_launched_kernel_query():
    """What AUTO launches where the table's activation-block stream covers more than one kernel: the streaming kernel at 65..128
    rows (not without its workspace where it shares K), tiles over M at 209..352; the plan's code everywhere else."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    ROWS, ROWSM, STREAM = 10, 12, 13
    for shape, ws_bytes, want in [((72, 4096, 4096), 1 << 30, STREAM), ((96, 7168, 2048), 1 << 30, STREAM), ((96, 2112, 7168), 1 << 30, STREAM),
                                  ((128, 2112, 7168), 1 << 30, ROWS), ((128, 36864, 7168), 1 << 30, ROWS), ((64, 14336, 4096), 1 << 30, ROWS),
                                  ((333, 27648, 5120), 0, ROWSM), ((209, 12288, 2048), 0, ROWSM), ((300, 4096, 14336), 1 << 30, ROWS)]:
        assert lib.mi355_block_fp8_gemm_launched(*shape, ws_bytes, 256) == want, shape
    seen = set()
    for m, n, k in _sweep_shapes(5, 3000):
        for ws_bytes in (0, 65536 + (8 << 20), 1 << 34):
            plan, v = (f(m, n, k, ws_bytes, 0) for f in (lib.mi355_block_fp8_gemm_plan, lib.mi355_block_fp8_gemm_launched))
            assert v == plan or (plan == ROWS and (v == STREAM and 65 <= m <= 128 or v == ROWSM and 209 <= m <= 352)), (m, n, k, plan, v)
            assert v != STREAM or lib.mi355_block_fp8_gemm_workspace_bytes(m, n, k, v) <= min(ws_bytes, 65536 + (8 << 20)), (m, n, k)
            seen.add(v)
    assert {ROWS, ROWSM, STREAM} <= seen


def test_over_m_query():
    """Tiles over M instead of the table's kernel: only from 80 rows on, on either side of the lines as timed."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    for shape, want in [((300, 4096, 4096), 1), ((340, 6144, 4096), 1), ((1700, 5120, 13824), 1), ((2500, 4096, 4096), 1),
                        ((380, 24576, 1536), 1), ((512, 4096, 4096), 1), ((333, 27648, 5120), 1), ((4096, 36864, 7168), 0),
                        ((1024, 7168, 18432), 0), ((640, 7168, 18432), 0), ((4096, 4096, 4096), 0), ((208, 4096, 4096), 1),
                        ((118, 5744, 1792), 1), ((79, 5744, 1792), 0), ((128, 24576, 1536), 0), ((5000, 4096, 4096), 0), ((300, 512, 4096), 0), ((300, 4096, 896), 0), ((300, 4096, 4096 + 64), 0)]:
        assert lib.mi355_block_fp8_gemm_over_m(*shape, 1 << 34, 256) == want, shape
    assert lib.mi355_block_fp8_gemm_over_m(300, 4096, 4096, 1 << 34, 64) == 0
    for m, n, k in _sweep_shapes(6, 2000):
        for ws_bytes in (0, 1 << 34):
            over = lib.mi355_block_fp8_gemm_over_m(m, n, k, ws_bytes, 256)
            if lib.mi355_block_fp8_gemm_launched(m, n, k, ws_bytes, 256) == 12:
                assert over == 1
            elif m < 80 or m > 4096:
                assert over == 0, (m, n, k)


def test_over_m_query_where_k_is_shared():
    """With the weights from HBM a step of few row blocks waits for its weight rows, so a kernel that shares K keeps these (us, over M
    / here: 566 x 640 x 6400 21.4 / 17.2, 250 x 2800 x 5504 23.8 / 19.2, 266 x 2112 x 7168 25.6 / 22.6, 929 x 1408 x 9216 36.4 / 33.3)."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    for shape, want in [((566, 640, 6400), 0), ((250, 2800, 5504), 0), ((266, 2112, 7168), 0), ((140, 912, 6144), 0), ((929, 1408, 9216), 0),
                        ((302, 4608, 7680), 0), ((300, 4096, 4096), 1), ((281, 3926, 2432), 1), ((184, 4464, 2560), 1)]:
        assert lib.mi355_block_fp8_gemm_over_m(*shape, 1 << 34, 256) == want, shape


def test_over_m_query_without_a_workspace():
    """A kernel that shares K runs it whole where its partial sums have no room, and is compared as that (us, K whole / over M: 300 x
    1024 x 18432 147 / 59, 768 x 2112 x 8192 104 / 34)."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    for shape in [(300, 1024, 18432), (202, 705, 18816), (768, 2112, 8192), (124, 15460, 14592)]:
        over = [lib.mi355_block_fp8_gemm_over_m(*shape, ws_bytes, 256) for ws_bytes in (0, 65536, 65536 + (8 << 20), 1 << 26, 1 << 34)]
        assert over == [1, 1, 1, 0, 0], (shape, over)


def test_tiles_over_m_ask_for_no_workspace():
    """An AUTO call that runs as tiles over M asks for none of the workspace of the kernel they stand in for (600 x 2560 x 8192: the
    128 MiB of stream-K), and runs as that without it."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    for shape in [(600, 2560, 8192), (1024, 2112, 8192), (300, 4096, 4096), (2500, 4096, 4096), (118, 5744, 1792)]:
        assert lib.mi355_block_fp8_gemm_workspace_bytes(*shape, 0) == 0, shape
    for m, n, k in _sweep_shapes(7, 2000):
        over = [lib.mi355_block_fp8_gemm_over_m(m, n, k, ws_bytes, 0) for ws_bytes in (0, 1 << 34)]
        need = lib.mi355_block_fp8_gemm_workspace_bytes(m, n, k, 0)
        assert need > 0 or not over[1] or over[0], (m, n, k)
        assert lib.mi355_block_fp8_gemm_over_m(m, n, k, need, 0) == over[1], (m, n, k)


_T256, _T128, _SKINNY, _GENERIC, _T256x128, _STREAMK, _XSHARE, _ROWS, _CU, _ROWSM = 1, 2, 3, 4, 5, 8, 9, 10, 11, 12


def _sweep_shapes(seed: int, count: int):
    import random

    rnd = random.Random(seed)
    model = [(28672, 4096), (4096, 14336), (36864, 7168), (7168, 18432), (2112, 7168), (24576, 1536), (6144, 4096),
             (5120, 13824), (128256, 4096), (10240, 8192), (7168, 2048), (4096, 7168), (1536, 7168), (512, 7168)]
    for _ in range(count):
        if rnd.random() < 0.6:
            n, k = rnd.choice(model)
        else:
            n, k = rnd.randrange(1, 400) * 64, rnd.randrange(1, 150) * 128
        m = rnd.choice([rnd.randrange(1, 65), rnd.randrange(65, 130), rnd.randrange(129, 385), rnd.randrange(385, 8193)])
        yield m, n, k


def test_auto_never_fails_for_want_of_a_workspace():
    """Whatever the table picks, an AUTO call without a workspace - or with the fixed scratch of the entry point
    that allocates nothing - ends in a kernel whose plan needs none (or no more than that): the ROWS128 band
    129 <= M <= 384 under a long K used to fall through to a stream-K plan that then reported MI355_EWORKSPACE."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    scratch = _lib.WS_COUNTER_BYTES + (8 << 20)
    # the shapes of the report, then a seeded sweep; cus = 0 plans for the current device, whose count
    # mi355_block_fp8_gemm_workspace_bytes uses as well
    shapes = [(200, 7168, 18432), (256, 4096, 14336), (300, 4096, 14336), (384, 4096, 14336), (320, 5120, 13824),
              (128, 7168, 18432), (8, 4096, 14336), (64, 28672, 4096), (512, 7168, 18432)]
    shapes += list(_sweep_shapes(11, 4000))
    optional = (_T256, _T128, _T256x128, _XSHARE, _GENERIC, _CU, _ROWSM)   # run unsplit / one workgroup per tile without one
    for ws_bytes in (0, scratch):
        for m, n, k in shapes:
            v = lib.mi355_block_fp8_gemm_plan(m, n, k, ws_bytes, 0)
            assert v in (_T256, _T128, _SKINNY, _GENERIC, _T256x128, _STREAMK, _XSHARE, _ROWS, _CU, _ROWSM), (m, n, k, v)
            if v not in optional:
                need = lib.mi355_block_fp8_gemm_workspace_bytes(m, n, k, v)
                assert need <= ws_bytes, (m, n, k, v, need, ws_bytes)
    # with room for everything the plan is the table's own choice
    for m, n, k in shapes[:200]:
        assert lib.mi355_block_fp8_gemm_plan(m, n, k, 1 << 34, 0) == lib.mi355_block_fp8_gemm_variant(m, n, k)


def test_no_stream_k_without_its_workspace():
    """Where the table shares K between 256x256 tiles and the workspace of that is missing (none, or the fixed scratch), the
    choice is the table's without stream-K: a few 256x256 tiles by themselves leave most of the device idle (us, 256x256 / here
    without a workspace: 175 x 6112 x 5888 65.0 / 49.2, 2831 x 176 x 8448 87.5 / 68.9, 204 x 9600 x 7424 80.3 / 62.4)."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    T256, T128, ROWS = 1, 2, 10
    for ws_bytes in (0, _lib.WS_COUNTER_BYTES + (8 << 20)):
        for shape, want in [((175, 6112, 5888), T128), ((204, 9600, 7424), T128), ((2831, 176, 8448), T128), ((4966, 16, 7552), T128),
                            ((1621, 528, 7296), T128), ((208, 10080, 7680), T128), ((3877, 240, 9472), T128), ((204, 31744, 5888), ROWS),
                            ((2048, 4096, 14336), T256)]:
            assert lib.mi355_block_fp8_gemm_plan(*shape, ws_bytes, 256) == want, (shape, ws_bytes)


def test_panel_split_on_a_narrow_n():
    """From 257 rows on the panel split of K is taken only where it is ahead of the 128x128 tiles with K shared (us, panel / 128x128:
    517 x 611 x 12288 31.6 / 21.2, 1058 x 128 x 23168 31.5 / 18.3, 1392 x 528 x 10112 33.9 / 29.1, 403 x 1232 x 32128 40.1 / 51.5)."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    T128, STREAMK = 2, 8
    for shape, want in [((517, 611, 12288), T128), ((1058, 128, 23168), T128), ((1392, 528, 10112), T128), ((787, 912, 7936), T128),
                        ((1457, 224, 24448), T128), ((1772, 3760, 27392), STREAMK), ((403, 1232, 32128), STREAMK), ((474, 1280, 28160), STREAMK),
                        ((462, 1840, 9344), T128), ((640, 7168, 18432), STREAMK), ((1024, 2560, 14336), STREAMK)]:
        assert lib.mi355_block_fp8_gemm_plan(*shape, 1 << 34, 256) == want, shape


def test_panel_split_at_201_to_256_rows():
    """One m tile on a large weight: the panel split of K takes over from the activation-block stream only where it has eight runs
    and more (us, panel / stream: 204 x 32336 x 6144 84.2 / 61.2, 211 x 9152 x 11520 61.3 / 44.9)."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    ROWS, STREAMK = 10, 8
    for shape, want in [((203, 31072, 5760), ROWS), ((211, 9152, 11520), ROWS), ((204, 32336, 6144), ROWS), ((203, 16000, 7040), ROWS),
                        ((240, 7168, 18432), STREAMK), ((256, 7168, 14336), STREAMK), ((200, 7168, 18432), ROWS)]:
        assert lib.mi355_block_fp8_gemm_plan(*shape, 1 << 34, 256) == want, shape


@pytest.mark.parametrize("cus", [8, 64, 128, 304])
def test_shape_table_off_256_compute_units(cus):
    """The table's thresholds are all relative to the compute-unit count but were measured at 256.  On other counts
    (a partitioned device, another bin) its rules must still hold together: every shape gets a kernel that exists,
    the weight-streaming kernels keep to their row limits, and a compute-bound shape with whole rounds of
    256 x 256 tiles gets those tiles."""
    from lightllm_amd import _lib

    lib = _lib.lib()
    for m, n, k in _sweep_shapes(cus, 3000):
        for ws_bytes in (0, 1 << 34):
            v = lib.mi355_block_fp8_gemm_plan(m, n, k, ws_bytes, cus)
            assert v in (_T256, _T128, _SKINNY, _T256x128, _STREAMK, _XSHARE, _ROWS, _CU, _ROWSM), (m, n, k, v)
            if v == _ROWSM:
                assert m > 384 and k <= 7168, (m, n, k, v)
            if v == _CU:
                assert m <= 16, (m, n, k, v)
            if v in (_SKINNY, _XSHARE):
                assert m <= 64, (m, n, k, v)
            if v == _ROWS:
                assert 16 <= m <= 384, (m, n, k, v)
            if v in (_T256, _STREAMK, _T256x128, _ROWSM):
                assert m > 64, (m, n, k, v)
            if m <= 64:
                assert v in (_SKINNY, _XSHARE, _ROWS, _T128, _CU), (m, n, k, v)
    # whole rounds of 256 x 256 tiles, K long enough to be compute-bound: the ping-pong tiles on every count
    rounds = 4
    n = 256 * max(cus // 8, 1)
    assert lib.mi355_block_fp8_gemm_plan(256 * 8 * rounds, n, 7168, 1 << 34, cus) == _T256
    # decode rows stream the weights on every count
    assert lib.mi355_block_fp8_gemm_plan(1, 28672, 4096, 1 << 34, cus) == _SKINNY
    assert lib.mi355_block_fp8_gemm_plan(8, 4096, 14336, 0, cus) in (_SKINNY, _T128, _CU)


def test_streaming_kernel_by_name_without_a_workspace():
    """The weight stream asked for by name at 17..64 rows runs K whole where its plan would share K and the workspace is missing
    (refused only where the launch would gain by sharing: a narrow N under a long K), and takes every N a plan of 64-row tiles has
    counters for (no memory is touched; the addresses are made up)."""
    from lightllm_amd import _lib

    if torch.cuda.is_available():
        pytest.skip("made-up addresses: only where a launch fails for want of a device")
    lib = _lib.lib()

    def call(m, n, k, ws_bytes):
        return lib.mi355_block_fp8_gemm(1 << 40, 2 << 40, 3 << 40, 4 << 40, 5 << 40, m, n, k, k, 1, k, n, k // 128, 1, 1, k // 128,
                                        128, 128, (6 << 40) if ws_bytes else None, ws_bytes, 3, None)

    for m, n, k in [(36, 25337, 22656), (49, 26940, 29824), (27, 31681, 35200), (36, 9509, 3840), (64, 530000, 7808),
                    (17, 12288, 20608), (40, 20000, 38400)]:
        for ws_bytes in (0, 1 << 34):
            assert call(m, n, k, ws_bytes) == -5, (m, n, k, ws_bytes)   # past every check: the launch itself fails here
    for m, n, k in [(32, 4096, 14336), (64, 2112, 7168)]:
        assert call(m, n, k, 0) == -4 and call(m, n, k, 1 << 34) == -5


def test_linear_call_is_the_c_entry():
    """The CPython entry of the one-call linear passes its integers (None: a null pointer) to the C entry as ctypes does and
    refuses anything else."""
    from lightllm_amd import _lib

    lib, call = _lib.lib(), _lib.linear_call()
    good = [64, 0, 64, 64, 64, 1, 128, 128, 128, 1, 1, 128, None, None, None, 0, 0, None]
    for place, value in [(0, None), (2, None), (4, 0), (5, -1), (6, -5), (7, 100), (8, 64), (11, 127), (16, 1), (16, 7), (5, 0), (6, 0)]:
        args = list(good)
        args[place] = value
        assert call(*args) == lib.mi355_block_fp8_linear(*args), (place, value)
    assert call((1 << 64) - 64, 0, None, 64, 64, 1, 128, 128, 128, 1, 1, 128, None, None, None, 0, 0, None) == -1
    for bad in (good[:-1], good + [0], [1.5] + good[1:], ["x"] + good[1:]):
        with pytest.raises(TypeError):
            call(*bad)
    with pytest.raises(OverflowError):
        call(1 << 64, *good[1:])


@pytest.mark.parametrize("with_entry", [True, False])
def test_linear_call_of_a_copied_package(tmp_path, with_entry):
    """A built package that was copied elsewhere calls the linear of its own library, the only one that is mapped; without
    the CPython entry beside it (not built for this interpreter) it does so through ctypes."""
    import shutil
    import subprocess
    import sys

    from lightllm_amd import _lib

    if with_entry and not os.path.exists(_lib.CALL_PATH):
        pytest.skip("the CPython entry is not built for this interpreter")
    skip = shutil.ignore_patterns("obj", "csrc", "__pycache__", *([] if with_entry else ["_mi355call*"]))
    shutil.copytree(os.path.join(ROOT, "lightllm_amd"), tmp_path / "lightllm_amd", ignore=skip)
    code = """
from lightllm_amd import _lib
call = _lib.linear_call()
args = [64, 0, 64, 64, 64, 1, 128, 128, 64, 1, 1, 128, None, None, None, 0, 0, None]
print(call(*args) == _lib.lib().mi355_block_fp8_linear(*args) == -2)
for name in sorted({line.split()[-1] for line in open("/proc/self/maps") if "mi355" in line}):
    print(name)
"""
    run = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, capture_output=True, text=True, timeout=300,
                         env={**os.environ, "PYTHONPATH": str(tmp_path)})
    assert run.returncode == 0, run.stderr[-2000:]
    lib_dir = str(tmp_path / "lightllm_amd" / "lib")
    want = [os.path.join(lib_dir, os.path.basename(p)) for p in ([_lib.CALL_PATH] if with_entry else []) + [_lib.LIB_PATH]]
    assert run.stdout.split("\n")[:-1] == ["True"] + want
