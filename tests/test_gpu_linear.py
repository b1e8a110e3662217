"""GPU parity of the linear in one library call (quantization method `apply`, mi355_block_fp8_linear): bit for bit the
stand-alone quantizer followed by the GEMM, whichever of the two the shape takes."""
import pytest
import torch

from tests import helpers as H

pytestmark = pytest.mark.gpu


def _composed(x, wq, ws, out_dtype):
    from lightllm_amd.quantization import per_token_group_quant_fp8, w8a8_block_fp8_matmul

    xq, xs = per_token_group_quant_fp8(x, 128)
    out = torch.full((x.shape[0], wq.shape[0]), float("nan"), dtype=out_dtype, device=x.device)
    return w8a8_block_fp8_matmul(xq, wq.t(), xs, ws.t(), out, [128, 128])


# one shape per kernel that quantizes in its stream (256 compute units): per-unit stream of 1..5 row blocks, the last one
# ragged; 64-row tiles with one K step per wave; 16-row tiles whole and with K shared, a K that the waves do not share
# evenly, a last tile of 8 rows and an N that is not a multiple of 8
SHAPES = [(4096, 4096), (4090, 2176), (7168, 2304), (12288, 2048), (16300, 2048), (20480, 2304), (28672, 512),
          (2112, 7168), (6144, 1024), (1004, 640), (72, 128)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,K", SHAPES)
def test_quantized_in_the_stream(hip, N, K, dtype):
    from lightllm_amd import _lib
    from lightllm_amd.quantization import QUANTMETHODS, WeightPack

    wq, ws = H.quantized_weights(N, K, seed=N + K, device="cuda")
    method, pack = QUANTMETHODS.get("fp8w8a8-b128"), WeightPack(wq, ws)
    for M in (1, 3, 4, 5, 8, 9):
        print(f"linear M={M} N={N} K={K} {dtype}", flush=True)
        fused = hip.mi355_block_fp8_linear_fused(M, N, K, _lib.DTYPE_CODES[dtype])
        assert fused == (M <= 8), (M, fused)
        x = H.activations(M, K, seed=M, outliers=True).to(dtype).cuda()
        x[M // 2, :128] = 0.0                       # a group on the eps floor
        if M > 1:
            x[M - 1, K - 3] = float("nan")          # a poisoned group stays in its row
        out = method.apply(x, pack)
        want = _composed(x, wq, ws, dtype)
        assert out.dtype == dtype and out.shape == (M, N)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), (M, N, K)
        assert not torch.isnan(out[: max(M - 1, 1)]).any()


# 64-row tiles with K whole over more steps than the stream stages activation scales for, K a multiple of 4096: the starts of
# the tiles are turned, in the quantizing stream and behind the quantizer alike; the per-unit stream of five row blocks, where
# they are not
@pytest.mark.parametrize("M,N,K,variant", [(1, 16384, 12288, 3), (4, 16384, 12288, 3), (3, 16380, 16384, 3), (4, 19200, 16384, 11)])
def test_quantized_in_the_stream_on_a_long_k(hip, M, N, K, variant):
    from lightllm_amd import _lib
    from lightllm_amd.quantization import QUANTMETHODS, WeightPack

    print(f"linear M={M} N={N} K={K}", flush=True)
    assert hip.mi355_block_fp8_linear_fused(M, N, K, _lib.DTYPE_CODES[torch.bfloat16]) == 1
    assert hip.mi355_block_fp8_gemm_variant(M, N, K) == variant
    wq, ws = H.quantized_weights(N, K, seed=N + K, device="cuda")
    x = H.activations(M, K, seed=M, outliers=True).cuda()
    method, want = QUANTMETHODS.get("fp8w8a8-b128"), _composed(x, wq, ws, torch.bfloat16)
    assert torch.equal(method.apply(x, WeightPack(wq, ws)), want)
    # an output over the activations takes the two launches
    buf = torch.zeros(M * max(N, K), dtype=torch.bfloat16, device="cuda")
    mine = buf[: M * K].view(M, K).copy_(x)
    out = buf[: M * N].view(M, N)
    assert torch.equal(method.apply(mine, WeightPack(wq, ws), out=out), want)


def test_output_argument_and_odd_operands(hip):
    """A caller's output tensor is filled and returned; activations that are not 16-byte aligned, a strided weight scale
    and fp32 outputs keep the behaviour of the step-by-step path."""
    from lightllm_amd.quantization import QUANTMETHODS, WeightPack

    M, N, K = 3, 512, 1024
    wq, ws = H.quantized_weights(N, K, seed=3, device="cuda")
    method = QUANTMETHODS.get("fp8w8a8-b128")
    x = H.activations(M, K, seed=4).cuda()
    want = _composed(x, wq, ws, torch.bfloat16)
    out = torch.empty_like(want)
    assert method.apply(x, WeightPack(wq, ws), out=out) is out and torch.equal(out, want)
    wide = torch.zeros((ws.shape[0], 2 * ws.shape[1]), dtype=torch.float32, device="cuda")
    wide[:, ::2] = ws
    assert torch.equal(method.apply(x, WeightPack(wq, wide[:, ::2])), want)
    buf = torch.empty(M * K + 1, dtype=torch.bfloat16, device="cuda")
    shifted = buf[1:].view(M, K).copy_(x)
    with pytest.raises(ValueError):                 # the quantizer needs 16-byte aligned activations
        method.apply(shifted, WeightPack(wq, ws))
    with pytest.raises(AssertionError):
        method.apply(x.float(), WeightPack(wq, ws))


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (4, 4096, 4096), (4, 6144, 4096), (8, 2048, 4096)])
def test_output_over_the_activations(hip, M, N, K):
    """An output that shares memory with the activations (whole, or its rows behind a part of them) holds what a separate one does."""
    from lightllm_amd.quantization import QUANTMETHODS, WeightPack

    wq, ws = H.quantized_weights(N, K, seed=N + K, device="cuda")
    x = H.activations(M, K, seed=M).cuda()
    want = _composed(x, wq, ws, torch.bfloat16)
    for shift in (0, 64):
        buf = torch.zeros(M * max(N, K) + shift, dtype=torch.bfloat16, device="cuda")
        mine = buf[: M * K].view(M, K).copy_(x)
        out = buf[shift: shift + M * N].view(M, N)
        assert QUANTMETHODS.get("fp8w8a8-b128").apply(mine, WeightPack(wq, ws), out=out) is out
        assert torch.equal(out, want), shift


@pytest.mark.parametrize("M", [2, 40])
def test_output_of_a_tensor_subclass(hip, M):
    """Activations of a tensor subclass give a plain tensor, as an output allocated by torch.empty is."""
    from lightllm_amd.quantization import QUANTMETHODS, WeightPack

    class Tagged(torch.Tensor):
        pass

    wq, ws = H.quantized_weights(512, 1024, seed=3, device="cuda")
    x = H.activations(M, 1024, seed=4).cuda()
    method, pack = QUANTMETHODS.get("fp8w8a8-b128"), WeightPack(wq, ws)
    for mine in (x.as_subclass(Tagged), torch.nn.Parameter(x, requires_grad=False)):
        out = method.apply(mine, pack)
        assert type(out) is torch.Tensor and torch.equal(out, method.apply(x, pack))
