"""The fp8w8a8-b128 quantization method on the gfx950 kernels.

Mirrors FP8w8a8B128QuantizationMethod / FP8w8a8B128TritonQuantizationMethod of the reference
(lightllm/common/quantization/w8a8.py:418-474, 505-533): 128x128 block-quantized e4m3fn weights with
``weight_scale_inv`` scales, dynamic per-token-group activation quantization, bf16 output, no bias.
"""
import functools
from typing import Callable, List, Optional, Tuple, Union

import torch

from .. import _lib
from .fp8act_quant_kernel import per_token_group_quant_fp8
from .fp8w8a8_block_gemm_kernel import w8a8_block_fp8_matmul
from .fp8w8a8_block_quant_kernel import weight_quant
from .quantize_method import QuantizationMethod, WeightPack
from .registry import QUANTMETHODS


@functools.lru_cache(maxsize=4096)
def _linear_plan(rows: int, n: int, k: int, dtype: torch.dtype, device_index: int) -> Tuple[bool, int]:
    """(quantized inside the GEMM's kernel, workspace bytes) of a linear: what the library says for the device."""
    lib, code = _lib.lib(), _lib.DTYPE_CODES[dtype]
    return (bool(lib.mi355_block_fp8_linear_fused(rows, n, k, code)),
            lib.mi355_block_fp8_linear_workspace_bytes(rows, n, k, code))


class FP8w8a8B128QuantizationMethod(QuantizationMethod):
    """``cache_manager`` may be any object with ``empty(shape, dtype=, device=)`` (LightLLM's g_cache_manager);
    without one, outputs come from torch.empty."""

    def __init__(self, cache_manager=None):
        super().__init__()
        self.cache_manager = cache_manager
        self.block_size = 128
        self.weight_scale_suffix = "weight_scale_inv"
        self.has_weight_scale = True
        self.has_weight_zero_point = False

    def quantize(self, weight: torch.Tensor, output: WeightPack) -> None:
        device = output.weight.device
        qweight, scale = weight_quant(weight.cuda(device).contiguous(), self.block_size)
        output.weight.copy_(qweight)
        output.weight_scale.copy_(scale)

    def _alloc_func(self, use_custom_tensor_mananger: bool) -> Callable:
        if use_custom_tensor_mananger and self.cache_manager is not None:
            return self.cache_manager.empty
        return torch.empty

    def _dynamic_quant_input(
        self,
        input_tensor: torch.Tensor,
        weight_pack: WeightPack,
        out: Optional[torch.Tensor] = None,
        use_custom_tensor_mananger: bool = True,
    ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
        """The five GEMM operands in the order of `w8a8_block_fp8_matmul`: quantized activations, the [K, N] view
        of the weight (strides (1, K)), activation scales, the [K/128, N/128] view of the weight scales, and the
        output (allocated here unless the caller brings one)."""
        alloc = self._alloc_func(use_custom_tensor_mananger)
        w_kn, ws_kn = weight_pack.weight.t(), weight_pack.weight_scale.t()
        x_q, x_s = per_token_group_quant_fp8(input_tensor, self.block_size, dtype=w_kn.dtype, alloc_func=alloc)
        if out is None:
            rows, cols = input_tensor.shape[0], w_kn.shape[1]
            out = alloc((rows, cols), dtype=input_tensor.dtype, device=input_tensor.device)
        return x_q, w_kn, x_s, ws_kn, out

    def _create_weight(
        self, out_dims: Union[int, List[int]], in_dim: int, dtype: torch.dtype, device_id: int, num_experts: int = 1
    ) -> Tuple[WeightPack, List[WeightPack]]:
        """One e4m3fn [sum(out_dims), in_dim] weight with its [.. // 128, .. // 128] fp32 scales (a leading expert
        axis when num_experts > 1), and one view pair per fused sub-weight, cut along the output rows."""
        b = self.block_size
        parts = list(out_dims) if isinstance(out_dims, (list, tuple)) else [out_dims]
        rows = sum(parts)
        lead = (num_experts,) if num_experts > 1 else ()
        device = torch.device("cuda", device_id)

        def storage(r: int, c: int, dt: torch.dtype) -> torch.Tensor:
            return torch.empty(lead + (r, c), dtype=dt, device=device)

        fused = WeightPack(
            weight=storage(rows, in_dim, torch.float8_e4m3fn),
            weight_scale=storage(rows // b, in_dim // b, torch.float32),
        )
        views = self._split_weight_pack(
            fused,
            weight_out_dims=parts,
            weight_split_dim=-2,
            weight_scale_out_dims=[p // b for p in parts],
            weight_scale_split_dim=-2,
        )
        return fused, views


@QUANTMETHODS.register(["fp8w8a8-b128-mi355", "fp8w8a8-b128-triton", "fp8w8a8-b128"], platform="cuda")
class FP8w8a8B128Mi355QuantizationMethod(FP8w8a8B128QuantizationMethod):
    def apply(
        self,
        input_tensor: torch.Tensor,
        weight_pack: WeightPack,
        out: Optional[torch.Tensor] = None,
        workspace: Optional[torch.Tensor] = None,
        use_custom_tensor_mananger: bool = True,
        bias: Optional[torch.Tensor] = None,
    ) -> torch.Tensor:
        assert bias is None, f"Bias addition is not supported in {self.method_name} for now"
        result = self._linear(input_tensor, weight_pack, out, use_custom_tensor_mananger)
        if result is not None:
            return result
        qinput_tensor, qweight, input_scale, weight_scale, out = self._dynamic_quant_input(
            input_tensor, weight_pack, out, use_custom_tensor_mananger
        )
        w8a8_block_fp8_matmul(
            qinput_tensor, qweight, input_scale, weight_scale, out, (self.block_size, self.block_size),
            dtype=input_tensor.dtype,
        )
        return out

    def _linear(self, x: torch.Tensor, weight_pack: WeightPack, out: Optional[torch.Tensor],
                use_custom_tensor_mananger: bool) -> Optional[torch.Tensor]:
        """The linear in one library call: packed 16-bit activations and outputs, a packed weight.  Anything else (and
        anything that is wrong) returns None and goes step by step, where every operator checks its own operands."""
        w, ws = weight_pack.weight, weight_pack.weight_scale
        dtype = x.dtype
        if (dtype is not torch.bfloat16 and dtype is not torch.float16) or x.ndim != 2 or w.ndim != 2 or ws.ndim != 2:
            return None
        (m, k), (n, wk) = x.shape, w.shape
        if k != wk or m == 0 or n == 0 or k % 128 != 0 or ws.shape != ((n + 127) // 128, k // 128):
            return None
        if not (x.is_cuda and w.is_cuda and ws.is_cuda and x.is_contiguous() and w.is_contiguous()
                and w.dtype is torch.float8_e4m3fn and ws.dtype is torch.float32):
            return None
        device = x.device
        alloc = self._alloc_func(use_custom_tensor_mananger)
        if out is None and alloc is torch.empty and type(x) is torch.Tensor:  # (a subclass would hand its type on)
            out, out_dtype = x.new_empty((m, n)), dtype
        else:
            if out is None:
                out = alloc((m, n), dtype=dtype, device=device)
            out_dtype = out.dtype
            if out.shape != (m, n) or not out.is_cuda or not out.is_contiguous() or out_dtype not in (torch.bfloat16, torch.float16):
                return None
        x_ptr, w_ptr = x.data_ptr(), w.data_ptr()
        if (x_ptr | w_ptr) & 15:
            return None
        fused, ws_need = _linear_plan(m, n, k, dtype, device.index)
        out_ptr = out.data_ptr()
        if fused and x_ptr < out_ptr + 2 * m * n and out_ptr < x_ptr + 2 * m * k:
            fused = False  # every workgroup of the stream reads all of x: one that is done must not store over it
        xq_ptr = xs_ptr = ws_ptr = None
        if not fused:
            x_q = alloc((m, k), dtype=torch.float8_e4m3fn, device=device)
            x_s = alloc((m, k // 128), dtype=torch.float32, device=device)
            xq_ptr, xs_ptr = x_q.data_ptr(), x_s.data_ptr()
        stream = _lib.stream_ptr(device)
        if ws_need:
            ws_ptr = _lib.workspace(device, ws_need, stream).data_ptr()
        ws_n, ws_k = ws.stride()
        code = _lib.linear_call()(
            x_ptr, _lib.DTYPE_CODES[dtype], w_ptr, ws.data_ptr(), out_ptr, m, n, k, k, ws_n, ws_k, n,
            xq_ptr, xs_ptr, ws_ptr, ws_need, _lib.DTYPE_CODES[out_dtype], stream,
        )
        if code:
            _lib.check(code, "fp8 linear")
        return out

    @property
    def method_name(self):
        return "fp8w8a8-b128-mi355"
