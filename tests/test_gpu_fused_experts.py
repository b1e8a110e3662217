"""GPU parity of the routed-expert FFN end to end (fused_experts_impl) against the CPU oracle's restatement of the
reference sequence.  Two chained block-FP8 GEMMs with a re-quantization in between: the GEMM tolerance of the path
(max-rel <= 1e-2, cosine >= 0.9999 against the same quantized operands) is applied to the final output, with the
max-rel bar doubled to 2e-2 because a bf16 rounding flip in the first GEMM moves an e4m3 byte of the second."""
import numpy as np
import pytest
import torch

import oracle
from oracle import torch_ref as tr
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _experts(E, I, Hd, seed):
    w1 = [H.quantized_weights(2 * I, Hd, seed=seed + e) for e in range(E)]
    w2 = [H.quantized_weights(Hd, I, seed=seed + 100 + e) for e in range(E)]
    st = lambda xs: torch.stack(list(xs)).contiguous()
    return st(q for q, _ in w1), st(s for _, s in w1), st(q for q, _ in w2), st(s for _, s in w2)


@pytest.mark.parametrize("T,E,topk,Hd,I", [(1, 8, 2, 256, 128), (48, 8, 2, 512, 256), (200, 16, 4, 1024, 256), (300, 6, 1, 256, 384),
                                           (512, 4, 2, 1024, 1024)])  # the last one takes the 256-row ping-pong blocks
def test_fused_experts_vs_oracle(hip, T, E, topk, Hd, I):
    from lightllm_amd.fused_moe import fused_experts_impl

    print(f"fused_experts T={T} E={E} topk={topk} H={Hd} I={I}", flush=True)
    x = H.activations(T, Hd, seed=T)
    w1q, w1s, w2q, w2s = _experts(E, I, Hd, seed=E * 7)
    ids, tw = H.routing(T, E, topk, seed=T + E)
    out = fused_experts_impl(x.cuda(), w1q.cuda(), w2q.cuda(), tw.cuda(), ids.cuda(), inplace=False,
                             use_fp8_w8a8=True, w1_scale=w1s.cuda(), w2_scale=w2s.cuda())
    torch.cuda.synchronize()
    want = tr.bf16_from_bits(oracle.fused_experts(tr.bits_of(x), tr.bits_of(w1q), w1s.numpy(), tr.bits_of(w2q),
                                                  w2s.numpy(), ids.numpy(), tw.numpy())).float()
    got = out.float().cpu()
    assert out.shape == x.shape and out.dtype == torch.bfloat16
    assert tr.cosine(got, want) >= 0.9999
    assert (got - want).abs().max() <= 2e-2 * want.abs().max()


def test_fused_experts_op_level_callers_and_bias(hip):
    """fused_experts / inplace_fused_experts_impl / outplace_fused_experts_impl (grouped_fused_moe.py:1118-1290,
    what FuseMoeTriton calls) give the bits of fused_experts_impl; w1_bias / w2_bias reach both grouped GEMMs
    (:1082, :1109) and match the oracle's sequence with the same biases."""
    from lightllm_amd.fused_moe import (fused_experts, fused_experts_impl, inplace_fused_experts_impl,
                                        outplace_fused_experts_impl)

    print("fused_experts op-level callers, bias", flush=True)
    T, E, topk, Hd, I = 160, 8, 2, 512, 256
    x = H.activations(T, Hd, seed=61)
    w1q, w1s, w2q, w2s = _experts(E, I, Hd, seed=62)
    ids, tw = H.routing(T, E, topk, seed=63)
    dev = [t.cuda() for t in (w1q, w2q, tw, ids)]
    kw = dict(use_fp8_w8a8=True, w1_scale=w1s.cuda(), w2_scale=w2s.cuda())
    base = fused_experts_impl(x.cuda(), *dev, inplace=False, **kw)
    out = fused_experts(x.cuda(), *dev, inplace=False, **kw)
    assert torch.equal(out.view(torch.int16), base.view(torch.int16))
    out = outplace_fused_experts_impl(x.cuda(), *dev, **kw)
    assert torch.equal(out.view(torch.int16), base.view(torch.int16))
    buf = x.cuda()
    assert inplace_fused_experts_impl(buf, *dev, **kw) is None
    assert torch.equal(buf.view(torch.int16), base.view(torch.int16))
    buf = x.cuda()
    assert fused_experts(buf, *dev, inplace=True, **kw) is buf
    assert torch.equal(buf.view(torch.int16), base.view(torch.int16))

    b1 = (torch.randn((E, 2 * I), generator=H.gen(64)) * 0.25).to(torch.bfloat16)
    b2 = (torch.randn((E, Hd), generator=H.gen(65)) * 0.25).float()
    out = fused_experts(x.cuda(), *dev, inplace=False, w1_bias=b1.cuda(), w2_bias=b2.cuda(), **kw)
    torch.cuda.synchronize()
    want = tr.bf16_from_bits(oracle.fused_experts(tr.bits_of(x), tr.bits_of(w1q), w1s.numpy(), tr.bits_of(w2q),
                                                  w2s.numpy(), ids.numpy(), tw.numpy(), w1_bias=b1.float().numpy(),
                                                  w2_bias=b2.numpy())).float()
    got = out.float().cpu()
    assert tr.cosine(got, want) >= 0.9999
    assert (got - want).abs().max() <= 2e-2 * want.abs().max()
    assert not torch.equal(out.view(torch.int16), base.view(torch.int16))


@pytest.mark.parametrize("layout,limit,alpha", [("interleaved", None, None), ("blocked", 7.0, 1.702), ("interleaved", 7.0, 1.702)])
def test_fused_experts_other_activation_forms(hip, layout, limit, alpha):
    """layout / limit / alpha are forwarded to silu_and_mul_fwd as in the reference (grouped_fused_moe.py:1084-1090);
    the product is then quantized by the stand-alone quantizer instead of the fused kernel."""
    from lightllm_amd.fused_moe import fused_experts_impl

    print(f"fused_experts layout={layout} limit={limit} alpha={alpha}", flush=True)
    T, E, topk, Hd, I = 96, 8, 2, 512, 256
    x = H.activations(T, Hd, seed=41)
    w1q, w1s, w2q, w2s = _experts(E, I, Hd, seed=43)
    ids, tw = H.routing(T, E, topk, seed=44)
    out = fused_experts_impl(x.cuda(), w1q.cuda(), w2q.cuda(), tw.cuda(), ids.cuda(), inplace=False, use_fp8_w8a8=True,
                             w1_scale=w1s.cuda(), w2_scale=w2s.cuda(), layout=layout, limit=limit, alpha=alpha)
    torch.cuda.synchronize()
    want = tr.bf16_from_bits(oracle.fused_experts(tr.bits_of(x), tr.bits_of(w1q), w1s.numpy(), tr.bits_of(w2q),
                                                  w2s.numpy(), ids.numpy(), tw.numpy(), layout, limit, alpha)).float()
    got = out.float().cpu()
    assert tr.cosine(got, want) >= 0.9999
    assert (got - want).abs().max() <= 2e-2 * want.abs().max()


def test_fused_experts_inplace_and_deterministic(hip):
    """Two runs give identical bits (ordered routing tables, no atomics on the output), and inplace writes the
    input tensor (unit_tests/common/fused_moe/test_grouped_fused_moe.py:200-215 checks the same determinism)."""
    from lightllm_amd.fused_moe import fused_experts_impl

    print("fused_experts determinism", flush=True)
    T, E, topk, Hd, I = 160, 8, 2, 512, 256
    x = H.activations(T, Hd, seed=3).cuda()
    w1q, w1s, w2q, w2s = (t.cuda() for t in _experts(E, I, Hd, seed=5))
    ids, tw = (t.cuda() for t in H.routing(T, E, topk, seed=8))
    kw = dict(use_fp8_w8a8=True, w1_scale=w1s, w2_scale=w2s)
    a = fused_experts_impl(x, w1q, w2q, tw, ids, **kw)
    b = fused_experts_impl(x, w1q, w2q, tw, ids, **kw)
    xin = x.clone()
    c = fused_experts_impl(xin, w1q, w2q, tw, ids, inplace=True, **kw)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    assert c.data_ptr() == xin.data_ptr() and torch.equal(c, a)


# the first launch's pair limit and one past it, single tokens and experts, more experts than it counts, ids that are not 16-byte
# aligned, schedules of two block sizes (E = 8, 12 rows per expert, K = 2048 / 768), 256-row blocks
@pytest.mark.parametrize("T,E,topk,Hd,I", [(1, 1, 1, 128, 128), (3, 1024, 8, 256, 128), (3, 1025, 8, 256, 128),
                                           (512, 16, 8, 256, 128), (513, 16, 8, 256, 128), (4095, 5, 1, 128, 128),
                                           (4097, 5, 1, 128, 128), (37, 7, 3, 384, 256), (48, 8, 2, 2048, 768),
                                           (300, 4, 2, 1024, 1024)])
@pytest.mark.parametrize("offset", [0, 1])
def test_fused_experts_in_one_call_equals_the_steps(hip, T, E, topk, Hd, I, offset):
    """An (empty) run_config sends the layer through the operators one by one: the same bits, in place too."""
    from lightllm_amd.fused_moe import fused_experts_impl

    print(f"fused_experts one call T={T} E={E} topk={topk} H={Hd} I={I} offset={offset}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + E)
    w1 = torch.randint(0, 0x70, (E, 2 * I, Hd), dtype=torch.uint8, device="cuda", generator=g).view(torch.float8_e4m3fn)
    w2 = torch.randint(0, 0x70, (E, Hd, I), dtype=torch.uint8, device="cuda", generator=g).view(torch.float8_e4m3fn)
    s1 = torch.rand((E, 2 * I // 128, Hd // 128), device="cuda", generator=g) * 1e-3
    s2 = torch.rand((E, Hd // 128, I // 128), device="cuda", generator=g) * 1e-3
    x = H.activations(T, Hd, seed=T).cuda()
    ids, tw = H.routing(T, E, topk, seed=T + E)
    ids_buf = torch.empty(offset + T * topk, dtype=torch.int32, device="cuda")
    ids_dev = ids_buf[offset:].view(T, topk).copy_(ids)
    kw = dict(use_fp8_w8a8=True, w1_scale=s1, w2_scale=s2)
    want = fused_experts_impl(x, w1, w2, tw.cuda(), ids_dev, run_config={}, **kw)
    got = fused_experts_impl(x, w1, w2, tw.cuda(), ids_dev, **kw)
    inp = x.clone()
    fused_experts_impl(inp, w1, w2, tw.cuda(), ids_dev, inplace=True, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert torch.equal(inp.view(torch.int16), want.view(torch.int16))


# up to 64 pairs the tables come from ballots: both sides of that, experts with more than one block, one pair, experts without any
@pytest.mark.parametrize("T,E,topk,Hd,I", [(64, 1, 1, 256, 128), (32, 2, 2, 2048, 768), (63, 3, 1, 256, 2048), (13, 5, 5, 256, 128),
                                           (16, 1024, 4, 256, 128), (8, 600, 8, 2048, 128)])
def test_fused_experts_with_few_pairs(hip, T, E, topk, Hd, I):
    test_fused_experts_in_one_call_equals_the_steps(hip, T, E, topk, Hd, I, 1)


# full chunks and a shorter last one (of another block size: 20 and 3 pairs per expert; 31 and 8), an odd topk, ids of a
# chunk that are not 16-byte aligned, biases
@pytest.mark.parametrize("T,E,topk,Hd,I,chunk", [(101, 7, 3, 256, 384, 47), (107, 12, 8, 1024, 1024, 47), (96, 5, 1, 128, 128, 48)])
@pytest.mark.parametrize("bias", [False, True])
def test_fused_experts_in_chunks(hip, monkeypatch, T, E, topk, Hd, I, chunk, bias):
    """More tokens than one pass takes: the one-call form, pass by pass over one scratch, gives the bits of the steps."""
    from lightllm_amd.fused_moe import fused_experts_impl, grouped_fused_moe

    print(f"fused_experts in chunks T={T} E={E} topk={topk} H={Hd} I={I} chunk={chunk} bias={bias}", flush=True)
    monkeypatch.setattr(grouped_fused_moe, "FFN_MOE_CHUNK_SIZE", chunk)
    x = H.activations(T, Hd, seed=T).cuda()
    w1q, w1s, w2q, w2s = (t.cuda() for t in _experts(E, I, Hd, seed=E))
    ids, tw = (t.cuda() for t in H.routing(T, E, topk, seed=T + E))
    kw = dict(use_fp8_w8a8=True, w1_scale=w1s, w2_scale=w2s)
    if bias:
        kw["w1_bias"] = torch.randn((E, 2 * I), generator=H.gen(1)).to(torch.bfloat16).cuda()
        kw["w2_bias"] = torch.randn((E, Hd), generator=H.gen(2)).cuda()
    want = fused_experts_impl(x, w1q, w2q, tw, ids, run_config={}, **kw)
    got = fused_experts_impl(x, w1q, w2q, tw, ids, **kw)
    inp = x.clone()
    fused_experts_impl(inp, w1q, w2q, tw, ids, inplace=True, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert torch.equal(inp.view(torch.int16), want.view(torch.int16))
    monkeypatch.undo()   # and those of a single pass
    whole = fused_experts_impl(x, w1q, w2q, tw, ids, **kw)
    assert tr.cosine(got.float().cpu(), whole.float().cpu()) >= 0.9999
