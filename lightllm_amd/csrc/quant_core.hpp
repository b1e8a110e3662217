// Device-side arithmetic of the 1x128 group quantizer (bf16 / fp16 / fp32 -> e4m3fn + fp32 scale), shared by the
// stand-alone quantizer and by the kernels that quantize what they have just computed.
//
// Arithmetic (must reproduce IEEE fp32 division results bit for bit, see
// lightllm/common/basemodel/triton_kernel/quantization/fp8act_quant_kernel.py:53-57, 239-251):
//     amax = max(max|x|, eps);  s = amax / 448;  q = e4m3fn_rtne(clamp(x / s, -448, 448))
// Doing two IEEE divisions per element would make the kernels VALU-bound, so:
//   * s = amax/448 is formed as q0 = amax*c, s = fma(fma(-q0,448,amax), c, q0) with c = RN(1/448);
//     this equals RN(amax/448) for every bf16 and every fp16 amax and for the default eps (checked exhaustively on
//     the CPU); calls with any other eps do not come here (they take quant_chunk_f32).
//   * x/s is formed as y = fma(x, r, x*d) from r, a little under 1/s (v_rcp_f32, two ulps taken off), and the rest
//     d = fma(-s, r, 1) * r >= 0: two operations per element.  r + d falls short of 1/s by e^2 of it, e = 1 - s*r being up
//     to three ulps: about 2^-42 at most, more where d is subnormal (the largest amax).  That is no proof by itself: for every
//     pair (amax, |x| <= amax) of bf16 or of fp16 values the e4m3 byte of y is that of RN(x/s), whatever the last bit of
//     the reciprocal is, checked exhaustively on the CPU (oracle_fast_quant_mismatches in the test oracle replays exactly these
//     operations for a reciprocal off by -1, 0 and +1 ulp).  With r and d positive -0 stays -0, as -0/s is.
// No contraction of a product and a sum anywhere in this arithmetic: the pragma stands inside each function so that it does
// not reach the rest of a file that includes this one.
#pragma once
#include "common.hpp"

namespace mi355 {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max_u32(uint32_t v) {
    uint32_t t = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
    return t > v ? t : v;
}

__device__ __forceinline__ uint32_t row16_max_u32(uint32_t v) {
    v = dpp_max_u32<0xB1>(v);   // quad_perm [1,0,3,2]
    v = dpp_max_u32<0x4E>(v);   // quad_perm [2,3,0,1]
    v = dpp_max_u32<0x141>(v);  // row_half_mirror: lane i <-> 7-i inside each half row
    v = dpp_max_u32<0x140>(v);  // row_mirror:      lane i <-> 15-i inside the row
    return v;
}

__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
    us2 x = __builtin_bit_cast(us2, a), y = __builtin_bit_cast(us2, b);
    us2 r = __builtin_elementwise_max(x, y);
    return __builtin_bit_cast(uint32_t, r);
}

// A group that holds a NaN or an infinity (outside the reference's contract: its max and clamp leave NaN
// unspecified) is poisoned as a whole: scale = NaN, every byte 0x7F with the sign bit of its element.
__device__ __forceinline__ void nonfinite_chunk(uint32_t s0, uint32_t s1, uint32_t s2, uint32_t s3, uint32_t s4,
                                                uint32_t s5, uint32_t s6, uint32_t s7, v2i &out, float &scale) {
    out[0] = (int)(0x7f7f7f7fu | (s0 << 7) | (s1 << 15) | (s2 << 23) | (s3 << 31));
    out[1] = (int)(0x7f7f7f7fu | (s4 << 7) | (s5 << 15) | (s6 << 23) | (s7 << 31));
    scale = as_f32(0x7fc00000u);
}

// Quantize 8 consecutive fp32 values (fp32 activations, or any with another eps, widened by the caller) with true IEEE
// divisions: the short quotient above is only proven for 16-bit inputs and the default eps.
__device__ __forceinline__ void quant_chunk_f32(const float (&f)[8], float eps, v2i &out, float &scale) {
#pragma clang fp contract(off)
    uint32_t mx = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t a = as_u32(f[i]) & 0x7fffffffu;
        mx = a > mx ? a : mx;
    }
    mx = row16_max_u32(mx);
    if (mx > 0x7f7fffffu) {
        nonfinite_chunk(as_u32(f[0]) >> 31, as_u32(f[1]) >> 31, as_u32(f[2]) >> 31, as_u32(f[3]) >> 31,
                        as_u32(f[4]) >> 31, as_u32(f[5]) >> 31, as_u32(f[6]) >> 31, as_u32(f[7]) >> 31, out, scale);
        return;
    }
    float amax = as_f32(mx);
    amax = amax > eps ? amax : eps;
    const float s = amax / 448.0f;
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        y[i] = f[i] / s;
        y[i] = y[i] > 448.0f ? 448.0f : y[i];
        y[i] = y[i] < -448.0f ? -448.0f : y[i];
    }
    int w0 = 0, w1 = 0;
    w0 = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], w0, false);
    w0 = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], w0, true);
    w1 = __builtin_amdgcn_cvt_pk_fp8_f32(y[4], y[5], w1, false);
    w1 = __builtin_amdgcn_cvt_pk_fp8_f32(y[6], y[7], w1, true);
    out[0] = w0;
    out[1] = w1;
    scale = s;
}

// Quantize N 16-byte chunks of bf16 (F16: fp16) with the default floor eps = 1e-10; the group amax is shared through the DPP row.
// About 50 vector operations per chunk.  (Chunks of one lane are interleaved; non-finite groups are handled behind one
// test that the whole wave takes or skips.)  No clamp is needed: |x| <= amax and s = RN(max(amax,eps)/448) bound |x/s| by
// 448*(1+2^-23), which the e4m3 cast rounds to 448, exactly what clamp-then-cast gives.
template <bool F16, int N>
__device__ __forceinline__ void quant_chunks(const v4i (&v)[N], v2i (&out)[N], float (&scale)[N]) {
#pragma clang fp contract(off)
    constexpr uint32_t kEps = 0x2edbe6ffu;  // 1e-10f
    uint32_t mx[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        // |x| as integers: for non-negative floats the integer order is the float order.
        const uint32_t m = pk_max_u16(pk_max_u16((uint32_t)v[k][0] & 0x7fff7fffu, (uint32_t)v[k][1] & 0x7fff7fffu),
                                      pk_max_u16((uint32_t)v[k][2] & 0x7fff7fffu, (uint32_t)v[k][3] & 0x7fff7fffu));
        const uint32_t hi = m >> 16, lo = m & 0xffffu, w = hi > lo ? hi : lo;
        if constexpr (F16) mx[k] = as_u32((float)__builtin_bit_cast(_Float16, (uint16_t)w));
        else mx[k] = w << 16;
    }
#pragma unroll
    for (int k = 0; k < N; ++k) mx[k] = row16_max_u32(mx[k]);
    uint32_t top = mx[0];
#pragma unroll
    for (int k = 1; k < N; ++k) top = mx[k] > top ? mx[k] : top;
    const float c = 1.0f / 448.0f;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const float amax = as_f32(mx[k] > kEps ? mx[k] : kEps);
        const float q0 = amax * c;
        const float s = __builtin_fmaf(__builtin_fmaf(-q0, 448.0f, amax), c, q0);
        const float r = as_f32(as_u32(__builtin_amdgcn_rcpf(s)) - 2u);
        const float d = __builtin_fmaf(-s, r, 1.0f) * r;
        float f[8];
        if constexpr (F16) {
            const h8 h = __builtin_bit_cast(h8, v[k]);
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = (float)h[i];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                f[2 * i] = as_f32((uint32_t)v[k][i] << 16);
                f[2 * i + 1] = as_f32((uint32_t)v[k][i] & 0xffff0000u);
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = __builtin_fmaf(f[i], r, f[i] * d);
        int w0 = 0, w1 = 0;
        w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], w0, false);
        w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], w0, true);
        w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], w1, false);
        w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], w1, true);
        out[k][0] = w0;
        out[k][1] = w1;
        scale[k] = s;
    }
    // (no asm in this block to hold its arithmetic behind the branch: even an empty one there cost a weight stream that
    // quantizes its activations 6 % - N = 28672, K = 4096, one row: 23.4 us against 22.0)
    if (__builtin_expect(__ballot(top > 0x7f7fffffu) != 0ull, 0)) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            if (mx[k] > 0x7f7fffffu) {  // the same for all 16 lanes of the group
                const uint32_t d0 = (uint32_t)v[k][0], d1 = (uint32_t)v[k][1], d2 = (uint32_t)v[k][2], d3 = (uint32_t)v[k][3];
                nonfinite_chunk((d0 >> 15) & 1u, d0 >> 31, (d1 >> 15) & 1u, d1 >> 31, (d2 >> 15) & 1u, d2 >> 31,
                                (d3 >> 15) & 1u, d3 >> 31, out[k], scale[k]);
            }
        }
    }
}

// One chunk of bf16.
__device__ __forceinline__ void quant_chunk(const v4i &v, v2i &out, float &scale) {
    const v4i a[1] = {v};
    v2i o[1];
    float s[1];
    quant_chunks<false, 1>(a, o, s);
    out = o[0];
    scale = s[0];
}

}  // namespace mi355
