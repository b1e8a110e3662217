// Block-scaled FP8 grouped GEMM for experts with few rows on gfx950: the weight stream of gemm_stream.hpp over a schedule
// of (expert, row block) entries.
//
// With one to a few rows per expert the launch is a single pass over the weights of the experts that were hit, and what
// holds for the dense decode stream holds here: plain 16-byte loads of whole 128-byte row segments, a few K steps in
// flight in registers per wave, the transposition into MFMA operand order through a wave-private LDS area, no barrier in
// the K loop.
//
//   workgroup = 4 waves = one schedule entry x 64 weight rows, whole K; the waves take the K steps round-robin and add
//   their accumulators through LDS at the end.  An entry of at most 16 rows runs one MFMA row block per step, one of up
//   to 32 two: how many is decided per entry, so uneven routing costs what it needs.  The activation rows are gathered
//   through expert_to_token_index, the scales of the workgroup's rows are staged in LDS once, outputs are scattered.
//
// What bounds it is the memory: 217 of 256 experts of N = 4096, K = 7168 (6.4 GB) in 911 us = 7.0 TB/s, N = 7168, K = 2048
// in 464 us = 6.9, where the ring tiles (16 x 128, DMA into LDS, a barrier per step) took 1043 and 524; Mixtral gate_up,
// 16 tokens, 147 us (6.4 TB/s) against 183.  Tried and not kept: the first weight requests ahead of the row indices (level,
// 10 % slower with K = 768); waves that stream 16-row units over the whole K by themselves with the activations staged in
// LDS once, for short K (K = 768, 4 / 64 tokens: 13.0 / 40.7 us against 11.5 / 41.5 for the ring tiles).
#pragma once
#include "gemm_stream.hpp"

namespace mi355 {

template <int MT>
struct GStreamCfg {
    static_assert(MT == 1 || MT == 2, "");
    static constexpr int TNW = 4, BN = 64;
    static constexpr int kDepth = MT == 1 ? 3 : 2;                // K steps in flight per wave
    static constexpr int kXOff = BN * 128;                        // X block behind the W block
    static constexpr int kWaveBytes = (BN + 16 * MT) * 128;       // >= one wave's accumulators (TNW * MT KiB)
    static constexpr int kScaleOff = kStreamWaves * kWaveBytes;   // X scales [KB][16*MT + 1]
    static constexpr int kScaleStride = 16 * MT + 1;
    static constexpr int lds_bytes(int KB) { return kScaleOff + KB * kScaleStride * 4; }
};

template <int MT, bool BIAS>
__device__ __forceinline__ void gstream_tile(const GemmArgs &p, uint8_t *lds, int tid, int expert, int m0, int rows, int n0) {
    using Cfg = GStreamCfg<MT>;
    constexpr int D = Cfg::kDepth, TNW = Cfg::TNW, NX = 2 * MT;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g4 = lane >> 4;
    const int sub = lane >> 3, pch = lane & 7;
    const int KB = p.K / kBlockK;
    const int steps = wave < KB ? (KB - wave + kStreamWaves - 1) / kStreamWaves : 0;

    const int32_t *idx_list = p.e2t_index + (int64_t)expert * p.num_pairs + m0;
    const uint8_t *wbase = p.W + (int64_t)expert * p.w_e + (int64_t)n0 * p.ldw;
    const int NB = (p.N + kBlockN - 1) / kBlockN;
    const float *wsp = p.Ws + (int64_t)expert * p.ws_e + (int64_t)min(n0 / kBlockN, NB - 1) * p.ws_n;

    // ---- per-lane offsets (rows past the matrix or the entry repeat the last one; their results are never stored)
    uint32_t woff[2 * TNW];
#pragma unroll
    for (int i = 0; i < 2 * TNW; ++i) woff[i] = (uint32_t)min(8 * i + sub, p.N - 1 - n0) * (uint32_t)p.ldw + (uint32_t)pch * 16u;
    uint32_t xoff[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i)
        xoff[i] = (uint32_t)idx_list[min(8 * i + sub, rows - 1)] / (uint32_t)p.topk * (uint32_t)p.ldx + (uint32_t)pch * 16u;

    struct Regs {
        v4i w[2 * TNW];
        v4i x[NX];
        float ws;
    };
    auto load = [&](Regs &r, int it) {
        const int kb = wave + it * kStreamWaves;
        const uint8_t *wk = wbase + (int64_t)kb * kBlockK;
        const uint8_t *xk = p.X + (int64_t)kb * kBlockK;
#pragma unroll
        for (int i = 0; i < 2 * TNW; ++i) r.w[i] = __builtin_nontemporal_load((const v4i *)(wk + woff[i]));
#pragma unroll
        for (int i = 0; i < NX; ++i) r.x[i] = *(const v4i *)(xk + xoff[i]);
        r.ws = wsp[(int64_t)kb * p.ws_k];
    };

    // ---- wave-private LDS (see gemm_stream.hpp)
    uint8_t *my = lds + wave * Cfg::kWaveBytes;
    uint32_t wst[2 * TNW];
#pragma unroll
    for (int i = 0; i < 2 * TNW; ++i) {
        const int nl = 8 * i + sub;
        const int a = nl / (4 * TNW), rem = nl % (4 * TNW);
        const int rho = 16 * (rem >> 2) + 4 * a + (rem & 3);
        wst[i] = (uint32_t)rho * 128u + (((uint32_t)pch ^ swz((uint32_t)rho)) * 16u);
    }
    uint32_t xst[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const int row = 8 * i + sub;
        xst[i] = (uint32_t)Cfg::kXOff + (uint32_t)row * 128u + (((uint32_t)pch ^ swz((uint32_t)row)) * 16u);
    }
    const uint32_t fr = swz((uint32_t)r16);
    const uint32_t c0 = ((uint32_t)(2 * g4)) ^ fr, c1 = c0 ^ 1u;
    const uint32_t rd0 = (uint32_t)r16 * 128u + c0 * 16u, rd1 = (uint32_t)r16 * 128u + c1 * 16u;
    float *xs_lds = (float *)(lds + Cfg::kScaleOff);

    v4f acc[MT][TNW];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int j = 0; j < TNW; ++j) acc[t][j] = v4f{0.f, 0.f, 0.f, 0.f};

    auto consume = [&](const Regs &r, int it) {
        const int kb = wave + it * kStreamWaves;
        float xsv[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) xsv[t] = xs_lds[kb * Cfg::kScaleStride + 16 * t + r16];
#pragma unroll
        for (int i = 0; i < 2 * TNW; ++i) *(v4i *)(my + wst[i]) = r.w[i];
#pragma unroll
        for (int i = 0; i < NX; ++i) *(v4i *)(my + xst[i]) = r.x[i];
        // LDS operations of one wave execute in order: the reads below see the writes above
        v8i wf[TNW];
#pragma unroll
        for (int j = 0; j < TNW; ++j) {
            const v4i lo = *(const v4i *)(my + rd0 + j * 2048);
            const v4i hi = *(const v4i *)(my + rd1 + j * 2048);
            wf[j] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const v4i lo = *(const v4i *)(my + Cfg::kXOff + rd0 + t * 2048);
            const v4i hi = *(const v4i *)(my + Cfg::kXOff + rd1 + t * 2048);
            const v8i xf = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            const float sc = xsv[t] * r.ws;
#pragma unroll
            for (int j = 0; j < TNW; ++j) {
                const v4f part = mfma_16x16x128_fp8(wf[j], xf, v4f{0.f, 0.f, 0.f, 0.f});
                acc[t][j] += part * sc;
            }
        }
    };

    Regs regs[D];
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d < steps) load(regs[d], d);
    // ---- stage the activation scales of the entry's rows behind the first weight requests: thread (row tid / 16, step
    // tid % 16 and on) reads a scale row as whole cache lines
    for (int r = tid >> 4; r < 16 * MT; r += 16) {
        const float *src = p.Xs + (int64_t)((uint32_t)idx_list[min(r, rows - 1)] / (uint32_t)p.topk) * p.xs_m;
        for (int kb = tid & 15; kb < KB; kb += 16) xs_lds[kb * Cfg::kScaleStride + r] = src[(int64_t)kb * p.xs_k];
    }
    __syncthreads();
    for (int j = 0; j < steps; j += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (j + d < steps) {
                consume(regs[d], j + d);
                if (j + d + D < steps) load(regs[d], j + d + D);
            }
        }
    }

    // ---- add the four waves' accumulators; wave w ends up with the MFMA blocks f = mt*TNW + tn, f % 4 == w
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int j = 0; j < TNW; ++j) *(v4f *)(my + ((t * TNW + j) * 64 + lane) * 16) = acc[t][j];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int j = wave;  // TNW == kStreamWaves
        v4f s = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kStreamWaves; ++w) s += *(const v4f *)(lds + w * Cfg::kWaveBytes + ((t * TNW + j) * 64 + lane) * 16);
        // lane (r16, g4) holds row 16*t + r16, columns n0 + 16*g4 + 4*j + [0, 4)
        const int rl = 16 * t + r16;
        const int ncol = n0 + 4 * TNW * g4 + 4 * j;
        if (rl >= rows) continue;
        const float rw = p.mul_weight ? p.e2t_weight[(int64_t)expert * p.num_pairs + m0 + rl] : 1.0f;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (BIAS) o[e] = (s[e] + bias_value(p.bias, p.bias_dtype, (int64_t)expert * p.bias_e + min(ncol + e, p.N - 1))) * rw;
            else o[e] = s[e] * rw;
        }
        uint16_t *cp = p.C + (int64_t)idx_list[rl] * p.ldc + ncol;
        if (p.vec_store && ncol + 4 <= p.N) {
            *(v2i *)cp = v2i{(int)pack_out2(o[0], o[1], p.out_f16), (int)pack_out2(o[2], o[3], p.out_f16)};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (ncol + e < p.N) cp[e] = (uint16_t)out_bits(o[e], p.out_f16);
        }
    }
}

// One workgroup per tile where most of the schedule is real.  LOOP: its length is only a bound (the padded layout of the
// expert-parallel caller); the grid is smaller than the schedule and a workgroup takes every gridDim.x-th tile until it
// meets the padding at the end.  A workgroup that finds nothing to do costs about 1 ns of the launch, and 16384 padded rows
// for 512 real ones made that 90 us of 350.
template <bool BIAS, bool LOOP>
__global__ __launch_bounds__(256, 2) void block_fp8_gemm_gstream_kernel(const GemmArgs p, int block_m) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    uint32_t tile = blockIdx.x;
    do {
        // n fastest: the tiles of an entry start together, and experts are handed out in schedule order
        const uint32_t tile_m = tile / (uint32_t)p.tiles_n, tile_n = tile - tile_m * (uint32_t)p.tiles_n;
        const v4i row = *(const v4i *)(p.table + (int64_t)tile_m * 4);
        const int expert = __builtin_amdgcn_readfirstlane(row[0]);
        if (expert < 0) return;
        const int mi = __builtin_amdgcn_readfirstlane(row[1]), m0 = mi * block_m;
        int rows = __builtin_amdgcn_readfirstlane(row[3]);
        if (block_m == 16) {
            // 16-row entries are taken in pairs (an expert's blocks 2i and 2i + 1 read the same weights): the even one
            // runs both, the odd one has nothing to do
            if (mi & 1) rows = 0;
            else if (rows == 16) rows = min(__builtin_amdgcn_readfirstlane(p.e_num[expert]) - m0, 32);
        }
        const int n0 = (int)tile_n * GStreamCfg<1>::BN;
        int tid = threadIdx.x;
        if constexpr (LOOP) asm volatile("" : "+v"(tid));  // nothing that depends on the lane stays in registers across tiles
        if (rows > 16) gstream_tile<2, BIAS>(p, lds, tid, expert, m0, rows, n0);
        else if (rows > 0) gstream_tile<1, BIAS>(p, lds, tid, expert, m0, rows, n0);
        if constexpr (LOOP) __syncthreads();  // the next tile lays its operands over this one's sums
        tile += gridDim.x;
    } while (LOOP && tile < (uint32_t)p.total_tiles);
}

}  // namespace mi355
