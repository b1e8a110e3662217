// The routed-expert FFN as one entry point: gate_up GEMM, SiLU-mul + quantizer, down GEMM, sum over the slots.
//
// With a few tokens the layer is a string of small launches around two reads of the weights: the ordered pair lists, the
// schedule table and the activation quantizer took a launch each (3.2, 2.5 and 2.5 us, none of them with enough work to
// matter) in front of the first GEMM.  None of the three needs another's result if every expert's workgroup counts the
// pairs of all experts by itself, so up to kProloguePairs pairs they are one launch (5.5 us).  Four layers of 128 experts,
// 4 tokens, launched eagerly: 338 us with seven launches from Python, 160 with five from here, which is what the GPU takes;
// one layer of 256 experts, 64 tokens: 1425 us and 1388.
#include <algorithm>

#include "moe_routing.hpp"
#include "quant_core.hpp"

namespace mi355 {

// One schedule to fill: `rows` table rows of blocks of `block_m` pairs (block_m = 0: none).
struct ScheduleOut {
    int32_t *table;
    int64_t rows;
    int32_t block_m;
};

constexpr int kPrologueThreads = 256;
using PrologueScan = PairScan<kPrologueThreads, 4>;
constexpr int64_t kProloguePairs = PrologueScan::kPass;  // one pass: an expert's workgroup holds every pair's expert in registers
constexpr int32_t kPrologueExperts = 1024;               // counters in LDS

constexpr int64_t kFewPairs = 64;  // one pair per lane of a wave

// The same for at most 64 pairs by one wave, a pair per lane, without LDS and barriers: which pairs precede one, which are of its
// expert and which are the first of a block are ballots.  Bound by the latency of its one load (four layers of 128 experts, 4
// tokens: 164.2 us with the counting form, 153.3).
__device__ __forceinline__ void few_pairs(const int32_t *topk_ids, const float *topk_weights, int32_t num_pairs, int32_t num_experts,
                                          int32_t *e2t_index, float *e2t_weight, int32_t *e_num, const ScheduleOut &first,
                                          const ScheduleOut &second, int expert, int lane) {
    const bool in = lane < num_pairs;
    const uint32_t id = in ? (uint32_t)topk_ids[lane] : ~0u;
    const float w = in ? topk_weights[lane] : 0.f;
    const bool valid = id < (uint32_t)num_experts, before = valid && id < (uint32_t)expert;
    const uint64_t lt = (1ull << lane) - 1ull, mine = __ballot(id == (uint32_t)expert);
    const int cnt = __popcll(mine);
    if (id == (uint32_t)expert) {
        const int64_t at = (int64_t)expert * num_pairs + __popcll(mine & lt);
        e2t_index[at] = lane;
        e2t_weight[at] = w;
    }
    if (lane == 0) e_num[expert] = cnt;
    // the pairs of this lane's expert, by the ten bits of its number
    uint64_t same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 10; ++b) {
        const uint64_t set = __ballot((id >> b) & 1u);
        same &= (id >> b) & 1u ? set : ~set;
    }
    const uint32_t rank = (uint32_t)__popcll(same & lt);
    const int tokens = __popcll(__ballot(before));
    auto blocks = [&](int32_t m) { return __popcll(__ballot(before && rank % (uint32_t)m == 0)); };
    if (first.block_m) schedule_rows<64>(expert, num_experts, cnt, tokens, blocks(first.block_m), first.block_m, first.rows, first.table, lane);
    if (second.block_m) schedule_rows<64>(expert, num_experts, cnt, tokens, blocks(second.block_m), second.block_m, second.rows, second.table, lane);
}

// Workgroups 0 .. E-1: the pair list, the count and the schedule rows of one expert.  The others: 256 chunks each of the
// activation quantizer (16 lanes of a DPP row = one group; scales [T, K/128] row-major).
template <bool FEW>
__global__ __launch_bounds__(kPrologueThreads) void moe_prologue_kernel(
    const int32_t *__restrict__ topk_ids, const float *__restrict__ topk_weights, int32_t num_pairs, int32_t num_experts,
    int32_t *__restrict__ e2t_index, float *__restrict__ e2t_weight, int32_t *__restrict__ e_num, ScheduleOut first,
    ScheduleOut second, const v4i *__restrict__ x, v2i *__restrict__ q, float *__restrict__ s, uint32_t total_chunks) {
    constexpr int T = kPrologueThreads, kW = T / 64;
    const int tid = threadIdx.x;
    if (blockIdx.x >= (uint32_t)num_experts) {
        const uint32_t c = (blockIdx.x - (uint32_t)num_experts) * T + tid;
        if (c >= total_chunks) return;  // a multiple of 16: a DPP row is active or idle as a whole
        v2i o;
        float sc;
        quant_chunk(__builtin_nontemporal_load(x + c), o, sc);
        q[c] = o;
        if ((tid & 15) == 0) s[c >> 4] = sc;
        return;
    }
    const int expert = blockIdx.x;
    if constexpr (FEW) {
        if (tid < 64)
            few_pairs(topk_ids, topk_weights, num_pairs, num_experts, e2t_index, e2t_weight, e_num, first, second, expert, tid);
    } else {
        __shared__ int hist[kPrologueExperts];
        __shared__ int wave_cnt[4 * kW];
        __shared__ int red[3][kW];
        v4i k[4], w[4];
        PrologueScan::load(topk_ids, (uint32_t)num_pairs, 0, tid, k);
        PrologueScan::load(topk_weights, (uint32_t)num_pairs, 0, tid, w);
        for (int e = tid; e < num_experts; e += T) hist[e] = 0;
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if ((uint32_t)k[c][j] < (uint32_t)num_experts) atomicAdd(&hist[k[c][j]], 1);  // others belong to no expert
        const int cnt = PrologueScan::append(k, w, expert, 0, tid, 0, e2t_index + (int64_t)expert * num_pairs,
                                             e2t_weight + (int64_t)expert * num_pairs, wave_cnt);
        if (tid == 0) e_num[expert] = cnt;
        // tokens and blocks of the experts before this one (the barriers of append() close the histogram)
        int before[3] = {0, 0, 0};
        for (int e = tid; e < expert; e += T) {
            const int n = hist[e];
            before[0] += n;
            if (first.block_m) before[1] += (n + first.block_m - 1) / first.block_m;
            if (second.block_m) before[2] += (n + second.block_m - 1) / second.block_m;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) before[i] += __shfl_xor(before[i], off);
            if ((tid & 63) == 0) red[i][tid >> 6] = before[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            before[i] = 0;
#pragma unroll
            for (int w = 0; w < kW; ++w) before[i] += red[i][w];
        }
        if (first.block_m)
            schedule_rows<T>(expert, num_experts, cnt, before[0], before[1], first.block_m, first.rows, first.table, tid);
        if (second.block_m)
            schedule_rows<T>(expert, num_experts, cnt, before[0], before[2], second.block_m, second.rows, second.table, tid);
    }
}

// Where everything between the input and the output lies in the caller's scratch.
struct FfnLayout {
    int32_t block_m1, block_m2;
    int64_t rows1, rows2;  // rows2 = 0: the down GEMM uses the schedule of the first
    size_t x_q, x_s, index, weight, count, table1, table2, gemm_out, act_q, act_s, bytes;
};

static FfnLayout ffn_layout(int64_t T, int64_t topk, int32_t E, int64_t hidden, int64_t inter) {
    FfnLayout f = {};
    const int64_t pairs = T * topk;
    f.block_m1 = mi355_grouped_block_m(pairs, E, 2 * inter, hidden);
    f.block_m2 = mi355_grouped_block_m(pairs, E, hidden, inter);
    f.rows1 = mi355_moe_align2_rows(pairs, E, f.block_m1);
    f.rows2 = f.block_m2 == f.block_m1 ? 0 : mi355_moe_align2_rows(pairs, E, f.block_m2);
    size_t at = 0;
    auto take = [&](int64_t n) {
        const size_t p = at;
        at += ((size_t)n + 255) & ~(size_t)255;
        return p;
    };
    f.x_q = take(T * hidden);
    f.x_s = take(T * (hidden / kBlockK) * 4);
    f.index = take((int64_t)E * pairs * 4);
    f.weight = take((int64_t)E * pairs * 4);
    f.count = take((int64_t)E * 4);
    f.table1 = take(f.rows1 * 16);
    f.table2 = take(f.rows2 * 16);
    f.gemm_out = take(pairs * std::max(2 * inter, hidden) * 2);  // the first GEMM's output is dead once it is quantized
    f.act_q = take(pairs * inter);
    f.act_s = take(pairs * (inter / kBlockK) * 4);
    f.bytes = at;
    return f;
}

static bool ffn_shape_ok(int64_t T, int32_t topk, int32_t E, int64_t hidden, int64_t inter) {
    return T >= 0 && topk > 0 && E > 0 && hidden > 0 && inter > 0 && hidden % kBlockK == 0 && inter % kBlockK == 0 &&
           T * topk < (1ll << 31) - 16384 && hidden < (1ll << 31) && inter < (1ll << 30);
}

}  // namespace mi355

using namespace mi355;

extern "C" size_t mi355_routed_ffn_scratch_bytes(int64_t T, int32_t topk, int32_t E, int64_t hidden, int64_t inter) {
    if (!ffn_shape_ok(T, topk, E, hidden, inter) || T == 0) return 0;
    return ffn_layout(T, topk, E, hidden, inter).bytes;
}

extern "C" size_t mi355_routed_ffn_workspace_bytes(int64_t T, int32_t topk, int32_t E, int64_t hidden, int64_t inter) {
    if (!ffn_shape_ok(T, topk, E, hidden, inter) || T == 0) return 0;
    const FfnLayout f = ffn_layout(T, topk, E, hidden, inter);
    size_t ws = 0;
    if (f.block_m1 == 256) ws = mi355_grouped_workspace_bytes(f.rows1);
    if (f.block_m2 == 256) ws = std::max(ws, mi355_grouped_workspace_bytes(f.rows2 ? f.rows2 : f.rows1));
    return ws;
}

extern "C" int mi355_routed_ffn(const void *x, const int32_t *topk_ids, const float *topk_weights, int64_t T, int32_t topk,
                                int32_t E, int64_t hidden, int64_t inter, const void *w1, const float *s1, const void *w2,
                                const float *s2, const void *b1, int32_t b1_dtype, int64_t b1_stride_e, const void *b2,
                                int32_t b2_dtype, int64_t b2_stride_e, void *out, void *scratch, size_t scratch_bytes,
                                void *ws, size_t ws_bytes, void *stream) {
    if (T < 0 || topk <= 0 || E <= 0 || hidden <= 0 || inter <= 0) return MI355_EINVAL;
    if (hidden % kBlockK != 0 || inter % kBlockK != 0) return MI355_ESHAPE;
    if (!ffn_shape_ok(T, topk, E, hidden, inter)) return MI355_EUNSUPPORTED;
    if (T == 0) return MI355_OK;
    if (!x || !topk_ids || !topk_weights || !w1 || !s1 || !w2 || !s2 || !out || !scratch) return MI355_EINVAL;
    if (((uintptr_t)x & 15) || ((uintptr_t)scratch & 15)) return MI355_EALIGN;
    const FfnLayout f = ffn_layout(T, topk, E, hidden, inter);
    if (scratch_bytes < f.bytes) return MI355_EWORKSPACE;
    hipStream_t st = (hipStream_t)stream;
    uint8_t *base = (uint8_t *)scratch;
    const int64_t pairs = T * topk, chunks = T * hidden / 8;
    int32_t *index = (int32_t *)(base + f.index), *count = (int32_t *)(base + f.count);
    int32_t *table1 = (int32_t *)(base + f.table1), *table2 = f.rows2 ? (int32_t *)(base + f.table2) : table1;
    float *weight = (float *)(base + f.weight), *x_s = (float *)(base + f.x_s), *act_s = (float *)(base + f.act_s);
    const int64_t rows2 = f.rows2 ? f.rows2 : f.rows1;
    int r;
    if (pairs <= kProloguePairs && E <= kPrologueExperts && chunks < (1ll << 30)) {
        const ScheduleOut first = {table1, f.rows1, f.block_m1};
        const ScheduleOut second = {table2, f.rows2, f.rows2 ? f.block_m2 : 0};
        r = launch(pairs <= kFewPairs ? moe_prologue_kernel<true> : moe_prologue_kernel<false>, dim3((uint32_t)(E + (chunks + kPrologueThreads - 1) / kPrologueThreads)),
                   dim3(kPrologueThreads), 0, st, topk_ids, topk_weights, (int32_t)pairs, E, index, weight, count, first, second,
                   (const v4i *)x, (v2i *)(base + f.x_q), x_s, (uint32_t)chunks);
        if (r != MI355_OK) return r;
    } else {
        if ((r = mi355_moe_align_fused(topk_ids, topk_weights, pairs, E, index, weight, count, stream)) != MI355_OK) return r;
        if ((r = mi355_group_quant_fp8(x, MI355_DTYPE_BF16, base + f.x_q, x_s, T, hidden, kBlockK, 1e-10f, hidden / kBlockK, 1,
                                       stream)) != MI355_OK)
            return r;
        if ((r = mi355_moe_align2(count, E, f.block_m1, f.rows1, table1, stream)) != MI355_OK) return r;
        if (f.rows2 && (r = mi355_moe_align2(count, E, f.block_m2, f.rows2, table2, stream)) != MI355_OK) return r;
    }
    uint8_t *gemm_out = base + f.gemm_out;
    r = mi355_grouped_block_fp8_gemm_bias(base + f.x_q, x_s, w1, s1, index, weight, count, table1, f.rows1, f.block_m1, pairs, T, E,
                                          topk, 2 * inter, hidden, 0, gemm_out, ws, ws_bytes, MI355_DTYPE_BF16, b1, b1_dtype,
                                          b1_stride_e, stream);
    if (r != MI355_OK) return r;
    r = mi355_silu_and_mul_group_quant_fp8(gemm_out, base + f.act_q, act_s, pairs, inter, 2 * inter, kBlockK, inter / kBlockK, 1,
                                           nullptr, 0, stream);
    if (r != MI355_OK) return r;
    r = mi355_grouped_block_fp8_gemm_bias(base + f.act_q, act_s, w2, s2, index, weight, count, table2, rows2, f.block_m2, pairs,
                                          pairs, E, 1, hidden, inter, 1, gemm_out, ws, ws_bytes, MI355_DTYPE_BF16, b2, b2_dtype,
                                          b2_stride_e, stream);
    if (r != MI355_OK) return r;
    return mi355_moe_sum_reduce(gemm_out, out, T, topk, hidden, stream);
}
