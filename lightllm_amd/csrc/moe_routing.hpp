// Device code of the routing tables: the ordered list of an expert's pairs, shared by the table kernels (moe_align.hip)
// and by the routed FFN's first launch (routed_ffn.hip).
#pragma once
#include "common.hpp"

namespace mi355 {

// THREADS * 4 * CH pairs per pass, four consecutive ones per lane and chunk.
template <int THREADS, int CH>
struct PairScan {
    static constexpr int kWaves = THREADS / 64;
    static constexpr int kChunk = THREADS * 4, kPass = kChunk * CH;
    static_assert(kWaves * CH <= 64, "one lane per count");

    // A pass of 4-byte values (keys: expert ids or the 0/1 entries of a mask row; or the routed weights), -1 past the end;
    // VEC: 16-byte aligned.
    template <bool VEC>
    static __device__ __forceinline__ void load_as(const int32_t *src, uint32_t num_pairs, uint32_t start, int tid, v4i (&k)[CH]) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const uint32_t p0 = start + c * kChunk + tid * 4;
            k[c] = v4i{-1, -1, -1, -1};
            if (VEC && p0 + 4 <= num_pairs) {
                k[c] = *(const v4i *)(src + p0);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (p0 + j < num_pairs) k[c][j] = src[p0 + j];
            }
        }
    }
    static __device__ __forceinline__ void load(const void *src, uint32_t num_pairs, uint32_t start, int tid, v4i (&k)[CH]) {
        if (((uintptr_t)src & 15) == 0) load_as<true>((const int32_t *)src, num_pairs, start, tid, k);
        else load_as<false>((const int32_t *)src, num_pairs, start, tid, k);
    }

    // Appends the pairs of a pass whose key is `want`, ascending, behind the `base` found so far; returns the new count.
    // Every thread has its keys before any writes (the barrier), so the indices may go over the keys themselves.  The weights
    // come with the keys: fetched hit by hit behind sixteen branches they were most of the kernel.
    static __device__ __forceinline__ int append(const v4i (&k)[CH], const v4i (&w)[CH], int want, uint32_t start, int tid, int base,
                                                 int32_t *out_i, float *out_w, int (&wave_cnt)[CH * kWaves]) {
        const int lane = tid & 63, wave = tid >> 6;
        const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
        int before[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            int total = 0;
            before[c] = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint64_t b = __ballot(k[c][j] == want);
                before[c] += __popcll(b & lt);
                total += __popcll(b);
            }
            if (lane == 0) wave_cnt[c * kWaves + wave] = total;
        }
        __syncthreads();
        // exclusive prefix over (chunk, wave): one count per lane
        const int mine = lane < CH * kWaves ? wave_cnt[lane] : 0;
        int incl = mine;
#pragma unroll
        for (int off = 1; off < CH * kWaves; off <<= 1) {
            const int t = __shfl_up(incl, off);
            if (lane >= off) incl += t;
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            int pos = base + __shfl(incl - mine, c * kWaves + wave) + before[c];
            const uint32_t p0 = start + c * kChunk + tid * 4;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (k[c][j] == want) {
                    out_i[pos] = (int32_t)(p0 + j);
                    out_w[pos] = as_f32((uint32_t)w[c][j]);
                    ++pos;
                }
        }
        const int all = __shfl(incl, CH * kWaves - 1);
        __syncthreads();
        return base + all;
    }
};

// The schedule rows of one expert: (expert, block, first token, tokens in the block); the last expert's workgroup also
// marks the padding rows behind its own.
template <int THREADS>
__device__ __forceinline__ void schedule_rows(int expert, int num_experts, int cnt, int token_start, int block_start,
                                              int block_m, int64_t rows, int32_t *table, int tid) {
    const int nblk = (cnt + block_m - 1) / block_m;
    for (int b = tid; b < nblk; b += THREADS) {
        const int64_t r = (int64_t)block_start + b;
        if (r < rows) {
            table[r * 4 + 0] = expert;
            table[r * 4 + 1] = b;
            table[r * 4 + 2] = token_start + b * block_m;
            table[r * 4 + 3] = min(cnt - b * block_m, block_m);
        }
    }
    if (expert == num_experts - 1)
        for (int64_t r = (int64_t)block_start + nblk + tid; r < rows; r += THREADS) table[r * 4] = -1;
}

}  // namespace mi355
