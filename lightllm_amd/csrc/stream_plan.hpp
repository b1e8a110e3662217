// Launch plans of the weight-streaming kernels (gemm_stream.hpp, gemm_streamcu.hpp): host code shared by the GEMM entry
// points (block_gemm.hip) and by the linear entry point that quantizes its activations in the stream (linear.hip).
#pragma once
#include "gemm_stream.hpp"
#include "gemm_streamcu.hpp"

namespace mi355 {

constexpr int kMaxLds = 160 * 1024;  // LDS per workgroup on gfx950

inline bool fast_layout_ok(const void *A, const void *B, int64_t K, int64_t lda, int64_t ldb_k, int64_t ldb_n) {
    return ldb_k == 1 && K % kBlockK == 0 && lda % 16 == 0 && ldb_n % 16 == 0 && ((uintptr_t)A & 15) == 0 &&
           ((uintptr_t)B & 15) == 0;
}

// ---- the stream in tiles of 16, 32 or 64 weight rows, M <= 64
inline int skinny_mt(int64_t M) { return M <= 16 ? 1 : (M <= 32 ? 2 : 4); }

struct SkinnyPlan {
    int tnw, splits, tiles;
};

inline SkinnyPlan skinny_plan(int64_t M, int64_t N, int64_t K, int cus) {
    SkinnyPlan pl;
    pl.splits = 1;
    const int64_t t64 = (N + 63) / 64;
    // 64-row tiles that come to just over one per unit leave half the units with twice the work of the others:
    // narrower tiles then (N = 18432, K = 7168, 288 tiles of 64 rows, M = 1 / 16: 22.6 / 26.8 us against 27.9 /
    // 29.9; N = 18944, K = 3584: 13.2 / 15.2 against 16.4 / 17.3); up to 1.5 per unit for M > 16, where the narrower
    // tiles have 32 rows (N = 24576, K = 1536, M = 32 / 64: 10.3 / 15.3 against 12.2 / 18.7)
    bool unbalanced = t64 > cus && t64 * 4 <= (int64_t)cus * (M <= 16 ? 5 : 6);
    // up to 8 rows under a long K the 16-row tiles also win wherever the 64-row ones fill less than 84 % of their
    // last round (N = 36864, K = 7168, 2.25 per unit, M = 1 / 8: 39.6 / 41.5 us against 45.4 / 46.2; N = 22016,
    // K = 5120, 1.34 per unit: 19.9 / 21.4 against 22.7 / 23.4); with whole rounds they lose (N = 49152, M = 8: 41.6
    // against 38.5), and so they do on K = 4096
    if (M <= 8 && K >= 5120 && t64 > cus) {
        const int64_t rounds = (t64 + cus - 1) / cus;
        if (t64 * 25 < rounds * cus * 21) unbalanced = true;
    }
    if (t64 >= cus && !unbalanced) {
        // N alone gives every compute unit a workgroup: 64-row tiles, whole K
        pl.tnw = 4;
        pl.tiles = (int)((N + 63) / 64);
        return pl;
    }
    // Otherwise narrow tiles first, then K splits, until there are about two workgroups per compute unit (measured
    // on N=4096, K=14336: 16-row tiles x 2 splits 13.1 us at M <= 8 against 14.1 for 64-row tiles x 4 splits;
    // at M > 16, 32-row tiles x 4 splits 16.1 / 20.0 us at M = 32 / 64, 16-row tiles 18.3 / 25.8), never below 16 K
    // steps per workgroup (4 per wave).
    pl.tnw = M <= 16 ? 1 : 2;
    pl.tiles = (int)((N + 16 * pl.tnw - 1) / (16 * pl.tnw));
    const int KB = (int)(K / kBlockK);
    pl.splits = (2 * cus + pl.tiles - 1) / pl.tiles;
    // from 1.5 tiles per unit on K stays whole: two splits would make 3 to 4 workgroups per unit and an exchange
    // (N = 7168, K = 8192, 448 tiles, M = 1 / 16: 12.8 / 13.7 us against 16.7 / 17.9; 14336 x 4096, M = 32: 15.1
    // against 18.8; 6912 x 6912, M = 1: 10.2 against 12.3)
    if (pl.tiles * 2 >= 3 * cus) pl.splits = 1;
    const int max_splits = KB / 16 > 0 ? KB / 16 : 1;
    if (pl.splits > max_splits) pl.splits = max_splits;
    if (pl.splits < 1) pl.splits = 1;
    // a workgroup stages the activation scales of its K range in LDS if the range is short enough; one more split
    // that gets it there pays (N=7168, K=18432, M=16: 72 steps unstaged 37.5 us, 48 steps staged 30.7)
    const int cap = skinny_mt(M) == 4 ? StreamCfg<4, 2>::kMaxScaleSteps : StreamCfg<1, 1>::kMaxScaleSteps;
    const int need = (KB + cap - 1) / cap;
    if (pl.splits < need && need <= max_splits) pl.splits = need;
    return pl;
}

inline size_t skinny_workspace(int64_t M, const SkinnyPlan &pl) {
    return (size_t)MI355_WS_COUNTER_BYTES + (size_t)pl.tiles * pl.splits * 16 * skinny_mt(M) * 16 * pl.tnw * 4;
}

// Preconditions of the stream kernel beyond the fast layout.
inline int skinny_check(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t as_m, int cus,
                        bool ws_usable, size_t ws_bytes) {
    if (M > 64) return MI355_EUNSUPPORTED;
    // rows are addressed from the matrix bases with 32-bit byte offsets
    if (N * ldw >= (1ll << 32) || M * lda >= (1ll << 32) || M * as_m >= (1ll << 32)) return MI355_EUNSUPPORTED;
    const SkinnyPlan pl = skinny_plan(M, N, K, cus);
    if ((int64_t)pl.tiles * 4 > MI355_WS_COUNTER_BYTES) return MI355_EUNSUPPORTED;
    if (pl.splits > 1 && (!ws_usable || ws_bytes < skinny_workspace(M, pl))) return MI355_EWORKSPACE;
    return MI355_OK;
}

// ---- the weight stream cut into one equal share per compute unit (gemm_streamcu.hpp): TNW 16-row blocks per
// workgroup with TNW = ceil(N / 16 / cus), one workgroup of 8 waves per tile, whole K.  Returns TNW, or 0 where the
// kernel does not apply: more than 16 rows, more than 5 blocks per unit, tiles that fill under 85 % of the units,
// fewer than two K steps per wave, offsets past 32 bits or scales that do not fit the LDS.
inline int streamcu_tnw(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t as_m, int cus) {
    if (M > 16 || cus <= 0) return 0;
    const int64_t blocks = (N + 15) / 16, KB = K / kBlockK;
    const int64_t tnw = (blocks + cus - 1) / cus;
    if (tnw > 5 || KB < 16 || KB > CuStreamCfg<1, 1>::max_steps()) return 0;
    const int64_t tiles = (blocks + tnw - 1) / tnw;
    if (tiles * 20 < (int64_t)cus * 17) return 0;
    if (N * ldw >= (1ll << 32) || M * lda >= (1ll << 32) || M * as_m >= (1ll << 32)) return 0;
    if (8 * ((16 * tnw + 16) * 128) + KB * (17 + 2) * 4 > kMaxLds) return 0;
    return (int)tnw;
}

// Where it is ahead of the streaming kernel (M = 1 / 8 / 16, weights rotated past the memory-side cache): wherever
// that kernel has to share K between workgroups (N = 4096, K = 14336: 12.3 - 13.0 / 12.6 - 13.4 / 13.6 - 14.4 us
// against 13.4 / 13.7 / 14.9; N = 7168, K = 18432: 23.1 / 23.9 / 25.4 against 26.6 / 28.8 / 30.9), and from three
// row blocks per unit on, where the 64-row tiles fill their last round badly (N = 14336, K = 4096: 13.4 / 13.5 / 14.0
// against 14.5 / 15.0 / 16.0; N = 18432, K = 7168: 23.4 / 23.3 / 23.6 against 23.0 / 24.0 / 27.1).  With one or two
// blocks per unit and K unshared the 16-row tiles of the streaming kernel are ahead (N = 7168, K = 8192: 16.6
// against 12.9).
inline bool streamcu_pays(int64_t M, int64_t N, int64_t K, int cus) {
    const int tnw = streamcu_tnw(M, N, K, K, K, K / kBlockK, cus);
    if (tnw == 0) return false;
    return skinny_plan(M, N, K, cus).splits > 1 || tnw >= 3;
}

}  // namespace mi355
