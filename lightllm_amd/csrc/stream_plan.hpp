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

// Where in its K range (of at least `steps` K steps) a tile starts: GemmArgs::turn_mask.  With rows a multiple of 4 KiB apart the
// same K step of every row lies in the same few memory channels, and tiles that walk K in step queue there; started at
// different steps they spread.  (K stands for the distance: a result does not depend on how a weight is padded.  It does depend
// on the tile a weight row lies in.)  With any other distance the rows do that by themselves and turning only costs
// (K = 14336: 0 to 5 % slower), and a range of fewer than 32 steps - 4 KiB of a row - is spread by its neighbours already.
// us, in step / turned: N = 6144, K = 4096, M = 1 8.1 / 7.4; 28672 x 4096 21.0 / 19.5; 12288 x 4096 13.7 / 11.7; 57344 x 8192
// 78.5 / 70.8; 8192 x 8192, M = 48, whole K on eight waves 21.8 / 17.3; a shared K of 16 steps is 1 to 3 % slower turned.
inline int stream_turn_mask(int64_t K, int steps) {
    if (K % 4096 != 0 || steps < 32) return 0;
    int m = 0;
    while (2 * m + 1 < steps) m = 2 * m + 1;
    return m;
}

// The same for the stream cut into one share per unit.  Not where tile t's weight rows start 5 t times 2^18 bytes on and its first
// step 5 t times 2^7: the two meet on the same channels again (N = 19200, K = 16384, M = 6 55.6 us in step, 57.6 turned).
inline int streamcu_turn_mask(int64_t K, int tnw) {
    return tnw == 5 && K == 16384 ? 0 : stream_turn_mask(K, (int)(K / kBlockK));
}

// ---- the stream in tiles of 16, 32 or 64 weight rows, M <= 64
inline int skinny_mt(int64_t M) { return M <= 16 ? 1 : (int)((M + 15) / 16); }

struct SkinnyPlan {
    int tnw, splits, tiles;
    int waves;
    bool staged = true;  // from 17 rows on: the activation scales of a workgroup's K range are staged in LDS
    bool deep = false;   // two K steps in flight per wave instead of one
};

// K whole without a workspace and for any K: 64-row tiles on four waves, the scales gathered step by step.
inline SkinnyPlan skinny_whole_plan(int64_t N) { return {4, 1, (int)((N + 63) / 64), 4, false}; }

// Where a caller's own choice of the streaming kernel runs so if the workspace of its plan is missing: N alone gives the units
// work.
inline bool skinny_runs_whole(int64_t M, int64_t N, int cus) { return M > 16 && M <= 64 && (N + 31) / 32 * 2 >= 3 * (int64_t)cus; }

// 17..64 rows: four or eight waves a workgroup, tiles of 16, 32 or 64 weight rows, K whole or shared by up to eight
// workgroups.  What a launch takes, in ns and beside what all of them have in common: for each of the busiest unit's workgroups
// 288, and for each of its K steps 14 for 16 weight rows and 16 for 16 rows of activations (they come from the L2; every
// workgroup reads all rows of its K range); 109 for each K step in a wave's sequence, 162 + 6.5 a wave for each accumulator (they
// are added up through LDS), 483 and 230 for each workgroup that shares a tile and 3.8 us for a further round.  Tiles of 64
// weight rows, one or none a unit, want 32 steps: under fewer, two of half the width are ahead (15616 x 2432, M = 23 9.6 us against
// 11.0).  K is shared from 32 steps on, so that a caller without a workspace keeps this kernel below (404 x 3456, M = 48, whole / in
// three 7.7 / 7.3 us), and the partial sums stay within what the entry point without a workspace holds.
// Fitted to every candidate timed on 1179 shapes (M = 17..64, N = 100..139000, K = 1024..21500, weights from HBM): the choice is
// 0.9 % behind the best candidate on average and on 8 shapes more than 4 % behind the plan of before the eight-wave
// forms, which ran 32- or 64-row tiles on four waves with K shared until there were two workgroups a unit.  (A fit to 22 shapes
// of model linears, part of whose weights came from the memory-side cache, charged the weights at 41 and nothing for the
// accumulators and was behind that plan on 70: 15722 x 1152, M = 62 12.1 us against 9.9; 8581 x 1280, M = 19 7.4 / 6.6.)  us,
// that plan in brackets: N = K = 4096, M = 20 / 48 / 64 7.3 / 8.6 / 9.7 (8.9 / 10.0 / 10.1), 6144 x 4096 8.5 / 10.3 / 11.6
// (10.2 / 12.3 / 12.8), 4096 x 14336 14.5 / 17.3 / 19.5 (14.9 / 18.8 / 20.1), 28672 x 4096 21.5 / 24.9 (23.8 / 30.1).
inline int64_t skinny_wide_lds(int waves, int tnw, int mt, int64_t steps) {
    const int64_t wave = (16 * tnw + 16 * (mt < 4 ? mt : 4)) * 128, acc = (int64_t)tnw * mt * 1024;
    return waves * (wave > acc ? wave : acc) + 16 + steps * (16 * mt + 1) * 4;
}

// K steps of a workgroup whose activation scales fit: the LDS behind eight waves, 15 KiB behind four (two workgroups a unit).
inline int64_t skinny_wide_cap(int waves, int tnw, int mt) {
    const int64_t room = waves == 8 ? kMaxLds - skinny_wide_lds(8, tnw, mt, 0) : 15 * 1024;
    const int64_t steps = room / ((16 * mt + 1) * 4), most = waves == 8 ? 160 : 64;
    return steps < most ? steps : most;
}

// Workgroups on a unit at a time, by registers (one or two waves a SIMD) and by LDS.
inline int64_t skinny_wide_slots(int waves, int tnw, int mt, int64_t steps) {
    const bool two = waves == 8 ? tnw > 1 : tnw * mt >= 8;
    const int64_t slots = tnw * mt == 16 ? 1 : (two ? 8 / waves : 4);
    const int64_t by_lds = kMaxLds / skinny_wide_lds(waves, tnw, mt, steps);
    return slots < by_lds ? slots : (by_lds > 0 ? by_lds : 1);
}

inline SkinnyPlan skinny_wide_plan(int64_t M, int64_t N, int64_t K, int cus) {
    const int mt = skinny_mt(M);
    const int64_t KB = K / kBlockK;
    SkinnyPlan best = {0, 1, 0, 8};
    int64_t best_cost = 0;
    // four row blocks in four rounds of 64-row tiles, K beyond what four waves stage: 76224 x 17152, M = 64 324 us, 362 for the
    // best staged form
    if (mt == 4 && KB > skinny_wide_cap(4, 4, mt) && (N + 63) / 64 >= 4 * (int64_t)cus) return skinny_whole_plan(N);
    for (int waves = 4; waves <= 8; waves += 4)
        for (int tnw = 1; tnw <= 4; tnw *= 2) {
            if (waves == 8 && tnw == 4 && mt == 4) continue;  // 128 KiB of LDS and half the registers: not built
            const int64_t tiles = (N + 16 * tnw - 1) / (16 * tnw), cap = skinny_wide_cap(waves, tnw, mt);
            if (tnw == 4 && KB < 32 && tiles <= cus) continue;
            if (tiles * 4 > MI355_WS_COUNTER_BYTES) continue;  // one arrival counter a tile
            for (int s = 1; s <= 8; ++s) {
                const int64_t wgs = tiles * s, steps = (KB + s - 1) / s;
                if (s > 1 && (KB < 32 || KB / s < 2 * waves || 2 * wgs > 5 * (int64_t)cus || wgs * mt * tnw > MI355_NOALLOC_PARTIAL_MIB * 1024)) break;
                if (steps > cap) continue;
                const int64_t slots = skinny_wide_slots(waves, tnw, mt, steps);
                const int64_t per_unit = (wgs + cus - 1) / cus, rounds = (wgs + cus * slots - 1) / (cus * slots);
                const int64_t cost = per_unit * (steps * (14 * tnw + 16 * mt) + 288) + 109 * ((steps + waves - 1) / waves) +
                                     (324 + 13 * waves) * tnw * mt / 2 + (s > 1 ? 483 + 230 * s : 0) + 3775 * (rounds - 1);
                if (best.tnw == 0 || cost < best_cost) {
                    best = {tnw, s, (int)tiles, waves};
                    best_cost = cost;
                }
            }
        }
    // a K range too long for the staged forms, on more tiles than share it: N = 72704, K = 21376, M = 39 335 us (366 with a second
    // K step in flight, 551 with K shared by two)
    if (best.tnw == 0) return skinny_whole_plan(N);
    // 32 rows: 64-row tiles in four rounds and more take a second K step in flight (N = 73856, K = 4864, M = 22 64.1 us against
    // 67.9 with one, 79744 x 2688, M = 24 40.6 / 43.2; level from 2 to 4 rounds; three row blocks lose a third by it)
    best.deep = mt == 2 && best.waves == 4 && best.tnw == 4 && best.splits == 1 && best.tiles >= 4 * (int64_t)cus;
    return best;
}

inline SkinnyPlan skinny_plan(int64_t M, int64_t N, int64_t K, int cus) {
    if (M > 16) return skinny_wide_plan(M, N, K, cus);
    SkinnyPlan pl;
    pl.splits = 1;
    pl.waves = 4;
    const int64_t t64 = (N + 63) / 64;
    // 64-row tiles that come to just over one per unit leave half the units with twice the work of the others:
    // narrower tiles then (N = 18432, K = 7168, 288 tiles of 64 rows, M = 1 / 16: 22.6 / 26.8 us against 27.9 /
    // 29.9; N = 18944, K = 3584: 13.2 / 15.2 against 16.4 / 17.3)
    bool unbalanced = t64 > cus && t64 * 4 <= (int64_t)cus * 5;
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
    // on N=4096, K=14336: 16-row tiles x 2 splits 13.1 us at M <= 8 against 14.1 for 64-row tiles x 4 splits), never
    // below 16 K steps per workgroup (4 per wave).
    pl.tnw = 1;
    pl.tiles = (int)((N + 15) / 16);
    const int KB = (int)(K / kBlockK);
    pl.splits = (2 * cus + pl.tiles - 1) / pl.tiles;
    // from 1.5 tiles per unit on K stays whole: two splits would make 3 to 4 workgroups per unit and an exchange
    // (N = 7168, K = 8192, 448 tiles, M = 1 / 16: 12.8 / 13.7 us against 16.7 / 17.9; 6912 x 6912, M = 1: 10.2 against
    // 12.3)
    if (pl.tiles * 2 >= 3 * cus) pl.splits = 1;
    const int max_splits = KB / 16 > 0 ? KB / 16 : 1;
    if (pl.splits > max_splits) pl.splits = max_splits;
    if (pl.splits < 1) pl.splits = 1;
    // a workgroup stages the activation scales of its K range in LDS if the range is short enough; one more split
    // that gets it there pays (N=7168, K=18432, M=16: 72 steps unstaged 37.5 us, 48 steps staged 30.7)
    const int cap = StreamCfg<1, 1>::kMaxScaleSteps;
    const int need = (KB + cap - 1) / cap;
    if (pl.splits < need && need <= max_splits) pl.splits = need;
    return pl;
}

// 65..128 rows: the same kernel on eight waves, one workgroup a unit in one round, against the weight stream with the
// activation block in LDS, whose tiles are wide and share K over a second launch where N is narrow.  Both times are models in
// ns, fitted to 38 (N, K) pairs (N = 512..28672, K = 1536..18432) at M = 65..128: this kernel's by what a workgroup does
// (234 points, 4 % rms), the other's by its rows and the weights' size (158 points, 6 % rms).  What is taken is 0.4 % behind
// the better of all candidates on average.  us, M = 72 / 96 / 128, before in brackets: N = K = 4096 11.3 / 12.4 / 14.6 (15.6
// / 17.0 / 18.7), 6144 x 4096 13.0 / 14.6 (16.0 / 17.1), 7168 x 2048 9.0 / 10.1 (15.2 / 16.6), 2112 x 7168 12.0 / 13.5 (16.0 /
// 17.2), M = 128 there stays.  32 weight rows stop at 112: with eight row blocks the accumulators spill (6144 x 4096, M =
// 128: 25.9 against 18.4).  Up to 512 weight rows the other kernel keeps the launch, whose sums are compared by name with the
// table's, although this one is ahead (512 x 7168, M = 80 / 128: 9.0 / 10.8 against 11.9 / 13.6).  tnw 0: not here.
inline SkinnyPlan skinny_many_rows_plan(int64_t M, int64_t N, int64_t K, int cus) {
    SkinnyPlan best = {0, 1, 0, 8};
    if (M <= 64 || M > 128 || N <= 512 || K % kBlockK != 0 || K / kBlockK < 16) return best;
    const int64_t mt = (M + 15) / 16, KB = K / kBlockK;
    const int64_t weights = (N * K + 999999) / 1000000;  // MB
    const int64_t alternative = 8228 + 713 * mt + weights * (902 + 109 * mt) / 10 + 19 * KB;
    int64_t best_cost = alternative - alternative / 33;
    for (int tnw = 1; tnw <= (mt < 8 ? 2 : 1); ++tnw) {
        const int64_t tiles = (N + 16 * tnw - 1) / (16 * tnw), cap = skinny_wide_cap(8, tnw, (int)mt);
        for (int s = 1; s <= 8; ++s) {
            const int64_t steps = (KB + s - 1) / s;
            if (tiles * s > cus || KB / s < 8) break;
            if (steps > cap) continue;
            const int64_t cost = 3433 + 264 * mt + steps * (145 * tnw + 220 * mt + 68 * mt * tnw) / 10 +
                                 124 * ((steps + 7) / 8) + (s > 1 ? 1764 + 169 * s : 0) + weights * 56;
            if (cost < best_cost) {
                best = {tnw, s, (int)tiles, 8};
                best_cost = cost;
            }
        }
    }
    return best;
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

// (K a multiple of 4096: the streaming kernel gains more from turned starts than this one, whose workgroups have most
// of the range in flight anyway - N = 12288, K = 4096, M = 1 / 16: 10.4 / 11.3 us against 11.7 / 12.2 here; 20480: 15.2 /
// 16.7 against 16.5 / 16.8; from four row blocks a unit and 9 rows on this one is level or ahead: 18432: 16.3 / 15.8.)
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
    if (skinny_plan(M, N, K, cus).splits > 1) return true;
    return K % 4096 == 0 ? tnw >= 4 && M > 8 : tnw >= 3;
}

}  // namespace mi355
