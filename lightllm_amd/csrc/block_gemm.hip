// Host side of the block-scaled FP8 GEMM entry points: argument checks, kernel choice, launches.
#include <algorithm>

#include "gemm_gstream.hpp"
#include "gemm_pp.hpp"
#include "gemm_small.hpp"
#include "gemm_stream.hpp"
#include "gemm_streamcu.hpp"
#include "gemm_xshare.hpp"
#include "rows128_launch.hpp"
#include "gemm_tile.hpp"
#include "stream_plan.hpp"

namespace mi355 {

// Correctness fallback for layouts the MFMA kernels do not take (B not K-contiguous, K not a multiple of
// 128, unaligned leading dimensions).  One thread per output element, same per-block arithmetic.
__device__ __forceinline__ float e4m3_to_f32(uint8_t b) {
    const uint32_t sign = (uint32_t)(b & 0x80u) << 24;
    const uint32_t e = (b >> 3) & 0xfu, m = b & 7u;
    float v;
    if (e == 0) v = (float)m * 0.001953125f;  // m * 2^-9
    else v = as_f32(((e + 120u) << 23) | (m << 20));
    return as_f32(as_u32(v) | sign);
}

__global__ __launch_bounds__(256) void block_fp8_gemm_generic_kernel(
    const uint8_t *__restrict__ A, const uint8_t *__restrict__ B, const float *__restrict__ As,
    const float *__restrict__ Bs, uint16_t *__restrict__ C, int M, int N, int K, int64_t lda, int64_t ldb_k,
    int64_t ldb_n, int64_t ldc, int64_t as_m, int64_t as_k, int64_t bs_k, int64_t bs_n, int block_n, int block_k,
    int out_f16) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)M * N) return;
    const int m = (int)(idx / N), n = (int)(idx % N);
    float acc = 0.f;
    int kb = 0;
    for (int k0 = 0; k0 < K; k0 += block_k, ++kb) {
        const int k1 = min(k0 + block_k, K);
        float d = 0.f;
        for (int k = k0; k < k1; ++k) d += e4m3_to_f32(A[m * lda + k]) * e4m3_to_f32(B[k * ldb_k + n * ldb_n]);
        acc += d * As[m * as_m + kb * as_k] * Bs[kb * bs_k + (n / block_n) * bs_n];
    }
    C[m * ldc + n] = (uint16_t)out_bits(acc, out_f16);
}

// X scales that can be fetched eight K steps at a time: row-major, 16-byte aligned rows, K/128 % 8 == 0.
static bool chunked_scales_ok(const GemmArgs &a) {
    return a.xs_k == 1 && (a.K / kBlockK) % 8 == 0 && a.xs_m % 4 == 0 && ((uintptr_t)a.Xs & 15) == 0;
}

template <int BM, int BN, int WM, int WN, int NSTAGE, int MODE, bool XS8, bool BIAS = false>
static int launch_tile_as(GemmArgs &a, int grid, hipStream_t st) {
    using Cfg = TileCfg<BM, BN, WM, WN, NSTAGE>;
    constexpr auto kernel = block_fp8_gemm_tile_kernel<BM, BN, WM, WN, NSTAGE, MODE, XS8, BIAS>;
    const int KB = a.K / kBlockK;
    // chunked scales keep two [BM rows][8 steps] buffers behind the common layout
    const int lds_bytes = XS8 ? ((Cfg::lds_bytes(KB) + 127) & ~127) + 2 * BM * 32 : Cfg::lds_bytes(KB);
    if (lds_bytes > kMaxLds) return MI355_EUNSUPPORTED;
    if (!allow_lds<kernel>(kMaxLds)) return MI355_ELAUNCH;
    return launch(kernel, dim3(grid), dim3(Cfg::kThreads), lds_bytes, st, a);
}

template <int BM, int BN, int WM, int WN, int NSTAGE, int MODE, bool BIAS = false>
static int launch_tile(GemmArgs &a, int grid, hipStream_t st) {
    using Cfg = TileCfg<BM, BN, WM, WN, NSTAGE>;
    constexpr bool kFits = ((Cfg::lds_bytes(144) + 127) & ~127) + 2 * BM * 32 <= kMaxLds;  // up to K = 18432
    if constexpr (kFits) {
        if (chunked_scales_ok(a)) {
            const int r = launch_tile_as<BM, BN, WM, WN, NSTAGE, MODE, true, BIAS>(a, grid, st);
            if (r != MI355_EUNSUPPORTED) return r;
        }
    }
    return launch_tile_as<BM, BN, WM, WN, NSTAGE, MODE, false, BIAS>(a, grid, st);
}

// A grouped launch of ring tiles, with or without the per-expert bias.
template <int BM, int BN, int WM, int WN, int NSTAGE>
static int launch_grouped_tile(GemmArgs &a, int grid, hipStream_t st) {
    if (a.bias) return launch_tile<BM, BN, WM, WN, NSTAGE, kGrouped, true>(a, grid, st);
    return launch_tile<BM, BN, WM, WN, NSTAGE, kGrouped, false>(a, grid, st);
}

// A grouped launch of weight streams over the entries of a 16- or 32-row schedule.
template <bool BIAS>
static int launch_gstream_as(GemmArgs &a, int block_m, int num_experts, hipStream_t st) {
    const int KB = a.K / kBlockK;
    const int lds_bytes = GStreamCfg<2>::lds_bytes(KB);
    if (lds_bytes > kMaxLds) return MI355_EUNSUPPORTED;
    a.tiles_n = (a.N + GStreamCfg<1>::BN - 1) / GStreamCfg<1>::BN;
    if ((int64_t)a.tiles_m * a.tiles_n >= (1ll << 31)) return MI355_EUNSUPPORTED;
    a.total_tiles = a.tiles_m * a.tiles_n;
    // an exact schedule has at most E more entries than it would with every block full
    const int64_t grid = std::max<int64_t>(4096, 2 * (int64_t)num_experts * a.tiles_n);
    if (a.total_tiles <= grid) {
        constexpr auto kernel = block_fp8_gemm_gstream_kernel<BIAS, false>;
        if (!allow_lds<kernel>(kMaxLds)) return MI355_ELAUNCH;
        return launch(kernel, dim3(a.total_tiles), dim3(256), lds_bytes, st, a, block_m);
    }
    constexpr auto kernel = block_fp8_gemm_gstream_kernel<BIAS, true>;
    if (!allow_lds<kernel>(kMaxLds)) return MI355_ELAUNCH;
    return launch(kernel, dim3((uint32_t)grid), dim3(256), lds_bytes, st, a, block_m);
}
static int launch_gstream(GemmArgs &a, int block_m, int num_experts, hipStream_t st) {
    return a.bias ? launch_gstream_as<true>(a, block_m, num_experts, st) : launch_gstream_as<false>(a, block_m, num_experts, st);
}

#ifndef MI355_SK_PANEL
#define MI355_SK_PANEL 1
#endif
// Runs per tile of the panel split (0 = none; otherwise tiles * runs is within the compute units).  A K step takes a
// workgroup 1.3 us and the partial tiles, written once and read once, 0.1 us each, so there are as many runs as make
// 1.3 steps + 0.1 tiles * runs least (us, runs: M = 256, N = 7168, K = 14336 54.3 / 51.7 / 48.6 / 49.5 / 50.2 with 5 .. 9, 7
// here; M = 512, N = 2560, K = 20480 46.1 / 44.5 / 46.0 with 9 .. 11, 10 here; M = 640, N = 7168, K = 18432 177.9 /
// 106.4 / 98.5 with 1 .. 3, which is what the units allow).
static int sk_panel_splits(int tiles_m, int tiles_n, int KB, int cus) {
    const int64_t tiles = (int64_t)tiles_m * tiles_n;
    int best = 0;
    int64_t best_cost = 0;
    for (int s = 2; s <= 32 && tiles * s <= cus && KB / s >= 8; ++s) {
        const int64_t cost = 13 * ((KB + s - 1) / s) + tiles * s;
        if (best == 0 || cost < best_cost) {
            best = s;
            best_cost = cost;
        }
    }
    return best;
}

// Stream-K plan of the 256x256 kernel: the number of workgroups (one per compute unit, a multiple of 8), or 0 when
// the tiles fill whole rounds anyway or there is too little work to give every unit 16 K steps (the 128x128
// split-K tiles take those shapes).
static int stream_k_groups(int64_t tiles, int64_t KB, int cus, int64_t tiles_m = 0) {
    if (cus < 8 || tiles <= 0) return 0;
    // a panel split (see launch_pp) stands in for the cut of the unit sequence wherever the shape has one
    if (MI355_SK_PANEL && tiles_m > 0 && tiles % tiles_m == 0 &&
        sk_panel_splits((int)tiles_m, (int)(tiles / tiles_m), (int)KB, cus) > 0)
        return cus / 8 * 8;
    const int64_t units = tiles * KB;
    if (units >= (1ll << 31)) return 0;
    const int64_t groups = cus / 8 * 8;
    if (units / 16 < groups || tiles % groups == 0) return 0;
    return (int)groups;
}

// Whether the shape table should take that plan.  A workgroup that shares tiles no longer runs in step with the
// ones that read the same X and W panels, so its K steps are served by the memory side instead of the L2 and take
// about 2.5 times as long: sharing pays only where the plain loop leaves most of the device idle.
static bool stream_k_pays(int64_t tiles, int64_t KB, int cus, int64_t tiles_m) {
    // a panel split that fills three eighths of the device with runs of a long K: measured ahead of every other
    // kernel from 385 rows on, behind them with K = 4096 (us, before / here, 5 % slower to 64 % faster over 260 shapes of 385..4096 rows:
    // 640 x 7168 x 18432 123 / 104, 640 x 4096 x 7168 57 / 40, 700 x 5120 x 13824 93 / 67, 1280 x 5120 x 8192 96 / 69,
    // 1772 x 3760 x 27392 281 / 177; 1024 x 7168 x 18432, one workgroup per tile, 164 / 135)
    const int panel = tiles % tiles_m == 0 ? sk_panel_splits((int)tiles_m, (int)(tiles / tiles_m), (int)KB, cus) : 0;
    // (one m tile on a narrow N: the 128-row tiles are ahead; more are compared in pick_variant)
    const bool few = tiles_m == 1 && (tiles * 64 < 3 * (int64_t)cus || (tiles * 32 < 3 * (int64_t)cus && KB < 96));
    // three m tiles under a short K or on a narrow N keep the name of the 256x128 tiles, which share K the same way and with which
    // launches by name are compared, although the panel split is ahead (600 x 5120 x 6144 52 us against 42, 768 x 2112 x 8192 36.5 /
    // 34.0); below K = 8192 AUTO runs them over M
    const bool kept = tiles_m == 3 && (KB <= 48 || (tiles <= 27 && KB <= 64));
    if (MI355_SK_PANEL && panel > 0 && KB >= 40 && tiles * panel * 8 >= (int64_t)cus * 3 && !few && !kept) return true;
    const int groups = stream_k_groups(tiles, KB, cus);
    if (groups == 0) return false;
    const int64_t plain = (tiles + groups - 1) / groups * KB, shared = (tiles * KB + groups - 1) / groups;
    if (shared * 5 <= plain * 2) return true;
    // every tile shared by the same whole number of workgroups, none of which straddles two tiles, is a plain split
    // of K with half the partial tiles: it still pays at two workgroups per tile when their runs are long
    // (N = 4096, K = 14336, M = 2048: 128 tiles, 111 us against 130; N = 16384, K = 7168, M = 512, 28 steps each: 70.0
    // against 77.8; with K = 4096, 16 steps each, 51.6 against 43.7)
    return groups % tiles == 0 && shared * 2 <= plain && shared >= 28;
}

static size_t stream_k_workspace(int groups) {
    return (size_t)MI355_WS_COUNTER_BYTES + (size_t)2 * groups * PPCfg::kPartialBytes;
}

// The 256x256 ping-pong kernel.  a.tiles_m / a.tiles_n / a.total_tiles are set by the caller.  With a workspace
// whose counter words are zero the launch is persistent (one workgroup per CU, tiles handed out per XCD);
// without one every workgroup runs a single tile.  `sk_groups` > 0 asks for the stream-K launch with that many
// workgroups (dense only; the workspace must hold stream_k_workspace(sk_groups)).  Returns MI355_EUNSUPPORTED
// when the K range does not fit the kernel's LDS layout.
template <bool GROUPED, bool SK, bool SC4, bool BIAS = false>
static int launch_pp_as(GemmArgs &a, int grid, int lds_bytes, hipStream_t st) {
    constexpr auto kernel = block_fp8_gemm_pp_kernel<GROUPED, SK, SC4, false, BIAS>;
    if (!allow_lds<kernel>(kMaxLds)) return MI355_ELAUNCH;
    return launch(kernel, dim3(grid), dim3(PPCfg::kThreads), lds_bytes, st, a);
}

template <bool GROUPED>
static int launch_pp(GemmArgs &a, void *ws, size_t ws_bytes, int cus, int sk_groups, hipStream_t st) {
    const int lds_bytes = PPCfg::lds_bytes(a.K / kBlockK);
    if (lds_bytes > kMaxLds) return MI355_EUNSUPPORTED;
    if (a.xs_m < 0 || a.xs_k < 0) return MI355_EUNSUPPORTED;
    const bool sc4 = chunked_scales_ok(a);
    a.blocks_per_xcd = (a.total_tiles + 7) / 8;
    int per_xcd = a.blocks_per_xcd;
    a.counters = nullptr;
    const bool ws_ok = ws && ((uintptr_t)ws & 15) == 0;
    if constexpr (!GROUPED) {
        if (sk_groups > 0) {
            if (!ws_ok || ws_bytes < stream_k_workspace(sk_groups)) return MI355_EWORKSPACE;
            a.counters = (uint32_t *)ws;
            a.partials = (float *)((uint8_t *)ws + MI355_WS_COUNTER_BYTES);
            // panel split where the shape allows it: every tile's K range in the same few runs (the grid is rounded up to the
            // 8 XCDs)
            a.splits = MI355_SK_PANEL ? sk_panel_splits(a.tiles_m, a.tiles_n, a.K / kBlockK, cus) : 0;
            if (a.splits > 0) sk_groups = (a.total_tiles * a.splits + 7) / 8 * 8;
            const int r = sc4 ? launch_pp_as<false, true, true>(a, sk_groups, lds_bytes, st)
                              : launch_pp_as<false, true, false>(a, sk_groups, lds_bytes, st);
            if (r != MI355_OK) return r;
            return launch(streamk_reduce_kernel, dim3(a.total_tiles * PPCfg::TM), dim3(PPCfg::kThreads), 0, st, a,
                          (uint32_t)sk_groups);
        }
    }
    // persistent only when there is more than one tile per CU (a single round gains nothing from the tile queue)
    if (ws_ok && ws_bytes >= (size_t)MI355_WS_COUNTER_BYTES && per_xcd > cus / 8 && cus >= 8) {
        a.counters = (uint32_t *)ws;
        per_xcd = cus / 8;
    }
    if constexpr (GROUPED) {
        if (a.bias)
            return sc4 ? launch_pp_as<true, false, true, true>(a, per_xcd * 8, lds_bytes, st)
                       : launch_pp_as<true, false, false, true>(a, per_xcd * 8, lds_bytes, st);
    }
    return sc4 ? launch_pp_as<GROUPED, false, true>(a, per_xcd * 8, lds_bytes, st)
               : launch_pp_as<GROUPED, false, false>(a, per_xcd * 8, lds_bytes, st);
}

// Grouped launch over a 256-row schedule.  With a workspace that also holds the two block lists
// (grouped_workspace) the blocks of at most 64 rows go to the 64x512 streaming tile inside the same persistent
// launch: some workgroups of every XCD start on them, the others on the large blocks, and each moves on to the
// other queue when its own is empty.
static size_t grouped_workspace(int64_t table_rows) {
    return (size_t)MI355_WS_COUNTER_BYTES + (((size_t)(2 + 2 * table_rows) * 4 + 255) & ~(size_t)255);
}

template <auto Kernel>
struct KernelTag {
    static constexpr auto value = Kernel;
};

static int launch_grouped_pp(GemmArgs &a, void *ws, size_t ws_bytes, int cus, hipStream_t st) {
    const int KB = a.K / kBlockK;
    const int lds_roles = PPCfg::roles_sched_off(KB) + 16;
    const bool ws_ok = ws && ((uintptr_t)ws & 15) == 0 && ws_bytes >= grouped_workspace(a.tiles_m);
    if (!ws_ok || cus < 8 || a.total_tiles <= cus || lds_roles > kMaxLds || a.xs_m < 0 || a.xs_k < 0)
        return launch_pp<true>(a, ws, ws_bytes, cus, 0, st);
    int32_t *lists = (int32_t *)((uint8_t *)ws + MI355_WS_COUNTER_BYTES);
    const int r = launch(grouped_split_kernel, dim3(1), dim3(1024), 0, st, a.table, a.tiles_m, lists);
    if (r != MI355_OK) return r;
    a.lists = lists;
    a.counters = (uint32_t *)ws;
    a.blocks_per_xcd = (a.total_tiles + 7) / 8;
    const int per_xcd = cus / 8;
    a.small_first = per_xcd * 3 / 8;  // measured on the 256-expert routed batch: 8..14 of 32 are within 3 %
    auto go = [&](auto kernel_tag) {
        constexpr auto kernel = decltype(kernel_tag)::value;
        if (!allow_lds<kernel>(kMaxLds)) return (int)MI355_ELAUNCH;
        return launch(kernel, dim3(per_xcd * 8), dim3(PPCfg::kThreads), lds_roles, st, a);
    };
    const bool sc4 = chunked_scales_ok(a);
    if (a.bias)
        return sc4 ? go(KernelTag<block_fp8_gemm_pp_kernel<true, false, true, true, true>>{})
                   : go(KernelTag<block_fp8_gemm_pp_kernel<true, false, false, true, true>>{});
    return sc4 ? go(KernelTag<block_fp8_gemm_pp_kernel<true, false, true, true>>{})
               : go(KernelTag<block_fp8_gemm_pp_kernel<true, false, false, true>>{});
}

template <int BM, int BN, int WM, int WN, int NSTAGE, int MODE = kDense>
static int launch_dense(GemmArgs &a, hipStream_t st) {
    a.tiles_m = (a.M + BM - 1) / BM;
    a.tiles_n = (a.N + BN - 1) / BN;
    a.total_tiles = a.tiles_m * a.tiles_n;
    a.blocks_per_xcd = (a.total_tiles + 7) / 8;
    return launch_tile<BM, BN, WM, WN, NSTAGE, MODE>(a, a.blocks_per_xcd * 8, st);
}

// Weight-streaming launches for M <= 64 (stream_plan.hpp has the plan).
template <int MT, int TNW, bool XSL, bool TURN, int WV, int DEEP = 0>
static int launch_stream_as(GemmArgs &a, const SkinnyPlan &pl, void *ws, int lds_bytes, hipStream_t st) {
    using Cfg = StreamCfg<MT, TNW, WV>;
    constexpr int max_lds = Cfg::kLds + (XSL ? Cfg::scale_lds_bytes(Cfg::kMaxScaleSteps) : 0);
    if (pl.splits <= 1) {
        constexpr auto whole_k = block_fp8_gemm_stream_kernel<MT, TNW, false, XSL, 0, false, WV, TURN, DEEP>;
        if (!allow_lds<whole_k>(max_lds)) return MI355_ELAUNCH;
        return launch(whole_k, dim3(pl.tiles), dim3(64 * WV), lds_bytes, st, a);
    }
    if constexpr (DEEP == 0 && (MT == 1 || XSL)) {
        constexpr auto split_k = block_fp8_gemm_stream_kernel<MT, TNW, true, XSL, 0, false, WV, TURN>;
        if (!allow_lds<split_k>(max_lds)) return MI355_ELAUNCH;
        a.splits = pl.splits;
        a.counters = (uint32_t *)ws;
        a.partials = (float *)((uint8_t *)ws + MI355_WS_COUNTER_BYTES);
        return launch(split_k, dim3(pl.tiles * pl.splits), dim3(64 * WV), lds_bytes, st, a);
    }
    return MI355_EUNSUPPORTED;
}

template <int MT, int TNW, bool XSL, int WV, int DEEP = 0>
static int launch_stream_form(GemmArgs &a, const SkinnyPlan &pl, void *ws, int lds_bytes, hipStream_t st) {
    return a.turn_mask ? launch_stream_as<MT, TNW, XSL, true, WV, DEEP>(a, pl, ws, lds_bytes, st)
                       : launch_stream_as<MT, TNW, XSL, false, WV, DEEP>(a, pl, ws, lds_bytes, st);
}

// The activation scales of a CTA's K range are staged in LDS when the range is short enough for the staging area; from 17
// rows on the plan says so, and only 64-row tiles on four waves run without.  Up to 8 rows the quantizing stream (linear.hip)
// runs the same K order, so that the linear has the bits of quantizer + GEMM.
template <int MT, int TNW, int WV = kStreamWaves>
static int launch_stream(GemmArgs &a, const SkinnyPlan &pl, void *ws, hipStream_t st) {
    using Cfg = StreamCfg<MT, TNW, WV>;
    const int KB = a.K / kBlockK;
    const int steps = (KB + pl.splits - 1) / pl.splits;
    a.turn_mask = stream_turn_mask(a.K, KB / pl.splits);
    if (pl.staged && steps <= Cfg::kMaxScaleSteps) {
        const int lds_bytes = Cfg::kLds + Cfg::scale_lds_bytes(steps);
        if constexpr (MT == 2 && TNW == 4 && WV == 4) {
            if (pl.deep) return launch_stream_form<MT, TNW, true, WV, 2>(a, pl, ws, lds_bytes, st);
        }
        return launch_stream_form<MT, TNW, true, WV>(a, pl, ws, lds_bytes, st);
    }
    if constexpr (MT == 1 || (MT <= 4 && TNW == 4 && WV == 4)) return launch_stream_form<MT, TNW, false, WV>(a, pl, ws, Cfg::kLds, st);
    return MI355_EUNSUPPORTED;
}

template <int MT>
static int launch_stream_mt(GemmArgs &a, const SkinnyPlan &pl, void *ws, hipStream_t st) {
    if constexpr (MT == 1) {
        switch (pl.tnw) {
            case 4: return launch_stream<1, 4>(a, pl, ws, st);
            case 1: return launch_stream<1, 1>(a, pl, ws, st);
            default: return MI355_EINVAL;
        }
    } else {
        if (pl.waves == 8) {
            switch (pl.tnw) {
                case 4:
                    if constexpr (MT < 4) return launch_stream<MT, 4, 8>(a, pl, ws, st);
                    return MI355_EINVAL;
                case 2: return launch_stream<MT, 2, 8>(a, pl, ws, st);
                case 1: return launch_stream<MT, 1, 8>(a, pl, ws, st);
                default: return MI355_EINVAL;
            }
        }
        switch (pl.tnw) {
            case 4: return launch_stream<MT, 4>(a, pl, ws, st);
            case 2: return launch_stream<MT, 2>(a, pl, ws, st);
            case 1: return launch_stream<MT, 1>(a, pl, ws, st);
            default: return MI355_EINVAL;
        }
    }
}

// 65..128 rows (skinny_many_rows_plan)
template <int MT>
static int launch_stream_many_rows(GemmArgs &a, const SkinnyPlan &pl, void *ws, hipStream_t st) {
    if constexpr (MT < 8) {
        if (pl.tnw == 2) return launch_stream<MT, 2, 8>(a, pl, ws, st);
    }
    return launch_stream<MT, 1, 8>(a, pl, ws, st);
}

// ---- the weight stream cut into one equal share per compute unit (gemm_streamcu.hpp)
template <int TNW, bool TURN>
static int launch_streamcu_turn(GemmArgs &a, hipStream_t st) {
    using Cfg = CuStreamCfg<1, TNW>;
    constexpr auto kernel_lo = block_fp8_gemm_streamcu_kernel<1, TNW, false, 0, false, TURN>;
    constexpr auto kernel_hi = block_fp8_gemm_streamcu_kernel<1, TNW, true, 0, false, TURN>;
    const int lds_bytes = Cfg::lds_bytes(a.K / kBlockK);
    if (lds_bytes > kMaxLds) return MI355_EUNSUPPORTED;
    const int tiles = (a.N + Cfg::BN - 1) / Cfg::BN;
    if (a.M <= 8) {
        if (!allow_lds<kernel_lo>(kMaxLds)) return MI355_ELAUNCH;
        return launch(kernel_lo, dim3(tiles), dim3(Cfg::kThreads), lds_bytes, st, a);
    }
    if (!allow_lds<kernel_hi>(kMaxLds)) return MI355_ELAUNCH;
    return launch(kernel_hi, dim3(tiles), dim3(Cfg::kThreads), lds_bytes, st, a);
}

template <int TNW>
static int launch_streamcu_as(GemmArgs &a, hipStream_t st) {
    a.turn_mask = streamcu_turn_mask(a.K, TNW);
    return a.turn_mask ? launch_streamcu_turn<TNW, true>(a, st) : launch_streamcu_turn<TNW, false>(a, st);
}

static int launch_streamcu(GemmArgs &a, int tnw, hipStream_t st) {
    switch (tnw) {
        case 1: return launch_streamcu_as<1>(a, st);
        case 2: return launch_streamcu_as<2>(a, st);
        case 3: return launch_streamcu_as<3>(a, st);
        case 4: return launch_streamcu_as<4>(a, st);
        case 5: return launch_streamcu_as<5>(a, st);
        default: return MI355_EUNSUPPORTED;
    }
}

// ---- the second streaming kernel (activation block shared by the workgroup).  Measured against the first one on
// the Llama decode shapes it wins only where the first is shortest of registers and N alone fills the device:
// M = 49..64 with 128-row workgroup tiles (N=28672, K=4096, M=64: 29.7 us against 34.4); with 64-row tiles, few
// tiles or smaller M its barrier per K step costs more than the shared activation block saves
// (N=4096, K=14336: 21.5-25.2 us against 13.9-19.8; N = 28672, M = 48: 28.7 against 24.9 for three row blocks on the
// first kernel).  Only that configuration is built.  Turned starts (K whole): N = 128256, K = 4096, M = 64 125 us, 102 turned.
constexpr int kXshareDepth = 4;
using XshareCfg = ShareCfg<4, 2, kXshareDepth>;

// 33..48 rows: three row blocks on the first kernel are ahead where they run turned or in up to five rounds of 64-row tiles over 8
// K steps and more (N = 66176, K = 7424, M = 38 98.0 us against 119 here), this one beyond (86144 x 12672, M = 46 227 against 210;
// 116480 x 1280, M = 40 38.9 / 35.2; 79616 x 256, M = 34 12.9 / 10.3).
static bool xshare_pays(int64_t M, int64_t N, int64_t K, int cus) {
    if (M <= 32 || M > 64 || K / kBlockK > XshareCfg::kMaxScaleSteps || (N + 127) / 128 < (int64_t)cus * 3 / 4) return false;
    return M > 48 || (K % 4096 != 0 && (K < 1024 || (N + 63) / 64 >= 5 * (int64_t)cus));
}

// 128-row workgroup tiles; the K range is split in two while that leaves fewer than two workgroups per compute unit
// (224 tiles unsplit take 34.7 us on N=28672, K=4096, M=64; split in two, 29.7), never below 8 K steps each.
static int xshare_splits(int64_t N, int64_t K, int cus) {
    const int64_t tiles = (N + XshareCfg::BN - 1) / XshareCfg::BN, KB = K / kBlockK;
    return tiles < 2 * (int64_t)cus && KB >= 16 ? 2 : 1;
}

static size_t xshare_workspace(int64_t N, int splits) {
    const int64_t tiles = (N + XshareCfg::BN - 1) / XshareCfg::BN;
    return (size_t)MI355_WS_COUNTER_BYTES + (size_t)tiles * splits * XshareCfg::kTileElems * 4;
}

static int launch_xshare(GemmArgs &a, int splits, void *ws, hipStream_t st) {
    const int KB = a.K / kBlockK;
    const int steps = (KB + splits - 1) / splits;
    if (steps > XshareCfg::kMaxScaleSteps) return MI355_EUNSUPPORTED;
    constexpr int max_lds = XshareCfg::kLds + XshareCfg::scale_lds_bytes(XshareCfg::kMaxScaleSteps);
    const int lds_bytes = XshareCfg::kLds + XshareCfg::scale_lds_bytes(steps);
    const int tiles = (a.N + XshareCfg::BN - 1) / XshareCfg::BN;
    a.turn_mask = splits > 1 ? 0 : stream_turn_mask(a.K, KB);
    if (a.turn_mask) {
        constexpr auto kernel = block_fp8_gemm_xshare_kernel<4, 2, kXshareDepth, false, true>;
        if (!allow_lds<kernel>(max_lds)) return MI355_ELAUNCH;
        return launch(kernel, dim3(tiles), dim3(256), lds_bytes, st, a);
    }
    if (splits <= 1) {
        constexpr auto kernel = block_fp8_gemm_xshare_kernel<4, 2, kXshareDepth, false>;
        if (!allow_lds<kernel>(max_lds)) return MI355_ELAUNCH;
        return launch(kernel, dim3(tiles), dim3(256), lds_bytes, st, a);
    }
    constexpr auto kernel = block_fp8_gemm_xshare_kernel<4, 2, kXshareDepth, true>;
    if (!allow_lds<kernel>(max_lds)) return MI355_ELAUNCH;
    a.splits = splits;
    a.counters = (uint32_t *)ws;
    a.partials = (float *)((uint8_t *)ws + MI355_WS_COUNTER_BYTES);
    return launch(kernel, dim3(tiles * splits), dim3(256), lds_bytes, st, a);
}

// ---- at most 384 rows: the weight stream with the activation block in LDS (gemm_rows128.hpp).  Up to 128 rows a
// workgroup takes 256 weight rows on three ring slots, beyond that 128 weight rows on two (the activation block of a
// step is two to three times as large).
constexpr int kRows128MinSteps = 6;

static int rows128_mt(int64_t M) { return (int)((M + 15) / 16); }

// Workgroup width, K sharing and tile count of a launch.  Up to 128 rows a workgroup is 8 waves x 32 weight rows;
// beyond, 8 waves x 16.  While the tiles leave compute units idle the K range is shared, never below
// kRows128MinSteps K steps for a workgroup.  Up to 128 rows there is a second way to occupy the idle units: narrower
// workgroups (5 or 6 waves) with K unshared - a unit's pull covers the X block and the W rows of a step alike, so
// more, narrower workgroups mean fewer bytes per unit.  It is taken when such a width gives between 0.55 cus and cus
// tiles (DeepSeek-V3 gate_up, N = 36864: 231 tiles of 160 rows, M = 64 / 128: 50.3 / 62.8 us against 59.4 / 68.8
// for 144 tiles of 256; q_b, N = 24576, K = 1536: 16.6 against 21.4 with K shared by two).
struct RowsMPlan {
    int mt, wv, tiles_m, tiles_n;
};
static RowsMPlan rowsm_plan(int64_t M, int64_t N, int64_t K, int cus);
static bool rows128_over_m(int64_t M, int64_t N, int64_t K, int cus);  // two to four tiles over M: rowsm_plan's launch

static Rows128Plan rows128_plan(int64_t M, int64_t N, int64_t K, int cus) {
    Rows128Plan pl;
    const int64_t KB = K / kBlockK;
    pl.turned = false;
    if (rows128_over_m(M, N, K, cus)) {
        const RowsMPlan mp = rowsm_plan(M, N, K, cus);
        return {mp.wv, 32 * mp.wv, 1, mp.tiles_m * mp.tiles_n, 2, false};
    }
    pl.wv = 8;
    pl.bn = M <= 128 ? 256 : 128;
    pl.tn = M <= 128 ? 2 : 1;
    if (M <= 128) {
        for (int wv = 5; wv <= 6; ++wv) {
            const int64_t tiles = (N + 32 * wv - 1) / (32 * wv);
            if (tiles <= cus && tiles * 20 >= (int64_t)cus * 11) {
                pl.wv = wv;
                pl.bn = 32 * wv;
                pl.splits = 1;
                pl.tiles = (int)tiles;
                return pl;
            }
        }
    }
    if (M > 128 && M <= kRows128NarrowMaxM) {
        // one round of workgroups of just the width that fits it: two 16-row blocks per wave (5..8 waves, 160..256
        // weight rows) where N is wide enough for that, else one (4..7 waves, 64..112 weight rows)
        const int64_t wv2 = (N + 32 * (int64_t)cus - 1) / (32 * (int64_t)cus);
        int64_t wv1 = (N + 16 * (int64_t)cus - 1) / (16 * (int64_t)cus);
        if (wv1 < 4) wv1 = 4;
        const int tn = wv2 >= 5 ? 2 : 1;
        const int64_t wv = tn == 2 ? wv2 : wv1, bn = 16 * tn * wv;
        const int64_t tiles = (N + bn - 1) / bn;
        // (four-wave workgroups fall behind the 128x128 tiles a little earlier: N = 16384, K = 7168, M = 208: 63.6 us
        // against 60.9)
        if (wv <= (tn == 2 ? 8 : 7) && (wv > 4 || M <= 192) && tiles <= cus && tiles * 20 >= (int64_t)cus * 11) {
            pl.wv = (int)wv;
            pl.bn = (int)bn;
            pl.splits = 1;
            pl.tiles = (int)tiles;
            pl.tn = tn;
            return pl;
        }
    }
    const int64_t tiles = (N + pl.bn - 1) / pl.bn;
    int64_t splits = cus / tiles;
    if (splits > KB / kRows128MinSteps) splits = KB / kRows128MinSteps;
    pl.splits = (int)(splits < 1 ? 1 : splits);
    pl.tiles = (int)tiles;
    return pl;
}

static int rows128_splits(int64_t M, int64_t N, int64_t K, int cus) { return rows128_plan(M, N, K, cus).splits; }

static size_t rows128_workspace(int64_t M, int64_t N, int64_t K, int cus) {
    const Rows128Plan pl = rows128_plan(M, N, K, cus);
    if (pl.splits <= 1) return 0;
    return (size_t)MI355_WS_COUNTER_BYTES + (size_t)pl.tiles * pl.splits * 16 * rows128_mt(M) * pl.bn * 4;
}

// What the two weight streams take at 17..64 rows, in ns, where K is not a multiple of 4096 (turned starts make their own rules
// below).  Fitted to 1066 shapes of 20 MB and more (N = 900..139000, K = 1024..21500, weights from HBM; 5.0 and 5.6 % rms):
// taking the smaller is 0.2 % behind the faster one on average.  (Rules drawn from 22 model linears took the streaming kernel
// where it is up to 29 % behind, us, this one / that: N = 20992, K = 8576, M = 46 40.6 / 52.3; 55680 x 10240, M = 47 103 / 126;
// 50069 x 2688, M = 46 31.4 / 39.1.)
static int64_t rows128_ns(int64_t M, int64_t N, int64_t K, const Rows128Plan &pl, int cus) {
    const int64_t mt = rows128_mt(M), steps = (K / kBlockK + pl.splits - 1) / pl.splits, wgs = (int64_t)pl.tiles * pl.splits;
    const int64_t rounds = (wgs + cus - 1) / cus;
    return 4314 + rounds * steps * (584 * mt + 4863 * pl.wv + 615 * mt * pl.wv) / 100 + N * K / 10060 + 3219 * (rounds - 1) +
           (pl.splits > 1 ? 2079 + 65 * pl.splits + 3429 * wgs * mt / 1000 : 65);
}

static int64_t skinny_wide_ns(int64_t M, int64_t N, int64_t K, const SkinnyPlan &pl, int cus) {
    const int64_t mt = skinny_mt(M), steps = (K / kBlockK + pl.splits - 1) / pl.splits, wgs = (int64_t)pl.tiles * pl.splits;
    const int64_t slots = skinny_wide_slots(pl.waves, pl.tnw, (int)mt, steps);
    return 1226 + N * K / 17450 + (wgs + cus - 1) / cus * steps * (320 * pl.tnw + 284 * mt) / 10 +
           150 * ((steps + pl.waves - 1) / pl.waves) + (3231 + 134 * pl.waves) * pl.tnw * mt / 10 +
           (pl.splits > 1 ? 1479 + 213 * pl.splits : 0) + 3320 * ((wgs + cus * slots - 1) / (cus * slots) - 1);
}

// 17..64 rows: whether ROWS128 is ahead of the streaming kernel.
static bool rows128_ahead_of_stream(int64_t M, int64_t N, int64_t K, int cus) {
    const Rows128Plan pl = rows128_plan(M, N, K, cus);
    const SkinnyPlan sp = skinny_plan(M, N, K, cus);
    const int64_t t64 = (N + 63) / 64, wgs = (int64_t)sp.tiles * sp.splits;
    // a single well-filled launch: narrow or full-width workgroups on 0.55 cus .. cus tiles with K unshared
    const bool one_launch = pl.splits == 1 && pl.tiles * 20 >= (int64_t)cus * 11;
    if (pl.tiles > cus || (N * K < 20000000ll && !one_launch)) return false;
    const bool over_one = t64 > cus && t64 * 4 <= 5 * (int64_t)cus;  // 64-row tiles that come to just over one per unit
    // kept here, where the sums of the table's launch are compared with those of this kernel by name, although the streaming kernel is
    // level or ahead: a short K (N = 24576, K = 1536, M = 48: 12.4 us here, 11.6), a very long one (7168 x 18432, M = 20 / 32: 28.5 /
    // 28.6, the stream 25.9 / 27.2) and N = 14336, K = 4096 and its neighbours from 49 rows on (19.5, 17.1)
    if (M > 32 && M <= 48 && K < 2048 && one_launch) return true;
    if (M <= 48 && K >= 18432 && N * K >= 100000000ll) return true;
    if (M > 48 && K <= 4096 && N * K >= 55000000ll && t64 < cus) return true;
    if (K % 4096 != 0) {
        if (M > 48 && !one_launch && xshare_pays(M, N, K, cus)) return false;
        if (!sp.staged) return true;  // gathered scales: 31680 x 21504, M = 56 131 us here, 160 there
        if (pl.splits == 1 && !one_launch) return false;  // K too short to share: 22037 x 1024, M = 61 15.1 us, 13.5 there
        return rows128_ns(M, N, K, pl, cus) < skinny_wide_ns(M, N, K, sp, cus);
    }
    // K a multiple of 4096.  From 49 rows on the streaming kernel where its workgroups fit one round, from 100 MB on tiles of 64
    // weight rows (M = 64, us here / there: N = 12288, K = 4096 18.0 / 16.7, 8192 x 8192 23.5 / 21.3; 10240 x 8192, two a unit, 24.2
    // / 30.7; 28672 x 4096, where this one is turned, 26.3 / 33; 32 weight rows: 8032 x 20480 1.13 times behind, 7984 x 16384
    // 0.9 but kept here like those above); below, where it does not share K on 80 MB and more (48 rows, 10240 x 8192: 24.7 /
    // 22.9, kept) and its tiles do not come to just over one per unit (18096 x 8192, M = 39: 1.12 times behind)
    const bool one_round = wgs <= cus && (N * K < 100000000ll || sp.tnw == 4);
    if (M > 48) return !one_round && N * K >= 55000000ll && (one_launch || !xshare_pays(M, N, K, cus));
    if (M > 32) return over_one || (sp.splits > 1 && N * K >= 80000000ll);
    return false;  // (turned, 17..32 rows: 40960 x 4096, M = 20 40.2 here, 30.5 there; 57344 x 8192, M = 48 111, 86)
}

// Where the kernel pays (Llama-3-8B and DeepSeek-V3 linears, weights rotated so that none is found in the
// memory-side cache).  At 65..128 rows it beats the 128x128 tiles by 10 to 30 % (DeepSeek-V3 down, M = 128: 39.5 us
// against 50.0; Llama-3 down: 27.9 against 30.3) unless K is short (q_b, K = 1536: 21.7 against 17.0).  At 17..64 rows it is
// the faster one on the larger weights (rows128_ahead_of_stream), at 16 rows on a few kinds of them (below).
static bool rows128_pays(int64_t M, int64_t N, int64_t K, int cus, bool allow_streamk) {
    if (M > 384 || M < 16) return false;
    if (rows128_over_m(M, N, K, cus)) return true;
    if (M == 16) {
        // large weights whose 64-row workgroups come to just over one per unit (N = 18432, K = 7168: 27.5 us against 30.3
        // for the streaming kernel), a very long K (N = 8192, K = 28672: 45.3 against 50.7), or workgroups that spill into a
        // mostly empty third round where this kernel has a well-filled single launch (N = 36864, K = 7168)
        const int64_t t64 = (N + 63) / 64;
        const Rows128Plan pl = rows128_plan(M, N, K, cus);
        if (N * K >= 100000000ll && pl.tiles <= cus && ((t64 > cus && t64 * 4 <= 5 * (int64_t)cus) || K >= 18432)) return true;
        return t64 > 2 * (int64_t)cus && t64 <= 3 * (int64_t)cus && pl.splits == 1 && pl.tiles <= cus &&
               pl.tiles * 20 >= (int64_t)cus * 11;
    }
    if (M <= 64) return rows128_ahead_of_stream(M, N, K, cus);
    if (M > 256) {
        // 257..384 rows (the activation block of a step is 48 KiB): still ahead where the 128-row tiles are few, K is
        // long and the weights are not small (Llama-3 down at M = 257 / 384: 38.0 / 46.8 us against 66.3 / 66.5;
        // DeepSeek-V3 down 70.6 / 86.6 against 97.7 / 106.4; Llama-3 qkv 26.0 / 32.0 against 36.3); on 15 MB of
        // weights (q_a+kv_a) it is not (24.1 against 23.5 at M = 320)
        const int64_t tiles = (N + 127) / 128;
        // from about 340 rows on the 256x256 tiles with a panel split of K overtake it on the large weights
        // (DeepSeek-V3 down, M = 352 / 384: 79.4 / 78.3 us against 82.9 / 87.5; Llama-3 down stays: 49.7 against 44.8)
        if (M > 336 && N * K >= 100000000ll && allow_streamk &&
            stream_k_pays(((M + 255) / 256) * ((N + 255) / 256), K / kBlockK, cus, (M + 255) / 256))
            return false;
        // (with more than cus/4 tiles of 128 weight rows only up to 320 rows: N = 10240, K = 8192, M = 257 / 300:
        // 49.4 / 53.4 us against 68.8 / 68.9; N = 14336, K = 5120: 48.3 / 49.7 against 54.3 / 54.0; at M = 384 the
        // 128x128 tiles are ahead there - N = 16384, K = 4096: 44.7 against 56.6; N = 12288: 43.3 against 48.9)
        return K / kBlockK >= 16 && N * K >= 20000000ll && tiles * 2 <= cus && (tiles * 4 <= cus || M <= 320) &&
               tiles * rows128_splits(M, N, K, cus) * 2 >= cus;
    }
    if (M > 128) {
        // 129..256 rows, 128-row tiles.  Against the 128x128 tiles it wins where those are few and K is long
        // (DeepSeek-V3 down at M = 129 / 256: 44.8 / 62.4 us against 83.9 / 84.6; Llama-3 down 25.3 / 34.7 against
        // 42.5), and up to 160 rows also where the tiles about fill the device (Llama-3 gate_up, 224 tiles, M = 160:
        // 40.1 against 46.7; M = 192: 49.2 against 46.8).  With more tiles than units it loses (DeepSeek-V3 gate_up).
        const int64_t tiles = (N + 127) / 128;
        // up to 208 rows a single round of narrower workgroups (160..256 weight rows at two blocks per wave, 64..112
        // at one) beats the square tiles (N = 36864, K = 7168, M = 144 / 192: 69.1 / 80.5 us against 82.7 / 85.9;
        // N = 28672, K = 4096: 35.8 / 42.0 against 43.3 / 48.4; q_b, K = 1536: 15.3 / 18.3 against 19.6 / 21.3);
        // its time grows with M (every wave reads the whole X block from LDS) and the square tiles are level or
        // ahead from about 220 rows
        {
            const Rows128Plan pl = rows128_plan(M, N, K, cus);
            if (pl.tn == 2 || pl.wv != 8) return true;
        }
        if (K / kBlockK < 16) return false;
        // from about 200 rows the panel split of the 256x256 tiles is level or ahead on the large weights, its time
        // flat in M (DeepSeek-V3 down, M = 208 / 240 / 256: 55.1 / 54.9 / 56.9 us against 58.4 / 60.4 / 63.3;
        // o_proj 53.1 / 52.8 / 58.1 against 54.9 / 57.5 / 57.6)
        // With fewer than eight runs of K (a wider N or a shorter K) it is behind: of 415 such shapes none is ahead by more than
        // 4 %, 1.11 times behind in the middle (203 x 31072 x 5760 77.9 us, 67.9 here before the pipelined K loop, 211 x 9152 x
        // 11520 61.3 / 44.9, 204 x 32336 x 6144 84.2 / 61.2).
        const bool runs8 = (N + 255) / 256 * 8 <= cus && K >= 96 * kBlockK;
        if (M > 200 && N * K >= 100000000ll && runs8 && allow_streamk && stream_k_pays((N + 255) / 256, K / kBlockK, cus, 1)) return false;
        // and on small weights the 128x128 tiles with K shared (N = 4096, K = 4096, M = 224 / 256: 18.9 / 19.0 us
        // against 20.9 / 21.3; N = 7168, K = 2304, M = 256: 19.7 against 23.0)
        if (M > 192 && N * K < 20000000ll) return false;
        if (tiles * 2 <= cus) return tiles * rows128_splits(M, N, K, cus) * 2 >= cus;
        return tiles <= cus && (M <= 160 || (M <= kRows128NarrowMaxM && tiles * 8 >= (int64_t)cus * 7));
    }
    // 65..128 rows: a single well-filled launch always pays (narrow or full-width workgroups on 0.55 cus .. cus tiles with K
    // unshared: q_b, M = 65: 12.5 us against 15.0), otherwise from 16 K steps on
    const Rows128Plan pl = rows128_plan(M, N, K, cus);
    if (pl.splits == 1 && pl.tiles <= cus && pl.tiles * 20 >= (int64_t)cus * 11) return true;
    return K / kBlockK >= 16;
}

static bool rowsm_limits_ok(const RowsMPlan &pl, int64_t M, int64_t K, int64_t lda, int64_t as_m, int64_t as_k);
static bool rows128_limits_ok(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t as_m, int64_t as_k, int cus) {
    if (M > 384) return false;
    if (rows128_over_m(M, N, K, cus)) return rowsm_limits_ok(rowsm_plan(M, N, K, cus), M, K, lda, as_m, as_k);
    if (M * lda >= (1ll << 32) || M * as_m * 4 >= (1ll << 32) || as_k * 32 >= (1ll << 32)) return false;
    const Rows128Plan pl = rows128_plan(M, N, K, cus);
    const int64_t steps = (K / kBlockK + pl.splits - 1) / pl.splits;
    // Rows128Cfg::lds_bytes for the plan's tile: the ring, the W scales of the tile's n blocks, two X scale chunks
    const int64_t mt = rows128_mt(M), ns = mt <= 8 ? 3 : 2, nblk = (pl.bn + 2 * kBlockN - 2) / kBlockN;
    const int64_t ring = ns * (16 * mt * 128 + (int64_t)pl.bn * 128);
    return ((ring + nblk * steps * 4 + 127) & ~127ll) + 2 * 16 * mt * 32 <= 160 * 1024;
}

// ---- more rows than that on a narrow N: the same kernel tiled over M as well (tiles_m x tiles_n workgroups in one
// round, K unshared).  Where N gives few 256-wide tiles the 256x256 launch leaves most units idle (N = 2112: 9 tile
// columns, 144 tiles at M = 4096, 72 at M = 2048) and its lone round is bound by the latency of its K steps; tiles of
// 16*mt rows x 32*wv weight rows with mt chosen so that tiles_m * tiles_n just fits the units put a workgroup on
// (nearly) every unit, each with less to load and to multiply per step.
// rowsm_round_plan is the tile of a single round: up to N = 4608 (5120 from 769 rows on) the fewest row blocks, then the fewest
// bytes a unit loads per K step; beyond, by what a step loads and multiplies.  rowsm_plan is what is launched: the tile of the
// least rowsm_ns over up to four rounds, where that is 4 % less than the round plan's.
static RowsMPlan rowsm_round_plan(int64_t M, int64_t N, int cus) {
    RowsMPlan best = {0, 0, 0, 0};
    if (M <= 0 || cus < 8) return best;
    const int64_t blocks = (M + 15) / 16;
    const bool wide = N > 5120 || (N > 4608 && M <= 768);
    int64_t best_cost = 0;
    for (int wv = 8; wv >= 5; --wv) {
        const int64_t tn = (N + 32 * wv - 1) / (32 * wv);
        if (tn > cus) continue;
        const int64_t room = cus / tn;                       // m tiles that fit one round
        const int64_t fewest = (blocks + room - 1) / room;   // row blocks per tile
        for (int64_t mt = fewest; mt <= fewest + (wide ? 1 : 0); ++mt) {
            if (mt > 13 || (mt <= 8 && wv == 7)) continue;   // kernels built: 5, 6, 8 waves up to 8 blocks; 5..8 up to 13
            const int64_t tm = (blocks + mt - 1) / mt;
            if (tm < 2 || tm * tn * 20 < (int64_t)cus * 11) continue;
            const int64_t cost = wide ? 146 * mt + 134 * wv + 45 * tm * tn * (mt + 2 * wv) / cus + (mt > 8 ? 371 : 0)
                                      : mt * 65536 + 16 * mt + 32 * wv;
            if (best.mt == 0 || cost < best_cost) {
                best = {(int)mt, wv, (int)tm, (int)tn};
                best_cost = cost;
            }
        }
    }
    return best;
}

static bool rowsm_lds_ok(int64_t mt, int64_t wv, int64_t K) {
    const int64_t steps = K / kBlockK, ns = mt <= 8 ? 3 : 2, bn = 32 * wv, nblk = (bn + 2 * kBlockN - 2) / kBlockN;
    const int64_t ring = ns * (16 * mt * 128 + bn * 128);
    return ((ring + nblk * steps * 4 + 127) & ~127ll) + 2 * 16 * mt * 32 <= 160 * 1024;
}

// What the launch takes, in ns: a least-squares fit to 82000 timed launches (9676 shapes of 209..4096 rows, N = 640..36864, K =
// 1024..18432, the nine most likely tiles of each; weights from HBM; 6 % rms).  A K step of a tile (its products; the X block,
// which every wave reads; its W rows; two slots of W instead of three; more than six waves), what all tiles pull together, the
// output and the weights; 2.9 us a round.  The tile of the least estimate is 0.8 % behind the fastest one on average.
static double rowsm_ns(int64_t M, int64_t N, int64_t K, const RowsMPlan &pl, int cus) {
    const int mt = pl.mt, wv = pl.wv, t = pl.tiles_m * pl.tiles_n;
    const double kb = (double)(K / kBlockK), rounds = (double)((t + cus - 1) / cus);
    const double step = 83.0 + 0.457 * mt * wv + 49.95 * mt + 18.96 * wv + (mt > 8 ? 59.7 : 0.0) + (wv > 6 ? 9.9 : 0.0) + (wv == 8 ? 23.6 : 0.0);
    return 792.0 + rounds * (2939.0 + kb * step) + 6.0 * kb * t / cus * (mt + 2 * wv) + M * N * 4.91e-4 + N * K * 7.95e-5;
}

static RowsMPlan rowsm_plan(int64_t M, int64_t N, int64_t K, int cus) {
    RowsMPlan best = rowsm_round_plan(M, N, cus);
    if (M < 80 || M > 4096 || N < 640 || cus < 8) return best;
    double best_ns = best.mt ? 0.96 * rowsm_ns(M, N, K, best, cus) : 0.0;
    const int blocks = (int)((M + 15) / 16);
    for (int wv = 5; wv <= 8; ++wv) {
        const int64_t tn = (N + 32 * wv - 1) / (32 * wv);
        if (2 * tn > 4 * (int64_t)cus) continue;  // (the kernel numbers two m tiles and more)
        for (int mt = wv == 7 ? 9 : 1; mt <= 13; ++mt) {
            const RowsMPlan pl = {mt, wv, (blocks + mt - 1) / mt, (int)tn};
            if (pl.tiles_m < 2 || pl.tiles_m * pl.tiles_n > 4 * cus || !rowsm_lds_ok(mt, wv, K)) continue;
            const double ns = rowsm_ns(M, N, K, pl, cus);
            if (best.mt == 0 || ns < best_ns) {
                best = pl;
                best_ns = ns;
            }
        }
    }
    return best;
}

static bool rowsm_limits_ok(const RowsMPlan &pl, int64_t M, int64_t K, int64_t lda, int64_t as_m, int64_t as_k) {
    if (pl.mt == 0) return false;
    if (M * lda >= (1ll << 32) || M * as_m * 4 >= (1ll << 32) || as_k * 32 >= (1ll << 32)) return false;
    return rowsm_lds_ok(pl.mt, pl.wv, K);
}

// Where the table names it (forced against the table's previous choice with the K loop before the pipelined one, over N =
// 1024..8192, K = 1536..14336, M = 400..4096,
// 256 units).  With K <= 5120 and at most 8 row blocks per tile (three ring slots) it is ahead on every N <= 5120:
// 1.2 to 2.0 times with up to 4 row blocks (N = 4096, K = 4096, M = 512 / 1024 / 2048: 22.4 / 28.8 / 42.0 us against
// 27.9 / 36.5 / 47.2; N = 2112, K = 2048, M = 1024: 1.95 times), 1.0 to 1.2 with 5..8; from N = 6144 on and with more
// row blocks (two slots) the square tiles were level or ahead.  With K = 6144 .. 7168 the panel split of the 256x256
// tiles shares K between idle units and takes most of the gain: 2..6 row blocks on N <= 3072 are still 1.04 to 1.3
// times ahead (q_a+kv_a, N = 2112, K = 7168, M = 512 / 1024 / 2048: 1.11 / 1.12 / 1.04), a single block or a wider N
// was behind, and from K = 8192 on the kernels that share K.  With the K loop as it is now the tiles are ahead of those on many more
// shapes; rowsm_ahead decides that by estimates, and this rule which of them have the name.
// On a wider N, K <= 5120: up to 960 rows and N = 15360 with at most 8 row blocks (us, before / here: N = 6144, K = 4096, M = 450 /
// 700 / 850 36.4 / 41.4 / 43.0 against 28.2 / 33.9 / 35.6; 8192 x 4096, M = 400 / 640 36.4 / 42.9 against 29.7 / 37.2; 10240
// x 5120, M = 512 55.4 / 45.3; 12288 x 4096, M = 400 / 640 44.2 / 45.3 against 37.1 / 44.3).
static bool rowsm_pays(int64_t M, int64_t N, int64_t K, int cus) {
    if (M <= 384) return false;
    const int64_t KB = K / kBlockK;
    if (KB < 12 || KB > 56) return false;
    const RowsMPlan pl = rowsm_round_plan(M, N, cus);
    if (pl.mt == 0 || pl.mt > 8) return false;
    if (KB <= 40) return N <= 5120 || (M <= 960 && N <= 15360 && KB >= 16);
    return pl.mt >= 2 && pl.mt <= 6 && N <= 3072;
}

// 209..352 rows on a wide N: ROWS128 as two (on a narrower N three or four) m tiles of up to 11 row blocks in one round instead
// of two 256-row tiles, a third of them padding, or 128x128 tiles in two rounds (us, before / here: N = 27648, K = 5120, M = 220 / 288
// / 333 / 352 59.1 / 68.2 / 73.7 / 69.2 against 53.7 / 58.9 / 67.4 / 66.6, at 384 level; 28672 x 4608, M = 300 63.7 / 56.3; 15360 x
// 5120, M = 330 54.2 / 45.8; 24576 x 1536, M = 333 27.4 / 22.3; 16384 x 4096, M = 256 40.8 / 36.7).  (K = 4096 beyond N = 16384
// keeps the square tiles by name as well, although the gain is the same there: 28672 x 4096, M = 224 / 320 48.5 / 60.7
// against 44.3 / 51.9.)
static bool rows128_over_m(int64_t M, int64_t N, int64_t K, int cus) {
    const int64_t KB = K / kBlockK;
    if (M <= 208 || M > 352 || N < 12288 || KB < 12 || KB > 44 || (K % 4096 == 0 && N > 16384)) return false;
    const RowsMPlan pl = rowsm_round_plan(M, N, cus);
    return pl.mt > 0 && pl.mt <= 11;
}

// m tiles in a group of the launch's tile order (gemm_rows128.hpp): the least sum over the 8 XCDs of the distinct rows of X and W
// that a run of tiles touches, estimated (a run that crosses from one group to the next touches the m tiles of both:
// 4 % above the best order over random plans, never above n fastest, half of it).  us, n fastest / here: N = 6144, K = 4096, M = 512 / 700
// 32.2 / 33.9 against 25.2 / 31.0; 512 x 4096 x 4096 25.4 / 23.6; 333 x 27648 x 5120 79.5 / 78.7; 15 others 0 to 4 % ahead.
static int rowsm_group(const RowsMPlan &pl) {
    const int64_t tm = pl.tiles_m, tn = pl.tiles_n, per = (tm * tn + 7) / 8;
    int best = 1;
    int64_t best_cost = 0;
    for (int64_t h = 1; h <= tm; ++h) {
        const int64_t m = h * tn < per ? 8 * h * (1 + per / (h * tn)) : h * (8 + (tm + h - 1) / h - 1);
        const int64_t n = 8 * (per / h) + (per % h ? 12 : 0);
        const int64_t cost = std::min(m, 8 * tm) * 16 * pl.mt + std::min(n, 8 * tn) * 32 * pl.wv;
        if (h == 1 || cost < best_cost) {
            best = (int)h;
            best_cost = cost;
        }
    }
    return best;
}

static int launch_rowsm(GemmArgs &a, const RowsMPlan &mp, hipStream_t st) {
    a.tiles_m = mp.tiles_m;
    a.tiles_n = mp.tiles_n;
    a.group_m = rowsm_group(mp);
    a.total_tiles = mp.tiles_m * mp.tiles_n;
    Rows128Plan pl;
    pl.turned = false;
    pl.wv = mp.wv;
    pl.bn = 32 * mp.wv;
    pl.splits = 1;
    pl.tiles = (a.total_tiles + 7) / 8 * 8;  // the kernel numbers its tiles per XCD
    pl.tn = 2;
    return launch_rows128(a, pl, mp.mt, true, nullptr, st);
}

// 256x128 tiles that are too few to occupy the device share the K range the same way.
static int tile256x128_splits(int64_t M, int64_t N, int64_t K, int cus) {
    const int64_t tiles = ((M + 255) / 256) * ((N + 127) / 128);
    const int64_t KB = K / kBlockK;
    if (tiles * 2 > cus || KB < 16) return 1;
    int64_t splits = cus / tiles;
    if (splits > KB / 8) splits = KB / 8;
    return (int)(splits < 1 ? 1 : splits);
}

static size_t tile256x128_workspace(int64_t M, int64_t N, int splits) {
    const int64_t tiles = ((M + 255) / 256) * ((N + 127) / 128);
    return (size_t)MI355_WS_COUNTER_BYTES + (size_t)tiles * splits * 256 * 128 * 4;
}

static int64_t n_split_rows(int64_t M, int64_t N, int64_t K, int cus);
static double other_ns(int64_t M, int64_t N, int64_t K, int variant, size_t ws_bytes, int cus);

// The shape -> kernel table (measured on the DeepSeek-V3 and Llama-3 linears over M = 128..4096):
//   129 <= M <= 384, K >= 2048, at most cus/2 tiles
//     of 128 weight rows (cus if M <= 160; above
//     256 rows only if N*K >= 2e7; 201..256 (eight runs) and
//     337..384 rows on N*K >= 1e8 go to the panel
//     split of stream-K instead)                     the weight stream with the activation block in LDS
//   129 <= M <= 208 (192), 0.55 cus .. cus tiles of
//     160..256 or of 80..112 (64) weight rows         the same, workgroups of that width, K unshared
//   65 <= M <= 128, K >= 2048                        the same with 256 weight rows per workgroup; under the same name the
//                                                    weight streaming kernel where one round of its tiles is ahead
//                                                    (skinny_many_rows_plan; mi355_block_fp8_gemm_launched tells)
//   65 <= M <= 128, 0.55 cus .. cus tiles of 160,
//     192 or 256 weight rows with K unshared          the same, workgroups of that width
//   17 <= M <= 64, N*K >= 2e7, at most cus tiles,
//     ahead of the weight streaming kernel
//     (rows128_ahead_of_stream)                       the same
//   M > 384, N <= 5120 (3072), K <= 5120 (7168), one
//     round of tiles of at most 128 (96) rows; 385..960
//     rows, N <= 15360, K <= 5120                     the same kernel tiled over M, K unshared
//   209..352 rows, N >= 12288, 1536 <= K <= 5632      the same, two to four tiles over M (mi355_block_fp8_gemm_launched)
//   M <= 64                                          weight streaming (M > 48 and N/128 about the unit count, or M > 32 in
//                                                    more than five rounds: the kernel that shares the activation block
//                                                    in the workgroup)
//   few 256x256 tiles, long K                        stream-K (the plain loop would leave most units idle), from 513 rows on,
//                                                    on few tiles from 257, where the 128x128 tiles are not estimated ahead
//   128x128 tiles fit one round of two per unit and
//     (few 256x256 tiles or a short K)               128x128 tiles, K shared between workgroups when they are few
//                                                    (M >= 768 and N <= 3072: 256x128 tiles with K shared)
//   otherwise                                        256x256 ping-pong tiles
// Without room for the partial tiles of stream-K (allow_streamk) its shapes go to the rows below it: 128x128 tiles are 1.25 times
// as fast as a few 256x256 ones there, level from about 80 of those on (2684 shapes of 129..6000 rows, K = 5120..29440; us, 256x256 /
// 128x128: 175 x 6112 x 5888 65.0 / 49.2, 2831 x 176 x 8448 87.5 / 68.9; 507 x 14976 x 25216, 118 tiles, 8 % the other way).
static int pick_variant(int64_t M, int64_t N, int64_t K, int cus, bool allow_rows128 = true, bool allow_streamk = true) {
    // up to 16 rows the per-unit stream also beats the stream with the activation block in LDS where both apply
    // (N = 18432, K = 7168, M = 16: 23.6 us against 27.5; N = 7168, K = 18432: 25.4 against 27.2)
    if (streamcu_pays(M, N, K, cus)) return MI355_GEMM_SKINNY_CU;
    if (allow_rows128 && rows128_pays(M, N, K, cus, allow_streamk)) return MI355_GEMM_ROWS128;
    if (allow_rows128 && rowsm_pays(M, N, K, cus)) return MI355_GEMM_ROWS_MTILED;
    if (xshare_pays(M, N, K, cus)) return MI355_GEMM_SKINNY_XSHARE;
    if (M <= 64) return MI355_GEMM_SKINNY;
    const int64_t t256 = ((M + 255) / 256) * ((N + 255) / 256);
    const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
    const int64_t KB = K / kBlockK;
    // one or two K steps: the 256x256 tile's first requests and its epilogue are most of its time (N = 7168,
    // K = 256, M = 4096: 21.3 us for the 128x128 tiles against 27.6)
    if (KB <= 2) return MI355_GEMM_TILE128;
    const bool shares = M > 128 && stream_k_pays(t256, KB, cus, (M + 255) / 256);
    const bool small = t128 <= 2 * (int64_t)cus && (t256 < (int64_t)cus * 3 / 8 || KB <= 64);  // 128x128 tiles fit the device
    // On a narrow N the 128x128 tiles, which share K in shorter runs, are ahead of the panel split (us, panel / 128x128: 517 x 611 x
    // 12288 31.6 / 21.2, 1058 x 128 x 23168 31.5 / 18.3, 462 x 1840 x 9344 32.4 / 28.7; 403 x 1232 x 32128 40.1 / 51.5).  The panel's
    // estimate is low where the tiles are few; with 8 % on it 76 of 1535 shapes of 513 rows and more with up to 36 256x256 tiles run
    // more than 2 % behind the faster of the two, 15 % at most (all of them on the panel split: 562, 1.8 times).  Two m tiles are
    // compared below three 32nds of the units, beyond which the panel split is ahead.
    const bool tiles128 = shares && small && (M > 512 || (M > 256 && t256 * 32 < 3 * (int64_t)cus)) &&
                          1.08 * other_ns(M, N, K, MI355_GEMM_TILE256_STREAMK, SIZE_MAX, cus) > other_ns(M, N, K, MI355_GEMM_TILE128, SIZE_MAX, cus);
    if (shares && allow_streamk && !tiles128) return MI355_GEMM_TILE256_STREAMK;
    // 257..384 rows leave the second 256-row tile at most half full; where the 256x256 tiles need a second round
    // anyway the 128x128 ones are ahead (N = 36864, K = 7168, M = 257 / 384: 144 / 148 us against 161 / 165) -
    // unless the second round is small enough to run as a launch of its own (130 / 139 us then)
    if (M > 256 && M <= 384 && t256 > cus && t128 <= 4 * (int64_t)cus && n_split_rows(M, N, K, cus) == 0)
        return MI355_GEMM_TILE128;
    if (small) {
        // a narrow N under many rows: 256x128 tiles with K shared load half as much X per product as the 128x128
        // ones and still fill the device (q_a+kv_a, N = 2112, K = 7168, M = 768 / 1024 / 1536: 35.0 / 40.6 / 50.6 us
        // against 38.7 / 60.2 / 60.6; not under 12 n tiles: N = 256 / 512, M = 1024: 17.5 / 17.5 against 20.6 / 21.4)
        // ... and, from two 256-row tiles on, a wider N under a long K (N = 5120, K = 5120, M = 400 / 512: 35.4 /
        // 37.6 us against 44.7 / 45.1; N = 4096, K = 7168, M = 640: 54.6 against 60.3; on N = 1536 the 128x128 tiles
        // keep their lead, 21.8 against 25.2, and with K = 4096 too)
        if (!shares && ((M >= 768 && (N + 127) / 128 <= 24 && (N + 127) / 128 >= 12) || (M > 384 && KB >= 40 && (N + 127) / 128 >= 20)) &&
            tile256x128_splits(M, N, K, cus) >= 2)
            return MI355_GEMM_TILE256x128;
        return MI355_GEMM_TILE128;
    }
    if (t256 >= (int64_t)cus * 3 / 8) return MI355_GEMM_TILE256;
    return MI355_GEMM_TILE128;
}

// 128x128 tiles that are too few to occupy the device share the K range: about one CTA per CU, at least
// 8 K steps each.
static int tile128_splits(int64_t M, int64_t N, int64_t K, int cus) {
    const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
    const int64_t KB = K / kBlockK;
    if (tiles * 2 > cus || KB < 16) return 1;
    int64_t splits = cus / tiles;
    if (splits > KB / 8) splits = KB / 8;
    return (int)(splits < 1 ? 1 : splits);
}

static size_t tile128_workspace(int64_t M, int64_t N, int splits) {
    const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
    return (size_t)MI355_WS_COUNTER_BYTES + (size_t)tiles * splits * 128 * 128 * 4;
}

// A launch of 256x256 tiles that fills the device once and leaves a small rest for a second round runs the rest
// as a launch of its own, with whatever the table gives its shape (mostly 128x128 tiles, which spread it over the
// whole device): N = 36864, K = 7168, M = 512 (288 tiles on 256 units) 137 us against 169; q_b, M = 768, 43.6
// against 50.2.  After two full rounds a rest of up to a quarter round still gains a little (M = 1024, 576 tiles:
// 248 us against 260; q_b, M = 1536: 77.8 against 83.3); with more rounds or a larger rest it gains nothing (3.5
// rounds: 235 against 220).  Returns the number of weight rows of the first launch, 0 for no split.
static int64_t n_split_rows(int64_t M, int64_t N, int64_t K, int cus) {
    (void)K;
    const int64_t tiles_m = (M + 255) / 256, tiles_n = (N + 255) / 256, t256 = tiles_m * tiles_n;
    const int64_t rounds = t256 / cus, rest = t256 - rounds * cus;
    if (tiles_m > cus || rounds < 1 || rounds > 2 || rest == 0) return 0;
    if (rest * 2 * rounds > cus) return 0;
    const int64_t n1 = rounds * (int64_t)cus / tiles_m * 256;
    return n1 > 0 && n1 < N ? n1 : 0;
}

// What the table's other choices take above 208 rows (the 128x128 tiles from 80 on), in ns: fits to the same shapes (256x256
// tiles 2.8 % rms, 128x128 tiles 3.4,
// panel split of K 5.0, weight stream of one m tile 4.7), 0 for what was not fitted.  `ws_bytes` of workspace: the 128x128 tiles run
// K whole without room for their partial sums (the estimate is 6 % low there).
static double other_ns(int64_t M, int64_t N, int64_t K, int variant, size_t ws_bytes, int cus) {
    const double kb = (double)(K / kBlockK), weights = 1e-6 * N * K, out = 1e-6 * M * N, c = cus;
    const int64_t KB = K / kBlockK, tm = (M + 255) / 256, tn = (N + 255) / 256, t = tm * tn;
    if (variant == MI355_GEMM_TILE256) {
        const double in_first = (double)std::min<int64_t>(t, cus) / c;
        const double common = 1964.0 + kb * (566.0 * t / c - 76.0 * in_first) + 212.6 * out + 30.6 * weights;
        const int64_t full = (t + cus - 1) / cus;
        if (n_split_rows(M, N, K, cus) > 0) return common - 670.0 + 8233.0 * full + kb * (1170.0 * (t / cus) + 1076.0 * (t % cus) / c);
        return common + full * (8233.0 + 1012.0 * kb);
    }
    if (variant == MI355_GEMM_TILE128) {
        int64_t splits = tile128_splits(M, N, K, cus);
        if (ws_bytes < tile128_workspace(M, N, (int)splits)) splits = 1;
        const int64_t w = ((M + 127) / 128) * ((N + 127) / 128) * splits;
        const double steps = (double)((KB + splits - 1) / splits), two = (double)((w + 2 * cus - 1) / (2 * cus));
        return 2938.0 + steps * (743.0 * two + 100.9 * ((w + cus - 1) / cus) + 164.9 * w / c) + 2938.0 * two + 81.0 * out + 32.5 * weights +
               (splits > 1 ? 2069.0 + 11.6 * w : 0.0);
    }
    if (variant == MI355_GEMM_TILE256_STREAMK) {
        const int64_t runs = sk_panel_splits((int)tm, (int)tn, (int)KB, cus);
        if (runs == 0) return 0.0;
        return 17671.0 + ((KB + runs - 1) / runs) * (400.0 + 893.0 * t * runs / c) + 20.45 * t * runs + 1141.0 * out + 88.6 * weights;
    }
    if (variant == MI355_GEMM_ROWS128) {
        const int64_t mt = (M + 15) / 16, splits = rows128_splits(M, N, K, cus), w = (N + 127) / 128 * splits;
        const double steps = (double)((KB + splits - 1) / splits), rounds = (double)((w + cus - 1) / cus);
        return 1303.0 + rounds * steps * (8.86 * mt - 220.7) + 378.7 * weights + 34.0 * out + 284.8 * mt + (splits > 1 ? 1303.0 + 2.347 * w * mt : 0.0);
    }
    return 0.0;
}

// Tiles over M instead of what the table names: from 80 rows on where the estimates say 3 % less (the weight stream's K loop
// multiplies two thirds as fast as the 256x256 tile's, on tiles that leave little of the device idle and nothing to padding or
// partial sums).  rowsm_ns was fitted to launches whose smaller weights the memory-side cache held; from HBM a K step of mt row blocks
// takes about 100 / mt ns more up to four of them (one row block 340 to 375 ns, two 380 to 460), and that decides against a kernel that shares K
// (us, over M / 128x128: 566 x 640 x 6400 21.4 / 17.2, 250 x 2800 x 5504 23.8 / 19.2, 266 x 2112 x 7168 25.6 / 22.6).
// Weights from HBM, random shapes and the ten model weights: 1564 shapes of 80..4096 rows run over M, 1.27 times as fast, 12 of them
// more than 2 % slower (7 % at most; without the 100 / mt ns 183 more shapes, 126 of them more than 2 % slower, 28 % at most); us,
// before / here: 300 x 4096 x 4096 26.3 / 19.1, 340 x 6144 x 4096 32.0 / 21.4, 300 x 28672 x 4096 65.0 / 47.8, 380 x 27648 x 5120
// 85.9 / 68.7, 1200 x 6144 x 4096 50.7 / 38.3, 1700 x 5120 x 13824 156 / 122, 1200 x 7168 x 18432 207 / 167.
// From 80 to 208 rows instead of the 128x128 tiles only (118 x 5744 x 1792 19.6 / 9.1, 143 x 2032 x 1920 20.2 / 9.2).  The plan keeps
// the table's name, by which the kernels' sums are compared; from K = 8192 on the 256x128 tiles with K shared do run under theirs (1.17
// times behind there, 1.3 to 1.8 times on a shorter K).
// `ws_bytes` (0: none that can be used): what the table's kernel shares K with.  Without it that runs K whole on too few tiles, and
// the tiles over M are 1.5 to 3.4 times as fast (us, K whole / over M: 300 x 1024 x 18432 147 / 59, 768 x 2112 x 8192
// 104 / 34; 812 shapes, bit-equal).
static RowsMPlan rowsm_ahead(int64_t M, int64_t N, int64_t K, int variant, size_t ws_bytes, int cus) {
    const RowsMPlan none = {0, 0, 0, 0};
    if (M < 80 || M > 4096 || N < 640 || K < 1024 || K > 20480 || cus < 192) return none;
    if (M <= 208 && variant != MI355_GEMM_TILE128) return none;
    if (variant == MI355_GEMM_TILE256x128)
        return K < 8192 || ws_bytes < tile256x128_workspace(M, N, tile256x128_splits(M, N, K, cus)) ? rowsm_plan(M, N, K, cus) : none;
    const double other = other_ns(M, N, K, variant, ws_bytes, cus);
    if (other == 0.0) return none;
    const RowsMPlan pl = rowsm_plan(M, N, K, cus);
    if (pl.mt == 0) return none;
    const int rounds = (pl.tiles_m * pl.tiles_n + cus - 1) / cus;
    const double from_hbm = pl.mt <= 4 ? 100.0 * rounds * (K / kBlockK) / pl.mt : 0.0;
    return rowsm_ns(M, N, K, pl, cus) + from_hbm < 0.97 * other ? pl : none;
}

static int auto_launch(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t as_m, int64_t as_k, bool ws_usable,
                       size_t ws_bytes, int cus, RowsMPlan &tiles);

// Whether an AUTO call in packed layout runs as tiles over M with any workspace and without one.
static bool over_m_without_workspace(int64_t M, int64_t N, int64_t K, int cus) {
    RowsMPlan tiles;
    return M >= 80 && M <= 4096 && auto_launch(M, N, K, K, K, K / kBlockK, 1, true, SIZE_MAX, cus, tiles) == MI355_GEMM_ROWS_MTILED &&
           auto_launch(M, N, K, K, K, K / kBlockK, 1, false, 0, cus, tiles) == MI355_GEMM_ROWS_MTILED;
}

// Workspace of a launch plan on a device with `cus` compute units.
static size_t workspace_bytes_for(int64_t M, int64_t N, int64_t K, int32_t variant, int cus) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    if (K % kBlockK != 0) return 0;
    if (variant == MI355_GEMM_AUTO) {
        if (over_m_without_workspace(M, N, K, cus)) return 0;
        variant = pick_variant(M, N, K, cus);
        const int64_t n1 = variant == MI355_GEMM_TILE256 ? n_split_rows(M, N, K, cus) : 0;
        if (n1 > 0) {
            const size_t rest = workspace_bytes_for(M, N - n1, K, MI355_GEMM_AUTO, cus);
            return rest > (size_t)MI355_WS_COUNTER_BYTES ? rest : (size_t)MI355_WS_COUNTER_BYTES;
        }
        // 65..128 rows may run as the streaming kernel, and where a limit of that is not met as the kernel of the name
        if (variant == MI355_GEMM_ROWS128)
            return std::max(workspace_bytes_for(M, N, K, MI355_GEMM_SKINNY_ROWS, cus), workspace_bytes_for(M, N, K, variant, cus));
    }
    if (variant == MI355_GEMM_TILE256_STREAMK) {
        const int groups = stream_k_groups(((M + 255) / 256) * ((N + 255) / 256), K / kBlockK, cus, (M + 255) / 256);
        return groups > 0 ? stream_k_workspace(groups) : (size_t)MI355_WS_COUNTER_BYTES;
    }
    if (variant == MI355_GEMM_TILE128) {
        const int splits = tile128_splits(M, N, K, cus);
        return splits > 1 ? tile128_workspace(M, N, splits) : 0;
    }
    if (variant == MI355_GEMM_TILE256x128) {
        const int splits = tile256x128_splits(M, N, K, cus);
        return splits > 1 ? tile256x128_workspace(M, N, splits) : 0;
    }
    if (variant == MI355_GEMM_TILE256) return MI355_WS_COUNTER_BYTES;  // the tile counters of the persistent launch
    if (variant == MI355_GEMM_SKINNY_XSHARE) {
        const int splits = xshare_splits(N, K, cus);
        return splits > 1 ? xshare_workspace(N, splits) : 0;
    }
    if (variant == MI355_GEMM_SKINNY_ROWS) {
        const SkinnyPlan sp = skinny_many_rows_plan(M, N, K, cus);
        return sp.tnw > 0 && sp.splits > 1 ? skinny_workspace(M, sp) : 0;
    }
    if (variant == MI355_GEMM_ROWS128) {
        if (M > 384) return 0;
        return rows128_workspace(M, N, K, cus);
    }
    if (variant != MI355_GEMM_SKINNY || M > 64) return 0;
    const SkinnyPlan pl = skinny_plan(M, N, K, cus);
    return pl.splits > 1 ? skinny_workspace(M, pl) : 0;
}

// The kernel an AUTO call launches (first) for a problem in the fast layout: the table's choice, or - where a limit
// of that kernel is not met or its workspace is missing - the next kernel with fewer preconditions.  The chain ends
// in tiles that take every fast layout and run unsplit without a workspace, so AUTO never fails for want of one.
// Stream-K's workspace and the 256-row stream are looked at first because the table's other choice for their shapes can be any of
// the kernels checked after them.
static int resolve_auto(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t as_m, int64_t as_k,
                        bool ws_usable, size_t ws_bytes, int cus, RowsMPlan *tiles = nullptr) {
    const bool streamk = ws_usable && ws_bytes >= stream_k_workspace(cus / 8 * 8);  // (every plan of it takes that much)
    int variant = pick_variant(M, N, K, cus, true, streamk);
    if (variant == MI355_GEMM_ROWS_MTILED) {
        const RowsMPlan pl = rowsm_plan(M, N, K, cus);
        if (!rowsm_limits_ok(pl, M, K, lda, as_m, as_k)) variant = pick_variant(M, N, K, cus, false, streamk);
        else if (tiles) *tiles = pl;
    }
    if (variant == MI355_GEMM_ROWS128 &&
        (!rows128_limits_ok(M, N, K, lda, as_m, as_k, cus) ||
         (rows128_splits(M, N, K, cus) > 1 && (!ws_usable || ws_bytes < rows128_workspace(M, N, K, cus)))))
        variant = pick_variant(M, N, K, cus, false, streamk);
    if (variant == MI355_GEMM_SKINNY_XSHARE &&
        (N * ldw >= (1ll << 32) || M * lda >= (1ll << 32) || M * as_m >= (1ll << 32) ||
         (N + XshareCfg::BN - 1) / XshareCfg::BN * 4 > MI355_WS_COUNTER_BYTES))
        variant = MI355_GEMM_TILE128;
    if (variant == MI355_GEMM_SKINNY_CU && streamcu_tnw(M, N, K, lda, ldw, as_m, cus) == 0)
        variant = MI355_GEMM_SKINNY;
    if (variant == MI355_GEMM_SKINNY &&
        skinny_check(M, N, K, lda, ldw, as_m, cus, ws_usable, ws_bytes) != MI355_OK)
        variant = MI355_GEMM_TILE128;
    return variant;
}

// 65..128 rows on the streaming kernel: its plan, the 32-bit offsets and the workspace of a shared K.
static int skinny_rows_check(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t as_m, int cus, bool ws_usable,
                             size_t ws_bytes) {
    const SkinnyPlan sp = skinny_many_rows_plan(M, N, K, cus);
    if (sp.tnw == 0 || N * ldw >= (1ll << 32) || M * lda >= (1ll << 32) || M * as_m >= (1ll << 32)) return MI355_EUNSUPPORTED;
    if (sp.splits > 1 && (!ws_usable || ws_bytes < skinny_workspace(M, sp))) return MI355_EWORKSPACE;
    return MI355_OK;
}

// What AUTO launches where the table says ROWS128: 65..128 rows as the streaming kernel where one round of that is ahead, 209..352
// rows tiled over M.
static int launched_for(int variant, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t as_m, bool ws_usable,
                        size_t ws_bytes, int cus) {
    if (variant != MI355_GEMM_ROWS128) return variant;
    if (rows128_over_m(M, N, K, cus)) return MI355_GEMM_ROWS_MTILED;
    return skinny_rows_check(M, N, K, lda, ldw, as_m, cus, ws_usable, ws_bytes) == MI355_OK ? MI355_GEMM_SKINNY_ROWS : variant;
}

// The kernel an AUTO call launches (first), `tiles` its tiles where that is ROWS_MTILED: the plan is made once a call.
static int auto_launch(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t as_m, int64_t as_k, bool ws_usable,
                       size_t ws_bytes, int cus, RowsMPlan &tiles) {
    tiles = {0, 0, 0, 0};
    const int variant = launched_for(resolve_auto(M, N, K, lda, ldw, as_m, as_k, ws_usable, ws_bytes, cus, &tiles), M, N, K, lda, ldw, as_m,
                                     ws_usable, ws_bytes, cus);
    if (variant == MI355_GEMM_ROWS_MTILED) {
        if (tiles.mt == 0) tiles = rowsm_plan(M, N, K, cus);
        return variant;
    }
    tiles = rowsm_ahead(M, N, K, variant, ws_usable ? ws_bytes : 0, cus);
    return rowsm_limits_ok(tiles, M, K, lda, as_m, as_k) ? MI355_GEMM_ROWS_MTILED : variant;
}

}  // namespace mi355

using namespace mi355;

extern "C" size_t mi355_block_fp8_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int32_t variant) {
    // sized from the launch plan of the current device (256 compute units when no device is visible)
    return workspace_bytes_for(M, N, K, variant, device_cus());
}

extern "C" int32_t mi355_block_fp8_gemm_plan(int64_t M, int64_t N, int64_t K, size_t ws_bytes, int32_t cus) {
    if (M <= 0 || N <= 0 || K <= 0 || K % kBlockK != 0) return MI355_GEMM_GENERIC;
    if (cus <= 0) cus = device_cus();
    return resolve_auto(M, N, K, K, K, K / kBlockK, 1, ws_bytes > 0, ws_bytes, cus);
}

extern "C" int32_t mi355_block_fp8_gemm_over_m(int64_t M, int64_t N, int64_t K, size_t ws_bytes, int32_t cus) {
    if (cus <= 0) cus = device_cus();
    if (M <= 0 || N <= 0 || K <= 0 || K % kBlockK != 0) return 0;
    RowsMPlan tiles;
    return auto_launch(M, N, K, K, K, K / kBlockK, 1, ws_bytes > 0, ws_bytes, cus, tiles) == MI355_GEMM_ROWS_MTILED ? 1 : 0;
}

extern "C" int32_t mi355_block_fp8_gemm_launched(int64_t M, int64_t N, int64_t K, size_t ws_bytes, int32_t cus) {
    if (cus <= 0) cus = device_cus();
    const int variant = mi355_block_fp8_gemm_plan(M, N, K, ws_bytes, cus);
    return launched_for(variant, M, N, K, K, K, K / kBlockK, ws_bytes > 0, ws_bytes, cus);
}

/* The kernel the shape table picks for a packed, aligned problem on the current device (256 compute units when no
 * device is visible): one of the MI355_GEMM_* codes.  A launch may still fall back when a limit or the workspace of
 * that kernel is not met. */
extern "C" int32_t mi355_block_fp8_gemm_variant(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % kBlockK != 0) return MI355_GEMM_GENERIC;
    return pick_variant(M, N, K, device_cus());
}

static int block_fp8_gemm_impl(const void *A, const void *B, const float *As, const float *Bs, void *C, int64_t M,
                               int64_t N, int64_t K, int64_t lda, int64_t ldb_k, int64_t ldb_n, int64_t ldc,
                               int64_t as_m, int64_t as_k, int64_t bs_k, int64_t bs_n, int32_t block_n,
                               int32_t block_k, void *ws, size_t ws_bytes, int32_t variant, int32_t c_dtype,
                               void *stream) {
    if (M < 0 || N < 0 || K < 0) return MI355_EINVAL;
    if (c_dtype != MI355_DTYPE_BF16 && c_dtype != MI355_DTYPE_F16) return MI355_EUNSUPPORTED;
    const int out_f16 = c_dtype == MI355_DTYPE_F16 ? 1 : 0;
    if (block_n <= 0 || block_k <= 0) return MI355_EINVAL;
    // the tiled kernels are built for 128x128 weight blocks; other block sizes run on the plain kernel
    const bool blocks128 = block_n == kBlockN && block_k == kBlockK;
    if (!blocks128 && variant != MI355_GEMM_AUTO && variant != MI355_GEMM_GENERIC) return MI355_EUNSUPPORTED;
    if (M == 0 || N == 0) return MI355_OK;
    if (K == 0) return MI355_ESHAPE;
    if (!A || !B || !As || !Bs || !C) return MI355_EINVAL;
    if (lda < K || ldc < N) return MI355_ESHAPE;
    if (M >= (1ll << 31) || N >= (1ll << 31) || K >= (1ll << 31)) return MI355_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const int cus = device_cus();

    const bool fast = fast_layout_ok(A, B, K, lda, ldb_k, ldb_n) &&
                      // 32-bit byte offsets inside a tile / scale column
                      256 * lda < (1ll << 32) && 256 * ldb_n < (1ll << 32) && 256 * as_m * 4 < (1ll << 32) &&
                      as_m >= 0 && as_k >= 0;
    const bool was_auto = variant == MI355_GEMM_AUTO;
    RowsMPlan over_m = {0, 0, 0, 0};
    if (was_auto) {
        const bool ws_usable = ws && ((uintptr_t)ws & 15) == 0;
        variant = fast && blocks128 ? auto_launch(M, N, K, lda, ldb_n, as_m, as_k, ws_usable, ws_bytes, cus, over_m) : MI355_GEMM_GENERIC;
    }
    if (was_auto && variant == MI355_GEMM_TILE256) {
        const int64_t n1 = n_split_rows(M, N, K, cus);
        if (n1 > 0 && ldb_n * n1 % 16 == 0) {
            const int r = block_fp8_gemm_impl(A, B, As, Bs, C, M, n1, K, lda, ldb_k, ldb_n, ldc, as_m, as_k, bs_k, bs_n,
                                              block_n, block_k, ws, ws_bytes, MI355_GEMM_TILE256, c_dtype, stream);
            if (r != MI355_OK) return r;
            return block_fp8_gemm_impl(A, (const uint8_t *)B + n1 * ldb_n, As, Bs + n1 / kBlockN * bs_n,
                                       (uint16_t *)C + n1, M, N - n1, K, lda, ldb_k, ldb_n, ldc, as_m, as_k, bs_k, bs_n,
                                       block_n, block_k, ws, ws_bytes, MI355_GEMM_AUTO, c_dtype, stream);
        }
    }
    if (variant != MI355_GEMM_GENERIC && !fast) return MI355_EALIGN;

    if (variant == MI355_GEMM_GENERIC) {
        const int64_t blocks = (M * N + 255) / 256;
        if (blocks >= (1ll << 31)) return MI355_EUNSUPPORTED;
        return launch(block_fp8_gemm_generic_kernel, dim3((uint32_t)blocks), dim3(256), 0, st, (const uint8_t *)A,
                      (const uint8_t *)B, As, Bs, (uint16_t *)C, (int)M, (int)N, (int)K, lda, ldb_k, ldb_n, ldc, as_m,
                      as_k, bs_k, bs_n, (int)block_n, (int)block_k, out_f16);
    }

    GemmArgs a = {};
    a.out_f16 = out_f16;
    a.X = (const uint8_t *)A;
    a.W = (const uint8_t *)B;
    a.Xs = As;
    a.Ws = Bs;
    a.C = (uint16_t *)C;
    a.M = (int)M;
    a.N = (int)N;
    a.K = (int)K;
    a.ldx = lda;
    a.ldw = ldb_n;
    a.ldc = ldc;
    a.xs_m = as_m;
    a.xs_k = as_k;
    a.ws_n = bs_n;
    a.ws_k = bs_k;
    a.vec_store = (((uintptr_t)C & 15) == 0 && ldc % 8 == 0 && N % 8 == 0) ? 1 : 0;

    switch (variant) {
        case MI355_GEMM_TILE256_ONCE:  // kept for comparison
            ws = nullptr;
            [[fallthrough]];
        case MI355_GEMM_TILE256:
        case MI355_GEMM_TILE256_STREAMK: {
            a.tiles_m = (a.M + 255) / 256;
            a.tiles_n = (a.N + 255) / 256;
            a.total_tiles = a.tiles_m * a.tiles_n;
            // stream-K when asked for and worth it on this device; the plain tile loop otherwise
            const int groups =
                variant == MI355_GEMM_TILE256_STREAMK ? stream_k_groups(a.total_tiles, a.K / kBlockK, cus, a.tiles_m) : 0;
            const int r = launch_pp<false>(a, ws, ws_bytes, cus, groups, st);
            if (r != MI355_EUNSUPPORTED) return r;
            return launch_dense<256, 256, 2, 4, 2>(a, st);  // K ranges past the ping-pong kernel's LDS layout
        }
        case MI355_GEMM_TILE256_RING:  // kept for comparison
            return launch_dense<256, 256, 2, 4, 2>(a, st);
        case MI355_GEMM_TILE256x128: {
            const int splits = tile256x128_splits(M, N, K, cus);
            if (splits <= 1 || !ws || ws_bytes < tile256x128_workspace(M, N, splits) || ((uintptr_t)ws & 15))
                return launch_dense<256, 128, 2, 4, 3>(a, st);
            a.tiles_m = (a.M + 255) / 256;
            a.tiles_n = (a.N + 127) / 128;
            a.total_tiles = a.tiles_m * a.tiles_n;
            a.splits = splits;
            a.counters = (uint32_t *)ws;
            a.partials = (float *)((uint8_t *)ws + MI355_WS_COUNTER_BYTES);  // the counter words stay untouched
            const int r = launch_tile<256, 128, 2, 4, 3, kSplitK>(a, a.total_tiles * splits, st);
            if (r != MI355_OK) return r;
            return launch(tile_splitk_reduce_kernel<256, 128, 2, 4>, dim3(a.total_tiles * 16), dim3(512), 0, st, a);
        }
        case MI355_GEMM_TILE128: {
            const int splits = tile128_splits(M, N, K, cus);
            if (splits <= 1 || !ws || ws_bytes < tile128_workspace(M, N, splits) || ((uintptr_t)ws & 15))
                return launch_dense<128, 128, 2, 2, 2>(a, st);  // without a workspace the split is simply not used
            a.tiles_m = (a.M + 127) / 128;
            a.tiles_n = (a.N + 127) / 128;
            a.total_tiles = a.tiles_m * a.tiles_n;
            a.splits = splits;
            a.counters = (uint32_t *)ws;
            a.partials = (float *)((uint8_t *)ws + MI355_WS_COUNTER_BYTES);
            const int r = launch_tile<128, 128, 2, 2, 2, kSplitK>(a, a.total_tiles * splits, st);
            if (r != MI355_OK) return r;
            return launch(tile_splitk_reduce_kernel<128, 128, 2, 2>, dim3(a.total_tiles * 16), dim3(256), 0, st, a);
        }
        case MI355_GEMM_SKINNY_XSHARE: {
            if (M <= 32 || M > 64) return MI355_EUNSUPPORTED;
            if (N * ldb_n >= (1ll << 32) || M * lda >= (1ll << 32) || M * as_m >= (1ll << 32)) return MI355_EUNSUPPORTED;
            if ((N + XshareCfg::BN - 1) / XshareCfg::BN * 4 > MI355_WS_COUNTER_BYTES) return MI355_EUNSUPPORTED;
            int splits = xshare_splits(N, K, cus);
            if (splits > 1 && (!ws || ws_bytes < xshare_workspace(N, splits) || ((uintptr_t)ws & 15))) {
                if (was_auto) splits = 1;  // the table's choice runs unsplit without a workspace
                else return MI355_EWORKSPACE;
            }
            return launch_xshare(a, splits, ws, st);
        }
        case MI355_GEMM_ROWS128: {
            if (!rows128_limits_ok(M, N, K, lda, as_m, as_k, cus)) return MI355_EUNSUPPORTED;
            if (rows128_over_m(M, N, K, cus)) return launch_rowsm(a, rowsm_plan(M, N, K, cus), st);
            Rows128Plan pl = rows128_plan(M, N, K, cus);
            pl.turned = was_auto || M <= 64;
            if (pl.splits > 1 && (!ws || ws_bytes < rows128_workspace(M, N, K, cus) || ((uintptr_t)ws & 15)))
                return MI355_EWORKSPACE;
            return launch_rows128(a, pl, rows128_mt(M), false, ws, st);
        }
        case MI355_GEMM_SKINNY_ROWS: {
            const int ok = skinny_rows_check(M, N, K, lda, ldb_n, as_m, cus, ws && ((uintptr_t)ws & 15) == 0, ws_bytes);
            if (ok != MI355_OK) return ok;
            const SkinnyPlan sp = skinny_many_rows_plan(M, N, K, cus);
            switch (skinny_mt(M)) {
                case 5: return launch_stream_many_rows<5>(a, sp, ws, st);
                case 6: return launch_stream_many_rows<6>(a, sp, ws, st);
                case 7: return launch_stream_many_rows<7>(a, sp, ws, st);
                default: return launch_stream_many_rows<8>(a, sp, ws, st);
            }
        }
        case MI355_GEMM_ROWS_MTILED: {
            const RowsMPlan mp = was_auto ? over_m : rowsm_plan(M, N, K, cus);
            if (!was_auto && rowsm_round_plan(M, N, cus).mt == 0) return MI355_EUNSUPPORTED;  // by name: a single round
            if (!rowsm_limits_ok(mp, M, K, lda, as_m, as_k)) return MI355_EUNSUPPORTED;
            return launch_rowsm(a, mp, st);
        }
        case MI355_GEMM_SKINNY_CU: {
            const int tnw = streamcu_tnw(M, N, K, lda, ldb_n, as_m, cus);
            if (tnw == 0) return MI355_EUNSUPPORTED;
            return launch_streamcu(a, tnw, st);
        }
        case MI355_GEMM_SKINNY: {
            const int ok = skinny_check(M, N, K, lda, ldb_n, as_m, cus, ws && ((uintptr_t)ws & 15) == 0, ws_bytes);
            const bool whole = ok == MI355_EWORKSPACE && skinny_runs_whole(M, N, cus);  // (AUTO does not come here then)
            if (ok != MI355_OK && !whole) return ok;
            const SkinnyPlan pl = whole ? skinny_whole_plan(N) : skinny_plan(M, N, K, cus);
            switch (skinny_mt(M)) {
                case 1: return launch_stream_mt<1>(a, pl, ws, st);
                case 2: return launch_stream_mt<2>(a, pl, ws, st);
                case 3: return launch_stream_mt<3>(a, pl, ws, st);
                default: return launch_stream_mt<4>(a, pl, ws, st);
            }
        }
        default:
            return MI355_EINVAL;
    }
}

extern "C" int mi355_block_fp8_gemm(const void *A, const void *B, const float *As, const float *Bs, void *C,
                                    int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb_k, int64_t ldb_n,
                                    int64_t ldc, int64_t as_m, int64_t as_k, int64_t bs_k, int64_t bs_n,
                                    int32_t block_n, int32_t block_k, void *ws, size_t ws_bytes, int32_t variant,
                                    void *stream) {
    return block_fp8_gemm_impl(A, B, As, Bs, C, M, N, K, lda, ldb_k, ldb_n, ldc, as_m, as_k, bs_k, bs_n, block_n,
                               block_k, ws, ws_bytes, variant, MI355_DTYPE_BF16, stream);
}

extern "C" int mi355_block_fp8_gemm_dtype(const void *A, const void *B, const float *As, const float *Bs, void *C,
                                          int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb_k,
                                          int64_t ldb_n, int64_t ldc, int64_t as_m, int64_t as_k, int64_t bs_k,
                                          int64_t bs_n, int32_t block_n, int32_t block_k, void *ws, size_t ws_bytes,
                                          int32_t variant, int32_t c_dtype, void *stream) {
    return block_fp8_gemm_impl(A, B, As, Bs, C, M, N, K, lda, ldb_k, ldb_n, ldc, as_m, as_k, bs_k, bs_n, block_n,
                               block_k, ws, ws_bytes, variant, c_dtype, stream);
}

namespace mi355 {

__global__ __launch_bounds__(256) void zero_words_kernel(uint32_t *p, uint32_t n) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n) p[i] = 0u;
}

}  // namespace mi355

// ---- the entry point that allocates nothing -------------------------------------------------------------
// Split-K partials, arrival counters and the tile counters of the persistent launch live in a fixed array in
// the library's own device image instead of a caller-owned workspace.  Every GPU holds its own copy of the
// array at its own address; in host code the array's name is only a handle for hipGetSymbolAddress.
namespace mi355 {

constexpr size_t kScratchBytes = (size_t)MI355_WS_COUNTER_BYTES + ((size_t)MI355_NOALLOC_PARTIAL_MIB << 20);
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

// Device address of `scratch` on the current device, looked up on the first call per device.
static void *scratch_ptr() {
    static std::atomic<void *> ptrs[kMaxDevices];
    const int dev = current_device();
    if (dev < 0 || dev >= kMaxDevices) return nullptr;
    void *p = ptrs[dev].load(std::memory_order_acquire);
    if (p) return p;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
    ptrs[dev].store(p, std::memory_order_release);
    return p;
}

}  // namespace mi355

extern "C" int mi355_block_fp8_gemm_noalloc(const void *A, const void *B, const float *As, const float *Bs, void *C,
                                            int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb_k,
                                            int64_t ldb_n, int64_t ldc, int64_t as_m, int64_t as_k, int64_t bs_k,
                                            int64_t bs_n, int32_t block_n, int32_t block_k, int32_t variant,
                                            void *stream) {
    const size_t need = mi355_block_fp8_gemm_workspace_bytes(M, N, K, variant);
    // a forced kernel that needs more than the array holds is an error; the shape table (MI355_GEMM_AUTO) gets
    // the whole array and takes the next best plan that fits into it
    if (need > kScratchBytes && variant != MI355_GEMM_AUTO &&
        !(variant == MI355_GEMM_SKINNY && skinny_runs_whole(M, N, device_cus())))
        return MI355_ESCRATCH;
    void *ws = nullptr;
    if (need > 0) {
        ws = scratch_ptr();
        if (!ws) return MI355_ELAUNCH;
        // The array keeps what the last call left.  The kernels need their counter words zero and leave them
        // zero, but a launch that was aborted would not have: clear them here (a fill kernel, not a memset node,
        // so that the call can be captured into a HIP graph).
        const uint32_t words = MI355_WS_COUNTER_BYTES / 4;
        const int rc = launch(zero_words_kernel, dim3(words / 256), dim3(256), 0, (hipStream_t)stream, (uint32_t *)ws, words);
        if (rc != MI355_OK) return rc;
    }
    return mi355_block_fp8_gemm(A, B, As, Bs, C, M, N, K, lda, ldb_k, ldb_n, ldc, as_m, as_k, bs_k, bs_n, block_n,
                                block_k, ws, ws ? kScratchBytes : 0, variant, stream);
}

/* Re-zeroes the counter words of a caller-owned workspace (recovery after an aborted launch). */
extern "C" int mi355_reset_workspace(void *ws, size_t ws_bytes, void *stream) {
    if (!ws || ws_bytes < (size_t)MI355_WS_COUNTER_BYTES || ((uintptr_t)ws & 3)) return MI355_EWORKSPACE;
    const uint32_t words = MI355_WS_COUNTER_BYTES / 4;
    return launch(zero_words_kernel, dim3(words / 256), dim3(256), 0, (hipStream_t)stream, (uint32_t *)ws, words);
}

// Whether the entries of a 16- or 32-row schedule run as weight streams or as ring tiles (16 or 32 x 128, DMA into LDS).
// The stream has no barrier in its K loop, but its 64-column tiles, two to a compute unit, need enough of them to even out.
// Over 8 to 256 experts, N = 512 to 7168, K = 2048 to 8192, even and uneven routing, weights from HBM, time of the stream
// over that of the ring tiles:
//  * fewer than 16 K steps give a wave too few (128 experts, N = 2048, K = 768, top-8, 4 / 8 tokens: 14.7 / 22.2 us against
//    11.5 / 19.3, level from 16 tokens on; K = 1408, 4 tokens: 16.4 against 14.9)
//  * up to 8 rows per expert it is ahead (0.73 - 0.97) except with 1 to 1.6 tiles per unit under a K below 7168 (1.02 - 1.09);
//    the ring tiles take rows that lie a multiple of 4096 bytes apart badly (0.75 - 0.9 wherever there are tiles enough)
//  * with 9 to 16 rows second entries come into it: one more round if the tiles fill one (1.04 - 1.24), half a round up to
//    3.1 tiles per unit under a short K (1.02 - 1.11); else 0.8 - 1.0
//  * from 17 rows on a stream step costs two row blocks: still ahead under a K of 2048 or 7168 (0.86 - 0.98), not between
//    (0.97 - 1.05), with a narrow N (N = 512, 1024: 1.04 - 1.09) or from 21 rows on (uneven routing: 1.04 - 1.1)
// With 8 experts or fewer the alternative to it is blocks of 64 rows, far behind where it is taken (mi355_grouped_block_m).
static bool grouped_streams(int64_t rows_per_expert, int64_t num_experts, int64_t N, int64_t K, int cus) {
    if (K < 16 * kBlockK) return false;
    if (num_experts <= 8) return true;
    const int64_t tiles = num_experts * ((N + 63) / 64);
    const bool ring_is_slow = K % 4096 == 0;
    if (rows_per_expert <= 8) return K >= 7168 || ring_is_slow || tiles <= cus || tiles * 5 > 8 * (int64_t)cus;
    if (rows_per_expert > 16 && !ring_is_slow && (rows_per_expert > 20 || N < 1536 || (K > 2176 && K < 7168))) return false;
    if (ring_is_slow || (K >= 4096 && rows_per_expert <= 16)) return tiles * 5 > 8 * (int64_t)cus;
    return tiles * 10 > 31 * (int64_t)cus;
}

extern "C" int32_t mi355_grouped_block_m(int64_t num_pairs, int32_t num_experts, int64_t N, int64_t K) {
    if (num_experts <= 0) return 64;
    const int64_t avg = num_pairs / num_experts;
    // 256-row schedule blocks run as the persistent launch with two queues: blocks of more than 64 rows on the
    // 256x256 ping-pong tile (it skips the empty 64-row halves of ragged blocks), the others on the 64x512
    // weight-streaming tile.  That launch needs more tiles than compute units, and its time hardly depends on how the rows
    // are spread.  With fewer rows the weight streams of 16- and 32-row schedules (gemm_gstream.hpp, where they are
    // taken) are ahead: they read at 6 to 7 TB/s, once per 32 rows of an expert, so what they cost follows the second reads
    // of popular experts.  Every line between the two lies where Zipf(1.1) popularity costs the stream its lead.
    const int cus = device_cus();
    const int64_t tiles256 = (int64_t)num_experts * ((N + 255) / 256);
    const bool two_queues = tiles256 > cus, stream = grouped_streams(avg, num_experts, N, K, cus);
    // Measured over Qwen3-MoE (128 experts), DeepSeek-V2-Lite (64), Mixtral (8), a DeepSeek-V3 expert-parallel slice
    // (32 experts, N = 512) and a 16-expert shape, 8 to 8192 tokens, uniform routing:
    //  * 128-row blocks are ahead of the 256-row launch up to a few hundred rows per expert where the whole launch
    //    is small - few tiles (32 experts x N = 512, 128 rows each: 63.9 us against 85.5; Mixtral down, 64 / 128
    //    rows: 128 / 150 against 154 / 163) or under 0.5 GB of weights with a short K (Qwen3-30B down, K = 768,
    //    64 / 128 rows: 60.5 / 89.9 against 81.1 / 105.6; DeepSeek-V2-Lite down, 96 rows: 52.3 against 87.1) -
    //    and behind it on the large ones (DeepSeek-V3, 128 rows: 2189 against 1747)
    if (avg > 32) {
        // (few tiles: from 33 rows per expert where an expert is large and a second block of it costs a second
        // read of its weights, from 65 where it is small - 32 experts x N = 512, 64 rows: 43.6 us for 64-row blocks
        // against 63.0 - and there up to 256 rows: 74.0 against 88.5)
        const bool large_expert = N * K >= 30000000ll;
        if (tiles256 * 2 <= cus && avg > (large_expert ? 32 : 64) && avg <= (large_expert ? 160 : 256)) return 128;
        if ((int64_t)num_experts * N * K <= 500000000ll && K <= 2048 && avg <= (K <= 1536 ? 224 : 112)) return 128;
    }
    //  * with 8 experts every block re-reads a large expert, and 64-row blocks beat ring tiles of the average size from 9
    //    rows per expert on, the weight streams from 21 (Mixtral gate_up, 20 rows, even / Zipf: 156 / 171 us for the 32-row
    //    stream against 215 / 214) - from 13 where the experts' 64-column tiles just fill the two workgroups a unit holds
    //    and the second entry of one expert starts another round (Mixtral down, 512 tiles, 12 rows: 74 / 78 against 82 /
    //    83; 14 rows, with a second entry: 101 against 83; N = 4096, K = 7168: 53 against 46)
    if (num_experts <= 8) {
        const int64_t tiles64 = (int64_t)num_experts * ((N + 63) / 64);
        const bool fills_one_round = tiles64 <= 2 * cus && tiles64 * 5 > 8 * (int64_t)cus;
        if (avg > (!stream ? 8 : fills_one_round ? 12 : 20) && avg <= 40) return 64;
    }
    //  * where an expert's N is wide the two-queue launch takes over from 12 rows per expert under a short K.  Against the
    //    streams it does so the earlier the more experts there are to be popular, and the less a step costs beside the
    //    outputs (us for the stream, even / Zipf routing, against the two-queue launch, which is the same for both within
    //    5 %.  256 experts, N = 4096, K = 7168, 12 / 14 / 16 / 20 rows: 1124 / 1252, 1144 / 1298, 1166 / 1371, 1230 / 1505
    //    against 1264 ... 1297; N = 7168, K = 2048, 12 / 16 rows: 615 / 683, 666 / 758 against 674 / 688.  128 experts, 16 /
    //    18 rows: 577 / 664, 595 / 697 against 641 / 677; 12 / 14 rows: 300 / 345, 312 / 351 against 345 / 348.  64 experts,
    //    20 rows: 298 / 358 against 331 / 374; 14 / 16 rows: 151 / 168, 158 / 192 against 185 / 185.  32 experts, 20 rows:
    //    145 / 173 against 176 / 221; 16 / 20 rows: 90 / 95, 93 / 104 against 101 / 103)
    //  * from 25 where N is not wide (Qwen3-30B gate_up, N = 1536, 24 rows: 88 / 100 us for the 32-row stream against 95)
    int64_t line = 25;
    if (N >= 4096) {
        if (!stream) line = 12;
        else if (K >= 4096) line = num_experts <= 64 ? 21 : num_experts <= 128 ? 17 : 13;
        else line = num_experts <= 32 ? 17 : num_experts <= 64 ? 16 : 12;
    }
    if (avg > 64 || (two_queues && avg >= line)) return 256;
    //  * a stream's 16-row entries run in pairs, and the workgroups of the second ones, which have nothing to do, show where
    //    an entry is short and an expert has few tiles (Qwen3-30B gate_up, 16 rows, even / Zipf: 80 / 86 us for 16-row
    //    entries, 75 / 82 for 32-row ones, 87 / 84 for the ring tiles; level with a longer K or a wide N)
    if (stream && K < 4096 && N < 4096 && avg > 8 && avg <= 32) return 32;
    if (avg <= 16) return 16;
    if (avg <= 32) return 32;
    return 64;
}

extern "C" size_t mi355_grouped_workspace_bytes(int64_t table_rows) {
    return grouped_workspace(table_rows < 0 ? 0 : table_rows);
}

static int grouped_block_fp8_gemm_impl(const void *Xq, const float *Xs, const void *W, const float *Ws,
                                       const int32_t *expert_to_token_index, const float *expert_to_weight,
                                       const int32_t *expert_token_num, const int32_t *table, int64_t table_rows,
                                       int32_t block_m, int64_t num_pairs, int64_t num_tokens, int32_t num_experts,
                                       int32_t topk_num, int64_t N, int64_t K, int32_t mul_routed_weight, void *out,
                                       void *ws, size_t ws_bytes, int32_t out_dtype, const void *bias,
                                       int32_t bias_dtype, int64_t bias_stride_e, void *stream) {
    if (out_dtype != MI355_DTYPE_BF16 && out_dtype != MI355_DTYPE_F16) return MI355_EUNSUPPORTED;
    if (bias && bias_dtype != MI355_DTYPE_BF16 && bias_dtype != MI355_DTYPE_F16 && bias_dtype != MI355_DTYPE_F32)
        return MI355_EUNSUPPORTED;
    if (bias && bias_stride_e < 0) return MI355_EINVAL;
    if (num_pairs < 0 || num_tokens < 0 || num_experts <= 0 || topk_num <= 0 || N < 0 || K < 0 || table_rows < 0)
        return MI355_EINVAL;
    if (num_pairs == 0 || N == 0 || table_rows == 0) return MI355_OK;
    if (!Xq || !Xs || !W || !Ws || !expert_to_token_index || !expert_to_weight || !expert_token_num || !table || !out)
        return MI355_EINVAL;
    if (K == 0 || K % kBlockK != 0) return MI355_ESHAPE;
    if (((uintptr_t)Xq & 15) || ((uintptr_t)W & 15)) return MI355_EALIGN;
    if (num_tokens * K >= (1ll << 32) || 256 * K >= (1ll << 32) || num_tokens * (K / kBlockK) * 4 >= (1ll << 32) ||
        N >= (1ll << 31) || num_pairs >= (1ll << 31))
        return MI355_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const int64_t KB = K / kBlockK, NB = (N + kBlockN - 1) / kBlockN;

    GemmArgs a = {};
    a.out_f16 = out_dtype == MI355_DTYPE_F16 ? 1 : 0;
    a.X = (const uint8_t *)Xq;
    a.W = (const uint8_t *)W;
    a.Xs = Xs;
    a.Ws = Ws;
    a.C = (uint16_t *)out;
    a.M = (int)num_pairs;
    a.N = (int)N;
    a.K = (int)K;
    a.ldx = K;
    a.ldw = K;
    a.ldc = N;
    a.xs_m = KB;
    a.xs_k = 1;
    a.ws_n = KB;
    a.ws_k = 1;
    a.vec_store = (((uintptr_t)out & 15) == 0 && N % 8 == 0) ? 1 : 0;
    a.table = table;
    a.e2t_index = expert_to_token_index;
    a.e2t_weight = expert_to_weight;
    a.e_num = expert_token_num;
    a.w_e = N * K;
    a.ws_e = NB * KB;
    a.num_pairs = (int)num_pairs;
    a.topk = topk_num;
    a.mul_weight = mul_routed_weight ? 1 : 0;
    a.bias = bias;
    a.bias_e = bias_stride_e;
    a.bias_dtype = bias_dtype;
    a.tiles_m = (int)table_rows;

    auto finish = [&](int BN) {
        a.tiles_n = (int)((N + BN - 1) / BN);
        a.total_tiles = a.tiles_m * a.tiles_n;
        a.blocks_per_xcd = (a.total_tiles + 7) / 8;
        return a.blocks_per_xcd * 8;
    };
    if ((int64_t)table_rows * ((N + 127) / 128) >= (1ll << 31)) return MI355_EUNSUPPORTED;
    switch (block_m) {
        case 16:
        case 32: {
            // (a padded layout's rows per expert are not known here: as many as its block holds)
            const int64_t rows = num_pairs >= num_tokens ? num_pairs / num_experts : block_m == 16 ? 16 : 20;
            if (grouped_streams(rows, num_experts, N, K, device_cus())) {
                const int r = launch_gstream(a, block_m, num_experts, st);
                if (r != MI355_EUNSUPPORTED) return r;  // (a K whose scales do not fit the LDS, or 2^31 tiles and more)
            }
            if (block_m == 16) return launch_grouped_tile<16, 128, 1, 4, 4>(a, finish(128), st);
            return launch_grouped_tile<32, 128, 1, 4, 4>(a, finish(128), st);
        }
        case 64: return launch_grouped_tile<64, 128, 1, 4, 4>(a, finish(128), st);
        case 128: return launch_grouped_tile<128, 128, 2, 2, 2>(a, finish(128), st);
        case 256:
            finish(256);
            return launch_grouped_pp(a, ws, ws_bytes, device_cus(), st);
        default: return MI355_EINVAL;
    }
}

extern "C" int mi355_grouped_block_fp8_gemm(const void *Xq, const float *Xs, const void *W, const float *Ws,
                                            const int32_t *expert_to_token_index, const float *expert_to_weight,
                                            const int32_t *expert_token_num, const int32_t *table,
                                            int64_t table_rows, int32_t block_m, int64_t num_pairs,
                                            int64_t num_tokens, int32_t num_experts, int32_t topk_num, int64_t N,
                                            int64_t K, int32_t mul_routed_weight, void *out, void *ws,
                                            size_t ws_bytes, void *stream) {
    return grouped_block_fp8_gemm_impl(Xq, Xs, W, Ws, expert_to_token_index, expert_to_weight, expert_token_num, table,
                                       table_rows, block_m, num_pairs, num_tokens, num_experts, topk_num, N, K,
                                       mul_routed_weight, out, ws, ws_bytes, MI355_DTYPE_BF16, nullptr, 0, 0, stream);
}

extern "C" int mi355_grouped_block_fp8_gemm_dtype(const void *Xq, const float *Xs, const void *W, const float *Ws,
                                                  const int32_t *expert_to_token_index,
                                                  const float *expert_to_weight, const int32_t *expert_token_num,
                                                  const int32_t *table, int64_t table_rows, int32_t block_m,
                                                  int64_t num_pairs, int64_t num_tokens, int32_t num_experts,
                                                  int32_t topk_num, int64_t N, int64_t K, int32_t mul_routed_weight,
                                                  void *out, void *ws, size_t ws_bytes, int32_t out_dtype,
                                                  void *stream) {
    return grouped_block_fp8_gemm_impl(Xq, Xs, W, Ws, expert_to_token_index, expert_to_weight, expert_token_num, table,
                                       table_rows, block_m, num_pairs, num_tokens, num_experts, topk_num, N, K,
                                       mul_routed_weight, out, ws, ws_bytes, out_dtype, nullptr, 0, 0, stream);
}

extern "C" int mi355_grouped_block_fp8_gemm_bias(const void *Xq, const float *Xs, const void *W, const float *Ws,
                                                 const int32_t *expert_to_token_index, const float *expert_to_weight,
                                                 const int32_t *expert_token_num, const int32_t *table,
                                                 int64_t table_rows, int32_t block_m, int64_t num_pairs,
                                                 int64_t num_tokens, int32_t num_experts, int32_t topk_num, int64_t N,
                                                 int64_t K, int32_t mul_routed_weight, void *out, void *ws,
                                                 size_t ws_bytes, int32_t out_dtype, const void *bias,
                                                 int32_t bias_dtype, int64_t bias_stride_e, void *stream) {
    return grouped_block_fp8_gemm_impl(Xq, Xs, W, Ws, expert_to_token_index, expert_to_weight, expert_token_num, table,
                                       table_rows, block_m, num_pairs, num_tokens, num_experts, topk_num, N, K,
                                       mul_routed_weight, out, ws, ws_bytes, out_dtype, bias, bias_dtype,
                                       bias_stride_e, stream);
}
