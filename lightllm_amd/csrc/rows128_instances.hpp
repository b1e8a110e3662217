// The launches of rows128_launch.hpp for one number of row blocks.
#pragma once
#include "gemm_rows128.hpp"
#include "rows128_launch.hpp"
#include "stream_plan.hpp"

namespace mi355 {

template <int MT, int WV, int TN = (MT <= 8 ? 2 : 1), int XS = 0>
static int launch_rows128_as(GemmArgs &a, const Rows128Plan &pl, void *ws, hipStream_t st) {
    using Cfg = Rows128Cfg<MT, TN, WV, XS>;
    const int KB = a.K / kBlockK;
    const int steps = (KB + pl.splits - 1) / pl.splits;
    const int lds_bytes = Cfg::lds_bytes(steps);
    if (lds_bytes > 160 * 1024) {
        // the weight scales of a very long K leave no room for a third slot of X: eight waves of 16 weight rows on two
        if constexpr (Cfg::NSX == 3 && MT > 8) {
            Rows128Plan two = pl;
            two.wv = 8;
            two.tn = 1;
            two.bn = 128;
            const int tiles_n = (a.N + 127) / 128;
            if (a.tiles_m > 1) {
                a.tiles_n = tiles_n;
                a.total_tiles = a.tiles_m * tiles_n;
                two.tiles = (a.total_tiles + 7) / 8 * 8;
            } else {
                two.tiles = tiles_n;
            }
            return launch_rows128_as<MT, 8, 1, 2>(a, two, ws, st);
        }
        return MI355_EUNSUPPORTED;
    }
    if (pl.splits <= 1) {
        // Turned starts (stream_turn_mask) where a step is mostly weights: up to 96 rows (80 beyond K = 16384), or weights of
        // 200 MB and more (450 at K = 16384) (us, in step / turned: N = 28672, K = 4096, M = 64 / 80 / 128 29.2 / 30.5 / 36.2
        // against 26.3 / 28.2 / 37.3; 57344 x 8192, M = 64 / 128 / 160 115 / 122 / 119 against 85 / 97 / 108; 36864 x 20480, M =
        // 128 172 / 180; 22656 x 16384, M = 128 124 / 128; 12288 x 4096, M = 160 31.8 / 33.1).  Not with narrow workgroups on K =
        // 8192: tile t's rows then start 5 t or 6 t times 2^18 bytes on, its steps 5 t times 128, and the two meet again on the
        // same channels (32768 x 8192, M = 64 63.3 / 82.1; 24576: 50.6 / 60.6; with 256 weight rows 45056: 1.18 times ahead).
        // Tiles over M share their activation rows in the L2 step by step and lose that (K = 8192: 2 to 6 %).  The two buffers
        // of scale chunks want a multiple of 16 steps.  From 65 rows on, where the square tiles run as well, a launch asked for
        // by name keeps K order: its sums are then theirs bit for bit.
        if constexpr (MT <= 10 && TN == 2) {
            const int64_t weights = (int64_t)a.N * a.K;
            const bool weights_lead = a.M <= (a.K <= 16384 ? 96 : 80) || (a.K <= 16384 && weights >= (a.K < 16384 ? 200000000ll : 450000000ll));
            const bool meets = WV < 8 && a.K == 8192;
            if (pl.turned && weights_lead && !meets && a.tiles_m <= 1 && KB % 16 == 0 && (a.turn_mask = stream_turn_mask(a.K, KB)) != 0) {
                constexpr auto turned = block_fp8_gemm_rows128_kernel<MT, TN, WV, false, true, XS>;
                if (!allow_lds<turned>(160 * 1024)) return MI355_ELAUNCH;
                return launch(turned, dim3(pl.tiles), dim3(Cfg::kThreads), lds_bytes, st, a);
            }
        }
        constexpr auto kernel = block_fp8_gemm_rows128_kernel<MT, TN, WV, false, false, XS>;
        if (!allow_lds<kernel>(160 * 1024)) return MI355_ELAUNCH;
        return launch(kernel, dim3(pl.tiles), dim3(Cfg::kThreads), lds_bytes, st, a);
    }
    if constexpr (WV == 8 && TN == (MT <= 8 ? 2 : 1)) {
        constexpr auto kernel = block_fp8_gemm_rows128_kernel<MT, TN, 8, true, false, XS>;
        if (!allow_lds<kernel>(160 * 1024)) return MI355_ELAUNCH;
        a.splits = pl.splits;
        a.partials = (float *)((uint8_t *)ws + MI355_WS_COUNTER_BYTES);  // the counter words stay untouched
        const int r = launch(kernel, dim3(pl.tiles * pl.splits), dim3(Cfg::kThreads), lds_bytes, st, a);
        if (r != MI355_OK) return r;
        return launch(rows128_reduce_kernel<MT, TN>, dim3((pl.tiles * Cfg::kWaves * MT + 3) / 4), dim3(256), 0, st, a);
    }
    return MI355_EINVAL;  // narrow workgroups never share K
}

template <int MT>
static int launch_rows128_mt(GemmArgs &a, const Rows128Plan &pl, void *ws, hipStream_t st) {
    if constexpr (MT <= 8) {
        if (pl.wv == 5) return launch_rows128_as<MT, 5>(a, pl, ws, st);
        if (pl.wv == 6) return launch_rows128_as<MT, 6>(a, pl, ws, st);
    } else if constexpr (MT <= (kRows128NarrowMaxM + 15) / 16) {
        if (pl.tn == 2) {
            switch (pl.wv) {
            case 5: return launch_rows128_as<MT, 5, 2>(a, pl, ws, st);
            case 6: return launch_rows128_as<MT, 6, 2>(a, pl, ws, st);
            case 7: return launch_rows128_as<MT, 7, 2>(a, pl, ws, st);
            case 8: return launch_rows128_as<MT, 8, 2>(a, pl, ws, st);
            default: return MI355_EINVAL;
            }
        }
        switch (pl.wv) {
        case 4: return launch_rows128_as<MT, 4>(a, pl, ws, st);
        case 5: return launch_rows128_as<MT, 5>(a, pl, ws, st);
        case 6: return launch_rows128_as<MT, 6>(a, pl, ws, st);
        case 7: return launch_rows128_as<MT, 7>(a, pl, ws, st);
        default: break;
        }
    }
    return launch_rows128_as<MT, 8>(a, pl, ws, st);
}

template <int MT>
static int launch_rowsm_mt(GemmArgs &a, const Rows128Plan &pl, hipStream_t st) {
    if constexpr (MT <= 8) {
        switch (pl.wv) {
            case 5: return launch_rows128_as<MT, 5>(a, pl, nullptr, st);
            case 6: return launch_rows128_as<MT, 6>(a, pl, nullptr, st);
            case 8: return launch_rows128_as<MT, 8>(a, pl, nullptr, st);
            default: return MI355_EINVAL;
        }
    } else {
        switch (pl.wv) {
            case 5: return launch_rows128_as<MT, 5, 2>(a, pl, nullptr, st);
            case 6: return launch_rows128_as<MT, 6, 2>(a, pl, nullptr, st);
            case 7: return launch_rows128_as<MT, 7, 2>(a, pl, nullptr, st);
            case 8: return launch_rows128_as<MT, 8, 2>(a, pl, nullptr, st);
            default: return MI355_EINVAL;
        }
    }
}

// One of FIRST..LAST row blocks.
template <int FIRST, int LAST>
static int launch_rows128_of(GemmArgs &a, const Rows128Plan &pl, int mt, bool over_m, void *ws, hipStream_t st) {
    if (mt == FIRST) {
        if constexpr (FIRST <= 13) {
            if (over_m) return launch_rowsm_mt<FIRST>(a, pl, st);
        }
        return over_m ? MI355_EINVAL : launch_rows128_mt<FIRST>(a, pl, ws, st);
    }
    if constexpr (FIRST < LAST) return launch_rows128_of<FIRST + 1, LAST>(a, pl, mt, over_m, ws, st);
    return MI355_EINVAL;
}

}  // namespace mi355
