// Host side of the weight stream with the activation block in LDS (gemm_rows128.hpp): one instantiation per number of row
// blocks, workgroup width and way to run it, by far the most of this library, so they are spread over the translation units
// rows128_few.hip, rows128_some.hip and rows128_many.hip.
#pragma once
#include "gemm_tile.hpp"

namespace mi355 {

constexpr int64_t kRows128NarrowMaxM = 208;  // the last row count with narrow workgroups above 128 rows

struct Rows128Plan {
    int wv, bn, splits, tiles, tn;
    bool turned;  // tiles may start at different K steps (launch_rows128_as)
};

// `mt` row blocks (1..24; over_m: 1..13, a.tiles_m x a.tiles_n tiles, pl.tiles workgroups).
int launch_rows128_few(GemmArgs &a, const Rows128Plan &pl, int mt, bool over_m, void *ws, hipStream_t st);   // 1..8
int launch_rows128_some(GemmArgs &a, const Rows128Plan &pl, int mt, bool over_m, void *ws, hipStream_t st);  // 9..13
int launch_rows128_many(GemmArgs &a, const Rows128Plan &pl, int mt, bool over_m, void *ws, hipStream_t st);  // 14..24

inline int launch_rows128(GemmArgs &a, const Rows128Plan &pl, int mt, bool over_m, void *ws, hipStream_t st) {
    if (mt <= 8) return launch_rows128_few(a, pl, mt, over_m, ws, st);
    if (mt <= 13) return launch_rows128_some(a, pl, mt, over_m, ws, st);
    return launch_rows128_many(a, pl, mt, over_m, ws, st);
}

}  // namespace mi355
