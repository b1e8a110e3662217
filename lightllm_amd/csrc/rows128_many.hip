// The weight stream with the activation block in LDS on 14 to 24 row blocks.
#include "rows128_instances.hpp"

namespace mi355 {

int launch_rows128_many(GemmArgs &a, const Rows128Plan &pl, int mt, bool over_m, void *ws, hipStream_t st) {
    return launch_rows128_of<14, 24>(a, pl, mt, over_m, ws, st);
}

}  // namespace mi355
