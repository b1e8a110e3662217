// The weight stream with the activation block in LDS on 1 to 8 row blocks.
#include "rows128_instances.hpp"

namespace mi355 {

int launch_rows128_few(GemmArgs &a, const Rows128Plan &pl, int mt, bool over_m, void *ws, hipStream_t st) {
    return launch_rows128_of<1, 8>(a, pl, mt, over_m, ws, st);
}

}  // namespace mi355
