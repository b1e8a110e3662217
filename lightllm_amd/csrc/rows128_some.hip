// The weight stream with the activation block in LDS on 9 to 13 row blocks.
#include "rows128_instances.hpp"

namespace mi355 {

int launch_rows128_some(GemmArgs &a, const Rows128Plan &pl, int mt, bool over_m, void *ws, hipStream_t st) {
    return launch_rows128_of<9, 13>(a, pl, mt, over_m, ws, st);
}

}  // namespace mi355
