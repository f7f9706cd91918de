// fp32 GEMM tiles for one pair of operand layouts (gemm_tile.hpp), a translation unit of its own.
#include "gemm_tile.hpp"

namespace nchip {

int sg_tile_nn(SgArgs &p, int id, int64_t count, hipStream_t st, const char *what) {
    return sg_tile_run<true, false>(p, id, count, st, what);
}

}  // namespace nchip
