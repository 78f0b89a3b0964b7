// The bf16 GEMM tiles for K a multiple of the 64-k stage.
#include "gemm_tile.h"

namespace mi {
template int gemm_tiles<bf16, false>(const GemmArgs&, int64_t, int, int, hipStream_t);
}  // namespace mi
