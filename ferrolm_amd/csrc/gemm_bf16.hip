// The tiled GEMM (gemm_tiles.h) on bf16 weights.
#include "gemm_tiles.h"

namespace fg {
template void run_mm<BF16>(hipStream_t, int, int, const GemvArgs&, hipEvent_t, hipEvent_t);
}
