// The tiled GEMM (gemm_tiles.h) on int8 weights.
#include "gemm_tiles.h"

namespace fg {
template void run_mm<INT8>(hipStream_t, int, int, const GemvArgs&, hipEvent_t, hipEvent_t);
}
