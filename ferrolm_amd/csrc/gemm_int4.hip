// The tiled GEMM (gemm_tiles.h) on int4 weights.
#include "gemm_tiles.h"

namespace fg {
template void run_mm<INT4>(hipStream_t, int, int, const GemvArgs&, hipEvent_t, hipEvent_t);
}
