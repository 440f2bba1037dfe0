// The grouped GEMM tiles of moe_gemm_tile.h: the plain instances with a bf16 store at 64 tokens per tile (a
// source each, so that they compile in parallel).
#include "moe_gemm_tile.h"

namespace glm52 {
template int launch_tile_plain<64>(const GemmArgs&, int, bool, hipStream_t);
}
