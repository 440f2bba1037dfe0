// The grouped GEMM tiles of moe_gemm_tile.h: the gated instances at 256 tokens per tile (a
// source each, so that they compile in parallel).
#include "moe_gemm_tile.h"

namespace glm52 {
template int launch_tile_gated<256>(const GemmArgs&, int, bool, hipStream_t);
}
