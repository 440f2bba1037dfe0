// The grouped GEMM tiles of moe_gemm_tile.h: the o_proj and atomic-merge instances at 64 tokens per tile (a
// source each, so that they compile in parallel).
#include "moe_gemm_tile.h"

namespace glm52 {
template int launch_tile_epi<64>(const GemmArgs&, int, bool, hipStream_t);
}
