// The 256 x 256 tile mapping (moe_gemm_t256.h): o_proj's epilogues (packed B only) and the
// atomic expert merge (weighted w2 only).
#include "moe_gemm_t256.h"

namespace glm52 {
int launch_t256_epi(const GemmArgs& a, int capacity, bool weighted, hipStream_t st) {
  if (a.merge_topk > 0) {
    if (!weighted || a.epi != 0) return GLM52_EUNSUPPORTED;
    return launch_t256_w<false, true, 4>(a, capacity, st);
  }
  if (weighted || !a.Wp) return GLM52_EUNSUPPORTED;
  if (a.epi == 1) return launch_t256_as<false, false, true, 1>(a, capacity, st);
  if (a.epi == 2) return launch_t256_as<false, false, true, 2>(a, capacity, st);
  return launch_t256_as<false, false, true, 3>(a, capacity, st);
}
}  // namespace glm52
