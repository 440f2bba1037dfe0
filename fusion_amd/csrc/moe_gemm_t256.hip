// The 256 x 256 tile mapping (moe_gemm_t256.h): the entry, and the gated instances.  The
// instances are spread over three sources so that they compile in parallel.
#include "moe_gemm_t256.h"

namespace glm52 {
int launch_t256(const GemmArgs& a, int capacity, bool gated, bool weighted, hipStream_t st) {
  if ((a.n_out % (gated ? 256 : 512)) || (a.K % 64)) return GLM52_EUNSUPPORTED;
  if (a.merge_topk > 0 || a.epi != 0) {
    if (gated) return GLM52_EUNSUPPORTED;
    return launch_t256_epi(a, capacity, weighted, st);
  }
  if (!gated) return launch_t256_plain(a, capacity, weighted, st);
  return weighted ? launch_t256_w<true, true, 0>(a, capacity, st)
                  : launch_t256_w<true, false, 0>(a, capacity, st);
}
}  // namespace glm52
