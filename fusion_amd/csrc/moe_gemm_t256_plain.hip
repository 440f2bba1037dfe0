// The 256 x 256 tile mapping (moe_gemm_t256.h): the plain instances with a bf16 store.
#include "moe_gemm_t256.h"

namespace glm52 {
int launch_t256_plain(const GemmArgs& a, int capacity, bool weighted, hipStream_t st) {
  return weighted ? launch_t256_w<false, true, 0>(a, capacity, st)
                  : launch_t256_w<false, false, 0>(a, capacity, st);
}
}  // namespace glm52
