// Entry of the grouped GEMM tiles (moe_gemm_tile.h), whose instances are in the sources
// moe_gemm_tile<tokens>_<kind>.hip.
#include "moe_gemm.h"
#include "tile_range.h"

namespace glm52 {
template <int MT>
int launch_tile_gated(const GemmArgs& a, int capacity, bool weighted, hipStream_t st);
template <int MT>
int launch_tile_plain(const GemmArgs& a, int capacity, bool weighted, hipStream_t st);
template <int MT>
int launch_tile_epi(const GemmArgs& a, int capacity, bool weighted, hipStream_t st);

namespace {
template <int MT>
int launch_mt(const GemmArgs& a, int capacity, bool gated, bool weighted, hipStream_t st) {
  if (a.merge_topk > 0 || a.epi != 0)
    return gated ? GLM52_EUNSUPPORTED : launch_tile_epi<MT>(a, capacity, weighted, st);
  return gated ? launch_tile_gated<MT>(a, capacity, weighted, st)
               : launch_tile_plain<MT>(a, capacity, weighted, st);
}
}  // namespace

int launch_tile(const GemmArgs& a, int capacity, bool gated, bool weighted, hipStream_t st) {
  if ((a.n_out % (gated ? 256 : 512)) || (a.K % 64)) return GLM52_EUNSUPPORTED;
  // row-major W: the rows of one expert are addressed with 32-bit byte offsets
  if (!a.Wp && !in_place_fits(gated ? a.gu_off : 0, a.n_out, a.swn, a.K)) return GLM52_EUNSUPPORTED;
  switch (a.BM) {
    case 64: return launch_mt<64>(a, capacity, gated, weighted, st);
    case 128: return launch_mt<128>(a, capacity, gated, weighted, st);
    case 256: return launch_mt<256>(a, capacity, gated, weighted, st);
    default: return GLM52_EUNSUPPORTED;
  }
}
}  // namespace glm52
