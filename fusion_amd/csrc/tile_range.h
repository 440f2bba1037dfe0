// The byte offsets and descriptor sizes of the grouped GEMM tiles' ring loads
// (moe_gemm_tile.h).  Plain C++, so that a host program can check them against every form of
// the buffer range check.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define GLM52_HD __host__ __device__ __forceinline__
#else
#define GLM52_HD inline
#endif

namespace glm52 {

constexpr uint32_t kTokenBytes = 0x7ffffff0u;  // descriptor size of the token rows (the entry
                                               // points refuse rows that reach past it)
constexpr uint32_t kInPlaceBytes = 0xfffffff0u;  // descriptor size of one expert's row-major W
constexpr uint32_t kNowhere = 0x90000000u;     // lane offset of a padding row: past kTokenBytes

// Whether one expert's row-major W rows -- 0 .. n_out - 1, and with gate_up > 0 those from
// gate_up on as well, k elements each at a stride of swn -- fit the descriptor, so that no
// lane's 32-bit offset wraps.
inline bool in_place_fits(int gate_up, int n_out, int64_t swn, int k) {
  return swn >= 0 &&
         (((int64_t)gate_up + n_out - 1) * swn + k) * 2 <= (int64_t)kInPlaceBytes;
}

// Stage s of nk (the item's first stage is krot, wrapping; `step` bytes from one stage to the
// next) of an operand of `bytes` bytes: the descriptor size and the scalar offsets of the stage
// and, where two are loaded together (nk, s and krot even, step 64), of the one after it.  The
// range check may compare a lane's offset with the size less the scalar offset, in 32 bits, so
// past the last stage both scalar offsets are 0, as the size is: no lane passes, a padding lane
// included, whether the check takes the scalar offset off the size, adds it or leaves it out.
struct StageLoad {
  uint32_t bytes, off, off1;
};
GLM52_HD StageLoad stage_load(int s, int nk, int krot, uint32_t step, uint32_t bytes) {
  const bool past = s >= nk;
  int k = s + krot;
  k = k >= nk ? k - nk : k;
  const uint32_t off = past ? 0u : (uint32_t)k * step;
  return {past ? 0u : bytes, off, past ? 0u : off + 64u};
}

}  // namespace glm52
