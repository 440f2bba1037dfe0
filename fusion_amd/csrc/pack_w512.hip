// The writer of the packed weight layout, which the grouped GEMM tiles (moe_gemm_tile.h) and
// the decode kernels read, and the tiles' debugging hooks.
#include "moe_gemm.h"

#include <atomic>

using namespace glm52;

namespace {

// The host side of glm52_debug_item_trace: the record the next launches write, or null.
std::atomic<unsigned long long*> g_item_trace{nullptr};

// The host side of glm52_debug_item_set.
thread_local int t_item_set = -1;

// One 16-byte chunk of the packed layout per thread and step: chunk d is lane d % 64 of
// stage (d / 64) % nk of load slot (d / (64 nk)) % 32 of tile d / (2048 nk), written at
// packed_slot_off(nk, slot) + stage * kPackStride (+ 16 lane bytes) of its tile.
template <bool GATED>
__global__ __launch_bounds__(256) void pack_w512_kernel(const uint16_t* __restrict__ w,
                                                        int64_t swe, int64_t swn, int64_t swk,
                                                        int gu_off, int num_n, int nk,
                                                        int64_t chunks,
                                                        uint16_t* __restrict__ out) {
  constexpr int NO = GATED ? 256 : 512;
  for (int64_t d = (int64_t)blockIdx.x * 256 + threadIdx.x; d < chunks;
       d += (int64_t)gridDim.x * 256) {
    const int l = (int)(d % 64);
    const int64_t q = d / 64;
    const int kt = (int)(q % nk);
    const int64_t rest = q / nk;  // tile * 32 + slot
    const int slot = (int)(rest % 32);
    const int64_t tile = rest / 32;
    uint16_t* dst = out + tile * packed_tile_elems(nk) + packed_slot_off(nk, slot) +
                    (int64_t)kt * kPackStride + l * 8;
    const int pid_n = (int)(tile % num_n);
    const int64_t e = tile / num_n;
    const int row = pid_n * NO + w512_row(GATED, gu_off, slot / 8, slot % 8, l);
    const int64_t k0 = (int64_t)kt * 32 + w512_chunk(l) * 8;
    const uint16_t* src = w + e * swe + (int64_t)row * swn + k0 * swk;
    if (swk == 1) {
      *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
    } else {  // k strided (a [K, N] operand packed as its transpose): gather 8 values
      uint16_t v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = src[q * swk];
      uint4 o;
      o.x = (uint32_t)v[0] | ((uint32_t)v[1] << 16);
      o.y = (uint32_t)v[2] | ((uint32_t)v[3] << 16);
      o.z = (uint32_t)v[4] | ((uint32_t)v[5] << 16);
      o.w = (uint32_t)v[6] | ((uint32_t)v[7] << 16);
      *reinterpret_cast<uint4*>(dst) = o;
    }
  }
}

}  // namespace

namespace glm52 {
unsigned long long* item_trace() { return g_item_trace.load(std::memory_order_relaxed); }
int note_item_set(int set) { return t_item_set = set; }
}  // namespace glm52

extern "C" int glm52_debug_item_trace(void* buf, int64_t bytes) {
  if (buf && bytes < 256 * 4 * (int64_t)sizeof(unsigned long long)) return GLM52_EINVAL;
  g_item_trace.store(static_cast<unsigned long long*>(buf), std::memory_order_relaxed);
  return GLM52_OK;
}

extern "C" int glm52_debug_item_set(void) { return t_item_set; }

namespace glm52 {
int64_t pack_w512(const uint16_t* w, int64_t swe, int64_t swn, int E, int n_out, int k,
                     int gate_up_offset, bool gated, uint16_t* out, hipStream_t st,
                     int64_t swk) {
  const int NO = gated ? 256 : 512;
  if (E <= 0 || n_out <= 0 || (n_out % NO) || k <= 0 || (k % 64)) return GLM52_EUNSUPPORTED;
  const int num_n = n_out / NO, nk = k / 32;
  const int64_t chunks = (int64_t)E * num_n * nk * 2048;  // 16-byte chunks written
  const int64_t bytes = (int64_t)E * num_n * packed_tile_elems(nk) * 2;
  if (!out) return bytes;
  const int64_t blocks = (chunks + 255) / 256;
  const int grid = (int)(blocks < 65536 ? blocks : 65536);
  if (gated)
    pack_w512_kernel<true><<<grid, 256, 0, st>>>(w, swe, swn, swk, gate_up_offset, num_n, nk, chunks, out);
  else
    pack_w512_kernel<false><<<grid, 256, 0, st>>>(w, swe, swn, swk, 0, num_n, nk, chunks, out);
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? bytes : -(int64_t)err;
}
}  // namespace glm52
