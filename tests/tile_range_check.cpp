// Checks the ring loads' offsets (fusion_amd/csrc/tile_range.h) under the three forms a raw
// buffer's range check can take: the lane's offset against the size less the scalar offset (in
// 32 bits), the sum of both against the size, and the lane's offset alone against the size.
// Prints each violation; the exit status is 1 if there was one.
#include "tile_range.h"

#include <cstdio>
#include <initializer_list>

using namespace glm52;

static int bad = 0;

static bool passes(int form, uint32_t lane, uint32_t scalar, uint32_t bytes) {
  if (form == 0) return lane < (uint32_t)(bytes - scalar);
  if (form == 1) return (uint64_t)lane + scalar < bytes;
  return lane < bytes;
}

static void check(const char* what, uint32_t lane, uint32_t scalar, uint32_t bytes, bool want, int nk,
                  int krot, int s) {
  for (int form = 0; form < 3; ++form)
    if (passes(form, lane, scalar, bytes) != want ||
        (want && !passes(form, lane + 15, scalar, bytes))) {
      ++bad;
      if (bad < 20)
        std::printf("%s: lane 0x%x scalar 0x%x bytes 0x%x form %d (nk %d, krot %d, stage %d)\n", what, lane,
                    scalar, bytes, form, nk, krot, s);
    }
}

// `lane`: the last lane offset of the operand's first stage; `pair`: two stages at a time
static void operand(const char* what, uint32_t bytes, uint32_t step, uint32_t lane, bool pair, int nk,
                    int krot) {
  for (int s = 0; s < nk + 16; s += pair ? 2 : 1) {
    const StageLoad l = stage_load(s, nk, krot, step, bytes);
    for (int h = 0; h < (pair ? 2 : 1); ++h) {
      const uint32_t so = h ? l.off1 : l.off;
      if (s < nk) {
        if (so != (uint32_t)((s + h + krot) % nk) * step) {
          ++bad;
          std::printf("%s: scalar 0x%x (nk %d, krot %d, stage %d + %d)\n", what, so, nk, krot, s, h);
        }
        check(what, 0, so, l.bytes, true, nk, krot, s);
        check(what, lane, so, l.bytes, true, nk, krot, s);
      } else {
        check(what, 0, so, l.bytes, false, nk, krot, s);
        check(what, lane, so, l.bytes, false, nk, krot, s);
      }
      if (bytes == kTokenBytes) check(what, kNowhere, so, l.bytes, false, nk, krot, s);
    }
  }
}

int main() {
  for (int nk : {2, 4, 6, 8, 34, 64, 130, 192, 512, 1024})
    for (int krot = 0; krot < nk; krot += 2) {
      // rows that end where the descriptor does; the last 16-byte chunk of their first stage
      operand("token rows", kTokenBytes, 64, kTokenBytes - nk * 64 + 48, true, nk, krot);
      operand("row-major W", kInPlaceBytes, 64, kInPlaceBytes - nk * 64 + 48, true, nk, krot);
      // a packed tile: 8 KB from a stage to the next, four groups of slots
      operand("packed W", (uint32_t)nk * 32768, 8192, (uint32_t)nk * 24576 + 8176, false, nk, krot);
    }
  return bad != 0;
}
