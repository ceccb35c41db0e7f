// The order in which consumers meet a queue's segments (gi_internal.h).
//   cover: every (segment, row) is met exactly once, in order of rows
//   even:  a consumer whose stride is a multiple of 16 meets each segment once
//          in four steps, from any of its places
#include <cstdio>
#include <vector>

#include "../../globillum_amd/csrc/gi_internal.h"

using namespace gi;

int main() {
  int bad = 0;
  for (uint32_t stride : {1u, 3u, 16u, 17u, 256u, 1000u, 4096u, 6144u, 8192u, 16384u}) {
    const uint32_t turn = queue_turn(stride), rows = 8192;
    std::vector<int> met(kShards * rows, 0);
    for (uint32_t j = 0; j < kShards * rows; ++j) {
      const uint32_t row = (j >> (2 * kShardShift)) << kShardShift | (j & (kShards - 1));
      ++met[queue_segment(j, turn) * rows + row];
    }
    for (int m : met) bad += m != 1;
  }
  std::printf("cover %d bad\n", bad);
  int uneven = 0;
  for (uint32_t stride = 16; stride <= 24576; stride += 16) {
    const uint32_t turn = queue_turn(stride);
    for (uint32_t w = 0; w < stride; w += 1 + stride / 37) {
      int n[kShards] = {};
      for (uint32_t i = 0; i < 64; ++i) ++n[queue_segment(w + i * stride, turn)];
      for (int c : n)
        if (c != 16) {
          if (++uneven < 10) std::printf("stride %u from %u: %d %d %d %d\n", stride, w, n[0], n[1], n[2], n[3]);
          break;
        }
    }
  }
  std::printf("even %d bad\n", uneven);
  return bad || uneven;
}
