// The kernels' sampler (halton_value of gi_internal.h, over the tables of
// halton_tables) on the host, against the plain digit loop with one FP64
// division, for every dimension a depth-32 render uses.
//   bounds:  what halton_value rests on (chunk and quotient sizes, exactness
//            of A and B, the distance of B from multiples of 2^29)
//   edges:   indices around the chunks' boundaries and the ends of the range
//   random:  <pairs> random indices per dimension
// usage: sampler_check <seed> <pairs>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <set>
#include <vector>

#include "../../globillum_amd/csrc/gi_internal.h"

using namespace gi;

static float digit_loop(uint32_t n, uint32_t p, const uint16_t *perm) {
  uint64_t rev = 0, pk = 1;
  for (; n; n /= p) {
    rev = rev * p + perm[n % p];
    pk *= p;
  }
  const double A = (double)(rev * (p - 1) + perm[0]), B = (double)(pk * (p - 1));
  const float f = (float)(A / B);
  return f >= 1.0f ? 0x1.fffffep-1f : f;
}

int main(int argc, char **argv) {
  const uint32_t seed = argc > 1 ? (uint32_t)std::strtoul(argv[1], nullptr, 10) : 0u;
  const long pairs = argc > 2 ? std::atol(argv[2]) : 1000;
  const int32_t nd = dims_for_depth(kMaxDepth);
  std::vector<HaltonDim> dims;
  std::vector<uint16_t> perms;
  uint32_t entries = 0;
  halton_tables(seed, nd, dims, perms, entries);
  std::vector<uint16_t> chunks(entries);
  long bounds = 0, edges = 0, random = 0, checked = 0;
  const uint64_t all = (uint64_t)1 << 32;
  std::mt19937 rng(seed + 1);
  for (int32_t d = 0; d < nd; ++d) {
    const HaltonDim &h = dims[d];
    const uint64_t p = h.prime, P = h.P;
    uint64_t pm = 1, pt = 1;
    for (uint32_t i = 0; i < h.m; ++i) pm *= p;
    for (uint32_t i = 0; i < h.mt; ++i) pt *= p;
    const unsigned __int128 span = (unsigned __int128)P * P * (h.full == 3 ? P : 1) * h.Ptop;
    const uint64_t B = (uint64_t)span * (p - 1), r29 = B % ((uint64_t)1 << 29);
    const uint64_t far29 = r29 < ((uint64_t)1 << 28) ? r29 : ((uint64_t)1 << 29) - r29;
    const bool ok = pm == P && pt == h.Ptop && P <= 65536 && h.Ptop <= 65536 &&     // 16-bit entries
                    (h.full == 2 || h.full == 3) && span >= all &&                  // every index is covered
                    (all - 1) / P < (1u << 24) && P < (1u << 24) &&                 // factors of mul24
                    (h.full == 2 || (unsigned __int128)P * h.Ptop <= all) &&        // lo and
                    (unsigned __int128)P * P <= all &&                              // hi below 2^32
                    span * (p - 1) < ((unsigned __int128)1 << 53) &&                // A < B, exact in FP64
                    (double)B == h.B && h.rB == 1.0 / h.B && h.p1 == (double)(p - 1) &&
                    h.c_hi == (double)((uint64_t)(span / (P * P)) * (p - 1)) && h.perm0d == (double)perms[h.perm_off] &&
                    h.magic == ~0ull / P + 1 && (far29 > 8 || (B & (B - 1)) == 0) &&
                    h.off + P == h.top_off && (d + 1 == nd ? entries : dims[d + 1].off) == h.top_off + h.Ptop;
    if (!ok) ++bounds, std::printf("bounds: dimension %d\n", d);
    // the second quotient, at the ends of its range
    for (uint64_t q : {(uint64_t)0, P - 1, P, (all - 1) / P, ((all - 1) / P) / P * P, ((all - 1) / P) / P * P - 1})
      if (q <= (all - 1) / P && mul_hi((uint32_t)q, (uint32_t)(h.magic >> 32) + 1u) != q / P) ++bounds;
    for (uint32_t c = 0; c < P + h.Ptop; ++c) chunks[h.off + c] = halton_entry(h, perms.data(), c);
    const uint16_t *perm = perms.data() + h.perm_off;
    auto differs = [&](uint32_t n) {
      const float a = halton_value(n, h, chunks.data()), b = digit_loop(n, (uint32_t)p, perm);
      ++checked;
      return std::memcmp(&a, &b, 4) != 0;
    };
    std::set<uint64_t> at;
    for (uint64_t b : {(uint64_t)0, p, P, 2 * P, P * P, 2 * P * P, P * P * P, P * P * (all / (P * P)), all, all / 2})
      for (int64_t o : {-2, -1, 0, 1})
        if ((int64_t)b + o >= 0 && b + o < all) at.insert(b + o);
    for (uint64_t n : at)
      if (differs((uint32_t)n)) ++edges, std::printf("edge: dimension %d index %llu\n", d, (unsigned long long)n);
    for (long i = 0; i < pairs; ++i) random += differs((uint32_t)rng() >> (i & 1 ? rng() % 32 : 0));
  }
  std::printf("%ld values, bad: bounds %ld edges %ld random %ld\n", checked, bounds, edges, random);
  return bounds || edges || random;
}
