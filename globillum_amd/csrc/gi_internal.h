// Internal declarations shared by the host sources of libgi_hip.so.
#pragma once

#include <cstdint>
#include <functional>
#include <string>
#include <vector>

#include "../../include/gi_hip.h"

namespace gi {

// ---------------------------------------------------------------- BVH ----
// Binary BVH node of the host builder.  Leaves hold [first, first+count) of
// the builder's triangle permutation.
struct Bvh2Node {
  float lo[3], hi[3];
  int32_t left, right;   // children (inner), -1 for leaves
  int32_t first, count;  // leaf range, count == 0 for inner nodes
};

// 4-wide node streamed by the traversal kernels: the six child-box planes
// as float4 (one lane per child) plus the child references -- 112 bytes,
// padded to one 128-byte cache line.
//   ref >= 0                 : inner node index
//   ref & 0x80000000         : leaf, bits 27..30 = triangle count (1..15),
//                              bits 0..26 = first triangle (leaf order)
//   ref == kEmptyRef         : empty slot
struct alignas(128) WideNode {
  float lox[4], hix[4], loy[4], hiy[4], loz[4], hiz[4];
  uint32_t child[4];
  uint32_t pad[4];
};
static_assert(sizeof(WideNode) == 128, "wide node must be one cache line");

// The traversal's copy of a WideNode, with the child planes in half
// precision: five 16-byte loads per visit instead of seven.
//   org, scale: the node box's min corner (f32) and a power of two s;
//   q[axis]: the four children's lo and hi planes on that axis as f16
//     offsets from org in units of s, packed lo0|lo1, lo2|lo3, hi0|hi1,
//     hi2|hi3 (low half first), rounded outward past a margin; empty slots
//     +inf (their box stays [+inf, +inf]);
//   child: the WideNode's child references.
// 80 bytes used of one 128-byte line, so nodes keep the WideNode indexing.
struct alignas(128) HalfNode {
  float org[3], scale;
  uint32_t q[3][4];
  uint32_t child[4];
  uint32_t pad[12];
};
static_assert(sizeof(HalfNode) == sizeof(WideNode), "half node keeps the wide node's stride");
constexpr uint32_t kLeafBit = 0x80000000u;
constexpr uint32_t kEmptyRef = 0x80000000u;  // a leaf with zero triangles
constexpr int kMaxLeafTris = 15;
constexpr uint32_t kMaxLeafFirst = (1u << 27) - 1;

#if defined(__HIP__)
#define GI_HOST_DEVICE __host__ __device__
#else
#define GI_HOST_DEVICE
#endif

// The slab tests' relative slack, and their limit: the nearer of the ray's
// limit and the largest float whose product with the slack is finite.  That
// product is FLT_MAX, so a ray without a limit reaches every box at a finite
// distance and no box at +inf.  A limit of NaN counts as none.
constexpr float kSlabSlack = 1.0f + 0x1p-21f;
constexpr float kMaxLim = 0x1.ffffeep127f;
static_assert(kMaxLim * kSlabSlack == 0x1.fffffep127f, "the largest limit stays finite, at FLT_MAX");
GI_HOST_DEVICE inline float slab_limit(float lim) { return lim < kMaxLim ? lim : kMaxLim; }
// A box entered at tn (at least 0) and left at tf (at most the limit).
GI_HOST_DEVICE inline bool slab_hit(float tn, float tf) { return tn <= tf * kSlabSlack; }

// An empty child slot: its box is [+inf, +inf] on every axis, so the slab
// test never reports it (each plane distance is +inf or -inf for any finite
// nonzero inverse direction: entered at +inf, or left at -inf, both beyond
// slab_limit) and the traversal needs no reference check.
GI_HOST_DEVICE inline void set_empty_slot(WideNode &nd, int k) {
  nd.lox[k] = nd.loy[k] = nd.loz[k] = __builtin_inff();
  nd.hix[k] = nd.hiy[k] = nd.hiz[k] = __builtin_inff();
  nd.child[k] = kEmptyRef;
}

// Triangle in leaf order for intersection: vertex a (w = original id as
// bits), edges b-a and c-a.  48 bytes.
struct alignas(16) IsectTri {
  float a[4];
  float e1[4];
  float e2[4];
};
static_assert(sizeof(IsectTri) == 48, "isect tri layout");

}  // namespace gi

struct gi_bvh {
  std::vector<gi::Bvh2Node> nodes;  // binary tree, root = 0
  std::vector<uint32_t> perm;       // leaf-order triangle ids
  int32_t max_depth = 0;
};

namespace gi {

// Binned-SAH build over the triangle list (host).  Boxes are padded by a
// relative 2^-20 so the float slab tests stay conservative.
// threads == 1 builds on the calling thread only; otherwise subtrees of at
// least 2^16 primitives near the root build on other threads.  Both give
// the same nodes in the same order.
void build_bvh2(const gi_tri *tris, int64_t n, int32_t max_leaf, gi_bvh &out, int32_t threads = 0);
// The same build from the triangles' boxes: corner by corner, lo[k] =
// min(lo[k], corner) from FLT_MAX and hi[k] = max(hi[k], corner) from
// -FLT_MAX.
struct TriBox {
  float lo[3], hi[3];
};
void build_bvh2(const TriBox *boxes, int64_t n, int32_t max_leaf, gi_bvh &out, int32_t threads = 0);
// Import a binary BVH in the reference's 2 x float4 layout.
bool import_bvh2(const float *nodes, int64_t n_nodes, const uint32_t *indices, int64_t n_indices,
                 int64_t n_tris, gi_bvh &out, std::string &err);
// Collapse to the 4-wide layout (surface-area cost, dynamic program over
// slot counts) and emit the leaf-ordered intersection triangles.
void collapse_wide(const gi_bvh &b, const gi_tri *tris, std::vector<WideNode> &nodes,
                   std::vector<IsectTri> &leaf_tris, int32_t &wide_depth, int32_t width = 4);
// The pieces of collapse_wide: leaf-ordered triangles (a.w = index in tris),
// and the 4-wide nodes with interior references offset by node_base and
// leaf references from leaf_ref (called for leaves with count > 0).  The
// collapse may turn a binary subtree of at most merge_limit primitives (a
// contiguous range) into one leaf; 1 keeps the binary leaves as they are.
// width (2..4) is the number of child slots it fills per wide node.
#ifndef GI_COLLAPSE_MERGE
#define GI_COLLAPSE_MERGE 4
#endif
constexpr int32_t kCollapseMergeLimit = GI_COLLAPSE_MERGE;
// Cost of a wide-node visit (four box tests, one 128-byte fetch) in
// triangle tests, for the collapse's surface-area cost.
#ifndef GI_COLLAPSE_NODE_COST
#define GI_COLLAPSE_NODE_COST 1.0
#endif
constexpr double kCollapseNodeCost = GI_COLLAPSE_NODE_COST;
// Binned SAH (host builder and its device counterpart): centroid bins per
// axis, and the depth from which nodes split at the object median.
constexpr int kSahBins = 32;
constexpr int kSahMaxDepth = 48;
void leaf_order_tris(const gi_bvh &b, const gi_tri *tris, std::vector<IsectTri> &leaf_tris);
void collapse_wide_nodes(const gi_bvh &b, const std::function<uint32_t(const Bvh2Node &)> &leaf_ref,
                         uint32_t node_base, std::vector<WideNode> &nodes, int32_t &wide_depth,
                         int32_t merge_limit, int32_t width = 4);
// Relative box padding of the builders (2^-20 of the largest coordinate
// magnitude / extent): keeps the float slab tests conservative.
void pad_box(float *lo, float *hi);
// Binned-SAH build over boxes (lo xyz, hi xyz per primitive), split down to
// max_leaf primitives per leaf.
void build_bvh2_boxes(const float *boxes, int64_t n, int32_t max_leaf, gi_bvh &out, int32_t threads = 0);

// Special references (count 0): an empty slot, the end of a traversal, the
// return from an instance to world space, and instance i (kLeafBit | i + 1).
constexpr uint32_t kDoneRef = kLeafBit | kMaxLeafFirst;
constexpr uint32_t kReturnRef = kLeafBit | (kMaxLeafFirst - 1);
constexpr uint32_t kMaxInstances = kMaxLeafFirst - 2;

// --------------------------------------------------------- ray queues ----
// Consumers take spans or tiles j, j + stride, j + 2 stride, ... of a queue
// of kShards segments: kShards consecutive ones of a segment, then as many of
// the next (16 j's: kShards rows of every segment).  In the next 16 the
// segments come in the same order, turned by one each time j passes a
// multiple of 2^turn (any turn of at least 4 keeps the order complete: 16 j's
// turn together).  With 2^turn the largest power of two that divides the
// stride, a multiple of 16 for any full grid, a consumer's step turns by an
// odd number: it meets the segments in turn, equally often.
constexpr uint32_t kShardShift = 2, kShards = 1u << kShardShift;
GI_HOST_DEVICE inline uint32_t queue_turn(uint32_t stride) {
  const uint32_t t = (uint32_t)__builtin_ctz(stride);
  return t > 2u * kShardShift ? t : 2u * kShardShift;
}
GI_HOST_DEVICE inline uint32_t queue_segment(uint32_t j, uint32_t turn) {
  return ((j >> kShardShift) + (j >> turn)) & (kShards - 1u);
}

// ------------------------------------------------------------- Halton ----
// Per-dimension constants of the scrambled radical inverse, laid out for
// the device.  An index n < 2^32 is split, lowest digits first, into `full`
// chunks of m digits (P = p^m, the largest <= 65536) and a top chunk of mt
// digits (Ptop = p^mt): P^full * Ptop >= 2^32.  Entry c of a chunk table is
// the scrambled reversed value sum_i perm[digit_i(c)] p^(m-1-i) of the m
// digits of c: below P, so 16 bits hold it.
struct HaltonDim {
  uint32_t prime;       // p
  uint32_t off;         // the table of the full chunks in the uint16 pool
  uint32_t top_off;     // the table of the top chunk
  uint32_t perm_off;    // perm in the pool of digit permutations
  uint32_t P, Ptop;
  uint32_t full;        // full chunks: 2 or 3
  uint32_t m, mt;       // digits of a full chunk and of the top chunk
  uint32_t perm0;       // perm[0]
  uint64_t magic;       // floor(2^64 / P) + 1
  // A = hi * c_hi + lo * (p - 1) + perm[0], B = P^full Ptop (p - 1), 1 / B:
  // integers below 2^53 (but for the last)
  double c_hi, p1, perm0d, B, rB;
};
static_assert(sizeof(HaltonDim) == 88, "halton dim layout");

// Chunk table entry c of dimension hd (the top chunk's table: c - P of the
// entries past the full chunks').
GI_HOST_DEVICE inline uint16_t halton_entry(const HaltonDim &hd, const uint16_t *perms, uint32_t c) {
  const bool top = c >= hd.P;
  uint32_t x = top ? c - hd.P : c, v = 0;
  const uint32_t m = top ? hd.mt : hd.m;
  for (uint32_t i = 0; i < m; ++i) {  // least significant digit first
    const uint32_t q = x / hd.prime;
    v = v * hd.prime + perms[hd.perm_off + (x - q * hd.prime)];
    x = q;
  }
  return (uint16_t)v;
}
// The product of two numbers below 2^24 (the hardware's full-rate one, which
// drops higher bits).
GI_HOST_DEVICE inline uint32_t mul24(uint32_t a, uint32_t b) { return (a & 0xffffffu) * (b & 0xffffffu); }
GI_HOST_DEVICE inline uint32_t mul_hi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }

// Scrambled radical inverse of n in the prime base p of a dimension: the
// digits d_k (K of them) map to perm[d_k] and the infinitely many leading
// zeros to perm[0], which is the exact rational
//   A / B,  A = rev*(p-1) + perm[0],  B = p^K (p-1),  rev = sum perm[d_k] p^(K-1-k).
// Leading zero digits may be counted as digits: each adds perm[0] to rev and
// a factor p to p^K, which multiplies A and B by p and leaves A / B as it
// is.  So every n < 2^32 is split into the same chunks of its dimension
// (HaltonDim), and A, B < 2^53 are exact in FP64.
//
// The value is RN32(RN64(A / B)), the FP64 division and one rounding, from
// rB = RN(1/B), q = RN(A rB) and one fused residual and correction
// (Markstein, IBM J. Res. Dev. 34(1), 1990): three instructions in place of
// the division's twenty.  q may be 1.5 ulp off, so RN64(A / B) itself is not
// assured; the FP32 value is.  With every rounding at most 2^-53, what is
// rounded last is x (1 + d), x = A / B, |d| <= 2^-104 (to first order).  The
// two roundings give another FP32 value than from x only if a half-way point
// of FP64 beside one of FP32, (j + 2^-29) / 2^(25+e) or (j - 2^-29) / 2^(25+e)
// with j odd and 2^-e-1 < x < 2^-e, lies that near x: then B 2^-29 is within
// 2^-26 of the integer |A 2^(25+e) - j B|, that is, B within 8 of a multiple
// of 2^29.  No dimension's is (the nearest is 1.8 million away), but for
// p = 2, whose B is a power of two and every step exact.
//
// The quarter-rate integer products are the two of n / P (the top 32 bits
// of the 96-bit n * magic; exact as the 64-bit mulhi) and one of the second
// quotient: for q < 2^32 / P, floor(q / P) = mul_hi(q, floor(2^32 / P) + 1),
// since q times the multiplier's excess (<= P / 2^32) stays below 1 / P.
// tests/csrc/sampler_check.cpp holds all these bounds for every dimension.
template <class Dim> GI_HOST_DEVICE inline float halton_value(uint32_t n, Dim &hd, const uint16_t *chunks) {
  const uint16_t *tab = chunks + hd.off, *top = chunks + hd.top_off;
  const uint32_t P = hd.P, mlo = (uint32_t)hd.magic, mhi = (uint32_t)(hd.magic >> 32);
  // (n * mhi + hi32(n * mlo)) >> 32 = hi64(n * magic): the low word of
  // n * mlo cannot carry into the top 32 bits of the 96-bit product
  const uint32_t q0 = (uint32_t)(((uint64_t)n * mhi + mul_hi(n, mlo)) >> 32);
  const uint32_t mq = mhi + 1u;  // floor(2^32 / P) + 1
  const uint32_t q1 = mul_hi(q0, mq);
  const uint32_t v0 = tab[n - mul24(q0, P)], v1 = tab[q0 - mul24(q1, P)];
  uint32_t lo;
  if (hd.full == 2) {  // uniform: one dimension per sample call
    lo = top[q1];
  } else {
    const uint32_t q2 = mul_hi(q1, mq);
    lo = mul24(tab[q1 - mul24(q2, P)], hd.Ptop) + top[q2];
  }
  const uint32_t hi = mul24(v0, P) + v1;
  const double A = __builtin_fma((double)hi, hd.c_hi, __builtin_fma((double)lo, hd.p1, hd.perm0d));
  const double q = A * hd.rB;
  const float f = (float)__builtin_fma(__builtin_fma(-q, hd.B, A), hd.rB, q);
  return f >= 1.0f ? 0x1.fffffep-1f : f;
}

int32_t prime_of(int32_t dim);
void halton_permutation(int32_t dim, uint32_t seed, uint16_t *perm);
// The dimensions' constants, the digit permutations they index and the
// number of chunk table entries (which halton_fill of gi_device.h computes
// on the device, one after another).
void halton_tables(uint32_t seed, int32_t ndims, std::vector<HaltonDim> &dims, std::vector<uint16_t> &perms,
                   uint32_t &entries);
float halton_host(uint64_t n, int32_t dim, uint32_t seed);

// Sample dimension map: jitter x/y, lens x/y, then per path vertex b:
// NEE x, y, light choice; BSDF x, y, lobe; Russian roulette.
constexpr int kDimJitterX = 0, kDimJitterY = 1, kDimLensX = 2, kDimLensY = 3;
constexpr int kDimVertex0 = 4, kDimsPerVertex = 7;
constexpr int kMaxDepth = 32;
inline int dims_for_depth(int depth) { return kDimVertex0 + kDimsPerVertex * depth; }

}  // namespace gi
