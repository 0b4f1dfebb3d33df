// small.h -- an LBVH over at most kSmallMax primitives, built by one workgroup.
//
// The staged build (lbvh.hip, batch.hip) is two dozen launches. On a few
// thousand primitives each of them leaves the chip idle and takes its 2 to 20
// us of launch, wait and cold caches: 37 scenes of 3,000 triangles took 220 us
// to build, and take 87 this way.  Here one workgroup holds a whole scene in LDS, does every
// stage with barriers between them and writes each result once, so a batch of
// such scenes is one launch of one workgroup per scene.  What bounds it is the
// length of that chain (4,096 triangles, us: box 7, codes 4, sort 20, leaves 13,
// hierarchy 21).
//
// The results are the staged build's bit for bit: the codes and the stable
// order are whole numbers, the tree is the one over the same unique codes, and
// boxes are unions, exact in any order.
#pragma once

#include <hip/hip_runtime.h>

#include "hrt_device.h"

namespace hrt {

// LDS holds nine words a primitive: 147,456 bytes of a CU's 163,840.
constexpr uint32_t kSmallMax = 4096;
// The box goes over every vertex, also unused ones: one workgroup reads this
// many in about 10 us, less than the staged build's launches take.
constexpr uint32_t kSmallVerts = 4 * kSmallMax;

// Where a build goes; what is null is not written.
struct SmallTree {
  NodePair* pairs;
  TriPre* tris;
  uint32_t* perm;         // sorted position -> primitive
  uint32_t* parent;       // per internal node but the root: parent << 1 | side
  uint32_t* parent_leaf;  // per leaf
  uint32_t* leaf_run;     // first sorted position per leaf
  uint2* range;           // leaf range per internal node
  uint32_t* leaves;       // one word
  uint32_t* max_run;      // one word
  float* box12;           // min xyzw, max xyzw, Morton scale xyzw
  // parity hooks
  uint32_t *codes_in, *codes_sorted, *ids_sorted, *run_start, *ucodes, *karras_lr;
  // nearest-hit nodes and their flag
  WideNode* wide;
  uint32_t* differ;
};

struct Child {
  float3 lo, hi;
  uint32_t ref;
};

__device__ inline Child pair_child(const NodePair* pairs, uint32_t k, uint32_t side) {
  const uint32_t* pw = reinterpret_cast<const uint32_t*>(pairs + k) + 8 * side;
  Child c;
  c.lo = make_float3(__uint_as_float(pw[0]), __uint_as_float(pw[1]), __uint_as_float(pw[2]));
  c.hi = make_float3(__uint_as_float(pw[4]), __uint_as_float(pw[5]), __uint_as_float(pw[6]));
  c.ref = pw[3];
  return c;
}

// The WideNode of internal node k (a one-leaf tree's pair 0 counts as one) into
// *out.  False when a child box is not the union of its own children's boxes,
// or one of those is inverted (a leaf of NaN vertices): the walk takes a
// child's distances from its children's.
__device__ inline bool make_wide_node(const NodePair* pairs, uint32_t k, WideNode* out) {
  Child g[4];
  uint32_t ref[2];
  bool exact = true;
  for (int side = 0; side < 2; side++) {
    const Child c = pair_child(pairs, k, side);
    Child &g0 = g[2 * side], &g1 = g[2 * side + 1];
    ref[side] = c.ref;
    if (c.ref & kLeafBit) {
      g0 = g1 = c;
      g1.ref = kInvalid;
      continue;
    }
    g0 = pair_child(pairs, c.ref, 0);
    g1 = pair_child(pairs, c.ref, 1);
    exact = exact && g0.lo.x <= g0.hi.x && g0.lo.y <= g0.hi.y && g0.lo.z <= g0.hi.z && g1.lo.x <= g1.hi.x &&
            g1.lo.y <= g1.hi.y && g1.lo.z <= g1.hi.z && c.lo.x == fminf(g0.lo.x, g1.lo.x) &&
            c.lo.y == fminf(g0.lo.y, g1.lo.y) && c.lo.z == fminf(g0.lo.z, g1.lo.z) &&
            c.hi.x == fmaxf(g0.hi.x, g1.hi.x) && c.hi.y == fmaxf(g0.hi.y, g1.hi.y) &&
            c.hi.z == fmaxf(g0.hi.z, g1.hi.z);
  }
  WideNode w;
  for (int i = 0; i < 4; i++) {
    w.g[2 * i] = make_float4(g[i].lo.x, g[i].lo.y, g[i].lo.z, __uint_as_float(g[i].ref));
    w.g[2 * i + 1] = make_float4(g[i].hi.x, g[i].hi.y, g[i].hi.z, __uint_as_float(ref[i >> 1]));
  }
  *out = w;
  return exact;
}

template <uint32_t kCap>
__device__ inline void put_box(float (&b)[6][kCap], uint32_t k, float3 lo, float3 hi) {
  b[0][k] = lo.x;
  b[1][k] = lo.y;
  b[2][k] = lo.z;
  b[3][k] = hi.x;
  b[4][k] = hi.y;
  b[5][k] = hi.z;
}
template <uint32_t kCap>
__device__ inline void get_box(const float (&b)[6][kCap], uint32_t k, float3& lo, float3& hi) {
  lo = make_float3(b[0][k], b[1][k], b[2][k]);
  hi = make_float3(b[3][k], b[4][k], b[5][k]);
}
__device__ inline float wave_min(float x) {
  for (int o = 32; o > 0; o >>= 1) x = fminf(x, __shfl_xor(x, o));
  return x;
}
__device__ inline float wave_max(float x) {
  for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o));
  return x;
}
__device__ inline uint32_t wave_exclusive_scan(uint32_t x, uint32_t lane) {
  uint32_t incl = x;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(incl, o);
    if (lane >= uint32_t(o)) incl += y;
  }
  return incl - x;
}

// The LDS of a workgroup of kThreads that builds over at most kThreads * kItems
// primitives.
template <uint32_t kThreads, uint32_t kItems>
struct SmallLds {
  static constexpr uint32_t kWaves = kThreads / 64, kCap = kThreads * kItems, kDigits = 256;
  uint32_t ucode[kCap];    // unique codes
  uint16_t run[kCap + 2];  // first sorted position of each, then the count
  union {
    uint16_t id[kCap];           // sorted primitives
    uint32_t nodes[kCap / 2];    // nodes that have yet to arrive at their split
  };
  union {
    struct {
      uint32_t key[kCap];
      uint32_t count[kDigits * kWaves];  // digit-major
    } sort;
    struct {
      float box[6][kCap];    // a node's or leaf's box, at its own number (see below)
      uint32_t word[kCap];   // per split: 0, or its first child's far leaf + 1 and side << 31
    } climb;
  };
  float4 box[2 * kWaves + 3];
  uint32_t sums[kWaves + 1];
  uint32_t flag, nnodes;
};

// Builds the tree over src's n primitives (n <= kThreads * kItems; all threads
// of the workgroup call it).
//
// The sort is four stable passes of 8 bits: a wave's items are consecutive, a
// lane's rank among the wave's equal digits comes from ballots, and the counts
// are scanned digit by digit, wave by wave.
//
// The hierarchy and its boxes grow from the leaves as in the batched build's
// leaf pass: node [l, r] is its parent's left child when l is the first leaf
// or its code at r differs less from the next than its code at l from the one
// before, and the second child to arrive at a split forms the parent.  A left
// child is node r, a right child node l, the root node 0.  A box waits at its
// node's own number: internal node m covers leaf m, whose box has been read by
// then.  While more nodes climb than there are threads, each takes one step
// and the formed ones are gathered: at most half as many as leaves after the
// first step, and no more after a later one (a node is formed by an arrival), so
// they fit `nodes`.  A thread that climbs with several leaves one after the
// other takes as many whole climbs (49 us instead of 33 on 4,096 triangles).
template <class Src, uint32_t kThreads, uint32_t kItems>
__device__ inline void small_build(const Src& src, uint32_t n, int cubic, const SmallTree& out,
                                   SmallLds<kThreads, kItems>& s) {
  using Lds = SmallLds<kThreads, kItems>;
  constexpr uint32_t kWaves = Lds::kWaves;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  // ---- scene box and Morton scale (k_box_final)
  {
    float4 lo = make_float4(kLbvhInf, kLbvhInf, kLbvhInf, kLbvhInf);
    float4 hi = make_float4(-kLbvhInf, -kLbvhInf, -kLbvhInf, -kLbvhInf);
    const uint32_t items = src.box_items();
    for (uint32_t i = tid; i < items; i += kThreads) {
      float4 a, b;
      src.box_item(i, a, b);
      lo = make_float4(fminf(lo.x, a.x), fminf(lo.y, a.y), fminf(lo.z, a.z), fminf(lo.w, a.w));
      hi = make_float4(fmaxf(hi.x, b.x), fmaxf(hi.y, b.y), fmaxf(hi.z, b.z), fmaxf(hi.w, b.w));
    }
    lo = make_float4(wave_min(lo.x), wave_min(lo.y), wave_min(lo.z), wave_min(lo.w));
    hi = make_float4(wave_max(hi.x), wave_max(hi.y), wave_max(hi.z), wave_max(hi.w));
    if (lane == 0) {
      s.box[wave] = lo;
      s.box[kWaves + wave] = hi;
    }
    __syncthreads();
    if (tid == 0) {
      for (uint32_t w = 1; w < kWaves; w++) {
        const float4 a = s.box[w], b = s.box[kWaves + w];
        lo = make_float4(fminf(lo.x, a.x), fminf(lo.y, a.y), fminf(lo.z, a.z), fminf(lo.w, a.w));
        hi = make_float4(fmaxf(hi.x, b.x), fmaxf(hi.y, b.y), fmaxf(hi.z, b.z), fmaxf(hi.w, b.w));
      }
      const float ex[4] = {(hi.x + kLbvhEpsBias) - (lo.x - kLbvhEpsBias), (hi.y + kLbvhEpsBias) - (lo.y - kLbvhEpsBias),
                           (hi.z + kLbvhEpsBias) - (lo.z - kLbvhEpsBias),
                           (hi.w + kLbvhEpsBias) - (lo.w - kLbvhEpsBias)};
      float z[4];
      if (cubic) {
        const float m = fmaxf(ex[0], fmaxf(ex[1], ex[2]));
        const float inv = (fabsf(m) < 1e-20f) ? 0.0f : 1.0f / m;
        z[0] = z[1] = z[2] = 1024.0f * inv;
        z[3] = 1024.0f * (1.0f / ex[3]);
      } else {
        for (int k = 0; k < 4; k++) {
          float inv = 1.0f / ex[k];
          if (k < 3 && fabsf(ex[k]) < 1e-20f) inv = 0.0f;
          z[k] = 1024.0f * inv;
        }
      }
      s.box[2 * kWaves] = lo;
      s.box[2 * kWaves + 1] = hi;
      s.box[2 * kWaves + 2] = make_float4(z[0], z[1], z[2], z[3]);
      s.flag = 0u;
      if (out.box12) {
        const float v[12] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w, z[0], z[1], z[2], z[3]};
        for (int k = 0; k < 12; k++) out.box12[k] = v[k];
      }
    }
    __syncthreads();
  }
  // ---- Morton codes (k_morton)
  uint32_t key[kItems], id[kItems];
  const uint32_t items = (n + kThreads - 1) / kThreads;  // a thread's share
  const uint32_t first = wave * 64 * items + lane;       // its item j is at first + 64 j
  {
    const float4 lo = s.box[2 * kWaves], z = s.box[2 * kWaves + 2];
#pragma unroll
    for (uint32_t j = 0; j < kItems; j++) {
      const uint32_t i = first + 64 * j;
      key[j] = 0u;
      id[j] = i;
      if (j >= items || i >= n) continue;
      const float3 c = src.centre(i, n);
      const int ix = int(z.x * (c.x - lo.x));
      const int iy = int(z.y * (c.y - lo.y));
      const int iz = int(z.z * (c.z - lo.z));
      key[j] = spread_bits(ix, 0) | spread_bits(iy, 1) | spread_bits(iz, 2);
      if (out.codes_in) out.codes_in[i] = key[j];
    }
  }
  // ---- sort
  for (uint32_t shift = 0; shift < 32; shift += 8) {
    for (uint32_t k = tid; k < Lds::kDigits * kWaves; k += kThreads) s.sort.count[k] = 0u;
    __syncthreads();
    uint32_t rank[kItems];
#pragma unroll
    for (uint32_t j = 0; j < kItems; j++) {
      rank[j] = 0u;
      if (j >= items) continue;
      const uint32_t d = (key[j] >> shift) & 255u;
      uint64_t same = __ballot(first + 64 * j < n);
      const bool valid = first + 64 * j < n;
#pragma unroll
      for (int bit = 0; bit < 8; bit++) {
        const bool b = (d >> bit) & 1u;
        const uint64_t m = __ballot(b);
        same &= b ? m : ~m;
      }
      uint32_t before = 0;
      const uint32_t below = lanes_below(same);
      if (valid && below == 0) before = atomicAdd(&s.sort.count[d * kWaves + wave], uint32_t(__popcll(same)));
      rank[j] = below + uint32_t(__shfl(before, valid ? __builtin_ctzll(same) : 0));
    }
    __syncthreads();
    {  // 4 counts a thread
      constexpr uint32_t kEach = Lds::kDigits / 64;
      uint32_t c[kEach], sum = 0;
#pragma unroll
      for (uint32_t k = 0; k < kEach; k++) {
        c[k] = s.sort.count[tid * kEach + k];
        sum += c[k];
      }
      uint32_t at = wave_exclusive_scan(sum, lane);
      if (lane == 63) s.sums[wave] = at + sum;
      __syncthreads();
      for (uint32_t w = 0; w < wave; w++) at += s.sums[w];
#pragma unroll
      for (uint32_t k = 0; k < kEach; k++) {
        s.sort.count[tid * kEach + k] = at;
        at += c[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kItems; j++) {
      if (j >= items || first + 64 * j >= n) continue;
      const uint32_t p = s.sort.count[((key[j] >> shift) & 255u) * kWaves + wave] + rank[j];
      s.sort.key[p] = key[j];
      s.id[p] = uint16_t(id[j]);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kItems; j++) {
      const uint32_t i = first + 64 * j;
      if (j >= items || i >= n) continue;
      key[j] = s.sort.key[i];
      id[j] = s.id[i];
    }
  }
  // ---- runs of one code
  uint32_t L;
  {
    bool head[kItems];
    uint32_t below[kItems], heads = 0;
#pragma unroll
    for (uint32_t j = 0; j < kItems; j++) {
      const uint32_t i = first + 64 * j;
      head[j] = j < items && i < n && (i == 0 || s.sort.key[i - 1] != key[j]);
      const uint64_t m = __ballot(head[j]);
      below[j] = heads + lanes_below(m);
      heads += uint32_t(__popcll(m));
      if (j < items && i < n) {
        if (out.perm) out.perm[i] = id[j];
        if (out.codes_sorted) out.codes_sorted[i] = key[j];
        if (out.ids_sorted) out.ids_sorted[i] = id[j];
      }
    }
    if (lane == 0) s.sums[wave] = heads;
    __syncthreads();
    uint32_t base = 0;
    L = 0;
    for (uint32_t w = 0; w < kWaves; w++) {
      if (w == wave) base = L;
      L += s.sums[w];
    }
#pragma unroll
    for (uint32_t j = 0; j < kItems; j++) {
      if (!head[j]) continue;
      const uint32_t m = base + below[j], i = first + 64 * j;
      s.ucode[m] = key[j];
      s.run[m] = uint16_t(i);
      if (out.leaf_run) out.leaf_run[m] = i;
      if (out.run_start) out.run_start[m] = i;
      if (out.ucodes) out.ucodes[m] = key[j];
    }
    if (tid == 0) s.run[L] = uint16_t(n);
    __syncthreads();  // the sort's arrays end here
  }
  // ---- boxes of the sorted primitives, and the triangles in leaf order
  for (uint32_t k = tid; k < L; k += kThreads) s.climb.word[k] = 0u;
  if (tid == 0) s.nnodes = 0u;
  {
    float3 lo[kItems], hi[kItems];
    uint32_t longest = 0;
    if constexpr (Src::kTris) {
      float4 va[kItems], vb[kItems], vc[kItems];
#pragma unroll
      for (uint32_t k = 0; k < kItems; k++) {
        const uint32_t j = tid + k * kThreads;
        src.corners(j < n ? s.id[j] : 0u, va[k], vb[k], vc[k]);
      }
#pragma unroll
      for (uint32_t k = 0; k < kItems; k++) {
        const uint32_t j = tid + k * kThreads;
        const float4 a = va[k], b = vb[k], c = vc[k];
        lo[k] = make_float3(fminf(a.x, fminf(b.x, c.x)), fminf(a.y, fminf(b.y, c.y)), fminf(a.z, fminf(b.z, c.z)));
        hi[k] = make_float3(fmaxf(a.x, fmaxf(b.x, c.x)), fmaxf(a.y, fmaxf(b.y, c.y)), fmaxf(a.z, fmaxf(b.z, c.z)));
        if (j >= n) continue;
        TriPre r;
        r.a = make_float4(a.x, a.y, a.z, __uint_as_float(uint32_t(s.id[j])));
        r.e1 = make_float4(b.x - a.x, b.y - a.y, b.z - a.z, 0.0f);
        r.e2 = make_float4(c.x - a.x, c.y - a.y, c.z - a.z, 0.0f);
        out.tris[j] = r;
      }
    } else {
#pragma unroll
      for (uint32_t k = 0; k < kItems; k++) {
        const uint32_t j = tid + k * kThreads;
        src.prim_box(j < n ? s.id[j] : 0u, lo[k], hi[k]);
      }
    }
#pragma unroll
    for (uint32_t k = 0; k < kItems; k++) {
      const uint32_t j = tid + k * kThreads;
      if (j < n) put_box(s.climb.box, j, lo[k], hi[k]);
    }
    __syncthreads();
    // a leaf's box: the union over its run (k_leaves)
#pragma unroll
    for (uint32_t k = 0; k < kItems; k++) {
      const uint32_t m = tid + k * kThreads;
      if (m >= L) continue;
      const uint32_t st = s.run[m], e = s.run[m + 1];
      longest = max(longest, e - st);
      lo[k] = make_float3(kLbvhInf, kLbvhInf, kLbvhInf);
      hi[k] = make_float3(-kLbvhInf, -kLbvhInf, -kLbvhInf);
      for (uint32_t j = st; j < e; j++) {
        float3 a, b;
        get_box(s.climb.box, j, a, b);
        lo[k] = make_float3(fminf(lo[k].x, a.x), fminf(lo[k].y, a.y), fminf(lo[k].z, a.z));
        hi[k] = make_float3(fmaxf(hi[k].x, b.x), fmaxf(hi[k].y, b.y), fmaxf(hi[k].z, b.z));
      }
    }
    for (int o = 32; o > 0; o >>= 1) longest = max(longest, uint32_t(__shfl_xor(longest, o)));
    if (lane == 0) s.sums[wave] = longest;
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < kItems; k++) {
      const uint32_t m = tid + k * kThreads;
      if (m < L) put_box(s.climb.box, m, lo[k], hi[k]);
    }
    if (tid == 0) {
      for (uint32_t w = 1; w < kWaves; w++) longest = max(longest, s.sums[w]);
      if (out.max_run) *out.max_run = longest;
      if (out.leaves) *out.leaves = L;
    }
    if (L == 1 && tid == 0) {
      // the root is a leaf: pair 0 = (root leaf, empty dummy), as in k_leaves
      store_box(out.pairs, 0, 0, lo[0], hi[0]);
      store_box(out.pairs, 0, 1, make_float3(0.f, 0.f, 0.f), make_float3(0.f, 0.f, 0.f));
      uint32_t* pw = reinterpret_cast<uint32_t*>(out.pairs);
      pw[3] = pack_leaf(0, n);
      pw[7] = 0u;
      pw[11] = 0x80000000u;
      pw[15] = 0u;
    }
    __syncthreads();
  }
  // ---- hierarchy and boxes
  // Node [l, r] (of a tree of several leaves, not the root) arrives at its
  // split.  The second child forms the parent: true with [l, r] = the parent,
  // its box in lo, hi and at its number, unless that is the root.
  auto arrive = [&](uint32_t& l, uint32_t& r, bool& left, float3& lo, float3& hi) {
    const uint32_t sib = left ? r + 1 : l - 1, g = left ? r : l - 1;
    const uint32_t old = __hip_atomic_exchange(&s.climb.word[g], left ? l + 1 : (r + 1) | 0x80000000u,
                                               __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (old == 0u) return false;
    const uint32_t far = (old & 0x7FFFFFFFu) - 1u;
    if (left) r = far;
    else l = far;
    const bool leaf0 = l == g, leaf1 = r == g + 1, root = l == 0 && r + 1 == L;
    const uint32_t r0 = s.run[g], r1 = s.run[g + 1], r2 = s.run[g + 2];
    float3 slo, shi;
    get_box(s.climb.box, sib, slo, shi);
    const bool up = root || l == 0 || (r + 1 != L && (s.ucode[r] ^ s.ucode[r + 1]) < (s.ucode[l - 1] ^ s.ucode[l]));
    const uint32_t k = root ? 0u : up ? r : l;
    const float3 lo0 = left ? lo : slo, hi0 = left ? hi : shi, lo1 = left ? slo : lo, hi1 = left ? shi : hi;
    const uint32_t c0 = leaf0 ? pack_leaf(r0, r1 - r0) : g, c1 = leaf1 ? pack_leaf(r1, r2 - r1) : g + 1;
    float4* pw = reinterpret_cast<float4*>(out.pairs + k);
    pw[0] = make_float4(lo0.x, lo0.y, lo0.z, __uint_as_float(c0));
    pw[1] = make_float4(hi0.x, hi0.y, hi0.z, 0.0f);
    pw[2] = make_float4(lo1.x, lo1.y, lo1.z, __uint_as_float(c1));
    pw[3] = make_float4(hi1.x, hi1.y, hi1.z, 0.0f);
    if (out.parent) {
      (leaf0 ? out.parent_leaf : out.parent)[g] = k << 1;
      (leaf1 ? out.parent_leaf : out.parent)[g + 1] = (k << 1) | 1u;
      out.range[k] = make_uint2(l, r);
    }
    if (out.karras_lr) {
      out.karras_lr[2 * k] = leaf0 ? L - 1 + g : g;
      out.karras_lr[2 * k + 1] = leaf1 ? L - 1 + g + 1 : g + 1;
    }
    if (root) return false;
    lo = make_float3(fminf(lo0.x, lo1.x), fminf(lo0.y, lo1.y), fminf(lo0.z, lo1.z));
    hi = make_float3(fmaxf(hi0.x, hi1.x), fmaxf(hi0.y, hi1.y), fmaxf(hi0.z, hi1.z));
    put_box(s.climb.box, k, lo, hi);
    left = up;
    return true;
  };
  if (L > 1) {
    uint32_t live = L;  // nodes that climb: the leaves first, then those in s.nodes (l, r << 12, left << 24)
    bool leaves = true;
    while (live > kThreads) {
      uint32_t formed[kItems];
#pragma unroll
      for (uint32_t k = 0; k < kItems; k++) {
        const uint32_t m = tid + k * kThreads;
        formed[k] = kInvalid;
        if (m < live) formed[k] = leaves ? m | m << 12 : s.nodes[m];
      }
      __syncthreads();
#pragma unroll
      for (uint32_t k = 0; k < kItems; k++) {
        uint32_t l = formed[k] & 4095u, r = (formed[k] >> 12) & 4095u;
        bool more = formed[k] != kInvalid;
        if (more) {
          bool left = leaves ? (l == 0 || (l + 1 != L && (s.ucode[l] ^ s.ucode[l + 1]) < (s.ucode[l - 1] ^ s.ucode[l])))
                             : (formed[k] >> 24) != 0u;
          float3 lo, hi;
          get_box(s.climb.box, left ? r : l, lo, hi);
          more = arrive(l, r, left, lo, hi);
          formed[k] = l | r << 12 | uint32_t(left) << 24;
        }
        const uint64_t m = __ballot(more);
        uint32_t at = 0;
        if (lane == 0 && m != 0) at = atomicAdd(&s.nnodes, uint32_t(__popcll(m)));
        at = __shfl(at, 0) + lanes_below(m);
        if (more) s.nodes[at] = formed[k];
      }
      __syncthreads();
      live = s.nnodes;
      leaves = false;
      __syncthreads();
      if (tid == 0) s.nnodes = 0u;
    }
    if (tid < live) {
      uint32_t l = tid, r = tid;
      bool left;
      if (leaves) {
        left = l == 0 || (l + 1 != L && (s.ucode[l] ^ s.ucode[l + 1]) < (s.ucode[l - 1] ^ s.ucode[l]));
      } else {
        const uint32_t v = s.nodes[tid];
        l = v & 4095u;
        r = (v >> 12) & 4095u;
        left = (v >> 24) != 0u;
      }
      float3 lo, hi;
      get_box(s.climb.box, left ? r : l, lo, hi);
      while (arrive(l, r, left, lo, hi)) {
      }
    }
  }
  if (out.wide) {
    __syncthreads();
    const uint32_t nodes = L > 1 ? L - 1 : 1;
    bool exact = true;
    for (uint32_t k = tid; k < nodes; k += kThreads) exact = make_wide_node(out.pairs, k, out.wide + k) && exact;
    if (!exact) s.flag = 1u;
    __syncthreads();
    if (tid == 0) *out.differ = s.flag;
  }
}

}  // namespace hrt
