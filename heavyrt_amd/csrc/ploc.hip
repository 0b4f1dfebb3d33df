// ploc.hip -- the agglomerative hierarchy of the any-hit tree.
//
// An any-hit answer (is there a triangle in (tNear, tFar)?) does not depend on
// the tree, so the tree that any-hit rays walk is this build's own choice
// (no reference counterpart).  Traversal time follows node visits, and a
// Morton split hierarchy is a poor one: this rebuilds the hierarchy above the
// LBVH leaves by parallel locally-ordered clustering (PLOC, Meister & Bittner
// 2018).  The leaves, their order and the leaf-order triangles stay those of
// the LBVH; only the internal nodes change.
//
// Rule (the oracle restates it, and the nodes match it one for one):
//   clusters = the leaves in Morton order;
//   repeat until one cluster is left:
//     each cluster i picks the j != i within [i - R, i + R] minimising the
//     union box's half area (ex*ey + ey*ez + ez*ex, NaN as +inf), ties to
//     the smaller j;
//     every mutual pair i < j becomes internal node (next_id - rank of i
//     among this round's merges), left = i, right = j, at position i; j is
//     dropped; survivors keep their order.
// The pick is a strict order on pairs, so the best pair of a round is always
// mutual and every round merges; ids count down from L - 2, so the root is 0.
//
// No round needs the host: its cluster count, next id and buffer are in a
// device-side record that the round before wrote.  Above kFinish clusters a
// round is two launches (pick and merge); from there on one workgroup does all
// remaining rounds with the clusters in LDS.  The host enqueues as many rounds
// as a tree of this size usually needs and looks at the result once.  The
// 564,235 leaves of 1.07 M triangles of hills with boxes (59 rounds) took 1.7 ms
// of kernels, about 480 launches and 59 waits of the host with separate
// neighbour, flag, scan and total passes, and take 0.7 ms of kernels in 64
// launches now: the rounds 0.49, the last 4,096 clusters 0.18.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "hrt_internal.h"

namespace hrt {
namespace {

constexpr int kBlock = 256;
constexpr uint32_t kPlocRadius = 8;  // window half-width; 4..32 measured, 8 visits fewest on AO rays

// A cluster: box, its reference as a pair child (packed leaf or internal node
// id) in lo.w; in hi.w its index in the left/right node layout (leaf L-1+m or
// internal id) in the low kLrBits bits and the height of its subtree above
// (0 for a leaf, stuck at kMaxHeight).
struct Cluster {
  float4 lo, hi;
};
constexpr uint32_t kLrBits = 25;  // 2 L - 1 < 2^25
constexpr uint32_t kLrMask = (1u << kLrBits) - 1u;
constexpr uint32_t kMaxHeight = 127;
static_assert(kMaxLevels4 < int(kMaxHeight), "a stuck height must not pass for a storable one");

// Where a round starts: clusters, the id of its first merge, the buffer they
// are in, and (once one is left) the height of the tree.
struct PlocState {
  uint32_t n, next_id, buf, height;
};

__device__ inline float union_half_area(float3 alo, float3 ahi, float3 blo, float3 bhi) {
  const float ex = fmaxf(ahi.x, bhi.x) - fminf(alo.x, blo.x);
  const float ey = fmaxf(ahi.y, bhi.y) - fminf(alo.y, blo.y);
  const float ez = fmaxf(ahi.z, bhi.z) - fminf(alo.z, blo.z);
  const float a = ex * ey + ey * ez + ez * ex;
  return (a == a) ? a : INFINITY;
}

// Boxes in LDS, a coordinate per array: conflict-free for neighbouring items.
template <int kN>
struct Boxes {
  float lx[kN], ly[kN], lz[kN], hx[kN], hy[kN], hz[kN];
  __device__ void put(int k, const Cluster& c) {
    lx[k] = c.lo.x;
    ly[k] = c.lo.y;
    lz[k] = c.lo.z;
    hx[k] = c.hi.x;
    hy[k] = c.hi.y;
    hz[k] = c.hi.z;
  }
  __device__ float3 lo(int k) const { return make_float3(lx[k], ly[k], lz[k]); }
  __device__ float3 hi(int k) const { return make_float3(hx[k], hy[k], hz[k]); }
  // The neighbour item i picks among n clusters; item j is at slot j - first.
  __device__ uint32_t pick(uint32_t i, uint32_t n, int64_t first) const {
    const int li = int(int64_t(i) - first);
    const float3 alo = lo(li), ahi = hi(li);
    const uint32_t from = i > kPlocRadius ? i - kPlocRadius : 0u;
    const uint32_t to = min(n - 1, i + kPlocRadius);
    float best = 0.0f;
    uint32_t bj = 0xFFFFFFFFu;
    for (uint32_t j = from; j <= to; j++) {
      if (j == i) continue;
      const int lj = int(int64_t(j) - first);
      const float a = union_half_area(alo, ahi, lo(lj), hi(lj));
      if (bj == 0xFFFFFFFFu || a < best) {
        best = a;
        bj = j;
      }
    }
    return bj;
  }
};

// Node `id` of clusters a (left) and b: its pair, its children's parent
// entries, and the cluster it becomes.
__device__ inline Cluster join(const Cluster& a, const Cluster& b, uint32_t id, NodePair* __restrict__ pairs,
                               uint32_t* __restrict__ parent, uint32_t* __restrict__ lr) {
  float4* w = reinterpret_cast<float4*>(pairs + id);
  w[0] = a.lo;
  w[1] = make_float4(a.hi.x, a.hi.y, a.hi.z, 0.0f);
  w[2] = b.lo;
  w[3] = make_float4(b.hi.x, b.hi.y, b.hi.z, 0.0f);
  const uint32_t ra = __float_as_uint(a.lo.w), rb = __float_as_uint(b.lo.w);
  const uint32_t xa = __float_as_uint(a.hi.w), xb = __float_as_uint(b.hi.w);
  if ((ra & kLeafBit) == 0u) parent[ra] = id << 1;
  if ((rb & kLeafBit) == 0u) parent[rb] = (id << 1) | 1u;
  if (lr) {
    lr[2 * id] = xa & kLrMask;
    lr[2 * id + 1] = xb & kLrMask;
  }
  const uint32_t h = min(max(xa >> kLrBits, xb >> kLrBits) + 1u, kMaxHeight);
  Cluster u;
  u.lo = make_float4(fminf(a.lo.x, b.lo.x), fminf(a.lo.y, b.lo.y), fminf(a.lo.z, b.lo.z), __uint_as_float(id));
  u.hi = make_float4(fmaxf(a.hi.x, b.hi.x), fmaxf(a.hi.y, b.hi.y), fmaxf(a.hi.z, b.hi.z),
                     __uint_as_float(id | (h << kLrBits)));
  return u;
}

// Leaves (boxes and refs from their parents' pairs) as the first clusters, and
// the first round's record.
__global__ __launch_bounds__(kBlock) void k_ploc_init(const NodePair* __restrict__ pairs,
                                                      const uint32_t* __restrict__ parent_leaf, uint32_t L,
                                                      Cluster* __restrict__ out, PlocState* __restrict__ st) {
  const uint32_t m = blockIdx.x * kBlock + threadIdx.x;
  if (m == 0) *st = PlocState{L, L - 2u, 0u, 0u};
  if (m >= L) return;
  const uint32_t pl = parent_leaf[m];
  const float4* w = reinterpret_cast<const float4*>(pairs + (pl >> 1)) + 2 * (pl & 1u);
  const float4 lo = w[0], hi = w[1];
  Cluster c;
  c.lo = lo;
  c.hi = make_float4(hi.x, hi.y, hi.z, __uint_as_float(L - 1 + m));
  out[m] = c;
}

// The first half of a round.  A workgroup picks the neighbours of a tile's
// clusters and of kPlocRadius more on either side (a pair is mutual if both
// picked each other), from boxes of twice that margin in LDS, and writes a byte
// per cluster -- its partner's offset, whether it starts a pair, whether it
// survives -- and the tile's two totals.
constexpr uint32_t kTile = 256;
constexpr uint8_t kStarts = 32, kSurvives = 64;  // above the offset + kPlocRadius (0..16)
constexpr uint32_t kPlocGrid = 4096;

__global__ __launch_bounds__(kBlock) void k_ploc_pick(const Cluster* __restrict__ c0, const Cluster* __restrict__ c1,
                                                      const PlocState* __restrict__ st, uint32_t stop,
                                                      uint8_t* __restrict__ code, uint2* __restrict__ counts) {
  constexpr int kR = int(kPlocRadius), kN = int(kTile) + 4 * kR;
  __shared__ Boxes<kN> boxes;
  __shared__ uint16_t nn[kTile + 2 * kR];  // slot of the picked neighbour
  __shared__ uint32_t total[2];
  const uint32_t n = st->n;
  if (n <= stop) return;
  const Cluster* __restrict__ c = st->buf ? c1 : c0;
  for (uint32_t tile = blockIdx.x; uint64_t(tile) * kTile < n; tile += gridDim.x) {
    const uint32_t base = tile * kTile;
    const int64_t first = int64_t(base) - 2 * kR;
    __syncthreads();
    if (threadIdx.x < 2) total[threadIdx.x] = 0u;
    for (int k = threadIdx.x; k < kN; k += kBlock) {
      const int64_t g = first + k;
      if (g >= 0 && g < int64_t(n)) boxes.put(k, c[g]);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < int(kTile) + 2 * kR; k += kBlock) {
      const int64_t g = first + kR + k;
      if (g >= 0 && g < int64_t(n)) nn[k] = uint16_t(int64_t(boxes.pick(uint32_t(g), n, first)) - first);
    }
    __syncthreads();
    uint32_t starts = 0, survives = 0;
    for (uint32_t k = threadIdx.x; k < kTile && base + k < n; k += kBlock) {
      const int me = int(k) + 2 * kR, other = int(nn[k + kR]);  // slots
      const bool mutual = int(nn[other - kR]) == me;
      const bool starts_k = mutual && me < other, survives_k = !(mutual && me > other);
      code[base + k] = uint8_t(other - me + kR) | (starts_k ? kStarts : 0) | (survives_k ? kSurvives : 0);
      starts += starts_k;
      survives += survives_k;
    }
    if (starts) atomicAdd(&total[0], starts);
    if (survives) atomicAdd(&total[1], survives);
    __syncthreads();
    if (threadIdx.x == 0) counts[tile] = make_uint2(total[0], total[1]);
  }
}

// The second half: every tile adds up the totals of the tiles before it, ranks
// its own clusters and writes nodes and surviving clusters.  The sums grow with
// the square of the tiles (on a million clusters 3,907 tiles read 16 KB each on
// average, from the L2), but stay the smaller part up to the largest tree: a
// commit that clusters 16 M triangles takes 14 ms, 23 with scans of the flags
// and the host between the rounds.  The last tile leaves the next round's
// record; a round that has nothing to do hands its own on.
__global__ __launch_bounds__(kBlock) void k_ploc_merge(Cluster* __restrict__ c0, Cluster* __restrict__ c1,
                                                       const PlocState* __restrict__ st, uint32_t stop,
                                                       const uint8_t* __restrict__ code,
                                                       const uint2* __restrict__ counts,
                                                       NodePair* __restrict__ pairs, uint32_t* __restrict__ parent,
                                                       uint32_t* __restrict__ lr, PlocState* __restrict__ next) {
  constexpr uint32_t kPer = kTile / kBlock, kWaves = kBlock / 64;
  __shared__ uint32_t before[2];
  __shared__ uint32_t wave_sum[kWaves];
  const PlocState s = *st;
  const uint32_t n = s.n;
  if (n <= stop) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *next = s;
    return;
  }
  const Cluster* __restrict__ cin = s.buf ? c1 : c0;
  Cluster* __restrict__ cout = s.buf ? c0 : c1;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  for (uint32_t tile = blockIdx.x; uint64_t(tile) * kTile < n; tile += gridDim.x) {
    const uint32_t base = tile * kTile;
    __syncthreads();
    if (threadIdx.x < 2) before[threadIdx.x] = 0u;
    __syncthreads();
    uint32_t bs = 0, bk = 0;
    for (uint32_t t = threadIdx.x; t < tile; t += kBlock) {
      bs += counts[t].x;
      bk += counts[t].y;
    }
    if (bs) atomicAdd(&before[0], bs);
    if (bk) atomicAdd(&before[1], bk);
    // this thread's kPer consecutive clusters; starts in the low half-word of
    // the running sums, survivors in the high one
    const uint32_t at = base + threadIdx.x * kPer;
    uint8_t cd[kPer];
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
      cd[k] = at + k < n ? code[at + k] : uint8_t(0);
      sum += ((cd[k] & kStarts) ? 1u : 0u) + ((cd[k] & kSurvives) ? 0x10000u : 0u);
    }
    uint32_t incl = sum;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(incl, o);
      if (lane >= uint32_t(o)) incl += y;
    }
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
    for (uint32_t w = 0; w < wave; w++) run += wave_sum[w];
    uint32_t ids = before[0] + (run & 0xFFFFu), pos = before[1] + (run >> 16);
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
      if (!(cd[k] & kSurvives)) continue;
      Cluster u = cin[at + k];
      if (cd[k] & kStarts) {
        u = join(u, cin[at + k + (cd[k] & 31u) - kPlocRadius], s.next_id - ids, pairs, parent, lr);
        ids++;
      }
      cout[pos++] = u;
    }
    if (uint64_t(tile + 1) * kTile >= n && threadIdx.x == 0) {
      uint32_t all = 0;
      for (uint32_t w = 0; w < kWaves; w++) all += wave_sum[w];
      *next = PlocState{before[1] + (all >> 16), s.next_id - before[0] - (all & 0xFFFFu), s.buf ^ 1u, 0u};
    }
  }
}

// All remaining rounds of at most kFinish clusters in one workgroup, the
// clusters in LDS.  Item i of a round belongs to thread i mod kFinishThreads.
// Ends with one cluster, or with more if a round merged nothing (the host sees
// the count).
constexpr uint32_t kFinish = 4096, kFinishThreads = 1024, kFinishPer = kFinish / kFinishThreads;

__global__ __launch_bounds__(kFinishThreads) void k_ploc_finish(const Cluster* __restrict__ c0,
                                                                const Cluster* __restrict__ c1,
                                                                PlocState* __restrict__ st,
                                                                NodePair* __restrict__ pairs,
                                                                uint32_t* __restrict__ parent,
                                                                uint32_t* __restrict__ lr) {
  constexpr uint32_t kWaves = kFinishThreads / 64;
  __shared__ Boxes<int(kFinish)> boxes;
  __shared__ uint32_t ref[kFinish], aux[kFinish];
  __shared__ uint16_t nn[kFinish];
  __shared__ uint32_t sums[kFinishPer * kWaves + 1];  // starts and survivors before each 64 items, packed
  const PlocState s = *st;
  uint32_t n = s.n, next_id = s.next_id;
  if (n > kFinish || n <= 1u) return;
  const Cluster* __restrict__ c = s.buf ? c1 : c0;
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  for (uint32_t i = t; i < n; i += kFinishThreads) {
    const Cluster x = c[i];
    boxes.put(int(i), x);
    ref[i] = __float_as_uint(x.lo.w);
    aux[i] = __float_as_uint(x.hi.w);
  }
  auto get = [&](uint32_t i) {
    Cluster x;
    x.lo = make_float4(boxes.lx[i], boxes.ly[i], boxes.lz[i], __uint_as_float(ref[i]));
    x.hi = make_float4(boxes.hx[i], boxes.hy[i], boxes.hz[i], __uint_as_float(aux[i]));
    return x;
  };
  __syncthreads();
  while (n > 1u) {
    for (uint32_t i = t; i < n; i += kFinishThreads) nn[i] = uint16_t(boxes.pick(i, n, 0));
    __syncthreads();
    bool starts[kFinishPer], survives[kFinishPer];
    uint32_t rank_s[kFinishPer], rank_k[kFinishPer];
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; k++) {
      const uint32_t i = t + k * kFinishThreads;
      starts[k] = survives[k] = false;
      if (i < n) {
        const uint32_t j = nn[i];
        const bool mutual = nn[j] == i;
        starts[k] = mutual && i < j;
        survives[k] = !(mutual && i > j);
      }
      const uint64_t ms = __ballot(starts[k]), mk = __ballot(survives[k]);
      rank_s[k] = lanes_below(ms);
      rank_k[k] = lanes_below(mk);
      if (lane == 0) sums[k * kWaves + wave] = uint32_t(__popcll(ms)) + (uint32_t(__popcll(mk)) << 16);
    }
    __syncthreads();
    if (wave == 0) {  // kFinishPer * kWaves == 64 sums: exclusive scan by one wave
      static_assert(kFinishPer * kWaves == 64, "one wave scans the sums");
      const uint32_t x = sums[lane];
      uint32_t incl = x;
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(incl, o);
        if (lane >= uint32_t(o)) incl += y;
      }
      sums[lane] = incl - x;
      if (lane == 63) sums[64] = incl;
    }
    __syncthreads();
    const uint32_t all = sums[64];
    Cluster u[kFinishPer];
    uint32_t pos[kFinishPer];
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; k++) {
      if (!survives[k]) continue;
      const uint32_t i = t + k * kFinishThreads, b = sums[k * kWaves + wave];
      u[k] = get(i);
      pos[k] = (b >> 16) + rank_k[k];
      if (starts[k]) u[k] = join(u[k], get(nn[i]), next_id - (b & 0xFFFFu) - rank_s[k], pairs, parent, lr);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < kFinishPer; k++) {
      if (!survives[k]) continue;
      boxes.put(int(pos[k]), u[k]);
      ref[pos[k]] = __float_as_uint(u[k].lo.w);
      aux[pos[k]] = __float_as_uint(u[k].hi.w);
    }
    __syncthreads();
    if ((all & 0xFFFFu) == 0u) break;
    next_id -= all & 0xFFFFu;
    n = all >> 16;
  }
  if (t == 0) *st = PlocState{n, next_id, s.buf, aux[0] >> kLrBits};
}

inline uint32_t blocks_for(uint64_t n) { return uint32_t(std::max<uint64_t>(1, (n + kBlock - 1) / kBlock)); }

}  // namespace

hipError_t blas_ploc(Blas& b, hipStream_t s, bool* replaced) {
  *replaced = false;
  const uint32_t L = b.leaves;
  if (L < 3) return hipSuccess;  // one or two leaves: nothing to cluster
  // Rounds to enqueue before the host looks: a round leaves 75 to 87 % of the
  // clusters (562,428 leaves of such hills are down to kFinish after 26 rounds,
  // 4,177,918 of a soup after 40), and one without work costs about 4 us.  With
  // its waits the hierarchy took 4.1 ms on them, 1.0 ms this way.
  uint32_t rounds = 0;
  for (double n = L; n > double(kFinish); n *= 0.85) rounds++;
  // device scratch: two cluster arrays, a byte per cluster, totals per tile,
  // the rounds' records
  const uint32_t ntiles = (L + kTile - 1) / kTile;
  size_t words = 0;
  auto take = [&](size_t n) { size_t o = words; words += (n + 63) & ~size_t(63); return o; };
  const size_t o_ca = take(8ull * L), o_cb = take(8ull * L), o_code = take((size_t(L) + 3) / 4);
  const size_t o_cnt = take(2ull * ntiles), o_st = take(4ull * (rounds + 2));
  NodePair* npairs = nullptr;
  uint32_t *nparent = nullptr, *nlr = nullptr;
  uint32_t* base = nullptr;
  // the same capacities as blas_alloc's (pairs for every triangle but one),
  // so the swapped arrays can stand in for the originals everywhere
  const size_t cap = std::max<size_t>(b.ntris > 1 ? b.ntris - 1 : 1, 1);
  hipError_t e = b.mem->alloc(&npairs, sizeof(NodePair) * cap);
  if (e == hipSuccess) e = b.mem->alloc(&nparent, 4ull * cap);
  if (e == hipSuccess && b.karras_lr) e = b.mem->alloc(&nlr, 8ull * cap);
  if (e == hipSuccess) e = b.mem->alloc(&base, 4 * words);
  Readback back(b.mem);
  bool ok = false;
  if (e == hipSuccess) {
    Cluster* ca = reinterpret_cast<Cluster*>(base + o_ca);
    Cluster* cb = reinterpret_cast<Cluster*>(base + o_cb);
    uint8_t* code = reinterpret_cast<uint8_t*>(base + o_code);
    uint2* counts = reinterpret_cast<uint2*>(base + o_cnt);
    PlocState* st = reinterpret_cast<PlocState*>(base + o_st);
    const uint32_t grid = std::min(ntiles, kPlocGrid);
    k_ploc_init<<<blocks_for(L), kBlock, 0, s>>>(b.pairs, b.parent_leaf, L, ca, st);
    PlocState now{L, L - 2, 0, 0};
    while (now.n > 1) {
      for (uint32_t r = 0; r < rounds; r++) {
        k_ploc_pick<<<grid, kBlock, 0, s>>>(ca, cb, st + r, kFinish, code, counts);
        k_ploc_merge<<<grid, kBlock, 0, s>>>(ca, cb, st + r, kFinish, code, counts, npairs, nparent, nlr, st + r + 1);
      }
      k_ploc_finish<<<1, kFinishThreads, 0, s>>>(ca, cb, st + rounds, npairs, nparent, nlr);
      PlocState after;
      if ((e = hipGetLastError()) != hipSuccess) break;
      if ((e = back.read(0, st + rounds, sizeof(after) / 4, s)) != hipSuccess) break;
      if ((e = hipStreamSynchronize(s)) != hipSuccess) break;
      std::memcpy(&after, back.words(), sizeof(after));
      // every round merges at least one pair (see the rule above), and each
      // merge takes one cluster and one id
      if (after.n == 0 || after.n >= now.n || now.n - after.n != now.next_id - after.next_id) {
        e = hipErrorIllegalState;
        break;
      }
      now = after;
      if (now.n > 1 && (e = hipMemcpyAsync(st, st + rounds, sizeof(*st), hipMemcpyDeviceToDevice, s)) != hipSuccess) break;
    }
    // the BVH4 traversal stack holds kStackDepth4 entries: at most kMaxLevels4
    // internal levels
    ok = e == hipSuccess && now.height <= uint32_t(kMaxLevels4);
  }
  const hipError_t werr = hipStreamSynchronize(s);  // the scratch may still be in use
  if (e == hipSuccess) e = werr;
  if (e == hipSuccess && ok) {
    std::swap(b.pairs, npairs);
    std::swap(b.parent, nparent);
    if (nlr) std::swap(b.karras_lr, nlr);
    b.clustered = true;
    *replaced = true;
  }
  b.mem->free(base);
  b.mem->free(npairs);
  b.mem->free(nparent);
  b.mem->free(nlr);
  return e;
}

}  // namespace hrt
