// Dense octree8 (drop-in mode): builder and classic walks over the
// reference's byte layout (OctreeNode8, src/sbh_ffi.cu:47-65).
//
// Builder (replaces src/sbh_ffi.cu:1039-1420):
//   codes -> stable radix sort (no atomics: intra-bin order = input order)
//   -> leaf records in sorted order -> one kernel per three levels, from the
//   deepest: cell starts, sums and complete node records.
// Walks (replace src/sbh_ffi.cu:1950-2144): 64 queries per wave share a depth-first
// traversal of the nodes that any of them opens, parameters passed by value.
#include <type_traits>

#include "common.hpp"
#include "o8walk.hpp"
#include "tree.hpp"

namespace sbh {
namespace {

constexpr int kB = 256;

struct BuildGeom {
  float min_x, min_y, min_z;
  float span;
  float cx, cy, cz, half_size;
};

__global__ __launch_bounds__(kB) void k_codes(const float* __restrict__ pts, int64_t n,
                                              BuildGeom g, int bits,
                                              uint32_t* __restrict__ codes) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * kB + threadIdx.x;
  if (i >= n) return;
  uint32_t qx = quantize_axis(pts[3 * i + 0], g.min_x, g.span, bits);
  uint32_t qy = quantize_axis(pts[3 * i + 1], g.min_y, g.span, bits);
  uint32_t qz = quantize_axis(pts[3 * i + 2], g.min_z, g.span, bits);
  codes[i] = morton3(qx, qy, qz);
}

__global__ __launch_bounds__(kB) void k_leaf_gather(const float* __restrict__ pts,
                                                    const float* __restrict__ nrm,
                                                    const float* __restrict__ ms, int64_t n,
                                                    const uint32_t* __restrict__ perm,
                                                    Leaf3* __restrict__ leaf) {
  int64_t r = static_cast<int64_t>(blockIdx.x) * kB + threadIdx.x;
  if (r >= n) return;
  int64_t i = perm[r];
  Leaf3 o;
  o.pos[0] = pts[3 * i + 0];
  o.pos[1] = pts[3 * i + 1];
  o.pos[2] = pts[3 * i + 2];
  o.normal[0] = nrm[3 * i + 0];
  o.normal[1] = nrm[3 * i + 1];
  o.normal[2] = nrm[3 * i + 2];
  o.mass = ms[i];
  o.alpha = 1.0f;
  leaf[r] = o;
}

// First position in [lo, hi) of the sorted codes with codes[pos] >= b (hi if none),
// by the 64 lanes of a wave: 64 probes a step.
__device__ __forceinline__ int64_t wave_lower_bound(const uint32_t* __restrict__ codes, int64_t lo,
                                                    int64_t hi, uint64_t b, int lane) {
  while (lo < hi) {
    const int64_t step = (hi - lo + 63) / 64;
    const int64_t p = lo + lane * step;
    const bool below = p < hi && codes[p] < b;
    const int k = __popcll(__ballot(below));  // the first k probes are below
    if (k == 0) return lo;
    const int64_t next = lo + k * step;
    lo = lo + (k - 1) * step + 1;
    hi = next < hi ? next : hi;
  }
  return lo;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2), aligned(4)));

// past: beyond what the caches hold, so not to be kept in them
__device__ __forceinline__ void store_pair(u32x2 v, u32x2* p, bool past) {
  if (past)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

// What a block leaves for the next one up about the cell that its nodes share.
struct CellSums {
  uint32_t cnt, start, mask;  // points below, first of them, children with points
  float a[7];                 // mass, sum m x (3), sum m n (3)
};

constexpr int kSpan = 3;                  // levels a block reduces
constexpr int kCells = 1 << (3 * kSpan);  // cells of its lowest level
constexpr int kStage = 2048;              // codes or records staged at a time
constexpr int kFewPoints = 16;            // a leaf of more is summed by a wave
constexpr int kNodeWords = sizeof(Node8) / 4;
constexpr int kRecWords = sizeof(Leaf3) / 4;
static_assert(sizeof(Node8) == 26 * 4 && sizeof(Leaf3) == 8 * 4, "records are copied by words");

// Node records of the dense octree (src/sbh_ffi.cu:1683-1876): one block takes
// the subtree below one cell of level `level` - `span` (blockIdx.x) and writes the
// nodes of levels level - span + 1 .. level (and the root's when span == level),
// leaving the cell's own sums in `up`.  BOTTOM: level is the deepest, its cells
// are summed from the sorted leaf records (in sorted order; counts and starts from
// the sorted codes); else they come from `down`, as the blocks below left them.
// A parent adds its occupied children in octant order.
//
// Bound by the writes of the records: 136 bytes a node, staged in LDS so that a
// wave writes them as one run.  At depth 8 (1.9e7 nodes) over 128^3 points 0.8 ms;
// one kernel each for the cells' starts, the leaf sums, every level's reduction and
// every level's records, a thread per bin or node, took 1.66.  A leaf of 75,000
// points: 1.2 ms instead of 10.
template <bool BOTTOM>
__global__ __launch_bounds__(kB) void k_subtree(
    const uint32_t* __restrict__ codes, const Leaf3* __restrict__ leaf, int64_t n,
    const CellSums* __restrict__ down, CellSums* __restrict__ up, int level, int span,
    int max_level, BuildGeom g, bool past, Node8* __restrict__ nodes,
    Leaf3* __restrict__ contrib_out) {
  constexpr int kWaves = kB / 64;
  // cells of the block, level by level from the lowest: kCells, kCells / 8, ..., 1
  constexpr int kAll = kCells + kCells / 8 + kCells / 64 + kCells / 512;
  __shared__ float s_sum[kAll][7];
  __shared__ uint32_t s_cnt[kAll];
  __shared__ uint32_t s_start[kCells + 1];
  __shared__ uint8_t s_mask[kAll];
  __shared__ int64_t s_range[2];
  __shared__ uint32_t s_stage[kWaves][64 * kNodeWords];
  static_assert(sizeof(s_stage) >= 4 * kStage, "the staged codes share the records' space");
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int cells = 1 << (3 * span);
  const uint64_t cell0 = static_cast<uint64_t>(blockIdx.x) << (3 * span);
  if (BOTTOM) {
    if (w < 2) {
      const int64_t r = wave_lower_bound(codes, 0, n, cell0 + (w == 0 ? 0 : cells), lane);
      if (lane == 0) s_range[w] = r;
    }
    __syncthreads();
    const int64_t r0 = s_range[0], r1 = s_range[1];
    uint32_t* staged = &s_stage[0][0];
    const bool in_lds = r1 - r0 <= kStage;
    if (in_lds)
      for (int64_t k = r0 + tid; k < r1; k += kB) staged[k - r0] = codes[k];
    __syncthreads();
    for (int c = tid; c <= cells; c += kB) {
      const uint64_t b = cell0 + c;
      int64_t lo = r0, hi = r1;
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((in_lds ? staged[mid - r0] : codes[mid]) < b)
          lo = mid + 1;
        else
          hi = mid;
      }
      s_start[c] = static_cast<uint32_t>(lo);
    }
    __syncthreads();
    // counts, and sums of the leaves in sorted order: few points by a thread ...
    for (int c = tid; c < cells; c += kB) {
      const uint32_t s = s_start[c], e = s_start[c + 1];
      s_cnt[c] = e - s;
      s_mask[c] = 0;
      if (e - s > kFewPoints) continue;
      float a[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (uint32_t j = s; j < e; ++j) {
        const Leaf3 L = leaf[j];
        const float m = L.mass;
        a[0] += m;
        a[1] += m * L.pos[0];
        a[2] += m * L.pos[1];
        a[3] += m * L.pos[2];
        a[4] += m * L.normal[0];
        a[5] += m * L.normal[1];
        a[6] += m * L.normal[2];
      }
      for (int k = 0; k < 7; ++k) s_sum[c][k] = a[k];
    }
    // ... and many by a wave that stages 64 records at a time, lane k < 7
    // adding up the k-th sum (a chain of adds in the same order)
    __syncthreads();
    uint32_t* buf = s_stage[w];
    for (int c0 = w; c0 < cells; c0 += 64 * kWaves) {
      const int mine = c0 + kWaves * lane;
      uint64_t many = __ballot(mine < cells && s_cnt[mine < cells ? mine : 0] > kFewPoints);
      while (many != 0) {
        const int c = c0 + kWaves * __builtin_ctzll(many);
        many &= many - 1;
        const uint32_t s = __builtin_amdgcn_readfirstlane(s_start[c]);
        const uint32_t e = __builtin_amdgcn_readfirstlane(s_start[c + 1]);
        float acc = 0.f;
        Leaf3 next = leaf[s + lane < e ? s + lane : s];
        for (uint32_t j = s; j < e; j += 64) {
          // word 0: mass; 1..6: position and normal; odd stride
          float* rec = reinterpret_cast<float*>(buf) + 7 * lane;
          rec[0] = next.mass;
          for (int k = 0; k < 3; ++k) rec[1 + k] = next.pos[k];
          for (int k = 0; k < 3; ++k) rec[4 + k] = next.normal[k];
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
          if (e - j > 64) next = leaf[j + 64 + lane < e ? j + 64 + lane : s];
          const int count = e - j < 64 ? static_cast<int>(e - j) : 64;
          if (lane < 7) {
            const float* p = reinterpret_cast<const float*>(buf);
            if (lane == 0) {
#pragma unroll 8
              for (int u = 0; u < count; ++u) acc += p[7 * u];
            } else {
#pragma unroll 8
              for (int u = 0; u < count; ++u) acc += p[7 * u] * p[7 * u + lane];
            }
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
        }
        if (lane < 7) s_sum[c][lane] = acc;
      }
    }
  } else {
    for (int c = tid; c < cells; c += kB) {
      const CellSums d = down[cell0 + c];
      s_cnt[c] = d.cnt;
      s_start[c] = d.start;
      s_mask[c] = static_cast<uint8_t>(d.mask);
      for (int k = 0; k < 7; ++k) s_sum[c][k] = d.a[k];
    }
  }
  __syncthreads();
  // parents from their children (src/sbh_ffi.cu:1745-1786)
  int base = 0;
  for (int m = cells / 8; m > 0; m /= 8) {
    const int pbase = base + 8 * m;
    if (tid < m) {
      uint32_t count = 0, mask = 0;
      float a[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < 8; ++c) {
        const int ch = base + 8 * tid + c;
        const uint32_t cc = s_cnt[ch];
        if (cc == 0) continue;
        count += cc;
        mask |= 1u << c;
        for (int k = 0; k < 7; ++k) a[k] += s_sum[ch][k];
      }
      s_cnt[pbase + tid] = count;
      s_mask[pbase + tid] = static_cast<uint8_t>(mask);
      for (int k = 0; k < 7; ++k) s_sum[pbase + tid][k] = a[k];
    }
    __syncthreads();
    base = pbase;
  }
  if (tid == 0 && up != nullptr) {
    CellSums d;
    d.cnt = s_cnt[base];
    d.start = s_start[0];
    d.mask = s_mask[base];
    for (int k = 0; k < 7; ++k) d.a[k] = s_sum[base][k];
    up[blockIdx.x] = d;
  }
  // the records, 64 nodes a wave at a time: level l holds `count` of them from
  // LDS slot lbase on; slot 0 of level l is node `first` of the level
  int lbase = 0, round = 0;
  const int top_level = span == level ? 0 : level - span + 1;
  for (int l = level; l >= top_level; --l) {
    const int up_by = level - l, count = cells >> (3 * up_by);
    const uint32_t first = static_cast<uint32_t>(cell0 >> (3 * up_by));
    // nodes of the levels above l: (8^l - 1) / 7
    auto nodes_above = [](int k) { return static_cast<uint32_t>(((uint64_t{1} << (3 * k)) - 1) / 7); };
    const uint32_t level_offset = nodes_above(l);
    for (int i0 = 0; i0 < count; i0 += 64, ++round) {
      if (round % kWaves != w) continue;
      const int i = i0 + lane, here = count - i0 < 64 ? count - i0 : 64;
      uint32_t* buf = s_stage[w];
      if (lane < here) {
        const uint32_t idx = first + i;
        const uint32_t node_idx = level_offset + idx;
        Node8 node;
        node.depth = static_cast<uint8_t>(l);
        node.parent = l == 0 ? node_idx : nodes_above(l - 1) + (idx >> 3);
        node.is_leaf = l == max_level ? 1 : 0;
        node.child_mask = 0;
        node.pad0 = 0;
        node.first_child = 0xFFFFFFFFu;
        node.start = s_start[i << (3 * up_by)];
        node.end = node.start + s_cnt[lbase + i];
        int ix = 0, iy = 0, iz = 0;
        for (int b = 0; b < l; ++b) {
          ix |= static_cast<int>((idx >> (3 * b + 0)) & 1u) << b;
          iy |= static_cast<int>((idx >> (3 * b + 1)) & 1u) << b;
          iz |= static_cast<int>((idx >> (3 * b + 2)) & 1u) << b;
        }
        {
#pragma clang fp contract(off)
          float step = g.half_size * 2.0f / static_cast<float>(1 << l);
          // (c - h) + (i + 0.5) * step with the a*b+c fused, as the reference's
          // compiler contracts it by default.
          node.cx = fmaf(static_cast<float>(ix) + 0.5f, step, g.cx - g.half_size);
          node.cy = fmaf(static_cast<float>(iy) + 0.5f, step, g.cy - g.half_size);
          node.cz = fmaf(static_cast<float>(iz) + 0.5f, step, g.cz - g.half_size);
          node.half_size = step * 0.5f;
          node.diameter = step * 1.7320508075688772f;
        }
        if (l < max_level) {
          const uint32_t child_base = nodes_above(l + 1) + (idx << 3);
          const uint32_t mask = s_mask[lbase + i];
          for (uint32_t c = 0; c < 8; ++c) node.child[c] = child_base + c;
          node.child_mask = static_cast<uint8_t>(mask);
          if (mask == 0)
            node.is_leaf = 1;
          else
            node.first_child = child_base + __builtin_ctz(mask);
        } else {
          for (int c = 0; c < 8; ++c) node.child[c] = 0xFFFFFFFFu;
        }
        const float* sum = s_sum[lbase + i];
        const float mass = sum[0];
        node.contrib.alpha = 1.0f;
        node.contrib.mass = mass;
        if (mass > 0.0f) {
          node.contrib.pos[0] = sum[1] / mass;
          node.contrib.pos[1] = sum[2] / mass;
          node.contrib.pos[2] = sum[3] / mass;
          node.contrib.normal[0] = sum[4] / mass;
          node.contrib.normal[1] = sum[5] / mass;
          node.contrib.normal[2] = sum[6] / mass;
        } else {
          for (int a = 0; a < 3; ++a) node.contrib.pos[a] = node.contrib.normal[a] = 0.0f;
        }
        uint32_t words[kNodeWords];
        __builtin_memcpy(words, &node, sizeof(node));
#pragma unroll
        for (int k = 0; k < kNodeWords; ++k) buf[lane * kNodeWords + k] = words[k];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const uint64_t n0 = static_cast<uint64_t>(level_offset) + first + i0;
      // words in pairs: 8-byte stores (both records are whole pairs)
      auto* out = reinterpret_cast<u32x2*>(nodes) + n0 * (kNodeWords / 2);
      const auto* in = reinterpret_cast<const u32x2*>(buf);
      for (int k = lane; k < here * (kNodeWords / 2); k += 64) store_pair(in[k], out + k, past);
      // the record's last words are its contribution
      auto* rec = reinterpret_cast<u32x2*>(contrib_out) + n0 * (kRecWords / 2);
      for (int k = lane; k < here * (kRecWords / 2); k += 64)
        store_pair(in[(k / (kRecWords / 2)) * (kNodeWords / 2) + (kNodeWords - kRecWords) / 2 +
                      k % (kRecWords / 2)],
                   rec + k, past);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    lbase += count;
  }
}

// ------------------------------------------------------------------ walks
using o8::WalkParams;
using o8::use_far_field;
using o8::should_prune;
using o8::contribution;
using o8::kGravGrad;
using o8::kSoftForce;
using o8::kSoftVjp;
using o8::kWinding;


// Point record read once per wave through the scalar data cache (the buffers
// are read-only during a walk; records are 4-byte aligned).
typedef uint32_t u32x8 __attribute__((ext_vector_type(8), aligned(4)));
typedef __attribute__((address_space(4))) const u32x8 cu32x8;

__device__ __forceinline__ Leaf3 sload_leaf3(const Leaf3* leaf, uint32_t j) {
  const u32x8 v = ((cu32x8*)(leaf))[j];
  Leaf3 r;
  uint32_t* d = reinterpret_cast<uint32_t*>(&r);
#pragma unroll
  for (int k = 0; k < 8; ++k) d[k] = v[k];
  return r;
}

constexpr int kRun = 4;              // points read together
constexpr int kWStack = 96;          // >= 7 * 10 + 8 entries for max_depth 10
constexpr uint32_t kRootEntry = ~0u;  // stack entry whose only child is node 0
constexpr int kAccs = 4;             // partial sums per query (kParts, kSplitParts)

// How a query's contributions add up: kAccs partial sums by subtree, kept by one
// wave or dealt to the kAccs waves of a block, or one running sum in the order
// of the reference's DFS.
enum WalkSums { kParts, kSplitParts, kRunning };

// Partial sum of the node in child slot c: the 8 octants twice over the 4
// sums, so that neighbours in every direction differ.
__device__ __forceinline__ uint32_t key_of(uint32_t c) { return (c + (c >> 2)) & 3u; }

// What the walk needs of a child node, as the lane that fetched it left it
// in LDS for the wave (read back as broadcasts).
struct alignas(16) Child {
  float cx, cy, cz;     // cell centre
  float open2;          // d^2 below this: nearer than beta diameters for sure
  float bx, by, bz;     // box times the periodic image of the wave's first query (PER)
  float far2;           // d^2 from this on: farther than beta diameters for sure
  float lx, ly, lz;     // cell box (prune)
  float mass;
  float hx, hy, hz;
  uint32_t id;
  float px, py, pz;     // centre of mass
  uint32_t start;
  uint32_t end, is_leaf, key, deep;  // key: partial sum; deep: at or below split_level
};
static_assert(sizeof(Child) == 96, "Child is read as six float4");

// Displacement q - p with the image shift b of a whole wave; *sure says that
// it is the minimum image, i.e. that min_image_floor gives the same bits: the
// shift is box * k with |k| <= 16 (infinite otherwise) and every component is
// within (0.5 - 1e-5) boxes, 2e-6 being the most that the rounding of
// d / box + 0.5 can move it there.
template <bool PER>
__device__ __forceinline__ float3 wave_delta(float qx, float qy, float qz, float px, float py,
                                             float pz, const Child& c, float limit, bool* sure) {
#pragma clang fp contract(off)
  float3 d = make_float3(qx - px, qy - py, qz - pz);
  *sure = true;
  if constexpr (PER) {
    d = make_float3(d.x - c.bx, d.y - c.by, d.z - c.bz);
    *sure = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z)) < limit;
  }
  return d;
}

// Squared distance as centre_dist() squares it (IEEE, not contracted).
__device__ __forceinline__ float square(float3 d) {
#pragma clang fp contract(off)
  return d.x * d.x + d.y * d.y + d.z * d.z;
}

// should_prune() for an image-shifted query.
__device__ __forceinline__ bool outside(const Child& c, float x, float y, float z, float r2) {
#pragma clang fp contract(off)
  const float dx = fmaxf(fmaxf(c.lx - x, x - c.hx), 0.0f);
  const float dy = fmaxf(fmaxf(c.ly - y, y - c.hy), 0.0f);
  const float dz = fmaxf(fmaxf(c.lz - z, z - c.hz), 0.0f);
  return dx * dx + dy * dy + dz * dz > r2;
}

// Wave-coherent form of the reference's per-query DFS
// (src/sbh_ffi.cu:1950-2144): the 64 queries of a wave share one stack of
// (opened node, lanes that opened it).  Popping an entry fetches the node's 8
// children at once, one per lane, which derives what is common to the wave
// (squared MAC bounds, cell box, image shift) and leaves it in LDS; each child
// is then tested by the lanes of the entry, which skip it (empty, pruned), use
// it (far field; a leaf is summed exactly) or open it.  The MAC decision is
// that of the reference's expression dist / diameter >= beta in IEEE fp32: the
// squared bounds stand 2^-14 to either side, and a lane between them evaluates
// the expression itself; likewise a displacement that may not be the minimum
// image falls back to min_image_floor.
//
// kParts, kSplitParts: every query keeps kAccs partial sums, combined in a fixed
// order at the end.  A node of level split_level, with all below it, belongs to one of them by
// its child slot, and so does each node above (for its own far field or leaf
// sum).  Each partial sum adds up in traversal order; a traversal restricted
// to an ancestor-closed subset keeps its order, so a query's result depends
// on the tree and on itself alone, bit for bit, not on the other lanes.  It
// is the same for both: with kSplitParts kAccs waves share a chunk of 64
// queries, all of them walk the levels above split_level, and each takes the
// subtrees and nodes of its own partial sum.  Queries run in Morton order
// (order[t]) so that the lanes of a wave share most of their paths.
//
// kRunning (see running_sums()): one sum per query in the order of the
// reference's DFS, the last child first, each with all below it before the next.
// An opened child is descended into at once, its parent put back with the
// children still to do, which costs the parent's fetch again.
//
// Bound by VALU issue where chunks fill the chip (the walk of a short-range
// force tests 2000 children per chunk, a quarter of the lanes of which then use
// each one), by the latency of the node fetches and by the longest chunk where
// they do not.  Measured against one popped node at a time, tested through the
// quotient, and one wave per chunk: softened walk of 100,003 Plummer points at
// depth 7 12.8 -> 4.5 ms, its VJP 15.1 -> 6.2 ms; periodic short-range walk of
// 128^3 particles 15.5 -> 11.8 ms.  Tried and dropped: deciding MAC and prune in the
// fetching lanes for the whole bounding box of the chunk (16.9 -> 15.9 ms for the
// pair of walks while every wave walked everything, but 13.4 -> 18.3 ms for the
// short-range walk, whose chunks are wider than its cells), splitting only
// the leaves' points between waves (16.9 against 13.3 ms), runs of 8 points
// (106 scalar registers, 15.9 against 13.3 ms).
// PER, CUT: periodicity and attenuation as template arguments: the walk without
// them carries no such arithmetic, and no branch inside a run of points keeps
// its loads from being issued together (same bits either way).
template <int KIND, bool PER, bool CUT, WalkSums SUMS>
__global__ __launch_bounds__(kB) __attribute__((amdgpu_waves_per_eu(
    KIND == kSoftVjp ? 5 : KIND == kSoftForce ? 6 : 8))) void k_walk8(const Leaf3* __restrict__ leaf,
                                              const Node8* __restrict__ nodes,
                                              const float* __restrict__ queries,
                                              const float* __restrict__ cot, int64_t nq,
                                              const uint32_t* __restrict__ order,
                                              float* __restrict__ out, WalkParams P,
                                              uint32_t num_nodes, uint32_t num_leaves,
                                              uint32_t split_level) {
  constexpr bool kScalar = o8::kScalarKind<KIND>;
  constexpr int kVec = kScalar ? 1 : 3;
  constexpr bool SPLIT = SUMS == kSplitParts, RUNNING = SUMS == kRunning;
  constexpr int kHeld = SUMS == kParts ? kAccs : 1;  // partial sums a wave holds
  static_assert(!SPLIT || kB / 64 == kAccs, "a split chunk is one block");
  P.periodic = PER ? 1 : 0;
  __shared__ uint32_t s_node[kB / 64][kWStack];
  __shared__ uint64_t s_lanes[kB / 64][kWStack];
  // partial sum of a deep node (and all below it), else kAccs; RUNNING: mask of
  // the children to do
  __shared__ uint8_t s_key[kB / 64][kWStack];
  __shared__ Child s_child[kB / 64][8];
  __shared__ float s_sum[SPLIT ? kAccs - 1 : 1][kVec][64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t chunk = SPLIT ? static_cast<int64_t>(blockIdx.x)
                              : static_cast<int64_t>(blockIdx.x) * (kB / 64) + w;
  const int64_t t = chunk * 64 + lane;
  const bool valid = t < nq;
  const int64_t q = !valid ? 0 : (order != nullptr ? static_cast<int64_t>(order[t]) : t);
  float qx = 0.f, qy = 0.f, qz = 0.f, gx = 0.f, gy = 0.f, gz = 0.f;
  if (valid) {
    qx = queries[3 * q + 0];
    qy = queries[3 * q + 1];
    qz = queries[3 * q + 2];
    if constexpr (KIND == kSoftVjp) {
      gx = cot[3 * q + 0];
      gy = cot[3 * q + 1];
      gz = cot[3 * q + 2];
    }
  }
  const uint64_t all = __ballot(valid);
  if (!SPLIT && all == 0) return;  // the whole wave is past the end
  const float limit = P.box * (0.5f - 1e-5f);
  // sum: the partial sum in use, number cur (SPLIT: the wave's own); the
  // others rest in acc
  float sum[3] = {}, acc[kHeld][3] = {};
  uint32_t cur = SPLIT ? w : 0;
  auto use_sum = [&](uint32_t k) {
    if (kHeld == 1 || k == cur) return;
#pragma unroll
    for (uint32_t m = 0; m < kHeld; ++m)
      if (cur == m)
        for (int a = 0; a < kVec; ++a) acc[m][a] = sum[a];
#pragma unroll
    for (uint32_t m = 0; m < kHeld; ++m)
      if (k == m)
        for (int a = 0; a < kVec; ++a) sum[a] = acc[m][a];
    cur = k;
  };
  uint32_t* stk_node = s_node[w];
  uint64_t* stk_lanes = s_lanes[w];
  uint8_t* stk_key = s_key[w];
  Child* slab = s_child[w];
  // the wave's first query picks the image shifts
  const float rx = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(qx)));
  const float ry = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(qy)));
  const float rz = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(qz)));
  int top = 0;
  if (all != 0) {
    if (lane == 0) {
      stk_node[0] = kRootEntry;
      stk_lanes[0] = all;
      stk_key[0] = RUNNING ? 0xff : kAccs;
    }
    top = 1;
  }
  __builtin_amdgcn_wave_barrier();
  while (top > 0) {
    --top;
    const uint32_t id = __builtin_amdgcn_readfirstlane(stk_node[top]);
    // the entry's lanes as a scalar mask
    const uint64_t entry_lanes = stk_lanes[top];
    const uint32_t lanes_lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(entry_lanes));
    const uint32_t lanes_hi =
        __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(entry_lanes >> 32));
    const uint64_t lanes = static_cast<uint64_t>(lanes_hi) << 32 | lanes_lo;
    const uint32_t key = __builtin_amdgcn_readfirstlane(stk_key[top]);
    // the children, one per lane
    bool have = false;
    if (lane < 8) {
      uint32_t ch = 0;
      have = lane == 0 && num_nodes > 0;
      if (id != kRootEntry) {
        ch = nodes[id].child[lane];
        have = ((nodes[id].child_mask >> lane) & 1) != 0 && ch < num_nodes;
      }
      if (have) {
        const Node8* nd = nodes + ch;
        Child c;
        c.mass = nd->contrib.mass;
        have = c.mass != 0.0f;
        c.cx = nd->cx;
        c.cy = nd->cy;
        c.cz = nd->cz;
        c.px = nd->contrib.pos[0];
        c.py = nd->contrib.pos[1];
        c.pz = nd->contrib.pos[2];
        c.id = ch;
        c.start = nd->start;
        c.end = nd->end < num_leaves ? nd->end : num_leaves;
        c.is_leaf = nd->is_leaf;
        c.deep = nd->depth >= split_level;
        c.key = key < kAccs ? key : key_of(lane);
        if (SPLIT && c.deep && c.key != static_cast<uint32_t>(w)) have = false;
        // (beta diameter)^2 and 2^-14 to either side; outside the range where
        // the square is exact to a few ulp, every lane evaluates the quotient
        const float r = P.beta * nd->diameter, r2 = r * r;
        const bool plain = r2 > 1e-30f && r2 < 1e30f;
        c.open2 = P.beta < 0.0f ? -1.0f : plain ? r2 * (1.0f - 6.1035156e-5f) : NAN;
        c.far2 = P.beta < 0.0f ? -1.0f : plain ? r2 * (1.0f + 6.1035156e-5f) : NAN;
        if constexpr (o8::kPrunedKind<KIND>) {
#pragma clang fp contract(off)
          const float h = nd->half_size;
          c.lx = c.cx - h;
          c.ly = c.cy - h;
          c.lz = c.cz - h;
          c.hx = c.cx + h;
          c.hy = c.cy + h;
          c.hz = c.cz + h;
        }
        if constexpr (PER) {
#pragma clang fp contract(off)
          const float kx = floorf((rx - c.cx) * P.inv_box + 0.5f);
          const float ky = floorf((ry - c.cy) * P.inv_box + 0.5f);
          const float kz = floorf((rz - c.cz) * P.inv_box + 0.5f);
          const bool small = fabsf(kx) <= 16.0f && fabsf(ky) <= 16.0f && fabsf(kz) <= 16.0f;
          c.bx = small ? P.box * kx : INFINITY;
          c.by = P.box * ky;
          c.bz = P.box * kz;
        }
        slab[lane] = c;
      }
    }
    uint32_t todo = static_cast<uint32_t>(__ballot(have)) & (RUNNING ? key : 0xffu);
    __builtin_amdgcn_wave_barrier();
    while (todo != 0) {
      const int slot = RUNNING ? 31 - __builtin_clz(todo) : __builtin_ctz(todo);
      todo &= ~(1u << slot);
      const Child c = slab[slot];
      const uint32_t own = __builtin_amdgcn_readfirstlane(c.key);
      const bool ours = !SPLIT || own == static_cast<uint32_t>(w);
      bool sure;
      const float3 d = wave_delta<PER>(qx, qy, qz, c.cx, c.cy, c.cz, c, limit, &sure);
      const bool all_sure = !PER || (lanes & __ballot(!sure)) == 0;
      // the lanes that do not prune the child
      uint64_t use = lanes;
      if constexpr (o8::kPrunedKind<KIND>) {
        if (P.prune) {
          if (all_sure) {
#pragma clang fp contract(off)
            use &= ~__ballot(PER ? outside(c, qx - c.bx, qy - c.by, qz - c.bz, P.r_cut_sq)
                                 : outside(c, qx, qy, qz, P.r_cut_sq));
          } else {
            use &= ~__ballot(should_prune(nodes + c.id, qx, qy, qz, P));
          }
          if (use == 0) continue;
        }
      }
      if (__builtin_amdgcn_readfirstlane(c.is_leaf) != 0) {
        // a leaf always takes the far branch: the exact sum of its points
        if (!ours) continue;
        use_sum(own);
        const uint32_t j1 = __builtin_amdgcn_readfirstlane(c.end);
        uint32_t j = __builtin_amdgcn_readfirstlane(c.start);
        if (__builtin_amdgcn_inverse_ballot_w64(use)) {
          auto run = [&](auto count, uint32_t j0) {
            constexpr int kCount = decltype(count)::value;
            Leaf3 r[kCount];
#pragma unroll
            for (int u = 0; u < kCount; ++u) r[u] = sload_leaf3(leaf, j0 + u);
#pragma unroll
            for (int u = 0; u < kCount; ++u) {
              if constexpr (kScalar) {
                contribution<KIND>(r[u], qx, qy, qz, gx, gy, gz, P, sum[0], sum[1], sum[2]);
              } else {
                bool ok;
                float3 e = wave_delta<PER>(qx, qy, qz, r[u].pos[0], r[u].pos[1], r[u].pos[2], c,
                                           limit, &ok);
                if (PER && __ballot(!ok) != 0)
                  e = make_float3(
                      min_image_floor(qx - r[u].pos[0], 1, P.box, P.inv_box),
                      min_image_floor(qy - r[u].pos[1], 1, P.box, P.inv_box),
                      min_image_floor(qz - r[u].pos[2], 1, P.box, P.inv_box));
                o8::pair_terms<KIND, CUT>(e.x, e.y, e.z, r[u].mass, gx, gy, gz, P, sum[0],
                                          sum[1], sum[2]);
              }
            }
          };
          for (; j + kRun <= j1; j += kRun) run(std::integral_constant<int, kRun>{}, j);
          if (j + 2 <= j1) {
            run(std::integral_constant<int, 2>{}, j);
            j += 2;
          }
          if (j < j1) run(std::integral_constant<int, 1>{}, j);
        }
        continue;
      }
      uint64_t far;
      if (all_sure) {
        const float d2 = square(d);
        far = __ballot(d2 >= c.far2);
        const uint64_t between = use & ~far & ~__ballot(d2 < c.open2);
        if (between != 0)
          far |= between & __ballot(use_far_field(nodes + c.id, qx, qy, qz, P));
      } else {
        far = __ballot(use_far_field(nodes + c.id, qx, qy, qz, P));
      }
      far &= use;
      if (far != 0 && ours) {
        use_sum(own);
        if (__builtin_amdgcn_inverse_ballot_w64(far)) {
          if constexpr (kScalar) {
            contribution<KIND>(nodes[c.id].contrib, qx, qy, qz, gx, gy, gz, P, sum[0], sum[1],
                               sum[2]);
          } else {
            bool ok;
            float3 e = wave_delta<PER>(qx, qy, qz, c.px, c.py, c.pz, c, limit, &ok);
            if (PER && __ballot(!ok) != 0)
              e = make_float3(min_image_floor(qx - c.px, 1, P.box, P.inv_box),
                              min_image_floor(qy - c.py, 1, P.box, P.inv_box),
                              min_image_floor(qz - c.pz, 1, P.box, P.inv_box));
            o8::pair_terms<KIND, CUT>(e.x, e.y, e.z, c.mass, gx, gy, gz, P, sum[0], sum[1],
                                      sum[2]);
          }
        }
      }
      const uint64_t open = use & ~far;
      if (RUNNING && open != 0 && todo != 0 && top < kWStack) {
        if (lane == 0) {
          stk_node[top] = id;
          stk_lanes[top] = lanes;
          stk_key[top] = static_cast<uint8_t>(todo);
        }
        ++top;
        todo = 0;
      }
      if (open != 0 && top < kWStack) {
        if (lane == 0) {
          stk_node[top] = c.id;
          stk_lanes[top] = open;
          stk_key[top] = static_cast<uint8_t>(RUNNING ? 0xff : c.deep ? own : kAccs);
        }
        ++top;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  float r[kVec];
  if constexpr (SPLIT) {
    if (w > 0)
      for (int a = 0; a < kVec; ++a) s_sum[w - 1][a][lane] = sum[a];
    __syncthreads();
    if (w > 0 || !valid) return;
    for (int a = 0; a < kVec; ++a)
      r[a] = (sum[a] + s_sum[0][a][lane]) + (s_sum[1][a][lane] + s_sum[2][a][lane]);
  } else if constexpr (RUNNING) {
    if (!valid) return;
    for (int a = 0; a < kVec; ++a) r[a] = sum[a];
  } else {
    if (!valid) return;
    use_sum(0);
    for (int a = 0; a < kVec; ++a)
      r[a] = (sum[a] + acc[1 % kHeld][a]) + (acc[2 % kHeld][a] + acc[3 % kHeld][a]);
  }
  if constexpr (kScalar) {
    out[q] = r[0];
  } else {
    out[3 * q + 0] = r[0];
    out[3 * q + 1] = r[1];
    out[3 * q + 2] = r[2];
  }
}

uint64_t total_nodes8(int max_depth) {
  uint64_t total = 0, level = 1;
  for (int l = 0; l <= max_depth; ++l) {
    total += level;
    level <<= 3;
  }
  return total;
}

using o8::check_walk_common;
using o8::make_walk_params;

template <int KIND, bool SOFT, WalkSums SUMS>
auto pick_walk(const WalkParams& P) {
  constexpr bool kPer = SUMS != kRunning;  // running sums: never periodic
  if constexpr (SOFT) {
    if (P.cutoff)
      return P.periodic ? k_walk8<KIND, kPer, true, SUMS> : k_walk8<KIND, false, true, SUMS>;
  }
  return P.periodic ? k_walk8<KIND, kPer, false, SUMS> : k_walk8<KIND, false, false, SUMS>;
}

int tree_depth(uint32_t num_nodes) {
  int depth = 0;
  while (depth < 10 && total_nodes8(depth) < num_nodes) ++depth;
  return depth;
}

// Level whose nodes the partial sums divide: two above the leaves, so that a
// query's neighbourhood spreads over all sums while few nodes lie above.
uint32_t split_level(int depth) { return static_cast<uint32_t>(depth > 3 ? depth - 2 : 1); }

// Whether a query's contributions go to one running sum (kRunning): large clouds
// in trees of few levels, whose full leaves give a query 1e5 terms and more.  A
// running sum loses terms below half an ulp of it, partial sums fewer of them:
// they are up to five times closer to 64 bits there, but move a force by 5e-5
// from what the reference's order gives (Plummer sphere of 262,144 points,
// depth 5, cutoff 0.5; 3e-5 at depth 6, 1.3e-5 at depth 7; without cutoff 1.8e-5,
// 1e-5 and 8e-6), and callers compare with that order.  From 98,304 points on at
// depth 5 (half as many more per level, twice as many without cutoff, whose tail
// of small terms is missing) the difference passes 1e-5: running sums, which give
// the same as the walk of one query after another to 3e-7.  Below, and in periodic
// boxes (short sums, 5e-7), partial sums: forces and VJP of 65,537 points at
// depth 6 with cutoff 9.4 ms against 15.5.  Above, little is lost: 150,001 points at
// depth 5 54 ms against 43, 262,144 126 against 123 (134 and 293 with a node
// at a time).  The rule looks at the tree alone, so that a query's bits do not
// depend on how many are asked.
bool running_sums(const WalkParams& P, uint32_t num_leaves, int depth) {
  if (P.periodic) return false;
  double line = P.cutoff ? 98304.0 : 196608.0;
  for (int d = 5; d < depth; ++d) line *= 1.5;
  for (int d = 5; d > depth; --d) line /= 1.5;
  return num_leaves >= line;
}

// Chunks of 64 queries below which each is walked by kAccs waves: 4096 chunks
// are 4 waves per SIMD, half of what fits, and the longest chunks then hold up
// the end of the launch.
constexpr int64_t kSplitChunks = 4096;

template <int KIND>
int launch_walk(void* stream, const SbhBuffer* leaf_bytes, const SbhBuffer* node_bytes,
                const SbhBuffer* queries, const SbhBuffer* cot, SbhBuffer* out,
                const WalkParams& P) {
  int64_t nq = queries->dims[0];
  if (nq == 0) return SBH_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint32_t* order = nullptr;
  // (not while the stream is captured: the ordering scratch may need an
  // allocation, and the unordered walk gives the same results)
  if (nq >= o8::kOrderMin && !stream_capturing(s)) {
    char* ws = static_cast<char*>(workspace(s, kWsWalk, tree::query_order_bytes(nq)));
    if (ws == nullptr) return fail_internal_msg("workspace allocation failed");
    int rc = tree::query_order(s, static_cast<const float*>(queries->data), nq, ws, &order);
    if (rc != SBH_OK) return rc;
  }
  const auto num_nodes = static_cast<uint32_t>(byte_count(node_bytes) / sizeof(Node8));
  const auto num_leaves = static_cast<uint32_t>(byte_count(leaf_bytes) / sizeof(Leaf3));
  const int depth = tree_depth(num_nodes);
  const bool running = running_sums(P, num_leaves, depth);
  const bool split = !running && (nq + 63) / 64 < kSplitChunks;
  constexpr bool kSoft = o8::kPrunedKind<KIND>;
  auto* walk = running ? pick_walk<KIND, kSoft, kRunning>(P)
               : split ? pick_walk<KIND, kSoft, kSplitParts>(P)
                       : pick_walk<KIND, kSoft, kParts>(P);
  walk<<<split ? grid_for(nq, 64) : grid_for(nq, kB), kB, 0, s>>>(
      static_cast<const Leaf3*>(leaf_bytes->data), static_cast<const Node8*>(node_bytes->data),
      static_cast<const float*>(queries->data),
      cot ? static_cast<const float*>(cot->data) : nullptr, nq, order,
      static_cast<float*>(out->data),
      P, num_nodes, num_leaves, split_level(depth));
  SBH_LAUNCH_CHECK();
  return SBH_OK;
}

}  // namespace
}  // namespace sbh

using namespace sbh;

extern "C" int sbh_build_octree8_buffers(void* stream, const SbhBuffer* points,
                                         const SbhBuffer* normals, const SbhBuffer* masses,
                                         const SbhBuffer* min_corner,
                                         const SbhBuffer* max_corner, SbhBuffer* leaf_out,
                                         SbhBuffer* node_out, SbhBuffer* contrib_out,
                                         int32_t max_depth) {
  clear_error();
  if (!buffer_ok(points, SBH_DTYPE_F32, 2) || points->dims[1] != 3)
    return fail_invalid("points must have shape (N, 3)");
  if (!buffer_ok(normals, SBH_DTYPE_F32, 2) || normals->dims[1] != 3)
    return fail_invalid("normals must have shape (N, 3)");
  if (points->dims[0] != normals->dims[0]) return fail_invalid("points/normals row mismatch");
  if (!buffer_ok(masses, SBH_DTYPE_F32, 1) || masses->dims[0] != points->dims[0])
    return fail_invalid("masses must have shape (N,)");
  if (!buffer_ok(min_corner, SBH_DTYPE_F32, 1) || min_corner->dims[0] != 3 ||
      !buffer_ok(max_corner, SBH_DTYPE_F32, 1) || max_corner->dims[0] != 3)
    return fail_invalid("min_corner/max_corner must have shape (3,)");
  if (max_depth < 1 || max_depth > 10) return fail_invalid("max_depth must be in [1, 10]");
  int64_t n = points->dims[0];
  uint64_t total = total_nodes8(max_depth);
  if (!buffer_ok(leaf_out, SBH_DTYPE_U8, -1) ||
      byte_count(leaf_out) != n * static_cast<int64_t>(sizeof(Leaf3)))
    return fail_invalid("leaf_out size mismatch");
  if (!buffer_ok(node_out, SBH_DTYPE_U8, -1) ||
      byte_count(node_out) != static_cast<int64_t>(total * sizeof(Node8)))
    return fail_invalid("node_out size mismatch");
  if (!buffer_ok(contrib_out, SBH_DTYPE_U8, -1) ||
      byte_count(contrib_out) != static_cast<int64_t>(total * sizeof(Leaf3)))
    return fail_invalid("contrib_out size mismatch");
  if (n > INT32_MAX) return fail_invalid("too many points");

  hipStream_t s = static_cast<hipStream_t>(stream);
  // Bounds are read back like the reference does (src/sbh_ffi.cu:1111-1126)
  // so that an empty span is reported as an argument error.
  float h[6];
  SBH_HIP_TRY(hipMemcpyAsync(h, min_corner->data, 3 * sizeof(float), hipMemcpyDeviceToHost, s));
  SBH_HIP_TRY(hipMemcpyAsync(h + 3, max_corner->data, 3 * sizeof(float), hipMemcpyDeviceToHost, s));
  SBH_HIP_TRY(hipStreamSynchronize(s));
  BuildGeom g;
  g.min_x = h[0];
  g.min_y = h[1];
  g.min_z = h[2];
  g.span = fmaxf(fmaxf(h[3] - h[0], h[4] - h[1]), h[5] - h[2]);
  if (!(g.span > 0.0f)) return fail_invalid("invalid bounds span");
  g.cx = h[0] + g.span * 0.5f;
  g.cy = h[1] + g.span * 0.5f;
  g.cz = h[2] + g.span * 0.5f;
  g.half_size = g.span * 0.5f;

  // Workspace: keys/vals x2, sort temp, sums of the cells between two launches
  // (levels max_depth - kSpan, max_depth - 2 kSpan, ...).
  size_t nn = static_cast<size_t>(n > 0 ? n : 1);
  size_t off_codes = 0;
  size_t off_idx = off_codes + nn * 4;
  size_t off_codes2 = off_idx + nn * 4;
  size_t off_perm = off_codes2 + nn * 4;
  size_t off_sort = (off_perm + nn * 4 + 255) & ~size_t{255};
  size_t ws_bytes = off_sort + ((order_temp_bytes(n) + 255) & ~size_t{255});
  size_t off_cells[4] = {};
  for (int k = 0, l = max_depth - kSpan; l > 0; l -= kSpan, ++k) {
    off_cells[k] = ws_bytes;
    ws_bytes += ((size_t{1} << (3 * l)) * sizeof(CellSums) + 255) & ~size_t{255};
  }
  char* ws = nullptr;
  if (int rcw = cached_workspace(s, kWsBuild, ws_bytes, &ws); rcw != SBH_OK) return rcw;
  auto* codes = reinterpret_cast<uint32_t*>(ws + off_codes);
  auto* pp = static_cast<const float*>(points->data);
  auto* leaf = static_cast<Leaf3*>(leaf_out->data);
  const uint32_t* codes_sorted = nullptr;
  if (n > 0) {
    k_codes<<<grid_for(n, kB), kB, 0, s>>>(pp, n, g, max_depth, codes);
    SBH_LAUNCH_CHECK();
    const uint32_t* perm = nullptr;
    int rc = order_by_key(s, codes, n, 3 * max_depth, reinterpret_cast<uint32_t*>(ws + off_idx),
                          reinterpret_cast<uint32_t*>(ws + off_codes2),
                          reinterpret_cast<uint32_t*>(ws + off_perm), ws + off_sort,
                          &codes_sorted, &perm);
    if (rc != SBH_OK) return rc;
    k_leaf_gather<<<grid_for(n, kB), kB, 0, s>>>(pp, static_cast<const float*>(normals->data),
                                                 static_cast<const float*>(masses->data), n,
                                                 perm, leaf);
    SBH_LAUNCH_CHECK();
  }
  auto* nodes = static_cast<Node8*>(node_out->data);
  auto* contrib = static_cast<Leaf3*>(contrib_out->data);
  // records beyond the 256 MB of the last cache (depth 7 and up) pass it by: depth 8
  // 3.84 -> 3.32 ms, depth 7 the same
  const bool past = total * (sizeof(Node8) + sizeof(Leaf3)) > (uint64_t{256} << 20);
  const CellSums* down = nullptr;
  for (int k = 0, l = max_depth;; ++k) {
    const int span = l < kSpan ? l : kSpan;
    const unsigned blocks = 1u << (3 * (l - span));
    auto* up = l > span ? reinterpret_cast<CellSums*>(ws + off_cells[k]) : nullptr;
    if (k == 0)
      k_subtree<true><<<blocks, kB, 0, s>>>(codes_sorted, leaf, n, nullptr, up, l, span, max_depth,
                                            g, past, nodes, contrib);
    else
      k_subtree<false><<<blocks, kB, 0, s>>>(nullptr, leaf, n, down, up, l, span, max_depth, g,
                                             past, nodes, contrib);
    SBH_LAUNCH_CHECK();
    if (l == span) break;
    down = up;
    l -= span;
  }
  return SBH_OK;
}

extern "C" int sbh_barnes_hut_force_octree8(void* stream, const SbhBuffer* leaf_bytes,
                                            const SbhBuffer* node_bytes,
                                            const SbhBuffer* queries, SbhBuffer* out,
                                            float beta, int32_t periodic, float box_length,
                                            int32_t threads) {
  clear_error();
  int rc = check_walk_common(leaf_bytes, node_bytes, queries, out, threads);
  if (rc != SBH_OK) return rc;
  WalkParams P = make_walk_params(beta, 0.0f, 0.0f, 0, 0.0f, periodic, box_length);
  return launch_walk<kGravGrad>(stream, leaf_bytes, node_bytes, queries, nullptr, out, P);
}

// Winding numbers over octree8 records built from oriented area elements
// (points = element centroids, normals = unit normals, masses = areas): the
// classic vote walk of src/sbh_gpu.cu:100-120 with signedSolidAngle<3>,
// include/kernel.h:73-80.  out: (M,).
extern "C" int sbh_barnes_hut_wn_octree8(void* stream, const SbhBuffer* leaf_bytes,
                                         const SbhBuffer* node_bytes, const SbhBuffer* queries,
                                         SbhBuffer* out, float beta, int32_t threads) {
  clear_error();
  int rc = check_walk_common(leaf_bytes, node_bytes, queries, out, threads, true);
  if (rc != SBH_OK) return rc;
  WalkParams P = make_walk_params(beta, 0.0f, 0.0f, 0, 0.0f, 0, 1.0f);
  return launch_walk<o8::kWinding>(stream, leaf_bytes, node_bytes, queries, nullptr, out, P);
}

// Potential -m / (r + 0.1) (gravityPotential, include/kernel.h:55-60) over
// octree8 records: the classic walk of src/sbh_gpu.cu:79-98, 324-361
// (evalBarnesHut_gravity).  out: (M,).
extern "C" int sbh_barnes_hut_potential_octree8(void* stream, const SbhBuffer* leaf_bytes,
                                                const SbhBuffer* node_bytes,
                                                const SbhBuffer* queries, SbhBuffer* out,
                                                float beta, int32_t threads) {
  clear_error();
  int rc = check_walk_common(leaf_bytes, node_bytes, queries, out, threads, true);
  if (rc != SBH_OK) return rc;
  WalkParams P = make_walk_params(beta, 0.0f, 0.0f, 0, 0.0f, 0, 1.0f);
  return launch_walk<o8::kPotential>(stream, leaf_bytes, node_bytes, queries, nullptr, out, P);
}

// Smooth distance field sum exp(-alpha r) (smoothDistExp, include/kernel.h:
// 82-87) over octree8 records (alpha = 1 in every record, as the builder of
// src/sbh_ffi.cu:1741, 1860 writes): src/sbh_gpu.cu:122-141, 400-434
// (evalBarnesHut_smoothdist).  out: (M,).
extern "C" int sbh_barnes_hut_smoothdist_octree8(void* stream, const SbhBuffer* leaf_bytes,
                                                 const SbhBuffer* node_bytes,
                                                 const SbhBuffer* queries, SbhBuffer* out,
                                                 float beta, int32_t threads) {
  clear_error();
  int rc = check_walk_common(leaf_bytes, node_bytes, queries, out, threads, true);
  if (rc != SBH_OK) return rc;
  WalkParams P = make_walk_params(beta, 0.0f, 0.0f, 0, 0.0f, 0, 1.0f);
  return launch_walk<o8::kSmoothDist>(stream, leaf_bytes, node_bytes, queries, nullptr, out, P);
}

extern "C" int sbh_barnes_hut_force_octree8_soft(
    void* stream, const SbhBuffer* leaf_bytes, const SbhBuffer* node_bytes,
    const SbhBuffer* queries, SbhBuffer* out, float beta, float softening_scale,
    float cutoff_scale, int32_t prune_enabled, float prune_r_cut_mult, int32_t periodic,
    float box_length, int32_t threads) {
  clear_error();
  int rc = check_walk_common(leaf_bytes, node_bytes, queries, out, threads);
  if (rc != SBH_OK) return rc;
  if (prune_enabled != 0 && prune_r_cut_mult <= 0.0f)
    return fail_invalid("prune_r_cut_mult must be > 0 when prune_enabled is set");
  WalkParams P = make_walk_params(beta, softening_scale, cutoff_scale, prune_enabled,
                                  prune_r_cut_mult, periodic, box_length);
  return launch_walk<kSoftForce>(stream, leaf_bytes, node_bytes, queries, nullptr, out, P);
}

extern "C" int sbh_barnes_hut_force_octree8_soft_vjp(
    void* stream, const SbhBuffer* leaf_bytes, const SbhBuffer* node_bytes,
    const SbhBuffer* queries, const SbhBuffer* cotangent, SbhBuffer* out, float beta,
    float softening_scale, float cutoff_scale, int32_t prune_enabled, float prune_r_cut_mult,
    int32_t periodic, float box_length, int32_t threads) {
  clear_error();
  int rc = check_walk_common(leaf_bytes, node_bytes, queries, out, threads);
  if (rc != SBH_OK) return rc;
  if (!buffer_ok(cotangent, SBH_DTYPE_F32, 2) || cotangent->dims[0] != queries->dims[0] ||
      cotangent->dims[1] != 3)
    return fail_invalid("cotangent shape mismatch");
  if (prune_enabled != 0 && prune_r_cut_mult <= 0.0f)
    return fail_invalid("prune_r_cut_mult must be > 0 when prune_enabled is set");
  WalkParams P = make_walk_params(beta, softening_scale, cutoff_scale, prune_enabled,
                                  prune_r_cut_mult, periodic, box_length);
  return launch_walk<kSoftVjp>(stream, leaf_bytes, node_bytes, queries, cotangent, out, P);
}
