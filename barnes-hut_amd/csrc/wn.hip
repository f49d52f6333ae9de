// Winding numbers of an oriented-area (dipole) cloud on the adaptive octree.
//
// Sources are area elements (centroid p, unit normal n, area a); the value at
// q is sum a n.(p - q) / (4 pi (|p - q|^3 + 1e-5)) (signedSolidAngle<3>,
// include/kernel.h:73-80).  The tree is built over the centroids with the
// areas as weights (tree::build: area-weighted centroid c and area A per
// node), then per node the dipole D = sum a n, so an accepted node counts as
// the dipole D at c -- the reference's node record (A, D / A) at c
// (src/sbh_gpu.cu:100-120 with src/sbh_ffi.cu:1840-1868).  A first-moment
// (sum a n (p - c)^T) correction was tried and rejected: for smooth surface
// patches at the MAC distance the next Taylor term is larger and of opposite
// sign, so the truncated series is less accurate than the dipole alone.
//
// Queries are a separate cloud with a tree of their own (topology only, in
// their own cube); its cell groups of <= 64 queries (one team of waves each) are
// walked against the element tree with the group MAC and traversal of the
// gravity walk.  (Plain runs of 64 Morton-sorted queries are not used: runs
// that cross a coarse cell boundary have boxes spanning much of the domain
// and accept almost nothing.)
#include "common.hpp"
#include "profile.hpp"
#include "groupwalk.hpp"
#include "tree.hpp"

namespace sbh {
namespace tree {
namespace {

using namespace gw;

constexpr float kInvFourPi = 0.07957747154594767f;
constexpr int kQueryDepth = kQueryTreeDepth;
constexpr int kQueryLeaf = kQueryTreeLeaf;

struct WnLayout {
  Layout t;      // element tree, at the workspace base
  size_t wd;     // per element-tree node: dipole (float4)
  size_t qbase;  // query tree, at workspace + qbase
  Layout qt;
  size_t total;
};

WnLayout wn_layout(int64_t n, int64_t m, int max_depth, int leaf_size) {
  auto align = [](size_t x) { return (x + 255) & ~size_t{255}; };
  WnLayout W;
  W.t = layout(n, max_depth, leaf_size);
  const size_t cap = static_cast<size_t>(W.t.cap) + 1;
  size_t o = W.t.total;
  W.wd = o; o = align(o + 16 * cap);
  W.qbase = o;
  W.qt = layout(m, kQueryDepth, kQueryLeaf);
  W.total = W.qbase + W.qt.total;
  return W;
}

// The dipoles are computed by the tree build's moment pass (tree::build with
// a dipole array), which also clears the sentinel node's entry.
// ------------------------------------------------------------------ walk
struct WnArgs {
  const Header* hdr;  // element tree
  Header* qhdr;       // query tree: group count, work queue, statistics
  const int2* groups; // query groups (start, count) in sorted query order
  const int4* topo;
  const float4* geo;
  const float4* mp;   // centroid, area
  const float4* wd;   // dipole
  const float4* sp;   // sorted centroid, area
  const float4* sn;   // sorted normal
  const float4* qs;   // sorted queries
  const uint32_t* qperm;
  int m;
  int sentinel;
  float beta;
  float* out;
  bool stats;
};

__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// C far nodes (sentinel-padded) against the lane's query; like the near batch
// below it returns 4 pi times the contribution (the caller scales once).
template <int C>
__device__ __forceinline__ float wn_far_batch(const WnArgs& A, float qx, float qy, float qz,
                                              const int* far) {
  float w = 0.f;
#pragma unroll
  for (int t = 0; t < C; ++t) {
    const int k = __builtin_amdgcn_readfirstlane(far[t]);
    const float4 c = sload4(A.mp, k);
    const float4 d = sload4(A.wd, k);
    const float Xx = c.x - qx, Xy = c.y - qy, Xz = c.z - qz;
    const float R2 = Xx * Xx + Xy * Xy + Xz * Xz;
    const float R = sqrt_hw(R2);
    w += (d.x * Xx + d.y * Xy + d.z * Xz) * rcp(fmaf(R, R2, 1e-5f));
  }
  return w;
}

// kChunk consecutive elements of one leaf from j0 (with PAD, entries at or
// beyond s1 carry zero area; without, the batch lies inside the range and
// reads its records as runs, which the scalar loads fetch 4 at a time).
template <bool PAD>
__device__ __forceinline__ float wn_near_batch(const WnArgs& A, float qx, float qy, float qz,
                                               int j0, int s1) {
  float w = 0.f;
  cfloat* rp = run_base(A.sp, j0);
  cfloat* rn = run_base(A.sn, j0);
#pragma unroll
  for (int u = 0; u < kChunk; ++u) {
    const int j = j0 + u;
    const int jj = min(j, s1 - 1);
    const float4 p = PAD ? sload4(A.sp, jj) : sload4_run(rp, u);
    const float4 nv = PAD ? sload4(A.sn, jj) : sload4_run(rn, u);
    const float a = (!PAD || j < s1) ? p.w : 0.0f;
    const float dx = p.x - qx, dy = p.y - qy, dz = p.z - qz;
    const float r2 = dx * dx + dy * dy + dz * dz;
    const float r = sqrt_hw(r2);
    w += a * (nv.x * dx + nv.y * dy + nv.z * dz) * rcp(fmaf(r, r2, 1e-5f));
  }
  return w;
}

// Elements [s0, s1) against the lane's query.
__device__ __forceinline__ float wn_range(const WnArgs& A, float qx, float qy, float qz, int s0,
                                          int s1) {
  float w = 0.f;
  int j0 = s0;
  for (; j0 + kChunk <= s1; j0 += kChunk) w += wn_near_batch<false>(A, qx, qy, qz, j0, s1);
  if (j0 < s1) w += wn_near_batch<true>(A, qx, qy, qz, j0, s1);
  return w;
}

// Walk with the TEAM waves of a block sharing each group of queries, as the
// teams of the gravity walk (tree.hip) do: the threads test candidate nodes, the
// accepted nodes and near leaves go to lists in LDS in a fixed order, and the
// lists are dealt to kShares shares in turn, each with a sum of its own,
// combined in order at the end: the values depend on tree and group alone, not
// on TEAM.
//
// Groups near the surface cost 10 times the mean and there are few groups (1e6
// queries: 17,500, two for each wave that fits the chip), so that one wave per
// group ended in a tail as long as the rest: half of the waves were done after
// 0.55 of 1.06 ms.  Whole calls, one wave per group -> teams: 204,020 elements at
// 2^20 queries 1.44 -> 1.17 ms, at 2^18 1.10 -> 0.75, at 10^4 3.0 -> 1.0, at 1000
// 19.8 -> 4.9; 1000 elements at 1000 queries 0.22 -> 0.15.
constexpr int kShares = 16;
constexpr int kWidth = 512;         // candidates tested at once
constexpr int kFarList = 1024;      // the lists are evaluated from here on
constexpr int kNearList = 256;
// Stack: a pop takes at most (kTeamSoft - top) / 7 nodes near the soft limit, so a
// push of <= 8 children each stays under kTeamStack.
constexpr int kTeamSoft = 2048;
constexpr int kTeamStack = kTeamSoft + 8 * 24;
constexpr int kLeafRun = 4;         // consecutive leaves of a share
constexpr int kBigLeaf = 128;       // a leaf of more elements is dealt 64 at a time

// Teams of 16 up to kWideQueries queries: few groups, so that each should be short
// (against teams of 8, 204,020 elements at 10^4 queries 1.03 and 1.55 ms, at 2^18 0.75
// and 0.78); above, teams of 8, which wait less at barriers (2^20: 1.17 against 1.36).
constexpr int64_t kWideQueries = int64_t{1} << 18;

template <int TEAM>
__global__ __launch_bounds__(64 * TEAM) __attribute__((amdgpu_waves_per_eu(8))) void k_wn_walk(
    WnArgs A) {
  static_assert(64 * TEAM >= kWidth && kShares % TEAM == 0, "team size");
  __shared__ int s_stack[kTeamStack];
  __shared__ int s_far[kFarList + kWidth + kChunk];
  __shared__ int2 s_near[kNearList + kWidth];
  __shared__ float s_sum[kShares][64];
  __shared__ int s_cnt[2][TEAM];
  __shared__ unsigned long long s_pairs[TEAM];  // statistics
  __shared__ int s_claim;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int num_groups = A.qhdr->num_groups, num_nodes = A.hdr->num_nodes;
  unsigned long long n_far = 0, n_groups = 0;
  if (lane == 0) s_pairs[w] = 0;
  // thread 0 claims groups, one ahead of its use: eighth by eighth from the
  // block's own XCD's on (see next_group)
  int tries = 0;
  auto claim = [&]() {
    for (; tries < 8; ++tries) {
      const int q = (static_cast<int>(blockIdx.x & 7u) + tries) & 7;
      const int2 r = eighth_range(num_groups, q);
      const int t = atomicAdd(&A.qhdr->tq[q], 1);
      if (t < r.y - r.x) return r.x + t;
    }
    return -1;
  };
  if (tid == 0) s_claim = claim();
  __syncthreads();
  while (true) {
    const int g = __builtin_amdgcn_readfirstlane(s_claim);
    if (g < 0) break;  // at most 8 failing claims: every block reaches this exit
    const int2 grp = A.groups[g];
    const int base = __builtin_amdgcn_readfirstlane(grp.x);
    const int cnt = __builtin_amdgcn_readfirstlane(grp.y);
    int next = -1;
    if (tid == 0) next = claim();
    if (cnt < 1 || cnt > 64 || base < 0 || base + cnt > A.m) {  // corrupt entry
      __syncthreads();
      if (tid == 0) s_claim = next;
      __syncthreads();
      continue;
    }
    const int i = base + (lane < cnt ? lane : 0);
    const float4 q = A.qs[i];
    const Box b = wave_box(q.x, q.y, q.z);
    for (int v = w; v < kShares; v += TEAM) s_sum[v][lane] = 0.f;
    int top = 1, nfar = 0, nnear = 0, iters = 0;
    if (tid == 0) s_stack[0] = 0;
    __syncthreads();
    while (true) {
      // (every node is pushed at most once and each round pops at least one)
      if (top > 0 && iters++ > num_nodes) top = 0;
      if (top > 0) {
        int k = min(kWidth, top);
        k = min(k, max(1, (kTeamSoft - top) / 7));
        top -= k;
        int node = -1, kind = 0, nch = 0, incl = 0;
        int4 t = make_int4(0, 0, 0, 0);
        if (w * 64 < k) {  // (waves without a candidate only keep the counts)
          node = tid < k ? s_stack[top + tid] : -1;
          const bool have = node >= 0 && node < num_nodes;
          const int nd = have ? node : 0;
          const float4 m = A.mp[nd];
          const float4 gg = A.geo[nd];
          t = A.topo[nd];
          if (have && m.w != 0.0f) {
            if (group_accept(b.lx, b.ly, b.lz, b.hx, b.hy, b.hz, gg, A.beta))
              kind = 1;
            else if (t.w == 0)
              kind = 2;
            else
              nch = t.w;
          }
          incl = wave_incl_scan(nch);
        }
        // per wave: accepted nodes | near leaves << 11; children
        const uint64_t bf = __ballot(kind == 1), bn = __ballot(kind == 2);
        if (lane == 63) {
          s_cnt[0][w] = __popcll(bf) | __popcll(bn) << 11;
          s_cnt[1][w] = incl;
        }
        __syncthreads();  // the popped entries are read, the counts written
        const int sum0 = wave_incl_scan(lane < TEAM ? s_cnt[0][lane] : 0);
        const int sum1 = wave_incl_scan(lane < TEAM ? s_cnt[1][lane] : 0);
        const int all0 = __builtin_amdgcn_readlane(sum0, TEAM - 1);
        const int pushed = __builtin_amdgcn_readlane(sum1, TEAM - 1);
        const int pre0 = w > 0 ? __builtin_amdgcn_readlane(sum0, w - 1) : 0;
        const int pre1 = w > 0 ? __builtin_amdgcn_readlane(sum1, w - 1) : 0;
        if (kind == 1) s_far[nfar + (pre0 & 2047) + lanes_below(bf)] = node;
        if (kind == 2) s_near[nnear + (pre0 >> 11) + lanes_below(bn)] = make_int2(t.x, t.y);
        nfar += all0 & 2047;
        nnear += all0 >> 11;
        if (top + pushed > kTeamStack) {  // unreachable for depth <= 10
          if (tid == 0) atomicOr(&A.qhdr->overflow, 4);
          top = 0;
        } else {
          int* dst = s_stack + (top + pre1 + incl - nch);
          for (int c = 0; c < nch; ++c) dst[c] = t.z + c;
          top += pushed;
        }
        __syncthreads();  // entries and lists written, the counts read
      }
      if (top > 0 && nfar < kFarList && nnear < kNearList) continue;
      // evaluate the lists
      const int runs = (nfar + kChunk - 1) / kChunk;
      if (tid < runs * kChunk - nfar) s_far[nfar + tid] = A.sentinel;
      __syncthreads();
      if (w == 0) n_far += static_cast<unsigned long long>(nfar) * cnt;
#pragma unroll 1
      for (int v = w; v < kShares; v += TEAM) {
        float sum = 0.f;
#pragma unroll 1
        for (int run = v; run < runs; run += kShares)
          sum += wn_far_batch<kChunk>(A, q.x, q.y, q.z, s_far + run * kChunk);
        int near = 0;
#pragma unroll 1
        for (int e0 = v * kLeafRun; e0 < nnear; e0 += kShares * kLeafRun) {
          const int e_end = min(e0 + kLeafRun, nnear);
          int e = e0;
          while (e < e_end) {
            // leaves whose elements adjoin, as one range
            const int s0 = __builtin_amdgcn_readfirstlane(s_near[e].x);
            int s1 = s0;
            do {
              const int c = __builtin_amdgcn_readfirstlane(s_near[e].y);
              if (c > kBigLeaf) break;
              s1 += c;
              ++e;
            } while (e < e_end && __builtin_amdgcn_readfirstlane(s_near[e].x) == s1);
            if (s1 == s0) {  // a large leaf (leaves are not empty): dealt below
              ++e;
              continue;
            }
            near += s1 - s0;
            sum += wn_range(A, q.x, q.y, q.z, s0, s1);
          }
        }
        // large leaves (elements that share a cell at the depth limit, or a large
        // leaf size), 64 elements at a time
#pragma unroll 1
        for (int e = 0; e < nnear; ++e) {
          const int s0 = __builtin_amdgcn_readfirstlane(s_near[e].x);
          const int s1 = s0 + __builtin_amdgcn_readfirstlane(s_near[e].y);
          if (s1 - s0 <= kBigLeaf) continue;
#pragma unroll 1
          for (int j = s0 + 64 * v; j < s1; j += 64 * kShares) {
            const int j1 = min(j + 64, s1);
            near += j1 - j;
            sum += wn_range(A, q.x, q.y, q.z, j, j1);
          }
        }
        if (lane == 0) s_pairs[w] += static_cast<unsigned long long>(near) * cnt;
        s_sum[v][lane] += sum;
      }
      nfar = nnear = 0;
      __syncthreads();  // the lists are read, the sums written
      if (top == 0) break;
    }
    if (w == 0 && lane < cnt) {
      float v = 0.f;
      for (int k = 0; k < kShares; ++k) v += s_sum[k][lane];
      A.out[A.qperm[i]] = v * kInvFourPi;
    }
    ++n_groups;
    if (tid == 0) s_claim = next;
    __syncthreads();  // the sums are read, the claim written
  }
  if (A.stats && lane == 0) {
    if (w == 0) {
      atomicAdd(&A.qhdr->stats[0], n_far);
      atomicAdd(&A.qhdr->stats[2], n_groups);
    }
    atomicAdd(&A.qhdr->stats[1], s_pairs[w]);
  }
}

__global__ void k_wn_copy_stats(const Header* __restrict__ hdr, const Header* __restrict__ qhdr,
                                int64_t* __restrict__ out) {
  if (threadIdx.x != 0) return;
  out[0] = static_cast<int64_t>(qhdr->stats[0]);
  out[1] = static_cast<int64_t>(qhdr->stats[1]);
  out[2] = static_cast<int64_t>(qhdr->stats[2]);
  out[3] = hdr->num_nodes;
  int levels = 0;
  for (int l = 0; l < kMaxLevels; ++l)
    if (hdr->level_count[l] > 0) levels = l + 1;
  out[4] = levels;
  out[5] = hdr->overflow | qhdr->overflow;
  out[6] = 0;
  out[7] = 0;
}

int check_wn(const SbhBuffer* points, const SbhBuffer* normals, const SbhBuffer* areas,
             const SbhBuffer* queries, const SbhBuffer* out, float beta, int max_depth,
             int leaf_size) {
  if (!buffer_ok(points, SBH_DTYPE_F32, 2) || points->dims[1] != 3)
    return fail_invalid("points must have shape (N, 3)");
  const int64_t n = points->dims[0];
  if (!buffer_ok(normals, SBH_DTYPE_F32, 2) || normals->dims[0] != n || normals->dims[1] != 3)
    return fail_invalid("normals must have shape (N, 3)");
  if (!buffer_ok(areas, SBH_DTYPE_F32, 1) || areas->dims[0] != n)
    return fail_invalid("areas must have shape (N,)");
  if (!buffer_ok(queries, SBH_DTYPE_F32, 2) || queries->dims[1] != 3)
    return fail_invalid("queries must have shape (M, 3)");
  if (!buffer_ok(out, SBH_DTYPE_F32, 1) || out->dims[0] != queries->dims[0])
    return fail_invalid("out must have shape (M,)");
  if (n > (int64_t{1} << 30) || queries->dims[0] > (int64_t{1} << 30))
    return fail_invalid("too many points");
  if (!(beta >= 0.0f)) return fail_invalid("beta must be >= 0");
  if (max_depth < 1 || max_depth > 10) return fail_invalid("max_depth must be in [1, 10]");
  if (leaf_size < 1) return fail_invalid("leaf_size must be >= 1");
  return SBH_OK;
}

}  // namespace

}  // namespace tree
}  // namespace sbh

using namespace sbh;

extern "C" int64_t sbh_winding_number_workspace_bytes(int64_t num_elements, int64_t num_queries,
                                                      int32_t max_depth, int32_t leaf_size) {
  if (num_elements < 0 || num_queries < 0 || max_depth < 1 || max_depth > 10 || leaf_size < 1)
    return -1;
  return static_cast<int64_t>(
      tree::wn_layout(num_elements, num_queries, max_depth, leaf_size).total);
}

extern "C" int sbh_winding_number(void* stream, const SbhBuffer* points, const SbhBuffer* normals,
                                  const SbhBuffer* areas, const SbhBuffer* queries,
                                  SbhBuffer* out, float beta, int32_t max_depth,
                                  int32_t leaf_size, SbhBuffer* workspace, SbhBuffer* stats) {
  clear_error();
  int rc = tree::check_wn(points, normals, areas, queries, out, beta, max_depth, leaf_size);
  if (rc != SBH_OK) return rc;
  if (stats != nullptr &&
      (!buffer_ok(stats, SBH_DTYPE_S64, -1) || elem_count(stats) < 8))
    return fail_invalid("stats must be an int64 buffer of at least 8 elements");
  const int64_t n = points->dims[0], m = queries->dims[0];
  hipStream_t s = static_cast<hipStream_t>(stream);
  const tree::WnLayout W = tree::wn_layout(n, m, max_depth, leaf_size);
  char* ws = nullptr;
  if (workspace != nullptr) {
    if (!buffer_ok(workspace, SBH_DTYPE_U8, -1) ||
        byte_count(workspace) < static_cast<int64_t>(W.total))
      return fail_invalid("workspace too small");
    ws = static_cast<char*>(workspace->data);
  } else {
    if ((rc = cached_workspace(s, kWsPipeline, W.total, &ws)) != SBH_OK) return rc;
  }
  const auto* pts = static_cast<const float*>(points->data);
  const auto* q = static_cast<const float*>(queries->data);
  prof::Scope pr(s, 2);
  const bool profiled = pr.on() && m > 0;
  // Source tree over the centroids with areas as weights; the normals ride
  // along as the gathered per-point vector.
  auto* wd = reinterpret_cast<float4*>(ws + W.wd);
  rc = tree::build(s, ws, W.t, pts, static_cast<const float*>(areas->data),
                   static_cast<const float*>(normals->data), n, max_depth, leaf_size, nullptr,
                   tree::kBuildAll, wd);
  if (rc != SBH_OK) return rc;
  auto* hdr = reinterpret_cast<tree::Header*>(ws + W.t.header);
  const auto* topo = reinterpret_cast<const int4*>(ws + W.t.topo);
  const auto* mp = reinterpret_cast<const float4*>(ws + W.t.mp);
  const auto* sp = reinterpret_cast<const float4*>(ws + W.t.sp);
  const auto* sn = reinterpret_cast<const float4*>(ws + W.t.sc);
  // Query tree (topology and groups only).
  char* qws = ws + W.qbase;
  rc = tree::build(s, qws, W.qt, q, nullptr, nullptr, m, tree::kQueryDepth, tree::kQueryLeaf,
                   nullptr, tree::kBuildGroups);
  if (rc != SBH_OK) return rc;
  auto* qhdr = reinterpret_cast<tree::Header*>(qws + W.qt.header);
  if (m > 0) {
    tree::WnArgs A;
    A.hdr = hdr;
    A.qhdr = qhdr;
    A.groups = reinterpret_cast<const int2*>(qws + W.qt.groups);
    A.topo = topo;
    A.geo = reinterpret_cast<const float4*>(ws + W.t.geo);
    A.mp = mp;
    A.wd = wd;
    A.sp = sp;
    A.sn = sn;
    A.qs = reinterpret_cast<const float4*>(qws + W.qt.sp);
    A.qperm = reinterpret_cast<const uint32_t*>(qws + W.qt.perm);
    A.m = static_cast<int>(m);
    A.sentinel = static_cast<int>(W.t.cap);
    A.beta = beta;
    A.out = static_cast<float*>(out->data);
    A.stats = stats != nullptr;
    // a block per 64 queries up to what fits the chip (32 waves a CU)
    const bool wide = m <= tree::kWideQueries;
    const unsigned grid = grid_for(m, 64, 256 * 32 / (wide ? 16 : 8));
    if (profiled) {
      SBH_HIP_TRY(hipEventRecord(pr.rec().ev[1], s));
      SBH_HIP_TRY(hipEventRecord(pr.rec().ev[2], s));
    }
    if (wide)
      tree::k_wn_walk<16><<<grid, 64 * 16, 0, s>>>(A);
    else
      tree::k_wn_walk<8><<<grid, 64 * 8, 0, s>>>(A);
    SBH_LAUNCH_CHECK();
    if (profiled) {
      SBH_HIP_TRY(hipEventRecord(pr.rec().ev[3], s));
      pr.commit();
    }
  }
  if (stats != nullptr) {
    tree::k_wn_copy_stats<<<1, 64, 0, s>>>(hdr, qhdr, static_cast<int64_t*>(stats->data));
    SBH_LAUNCH_CHECK();
  }
  return SBH_OK;
}
