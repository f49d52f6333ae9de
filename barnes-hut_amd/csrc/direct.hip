// Direct O(N*M) sums in FP32 (no MFMA: there is no dense contraction).
//
// The softened sums (force, query-side VJP, full adjoint): one wave owns a
// chunk of 64 queries, one per lane, and a range of the sources, whose records
// it reads through the scalar cache (they are the same for all lanes), 8 at a
// time.  The ranges split the sources over the 4 waves of a block and over
// gridDim.y blocks; partial sums are combined in a fixed order, first in LDS,
// then (gridDim.y > 1) by k_direct_combine.  Attenuated sums over many sources
// keep one running sum per query instead (k_direct_running).
// The brute-force fields below: one thread per query, sources staged through
// LDS tiles of 256 records.
//
// Pair arithmetic follows src/sbh_ffi.cu:431-501 (forward and query-side VJP)
// and src/sbh_ffi.cu:399-429 (potential brute force).
#include <mutex>
#include <utility>

#include "common.hpp"

namespace sbh {
namespace {

constexpr int kBlock = 256;

struct PairParams {
  float eps2;     // max(eps, 0)^2
  float rc;       // cutoff scale (used when CUT)
  float box;      // periodic box length
  float inv_box;  // 1 / box
  int periodic;
};

// Source records through the scalar data cache: the arrays are not written
// while a sum runs, so they may be read as constant memory.
typedef __attribute__((address_space(4))) const float cfloat;

constexpr int kSplit = 4;  // waves of a block, each with its own source range
constexpr int kRun = 8;    // sources read together

template <bool PER>
__device__ __forceinline__ float pair_delta(float q, float s, const PairParams& P) {
  const float d = q - s;
  return PER ? fmaf(-P.box, rintf(d * P.inv_box), d) : d;
}

// att s^3 and 3 att s^5 + cutoff term of one pair (att = 1 without CUT).
template <bool CUT>
__device__ __forceinline__ void pair_kernel(float dx, float dy, float dz, const PairParams& P,
                                            float& lin, float& rad) {
  if constexpr (CUT) {
    const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
    const float s = rsq_softened(r2 + P.eps2 + 1e-12f);
    const float s2 = s * s, s3 = s2 * s;
    float e, dist;
    const float att = attenuation(r2, P.rc, &e, &dist);
    lin = att * s3;
    rad = fmaf(3.0f * s2, lin, s3 * (dist * e) * radial_cutoff(P.rc));
  } else {
    const float s =
        rsq_softened(fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, P.eps2 + 1e-12f))));
    const float s2 = s * s;
    lin = s2 * s;
    rad = 3.0f * s2 * lin;
  }
}

// Which sum: the forces, the query-side gradient J^T g, or the full
// self-gravity adjoint (queries = points).
enum DirectKind { kForce = 0, kVjp = 1, kFull = 2 };

template <int KIND>
constexpr int kComps = KIND == kFull ? 4 : 3;

// Sums of one query.  kFull, for the pair (k = this query, j = source) and
// d = minimage(x_k - x_j), lin = att s^3, K = 3 att s^5 + cutoff term:
//   v_kj = -m_j (lin c_k - (d.c_k) K d),  v_jk = -m_k (lin c_j - (d.c_j) K d),
//   grad_x[k] += v_kj - v_jk,   grad_m[k] += lin (c_j . d),
// regrouped as  -c_k sum m_j lin + m_k sum lin c_j
//               + sum K (m_j (d.c_k) - m_k (d.c_j)) d.
struct Query {
  float x, y, z, m;     // position (and mass, kFull)
  float gx, gy, gz;     // cotangent (kVjp, kFull)
  float ax, ay, az;     // sum of the radial terms (kForce: of the forces)
  float lm;             // sum m_j lin (kVjp, kFull)
  float bx, by, bz;     // sum lin c_j (kFull)
  float am;             // sum lin (c_j . d) (kFull)
};

template <int KIND, bool CUT, bool PER>
__device__ __forceinline__ void add_pair(Query& q, float sx, float sy, float sz, float sm,
                                         float cx, float cy, float cz, bool self,
                                         const PairParams& P) {
  const float dx = pair_delta<PER>(q.x, sx, P), dy = pair_delta<PER>(q.y, sy, P),
              dz = pair_delta<PER>(q.z, sz, P);
  float lin, rad;
  pair_kernel<CUT>(dx, dy, dz, P, lin, rad);
  if constexpr (KIND == kForce) {
    const float c = -sm * lin;
    q.ax = fmaf(c, dx, q.ax);
    q.ay = fmaf(c, dy, q.ay);
    q.az = fmaf(c, dz, q.az);
  } else if constexpr (KIND == kVjp) {
    const float u = fmaf(dz, q.gz, fmaf(dy, q.gy, dx * q.gx));
    const float t = sm * rad * u;
    q.lm = fmaf(sm, lin, q.lm);
    q.ax = fmaf(t, dx, q.ax);
    q.ay = fmaf(t, dy, q.ay);
    q.az = fmaf(t, dz, q.az);
  } else {
    // the self pair is zero in exact arithmetic (its two halves cancel); left out,
    // not weighted with 0: its cotangent may be infinite or NaN, and the
    // point's mass gradient does not depend on that
    if (self) return;
    const float u = fmaf(dz, q.gz, fmaf(dy, q.gy, dx * q.gx));
    const float v = fmaf(dz, cz, fmaf(dy, cy, dx * cx));
    const float t = rad * fmaf(sm, u, -(q.m * v));
    q.ax = fmaf(t, dx, q.ax);
    q.ay = fmaf(t, dy, q.ay);
    q.az = fmaf(t, dz, q.az);
    q.lm = fmaf(sm, lin, q.lm);
    q.bx = fmaf(lin, cx, q.bx);
    q.by = fmaf(lin, cy, q.by);
    q.bz = fmaf(lin, cz, q.bz);
    q.am = fmaf(lin, v, q.am);
  }
}

// The values of a query's sums.
template <int KIND>
__device__ __forceinline__ void finish(const Query& q, float (&v)[kComps<KIND>]) {
  if constexpr (KIND == kForce) {
    v[0] = q.ax;
    v[1] = q.ay;
    v[2] = q.az;
  } else {
    v[0] = fmaf(-q.lm, q.gx, q.ax);
    v[1] = fmaf(-q.lm, q.gy, q.ay);
    v[2] = fmaf(-q.lm, q.gz, q.az);
    if constexpr (KIND == kFull) {
      v[0] = fmaf(q.m, q.bx, v[0]);
      v[1] = fmaf(q.m, q.by, v[1]);
      v[2] = fmaf(q.m, q.bz, v[2]);
      v[3] = q.am;
    }
  }
}

// C consecutive sources from j.  SELF: the run may hold a query of the chunk
// (lane's own index i).
template <int KIND, bool CUT, bool PER, int C, bool SELF>
__device__ __forceinline__ void add_run(Query& q, cfloat* pts, cfloat* ms, cfloat* cot, int j,
                                        int i, const PairParams& P) {
  float s[3 * C], m[C], c[3 * C];
#pragma unroll
  for (int k = 0; k < 3 * C; ++k) s[k] = pts[3 * static_cast<int64_t>(j) + k];
#pragma unroll
  for (int k = 0; k < C; ++k) m[k] = ms[j + k];
  if constexpr (KIND == kFull) {
#pragma unroll
    for (int k = 0; k < 3 * C; ++k) c[k] = cot[3 * static_cast<int64_t>(j) + k];
  }
#pragma unroll
  for (int k = 0; k < C; ++k)
    add_pair<KIND, CUT, PER>(q, s[3 * k], s[3 * k + 1], s[3 * k + 2], m[k],
                             KIND == kFull ? c[3 * k] : 0.f, KIND == kFull ? c[3 * k + 1] : 0.f,
                             KIND == kFull ? c[3 * k + 2] : 0.f, SELF && j + k == i, P);
}

// Softened direct sums of the 64 queries of chunk blockIdx.x over source
// range blockIdx.y * kSplit + wave of `per` sources.  With one block per chunk
// the results go to out (nq x 3) and, kFull, out_m (nq); else the block's sums
// go to part[blockIdx.y] (nq x kComps).
//
// VALU-issue bound where the chip is full: 16 issue slots per pair for the
// force (the reciprocal square root takes 4 of them), 26 for the query-side
// VJP, 31 for the full adjoint.  Split so that small calls fill it too: one
// thread per query and all the sources left 10,000 queries on 40 of the 256
// CUs.  The scalar loads leave LDS and the barriers of a staged tile out.
// Measured, before -> after: force and full adjoint of 10,000 points 1.89 ->
// 0.10 ms; 65,536 sources at 4,099 queries with cutoff and periodic box 6.05 ->
// 0.28 ms; 131,072 x 131,072 pairs (chip full both ways) force 6.94 -> 5.27,
// query-side VJP 10.7 -> 7.2, full adjoint 18.7 -> 11.6 ms; 262,144 sources at
// 64 queries 9.05 -> 0.034 ms (a captured call has one block per chunk: 2.3).  The
// bits of a query depend on the number of blocks, and so on how many queries are
// asked and on capture (ranges and an order of adding that do not took 5 to 15% longer
// in attenuated sums).  The shorter sums are also more exact (10,000
// points: 1.4e-6 -> 7.5e-8 against 64 bits).
template <int KIND, bool CUT, bool PER>
__global__ __launch_bounds__(64 * kSplit) void k_direct(
    const float* __restrict__ pts_, const float* __restrict__ ms_,
    const float* __restrict__ cot_, int n, const float* __restrict__ qs,
    const float* __restrict__ qcot, int nq, int per, float* __restrict__ out,
    float* __restrict__ out_m, float* __restrict__ part, PairParams P) {
  constexpr int C = kComps<KIND>;
  __shared__ float red[kSplit - 1][C][64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  cfloat* pts = (cfloat*)(pts_);
  cfloat* ms = (cfloat*)(ms_);
  cfloat* cot = (cfloat*)(cot_);
  const int q0 = static_cast<int>(blockIdx.x) * 64;
  const int i = q0 + lane;
  const bool ok = i < nq;
  Query q = {};
  if (ok) {
    const int64_t o = 3 * static_cast<int64_t>(i);
    q.x = qs[o];
    q.y = qs[o + 1];
    q.z = qs[o + 2];
    if constexpr (KIND != kForce) {
      q.gx = qcot[o];
      q.gy = qcot[o + 1];
      q.gz = qcot[o + 2];
    }
    if constexpr (KIND == kFull) q.m = ms_[i];
  }
  // (64-bit: the last ranges of a ragged split may start beyond n)
  const int64_t b = (static_cast<int64_t>(blockIdx.y) * kSplit + w) * per;
  const int j0 = static_cast<int>(b < n ? b : n);
  const int j1 = static_cast<int>(b + per < n ? b + per : n);
  int j = j0;
  for (; j <= j1 - kRun; j += kRun) {
    if (KIND == kFull && j < q0 + 64 && j + kRun > q0)
      add_run<KIND, CUT, PER, kRun, true>(q, pts, ms, cot, j, i, P);
    else
      add_run<KIND, CUT, PER, kRun, false>(q, pts, ms, cot, j, i, P);
  }
  for (; j < j1; ++j) add_run<KIND, CUT, PER, 1, true>(q, pts, ms, cot, j, i, P);
  float v[C];
  finish<KIND>(q, v);
  if (w > 0)
    for (int c = 0; c < C; ++c) red[w - 1][c][lane] = v[c];
  __syncthreads();
  if (w > 0 || !ok) return;
  for (int k = 0; k < kSplit - 1; ++k)
    for (int c = 0; c < C; ++c) v[c] += red[k][c][lane];
  if (gridDim.y > 1) {
    float* p = part + (static_cast<int64_t>(blockIdx.y) * nq + i) * C;
    for (int c = 0; c < C; ++c) p[c] = v[c];
  } else {
    for (int c = 0; c < 3; ++c) out[3 * static_cast<int64_t>(i) + c] = v[c];
    if constexpr (KIND == kFull) out_m[i] = v[3];
  }
}

// Sums of the `splits` partials of k_direct (rows x COMPS values each) in a
// fixed order: 8 threads per value, 32 values per block.
template <int COMPS>
__global__ __launch_bounds__(256) void k_direct_combine(const float* __restrict__ part,
                                                        int splits, int64_t rows,
                                                        float* __restrict__ out,
                                                        float* __restrict__ out_m) {
  __shared__ float sh[8][32];
  const int e = threadIdx.x & 31, k = threadIdx.x >> 5;
  const int64_t total = rows * COMPS;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 32 + e;
  float v = 0.0f;
  if (i < total)
    for (int s = k; s < splits; s += 8) v += part[s * total + i];
  sh[k][e] = v;
  __syncthreads();
  if (k > 0 || i >= total) return;
  for (int t = 1; t < 8; ++t) v += sh[t][e];
  if constexpr (COMPS == 3) {
    out[i] = v;
  } else {
    const int64_t r = i / COMPS, c = i % COMPS;
    if (c < 3)
      out[3 * r + c] = v;
    else
      out_m[r] = v;
  }
}

// Adds the values of each run of 4 or 16 lanes, one after another, to the run's
// sums.
template <int C, int... E>
__device__ __forceinline__ void add_lanes(float (&sum)[C], const float (&v)[C],
                                          std::integer_sequence<int, E...>) {
  auto lane = [](float x, auto e) {
    // quad_perm or row_newbcast: lane e of the four or the sixteen
    constexpr int kCtrl = sizeof...(E) == 4 ? 0x55 * decltype(e)::value : 0x150 + decltype(e)::value;
    return __uint_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_uint(x), kCtrl, 0xf, 0xf, true));
  };
  auto add = [&](auto e) {
#pragma unroll
    for (int c = 0; c < C; ++c) sum[c] += lane(v[c], e);
  };
  (add(std::integral_constant<int, E>{}), ...);
}

// The forces and the query-side VJP with every query's terms added one after
// another in the order of the sources (running_sums() says when).  LANES lanes own
// a query and take as many sources at a time, whose terms they then add up in turn,
// the same chain of adds for either LANES.
template <int KIND, bool CUT, int LANES>
__global__ __launch_bounds__(256) void k_direct_running(
    const float* __restrict__ pts, const float* __restrict__ ms, int n,
    const float* __restrict__ qs, const float* __restrict__ qcot, int nq,
    float* __restrict__ out, PairParams P) {
  static_assert(KIND == kForce || KIND == kVjp, "three values a query");
  constexpr int kTiles = 4;
  const int e = threadIdx.x % LANES;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * (256 / LANES) + threadIdx.x / LANES;
  const int64_t o = 3 * (row < nq ? row : nq - 1);
  Query q = {};
  q.x = qs[o];
  q.y = qs[o + 1];
  q.z = qs[o + 2];
  if constexpr (KIND == kVjp) {
    q.gx = qcot[o];
    q.gy = qcot[o + 1];
    q.gz = qcot[o + 2];
  }
  float sum[3] = {};
  // the loads of kTiles tiles of LANES sources together
  for (int64_t j0 = e; j0 - e < n; j0 += LANES * kTiles) {
    float4 s[kTiles];
#pragma unroll
    for (int u = 0; u < kTiles; ++u) {
      const int64_t j = j0 + LANES * u < n ? j0 + LANES * u : n - 1;
      s[u] = make_float4(pts[3 * j], pts[3 * j + 1], pts[3 * j + 2], ms[j]);
    }
#pragma unroll
    for (int u = 0; u < kTiles; ++u) {
      Query t = q;
      add_pair<KIND, CUT, false>(t, s[u].x, s[u].y, s[u].z, s[u].w, 0.f, 0.f, 0.f, false, P);
      float v[3];
      finish<KIND>(t, v);
      if (j0 + LANES * u >= n) v[0] = v[1] = v[2] = 0.0f;
      add_lanes(sum, v, std::make_integer_sequence<int, LANES>{});
    }
  }
  if (row >= nq || e > 0) return;
  for (int c = 0; c < 3; ++c) out[o + c] = sum[c];
}

// Whether a query's terms go to one running sum: attenuated sums over many
// sources.  Most of their terms are small, and a running sum loses those below half
// an ulp of it: split sums are closer to 64 bits, but leave the sums in
// source order, which callers compare with, by 5.3e-6 at 65,536 sources,
// 1.1e-5 at 131,072 and 2.3e-5 at 262,144 (uniform cube, cutoff 0.05; running
// sums: 1.6e-7).  Without attenuation it is 7.7e-6 at 262,144 and in a periodic box
// 5e-6: split.  So is the full adjoint, which is not asked for at such sizes.  The
// rule leaves the number of queries out, so that a query's bits do not depend on it.
// 262,144 sources at 64, 1001 and 16,384 queries, split and running: 0.054, 0.26 and 3.6
// against 3.4, 3.4 and 9.5 ms (one thread per query: 54, 55 and 58).
constexpr int64_t kRunningMin = 65536;
bool running_sums(int64_t n, bool cut, bool periodic) {
  return cut && !periodic && n >= kRunningMin;
}
// Queries from which 4 lanes own one, below 16: 4 do less adding beside the pairs, but
// fill the chip later (262,144 sources at 8192 queries 9.3 and 5.8 ms, at 16,384
// 9.5 and 10.9, at 131,072 52 and 82).
constexpr int64_t kFourLanes = 16384;

// Blocks per chunk of 64 queries: as many whole blocks as give at most 8 waves to
// each of the 1024 SIMDs (more than 2048 blocks would end in a second, nearly empty
// round: 65,536 attenuated sources at 4099 queries 0.29 ms with 31 blocks per chunk,
// 0.33 with 32), one from 65,537 queries on; at least 64 sources per wave (below
// that the wave's start, the combine and its launch, about 4 us, cost more than
// they save); at most 256 partials per query.  Up to 1024 sources (512 with attenuation, whose
// pairs take three times as long) a wave's quarter is short: 1000 sources 14.0 us a call
// unsplit and 16.4 split, 2048 21 and 16; 700 attenuated 16.4 and 17.1, 1000 22.9 and
// 16.9.
int direct_blocks(int64_t n, int64_t nq, bool cut) {
  if (n <= (cut ? 512 : 1024)) return 1;
  const int64_t chunks = (nq + 63) / 64;
  int64_t y = 2048 / chunks;
  y = y < n / (64 * kSplit) ? y : n / (64 * kSplit);
  y = y < 256 ? y : 256;
  return static_cast<int>(y > 1 ? y : 1);
}

// The partial sums live in a scratch buffer of the stream, so another host
// thread's call on the same stream must not launch between a call's two
// kernels.
std::mutex g_direct_mu;

template <int KIND, bool CUT, bool PER>
int launch_direct_as(hipStream_t s, const float* pts, const float* ms, const float* cot, int n,
                     const float* qs, const float* qcot, int nq, float* out, float* out_m,
                     const PairParams& P) {
  constexpr int C = kComps<KIND>;
  if constexpr (KIND != kFull && CUT && !PER) {
    if (running_sums(n, CUT, PER)) {
      auto* run = nq >= kFourLanes ? k_direct_running<KIND, CUT, 4> : k_direct_running<KIND, CUT, 16>;
      run<<<grid_for(nq, nq >= kFourLanes ? 64 : 16), 256, 0, s>>>(pts, ms, n, qs, qcot, nq, out, P);
      SBH_LAUNCH_CHECK();
      return SBH_OK;
    }
  }
  std::lock_guard<std::mutex> lock(g_direct_mu);
  int blocks = direct_blocks(n, nq, CUT);
  float* part = nullptr;
  if (blocks > 1) {
    // unsplit under stream capture (the scratch could need an allocation), on the
    // per-thread default stream (one handle, but a stream for each host thread), and
    // where there is no memory for the scratch
    if (s != hipStreamPerThread && !stream_capturing(s))
      part = static_cast<float*>(
          workspace(s, kWsDirect, sizeof(float) * C * static_cast<size_t>(blocks) * nq));
    if (part == nullptr) blocks = 1;
  }
  const int64_t ranges = static_cast<int64_t>(blocks) * kSplit;
  const int per = static_cast<int>(((n + ranges - 1) / ranges + kRun - 1) / kRun * kRun);
  const dim3 grid((static_cast<unsigned>(nq) + 63u) / 64u, static_cast<unsigned>(blocks));
  k_direct<KIND, CUT, PER><<<grid, 64 * kSplit, 0, s>>>(pts, ms, cot, n, qs, qcot, nq, per, out,
                                                        out_m, part, P);
  SBH_LAUNCH_CHECK();
  if (blocks > 1) {
    k_direct_combine<C><<<grid_for(static_cast<int64_t>(nq) * C, 32), 256, 0, s>>>(
        part, blocks, nq, out, out_m);
    SBH_LAUNCH_CHECK();
  }
  return SBH_OK;
}

template <int KIND>
int launch_direct(hipStream_t s, const float* pts, const float* ms, const float* cot, int64_t n,
                  const float* qs, const float* qcot, int64_t nq, float* out, float* out_m,
                  const PairParams& P, bool cut) {
  const int n32 = static_cast<int>(n), nq32 = static_cast<int>(nq);
  if (cut)
    return P.periodic
               ? launch_direct_as<KIND, true, true>(s, pts, ms, cot, n32, qs, qcot, nq32, out, out_m, P)
               : launch_direct_as<KIND, true, false>(s, pts, ms, cot, n32, qs, qcot, nq32, out, out_m, P);
  return P.periodic
             ? launch_direct_as<KIND, false, true>(s, pts, ms, cot, n32, qs, qcot, nq32, out, out_m, P)
             : launch_direct_as<KIND, false, false>(s, pts, ms, cot, n32, qs, qcot, nq32, out, out_m, P);
}

__device__ __forceinline__ void load_tile(float4* tile, const float* __restrict__ pts,
                                          const float* __restrict__ ms, int n, int base,
                                          int dim) {
  int j = base + static_cast<int>(threadIdx.x);
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (j < n) {
    const float* p = pts + static_cast<int64_t>(j) * dim;
    v.x = p[0];
    v.y = p[1];
    v.z = dim == 3 ? p[2] : 0.0f;
    v.w = ms[j];
  }
  tile[threadIdx.x] = v;
}

// Potential brute force (src/sbh_ffi.cu:399-429), dim 2 or 3.
__global__ __launch_bounds__(kBlock) void k_bruteforce_gravity(
    const float* __restrict__ pts, const float* __restrict__ ms, int n,
    const float* __restrict__ qs, int nq, int dim, float* __restrict__ out, int periodic,
    float box) {
  __shared__ float4 tile[kBlock];
  int i = blockIdx.x * kBlock + threadIdx.x;
  float qx = 0.f, qy = 0.f, qz = 0.f;
  if (i < nq) {
    const float* q = qs + static_cast<int64_t>(i) * dim;
    qx = q[0];
    qy = q[1];
    qz = dim == 3 ? q[2] : 0.0f;
  }
  float acc = 0.0f;
  for (int base = 0; base < n; base += kBlock) {
    load_tile(tile, pts, ms, n, base, dim);
    __syncthreads();
    int cnt = min(kBlock, n - base);
    for (int k = 0; k < cnt; ++k) {
      float4 s = tile[k];
      float dx = s.x - qx, dy = s.y - qy, dz = s.z - qz;
      if (periodic) {
        dx -= box * rintf(dx / box);
        dy -= box * rintf(dy / box);
        dz -= box * rintf(dz / box);
      }
      float dist = sqrtf(dx * dx + dy * dy + dz * dz);
      acc += -s.w / (dist + 1e-1f);
    }
    __syncthreads();
  }
  if (i < nq) out[i] = acc;
}

// Winding-number brute force (src/sbh_gpu.cu:53-64 with brute_force_gpu.h:18-66):
// per query, the compensated (Kahan) sum of signedSolidAngle<3> over all
// oriented area elements, staged through LDS one tile at a time.
__global__ __launch_bounds__(kBlock) void k_bruteforce_wn(
    const float* __restrict__ pts, const float* __restrict__ nrm,
    const float* __restrict__ area, int n, const float* __restrict__ qs, int nq,
    float* __restrict__ out) {
  __shared__ float4 tp[kBlock];
  __shared__ float4 tn[kBlock];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  float qx = 0.f, qy = 0.f, qz = 0.f;
  if (i < nq) {
    qx = qs[3 * static_cast<int64_t>(i)];
    qy = qs[3 * static_cast<int64_t>(i) + 1];
    qz = qs[3 * static_cast<int64_t>(i) + 2];
  }
  float total = 0.0f, comp = 0.0f;
  for (int base = 0; base < n; base += kBlock) {
    const int j = base + threadIdx.x;
    if (j < n) {
      const int64_t o = 3 * static_cast<int64_t>(j);
      tp[threadIdx.x] = make_float4(pts[o], pts[o + 1], pts[o + 2], area[j]);
      tn[threadIdx.x] = make_float4(nrm[o], nrm[o + 1], nrm[o + 2], 0.f);
    }
    __syncthreads();
    const int cnt = min(kBlock, n - base);
    for (int k = 0; k < cnt; ++k) {
      const float4 p = tp[k], nv = tn[k];
      const float dx = p.x - qx, dy = p.y - qy, dz = p.z - qz;
      const float r = sqrtf(dx * dx + dy * dy + dz * dz);
      const float v = p.w * (nv.x * dx + nv.y * dy + nv.z * dz) * 0.07957747154594767f /
                      (r * r * r + 1e-5f);
      const float y = v - comp;
      const float t = total + y;
      comp = (t - total) - y;
      total = t;
    }
    __syncthreads();
  }
  if (i < nq) out[i] = total;
}

// smoothDistExp brute force (src/sbh_gpu.cu:66-77, 287-322): sum over all
// points of exp(-alpha_j |p_j - q|), Kahan-compensated as
// include/brute_force_gpu.h:18-66, points staged through LDS tiles.
__global__ __launch_bounds__(kBlock) void k_bruteforce_smoothdist(
    const float* __restrict__ pts, const float* __restrict__ alpha, int n,
    const float* __restrict__ qs, int nq, float* __restrict__ out) {
  __shared__ float4 tp[kBlock];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  float qx = 0.f, qy = 0.f, qz = 0.f;
  if (i < nq) {
    qx = qs[3 * static_cast<int64_t>(i)];
    qy = qs[3 * static_cast<int64_t>(i) + 1];
    qz = qs[3 * static_cast<int64_t>(i) + 2];
  }
  float total = 0.0f, comp = 0.0f;
  for (int base = 0; base < n; base += kBlock) {
    const int j = base + threadIdx.x;
    if (j < n) {
      const int64_t o = 3 * static_cast<int64_t>(j);
      tp[threadIdx.x] = make_float4(pts[o], pts[o + 1], pts[o + 2], alpha[j]);
    }
    __syncthreads();
    const int cnt = min(kBlock, n - base);
    for (int k = 0; k < cnt; ++k) {
      const float4 p = tp[k];
      const float dx = p.x - qx, dy = p.y - qy, dz = p.z - qz;
      const float v = expf(-p.w * sqrtf(dx * dx + dy * dy + dz * dz));
      const float y = v - comp;
      const float t = total + y;
      comp = (t - total) - y;
      total = t;
    }
    __syncthreads();
  }
  if (i < nq) out[i] = total;
}

PairParams make_params(float softening, float cutoff, int periodic, float box) {
  PairParams P;
  float eps = fmaxf(softening, 0.0f);
  P.eps2 = eps * eps;
  P.rc = cutoff;
  P.periodic = (periodic != 0 && box > 0.0f) ? 1 : 0;
  P.box = box;
  P.inv_box = box > 0.0f ? 1.0f / box : 0.0f;
  return P;
}

// A finite positive cutoff applies the erfc attenuation; +inf gives exactly 1.
inline bool cutoff_active(float cutoff) { return cutoff > 0.0f && std::isfinite(cutoff); }

int check_direct_common(const SbhBuffer* points, const SbhBuffer* masses,
                        const SbhBuffer* queries, float softening, float cutoff,
                        int threads) {
  if (!buffer_ok(points, SBH_DTYPE_F32, -1) || !buffer_ok(queries, SBH_DTYPE_F32, -1) ||
      !buffer_ok(masses, SBH_DTYPE_F32, -1))
    return fail_invalid("points/masses/queries must be float32 device buffers");
  if (points->rank != 2 || queries->rank != 2)
    return fail_invalid("points/queries must be rank-2");
  if (points->dims[1] != 3 || queries->dims[1] != 3)
    return fail_invalid("points/queries must have dim=3");
  if (elem_count(masses) != points->dims[0]) return fail_invalid("masses length mismatch");
  if (softening < 0.0f) return fail_invalid("softening_scale must be >= 0");
  if (!(cutoff > 0.0f)) return fail_invalid("cutoff_scale must be > 0");
  if (threads <= 0 || threads > 1024) return fail_invalid("threads must be in [1, 1024]");
  if (points->dims[0] > INT32_MAX || queries->dims[0] > INT32_MAX)
    return fail_invalid("too many points");
  return SBH_OK;
}

}  // namespace
}  // namespace sbh

using namespace sbh;

extern "C" int sbh_bruteforce_gravity(void* stream, const SbhBuffer* points,
                                      const SbhBuffer* masses, const SbhBuffer* queries,
                                      SbhBuffer* out, int32_t periodic, float box_length,
                                      int32_t threads) {
  clear_error();
  if (!buffer_ok(points, SBH_DTYPE_F32, -1) || !buffer_ok(queries, SBH_DTYPE_F32, -1) ||
      !buffer_ok(masses, SBH_DTYPE_F32, -1) || !buffer_ok(out, SBH_DTYPE_F32, -1))
    return fail_invalid("points/masses/queries/out must be float32 device buffers");
  if (points->rank != 2 || queries->rank != 2)
    return fail_invalid("points/queries must be rank-2");
  int64_t n = points->dims[0], dim = points->dims[1], nq = queries->dims[0];
  if (queries->dims[1] != dim) return fail_invalid("queries dim mismatch");
  if (elem_count(masses) != n) return fail_invalid("masses length mismatch");
  if (dim != 2 && dim != 3) return fail_invalid("only dim=2 or dim=3 supported");
  if (threads <= 0 || threads > 1024) return fail_invalid("threads must be in [1, 1024]");
  if (elem_count(out) != nq) return fail_invalid("out shape mismatch");
  if (n > INT32_MAX || nq > INT32_MAX) return fail_invalid("too many points");
  if (nq == 0) return SBH_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int per = (periodic != 0 && box_length > 0.0f) ? 1 : 0;
  k_bruteforce_gravity<<<grid_for(nq, kBlock), kBlock, 0, s>>>(
      static_cast<const float*>(points->data), static_cast<const float*>(masses->data),
      static_cast<int>(n), static_cast<const float*>(queries->data), static_cast<int>(nq),
      static_cast<int>(dim), static_cast<float*>(out->data), per, box_length);
  SBH_LAUNCH_CHECK();
  return SBH_OK;
}

extern "C" int sbh_bruteforce_wn(void* stream, const SbhBuffer* points,
                                 const SbhBuffer* normals, const SbhBuffer* areas,
                                 const SbhBuffer* queries, SbhBuffer* out, int32_t threads) {
  clear_error();
  if (!buffer_ok(points, SBH_DTYPE_F32, 2) || points->dims[1] != 3)
    return fail_invalid("points must have shape (N, 3)");
  const int64_t n = points->dims[0];
  if (!buffer_ok(normals, SBH_DTYPE_F32, 2) || normals->dims[0] != n || normals->dims[1] != 3)
    return fail_invalid("normals must have shape (N, 3)");
  if (!buffer_ok(areas, SBH_DTYPE_F32, 1) || areas->dims[0] != n)
    return fail_invalid("areas must have shape (N,)");
  if (!buffer_ok(queries, SBH_DTYPE_F32, 2) || queries->dims[1] != 3)
    return fail_invalid("queries must have shape (M, 3)");
  const int64_t nq = queries->dims[0];
  if (!buffer_ok(out, SBH_DTYPE_F32, 1) || out->dims[0] != nq)
    return fail_invalid("out must have shape (M,)");
  if (threads <= 0 || threads > 1024) return fail_invalid("threads must be in [1, 1024]");
  if (n > INT32_MAX || nq > INT32_MAX) return fail_invalid("too many points");
  if (nq == 0) return SBH_OK;
  k_bruteforce_wn<<<grid_for(nq, kBlock), kBlock, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const float*>(points->data), static_cast<const float*>(normals->data),
      static_cast<const float*>(areas->data), static_cast<int>(n),
      static_cast<const float*>(queries->data), static_cast<int>(nq),
      static_cast<float*>(out->data));
  SBH_LAUNCH_CHECK();
  return SBH_OK;
}

extern "C" int sbh_bruteforce_smoothdist(void* stream, const SbhBuffer* points,
                                         const SbhBuffer* alphas, const SbhBuffer* queries,
                                         SbhBuffer* out, int32_t threads) {
  clear_error();
  if (!buffer_ok(points, SBH_DTYPE_F32, 2) || points->dims[1] != 3)
    return fail_invalid("points must have shape (N, 3)");
  const int64_t n = points->dims[0];
  if (!buffer_ok(alphas, SBH_DTYPE_F32, 1) || alphas->dims[0] != n)
    return fail_invalid("alphas must have shape (N,)");
  if (!buffer_ok(queries, SBH_DTYPE_F32, 2) || queries->dims[1] != 3)
    return fail_invalid("queries must have shape (M, 3)");
  const int64_t nq = queries->dims[0];
  if (!buffer_ok(out, SBH_DTYPE_F32, 1) || out->dims[0] != nq)
    return fail_invalid("out must have shape (M,)");
  if (threads <= 0 || threads > 1024) return fail_invalid("threads must be in [1, 1024]");
  if (n > INT32_MAX || nq > INT32_MAX) return fail_invalid("too many points");
  if (nq == 0) return SBH_OK;
  k_bruteforce_smoothdist<<<grid_for(nq, kBlock), kBlock, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const float*>(points->data), static_cast<const float*>(alphas->data),
      static_cast<int>(n), static_cast<const float*>(queries->data), static_cast<int>(nq),
      static_cast<float*>(out->data));
  SBH_LAUNCH_CHECK();
  return SBH_OK;
}

extern "C" int sbh_direct_force_soft(void* stream, const SbhBuffer* points,
                                     const SbhBuffer* masses, const SbhBuffer* queries,
                                     SbhBuffer* out, float softening_scale,
                                     float cutoff_scale, int32_t periodic,
                                     float box_length, int32_t threads) {
  clear_error();
  int rc = check_direct_common(points, masses, queries, softening_scale, cutoff_scale,
                               threads);
  if (rc != SBH_OK) return rc;
  int64_t n = points->dims[0], nq = queries->dims[0];
  if (!buffer_ok(out, SBH_DTYPE_F32, 2) || out->dims[0] != nq || out->dims[1] != 3)
    return fail_invalid("out shape mismatch");
  if (nq == 0) return SBH_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  PairParams P = make_params(softening_scale, cutoff_scale, periodic, box_length);
  auto* pp = static_cast<const float*>(points->data);
  auto* pm = static_cast<const float*>(masses->data);
  auto* pq = static_cast<const float*>(queries->data);
  auto* po = static_cast<float*>(out->data);
  return launch_direct<kForce>(s, pp, pm, nullptr, n, pq, nullptr, nq, po, nullptr, P, cutoff_active(cutoff_scale));
}

extern "C" int sbh_direct_force_soft_vjp(void* stream, const SbhBuffer* points,
                                         const SbhBuffer* masses, const SbhBuffer* queries,
                                         const SbhBuffer* cotangent, SbhBuffer* out,
                                         float softening_scale, float cutoff_scale,
                                         int32_t periodic, float box_length,
                                         int32_t threads) {
  clear_error();
  if (points == nullptr || queries == nullptr || cotangent == nullptr ||
      points->rank != 2 || queries->rank != 2 || cotangent->rank != 2)
    return fail_invalid("points/queries/cotangent must be rank-2");
  if (!buffer_ok(cotangent, SBH_DTYPE_F32, 2))
    return fail_invalid("cotangent must be a float32 device buffer");
  if (points->dims[1] != 3 || queries->dims[1] != 3 || cotangent->dims[1] != 3)
    return fail_invalid("points/queries/cotangent must have dim=3");
  if (cotangent->dims[0] != queries->dims[0]) return fail_invalid("cotangent shape mismatch");
  int rc = check_direct_common(points, masses, queries, softening_scale, cutoff_scale,
                               threads);
  if (rc != SBH_OK) return rc;
  int64_t n = points->dims[0], nq = queries->dims[0];
  if (!buffer_ok(out, SBH_DTYPE_F32, 2) || out->dims[0] != nq || out->dims[1] != 3)
    return fail_invalid("out shape mismatch");
  if (nq == 0) return SBH_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  PairParams P = make_params(softening_scale, cutoff_scale, periodic, box_length);
  auto* pp = static_cast<const float*>(points->data);
  auto* pm = static_cast<const float*>(masses->data);
  auto* pq = static_cast<const float*>(queries->data);
  auto* pc = static_cast<const float*>(cotangent->data);
  auto* po = static_cast<float*>(out->data);
  return launch_direct<kVjp>(s, pp, pm, nullptr, n, pq, pc, nq, po, nullptr, P, cutoff_active(cutoff_scale));
}

extern "C" int sbh_direct_force_soft_full_vjp(void* stream, const SbhBuffer* points,
                                              const SbhBuffer* masses,
                                              const SbhBuffer* cotangent,
                                              SbhBuffer* grad_points,
                                              SbhBuffer* grad_masses,
                                              float softening_scale, float cutoff_scale,
                                              int32_t periodic, float box_length,
                                              int32_t threads) {
  clear_error();
  int rc = check_direct_common(points, masses, points, softening_scale, cutoff_scale,
                               threads);
  if (rc != SBH_OK) return rc;
  int64_t n = points->dims[0];
  if (!buffer_ok(cotangent, SBH_DTYPE_F32, 2) || cotangent->dims[0] != n ||
      cotangent->dims[1] != 3)
    return fail_invalid("cotangent shape mismatch");
  if (!buffer_ok(grad_points, SBH_DTYPE_F32, 2) || grad_points->dims[0] != n ||
      grad_points->dims[1] != 3)
    return fail_invalid("grad_points shape mismatch");
  if (!buffer_ok(grad_masses, SBH_DTYPE_F32, -1) || elem_count(grad_masses) != n)
    return fail_invalid("grad_masses shape mismatch");
  if (n == 0) return SBH_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  PairParams P = make_params(softening_scale, cutoff_scale, periodic, box_length);
  auto* pp = static_cast<const float*>(points->data);
  auto* pm = static_cast<const float*>(masses->data);
  auto* pc = static_cast<const float*>(cotangent->data);
  auto* gx = static_cast<float*>(grad_points->data);
  auto* gm = static_cast<float*>(grad_masses->data);
  return launch_direct<kFull>(s, pp, pm, pc, n, pp, pc, n, gx, gm, P, cutoff_active(cutoff_scale));
}
