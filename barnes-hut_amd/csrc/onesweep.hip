// Stable LSD radix sort of 30-bit Morton codes (and of set ids) producing the
// sorted order as a permutation, in 2 + passes launches above 4096 keys, else in
// one (Adinets & Merrill,
// "Onesweep: A Faster Least Significant Digit Radix Sort for GPUs", 2022):
//
//   k_os_hist    per-block digit histograms of every pass (one read of the
//                codes) and zeroing of the look-back words
//   k_os_offsets global exclusive digit offsets of every pass; resets the
//                tile tickets
//   k_os_pass    one launch per 8-bit digit: each block takes the next tile
//                ticket, counts the tile's digits, publishes them, looks back
//                over the earlier tiles' published counts (decoupled look-back)
//                for its exclusive prefix per digit, ranks the tile's keys in
//                (wave, round, lane) order (which keeps the sort stable),
//                stages them in LDS sorted by digit and writes them out so
//                that consecutive threads fill consecutive slots of a digit
//
// Up to 4096 keys one launch (k_os_one) does all passes in one block.
//
// Code passes move (key, value) pairs, value = input row (the first pass
// reads the keys in input order and makes the values); set passes move
// values only, their digit being that of the set holding the row (sets are
// contiguous input row ranges), so the result is the order by (set, code,
// row).
//
// Every wait ends: a block spins only on tiles with smaller tickets, which
// were taken by blocks already running that publish their counts before
// they wait themselves.  A thread that has spun kSpinLimit times all the same
// counts its digit in the earlier tiles itself, so that the result is right in any
// case.
#include "common.hpp"
#include "tree.hpp"

namespace sbh {
namespace {

constexpr int kBlock = 512;
// Keys per thread: a tile of kBlock items(n) keys.  A pass waits for one key's
// ranking after another, so few keys are better with few tiles; the look-back
// reads grow with the square of the tiles, which bounds large sorts: 10^4
// keys 7 us a pass with 2 and 12 with 8 (2^20 keys: 21 with 8, 27 with 2048 keys a
// tile).
constexpr int kMaxItems = 8;
constexpr int64_t kTwoItems = int64_t{1} << 15, kFourItems = int64_t{1} << 17;
int items_for(int64_t n) { return n <= kTwoItems ? 2 : n <= kFourItems ? 4 : kMaxItems; }
int64_t tiles_for(int64_t n) {
  const int64_t tile = static_cast<int64_t>(kBlock) * items_for(n);
  return (n + tile - 1) / tile;
}
// Tiles to reserve scratch for: those of any sort of at most n keys (the tiles
// grow at kTwoItems and kFourItems, so that a larger sort may have fewer), so that
// scratch of a given size also holds every smaller sort.
int64_t tiles_reserved(int64_t n) {
  return std::max({tiles_for(n), tiles_for(std::min(n, kTwoItems)),
                   tiles_for(std::min(n, kFourItems))});
}
constexpr int kRadix = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kHistBlocks = 128;
constexpr int kHistBlock = 1024;
constexpr int kMaxPasses = 8;
constexpr int kBack = 16;  // tiles looked back over per round trip
constexpr uint32_t kAgg = 1u << 30;    // status: tile count published
constexpr uint32_t kIncl = 2u << 30;   // status: inclusive prefix published
constexpr uint32_t kValue = (1u << 30) - 1u;
constexpr int kSpinLimit = 1 << 22;
constexpr int64_t kMaxKeys = int64_t{1} << 30;  // counts share a word with two flags

// Blocks of k_os_hist for n keys.
int hist_blocks(int64_t n) {
  return static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>(kHistBlocks, (n + kHistBlock - 1) / kHistBlock)));
}

struct OsLayout {
  size_t hist;    // hist_blocks(n) x kMaxPasses x 256 u32
  size_t offs;    // passes x 256 u32: global exclusive digit offsets
  size_t ticket;  // passes u32 (padded)
  size_t status;  // passes x tiles x 256 u32
  size_t total;
};

OsLayout os_layout(int64_t n, int passes) {
  auto align = [](size_t x) { return (x + 255) & ~size_t{255}; };
  const size_t tiles = static_cast<size_t>(tiles_reserved(n));
  OsLayout L;
  size_t o = 0;
  L.hist = o; o = align(o + 4ull * hist_blocks(n) * kMaxPasses * kRadix);
  L.offs = o; o = align(o + 4ull * kMaxPasses * kRadix);
  L.ticket = o; o = align(o + 4ull * 64);
  L.status = o; o = align(o + 4ull * static_cast<size_t>(passes) * tiles * kRadix);
  L.total = o;
  return L;
}

__device__ __forceinline__ int row_set(const int32_t* __restrict__ set_offs, int nsets,
                                       uint32_t row) {
  return tree::set_of(set_offs, nsets, static_cast<int>(row));
}

// Per-block digit histograms of every pass: code passes from the codes, set
// passes from the set of each row (the same set_of the passes use, so the
// counts match the digits scattered whatever the offsets hold).
// Blocks of kHistBlock threads: the reads are few and each is followed by LDS
// adds (and a search for the row's set), so it takes many waves to hide them.
// 2^20 keys 7 us, 2.3e6 rows of 48 sets 19 (blocks of 256: 15 and 48).
__global__ __launch_bounds__(kHistBlock) void k_os_hist(const uint32_t* __restrict__ codes, int64_t n,
                                                    int code_passes, int set_passes,
                                                    const int32_t* __restrict__ set_offs,
                                                    int nsets, uint32_t* __restrict__ hist,
                                                    uint32_t* __restrict__ status,
                                                    int64_t status_words) {
  __shared__ uint32_t cnt[kMaxPasses][kRadix];
  const int passes = code_passes + set_passes;
  for (int p = threadIdx.x; p < kMaxPasses * kRadix; p += kHistBlock) cnt[p / kRadix][p % kRadix] = 0;
  __syncthreads();
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kHistBlock + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * kHistBlock) {
    const uint32_t k = codes[i];
    for (int p = 0; p < code_passes; ++p) atomicAdd(&cnt[p][(k >> (8 * p)) & 255u], 1u);
    if (set_passes > 0) {
      const uint32_t sid = static_cast<uint32_t>(row_set(set_offs, nsets, static_cast<uint32_t>(i)));
      for (int q = 0; q < set_passes; ++q)
        atomicAdd(&cnt[code_passes + q][(sid >> (8 * q)) & 255u], 1u);
    }
  }
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kHistBlock + threadIdx.x; i < status_words;
       i += static_cast<int64_t>(gridDim.x) * kHistBlock)
    status[i] = 0u;
  __syncthreads();
  for (int p = threadIdx.x; p < passes * kRadix; p += kHistBlock)
    hist[static_cast<int64_t>(blockIdx.x) * kMaxPasses * kRadix + p] = cnt[p / kRadix][p % kRadix];
}

// Global exclusive digit offsets, one block per pass; resets the pass's tile
// ticket.  Thread (quarter q, digit d) sums a quarter of the block histograms;
// the digits are then scanned in four waves.  (One block for all passes took
// 12.5 us for four, whatever n.)
__global__ __launch_bounds__(4 * kRadix) void k_os_offsets(const uint32_t* __restrict__ hist,
                                                           int blocks,
                                                           uint32_t* __restrict__ offs,
                                                           uint32_t* __restrict__ ticket) {
  __shared__ uint32_t part[4][kRadix];
  __shared__ uint32_t s_wave[4];
  const int d = threadIdx.x & (kRadix - 1), q = threadIdx.x / kRadix;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, p = blockIdx.x;
  uint32_t c = 0;
#pragma unroll 8
  for (int b = q; b < blocks; b += 4)
    c += hist[(static_cast<int64_t>(b) * kMaxPasses + p) * kRadix + d];
  part[q][d] = c;
  __syncthreads();
  const uint32_t tot = part[0][d] + part[1][d] + part[2][d] + part[3][d];
  uint32_t incl = tot;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(incl, o, 64);
    if (lane >= o) incl += t;
  }
  if (lane == 63 && w < 4) s_wave[w] = incl;
  __syncthreads();
  if (q == 0) {
    uint32_t before = 0;
    for (int k = 0; k < w; ++k) before += s_wave[k];
    offs[p * kRadix + d] = before + incl - tot;
  }
  if (threadIdx.x == 0) ticket[p] = 0u;
}

// One digit pass: (key, value) pairs move to their sorted slots.  The digit
// is a byte of the key (code pass) or of the set holding the row (set pass);
// on the first pass vals_in == nullptr makes the values the rows.  A wave ranks
// a run of 64 kItems consecutive keys of the tile by itself, round after round,
// with counts of its own in LDS, and the waves' counts are joined once; with
// rounds across the block and three barriers in each a pass over one tile took 9.5
// us instead of 7.
template <bool SET_PASS, int kItems>
__global__ __launch_bounds__(kBlock) void k_os_pass(
    const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in, int64_t n,
    int shift, const uint32_t* __restrict__ offs, uint32_t* __restrict__ ticket,
    uint32_t* __restrict__ status, const int32_t* __restrict__ set_offs, int nsets,
    uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out) {
  constexpr int kTile = kBlock * kItems;
  __shared__ uint32_t s_tile;
  __shared__ uint32_t s_base[kRadix];
  __shared__ uint32_t s_lstart[kRadix];
  __shared__ uint32_t s_wcnt[kWaves][kRadix];
  __shared__ uint32_t s_wave[kWaves];
  __shared__ uint32_t s_key[kTile];
  __shared__ uint32_t s_val[kTile];
  __shared__ uint8_t s_dig[kTile];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  if (tid == 0) s_tile = atomicAdd(ticket, 1u);
  for (int k = tid; k < kWaves * kRadix; k += kBlock) (&s_wcnt[0][0])[k] = 0u;
  __syncthreads();
  const uint32_t tile = s_tile;
  const int64_t base = static_cast<int64_t>(tile) * kTile;
  const int64_t run = base + wave * (64 * kItems) + lane;
  auto value = [&](int64_t i) {
    return vals_in != nullptr ? vals_in[i] : static_cast<uint32_t>(i);
  };
  auto digit_of = [&](uint32_t k, uint32_t v) {
    const uint32_t d = SET_PASS ? static_cast<uint32_t>(row_set(set_offs, nsets, v)) : k;
    return (d >> shift) & 255u;
  };
  uint32_t key[kItems], val[kItems], dig[kItems], loc[kItems];
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const int64_t i = run + r * 64;
    const bool ok = i < n;
    key[r] = ok ? keys_in[i] : 0u;
    val[r] = ok ? value(i) : 0u;
    dig[r] = ok ? digit_of(key[r], val[r]) : kRadix;
  }
  // rank the keys in (wave, round, lane) order, the input's: loc = the key's
  // offset among its wave's keys of the digit.  Only this wave touches its counts
  // here, and its LDS operations complete in order.
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const bool ok = dig[r] < kRadix;
    uint64_t peers = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (dig[r] >> b) & 1u;
      const uint64_t bal = __ballot(bit);
      peers &= bit ? bal : ~bal;
    }
    const uint32_t rank = static_cast<uint32_t>(__popcll(peers & lt));
    const uint32_t have = ok ? s_wcnt[wave][dig[r]] : 0u;
    loc[r] = have + rank;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (ok && rank == 0) s_wcnt[wave][dig[r]] = have + static_cast<uint32_t>(__popcll(peers));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // counts of the tile per digit; each wave's become the keys before its own
  const bool digit = tid < kRadix;  // the first kRadix threads: one per digit
  uint32_t mine = 0;
  if (digit) {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t c = s_wcnt[w][tid];
      s_wcnt[w][tid] = mine;
      mine += c;
    }
  }
  // publish this tile's counts, then look back for the exclusive prefix
  uint32_t* st = status + static_cast<int64_t>(tile) * kRadix;
  if (digit)
    __hip_atomic_store(st + tid, kAgg | mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // look back kBack tiles per round trip: their status words are loaded
  // together and the published ones consumed nearest first (aggregates added) up
  // to the first inclusive prefix; from the first not yet published, again
  uint32_t excl = 0;
  int spins = 0;
  bool done = !digit;
  for (int64_t k = static_cast<int64_t>(tile) - 1; k >= 0 && !done;) {
    uint32_t v[kBack];
#pragma unroll
    for (int j = 0; j < kBack; ++j)
      v[j] = k - j >= 0 ? __hip_atomic_load(status + (k - j) * kRadix + tid, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT)
                        : kIncl;
    bool ready = true;
    int used = 0;
#pragma unroll
    for (int j = 0; j < kBack; ++j) {
      ready = ready && !done && (v[j] & ~kValue) != 0u;
      excl += ready ? v[j] & kValue : 0u;
      used += ready ? 1 : 0;
      done = done || (ready && (v[j] & kIncl) != 0u);
    }
    k -= used;
    if (used == 0) {
      if (++spins >= kSpinLimit) {
        for (int64_t i = 0; i < (k + 1) * kTile; ++i)
          excl += digit_of(keys_in[i], value(i)) == static_cast<uint32_t>(tid) ? 1u : 0u;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    } else {
      spins = 0;
    }
  }
  if (digit) {
    __hip_atomic_store(st + tid, kIncl | ((excl + mine) & kValue), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    s_base[tid] = offs[tid] + excl;
  }
  // local start of each digit inside the tile (exclusive scan of the counts)
  {
    uint32_t incl = mine;
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t t = __shfl_up(incl, d, 64);
      if (lane >= d) incl += t;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
    for (int w = 0; w < wave; ++w) before += s_wave[w];
    if (digit) s_lstart[tid] = before + incl - mine;
    __syncthreads();
  }
  // stage the tile in LDS sorted by digit (stable: loc keeps the order)
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    if (dig[r] < kRadix) {
      const uint32_t lp = s_lstart[dig[r]] + s_wcnt[wave][dig[r]] + loc[r];
      s_key[lp] = key[r];
      s_val[lp] = val[r];
      s_dig[lp] = static_cast<uint8_t>(dig[r]);
    }
  }
  __syncthreads();
  // write the staged tile out: consecutive threads, consecutive slots of a digit
  const int64_t left = n - base;
  const int valid = left < kTile ? static_cast<int>(left) : kTile;
  for (int i = tid; i < valid; i += kBlock) {
    const uint32_t d = s_dig[i];
    const uint32_t dst = s_base[d] + (static_cast<uint32_t>(i) - s_lstart[d]);
    if (keys_out != nullptr) keys_out[dst] = s_key[i];
    vals_out[dst] = s_val[i];
  }
}

// All passes of a sort of at most kOneBlock * kItems keys by one block: the keys
// stay in registers and change places through LDS.  A launch and its waits for
// memory cost more than such a pass (forces of 2003 points 105 -> 88 us, of 4096 126 ->
// 112); with more keys a thread the one block ranks too long (8192 points 157 and 154
// us, 10,000 with 16 keys a thread 166 -> 191).  keys_out may be codes.
constexpr int kOneBlock = 1024;
constexpr int64_t kOneMax = 4 * kOneBlock;

template <int kItems>
__global__ __launch_bounds__(kOneBlock) void k_os_one(
    const uint32_t* codes, int n, int code_passes, int passes,
    const int32_t* __restrict__ set_offs, int nsets, uint32_t* keys_out,
    uint32_t* __restrict__ vals_out) {
  constexpr int kWaveCount = kOneBlock / 64;
  __shared__ uint32_t s_wcnt[kWaveCount][kRadix];
  __shared__ uint32_t s_lstart[kRadix];
  __shared__ uint32_t s_wave[kRadix / 64];
  __shared__ uint32_t s_key[kOneBlock * kItems];
  __shared__ uint32_t s_val[kOneBlock * kItems];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const int run = wave * (64 * kItems) + lane;  // a wave's keys are consecutive
  uint32_t key[kItems], val[kItems], dig[kItems], loc[kItems];
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const int i = run + r * 64;
    key[r] = i < n ? codes[i] : 0u;
    val[r] = static_cast<uint32_t>(i);
  }
  for (int p = 0; p < passes; ++p) {
    for (int k = tid; k < kWaveCount * kRadix; k += kOneBlock) (&s_wcnt[0][0])[k] = 0u;
    const int shift = 8 * (p < code_passes ? p : p - code_passes);
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
      const bool ok = run + r * 64 < n;
      uint32_t d = key[r];
      if (p >= code_passes) d = ok ? static_cast<uint32_t>(row_set(set_offs, nsets, val[r])) : 0u;
      dig[r] = ok ? (d >> shift) & 255u : kRadix;
    }
    __syncthreads();
    // ranks within the wave, as in k_os_pass
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
      const bool ok = dig[r] < kRadix;
      uint64_t peers = __ballot(ok);
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const bool bit = (dig[r] >> b) & 1u;
        const uint64_t bal = __ballot(bit);
        peers &= bit ? bal : ~bal;
      }
      const uint32_t rank = static_cast<uint32_t>(__popcll(peers & lt));
      const uint32_t have = ok ? s_wcnt[wave][dig[r]] : 0u;
      loc[r] = have + rank;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (ok && rank == 0) s_wcnt[wave][dig[r]] = have + static_cast<uint32_t>(__popcll(peers));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // each wave's counts become the keys of the digit before its own; digit starts
    uint32_t mine = 0, incl = 0;
    if (tid < kRadix) {
#pragma unroll
      for (int w = 0; w < kWaveCount; ++w) {
        const uint32_t c = s_wcnt[w][tid];
        s_wcnt[w][tid] = mine;
        mine += c;
      }
      incl = mine;
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
      }
      if (lane == 63) s_wave[wave] = incl;
    }
    __syncthreads();
    if (tid < kRadix) {
      uint32_t before = 0;
      for (int w = 0; w < wave; ++w) before += s_wave[w];
      s_lstart[tid] = before + incl - mine;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
      if (dig[r] < kRadix) {
        const uint32_t dst = s_lstart[dig[r]] + s_wcnt[wave][dig[r]] + loc[r];
        s_key[dst] = key[r];
        s_val[dst] = val[r];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
      const int i = run + r * 64;
      if (i < n) {
        key[r] = s_key[i];
        val[r] = s_val[i];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const int i = run + r * 64;
    if (i < n) {
      keys_out[i] = key[r];
      vals_out[i] = val[r];
    }
  }
}

}  // namespace

size_t morton_sort_temp_bytes(int64_t n, int nsets) {
  int set_passes = 0;
  while (nsets > 1 && (int64_t{1} << (8 * set_passes)) < nsets) ++set_passes;
  return os_layout(n, 4 + set_passes).total;
}

int morton_sort(hipStream_t s, const uint32_t* codes, int64_t n, int key_bits,
                const int32_t* set_offs, int nsets, uint32_t* keys_a, uint32_t* vals_a,
                uint32_t* keys_b, uint32_t* vals_b, void* temp,
                const uint32_t** keys, const uint32_t** perm) {
  *keys = nullptr;
  *perm = nullptr;
  if (n <= 0) return SBH_OK;
  if (n >= kMaxKeys) return fail_invalid("too many points for the sort");
  const int code_passes = key_bits <= 0 ? 1 : (key_bits + 7) / 8;
  int set_passes = 0;
  while (nsets > 1 && (int64_t{1} << (8 * set_passes)) < nsets) ++set_passes;
  const int passes = code_passes + set_passes;
  if (code_passes > 4 || passes > kMaxPasses) return fail_invalid("sort key too wide");
  if (n <= kOneMax) {
    auto one = [&](auto kernel) {
      kernel<<<1, kOneBlock, 0, s>>>(codes, static_cast<int>(n), code_passes, passes, set_offs,
                                     nsets, keys_b, vals_b);
    };
    if (n <= 2 * kOneBlock)
      one(k_os_one<2>);
    else
      one(k_os_one<4>);
    SBH_LAUNCH_CHECK();
    *keys = keys_b;
    *perm = vals_b;
    return SBH_OK;
  }
  const OsLayout L = os_layout(n, passes);
  char* t = static_cast<char*>(temp);
  auto* hist = reinterpret_cast<uint32_t*>(t + L.hist);
  auto* offs = reinterpret_cast<uint32_t*>(t + L.offs);
  auto* ticket = reinterpret_cast<uint32_t*>(t + L.ticket);
  auto* status = reinterpret_cast<uint32_t*>(t + L.status);
  const int items = items_for(n);
  const int64_t tiles = tiles_for(n);
  const int blocks = hist_blocks(n);
  k_os_hist<<<blocks, kHistBlock, 0, s>>>(codes, n, code_passes, set_passes, set_offs, nsets,
                                            hist, status,
                                            static_cast<int64_t>(passes) * tiles * kRadix);
  SBH_LAUNCH_CHECK();
  k_os_offsets<<<passes, 4 * kRadix, 0, s>>>(hist, blocks, offs, ticket);
  SBH_LAUNCH_CHECK();
  const uint32_t* kin = codes;
  const uint32_t* vin = nullptr;
  for (int p = 0; p < passes; ++p) {
    uint32_t* kout = (p & 1) ? keys_b : keys_a;
    uint32_t* vout = (p & 1) ? vals_b : vals_a;
    uint32_t* st = status + static_cast<int64_t>(p) * tiles * kRadix;
    // the keys travel through every pass: the last one leaves them sorted
    const bool set_pass = p >= code_passes;
    auto pass = [&](auto kernel) {
      kernel<<<static_cast<unsigned>(tiles), kBlock, 0, s>>>(
          kin, vin, n, 8 * (set_pass ? p - code_passes : p), offs + p * kRadix, ticket + p, st,
          set_offs, nsets, kout, vout);
    };
    if (items == 2)
      set_pass ? pass(k_os_pass<true, 2>) : pass(k_os_pass<false, 2>);
    else if (items == 4)
      set_pass ? pass(k_os_pass<true, 4>) : pass(k_os_pass<false, 4>);
    else
      set_pass ? pass(k_os_pass<true, kMaxItems>) : pass(k_os_pass<false, kMaxItems>);
    SBH_LAUNCH_CHECK();
    kin = kout;
    vin = vout;
  }
  *keys = kin;
  *perm = vin;
  return SBH_OK;
}

namespace {
__global__ __launch_bounds__(kBlock) void k_rows(uint32_t* __restrict__ vals, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i < n) vals[i] = static_cast<uint32_t>(i);
}
}  // namespace

size_t order_temp_bytes(int64_t n) {
  return n < kMaxKeys ? morton_sort_temp_bytes(n, 1) : radix_sort_temp_bytes(n);
}

int order_by_key(hipStream_t s, uint32_t* keys, int64_t n, int key_bits, uint32_t* vals,
                 uint32_t* keys2, uint32_t* vals2, void* temp, const uint32_t** sorted,
                 const uint32_t** perm) {
  if (n < kMaxKeys)
    return morton_sort(s, keys, n, key_bits, nullptr, 1, keys2, vals2, keys, vals, temp, sorted,
                       perm);
  k_rows<<<grid_for(n, kBlock), kBlock, 0, s>>>(vals, n);
  SBH_LAUNCH_CHECK();
  *sorted = keys2;
  *perm = vals2;
  return radix_sort_pairs(s, keys, vals, keys2, vals2, n, key_bits, temp);
}

}  // namespace sbh
