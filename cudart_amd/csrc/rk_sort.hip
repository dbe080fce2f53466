// Stable LSD radix sort for gfx950, 8-bit digits, onesweep style:
//   1. one kernel counts the digits of every pass in a single read (or the
//      kernel that makes the keys does, rk_sort.h);
//   2. one scatter kernel per pass. Each 512-thread workgroup sorts the tile
//      of its block index (2048, 4096 or 8192 keys): it ranks its keys stably
//      with per-(wave, digit) lane masks in LDS, publishes its per-digit
//      counts, resolves its global per-digit prefix by decoupled look-back
//      over earlier tiles, reorders the tile by digit in LDS and writes it
//      out in per-digit runs, keys first, then values through the same LDS.
// Up to 4096 keys, one workgroup does all passes in LDS in a single launch
// instead (k_sort_one: a 3,042-face build 43 us against 52).
// Below 2^21 keys a pass is bound by latency, at most a few tiles per CU, and
// the look-back has two levels: a tile adds the counts of the tiles before it
// in its group of 16, all in flight at once, and looks back over groups (1M
// pairs: 15.2 against 16.8 us per pass; with one level the prefixes advance 8
// tiles per round trip). Above, tiles queue on every CU and overlap each other.
// Slower: ranks from eight ballots per key (158 against 155 us per 1M-face
// build, 1613 against 1577 for 10M); wider digits, 10 bits (three passes for
// 30-bit keys) at 25.9 us per pass on 1M pairs, 9 bits (seven for 63) at 85.6
// us on 10M 64-bit pairs against 59.7, for their shorter runs and more counts to
// look back over.
// Tiles follow the block index rather than a counter that every workgroup
// increments (on MI355X such a counter serialises the workgroups' start
// across the eight XCDs). A workgroup only waits on lower tiles; workgroups
// are dispatched in block order on each XCD, so the lowest unfinished tile is
// always resident or next to be dispatched on its XCD, whose earlier
// workgroups have all finished. Look-back waits are bounded (kSpinLimit); on
// expiry the kernel sets an error bit and finishes, so a fault in the
// protocol cannot hang the GPU.
//
// The reference's sorts (CUDA_radixSortGeneral.cu, CUDA_radixSort.cu,
// CUDA_bitonicSortGeneral.cu, CUDA_bitonicSort.cu, CUDA_bubbleSort512.cu)
// differ in tie order by size class; rk_radix_sort_general reproduces that
// order (see the size-class notes at the entry point).
#include <algorithm>
#include <utility>

#include "rk_sort.h"

namespace {

#ifndef RK_SCATTER_WAVES
#define RK_SCATTER_WAVES 8
#endif
#ifndef RK_SCATTER_ITEMS
#define RK_SCATTER_ITEMS 16
#endif
constexpr int kWaves = RK_SCATTER_WAVES;    // waves per scatter workgroup
constexpr int kThreads = 64 * kWaves;
constexpr int kItems = RK_SCATTER_ITEMS;    // keys per lane, at most
// Keys per tile: 8192 from 2^21 keys on, 4096 below (8192 would leave most of
// the 256 CUs idle on 1M keys: 214 against 224 us per build; 10M keys 1.73 ms
// with 8192 against 1.80), 2048 below 2^19 (a 180K-face build 97.7 against
// 104.5 us, the 20,480-face icosphere 64 against 70; 1M 156.5 against 155.6).
constexpr int kItemsMid = 8, kItemsSmall = 4;
constexpr size_t kMidTilesBelow = size_t(1) << 21, kSmallTilesBelow = size_t(1) << 19;
static_assert(kThreads >= 256, "one thread per digit");
constexpr uint32_t kAgg = 1u << 30;
constexpr uint32_t kInc = 2u << 30;
constexpr uint32_t kCountMask = (1u << 30) - 1u;
constexpr uint32_t kSpinLimit = 1u << 20;
constexpr int kMaxPasses = 8;
constexpr uint32_t kOneMax = 4096;  // up to this many keys one workgroup sorts them in LDS
#ifndef RK_SORT_LOOK
#define RK_SORT_LOOK 8
#endif
constexpr int kLook = RK_SORT_LOOK;  // look-back status loads in flight per digit

constexpr uint32_t kGroup = 16;  // tiles per look-back group
constexpr uint32_t kMaxCopies = 8;  // of the digit counts

// Exclusive scan over a block of kT threads of kPer consecutive values each.
template <int kT, int kPer>
__device__ __forceinline__ void block_excl_scan(const uint32_t (&v)[kPer], uint32_t (&ex)[kPer],
                                                uint32_t* s_tmp /*>= kT / 64*/) {
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t sum = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) sum += v[u];
  uint32_t incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t y = __shfl_up(incl, off, 64);
    if (lane >= (uint32_t)off) incl += y;
  }
  if (lane == 63) s_tmp[wave] = incl;
  __syncthreads();
  uint32_t run = incl - sum;
#pragma unroll
  for (int w = 0; w < kT / 64; ++w) run += (w < (int)wave) ? s_tmp[w] : 0u;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    ex[u] = run;
    run += v[u];
  }
}

// Digit counts of every pass in one read. Block b counts keys
// [b * chunk, (b + 1) * chunk), eight loads in flight per thread; a wave whose
// 64 keys share a digit (the high digits of spatially ordered keys) adds them
// with one LDS atomic instead of 64 to the same address. Each block adds to one
// of 'copies' copies of the counts, so that fewer meet on one address.
constexpr int kHistUnroll = 8;
constexpr uint32_t kHistMaxBlocks = 1024;
constexpr size_t kHistKeysPerBlock = 256 * kHistUnroll * 2;

// Also zeroes the look-back words of the first pass (zero, zero_words), which
// saves a fill launch per sort.
template <typename K>
__global__ __launch_bounds__(256) void k_rs_hist(const K* __restrict__ keys, uint32_t n, int passes, uint32_t chunk,
                                                 uint32_t* __restrict__ hist, uint32_t copies,
                                                 uint32_t* __restrict__ zero, size_t zero_words) {
  constexpr uint32_t D = 256;
  __shared__ uint32_t s[kMaxPasses * D];
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < zero_words; i += (size_t)gridDim.x * 256) zero[i] = 0u;
  for (uint32_t i = threadIdx.x; i < (uint32_t)passes * D; i += 256) s[i] = 0;
  __syncthreads();
  const size_t b0 = (size_t)blockIdx.x * chunk;
  const size_t b1 = b0 + chunk < (size_t)n ? b0 + chunk : (size_t)n;
  for (size_t i0 = b0; i0 < b1; i0 += 256 * kHistUnroll) {
    K k[kHistUnroll];
    bool ok[kHistUnroll];
#pragma unroll
    for (int u = 0; u < kHistUnroll; ++u) {
      const size_t i = i0 + (size_t)u * 256 + threadIdx.x;
      ok[u] = i < b1;
      k[u] = ok[u] ? keys[i] : (K)0;
    }
#pragma unroll
    for (int u = 0; u < kHistUnroll; ++u) {
      const uint64_t active = __ballot(ok[u]);
      if (!ok[u]) continue;
      for (int p = 0; p < passes; ++p) {
        const uint32_t d = (uint32_t)(k[u] >> (8 * p)) & (D - 1u);
        const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);
        if (__ballot(d == d0) == active) {
          if (__lane_id() == (uint32_t)__builtin_ctzll(active)) atomicAdd(&s[p * D + d0], (uint32_t)__popcll(active));
        } else {
          atomicAdd(&s[p * D + d], 1u);
        }
      }
    }
  }
  __syncthreads();
  uint32_t* g = hist + (size_t)(blockIdx.x % copies) * passes * D;
  for (uint32_t i = threadIdx.x; i < (uint32_t)passes * D; i += 256) {
    uint32_t c = s[i];
    if (c) atomicAdd(&g[i], c);
  }
}

// Stable ranks of a wave's keys (kIt per lane, iteration j of lane l being the
// wave's key 64 j + l) among its keys of the same digit, and the wave's digit
// counts in cnt (zero before). Each lane ORs its bit into its digit's mask and
// reads it back: the lanes that share the digit. The last of them advances the
// digit's counter and clears the mask. wmask: the wave's 256 zero words, left zero.
template <typename K, int kIt>
__device__ __forceinline__ void wave_ranks(const K (&key)[kIt], const bool (&valid)[kIt], int shift,
                                           uint64_t* __restrict__ wmask, uint32_t* __restrict__ cnt,
                                           uint32_t (&rank)[kIt]) {
  const uint64_t my_bit = 1ull << __lane_id(), lower_lanes = my_bit - 1;
#pragma unroll
  for (int j = 0; j < kIt; ++j) {
    const uint32_t d = (uint32_t)(key[j] >> shift) & 0xFFu;
    if (valid[j]) __hip_atomic_fetch_or(wmask + d, my_bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __builtin_amdgcn_wave_barrier();
    const uint64_t peers =
        valid[j] ? __hip_atomic_load(wmask + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0ull;
    const uint32_t lower = (uint32_t)__popcll(peers & lower_lanes);
    const uint32_t all = (uint32_t)__popcll(peers);
    const uint32_t old = cnt[d];
    rank[j] = old + lower;
    __builtin_amdgcn_wave_barrier();
    if (valid[j] && lower + 1 == all) {
      cnt[d] = old + all;
      __hip_atomic_store(wmask + d, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// One pass over one tile of kThreads * kIt keys. The tile's keys are ranked stably
// per digit and moved to their place in the tile's digit order in LDS before
// the look-back, so their registers are free while it waits; the values are
// loaded during the look-back and follow through the same LDS buffer once the
// keys are out, so a workgroup holds a tile of keys in LDS, not keys and values.
// kGroups (fewer than 2^21 keys): status holds a row of words per tile, then
// one per group of tiles, all tagged with the pass, so that what the pass
// before left counts as unpublished. Otherwise a row per tile, and next is the
// other buffer, which this pass zeroes for the next (NULL after the last).
template <typename K, bool kVals, int kIt, bool kGroups>
__global__ __launch_bounds__(kThreads) void k_rs_scatter(const K* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                         K* __restrict__ kout, uint32_t* __restrict__ vout, uint32_t n,
                                                         int pass, const uint32_t* __restrict__ hist,
                                                         uint32_t copies, uint32_t copy_words,
                                                         uint32_t* __restrict__ status, uint32_t* __restrict__ next,
                                                         uint32_t* __restrict__ err) {
  constexpr int kTileT = kThreads * kIt, kWaveTileT = 64 * kIt;  // keys per tile and per wave
  constexpr uint32_t D = 256;
  // words: flag (2 bits), with kGroups the pass's tag (4 bits, not 0), count
  constexpr uint32_t kCount = kGroups ? (1u << 26) - 1u : kCountMask;
  const uint32_t tag = kGroups ? (uint32_t)(pass + 1) << 26 : 0u;
  const int shift = 8 * pass;
  __shared__ uint32_t s_cnt[kWaves][D];
  __shared__ uint32_t s_gbase[D];
  __shared__ uint32_t s_tmp[kWaves];
  // while ranking, s_buf holds 256 64-bit lane masks per wave
  constexpr int kBuf = sizeof(K) * kTileT >= sizeof(uint64_t) * kWaves * D ? kTileT
                                                                          : (int)(sizeof(uint64_t) * kWaves * D / sizeof(K));
  __shared__ K s_buf[kBuf];

  const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  uint64_t* s_mask = reinterpret_cast<uint64_t*>(s_buf);
  for (uint32_t i = tid; i < kWaves * D; i += kThreads) {
    (&s_cnt[0][0])[i] = 0;
    s_mask[i] = 0;
  }
  const uint32_t tile = blockIdx.x, group = tile / kGroup, place = tile % kGroup;
  const size_t base = (size_t)tile * kTileT;
  const size_t wbase = base + (size_t)wave * kWaveTileT;
  uint32_t* gstatus = status + (size_t)gridDim.x * D;
  if (!kGroups && next && tid < D) next[(size_t)tile * D + tid] = 0u;
  K key[kIt];
  bool valid[kIt];
  uint32_t rank[kIt];
#pragma unroll
  for (int j = 0; j < kIt; ++j) {
    size_t idx = wbase + (size_t)j * 64 + lane;
    valid[j] = idx < n;
    key[j] = valid[j] ? kin[idx] : (K)0;
  }
  __syncthreads();
  wave_ranks<K, kIt>(key, valid, shift, s_mask + wave * 256, s_cnt[wave], rank);
  __syncthreads();

  // Per digit (thread d < 256): the tile's count, published at once for the
  // look-back of later tiles, and each wave's start within the digit's run.
  const uint32_t d = tid;
  const bool mine = tid < D;
  uint32_t total[1] = {0u}, local[1], counted[1] = {0u}, global[1];
  if (mine) {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t c = s_cnt[w][d];
      s_cnt[w][d] = total[0];
      total[0] += c;
    }
    rk::atomic_store_relaxed(status + (size_t)tile * D + d, (!kGroups && tile == 0 ? kInc : kAgg) | tag | total[0]);
    // all loads in flight: one after the other, copies cost a pass on 100,000 keys 1 us
    // of its 8 (a sort of them 47.6 against 42.8 us; 1M 67 against 62)
    uint32_t part[kMaxCopies];
#pragma unroll
    for (uint32_t c = 0; c < kMaxCopies; ++c) part[c] = hist[(size_t)min(c, copies - 1u) * copy_words + d];
#pragma unroll
    for (uint32_t c = 0; c < kMaxCopies; ++c) counted[0] += c < copies ? part[c] : 0u;
  }
  block_excl_scan<kThreads, 1>(total, local, s_tmp);
  if (mine) {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s_cnt[w][d] += local[0];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kIt; ++j) {
    if (valid[j]) {
      rank[j] += s_cnt[wave][(uint32_t)(key[j] >> shift) & 0xFFu];  // position in the tile's digit order
      s_buf[rank[j]] = key[j];
    }
  }
  uint32_t val[kIt];
  if (kVals) {
#pragma unroll
    for (int j = 0; j < kIt; ++j) val[j] = valid[j] ? vin[wbase + (size_t)j * 64 + lane] : 0u;
  }
  block_excl_scan<kThreads, 1>(counted, global, s_tmp);

  if (mine) {
    // a word of this pass: its flag (0: not published yet)
    auto flag_of = [&](uint32_t w) { return ((w ^ tag) & ~(kAgg | kInc | kCount)) == 0u ? w & (kAgg | kInc) : 0u; };
    uint32_t prefix = 0, spins = 0;
    if (kGroups && place > 0u) {
      // the tiles before this one in its group, all in flight; again until all are published
      for (;;) {
        uint32_t sv[kGroup - 1];
#pragma unroll
        for (uint32_t w = 0; w < kGroup - 1; ++w)
          sv[w] = w < place ? rk::atomic_load_relaxed(status + (size_t)(group * kGroup + w) * D + d) : kAgg | tag;
        bool ready = true;
        prefix = 0;
#pragma unroll
        for (uint32_t w = 0; w < kGroup - 1; ++w) {
          ready = ready && flag_of(sv[w]) != 0u;
          prefix += sv[w] & kCount;
        }
        if (ready) break;
        if (++spins > kSpinLimit) {
          atomicOr(err, (uint32_t)RK_FLAG_SPIN_LIMIT);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    // The rows looked back over: the groups', or the tiles'. The inclusive
    // prefix goes out for a group by its last tile, or for every tile.
    const uint32_t* rows = kGroups ? gstatus : status;
    const uint32_t row = kGroups ? group : tile;
    const bool publish = !kGroups || place == kGroup - 1u;
    uint32_t* out = (kGroups ? gstatus : status) + (size_t)row * D + d;
    if (kGroups && publish)
      rk::atomic_store_relaxed(out, (group == 0u ? kInc : kAgg) | tag | ((prefix + total[0]) & kCount));
    // Decoupled look-back, kLook predecessors' words per round trip: add counts
    // from row j down until an inclusive prefix; stop the round at a row that
    // has published nothing yet and reload from there.
    if (row > 0u) {
      int32_t j = (int32_t)row - 1;
      for (;;) {
        uint32_t sv[kLook];
#pragma unroll
        for (int w = 0; w < kLook; ++w)
          sv[w] = (j - w >= 0) ? rk::atomic_load_relaxed(rows + (size_t)(j - w) * D + d) : kInc | tag;
        int used = 0;
        bool inc = false, stalled = false;
#pragma unroll
        for (int w = 0; w < kLook; ++w) {
          if (inc || stalled) continue;
          const uint32_t flag = flag_of(sv[w]);
          if (flag == 0) {
            stalled = true;
            continue;
          }
          prefix += sv[w] & kCount;
          ++used;
          if (flag == kInc) inc = true;
        }
        if (inc) break;
        j -= used;
        if (used == 0) {
          if (++spins > kSpinLimit) {
            atomicOr(err, (uint32_t)RK_FLAG_SPIN_LIMIT);
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
      }
      if (publish) rk::atomic_store_relaxed(out, kInc | tag | ((prefix + total[0]) & kCount));
    }
    s_gbase[d] = global[0] + prefix - local[0];
  }
  __syncthreads();

  const uint32_t tile_n = (n - base) < (size_t)kTileT ? (uint32_t)(n - base) : (uint32_t)kTileT;
  uint32_t opos[kIt];
#pragma unroll
  for (int m = 0; m < kIt; ++m) {
    const uint32_t i = tid + (uint32_t)m * kThreads;
    opos[m] = 0xFFFFFFFFu;
    if (i < tile_n) {
      const K k = s_buf[i];
      const uint32_t dd = (uint32_t)(k >> shift) & 0xFFu;
      const size_t o = (size_t)s_gbase[dd] + i;
      if (o < n) {  // always true unless the look-back failed (err is set then)
        kout[o] = k;
        opos[m] = (uint32_t)o;
      }
    }
  }
  if (kVals) {
    uint32_t* s_val = reinterpret_cast<uint32_t*>(s_buf);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kIt; ++j) {
      if (valid[j]) s_val[rank[j]] = val[j];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kIt; ++m) {
      const uint32_t i = tid + (uint32_t)m * kThreads;
      if (i < tile_n && opos[m] != 0xFFFFFFFFu) vout[opos[m]] = s_val[i];
    }
  }
}

// All passes of a small sort in one workgroup: its keys and values stay in
// registers and change places through LDS, with the scatter kernel's stable
// ranks. 16 waves, kIt keys per lane. In place when kin is kout (every load
// comes before every store). clear (may be NULL) is set to 0.
constexpr int kOneThreads = 1024, kOneWaves = kOneThreads / 64;
template <typename K, bool kVals, int kIt>
__global__ __launch_bounds__(kOneThreads) void k_sort_one(const K* kin, const uint32_t* vin, K* kout, uint32_t* vout,
                                                          uint32_t n, int passes, uint32_t* clear) {
  constexpr uint32_t D = 256;
  __shared__ uint32_t s_cnt[kOneWaves][D];
  __shared__ uint32_t s_tmp[kOneWaves];
  __shared__ K s_buf[kOneThreads * kIt];
  __shared__ uint64_t s_mask[kOneWaves * D];  // zero between the passes
  uint32_t* s_val = reinterpret_cast<uint32_t*>(s_buf);
  const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (clear && tid == 0) *clear = 0u;
  for (uint32_t i = tid; i < kOneWaves * D; i += kOneThreads) s_mask[i] = 0;
  const uint32_t first = wave * (64u * kIt) + lane;
  K key[kIt];
  uint32_t val[kIt], rank[kIt];
  bool valid[kIt];
#pragma unroll
  for (int j = 0; j < kIt; ++j) {
    const uint32_t i = first + 64u * j;
    valid[j] = i < n;
    key[j] = valid[j] ? kin[i] : (K)0;
    val[j] = kVals && valid[j] ? vin[i] : 0u;
  }
  for (int p = 0; p < passes; ++p) {
    const int shift = p * 8;
    for (uint32_t i = tid; i < kOneWaves * D; i += kOneThreads) (&s_cnt[0][0])[i] = 0;
    __syncthreads();
    wave_ranks<K, kIt>(key, valid, shift, s_mask + wave * D, s_cnt[wave], rank);
    __syncthreads();
    uint32_t total[1] = {0u}, excl[1];
    if (tid < D) {
#pragma unroll
      for (int w = 0; w < kOneWaves; ++w) total[0] += s_cnt[w][tid];
    }
    block_excl_scan<kOneThreads, 1>(total, excl, s_tmp);
    if (tid < D) {
      uint32_t run = excl[0];
#pragma unroll
      for (int w = 0; w < kOneWaves; ++w) {
        const uint32_t c = s_cnt[w][tid];
        s_cnt[w][tid] = run;
        run += c;
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kIt; ++j) {
      if (valid[j]) {
        rank[j] += s_cnt[wave][(uint32_t)(key[j] >> shift) & (D - 1u)];
        s_buf[rank[j]] = key[j];
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kIt; ++j)
      if (valid[j]) key[j] = s_buf[first + 64u * j];
    if (kVals) {
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kIt; ++j)
        if (valid[j]) s_val[rank[j]] = val[j];
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kIt; ++j)
        if (valid[j]) val[j] = s_val[first + 64u * j];
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < kIt; ++j) {
    if (valid[j]) {
      kout[first + 64u * j] = key[j];
      if (kVals) vout[first + 64u * j] = val[j];
    }
  }
}

__global__ __launch_bounds__(256) void k_sort_clear(uint32_t* __restrict__ head, size_t head_words,
                                                    uint32_t* __restrict__ status, size_t status_words,
                                                    uint32_t* __restrict__ info) {
  const size_t stride = (size_t)gridDim.x * 256, t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (info && t < RK_INFO_WORDS) info[t] = 0u;
  for (size_t i = t; i < head_words; i += stride) head[i] = 0u;
  for (size_t i = t; i < status_words; i += stride) status[i] = 0u;
}

template <typename K, bool kVals>
__global__ __launch_bounds__(256) void k_copy_back(const K* __restrict__ ks, const uint32_t* __restrict__ vs,
                                                   K* __restrict__ kd, uint32_t* __restrict__ vd, uint32_t n) {
  size_t stride = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    kd[i] = ks[i];
    if (kVals) vd[i] = vs[i];
  }
}

// The reference's middle size class (CUDA_bitonicSortGeneral.cu:39-169):
// each full 128-element chunk goes through the bitonic network on (key, value);
// the partial last chunk is sorted stably (odd-even transposition in the
// reference, :107-162). A stable key sort afterwards reproduces the order of
// the reference's stable '<=' merges (:172-481).
__global__ __launch_bounds__(128) void k_bitonic_chunks(uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                        uint32_t n) {
  __shared__ uint32_t sk[128], sv[128];
  const uint32_t t = threadIdx.x, o = blockIdx.x * 128u;
  const uint32_t size = (n - o) < 128u ? (n - o) : 128u;
  if (size <= 1) return;
  if (t < size) { sk[t] = keys[o + t]; sv[t] = vals[o + t]; }
  __syncthreads();
  if (size == 128) {
    for (uint32_t i = 2; i <= 128; i <<= 1) {
      for (uint32_t j = i >> 1; j > 0; j >>= 1) {
        uint32_t ixj = t ^ j;
        if (ixj > t) {
          uint32_t ka = sk[t], kb = sk[ixj];
          bool sw = ((t & i) == 0) ? (ka > kb) : (ka < kb);
          if (sw) {
            uint32_t va = sv[t], vb = sv[ixj];
            sk[t] = kb; sk[ixj] = ka; sv[t] = vb; sv[ixj] = va;
          }
        }
        __syncthreads();
      }
    }
    keys[o + t] = sk[t];
    vals[o + t] = sv[t];
  } else if (t < size) {
    uint32_t k = sk[t], r = 0;
    for (uint32_t u = 0; u < size; ++u) r += (sk[u] < k || (sk[u] == k && u < t)) ? 1u : 0u;
    keys[o + r] = k;
    vals[o + r] = sv[t];
  }
}

// Stable sort of at most 512 keys (and values) in one workgroup: each thread
// ranks its key by counting the smaller keys and the equal keys before it. This
// is the order of the reference's odd-even transposition sort, which swaps only
// on '>' (CUDA_bubbleSort512.cu:42-96) and is therefore stable. 'init' takes
// the values to be 0..n-1 (kernel_bubbleSortInit, CUDA_bubbleSort512.cu:98-104).
// 'clear' (may be NULL) is set to 0. Every global read happens before the
// barrier and every write after it, so the sort is in place.
constexpr uint32_t kSmallSort = 512;
__global__ __launch_bounds__(512) void k_small_sort(uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                    uint32_t n, int init, uint32_t* __restrict__ clear) {
  __shared__ uint32_t sk[kSmallSort];
  const uint32_t t = threadIdx.x;
  if (clear && t == 0) *clear = 0u;
  uint32_t k = 0, v = 0;
  if (t < n) {
    k = keys[t];
    sk[t] = k;
    if (vals) v = init ? t : vals[t];
  }
  __syncthreads();
  if (t < n) {
    uint32_t r = 0;
    for (uint32_t u = 0; u < n; ++u) {
      const uint32_t x = sk[u];
      r += (x < k || (x == k && u < t)) ? 1u : 0u;
    }
    keys[r] = k;
    if (vals) vals[r] = v;
  }
}

__global__ __launch_bounds__(256) void k_iota(uint32_t* __restrict__ v, uint32_t n) {
  size_t stride = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) v[i] = (uint32_t)i;
}

inline int items_of(uint32_t n) {
  return (size_t)n < kSmallTilesBelow ? kItemsSmall : ((size_t)n < kMidTilesBelow ? kItemsMid : kItems);
}
inline uint32_t tiles_of(uint32_t n, int items) {
  const uint32_t tile = (uint32_t)(kThreads * items);
  return (uint32_t)(((size_t)n + tile - 1) / tile);
}
// The error word of a sort called with this workspace: its first 4 bytes.
inline uint32_t* ws_flags_word(void* ws, size_t ws_bytes) {
  return (ws && ws_bytes >= 4) ? static_cast<uint32_t*>(ws) : nullptr;
}
inline rk_status clear_ws_flags(hipStream_t st, void* ws, size_t ws_bytes) {
  uint32_t* w = ws_flags_word(ws, ws_bytes);
  return w ? rk_fill_u32(reinterpret_cast<rk_stream>(st), w, 1, 0u) : RK_SUCCESS;
}
rk_status launch_small_sort(hipStream_t st, uint32_t* keys, uint32_t* vals, uint32_t n, int init, uint32_t* clear) {
  hipLaunchKernelGGL(k_small_sort, dim3(1), dim3(kSmallSort), 0, st, keys, vals, n, init, clear);
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}
inline unsigned grid_for(size_t n, size_t per_block, unsigned cap) {
  size_t g = (n + per_block - 1) / per_block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}

}  // namespace

// Size of the workspace for a sort of 'length' keys of 'key_bytes' bytes.
extern "C" size_t rk_sort_workspace_size(uint32_t length, uint32_t key_bytes) {
  size_t n = length ? length : 1;
  const size_t tile = (size_t)kThreads * (n < kMidTilesBelow ? kItemsMid : kItems), T = (n + tile - 1) / tile;
  size_t P = key_bytes >= 8 ? 8 : 4;
  return rk_align_up(P * 256 * 4 + P * 4 + 4 + P * T * 256 * 4) + rk_align_up(n * (key_bytes >= 8 ? 8 : 4)) +
         rk_align_up(n * 4) + 1024;
}

// The look-back words count keys in 30 bits, so n < 2^30.
template <typename K>
rk_status rk_sort_plan(uint32_t n, int bits, bool anywhere, K* keys, uint32_t* vals, void* ws, size_t ws_bytes,
                       RkSortPlan<K>& p) {
  if (n >= kAgg) return RK_ERROR_UNSUPPORTED;
  if (!keys || bits <= 0 || bits > (int)sizeof(K) * 8) return RK_ERROR_INVALID_VALUE;
  p.n = n;
  p.one = n <= kOneMax;
  p.passes = (bits + 7) / 8;
  p.dst = p.src = keys;
  p.vdst = p.vsrc = vals;
  // rk_sort_workspace_size has one count and one status row per pass and tile of
  // 4096 or 8192 keys: room for these copies of the counts and rows. A caller's
  // smaller workspace may still have room for fewer: one copy, tiles of 8192 keys
  // and two rows each, which fit wherever 'least_ws' bytes do.
  auto fits = [&](int items, bool copies) {
    const bool groups = items != kItems;
    p.items = items;
    p.tiles = tiles_of(n, items);
    p.copies = copies ? std::min(kMaxCopies, 1u + p.tiles / 8u) : 1u;
    p.head_words = p.one ? 1 : 1 + (size_t)p.copies * p.passes * 256;
    p.status_words = p.one ? 0 : ((size_t)p.tiles + (groups ? (p.tiles + kGroup - 1) / kGroup : 0)) * 256;
    RkArena ar(ws, ws_bytes);
    p.head = ar.take<uint32_t>(p.head_words + (groups || p.passes < 2 ? 1 : 2) * p.status_words);
    if (!p.head) return false;
    p.status = p.head + p.head_words;
    if (p.one) return true;
    p.alt = ar.take<K>(n);
    p.valt = vals ? ar.take<uint32_t>(n) : nullptr;
    return p.alt && (!vals || p.valt);
  };
  if (!fits(items_of(n), true) && !fits(kItems, false)) return RK_ERROR_WORKSPACE;
  if (p.one) return RK_SUCCESS;
  if (anywhere && (p.passes & 1)) {
    p.src = p.alt;
    p.vsrc = p.valt;
  }
  return RK_SUCCESS;
}

template <typename K>
rk_status rk_sort_clear(hipStream_t st, const RkSortPlan<K>& p, uint32_t* info) {
  const size_t words = p.head_words + p.status_words;
  hipLaunchKernelGGL(k_sort_clear, dim3(grid_for(words, 256 * 4, 1024)), dim3(256), 0, st, p.head, p.head_words,
                     p.status, p.status_words, info);
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

namespace {

template <typename K>
rk_status launch_one(hipStream_t st, const RkSortPlan<K>& p, uint32_t* clear) {
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kOneThreads), 0, st, p.src, p.vsrc, p.dst, p.vdst, p.n, p.passes, clear);
  };
  static_assert(kOneMax == 4 * kOneThreads, "4 keys per thread at most");
  const bool two = p.n <= 2 * kOneThreads;
  if (p.vsrc) go(two ? k_sort_one<K, true, 2> : k_sort_one<K, true, 4>);
  else go(two ? k_sort_one<K, false, 2> : k_sort_one<K, false, 4>);
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

}  // namespace

template <typename K>
rk_status rk_sort_run(hipStream_t st, const RkSortPlan<K>& p, bool counted, uint32_t* err) {
  // One key is in its place: sorting it had made a tree of one face cost 21.8 us instead
  // of 18.7, a sorted trace of one ray 22.2 instead of 18.4.
  if (p.n <= 1)
    return err || counted ? RK_SUCCESS : rk_fill_u32(reinterpret_cast<rk_stream>(st), p.head, 1, 0u);
  if (p.one) return launch_one<K>(st, p, err || counted ? nullptr : p.head);
  uint32_t* hist = p.head + 1;
  if (!counted) {
    rk_status s = rk_fill_u32(reinterpret_cast<rk_stream>(st), p.head, p.head_words, 0u);
    if (s != RK_SUCCESS) return s;
    const unsigned blocks = grid_for(p.n, kHistKeysPerBlock, kHistMaxBlocks);
    const uint32_t chunk = (uint32_t)(((size_t)p.n + blocks - 1) / blocks);
    hipLaunchKernelGGL(k_rs_hist<K>, dim3(blocks), dim3(256), 0, st, p.src, p.n, p.passes, chunk, hist, p.copies,
                       p.status, p.status_words);
    RK_CHECK_LAUNCH();
  }
  if (!err) err = p.head;
  K *ks = p.src, *kd = p.src == p.dst ? p.alt : p.dst;
  uint32_t *vs = p.vsrc, *vd = p.vsrc == p.vdst ? p.valt : p.vdst;
  for (int i = 0; i < p.passes; ++i) {
    const bool groups = p.items != kItems;
    uint32_t* status = p.status + (groups ? 0 : (i & 1) * p.status_words);
    uint32_t* next = !groups && i + 1 < p.passes ? p.status + ((i + 1) & 1) * p.status_words : nullptr;
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(p.tiles), dim3(kThreads), 0, st, ks, vs, kd, vd, p.n, i, hist + (size_t)i * 256,
                         p.copies, (uint32_t)p.passes * 256u, status, next, err);
    };
    if (p.vsrc) {
      if (p.items == kItemsSmall) go(k_rs_scatter<K, true, kItemsSmall, true>);
      else if (groups) go(k_rs_scatter<K, true, kItemsMid, true>);
      else go(k_rs_scatter<K, true, kItems, false>);
    } else {
      if (p.items == kItemsSmall) go(k_rs_scatter<K, false, kItemsSmall, true>);
      else if (groups) go(k_rs_scatter<K, false, kItemsMid, true>);
      else go(k_rs_scatter<K, false, kItems, false>);
    }
    RK_CHECK_LAUNCH();
    std::swap(ks, kd);
    std::swap(vs, vd);
  }
  if (ks != p.dst) {
    if (p.vsrc)
      hipLaunchKernelGGL((k_copy_back<K, true>), dim3(grid_for(p.n, 256 * 8, 4096)), dim3(256), 0, st, ks, vs, p.dst,
                         p.vdst, p.n);
    else
      hipLaunchKernelGGL((k_copy_back<K, false>), dim3(grid_for(p.n, 256 * 8, 4096)), dim3(256), 0, st, ks,
                         (const uint32_t*)nullptr, p.dst, (uint32_t*)nullptr, p.n);
    RK_CHECK_LAUNCH();
  }
  return RK_SUCCESS;
}

#define RK_SORT_INSTANCES(K)                                                                                      \
  template rk_status rk_sort_plan<K>(uint32_t, int, bool, K*, uint32_t*, void*, size_t, RkSortPlan<K>&);          \
  template rk_status rk_sort_clear<K>(hipStream_t, const RkSortPlan<K>&, uint32_t*);                              \
  template rk_status rk_sort_run<K>(hipStream_t, const RkSortPlan<K>&, bool, uint32_t*);
RK_SORT_INSTANCES(uint32_t)
RK_SORT_INSTANCES(uint64_t)
#undef RK_SORT_INSTANCES

// The workspace that a sort of n > 1 keys asks for whichever way it goes, the
// one-workgroup sort included: a count and a status row per pass and tile of 4096 or
// 8192 keys, and the other halves of the keys and values.
template <typename K>
static size_t least_ws(uint32_t n, int passes, bool vals) {
  const size_t T = tiles_of(n, n < kMidTilesBelow ? kItemsMid : kItems), P = (size_t)passes, keys = n * sizeof(K);
  return rk_align_up((1 + P * 256 + P * T * 256) * 4) + (vals ? rk_align_up(keys) + (size_t)n * 4 : keys);
}

// Sorts keys (and values, when not NULL) stably on their low 'bits' bits. 'err'
// (device, may be NULL) receives RK_FLAG_SPIN_LIMIT on a look-back timeout; when
// it is NULL the first word of 'ws' does, cleared by this call.
template <typename K>
static rk_status sort_keys(hipStream_t st, K* keys, uint32_t* vals, uint32_t n, int bits, void* ws, size_t ws_bytes,
                           uint32_t* err) {
  if (n >= kAgg) return RK_ERROR_UNSUPPORTED;
  if (n <= 1) return err ? RK_SUCCESS : clear_ws_flags(st, ws, ws_bytes);
  RkSortPlan<K> p;
  rk_status s = rk_sort_plan<K>(n, bits, false, keys, vals, ws, ws_bytes, p);
  if (s == RK_SUCCESS && ws_bytes < least_ws<K>(n, p.passes, vals != nullptr)) s = RK_ERROR_WORKSPACE;
  return s == RK_SUCCESS ? rk_sort_run<K>(st, p, false, err) : s;
}

// The reference tie order of CUDA_radixSortGeneral (CUDA_radixSortGeneral.cu:397-482):
//  length <= 512 (bubble, CUDA_bubbleSort512.cu): stable by key;
//  length <= byte_depth*8192 (bitonic general): network order inside each
//   128-chunk, then stable by key;
//  larger (LSD radix on the low byte_depth bytes): stable by those bytes.
rk_status rk_sort_general_impl(hipStream_t st, uint32_t* keys, uint32_t* indices, uint32_t length,
                               uint32_t bit_depth, int init_indices, void* ws, size_t ws_bytes, uint32_t* err) {
  if (bit_depth == 0 || bit_depth > 32) return RK_ERROR_INVALID_VALUE;
  if (length >= kAgg) return RK_ERROR_UNSUPPORTED;
  if (length == 0) return err ? RK_SUCCESS : clear_ws_flags(st, ws, ws_bytes);
  if (!keys || !indices) return RK_ERROR_INVALID_VALUE;
  const uint32_t byte_depth = 1 + (bit_depth - 1) / 8;
  if (length <= kSmallSort)
    return launch_small_sort(st, keys, indices, length, init_indices, err ? nullptr : ws_flags_word(ws, ws_bytes));
  if (init_indices) {
    hipLaunchKernelGGL(k_iota, dim3(grid_for(length, 256 * 8, 4096)), dim3(256), 0, st, indices, length);
    RK_CHECK_LAUNCH();
  }
  if (length <= byte_depth * 8192u) {
    hipLaunchKernelGGL(k_bitonic_chunks, dim3((length + 127) / 128), dim3(128), 0, st, keys, indices, length);
    RK_CHECK_LAUNCH();
    return sort_keys<uint32_t>(st, keys, indices, length, 32, ws, ws_bytes, err);
  }
  return sort_keys<uint32_t>(st, keys, indices, length, 8 * (int)byte_depth, ws, ws_bytes, err);
}

extern "C" rk_status rk_radix_sort_general(rk_stream stream, uint32_t* keys, uint32_t* indices, uint32_t length,
                                           uint32_t bit_depth, int init_indices, void* ws, size_t ws_bytes) {
  return rk_sort_general_impl(rk_hip_stream(stream), keys, indices, length, bit_depth, init_indices, ws, ws_bytes,
                              nullptr);
}

// CUDA_radixSort (CUDA_radixSort.cu:357-392): values only, sorted on the low
// byte_depth bytes (the bitonic class compares whole values; for values below
// 2^(8*byte_depth) both agree, and equal values are indistinguishable).
extern "C" rk_status rk_radix_sort(rk_stream stream, uint32_t* values, uint32_t length, uint32_t bit_depth, void* ws,
                                   size_t ws_bytes) {
  if (bit_depth == 0 || bit_depth > 32) return RK_ERROR_INVALID_VALUE;
  if (length >= kAgg) return RK_ERROR_UNSUPPORTED;
  if (length > 1 && !values) return RK_ERROR_INVALID_VALUE;
  if (length <= kSmallSort)
    return launch_small_sort(rk_hip_stream(stream), values, nullptr, length, 0, ws_flags_word(ws, ws_bytes));
  const uint32_t byte_depth = 1 + (bit_depth - 1) / 8;
  int passes = (length <= byte_depth * 8192u) ? 4 : (int)byte_depth;
  return sort_keys<uint32_t>(rk_hip_stream(stream), values, nullptr, length, 8 * passes, ws, ws_bytes, nullptr);
}

extern "C" rk_status rk_radix_sort_pairs_u64(rk_stream stream, uint64_t* keys, uint32_t* values, uint32_t length,
                                             uint32_t bit_depth, void* ws, size_t ws_bytes) {
  if (bit_depth == 0 || bit_depth > 64) return RK_ERROR_INVALID_VALUE;
  int passes = (int)(1 + (bit_depth - 1) / 8);
  return sort_keys<uint64_t>(rk_hip_stream(stream), keys, values, length, 8 * passes, ws, ws_bytes, nullptr);
}

// template <typename T> void CUDA_bitonicSort(T* values, uint length),
// samples/09_how_to_use_a_sorter.cpp:39-40 / CUDA_bitonicSort.cu:402-518
// (instantiated for unsigned int, :523-537). The values are their own keys, so
// any correct sort gives the reference's result: at most 512 values in one
// workgroup, more by the radix passes over all 32 bits.
extern "C" rk_status rk_bitonic_sort(rk_stream stream, uint32_t* values, uint32_t length, void* ws, size_t ws_bytes) {
  if (length >= kAgg) return RK_ERROR_UNSUPPORTED;
  if (length > 1 && !values) return RK_ERROR_INVALID_VALUE;
  hipStream_t st = rk_hip_stream(stream);
  if (length <= kSmallSort) return launch_small_sort(st, values, nullptr, length, 0, ws_flags_word(ws, ws_bytes));
  return sort_keys<uint32_t>(st, values, nullptr, length, 32, ws, ws_bytes, nullptr);
}

// template <typename K, typename V> void CUDA_bitonicSortGeneral(K* keys, V* values, uint length),
// samples/09_how_to_use_a_sorter.cpp:42-43 / CUDA_bitonicSortGeneral.cu:504-690
// (instantiated for <uint, uint>, :694-697), at any length. The reference sorts
// each full 128-element chunk with a bitonic network, the partial last chunk
// by odd-even transposition, then merges chunk pairs and buckets of doubling
// size with stable '<=' merges (:172-481) until one bucket remains, carrying a
// local index array that finally permutes the values. The same order is the
// chunk networks followed by a stable sort on the whole key.
extern "C" rk_status rk_bitonic_sort_general(rk_stream stream, uint32_t* keys, uint32_t* values, uint32_t length,
                                             void* ws, size_t ws_bytes) {
  hipStream_t st = rk_hip_stream(stream);
  if (length >= kAgg) return RK_ERROR_UNSUPPORTED;
  if (length <= 1) return clear_ws_flags(st, ws, ws_bytes);
  if (!keys || !values) return RK_ERROR_INVALID_VALUE;
  hipLaunchKernelGGL(k_bitonic_chunks, dim3((length + 127) / 128), dim3(128), 0, st, keys, values, length);
  RK_CHECK_LAUNCH();
  if (length <= 128) return clear_ws_flags(st, ws, ws_bytes);
  return sort_keys<uint32_t>(st, keys, values, length, 32, ws, ws_bytes, nullptr);
}

// void CUDA_bubbleSort512(uint* keys, uint* indices, uint length, bool init_indices),
// CUDA_radixSortGeneral.cu:27 / CUDA_bubbleSort512.cu:114-167: a stable sort of
// at most 512 (key, index) pairs; init_indices first sets indices[i] = i. The
// reference asserts on length > 512 (:116); here that is RK_ERROR_INVALID_VALUE.
extern "C" rk_status rk_bubble_sort512(rk_stream stream, uint32_t* keys, uint32_t* indices, uint32_t length,
                                       int init_indices) {
  if (length > kSmallSort) return RK_ERROR_INVALID_VALUE;
  if (length == 0) return RK_SUCCESS;
  if (!keys || !indices) return RK_ERROR_INVALID_VALUE;
  return launch_small_sort(rk_hip_stream(stream), keys, indices, length, init_indices, nullptr);
}

// The RK_FLAG_* bits a sort left in the first word of its workspace (waits for 'stream').
extern "C" rk_status rk_workspace_flags(rk_stream stream, const void* ws, uint32_t* flags) {
  if (!ws || !flags) return RK_ERROR_INVALID_VALUE;
  hipStream_t st = rk_hip_stream(stream);
  uint32_t h = 0;
  RK_HIP(hipMemcpyAsync(&h, ws, 4, hipMemcpyDeviceToHost, st));
  RK_HIP(hipStreamSynchronize(st));
  *flags = h;
  return RK_SUCCESS;
}
