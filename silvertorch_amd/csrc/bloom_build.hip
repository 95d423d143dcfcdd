// Bloom index build for gfx950.
//
// Replaces bloom_index_build (bloom_indexer.cpp:26-113 on CPU,
// bloom_indexer_cuda.cu:253-389 and :137-251 / :506-711 on CUDA) with three
// kernels:
//   widths_kernel   one workgroup per bundle of 2048 docs: per-doc term count
//                   (feature_offsets[(d+1)F] - feature_offsets[dF]), bundle
//                   max, b = (int64)((double)(max * k) * b_multiplier); also
//                   checks that feature_offsets never decreases.
//   scan_kernel     one workgroup: exclusive prefix sum of the widths into
//                   bundle_b_offsets, plus the totals the host needs.
//   scatter_kernel  one workgroup per part of a bundle (16 of its 32 columns,
//                   fewer where bundles are wide or docs few): clears a tile of
//                   b rows in LDS, hashes every (doc, feature, value) term of
//                   the part (one thread per value, its place from an LDS map
//                   of the slot group), ORs its k bits into the tile with LDS
//                   atomics and stores the tile.  A bundle too wide for the
//                   part's tile goes in passes over fewer columns, one that no
//                   tile holds ORs straight into global memory.
// The reference's per-doc byte signatures and 64-way transpose
// (bloom_indexer_cuda.cu:137-251, ~N*b/8 bytes of scratch) are not needed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>

#include "st_common.hpp"
#include "st_errors.hpp"

namespace st {
int cu_count();

namespace {

constexpr int kWidthThreads = 256;        // of a bundle, many bundles
constexpr int kWidthThreadsFew = 1024;    // of a bundle, few bundles
constexpr int kScanThreads = 1024;
constexpr int kBuildThreads = 1024;     // of a workgroup that takes a whole CU
constexpr int kBuildHalfThreads = 512;  // of two workgroups that share one
constexpr int kLdsBytes = 160 * 1024;
constexpr int kBuildFeatureCache = 64;     // murmur_mix_x of the first feature ids, in LDS
constexpr int kBuildMapBytes = 12288;      // the places of a window's values, in LDS
constexpr int kBuildMapFeatures = 1 << 20; // features that a 32-bit place names
constexpr int kBuildQueueWords = 2 * 64;   // a wave's queue of values with colliding positions, in LDS
constexpr int kBuildStaticLds = 64;        // BundleMod and alignment
constexpr int kBuildRestLds = 256;         // the same and scatter_rest_kernel's list

// stats layout (int64[6]):
//   [0] total rows  [1] max bundle width  [2] non-decreasing violation flag
//   [3] feature_offsets[0]  [4] feature_offsets[N*F]  [5] reserved

// 64-bit min / max (the device library's overloads go through doubles).
__device__ __forceinline__ int64_t lesser(int64_t a, int64_t b) { return a < b ? a : b; }
__device__ __forceinline__ int64_t greater(int64_t a, int64_t b) { return a > b ? a : b; }

__device__ __forceinline__ int64_t wave_max(int64_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const int64_t o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

// Feature counts up to this stage a chunk's offsets in LDS (below).
constexpr int kWidthStageFeatures = 16;
constexpr int kWidthFewFeatures = 7;  // 1,024 docs' offsets within 64 KB of LDS

// Marks a bundle whose offsets decrease somewhere, in the sign of its width.
constexpr int64_t kDecreasing = INT64_MIN;

// One workgroup of T threads per bundle.  256 threads keep eight workgroups on
// a CU when there are many bundles; with fewer bundles than would fill the
// chip so, 1,024 threads take a bundle in a quarter of the dependent steps
// (100,000 docs of 2 features, 49 bundles: 12.3 against 6.1 us).
template <int T>
__global__ __launch_bounds__(T) void widths_kernel(
    const int64_t* __restrict__ offsets, int64_t num_docs, int64_t num_features,
    int64_t k, double b_multiplier, int64_t* __restrict__ bundle_b_offsets) {
  extern __shared__ __attribute__((aligned(16))) int64_t stage[];  // T * F + 1 up to 16 features
  __shared__ int64_t red[T / 64];
  __shared__ int any_bad;
  const int64_t bundle = blockIdx.x;
  const int64_t doc0 = bundle * kDocsPerBundle;
  const int64_t doc1 = lesser(doc0 + kDocsPerBundle, num_docs);
  const int64_t F = num_features;
  if (threadIdx.x == 0) any_bad = 0;
  int bad = 0;
  int64_t best = 0;
  if (F <= kWidthStageFeatures) {
    // Chunks of T docs: the chunk's offsets (F per doc and the next doc's
    // first) are loaded once with coalesced loads into registers, the next
    // chunk's loads are issued before this chunk is evaluated, and the values
    // pass through LDS so that thread t can check that its doc's offsets never
    // decrease and take its count from the first and the last.
    constexpr int kPer = kWidthStageFeatures + 1;  // ns <= kPer * T
    int64_t r[kPer];
    const auto load = [&](int64_t c0) {
      const int64_t ns = lesser(T, doc1 - c0) * F + 1;
      const int64_t* src = offsets + c0 * F;
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int64_t i = threadIdx.x + u * T;
        r[u] = i < ns ? src[i] : 0;
      }
    };
    if (doc0 < doc1) load(doc0);
    for (int64_t c0 = doc0; c0 < doc1; c0 += T) {
      const int64_t nd = lesser(T, doc1 - c0);
      const int64_t ns = nd * F + 1;
      __syncthreads();  // the previous chunk's readers are done with stage
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int64_t i = threadIdx.x + u * T;
        if (i < ns) stage[i] = r[u];
      }
      __syncthreads();
      if (c0 + T < doc1) load(c0 + T);
      if (threadIdx.x < nd) {
        const int64_t* o = stage + threadIdx.x * F;
        for (int64_t f = 0; f < F; ++f) bad |= o[f + 1] < o[f];
        const int64_t cnt = o[F] - o[0];
        best = cnt > best ? cnt : best;
      }
    }
  } else {
    // Wide docs: every offset is read once for the monotonicity check, the
    // doc boundaries again for the counts (L2 hits).
    for (int64_t s = doc0 * F + threadIdx.x; s < doc1 * F; s += T)
      bad |= offsets[s + 1] < offsets[s];
    for (int64_t d = doc0 + threadIdx.x; d < doc1; d += T) {
      const int64_t cnt = offsets[(d + 1) * F] - offsets[d * F];
      best = cnt > best ? cnt : best;
    }
    __syncthreads();  // any_bad is set
  }
  best = wave_max(best);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
  if (__any(bad) && (threadIdx.x & 63) == 0) any_bad = 1;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t m = red[0];
    for (int i = 1; i < T / 64; ++i) m = red[i] > m ? red[i] : m;
    const int64_t b = static_cast<int64_t>(static_cast<double>(m * k) * b_multiplier);
    bundle_b_offsets[bundle + 1] = any_bad ? (b | kDecreasing) : b;
  }
}

// In-place exclusive scan: on entry bundle_b_offsets[i+1] holds width i (its
// sign set where the bundle's offsets decrease).  The stats are stored once,
// with plain stores: they may lie in host memory that the device can write.
__global__ __launch_bounds__(kScanThreads) void scan_kernel(
    const int64_t* __restrict__ offsets, int64_t num_slots, int64_t nb,
    int64_t* __restrict__ bundle_b_offsets, int64_t* __restrict__ stats) {
  __shared__ int64_t part[kScanThreads / 64];
  __shared__ int64_t wide[kScanThreads / 64];
  __shared__ int any_bad;
  const int t = threadIdx.x;
  const int64_t per = (nb + kScanThreads - 1) / kScanThreads;
  const int64_t lo = lesser(t * per, nb);
  const int64_t hi = lesser(lo + per, nb);
  if (t == 0) any_bad = 0;
  int64_t sum = 0, most = 0;
  bool bad = false;
#pragma unroll 8
  for (int64_t i = lo; i < hi; ++i) {
    const int64_t v = bundle_b_offsets[i + 1];
    const int64_t b = v & ~kDecreasing;
    bad |= v < 0;
    most = greater(most, b);
    sum += b;
  }
  // inclusive scan within the wave, then over the waves
  int64_t incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int64_t v = __shfl_up(incl, off, 64);
    if ((t & 63) >= off) incl += v;
  }
  most = wave_max(most);
  if ((t & 63) == 63) part[t >> 6] = incl;
  if ((t & 63) == 0) wide[t >> 6] = most;
  __syncthreads();
  if (__any(bad) && (t & 63) == 0) any_bad = 1;
  int64_t before = 0, total = 0;
  for (int w = 0; w < kScanThreads / 64; ++w) {
    if (w < (t >> 6)) before += part[w];
    total += part[w];
    most = greater(most, wide[w]);
  }
  __syncthreads();
  int64_t run = before + incl - sum;
#pragma unroll 8
  for (int64_t i = lo; i < hi; ++i) {
    run += bundle_b_offsets[i + 1] & ~kDecreasing;
    bundle_b_offsets[i + 1] = run;
  }
  if (t == 0) {
    bundle_b_offsets[0] = 0;
    stats[0] = total;
    stats[1] = most;
    stats[2] = any_bad;
    stats[3] = offsets[0];
    stats[4] = offsets[num_slots];
    stats[5] = 0;
  }
}

// h mod d of a 64-bit hash for a bundle width d < 2^15, without a correction
// step: h / d = hi * (2^32 / d) + lo * (1 / d), and only the fraction of that
// sum matters, in 32 bits.  a ~ frac(2^32 / d) and b ~ 1 / d, rounded up, in
// 64 fraction bits; frac = top 32 bits of hi * a + lo * b (mod 1) plus 2 for the
// two truncated products lies above r / d by less than (d + 4) / 2^32, so
// floor(frac * d / 2^32) is the remainder r itself while d^2 < 2^31.  Five
// 32-bit multiplies and three adds against the general form's seven multiplies
// and two compare-and-subtract corrections.
struct BundleMod {
  uint32_t d, a_lo, a_hi, b_lo, b_hi;
};
constexpr int64_t kBundleModMax = 1 << 15;

__device__ __forceinline__ BundleMod make_bundle_mod(uint32_t d) {
  const uint64_t q = make_fastmod_dev(d).magic;  // floor((2^64 - 1) / d)
  const uint64_t r = 0ull - q * d;               // 2^64 = q d + r, 0 < r <= d
  const uint32_t c = static_cast<uint32_t>((1ull << 32) % d);
  // c * 2^64 / d = c q + c r / d <= c q + r; at most d units of 2^-64 too large
  const uint64_t a = c == 0 ? 0 : c * q + r;
  const uint64_t b = q + 1;
  return {d, static_cast<uint32_t>(a), static_cast<uint32_t>(a >> 32), static_cast<uint32_t>(b),
          static_cast<uint32_t>(b >> 32)};
}

__device__ __forceinline__ uint32_t bundle_mod(uint64_t h, const BundleMod& m) {
  const uint32_t lo = static_cast<uint32_t>(h), hi = static_cast<uint32_t>(h >> 32);
  const uint32_t frac = __umulhi(hi, m.a_lo) + hi * m.a_hi + (__umulhi(lo, m.b_lo) + lo * m.b_hi) + 2u;
  uint32_t r = __umulhi(frac, m.d);
  asm("" : "+v"(r));  // a 32-bit value from here on (not a shifted 64-bit product)
  return r;
}

// The term's row position under one seed: a bundle in an LDS tile uses
// BundleMod, one that ORs into global memory the general form.
struct TileMod {
  BundleMod m;
  __device__ __forceinline__ uint32_t operator()(uint64_t h) const { return bundle_mod(h, m); }
};
struct WideMod {
  FastMod64 m;
  __device__ __forceinline__ uint32_t operator()(uint64_t h) const {
    return static_cast<uint32_t>(fast_mod(h, m));
  }
};

// First K distinct positions murmur(fid, value, seed) % b over seeds
// 0, 1, 2, ... (assign_one_bits_position, bloom_index_util.cuh:183-207).
// b >= K always holds for bundles that have terms (b >= floor(K *
// b_multiplier) >= K), so the loop ends.  The first K seeds are hashed
// unrolled with constant seeds; only when two of them collide (about K^2 / 2b
// of the keys) does the key go on with seeds K, K + 1, ...  rx and ry are the
// feature's and the value's halves of the hash, rotated once per key
// (rotl(mx, 27), rotl(my, 31)); seeds stay far below 2^27 (k distinct positions
// out of b >= k need few more than k seeds).

// The positions of seeds 0 .. K - 1; true when they are distinct.
template <int K, typename Mod>
__device__ __forceinline__ bool first_positions(uint64_t rx, uint64_t ry, const Mod& mod, uint32_t (&found)[K]) {
  bool distinct = true;
#pragma unroll
  for (int j = 0; j < K; ++j) found[j] = mod(murmur_finish_rot(rx, ry, static_cast<uint64_t>(j)));
#pragma unroll
  for (int j = 0; j < K; ++j)
#pragma unroll
    for (int i = 0; i < j; ++i) distinct &= found[i] != found[j];
  return distinct;
}

// first_positions' K positions with repetitions: the first occurrence of each,
// in seed order, then further seeds' as the sequential search takes them.
template <int K, typename Mod>
__device__ __forceinline__ void further_positions(uint64_t rx, uint64_t ry, const Mod& mod, uint32_t (&found)[K]) {
  uint32_t first[K];
#pragma unroll
  for (int j = 0; j < K; ++j) first[j] = found[j];
  int cnt = 0;
#pragma unroll
  for (int j = 0; j < K; ++j) {
    bool dup = false;
#pragma unroll
    for (int i = 0; i < j; ++i) dup |= first[i] == first[j];
    if (!dup) {
#pragma unroll
      for (int s = 0; s < K; ++s)
        if (s == cnt) found[s] = first[j];
      ++cnt;
    }
  }
  uint64_t seed = K;
  while (cnt < K) {
    const uint64_t h = seed < (1ull << 27) ? murmur_finish_rot(rx, ry, seed)
                                           : murmur_finish(rotl64(rx, 37), rotl64(ry, 33), seed);
    ++seed;
    const uint32_t p = mod(h);
    bool dup = false;
#pragma unroll
    for (int j = 0; j < K; ++j) dup |= (j < cnt) && (found[j] == p);
    if (!dup) {
#pragma unroll
      for (int j = 0; j < K; ++j)
        if (j == cnt) found[j] = p;
      ++cnt;
    }
  }
}

// set(p) for each of the term's k positions p.
template <int K, typename Mod, typename Set>
__device__ __forceinline__ void scatter_value(int64_t k, uint64_t rx, int64_t value, const Mod& mod, Set set) {
  const uint64_t my = murmur_mix_y(static_cast<uint64_t>(value));
  if constexpr (K > 0) {
    const uint64_t ry = rotl64(my, 31);
    uint32_t found[K];
    if (!first_positions<K>(rx, ry, mod, found)) further_positions<K>(rx, ry, mod, found);
#pragma unroll
    for (int j = 0; j < K; ++j) set(found[j]);
  } else {  // k above the templated range (k <= 64)
    const uint64_t mx = rotl64(rx, 37);
    uint32_t found[kMaxBuildK];
    int cnt = 0;
    uint64_t seed = 0;
    while (cnt < k) {
      const uint32_t p = mod(murmur_finish(mx, my, seed++));
      bool dup = false;
      for (int j = 0; j < cnt; ++j) dup |= found[j] == p;
      if (!dup) found[cnt++] = p;
    }
    for (int j = 0; j < k; ++j) set(found[j]);
  }
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// LDS of a workgroup besides its tile.
constexpr int fixed_lds(int threads) {
  return 8 * kBuildFeatureCache + kBuildMapBytes + 4 * kBuildQueueWords * (threads / 64);
}

// Words of the tile when a workgroup of `threads` may use `lds` bytes.
constexpr int tile_words_in(int lds, int threads) { return (lds - fixed_lds(threads)) / 4; }

// The tiles of two workgroups a CU, of one, and of one of scatter_rest_kernel.
constexpr int kHalfWords = tile_words_in(kLdsBytes / 2 - kBuildStaticLds, kBuildHalfThreads);
constexpr int kWholeWords = tile_words_in(kLdsBytes - kBuildStaticLds, kBuildThreads);
constexpr int kRestWords = tile_words_in(kLdsBytes - kBuildRestLds, kBuildThreads);

enum ScatterKind { kScatterEven, kScatterPasses, kScatterRest };

struct ScatterArgs {
  const int32_t* feature_ids;
  const int64_t* offsets;
  const int64_t* values;
  int64_t num_values;
  int64_t num_features;
  int64_t num_docs;
  int64_t num_bundles;
  int64_t k;
  const int64_t* bundle_b_offsets;
  unsigned long long* index;
  int lc;          // a workgroup's part of a bundle: 2^lc columns (64 * 2^lc docs)
  int tile_words;  // 32-bit words of its LDS tile
  int rest_words;  // one column's words above which a bundle is scatter_rest_kernel's (0: no such launch)
};

// A tile row: the part's columns as 32-bit words, one word of padding so that
// the rows' words of one column lie on different LDS banks (64 lanes mostly
// share a column and differ in the row).
__host__ __device__ constexpr int tile_stride(int lc) { return (2 << lc) + 1; }
static_assert(kLdsBytes / (4 * tile_stride(0)) < kBundleModMax, "BundleMod takes every tiled width");

// A value's place, as the slot threads record it in the value map: the doc's
// bit (doc % 32) in bits 0-4, its 32-bit word in a tile row in bits 5-9 (the
// high half of a 64-bit column, docs 0-31, is the odd word), the feature above:
// 16 bits hold the first kBuildFeatureCache features, 32 bits the first
// kBuildMapFeatures.
__device__ __forceinline__ uint32_t place(uint32_t d, uint32_t f, uint32_t c0) {
  return (d & 31u) | ((((d >> 5) ^ 1u) - 2 * c0) << 5) | (f << 10);
}
__device__ __forceinline__ uint32_t place_bit(uint32_t m) { return 0x80000000u >> (m & 31u); }
__device__ __forceinline__ uint32_t place_word(uint32_t m) { return (m >> 5) & 31u; }
__device__ __forceinline__ uint32_t place_feature(uint32_t m) { return m >> 10; }

// one(value, place, index, mine) for each value of the part's slots [slot_lo, slot_hi)
// (slot = doc * F + feature, doc relative to the bundle).
// Slots go in groups of kSlots per thread, a group's values in windows of
// the map's entries, for which every slot thread records its place in an LDS map,
// so that the threads then take the window's values one each (all lanes hash,
// value loads coalesce).  A thread's next value is loaded before the current
// one is hashed: the load is an atomic one of wavefront scope, an ordinary
// load whose order the compiler keeps (a plain load it sinks to the value's
// use, where every value waits for memory).
template <typename Place, typename One>
__device__ __forceinline__ void for_each_value(const ScatterArgs& a, const int64_t* offs, uint32_t c0,
                                               int64_t slot_lo, int64_t slot_hi, Place* vmap, One one) {
  constexpr int kSlots = 4;
  constexpr int kWindow = kBuildMapBytes / sizeof(Place);
  const int tid = threadIdx.x, T = blockDim.x;
  const uint32_t F = static_cast<uint32_t>(a.num_features);
  const uint32_t step_d = T / F, step_f = T % F;
  // Values outside [0, num_values) are never read (the host rejects offsets
  // that would point there before launching).
  auto clampv = [&](int64_t v) { return lesser(greater(v, 0), a.num_values); };
  const uint32_t first = static_cast<uint32_t>(slot_lo) + tid;
  uint32_t d = first / F, f = first % F;
  for (int64_t g = slot_lo; g < slot_hi; g += kSlots * T) {
    int64_t v0[kSlots], v1[kSlots];
    uint32_t at[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      // clamped, not predicated: the loads go out together
      const int64_t rel = g + s * T + tid;
      const int64_t* o = offs + lesser(rel, slot_hi - 1);
      v0[s] = o[0];
      v1[s] = rel < slot_hi ? o[1] : o[0];
      at[s] = place(d, f, c0);
      d += step_d;
      f += step_f;
      if (f >= F) {
        f -= F;
        ++d;
      }
    }
    const int64_t gv0 = clampv(offs[g]);
    const int64_t gv1 = clampv(offs[lesser(g + kSlots * T, slot_hi)]);
    for (int64_t w = gv0; w < gv1; w += kWindow) {
      const int n = static_cast<int>(lesser(kWindow, gv1 - w));
      const int64_t* vals = a.values + w;
      auto load = [&](int i) {
        const uint32_t c = static_cast<uint32_t>(i < n ? i : n - 1);
        return __hip_atomic_load(vals + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      };
      int64_t value = load(tid);
      __syncthreads();  // the previous window's readers are done with vmap
#pragma unroll
      for (int s = 0; s < kSlots; ++s) {
        const int lo = static_cast<int>(lesser(greater(v0[s] - w, 0), n));
        const int hi = static_cast<int>(lesser(greater(v1[s] - w, 0), n));
        for (int i = lo; i < hi; ++i) vmap[i] = static_cast<Place>(at[s]);
      }
      __syncthreads();
      // whole waves: the last values' wave runs with its spare lanes repeating
      // the window's last value, `mine` false
      for (int i0 = __builtin_amdgcn_readfirstlane(tid & ~63); i0 < n; i0 += T) {
        const int i = i0 + (tid & 63);
        const int64_t next = load(i + T);
        one(value, vmap[i < n ? i : n - 1], w + i, i < n);
        value = next;
      }
    }
  }
}

// Part `part` of a bundle of b > 0 rows (2^a.lc of its 32 columns): clears the
// tile of the part's rows in LDS, hashes the part's values one per thread, ORs
// their bits into the tile and stores it.  Except in an even index, a bundle
// whose rows the tile does not hold at the part's columns is taken in passes of
// as many as fit (a pass hashes its own docs only, so that no work is done
// twice).  The bits of a bundle that the tile does not hold are ORed in global
// memory, cleared before by this workgroup or (kScatterRest) by scatter_kernel.
// Ends without a barrier.
template <int K, ScatterKind kKind>
__device__ __forceinline__ void scatter_part(const ScatterArgs& a, int64_t bundle, int part, int64_t start,
                                             int64_t b, uint32_t* lds, BundleMod& s_mod) {
  const int tid = threadIdx.x, T = blockDim.x;
  uint64_t* rxc = reinterpret_cast<uint64_t*>(lds);  // rotl(murmur_mix_x(id), 27)
  uint32_t* vmap = lds + 2 * kBuildFeatureCache;
  uint16_t* vmap16 = reinterpret_cast<uint16_t*>(vmap);
  uint32_t* queues = vmap + kBuildMapBytes / 4;
  uint32_t* tile = queues + kBuildQueueWords * (T >> 6);
  int lc = a.lc;  // 2^lc columns a pass
  if constexpr (kKind != kScatterEven) {
    while (lc > 0 && b * tile_stride(lc) > a.tile_words) --lc;
  }
  const bool tiled = b * tile_stride(lc) <= a.tile_words;
  if (!tiled) lc = a.lc;
  const int stride = tile_stride(lc);
  const uint32_t part_begin = static_cast<uint32_t>(part) << a.lc, part_end = part_begin + (1u << a.lc);
  const int64_t F = a.num_features;
  auto rx_id = [&](int64_t f) {
    return rotl64(murmur_mix_x(static_cast<uint64_t>(static_cast<int64_t>(a.feature_ids[f]))), 27);
  };

  const int64_t words = b << lc;
  if (tiled) {
    for (int i = tid; i < static_cast<int>(lesser(F, kBuildFeatureCache)); i += T) rxc[i] = rx_id(i);
    if (tid == T - 1) s_mod = make_bundle_mod(static_cast<uint32_t>(b));
  }
  const int64_t doc0 = bundle * kDocsPerBundle;
  const int64_t docs = lesser(doc0 + kDocsPerBundle, a.num_docs) - doc0;
  const int64_t* offs = a.offsets + doc0 * F;
  for (uint32_t c0 = part_begin; c0 < part_end; c0 += 1u << lc) {
    unsigned long long* gbase = a.index + start * 32 + c0;
    if (tiled) {
      if (c0 != part_begin) __syncthreads();  // the last pass's tile is stored
      u32x4* clear = reinterpret_cast<u32x4*>(tile);
      for (int w = tid; w < (static_cast<int>(b) * stride + 3) / 4; w += T) clear[w] = u32x4{0, 0, 0, 0};
    } else if constexpr (kKind != kScatterRest) {
      for (int64_t w = tid; w < words; w += T) gbase[(w >> lc) * 32 + (w & ((1 << lc) - 1))] = 0;
      __threadfence();
    }
    __syncthreads();
    const int64_t dlo = static_cast<int64_t>(c0) * 64;
    const int64_t dhi = lesser(dlo + (64 << lc), docs);
    const int64_t slot_lo = dlo * F, slot_hi = dhi > dlo ? dhi * F : slot_lo;
    if (tiled && F <= kBuildFeatureCache) {
      TileMod mod{s_mod};
      mod.m.d = __builtin_amdgcn_readfirstlane(mod.m.d);
      mod.m.a_lo = __builtin_amdgcn_readfirstlane(mod.m.a_lo);
      mod.m.a_hi = __builtin_amdgcn_readfirstlane(mod.m.a_hi);
      mod.m.b_lo = __builtin_amdgcn_readfirstlane(mod.m.b_lo);
      mod.m.b_hi = __builtin_amdgcn_readfirstlane(mod.m.b_hi);
      const uint32_t row_bytes = 4 * stride;
      auto set = [&](uint32_t p, uint32_t m) {
        atomicOr(reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(tile) +
                                             (__umul24(p, row_bytes) + 4 * place_word(m))),
                 place_bit(m));
      };
      if constexpr (K > 1) {
        // Values whose first K positions collide (0.6% of the values, but a third
        // of the waves hold one, at b = 470 and K = 3) wait in the wave's queue
        // until it is full, and are then hashed again and further together.
        uint32_t* queue = queues + (tid >> 6) * kBuildQueueWords;
        const int lane = tid & 63;
        const int64_t base = slot_hi > slot_lo ? lesser(greater(offs[slot_lo], 0), a.num_values) : 0;
        int queued = 0;  // wave-uniform
        auto drain = [&] {
          if (lane < queued) {
            const uint32_t i = queue[2 * lane], m = queue[2 * lane + 1];
            scatter_value<K>(a.k, rxc[place_feature(m)], a.values[base + i], mod, [&](uint32_t p) { set(p, m); });
          }
          queued = 0;
        };
        for_each_value(a, offs, c0, slot_lo, slot_hi, vmap16, [&](int64_t value, uint32_t m, int64_t index, bool mine) {
          const uint64_t rx = rxc[place_feature(m)];
          const uint64_t ry = rotl64(murmur_mix_y(static_cast<uint64_t>(value)), 31);
          uint32_t found[K];
          const bool distinct = first_positions<K>(rx, ry, mod, found);
          if (mine && distinct) {
#pragma unroll
            for (int j = 0; j < K; ++j) set(found[j], m);
          }
          const bool wait = mine && !distinct;
          const uint64_t again = __ballot(wait);
          if (again != 0) {
            const int more = __popcll(again);
            if (queued + more > 64) {
              __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
              drain();
              __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
            if (wait) {
              const int at_q = queued + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(again >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(again), 0));
              queue[2 * at_q] = static_cast<uint32_t>(index - base);
              queue[2 * at_q + 1] = m;
            }
            queued += more;
          }
        });
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        drain();
      } else {
        for_each_value(a, offs, c0, slot_lo, slot_hi, vmap16, [&](int64_t value, uint32_t m, int64_t, bool mine) {
          if (mine) scatter_value<K>(a.k, rxc[place_feature(m)], value, mod, [&](uint32_t p) { set(p, m); });
        });
      }
    } else {
      // A bundle wider than the tile (its bits go straight to global memory),
      // or more features than the cache (300,000 docs of 60 features and 3 or 12
      // values 0.140 and 0.160 ms, of 65 features 0.150 and 0.175 ms) or than a
      // place names (a thread per slot then).
      uint64_t width = static_cast<uint64_t>(b);
      asm volatile("" : "+s"(width));  // formed here: hoisted, its registers would spill the other path's
      const WideMod mod{make_fastmod(width)};
      auto one = [&](int64_t value, int64_t f, uint32_t word, uint32_t doc) {
        scatter_value<K>(a.k, rx_id(f), value, mod, [&](uint32_t p) {
          if (tiled) {
            atomicOr(tile + (p * stride + word), 0x80000000u >> doc);
          } else {
            atomicOr(gbase + static_cast<uint64_t>(p) * 32 + (word >> 1),
                     1ull << (((word & 1u) << 5) + 31u - doc));
          }
        });
      };
      if (F < kBuildMapFeatures) {
        for_each_value(a, offs, c0, slot_lo, slot_hi, vmap, [&](int64_t value, uint32_t m, int64_t, bool mine) {
          if (mine) one(value, place_feature(m), place_word(m), m & 31u);
        });
      } else {
        for (int64_t rel = slot_lo + tid; rel < slot_hi; rel += T) {
          const int64_t d = rel / F, f = rel - d * F;
          const int64_t v0 = lesser(greater(offs[rel], 0), a.num_values);
          const int64_t v1 = lesser(greater(offs[rel + 1], 0), a.num_values);
          for (int64_t v = v0; v < v1; ++v)
            one(a.values[v], f, static_cast<uint32_t>(((d >> 5) ^ 1) - 2 * c0), static_cast<uint32_t>(d & 31));
        }
      }
    }
    if (!tiled) return;
    __syncthreads();
    for (int w = tid; w < static_cast<int>(words); w += T) {
      const int p = w >> lc, c = w & ((1 << lc) - 1);
      const uint32_t* src = tile + p * stride + 2 * c;
      const unsigned long long v = (static_cast<unsigned long long>(src[1]) << 32) | src[0];
      unsigned long long* dst = gbase + static_cast<int64_t>(p) * 32 + c;
      // whole 128-byte lines stream past the caches; parts of a line meet in L2
      if (lc >= 4) __builtin_nontemporal_store(v, dst);
      else *dst = v;
    }
    if constexpr (kKind == kScatterEven) return;
  }
}

// One workgroup per part of a bundle (2^lc of its 32 columns).  The parts of a
// bundle lie 8 workgroups apart, on one XCD, so that the lines they share
// meet in its L2.  Parts rather than whole bundles: two tiles fit a CU, so one
// workgroup hashes while the other clears, loads offsets or stores, and a
// small corpus (49 bundles at 100,000 docs) still fills the chip.
// kScatterPasses: some bundles are wider than the tile holds at the part's
// columns; the loop over passes costs the others 2-8% (registers), so that
// indices without such bundles run without it.  What scatter_rest_kernel ORs in
// global memory is cleared here, whole rows by each workgroup.
// Bound by VALU issue: 242 wave instructions per 64 values at k = 3, one per 4.3
// cycles (nearly every instruction of the hash, 32-bit multiplies and
// v_mad_u64_u32 included, takes 4).  100M docs x 4 features, 1.8e9 values, 470
// rows: 12.0 ms; 17.0 ms with a whole bundle per workgroup (one a CU), the
// general remainder and 64-bit tile words (315 instructions).  100,000 docs x 2
// features: 11.8 against 29.9 us.
template <int K, ScatterKind kKind>
__global__ __launch_bounds__(kBuildThreads) void scatter_kernel(ScatterArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  __shared__ BundleMod s_mod;
  const int parts = 32 >> a.lc;
  const int64_t run = blockIdx.x / (8 * parts), at = blockIdx.x % (8 * parts);
  const int64_t bundle = run * 8 + at % 8;
  const int part = static_cast<int>(at / 8);
  if (bundle >= a.num_bundles) return;
  const int64_t start = a.bundle_b_offsets[bundle];
  const int64_t b = a.bundle_b_offsets[bundle + 1] - start;
  if (b <= 0) return;
  if constexpr (kKind == kScatterPasses) {
    if (a.rest_words != 0 && b * tile_stride(0) > a.rest_words) {
      if (b * tile_stride(0) > kRestWords) {
        const int64_t end = (start + b * (part + 1) / parts) * 32;
        for (int64_t w = (start + b * part / parts) * 32 + threadIdx.x; w < end; w += blockDim.x)
          __builtin_nontemporal_store(0ull, a.index + w);
      }
      return;
    }
  }
  scatter_part<K, kKind>(a, bundle, part, start, b, lds, s_mod);
}

// The bundles that scatter_kernel's tile does not hold at any number of columns,
// with the tile of a whole CU: persistent workgroups, each of which looks all
// bundle widths through (1,024 at a time) and takes its share of the wide
// bundles' parts.  The parts of a bundle are taken on one XCD (workgroup i runs
// on XCD i % 8; the n-th wide bundle is XCD n % 8's).
template <int K>
__global__ __launch_bounds__(kBuildThreads) void scatter_rest_kernel(ScatterArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  __shared__ BundleMod s_mod;
  __shared__ unsigned long long wide[kBuildThreads / 64];  // bundles of the 1,024, by wave and lane
  const int tid = threadIdx.x;
  const int64_t parts = 32 >> a.lc, xcd = blockIdx.x % 8, per_xcd = gridDim.x / 8;
  // this workgroup's next part of its XCD's wide bundles; wide bundles before the 1,024
  int64_t item = blockIdx.x / 8, seen = 0;
  for (int64_t base = 0; base < a.num_bundles; base += kBuildThreads) {
    const int64_t i = base + tid;
    const int64_t b = i < a.num_bundles ? a.bundle_b_offsets[i + 1] - a.bundle_b_offsets[i] : 0;
    const uint64_t mask = __ballot(b * tile_stride(0) > a.rest_words);
    __syncthreads();  // the last 1,024's readers are done
    if ((tid & 63) == 0) wide[tid >> 6] = mask;
    __syncthreads();
    int64_t n = 0;
    for (int w = 0; w < kBuildThreads / 64; ++w) n += __popcll(wide[w]);
    for (; item / parts * 8 + xcd < seen + n; item += per_xcd) {
      int nth = static_cast<int>(item / parts * 8 + xcd - seen), w = 0;
      while (nth >= __popcll(wide[w])) nth -= __popcll(wide[w++]);
      uint64_t m = wide[w];
      for (; nth > 0; --nth) m &= m - 1;
      const int64_t bundle = base + 64 * w + __builtin_ctzll(m);
      const int64_t start = a.bundle_b_offsets[bundle];
      scatter_part<K, kScatterRest>(a, bundle, static_cast<int>(item % parts), start,
                                    a.bundle_b_offsets[bundle + 1] - start, lds, s_mod);
      __syncthreads();  // the tile is stored
    }
    seen += n;
  }
}

using ScatterFn = void (*)(ScatterArgs);

template <int K>
ScatterFn scatter_of(ScatterKind kind) {
  return kind == kScatterRest ? scatter_rest_kernel<K>
         : kind == kScatterPasses ? scatter_kernel<K, kScatterPasses>
                                  : scatter_kernel<K, kScatterEven>;
}

ScatterFn select_scatter(int64_t k, ScatterKind kind) {
  switch (k) {
    case 1: return scatter_of<1>(kind);
    case 2: return scatter_of<2>(kind);
    case 3: return scatter_of<3>(kind);
    case 4: return scatter_of<4>(kind);
    case 5: return scatter_of<5>(kind);
    case 6: return scatter_of<6>(kind);
    case 7: return scatter_of<7>(kind);
    case 8: return scatter_of<8>(kind);
    case 9: return scatter_of<9>(kind);
    case 10: return scatter_of<10>(kind);
    default: return scatter_of<0>(kind);
  }
}

void check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    throw Error(ST_ERR_HIP, cat(what, " launch failed: ", hipGetErrorString(e)));
}

// The tile may take more than the 64 KB default limit.
void set_lds_limits() {
  static std::once_flag once;
  static hipError_t status = hipSuccess;
  std::call_once(once, [] {
    for (int64_t k = 0; k <= 10; ++k) {
      for (const ScatterKind kind : {kScatterEven, kScatterPasses, kScatterRest}) {
        const hipError_t e = hipFuncSetAttribute(
            reinterpret_cast<const void*>(select_scatter(k, kind)), hipFuncAttributeMaxDynamicSharedMemorySize,
            kLdsBytes - (kind == kScatterRest ? kBuildRestLds : kBuildStaticLds));
        if (e != hipSuccess && status == hipSuccess) status = e;
      }
    }
  });
  if (status != hipSuccess)
    throw Error(ST_ERR_HIP, cat("hipFuncSetAttribute failed: ", hipGetErrorString(status)));
}

struct ScatterShape {
  int lc, tile_words, threads;
  bool passes;  // some bundle is wider than the tile holds at 2^lc columns
  bool rest;    // ... than it holds at one column
};

// The part of a bundle a workgroup takes: as many columns as let two tiles of a
// typical bundle share a CU (16 columns up to 492 rows, 8 up to 955, 4 up to
// 1,804), else as many as fit the whole CU (4 up to 3,966 rows, 2 up to 7,139, 1
// up to 11,898).  Typical is a quarter above the mean width, or the widest where
// that is less: a few wide bundles among narrow ones go in passes, and those
// that the tile does not hold at one column (5,413 or 11,898 rows) in a launch
// of their own, so that they do not change the parts of the others.
// 20M docs of 1-2 values (20 rows), 2% of the bundles wider, ms by their rows
// (1,200 / 3,000 / 6,000 / 12,500): parts for the widest bundle 1.15 / 2.14 /
// 1.68 / 1.80, these 0.60 / 0.74 / 0.79 / 0.95, without wide bundles 0.49.
// 1M docs of 8 features, a fifth of the bundles 3,000 rows: 0.284 -> 0.241; all
// bundles 12,500 rows: 3.67 -> 2.77 (whole rows cleared, 16 parts OR).
// A corpus too small to give every CU two workgroups is split further, one of
// over half a million bundles less far than its widths ask for where the grid
// would pass 2^32 threads (the passes do the rest).
ScatterShape scatter_shape(int64_t max_b, int64_t total_rows, int64_t nb) {
  const int64_t widest = std::min<int64_t>(max_b, INT32_MAX);
  const int64_t typical = std::min(widest, (total_rows + nb - 1) / nb * 5 / 4);
  ScatterShape s{0, kWholeWords, kBuildThreads, false, false};
  for (int lc = 1; lc <= 2; ++lc)
    if (typical * tile_stride(lc) <= kWholeWords) s.lc = lc;
  for (int lc = 2; lc <= 4; ++lc)
    if (typical * tile_stride(lc) <= kHalfWords) s = {lc, kHalfWords, kBuildHalfThreads, false, false};
  while (s.lc > 2 && s.threads == kBuildHalfThreads && nb * (32 >> s.lc) < 2 * cu_count()) --s.lc;
  while (s.lc < 4 && (nb + 7) / 8 * 8 * (32 >> s.lc) * s.threads > int64_t{UINT32_MAX}) ++s.lc;
  s.passes = widest * tile_stride(s.lc) > s.tile_words;
  s.rest = widest * tile_stride(0) > s.tile_words;
  if (!s.passes) s.tile_words = static_cast<int>(widest) * tile_stride(s.lc);
  return s;
}

void launch_scatter(ScatterArgs a, ScatterKind kind, int64_t grid, int threads, hipStream_t s) {
  const int lds = fixed_lds(threads) + (4 * a.tile_words + 15) / 16 * 16;
  hipLaunchKernelGGL(select_scatter(a.k, kind), dim3(static_cast<unsigned>(grid)), dim3(threads), lds, s, a);
  check_launch(kind == kScatterRest ? "scatter_rest_kernel" : "scatter_kernel");
}

}  // namespace
}  // namespace st

extern "C" int st_bloom_build_bundle_offsets(const int64_t* feature_offsets,
                                             int64_t num_docs,
                                             int64_t num_features, int64_t k,
                                             double b_multiplier,
                                             int64_t* bundle_b_offsets,
                                             int64_t* stats, void* stream) {
  using namespace st;
  return guarded([&] {
    ST_CHECK(num_features >= 1, "feature_ids must not be empty");
    ST_CHECK(num_docs >= 0, "negative document count");
    ST_CHECK(k >= 0 && k <= kMaxBuildK, "k must be in [0, ", kMaxBuildK,
             "], got ", k);
    ST_CHECK(b_multiplier > 1.0, "b_multiplier must be greater than 1.0");
    ST_CHECK(feature_offsets && bundle_b_offsets && stats, "null device pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t nb = (num_docs + kDocsPerBundle - 1) / kDocsPerBundle;
    if (nb > 0) {
      const int64_t staged = num_features <= kWidthStageFeatures ? num_features : 0;
      const bool few = nb < 4 * cu_count() && staged <= kWidthFewFeatures;
      const int threads = few ? kWidthThreadsFew : kWidthThreads;
      hipLaunchKernelGGL(few ? widths_kernel<kWidthThreadsFew> : widths_kernel<kWidthThreads>,
                         dim3(static_cast<unsigned>(nb)), dim3(threads), 8 * (threads * staged + 1), s,
                         feature_offsets, num_docs, num_features, k, b_multiplier, bundle_b_offsets);
      check_launch("widths_kernel");
    }
    hipLaunchKernelGGL(scan_kernel, dim3(1), dim3(kScanThreads), 0, s,
                       feature_offsets, num_docs * num_features, nb,
                       bundle_b_offsets, stats);
    check_launch("scan_kernel");
  });
}

extern "C" int st_bloom_index_build(const int32_t* feature_ids,
                                    const int64_t* feature_offsets,
                                    const int64_t* feature_values,
                                    int64_t num_features, int64_t num_docs,
                                    int64_t num_values, int64_t k,
                                    const int64_t* bundle_b_offsets,
                                    int64_t max_b, int64_t* bloom_index,
                                    int64_t bloom_index_numel, void* stream) {
  using namespace st;
  return guarded([&] {
    ST_CHECK(num_features >= 1, "feature_ids must not be empty");
    ST_CHECK(num_docs >= 0 && num_values >= 0, "negative sizes");
    ST_CHECK(k >= 0 && k <= kMaxBuildK, "k must be in [0, ", kMaxBuildK,
             "], got ", k);
    const int64_t nb = (num_docs + kDocsPerBundle - 1) / kDocsPerBundle;
    if (nb == 0 || bloom_index_numel == 0) return;
    ST_CHECK(feature_ids && feature_offsets && bundle_b_offsets && bloom_index,
             "null device pointer");
    ST_CHECK(num_values == 0 || feature_values, "feature_values is null");
    set_lds_limits();
    // any max_b gives the same index: one below the widths (a negative one as
    // zero) sends the wider bundles through global memory
    const ScatterShape shape =
        scatter_shape(std::max<int64_t>(max_b, 0), bloom_index_numel / kColumnsPerBundle, nb);
    ScatterArgs a;
    a.feature_ids = feature_ids;
    a.offsets = feature_offsets;
    a.values = feature_values;
    a.num_values = num_values;
    a.num_features = num_features;
    a.num_docs = num_docs;
    a.k = k;
    a.bundle_b_offsets = bundle_b_offsets;
    a.index = reinterpret_cast<unsigned long long*>(bloom_index);
    a.num_bundles = nb;
    a.lc = shape.lc;
    a.tile_words = shape.tile_words;
    a.rest_words = shape.rest ? shape.tile_words : 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    launch_scatter(a, shape.passes ? kScatterPasses : kScatterEven, (nb + 7) / 8 * 8 * (32 >> shape.lc),
                   shape.threads, s);
    if (shape.rest) {
      a.lc = 1;
      a.tile_words = kRestWords;
      launch_scatter(a, kScatterRest, std::max(8, cu_count() / 8 * 8), kBuildThreads, s);
    }
  });
}
