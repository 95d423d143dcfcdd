// Fused bloom filter + top-k scoring for gfx950.
//
// No reference operator: the closest relatives are the bloom-filtered
// scoring of fused_kmean_ann (fused_kmean_ann_cuda.cu:545-551, :1797-1926)
// and at::topk in fresh_index_post_processing.cpp:245-250.  For every query
// q, among docs d < num_docs whose bit is set in the packed search output
// (doc 64c+i of row q at bit 63-i of word c), return the `topk` best by
//   score(q, d) = sum_j bf16(emb[d, j]) * bf16(x[q, j])   (fp32 accumulation)
// ordered by score descending, then doc id ascending; missing entries are
// id -1 and score -inf (the reference's padding, fused_kmean_ann.cpp:139-167).
//
// Scoring is a dense bf16 contraction on the matrix cores
// (v_mfma_f32_32x32x16_bf16): each wave keeps the fragments of its 32 or 64
// queries in registers (B operands) for the whole launch, the workgroup
// streams 64 KB steps of doc rows and their filter words through LDS (the
// next step is loaded into registers while the current one is scored), and
// one LDS read of a doc fragment feeds the MFMAs of every query tile of the
// wave.  A doc tile whose filter bits are all zero for the wave is skipped.
//
// Selection is exact and runs in rounds over growing doc ranges: a scored
// pair enters query q's candidate list when it passes the filter and its
// score is at least thr[q]; after each round one workgroup per query keeps
// the best `topk` of its candidates (a radix select in LDS; the last round
// sorts them, bitonic) and sets thr[q] to the score of the topk-th, so later
// rounds emit only pairs that can still enter.  A candidate list has a fixed
// capacity; a round that overflows one changes nothing, nor do the rounds after
// it, and the call goes on from that round with smaller ones.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <utility>
#include <vector>

#include "st_common.hpp"
#include "st_errors.hpp"

namespace st {
int cu_count();

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kScoreThreads = 512;   // 8 waves; one workgroup per CU
constexpr int kScoreWaves = kScoreThreads / 64;
constexpr int kQueryTile = 32;
constexpr int kLdsBytes = 160 * 1024;
// topk_score_few_kernel (a dim-256 tile's operands need 256 registers a lane)
template <int D>
constexpr int kFewThreads = D <= 128 ? 1024 : 512;
constexpr int kFewTiles = 4;
constexpr int64_t kFewBytes = 128 << 20;
constexpr int kSelectThreads = 256;
constexpr int kSelectSlots = 4096;   // candidates gathered into LDS for the selection
constexpr int kMaxTopk = 2048;
constexpr uint32_t kCandidateCapacity = 32768;  // per query
// A query's candidate list: the best kept so far in slots [0, kMaxTopk), then
// one segment per scoring workgroup (at most kMaxSegments of them), each
// filled by its workgroup alone.
constexpr int kMaxSegments = 256;
constexpr uint32_t kSegmentSlots = kCandidateCapacity - kMaxTopk;
constexpr int64_t kRoundAlign = 2048;
constexpr int64_t kRoundCandidates = 1 << 17;

// Monotone map of floats to unsigned ints (larger float -> larger int).
__device__ __forceinline__ uint32_t ordered_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float from_ordered(uint32_t o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o);
}

// Sort key: score descending, then doc id ascending, as one descending
// 64-bit key.  Key 0 sorts below every real key.
__device__ __forceinline__ uint64_t make_key(float score, int64_t doc) {
  return (static_cast<uint64_t>(ordered_bits(score)) << 32) |
         (0xFFFFFFFFu - static_cast<uint32_t>(doc));
}

struct TopkState {
  uint32_t* counts;    // [Q] best candidates kept (<= topk)
  float* thr;          // [Q] entry threshold
  uint64_t* cand;      // [Q * capacity] keys
  uint32_t* segn;      // [Q * kMaxSegments] entries in each segment
  uint32_t* stop;      // [1] number of the round that overflowed a segment, or 0
  uint32_t capacity;
  uint32_t seg;        // slots per segment in the current round
  uint32_t round;      // number of the current round in the schedule, from 1
  int first_round;     // counts and thr are not written yet: none kept, -inf
  int check;           // a round before this one (for the selection: up to this one) may have set stop
};

// Whether an earlier round overflowed (this one's number may appear while it
// runs).
__device__ __forceinline__ bool stopped_before(const TopkState& st) {
  if (st.check == 0) return false;
  const uint32_t stop = *st.stop;
  return stop != 0u && stop != st.round;
}

// Scoring geometry for embedding dimension D.  Each of the 8 waves keeps
// QT query tiles (32 queries each) as MFMA B operands in registers, so one
// launch pass covers 8 * 32 * QT queries; the workgroup streams its docs in
// steps of kDocs rows (32 KB of embeddings) through two LDS buffers, each with
// the queries' filter words for those docs.
template <int D>
struct ScoreShape {
  static constexpr int S = D / 16;                     // MFMA k-steps
  static constexpr int QT = D <= 128 ? 2 : 1;          // query tiles per wave
  static constexpr int kQueries = kScoreWaves * kQueryTile * QT;  // per pass
  static constexpr int kStepBytes = 32768;
  static constexpr int kDocs = kStepBytes / (2 * D);   // docs per step
  static constexpr int kDocTiles = kDocs / 32;
  static constexpr int kPieces = D / 8;                // 16-byte pieces per doc row
  // Rows padded by 16 bytes: the 16 rows an A-operand read serves at once
  // start 4 banks apart, and every piece sits at a fixed offset of its row.
  static constexpr int kRowBytes = 2 * D + 16;
  static constexpr int kCols = kDocs / 64;             // mask columns per step
  static constexpr int kMaskWords = kDocTiles + 1;     // u32 per query, padded
  static constexpr int kDocBuf = kDocs * kRowBytes;
  static constexpr int kMaskBuf = kQueries * kMaskWords * 4;
  static constexpr int kBuf = kDocBuf + kMaskBuf;
  static constexpr int kLds = 2 * kBuf + kQueries * 4;  // + segment slot counters
  static constexpr int kDocLoads = kStepBytes / 16 / kScoreThreads;  // u32x4 per thread
  static constexpr int kMaskLoads = (kQueries * kCols + kScoreThreads - 1) / kScoreThreads;
  static_assert(kLds <= kLdsBytes, "two steps must fit in LDS");
  static_assert(kDocs % 64 == 0 && kStepBytes % (16 * kScoreThreads) == 0, "step shape");
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Filter bits of the 32 docs from g0 that lie below hi (doc g0 at bit 31).
__device__ __forceinline__ uint32_t valid_doc_mask(int64_t g0, int64_t hi) {
  const int64_t left = hi - g0;
  return left >= 32 ? ~0u : (left <= 0 ? 0u : ~0u << (32 - static_cast<int>(left)));
}

// acc[j] of a 32 x 32 MFMA result holds doc row 8 (j / 4) + 4 h + j % 4 of
// the tile for lane half h = lane / 32 (query column lane % 32).  Returns the
// filter bits of those rows, row of acc[j] at bit j (doc row r of m at bit
// 31 - r).
__device__ __forceinline__ uint32_t lane_rows(uint32_t m, int h) {
  uint32_t x = (__builtin_bitreverse32(m) >> (4 * h)) & 0x0F0F0F0Fu;
  x = (x | (x >> 4)) & 0x00FF00FFu;
  return (x | (x >> 8)) & 0xFFFFu;
}

// Whether this lane's part of a 32 x 32 score tile (16 docs of its query)
// may hold a candidate: a filter bit, and a score at the threshold.
__device__ __forceinline__ bool tile_gate(const f32x16& acc, uint32_t m, float th) {
  float mx = acc[0];
#pragma unroll
  for (int j = 1; j < 16; ++j) mx = fmaxf(mx, acc[j]);
  return m != 0u && mx >= th;
}

// Candidates of one 32 x 32 score tile (docs x this lane's query): pairs that
// pass the filter with a score >= th go to the query's candidate list.
// Called by the whole wave.
__device__ __forceinline__ void tile_candidates(const TopkState& st, const f32x16& acc, uint32_t m,
                                                float th, int64_t q, uint32_t* slot_count,
                                                int64_t doc0, int lane) {
  uint32_t ge = 0u;
#pragma unroll
  for (int j = 15; j >= 0; --j) ge = (ge << 1) | (acc[j] >= th ? 1u : 0u);
  const int h = lane >> 5;
  uint32_t hits = ge & lane_rows(m, h);
  if (__ballot(hits != 0u) == 0) return;
  const uint32_t cnt = __builtin_popcount(hits);
  const uint32_t cnt_pair = __shfl_xor(cnt, 32, 64);  // lanes l, l ^ 32: same query
  // slots of this workgroup's segment, counted in LDS
  uint32_t base = 0u;
  if (lane < 32 && cnt + cnt_pair > 0u) base = atomicAdd(slot_count, cnt + cnt_pair);
  const uint32_t base_pair = __shfl_xor(base, 32, 64);
  uint32_t slot = lane < 32 ? base : base_pair + cnt_pair;
  uint64_t* seg = st.cand + q * st.capacity + kMaxTopk + static_cast<uint64_t>(blockIdx.x) * st.seg;
  while (__ballot(hits != 0u) != 0) {
    if (hits != 0u) {
      const int j = __builtin_ctz(hits);
      hits &= hits - 1u;
      float v = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) v = j == i ? acc[i] : v;
      const int64_t doc = doc0 + 8 * (j >> 2) + 4 * h + (j & 3);
      if (slot < st.seg) seg[slot] = make_key(v, doc);
      ++slot;
    }
  }
}

// Scores docs [lo, hi) against queries [q_begin, q_begin + q_count)
// (q_count <= ScoreShape<D>::kQueries).  Wave w holds queries
// w * 32 * QT + 32 t + (lane & 31) of tile t as B operands (lanes 32-63
// carry the second half of each 16-wide k step); the workgroups take the steps
// in turn, so that docs of one kind that lie together (a query's cluster) are
// spread over the segments.  A step's rows and filter words are loaded into
// registers while the step before is scored and stored into the other LDS
// buffer after it, so each step needs one barrier.  Steps in turn and not in
// runs: 64 queries of 10 over 2M docs in 1,000 clusters 2.31 -> 0.54 ms, 512 of
// 100 over 20M docs in random order 2.91 -> 2.93 ms.
template <int D>
__global__ __launch_bounds__(kScoreThreads) void topk_score_kernel(
    const uint16_t* __restrict__ emb, const uint16_t* __restrict__ qv,
    const uint64_t* __restrict__ mask64, int64_t num_columns, int64_t q_begin,
    int64_t q_count, int64_t lo, int64_t hi, TopkState st) {
  using SS = ScoreShape<D>;
  constexpr int S = SS::S, QT = SS::QT;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int h = lane >> 5;

  if (st.round == 1 && blockIdx.x == 0 && tid == 0) *st.stop = 0u;
  if (stopped_before(st)) return;
  const int64_t first = lo + static_cast<int64_t>(blockIdx.x) * SS::kDocs;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * SS::kDocs;
  uint32_t* segn = st.segn + q_begin * kMaxSegments + blockIdx.x;  // query stride kMaxSegments
  if (first >= hi) {  // whole workgroup; its segments stay empty
    for (int i = tid; i < q_count; i += kScoreThreads) segn[i * kMaxSegments] = 0u;
    return;
  }
  // Entries this workgroup put in each query's segment.
  uint32_t* slot_count = reinterpret_cast<uint32_t*>(lds + 2 * SS::kBuf);
  for (int i = tid; i < SS::kQueries; i += kScoreThreads) slot_count[i] = 0u;

  // This wave's query fragments (zero past q_count) and entry thresholds
  // (fixed for the launch).
  bf16x8 b[QT][S];
  int ql[QT];
  float th[QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    ql[t] = (wave * QT + t) * kQueryTile + (lane & 31);
    const bool valid = ql[t] < q_count;
    const uint16_t* row = qv + (q_begin + (valid ? ql[t] : 0)) * D + h * 8;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      b[t][s] = *reinterpret_cast<const bf16x8*>(row + s * 16);
      if (!valid) b[t][s] = bf16x8{};
    }
    th[t] = st.first_round ? -INFINITY : st.thr[q_begin + (valid ? ql[t] : 0)];
  }

  u32x4 dpre[SS::kDocLoads];
  uint64_t mpre[SS::kMaskLoads];
  // Step d0's rows and filter words into registers: rows at or past hi read
  // as zero, and so do columns past the last and queries past the chunk.
  // d0 is a multiple of 64; a mask row is only 8-byte aligned.
  auto prefetch = [&](int64_t d0) {
    const int64_t rows = hi - d0 < SS::kDocs ? hi - d0 : SS::kDocs;
    const u32x4* src = reinterpret_cast<const u32x4*>(emb + d0 * D);
#pragma unroll
    for (int i = 0; i < SS::kDocLoads; ++i) {
      const int c = tid + i * kScoreThreads;
      dpre[i] = (c / SS::kPieces < rows) ? __builtin_nontemporal_load(src + c) : u32x4{0, 0, 0, 0};
    }
    const int64_t col0 = d0 >> 6;
#pragma unroll
    for (int i = 0; i < SS::kMaskLoads; ++i) {
      const int w = tid + i * kScoreThreads;
      const int qq = w / SS::kCols, cc = w - qq * SS::kCols;
      const bool ok = qq < q_count && col0 + cc < num_columns;
      mpre[i] = ok ? mask64[(q_begin + qq) * num_columns + col0 + cc] : 0ull;
    }
  };
  // The registers into LDS buffer buf, with the filter bits of docs at or
  // past hi cleared.  A column word holds docs 0-31 in its high half.
  auto stage = [&](int buf, int64_t d0) {
    uint8_t* docs = lds + buf * SS::kBuf;
    uint32_t* masks = reinterpret_cast<uint32_t*>(docs + SS::kDocBuf);
#pragma unroll
    for (int i = 0; i < SS::kDocLoads; ++i) {
      const int c = tid + i * kScoreThreads;
      const int r = c / SS::kPieces, k = c - r * SS::kPieces;
      *reinterpret_cast<u32x4*>(docs + r * SS::kRowBytes + k * 16) = dpre[i];
    }
#pragma unroll
    for (int i = 0; i < SS::kMaskLoads; ++i) {
      const int w = tid + i * kScoreThreads;
      if (w >= SS::kQueries * SS::kCols) continue;
      const int qq = w / SS::kCols, cc = w - qq * SS::kCols;
      const int64_t g0 = d0 + 64 * cc;
      uint32_t* dst = masks + qq * SS::kMaskWords + 2 * cc;
      dst[0] = static_cast<uint32_t>(mpre[i] >> 32) & valid_doc_mask(g0, hi);
      dst[1] = static_cast<uint32_t>(mpre[i]) & valid_doc_mask(g0 + 32, hi);
    }
  };

  prefetch(first);
  stage(0, first);
  if (first + stride < hi) prefetch(first + stride);
  __syncthreads();
  // Scored tiles whose epilogue is still to run (two accumulator sets).
  f32x16 acc[2][QT];
  uint32_t mb[2][QT];
  int64_t docb[2] = {0, 0};
  bool pend[2] = {false, false};
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      acc[x][t] = f32x16{};
      mb[x][t] = 0u;
    }
  int buf = 0;
  for (int64_t d0 = first; d0 < hi; d0 += stride, buf ^= 1) {
    const uint8_t* docs = lds + buf * SS::kBuf;
    const uint32_t* masks = reinterpret_cast<const uint32_t*>(docs + SS::kDocBuf);
    uint32_t m[QT][SS::kDocTiles];
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
      for (int dt = 0; dt < SS::kDocTiles; ++dt)
        m[t][dt] = masks[ql[t] * SS::kMaskWords + dt];  // zero past q_count
    // A operands: doc row 32 dt + (lane & 31), k half h.  The step's
    // fragments are read from LDS in one stream, kAhead ahead of their MFMAs
    // and across tile boundaries (rows past hi are zero in LDS and carry no
    // filter bit).  The epilogue of a tile is deferred to the next tile,
    // whose MFMAs its gate is interleaved with, so each wave keeps the
    // matrix cores fed by itself.  Tiles alternate between the two
    // accumulator sets; pend[x] says set x holds a tile still to finish.  A
    // step with no filter bit for any of the wave's queries is skipped.
    bool any = false;
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
      for (int dt = 0; dt < SS::kDocTiles; ++dt) any |= m[t][dt] != 0u;
    if (__ballot(any) != 0) {
      constexpr int kFrags = SS::kDocTiles * S;
      constexpr int kAhead = 3;
      const uint8_t* arow = docs + (lane & 31) * SS::kRowBytes + h * 16;
      bf16x8 fr[kAhead + 1];
      auto read = [&](int g) {
        fr[g % (kAhead + 1)] = *reinterpret_cast<const bf16x8*>(
            arow + (g / S) * 32 * SS::kRowBytes + (g % S) * 32);
      };
#pragma unroll
      for (int g = 0; g < kAhead; ++g) read(g);
#pragma unroll
      for (int dt = 0; dt < SS::kDocTiles; ++dt) {
        const int cb = dt & 1, pb = cb ^ 1;
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const int g = dt * S + s;
          if (g + kAhead < kFrags) read(g + kAhead);
#pragma unroll
          for (int t = 0; t < QT; ++t)
            acc[cb][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[g % (kAhead + 1)], b[t][s],
                                                                 s == 0 ? f32x16{} : acc[cb][t], 0, 0, 0);
        }
        bool gate[QT];
#pragma unroll
        for (int t = 0; t < QT; ++t) gate[t] = tile_gate(acc[pb][t], mb[pb][t], th[t]) & pend[pb];
        // MFMAs with a fragment read and the pending tile's gate VALU work
        // between them
#pragma unroll
        for (int i = 0; i < S; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
          for (int t = 0; t < QT; ++t) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
          }
        }
#pragma unroll
        for (int t = 0; t < QT; ++t)
          if (__ballot(gate[t]) != 0)
            tile_candidates(st, acc[pb][t], mb[pb][t], th[t], q_begin + ql[t], slot_count + ql[t],
                            docb[pb], lane);
        pend[cb] = true;
        pend[pb] = false;
#pragma unroll
        for (int t = 0; t < QT; ++t) mb[cb][t] = m[t][dt];
        docb[cb] = d0 + dt * 32;
      }
    }
    const int64_t next = d0 + stride;
    if (next < hi) {
      stage(buf ^ 1, next);
      if (next + stride < hi) prefetch(next + stride);
    }
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    if (pend[x]) {
#pragma unroll
      for (int t = 0; t < QT; ++t)
        if (__ballot(tile_gate(acc[x][t], mb[x][t], th[t])) != 0)
          tile_candidates(st, acc[x][t], mb[x][t], th[t], q_begin + ql[t], slot_count + ql[t],
                          docb[x], lane);
    }
  }
  __syncthreads();
  for (int i = tid; i < q_count; i += kScoreThreads) {
    segn[i * kMaxSegments] = slot_count[i];
    if (slot_count[i] > st.seg) *st.stop = st.round;
  }
}

// Scores docs [lo, hi) for few queries: grid.y tiles of 32, of which each wave
// holds one as B operands.  The waves share out the 64-doc columns of the mask
// and read their rows straight from memory as A operands, so that nothing is
// staged and a small corpus has every column in flight at once (topk_score_kernel
// gives a CU's waves different queries and takes the docs in steps: with 16
// queries one wave of eight works, 10 us for a step or two).  Rows that no
// query of the tile passes are not read.  The same products in the same order
// as topk_score_kernel's.  Latency-bound on small corpora (16 queries, 200,000
// docs, dim 64: the call 134 -> 55 us with this kernel, two rounds and the
// overflow flag in host memory), bandwidth-bound on large ones (16 queries, 20M
// docs, dim 128: 1.34 -> 0.78 ms).
template <int D>
__global__ __launch_bounds__(kFewThreads<D>) void topk_score_few_kernel(
    const uint16_t* __restrict__ emb, const uint16_t* __restrict__ qv,
    const uint64_t* __restrict__ mask64, int64_t num_columns, int64_t num_queries, int64_t lo,
    int64_t hi, TopkState st) {
  constexpr int S = D / 16;
  __shared__ uint32_t slot_count[kQueryTile];
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, row = lane & 31;
  const int64_t q0 = static_cast<int64_t>(blockIdx.y) * kQueryTile;
  const int64_t q = q0 + row;
  const bool valid = q < num_queries;
  if (st.round == 1 && blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) *st.stop = 0u;
  if (stopped_before(st)) return;
  if (tid < kQueryTile) slot_count[tid] = 0u;
  __syncthreads();
  const int64_t columns = (hi + 63) >> 6;
  const int64_t wave = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(tid >> 6)) * gridDim.x + blockIdx.x;
  const int64_t waves = static_cast<int64_t>(kFewThreads<D> / 64) * gridDim.x;
  const uint64_t* mrow = mask64 + (valid ? q : q0) * num_columns;
  int64_t col = (lo >> 6) + wave;
  uint64_t next = valid && col < columns ? mrow[col] : 0ull;
  if (col < columns) {
    bf16x8 b[S];
    const uint16_t* src = qv + (valid ? q : q0) * D + h * 8;
#pragma unroll
    for (int s = 0; s < S; ++s) b[s] = *reinterpret_cast<const bf16x8*>(src + s * 16);
    const float th = st.first_round ? -INFINITY : st.thr[valid ? q : q0];
    for (; col < columns; col += waves) {
      uint64_t m = next;
      const int64_t ahead = col + waves;
      next = valid && ahead < columns ? mrow[ahead] : 0ull;
      const int64_t left = hi - (col << 6);
      if (left < 64) m &= ~0ull << (64 - static_cast<int>(left));
      // docs that some query of the tile passes
      uint32_t any[2] = {static_cast<uint32_t>(m >> 32), static_cast<uint32_t>(m)};
#pragma unroll
      for (int x = 0; x < 2; ++x) {
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) any[x] |= __shfl_xor(any[x], d, 64);
      }
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        if (__builtin_amdgcn_readfirstlane(any[x]) == 0u) continue;
        const int64_t doc0 = (col << 6) + 32 * x;
        bf16x8 a[S];
        if ((any[x] >> (31 - row)) & 1u) {
          const uint16_t* r = emb + (doc0 + row) * D + h * 8;
#pragma unroll
          for (int s = 0; s < S; ++s) a[s] = *reinterpret_cast<const bf16x8*>(r + s * 16);
        } else {
#pragma unroll
          for (int s = 0; s < S; ++s) a[s] = bf16x8{};
        }
        f32x16 acc = {};
#pragma unroll
        for (int s = 0; s < S; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s], b[s], acc, 0, 0, 0);
        const uint32_t mx = x == 0 ? static_cast<uint32_t>(m >> 32) : static_cast<uint32_t>(m);
        if (__ballot(tile_gate(acc, mx, th)) != 0)
          tile_candidates(st, acc, mx, th, q, slot_count + row, doc0, lane);
      }
    }
  }
  __syncthreads();
  if (tid < kQueryTile && q < num_queries) {
    st.segn[q * kMaxSegments + blockIdx.x] = slot_count[tid];
    if (slot_count[tid] > st.seg) *st.stop = st.round;
  }
}

// Descending bitonic sort of the first `size` keys in LDS (a power of two).
__device__ void bitonic_sort_desc(uint64_t* keys, int size) {
  for (int k = 2; k <= size; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < size / 2; i += kSelectThreads) {
        // i-th compare pair of this stage: lower index lo, partner lo + j
        const int lo = ((i & ~(j - 1)) << 1) | (i & (j - 1));
        const int hi = lo + j;
        const bool desc = (lo & k) == 0;  // direction of this k-block
        const uint64_t x = keys[lo], y = keys[hi];
        if ((x < y) == desc) {
          keys[lo] = y;
          keys[hi] = x;
        }
      }
      __syncthreads();
    }
  }
}

// Writes the best m = min(n, k) of the n distinct keys key_at(0 .. n-1) to
// keys[0, m) in no particular order and returns m; *min_key receives the
// smallest of them.  key_at may read keys[] itself (the keys are gathered
// before keys[] is written).  A radix select over the bits in which the keys differ
// (8 bits a pass, one LDS histogram per wave) finds the lower bound L of the
// best m (the m-th key itself, or the start of a digit bucket that holds
// exactly the keys still needed), then the keys >= L are gathered.  Called
// by the whole workgroup; the keys stay in LDS.
template <typename Key>
__device__ uint32_t select_best(Key key_at, uint64_t* keys, uint32_t n, uint32_t k, uint64_t* min_key) {
  constexpr int kWaves = kSelectThreads / 64;
  __shared__ uint32_t hist[kWaves][256];
  __shared__ uint64_t red_and[kWaves], red_or[kWaves];
  __shared__ uint64_t s_prefix, s_min;
  __shared__ uint32_t s_remaining, s_done, s_count;
  __shared__ uint64_t picked[kMaxTopk];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t m = min(n, k);
  uint64_t bound = 0ull;  // keys >= bound are the best m
  if (n > k) {
    uint64_t kand = ~0ull, kor = 0ull;
    for (uint32_t i = tid; i < n; i += kSelectThreads) {
      const uint64_t key = key_at(i);
      kand &= key;
      kor |= key;
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
      kand &= __shfl_xor(kand, d, 64);
      kor |= __shfl_xor(kor, d, 64);
    }
    if (lane == 0) {
      red_and[wave] = kand;
      red_or[wave] = kor;
    }
    for (int i = tid; i < kWaves * 256; i += kSelectThreads) (&hist[0][0])[i] = 0u;
    __syncthreads();
    kand = ~0ull;
    kor = 0ull;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      kand &= red_and[w];
      kor |= red_or[w];
    }
    const uint64_t diff = kand ^ kor;  // nonzero: n > k >= 1 distinct keys
    uint64_t prefix = kand & ~(~0ull >> __builtin_clzll(diff));
    uint32_t remaining = k;
    for (int shift = ((63 - __builtin_clzll(diff)) / 8) * 8; shift >= 0; shift -= 8) {
      const uint64_t hi_mask = shift + 8 >= 64 ? 0ull : (~0ull << (shift + 8));
      for (uint32_t i = tid; i < n; i += kSelectThreads) {
        const uint64_t key = key_at(i);
        if ((key & hi_mask) == (prefix & hi_mask)) atomicAdd(&hist[wave][(key >> shift) & 0xFFu], 1u);
      }
      __syncthreads();
      if (wave == 0) {
        // bins from the top digit down: 4 per lane, lane 0 holding 255..252
        uint32_t c[4], sum = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          c[i] = 0;
#pragma unroll
          for (int w = 0; w < kWaves; ++w) c[i] += hist[w][255 - (lane * 4 + i)];
          sum += c[i];
        }
        uint32_t incl = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const uint32_t y = __shfl_up(incl, d, 64);
          if (lane >= d) incl += y;
        }
        uint32_t run = incl - sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (run < remaining && run + c[i] >= remaining) {
            const int digit = 255 - (lane * 4 + i);
            s_prefix = (prefix & hi_mask) | (static_cast<uint64_t>(digit) << shift);
            s_remaining = remaining - run;
            s_done = run + c[i] == remaining ? 1u : 0u;  // the whole bucket is needed
          }
          run += c[i];
        }
      }
      __syncthreads();
      prefix = s_prefix;
      remaining = s_remaining;
      const bool done = s_done != 0u;
      for (int i = tid; i < kWaves * 256; i += kSelectThreads) (&hist[0][0])[i] = 0u;
      __syncthreads();
      if (done) break;
    }
    bound = prefix;  // the bucket's lowest key, or the m-th key after the last pass
  }
  if (tid == 0) {
    s_count = 0u;
    s_min = ~0ull;
  }
  __syncthreads();
  for (uint32_t i = tid; i < n; i += kSelectThreads) {
    const uint64_t key = key_at(i);
    if (key >= bound) {
      picked[atomicAdd(&s_count, 1u)] = key;
      atomicMin(&s_min, key);
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < m; i += kSelectThreads) keys[i] = picked[i];
  *min_key = s_min;
  __syncthreads();
  return m;
}

// One workgroup per query: keeps the best `topk` candidates (unordered
// between rounds), sets the entry threshold, and on the last round writes
// the outputs, sorted.  The
// candidates are the kept best (slots [0, counts[q])) followed by the entries
// of the round's nseg segments, gathered in that order.  After an overflow
// nothing is touched, and the last round stores the number of the round that
// overflowed to host memory.
__global__ __launch_bounds__(kSelectThreads) void topk_select_kernel(
    TopkState st, int64_t topk, int nseg, int final_round, int64_t* __restrict__ out_ids,
    float* __restrict__ out_scores, uint32_t* __restrict__ overflowed) {
  static_assert(kSelectThreads == kMaxSegments, "one thread per segment");
  __shared__ uint64_t keys[kSelectSlots];
  __shared__ uint32_t start[kMaxSegments + 1];  // virtual index of each segment's first entry
  const int64_t q = blockIdx.x;
  if (st.check != 0) {
    const uint32_t stop = *st.stop;
    if (stop != 0u) {
      if (final_round && q == 0 && threadIdx.x == 0) *overflowed = stop;  // host memory
      return;
    }
  }
  uint64_t* cand = st.cand + q * st.capacity;
  const uint32_t kept = st.first_round ? 0u : st.counts[q];
  // Exclusive scan of the segment counts, one thread per segment.
  const int g = threadIdx.x;
  start[g + 1] = g < nseg ? st.segn[q * kMaxSegments + g] : 0u;
  if (g == 0) start[0] = 0u;
  __syncthreads();
  for (int off = 1; off < kMaxSegments; off <<= 1) {
    const uint32_t v = g + 1 - off >= 1 ? start[g + 1 - off] : 0u;
    __syncthreads();
    start[g + 1] += v;
    __syncthreads();
  }
  const uint32_t n = kept + start[kMaxSegments];
  // Candidate v of the virtual list: the kept best, then the segments.
  auto at = [&](uint32_t v) -> uint64_t {
    if (v < kept) return cand[v];
    const uint32_t w = v - kept;
    int lo = 0, hi = nseg;  // last segment with start <= w
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (start[mid] <= w) lo = mid;
      else hi = mid;
    }
    return cand[kMaxTopk + static_cast<uint64_t>(lo) * st.seg + (w - start[lo])];
  };
  // the best min(n, topk) to the front of keys[], unordered: candidates
  // gathered into LDS when they fit (several radix passes read them), else
  // read from their segments on each pass
  uint64_t sel_min = 0ull;
  uint32_t best;
  if (n <= static_cast<uint32_t>(kSelectSlots)) {
    for (int i = threadIdx.x; i < static_cast<int>(n); i += kSelectThreads) keys[i] = at(i);
    __syncthreads();
    best = select_best([&](uint32_t i) { return keys[i]; }, keys, n, static_cast<uint32_t>(topk), &sel_min);
  } else {
    best = select_best(at, keys, n, static_cast<uint32_t>(topk), &sel_min);
  }
  if (final_round) {
    int size = 64;
    while (size < static_cast<int>(best)) size <<= 1;
    for (int i = static_cast<int>(best) + threadIdx.x; i < size; i += kSelectThreads) keys[i] = 0ull;
    __syncthreads();
    bitonic_sort_desc(keys, size);
    for (int64_t i = threadIdx.x; i < topk; i += kSelectThreads) {
      const bool have = i < best;
      out_ids[q * topk + i] = have ? static_cast<int64_t>(0xFFFFFFFFu - static_cast<uint32_t>(keys[i])) : -1;
      out_scores[q * topk + i] = have ? from_ordered(static_cast<uint32_t>(keys[i] >> 32)) : -INFINITY;
    }
    return;
  }
  for (uint32_t i = threadIdx.x; i < best; i += kSelectThreads) cand[i] = keys[i];
  if (threadIdx.x == 0) {
    st.counts[q] = best;
    st.thr[q] = best == topk ? from_ordered(static_cast<uint32_t>(sel_min >> 32)) : -INFINITY;
  }
}

void check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw Error(ST_ERR_HIP, cat(what, " launch failed: ", hipGetErrorString(e)));
}

// Segments of a round (a scoring workgroup each), and whether they hold every
// doc that their workgroup scores: such a round cannot overflow.
struct Segments {
  int count;
  uint32_t slots;
  bool safe;
};

// Segments when the docs [lo, hi) are taken in steps by one workgroup per CU.
Segments segments_of(int64_t lo, int64_t hi, int64_t step_docs) {
  const int64_t steps = (hi - lo + step_docs - 1) / step_docs;
  const int64_t groups = std::min<int64_t>(cu_count(), kMaxSegments);
  const int64_t per_group = (steps + groups - 1) / groups;
  const int64_t count = std::max<int64_t>(1, (steps + per_group - 1) / per_group);
  const int64_t slots = kSegmentSlots / count;
  return {static_cast<int>(count), static_cast<uint32_t>(slots), slots >= per_group * step_docs};
}

// Scores docs [lo, hi) for every query.
template <int D>
Segments launch_score(const uint16_t* emb, const uint16_t* qv, const uint64_t* mask64,
                      int64_t num_columns, int64_t num_queries, int64_t lo, int64_t hi,
                      TopkState st, hipStream_t s) {
  using SS = ScoreShape<D>;
  const Segments segs = segments_of(lo, hi, SS::kDocs);
  st.seg = segs.slots;
  for (int64_t qb = 0; qb < num_queries; qb += SS::kQueries) {
    const int64_t qn = std::min<int64_t>(SS::kQueries, num_queries - qb);
    hipLaunchKernelGGL(topk_score_kernel<D>, dim3(segs.count), dim3(kScoreThreads), SS::kLds, s, emb,
                       qv, mask64, num_columns, qb, qn, lo, hi, st);
    check_launch("topk_score_kernel");
  }
  return segs;
}

// The same for few queries, with topk_score_few_kernel (lo is a multiple of 64).
template <int D>
Segments launch_score_few(const uint16_t* emb, const uint16_t* qv, const uint64_t* mask64,
                          int64_t num_columns, int64_t num_queries, int64_t lo, int64_t hi,
                          TopkState st, hipStream_t s) {
  const Segments segs = segments_of(lo, hi, 64);
  const unsigned tiles = static_cast<unsigned>((num_queries + kQueryTile - 1) / kQueryTile);
  st.seg = segs.slots;
  hipLaunchKernelGGL(topk_score_few_kernel<D>, dim3(segs.count, tiles), dim3(kFewThreads<D>), 0, s, emb, qv,
                     mask64, num_columns, num_queries, lo, hi, st);
  check_launch("topk_score_few_kernel");
  return segs;
}

using ScoreFn = Segments (*)(const uint16_t*, const uint16_t*, const uint64_t*, int64_t, int64_t,
                             int64_t, int64_t, TopkState, hipStream_t);

// One tile of queries reads every row once; more tiles read the rows again, from
// the last-level cache while they fit it (64 queries over 400,000 docs of dim
// 128: 211 us staged, 148 us so; 128 queries: 220 and 184 us).
bool few_queries(int64_t num_queries, int64_t num_docs, int64_t dim) {
  const int64_t tiles = (num_queries + kQueryTile - 1) / kQueryTile;
  return tiles == 1 || (tiles <= kFewTiles && num_docs * dim * 2 <= kFewBytes);
}

ScoreFn score_fn(int64_t dim, bool few) {
  switch (dim) {
    case 64: return few ? launch_score_few<64> : launch_score<64>;
    case 128: return few ? launch_score_few<128> : launch_score<128>;
    case 256: return few ? launch_score_few<256> : launch_score<256>;
    default: fail("embedding dimension ", dim, " is not supported (64, 128 or 256)");
  }
}

// The scoring kernel stages a step of doc rows and filter words in LDS
// (more than the 64 KB default limit).
void set_lds_limits() {
  static std::once_flag once;
  static hipError_t status = hipSuccess;
  std::call_once(once, [] {
    const std::pair<const void*, int> kernels[] = {
        {reinterpret_cast<const void*>(topk_score_kernel<64>), ScoreShape<64>::kLds},
        {reinterpret_cast<const void*>(topk_score_kernel<128>), ScoreShape<128>::kLds},
        {reinterpret_cast<const void*>(topk_score_kernel<256>), ScoreShape<256>::kLds}};
    for (const auto& k : kernels) {
      const hipError_t e = hipFuncSetAttribute(k.first, hipFuncAttributeMaxDynamicSharedMemorySize, k.second);
      if (e != hipSuccess && status == hipSuccess) status = e;
    }
  });
  if (status != hipSuccess)
    throw Error(ST_ERR_HIP, cat("hipFuncSetAttribute failed: ", hipGetErrorString(status)));
}

// A schedule of rounds: `small` rounds of `first` docs, then each round `growth`
// times what the schedule has covered.
struct Schedule {
  int64_t first, small;
  double growth;
};

// A call's first schedule: a round after the first leaves about growth x topk
// candidates per query where docs lie in random order.  A round takes about
// 20 us of fixed time; a candidate costs its tile's slow path, and more where the
// staged kernel's waves hold more queries.  Over 1-512 queries of 200,000-8M
// docs, each time over the better of the two schedules that this one took the
// place of (8,192 docs and x8; 2,048 and up to x2,048): read directly, top 1 and
// 10 x128 0.89-1.02 (x512 up to 1.95), top 50 x32 0.97-1.04; staged, top 1 x32
// 0.97-1.04 (x512 1.0-1.6), top 10 x16 1.03-1.08 (x128 1.04-1.2), top 50 and 100
// 8,192 and x8 1.00-1.06 (2,048 and x16 1.08-1.15).
// Read directly, the rounds that a growth gives grow by equal factors, which
// leaves the fewest candidates; staged this measured 0-4% slower.
Schedule first_schedule(bool few, int64_t num_queries, int64_t num_docs, int64_t topk) {
  const int64_t first = topk <= (few || num_docs < int64_t{1} << 20 ? 64 : 16) ? 2048 : 8192;
  if (!few && num_docs >= int64_t{1} << 20) return {first, 1, topk <= 4 ? 32.0 : topk <= 16 ? 16.0 : 8.0};
  int64_t growth = std::min(kSelectSlots / 2 / topk, kRoundCandidates / (num_queries * topk));
  growth = std::max<int64_t>(8, std::min(growth, std::max<int64_t>(256, 2048 / num_queries)));
  if (!few) return {first, 1, static_cast<double>(growth)};
  const double all = std::max(1.0, static_cast<double>(num_docs) / static_cast<double>(first));
  const double rounds = std::max(1.0, std::ceil(std::log(all) / std::log(1.0 + static_cast<double>(growth))));
  return {first, 1, std::pow(all, 1.0 / rounds) - 1.0};
}

// The schedule from the n-th round that overflowed on (docs that come in an
// order, by which those before do not predict those after): small rounds that
// cannot overflow, more of them each time.  Going on from that round and not
// from the first doc in rounds of 30,720: 16 queries of 10 over 2M docs in 1,000
// clusters 1.69 -> 0.24 ms, 64 queries 2.55 -> 0.54; a filter that passes
// nothing in the first 4,000 of 200,000 docs 0.78 -> 0.10 ms.
Schedule next_schedule(int n) {
  if (n <= 2) return {n == 1 ? 8192 : 16384, 1, 8.0};
  return {kSegmentSlots, int64_t{1} << std::min(n - 3, 30), n == 3 ? 4.0 : n == 4 ? 2.0 : 1.0};
}

// Doc bounds of a schedule's rounds from doc `from` on, aligned to bundles.
std::vector<int64_t> round_bounds(const Schedule& sc, int64_t from, int64_t num_docs) {
  static_assert(kSegmentSlots % kRoundAlign == 0, "small rounds stay aligned");
  std::vector<int64_t> b{from};
  for (int64_t pos = from; pos < num_docs;) {
    const int64_t done = pos - from;
    const int64_t step = done < sc.small * sc.first
                             ? sc.first
                             : std::max<int64_t>(1, static_cast<int64_t>(std::ceil(sc.growth * static_cast<double>(done))));
    pos = std::min(num_docs, pos + (step + kRoundAlign - 1) / kRoundAlign * kRoundAlign);
    b.push_back(pos);
  }
  return b;
}

// Words of pinned host memory that the last kernel of a schedule stores the
// overflowed round to (a copy of the word and the wait for it cost more than the
// small selections themselves).  A call holds one from before its first launch
// until it has waited for its stream; there are as many as calls ever ran at
// once.
class HostFlag {
 public:
  HostFlag() {
    {
      std::lock_guard<std::mutex> lk(mutex());
      if (!spare().empty()) {
        word_ = spare().back();
        spare().pop_back();
      }
    }
    if (word_ == nullptr) {
      void* p = nullptr;
      const hipError_t e = hipHostMalloc(&p, 64, hipHostMallocCoherent | hipHostMallocPortable);
      if (e != hipSuccess) throw Error(ST_ERR_HIP, cat("hipHostMalloc failed: ", hipGetErrorString(e)));
      word_ = static_cast<uint32_t*>(p);
    }
    take();
  }
  ~HostFlag() {
    if (pending) return;  // a kernel may still store to the word: it is not used again
    std::lock_guard<std::mutex> lk(mutex());
    spare().push_back(word_);
  }
  HostFlag(const HostFlag&) = delete;
  HostFlag& operator=(const HostFlag&) = delete;
  uint32_t* word() const { return word_; }
  // The word, cleared for the next schedule.
  uint32_t take() { return __atomic_exchange_n(word_, 0u, __ATOMIC_ACQ_REL); }
  bool pending = false;  // kernels that store to the word are in flight

 private:
  static std::mutex& mutex() {
    static std::mutex* m = new std::mutex;
    return *m;
  }
  static std::vector<uint32_t*>& spare() {
    static auto* v = new std::vector<uint32_t*>;
    return *v;
  }
  uint32_t* word_ = nullptr;
};

}  // namespace
}  // namespace st

extern "C" int64_t st_filtered_topk_workspace_bytes(int64_t num_queries) {
  if (num_queries <= 0) return 0;
  return num_queries * (4 + 4 + 8 * static_cast<int64_t>(st::kCandidateCapacity) +
                       4 * static_cast<int64_t>(st::kMaxSegments)) +
         256;
}

extern "C" int st_filtered_topk(const int64_t* packed, int64_t num_queries,
                                int64_t num_columns, int64_t num_docs,
                                const void* doc_embeddings, const void* query_embeddings,
                                int64_t dim, int64_t topk, void* workspace,
                                int64_t* out_ids, float* out_scores, void* stream) {
  using namespace st;
  return guarded([&] {
    ST_CHECK(num_queries >= 0 && num_columns >= 0 && num_docs >= 0, "negative sizes");
    ST_CHECK(topk >= 1 && topk <= kMaxTopk, "topk must be in [1, ", kMaxTopk, "], got ", topk);
    ST_CHECK(num_docs <= num_columns * kBitsPerColumn,
             "num_docs ", num_docs, " exceeds the mask's ", num_columns * kBitsPerColumn, " docs");
    ST_CHECK(num_docs <= 0xFFFFFFFFll, "doc ids must fit 32 bits");
    if (num_queries == 0) return;
    ST_CHECK(out_ids && out_scores && workspace, "null device pointer");
    ST_CHECK(num_docs == 0 || (packed && doc_embeddings && query_embeddings), "null device pointer");
    ST_CHECK(reinterpret_cast<uintptr_t>(doc_embeddings) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(query_embeddings) % 16 == 0,
             "embeddings must be 16-byte aligned");
    const bool few = few_queries(num_queries, num_docs, dim);
    const ScoreFn score = score_fn(dim, few);
    set_lds_limits();
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    TopkState state;
    state.counts = reinterpret_cast<uint32_t*>(ws);
    state.thr = reinterpret_cast<float*>(ws + 4 * num_queries);
    state.stop = reinterpret_cast<uint32_t*>(ws + 8 * num_queries);
    state.cand = reinterpret_cast<uint64_t*>(ws + ((8 * num_queries + 4 + 255) / 256) * 256);
    state.capacity = kCandidateCapacity;
    state.segn = reinterpret_cast<uint32_t*>(state.cand + num_queries * static_cast<int64_t>(kCandidateCapacity));
    state.seg = 0;
    const uint16_t* emb = static_cast<const uint16_t*>(doc_embeddings);
    const uint16_t* qv = static_cast<const uint16_t*>(query_embeddings);
    const uint64_t* m64 = reinterpret_cast<const uint64_t*>(packed);
    const unsigned qgrid = static_cast<unsigned>(num_queries);
    auto run_select = [&](TopkState st, int nseg, bool last, uint32_t* word) {
      hipLaunchKernelGGL(topk_select_kernel, dim3(qgrid), dim3(kSelectThreads), 0, s, st, topk, nseg,
                         last ? 1 : 0, out_ids, out_scores, word);
      check_launch("topk_select_kernel");
    };
    if (num_docs == 0) {  // every output is padding
      state.first_round = 1;
      state.check = 0;
      run_select(state, 0, true, nullptr);
      return;
    }

    HostFlag overflowed;
    Schedule schedule = first_schedule(few, num_queries, num_docs, topk);
    int64_t from = 0;
    for (int n = 0;;) {
      const std::vector<int64_t> bounds = round_bounds(schedule, from, num_docs);
      state.check = 0;
      for (size_t r = 0; r + 1 < bounds.size(); ++r) {
        state.first_round = bounds[r] == 0 ? 1 : 0;
        state.round = static_cast<uint32_t>(r + 1);
        const Segments segs = score(emb, qv, m64, num_columns, num_queries, bounds[r], bounds[r + 1], state, s);
        // the first round clears `stop`, and each schedule has to get on
        if (static_cast<int64_t>(r) < schedule.small && !segs.safe)
          fail("internal: ", segs.count, " segments of ", segs.slots, " slots cannot hold docs ", bounds[r],
               " to ", bounds[r + 1]);
        if (!segs.safe) {
          state.check = 1;
          overflowed.pending = true;
        }
        TopkState st = state;
        st.seg = segs.slots;
        run_select(st, segs.count, r + 2 == bounds.size(), overflowed.word());
      }
      if (n > 0 && state.check == 0) return;  // no round of this schedule could overflow
      const hipError_t e = hipStreamSynchronize(s);
      if (e != hipSuccess)
        throw Error(ST_ERR_HIP, cat("waiting for the selection failed: ", hipGetErrorString(e)));
      overflowed.pending = false;
      const uint32_t round = overflowed.take();
      if (round == 0) return;
      from = bounds[round - 1];
      schedule = next_schedule(++n);
    }
  });
}
