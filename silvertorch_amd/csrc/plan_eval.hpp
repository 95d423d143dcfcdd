// Evaluation of one compiled program (search_plan.hpp layouts) on one
// 64-bit column word per lane, with the row positions resolved by the lane
// itself from the term hashes (no width binding, no LDS).  Used by the
// cluster-restricted search and by the generic search kernel, which runs
// the programs the batch kernels do not take (deep stacks, very long
// queries).
#pragma once

#include <hip/hip_runtime.h>

#include "search_plan.hpp"
#include "st_common.hpp"

namespace st {

#define ST_EVAL_CONST __attribute__((address_space(4)))

struct EvalArgs {
  const int64_t* index;
  int64_t index_numel;
  int32_t hash_k;
  uint32_t pos_bytes;  // program term references are term * pos_bytes
};

// Where a lane's column sits.
struct Column {
  int64_t start;  // first row of the bundle
  int64_t b;      // bundle width
  int64_t cib;    // column within the bundle
  FastMod64 fm;
};

__device__ __forceinline__ Column column_of(const int64_t* bbo, int64_t col) {
  Column c;
  const int64_t bundle = col / kColumnsPerBundle;
  c.start = bbo[bundle];
  c.b = bbo[bundle + 1] - c.start;
  if (c.b < 0) c.b = 0;
  c.cib = col % kColumnsPerBundle;
  c.fm = make_fastmod_dev(static_cast<uint64_t>(c.b > 0 ? c.b : 1));
  return c;
}

// Word of one term on the lane's column: the AND of the rows at its first K
// distinct positions (int16)(h[p] % b), p < hash_k (signature_match,
// bloom_index_search.cpp:40-61); a bundle of width 0 matches nothing, a row
// outside the index reads as zero.
template <int K>
__device__ __forceinline__ uint64_t eval_term_word(const EvalArgs& a, const Column& c,
                                                   const ST_EVAL_CONST uint64_t* h) {
  int16_t found[K];
  int cnt = 0;
  uint64_t r = ~0ull;
  for (int p = 0; p < a.hash_k && cnt < K; ++p) {
    const int16_t bp = static_cast<int16_t>(fast_mod(h[p], c.fm));
    bool dup = false;
#pragma unroll
    for (int j = 0; j < K; ++j) dup |= (j < cnt) && (found[j] == bp);
    if (dup) continue;
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (j == cnt) found[j] = bp;
    ++cnt;
    const int64_t w = (c.start + bp) * kColumnsPerBundle + c.cib;
    r &= (w >= 0 && w < a.index_numel) ? static_cast<uint64_t>(a.index[w]) : 0ull;
  }
  return r;
}

// Terms whose rows are read together at most (kTermsAhead x K words in flight a
// lane).  Two at k = 4 and 5 keep 8 waves a SIMD (five or six with four terms)
// and measured the same or faster; at k = 3 four cost one wave of eight and
// gain 10% on trees.
template <int K>
constexpr int kTermsAhead = K <= 3 ? 4 : 2;

// out[u] = the word of the u-th of N terms, hashes_of(u) its hashes.  The rows
// are scattered over the index, so each read is a miss, and what bounds an item
// is how many of them wait for each other: the first K positions of every term
// are formed without a branch and their rows read back to back; only a term
// whose first K positions collide (about K^2 / 2b of them), or with a row
// outside the index, is evaluated position by position.  K = min(k, hash_k):
// there are K hashes.
template <int K, int N, typename HashesOf>
__device__ __forceinline__ void eval_term_group(const EvalArgs& a, const Column& c, HashesOf hashes_of,
                                                uint64_t* out) {
  uint64_t w[N][K];
  uint32_t again = 0;  // terms to evaluate position by position
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const ST_EVAL_CONST uint64_t* h = hashes_of(u);
    int16_t found[K];
    bool plain = true;
#pragma unroll
    for (int j = 0; j < K; ++j) found[j] = static_cast<int16_t>(fast_mod(h[j], c.fm));
#pragma unroll
    for (int j = 0; j < K; ++j) {
#pragma unroll
      for (int i = 0; i < j; ++i) plain &= found[i] != found[j];
      const int64_t at = (c.start + found[j]) * kColumnsPerBundle + c.cib;
      const bool inside = at >= 0 && at < a.index_numel;
      plain &= inside;
      w[u][j] = static_cast<uint64_t>(a.index[inside ? at : 0]);
    }
    again |= plain ? 0u : 1u << u;
  }
#pragma unroll
  for (int u = 0; u < N; ++u) {
    out[u] = w[u][0];
#pragma unroll
    for (int j = 1; j < K; ++j) out[u] &= w[u][j];
  }
  if (again != 0) {
#pragma unroll
    for (int u = 0; u < N; ++u)
      if ((again >> u) & 1u) out[u] = eval_term_word<K>(a, c, hashes_of(u));
  }
}

// out[u] = the word of the u-th of n terms (0 < n <= kTermsAhead, uniform over
// the wave).  A program's last group is as large as what is left of it: with
// many small clusters the work is bound by issue, and terms repeated to fill the
// group cost as much as real ones.  Partial search kernel, k = 3, 512 queries x
// 24 clusters of 200 docs, us by terms of a query (1 / 2 / 5 / trees of 3-12):
// row by row 10.4 / 14.1 / 26.2 / 103, groups filled up 20.4 / 18.8 / 29.8 /
// 50.6, these 11.8 / 14.1 / 22.6 / 46.8.
template <int K, typename HashesOf>
__device__ __forceinline__ void eval_term_words(const EvalArgs& a, const Column& c, uint32_t n, HashesOf hashes_of,
                                                uint64_t (&out)[kTermsAhead<K>]) {
  constexpr int A = kTermsAhead<K>;
  if constexpr (K == 0) {
#pragma unroll
    for (int u = 0; u < A; ++u) out[u] = ~0ull;
  } else {
#pragma unroll
    for (int u = 0; u < A; ++u) out[u] = 0;
    if (c.b <= 0 || a.index_numel <= 0) return;
    if (n >= A) {
      eval_term_group<K, A>(a, c, hashes_of, out);
    } else if (n == 1) {
      eval_term_group<K, 1>(a, c, hashes_of, out);
    } else if constexpr (A > 2) {
      if (n == 2)
        eval_term_group<K, 2>(a, c, hashes_of, out);
      else
        eval_term_group<K, 3>(a, c, hashes_of, out);
    }
  }
}

__device__ __forceinline__ uint64_t eval_combine(uint32_t op, uint64_t acc, uint64_t v) {
  if (op & 32u) v = ~v;
  const uint32_t mode = (op >> 3) & 3u;
  return mode == kModeSet ? v : (mode == kModeAnd ? (acc & v) : (acc | v));
}

// The program on the lane's column: flat form (OR of AND-groups) or stack
// form (accumulator machine with a stack of at most kStack words).
template <int K, int kStack>
__device__ uint64_t eval_program(const EvalArgs& a, const Column& c,
                                 const ST_EVAL_CONST uint32_t* prog,
                                 const ST_EVAL_CONST uint64_t* hashes) {
  const uint32_t hdr = prog[0];
  const uint32_t T = program_terms(hdr);
  auto term_hashes = [&](uint32_t ref) {
    return hashes + static_cast<uint64_t>(ref / a.pos_bytes) * a.hash_k;
  };
  constexpr uint32_t A = kTermsAhead<K>;
  uint64_t words[A];
  if (hdr & kFlatForm) {  // OR of AND-groups: [term ref, negate mask, group mask, 0]
    typedef uint32_t v4 __attribute__((ext_vector_type(4)));
    const ST_EVAL_CONST v4* lit = (const ST_EVAL_CONST v4*)(prog + kProgHeaderWords);
    uint64_t res = 0, acc = 0;
    for (uint32_t j = 0; j < T; j += A, lit += A) {
      const uint32_t n = T - j < A ? T - j : A;
      v4 rec[A];  // whole records at once: one wait for the scalar cache a group
#pragma unroll
      for (uint32_t u = 0; u < A; ++u) rec[u] = lit[u < n ? u : n - 1];
      eval_term_words<K>(a, c, n, [&](uint32_t u) { return term_hashes(rec[u].x); }, words);
#pragma unroll
      for (uint32_t u = 0; u < A; ++u) {
        if (u >= n) break;
        const uint64_t neg = rec[u].y ? ~0ull : 0ull;
        const uint64_t grp = rec[u].z ? ~0ull : 0ull;
        res |= acc & grp;
        acc = (acc | grp) & (words[u] ^ neg);
      }
    }
    res |= acc;
    return (hdr & kFlatComplement) ? ~res : res;
  }
  // stack form: T term references, then the operations
  const ST_EVAL_CONST uint32_t* tref = prog + kProgHeaderWords;
  const ST_EVAL_CONST uint32_t* ops = tref + T;
  const uint32_t nops = prog[2];
  uint64_t acc = 0;
  uint64_t stk[kStack];
  uint32_t sp = 0, t = 0;
  for (uint32_t i = 0; i < nops; ++i) {
    const uint32_t op = ops[i];
    const uint32_t code = op & 7u;
    if (code == kInsTerm) {
      if (t % A == 0) {
        const uint32_t n = T - t < A ? T - t : A;
        eval_term_words<K>(a, c, n, [&](uint32_t u) { return term_hashes(tref[t + u]); }, words);
      }
      uint64_t word = words[0];
#pragma unroll
      for (uint32_t u = 1; u < A; ++u) word = t % A == u ? words[u] : word;
      ++t;
      acc = eval_combine(op, acc, word);
    } else if (code == kInsConst) {
      acc = eval_combine(op, acc, ~0ull);
    } else if (code == kInsPush) {
      stk[sp < kStack ? sp : kStack - 1] = acc;  // the compiler bounds sp by kStack
      ++sp;
    } else if (code == kInsPop) {
      const uint64_t v = acc;
      --sp;
      acc = stk[sp < kStack ? sp : kStack - 1];
      acc = eval_combine(op, acc, v);
    } else {  // kInsNot
      acc = ~acc;
    }
  }
  return acc;
}

}  // namespace st
