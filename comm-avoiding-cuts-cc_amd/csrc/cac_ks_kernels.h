// cac_ks_kernels.h -- device side of the dense Karger-Stein recursive contraction.
//
// One workgroup contracts one child of the recursion tree (indexed_adjacency_matrix /
// lazy_adjacency_matrix semantics, src/karger-stein/indexed_adjacency_matrix.hpp:137-191,
// lazy_adjacency_matrix.hpp:120-216):
//   - the parent matrix and its row sums are shared read-only by both children; a
//     child writes only the rows it merges into, into rows of its own pool (copy
//     on write, the row's pool index kept in LDS);
//   - capacities live in LDS with 64-entry block sums, so the row pick is a
//     two-level search by one wavefront;
//   - every thread owns the same entries of every row for the whole kernel, in
//     16-byte pieces interleaved over the block (thread t of B owns entries
//     (q B + t) V .. + V of piece q, V = 16 / entry size), so each load or store
//     instruction of a wavefront covers 1 KiB of a row; the picked row stays in
//     registers for the column pick and the merge, the last merged row stays
//     there too and is written to its pool row only when another merged row takes
//     its place while it is live, or when the child ends, and a thread only ever
//     reads back what it wrote itself;
//   - a PR pass (co_mincut.h:50-63) may follow; the kernel ends by writing the
//     lists of live rows and columns and of merged-away columns, and the live
//     rows' sums (their capacities), and a separate many-workgroup kernel compacts
//     the live rows into the child's t x t matrix.
// Entry type E: uint32_t when the root matrix's entries sum to less than 2^32 (no
// entry, row sum or merged entry of the recursion can then exceed it), int64_t
// otherwise.  The draws, the picks and the cuts are the same numbers either way.
// Leaves (<= 128 vertices) get a lower-bound certificate from those row sums and
// maxima; Stoer-Wagner runs only on the leaves it does not settle.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cac_common.h"
#include "cac_wave.h"

namespace cac {

constexpr uint32_t kKsBase = 128;        // base_case_size (co_mincut.h:24)
constexpr uint32_t kKsMaxS = 8192;       // LDS holds caps, reps and row slots for s <= this
constexpr uint32_t kKsChunk = 8;         // row entries per thread (s <= 8 * block size), x = k * B + t
constexpr uint32_t kKsUnit = 64;         // a pool row is padded to whole units of 64 entries
constexpr uint32_t kKsListMax = 4096;    // a root of at most this many vertices may be given as row lists
constexpr uint32_t kListBuildMax = 2048;  // lists built by one workgroup: two rows per thread
constexpr uint64_t kListShare = 20;      // a root goes as row lists at n / kListShare entries a row or fewer
constexpr uint32_t kKsListBits = 12, kKsListLen = (1u << kKsListBits) - 1;
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;
constexpr uint16_t kNoRow = 0xFFFFu;         // LDS: the row has no pool row (pool rows per child <= s <= 8192)
constexpr uint32_t kLiveWork = 0x80000000u;  // live[] entry: pool row of the child
constexpr uint32_t kKsBad = 0xFFFFFFFFu;       // k_out: selection out of range
constexpr uint32_t kKsOverflow = 0xFFFFFFFEu;  // k_out: row pool exhausted, rerun the child

// Row stride (entries) of a k x k matrix the engine reads: 32-bit rows are padded
// to whole 16-byte pieces.  A 64-bit matrix may come from a caller and is dense.
template <typename E>
__host__ __device__ inline uint32_t ks_stride(uint32_t k) {
  return sizeof(E) == 4 ? (k + 3u) & ~3u : k;
}
// Entries of a pool row.
__host__ __device__ inline uint32_t ks_pool_stride(uint32_t s) { return (s + kKsUnit - 1) / kKsUnit * kKsUnit; }

// 16-byte pieces of a row; a 64-bit row may start on any 8-byte boundary.
template <typename E>
struct KsPiece;
template <>
struct KsPiece<uint32_t> {
  typedef uint32_t type __attribute__((ext_vector_type(4), aligned(16)));
};
template <>
struct KsPiece<int64_t> {
  typedef int64_t type __attribute__((ext_vector_type(2), aligned(8)));
};
template <typename E>
constexpr uint32_t kPiece = 16 / sizeof(E);  // V: entries of a piece
template <typename E>
constexpr uint32_t kPieces = kKsChunk / kPiece<E>;  // pieces per thread

template <typename E>
struct KsChild {
  const E* parent;   // s x s, row stride ps
  const E* prsum;    // parent row sums [s]
  E* out;            // k x k compacted (k <= tgt), row stride ks_stride<E>(k)
  E* orsum;          // [tgt] row sums of out
  E* ormax;          // [tgt] row maxima of out
  E* pool;           // pool_rows merged rows of ks_pool_stride(s) entries
  uint32_t* live;    // [tgt] output row -> parent row, or kLiveWork | pool row
  uint16_t* repcol;  // [tgt] output column -> parent column that represents it
  uint32_t* dead;    // [s - k] merged-away columns: column | representative << 16
  uint32_t s, ps, tgt, trial, nid;
  uint32_t slot, seed;  // seed: Philox key word 0 of the child's trial
  uint32_t pool_rows;
  int64_t bound;
  const uint32_t* rp;    // a parent of row lists (parent null): see KsRoot
  const uint16_t* cols;
  const E* ws;
};

template <typename E>
struct KsLeaf {
  const E* mat;   // k x k, row stride ks
  const E* rsum;  // [k] row sums, or null
  const E* rmax;  // [k] row maxima, or null
  uint32_t k, ks, slot;
  int64_t bound;
};

// ---- wave / block reductions (wave primitives in cac_wave.h) --------------------
// Unsigned type of the sums over entries of type E.
template <typename E>
struct KsSum {
  typedef uint64_t type;
};
template <>
struct KsSum<uint32_t> {
  typedef uint32_t type;
};
template <typename E>
using ks_sum_t = typename KsSum<E>::type;

// Block sum over B threads; every thread gets the total.  lds: >= B/64 u64.
template <int B>
__device__ inline uint64_t block_sum_u64(uint64_t x, uint64_t* lds) {
  x = wave_sum<uint64_t>(x);
  if (B == 64) return x;
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = x;
  __syncthreads();
  uint64_t t = 0;
#pragma unroll
  for (int w = 0; w < B / 64; ++w) t += lds[w];
  __syncthreads();
  return t;
}
// Block sum over B threads, without a trailing barrier: the caller reaches a
// barrier before lds (>= B/64 entries) is written again.
template <int B, typename U>
__device__ inline U block_sum_open(U x, U* lds) {
  x = wave_sum<U>(x);
  if (B == 64) return x;
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = x;
  __syncthreads();
  U t = 0;
#pragma unroll
  for (int w = 0; w < B / 64; ++w) t += lds[w];
  return t;
}
template <int B>
__device__ inline uint32_t block_min_u32(uint32_t x, uint32_t* lds) {
  x = wave_min<uint32_t>(x);
  if (B == 64) return x;
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = x;
  __syncthreads();
  uint32_t t = 0xFFFFFFFFu;
#pragma unroll
  for (int w = 0; w < B / 64; ++w) t = min(t, lds[w]);
  __syncthreads();
  return t;
}

// First index i in [0, s) whose inclusive prefix of cap reaches r (1 <= r <= total),
// by one wavefront: 64-entry block sums first (lane l owns blocks 2l, 2l + 1),
// then the 64 entries of the chosen block.  kNoSlot when r exceeds the total.
template <typename U>
__device__ inline uint32_t wave_select_two_level(const U* cap, const U* cbs, uint32_t s, uint32_t nb, U r) {
  const int lane = threadIdx.x & 63;
  const uint32_t b0 = 2 * lane, b1 = b0 + 1;
  const U c0 = b0 < nb ? cbs[b0] : 0, c1 = b1 < nb ? cbs[b1] : 0;
  const U incl = wave_incl_scan<U>(c0 + c1);
  const uint64_t hit = __ballot(incl >= r);
  if (!hit) return kNoSlot;
  const int owner = __ffsll((long long)hit) - 1;
  const U before = readlane((U)(incl - c0 - c1), owner);
  const U oc0 = readlane(c0, owner);
  uint32_t blk = 2 * owner;
  U rr = r - before;
  if (rr > oc0) {
    rr -= oc0;
    blk += 1;
  }
  const uint32_t x = blk * 64 + lane;
  const U v = x < s ? cap[x] : 0;
  const U inc2 = wave_incl_scan<U>(v);
  const uint64_t hit2 = __ballot(x < s && inc2 >= rr);
  if (!hit2) return kNoSlot;
  return blk * 64 + (uint32_t)(__ffsll((long long)hit2) - 1);
}

// First index (natural column order) of a row whose inclusive prefix reaches r
// (1 <= r), with the row held in registers by pieces: thread t holds entries
// x = (q B + t) V + j, q < qc, j < V, and 0 for x >= s.  Natural order is segment
// q by segment q (B V entries each), thread by thread inside a segment, so a
// thread's sum of a piece is one term of its segment's scan: every wave's
// segment totals go to LDS (one barrier); then each thread finds the segment
// where the prefix reaches r and its wave's offset inside it, and the one thread
// whose piece holds r walks its V entries and publishes the index (a second
// barrier), with rep[index] in lds_idx[1]: it reads that entry before the
// barrier, so a merge that relabels representatives right after cannot race with
// it.  lds: kPieces * B/64 sums.  kNoSlot if the row total is below r.  The
// caller reaches a barrier before lds or lds_idx is written again.
template <int B, typename E>
__device__ inline uint32_t block_select_row(const E (&v)[kKsChunk], uint32_t qc, ks_sum_t<E> r, ks_sum_t<E>* lds,
                                            uint32_t* lds_idx, const uint16_t* rep) {
  typedef ks_sum_t<E> U;
  constexpr int W = B / 64;
  constexpr uint32_t V = kPiece<E>, Q = kPieces<E>;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  U inc[Q], sum[Q];
#pragma unroll
  for (uint32_t q = 0; q < Q; ++q) {
    inc[q] = sum[q] = 0;
    if (q < qc) {
#pragma unroll
      for (uint32_t j = 0; j < V; ++j) sum[q] += (U)v[q * V + j];
      inc[q] = wave_incl_scan<U>(sum[q]);
      if (lane == 63) lds[q * W + wave] = inc[q];
    }
  }
  __syncthreads();
  // a segment's wave totals are scanned by the first W lanes of every wave, or read
  // by all where there are two at most (square_root of G(1000, 0.04) with weights to
  // 2^30, 64-bit entries: the solve 1.51 -> 1.48 ms)
  U before = 0, ex = 0, piece = 0;
  uint32_t qs = kNoSlot;
#pragma unroll
  for (uint32_t q = 0; q < Q; ++q) {
    if (q < qc && qs == kNoSlot) {
      U tot = 0, earlier = 0;
      if constexpr (W <= 2) {
#pragma unroll
        for (int w = 0; w < W; ++w) {
          const U t = lds[q * W + w];
          earlier += w < wave ? t : 0;
          tot += t;
        }
      } else {
        const U sc = row_incl_scan<U>(lane < W ? lds[q * W + lane] : 0);
        tot = readlane(sc, W - 1);
        earlier = wave > 0 ? readlane(sc, wave - 1) : 0;
      }
      if (before + tot >= r) {
        qs = q;
        piece = sum[q];
        ex = before + earlier + inc[q] - sum[q];
      } else {
        before += tot;
      }
    }
  }
  if (qs == kNoSlot) return kNoSlot;  // the same for every thread
  if (piece != 0 && ex < r && r <= ex + piece) {  // exactly one thread
    uint32_t j = 0;
#pragma unroll
    for (uint32_t q = 0; q < Q; ++q) {
      if (q == qs) {
        U p = ex;
        bool open = true;
#pragma unroll
        for (uint32_t k = 0; k < V; ++k) {
          p += (U)v[q * V + k];
          if (open && p >= r) {
            j = k;
            open = false;
          }
        }
      }
    }
    const uint32_t x = (qs * B + threadIdx.x) * V + j;
    lds_idx[0] = x;
    lds_idx[1] = rep[x];
  }
  __syncthreads();
  return *lds_idx;
}

}  // namespace cac
