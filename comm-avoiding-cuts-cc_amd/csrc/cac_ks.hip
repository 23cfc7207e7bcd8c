// cac_ks.hip -- dense Karger-Stein on gfx950: breadth-first recursive contraction
// over all trials at once, a many-workgroup compaction per level, and
// certificate-first leaves.
//
// Replaces comincut::minimum_cut_trials_start (dense, src/karger-stein/co_mincut.h:370-390),
// minimum_cut_trials (:315-342), recursive_contraction_inner (:176-223),
// contract_graph (:38-66) and the base case deterministic_cut_pr
// (co_mincut_base_case.hpp:164-185).  Sizes follow
// target_number_of_vertices_for_contraction (co_mincut.cpp:18-20).
//
// Per level of the recursion tree:
//   1. k_ks_contract<B>: one workgroup per child (B = 64 to 1024 threads by size)
//      draws s - t' picks, merges rows into pool rows, runs the PR pass and writes
//      the lists of live rows, live columns and merged-away columns.  The parent is
//      a matrix, or at the root the lists of its rows;
//   2. k_ks_compact: teams of threads each fold a live row's merged-away columns
//      into their representatives in LDS and write the child's row;
//   3. children of at most 128 vertices are leaves: k_ks_cert settles most of them
//      from row sums and maxima; k_ks_sw runs the phases of Stoer and Wagner with
//      the contractions of Nagamochi and Ibaraki on the rest.
// Entries are 32-bit where a root's total weight is below 2^32, else 64-bit.
// Device memory for a level comes from two grow-only buffers of the context used
// alternately (the parents live in one, the children in the other).
#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <vector>

#include "cac_internal.h"
#include "cac_ks.h"
#include "cac_ks_kernels.h"

namespace cac {
namespace {

// ---- leaves ------------------------------------------------------------------
// One wavefront per leaf: lane l owns vertices l and l + 64.
constexpr int kLeafMax = 128;
// Row stride of a leaf matrix in LDS: one entry more than a row, so a column
// (lane x reading or writing entry (x, c), as a merge and the PR scan do) spans
// the banks instead of hitting one: with 128 int64 per row every row starts on
// the same bank and a column access is a 64-way bank conflict.
constexpr int kLeafStride = kLeafMax + 1;

__device__ inline int64_t wave_sum_i64(int64_t x) { return (int64_t)wave_sum<uint64_t>((uint64_t)x); }

// d - (q-1) M, saturating to a large negative value instead of overflowing
// (a negative term only weakens the bound).
__device__ inline int64_t leaf_f(int64_t d, int64_t M, uint32_t q) {
  const int64_t k = (int64_t)q - 1;
  if (M != 0 && k > INT64_MAX / 256 / M) return INT64_MIN / 256;
  return d - k * M;
}

// Lower bound on the minimum cut of a leaf: for a side S with |S| = q <= V/2,
// cut(S) = sum over u in S of (d(u) - w(u, S \ u)) >= sum of f_q(u) over S, with
// f_q(u) = d(u) - (q-1) M(u) and M(u) the heaviest edge at u; so the min over q
// of the sum of the q smallest f_q bounds every cut from below.
__device__ int64_t leaf_lower_bound(const int64_t d[2], const int64_t M[2], const bool alive[2], uint32_t V,
                                    int64_t stop_at) {
  const int lane = threadIdx.x & 63;
  int64_t best = INT64_MAX;
  for (uint32_t q = 1; q <= V / 2; ++q) {
    int64_t f0 = alive[0] ? leaf_f(d[0], M[0], q) : INT64_MAX;
    int64_t f1 = alive[1] ? leaf_f(d[1], M[1], q) : INT64_MAX;
    // bitonic sort of 128 keys: element e = lane + 64 * r lives in register r
#pragma unroll
    for (int k = 2; k <= 128; k <<= 1) {
#pragma unroll
      for (int j = k >> 1; j > 0; j >>= 1) {
        if (j == 64) {
          // partner of lane's element 0 is its element 1
          bool up = (lane & k) == 0;  // k == 128 -> up for all
          if ((f0 > f1) == up) {
            int64_t t = f0;
            f0 = f1;
            f1 = t;
          }
        } else {
          int64_t p0 = __shfl_xor(f0, j, 64), p1 = __shfl_xor(f1, j, 64);
          bool lower = (lane & j) == 0;
          bool up0 = ((lane) & k) == 0, up1 = ((lane + 64) & k) == 0;
          int64_t mn0 = f0 < p0 ? f0 : p0, mx0 = f0 < p0 ? p0 : f0;
          int64_t mn1 = f1 < p1 ? f1 : p1, mx1 = f1 < p1 ? p1 : f1;
          f0 = (lower == up0) ? mn0 : mx0;
          f1 = (lower == up1) ? mn1 : mx1;
        }
      }
    }
    // sum of the q smallest: elements 0..q-1 (element e in register e / 64 of lane e % 64)
    int64_t part = ((uint32_t)lane < q ? f0 : 0) + ((uint32_t)(lane + 64) < q ? f1 : 0);
    const int64_t lb = wave_sum_i64(part);
    if (lb < best) best = lb;
    if (best < stop_at) break;
  }
  return best;
}

// Certificate first: a leaf whose lower bound reaches the trial's bound
// contributes the bound; the others are queued for Stoer-Wagner.
template <typename E>
__global__ void __launch_bounds__(64) k_ks_cert(const KsLeaf<E>* __restrict__ leaves, int64_t* __restrict__ results,
                                                uint32_t* __restrict__ sw_list, uint32_t* __restrict__ sw_count) {
  const KsLeaf<E> lf = leaves[blockIdx.x];
  const uint32_t V = lf.k;
  const int lane = threadIdx.x;
  const bool alive[2] = {(uint32_t)lane < V, (uint32_t)lane + 64 < V};
  int64_t d[2] = {0, 0}, M[2] = {0, 0};
  for (int h = 0; h < 2; ++h) {
    const uint32_t u = lane + 64 * h;
    if (!alive[h]) continue;
    if (lf.rsum && lf.rmax) {
      d[h] = (int64_t)lf.rsum[u];
      M[h] = (int64_t)lf.rmax[u];
    } else {
      int64_t sm = 0, mx = 0;
      for (uint32_t x = 0; x < V; ++x) {
        const int64_t v = (int64_t)lf.mat[(size_t)u * lf.ks + x];
        sm += v;
        mx = v > mx ? v : mx;
      }
      d[h] = sm;
      M[h] = mx;
    }
  }
  const int64_t lb = V >= 2 ? leaf_lower_bound(d, M, alive, V, lf.bound) : 0;
  // leaves whose total weight is below 2^32 (every entry and every merged
  // entry fits 32 bits) go to the front of the list, the others to the back
  const uint64_t total = wave_sum<uint64_t>((uint64_t)(d[0] + d[1]));
  if (lane == 0) {
    if (lb >= lf.bound) atomicMin((long long*)&results[lf.slot], (long long)lf.bound);
    else if (total < (1ull << 32)) sw_list[atomicAdd(&sw_count[0], 1u)] = blockIdx.x;
    else sw_list[gridDim.x - 1 - atomicAdd(&sw_count[1], 1u)] = blockIdx.x;
  }
}

// The base case of co_mincut_base_case.hpp:164-185 on a leaf in LDS: result
// min(bound, minimum cut).  Phases of maximum adjacency orders (Stoer and
// Wagner, J. ACM 44(4), 1997), each followed by the contractions of Nagamochi
// and Ibaraki (SIAM J. Discrete Math. 5(1), 1992): with `best` the smallest cut
// seen (the bound and the smallest degree to begin with), a vertex whose weight
// to the vertices ordered before it reaches `best` is connected to its
// predecessor by at least that much, so no cut below `best` separates the two.
// All such pairs of a phase are contracted at once; they are runs of
// consecutive vertices of the order.  The last vertex's weight is its degree
// and lowers `best` if it is smaller, so every phase contracts its last pair.
//
// A phase is a chain of V - 1 steps (a wave maximum, two ballots, one LDS row),
// so the phases are the cost.  Contracting only the last pair (and edges that
// alone reach the bound) took V - 1 phases of a leaf that no such edge
// collapses: 49 trials of a complete graph of 700 vertices, 1568 leaves of 128
// in 64-bit entries, took 21.4 of the solve's 25.3 ms; a phase contracts most of
// such a leaf at once, and the solve takes 5.7 ms.
// T: the LDS entry type, uint32_t for a leaf of total weight below 2^32 (66 KiB,
// two leaves per CU) and int64_t otherwise (132 KiB, one per CU).
template <typename T, typename E>
__global__ void __launch_bounds__(64) k_ks_sw(const KsLeaf<E>* __restrict__ leaves,
                                              const uint32_t* __restrict__ sw_list, int64_t* __restrict__ results) {
  typedef ks_sum_t<T> U;
  __shared__ T A[kLeafMax * kLeafStride];
  const KsLeaf<E> lf = leaves[sw_list[blockIdx.x]];
  const uint32_t V = lf.k;
  if (V < 2) return;  // no cut: the result keeps the bound
  const uint32_t lane = threadIdx.x;
  bool alive[2] = {lane < V, lane + 64 < V};
  U deg[2] = {0, 0};
#pragma unroll 8
  for (uint32_t r = 0; r < V; ++r)
    for (int h = 0; h < 2; ++h) {
      const uint32_t x = lane + 64 * h;
      if (x < V) {
        const U a = (U)lf.mat[(size_t)r * lf.ks + x];
        A[r * kLeafStride + x] = (T)a;
        deg[h] += a;  // symmetric: the column sum is the degree
      }
    }
  __syncthreads();
  U best = lf.bound <= 0 ? 0 : (uint64_t)lf.bound > (uint64_t)(U)~(U)0 ? (U)~(U)0 : (U)lf.bound;
  uint32_t nalive = V;
  {
    const U d0 = alive[0] ? deg[0] : (U)~(U)0, d1 = alive[1] ? deg[1] : (U)~(U)0;
    const U dmin = wave_min<U>(d0 < d1 ? d0 : d1);
    best = dmin < best ? dmin : best;
  }
  while (nalive > 1 && best > 0) {
    U key[2] = {0, 0};
    bool added[2] = {!alive[0], !alive[1]};
    uint32_t ord0 = 0, ord1 = 0;    // lane l: the vertices at positions l and l + 64 of the order
    uint64_t join0 = 0, join1 = 0;  // bit t: the vertex at position t (t + 64) joins its predecessor
    uint32_t merged = 0;
    const uint64_t live_lo = __ballot(alive[0]), live_hi = __ballot(alive[1]);
    uint32_t v = live_lo ? (uint32_t)(__ffsll((long long)live_lo) - 1)
                         : 64u + (uint32_t)(__ffsll((long long)live_hi) - 1);
    for (uint32_t step = 0;; ++step) {  // v takes position `step`
      ord0 = lane == step ? v : ord0;
      ord1 = lane + 64 == step ? v : ord1;
      added[0] = added[0] || lane == v;
      added[1] = added[1] || lane + 64 == v;
      if (step + 1 == nalive) break;
      for (int h = 0; h < 2; ++h) key[h] += (U)A[v * kLeafStride + lane + 64 * h];
      const U k0 = added[0] ? 0 : key[0], k1 = added[1] ? 0 : key[1];
      const U m = wave_max<U>(k0 > k1 ? k0 : k1);
      const uint64_t b0 = __ballot(!added[0] && key[0] == m), b1 = __ballot(!added[1] && key[1] == m);
      v = b0 ? (uint32_t)(__ffsll((long long)b0) - 1) : 64u + (uint32_t)(__ffsll((long long)b1) - 1);
      if (step + 2 == nalive && m < best) best = m;  // the last vertex: its degree, a cut
      if (m >= best) {
        if (step + 1 < 64) join0 |= 1ull << (step + 1);
        else join1 |= 1ull << (step - 63);
        ++merged;
      }
    }
    // Rows, then columns, of every run into its first vertex; a lane owns its
    // two columns in the first pass and its two rows in the second.
    auto joins = [&](uint32_t t) { return ((t < 64 ? join0 >> t : join1 >> (t - 64)) & 1ull) != 0; };
    auto at = [&](uint32_t t) { return t < 64 ? readlane_u32(ord0, (int)t) : readlane_u32(ord1, (int)(t - 64)); };
    bool dead[2] = {false, false};
    for (int pass = 0; pass < 2; ++pass) {
      const uint32_t sv = pass == 0 ? kLeafStride : 1, sl = pass == 0 ? 1 : kLeafStride;
      for (uint32_t p = 0; p + 1 < nalive;) {
        uint32_t e = p + 1;
        if (!joins(e)) {
          p = e;
          continue;
        }
        T* first = A + at(p) * sv + lane * sl;
        T a0 = first[0], a1 = first[64 * sl];
        for (; e < nalive && joins(e); ++e) {
          const uint32_t w = at(e);
          const T* row = A + w * sv + lane * sl;
          a0 += row[0];
          a1 += row[64 * sl];
          dead[0] = dead[0] || lane == w;
          dead[1] = dead[1] || lane + 64 == w;
        }
        first[0] = a0;
        first[64 * sl] = a1;
        p = e;
      }
      __syncthreads();
    }
    for (int h = 0; h < 2; ++h) {
      if (dead[h]) alive[h] = false;
      if (alive[h]) A[(lane + 64 * h) * (kLeafStride + 1)] = 0;  // loops of the merged vertices
    }
    __syncthreads();
    nalive -= merged;
  }
  const int64_t res = (int64_t)best < lf.bound ? (int64_t)best : lf.bound;
  if (lane == 0) atomicMin((long long*)&results[lf.slot], (long long)res);
}

// ---- contraction -------------------------------------------------------------
// LDS layout for a child of s vertices (U: unsigned sums of E): cap[s] U |
// cbs[nb] U | red[(kPieces + 1) B/64] U | misc[8] u32 | rep[s] u16 | wslot[s] u16,
// rep and cap padded to 16 bytes.  With 32-bit entries that is 8 s bytes: two
// 1024-thread workgroups of s = 8192 share a CU.
// A parent of row lists adds row[s] U, 16-byte aligned.
template <typename E>
__host__ __device__ inline size_t contract_lds_bytes(uint32_t s, int B, bool list = false) {
  const size_t e = sizeof(E), s8 = (s + 7) & ~size_t(7), nb2 = ((s + 63) / 64 + 3) & ~size_t(3);
  return e * s8 + e * nb2 + e * (size_t)(kPieces<E> + 1) * (B / 64) + 32 + 4 * s8 + 16 +
         (list ? e * s8 + 16 : 0);
}

template <typename E>
struct KsLds {
  ks_sum_t<E>* cap;
  ks_sum_t<E>* cbs;
  ks_sum_t<E>* red;
  uint32_t* misc;   // [0] i  [1] k  [2] rep[k]  [3], [4], [7] chains  [5] spare pool row  [6] pool rows handed out
  uint16_t* rep;    // padded entries past s hold 0xFFFF
  uint16_t* wslot;  // pool row of a merged row, or kNoRow
  ks_sum_t<E>* row;  // row lists: a row being assembled, 0 between; in a chain row cb
};

template <typename E>
__device__ inline const E* ks_row(const KsChild<E>& c, uint16_t slot, uint32_t r) {
  return slot == kNoRow ? c.parent + (size_t)r * c.ps : c.pool + (size_t)slot * ks_pool_stride(c.s);
}

// This thread's pieces of a row (0 past s).  The row pointer is generic (it comes
// from a struct in memory); as a global-address-space pointer the loads are
// global loads, which unlike flat loads do not count against the LDS wait
// counter, so the block's LDS waits between picks do not also wait for row loads
// in flight.  The last piece of a row is loaded entry by entry where it is not
// whole: what lies past s is not the row's.
template <int B, typename E>
__device__ inline void load_row(const E* row, uint32_t qc, uint32_t s, E (&v)[kKsChunk]) {
  typedef typename KsPiece<E>::type piece_t;
  typedef const __attribute__((address_space(1))) piece_t g_piece;
  typedef const __attribute__((address_space(1))) E g_e;
  constexpr uint32_t V = kPiece<E>, Q = kPieces<E>;
  g_e* g = (g_e*)row;
#pragma unroll
  for (uint32_t q = 0; q < Q; ++q) {
    const uint32_t x = (q * B + threadIdx.x) * V;
    if (q < qc && x + V <= s) {
      const piece_t p = *(g_piece*)(g + x);
#pragma unroll
      for (uint32_t j = 0; j < V; ++j) v[q * V + j] = p[j];
    } else {
#pragma unroll
      for (uint32_t j = 0; j < V; ++j) v[q * V + j] = q < qc && x + j < s ? g[x + j] : (E)0;
    }
  }
}

// This thread's pieces of row r, whose pool row is `slot`.  A row of a parent of
// lists is assembled in LDS, its entries written over zeros and the zeros put back
// by the threads that read them; between two rows the block meets a barrier (one
// wavefront's LDS accesses run in order).
template <int B, bool kList, typename E>
__device__ inline void fetch_row(const KsChild<E>& c, const KsLds<E>& L, uint16_t slot, uint32_t r, uint32_t qc,
                                 uint32_t s, E (&v)[kKsChunk]) {
  if constexpr (kList) {
    if (slot == kNoRow) {
      typedef ks_sum_t<E> U;
      typedef const __attribute__((address_space(1))) E g_e;
      typedef const __attribute__((address_space(1))) uint16_t g_u16;
      constexpr uint32_t V = kPiece<E>, Q = kPieces<E>;
      const uint32_t at = __builtin_amdgcn_readfirstlane(c.rp[r]), len = at & kKsListLen;
      g_u16* cols = (g_u16*)c.cols + (at >> kKsListBits);
      g_e* ws = (g_e*)c.ws + (at >> kKsListBits);
      for (uint32_t p = threadIdx.x; p < len; p += B) L.row[cols[p]] = (U)ws[p];
      __syncthreads();
      typedef U piece_t __attribute__((ext_vector_type(V)));
#pragma unroll
      for (uint32_t q = 0; q < Q; ++q) {
        const uint32_t x = (q * B + threadIdx.x) * V;
        const bool in = q < qc && x < s;  // the row's LDS is padded to whole pieces
        piece_t t = {};
        if (in) {
          t = *(piece_t*)(L.row + x);
          *(piece_t*)(L.row + x) = piece_t{};
        }
#pragma unroll
        for (uint32_t j = 0; j < V; ++j) v[q * V + j] = (E)t[j];
      }
      return;
    }
  }
  load_row<B>(ks_row(c, slot, r), qc, s, v);
}

// A pool row: whole pieces, the padding past s (0 in registers) included.
template <int B, typename E>
__device__ inline void store_row(E* row, uint32_t qc, uint32_t s, const E (&v)[kKsChunk]) {
  typedef typename KsPiece<E>::type piece_t;
  constexpr uint32_t V = kPiece<E>, Q = kPieces<E>;
#pragma unroll
  for (uint32_t q = 0; q < Q; ++q) {
    const uint32_t x = (q * B + threadIdx.x) * V;
    if (q < qc && x < s) {
      piece_t p;
#pragma unroll
      for (uint32_t j = 0; j < V; ++j) p[j] = v[q * V + j];
      *(piece_t*)(row + x) = p;
    }
  }
}

// Merge row a into row b (a dies, b keeps its index).  The calling threads hold
// their pieces of row `held` (a or b) in v, and in u the last merged row, row
// `cached` (kNoSlot before the first merge), which is the other row when
// u_has_other.  That row is written back lazily: its pool row is stale until it
// leaves the registers.  Otherwise the other row is loaded into u here, after
// row `cached` is written to its pool row if it is still live and not a or b
// (merged into b's new row or dead, it needs no write).  On return u holds the
// merged row (0 past s), not yet written.  Its pool row is b's, else a's (a
// dies), else the child's spare pool row (misc[5]), which thread 0 then
// replaces with a fresh one.  Every thread derives that destination from the
// same LDS words; thread 0 changes them only after the block sum's barrier,
// which every thread reaches after its reads, and the merge ends with one more
// barrier.  Each thread relabels only the representatives of the columns it
// owns.  Returns the contracted weight (cap[a] + cap[b] - cap_new) / 2 in w;
// false when the pool is exhausted.  Called by the whole block.
template <int B, bool kList, typename E>
__device__ bool ks_merge(const KsChild<E>& c, const KsLds<E>& L, uint32_t a, uint32_t b, uint32_t held,
                         const E (&v)[kKsChunk], E (&u)[kKsChunk], uint32_t cached, bool u_has_other, uint32_t qc,
                         ks_sum_t<E>& w) {
  typedef ks_sum_t<E> U;
  constexpr uint32_t V = kPiece<E>, Q = kPieces<E>;
  typedef uint16_t rep_t __attribute__((ext_vector_type(V), aligned(2 * V)));
  const uint32_t s = c.s;
  const uint32_t other = held == a ? b : a;
  const uint16_t slot_a = L.wslot[a], slot_b = L.wslot[b];
  const bool spare = slot_b == kNoRow && slot_a == kNoRow;
  const uint32_t db = slot_b != kNoRow ? slot_b : slot_a != kNoRow ? slot_a : L.misc[5];
  if (db == kNoSlot) return false;  // only a spare can be missing: the pool is exhausted
  if (!u_has_other) {
    if (cached != kNoSlot && cached != a && cached != b)  // a merged row has a pool row
      store_row<B>(c.pool + (size_t)L.wslot[cached] * ks_pool_stride(s), qc, s, u);
    fetch_row<B, kList>(c, L, other == a ? slot_a : slot_b, other, qc, s, u);
  }
  U sum = 0;
#pragma unroll
  for (uint32_t q = 0; q < Q; ++q) {
    const uint32_t x = (q * B + threadIdx.x) * V;
    if (q < qc && x < s) {
      rep_t rx = *(const rep_t*)(L.rep + x);
      bool hit_a = false;
#pragma unroll
      for (uint32_t j = 0; j < V; ++j) {
        E t = v[q * V + j] + u[q * V + j];
        if (rx[j] == a || rx[j] == b) t = 0;  // loop of the merged vertex
        if (rx[j] == a) {
          rx[j] = (uint16_t)b;
          hit_a = true;
        }
        u[q * V + j] = t;
        sum += (U)t;
      }
      if (hit_a) *(rep_t*)(L.rep + x) = rx;
    }
  }
  const U ca = L.cap[a], cb = L.cap[b];
  const U newcap = block_sum_open<B, U>(sum, L.red);
  w = (ca + cb - newcap) / 2;
  if (B == 64) __syncthreads();  // every lane has read the slots and capacities
  if (threadIdx.x == 0) {
    if (slot_b == kNoRow) {
      L.wslot[b] = (uint16_t)db;
      L.wslot[a] = kNoRow;
    }
    if (spare) {
      const uint32_t next = L.misc[6];
      L.misc[5] = next < c.pool_rows ? next : kNoSlot;
      L.misc[6] = next + 1;
    }
    L.cbs[a / 64] -= ca;
    L.cap[a] = 0;
    L.cbs[b / 64] += newcap - cb;
    L.cap[b] = newcap;
  }
  __syncthreads();
  return true;
}

// Waves per SIMD the contraction is compiled for.  32-bit entries: the two rows a
// thread keeps (the picked row and the last merged row) take 16 registers and
// the kernel fits 64 (8 waves: two 1024-thread workgroups per CU).  64-bit
// entries take 32: at most 96 registers below 1024 threads (5 waves; at 80 the
// kernel spills and is slower).  Row lists in 32-bit entries: 64 registers at 256
// threads, for 8 workgroups per CU of up to 1700 vertices although a few values
// spill (Watts-Strogatz, 32000 vertices: 34.1 ms, 38.2 with 80 registers and 6
// workgroups), 80 otherwise, where LDS leaves 6 waves.
template <int B, bool kList, typename E>
constexpr int kContractWaves =
    sizeof(E) == 4 ? (kList && B != 256 ? 6 : 8) : B >= 1024 ? 1 : kList ? 4 : 5;

// ---- chains ------------------------------------------------------------------
// With a parent of row lists nearly every merge of a sparse graph joins the heavy
// class cb and a vertex not merged before (439 picks and 1064 PR merges of a child
// of 1505 vertices had 17 others).  Wavefront 0 follows a chain of such merges
// alone: row cb stands in LDS, and a merge adds the vertex's list to it, where a
// merge by the block assembles rows and meets barriers.  The class's columns keep
// their label, cb at the chain's start, while its index `at` moves; chain_close
// puts the row back in u and the index in rep.  One hop is a chain of LDS and list
// loads: the 7974 children of 3987 such roots take 10.5 ms, 21.4 by the block alone
// (16.1 ms for 6472 as matrices).
template <int B, typename E>
__device__ void chain_open(const KsChild<E>& c, const KsLds<E>& L, uint32_t qc, const E (&u)[kKsChunk]) {
  typedef ks_sum_t<E> U;
  constexpr uint32_t V = kPiece<E>, Q = kPieces<E>;
  typedef U row_piece __attribute__((ext_vector_type(V)));
  __syncthreads();  // every thread has read the state that led here
#pragma unroll
  for (uint32_t q = 0; q < Q; ++q) {
    const uint32_t x = (q * B + threadIdx.x) * V;
    row_piece t;
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) t[j] = (U)u[q * V + j];
    if (q < qc && x < c.s) *(row_piece*)(L.row + x) = t;
  }
  __syncthreads();
}

// After wavefront 0 has written misc[3] = at: a barrier, then u, cb, rep and wslot.
template <int B, typename E>
__device__ void chain_close(const KsChild<E>& c, const KsLds<E>& L, uint32_t qc, E (&u)[kKsChunk], uint32_t& cb) {
  typedef ks_sum_t<E> U;
  constexpr uint32_t V = kPiece<E>, Q = kPieces<E>;
  typedef U row_piece __attribute__((ext_vector_type(V)));
  __syncthreads();
  const uint32_t label = cb;
  cb = L.misc[3];
#pragma unroll
  for (uint32_t q = 0; q < Q; ++q) {
    const uint32_t x = (q * B + threadIdx.x) * V;
    row_piece t = {};
    if (q < qc && x < c.s) {
      t = *(row_piece*)(L.row + x);
      *(row_piece*)(L.row + x) = row_piece{};
    }
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) u[q * V + j] = (E)t[j];
  }
  if (cb != label) {
    for (uint32_t x = threadIdx.x; x < c.s; x += B)
      if (L.rep[x] == label) L.rep[x] = (uint16_t)cb;
    if (threadIdx.x == 0) {  // the vertices that joined had no pool rows
      L.wslot[cb] = L.wslot[label];
      L.wslot[label] = kNoRow;
    }
  }
  __syncthreads();
}

// The first 64 entries of a row list, one per lane.
template <typename E>
struct ListHead {
  uint32_t p0, p1, x;
  ks_sum_t<E> w;
};
template <typename E>
__device__ inline ListHead<E> list_head(const KsChild<E>& c, const KsLds<E>& L, uint32_t y) {
  typedef const __attribute__((address_space(1))) E g_e;
  typedef const __attribute__((address_space(1))) uint16_t g_u16;
  ListHead<E> h;
  const uint32_t at = __builtin_amdgcn_readfirstlane(c.rp[__builtin_amdgcn_readfirstlane(y)]);
  h.p0 = at >> kKsListBits;
  h.p1 = h.p0 + (at & kKsListLen);
  const uint32_t p = h.p0 + (threadIdx.x & 63);
  h.x = p < h.p1 ? ((g_u16*)c.cols)[p] : 0u;
  h.w = p < h.p1 ? (ks_sum_t<E>)((g_e*)c.ws)[p] : 0;
  return h;
}

// Adds vertex y's list to the chain's row (label: the class's columns, which take
// nothing), and y to the class: returns the weight between them.  *low gets the
// smallest column whose entry reached the bound, or kNoSlot.
template <typename E>
__device__ inline ks_sum_t<E> chain_add(const KsChild<E>& c, const KsLds<E>& L, uint32_t y, const ListHead<E>& h,
                                        uint32_t label, ks_sum_t<E> bound, uint32_t* low) {
  typedef ks_sum_t<E> U;
  typedef const __attribute__((address_space(1))) E g_e;
  typedef const __attribute__((address_space(1))) uint16_t g_u16;
  const uint32_t lane = threadIdx.x & 63;
  uint32_t m = kNoSlot, x = h.x;
  U w = h.w;
  for (uint32_t p = h.p0 + lane; p < h.p1; p += 64) {
    if (p >= h.p0 + 64) {
      x = ((g_u16*)c.cols)[p];
      w = (U)((g_e*)c.ws)[p];
    }
    if (L.rep[x] != label) {  // a column once: no two lanes meet
      const U now = L.row[x] + w;
      L.row[x] = now;
      if (now >= bound && x < m) m = x;
    }
  }
  *low = wave_min<uint32_t>(m);
  const U between = readlane((U)L.row[y], 0);
  if (lane == 0) {
    L.row[y] = 0;
    L.rep[y] = (uint16_t)label;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  return between;
}

template <typename E>
__device__ inline bool chain_single(const KsLds<E>& L, uint32_t y) {  // not merged before: its row is the parent's
  return readlane_u32((uint32_t)L.rep[y], 0) == y && readlane_u32((uint32_t)L.wslot[y], 0) == kNoRow;
}

// Picks from number p on, while they join the class of cb and a single vertex.
// Returns the first pick left to the block; W, u, cb, nv and pr1 follow.
template <int B, typename E>
__device__ uint32_t pick_chain(const KsChild<E>& c, const KsLds<E>& L, uint32_t p, ks_sum_t<E> bound, uint32_t qc,
                               uint32_t nb, uint64_t& W, E (&u)[kKsChunk], uint32_t& cb, uint32_t& nv,
                               uint32_t& pr1) {
  typedef ks_sum_t<E> U;
  constexpr uint32_t V = kPiece<E>;
  typedef U row_piece __attribute__((ext_vector_type(V)));
  const uint32_t s = c.s, label = cb, lane = threadIdx.x & 63;
  chain_open<B>(c, L, qc, u);
  if (threadIdx.x < 64) {
    uint32_t at = cb;
    const uint32_t span = ((s + 63) / 64 + V - 1) / V * V;  // a lane's columns of the row
    for (; p + c.tgt < s && W != 0; ++p) {
      const u32x4 rnd = philox4x32(c.trial, c.nid, p, 0u, c.seed, kDomKs);
      const uint32_t i = wave_select_two_level<U>(L.cap, L.cbs, s, nb, (U)uniform1(lo64(rnd), W));
      if (i >= s) break;
      const U r = (U)uniform1(hi64(rnd), (uint64_t)readlane((U)L.cap[i], 0));
      uint32_t y = i;
      if (i == at) {  // the column of row cb whose prefix reaches r
        U sum = 0;
        const uint32_t x0 = lane * span, x1 = min(x0 + span, (s + V - 1) / V * V);  // padded to pieces of 0
        for (uint32_t x = x0; x < x1; x += V) {
          const row_piece t = *(const row_piece*)(L.row + x);
#pragma unroll
          for (uint32_t j = 0; j < V; ++j) sum += t[j];
        }
        const U inc = wave_incl_scan<U>(sum);
        const uint64_t hit = __ballot(inc >= r);
        if (!hit) break;
        const int owner = __ffsll((long long)hit) - 1;
        const U before = readlane((U)(inc - sum), owner);
        const uint32_t x = owner * span + lane;
        const U e = lane < span && x < s ? L.row[x] : 0;
        const U inc2 = wave_incl_scan<U>(e);
        const uint64_t hit2 = __ballot(lane < span && x < s && inc2 + before >= r);
        if (!hit2) break;
        y = owner * span + (uint32_t)(__ffsll((long long)hit2) - 1);
      }
      if (!chain_single(L, y)) break;
      const ListHead<E> h = list_head(c, L, y);
      if (i != at) {  // the column of the list whose prefix, in column order, reaches r
        const uint32_t len = h.p1 - h.p0;
        if (len > 64) break;
        U below = 0;
        for (uint32_t k = 0; k < len; ++k) {
          const uint32_t x = readlane_u32(h.x, k);
          const U w = readlane(h.w, k);
          below += x < h.x ? w : 0;
        }
        const uint64_t hit = __ballot(lane < len && below < r && r <= below + h.w);
        if (!hit) break;
        const uint32_t x = readlane_u32(h.x, __ffsll((long long)hit) - 1);
        if (readlane_u32((uint32_t)L.rep[x], 0) != label) break;
      }
      uint32_t low;
      const U w = chain_add(c, L, y, h, label, bound, &low);
      const uint32_t a = max(at, y), b = min(at, y);
      if (lane == 0) {
        const U ca = L.cap[a], cb0 = L.cap[b], now = ca + cb0 - 2 * w;
        L.cbs[a / 64] -= ca;
        L.cap[a] = 0;
        L.cbs[b / 64] += now - cb0;
        L.cap[b] = now;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      at = b;
      W -= 2 * (uint64_t)w;
      --nv;
      if (w >= bound) ++pr1;
    }
    if (lane == 0) {
      L.misc[0] = p;
      L.misc[3] = at;
      L.misc[4] = nv;
      L.misc[7] = pr1;
      ((uint32_t*)L.red)[0] = (uint32_t)W;
      ((uint32_t*)L.red)[1] = (uint32_t)(W >> 32);
    }
  }
  chain_close<B>(c, L, qc, u, cb);
  nv = L.misc[4];
  pr1 = L.misc[7];
  W = ((uint64_t)((uint32_t*)L.red)[1] << 32) | ((uint32_t*)L.red)[0];
  p = L.misc[0];
  __syncthreads();
  return p;
}

// Rows of the PR pass from i = cb on, while more than two vertices are left: row cb
// whose first entry of weight >= bound leads to a single vertex (the class takes its
// index), and single vertices whose first such entry leads to the class.  Returns
// the row left to the block, kNoSlot if none; u, cb and nv follow.
template <int B, typename E>
__device__ uint32_t pr_chain(const KsChild<E>& c, const KsLds<E>& L, uint32_t i, ks_sum_t<E> bound, uint32_t qc,
                             E (&u)[kKsChunk], uint32_t& cb, uint32_t& nv) {
  typedef ks_sum_t<E> U;
  typedef const __attribute__((address_space(1))) E g_e;
  typedef const __attribute__((address_space(1))) uint16_t g_u16;
  constexpr uint32_t V = kPiece<E>;
  typedef U row_piece __attribute__((ext_vector_type(V)));
  const uint32_t s = c.s, label = cb, lane = threadIdx.x & 63;
  chain_open<B>(c, L, qc, u);
  if (threadIdx.x < 64) {
    uint32_t at = cb, from = 0;  // no entry before column `from` reaches the bound
    ListHead<E> ahead;           // of vertex `guess`, the entry after the one taken
    uint32_t guess = kNoSlot;
    while (nv > 2) {
      uint32_t first = kNoSlot, second = kNoSlot, low = kNoSlot;
      if (i == at) {
        for (uint32_t b = from & ~(64 * V - 1); b < s && first == kNoSlot; b += 64 * V) {
          const uint32_t x = b + lane * V;
          const row_piece t = x < s ? *(const row_piece*)(L.row + x) : row_piece{};
          uint32_t bits = 0;
#pragma unroll
          for (uint32_t k = 0; k < V; ++k) bits |= t[k] >= bound ? 1u << k : 0u;
          uint64_t hit = __ballot(bits != 0);
          if (hit) {
            const int l = __ffsll((long long)hit) - 1;
            first = b + (uint32_t)l * V + (uint32_t)(__ffs((int)readlane_u32(bits, l)) - 1);
            if ((int)lane == l) bits &= bits - 1;
            hit = __ballot(bits != 0);
            if (hit) {
              const int l2 = __ffsll((long long)hit) - 1;
              second = b + (uint32_t)l2 * V + (uint32_t)(__ffs((int)readlane_u32(bits, l2)) - 1);
            }
          }
        }
        if (first != kNoSlot) {
          if (!chain_single(L, first)) break;
          const ListHead<E> h = guess == first ? ahead : list_head(c, L, first);
          guess = second;
          if (second != kNoSlot) ahead = list_head(c, L, second);
          const U w = chain_add(c, L, first, h, label, bound, &low);
          if (lane == 0) {
            L.cap[first] += L.cap[at] - 2 * w;
            L.cap[at] = 0;
          }
          from = min(first + 1, low);
          at = first;
          --nv;
        }
      } else {
        if (!chain_single(L, i)) break;
        const ListHead<E> h = guess == i ? ahead : list_head(c, L, i);
        uint32_t x = h.x;
        U w = h.w;
        for (uint32_t p = h.p0 + lane; p < h.p1; p += 64) {
          if (p >= h.p0 + 64) {
            x = ((g_u16*)c.cols)[p];
            w = (U)((g_e*)c.ws)[p];
          }
          if (w >= bound && x < first) first = x;
        }
        first = wave_min<uint32_t>(first);
        if (first != kNoSlot) {
          if (readlane_u32((uint32_t)L.rep[first], 0) != label) break;
          const U between = chain_add(c, L, i, h, label, bound, &low);
          if (lane == 0) {
            L.cap[at] += L.cap[i] - 2 * between;
            L.cap[i] = 0;
          }
          from = min(from, low);
          --nv;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      // the next row to check: a live one, or the class itself if its index is past i
      uint32_t next = kNoSlot;
      for (uint32_t b = (i + 1) & ~63u; b < s && next == kNoSlot; b += 64) {
        const uint32_t x = b + lane;
        const uint64_t hit = __ballot(x > i && x < s && (L.rep[x] == x || x == at) && L.cap[x] >= bound);
        if (hit) next = b + (uint32_t)(__ffsll((long long)hit) - 1);
      }
      i = next;
      if (next == kNoSlot) break;
      if (next != at && next != guess) {
        guess = next;
        ahead = list_head(c, L, next);
      }
    }
    if (lane == 0) {
      L.misc[0] = i;
      L.misc[3] = at;
      L.misc[4] = nv;
    }
  }
  chain_close<B>(c, L, qc, u, cb);
  nv = L.misc[4];
  i = L.misc[0];
  __syncthreads();
  return i;
}

// kList: the parents are row lists.  A sparse graph's matrix costs its n^2 entries
// three times, written once and read about once by each child, where the lists
// cost its edges.
template <int B, bool kList, typename E>
__global__ void __launch_bounds__(B, (kContractWaves<B, kList, E>))
    k_ks_contract(const KsChild<E>* __restrict__ children, uint32_t* __restrict__ k_out,
                  int64_t* __restrict__ results) {
  typedef ks_sum_t<E> U;
  constexpr uint32_t V = kPiece<E>, Q = kPieces<E>;
  extern __shared__ __align__(16) unsigned char smem[];
  const KsChild<E> c = children[blockIdx.x];
  const uint32_t s = c.s, nb = (s + 63) / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t s8 = (s + 7) & ~size_t(7), nb2 = (nb + 3) & ~size_t(3);
  KsLds<E> L;
  L.cap = (U*)smem;
  L.cbs = L.cap + s8;
  L.red = L.cbs + nb2;
  L.misc = (uint32_t*)(L.red + (kPieces<E> + 1) * (B / 64));
  L.rep = (uint16_t*)(((uintptr_t)(L.misc + 8) + 15) & ~uintptr_t(15));
  L.wslot = L.rep + s8;
  if constexpr (kList) {
    L.row = (U*)(((uintptr_t)(L.wslot + s8) + 15) & ~uintptr_t(15));
    for (uint32_t x = threadIdx.x; x < s8; x += B) L.row[x] = 0;
  }

  for (uint32_t x = threadIdx.x; x < s8; x += B) {
    L.cap[x] = x < s ? (U)c.prsum[x] : 0;
    L.rep[x] = x < s ? (uint16_t)x : (uint16_t)0xFFFF;
    L.wslot[x] = kNoRow;
  }
  if (threadIdx.x == 0) {  // the spare pool row of the first merge of two original rows
    L.misc[5] = c.pool_rows > 0 ? 0 : kNoSlot;
    L.misc[6] = 1;
  }
  __syncthreads();
  for (uint32_t blk = wave; blk < nb; blk += B / 64) {
    const uint32_t x = blk * 64 + lane;
    const U t = wave_sum<U>(x < s ? L.cap[x] : 0);
    if (lane == 0) L.cbs[blk] = t;
  }
  __syncthreads();
  uint64_t W = 0;
  for (uint32_t blk = 0; blk < nb; ++blk) W += L.cbs[blk];

  // A bound that no entry of the type reaches compares like the type's maximum.
  const U bound = c.bound > 0 && (uint64_t)c.bound > (uint64_t)(U)~(U)0 ? (U)~(U)0 : (U)c.bound;
  const uint32_t qc = (s + B * V - 1) / (B * V);  // pieces per thread, <= Q
  const uint32_t cc = (s + B - 1) / B;            // entries per thread in the closing pass
  const uint32_t lo = threadIdx.x * cc;
  uint32_t nv = s, pr1 = 0;
  int status = 0;  // 1 disconnected, 2 bad selection, 3 pool exhausted
  // v: the row being picked or checked; u: the last merged row, whose index is
  // cb (most picks touch it: the heavy super-vertex is picked or is the picked
  // row's partner, and the PR pass checks it next after merging into it), so
  // it is not loaded again
  E v[kKsChunk], u[kKsChunk];
  uint32_t cb = kNoSlot;
  bool chain = false;  // row lists: the last pick joined cb and a single vertex
  for (uint32_t p = 0; p + c.tgt < s; ++p) {
    if constexpr (kList) {
      if (chain) {
        p = pick_chain<B>(c, L, p, bound, qc, nb, W, u, cb, nv, pr1);
        if (p + c.tgt >= s) break;
      }
    }
    if (W == 0) {
      status = 1;
      break;
    }
    const u32x4 rnd = philox4x32(c.trial, c.nid, p, 0u, c.seed, kDomKs);
    if (wave == 0) {
      const uint32_t i = wave_select_two_level<U>(L.cap, L.cbs, s, nb, (U)uniform1(lo64(rnd), W));
      if (lane == 0) L.misc[0] = i;
    }
    __syncthreads();
    const uint32_t i = L.misc[0];
    if (i >= s) {
      status = 2;
      break;
    }
    if (i == cb) {
#pragma unroll
      for (uint32_t q = 0; q < kKsChunk; ++q) v[q] = u[q];
    } else {
      fetch_row<B, kList>(c, L, L.wslot[i], i, qc, s, v);
    }
    const uint32_t k =
        block_select_row<B, E>(v, qc, (U)uniform1(hi64(rnd), (uint64_t)L.cap[i]), L.red, L.misc + 1, L.rep);
    if (k >= s) {
      status = 2;
      break;
    }
    const uint32_t j = L.misc[2];  // rep[k], read by the selecting thread before the merge relabels
    const uint32_t a = i > j ? i : j, b = i > j ? j : i;
    if constexpr (kList)
      chain = (i == cb && L.wslot[j] == kNoRow) || (j == cb && L.wslot[i] == kNoRow);
    U w = 0;
    if (!ks_merge<B, kList, E>(c, L, a, b, i, v, u, cb, j == cb, qc, w)) {
      status = 3;
      break;
    }
    cb = b;
    W -= 2 * (uint64_t)w;
    --nv;
    if (w >= bound) ++pr1;
  }
  // PR pass (indexed_adjacency_matrix::pr_pass): contract every edge of weight >= bound
  if (status == 0 && pr1 > 0 && c.bound > 0) {
    for (uint32_t i = 0; i < s && nv > 2; ++i) {
      if (L.rep[i] != i || L.cap[i] < bound) continue;
      if constexpr (kList) {
        // the heavy class merges into one vertex after the other, its index each
        // time the next row to check
        if (i == cb) {
          i = pr_chain<B>(c, L, i, bound, qc, u, cb, nv);
          if (i >= s || nv <= 2) break;
        }
      }
      if (i == cb) {
#pragma unroll
        for (uint32_t q = 0; q < kKsChunk; ++q) v[q] = u[q];
      } else {
        fetch_row<B, kList>(c, L, L.wslot[i], i, qc, s, v);
      }
      uint32_t first = kNoSlot;
#pragma unroll
      for (uint32_t q = 0; q < Q; ++q) {
#pragma unroll
        for (uint32_t j = 0; j < V; ++j)  // an entry past s is 0, below the bound
          if (first == kNoSlot && (U)v[q * V + j] >= bound) first = (q * B + threadIdx.x) * V + j;
      }
      first = block_min_u32<B>(first, (uint32_t*)L.red);
      if (first == kNoSlot) continue;
      // rep[first] is not i: row i's entries of its own class are 0, below the
      // bound, so this merge's relabelling (of class i) leaves it unchanged
      U w = 0;
      const uint32_t tgt = L.rep[first];
      if (!ks_merge<B, kList, E>(c, L, i, tgt, i, v, u, cb, tgt == cb, qc, w)) {
        status = 3;
        break;
      }
      cb = tgt;
      --nv;
    }
  }
  if (status == 0 && cb != kNoSlot) store_row<B>(c.pool + (size_t)L.wslot[cb] * ks_pool_stride(s), qc, s, u);
  if (status != 0) {
    if (threadIdx.x == 0) {
      k_out[blockIdx.x] = status == 1 ? 0u : status == 2 ? kKsBad : kKsOverflow;
      if (status == 1) atomicMin((long long*)&results[c.slot], 0ll);
    }
    return;
  }
  // live rows and columns in natural order with the rows' sums (their
  // capacities), and the merged-away columns with their representatives
  __syncthreads();
  uint32_t cnt = 0;
#pragma unroll
  for (uint32_t k = 0; k < kKsChunk; ++k)
    if (k < cc && lo + k < s && L.rep[lo + k] == lo + k) ++cnt;
  uint32_t inc = cnt;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(inc, d, 64);
    if (lane >= d) inc += y;
  }
  if (lane == 63) L.red[wave] = inc;
  __syncthreads();
  uint32_t ex = inc - cnt, total = 0;
  for (int w2 = 0; w2 < B / 64; ++w2) {
    if (w2 < wave) ex += (uint32_t)L.red[w2];
    total += (uint32_t)L.red[w2];
  }
#pragma unroll
  for (uint32_t k = 0; k < kKsChunk; ++k) {
    const uint32_t x = lo + k;
    if (k >= cc || x >= s) break;
    const uint32_t rx = L.rep[x];
    if (rx == x) {
      const uint16_t sl = L.wslot[x];
      c.live[ex] = sl == kNoRow ? x : (kLiveWork | sl);
      c.repcol[ex] = (uint16_t)x;
      c.orsum[ex] = (E)L.cap[x];
      ++ex;
    } else {
      c.dead[x - ex] = x | (rx << 16);
    }
  }
  if (threadIdx.x == 0) k_out[blockIdx.x] = total;
}

// Threads per compaction workgroup of a class of children whose longest parent
// row takes row_bytes: the context's CAC_TUNE_KS_COMPACT_BLOCK setting for tgt's
// class, or 256, and 512 for rows above 16 KiB.
inline int compact_block(const cac_ctx* ctx, uint32_t tgt, size_t row_bytes) {
  const int cls = tgt <= 512 ? 0 : tgt <= 1024 ? 1 : tgt <= 2048 ? 2 : tgt <= 4096 ? 3 : 4;
  const int v = ctx->ks_compact_block[cls];
  return v ? v : row_bytes <= 16384 ? 256 : 512;
}
// A wavefront takes a row of its own up to this size, the whole workgroup above.
constexpr size_t kCompactWaveRow = 8192;

// Output rows per compaction workgroup.
__host__ __device__ inline uint32_t compact_rows(uint32_t tgt) {
  const uint32_t r = 8192 / (tgt ? tgt : 1);
  return r < 4 ? 4 : (r > 64 ? 64 : r);
}

// Team barrier: a team of one wavefront runs its LDS accesses in order, so only
// the compiler has to keep them in order.
template <int TEAM>
__device__ inline void team_sync() {
  if constexpr (TEAM == 64) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// One workgroup per (child, group of output rows), its rows dealt to teams of
// TEAM threads.  A team copies a live row to LDS with 16-byte loads, adds the
// entries of the merged-away columns to their representatives' (the only
// atomics), and writes the representatives' entries in column order.  The work
// item's child comes from a binary search of the per-child item prefix
// (item_prefix).  The bound is the rows' HBM traffic plus the LDS passes; adding
// every column into an accumulator by its class took s atomics per row instead
// of s - k.  Row maxima are written for leaves only, which alone read them.
// kList: the parents are row lists, a row's entries are written over zeros in LDS.
template <int CB, int TEAM, bool kList, typename E>
__global__ void __launch_bounds__(CB) k_ks_compact(const KsChild<E>* __restrict__ children,
                                                   const uint32_t* __restrict__ k_out,
                                                   const uint32_t* __restrict__ item_prefix, uint32_t nchild,
                                                   uint32_t row_stride) {
  typedef typename std::conditional<sizeof(E) == 4, uint32_t, unsigned long long>::type AccT;
  typedef typename KsPiece<E>::type piece_t;
  typedef ks_sum_t<E> U;
  constexpr uint32_t V = kPiece<E>;
  extern __shared__ __align__(16) unsigned char row_lds[];
  __shared__ U wave_top[CB / 64];
  const uint32_t team = threadIdx.x / TEAM, t = threadIdx.x % TEAM;
  AccT* row = reinterpret_cast<AccT*>(row_lds) + (size_t)team * row_stride;
  const uint32_t item = blockIdx.x;
  uint32_t lo = 0, hi = nchild;  // last child with item_prefix[child] <= item
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) / 2;
    if (item_prefix[mid] <= item) lo = mid;
    else hi = mid;
  }
  const KsChild<E> c = children[lo];
  const uint32_t kk = k_out[lo];
  if (kk == 0 || kk > c.tgt) return;  // disconnected child, or an error code
  const uint32_t R = compact_rows(c.tgt);
  const uint32_t r0 = (item - item_prefix[lo]) * R;
  if (r0 >= kk) return;
  const uint32_t r1 = min(r0 + R, kk);
  const uint32_t s = c.s, os = ks_stride<E>(kk), nd = s - kk;
  // Rows and lists are global memory (the struct's pointers are generic, which
  // would give flat loads).
  typedef const __attribute__((address_space(1))) piece_t g_piece;
  typedef const __attribute__((address_space(1))) E g_e;
  typedef const __attribute__((address_space(1))) uint16_t g_u16;
  typedef const __attribute__((address_space(1))) uint32_t g_u32;
  g_u16* repcol = (g_u16*)c.repcol;
  g_u32* dead = (g_u32*)c.dead;
  for (uint32_t r = r0 + team; r < r1; r += CB / TEAM) {
    const uint32_t e = c.live[r];
    if (kList && !(e & kLiveWork)) {
      for (uint32_t x = t; x < s; x += TEAM) row[x] = 0;
      team_sync<TEAM>();
      const uint32_t at = c.rp[e], len = at & kKsListLen;
      const uint16_t* cols = c.cols + (at >> kKsListBits);
      const E* ws = c.ws + (at >> kKsListBits);
      for (uint32_t p = t; p < len; p += TEAM) row[cols[p]] = (AccT)ws[p];
    } else {
      g_e* src = (g_e*)((e & kLiveWork) ? c.pool + (size_t)(e & ~kLiveWork) * ks_pool_stride(s)
                                        : c.parent + (size_t)e * c.ps);
#pragma unroll 4
      for (uint32_t x = t * V; x + V <= s; x += TEAM * V) *(piece_t*)(row + x) = *(g_piece*)(src + x);
      for (uint32_t x = s / V * V + t; x < s; x += TEAM) row[x] = (AccT)src[x];
    }
    team_sync<TEAM>();
#pragma unroll 4
    for (uint32_t i = t; i < nd; i += TEAM) {
      const uint32_t d = dead[i];
      const AccT v = row[d & 0xFFFFu];
      if (v) atomicAdd(&row[d >> 16], v);
    }
    team_sync<TEAM>();
    E* dst = c.out + (size_t)r * os;
    U mx = 0;
#pragma unroll 4
    for (uint32_t x = t; x < kk; x += TEAM) {
      const U v = (U)row[repcol[x]];
      dst[x] = (E)v;
      mx = v > mx ? v : mx;
    }
    if (kk <= kKsBase) {  // entries are non-negative, so the unsigned maximum is the maximum
      mx = wave_max<U>(mx);
      if (TEAM == 64) {
        if (t == 0) c.ormax[r] = (E)mx;
      } else {
        if ((t & 63) == 0) wave_top[t >> 6] = mx;
        __syncthreads();
        if (t == 0) {
          for (int w = 1; w < TEAM / 64; ++w) mx = wave_top[w] > mx ? wave_top[w] : mx;
          c.ormax[r] = (E)mx;
        }
      }
    }
    team_sync<TEAM>();
  }
}

// Row sums of a dense matrix (one wavefront per row) and their minimum, and on
// the way the matrix and the sums cut to 32 bits, row stride
// ks_stride<uint32_t>(n): exact copies when the sums add up to less than 2^32,
// which the host decides from the 64-bit sums.
__global__ void __launch_bounds__(256) k_row_sums(const int64_t* __restrict__ A, uint32_t n, int64_t* __restrict__ rsum,
                                                  int64_t* out_min, uint32_t* __restrict__ A32,
                                                  uint32_t* __restrict__ rsum32) {
  __shared__ long long wmin[4];
  long long best = INT64_MAX;
  const uint32_t st = ks_stride<uint32_t>(n);
  for (uint32_t r = blockIdx.x * 4 + (threadIdx.x >> 6); r < n; r += gridDim.x * 4) {
    const int64_t* row = A + (size_t)r * n;
    uint32_t* row32 = A32 + (size_t)r * st;
    uint64_t acc = 0;
    for (uint32_t x = threadIdx.x & 63; x < n; x += 64) {
      const uint64_t v = (uint64_t)row[x];
      acc += v;
      row32[x] = (uint32_t)v;
    }
    acc = wave_sum<uint64_t>(acc);
    if ((threadIdx.x & 63) == 0) {
      rsum[r] = (int64_t)acc;
      rsum32[r] = (uint32_t)acc;
    }
    best = (long long)acc < best ? (long long)acc : best;
  }
  if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    long long b = wmin[0];
    for (int w = 1; w < 4; ++w) b = wmin[w] < b ? wmin[w] : b;
    atomicMin((long long*)out_min, b);
  }
}

__global__ void k_fill_i64(int64_t* p, uint32_t count, int64_t v) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_zero_words(unsigned long long* p, uint32_t count) {
  for (uint32_t i = threadIdx.x; i < count; i += blockDim.x) p[i] = 0ull;
}

// Block size for a child of s vertices: the smallest power of two from 64 up
// with at most kKsChunk row entries per thread, unless the context holds a
// tuned size for the row-size class of s (cac_tune_set); any power of two from
// that minimum to 1024 gives the same results.
inline int contract_block(const cac_ctx* ctx, uint32_t s) {
  int B = 64;
  while (B < 1024 && (uint32_t)B * kKsChunk < s) B *= 2;
  const int cls = B == 64 ? 0 : B == 128 ? 1 : B == 256 ? 2 : B == 512 ? 3 : -1;
  if (cls >= 0 && ctx->ks_contract_block[cls] >= B) B = ctx->ks_contract_block[cls];
  return B;
}

constexpr uint32_t kFewChildren = 256;  // the CU count of an MI355X

// Bump carving with 64-byte alignment (level buffers hold millions of small arrays).
struct Carve64 {
  char* base;
  size_t off = 0;
  explicit Carve64(void* b) : base((char*)b) {}
  template <class T>
  T* take(size_t count) {
    off = (off + 63) & ~size_t(63);
    T* p = (T*)(base + off);
    off += count * sizeof(T);
    return p;
  }
};
inline size_t c64(size_t bytes) { return (bytes + 63) & ~size_t(63); }

}  // namespace

// Host mirror of co_mincut.cpp:18-20 (same double arithmetic).
uint32_t ks_target_host(uint32_t s) {
  int t = (int)std::ceil((double)s / std::sqrt((double)2)) + 1;
  return t > (int)kKsBase ? (uint32_t)t : kKsBase;
}

namespace {
inline uint32_t ks_target(uint32_t s) { return ks_target_host(s); }

// Grow-only level buffer `which` of the context.
int ks_reserve(cac_ctx* ctx, int which, size_t bytes, void** out) {
  int rc = grow_buffer(ctx, &ctx->ks_buf[which], &ctx->ks_bytes[which], bytes);
  *out = ctx->ks_buf[which];
  return rc;
}

// Device bytes of the per-child arrays of one child (out, sums, maxima, lists).
size_t child_bytes(uint32_t s, uint32_t t, size_t esize) {
  const size_t stride = esize == 4 ? ks_stride<uint32_t>(t) : ks_stride<int64_t>(t);
  return c64(stride * t * esize) + 2 * c64((size_t)t * esize) + c64((size_t)t * 4) + c64((size_t)t * 2) +
         c64((size_t)s * 4);
}
// Pool rows of a child in the first pass: one for every pick and 1/8 spare (at
// least 8) for the PR pass.  A child that needs more comes back as kKsOverflow.
uint32_t child_pool_rows(uint32_t s, uint32_t t) { return std::min(s, (s - t) + (s - t) / 8 + 8); }

template <typename E>
int run_leaves(cac_ctx* ctx, const std::vector<KsLeaf<E>>& leaves, int buf, int64_t* d_results, hipStream_t s) {
  typedef KsLeaf<E> Leaf;
  const size_t n = leaves.size();
  void* base = nullptr;
  int rc = ks_reserve(ctx, buf, c64(n * sizeof(Leaf)) + c64(n * 4) + 128, &base);
  if (rc) return rc;
  Carve64 cv(base);
  Leaf* d_leaves = cv.take<Leaf>(n);
  uint32_t* d_list = cv.take<uint32_t>(n);
  uint32_t* d_count = cv.take<uint32_t>(2);  // [0] 32-bit leaves (list front), [1] the others (list back)
  CAC_HIP(ctx, hipMemcpyAsync(d_leaves, leaves.data(), n * sizeof(Leaf), hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(64), 0, s, (unsigned long long*)d_count, 1u);
  prof_begin(ctx, "ks_cert", s);
  hipLaunchKernelGGL(k_ks_cert<E>, dim3((unsigned)n), dim3(64), 0, s, (const Leaf*)d_leaves, d_results, d_list,
                     d_count);
  prof_end(ctx, s);
  CAC_LAUNCH_CHECK(ctx, "ks certificate");
  CAC_HIP(ctx, hipMemcpyAsync(ctx->pinned, d_count, 8, hipMemcpyDeviceToHost, s));
  CAC_HIP(ctx, hipStreamSynchronize(s));
  const uint32_t n32 = ((uint32_t*)ctx->pinned)[0], n64 = ((uint32_t*)ctx->pinned)[1];
  if (n32 + n64) {
    prof_begin(ctx, "ks_sw", s);
    if (n32)
      hipLaunchKernelGGL((k_ks_sw<uint32_t, E>), dim3(n32), dim3(64), 0, s, (const Leaf*)d_leaves,
                         (const uint32_t*)d_list, d_results);
    if constexpr (sizeof(E) == 8) {  // a 32-bit leaf always goes to the front
      if (n64)
        hipLaunchKernelGGL((k_ks_sw<int64_t, E>), dim3(n64), dim3(64), 0, s, (const Leaf*)d_leaves,
                           (const uint32_t*)(d_list + (n - n64)), d_results);
    }
    prof_end(ctx, s);
    CAC_LAUNCH_CHECK(ctx, "ks stoer-wagner");
  }
  CAC_HIP(ctx, hipStreamSynchronize(s));
  return CAC_OK;
}

template <int B, typename E>
void launch_contract(const KsChild<E>* d_children, uint32_t count, uint32_t smax, bool list, uint32_t* d_kout,
                     int64_t* d_results, hipStream_t s) {
  const size_t lds = contract_lds_bytes<E>(smax, B, list);
  if (list)
    hipLaunchKernelGGL((k_ks_contract<B, true, E>), dim3(count), dim3(B), lds, s, d_children, d_kout, d_results);
  else
    hipLaunchKernelGGL((k_ks_contract<B, false, E>), dim3(count), dim3(B), lds, s, d_children, d_kout, d_results);
}
// TEAM 0: the whole workgroup.
template <int TEAM, typename E>
void launch_compact(int cb, dim3 grid, size_t lds, bool list, const KsChild<E>* dc, const uint32_t* dk,
                    const uint32_t* dp, uint32_t nc, uint32_t stride, hipStream_t s) {
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3((unsigned)cb), lds, s, dc, dk, dp, nc, stride); };
  auto pick = [&](auto block) {
    constexpr int CB = decltype(block)::value, T = TEAM ? TEAM : CB;
    go(list ? k_ks_compact<CB, T, true, E> : k_ks_compact<CB, T, false, E>);
  };
  if (cb == 1024) pick(std::integral_constant<int, 1024>{});
  else if (cb == 512) pick(std::integral_constant<int, 512>{});
  else pick(std::integral_constant<int, 256>{});
}

// One level's launches for the children ch (already in d_children's order, by
// block-size class and form of the parent): contraction per class; waits for the children's k_out;
// then the compaction, sized by those k (a child that the PR pass collapsed
// takes a few workgroups, not t' / rows of them), left running on the stream
// (the next level's work follows it there).
template <typename E>
int contract_level(cac_ctx* ctx, const std::vector<KsChild<E>>& ch, KsChild<E>* d_children, uint32_t* d_prefix,
                   uint32_t* d_kout, int64_t* d_results, std::vector<uint32_t>& kout, hipStream_t s) {
  const size_t nchild = ch.size();
  CAC_HIP(ctx, hipMemcpyAsync(d_children, ch.data(), nchild * sizeof(KsChild<E>), hipMemcpyHostToDevice, s));
  prof_begin(ctx, "ks_contract", s);
  std::vector<size_t> group;  // first child of each block-size class, then nchild
  size_t c0 = 0;
  while (c0 < nchild) {
    const int B = contract_block(ctx, ch[c0].s);
    size_t c1 = c0;
    uint32_t smax = 0;
    const bool list = ch[c0].parent == nullptr;
    while (c1 < nchild && contract_block(ctx, ch[c1].s) == B && (ch[c1].parent == nullptr) == list)
      smax = std::max(smax, ch[c1++].s);
    const uint32_t cnt = (uint32_t)(c1 - c0);
    group.push_back(c0);
    // The narrow block also where children are fewer than CUs: its wavefronts have
    // several pieces of a row to scan and fewer barriers to wait at (square_root of
    // G(1000, 0.05): contraction 0.82 ms with 64 threads, 0.86 with 128, 0.90 with
    // 256; of G(1000, 0.02) with weights to 2^30, 64-bit entries: the solve 1.37
    // ms with 64, 1.38 with 128, 1.42 with 256).
    if (B == 1024) launch_contract<1024, E>(d_children + c0, cnt, smax, list, d_kout + c0, d_results, s);
    else if (B == 512) launch_contract<512, E>(d_children + c0, cnt, smax, list, d_kout + c0, d_results, s);
    else if (B == 256) launch_contract<256, E>(d_children + c0, cnt, smax, list, d_kout + c0, d_results, s);
    else if (B == 128) launch_contract<128, E>(d_children + c0, cnt, smax, list, d_kout + c0, d_results, s);
    else launch_contract<64, E>(d_children + c0, cnt, smax, list, d_kout + c0, d_results, s);
    c0 = c1;
  }
  group.push_back(nchild);
  prof_end(ctx, s);
  CAC_LAUNCH_CHECK(ctx, "ks contract");
  CAC_HIP(ctx, hipMemcpyAsync(kout.data(), d_kout, nchild * 4, hipMemcpyDeviceToHost, s));
  CAC_HIP(ctx, hipStreamSynchronize(s));
  // compaction work items: ceil(k / rows) per child of 1 <= k <= t' (0 for a
  // disconnected child and for the error codes); one launch per block-size
  // class, so that a class of small children does not take the large ones' LDS
  std::vector<uint32_t>& item_prefix = ctx->ks_items;  // rewritten only after the next synchronisation
  item_prefix.clear();
  std::vector<uint32_t> items(group.size() - 1);
  for (size_t g = 0; g + 1 < group.size(); ++g) {
    uint32_t n = 0;
    for (size_t i = group[g]; i < group[g + 1]; ++i) {
      item_prefix.push_back(n);
      const uint32_t k = kout[i];
      if (k >= 1 && k <= ch[i].tgt) n += (k + compact_rows(ch[i].tgt) - 1) / compact_rows(ch[i].tgt);
    }
    items[g] = n;
  }
  CAC_HIP(ctx, hipMemcpyAsync(d_prefix, item_prefix.data(), nchild * 4, hipMemcpyHostToDevice, s));
  prof_begin(ctx, "ks_compact", s);
  for (size_t g = 0; g + 1 < group.size(); ++g) {
    if (items[g] == 0) continue;
    uint32_t smax = 0, tmax = 0;
    for (size_t i = group[g]; i < group[g + 1]; ++i) {
      smax = std::max(smax, ch[i].s);
      tmax = std::max(tmax, ch[i].tgt);
    }
    const uint32_t stride = (smax + 15) & ~15u;
    const size_t row_bytes = stride * sizeof(E);
    const bool waves = row_bytes <= kCompactWaveRow;
    const int cb = compact_block(ctx, tmax, row_bytes);
    const size_t lds = (waves ? cb / 64 : 1) * row_bytes;
    const KsChild<E>* dc = d_children + group[g];
    const uint32_t* dk = d_kout + group[g];
    const uint32_t* dp = d_prefix + group[g];
    const uint32_t nc = (uint32_t)(group[g + 1] - group[g]);
    const bool list = ch[group[g]].parent == nullptr;
    if (waves) launch_compact<64, E>(cb, dim3(items[g]), lds, list, dc, dk, dp, nc, stride, s);
    else launch_compact<0, E>(cb, dim3(items[g]), lds, list, dc, dk, dp, nc, stride, s);
  }
  prof_end(ctx, s);
  CAC_LAUNCH_CHECK(ctx, "ks compact");
  return CAC_OK;
}

}  // namespace

size_t ks_wave_trials(const cac_ctx* ctx, uint32_t t) {
  return (size_t)kFewChildren * (2048 / contract_block(ctx, t)) / 2;  // 2048 threads per CU
}

size_t ks_live_bytes_per_root(uint32_t n, bool w32) {
  // children of every node at one depth with their pool rows; a depth's
  // children go to the buffer its parents are not in, so the two buffers hold
  // the largest even and the largest odd depth
  const size_t esize = w32 ? 4 : 8;
  size_t best[2] = {0, 0};
  uint64_t nodes = 1;
  int depth = 0;
  for (uint32_t sz = n; sz > kKsBase; sz = ks_target(sz), nodes *= 2, ++depth) {
    const uint32_t t = ks_target(sz);
    // matrix, sums, live list, column list and node of a child, then its pool
    // rows; the few spare rows beyond 1/8 are not counted: a served query's
    // admitted bytes rest on this sum
    const size_t stride = w32 ? ks_stride<uint32_t>(t) : t;
    const size_t b = 2 * nodes * (c64(stride * t * esize) + 2 * c64((size_t)t * esize) + c64((size_t)sz * 4) +
                                  c64((size_t)t * 4) + 104 +
                                  (size_t)(sz - t) * ks_pool_stride(sz) * esize * 9 / 8);
    best[depth & 1] = std::max(best[depth & 1], b);
  }
  return best[0] + best[1] + 8192;
}

namespace {

// The contraction's and the compaction's dynamic LDS may exceed the default
// limit: raise it once.
template <typename E>
int contract_attr(cac_ctx* ctx) {
  static std::once_flag once;
  static hipError_t err = hipSuccess;
  std::call_once(once, [] {
    err = hipFuncSetAttribute((const void*)k_ks_contract<1024, false, E>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)contract_lds_bytes<E>(kKsMaxS, 1024));
    if (err == hipSuccess)
      err = hipFuncSetAttribute((const void*)k_ks_contract<512, false, E>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)contract_lds_bytes<E>(512 * kKsChunk, 512));
    if (err == hipSuccess)
      err = hipFuncSetAttribute((const void*)k_ks_contract<512, true, E>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)contract_lds_bytes<E>(kKsListMax, 512, true));
    if (err == hipSuccess)
      err = hipFuncSetAttribute((const void*)k_ks_contract<1024, true, E>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)contract_lds_bytes<E>(kKsListMax, 1024, true));
    const void* compact[] = {(const void*)k_ks_compact<1024, 64, false, E>,
                             (const void*)k_ks_compact<1024, 1024, false, E>,
                             (const void*)k_ks_compact<512, 512, false, E>,
                             (const void*)k_ks_compact<256, 256, false, E>,
                             (const void*)k_ks_compact<1024, 64, true, E>};
    for (const void* f : compact)
      if (err == hipSuccess)
        err = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)std::max<size_t>(16 * kCompactWaveRow, kKsMaxS * sizeof(E)));
  });
  CAC_HIP(ctx, err);
  return CAC_OK;
}

// Runs one Karger-Stein trial per root of entry type E.  roots[i]: device matrix
// (n_i x n_i, row stride ks_stride<E>(n_i)) with its row sums, trial id, result
// slot and bound; d_results[slot] must hold the bound already and receives
// min(bound, every leaf) by atomicMin.
template <typename E>
int ks_run_typed(cac_ctx* ctx, const std::vector<KsRoot>& roots, int64_t* d_results, hipStream_t s) {
  typedef KsChild<E> Child;
  struct Node {
    const E* mat;
    const E* rsum;
    const E* rmax;
    uint32_t s, trial, nid, slot;
    int64_t bound;
    uint32_t seed;
    const uint32_t* rp = nullptr;  // row lists in place of mat
    const uint16_t* cols = nullptr;
    const E* ws = nullptr;
  };
  int rc = contract_attr<E>(ctx);
  if (rc) return rc;
  // parents and children of a level live in the two level buffers
  BufPin pin0(ctx, kBufKs0), pin1(ctx, kBufKs1);

  std::vector<Node> level;
  for (const KsRoot& r : roots) {
    if (r.n > kKsMaxS) return fail(ctx, CAC_EINVAL, "dense Karger-Stein supports at most 8192 vertices");
    if (!r.mat && (r.n <= kKsBase || r.n > kKsListMax || !r.rp))
      return fail(ctx, CAC_EINVAL, "dense Karger-Stein root without a matrix");
    level.push_back({(const E*)r.mat, (const E*)r.rsum, nullptr, r.n, r.trial, r.nid, r.slot, r.bound, r.seed, r.rp,
                     r.cols, (const E*)r.ws});
  }
  int buf = 0;  // level buffer for the children of this level; the parents are in the other one
  while (!level.empty()) {
    std::vector<KsLeaf<E>> leaves;
    std::vector<Node> internal;
    for (auto& nd : level) {
      if (nd.s <= kKsBase) leaves.push_back({nd.mat, nd.rsum, nd.rmax, nd.s, ks_stride<E>(nd.s), nd.slot, nd.bound});
      else internal.push_back(nd);
    }
    if (!leaves.empty()) {
      rc = run_leaves<E>(ctx, leaves, buf, d_results, s);
      if (rc) return rc;
    }
    if (internal.empty()) break;
    // children sorted by block-size class (1024, 256, 64) and form of the parent,
    // two per internal node
    std::vector<std::pair<int, uint32_t>> order;
    for (uint32_t i = 0; i < internal.size(); ++i)
      order.push_back({-2 * contract_block(ctx, internal[i].s) + (internal[i].mat ? 0 : 1), i});
    std::stable_sort(order.begin(), order.end());
    const size_t nchild = 2 * internal.size();
    size_t arrays = 0;
    for (auto& nd : internal) {
      const uint32_t t = ks_target(nd.s);
      arrays += 2 * (child_bytes(nd.s, t, sizeof(E)) +
                     c64((size_t)child_pool_rows(nd.s, t) * ks_pool_stride(nd.s) * sizeof(E)));
    }
    std::vector<Child> ch(nchild);
    std::vector<uint32_t> kout(nchild);
    const size_t bytes = c64(nchild * sizeof(Child)) + c64((nchild + 1) * 4) + c64(nchild * 4) + arrays + 1024;
    void* base = nullptr;
    rc = ks_reserve(ctx, buf, bytes, &base);
    if (rc) return rc;
    Carve64 cv(base);
    Child* d_children = cv.take<Child>(nchild);
    uint32_t* d_prefix = cv.take<uint32_t>(nchild + 1);
    uint32_t* d_kout = cv.take<uint32_t>(nchild);
    size_t ci = 0;
    for (auto& o : order) {
      const Node& nd = internal[o.second];
      const uint32_t t = ks_target(nd.s);
      for (uint32_t k = 0; k < 2; ++k, ++ci) {
        Child& x = ch[ci];
        x.parent = nd.mat;
        x.prsum = nd.rsum;
        x.out = cv.take<E>((size_t)t * ks_stride<E>(t));
        x.orsum = cv.take<E>(t);
        x.ormax = cv.take<E>(t);
        x.live = cv.take<uint32_t>(t);
        x.repcol = cv.take<uint16_t>(t);
        x.dead = cv.take<uint32_t>(nd.s);
        x.pool_rows = child_pool_rows(nd.s, t);
        x.pool = cv.take<E>((size_t)x.pool_rows * ks_pool_stride(nd.s));
        x.s = nd.s;
        x.ps = ks_stride<E>(nd.s);
        x.tgt = t;
        x.trial = nd.trial;
        x.nid = 2 * nd.nid + k;
        x.slot = nd.slot;
        x.seed = nd.seed;
        x.bound = nd.bound;
        x.rp = nd.rp;
        x.cols = nd.cols;
        x.ws = nd.ws;
      }
    }
    rc = contract_level<E>(ctx, ch, d_children, d_prefix, d_kout, d_results, kout, s);
    if (rc) return rc;
    // children that ran out of pool rows: again, with s pool rows each (a child
    // merges at most s - 2 times, so this cannot overflow)
    std::vector<uint32_t> over;
    for (uint32_t i = 0; i < nchild; ++i)
      if (kout[i] == kKsOverflow) over.push_back(i);
    if (!over.empty()) {
      std::vector<Child> rch;
      size_t rpool = 0;
      for (uint32_t i : over) {
        rch.push_back(ch[i]);
        rpool += c64((size_t)ch[i].s * ks_pool_stride(ch[i].s) * sizeof(E));
      }
      const size_t no = rch.size();
      const size_t rbytes = c64(no * sizeof(Child)) + c64((no + 1) * 4) + c64(no * 4) + rpool + 1024;
      rc = grow_buffer(ctx, &ctx->ks_retry_buf, &ctx->ks_retry_bytes, rbytes);
      if (rc) return rc;
      Carve64 rv(ctx->ks_retry_buf);
      Child* d_rch = rv.take<Child>(no);
      uint32_t* d_rprefix = rv.take<uint32_t>(no + 1);
      uint32_t* d_rkout = rv.take<uint32_t>(no);
      for (Child& x : rch) {
        x.pool_rows = x.s;
        x.pool = rv.take<E>((size_t)x.s * ks_pool_stride(x.s));
      }
      std::vector<uint32_t> rkout(no);
      rc = contract_level<E>(ctx, rch, d_rch, d_rprefix, d_rkout, d_results, rkout, s);
      if (rc) return rc;
      for (size_t k = 0; k < no; ++k) {
        if (rkout[k] == kKsOverflow) return fail(ctx, CAC_EDEVICE, "Karger-Stein row pool overflow");
        kout[over[k]] = rkout[k];
      }
    }
    std::vector<Node> next;
    for (size_t i = 0; i < nchild; ++i) {
      if (kout[i] == kKsBad) return fail(ctx, CAC_EDEVICE, "Karger-Stein selection out of range");
      if (kout[i] == 0) continue;  // disconnected child: its 0 is already recorded
      next.push_back({ch[i].out, ch[i].orsum, ch[i].ormax, kout[i], ch[i].trial, ch[i].nid, ch[i].slot, ch[i].bound,
                      ch[i].seed, nullptr, nullptr, nullptr});
    }
    level.swap(next);
    buf ^= 1;
  }
  CAC_HIP(ctx, hipStreamSynchronize(s));
  return CAC_OK;
}

}  // namespace

// Roots of 32-bit and of 64-bit entries run one kind after the other.
int ks_run(cac_ctx* ctx, const std::vector<KsRoot>& roots, int64_t* d_results, hipStream_t s) {
  std::vector<KsRoot> kind[2];
  for (const KsRoot& r : roots) kind[r.w32 ? 1 : 0].push_back(r);
  int rc = CAC_OK;
  if (!kind[1].empty()) rc = ks_run_typed<uint32_t>(ctx, kind[1], d_results, s);
  if (rc == CAC_OK && !kind[0].empty()) rc = ks_run_typed<int64_t>(ctx, kind[0], d_results, s);
  return rc;
}

// Validates a host matrix: symmetric, zero diagonal, non-negative, no overflow.
int ks_check_matrix(cac_ctx* ctx, const int64_t* adj, uint32_t n) {
  long double total = 0;
  for (uint32_t i = 0; i < n; ++i) {
    if (adj[(size_t)i * n + i] != 0) return fail(ctx, CAC_EINVAL, "adjacency diagonal must be zero");
    for (uint32_t j = 0; j < n; ++j) {
      const int64_t v = adj[(size_t)i * n + j];
      if (v < 0) return fail(ctx, CAC_EINVAL, "negative edge weight");
      if (j > i && v != adj[(size_t)j * n + i]) return fail(ctx, CAC_EINVAL, "adjacency matrix is not symmetric");
      total += v;
    }
  }
  if (total >= 4.0e18L) return fail(ctx, CAC_ERANGE, "total weight exceeds int64 range");
  return CAC_OK;
}

int ks_dense_run(cac_ctx* ctx, const int64_t* d_adj, uint32_t n, uint32_t seed, uint32_t first_trial,
                 uint32_t ntrials, int64_t* raw_cuts, int64_t* min_cut, hipStream_t s) {
  if (ntrials == 0) return fail(ctx, CAC_EINVAL, "ntrials must be >= 1");
  if (n > kKsMaxS) return fail(ctx, CAC_EINVAL, "dense Karger-Stein supports at most 8192 vertices");
  // the root's row sums, bound and trial results, and its 32-bit copy
  const size_t n32 = (size_t)n * ks_stride<uint32_t>(n);
  int rc = grow_buffer(ctx, &ctx->sp_dense_buf, &ctx->sp_dense_bytes,
                       carve_size(8) + carve_size(8 * (size_t)n) + carve_size(8 * (size_t)ntrials) +
                           carve_size(4 * (size_t)n) + carve_size(4 * n32));
  if (rc) return rc;
  BufPin pin(ctx, kBufSpDense);
  Carver cv(ctx->sp_dense_buf);
  int64_t* d_bound = cv.take<int64_t>(1);
  int64_t* d_rsum = cv.take<int64_t>(n);
  int64_t* d_res = cv.take<int64_t>(ntrials);
  uint32_t* d_rsum32 = cv.take<uint32_t>(n);
  uint32_t* d_adj32 = cv.take<uint32_t>(n32);
  hipLaunchKernelGGL(k_fill_i64, dim3(1), dim3(64), 0, s, d_bound, 1u, (int64_t)INT64_MAX);
  hipLaunchKernelGGL(k_row_sums, dim3(grid_for(n, 4, 2048)), dim3(256), 0, s, d_adj, n, d_rsum, d_bound, d_adj32,
                     d_rsum32);
  CAC_LAUNCH_CHECK(ctx, "row sums");
  int64_t bound = 0;
  std::vector<int64_t> rs(n);  // the row sums: their total decides the entry type
  hipError_t e = hipMemcpyAsync(&bound, d_bound, 8, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipMemcpyAsync(rs.data(), d_rsum, 8 * (size_t)n, hipMemcpyDeviceToHost, s);
  const hipError_t e_sync = hipStreamSynchronize(s);
  if (e == hipSuccess) e = e_sync;
  if (e != hipSuccess) return hip_fail(ctx, e, "row sums");
  bool w32 = true;  // total weight below 2^32, checked without wrapping
  uint64_t total = 0;
  for (int64_t r : rs) {
    if (r < 0 || (uint64_t)r >= (1ull << 32) || (total += (uint64_t)r) >= (1ull << 32)) {
      w32 = false;
      break;
    }
  }
  hipLaunchKernelGGL(k_fill_i64, dim3(grid_for(ntrials, 256, 64)), dim3(256), 0, s, d_res, ntrials, bound);
  // trials run in batches whose two live levels fit in 3/4 of the free
  // memory: the top levels are chains of picks with one workgroup per child,
  // so the more trials a batch holds, the more CUs they keep busy.  Every
  // batch but the last is as large as that allows: at n = 8192 the first of
  // two then fills the CUs at the levels where children outnumber them (two
  // even batches of 85 left a partial round of workgroups in each)
  size_t avail = 0;
  rc = device_memory_available(ctx, &avail);
  const size_t per_trial = ks_live_bytes_per_root(n, w32);
  size_t batch = std::max<size_t>(1, (size_t)(0.75 * (double)avail) / per_trial);
  batch = std::min<size_t>(batch, ntrials);
  for (uint32_t t0 = 0; t0 < ntrials && rc == CAC_OK; t0 += (uint32_t)batch) {
    std::vector<KsRoot> roots;
    for (uint32_t t = t0; t < std::min<uint32_t>(ntrials, t0 + (uint32_t)batch); ++t)
      roots.push_back({w32 ? (const void*)d_adj32 : (const void*)d_adj,
                       w32 ? (const void*)d_rsum32 : (const void*)d_rsum, n, first_trial + t, t, bound, seed, 1, w32});
    rc = ks_run(ctx, roots, d_res, s);
  }
  if (rc == CAC_OK) {
    std::vector<int64_t> res(ntrials);
    hipError_t e2 = hipMemcpyAsync(res.data(), d_res, 8 * (size_t)ntrials, hipMemcpyDeviceToHost, s);
    if (e2 == hipSuccess) e2 = hipStreamSynchronize(s);
    if (e2 != hipSuccess) rc = hip_fail(ctx, e2, "trial results");
    int64_t mn = INT64_MAX;
    for (uint32_t t = 0; t < ntrials && rc == CAC_OK; ++t) {
      if (raw_cuts) raw_cuts[t] = res[t];
      mn = std::min(mn, res[t]);
    }
    if (rc == CAC_OK && min_cut) *min_cut = mn;
  }
  (void)hipStreamSynchronize(s);
  return rc;
}

}  // namespace cac

extern "C" {

int cac_ks_dense_dev(cac_ctx* ctx, const int64_t* d_adj, uint32_t n, uint32_t seed, uint32_t first_trial,
                     uint32_t ntrials, int64_t* raw_cuts, int64_t* min_cut, void* stream) {
  int rc = cac::bind(ctx);
  if (rc) return rc;
  if (!d_adj || n < 2) return cac::fail(ctx, CAC_EINVAL, "need a matrix with at least 2 vertices");
  return cac::ks_dense_run(ctx, d_adj, n, seed, first_trial, ntrials, raw_cuts, min_cut, cac::pick_stream(ctx, stream));
}

int cac_ks_dense(cac_ctx* ctx, const int64_t* adj, uint32_t n, uint32_t seed, uint32_t first_trial, uint32_t ntrials,
                 int64_t* raw_cuts, int64_t* min_cut) {
  int rc = cac::bind(ctx);
  if (rc) return rc;
  if (!adj || n < 2) return cac::fail(ctx, CAC_EINVAL, "need a matrix with at least 2 vertices");
  rc = cac::ks_check_matrix(ctx, adj, n);
  if (rc) return rc;
  hipStream_t s = ctx->stream;
  int64_t* d_adj = nullptr;
  CAC_HIP(ctx, hipMalloc((void**)&d_adj, (size_t)n * n * 8));
  hipError_t e = hipMemcpyAsync(d_adj, adj, (size_t)n * n * 8, hipMemcpyHostToDevice, s);
  if (e != hipSuccess) {
    (void)hipFree(d_adj);
    return cac::hip_fail(ctx, e, "upload matrix");
  }
  rc = cac::ks_dense_run(ctx, d_adj, n, seed, first_trial, ntrials, raw_cuts, min_cut, s);
  (void)hipStreamSynchronize(s);
  (void)hipFree(d_adj);
  return rc;
}

}  // extern "C"
