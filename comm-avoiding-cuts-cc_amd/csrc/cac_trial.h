// cac_trial.h -- one sqrt-cut trial's device scratch, shared by the
// workgroup-per-trial sampling kernels and the wide (grid-per-trial) ones
// (internal).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "cac_internal.h"

namespace cac {

// One sampling job = one sqrt-cut trial of one graph; a launch runs one
// workgroup per job, so trials of different graphs share a launch.
struct TrialScratch {
  const cac_edge* edges;  // the job's graph (ids local to it)
  uint64_t m;
  uint32_t n, t;          // vertices, intermediate size
  uint32_t trial, slot;   // Philox trial id, result slot
  uint32_t seed;          // Philox key word 0 of the trial
  uint32_t dpr;           // draws per round: 0 = |V| (low-concurrency rule), else that many
  uint32_t* lab;          // [n]
  uint32_t* par;          // [n]
  uint64_t* pre;          // [m]
  uint2* draws;           // [n]
  void* mat;              // [t x t] entries of trial_w32's type, row stride ks_stride
  void* rsum;             // [t] row sums of mat, same type (may be null)
  uint32_t* nv_out;       // [1]
  // [1] of the job's graph, nonzero when an edge is a loop or two weights
  // differ (may be null: then every round builds the prefix)
  const uint32_t* mixed;
  // [1] total edge weight of the job's graph, saturating (null: entries are 64-bit)
  const unsigned long long* total;
  // The graph packed for trials in 32-bit arithmetic (null: not packed): endpoints
  // u | v << 16 and the inclusive prefix of the weights with loops counted as 0
  // (unless every edge weighs the same, with no loop).  Such a trial keeps its
  // labels as u16 in lab, its surviving edges and their prefix in pre's 2 m
  // words, its draws as la | lb << 16, and leaves in live[0] the number of edges
  // of its last scan and in live[1] whether they are its own list's.
  const uint32_t* pk;
  const uint32_t* pre0;
  uint32_t* live;  // live[1] = 2 when the contracted graph is left as row lists (TrialLists) in mat's place
};
// Of a trial that is not packed, once k_trial_rows has run: live[1] = 0 when its
// 32-bit matrix is followed by its row lists (live[0] entries), else 3.

// Row lists of a packed trial's contracted graph (the form of KsRoot) in the t^2
// words of its matrix; cap entries, and as many placed ones before they are merged.
struct TrialLists {
  uint32_t cap;
  uint32_t *rp, *ws, *pws;
  uint16_t *cols, *pcols;
  __host__ __device__ TrialLists(void* mat, uint32_t k, uint32_t share) : cap(k * k / share) {
    rp = (uint32_t*)mat;
    ws = rp + k;
    pws = ws + cap;
    cols = (uint16_t*)(pws + cap);
    pcols = cols + cap;
  }
};

// The contracted matrix's entries add up to at most twice the graph's total
// weight: below 2^32 the matrix and its row sums are uint32_t, else int64_t.
constexpr unsigned long long kTrialW32Total = 1ull << 31;
__device__ inline bool trial_w32(const TrialScratch& S) { return S.total && *S.total < kTrialW32Total; }
__device__ inline bool trial_packed(const TrialScratch& S) { return S.pk && trial_w32(S); }

// What makes two jobs' graphs one: the jobs of a batch may take different parts of
// one edge list from the same place (prefixes of it), and a graph's flag, total
// and packed form belong to all of its m edges; n decides whether it is packed.
struct GraphKey {
  const cac_edge* edges;
  uint64_t m;
  uint32_t n;
  bool operator==(const GraphKey& o) const { return edges == o.edges && m == o.m && n == o.n; }
};
struct GraphHash {
  size_t operator()(const GraphKey& k) const {
    uint64_t h = (uint64_t)(uintptr_t)k.edges;
    for (const uint64_t x : {k.m, (uint64_t)k.n}) h = (h ^ (h >> 29)) * 0x9E3779B97F4A7C15ull + x;
    return (size_t)(h ^ (h >> 32));
  }
};

// Device bytes of the per-trial state of the wide form beside TrialScratch's
// buffers (tile totals and the round's control words).
size_t wide_trial_bytes(uint64_t m, uint32_t n);

// Wide trials: every trial of h (device copies at d_scr, k = h.size()) runs its
// sampling rounds as grid-wide kernels over its edge list instead of in one
// workgroup, with the same draws, draw-prefix lengths and canonical labels.
// work holds k * wide_trial_bytes(m, n) bytes carved in order (the caller's
// sizes).  On return (queued on s, after two host synchronisations per round)
// lab holds the canonical labels and *nv_out the super-vertex count.
int wide_sample(cac_ctx* ctx, const std::vector<TrialScratch>& h, const TrialScratch* d_scr, void* work,
                hipStream_t s);
// Then the t x t matrix, row sums and bound of each trial, as k_densify_trials
// writes them: bounds[i] (i indexes h) and results[h[i].slot].
int wide_densify(cac_ctx* ctx, const std::vector<TrialScratch>& h, const TrialScratch* d_scr, void* work,
                 int64_t* bounds, int64_t* results, hipStream_t s);

// Smallest edge count that runs a trial in the wide form (the context's
// setting or the built-in 2^20).
uint64_t wide_min_edges(const cac_ctx* ctx);

}  // namespace cac
