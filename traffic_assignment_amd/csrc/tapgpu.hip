// tapgpu.hip -- gfx950 Frank-Wolfe user-equilibrium engine (C ABI in
// include/tapgpu.h).
//
// Replaces the reference's per-iteration work (trunk/tap/tap_frankwolfe_*.c,
// trunk/tap/pape_*.cu, trunk/tap/volume_update_*.cu) with HBM-resident state
// and these kernel families, all FP64 and none of them MFMA-shaped:
//
//  * shortest paths and loading, one origin per workgroup: the path of almost
//    every call, with labels in LDS (k_origin_lds) where they fit and in HBM
//    (k_origin_hbm) where not; a batch's variants in the lanes of a wavefront
//    where that is faster (taplanes.inc); whole iterations of the smallest
//    networks in one workgroup (taptiny.inc).
//  * all-origin shortest paths (any size): node-major labels dist[v][col] with one
//    origin per wavefront lane (64 origins per "group"); pull relaxations
//    over an explicit worklist of (node, group) items; a node's out-neighbours
//    are queued for the next sweep when any lane improved, deduplicated by a
//    per-(node, group) stamp and compacted with a wavefront ballot/prefix.
//    Labels are the least fixed point of fl(dist[u] + w) over paths whose
//    inner nodes are not zones (trunk/tap/sssp_pape.c:355), so they are
//    bit-identical to d'Esopo-Pape's for any relaxation order.
//  * their all-or-nothing loading: bottom-up accumulation on the predecessor trees
//    (children counted in a dense pass, then ready nodes push their subtree
//    demand to the parent level by level); per-group partial link volumes are
//    summed in a fixed order, so volumes are deterministic (and exact for
//    integer demand, where the reference's path walk is exact too).
//  * link passes: one fused pass evaluates g(0) = sum c*d, the Beckmann
//    objective, VHT and g(2^-j) for a window of j (the only step sizes the
//    reference's bisection ever tests, trunk/tap/tap_functions.c:469-507)
//    with compensated block sums, and the last of a variant's blocks picks
//    lambda and updates gap / relative gap; an update pass does
//    x += lambda*d and BPR.
//  * everything is per "variant": a batch of TAPs over one union topology
//    (uneven link sets via a presence mask) runs in the same launches.
//
// Build: hipcc --offload-arch=gfx950 -O3 -ffp-contract=off (no FMA
// contraction: every + and * is one IEEE rounding, as on the reference host).

#include <hip/hip_runtime.h>

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <climits>
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "../../include/tapgpu.h"
#include "tapmath.h"

namespace {

constexpr int kWave = 64;
constexpr int kBlock = 256;                 // 4 wavefronts
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kGridVariants = 65535;        // variants of a launch in the grid's second dimension
constexpr int kJ = 16;                      // step sizes 2^-j evaluated per link pass
constexpr int kQ = 3 + kJ;                  // g0, objective, vht, g(2^-j)...
constexpr int kMaxHalvings = 1001;          // lambda = 2^-1 ... 2^-1001

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

__device__ __forceinline__ unsigned long long ballot(bool p) { return __ballot(p); }

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// ---------------------------------------------------------------------------
// kernel arguments
// ---------------------------------------------------------------------------

struct Graph {
  int N, E, ft0;                  // ft0 = first_thru_node - 1 (0-based)
  const int* fw_off;              // [N+1]
  const int* fw_dst;              // [E]  head of link k (CSR edge k == link k)
  const int* rv_off;              // [N+1] in-links of v
  const int* rv_src;              // [E]  tail, reverse order
  const int* rv_eid;              // [E]  link index, reverse order
  const int* tail;                // [E]  tail of link k
};

struct Labels {
  double* dist;                   // [N * P]   (flow during loading)
  int* pred;                      // [N * P]
  int* pend;                      // [N * P]   children left / -1 done
  long long P;                    // row stride (columns allocated)
  int Galloc;                     // group stride of stamp / items
  const int* col_src;             // [P] origin node of each column, -1 = padding
  const int* grp_var;             // [Galloc] variant of each group
  const unsigned char* var_on;    // [V] or null (all on)
  const double* rvw;              // [V * E] link costs in reverse-CSR order
};

__device__ __forceinline__ bool group_on(const Labels& L, int g) {
  return L.var_on == nullptr || L.var_on[L.grp_var[g]] != 0;
}

// Frontier bookkeeping: stamp[v * Galloc + g] holds the tag of the round in
// which item (v, g) must be processed; flags[r] != 0 iff round r has work.
// Writers only store (no atomics); a round's kernel finds its items with a
// dense scan compacted per block in LDS.  An item whose stamp is advanced to
// the next round before the scan reads it is simply processed one round
// later, which both worklists tolerate (labels only decrease; loading lanes
// carry the round from which they may run).
struct Frontier {
  int* stamp;     // [N * Galloc]
  int* flags;     // [rounds]
  unsigned long long* counters;   // [4] items, in-links scanned, lanes improved, out-links
};

// per-block scan of slots [blockIdx.x*kBlock, +kBlock) of the (v, g) space
// of groups [g0, g0+Gn); returns the number of items compacted into s_items
__device__ __forceinline__ int scan_slots(const Frontier& F, int N, int Galloc, int g0, int Gn,
                                          int tag, unsigned* s_items, int* s_n) {
  const long long slot = (long long)blockIdx.x * kBlock + threadIdx.x;
  const long long total = (long long)N * Gn;
  bool act = false;
  unsigned item = 0;
  if (slot < total) {
    const int v = (int)(slot / Gn);
    const int g = g0 + (int)(slot - (long long)v * Gn);
    item = (unsigned)v * (unsigned)Galloc + (unsigned)g;
    act = F.stamp[item] == tag;
  }
  const unsigned long long m = ballot(act);
  const int lane = lane_id();
  int base = 0;
  if (lane == 0 && m) base = atomicAdd(s_n, (int)__popcll(m));
  base = __shfl(base, 0);
  if (act) s_items[base + (int)__popcll(m & ((1ull << lane) - 1ull))] = item;
  __syncthreads();
  return *s_n;
}

// Mark the out-neighbours of v for group g in the next round (wave-wide).
__device__ __forceinline__ void mark_out(const Graph& G, const Frontier& F, int v, int g, int Galloc,
                                         int tag_next) {
  const int beg = G.fw_off[v], end = G.fw_off[v + 1];
  for (int e = beg + lane_id(); e < end; e += kWave)
    F.stamp[(size_t)G.fw_dst[e] * Galloc + g] = tag_next;
}

__device__ __forceinline__ void block_flush(const Frontier& F, int* s_any, int* flag_next,
                                            unsigned long long c0, unsigned long long c1,
                                            unsigned long long c2, unsigned long long c3,
                                            unsigned long long* s_cnt) {
  // c0..c3 are per-wave totals held by lane 0
  if (lane_id() == 0) {
    atomicAdd(&s_cnt[0], c0); atomicAdd(&s_cnt[1], c1);
    atomicAdd(&s_cnt[2], c2); atomicAdd(&s_cnt[3], c3);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (*s_any) *flag_next = 1;
    if (s_cnt[0]) {
      atomicAdd(&F.counters[0], s_cnt[0]); atomicAdd(&F.counters[1], s_cnt[1]);
      atomicAdd(&F.counters[2], s_cnt[2]); atomicAdd(&F.counters[3], s_cnt[3]);
    }
  }
}

// ---------------------------------------------------------------------------
// shortest paths
// ---------------------------------------------------------------------------

// dist = DBL_MAX, pred = -1 over the rows of groups [g0, g0+G).
__global__ __launch_bounds__(kBlock) void k_fill_labels(Graph G, Labels L, int g0, int Gn) {
  const long long waves = (long long)gridDim.x * kWavesPerBlock;
  const long long items = (long long)G.N * Gn;
  const int lane = lane_id();
  for (long long it = (long long)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; it < items;
       it += waves) {
    const int v = (int)(it / Gn);
    const int g = g0 + (int)(it - (long long)v * Gn);
    if (!group_on(L, g)) continue;
    const size_t idx = (size_t)v * L.P + (size_t)g * kWave + lane;
    L.dist[idx] = DBL_MAX;
    L.pred[idx] = -1;
  }
}

// Origins get label 0; their out-neighbours form round 0.
__global__ __launch_bounds__(kBlock) void k_sssp_seed(Graph G, Labels L, Frontier F, int g0,
                                                       int Gn, int tag0) {
  const int wave = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  if (wave >= Gn) return;
  const int g = g0 + wave;
  if (!group_on(L, g)) return;
  const int col = g * kWave + lane_id();
  const int src = L.col_src[col];
  bool any = false;
  if (src >= 0) {
    L.dist[(size_t)src * L.P + col] = 0.0;
    for (int e = G.fw_off[src]; e < G.fw_off[src + 1]; ++e) {
      F.stamp[(size_t)G.fw_dst[e] * L.Galloc + g] = tag0;
      any = true;
    }
  }
  if (ballot(any) && lane_id() == 0) F.flags[0] = 1;
}

// Round r: every marked (v, g) pulls min over in-links of dist[u] + w for its
// 64 origins (zones other than the lane's origin are not expanded).
__global__ __launch_bounds__(kBlock) void k_sssp_sweep(Graph G, Labels L, Frontier F, int g0,
                                                        int Gn, int r, int tag, int tag_next) {
  __shared__ unsigned s_items[kBlock];
  __shared__ int s_n, s_any;
  __shared__ unsigned long long s_cnt[4];
  if (threadIdx.x < 4) s_cnt[threadIdx.x] = 0;
  if (threadIdx.x == 0) { s_n = 0; s_any = 0; }
  __syncthreads();
  const int n = scan_slots(F, G.N, L.Galloc, g0, Gn, tag, s_items, &s_n);
  const int lane = lane_id();
  unsigned long long c_items = 0, c_scan = 0, c_upd = 0, c_out = 0;
  for (int it = threadIdx.x / kWave; it < n; it += kWavesPerBlock) {
    const unsigned item = s_items[it];
    const int v = uniform((int)(item / (unsigned)L.Galloc));
    const int g = uniform((int)(item - (unsigned)v * (unsigned)L.Galloc));
    const int col = g * kWave + lane;
    const int src = L.col_src[col];
    const double* __restrict__ w = L.rvw + (size_t)L.grp_var[g] * G.E;
    const size_t me = (size_t)v * L.P + col;
    const double cur = L.dist[me];
    double best = cur, arg_du = INFINITY;
    int arg = -1;
    const int kb = G.rv_off[v], ke = G.rv_off[v + 1];
    for (int k = kb; k < ke; ++k) {
      const int u = G.rv_src[k];
      if (u == v || (u < G.ft0 && u != src)) continue;   // zone: not a through node
      const double du = L.dist[(size_t)u * L.P + col];
      if (du < DBL_MAX) {
        const double cand = du + w[k];
        // equal-cost candidates: the tail with the smaller label wins (the
        // one a label-ordered search expands first)
        if (cand < best || (cand == best && du < arg_du)) {
          best = cand;
          arg = G.rv_eid[k];
          arg_du = du;
        }
      }
    }
    const bool improved = best < cur;
    if (improved) {
      L.dist[me] = best;
      L.pred[me] = arg;
    } else if (arg >= 0 && arg_du < cur && L.pred[me] != arg) {
      L.pred[me] = arg;     // same label, tail with a strictly smaller label
    }
    const unsigned long long m = ballot(improved);
    c_items += 1;
    c_scan += (unsigned long long)(ke - kb);
    c_upd += (unsigned long long)__popcll(m);
    if (ballot(improved && (v >= G.ft0 || v == src))) {
      mark_out(G, F, v, g, L.Galloc, tag_next);
      c_out += (unsigned long long)(G.fw_off[v + 1] - G.fw_off[v]);
      if (lane == 0) s_any = 1;
    }
  }
  block_flush(F, &s_any, &F.flags[r + 1], c_items, c_scan, c_upd, c_out, s_cnt);
}

// ---------------------------------------------------------------------------
// all-or-nothing loading on the predecessor trees
// ---------------------------------------------------------------------------

struct Loading {
  const double* odc;     // [Z * Pv] demand origin(col) -> zone row
  long long Pv;          // columns per variant
  int Z;
  double* ypart;         // [Galloc * E] per-group link volumes
  int* err;              // [3] flag, origin, dest (0-based)
};

// Lane state in pend[]: >= 0 children still to report; -1 done or not in the
// tree; -(L+2) ready from round L on (its subtree flow is complete once all
// launches before round L have finished).

// Dense pass: children count, initial node flow (= demand to this zone),
// no-path check, leaves marked for round 0.
__global__ __launch_bounds__(kBlock) void k_aon_init(Graph G, Labels L, Loading A, Frontier F,
                                                      int g0, int Gn, int tag0) {
  const long long waves = (long long)gridDim.x * kWavesPerBlock;
  const long long items = (long long)G.N * Gn;
  const int lane = lane_id();
  bool any = false;
  for (long long it = (long long)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; it < items;
       it += waves) {
    const int v = uniform((int)(it / Gn));
    const int g = uniform(g0 + (int)(it - (long long)v * Gn));
    if (!group_on(L, g)) continue;
    const int col = g * kWave + lane;
    const int src = L.col_src[col];
    const size_t me = (size_t)v * L.P + col;
    const int p = L.pred[me];
    int kids = 0;
    for (int e = G.fw_off[v]; e < G.fw_off[v + 1]; ++e) {
      const int x = G.fw_dst[e];
      kids += (L.pred[(size_t)x * L.P + col] == e) ? 1 : 0;
    }
    double f = 0.0;
    if (v < A.Z && src >= 0 && v != src) {
      const double d = A.odc[(size_t)v * A.Pv + (col % A.Pv)];
      if (d > 0.0) {
        f = d;
        if (p < 0 && atomicCAS(&A.err[0], 0, 1) == 0) {
          A.err[1] = src;
          A.err[2] = v;
        }
      }
    }
    L.dist[me] = f;
    L.pend[me] = (p < 0) ? -1 : (kids > 0 ? kids : -2);
    if (ballot(p >= 0 && kids == 0)) {
      if (lane == 0) F.stamp[(size_t)v * L.Galloc + g] = tag0;
      any = true;
    }
  }
  if (ballot(any) && lane == 0) F.flags[0] = 1;
}

// Round r: ready lanes of each marked (v, g) add their subtree demand to the
// in-link on their path, pass it to the tail node and release it.
__global__ __launch_bounds__(kBlock) void k_aon_level(Graph G, Labels L, Loading A, Frontier F,
                                                       int g0, int Gn, int r, int tag,
                                                       int tag_next) {
  __shared__ unsigned s_items[kBlock];
  __shared__ int s_n, s_any;
  __shared__ unsigned long long s_cnt[4];
  if (threadIdx.x < 4) s_cnt[threadIdx.x] = 0;
  if (threadIdx.x == 0) { s_n = 0; s_any = 0; }
  __syncthreads();
  const int n = scan_slots(F, G.N, L.Galloc, g0, Gn, tag, s_items, &s_n);
  const int lane = lane_id();
  unsigned long long c_items = 0, c_lanes = 0;
  for (int it = threadIdx.x / kWave; it < n; it += kWavesPerBlock) {
    const unsigned item = s_items[it];
    const int v = uniform((int)(item / (unsigned)L.Galloc));
    const int g = uniform((int)(item - (unsigned)v * (unsigned)L.Galloc));
    const int col = g * kWave + lane;
    const int src = L.col_src[col];
    const size_t me = (size_t)v * L.P + col;
    const int pe = L.pend[me];
    const int p = L.pred[me];
    // lanes released for this round or an earlier one (a lane released in
    // this round carries -(r+3) and waits for the next launch)
    const bool ready = (pe <= -2) && (-(pe + 2) <= r) && (p >= 0);
    const double f = ready ? L.dist[me] : 0.0;
    bool release = false;   // this lane's parent became ready
    if (ready) {
      const int parent = G.tail[p];
      L.pend[me] = -1;
      if (parent != src) {
        const size_t pi = (size_t)parent * L.P + col;
        if (f != 0.0) unsafeAtomicAdd(&L.dist[pi], f);
        if (atomicSub(&L.pend[pi], 1) == 1) {
          L.pend[pi] = -(r + 3);
          release = true;
        }
      }
    }
    c_items += 1;
    c_lanes += (unsigned long long)__popcll(ballot(ready));
    // per in-link: wave sum of the flow routed through it (fixed order)
    double* __restrict__ yp = A.ypart + (size_t)g * G.E;
    for (int k = G.rv_off[v]; k < G.rv_off[v + 1]; ++k) {
      const int eid = G.rv_eid[k];
      const bool mine = ready && p == eid;
      if (!ballot(mine)) continue;
      double s = mine ? f : 0.0;
      for (int off = kWave / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
      const bool rel = ballot(mine && release) != 0ull;
      if (lane == 0) {
        if (s != 0.0) yp[eid] += s;
        if (rel) {
          F.stamp[(size_t)G.rv_src[k] * L.Galloc + g] = tag_next;
          s_any = 1;
        }
      }
    }
  }
  block_flush(F, &s_any, &F.flags[r + 1], c_items, c_lanes, 0, 0, s_cnt);
}

// After the level rounds have drained every lane of a tree is done (-1).  A
// lane still waiting for children (>= 0) or released but never run (<= -2)
// lies on a predecessor cycle or hangs from one: flag it (err code 4).
__global__ __launch_bounds__(kBlock) void k_aon_check(Graph G, Labels L, Loading A, int g0, int Gn) {
  const long long n = (long long)G.N * Gn * kWave;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (long long)gridDim.x * kBlock) {
    const long long item = i / kWave;
    const int v = (int)(item / Gn);
    const int g = g0 + (int)(item - (long long)v * Gn);
    if (!group_on(L, g)) continue;
    const int col = g * kWave + (int)(i % kWave);
    if (L.col_src[col] < 0) continue;
    if (L.pend[(size_t)v * L.P + col] != -1 && atomicCAS(&A.err[0], 0, 4) == 0) {
      A.err[1] = L.col_src[col];
      A.err[2] = v;
    }
  }
}

// y[var][e] = sum over the variant's groups of ypart (fixed order); clears
// ypart for the next loading.
__global__ __launch_bounds__(kBlock) void k_aon_reduce(int E, int Gv, int v0, int Vn,
                                                        const unsigned char* var_on,
                                                        double* ypart, double* y) {
  const long long n = (long long)E * Vn;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (long long)gridDim.x * kBlock) {
    const int var = v0 + (int)(i / E);
    const int e = (int)(i - (long long)(var - v0) * E);
    if (var_on && !var_on[var]) continue;
    double s = 0.0;
    for (int j = 0; j < Gv; ++j) {
      double* p = ypart + ((size_t)var * Gv + j) * E + e;
      s += *p;
      *p = 0.0;
    }
    y[(size_t)var * E + e] = s;
  }
}

// ---------------------------------------------------------------------------
// one origin per workgroup, labels in LDS (networks up to ~13k nodes)
// ---------------------------------------------------------------------------
//
// For a metro-sized network one origin's labels (8 B/node) fit in a CU's
// 160 KB LDS, so a 1024-thread workgroup runs the whole origin: rounds of
// label-correcting relaxation (64-bit LDS atomicMin on the label bits --
// non-negative doubles order like their bit patterns; the nodes lowered in a
// round form the next round's frontier, marked by a bit of the label itself
// and listed in an LDS queue, kGroup lanes expanding each), then
// predecessor selection, then loading: each destination walks its tree path
// adding its demand to LDS node flows (FP64 LDS atomics), and every tree
// link with flow adds it to the HBM link volumes (FP64 atomics).  One launch
// covers every (variant, origin).
//
// Predecessor rule: among in-links u->v with fl(dist[u] + w) == dist[v]
// (u expandable) and dist[u] < dist[v], take the tail with the smallest
// label (the one a label-ordered search such as d'Esopo-Pape-LLL normally
// expands first), then the smallest tail id, then the first such link in
// link order -- the choice of the node-major sweeps too, and independent of
// thread timing.  A node whose tight tails all carry its own label
// (zero-cost links, or costs below half an ulp of the label) has none; such
// nodes join the tree level by level (attach_level_ties): each pass gives
// every one of them the smallest-id tight tail that was in the tree before
// the pass.  Along the chosen links the label decreases, or stays equal
// while the level decreases, so the tree is acyclic.  Where the shortest
// path is unique this is the reference's predecessor.

// Workgroup sizes of the LDS kernel; a size serves networks of up to
// kLdsPerThread nodes per thread: a wavefront of the predecessor phase takes
// that many slices of 64 nodes at most, whose bounds it keeps one a lane.
// 1024 by default; the schedule tuner may pick a smaller one where it fits.
constexpr int kLdsBlock = 1024;
constexpr int kLdsBlocks[] = {1024, 512, 256};
constexpr int kDefaultChase = 4;               // before tuning / shortest-path-only calls
constexpr int kLdsPerThread = 16;
constexpr int kLdsMaxNodes = kLdsPerThread * kLdsBlock;
#ifndef TAPGPU_LDS_QUEUE_MAX
#define TAPGPU_LDS_QUEUE_MAX 4096
#endif
constexpr int kLdsQueueMax = TAPGPU_LDS_QUEUE_MAX;   // frontier queue entries per round
constexpr int kGroup = 4;                            // lanes per expanded node (one link each)
constexpr int kGroupsPerWave = kWave / kGroup;
constexpr unsigned kNoPred = 0xFFFF;

// Mirrors of the graph and of each variant's costs that the LDS kernel
// reads, written wherever a cost is (store_cost).  Neither holds self-loops
// (they never lower a label and are never a tree link).
//  * Out-link records, 64 bytes per node: kRecLinks costs, then as many
//    16-bit heads; only links to through nodes (a zone's label is needed by
//    no other node, so it is taken from its in-links at the end).  A slot
//    without a link has the node itself as its head and an infinite cost.
//    kRecMore marks every head of a node with more than kGroup links,
//    kRecCsr those of one with more than kRecLinks, whose links are then
//    read from the CSR.
//  * In-links in slices of 64 nodes, slot-major (SELL): row s of a slice
//    holds the s-th in-link of its 64 nodes, a word of link id and tail and
//    the cost.  Only links between through nodes: those of zones are looked
//    at by themselves.  An entry without a link has the node itself as its
//    tail and an infinite cost.
//    At most kSellWidth rows a slice; a node with more in-links is looked at
//    after the slices, from the CSR.
constexpr int kRecDoubles = 8, kRecLinks = 6;
constexpr unsigned kRecNode = 0x3FFF, kRecMore = 0x4000, kRecCsr = 0x8000;
static_assert(kRecLinks * 10 <= 64 && kRecLinks <= 2 * kGroup, "an out-link record is 64 bytes");
static_assert(kLdsMaxNodes <= (int)kRecNode + 1, "heads are 14-bit");
constexpr int kSellWidth = 16;
constexpr int kSellFetch = 4;        // rows of a slice loaded ahead
constexpr unsigned kSellNone = 0xFFFF0000u;

// A barrier in a loop whose LDS writes of one pass are read in the next.  The
// wait is written out: the compiler drops its own where the writes reach the
// barrier over the loop's back edge only, and another wavefront's read can
// then overtake a write (seen with 512 threads: one label in 10^7 stayed
// too high).
__device__ __forceinline__ void loop_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();
}

// LDS atomicAdd by one lane.  The address is made to look divergent: for a
// uniform one the compiler adds a wave-wide reduction around the atomic.
__device__ __forceinline__ int lds_add(int* p, int n) {
  int z = 0;
  asm("" : "+v"(z));
  return atomicAdd(p + z, n);
}

struct OriginArgs {
  int N, E, ft0, Z;
  const int *fw_off, *fw_dst, *rv_off, *rv_src, *rv_eid, *tail;
  const double* fww;                 // [V * E] forward costs (INF: absent)
  const double* rvw;                 // [V * E] reverse-order costs
  const double* rec;                 // [V][N] out-link records (LDS kernel)
  const double* sellw;               // [V][sell_n] sliced in-link costs
  const unsigned* sell_id;           // [sell_n] link id << 16 | tail
  const int* sell_ptr;               // [ceil(N/64) + 1] first entry of each slice
  const void* hrec;                  // [variants of the launch][hrec_n] out-link records (labels-in-HBM kernel)
  const struct HbmRecOf* hrec_of;    // [hrec_n]
  int hrec_n;
  const uint2* hsell_id;             // [hsell_n] tail, link id
  const double* hsellw;              // [variants of the launch][hsell_n]
  const int* hsell_ptr;
  long long hsell_n;
  const int *place, *node;           // its numbering: node -> place, place -> node
  long long sell_n;
  const long long* od_start;         // [Z + 1]
  const int* od_dest;                // 0-based zone
  const double* od_val;
  const unsigned char* var_on;       // [V] or null
  int chase;                         // expansions a thread chains per round
  int qcap;                          // LDS frontier queue entries per round (0: bitmap scan only)
  int hqcap;                         // labels-in-HBM kernel: entries of a queue
  double delta;                      // labels-in-HBM kernel: bucket width (< 0: the first of one that adapts)
  int z0, zn;                        // labels-in-HBM kernel: origins [z0, z0 + zn) of each variant
  double* y;                         // [V * E], zeroed by the caller
  int* err;                          // [3]
  unsigned long long* counters;      // [16] expansions, links scanned, updates,
                                     //     relax rounds, longest loading walk,
                                     //     tree links loaded, walk steps, -,
                                     //     wall-clock ticks of relaxation,
                                     //     predecessors, loading; [12] rounds
                                     //     that overflowed the LDS queue
  // block x handles origin src_list[x] (shortest-path-only mode: start
  // nodes; LDS loadings: origins longest first)
  const int* src_list;
  int* work;                         // [Z] relaxation rounds per origin, recorded when non-null
  // labels-in-HBM loadings: items taken from a counter (null: block-strided),
  // origin-major in `order` (origins by decreasing rounds) when non-null
  int* next;
  const int* order;
  int vn;                            // variants of the launch (with order)
  double* out_dist;                  // [(N) * ld] node-major, row v = node v+1
  int* out_pred;
  long long ld;
  // labels-in-HBM kernel: per-block scratch rows of N entries
  unsigned long long* h_dist;        // labels, then flows
  int* h_pred;                       // tree link
  int* h_ptail;                      // its tail
};

__device__ __forceinline__ double as_d(unsigned long long b) { return __longlong_as_double((long long)b); }

// wavefront-wide sum / max (every lane of the wavefront active), so that
// per-thread counters reach a workgroup total with one LDS atomic per wave
__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long x) {
  for (int o = kWave / 2; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}
__device__ __forceinline__ int wave_max_i32(int x) {
  for (int o = kWave / 2; o > 0; o >>= 1) x = max(x, __shfl_xor(x, o));
  return x;
}
__device__ __forceinline__ unsigned long long as_b(double d) { return (unsigned long long)__double_as_longlong(d); }

// LDS layout (bytes): labels 8N (flows while loading) | two bitmaps 2*8W |
// pred 2A | ptail 2A | two frontier queues 2*2(Q+2), with W = ceil(N/64),
// A = N+1 rounded up to 4, Q = queue entries (entry Q takes what overflows).
size_t origin_lds_bytes(int N, int qcap) {
  const size_t W = (size_t)(N + 63) / 64, A = (size_t)((N + 1 + 3) & ~3);
  return 8ull * N + 16ull * W + 4ull * A + 4ull * ((size_t)qcap + 2);
}

// Second step of the predecessor rule: the nodes flagged in `pending` have
// no tight tail with a smaller label.  Each pass gives every pending node
// the smallest-id tight tail with its own label that was in the tree before
// the pass (not pending), and clears the flags after a barrier, so a pass's
// result does not depend on thread timing.  Every pending node hangs from a
// tree node through such links (its label came along them), so each pass
// attaches at least one node; false if a pass attaches none.  All threads
// of the workgroup call it; label(v) reads a label, set_pred(v, link, tail)
// records a choice.
template <int kThreads, class Label, class SetPred>
__device__ bool attach_level_ties(const OriginArgs& A, const double* __restrict__ rw, int src,
                                  unsigned long long* pending, unsigned long long* added,
                                  int* s_left, int* s_added, Label label, SetPred set_pred) {
  const int N = A.N, W = (N + 63) >> 6, tid = threadIdx.x;
  for (int w = tid; w < W; w += kThreads) added[w] = 0;
  for (;;) {
    if (tid == 0) { *s_left = 0; *s_added = 0; }
    __syncthreads();
    for (int v = tid; v < N; v += kThreads) {
      if (!((pending[v >> 6] >> (v & 63)) & 1ull)) continue;
      const unsigned long long dv = label(v);
      int bu = -1, be = -1;
      for (int k = A.rv_off[v]; k < A.rv_off[v + 1]; ++k) {
        const int u = A.rv_src[k];
        if (u == v || (u < A.ft0 && u != src)) continue;
        if ((pending[u >> 6] >> (u & 63)) & 1ull) continue;       // not in the tree yet
        const unsigned long long du = label(u);
        if (du != dv || as_b(as_d(du) + rw[k]) != dv) continue;
        if (bu < 0 || u < bu) { bu = u; be = A.rv_eid[k]; }
      }
      if (be >= 0) {
        set_pred(v, be, bu);
        atomicOr(&added[v >> 6], 1ull << (v & 63));
        atomicAdd(s_added, 1);
      } else {
        atomicAdd(s_left, 1);
      }
    }
    __syncthreads();
    const int left = *s_left, got = *s_added;
    for (int w = tid; w < W; w += kThreads) { pending[w] &= ~added[w]; added[w] = 0; }
    if (left == 0 || got == 0) return left == 0;
    __syncthreads();
  }
}

template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_origin_lds(OriginArgs A, int load) {
  extern __shared__ unsigned long long sm[];
  constexpr int kWaves = BLOCK / kWave;
  const int N = A.N;
  const int W = (N + 63) >> 6;
  const int Al = (N + 1 + 3) & ~3;
  unsigned long long* key = sm;                                    // [N] label << 1 | listed
  double* flow = (double*)sm;                                      //     (flows while loading)
  unsigned long long* bmB = key + N;                               // 2 x [W] (attach_level_ties)
  unsigned long long* bmC = bmB + W;
  unsigned short* pred = (unsigned short*)(bmC + W);               // [N]
  unsigned short* ptail = pred + Al;                               // [N]
  unsigned short* queue0 = ptail + Al;                             // 2 x [qcap + 2]
  __shared__ int s_qn[3];
  __shared__ unsigned long long s_cnt[8];

  const int var = blockIdx.y;
  if (A.var_on && !A.var_on[var]) return;
  const int src = A.src_list ? A.src_list[blockIdx.x] : (int)blockIdx.x;
  const int tid = threadIdx.x;
  const int wave = uniform(tid / kWave);
  const int lane = tid & (kWave - 1);
  const double* __restrict__ fw = A.fww + (size_t)var * A.E;
  const double* __restrict__ rw = A.rvw + (size_t)var * A.E;
  const double* __restrict__ rec = A.rec + (size_t)var * N * kRecDoubles;
  const double* __restrict__ sellw = A.sellw + (size_t)var * A.sell_n;
  const unsigned long long kMax = as_b(DBL_MAX);

  for (int v = tid; v < N; v += BLOCK) key[v] = kMax << 1;
  for (int w = tid; w < 2 * W; w += BLOCK) bmB[w] = 0;
  if (tid < 3) s_qn[tid] = tid == 0 ? 1 : 0;
  if (tid < 8) s_cnt[tid] = 0;
  __syncthreads();
  if (tid == 0) {
    key[src] = 1ull;                      // +0.0, listed
    queue0[0] = (unsigned short)src;
  }
  __syncthreads();

  unsigned n_exp = 0, n_scan = 0, n_upd = 0;
  const long long clk0 = wall_clock64();
  // ---- label-correcting rounds, one barrier each.  Round r expands the
  //      nodes lowered in round r-1.  Normally they are listed in a queue
  //      (count s_qn[cnt]) and each gets a group of kGroup lanes of one
  //      wavefront, one out-link per lane, whose costs and heads are one
  //      64-byte record.  When more nodes were lowered than the queue holds,
  //      the round looks for their flags among the labels instead, a lane
  //      expanding each (and chaining up to A.chase further expansions of
  //      nodes it lowers itself).
  //      A label is kept as (bits << 1) | listed: labels are non-negative,
  //      so the sign bit is free and the keys order like the labels.  An
  //      expansion reads the label and clears the flag in one atomic, and a
  //      lane that lowers a label sets it in the same atomic min: the old
  //      key it gets back tells whether the node waits in a queue already.
  //      So one LDS atomic lowers and deduplicates, and a node lowered again
  //      before its expansion is not listed twice.  Labels are the same
  //      least fixed point for any such order.
  //      A round is a chain of five latencies (queue entry, record, label
  //      atomic, append, barrier) and of the instructions between them, and
  //      4 wavefronts share a SIMD's issue slots, so what bounds it is the
  //      instructions of the few wavefronts with nodes to expand (~73 nodes
  //      a round on metro: 5 of 16).  Hence links to zones are left out
  //      (they would need a 5th and 6th lane for one node in five), empty
  //      record slots relax like links instead of being masked, control flow
  //      is wave-uniform, and the lane that lists a node starts a load of
  //      its record, which has the line in the CU's L1 before the next
  //      round asks for it.  Taken branches cost as much as an LDS read, so
  //      the common round is laid out straight.  Measured on metro (1,000
  //      origins, 146 rounds; us per workgroup): 69, and 143 with 6 lanes
  //      per node, CSR reads, a bitmap atomic beside the label's and
  //      divergent loop control. ----
  const int qcap = A.qcap, ft0 = A.ft0;
  int c_now = 0, c_next = 1, c_free = 2;   // s_qn slots, in turn: written, cleared, idle
  const int qstride = qcap + 2;
  int qoff = 0;                            // the queue written last
  int pf_node = -1;                        // listed by this lane in the last round
  unsigned pf_sink = 0;
  // relaxes a link to the through node v at label bits cb and, if this lane
  // lowered v and `want`, lists it unless listed already; returns whether
  // this lane lowered v (without `want` the lane then expands v itself,
  // which clears the flag set here)
  auto relax = [&](unsigned long long cb, int v, bool want) {
    // no pre-read of key[v]: one LDS round trip, and measured faster
    const unsigned long long kb = (cb << 1) | 1ull;
    const unsigned long long old = atomicMin(&key[v], kb);
    const bool low = kb < old;
    n_upd += low;
    if (low && want && !(old & 1ull)) {
      // one LDS atomic for the wavefront's appends
      const unsigned long long m = __builtin_amdgcn_read_exec();
      const int rank = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      int b0 = 0;
      if (rank == 0) b0 = lds_add(&s_qn[c_now], __popcll(m));
      queue0[qoff + min(uniform(b0) + rank, qcap)] = (unsigned short)v;
      pf_node = v;
    }
    return low;
  };
  // the label of a node about to be expanded; clears its flag
  auto take = [&](int u) { return as_d(atomicAnd(&key[u], ~1ull) >> 1); };
  const char* recb = (const char*)rec;
  const unsigned g = lane % kGroup;
  // expands a listed node with the kGroup lanes of a group
  auto expand = [&](int u) {
    const unsigned at = (unsigned)u * 64u;
    const double w = *(const double*)(recb + (at + g * 8u));
    const unsigned h = *(const unsigned short*)(recb + (at + 8u * kRecLinks + g * 2u));
    const double du = take(u);
    relax(as_b(du + w), (int)(h & kRecNode), true);
    n_scan += (int)(h & kRecNode) != u;
    if (__builtin_expect(h & kRecMore, 0)) {          // more out-links than lanes
      if (h & kRecCsr) {                              // ... than the record holds
        // (the first kGroup links of the CSR are among those just relaxed)
        const int ee = A.fw_off[u + 1] - kGroup;
        for (int e0 = A.fw_off[u] + (int)g; e0 < ee; e0 += kGroup) {
          const int e = e0 + kGroup;
          const int v = A.fw_dst[e];
          if (v < ft0) continue;
          ++n_scan;
          relax(as_b(du + fw[e]), v, true);
        }
      } else if (g < kRecLinks - kGroup) {
        const double w2 = *(const double*)(recb + (at + (g + kGroup) * 8u));
        const unsigned h2 = *(const unsigned short*)(recb + (at + 8u * kRecLinks + (g + kGroup) * 2u));
        n_scan += (int)(h2 & kRecNode) != u;
        relax(as_b(du + w2), (int)(h2 & kRecNode), true);
      }
    }
  };
  constexpr int kPass = kWaves * kGroupsPerWave;       // nodes expanded at once
  const int j0 = wave * kGroupsPerWave + lane / kGroup;
  const int jq = min(j0, qcap);
  const int pass = min(kPass, qcap);
  int r = 0, qn;
  unsigned n_listed = 0, n_scans = 0;      // (wave-uniform)
  for (;;) {
    unsigned pf = 0;
    if (pf_node >= 0)
      pf = __hip_atomic_load((const unsigned*)(recb + (unsigned)pf_node * 64u), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WAVEFRONT);
    pf_node = -1;
    loop_barrier();
    int u0 = queue0[qoff + jq], n0 = s_qn[c_now];
    asm volatile("" : "+v"(u0), "+v"(n0));              // (both read before either is used)
    qn = uniform(n0);
    if (qn == 0 || r > N + 8) break;
    ++r;
    qoff = qstride - qoff;
    // (this slot was read before the barrier and is written after the next)
    s_qn[c_free] = 0;
    { const int t = c_now; c_now = c_next; c_next = c_free; c_free = t; }
    if (__builtin_expect(qn <= pass, 1)) {
      if (j0 < qn) expand(u0);
      n_listed += (unsigned)qn;
    } else if (qn <= qcap) {
      const unsigned short* qr = queue0 + (qstride - qoff);
      for (int j = j0; j < qn; j += kPass) expand(qr[j]);
      n_listed += (unsigned)qn;
    } else {
      ++n_scans;
      for (int v0 = tid; v0 < N; v0 += BLOCK) {
        if (!(__hip_atomic_load(&key[v0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) & 1ull)) continue;
        int x = v0;
        for (int hops = 0;; ++hops) {
          const double du = take(x);
          const int eb = A.fw_off[x], ee = A.fw_off[x + 1];
          ++n_exp;
          int next = -1;
          for (int e = eb; e < ee; ++e) {
            const int v = A.fw_dst[e];
            if (v < ft0) continue;
            ++n_scan;
            // the first node this lane lowers is chained, not listed
            const bool chain = next < 0 && hops < A.chase;
            if (relax(as_b(du + fw[e]), v, !chain) && chain) next = v;
          }
          if (next < 0) break;
          x = next;
        }
      }
    }
    pf_sink ^= pf;
  }
  if (tid == 0) n_exp += n_listed;
  if (n_scans && tid == 0 && A.counters) atomicAdd(&A.counters[12], (unsigned long long)n_scans);
  if (qn) {                     // only possible with negative costs
    if (tid == 0 && atomicCAS(&A.err[0], 0, 2) == 0) { A.err[1] = src; A.err[2] = 0; }
    return;
  }
  if (N < 0) s_cnt[7] = pf_sink;            // (never: keeps the loads)
  const int relax_rounds = r;
  const long long clk1 = wall_clock64();
  if (A.work && tid == 0 && blockIdx.y == 0) A.work[src] = relax_rounds;

  // ---- predecessor links (label, then tail id; see above), every flag
  //      being clear now.  Through nodes first.  A wavefront takes slices of
  //      64 consecutive nodes; row s of a slice (the s-th in-links) is
  //      contiguous in the sliced copy, so every line is read once, and the
  //      first kSellFetch rows of the next slice are on their way while a
  //      slice is processed.  Zones other than the origin still have no
  //      label, so no test keeps them from being tails, and the links of an
  //      origin that is a zone (which are in no slice) are looked at before
  //      the slices: its label 0 is the smallest there is, and its id too,
  //      so such a link wins where it is tight.  Then the zones, whose
  //      labels are the minimum over their in-links.  Bound by instruction
  //      issue (about 15 a row; 156 slices of 4 rows on metro): 14.5 us per
  //      workgroup, 25.6 with a thread reading its node's in-links from the
  //      CSR. ----
  __shared__ int s_level_ties;
  if (tid == 0) s_level_ties = 0;
  // this thread's first destination, on its way while the links are chosen
  long long od0 = 0, od1 = 0;
  int d0 = 0;
  double f0 = 0.0;
  if (load) {
    od0 = A.od_start[src];
    od1 = A.od_start[src + 1];
    if (od0 + tid < od1) { d0 = A.od_dest[od0 + tid]; f0 = A.od_val[od0 + tid]; }
  }
  if (src < ft0)
    for (int e = A.fw_off[src] + tid; e < A.fw_off[src + 1]; e += BLOCK) {
      const int v = A.fw_dst[e];
      const unsigned long long wb = as_b(0.0 + fw[e]);
      if (v < ft0 || wb == 0ull || key[v] >> 1 != wb || wb >= kMax) continue;
      bool first = true;                     // of equal parallel links
      for (int k = A.fw_off[src]; k < e; ++k) first = first && !(A.fw_dst[k] == v && fw[k] == fw[e]);
      if (!first) continue;
      pred[v] = (unsigned short)e;
      ptail[v] = (unsigned short)src;
      atomicOr(&bmC[v >> 6], 1ull << (v & 63));        // chosen
    }
  __syncthreads();
  // records v's choice `id` (link and tail; kSellNone's link: none)
  auto choose = [&](int v, unsigned id, unsigned long long dk) {
    const bool none = id >= kSellNone, reached = v != src && dk != kMax << 1;
    pred[v] = (unsigned short)(id >> 16);
    ptail[v] = (unsigned short)id;
    // reached, not the origin, and no tight tail with a smaller label:
    // every tight tail has this label
    const bool level_tie = none && reached;
    if (level_tie) {
      atomicOr(&bmB[v >> 6], 1ull << (v & 63));
      s_level_ties = 1;
    }
    if (A.out_dist) {
      const size_t o = (size_t)v * A.ld + blockIdx.x;
      A.out_dist[o] = as_d(dk >> 1);
      if (!level_tie) A.out_pred[o] = none ? -1 : (int)(id >> 16);
    }
  };
  {
    constexpr int kSlices = kLdsPerThread;             // slices per wavefront, at most
    const int sl0 = ft0 / kWave + wave;                // its first
    int first = 0, last = 0;                           // lane k: entries of the k-th slice
    if (lane < kSlices && sl0 + lane * kWaves < W) {
      first = A.sell_ptr[sl0 + lane * kWaves];
      last = A.sell_ptr[sl0 + lane * kWaves + 1];
    }
    struct Rows { unsigned id[kSellFetch]; double w[kSellFetch]; };
    auto rows_of = [&](int k) {
      return (__builtin_amdgcn_readlane(last, k) - __builtin_amdgcn_readlane(first, k)) / kWave;
    };
    auto fetch = [&](int k, Rows& R) {
      // (no load is left out: one under a branch waits for those before it)
      const int rows = rows_of(k);
      const unsigned at = (unsigned)((rows ? __builtin_amdgcn_readlane(first, k) : 0) + lane);
#pragma unroll
      for (int i = 0; i < kSellFetch; ++i) {
        const unsigned a = at + (unsigned)(max(min(i, rows - 1), 0) * kWave);
        R.id[i] = A.sell_id[a];
        R.w[i] = sellw[a];
      }
    };
    auto select = [&](int k, const Rows& R) {
      const int sl = sl0 + k * kWaves, v = sl * kWave + lane, rows = rows_of(k);
      const unsigned long long dk = v < N ? key[v] : kMax << 1, dv = dk >> 1;
      // starting from (dv, tail 0) only tails with a smaller label can win
      unsigned best = kSellNone;
      unsigned long long best_du = dk;
      auto offer = [&](unsigned id, double w) {
        const unsigned u = id & 0xFFFFu;
        const unsigned long long du = key[u];
        const bool tight = as_b(as_d(du >> 1) + w) == dv;
        if (__ballot(tight && du == best_du) && tight && du == best_du && u < (best & 0xFFFFu)) best = id;
        if (tight && du < best_du) { best = id; best_du = du; }
      };
#pragma unroll
      for (int i = 0; i < kSellFetch; ++i)
        if (i < rows) offer(R.id[i], R.w[i]);
      if (rows > kSellFetch) {
        const unsigned at = (unsigned)(__builtin_amdgcn_readlane(first, k) + lane);
        for (int i = kSellFetch; i < rows; ++i) offer(A.sell_id[at + i * kWave], sellw[at + i * kWave]);
      }
      const bool chosen = (bmC[min(sl, W - 1)] >> lane) & 1ull;
      if (v < N && v >= ft0) {
        if (dk == kMax << 1 || v == src) best = kSellNone | 0xFFFFu;
        if (!chosen)
          choose(v, best, dk);
        else if (A.out_dist)
          choose(v, (unsigned)pred[v] << 16 | (unsigned)src, dk);
      }
    };
    const int n = sl0 < W ? (W - sl0 + kWaves - 1) / kWaves : 0;
    Rows Ra, Rb;
    if (n > 0) fetch(0, Ra);
    for (int k = 0; k < n; k += 2) {
      if (k + 1 < n) fetch(k + 1, Rb);
      select(k, Ra);
      if (k + 2 < n) fetch(k + 2, Ra);
      if (k + 1 < n) select(k + 1, Rb);
    }
    // Nodes with more in-links than a slice has rows are looked at again, each
    // by the whole wavefront (100 origins on a star of 10,000 links: 4.3 ms a
    // loading, 6.1 with a lane reading them all in the loop above).
    for (unsigned long long ks = __ballot(last - first >= kSellWidth * kWave); ks; ks &= ks - 1) {
      const int sl = sl0 + (__ffsll((long long)ks) - 1) * kWaves, v = sl * kWave + lane;
      const bool more = v < N && v >= ft0 && v != src && key[v] != kMax << 1 &&
                        !((bmC[sl] >> lane) & 1ull) && A.rv_off[v + 1] - A.rv_off[v] > kSellWidth;
      for (unsigned long long m = __ballot(more); m; m &= m - 1) {
        const int l = __ffsll((long long)m) - 1, x = sl * kWave + l;
        const unsigned long long dx = key[x];
        unsigned long long du = dx, id = ~0ull;        // the lane's choice: label, then tail, then link
        for (int e = A.rv_off[x] + lane; e < A.rv_off[x + 1]; e += kWave) {
          const int u = A.rv_src[e];
          const unsigned long long d = key[u], i = (unsigned long long)u << 32 | (unsigned)A.rv_eid[e];
          if (u < ft0 || d >= dx || as_b(as_d(d >> 1) + rw[e]) != dx >> 1) continue;
          if (d < du || (d == du && i < id)) { du = d; id = i; }
        }
        for (int o = kWave / 2; o > 0; o >>= 1) {
          const unsigned long long d = __shfl_xor(du, o), i = __shfl_xor(id, o);
          if (d < du || (d == du && i < id)) { du = d; id = i; }
        }
        if (lane == l && id != ~0ull) {
          atomicAnd(&bmB[x >> 6], ~(1ull << (x & 63)));  // (the first rows may have had none)
          choose(x, (unsigned)(id >> 32) | (unsigned)id << 16, dx);
        }
      }
    }
  }
  if (ft0 > 0) {
    __syncthreads();                        // the through nodes' selections read no zone label
    for (int v = tid; v < ft0 && v < N; v += BLOCK) {
      unsigned id = kSellNone | 0xFFFFu;
      unsigned long long dk = key[v];
      if (v != src) {
        auto tails = [&](auto&& f) {        // f(tail, link, label bits through it)
          for (int e = A.rv_off[v]; e < A.rv_off[v + 1]; ++e) {
            const int u = A.rv_src[e];
            if (u == v || (u < ft0 && u != src)) continue;
            const unsigned long long du = key[u];
            if (du != kMax << 1) f(u, A.rv_eid[e], du, as_b(as_d(du >> 1) + rw[e]) << 1);
          }
        };
        tails([&](int, int, unsigned long long, unsigned long long c) { dk = min(dk, c); });
        unsigned long long best_du = dk;
        tails([&](int u, int e, unsigned long long du, unsigned long long c) {
          if (c == dk && (du < best_du || (du == best_du && (unsigned)u < (id & 0xFFFFu) && id < kSellNone))) {
            best_du = du;
            id = (unsigned)u | (unsigned)e << 16;
          }
        });
        if (dk == kMax << 1) id = kSellNone | 0xFFFFu;
        key[v] = dk;
      }
      choose(v, id, dk);
    }
  }
  __syncthreads();
  const long long clk2 = wall_clock64();
  if (s_level_ties) {
    __shared__ int s_left, s_added;
    const bool ok = attach_level_ties<BLOCK>(
        A, rw, src, bmB, bmC, &s_left, &s_added, [&](int v) { return key[v] >> 1; },
        [&](int v, int e, int u) {
          pred[v] = (unsigned short)e;
          ptail[v] = (unsigned short)u;
          if (A.out_dist) A.out_pred[(size_t)v * A.ld + blockIdx.x] = e;
        });
    if (!ok && tid == 0 && atomicCAS(&A.err[0], 0, 3) == 0) { A.err[1] = src; A.err[2] = 0; }
  }
  auto flush_counts = [&]() {
    const unsigned long long a = wave_sum_u64(n_exp), b = wave_sum_u64(n_scan), c = wave_sum_u64(n_upd);
    if (lane == 0) { atomicAdd(&s_cnt[0], a); atomicAdd(&s_cnt[1], b); atomicAdd(&s_cnt[2], c); }
  };
  if (!load) {
    if (A.counters) {
      flush_counts();
      __syncthreads();
      if (tid == 0) {
        atomicAdd(&A.counters[0], s_cnt[0]); atomicAdd(&A.counters[1], s_cnt[1]);
        atomicAdd(&A.counters[2], s_cnt[2]); atomicAdd(&A.counters[3], (unsigned long long)relax_rounds);
      }
    }
    return;
  }

  // ---- all-or-nothing loading: every destination with demand walks its
  //      tree path to the origin, adding its demand to each node's flow
  //      (the flow on the node's tree in-link); no rounds, no barriers.
  //      Integer demands make every partial sum exact, so the order of the
  //      LDS atomics does not matter. ----
  __syncthreads();                 // every label read is done
  for (int v = tid; v < N; v += BLOCK) flow[v] = 0.0;
  __shared__ unsigned long long s_steps;
  __shared__ int s_maxlen, s_loaded;
  if (tid == 0) { s_steps = 0; s_maxlen = 0; s_loaded = 0; ptail[src] = (unsigned short)src; }
  __syncthreads();
  unsigned long long steps = 0;
  int maxlen = 0;
  for (long long i = od0 + tid; i < od1; i += BLOCK) {
    const int d = i == od0 + tid ? d0 : A.od_dest[i];
    const double f = i == od0 + tid ? f0 : A.od_val[i];
    if (d == src || !(f > 0.0)) continue;
    if (pred[d] == kNoPred) {
      if (atomicCAS(&A.err[0], 0, 1) == 0) { A.err[1] = src; A.err[2] = d; }
      continue;
    }
    // The longest walk (one LDS read a step) sets the time, so four steps
    // go without a branch: a walk that has arrived stays at the origin, its
    // own tail here, and adds zero to a node of its lane's own (metro: 15 us
    // per workgroup for the loading, 22.9 with a branch a step).
    int v = d, len = 0;
    const int idle = min(lane, N - 1);
    do {
      if (len > N) {        // a predecessor cycle
        if (atomicCAS(&A.err[0], 0, 3) == 0) { A.err[1] = src; A.err[2] = 0; }
        break;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int next = ptail[v];
        const bool on = v != src;
        atomicAdd(&flow[on ? v : idle], on ? f : 0.0);
        len += on;
        v = next;
      }
    } while (v != src);
    steps += (unsigned long long)len;
    maxlen = max(maxlen, len);
  }
  __syncthreads();
  double* __restrict__ yv = A.y + (size_t)var * A.E;
  int loaded = 0;
  for (int v = tid; v < N; v += BLOCK) {
    const double f = flow[v];
    if (f != 0.0 && pred[v] != kNoPred) {
      unsafeAtomicAdd(&yv[pred[v]], f);
      ++loaded;
    }
  }
  if (A.counters) {
    flush_counts();
    steps = wave_sum_u64(steps);
    maxlen = wave_max_i32(maxlen);
    const unsigned long long ld = wave_sum_u64((unsigned long long)loaded);
    if (lane == 0) {
      atomicAdd(&s_steps, steps);
      atomicMax(&s_maxlen, maxlen);
      atomicAdd(&s_loaded, (int)ld);
    }
  }
  __syncthreads();
  if (tid == 0 && A.counters) {
    atomicAdd(&A.counters[0], s_cnt[0]); atomicAdd(&A.counters[1], s_cnt[1]);
    atomicAdd(&A.counters[2], s_cnt[2]); atomicAdd(&A.counters[3], (unsigned long long)relax_rounds);
    atomicAdd(&A.counters[4], (unsigned long long)s_maxlen);
    atomicAdd(&A.counters[5], (unsigned long long)s_loaded);
    atomicAdd(&A.counters[6], s_steps);
    const long long clk3 = wall_clock64();
    atomicAdd(&A.counters[8], (unsigned long long)(clk1 - clk0));
    atomicAdd(&A.counters[9], (unsigned long long)(clk2 - clk1));
    atomicAdd(&A.counters[10], (unsigned long long)(clk3 - clk2));
  }
}


// ---------------------------------------------------------------------------
// one origin per workgroup, labels in HBM (networks of any size)
// ---------------------------------------------------------------------------
//
// The same three phases as k_origin_lds for networks whose labels do not fit
// LDS: only a node bitmap (8 x ceil(N/64) bytes) and the frontier
// queues live in LDS; labels, predecessors and flows are a per-workgroup
// scratch row in HBM (L2 / infinity cache resident while the workgroup
// runs).  A persistent grid loops over (origin, variant) items.  A row is
// private to its workgroup, whose waves share one CU, so every scratch
// access is a workgroup-scope atomic: loads skip the CU's L1 and read the
// XCD's L2, and the barrier closing a round orders them.  (Device-scope
// accesses would have to be coherent across the XCDs' L2s and cost an L2
// writeback and invalidation per round.)  Relaxation within a round may read
// a label another thread is lowering; the lowered node is queued for the
// next round, so the fixed point is the same as with strict rounds.

#ifndef TAPGPU_HBM_BLOCK
#define TAPGPU_HBM_BLOCK 512
#endif
constexpr int kHbmBlock = TAPGPU_HBM_BLOCK;    // 512: 2 workgroups per CU, each with room for queues
#ifndef TAPGPU_HBM_PER_CU
#define TAPGPU_HBM_PER_CU (1024 / TAPGPU_HBM_BLOCK)
#endif
constexpr int kHbmPerCu = TAPGPU_HBM_PER_CU;    // workgroups sharing a CU's LDS (registers: <= 128 VGPRs)
constexpr int kHbmQueueMax = 4096;              // entries of a frontier queue

__global__ void k_zero_i32(int* p) { *p = 0; }

// LDS of the labels-in-HBM kernel: a bitmap 8W | the table, two near queues
// and a far queue of twice their size, of (label 8 B, node 4 B) entries; the
// predecessors' second bitmap takes the place of these.
constexpr int kHbmQueueMin = 64;                // entries there is room for at least (fewer can be asked for)
constexpr size_t kHbmQueueBytes = 48;           // per entry of the queue size
constexpr int kHbmCand = 3;                     // links per lane of an expanded node
constexpr int kHbmRedo = 64;                    // places kept for entries to be followed up again
constexpr int kHbmFew = 32;                     // entries brought near at once, below which the far queue is weeded
constexpr int kHbmSlots = 1024;                 // of the table that settles which lane lowers a label
size_t origin_hbm_lds_bytes(int N, int hqcap) {
  const size_t bitmap = 8ull * (size_t)((N + 63) / 64);
  return bitmap + std::max<size_t>(bitmap, 12 * kHbmSlots + kHbmQueueBytes * (size_t)hqcap);
}

// Mirrors of the graph and of each variant's costs that the labels-in-HBM
// kernel reads, written before each of its launches (a pass over the links:
// 20 us on regional, against 40 ms): the LDS kernel's records and sliced
// in-links with 32-bit nodes and links.  A record is one 64-byte line of
// kHrecLinks links to through nodes, self-loops left out; a node with more
// of them has further records behind those of the nodes, so that its links
// come in lines too: a search takes them as entries of their own, a round
// later.  Read from the CSR instead, two links at a time and past the table
// that settles which label is stored, such nodes held up their wavefronts:
// a grid of 22,500 nodes with 12 through links each, 200 origins, 3
// iterations 13.2 ms, and 9.5 so; a star of 20,000 nodes, 100 origins, one
// loading 44 and 11; regional, where one node in a thousand has more than 5,
// 39.2 and 36.7 ms a loading.  (Following the records within the round, the
// workgroup waiting for those that have more: 10.5, - and 39.5.)
// The kernel has a numbering of its own: zones keep their numbers, through
// nodes get places such that each 128-byte line of labels (16 nodes) holds
// neighbours of each other (hbm_places).  A search's front is a ring; with
// nodes numbered along rows of a city every node of it brings a line of its
// own, which 64 workgroups an XCD cannot keep in 4 MB of L2.  Ties are
// broken by node numbers, not places, so the trees do not depend on it.
// Records of 5 links (a line) are read by 2 lanes.  Where most nodes have
// more than 5 links and no more than 10, records hold 10 and are read by 4,
// so that a node is expanded in one round.  Measured ms with records of 10
// and of 5 links: grids of 22,500 nodes with 4, 6, 8 and 12 links each, 200
// origins, 3 iterations 4.9 and 4.9, 7.0 and 8.5, 6.1 and 8.1, 10.4 and 9.6;
// 48,400 nodes with 6, 12 origins, 10 iterations 30 and 37; regional (4 links)
// 125 and 109 for two iterations.
constexpr int hrec_links(int group) { return group == 2 ? 5 : 10; }
constexpr size_t hrec_bytes(int group) { return 32 * (size_t)group; }
template <int kGroup>
struct __align__(64) HbmRec {
  double w[hrec_links(kGroup)];
  int head[hrec_links(kGroup)];
  int more;
  static_assert(hrec_links(kGroup) <= kHbmCand * kGroup, "a lane takes kHbmCand links");
};
static_assert(sizeof(HbmRec<2>) == hrec_bytes(2) && sizeof(HbmRec<4>) == hrec_bytes(4), "whole lines");
// HbmRec::more: the record that follows, whether the one after that follows
// too (a node's further records are a row that is read as a heap: record k
// leads to 2k + 1 and 2k + 2), and whether the row goes on
constexpr int kHrecNext = 0x0FFFFFFF, kHrecRow = 1 << 29, kHrecTwo = 1 << 30;
struct HbmRecOf {
  int first, end;                    // its links: those of [first, end) to through nodes
  int more;                          // HbmRec::more
  int node;                          // place of its node
};

// a thread per (variant, record), and per padding lane of the last slice
template <int kGroup>
__global__ __launch_bounds__(kBlock) void k_hbm_mirrors(OriginArgs A, int Vn, HbmRec<kGroup>* hrec,
                                                        uint2* sell_id, double* sellw_all) {
  constexpr int kLinks = hrec_links(kGroup);
  const int i = blockIdx.x * kBlock + threadIdx.x;       // record; below N the place of its node
  const int N = A.N, sl = i / kWave;
  const bool slice = sl < (N + kWave - 1) / kWave;
  if (!slice && i >= A.hrec_n) return;
  const int v = i < N ? A.node[i] : -1;
  const int begin = slice ? A.hsell_ptr[sl] + i % kWave : 0, end = slice ? A.hsell_ptr[sl + 1] : 0;
  for (int var = blockIdx.y; var < Vn; var += gridDim.y) {
    const double* fw = A.fww + (size_t)var * A.E;
    const double* rw = A.rvw + (size_t)var * A.E;
    double* sellw = sellw_all + (size_t)var * A.hsell_n;
    int at = begin;
    if (i < A.hrec_n) {
      const HbmRecOf of = A.hrec_of[i];
      HbmRec<kGroup> R;
      int n = 0;
#pragma unroll
      for (int g = 0; g < kLinks; ++g) { R.w[g] = INFINITY; R.head[g] = min(i, N - 1); }
      for (int k = of.first; k < of.end; ++k) {
        const int d = A.fw_dst[k];
        if (d < A.ft0 || d == A.tail[k]) continue;
#pragma unroll
        for (int g = 0; g < kLinks; ++g)
          if (g == n) { R.w[g] = fw[k]; R.head[g] = A.place[d]; }
        ++n;
      }
      R.more = of.more;
      hrec[(size_t)var * A.hrec_n + i] = R;
    }
    if (v >= 0) {
      for (int k = A.rv_off[v]; k < A.rv_off[v + 1] && at < end; ++k) {
        const int u = A.rv_src[k];
        if (v < A.ft0 || u < A.ft0 || u == v) continue;
        if (var == 0) sell_id[at] = make_uint2((unsigned)A.place[u], (unsigned)A.rv_eid[k]);
        sellw[at] = rw[k];
        at += kWave;
      }
    }
    for (; at < end; at += kWave) {
      if (var == 0) sell_id[at] = make_uint2((unsigned)min(i, N - 1), 0u);
      sellw[at] = INFINITY;
    }
  }
}

// workgroup-scope loads of a workgroup's private scratch row
__device__ __forceinline__ unsigned long long ldg_u64(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int ldg_i32(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int kGroup>
__global__ __launch_bounds__(kHbmBlock, kHbmPerCu * kHbmBlock / kWave / 4) void k_origin_hbm(OriginArgs A, int load, int items) {
  extern __shared__ unsigned long long sm[];
  constexpr int kLinks = hrec_links(kGroup), kRecBytes = (int)hrec_bytes(kGroup);
  constexpr int kWaves = kHbmBlock / kWave;
  const int N = A.N, ft0 = A.ft0, qcap = A.hqcap;
  const int W = (N + 63) >> 6;
  unsigned long long* bmA = sm;
  unsigned long long* bmB = bmA;                        // (the predecessors' use of the two bitmaps)
  unsigned long long* bmC = bmA + W;
  const int fcap = 2 * qcap;
  unsigned long long* tab_lab = bmA + W;                // [kHbmSlots] smallest label offered
  unsigned long long* far_lab = tab_lab + kHbmSlots;    // [fcap] labels when listed
  unsigned long long* near_lab = far_lab + fcap;        // 2 x [qcap]
  unsigned* far_node = (unsigned*)(near_lab + 2 * (size_t)qcap);
  unsigned* near_node = far_node + fcap;
  unsigned* tab_node = near_node + 2 * (size_t)qcap;    // [kHbmSlots] node + 1, 0: free
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  __shared__ int s_near[3], s_redo[3], s_far[2], s_wide[2];
  __shared__ unsigned long long s_min[3];
  __shared__ unsigned long long s_cnt[8];
  __shared__ int s_maxlen;
  __shared__ int s_level_ties, s_left, s_added;
  const int tid = threadIdx.x, wave = uniform(tid / kWave);
  const unsigned long long kMax = as_b(DBL_MAX);
  unsigned long long* dist = A.h_dist + (size_t)blockIdx.x * N;
  int* pred = A.h_pred + (size_t)blockIdx.x * N;
  int* ptail = A.h_ptail + (size_t)blockIdx.x * N;
  double* flow = (double*)dist;
  if (tid < 8) s_cnt[tid] = 0;
  if (tid == 0) s_maxlen = 0;
  unsigned n_exp = 0, n_scan = 0, n_upd = 0, n_steps = 0, n_loaded = 0, n_def = 0;   // (a lane's share)
  unsigned long long n_rounds = 0;
  unsigned long long c_relax = 0, c_pred = 0, c_load = 0;

  __shared__ int s_item;
  for (int k = 0;; ++k) {
    // the next item: from the launch's counter (the first free workgroup
    // takes it), or block-strided
    if (tid == 0) s_item = A.next ? atomicAdd(A.next, 1) : (int)blockIdx.x + k * (int)gridDim.x;
    __syncthreads();
    const int item = uniform(s_item);
    __syncthreads();
    if (item >= items) break;
    int var, origin;
    if (A.src_list) {
      var = 0;
      origin = A.src_list[item];
    } else if (A.order) {                     // longest origins first, all variants of each
      const int rank = item / A.vn;
      var = item - rank * A.vn;
      origin = A.order[rank];
    } else {
      var = item / A.zn;
      origin = A.z0 + item - var * A.zn;
    }
    if (A.var_on && !A.var_on[var]) continue;
    const int src = A.place[origin];          // (nodes below are places, unless they come from the CSR)
    const double* __restrict__ fw = A.fww + (size_t)var * A.E;
    const double* __restrict__ rw = A.rvw + (size_t)var * A.E;
    const char* recb = (const char*)A.hrec + (size_t)var * A.hrec_n * kRecBytes;
    const double* __restrict__ sellw = A.hsellw + (size_t)var * A.hsell_n;
    const long long clk0 = wall_clock64();
    // ---- label-correcting rounds in buckets.  Round r expands the near
    //      nodes: those lowered below T in round r-1, listed in an LDS queue
    //      with their label.  A node lowered to T or above goes to the far
    //      queue.  A round that leaves nothing near moves T to the smallest
    //      far label plus the bucket width and the far entries below it over.
    //      The width is delta; where none is set (delta < 0) it doubles when
    //      a bucket has fewer nodes than half a pass and halves when one has
    //      more than two passes.
    //      Labels are lowered with plain stores: an atomic at L2 is forwarded
    //      to memory (it must be seen by the other XCDs) and takes the line
    //      out of this one's L2, which made 0.57 G memory atomics and as many
    //      misses a loading of regional.  Two lanes that lower a label in the
    //      same round may leave the larger value, so every store is followed
    //      up: its queue entry (v, lab) is compared with v's label when it is
    //      taken out, in a later round.  Equal: v is expanded (once a round:
    //      `taken` flags).  The label is smaller: another entry stands for
    //      it.  Larger: it is stored again, with a new entry.  An entry is
    //      thus dropped only where the label at most equals its own, and a
    //      round never leaves a label above what it was at its start, so the
    //      labels that are left are the least.  Most such races are settled
    //      before the store, in a table of labels offered in the round: only
    //      the smallest offered to a node goes on (a node that finds no slot
    //      goes on anyway).  Without it the larger value wins half of the
    //      races and is expanded: 2.6 times the rounds on regional.
    //      Nodes that find the near queue full go to the far one; no store
    //      without an entry: where that is full too, the search turns wide
    //      (below), with the nodes of every entry flagged, the round's own
    //      among them.  Entries to be followed up once more grow from the end
    //      of the near queue, where kHbmRedo places are kept for them; should
    //      a round have more, the search turns wide too.
    //      A far entry whose node has a smaller label by now is of no use.
    //      When T moves they are weeded out if the far queue is half full or
    //      the last move brought few entries near: where some links cost far
    //      more than the others, the search would otherwise end in a move and
    //      a round for each of thousands of them (regional with 5% of its
    //      links at a million times their cost: 2,360 moves an origin and
    //      160 ms a loading, 39 weeded, as without such links).
    //      A round is a chain of trips to the XCD's L2 and beyond, so what
    //      counts is their number and the lines they touch: kGroup lanes
    //      share an expanded node, whose links are one line that is read
    //      beside its label; the labels of the heads are next.  Links to
    //      zones are left out (their labels are pulled at the end), and
    //      keeping a node for a later bucket costs nothing in the rounds
    //      between.  Measured on regional (4,000 origins, 94,000 nodes, 500
    //      rounds an origin): 2.9 ms an origin and workgroup for the labels,
    //      0.9 for the predecessors, 0.5 for the loading, 37 ms a loading;
    //      with one lane a node, CSR reads, an L2 atomic a lowered label and
    //      queued nodes looked at in every round 6.0, 1.2 and 0.8, 66 ms. ----
    const bool adapt = A.delta < 0.0;
    double width = fabs(A.delta);
    unsigned long long T = 0;
    int r = 1, fb = 0, lim = qcap;             // lim: places of the near queue for lowered nodes
    bool wide = false;
    constexpr int kPass = kHbmBlock / kGroup;     // nodes taken at once
    const int g = lane & (kGroup - 1), grp = lane / kGroup;
    // this lane's place among the lanes with `want`, counted on *n
    auto place = [&](bool want, int* n) {
      const unsigned long long bal = __ballot(want);
      int b0 = 0;
      if (bal) {
        const int leader = __ffsll((long long)bal) - 1;
        if (lane == leader) b0 = lds_add(n, __popcll(bal));
        b0 = __builtin_amdgcn_readlane(b0, leader);
      }
      return b0 + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32),
                                                 __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u));
    };
    auto put = [&](unsigned long long* lab, unsigned* node, int at, unsigned long long l, int v) {
      lab[at] = l;
      node[at] = (unsigned)v;
    };
    auto set_label = [&](int v, unsigned long long lab) {
      __hip_atomic_store(&dist[v], lab, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    // offers v the label cb; the slot it went to, -1: none of its two
    auto offer_label = [&](int v, unsigned long long cb) {
      const unsigned h = ((unsigned)v * 0x9E3779B1u) >> 22;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int s = (int)(h ^ k);
        const unsigned old = atomicCAS(&tab_node[s], 0u, (unsigned)v + 1u);
        if (old == 0u || old == (unsigned)v + 1u) {
          atomicMin(&tab_lab[s], cb);
          return s;
        }
      }
      return -1;
    };
    // gives v[i] the label cb[i] where low[i]: lowers and lists them, one LDS
    // atomic for both queues and all of the wavefront's
    auto relax = [&](auto& v, auto& cb, auto& low, int room) {
      constexpr int K = sizeof(low) / sizeof(low[0]);
      unsigned long long bn[K], bf[K];
      int nn = 0, nf = 0;
#pragma unroll
      for (int i = 0; i < K; ++i) {
        bn[i] = __ballot(low[i] && cb[i] < T);
        bf[i] = __ballot(low[i] && cb[i] >= T);
        nn += __popcll(bn[i]);
        nf += __popcll(bf[i]);
      }
      if (!(nn + nf)) return;
      int base = 0;
      if (lane < 2) base = lds_add(lane ? &s_far[fb] : &s_near[r % 3], lane ? nf : nn);
      int pn = __builtin_amdgcn_readlane(base, 0), pf = __builtin_amdgcn_readlane(base, 1);
      auto rank = [&](unsigned long long m) {
        return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      };
#pragma unroll
      for (int i = 0; i < K; ++i) {
        const bool near = low[i] && cb[i] < T && pn + rank(bn[i]) < room;
        int at = pf + rank(bf[i]);
        if (pn + __popcll(bn[i]) > room) {             // the rest of the near ones to the far queue
          const bool rest = low[i] && cb[i] < T && !near;
          const int k = place(rest, &s_far[fb]);
          if (rest) at = k;
        }
        if (near) {
          put(near_lab, near_node, (r & 1) * qcap + pn + rank(bn[i]), cb[i], v[i]);
        } else if (low[i] && at < fcap) {
          put(far_lab, far_node, at, cb[i], v[i]);
          ++n_def;
        } else if (low[i]) {
          s_wide[r & 1] = 1;
          low[i] = false;
        }
        if (low[i]) {
          set_label(v[i], cb[i]);
          ++n_upd;
        }
        pn += __popcll(bn[i]);
        pf += __popcll(bf[i]);
      }
    };
#pragma unroll 4
    for (int v = tid; v < N; v += kHbmBlock)
      __hip_atomic_store(&dist[v], kMax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    for (int w = tid; w < W; w += kHbmBlock) bmA[w] = 0;
    if (tid < 3) { s_near[tid] = tid == 0 ? 1 : 0; s_redo[tid] = 0; s_min[tid] = ~0ull; }
    if (tid < 2) { s_far[tid] = 0; s_wide[tid] = 0; }
    __syncthreads();
    if (tid == 0) {
      __hip_atomic_store(&dist[src], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      near_node[0] = (unsigned)src;
      near_lab[0] = 0ull;
    }
    __syncthreads();
    T = as_b(width);
    bool few = false;                        // the last move of T brought few entries near
    for (;;) {
      const int n1 = min(uniform(s_near[(r - 1) % 3]), lim);
      const int qn = n1 + min(uniform(s_redo[(r - 1) % 3]), qcap - lim);
      const int from = ((r - 1) & 1) * qcap, to = (r & 1) * qcap;
      const int room = qcap - min(qn, kHbmRedo);
      for (int s = tid; s < kHbmSlots; s += kHbmBlock) { tab_node[s] = 0u; tab_lab[s] = ~0ull; }
      for (int j0 = 0; j0 < qn; j0 += kPass) {
        // ---- the lanes of a group take an entry (all lanes come here) ----
        const int j = j0 + wave * (kWave / kGroup) + grp;
        const bool on = j < qn;
        const int at = from + (j < n1 ? j : qcap - 1 - (j - n1));
        const int u = on ? (int)near_node[at] : src;
        const unsigned long long lab = on ? near_lab[at] : kMax;
        const unsigned ro = (unsigned)u * kRecBytes;
        // (an entry from N on is a further record of a node that was expanded)
        // (no load is masked: a merge with a default waits for each of them)
        double w[kHbmCand];
        int v[kHbmCand];
        const unsigned long long seen = ldg_u64(&dist[min(u, N - 1)]), have = u < N ? seen : lab;
        const int more = *(const int*)(recb + (ro + 12u * kLinks));
#pragma unroll
        for (int i = 0; i < kHbmCand; ++i) {
          const unsigned k = min((unsigned)(g + i * kGroup), (unsigned)(kLinks - 1));
          w[i] = *(const double*)(recb + (ro + k * 8u));
          v[i] = *(const int*)(recb + (ro + 8u * kLinks + k * 4u));
        }
        if (j0 == 0) __syncthreads();                  // (the table is clear; the loads are on their way)
        const bool lost = on && g == 0 && have > lab;
        if (__builtin_expect(__ballot(lost) != 0, 0)) {
          const int k = place(lost, &s_redo[r % 3]);
          if (lost && k < qcap - room) {
            set_label(u, lab);
            put(near_lab, near_node, to + qcap - 1 - k, lab, u);
          } else if (lost) {
            s_wide[r & 1] = 1;
          }
        }
        bool first = on && g == 0 && have == lab;
        const unsigned long long bit = 1ull << (u & 63);
        if (first && u < N) first = !(atomicOr(&bmA[u >> 6], bit) & bit);
        const bool go = (__ballot(first) >> (lane & ~(kGroup - 1))) & 1ull;
        n_exp += first && u < N;
        unsigned long long cb[kHbmCand], hv[kHbmCand];
        bool low[kHbmCand];
        int slot[kHbmCand];
#pragma unroll
        for (int i = 0; i < kHbmCand; ++i) {
          cb[i] = as_b(as_d(lab) + w[i]);
          hv[i] = ldg_u64(&dist[v[i]]);
        }
#pragma unroll
        for (int i = 0; i < kHbmCand; ++i) {
          const bool in = go && cb[i] < kMax && g + i * kGroup < kLinks;
          n_scan += in;
          low[i] = in && cb[i] < hv[i];
          slot[i] = -1;
          if (low[i]) slot[i] = offer_label(v[i], cb[i]);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kHbmCand; ++i)
          if (slot[i] >= 0) low[i] = tab_lab[slot[i]] == cb[i];   // else a smaller one is stored
        relax(v, cb, low, room);
        const bool rec = go && (g == 0 ? more & kHrecNext : g == 1 && (more & kHrecTwo));
        if (__ballot(rec)) {                           // the records that follow
          int k = place(rec, &s_near[r % 3]);
          const bool rest = rec && k >= room;
          const int f = place(rest, &s_far[fb]);
          if (rec && !rest) put(near_lab, near_node, to + k, lab, (more & kHrecNext) + g);
          if (rest && f < fcap) put(far_lab, far_node, f, lab, (more & kHrecNext) + g);
          if (rest && f >= fcap) s_wide[r & 1] = 1;
        }
      }
      // (every entry is taken: the last pass's barrier)
      for (int j = tid; j < qn; j += kHbmBlock) {
        const unsigned u = near_node[from + (j < n1 ? j : qcap - 1 - (j - n1))];
        if (u < (unsigned)N) bmA[u >> 6] = 0ull;
      }
      if (tid == 0) { s_near[(r + 1) % 3] = 0; s_redo[(r + 1) % 3] = 0; }
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // (the round's stores are done)
      __syncthreads();
      lim = room;
      if (__builtin_expect(uniform(s_wide[r & 1]), 0)) {                    // an entry found no place
        const int nn = min(uniform(s_near[r % 3]), lim), nr = min(uniform(s_redo[r % 3]), qcap - lim);
        const int nf = min(uniform(s_far[fb]), fcap);
        for (int j = tid; j < qn + nn + nr + nf; j += kHbmBlock) {
          const int k = j - qn, at = j < qn ? from + (j < n1 ? j : qcap - 1 - (j - n1))
                                            : to + (k < nn ? k : qcap - 1 - (k - nn));
          const bool near = k < nn + nr;
          const unsigned long long lab = near ? near_lab[at] : far_lab[k - nn - nr];
          int v = (int)(near ? near_node[at] : far_node[k - nn - nr]);
          if (v >= N) v = A.hrec_of[v].node;
          if (k >= 0 && ldg_u64(&dist[v]) < lab) continue;   // (another entry stands for it)
          (void)__hip_atomic_fetch_min(&dist[v], lab, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          atomicOr(&bmA[v >> 6], 1ull << (v & 63));
        }
        wide = true;
        break;
      }
      bool done = false;
      while (!(min(uniform(s_near[r % 3]), lim) + uniform(s_redo[r % 3]))) {   // T moves
        const int fc = min(uniform(s_far[fb]), fcap);
        done = fc == 0;
        if (done) break;
        const bool weed = few || fc > fcap / 2;
        unsigned long long m = ~0ull;
        for (int i = tid; i < fc; i += kHbmBlock) {
          const unsigned long long lab = far_lab[i];
          if (weed && far_node[i] < (unsigned)N && ldg_u64(&dist[far_node[i]]) < lab)
            far_lab[i] = ~0ull;
          else
            m = min(m, lab);
        }
        for (int o = kWave / 2; o > 0; o >>= 1) m = min(m, __shfl_xor(m, o));
        if (lane == 0 && m != ~0ull) atomicMin(&s_min[fb], m);
        if (tid == 0) { s_far[fb ^ 1] = 0; s_near[r % 3] = 0; }
        __syncthreads();
        // 7/8 of the near queue at most, so that the entries find room for what
        // they lower; far entries first, so that the far queue empties
        const int fill = qcap - qcap / 8;
        lim = fill;
        const unsigned long long mn = s_min[fb];
        // (above the smallest label also where delta is below its last bit)
        if (mn != ~0ull) T = max(T, max(as_b(as_d(mn) + width), mn + 1));
        if (tid == 0) s_min[fb ^ 1] = ~0ull;
        for (int i0 = 0; i0 < fc; i0 += kHbmBlock) {   // (what stays closes up in place)
          const int i = i0 + tid;
          const unsigned long long lab = i < fc ? far_lab[i] : ~0ull;
          const bool on = lab != ~0ull;
          const int v = on ? (int)far_node[i] : src;
          __syncthreads();
          const bool near = on && lab < T;
          const int pn = place(near, &s_near[r % 3]);
          const bool keep = on && !(near && pn < fill);
          if (near && pn < fill) put(near_lab, near_node, to + pn, lab, v);
          const int pf = place(keep, &s_far[fb ^ 1]);
          if (keep) put(far_lab, far_node, pf, lab, v);
        }
        fb ^= 1;
        __syncthreads();
        const int moved = uniform(s_near[r % 3]);
        few = moved < kHbmFew;
        if (adapt) {
          if (moved > 2 * kPass)
            width *= 0.5;
          else if (moved < kPass / 2)
            width *= 2.0;
        }
      }
      if (done) break;
      if (r > 64 * N + 64) {
        if (tid == 0 && atomicCAS(&A.err[0], 0, 2) == 0) { A.err[1] = origin; A.err[2] = 0; }
        break;
      }
      ++r;
    }
    // ---- wide: more nodes wait than the queues hold.  They are flagged in
    //      bitmaps, one for the round, one for the next and one of those at
    //      T or above (which are flagged for the next round too where LDS has
    //      no room for three), and listed by node alone; a round of more
    //      nodes than its list holds goes by the flags, a wavefront taking
    //      every 8th word (64 nodes).  A lane expands a node.  Labels are
    //      lowered by atomics here, so nothing needs to be followed up.
    //      Measured, ms a loading: a random graph (40,000 nodes of 5 links,
    //      100 origins, fronts of thousands) 1.8; 4.9 with the tails of links
    //      that found no place expanded again at each move of T, and 2.1 with
    //      every listed node looked at in every round.  23,500 nodes of a
    //      city and 1,000 origins, costs spread by a log-normal factor of
    //      sigma 2: 4.9, 9.4 and 5.9. ----
    if (__builtin_expect(wide, 0)) {
      unsigned long long *cur = bmA, *nxt = bmC;         // (the queues' place)
      const int room = (int)((12 * kHbmSlots + kHbmQueueBytes * (size_t)qcap) / 8) - W;
      const bool three = room - W >= kHbmBlock;
      const int listed = max(0, three ? room - W : room);            // entries of a list
      unsigned long long* far = nxt + W;
      int* list = (int*)(three ? far + W : nxt + W);     // 2 x [listed]
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __syncthreads();
      for (int w = tid; w < (three ? 2 * W : W); w += kHbmBlock) nxt[w] = 0;
      // in s_near the flagged nodes of a round (the first goes by the flags),
      // in s_redo the expanded ones, in s_far[0] whether a node waits for T
      if (tid < 3) { s_near[tid] = tid == r % 3 ? INT_MAX : 0; s_redo[tid] = 0; s_min[tid] = ~0ull; }
      if (tid == 0) s_far[0] = 0;
      __syncthreads();
      // f(node of this lane, flagged, label) for every word of `bm` with a
      // flag, which are cleared; the next word's labels are on their way
      // meanwhile
      auto words = [&](unsigned long long* bm, auto&& f) {
        for (int w0 = wave; w0 < W; w0 += kWaves * kWave) {
          const int wi = w0 + lane * kWaves;
          unsigned long long mine = 0ull;
          if (wi < W) {
            mine = bm[wi];
            if (mine) bm[wi] = 0ull;
          }
          auto label = [&](unsigned long long m) {
            const int k = m ? __ffsll((long long)m) - 1 : 0;
            return ldg_u64(&dist[min((w0 + k * kWaves) * kWave + lane, N - 1)]);
          };
          unsigned long long m = __ballot(mine != 0ull), ahead = label(m);
          while (m) {
            const int k = __ffsll((long long)m) - 1;
            const unsigned long long lab = ahead;
            m &= m - 1;
            ahead = label(m);
            const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)mine, k);
            const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(mine >> 32), k);
            f((w0 + k * kWaves) * kWave + lane, ((lane < 32 ? lo : hi) >> (lane & 31)) & 1u, lab);
          }
        }
      };
      // flags v[i] where want[i] for round r + 1 and lists it there, unless it is
      auto flag = [&](auto& v, auto& want) {
        constexpr int K = sizeof(want) / sizeof(want[0]);
        unsigned long long bal[K];
        int n = 0;
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const unsigned long long bit = 1ull << (v[i] & 63);
          if (want[i]) want[i] = !(atomicOr(&nxt[v[i] >> 6], bit) & bit);
        }
#pragma unroll
        for (int i = 0; i < K; ++i) { bal[i] = __ballot(want[i]); n += __popcll(bal[i]); }
        if (!n) return;
        int at = 0;
        if (lane == 0) at = lds_add(&s_near[r % 3], n);
        at = __builtin_amdgcn_readlane(at, 0);
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const int k = at + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bal[i] >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((unsigned)bal[i], 0u));
          if (want[i] && k < listed) list[(r & 1) * listed + k] = v[i];
          at += __popcll(bal[i]);
        }
      };
      unsigned long long kept = ~0ull;
      int taken = 0, since = 0;                          // nodes expanded in this round, since T moved
      auto lower = [&](auto& v, auto& c, auto& have, bool go) {
        constexpr int K = sizeof(v) / sizeof(v[0]);
        bool want[K];
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const bool in = go && c[i] < kMax, low = in && c[i] < have[i], later = three && c[i] >= T;
          n_scan += in;
          n_upd += low;
          want[i] = low && !later;
          if (low) (void)__hip_atomic_fetch_min(&dist[v[i]], c[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          if (low && later) {
            atomicOr(&far[v[i] >> 6], 1ull << (v[i] & 63));
            s_far[0] = 1;
          }
        }
        flag(v, want);
      };
      auto expand = [&](int u, bool on, unsigned long long lab) {    // (all lanes)
        bool go = on && lab < T;
        const bool keep = on && !go;
        if (__ballot(keep)) {
          if (three) {
            if (keep) { atomicOr(&far[u >> 6], 1ull << (u & 63)); s_far[0] = 1; }
          } else {
            if (keep) kept = min(kept, lab);
            int x[1] = {u};
            bool want[1] = {keep};
            flag(x, want);
          }
        }
        const unsigned long long m = __ballot(go);
        if (!m) return;
        taken += __popcll(m);
        n_exp += go;
        for (int q = go ? u : src;;) {                   // its records
          const HbmRec<kGroup>* rec = (const HbmRec<kGroup>*)recb + q;
          constexpr int K = 5;                           // links at once
          const int more = rec->more;
#pragma unroll 1
          for (int k = 0; k < kLinks; k += K) {
            int x[K];
            unsigned long long c[K], have[K];
#pragma unroll
            for (int i = 0; i < K; ++i) { x[i] = rec->head[k + i]; c[i] = as_b(as_d(lab) + rec->w[k + i]); }
#pragma unroll
            for (int i = 0; i < K; ++i) have[i] = ldg_u64(&dist[x[i]]);
            lower(x, c, have, go);
          }
          go = go && more & kHrecRow;
          if (!__ballot(go)) break;
          if (go) q = q < N ? more & kHrecNext : q + 1;
        }
      };
      for (++r;; ++r) {
        const int sl = r % 3, n = uniform(s_near[(r - 1) % 3]);
        taken = 0;
        if (n <= listed) {
          const int* q = list + ((r - 1) & 1) * listed;
          for (int j0 = 0; j0 < n; j0 += kHbmBlock) {
            const bool on = j0 + tid < n;
            const int u = on ? q[j0 + tid] : src;
            if (on) cur[u >> 6] = 0ull;
            expand(u, on, ldg_u64(&dist[u]));
          }
        } else {
          words(cur, expand);
        }
        auto smallest = [&](unsigned long long x) {      // of the wavefront's, to s_min[sl]
          for (int o = kWave / 2; o > 0; o >>= 1) x = min(x, __shfl_xor(x, o));
          if (lane == 0 && x != ~0ull) atomicMin(&s_min[sl], x);
        };
        if (!three) smallest(kept);
        kept = ~0ull;
        if (lane == 0 && taken) atomicAdd(&s_redo[sl], taken);
        if (tid == 0) { const int sn = (r + 1) % 3; s_near[sn] = 0; s_redo[sn] = 0; s_min[sn] = ~0ull; }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
        const int got = uniform(s_redo[sl]);
        const bool work = uniform(s_near[sl]) != 0;
        since += got;
        if (!work && !(three && uniform(s_far[0]))) break;
        if (three ? !work : !got) {                      // T moves
          if (three) {
            // (a far node below T by now was expanded since)
            unsigned long long m = ~0ull;
            words(far, [&](int u, bool on, unsigned long long lab) {
              const unsigned long long live = __ballot(on && lab >= T);
              if (on && lab >= T) m = min(m, lab);
              if (lane == 0) far[u >> 6] = live;
            });
            smallest(m);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __syncthreads();
          }
          const unsigned long long mn = s_min[sl];
          if (mn == ~0ull) break;
          if (adapt) width *= since < kPass ? 2.0 : since > 4 * kHbmBlock ? 0.5 : 1.0;
          T = max(T, max(as_b(as_d(mn) + width), mn + 1));
          since = 0;
          if (three) {
            words(far, [&](int u, bool on, unsigned long long lab) {
              const unsigned long long later = __ballot(on && lab >= T);
              if (lane == 0) far[u >> 6] = later;
              int x[1] = {u};
              bool want[1] = {on && lab < T};
              flag(x, want);
            });
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __syncthreads();
          }
        }
        if (r > 64 * N + 64) {
          if (tid == 0 && atomicCAS(&A.err[0], 0, 2) == 0) { A.err[1] = origin; A.err[2] = 0; }
          break;
        }
        unsigned long long* t = cur; cur = nxt; nxt = t;
      }
    }
    n_rounds += (unsigned long long)r;
    if (A.work && tid == 0 && var == 0) A.work[origin] = r;
    const long long clk1 = wall_clock64();

    // ---- predecessor links: smallest tail label below the node's, then
    //      tail id; nodes with none join by attach_level_ties.  Through
    //      nodes by slices of 64, whose in-links are contiguous row by row;
    //      the next slice's rows are on their way while a slice's tails are
    //      looked up.  The links of an origin that is a zone are in no slice
    //      and come first (label 0 and the smallest id: they win where they
    //      are tight).  Then the zones, whose labels are the minimum over
    //      their in-links. ----
    for (int w = tid; w < 2 * W; w += kHbmBlock) bmB[w] = 0;   // level ties | chosen
    if (tid == 0) s_level_ties = 0;
    __syncthreads();
    auto choose = [&](int v, int p, int pt, unsigned long long dv) {
      __hip_atomic_store(&pred[v], p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __hip_atomic_store(&ptail[v], pt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      // reached, not the origin, and no tight tail with a smaller label
      const bool level_tie = p < 0 && v != src && dv != kMax;
      if (level_tie) {                                 // (by node)
        const int n = A.node[v];
        atomicOr(&bmB[n >> 6], 1ull << (n & 63));
        s_level_ties = 1;
      }
      if (A.out_dist) {
        const size_t o = (size_t)A.node[v] * A.ld + item;
        A.out_dist[o] = as_d(dv);
        if (!level_tie) A.out_pred[o] = p;
      }
    };
    if (src < ft0)
      for (int e = A.fw_off[src] + tid; e < A.fw_off[src + 1]; e += kHbmBlock) {
        const int v = A.place[A.fw_dst[e]];
        const unsigned long long wb = as_b(0.0 + fw[e]);
        if (v < ft0 || wb == 0ull || wb >= kMax || ldg_u64(&dist[v]) != wb) continue;
        bool first = true;                             // of equal parallel links
        for (int k = A.fw_off[src]; k < e; ++k) first = first && !(A.fw_dst[k] == A.fw_dst[e] && fw[k] == fw[e]);
        if (!first) continue;
        choose(v, e, src, wb);
        atomicOr(&bmC[v >> 6], 1ull << (v & 63));      // chosen
      }
    __syncthreads();
    {
      constexpr int kFetch = 5;                        // rows of a slice loaded ahead
      struct Rows { uint2 id[kFetch]; double w[kFetch]; unsigned long long dv; int at, rows; };
      auto fetch = [&](int sl, Rows& R) {
        const int p0 = A.hsell_ptr[sl];
        R.at = p0 + lane;
        R.rows = (A.hsell_ptr[sl + 1] - p0) / kWave;
#pragma unroll
        for (int i = 0; i < kFetch; ++i)
          if (i < R.rows) { R.id[i] = A.hsell_id[R.at + i * kWave]; R.w[i] = sellw[R.at + i * kWave]; }
        const int v = sl * kWave + lane;
        R.dv = v < N && v >= ft0 ? ldg_u64(&dist[v]) : kMax;
      };
      auto select = [&](int sl, const Rows& R) {
        const int v = sl * kWave + lane;
        const unsigned long long dv = R.dv;
        unsigned long long best_du = dv, du[kFetch];   // only tails with a smaller label can win
        int p = -1, pt = INT_MAX;
        auto offer = [&](int u, int e, double w, unsigned long long d) {
          const bool tight = as_b(as_d(d) + w) == dv;
          if (tight && (d < best_du || (d == best_du && p >= 0 && A.node[u] < A.node[pt]))) {
            best_du = d; p = e; pt = u;
          }
        };
#pragma unroll
        for (int i = 0; i < kFetch; ++i)
          if (i < R.rows) du[i] = ldg_u64(&dist[R.id[i].x]);
#pragma unroll
        for (int i = 0; i < kFetch; ++i)
          if (i < R.rows) offer((int)R.id[i].x, (int)R.id[i].y, R.w[i], du[i]);
        for (int i = kFetch; i < R.rows; ++i) {
          const uint2 id = A.hsell_id[R.at + i * kWave];
          offer((int)id.x, (int)id.y, sellw[R.at + i * kWave], ldg_u64(&dist[id.x]));
        }
        if (v >= N || v < ft0) return;
        if (R.rows == kSellWidth)
          for (int n = A.node[v], e = A.rv_off[n]; e < A.rv_off[n + 1]; ++e) {
            const int u = A.place[A.rv_src[e]];
            if (u >= ft0 && u != v) offer(u, A.rv_eid[e], rw[e], ldg_u64(&dist[u]));
          }
        if ((bmC[sl] >> lane) & 1ull) return;          // chosen
        if (dv == kMax || v == src) p = -1;
        choose(v, p, p < 0 ? -1 : pt, dv);
      };
      for (int sl = ft0 / kWave + wave; sl < W; sl += kWaves) {
        Rows R;
        fetch(sl, R);
        select(sl, R);
      }
    }
    for (int v = tid; v < ft0 && v < N; v += kHbmBlock) {
      int p = -1, pt = -1;
      unsigned long long dk = v == src ? 0ull : kMax;
      if (v != src) {
        auto tails = [&](auto&& f) {                   // f(tail, link, its label, label through it)
          for (int e = A.rv_off[v]; e < A.rv_off[v + 1]; ++e) {
            const int u = A.place[A.rv_src[e]];
            if (u == v || (u < ft0 && u != src)) continue;
            const unsigned long long du = u == src ? 0ull : ldg_u64(&dist[u]);
            if (du != kMax) f(u, A.rv_eid[e], du, as_b(as_d(du) + rw[e]));
          }
        };
        tails([&](int, int, unsigned long long, unsigned long long c) { dk = min(dk, c); });
        unsigned long long best_du = dk;
        if (dk != kMax)
          tails([&](int u, int e, unsigned long long du, unsigned long long c) {
            if (c == dk && (du < best_du || (du == best_du && p >= 0 && A.node[u] < A.node[pt]))) {
              best_du = du;
              p = e;
              pt = u;
            }
          });
        __hip_atomic_store(&dist[v], dk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      choose(v, p, pt, dk);
    }
    __syncthreads();
    if (s_level_ties) {
      const bool ok = attach_level_ties<kHbmBlock>(
          A, rw, origin, bmB, bmC, &s_left, &s_added, [&](int v) { return ldg_u64(&dist[A.place[v]]); },
          [&](int v, int e, int u) {                   // (v and u are nodes here)
            const int i = A.place[v];
            __hip_atomic_store(&pred[i], e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_store(&ptail[i], A.place[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (A.out_dist) A.out_pred[(size_t)v * A.ld + item] = e;
          });
      if (!ok && tid == 0 && atomicCAS(&A.err[0], 0, 3) == 0) { A.err[1] = origin; A.err[2] = 0; }
      __syncthreads();
    }
    // every label read is done: the row now holds flows
    const long long clk2 = wall_clock64();
    c_relax += (unsigned long long)(clk1 - clk0);
    c_pred += (unsigned long long)(clk2 - clk1);
    if (!load) continue;

    // ---- loading: destination walks, then tree links with flow ----
#pragma unroll 4
    for (int v = tid; v < N; v += kHbmBlock)
      __hip_atomic_store(&dist[v], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // +0.0
    __syncthreads();
    int maxlen = 0;
    for (long long i = A.od_start[origin] + tid; i < A.od_start[origin + 1]; i += kHbmBlock) {
      const int d = A.place[A.od_dest[i]];
      const double f = A.od_val[i];
      if (d == src || !(f > 0.0)) continue;
      if (ldg_i32(&pred[d]) < 0) {
        if (atomicCAS(&A.err[0], 0, 1) == 0) { A.err[1] = origin; A.err[2] = A.od_dest[i]; }
        continue;
      }
      int v = d, len = 0;
      while (v != src) {
        if (len > N || v < 0) {
          if (atomicCAS(&A.err[0], 0, 3) == 0) { A.err[1] = origin; A.err[2] = 0; }
          break;
        }
        __hip_atomic_fetch_add(&flow[v], f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        v = ldg_i32(&ptail[v]);
        ++len;
      }
      n_steps += (unsigned)len;
      maxlen = max(maxlen, len);
    }
    if (maxlen) atomicMax(&s_maxlen, maxlen);
    __syncthreads();
    double* __restrict__ yv = A.y + (size_t)var * A.E;
    constexpr int kScan = 4;                           // nodes a thread has in flight
    for (int v0 = tid; v0 < N; v0 += kScan * kHbmBlock) {
      double f[kScan];
      int p[kScan];
#pragma unroll
      for (int i = 0; i < kScan; ++i)
        f[i] = v0 + i * kHbmBlock < N ? as_d(ldg_u64(&dist[v0 + i * kHbmBlock])) : 0.0;
#pragma unroll
      for (int i = 0; i < kScan; ++i) p[i] = f[i] != 0.0 ? ldg_i32(&pred[v0 + i * kHbmBlock]) : -1;
#pragma unroll
      for (int i = 0; i < kScan; ++i)
        if (p[i] >= 0) {
          unsafeAtomicAdd(&yv[p[i]], f[i]);
          ++n_loaded;
        }
    }
    __syncthreads();          // the row is reused by the next item
    c_load += (unsigned long long)(wall_clock64() - clk2);
  }
  if (A.counters) {
    const unsigned long long cnt[8] = {n_exp, n_scan, n_upd, 0, 0, n_loaded, n_steps, n_def};
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < 3 || i > 4) atomicAdd(&s_cnt[i], cnt[i]);
    __syncthreads();
    if (tid == 0) {
      atomicAdd(&A.counters[7], s_cnt[7]);
      atomicAdd(&A.counters[0], s_cnt[0]); atomicAdd(&A.counters[1], s_cnt[1]);
      atomicAdd(&A.counters[2], s_cnt[2]); atomicAdd(&A.counters[3], n_rounds);
      atomicAdd(&A.counters[4], (unsigned long long)s_maxlen);
      atomicAdd(&A.counters[5], s_cnt[5]); atomicAdd(&A.counters[6], s_cnt[6]);
      atomicAdd(&A.counters[8], c_relax); atomicAdd(&A.counters[9], c_pred);
      atomicAdd(&A.counters[10], c_load);
    }
  }
}


// ---------------------------------------------------------------------------
// link passes
// ---------------------------------------------------------------------------

struct Links {
  int E, V;
  const double *t0, *cap, *B, *pw;   // [V * E]
  const unsigned char* present;      // [V * E]
  const int* rvpos;                  // [E] position of link k in reverse order
  double *x, *y, *c;                 // [V * E]
  double* rvw;                       // [V * E]  costs, reverse-CSR order, INF: absent
  double* fww;                       // [V * E]  costs, link order, INF: absent
  // mirrors of the LDS kernel (null: it does not apply to this network)
  double *rec, *sellw;
  const int *recpos, *sellpos;       // [E] position of link k in a variant's mirror, -1: none
  long long rec_n, sell_n;           // their sizes per variant
};

// The cost of link k of variant var, in every order a search reads it.
__device__ __forceinline__ void store_cost(const Links& K, int var, int k, double c) {
  const size_t off = (size_t)var * K.E;
  const double wv = K.present[off + k] ? c : INFINITY;
  K.rvw[off + K.rvpos[k]] = wv;
  K.fww[off + k] = wv;
  if (K.rec) {
    const int a = K.recpos[k], b = K.sellpos[k];
    if (a >= 0) K.rec[(size_t)var * K.rec_n + a] = wv;
    if (b >= 0) K.sellw[(size_t)var * K.sell_n + b] = wv;
  }
}

// The fixed parts of the LDS kernel's mirrors (heads, tails, link ids and
// every link's positions) and infinite costs where a slot holds no link; a
// thread per node, and per padding lane of the last slice.
__global__ __launch_bounds__(kBlock) void k_mirrors(Graph G, Links K, const int* sell_ptr,
                                                    unsigned* sell_id, int* recpos, int* sellpos) {
  const int v = blockIdx.x * kBlock + threadIdx.x;
  const int sl = v / kWave;
  if (sl >= (G.N + kWave - 1) / kWave) return;
  const int base = sell_ptr[sl] + v % kWave, end = sell_ptr[sl + 1];
  int at = base;
  if (v < G.N) {
    unsigned short head[8] = {};
    int n = 0;
    for (int g = 0; g < kRecLinks; ++g) head[g] = (unsigned short)v;
    for (int k = G.fw_off[v]; k < G.fw_off[v + 1]; ++k) {
      const int d = G.fw_dst[k];
      recpos[k] = -1;
      if (d < G.ft0 || d == v) continue;
      if (n < kRecLinks) {
        head[n] = (unsigned short)d;
        recpos[k] = v * kRecDoubles + n;
      }
      ++n;
    }
    const unsigned mark = (n > kGroup ? kRecMore : 0u) | (n > kRecLinks ? kRecCsr : 0u);
    for (int g = 0; g < kRecLinks; ++g) head[g] |= (unsigned short)mark;
    for (int var = 0; var < K.V; ++var) {
      double* r = K.rec + (size_t)var * K.rec_n + (size_t)v * kRecDoubles;
      for (int g = 0; g < kRecLinks; ++g) r[g] = INFINITY;
      __builtin_memcpy(r + kRecLinks, head, 16);
    }
    for (int k = G.rv_off[v]; k < G.rv_off[v + 1]; ++k) {
      const int u = G.rv_src[k], e = G.rv_eid[k];
      sellpos[e] = -1;
      if (v < G.ft0 || u < G.ft0 || u == v || at >= end) continue;
      sell_id[at] = (unsigned)u | (unsigned)e << 16;
      sellpos[e] = at;
      at += kWave;
    }
  }
  for (; at < end; at += kWave) {
    sell_id[at] = kSellNone | (unsigned)min(v, G.N - 1);
    for (int var = 0; var < K.V; ++var) K.sellw[(size_t)var * K.sell_n + at] = INFINITY;
  }
}

struct VarState {
  double best_lb, relgap, lambda, objective, total_demand, vht;
  int iter, active, stepping, need_more, jnext, found;
};

constexpr int kMaxGraphIters = 8;    // iterations per whole-iteration replay, at most

// Arguments of a tapgpu_fw_run call that the decision kernel reads from
// device memory, so a captured iteration graph serves every call.
struct FwParams {
  tapgpu_iter* trace;
  int trace_cap;
  int max_iters;
  double target;
  int jwin;                 // step sizes a line-search window decides on (<= kJ)
};

// The LDS kernel's mirrors of the current costs (after passes that did not
// keep them).
__global__ __launch_bounds__(kBlock) void k_mirror_costs(Links K) {
  const long long n = (long long)K.E * K.V;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (long long)gridDim.x * kBlock) {
    const int var = (int)(i / K.E), k = (int)(i - (long long)var * K.E);
    const int a = K.recpos[k], b = K.sellpos[k];
    if (a >= 0) K.rec[(size_t)var * K.rec_n + a] = K.fww[i];
    if (b >= 0) K.sellw[(size_t)var * K.sell_n + b] = K.fww[i];
  }
}

// mode 0: c = t0 (free-flow, initial Wa); mode 1: c = BPR(x); mode 2: c given
__global__ __launch_bounds__(kBlock) void k_costs(Links K, int mode, const unsigned char* var_on,
                                                  int v0, int Vn) {
  const long long n = (long long)K.E * Vn;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (long long)gridDim.x * kBlock) {
    const int var = v0 + (int)(i / K.E);
    const int k = (int)(i - (long long)(var - v0) * K.E);
    if (var_on && !var_on[var]) continue;
    const size_t j = (size_t)var * K.E + k;
    double c;
    if (mode == 0) c = K.t0[j];
    else if (mode == 1) c = tap_bpr(K.t0[j], K.cap[j], K.B[j], K.pw[j], K.x[j]);
    else c = K.c[j];
    K.c[j] = c;
    store_cost(K, var, k, c);
  }
}

// All kQ compensated sums of a block at once, in a fixed order.  Inside a
// wavefront by recursive halving: at each step a lane hands half of the sums
// it still carries to its partner and merges the partner's share of the
// other half (10 + 5 + 3 + 2 + 1 + 1 merges, where a butterfly of all 19
// sums takes 114), then one thread per sum merges the wavefronts.  The
// result is in out[] for every thread after the call's last barrier; sh
// holds a row per wavefront.
//
// The exchanges are register moves, not LDS permutes: between the halves of
// 32 and of 16 lanes the swap instructions, which hand over and keep in
// one, inside a row of 16 the data-parallel moves.  (kOff 4 is i ^ 7: it
// also turns the lanes of a quad round, whose shares are all different yet.)
template <int kOff>
__device__ __forceinline__ unsigned xchg_u32(unsigned x) {
  constexpr int ctrl = kOff == 8 ? 0x128 /* row_ror:8 */ : kOff == 4 ? 0x141 /* row_half_mirror */
                       : kOff == 2 ? 0x4E /* quad_perm 2,3,0,1 */ : 0xB1 /* quad_perm 1,0,3,2 */;
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, ctrl, 0xf, 0xf, false);
}
template <int kOff>
__device__ __forceinline__ double xchg(double x) {
  const unsigned long long b = as_b(x);
  const unsigned lo = xchg_u32<kOff>((unsigned)b), hi = xchg_u32<kOff>((unsigned)(b >> 32));
  return as_d((unsigned long long)hi << 32 | lo);
}
// lower half: {own a, partner's a}; upper half: {partner's b, own b}
template <int kOff>
__device__ __forceinline__ void swap_halves(double& a, double& b) {
  const unsigned long long x = as_b(a), y = as_b(b);
  unsigned r0[2], r1[2];
  if constexpr (kOff == 32) {
    auto p = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    auto q = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    r0[0] = p[0]; r0[1] = p[1]; r1[0] = q[0]; r1[1] = q[1];
  } else {
    auto p = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    auto q = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    r0[0] = p[0]; r0[1] = p[1]; r1[0] = q[0]; r1[1] = q[1];
  }
  a = as_d((unsigned long long)r1[0] << 32 | r0[0]);
  b = as_d((unsigned long long)r1[1] << 32 | r0[1]);
}

template <int kOff, int kHave>
__device__ __forceinline__ void halve_acc(tap_acc* v, int lane) {
  constexpr int kKeep = (kHave + 1) / 2;
#pragma unroll
  for (int i = 0; i < kKeep; ++i) {
    tap_acc lo = v[i], hi{0.0, 0.0};
    if (kKeep + i < kHave) hi = v[kKeep + i];
    if constexpr (kOff >= 16) {
      swap_halves<kOff>(lo.s, hi.s);
      swap_halves<kOff>(lo.c, hi.c);
      tap_acc_merge(&lo, hi);
      v[i] = lo;
    } else {
      const bool up = lane & kOff;
      const tap_acc give = up ? lo : hi;
      tap_acc keep = up ? hi : lo, got;
      got.s = xchg<kOff>(give.s);
      got.c = xchg<kOff>(give.c);
      tap_acc_merge(&keep, got);
      v[i] = keep;
    }
  }
}

// One sum, whose shares are in both lanes of a pair: merged in both, the
// lower lane's share first.
template <int kOff>
__device__ __forceinline__ void pair_acc(tap_acc* v, int lane) {
  tap_acc got;
  got.s = xchg<kOff>(v->s);
  got.c = xchg<kOff>(v->c);
  tap_acc a = (lane & kOff) ? got : *v;
  tap_acc_merge(&a, (lane & kOff) ? *v : got);
  *v = a;
}

template <int kWaves>
__device__ void block_reduce_acc(tap_acc* v, tap_acc* sh /* [kWaves][kQ] */, tap_acc* out /* [kQ] */) {
  static_assert(kQ == 19, "the halving below is written for 19 sums");
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  halve_acc<32, 19>(v, lane);      // 10 and 9
  halve_acc<16, 10>(v, lane);      // 5 and 5
  halve_acc<8, 5>(v, lane);        // 3 and 2
  halve_acc<4, 3>(v, lane);        // 2 and 1
  halve_acc<2, 2>(v, lane);        // 1 and 1
  pair_acc<1>(v, lane);
  const int b5 = lane >> 5 & 1, b4 = lane >> 4 & 1, b3 = lane >> 3 & 1, b2 = lane >> 2 & 1, b1 = lane >> 1 & 1;
  const int in5 = 3 * b3 + 2 * b2 + b1;                       // of the 5 sums of this 8-lane group
  const int q = 10 * b5 + 5 * b4 + in5;
  const bool holds = (b3 ? !b2 : !(b2 && b1)) && q < kQ && !(lane & 1);
  if (holds) sh[w * kQ + q] = v[0];
  __syncthreads();
  if (threadIdx.x < kQ) {
    tap_acc a = sh[threadIdx.x];
    for (int j = 1; j < kWaves; ++j) tap_acc_merge(&a, sh[j * kQ + threadIdx.x]);
    out[threadIdx.x] = a;
  }
  __syncthreads();
}

// acc[3 + j] += BPR(x + 2^-(jbase+j) d) * d for the kJ step sizes of a
// window (lam0 = 2^-jbase).  Halving is exact for every step size used
// (2^-1016 is still a normal double), so lam equals ldexp(1, -(jbase + j)).
// Unrolled, so the sums stay in registers.
__device__ __forceinline__ void step_sums(tap_acc* acc, double lam0, double x, double d, double t0,
                                          double cap, double B, double pw) {
  double lam = lam0;
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    const double q = x + lam * d;
    tap_acc_add(&acc[3 + j], tap_bpr(t0, cap, B, pw, q) * d);
    lam *= 0.5;
  }
}

// acc += a link's terms of a window; the first window also sums g(0) = c d,
// the objective and VHT.
__device__ __forceinline__ void link_sums(tap_acc* acc, const Links& K, size_t i, double lam0, bool first) {
  const double x = K.x[i];
  const double d = K.y[i] - x;
  const double t0 = K.t0[i], cap = K.cap[i], B = K.B[i], pw = K.pw[i];
  if (first) {
    const double c = K.c[i];
    tap_acc_add(&acc[0], c * d);
    tap_acc_add(&acc[1], tap_integral(t0, cap, B, pw, x));
    tap_acc_add(&acc[2], x * c);
  }
  step_sums(acc, lam0, x, d, t0, cap, B, pw);
}

// Per variant: lambda (first 2^-j with g <= 0, the reference's rule), then
// gap, objective, lower bound, relative gap, average excess cost, trace
// record, stop test.
// The decision of one window for one variant from its merged sums acc[kQ],
// by one wavefront (all its lanes keep the same state; lane 0 writes): on
// the first window the iteration's scalars and trace record, then lambda =
// the first 2^-j with g <= 0 (a lane looks at each j), or a request for the
// next window (need_more, jnext).
__device__ __forceinline__ void decide_window(VarState& s, const tap_acc* acc, int only_g,
                                              const FwParams& prm, int var) {
  const int lane = lane_id();
  const int jbase = only_g ? s.jnext : 0;
  const int jl = min(lane, kJ - 1);
  const unsigned long long neg = ballot(tap_acc_value(acc[3 + jl]) <= 0) & ((1ull << kJ) - 1ull);
  tapgpu_iter* const rec = s.iter < prm.trace_cap ? prm.trace + (size_t)var * prm.trace_cap + s.iter : nullptr;
  if (!only_g) {
    const double g0 = tap_acc_value(acc[0]);
    s.objective = tap_acc_value(acc[1]);
    s.vht = tap_acc_value(acc[2]);
    s.found = 0;
    s.need_more = 0;
    if (g0 >= 0) {
      s.lambda = 0.0; s.found = 1;
    } else if (neg & 1ull) {
      s.lambda = 1.0; s.found = 1;
    }
    // record the iteration's scalars (lambda filled below)
    const double gap = -g0;
    const double lb = s.objective - gap;
    if (lb > s.best_lb) s.best_lb = lb;
    if (s.best_lb != 0) s.relgap = (s.objective - s.best_lb) / fabs(s.best_lb);
    if (rec && lane == 0) {
      tapgpu_iter t;
      t.lambda = 0.0; t.gap = gap; t.objective = s.objective; t.lowerbound = lb;
      t.best_lowerbound = s.best_lb; t.relgap = s.relgap;
      t.avg_excess = -g0 / s.total_demand; t.vht = s.vht;
      *rec = t;
    }
  }
  if (!s.found) {
    // steps jbase .. jbase + jwin - 1, from 2^-1 on and down to 2^-kMaxHalvings
    const int n = min(prm.jwin, kMaxHalvings + 1 - jbase);
    unsigned long long m = neg & ((1ull << n) - 1ull);
    if (jbase == 0) m &= ~1ull;
    if (m) {
      s.lambda = ldexp(1.0, -(jbase + __ffsll((long long)m) - 1));
      s.found = 1;
    } else if (jbase + prm.jwin > kMaxHalvings) {
      s.lambda = 0.0;            // bisection cap reached: lambda_left == 0
      s.found = 1;
    } else {
      s.need_more = 1;
      s.jnext = jbase + prm.jwin;
    }
  }
  if (s.found) {
    s.need_more = 0;
    if (rec && lane == 0) rec->lambda = s.lambda;
    s.iter += 1;
    s.active = (prm.max_iters <= 0 || s.iter < prm.max_iters) && (prm.target <= 0 || s.relgap > prm.target);
  }
}

// x += lambda * (y - x), c = BPR(x) and its mirrors; clears y for the next
// loading.
__device__ __forceinline__ void step_link(const Links& K, int var, int k, double lambda) {
  const size_t i = (size_t)var * K.E + k;
  const double x = K.x[i] + lambda * (K.y[i] - K.x[i]);
  K.x[i] = x;
  K.y[i] = 0.0;
  const double c = tap_bpr(K.t0[i], K.cap[i], K.B[i], K.pw[i], x);
  K.c[i] = c;
  store_cost(K, var, k, c);
}

// Hands this block's sums[kQ] over and, in the last of the gridDim.x blocks
// to do so, leaves the merged sums (in a fixed order) in sums[] and returns
// true.  part: [gridDim.x][kQ]; done: a counter, 0 before and after; sh:
// [kMergeGroups][kQ].  The sums go through the XCDs' caches as device-scope
// stores and loads, and the stores have arrived before the count: no fence,
// which would write back a whole L2 for every block (512 variants of metro:
// 13 ms a step).
constexpr int kMergeGroups = kBlock / kQ;
__device__ bool merge_blocks(tap_acc* sums, tap_acc* sh, tap_acc* part, unsigned* done) {
  __shared__ int s_last;
  const int tid = threadIdx.x, nb = gridDim.x;
  if (tid < kQ) {
    tap_acc* mine = part + (size_t)blockIdx.x * kQ + tid;
    __hip_atomic_store(&mine->s, sums[tid].s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&mine->c, sums[tid].c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __syncthreads();
  if (tid == 0)
    s_last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)nb - 1;
  __syncthreads();
  if (!s_last) return false;
  if (tid < kMergeGroups * kQ) {
    const int q = tid % kQ, g = tid / kQ;
    tap_acc a{0.0, 0.0};
    for (int b = g; b < nb; b += kMergeGroups) {
      tap_acc t;
      t.s = __hip_atomic_load(&part[(size_t)b * kQ + q].s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      t.c = __hip_atomic_load(&part[(size_t)b * kQ + q].c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      tap_acc_merge(&a, t);
    }
    sh[g * kQ + q] = a;
  }
  if (tid == 0) *done = 0;
  __syncthreads();
  if (tid < kQ) {
    tap_acc a = sh[tid];
    for (int g = 1; g < kMergeGroups; ++g) tap_acc_merge(&a, sh[g * kQ + tid]);
    sums[tid] = a;
  }
  __syncthreads();
  return true;
}

// The line search of an iteration in one launch: `blocks` blocks a variant
// sum the first window, and the last one to finish merges their sums and
// decides.  A step below the first window (2^-15: rare) needs further ones:
// on networks of up to kSoloLinks links that block sums them by itself; on
// larger ones each takes a launch with `more`, which the host issues when it
// sees need_more.  Until then the variant is off, so that the iterations
// left in a replay pass it by and its loading stays.
// A variant that is off, and every variant after a loading that reported an
// error (a level tie in the lanes kernel, redone by the host), takes no step:
// its state stays as it was.  With one block a variant (small networks) the
// block sums every window and takes the step, so an iteration's link work is
// one launch; else k_link_step follows.
//
// A link costs 16 cost evaluations (~1,000 instructions) and a block's
// reduction ~450, so a thread takes one link while that leaves the chip
// unfilled, and up to kLinkPer where a batch or a large network fills it
// anyway.  Measured: metro (43,600 links) search and step 22 us an
// iteration, and ~58 as eight launches (two windows of 120 single-wavefront
// blocks with a butterfly reduction, two decisions, step, flags, clears);
// 512 variants of metro 1.0 ms with 8 links a thread, 2.0 ms with one;
// town (3,840 links) 15 us, and ~40 for one block doing all of it (rocprof).
constexpr int kLinkPer = 8;
constexpr long long kLinkFill = 1 << 20;   // links a launch has per link of a thread
constexpr int kSmallLinks = 512;     // links up to which one block a variant is faster
// Links up to which one block sums a further window as fast as the host has it
// done by many: ~2 us for each link of a thread, against ~100 us.  Measured, ms
// for solves with such steps, one block and the host: 200 iterations with 64 of
// them on 3,800 links 13.3 and 15.6, with 70 on 28,000 60.4 and 41.4, with 49 on
// 57,000 117 and 78.
constexpr int kSoloLinks = 16384;

int link_blocks(long long E, long long V, bool alone) {
  const long long per = std::min<long long>(kLinkPer, 1 + E * V / kLinkFill + E / 65536);
  return alone ? 1 : (int)std::max<long long>(1, (E + kBlock * per - 1) / (kBlock * per));
}

__global__ __launch_bounds__(kBlock) void k_link_search(Links K, VarState* st, unsigned char* var_on,
                                                        tap_acc* part, unsigned* done, const int* err,
                                                        const FwParams* prm, int v0, int alone, int solo, int more) {
  constexpr int kWaves = kBlock / kWave;
  const int var = v0 + blockIdx.y, tid = threadIdx.x;
  if (more ? !st[var].need_more : (!var_on[var] || err[0] != 0)) {
    if (blockIdx.x == 0 && tid == 0) st[var].stepping = 0;
    return;
  }
  __shared__ tap_acc sh[kMergeGroups * kQ], sums[kQ];
  __shared__ int s_more, s_jnext;
  __shared__ double s_lambda;
  const size_t off = (size_t)var * K.E;
  const int nb = gridDim.x;
  auto window = [&](int jbase, bool first, int k0, int stride) {
    tap_acc acc[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) acc[q] = tap_acc{0.0, 0.0};
    const double lam0 = ldexp(1.0, -jbase);
    for (int k = k0; k < K.E; k += stride)
      if (K.present[off + k]) link_sums(acc, K, off + k, lam0, first);
    block_reduce_acc<kWaves>(acc, sh, sums);
  };
  window(more ? st[var].jnext : 0, !more, blockIdx.x * kBlock + tid, nb * kBlock);
  if (nb > 1 && !merge_blocks(sums, sh, part + (size_t)var * nb * kQ, &done[var])) return;
  VarState s{};                                              // (kept by wavefront 0)
  FwParams p{};
  if (tid < kWave) { s = st[var]; p = *prm; }
  for (int only_g = more;; only_g = 1) {
    if (tid < kWave) {
      decide_window(s, sums, only_g, p, var);
      if (tid == 0) {
        s_more = s.need_more;
        s_jnext = s.jnext;
        s_lambda = s.lambda;
      }
    }
    __syncthreads();
    if (!s_more || !solo) break;
    window(s_jnext, false, tid, kBlock);
  }
  if (alone)
    for (int k = tid; k < K.E; k += kBlock) step_link(K, var, k, s_lambda);
  if (tid == 0) {
    s.stepping = !alone && !s.need_more;
    st[var] = s;
    var_on[var] = (unsigned char)(s.active && !s.need_more);
  }
}

__global__ __launch_bounds__(kBlock) void k_link_step(Links K, const VarState* st, int v0) {
  const int var = v0 + blockIdx.y;
  if (!st[var].stepping) return;
  const double lambda = st[var].lambda;
  for (int k = blockIdx.x * kBlock + threadIdx.x; k < K.E; k += gridDim.x * kBlock) step_link(K, var, k, lambda);
}

// Per variant at the current volumes: out[2v] = VHT = sum x * c, out[2v+1]
// = the Beckmann objective (sum of the link cost integrals), compensated
// sums in a fixed order.
__global__ __launch_bounds__(kBlock) void k_totals(Links K, tap_acc* part, unsigned* done, double* out,
                                                   int v0) {
  const int var = v0 + blockIdx.y, nb = gridDim.x;
  tap_acc acc[kQ];
#pragma unroll
  for (int q = 0; q < kQ; ++q) acc[q] = tap_acc{0.0, 0.0};
  const size_t off = (size_t)var * K.E;
  for (int k = blockIdx.x * kBlock + threadIdx.x; k < K.E; k += nb * kBlock) {
    const size_t i = off + k;
    if (!K.present[i]) continue;
    tap_acc_add(&acc[0], K.x[i] * K.c[i]);
    tap_acc_add(&acc[1], tap_integral(K.t0[i], K.cap[i], K.B[i], K.pw[i], K.x[i]));
  }
  __shared__ tap_acc sh[kMergeGroups * kQ], sums[kQ];
  block_reduce_acc<kBlock / kWave>(acc, sh, sums);
  if (nb > 1 && !merge_blocks(sums, sh, part + (size_t)var * nb * kQ, &done[var])) return;
  if (threadIdx.x < 2) out[2 * var + threadIdx.x] = tap_acc_value(sums[threadIdx.x]);
}

// Opens an FW iteration (or a replay of several) in one launch: the error
// flag and the counters, and the loading's volumes (the step clears them
// for the iteration after it).
__global__ __launch_bounds__(kBlock) void k_iter_begin(int* err, unsigned long long* counters, double* y,
                                                       long long ny) {
  const long long i0 = (long long)blockIdx.x * kBlock + threadIdx.x;
  const long long stride = (long long)gridDim.x * kBlock;
  if (i0 < 4) err[i0] = 0;
  if (i0 < 16) counters[i0] = 0ull;
  for (long long i = i0; i < ny; i += stride) y[i] = 0.0;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

template <class T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
};

}  // namespace

constexpr int kStageSlots = 8;          // slabs of results in flight to the host

struct tapgpu_ctx {
  std::string err;
  hipStream_t stream = nullptr;
  int device = 0;
  // sizes
  int N = 0, E = 0, Z = 0, ft0 = 0, V = 1, Gv = 0, Galloc = 0;
  long long Pv = 0, P = 0;
  double total_demand = 0;
  // graph
  int *fw_off = nullptr, *fw_dst = nullptr, *rv_off = nullptr, *rv_src = nullptr,
      *rv_eid = nullptr, *tail = nullptr, *rvpos = nullptr;
  // link records per variant
  double *t0 = nullptr, *cap = nullptr, *B = nullptr, *pw = nullptr;
  unsigned char* present = nullptr;
  double *x = nullptr, *y = nullptr, *c = nullptr, *rvw = nullptr, *fww = nullptr;
  // the LDS kernel's mirrors of the graph and the costs
  double *rec = nullptr, *sellw = nullptr;
  int *recpos = nullptr, *sellpos = nullptr, *sell_ptr = nullptr;
  unsigned char* hrec = nullptr;      // the labels-in-HBM kernel's mirrors (alloc_hbm_mirrors)
  int hgroup = 2;                     // lanes per expanded node (with the records' size)
  int hvars = 0, hvars_max = INT_MAX; // variants they hold, and may hold
  HbmRecOf* hrec_of = nullptr;
  int hrec_n = 0;
  uint2* hsell_id = nullptr;
  double* hsellw = nullptr;
  int* hplace = nullptr;              // [N] place of a node | [N] node of a place | slices
  long long hsell_n = 0;
  unsigned* sell_id = nullptr;
  long long sell_n = 0;
  bool mirrors_stale = false;         // not kept since the last lanes loading
  // origin-major demand (per-origin workgroups)
  long long* od_start = nullptr;
  int* od_dest = nullptr;
  double* od_val = nullptr;
  // strategy: 0 auto, 1 node-major sweeps, 2 one origin per workgroup (LDS)
  int strategy = 0;
  int chase = -1;                     // LDS path: chained expansions (-1: tune)
  int lds_block = -1;                 // LDS path: workgroup size (-1: tune)
  // LDS loadings dispatch origins longest first: the first loading records
  // each origin's relaxation rounds, later ones launch in that order
  int* d_origin_work = nullptr;          // [Z] rounds per origin
  int* d_hbm_next = nullptr;          // item counter of a labels-in-HBM loading
  int* d_origin_order = nullptr;         // [Z] origins by decreasing rounds
  bool origin_recorded = false, origin_order_ready = false;
  std::vector<int> h_origin_order;       // its host copy (the upload's source)
  bool qcap_auto = true;              // LDS path: queue size picked with the workgroup size
  int split = 0;                      // LDS path: origins per variant run by the HBM kernel
                                      // alongside it (-1: tune, 0: none)
  hipStream_t stream2 = nullptr;      // second queue for that co-running kernel
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  bool hbm_ok = false;                // labels-in-HBM path: bitmaps fit LDS
  size_t hbm_lds = 0;
  int hbm_grid = 0;                   // persistent workgroups
  double delta_mult = -1;             // bucket width / mean free-flow time (-1: tune)
  double mean_t0 = 1;                 // mean free-flow time of variant 0's links
  unsigned long long* h_dist = nullptr;
  int *h_pred = nullptr, *h_ptail = nullptr;
  int clock_khz = 0;                  // device wall clock
  bool labels_ready = false;          // node-major buffers allocated
  std::vector<double> h_odc;          // demand by (zone row, column), host copy
  std::vector<long long> h_od_start;  // origin-major demand, host copy (input order)
  std::vector<int> h_od_dest;
  std::vector<double> h_od_val;
  std::vector<int> h_tail;            // tail node of each link (0-based)
  std::vector<int> h_head;            // head node of each link (0-based)
  bool lds_ok = false;
  size_t lds_bytes = 0;
  int qcap = 0;                       // LDS frontier queue entries in use (per buffer)
  int qcap_max = 0;                   // entries the LDS allocation holds
  int hqcap = 0;                      // labels-in-HBM kernel: queue entries in use (per buffer)
  int hqcap_max = 0;                  // entries its LDS allocation holds
  // labels
  double* dist = nullptr;
  int *pred = nullptr, *pend = nullptr, *col_src = nullptr, *grp_var = nullptr;
  int *stamp = nullptr, *flags = nullptr;
  unsigned long long* counters = nullptr;
  int flags_cap = 0;
  int tag = 0;
  std::vector<int> zone_order;   // column -> zone (landmark order)
  // loading
  double *odc = nullptr, *ypart = nullptr;
  int* err_dev = nullptr;
  // FW state
  unsigned char* var_on = nullptr;
  VarState* st = nullptr;
  tap_acc* part = nullptr;            // [V][link_blocks][kQ] sums of the line search's blocks
  unsigned* done = nullptr;           // [V] its blocks that have finished
  double* vht = nullptr;              // [2V] VHT, objective at the current volumes
  FwParams* prm = nullptr;            // the fw_run call's limits and trace
  // captured iteration graphs (replayed while profiling is off):
  // g_iter = iteration begin + per-origin loading + link passes + readback,
  // g_link = link passes + readback (for the lanes path)
  bool graphs = true;
  int link_mode = 0;                  // link passes: 0 by size, 1 one workgroup per variant, 2 multi-block
  int line_window = kJ;               // step sizes per line-search window
  int g_link_mode = 0;                // the mode g_link was captured with
  int graph_iters = 0;                // iterations per whole-iteration replay (0: from the iteration time)
  double last_iter_ms = 0;            // wall time of the last iteration (per iteration of a replay)
  hipGraphExec_t g_iter = nullptr, g_link = nullptr;
  long long g_iter_key[6] = {-1, -1, -1, -1, -1, -1};
  int64_t graph_launches = 0;
  tapgpu_iter* trace = nullptr;
  int trace_cap = 0;
  bool initialised = false;
  // pinned host scratch
  int* h_int = nullptr;
  // results on their way to the caller's arrays (tapstage.inc)
  char* stage_dev = nullptr;
  size_t stage_dev_bytes = 0;
  char* stage_pin = nullptr;
  size_t stage_pin_bytes = 0;
  hipEvent_t stage_ev[kStageSlots] = {};
  unsigned char* aon_on = nullptr;    // [V] the variant that an all-or-nothing call loads
  // pinned readback of one FW iteration: error flag, origin-kernel
  // counters, variant states and flags (one synchronisation per iteration)
  int* pin_err = nullptr;                   // [4]
  unsigned long long* pin_cnt = nullptr;    // [16]
  VarState* pin_st = nullptr;               // [V]
  unsigned char* pin_on = nullptr;          // [V]
  void* pin_block = nullptr;
  // loading whose counters and error flag are read at the next
  // synchronisation instead of right after the launch
  bool defer_origin = false;
  bool origin_pending = false;
  int pending_Vn = 0;
  // the volumes, error flag and counters of the next loading were cleared
  // by k_iter_begin (the loading skips its own clears)
  bool pre_cleared = false;
  // error flag, counters, variant states and flags: one device block laid
  // out like pin_block, read back with one copy
  unsigned char* iter_dev = nullptr;
  size_t iter_bytes = 0;
  // lanes kernel (batched loading, variants in wavefront lanes)
  int lanes_min = 0;                  // active variants needed to use it (0: never)
  bool lanes_auto = true;             // lanes_min is the default
  int cus = 0;                        // compute units of the device
  bool tiny_ok = false;               // the one-workgroup kernel holds this network, and is the faster one
  bool lanes_ok = false;              // its LDS (bitmaps + queues) fits
  int lanes_qcap = 0;                 // LDS frontier queue entries per round
  int lanes_qcap_max = 0;             // entries its LDS allocation holds
  double lanes_delta_mult = -1;       // bucket width / mean free-flow time (-1: tune)
  size_t lanes_lds = 0;
  int lanes_grid = 0;                 // persistent workgroups (rows allocated)
  int lanes_grid_max = 0;             // resident workgroups on this device
  unsigned long long *l_dist = nullptr, *l_memo = nullptr;   // [grid][N][64]
  double *l_W = nullptr, *l_Y = nullptr;                     // [groups][E][64]
  int* l_lane_var = nullptr;          // [groups * 64]
  std::vector<int> h_lane_var;        // its host copy (as uploaded)
  unsigned l_stamp = 1;               // stamp of the next task's memo entries
  unsigned* l_stamp_dev = nullptr;    // its device copy, read by the kernel
  int* l_next = nullptr;              // task counter of a lanes launch
  bool capturing = false;             // launches are being recorded into a graph
  // stats
  tapgpu_stats stats{};
  bool profiling = false;
  hipEvent_t ev[2 * 8] = {};
  std::vector<void*> allocs;
  unsigned char* block_at = nullptr;  // balloc: the rest of the current block
  size_t block_left = 0;

  int fail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    err = buf;
    return code;
  }
};

namespace {

thread_local std::string g_create_error;   // message of this thread's last failed create

#define HIPCHK(ctx, call)                                                               \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess)                                                               \
      return (ctx)->fail(TAPGPU_E_HIP, "%s failed: %s", #call, hipGetErrorString(e_));  \
  } while (0)

template <class T>
int dalloc(tapgpu_ctx* ctx, T** p, size_t n) {
  *p = nullptr;
  if (n == 0) n = 1;
  hipError_t e = hipMalloc((void**)p, n * sizeof(T));
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return ctx->fail(TAPGPU_E_NOMEM, "hipMalloc of %zu bytes failed: %s", n * sizeof(T),
                     hipGetErrorString(e));
  }
  ctx->allocs.push_back(*p);
  return TAPGPU_OK;
}

// dalloc for the arrays a context keeps for life: carved out of blocks, so
// that creating a small context costs a few device allocations.
template <class T>
int balloc(tapgpu_ctx* ctx, T** p, size_t n) {
  constexpr size_t kBlockBytes = 4ull << 20;
  const size_t bytes = (std::max<size_t>(n, 1) * sizeof(T) + 255) & ~(size_t)255;
  *p = nullptr;
  if (bytes > ctx->block_left) {
    unsigned char* b = nullptr;
    if (int rc = dalloc(ctx, &b, std::max(bytes, kBlockBytes))) return rc;
    if (bytes >= kBlockBytes) {                  // (a block of its own)
      *p = (T*)b;
      return TAPGPU_OK;
    }
    ctx->block_at = b;
    ctx->block_left = kBlockBytes;
  }
  *p = (T*)ctx->block_at;
  ctx->block_at += bytes;
  ctx->block_left -= bytes;
  return TAPGPU_OK;
}

void dfree(tapgpu_ctx* ctx, void* p) {
  if (!p) return;
  ctx->allocs.erase(std::remove(ctx->allocs.begin(), ctx->allocs.end(), p), ctx->allocs.end());
  (void)hipFree(p);
}

template <class T>
int upload(tapgpu_ctx* ctx, T* d, const T* h, size_t n) {
  if (n == 0) return TAPGPU_OK;
  HIPCHK(ctx, hipMemcpyAsync(d, h, n * sizeof(T), hipMemcpyHostToDevice, ctx->stream));
  return TAPGPU_OK;
}

int grid_for(long long waves) {
  long long b = (waves + kWavesPerBlock - 1) / kWavesPerBlock;
  if (b < 1) b = 1;
  if (b > 8192) b = 8192;
  return (int)b;
}

constexpr int kSweepBlocks = 2048;
constexpr int kCheckEvery = 8;

Graph make_graph(tapgpu_ctx* c) {
  return Graph{c->N, c->E, c->ft0, c->fw_off, c->fw_dst, c->rv_off, c->rv_src, c->rv_eid, c->tail};
}

Labels make_labels(tapgpu_ctx* c, const int* col_src, const int* grp_var,
                   const unsigned char* var_on) {
  return Labels{c->dist, c->pred, c->pend, c->P, c->Galloc, col_src, grp_var, var_on, c->rvw};
}

// Without `mirrors` the passes do not keep the LDS kernel's copies of the
// costs (batches on the lanes kernel, where they would double the writes of
// a step); launch_lds brings them up to date when it needs them.
Links make_links(tapgpu_ctx* c, bool mirrors = true) {
  if (!mirrors) {
    c->mirrors_stale = c->mirrors_stale || c->rec;
    Links K = make_links(c);
    K.rec = nullptr;
    return K;
  }
  return Links{c->E, c->V, c->t0, c->cap, c->B, c->pw, c->present, c->rvpos,
               c->x, c->y, c->c, c->rvw, c->fww, c->rec, c->sellw, c->recpos, c->sellpos,
               (long long)c->N * kRecDoubles, c->sell_n};
}

// Round loop shared by the sweeps and the loading levels: launch
// kCheckEvery rounds, then read whether the next round has work.
template <class Launch>
int run_rounds(tapgpu_ctx* c, Launch launch, int64_t* rounds_out, double* kernel_ms,
               int64_t* launches) {
  int r = 0;
  for (;;) {
    if (r + kCheckEvery + 2 >= c->flags_cap)
      return c->fail(TAPGPU_E_LIMIT, "worklist did not drain in %d rounds", r);
    for (int k = 0; k < kCheckEvery; ++k, ++r) {
      if (c->profiling) HIPCHK(c, hipEventRecord(c->ev[2 * k], c->stream));
      launch(r, c->tag + r, c->tag + r + 1);
      if (c->profiling) HIPCHK(c, hipEventRecord(c->ev[2 * k + 1], c->stream));
    }
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipMemcpyAsync(c->h_int, c->flags + r - kCheckEvery + 1, sizeof(int) * kCheckEvery,
                             hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (c->profiling) {
      // rounds without work still launch; count every launch that was timed
      for (int k = 0; k < kCheckEvery; ++k) {
        float ms = 0.f;
        HIPCHK(c, hipEventElapsedTime(&ms, c->ev[2 * k], c->ev[2 * k + 1]));
        *kernel_ms += ms;
        *launches += 1;
      }
    }
    if (c->h_int[kCheckEvery - 1] == 0) {
      if (rounds_out) {
        int last = r - kCheckEvery;
        for (int k = 0; k < kCheckEvery; ++k)
          if (c->h_int[k]) last = r - kCheckEvery + 1 + k;
        *rounds_out += last + 1;
      }
      break;
    }
  }
  c->tag += r + 2;
  return TAPGPU_OK;
}

// tags are compared for equality with stamp[]; restart them long before
// 32-bit overflow
int maybe_reset_tags(tapgpu_ctx* c) {
  if (c->tag < 2000000000) return TAPGPU_OK;
  HIPCHK(c, hipMemsetAsync(c->stamp, 0xFF, sizeof(int) * (size_t)c->N * c->Galloc, c->stream));
  c->tag = 0;
  return TAPGPU_OK;
}

int scan_blocks(tapgpu_ctx* c, int Gn) {
  return (int)(((long long)c->N * Gn + kBlock - 1) / kBlock);
}

int read_counters(tapgpu_ctx* c, int64_t* a, int64_t* b, int64_t* d, int64_t* e) {
  unsigned long long h[4];
  HIPCHK(c, hipMemcpyAsync(h, c->counters, sizeof h, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (a) *a += (int64_t)h[0];
  if (b) *b += (int64_t)h[1];
  if (d) *d += (int64_t)h[2];
  if (e) *e += (int64_t)h[3];
  return TAPGPU_OK;
}

// Node-major buffers of the multi-origin sweep path, allocated on first use
// (the one-origin-per-workgroup path never needs them).
int ensure_labels(tapgpu_ctx* c) {
  if (c->labels_ready) return TAPGPU_OK;
  const size_t NP = (size_t)c->N * c->P;
  int rc;
  if ((rc = dalloc(c, &c->dist, NP))) return rc;
  if ((rc = dalloc(c, &c->pred, NP))) return rc;
  if ((rc = dalloc(c, &c->pend, NP))) return rc;
  if ((rc = dalloc(c, &c->stamp, (size_t)c->N * c->Galloc))) return rc;
  if ((rc = dalloc(c, &c->odc, c->h_odc.size()))) return rc;
  if ((rc = dalloc(c, &c->ypart, (size_t)c->Galloc * c->E))) return rc;
  if ((rc = upload(c, c->odc, c->h_odc.data(), c->h_odc.size()))) return rc;
  HIPCHK(c, hipMemsetAsync(c->stamp, 0xFF, sizeof(int) * (size_t)c->N * c->Galloc, c->stream));
  HIPCHK(c, hipMemsetAsync(c->ypart, 0, sizeof(double) * (size_t)c->Galloc * c->E, c->stream));
  c->labels_ready = true;
  return TAPGPU_OK;
}

// Shortest paths for groups [g0, g0+Gn).
int sssp_groups(tapgpu_ctx* c, int g0, int Gn, const int* col_src, const int* grp_var,
                const unsigned char* var_on) {
  int rc = ensure_labels(c);
  if (rc) return rc;
  rc = maybe_reset_tags(c);
  if (rc) return rc;
  auto t0 = std::chrono::steady_clock::now();
  Graph G = make_graph(c);
  Labels L = make_labels(c, col_src, grp_var, var_on);
  Frontier F{c->stamp, c->flags, c->counters};
  HIPCHK(c, hipMemsetAsync(c->flags, 0, sizeof(int) * c->flags_cap, c->stream));
  HIPCHK(c, hipMemsetAsync(c->counters, 0, sizeof(unsigned long long) * 4, c->stream));
  hipLaunchKernelGGL(k_fill_labels, dim3(grid_for((long long)c->N * Gn)), dim3(kBlock), 0,
                     c->stream, G, L, g0, Gn);
  hipLaunchKernelGGL(k_sssp_seed, dim3((Gn + kWavesPerBlock - 1) / kWavesPerBlock), dim3(kBlock), 0,
                     c->stream, G, L, F, g0, Gn, c->tag);
  const int nb = scan_blocks(c, Gn);
  rc = run_rounds(
      c,
      [&](int r, int tag, int tag_next) {
        hipLaunchKernelGGL(k_sssp_sweep, dim3(nb), dim3(kBlock), 0, c->stream, G, L, F, g0, Gn, r,
                           tag, tag_next);
      },
      &c->stats.sssp_sweeps, &c->stats.sweep_kernel_ms, &c->stats.sweep_launches);
  if (rc) return rc;
  rc = read_counters(c, &c->stats.sssp_items, &c->stats.sssp_inlinks, &c->stats.sssp_updates,
                     &c->stats.sssp_outlinks);
  c->stats.sssp_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return rc;
}

// Loading for groups [g0, g0+Gn) of variants [v0, v0+Vn) into y.  With
// check_tree the predecessor links came from the caller: lanes that never
// drained (a cycle) are reported as TAPGPU_E_ARG.
int aon_groups(tapgpu_ctx* c, int g0, int Gn, int v0, int Vn, const unsigned char* var_on,
               bool check_tree = false) {
  int rc = ensure_labels(c);
  if (rc) return rc;
  rc = maybe_reset_tags(c);
  if (rc) return rc;
  auto t0 = std::chrono::steady_clock::now();
  Graph G = make_graph(c);
  Labels L = make_labels(c, c->col_src, c->grp_var, var_on);
  Loading A{c->odc, c->Pv, c->Z, c->ypart, c->err_dev};
  Frontier F{c->stamp, c->flags, c->counters};
  HIPCHK(c, hipMemsetAsync(c->flags, 0, sizeof(int) * c->flags_cap, c->stream));
  HIPCHK(c, hipMemsetAsync(c->counters, 0, sizeof(unsigned long long) * 4, c->stream));
  HIPCHK(c, hipMemsetAsync(c->err_dev, 0, sizeof(int) * 3, c->stream));
  hipLaunchKernelGGL(k_aon_init, dim3(grid_for((long long)c->N * Gn)), dim3(kBlock), 0, c->stream,
                     G, L, A, F, g0, Gn, c->tag);
  const int nb = scan_blocks(c, Gn);
  rc = run_rounds(
      c,
      [&](int r, int tag, int tag_next) {
        hipLaunchKernelGGL(k_aon_level, dim3(nb), dim3(kBlock), 0, c->stream, G, L, A, F, g0, Gn,
                           r, tag, tag_next);
      },
      &c->stats.aon_levels, &c->stats.level_kernel_ms, &c->stats.level_launches);
  if (rc) return rc;
  if ((rc = read_counters(c, &c->stats.aon_items, &c->stats.aon_lanes, nullptr, nullptr))) return rc;
  if (check_tree) {
    hipLaunchKernelGGL(k_aon_check, dim3(grid_for((long long)c->N * Gn)), dim3(kBlock), 0,
                       c->stream, G, L, A, g0, Gn);
    HIPCHK(c, hipGetLastError());
  }
  int herr[3];
  HIPCHK(c, hipMemcpyAsync(herr, c->err_dev, sizeof herr, hipMemcpyDeviceToHost, c->stream));
  hipLaunchKernelGGL(k_aon_reduce, dim3(grid_for((long long)c->E * Vn / kWave + 1)), dim3(kBlock), 0,
                     c->stream, c->E, c->Gv, v0, Vn, var_on, c->ypart, c->y);
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->stats.aon_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  if (herr[0] == 4)
    return c->fail(TAPGPU_E_ARG, "predecessor links do not form a tree (origin %d, node %d)",
                   herr[1] + 1, herr[2] + 1);
  if (herr[0])
    return c->fail(TAPGPU_E_NOPATH, "no path from %d to %d", herr[1] + 1, herr[2] + 1);
  return TAPGPU_OK;
}

bool use_lds(tapgpu_ctx* c) {
  return c->lds_ok && (c->strategy == 0 || c->strategy == 2);
}

// auto: labels in LDS where they fit, else labels in HBM
bool use_hbm(tapgpu_ctx* c) {
  return c->hbm_ok && (c->strategy == 3 || (c->strategy == 0 && !c->lds_ok));
}

OriginArgs make_origin_args(tapgpu_ctx* c, const unsigned char* var_on) {
  OriginArgs A{};
  A.N = c->N; A.E = c->E; A.ft0 = c->ft0; A.Z = c->Z;
  A.fw_off = c->fw_off; A.fw_dst = c->fw_dst; A.rv_off = c->rv_off; A.rv_src = c->rv_src;
  A.rv_eid = c->rv_eid; A.tail = c->tail; A.fww = c->fww; A.rvw = c->rvw;
  A.rec = c->rec; A.sellw = c->sellw; A.sell_id = c->sell_id; A.sell_ptr = c->sell_ptr;
  A.sell_n = c->sell_n;
  A.hrec = c->hrec; A.hrec_of = c->hrec_of; A.hrec_n = c->hrec_n; A.hsell_id = c->hsell_id; A.hsellw = c->hsellw; A.hsell_n = c->hsell_n;
  A.place = c->hplace; A.node = c->hplace + c->N; A.hsell_ptr = c->hplace + 2 * (size_t)c->N;
  A.od_start = c->od_start; A.od_dest = c->od_dest; A.od_val = c->od_val;
  A.var_on = var_on; A.y = c->y; A.err = c->err_dev; A.counters = c->counters;
  A.chase = c->chase >= 0 ? c->chase : kDefaultChase;
  A.qcap = c->qcap;
  A.hqcap = std::max(c->hqcap, 1);            // (with 1 a search goes on with bitmaps from its first nodes)
  A.h_dist = c->h_dist; A.h_pred = c->h_pred; A.h_ptail = c->h_ptail;
  // (negative: a width to start from; before tuning, or without buckets)
  A.delta = c->delta_mult > 0 ? c->delta_mult * c->mean_t0 : c->mean_t0 > 0 ? -4.0 * c->mean_t0 : -1.0;
  A.z0 = 0;
  A.zn = c->Z;
  return A;
}

// The cost arrays of A moved to variant v (the kernels' variant 0; the
// labels-in-HBM kernel's mirrors are those of a launch's variants).
void advance_variant(tapgpu_ctx* c, OriginArgs& A, int64_t v) {
  A.fww += (size_t)v * c->E;
  A.rvw += (size_t)v * c->E;
  if (c->rec) {
    A.rec += (size_t)v * c->N * kRecDoubles;
    A.sellw += (size_t)v * c->sell_n;
  }
}

// Arguments of a loading of the variants from v on.
OriginArgs variant_args(tapgpu_ctx* c, const unsigned char* var_on, int v) {
  OriginArgs A = make_origin_args(c, var_on ? var_on + v : nullptr);
  advance_variant(c, A, v);
  A.y += (size_t)v * c->E;
  return A;
}

// (before any capture too: a replay takes the mirrors as the passes keep them)
void refresh_mirrors(tapgpu_ctx* c) {
  if (!c->mirrors_stale || c->capturing) return;
  hipLaunchKernelGGL(k_mirror_costs, dim3(grid_for((long long)c->E * c->V / kWave + 1)), dim3(kBlock), 0,
                     c->stream, make_links(c));
  c->mirrors_stale = false;
}

// Workgroup size the LDS kernel runs with (before tuning: kLdsBlock).
int lds_threads(const tapgpu_ctx* c) { return c->lds_block > 0 ? c->lds_block : kLdsBlock; }

// One launch of the LDS kernel at the context's workgroup size, with the
// LDS its queue size needs (a smaller queue leaves room for more
// workgroups per CU).
void launch_lds(tapgpu_ctx* c, dim3 grid, hipStream_t st, const OriginArgs& A, int load) {
  refresh_mirrors(c);
  const size_t sh = origin_lds_bytes(c->N, A.qcap);
  switch (lds_threads(c)) {
    case 256: hipLaunchKernelGGL(k_origin_lds<256>, grid, dim3(256), sh, st, A, load); break;
    case 512: hipLaunchKernelGGL(k_origin_lds<512>, grid, dim3(512), sh, st, A, load); break;
    default: hipLaunchKernelGGL(k_origin_lds<1024>, grid, dim3(1024), sh, st, A, load); break;
  }
}

// Shortest paths + loading for variants [v0, v0+Vn) with one workgroup per
// (origin, variant); y of those variants is overwritten.
//
// Worklist schedule tuning: the first loading on a context with chase < 0
// times one full launch for each candidate chain length and keeps the
// fastest (the result is the same for every candidate; the last launch
// below, with the chosen value, is the one whose volumes are kept).
constexpr int kChaseCandidates[] = {0, 2, 4, 8, 16, 32};
constexpr int kTuneBlocks = 4096;              // workgroups of a tuning launch on a batch

int ensure_hbm(tapgpu_ctx* c, int Vn);
void launch_hbm_kernel(tapgpu_ctx* c, const OriginArgs& A, int Vn, int load, int items, int blocks, hipStream_t st,
                       bool mirrors = true);

// Per-origin round counts of the recording loading (zeroed: origins a
// loading skips keep 0 and go last).
int ensure_origin_work(tapgpu_ctx* c) {
  int rc = dalloc(c, &c->d_origin_work, (size_t)c->Z);
  if (rc) return rc;
  HIPCHK(c, hipMemsetAsync(c->d_origin_work, 0, sizeof(int) * (size_t)c->Z, c->stream));
  return TAPGPU_OK;
}

// One loading launch of the LDS path.  With split > 0 the last `split`
// origins of every variant go to the labels-in-HBM kernel on a second queue,
// running on the same CUs at the same time: the LDS kernel's workgroup takes
// most of a CU's LDS but only half of its wave slots, and the HBM kernel's
// workgroups (a few KB of LDS each) fill the rest.  Both add integer flows
// to y with atomics, so the split changes no result.
int launch_origin(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on, float* ms) {
  if (!c->pre_cleared)
    HIPCHK(c, hipMemsetAsync(c->y + (size_t)v0 * c->E, 0, sizeof(double) * (size_t)Vn * c->E, c->stream));
  if (c->Z > 0) {
    const int zh = (c->hbm_ok && c->split > 0) ? std::min(c->split, c->Z - 1) : 0;
    const int zl = c->Z - zh;
    if (zh > 0)
      if (int rc = ensure_hbm(c, Vn)) return rc;
    OriginArgs A = variant_args(c, var_on, v0);
    if (zh == 0) {
      if (c->origin_order_ready) {
        A.src_list = c->d_origin_order;
      } else if (!c->capturing && c->Z > 1) {
        if (!c->d_origin_work) {
          int rc = ensure_origin_work(c);
          if (rc) return rc;
        }
        A.work = c->d_origin_work;
        c->origin_recorded = true;
      }
    }
    if (ms) HIPCHK(c, hipEventRecord(c->ev[0], c->stream));
    if (zh > 0) {
      HIPCHK(c, hipEventRecord(c->ev_fork, c->stream));
      HIPCHK(c, hipStreamWaitEvent(c->stream2, c->ev_fork, 0));
      for (int v = 0; v < Vn; v += c->hvars) {
        const int n = std::min(c->hvars, Vn - v), items = zh * n;
        OriginArgs B = variant_args(c, var_on, v0 + v);
        B.z0 = zl;
        B.zn = zh;
        launch_hbm_kernel(c, B, n, 1, items, c->hbm_grid, c->stream2);
        HIPCHK(c, hipGetLastError());
      }
      HIPCHK(c, hipEventRecord(c->ev_join, c->stream2));
    }
    for (int v = 0; v < Vn; v += kGridVariants) {
      OriginArgs B = variant_args(c, var_on, v0 + v);
      B.src_list = A.src_list;
      B.work = v == 0 ? A.work : nullptr;
      launch_lds(c, dim3(zl, std::min(Vn - v, kGridVariants)), c->stream, B, 1);
    }
    HIPCHK(c, hipGetLastError());
    if (zh > 0) HIPCHK(c, hipStreamWaitEvent(c->stream, c->ev_join, 0));
    if (ms) HIPCHK(c, hipEventRecord(c->ev[1], c->stream));
    if (ms) {
      HIPCHK(c, hipEventSynchronize(c->ev[1]));
      HIPCHK(c, hipEventElapsedTime(ms, c->ev[0], c->ev[1]));
    }
  }
  return TAPGPU_OK;
}

// Share of origins for the co-running HBM kernel: each candidate (as a
// fraction of Z) is timed on the full launch; the fastest is kept.
constexpr int kSplitCandidates[] = {0, 10, 15, 20, 25, 33};   // percent of Z

int tune_split(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on) {
  if (!c->hbm_ok || c->Z < 8) {
    c->split = 0;
    return TAPGPU_OK;
  }
  if (!c->ev[0])
    for (auto& e : c->ev) HIPCHK(c, hipEventCreate(&e));
  float best_ms = 0.f;
  int best = 0;
  for (int pct : kSplitCandidates) {
    c->split = (int)((long long)c->Z * pct / 100);
    float ms = 0.f;
    int rc = launch_origin(c, v0, Vn, var_on, &ms);
    if (rc) return rc;
    int herr = 0;
    HIPCHK(c, hipMemcpyAsync(&herr, c->err_dev, sizeof herr, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (herr) break;
    if (best_ms == 0.f || ms < best_ms) { best_ms = ms; best = c->split; }
  }
  c->split = best;
  c->stats.origin_tune_ms += best_ms;
  return TAPGPU_OK;
}

int tune_chase(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on) {
  if (!c->ev[0])
    for (auto& e : c->ev) HIPCHK(c, hipEventCreate(&e));
  float best_ms = 0.f;
  int best = kDefaultChase;
  HIPCHK(c, hipMemsetAsync(c->counters, 0, sizeof(unsigned long long) * 16, c->stream));
  for (int k : kChaseCandidates) {
    c->chase = k;
    float ms = 0.f;
    int rc = launch_origin(c, v0, Vn, var_on, &ms);
    if (rc) return rc;
    int herr = 0;
    unsigned long long scans = 0;
    HIPCHK(c, hipMemcpyAsync(&herr, c->err_dev, sizeof herr, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipMemcpyAsync(&scans, c->counters + 12, sizeof scans, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (herr) break;                    // reported by the caller's launch
    if (best_ms == 0.f || ms < best_ms) { best_ms = ms; best = k; }
    if (!scans) break;                  // every round ran from the queue: the length plays no part
  }
  c->chase = best;
  c->stats.origin_tune_ms += best_ms;
  return TAPGPU_OK;
}

// Workgroup size and queue size of the LDS kernel: every allowed size
// (kLdsPerThread nodes per thread at most) with, unless the queue size was
// set, the full queue and two shorter ones (less LDS per workgroup, so more
// workgroups per CU), each timed on one launch over the variants given (of a
// batch, enough of them to fill the chip); the fastest pair is kept.  Results
// do not depend on them.
int tune_lds_shape(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on) {
  if (!c->ev[0])
    for (auto& e : c->ev) HIPCHK(c, hipEventCreate(&e));
  std::vector<int> qs{c->qcap};
  if (c->qcap_auto) {
    qs = {c->qcap_max};
    for (int q : {1024, 256})
      if (q < c->qcap_max) qs.push_back(q);
  }
  float best_ms = 0.f;
  int best_b = kLdsBlock, best_q = c->qcap;
  for (int b : kLdsBlocks) {
    if (c->N > kLdsPerThread * b) continue;
    for (int q : qs) {
      c->lds_block = b;
      c->qcap = q;
      float ms = 0.f;
      int rc = launch_origin(c, v0, Vn, var_on, &ms);
      if (rc) return rc;
      int herr = 0;
      HIPCHK(c, hipMemcpyAsync(&herr, c->err_dev, sizeof herr, hipMemcpyDeviceToHost, c->stream));
      HIPCHK(c, hipStreamSynchronize(c->stream));
      if (herr) {                       // reported by the caller's launch
        c->lds_block = best_b;
        c->qcap = best_q;
        return TAPGPU_OK;
      }
      if (best_ms == 0.f || ms < best_ms) { best_ms = ms; best_b = b; best_q = q; }
    }
  }
  c->lds_block = best_b;
  c->qcap = best_q;
  c->stats.origin_tune_ms += best_ms;
  return TAPGPU_OK;
}

int absorb_origin(tapgpu_ctx* c, const int* herr, const unsigned long long* hc, int Vn,
                  std::chrono::steady_clock::time_point t0);

// Reads the error flag and counters of an origin-kernel launch into stats:
// now, or (defer_origin) from the pinned copy of the iteration block that
// the caller makes, absorbed by absorb_pending after its synchronisation.
int finish_origin(tapgpu_ctx* c, int Vn, std::chrono::steady_clock::time_point t0) {
  if (c->defer_origin) {            // read back with the iteration's block copy
    c->origin_pending = true;
    c->pending_Vn = Vn;
    return TAPGPU_OK;
  }
  int herr[3];
  unsigned long long hc[16];
  HIPCHK(c, hipMemcpyAsync(herr, c->err_dev, sizeof herr, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(hc, c->counters, sizeof hc, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return absorb_origin(c, herr, hc, Vn, t0);
}

// The deferred readback of finish_origin, after the stream has synchronised.
int absorb_pending(tapgpu_ctx* c) {
  if (!c->origin_pending) return TAPGPU_OK;
  c->origin_pending = false;
  return absorb_origin(c, c->pin_err, c->pin_cnt, c->pending_Vn, std::chrono::steady_clock::now());
}

int absorb_origin(tapgpu_ctx* c, const int* herr, const unsigned long long* hc, int Vn,
                  std::chrono::steady_clock::time_point t0) {
  c->stats.origin_expansions += (int64_t)hc[0];
  c->stats.origin_scanned += (int64_t)hc[1];
  c->stats.origin_updates += (int64_t)hc[2];
  c->stats.origin_relax_rounds += (int64_t)hc[3];
  c->stats.origin_load_rounds += (int64_t)hc[4];
  c->stats.origin_loaded += (int64_t)hc[5];
  c->stats.origin_walk_steps += (int64_t)hc[6];
  c->stats.origin_deferred += (int64_t)hc[7];
  if (c->clock_khz > 0) {
    c->stats.origin_relax_ms += (double)hc[8] / c->clock_khz;
    c->stats.origin_pred_ms += (double)hc[9] / c->clock_khz;
    c->stats.origin_load_ms += (double)hc[10] / c->clock_khz;
  }
  if (c->profiling && c->Z > 0) {
    float ms = 0.f;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    c->stats.origin_kernel_ms += ms;
    c->stats.origin_launches += 1;
  }
  c->stats.origin_blocks += (int64_t)c->Z * Vn;
  c->stats.origin_chase = c->chase;
  c->stats.origin_block = use_lds(c) ? lds_threads(c) : 0;
  c->stats.origin_queue = use_lds(c) ? c->qcap : c->hqcap;
  c->stats.origin_split = c->split;
  c->stats.aon_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  if (herr[0] == 1)
    return c->fail(TAPGPU_E_NOPATH, "no path from %d to %d", herr[1] + 1, herr[2] + 1);
  if (herr[0] == 2)
    return c->fail(TAPGPU_E_LIMIT, "label-correcting rounds exceeded from origin %d (negative costs?)",
                   herr[1] + 1);
  if (herr[0] == 3)
    return c->fail(TAPGPU_E_LIMIT, "predecessor cycle in the tree of origin %d", herr[1] + 1);
  return TAPGPU_OK;
}

// After a loading that recorded each origin's relaxation rounds: the
// origins sorted by decreasing rounds (then id), the dispatch order of later
// LDS loadings.  The hardware starts workgroups in block order as slots
// free up, so the longest searches start first and the short ones fill the
// tail.  Results do not depend on the order.
int origin_order_update(tapgpu_ctx* c) {
  if (!c->origin_recorded || c->origin_order_ready || c->capturing) return TAPGPU_OK;
  std::vector<int> work(c->Z), order(c->Z);
  HIPCHK(c, hipMemcpyAsync(work.data(), c->d_origin_work, sizeof(int) * c->Z, hipMemcpyDeviceToHost,
                           c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  for (int z = 0; z < c->Z; ++z) order[z] = z;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return work[a] > work[b]; });
  int rc;
  if (!c->d_origin_order && (rc = dalloc(c, &c->d_origin_order, (size_t)c->Z))) return rc;
  if ((rc = upload(c, c->d_origin_order, order.data(), (size_t)c->Z))) return rc;
  c->h_origin_order = std::move(order);
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->origin_order_ready = true;
  return TAPGPU_OK;
}

int aon_lds(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on) {
  auto t0 = std::chrono::steady_clock::now();
  if (int rc = origin_order_update(c)) return rc;
  if (!c->pre_cleared) HIPCHK(c, hipMemsetAsync(c->err_dev, 0, sizeof(int) * 3, c->stream));
  // candidates run on as many variants as fill the chip several times over
  const int Vt = var_on ? Vn : (int)std::min<long long>(Vn, 1 + kTuneBlocks / std::max(c->Z, 1));
  if (c->lds_block < 0 && c->Z > 0) {
    // workgroup and queue size first, then the chain length, on the LDS
    // kernel alone
    const int keep = c->split;
    c->split = 0;
    int rc = tune_lds_shape(c, v0, Vt, var_on);
    c->split = keep;
    if (rc) return rc;
    HIPCHK(c, hipMemsetAsync(c->err_dev, 0, sizeof(int) * 3, c->stream));
  }
  if (c->chase < 0 && c->Z > 0) {
    const int keep = c->split;
    c->split = 0;
    int rc = tune_chase(c, v0, Vt, var_on);
    c->split = keep;
    if (rc) return rc;
    HIPCHK(c, hipMemsetAsync(c->err_dev, 0, sizeof(int) * 3, c->stream));
  }
  if (c->split < 0 && c->Z > 0) {
    int rc = tune_split(c, v0, Vn, var_on);
    if (rc) return rc;
    HIPCHK(c, hipMemsetAsync(c->err_dev, 0, sizeof(int) * 3, c->stream));
  }
  if (!c->pre_cleared)
    HIPCHK(c, hipMemsetAsync(c->counters, 0, sizeof(unsigned long long) * 16, c->stream));
  if (c->Z > 0) {
    if (c->profiling) HIPCHK(c, hipEventRecord(c->ev[0], c->stream));
    int rc = launch_origin(c, v0, Vn, var_on, nullptr);
    if (rc) return rc;
    if (c->profiling) HIPCHK(c, hipEventRecord(c->ev[1], c->stream));
  }
  return finish_origin(c, Vn, t0);
}

// Places of the nodes in the labels-in-HBM kernel's rows: zones first, as
// they are numbered; then, line by line, groups of through nodes grown from
// a node beside the last ones, each time by the node with the most links to
// the group.
void hbm_places(int N, int ft0, const std::vector<int>& off, const std::vector<int>& dst,
                const std::vector<int>& roff, const std::vector<int>& rsrc, int* place) {
  constexpr int kLine = 16;                            // labels in 128 bytes
  std::vector<char> done(N, 0);
  std::vector<int> beside, links(N, 0), group;
  size_t head = 0;
  int next = std::min(ft0, N), scan = next;
  for (int v = 0; v < next; ++v) { place[v] = v; done[v] = 1; }
  while (next < N) {
    int left = kLine - next % kLine;
    while (left > 0 && next < N) {
      while (head < beside.size() && done[beside[head]]) ++head;
      if (head == beside.size())
        while (done[scan]) ++scan;
      group.assign(1, head < beside.size() ? beside[head] : scan);
      while (!group.empty() && left > 0) {
        size_t best = 0;
        for (size_t i = 1; i < group.size(); ++i)
          if (links[group[i]] > links[group[best]]) best = i;
        const int v = group[best];
        group.erase(group.begin() + best);
        links[v] = 0;
        done[v] = 1;
        place[v] = next++;
        --left;
        auto grow = [&](int u) {
          if (u < ft0 || done[u]) return;
          if (links[u]++ == 0) group.push_back(u);
        };
        for (int k = off[v]; k < off[v + 1]; ++k) grow(dst[k]);
        for (int k = roff[v]; k < roff[v + 1]; ++k) grow(rsrc[k]);
      }
      for (int u : group) { links[u] = 0; beside.push_back(u); }
    }
  }
}

// The labels-in-HBM kernel's mirrors, of Vn variants or of as many as
// kHbmMirrorBytes hold: launches over more variants go by parts (58 variants
// of regional are 232,000 items, for 512 workgroups).  Those of one variant
// are made with the context where its labels do not fit LDS, since
// tapgpu_sssp_noalloc allocates nothing, otherwise when the kernel is chosen
// or first runs; a batch that only the lanes kernel loads holds no more (512
// variants of regional: 5 GB).  They grow before an iteration is captured.
constexpr size_t kHbmMirrorBytes = 512ull << 20;

int alloc_hbm_mirrors(tapgpu_ctx* c, int Vn) try {
  auto grow = [&]() -> int {
    const size_t recs = hrec_bytes(c->hgroup) * (size_t)c->hrec_n, each = recs + sizeof(double) * (size_t)c->hsell_n;
    const int most = std::min<int>(c->hvars_max, (int)std::max<size_t>(1, kHbmMirrorBytes / each));
    for (int n = std::min(Vn, most); n > c->hvars; n /= 2) {
      unsigned char* rec = nullptr;
      double* w = nullptr;
      int rc = dalloc(c, &rec, n * recs);
      if (!rc && (rc = dalloc(c, &w, (size_t)n * c->hsell_n))) dfree(c, rec);
      if (rc && (n == 1 || rc != TAPGPU_E_NOMEM)) return rc;
      if (rc) {                                        // with fewer at a time, then and later
        c->hvars_max = std::max(1, n / 2);
        continue;
      }
      HIPCHK(c, hipStreamSynchronize(c->stream));
      dfree(c, c->hrec);
      dfree(c, c->hsellw);
      c->hrec = rec;
      c->hsellw = w;
      c->hvars = n;
      break;
    }
    return TAPGPU_OK;
  };
  if (c->hvars) return grow();
  const int N = c->N, W = (N + kWave - 1) / kWave;
  std::vector<int> off(N + 1), dst(c->E), roff(N + 1), rsrc(c->E);
  auto get = [&](std::vector<int>& h, const int* d) {
    return hipMemcpyAsync(h.data(), d, sizeof(int) * h.size(), hipMemcpyDeviceToHost, c->stream);
  };
  HIPCHK(c, get(off, c->fw_off));
  HIPCHK(c, get(dst, c->fw_dst));
  HIPCHK(c, get(roff, c->rv_off));
  HIPCHK(c, get(rsrc, c->rv_src));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  std::vector<int> h(2 * (size_t)N + W + 1, 0);
  hbm_places(N, c->ft0, off, dst, roff, rsrc, h.data());
  for (int v = 0; v < N; ++v) h[(size_t)N + h[v]] = v;
  int* ptr = h.data() + 2 * (size_t)N;
  for (int v = c->ft0; v < N; ++v) {
    int n = 0;
    for (int k = roff[v]; k < roff[v + 1]; ++k) n += rsrc[k] != v && rsrc[k] >= c->ft0;
    int& rows = ptr[h[v] / kWave + 1];
    rows = std::max(rows, std::min(kSellWidth, n));
  }
  for (int i = 0; i < W; ++i) ptr[i + 1] = ptr[i] + ptr[i + 1] * kWave;
  c->hsell_n = ptr[W];
  // a node's records: the first at its place, further ones in a row behind
  // all places
  std::vector<HbmRecOf> of(N);
  auto counts = [&](int v, int k) { return dst[k] >= c->ft0 && dst[k] != v; };
  int large = 0;
  for (int v = 0; v < N; ++v) {
    int n = 0;
    for (int k = off[v]; k < off[v + 1]; ++k) n += counts(v, k);
    large += n > hrec_links(2) && n <= hrec_links(4);
  }
  c->hgroup = large > N / 2 ? 4 : 2;
  for (int i = 0; i < N; ++i) {
    const int v = h[(size_t)N + i], base = (int)of.size() - 1;
    int at = i, n = 0;
    of[i] = {off[v], off[v + 1], 0, i};
    for (int k = off[v]; k < off[v + 1]; ++k) {
      if (!counts(v, k) || n++ < hrec_links(c->hgroup)) continue;
      n = 1;
      of[at].end = k;
      at = (int)of.size();
      of.push_back({k, off[v + 1], 0, i});
    }
    const int m = (int)of.size() - 1 - base;           // records after the first
    for (int k = 0; k <= m; ++k)
      of[k ? base + k : i].more = (2 * k + 1 <= m ? base + 2 * k + 1 : 0) | (2 * k + 2 <= m ? kHrecTwo : 0) |
                                  (k < m ? kHrecRow : 0);
  }
  c->hrec_n = (int)of.size();
  int rc;
  if (!c->hplace && (rc = dalloc(c, &c->hplace, h.size()))) return rc;
  if (!c->hrec_of && (rc = dalloc(c, &c->hrec_of, of.size()))) return rc;
  if ((rc = upload(c, c->hrec_of, of.data(), of.size()))) return rc;
  if (!c->hsell_id && (rc = dalloc(c, &c->hsell_id, (size_t)c->hsell_n))) return rc;
  if ((rc = upload(c, c->hplace, h.data(), h.size()))) return rc;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return grow();
} catch (const std::bad_alloc&) {
  return c->fail(TAPGPU_E_NOMEM, "out of host memory for the node numbering");
}

// Before a launch of the labels-in-HBM kernel: the mirrors of Vn variants
// (A is advanced to the first, and hvars holds them).
void launch_hbm_mirrors(tapgpu_ctx* c, const OriginArgs& A, int Vn, hipStream_t st) {
  const int nodes = std::max((c->N + kWave - 1) / kWave * kWave, c->hrec_n);
  const dim3 grid((nodes + kBlock - 1) / kBlock, std::min(Vn, kGridVariants));
  uint2* id = const_cast<uint2*>(A.hsell_id);
  double* w = const_cast<double*>(A.hsellw);
  if (c->hgroup == 4)
    hipLaunchKernelGGL(k_hbm_mirrors<4>, grid, dim3(kBlock), 0, st, A, Vn, (HbmRec<4>*)c->hrec, id, w);
  else
    hipLaunchKernelGGL(k_hbm_mirrors<2>, grid, dim3(kBlock), 0, st, A, Vn, (HbmRec<2>*)c->hrec, id, w);
}

// The mirrors of Vn variants, then the kernel over `items` of theirs by at
// most `blocks` workgroups.
void launch_hbm_kernel(tapgpu_ctx* c, const OriginArgs& A, int Vn, int load, int items, int blocks, hipStream_t st,
                       bool mirrors) {
  if (mirrors) launch_hbm_mirrors(c, A, Vn, st);
  const dim3 grid(std::min(blocks, items));
  if (c->hgroup == 4)
    hipLaunchKernelGGL(k_origin_hbm<4>, grid, dim3(kHbmBlock), c->hbm_lds, st, A, load, items);
  else
    hipLaunchKernelGGL(k_origin_hbm<2>, grid, dim3(kHbmBlock), c->hbm_lds, st, A, load, items);
}

// Per-workgroup scratch rows of the labels-in-HBM kernel (allocated on
// first use: hbm_grid rows of N labels, predecessors and tails).
int ensure_hbm(tapgpu_ctx* c, int Vn) {
  if (int rc = alloc_hbm_mirrors(c, Vn)) return rc;
  if (c->h_dist) return TAPGPU_OK;
  const size_t n = (size_t)c->hbm_grid * c->N;
  int rc;
  if ((rc = dalloc(c, &c->d_hbm_next, 1))) return rc;
  if ((rc = dalloc(c, &c->h_dist, n))) return rc;
  if ((rc = dalloc(c, &c->h_pred, n))) return rc;
  if ((rc = dalloc(c, &c->h_ptail, n))) return rc;
  return TAPGPU_OK;
}

// Shortest paths + loading of variants [v0, v0+Vn) with the labels-in-HBM
// kernel (persistent grid over the Z * Vn (origin, variant) items).
//
// Bucket-width tuning: the first loading on a context with delta_mult < 0
// runs one wave of workgroups (the first hbm_grid items) for each candidate
// width, in units of the mean free-flow link time, and keeps the one with
// the smallest busy time summed over the workgroups; the full launch
// follows.  Results do not depend on the width.
// From narrow to wide, ending with the first that is clearly slower: a width
// that lists more nodes than the queues hold is many times slower.
constexpr double kDeltaCandidates[] = {1.0, 2.0, 4.0, 8.0, 16.0};
constexpr double kDeltaStop = 1.2;

int launch_hbm(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on, int items_cap,
               float* ms) {
  if (!c->pre_cleared)
    HIPCHK(c, hipMemsetAsync(c->y + (size_t)v0 * c->E, 0, sizeof(double) * (size_t)Vn * c->E, c->stream));
  if (c->Z == 0) return TAPGPU_OK;
  if (int rc = ensure_hbm(c, Vn)) return rc;    // (no allocation once made)
  int* work = nullptr;
  if (!c->origin_order_ready && !c->capturing && c->Z > 1) {
    if (!c->d_origin_work) {
      int rc = ensure_origin_work(c);
      if (rc) return rc;
    }
    work = c->d_origin_work;
    c->origin_recorded = true;
  }
  if (ms) HIPCHK(c, hipEventRecord(c->ev[0], c->stream));
  for (int v = 0; v < Vn && items_cap > 0; v += c->hvars) {
    const int n = std::min(c->hvars, Vn - v), items = std::min(c->Z * n, items_cap);
    items_cap -= items;
    OriginArgs A = variant_args(c, var_on, v0 + v);
    if (c->origin_order_ready) {
      A.order = c->d_origin_order;
      A.vn = n;
    }
    A.work = work;
    A.next = c->d_hbm_next;
    hipLaunchKernelGGL(k_zero_i32, dim3(1), dim3(1), 0, c->stream, c->d_hbm_next);
    launch_hbm_kernel(c, A, n, 1, items, c->hbm_grid, c->stream);
    HIPCHK(c, hipGetLastError());
  }
  if (ms) {
    HIPCHK(c, hipEventRecord(c->ev[1], c->stream));
    HIPCHK(c, hipEventSynchronize(c->ev[1]));
    HIPCHK(c, hipEventElapsedTime(ms, c->ev[0], c->ev[1]));
  }
  return TAPGPU_OK;
}

// Busy time of a tuning launch: the workgroups' phase clocks (relaxation,
// predecessors, loading), summed over its tasks.  At full occupancy the
// smallest sum is the highest throughput; one wave's wall time would be set
// by its slowest task alone.
int tuning_work(tapgpu_ctx* c, double* work, int* herr) {
  unsigned long long hc[16];
  HIPCHK(c, hipMemcpyAsync(hc, c->counters, sizeof hc, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(herr, c->err_dev, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  *work = (double)hc[8] + (double)hc[9] + (double)hc[10];
  return TAPGPU_OK;
}

int tune_delta(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on) {
  if (!c->ev[0])
    for (auto& e : c->ev) HIPCHK(c, hipEventCreate(&e));
  float best_ms = 0.f;
  double best = 4.0, best_work = 0.0;
  for (double m : kDeltaCandidates) {
    c->delta_mult = m;
    HIPCHK(c, hipMemsetAsync(c->counters, 0, sizeof(unsigned long long) * 16, c->stream));
    float ms = 0.f;
    int rc = launch_hbm(c, v0, Vn, var_on, c->hbm_grid, &ms);
    if (rc) return rc;
    int herr = 0;
    double work = 0.0;
    if ((rc = tuning_work(c, &work, &herr))) return rc;
    if (herr) break;
    if (best_work == 0.0 || work < best_work) { best_work = work; best_ms = ms; best = m; }
    if (work > kDeltaStop * best_work) break;
  }
  c->delta_mult = best;
  c->stats.origin_tune_ms += best_ms;
  HIPCHK(c, hipMemsetAsync(c->err_dev, 0, sizeof(int) * 3, c->stream));
  HIPCHK(c, hipMemsetAsync(c->counters, 0, sizeof(unsigned long long) * 16, c->stream));
  return TAPGPU_OK;
}

int aon_hbm(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on) {
  auto t0 = std::chrono::steady_clock::now();
  int rc = ensure_hbm(c, Vn);
  if (rc) return rc;
  if ((rc = origin_order_update(c))) return rc;
  if (!c->pre_cleared) HIPCHK(c, hipMemsetAsync(c->err_dev, 0, sizeof(int) * 3, c->stream));
  if (c->delta_mult < 0 && c->Z > 0 && (rc = tune_delta(c, v0, Vn, var_on))) return rc;
  if (!c->pre_cleared)
    HIPCHK(c, hipMemsetAsync(c->counters, 0, sizeof(unsigned long long) * 16, c->stream));
  if (c->profiling && c->Z > 0) HIPCHK(c, hipEventRecord(c->ev[0], c->stream));
  if ((rc = launch_hbm(c, v0, Vn, var_on, INT32_MAX, nullptr))) return rc;
  if (c->profiling && c->Z > 0) HIPCHK(c, hipEventRecord(c->ev[1], c->stream));
  c->stats.origin_delta = c->delta_mult;
  return finish_origin(c, Vn, t0);
}

#include "taplanes.inc"
#include "tapstage.inc"
#include "taptiny.inc"

// Whether the lanes kernel is the faster loading of n variants, where the
// labels fit LDS.  A lanes task walks its network at ~1.1 us a node however
// few of its lanes are used, and 1,024 tasks run at once; an LDS workgroup
// takes ~10 ns a node (23 us at least), one variant and origin each, over
// the CUs.  So few variants or few origins leave the lanes kernel waiting
// on its own latency.  Measured ms a loading, lanes and per-origin: 990
// nodes, 90 zones, 40 variants 1.06 and 0.39, 256 variants 1.43 and 2.11;
// 2,750 nodes, 250 zones, 64 variants 3.1 and 1.8, 256 variants 5.0 and 6.5;
// 5,390 nodes, 490 zones, 40 variants 7.1 and 3.6, 128 variants 9.4 and
// 11.1; metro (11,000 nodes, 1,000 zones) 16 variants 14.9 and 7.0, 64
// variants 17.1 and 27.4.  Networks with denser nodes cost the LDS kernel
// up to 1.7 times this estimate (8,460 nodes with shortcuts, 360 zones, 64
// variants: 8.9 and 12.7), hence the factor.
bool lanes_pay(const tapgpu_ctx* c, int n) {
  const double nodes = c->N, tasks = (double)c->Z * ((n + kWave - 1) / kWave);
  const double lanes = 1.1e-6 * nodes + 0.9e-9 * nodes * tasks;
  const double origin = (double)n * c->Z * std::max(23e-6, 10e-9 * nodes) / std::max(c->cus, 1);
  return 1.6 * origin >= lanes;
}

// The lanes kernel loads a batch when at least lanes_min of its variants
// are active (lanes_min 0: never) and, unless the number was asked for, it
// is the faster one.
bool use_lanes(tapgpu_ctx* c, int v0, int Vn, const unsigned char* h_on) {
  if (c->lanes_min <= 0 || !c->lanes_ok) return false;
  int n = 0;
  for (int v = v0; v < v0 + Vn; ++v) n += (!h_on || h_on[v]) ? 1 : 0;
  return n >= c->lanes_min && (!c->lanes_auto || !use_lds(c) || lanes_pay(c, n));
}

// Whether iterations run in the one-workgroup kernel: a network it holds, on
// the LDS strategy and the default link passes (h_on as for use_lanes; a
// batch for which the lanes kernel was asked for keeps it).
bool use_tiny(tapgpu_ctx* c, const unsigned char* h_on) {
  return c->tiny_ok && c->graphs && !c->profiling && use_lds(c) && c->split == 0 && c->link_mode == 0 &&
         (c->lanes_auto || !use_lanes(c, 0, c->V, h_on));
}

// All-or-nothing loading of variants [v0, v0 + Vn) (groups of those
// variants) with the current costs, by the configured strategy.  h_on is
// the host copy of var_on (null: every variant of the range).
int load_per_origin(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on) {
  if (use_lds(c)) return aon_lds(c, v0, Vn, var_on);
  if (use_hbm(c)) return aon_hbm(c, v0, Vn, var_on);
  int rc = sssp_groups(c, v0 * c->Gv, Vn * c->Gv, c->col_src, c->grp_var, var_on);
  if (!rc) rc = aon_groups(c, v0 * c->Gv, Vn * c->Gv, v0, Vn, var_on);
  return rc;
}

// A loading redone by the per-origin strategy after the lanes kernel met a
// level tie: from cleared volumes, error flag and counters.
int redo_per_origin(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on) {
  const bool pc = c->pre_cleared;
  c->pre_cleared = false;
  const int rc = load_per_origin(c, v0, Vn, var_on);
  c->pre_cleared = pc;
  return rc;
}

int load_variants(tapgpu_ctx* c, int v0, int Vn, const unsigned char* var_on,
                  const unsigned char* h_on) {
  if (use_lanes(c, v0, Vn, h_on)) {
    bool fallback = false;
    int rc = aon_lanes(c, v0, Vn, var_on, h_on, &fallback);
    if (rc || !fallback) return rc;
    return redo_per_origin(c, v0, Vn, var_on);
  }
  return load_per_origin(c, v0, Vn, var_on);
}

int launch_costs(tapgpu_ctx* c, int mode, const unsigned char* var_on, int v0, int Vn) {
  hipLaunchKernelGGL(k_costs, dim3(grid_for((long long)c->E * Vn / kWave + 1)), dim3(kBlock), 0,
                     c->stream, make_links(c, !use_lanes(c, v0, Vn, nullptr)), mode, var_on, v0, Vn);
  HIPCHK(c, hipGetLastError());
  return TAPGPU_OK;
}

// Free-flow shortest-path distances from one node (binary-heap Dijkstra on
// the host; zones other than the start are labelled but not expanded).
std::vector<double> host_dijkstra(int N, int ft0, const std::vector<int>& off,
                                  const std::vector<int>& dst, const std::vector<double>& w,
                                  int s) {
  std::vector<double> d(N, INFINITY);
  std::vector<std::pair<double, int>> heap;
  d[s] = 0.0;
  heap.push_back({0.0, s});
  auto cmp = [](const std::pair<double, int>& a, const std::pair<double, int>& b) {
    return a.first > b.first;
  };
  while (!heap.empty()) {
    std::pop_heap(heap.begin(), heap.end(), cmp);
    const auto [du, u] = heap.back();
    heap.pop_back();
    if (du > d[u] || (u < ft0 && u != s)) continue;
    for (int e = off[u]; e < off[u + 1]; ++e) {
      const double nd = du + w[e];
      if (nd < d[dst[e]]) {
        d[dst[e]] = nd;
        heap.push_back({nd, dst[e]});
        std::push_heap(heap.begin(), heap.end(), cmp);
      }
    }
  }
  return d;
}

// Column order of the zones: origins that are close in the network share a
// 64-lane group, so their wavefronts reach each node in nearby rounds.  The
// "coordinates" of a zone are its free-flow distances from two far-apart
// landmark nodes; zones are sorted along the Morton curve of those.  Results
// do not depend on the order (each column is an independent search and the
// group partial volumes are exact for integer demand).
std::vector<int> landmark_zone_order(int N, int Z, int ft0, const std::vector<int>& off,
                                     const std::vector<int>& dst, const std::vector<double>& w) {
  std::vector<int> order(Z);
  for (int z = 0; z < Z; ++z) order[z] = z;
  if (Z <= kWave) return order;
  auto farthest = [&](const std::vector<double>& d) {
    int best = 0;
    double bd = -1;
    for (int v = 0; v < N; ++v)
      if (std::isfinite(d[v]) && d[v] > bd) { bd = d[v]; best = v; }
    return best;
  };
  const int l1 = farthest(host_dijkstra(N, ft0, off, dst, w, 0));
  const std::vector<double> d1 = host_dijkstra(N, ft0, off, dst, w, l1);
  const int l2 = farthest(d1);
  const std::vector<double> d2 = host_dijkstra(N, ft0, off, dst, w, l2);
  double m1 = 0, m2 = 0;
  for (int z = 0; z < Z; ++z) {
    if (std::isfinite(d1[z])) m1 = std::max(m1, d1[z]);
    if (std::isfinite(d2[z])) m2 = std::max(m2, d2[z]);
  }
  auto q = [](double x, double m) -> uint32_t {
    if (!std::isfinite(x) || m <= 0) return 0xFFFFu;
    return (uint32_t)std::min(65535.0, std::floor(x / m * 65535.0));
  };
  auto spread = [](uint32_t x) -> uint64_t {
    uint64_t r = 0;
    for (int b = 0; b < 16; ++b) r |= (uint64_t)((x >> b) & 1u) << (2 * b);
    return r;
  };
  std::vector<uint64_t> key(Z);
  for (int z = 0; z < Z; ++z) key[z] = spread(q(d1[z], m1)) | (spread(q(d2[z], m2)) << 1);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return key[a] < key[b]; });
  return order;
}

int build(tapgpu_ctx* c, const tapgpu_network* net, const tapgpu_demand* dem, int64_t V,
          const uint8_t* present, const double* cap_v, const double* t0_v, const double* B_v,
          const double* pw_v) {
  if (!net || !dem) return c->fail(TAPGPU_E_ARG, "null network or demand");
  const int64_t N = net->num_nodes, E = net->num_links, Z = net->num_zones;
  if (N < 1 || E < 0 || Z < 0 || Z > N || V < 1)
    return c->fail(TAPGPU_E_ARG, "bad sizes N=%lld E=%lld Z=%lld V=%lld", (long long)N,
                   (long long)E, (long long)Z, (long long)V);
  if (N >= (1LL << 30) || E >= (1LL << 30))
    return c->fail(TAPGPU_E_LIMIT, "network too large for 32-bit indices");
  if (dem->num_zones != Z)
    return c->fail(TAPGPU_E_ARG, "demand has %lld zones, network %lld", (long long)dem->num_zones,
                   (long long)Z);
  c->N = (int)N; c->E = (int)E; c->Z = (int)Z; c->V = (int)V;
  int64_t ft = net->first_thru_node;
  if (ft < 1) ft = 1;
  if (ft > N + 1) ft = N + 1;
  c->ft0 = (int)(ft - 1);
  c->Gv = (int)((std::max<int64_t>(Z, 1) + kWave - 1) / kWave);
  c->Pv = (long long)c->Gv * kWave;
  c->Galloc = c->Gv * c->V;
  c->P = c->Pv * c->V;
  if ((unsigned long long)N * (unsigned long long)c->Galloc >= (1ull << 32))
    return c->fail(TAPGPU_E_LIMIT, "nodes x origin groups exceeds 2^32");

  // --- graph (host build) ---
  std::vector<int> fw_off(N + 1, 0), fw_dst(E), rv_off(N + 1, 0), rv_src(E), rv_eid(E), tail(E),
      rvpos(E);
  for (int64_t k = 0; k < E; ++k) {
    const int64_t a = net->init_node[k], b = net->term_node[k];
    if (a < 1 || a > N || b < 1 || b > N)
      return c->fail(TAPGPU_E_ARG, "link %lld has node out of range (%lld, %lld)", (long long)k,
                     (long long)a, (long long)b);
    if (k > 0 && a < net->init_node[k - 1])
      return c->fail(TAPGPU_E_ARG, "links not grouped by init node at %lld", (long long)k);
    fw_off[a]++;  // count into slot a (0-based a-1 -> prefix below)
    rv_off[b]++;
    fw_dst[k] = (int)(b - 1);
    tail[k] = (int)(a - 1);
  }
  for (int64_t v = 0; v < N; ++v) {
    fw_off[v + 1] += fw_off[v];
    rv_off[v + 1] += rv_off[v];
  }
  {
    std::vector<int> fill(rv_off.begin(), rv_off.end() - 1);
    for (int64_t k = 0; k < E; ++k) {   // stable: in-links of v in link order
      const int b = fw_dst[k];
      const int pos = fill[b]++;
      rv_src[pos] = tail[k];
      rv_eid[pos] = (int)k;
      rvpos[k] = pos;
    }
  }
  // --- origin columns in landmark order ---
  {
    std::vector<double> w0(E);
    for (int64_t k = 0; k < E; ++k)
      w0[k] = (present && !present[k]) ? INFINITY : (t0_v ? t0_v[k] : net->free_flow_time[k]);
    c->zone_order = landmark_zone_order(c->N, c->Z, c->ft0, fw_off, fw_dst, w0);
  }
  std::vector<int> col_of_zone(Z);
  for (int64_t j = 0; j < Z; ++j) col_of_zone[c->zone_order[j]] = (int)j;
  // --- demand: dense per zone row in column order ---
  std::vector<double> odc((size_t)std::max<int64_t>(Z, 1) * c->Pv, 0.0);
  double tot = 0;
  for (int64_t o = 1; o <= Z; ++o) {
    for (int64_t i = dem->od_start[o - 1]; i < dem->od_start[o]; ++i) {
      const int64_t d = dem->od_dest[i];
      const double f = dem->od_demand[i];
      tot += f;
      if (d == o || !(f > 0)) continue;
      if (d < 1 || d > Z)
        return c->fail(TAPGPU_E_ARG, "demand destination %lld is not a zone", (long long)d);
      odc[(size_t)(d - 1) * c->Pv + col_of_zone[o - 1]] += f;
    }
  }
  c->total_demand = tot;
  std::vector<long long> h_od_start(Z + 1, 0);
  std::vector<int> h_od_dest;
  std::vector<double> h_od_val;
  for (int64_t o = 1; o <= Z; ++o) {
    for (int64_t i = dem->od_start[o - 1]; i < dem->od_start[o]; ++i) {
      const int64_t d = dem->od_dest[i];
      const double f = dem->od_demand[i];
      if (d == o || !(f > 0)) continue;
      h_od_dest.push_back((int)(d - 1));
      h_od_val.push_back(f);
    }
    h_od_start[o] = (long long)h_od_dest.size();
  }
  // one-origin-per-workgroup path: labels must fit LDS, link ids and CSR
  // offsets 16-bit
  {
    int dev = 0, lds_max = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
      lds_max = 0;
    // (8W bytes more than the layout: room for a queue on the largest networks)
    c->lds_bytes = origin_lds_bytes(c->N, 0) + 8ull * ((N + 63) / 64);
    if (hipDeviceGetAttribute(&c->clock_khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess)
      c->clock_khz = 0;
    c->lds_ok = c->lds_bytes + 128 <= (size_t)lds_max && E < 65535 && N <= kLdsMaxNodes;
    if (c->lds_ok) {
      // the rest of the LDS, up to kLdsQueueMax entries, holds the frontier queues
      const size_t spare = (size_t)lds_max - 128 - origin_lds_bytes(c->N, 0);
      c->qcap_max = (int)std::min<size_t>(kLdsQueueMax, spare / 4) & ~63;
      c->qcap = c->qcap_max;
      c->lds_bytes = origin_lds_bytes(c->N, c->qcap_max);
    }
    // (the networks it takes: 24 bytes of LDS for 64 nodes)
    c->hbm_ok = 24 * (((size_t)N + 63) / 64) + 256 <= (size_t)lds_max;
    if (c->hbm_ok) {
      // queues from the LDS share of one of the kHbmPerCu workgroups on a CU
      int lds_cu = 0;
      if (hipDeviceGetAttribute(&lds_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) !=
              hipSuccess || lds_cu <= 0)
        lds_cu = lds_max;
      const size_t share = std::min<size_t>((size_t)lds_cu / kHbmPerCu, (size_t)lds_max) - 256;
      const size_t fixed = 8 * (((size_t)N + 63) / 64) + 12 * kHbmSlots;
      const size_t spare = share > fixed ? share - fixed : 0;
      c->hqcap_max = std::max((int)std::min<size_t>(kHbmQueueMax, spare / kHbmQueueBytes) & ~63, kHbmQueueMin);
      c->hqcap = c->hqcap_max;
      c->hbm_lds = origin_hbm_lds_bytes(N, c->hqcap_max);
    }
    int ncu = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) ncu = 1;
    c->cus = ncu;
    if (c->lds_ok && tiny_fits(c->N, c->E, c->Z) && tiny_lds_bytes(c->N, c->E) + 128 <= (size_t)lds_max) {
      int in = 0, zone_in = 0;                    // most in-links of a through node (that count) and of a zone
      for (int v = 0; v < c->N; ++v) {
        int n = 0;
        for (int k = rv_off[v]; k < rv_off[v + 1]; ++k) n += v < c->ft0 || (rv_src[k] >= c->ft0 && rv_src[k] != v);
        (v < c->ft0 ? zone_in : in) = std::max(v < c->ft0 ? zone_in : in, n);
      }
      bool pow4 = true;
      for (int64_t j = 0; j < (pw_v ? V * E : E); ++j) pow4 = pow4 && (pw_v ? pw_v : net->power)[j] == 4.0;
      c->tiny_ok = pow4 && tiny_pays(c->N, c->Z, in, zone_in, c->V, ncu);
    }
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_origin_hbm<2>, kHbmBlock, c->hbm_lds) !=
        hipSuccess || per_cu < 1)
      per_cu = 1;
    c->hbm_grid = std::max(1, ncu * per_cu);
    // lanes kernel: three bitmaps, then queues from the LDS share of the
    // kLanesPerCu workgroups on a CU
    {
      int lds_cu = 0;
      if (hipDeviceGetAttribute(&lds_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) !=
              hipSuccess || lds_cu <= 0)
        lds_cu = lds_max;
      const size_t base = lanes_lds_bytes(c->N, 0);
      c->lanes_ok = base + 256 <= (size_t)lds_max;
      if (c->lanes_ok) {
        const size_t share = std::min<size_t>((size_t)lds_cu / kLanesPerCu, (size_t)lds_max) - 256;
        const size_t spare = share > base ? share - base : 0;
        c->lanes_qcap_max = (int)std::min<size_t>(kLanesQueueMax, spare / 24) & ~63;
        c->lanes_qcap = c->lanes_qcap_max;
        c->lanes_lds = lanes_lds_bytes(c->N, c->lanes_qcap_max);
        int pc = 0;
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(k_origin_lanes),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)c->lanes_lds) !=
                hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&pc, k_origin_lanes, kLanesBlock,
                                                          c->lanes_lds) != hipSuccess ||
            pc < 1)
          pc = 1;
        c->lanes_grid_max = std::max(1, ncu * pc);
      }
      c->lanes_min = V > 1 ? kLanesMinDefault : 0;
    }
    double sum = 0;
    int cnt = 0;
    for (int64_t k = 0; k < E; ++k) {
      const double t = (t0_v ? t0_v[k] : net->free_flow_time[k]);
      const bool on = !present || present[k];
      if (on && t > 0 && std::isfinite(t)) { sum += t; ++cnt; }
    }
    c->mean_t0 = cnt ? sum / cnt : 1.0;
  }

  // --- link records per variant (capacity fix-up per variant) ---
  const size_t VE = (size_t)V * E;
  std::vector<double> hcap(VE), ht0(VE), hB(VE), hpw(VE);
  std::vector<unsigned char> hpres(VE, 1);
  for (int64_t v = 0; v < V; ++v) {
    double minpos = DBL_MAX;
    for (int64_t k = 0; k < E; ++k) {
      const size_t j = (size_t)v * E + k;
      hcap[j] = cap_v ? cap_v[j] : net->capacity[k];
      ht0[j] = t0_v ? t0_v[j] : net->free_flow_time[k];
      hB[j] = B_v ? B_v[j] : net->B[k];
      hpw[j] = pw_v ? pw_v[j] : net->power[k];
      if (present) hpres[j] = present[j] ? 1 : 0;
      if (hpres[j] && hcap[j] > 0.0 && hcap[j] < minpos) minpos = hcap[j];
      // the kernels order labels by their bit patterns, which holds for
      // non-negative costs only: BPR costs are non-negative when t0 and B are
      if (hpres[j] && !(ht0[j] >= 0.0 && hB[j] >= 0.0))
        return c->fail(TAPGPU_E_ARG, "link %lld of variant %lld: negative or NaN free-flow time or B",
                       (long long)k, (long long)v);
    }
    for (int64_t k = 0; k < E; ++k) {
      const size_t j = (size_t)v * E + k;
      if (!(hcap[j] > 0.0)) hcap[j] = minpos;
    }
  }
  std::vector<int> col_src(c->P, -1), grp_var(c->Galloc);
  for (int v = 0; v < c->V; ++v) {
    for (int64_t j = 0; j < Z; ++j) col_src[(size_t)v * c->Pv + j] = c->zone_order[j];
    for (int g = 0; g < c->Gv; ++g) grp_var[v * c->Gv + g] = v;
  }

  // --- device ---
  HIPCHK(c, hipGetDevice(&c->device));
  HIPCHK(c, hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  HIPCHK(c, hipStreamCreateWithFlags(&c->stream2, hipStreamNonBlocking));
  HIPCHK(c, hipEventCreateWithFlags(&c->ev_fork, hipEventDisableTiming));
  HIPCHK(c, hipEventCreateWithFlags(&c->ev_join, hipEventDisableTiming));
  HIPCHK(c, hipHostMalloc((void**)&c->h_int, 64 * sizeof(int), hipHostMallocDefault));
  {
    const size_t bytes = 16 + 128 + sizeof(VarState) * (size_t)V + (size_t)V;   // as iter_dev
    HIPCHK(c, hipHostMalloc(&c->pin_block, bytes, hipHostMallocDefault));
    unsigned char* b = (unsigned char*)c->pin_block;
    c->pin_err = (int*)b;
    c->pin_cnt = (unsigned long long*)(b + 16);
    c->pin_st = (VarState*)(b + 144);
    c->pin_on = b + 144 + sizeof(VarState) * (size_t)V;
  }
  int rc;
#define ALLOC(ptr, n) if ((rc = balloc(c, &c->ptr, (n)))) return rc
  ALLOC(fw_off, N + 1); ALLOC(fw_dst, E); ALLOC(rv_off, N + 1); ALLOC(rv_src, E);
  ALLOC(rv_eid, E); ALLOC(tail, E); ALLOC(rvpos, E);
  ALLOC(t0, VE); ALLOC(cap, VE); ALLOC(B, VE); ALLOC(pw, VE); ALLOC(present, VE);
  ALLOC(x, VE); ALLOC(y, VE); ALLOC(c, VE); ALLOC(rvw, VE); ALLOC(fww, VE);
  ALLOC(col_src, c->P); ALLOC(grp_var, c->Galloc);
  c->flags_cap = (int)std::min<int64_t>(std::max<int64_t>(4 * N + 64, 1024), 1 << 24);
  ALLOC(flags, c->flags_cap);
  {
    c->iter_bytes = 16 + 128 + sizeof(VarState) * (size_t)V + (size_t)V;
    if ((rc = balloc(c, &c->iter_dev, c->iter_bytes))) return rc;
    c->err_dev = (int*)c->iter_dev;
    c->counters = (unsigned long long*)(c->iter_dev + 16);
    c->st = (VarState*)(c->iter_dev + 144);
    c->var_on = c->iter_dev + 144 + sizeof(VarState) * (size_t)V;
  }


  ALLOC(part, (size_t)V * link_blocks(c->E, V, false) * kQ);
  ALLOC(done, V);
  ALLOC(prm, 1);
  // the LDS kernel's mirrors (k_mirrors fills them in, store_cost their costs)
  const int W = (int)((N + 63) / 64);
  std::vector<int> sell_ptr;
  if (c->lds_ok) {
    sell_ptr.assign(W + 1, 0);
    for (int64_t v = c->ft0; v < N; ++v) {
      int n = 0;
      for (int k = rv_off[v]; k < rv_off[v + 1]; ++k) n += rv_src[k] != v && rv_src[k] >= c->ft0;
      int& rows = sell_ptr[v / kWave + 1];
      rows = std::max(rows, std::min(kSellWidth, n));
    }
    for (int i = 0; i < W; ++i) sell_ptr[i + 1] = sell_ptr[i] + sell_ptr[i + 1] * kWave;
    c->sell_n = std::max(sell_ptr[W], kWave);          // (a slice without rows reads the first one's)
    ALLOC(rec, (size_t)V * (N * kRecDoubles + c->sell_n));
    ALLOC(recpos, 2 * (size_t)E + W + 1 + c->sell_n);
    c->sellw = c->rec + (size_t)V * N * kRecDoubles;
    c->sellpos = c->recpos + E;
    c->sell_ptr = c->sellpos + E;
    c->sell_id = (unsigned*)(c->sell_ptr + W + 1);
  }
#undef ALLOC
  if ((rc = upload(c, c->fw_off, fw_off.data(), N + 1))) return rc;
  if ((rc = upload(c, c->fw_dst, fw_dst.data(), E))) return rc;
  if ((rc = upload(c, c->rv_off, rv_off.data(), N + 1))) return rc;
  if ((rc = upload(c, c->rv_src, rv_src.data(), E))) return rc;
  if ((rc = upload(c, c->rv_eid, rv_eid.data(), E))) return rc;
  if ((rc = upload(c, c->tail, tail.data(), E))) return rc;
  if ((rc = upload(c, c->rvpos, rvpos.data(), E))) return rc;
  if ((rc = upload(c, c->t0, ht0.data(), VE))) return rc;
  if ((rc = upload(c, c->cap, hcap.data(), VE))) return rc;
  if ((rc = upload(c, c->B, hB.data(), VE))) return rc;
  if ((rc = upload(c, c->pw, hpw.data(), VE))) return rc;
  if ((rc = upload(c, c->present, hpres.data(), VE))) return rc;
  if ((rc = upload(c, c->col_src, col_src.data(), c->P))) return rc;
  if ((rc = upload(c, c->grp_var, grp_var.data(), c->Galloc))) return rc;
  if (!c->lds_ok && c->hbm_ok && (rc = alloc_hbm_mirrors(c, 1))) return rc;   // (tapgpu_sssp_noalloc allocates nothing)
  if (c->lds_ok) {
    if ((rc = upload(c, c->sell_ptr, sell_ptr.data(), sell_ptr.size()))) return rc;
    hipLaunchKernelGGL(k_mirrors, dim3((W * kWave + kBlock - 1) / kBlock), dim3(kBlock), 0, c->stream,
                       make_graph(c), make_links(c), c->sell_ptr, c->sell_id, c->recpos, c->sellpos);
    HIPCHK(c, hipGetLastError());
  }
  c->h_odc = std::move(odc);
  if ((rc = balloc(c, &c->od_start, Z + 1))) return rc;
  if ((rc = balloc(c, &c->od_dest, h_od_dest.size()))) return rc;
  if ((rc = balloc(c, &c->od_val, h_od_val.size()))) return rc;
  if ((rc = upload(c, c->od_start, h_od_start.data(), Z + 1))) return rc;
  if ((rc = upload(c, c->od_dest, h_od_dest.data(), h_od_dest.size()))) return rc;
  if ((rc = upload(c, c->od_val, h_od_val.data(), h_od_val.size()))) return rc;
  if (c->tiny_ok)
    HIPCHK(c, hipFuncSetAttribute(tiny_kernel(c->N), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)tiny_lds_bytes(c->N, c->E)));
  if (c->lds_ok) {
    HIPCHK(c, hipFuncSetAttribute(reinterpret_cast<const void*>(k_origin_lds<1024>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)c->lds_bytes));
    HIPCHK(c, hipFuncSetAttribute(reinterpret_cast<const void*>(k_origin_lds<512>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)c->lds_bytes));
    HIPCHK(c, hipFuncSetAttribute(reinterpret_cast<const void*>(k_origin_lds<256>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)c->lds_bytes));
  }

  c->h_od_start = std::move(h_od_start);
  c->h_od_dest = std::move(h_od_dest);
  c->h_od_val = std::move(h_od_val);
  c->h_tail = std::move(tail);
  c->h_head = fw_dst;

  HIPCHK(c, hipMemsetAsync(c->x, 0, sizeof(double) * VE, c->stream));
  HIPCHK(c, hipMemsetAsync(c->y, 0, sizeof(double) * VE, c->stream));
  HIPCHK(c, hipMemsetAsync(c->var_on, 1, V, c->stream));
  HIPCHK(c, hipMemsetAsync(c->done, 0, sizeof(unsigned) * V, c->stream));
  // Wa = free-flow time (trunk/tap/tap_functions.c:331)
  if ((rc = launch_costs(c, 0, nullptr, 0, c->V))) return rc;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return TAPGPU_OK;
}

int check_variant(tapgpu_ctx* c, int64_t v) {
  if (v < 0 || v >= c->V) return c->fail(TAPGPU_E_ARG, "variant %lld out of range", (long long)v);
  return TAPGPU_OK;
}

}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

extern "C" {

int tapgpu_create_batched(tapgpu_ctx** out, const tapgpu_network* net, const tapgpu_demand* dem,
                          int64_t num_variants, const uint8_t* present, const double* capacity_v,
                          const double* free_flow_time_v, const double* B_v,
                          const double* power_v) {
  if (!out) return TAPGPU_E_ARG;
  *out = nullptr;
  tapgpu_ctx* c = new (std::nothrow) tapgpu_ctx();
  if (!c) return TAPGPU_E_NOMEM;
  const int rc = build(c, net, dem, num_variants, present, capacity_v, free_flow_time_v, B_v,
                       power_v);
  if (rc) {
    g_create_error = c->err;
    tapgpu_destroy(c);
    return rc;
  }
  *out = c;
  return TAPGPU_OK;
}

int tapgpu_create(tapgpu_ctx** out, const tapgpu_network* net, const tapgpu_demand* dem) {
  return tapgpu_create_batched(out, net, dem, 1, nullptr, nullptr, nullptr, nullptr, nullptr);
}

void tapgpu_destroy(tapgpu_ctx* c) {
  if (!c) return;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  if (c->g_iter) (void)hipGraphExecDestroy(c->g_iter);
  if (c->g_link) (void)hipGraphExecDestroy(c->g_link);
  for (void* p : c->allocs) (void)hipFree(p);
  if (c->trace) (void)hipFree(c->trace);
  if (c->h_int) (void)hipHostFree(c->h_int);
  if (c->pin_block) (void)hipHostFree(c->pin_block);
  if (c->stage_pin) (void)hipHostFree(c->stage_pin);
  if (c->stage_dev) (void)hipFree(c->stage_dev);
  for (auto& e : c->stage_ev)
    if (e) (void)hipEventDestroy(e);
  for (auto& e : c->ev)
    if (e) (void)hipEventDestroy(e);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  if (c->stream2) (void)hipStreamDestroy(c->stream2);
  if (c->ev_fork) (void)hipEventDestroy(c->ev_fork);
  if (c->ev_join) (void)hipEventDestroy(c->ev_join);
  delete c;
}

const char* tapgpu_last_error(const tapgpu_ctx* c) {
  return c ? c->err.c_str() : g_create_error.c_str();
}

int64_t tapgpu_num_variants(const tapgpu_ctx* c) { return c ? c->V : 0; }

int tapgpu_set_costs(tapgpu_ctx* c, int64_t variant, const double* costs) {
  if (!c || !costs) return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  int bad = 0;                                   // (no early exit: the loop takes vectors)
  for (int k = 0; k < c->E; ++k) bad |= !(costs[k] >= 0.0);
  for (int k = 0; bad && k < c->E; ++k)
    if (!(costs[k] >= 0.0))
      return c->fail(TAPGPU_E_ARG, "link %d: negative or NaN cost", k);
  if ((rc = upload(c, c->c + (size_t)variant * c->E, costs, c->E))) return rc;
  if ((rc = launch_costs(c, 2, nullptr, (int)variant, 1))) return rc;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return TAPGPU_OK;
}

int tapgpu_sssp(tapgpu_ctx* c, int64_t variant, const int64_t* start_nodes, int64_t num_start,
                double* dist, int64_t* pred, int64_t ld, int64_t col_base) {
  if (!c || (num_start > 0 && !start_nodes) || num_start < 0 || col_base < 0)
    return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  // row v starts at v * ld; with pape_cuda's layout (ld = num_start,
  // col_base = 1) the last column of row v is the unused column 0 of v + 1
  if (ld < num_start || (col_base > 0 && ld < num_start + col_base - 1))
    return c->fail(TAPGPU_E_ARG, "ld %lld too small for %lld columns", (long long)ld,
                   (long long)num_start);
  for (int64_t i = 0; i < num_start; ++i)
    if (start_nodes[i] < 1 || start_nodes[i] > c->N)
      return c->fail(TAPGPU_E_ARG, "start node %lld out of range", (long long)start_nodes[i]);
  const int64_t N1 = (int64_t)c->N + 1;
  // node 0 does not exist: row 0 stays unreachable
  for (int64_t i = 0; i < num_start; ++i) {
    if (dist) dist[col_base + i] = DBL_MAX;
    if (pred) pred[col_base + i] = -1;
  }
  if (use_lds(c) || use_hbm(c)) {
    // one workgroup per start node (labels in LDS), or the persistent
    // labels-in-HBM grid; chunks of up to 1024 starts
    const bool hbm = !use_lds(c);
    if (hbm && (rc = ensure_hbm(c, 1))) return rc;
    const int64_t chunk = std::min<int64_t>(std::max<int64_t>(num_start, 1), 1024);
    SsspStage S;
    rc = stage_sssp(c, chunk, &S);
    for (int64_t s0 = 0; !rc && s0 < num_start; s0 += chunk) {
      const int ns = (int)std::min<int64_t>(chunk, num_start - s0);
      for (int j = 0; j < ns; ++j) S.src[j] = (int)(start_nodes[s0 + j] - 1);
      OriginArgs A = make_origin_args(c, nullptr);
      advance_variant(c, A, variant);
      A.src_list = S.src; A.err = S.err; A.out_dist = S.dist; A.out_pred = S.pred; A.ld = ns;
      hipLaunchKernelGGL(k_sssp_begin, dim3(grid_for((long long)c->N * ns / kWave + 1)), dim3(kBlock), 0,
                         c->stream, S.pred, (long long)c->N * ns, S.err);
      if (hbm)
        launch_hbm_kernel(c, A, 1, 0, ns, c->hbm_grid, c->stream, s0 == 0);
      else
        launch_lds(c, dim3(ns, 1), c->stream, A, 0);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess)
        rc = c->fail(TAPGPU_E_HIP, "shortest-path launch failed: %s", hipGetErrorString(e));
      else
        rc = deliver_sssp(c, S, ns, dist, pred, ld, col_base + s0);
    }
    stage_trim(c);
    return rc;
  }
  // chunks of the variant's columns; groups [0, Gv) of a private mapping
  int* d_col = nullptr;
  int* d_gv = nullptr;
  if ((rc = dalloc(c, &d_col, c->Pv))) return rc;
  if ((rc = dalloc(c, &d_gv, c->Gv))) return rc;
  std::vector<int> hgv(c->Gv, (int)variant), hcol(c->Pv);
  std::vector<double> hd((size_t)c->N * c->Pv);
  std::vector<int> hp((size_t)c->N * c->Pv);
  rc = upload(c, d_gv, hgv.data(), c->Gv);
  for (int64_t s0 = 0; !rc && s0 < num_start; s0 += c->Pv) {
    const int64_t ns = std::min<int64_t>(c->Pv, num_start - s0);
    for (int64_t j = 0; j < c->Pv; ++j) hcol[j] = j < ns ? (int)(start_nodes[s0 + j] - 1) : -1;
    if ((rc = upload(c, d_col, hcol.data(), c->Pv))) break;
    const int Gn = (int)((ns + kWave - 1) / kWave);
    if ((rc = sssp_groups(c, 0, Gn, d_col, d_gv, nullptr))) break;
    // rows are P apart on the device; copy the first Pv columns of each row
    const hipError_t e1 = hipMemcpy2DAsync(hd.data(), c->Pv * sizeof(double), c->dist,
                                           c->P * sizeof(double), c->Pv * sizeof(double), c->N,
                                           hipMemcpyDeviceToHost, c->stream);
    const hipError_t e2 = hipMemcpy2DAsync(hp.data(), c->Pv * sizeof(int), c->pred,
                                           c->P * sizeof(int), c->Pv * sizeof(int), c->N,
                                           hipMemcpyDeviceToHost, c->stream);
    const hipError_t e3 = hipStreamSynchronize(c->stream);
    if (e1 != hipSuccess || e2 != hipSuccess || e3 != hipSuccess) {
      rc = c->fail(TAPGPU_E_HIP, "copy of labels failed");
      break;
    }
    for (int64_t v = 1; v < N1; ++v) {
      const size_t row = (size_t)(v - 1) * c->Pv;
      for (int64_t j = 0; j < ns; ++j) {
        const size_t o = (size_t)v * ld + col_base + s0 + j;
        if (dist) dist[o] = hd[row + j];
        if (pred) pred[o] = hp[row + j];
      }
    }
  }
  // private buffers are freed here (not kept in allocs)
  c->allocs.erase(std::remove(c->allocs.begin(), c->allocs.end(), (void*)d_col), c->allocs.end());
  c->allocs.erase(std::remove(c->allocs.begin(), c->allocs.end(), (void*)d_gv), c->allocs.end());
  (void)hipFree(d_col);
  (void)hipFree(d_gv);
  return rc;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// shortest paths without allocation (tapgpu_sssp_noalloc)
// ---------------------------------------------------------------------------
//
// The per-origin kernels' scratch (the labels-in-HBM kernel's label,
// predecessor and tail rows, and the 0-based start list of either kernel)
// lives in this file-scope device array instead of buffers allocated by the
// context.  Each GPU holds its own copy for the life of the process; host
// code reaches it only through the address hipGetSymbolAddress returns for
// the current device (kept per device in g_scratch_ptr).  Every call on a
// GPU shares that GPU's copy: calls that overlap on one GPU race.

constexpr size_t kNoAllocScratchBytes = 64ull << 20;       // 64 MiB per GPU
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on device `dev` (which is current).
int scratch_address(tapgpu_ctx* c, int dev, void** out) {
  if (dev < 0 || dev >= kMaxDevices) return c->fail(TAPGPU_E_ARG, "device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return c->fail(TAPGPU_E_HIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return TAPGPU_OK;
}

// 1-based start nodes -> 0-based list; clears the error flag first; a start
// node outside 1..N is flagged (code 5) and replaced by node 0.  One block.
__global__ __launch_bounds__(kBlock) void k_noalloc_starts(const int64_t* starts, int64_t n, int N,
                                                           int* out, int* err) {
  if (threadIdx.x < 3) err[threadIdx.x] = 0;
  __syncthreads();
  for (int64_t i = threadIdx.x; i < n; i += kBlock) {
    const int64_t s = starts[i];
    if (s < 1 || s > N) {
      if (atomicCAS(&err[0], 0, 5) == 0) err[1] = (int)i;
      out[i] = 0;
    } else {
      out[i] = (int)(s - 1);
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_fill_i32(int* p, long long n, int v) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (long long)gridDim.x * kBlock)
    p[i] = v;
}

}  // namespace

extern "C" {

int tapgpu_sssp_noalloc(tapgpu_ctx* c, int64_t variant, const int64_t* d_start_nodes,
                        int64_t num_start, double* d_dist, int32_t* d_pred, int64_t ld) {
  if (!c || num_start < 0 || (num_start > 0 && (!d_start_nodes || !d_dist || !d_pred)))
    return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  if (num_start == 0) return TAPGPU_OK;
  if (ld < num_start)
    return c->fail(TAPGPU_E_ARG, "ld %lld too small for %lld columns", (long long)ld,
                   (long long)num_start);
  if (num_start > INT32_MAX) return c->fail(TAPGPU_E_LIMIT, "too many start nodes");
  int dev = -1;
  HIPCHK(c, hipGetDevice(&dev));
  if (dev != c->device)
    return c->fail(TAPGPU_E_STATE, "the context belongs to device %d, device %d is current",
                   c->device, dev);
  const bool lds = use_lds(c);
  if (!lds && !c->hbm_ok)
    return c->fail(TAPGPU_E_LIMIT, "the per-origin kernels do not fit this network");
  // scratch: the start list, then (labels-in-HBM kernel) rows of 16 B per node
  const size_t list_bytes = ((size_t)num_start * sizeof(int) + 255) & ~(size_t)255;
  const size_t row_bytes = 16ull * (size_t)c->N;
  if (list_bytes + (lds ? 0 : row_bytes) > kNoAllocScratchBytes)
    return c->fail(TAPGPU_E_LIMIT,
                   "%lld start nodes on %d nodes exceed the %zu-byte scratch of the no-allocation "
                   "entry point", (long long)num_start, c->N, kNoAllocScratchBytes);
  void* base = nullptr;
  if ((rc = scratch_address(c, dev, &base))) return rc;
  unsigned char* p = (unsigned char*)base;
  int* d_src = (int*)p;
  OriginArgs A = make_origin_args(c, nullptr);
  advance_variant(c, A, variant);
  A.src_list = d_src;
  A.out_dist = d_dist;
  A.out_pred = d_pred;
  A.ld = ld;
  int rows = 0;
  if (!lds) {
    rows = (int)std::min<size_t>((size_t)c->hbm_grid, (kNoAllocScratchBytes - list_bytes) / row_bytes);
    const size_t rN = (size_t)rows * c->N;
    A.h_dist = (unsigned long long*)(p + list_bytes);
    A.h_pred = (int*)(p + list_bytes + 8 * rN);
    A.h_ptail = (int*)(p + list_bytes + 12 * rN);
  }
  hipLaunchKernelGGL(k_noalloc_starts, dim3(1), dim3(kBlock), 0, c->stream, d_start_nodes, num_start,
                     c->N, d_src, c->err_dev);
  // predecessors start at -1, so a failed search hands back no stale link
  const long long npred = (long long)c->N * ld;
  hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(npred / kWave + 1)), dim3(kBlock), 0, c->stream,
                     d_pred, npred, -1);
  if (lds) {
    launch_lds(c, dim3((unsigned)num_start, 1), c->stream, A, 0);
  } else {
    launch_hbm_kernel(c, A, 1, 0, (int)num_start, rows, c->stream);
  }
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipMemcpyAsync(c->h_int, c->err_dev, sizeof(int) * 3, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  const int* herr = c->h_int;
  if (herr[0] == 5)
    return c->fail(TAPGPU_E_ARG, "start node %d of the list is out of range", herr[1]);
  return sssp_error(c, herr);
}

int tapgpu_aon(tapgpu_ctx* c, int64_t variant, double* volumes) {
  if (!c) return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  const int v = (int)variant;
  std::vector<unsigned char> on(c->V, 0);
  on[v] = 1;
  if (!c->aon_on && (rc = dalloc(c, &c->aon_on, c->V))) return rc;
  if ((rc = upload(c, c->aon_on, on.data(), c->V))) return rc;
  if ((rc = load_variants(c, v, 1, c->aon_on, on.data()))) return rc;
  if (volumes) {
    const hipError_t e = hipMemcpy(volumes, c->y + (size_t)v * c->E, sizeof(double) * c->E,
                                   hipMemcpyDeviceToHost);
    if (e != hipSuccess) return c->fail(TAPGPU_E_HIP, "copy of volumes failed");
  }
  return TAPGPU_OK;
}

static int ensure_trace(tapgpu_ctx* c, int need) {
  if (need <= c->trace_cap) return TAPGPU_OK;
  int cap = std::max(need, 1024);
  tapgpu_iter* t = nullptr;
  hipError_t e = hipMalloc((void**)&t, sizeof(tapgpu_iter) * (size_t)cap * c->V);
  if (e != hipSuccess) return c->fail(TAPGPU_E_NOMEM, "trace allocation failed");
  HIPCHK(c, hipMemsetAsync(t, 0, sizeof(tapgpu_iter) * (size_t)cap * c->V, c->stream));
  if (c->trace) {
    for (int v = 0; v < c->V; ++v)
      HIPCHK(c, hipMemcpyAsync(t + (size_t)v * cap, c->trace + (size_t)v * c->trace_cap,
                               sizeof(tapgpu_iter) * c->trace_cap, hipMemcpyDeviceToDevice,
                               c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    (void)hipFree(c->trace);
  }
  c->trace = t;
  c->trace_cap = cap;
  return TAPGPU_OK;
}

int tapgpu_fw_init(tapgpu_ctx* c, const double* warm_volumes) {
  if (!c) return TAPGPU_E_ARG;
  int rc = ensure_trace(c, 1024);
  if (rc) return rc;
  std::vector<VarState> hs(c->V);
  for (auto& s : hs) {
    s = VarState{};
    s.best_lb = -DBL_MAX;
    s.relgap = DBL_MAX;
    s.total_demand = c->total_demand;
    s.active = 1;
  }
  if ((rc = upload(c, c->st, hs.data(), c->V))) return rc;
  HIPCHK(c, hipMemsetAsync(c->var_on, 1, c->V, c->stream));
  if (warm_volumes) {
    if ((rc = upload(c, c->x, warm_volumes, (size_t)c->V * c->E))) return rc;
  } else if (use_tiny(c, nullptr)) {
    // the loading, x = y and c = BPR(x) in one launch
    hipLaunchKernelGGL(k_iter_begin, dim3(1), dim3(kBlock), 0, c->stream, c->err_dev, c->counters, c->y, 0ll);
    if ((rc = launch_tiny(c, 1))) return rc;
    if ((rc = finish_origin(c, c->V, std::chrono::steady_clock::now()))) return rc;
    c->initialised = true;
    return TAPGPU_OK;
  } else {
    if ((rc = launch_costs(c, 0, nullptr, 0, c->V))) return rc;   // Wa = t0
    if ((rc = load_variants(c, 0, c->V, nullptr, nullptr))) return rc;
    HIPCHK(c, hipMemcpyAsync(c->x, c->y, sizeof(double) * (size_t)c->V * c->E,
                             hipMemcpyDeviceToDevice, c->stream));
  }
  if ((rc = launch_costs(c, 1, nullptr, 0, c->V))) return rc;      // c = BPR(x)
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->initialised = true;
  return TAPGPU_OK;
}

__global__ void k_set_params(FwParams* p, FwParams v) { *p = v; }

// (a kernel argument, not a copy from host memory that the next call
// overwrites)
static int upload_params(tapgpu_ctx* c, int max_iters, double target) {
  hipLaunchKernelGGL(k_set_params, dim3(1), dim3(1), 0, c->stream, c->prm,
                     FwParams{c->trace, c->trace_cap, max_iters, target, c->line_window});
  HIPCHK(c, hipGetLastError());
  return TAPGPU_OK;
}

// The link passes of an iteration: the line search (with the flags) and the
// step, and the copy of the iteration block (error flag, counters, states,
// flags) to pinned host memory.  With `more` the next window of the variants
// whose step is below the last one.
static int issue_link_passes(tapgpu_ctx* c, const Links& K, bool readback = true, int more = 0) {
  const bool alone = c->link_mode == 1 || (c->link_mode == 0 && c->E <= kSmallLinks);
  const int nb = link_blocks(c->E, c->V, alone);
  for (int v = 0; v < c->V; v += kGridVariants)
    hipLaunchKernelGGL(k_link_search, dim3(nb, std::min(c->V - v, kGridVariants)), dim3(kBlock), 0,
                       c->stream, K, c->st, c->var_on, c->part, c->done, c->err_dev, c->prm, v,
                       alone ? 1 : 0, alone || c->E <= kSoloLinks ? 1 : 0, more);
  for (int v = 0; v < c->V && !alone; v += kGridVariants)
    hipLaunchKernelGGL(k_link_step, dim3(nb, std::min(c->V - v, kGridVariants)), dim3(kBlock), 0,
                       c->stream, K, c->st, v);
  HIPCHK(c, hipGetLastError());
  if (readback)
    HIPCHK(c, hipMemcpyAsync(c->pin_block, c->iter_dev, c->iter_bytes, hipMemcpyDeviceToHost,
                             c->stream));
  return TAPGPU_OK;
}

static void launch_totals(tapgpu_ctx* c) {
  const int nb = link_blocks(c->E, c->V, false);
  for (int v = 0; v < c->V; v += kGridVariants)
    hipLaunchKernelGGL(k_totals, dim3(nb, std::min(c->V - v, kGridVariants)), dim3(kBlock), 0, c->stream,
                       make_links(c), c->part, c->done, c->vht, v);
}

// Records what `issue` puts on the context's stream into an executable
// graph (replacing *exec).  Nothing in a captured sequence may allocate,
// synchronise, record events or clear memory with a memset: the captured
// kernels clear what they need themselves.
extern "C++" template <class F>
static int capture(tapgpu_ctx* c, hipGraphExec_t* exec, F&& issue) {
  if (*exec) {
    HIPCHK(c, hipGraphExecDestroy(*exec));
    *exec = nullptr;
  }
  HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  c->capturing = true;               // (launch paths then skip host-side set-up)
  const int rc = issue();
  c->capturing = false;
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(c->stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess || !g) return c->fail(TAPGPU_E_HIP, "stream capture failed: %s", hipGetErrorString(e));
  const hipError_t ei = hipGraphInstantiate(exec, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (ei != hipSuccess) {
    *exec = nullptr;
    return c->fail(TAPGPU_E_HIP, "graph instantiation failed: %s", hipGetErrorString(ei));
  }
  return TAPGPU_OK;
}

// The whole iteration of a tuned per-origin schedule as one graph:
// k_iter_begin, the loading kernel, the link passes and the readback.  It is
// captured again when the schedule that its launches bake in changes.
// With m > 1 the graph holds m iterations back to back and one readback: a
// variant that stops (or converges) in one of them is skipped by the rest
// (its flag is off), so the results are those of m single replays.  Used
// where an iteration is short enough for the launch and synchronisation
// to matter.
static int iter_graph(tapgpu_ctx* c, const Links& K, int m) {
  const bool lds = use_lds(c);
  if (!lds) {
    int rc = ensure_hbm(c, c->V);
    if (rc) return rc;
  }
  long long dbits;
  std::memcpy(&dbits, &c->delta_mult, sizeof dbits);
  const long long key[6] = {(lds ? 1 : 2) + 4 * m + (c->origin_order_ready ? 64 : 0) + 128 * c->link_mode,
                            c->chase, c->qcap, c->hqcap, dbits, lds_threads(c)};
  if (c->g_iter && std::equal(key, key + 6, c->g_iter_key)) return TAPGPU_OK;
  int rc = capture(c, &c->g_iter, [&]() -> int {
    const long long ny = (long long)c->V * c->E;
    hipLaunchKernelGGL(k_iter_begin, dim3(grid_for(ny / kWave + 1)), dim3(kBlock), 0, c->stream,
                       c->err_dev, c->counters, c->y, ny);
    for (int it = 0; it < m; ++it) {
      c->defer_origin = true;
      c->pre_cleared = true;
      int r = lds ? aon_lds(c, 0, c->V, c->var_on) : aon_hbm(c, 0, c->V, c->var_on);
      c->defer_origin = false;
      c->pre_cleared = false;
      c->origin_pending = false;
      if (r) return r;
      if ((r = issue_link_passes(c, K, it == m - 1))) return r;
    }
    return TAPGPU_OK;
  });
  if (rc) return rc;
  std::copy(key, key + 6, c->g_iter_key);
  return TAPGPU_OK;
}

// The whole iteration of a batch on the lanes kernel as one graph:
// k_iter_begin (error flag, counters), pack, the lanes kernel, unpack, the
// link passes and the readback.  The lane map and the memo
// stamps are device data, set before each replay; the graph is captured
// again when the number of groups or the kernel's schedule changes.
static int lanes_graph(tapgpu_ctx* c, const Links& K, int G) {
  long long dbits;
  std::memcpy(&dbits, &c->lanes_delta_mult, sizeof dbits);
  const long long key[6] = {3 + (c->origin_order_ready ? 64 : 0) + 128 * c->link_mode, G, c->lanes_qcap,
                            dbits, (long long)c->lanes_lds, c->lanes_grid};
  if (c->g_iter && std::equal(key, key + 6, c->g_iter_key)) return TAPGPU_OK;
  int rc = capture(c, &c->g_iter, [&]() {
    hipLaunchKernelGGL(k_iter_begin, dim3(1), dim3(kBlock), 0, c->stream, c->err_dev, c->counters,
                       c->y, 0ll);
    int r = launch_lanes(c, G, (long long)c->Z * G, nullptr);
    if (r) return r;
    return issue_link_passes(c, K);
  });
  if (rc) return rc;
  std::copy(key, key + 6, c->g_iter_key);
  return TAPGPU_OK;
}

static int link_graph(tapgpu_ctx* c, const Links& K) {
  if (c->g_link && c->g_link_mode == c->link_mode) return TAPGPU_OK;
  c->g_link_mode = c->link_mode;
  return capture(c, &c->g_link, [&]() { return issue_link_passes(c, K); });
}

int tapgpu_set_link_passes(tapgpu_ctx* c, int mode, int window) {
  if (!c || mode < 0 || mode > 2 || window < 0 || window > kJ) return TAPGPU_E_ARG;
  c->link_mode = mode;
  c->line_window = window > 0 ? window : kJ;
  return TAPGPU_OK;
}

int tapgpu_set_graphs(tapgpu_ctx* c, int mode) {
  if (!c || mode < 0 || mode > kMaxGraphIters) return TAPGPU_E_ARG;
  c->graphs = mode != 0;
  c->graph_iters = mode > 1 ? mode : 0;
  return TAPGPU_OK;
}

int tapgpu_get_graphs(tapgpu_ctx* c, int* mode) {
  if (!c || !mode) return TAPGPU_E_ARG;
  *mode = !c->graphs ? 0 : (c->graph_iters > 1 ? c->graph_iters : 1);
  return TAPGPU_OK;
}

int tapgpu_fw_run(tapgpu_ctx* c, int max_iters, double target_relgap, tapgpu_result* results) {
  if (!c) return TAPGPU_E_ARG;
  if (!c->initialised) return c->fail(TAPGPU_E_STATE, "tapgpu_fw_init was not called");
  int rc = ensure_trace(c, max_iters > 0 ? max_iters : 1024);
  if (rc) return rc;
  c->stats = tapgpu_stats{};
  auto t_start = std::chrono::steady_clock::now();
  Links K = make_links(c);
  std::vector<unsigned char> hon(c->V);
  std::vector<VarState> hs(c->V);
  // variants already past the stop rule do not run (the loop test comes first)
  HIPCHK(c, hipMemcpy(hs.data(), c->st, sizeof(VarState) * c->V, hipMemcpyDeviceToHost));
  for (int v = 0; v < c->V; ++v) {
    hs[v].need_more = 0;                // (a run that ended in an error may have left it)
    hs[v].active = (max_iters <= 0 || hs[v].iter < max_iters) &&
                   (target_relgap <= 0 || hs[v].relgap > target_relgap);
    hon[v] = (unsigned char)hs[v].active;
  }
  if ((rc = upload(c, c->st, hs.data(), c->V))) return rc;
  if ((rc = upload(c, c->var_on, hon.data(), c->V))) return rc;
  // One synchronisation per iteration (or per replay of several): the
  // loading's error flag and counters, the variants' states and flags are
  // read back together at the end.
  if (!c->ev[2])
    for (auto& e : c->ev) HIPCHK(c, hipEventCreate(&e));
  if ((rc = upload_params(c, max_iters, target_relgap))) return rc;
  for (;;) {
    bool any = false;
    for (int v = 0; v < c->V; ++v) any = any || hon[v];
    if (!any) break;
    if (c->trace_cap < 1 << 30) {
      int maxit = 0;
      for (int v = 0; v < c->V; ++v) maxit = std::max(maxit, hs[v].iter);
      const int ahead = std::max(kMaxGraphIters, kTinyIters);       // iterations before the next look
      if (maxit + ahead >= c->trace_cap) {
        if ((rc = ensure_trace(c, std::max(2 * c->trace_cap, maxit + ahead + 1)))) return rc;
        if ((rc = upload_params(c, max_iters, target_relgap))) return rc;
      }
    }
    auto t_it = std::chrono::steady_clock::now();
    if (use_tiny(c, hon.data())) {
      // up to kTinyIters iterations of every variant in one launch
      hipLaunchKernelGGL(k_iter_begin, dim3(1), dim3(kBlock), 0, c->stream, c->err_dev, c->counters, c->y, 0ll);
      if ((rc = launch_tiny(c, 0))) return rc;
      HIPCHK(c, hipMemcpyAsync(c->pin_block, c->iter_dev, c->iter_bytes, hipMemcpyDeviceToHost, c->stream));
      HIPCHK(c, hipStreamSynchronize(c->stream));
      int64_t done = 0;
      for (int v = 0; v < c->V; ++v) done += c->pin_st[v].iter - hs[v].iter;
      if ((rc = absorb_origin(c, c->pin_err, c->pin_cnt, 0, std::chrono::steady_clock::now()))) return rc;
      c->stats.origin_blocks += (int64_t)c->Z * done;
      c->stats.link_passes += done / c->V;
      std::copy(c->pin_st, c->pin_st + c->V, hs.begin());
      std::copy(c->pin_on, c->pin_on + c->V, hon.begin());
      c->stats.link_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_it).count();
      continue;
    }
    if ((rc = origin_order_update(c))) return rc;      // (before any capture)
    // with the schedule already tuned, one kernel opens the iteration and
    // clears what the loading would clear
    const bool tuned = use_lds(c) ? (c->chase >= 0 && c->split >= 0 && c->lds_block > 0)
                                  : (use_hbm(c) && c->delta_mult >= 0);
    const bool graphs = c->graphs && !c->profiling;
    const bool lanes_now = use_lanes(c, 0, c->V, hon.data());
    float aon = 0.f;
    // how the iteration runs: a captured graph of all of it (per-origin
    // kernel or lanes kernel), or the loading issued launch by launch and
    // the link passes (captured or not) after it
    int mode = 0;
    int G = 0;
    if (graphs && lanes_now && c->lanes_delta_mult >= 0 && c->l_dist && c->Z > 0) {
      if ((rc = lanes_map(c, 0, c->V, hon.data(), &G))) return rc;
      if (G > 0) mode = 2;
    } else if (graphs && tuned && !lanes_now && (use_lds(c) ? c->split == 0 : use_hbm(c))) {
      mode = 1;
    }
    int m = 1;                          // iterations in this replay
    if (mode == 1) {
      // short iterations go several to a replay: one host synchronisation
      // per replay instead of per iteration (on metro, ~0.9 ms iterations,
      // 8 per replay beat 2 by 0.9%; the iterations a replay runs past
      // convergence are gated off and cost little)
      m = c->graph_iters > 0 ? c->graph_iters
          : (c->last_iter_ms > 0 && c->last_iter_ms < 2.0) ? kMaxGraphIters : 1;
      // the loading's error flag and counters come back in the iteration block
      refresh_mirrors(c);
      if ((rc = iter_graph(c, K, m))) return rc;
      HIPCHK(c, hipGraphLaunch(c->g_iter, c->stream));
      c->graph_launches += 1;
      c->origin_pending = true;
      c->pending_Vn = c->V;
      c->stats.origin_blocks += (int64_t)(m - 1) * c->Z * c->V;
      c->stats.link_passes += m - 1;
      if (!use_lds(c)) c->stats.origin_delta = c->delta_mult;
    } else if (mode == 2) {
      const long long tasks = (long long)c->Z * G;
      if ((rc = lanes_reserve(c, tasks))) return rc;
      if ((rc = lanes_graph(c, make_links(c, false), G))) return rc;
      HIPCHK(c, hipGraphLaunch(c->g_iter, c->stream));
      c->graph_launches += 1;
      HIPCHK(c, hipStreamSynchronize(c->stream));
      bool fallback = false;
      if ((rc = absorb_lanes(c, c->pin_err, c->pin_cnt, tasks, c->V, std::chrono::steady_clock::now(),
                             &fallback)))
        return rc;
      if (fallback) {
        // the error flag kept every variant from stepping: load with a
        // per-origin kernel and run the link passes
        if ((rc = redo_per_origin(c, 0, c->V, c->var_on))) return rc;
        if ((rc = issue_link_passes(c, K))) return rc;
      }
    } else {
      if (tuned) {
        const long long ny = (long long)c->V * c->E;
        hipLaunchKernelGGL(k_iter_begin, dim3(grid_for(ny / kWave + 1)), dim3(kBlock), 0, c->stream,
                           c->err_dev, c->counters, c->y, ny);
      }
      HIPCHK(c, hipEventRecord(c->ev[2], c->stream));
      c->defer_origin = true;
      c->pre_cleared = tuned;
      rc = load_variants(c, 0, c->V, c->var_on, hon.data());
      c->defer_origin = false;
      c->pre_cleared = false;
      if (rc) return rc;
      HIPCHK(c, hipEventRecord(c->ev[3], c->stream));
      if (graphs) {
        if ((rc = link_graph(c, K))) return rc;
        HIPCHK(c, hipGraphLaunch(c->g_link, c->stream));
        c->graph_launches += 1;
      } else if ((rc = issue_link_passes(c, lanes_now ? make_links(c, false) : K))) {
        return rc;
      }
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if ((rc = absorb_pending(c))) return rc;
    c->stats.link_passes += 1;
    auto undecided = [&]() {
      return std::any_of(c->pin_st, c->pin_st + c->V, [](const VarState& s) { return s.need_more != 0; });
    };
    while (undecided()) {
      if ((rc = issue_link_passes(c, lanes_now ? make_links(c, false) : K, true, 1))) return rc;
      HIPCHK(c, hipStreamSynchronize(c->stream));
      c->stats.link_passes += 1;
    }
    std::copy(c->pin_st, c->pin_st + c->V, hs.begin());
    std::copy(c->pin_on, c->pin_on + c->V, hon.begin());
    const double it_ms =
        std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_it).count();
    c->last_iter_ms = it_ms / m;
    // (a captured iteration is timed as a whole, in link_ms)
    if (mode == 0) HIPCHK(c, hipEventElapsedTime(&aon, c->ev[2], c->ev[3]));
    c->stats.aon_ms += aon;
    c->stats.link_ms += std::max(0.0, it_ms - aon);
  }
  c->stats.graph_launches = c->graph_launches;
  c->graph_launches = 0;
  c->stats.total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
  if (results) {
    // VHT after the last step: sum x*c per variant on the device (fixed
    // order), read back with the variant states
    if (!c->vht) {
      int rc2 = dalloc(c, &c->vht, 2 * (size_t)c->V);
      if (rc2) return rc2;
    }
    launch_totals(c);
    HIPCHK(c, hipGetLastError());
    std::vector<double> tot(2 * (size_t)c->V);
    HIPCHK(c, hipMemcpyAsync(hs.data(), c->st, sizeof(VarState) * c->V, hipMemcpyDeviceToHost,
                             c->stream));
    HIPCHK(c, hipMemcpyAsync(tot.data(), c->vht, sizeof(double) * 2 * c->V, hipMemcpyDeviceToHost,
                             c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    for (int v = 0; v < c->V; ++v) {
      tapgpu_result& r = results[v];
      r.iterations = hs[v].iter;
      r.relgap = hs[v].relgap;
      r.objective = hs[v].objective;
      r.converged = (target_relgap > 0 && hs[v].relgap <= target_relgap) ? 1 : 0;
      r.vht = tot[2 * (size_t)v];
    }
  }
  return TAPGPU_OK;
}

int tapgpu_get_flows(tapgpu_ctx* c, int64_t variant, double* volumes, double* costs) {
  if (!c) return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  if (volumes)
    HIPCHK(c, hipMemcpy(volumes, c->x + (size_t)variant * c->E, sizeof(double) * c->E,
                        hipMemcpyDeviceToHost));
  if (costs)
    HIPCHK(c, hipMemcpy(costs, c->c + (size_t)variant * c->E, sizeof(double) * c->E,
                        hipMemcpyDeviceToHost));
  return TAPGPU_OK;
}

int tapgpu_get_totals(tapgpu_ctx* c, int64_t variant, double* objective, double* vht) {
  if (!c) return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  if (!c->initialised) return c->fail(TAPGPU_E_STATE, "tapgpu_fw_init was not called");
  if (!c->vht && (rc = dalloc(c, &c->vht, 2 * (size_t)c->V))) return rc;
  launch_totals(c);
  HIPCHK(c, hipGetLastError());
  double t[2];
  HIPCHK(c, hipMemcpyAsync(t, c->vht + 2 * variant, sizeof t, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (vht) *vht = t[0];
  if (objective) *objective = t[1];
  return TAPGPU_OK;
}

int tapgpu_set_links(tapgpu_ctx* c, int64_t variant, const double* capacity,
                     const double* free_flow_time) {
  if (!c) return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  if (free_flow_time)       // (costs must stay non-negative; checked before any change)
    for (int k = 0; k < c->E; ++k)
      if (!(free_flow_time[k] >= 0.0))
        return c->fail(TAPGPU_E_ARG, "link %d: negative or NaN free-flow time", k);
  const size_t off = (size_t)variant * c->E;
  if (capacity) {
    std::vector<unsigned char> pres(c->E);
    HIPCHK(c, hipMemcpy(pres.data(), c->present + off, c->E, hipMemcpyDeviceToHost));
    std::vector<double> cap(capacity, capacity + c->E);
    double minpos = DBL_MAX;
    for (int64_t k = 0; k < c->E; ++k)
      if (pres[k] && cap[k] > 0.0 && cap[k] < minpos) minpos = cap[k];
    for (auto& v : cap)
      if (!(v > 0.0)) v = minpos;
    HIPCHK(c, hipMemcpy(c->cap + off, cap.data(), sizeof(double) * c->E, hipMemcpyHostToDevice));
  }
  if (free_flow_time)
    HIPCHK(c, hipMemcpy(c->t0 + off, free_flow_time, sizeof(double) * c->E, hipMemcpyHostToDevice));
  // the volumes no longer belong to these links: fw_init comes next
  c->initialised = false;
  return TAPGPU_OK;
}

int tapgpu_get_trace(tapgpu_ctx* c, int64_t variant, tapgpu_iter* trace, int cap, int* count) {
  if (!c) return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  VarState s;
  HIPCHK(c, hipMemcpy(&s, c->st + variant, sizeof s, hipMemcpyDeviceToHost));
  const int held = std::min(s.iter, c->trace_cap);
  if (count) *count = s.iter;
  const int n = std::min(held, cap);
  if (trace && n > 0)
    HIPCHK(c, hipMemcpy(trace, c->trace + (size_t)variant * c->trace_cap, sizeof(tapgpu_iter) * n,
                        hipMemcpyDeviceToHost));
  return TAPGPU_OK;
}

int tapgpu_load_pred(tapgpu_ctx* c, int64_t variant, const int64_t* predlink, int64_t ld,
                     int64_t col_base, double* volumes) {
  if (!c || !predlink) return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  if ((rc = ensure_labels(c))) return rc;
  const int v = (int)variant;
  // predecessor links of zone origins into the variant's columns
  std::vector<int> hp((size_t)c->N * c->Pv, -1);
  for (int64_t node = 1; node <= c->N; ++node)
    for (int64_t j = 0; j < c->Z; ++j) {
      const int64_t e = predlink[(size_t)node * ld + col_base + c->zone_order[j]];
      if (e < -1 || e >= c->E)
        return c->fail(TAPGPU_E_ARG, "predecessor link %lld out of range", (long long)e);
      if (e >= 0 && c->h_head[e] != node - 1)
        return c->fail(TAPGPU_E_ARG, "predecessor link %lld of node %lld (origin %d) ends at node %d",
                       (long long)e, (long long)node, c->zone_order[j] + 1, c->h_head[e] + 1);
      hp[(size_t)(node - 1) * c->Pv + j] = (int)e;
    }
  HIPCHK(c, hipMemcpy2DAsync(c->pred + (size_t)v * c->Pv, c->P * sizeof(int), hp.data(),
                             c->Pv * sizeof(int), c->Pv * sizeof(int), c->N,
                             hipMemcpyHostToDevice, c->stream));
  std::vector<unsigned char> on(c->V, 0);
  on[v] = 1;
  unsigned char* d_on = nullptr;
  if ((rc = dalloc(c, &d_on, c->V))) return rc;
  rc = upload(c, d_on, on.data(), c->V);
  if (!rc) rc = aon_groups(c, v * c->Gv, c->Gv, v, 1, d_on, true);
  if (!rc && volumes) {
    const hipError_t e = hipMemcpy(volumes, c->y + (size_t)v * c->E, sizeof(double) * c->E,
                                   hipMemcpyDeviceToHost);
    if (e != hipSuccess) rc = c->fail(TAPGPU_E_HIP, "copy of volumes failed");
  }
  c->allocs.erase(std::remove(c->allocs.begin(), c->allocs.end(), (void*)d_on), c->allocs.end());
  (void)hipFree(d_on);
  return rc;
}

int tapgpu_get_iter(tapgpu_ctx* c, int64_t variant, int index, tapgpu_iter* rec) {
  if (!c || !rec) return TAPGPU_E_ARG;
  int rc = check_variant(c, variant);
  if (rc) return rc;
  if (index < 0 || index >= c->trace_cap) return c->fail(TAPGPU_E_ARG, "iteration %d not held", index);
  HIPCHK(c, hipMemcpy(rec, c->trace + (size_t)variant * c->trace_cap + index, sizeof(tapgpu_iter),
                      hipMemcpyDeviceToHost));
  return TAPGPU_OK;
}

int tapgpu_device_state(tapgpu_ctx* c, const double** d_volumes, const double** d_costs) {
  if (!c) return TAPGPU_E_ARG;
  if (d_volumes) *d_volumes = c->x;
  if (d_costs) *d_costs = c->c;
  return TAPGPU_OK;
}

int tapgpu_get_stats(tapgpu_ctx* c, tapgpu_stats* s) {
  if (!c || !s) return TAPGPU_E_ARG;
  *s = c->stats;
  return TAPGPU_OK;
}

int tapgpu_set_strategy(tapgpu_ctx* c, int strategy) {
  if (!c || strategy < 0 || strategy > 3) return TAPGPU_E_ARG;
  if (strategy == 2 && !c->lds_ok)
    return c->fail(TAPGPU_E_ARG, "network does not fit the one-origin-per-workgroup path");
  if (strategy == 3 && !c->hbm_ok)
    return c->fail(TAPGPU_E_ARG, "frontier bitmaps of this network do not fit LDS");
  const int before = c->strategy;
  c->strategy = strategy;
  // (tapgpu_sssp_noalloc allocates nothing, and takes this kernel then)
  if (!use_lds(c) && c->hbm_ok)
    if (int rc = alloc_hbm_mirrors(c, 1)) {
      c->strategy = before;
      return rc;
    }
  return TAPGPU_OK;
}

int tapgpu_set_origin_chase(tapgpu_ctx* c, int chase) {
  if (!c || chase < -1 || chase > 1024) return TAPGPU_E_ARG;
  c->chase = chase;
  return TAPGPU_OK;
}

int tapgpu_set_origin_delta(tapgpu_ctx* c, double mult) {
  if (!c || !(mult >= -1.0) || !std::isfinite(mult)) return TAPGPU_E_ARG;
  c->delta_mult = mult < 0 ? -1.0 : mult;
  return TAPGPU_OK;
}

double tapgpu_get_origin_delta(const tapgpu_ctx* c) { return c ? c->delta_mult : -2.0; }

int tapgpu_set_origin_split(tapgpu_ctx* c, int origins) {
  if (!c || origins < -1) return TAPGPU_E_ARG;
  c->split = origins;
  return TAPGPU_OK;
}

int tapgpu_get_origin_split(const tapgpu_ctx* c) { return c ? c->split : TAPGPU_E_ARG; }

int tapgpu_set_origin_block(tapgpu_ctx* c, int threads) {
  if (!c) return TAPGPU_E_ARG;
  if (threads == -1) {
    c->lds_block = -1;
    return TAPGPU_OK;
  }
  bool known = false;
  for (int b : kLdsBlocks) known = known || b == threads;
  if (!known) return c->fail(TAPGPU_E_ARG, "workgroup size %d: 1024, 512, 256 or -1", threads);
  if (c->N > kLdsPerThread * threads)
    return c->fail(TAPGPU_E_ARG, "%d threads per workgroup hold at most %d nodes", threads,
                   kLdsPerThread * threads);
  c->lds_block = threads;
  return TAPGPU_OK;
}

int tapgpu_get_origin_block(const tapgpu_ctx* c) {
  if (!c) return TAPGPU_E_ARG;
  return c->lds_block;
}

int tapgpu_get_origin_chase(const tapgpu_ctx* c) {
  if (!c) return TAPGPU_E_ARG;
  return c->chase;
}

int tapgpu_set_origin_queue(tapgpu_ctx* c, int entries) {
  if (!c || entries < -1) return TAPGPU_E_ARG;
  c->qcap = entries < 0 ? c->qcap_max : std::min(entries, c->qcap_max);
  c->qcap_auto = entries < 0;
  if (entries < 0) c->lds_block = -1;     // picked again with the workgroup size
  c->hqcap = entries < 0 ? c->hqcap_max : std::min(entries, c->hqcap_max);
  c->lanes_qcap = entries < 0 ? c->lanes_qcap_max : std::min(entries, c->lanes_qcap_max);
  return TAPGPU_OK;
}

int tapgpu_get_origin_queue(const tapgpu_ctx* c) {
  if (!c) return TAPGPU_E_ARG;
  tapgpu_ctx* m = const_cast<tapgpu_ctx*>(c);
  return use_hbm(m) ? c->hqcap : c->qcap;
}

int tapgpu_get_strategy(const tapgpu_ctx* c) {
  if (!c) return TAPGPU_E_ARG;
  tapgpu_ctx* m = const_cast<tapgpu_ctx*>(c);
  return use_lds(m) ? 2 : (use_hbm(m) ? 3 : 1);
}

int tapgpu_set_lanes(tapgpu_ctx* c, int min_active) {
  if (!c || min_active < -1) return TAPGPU_E_ARG;
  if (min_active != 0 && !c->lanes_ok)
    return c->fail(TAPGPU_E_ARG, "frontier bitmaps of this network do not fit LDS");
  c->lanes_min = min_active < 0 ? (c->V > 1 ? kLanesMinDefault : 0) : min_active;
  c->lanes_auto = min_active < 0;
  return TAPGPU_OK;
}

int tapgpu_get_lanes(const tapgpu_ctx* c) { return c ? c->lanes_min : TAPGPU_E_ARG; }

int tapgpu_set_lanes_delta(tapgpu_ctx* c, double mult) {
  if (!c || !(mult >= -1.0) || !std::isfinite(mult)) return TAPGPU_E_ARG;
  c->lanes_delta_mult = mult < 0 ? -1.0 : mult;
  return TAPGPU_OK;
}

double tapgpu_get_lanes_delta(const tapgpu_ctx* c) { return c ? c->lanes_delta_mult : -2.0; }

int tapgpu_set_profiling(tapgpu_ctx* c, int on) {
  if (!c) return TAPGPU_E_ARG;
  if (on && !c->ev[0])
    for (auto& e : c->ev) HIPCHK(c, hipEventCreate(&e));
  c->profiling = on != 0;
  return TAPGPU_OK;
}

}  // extern "C"

#include "tapgrad.inc"
#include "tapgreedy.inc"
