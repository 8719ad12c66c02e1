// Coarsening kernels for gfx950: heavy-edge candidate matching, grouping of
// the candidate pseudo-forest by walking to the root pairs (pointer jumping in
// deep trees), chunking into coarse vertices, and CSR contraction (relabel,
// per-row sort, merge of parallel edges) -- the work of gkway/coarsen.hpp.
// Every kernel is integer-exact and writes results that do not depend on the
// launch schedule: atomics are used only for commutative integer max/add or for
// slot reservation whose order is discarded by a later rank or sort.
#include <algorithm>

#include "kernels.hpp"
#include "prim.hpp"
#include "steal.hpp"
#include "../../include/gkway.h"

namespace gkd {

// About one lane per two to four entries: measured on MI355X, 4 lanes beat 8
// on meshes of average degree 4.5-6 (up to 24% at 2^24 vertices), 8 beat 16
// at degree 7-16 and 16 beat 32 at degree 16-22.
int lanes_for_degree(double avg) {
  if (avg <= 8.0) return 4;
  if (avg <= 16.0) return 8;
  if (avg <= 32.0) return 16;
  if (avg <= 64.0) return 32;
  return 64;
}

static inline int hip_status() { return hipGetLastError() == hipSuccess ? 0 : GK_ERR_HIP; }

// --------------------------------------------------------------- matching
constexpr int32_t kDegMore = 255;

// matching_with_score (gkway/coarsen.hpp:39-78) with S lanes per vertex: the
// lanes stride over the row, then reduce the packed preference
// (weight desc, neighbour degree asc, neighbour id asc) by xor-shuffles.
// Global thread slot gt serves vertex gt / S as lane gt % S of its group.
// deg (may be null): the neighbours' degrees as bytes, kDegMore for that many
// or more.
template <int S>
__device__ __forceinline__ void match_slot(int64_t gt, int32_t n, const int32_t* __restrict__ xadj,
                                           const int32_t* __restrict__ adj, const int32_t* __restrict__ w,
                                           const uint8_t* __restrict__ deg, int32_t* __restrict__ cand) {
  const int32_t v = static_cast<int32_t>(gt / S);
  const int sub = static_cast<int>(gt % S);
  if (v >= n) return;
  int bw = 0, bd = 0, bu = v;
  const int s = xadj[v], e = xadj[v + 1];
  auto better = [&](int wj, int d, int u) {
    if (wj > bw || (wj == bw && (d < bd || (d == bd && u < bu)))) { bw = wj; bd = d; bu = u; }
  };
  if (deg) {
    for (int j = s + sub; j < e; j += S) {
      const int u = adj[j];
      const int wj = w[j];
      int d = deg[u];
      if (d == kDegMore) d = xadj[u + 1] - xadj[u];
      better(wj, d, u);
    }
  } else {
    for (int j = s + sub; j < e; j += S) {
      const int u = adj[j];
      const int wj = w[j];
      better(wj, xadj[u + 1] - xadj[u], u);
    }
  }
#pragma unroll
  for (int o = S / 2; o > 0; o >>= 1) {
    const int ow = __shfl_xor(bw, o, S), od = __shfl_xor(bd, o, S), ou = __shfl_xor(bu, o, S);
    if (ow > bw || (ow == bw && (od < bd || (od == bd && ou < bu)))) { bw = ow; bd = od; bu = ou; }
  }
  if (sub == 0) cand[v] = bu;
}

template <int S, int B>
__global__ void __launch_bounds__(B) k_match(int32_t n, const int32_t* __restrict__ xadj,
                                             const int32_t* __restrict__ adj,
                                             const int32_t* __restrict__ w, const uint8_t* __restrict__ deg,
                                             int32_t* __restrict__ cand) {
  match_slot<S>(int64_t(xcd_block()) * B + threadIdx.x, n, xadj, adj, w, deg, cand);
}

// The same slots, taken from the work-stealing queues.
template <int S, int B>
__global__ void __launch_bounds__(B) k_match_ws(int32_t n, const int32_t* __restrict__ xadj,
                                                const int32_t* __restrict__ adj,
                                                const int32_t* __restrict__ w, const uint8_t* __restrict__ deg,
                                                int32_t* __restrict__ cand, unsigned long long* __restrict__ ctr) {
  const int64_t sweeps = (int64_t(n) * S + 63) / 64;
  steal_sweeps(ctr, sweeps, [&](int64_t sw) { match_slot<S>(sw * 64 + lane_id(), n, xadj, adj, w, deg, cand); });
}

template <int S, int B>
static void match_go(const DGraph& g, const uint8_t* deg, int32_t* cand, const Steal* ws, hipStream_t st) {
  const unsigned grid = grid_for(int64_t(g.n) * S, B);
  if (!ws) {
    gk_launch(k_match<S, B>, dim3(grid), dim3(B), 0, st, g.n, g.xadj, g.adj, g.w, deg, cand);
    return;
  }
  const unsigned pg = steal_grid(reinterpret_cast<const void*>(&k_match_ws<S, B>), B, *ws, grid);
  unsigned long long* ctr = nullptr;  // queues cleared and used only when the work has a tail
  if (steal_tail((int64_t(g.n) * S + 63) / 64, int64_t(pg) * (B / 64)) > 0) {
    fill<unsigned long long>(ws->ctr, 0ull, kStealWords, st);
    ctr = ws->ctr;
  }
  gk_launch(k_match_ws<S, B>, dim3(pg), dim3(B), 0, st, g.n, g.xadj, g.adj, g.w, deg, cand, ctr);
}

template <int B>
static void match_block(const DGraph& g, int lanes, const uint8_t* deg, int32_t* cand, const Steal* ws,
                        hipStream_t st) {
  switch (lanes) {
    case 1: match_go<1, B>(g, deg, cand, ws, st); break;
    case 2: match_go<2, B>(g, deg, cand, ws, st); break;
    case 4: match_go<4, B>(g, deg, cand, ws, st); break;
    case 8: match_go<8, B>(g, deg, cand, ws, st); break;
    case 16: match_go<16, B>(g, deg, cand, ws, st); break;
    case 32: match_go<32, B>(g, deg, cand, ws, st); break;
    default: match_go<64, B>(g, deg, cand, ws, st); break;
  }
}

// Every entry's degree is a random gather: the bound of the matching of a large
// mesh numbered without locality (2^22 vertices, 25 M entries: 372 us, 67 G/s
// out of 16 MB of row bounds).  From kDegTable vertices on the row bounds are
// larger than an XCD's 4 MB L2 and a table of bytes pays (the same mesh: 209 us
// and 9 for the table; a DAG of 1 M vertices, 32 us, is as fast without).
__global__ void __launch_bounds__(256) k_deg_table(int32_t n, const int32_t* __restrict__ xadj,
                                                   uint8_t* __restrict__ deg) {
  const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  int32_t x[5];
  uint32_t packed = 0;
#pragma unroll
  for (int j = 0; j < 5; ++j) x[j] = xadj[i + j <= n ? i + j : n];
#pragma unroll
  for (int j = 0; j < 4; ++j) packed |= uint32_t(min(x[j + 1] - x[j], kDegMore)) << (8 * j);
  *reinterpret_cast<uint32_t*>(deg + i) = packed;
}

int launch_deg_table(const DGraph& g, uint8_t* deg, hipStream_t st) {
  if (g.n <= 0) return 0;
  k_deg_table<<<grid_for(g.n, 1024), 256, 0, st>>>(g.n, g.xadj, deg);
  return hip_status();
}

int launch_match(const DGraph& g, int lanes, int block, const uint8_t* deg, int32_t* cand, hipStream_t st,
                 const Steal* ws) {
  if (g.n <= 0) return 0;
  switch (block) {
    case 128: match_block<128>(g, lanes, deg, cand, ws, st); break;
    case 512: match_block<512>(g, lanes, deg, cand, ws, st); break;
    default: match_block<256>(g, lanes, deg, cand, ws, st); break;
  }
  return hip_status();
}

// --------------------------------------------------------------- grouping
// The candidate graph {v, cand[v]} is a pseudo-forest whose only cycles are
// mutual pairs (or a self loop for an isolated vertex).  Pointer jumping
// finds for every vertex its root pair and the hop distance to it.
__global__ void __launch_bounds__(256) k_jump_init(int32_t n, const int32_t* __restrict__ cand,
                                                   int32_t* __restrict__ next, int32_t* __restrict__ dist) {
  const int64_t v = int64_t(xcd_block()) * 256 + threadIdx.x;
  if (v >= n) return;
  const int32_t c = cand[v];
  const bool root = cand[c] == v;
  next[v] = root ? int32_t(v) : c;
  dist[v] = root ? 0 : 1;
}

__global__ void __launch_bounds__(256) k_jump_round(int32_t n, const int32_t* __restrict__ next_in,
                                                    const int32_t* __restrict__ dist_in,
                                                    int32_t* __restrict__ next_out,
                                                    int32_t* __restrict__ dist_out,
                                                    int32_t* __restrict__ flags, int32_t round) {
  if (round > 0 && flags[round - 1] == 0) return;  // converged in an earlier round
  const int64_t v = int64_t(xcd_block()) * 256 + threadIdx.x;
  bool moved = false;
  if (v < n) {
    const int32_t nx = next_in[v];
    const int32_t nn = next_in[nx];
    if (nn == nx) {
      next_out[v] = nx;
      dist_out[v] = dist_in[v];
    } else {
      next_out[v] = nn;
      dist_out[v] = dist_in[v] + dist_in[nx];
      moved = true;
    }
  }
  if (ballot(moved) != 0 && lane_id() == 0) flags[round] = 1;
}

int launch_jump_init(int32_t n, const int32_t* cand, int32_t* next, int32_t* dist, hipStream_t st) {
  if (n <= 0) return 0;
  k_jump_init<<<grid_for(n, 256), 256, 0, st>>>(n, cand, next, dist);
  return hip_status();
}

int launch_jump_round(int32_t n, const int32_t* cand, const int32_t* next_in, const int32_t* dist_in,
                      int32_t* next_out, int32_t* dist_out, int32_t* flags, int32_t round,
                      hipStream_t st) {
  (void)cand;
  if (n <= 0) return 0;
  k_jump_round<<<grid_for(n, 256), 256, 0, st>>>(n, next_in, dist_in, next_out, dist_out, flags, round);
  return hip_status();
}

// One vertex more in the component of key, its root pair's larger id and so one
// of its members: the largest id above key in comp[key].x (0: none), its members
// counted in comp[key].y; returns v's (arbitrary) place among them.  Most
// vertices are not above their key, which saves their atomicMax (in a random
// numbering four of five).  Components are small, so the atomics rarely collide;
// lanes that share the first active lane's key (hubs, stars) are added with one
// atomic pair, since same-address atomics serialise.
__device__ __forceinline__ int32_t comp_add(int2* __restrict__ comp, int32_t key, int32_t v, bool live) {
  const uint64_t lm = ballot(live);
  if (lm == 0) return 0;
  const int first = __ffsll(static_cast<long long>(lm)) - 1;
  const uint64_t same = ballot(live && key == __shfl(key, first, 64));
  int32_t slot = 0;
  if (popc64(same) > 4) {
    int32_t base = 0;
    const int lead = 63 - __clzll(static_cast<long long>(same));  // ids grow with the lane: its id is the largest
    if (lane_id() == lead) {
      if (v > key) atomicMax(&comp[key].x, v);
      base = atomicAdd(&comp[key].y, popc64(same));
    }
    base = __shfl(base, lead, 64);
    if ((same >> lane_id()) & 1ull) return base + popc64(same & lanemask_lt());
  }
  if (live) {
    if (v > key) atomicMax(&comp[key].x, v);
    slot = atomicAdd(&comp[key].y, 1);
  }
  return slot;
}

// Grouping in one pass: every vertex follows its candidates to the mutual
// pair at the root of its tree (a self loop for an isolated vertex), counting
// hops.  Vertices sit on average less than one hop from their pair and
// rarely more than ten, so the walk reads cand[] about three times per vertex
// where the jumping rounds read and write pointer and distance arrays four
// times over.  On a 2^22-vertex mesh numbered at random (every read a cache
// line): 244 us with the component atomics, which bound it (327 us with an
// atomicMax for every vertex), where init and jumping rounds took 60 + 269 us
// and the label kernels 148 + 98 us (now 64).  flags[r] is set when some vertex
// is more than 2^r hops away, which tells the jumping rounds that the walk
// replaces; a vertex more than kWalkMax hops away sets flags[kWalkBits], and
// the caller falls back to the jumping rounds (long chains would make the walk
// linear).
__global__ void __launch_bounds__(256) k_walk(int32_t n, const int32_t* __restrict__ cand, int2* __restrict__ comp,
                                              int32_t* __restrict__ key_out, int32_t* __restrict__ dist,
                                              int32_t* __restrict__ slot, int32_t* __restrict__ flags) {
  const int64_t i = int64_t(xcd_block()) * 256 + threadIdx.x;
  const bool live = i < n;
  const int32_t v = live ? int32_t(i) : 0;
  int32_t a = v, d = 0, key = 0;
  if (live) {
    int32_t b = cand[a], c = cand[b];
    while (c != a && d <= kWalkMax) {
      a = b;
      b = c;
      c = cand[b];
      ++d;
    }
    key = max(a, b);
    if (c != a) {
      // Unresolved: a component of its own.  A key must be a member of its
      // component, or the members' places would not fit their groups.
      key = v;
      d = kWalkMax + 1;
    }
    key_out[v] = key;
    dist[v] = d;
  }
  const int32_t s = comp_add(comp, key, v, live);
  if (live) slot[v] = s;
  // highest power of two below the wave's largest distance
  int r = -1;
#pragma unroll
  for (int x = 0; x <= kWalkBits; ++x)
    if (ballot(d > (1 << x)) != 0) r = x;
  if (r >= 0 && lane_id() == 0 && flags[r] == 0) flags[r] = 1;
}

int launch_walk(int32_t n, const int32_t* cand, int2* comp, int32_t* key, int32_t* dist, int32_t* slot,
                int32_t* ctl, hipStream_t st) {
  if (n <= 0) return 0;
  Copies zero;
  zero.add(comp, nullptr, sizeof(int2) * size_t(n));
  zero.add(ctl, nullptr, sizeof(int32_t) * (kCtlInts + kRowCtlInts));
  const int rc = launch_copies(zero, st);
  if (rc) return rc;
  int32_t* flags = ctl + kCtlFlags;
  k_walk<<<grid_for(n, 256), 256, 0, st>>>(n, cand, comp, key, dist, slot, flags);
  return hip_status();
}

// The same from the jumping rounds' root pointers (root pair of every vertex).
__global__ void __launch_bounds__(256) k_comp_count(int32_t n, const int32_t* __restrict__ cand,
                                                    const int32_t* __restrict__ next, int2* __restrict__ comp,
                                                    int32_t* __restrict__ key_out, int32_t* __restrict__ slot) {
  const int64_t i = int64_t(xcd_block()) * 256 + threadIdx.x;
  const bool live = i < n;
  int32_t key = 0;
  if (live) {
    const int32_t r = next[i];
    key = max(r, cand[r]);
    key_out[i] = key;
  }
  const int32_t s = comp_add(comp, key, int32_t(i), live);
  if (live) slot[i] = s;
}

int launch_comp_count(int32_t n, const int32_t* cand, const int32_t* next, int2* comp, int32_t* key, int32_t* slot,
                      hipStream_t st) {
  if (n <= 0) return 0;
  fill<int2>(comp, int2{0, 0}, n, st);
  k_comp_count<<<grid_for(n, 256), 256, 0, st>>>(n, cand, next, comp, key, slot);
  return hip_status();
}

// label[v] = the largest id of v's component; size[label] = its member count,
// 0 for every other index.  key may be label.
__global__ void __launch_bounds__(256) k_label_size(int32_t n, const int32_t* key, const int2* __restrict__ comp,
                                                    int32_t* label, int32_t* __restrict__ size) {
  const int64_t v = int64_t(xcd_block()) * 256 + threadIdx.x;
  if (v >= n) return;
  const int32_t k = key[v];
  const int2 c = comp[k];
  const int32_t l = max(c.x, k);
  label[v] = l;
  size[v] = l == int32_t(v) ? c.y : 0;
}

int launch_label_size(int32_t n, const int32_t* key, const int2* comp, int32_t* label, int32_t* size,
                      hipStream_t st) {
  if (n <= 0) return 0;
  k_label_size<<<grid_for(n, 256), 256, 0, st>>>(n, key, comp, label, size);
  return hip_status();
}

// size[l] = vertices with label l, slot[v] = v's (arbitrary) place among them,
// for labels that come without a grouping and so from a caller: those outside
// [0, n) are left out and flagged (kCtlFlags, and [1], so that nobody orders
// the members).
__global__ void __launch_bounds__(256) k_label_count(int32_t n, const int32_t* __restrict__ label,
                                                     int32_t* __restrict__ size, int32_t* __restrict__ slot,
                                                     int32_t* __restrict__ ctl) {
  const int64_t v = int64_t(xcd_block()) * 256 + threadIdx.x;
  const int32_t l = v < n ? label[v] : -1;
  const bool live = uint32_t(l) < uint32_t(n);
  const uint64_t lm = ballot(live);
  if (ballot(v < n && !live) != 0 && lane_id() == 0) {
    ctl[1] = 1;
    ctl[kCtlFlags] = 1;
  }
  if (lm == 0) return;
  // one atomic, by the first live lane, for the lanes that share its label
  const int first = __ffsll(static_cast<long long>(lm)) - 1;
  const int32_t lf = __shfl(l, first, 64);
  const uint64_t same = ballot(live && l == lf);
  if (popc64(same) > 4) {
    int32_t base = 0;
    if (lane_id() == first) base = atomicAdd(&size[lf], popc64(same));
    base = __shfl(base, first, 64);
    if ((same >> lane_id()) & 1ull) {
      slot[v] = base + popc64(same & lanemask_lt());
      return;
    }
  }
  if (live) slot[v] = atomicAdd(&size[l], 1);
}

int launch_label_count(int32_t n, const int32_t* label, int32_t* size, int32_t* slot, int32_t* ctl, hipStream_t st) {
  Copies zero;
  zero.add(ctl, nullptr, sizeof(int32_t) * (kCtlInts + kRowCtlInts));
  if (n > 0) zero.add(size, nullptr, sizeof(int32_t) * size_t(n));
  const int rc = launch_copies(zero, st);
  if (rc || n <= 0) return rc;
  k_label_count<<<grid_for(n, 256), 256, 0, st>>>(n, label, size, slot, ctl);
  return hip_status();
}

// --------------------------------------------------------------- members
// Order of the vertices by (label, stamp, id) and their chunks of at most G,
// by counting instead of sorting: the member counts are scanned over the
// labels (first place and first coarse id of every group), every vertex is
// written to its group's places in arbitrary order, and then finds its rank
// among its group's members.  Groups average 3 to 6 members, so the quadratic
// ranking is cheaper than the four 8-bit passes of a radix sort over (label,
// stamp).  2^22 vertices numbered at random: scan 35, scatter 190, rank 79 us,
// where keys, passes, chunk flags and ids took 530 us and the gathers of the
// members' rows and weights, which the records now carry, another 120 us.  The
// scatter is bound by its random 32-byte writes.  A group of more than kRankMax
// members sets ctl[1] and the caller sorts instead (at 512 members for every
// vertex the ranking costs about what the passes cost).
constexpr int kSizeIPT = 8;
constexpr int kSizeTile = 256 * kSizeIPT;
constexpr int64_t kSizeDirect = 8192;  // up to this many tiles every block sums the tiles before it itself

__device__ __forceinline__ int32_t chunks_of(int32_t size, int32_t G) {
  return size == 0 ? 0 : (size - 1) / G + 1;
}

// Members and chunks of each tile.
__global__ void __launch_bounds__(256) k_size_reduce(int32_t n, const int32_t* __restrict__ size, int32_t G,
                                                     int2* __restrict__ partial, int32_t* __restrict__ ctl) {
  __shared__ int2 ws[4];
  const int64_t base = int64_t(blockIdx.x) * kSizeTile;
  int32_t m = 0, c = 0, big = 0;
#pragma unroll
  for (int j = 0; j < kSizeIPT; ++j) {
    const int64_t i = base + j * 256 + threadIdx.x;
    if (i < n) {
      const int32_t s = size[i];
      m += s;
      c += chunks_of(s, G);
      big |= s > kRankMax;
    }
  }
  if (ballot(big) != 0 && lane_id() == 0) ctl[1] = 1;
  m = wave_sum(m);
  c = wave_sum(c);
  if (lane_id() == 0) ws[threadIdx.x >> 6] = make_int2(m, c);
  __syncthreads();
  if (threadIdx.x == 0)
    partial[blockIdx.x] = make_int2(ws[0].x + ws[1].x + ws[2].x + ws[3].x, ws[0].y + ws[1].y + ws[2].y + ws[3].y);
}

// Many tiles: their exclusive sums, in place, by one block.
__global__ void __launch_bounds__(256) k_size_mid(int64_t nb, int2* __restrict__ partial) {
  __shared__ int lds[8];
  int32_t rm = 0, rc = 0;
  for (int64_t b0 = 0; b0 < nb; b0 += 256) {
    const int64_t b = b0 + threadIdx.x;
    const int2 p = b < nb ? partial[b] : make_int2(0, 0);
    int tm, tc;
    const int em = block_excl_scan_256(p.x, &tm, lds);
    const int ec = block_excl_scan_256(p.y, &tc, lds);
    if (b < nb) partial[b] = make_int2(rm + em, rc + ec);
    rm += tm;
    rc += tc;
  }
}

// offc[l] = first place and first coarse id of label l's group, offc[n] the
// totals; ctl[0] (and the host's copy) = the number of coarse ids; words 1.. of host
// = the flags.
__global__ void __launch_bounds__(256) k_size_apply(int32_t n, const int32_t* __restrict__ size, int32_t G,
                                                    const int2* __restrict__ partial, int scanned,
                                                    int2* __restrict__ offc, int32_t* __restrict__ ctl,
                                                    const HostWords host) {
  __shared__ int lds[8];
  int32_t pm = 0, pc = 0;
  if (scanned) {
    const int2 p = partial[blockIdx.x];
    pm = p.x;
    pc = p.y;
  } else {
    int32_t sm = 0, sc = 0;
    for (int64_t b = threadIdx.x; b < int64_t(blockIdx.x); b += 256) {
      const int2 p = partial[b];
      sm += p.x;
      sc += p.y;
    }
    int t;
    (void)block_excl_scan_256(sm, &t, lds);
    pm = t;
    (void)block_excl_scan_256(sc, &t, lds);
    pc = t;
  }
  const int64_t base = int64_t(blockIdx.x) * kSizeTile + int64_t(threadIdx.x) * kSizeIPT;
  int32_t s[kSizeIPT];
  int32_t m = 0, c = 0;
#pragma unroll
  for (int j = 0; j < kSizeIPT; ++j) {
    s[j] = base + j < n ? size[base + j] : 0;
    m += s[j];
    c += chunks_of(s[j], G);
  }
  int t;
  int32_t rm = pm + block_excl_scan_256(m, &t, lds);
  int32_t rc = pc + block_excl_scan_256(c, &t, lds);
#pragma unroll
  for (int j = 0; j < kSizeIPT; ++j) {
    if (base + j < n) offc[base + j] = make_int2(rm, rc);
    rm += s[j];
    rc += chunks_of(s[j], G);
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 255) {
    offc[n] = make_int2(rm, rc);
    ctl[0] = rc;
    int32_t word[kCtlInts];  // read first: the loads would wait for the stores
    word[0] = rc;
#pragma unroll
    for (int i = 1; i < kCtlInts; ++i) word[i] = ctl[i];
#pragma unroll
    for (int i = 0; i < kCtlInts; ++i) tell(host, i, word[i]);
  }
}

int64_t size_partials(int64_t n) { return (n + kSizeTile - 1) / kSizeTile; }

int launch_size_scan(int32_t n, const int32_t* size, int32_t G, int2* partial, int2* offc, int32_t* ctl,
                     const HostWords& host, hipStream_t st) {
  if (n <= 0) return 0;
  const int64_t nb = size_partials(n);
  k_size_reduce<<<unsigned(nb), 256, 0, st>>>(n, size, G, partial, ctl);
  const bool mid = nb > kSizeDirect;
  if (mid) k_size_mid<<<1, 256, 0, st>>>(nb, partial);
  k_size_apply<<<unsigned(nb), 256, 0, st>>>(n, size, G, partial, mid ? 1 : 0, offc, ctl, host);
  return hip_status();
}

// Every vertex to a place of its group, with what its later readers need (its
// row and weight), so that they read consecutive records: memb[2p] = (vertex,
// stamp, group's first place, group's first coarse id), memb[2p + 1] = (row
// start, row length, weight, members of the group).
__global__ void __launch_bounds__(256) k_member_scatter(int32_t n, const int32_t* __restrict__ label,
                                                        const int32_t* __restrict__ stamp,
                                                        const int32_t* __restrict__ slot,
                                                        const int2* __restrict__ offc,
                                                        const int32_t* __restrict__ xadj,
                                                        const int32_t* __restrict__ vw, int4* __restrict__ memb) {
  const int64_t v = int64_t(xcd_block()) * 256 + threadIdx.x;
  if (v >= n) return;
  const int32_t l = label[v];
  if (uint32_t(l) >= uint32_t(n)) return;  // flagged by k_label_count
  const int2 oc = offc[l];
  const int32_t cnt = offc[l + 1].x - oc.x;
  int32_t a = 0, d = 0;
  if (xadj) {
    a = xadj[v];
    d = xadj[v + 1] - a;
  }
  const int64_t p = int64_t(oc.x) + slot[v];
  memb[2 * p] = make_int4(int32_t(v), stamp ? stamp[v] : 0, oc.x, oc.y);
  memb[2 * p + 1] = make_int4(a, d, vw ? vw[v] : 0, cnt);
}

// Rank of every member in its group, and with it the vertex order, the coarse
// ids, the first place of every coarse id and the members' rows and weights
// in that order (each output but cptr may be null).
__global__ void __launch_bounds__(256) k_member_rank(int32_t n, const int4* __restrict__ memb, int32_t G,
                                                     const int32_t* __restrict__ ctl, int32_t* __restrict__ order,
                                                     int32_t* __restrict__ cmap, int32_t* __restrict__ cptr,
                                                     int2* __restrict__ mrow, int32_t* __restrict__ mvw) {
  const int64_t i = int64_t(xcd_block()) * 256 + threadIdx.x;
  if (i >= n) return;
  if (ctl[1]) return;  // some group is too large: the caller sorts
  if (i == n - 1) cptr[ctl[0]] = n;
  const int4 a = memb[2 * i], b = memb[2 * i + 1];
  const int32_t cnt = b.w;
  int32_t r = 0;
  for (int32_t j = 0; j < cnt; ++j) {
    const int4 o = memb[2 * (int64_t(a.z) + j)];
    r += (o.y < a.y || (o.y == a.y && o.x < a.x)) ? 1 : 0;
  }
  const int32_t p = a.z + r;
  const int32_t q = r / G;
  if (cmap) cmap[a.x] = a.w + q;
  if (r - q * G == 0) cptr[a.w + q] = p;
  if (order) order[p] = a.x;
  if (mrow) mrow[p] = make_int2(b.x, b.y);
  if (mvw) mvw[p] = b.z;
}

int launch_members(int32_t n, const int32_t* label, const int32_t* stamp, const int32_t* slot, const int2* offc,
                   const int32_t* xadj, const int32_t* vw, int4* memb, int32_t G, const int32_t* ctl,
                   int32_t* order, int32_t* cmap, int32_t* cptr, int2* mrow, int32_t* mvw, hipStream_t st) {
  if (n <= 0) return 0;
  k_member_scatter<<<grid_for(n, 256), 256, 0, st>>>(n, label, stamp, slot, offc, xadj, vw, memb);
  k_member_rank<<<grid_for(n, 256), 256, 0, st>>>(n, memb, G, ctl, order, cmap, cptr, mrow, mvw);
  return hip_status();
}

// Grouping, coarse ids and members of a small graph by one workgroup, in LDS:
// the walk, the component counts, the scan over the labels, the places and the
// ranks are the steps of the kernels above.  Their eight launches on a few
// thousand vertices took 24 us and the gaps between them as much again.
constexpr int kSmallThreads = 1024;
constexpr int kSmallPer = kSmallGroup / kSmallThreads;
static_assert(kSmallPer == 4 && kSmallGroup <= 65536, "16-bit ids, four vertices a thread");

// Exclusive scan over the block (16 waves); *tot the sum.  ws: 16 ints, not
// read by the scan before after this one's first barrier.
__device__ __forceinline__ int small_scan(int x, int* tot, int32_t* ws) {
  const int wave = threadIdx.x >> 6;
  const int incl = wave_incl_scan(x);
  if (lane_id() == 63) ws[wave] = incl;
  __syncthreads();
  int below = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kSmallThreads / 64; ++w) {
    below += w < wave ? ws[w] : 0;
    all += ws[w];
  }
  *tot = all;
  return incl - x + below;
}

__global__ void __launch_bounds__(kSmallThreads) k_group_small(int32_t n, const int32_t* __restrict__ cand, int32_t G,
                                                               const int32_t* __restrict__ xadj,
                                                               const int32_t* __restrict__ vw,
                                                               int32_t* __restrict__ order,
                                                               int32_t* __restrict__ cmap, int32_t* __restrict__ cptr,
                                                               int2* __restrict__ mrow, int32_t* __restrict__ mvw,
                                                               int32_t* __restrict__ ctl, const HostWords host) {
  __shared__ uint16_t cd[kSmallGroup];                     // candidates; then the vertices by place
  __shared__ int32_t mx[kSmallGroup], ct[kSmallGroup];     // by key: largest id above it, members
  __shared__ uint16_t sz[kSmallGroup];                     // by label: members,
  __shared__ uint16_t off[kSmallGroup], ch[kSmallGroup];   // first place, first coarse id
  __shared__ uint8_t ds[kSmallGroup];
  __shared__ int32_t wsm[16], wsc[16];
  __shared__ int32_t deepest, largest;
  const int t = threadIdx.x;
  int32_t row[kSmallPer], len[kSmallPer], wt[kSmallPer];
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    const int32_t v = t + j * kSmallThreads;
    mx[v] = 0;
    ct[v] = 0;
    row[j] = len[j] = wt[j] = 0;
    if (v < n) {
      cd[v] = uint16_t(cand[v]);
      row[j] = xadj[v];
      len[j] = xadj[v + 1] - row[j];
      wt[j] = vw[v];
    }
  }
  if (t == 0) deepest = largest = 0;
  for (int i = t; i < kCtlInts + kRowCtlInts; i += kSmallThreads) ctl[i] = 0;
  __syncthreads();
  int32_t key[kSmallPer], slot[kSmallPer];
  int far = 0;
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    const int32_t v = t + j * kSmallThreads;
    key[j] = slot[j] = 0;
    if (v >= n) continue;
    int32_t a = v, d = 0, b = cd[a], c = cd[b];
    while (c != a && d <= kWalkMax) {
      a = b;
      b = c;
      c = cd[b];
      ++d;
    }
    int32_t k = max(a, b);
    if (c != a) {
      k = v;
      d = kWalkMax + 1;
    }
    key[j] = k;
    ds[v] = uint8_t(d);
    far = max(far, d);
    if (v > k) atomicMax(&mx[k], v);
    slot[j] = atomicAdd(&ct[k], 1);
  }
  far = wave_max(far);
  if (lane_id() == 0) atomicMax(&deepest, far);
  __syncthreads();
  int32_t label[kSmallPer];
  int big = 0;
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    const int32_t v = t + j * kSmallThreads;
    label[j] = max(mx[key[j]], key[j]);
    const int32_t s = v < n && label[j] == v ? ct[key[j]] : 0;
    sz[v] = uint16_t(s);
    big = max(big, s);
  }
  big = wave_max(big);
  if (lane_id() == 0) atomicMax(&largest, big);
  __syncthreads();
  {
    int32_t s[kSmallPer];
    int m = 0, c = 0;
#pragma unroll
    for (int j = 0; j < kSmallPer; ++j) {
      s[j] = sz[t * kSmallPer + j];
      m += s[j];
      c += chunks_of(s[j], G);
    }
    int tm, tc;
    int32_t rm = small_scan(m, &tm, wsm), rc = small_scan(c, &tc, wsc);
#pragma unroll
    for (int j = 0; j < kSmallPer; ++j) {
      off[t * kSmallPer + j] = uint16_t(rm);
      ch[t * kSmallPer + j] = uint16_t(rc);
      rm += s[j];
      rc += chunks_of(s[j], G);
    }
    if (t == 0) {
      cptr[tc] = n;
      ctl[0] = tc;
      tell(host, 0, tc);
      tell(host, 1, largest > kRankMax ? 1 : 0);
#pragma unroll
      for (int b = 0; b <= kWalkBits; ++b) tell(host, kCtlFlags + b, deepest > (1 << b) ? 1 : 0);
    }
  }
  __syncthreads();
  uint16_t* mem = cd;  // the walk has ended
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    const int32_t v = t + j * kSmallThreads;
    if (v < n) mem[off[label[j]] + slot[j]] = uint16_t(v);
  }
  __syncthreads();
  if (largest > kRankMax) return;
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    const int32_t v = t + j * kSmallThreads;
    if (v >= n) continue;
    const int32_t l = label[j], base = off[l], d = ds[v];
    int32_t r = 0;
    for (int32_t i = base; i < base + sz[l]; ++i) {
      const int32_t u = mem[i];
      r += (ds[u] < d || (ds[u] == d && u < v)) ? 1 : 0;
    }
    const int32_t p = base + r, q = r / G;
    cmap[v] = ch[l] + q;
    if (r - q * G == 0) cptr[ch[l] + q] = p;
    if (order) order[p] = v;
    mrow[p] = make_int2(row[j], len[j]);
    mvw[p] = wt[j];
  }
}

int launch_group_small(int32_t n, const int32_t* cand, int32_t G, const int32_t* xadj, const int32_t* vw,
                       int32_t* order, int32_t* cmap, int32_t* cptr, int2* mrow, int32_t* mvw, int32_t* ctl,
                       const HostWords& host, hipStream_t st) {
  if (n <= 0 || n > kSmallGroup) return GK_ERR_LIMIT;
  k_group_small<<<1, kSmallThreads, 0, st>>>(n, cand, G, xadj, vw, order, cmap, cptr, mrow, mvw, ctl, host);
  return hip_status();
}

// The members' rows by group, in arbitrary order inside a group, and each
// group's first place, for readers to whom that order is all the same.
__global__ void __launch_bounds__(256) k_member_place(int32_t n, const int32_t* __restrict__ label,
                                                      const int32_t* __restrict__ slot,
                                                      const int2* __restrict__ offc,
                                                      const int32_t* __restrict__ xadj,
                                                      const int32_t* __restrict__ ctl, int32_t* __restrict__ cptr,
                                                      int2* __restrict__ mrow) {
  const int64_t v = int64_t(xcd_block()) * 256 + threadIdx.x;
  if (v >= n) return;
  const int32_t a = xadj[v], l = label[v];
  if (uint32_t(l) < uint32_t(n)) mrow[int64_t(offc[l].x) + slot[v]] = make_int2(a, xadj[v + 1] - a);
  // index v as a label: the first place of its group, if it has members
  const int2 o = offc[v];
  if (offc[v + 1].x > o.x) cptr[o.y] = o.x;
  if (v == n - 1) cptr[ctl[0]] = n;
}

int launch_member_place(int32_t n, const int32_t* label, const int32_t* slot, const int2* offc, const int32_t* xadj,
                        const int32_t* ctl, int32_t* cptr, int2* mrow, hipStream_t st) {
  if (n <= 0) return 0;
  k_member_place<<<grid_for(n, 256), 256, 0, st>>>(n, label, slot, offc, xadj, ctl, cptr, mrow);
  return hip_status();
}

// The members' rows and weights in a given vertex order (after a sort).
__global__ void __launch_bounds__(256) k_member_rows(int32_t n, const int32_t* __restrict__ order,
                                                     const int32_t* __restrict__ xadj,
                                                     const int32_t* __restrict__ vw, int2* __restrict__ mrow,
                                                     int32_t* __restrict__ mvw) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const int32_t v = order[i];
  if (mrow) {
    const int32_t a = xadj[v];
    mrow[i] = make_int2(a, xadj[v + 1] - a);
  }
  if (mvw) mvw[i] = vw[v];
}

int launch_member_rows(int32_t n, const int32_t* order, const int32_t* xadj, const int32_t* vw, int2* mrow,
                       int32_t* mvw, hipStream_t st) {
  if (n <= 0) return 0;
  k_member_rows<<<grid_for(n, 256), 256, 0, st>>>(n, order, xadj, vw, mrow, mvw);
  return hip_status();
}

// --------------------------------------------------------------- sorted order
// The order by a radix sort of (label, stamp), for groups too large to rank.
__global__ void __launch_bounds__(256) k_make_keys(int32_t n, const int32_t* __restrict__ label,
                                                   const int32_t* __restrict__ dist, int sbits,
                                                   uint64_t* __restrict__ keys, int32_t* __restrict__ ids) {
  const int64_t v = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (v >= n) return;
  keys[v] = (uint64_t(uint32_t(label[v])) << sbits) | uint64_t(uint32_t(dist[v]));
  ids[v] = int32_t(v);
}

int launch_make_keys(int32_t n, const int32_t* label, const int32_t* dist, int sbits,
                     uint64_t* keys, int32_t* ids, hipStream_t st) {
  if (n <= 0) return 0;
  k_make_keys<<<grid_for(n, 256), 256, 0, st>>>(n, label, dist, sbits, keys, ids);
  return hip_status();
}

// --------------------------------------------------------------- chunking
// constraint_group_size + coarse numbering (gkway/coarsen.hpp:361-421,
// 120-155): in the sorted order, an item starts a chunk when its rank in its
// group is a multiple of G; coarse ids are the running count of chunk starts.
__global__ void __launch_bounds__(256) k_group_start(int32_t n, const uint64_t* __restrict__ skeys, int sbits,
                                                     int32_t* __restrict__ gstart) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const uint64_t lab = skeys[i] >> sbits;
  if (i == 0 || (skeys[i - 1] >> sbits) != lab) gstart[lab] = int32_t(i);
}

struct ChunkFlag {
  const uint64_t* skeys;
  const int32_t* gstart;
  int sbits;
  int32_t G;
  __device__ int operator()(int64_t i) const {
    const int32_t r = int32_t(i) - gstart[skeys[i] >> sbits];
    return (r % G) == 0 ? 1 : 0;
  }
};
struct StoreExcl {
  int32_t* out;
  __device__ void operator()(int64_t i, int excl, int) const { out[i] = excl; }
};

__global__ void __launch_bounds__(256) k_cmap(int32_t n, const uint64_t* __restrict__ skeys,
                                              const int32_t* __restrict__ sids, int sbits,
                                              const int32_t* __restrict__ gstart, int32_t G,
                                              const int32_t* __restrict__ excl,
                                              int32_t* __restrict__ cmap, int32_t* __restrict__ cptr) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const int32_t r = int32_t(i) - gstart[skeys[i] >> sbits];
  const int f = (r % G) == 0;
  const int32_t c = f ? excl[i] : excl[i] - 1;
  cmap[sids[i]] = c;
  if (f) cptr[c] = int32_t(i);
  if (i == n - 1) cptr[c + 1] = n;
}

int launch_cluster(int32_t n, const uint64_t* skeys, const int32_t* sids, int sbits, int32_t G, int32_t* gstart,
                   int32_t* flagscan, int32_t* cmap, int32_t* cptr, int32_t* nc_dev, int32_t* scratch,
                   hipStream_t st) {
  if (n <= 0) return 0;
  k_group_start<<<grid_for(n, 256), 256, 0, st>>>(n, skeys, sbits, gstart);
  int rc = scan(n, ChunkFlag{skeys, gstart, sbits, G}, StoreExcl{flagscan}, nc_dev, scratch, st);
  if (rc) return GK_ERR_HIP;
  k_cmap<<<grid_for(n, 256), 256, 0, st>>>(n, skeys, sids, sbits, gstart, G, flagscan, cmap, cptr);
  return hip_status();
}

// cal_coarsen_vwgt (gkway/coarsen.hpp:157-171) as an ordered sum over the
// (at most G) members of each chunk, their weights in member order; no
// atomics, destination fully written.  With ctl the chunks are counted there
// (nc: no more than that), and nothing is done where the members are not in
// order (ctl[1]).
__global__ void __launch_bounds__(256) k_cvwgt(int32_t nc, const int32_t* __restrict__ ctl,
                                               const int32_t* __restrict__ cptr,
                                               const int32_t* __restrict__ mvw, int32_t* __restrict__ cvw) {
  const int64_t c = int64_t(xcd_block()) * 256 + threadIdx.x;
  if (ctl) nc = ctl[1] ? 0 : min(nc, ctl[0]);
  if (c >= nc) return;
  int32_t s = 0;
  for (int32_t j = cptr[c]; j < cptr[c + 1]; ++j) s += mvw[j];
  cvw[c] = s;
}

int launch_cvwgt(int32_t nc, const int32_t* ctl, const int32_t* cptr, const int32_t* mvw, int32_t* cvw,
                 hipStream_t st) {
  if (nc <= 0) return 0;
  k_cvwgt<<<grid_for(nc, 256), 256, 0, st>>>(nc, ctl, cptr, mvw, cvw);
  return hip_status();
}

// --------------------------------------------------------------- contraction
// Per coarse row: the upper bound of its entries (sum of member degrees), its
// class (16, 32 or 64 lanes, a workgroup, or the global sort), and room for
// them in the temporary rows (toff).  Row ids are appended to one list per
// class, each with its member range in member order (desc: first member,
// member count); a row of the last two classes leaves its bound in len until
// it is merged.  The members' rows (mrow) and weights (mvw, with cvw the
// coarse weights' destination; both may be null) lie in member order, so a
// row's members are consecutive reads.  A block takes kBoundsPer rows a thread
// and adds to the class counters and the room once: same-address atomics
// serialise, and with one row a thread they, not the reads, were the time
// (2^22 vertices, 1 M rows: 52 us with one, 23 us with four rows a thread and
// the counters kRowCtlStride ints apart).  Up to kRowsAllMax rows there are few
// blocks, and one row a thread is the shorter chain (20000 rows: 9 us with
// four).
template <int kBoundsPer>
__global__ void __launch_bounds__(256) k_row_bounds(int32_t nc, const int32_t* __restrict__ cptr,
                                                    const int2* __restrict__ mrow, const int32_t* __restrict__ mvw,
                                                    int32_t* __restrict__ toff, int32_t* __restrict__ lists,
                                                    int2* __restrict__ desc, int32_t* __restrict__ len,
                                                    int32_t* __restrict__ cvw, int32_t* __restrict__ cnt) {
  // per class: rows of each wave and pass; then entries likewise
  __shared__ int wcnt[kRowClasses][4 * kBoundsPer];
  __shared__ int wub[4 * kBoundsPer];
  __shared__ int base[kRowClasses + 1];
  const int wave = threadIdx.x >> 6;
  const uint64_t lt = lanemask_lt();
  const int64_t c0 = int64_t(xcd_block()) * (256 * kBoundsPer) + threadIdx.x;
  int32_t m0[kBoundsPer], nm[kBoundsPer], ub[kBoundsPer], pre[kBoundsPer];
  int cls[kBoundsPer];
  int big = 0;
#pragma unroll
  for (int r = 0; r < kBoundsPer; ++r) {
    const int64_t c = c0 + r * 256;
    cls[r] = -1;
    m0[r] = nm[r] = ub[r] = 0;
    if (c < nc) {
      m0[r] = cptr[c];
      nm[r] = cptr[c + 1] - m0[r];
      int32_t s = 0, x = 0;
      for (int32_t j = m0[r]; j < m0[r] + nm[r]; ++j) {
        s += mrow[j].y;
        if (mvw) x += mvw[j];
      }
      if (mvw) cvw[c] = x;
      ub[r] = s;
      cls[r] = s <= 16 ? 0 : (s <= 32 ? 1 : (s <= 64 ? 2 : (s <= kMidMax ? 3 : 4)));
      if (cls[r] == 4) big += s;
      if (cls[r] >= 3) len[c] = s;
    }
    const int incl = wave_incl_scan(ub[r]);
    pre[r] = incl - ub[r];
    if (lane_id() == 63) wub[r * 4 + wave] = incl;
#pragma unroll
    for (int k = 0; k < kRowClasses; ++k) {
      const int x = popc64(ballot(cls[r] == k));
      if (lane_id() == 0) wcnt[k][r * 4 + wave] = x;
    }
  }
  if (ballot(big > 0) != 0) {
    big = wave_sum(big);
    if (lane_id() == 0) atomicAdd(&cnt[kRowBigEntries * kRowCtlStride], big);
  }
  __syncthreads();
  if (threadIdx.x <= kRowClasses) {
    int* w = threadIdx.x < kRowClasses ? wcnt[threadIdx.x] : wub;
    int run = 0;
#pragma unroll
    for (int i = 0; i < 4 * kBoundsPer; ++i) {
      const int q = w[i];
      w[i] = run;
      run += q;
    }
    base[threadIdx.x] = run ? atomicAdd(&cnt[threadIdx.x * kRowCtlStride], run) : 0;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kBoundsPer; ++r) {
    const int64_t c = c0 + r * 256;
    uint64_t mine = 0;
#pragma unroll
    for (int k = 0; k < kRowClasses; ++k) {
      const uint64_t m = ballot(cls[r] == k);
      if (cls[r] == k) mine = m;
    }
    if (c >= nc) continue;
    toff[c] = base[kRowClasses] + wub[r * 4 + wave] + pre[r];
    const int64_t slot = int64_t(cls[r]) * nc + base[cls[r]] + wcnt[cls[r]][r * 4 + wave] + popc64(mine & lt);
    lists[slot] = int32_t(c);
    desc[slot] = make_int2(m0[r], nm[r]);
  }
}

int launch_contract_bounds(int32_t nc, const int32_t* cptr, const int2* mrow, const int32_t* mvw, int32_t* toff,
                           int32_t* lists, int2* desc, int32_t* len, int32_t* cvw, int32_t* cnt, hipStream_t st) {
  if (nc <= 0) return 0;
  if (nc <= kRowsAllMax)
    k_row_bounds<1><<<grid_for(nc, 256), 256, 0, st>>>(nc, cptr, mrow, mvw, toff, lists, desc, len, cvw, cnt);
  else
    k_row_bounds<4><<<grid_for(nc, 1024), 256, 0, st>>>(nc, cptr, mrow, mvw, toff, lists, desc, len, cvw, cnt);
  return hip_status();
}

// Rows whose upper bound fits S lanes, any coarse id width: one entry per
// lane, bitonic sort of (coarse neighbour, weight) pairs across the S lanes
// by shuffles, segmented sum of equal neighbours, self entries dropped, run
// tails compacted with a ballot.  Used when the coarse ids do not leave room
// for the lane number beside them in 32 bits (k_contract_rows).
template <int S, int B>
__global__ void __launch_bounds__(B) k_contract_rows_wide(const int32_t* __restrict__ rows,
                                                       const int2* __restrict__ desc, int32_t nrows,
                                                       const int2* __restrict__ mrow,
                                                       const int32_t* __restrict__ adj,
                                                       const int32_t* __restrict__ w,
                                                       const int32_t* __restrict__ cmap,
                                                       const int32_t* __restrict__ toff,
                                                       int32_t* __restrict__ tadj, int32_t* __restrict__ tw,
                                                       int32_t* __restrict__ len) {
  const int64_t gt = int64_t(xcd_block()) * B + threadIdx.x;
  const int64_t ri = gt / S;
  const int sub = static_cast<int>(gt % S);
  if (ri >= nrows) return;
  const int32_t c = rows[ri];
  const int2 d = desc[ri];
  const int32_t m0 = d.x, nm = d.y;
  // Locate this lane's entry in the concatenation of the member rows: lane m
  // loads member m's row start and length, a shuffle scan gives the offsets,
  // and each lane finds its member among them.  More members than lanes
  // (max_group > S): member by member.
  int32_t j = -1;
  if (nm <= S) {
    int32_t ms = 0, md = 0;
    if (sub < nm) {
      const int2 r = mrow[m0 + sub];
      ms = r.x;
      md = r.y;
    }
    int32_t inc = md;
#pragma unroll
    for (int o = 1; o < S; o <<= 1) {
      const int32_t y = __shfl_up(inc, o, S);
      if (sub >= o) inc += y;
    }
    for (int m = 0; m < nm; ++m) {
      const int32_t im = __shfl(inc, m, S), sm = __shfl(ms, m, S), dm = __shfl(md, m, S);
      if (sub < im && sub >= im - dm) j = sm + (sub - (im - dm));
    }
  } else {
    int32_t pre = 0;
    for (int32_t m = m0; m < m0 + nm; ++m) {
      const int2 r = mrow[m];
      if (sub >= pre && sub < pre + r.y) j = r.x + (sub - pre);
      pre += r.y;
    }
  }
  int32_t key = INT32_MAX, val = 0;
  if (j >= 0) { key = cmap[adj[j]]; val = w[j]; }
#pragma unroll
  for (int k2 = 2; k2 <= S; k2 <<= 1) {
#pragma unroll
    for (int j2 = k2 >> 1; j2 > 0; j2 >>= 1) {
      const int32_t ok = __shfl_xor(key, j2, S);
      const int32_t ov = __shfl_xor(val, j2, S);
      const bool up = (sub & k2) == 0;
      const bool lower = (sub & j2) == 0;
      const bool take = lower ? (up ? ok < key : ok > key) : (up ? ok > key : ok < key);
      if (take) { key = ok; val = ov; }
    }
  }
  int32_t x = val;
#pragma unroll
  for (int o = 1; o < S; o <<= 1) {
    const int32_t y = __shfl_up(x, o, S);
    const int32_t ky = __shfl_up(key, o, S);
    if (sub >= o && ky == key) x += y;
  }
  const int32_t kn = __shfl_down(key, 1, S);
  const bool tail = (sub == S - 1) || kn != key;
  const bool out = tail && key != c && key != INT32_MAX;
  const uint64_t b = ballot(out);
  const int base_lane = lane_id() & ~(S - 1);
  const uint64_t seg = (S == 64) ? b : ((b >> base_lane) & ((1ull << S) - 1));
  const int pos = popc64(seg & ((1ull << sub) - 1));
  if (out) {
    const int32_t o = toff[c] + pos;
    tadj[o] = key;
    tw[o] = x;
  }
  if (sub == 0) len[c] = popc64(seg);
}

// Rows whose upper bound fits S lanes (S = 16, 32, 64; B / S rows per
// block), coarse ids below 2^(32 - log2 S) - 1.  Per row:
//   1. lane m < nm loads member m's row bounds (mrow); an add-scan of the
//      lengths gives each member's first lane, which the member marks in a
//      per-wave LDS slot array; lane i takes the entry of the last member
//      marked at or below it (a ballot of the marks);
//   2. its entry (coarse neighbour, weight); self entries become the
//      sentinel 0xffffffff, others the key neighbour << log2 S | lane;
//   3. an in-register bitonic sort of the keys (DPP partners), the weight
//      follows its key by one ds_bpermute;
//   4. runs of equal neighbours: a segmented add-scan minus the exclusive
//      sum at the run's head gives the run total at its tail; tails are
//      compacted with a ballot.
// The dependent loads per entry: the row's list slot (id and member range),
// the members' row bounds, the entry, its coarse id.
// Global thread slot gt serves row gt / S as lane gt % S of its segment; wm
// is the wave's 64-slot LDS mark array.  The whole wave calls it together.
template <int S>
__device__ __forceinline__ void contract_row_slot(int64_t gt, int32_t* wm, const int32_t* __restrict__ rows,
                                                  const int2* __restrict__ desc, int32_t nrows,
                                                  const int2* __restrict__ mrow, const int32_t* __restrict__ adj,
                                                  const int32_t* __restrict__ w, const int32_t* __restrict__ cmap,
                                                  const int32_t* __restrict__ toff, int32_t* __restrict__ tadj,
                                                  int32_t* __restrict__ tw, int32_t* __restrict__ len) {
  static_assert(S == 16 || S == 32 || S == 64, "segment of 16, 32 or 64 lanes");
  constexpr int LB = S == 16 ? 4 : (S == 32 ? 5 : 6);
  constexpr uint32_t kNone = 0xffffffffu;
  const int64_t ri = gt >> LB;
  const int lane = lane_id();
  const int sub = lane & (S - 1);
  const int base = lane - sub;
  // Segments past the last row stay active (masked stores) so that every
  // cross-lane step runs on whole segments.
  const bool live = ri < nrows;
  int32_t c = -1, m0 = 0, nm = 0, to = 0;
  if (live) {
    c = rows[ri];
    const int2 d = desc[ri];
    m0 = d.x;
    nm = d.y;
    to = toff[c];
  }
  int32_t j = -1;
  if (nm <= S) {
    int32_t ms = 0, md = 0;
    if (sub < nm) {
      const int2 r = mrow[m0 + sub];
      ms = r.x;
      md = r.y;
    }
    const int32_t inc = seg_incl_scan<S>(md);
    const int32_t e = inc - md;
    const int32_t tot = __shfl(inc, base + S - 1, 64);
    wm[lane] = INT32_MIN;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (md > 0) wm[base + e] = ms - e;  // distinct lanes: members with entries start apart
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint64_t starts = ballot(wm[lane] != INT32_MIN);
    if (sub < tot) j = wm[last_set_at_or_below(starts, lane)] + sub;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    // More members than lanes (members without entries): member by member.
    int32_t pre = 0;
    for (int32_t m = m0; m < m0 + nm; ++m) {
      const int2 r = mrow[m];
      if (sub >= pre && sub < pre + r.y) j = r.x + (sub - pre);
      pre += r.y;
    }
  }
  uint32_t key = kNone;
  int32_t val = 0;
  if (j >= 0) {
    const int32_t q = cmap[adj[j]];
    val = w[j];
    if (q != c) key = (uint32_t(q) << LB) | uint32_t(sub);
  }
  key = seg_sort_u32<S>(key);
  const bool valid = key != kNone;
  const int32_t sv = __shfl(val, base + int(key & (S - 1)), 64);
  const uint32_t nb = key >> LB;
  const uint32_t prev = dpp_mov<dpp::kWaveShr1>(key), next = dpp_mov<dpp::kWaveShl1>(key);
  const bool head = valid && (sub == 0 || (prev >> LB) != nb);
  const bool tail = valid && (sub == S - 1 || (next >> LB) != nb);
  const int32_t x = valid ? sv : 0;
  const int32_t p = seg_incl_scan<S>(x);
  const int h = last_set_at_or_below(ballot(head), lane);
  const int32_t eh = __shfl(p - x, h < 0 ? lane : h, 64);
  const uint64_t tails = ballot(tail);
  const uint64_t segm = S == 64 ? ~0ull : (((1ull << S) - 1) << base);
  if (live && tail) {
    const int32_t o = to + popc64(tails & segm & lanemask_lt());
    tadj[o] = int32_t(nb);
    tw[o] = p - eh;
  }
  if (live && sub == 0) len[c] = popc64(tails & segm);
}

template <int S, int B>
__global__ void __launch_bounds__(B) k_contract_rows(const int32_t* __restrict__ rows,
                                                       const int2* __restrict__ desc, int32_t nrows,
                                                       const int2* __restrict__ mrow,
                                                       const int32_t* __restrict__ adj,
                                                       const int32_t* __restrict__ w,
                                                       const int32_t* __restrict__ cmap,
                                                       const int32_t* __restrict__ toff,
                                                       int32_t* __restrict__ tadj, int32_t* __restrict__ tw,
                                                       int32_t* __restrict__ len) {
  static_assert(B % 64 == 0, "whole waves");
  __shared__ int32_t mark[B];
  contract_row_slot<S>(int64_t(xcd_block()) * B + threadIdx.x, mark + (threadIdx.x & ~63u), rows, desc, nrows, mrow,
                       adj, w, cmap, toff, tadj, tw, len);
}

// The same slots, taken from the work-stealing queues.
template <int S, int B>
__global__ void __launch_bounds__(B) k_contract_rows_ws(const int32_t* __restrict__ rows,
                                                          const int2* __restrict__ desc, int32_t nrows,
                                                          const int2* __restrict__ mrow,
                                                          const int32_t* __restrict__ adj,
                                                          const int32_t* __restrict__ w,
                                                          const int32_t* __restrict__ cmap,
                                                          const int32_t* __restrict__ toff,
                                                          int32_t* __restrict__ tadj, int32_t* __restrict__ tw,
                                                          int32_t* __restrict__ len,
                                                          unsigned long long* __restrict__ ctr) {
  static_assert(B % 64 == 0, "whole waves");
  __shared__ int32_t mark[B];
  int32_t* wm = mark + (threadIdx.x & ~63u);
  const int64_t sweeps = (int64_t(nrows) * S + 63) / 64;
  steal_sweeps(ctr, sweeps, [&](int64_t sw) {
    contract_row_slot<S>(sw * 64 + lane_id(), wm, rows, desc, nrows, mrow, adj, w, cmap, toff, tadj, tw, len);
  });
}

// Largest coarse id count for k_contract_rows<64, B> (ids below 2^26 - 1);
// the 16- and 32-lane kernels allow more, one limit keeps the choice simple.
constexpr int32_t kNarrowIdsMax = (1 << 26) - 1;

// Wide rows (coarse graphs of 2^26 - 1 vertices or more) always take the
// direct launch; the narrow ones may take the work-stealing form.
template <int B, bool Wide>
static void contract_rows_block(const DGraph& g, int lanes, const int32_t* rows, const int2* desc, int32_t nrows,
                                const int2* mrow, const int32_t* cmap, const int32_t* toff, int32_t* tadj,
                                int32_t* tw, int32_t* len, const Steal* ws, hipStream_t st) {
  const unsigned grid = grid_for(int64_t(nrows) * lanes, B);
  auto go = [&](auto kern) {
    gk_launch(kern, dim3(grid), dim3(B), 0, st, rows, desc, nrows, mrow, g.adj, g.w, cmap, toff, tadj, tw, len);
  };
  auto go_ws = [&](auto kern, int S) {
    const unsigned pg = steal_grid(reinterpret_cast<const void*>(kern), B, *ws, grid);
    unsigned long long* ctr = nullptr;  // queues cleared and used only when the work has a tail
    if (steal_tail((int64_t(nrows) * S + 63) / 64, int64_t(pg) * (B / 64)) > 0) {
      fill<unsigned long long>(ws->ctr, 0ull, kStealWords, st);
      ctr = ws->ctr;
    }
    gk_launch(kern, dim3(pg), dim3(B), 0, st, rows, desc, nrows, mrow, g.adj, g.w, cmap, toff, tadj, tw, len, ctr);
  };
  if (!Wide && ws) {
    switch (lanes) {
      case 16: go_ws(k_contract_rows_ws<16, B>, 16); break;
      case 32: go_ws(k_contract_rows_ws<32, B>, 32); break;
      default: go_ws(k_contract_rows_ws<64, B>, 64); break;
    }
    return;
  }
  switch (lanes) {
    case 16: Wide ? go(k_contract_rows_wide<16, B>) : go(k_contract_rows<16, B>); break;
    case 32: Wide ? go(k_contract_rows_wide<32, B>) : go(k_contract_rows<32, B>); break;
    default: Wide ? go(k_contract_rows_wide<64, B>) : go(k_contract_rows<64, B>); break;
  }
}

template <bool Wide>
static void contract_rows_any(const DGraph& g, int lanes, int block, const int32_t* rows, const int2* desc,
                              int32_t nrows, const int2* mrow, const int32_t* cmap, const int32_t* toff,
                              int32_t* tadj, int32_t* tw, int32_t* len, const Steal* ws, hipStream_t st) {
  switch (block) {
    case 64: contract_rows_block<64, Wide>(g, lanes, rows, desc, nrows, mrow, cmap, toff, tadj, tw, len, ws, st); break;
    case 128: contract_rows_block<128, Wide>(g, lanes, rows, desc, nrows, mrow, cmap, toff, tadj, tw, len, ws, st); break;
    case 512: contract_rows_block<512, Wide>(g, lanes, rows, desc, nrows, mrow, cmap, toff, tadj, tw, len, ws, st); break;
    default: contract_rows_block<256, Wide>(g, lanes, rows, desc, nrows, mrow, cmap, toff, tadj, tw, len, ws, st); break;
  }
}

int launch_contract_rows(const DGraph& g, int lanes, int block, const int32_t* rows, const int2* desc,
                         int32_t nrows, int32_t nc, const int2* mrow, const int32_t* cmap, const int32_t* toff,
                         int32_t* tadj, int32_t* tw, int32_t* len, bool force_wide, hipStream_t st,
                         const Steal* ws) {
  if (nrows <= 0) return 0;
  if (force_wide || nc > kNarrowIdsMax)
    contract_rows_any<true>(g, lanes, block, rows, desc, nrows, mrow, cmap, toff, tadj, tw, len, nullptr, st);
  else
    contract_rows_any<false>(g, lanes, block, rows, desc, nrows, mrow, cmap, toff, tadj, tw, len, ws, st);
  return hip_status();
}

// The rows of all three lane classes in one launch, their counts read on the
// device: the waves stride over the classes' waves one after another.  For
// levels of up to kRowsAllMax coarse rows, whose launches and the read-back of
// the counts took longer than the rows (mesh of 60000 vertices, 3 levels: 7 us
// a level here; three launches of 4 us and a read-back of 15 us before).
__global__ void __launch_bounds__(256) k_contract_rows_all(int32_t nc, const int32_t* __restrict__ cnt,
                                                           const int32_t* __restrict__ lists,
                                                           const int2* __restrict__ desc,
                                                           const int2* __restrict__ mrow,
                                                           const int32_t* __restrict__ adj,
                                                           const int32_t* __restrict__ w,
                                                           const int32_t* __restrict__ cmap,
                                                           const int32_t* __restrict__ toff,
                                                           int32_t* __restrict__ tadj, int32_t* __restrict__ tw,
                                                           int32_t* __restrict__ len) {
  __shared__ int32_t mark[256];
  int32_t* wm = mark + (threadIdx.x & ~63u);
  const int32_t r0 = cnt[0], r1 = cnt[kRowCtlStride], r2 = cnt[2 * kRowCtlStride];
  const int32_t w0 = (r0 + 3) / 4, w1 = (r1 + 1) / 2;
  const int32_t total = w0 + w1 + r2;
  for (int32_t u = int32_t(blockIdx.x) * 4 + int32_t(threadIdx.x >> 6); u < total; u += int32_t(gridDim.x) * 4) {
    if (u < w0)
      contract_row_slot<16>(int64_t(u) * 64 + lane_id(), wm, lists, desc, r0, mrow, adj, w, cmap, toff, tadj, tw, len);
    else if (u < w0 + w1)
      contract_row_slot<32>(int64_t(u - w0) * 64 + lane_id(), wm, lists + nc, desc + nc, r1, mrow, adj, w, cmap, toff,
                            tadj, tw, len);
    else
      contract_row_slot<64>(int64_t(u - w0 - w1) * 64 + lane_id(), wm, lists + 2 * int64_t(nc), desc + 2 * int64_t(nc),
                            r2, mrow, adj, w, cmap, toff, tadj, tw, len);
  }
}

// Rows of 65 to kMidMax entries: a workgroup per row sums the entries by
// coarse neighbour in an LDS hash table, collects the (distinct) neighbours
// and sorts them.  The rows of a weighted DAG's coarse levels are of this kind;
// sorting all their entries in global memory took a read-back, 69 + 35 us of
// scatters and histograms and 70 us of scans on a DAG of 1 M vertices, which is
// 11 us here.  Grid-stride over
// the class's list, whose count is read on the device.
constexpr int kMidThreads = 256;

__global__ void __launch_bounds__(kMidThreads) k_contract_mid(const int32_t* __restrict__ cnt,
                                                              const int32_t* __restrict__ rows,
                                                              const int2* __restrict__ desc,
                                                              const int2* __restrict__ mrow,
                                                              const int32_t* __restrict__ adj,
                                                              const int32_t* __restrict__ w,
                                                              const int32_t* __restrict__ cmap,
                                                              const int32_t* __restrict__ toff,
                                                              int32_t* __restrict__ tadj, int32_t* __restrict__ tw,
                                                              int32_t* __restrict__ len) {
  __shared__ int32_t key[2 * kMidMax];
  __shared__ int32_t sum[2 * kMidMax];
  __shared__ uint64_t srt[kMidMax];
  __shared__ int32_t m;
  const int t = threadIdx.x;
  const int32_t nrows = cnt[3 * kRowCtlStride];
  for (int32_t i = blockIdx.x; i < nrows; i += gridDim.x) {
    const int32_t c = rows[i];
    const int2 d = desc[i];
    // entries of the row, and the table: a power of two, at least twice as many
    const int32_t ub = len[c];
    int32_t tab = 256;
    while (tab < 2 * ub) tab <<= 1;
    const int shift = __clz(tab) + 1;  // 32 - log2(tab)
    for (int32_t x = t; x < tab; x += kMidThreads) {
      key[x] = -1;
      sum[x] = 0;
    }
    if (t == 0) m = 0;
    __syncthreads();
    // a wave per member in turn: its entries are consecutive reads
    for (int32_t x = d.x + (t >> 6); x < d.x + d.y; x += kMidThreads / 64) {
      const int2 r = mrow[x];
      for (int32_t e = r.x + lane_id(); e < r.x + r.y; e += 64) {
        const int32_t q = cmap[adj[e]];
        if (q == c) continue;
        const int32_t we = w[e];
        uint32_t s = (uint32_t(q) * 0x9E3779B1u) >> shift;
        while (true) {
          const int32_t o = atomicCAS(&key[s], -1, q);
          if (o == -1 || o == q) break;
          s = (s + 1) & uint32_t(tab - 1);
        }
        atomicAdd(&sum[s], we);
      }
    }
    __syncthreads();
    // the distinct neighbours with their sums
    for (int32_t x0 = 0; x0 < tab; x0 += kMidThreads) {
      const int32_t q = key[x0 + t];
      const uint64_t b = ballot(q >= 0);
      int32_t o = 0;
      if (lane_id() == 0 && b) o = atomicAdd(&m, popc64(b));
      o = __shfl(o, 0, 64);
      if (q >= 0) srt[o + popc64(b & lanemask_lt())] = (uint64_t(uint32_t(q)) << 32) | uint32_t(sum[x0 + t]);
    }
    __syncthreads();
    const int32_t cntc = m;
    int32_t P = 64;
    while (P < cntc) P <<= 1;
    for (int32_t x = cntc + t; x < P; x += kMidThreads) srt[x] = ~0ull;
    __syncthreads();
    for (int32_t k2 = 2; k2 <= P; k2 <<= 1)
      for (int32_t j2 = k2 >> 1; j2 > 0; j2 >>= 1) {
        for (int32_t p = t; p < (P >> 1); p += kMidThreads) {
          const int32_t lo = ((p & ~(j2 - 1)) << 1) | (p & (j2 - 1));
          const int32_t hi = lo + j2;
          const uint64_t a = srt[lo], b = srt[hi];
          if ((lo & k2) == 0 ? a > b : a < b) {
            srt[lo] = b;
            srt[hi] = a;
          }
        }
        __syncthreads();
      }
    const int32_t to = toff[c];
    for (int32_t x = t; x < cntc; x += kMidThreads) {
      const uint64_t e = srt[x];
      tadj[to + x] = int32_t(e >> 32);
      tw[to + x] = int32_t(uint32_t(e));
    }
    if (t == 0) len[c] = cntc;
    __syncthreads();  // the table and the sorted row are read
  }
}

int launch_contract_rows_all(const DGraph& g, int32_t nc, const int32_t* cnt, const int32_t* lists, const int2* desc,
                             const int2* mrow, const int32_t* cmap, const int32_t* toff, int32_t* tadj, int32_t* tw,
                             int32_t* len, hipStream_t st) {
  if (nc <= 0) return 0;
  gk_launch(k_contract_rows_all, dim3(std::min<unsigned>(grid_for(nc, 4), 4096)), dim3(256), 0, st, nc, cnt, lists,
            desc, mrow, g.adj, g.w, cmap, toff, tadj, tw, len);
  return hip_status();
}

int launch_contract_mid(const DGraph& g, int32_t nc, int32_t max_rows, const int32_t* cnt, const int32_t* lists,
                        const int2* desc, const int2* mrow, const int32_t* cmap, const int32_t* toff, int32_t* tadj,
                        int32_t* tw, int32_t* len, hipStream_t st) {
  // More than 64 entries a row: no more rows than that.
  const int64_t rows = std::min<int64_t>(std::min<int64_t>(max_rows, nc), int64_t(g.nnz) / 65);
  if (rows <= 0) return 0;
  gk_launch(k_contract_mid, dim3(unsigned(std::min<int64_t>(rows, 2048))), dim3(kMidThreads), 0, st, cnt,
            lists + 3 * int64_t(nc), desc + 3 * int64_t(nc), mrow, g.adj, g.w, cmap, toff, tadj, tw, len);
  return hip_status();
}

struct BigUbLoad {
  const int32_t* rows;
  const int32_t* ub;
  int32_t nrows;
  __device__ int operator()(int64_t i) const { return i < nrows ? ub[rows[i]] : 0; }
};

int launch_big_offsets(const int32_t* rows, const int32_t* ub, int32_t nrows, int32_t* boff, int32_t* scratch,
                       hipStream_t st) {
  int rc = scan(int64_t(nrows) + 1, BigUbLoad{rows, ub, nrows}, StoreExcl{boff}, nullptr, scratch, st);
  return rc ? GK_ERR_HIP : hip_status();
}

// Big rows: every entry becomes the key (row rank << 32 | coarse neighbour);
// one block per row walks the members in order.
__global__ void __launch_bounds__(256) k_big_gather(const int32_t* __restrict__ rows,
                                                    const int32_t* __restrict__ boff,
                                                    const int32_t* __restrict__ cptr,
                                                    const int2* __restrict__ mrow,
                                                    const int32_t* __restrict__ adj,
                                                    const int32_t* __restrict__ w,
                                                    const int32_t* __restrict__ cmap,
                                                    uint64_t* __restrict__ keys, int32_t* __restrict__ vals) {
  const int32_t i = blockIdx.x;
  const int32_t c = rows[i];
  int32_t o = boff[i];
  for (int32_t m = cptr[c]; m < cptr[c + 1]; ++m) {
    const int32_t s = mrow[m].x, d = mrow[m].y;
    for (int32_t t = threadIdx.x; t < d; t += 256) {
      keys[o + t] = (uint64_t(uint32_t(i)) << 32) | uint64_t(uint32_t(cmap[adj[s + t]]));
      vals[o + t] = w[s + t];
    }
    o += d;
  }
}

int launch_contract_big_gather(const DGraph& g, const int32_t* rows, int32_t nrows,
                               const int32_t* boff, const int32_t* cptr, const int2* mrow,
                               const int32_t* cmap, uint64_t* keys, int32_t* vals, hipStream_t st) {
  if (nrows <= 0) return 0;
  k_big_gather<<<nrows, 256, 0, st>>>(rows, boff, cptr, mrow, g.adj, g.w, cmap, keys, vals);
  return hip_status();
}

// One wave per big row walks its sorted entries in chunks of 64 with a
// segmented sum carried across chunks.
__global__ void __launch_bounds__(64) k_big_merge(const int32_t* __restrict__ rows,
                                                  const int32_t* __restrict__ boff,
                                                  const uint64_t* __restrict__ keys,
                                                  const int32_t* __restrict__ vals,
                                                  const int32_t* __restrict__ toff,
                                                  int32_t* __restrict__ tadj, int32_t* __restrict__ tw,
                                                  int32_t* __restrict__ len) {
  const int32_t i = blockIdx.x;
  const int32_t c = rows[i];
  const int32_t b0 = boff[i], b1 = boff[i + 1];
  const int lane = lane_id();
  const uint64_t lt = lanemask_lt();
  int32_t carry_key = -1, carry_sum = 0;
  int32_t count = 0;
  const int32_t obase = toff[c];
  for (int32_t base = b0; base < b1; base += 64) {
    const int32_t e = base + lane;
    const bool valid = e < b1;
    const int32_t key = valid ? int32_t(uint32_t(keys[e])) : INT32_MAX;
    int32_t x = valid ? vals[e] : 0;
    if (valid && key == carry_key) x += (lane == 0) ? carry_sum : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t y = __shfl_up(x, o, 64);
      const int32_t ky = __shfl_up(key, o, 64);
      if (lane >= o && ky == key) x += y;
    }
    // Tail: the next element (possibly in the next chunk) has another key.
    int32_t kn = __shfl_down(key, 1, 64);
    if (lane == 63) kn = (e + 1 < b1) ? int32_t(uint32_t(keys[e + 1])) : INT32_MAX;
    const bool tail = valid && (e + 1 == b1 || kn != key);
    const bool out = tail && key != c;
    const uint64_t bm = ballot(out);
    if (out) {
      const int32_t o = obase + count + popc64(bm & lt);
      tadj[o] = key;
      tw[o] = x;
    }
    count += popc64(bm);
    // Carry the last run into the next chunk when it continues.
    const int32_t last_key = __shfl(key, 63, 64);
    const int32_t last_x = __shfl(x, 63, 64);
    const bool last_tail = __shfl(static_cast<int>(tail), 63, 64) != 0;
    carry_key = last_tail ? -1 : last_key;
    carry_sum = last_x;
  }
  if (lane == 0) len[c] = count;
}

int launch_contract_big_merge(const int32_t* rows, int32_t nrows, const int32_t* boff,
                              const uint64_t* keys, const int32_t* vals, const int32_t* toff,
                              int32_t* tadj, int32_t* tw, int32_t* len, hipStream_t st) {
  if (nrows <= 0) return 0;
  k_big_merge<<<nrows, 64, 0, st>>>(rows, boff, keys, vals, toff, tadj, tw, len);
  return hip_status();
}

// Row starts of the coarse CSR from the rows' lengths: per-tile sums, then
// every tile adds up the sums before it (many tiles: scanned by one block; up to
// kLenDirect tiles: the lengths before it, which saves the first launch).
// The last tile writes the entry count and the row class counters to the host.
__global__ void __launch_bounds__(256) k_len_reduce(int32_t nc, const int32_t* __restrict__ len,
                                                    int32_t* __restrict__ partial) {
  __shared__ int ws[4];
  const int64_t base = int64_t(blockIdx.x) * kSizeTile;
  int32_t s = 0;
#pragma unroll
  for (int j = 0; j < kSizeIPT; ++j) {
    const int64_t i = base + j * 256 + threadIdx.x;
    if (i < nc) s += len[i];
  }
  s = wave_sum(s);
  if (lane_id() == 0) ws[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

__global__ void __launch_bounds__(256) k_len_mid(int64_t nb, int32_t* __restrict__ partial) {
  __shared__ int lds[8];
  int32_t run = 0;
  for (int64_t b0 = 0; b0 < nb; b0 += 256) {
    const int64_t b = b0 + threadIdx.x;
    int t;
    const int e = block_excl_scan_256(b < nb ? partial[b] : 0, &t, lds);
    if (b < nb) partial[b] = run + e;
    run += t;
  }
}

__global__ void __launch_bounds__(256) k_len_apply(int32_t nc, const int32_t* __restrict__ len,
                                                   const int32_t* __restrict__ partial, int scanned,
                                                   int32_t* __restrict__ cxadj, const int32_t* __restrict__ cnt,
                                                   const HostWords host) {
  __shared__ int lds[8];
  int32_t pre = 0;
  int t;
  if (scanned) {
    pre = partial[blockIdx.x];
  } else {
    // partial: the sums of the tiles before this one, or null and the lengths themselves
    const int64_t nb = partial ? int64_t(blockIdx.x) : int64_t(blockIdx.x) * kSizeTile;
    const int32_t* from = partial ? partial : len;
    int32_t s = 0;
    for (int64_t b = threadIdx.x; b < nb; b += 256) s += from[b];
    (void)block_excl_scan_256(s, &t, lds);
    pre = t;
  }
  const int64_t base = int64_t(blockIdx.x) * kSizeTile + int64_t(threadIdx.x) * kSizeIPT;
  int32_t l[kSizeIPT];
  int32_t s = 0;
#pragma unroll
  for (int j = 0; j < kSizeIPT; ++j) {
    l[j] = base + j < nc ? len[base + j] : 0;
    s += l[j];
  }
  int32_t run = pre + block_excl_scan_256(s, &t, lds);
#pragma unroll
  for (int j = 0; j < kSizeIPT; ++j) {
    if (base + j < nc) cxadj[base + j] = run;
    run += l[j];
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 255) {
    cxadj[nc] = run;
    int32_t word[kRowCtlWords];
#pragma unroll
    for (int k = 0; k < kRowCtlWords; ++k) word[k] = cnt[k * kRowCtlStride];
    tell(host, 0, run);
#pragma unroll
    for (int k = 0; k < kRowCtlWords; ++k) tell(host, 1 + k, word[k]);
  }
}

int launch_len_scan(int32_t nc, const int32_t* len, int32_t* partial, int32_t* cxadj, const int32_t* cnt,
                    const HostWords& host, hipStream_t st) {
  const int64_t nb = std::max<int64_t>(1, size_partials(nc));
  constexpr int64_t kLenDirect = 4;
  if (nb <= kLenDirect) {
    k_len_apply<<<unsigned(nb), 256, 0, st>>>(nc, len, nullptr, 0, cxadj, cnt, host);
    return hip_status();
  }
  k_len_reduce<<<unsigned(nb), 256, 0, st>>>(nc, len, partial);
  const bool mid = nb > kSizeDirect;
  if (mid) k_len_mid<<<1, 256, 0, st>>>(nb, partial);
  k_len_apply<<<unsigned(nb), 256, 0, st>>>(nc, len, partial, mid ? 1 : 0, cxadj, cnt, host);
  return hip_status();
}

// Copy merged rows to the final CSR (8 lanes per row).
__global__ void __launch_bounds__(256) k_contract_copy(int32_t nc, const int32_t* __restrict__ toff,
                                                       const int32_t* __restrict__ len,
                                                       const int32_t* __restrict__ cxadj,
                                                       const int32_t* __restrict__ tadj,
                                                       const int32_t* __restrict__ tw,
                                                       int32_t* cadj, int32_t* cw, int32_t* xout) {
  const int64_t gt = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int64_t c = gt / 8;
  const int sub = static_cast<int>(gt % 8);
  if (c >= nc) return;
  const int32_t s = toff[c], d = cxadj[c], l = len[c];
  if (xout && sub == 0) {
    xout[c] = d;
    if (c == nc - 1) xout[nc] = d + l;
  }
  for (int32_t t = sub; t < l; t += 8) {
    cadj[d + t] = tadj[s + t];
    cw[d + t] = tw[s + t];
  }
}

int launch_contract_copy(int32_t nc, const int32_t* toff, const int32_t* len, const int32_t* cxadj,
                         const int32_t* tadj, const int32_t* tw, int32_t* cadj, int32_t* cw, int32_t* xout,
                         hipStream_t st) {
  if (nc <= 0) return 0;
  k_contract_copy<<<grid_for(int64_t(nc) * 8, 256), 256, 0, st>>>(nc, toff, len, cxadj, tadj, tw, cadj, cw, xout);
  return hip_status();
}

}  // namespace gkd
