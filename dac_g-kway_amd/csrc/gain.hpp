// Gain of the vertices of a worklist pass (update_vertex_info +
// calculate_gain, gkway/uncoarsen.hpp:175-237, 82-109), shared by the gain pass
// over the whole device (refine.hip) and the one inside the round loop
// (rounds.hip).
#pragma once
#include "dev_common.hpp"

namespace gkd {

// 64 / S vertices of a wave, S lanes each: a lane group takes vertex v with row
// [s, s + d), d <= S, when has is set.  Each lane holds one (part, weight)
// entry of the row and sums the weights of the lanes with the same part (an
// O(S) shuffle loop), which gives the connectivity to every adjacent part
// without a histogram.  Gain is the signed max over the adjacent parts of
// conn_q - conn_p, floored at 0, lowest q on ties.  emit(v, p, any, g, q, d) is
// called once per vertex by one lane: own part, whether a neighbour lies in
// another part, best gain (any sign) and its part, row length.
template <int S, class Emit>
__device__ __forceinline__ void gain_short(bool has, int32_t v, int32_t s, int32_t d, const int32_t* __restrict__ adj,
                                           const int32_t* __restrict__ w, const int32_t* part, Emit&& emit) {
  const int sub = lane_id() & (S - 1);
  if (!has) return;
  const int32_t p = part[v];
  int32_t q = -1, wj = 0;
  if (sub < d) {
    q = part[adj[s + sub]];
    wj = w[s + sub];
  }
  int32_t conn = 0, id = 0;
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const int32_t qi = __shfl(q, i, S);
    const int32_t wi = __shfl(wj, i, S);
    conn += (qi == q) ? wi : 0;
    id += (qi == p) ? wi : 0;
  }
  const bool ext = q >= 0 && q != p;
  int32_t g = ext ? conn - id : INT32_MIN;
  int32_t bq = ext ? q : INT32_MAX;
  int32_t anyext = ext ? 1 : 0;
#pragma unroll
  for (int o = S / 2; o > 0; o >>= 1) {
    const int32_t og = __shfl_xor(g, o, S), oq = __shfl_xor(bq, o, S);
    if (og > g || (og == g && oq < bq)) { g = og; bq = oq; }
    anyext |= __shfl_xor(anyext, o, S);
  }
  if (sub == 0) emit(v, p, anyext != 0, g, bq, d);
}

// The same for one vertex of any row length by the whole wave, with a
// histogram of the k parts (hist: k ints of LDS for this wave).
template <class Emit>
__device__ __forceinline__ void gain_long(int32_t v, int32_t s, int32_t e, const int32_t* __restrict__ adj,
                                          const int32_t* __restrict__ w, const int32_t* part, int32_t k,
                                          int32_t* hist, Emit&& emit) {
  const int lane = lane_id();
  for (int32_t q = lane; q < k; q += 64) hist[q] = 0;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int32_t p = part[v];
  bool ext = false;
  for (int32_t j = s + lane; j < e; j += 64) {
    const int32_t q = part[adj[j]];
    atomicAdd(&hist[q], w[j]);
    ext |= (q != p);
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const bool any = ballot(ext) != 0;
  const int32_t id = hist[p];
  int32_t g = INT32_MIN, bq = INT32_MAX;
  for (int32_t q = lane; q < k; q += 64) {
    const int32_t h = hist[q];
    if (q != p && h > 0) {
      const int32_t gq = h - id;
      if (gq > g || (gq == g && q < bq)) { g = gq; bq = q; }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const int32_t og = __shfl_xor(g, o, 64), oq = __shfl_xor(bq, o, 64);
    if (og > g || (og == g && oq < bq)) { g = og; bq = oq; }
  }
  if (lane == 0) emit(v, p, any, g, bq, e - s);
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Both for a pass of a wave: rows longer than S by the whole wave afterwards,
// one at a time; without a histogram they are left to the caller.
template <int S, class Emit>
__device__ __forceinline__ void gain_pass(bool has, int32_t v, int32_t s, int32_t d, const int32_t* __restrict__ adj,
                                          const int32_t* __restrict__ w, const int32_t* part, int32_t k,
                                          int32_t* hist, Emit&& emit) {
  const bool long_row = has && d > S;
  gain_short<S>(has && d <= S, v, s, d, adj, w, part, emit);
  if (!hist) return;
  uint64_t lm = ballot(long_row && (lane_id() & (S - 1)) == 0);
  while (lm) {
    const int src = __ffsll(static_cast<long long>(lm)) - 1;
    lm &= lm - 1;
    const int32_t hv = __shfl(v, src, 64), hs = __shfl(s, src, 64), he = hs + __shfl(d, src, 64);
    gain_long(hv, hs, he, adj, w, part, k, hist, emit);
  }
}

// Candidate bitmask: bit v set iff v is a boundary vertex with positive gain
// (the vertices the selection looks at).
__device__ __forceinline__ void set_cand(uint64_t* cand, int32_t v, bool on) {
  const uint64_t b = 1ull << (v & 63);
  if (on) atomicOr(reinterpret_cast<unsigned long long*>(&cand[v >> 6]), (unsigned long long)b);
  else atomicAnd(reinterpret_cast<unsigned long long*>(&cand[v >> 6]), (unsigned long long)~b);
}

}  // namespace gkd
