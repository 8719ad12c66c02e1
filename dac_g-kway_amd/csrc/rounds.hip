// The refinement rounds of a level in one launch: one workgroup per job runs
// the whole round -- movable set, independent selection, ordered moves,
// balanced prefix, apply, gain pass -- and goes on to the next round itself.
//
// What bounds a refinement round is latency, not bandwidth: late rounds move
// three to ten vertices and update a few dozen, out of some hundred
// candidates.  As five launches (three of the selection, the round kernel, the
// gain pass), each waiting for the one before, such a round took 40 us, and
// the host looked in every four rounds.  One workgroup needs a barrier where
// the launches needed a kernel boundary; the candidates (boundary vertices
// with positive gain) stay in LDS with their gain, destination and weight for
// the whole level, corrected after each round for the vertices it updated; the
// movable set is a bitmap in LDS that neighbours are tested against; part
// weights stay in LDS.  Jobs of a batch share no vertex and no part, so each
// runs at its own pace and none waits for another's rounds.  Refinement of a
// DAG of 300k vertices, k = 256 (375 rounds): 15.8 ms with separate kernels,
// 7.9 ms here; a late round takes 22k to 35k cycles, about a quarter of them
// the gains of the updated vertices (three dependent reads), the rest shared
// between finding the movable vertices, their best, the tests and the sort.
//
// The state in memory after a launch is the one the separate kernels would
// leave after as many rounds, so the two can take turns: a job with more
// candidates than the list holds is left to them, and a round that updates
// more vertices than one workgroup should (a large graph's first rounds)
// appends them to the worklist and leaves, for the gain pass over the whole
// device and another launch.
#include "balance.hpp"
#include "batch.hpp"
#include "gain.hpp"
#include "kernels.hpp"
#include "rounds.hpp"
#include "../../include/gkway.h"

namespace gkd {

static inline int hip_status() { return hipGetLastError() == hipSuccess ? 0 : GK_ERR_HIP; }

constexpr int kMovableBits = 1 << 16;  // bitmap of the movable set, by id modulo its size
constexpr int kLoopItems = 512;        // movers and neighbours that a round updates inside the workgroup
constexpr int32_t kLoopShortRow = 32;  // longer rows are tested by the whole wave, 64 neighbours a step
constexpr int kTop = 256;              // best movable vertices that the short way looks at
constexpr int kTopMin = 32;            // fewer than this many in its gain classes: the long way
constexpr int kTopIdBits = 21;         // vertex ids of a job in a sort key of the short way
constexpr int kGainClasses = 512;
constexpr int32_t kNoClass = -1;       // too few in the classes that fit: the long way

static_assert(kLoopItems <= 1024 / 2, "the table of first occurrences stays half empty");
static_assert(kGainClasses <= kBalMax, "the class counts lie in the cover array");

template <int CAP>
struct LoopLds {
  RoundLds r;
  int32_t lv[CAP], lg[CAP], lw[CAP];  // candidates: vertex (-1: dropped), gain, weight
  uint8_t ld[CAP], lp[CAP];           // destination, own part
  uint16_t mi[CAP], si[CAP];          // list indexes: movable with gain >= threshold; selected
  uint32_t bits[kMovableBits / 32];
  int32_t spw[kGainInlineK], dpw[kGainInlineK];  // part weights, and the balanced prefix's scratch
  int32_t outw[kGainInlineK];                    // movable weight by own part
  uint16_t ti[kTop], tj[kTop];                   // the best selected; the best movable, not yet tested
  int32_t wv[kLoopItems], ws[kLoopItems], wd[kLoopItems], ww[kLoopItems];  // worklist: vertex, row, weight
  long long cut;
  int32_t n, nmov, nsel, ntop, nts, nshort, nlong, tot, thr, pos, code;
};

// Selected candidates by list index.
template <int CAP>
struct SelectedIndex {
  const LoopLds<CAP>* L;
  __device__ int32_t vertex(int32_t i) const { return L->lv[L->si[i]]; }
  __device__ uint32_t gain_key(int32_t i, int32_t) const { return uint32_t(0x7fffffff - L->lg[L->si[i]]); }
};

// Appends x to list at *count for the lanes with on set: one LDS atomic per
// wave.  The whole wave calls it.
__device__ __forceinline__ void wave_append(bool on, uint16_t x, uint16_t* list, int32_t* count) {
  const uint64_t m = ballot(on);
  if (m == 0) return;
  int base = 0;
  if (lane_id() == 0) base = atomicAdd(count, popc64(m));
  base = __shfl(base, 0, 64);
  if (on) list[base + popc64(m & lanemask_lt())] = x;
}

// A barrier for LDS alone: stores to memory may still be under way after it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Gain class, monotone in the gain: its exponent and the four bits below.
__device__ __forceinline__ int32_t gain_class(int32_t g) {
  const int e = 31 - __clz(g);
  return (e << 4) | ((e >= 4 ? g >> (e - 4) : g << (4 - e)) & 15);
}

// Ascending sort of one key per lane over the wave, and the 64 smallest of two
// ascending waves' keys, ascending.
__device__ __forceinline__ uint64_t wave_merge_u64(uint64_t x) {
  for_pow2_down<32>([&](auto jc) {
    constexpr int J = decltype(jc)::value;
    const uint64_t y = lane_xor<J>(x);
    x = ((lane_id() & J) == 0) == (y < x) ? y : x;
  });
  return x;
}
template <int K>
__device__ __forceinline__ void wave_sort_step(uint64_t& x) {
  const bool up = K == 64 || (lane_id() & K) == 0;
  for_pow2_down<K / 2>([&](auto jc) {
    constexpr int J = decltype(jc)::value;
    const uint64_t y = lane_xor<J>(x);
    const bool keep_min = ((lane_id() & J) == 0) == up;
    x = keep_min == (y < x) ? y : x;
  });
}
__device__ __forceinline__ uint64_t wave_sort_u64(uint64_t x) {
  wave_sort_step<2>(x);
  wave_sort_step<4>(x);
  wave_sort_step<8>(x);
  wave_sort_step<16>(x);
  wave_sort_step<32>(x);
  wave_sort_step<64>(x);
  return x;
}

template <int S, int CAP>
__global__ void __launch_bounds__(kBalThreads) k_rounds(const RoundsArgs a) {
  static_assert(CAP <= 4 * kBalThreads, "the ordered list keeps four keys per thread");
  constexpr int kFull = CAP - kLoopItems;  // a round may add so many entries
  __shared__ LoopLds<CAP> L;
  RoundLds& R = L.r;
  const int t = threadIdx.x;
  const int lane = lane_id();
  const int wave = t >> 6;
  const int32_t j = blockIdx.x;
  if (j == 0 && t == 0) {  // the next launch's worklist counts and status
    a.next_wlc[0] = 0;
    a.next_wlc[1] = 0;
    a.next_status[0] = 0;
    a.next_status[1] = 0;
  }
  if (a.lastcnt[j] == 0) {  // converged in an earlier launch
    if (a.host.host && t == 0) {
      tell(a.host, 0, 0);
      tell(a.host, 1, 0);
      tell(a.host, 2, a.rounds[j]);
    }
    return;
  }
  const int32_t vb = a.v_off[j], ve = a.v_off[j + 1];
  const int32_t kj = a.kk[j];
  const long long cap = a.cap[j];
  int32_t* pwj = a.pw + a.pw_off[j];
  const bool exact_bits = ve - vb <= kMovableBits;
  // The candidates of the job's id range.
  const int64_t w0 = int64_t(vb) >> 6, w1 = ve > vb ? (int64_t(ve) - 1) >> 6 : w0 - 1;
  auto range_of = [&](int64_t w) -> uint64_t {
    const int64_t lo = vb > (w << 6) ? vb - (w << 6) : 0;
    const int64_t hi = ve < (w << 6) + 64 ? ve - (w << 6) : 64;
    return hi - lo == 64 ? ~0ull : (((1ull << (hi - lo)) - 1) << lo);
  };
  auto word_of = [&](int64_t w) -> uint64_t { return a.cand[w] & range_of(w); };
  int c = 0;
  for (int64_t w = w0 + t; w <= w1; w += kBalThreads) c += popc64(word_of(w));
  int n;
  int at = block_excl_scan_1024(c, &n, R.ws);
  if (n > kFull) {  // left to the kernels that select over the whole device
    if (t == 0) {
      atomicAdd(&a.status[0], 1);
      atomicAdd(&a.status[1], 1);
      if (a.host.host) {
        tell(a.host, 0, 1);
        tell(a.host, 1, 1);
        tell(a.host, 2, a.rounds[j]);
      }
    }
    return;
  }
  for (int64_t w = w0 + t; w <= w1; w += kBalThreads)
    for (uint64_t x = word_of(w); x; x &= x - 1) L.lv[at++] = int32_t((w << 6) + __ffsll(static_cast<long long>(x)) - 1);
  if (t < kj) L.spw[t] = pwj[t];
  if (t == 0) {
    L.n = n;
    L.thr = a.thr[j];
    L.cut = a.cut[j];
  }
  // What a round starts from: no movable vertex, empty lists.
  auto clear = [&]() {
    L.bits[t] = 0;
    L.bits[t + kBalThreads] = 0;
    static_assert(kMovableBits / 32 == 2 * kBalThreads, "two bitmap words per thread");
    if (t < kGainInlineK) L.outw[t] = 0;
    if (t == 0) {
      L.nmov = 0;
      L.nsel = 0;
      L.ntop = 0;
      L.nts = 0;
      R.lz[2] = 1;  // next threshold: test everything unless set below
    }
  };
  clear();
  __syncthreads();
  for (int i = t; i < n; i += kBalThreads) {
    const int32_t v = L.lv[i];
    L.lg[i] = a.gain[v];
    L.ld[i] = uint8_t(a.dest[v]);
    L.lp[i] = uint8_t(a.part[v]);
    L.lw[i] = a.vw[v];
  }
  // Movable: the candidate's move fits the cap.
  auto fits = [&](int32_t d, int32_t w) { return (long long)L.spw[d] + w <= cap; };
  // Whether neighbour u of v stands in v's way: a smaller id, and movable.
  // The bitmap decides for jobs of up to kMovableBits vertices; above that a
  // set bit may be another vertex's, and u's own state decides.
  auto blocks = [&](int32_t u, int32_t v) -> bool {
    const uint32_t b = uint32_t(u - vb) & (kMovableBits - 1);
    if (u >= v || !((L.bits[b >> 5] >> (b & 31)) & 1u)) return false;
    return exact_bits || (a.gain[u] > 0 && fits(a.dest[u], a.vw[u]));
  };
  long long tested = 0;           // row entries of the tested vertices
  int32_t upd_v = 0, upd_e = 0;   // vertices and row entries of the gain passes
  long long rounds_bytes = 0;     // thread 0: the rest of the algorithmic bytes
  // Tests list entries [0, m) named by index(i) (< 0: none) and appends the
  // selected ones to list: a lane per row of up to kLoopShortRow entries, eight
  // neighbours a step, longer rows by the whole wave.
  auto test = [&](int32_t m, auto&& index, uint16_t* list, int32_t* cnt) {
    for (int32_t i0 = wave * 64; i0 < m; i0 += kBalThreads) {
      const int32_t idx = i0 + lane < m ? index(i0 + lane) : -1;
      int32_t v = 0, s = 0, e = 0;
      bool sel = idx >= 0, long_row = false;
      if (sel) {
        v = L.lv[idx];
        s = a.xadj[v];
        e = a.xadj[v + 1];
        tested += e - s;
        long_row = e - s > kLoopShortRow;
        if (!long_row)
          for (int32_t x = s; x < e && sel; x += 8) {
            int32_t u[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) u[q] = x + q < e ? a.adj[x + q] : v;
#pragma unroll
            for (int q = 0; q < 8; ++q)
              if (blocks(u[q], v)) sel = false;
          }
      }
      uint64_t lm = ballot(long_row);
      while (lm) {
        const int src = __ffsll(static_cast<long long>(lm)) - 1;
        lm &= lm - 1;
        const int32_t lv = __shfl(v, src, 64), ls = __shfl(s, src, 64), le = __shfl(e, src, 64);
        bool blocked = false;
        for (int32_t x0 = ls; x0 < le && !blocked; x0 += 64) {
          const int32_t x = x0 + lane;
          blocked = ballot(x < le && blocks(a.adj[x], lv)) != 0;
        }
        if (lane == src && blocked) sel = false;
      }
      wave_append(sel, uint16_t(idx), list, cnt);
    }
  };

  int32_t rounds0 = 0;
  long long moved0 = 0;
  if (t == 0) {
    rounds0 = a.rounds[j];
    moved0 = a.moved[j];
  }
  int32_t count = 0;
  const bool may_short = !a.hist && !a.order && ve - vb <= (1 << kTopIdBits);
  __syncthreads();
  for (int32_t r = 0; r < a.max_rounds; ++r) {
    // 1. movable candidates: bitmap, the list of those at or above the gain
    // threshold, their weight by part
    n = L.n;
    const int32_t thr = L.thr;
    for (int32_t i0 = wave * 64; i0 < n; i0 += kBalThreads) {
      const int32_t i = i0 + lane;
      bool mv = false;
      if (i < n && L.lv[i] >= 0 && fits(L.ld[i], L.lw[i])) {
        const uint32_t b = uint32_t(L.lv[i] - vb) & (kMovableBits - 1);
        atomicOr(&L.bits[b >> 5], 1u << (b & 31));
        atomicAdd(&L.outw[L.lp[i]], L.lw[i]);
        mv = L.lg[i] >= thr;
      }
      wave_append(mv, uint16_t(i), L.mi, &L.nmov);
    }
    R.ht[t] = -1;
    if (t < kGainClasses) R.b.cover[t] = 0;
    if (t == 0) {
      L.nshort = 0;
      L.nlong = 0;
    }
    __syncthreads();
    const int32_t nmov = L.nmov;
    if (nmov == 0 && thr == 1) {
      count = 0;
      break;
    }
    // 2. The short way.  Late rounds select hundreds of vertices and move the
    // first three to ten of them: the part weights forbid the rest.  So the
    // kTop best are enough to begin with: one wave applies the 64 best
    // selected ones among them one after another, and stops where some part
    // is above the cap by more than all movable vertices of that part that are
    // still to come weigh -- it then stays above it, so no later prefix is
    // balanced.  Without that proof within 64 moves the long way follows (all
    // of the sequence, sorted, and all of its weight changes); it found itself
    // needed in one round of ten (DAG of 300k, k = 256).  The number selected
    // matters beyond M movable vertices (which M are ordered, the next gain
    // threshold) and while a threshold is set: then all are tested first, and
    // the best are taken from the selected ones.
    const bool few = nmov <= a.M && thr == 1;
    const bool may = may_short && few;
    bool tested_all = false;
    int pos = -2;  // -2: not decided yet
    const uint16_t* pick = L.mi;
    int32_t npick = nmov;
    if (!may) {
      // selection: no smaller-id movable neighbour; the movable vertices below
      // the threshold only when it leaves fewer than M
      test(nmov, [&](int32_t i) { return int32_t(L.mi[i]); }, L.si, &L.nsel);
      __syncthreads();
      count = L.nsel;
      if (count < a.M && thr > 1) {
        if (a.paths && t == 0) a.paths[3 * int64_t(j) + 2] += 1;
        __syncthreads();  // every thread has read nsel
        test(n, [&](int32_t i) { return L.lv[i] >= 0 && L.lg[i] < thr && fits(L.ld[i], L.lw[i]) ? i : -1; }, L.si,
             &L.nsel);
        __syncthreads();
        count = L.nsel;
      }
      if (count == 0) {
        if (t == 0) L.thr = 1;
        break;
      }
      tested_all = true;
      pick = L.si;
      npick = count;
    }
    if (may || (may_short && count <= kLazyFactor * a.M)) {
      const uint16_t* top = pick;
      int32_t ntop = npick;
      if (npick > kTop) {
        // the classes of highest gain that hold up to kTop of them
        for (int32_t i = t; i < npick; i += kBalThreads) {
          const int32_t g = L.lg[pick[i]];
          atomicAdd(&R.b.cover[gain_class(g)], 1);
        }
        __syncthreads();
        if (wave == 0) {
          constexpr int kPer = kGainClasses / 64;
          int32_t h[kPer], sum = 0;
#pragma unroll
          for (int i = 0; i < kPer; ++i) {
            h[i] = R.b.cover[kGainClasses - 1 - (kPer * lane + i)];
            sum += h[i];
          }
          int32_t run = wave_incl_scan(sum) - sum;
          int32_t code = kGainClasses, cnt = 0;  // lowest class that fits, vertices down to it
#pragma unroll
          for (int i = 0; i < kPer; ++i) {
            run += h[i];
            if (run <= kTop) {
              code = kGainClasses - 1 - (kPer * lane + i);
              cnt = run;
            }
          }
          // lanes that hold a class that fits are the first ones
          const uint64_t m = ballot(code < kGainClasses);
          const int last = m ? 63 - __clzll(static_cast<long long>(m)) : 0;
          if (lane == last) L.code = cnt >= kTopMin ? code : kNoClass;
        }
        __syncthreads();
        ntop = 0;
        // decided by a word that nobody writes again before the next round's
        // barriers: L.ntop counts up below while other waves still arrive here
        const int32_t code = L.code;
        if (code != kNoClass) {
          for (int32_t i0 = wave * 64; i0 < npick; i0 += kBalThreads) {
            const int32_t idx = i0 + lane < npick ? pick[i0 + lane] : -1;
            wave_append(idx >= 0 && gain_class(L.lg[idx]) >= code, uint16_t(idx), L.tj, &L.ntop);
          }
          __syncthreads();
          top = L.tj;
          ntop = L.ntop;
        }
      }
      if (ntop > 0) {
        if (!tested_all) {
          // Tests by four lanes per vertex; long rows as in test().
          const int32_t i = t >> 2;
          const int sub = lane & 3;
          const int32_t idx = i < ntop ? top[i] : -1;
          int32_t v = 0, s = 0, e = 0;
          bool blocked = false, long_row = false;
          if (idx >= 0) {
            v = L.lv[idx];
            s = a.xadj[v];
            e = a.xadj[v + 1];
            if (sub == 0) tested += e - s;
            long_row = e - s > kLoopShortRow;
            if (!long_row) {
              int32_t u[kLoopShortRow / 4];
#pragma unroll
              for (int q = 0; q < kLoopShortRow / 4; ++q) u[q] = s + 4 * q + sub < e ? a.adj[s + 4 * q + sub] : v;
#pragma unroll
              for (int q = 0; q < kLoopShortRow / 4; ++q)
                if (blocks(u[q], v)) blocked = true;
            }
          }
          uint64_t lm = ballot(long_row && sub == 0);
          while (lm) {
            const int src = __ffsll(static_cast<long long>(lm)) - 1;
            lm &= lm - 1;
            const int32_t lv = __shfl(v, src, 64), ls = __shfl(s, src, 64), le = __shfl(e, src, 64);
            bool b = false;
            for (int32_t x0 = ls; x0 < le && !b; x0 += 64) {
              const int32_t x = x0 + lane;
              b = ballot(x < le && blocks(a.adj[x], lv)) != 0;
            }
            if (lane == src && b) blocked = true;
          }
          const uint64_t bm = ballot(blocked);
          const bool sel = idx >= 0 && sub == 0 && ((bm >> lane) & 15u) == 0;
          wave_append(sel, uint16_t(idx), L.ti, &L.nts);
          __syncthreads();
          top = L.ti;
        }
        const int32_t nts = tested_all ? ntop : L.nts;
        // The 64 best of them, by (gain desc, id asc); the list index rides
        // in the key's low bits.
        uint64_t key = ~0ull;
        if (t < nts) {
          const int32_t idx = top[t];
          key = (uint64_t(uint32_t(0x7fffffff - L.lg[idx])) << (kTopIdBits + 12)) |
                (uint64_t(uint32_t(L.lv[idx] - vb)) << 12) | uint64_t(idx);
        }
        if (wave * 64 < nts) {
          key = wave_sort_u64(key);
          if (wave > 0) R.b.sk[t] = key;
        }
        if (nts > 64) __syncthreads();
        if (wave == 0) {
          for (int32_t w = 64; w < nts; w += 64) {
            const uint64_t y = R.b.sk[w + 63 - lane];
            key = wave_merge_u64(y < key ? y : key);
          }
          int32_t K = nts < 64 ? nts : 64;
          if (a.M < K) K = a.M;
          const int32_t idx = int32_t(key & 4095);
          int32_t src = -1, dst = -2, w = 0, left = 0, g = 0, pwd = 0, v = 0;
          if (lane < K) {
            v = L.lv[idx];
            g = L.lg[idx];
            src = L.lp[idx];
            dst = L.ld[idx];
            w = L.lw[idx];
            pwd = L.spw[dst];
            left = L.outw[dst];  // of dst's movable vertices, those still to come
          }
          const int32_t cap32 = cap > INT32_MAX ? INT32_MAX : int32_t(cap);
          int32_t delta = 0, p = -1;
          bool proven = false;
          // four moves a step, the proof asked for after each step; lanes K
          // and above are no moves (their parts match none, weight 0), and
          // positions from K on do not count
          for (int32_t m0 = 0; m0 < K && !proven; m0 += 4) {
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              const int m = m0 + x;
              const int32_t sm = __builtin_amdgcn_readlane(src, m), dm = __builtin_amdgcn_readlane(dst, m);
              const int32_t wm = __builtin_amdgcn_readlane(w, m);
              delta += dst == dm ? wm : 0;
              const int32_t out = dst == sm ? wm : 0;
              delta -= out;
              left -= out;
              const bool over = delta > 0 && pwd + delta > cap32;
              if (m < K && ballot(over) == 0) p = m;
            }
            const int32_t least = delta - left;
            proven = ballot(least > 0 && pwd + least > cap32) != 0;
          }
          // The sequence ends here: M moves, or every selected vertex.
          if (K == a.M || (nts <= 64 && ntop == npick)) proven = true;
          if (proven) {
            const bool mv = lane <= p;
            if (mv) {
              R.b.sv[lane] = v;
              R.mdst[lane] = dst;
              atomicAdd(&L.spw[src], -w);
              atomicAdd(&L.spw[dst], w);
            }
            const long long gs = wave_sum64(mv ? g : 0);
            if (lane == 0) {
              L.cut -= gs;
              L.thr = 1;
              rounds0 += 1;
              moved0 += p + 1;
              rounds_bytes += 8LL * ntop + 16LL * nts;
            }
          }
          if (lane == 0) L.pos = proven ? p : -2;
        }
        __syncthreads();
        pos = L.pos;
      }
    }
    if (!tested_all) count = nmov;  // some are selected: the movable vertex of smallest id is
    // 3. The long way.
    if (pos == -2) {
      if (!tested_all) {
        test(nmov, [&](int32_t i) { return int32_t(L.mi[i]); }, L.si, &L.nsel);
        __syncthreads();
        count = L.nsel;
      }
      // the best moves in order, and their balanced prefix
      const int32_t B = count < a.M ? count : a.M;
      const bool narrow = order_moves<4>(R, count, a.M, vb, ve, nullptr, SelectedIndex<CAP>{&L});
      BalanceOpt bo;
      bo.spw = L.spw;
      bo.mdst = R.mdst;
      bo.gain_in_key = true;
      bo.cut_given = true;
      if (t == 0) bo.cut_now = L.cut;
      pos = balance_prefix(R.b, L.dpw, kj, B, 0xffffffffull, a.part, a.dest, a.gain, a.vw, L.spw, cap, nullptr, nullptr,
                           &L.cut, bo);
      if (t == 0) {
        if (a.paths && count > a.M) {
          a.paths[3 * int64_t(j)] += 1;
          if (!narrow) a.paths[3 * int64_t(j) + 1] += 1;
        }
        if (a.hist) {
          a.hist[2 * rounds0] = B;
          a.hist[2 * rounds0 + 1] = pos;
        }
        L.thr = R.lz[2];
        rounds0 += 1;
        moved0 += pos + 1;
        rounds_bytes += 8LL * count + 16LL * B;
      }
      if (a.order) {
        int32_t* o = a.order + int64_t(j) * (a.M + 2);
        if (t < B) o[2 + t] = R.b.sv[t];
        if (t == 0) {
          o[0] = B;
          o[1] = pos;
        }
      }
    }
    // 4. apply: the movers and their neighbours are items [0, tot) -- mover m
    // owns [istart[m], istart[m] + deg + 1), first itself, then its row
    int32_t* istart = R.b.sw;  // free after the prefix
    int32_t* rstart = R.b.sw + 64;
    if (pos < 64 && t < 64) {
      int32_t es = 0, cnt = 0;
      if (t <= pos) {
        const int32_t v = R.b.sv[t];
        a.part[v] = R.mdst[t];
        es = a.xadj[v];
        cnt = a.xadj[v + 1] - es + 1;
      }
      const int32_t incl = seg_incl_scan<64>(cnt);
      istart[t] = incl - cnt;
      rstart[t] = es;
      if (t == 63) L.tot = incl;
    }
    __syncthreads();
    if (pos >= 64 || L.tot > kLoopItems) {
      // More than this workgroup should update: the worklist in memory, and
      // out, for the gain pass over the whole device.
      // Its table of first occurrences lies over the candidates' gains and
      // weights, which nobody reads any more.
      static_assert(offsetof(LoopLds<CAP>, lw) == offsetof(LoopLds<CAP>, lg) + sizeof(L.lg), "one array of 2 * CAP");
      constexpr int kBits = CAP == 4096 ? 13 : 11;
      static_assert((1 << kBits) == 2 * CAP, "slots");
      int32_t* table = &L.lg[0];
      for (int i = t; i < 2 * CAP; i += kBalThreads) table[i] = -1;
      __syncthreads();
      int32_t unused = 0;
      const int tot = apply_moves(R, pos, a.part, a.xadj, a.adj, a.upd, a.wl, a.wlc, false, &unused, table, kBits);
      if (t == 0) rounds_bytes += 12LL * tot;
      break;
    }
    const int tot = L.tot;
    if (t == 0) rounds_bytes += 12LL * tot;
    if (t < tot) {
      int lo = 0, hi = pos;  // last mover m with istart[m] <= t
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (istart[mid] <= t) lo = mid; else hi = mid - 1;
      }
      const int off = t - istart[lo];
      const int32_t u = off == 0 ? R.b.sv[lo] : a.adj[rstart[lo] + off - 1];
      uint32_t sl = (uint32_t(u) * 0x9E3779B1u) >> 22;  // 10 bits: the table's slots
      while (true) {
        const int32_t o = atomicCAS(&R.ht[sl], -1, u);
        if (o == -1) {
          // first occurrence: onto the worklist, with its row and weight
          const int32_t rs = a.xadj[u], d = a.xadj[u + 1] - rs;
          const bool lg = d > S;
          const int i = lg ? kLoopItems - 1 - atomicAdd(&L.nlong, 1) : atomicAdd(&L.nshort, 1);
          L.wv[i] = u;
          L.ws[i] = rs;
          L.wd[i] = d;
          L.ww[i] = a.vw[u];
          break;
        }
        if (o == u) break;
        sl = (sl + 1) & 1023;
      }
    }
    __syncthreads();
    // 5. the updated vertices leave the candidate list, their gains are
    // computed anew, and those that are candidates now are appended; the next
    // round's lists are cleared meanwhile
    clear();
    for (int32_t i = t; i < n; i += kBalThreads) {
      const int32_t v = L.lv[i];
      if (v < 0) continue;
      uint32_t sl = (uint32_t(v) * 0x9E3779B1u) >> 22;
      int32_t o;
      while ((o = R.ht[sl]) != -1) {
        if (o == v) {
          L.lv[i] = -1;
          break;
        }
        sl = (sl + 1) & 1023;
      }
    }
    // Units of work for a wave: a long row, or 64 / S short ones.
    const int32_t nshort = L.nshort, nlong = L.nlong;
    int32_t* hist = (wave < 8 ? reinterpret_cast<int32_t*>(R.b.sk) + wave * kGainInlineK
                              : reinterpret_cast<int32_t*>(R.b.ev2) + (wave - 8) * kGainInlineK);
    for (int32_t x = wave; x < nlong + (nshort + 64 / S - 1) / (64 / S); x += kBalThreads / 64) {
      const bool lg = x < nlong;
      const int32_t i = lg ? kLoopItems - 1 - x : (x - nlong) * (64 / S) + lane / S;
      const bool has = lg || i < nshort;
      int32_t v = 0, s = 0, d = 0, w = 0;
      if (has) {
        v = L.wv[i];
        s = L.ws[i];
        d = L.wd[i];
        w = L.ww[i];
      }
      auto emit = [&](int32_t u, int32_t p, bool any, int32_t g, int32_t q, int32_t du) {
        const bool up = any && g > 0;
        a.bnd[u] = any ? 1 : 0;
        a.gain[u] = up ? g : 0;
        a.dest[u] = up ? q : p;
        if (up) {
          const int y = atomicAdd(&L.n, 1);  // below CAP: n <= kFull before, and kLoopItems updated at most
          L.lv[y] = u;
          L.lg[y] = g;
          L.ld[y] = uint8_t(q);
          L.lp[y] = uint8_t(p);
          L.lw[y] = w;
        }
        ++upd_v;
        upd_e += du;
      };
      if (lg) gain_long(v, s, s + d, a.adj, a.w, a.part, kj, hist, emit);
      else gain_short<S>(has, v, s, d, a.adj, a.w, a.part, emit);
    }
    // The stores of part, gain and destination may take their time: the
    // barrier after the next round's first step comes before anyone reads them.
    lds_barrier();
    // Dropped entries are squeezed out when the next round might not find room.
    if (L.n > kFull) {
      n = L.n;
      int32_t ev[CAP / kBalThreads], eg[CAP / kBalThreads], ew[CAP / kBalThreads];
      uint8_t ed[CAP / kBalThreads], ep[CAP / kBalThreads];
#pragma unroll
      for (int x = 0; x < CAP / kBalThreads; ++x) {
        const int32_t i = t + x * kBalThreads;
        ev[x] = i < n ? L.lv[i] : -1;
        eg[x] = L.lg[i];
        ew[x] = L.lw[i];
        ed[x] = L.ld[i];
        ep[x] = L.lp[i];
      }
      __syncthreads();
      if (t == 0) L.n = 0;
      __syncthreads();
#pragma unroll
      for (int x = 0; x < CAP / kBalThreads; ++x) {
        const uint64_t m = ballot(ev[x] >= 0);
        if (m == 0) continue;
        int base = 0;
        if (lane == 0) base = atomicAdd(&L.n, popc64(m));
        base = __shfl(base, 0, 64);
        if (ev[x] >= 0) {
          const int i = base + popc64(m & lanemask_lt());
          L.lv[i] = ev[x];
          L.lg[i] = eg[x];
          L.lw[i] = ew[x];
          L.ld[i] = ed[x];
          L.lp[i] = ep[x];
        }
      }
      __syncthreads();
      if (L.n > kFull) break;  // too many candidates: left to the other kernels
    }
  }
  static_assert(sizeof(R.b.sk) == 8 * kGainInlineK * sizeof(int32_t) && sizeof(R.b.ev2) == sizeof(R.b.sk),
                "a histogram per wave in the sort buffers");
  __syncthreads();
  if (t < kj) pwj[t] = L.spw[t];
  // The candidate bits of the job's vertices: the list's, and for a round that
  // left the gains of its updates to the other pass, their own follow from it.
  // Words are shared with the neighbouring jobs: by atomics.
  for (int64_t w = w0 + t; w <= w1; w += kBalThreads)
    atomicAnd(reinterpret_cast<unsigned long long*>(&a.cand[w]), ~((unsigned long long)range_of(w)));
  __syncthreads();
  for (int i = t; i < L.n && i < CAP; i += kBalThreads)
    if (L.lv[i] >= 0) set_cand(a.cand, L.lv[i], true);
  // Algorithmic bytes: the rounds' own, tested rows' bounds and entries, and
  // the gain passes' (as the gain kernels count them).
  if (a.abytes) {
    const long long b = wave_sum64(4 * tested + 28LL * upd_v + 12LL * upd_e);
    if (lane == 0) atomicAdd(reinterpret_cast<unsigned long long*>(&a.abytes[j]), (unsigned long long)b);
  }
  if (t == 0) {
    if (a.abytes) atomicAdd(reinterpret_cast<unsigned long long*>(&a.abytes[j]), (unsigned long long)rounds_bytes);
    a.cut[j] = L.cut;
    a.thr[j] = L.thr;
    a.rounds[j] = rounds0;
    a.moved[j] = moved0;
    a.lastcnt[j] = count;
    if (count) atomicAdd(&a.status[0], 1);
    if (a.host.host) {
      tell(a.host, 0, count ? 1 : 0);
      tell(a.host, 1, 0);
      tell(a.host, 2, rounds0);
    }
  }
}

template <int S>
static void rounds_go(const RoundsArgs& a, int32_t nj, hipStream_t st) {
  // A long candidate list takes most of a compute unit's LDS; with more jobs
  // than compute units a short one lets two jobs share a unit.
  if (nj > 256) gk_launch(k_rounds<S, 1024>, dim3(nj), dim3(kBalThreads), 0, st, a);
  else gk_launch(k_rounds<S, 4096>, dim3(nj), dim3(kBalThreads), 0, st, a);
}

int launch_rounds(const RoundsArgs& a, int32_t nj, int lanes, hipStream_t st) {
  if (nj <= 0) return 0;
  if (a.M > kBalMax) return GK_ERR_LIMIT;
  if (lanes <= 8) rounds_go<8>(a, nj, st);
  else if (lanes <= 16) rounds_go<16>(a, nj, st);
  else rounds_go<32>(a, nj, st);
  return hip_status();
}

}  // namespace gkd
