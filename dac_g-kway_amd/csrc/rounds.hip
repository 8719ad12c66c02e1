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
// runs at its own pace and none waits for another's rounds.
//
// The state in memory after a launch is the one the separate kernels would
// leave after as many rounds, so the two can take turns: a job with more
// candidates than the list holds is left to them, and a round that updates
// more vertices than one workgroup should (a large graph's first rounds)
// appends them to the worklist and leaves, for the gain pass over the whole
// device and another launch.
#include <algorithm>

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

static_assert(kLoopItems <= 1024 / 2, "the table of first occurrences stays half empty");
static_assert(kLoopItems <= kBalMax, "the worklist lies in the cover array");

template <int CAP>
struct LoopLds {
  RoundLds r;
  int32_t lv[CAP], lg[CAP], ld[CAP], lw[CAP];  // candidates: vertex, gain, destination, weight
  uint16_t mi[CAP], si[CAP];                   // list indexes: movable with gain >= threshold; selected
  uint32_t bits[kMovableBits / 32];
  int32_t spw[kGainInlineK], dpw[kGainInlineK];  // part weights, and the balanced prefix's scratch
  long long cut;
  int32_t n, nmov, nsel, nwl, tot, thr;
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

template <int S, int CAP>
__global__ void __launch_bounds__(kBalThreads) k_rounds(const RoundsArgs a) {
  static_assert(CAP <= 4 * kBalThreads, "the ordered list keeps four keys per thread");
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
  if (a.lastcnt[j] == 0) return;  // converged in an earlier launch
  const int32_t vb = a.v_off[j], ve = a.v_off[j + 1];
  const int32_t kj = a.kk[j];
  const long long cap = a.cap[j];
  int32_t* pwj = a.pw + a.pw_off[j];
  const bool exact_bits = ve - vb <= kMovableBits;
  // The candidates of the job's id range.
  const int64_t w0 = int64_t(vb) >> 6, w1 = ve > vb ? (int64_t(ve) - 1) >> 6 : w0 - 1;
  auto word_of = [&](int64_t w) -> uint64_t {
    const int64_t lo = vb > (w << 6) ? vb - (w << 6) : 0;
    const int64_t hi = ve < (w << 6) + 64 ? ve - (w << 6) : 64;
    return a.cand[w] & (hi - lo == 64 ? ~0ull : (((1ull << (hi - lo)) - 1) << lo));
  };
  int c = 0;
  for (int64_t w = w0 + t; w <= w1; w += kBalThreads) c += popc64(word_of(w));
  int n;
  int at = block_excl_scan_1024(c, &n, R.ws);
  if (n > CAP) {  // left to the kernels that select over the whole device
    if (t == 0) {
      atomicAdd(&a.status[0], 1);
      atomicAdd(&a.status[1], 1);
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
  __syncthreads();
  for (int i = t; i < n; i += kBalThreads) {
    const int32_t v = L.lv[i];
    L.lg[i] = a.gain[v];
    L.ld[i] = a.dest[v];
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
  // selected ones to L.si: a lane per row of up to kLoopShortRow entries, eight
  // neighbours a step, longer rows by the whole wave.
  auto test = [&](int32_t m, auto&& index) {
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
      wave_append(sel, uint16_t(idx), L.si, &L.nsel);
    }
  };

  int32_t rounds0 = 0;
  long long moved0 = 0;
  if (t == 0) {
    rounds0 = a.rounds[j];
    moved0 = a.moved[j];
  }
  int32_t count = 0;
  for (int32_t r = 0; r < a.max_rounds; ++r) {
    // 1. movable candidates: bitmap, and the list of those at or above the
    // gain threshold
    L.bits[t] = 0;
    L.bits[t + kBalThreads] = 0;
    static_assert(kMovableBits / 32 == 2 * kBalThreads, "two bitmap words per thread");
    R.ht[t] = -1;
    if (t == 0) {
      L.nmov = 0;
      L.nsel = 0;
      L.nwl = 0;
      R.lz[2] = 1;  // next threshold: test everything unless set below
    }
    __syncthreads();
    n = L.n;
    const int32_t thr = L.thr;
    for (int32_t i0 = wave * 64; i0 < n; i0 += kBalThreads) {
      const int32_t i = i0 + lane;
      bool mv = false;
      if (i < n && fits(L.ld[i], L.lw[i])) {
        const uint32_t b = uint32_t(L.lv[i] - vb) & (kMovableBits - 1);
        atomicOr(&L.bits[b >> 5], 1u << (b & 31));
        mv = L.lg[i] >= thr;
      }
      wave_append(mv, uint16_t(i), L.mi, &L.nmov);
    }
    __syncthreads();
    // 2. selection: no smaller-id movable neighbour; the movable vertices
    // below the threshold only when it leaves fewer than M
    const int32_t nmov = L.nmov;
    test(nmov, [&](int32_t i) { return int32_t(L.mi[i]); });
    __syncthreads();
    count = L.nsel;
    if (count < a.M && thr > 1) {
      if (a.paths && t == 0) a.paths[3 * int64_t(j) + 2] += 1;
      __syncthreads();  // every thread has read nsel
      test(n, [&](int32_t i) { return L.lg[i] < thr && fits(L.ld[i], L.lw[i]) ? i : -1; });
      __syncthreads();
      count = L.nsel;
    }
    if (count == 0) {
      if (t == 0) L.thr = 1;
      break;
    }
    // 3. the best moves in order, and their balanced prefix
    const int32_t B = count < a.M ? count : a.M;
    const bool narrow = order_moves(R, count, a.M, vb, ve, nullptr, SelectedIndex<CAP>{&L});
    BalanceOpt bo;
    bo.spw = L.spw;
    bo.mdst = R.mdst;
    bo.gain_in_key = true;
    bo.cut_given = true;
    if (t == 0) bo.cut_now = L.cut;
    const int pos = balance_prefix(R.b, L.dpw, kj, B, 0xffffffffull, a.part, a.dest, a.gain, a.vw, L.spw, cap, nullptr,
                                   nullptr, &L.cut, bo);
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
    }
    if (a.order) {
      int32_t* o = a.order + int64_t(j) * (a.M + 2);
      if (t < B) o[2 + t] = R.b.sv[t];
      if (t == 0) {
        o[0] = B;
        o[1] = pos;
      }
    }
    // 4. apply: the movers and their neighbours are items [0, tot) -- mover m
    // owns [istart[m], istart[m] + deg + 1), first itself, then its row
    int32_t* istart = R.b.sw;  // free after balance_prefix
    int32_t* rstart = R.b.sw + 64;
    int32_t* wl = R.b.cover;
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
      int32_t unused = 0;
      const int tot = apply_moves(R, pos, a.part, a.xadj, a.adj, a.upd, a.wl, a.wlc, false, &unused);
      if (t == 0) rounds_bytes += 8LL * count + 16LL * B + 12LL * tot;
      break;
    }
    const int tot = L.tot;
    if (t == 0) rounds_bytes += 8LL * count + 16LL * B + 12LL * tot;
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
          wl[atomicAdd(&L.nwl, 1)] = u;
          break;
        }
        if (o == u) break;
        sl = (sl + 1) & 1023;
      }
    }
    __syncthreads();
    // 5. gains of the updated vertices; the candidate list without the
    // updated vertices, and with those that are candidates now
    int32_t ev[CAP / kBalThreads], eg[CAP / kBalThreads], ed[CAP / kBalThreads], ew[CAP / kBalThreads];
    bool keep[CAP / kBalThreads];
#pragma unroll
    for (int x = 0; x < CAP / kBalThreads; ++x) {
      const int32_t i = t + x * kBalThreads;
      keep[x] = i < n;
      if (keep[x]) {
        ev[x] = L.lv[i];
        eg[x] = L.lg[i];
        ed[x] = L.ld[i];
        ew[x] = L.lw[i];
        uint32_t sl = (uint32_t(ev[x]) * 0x9E3779B1u) >> 22;
        int32_t o;
        while ((o = R.ht[sl]) != -1) {
          if (o == ev[x]) {
            keep[x] = false;
            break;
          }
          sl = (sl + 1) & 1023;
        }
      }
    }
    if (t == 0) L.n = 0;
    const int32_t nwl = L.nwl;
    __syncthreads();
#pragma unroll
    for (int x = 0; x < CAP / kBalThreads; ++x) {
      const uint64_t m = ballot(keep[x]);
      if (m == 0) continue;
      int base = 0;
      if (lane == 0) base = atomicAdd(&L.n, popc64(m));
      base = __shfl(base, 0, 64);
      if (keep[x]) {
        const int i = base + popc64(m & lanemask_lt());  // below CAP while only kept entries
        if (i < CAP) {                                    // are in; new ones may come between
          L.lv[i] = ev[x];
          L.lg[i] = eg[x];
          L.ld[i] = ed[x];
          L.lw[i] = ew[x];
        }
      }
    }
    int32_t* hist = (wave < 8 ? reinterpret_cast<int32_t*>(R.b.sk) + wave * kGainInlineK
                              : reinterpret_cast<int32_t*>(R.b.ev2) + (wave - 8) * kGainInlineK);
    for (int32_t e0 = wave * (64 / S); e0 < nwl; e0 += kBalThreads / S) {
      const int32_t e = e0 + lane / S;
      int32_t v = 0, s = 0, d = 0;
      if (e < nwl) {
        v = wl[e];
        s = a.xadj[v];
        d = a.xadj[v + 1] - s;
      }
      gain_pass<S>(e < nwl, v, s, d, a.adj, a.w, a.part, kj, hist,
                   [&](int32_t u, int32_t p, bool any, int32_t g, int32_t q, int32_t du) {
                     const bool up = any && g > 0;
                     a.bnd[u] = any ? 1 : 0;
                     a.gain[u] = up ? g : 0;
                     a.dest[u] = up ? q : p;
                     set_cand(a.cand, u, up);
                     if (up) {
                       const int i = atomicAdd(&L.n, 1);
                       if (i < CAP) {
                         L.lv[i] = u;
                         L.lg[i] = g;
                         L.ld[i] = q;
                         L.lw[i] = a.vw[u];
                       }
                     }
                     ++upd_v;
                     upd_e += du;
                   });
    }
    __syncthreads();
    if (L.n > CAP) break;  // the next launch builds the list anew, or leaves the job to the other kernels
  }
  static_assert(sizeof(R.b.sk) == 8 * kGainInlineK * sizeof(int32_t) && sizeof(R.b.ev2) == sizeof(R.b.sk),
                "a histogram per wave in the sort buffers");
  __syncthreads();
  if (t < kj) pwj[t] = L.spw[t];
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

// State of a level's rounds before the first one: per job the counters, and
// the words that the launches share.
__global__ void __launch_bounds__(256) k_rounds_init(int32_t nj, int32_t* __restrict__ lastcnt,
                                                     int32_t* __restrict__ thr, int32_t* __restrict__ rounds,
                                                     long long* __restrict__ moved, long long* __restrict__ abytes,
                                                     int32_t* __restrict__ wlc, int32_t* __restrict__ status) {
  const int32_t j = blockIdx.x * 256 + threadIdx.x;
  if (j < 4) {
    wlc[j] = 0;
    status[j] = 0;
  }
  if (j >= nj) return;
  lastcnt[j] = 1;
  thr[j] = 1;
  rounds[j] = 0;
  moved[j] = 0;
  abytes[j] = 0;
}

int launch_rounds_init(int32_t nj, int32_t* lastcnt, int32_t* thr, int32_t* rounds, long long* moved,
                       long long* abytes, int32_t* wlc, int32_t* status, hipStream_t st) {
  k_rounds_init<<<grid_for(std::max(nj, 4), 256), 256, 0, st>>>(nj, lastcnt, thr, rounds, moved, abytes, wlc, status);
  return hip_status();
}

}  // namespace gkd
