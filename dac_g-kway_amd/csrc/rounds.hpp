// Pieces of a refinement round that the two round kernels share (batch.hip:
// one round, one workgroup per job, after the selection kernels; rounds.hip:
// many rounds, one workgroup per job): the workgroup's LDS and the ordered
// list of the best moves.
#pragma once
#include "balance.hpp"
#include "dev_common.hpp"

namespace gkd {

struct RoundLds {
  BalanceLds b;  // b.sk doubles as the 2048-bin radix histogram
  int32_t mdst[kBalMax];  // each ordered move's destination
  int32_t ht[1024];  // the apply's table of first occurrences (cleared at the start)
  int32_t ws[40];
  int32_t misc[4];
  int32_t lz[4];  // deferred tests: selected count; next threshold's digit; next threshold
};

// Gain threshold of the next round's selection: aim at about
// kLazyFactor * M tested vertices per job.
constexpr int kLazyFactor = 2;

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t x) {
  return wave_reduce(x, [](uint32_t a, uint32_t b) { return b < a ? b : a; });
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
  return wave_reduce(x, [](uint32_t a, uint32_t b) { return b > a ? b : a; });
}

// Bits needed to hold values 0..x (at least 1).
__device__ __forceinline__ int bits_of(uint32_t x) { return x ? 32 - __clz(x) : 1; }

// Selected vertices in a list, gains by vertex.
struct SelectedList {
  const int32_t* seg;
  const int32_t* gain;
  __device__ int32_t vertex(int32_t i) const { return seg[i]; }
  // ascending order = gain descending (the mvRequest order of
  // gkway/move_request.hpp:36-41, with the id below it)
  __device__ uint32_t gain_key(int32_t, int32_t v) const { return uint32_t(0x7fffffff - gain[v]); }
};

// The min(count, M) best of the count selected vertices of a job with ids
// [vb, ve), by (gain desc, id asc), sorted into R.b.sk as (gain key << 32 |
// vertex), slots behind them the largest key.  sel.vertex(i) and
// sel.gain_key(i, vertex) give the selected vertices.  hk: scratch for count
// keys, used beyond kKeep * kBalThreads selected (kKeep a thread stay in
// registers).  R.lz[2] gets the gain threshold
// of the job's next round when one is due.  Returns whether the keys were
// sorted as 32-bit words.  Every thread of the block calls it after a barrier;
// it ends with one.
template <int kKeep, class Sel>
__device__ __forceinline__ bool order_moves(RoundLds& R, int32_t count, int32_t M, int32_t vb, int32_t ve, uint32_t* hk,
                                            const Sel& sel) {
  const int t = threadIdx.x;
  const int32_t B = count < M ? count : M;
  bool narrow = false;  // keys already sorted as 32-bit compressed keys
  if (count <= M) {
    R.b.sk[t] = ~0ull;
    if (t < count) {
      const int32_t v = sel.vertex(t);
      R.b.sk[t] = (uint64_t(sel.gain_key(t, v)) << 32) | uint64_t(uint32_t(v));
    }
  } else {
    // Exact top-B by radix select on a compressed key: (gain key - its
    // minimum) above (id - first id of the job); the key is monotone in
    // (gain desc, id asc) and has only as many bits as the ranges need.
    // Pass 0 gathers the gain keys and finds their range; the passes then
    // use 11-bit digits from the top.  Up to kKeep keys per thread stay in
    // registers across the passes (with their vertices); more go through the
    // scratch hk.
    const bool inreg = count <= kKeep * kBalThreads;
    uint32_t hr[kKeep];
    int32_t vr[kKeep];
    uint32_t lo = 0xffffffffu, hi = 0;
    if (inreg) {
#pragma unroll
      for (int r = 0; r < kKeep; ++r) {
        const int32_t i = t + r * kBalThreads;
        vr[r] = i < count ? sel.vertex(i) : vb;
      }
#pragma unroll
      for (int r = 0; r < kKeep; ++r) {
        if (t + r * kBalThreads < count) {
          const uint32_t h = sel.gain_key(t + r * kBalThreads, vr[r]);
          hr[r] = h;
          lo = h < lo ? h : lo;
          hi = h > hi ? h : hi;
        }
      }
    } else {
      for (int32_t i = t; i < count; i += kBalThreads) {
        const uint32_t h = sel.gain_key(i, sel.vertex(i));
        hk[i] = h;
        lo = h < lo ? h : lo;
        hi = h > hi ? h : hi;
      }
    }
    // fn(gain key, vertex) for every selected vertex this thread holds
    auto each = [&](auto&& fn) {
      if (inreg) {
#pragma unroll
        for (int r = 0; r < kKeep; ++r)
          if (t + r * kBalThreads < count) fn(hr[r], vr[r]);
      } else {
        for (int32_t i = t; i < count; i += kBalThreads) fn(hk[i], sel.vertex(i));
      }
    };
    lo = wave_min_u32(lo);
    hi = wave_max_u32(hi);
    if (lane_id() == 0) {
      R.ws[t >> 6] = int32_t(lo);
      R.ws[16 + (t >> 6)] = int32_t(hi);
    }
    __syncthreads();
    if (t == 0) {
      uint32_t a2 = 0xffffffffu, b2 = 0;
      for (int w = 0; w < kBalThreads / 64; ++w) {
        a2 = uint32_t(R.ws[w]) < a2 ? uint32_t(R.ws[w]) : a2;
        b2 = uint32_t(R.ws[16 + w]) > b2 ? uint32_t(R.ws[16 + w]) : b2;
      }
      R.ws[32] = int32_t(a2);
      R.ws[33] = int32_t(b2);
    }
    __syncthreads();
    const uint32_t hmin = uint32_t(R.ws[32]), hrange = uint32_t(R.ws[33]) - hmin;
    const int ib = bits_of(uint32_t(ve - vb - 1));
    const int tb = bits_of(hrange) + ib;
    auto ckey = [&](uint32_t h, int32_t v) -> uint64_t {
      return (uint64_t(h - hmin) << ib) | uint64_t(uint32_t(v - vb));
    };
    constexpr int kDigit = 11;
    int32_t* hist = reinterpret_cast<int32_t*>(R.b.sk);  // 2048 ints, free until the keys are collected
    uint64_t prefix = 0, pmask = 0;
    int32_t need = B;
    for (int shift = ((tb + kDigit - 1) / kDigit - 1) * kDigit; shift >= 0; shift -= kDigit) {
      hist[2 * t] = 0;
      hist[2 * t + 1] = 0;
      __syncthreads();
      each([&](uint32_t h, int32_t v) {
        const uint64_t key = ckey(h, v);
        if ((key & pmask) == prefix) atomicAdd(&hist[(key >> shift) & 2047], 1);
      });
      __syncthreads();
      // The digit where the running count reaches `need`: a block scan over
      // the 2048 bins, two per thread.
      const int32_t h0 = hist[2 * t], h1 = hist[2 * t + 1];
      int tot;
      const int32_t ex = block_excl_scan_1024(h0 + h1, &tot, R.ws);
      if (ex < need && need <= ex + h0) {
        R.misc[0] = 2 * t;
        R.misc[1] = ex;
        R.misc[3] = h0;
      } else if (ex + h0 < need && need <= ex + h0 + h1) {
        R.misc[0] = 2 * t + 1;
        R.misc[1] = ex + h0;
        R.misc[3] = h1;
      }
      // First digit: also the digit holding rank kLazyFactor * M, for the
      // next round's gain threshold.
      const bool lazy = pmask == 0 && count > kLazyFactor * M;
      const int32_t r2 = kLazyFactor * M;
      if (lazy && ex < r2 && r2 <= ex + h0) R.lz[1] = 2 * t;
      else if (lazy && ex + h0 < r2 && r2 <= ex + h0 + h1) R.lz[1] = 2 * t + 1;
      __syncthreads();
      if (lazy && t == 0) {
        // every key in digits <= lz[1] has a gain key <= hu, i.e. a gain >= 0x7fffffff - hu
        const uint64_t top = ((uint64_t(R.lz[1]) + 1) << shift) - 1;
        const uint64_t hu = uint64_t(hmin) + (top >> ib);
        R.lz[2] = hu >= 0x7ffffffeull ? 1 : int32_t(0x7fffffffull - hu);
      }
      need -= R.misc[1];
      prefix |= uint64_t(R.misc[0]) << shift;
      pmask |= 2047ull << shift;
      // Every key of the chosen bucket is needed: the B best are the keys
      // whose digits so far are <= prefix, and the lower digits can stay
      // unread.  (Only R.misc[2], R.b.sk and R.b.sv are written next; none
      // of them is read in this pass after its last barrier.)
      if (need == R.misc[3]) break;
      __syncthreads();
    }
    // (key & pmask) <= prefix holds for exactly the B best keys: prefix is
    // the B-th smallest key's leading digits and the keys are distinct.
    // Compressed keys of at most 32 bits are sorted as 32-bit words (half the
    // shuffle and LDS traffic of the 64-bit keys) and expanded afterwards.
    narrow = tb <= 32;
    uint32_t* nk = reinterpret_cast<uint32_t*>(R.b.sv);  // free until balance_prefix
    if (t == 0) R.misc[2] = 0;
    if (narrow) nk[t] = 0xffffffffu;
    else R.b.sk[t] = ~0ull;
    __syncthreads();
    each([&](uint32_t h, int32_t v) {
      const uint64_t ck = ckey(h, v);
      if ((ck & pmask) <= prefix) {
        const int slot = atomicAdd(&R.misc[2], 1);
        if (narrow) nk[slot] = uint32_t(ck);
        else R.b.sk[slot] = (uint64_t(h) << 32) | uint64_t(uint32_t(v));
      }
    });
    if (narrow) {
      __syncthreads();
      int P = 128;
      while (P < B) P <<= 1;
      bitonic_lds(nk, P);
      const uint32_t ck = nk[t];
      const uint32_t idm = uint32_t((1ull << ib) - 1);
      R.b.sk[t] = t < B ? (uint64_t(hmin + (ck >> ib)) << 32) | uint64_t(uint32_t(vb) + (ck & idm)) : ~0ull;
    }
  }
  __syncthreads();
  if (!narrow) lds_bitonic(R.b, B);
  return narrow;
}

// Applies moves 0..pos in R.b.sv to R.mdst (balance_prefix read part[] before
// its last barrier) and appends the movers and their neighbours to the gain
// worklist, each once: wl at *wlc, by an atomic per pass, or with sole (one
// workgroup owns the list, empty before) at a running offset whose end thread
// 0 gets in *wrun_out.  R.ht is all -1 before, and so are the 2^big_bits slots
// of LDS at big, if there are any (big_bits > 0).  Returns the items looked at.
__device__ __forceinline__ int apply_moves(RoundLds& R, int pos, int32_t* part, const int32_t* __restrict__ xadj,
                                           const int32_t* __restrict__ adj, int32_t* upd, int32_t* wl, int32_t* wlc,
                                           bool sole, int32_t* wrun_out, int32_t* big, int big_bits) {
  const int t = threadIdx.x;
  // The movers and their neighbours are items [0, tot) -- mover m owns
  // [istart[m], istart[m] + deg + 1), first itself, then its row -- dealt out
  // in passes of kApplyPer items per thread.  An item's vertex joins the gain
  // worklist if its update flag was clear.  One workgroup (one job) owns the
  // worklist count, which the selection zeroed: it appends at a running
  // offset and stores the count at the end; several jobs append with one
  // global atomic per pass.
  constexpr int kApplyPer = 8;
  int32_t* istart = R.b.sw;     // free after balance_prefix
  int32_t* rstart = R.b.cover;  // likewise
  int tot = 0;
  // Items [a0, a0 + kApplyPer) of [0, tot): their vertices (-1 past the end)
  // and the bit mask of the first occurrences.  With a table ht (LDS, 2^bits
  // slots, all -1, at least twice the items): first occurrences within the
  // round by insertion into ht, the update flag then set by a plain store --
  // every flag is clear when a round starts (the gain pass of the previous
  // round cleared those it set).  Without: by the update flag's atomic swap,
  // which a workgroup waits for (7100 items: 25 us, with the table 19).
  constexpr int kHt = sizeof(R.ht) / sizeof(int32_t);
  static_assert(kHt == 1024, "10-bit table index");
  auto take = [&](int a0, int32_t (&us)[kApplyPer], int32_t* ht, int bits) -> uint32_t {
    uint32_t win = 0;
#pragma unroll
    for (int i = 0; i < kApplyPer; ++i) us[i] = -1;
    if (a0 >= tot) return 0;
    int lo = 0, hi = pos;  // last mover m with istart[m] <= a0
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (istart[mid] <= a0) lo = mid; else hi = mid - 1;
    }
    int m = lo;
#pragma unroll
    for (int i = 0; i < kApplyPer; ++i) {
      const int e2 = a0 + i;
      if (e2 < tot) {
        while (m < pos && istart[m + 1] <= e2) ++m;
        const int off = e2 - istart[m];
        us[i] = off == 0 ? R.b.sv[m] : adj[rstart[m] + off - 1];
      }
    }
    if (ht) {
#pragma unroll
      for (int i = 0; i < kApplyPer; ++i) {
        if (us[i] < 0) continue;
        uint32_t sl = (uint32_t(us[i]) * 0x9E3779B1u) >> (32 - bits);
        while (true) {
          const int32_t o = atomicCAS(&ht[sl], -1, us[i]);
          if (o == -1) {
            win |= 1u << i;
            upd[us[i]] = 1;
            break;
          }
          if (o == us[i]) break;
          sl = (sl + 1) & ((1u << bits) - 1);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < kApplyPer; ++i)
        if (us[i] >= 0 && atomicExch(&upd[us[i]], 1) == 0) win |= 1u << i;
    }
    return win;
  };
  int32_t& wrun = *wrun_out;
  if (pos < 64) {
    // At most 64 movers (the usual case once the parts sit at the cap): wave
    // 0 alone, with wave-level scans and no block barriers.
    if (t < 64) {
      const bool mv = t <= pos;
      int32_t es = 0, cnt = 0;
      if (mv) {
        const int32_t v = R.b.sv[t];
        part[v] = R.mdst[t];
        es = xadj[v];
        cnt = xadj[v + 1] - es + 1;
      }
      const int32_t incl = seg_incl_scan<64>(cnt);
      tot = __shfl(incl, 63, 64);
      if (mv) {
        istart[t] = incl - cnt;
        rstart[t] = es;
      }
      // first occurrences in LDS when the items fit the table
      int32_t* ht = tot <= kHt / 2 ? R.ht : nullptr;
      int bits = 10;
      if (!ht && big_bits > 0 && 2 * int64_t(tot) <= (int64_t(1) << big_bits)) {
        ht = big;
        bits = big_bits;
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (int pb = 0; pb < tot; pb += kApplyPer * 64) {
        int32_t us[kApplyPer];
        const uint32_t win = take(pb + kApplyPer * t, us, ht, bits);
        const int c = __popc(win);
        const int wincl = seg_incl_scan<64>(c);
        const int wtot = __shfl(wincl, 63, 64);
        int base = wrun;
        if (!sole) {
          int b0 = 0;
          if (t == 0 && wtot > 0) b0 = atomicAdd(&wlc[0], wtot);
          base = __shfl(b0, 0, 64);
        }
        int r = base + wincl - c;
#pragma unroll
        for (int i = 0; i < kApplyPer; ++i)
          if ((win >> i) & 1u) wl[r++] = us[i];
        wrun += wtot;
      }
    }
  } else {
    const bool mv = t <= pos;
    int32_t es = 0, deg = 0;
    if (mv) {
      const int32_t v = R.b.sv[t];
      part[v] = R.mdst[t];
      es = xadj[v];
      deg = xadj[v + 1] - es;
    }
    const int ib = block_excl_scan_1024(mv ? deg + 1 : 0, &tot, R.ws);
    if (mv) {
      istart[t] = ib;
      rstart[t] = es;
    }
    __syncthreads();
    int32_t* ht = big_bits > 0 && 2 * int64_t(tot) <= (int64_t(1) << big_bits) ? big : nullptr;
    for (int pb = 0; pb < tot; pb += kApplyPer * kBalThreads) {
      int32_t us[kApplyPer];
      const uint32_t win = take(pb + kApplyPer * t, us, ht, big_bits);
      int wtot;
      const int wex = block_excl_scan_1024(__popc(win), &wtot, R.ws);
      if (t == 0) {
        if (sole) {
          R.misc[0] = wrun;
          wrun += wtot;
        } else if (wtot > 0) {
          R.misc[0] = atomicAdd(&wlc[0], wtot);
        }
      }
      __syncthreads();
      const int wbase = R.misc[0] + wex;
      int r = 0;
#pragma unroll
      for (int i = 0; i < kApplyPer; ++i)
        if ((win >> i) & 1u) wl[wbase + r++] = us[i];
      __syncthreads();  // R.misc[0] is reused by the next pass
    }
  }
  return tot;
}

}  // namespace gkd
