// Kernels of the batched form: many graphs (jobs) packed into one CSR with
// global vertex ids, processed by one launch per stage.  Jobs never share an
// edge, so the coarsening kernels of coarsen.hip run on the pack unchanged;
// this file adds the per-job glue:
//   pack / unpack    descriptor-driven copies from per-job slices (local ids)
//                    into a pack (global ids), and of partitions back out;
//   job offsets      first coarse id / first coarse entry of every job;
//   rounds           independent-set selection with per-job caps and part
//                    weights as a bitmask, then one workgroup per job for the
//                    ordered move list, the best moves by (gain desc, id asc),
//                    the balanced prefix (balance.hpp) and the apply;
//   cut              final cut and part weights with per-job offsets.
// Every per-job result equals the single-graph path's: ids keep their order
// inside a job and every order-sensitive step is segmented by job.
#include <algorithm>

#include "balance.hpp"
#include "batch.hpp"
#include "kernels.hpp"
#include "prim.hpp"
#include "rounds.hpp"
#include "../../include/gkway.h"

namespace gkd {

static inline int hip_status() { return hipGetLastError() == hipSuccess ? 0 : GK_ERR_HIP; }

// Index j in [lo, hi) with off[j] <= i < off[j+1] (off is nondecreasing;
// the caller knows off[lo] <= i < off[hi]).
__device__ __forceinline__ int32_t job_in(const int32_t* __restrict__ off, int32_t lo, int32_t hi, int64_t i) {
  while (hi - lo > 1) {
    const int32_t mid = (lo + hi) >> 1;
    if (off[mid] <= i) lo = mid; else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ int32_t job_of(const int32_t* __restrict__ off, int32_t nj, int64_t i) {
  return job_in(off, 0, nj, i);
}

// Descriptor-driven copies: a block covers kPackPer * 256 consecutive items
// (vertices or entries) and looks up the jobs of its first and last item
// once; items of a block inside one job (nearly all) then need no per-item
// search.
constexpr int kPackPer = 8;

__device__ __forceinline__ void block_jobs(const int32_t* __restrict__ off, int32_t nj, int64_t total, int64_t i0,
                                           int32_t* sj) {
  if (threadIdx.x == 0) {
    const int64_t last = (i0 + int64_t(kPackPer) * 256 < total ? i0 + int64_t(kPackPer) * 256 : total) - 1;
    sj[0] = job_of(off, nj, i0);
    sj[1] = job_in(off, sj[0], nj, last);
  }
  __syncthreads();
}

// ---------------------------------------------------------------- pack
__global__ void __launch_bounds__(256) k_pack_vert(int32_t nj, const PackSrc* __restrict__ src,
                                                   const int32_t* __restrict__ v_off,
                                                   const int32_t* __restrict__ e_off, int32_t ntot, int32_t etot,
                                                   int32_t* __restrict__ xadj, int32_t* __restrict__ vw) {
  __shared__ int32_t sj[2];
  const int64_t i0 = int64_t(blockIdx.x) * kPackPer * 256;
  block_jobs(v_off, nj, ntot, i0, sj);
  if (blockIdx.x == 0 && threadIdx.x == 0) xadj[ntot] = etot;
  for (int r = 0; r < kPackPer; ++r) {
    const int64_t i = i0 + r * 256 + threadIdx.x;
    if (i >= ntot) break;
    const int32_t j = sj[0] == sj[1] ? sj[0] : job_in(v_off, sj[0], sj[1] + 1, i);
    const PackSrc& s = src[j];
    const int32_t li = int32_t(i - v_off[j]);
    xadj[i] = e_off[j] + (s.xadj[li] - s.xbase);
    vw[i] = s.vw[li];
  }
}

// The vertex side of a refinement pack, with the start of its rounds: rows and
// weights, expand_partition (gkway/uncoarsen.hpp:325-356) straight from the
// coarse level's arrays (levels entered by projection) or the carried state
// (resumed ones), the candidate bits, the worklist of the projected boundary
// and the jobs' state words.  Five kernels (pack, packed coarse arrays,
// projection, candidates, compaction) took 18 + 12 + 4 + 2 + 9 us a step before,
// most of it launches and chains of small loads (160 graphs of 500 to 50000
// vertices).
__global__ void __launch_bounds__(256) k_pack_refine(int32_t nj, const PackSrc* __restrict__ src,
                                                     const int32_t* __restrict__ v_off,
                                                     const int32_t* __restrict__ e_off, int32_t ntot, int32_t etot,
                                                     int32_t* __restrict__ xadj, int32_t* __restrict__ vw,
                                                     const RefineStart o) {
  __shared__ int32_t sj[2];
  __shared__ int wsum[4];
  __shared__ int base_s;
  const int64_t i0 = int64_t(blockIdx.x) * kPackPer * 256;
  const int wave = threadIdx.x >> 6;
  block_jobs(v_off, nj, ntot, i0, sj);
  if (blockIdx.x == 0 && threadIdx.x == 0) xadj[ntot] = etot;
  for (int64_t j = int64_t(blockIdx.x) * 256 + threadIdx.x; j < nj; j += int64_t(gridDim.x) * 256) {
    o.lastcnt[j] = 1;
    o.thr[j] = 1;
  }
  uint64_t m[kPackPer];
  int tot = 0;
#pragma unroll
  for (int r = 0; r < kPackPer; ++r) {
    const int64_t i = i0 + r * 256 + threadIdx.x;
    bool up = false, cnd = false;
    if (i < ntot) {
      const int32_t j = sj[0] == sj[1] ? sj[0] : job_in(v_off, sj[0], sj[1] + 1, i);
      const PackSrc& s = src[j];
      const int32_t li = int32_t(i - v_off[j]);
      xadj[i] = e_off[j] + (s.xadj[li] - s.xbase);
      vw[i] = s.vw[li];
      o.vjob[i] = j;
      // No source map: the coarse side has the level's own ids (resumed).
      const int32_t c = s.cmap ? s.cmap[li] - s.cbase : li;
      const int32_t p = s.cpart[c];
      const bool b = s.cbnd[c] != 0;
      int32_t g = 0, d = p;
      if (s.cgain) {
        g = s.cgain[c];
        d = s.cdest[c];
      } else {
        up = b;
      }
      o.part[i] = p;
      o.bnd[i] = b ? 1 : 0;
      o.gain[i] = g;
      o.dest[i] = d;
      o.upd[i] = up ? 1 : 0;
      cnd = b && g > 0;
    }
    m[r] = ballot(up);
    tot += popc64(m[r]);
    const uint64_t cb = ballot(cnd);
    if (lane_id() == 0 && i < ntot) o.cand[i >> 6] = cb;
  }
  if (lane_id() == 0) wsum[wave] = tot;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int t = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    base_s = t ? atomicAdd(o.cnt, t) : 0;
  }
  __syncthreads();
  int off = base_s;
  for (int w = 0; w < wave; ++w) off += wsum[w];
  const uint64_t lt = lanemask_lt();
#pragma unroll
  for (int r = 0; r < kPackPer; ++r) {
    if ((m[r] >> lane_id()) & 1ull) o.wl[off + popc64(m[r] & lt)] = int32_t(i0 + r * 256 + threadIdx.x);
    off += popc64(m[r]);
  }
}

__global__ void __launch_bounds__(256) k_pack_edge(int32_t nj, const PackSrc* __restrict__ src,
                                                   const int32_t* __restrict__ v_off,
                                                   const int32_t* __restrict__ e_off, int32_t etot,
                                                   int32_t* __restrict__ adj, int32_t* __restrict__ w) {
  __shared__ int32_t sj[2];
  const int64_t i0 = int64_t(blockIdx.x) * kPackPer * 256;
  block_jobs(e_off, nj, etot, i0, sj);
  if (sj[0] == sj[1]) {
    const int32_t j = sj[0];
    const int32_t* __restrict__ sa = src[j].adj;
    const int32_t* __restrict__ sw = src[j].w;
    const int32_t shift = v_off[j] - src[j].abase;
    const int32_t eo = e_off[j];
#pragma unroll
    for (int r = 0; r < kPackPer; ++r) {
      const int64_t e = i0 + r * 256 + threadIdx.x;
      if (e < etot) {
        adj[e] = sa[e - eo] + shift;
        w[e] = sw[e - eo];
      }
    }
    return;
  }
  for (int r = 0; r < kPackPer; ++r) {
    const int64_t e = i0 + r * 256 + threadIdx.x;
    if (e >= etot) break;
    const int32_t j = job_in(e_off, sj[0], sj[1] + 1, e);
    const PackSrc& s = src[j];
    const int32_t le = int32_t(e - e_off[j]);
    adj[e] = v_off[j] + (s.adj[le] - s.abase);
    w[e] = s.w[le];
  }
}

int launch_pack(int32_t nj, const PackSrc* src, const int32_t* v_off, const int32_t* e_off, int32_t ntot, int32_t etot,
                int32_t* xadj, int32_t* adj, int32_t* w, int32_t* vw, const RefineStart* refine, hipStream_t st) {
  constexpr int kTile = kPackPer * 256;
  if (ntot <= 0) {
    fill<int32_t>(xadj, 0, 1, st);
    return hip_status();
  }
  if (refine)
    k_pack_refine<<<grid_for(ntot, kTile), 256, 0, st>>>(nj, src, v_off, e_off, ntot, etot, xadj, vw, *refine);
  else
    k_pack_vert<<<grid_for(ntot, kTile), 256, 0, st>>>(nj, src, v_off, e_off, ntot, etot, xadj, vw);
  if (etot > 0) k_pack_edge<<<grid_for(etot, kTile), 256, 0, st>>>(nj, src, v_off, e_off, etot, adj, w);
  return hip_status();
}

// Candidate bitmask from boundary flags and gains, one wave per word.
__global__ void __launch_bounds__(256) k_cand_init(int32_t n, const int32_t* __restrict__ bnd,
                                                   const int32_t* __restrict__ gain, uint64_t* __restrict__ cand) {
  const int64_t v = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const bool c = v < n && bnd[v] && gain[v] > 0;
  const uint64_t m = ballot(c);
  if (lane_id() == 0 && (v >> 6) <= (int64_t(n) - 1) / 64) cand[v >> 6] = m;
}

int launch_cand_init(int32_t n, const int32_t* bnd, const int32_t* gain, uint64_t* cand, hipStream_t st) {
  if (n > 0) k_cand_init<<<grid_for(n, 256), 256, 0, st>>>(n, bnd, gain, cand);
  return hip_status();
}

// Total vertex weight of every job (one block per job).
__global__ void __launch_bounds__(256) k_job_sum(const int32_t* __restrict__ v_off, const int32_t* __restrict__ vw,
                                                 long long* __restrict__ out) {
  __shared__ long long ws[4];
  const int32_t j = blockIdx.x;
  long long s = 0;
  for (int64_t i = v_off[j] + threadIdx.x; i < v_off[j + 1]; i += 256) s += vw[i];
  s = wave_sum64(s);
  if (lane_id() == 0) ws[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[j] = ws[0] + ws[1] + ws[2] + ws[3];
}

int launch_job_sum(int32_t nj, const int32_t* v_off, const int32_t* vw, long long* out, hipStream_t st) {
  if (nj > 0) k_job_sum<<<nj, 256, 0, st>>>(v_off, vw, out);
  return hip_status();
}

// ---------------------------------------------------------------- job offsets
// After clustering the pack: job j's coarse ids start at the coarse id of its
// first vertex in sorted order (jobs occupy consecutive sorted ranges because
// labels stay inside a job's id range).
__global__ void k_job_coff(int32_t nj, const int32_t* __restrict__ v_off, const int32_t* __restrict__ order,
                           const int32_t* __restrict__ cmap, int32_t nc, int32_t* __restrict__ c_off) {
  const int32_t j = blockIdx.x * 256 + threadIdx.x;
  if (j > nj) return;
  if (j == nj) { c_off[j] = nc; return; }
  c_off[j] = cmap[order[v_off[j]]];
}

__global__ void k_job_eoff(int32_t nj, const int32_t* __restrict__ c_off, const int32_t* __restrict__ cxadj,
                           int32_t* __restrict__ ce_off) {
  const int32_t j = blockIdx.x * 256 + threadIdx.x;
  if (j > nj) return;
  ce_off[j] = cxadj[c_off[j]];
}

int launch_job_offsets(int32_t nj, const int32_t* v_off, const int32_t* order, const int32_t* cmap, int32_t nc,
                       int32_t* c_off, hipStream_t st) {
  k_job_coff<<<grid_for(int64_t(nj) + 1, 256), 256, 0, st>>>(nj, v_off, order, cmap, nc, c_off);
  return hip_status();
}

int launch_job_eoffsets(int32_t nj, const int32_t* c_off, const int32_t* cxadj, int32_t* ce_off, hipStream_t st) {
  k_job_eoff<<<grid_for(int64_t(nj) + 1, 256), 256, 0, st>>>(nj, c_off, cxadj, ce_off);
  return hip_status();
}

// ---------------------------------------------------------------- unpack
// Refined partition of the pack -> per-job arrays.
__global__ void __launch_bounds__(256) k_unpack_part(int32_t nj, const UnpackDst* __restrict__ dst,
                                                     const int32_t* __restrict__ v_off, int32_t n,
                                                     const int32_t* __restrict__ part,
                                                     const int32_t* __restrict__ bnd) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const int32_t j = job_of(v_off, nj, i);
  const UnpackDst d = dst[j];
  const int32_t li = int32_t(i - v_off[j]);
  if (d.part) d.part[li] = part[i];
  if (d.bnd) d.bnd[li] = bnd[i];
}

int launch_unpack_part(int32_t nj, const UnpackDst* dst, const int32_t* v_off, int32_t n, const int32_t* part,
                       const int32_t* bnd, hipStream_t st) {
  if (n > 0) k_unpack_part<<<grid_for(n, 256), 256, 0, st>>>(nj, dst, v_off, n, part, bnd);
  return hip_status();
}

// ---------------------------------------------------------------- rounds
// Selection of a refinement round: create_independent_move_buffer
// (gkway/uncoarsen.hpp:111-173) with the cap and part weights of the vertex's
// job, over the candidate bitmask kept by the gain kernels (boundary vertices
// with positive gain), so vertices outside the mask cost one bit of a
// coalesced load.  k_select_list keeps the movable candidates (move fits the
// cap) with no smaller-id movable neighbour, as a bitmask; a scan turns
// the bitmask into a list ordered by vertex id, in which every job's selected
// vertices form one slice.  No kernel of the selection shares a counter
// between waves (same-address atomics serialise in L2).  vjob == null: one
// job.
// Candidate bitmask words read per wave by k_select_list, and
// per 256-thread block.
constexpr int kSelectWords = 8;
constexpr int kSelectBlockWords = 4 * kSelectWords;
// Rows longer than this are tested by the whole wave, 64 neighbours a step.
constexpr int32_t kSelectShortRow = 32;

// Position of the k-th (0-based) set bit of w (k < popcount(w)).
__device__ __forceinline__ int nth_set_bit(uint64_t w, int k) {
  int bit = 0;
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) {
    const int pc = popc64((w >> bit) & ((1ull << s) - 1));
    if (pc <= k) {
      k -= pc;
      bit += s;
    }
  }
  return bit;
}

// The wave's bit of rank r among the set bits of its kSelectWords words: lane
// l holds word l and the running count incl of words 0..l.  Every lane
// calls it (wave shuffles); the result is meaningful for r < the total.
__device__ __forceinline__ void deal_bit(int incl, uint64_t word, int r, int* wi_out, int* bit_out) {
  int wi = 0;
#pragma unroll
  for (int s = kSelectWords / 2; s >= 1; s >>= 1) {
    const int x = __shfl(incl, wi + s - 1, 64);
    if (x <= r) wi += s;
  }
  const int before = __shfl(incl, wi > 0 ? wi - 1 : 0, 64);
  const uint64_t wd = __shfl(word, wi < kSelectWords ? wi : 0, 64);
  *wi_out = wi;
  *bit_out = nth_set_bit(wd, r - (wi > 0 ? before : 0));
}

// Selection of a round: a candidate (boundary, positive gain) is movable when
// its move fits its job's cap, and a movable vertex is selected when no
// smaller-id neighbour is movable.  Each wave reads kSelectWords words of the
// candidate mask with one load and deals their set bits out to its lanes, 64
// per pass.  A neighbour's candidate bit is looked up first, and only for the
// few that are candidates whether their move fits, so no second launch over a
// finished movable mask is needed (that took 5 us and a gap of 2 a round on a
// mesh of 2 M vertices).  Only vertices with gain >= thr[job] are tested; the
// others get a bit in defbits, and the round kernel tests them, against the
// movable mask, only when fewer than M were selected (every key above the
// threshold beats every key below it).  A lane tests a row of up to
// kSelectShortRow entries itself; longer rows of a dealing pass are then tested
// one after another by the whole wave, 64 neighbours per step.  Results are
// bitmask words (movable, selbits, defbits), all written, so no counter is
// shared between waves.  Thread 0 also clears the worklist counters and the
// round's move counter, which only the round kernel adds to.
__global__ void __launch_bounds__(256) k_select_list(int32_t n, const int32_t* __restrict__ xadj,
                                                     const int32_t* __restrict__ adj,
                                                     const int32_t* __restrict__ vw,
                                                     const int32_t* __restrict__ vjob,
                                                     const int32_t* __restrict__ gain,
                                                     const int32_t* __restrict__ dest,
                                                     const int32_t* __restrict__ pw,
                                                     const int32_t* __restrict__ pw_off,
                                                     const long long* __restrict__ cap,
                                                     const int32_t* __restrict__ thr,
                                                     const uint64_t* __restrict__ cand,
                                                     uint64_t* __restrict__ movable, uint64_t* __restrict__ selbits,
                                                     uint64_t* __restrict__ defbits, int32_t* __restrict__ bsum,
                                                     int32_t* __restrict__ reset, int32_t* __restrict__ active,
                                                     unsigned long long* __restrict__ abytes) {
  __shared__ unsigned long long sw[4][3][kSelectWords];  // selected, deferred, movable
  __shared__ int32_t wsum[4];
  __shared__ long long wbytes[4];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    reset[0] = 0;
    reset[1] = 0;
    active[0] = 0;
  }
  const int lane = lane_id();
  const int wv = threadIdx.x >> 6;
  if (lane < kSelectWords) {
    sw[wv][0][lane] = 0;
    sw[wv][1][lane] = 0;
    sw[wv][2][lane] = 0;
  }
  __syncthreads();
  const int64_t nwords = (int64_t(n) + 63) >> 6;
  const int64_t w0 = ((int64_t(blockIdx.x) * 256 + threadIdx.x) >> 6) * kSelectWords;
  uint64_t word = 0;
  if (lane < kSelectWords && w0 + lane < nwords) word = cand[w0 + lane];
  const int incl = wave_incl_scan(popc64(word));
  const int total = __shfl(incl, kSelectWords - 1, 64);
  long long tested = 0;  // row entries of the tested vertices
  int fitting = 0;       // movable vertices
  for (int base = 0; base < total; base += 64) {
    const int r = base + lane;
    int wi, bit;
    deal_bit(incl, word, r, &wi, &bit);
    int32_t v = 0, s = 0, e = 0;
    int which = -1;  // 0 selected, 1 deferred
    bool long_row = false;
    const int32_t* pj = pw;  // part weights and cap of the vertex's job, and so of its neighbours'
    long long cj = 0;
    auto fits = [&](int32_t u) { return (long long)pj[dest[u]] + vw[u] <= cj; };
    if (r < total) {
      v = int32_t(((w0 + wi) << 6) + bit);
      const int32_t j = vjob ? vjob[v] : 0;
      pj = pw + pw_off[j];
      cj = cap[j];
      s = xadj[v];
      e = xadj[v + 1];
      if (fits(v)) {
        ++fitting;
        atomicOr(&sw[wv][2][wi], 1ull << bit);
        if (gain[v] < thr[j]) {
          which = 1;
        } else if (e - s > kSelectShortRow) {
          tested += e - s;
          long_row = true;
        } else {
          tested += e - s;
          // eight neighbours per step: their ids, their candidate bits, and
          // whether those that are candidates fit
          bool sel = true;
          for (int32_t x = s; x < e && sel; x += 8) {
            int32_t u[8];
            uint32_t c = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) u[i] = x + i < e ? adj[x + i] : v;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const uint64_t cw = cand[u[i] >> 6];
              if (u[i] < v && ((cw >> (u[i] & 63)) & 1ull)) c |= 1u << i;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i)
              if (((c >> i) & 1u) && sel && fits(u[i])) sel = false;
          }
          if (sel) which = 0;
        }
      }
    }
    // The pass's long rows, one at a time, by the whole wave.
    uint64_t lm = ballot(long_row);
    while (lm) {
      const int src = __ffsll(static_cast<long long>(lm)) - 1;
      lm &= lm - 1;
      const int32_t lv = __shfl(v, src, 64), ls = __shfl(s, src, 64), le = __shfl(e, src, 64);
      const int32_t lj = vjob ? vjob[lv] : 0;
      const int32_t* lp = pw + pw_off[lj];
      const long long lc = cap[lj];
      bool blocked = false;
      for (int32_t x0 = ls; x0 < le && !blocked; x0 += 64) {
        const int32_t x = x0 + lane;
        bool b = false;
        if (x < le) {
          const int32_t u = adj[x];
          b = u < lv && ((cand[u >> 6] >> (u & 63)) & 1ull) && (long long)lp[dest[u]] + vw[u] <= lc;
        }
        blocked = ballot(b) != 0;
      }
      if (lane == src && !blocked) which = 0;
    }
    if (which >= 0) atomicOr(&sw[wv][which][wi], 1ull << bit);
  }
  __syncthreads();
  int c = 0;
  if (lane < kSelectWords && w0 + lane < nwords) {
    selbits[w0 + lane] = sw[wv][0][lane];
    defbits[w0 + lane] = sw[wv][1][lane];
    movable[w0 + lane] = sw[wv][2][lane];
    c = popc64(sw[wv][0][lane]);
  }
  // selected vertices of the block's kSelectBlockWords words
  c = wave_sum(c);
  tested = wave_sum64(tested);
  fitting = wave_sum(fitting);
  if (lane == 0) {
    wsum[wv] = c;
    // per candidate its job, destination, part weight and vertex weight, per
    // movable vertex its row bounds, job and gain, per tested entry the
    // neighbour id and one movable bit
    wbytes[wv] = 16LL * total + 8LL * fitting + 4LL * tested + tested / 8;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    bsum[blockIdx.x] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    // and the block's candidate, movable, selected and deferred words
    if (abytes)
      atomicAdd(&abytes[blockIdx.x % kSelectByteSlots],
                (unsigned long long)(40LL * kSelectBlockWords + wbytes[0] + wbytes[1] + wbytes[2] + wbytes[3]));
  }
}

// Ordered list of the selected vertices: every word's first list slot
// (wpos) is the number of selected vertices before it.  Block b covers
// kScatterWords words; its offset is the sum of the selection blocks' counts
// (bsum) before its first word, then a block scan over its words.  One launch,
// no shared counter.  wpos[nwords] receives the total.
constexpr int kScatterWords = 2048;

__global__ void __launch_bounds__(256) k_sel_scatter(int64_t nwords, const uint64_t* __restrict__ selbits,
                                                     const int32_t* __restrict__ bsum, int32_t* __restrict__ wpos,
                                                     int32_t* __restrict__ list,
                                                     unsigned long long* __restrict__ abytes) {
  __shared__ int lds[8];
  const int64_t wb = int64_t(blockIdx.x) * kScatterWords;
  // offset: selection blocks [0, wb / kSelectBlockWords)
  const int64_t nb = wb / kSelectBlockWords;
  int off = 0;
  for (int64_t i = threadIdx.x; i < nb; i += 256) off += bsum[i];
  int tot;
  (void)block_excl_scan_256(off, &tot, lds);
  off = tot;
  constexpr int kPer = kScatterWords / 256;
  const int64_t w0 = wb + int64_t(threadIdx.x) * kPer;
  uint64_t b[kPer];
  int c = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    b[i] = w0 + i < nwords ? selbits[w0 + i] : 0;
    c += popc64(b[i]);
  }
  int r = off + block_excl_scan_256(c, &tot, lds);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    if (w0 + i < nwords) wpos[w0 + i] = r;
    uint64_t x = b[i];
    while (x) {
      const int bit = __ffsll(static_cast<long long>(x)) - 1;
      x &= x - 1;
      list[r++] = int32_t(((w0 + i) << 6) + bit);
    }
  }
  if (wb + kScatterWords >= nwords && threadIdx.x == 255) wpos[nwords] = r;
  // Algorithmic bytes: the block's selected words read and word positions
  // written, and one list slot per selected vertex (tot: the block's count).
  if (abytes && threadIdx.x == 0)
    atomicAdd(&abytes[blockIdx.x % kSelectByteSlots], (unsigned long long)(12LL * kScatterWords + 4LL * tot));
}

// List slot of vertex x (the number of selected vertices before it).
__device__ __forceinline__ int32_t sel_slot(const int32_t* __restrict__ wpos, const uint64_t* __restrict__ selbits,
                                            int64_t x) {
  const int64_t w = x >> 6;
  const int b = int(x & 63);
  return wpos[w] + (b ? popc64(selbits[w] & ((1ull << b) - 1)) : 0);
}

int select_scratch_ints(int64_t n) {
  const int64_t nwords = (n + 63) / 64;
  return static_cast<int>((nwords + kSelectBlockWords - 1) / kSelectBlockWords + 1);
}

int launch_select_list(const DGraph& g, const int32_t* vjob, const int32_t* gain, const int32_t* dest,
                       const int32_t* pw, const int32_t* pw_off, const long long* cap, const int32_t* thr,
                       const uint64_t* cand, const SelectBufs& sb, int32_t* reset, int32_t* active,
                       hipStream_t st) {
  if (g.n <= 0) return 0;
  const int64_t nwords = (int64_t(g.n) + 63) / 64;
  const int64_t waves = (nwords + kSelectWords - 1) / kSelectWords;
  const unsigned grid = grid_for(waves * 64, 256);
  gk_launch(k_select_list, dim3(grid), dim3(256), 0, st, g.n, g.xadj, g.adj, g.vw, vjob, gain, dest, pw, pw_off, cap,
            thr, cand, sb.movable, sb.selbits, sb.defbits, sb.scratch, reset, active, sb.abytes);
  gk_launch(k_sel_scatter, dim3(grid_for(nwords, kScatterWords)), dim3(256), 0, st, nwords, sb.selbits, sb.scratch,
            sb.wpos, sb.list, sb.abytes);
  return hip_status();
}

// One refinement round of one job per workgroup, after k_select_list:
//   1. the job's selected vertices: its slice of the selection list (plus,
//      when fewer than M and a gain threshold deferred some, those of the
//      deferred vertices that pass the test);
//   2. the min(count, M) best moves by (gain desc, id asc): all of them when
//      count <= M, else an exact radix select on a compressed key -- keys are
//      distinct, so exactly M are taken -- whose first digit also gives the
//      gain threshold of the job's next round;
//   3. LDS bitonic sort, balanced prefix (balance_prefix);
//   4. apply of the prefix: part, update flags and the gain worklist
//      (apply_sequence_move, gkway/uncoarsen.hpp:290-323).
// A job with nothing selected is left untouched, so extra rounds after the
// last productive one change nothing.
template <int kBigBits>
__global__ void __launch_bounds__(kBalThreads) k_round_b(
    const int32_t* __restrict__ v_off, int32_t M, int32_t kmax, const int32_t* __restrict__ kk,
    const long long* __restrict__ cap,
    const int32_t* __restrict__ pw_off, const int32_t* __restrict__ xadj, const int32_t* __restrict__ adj,
    int32_t* __restrict__ part, const int32_t* __restrict__ dest, const int32_t* __restrict__ gain,
    const int32_t* __restrict__ vw, int32_t* __restrict__ pw, long long* __restrict__ cut,
    int32_t* __restrict__ rounds, long long* __restrict__ moved, const SelectBufs sb, int32_t* __restrict__ xlist,
    uint32_t* __restrict__ hkey, int32_t* __restrict__ upd, int32_t* __restrict__ wl, int32_t* __restrict__ wlc,
    int32_t* __restrict__ lastcnt, int32_t* __restrict__ active, uint64_t* __restrict__ cand,
    int32_t* __restrict__ thr, long long* __restrict__ paths, int32_t* __restrict__ order,
    int32_t* __restrict__ hist, long long* __restrict__ abytes, int32_t* __restrict__ movers) {
  __shared__ RoundLds R;
  __shared__ int32_t big[1 << kBigBits];  // the apply's table for rounds of many moves
  if (kBigBits > 0)
    for (int i = threadIdx.x; i < (1 << kBigBits); i += kBalThreads) big[i] = -1;
  extern __shared__ int32_t dpw[];  // 2 * kmax ints: part weight changes, then the part weights
  int32_t* spw = dpw + kmax;
  const int t = threadIdx.x;
  const int32_t j = blockIdx.x;
  const int32_t vb = v_off[j], ve = v_off[j + 1];
  // Loads that the end of the round needs are issued now, off its critical
  // path: the job's first kBalThreads part weights (stored to LDS before the
  // balanced prefix) and its counters (thread 0).
  const int32_t kj = kk[j];
  const int32_t* pwj = pw + pw_off[j];
  const int32_t pw_t = t < kj ? pwj[t] : 0;
  R.ht[t] = -1;  // kBalThreads == table slots; the barriers before the apply order it
  long long cut0 = 0, moved0 = 0, ab0 = 0;
  int32_t rounds0 = 0;
  if (t == 0) {
    cut0 = cut[j];
    moved0 = moved[j];
    rounds0 = rounds[j];
    if (abytes) ab0 = abytes[j];
    R.misc[3] = sel_slot(sb.wpos, sb.selbits, vb);
    R.misc[1] = sel_slot(sb.wpos, sb.selbits, ve);
    R.misc[2] = lastcnt[j];
  }
  __syncthreads();
  const int32_t* seg = sb.list + R.misc[3];
  int32_t count = R.misc[1] - R.misc[3];
  const int32_t prev = R.misc[2];
  const bool deferred = count < M && thr[j] > 1;
  if (paths && deferred && t == 0) paths[3 * j + 2] += 1;
  if (deferred) {
    // The threshold left fewer than M selected: test the deferred (lower
    // gain) movable vertices of the job too, into the job's segment of xlist
    // after the selected ones, so that it holds every selected vertex.
    int32_t* xs = xlist + vb;
    for (int32_t i = t; i < count; i += kBalThreads) xs[i] = seg[i];
    if (t == 0) R.lz[0] = count;
    __syncthreads();
    for (int64_t w = (int64_t(vb) >> 6) + t; ve > vb && w <= ((int64_t(ve) - 1) >> 6); w += kBalThreads) {
      const int64_t lo = (vb > (w << 6) ? vb : (w << 6)) - (w << 6);
      const int64_t hi = (ve < (w << 6) + 64 ? ve : (w << 6) + 64) - (w << 6);
      uint64_t db = sb.defbits[w] & ((hi - lo == 64) ? ~0ull : (((1ull << (hi - lo)) - 1) << lo));
      while (db) {
        const int bit = __ffsll(static_cast<long long>(db)) - 1;
        db &= db - 1;
        const int32_t v = int32_t((w << 6) + bit);
        bool blocked = false;
        for (int32_t x = xadj[v]; x < xadj[v + 1] && !blocked; ++x) {
          const int32_t u = adj[x];
          blocked = u < v && ((sb.movable[u >> 6] >> (u & 63)) & 1ull);
        }
        if (!blocked) xs[atomicAdd(&R.lz[0], 1)] = v;
      }
    }
    __syncthreads();
    count = R.lz[0];
    seg = xs;
  }
  if (t == 0) {
    lastcnt[j] = count;
    if (count) atomicAdd(active, count);
    R.lz[2] = 1;  // next threshold: test everything unless set below
  }
  if (count == 0) {
    if (t == 0) thr[j] = 1;
    if (movers && t == 0) movers[0] = 0;
    // Nothing selected: the job's state (partition, gains, part weights) is
    // unchanged, so every later round of this level selects nothing either.
    // The first time, its candidate bits are dropped so that the selection
    // stops re-checking them (with one job the rounds end at the next check
    // anyway).
    if (prev != 0 && gridDim.x > 1) {
      const int64_t a = v_off[j], b = v_off[j + 1];
      for (int64_t w = (a >> 6) + t; b > a && w <= ((b - 1) >> 6); w += kBalThreads) {
        const int64_t lo = (a > (w << 6) ? a : (w << 6)) - (w << 6);
        const int64_t hi = (b < (w << 6) + 64 ? b : (w << 6) + 64) - (w << 6);
        const uint64_t m = (hi - lo == 64) ? ~0ull : (((1ull << (hi - lo)) - 1) << lo);
        if (m == ~0ull) cand[w] = 0;
        else atomicAnd(reinterpret_cast<unsigned long long*>(&cand[w]), (unsigned long long)~m);
      }
    }
    return;
  }
  const int32_t B = count < M ? count : M;
  // 2. and 3. the B best keys into R.b.sk, sorted; the balanced prefix
  const bool narrow = order_moves<8>(R, count, M, vb, ve, hkey + vb, SelectedList{seg, gain});
  if (t < kj) spw[t] = pw_t;
  for (int32_t q = t + kBalThreads; q < kj; q += kBalThreads) spw[q] = pwj[q];
  BalanceOpt bo;
  bo.spw = spw;
  bo.mdst = R.mdst;
  bo.gain_in_key = true;
  bo.cut_given = true;
  bo.cut_now = cut0;
  const int pos = balance_prefix(R.b, dpw, kj, B, 0xffffffffull, part, dest, gain, vw, pw + pw_off[j], cap[j],
                                 nullptr, nullptr, &cut[j], bo);
  // Optional trace of the round: which ordering path ran (top-M radix
  // select; compressed keys wider than 32 bits) and the ordered moves with B
  // and pos.  R.b.sv keeps the ordered vertices through the apply below.
  if (paths && t == 0 && count > M) {
    paths[3 * j] += 1;
    if (!narrow) paths[3 * j + 1] += 1;
  }
  if (order) {
    int32_t* o = order + int64_t(j) * (M + 2);
    if (t < B) o[2 + t] = R.b.sv[t];
    if (t == 0) {
      o[0] = B;
      o[1] = pos;
    }
  }
  if (hist && t == 0) {
    hist[2 * rounds0] = B;
    hist[2 * rounds0 + 1] = pos;
  }
  // 4. the apply
  const bool sole = gridDim.x == 1;
  int32_t wrun = 0;
  if (movers && t == 0) movers[0] = pos < 64 ? 0 : pos + 1;
  if (movers && pos >= 64) {
    // More than a wave's worth, and one job: the whole device expands them
    // (k_expand_moves).
    if (t <= pos) {
      const int32_t v = R.b.sv[t];
      part[v] = R.mdst[t];
      movers[1 + t] = v;
    }
    if (t == 0) {
      thr[j] = R.lz[2];
      rounds[j] = rounds0 + 1;
      moved[j] = moved0 + pos + 1;
      if (abytes) abytes[j] = ab0 + 8LL * count + 16LL * B + 4LL * kj;
    }
    return;
  }
  const int tot = apply_moves(R, pos, part, xadj, adj, upd, wl, wlc, sole, &wrun, big, kBigBits);
  if (t == 0) {
    if (sole) wlc[0] = wrun;
    thr[j] = R.lz[2];
    rounds[j] = rounds0 + 1;
    moved[j] = moved0 + pos + 1;
    // Algorithmic bytes of the round: each selected vertex's id and gain,
    // each ordered move's weight, gain, part and destination, the job's part
    // weights, and per applied item (a mover or a neighbour) its id, update
    // flag and worklist slot.
    if (abytes) abytes[j] = ab0 + 8LL * count + 16LL * B + 4LL * kj + 12LL * tot;
  }
}

// The movers of a round that moved 64 or more (movers[0] of them, else 0;
// their parts are set): they and their neighbours, items dealt out over the
// device, each once onto the gain worklist.  The round's own workgroup took 19
// to 25 us for the 7100 items of 1024 movers, bound by the scattered accesses
// of one compute unit.  Every block adds up the movers' rows for itself.
__global__ void __launch_bounds__(256) k_expand_moves(const int32_t* __restrict__ movers,
                                                      const int32_t* __restrict__ xadj,
                                                      const int32_t* __restrict__ adj, int32_t* __restrict__ upd,
                                                      int32_t* __restrict__ wl, int32_t* __restrict__ wlc,
                                                      long long* __restrict__ abytes) {
  __shared__ int32_t mv[kBalMax], rstart[kBalMax], istart[kBalMax];
  __shared__ int lds[8];
  constexpr int kPer = kBalMax / 256;
  const int32_t cnt = movers[0];
  if (cnt == 0) return;
  const int t = threadIdx.x;
  int32_t v[kPer], s[kPer], c[kPer];
  int sum = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int m = t * kPer + i;
    v[i] = m < cnt ? movers[1 + m] : -1;
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    s[i] = v[i] >= 0 ? xadj[v[i]] : 0;
    c[i] = v[i] >= 0 ? xadj[v[i] + 1] - s[i] + 1 : 0;
    sum += c[i];
  }
  int tot;
  int run = block_excl_scan_256(sum, &tot, lds);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int m = t * kPer + i;
    mv[m] = v[i];
    rstart[m] = s[i];
    istart[m] = run;
    run += c[i];
  }
  __syncthreads();
  if (abytes && blockIdx.x == 0 && t == 0) atomicAdd(reinterpret_cast<unsigned long long*>(abytes), 12ull * tot);
  const int64_t step = int64_t(gridDim.x) * 256;
  // whole waves stay together
  for (int64_t b = int64_t(blockIdx.x) * 256 + (t & ~63); b < tot; b += step) {
    const int64_t x = b + lane_id();
    bool first = false;
    int32_t u = 0;
    if (x < tot) {
      int lo = 0, hi = cnt - 1;  // last mover m with istart[m] <= x
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (istart[mid] <= x) lo = mid; else hi = mid - 1;
      }
      const int off = int(x) - istart[lo];
      u = off == 0 ? mv[lo] : adj[rstart[lo] + off - 1];
      first = atomicExch(&upd[u], 1) == 0;
    }
    const uint64_t m = ballot(first);
    int base = 0;
    if (lane_id() == 0 && m) base = atomicAdd(wlc, popc64(m));
    base = __shfl(base, 0, 64);
    if (first) wl[base + popc64(m & lanemask_lt())] = u;
  }
}

int launch_round_b(int32_t nj, int32_t kmax, const int32_t* v_off, int32_t M, const int32_t* kk, const long long* cap,
                   const int32_t* pw_off, const DGraph& g, int32_t* part, const int32_t* dest, const int32_t* gain,
                   int32_t* pw, long long* cut, int32_t* rounds, long long* moved, const SelectBufs& sb,
                   int32_t* xlist, uint32_t* hkey, int32_t* upd, int32_t* wl, int32_t* wlc, int32_t* lastcnt,
                   int32_t* active, uint64_t* cand, int32_t* thr, long long* paths, int32_t* order, int32_t* hist,
                   long long* abytes, int32_t* movers, hipStream_t st) {
  if (nj <= 0) return 0;
  if (M > kBalMax) return GK_ERR_LIMIT;
  if (nj != 1) movers = nullptr;
  // 64 KB of LDS for the apply's table, unless the device expands the moves,
  // the jobs need to share a compute unit, or the part weights (8 kmax bytes)
  // take the room.
  if (!movers && nj <= 256 && kmax <= 4096)
    gk_launch(k_round_b<14>, dim3(nj), dim3(kBalThreads), uint32_t(2 * sizeof(int32_t) * kmax), st, v_off, M, kmax, kk, cap,
              pw_off,
              g.xadj, g.adj, part, dest, gain, g.vw, pw, cut, rounds, moved, sb, xlist, hkey, upd, wl, wlc, lastcnt,
              active, cand, thr, paths, order, hist, abytes, movers);
  else
    gk_launch(k_round_b<0>, dim3(nj), dim3(kBalThreads), uint32_t(2 * sizeof(int32_t) * kmax), st, v_off, M, kmax, kk, cap,
              pw_off,
              g.xadj, g.adj, part, dest, gain, g.vw, pw, cut, rounds, moved, sb, xlist, hkey, upd, wl, wlc, lastcnt,
              active, cand, thr, paths, order, hist, abytes, movers);
  if (movers)
    gk_launch(k_expand_moves, dim3(64), dim3(256), 0, st, movers, g.xadj, g.adj, upd, wl, wlc, abytes);
  return hip_status();
}

// Largest row length of a graph (atomicMax per wave into *out, zeroed here).
// Grid-stride; one atomic per block.
__global__ void __launch_bounds__(256) k_max_deg(int32_t n, const int32_t* __restrict__ xadj, int32_t* __restrict__ out) {
  __shared__ int wm[4];
  int d = 0;
  for (int64_t v = int64_t(blockIdx.x) * 256 + threadIdx.x; v < n; v += int64_t(gridDim.x) * 256) {
    const int x = xadj[v + 1] - xadj[v];
    d = x > d ? x : d;
  }
  d = wave_max(d);
  if (lane_id() == 0) wm[threadIdx.x >> 6] = d;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int m = max(max(wm[0], wm[1]), max(wm[2], wm[3]));
    if (m > 0) atomicMax(out, m);
  }
}

int launch_max_deg(const DGraph& g, int32_t* out, hipStream_t st) {
  fill<int32_t>(out, 0, 1, st);
  unsigned grid = grid_for(g.n, 256);
  if (grid > 1024) grid = 1024;
  if (g.n > 0) k_max_deg<<<grid, 256, 0, st>>>(g.n, g.xadj, out);
  return hip_status();
}

// Final cut and part weights (calculate_cutsize + calculate_partition_wgt,
// gkway/uncoarsen.hpp:398-424, gkway/cuda_check.hpp:61-73) per chunk of one
// job's vertices: the block sums its vertex weights per part in an LDS
// histogram and its cut edges in registers (8 lanes a vertex), then adds them
// to the job's totals with one atomic per touched part and one for the cut.
// The finished partition goes to its job's destination on the way.  Few jobs
// end in one step, so a chunk is short: with 2048 vertices of a chunk and one
// lane a vertex a launch took 67 us, nearly all of it one block's chain.
__global__ void __launch_bounds__(256) k_cut_chunks(const int32_t* __restrict__ cj, const int32_t* __restrict__ cs,
                                                    const int32_t* __restrict__ ce, const int32_t* __restrict__ kk,
                                                    const int32_t* __restrict__ v_off,
                                                    const int32_t* __restrict__ xadj,
                                                    const int32_t* __restrict__ adj, const int32_t* __restrict__ w,
                                                    const int32_t* __restrict__ vw,
                                                    const int32_t* __restrict__ part,
                                                    const int32_t* __restrict__ pw_off,
                                                    const UnpackDst* __restrict__ dst,
                                                    unsigned long long* __restrict__ cut,
                                                    unsigned long long* __restrict__ pw64) {
  extern __shared__ unsigned int hist[];
  __shared__ long long wsum[4];
  const int32_t c = static_cast<int32_t>(xcd_block());
  const int32_t j = cj[c], k = kk[j], e0 = ce[c];
  int32_t* out = dst[j].part - v_off[j];
  for (int32_t q = threadIdx.x; q < k; q += 256) hist[q] = 0;
  __syncthreads();
  long long cc = 0;
  const int sub = threadIdx.x & 7;
  for (int32_t v = cs[c] + int32_t(threadIdx.x >> 3); v < e0; v += 32) {
    const int32_t p = part[v];
    for (int32_t e = xadj[v] + sub; e < xadj[v + 1]; e += 8) {
      const int32_t u = adj[e];
      if (v < u && part[u] != p) cc += w[e];
    }
    if (sub == 0) {
      atomicAdd(&hist[p], (unsigned int)vw[v]);
      out[v] = p;
    }
  }
  cc = wave_sum64(cc);
  if (lane_id() == 0) wsum[threadIdx.x >> 6] = cc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const long long s = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    if (s) atomicAdd(&cut[j], (unsigned long long)s);
  }
  for (int32_t q = threadIdx.x; q < k; q += 256)
    if (hist[q]) atomicAdd(&pw64[pw_off[j] + q], (unsigned long long)hist[q]);
}

int launch_cut_chunks(int32_t nchunks, const int32_t* cj, const int32_t* cs, const int32_t* ce, int32_t kmax,
                      const int32_t* kk, const int32_t* v_off, const DGraph& g, const int32_t* part,
                      const int32_t* pw_off, const UnpackDst* dst, unsigned long long* cut, unsigned long long* pw64,
                      hipStream_t st) {
  if (nchunks <= 0) return 0;
  k_cut_chunks<<<nchunks, 256, sizeof(unsigned int) * kmax, st>>>(cj, cs, ce, kk, v_off, g.xadj, g.adj, g.w, g.vw,
                                                                  part, pw_off, dst, cut, pw64);
  return hip_status();
}

}  // namespace gkd
