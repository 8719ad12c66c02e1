// Host driver of the MI355X partitioner: context, device memory pool, the
// multilevel V-cycle, and the C ABI entry points that launch device work.
//
// Flow of one gk_partition_device call (the reference's graph_partitioner,
// gkway/graph_partitioner.hpp:222-365):
//   coarsening levels  -> match, grouping by a walk to the root pairs (deep
//                         trees: pointer jumping), order, chunks and coarse ids
//                         by counting (large groups: a radix sort by (label,
//                         stamp, id)), contraction
//   coarsest level     -> copy to host, gk_initpart (METIS's role), copy back
//   uncoarsening       -> per finer level: projection and gain pass, then rounds
//                         by the round loop or by separate kernels (select,
//                         order and balance, apply, gain) until no move
//   final              -> weighted cut and part weights of level 0
// One stream per context.  The host waits for the counts that size a coarsening
// level's next launches (two or three of them), for the coarsest graph, and in
// refinement at the end of a launch of the round loop (up to 64 rounds) or every
// 4 to 32 rounds of the separate kernels; kernels tell it most counts in words
// it watches.
#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "../../include/gkway.h"
#include "host_graph.hpp"
#include "batch.hpp"
#include "kernels.hpp"
#include "prim.hpp"
#include "round_plan.hpp"
#include "runtime.hpp"


using gkd::DGraph;

using namespace gkrt;

namespace gkd {
bool kernel_events(hipEvent_t* start, hipEvent_t* stop) { return gkrt::StageClock::kernel_pair(start, stop); }
}  // namespace gkd

namespace gkrt {

// Smallest launches worth timing candidates for: matching over at least
// 1 Mi entries, a contraction row class of at least 16 Ki rows.
constexpr int64_t kTuneMinEntries = int64_t(1) << 20;
constexpr int32_t kTuneMinRows = 1 << 14;

int wait_words(gk_ctx* ctx, hipStream_t st, const gkd::HostWords& h, int n, int32_t* out) {
  bool ended = false;  // the stream has run out
  for (int i = 0, spins = 0; i < n;) {
    const unsigned long long w = __atomic_load_n(&ctx->hctl[i], __ATOMIC_ACQUIRE);
    if (uint32_t(w >> 32) == h.number) {
      out[i++] = int32_t(uint32_t(w));
      continue;
    }
    if (ended) {
      gkh::set_error("a kernel did not report to the host");
      return GK_ERR_INTERNAL;
    }
    __builtin_ia32_pause();
    if (++spins % 4096) continue;
    const hipError_t e = hipStreamQuery(st);
    if (e == hipSuccess) {
      ended = true;
    } else if (e == hipErrorNotReady) {
      (void)hipGetLastError();  // no error, but remembered as one
    } else {
      gkh::set_error(std::string("waiting for a kernel: ") + hipGetErrorString(e));
      return GK_ERR_HIP;
    }
  }
  return GK_OK;
}

// ---------------------------------------------------------------- stages
// Labels, hops (to dist_out, or dist) and member counts of the groups by
// walking to the root pairs.
// The control words hold whether every vertex reached its pair.
int Groups::walk(gk_ctx* ctx, hipStream_t st, int32_t n, const int32_t* cand, int32_t* label, int32_t* dist_out) {
  Pool& P = ctx->pool;
  GK_TRY(ctl.alloc(P, gkd::kCtlInts + gkd::kRowCtlInts));
  GK_TRY(comp.alloc(P, int64_t(n) + 1));
  if (!dist_out) GK_TRY(dist.alloc(P, n));
  GK_TRY(slot.alloc(P, n));
  GK_TRY(size.alloc(P, n));
  GK_STAGE(ctx, GK_ST_GROUP, 52LL * n,
           (gkd::launch_walk(n, cand, comp.p, label, dist_out ? dist_out : dist.p, slot.p, ctl.p, st) ||
                    gkd::launch_label_size(n, label, comp.p, label, size.p, st)
                ? GK_ERR_HIP
                : GK_OK));
  return GK_OK;
}

// Jumping rounds that the walk's flags (words kCtlFlags.. of the control
// words) stand for: every round halves the largest distance.
int32_t Groups::rounds(const int32_t* words) {
  int32_t r = 0;
  for (int b = 0; b <= gkd::kWalkBits; ++b)
    if (words[gkd::kCtlFlags + b]) r = b + 1;
  return r;
}

// The same by pointer jumping, for trees deeper than the walk goes; returns
// the jump rounds in *rounds.
int Groups::jump(gk_ctx* ctx, hipStream_t st, int32_t n, const int32_t* cand, int32_t* label, int32_t* rounds) {
  Pool& P = ctx->pool;
  Buf<int32_t> nx[2], ds[2], flags;
  GK_TRY(nx[0].alloc(P, n));
  GK_TRY(nx[1].alloc(P, n));
  GK_TRY(ds[0].alloc(P, n));
  GK_TRY(ds[1].alloc(P, n));
  GK_TRY(flags.alloc(P, kMaxJumpRounds + 8));
  gkd::fill<int32_t>(flags.p, 0, kMaxJumpRounds + 8, st);
  gkd::fill<int32_t>(ctl.p, 0, gkd::kCtlInts, st);
  GK_STAGE(ctx, GK_ST_GROUP, 16LL * n, gkd::launch_jump_init(n, cand, nx[0].p, ds[0].p, st));
  int32_t f = -1;
  int32_t r = 0;
  constexpr int kBatch = 4;
  while (f < 0) {
    if (r >= kMaxJumpRounds) {
      gkh::set_error("candidate graph did not reduce to pairs (asymmetric input?)");
      return GK_ERR_GRAPH;
    }
    ctx->clock.begin(GK_ST_GROUP);
    for (int i = 0; i < kBatch && r + i < kMaxJumpRounds; ++i) {
      const int rr = r + i;
      GK_TRY(gkd::launch_jump_round(n, cand, nx[rr & 1].p, ds[rr & 1].p, nx[(rr + 1) & 1].p,
                                    ds[(rr + 1) & 1].p, flags.p, rr, st));
    }
    ctx->clock.end(GK_ST_GROUP);
    int32_t hf[kBatch];
    const int cnt = std::min(kBatch, kMaxJumpRounds - r);
    GK_TRY(fetch(ctx, st, {{hf, flags.p + r, sizeof(int32_t) * cnt}}));
    for (int i = 0; i < cnt; ++i)
      if (hf[i] == 0) { f = r + i; break; }
    r += cnt;
  }
  // Round f moved nothing: buffers f&1 and (f+1)&1 agree.
  // Rounds 0..f ran in full (24 bytes per vertex each); later ones exit early.
  count_stage(ctx, GK_ST_GROUP, 24LL * n * (f + 1));
  GK_STAGE(ctx, GK_ST_GROUP, 40LL * n,
           (gkd::launch_comp_count(n, cand, nx[f & 1].p, comp.p, label, slot.p, st) ||
                    gkd::launch_label_size(n, label, comp.p, label, size.p, st)
                ? GK_ERR_HIP
                : GK_OK));
  dist = std::move(ds[f & 1]);
  *rounds = f;
  return GK_OK;
}

// Labels that come without a grouping: member counts only.  The control word
// kCtlFlags tells of labels outside [0, n).
int Groups::count(gk_ctx* ctx, hipStream_t st, int32_t n, const int32_t* label) {
  Pool& P = ctx->pool;
  GK_TRY(ctl.alloc(P, gkd::kCtlInts + gkd::kRowCtlInts));
  GK_TRY(comp.alloc(P, int64_t(n) + 1));
  GK_TRY(slot.alloc(P, n));
  GK_TRY(size.alloc(P, n));
  GK_STAGE(ctx, GK_ST_SORT, 16LL * n, gkd::launch_label_count(n, label, size.p, slot.p, ctl.p, st));
  return GK_OK;
}

// Order, coarse ids and member records by counting, from the groups' sizes
// and slots.  The control words (kCtlInts) are told the host; [1] != 0: some
// group is too large, the results are incomplete and sort_members is needed.
// So it is with *no_room: the pool had none for the members' records (32 bytes
// a vertex beside the counts; the sort's arrays come after the counts are
// given back), and nothing but the control words is written.
static int count_members(gk_ctx* ctx, hipStream_t st, int32_t n, const int32_t* label, const int32_t* stamp,
                         Groups& gr, const int32_t* xadj, const int32_t* vw, int32_t G, const MemberOut& out,
                         gkd::HostWords* told_out, bool* no_room) {
  Buf<int2> partial;
  Buf<int4> memb;
  const gkd::HostWords told = host_words(ctx);
  GK_TRY(partial.alloc(ctx->pool, gkd::size_partials(n)));
  *no_room = memb.alloc(ctx->pool, 2 * int64_t(n)) != GK_OK;
  GK_STAGE(ctx, GK_ST_SORT, 16LL * n,
           gkd::launch_size_scan(n, gr.size.p, G, partial.p, gr.comp.p, gr.ctl.p, told, st));
  *told_out = told;
  if (*no_room) return GK_OK;
  // The counts come back while the members are ordered.
  GK_STAGE(ctx, GK_ST_SORT, 120LL * n,
           gkd::launch_members(n, label, stamp, gr.slot.p, gr.comp.p, xadj, vw, memb.p, G, gr.ctl.p, out.order,
                               out.cmap, out.cptr, out.mrow, out.mvw, st));
  return GK_OK;
}

// The same by a radix sort of (label, stamp), stamps below 2^sbits.  The rows
// and weights (out.mrow and out.mvw are not used) are allocated when the keys
// have been given back: 12 bytes a vertex less at the peak.
static int sort_members(gk_ctx* ctx, hipStream_t st, int32_t n, const int32_t* label, const int32_t* stamp, int sbits,
                        const int32_t* xadj, const int32_t* vw, int32_t G, const MemberOut& out, Buf<int2>* mrow,
                        Buf<int32_t>* mvw, int32_t* nc) {
  Pool& P = ctx->pool;
  const int lbits = bits_for(n > 0 ? n - 1 : 0);
  Buf<uint64_t> keys, keys2;
  Buf<int32_t> ids, ids2, scratch, gstart, flagscan, ncd, zero, cm;
  if (!stamp) {
    GK_TRY(zero.alloc(P, n));
    gkd::fill<int32_t>(zero.p, 0, n, st);
    stamp = zero.p;
  }
  if (mrow) mrow->release();
  mvw->release();
  int32_t* cmap = out.cmap;
  if (!cmap) {
    GK_TRY(cm.alloc(P, n));
    cmap = cm.p;
  }
  GK_TRY(keys.alloc(P, n));
  GK_TRY(keys2.alloc(P, n));
  GK_TRY(ids.alloc(P, n));
  GK_TRY(ids2.alloc(P, n));
  GK_TRY(scratch.alloc(P, gkd::sort_scratch_ints(n) + gkd::scan_scratch_ints(n)));
  GK_TRY(gstart.alloc(P, n));
  GK_TRY(flagscan.alloc(P, n));
  GK_TRY(ncd.alloc(P, 1));
  bool alt = false;
  const int passes = (sbits + lbits + 7) / 8;
  GK_STAGE(ctx, GK_ST_SORT, 20LL * n + 32LL * n * passes,
           (gkd::launch_make_keys(n, label, stamp, sbits, keys.p, ids.p, st) ||
                    gkd::radix_sort_pairs<uint64_t>(keys.p, ids.p, keys2.p, ids2.p, n, 0, sbits + lbits, scratch.p, st, &alt)
                ? GK_ERR_HIP
                : GK_OK));
  const int32_t* sid = alt ? ids2.p : ids.p;
  auto rows = [&]() -> int {
    keys.release();
    keys2.release();
    gstart.release();
    flagscan.release();
    if (mrow) GK_TRY(mrow->alloc(P, n));
    GK_TRY(mvw->alloc(P, n));
    return gkd::launch_member_rows(n, sid, xadj, vw, mrow ? mrow->p : nullptr, mvw->p, st);
  };
  ctx->clock.begin(GK_ST_CLUSTER);
  int rc = gkd::launch_cluster(n, alt ? keys2.p : keys.p, sid, sbits, G, gstart.p, flagscan.p, cmap, out.cptr, ncd.p,
                               scratch.p, st);
  if (!rc) rc = rows();
  ctx->clock.end(GK_ST_CLUSTER);
  if (rc) return rc;
  count_stage(ctx, GK_ST_CLUSTER, 80LL * n);
  if (out.order)
    GK_HIP(hipMemcpyAsync(out.order, sid, sizeof(int32_t) * size_t(n), hipMemcpyDeviceToDevice, st));
  GK_TRY(fetch(ctx, st, {{nc, ncd.p, sizeof(int32_t)}}));
  return GK_OK;
}

// Coarse ids of the vertices from their candidates: groups, their members in
// (label, stamp, id) order, chunks of at most G.
int coarse_ids(gk_ctx* ctx, hipStream_t st, const DGraph& g, const int32_t* cand, int32_t G, bool want_order,
               int32_t* cmap, Members& m, int32_t* nc, int32_t* rounds) {
  Pool& P = ctx->pool;
  const int32_t n = g.n;
  Buf<int32_t> label;
  Groups gr;
  if (want_order) GK_TRY(m.order.alloc(P, n));
  GK_TRY(m.cptr.alloc(P, int64_t(n) + 1));
  GK_TRY(m.mrow.alloc(P, n));
  GK_TRY(m.mvw.alloc(P, n));
  int32_t words[gkd::kCtlInts];
  // Small graphs in one launch, unless a tree is too deep or a group too large.
  if (n > 0 && n <= gkd::kSmallGroup) {
    GK_TRY(m.ctl.alloc(P, gkd::kCtlInts + gkd::kRowCtlInts));
    const gkd::HostWords told = host_words(ctx);
    GK_STAGE(ctx, GK_ST_GROUP, 40LL * n,
             gkd::launch_group_small(n, cand, G, g.xadj, g.vw, m.order.p, cmap, m.cptr.p, m.mrow.p, m.mvw.p, m.ctl.p,
                                     told, st));
    GK_TRY(wait_words(ctx, st, told, gkd::kCtlInts, words));
    *rounds = Groups::rounds(words);
    *nc = words[0];
    if (!words[1] && !words[gkd::kCtlFlags + gkd::kWalkBits]) return GK_OK;
  }
  GK_TRY(label.alloc(P, n));
  const MemberOut out{m.order.p, cmap, m.cptr.p, m.mrow.p, m.mvw.p};
  gkd::HostWords told;
  bool no_room = false;
  GK_TRY(gr.walk(ctx, st, n, cand, label.p));
  GK_TRY(count_members(ctx, st, n, label.p, gr.dist.p, gr, g.xadj, g.vw, G, out, &told, &no_room));
  GK_TRY(wait_words(ctx, st, told, gkd::kCtlInts, words));
  *rounds = Groups::rounds(words);
  if (words[gkd::kCtlFlags + gkd::kWalkBits]) {
    GK_TRY(gr.jump(ctx, st, n, cand, label.p, rounds));
    GK_TRY(count_members(ctx, st, n, label.p, gr.dist.p, gr, g.xadj, g.vw, G, out, &told, &no_room));
    GK_TRY(wait_words(ctx, st, told, gkd::kCtlInts, words));
  }
  *nc = words[0];
  // Distances are at most 2^rounds.
  if (words[1] || no_room) {
    gr.counts_done();
    GK_TRY(sort_members(ctx, st, n, label.p, gr.dist.p, *rounds + 1, g.xadj, g.vw, G, out, &m.mrow, &m.mvw, nc));
  }
  m.ctl = std::move(gr.ctl);
  return GK_OK;
}

// Contraction of g under cmap, with its members by coarse id (m: first places,
// rows, and, unless null, weights), into the coarse level c; with weights also
// the coarse weights into c.vw (allocated by the caller).  With out the coarse
// CSR goes to its arrays, written after everything else has been read.
int contract_stage(gk_ctx* ctx, hipStream_t st, const DGraph& g, int32_t nc, const int32_t* cmap, const Members& m,
                   Level& c, const CsrOut* out) {
  Pool& P = ctx->pool;
  Buf<int32_t> toff, lists, scratch, tadj, tw, len;
  Buf<int2> desc;
  const int32_t* cnt = m.ctl.p + gkd::kCtlInts;
  GK_TRY(toff.alloc(P, nc));
  GK_TRY(lists.alloc(P, int64_t(gkd::kRowClasses) * nc));
  GK_TRY(desc.alloc(P, int64_t(gkd::kRowClasses) * nc));
  GK_TRY(tadj.alloc(P, g.nnz));
  GK_TRY(tw.alloc(P, g.nnz));
  GK_TRY(len.alloc(P, nc));
  GK_TRY(scratch.alloc(P, gkd::size_partials(nc)));
  GK_TRY(c.xadj.alloc(P, int64_t(nc) + 1));
  GK_STAGE(ctx, GK_ST_CONTRACT_AUX, (m.mvw.p ? 12LL : 8LL) * g.n + 28LL * nc,
           gkd::launch_contract_bounds(nc, m.cptr.p, m.mrow.p, m.mvw.p, toff.p, lists.p, desc.p, len.p,
                                       c.vw.p, m.ctl.p + gkd::kCtlInts, st));
  // GK_CONTRACT_WIDE=1 runs the row kernels that sort (id, weight) pairs,
  // which otherwise serve only coarse graphs of 2^26 - 1 vertices or more.
  const char* wide_env = std::getenv("GK_CONTRACT_WIDE");
  const bool wide = wide_env && wide_env[0] == '1';
  int32_t words[1 + gkd::kRowCtlWords];  // entries, then the class counters
  const int32_t* hc = words + 1;
  if (nc <= gkd::kRowsAllMax && !wide && !ctx->autotune && !steal_of(ctx)) {
    GK_STAGE(ctx, GK_ST_CONTRACT, 0,
             gkd::launch_contract_rows_all(g, nc, cnt, lists.p, desc.p, m.mrow.p, cmap, toff.p, tadj.p, tw.p, len.p,
                                           st));
    GK_STAGE(ctx, GK_ST_CONTRACT_BIG, 0,
             gkd::launch_contract_mid(g, nc, nc, cnt, lists.p, desc.p, m.mrow.p, cmap, toff.p, tadj.p, tw.p, len.p,
                                      st));
  } else {
    std::vector<int32_t> h(gkd::kRowCtlInts);
    GK_TRY(fetch(ctx, st, {{h.data(), cnt, sizeof(int32_t) * gkd::kRowCtlInts}}));
    for (int i = 0; i < gkd::kRowCtlWords; ++i) words[1 + i] = h[i * gkd::kRowCtlStride];
    const int lanes[3] = {16, 32, 64};
    auto row_classes = [&]() -> int {
      for (int cls = 0; cls < 3; ++cls) {
        const int32_t* rows = lists.p + int64_t(cls) * nc;
        auto run = [&](const Tuner::Shape& x) {
          return gkd::launch_contract_rows(g, x.lanes, x.block, rows, desc.p + int64_t(cls) * nc, hc[cls], nc,
                                           m.mrow.p, cmap, toff.p, tadj.p, tw.p, len.p, wide, st, steal_of(ctx));
        };
        Tuner::Shape shape{lanes[cls], 256};
        if (ctx->autotune && hc[cls] >= kTuneMinRows) {
          // Block size per row class; the lanes of a class are fixed by its rows.
          const uint64_t key = Tuner::key(1 + cls, g.n, g.nnz);
          if (const Tuner::Shape* s = ctx->tuner.find(key)) {
            shape = *s;
          } else {
            const int L = lanes[cls];
            GK_TRY(ctx->tuner.tune(key, {{L, 256}, {L, 64}, {L, 128}, {L, 512}}, st, run, &shape));
            continue;  // every candidate wrote the rows
          }
        }
        GK_TRY(run(shape));
      }
      return GK_OK;
    };
    ctx->clock.begin(GK_ST_CONTRACT);
    const int rc_rows = row_classes();
    ctx->clock.end(GK_ST_CONTRACT);
    if (rc_rows != GK_OK) return rc_rows;
    count_stage(ctx, GK_ST_CONTRACT, 0);  // bytes added once the coarse entry count is known
    if (hc[3] > 0)
      GK_STAGE(ctx, GK_ST_CONTRACT_BIG, 0,
               gkd::launch_contract_mid(g, nc, hc[3], cnt, lists.p, desc.p, m.mrow.p, cmap, toff.p, tadj.p, tw.p,
                                        len.p, st));
  }
  // The entry count comes back with the class counters; rows for the global
  // sort, if there are any, are merged then, and the lengths scanned again.
  // Graphs of up to kEarlyEntries get arrays as large as their own, so that the
  // rows are copied while the host still waits for their number.  (A caller's
  // arrays need not be so large.)  They stay as large as that (levels of 8 MB at
  // most): under a pool limit, without room, or with rows for the global sort,
  // which needs the room, the rows are copied once it is known.
  constexpr int32_t kEarlyEntries = 1 << 20;
  bool early = !out && !P.limited() && g.nnz <= kEarlyEntries && c.adj.alloc(P, g.nnz) == GK_OK &&
               c.w.alloc(P, g.nnz) == GK_OK;
  auto not_early = [&]() {
    early = false;
    c.adj.release();
    c.w.release();
  };
  if (!early) not_early();
  auto copy_rows = [&](int32_t room) -> int {
    if (!out && !early) {
      GK_TRY(c.adj.alloc(P, room));
      GK_TRY(c.w.alloc(P, room));
    }
    return gkd::launch_contract_copy(nc, toff.p, len.p, c.xadj.p, tadj.p, tw.p, out ? out->adj : c.adj.p,
                                     out ? out->w : c.w.p, out ? out->xadj : nullptr, st);
  };
  auto scan_lengths = [&]() -> int {
    const gkd::HostWords told = host_words(ctx);
    GK_STAGE(ctx, GK_ST_CONTRACT_AUX, 12LL * nc,
             gkd::launch_len_scan(nc, len.p, scratch.p, c.xadj.p, cnt, told, st));
    if (early) GK_STAGE(ctx, GK_ST_CONTRACT_AUX, 12LL * nc, copy_rows(g.nnz));
    return wait_words(ctx, st, told, 1 + gkd::kRowCtlWords, words);
  };
  GK_TRY(scan_lengths());
  if (hc[4] > 0) {
    const int32_t nbig = hc[4], eb = hc[gkd::kRowBigEntries];
    not_early();
    const int32_t* rows = lists.p + int64_t(4) * nc;
    Buf<int32_t> boff, bscr;
    GK_TRY(boff.alloc(P, int64_t(nbig) + 1));
    GK_TRY(bscr.alloc(P, gkd::scan_scratch_ints(int64_t(nbig) + 1) + 64));
    GK_STAGE(ctx, GK_ST_CONTRACT_BIG, 16LL * nbig,
             gkd::launch_big_offsets(rows, len.p, nbig, boff.p, bscr.p, st));
    Buf<uint64_t> k1, k2;
    Buf<int32_t> v1, v2, sscr;
    GK_TRY(k1.alloc(P, eb));
    GK_TRY(k2.alloc(P, eb));
    GK_TRY(v1.alloc(P, eb));
    GK_TRY(v2.alloc(P, eb));
    GK_TRY(sscr.alloc(P, gkd::sort_scratch_ints(eb)));
    bool alt = false;
    const int bpasses = (32 + bits_for(nbig - 1) + 7) / 8;
    GK_STAGE(ctx, GK_ST_CONTRACT_BIG, 24LL * eb + 36LL * eb * bpasses + 24LL * eb,
             (gkd::launch_contract_big_gather(g, rows, nbig, boff.p, m.cptr.p, m.mrow.p, cmap, k1.p, v1.p, st) ||
                      gkd::radix_sort_pairs<uint64_t>(k1.p, v1.p, k2.p, v2.p, eb, 0, 32 + bits_for(nbig - 1),
                                                      sscr.p, st, &alt) ||
                      gkd::launch_contract_big_merge(rows, nbig, boff.p, alt ? k2.p : k1.p, alt ? v2.p : v1.p,
                                                     toff.p, tadj.p, tw.p, len.p, st)
                  ? GK_ERR_HIP
                  : GK_OK));
    GK_TRY(scan_lengths());
  }
  const int32_t cnnz = words[0];
  // Row merge: member rows and the cmap gathers read once, merged rows
  // written once (known now that cnnz is).
  if (ctx->cur) ctx->cur->stage_bytes[GK_ST_CONTRACT] += 8LL * g.n + 20LL * nc + 12LL * g.nnz + 8LL * cnnz;
  if (early) {
    if (ctx->cur) ctx->cur->stage_bytes[GK_ST_CONTRACT_AUX] += 16LL * cnnz;
  } else {
    GK_STAGE(ctx, GK_ST_CONTRACT_AUX, 12LL * nc + 16LL * cnnz, copy_rows(cnnz));
  }
  c.g.n = nc;
  c.g.nnz = cnnz;
  c.g.xadj = c.xadj.p;
  c.g.adj = c.adj.p;
  c.g.w = c.w.p;
  return GK_OK;
}

// Degrees as bytes, for graphs on which the matching is faster with them; left
// out where the pool has no room (they only save time).
int degree_table(gk_ctx* ctx, hipStream_t st, const DGraph& g, Buf<uint8_t>& deg) {
  if (g.n < gkd::kDegTable || deg.alloc(ctx->pool, (int64_t(g.n) + 3) & ~int64_t(3)) != GK_OK) return GK_OK;
  return gkd::launch_deg_table(g, deg.p, st);
}

int match_stage(gk_ctx* ctx, hipStream_t st, const DGraph& g, int32_t* cand) {
  const int def = gkd::lanes_for_degree(g.n ? double(g.nnz) / g.n : 0.0);
  Tuner::Shape shape{def, 256};
  Buf<uint8_t> deg;
  GK_TRY(degree_table(ctx, st, g, deg));
  auto run = [&](const Tuner::Shape& x) {
    return gkd::launch_match(g, x.lanes, x.block, deg.p, cand, st, steal_of(ctx));
  };
  if (ctx->autotune && g.nnz >= kTuneMinEntries) {
    const uint64_t key = Tuner::key(0, g.n, g.nnz);
    if (const Tuner::Shape* s = ctx->tuner.find(key)) {
      shape = *s;
    } else {
      // Vertices per wavefront around the degree table's choice, three block sizes.
      std::vector<Tuner::Shape> c;
      for (int l : {def, def / 2, def * 2})
        if (l >= 1 && l <= 64)
          for (int b : {256, 128, 512}) c.push_back({l, b});
      return ctx->tuner.tune(key, c, st, run, &shape);  // every candidate wrote cand
    }
  }
  return run(shape);
}

int gain_lanes(const DGraph& g) {
  const double avg = g.n > 0 ? double(g.nnz) / g.n : 0.0;
  int s = 4;
  while (s < 64 && s < 2.0 * avg) s <<= 1;
  return s;
}

// ---------------------------------------------------------------- rounds
namespace {

// One round by the separate kernels.
int wide_round(gk_ctx* ctx, hipStream_t st, const RoundState& s) {
  GK_STAGE(ctx, GK_ST_SELECT, 0,
           gkd::launch_select_list(s.g, s.vjob, s.gain, s.dest, s.pw, s.pw_off, s.cap, s.thr, s.cand, s.sb, s.hcnt,
                                   s.active, st));
  GK_STAGE(ctx, GK_ST_BALANCE, 0,
           gkd::launch_round_b(s.nj, s.kmax, s.v_off, s.M, s.kk, s.cap, s.pw_off, s.g, s.part, s.dest, s.gain, s.pw,
                               s.cut, s.rounds, s.moved, s.sb, s.xlist, s.hkey, s.upd, s.wl, s.hcnt, s.lastcnt,
                               s.active, s.cand, s.thr, s.paths, s.order, s.hist, s.abytes, s.movers, st));
  GK_STAGE(ctx, GK_ST_GAIN, 0,
           gkd::launch_gain_wl(s.g, s.kmax, s.lanes, s.wl, s.hcnt, s.heavy, s.part, s.upd, s.bnd, s.gain, s.dest,
                               s.work, s.wl_items, s.cand, st, steal_of(ctx)));
  if (s.heavy_rows)
    GK_STAGE(ctx, GK_ST_GAIN_HEAVY, 0,
             gkd::launch_gain_heavy(s.g, s.kmax, s.heavy, s.hcnt, s.part, s.upd, s.bnd, s.gain, s.dest, s.work, s.cand,
                                    st));
  return GK_OK;
}

// A launch of the round loop; pair: which pair of counts and status words it
// uses.
int loop_rounds(gk_ctx* ctx, hipStream_t st, const RoundState& s, int max_rounds, int pair,
                const gkd::HostWords& told) {
  const int o = 2 * pair, e = 2 * (1 - pair);
  const gkd::RoundsArgs a{s.v_off,     s.M,        max_rounds, s.kk,         s.cap,        s.pw_off,  s.g.xadj,
                          s.g.adj,     s.g.w,      s.g.vw,     s.part,       s.bnd,        s.gain,    s.dest,
                          s.pw,        s.cut,      s.rounds,   s.moved,      s.cand,       s.upd,     s.wl,
                          s.hcnt + o,  s.hcnt + e, s.lastcnt,  s.status + o, s.status + e, s.thr,     s.paths,
                          s.abytes,    s.order,    s.hist,     told};
  GK_STAGE(ctx, GK_ST_BALANCE, 0, gkd::launch_rounds(a, s.nj, s.lanes, st));
  return GK_OK;
}

// The gain pass over what a launch of the round loop left; none is needed
// after one in which every job converged.
int loop_gains(gk_ctx* ctx, hipStream_t st, const RoundState& s, int pair) {
  GK_STAGE(ctx, GK_ST_GAIN, 0,
           gkd::launch_gain_wl(s.g, s.kmax, s.lanes, s.wl, s.hcnt + 2 * pair, s.heavy, s.part, s.upd, s.bnd, s.gain, s.dest,
                               s.work, s.wl_items, s.cand, st, steal_of(ctx)));
  return GK_OK;
}

}  // namespace

int refine_rounds(gk_ctx* ctx, hipStream_t st, const RoundState& s, int max_rounds, bool exact, bool graph, int* ran) {
  graph = graph && !exact && !ctx->clock.timed(GK_ST_SELECT) && !ctx->clock.timed(GK_ST_BALANCE) &&
          !ctx->clock.timed(GK_ST_GAIN) && !ctx->clock.timed(GK_ST_GAIN_HEAVY);
  RoundPlan plan(s.kmax <= gkd::kGainInlineK, s.g.n, s.nj, max_rounds, exact, graph);
  RoundGraph wide_graph, loop_graph;
  // Jobs that go on, jobs left out, and with one job the ordering rounds so
  // far; one job's kernel writes them to pinned memory itself.
  const bool one = s.nj == 1;
  auto status = [&](int p, const gkd::HostWords& told, int32_t* words) -> int {
    if (one) return wait_words(ctx, st, told, 3, words);
    const gkd::HostWords t2 = host_words(ctx);
    GK_TRY(gkd::launch_tell(s.status + 2 * p, 2, t2, st));
    return wait_words(ctx, st, t2, 2, words);
  };
  auto listen = [&]() { return one ? host_words(ctx) : gkd::HostWords{}; };
  while (!plan.ended()) {
    const int rounds = plan.rounds();
    if (plan.loop()) {
      const int pair = plan.pair();
      int32_t words[3] = {0, 0, 0};
      if (plan.captured()) {
        if (!loop_graph.ready())
          GK_TRY(loop_graph.capture(ctx, st, [&]() -> int {
            GK_TRY(loop_rounds(ctx, st, s, rounds / 2, pair, gkd::HostWords{}));
            GK_TRY(loop_gains(ctx, st, s, pair));
            GK_TRY(loop_rounds(ctx, st, s, rounds / 2, 1 - pair, gkd::HostWords{}));
            return loop_gains(ctx, st, s, 1 - pair);
          }));
        GK_TRY(loop_graph.replay(ctx, st));
        const gkd::HostWords told = host_words(ctx);
        GK_TRY(gkd::launch_tell(s.status + 2 * (1 - pair), 2, told, st));
        GK_TRY(wait_words(ctx, st, told, 2, words));
      } else {
        const gkd::HostWords told = listen();
        GK_TRY(loop_rounds(ctx, st, s, rounds, pair, told));
        // Of several jobs some usually go on, and the wait is the longer part.
        if (!one) GK_TRY(loop_gains(ctx, st, s, pair));
        GK_TRY(status(pair, told, words));
        if (one && words[0] != 0) GK_TRY(loop_gains(ctx, st, s, pair));
      }
      plan.loop_ran(words[0], words[1], words[2]);
    } else {
      if (plan.captured()) {
        if (!wide_graph.ready())
          GK_TRY(wide_graph.capture(ctx, st, [&]() -> int {
            for (int r = 0; r < RoundPlan::kWideRounds; ++r) GK_TRY(wide_round(ctx, st, s));
            return GK_OK;
          }));
        for (int r = 0; r < rounds; r += RoundPlan::kWideRounds) GK_TRY(wide_graph.replay(ctx, st));
      } else {
        for (int r = 0; r < rounds; ++r) GK_TRY(wide_round(ctx, st, s));
      }
      int32_t live = 0;
      const gkd::HostWords told = host_words(ctx);
      GK_TRY(gkd::launch_tell(s.active, 1, told, st));
      GK_TRY(wait_words(ctx, st, told, 1, &live));
      if (plan.wide_ran(live)) {
        gkd::fill<int32_t>(s.hcnt, 0, 4, st);
        gkd::fill<int32_t>(s.status, 0, 4, st);
      }
    }
  }
  if (ran) *ran = plan.done();
  return GK_OK;
}

}  // namespace gkrt

namespace {

// ---------------------------------------------------------------- V-cycle
// The partition goes to dpart_out (device) or, if that is null, to part (host).
int run_vcycle(gk_ctx* ctx, hipStream_t st, const DGraph& g0in, const gk_params& prm,
               int32_t* dpart_out, gk_stats* stats, int32_t* part = nullptr) {
  using clk = std::chrono::steady_clock;
  const auto t0 = clk::now();
  Pool& P = ctx->pool;
  const int32_t k = prm.k;
  const bool trace = (prm.flags & GK_FLAG_TRACE) != 0;
  gk_stats S;
  std::memset(&S, 0, sizeof S);
  ctx->cur = &S;
  ctx->clock.start((prm.flags & GK_FLAG_STAGE_TIME) != 0, st);
  HostBlock top_down, part_up;
  StageGuard stage_guard{ctx, st};
  struct Reset {
    gk_ctx* c;
    ~Reset() {
      c->cur = nullptr;
      c->clock.start(false, nullptr);
      gkrt::clear_launch_options(c);
    }
  } reset{ctx};
  GK_TRY(gkrt::set_launch_options(ctx, prm.flags));

  std::vector<Level> L;
  L.reserve(GK_MAX_LEVELS + 1);
  L.emplace_back();
  L[0].g = g0in;
  const int32_t n0 = g0in.n;
  if (!g0in.w && g0in.nnz > 0) {
    GK_TRY(L[0].w.alloc(P, g0in.nnz));
    gkd::fill<int32_t>(L[0].w.p, 1, g0in.nnz, st);
    L[0].g.w = L[0].w.p;
  }
  if (!g0in.vw) {
    GK_TRY(L[0].vw.alloc(P, n0));
    gkd::fill<int32_t>(L[0].vw.p, 1, n0, st);
    L[0].g.vw = L[0].vw.p;
  }
  // The total weight comes back with the coarsest graph.
  Buf<unsigned long long> tw;
  GK_TRY(tw.alloc(P, 1));
  GK_TRY(gkd::launch_sum(L[0].g.vw, n0, tw.p, st));
  const int32_t floor_n = gk_coarsen_floor(n0, k, prm.coarsen_policy, prm.coarsen_to);
  const int32_t maxlv = prm.max_levels > 0 ? std::min(prm.max_levels, GK_MAX_LEVELS) : GK_MAX_LEVELS;

  // ---------------------------------------------------------- coarsening
  while (static_cast<int32_t>(L.size()) < maxlv) {
    Level& f = L.back();
    const int32_t n = f.g.n;
    if (!(n > floor_n)) break;
    gk_level_stats& ls = S.levels[L.size() - 1];
    Buf<int32_t> cand, cmap;
    Members mem;
    GK_TRY(cand.alloc(P, n));
    GK_TRY(cmap.alloc(P, n));
    GK_STAGE(ctx, GK_ST_MATCH, 16LL * f.g.nnz + 8LL * n + 4,
             match_stage(ctx, st, f.g, cand.p));
    int32_t rounds = 0, nc = 0;
    GK_TRY(coarse_ids(ctx, st, f.g, cand.p, prm.max_group, false, cmap.p, mem, &nc, &rounds));
    if (nc == n || nc < k + 1) break;
    if (prm.coarsen_policy != GK_COARSEN_REF && nc < floor_n) break;
    Level c;
    GK_TRY(c.vw.alloc(P, nc));
    c.g.vw = c.vw.p;
    if (!trace) cand.release();
    GK_TRY(contract_stage(ctx, st, f.g, nc, cmap.p, mem, c));
    ls.sweeps = rounds;
    if (trace) {
      std::vector<int32_t> h;
      GK_TRY(to_host(st, h, cand.p, n));
      ls.h_cand = fnv_host(h);
      GK_TRY(to_host(st, h, cmap.p, n));
      ls.h_cmap = fnv_host(h);
      std::vector<int32_t> a, b, d, e;
      GK_TRY(to_host(st, a, c.g.xadj, int64_t(nc) + 1));
      GK_TRY(to_host(st, b, c.g.adj, c.g.nnz));
      GK_TRY(to_host(st, d, c.g.w, c.g.nnz));
      GK_TRY(to_host(st, e, c.g.vw, nc));
      ls.h_coarse = fnv_host(e, fnv_host(d, fnv_host(b, fnv_host(a))));
    }
    f.cmap = std::move(cmap);
    L.push_back(std::move(c));
  }
  const int32_t nl = static_cast<int32_t>(L.size());

  // ---------------------------------------------------------- initial partition
  Level& top = L.back();
  const int32_t nt = top.g.n;
  // The largest row of every level refined later decides whether a level
  // needs the heavy-row gain kernel, which serves only large k.
  const bool heavy_k = gkd::gain_heavy_separate(k) && nl > 1;
  Buf<int32_t> dmaxall;
  if (heavy_k) {
    GK_TRY(dmaxall.alloc(P, nl));
    for (int32_t l = 0; l + 1 < nl; ++l) GK_TRY(gkd::launch_max_deg(L[l].g, dmaxall.p + l, st));
  }
  // The coarsest graph comes back into the context's pinned staging in one
  // launch, which writes there, and is partitioned from there.
  const int64_t tn = top.g.nnz;
  auto up4 = [](size_t ints) { return (ints + 3) & ~size_t(3); };  // 16-byte places
  GK_TRY(top_down.get(ctx->dl, st, sizeof(int32_t) * (4 + up4(nl) + up4(size_t(nt) + 1) + 2 * up4(tn) + up4(nt))));
  unsigned long long* ht = static_cast<unsigned long long*>(top_down.p());
  int32_t* hmaxdeg = reinterpret_cast<int32_t*>(ht + 2);
  int32_t* hx = hmaxdeg + up4(nl);
  int32_t* ha = hx + up4(size_t(nt) + 1);
  int32_t* hw = ha + up4(tn);
  int32_t* hv = hw + up4(tn);
  std::memset(hmaxdeg, 0, sizeof(int32_t) * size_t(nl));
  gkd::Copies dn;
  auto down = [&](void* dst, const void* src, size_t words) -> int {
    return top_down.copy(dn, st, dst, src, sizeof(int32_t) * words, hipMemcpyDeviceToHost);
  };
  GK_TRY(down(ht, tw.p, 2));
  if (heavy_k) GK_TRY(down(hmaxdeg, dmaxall.p, size_t(nl - 1)));
  GK_TRY(down(hx, top.g.xadj, size_t(nt) + 1));
  GK_TRY(down(ha, top.g.adj, size_t(tn)));
  GK_TRY(down(hw, top.g.w, size_t(tn)));
  GK_TRY(down(hv, top.g.vw, size_t(nt)));
  GK_TRY(gkd::launch_copies(dn, st));
  GK_HIP(hipStreamSynchronize(st));
  const std::vector<int32_t> maxdeg_of(hmaxdeg, hmaxdeg + nl);
  const auto t1 = clk::now();
  const int64_t T = static_cast<int64_t>(*ht);
  if (T >= (int64_t(1) << 31)) { gkh::set_error("total vertex weight >= 2^31"); return GK_ERR_LIMIT; }
  const int64_t cap = gk_part_cap(T, k, prm.ubfactor);
  S.total_vwgt = T;
  S.cap = cap;
  gk_csr hc;
  hc.n = nt;
  hc.nnz = tn;
  hc.xadj = hx;
  hc.adjncy = ha;
  hc.adjwgt = hw;
  hc.vwgt = hv;
  // The initial part goes up through pinned staging, and with it the words
  // of the refinement's state (64-bit, then 32-bit ones): per level cut after
  // the level, moves and algorithmic bytes, rounds, worklist counts and round
  // loop status; what the kernels take as one job's tables.
  const int nl64 = 3 * nl + 4, nl32 = 11 * nl + 7;
  const size_t state_bytes = sizeof(long long) * nl64 + sizeof(int32_t) * up4(nl32);
  struct State {
    long long *cut, *moved, *abytes, *paths, *cap;
    int32_t *rounds, *hcnt, *status, *voff, *pwoff, *kk, *thr, *lastcnt, *active;
  };
  auto state_at = [&](void* base) {
    State s;
    s.cut = static_cast<long long*>(base);
    s.moved = s.cut + nl;
    s.abytes = s.moved + nl;
    s.paths = s.abytes + nl;
    s.cap = s.paths + 3;
    s.rounds = reinterpret_cast<int32_t*>(s.cut + nl64);
    s.hcnt = s.rounds + nl;      // 4 per level: two pairs of (worklist, heavy rows)
    s.status = s.hcnt + 4 * nl;  // 4 per level
    s.voff = s.status + 4 * nl;  // 2 per level
    s.pwoff = s.voff + 2 * nl;
    s.kk = s.pwoff + 2;
    s.thr = s.kk + 1;
    s.lastcnt = s.thr + 1;
    s.active = s.lastcnt + 1;
    return s;
  };
  GK_TRY(part_up.get(ctx->up, st, sizeof(int32_t) * size_t(nt), state_bytes));
  void* hup = part_up.head();
  int32_t* hp = static_cast<int32_t*>(part_up.p());
  int64_t cut0 = 0;
  GK_TRY(gk_initpart(&hc, k, cap, prm.seed, prm.initpart_threads, hp, &cut0));
  std::memset(hup, 0, state_bytes);
  const State hs = state_at(hup);
  hs.cut[nl - 1] = cut0;
  *hs.cap = cap;
  for (int32_t l = 0; l < nl; ++l) hs.voff[2 * l + 1] = L[l].g.n;
  hs.pwoff[1] = k;
  *hs.kk = k;
  S.init_cut = cut0;
  Buf<int32_t> partA, partB, bndA, bndB, pw;
  GK_TRY(partA.alloc(P, n0));
  GK_TRY(partB.alloc(P, n0));
  GK_TRY(bndA.alloc(P, n0));
  GK_TRY(bndB.alloc(P, n0));
  GK_TRY(pw.alloc(P, k));
  // Gain statistics: a (vertices, entries) pair per block of the gain launches
  // (grids of at most kGainSlots blocks), and the selection kernels'
  // algorithmic bytes, likewise per block slot; summed at the end.
  constexpr int kGainSlots = gkd::kGainMaxBlocks;
  constexpr int kWork = 2 * kGainSlots + gkd::kSelectByteSlots;
  const int64_t nwords0 = (int64_t(n0) + 63) / 64;
  Buf<char> dstate;
  Buf<unsigned long long> work;
  Buf<uint64_t> selbits;
  GK_TRY(dstate.alloc(P, int64_t(state_bytes)));
  const State ds = state_at(dstate.p);
  gkd::Copies upc;
  upc.add(dstate.p, hup, state_bytes);
  GK_TRY(part_up.copy(upc, st, partA.p, hp, sizeof(int32_t) * size_t(nt), hipMemcpyHostToDevice));
  if (nl > 1) {
    GK_TRY(work.alloc(P, kWork));
    GK_TRY(selbits.alloc(P, nwords0 + 1));
    upc.add(pw.p, nullptr, sizeof(int32_t) * size_t(k));
    upc.add(work.p, nullptr, sizeof(unsigned long long) * kWork);
    upc.add(selbits.p, nullptr, sizeof(uint64_t) * size_t(nwords0 + 1));
  }
  GK_TRY(gkd::launch_copies(upc, st));
  if (nl > 1) GK_TRY(gkd::launch_part_state(top.g, k, partA.p, bndA.p, pw.p, st));
  S.levels[nl - 1].cut_after = cut0;
  if (trace) S.levels[nl - 1].h_part = fnv_host(std::vector<int32_t>(hp, hp + nt));
  const auto t2 = clk::now();

  // ---------------------------------------------------------- uncoarsening
  // Rounds run back to back on the device (refine_rounds).
  int32_t* cur_part = partA.p;
  int32_t* cur_bnd = bndA.p;
  int32_t* oth_part = partB.p;
  int32_t* oth_bnd = bndB.p;
  if (nl > 1) {
    const int32_t M = prm.max_moves;
    Buf<int32_t> movers, xlist, wpos, sscr, gain, dest, upd, heavy, wl, list;
    Buf<uint64_t> cand, movable, defbits;
    Buf<uint32_t> hkey;
    GK_TRY(gain.alloc(P, n0));
    GK_TRY(dest.alloc(P, n0));
    GK_TRY(upd.alloc(P, n0));
    GK_TRY(heavy.alloc(P, n0));
    GK_TRY(wl.alloc(P, n0));
    GK_TRY(list.alloc(P, n0));
    GK_TRY(hkey.alloc(P, n0));
    GK_TRY(cand.alloc(P, nwords0 + 1));
    GK_TRY(movable.alloc(P, nwords0 + 1));
    GK_TRY(defbits.alloc(P, nwords0 + 1));
    GK_TRY(wpos.alloc(P, nwords0 + 1));
    GK_TRY(sscr.alloc(P, gkd::select_scratch_ints(n0)));
    GK_TRY(xlist.alloc(P, n0));
    GK_TRY(movers.alloc(P, int64_t(M) + 1));
    const gkd::SelectBufs sb{movable.p, selbits.p, defbits.p, wpos.p, list.p, sscr.p, work.p + 2 * kGainSlots};
    for (int32_t l = nl - 2; l >= 0; --l) {
      Level& f = L[l];
      const DGraph& g = f.g;
      gk_level_stats& ls = S.levels[l];
      int32_t* hcnt = ds.hcnt + 4 * l;
      // The projected boundary becomes the first gain worklist; every gain is
      // 0, so there is no candidate yet.
      GK_STAGE(ctx, GK_ST_PROJECT, 32LL * g.n,
               gkd::launch_level_start(g.n, f.cmap.p, cur_part, cur_bnd, oth_part, oth_bnd, gain.p, dest.p, upd.p,
                                       cand.p, wl.p, hcnt, ds.cut + l + 1, ds.cut + l, ds.thr, ds.lastcnt, st));
      std::swap(cur_part, oth_part);
      std::swap(cur_bnd, oth_bnd);
      const int lanes = gain_lanes(g);
      // Rows longer than the lane count: the gain pass takes them itself for
      // k <= kGainInlineK, else they go to the heavy-row kernel, whose
      // launches are skipped when there are none.
      const bool heavy_rows = heavy_k && maxdeg_of[l] > lanes;
      GK_STAGE(ctx, GK_ST_GAIN, 0,
               gkd::launch_gain_wl(g, k, lanes, wl.p, hcnt, heavy.p, cur_part, upd.p, cur_bnd, gain.p, dest.p,
                                   work.p, g.n, cand.p, st, steal_of(ctx)));
      if (heavy_rows)
        GK_STAGE(ctx, GK_ST_GAIN_HEAVY, 0,
                 gkd::launch_gain_heavy(g, k, heavy.p, hcnt, cur_part, upd.p, cur_bnd, gain.p, dest.p, work.p,
                                        cand.p, st));
      // A round updates at most M movers and their neighbours.
      const int64_t avg_deg = g.n > 0 ? (int64_t(g.nnz) + g.n - 1) / g.n : 0;
      const int64_t wl_items = std::min<int64_t>(g.n, int64_t(M) * (1 + 2 * avg_deg));
      RoundState rs;
      rs.g = g;
      rs.kmax = k;
      rs.M = M;
      rs.lanes = lanes;
      rs.heavy_rows = heavy_rows;
      rs.wl_items = wl_items;
      rs.v_off = ds.voff + 2 * l;
      rs.kk = ds.kk;
      rs.pw_off = ds.pwoff;
      rs.cap = ds.cap;
      rs.part = cur_part;
      rs.bnd = cur_bnd;
      rs.gain = gain.p;
      rs.dest = dest.p;
      rs.pw = pw.p;
      rs.upd = upd.p;
      rs.cut = ds.cut + l;
      rs.moved = ds.moved + l;
      rs.paths = ds.paths;
      rs.abytes = ds.abytes + l;
      rs.rounds = ds.rounds + l;
      rs.lastcnt = ds.lastcnt;
      rs.thr = ds.thr;
      rs.active = ds.active;
      rs.cand = cand.p;
      rs.sb = sb;
      rs.xlist = xlist.p;
      rs.movers = movers.p;
      rs.wl = wl.p;
      rs.hcnt = hcnt;
      rs.heavy = heavy.p;
      rs.status = ds.status + 4 * l;
      rs.hkey = hkey.p;
      rs.work = work.p;
      GK_TRY(refine_rounds(ctx, st, rs, 0, false, (prm.flags & GK_FLAG_GRAPH_ROUNDS) != 0, nullptr));
      if (trace) {
        std::vector<int32_t> h;
        GK_TRY(to_host(st, h, cur_part, g.n));
        ls.h_part = fnv_host(h);
      }
    }
  }
  const auto t3 = clk::now();

  // ---------------------------------------------------------- final metrics
  {
    Buf<unsigned long long> cut, pw64, cscr;
    GK_TRY(cut.alloc(P, 1));
    GK_TRY(pw64.alloc(P, k));
    GK_TRY(cscr.alloc(P, gkd::cut_scratch(L[0].g.n, k)));
    GK_STAGE(ctx, GK_ST_CUT, 16LL * n0 + 12LL * L[0].g.nnz,
             gkd::launch_cut(L[0].g, k, cur_part, cut.p, pw64.p, cscr.p, st));
    // The partition, the metrics and the levels' figures, in one launch.
    void* hend = nullptr;
    const size_t part_bytes = sizeof(int32_t) * size_t(n0);
    const bool staged = !dpart_out && part_bytes <= kStageMax;
    const size_t own = (state_bytes + 32 + sizeof(unsigned long long) * (size_t(k) + 2 + kWork) + 15) & ~size_t(15);
    GK_TRY(ctx->dl.get(st, own + (staged ? part_bytes : 0), &hend));
    unsigned long long* hcut = static_cast<unsigned long long*>(hend);
    unsigned long long* hpw64 = hcut + 2;
    unsigned long long* hwork = hpw64 + ((size_t(k) + 1) & ~size_t(1));
    void* hstate = hwork + kWork;
    gkd::Copies fin;
    void* hpart = static_cast<char*>(hend) + own;
    if (dpart_out) fin.add(dpart_out, cur_part, part_bytes);
    else if (staged) fin.add(hpart, cur_part, part_bytes);
    fin.add(hcut, cut.p, sizeof *hcut);
    fin.add(hpw64, pw64.p, sizeof *hpw64 * size_t(k));
    fin.add(hstate, dstate.p, state_bytes);
    if (nl > 1) fin.add(hwork, work.p, sizeof *hwork * size_t(kWork));
    GK_TRY(gkd::launch_copies(fin, st));
    GK_HIP(hipStreamSynchronize(st));
    if (!dpart_out && *hcut == static_cast<unsigned long long>(state_at(hstate).cut[0])) {
      if (staged) std::memcpy(part, hpart, part_bytes);
      else GK_HIP(hipMemcpy(part, cur_part, part_bytes, hipMemcpyDeviceToHost));
    }
    const State fs = state_at(hstate);
    S.cut = static_cast<int64_t>(*hcut);
    S.cut_tracked = fs.cut[0];
    for (int i = 0; i < 3; ++i) S.round_paths[i] = fs.paths[i];
    for (int32_t l = 0; l + 1 < nl; ++l) {
      gk_level_stats& ls = S.levels[l];
      // The round kernel's algorithmic bytes, counted on the device.
      S.stage_bytes[GK_ST_BALANCE] += fs.abytes[l];
      ls.rounds = fs.rounds[l];
      ls.moves = fs.moved[l];
      ls.cut_after = fs.cut[l];
    }
    if (nl > 1) {
      // Data-dependent bytes of the gain passes and the selection.
      unsigned long long wv = 0, we = 0;
      for (int i = 0; i < kGainSlots; ++i) {
        wv += hwork[2 * i];
        we += hwork[2 * i + 1];
      }
      S.stage_bytes[GK_ST_GAIN] += int64_t(28 * wv + 12 * we);
      for (int i = 0; i < gkd::kSelectByteSlots; ++i) S.stage_bytes[GK_ST_SELECT] += int64_t(hwork[2 * kGainSlots + i]);
    }
    stage_guard.done = true;
    unsigned long long mx = 0;
    for (int32_t q = 0; q < k; ++q) mx = std::max(mx, hpw64[q]);
    S.max_part_wgt = static_cast<int64_t>(mx);
    S.imbalance = T > 0 ? double(mx) * k / double(T) : 1.0;
  }
  S.nlevels = nl;
  S.coarsest_n = nt;
  for (int32_t l = 0; l < nl; ++l) {
    S.levels[l].n = L[l].g.n;
    S.levels[l].nnz = L[l].g.nnz;
  }
  auto ms = [](clk::time_point a, clk::time_point b) {
    return std::chrono::duration<double, std::milli>(b - a).count();
  };
  S.t_coarsen_ms = ms(t0, t1);
  S.t_init_ms = ms(t1, t2);
  S.t_refine_ms = ms(t2, t3);
  GK_TRY(ctx->clock.collect(S));
  S.t_total_ms = ms(t0, clk::now());
  for (int i = 0; i < GK_ST_COUNT; ++i) S.alg_bytes += S.stage_bytes[i];
  if (stats) *stats = S;
  if (S.cut != S.cut_tracked) {
    gkh::set_error("tracked cut " + std::to_string(S.cut_tracked) + " != recomputed cut " +
                   std::to_string(S.cut));
    return GK_ERR_INTERNAL;
  }
  return GK_OK;
}

// Entries from which a host graph is checked on the device.
constexpr int32_t kDeviceCheckEntries = 1 << 15;

// A host graph to the device, and, with check, its validity.  Up to kStageMax
// bytes go through pinned staging memory in pieces, a launch carrying one while
// the next is staged (2.4 MB: 36 us to stage and 52 us to carry, 97 us by the
// runtime's copy from pageable memory), and a few thousand vertices in one
// launch instead of four copies of 25 us: a whole call on 2048 vertices went
// from 617 to 558 us, and one on 100 k vertices, with the check on the device,
// from 2880 to 2031 us.
int upload_graph(gk_ctx* ctx, hipStream_t st, const gk_csr& h, bool check, Buf<int32_t>& x, Buf<int32_t>& a,
                 Buf<int32_t>& w, Buf<int32_t>& v, DGraph* g) {
  Pool& P = ctx->pool;
  const size_t nb = sizeof(int32_t) * size_t(h.n), eb = sizeof(int32_t) * size_t(h.nnz);
  struct Array {
    Buf<int32_t>& dev;
    const int32_t* host;
    size_t bytes;
  };
  const Array arrays[4] = {{x, h.xadj, nb + sizeof(int32_t)}, {a, h.adjncy, eb}, {w, h.adjwgt, eb}, {v, h.vwgt, nb}};
  size_t total = 0;
  if (!eb) GK_TRY(a.alloc(P, 1));
  for (const Array& y : arrays) {
    if (!y.host || !y.bytes) continue;
    GK_TRY(y.dev.alloc(P, int64_t(y.bytes / sizeof(int32_t))));
    total += (y.bytes + 15) & ~size_t(15);
  }
  Buf<unsigned long long> verdict;
  GK_TRY(verdict.alloc(P, 3));
  gkd::Copies c;
  if (check) c.add(verdict.p, nullptr, 3 * sizeof(unsigned long long));
  if (total <= kStageMax) {
    void* stage = nullptr;
    GK_TRY(ctx->up.get(st, total, &stage));
    char* to = static_cast<char*>(stage);
    size_t pending = 0;
    for (const Array& y : arrays) {
      if (!y.host || !y.bytes) continue;
      for (size_t o = 0; o < y.bytes; o += kStagePiece) {
        const size_t b = std::min(kStagePiece, y.bytes - o);
        std::memcpy(to, reinterpret_cast<const char*>(y.host) + o, b);
        c.add(reinterpret_cast<char*>(y.dev.p) + o, to, b);
        to += (b + 15) & ~size_t(15);
        pending += b;
        if (pending >= kStagePiece || c.n == gkd::Copies::kMax) {
          GK_TRY(gkd::launch_copies(c, st));
          c = gkd::Copies{};
          pending = 0;
        }
      }
    }
    GK_TRY(gkd::launch_copies(c, st));
  } else {
    GK_TRY(gkd::launch_copies(c, st));
    for (const Array& y : arrays)
      if (y.host && y.bytes) GK_HIP(hipMemcpyAsync(y.dev.p, y.host, y.bytes, hipMemcpyHostToDevice, st));
  }
  g->n = h.n;
  g->nnz = h.nnz;
  g->xadj = x.p;
  g->adj = a.p;
  g->w = h.adjwgt ? w.p : nullptr;
  g->vw = h.vwgt ? v.p : nullptr;
  if (!check) return GK_OK;
  GK_TRY(gkd::launch_graph_check(*g, verdict.p, st));
  unsigned long long r[3];
  int32_t halves[6];
  const gkd::HostWords told = host_words(ctx);
  GK_TRY(gkd::launch_tell(reinterpret_cast<const int32_t*>(verdict.p), 6, told, st));
  GK_TRY(wait_words(ctx, st, told, 6, halves));
  std::memcpy(r, halves, sizeof r);
  const unsigned long long limit = 1ull << 31;
  if (r[0] != 0 || r[1] >= limit || r[2] / 2 >= limit) {
    gkh::set_error("graph changed while it was read");  // unless the host's check names its fault
    return GK_ERR_GRAPH;
  }
  return GK_OK;
}

int check_params(const gk_params* p) {
  if (!p) { gkh::set_error("null params"); return GK_ERR_ARG; }
  if (p->k < 1 || p->k > kMaxK) { gkh::set_error("k must be in [1, 8192]"); return GK_ERR_ARG; }
  if (p->ubfactor < 0) { gkh::set_error("ubfactor < 0"); return GK_ERR_ARG; }
  if (p->max_group < 1 || p->max_group > 64) { gkh::set_error("max_group must be in [1, 64]"); return GK_ERR_ARG; }
  if (p->max_moves < 1 || p->max_moves > 1024) { gkh::set_error("max_moves must be in [1, 1024]"); return GK_ERR_ARG; }
  return GK_OK;
}

struct DeviceGuard {
  explicit DeviceGuard(int d) { (void)hipSetDevice(d); }
};

// ---------------------------------------------------------------- no-alloc cut
// gk_k_cut_noalloc keeps the cut kernel's per-block slots (one 64-bit cut
// share per block, then k 64-bit part weights per block) in `scratch` instead
// of pool memory: 2^18 slots = 2 MiB on every device the library runs on,
// held until the process ends.  Every slot a launch reads was written by the
// same launch, so nothing needs clearing between calls.
constexpr int64_t kCutScratchSlots = int64_t(1) << 18;
static_assert(kCutScratchSlots >= 2 * (int64_t(kMaxK) + 1), "two blocks of slots at the largest k");
static __device__ __align__(256) unsigned long long scratch[kCutScratchSlots];

// On the host, `scratch` names a host-side shadow, not device memory.  Its
// device address on each device is looked up once, with that device current
// (gk_ctx_create), and only that address is ever handed to kernels.
constexpr int kScratchDevices = 256;
std::mutex g_scratch_mu;
unsigned long long* g_scratch_addr[kScratchDevices] = {};

int scratch_setup(int device) {
  if (device < 0 || device >= kScratchDevices) return GK_OK;  // gk_k_cut_noalloc rejects such devices
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_addr[device]) return GK_OK;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    (void)hipGetLastError();
    gkh::set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    return GK_ERR_NODEVICE;
  }
  g_scratch_addr[device] = static_cast<unsigned long long*>(p);
  return GK_OK;
}

unsigned long long* scratch_addr(int device) {
  if (device < 0 || device >= kScratchDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return g_scratch_addr[device];
}

}  // namespace

extern "C" {

int gk_ctx_create(int device, gk_ctx** out) {
  if (!out) { gkh::set_error("null out"); return GK_ERR_ARG; }
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
    (void)hipGetLastError();
    gkh::set_error("no HIP device");
    return GK_ERR_NODEVICE;
  }
  if (device < 0 || device >= ndev) { gkh::set_error("device out of range"); return GK_ERR_ARG; }
  GK_HIP(hipSetDevice(device));
  GK_TRY(scratch_setup(device));
  gk_ctx* c = new gk_ctx;
  c->device = device;
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    gkh::set_error("hipStreamCreate failed");
    return GK_ERR_HIP;
  }
  if (hipHostMalloc(reinterpret_cast<void**>(&c->hpin), kPinFetch + kPinCtl, hipHostMallocDefault) != hipSuccess) {
    (void)hipStreamDestroy(c->stream);
    delete c;
    gkh::set_error("hipHostMalloc failed");
    return GK_ERR_NOMEM;
  }
  c->hctl = reinterpret_cast<unsigned long long*>(c->hpin + kPinFetch);
  std::memset(c->hctl, 0, kPinCtl);
  *out = c;
  return GK_OK;
}

int gk_ctx_set_stage_mask(gk_ctx* c, uint32_t mask) {
  if (!c) return GK_ERR_ARG;
  c->clock.set_mask(mask);
  return GK_OK;
}

int gk_ctx_set_pool_limit(gk_ctx* c, int64_t bytes) {
  if (!c || bytes < 0) { gkh::set_error("bad argument"); return GK_ERR_ARG; }
  c->pool.set_limit(bytes);
  return GK_OK;
}

int gk_ctx_destroy(gk_ctx* c) {
  if (!c) return GK_OK;
  DeviceGuard dg(c->device);
  (void)hipStreamSynchronize(c->stream);
  c->pool.release_all();
  (void)hipHostFree(c->hpin);
  (void)hipStreamDestroy(c->stream);
  delete c;
  return GK_OK;
}

int gk_partition_device(gk_ctx* ctx, const gk_csr* dg, const gk_params* prm, int32_t* dpart,
                        gk_stats* stats, void* stream) {
  if (!ctx || !dg || !dpart) { gkh::set_error("null argument"); return GK_ERR_ARG; }
  GK_TRY(check_params(prm));
  if (dg->n < 0 || dg->nnz < 0 || !dg->xadj || (dg->nnz > 0 && !dg->adjncy)) {
    gkh::set_error("bad graph description");
    return GK_ERR_ARG;
  }
  DeviceGuard guard(ctx->device);
  hipStream_t st = stream ? static_cast<hipStream_t>(stream) : ctx->stream;
  if (dg->n == 0) {
    if (stats) std::memset(stats, 0, sizeof *stats);
    return GK_OK;
  }
  DGraph g;
  g.n = dg->n;
  g.nnz = dg->nnz;
  g.xadj = dg->xadj;
  g.adj = dg->adjncy;
  g.w = dg->adjwgt;
  g.vw = dg->vwgt;
  return run_vcycle(ctx, st, g, *prm, dpart, stats);
}

int gk_partition(gk_ctx* ctx, const gk_csr* hg, const gk_params* prm, int32_t* part, gk_stats* stats) {
  if (!ctx || !hg || !part) { gkh::set_error("null argument"); return GK_ERR_ARG; }
  GK_TRY(check_params(prm));
  const bool symmetry = (prm->flags & GK_FLAG_CHECK) != 0;
  const int32_t n = hg->n, nnz = hg->nnz;
  // Graphs of kDeviceCheckEntries entries or more whose ends are sound are
  // checked on the device: three launches and a wait, some 20 us, against 1.3 ns
  // an entry on the host (12 k entries 10 us, 600 k entries 810 us).  A graph
  // that fails there is checked again here, for its error.
  const bool device_check = !symmetry && n > 0 && hg->xadj && hg->xadj[0] == 0 && hg->xadj[n] == nnz && hg->adjncy &&
                            nnz >= kDeviceCheckEntries;
  if (!device_check) GK_TRY(gk_graph_check(hg, symmetry));
  DeviceGuard guard(ctx->device);
  hipStream_t st = ctx->stream;
  if (n == 0) {
    if (stats) std::memset(stats, 0, sizeof *stats);
    return GK_OK;
  }
  Buf<int32_t> x, a, w, v;
  DGraph g;
  const int rc = upload_graph(ctx, st, *hg, device_check, x, a, w, v, &g);
  if (rc != GK_OK) {
    (void)hipStreamSynchronize(st);
    ctx->up.drained();
    // a wrong graph is refused as such, whatever else went wrong
    if (device_check) GK_TRY(gk_graph_check(hg, symmetry));
    return rc;
  }
  return run_vcycle(ctx, st, g, *prm, nullptr, stats, part);
}

int gk_partition_file(gk_ctx* ctx, const char* graph_file, const char* out_file, int32_t k,
                      gk_stats* stats) {
  if (!ctx || !graph_file || !out_file) { gkh::set_error("null argument"); return GK_ERR_ARG; }
  gk_csr g;
  GK_TRY(gk_graph_read(graph_file, &g));
  gk_params p;
  gk_params_default(&p, k);
  std::vector<int32_t> part(g.n > 0 ? g.n : 1);
  int rc = gk_partition(ctx, &g, &p, part.data(), stats);
  if (rc == GK_OK) rc = gk_write_partition((std::string(out_file) + ".out").c_str(), part.data(), g.n);
  gk_graph_free(&g);
  return rc;
}

// ---------------------------------------------------------------- stage hooks
static DGraph dview(const gk_csr* g) {
  DGraph d;
  d.n = g->n;
  d.nnz = g->nnz;
  d.xadj = g->xadj;
  d.adj = g->adjncy;
  d.w = g->adjwgt;
  d.vw = g->vwgt;
  return d;
}

static hipStream_t pick(gk_ctx* ctx, void* s) { return s ? static_cast<hipStream_t>(s) : ctx->stream; }

int gk_k_match(gk_ctx* ctx, const gk_csr* dg, int32_t* cand, void* stream) {
  if (!ctx || !dg || !cand || !dg->adjwgt) { gkh::set_error("null argument (adjwgt required)"); return GK_ERR_ARG; }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  DGraph g = dview(dg);
  Buf<uint8_t> deg;
  GK_TRY(gkrt::degree_table(ctx, st, g, deg));
  GK_TRY(gkd::launch_match(g, gkd::lanes_for_degree(g.n ? double(g.nnz) / g.n : 0.0), 256, deg.p, cand, st));
  GK_HIP(hipStreamSynchronize(st));
  return GK_OK;
}

int gk_k_group(gk_ctx* ctx, int32_t n, const int32_t* cand, int32_t* label, int32_t* stamp,
               int32_t* sweeps, void* stream) {
  if (!ctx || !cand || !label || !stamp) { gkh::set_error("null argument"); return GK_ERR_ARG; }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  if (n <= 0) { if (sweeps) *sweeps = 0; return GK_OK; }
  Groups gr;
  int32_t words[gkd::kCtlInts];
  // The walk writes labels and hops while it reads candidates: where those lie
  // in the same place, it works on a copy.
  Buf<int32_t> own;
  StageGuard drain{ctx, st};  // an early end leaves nothing queued on memory that goes back
  auto apart = [&](const int32_t* x) { return x + n <= cand || cand + n <= x; };
  if (!apart(stamp) || !apart(label)) {
    GK_TRY(own.alloc(ctx->pool, n));
    GK_HIP(hipMemcpyAsync(own.p, cand, sizeof(int32_t) * n, hipMemcpyDeviceToDevice, st));
    cand = own.p;
  }
  const gkd::HostWords told = gkrt::host_words(ctx);
  GK_TRY(gr.walk(ctx, st, n, cand, label, stamp));
  GK_TRY(gkd::launch_tell(gr.ctl.p, gkd::kCtlInts, told, st));
  GK_HIP(hipStreamSynchronize(st));
  GK_TRY(gkrt::wait_words(ctx, st, told, gkd::kCtlInts, words));
  int32_t rounds = Groups::rounds(words);
  if (words[gkd::kCtlFlags + gkd::kWalkBits]) {
    GK_TRY(gr.jump(ctx, st, n, cand, label, &rounds));
    GK_HIP(hipMemcpyAsync(stamp, gr.dist.p, sizeof(int32_t) * n, hipMemcpyDeviceToDevice, st));
    GK_HIP(hipStreamSynchronize(st));
  }
  drain.done = true;
  if (sweeps) *sweeps = rounds;
  return GK_OK;
}

int gk_k_cluster(gk_ctx* ctx, int32_t n, const int32_t* label, const int32_t* stamp, const int32_t* vwgt,
                 int32_t max_group, int32_t* order, int32_t* cmap, int32_t* cvwgt, int32_t* nc,
                 void* stream) {
  if (!ctx || !label || !stamp || !vwgt || !order || !cmap || !cvwgt || !nc || max_group < 1) {
    gkh::set_error("bad argument");
    return GK_ERR_ARG;
  }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  if (n <= 0) { *nc = 0; return GK_OK; }
  Groups gr;
  Buf<int32_t> cptr, mvw;
  GK_TRY(cptr.alloc(ctx->pool, int64_t(n) + 1));
  GK_TRY(mvw.alloc(ctx->pool, n));
  const MemberOut out{order, cmap, cptr.p, nullptr, mvw.p};
  int32_t words[gkd::kCtlInts];
  StageGuard drain{ctx, st};
  GK_TRY(gr.count(ctx, st, n, label));
  gkd::HostWords told;
  bool no_room = false;
  GK_TRY(count_members(ctx, st, n, label, stamp, gr, nullptr, vwgt, max_group, out, &told, &no_room));
  if (!no_room) GK_TRY(gkd::launch_cvwgt(n, gr.ctl.p, cptr.p, mvw.p, cvwgt, st));
  GK_HIP(hipStreamSynchronize(st));
  GK_TRY(gkrt::wait_words(ctx, st, told, gkd::kCtlInts, words));
  if (words[gkd::kCtlFlags]) { gkh::set_error("label outside [0, n)"); return GK_ERR_ARG; }
  *nc = words[0];
  if (words[1] || no_room) {
    gr.counts_done();
    // The stamp bit width is taken from the data (max stamp).
    std::vector<int32_t> hs;
    GK_TRY(to_host(st, hs, stamp, n));
    int32_t mx = 0;
    for (int32_t x : hs) mx = std::max(mx, x);
    GK_TRY(sort_members(ctx, st, n, label, stamp, bits_for(mx), nullptr, vwgt, max_group, out, nullptr, &mvw, nc));
    GK_TRY(gkd::launch_cvwgt(*nc, nullptr, cptr.p, mvw.p, cvwgt, st));
    GK_HIP(hipStreamSynchronize(st));
  }
  drain.done = true;
  return GK_OK;
}

int gk_k_contract(gk_ctx* ctx, const gk_csr* dg, const int32_t* cmap, int32_t nc, int32_t* cxadj,
                  int32_t* cadjncy, int32_t* cadjwgt, int32_t* cnnz, void* stream) {
  if (!ctx || !dg || !cmap || !cxadj || !cadjncy || !cadjwgt || !cnnz || !dg->adjwgt) {
    gkh::set_error("bad argument");
    return GK_ERR_ARG;
  }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  Pool& P = ctx->pool;
  const int32_t n = dg->n;
  // Members of each coarse vertex, in any order (the rows are sorted).
  Members m;
  Groups gr;
  Buf<int2> partial;
  GK_TRY(m.cptr.alloc(P, int64_t(n) + 1));
  GK_TRY(m.mrow.alloc(P, n));
  GK_TRY(partial.alloc(P, gkd::size_partials(n)));
  int32_t words[gkd::kCtlFlags + 1] = {};  // coarse vertices counted, flags
  StageGuard drain{ctx, st};
  GK_TRY(gr.count(ctx, st, n, cmap));
  if (n > 0) {
    const gkd::HostWords told = gkrt::host_words(ctx);
    GK_TRY(gkd::launch_size_scan(n, gr.size.p, INT32_MAX, partial.p, gr.comp.p, gr.ctl.p, told, st));
    GK_TRY(gkd::launch_member_place(n, cmap, gr.slot.p, gr.comp.p, dg->xadj, gr.ctl.p, m.cptr.p, m.mrow.p, st));
    GK_TRY(gkrt::wait_words(ctx, st, told, gkd::kCtlFlags + 1, words));
  }
  m.ctl = std::move(gr.ctl);
  // With G = INT32_MAX every label is one chunk, so chunks are the coarse
  // vertices in id order exactly when cmap is onto [0, nc).
  if (words[0] != nc || words[gkd::kCtlFlags]) { gkh::set_error("cmap is not onto [0, nc)"); return GK_ERR_ARG; }
  Level c;
  DGraph g = dview(dg);
  const CsrOut out{cxadj, cadjncy, cadjwgt};
  GK_TRY(contract_stage(ctx, st, g, nc, cmap, m, c, &out));
  if (nc == 0) gkd::fill<int32_t>(cxadj, 0, 1, st);
  GK_HIP(hipStreamSynchronize(st));
  drain.done = true;
  *cnnz = c.g.nnz;
  return GK_OK;
}

int gk_k_project(gk_ctx* ctx, int32_t n, const int32_t* cmap, const int32_t* cpart, const int32_t* cbnd,
                 int32_t* part, int32_t* bnd, int32_t* gain, int32_t* dest, int32_t* upd, void* stream) {
  if (!ctx) return GK_ERR_ARG;
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  GK_TRY(gkd::launch_project(n, cmap, cpart, cbnd, part, bnd, gain, dest, upd, st));
  GK_HIP(hipStreamSynchronize(st));
  return GK_OK;
}

int gk_k_gain(gk_ctx* ctx, const gk_csr* dg, int32_t k, const int32_t* part, const int32_t* upd,
              int32_t* bnd, int32_t* gain, int32_t* dest, void* stream) {
  if (!ctx || !dg || !dg->adjwgt || k < 1 || k > kMaxK) { gkh::set_error("bad argument"); return GK_ERR_ARG; }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  DGraph g = dview(dg);
  const int lanes = gain_lanes(g);
  Buf<int32_t> wl, heavy, cnt;
  GK_TRY(wl.alloc(ctx->pool, g.n));
  GK_TRY(heavy.alloc(ctx->pool, g.n));
  GK_TRY(cnt.alloc(ctx->pool, 2));
  gkd::fill<int32_t>(cnt.p, 0, 2, st);
  // The caller's flags stay as they are (none given to the gain kernels).
  GK_TRY(gkd::launch_compact(g.n, upd, wl.p, cnt.p, st));
  GK_TRY(gkd::launch_gain_wl(g, k, lanes, wl.p, cnt.p, heavy.p, part, nullptr, bnd, gain, dest, nullptr, g.n, nullptr,
                              st));
  if (gkd::gain_heavy_separate(k))
    GK_TRY(gkd::launch_gain_heavy(g, k, heavy.p, cnt.p, part, nullptr, bnd, gain, dest, nullptr, nullptr, st));
  GK_HIP(hipStreamSynchronize(st));
  return GK_OK;
}

int gk_k_select(gk_ctx* ctx, const gk_csr* dg, const int32_t* part, const int32_t* bnd, const int32_t* gain,
                const int32_t* dest, const int32_t* pw, int64_t cap, int32_t max_moves, int32_t* upd,
                int32_t* moves, int32_t* nsel, void* stream) {
  (void)part;
  if (!ctx || !dg || !dg->vwgt || !moves || !nsel || max_moves < 1) { gkh::set_error("bad argument"); return GK_ERR_ARG; }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  DGraph g = dview(dg);
  Pool& P = ctx->pool;
  Buf<uint64_t> keys, keys2;
  Buf<int32_t> ctl, sscr;
  GK_TRY(keys.alloc(P, g.n));
  GK_TRY(keys2.alloc(P, g.n));
  GK_TRY(ctl.alloc(P, 4));
  GK_TRY(sscr.alloc(P, gkd::sort_scratch_ints(g.n)));
  const int idbits = bits_for(g.n > 0 ? g.n - 1 : 0);
  GK_TRY(gkd::launch_select(g, bnd, gain, dest, pw, cap, idbits, upd, keys.p, ctl.p, nullptr, 1, nullptr, st));
  int32_t hc[2];
  GK_TRY(fetch(ctx, st, {{hc, ctl.p, sizeof hc}}));
  *nsel = hc[0];
  if (hc[0] == 0) return GK_OK;
  bool alt = false;
  if (gkd::radix_sort_pairs<uint64_t>(keys.p, nullptr, keys2.p, nullptr, hc[0], 0, idbits + bits_for(hc[1]),
                                      sscr.p, st, &alt))
    GK_HIP(hipGetLastError());
  std::vector<uint64_t> hk;
  GK_TRY(to_host(st, hk, alt ? keys2.p : keys.p, hc[0]));
  const int32_t B = std::min(hc[0], max_moves);
  std::vector<int32_t> mv(B);
  const uint64_t mask = (1ull << idbits) - 1;
  for (int32_t i = 0; i < B; ++i) mv[i] = int32_t(hk[i] & mask);
  GK_HIP(hipMemcpyAsync(moves, mv.data(), sizeof(int32_t) * B, hipMemcpyHostToDevice, st));
  GK_HIP(hipStreamSynchronize(st));
  return GK_OK;
}

int gk_k_balance(gk_ctx* ctx, const gk_csr* dg, int32_t k, const int32_t* moves, int32_t nmoves,
                 const int32_t* part, const int32_t* dest, int32_t* pw, int64_t cap, int32_t* pos,
                 void* stream) {
  if (!ctx || !dg || !dg->vwgt || !pos || k < 1 || k > kMaxK || nmoves > 1024) {
    gkh::set_error("bad argument");
    return GK_ERR_ARG;
  }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  if (nmoves <= 0) { *pos = -1; return GK_OK; }
  DGraph g = dview(dg);
  Pool& P = ctx->pool;
  // Keys in the given order: the vertex id with idbits = 32 (presorted).
  std::vector<int32_t> hm;
  GK_TRY(to_host(st, hm, moves, nmoves));
  std::vector<uint64_t> hk(nmoves);
  for (int32_t i = 0; i < nmoves; ++i) hk[i] = uint64_t(uint32_t(hm[i]));
  Buf<uint64_t> keys;
  Buf<int32_t> out, ctl, gz;
  Buf<long long> cut;
  GK_TRY(keys.alloc(P, nmoves));
  GK_TRY(out.alloc(P, nmoves));
  GK_TRY(ctl.alloc(P, 4));
  GK_TRY(gz.alloc(P, g.n));
  GK_TRY(cut.alloc(P, 1));
  gkd::fill<int32_t>(gz.p, 0, g.n, st);
  gkd::fill<long long>(cut.p, 0, 1, st);
  GK_HIP(hipMemcpyAsync(keys.p, hk.data(), sizeof(uint64_t) * nmoves, hipMemcpyHostToDevice, st));
  GK_TRY(gkd::launch_balance(g, k, keys.p, nmoves, nmoves, true, 32, part, dest, gz.p, pw, cap, out.p,
                             ctl.p, cut.p, st));
  int32_t hc[3];
  GK_TRY(fetch(ctx, st, {{hc, ctl.p, sizeof hc}}));
  *pos = hc[2];
  return GK_OK;
}

int gk_k_apply(gk_ctx* ctx, const gk_csr* dg, const int32_t* moves, int32_t pos, const int32_t* gain,
               const int32_t* dest, int32_t* part, int32_t* upd, int64_t* gain_sum, void* stream) {
  if (!ctx || !dg || !moves || !gain_sum) { gkh::set_error("bad argument"); return GK_ERR_ARG; }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  DGraph g = dview(dg);
  *gain_sum = 0;
  if (pos < 0) return GK_OK;
  std::vector<int32_t> hm, hg;
  GK_TRY(to_host(st, hm, moves, int64_t(pos) + 1));
  GK_TRY(to_host(st, hg, gain, g.n));
  int64_t s = 0;
  for (int32_t v : hm) s += hg[v];
  Buf<int32_t> ctl, wl, wlc;
  GK_TRY(ctl.alloc(ctx->pool, 4));
  GK_TRY(wl.alloc(ctx->pool, g.n));
  GK_TRY(wlc.alloc(ctx->pool, 2));
  gkd::fill<int32_t>(ctl.p, pos, 4, st);
  gkd::fill<int32_t>(wlc.p, 0, 2, st);
  GK_TRY(gkd::launch_apply(g, pos + 1, moves, ctl.p, dest, part, upd, wl.p, wlc.p, st));
  GK_HIP(hipStreamSynchronize(st));
  *gain_sum = s;
  return GK_OK;
}

int gk_k_round(gk_ctx* ctx, const gk_csr* dg, int32_t k, int64_t cap, int32_t max_moves, int32_t nrounds,
               int32_t* part, int32_t* bnd, int32_t* gain, int32_t* dest, int32_t* pw, int32_t* nmoves,
               int32_t* pos, int64_t* gain_sum, int32_t* order, int64_t* paths, void* stream) {
  if (!ctx || !dg || !dg->adjwgt || !dg->vwgt || !part || !bnd || !gain || !dest || !pw || !gain_sum ||
      k < 1 || k > kMaxK || max_moves < 1 || max_moves > 1024 || nrounds < 0) {
    gkh::set_error("bad argument");
    return GK_ERR_ARG;
  }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  *gain_sum = 0;
  if (paths) paths[0] = paths[1] = paths[2] = 0;
  DGraph g = dview(dg);
  if (g.n <= 0 || nrounds == 0) {
    for (int32_t r = 0; r < nrounds; ++r) {
      if (nmoves) nmoves[r] = 0;
      if (pos) pos[r] = -1;
    }
    return GK_OK;
  }
  Pool& P = ctx->pool;
  const int32_t n = g.n, M = max_moves;
  const int64_t nwords = (int64_t(n) + 63) / 64;
  // The round state of run_vcycle's refinement, for one job.
  Buf<int32_t> movers, upd, wl, heavy, list, xlist, wpos, sscr, dorder, dmax, hist;
  Buf<char> state;
  Buf<uint64_t> cand, movable, selbits, defbits;
  Buf<uint32_t> hkey;
  GK_TRY(upd.alloc(P, n));
  GK_TRY(wl.alloc(P, n));
  GK_TRY(heavy.alloc(P, n));
  // The round loop orders all of a round's moves when a caller wants to see
  // them, and else only as many as decide the round.
  const bool want_hist = nmoves || pos;
  if (want_hist) GK_TRY(hist.alloc(P, 2 * int64_t(nrounds)));
  GK_TRY(list.alloc(P, n));
  GK_TRY(xlist.alloc(P, n));
  GK_TRY(hkey.alloc(P, n));
  GK_TRY(wpos.alloc(P, nwords + 1));
  GK_TRY(sscr.alloc(P, gkd::select_scratch_ints(n)));
  GK_TRY(cand.alloc(P, nwords + 1));
  GK_TRY(movable.alloc(P, nwords + 1));
  GK_TRY(selbits.alloc(P, nwords + 1));
  GK_TRY(defbits.alloc(P, nwords + 1));
  GK_TRY(movers.alloc(P, int64_t(M) + 1));
  if (order) GK_TRY(dorder.alloc(P, int64_t(M) + 2));
  GK_TRY(dmax.alloc(P, 1));
  // The words of the one job's state, which go up and come back as one block.
  struct State {
    long long cut, cap, moved, abytes, paths[3], pad;
    int32_t voff[2], pwoff[2], hcnt[4], status[4], kk, thr, lastcnt, rounds, active, pad2[3];
  };
  static_assert(sizeof(State) % 16 == 0, "whole 16-byte words");
  GK_TRY(state.alloc(P, sizeof(State)));
  State* ds = reinterpret_cast<State*>(state.p);
  HostBlock hist_down;
  StageGuard staged{ctx, st};
  void* hup = nullptr;
  GK_TRY(ctx->up.get(st, sizeof(State), &hup));
  State* hs = static_cast<State*>(hup);
  std::memset(hs, 0, sizeof *hs);
  hs->cap = cap;
  hs->voff[1] = n;
  hs->pwoff[1] = k;
  hs->kk = k;
  hs->thr = 1;
  hs->lastcnt = 1;
  gkd::Copies begin;
  begin.add(ds, hs, sizeof *hs);
  begin.add(upd.p, nullptr, sizeof(int32_t) * size_t(n));
  begin.add(selbits.p, nullptr, sizeof(uint64_t) * size_t(nwords + 1));
  GK_TRY(gkd::launch_copies(begin, st));
  GK_TRY(gkd::launch_cand_init(n, bnd, gain, cand.p, st));
  RoundState rs;
  rs.g = g;
  rs.kmax = k;
  rs.M = M;
  rs.lanes = gain_lanes(g);
  if (gkd::gain_heavy_separate(k)) {
    GK_TRY(gkd::launch_max_deg(g, dmax.p, st));
    int32_t maxdeg = 0;
    GK_TRY(fetch(ctx, st, {{&maxdeg, dmax.p, sizeof maxdeg}}));
    rs.heavy_rows = maxdeg > rs.lanes;
  }
  rs.wl_items = n;
  rs.v_off = ds->voff;
  rs.kk = &ds->kk;
  rs.pw_off = ds->pwoff;
  rs.cap = &ds->cap;
  rs.part = part;
  rs.bnd = bnd;
  rs.gain = gain;
  rs.dest = dest;
  rs.pw = pw;
  rs.upd = upd.p;
  rs.cut = &ds->cut;
  rs.moved = &ds->moved;
  rs.paths = ds->paths;
  rs.abytes = &ds->abytes;
  rs.rounds = &ds->rounds;
  rs.lastcnt = &ds->lastcnt;
  rs.thr = &ds->thr;
  rs.active = &ds->active;
  rs.cand = cand.p;
  rs.sb = gkd::SelectBufs{movable.p, selbits.p, defbits.p, wpos.p, list.p, sscr.p, nullptr};
  rs.xlist = xlist.p;
  rs.movers = movers.p;
  rs.wl = wl.p;
  rs.hcnt = ds->hcnt;
  rs.heavy = heavy.p;
  rs.status = ds->status;
  rs.hkey = hkey.p;
  rs.order = dorder.p;
  rs.hist = hist.p;
  GK_TRY(refine_rounds(ctx, st, rs, nrounds, true, false, nullptr));
  // Rounds that ordered no move came after those that did (an unchanged state
  // stays so): no moves, position -1.
  const size_t hist_bytes = want_hist ? sizeof(int32_t) * 2 * size_t(nrounds) : 0;
  GK_TRY(hist_down.get(ctx->dl, st, hist_bytes, sizeof(State)));
  void* hend = hist_down.head();
  const State* he = static_cast<const State*>(hend);
  const int32_t* hh = static_cast<const int32_t*>(hist_down.p());
  gkd::Copies end;
  end.add(hend, ds, sizeof *ds);
  GK_TRY(hist_down.copy(end, st, hist_down.p(), hist.p, hist_bytes, hipMemcpyDeviceToHost));
  GK_TRY(gkd::launch_copies(end, st));
  GK_HIP(hipStreamSynchronize(st));
  staged.done = true;
  const int32_t made = he->rounds;
  for (int32_t r = 0; r < nrounds; ++r) {
    if (nmoves) nmoves[r] = r < made ? hh[2 * r] : 0;
    if (pos) pos[r] = r < made ? hh[2 * r + 1] : -1;
  }
  if (order && made > 0) {
    int32_t ordered = 0;
    GK_TRY(fetch(ctx, st, {{&ordered, dorder.p, sizeof ordered}}));
    GK_HIP(hipMemcpyAsync(order, dorder.p + 2, sizeof(int32_t) * size_t(ordered), hipMemcpyDeviceToDevice, st));
  }
  GK_HIP(hipStreamSynchronize(st));
  *gain_sum = -he->cut;
  if (paths)
    for (int i = 0; i < 3; ++i) paths[i] = he->paths[i];
  return GK_OK;
}

int gk_k_cut(gk_ctx* ctx, const gk_csr* dg, int32_t k, const int32_t* part, int64_t* cut, int64_t* pw,
             void* stream) {
  if (!ctx || !dg || !dg->adjwgt || !dg->vwgt || !cut || k < 1) { gkh::set_error("bad argument"); return GK_ERR_ARG; }
  if (k > gkd::kCutMaxK) {
    gkh::set_error("k = " + std::to_string(k) + " exceeds " + std::to_string(gkd::kCutMaxK) +
                   ", the part weights that fit a compute unit's LDS");
    return GK_ERR_LIMIT;
  }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  DGraph g = dview(dg);
  Buf<unsigned long long> c, p, cscr;
  GK_TRY(c.alloc(ctx->pool, 1));
  GK_TRY(p.alloc(ctx->pool, k));
  GK_TRY(cscr.alloc(ctx->pool, gkd::cut_scratch(g.n, k)));
  StageGuard drain{ctx, st};
  GK_TRY(gkd::launch_cut(g, k, part, c.p, p.p, cscr.p, st));
  void* h = nullptr;
  GK_TRY(ctx->dl.get(st, sizeof(unsigned long long) * (size_t(k) + 2), &h));
  unsigned long long* hc = static_cast<unsigned long long*>(h);
  gkd::Copies back;
  back.add(hc, c.p, sizeof *hc);
  if (pw) back.add(hc + 2, p.p, sizeof *hc * size_t(k));
  GK_TRY(gkd::launch_copies(back, st));
  GK_HIP(hipStreamSynchronize(st));
  drain.done = true;
  *cut = static_cast<int64_t>(*hc);
  if (pw)
    for (int32_t q = 0; q < k; ++q) pw[q] = static_cast<int64_t>(hc[2 + q]);
  return GK_OK;
}

int gk_k_cut_noalloc(gk_ctx* ctx, const gk_csr* dg, int32_t k, const int32_t* part, int64_t* dev_cut,
                     int64_t* dev_pw, void* stream) {
  if (!ctx || !dg || !dg->adjwgt || !dg->vwgt || !dev_cut || !dev_pw || k < 1 || dg->n < 0 ||
      (dg->n > 0 && (!part || !dg->xadj || !dg->adjncy))) {
    gkh::set_error("bad argument");
    return GK_ERR_ARG;
  }
  if (k > kMaxK) {
    gkh::set_error("k = " + std::to_string(k) + " exceeds " + std::to_string(kMaxK) +
                   ", the largest k of the no-allocation cut (its scratch holds 2^18 slots)");
    return GK_ERR_LIMIT;
  }
  unsigned long long* scr = scratch_addr(ctx->device);
  if (!scr) { gkh::set_error("no scratch address for this device"); return GK_ERR_INTERNAL; }
  DeviceGuard guard(ctx->device);
  hipStream_t st = pick(ctx, stream);
  const int rc = gkd::launch_cut(dview(dg), k, part, reinterpret_cast<unsigned long long*>(dev_cut),
                                 reinterpret_cast<unsigned long long*>(dev_pw), scr, st, kCutScratchSlots);
  if (rc != GK_OK) gkh::set_error("cut launch failed");
  return rc;
}

}  // extern "C"
