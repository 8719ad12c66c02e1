// Coarsest-level initial partitioner (host C++).
//
// The reference hands its coarsest graph to METIS_PartGraphKway
// (gkway/metis_partition.hpp:46-47).  The METIS it uses exists only as a
// prebuilt binary, so this library supplies its own deterministic
// partitioner for that step:
//   multilevel recursive bisection
//     - coarsening by sequential heavy-edge matching in a seeded random order,
//     - initial bisection by greedy graph growing from several seeds,
//     - 2-way Fiduccia-Mattheyses refinement at every level,
//   followed by a k-way greedy boundary pass that repairs any part above the
//   cap and takes positive-gain moves.
// Every random choice comes from a SplitMix64 stream seeded by (seed, depth,
// first part id), so the output depends only on the input graph, k, cap and
// seed -- never on the number of threads.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <deque>
#include <functional>
#include <memory>
#include <mutex>
#include <numeric>
#include <thread>
#include <vector>

#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include "../../include/gkway.h"
#include "host_graph.hpp"

#ifndef GKIP_NCUTS0
#define GKIP_NCUTS0 4
#endif
#ifndef GKIP_NCUTS1
#define GKIP_NCUTS1 3
#endif
#ifndef GKIP_NCUTS2
#define GKIP_NCUTS2 2
#endif
#ifndef GKIP_FMPASS
#define GKIP_FMPASS 6
#endif
#ifndef GKIP_TRIALS
#define GKIP_TRIALS 8
#endif
#ifndef GKIP_SPAWN_MIN
#define GKIP_SPAWN_MIN 200  // smallest subgraph whose trials / halves become pool tasks
#endif

namespace {

struct Rng {
  uint64_t s;
  explicit Rng(uint64_t seed) : s(seed) {}
  uint64_t next() {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  }
  uint32_t below(uint32_t m) { return static_cast<uint32_t>((static_cast<uint64_t>(next() >> 32) * m) >> 32); }
};

// ------------------------------------------------------------------ memory
// Per-thread stack of memory for the graphs and work arrays of a bisection:
// they are made and dropped in last-in first-out order (a task that a waiting
// thread runs meanwhile begins and ends above what the waiter holds), so
// nothing is zeroed, returned to the system or faulted in again between
// levels and trials.
class Arena {
 public:
  static Arena& get() {
    thread_local Arena a;
    return a;
  }
  template <class T>
  T* take(size_t count) {
    const size_t bytes = (count * sizeof(T) + 63) & ~size_t(63);
    while (cur_ < blocks_.size() && used_ + bytes > blocks_[cur_].size) {
      ++cur_;
      used_ = 0;
    }
    if (cur_ == blocks_.size()) {
      const size_t size = std::max(bytes, std::max<size_t>(size_t(1) << 20, 2 * (blocks_.empty() ? 0 : blocks_.back().size)));
      blocks_.push_back({std::unique_ptr<char[]>(new char[size + 64]), size});
    }
    char* base = blocks_[cur_].mem.get();
    char* p = base + ((64 - (reinterpret_cast<uintptr_t>(base) & 63)) & 63) + used_;
    used_ += bytes;
    return reinterpret_cast<T*>(p);
  }
  // Gives back the end of the latest take: it keeps `count` elements at p.
  template <class T>
  void keep(T* p, size_t count) {
    char* base = blocks_[cur_].mem.get();
    base += (64 - (reinterpret_cast<uintptr_t>(base) & 63)) & 63;
    used_ = static_cast<size_t>(reinterpret_cast<char*>(p) - base) + ((count * sizeof(T) + 63) & ~size_t(63));
  }
  // Everything taken while a Scope lives is dropped with it.  A thread keeps
  // at most kIdle bytes between its outermost scopes.
  class Scope {
   public:
    Scope() : a_(Arena::get()), cur_(a_.cur_), used_(a_.used_) { ++a_.depth_; }
    ~Scope() {
      a_.cur_ = cur_;
      a_.used_ = used_;
      if (--a_.depth_ == 0) a_.trim();
    }
    Scope(const Scope&) = delete;
    Scope& operator=(const Scope&) = delete;

   private:
    Arena& a_;
    size_t cur_, used_;
  };

 private:
  static constexpr size_t kIdle = size_t(32) << 20;
  struct Block {
    std::unique_ptr<char[]> mem;
    size_t size;
  };
  void trim() {
    size_t total = 0;
    for (const Block& b : blocks_) total += b.size;
    if (total > kIdle) blocks_.clear();
    cur_ = 0;
    used_ = 0;
  }
  std::vector<Block> blocks_;
  size_t cur_ = 0, used_ = 0;
  int depth_ = 0;
};

struct Edge {
  int32_t u, w;
};

// A vertex: its row is the edges [lo, hi), inc their summed weight.
struct V {
  int32_t lo, hi, vw, inc;
};

// A graph in arena memory.
struct G {
  int32_t n = 0;
  V* v = nullptr;
  Edge* e = nullptr;
  int64_t tw = 0;    // total vertex weight
  int64_t rows = 0;  // entries of all rows
};

// ------------------------------------------------------------------ heap
// State of a vertex in a two-way refinement: weight to its own side and to
// the other, place in its side's queue (-1: not queued), side, and whether it
// has moved in this pass or been listed as a boundary vertex.  One record, so
// that an update of a neighbour touches one cache line.
struct FV {
  int32_t id, ed, pos;
  uint8_t side, locked, listed, pad;
};

// Indexed binary max-heap of vertices ordered by (gain desc, vertex asc).
// Both go into one 64-bit key: the gain in the high 32 bits (a gain is
// bounded by a vertex's weighted degree, below 2^31) and the complemented
// vertex id in the low 32, so one integer compare orders two entries.  Keys
// are distinct, so the order in which vertices leave the heap depends on the
// keys alone, never on the heap's layout: building it in O(n) by sift-down
// gives the same sequence as n pushes.  Places are kept in the vertex records.
class Heap {
 public:
  static int64_t pack(int32_t g, int32_t v) {
    return static_cast<int64_t>(static_cast<uint64_t>(static_cast<int64_t>(g)) << 32) |
           int64_t(0xFFFFFFFFu - static_cast<uint32_t>(v));
  }
  static int32_t vertex(int64_t key) { return static_cast<int32_t>(0xFFFFFFFFu - static_cast<uint32_t>(key)); }
  void use(FV* fv) { fv_ = fv; }
  // Empties the heap, clearing the places of what is still queued.
  void drop() {
    for (int64_t k : h_) fv_[vertex(k)].pos = -1;
    h_.clear();
  }
  std::vector<int64_t>& keys() { return h_; }  // filled by the caller while empty, then heapify()
  void heapify() {
    const int32_t n = static_cast<int32_t>(h_.size());
    for (int32_t i = n / 2 - 1; i >= 0; --i) sift_down(i);
    for (int32_t i = 0; i < n; ++i) fv_[vertex(h_[i])].pos = i;
  }
  bool empty() const { return h_.empty(); }
  int32_t top() const { return vertex(h_[0]); }
  int64_t top_key() const { return h_[0] >> 32; }  // the gain of the top vertex
  void push(int32_t v, int32_t g) {
    const int32_t i = static_cast<int32_t>(h_.size());
    h_.push_back(0);
    up(i, pack(g, v));
  }
  void update(int32_t v, int32_t g) {
    const int32_t i = fv_[v].pos;
    const int64_t k = pack(g, v);
    if (k > h_[i]) up(i, k); else down(i, k);
  }
  void remove(int32_t v) {
    const int32_t i = fv_[v].pos;
    fv_[v].pos = -1;
    const int64_t old = h_[i], last = h_.back();
    h_.pop_back();
    if (i == static_cast<int32_t>(h_.size())) return;
    if (last > old) up(i, last); else down(i, last);
  }

 private:
  void up(int32_t i, int64_t k) {
    while (i > 0) {
      const int32_t p = (i - 1) / 2;
      if (h_[p] >= k) break;
      h_[i] = h_[p];
      fv_[vertex(h_[i])].pos = i;
      i = p;
    }
    h_[i] = k;
    fv_[vertex(k)].pos = i;
  }
  void down(int32_t i, int64_t k) {
    const int32_t n = static_cast<int32_t>(h_.size());
    while (true) {
      int32_t c = 2 * i + 1;
      if (c >= n) break;
      if (c + 1 < n) c += h_[c + 1] > h_[c];
      if (h_[c] <= k) break;
      h_[i] = h_[c];
      fv_[vertex(h_[i])].pos = i;
      i = c;
    }
    h_[i] = k;
    fv_[vertex(k)].pos = i;
  }
  // down() without place updates, for heapify().
  void sift_down(int32_t i) {
    const int32_t n = static_cast<int32_t>(h_.size());
    const int64_t k = h_[i];
    while (true) {
      int32_t c = 2 * i + 1;
      if (c >= n) break;
      if (c + 1 < n) c += h_[c + 1] > h_[c];
      if (h_[c] <= k) break;
      h_[i] = h_[c];
      i = c;
    }
    h_[i] = k;
  }
  std::vector<int64_t> h_;
  FV* fv_ = nullptr;
};

// ------------------------------------------------------------------ fork-join
// Process-wide worker threads for the independent pieces of the recursive
// bisection (the trial bisections of a node and the two halves below it).
// A thread waiting for a task that nobody has begun runs it itself; it takes
// no other task meanwhile, which could hold it up long after its own is done
// (a 7 ms stall of a node's halves was seen).  Every queued task is so run by
// its waiter or by a worker.  Threads look for a short while before they
// sleep: tasks follow each other closely, and a wake-up takes longer than
// many of them.  Results never depend on which thread runs a task.
class ForkJoin {
 public:
  struct Task {
    std::function<void()> fn;
    std::atomic<int> state{0};  // 0 queued, 1 running, 2 done
  };
  static ForkJoin& get() {
    static ForkJoin pool;
    return pool;
  }
  int workers() const { return static_cast<int>(th_.size()); }
  std::shared_ptr<Task> spawn(std::function<void()> fn) {
    auto t = std::make_shared<Task>();
    t->fn = std::move(fn);
    bool wake;
    {
      std::lock_guard<std::mutex> lk(m_);
      q_.push_back(t);
      queued_.store(static_cast<int>(q_.size()));
      wake = idle_ > 0;
    }
    if (wake) cv_.notify_one();
    return t;
  }
  void wait(const std::shared_ptr<Task>& t) {
    int queued = 0;
    if (t->state.compare_exchange_strong(queued, 1)) {
      run(*t);
      return;
    }
    for (int i = 0; i < kSpin; ++i) {
      if (t->state.load() == 2) return;
      relax();
    }
    std::unique_lock<std::mutex> lk(m_);
    ++waiters_;
    done_cv_.wait(lk, [&] { return t->state.load() == 2; });
    --waiters_;
  }

 private:
  static constexpr int kSpin = 4000;
  static void relax() {
#if defined(__x86_64__)
    __builtin_ia32_pause();
#endif
  }
  ForkJoin() {
    const unsigned hw = std::thread::hardware_concurrency();
    const int n = static_cast<int>(hw ? std::min(hw, 16u) : 1u) - 1;
    for (int i = 0; i < n; ++i)
      th_.emplace_back([this] {
        while (true) {
          for (int s = 0; s < kSpin && queued_.load() == 0; ++s) relax();
          std::shared_ptr<Task> t;
          {
            std::unique_lock<std::mutex> lk(m_);
            ++idle_;
            cv_.wait(lk, [this] { return stop_ || !q_.empty(); });
            --idle_;
            if (stop_ && q_.empty()) return;
            t = std::move(q_.front());
            q_.pop_front();
            queued_.store(static_cast<int>(q_.size()));
          }
          int queued = 0;
          if (t->state.compare_exchange_strong(queued, 1)) run(*t);
        }
      });
  }
  ~ForkJoin() {
    {
      std::lock_guard<std::mutex> lk(m_);
      stop_ = true;
    }
    cv_.notify_all();
    for (auto& t : th_) t.join();
  }
  void run(Task& t) {
    t.fn();
    t.state.store(2);
    if (waiters_.load() > 0) {
      std::lock_guard<std::mutex> lk(m_);
      done_cv_.notify_all();
    }
  }
  std::vector<std::thread> th_;
  std::deque<std::shared_ptr<Task>> q_;
  std::mutex m_;
  std::condition_variable cv_, done_cv_;
  std::atomic<int> queued_{0}, waiters_{0};
  int idle_ = 0;  // guarded by m_
  bool stop_ = false;
};

// Runs fn(c) for c in [0, chunks): chunk 0 on the calling thread, the others
// as pool tasks (the caller may itself be a pool task).
template <class F>
void par_chunks(int chunks, const F& fn) {
  if (chunks <= 1) {
    if (chunks == 1) fn(0);
    return;
  }
  std::vector<std::shared_ptr<ForkJoin::Task>> ts;
  for (int c = 1; c < chunks; ++c) ts.push_back(ForkJoin::get().spawn([&fn, c] { fn(c); }));
  fn(0);
  for (auto& t : ts) ForkJoin::get().wait(t);
}

// ------------------------------------------------------------------ coarsening
// The rows of coarse vertices [lo, hi): coarse vertex cv is first reached at
// its smaller member v (v <= match[v]); its row lists the neighbours of v,
// then of match[v], in order of first appearance, weights summed.  out holds
// the rows from index `top` on, and one entry more at index trash, where edges
// between the two members go; slot: c.n ints, all -1.  Returns the end.
int32_t coarse_rows(const G& g, const int32_t* match, const int32_t* cmap, int32_t v0, int32_t v1, G& c, int32_t top,
                    int32_t trash, int32_t* slot) {
  Edge* out = c.e;
  for (int32_t v = v0; v < v1; ++v) {
    const int32_t m = match[v];
    // the partners' rows lie anywhere: fetched some vertices ahead
    if (v + 8 < v1) __builtin_prefetch(&g.v[match[v + 8]]);
    if (v + 4 < v1) __builtin_prefetch(&g.e[g.v[match[v + 4]].lo]);
    if (m < v) continue;  // second member: taken with the first
    const int32_t cv = cmap[v];
    const int32_t start = top;
    out[trash].w = 0;
    slot[cv] = trash;
    int32_t x = v;
    while (true) {
      for (int32_t j = g.v[x].lo; j < g.v[x].hi; ++j) {
        const int32_t cu = cmap[g.e[j].u];
        const int32_t s = slot[cu];
        const bool seen = s >= start;
        const int32_t at = seen ? s : top;
        slot[cu] = at;
        out[at].u = cu;
        out[at].w = (seen ? out[at].w : 0) + g.e[j].w;
        top += !seen;
      }
      if (x == m) break;
      x = m;
    }
    slot[cv] = -1;
    c.v[cv] = V{start, top, g.v[v].vw + (m != v ? g.v[m].vw : 0), g.v[v].inc + (m != v ? g.v[m].inc : 0) - out[trash].w};
  }
  return top;
}

// Heavy-edge matching in a seeded random visiting order.  Ties between equal
// edge weights go to the lighter neighbour, then the lower id.  cmap (n, in
// the arena) gets the coarse id of every vertex; returns the coarse graph.
G coarsen_hem(const G& g, Rng& rng, int64_t maxvw, int32_t* cmap, bool par) {
  const int32_t n = g.n;
  Arena& A = Arena::get();
  // The coarse graph comes first in the arena, its arrays sized for n, so that
  // the work arrays behind it can be dropped.
  G c;
  c.v = A.take<V>(n);
  c.tw = g.tw;
  c.e = A.take<Edge>(static_cast<size_t>(g.rows) + 1);
  int64_t end = 0;  // entries of c.e in use
  {
    Arena::Scope work;
    int32_t* perm = A.take<int32_t>(n);
    int32_t* match = A.take<int32_t>(n);
    // what the matching asks of a neighbour: matched already, and its weight
    struct Free {
      int32_t matched, vw;
    };
    Free* fr = A.take<Free>(n);
    std::iota(perm, perm + n, 0);
    for (int32_t i = n - 1; i > 0; --i) std::swap(perm[i], perm[rng.below(static_cast<uint32_t>(i + 1))]);
    for (int32_t v = 0; v < n; ++v) fr[v] = Free{0, g.v[v].vw};
    for (int32_t i = 0; i < n; ++i) {
      const int32_t v = perm[i];
      // the visits jump: vertices and rows are fetched some visits ahead
      if (i + 16 < n) __builtin_prefetch(&g.v[perm[i + 16]]);
      if (i + 8 < n) __builtin_prefetch(&g.e[g.v[perm[i + 8]].lo]);
      if (fr[v].matched) continue;
      int32_t best = v;  // alone, if nothing fits
      int32_t bw = INT32_MIN, bvw = 0;
      const V me = g.v[v];
      const int64_t room = maxvw - me.vw;
      for (int32_t j = me.lo; j < me.hi; ++j) {
        const int32_t u = g.e[j].u, w = g.e[j].w;
        if (w < bw) continue;
        const Free f = fr[u];
        if (f.matched || f.vw > room) continue;
        if (w > bw || f.vw < bvw || (f.vw == bvw && u < best)) {
          best = u;
          bw = w;
          bvw = f.vw;
        }
      }
      fr[v].matched = 1;
      fr[best].matched = 1;
      match[v] = best;
      match[best] = v;
    }
    int32_t nc = 0;
    for (int32_t v = 0; v < n; ++v)
      if (match[v] >= v) cmap[v] = nc++; else cmap[v] = cmap[match[v]];
    c.n = nc;
    const int chunks = par ? static_cast<int>(std::min<int64_t>(8, g.rows / 32768)) : 1;
    if (chunks > 1) {
      // Rows are independent: vertex ranges are taken by pool threads, each
      // into the entries that its rows could fill at most (a range's rows read
      // the rows of its own vertices and of their partners behind them).
      std::vector<int32_t> first(chunks + 1), at(chunks + 1, 0), tops(chunks);
      for (int i = 0; i <= chunks; ++i) first[i] = static_cast<int32_t>(int64_t(n) * i / chunks);
      for (int i = 0; i < chunks; ++i) {
        int32_t ub = 0;
        for (int32_t v = first[i]; v < first[i + 1]; ++v) {
          const int32_t m = match[v];
          if (m < v) continue;
          ub += g.v[v].hi - g.v[v].lo + (m != v ? g.v[m].hi - g.v[m].lo : 0);
        }
        at[i + 1] = at[i] + ub;
      }
      // every range's trash entry in an array of its own behind the rows: the
      // ranges' rows and trash must be indexes of one array
      Edge* wide = A.take<Edge>(static_cast<size_t>(g.rows) + chunks);
      G cw = c;
      cw.e = wide;
      par_chunks(chunks, [&](int i) {
        Arena::Scope own;
        int32_t* slot = Arena::get().take<int32_t>(nc);
        std::fill(slot, slot + nc, -1);
        tops[i] = coarse_rows(g, match, cmap, first[i], first[i + 1], cw, at[i], static_cast<int32_t>(g.rows) + i, slot);
      });
      // together, without the gaps
      par_chunks(chunks, [&](int i) {
        int64_t to = 0;
        for (int q = 0; q < i; ++q) to += tops[q] - at[q];
        std::copy(wide + at[i], wide + tops[i], c.e + to);
        const int32_t shift = static_cast<int32_t>(to) - at[i];
        for (int32_t v = first[i]; v < first[i + 1]; ++v)
          if (match[v] >= v) {
            c.v[cmap[v]].lo += shift;
            c.v[cmap[v]].hi += shift;
          }
      });
      for (int q = 0; q < chunks; ++q) end += tops[q] - at[q];
    } else {
      int32_t* slot = A.take<int32_t>(nc);
      std::fill(slot, slot + nc, -1);
      end = coarse_rows(g, match, cmap, 0, n, c, 0, static_cast<int32_t>(g.rows), slot);
    }
  }
  A.keep(c.e, static_cast<size_t>(end));
  c.rows = end;
  return c;
}

// ------------------------------------------------------------------ 2-way FM
struct Bal {
  int64_t max[2];
};

inline int64_t overload(const int64_t pw[2], const Bal& b) {
  return std::max<int64_t>(0, pw[0] - b.max[0]) + std::max<int64_t>(0, pw[1] - b.max[1]);
}

// Buffers of fm2, one set per thread (fm2 never waits on the pool, so no
// other fm2 call can run on its thread while it holds them).
struct FmWork {
  std::vector<int32_t> moved, list;
  Heap q[2];
};

// Boundary FM refinement.  Moves that keep both sides within their maxima
// (or reduce the overload) are taken in max-gain order; the best prefix of a
// pass (lowest (overload, cut)) is kept.  fv holds every vertex's side and
// degrees (exact on entry, kept exact through the moves of a pass and their
// rollback), pos -1, locked and listed 0; pw the sides' weights.
void fm2(const G& g, FV* fv, int64_t pw[2], const Bal& bal, int passes, int64_t& cut) {
  const int32_t n = g.n;
  thread_local FmWork W;
  Heap* q = W.q;
  q[0].use(fv);
  q[1].use(fv);
  std::vector<int32_t>& moved = W.moved;
  // Vertices that are or were on the boundary: what a pass starts from.
  std::vector<int32_t>& list = W.list;
  list.clear();
  for (int32_t v = 0; v < n; ++v)
    if (fv[v].ed > 0) {
      fv[v].listed = 1;
      list.push_back(v);
    }
  const int32_t limit = std::max<int32_t>(25, std::min<int32_t>(n / 20, 300));
  for (int pass = 0; pass < passes; ++pass) {
    for (int32_t v : list)
      if (fv[v].ed > 0) q[fv[v].side].keys().push_back(Heap::pack(fv[v].ed - fv[v].id, v));
    q[0].heapify();
    q[1].heapify();
    moved.clear();
    int64_t cur_cut = cut, best_cut = cut;
    int64_t best_ol = overload(pw, bal);
    int32_t best_len = 0, since_best = 0;
    int64_t cur_pw[2] = {pw[0], pw[1]};
    while (true) {
      // Pick the source side: an overloaded side must shed weight; otherwise
      // take the better top among moves that keep the target within bounds.
      int from = -1;
      const bool ol0 = cur_pw[0] > bal.max[0], ol1 = cur_pw[1] > bal.max[1];
      if (ol0 && !q[0].empty()) from = 0;
      else if (ol1 && !q[1].empty()) from = 1;
      else {
        int64_t bg = INT64_MIN;
        for (int s = 0; s < 2; ++s) {
          if (q[s].empty()) continue;
          int32_t v = q[s].top();
          if (cur_pw[1 - s] + g.v[v].vw > bal.max[1 - s]) continue;
          if (q[s].top_key() > bg) { bg = q[s].top_key(); from = s; }
        }
      }
      if (from < 0) break;
      int32_t v = q[from].top();
      q[from].remove(v);
      const int to = 1 - from;
      if (!(ol0 || ol1) && cur_pw[to] + g.v[v].vw > bal.max[to]) continue;
      FV& f = fv[v];
      cur_cut -= f.ed - f.id;
      cur_pw[from] -= g.v[v].vw;
      cur_pw[to] += g.v[v].vw;
      f.side = static_cast<uint8_t>(to);
      f.locked = 1;
      std::swap(f.id, f.ed);
      moved.push_back(v);
      for (int32_t j = g.v[v].lo; j < g.v[v].hi; ++j) {
        const int32_t u = g.e[j].u;
        FV& x = fv[u];
        const int32_t w = x.side == to ? g.e[j].w : -g.e[j].w;
        x.id += w;
        x.ed -= w;
        if (x.locked) continue;
        if (x.pos >= 0) {
          if (x.ed > 0) q[x.side].update(u, x.ed - x.id); else q[x.side].remove(u);
        } else if (x.ed > 0) {
          q[x.side].push(u, x.ed - x.id);
          if (!x.listed) {
            x.listed = 1;
            list.push_back(u);
          }
        }
      }
      // a mover that was interior cannot be: it came from a queue, so listed
      int64_t ol = overload(cur_pw, bal);
      if (ol < best_ol || (ol == best_ol && cur_cut < best_cut)) {
        best_ol = ol;
        best_cut = cur_cut;
        best_len = static_cast<int32_t>(moved.size());
        since_best = 0;
      } else if (++since_best > limit) {
        break;
      }
    }
    // Roll back past the best prefix, newest first, undoing each move's
    // degree updates.
    for (int32_t i = static_cast<int32_t>(moved.size()) - 1; i >= best_len; --i) {
      const int32_t v = moved[i];
      FV& f = fv[v];
      const int to = f.side, from = 1 - to;
      for (int32_t j = g.v[v].lo; j < g.v[v].hi; ++j) {
        FV& x = fv[g.e[j].u];
        const int32_t w = x.side == to ? g.e[j].w : -g.e[j].w;
        x.id -= w;
        x.ed += w;
      }
      std::swap(f.id, f.ed);
      f.side = static_cast<uint8_t>(from);
      cur_pw[to] -= g.v[v].vw;
      cur_pw[from] += g.v[v].vw;
    }
    for (int32_t v : moved) fv[v].locked = 0;
    q[0].drop();
    q[1].drop();
    pw[0] = cur_pw[0];
    pw[1] = cur_pw[1];
    bool improved = best_cut < cut || best_len > 0;
    cut = best_cut;
    if (!improved || best_len == 0) break;
  }
}

// First index of the largest of a[0, n), n a multiple of 8.
int32_t first_max(const int32_t* a, int32_t n) {
  int32_t at = 0;
  for (int32_t i = 1; i < n; ++i)
    if (a[i] > a[at]) at = i;
  return at;
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) int32_t first_max_avx2(const int32_t* a, int32_t n) {
  __m256i m = _mm256_loadu_si256(reinterpret_cast<const __m256i*>(a));
  for (int32_t i = 8; i < n; i += 8) m = _mm256_max_epi32(m, _mm256_loadu_si256(reinterpret_cast<const __m256i*>(a + i)));
  __m128i h = _mm_max_epi32(_mm256_castsi256_si128(m), _mm256_extracti128_si256(m, 1));
  h = _mm_max_epi32(h, _mm_shuffle_epi32(h, 0x4E));
  h = _mm_max_epi32(h, _mm_shuffle_epi32(h, 0xB1));
  const __m256i x = _mm256_broadcastd_epi32(h);
  for (int32_t i = 0;; i += 8) {
    const int b = _mm256_movemask_ps(
        _mm256_castsi256_ps(_mm256_cmpeq_epi32(x, _mm256_loadu_si256(reinterpret_cast<const __m256i*>(a + i)))));
    if (b) return i + __builtin_ctz(static_cast<unsigned>(b));
  }
}
const auto kFirstMax = __builtin_cpu_supports("avx2") ? first_max_avx2 : first_max;
#else
const auto kFirstMax = first_max;
#endif

// Growing takes the best vertex by a scan of all gains instead of from a heap
// on graphs of up to kFlatMax vertices with kFlatDegree entries a row or more:
// the coarsest graphs have about 60 to 120 vertices, and one vector scan costs
// less than a heap's pop and the key changes of a row (64 coarsest graphs of a
// batch: growing 25% -> 15% of the time).  On road networks, with two entries
// a row, the heap holds a handful of vertices and stays cheaper.
constexpr int32_t kFlatMax = 256;
constexpr int32_t kFlatDegree = 4;

// Greedy graph growing from `seedv`: side 0 grows by max gain (then lowest
// id) until it reaches its target weight.  Leaves side and degrees of every
// vertex in fv and the sides' weights in pw; returns the cut of the result
// (each added vertex turns its edges to side 0 internal and the rest cut).
int64_t grow(const G& g, FV* fv, int32_t seedv, int64_t target0, int64_t pw[2]) {
  const int32_t n = g.n;
  const bool flat = n <= kFlatMax && g.rows >= int64_t(kFlatDegree) * n;
  thread_local Heap q;  // growing never waits on the pool
  q.use(fv);
  // While growing, id is the vertex's weight to side 0; gains[v] (flat) the
  // gain of a side-1 vertex next to side 0, kNone for the others.
  constexpr int32_t kNone = INT32_MIN;
  int32_t gains[kFlatMax];
  const int32_t n8 = (n + 7) & ~7;
  if (flat) std::fill(gains, gains + n8, kNone);
  for (int32_t v = 0; v < n; ++v) fv[v] = FV{0, 0, -1, 1, 0, 0, 0};
  int64_t w0 = 0, cut = 0;
  int32_t next_unreached = 0;
  auto add = [&](int32_t v) {
    fv[v].side = 0;
    const V me = g.v[v];
    w0 += me.vw;
    cut += me.inc - 2 * int64_t(fv[v].id);
    for (int32_t j = me.lo; j < me.hi; ++j) {
      const int32_t u = g.e[j].u;
      FV& x = fv[u];
      x.id += g.e[j].w;
      // gain of moving u to side 0: 2 * its weight to side 0 - its weight
      const int32_t gain = static_cast<int32_t>(2 * int64_t(x.id) - g.v[u].inc);
      if (flat) gains[u] = x.side != 0 ? gain : kNone;
      else if (x.side == 0) continue;
      else if (x.pos >= 0) q.update(u, gain);
      else q.push(u, gain);
    }
  };
  add(seedv);
  while (w0 < target0) {
    int32_t v = -1;
    if (flat) {
      v = kFirstMax(gains, n8);
      if (gains[v] == kNone) v = -1;
      else gains[v] = kNone;
    } else if (!q.empty()) {
      v = q.top();
      q.remove(v);
    }
    if (v < 0) {
      while (next_unreached < n && fv[next_unreached].side == 0) ++next_unreached;
      if (next_unreached >= n) break;
      v = next_unreached;
    }
    // Stop before overshooting by more than half the vertex weight.
    if (w0 + g.v[v].vw > target0 && (w0 + g.v[v].vw - target0) > (target0 - w0)) break;
    add(v);
  }
  if (!flat) q.drop();
  for (int32_t v = 0; v < n; ++v) {
    FV& f = fv[v];
    const int32_t own = f.side == 0 ? f.id : g.v[v].inc - f.id;
    f.id = own;
    f.ed = g.v[v].inc - own;
  }
  pw[0] = w0;
  pw[1] = g.tw - w0;
  return cut;
}

// Multilevel bisection of g.  target0 = desired weight of side 0.  side[v]
// (n) receives the result; returns its cut (tracked exactly through growth,
// FM and projection), and its side-0 weight in *w0.
int64_t ml_bisect(const G& g, int64_t target0, double tol, uint64_t seed, uint8_t* side, int64_t* w0, bool par) {
  Arena::Scope all;
  Arena& A = Arena::get();
  Rng rng(seed);
  const int64_t t1 = g.tw - target0;
  Bal bal;
  bal.max[0] = static_cast<int64_t>(std::floor(double(target0) * (1.0 + tol)));
  bal.max[1] = static_cast<int64_t>(std::floor(double(t1) * (1.0 + tol)));
  // Coarsen.
  std::vector<G> levels;
  std::vector<int32_t*> cmaps;
  levels.reserve(64);
  const G* cur = &g;
  const int64_t maxvw = std::max<int64_t>(1, static_cast<int64_t>(1.5 * double(g.tw) / 60.0));
  while (cur->n > 120) {
    int32_t* cm = A.take<int32_t>(cur->n);
    G c = coarsen_hem(*cur, rng, maxvw, cm, par);
    if (c.n > 0.92 * cur->n) break;
    cmaps.push_back(cm);
    levels.push_back(c);
    cur = &levels.back();
  }
  // Initial bisection: best of several grown regions.
  const G& cg = *cur;
  FV* best = A.take<FV>(cg.n);
  FV* trial = A.take<FV>(cg.n);
  int64_t best_cut = INT64_MAX, best_ol = INT64_MAX;
  int64_t pw[2] = {0, 0};
  const int trials = cg.n <= 1 ? 1 : GKIP_TRIALS;
  for (int t = 0; t < trials; ++t) {
    int32_t s = static_cast<int32_t>(rng.below(static_cast<uint32_t>(std::max(1, cg.n))));
    int64_t tpw[2];
    int64_t c = grow(cg, trial, s, target0, tpw);
    fm2(cg, trial, tpw, bal, 4, c);
    int64_t ol = overload(tpw, bal);
    if (ol < best_ol || (ol == best_ol && c < best_cut)) {
      best_ol = ol;
      best_cut = c;
      std::swap(best, trial);
      pw[0] = tpw[0];
      pw[1] = tpw[1];
    }
  }
  // Uncoarsen with refinement.  A vertex whose coarse vertex has no cut edge
  // has none either: only the rows of the others are read for their degrees.
  FV* coarse = best;
  for (int32_t l = static_cast<int32_t>(levels.size()) - 1; l >= 0; --l) {
    const G& fine = (l == 0) ? g : levels[l - 1];
    const int32_t* cm = cmaps[l];
    FV* fv = A.take<FV>(fine.n);
    uint8_t* sd = A.take<uint8_t>(fine.n);
    for (int32_t v = 0; v < fine.n; ++v) {
      const FV& c = coarse[cm[v]];
      sd[v] = c.side;
      fv[v] = FV{fine.v[v].inc, c.ed, -1, c.side, 0, 0, 0};
    }
    for (int32_t v = 0; v < fine.n; ++v) {
      if (fv[v].ed == 0) continue;
      const uint8_t sv = sd[v];
      int32_t a = 0;
      for (int32_t j = fine.v[v].lo; j < fine.v[v].hi; ++j) a += sd[fine.e[j].u] == sv ? fine.e[j].w : 0;
      fv[v].ed = fv[v].id - a;
      fv[v].id = a;
    }
    fm2(fine, fv, pw, bal, GKIP_FMPASS, best_cut);  // projection preserves the cut
    coarse = fv;
  }
  for (int32_t v = 0; v < g.n; ++v) side[v] = coarse[v].side;
  *w0 = pw[0];
  return best_cut;
}

// Induced subgraph (in the arena) of the vertices with side[v] == s; ids (its
// vertices' numbers, in the arena) from the parent's.
G induced(const G& g, const uint8_t* side, uint8_t s, const int32_t* parent_ids, int32_t** ids) {
  Arena& A = Arena::get();
  int32_t cnt = 0;
  int64_t ub = 0;  // entries of the kept rows: room for the induced rows
  for (int32_t v = 0; v < g.n; ++v)
    if (side[v] == s) {
      ++cnt;
      ub += g.v[v].hi - g.v[v].lo;
    }
  G h;
  h.n = cnt;
  h.v = A.take<V>(cnt);
  *ids = A.take<int32_t>(cnt);
  h.e = A.take<Edge>(static_cast<size_t>(ub));
  int32_t top = 0;
  {
    Arena::Scope work;
    int32_t* loc = A.take<int32_t>(g.n);
    int32_t i = 0;
    for (int32_t v = 0; v < g.n; ++v) loc[v] = side[v] == s ? i++ : -1;
    i = 0;
    for (int32_t v = 0; v < g.n; ++v) {
      if (side[v] != s) continue;
      (*ids)[i] = parent_ids[v];
      h.v[i].vw = g.v[v].vw;
      h.tw += g.v[v].vw;
      h.v[i].lo = top;
      int32_t sum = 0;
      for (int32_t j = g.v[v].lo; j < g.v[v].hi; ++j) {
        const int32_t u = loc[g.e[j].u];
        const bool in = u >= 0;
        if (in) {
          h.e[top] = Edge{u, g.e[j].w};
          sum += g.e[j].w;
        }
        top += in;
      }
      h.v[i].hi = top;
      h.v[i].inc = sum;
      ++i;
    }
  }
  A.keep(h.e, static_cast<size_t>(top));
  h.rows = top;
  return h;
}

struct RBCtx {
  double tol;
  int ncuts0, ncuts1, ncuts2;
  uint64_t seed;
  bool parallel;  // use the fork-join pool
};

void rb(const G& g, int32_t k, int32_t part0, int depth, RBCtx& ctx, int32_t* out, const int32_t* ids) {
  if (k == 1 || g.n <= 1) {
    for (int32_t i = 0; i < g.n; ++i) out[ids[i]] = part0;
    return;
  }
  Arena::Scope all;
  const int32_t k0 = k / 2, k1 = k - k0;
  const int64_t target0 = g.tw * k0 / k;
  const uint64_t s = ctx.seed * 0x9E3779B97F4A7C15ull ^ (uint64_t(depth) << 40) ^ uint64_t(part0) * 0xD1B54A32D192ED03ull;
  // Several independent multilevel bisections (more near the root, where a
  // bisection decides the most); keep the lowest (overload, cut, trial).
  // Trials run on spare threads; the pick does not depend on scheduling.
  const int ncuts = depth == 0 ? ctx.ncuts0 : (depth < 3 ? ctx.ncuts1 : ctx.ncuts2);
  uint8_t* trial = Arena::get().take<uint8_t>(size_t(ncuts) * g.n);
  std::vector<int64_t> key_ol(ncuts), key_cut(ncuts);
  auto run_trial = [&](int c) {
    int64_t pw0 = 0;
    key_cut[c] = ml_bisect(g, target0, ctx.tol, s + 0x51ED2701ull * uint64_t(c), trial + size_t(c) * g.n, &pw0, ctx.parallel);
    const int64_t t1 = g.tw - target0;
    const int64_t m0 = static_cast<int64_t>(std::floor(double(target0) * (1.0 + ctx.tol)));
    const int64_t m1 = static_cast<int64_t>(std::floor(double(t1) * (1.0 + ctx.tol)));
    key_ol[c] = std::max<int64_t>(0, pw0 - m0) + std::max<int64_t>(0, (g.tw - pw0) - m1);
  };
  const bool spawn = ctx.parallel && g.n > GKIP_SPAWN_MIN;
  if (spawn) {
    std::vector<std::shared_ptr<ForkJoin::Task>> ts;
    for (int c = 1; c < ncuts; ++c) ts.push_back(ForkJoin::get().spawn([&, c] { run_trial(c); }));
    run_trial(0);
    for (auto& t : ts) ForkJoin::get().wait(t);
  } else {
    for (int c = 0; c < ncuts; ++c) run_trial(c);
  }
  int bc = 0;
  for (int c = 1; c < ncuts; ++c)
    if (key_ol[c] < key_ol[bc] || (key_ol[c] == key_ol[bc] && key_cut[c] < key_cut[bc])) bc = c;
  const uint8_t* side = trial + size_t(bc) * g.n;
  // The two halves are independent: each makes its own graph, one may run on
  // another thread.
  auto half = [&](uint8_t x) {
    Arena::Scope own;
    int32_t* hid = nullptr;
    const G h = induced(g, side, x, ids, &hid);
    if (x == 0) rb(h, k0, part0, depth + 1, ctx, out, hid);
    else rb(h, k1, part0 + k0, depth + 1, ctx, out, hid);
  };
  if (spawn) {
    auto t = ForkJoin::get().spawn([&] { half(0); });
    half(1);
    ForkJoin::get().wait(t);
  } else {
    half(0);
    half(1);
  }
}

// k-way greedy boundary pass: repair parts above cap, then positive-gain
// moves that respect the cap.  Vertices are visited in id order each sweep.
// A visit changes nothing, and will not until a neighbour moves, unless the
// vertex's part is above the cap or some part would give a positive gain (only
// the cap can then hold it back): after the first sweep only such vertices and
// the movers' neighbours are visited.  With par the first sweep's vertices are
// picked on the pool threads beforehand.
void kway_polish(const G& g, int32_t k, int64_t cap, int32_t* part, int sweeps, bool par) {
  Arena::Scope all;
  const int32_t n = g.n;
  std::vector<int64_t> pw(k, 0);
  for (int32_t v = 0; v < n; ++v) pw[part[v]] += g.v[v].vw;
  const int32_t words = (n + 63) / 64;
  uint64_t* due = Arena::get().take<uint64_t>(words);
  // Weights of v to the parts around it (conn, all 0 before; touched lists
  // them); false when every neighbour is in v's own part.
  auto connect = [&](int32_t v, int32_t* conn, std::vector<int32_t>& touched) -> bool {
    const int32_t p = part[v];
    int32_t j = g.v[v].lo;
    while (j < g.v[v].hi && part[g.e[j].u] == p) ++j;
    if (j == g.v[v].hi) return false;
    touched.clear();
    for (j = g.v[v].lo; j < g.v[v].hi; ++j) {
      const int32_t q = part[g.e[j].u];
      if (conn[q] == 0) touched.push_back(q);
      conn[q] += g.e[j].w;
    }
    return true;
  };
  auto may_move = [&](int32_t v, const int32_t* conn, const std::vector<int32_t>& touched) -> bool {
    const int32_t p = part[v];
    if (pw[p] > cap) return true;
    for (int32_t q : touched)
      if (q != p && conn[q] > conn[p]) return true;
    return false;
  };
  const int chunks = par ? static_cast<int>(std::min<int64_t>(16, g.rows / 8192)) : 1;
  if (chunks > 1) {
    par_chunks(chunks, [&](int c) {
      std::vector<int32_t> conn(k, 0), touched;
      for (int32_t w = int32_t(int64_t(words) * c / chunks); w < int32_t(int64_t(words) * (c + 1) / chunks); ++w) {
        uint64_t b = 0;
        for (int32_t v = 64 * w; v < std::min(n, 64 * w + 64); ++v) {
          if (!connect(v, conn.data(), touched)) continue;
          if (may_move(v, conn.data(), touched)) b |= 1ull << (v & 63);
          for (int32_t q : touched) conn[q] = 0;
        }
        due[w] = b;
      }
    });
  } else {
    for (int32_t w = 0; w < words; ++w) due[w] = w + 1 < words || n % 64 == 0 ? ~0ull : (1ull << (n % 64)) - 1;
  }
  std::vector<int32_t> conn(k, 0), touched;
  for (int s = 0; s < sweeps; ++s) {
    int64_t moves = 0;
    for (int32_t w = 0; w < words; ++w) {
      // Bits set meanwhile: those behind the current vertex are still visited
      // in this sweep, those before it in the next one.
      uint64_t seen = 0;
      while (uint64_t left = due[w] & ~seen) {
        const int bit = __builtin_ctzll(left);
        const int32_t v = 64 * w + bit;
        seen |= bit == 63 ? ~0ull : (2ull << bit) - 1;
        due[w] &= ~(1ull << bit);
        if (!connect(v, conn.data(), touched)) continue;
        const int32_t p = part[v];
        const bool over = pw[p] > cap;
        int32_t bestq = -1;
        int64_t bestg = 0;
        for (int32_t q : touched) {
          if (q == p) continue;
          if (pw[q] + g.v[v].vw > cap) continue;
          int64_t gain = int64_t(conn[q]) - conn[p];
          bool better;
          if (over) better = bestq < 0 || gain > bestg || (gain == bestg && (pw[q] < pw[bestq] || (pw[q] == pw[bestq] && q < bestq)));
          else better = gain > bestg || (gain == bestg && gain > 0 && q < bestq);
          if (better) { bestq = q; bestg = gain; }
        }
        if (bestq >= 0 && (over || bestg > 0)) {
          pw[p] -= g.v[v].vw;
          pw[bestq] += g.v[v].vw;
          part[v] = bestq;
          ++moves;
          due[w] |= 1ull << bit;
          for (int32_t j = g.v[v].lo; j < g.v[v].hi; ++j) due[g.e[j].u >> 6] |= 1ull << (g.e[j].u & 63);
        } else if (may_move(v, conn.data(), touched)) {
          due[w] |= 1ull << bit;
        }
        for (int32_t q : touched) conn[q] = 0;
      }
    }
    if (moves == 0) break;
  }
}

}  // namespace

extern "C" int64_t gk_part_cap(int64_t total_vwgt, int32_t k, int32_t ubfactor) {
  if (k < 1) return total_vwgt;
  int64_t a = total_vwgt * (1000 + int64_t(ubfactor)) / (1000 * int64_t(k));
  int64_t b = (total_vwgt + k - 1) / k;
  return std::max(a, b);
}

extern "C" int gk_initpart(const gk_csr* hg, int32_t k, int64_t cap, int32_t seed,
                           int32_t nthreads, int32_t* part, int64_t* cut) {
  if (!hg || !part || k < 1 || hg->n < 0) return GK_ERR_ARG;
  const int32_t n = hg->n;
  if (k == 1) {
    std::fill(part, part + n, 0);
    if (cut) *cut = 0;
    return GK_OK;
  }
  Arena::Scope all;
  Arena& A = Arena::get();
  const bool parallel = nthreads != 1 && ForkJoin::get().workers() > 0;
  G g;
  g.n = n;
  g.rows = hg->xadj[n];
  g.v = A.take<V>(n);
  g.e = A.take<Edge>(static_cast<size_t>(g.rows));
  const int chunks = parallel ? static_cast<int>(std::min<int64_t>(16, std::max<int64_t>(1, g.rows / 16384))) : 1;
  std::vector<int64_t> tw(chunks, 0);
  par_chunks(chunks, [&](int c) {
    for (int32_t v = int32_t(int64_t(n) * c / chunks); v < int32_t(int64_t(n) * (c + 1) / chunks); ++v) {
      int32_t sum = 0;
      for (int32_t j = hg->xadj[v]; j < hg->xadj[v + 1]; ++j) {
        const int32_t w = hg->adjwgt ? hg->adjwgt[j] : 1;
        g.e[j] = Edge{hg->adjncy[j], w};
        sum += w;
      }
      g.v[v] = V{hg->xadj[v], hg->xadj[v + 1], hg->vwgt ? hg->vwgt[v] : 1, sum};
      tw[c] += g.v[v].vw;
    }
  });
  for (int64_t x : tw) g.tw += x;
  // Per-bisection tolerance: (cap / (T/k))^(1/levels) - 1, slightly tightened
  // so that rounding of the recursive targets stays inside the cap.
  const int levels = static_cast<int>(std::ceil(std::log2(double(k))));
  const double ratio = double(cap) * k / std::max<double>(1.0, double(g.tw));
  double tol = std::pow(std::max(1.0, ratio), 1.0 / std::max(1, levels)) - 1.0;
  tol = std::max(0.0, tol * 0.9);
  RBCtx ctx;
  ctx.tol = tol;
  ctx.ncuts0 = GKIP_NCUTS0;
  ctx.ncuts1 = GKIP_NCUTS1;
  ctx.ncuts2 = GKIP_NCUTS2;
  ctx.seed = static_cast<uint64_t>(seed) + 1;
  // nthreads == 1: everything on the calling thread; otherwise the
  // process-wide pool (up to 16 threads) helps.
  ctx.parallel = parallel;
  int32_t* ids = A.take<int32_t>(n);
  std::iota(ids, ids + n, 0);
  rb(g, k, 0, 0, ctx, part, ids);
  kway_polish(g, k, cap, part, 4, parallel);
  if (cut) {
    std::vector<int64_t> cs(chunks, 0);
    par_chunks(chunks, [&](int c) {
      int64_t x = 0;
      for (int32_t v = int32_t(int64_t(n) * c / chunks); v < int32_t(int64_t(n) * (c + 1) / chunks); ++v)
        for (int32_t j = g.v[v].lo; j < g.v[v].hi; ++j)
          x += v < g.e[j].u && part[v] != part[g.e[j].u] ? g.e[j].w : 0;
      cs[c] = x;
    });
    *cut = 0;
    for (int64_t x : cs) *cut += x;
  }
  return GK_OK;
}
