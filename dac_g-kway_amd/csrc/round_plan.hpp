// Which launches a level's refinement rounds are run by, one after another:
// host-only bookkeeping of refine_rounds (driver.hip), apart from it so that
// its bounds can be tested without a device.
#pragma once
#include <algorithm>
#include <cstdint>

namespace gkrt {

// Two ways to run rounds, which leave the same state.  The round loop (one
// workgroup per job) is the faster one while a job has up to some thousand
// candidates; the separate kernels select over the whole device, and start on
// graphs so large that their first rounds will have more.  The host looks at
// the end of a round loop's launch, and every 4 rounds of the separate kernels
// (every 8, 16, then 32 once they ran 32: a look costs a copy and a
// synchronisation; a round with nothing selected changes nothing).
class RoundPlan {
 public:
  static constexpr int kWideRounds = 4;
  static constexpr int kLoopRounds = 64;

  // max_rounds: as for refine_rounds; graph: launches may be captured.
  RoundPlan(bool can_loop, int64_t n, int32_t nj, int max_rounds, bool exact, bool graph)
      : max_(max_rounds), exact_(exact), graph_(graph), step_(max_rounds > 0 && !exact),
        wide_most_(std::max(kWideRounds, max_rounds / 4)), jobs_(nj), may_return_(can_loop),
        loop_(can_loop && n <= kLoopVertices * nj) {}

  bool ended() const { return ended_ || (max_ > 0 && done_ >= max_); }
  bool loop() const { return loop_; }
  // Rounds of the next launch (of the round loop) or of the launches up to the
  // next look (separate kernels).
  int rounds() const {
    const int most = loop_ ? kLoopRounds : per_check_;
    return max_ > 0 ? std::min(most, max_ - done_) : most;
  }
  // Whether they are replayed from a graph: two launches of half the loop's
  // rounds each, so that every replay begins with the same pair of counts; or
  // kWideRounds rounds of the separate kernels at a time.
  bool captured() const {
    return graph_ && (loop_ ? rounds() == kLoopRounds && pair_ == kFirstPair : rounds() % kWideRounds == 0);
  }
  // The pair of counts and status words that the next launch of the loop uses,
  // zero before it; the launch clears the other pair for the next one.  A graph
  // holds the pair it was captured with, so only the first pair is captured.
  int pair() const { return pair_; }
  int done() const { return done_; }

  // What the host saw after them.  live: jobs that go on; left_out: of those,
  // jobs whose candidates were too many, which did no round; ordered (exact,
  // one job): rounds that ordered moves so far.
  void loop_ran(int32_t live, int32_t left_out, int32_t ordered) {
    const int given = rounds();
    if (!captured()) pair_ = 1 - pair_;
    // a launch that leaves a job out gives its rounds back
    if (exact_) done_ = ordered;
    else if (live == 0 || left_out == 0) done_ += given;
    if (live == 0) ended_ = true;
    if (live == 0 || left_out == 0) return;
    loop_ = false;
    if (step_ && left_out > left_out_ / 2) may_return_ = false;
    left_out_ = left_out;
  }
  // live: vertices selected in the last round.  Returns whether the loop takes
  // over, with cleared counts and status words.
  bool wide_ran(int32_t live) {
    const int given = rounds();
    done_ += given;
    wide_done_ += given;
    if (live == 0 || (step_ && wide_done_ >= wide_most_)) {
      ended_ = true;
      return false;
    }
    if (may_return_ && live <= kLoopSelected * jobs_) {
      loop_ = true;
      pair_ = kFirstPair;  // both are cleared
    }
    if (wide_done_ >= 32 && per_check_ < 32) per_check_ *= 2;
    return loop_;
  }

 private:
  static constexpr int64_t kLoopVertices = int64_t(1) << 20;  // per job, to begin with the loop
  static constexpr int32_t kLoopSelected = 1024;              // selected per round, to come back to it
  static constexpr int kFirstPair = 1;                        // the compaction before the rounds uses pair 0
  const int max_;
  const bool exact_, graph_;
  // A step of a batch: new requests wait for its end.  Launches of the loop
  // that leave a job out give their rounds back, so max_rounds alone does not
  // bound the rounds by the separate kernels; they get a quarter of it, and the
  // loop is tried again only while each attempt leaves out at most half as many
  // jobs as the last.  Poisson arrivals at 200 a second, 500 graphs of up to
  // 2 M vertices, 20 s: without the bound 3000 such rounds and 100 attempts in
  // a step of 350 ms, half of the requests later than 3.4-3.6 s; with it 46-47
  // ms.
  const bool step_;
  const int wide_most_;
  const int32_t jobs_;
  bool may_return_;  // from the separate kernels to the loop
  bool loop_;
  bool ended_ = false;
  int pair_ = kFirstPair;
  int done_ = 0, wide_done_ = 0, per_check_ = kWideRounds;
  int32_t left_out_ = INT32_MAX;  // by the loop's last launch that left any
};

}  // namespace gkrt
