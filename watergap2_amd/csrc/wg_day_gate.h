// wg_day_gate.h -- keeps launches of the many-days kernel apart that do not fit on a
// GPU together.
//
// Its wavefronts wait for wavefronts before them.  Within one launch those have started,
// because each XCD starts a launch's workgroups in index order.  Two handles' launches
// that compete for slots have no such order between them: each can hold all the slots of
// an XCD that the other's first unfinished workgroup needs.  So launches run side by side
// only while all their wavefronts together are few enough to have slots at once, three
// for four SIMDs: a CU that has no room for a workgroup of one or two holds at least four
// (32,000 bytes of LDS for one, 40,960 for two, of 160 KB), and the rest is for the
// rounding of each launch's share of an XCD.  Others run one after another, in the
// order they came.  (A handle's own launches are on one stream.)
#ifndef WG_DAY_GATE_H
#define WG_DAY_GATE_H

#include <condition_variable>
#include <cstdint>
#include <mutex>

class WgDayGate {
 public:
  // Returns when `waves` wavefronts may run: nothing else does, or all together are at most `limit`.
  void enter(int64_t waves, int64_t limit) {
    std::unique_lock<std::mutex> lock(mutex_);
    const uint64_t turn = last_turn_++;
    changed_.wait(lock, [&] { return turn == turn_ && (running_ == 0 || running_ + waves <= limit); });
    turn_++;
    running_ += waves;
    changed_.notify_all();
  }
  void leave(int64_t waves) {
    std::lock_guard<std::mutex> lock(mutex_);
    running_ -= waves;
    changed_.notify_all();
  }

 private:
  std::mutex mutex_;
  std::condition_variable changed_;
  uint64_t last_turn_ = 0, turn_ = 0;
  int64_t running_ = 0;
};

#endif  // WG_DAY_GATE_H
