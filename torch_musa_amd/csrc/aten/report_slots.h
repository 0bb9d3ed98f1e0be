// Which call holds which of the host's report slots (tmq_host_report); host code without a GPU call.
#pragma once

#include <condition_variable>
#include <cstdint>
#include <mutex>
#include <vector>

#include "tmq.h"

namespace tmq {

// `count` slots, each with one call at a time.  A call that cannot say whether the device still writes to
// its slot loses it: it is not handed out again.
class ReportSlots {
 public:
  explicit ReportSlots(int count) : count_(count) {
    for (int i = 0; i < count; ++i) free_.push_back(i);
  }
  // A slot and the ticket of its use; waits for one.  -1: all are lost, none will come.
  int take(uint32_t* ticket) {
    std::unique_lock<std::mutex> lock(mu_);
    changed_.wait(lock, [&] { return !free_.empty() || lost_ == count_; });
    if (free_.empty()) return -1;
    const int slot = free_.back();
    free_.pop_back();
    if (++ticket_ == 0) ++ticket_;  // (fresh memory is zero)
    *ticket = ticket_;
    return slot;
  }
  void give_back(int slot) {
    {
      std::lock_guard<std::mutex> lock(mu_);
      free_.push_back(slot);
    }
    changed_.notify_one();
  }
  void lose() {
    {
      std::lock_guard<std::mutex> lock(mu_);
      ++lost_;
    }
    changed_.notify_all();
  }

 private:
  const int count_;
  std::mutex mu_;
  std::condition_variable changed_;
  std::vector<int> free_;
  int lost_ = 0;
  uint32_t ticket_ = 0;
};

// One call's slot.
class ReportHold {
 public:
  explicit ReportHold(ReportSlots& slots) : slots_(slots), slot_(slots.take(&ticket_)) {}
  ~ReportHold() {
    if (slot_ < 0) return;
    if (pending_) slots_.lose();
    else slots_.give_back(slot_);
  }
  ReportHold(const ReportHold&) = delete;
  ReportHold& operator=(const ReportHold&) = delete;

  int slot() const { return slot_; }  // -1: none
  uint32_t ticket() const { return ticket_; }
  // Runs `call`, which queues the kernels that write to the slot, and returns its status.  A chain of launches can
  // fail behind the first one, whose kernel then still runs: the slot is the device's from before the call on.  After a
  // failure `drain` waits for the stream; only if it can say that nothing runs any more is the slot free again.
  template <class Call, class Drain>
  int queue(Call&& call, Drain&& drain) {
    pending_ = true;
    const int status = call();
    if (status != TMQ_OK && drain()) pending_ = false;
    return status;
  }
  void done() { pending_ = false; }  // the report is here: the device has written its last word

 private:
  ReportSlots& slots_;
  uint32_t ticket_ = 0;
  int slot_;
  bool pending_ = false;
};

}  // namespace tmq
