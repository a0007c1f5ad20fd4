// Who may put a team of workgroups on a device.  The workgroups of an ePIE team wait for one another, so
// all of them have to be there at once: iterations of several handles (from several threads) take their
// workgroups out of one budget per device and wait when it is spent, in the order in which they came (a
// large team behind many small ones would else find the budget too low for as long as they go on).
#pragma once
#include <condition_variable>
#include <mutex>

namespace ptyk {

struct TeamBudget {
  std::mutex mu;
  std::condition_variable cv;
  int left = -1;                // workgroups; set by the first use
  unsigned long came = 0, let = 0;  // tickets handed out, and let in
};

class TeamSlots {
 public:
  // b null or want 0: nothing to wait for.  want is at most total.
  TeamSlots(TeamBudget* b, int total, int want) : b_(want > 0 ? b : nullptr), want_(want) {
    if (!b_) return;
    std::unique_lock<std::mutex> l(b_->mu);
    if (b_->left < 0) b_->left = total;
    const unsigned long me = b_->came++;
    b_->cv.wait(l, [&] { return b_->let == me && b_->left >= want_; });
    ++b_->let;
    b_->left -= want_;
    l.unlock();
    b_->cv.notify_all();  // the next in turn may fit as well
  }
  ~TeamSlots() {
    if (!b_) return;
    {
      std::lock_guard<std::mutex> l(b_->mu);
      b_->left += want_;
    }
    b_->cv.notify_all();
  }
  TeamSlots(const TeamSlots&) = delete;
  TeamSlots& operator=(const TeamSlots&) = delete;

 private:
  TeamBudget* b_;
  int want_;
};

}  // namespace ptyk
