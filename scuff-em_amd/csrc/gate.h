// gate.h -- admission of launches whose workgroups wait for each other.
//
// The panels of a factorization pass data between workgroups, so all of a
// panel's workgroups have to be on the GPU at once.  One panel fits (checked
// at every factorization), but two factorizations on streams of their own
// could each hold a part of the workgroup slots and wait for the rest until
// their bounded waits expire.  A factorization therefore enters its device's
// gate with the share of the slots that its panels take and leaves it when
// it has completed.
//
// Admitted together are shares of at most one half in all, or one of any
// size by itself.  A half suffices however the kernels mix: a waiting kernel
// with p >= 2 workgroups to a CU needs at most 1/p <= 1/2 of any of a CU's
// resources, so a CU that cannot take it is more than half full of admitted
// workgroups (all others retire), and not every CU can be.  A kernel with one
// workgroup to a CU takes the whole share.
//
// Host threads wait in order of arrival.  Other processes on the same GPU are
// not counted: against them the panels' waits stay bounded, and the
// factorization reports the time-out.
#pragma once

#include <condition_variable>
#include <mutex>

namespace scuffx {

class Gate {
 public:
  void enter(double share)
  {
    std::unique_lock<std::mutex> lk(mu_);
    const unsigned long me = tail_++;
    cv_.wait(lk, [&] { return me == head_ && (inside_ == 0 || used_ + share <= 0.5); });
    head_++;
    inside_++;
    used_ += share;
    cv_.notify_all();
  }
  void leave(double share)
  {
    std::lock_guard<std::mutex> lk(mu_);
    used_ = --inside_ ? used_ - share : 0.0;
    cv_.notify_all();
  }

 private:
  std::mutex mu_;
  std::condition_variable cv_;
  unsigned long head_ = 0, tail_ = 0;   // next to be admitted, next to arrive
  int inside_ = 0;
  double used_ = 0.0;
};

}  // namespace scuffx
