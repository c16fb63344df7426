// Admission of resident launches (fe_resident.h) to a device: what is inside
// fits it at the same time, in the order of arrival, so that small solves of
// several threads overlap and one that needs the whole device is not passed
// over.  Host code only.
//
// The unit is a CU of every shader engine (8 per engine): workgroups go round
// the engines, and a launch is charged its largest number on one of them, so
// no engine has more workgroups than CUs whatever the launches started at.
#pragma once

#include <condition_variable>
#include <mutex>

class FeResidentGate {
 public:
  void enter(int need, int cap)
  {
    std::unique_lock<std::mutex> lock(m_);
    const unsigned long long mine = arrived_++;
    cv_.wait(lock, [&] { return admitted_ == mine && (used_ == 0 || used_ + need <= cap); });
    used_ += need;
    ++admitted_;
    cv_.notify_all();
  }
  void leave(int need)
  {
    std::lock_guard<std::mutex> lock(m_);
    used_ -= need;
    cv_.notify_all();
  }
  bool busy()
  {
    std::lock_guard<std::mutex> lock(m_);
    return used_ > 0 || admitted_ != arrived_;
  }
  // Held while a kernel's LDS limit, which all threads share, is set and the
  // kernel launched with it.
  std::mutex &launching() { return launch_; }

 private:
  std::mutex m_, launch_;
  std::condition_variable cv_;
  int used_ = 0;
  unsigned long long arrived_ = 0, admitted_ = 0;
};

// CUs of an engine that a launch of G workgroups takes, on a device of `cus`.
constexpr int kGateCus = 8;
inline int feGateNeed(int G, int cus)
{
  const int engines = cus >= kGateCus ? cus / kGateCus : 1, need = (G + engines - 1) / engines;
  return need < kGateCus ? need : kGateCus;
}
