// ticket.h — how many work-groups that wait for each other may be in flight.
#pragma once

#include <atomic>

namespace cloth {

// A launch whose `blocks` work-groups wait for each other may go ahead while
// the holders on that device, this one included, have at most one work-group
// for each of its `cus` compute units.  Then none can keep part of another
// from becoming resident: a compute unit can hold a work-group of any of these
// kernels, and while one is still to be placed some unit has none of them
// (work-groups of other kernels end by themselves).  Work-groups are dealt to
// the eight XCDs in turn and stay there, so a launch counts as whole rounds
// of eight and the same holds within each XCD.  A caller that gets no ticket
// takes its path of separate kernels (the same results).  Host code without
// HIP.
class CoopTicket {
 public:
  static constexpr int kMaxDevices = 64;
  static constexpr unsigned kRound = 8;
  CoopTicket(int device, unsigned blocks, unsigned cus) : units_((blocks + kRound - 1) / kRound * kRound) {
    if (device < 0 || device >= kMaxDevices || units_ > cus) return;
    std::atomic<unsigned>& n = in_flight(device);
    unsigned have = n.load();
    do {
      if (have + units_ > cus) return;
    } while (!n.compare_exchange_weak(have, have + units_));
    held_ = &n;
  }
  ~CoopTicket() {
    if (held_) held_->fetch_sub(units_);
  }
  CoopTicket(const CoopTicket&) = delete;
  CoopTicket& operator=(const CoopTicket&) = delete;
  explicit operator bool() const { return held_ != nullptr; }

 private:
  static std::atomic<unsigned>& in_flight(int device) {
    static std::atomic<unsigned> n[kMaxDevices] = {};
    return n[device];
  }
  unsigned units_;
  std::atomic<unsigned>* held_ = nullptr;
};

}  // namespace cloth
