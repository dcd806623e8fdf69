// sdpd_threads.h -- host threads of one call.
#pragma once

#include <thread>

namespace sdpd {

// work(0) here and work(1) .. work(slots - 1) on threads of their own, all
// ended on return.  Slots whose thread cannot be started (no threads or no memory
// left) are not run: work takes its share from a common pile.  Nothing is thrown
// unless work throws.
template <int MAX, class F>
void run_slots(int slots, F&& work) {
  std::thread helper[MAX];
  for (int k = 1; k < slots && k < MAX; ++k) {
    try {
      helper[k] = std::thread([&work, k] { work(k); });
    } catch (...) {
      break;
    }
  }
  work(0);
  for (std::thread& t : helper)
    if (t.joinable()) t.join();
}

}  // namespace sdpd
