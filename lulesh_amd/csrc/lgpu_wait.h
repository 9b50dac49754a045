// lgpu_wait.h -- waiting on the host for a count that a kernel stores in pinned
// memory.
#pragma once

#include <chrono>
#include <stdint.h>

namespace lgpu {

// Waits until a kernel's count in pinned memory has reached `want`, for up to
// 2 ms: false if it has not, and the caller then waits for the stream.  A
// kernel's store is seen about 5 us sooner than hipStreamSynchronize returns
// (launch and wait 5.8 against 11.3 us), of no weight after 2 ms.
inline bool host_reached(const uint32_t *count, uint32_t want)
{
   const auto start = std::chrono::steady_clock::now();
   for (;;) {
      for (int i = 0; i < 64; ++i) {
         if ((int32_t)(__atomic_load_n(count, __ATOMIC_ACQUIRE) - want) >= 0) return true;
         __builtin_ia32_pause();
      }
      if (std::chrono::steady_clock::now() - start > std::chrono::milliseconds(2)) return false;
   }
}

} // namespace lgpu
