// How the parts of an environment come together in the partitioned frame.
// Host and device code, so that the protocol can be run by threads on the host.
#pragma once

#include <cstdint>

namespace ffsrl {

// Set in an env's assembly word when its parts gave up waiting for each other.
constexpr uint32_t kWithdrawn = 1u << 31;

// One thread of a part waits for the env's np parts to arrive at the env's
// word; false when they withdraw from the env.  The first to give up sets
// kWithdrawn, and can only while fewer than np have arrived; so either all np
// see np arrivals, or all see the flag.
//
// A part gives up after `polls` polls, or after idle_polls of them in a row
// with no workgroup of the launch at work on the XCD (0: not for that; an env
// that only its parts can run waits for them as long as the frame's other
// waits do, whatever else holds the CUs).
//
// Word: add(n) and cas(expected, desired) return the word before, idle()
// whether no workgroup is at work (asked every kIdleEvery polls), pause(k) passes
// the time after the k-th poll.
constexpr int kIdleEvery = 8;

template <class Word>
__host__ __device__ inline bool parts_assemble(Word word, uint32_t np, int idle_polls, int polls) {
  uint32_t v = word.add(1u) + 1u;
  int idle = 0;
  for (int k = 1; !(v & kWithdrawn) && v < np; ++k) {
    if (idle_polls && k % kIdleEvery == 0) idle = word.idle() ? idle + kIdleEvery : 0;
    if (idle > idle_polls || k > polls) {
      const uint32_t seen = word.cas(v, v | kWithdrawn);
      if (seen == v) return false;
      v = seen;
      continue;  // another part arrived or withdrew meanwhile
    }
    word.pause(k);
    v = word.add(0u);
  }
  return !(v & kWithdrawn);
}

}  // namespace ffsrl
