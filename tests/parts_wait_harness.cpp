// Runs the partitioned frame's assembly (parts_wait.hpp) with one thread per
// part.  Arguments: scenario, parts, rounds.  Exit status 1 if in any round the
// parts disagree, or agree on the wrong thing.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <thread>
#include <vector>

#include "../ff-srl_amd/csrc/parts_wait.hpp"

using namespace ffsrl;

struct Word {
  std::atomic<uint32_t>* w;
  std::atomic<int>* working;
  std::atomic<long>* polls;
  uint32_t add(uint32_t n) { return w->fetch_add(n); }
  uint32_t cas(uint32_t expected, uint32_t desired) {
    w->compare_exchange_strong(expected, desired);
    return expected;
  }
  bool idle() { return working->load() == 0; }
  void pause(int) {
    polls->fetch_add(1);
    std::this_thread::yield();
  }
};

int main(int argc, char** argv) {
  const char* scenario = argv[1];
  const int np = atoi(argv[2]), rounds = atoi(argv[3]);
  auto is = [&](const char* s) { return !strcmp(scenario, s); };
  std::mt19937 rng(1);
  long went = 0, left = 0;
  for (int r = 0; r < rounds; ++r) {
    std::atomic<uint32_t> w{0};
    std::atomic<int> working{is("busy") ? 1 : 0};
    std::atomic<long> polls{0};
    int idle_polls = 1 << 28, limit = 1 << 28;
    if (is("absent")) idle_polls = 50;              // one part is claimed after the others withdrew
    if (is("race")) idle_polls = 1 + (int)(rng() % 40);  // one part arrives about when they do
    if (is("busy")) idle_polls = 1;                 // a workgroup at work on the XCD: no idle withdrawal
    if (is("large")) idle_polls = 0;                // no other form of the env: the same
    if (is("limit")) idle_polls = 0, limit = 50;    // ... but not for ever
    const bool late = is("absent") || is("race") || is("busy") || is("large") || is("limit");
    std::vector<int> go((size_t)np, -1);
    std::vector<std::thread> th;
    std::atomic<bool> start{!is("race")};
    auto part = [&](int i) {
      while (!start.load()) std::this_thread::yield();
      go[(size_t)i] = parts_assemble(Word{&w, &working, &polls}, (uint32_t)np, idle_polls, limit);
    };
    const long k = (long)(rng() % 60) * (np - 1);
    auto late_part = [&] {  // after k polls of the others, or when they have withdrawn
      while (!start.load()) std::this_thread::yield();
      while (is("race") && polls.load() < k && !(w.load() & kWithdrawn)) std::this_thread::yield();
      part(np - 1);
    };
    if (is("race")) th.emplace_back(late_part);
    for (int i = 0; i < np - (late ? 1 : 0); ++i) th.emplace_back(part, i);
    start = true;
    if (is("busy") || is("large"))
      while (polls.load() < 2000) std::this_thread::yield();  // far beyond the idle limit
    if (is("absent") || is("limit")) {
      for (auto& t : th) t.join();  // they end by themselves
      th.clear();
    }
    if (late && !is("race")) th.emplace_back(late_part);
    for (auto& t : th) t.join();
    for (int i = 1; i < np; ++i)
      if (go[(size_t)i] != go[0]) return printf("round %d: parts disagree\n", r), 1;
    const bool all = go[0] != 0;
    (all ? went : left) += 1;
    if (all != !(w.load() & kWithdrawn)) return printf("round %d: the word does not say so\n", r), 1;
    if ((is("all") || is("busy") || is("large")) && !all) return printf("round %d: withdrew\n", r), 1;
    if ((is("absent") || is("limit")) && all) return printf("round %d: went on without a part\n", r), 1;
  }
  printf("went %ld left %ld\n", went, left);
  return 0;
}
