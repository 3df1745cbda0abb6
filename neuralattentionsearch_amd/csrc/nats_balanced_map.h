// The map of a prefill launch that starts its heavy streams first: host and device code without anything else of the
// library, so that a host program can enumerate it.
#pragma once

#include <stdint.h>

namespace nats {

// Workgroup `bid` of ns * n_hg * n_qg -> its item, where the streams in `heavy` (a set of the first ns <= 64) come first.
__host__ __device__ inline void balanced_item(uint64_t heavy, int ns, int n_hg, int n_qg, int bid, int& ks, int& hg, int& rank) {
  const uint64_t light = ~heavy & (ns < 64 ? (uint64_t(1) << ns) - 1 : ~uint64_t(0));
  const uint64_t every8 = 0x0101010101010101ull;
  const int total = ns * n_hg * n_qg;
  const int n_heavy = (int)__builtin_popcountll(heavy) * n_hg * n_qg;
  uint64_t set = heavy;
  int i = bid;  // the item's place among those of the streams in `set`, rank by rank
  if (bid >= n_heavy) {
    // Workgroup i runs on XCD i mod 8.  An XCD works through the light streams that are its own as far as its workgroups
    // reach; what is left of them (their lightest query groups) goes to the XCDs that have workgroups to spare.
    auto own = [&](int y) -> int { return (int)__builtin_popcountll(light & (every8 << y)) * n_hg * n_qg; };
    auto slots = [&](int y) -> int { return (total + 7 - y) / 8 - (n_heavy + 7 - y) / 8; };  // workgroups of [n_heavy, total) on XCD y
    auto kept = [&](int y) -> int { return own(y) < slots(y) ? own(y) : slots(y); };
    const int x = bid & 7;
    i = (bid - x) / 8 - (n_heavy + 7 - x) / 8;  // this workgroup's place among those of its XCD
    int home = x;
    if (i >= kept(x)) {
      int o = i - kept(x);  // ... among the workgroups to spare, then among the items left over
      for (int y = 0; y < x; ++y) o += slots(y) - kept(y);
      for (home = 0; home < 7 && o >= own(home) - kept(home); ++home) o -= own(home) - kept(home);
      i = kept(home) + o;
    }
    set = light & (every8 << home);
  }
  const int n_slot = (int)__builtin_popcountll(set) * n_hg;
  rank = i / n_slot;
  const int slot = i % n_slot;
  hg = slot % n_hg;
  for (int n = slot / n_hg; n > 0; --n) set &= set - 1;
  ks = __builtin_ctzll(set);
}

}  // namespace nats
