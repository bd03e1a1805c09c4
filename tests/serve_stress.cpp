// Host-thread stress of a serving slot's arena (serve_take in
// hvm-64_amd/csrc/hvm64_rules.h, built for the host): argv[1] threads take
// node blocks of 1 to argv[3] nodes until each has been refused argv[4]
// times, then what is left is taken node by node; argv[2] rounds on a cleared
// slot.  Checks that no two blocks overlap, that every block lies in one
// sub-arena, that a block is refused only if no sub-arena has room for it at
// the end, and that node by node everything is handed out.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#include "hvm64_rules.h"

using namespace hvm;

int main(int, char **argv) {
  const u32 threads = (u32)atoi(argv[1]), rounds = (u32)atoi(argv[2]), most = (u32)atoi(argv[3]);
  const u32 refusals = (u32)atoi(argv[4]);
  const u64 len = 1024;
  u64 words[SERVE_WORDS];
  u64 blocks = 0, overlaps = 0, outside = 0, wrongly_refused = 0, lost = 0;
  for (u32 round = 0; round < rounds; round++) {
    serve_clear(words);
    std::vector<std::vector<std::pair<u64, u64>>> got(threads);
    std::vector<u32> least(threads, ~0u);  // smallest block refused
    std::vector<std::thread> pool;
    for (u32 t = 0; t < threads; t++)
      pool.emplace_back([&, t] {
        u64 x = 0x9E3779B97F4A7C15ull * (round * threads + t + 1);
        for (u32 no = 0; no < refusals;) {
          x ^= x << 13;
          x ^= x >> 7;
          x ^= x << 17;
          const u32 n = 1 + (u32)((x >> 8) % (x & 3 ? std::min(most, 6u) : most));
          const u64 p = serve_take(words, len, (u32)(x >> 40), n);
          if (p != NO_NODES) got[t].push_back({p, p + n});
          else no++, least[t] = std::min(least[t], n);
        }
      });
    for (auto &th : pool) th.join();
    u32 n_least = ~0u;
    for (u32 v : least) n_least = std::min(n_least, v);
    std::vector<std::pair<u64, u64>> all;
    for (auto &g : got) all.insert(all.end(), g.begin(), g.end());
    // (room is never made while a net runs, so what is refused now was short then)
    if (n_least != ~0u && serve_take(words, len, round, n_least) != NO_NODES) wrongly_refused++;
    for (u64 p; (p = serve_take(words, len, round, 1)) != NO_NODES;) all.push_back({p, p + 1});
    std::sort(all.begin(), all.end());
    u64 nodes = 0;
    for (size_t i = 0; i < all.size(); i++) {
      nodes += all[i].second - all[i].first;
      if (i && all[i].first < all[i - 1].second) overlaps++;
      if (all[i].second > SERVE_SUB * len || all[i].first / len != (all[i].second - 1) / len) outside++;
    }
    blocks += all.size();
    lost += SERVE_SUB * len - nodes;
  }
  printf("blocks %llu overlaps %llu outside %llu refused %llu lost %llu\n", (unsigned long long)blocks,
         (unsigned long long)overlaps, (unsigned long long)outside, (unsigned long long)wrongly_refused,
         (unsigned long long)lost);
  return overlaps || outside || wrongly_refused || lost ? 1 : 0;
}
