// Host-side dump of the attention kernels' launch order (spread_workgroup, then
// work_position, attn_common.h) and of fast_div, for tests/test_work_map.py:
//   work_map_dump groups m_blocks group ilv [workgroups per CU [causal]]  ->  one line per workgroup: "bid group item" (-1 -1: none)
//   work_map_dump --div                      ->  the number of wrong quotients over edges and a sweep
#include <cstdio>
#include <cstdlib>

#include "attn_common.h"

int main(int argc, char** argv) {
  if (argc == 2) {
    long wrong = 0;
    const int big[] = {1 << 20, 65536, 65537, 1000003, (1 << 30) - 1, 1 << 30, (1 << 30) + 1, 2147483646, 2147483647};
    for (int i = 0; i < 4096 + 9; ++i) {
      const int d = i < 4096 ? i + 1 : big[i - 4096];
      const tmx::FastDiv f = tmx::make_fast_div(d);
      for (int k = 0; k < 200; ++k) {
        // multiples of d and their neighbours up to 2^31 - 1
        const int64_t base = ((int64_t)2147483647 / d) * k / 199 * d;
        for (int64_t n = base - 1; n <= base + 1; ++n)
          if (n >= 0 && n <= 2147483647) wrong += tmx::fast_div((int)n, f) != (int)(n / d);
      }
      wrong += tmx::fast_div(2147483647, f) != 2147483647 / d;
    }
    printf("%ld\n", wrong);
    return 0;
  }
  if (argc < 5 || argc > 7) return 2;
  const int groups = atoi(argv[1]), m_blocks = atoi(argv[2]), group = atoi(argv[3]), ilv = atoi(argv[4]);
  const int ipg = m_blocks * group;
  const tmx::WorkMap w = tmx::make_work_map(groups * ipg, ipg, ilv, group, 1, argc < 7 || atoi(argv[6]) != 0,
                                            argc > 5 ? atoi(argv[5]) : 2);
  for (int bid = 0; bid < 8 * w.per_xcd; ++bid) {
    int grp = -1, item = -1;
    if (!tmx::work_position(w, tmx::spread_workgroup(w, bid), grp, item)) grp = item = -1;
    printf("%d %d %d\n", bid, grp, item);
  }
  return 0;
}
