// Host-side dump of the attention kernels' position -> work-item mapping
// (work_position in attn_common.h, before spread_workgroup orders the positions) for
// tests/test_work_item.py:
//   work_item_dump groups m_blocks group ilv  ->  one line per position: "position item"
//   work_item_dump --ilv max_seqlen_k head_dim  ->  interleave_groups
#include <cstdio>
#include <cstdlib>

#include "attn_common.h"

int main(int argc, char** argv) {
  if (argc == 4 && argv[1][0] == '-') {
    printf("%d\n", tmx::interleave_groups(atol(argv[2]), atoi(argv[3])));
    return 0;
  }
  if (argc != 5) return 2;
  const long groups = atol(argv[1]), m_blocks = atol(argv[2]), group = atol(argv[3]);
  const int ilv = atoi(argv[4]);
  const long ipg = m_blocks * group;
  const long total = groups * ipg;
  const long grid = 8 * tmx::work_items_per_xcd(groups, ipg);
  const tmx::WorkMap w = tmx::make_work_map((int)total, (int)ipg, ilv, 1, 1);
  for (long p = 0; p < grid; ++p) {
    int grp, item;
    printf("%ld %ld\n", p, tmx::work_position(w, (int)p, grp, item) ? grp * ipg + item : -1L);
  }
  return 0;
}
