// Host run of the varlen work order (csrc/fa_common.h): every item of a launch is handed out once, whatever the span
// the launcher chooses.  Prints the number of launches whose items are not a permutation.
#include <cstdio>
#include <vector>

#include "fa_common.h"

static bool permutation(int n_kv, int group, int n_mblocks, bool heavy, int span) {
  const int total = n_kv * group * n_mblocks;
  std::vector<char> seen(total, 0);
  for (int L = 0; L < total; ++L) {
    int mb = -1, grp = -1;
    if (!fa::work_item_kv_rr(L, total, n_mblocks, group, heavy, span, mb, grp)) return false;
    if (mb < 0 || mb >= n_mblocks || grp < 0 || grp >= n_kv * group || seen[grp * n_mblocks + mb]++) return false;
  }
  return true;
}

int main() {
  int wrong = 0;
  for (int n_kv : {1, 3, 7, 8, 9, 16, 27, 40})
    for (int group : {1, 4, 8})
      for (int n_mblocks : {1, 2, 5, 16})
        for (int64_t rows : {1, 4, 64, 300, 2048, 16384, 1 << 20})
          for (int heavy = 0; heavy < 2; ++heavy)
            wrong += !permutation(n_kv, group, n_mblocks, heavy, fa::kv_rr_span(rows, 64, 1, n_kv));
  // 1 M and 2 M queries of 64 heads per K/V head against a handful of keys: 4096 spans' worth of items is 2^31, 2^32.
  for (int n_mblocks : {8192, 16384})
    for (int n_kv : {1, 8, 9}) wrong += !permutation(n_kv, 64, n_mblocks, true, fa::kv_rr_span(4, 64, 1, n_kv));
  std::printf("wrong %d\n", wrong);
  return wrong != 0;
}
