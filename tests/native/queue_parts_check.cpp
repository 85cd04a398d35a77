// Host-side check of the work-item map with split video tiles in any number
// of parts (lvsa_attn_kernels.h: queue_shape, queue_item, static_grid): every
// tile is taken once, whole or once per part with one slot, and the grid of a
// launch without queues reaches every item.  Prints "queue parts ok".
#include "lvsa_attn_kernels.h"

#include <cstdio>
#include <map>
#include <random>
#include <set>
#include <vector>

using namespace lvsa;

int main() {
  std::mt19937 rng(2);
  for (int trial = 0; trial < 5000; ++trial) {
    AttnParams p{};
    p.B = 1 + rng() % 2;
    p.H = 1 + rng() % 24;
    p.n_vt = rng() % 30;
    p.n_tt = rng() % 2;
    p.text_chunks = p.n_tt ? 1 + rng() % 4 : 1;
    p.text_first = p.text_chunks == 1;
    p.vsplit = rng() % 20;
    p.vparts = 2 + rng() % 7;
    p.n_vwork = p.n_vt * p.H * p.B;
    p.n_twork = p.n_tt * p.text_chunks * p.H * p.B;
    std::vector<int> whole(p.n_vwork, 0);
    std::vector<std::set<int>> parts(p.n_vwork);
    std::map<int, int> tile_of_slot;
    int text = 0, items = 0;
    for (int b = 0; b < static_grid(p); ++b) {
      const int x = b % kXcds, j = b / kXcds;
      if (j >= queue_items(queue_shape(p, x))) continue;
      const WorkItem it = queue_item(p, x, j);
      ++items;
      if (it.text) {
        ++text;
        continue;
      }
      const int w = (it.batch * p.H + it.head) * p.n_vt + it.tile;
      if (it.vhalf < 0) {
        ++whole[w];
        continue;
      }
      if (it.vhalf >= p.vparts || it.vslot >= kXcds * p.vsplit || !parts[w].insert(it.vhalf).second ||
          (tile_of_slot.count(it.vslot) && tile_of_slot[it.vslot] != w)) {
        printf("trial %d: part %d of slot %d\n", trial, it.vhalf, it.vslot);
        return 1;
      }
      tile_of_slot[it.vslot] = w;
    }
    long expect = p.n_twork;
    for (int w = 0; w < p.n_vwork; ++w) {
      if (!((whole[w] == 1 && parts[w].empty()) || (whole[w] == 0 && (int)parts[w].size() == p.vparts))) {
        printf("trial %d: tile %d taken %d times and in %d parts\n", trial, w, whole[w], (int)parts[w].size());
        return 1;
      }
      expect += whole[w] ? 1 : p.vparts;
    }
    if (text != p.n_twork || items != expect) {
      printf("trial %d: %d text items of %d, %d items of %ld\n", trial, text, p.n_twork, items, expect);
      return 1;
    }
  }
  printf("queue parts ok\n");
  return 0;
}
