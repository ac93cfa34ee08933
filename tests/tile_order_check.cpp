// Host check of the order in which the persistent grid takes its work
// (tile_of_ticket in flash_attn_npu_amd/csrc/fa_plan.cpp), built and run by
// tests/test_tile_order.py: against lists written out by plain loops, every
// (head, m-tile, KV run) comes exactly once, at the ticket that its list gives,
// and a grid of one workgroup per unit has as many workgroups on a queue as the
// queue has tickets.
#include <stdio.h>
#include <stdlib.h>

#include <vector>

#include "fa_plan.cpp"

struct Unit {
  int bh, mt, split;
};

static void check(int heads, int m, int splits, int nq, bool causal, int grid) {
  // The queues' lists by loops: groups of 8 of a queue's own heads x, x + nq, ...;
  // KV run by KV run, heaviest m-tile first, head by head.  The tiles of the heads
  // left over go to the queues in turn, with the last group, after each rank's own
  // heads (with fewer than 8 queues the last group's heads all go in turn);
  // or, non-causal, one is a whole head of queue 0's.
  std::vector<std::vector<Unit>> queue(nq);
  const int per_queue = heads / nq, left = heads % nq, own = heads - left, units = heads * m * splits;
  const TileOrder o = make_tile_order(heads, m, splits, nq, causal, grid, 256);
  const bool whole = o.heads0 != o.heads;
  if (whole && (causal || left != 1 || units <= grid)) {
    printf("FAIL whole: heads %d m %d splits %d nq %d causal %d grid %d\n", heads, m, splits, nq, (int)causal, grid);
    exit(1);
  }
  const bool turns = left != 0 && !whole;
  int turn = 0;
  for (int h0 = 0; h0 < per_queue; h0 += 8) {
    const bool last = h0 + 8 >= per_queue;
    const int lo = nq * h0, hi = last ? own : nq * (h0 + 8);
    for (int s = 0; s < splits; ++s)
      for (int k = 0; k < m; ++k) {
        const int mt = causal ? m - 1 - k : k;
        for (int h = lo; h < hi; ++h) queue[last && turns && nq != 8 ? turn++ % nq : h % nq].push_back({h, mt, s});
        if (last)
          for (int h = own; h < heads; ++h) queue[whole ? 0 : turn++ % nq].push_back({h, mt, s});
      }
  }
  std::vector<int> seen((size_t)units);
  for (int x = 0; x < nq; ++x) {
    const uint32_t n = queue_tickets(o, x);
    bool ok = n == queue[x].size() && (whole || n == (uint32_t)(units - x + nq - 1) / nq);
    for (uint32_t t = 0; ok && t < n; ++t) {
      int bh = -1, mt = -1, split = -1;
      tile_of_ticket(o, x, t, causal, &bh, &mt, &split);
      const Unit &u = queue[x][t];
      ok = bh == u.bh && mt == u.mt && split == u.split && ++seen[((size_t)bh * m + mt) * splits + split] == 1;
    }
    if (!ok) {
      printf("FAIL heads %d m %d splits %d nq %d causal %d queue %d\n", heads, m, splits, nq, (int)causal, x);
      exit(1);
    }
  }
}

int main() {
  long n = 0;
  for (int heads = 1; heads <= 140; ++heads)
    for (int nq = 1; nq <= 8 && nq <= heads; ++nq)
      for (int m : {1, 2, 3, 7, 8, 29})
        for (int splits : {1, 2, 3, 7})
          for (int causal = 0; causal < 2; ++causal)
            for (int grid : {nq, 64, 512, heads * m * splits}) {
              if (grid > heads * m * splits) grid = heads * m * splits;
              check(heads, m, splits, nq, causal != 0, grid);
              ++n;
            }
  check(1023, 5, 1, 8, true, 512);
  check(1025, 5, 1, 8, false, 512);
  check(8, 4099, 1, 8, true, 512);
  // The largest counts the planner lets through, up to 2^31 - 1 units: the last tickets.
  const int big[4][2] = {{1, 2147483647}, {2147483647, 1}, {715827881, 3}, {9, 238609294}};
  for (const auto &b : big) {
    const TileOrder o = make_tile_order(b[0], b[1], 1, b[0] < 8 ? 1 : 8, false, 512, 256);
    for (int x = 0; x < o.nq; ++x) {
      int bh = -1, mt = -1, split = -1;
      tile_of_ticket(o, x, queue_tickets(o, x) - 1, false, &bh, &mt, &split);
      if (bh < 0 || bh >= b[0] || mt < 0 || mt >= b[1] || split != 0) {
        printf("FAIL big %d %d: %d %d %d\n", b[0], b[1], bh, mt, split);
        return 1;
      }
    }
  }
  printf("tile order ok: %ld forms\n", n);
}
