// The launch choices of 15642_moe_amd/csrc/plan.h as C functions for tests/test_plan.py.
#include "plan.h"

extern "C" {

int plan_router_k_parts(int T) { return moe::router_k_parts(T); }
int plan_router_waves(int T, int cus) { return moe::router_waves(T, cus); }

int plan_stage2_decode_waves(int T, int e_local, int cus) { return moe::stage2_decode_waves(T, e_local, cus); }
int plan_prefill_wide(int T, int e_local, int cus) { return moe::prefill_wide(T, e_local, cus); }

// The tile size (fragments) that a wide prefill GEMM with nblk weight blocks per expert takes.
int plan_wide_tile(const int* counts, int e_local, int nblk, int workgroups) {
  float est[moe::TILE_SIZES];
  bool fine = false;
  for (int i = 0; i < moe::TILE_SIZES; ++i) {
    int tiles = 0, frags = 0;
    for (int e = 0; e < e_local; ++e) {
      tiles += moe::route_tiles(moe::route_frags(counts[e]), moe::TILE_FRAGS[i]);
      frags += moe::route_frags(counts[e]);
    }
    est[i] = moe::launch_estimate(tiles, frags, nblk, workgroups);
    if (i == moe::TILE_COARSE - 1) fine = tiles * nblk <= workgroups;
  }
  return moe::TILE_FRAGS[moe::pick_tile(est, fine)];
}

// Its items with that tile size, queue by queue: (queue, expert, weight block, first route, routes) each.
// Returns their number, or -1 where `room` items are not enough.
int plan_wide_items(const int* counts, int e_local, int nblk, int tile, int* items, int room) {
  int nt[moe::MAX_E_LOCAL], key[moe::MAX_E_LOCAL], ord[moe::MAX_E_LOCAL], n = 0;
  for (int e = 0; e < moe::MAX_E_LOCAL; ++e) {
    const int f = e < e_local ? moe::route_frags(counts[e]) : 0;
    nt[e] = moe::route_tiles(f, tile);
    key[e] = nt[e] ? moe::route_tiles(f, nt[e]) : 0;
  }
  for (int e = 0; e < moe::MAX_E_LOCAL; ++e) {
    int rank = 0;
    for (int j = 0; j < moe::MAX_E_LOCAL; ++j) rank += moe::expert_before(key[j], j, key[e], e);
    ord[rank] = e;
  }
  for (int x = 0; x < moe::XCDS; ++x)
    for (int i = 0; i < moe::MAX_E_LOCAL; ++i) {
      const int p = moe::order_place(x, i), e = ord[p], count = moe::queue_items(x, nblk / 4, p, nt[e]);
      for (int local = 0; local < count; ++local, ++n) {
        if (n == room) return -1;
        int blk, mt;
        moe::queue_item(x, nblk / 4, p, nt[e], local, blk, mt);
        const int f = moe::route_frags(counts[e]), first = moe::tile_first_route(mt, f, nt[e]);
        const int end = moe::tile_first_route(mt + 1, f, nt[e]);
        int* it = items + 5 * n;
        it[0] = x, it[1] = e, it[2] = blk, it[3] = first, it[4] = (end < counts[e] ? end : counts[e]) - first;
      }
    }
  return n;
}

}
