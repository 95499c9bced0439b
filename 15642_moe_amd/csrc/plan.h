// The choices of a launch that follow from sizes alone.  No HIP here: the CPU
// tests compile this file by itself.
#pragma once

#include "common.h"

#ifdef __HIPCC__
#define MOE_HD __host__ __device__ __forceinline__
#else
#define MOE_HD inline
#endif

namespace moe {

// ---------------------------------------------------------------------------
// Upstream producer (upstream.hip): a workgroup covers RQ_TOK tokens x one
// 16-expert tile per wave x one of router_k_parts(T) ranges of K-blocks.
// ---------------------------------------------------------------------------
constexpr int RQ_TOK = 64;            // tokens per workgroup (4 tiles of 16)
constexpr int RQ_ET = E_GLOBAL / 16;  // expert tiles of 16, one per wave

// K parts per launch: the fewest that give at least 448 workgroups of four waves (about
// two per CU; the K loop's dependent steps leave one workgroup per CU short
// of the HBM rate), each part a multiple of the ring depth in K-blocks.
// Measured: T=4096 51.5 -> 42.7 us with 2 parts (512 workgroups) instead of
// 1; more parts than that lose to the partial sums' traffic and reduction
// (T=8192 with 2 parts: 77 -> 81 us; T=1024 with 14: 19.9 -> 25.5 us).
inline int router_k_parts(int T) {
  const int groups = 4 * ((T + RQ_TOK - 1) / RQ_TOK);
  const int parts[] = {1, 2, 7, 14};
  for (int p : parts)
    if (groups * p >= 448) return p;
  return 14;
}

// Waves per workgroup: 16, 8 or 4, on a GPU of `cus` CUs.  One workgroup of 16
// or 8 waves runs per CU, and all workgroups of a token tile run on one XCD
// (tile t on XCD t % XCDS), so a round is an XCD's CUs and the XCD with the
// most token tiles sets the rounds.  16 waves are taken where they fill 7/10
// of their rounds and 8 waves where they fill 8/10 (9/10 for several rounds
// over the whole K range, whose last one is long); parts of a single ring
// (14 K parts, small T) stay with four waves, which spread over more CUs.
// Counted over the chip instead of an XCD, T=2198..2560 (35 workgroups of 16
// waves for 32 CUs) took 35.7 us where four waves take 33.5, and T=3222 47.0
// with 8 waves where 16 take 38.9.
// Same K parts, 4 / 8 / 16 waves, us: T=2048 29.3 / 27.9 / 23.4, T=2560 35.0 /
// 36.3 / 36.2, T=3072 40.9 / 39.4 / 38.1, T=3222 45.0 / 46.9 / 38.9, T=4096
// 33.2 / 29.6 / 40.0, T=6144 45.6 / 52.1 / 42.4, T=8192 63.3 / 53.3 / 77.5,
// T=10752 95.5 / 110.8 / 95.6, T=13312 120.9 / 116.8 / 101.3, T=16384 132.7 /
// 126.1 / 110.1, T=20480 163.3 / 180.9 / 192.8, T=24064 193.3 / 186.8 / 200.1.
inline int router_waves(int T, int cus) {
  const int n_kp = router_k_parts(T), xcd_cus = cus / XCDS > 0 ? cus / XCDS : 1;
  const int tiles = (T + RQ_TOK - 1) / RQ_TOK, xcd_tiles = (tiles + XCDS - 1) / XCDS;
  if (n_kp == 14) return 4;
  for (int waves = 16; waves > 4; waves /= 2) {
    const int groups = RQ_ET / waves * xcd_tiles * n_kp;
    const int rounds = (groups + xcd_cus - 1) / xcd_cus;
    const int tenths = n_kp == 1 && rounds > 1 ? 9 : waves == 16 ? 7 : 8;
    if (10 * groups >= tenths * rounds * xcd_cus) return waves;
  }
  return 4;
}

// The most local experts that T tokens can hit.
inline int decode_experts(int T, int e_local) { return T * TOP_K < e_local ? T * TOP_K : e_local; }

// Waves that share the K range of a decode GEMM2 item (expert, 64 weight rows):
// four, so that an item has more loads in flight; one above 64 tokens where
// the items nearly fill the chip and are all resident at once as single waves
// (two per SIMD: more than 6 and at most 8 per CU, 14 to 18 local experts), which
// four-wave workgroups, two per CU, need 3.1 to 3.9 rounds for.  Whole call,
// weights not in cache, four waves / one, us: even routing, 16 local experts T=72
// 122.3 / 119.3, T=128 128.5 / 125.2 (and the next call's GEMM1 with it), 14 T=96
// 117.5 / 114.6, 18 T=96 145.7 / 144.2; uneven, 16 T=128 86.3 / 87.1; skewed,
// 16 T=128 220 / 230 (231 before the split).  Outside: 12, even T=128 99.0 /
// 99.0, 19 149.6 / 151.5, 32 231.9 / 239.1; 16, even T=48 115.1 / 114.3, T=64
// 119.2 / 118.8.
inline int stage2_decode_waves(int T, int e_local, int cus) {
  const int items = decode_experts(T, e_local) * (H / 64);
  return T > 64 && items > 6 * cus && items <= 8 * cus ? 1 : 4;
}

// Whether both prefill GEMMs of T tokens run in the 256 x 256-tile kernels of
// prefill_wide.hip: with at least 16 local experts, from T = 3072 on (96 expected
// routes per expert), or 3456 (108) where an item per weight block is at most one
// per CU: such a launch is a single round of the kernels of prefill.hip too, as
// long as no expert has more than 128 routes (108 and twice the deviation of
// even routing), and a wide item takes longer to stream its weights.
// Whole forward, weights not in cache, prefill.hip / wide, us:
//   32 local experts, even  T=2800 306 / 316, 3072 319 / 322, 3200 333 / 325, 3500
//     368 / 330, 4096 418 / 347, 8192 576 / 542, 16384 996 / 909
//     uneven 2500 / 3072 / 4096 / 8192: 0.96, 0.97, 0.95, 0.93 of prefill.hip's
//     time; skewed 3072 885 / 812, 4096 1098 / 985
//   24, even   3072 262 / 267, 3500 271 / 273, 4096 331 / 283; uneven 3072 297 / 281
//   17, even   3072 224 / 226, 3500 227 / 229, 5000 270 / 259; uneven 3072 219 / 220
//   16, even   3072 175 / 185, 3231 177 / 188, 3341 176 / 189, 3474 189 / 192, 3526
//     215 / 194, 4096 236 / 196, 4329 195 / 199, 4910 206 / 206, 5500 252 / 222, 8192
//     317 / 314; uneven 3176 190 / 186, 3326 218 / 207, 3561 232 / 220; skewed 3335
//     848 / 780
// With 8 local experts a 256-row item per weight block leaves CUs without work
// unless the routing is skewed: T=4096 143 / 163, T=8192 199 / 207, skewed
// T=4096 936 / 835.
inline bool prefill_wide(int T, int e_local, int cus) {
  return e_local >= 16 && T >= (e_local * IB <= cus ? 3456 : 3072);
}

// ---------------------------------------------------------------------------
// Work lists of the wide prefill GEMMs (prefill_wide.hip): which tile size a
// launch takes, which items an XCD's queue holds and in which order.
// ---------------------------------------------------------------------------
constexpr int WORK_BAND = 8;  // route tiles of a band (see decode_work in gemm_util.h)

// A launch's tile sizes, in 32-route fragments, and an item's cost by its
// fragments, of which only the ratio matters: what a K-block of an item takes
// beside its fragments (weights, barriers, LDS latency) is worth about 8
// fragments where most items of a launch have few of them.
// The launch's length is estimated as whole rounds of items over the
// workgroups x the mean item, and the least one's size is taken; sizes 3 and 2
// only where tiles of 4 leave some workgroup without an item, since cutting
// finer only then puts idle CUs to work.  Over 1000 launches (16 to 32 local
// experts, T = 3072 .. 16384, even, uneven and skewed routing) the choice takes
// 1.0% more than the best of the five sizes in the mean and 6% in the worst
// 20th; with sizes 3 and 2 always open 1.2% and 7% (even routing, T=3300 with
// 18 experts: 5% slower than the kernels of prefill.hip instead of equal).
// An estimate from the items' sum, max(largest item, sum / CUs + half an item),
// is 2.8 to 3.7% off for GEMM1, with these costs or with a full tile's clocks.
constexpr int TILE_SIZES = 5, TILE_COARSE = 3;  // the first TILE_COARSE are always open
constexpr int TILE_FRAGS[TILE_SIZES] = {8, 6, 4, 3, 2};
constexpr float ITEM_COST = 1500.0f, FRAG_COST = 190.0f;

MOE_HD int route_frags(int routes) { return (routes + 31) >> 5; }
MOE_HD int route_tiles(int frags, int tile_frags) { return (frags + tile_frags - 1) / tile_frags; }
// First route of tile mt (0 .. nt) of an expert with f fragments in nt tiles:
// the fragments are dealt evenly.
MOE_HD int tile_first_route(int mt, int f, int nt) { return 32 * ((mt * f) / nt); }

// A launch of `tiles` route tiles with `frags` fragments in all, each x nblk
// weight blocks, over `workgroups`.
MOE_HD float launch_estimate(int tiles, int frags, int nblk, int workgroups) {
  const int rounds = (tiles * nblk + workgroups - 1) / workgroups;
  return (float)rounds * (ITEM_COST + FRAG_COST * ((float)frags / (float)(tiles > 0 ? tiles : 1)));
}
// Index into TILE_FRAGS; `fine`: tiles of 4 give at most one item per workgroup.
MOE_HD int pick_tile(const float* est, bool fine) {
  int best = 0;
  for (int i = 1; i < TILE_SIZES; ++i)
    if ((i < TILE_COARSE || fine) && est[i] < est[best]) best = i;
  return best;
}

// Order of the experts: by fragments per item (key), descending.
MOE_HD bool expert_before(int key_a, int a, int key_b, int b) { return key_a > key_b || (key_a == key_b && a < b); }
// Place in the order of the i-th expert of queue x: descending in the even
// queues, ascending in the odd ones.
MOE_HD int order_place(int x, int i) { return x & 1 ? MAX_E_LOCAL - 1 - i : i; }
// Items of queue x from the expert at place p of the order, which has nt route
// tiles and U quads of weight blocks: quad j is queue (U * p + j) % XCDS's.
MOE_HD int queue_items(int x, int U, int p, int nt) { return ((x - U * p) & (XCDS - 1)) < U ? 4 * nt : 0; }
// Weight block and route tile of the local-th of them: bands of WORK_BAND
// route tiles, then weight block, then route tile.
MOE_HD void queue_item(int x, int U, int p, int nt, int local, int& blk, int& mt) {
  const int full = nt / WORK_BAND, b = local / (4 * WORK_BAND), band = b < full ? b : full;
  const int width = b < full ? WORK_BAND : nt - full * WORK_BAND;
  const int r = local - band * 4 * WORK_BAND;
  blk = 4 * ((x - U * p) & (XCDS - 1)) + r / width;
  mt = band * WORK_BAND + r % width;
}

}  // namespace moe
