// Sizes of the layer, the fixed DeepSeek-V3/R1 routed-expert layer of the
// reference (kernels/moe.cu:41-53, reference/moe_ref.py:27-46), and the choices
// of a launch that follow from sizes alone.  No HIP here: the CPU tests compile
// this file by itself.
#pragma once

namespace moe {

constexpr int H = 7168;            // hidden size
constexpr int I = 2048;            // expert intermediate size
constexpr int G1 = 2 * I;          // W13 rows (gate rows 0..I-1, up rows I..2I-1)
constexpr int E_GLOBAL = 256;
constexpr int N_GROUP = 8;
constexpr int GROUP_SIZE = E_GLOBAL / N_GROUP;  // 32
constexpr int TOP_K = 8;
constexpr int TOPK_GROUP = 4;
constexpr int BLK = 128;           // scale block along every K/N axis
constexpr int HB = H / BLK;        // 56 hidden blocks
constexpr int IB = I / BLK;        // 16 intermediate blocks
constexpr int G1B = G1 / BLK;      // 32 W13 row blocks
constexpr int MAX_E_LOCAL = 32;    // dispatch uses a 32-bit local-expert mask per token
constexpr float E4M3_MAX = 448.0f;
// Largest token count served by the decode kernels (dispatch fused into GEMM1).
constexpr int DECODE_MAX_T = 128;
// Work-queue words of the prefill GEMMs, for each of the two: a claim
// counter per XCD, then a mask of the XCD segments found drained.
constexpr int XCDS = 8;
constexpr int QUEUE_COUNTERS = 2 * (XCDS + 1);

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

}  // namespace moe
