// Prefill grouped FP8 GEMMs for large batches (launch_stage1_wide /
// launch_stage2_wide) on v_mfma_f32_32x32x64_f8f6f4: the math, packed weights
// and results of prefill.hip's kernels (bit for bit), another structure.
//
// Item = (expert, 256 weight rows, up to 256 routes).  Eight waves in 4 row
// groups x 2 route groups, so a wave owns 64 rows (two 32-row operands) x up
// to 4 route tiles of 32, and each B fragment read from LDS feeds two MFMA
// chains.  Both operands reach LDS by direct global -> LDS loads
// (global_load_lds, no staging registers or LDS stores), which leaves the
// registers for the 128 accumulators that a 256 x 256 tile needs: 64 KB of
// operands per 16.8 MFLOP K-block step, where the register-staged 256 x 192
// tile moves 56 KB per 12.6.
//
// What a step is bound by.  The MFMA pipe alone needs 2048 clocks per K-block of
// a full tile.  Timing copies at skewed T=4096, before the wait states in front
// of the loads (dma16), took 2640 without any loads -- the two barriers and the
// weight fragments' LDS latency, ~400, and 280-290 per route tile where the pipe
// needs 256 -- and 2640-2840 with them.  The instruction order inside a route
// tile matters more than anything else (below); all loads at the step's start
// instead of one behind each MFMA cost 540 clocks.  Over whole launches, where
// most tiles are partial, the counters point to the operands' arrival: at T=8192
// the pipe is busy 44% (GEMM1) and 35% (GEMM2) of the cycles, the waves wait 42%
// and 48% of theirs, and the L1 is stalled ~40% on L2 data; GEMM1 moves 1.37 GB
// from beyond L2 (1.7x its algorithmic bytes) at 4.7 TB/s.  At full density the chip lowers
// its clock (2.2 -> 1.7-1.9 GHz), which takes back about half of what the step
// gains.  The wait states cost 1 to 5% of GEMM1.
//
// Measured against the register-staged kernels on the same box (GEMM1 / GEMM2
// us): T=16384 even routing 557 / 342 -> 500 / 328, T=8192 uneven 314 / 179 ->
// 290 / 179, skewed T=4096 623 / 381 -> 519 / 355, T=4096 even 248 / 137 -> 198
// / 132.
#include "common.h"
#include "gemm_util.h"
#include "launch.h"

#include <type_traits>

namespace moe {
namespace {

constexpr int WNT = 512;                       // 8 waves: 4 row groups x 2 route groups
constexpr int RT = 32;                         // routes per route tile
constexpr int FRAG = 4096;                     // one 32-row operand's K-block
constexpr int W_SLOT = 8 * FRAG;               // a K-block of the item's weights in LDS

// MAXC route tiles of 32 per wave at most; an item has up to 2 * MAXC.
template <int MAXC>
struct WideGeom {
  static constexpr int BM = 2 * MAXC * RT;
  static constexpr int ACT_SLOT = 2 * MAXC * FRAG;
  static constexpr int SCL_SLOT = 2 * MAXC * 64;  // floats
};

// Direct global -> LDS loads: lane l's 16 (4) bytes at sbase + voff land at
// LDS address lds + 16 l (4 l).  M0 holds the LDS address.  It is an operand
// that the compiler writes: it uses M0 too (as the lane select of v_writelane,
// in the wave reduction around the queue's atomics).  The loads are counted by
// vmcnt like any other, and the compiler knows nothing of them: every wait is
// explicit (landed_barrier, wait_loads).  The wait states in front cover M0's
// write and a base address that a VALU instruction has just written (the
// reload of a spilled scalar register; five states to its use by a memory
// instruction, which the compiler does not insert for inline assembly).
// NTL: non-temporal.  K, which the assembly carries as a comment: what the load
// brings, by which a test follows the counted waits.
enum LoadKind { K_WEIGHTS, K_ACTIVATIONS, K_TABLES };
template <bool NTL, LoadKind K>
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t voff, const void* sbase) {
  if constexpr (NTL)
    __asm__ volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2 nt ; kind %3"
                     ::"{m0}"(lds), "v"(voff), "s"(sbase), "n"(K) : "memory");
  else
    __asm__ volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2 ; kind %3"
                     ::"{m0}"(lds), "v"(voff), "s"(sbase), "n"(K) : "memory");
}
template <LoadKind K>
__device__ __forceinline__ void dma4(uint32_t lds, uint32_t voff, const void* sbase) {
  __asm__ volatile("s_nop 4\n\tglobal_load_lds_dword %1, %2 ; kind %3"
                   ::"{m0}"(lds), "v"(voff), "s"(sbase), "n"(K) : "memory");
}
// All but this wave's N youngest loads have landed and its LDS reads are done;
// then all waves meet.
template <int N>
__device__ __forceinline__ void landed_barrier() {
  __asm__ volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
__device__ __forceinline__ void plain_barrier() { __asm__ volatile("s_barrier" ::: "memory"); }

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
__device__ __forceinline__ float lane_value(float v, int k) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
}
__device__ __forceinline__ uint32_t a_lane_offset(int lane) {
  return (uint32_t)(((lane & 31) >> 4) * TILE_BYTES + (16 * (lane >> 5) + (lane & 15)) * 16);
}
// Reads at 32-bit LDS addresses (constant parts fold into the instruction's offset).
using lds_u32x4 = const __attribute__((address_space(3))) u32x4;
using lds_float = const __attribute__((address_space(3))) float;
__device__ __forceinline__ v8i lds_op(uint32_t lo, uint32_t hi) {
  const u32x4 l = *(lds_u32x4*)(uintptr_t)lo, h = *(lds_u32x4*)(uintptr_t)hi;
  return frag(l, h);
}
__device__ __forceinline__ float lds_f32(uint32_t a) { return *(lds_float*)(uintptr_t)a; }

// One wave's accumulators and products: 64 weight rows (two 32-row operands)
// x NC route tiles.  NS: weight scales per route tile (2: gate and up, 1).
template <int NC, int NS>
struct WideAcc {
  static constexpr int ND = NC > 0 ? NC : 1;
  v16f acc[2][ND];
  v16f p[2];
  float sg[2], su[2];

  // acc += p * scale for half h (8 registers) of operand op's product.
  __device__ __forceinline__ void finish(int op, int cc, int ss, int h) {
#pragma unroll
    for (int r = 8 * h; r < 8 * h + 8; ++r) acc[op][cc][r] += p[op][r] * ((NS == 2 && r >= 8) ? su[ss] : sg[ss]);
    __asm__ volatile("" : "+v"(acc[op][cc]));
  }
};

// An item as one wave sees it (wave-uniform values).
struct WideItem {
  int nb, rows, rb, ncw, tile0;
  bool nt;
  const uint8_t* wsrc;
  uint32_t sofs;  // byte offset of the item's first weight scales
};

// The lane number, computed afresh where it is used: derived per-lane offsets
// then need no registers across the K loop (hoisted, they were spilled, and
// every reload waited for the loads in flight).
__device__ __forceinline__ int fresh_lane() {
  int l = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  __asm__ volatile("" : "+v"(l));
  return l;
}
__device__ __forceinline__ void lds_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
template <int N>
__device__ __forceinline__ void wait_loads() { __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// ---------------------------------------------------------------------------
// Work distribution.  A launch's items are (local expert, weight block of 256
// rows, route tile); WideWork lists them per XCD queue.
//
// The arithmetic is plan.h's, which a CPU test compiles.
//
// Tile size: each expert's 32-route fragments are dealt evenly over
// ceil(fragments / tile) route tiles, with one tile size per launch, chosen
// from TILE_FRAGS by the launch's estimated length: a few experts with many
// routes are cut finer where whole tiles would leave CUs without an item.
// Order: experts by fragments per item, descending in the even queues and
// ascending in the odd ones: items of few routes stream weights from HBM and
// large ones keep the MFMA pipe busy, and the launch is shortest with both
// running at once (skewed T=4096 GEMM1: 493 us, all queues descending 520, ascending
// in queues 4-7 508; T=16384: 485, 489, 489).
// Queues: an expert's weight blocks are cut into quads (U per expert); quad j
// of the expert at place p belongs to XCD (U * p + j) % 8, so an expert's quads lie
// on different XCDs and each XCD has at most one of them (U <= 8), holds a
// share of every cost class, and runs 4 weight blocks x up to 8 route tiles at
// a time, which share their fetches into its L2 as far as they stay in step
// (skewed T=4096: GEMM1 moves 1.9x its algorithmic bytes, the register-staged
// kernels 2.0x; T=8192: 1.7x and 1.5x).  Within a quad: bands of
// WORK_BAND route tiles, then weight block, then route tile.
// ---------------------------------------------------------------------------
struct WideWork {
  int ord[MAX_E_LOCAL];                   // the expert at each place of the order
  int cnt[MAX_E_LOCAL], off[MAX_E_LOCAL], nt[MAX_E_LOCAL];  // per expert: routes, first route, route tiles
  int first[XCDS][MAX_E_LOCAL + 1];       // first[x][i]: items of queue x before its i-th expert's
  float est[TILE_SIZES];                  // the launch's estimated length with each tile size
  int fine;                               // sizes below 4 fragments are open
};

__device__ __forceinline__ int sum32(int v) {
#pragma unroll
  for (int d = 1; d < 32; d <<= 1) v += __shfl_xor(v, d, 32);
  return v;
}

template <int NBLK, int U>
__device__ __forceinline__ void build_work(WideWork& wk, const int32_t* __restrict__ counts,
                                           const int32_t* __restrict__ offsets, int e_local) {
  static_assert(NBLK == 4 * U && U <= XCDS, "quads");
  static_assert(TILE_SIZES <= WNT / 64 && TILE_FRAGS[TILE_COARSE - 1] == 4, "one tile size per wave");
  const int e = threadIdx.x & 31, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = e < e_local ? counts[e] : 0, o = e < e_local ? offsets[e] : 0;
  const int f = route_frags(c);
  if (wave < TILE_SIZES) {
    const int tiles = sum32(route_tiles(f, TILE_FRAGS[wave])), frags = sum32(f);
    if (threadIdx.x % 64 == 0) {
      wk.est[wave] = launch_estimate(tiles, frags, NBLK, (int)gridDim.x);
      if (wave == TILE_COARSE - 1) wk.fine = tiles * NBLK <= (int)gridDim.x;
    }
  }
  __syncthreads();
  const int k = TILE_FRAGS[pick_tile(wk.est, wk.fine)];
  if (threadIdx.x < MAX_E_LOCAL) {
    const int nt = route_tiles(f, k), key = nt ? route_tiles(f, nt) : 0;
    int rank = 0;
#pragma unroll
    for (int j = 0; j < MAX_E_LOCAL; ++j) {
      rank += expert_before(__builtin_amdgcn_readlane(key, j), j, key, e) ? 1 : 0;
    }
    wk.ord[rank] = e;
    wk.cnt[e] = c;
    wk.off[e] = o;
    wk.nt[e] = nt;
  }
  __syncthreads();
  if (threadIdx.x < XCDS * MAX_E_LOCAL) {
    const int x = threadIdx.x >> 5, i = e, p = order_place(x, i);
    int inc = queue_items(x, U, p, wk.nt[wk.ord[p]]);
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
      const int y = __shfl_up(inc, d, 32);
      if (i >= d) inc += y;
    }
    wk.first[x][i + 1] = inc;
    if (i == 0) wk.first[x][0] = 0;
  }
  __syncthreads();
}

// Item idx of queue x -> expert, weight block, route tile.
template <int U>
__device__ __forceinline__ void work_item(const WideWork& wk, int x, int idx, int& e, int& blk, int& mt) {
  const int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) & 31;
  const int i = __builtin_ctzll(__ballot(wk.first[x][l] <= idx && idx < wk.first[x][l + 1]));
  const int p = order_place(x, i);
  e = __builtin_amdgcn_readfirstlane(wk.ord[p]);
  const int nt = __builtin_amdgcn_readfirstlane(wk.nt[e]);
  const int local = idx - __builtin_amdgcn_readfirstlane(wk.first[x][i]);
  queue_item(x, U, p, nt, local, blk, mt);
}

// Claims of a persistent workgroup (wave 0's lane 0): its own XCD's queue
// first, then the others', as ItemQueue in gemm_util.h.  An item is
// (queue << 24) + index, -1 when every queue is drained.
struct WideQueue {
  int cur, claimed;
  __device__ __forceinline__ void claim(int32_t* queue) { claimed = atomicAdd(&queue[cur], 1); }
  __device__ __forceinline__ int next(int32_t* queue, const WideWork& wk) {
    constexpr unsigned all = (1u << XCDS) - 1u;
    for (;;) {
      if (claimed < wk.first[cur][MAX_E_LOCAL]) return (cur << 24) + claimed;
      const unsigned m = atomicOr(reinterpret_cast<unsigned*>(&queue[XCDS]), 1u << cur) | (1u << cur);
      if ((m & all) == all) return -1;
      do cur = (cur + 1) & (XCDS - 1);
      while ((m >> cur) & 1u);
      claim(queue);
    }
  }
};

// The K loop.  LDS holds two K-blocks of weights and two of activations and
// activation scales.  Step kb opens with a barrier (its K-block landed; every
// wave is done with kb - 1).  Each wave reads its two weight operands into
// registers, then walks its route tiles; behind each MFMA it issues one load:
// first the activations of kb + 1, then, past a second barrier in the first
// or second route tile (every wave holds its operands of kb, so their slot is
// free), the weights of kb + 2.  At the next opening barrier only those 4
// weight loads may be outstanding: weights have up to 1.7 steps to arrive,
// activations one.
//
// Order inside a route tile: M(a0,k0) F M(a0,k1) F M(a1,k0) F M(a1,k1) F, each
// F half (8) of the scale FMAs of the product finished before: the second
// operand's of the previous route tile, then the first operand's of this one.
// Two product buffers suffice, no FMA waits for the MFMA right before it, and
// the pipe always holds the next MFMA.  With all of a product's 16 FMAs in one
// place between MFMAs a full tile's step took a quarter longer.
//
// Between items: the next item is claimed during the last two steps; its
// tables, first weights and (stage 2) activations are loaded under the
// epilogue, and land before any store is issued, since loads and stores
// retire in order from one counter: the next item's first step waits for
// nothing.
template <int MAXC, bool S1>
__global__ void __launch_bounds__(WNT)
wide_kernel(const uint8_t* __restrict__ act, const float* __restrict__ ascale, const uint8_t* __restrict__ wp_all,
            const float* __restrict__ wscale, const int32_t* __restrict__ counts, const int32_t* __restrict__ offsets,
            const float* __restrict__ route_weight, const int32_t* __restrict__ route_token, uint8_t* __restrict__ Cq,
            float* __restrict__ Cs, float* __restrict__ Y, uint16_t* __restrict__ out, int T, int e_local,
            int32_t* __restrict__ queue) {
  using G = WideGeom<MAXC>;
  constexpr int BM = G::BM, KB = S1 ? HB : IB, NBLK = S1 ? IB : HB / 2, U = NBLK / 4;
  constexpr int KROW = S1 ? H : I;  // bytes per activation row
  constexpr size_t WKB = S1 ? W13_KB_BYTES : W2_KB_BYTES;
  constexpr int CQ_STRIDE = BLK + 16;
  static_assert(KB % 2 == 0 && KB >= 6, "two slots");
  // LDS: weight slots, activation slots, then bytes that extend the second
  // activation slot to stage 1's FP8 rows, and the scale slots.
  constexpr int EPI = S1 ? BM * CQ_STRIDE : 0;
  constexpr int L_A = 2 * W_SLOT, L_E = L_A + G::ACT_SLOT, L_S = L_E + (EPI > G::ACT_SLOT ? EPI : G::ACT_SLOT);
  static_assert(S1 || (RT * 2 * BLK * 4 <= W_SLOT && RT * 2 * BLK * 4 <= G::ACT_SLOT), "stage 2's fp32 rows fit a slot");
  __shared__ __attribute__((aligned(16))) uint8_t pool[L_S + 2 * G::SCL_SLOT * 4];
  __shared__ float s_red[S1 ? 4 : 1][S1 ? BM : 1], s_sc[S1 ? BM : 1];  // stage 1: amax per row group, scales
  __shared__ int s_rt[2][2][BM];   // route tokens and (stage 2) route weights of the current and the next item
  __shared__ float s_ws[2][2][64];  // their weight-block scales, K-block k at k
  __shared__ WideWork wk;
  __shared__ int s_item;

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w & 3, wc = w >> 2;
  WideQueue iq{(int)blockIdx.x & (XCDS - 1), 0};
  // Nothing of a claim stays in a register between take() and the next claim().
  auto claim = [&]() __attribute__((always_inline)) {
    iq.claimed = 0;
    if (w == 0 && fresh_lane() == 0) iq.claim(queue);
  };
  auto take = [&]() __attribute__((always_inline)) {
    if (w == 0 && fresh_lane() == 0) s_item = iq.next(queue, wk);
    iq.cur = __builtin_amdgcn_readfirstlane(iq.cur);
    iq.claimed = 0;
  };
  claim();  // the first claim's round trip runs under the table's loads
  build_work<NBLK, U>(wk, counts, offsets, e_local);
  const int op_w = 2 * wr + wc;  // the operand this wave loads
  const uint32_t lw = lds_addr(pool), la = lw + L_A, ls = lw + L_S;
  uint32_t aoff[MAXC], soff = 0;

  // Work item L for this wave.
  auto decode = [&](int L) __attribute__((always_inline)) {
    WideItem it;
    int e, mt;
    work_item<U>(wk, L >> 24, L & 0xFFFFFF, e, it.nb, mt);
    it.nb = __builtin_amdgcn_readfirstlane(it.nb);
    mt = __builtin_amdgcn_readfirstlane(mt);
    // fragments [mt * f / nt, (mt + 1) * f / nt) of the expert's f
    const int cnt = __builtin_amdgcn_readfirstlane(wk.cnt[e]), nt = __builtin_amdgcn_readfirstlane(wk.nt[e]);
    const int f = route_frags(cnt), m0 = tile_first_route(mt, f, nt);
    it.rows = min(cnt, tile_first_route(mt + 1, f, nt)) - m0;
    it.rb = __builtin_amdgcn_readfirstlane(wk.off[e]) + m0;
    const int ncc = (it.rows + RT - 1) / RT, nc0 = (ncc + 1) >> 1;
    it.ncw = wc ? ncc - nc0 : nc0;
    it.tile0 = wc ? nc0 : 0;
    it.nt = nt == 1;
    if constexpr (S1) {
      it.wsrc = wp_all + (size_t)(e * IB + it.nb) * W13_SLAB_BYTES + (size_t)op_w * FRAG;
      it.sofs = (uint32_t)(e * G1B + it.nb) * HB * 4u;
    } else {
      it.wsrc = wp_all + (size_t)(e * HB + 2 * it.nb + (op_w >> 2)) * W2_SLAB_BYTES + (size_t)(op_w & 3) * FRAG;
      it.sofs = (uint32_t)(e * HB + 2 * it.nb) * IB * 4u;
    }
    return it;
  };
  // Load i (of 4) of this wave's operand of K-block kb.
  auto issue_w1 = [&](const WideItem& it, uint32_t alane, int kb, int slot, int i) __attribute__((always_inline)) {
    const uint8_t* p = it.wsrc + (size_t)kb * WKB + (i >> 1) * 512 + (i & 1) * 1024;
    const uint32_t d = lw + slot * W_SLOT + op_w * FRAG + i * 1024;
    if (it.nt) dma16<true, K_WEIGHTS>(d, alane, p);
    else dma16<false, K_WEIGHTS>(d, alane, p);
  };
  auto issue_w = [&](const WideItem& it, int kb, int slot) __attribute__((always_inline)) {
    const uint32_t alane = a_lane_offset(fresh_lane());
#pragma unroll
    for (int i = 0; i < 4; ++i) issue_w1(it, alane, kb, slot, i);
  };
  auto issue_a1 = [&](const WideItem& it, int kb, int slot, int i) __attribute__((always_inline)) {
    dma16<false, K_ACTIVATIONS>(la + slot * G::ACT_SLOT + (it.tile0 + i) * FRAG + wr * 1024, aoff[i], act + (size_t)kb * BLK);
  };
  // 64 lanes: the 32 scales of one of the wave's route tiles, twice
  auto issue_s = [&](const WideItem& it, int kb, int slot) __attribute__((always_inline)) {
    dma4<K_ACTIVATIONS>(ls + slot * (G::SCL_SLOT * 4) + (it.tile0 + min(wr, it.ncw - 1)) * 256, soff,
         S1 ? ascale + (size_t)kb * T : ascale + kb);
  };
  // The item's tables, one load per wave: route tokens (waves 0-3), stage 2's
  // route weights (waves 4-7) or stage 1's weight scales (waves 4 and 5).
  auto issue_tables = [&](const WideItem& it, int par) __attribute__((always_inline)) {
    const int lane = fresh_lane();
    const int r = 64 * wr + lane;
    const uint32_t off = (uint32_t)(it.rb + (r < it.rows ? r : 0)) * 4u;
    if (wc == 0) {
      dma4<K_TABLES>(lds_addr(&s_rt[par][0][64 * wr]), off, route_token);
    } else if constexpr (!S1) {
      dma4<K_TABLES>(lds_addr(&s_rt[par][1][64 * wr]), off, route_weight);
    }
    if (wc == 1 && wr < 2)  // gate / up blocks nb, IB + nb; H blocks 2nb, 2nb + 1
      dma4<K_TABLES>(lds_addr(&s_ws[par][wr][0]), it.sofs + (uint32_t)(wr * (S1 ? IB * HB : IB) + min(lane, KB - 1)) * 4u, wscale);
  };
  // Per-lane row offsets of an item's activations and scales (stage 1: its
  // route tokens are in s_rt[par][0]).  Activation chunks: lane = route
  // lane / 8 of the wave's quarter of a tile, chunk (lane % 8) ^ (route / 2 % 8).
  auto bind = [&](const WideItem& it, int par) __attribute__((always_inline)) {
    const int lane = fresh_lane();
    const int di = 8 * wr + (lane >> 3), dc = (lane & 7) ^ ((di >> 1) & 7);
    auto row = [&](int r) {
      if constexpr (S1) return s_rt[par][0][r] & ROUTE_TOKEN_MASK;
      else return it.rb + (r < it.rows ? r : 0);
    };
#pragma unroll
    for (int j = 0; j < MAXC; ++j)
      aoff[j] = (uint32_t)row(min(it.tile0 + j, 2 * MAXC - 1) * RT + di) * KROW + dc * 16;
    soff = (uint32_t)row((it.tile0 + max(0, min(wr, it.ncw - 1))) * RT + (lane & 31)) * (S1 ? 4u : IB * 4u);
  };
  auto issue_a = [&](const WideItem& it) __attribute__((always_inline)) {  // K-block 0
#pragma unroll
    for (int j = 0; j < MAXC; ++j)
      if (j < it.ncw) issue_a1(it, 0, 0, j);
    if (it.ncw > 0) issue_s(it, 0, 0);
  };

  take();
  __syncthreads();
  int L = __builtin_amdgcn_readfirstlane(s_item);
  if (L < 0) return;
  WideItem cur = decode(L);
  issue_tables(cur, 0);
  issue_w(cur, 0, 0);
  wait_loads<4>();
  lds_barrier();
  bind(cur, 0);
  issue_a(cur);
  if constexpr (S1) {
    issue_w(cur, 1, 1);
    wait_loads<4>();
  } else {
    wait_loads<0>();
  }
  int par = 0;

  for (;;) {
    WideItem nxt = cur;
    int Ln = 0;
    auto item = [&](auto nct) __attribute__((always_inline)) {
      constexpr int NC = decltype(nct)::value;
      WideAcc<NC, S1 ? 2 : 1> lp;
      if constexpr (NC > 0) {
#pragma unroll
        for (int op = 0; op < 2; ++op)
#pragma unroll
          for (int cc = 0; cc < NC; ++cc)
#pragma unroll
            for (int r = 0; r < 16; ++r) lp.acc[op][cc][r] = 0.0f;
#pragma unroll
        for (int op = 0; op < 2; ++op)
#pragma unroll
          for (int r = 0; r < 16; ++r) lp.p[op][r] = 0.0f;
        lp.sg[0] = lp.sg[1] = lp.su[0] = lp.su[1] = 0.0f;
      }
      uint32_t alane, aw, b0, b1, b2, b3, sp;
      {
        const int lane = fresh_lane(), bi = lane & 31;
        // B operand reads: chunk 4kh + 2g + p of route i sits at slot chunk ^ (i / 2 % 8)
        const uint32_t bx = (uint32_t)((((lane >> 5) << 1) ^ ((bi >> 1) & 7)) << 4);
        const uint32_t ba = la + cur.tile0 * FRAG + bi * 128;
        alane = a_lane_offset(lane);
        aw = lw + (2 * wr) * FRAG + lane * 16;
        b0 = ba + bx, b1 = ba + (bx ^ 16), b2 = ba + (bx ^ 64), b3 = ba + (bx ^ 80);
        sp = ls + cur.tile0 * 256 + lane * 4;
        __asm__ volatile("" : "+v"(b0), "+v"(b1), "+v"(b2), "+v"(b3), "+v"(aw), "+v"(sp), "+v"(alane));
      }
      float wsa_l = 0.0f, wsb_l = 0.0f;  // weight-block scales, K-block k in lane k

      // One K-block.  LEFT: K-blocks left after it, at most 2.  OUT: loads
      // that may be outstanding at its opening barrier (-1: nothing to wait
      // for, its K-block landed before the previous item's stores).
      auto step = [&](int kb, auto slot_c, auto left_c, auto out_c) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_c)::value, LEFT = decltype(left_c)::value, OUT = decltype(out_c)::value;
        constexpr bool FIRST = OUT < 0;
        if constexpr (FIRST) lds_barrier();
        else landed_barrier<OUT>();
        // stage 2: the previous item's rows were in slot 1 up to here
        if constexpr (FIRST && !S1) issue_w(cur, 1, 1);
        if constexpr (NC > 0) {
          constexpr int WS = slot * W_SLOT, AS = slot * G::ACT_SLOT;
          v16f zero16;
#pragma unroll
          for (int r = 0; r < 16; ++r) zero16[r] = 0.0f;
          v8i b[3], a[2][2];
          a[0][0] = lds_op(aw + WS, aw + WS + 1024);
          b[0] = lds_op(b0 + AS, b1 + AS);
          a[0][1] = lds_op(aw + WS + 2048, aw + WS + 3072);
          b[1] = lds_op(b2 + AS, b3 + AS);
          a[1][0] = lds_op(aw + WS + FRAG, aw + WS + FRAG + 1024);
          a[1][1] = lds_op(aw + WS + FRAG + 2048, aw + WS + FRAG + 3072);
          if constexpr (FIRST) {
            const int lane = fresh_lane();
            wsa_l = s_ws[par][S1 ? 0 : wr >> 1][lane];
            if constexpr (S1) wsb_l = s_ws[par][1][lane];
          }
          const float wk0 = lane_value(wsa_l, kb), wk1 = S1 ? lane_value(wsb_l, kb) : 0.0f;
          __builtin_amdgcn_sched_barrier(0);
          // after MFMA i of route tile cc: the step's loads, one at a time
          auto hook = [&](int n) __attribute__((always_inline)) {
            constexpr int NA = NC + 1;
            constexpr int WB = NC == 1 ? 3 : NA + 1 > 3 ? NA + 1 : 3, WSTEP = NC >= 3 ? 2 : NC == 2 ? 1 : 0;
            if constexpr (LEFT >= 1) {
#pragma unroll
              for (int i = 0; i < NA; ++i)
                if (n == (NC == 1 ? 0 : i)) {
                  if (i < NC) issue_a1(cur, kb + 1, slot ^ 1, i);
                  else issue_s(cur, kb + 1, slot ^ 1);
                }
            }
            if constexpr (LEFT >= 2) {
              if (n == WB) plain_barrier();  // every wave holds its weight fragments of kb
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int at = WB + 1 + i * WSTEP;
                if (n == (at < 4 * NC ? at : 4 * NC - 1)) issue_w1(cur, alane, kb + 2, slot, i);
              }
            }
            __builtin_amdgcn_sched_barrier(0);
          };
#pragma unroll
          for (int cc = 0; cc < NC; ++cc) {
            const int u = (slot * NC + cc) & 1;  // scale set: 2 * NC units per two steps is even
            const int pc = cc >= 1 ? cc - 1 : NC - 1;
            lp.p[0] = mfma_32x32x64_fp8(a[0][0], b[(2 * cc) % 3], zero16);
            if (cc + 1 < NC) b[(2 * cc + 2) % 3] = lds_op(b0 + AS + (cc + 1) * FRAG, b1 + AS + (cc + 1) * FRAG);
            const float s = lds_f32(sp + slot * (G::SCL_SLOT * 4) + cc * 256);
            hook(4 * cc);
            lp.finish(1, pc, u ^ 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            lp.p[0] = mfma_32x32x64_fp8(a[0][1], b[(2 * cc + 1) % 3], lp.p[0]);
            hook(4 * cc + 1);
            lp.finish(1, pc, u ^ 1, 1);
            lp.sg[u] = s * wk0;
            if constexpr (S1) lp.su[u] = s * wk1;
            __builtin_amdgcn_sched_barrier(0);
            lp.p[1] = mfma_32x32x64_fp8(a[1][0], b[(2 * cc) % 3], zero16);
            if (cc + 1 < NC) b[(2 * cc + 3) % 3] = lds_op(b2 + AS + (cc + 1) * FRAG, b3 + AS + (cc + 1) * FRAG);
            hook(4 * cc + 2);
            lp.finish(0, cc, u, 0);
            __builtin_amdgcn_sched_barrier(0);
            lp.p[1] = mfma_32x32x64_fp8(a[1][1], b[(2 * cc + 1) % 3], lp.p[1]);
            hook(4 * cc + 3);
            lp.finish(0, cc, u, 1);
            __builtin_amdgcn_sched_barrier(0);
          }
        } else {
          if constexpr (LEFT >= 2) {
            plain_barrier();
#pragma unroll
            for (int i = 0; i < 4; ++i) issue_w1(cur, alane, kb + 2, slot, i);
          }
        }
      };
      using std::integral_constant;
      step(0, integral_constant<int, 0>{}, integral_constant<int, 2>{}, integral_constant<int, -1>{});
      step(1, integral_constant<int, 1>{}, integral_constant<int, 2>{}, integral_constant<int, 4>{});
#pragma unroll 1
      for (int kb0 = 2; kb0 < KB - 2; kb0 += 2) {
        step(kb0, integral_constant<int, 0>{}, integral_constant<int, 2>{}, integral_constant<int, 4>{});
        step(kb0 + 1, integral_constant<int, 1>{}, integral_constant<int, 2>{}, integral_constant<int, 4>{});
      }
      claim();
      step(KB - 2, integral_constant<int, 0>{}, integral_constant<int, 1>{}, integral_constant<int, 4>{});
      take();
      step(KB - 1, integral_constant<int, 1>{}, integral_constant<int, 0>{}, integral_constant<int, 0>{});
      // Every wave has passed the last step's opening barrier: slot 0 is free
      // for the next item, and s_item holds it.
      Ln = __builtin_amdgcn_readfirstlane(s_item);
      const bool more = Ln >= 0;
      if (more) {
        nxt = decode(Ln);
        issue_tables(nxt, par ^ 1);
        issue_w(nxt, 0, 0);
        if constexpr (!S1) {
          bind(nxt, par ^ 1);
          issue_a(nxt);
        }
      }
      if constexpr (NC > 0) {
        constexpr int ul = (NC + NC - 1) & 1;
        lp.finish(1, NC - 1, ul, 0);
        lp.finish(1, NC - 1, ul, 1);
      }
      const int rows = cur.rows, rb = cur.rb, nb = cur.nb, tile0 = cur.tile0;

      if constexpr (S1) {
        // SwiGLU, per-route amax, FP8 requant (see prefill.hip)
        if constexpr (NC > 0) {
          const int lane = fresh_lane();
#pragma unroll
          for (int cc = 0; cc < NC; ++cc) {
            float m = 0.0f;
#pragma unroll
            for (int op = 0; op < 2; ++op)
#pragma unroll
              for (int r = 0; r < 8; ++r) {
                const float g = lp.acc[op][cc][r], u = lp.acc[op][cc][r + 8];
                const float c = (u * __builtin_amdgcn_rcpf(1.0f + __expf(-u))) * g;
                lp.acc[op][cc][r] = c;
                m = fmaxf(m, fabsf(c));
              }
            m = fmaxf(m, __shfl_xor(m, 32));
            if (lane < 32) s_red[wr][(tile0 + cc) * RT + lane] = m;
          }
        }
        wait_loads<4>();  // the next item's tables
        lds_barrier();    // also: every wave is past its K loop
        if (more) {
          bind(nxt, par ^ 1);
          issue_a(nxt);
          issue_w(nxt, 1, 1);
        }
        uint8_t* s_e = pool + L_E;
        if constexpr (NC > 0) {
          const int lane = fresh_lane(), bi = lane & 31;
#pragma unroll
          for (int cc = 0; cc < NC; ++cc) {
            const int row = (tile0 + cc) * RT + bi;
            if (row < rows) {
              const float am = fmaxf(fmaxf(s_red[0][row], s_red[1][row]), fmaxf(s_red[2][row], s_red[3][row]));
              const float sc = fmaxf(am / E4M3_MAX, 1.0e-8f);
              const float isc = __builtin_amdgcn_rcpf(sc);
#pragma unroll
              for (int op = 0; op < 2; ++op) {
                uint8_t* crow = s_e + row * CQ_STRIDE + 16 * (2 * wr + op) + 4 * (lane >> 5);
#pragma unroll
                for (int hq = 0; hq < 2; ++hq) {
                  float v[4];
#pragma unroll
                  for (int i = 0; i < 4; ++i)
                    v[i] = fminf(fmaxf(lp.acc[op][cc][4 * hq + i] * isc, -E4M3_MAX), E4M3_MAX);
                  *reinterpret_cast<uint32_t*>(crow + 8 * hq) = cvt4_e4m3(v[0], v[1], v[2], v[3]);
                }
              }
              if (wr == 0 && lane < 32) s_sc[row] = sc;
            }
          }
        }
        wait_loads<4>();  // the next item's first K-block has landed before any store is issued
        lds_barrier();
        const int tid = w * 64 + fresh_lane();
        for (int row = tid >> 3; row < rows; row += WNT / 8) {
          const uint4 v = *reinterpret_cast<const uint4*>(s_e + row * CQ_STRIDE + 16 * (tid & 7));
          *reinterpret_cast<uint4*>(Cq + (size_t)(rb + row) * I + nb * BLK + 16 * (tid & 7)) = v;
        }
        if (tid < rows) Cs[(size_t)(rb + tid) * IB + nb] = s_sc[tid];
      } else {
        // One route tile of each route group at a time through LDS (group 0:
        // weight slot 1, group 1: activation slot 1), out as whole 1 KB (Y) or
        // 512-byte (bf16 output) rows.  16-byte column chunk c of route i sits
        // at chunk c ^ (i % 16).
        const int lane = fresh_lane(), bi = lane & 31;
        const int np = (rows + 2 * RT - 1) / (2 * RT);  // route tiles of group 0
        uint8_t* s_y = pool + (wc ? L_E : W_SLOT);
        const size_t hcol = (size_t)nb * (2 * BLK) + 4 * lane;
        lds_barrier();  // every wave is past its K loop
#pragma unroll
        for (int cc = 0; cc < MAXC; ++cc) {
          if (cc >= np) break;
          if constexpr (NC > 0) {
            if (cc < NC) {
              const int c2 = cc < NC ? cc : 0;
              const float rw = __int_as_float(s_rt[par][1][(tile0 + cc) * RT + bi]);
#pragma unroll
              for (int op = 0; op < 2; ++op)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  const int c = 16 * wr + 8 * op + 2 * j + (lane >> 5);
                  *reinterpret_cast<float4*>(s_y + bi * 1024 + ((c ^ (bi & 15)) << 4)) =
                      make_float4(lp.acc[op][c2][4 * j] * rw, lp.acc[op][c2][4 * j + 1] * rw,
                                  lp.acc[op][c2][4 * j + 2] * rw, lp.acc[op][c2][4 * j + 3] * rw);
                }
            }
          }
          lds_barrier();
          float4 v[RT / 4];
          int tk[RT / 4];
          if (NC > 0 && cc < NC) {
#pragma unroll
            for (int k = 0; k < RT / 4; ++k) {
              const int rt = wr + 4 * k;
              v[k] = *reinterpret_cast<const float4*>(s_y + rt * 1024 + ((lane ^ (rt & 15)) << 4));
              tk[k] = s_rt[par][0][(tile0 + cc) * RT + rt];
            }
          }
          if (cc + 1 < np) lds_barrier();  // the next tile's rows may be written
          if (cc == 0) wait_loads<0>();    // the next item's first K-block lands before any store is issued
          if (NC > 0 && cc < NC) {
#pragma unroll
            for (int k = 0; k < RT / 4; ++k) {
              const int row = (tile0 + cc) * RT + wr + 4 * k;
              if (row < rows) {
                const int t = __builtin_amdgcn_readfirstlane(tk[k]);
                if (t < 0)  // SINGLE_ROUTE_BIT
                  store_out_bf16x4(out + (size_t)(t & ROUTE_TOKEN_MASK) * H + hcol, v[k]);
                else
                  *reinterpret_cast<float4*>(Y + (size_t)(rb + row) * H + hcol) = v[k];
              }
            }
          }
        }
      }
    };
    // wave-uniform instantiation by the wave's route-tile count
    switch (cur.ncw) {
      case 0: item(std::integral_constant<int, 0>{}); break;
      case 1: item(std::integral_constant<int, 1>{}); break;
      case 2: item(std::integral_constant<int, 2>{}); break;
      case 3: item(std::integral_constant<int, 3>{}); break;
      default: item(std::integral_constant<int, MAXC>{}); break;
    }
    if (Ln < 0) break;
    cur = nxt;
    par ^= 1;
  }
}

}  // namespace

hipError_t launch_stage1_wide(const uint8_t* hidden, const float* hs, const uint8_t* w13p, const float* w13s,
                              const int32_t* counts, const int32_t* offsets, const int32_t* route_token, uint8_t* Cq,
                              float* Cs, int T, int e_local, int max_routes, int32_t* queue, hipStream_t stream) {
  constexpr int MAXC = 4;
  auto k = wide_kernel<MAXC, true>;
  const long long bound = ((long long)e_local + max_routes / WideGeom<MAXC>::BM + 1) * IB;
  k<<<persistent_grid(bound, device_cus()), WNT, 0, stream>>>(hidden, hs, w13p, w13s, counts, offsets, nullptr,
                                                               route_token, Cq, Cs, nullptr, nullptr, T, e_local, queue);
  return hipGetLastError();
}

hipError_t launch_stage2_wide(const uint8_t* Cq, const float* Cs, const uint8_t* w2p, const float* w2s,
                              const int32_t* counts, const int32_t* offsets, const float* rw,
                              const int32_t* route_token, float* Y, uint16_t* out, int T, int e_local, int max_routes,
                              int32_t* queue, hipStream_t stream) {
  constexpr int MAXC = 4;
  auto k = wide_kernel<MAXC, false>;
  const long long bound = ((long long)e_local + max_routes / WideGeom<MAXC>::BM + 1) * (HB / 2);
  k<<<persistent_grid(bound, device_cus()), WNT, 0, stream>>>(Cq, Cs, w2p, w2s, counts, offsets, rw, route_token,
                                                               nullptr, nullptr, Y, out, T, e_local, queue);
  return hipGetLastError();
}

}  // namespace moe
