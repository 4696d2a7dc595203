// Fused half-layout-RoPE flash-attention backward for gfx950: the dK/dV kernel and the dQ kernel.
//
// Device counterparts of the reference's _attn_bwd_dkdv / _attn_bwd_dq
// (fused-rope/fused_rope_attn.py:342-404, :409-470, driver :474-649).  The reference runs both halves in one
// program and re-rotates Q (resp. K) in registers on every inner iteration; here each half is its own kernel
// and the streamed operand is rotated once per workgroup per tile while it is staged into LDS.  No atomics:
// dK/dV are owned by the key block's workgroup, dQ by the query block's.
//
// Scaling contract (same as the reference's, :385, :457, :574-575, :643-644, with the host-side K pre-scale
// :746-748 folded in): P = exp2(s * sm_scale * log2e - M) with M the forward's base-2 statistic;
// dS = P o (dP - delta); dK_r = sm_scale * dS^T Q_r; dQ_r = sm_scale * dS K_r; both un-rotated in fp32
// before the single rounding to bf16.
//
// Operands that must be read "transposed" (contraction along the sequence axis of a row-major tile) use the
// gfx950 transposing LDS read, so every tile is staged row-major exactly once.
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "kernels.hpp"

namespace COROPE_NS {

// Layout of LDS tiles that are read both row-wise (16 bytes per lane, lane = row) and through the transposing read
// (8 bytes per lane, 4 rows x 32 bytes per 16 lanes).  With plain row padding, 16 bytes keep the row-wise reads free of
// bank conflicts and leave the transposing ones four-way conflicted, 64 bytes do the opposite; measured on the fused
// dK+dV kernel at B2 H32 N4096 D128, paddings of 16 / 32 / 48 / 64 / 80 bytes gave 0.551 / 0.524 / 0.512 / 0.561 /
// 0.523 ms.  The staggered layout (free of conflicts both ways, 68 bytes a row) gains another 1.4 % there, side by side
// on one device; in the dQ kernel it loses 2.8 % to the 48-byte padding (more registers spilled for its addresses).
constexpr int kBothWaysPad = 24;
constexpr int kDkdvBothWaysPad = kStaggerPad;

// ===================================================================================== dK / dV
// Workgroup = NWAVES waves x 32 keys.  K_r and V rows of the wave stay in registers as B operands.
// Per query tile (BLOCK_M rows, staged: rotated Q and dO, plus M and delta):
//   S  = Q_r K_r^T            (A = Q_r rows from LDS,      B = K_r regs)   lane = key, registers = queries
//   dP = dO V^T               (A = dO rows from LDS,       B = V regs)
//   P  = exp2(S*c - M), dS = P o (dP - delta)                               (bf16, already B-operand shaped)
//   dV^T   += dO^T  P         (A = dO tile read transposed, B = P)
//   dK_r^T += Q_r^T dS        (A = Q_r tile read transposed, B = dS)
// DO_PAD: row padding of the dO tile.  The dV-only kernel reads dO through the transposing load alone and takes the
// padding that is conflict-free for it (32); the dK kernel reads dO row-wise (8).
// V_LDS: the waves' V rows live in LDS instead of registers -- the fused dK+dV kernel up to D = 128, whose two sets of accumulators
// leave no room for them (at D = 256, with one wave per SIMD, they do).
//
// Persistent, like the other attention kernels: one workgroup per compute unit walks a balanced list of (key/value slab,
// key block) items and the stream of query tiles runs on from item to item.  Behind the two tile stages every wave has an
// LDS slot of its own (32 padded rows): its V rows during an item (V_LDS), and at the change of items the tile through
// which its dV and dK rows leave and its next K_r rows come in -- nothing there needs a workgroup barrier.
template <int D, int NWAVES, int BLOCK_M, int DO_PAD, int Q_PAD>
struct DkdvCfg {
  static constexpr int kThreads = NWAVES * kWave;
  static constexpr int kBlockN = NWAVES * 32;
  static constexpr int kTileBytes = RowTile<D, Q_PAD>::bytes(BLOCK_M);
  static constexpr int kDoTileBytes = RowTile<D, DO_PAD>::bytes(BLOCK_M);
  static constexpr int kStatBytes = BLOCK_M * 4;
  static constexpr int kStageBytes = kTileBytes + kDoTileBytes + 2 * kStatBytes;
  static constexpr int kRingBytes = 2 * kStageBytes;
  static constexpr int kWaveBytes = RowTile<D>::bytes(32);
  static_assert(kWaveBytes >= WaveTile<D>::kBytes, "a wave's slot holds its unpadded tile too");
  static constexpr int kLdsBytes = kRingBytes + NWAVES * kWaveBytes;
  static_assert(kLdsBytes <= 160 * 1024, "LDS of a compute unit");
};

// v and d_o may be strided views (BwdParams) on rotated copies up to D = 128; the kernels' STRIDED says whether they read them through
// run-time strides.  At D = 256 the registers for these cost the dK+dV kernel 10 % (222 -> 245 us at B2 H16 N2048).  On unrotated
// operands, which have none, they cost dK and dV up to 3 % (dK B6 H4 N274 D128 not causal 24.7 -> 25.5 us, dV B4 H32 N900 D64 33.7 -> 34.3),
// and dQ nothing (B4 H32 N448 D128 44.1 us with, 44.5 without).
template <int D, bool STRIDED>
__device__ __forceinline__ uint32_t do_row_bytes(const BwdParams& p) { return STRIDED ? (uint32_t)p.do_sn * 2 : D * 2; }
template <int D, bool STRIDED>
__device__ __forceinline__ uint32_t v_row_bytes(const BwdParams& p) { return STRIDED ? (uint32_t)p.v_sn * 2 : D * 2; }
template <int D, bool STRIDED>
__device__ __forceinline__ const uint16_t* v_slab_of(const BwdParams& p, int kvs) {
  return STRIDED ? p.v_slab(kvs) : p.v + (int64_t)kvs * p.N * D;
}

// What a workgroup of the dK+dV kernel works on.  CUT = false: whole items dealt in rounds (ItemList).  CUT = true: the query
// tiles of all items, slab after slab, form one list that the workgroups cut into equal pieces, so that few or unequal items
// (short sequences, few heads, grouped-query attention, where one key block sweeps the query tiles of several heads) still
// keep every compute unit busy equally long.  A piece that holds all of an item writes its result; others leave fp32
// accumulators in a slot of their own -- at most one at each end of a piece -- and rope_attn_bwd_dkdv_sum_kernel adds an
// item's slots in list order.  Both number the items heaviest first: item i is key block i / slabs of slab i % slabs.
template <bool CUT>
struct DkdvWork;

template <>
struct DkdvWork<false> {
  ItemList items;
  int total;
  __device__ __forceinline__ DkdvWork(int num_blocks, int slabs, int, int, int) : total(num_blocks * slabs) {}
  __device__ __forceinline__ int at(int round) const { return items.at(round); }   // >= total: no such item
  __device__ __forceinline__ int begin(int) const { return 0; }
  __device__ __forceinline__ int end(int, int iters) const { return iters; }
  __device__ __forceinline__ int share() const { return 0; }
};

struct DkdvTiles {
  int nb, slabs, group, m_tiles, step, per_slab, total_tiles;
  // step: query tiles by which a key block sees fewer than the one before it (0 when every key sees every query)
  __host__ __device__ DkdvTiles(int nb_, int slabs_, int group_, int m_tiles_, int step_)
      : nb(nb_), slabs(slabs_), group(group_), m_tiles(m_tiles_), step(step_) {
    per_slab = first(nb);
    total_tiles = per_slab * slabs;
  }
  __host__ __device__ int first(int kb) const { return group * (kb * m_tiles - step * (kb * (kb - 1) / 2)); }   // tiles of a slab before block kb
  __device__ int start(int item) const { return (item % slabs) * per_slab + first(item / slabs); }
  __device__ int begin_of_share(int w, int shares) const { return (int)((int64_t)w * total_tiles / shares); }
  __device__ int share_of(int tile, int shares) const { return (int)((((int64_t)tile + 1) * shares - 1) / total_tiles); }
};

template <>
struct DkdvWork<true> {
  DkdvTiles t;
  int total, t0, t1, li0, piece;
  __device__ __forceinline__ DkdvWork(int num_blocks, int slabs, int group, int m_tiles, int step)
      : t(num_blocks, slabs, group, m_tiles, step), total(num_blocks * slabs) {
    // workgroup ids go round-robin to the 8 XCDs: neighbouring pieces, which share slabs, stay on one
    const int n = gridDim.x, id = blockIdx.x;
    piece = n % 8 == 0 ? (id % 8) * (n / 8) + id / 8 : id;
    t0 = t.begin_of_share(piece, n);
    t1 = t.begin_of_share(piece + 1, n);
    const int slab = t0 / t.per_slab, rem = t0 % t.per_slab;
    int kb = 0;
    while (kb + 1 < t.nb && t.first(kb + 1) <= rem) ++kb;
    li0 = slab * t.nb + kb;
  }
  __device__ __forceinline__ int at(int round) const {
    const int li = li0 + round, slab = li / t.nb, kb = li % t.nb;
    return li < total && slab * t.per_slab + t.first(kb) < t1 ? kb * t.slabs + slab : total;
  }
  __device__ __forceinline__ int begin(int item) const { return max(0, t0 - t.start(item)); }
  __device__ __forceinline__ int end(int item, int iters) const { return min(iters, t1 - t.start(item)); }
  __device__ __forceinline__ int share() const { return piece; }
};

// A slot of partial sums: NWAVES x 32 keys x D of dV, then of dK_r, as the accumulators lie ([32-key block][register quad][lane]).
template <int D, int NWAVES>
constexpr int64_t kDkdvSlotFloats = 2ll * NWAVES * 32 * D;

// PREROT: Q and K come from copies that rope_rotate_kernel rotated beforehand (no table reads in the loop).
template <int D, int NWAVES, int BLOCK_M, bool CAUSAL, bool DO_DV, bool DO_DK, bool PREROT, bool CUT = false>
__global__ __launch_bounds__(NWAVES* kWave) __attribute__((amdgpu_waves_per_eu(kWavesPerSimd<D>, kWavesPerSimd<D>))) void rope_attn_bwd_dkdv_kernel(BwdParams p) {
  constexpr int DO_PAD = DO_DK ? (DO_DV ? kDkdvBothWaysPad : 8) : 32;
  constexpr int Q_PAD = DO_DK ? kDkdvBothWaysPad : 8;
  constexpr bool V_LDS = DO_DV && DO_DK && D <= 128, STRIDED = PREROT && D <= 128, PIPED = DO_DV && DO_DK && D > 128;
  // The next rows are requested behind a cut block's partial sums: in both branches of the change of items, 27 of the loads went to scratch memory one
  // by one, each waiting for the memory's full latency (B1 H4 N4096 154 -> 104 us, B1 H1 N30000 fp16 1585 -> 990).
  constexpr bool LATE = CUT && PIPED;
  using Cfg = DkdvCfg<D, NWAVES, BLOCK_M, DO_PAD, Q_PAD>;
  constexpr int NT = Cfg::kThreads;
  constexpr int KC = D / 16, NDB = D / 32, NQB = BLOCK_M / 32;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int lq = lane % 32, lh = lane / 32;
  // 32-key block of the item this wave owns; waves w and w + 4 share a SIMD, blocks (0,7), (1,6), (2,5), (3,4) give
  // every SIMD the same number of diagonal tiles
  const int rb = NWAVES == 8 ? (wave < 4 ? wave : 11 - wave) : wave;
  [[maybe_unused]] constexpr int TT = 0;   // stamping thread: first lane of the wave with the first keys (it sees every tile)
  const int N = p.N;
  uint8_t* const wave_slot = smem + Cfg::kRingBytes + wave * Cfg::kWaveBytes;
  uint16_t* const vrows = reinterpret_cast<uint16_t*>(wave_slot);   // V_LDS: the wave's V rows, row-major, padded

  // An item: a key block of one key/value slab; its workgroup sweeps the query tiles of every query head of the group
  // (one head without grouped-query attention), accumulating dK and dV over all of them.  Heaviest first: causal key
  // blocks see fewer query tiles the later they lie.
  const int BHkv = p.BH / p.H * p.Hkv, GQ = p.H / p.Hkv;
  const int m_tiles = (N + BLOCK_M - 1) / BLOCK_M;
  const DkdvWork<CUT> items(p.num_blocks, BHkv, GQ, m_tiles, CAUSAL ? Cfg::kBlockN / BLOCK_M : 0);
  const int total = items.total;           // item i: key block i / BHkv of slab i % BHkv
  const uint16_t* q_all = PREROT ? p.q_rot : p.q;

  // ---- the stream of query tiles: a cursor one tile ahead of the tile being consumed -----------------------------------
  RopeStage<D, BLOCK_M, NT, PREROT, true, Q_PAD> qst;   // Q_r tiles carry qk_scale: S leaves the matrix cores in base-2 units
  qst.out_scale = p.qk_scale;
  CopyStage<D, BLOCK_M, NT, DO_PAD> dst;
  float st_lse = 0.f, st_delta = 0.f;
  [[maybe_unused]] int st_row = 0;
  int l_round = 0, l_it, l_iters, l_slab0, l_mt0, l_tph;
  const uint16_t* l_do;
  auto load_item = [&](int r) {    // false: no such item
    const int i = items.at(r);
    if (i >= total) return false;
    const int bkv = i % BHkv, n0 = (i / BHkv) * Cfg::kBlockN;
    l_slab0 = (bkv / p.Hkv) * p.H + (bkv % p.Hkv) * GQ;   // first query head of the group
    if constexpr (STRIDED) l_do = p.do_slab(l_slab0);
    l_mt0 = CAUSAL ? n0 / BLOCK_M : 0;
    l_tph = max(m_tiles - l_mt0, 0);
    l_it = items.begin(i);
    l_iters = items.end(i, GQ * l_tph);
    return true;
  };
  // iteration it of an item -> query head slab0 + it / tph, query tile mt0 + it % tph
  auto load_next_tile = [&](bool advance) __attribute__((always_inline)) {
    if (advance) {
      if (l_it + 1 < l_iters) {
        ++l_it;
      } else if (load_item(l_round + 1)) {
        ++l_round;
      }   // else: past the last tile of the last item; the same tile is requested again and never used
    }
    const int qs = l_slab0 + l_it / l_tph, m0 = (l_mt0 + l_it % l_tph) * BLOCK_M;
    qst.load(q_all + (int64_t)qs * N * D, p.cos, p.sin, p.fstride, m0, N);
    dst.load(STRIDED ? l_do + (qs - l_slab0) * p.do_sh : p.d_o + (int64_t)qs * N * D, m0, N, do_row_bytes<D, STRIDED>(p));
    if constexpr (PIPED) {
      // As they lie in memory: a sign changed here waits for the loads, and for the tile's before them, on the spot.  With one wave per SIMD
      // that was 0.6 us of a tile's 1.85; with two the other wave fills it, and this form is no faster (D = 128) or 2 % slower (64).
      st_row = m0 + threadIdx.x;
      if (threadIdx.x < BLOCK_M) {
        const int64_t at = (int64_t)qs * N + min(st_row, N - 1);
        st_lse = p.lse[at];
        st_delta = p.delta[at];
      }
    } else if (threadIdx.x < BLOCK_M) {
      int qi = m0 + threadIdx.x;
      // -M and -delta: what the S and dP products start from.  Rows past the end: M = +inf makes P = 0, so they
      // contribute nothing
      st_lse = qi < N ? -p.lse[(int64_t)qs * N + qi] : -INFINITY;
      if constexpr (DO_DK) st_delta = qi < N ? -p.delta[(int64_t)qs * N + qi] : 0.f;
    }
  };
  auto q_tile = [&](int buf) { return reinterpret_cast<uint16_t*>(smem + buf * Cfg::kStageBytes); };
  auto do_tile = [&](int buf) { return reinterpret_cast<uint16_t*>(smem + buf * Cfg::kStageBytes + Cfg::kTileBytes); };
  auto lse_tile = [&](int buf) {
    return reinterpret_cast<float*>(smem + buf * Cfg::kStageBytes + Cfg::kTileBytes + Cfg::kDoTileBytes);
  };
  auto delta_tile = [&](int buf) {
    return reinterpret_cast<float*>(smem + buf * Cfg::kStageBytes + Cfg::kTileBytes + Cfg::kDoTileBytes + Cfg::kStatBytes);
  };
  auto store_tile = [&](int buf) __attribute__((always_inline)) {
    qst.store_rows(q_tile(buf));
    dst.store_rows(do_tile(buf));
    if (threadIdx.x < BLOCK_M) {
      lse_tile(buf)[threadIdx.x] = !PIPED ? st_lse : st_row < N ? -st_lse : -INFINITY;
      if constexpr (DO_DK) delta_tile(buf)[threadIdx.x] = !PIPED ? st_delta : st_row < N ? -st_delta : 0.f;
    }
  };
  int cur = 0;   // ring stage of the tile being consumed

  // ---- the wave's K_r (and V) rows of an item ----------------------------------------------------------------------
  // (the lane index goes in as a value the optimiser cannot see through: the per-lane address parts of these steps are
  // then recomputed per item instead of being kept in registers, or in scratch memory, across the whole loop)
  auto opaque_lane = [&]() __attribute__((always_inline)) {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  WaveRows<D, !PREROT> krows;
  WaveRows<D, false> vrows_regs;
  u32x4 kb[KC], vb[(DO_DK && !V_LDS) ? KC : 1];
  auto request_rows = [&](int i) __attribute__((always_inline)) {
    const int64_t base = (int64_t)(i % BHkv) * N * D;
    const int row0 = (i / BHkv) * Cfg::kBlockN + rb * 32, l = opaque_lane();
    krows.load((PREROT ? p.k_rot : p.k) + base, p.cos, p.sin, p.fstride, row0, N, l);
    if constexpr (DO_DK) vrows_regs.load(v_slab_of<D, STRIDED>(p, i % BHkv), nullptr, nullptr, 0, row0, N, l, v_row_bytes<D, STRIDED>(p));
  };
  auto take_rows = [&]() __attribute__((always_inline)) {
    const int l = opaque_lane();
    park_rows<D>(krows, kb, wave_slot, 1.f, l);
    if constexpr (DO_DK && !V_LDS) park_plain_rows<D>(vrows_regs, vb, wave_slot, l);
    if constexpr (V_LDS) {
      using WR = WaveRows<D, false>;
      lds_order();
#pragma unroll
      for (int i = 0; i < WR::IT; ++i)
        *reinterpret_cast<u32x4*>(vrows + RowTile<D>::off(WR::RPI * i + l / WR::CPR, (l % WR::CPR) * 8)) = vrows_regs.x[i];
      lds_order();
    }
  };

  // ---- first item: nothing to hide its prologue behind ----------------------------------------------------------------
  int item = items.at(0);
  COROPE_ISTAMP(0);
  load_item(0);
  load_next_tile(false);
  request_rows(item);
  take_rows();
  store_tile(0);
  __syncthreads();

  for (int round = 0;; ++round) {
    const int bkv = item % BHkv, n0 = (item / BHkv) * Cfg::kBlockN;
    const int64_t base = (int64_t)bkv * N * D;                           // k, v, dk, dv
    const int mt0 = CAUSAL ? n0 / BLOCK_M : 0;
    const int tiles_per_head = max(m_tiles - mt0, 0), n_iter = GQ * tiles_per_head;
    const int it_begin = items.begin(item), it_end = items.end(item, n_iter);
    const int wk_lo = n0 + rb * 32, wk_hi = wk_lo + 31;
    const int key = wk_lo + lq;
    COROPE_ISTAMP(1);
    COROPE_ISTAMP_ID(n_iter);
#ifdef COROPE_TRACE
    const uint64_t clk0 = __builtin_readcyclecounter();
#endif

    f32x16 dvacc[DO_DV ? NDB : 1], dkacc[DO_DK ? NDB : 1];
#pragma unroll
    for (int i = 0; i < NDB; ++i) {
      if constexpr (DO_DV) dvacc[i] = f32x16{0};
      if constexpr (DO_DK) dkacc[i] = f32x16{0};
    }
    // The wave's K_r (and V) rows must have landed on EVERY path into the loop: left to the first product that reads
    // them, the wait for them is placed inside the loop, where each time round it also waits for the next tile's loads
    // issued a few instructions earlier, and the prefetch hides less.
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      asm volatile("" ::"v"(kb[kc]));
      if constexpr (DO_DK && !V_LDS) asm volatile("" ::"v"(vb[kc]));
    }

    for (int it = it_begin; it < it_end; ++it) {
      const int m0 = (mt0 + it % tiles_per_head) * BLOCK_M;
#ifdef COROPE_TRACE
      if (it == 1) COROPE_ISTAMP(3);
      if (it == Cfg::kBlockN / BLOCK_M) COROPE_ISTAMP(4);   // first tile past the diagonal block
#endif
      load_next_tile(true);

      const uint16_t* qs = q_tile(cur);
      const uint16_t* dos = do_tile(cur);
      const float* lses = lse_tile(cur);
      const float* deltas = delta_tile(cur);
      if constexpr (PIPED) {
        // One wave per SIMD: nothing overlaps what the wave itself does not, so the tile is one stream of 4 x 16 products with its operands
        // RING ahead, the exponentials between the dP products, dS between the dV products, and the next tile's staging between the dK products.
        // What bounds it: LDS reads (64 KB a tile) and products in about equal parts, and what of the latencies is still seen.  As the compiler scheduled it, V
        // read from the LDS for every product: B2 H16 N2048 245 -> 187 us, B7 Hq10 Hkv5 N2371 700 -> 487 (RING 6 or later staging: no difference).
        static_assert(NQB == 1 && kWavesPerSimd<D> == 1, "one 32-row block per tile");
        if (CAUSAL && m0 + 31 < wk_lo) {   // queries that lie above every key of the wave: it only stages its share
          store_tile(cur ^ 1);
        } else {
          constexpr int RING = 4, TOTAL = 4 * KC;
          const uint32_t tr = (4 * lh + lane % 16 / 4) * RowTile<D, Q_PAD>::kStride + RowTile<D, Q_PAD>::stagger(4 * lh) + 16 * (lane / 16 % 2) + 4 * (lane % 4);
          const uint16_t *q_l = qs + RowTile<D, Q_PAD>::off(lq, 8 * lh), *do_l = dos + RowTile<D, DO_PAD>::off(lq, 8 * lh), *q_t = qs + tr, *do_t = dos + tr;
          auto operand = [&](int n) __attribute__((always_inline)) {
            const int i = n % KC;
            return n < KC       ? *reinterpret_cast<const u32x4*>(q_l + 16 * i)
                   : n < 2 * KC ? *reinterpret_cast<const u32x4*>(do_l + 16 * i)
                   : n < 3 * KC ? load_a_trans_lane<RowTile<D, DO_PAD>>(do_t, 16 * (i / NDB), i % NDB * 32)
                                : load_a_trans_lane<RowTile<D, Q_PAD>>(q_t, 16 * (i / NDB), i % NDB * 32);
          };
          u32x4 ring[RING];
          f32x16 sacc, dpacc;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 m4 = *reinterpret_cast<const f32x4*>(lses + 8 * g + 4 * lh);
#pragma unroll
            for (int e = 0; e < 4; ++e) sacc[4 * g + e] = m4[e];
          }
#pragma unroll
          for (int n = 0; n < RING; ++n) ring[n] = operand(n);
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 d4 = *reinterpret_cast<const f32x4*>(deltas + 8 * g + 4 * lh);
#pragma unroll
            for (int e = 0; e < 4; ++e) dpacc[4 * g + e] = d4[e];
          }
          u32x4 pb[2], dsb[2];
          __builtin_amdgcn_sched_barrier(0);
          static_for<TOTAL>([&](auto n_c) __attribute__((always_inline)) {
            constexpr int n = decltype(n_c)::value, slot = n / KC, i = n % KC;
            const u32x4 a = ring[n % RING];
            if constexpr (slot == 0) mfma32_acc_v(sacc, a, kb[i]);
            if constexpr (slot == 1) mfma32_acc_v(dpacc, a, vb[i]);
            if constexpr (slot == 2) dvacc[i % NDB] = mfma32(a, pb[i / NDB], dvacc[i % NDB]);
            if constexpr (slot == 3) dkacc[i % NDB] = mfma32(a, dsb[i / NDB], dkacc[i % NDB]);
            if constexpr (n + RING < TOTAL) ring[n % RING] = operand(n + RING);
            if constexpr (n == 3 * KC + 1) store_tile(cur ^ 1);
            // what the asm statements of the slot before left: nothing reads it behind product 0, which waits a little instead
            if constexpr ((slot == 1 || slot == 2) && i == 0) asm volatile("s_nop 7");
            if constexpr (slot == 1 && i == 1) {
              if (CAUSAL && m0 < wk_hi) {
                int rel = key - m0 - 4 * lh;
                asm volatile("" : "+v"(rel));
#pragma unroll
                for (int x = 0; x < 16; ++x)
                  if (8 * (x / 4) + x % 4 < rel) sacc[x] = -INFINITY;
              }
            }
            // eight pairs over the products 1 .. KC - 1 of a slot
            constexpr int lo = i == 0 ? 0 : (i - 1) * 8 / (KC - 1), hi = i == 0 ? 0 : i * 8 / (KC - 1);
            if constexpr (slot == 1) {
#pragma unroll
              for (int j = lo; j < hi; ++j) {
                sacc[2 * j] = fast_exp2(sacc[2 * j]);
                sacc[2 * j + 1] = fast_exp2(sacc[2 * j + 1]);
                pb[j / 4][j % 4] = pack_elts(sacc[2 * j], sacc[2 * j + 1]);
              }
            }
            if constexpr (slot == 2) {
#pragma unroll
              for (int j = lo; j < hi; ++j) dsb[j / 4][j % 4] = pack_elts(sacc[2 * j] * dpacc[2 * j], sacc[2 * j + 1] * dpacc[2 * j + 1]);
            }
            __builtin_amdgcn_sched_barrier(0);
          });
        }
      }
#pragma unroll
      for (int qb = 0; qb < (PIPED ? 0 : NQB); ++qb) {
        const int mq0 = m0 + qb * 32;
        // queries of this 32-row block that lie above every key of the wave see none of them
        if (CAUSAL && mq0 + 31 < wk_lo) continue;
        // The products start from -M and -delta of their rows (register i holds query 8*(i/4) + 4*lh + i%4 of the block):
        // S - M and dP - delta leave the matrix cores, no vector instruction applies them.
        f32x16 sacc, dpacc = f32x16{0};
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 m4 = *reinterpret_cast<const f32x4*>(lses + qb * 32 + 8 * g + 4 * lh);
#pragma unroll
          for (int e = 0; e < 4; ++e) sacc[4 * g + e] = m4[e];
          if constexpr (DO_DK) {
            const f32x4 d4 = *reinterpret_cast<const f32x4*>(deltas + qb * 32 + 8 * g + 4 * lh);
#pragma unroll
            for (int e = 0; e < 4; ++e) dpacc[4 * g + e] = d4[e];
          }
        }
        const uint16_t* qrow = qs + RowTile<D, Q_PAD>::off(qb * 32 + lq, 8 * lh);
        const uint16_t* dorow = dos + RowTile<D, DO_PAD>::off(qb * 32 + lq, 8 * lh);
        constexpr bool V_FORM = kWavesPerSimd<D> == 1;   // see mfma32_acc_v
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
          const u32x4 a = *reinterpret_cast<const u32x4*>(qrow + 16 * kc);
          if constexpr (V_FORM) mfma32_acc_v(sacc, a, kb[kc]); else sacc = mfma32(a, kb[kc], sacc);
        }
        if constexpr (DO_DK) {
#pragma unroll
          for (int kc = 0; kc < KC; ++kc) {
            const u32x4 a = *reinterpret_cast<const u32x4*>(dorow + 16 * kc);
            const u32x4 b = V_LDS ? *reinterpret_cast<const u32x4*>(vrows + RowTile<D>::off(lq, 8 * lh + 16 * kc)) : vb[V_LDS ? 0 : kc];
            if constexpr (V_FORM) mfma32_acc_v(dpacc, a, b); else dpacc = mfma32(a, b, dpacc);
          }
        }
        if constexpr (V_FORM) mfma32_settle(DO_DK ? dpacc : sacc);

        // Causal mask on the raw scores, under a wave-uniform branch of its own (written into the exponential loop it
        // is turned into compare + select on every tile).  Register i holds query mq0 + 8*(i/4) + 4*lh + i%4; the
        // lane-dependent part of the threshold goes into one opaque value so that the 16 thresholds stay immediates.
        if (CAUSAL && mq0 < wk_hi) {
          int rel = key - mq0 - 4 * lh;
          asm volatile("" : "+v"(rel));
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (8 * (i / 4) + i % 4 < rel) sacc[i] = -INFINITY;
        }
        u32x4 pb[2], dsb[2];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float pv[4], ds[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            pv[e] = fast_exp2(sacc[4 * g + e]);
            ds[e] = pv[e] * dpacc[4 * g + e];
          }
          if constexpr (DO_DV) {
            pb[g / 2][2 * (g % 2)] = pack_elts(pv[0], pv[1]);
            pb[g / 2][2 * (g % 2) + 1] = pack_elts(pv[2], pv[3]);
          }
          if constexpr (DO_DK) {
            dsb[g / 2][2 * (g % 2)] = pack_elts(ds[0], ds[1]);
            dsb[g / 2][2 * (g % 2) + 1] = pack_elts(ds[2], ds[3]);
          }
        }
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
          const int kbase = qb * 32 + 16 * cc;
#pragma unroll
          for (int db = 0; db < NDB; ++db) {
            if constexpr (DO_DV) dvacc[db] = mfma32(load_a_trans_of<RowTile<D, DO_PAD>>(dos, kbase, db * 32), pb[cc], dvacc[db]);
            if constexpr (DO_DK) dkacc[db] = mfma32(load_a_trans_of<RowTile<D, Q_PAD>>(qs, kbase, db * 32), dsb[cc], dkacc[db]);
          }
        }
        // without the causal branches the two blocks of a tile are one stretch of code: kept apart, or the scheduler
        // interleaves them and needs both blocks' score registers at once
        if constexpr (!CAUSAL) __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kWavesPerSimd<D> == 1) {
        // one wave per SIMD: the accumulators' home is the accumulation half of the register file, where the MFMAs the
        // compiler selects update them; said here, or it carries them round the loop in the other half and copies all of
        // them over and back on every tile
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
          if constexpr (DO_DV) asm volatile("" : "+a"(dvacc[db]));
          if constexpr (DO_DK) asm volatile("" : "+a"(dkacc[db]));
        }
      }
      if constexpr (!PIPED) store_tile(cur ^ 1);
      cur ^= 1;
      __syncthreads();
    }

    COROPE_ISTAMP(5);
#ifdef COROPE_TRACE
    if (p.trace != nullptr && threadIdx.x == TT) p.trace[(int64_t)item * 16 + 7] = __builtin_readcyclecounter() - clk0;
#endif
    // ---- change of items, all within the wave's own LDS slot.  The table values dK needs on its way out are requested
    // first and land while dV leaves (which waits for nothing); behind them (loads return in the order they were issued)
    // the next item's rows, which land while dK leaves.  After the last item its own rows are requested once more and
    // never used: the request is then unconditional, and the registers it fills are free during the tile loop on every path.
    const int next_item = items.at(round + 1);
    const bool has_next = next_item < total;
    if (!CUT || (it_begin == 0 && it_end == n_iter)) {   // workgroup-uniform
      UnrotateTables<D> tb;
      if constexpr (DO_DK && PREROT) tb.load(p.cos, p.sin, p.fstride, wk_lo, N, opaque_lane());
      if constexpr (DO_DV) store_rows_via_wave_tile<D>(dvacc, p.dv + base, wk_lo, N, 1.f, wave_slot, opaque_lane());
      if constexpr (!LATE) request_rows(has_next ? next_item : item);
      if constexpr (DO_DK) {
        if constexpr (!PREROT) tb.load(p.cos, p.sin, p.fstride, wk_lo, N, opaque_lane());
        // the Q_r operand carried sm_scale * log2(e): ln 2 is what is left of sm_scale
        store_unrotated_rows_via_wave_tile<D>(dkacc, tb, p.dk + base, wk_lo, N, 0.6931471805599453f, wave_slot, opaque_lane());
      }
    } else if constexpr (CUT) {   // a piece of the item: its partial sums
      float* slot = p.parts + piece_slot(items.share(), it_begin == 0) * kDkdvSlotFloats<D, NWAVES> + (int64_t)rb * 32 * D + 4 * opaque_lane();
#pragma unroll
      for (int i = 0; i < NDB * 4; ++i) {
        const int db = i / 4, g = i % 4;
        *reinterpret_cast<f32x4*>(slot + i * 4 * kWave) = f32x4{dvacc[db][4 * g], dvacc[db][4 * g + 1], dvacc[db][4 * g + 2], dvacc[db][4 * g + 3]};
        *reinterpret_cast<f32x4*>(slot + NWAVES * 32 * D + i * 4 * kWave) = f32x4{dkacc[db][4 * g], dkacc[db][4 * g + 1], dkacc[db][4 * g + 2], dkacc[db][4 * g + 3]};
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!LATE) request_rows(has_next ? next_item : item);
    }
    if constexpr (LATE) request_rows(has_next ? next_item : item);
    COROPE_ISTAMP(6);
    if (!has_next) break;
    item = next_item;
    COROPE_ISTAMP(0);
    take_rows();
  }
}

// dV and dK of the items that were cut: one wave per 32 keys of an item (blockIdx.x) and output (blockIdx.y: dV, dK) adds the
// partial accumulators and stores them as the dK+dV kernel would have.
template <int D, int NWAVES, int BLOCK_M, bool CAUSAL>
__global__ __launch_bounds__(kWave) void rope_attn_bwd_dkdv_sum_kernel(BwdParams p, int shares) {
  constexpr int NDB = D / 32, BLOCK_N = NWAVES * 32;
  __shared__ __attribute__((aligned(16))) uint8_t tile[WaveTile<D>::kBytes];
  const int N = p.N, slabs = p.BH / p.H * p.Hkv, GQ = p.H / p.Hkv, m_tiles = (N + BLOCK_M - 1) / BLOCK_M;
  const DkdvTiles t(p.num_blocks, slabs, GQ, m_tiles, CAUSAL ? BLOCK_N / BLOCK_M : 0);
  const int item = blockIdx.x / NWAVES, rb = blockIdx.x % NWAVES, kb = item / slabs, slab = item % slabs;
  const int start = t.start(item), w0 = t.share_of(start, shares), w1 = t.share_of(start + t.first(kb + 1) - t.first(kb) - 1, shares);
  const int row0 = kb * BLOCK_N + rb * 32;
  if (w0 == w1 || row0 >= N) return;   // one piece holds all of the item and has written it
  const float* src = p.parts + blockIdx.y * (NWAVES * 32 * D) + (int64_t)rb * 32 * D + 4 * threadIdx.x;
  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = f32x16{0};
#pragma unroll 1
  for (int w = w0; w <= w1; ++w) {
    const float* slot = src + piece_slot(w, w == w0) * kDkdvSlotFloats<D, NWAVES>;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(slot + (4 * db + g) * 4 * kWave);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[db][4 * g + e] += x[e];
      }
  }
  const int64_t base = (int64_t)slab * N * D;
  if (blockIdx.y == 0) {
    store_rows_via_wave_tile<D>(acc, p.dv + base, row0, N, 1.f, tile);
  } else {
    UnrotateTables<D> tb;
    tb.load(p.cos, p.sin, p.fstride, row0, N);
    store_unrotated_rows_via_wave_tile<D>(acc, tb, p.dk + base, row0, N, 0.6931471805599453f, tile);
  }
}

// The same for few items, whose many pieces one wave would fetch one after the other: a workgroup per 32 keys, output and 64 columns
// (blockIdx.z), a wave per register quad and its partner (columns d and d + D / 2), four pieces in flight.
constexpr int kDkdvSumThreads = 4 * kWave;
constexpr unsigned kSplitSumBlocks = 512;

template <int D, int NWAVES, int BLOCK_M, bool CAUSAL>
__global__ __launch_bounds__(kDkdvSumThreads) void rope_attn_bwd_dkdv_sum_split_kernel(BwdParams p, int shares) {
  constexpr int BLOCK_N = NWAVES * 32, PARTNER = D / 16 * 4 * kWave;
  const int N = p.N, slabs = p.BH / p.H * p.Hkv, GQ = p.H / p.Hkv, m_tiles = (N + BLOCK_M - 1) / BLOCK_M;
  const DkdvTiles t(p.num_blocks, slabs, GQ, m_tiles, CAUSAL ? BLOCK_N / BLOCK_M : 0);
  const int item = blockIdx.x / NWAVES, rb = blockIdx.x % NWAVES, kb = item / slabs, slab = item % slabs;
  const int start = t.start(item), w0 = t.share_of(start, shares), w1 = t.share_of(start + t.first(kb + 1) - t.first(kb) - 1, shares);
  const int lane = threadIdx.x % kWave, i = blockIdx.z * 4 + threadIdx.x / kWave, row = kb * BLOCK_N + rb * 32 + lane % 32;
  if (w0 == w1 || row >= N) return;   // one piece holds all of the item and has written it
  const float* src = p.parts + blockIdx.y * (NWAVES * 32 * D) + (int64_t)rb * 32 * D + 4 * (i * kWave + lane);
  f32x4 a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
  int w = w0;
  auto add = [&](auto count_c) __attribute__((always_inline)) {   // that many pieces
    constexpr int COUNT = decltype(count_c)::value;
    f32x4 x[COUNT], y[COUNT];
#pragma unroll
    for (int u = 0; u < COUNT; ++u) {
      const float* slot = src + piece_slot(w + u, w + u == w0) * kDkdvSlotFloats<D, NWAVES>;
      x[u] = *reinterpret_cast<const f32x4*>(slot);
      y[u] = *reinterpret_cast<const f32x4*>(slot + PARTNER);
    }
#pragma unroll
    for (int u = 0; u < COUNT; ++u) a += x[u], b += y[u];
    w += COUNT;
  };
  while (w + 3 <= w1) add(std::integral_constant<int, 4>{});
  if (w + 1 <= w1) add(std::integral_constant<int, 2>{});
  if (w <= w1) add(std::integral_constant<int, 1>{});
  const int col = 8 * i + 4 * (lane / 32);
  f32x4 o1 = a, o2 = b;
  if (blockIdx.y == 1) {   // (the Q_r operand carried sm_scale * log2(e): ln 2 is what is left of sm_scale)
    const f32x4 c = *reinterpret_cast<const f32x4*>(p.cos + row * p.fstride + col), s = *reinterpret_cast<const f32x4*>(p.sin + row * p.fstride + col);
    a *= 0.6931471805599453f, b *= 0.6931471805599453f;
    o1 = a * c + b * s, o2 = b * c - a * s;
  }
  uint16_t* out = (blockIdx.y == 0 ? p.dv : p.dk) + ((int64_t)slab * N + row) * D + col;
  *reinterpret_cast<u32x2*>(out) = u32x2{pack_elts(o1[0], o1[1]), pack_elts(o1[2], o1[3])};
  *reinterpret_cast<u32x2*>(out + D / 2) = u32x2{pack_elts(o2[0], o2[1]), pack_elts(o2[2], o2[3])};
}

// ===================================================================================== dQ
// Workgroup = NWAVES waves x 32 queries.  Rotated Q rows and dO rows of the wave stay in registers.
// Per key tile (BLOCK_N rows, staged: rotated K and V):
//   S^T  = K_r Q_r^T          (A = K_r rows from LDS, B = Q_r regs)    lane = query, registers = keys
//   dP^T = V dO^T             (A = V rows from LDS,   B = dO regs)
//   dS^T = P^T o (dP^T - delta)                                        (bf16, B-operand shaped)
//   dQ_r^T += K_r^T dS^T      (A = K_r tile read transposed, B = dS^T)
template <int D, int NWAVES, int BLOCK_N>
struct DqCfg {
  static constexpr int kThreads = NWAVES * kWave;
  static constexpr int kBlockM = NWAVES * 32;
  static constexpr int kKTileBytes = RowTile<D, kBothWaysPad>::bytes(BLOCK_N);   // K_r: read row-wise and transposed
  static constexpr int kVTileBytes = RowTile<D>::bytes(BLOCK_N);                 // V: read row-wise
  static constexpr int kStageBytes = kKTileBytes + kVTileBytes;
  static constexpr int kRingBytes = 2 * kStageBytes;
  // behind the ring, per wave: a private tile for its operand rows on their way in and its dQ rows on their way out, and
  // the 32 delta values of its rows
  static constexpr int kWaveBytes = WaveTile<D>::kBytes + 32 * 4;
  static constexpr int kLdsBytes = kRingBytes + NWAVES * kWaveBytes;
  static_assert(kLdsBytes <= 160 * 1024, "LDS of a compute unit");
};

// A slot of partial sums: NWAVES x 32 queries x D of dQ_r, as the accumulators lie ([32-row block][register quad][lane]).
template <int D, int NWAVES>
constexpr int64_t kDqSlotFloats = (int64_t)NWAVES * 32 * D;

// Persistent, like the forward on a pre-rotated K: one workgroup per compute unit walks a balanced list of (head, query
// block) items, the stream of K/V tiles runs on from item to item, and nothing at the change of items needs a workgroup
// barrier (a wave's operand rows and its dQ rows go through an LDS tile of its own).
template <int D, int NWAVES, int BLOCK_N, bool CAUSAL, bool PREROT, bool CUT = false>
__global__ __launch_bounds__(NWAVES* kWave) __attribute__((amdgpu_waves_per_eu(kWavesPerSimd<D>, kWavesPerSimd<D>))) void rope_attn_bwd_dq_kernel(BwdParams p) {
  using Cfg = DqCfg<D, NWAVES, BLOCK_N>;
  constexpr int NT = Cfg::kThreads;
  // (A causal launch that is cut changes items often, and more of a change goes through scratch memory in this form: B1 H2 N8000 270 -> 324 us.)
  constexpr bool PIPED = D > 128 && PREROT && !(CUT && CAUSAL);
  constexpr bool STRIDED = D <= 128, DELTA_ACC = D == 64;
  constexpr int KC = D / 16, NDB = D / 32, NKB = BLOCK_N / 32;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int lq = lane % 32, lh = lane / 32;
  // 32-row block of the item this wave owns; waves w and w + 4 share a SIMD, blocks (0,7), (1,6), (2,5), (3,4) give
  // every SIMD the same number of diagonal tiles
  const int rb = NWAVES == 8 ? (wave < 4 ? wave : 11 - wave) : wave;
  [[maybe_unused]] constexpr int TT = NWAVES == 8 ? 4 * kWave : (NWAVES - 1) * kWave;   // stamping thread: first lane of the wave with the last rows
  const int N = p.N;
  uint8_t* const wave_tile = smem + Cfg::kRingBytes + wave * Cfg::kWaveBytes;
  float* const wave_delta = reinterpret_cast<float*>(wave_tile + WaveTile<D>::kBytes);

  const int n_k_tiles = (N + BLOCK_N - 1) / BLOCK_N;
  const QueryWork<CUT> items(p.num_blocks, p.BH, n_k_tiles, CAUSAL ? Cfg::kBlockM / BLOCK_N : 0);
  const int total = items.total;   // item i (heaviest first): query block num_blocks - 1 - i / BH of head i % BH
  auto tiles_of = [&](int mb) {
    return CAUSAL ? min((mb * Cfg::kBlockM + Cfg::kBlockM + BLOCK_N - 1) / BLOCK_N, n_k_tiles) : n_k_tiles;
  };

  // ---- the stream of K/V tiles: a cursor one tile ahead of the tile being consumed -------------------------------------
  RopeStage<D, BLOCK_N, NT, PREROT, false, kBothWaysPad> kst;
  CopyStage<D, BLOCK_N, NT> vst;
  int l_round = 0, l_tile = 0, l_tiles;
  const uint16_t *l_kg, *l_vg;
  auto load_item = [&](int r) {    // false: no such item
    const int i = items.at(r);
    if (i >= total) return false;
    const int64_t kv_base = (int64_t)kv_slab(i % p.BH, p.H, p.Hkv) * N * D;
    l_kg = (PREROT ? p.k_rot : p.k) + kv_base;
    l_vg = v_slab_of<D, STRIDED>(p, kv_slab(i % p.BH, p.H, p.Hkv));
    l_tile = items.begin(i);
    l_tiles = items.end(i, tiles_of(p.num_blocks - 1 - i / p.BH));
    return true;
  };
  auto load_next_tile = [&]() __attribute__((always_inline)) {   // moves the cursor on and requests that tile
    if (l_tile + 1 < l_tiles) {
      ++l_tile;
    } else if (load_item(l_round + 1)) {
      ++l_round;
    }   // else: past the last tile of the last item; the same tile is requested again and never used
    kst.load(l_kg, p.cos, p.sin, p.fstride, l_tile * BLOCK_N, N);
    vst.load(l_vg, l_tile * BLOCK_N, N, v_row_bytes<D, STRIDED>(p));
  };
  auto k_tile = [&](int buf) { return reinterpret_cast<uint16_t*>(smem + buf * Cfg::kStageBytes); };
  auto v_tile = [&](int buf) { return reinterpret_cast<uint16_t*>(smem + buf * Cfg::kStageBytes + Cfg::kKTileBytes); };
  int cur = 0;   // ring stage of the tile being consumed

  // ---- operand rows of an item: Q_r (rotated and scaled here unless a pre-rotated copy is given), dO, O for delta ------
  // (the lane index goes in as a value the optimiser cannot see through: the per-lane address parts of these steps are
  // then recomputed per item instead of being kept in registers, or in scratch memory, across the whole loop)
  auto opaque_lane = [&]() __attribute__((always_inline)) {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  WaveRows<D, !PREROT> qrows;
  WaveRows<D, false> dorows, orows;
  float lse_q, delta_in;
  u32x4 qb[KC], dob[KC];
  float delta_q;
  auto request_rows = [&](int i) __attribute__((always_inline)) {
    const int bh = i % p.BH, row0 = (p.num_blocks - 1 - i / p.BH) * Cfg::kBlockM + rb * 32;
    const int64_t base = (int64_t)bh * N * D;
    const int l = opaque_lane();
    qrows.load((PREROT ? p.q_rot : p.q) + base, p.cos, p.sin, p.fstride, row0, N, l);
    const uint16_t* dog = STRIDED ? p.do_slab(bh) : p.d_o + base;
    dorows.load(dog, nullptr, nullptr, 0, row0, N, l, do_row_bytes<D, STRIDED>(p));
    // (without O the dO rows are requested twice: the request is then unconditional and the registers it fills are free
    // during the tile loop on every path)
    orows.load(p.o != nullptr ? p.o + base : dog, nullptr, nullptr, 0, row0, N, l, p.o != nullptr ? (uint32_t)D * 2 : do_row_bytes<D, STRIDED>(p));
    const int q_c = min(row0 + l % 32, N - 1);
    lse_q = p.lse[(int64_t)bh * N + q_c];
    // delta_i = sum_d o_id * do_id (reference _attn_bwd_preprocess, :324-337): read from the preprocess pass, or -- when the
    // caller hands over O instead -- computed here for the rows this workgroup owns and written out for the dK kernel,
    // which then has to run after this one.
    delta_in = 0.f;
    if (p.o == nullptr) delta_in = p.delta[(int64_t)bh * N + q_c];
  };
  auto take_rows = [&](int i) __attribute__((always_inline)) {
    const int bh = i % p.BH, row0 = (p.num_blocks - 1 - i / p.BH) * Cfg::kBlockM + rb * 32;
    const int l = opaque_lane();
    park_rows<D>(qrows, qb, wave_tile, p.qk_scale, l);   // Q_r carries qk_scale (a pre-rotated copy already does)
    park_plain_rows<D>(dorows, dob, wave_tile, l);
    delta_q = delta_in;
    if (p.o != nullptr) {
      // 16 lanes per row: O and dO in registers, same chunk order
      constexpr int CPR = D / 8, RPI = kWave / CPR;
#pragma unroll
      for (int i2 = 0; i2 < 32 / RPI; ++i2) {
        const int r = RPI * i2 + l / CPR, ch = l % CPR;
        const u32x4 ow = orows.x[i2], dw = dorows.x[i2];
        float acc = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) acc += elt_lo(ow[w]) * elt_lo(dw[w]) + elt_hi(ow[w]) * elt_hi(dw[w]);
        if constexpr (CPR == 16) {
          acc = row16_sum(acc);
        } else {
#pragma unroll
          for (int m = CPR / 2; m >= 1; m >>= 1) acc += __shfl_xor(acc, m);
        }
        if (ch == 0) wave_delta[r] = acc;
      }
      lds_order();
      delta_q = wave_delta[l % 32];
      lds_order();
      if (l / 32 == 0 && row0 + l % 32 < N) p.delta[(int64_t)bh * N + row0 + l % 32] = delta_q;
    }
  };

  // ---- first item: nothing to hide its prologue behind ----------------------------------------------------------------
  int item = items.at(0);
  COROPE_ISTAMP(0);
  load_item(0);
  kst.load(l_kg, p.cos, p.sin, p.fstride, l_tile * BLOCK_N, N);
  vst.load(l_vg, l_tile * BLOCK_N, N, v_row_bytes<D, STRIDED>(p));
  request_rows(item);
  take_rows(item);
  kst.store_rows(k_tile(0));
  vst.store_rows(v_tile(0));
  __syncthreads();

  for (int round = 0;; ++round) {
    const int bh = item % p.BH, mb = p.num_blocks - 1 - item / p.BH;
    const int m0 = mb * Cfg::kBlockM;
    const int t_begin = items.begin(item), n_tiles = items.end(item, tiles_of(mb));   // of this workgroup's piece of the item
    const int q_row = m0 + rb * 32 + lq;
    const int wq_lo = m0 + rb * 32, wq_hi = wq_lo + 31;
    const int key_limit = CAUSAL ? q_row : N - 1;   // last key this lane's query attends to
    // last tile this wave's rows can see
    const int t_last = __builtin_amdgcn_readfirstlane(CAUSAL ? min(n_tiles - 1, wq_hi / BLOCK_N) : n_tiles - 1);
    COROPE_ISTAMP(1);
    COROPE_ISTAMP_ID(n_tiles);
#ifdef COROPE_TRACE
    const uint64_t clk0 = __builtin_readcyclecounter();
#endif

    f32x16 dqacc[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i) dqacc[i] = f32x16{0};
    // S - M leaves the matrix cores: the score products start from -M of the lane's query in every register
    f32x16 msb;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float x = -lse_q;
      asm volatile("" : "+v"(x));   // sixteen values of their own: one value in sixteen places is tied to the first of them
      msb[i] = x;
    }
    // the wave's operands have landed on every path into the loop (left to their first use, the wait would sit inside
    // the loop and there also wait for the next tile's loads)
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) asm volatile("" ::"v"(qb[kc]), "v"(dob[kc]));
    asm volatile("" ::"v"(delta_q));
    // ... and dP - delta, where the registers for it are there (D = 64: B2 H16 N4096 128 -> 122.5 us; at D = 128, with -delta from the LDS, 440 -> 460)
    f32x16 mdb;
    if constexpr (DELTA_ACC) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float x = -delta_q;
        asm volatile("" : "+v"(x));
        mdb[i] = x;
      }
    }

    if constexpr (PIPED) {   // the operand rows' home, and the accumulators', is the accumulation half of the register file
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) asm volatile("" : "+a"(qb[kc]), "+a"(dob[kc]));
#pragma unroll
      for (int db = 0; db < NDB; ++db) asm volatile("" : "+a"(dqacc[db]));
    }

    auto stage_next = [&]() __attribute__((always_inline)) {
      kst.store_rows(k_tile(cur ^ 1));
      vst.store_rows(v_tile(cur ^ 1));
    };

    for (int t = t_begin; t <= t_last; ++t) {
      const int n0 = t * BLOCK_N;
#ifdef COROPE_TRACE
      if (t == 1) COROPE_ISTAMP(3);
      if (n0 == m0) COROPE_ISTAMP(4);
#endif
      load_next_tile();
      const uint16_t* ks = k_tile(cur);
      const uint16_t* vs = v_tile(cur);
      const bool need_mask = (CAUSAL && n0 + BLOCK_N - 1 > wq_lo) || (!CAUSAL && n0 + BLOCK_N > N);
      u32x4 dsb[BLOCK_N / 16];
      if constexpr (PIPED) {
        // One stream of 3 x 16 products as in the dK+dV kernel at this head dim: the exponentials between the dP products, the second half of dS
        // between the first half of the dQ products (the first half of dS is all that waits), then the next tile's staging.  As the compiler scheduled
        // it: B2 H16 N2048 171 -> 158 us, B2 H8 N3000 not causal 285 -> 253.
        static_assert(NKB == 1, "one 32-key block per tile");
        constexpr int RING = 4, TOTAL = 3 * KC;
        using KT = RowTile<D, kBothWaysPad>;
        const uint16_t *k_l = ks + KT::off(lq, 8 * lh), *v_l = vs + RowTile<D>::off(lq, 8 * lh);
        const uint16_t* k_t = ks + KT::off(4 * lh + lane % 16 / 4, 16 * (lane / 16 % 2) + 4 * (lane % 4));
        auto operand = [&](int n) __attribute__((always_inline)) {
          const int i = n % KC;
          return n < KC       ? *reinterpret_cast<const u32x4*>(k_l + 16 * i)
                 : n < 2 * KC ? *reinterpret_cast<const u32x4*>(v_l + 16 * i)
                              : load_a_trans_lane<KT>(k_t, 16 * (i / NDB), i % NDB * 32);
        };
        u32x4 ring[RING];
#pragma unroll
        for (int n = 0; n < RING; ++n) ring[n] = operand(n);
        f32x16 sacc, dpacc;
        auto ds_pair = [&](int j) __attribute__((always_inline)) {
          dsb[j / 4][j % 4] = pack_elts(sacc[2 * j] * (dpacc[2 * j] - delta_q), sacc[2 * j + 1] * (dpacc[2 * j + 1] - delta_q));
        };
        __builtin_amdgcn_sched_barrier(0);
        static_for<TOTAL>([&](auto n_c) __attribute__((always_inline)) {
          constexpr int n = decltype(n_c)::value, slot = n / KC, i = n % KC;
          if constexpr (slot == 2 && i == 0) {
            mfma32_settle(dpacc);
#pragma unroll
            for (int j = 0; j < 4; ++j) ds_pair(j);
            __builtin_amdgcn_sched_barrier(0);
          }
          const u32x4 a = ring[n % RING];
          if constexpr (slot == 0) { if constexpr (i == 0) sacc = mfma32_from_aq(a, qb[0], msb); else mfma32_acc_aq(sacc, a, qb[i]); }
          if constexpr (slot == 1) { if constexpr (i == 0) dpacc = mfma32_zero_aq(a, dob[0]); else mfma32_acc_aq(dpacc, a, dob[i]); }
          if constexpr (slot == 2) dqacc[i % NDB] = mfma32(a, dsb[i / NDB], dqacc[i % NDB]);
          if constexpr (n + RING < TOTAL) ring[n % RING] = operand(n + RING);
          if constexpr (slot == 1 && i == 0) asm volatile("s_nop 7");   // (nothing reads the scores behind product 0, which waits a little instead)
          if constexpr (slot == 1 && i == 1) {
            if (need_mask) {
              int rel = key_limit - n0 - 4 * lh;
              asm volatile("" : "+v"(rel));
#pragma unroll
              for (int x = 0; x < 16; ++x)
                if (8 * (x / 4) + x % 4 > rel) sacc[x] = -INFINITY;
            }
          }
          if constexpr (slot == 1) {
#pragma unroll
            for (int e = (i == 0 ? 0 : (i - 1) * 16 / (KC - 1)); e < (i == 0 ? 0 : i * 16 / (KC - 1)); ++e) sacc[e] = fast_exp2(sacc[e]);
          }
          if constexpr (slot == 2 && i < 4) ds_pair(4 + i);
          if constexpr (slot == 2 && i == KC - 2) stage_next();
          __builtin_amdgcn_sched_barrier(0);
        });
#pragma unroll
        for (int db = 0; db < NDB; ++db) asm volatile("" : "+a"(dqacc[db]));
      }
#pragma unroll
      for (int kb = 0; kb < (PIPED ? 0 : NKB); ++kb) {
        f32x16 sacc, dpacc;   // dP starts from a literal zero, S from -M
        const uint16_t* krow = ks + RowTile<D, kBothWaysPad>::off(kb * 32 + lq, 8 * lh);
        const uint16_t* vrow = vs + RowTile<D>::off(kb * 32 + lq, 8 * lh);
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
          // (mfma32_from is for builds whose accumulators stay in the registers it names: with one wave per SIMD the
          // compiler keeps them in the other half of the register file and would copy the result there at once)
          sacc = kc > 0 ? mfma32(*reinterpret_cast<const u32x4*>(krow + 16 * kc), qb[kc], sacc)
                 : kWavesPerSimd<D> == 2 ? mfma32_from(*reinterpret_cast<const u32x4*>(krow), qb[0], msb)
                                         : mfma32(*reinterpret_cast<const u32x4*>(krow), qb[0], msb);
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
          dpacc = kc > 0 ? mfma32(*reinterpret_cast<const u32x4*>(vrow + 16 * kc), dob[kc], dpacc)
                  : DELTA_ACC ? mfma32_from(*reinterpret_cast<const u32x4*>(vrow), dob[0], mdb)
                              : mfma32(*reinterpret_cast<const u32x4*>(vrow), dob[0], f32x16{0});
        // mask on the raw scores under a wave-uniform branch of its own; register i holds key
        // n0 + 32*kb + 8*(i/4) + 4*lh + i%4, the lane-dependent part of the threshold goes into one opaque value
        if (need_mask) {
          int rel = key_limit - n0 - 4 * lh;
          asm volatile("" : "+v"(rel));
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (kb * 32 + 8 * (i / 4) + i % 4 > rel) sacc[i] = -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
          float ds[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            float pv = fast_exp2(sacc[i + e]);
            ds[e] = DELTA_ACC ? pv * dpacc[i + e] : pv * (dpacc[i + e] - delta_q);
          }
          dsb[2 * kb + i / 8][(i % 8) / 2] = pack_elts(ds[0], ds[1]);
        }
      }
#pragma unroll
      for (int c = 0; c < (PIPED ? 0 : BLOCK_N / 16); ++c)
#pragma unroll
        for (int db = 0; db < NDB; ++db)
          dqacc[db] = mfma32(load_a_trans_of<RowTile<D, kBothWaysPad>>(ks, 16 * c, db * 32), dsb[c], dqacc[db]);
      if constexpr (!PIPED) stage_next();
      cur ^= 1;
      __syncthreads();
    }
    COROPE_ISTAMP(5);
#ifdef COROPE_TRACE
    if (p.trace != nullptr && threadIdx.x == TT) p.trace[(int64_t)item * 16 + 7] = __builtin_readcyclecounter() - clk0;
#endif
    // The next item's rows are requested as soon as the registers of this item's rows are free.  (After the last item its
    // own rows are requested once more and never used: the request is then unconditional, and the registers it fills are
    // free during the tile loop on every path.)
    // Ahead of them go the table values that the item's dQ rows need on their way out: loads return in the order they
    // were issued, and those must not wait for the next item's rows.
    // (Only on pre-rotated operands: rows that are rotated here travel with their own table values, and both sets do not
    // fit the registers.)
    UnrotateTables<D> tb;
    if constexpr (PREROT) tb.load(p.cos, p.sin, p.fstride, wq_lo, N, opaque_lane());
    const int next_item = items.at(round + 1);
    const bool has_next = next_item < total;
    request_rows(has_next ? next_item : item);
    // of the tiles entirely above this wave's diagonal it only stages its share
    for (int t = CUT ? max(t_begin, t_last + 1) : t_last + 1; t < n_tiles; ++t) {
      load_next_tile();
      stage_next();
      cur ^= 1;
      __syncthreads();
    }
    // dQ_r -> dQ: scaled, un-rotated in fp32, rounded once, whole rows per store
    if constexpr (!PREROT) tb.load(p.cos, p.sin, p.fstride, wq_lo, N, opaque_lane());
    if (!CUT || (t_begin == 0 && n_tiles == tiles_of(mb))) {   // workgroup-uniform
      store_unrotated_rows_via_wave_tile<D>(dqacc, tb, p.dq + (int64_t)bh * N * D, wq_lo, N, p.sm_scale, wave_tile, opaque_lane());
    } else if constexpr (CUT) {   // a piece of the item: its partial sums
      float* slot = p.dq_parts + piece_slot(items.share(), t_begin == 0) * kDqSlotFloats<D, NWAVES> + (int64_t)rb * 32 * D + 4 * opaque_lane();
#pragma unroll
      for (int i = 0; i < NDB * 4; ++i)
        *reinterpret_cast<f32x4*>(slot + i * 4 * kWave) =
            f32x4{dqacc[i / 4][4 * (i % 4)], dqacc[i / 4][4 * (i % 4) + 1], dqacc[i / 4][4 * (i % 4) + 2], dqacc[i / 4][4 * (i % 4) + 3]};
    }
    COROPE_ISTAMP(6);
    if (!has_next) break;
    item = next_item;
    COROPE_ISTAMP(0);
    take_rows(item);
  }
}

// dQ of the items that were cut: a workgroup per 32 rows of an item, a wave per register quad and its partner (columns d and d + D / 2): adds the
// pieces' accumulators, un-rotates, rounds.
template <int D, int NWAVES, int BLOCK_N, bool CAUSAL>
__global__ __launch_bounds__(D / 16 * kWave) void rope_attn_bwd_dq_sum_kernel(BwdParams p, int shares) {
  constexpr int BLOCK_M = NWAVES * 32, PARTNER = D / 16 * 4 * kWave;
  const int N = p.N;
  const QueryTiles t(p.num_blocks, p.BH, (N + BLOCK_N - 1) / BLOCK_N, CAUSAL ? BLOCK_M / BLOCK_N : 0);
  const int item = blockIdx.x / NWAVES, rb = blockIdx.x % NWAVES, mb = p.num_blocks - 1 - item / p.BH;
  const int start = t.start(item), w0 = t.share_of(start, shares), w1 = t.share_of(start + t.first(mb + 1) - t.first(mb) - 1, shares);
  const int lane = threadIdx.x % kWave, i = threadIdx.x / kWave, row = mb * BLOCK_M + rb * 32 + lane % 32;
  if (w0 == w1 || row >= N) return;   // one piece holds all of the item and has written it
  const float* src = p.dq_parts + (int64_t)rb * 32 * D + 4 * (i * kWave + lane);
  const int col = 8 * i + 4 * (lane / 32);
  const f32x4 c = *reinterpret_cast<const f32x4*>(p.cos + row * p.fstride + col), s = *reinterpret_cast<const f32x4*>(p.sin + row * p.fstride + col);
  f32x4 a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
  for (int w = w0; w <= w1; w += 4) {   // eight loads in flight
    f32x4 x[4], y[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float* slot = src + piece_slot(min(w + u, w1), min(w + u, w1) == w0) * kDqSlotFloats<D, NWAVES>;
      x[u] = *reinterpret_cast<const f32x4*>(slot);
      y[u] = *reinterpret_cast<const f32x4*>(slot + PARTNER);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (w + u <= w1) a += x[u], b += y[u];
  }
  a *= p.sm_scale, b *= p.sm_scale;
  const f32x4 o1 = a * c + b * s, o2 = b * c - a * s;
  uint16_t* out = p.dq + ((int64_t)(item % p.BH) * N + row) * D + col;
  *reinterpret_cast<u32x2*>(out) = u32x2{pack_elts(o1[0], o1[1]), pack_elts(o1[2], o1[3])};
  *reinterpret_cast<u32x2*>(out + D / 2) = u32x2{pack_elts(o2[0], o2[1]), pack_elts(o2[2], o2[3])};
}

// ===================================================================================== launchers
template <int D>
constexpr int kDkdvBlockM = D > 128 ? 32 : 64;   // what fits the LDS beside the waves' own slots
template <int D>
constexpr int kDkdvCutWaves = D > 128 ? 4 : 8;
template <int D, bool DO_DV, bool DO_DK, int NWAVES>
using DkdvCfgOf = DkdvCfg<D, NWAVES, kDkdvBlockM<D>, DO_DK ? (DO_DV ? kDkdvBothWaysPad : 8) : 32, DO_DK ? kDkdvBothWaysPad : 8>;

template <int D, bool CAUSAL, bool DO_DV, bool DO_DK, bool PREROT, int NWAVES>
static hipError_t launch_dkdv_waves(BwdParams p, hipStream_t stream) {
  using Cfg = DkdvCfgOf<D, DO_DV, DO_DK, NWAVES>;
  auto kern = rope_attn_bwd_dkdv_kernel<D, NWAVES, kDkdvBlockM<D>, CAUSAL, DO_DV, DO_DK, PREROT>;
  static std::atomic<uint64_t> lds_ok{0};
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes, lds_ok); e != hipSuccess) return e;
  p.num_blocks = (p.N + Cfg::kBlockN - 1) / Cfg::kBlockN;
#ifdef COROPE_TRACE
  p.trace = g_trace_buf;
#endif
  const unsigned grid = persistent_grid((int64_t)p.num_blocks * (p.BH / p.H * p.Hkv), NWAVES, Cfg::kLdsBytes);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(Cfg::kThreads), Cfg::kLdsBytes, stream, p);
  return hipGetLastError();
}

template <int D, bool DO_DV, bool DO_DK>
static bool dkdv_small_tiles(int N, int slabs) {
  return use_small_tiles(N, slabs, DkdvCfgOf<D, DO_DV, DO_DK, 4>::kLdsBytes);
}

// How many pieces the tiles of the fused dK+dV launch on rotated operands are cut into; 0: whole items.  Whole items take as
// long as the workgroup that is dealt the most.  Cut, every workgroup has the same number of tiles, and what is added is the
// partial sums' way through memory (each of the about `shares` + `items` pieces written and read once) and one more launch.
// The constants are measured ones: microseconds per tile of a full chip (a tile of a 128-key item with four waves on its
// compute unit takes 0.85 of a 256-key item's; with part of the chip idle the clock is higher and tiles are up to a quarter
// shorter), 6 TB/s for the partial sums, 10 us for the launch and the longer change of items.  Backward, whole / cut, B Hq Hkv N at
// D = 128: 1 32 8 3001 676 / 285 us, 4 8 1 1500 633 / 129, 1 8 8 4096 337 / 244, 1 16 16 2048 181 / 150, and on the other side
// 2 16 16 2048 182 / 188, 2 40 40 1500 196 / 254.
// At D = 256 (one wave per SIMD) what is not tiles weighs more: the constants there are those of a fit to both forms' launches at 660 shapes, 1 to 96
// heads of 200 to 8000 rows, grouped ones among them, with the most items that a piece meets; 3 to 5 % of a launch off at the root mean square.  The form chosen
// is more than 3 % slower than the other at 9 of them (with the constants of D = 128: 39, by up to 26 %).  dK+dV launch, whole / cut with its sums, B1 H N:
// causal 1 2048 115 / 32, 4 4096 219 / 126, 10 2048 119 / 103, 10 500 40 / 29, not 24 1500 182 / 150, and on the other side causal 16 2048 123 / 135, 20 1024
// 68 / 76, 10 4096 236 / 257, not 40 1500 194 / 222.
template <int D>
static int dkdv_shares(int N, int slabs, int group, bool causal) {
  constexpr int BM = kDkdvBlockM<D>, CW = kDkdvCutWaves<D>, kMost = 16;
  if (g_tile_rows.load(std::memory_order_relaxed) != 0) return 0;   // a form was asked for
  const int m_tiles = (N + BM - 1) / BM, cus = device_cu_count();
  const bool small = D <= 128 && dkdv_small_tiles<D, true, true>(N, slabs);
  const int block = small || D > 128 ? 128 : 256, nb = (N + block - 1) / block;
  const int slots = cus * (small && fits_twice(DkdvCfgOf<D, true, true, 4>::kLdsBytes) ? 2 : 1);
  const int64_t n_items = (int64_t)nb * slabs;
  if (n_items > (int64_t)kMost * slots || (int64_t)n_items * group * m_tiles >= (1ll << 30)) return 0;   // many rounds even out
  const int grid = (int)std::min<int64_t>(n_items, slots);
  const int64_t longest = most_tiles_dealt(n_items, grid, [&](int64_t i) -> int64_t { return group * (m_tiles - (causal ? (int)(i / slabs) * (block / BM) : 0)); });
  const DkdvTiles t((N + CW * 32 - 1) / (CW * 32), slabs, group, m_tiles, causal ? CW * 32 / BM : 0);
  const int shares = std::max(1, std::min(cus, t.total_tiles / 4));
  const float moved = (float)(shares + std::min<int64_t>(t.nb * (int64_t)slabs, shares)) * kDkdvSlotFloats<D, CW> * 8;
  if constexpr (D > 128) {
    const float busy = std::min(1.f, (float)t.total_tiles / ((float)longest * cus));
    const float whole = 1.9f * longest * (0.75f + 0.25f * busy) + 4.f * ((n_items + grid - 1) / grid) + 11.f;
    const int tiles = (t.total_tiles + shares - 1) / shares;
    return (causal ? 2.3f : 1.92f) * tiles + 4.5f * most_items_met(t, t.per_slab, shares) + 11.5f + moved / 9e6f < whole ? shares : 0;
  }
  const float tile_us = D == 64 ? 1.7f : 3.3f;
  const float busy = std::min(1.f, (float)t.total_tiles * (block == CW * 32 ? 1.f : 2.f) / ((float)longest * cus));
  const float whole = (small ? 0.85f : 1.f) * longest * tile_us * (0.75f + 0.25f * busy);
  const float cut = t.total_tiles * tile_us / shares + 10.f + moved / 6e6f;
  return cut < 0.95f * whole ? shares : 0;
}

int64_t bwd_dkdv_parts_bytes(int B, int H, int Hkv, int N, int D, bool causal) {
  const int slabs = B * Hkv, group = H / Hkv;
  if (D == 64) return 8 * dkdv_shares<64>(N, slabs, group, causal) * kDkdvSlotFloats<64, kDkdvCutWaves<64>>;
  if (D == 128) return 8 * dkdv_shares<128>(N, slabs, group, causal) * kDkdvSlotFloats<128, kDkdvCutWaves<128>>;
  return 8 * dkdv_shares<256>(N, slabs, group, causal) * kDkdvSlotFloats<256, kDkdvCutWaves<256>>;
}

template <int D, bool CAUSAL>
static hipError_t launch_dkdv_cut(BwdParams p, int shares, hipStream_t stream) {
  constexpr int NWAVES = kDkdvCutWaves<D>, BM = kDkdvBlockM<D>;
  using Cfg = DkdvCfgOf<D, true, true, NWAVES>;
  auto kern = rope_attn_bwd_dkdv_kernel<D, NWAVES, BM, CAUSAL, true, true, true, true>;
  static std::atomic<uint64_t> lds_ok{0};
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes, lds_ok); e != hipSuccess) return e;
  p.num_blocks = (p.N + Cfg::kBlockN - 1) / Cfg::kBlockN;
#ifdef COROPE_TRACE
  p.trace = nullptr;
#endif
  hipLaunchKernelGGL(kern, dim3(shares), dim3(Cfg::kThreads), Cfg::kLdsBytes, stream, p);
  const unsigned blocks = (unsigned)p.num_blocks * (p.BH / p.H * p.Hkv) * NWAVES;
  // One wave per 32 keys reads its pieces at the memory's rate once there are waves enough; below that the pieces' latencies set the time.
  // us, one wave / split, by blocks of 32 keys: 24 (B1 Hq8 Hkv1 N700 D128) 12.8 / 5.4, 64 (B2 Hq16 Hkv2 N512 D256) 28.0 / 12.2, 128 (B1 Hq16 Hkv4 N1024 D128)
  // 11.4 / 8.5, 496 (B1 H4 N3900 D256) 21.4 / 19.2, 512 (B1 H8 N2048 D128) 15.3 / 15.3, 768 (B1 Hq32 Hkv8 N3001 D128) 17.7 / 18.9, 1536 (B2 H8 N3000 D256) 19.3 / 25.5.
  if (blocks < kSplitSumBlocks)
    hipLaunchKernelGGL((rope_attn_bwd_dkdv_sum_split_kernel<D, NWAVES, BM, CAUSAL>), dim3(blocks, 2, D / 64), dim3(kDkdvSumThreads), 0, stream, p, shares);
  else
    hipLaunchKernelGGL((rope_attn_bwd_dkdv_sum_kernel<D, NWAVES, BM, CAUSAL>), dim3(blocks, 2), dim3(kWave), 0, stream, p, shares);
  return hipGetLastError();
}

template <int D, bool CAUSAL, bool DO_DV, bool DO_DK, bool PREROT>
static hipError_t launch_dkdv_cfg(const BwdParams& p, hipStream_t stream) {
  if constexpr (DO_DV && DO_DK && PREROT)
    if (p.parts != nullptr)
      if (const int shares = dkdv_shares<D>(p.N, p.BH / p.H * p.Hkv, p.H / p.Hkv, CAUSAL); shares > 0)
        return launch_dkdv_cut<D, CAUSAL>(p, shares, stream);
  if constexpr (D > 128) {
    return launch_dkdv_waves<D, CAUSAL, DO_DV, DO_DK, PREROT, 4>(p, stream);   // 4 waves x 512 registers
  } else {
    return dkdv_small_tiles<D, DO_DV, DO_DK>(p.N, p.BH / p.H * p.Hkv) ? launch_dkdv_waves<D, CAUSAL, DO_DV, DO_DK, PREROT, 4>(p, stream)
                                                                      : launch_dkdv_waves<D, CAUSAL, DO_DV, DO_DK, PREROT, 8>(p, stream);
  }
}

template <int D>
constexpr int kDqBlockN = D > 128 ? 32 : 64;   // what fits the LDS beside the waves' own tiles
template <int D>
constexpr int kDqCutWaves = D > 128 ? 4 : 8;
template <int D, bool CAUSAL, bool PREROT, int NWAVES>
static hipError_t launch_dq_waves(BwdParams p, hipStream_t stream) {
  constexpr int BLOCK_N = kDqBlockN<D>;
  using Cfg = DqCfg<D, NWAVES, BLOCK_N>;
  auto kern = rope_attn_bwd_dq_kernel<D, NWAVES, BLOCK_N, CAUSAL, PREROT>;
  static std::atomic<uint64_t> lds_ok{0};
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes, lds_ok); e != hipSuccess) return e;
  p.num_blocks = (p.N + Cfg::kBlockM - 1) / Cfg::kBlockM;
#ifdef COROPE_TRACE
  p.trace = g_trace_buf;
#endif
  const unsigned grid = persistent_grid((int64_t)p.num_blocks * p.BH, NWAVES, Cfg::kLdsBytes);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(Cfg::kThreads), Cfg::kLdsBytes, stream, p);
  return hipGetLastError();
}

// How many pieces the key tiles of the dQ launch on rotated operands are cut into; 0: whole items.  As dkdv_shares: with few heads the longest
// whole item (a sequence's last queries, which see all of its keys) sets the time however many compute units are idle.  Measured
// constants, in microseconds: a tile of a full chip, a change of items (items_crossed: at most so many a piece, and one), the launch.  dQ launch, whole / cut
// with its sums, B1 H N: D = 128: 8 4096 159 / 87, 4 8192 296 / 132, 1 10000 330 / 66, 8 3000 not causal 119 / 80, and on the other side 16 4096 153 / 152, 40 1100 53 / 64; D = 64: 8 4096 63 / 50, 4 16384 276 / 239, 2 3000
// not causal 46 / 27, 16 1500 27.5 / 28.2.
// At D = 256 nothing hides a change of items with one wave per SIMD, and the cut kernels send 130 to 147 registers through scratch there (none in the tile
// loop): the constants are those of a fit as in dkdv_shares, with the most items that a piece meets.  The form chosen is more than 3 % slower than the
// other at 4 of the 660 shapes (with the constants of the kernels before: 56, by up to 50 %).  Causal 2 2048 92 / 58, 4 1500 73 / 58, 1 1024 54 / 48, and on the other side 3 8000 308 / 367, 4 4096
// 168 / 187, 8 2048 95 / 131; not causal 4 1024 57 / 43, 12 4096 373 / 341, 24 1500 162 / 148, and on the other side 6 700 45 / 66, 10 2048 103 / 120, 40 1500 171 / 235.
template <int D>
static int dq_shares(int N, int BH, bool causal) {
  constexpr int BN = kDqBlockN<D>, CW = kDqCutWaves<D>, kMost = 16;
  if (g_tile_rows.load(std::memory_order_relaxed) != 0) return 0;   // a form was asked for
  const int k_tiles = (N + BN - 1) / BN, cus = device_cu_count();
  const bool small = D <= 128 && use_small_tiles(N, BH, DqCfg<D, 4, BN>::kLdsBytes);
  const int block = small || D > 128 ? 128 : 256, nb = (N + block - 1) / block;
  const int slots = cus * (small && fits_twice(DqCfg<D, 4, BN>::kLdsBytes) ? 2 : 1);
  const int64_t n_items = (int64_t)nb * BH;
  if (n_items > (int64_t)kMost * slots || n_items * k_tiles >= (1ll << 30)) return 0;   // many rounds even out
  const int grid = (int)std::min<int64_t>(n_items, slots);
  const int64_t longest = most_tiles_dealt(n_items, grid, [&](int64_t i) -> int64_t { return causal ? std::min((nb - (int)(i / BH)) * (block / BN), k_tiles) : k_tiles; });
  const QueryTiles t((N + CW * 32 - 1) / (CW * 32), BH, k_tiles, causal ? CW * 32 / BN : 0);
  const int shares = std::max(1, std::min(cus, t.total_tiles / 4));
  const float moved = (float)(shares + std::min<int64_t>(t.nb * (int64_t)BH, shares)) * kDqSlotFloats<D, CW> * 8;
  const int rounds = (int)((n_items + grid - 1) / grid);
  if constexpr (D > 128) {
    const float busy = std::min(1.f, (float)t.total_tiles / ((float)longest * cus));
    const float whole = 1.5f * longest * (0.75f + 0.25f * busy) + 6.4f * rounds + 11.6f;
    const int tiles = (t.total_tiles + shares - 1) / shares, met = most_items_met(t, t.per_head, shares);
    const float cut = causal ? 3.5f * tiles + 3.3f * met + 22.f + moved / 3.4e6f : 1.45f * tiles + 21.f * met + 3.f + moved / 5.4e6f;
    return cut < whole ? shares : 0;
  }
  constexpr float kWholeTile = D == 64 ? 1.25f : 2.8f, kTile = D == 64 ? 1.5f : 2.9f, kChange = D == 64 ? 3.5f : 5.f;
  const float busy = std::min(1.f, (float)t.total_tiles * (block == CW * 32 ? 1.f : 2.f) / ((float)longest * cus));
  const float whole = (small ? 0.85f : 1.f) * longest * kWholeTile * (0.75f + 0.25f * busy) + kChange * rounds;
  const float tiles = (float)t.total_tiles / shares;
  const float cut = tiles * kTile + kChange * (1.f + items_crossed(t, tiles)) + 9.f + moved / 12e6f;
  return cut < 0.9f * whole ? shares : 0;
}

int64_t bwd_dq_parts_bytes(int B, int H, int N, int D, bool causal) {
  if (D == 64) return 8 * dq_shares<64>(N, B * H, causal) * kDqSlotFloats<64, kDqCutWaves<64>>;
  if (D == 128) return 8 * dq_shares<128>(N, B * H, causal) * kDqSlotFloats<128, kDqCutWaves<128>>;
  return 8 * dq_shares<256>(N, B * H, causal) * kDqSlotFloats<256, kDqCutWaves<256>>;
}

template <int D, bool CAUSAL>
static hipError_t launch_dq_cut(BwdParams p, int shares, hipStream_t stream) {
  constexpr int NWAVES = kDqCutWaves<D>, BN = kDqBlockN<D>;
  using Cfg = DqCfg<D, NWAVES, BN>;
  auto kern = rope_attn_bwd_dq_kernel<D, NWAVES, BN, CAUSAL, true, true>;
  static std::atomic<uint64_t> lds_ok{0};
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes, lds_ok); e != hipSuccess) return e;
  p.num_blocks = (p.N + Cfg::kBlockM - 1) / Cfg::kBlockM;
#ifdef COROPE_TRACE
  p.trace = nullptr;
#endif
  hipLaunchKernelGGL(kern, dim3(shares), dim3(Cfg::kThreads), Cfg::kLdsBytes, stream, p);
  hipLaunchKernelGGL((rope_attn_bwd_dq_sum_kernel<D, NWAVES, BN, CAUSAL>), dim3((unsigned)p.num_blocks * p.BH * NWAVES), dim3(D / 16 * kWave), 0,
                     stream, p, shares);
  return hipGetLastError();
}

template <int D, bool CAUSAL, bool PREROT>
static hipError_t launch_dq_cfg(const BwdParams& p, hipStream_t stream) {
  if constexpr (PREROT)
    if (p.dq_parts != nullptr)
      if (const int shares = dq_shares<D>(p.N, p.BH, CAUSAL); shares > 0) return launch_dq_cut<D, CAUSAL>(p, shares, stream);
  if constexpr (D > 128) {
    return launch_dq_waves<D, CAUSAL, PREROT, 4>(p, stream);   // 4 waves x 512 registers
  } else {
    return use_small_tiles(p.N, p.BH, DqCfg<D, 4, 64>::kLdsBytes) ? launch_dq_waves<D, CAUSAL, PREROT, 4>(p, stream)
                                      : launch_dq_waves<D, CAUSAL, PREROT, 8>(p, stream);
  }
}

// Dispatch on the run-time switches (head dim, causal, pre-rotated operands present).
template <bool DO_DV, bool DO_DK>
static hipError_t launch_dkdv(const BwdParams& p, int D, bool causal, hipStream_t stream) {
  const bool pre = p.q_rot != nullptr && p.k_rot != nullptr;
#define COROPE_DKDV(DD, CC, PP) launch_dkdv_cfg<DD, CC, DO_DV, DO_DK, PP>(p, stream)
  if (D == 256) {   // separate dV and dK only: both in one launch is built for rotated copies alone (launch_bwd_dkdv_fused)
    if (DO_DV && DO_DK) return hipErrorInvalidValue;
    if constexpr (!(DO_DV && DO_DK)) {
      if (pre) return causal ? COROPE_DKDV(256, true, true) : COROPE_DKDV(256, false, true);
      return causal ? COROPE_DKDV(256, true, false) : COROPE_DKDV(256, false, false);
    }
  }
  if (D == 128) {
    if (pre) return causal ? COROPE_DKDV(128, true, true) : COROPE_DKDV(128, false, true);
    return causal ? COROPE_DKDV(128, true, false) : COROPE_DKDV(128, false, false);
  }
  if (D != 64) return hipErrorInvalidValue;
  if (pre) return causal ? COROPE_DKDV(64, true, true) : COROPE_DKDV(64, false, true);
  return causal ? COROPE_DKDV(64, true, false) : COROPE_DKDV(64, false, false);
#undef COROPE_DKDV
}

hipError_t launch_bwd_dkdv_fused(const BwdParams& p, int D, bool causal, hipStream_t stream) {
  if (D == 256) {
    if (p.q_rot != nullptr && p.k_rot != nullptr)   // on rotated copies: fused, both sets of accumulators in the accumulation registers
      return causal ? launch_dkdv_cfg<256, true, true, true, true>(p, stream) : launch_dkdv_cfg<256, false, true, true, true>(p, stream);
    if (hipError_t e = launch_dkdv<true, false>(p, D, causal, stream); e != hipSuccess) return e;
    return launch_dkdv<false, true>(p, D, causal, stream);
  }
  return launch_dkdv<true, true>(p, D, causal, stream);
}

hipError_t launch_bwd_dv(const BwdParams& p, int D, bool causal, hipStream_t stream) {
  return launch_dkdv<true, false>(p, D, causal, stream);
}

hipError_t launch_bwd_dk(const BwdParams& p, int D, bool causal, hipStream_t stream) {
  return launch_dkdv<false, true>(p, D, causal, stream);
}

hipError_t launch_bwd_dq(const BwdParams& p, int D, bool causal, hipStream_t stream) {
  const bool pre = p.q_rot != nullptr && p.k_rot != nullptr;
  if (D == 256) {
    if (pre) return causal ? launch_dq_cfg<256, true, true>(p, stream) : launch_dq_cfg<256, false, true>(p, stream);
    return causal ? launch_dq_cfg<256, true, false>(p, stream) : launch_dq_cfg<256, false, false>(p, stream);
  }
  if (D == 128) {
    if (pre) return causal ? launch_dq_cfg<128, true, true>(p, stream) : launch_dq_cfg<128, false, true>(p, stream);
    return causal ? launch_dq_cfg<128, true, false>(p, stream) : launch_dq_cfg<128, false, false>(p, stream);
  }
  if (D != 64) return hipErrorInvalidValue;
  if (pre) return causal ? launch_dq_cfg<64, true, true>(p, stream) : launch_dq_cfg<64, false, true>(p, stream);
  return causal ? launch_dq_cfg<64, true, false>(p, stream) : launch_dq_cfg<64, false, false>(p, stream);
}

}  // namespace COROPE_NS
