// Co-RoPE grouped-query attention forward for gfx950 (causal).
//
// Device counterpart of the reference's _corope_fwd_backbone
// (corope-exp/flash_attn_co_rope_gqa_triton.py:48-400); the definition it must reproduce is
// corope-exp/corope_attn_gqa_pytorch.py:16-134.
//
//   z[i,j]     = sigmoid(s * q_leader[i] . k[j])                      (leader = first query head of the group)
//   delta[i,j] = sum_{j < t <= i} z[i,t]                              (the reference's a[i,i] - a[i,j])
//   score[i,j] = s * sum_d ( (q1 k1 + q2 k2) cos(delta w_d) - (q2 k1 - q1 k2) sin(delta w_d) )
//              = s * q[i] . R(delta[i,j]) k[j]      with R rotating each (k1, k2) pair by -delta w_d
//
// Four restatements keep the work down.  (1) delta is a suffix sum that starts at the diagonal, so key chunks are
// swept right to left and delta accumulates directly: the reference's extra pass over all keys (:103-135) and the
// cancellation in a[i,i] - a[i,j] disappear (online softmax does not care about chunk order).  (2) The angle is
// shared by the whole group, so the key is rotated once per (i, j, d).
// (3) Everything that is a dot product with a key or value row runs on the matrix cores: the leader logits q_leader K^T (bf16 x
// bf16: exact products), the scores q^h Kt^T and O^T += V^T P^T.  The rotated keys are rounded to fp16, not bf16, and the score
// product runs in fp16 (the bf16 queries convert exactly): 11 significant bits keep the scores as accurate as the bf16 rounding of P
// afterwards, also at sm_scale = 1 where a bf16 key would cost several percent of a weight.  (4) The pairs that turn slowly are not rotated
// per key at all: over a chunk of 64 keys their rotation is a short polynomial in delta (common.hpp, "Co-RoPE's slow pairs"), so their
// scores are four to seven products with the unrotated keys for all rows at once, and sines and cosines are taken per (row, head, pair)
// and chunk.  With theta = 10000 those are half of the pairs (LOW groups of 16).
//
// Mapping: a wave owns R query rows of one (batch, kv head) group; four waves share a workgroup and the K and V tiles of 64 keys
// it stages in LDS, sweeping from the diagonal to key 0.  Everything is laid out for 16x16x32 MFMAs with the R x G (row, head)
// pairs as the 16 columns:
//   logits   A = leaders (row m of A is the leader of query row m R / 16), B = keys: lane (key % 16, row group) finds the logits
//            of its own rows in its own registers; gates and their suffix sums run along the 16 lanes of a DPP row and then over the
//            four 16-key blocks in registers; delta crosses the lanes once, through LDS.
//   rotation lane (key % 16, g) holds four columns of every 16 of its key and their partners (eight of every 32 where every pair is
//            rotated), exactly as the A operand of the score product wants them: the rotated keys never leave the registers.  Keys are
//            unpacked once for all R rows.
//   scores   S^T = Kt Q^T per row: all 16 columns are multiplied, the row's own G are taken over.  The accumulators of the R rows
//            together are one full tile: lane = (row, head), registers = 16 keys of the chunk, so the softmax has no idle lane and its
//            row statistics are one register per lane.
//   O^T += V^T P^T  for all R rows at once; P is the B operand as the scores left it (the keys of a contraction step in accumulator
//            order, V read transposed in the same order).
// What bounds it: the vector units, for the pairs that are rotated 9 or 10 issue slots per (row, key, pair) -- one multiply, a range
// reduction where the phase can leave the sine unit's domain (REDUCED: in that many groups of 16 pairs), sine and cosine at two slots each, two
// multiplies, two multiply-adds that round to fp16 -- and about 760 per chunk, wave and 16 columns for everything else, of which the slow
// pairs take 350 where rotating them took 1220 with four rows per wave.
// Measured, every pair rotated -> slow pairs as polynomials, the rows of a wave unrolled and the workgroups of a short launch dealt in turn:
// B2 Hq32 Hkv8 N4096 D128 3.20 -> 2.23 ms (2.32 before the rows were unrolled), fp16 B1 Hq32 Hkv8 N1111 D128 143 -> 103 us, B2 Hq8 Hkv8 N3500 D64 1219 -> 780 us.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace COROPE_NS {

struct CoropeFreqs {
  alignas(16) float w[64];  // inverse frequencies divided by 2*pi (revolutions per unit of delta), D/2 entries used
};

constexpr int kCoropeWaves = 4, kCoropeKeys = 64;

template <int D, int R>
struct CoropeFwdCfg {
  static constexpr int kKStride = D + 8;    // K tile rows: 16 keys read at one column hit 16 different bank groups
  static constexpr int kVStride = D + 16;   // V tile rows: the 4 rows x 32 bytes of a transposing read cover 32 banks once
  static constexpr int kTileElems = kCoropeKeys * (kKStride + kVStride);
  static constexpr int kMids = 4 * R * 16, kDeltaFloats = kMids + (R + 3) / 4 * 4;   // per wave: [16-key block][row][key % 16], [row] the chunk's middle
  static constexpr int kLdsBytes = 2 * kTileElems * 2 + kCoropeWaves * kDeltaFloats * 4;
  static_assert(2 * kLdsBytes <= 160 * 1024, "two workgroups per compute unit");
};

// (At D = 64 the registers allow more than two waves per SIMD: with several rows per wave that is 4 % faster, B2 Hq16 Hkv16 N2688
// 1458 -> 1397 us; with one, where the longest rows set the time, 7 % slower, B1 Hq2 Hkv1 N4096 173 -> 185 us.)
template <int D, int G, int R, int REDUCED, int LOW>
__global__ __launch_bounds__(kCoropeWaves* kWave) __attribute__((amdgpu_waves_per_eu(2, R == 1 ? 2 : 8))) void corope_gqa_fwd_kernel(CoropeParams p,
                                                                                                       CoropeFreqs fr) {
  using Cfg = CoropeFwdCfg<D, R>;
  constexpr int KS = Cfg::kKStride, VS = Cfg::kVStride, NT = kCoropeWaves * kWave, PIECES = D / 8;
  constexpr int NG = D / 32, NH = NG - LOW, NOB = D / 16, PER = kCoropeKeys * PIECES / NT;   // groups of 16 rotation pairs, those rotated per key
  constexpr int ZR = R > 4 ? R / 4 : 1;     // query rows whose gates a lane holds
  static_assert(R * G <= 16 && 64 % (kCoropeWaves * R) == 0, "columns of a product; a workgroup's rows lie in one chunk");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int n = lane % 16, g = lane / 16;   // matrix-core identity: A row / B column, contraction group
  uint16_t* const tiles = reinterpret_cast<uint16_t*>(smem);
  float* const dbuf = reinterpret_cast<float*>(smem + 2 * Cfg::kTileElems * 2) + wave * Cfg::kDeltaFloats;

  const int n_groups = p.B * p.Hkv;
  // Longest rows first; where the workgroups that start beside those (two fit a compute unit) are its last ones they run the other way
  // round, so that the compute units end up with equal work (launch_corope_rows).
  int item = blockIdx.x;
  if (item >= p.turn_from && item < p.turn_to) item = p.turn_to - 8 - ((item - p.turn_from) & ~7) + (item & 7);
  const int grp = item % n_groups;
  const int i0 = (p.num_m_blocks - 1 - item / n_groups) * (kCoropeWaves * R);
  const int N = p.N, iw = i0 + wave * R;
  const int head0 = (grp / p.Hkv) * p.Hq + (grp % p.Hkv) * G;
  const uint16_t* kbase = p.k + (int64_t)grp * N * D;
  const uint16_t* vbase = p.v + (int64_t)grp * N * D;
  const int n_chunks = i0 / kCoropeKeys + 1;

  // column n of the score product: (query row, head) = (iw + n / G, n % G); columns from R G on are idle
  const int crow = n < R * G ? n / G : 0, chead = n < R * G ? n % G : 0;
  // An operand holds 32 columns, 8 a lane.  With slow groups operand u is the 16 pairs 16 u .. + 15: lane g holds four columns of the first
  // half, then their partners.  Without, operands come in twos, 8 columns of the first half and 8 of the second (one load of 16 bytes each).
  constexpr int P = LOW > 0 ? 4 : 8;        // pairs per lane and unit of one or two operands
  auto first_col = [&](int unit) __attribute__((always_inline)) { return 4 * P * unit + P * g; };
  auto operands_of = [&](auto& out, const uint16_t* row, int u0) __attribute__((always_inline)) {
    constexpr int COUNT = sizeof(out) / sizeof(out[0]);
#pragma unroll
    for (int u = 0; u < COUNT; u += P / 4) {
      const uint16_t* at = row + first_col((u0 + u) / (P / 4));
      if constexpr (LOW > 0) {
        const u32x2 a = *reinterpret_cast<const u32x2*>(at), b = *reinterpret_cast<const u32x2*>(at + D / 2);
        out[u] = u32x4{a[0], a[1], b[0], b[1]};
      } else {
        out[u] = *reinterpret_cast<const u32x4*>(at);
        out[u + 1] = *reinterpret_cast<const u32x4*>(at + D / 2);
      }
    }
  };
  u32x4 qop[NG], lop[NG];   // B operand of the score product (fp16; the low groups' as they are), A operand of the logit product (element type)
  {
    const uint16_t* qrow = p.q + ((int64_t)(head0 + chead) * N + min(iw + crow, N - 1)) * D;
    const uint16_t* lrow = p.q + ((int64_t)head0 * N + min(iw + n * R / 16, N - 1)) * D;
    operands_of(qop, qrow, 0);
    operands_of(lop, lrow, 0);
#pragma unroll
    for (int u = 0; u < NG; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) qop[u][e] = n >= R * G ? 0u : u < NH ? pack_f16(elt_lo(qop[u][e]), elt_hi(qop[u][e])) : qop[u][e];
  }
  float turns[NG * 4 / P][P];  // w_d / 2 pi of this lane's columns
#pragma unroll
  for (int u = 0; u < NG * 4 / P; ++u)
#pragma unroll
    for (int e = 0; e < P; e += 4) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(fr.w + first_col(u) + e);
#pragma unroll
      for (int x = 0; x < 4; ++x) turns[u][e + x] = t[x];
    }

#pragma unroll
  for (int u = 0; u < NG * 4 / P; ++u)
#pragma unroll
    for (int e = 0; e < P; ++e) asm volatile("" ::"v"(turns[u][e]));   // landed before the loop: left to their first use, the wait sits in it

  // K and V of a chunk: global memory -> registers one chunk ahead -> the other LDS stage
  u32x4 kst[PER], vst[PER];
  auto fetch = [&](int c, auto may_run_past_end) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = threadIdx.x + u * NT;
      int row = c * kCoropeKeys + e / PIECES;
      if (decltype(may_run_past_end)::value) row = min(row, N - 1);   // only the chunk on the diagonal can
      const uint32_t off = (uint32_t)row * (D * 2) + (e % PIECES) * 16;
      kst[u] = *reinterpret_cast<const u32x4*>(byte_offset(kbase, off));
      vst[u] = *reinterpret_cast<const u32x4*>(byte_offset(vbase, off));
    }
  };
  auto park = [&](int buf) __attribute__((always_inline)) {
    uint16_t* kt = tiles + buf * Cfg::kTileElems;
    uint16_t* vt = kt + kCoropeKeys * KS;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = threadIdx.x + u * NT;
      *reinterpret_cast<u32x4*>(kt + (e / PIECES) * KS + 8 * (e % PIECES)) = kst[u];
      *reinterpret_cast<u32x4*>(vt + (e / PIECES) * VS + 8 * (e % PIECES)) = vst[u];
    }
  };

  f32x4 oacc[NOB];            // O^T: column n, d = 16 db + 4 g + e
#pragma unroll
  for (int db = 0; db < NOB; ++db) oacc[db] = f32x4{0, 0, 0, 0};
  // reference value of the exponentials of this lane's column (base-2 units; far below every score until the first chunk) and
  // this lane's share of its denominator
  float m_run = -1e30f, l_run = 0.f;
  float carry[ZR];            // sum of the gates to the right of the chunk
#pragma unroll
  for (int z = 0; z < ZR; ++z) carry[z] = 0.f;

  fetch(n_chunks - 1, std::true_type{});
  float scale2 = p.sm_scale * 1.4426950408889634f;   // scores in the base-2 domain, of this lane's column
  if constexpr (LOW > 0 && kEltIsF16) scale2 *= corope_scaled_query(qop);   // (waits for the query under the first tiles' requests)
  park(0);
  __syncthreads();
  int buf = 0;
#pragma unroll 1
  for (int c = n_chunks - 1; c >= 0; --c) {
    if (LOW == 0 && c > 0) fetch(c - 1, std::false_type{});
    const uint16_t* kt = tiles + buf * Cfg::kTileElems;
    const uint16_t* vt = kt + kCoropeKeys * KS;
    const bool diagonal = c == n_chunks - 1;   // wave-uniform

    // ---- leader logits, gates, delta: lane (key 16 b + n, query rows (4 g + e) R / 16) -------------------------------------
    {
      f32x4 lg[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        lg[b] = f32x4{0, 0, 0, 0};
        u32x4 kf[NG];
        operands_of(kf, kt + (16 * b + n) * KS, 0);
#pragma unroll
        for (int u = 0; u < NG; ++u) lg[b] = mfma16(lop[u], kf[u], lg[b]);
      }
#pragma unroll
      for (int z = 0; z < ZR; ++z) {
        const int r = R > 4 ? g * ZR + z : 4 * g * R / 16;
        float pre[4], tot[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          float x = sigmoid(lg[b][z * (4 / ZR)] * p.sm_scale);
          if (diagonal && c * kCoropeKeys + 16 * b + n > iw + r) x = 0.f;   // gates beyond the diagonal do not count
          pre[b] = row16_prefix_sum(x);
          tot[b] = row16_last(pre[b]);
        }
        float right = carry[z];
#pragma unroll
        for (int b = 3; b >= 0; --b) {
          dbuf[(b * R + r) * 16 + n] = right + (tot[b] - pre[b]);   // gates strictly to the right of the key, up to the diagonal
          right += tot[b];
        }
        if constexpr (LOW > 0) dbuf[Cfg::kMids + r] = 0.5f * (carry[z] + right);
        carry[z] = right;
      }
    }
    lds_order();

    // ---- scores, the slow pairs: a polynomial in delta ---------------------------------------------------------------------
    f32x4 sacc[4];
    if constexpr (LOW > 0) {
      CoropeLowOps<LOW> ops;
      ops.build(qop + NH, turns + NH, dbuf[Cfg::kMids + crow]);
      const float mid = dbuf[Cfg::kMids + crow];
      constexpr int NB = 2;   // blocks at a time (with all four the kernel spills at D = 128)
#pragma unroll
      for (int b0 = 0; b0 < 4; b0 += NB) {
        f32x4 y[NB], s[NB];
        u32x4 kf[NB][LOW];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          y[b] = *reinterpret_cast<const f32x4*>(dbuf + ((b0 + b) * R + crow) * 16 + 4 * g);
#pragma unroll
          for (int e = 0; e < 4; ++e) y[b][e] = (y[b][e] - mid) * (1.f / kCoropeReach);
          operands_of(kf[b], kt + (16 * (b0 + b) + n) * KS, NH);
        }
        ops.scores(kf, y, s);
#pragma unroll
        for (int b = 0; b < NB; ++b) sacc[b0 + b] = s[b];
      }
      if (c > 0) fetch(c - 1, std::false_type{});   // (behind the polynomial, which needs the registers)
    } else {
#pragma unroll
      for (int b = 0; b < 4; ++b) sacc[b] = f32x4{0, 0, 0, 0};
    }

    // ---- the others: rotated keys, 16 keys at a time ---------------------------------------------------------------------
    static_for<4>([&](auto b_c) __attribute__((always_inline)) {
      constexpr int b = decltype(b_c)::value;
      constexpr int UNITS = NH * 4 / P;
      float k1[UNITS][P], k2[UNITS][P];
      u32x4 kf[NH];
      operands_of(kf, kt + (16 * b + n) * KS, 0);
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
#pragma unroll
        for (int e = 0; e < P / 2; ++e) {
          const uint32_t w1 = P == 4 ? kf[u][e] : kf[2 * u % NH][e], w2 = P == 4 ? kf[u][2 + e % 2] : kf[(2 * u + 1) % NH][e];
          k1[u][2 * e] = elt_lo(w1);
          k1[u][2 * e + 1] = elt_hi(w1);
          k2[u][2 * e] = elt_lo(w2);
          k2[u][2 * e + 1] = elt_hi(w2);
        }
      const f32x4 low = sacc[b];
      // The rows are unrolled, which hides a row's chain behind the next row's: bf16 B2 Hq32 Hkv8 N4096 D128 2.32 -> 2.23 ms.  fp16 at D = 128 has no registers
      // for that (84 to 134 of them went through scratch): with eight rows the scheduler is kept from mixing them, and where every pair is
      // rotated they stay a loop.  All unrolled -> this, us: N4096 Hq32 Hkv32 5523 -> 3674 and Hkv16 2787 -> 1865; theta = 1000 (every pair
      // rotated) Hkv32 6815 -> 5770, Hkv8 1740 -> 1557, Hkv4 902 -> 880.
      constexpr bool kRowByRow = kEltIsF16 && D == 128 && LOW > 0 && R == 8, kLoop = kEltIsF16 && D == 128 && LOW == 0;
      constexpr int kUnroll = kLoop ? 1 : R;
      float delta[kLoop ? 1 : R];   // (in the loop: of the next row)
#pragma unroll
      for (int r = 0; r < (kLoop ? 1 : R); ++r) delta[r] = dbuf[(b * R + r) * 16 + n];
#pragma unroll kUnroll
      for (int r = 0; r < R; ++r) {
        const float delta_r = delta[kLoop ? 0 : r];
        if constexpr (kLoop) delta[0] = dbuf[(b * R + min(r + 1, R - 1)) * 16 + n];
        f32x4 acc = low;
        static_for<UNITS>([&](auto u_c) __attribute__((always_inline)) {
          constexpr int u = decltype(u_c)::value;
          _Float16 y[2 * P];
#pragma unroll
          for (int e = 0; e < P; ++e) {
            const float x = corope_phase<(P / 4 * u < REDUCED)>(delta_r * turns[u][e]);
            const float sn = __builtin_amdgcn_sinf(x), cs = __builtin_amdgcn_cosf(x);
            y[e] = (_Float16)__builtin_fmaf(cs, k1[u][e], sn * k2[u][e]);
            y[P + e] = (_Float16)__builtin_fmaf(cs, k2[u][e], -(sn * k1[u][e]));
          }
#pragma unroll
          for (int t = 0; t < P / 4; ++t) {
            f16x8 op;
#pragma unroll
            for (int e = 0; e < 8; ++e) op[e] = y[8 * t + e];
            acc = mfma16_f16(__builtin_bit_cast(u32x4, op), qop[P / 4 * u + t], acc);
          }
        });
#pragma unroll
        for (int e = 0; e < 4; ++e) sacc[b][e] = crow == r ? acc[e] : sacc[b][e];
        if constexpr (kRowByRow) __builtin_amdgcn_sched_barrier(0);
      }
    });

    // ---- softmax: lane = (row, head), 16 keys 16 b + 4 g + e of the chunk ------------------------------------------------
    // Keys beyond the diagonal are masked behind the scaling: sm_scale may be zero or negative.
    auto mask = [&](float (&y)[4][4]) __attribute__((always_inline)) {
      if (!diagonal) return;
      const int rel = iw + crow - c * kCoropeKeys - 4 * g;   // last key the row sees, relative to this lane's first
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (16 * b + e > rel) y[b][e] = -INFINITY;
    };
    // The reference value only has to keep the exponentials in range, it need not be the running maximum: it moves (to the exact
    // maximum so far, with the usual rescaling) only when some score of the chunk lies more than kLazyMargin above it, which after
    // the first chunks of a row is rare.  On the diagonal, a row's first chunk, it always does, so only that branch masks.
    constexpr float kLazyMargin = 8.f;   // base-2 units: weights stay below 2^8
    float x[4][4], top = -INFINITY;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[b][e] = __builtin_fmaf(sacc[b][e], scale2, -m_run);
        top = fmaxf(top, x[b][e]);
      }
    if (diagonal || __builtin_amdgcn_ballot_w64(top > kLazyMargin) != 0) {   // wave-uniform
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[b][e] = sacc[b][e] * scale2;
      mask(x);
      top = -INFINITY;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) top = fmaxf(top, x[b][e]);
      top = fmaxf(top, __shfl_xor(top, 16));
      top = fmaxf(top, __shfl_xor(top, 32));
      const float m_new = fmaxf(m_run, top);   // finite: the chunk holds a key <= row
      const float al = fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= al;
#pragma unroll
      for (int db = 0; db < NOB; ++db)
#pragma unroll
        for (int e = 0; e < 4; ++e) oacc[db][e] *= al;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[b][e] = __builtin_fmaf(sacc[b][e], scale2, -m_run);
      mask(x);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {   // 32 keys per product
      float w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        w[j] = fast_exp2(x[2 * t + j / 4][j % 4]);   // 0 for the keys beyond the diagonal
        l_run += w[j];
      }
      const u32x4 bop = {pack_elts(w[0], w[1]), pack_elts(w[2], w[3]), pack_elts(w[4], w[5]), pack_elts(w[6], w[7])};
#pragma unroll
      for (int db = 0; db < NOB; ++db) oacc[db] = mfma16(load_a_trans16_acc(vt, VS, 32 * t, 16 * db), bop, oacc[db]);
    }
    if (c > 0) park(buf ^ 1);
    buf ^= 1;
    __syncthreads();
  }

  float l = l_run + __shfl_xor(l_run, 16);
  l += __shfl_xor(l, 32);
  const float inv_l = l > 0.f ? 1.f / l : 0.f;   // same guard as the reference's epilogue (:343-345)
  if (n < R * G && iw + crow < N) {
    uint16_t* op = p.o + ((int64_t)(head0 + chead) * N + iw + crow) * D;
#pragma unroll
    for (int db = 0; db < NOB; ++db) {
      const u32x2 w = {pack_elts(oacc[db][0] * inv_l, oacc[db][1] * inv_l), pack_elts(oacc[db][2] * inv_l, oacc[db][3] * inv_l)};
      *reinterpret_cast<u32x2*>(op + db * 16 + 4 * g) = w;
    }
  }
}

template <int D, int G, int R, int REDUCED, int LOW>
static hipError_t launch_corope_rows(CoropeParams p, const CoropeFreqs& fr, hipStream_t stream) {
  using Cfg = CoropeFwdCfg<D, R>;
  auto kern = corope_gqa_fwd_kernel<D, G, R, REDUCED, LOW>;
  static std::atomic<uint64_t> lds_ok{0};
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes, lds_ok); e != hipSuccess) return e;
  p.num_m_blocks = (p.N + kCoropeWaves * R - 1) / (kCoropeWaves * R);
  const int64_t items = (int64_t)p.num_m_blocks * p.B * p.Hkv, cus = device_cu_count() & ~7;
  // Workgroups i and i + cus start on the same compute unit: the second of them takes the items from the other end, so that the two
  // are equal work together.  (In whole rounds of the eight XCDs.)  Four rows per wave, longest first -> in turn: fp16 B1 Hq32 Hkv8 N1111 D128 124 -> 115 us, B1 Hq8
  // Hkv2 N4096 D128 431 -> 404, B1 Hq32 Hkv8 N1300 D64 93 -> 77; from four workgroups per compute unit on no difference.  With one row per wave the items
  // that start last are short and longest first evens out by itself: B2 Hq8 Hkv4 N300 D64 13.3 us against 13.7 in turn.
  const bool turn = R > 1 ? items < 4 * cus : 4 * items <= 9 * cus;
  p.turn_from = turn ? (int)cus : 0;
  p.turn_to = turn ? (int)std::min<int64_t>(items & ~7, 2 * cus) : 0;
  hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(kCoropeWaves * kWave), Cfg::kLdsBytes, stream, p, fr);
  return hipGetLastError();
}

// reduced: leading groups of 16 pairs whose phase has to be reduced (a template argument, rounded up to one that is built); low: trailing
// groups that may go through the polynomial.
template <int D, int G, int R, int LOW>
static hipError_t launch_corope_reduced(const CoropeParams& p, const CoropeFreqs& fr, int reduced, hipStream_t stream) {
  if (reduced == 0) return launch_corope_rows<D, G, R, 0, LOW>(p, fr, stream);
  if constexpr (LOW > 0) {
    constexpr int NH = D / 32 - LOW;
    if (NH == 1 || reduced == 1) return launch_corope_rows<D, G, R, 1, LOW>(p, fr, stream);
    return launch_corope_rows<D, G, R, NH, LOW>(p, fr, stream);
  } else {
    if (D == 64 || reduced <= 2) return launch_corope_rows<D, G, R, 2, LOW>(p, fr, stream);
    return launch_corope_rows<D, G, R, D / 32, LOW>(p, fr, stream);
  }
}

template <int D, int G>
static hipError_t launch_corope_cfg(const CoropeParams& p, const CoropeFreqs& fr, int reduced, int low, hipStream_t stream) {
  // Rows per wave: as many as fill the 16 columns, where the waves then still fill the chip; below that the longest rows, whose chunks
  // follow one after the other, set the time, and fewer rows per wave shorten it.
  // The slow pairs' products cost the same for one row as for all: they pay from two rows per wave on, and make more rows pay earlier.
  // Whether they are used depends on the rows of one batch entry, so that an entry's scores are computed the same way whatever it is batched with (its
  // bits may still differ: the rows of a wave, which depend on the whole batch, move their reference values together).  From `least` on, two rows
  // per wave are no slower than one with every pair rotated; at D = 128 an entry alone needs 3.375 rows a SIMD for that, where the launch of
  // one row per wave has just begun another round: us, every pair rotated / products, B1 Hq4 Hkv1 N3200 191 / 206, N3400 215 / 222, N3600 241 / 234; B2 Hq8 Hkv2 N1600
  // (3200 rows an entry) 183 / 139.
  // us with one (every pair rotated) / two / four rows, B1 Hq32 Hkv8, D = 64: N256 9.8 / 13.8 / 16.7, N512 26.5 / 24.9 / 29.8, N700 46 / 35 / 40, N900 73 / 54 / 53, N1024
  // 106 / 65 / 57; D = 128: N256 15.4 / 19.9 / 26.6, N400 34.5 / 33.0 / 43.0, N700 79 / 60 / 66, N900 126 / 92 / 87, N1300 273 / 175 / 139.  Every pair
  // rotated: fp16 B1 Hq32 Hkv8 N1111 D128 179 / 143 / 171, B2 Hq16 Hkv4 N2048 D128 582 / 466 / 418.
  constexpr int kMost = G <= 2 ? 8 : G <= 4 ? 4 : 2, kLow = D / 64;
  const int64_t rows = (int64_t)p.N * p.B * p.Hkv, simds = 4 * device_cu_count(), least = (D == 64 ? 4 : 3) * simds;
  if (low >= kLow && (int64_t)p.N * p.Hkv >= least && rows >= (D == 64 ? least : least + 3 * simds / 8)) {
    if constexpr (kMost > 4) {
      if (rows >= 14 * simds) return launch_corope_reduced<D, G, kMost, kLow>(p, fr, reduced, stream);
    }
    if constexpr (kMost > 2) {
      if (rows >= 7 * simds) return launch_corope_reduced<D, G, 4, kLow>(p, fr, reduced, stream);
    }
    return launch_corope_reduced<D, G, 2, kLow>(p, fr, reduced, stream);
  }
  if (rows >= 4 * simds * kMost) return launch_corope_reduced<D, G, kMost, 0>(p, fr, reduced, stream);
  if (kMost > 2 && rows >= 8 * simds) return launch_corope_reduced<D, G, 2, 0>(p, fr, reduced, stream);
  return launch_corope_reduced<D, G, 1, 0>(p, fr, reduced, stream);
}

template <int D>
static hipError_t launch_corope_d(const CoropeParams& p, const CoropeFreqs& fr, hipStream_t stream) {
  const int reduced = corope_reduced_groups(fr.w, D, p.N), low = corope_low_groups(fr.w, D);
  switch (p.Hq / p.Hkv) {
    case 1: return launch_corope_cfg<D, 1>(p, fr, reduced, low, stream);
    case 2: return launch_corope_cfg<D, 2>(p, fr, reduced, low, stream);
    case 3: return launch_corope_cfg<D, 3>(p, fr, reduced, low, stream);
    case 4: return launch_corope_cfg<D, 4>(p, fr, reduced, low, stream);
    case 5: return launch_corope_cfg<D, 5>(p, fr, reduced, low, stream);
    case 6: return launch_corope_cfg<D, 6>(p, fr, reduced, low, stream);
    case 7: return launch_corope_cfg<D, 7>(p, fr, reduced, low, stream);
    case 8: return launch_corope_cfg<D, 8>(p, fr, reduced, low, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_corope_gqa_fwd(const CoropeParams& p, int D, hipStream_t stream) {
  CoropeFreqs fr{};
  // theta^(-2d/D) evaluated like the reference's torch expression (fp32 exponent, fp32 power), then / 2 pi
  for (int d = 0; d < D / 2; ++d) {
    float e = (float)(2 * d) / (float)D;
    float inv = 1.0f / powf(p.theta, e);
    fr.w[d] = (float)((double)inv / 6.283185307179586);
  }
  return D == 64 ? launch_corope_d<64>(p, fr, stream) : launch_corope_d<128>(p, fr, stream);
}

}  // namespace COROPE_NS
