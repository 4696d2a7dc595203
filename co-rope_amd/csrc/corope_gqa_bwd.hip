// Co-RoPE grouped-query attention backward for gfx950.
//
// The reference's "fused" Co-RoPE operator falls back to a dense PyTorch backward that materialises (B, Hq, N, N, D/2)
// temporaries (corope-exp/flash_attn_co_rope_gqa_triton.py:459-577; same mathematics as the manual backward of
// corope-exp/corope_attn_gqa_pytorch.py:137-300).  This file computes the same gradients with O(N^2) scalars per head
// in a caller-supplied workspace (packed lower-triangular matrices) and no D-sized temporaries.
//
// Mathematics (group = the Hq/Hkv query heads sharing one key/value head; leader = first head of the group;
// c = sm_scale; w_d = theta^(-2d/D); pairs (d, d + D/2) as in the forward):
//   z_it    = sigmoid(c qL_i . k_t)                      delta_ij = sum_{j < t <= i} z_it
//   S^h_ij  = c sum_d [ q1 (k1 cos phi + k2 sin phi) + q2 (k2 cos phi - k1 sin phi) ],   phi = delta_ij w_d
//           = c q^h_i . kt_ij  =  c k_j . qt^h_ij       (kt, qt: the key / the query rotated by -/+ phi)
//   P = softmax_j(S),  dP^h_ij = dO^h_i . v_j,  dS = P o (dP - rowsum(P o dP))
//   dv_j    = sum_{h,i} P^h_ij dO^h_i
//   dq^h_i  = c sum_j dS^h_ij kt_ij                      dk_j = c sum_{h,i} dS^h_ij qt^h_ij      (paths with delta fixed)
//   through delta:  g^h_ij = dS/ddelta = c sum_d w_d (q1 kt2 - q2 kt1),   G_ij = sum_h dS^h_ij g^h_ij,
//                   dz_it = sum_{j < t} G_ij,   W_it = dz_it z_it (1 - z_it)   (gradient of the leader's logit),
//                   dqL_i += c sum_t W_it k_t,   dk_t += c sum_i W_it qL_i.
//
// Sines and cosines are evaluated in two places only, once per (i, j, d) each: where the key is rotated (scores kernel)
// and where the dS-weighted sum of the group's queries is rotated (dk kernel) - the angle is shared by the group and
// rotation is linear, so one vector is rotated per (i, j), not one per head.  Everything that is a dot product with an
// already rotated or an unrotated row runs on the matrix cores.  Launches, in order:
//   scores       a wave per R query rows of a group, 16 keys at a time:
//                  right to left: leader logits, z, delta by a scan, the rotated keys Kt in registers (fp16); on the matrix cores
//                  dP = V dO^T, S = Kt q^T and dS/ddelta = Kt [-w q2, w q1]^T for all heads, then - with running softmax
//                  statistics, flash-attention style - the two sums that make dq: sum_j e_j dP_j kt_j and sum_j e_j kt_j;
//                  left to right: dP again, dS, G and its running sum, W;
//                  writes dq of the heads 1..G-1, the leader's dq without its gate path (fp32, workspace), the workspace
//                  matrices DELTA, W [group] and S, DS [head] (packed lower triangles) and the row statistics that make P of S
//   dv           dq_leader = c (partial + W K), 32 rows per workgroup, and beside it dv^T += dO^T P, P from S and the row statistics, 128
//                keys per workgroup: plain products on the matrix cores
//   dk           one workgroup per (group, 128 keys): sum_h dS^h q^h on the matrix cores, then lane = rotation pair x 16
//                keys rotates it per (i, j) and adds the gate path W qL; tiles of DELTA, W, DS staged through LDS
// Rounding: the rotated keys and what multiplies them (queries, the softmax weights e and e dP) are fp16 - the bf16
// queries convert exactly, and 11 significant bits keep scores accurate at sm_scale = 1 too; the products on unrotated
// rows (W K, P dO, the row dots) take bf16 operands; sums, statistics, delta, dS/ddelta and everything stored in the
// workspace are fp32.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace COROPE_NS {

struct CoropeBwdFreqs {
  alignas(16) float turns[64];   // w_d / (2 pi): phase in revolutions per unit of delta (what v_sin_f32 / v_cos_f32 take)
  alignas(16) float rad[64];     // w_d
};

// Row i of a workspace matrix holds the keys j <= i only: rows are packed, each padded to the 64-key chunk it ends in
// (rows 64 c .. 64 c + 63 take 64 (c + 1) floats each), so every row starts on a 256-byte boundary.
__device__ __host__ inline int64_t tri_row_start(int i) {
  const int64_t c = i / 64, r = i % 64;
  return 2048 * c * (c + 1) + 64 * (c + 1) * r;
}

// Workspace layout, in floats; NN = tri_row_start(N) is the size of one packed lower-triangular matrix.
struct CoropeBwdWs {
  float* base;
  int64_t NN;
  int n_groups, n_heads;
  __device__ __host__ float* delta(int g) const { return base + (int64_t)g * NN; }
  __device__ __host__ float* w(int g) const { return base + (int64_t)(n_groups + g) * NN; }
  __device__ __host__ float* s(int h) const { return base + (int64_t)(2 * n_groups + h) * NN; }               // scores, base-2 units
  __device__ __host__ float* ds(int h) const { return base + (int64_t)(2 * n_groups + n_heads + h) * NN; }    // dS/ddelta, then dS
  // What the last n_heads matrices' worth of space holds, per group: the partial sums of dv, then of dk, from the front, and per
  // head and query row, at the end, the reference value of the exponentials and 1 / their sum.
  __device__ __host__ static int padded_rows(int N) { return (N + 15) / 16 * 16; }
  __device__ __host__ int64_t part_floats(int G, int N) const { return G * (NN - 2 * padded_rows(N)); }
  __device__ __host__ float* parts(int g, int G) const { return base + (int64_t)(2 * n_groups + 2 * n_heads + g * G) * NN; }
  __device__ __host__ float* row_max(int g, int G, int N, int h) const { return parts(g, G) + part_floats(G, N) + h * padded_rows(N); }
  __device__ __host__ float* row_inv(int g, int G, int N, int h) const { return row_max(g, G, N, G + h); }
  // (N, D) per group: the leader head's dq without the gate path and without the factor sm_scale
  __device__ __host__ float* dql(int g, int N, int D) const {
    return base + (int64_t)(2 * n_groups + 3 * n_heads) * NN + (int64_t)g * N * D;
  }
};

// ---------------------------------------------------------------------------------------------------- scores
// A wave owns R query rows of one (batch, kv head) group, all G heads at once, and sweeps 16 keys at a time.  The R x G (row, head)
// pairs are columns of 16x16 products: rows 0 .. R/2 - 1 are columns 0 .. 7, the others columns 8 .. 15 (R = 1: columns 0 .. 7).
//   keys     lane (key % 16, g) holds columns 8 g .. 8 g + 7 of every 32 of its key, fetched straight from global memory (a key
//            block is 4 KB, read once for all R rows) and unpacked once; the rotation happens in that layout, row by row.
//   scores   the rotated keys are the A operand as they are.  A row needs its own columns of S = Kt q^T only, and of
//            dS/ddelta = Kt [-w q2, w q1]^T; one product gives both: the B operand of a row of the lower half carries q in columns
//            0 .. 7 and the derivative's rows in columns 8 .. 15, of the upper half the other way round.
//   softmax  lane = (row, head), registers = 4 of the 16 keys: no idle lane, row statistics are one register per lane.
//   dq       needs the rotated keys transposed: they go through LDS (16 keys x D x R rows per wave) and come back through the
//            transposing read.  The weights of the two sums, e (dP - ref) and e, share the 16 columns in the same way (a rotation by 8
//            lanes), and two rows share the 32 contraction slots of a product (the other row's columns of B are zero).
// No barriers: a wave is a workgroup.  What bounds it: in the first sweep the vector units (busy 71 % of both sweeps together; 9 or 10 issue slots per (row, key,
// pair) as in the forward, of about 12 in all), in the second the memory (9 floats in, 5 out per (row, key) at G = 4); two waves a
// SIMD hide one under the other only in part.  dP is computed in both sweeps, and P is left to the dv kernel: kept in the workspace they cost
// 12 floats more per (row, key) and a launch.
// Measured at B2 Hq32 Hkv8 N4096 D128: 8.2 -> 6.1 ms, three quarters of it the first sweep (one wave per row with the rotated keys in LDS, behind launches for the
// logits and dP); B2 Hq8 Hkv2 N512 D64 52 -> 40 us.
template <int D, int G, int R, int REDUCED>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(2))) void corope_bwd_scores_kernel(CoropeBwdParams p, CoropeBwdWs ws,
                                                                                                          CoropeBwdFreqs fr) {
  constexpr int TS = D + 16, HALF = D / 2;   // LDS row stride: the row-wise writes and the transposing reads both spread over the banks
  constexpr int NKS = D / 32, HK = D / 64, NDB = D / 16;
  constexpr int NS = R > 1 ? 2 : 1, RH = R / NS;             // halves of the columns, rows in each
  static_assert(RH * G <= 8 && (R == 1 || R == 2 || R == 4), "eight columns for each half of the rows");
  // [row][key][d]: rotated keys, fp16.  Before they come and after they have been used, a block of 16 rows of K or V on its way from whole
  // cache lines to operand order; second sweep: such a block, and behind it dP [column][key], fp32
  constexpr int BS = D + 8, PS = kWave + 4;   // row strides: block (elements), dP (floats)
  constexpr int kKtElems = R * 16 * TS, kBlockElems = 2 * 16 * BS, kSecondElems = 16 * BS + NS * 8 * PS * 2;
  __shared__ __attribute__((aligned(16))) uint16_t kt[std::max({kKtElems, kBlockElems, kSecondElems})];
  __shared__ __attribute__((aligned(16))) uint16_t lead[R * (D + 8)];  // the leader's rows
  const int lane = threadIdx.x, n = lane % 16, g = lane / 16;
  // longest rows of all groups first: with one group after the other the last group's longest rows started when the chip was
  // already running empty (23 % of the compute units' time idle)
  const int n_groups = p.B * p.Hkv, grp = (int)(blockIdx.x % n_groups);
  const int iw = R * ((int)(gridDim.x / n_groups) - 1 - (int)(blockIdx.x / n_groups));
  const int N = p.N, b_ = grp / p.Hkv, kvh = grp % p.Hkv;
  const int head0 = b_ * p.Hq + kvh * G;   // first head of the group, as a (batch, head) slab index
  const int sub = n % 8;                   // place within a half
  const bool low = n < 8;
  // Idle columns repeat the first one of their half, rows past the end the last row, operands and all: they come to the same values
  // and may store them to the same places.  With no lane switched off around the loops' stores their number is known to the compiler,
  // and a wait for a prefetched load does not wait for the stores behind it.
  const bool busy = sub / G < RH;
  const int place = busy ? sub / G : 0, head = busy ? sub % G : 0;      // this lane's column: row of the half, head
  const int half = NS > 1 ? n / 8 : 0;                                  // (R = 1: the lanes from 8 on hold dS/ddelta only)
  const int own_row = min(iw + half * RH + place, N - 1);
  const float scale2 = p.sm_scale * 1.4426950408889634f;                // scores in the base-2 domain

  // w_d / 2 pi and w_d of this lane's columns d = 32 hk + 8 g + e
  float turns[HK][8], rad[HK][8];
#pragma unroll
  for (int hk = 0; hk < HK; ++hk)
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(fr.turns + 32 * hk + 8 * g + e);
      const f32x4 w = *reinterpret_cast<const f32x4*>(fr.rad + 32 * hk + 8 * g + e);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        turns[hk][e + x] = t[x];
        rad[hk][e + x] = w[x];
      }
    }

  // B operands of the score products (fp16): columns of half s, the derivative's rows in the other half's places
  u32x4 qop[NS][NKS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const bool deriv = n / 8 != s;
    const uint16_t* qrow = p.q + ((int64_t)(head0 + head) * N + min(iw + s * RH + place, N - 1)) * D;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int d0 = 32 * ks + 8 * g;
      const u32x4 raw = *reinterpret_cast<const u32x4*>(qrow + (deriv ? d0 ^ HALF : d0));
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float w = rad[ks % HK][e], qv = e % 2 ? elt_hi(raw[e / 2]) : elt_lo(raw[e / 2]);
        x[e] = (deriv ? (2 * ks < NKS ? -w : w) : 1.f) * qv;   // first half of the columns: -w q2, second: w q1
      }
      qop[s][ks] = u32x4{pack_f16(x[0], x[1]), pack_f16(x[2], x[3]), pack_f16(x[4], x[5]), pack_f16(x[6], x[7])};
    }
  }
  // dq^h = c sum_j dS_j kt_j = c (sum_j e_j dP_j kt_j - Delta sum_j e_j kt_j) / L with e_j = exp(s_j - m): both sums are
  // accumulated on the matrix cores, rescaled flash-attention style when the row's reference value m moves.
  // Reference value for Delta = rowsum(P o dP), which is only known at the end of the row: the dq sums take e (dP - ref)
  // as weights and are corrected by (Delta - ref) afterwards, which is exact for any ref; the closer ref is to Delta, the
  // less the two sums cancel (rows dominated by one key would otherwise lose the 11 bits of the weights).  With the forward
  // output at hand ref = rowsum(O o dO), equal to Delta up to O's rounding; without it ref = 0.
  // The weights e (dP - ref) go to the matrix cores as fp16, whose 5 exponent bits would tie the result to the scale of
  // dO (overflow from |dP - ref| ~ 1e3 on, nothing left of a mean-reduced loss's 1e-7): they are divided by a power of two
  // w_scale >= 4 |dO_i| first (|dP_ij| <= |dO_i| |v_j|, so the scaled weights are at most 2^5 |v_j| / 4 whatever dO is)
  // and the sum is multiplied back afterwards -- exact both ways.
  float dref = 0.f, w_mul, w_inv;
  const uint16_t* const do_l = p.d_o + ((int64_t)(head0 + head) * N + own_row) * D + 8 * g;   // B operand of dP = V dO^T, column n
  {
    float sq = 0.f;
    const int64_t off = ((int64_t)(head0 + head) * N + own_row) * D + 8 * g;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const u32x4 x = *reinterpret_cast<const u32x4*>(do_l + 32 * ks);
      u32x4 y = u32x4{0, 0, 0, 0};
      if (p.o != nullptr) y = *reinterpret_cast<const u32x4*>(p.o + off + 32 * ks);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sq = __builtin_fmaf(elt_lo(x[e]), elt_lo(x[e]), __builtin_fmaf(elt_hi(x[e]), elt_hi(x[e]), sq));
        dref = __builtin_fmaf(elt_lo(x[e]), elt_lo(y[e]), __builtin_fmaf(elt_hi(x[e]), elt_hi(y[e]), dref));
      }
    }
    sq += __shfl_xor(sq, 16);
    sq += __shfl_xor(sq, 32);
    dref += __shfl_xor(dref, 16);
    dref += __shfl_xor(dref, 32);
    int ex = 0;
    (void)frexpf(__builtin_sqrtf(sq), &ex);       // |dO_i| = m 2^ex with m in [0.5, 1); 0 gives ex = 0
    const int w_exp = max(-100, min(100, ex + 2));
    w_mul = ldexpf(1.f, w_exp);
    w_inv = ldexpf(1.f, -w_exp);
  }
  const float ref_scaled = dref * w_inv;

  const uint16_t* kbase = p.k + (int64_t)grp * N * D;
  const uint16_t* vbase = p.v + (int64_t)grp * N * D;
  const int row_len = 64 * (iw / 64 + 1);                    // the rows of a wave lie in one 64-row band: one row length
  const int64_t rows0 = tri_row_start(iw);
  // this lane's places in the matrices: the score of a column; dS/ddelta of the column eight on; gates of key n
  // of query row z_row
  const int z_row = min(iw + g * R / 4, N - 1);
  // (stored by lane (column, keys) = (lane / 4, 4 (lane % 4) ..): four lanes complete a 64-byte piece)
  float *s_l, *g_l;
  const int from = lane / 4 + 16 * (lane % 4);   // the lane that computes what this one stores
  {
    const int c = lane / 4, csub = c % 8, chalf = NS > 1 ? c / 8 : 0;
    const int cplace = csub / G < RH ? csub / G : 0, chead = csub / G < RH ? csub % G : 0;
    const int64_t c_own = rows0 + row_len * (min(iw + chalf * RH + cplace, N - 1) - iw) + 4 * (lane % 4);
    const int64_t c_other = rows0 + row_len * (min(iw + (NS - 1 - chalf) * RH + cplace, N - 1) - iw) + 4 * (lane % 4);
    s_l = (NS == 1 && c >= 8 ? ws.ds(head0 + chead) : ws.s(head0 + chead)) + c_own;
    g_l = ws.ds(head0 + chead) + c_other;
  }
  float* const d_l = ws.delta(grp) + rows0 + row_len * (z_row - iw) + n;
  float* const slope_l = ws.w(grp) + rows0 + row_len * (z_row - iw) + n;

  f32x4 dqa[NS][NDB];    // half s: columns 0..7 sum e (dP - ref) kt, 8..15 sum e kt of the half's columns; d = 16 db + 4 g + e
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int db = 0; db < NDB; ++db) dqa[s][db] = f32x4{0, 0, 0, 0};
  float m_run = -1e30f, l_run = 0.f, pd_run = 0.f;   // reference value of the exponentials; this lane's sums of e and e dP
  float carry = 0.f;                                  // gates to the right of the block, up to the diagonal

  const int nb = iw / 16 + 1;
  // A block of 16 rows of K or V: an operand piece read straight from memory is 16 bytes of a row per lane, neighbouring lanes in different
  // rows, and the address unit then handles one lane per cycle (which bound this kernel).  So a block is requested with
  // consecutive pieces in consecutive lanes and takes its operand order in LDS.
  auto request = [&](u32x4 (&x)[NKS], const uint16_t* base, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NKS; ++u) {
      const int e = lane + u * kWave;
      const uint32_t row = min(16 * b + e / (D / 8), N - 1);   // (only the block on the diagonal can reach past the end)
      x[u] = *reinterpret_cast<const u32x4*>(byte_offset(base, row * (D * 2) + e % (D / 8) * 16));
    }
  };
  auto park = [&](const u32x4 (&x)[NKS], uint16_t* tile) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NKS; ++u) {
      const int e = lane + u * kWave;
      *reinterpret_cast<u32x4*>(tile + e / (D / 8) * BS + e % (D / 8) * 8) = x[u];
    }
  };
  auto take = [&](u32x4 (&x)[NKS], const uint16_t* tile) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) x[ks] = *reinterpret_cast<const u32x4*>(tile + n * BS + 32 * ks + 8 * g);
  };
  u32x4 kraw[NKS];
  u32x4 va[NKS], da[NKS];
  f32x4 dp;   // dP of this lane's column for the block at hand
  auto fetch_dp = [&](int b) __attribute__((always_inline)) {
    request(va, vbase, b);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) da[ks] = *reinterpret_cast<const u32x4*>(do_l + 32 * ks);
  };
  // What a block needs before its keys can be rotated, done for the next block at the end of this one: its keys and values in operand order,
  // dP, the leader logits (row m of A is the leader of query row m R / 16, so lane (key n, g) finds the logit of its own query row z_row),
  // gates and delta of (z_row, key n).  The steps are short and each waits for the one before: together their waits overlap.
  float z, delta;
  auto prepare = [&](int b, bool diagonal) __attribute__((always_inline)) {
    lds_order();
    park(va, kt);
    park(kraw, kt + 16 * BS);
    lds_order();
    take(va, kt);
    take(kraw, kt + 16 * BS);
    lds_order();
    f32x4 lg = f32x4{0, 0, 0, 0};
    dp = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      lg = mfma16(*reinterpret_cast<const u32x4*>(lead + n * R / 16 * (D + 8) + 32 * ks + 8 * g), kraw[ks], lg);
      dp = mfma16(va[ks], da[ks], dp);
    }
    z = sigmoid(lg[0] * p.sm_scale);
    if (diagonal && 16 * b + n > z_row) z = 0.f;
    const float zpre = row16_prefix_sum(z), ztot = row16_last(zpre);
    delta = carry + (ztot - zpre);   // gates strictly to the right, up to and including the diagonal
    carry += ztot;
  };
  fetch_dp(nb - 1);
  for (int e = lane; e < R * (D / 8); e += kWave)
    *reinterpret_cast<u32x4*>(lead + e / (D / 8) * (D + 8) + e % (D / 8) * 8) =
        *reinterpret_cast<const u32x4*>(p.q + ((int64_t)head0 * N + min(iw + e / (D / 8), N - 1)) * D + e % (D / 8) * 8);
  lds_order();
  request(kraw, kbase, nb - 1);
  prepare(nb - 1, true);
#pragma unroll
  for (int hk = 0; hk < HK; ++hk)
#pragma unroll
    for (int e = 0; e < 8; ++e) asm volatile("" ::"v"(turns[hk][e]));
#pragma unroll 1
  for (int b = nb - 1; b >= 0; --b) {
    const bool diagonal = b == nb - 1;   // wave-uniform
    float k1[HK][8], k2[HK][8];
#pragma unroll
    for (int hk = 0; hk < HK; ++hk)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        k1[hk][2 * e] = elt_lo(kraw[hk][e]);
        k1[hk][2 * e + 1] = elt_hi(kraw[hk][e]);
        k2[hk][2 * e] = elt_lo(kraw[HK + hk][e]);
        k2[hk][2 * e + 1] = elt_hi(kraw[HK + hk][e]);
      }
    request(kraw, kbase, max(b - 1, 0));
    *byte_offset(d_l, 64u * b) = delta;
    *byte_offset(slope_l, 64u * b) = z * (1.f - z);   // the sigmoid's slope; replaced by W in the second sweep

    // rotated keys -> LDS, scores and dS/ddelta
    f32x4 m[NS];
    static_for<R>([&](auto r_c) __attribute__((always_inline)) {
      constexpr int r = decltype(r_c)::value, s = r / RH;
      const float delta_r = R == 1 ? delta : __shfl(delta, 64 / R * r + n);
      f32x4 acc = f32x4{0, 0, 0, 0};
      static_for<HK>([&](auto hk_c) __attribute__((always_inline)) {
        constexpr int hk = decltype(hk_c)::value;
        f16x8 y1, y2;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x = corope_phase<(hk < REDUCED)>(delta_r * turns[hk][e]);
          const float sn = __builtin_amdgcn_sinf(x), cs = __builtin_amdgcn_cosf(x);
          y1[e] = (_Float16)__builtin_fmaf(cs, k1[hk][e], sn * k2[hk][e]);
          y2[e] = (_Float16)__builtin_fmaf(cs, k2[hk][e], -(sn * k1[hk][e]));
        }
        const u32x4 w1 = __builtin_bit_cast(u32x4, y1), w2 = __builtin_bit_cast(u32x4, y2);
        uint16_t* dst = kt + (r * 16 + n) * TS + 32 * hk + 8 * g;
        *reinterpret_cast<u32x4*>(dst) = w1;
        *reinterpret_cast<u32x4*>(dst + HALF) = w2;
        acc = mfma16_f16(w1, qop[s][hk], acc);
        acc = mfma16_f16(w2, qop[s][HK + hk], acc);
      });
      if (r % RH == 0) {
        m[s] = acc;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) m[s][e] = place == r % RH ? acc[e] : m[s][e];
      }
    });
    // The operands of the next block's dP take the registers that this block's keys have left: requested here, used at the end
    __builtin_amdgcn_sched_barrier(0);
    fetch_dp(max(b - 1, 0));
    __builtin_amdgcn_sched_barrier(0);
    f32x4 sc, gd;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x0 = m[0][e], x1 = m[NS - 1][e];
      sc[e] = (low ? x0 : x1) * scale2;
      gd[e] = (NS > 1 && low ? x1 : x0) * p.sm_scale;
    }
    {
      f32x4 s_out, g_out;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s_out[e] = __shfl(NS == 1 && !low ? gd[e] : sc[e], from);
        if constexpr (NS > 1) g_out[e] = __shfl(gd[e], from);
      }
      *reinterpret_cast<f32x4*>(byte_offset(s_l, 64u * b)) = s_out;
      if constexpr (NS > 1) *reinterpret_cast<f32x4*>(byte_offset(g_l, 64u * b)) = g_out;
    }
    // Two rows share the contraction slots of the dq products, the other row's columns of B being zero: a rotated key that is not
    // finite (a leader's row that is not, a key beyond fp16 once rotated) would reach the other row's dq.  It shows in its own row's scores,
    // and through them in that row's statistics and dq; in LDS it is then replaced by zero.  Rare: the common case costs five instructions a
    // block.
    if constexpr (RH > 1) {
      float poison = 0.f;   // NaN if a score is not finite
#pragma unroll
      for (int e = 0; e < 4; ++e) poison = __builtin_fmaf(sc[e], 0.f, poison);
      if (__builtin_amdgcn_ballot_w64(poison != poison) != 0) {   // wave-uniform
        lds_order();
#pragma unroll 1
        for (int e = lane; e < R * 16 * (D / 2); e += kWave) {
          uint32_t* at = reinterpret_cast<uint32_t*>(kt + e / (D / 2) * TS) + e % (D / 2);
          uint32_t w = *at;
          if ((w & 0x7c00u) == 0x7c00u) w &= 0xffff0000u;
          if ((w & 0x7c000000u) == 0x7c000000u) w &= 0xffffu;
          *at = w;
        }
        lds_order();
      }
    }
    if (diagonal) {
      const int rel = own_row - 16 * b - 4 * g;   // last key the row sees, relative to this lane's first
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sc[e] = e > rel ? -INFINITY : sc[e];
        dp[e] = e > rel ? 0.f : dp[e];              // not defined there
      }
    }
    // The reference value only has to keep the exponentials in range, it need not be the running maximum (any value gives the
    // same P once the row is normalised): it moves, to the exact maximum so far and with the usual rescaling, only when some score
    // of the block lies more than kLazyMargin above it.  The margin bounds the weights that go to the matrix cores as fp16.
    constexpr float kLazyMargin = 5.f;   // base-2 units
    float x[4], top = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = sc[e] - m_run;
      top = fmaxf(top, x[e]);
    }
    if (__builtin_amdgcn_ballot_w64(top > kLazyMargin) != 0) {   // wave-uniform
      top = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
      top = fmaxf(top, __shfl_xor(top, 16));
      top = fmaxf(top, __shfl_xor(top, 32));
      const float m_new = fmaxf(m_run, top);   // finite: the block holds a key <= row
      const float al = fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= al;
      pd_run *= al;
      const float al_x = __shfl_xor(al, 8);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const float f = (n / 8 == s) ? al : al_x;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int e = 0; e < 4; ++e) dqa[s][db][e] *= f;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = sc[e] - m_run;
    }
    float we[4], wd[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      we[e] = fast_exp2(x[e]);   // 0 for the keys beyond the diagonal
      l_run += we[e];
      pd_run = __builtin_fmaf(we[e], dp[e], pd_run);
      // (clamped to fp16's range: a value row |v_j| in the thousands saturates instead of turning into infinity)
      wd[e] = fminf(fmaxf(we[e] * __builtin_fmaf(dp[e], w_inv, -ref_scaled), -65504.f), 65504.f);
    }
    const u32x2 pd = {pack_f16(wd[0], wd[1]), pack_f16(wd[2], wd[3])}, pe = {pack_f16(we[0], we[1]), pack_f16(we[2], we[3])};
    u32x2 wts[NS];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint32_t pe_x = row16_ror8(pe[t]), pd_x = row16_ror8(pd[t]);   // all lanes active
      wts[0][t] = low ? pd[t] : pe_x;
      if constexpr (NS > 1) wts[NS - 1][t] = low ? pd_x : pe[t];
    }
    lds_order();   // rotated keys are in LDS
    static_for<NS>([&](auto s_c) __attribute__((always_inline)) {
      constexpr int s = decltype(s_c)::value;
      u32x4 bop;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        bop[t] = busy && place == 0 ? wts[s][t] : 0u;
        bop[2 + t] = place == 1 ? wts[s][t] : 0u;
      }
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        const u32x2 a0 = load_a_trans16_block(kt + s * RH * 16 * TS, TS, 16 * db);
        if constexpr (RH > 1) {
          const u32x2 a1 = load_a_trans16_block(kt + (s * RH + 1) * 16 * TS, TS, 16 * db);
          dqa[s][db] = mfma16_f16(u32x4{a0[0], a0[1], a1[0], a1[1]}, bop, dqa[s][db]);
        } else {
          dqa[s][db] = mfma16x16_f16(a0, u32x2{bop[0], bop[1]}, dqa[s][db]);
        }
      }
    });
    lds_order();   // ... and consumed: the next block may overwrite them
    prepare(b - 1, false);   // (before block 0: again block 0, unused)
  }
  // row statistics: 1 / sum of exponentials, rowsum(P o dP)
  l_run += __shfl_xor(l_run, 16);
  l_run += __shfl_xor(l_run, 32);
  pd_run += __shfl_xor(pd_run, 16);
  pd_run += __shfl_xor(pd_run, 32);
  const float inv_l = 1.f / l_run, dsum = pd_run * inv_l;

  if ((NS > 1 || low) && busy && g == 0 && iw + half * RH + place < N) {   // for the dv kernel
    ws.row_max(grp, G, N, head)[own_row] = m_run;
    ws.row_inv(grp, G, N, head)[own_row] = inv_l;
  }

  // (sum e (dP - ref) kt - (Delta - ref) sum e kt) / L, the second sum sitting eight lanes up.  dq of the heads 1..G-1 is final; the
  // leader's still lacks the gate path W K, which a separate plain matrix product adds (corope_bwd_dq_leader): its row
  // goes to the workspace in fp32, unscaled
  {
    const float corr = dsum - dref;
    const float inv_x = __shfl_xor(inv_l, 8), corr_x = __shfl_xor(corr, 8), mul_x = __shfl_xor(w_mul, 8);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int row = iw + s * RH + place;
      const float my_inv = s == 0 ? inv_l : inv_x, my_corr = s == 0 ? corr : corr_x, my_mul = s == 0 ? w_mul : mul_x;
      const bool mine = low && busy && row < N;
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        f32x4 val;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = dqa[s][db][e], plain = __shfl_xor(a, 8);
          val[e] = (a * my_mul - my_corr * plain) * my_inv;
        }
        if (mine) {
          if (head == 0)
            *reinterpret_cast<f32x4*>(ws.dql(grp, N, D) + (int64_t)row * D + db * 16 + 4 * g) = val;
          else
            *reinterpret_cast<u32x2*>(p.dq + ((int64_t)(head0 + head) * N + row) * D + db * 16 + 4 * g) =
                u32x2{pack_elts(val[0] * p.sm_scale, val[1] * p.sm_scale), pack_elts(val[2] * p.sm_scale, val[3] * p.sm_scale)};
        }
      }
    }
  }

  // ---- left to right: dS, G_ij = sum_h dS dS/ddelta, its running sum over the keys, W: 64 keys at a time, lane = (row, R keys) ------
  // dP once more from V and dO: lane = column there, through LDS to lane = (row, keys).  What the lanes read here other lanes of this
  // wave wrote above.
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  constexpr int SEG = kWave / R;   // lanes of a row
  typedef float keys_t __attribute__((ext_vector_type(R)));
  float* const dpt = reinterpret_cast<float*>(kt + 16 * BS);
  const int row2 = lane / SEG, key0 = (lane % SEG) * R, i2 = min(iw + row2, N - 1);
  const int col2 = row2 / RH * 8 + row2 % RH * G;   // column of (row2, head 0)
  float m_row[G], l_row[G], d_row[G];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    m_row[h] = __shfl(m_run, col2 + h);
    l_row[h] = __shfl(inv_l, col2 + h);
    d_row[h] = __shfl(dsum, col2 + h);
  }
  const uint32_t at = 4u * (row_len * (i2 - iw) + key0);
  float* const w_base = ws.w(grp) + rows0;   // wave-uniform bases, addressed with 32-bit byte offsets
  const float* const s_base = ws.s(head0) + rows0;
  float* const ds_base = ws.ds(head0) + rows0;
  u32x4 dop[NKS], vraw[4][NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) dop[ks] = *reinterpret_cast<const u32x4*>(do_l + 32 * ks);
  // The matrices come from memory and are requested two chunks ahead, in two register sets; V comes from the cache, one chunk ahead.
  keys_t sl_n[2], sv_n[2][G], gv_n[2][G];
  const int n_chunks = iw / kWave + 1;
  auto fetch_v = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 4; ++t) request(vraw[t], vbase, 4 * c + t);
  };
  auto fetch_rows = [&](int c, auto set_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
    const uint32_t off = at + 256u * c;
    sl_n[set] = *reinterpret_cast<const keys_t*>(byte_offset(w_base, off));
#pragma unroll
    for (int h = 0; h < G; ++h) {
      sv_n[set][h] = *reinterpret_cast<const keys_t*>(byte_offset(s_base + h * ws.NN, off));
      gv_n[set][h] = *reinterpret_cast<const keys_t*>(byte_offset(ds_base + h * ws.NN, off));
    }
  };
  float gcarry = 0.f;
  auto chunk = [&](int c, auto set_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      lds_order();
      park(vraw[t], kt);
      lds_order();
      take(vraw[t], kt);
      f32x4 dp = f32x4{0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) dp = mfma16(vraw[t][ks], dop[ks], dp);
      *reinterpret_cast<f32x4*>(dpt + (half * 8 + sub) * PS + 16 * t + 4 * g) = dp;
    }
    // take this chunk's values out of the look-ahead registers and request the later chunks' before anything is stored,
    // so that waiting for them never waits for this chunk's stores
    const keys_t slope = sl_n[set];
    keys_t sv[G], gv[G];
#pragma unroll
    for (int h = 0; h < G; ++h) {
      sv[h] = sv_n[set][h];
      gv[h] = gv_n[set][h];
    }
    fetch_v(min(c + 1, n_chunks - 1));
    fetch_rows(min(c + 2, n_chunks - 1), set_c);
    lds_order();   // dP is in LDS
    float gij[R];
#pragma unroll
    for (int x = 0; x < R; ++x) gij[x] = 0.f;
#pragma unroll
    for (int h = 0; h < G; ++h) {
      const keys_t dp = *reinterpret_cast<const keys_t*>(dpt + (col2 + h) * PS + key0);
#pragma unroll
      for (int x = 0; x < R; ++x) {
        const float pr = fast_exp2(sv[h][x] - m_row[h]) * l_row[h];
        const float ds = pr * (dp[x] - d_row[h]);
        gij[x] = __builtin_fmaf(ds, gv[h][x], gij[x]);
        gv[h][x] = ds;
      }
    }
    lds_order();   // ... and read: the next chunk's may overwrite it
    float tot = 0.f;
#pragma unroll
    for (int x = 0; x < R; ++x) {
      if (c * kWave + key0 + x > i2) gij[x] = 0.f;   // nothing beyond the diagonal is defined
      tot += gij[x];
    }
    const float pre = segment_prefix_sum<SEG>(tot);
    float left = gcarry + (pre - tot);               // G over the keys to the left of this lane's first
    gcarry += segment_last<SEG>(pre);
    keys_t wij;
#pragma unroll
    for (int x = 0; x < R; ++x) {
      wij[x] = left * slope[x];                      // (sum of G over the keys j < t) z'(t)
      left += gij[x];
    }
    const uint32_t off = at + 256u * c;
#pragma unroll
    for (int h = 0; h < G; ++h) *reinterpret_cast<keys_t*>(byte_offset(ds_base + h * ws.NN, off)) = gv[h];
    *reinterpret_cast<keys_t*>(byte_offset(w_base, off)) = wij;
  };
  fetch_rows(0, std::integral_constant<int, 0>{});
  fetch_v(0);
  fetch_rows(min(1, n_chunks - 1), std::integral_constant<int, 1>{});
#pragma unroll 1
  for (int c = 0; c < n_chunks; c += 2) {
    chunk(c, std::integral_constant<int, 0>{});
    if (c + 1 == n_chunks) break;
    chunk(c + 1, std::integral_constant<int, 1>{});
  }
}

// ---------------------------------------------------------------------------------------------------- leader's dq
// dq_leader_i = c (partial_i + sum_{t <= i} W_it k_t): a plain (rows x keys) x (keys x D) product on the matrix cores,
// computed transposed (dq^T += K^T W^T) so that W is read along its packed rows: lane = query row, 8 consecutive keys per
// step, each value split into two bf16 parts (the keys are exact, so the product carries W to about 16 bits).  One
// workgroup of 4 waves owns 32 rows of one group; every wave takes each fourth step of 16 keys, staged in LDS of its own and read
// transposed, and the four sums are added at the end.  Its workgroups come first in the dv launch.
// What bounds it: the chain of steps of the last rows (short sequences), the reads of W (long ones).  128 rows per workgroup, 32 a wave, every wave all
// steps behind two barriers each -> this: the dv launch B2 Hq8 Hkv2 N512 D64 25.3 -> 11.0 us, B2 Hq32 Hkv8 N4096 D128 990 -> 921 us; forward +
// backward B1 Hq8 Hkv2 N1024 D64 190 -> 157 us, B2 Hq16 Hkv16 N700 D64 fp16 435 -> 386 us.
constexpr int kLeaderRows = 32;

template <int D>
struct CoropeLeaderCfg {
  static constexpr int TS = D + 16, STEP = 16, kSumStride = 36;   // key rows; a wave's sums, [row][32 columns], fp32
  static constexpr int kElems = std::max(4 * STEP * TS, 4 * kLeaderRows * kSumStride * 2);
};

template <int D>
__device__ __forceinline__ void corope_bwd_dq_leader(const CoropeBwdParams& p, const CoropeBwdWs& ws, uint16_t* lds, int g, int rb) {
  using Cfg = CoropeLeaderCfg<D>;
  constexpr int TS = Cfg::TS, NDB = D / 32, STEP = Cfg::STEP, PER = STEP * (D / 8) / kWave, SS = Cfg::kSumStride;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r = lane % 32, hf = lane / 32;
  const int N = p.N, b = g / p.Hkv, kvh = g % p.Hkv, G = p.Hq / p.Hkv;
  const int i0 = rb * kLeaderRows, i = i0 + r;                           // the workgroup's first row, this lane's row
  const uint16_t* kbase = p.k + (int64_t)g * N * D;
  const float* wrow = ws.w(g) + tri_row_start(min(i, N - 1));
  uint16_t* const tile = lds + wave * STEP * TS;
  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = f32x16{0};
  const int steps = (min(N, i0 + kLeaderRows) + STEP - 1) / STEP;        // up to the last row's diagonal
  // the key rows and this lane's W values are fetched into registers two of the wave's steps ahead
  u32x4 kreg[2][PER];
  f32x4 w0[2], w1[2];
  auto fetch = [&](int step, auto set_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
    const int t0 = min(step, steps - 1) * STEP;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = lane + u * kWave;
      kreg[set][u] = *reinterpret_cast<const u32x4*>(kbase + (int64_t)min(t0 + e / (D / 8), N - 1) * D + 8 * (e % (D / 8)));
    }
    const int t = t0 + 8 * hf;     // first of this lane's 8 keys; t <= i keeps the 32-byte read inside the padded row
    w0[set] = w1[set] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (i < N && t <= i) {
      w0[set] = *reinterpret_cast<const f32x4*>(wrow + t);
      w1[set] = *reinterpret_cast<const f32x4*>(wrow + t + 4);
    }
  };
  auto multiply = [&](int step, auto set_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
    lds_order();   // the previous step's reads of the tile are done
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = lane + u * kWave;
      *reinterpret_cast<u32x4*>(tile + (e / (D / 8)) * TS + 8 * (e % (D / 8))) = kreg[set][u];
    }
    const int t = step * STEP + 8 * hf;
    float hi[8], lo[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const float wv = (i < N && t + x <= i) ? (x < 4 ? w0[set][x] : w1[set][x - 4]) : 0.f;   // nothing beyond the diagonal is defined
      hi[x] = elt_to_f(f_to_elt(wv));
      lo[x] = wv - hi[x];
    }
    const u32x4 bhi = {pack_elts(hi[0], hi[1]), pack_elts(hi[2], hi[3]), pack_elts(hi[4], hi[5]), pack_elts(hi[6], hi[7])};
    const u32x4 blo = {pack_elts(lo[0], lo[1]), pack_elts(lo[2], lo[3]), pack_elts(lo[4], lo[5]), pack_elts(lo[6], lo[7])};
    fetch(step + 8, set_c);
    lds_order();
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      const u32x4 a = load_a_trans_natural(tile, TS, 0, 32 * db);
      acc[db] = mfma32(a, bhi, acc[db]);
      acc[db] = mfma32(a, blo, acc[db]);
    }
  };
  fetch(wave, std::integral_constant<int, 0>{});
  fetch(wave + 4, std::integral_constant<int, 1>{});
#pragma unroll 1
  for (int step = wave; step < steps; step += 8) {
    multiply(step, std::integral_constant<int, 0>{});
    if (step + 4 >= steps) break;
    multiply(step + 4, std::integral_constant<int, 1>{});
  }
  // the four waves' sums, 32 columns at a time: thread = (row, 4 columns)
  float* const sums = reinterpret_cast<float*>(lds);
  const int row = threadIdx.x / 8, d4 = threadIdx.x % 8 * 4;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    __syncthreads();
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
      *reinterpret_cast<f32x4*>(sums + (wave * kLeaderRows + r) * SS + 8 * g4 + 4 * hf) =
          f32x4{acc[db][4 * g4], acc[db][4 * g4 + 1], acc[db][4 * g4 + 2], acc[db][4 * g4 + 3]};
    __syncthreads();
    if (i0 + row < N) {
      f32x4 sum = *reinterpret_cast<const f32x4*>(ws.dql(g, N, D) + (int64_t)(i0 + row) * D + db * 32 + d4);
#pragma unroll
      for (int w = 0; w < 4; ++w) sum += *reinterpret_cast<const f32x4*>(sums + (w * kLeaderRows + row) * SS + d4);
      *reinterpret_cast<u32x2*>(p.dq + ((int64_t)(b * p.Hq + kvh * G) * N + i0 + row) * D + db * 32 + d4) =
          u32x2{pack_elts(sum[0] * p.sm_scale, sum[1] * p.sm_scale), pack_elts(sum[2] * p.sm_scale, sum[3] * p.sm_scale)};
    }
  }
}

// ---------------------------------------------------------------------------------------------------- equal shares
// The dv and dk kernels sum over query rows into blocks of 128 keys.  Key block kb sees the rows from its first key on, so
// the blocks of a group differ in work by their number, and a group of 512 rows has four of them: a workgroup per block (or
// per pair of a long and a short one) left most of the chip idle on short sequences.  Instead the row tiles of a group's
// blocks, block after block, form one list that `shares` workgroups cut into equal pieces.  A piece that holds all of a block
// writes the block's result; the others leave fp32 partial sums in a slot of their own, at most one at each end of a piece,
// and corope_bwd_sum_kernel adds a block's slots in list order.  The cut depends on the sizes alone and not on how many
// groups a pass handles, so a smaller workspace gives the same bits.
// Measured: B2 Hq8 Hkv2 N512 D64 dk 414 -> 33 us and dv 55 -> 9 us, plus 7 us each for the sums; B2 Hq32 Hkv8 N4096 D128 dk
// 4.69 -> 4.05 ms (two workgroups per compute unit, all of equal length, instead of one) and dv 0.67 -> 0.48 ms.
constexpr int kDkKeys = 128;   // keys per block

template <int ROWS>
struct CoropeShares {
  static_assert(kDkKeys % ROWS == 0, "a block starts on a tile");
  int n_tiles, n_blocks, total;   // row tiles of block 0, key blocks, tiles of a whole group
  __device__ __host__ explicit CoropeShares(int N) {
    n_tiles = (N + ROWS - 1) / ROWS;
    n_blocks = (N + kDkKeys - 1) / kDkKeys;
    total = first(n_blocks);
  }
  __device__ __host__ int first(int kb) const { return kb * n_tiles - kDkKeys / ROWS * (kb * (kb - 1) / 2); }   // tiles before block kb
  __device__ int begin(int share, int shares) const { return (int)((int64_t)share * total / shares); }
  __device__ int owner(int tile, int shares) const { return (int)((((int64_t)tile + 1) * shares - 1) / total); }   // begin(owner) <= tile
  // A piece's partial sums: slot 1 if they start at the block's first tile, slot 0 if an earlier piece started the block.
  __device__ static int64_t slot(int share, bool starts_block) { return 2 * (int64_t)share + (starts_block ? 1 : 0); }
};

// Adds the partial sums of the blocks that were cut: out[key][d] = scale * sum over the block's pieces.
template <int D, int ROWS>
__global__ __launch_bounds__(256) void corope_bwd_sum_kernel(const float* parts, int64_t group_floats, uint16_t* out, int N, int shares,
                                                             float scale) {
  const CoropeShares<ROWS> sh(N);
  const int kb = blockIdx.x, g = blockIdx.y;
  const int w0 = sh.owner(sh.first(kb), shares), w1 = sh.owner(sh.first(kb + 1) - 1, shares);
  if (w0 == w1) return;   // one piece holds all of the block and has written it
  const float* src = parts + (int64_t)g * group_floats;
  for (int e = blockIdx.z * 256 + threadIdx.x; e < kDkKeys * D / 4; e += 256 * gridDim.z) {
    const int j = kb * kDkKeys + e / (D / 4);
    if (j >= N) break;
    f32x4 sum = *reinterpret_cast<const f32x4*>(src + sh.slot(w0, true) * (kDkKeys * D) + 4 * e);
    for (int w = w0 + 1; w <= w1; w += 4) {   // four loads in flight
      f32x4 x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const f32x4*>(src + sh.slot(min(w + u, w1), false) * (kDkKeys * D) + 4 * e);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (w + u <= w1) sum += x[u];
    }
    *reinterpret_cast<u32x2*>(out + ((int64_t)g * N + kb * kDkKeys) * D + 4 * e) =
        u32x2{pack_elts(sum[0] * scale, sum[1] * scale), pack_elts(sum[2] * scale, sum[3] * scale)};
  }
}

// ---------------------------------------------------------------------------------------------------- dv
// dv_j = sum_{h, i} P^h_ij dO^h_i on the matrix cores: dv^T (d x keys) += dO^T (d x rows) P (rows x keys), 16 rows per
// step.  A workgroup of 4 waves takes 128 keys at a time (32 per wave) of one group, equal shares of the rows as above; the 16 dO
// rows of every head are staged in LDS and read transposed; S comes straight from the workspace (lane = key: 128-byte lines), becomes P
// with the row's statistics and is rounded to the element type.
// The leader's dq needs nothing of dv's and both wait for memory, so their workgroups share a launch: forward + backward
// B2 Hq8 Hkv2 N512 D64 129.7 -> 127.3 us, and 5 % where the groups are fewer; at N = 4096, where each fills the chip by itself, no difference.
constexpr int kDvRows = 16;

template <int D, int G>
__global__ __launch_bounds__(4 * kWave) void corope_bwd_dv_kernel(CoropeBwdParams p, CoropeBwdWs ws, float* parts, int64_t group_floats,
                                                                     int shares) {
  constexpr int TS = D + 16, NDB = D / 32, NT = 4 * kWave, ROWS = kDvRows;
  constexpr int UNITS = G * ROWS * (D / 8), PER = (UNITS + NT - 1) / NT;   // 16-byte pieces of a dO tile, per thread
  __shared__ __attribute__((aligned(16))) uint16_t tile[std::max(G * ROWS * TS, CoropeLeaderCfg<D>::kElems)];
  __shared__ __attribute__((aligned(16))) float stat[2][2 * G * ROWS];   // two steps' [reference values, 1 / sums][head][row]
  static_assert(2 * G * ROWS <= NT, "one statistic per thread");
  const int n_groups = p.B * p.Hkv, leader_blocks = (p.N + kLeaderRows - 1) / kLeaderRows * n_groups;
  if ((int)blockIdx.x < leader_blocks) {   // the last row blocks of all groups see the most keys: first
    corope_bwd_dq_leader<D>(p, ws, tile, blockIdx.x % n_groups, (leader_blocks - 1 - (int)blockIdx.x) / n_groups);
    return;
  }
  const int g = ((int)blockIdx.x - leader_blocks) / shares, share = ((int)blockIdx.x - leader_blocks) % shares;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int r = lane % 32, hf = lane / 32;
  const int N = p.N, b = g / p.Hkv, kvh = g % p.Hkv;
  const int head0 = b * p.Hq + kvh * G;
  const CoropeShares<ROWS> sh(N);
  int kb = 0;
#pragma unroll 1
  for (int t = sh.begin(share, shares), t_end = sh.begin(share + 1, shares); t < t_end;) {
    while (sh.first(kb + 1) <= t) ++kb;
    const int b0 = sh.first(kb), b1 = sh.first(kb + 1), seg_end = min(t_end, b1);
    const int jb = kb * kDkKeys, row_end = min(N, jb + ROWS * (seg_end - b0));
    const int jw = jb + 32 * wave, j = jw + r;
    f32x16 acc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = f32x16{0};

    // Both streams run one step ahead in registers: the steps of a piece follow one after the other, and with a step's loads
    // issued only when the step begins its time is that many memory latencies.
    u32x4 dreg[PER];
    float pnext[G][8], stat_next = 0.f;
    auto fetch_stat = [&](int i0) __attribute__((always_inline)) {
      const int i = i0 + threadIdx.x % ROWS;
      if (threadIdx.x < 2 * G * ROWS) stat_next = i < N ? ws.row_max(g, G, N, threadIdx.x / ROWS)[i] : 0.f;
    };
    auto park_stat = [&](int step) __attribute__((always_inline)) {
      if (threadIdx.x < 2 * G * ROWS) stat[step % 2][threadIdx.x] = stat_next;
    };
    auto fetch = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int e = min((int)threadIdx.x + u * NT, UNITS - 1);
        const int h = e / (ROWS * (D / 8)), rr = (e / (D / 8)) % ROWS, v8 = e % (D / 8);
        dreg[u] = *reinterpret_cast<const u32x4*>(p.d_o + ((int64_t)(head0 + h) * N + min(i0 + rr, N - 1)) * D + 8 * v8);
      }
      const bool wave_on = i0 + ROWS - 1 >= jw && jw < N;   // wave-uniform: some row of the step sees a key of this wave
      const int64_t row_len = 64 * (i0 / 64 + 1);           // the 16 rows of a step share a row length
#pragma unroll
      for (int h = 0; h < G; ++h) {
        const float* srow = ws.s(head0 + h) + tri_row_start(min(i0, N - 1)) + j;
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          const int i = i0 + 8 * hf + x;
          pnext[h][x] = (wave_on && i < N && j <= i) ? srow[row_len * (8 * hf + x)] : 0.f;   // nothing outside the triangle is defined
        }
      }
    };
    const int row_begin = jb + ROWS * (t - b0);
    fetch(row_begin);
    fetch_stat(row_begin);
    __syncthreads();   // the previous piece's reads are done
    park_stat(0);
    fetch_stat(row_begin + ROWS);
#pragma unroll 1
    for (int i0 = row_begin, step = 0; i0 < row_end; i0 += ROWS, ++step) {
      __syncthreads();   // the previous step's reads of the tile are done, this step's statistics are there
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int e = threadIdx.x + u * NT;
        if (UNITS % NT == 0 || e < UNITS)
          *reinterpret_cast<u32x4*>(tile + (e / (D / 8)) * TS + 8 * (e % (D / 8))) = dreg[u];   // rows are (head, row) pairs
      }
      park_stat(step + 1);   // (two steps ahead of their use, so that the weights are ready when the tile is)
      fetch_stat(i0 + 2 * ROWS);
      const float* st = stat[step % 2];
      u32x4 bop[G];
#pragma unroll
      for (int h = 0; h < G; ++h) {
        float w[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {   // (a key the row does not see has weight zero also where the row's statistics are NaN)
          const float e = fast_exp2(pnext[h][x] - st[h * ROWS + 8 * hf + x]) * st[(G + h) * ROWS + 8 * hf + x];
          w[x] = j <= i0 + 8 * hf + x ? e : 0.f;
        }
        bop[h] = u32x4{pack_elts(w[0], w[1]), pack_elts(w[2], w[3]), pack_elts(w[4], w[5]), pack_elts(w[6], w[7])};
      }
      const bool wave_on = i0 + ROWS - 1 >= jw && jw < N;
      if (i0 + ROWS < row_end) fetch(i0 + ROWS);
      __syncthreads();
      if (wave_on) {
#pragma unroll
        for (int h = 0; h < G; ++h)
#pragma unroll
          for (int db = 0; db < NDB; ++db)
            acc[db] = mfma32(load_a_trans_natural(tile + h * ROWS * TS, TS, 0, 32 * db), bop[h], acc[db]);
      }
    }
    const bool whole = t == b0 && seg_end == b1;
    if (j < N) {
      uint16_t* op = p.dv + ((int64_t)g * N + j) * D;
      float* pp = parts + (int64_t)g * group_floats + sh.slot(share, t == b0) * (kDkKeys * D) + (j - jb) * D;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const f32x4 x = {acc[db][4 * g4], acc[db][4 * g4 + 1], acc[db][4 * g4 + 2], acc[db][4 * g4 + 3]};
          if (whole)
            *reinterpret_cast<u32x2*>(op + db * 32 + 8 * g4 + 4 * hf) = u32x2{pack_elts(x[0], x[1]), pack_elts(x[2], x[3])};
          else
            *reinterpret_cast<f32x4*>(pp + db * 32 + 8 * g4 + 4 * hf) = x;
        }
    }
    t = seg_end;
  }
}

// ---------------------------------------------------------------------------------------------------- dk
// dk_j = c sum_i [ R(+delta_ij)(sum_h dS^h_ij q^h_i) + W_ij qL_i ].  A workgroup of 4 waves takes 128 keys of one group at a time
// (32 per wave) and walks query rows, 8 per staged tile.  Per row:
//   u = sum_h dS^h q^h for the wave's 32 keys and all D columns: a (32 keys x heads) x (heads x D) product on the
//       matrix cores - the contraction is only G long, but it takes 2G multiply-adds per (key, pair) off the vector
//       units; the result lands as lane = column (mod 32), registers = 16 of the wave's keys;
//   rotation and accumulation on the vector units: lane (c, half) owns pairs c and c + 32 (D = 128) for the 16 keys of
//       its half: one (sin, cos) and four multiply-adds per (row, key, pair).
// The gate path W qL contracts over rows, so a tile's 8 rows are one more product into the same accumulators (on the vector units it was 2 of
// 12 issue slots per (row, key, pair)).  W is split into three bf16 parts, 24 bits whatever its scale, and an fp16 query into two.
// The slow pairs (common.hpp; D = 128: half of all with theta = 10000) are not rotated per (row, key): with delta = mid_i + x, |x| <= kDkReach over
// the block's 128 keys, and complex numbers for the pairs,
//   dk_j = sum_i e^(i delta w) sum_h dS^h_ij q^h_i = sum_n sum_{i, h} (x_ij^n dS^h_ij) [ (i w)^n / n! e^(i mid_i w) q^h_i ] :
// products that contract over rows and heads, one per power.  The bracket is shared by the block's keys: the four waves prepare it once per tile,
// a wave per head.  Class 0 (|x w| <= 0.68) takes the powers 0 .. 5, class 1 (<= 0.08) 0 .. 2, the last coefficients lowered to spread the
// remainder: below 1e-5 and 2.2e-5.  Operands are bf16 parts: two of dS and two of the bracket (16 bits) up to power 2 (fp16: 3) of class 0 and 1 of
// class 1; one part of the powers above leaves an error of 4.8e-5 (fp16: 0.9e-5) and 1.6e-5 of dk for the fastest pair with every gate open, beside
// 1.7e-3 (3e-4) of its rounding.  (With one part from power 2, fp16 3, and class 1's power 1 on it was 2.4e-4, 4.8e-5 and 1.1e-4, and the kernel 3.06 instead of 3.15 ms.)  Built for up
// to five heads a group (fp16: four), whose LDS leaves two workgroups to a compute unit.
// What bounds it: the vector units, 9 or 10 issue slots per (row, key, pair) that is rotated.  Measured with the gate path moved: B2 Hq32 Hkv8 N4096 D128
// forward + backward 15.0 -> 14.6 ms, B2 Hq8 Hkv2 N512 D64 133 -> 130.5 us; with the slow pairs as products the former 13.43 -> 12.70 ms, error of
// dk against 64 bits 1.68e-3 (bf16) and 3.18e-4 (fp16) as before.
// A workgroup takes its share of the group's (block, row tile) list as above.  Tiles of DELTA, W, DS^h ([row][matrix][key], fp32) and the rows' queries
// ([row][column][head], bf16, heads padded to 8 with zeros: the B operand is then one 16-byte read) go through LDS,
// fetched into registers one tile ahead.
constexpr int kDkRows = 8, kDkWaves = 4;
constexpr float kDkReach = kDkKeys / 2, kDkLow0 = kCoropeLow0 * kDkReach / kCoropeReach, kDkLow1 = kCoropeLow1 * kDkReach / kCoropeReach;

// Where column c of a query row lies in its tile, 16 bytes (8 heads) a column.  The rows arrive eight columns a lane, so that the lanes of a store
// lie 128 bytes apart, on 4 of the 64 banks; with the bits of c / 16 below D / 2 folded into its lowest ones they spread over D / 8 of them,
// 16 neighbours still fill 16 groups of four banks, and a column's partner stays D / 2 columns on.
// B2 Hq32 Hkv8 N4096 D128: bank conflicts 3.6e8 -> 2.1e8 cycles, the kernel 3.17 -> 3.06 ms, forward + backward 12.61 -> 12.42 ms.
template <int D>
__device__ __forceinline__ constexpr int dk_slot(int c) { return c ^ (c >> 4 & (D / 32 - 1)); }

template <int D, int G, int LOW>
struct CoropeDkCfg {
  static constexpr int kMats = 2 + G;                                       // DELTA, W, DS^h
  static constexpr int kMatBytes = kDkRows * kMats * kDkKeys * 4;
  static constexpr int kQBytes = kDkRows * D * 8 * 2;                       // [row][column][8 heads] bf16
  // slow pairs: [part][head][column][row] bf16, the parts of class 0, then of class 1; the rows' reference values of delta behind them
  static constexpr int kParts0 = kEltIsF16 ? 10 : 9, kParts1 = 5;
  static constexpr int kSlowElems = (LOW > 0 ? kParts0 : 0) * G * 32 * kDkRows + (LOW > 1 ? kParts1 : 0) * G * 32 * kDkRows;
  static constexpr int kLdsBytes = kMatBytes + kQBytes + kSlowElems * 2 + (LOW > 0 ? kDkRows * 4 : 0);
};

template <int D, int G, int REDUCED, int LOW>
__global__ __launch_bounds__(kDkWaves* kWave) __attribute__((amdgpu_waves_per_eu(2))) void corope_bwd_dk_kernel(CoropeBwdParams p, CoropeBwdWs ws,
                                                                       CoropeBwdFreqs fr, float* parts, int64_t group_floats) {
  using Cfg = CoropeDkCfg<D, G, LOW>;
  constexpr int HALF = D / 2, NT = kDkWaves * kWave, MATS = Cfg::kMats;
  constexpr int FAST = HALF - 16 * LOW, NP = FAST / 32;   // pairs rotated per (row, key), in blocks of 32
  static_assert((D == 64 || D == 128) && FAST % 32 == 0, "pairs per lane are laid out for these head dims");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  float* tile = reinterpret_cast<float*>(smem);                                   // [row][matrix][key]
  uint16_t* qT = reinterpret_cast<uint16_t*>(smem + Cfg::kMatBytes);             // [row][column][8 heads]
  uint16_t* slow_q = qT + Cfg::kQBytes / 2;                                       // [part][head][column][row]
  float* mids = reinterpret_cast<float*>(slow_q + Cfg::kSlowElems);

  const int g = blockIdx.y;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int col = lane % 32, hf = lane / 32;
  const int N = p.N, b = g / p.Hkv, kvh = g % p.Hkv;
  const int head0 = b * p.Hq + kvh * G;
  const CoropeShares<kDkRows> sh(N);
  const int shares = gridDim.x, share = blockIdx.x;
  float w_turn[NP];
#pragma unroll
  for (int np = 0; np < NP; ++np) w_turn[np] = fr.turns[32 * np + col];
  float slow_turn[LOW > 0 ? LOW : 1] = {};   // of the pair whose queries this lane prepares
#pragma unroll
  for (int u = 0; u < LOW; ++u) slow_turn[u] = fr.turns[FAST + 16 * u + lane % 16];

  // heads G..7 of the query tile stay zero for the whole kernel
  for (int e = threadIdx.x; e < Cfg::kQBytes / 16; e += NT) reinterpret_cast<u32x4*>(qT)[e] = u32x4{0, 0, 0, 0};

  constexpr int kTileElems = kDkRows * MATS * kDkKeys, TI = kTileElems / NT;      // fp32 values per thread and tile
  constexpr int kRowItems = kDkRows * G * (D / 8), RI = (kRowItems + NT - 1) / NT;  // 16-byte pieces of q rows
  static_assert(kTileElems % (4 * NT) == 0, "tile elements divide evenly over the threads, four keys at a time");
  // A thread fetches four keys of (row, matrix) number first_unit + k STEP, k = 0 .. MATS - 1; the matrices come round with period PERIOD and the rows
  // then lie ROWS_ON further, so what depends on the matrix is looked up once (per tile it was a tenth of the kernel's instructions), and keys are
  // looked at one by one only where a row of the tile does not see all of them: B2 Hq32 Hkv8 N4096 D128 3.18 -> 3.06 ms.  (One head a group has few
  // matrices, and the registers cost it more: B2 H16 N2000 D64 fp16 930 -> 960 us.)
  constexpr bool KEPT = G > 1;
  constexpr int STEP = 4 * NT / kDkKeys, PERIOD = MATS % 8 == 0 ? MATS / 8 : MATS % 4 == 0 ? MATS / 4 : MATS % 2 == 0 ? MATS / 2 : MATS;
  constexpr int ROWS_ON = STEP * PERIOD / MATS;
  static_assert(STEP == 8 && STEP * PERIOD % MATS == 0, "period of the matrices");
  const int key0 = 4 * (threadIdx.x % (kDkKeys / 4));
  const float* mat_at[PERIOD];
  int row_at[PERIOD];
#pragma unroll
  for (int j = 0; j < (KEPT ? PERIOD : 0); ++j) {
    const int unit = threadIdx.x / (kDkKeys / 4) + j * STEP;
    row_at[j] = unit / MATS;
    const int m = unit % MATS, mat = m == 0 ? g : m == 1 ? ws.n_groups + g : 2 * ws.n_groups + ws.n_heads + head0 + m - 2;   // (as CoropeBwdWs counts them)
    mat_at[j] = ws.base + mat * ws.NN;
  }

  int kb = 0;
#pragma unroll 1
  for (int t = sh.begin(share, shares), t_end = sh.begin(share + 1, shares); t < t_end;) {
    while (sh.first(kb + 1) <= t) ++kb;
    const int b0 = sh.first(kb), b1 = sh.first(kb + 1), seg_end = min(t_end, b1);
    const int jb = kb * kDkKeys, jw = jb + 32 * wave;
    const int row_begin = jb + kDkRows * (t - b0), row_end = min(N, jb + kDkRows * (seg_end - b0));

    f32x4 mv[TI / 4];
    u32x4 qv[RI];
    auto fetch = [&](int i0) __attribute__((always_inline)) {
      // the 8 rows of a tile share a row length; rows past the end repeat the last one
      const int64_t tile0 = tri_row_start(i0);
      const int row_len = 64 * (i0 / 64 + 1);
      static_for<TI / 4>([&](auto k_c) __attribute__((always_inline)) {
        constexpr int k = decltype(k_c)::value;
        // four keys with one load, always inside the padded row (no branch); what is not defined there becomes zero on its way into
        // LDS (here the select would wait for the load)
        if constexpr (KEPT) {
          const uint32_t off = (uint32_t)row_len * min(row_at[k % PERIOD] + k / PERIOD * ROWS_ON, N - 1 - i0) + min(jb + key0, row_len - 4);
          mv[k] = *reinterpret_cast<const f32x4*>(mat_at[k % PERIOD] + tile0 + off);
        } else {
          const int e = 4 * (threadIdx.x + k * NT);
          const int key = e % kDkKeys, m = (e / kDkKeys) % MATS, r = e / (kDkKeys * MATS);
          const int mat = m == 0 ? g : m == 1 ? ws.n_groups + g : 2 * ws.n_groups + ws.n_heads + head0 + m - 2;
          const float* src = ws.base + mat * ws.NN;
          mv[k] = *reinterpret_cast<const f32x4*>(src + tile0 + (int64_t)row_len * min(r, N - 1 - i0) + min(jb + key, row_len - 4));
        }
      });
      static_for<RI>([&](auto k_c) __attribute__((always_inline)) {
        constexpr int k = decltype(k_c)::value;
        const int e = threadIdx.x + k * NT;
        if (kRowItems % NT == 0 || e < kRowItems) {
          const int r = e / (G * (D / 8)), h = (e / (D / 8)) % G, v8 = e % (D / 8);
          qv[k] = *reinterpret_cast<const u32x4*>(p.q + ((int64_t)(head0 + h) * N + min(i0 + r, N - 1)) * D + 8 * v8);
        }
      });
    };
    f32x16 dk1[NP], dk2[NP];
#pragma unroll
    for (int np = 0; np < NP; ++np) dk1[np] = dk2[np] = f32x16{0};
    // slow group u: lane = column, 16 of the first half and their 16 partners
    f32x16 slow[LOW > 0 ? LOW : 1];
#pragma unroll
    for (int u = 0; u < (LOW > 0 ? LOW : 1); ++u) slow[u] = f32x16{0};
    auto slow_column = [&](int u) __attribute__((always_inline)) { return FAST + 16 * u + col % 16 + (col < 16 ? 0 : HALF); };

    fetch(row_begin);
#pragma unroll 1
    for (int i0 = row_begin; i0 < row_end; i0 += kDkRows) {
      __syncthreads();   // the previous tile has been consumed
      const bool inside = i0 >= jb + kDkKeys - 1 && i0 + kDkRows <= N;   // every row of the tile sees every key of the block
      static_for<TI / 4>([&](auto k_c) __attribute__((always_inline)) {
        constexpr int k = decltype(k_c)::value;
        const int e = 4 * (threadIdx.x + k * NT), j = jb + (KEPT ? key0 : e % kDkKeys);
        const int i = i0 + (KEPT ? row_at[k % PERIOD] + k / PERIOD * ROWS_ON : e / (kDkKeys * MATS));
        f32x4 v = mv[k];
        if (!KEPT || !inside) {   // wave-uniform
#pragma unroll
          for (int x = 0; x < 4; ++x) v[x] = (i < N && j + x <= i) ? mv[k][x] : 0.f;   // outside the causal triangle or past N
        }
        *reinterpret_cast<f32x4*>(tile + e) = v;
      });
      static_for<RI>([&](auto k_c) __attribute__((always_inline)) {
        constexpr int k = decltype(k_c)::value;
        const int e = threadIdx.x + k * NT;
        if (kRowItems % NT == 0 || e < kRowItems) {
          const int r = e / (G * (D / 8)), h = (e / (D / 8)) % G, v8 = e % (D / 8);
          uint16_t* dst = qT + (r * D + 8 * v8) * 8 + h;
#pragma unroll
          for (int x = 0; x < 8; ++x) dst[8 * (x ^ (v8 >> 1 & (D / 32 - 1)))] = (uint16_t)(x % 2 ? qv[k][x / 2] >> 16 : qv[k][x / 2] & 0xffffu);
        }
      });
      __syncthreads();
      if (i0 + kDkRows < row_end) fetch(i0 + kDkRows);
      if constexpr (LOW > 0) {
        // the slow pairs' B operands: lane = (pair, two rows), a wave = one head
#pragma unroll 1
        for (int h = wave; h < G; h += kDkWaves) {
          const int pair = lane % 16, r0 = lane / 16 * 2;
          float mid[2];
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const float* trow = tile + (r0 + x) * MATS * kDkKeys;   // (keys beyond the diagonal hold zero, what delta comes to there)
            const float m = 0.5f * (trow[0] + trow[kDkKeys - 1]);
            mid[x] = __builtin_fabsf(m) < 1e30f ? m : 0.f;          // (NaN: or keys the row does not see would meet it)
            if (h == 0 && pair == 0) mids[r0 + x] = mid[x];
          }
          static_for<LOW>([&](auto u_c) __attribute__((always_inline)) {
            constexpr int u = decltype(u_c)::value;
            float v1[2], v2[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
              const uint16_t* src = qT + ((r0 + x) * D + dk_slot<D>(FAST + 16 * u + pair)) * 8 + h;
              const float q1 = elt_to_f(src[0]), q2 = elt_to_f(src[HALF * 8]);
              const float ph = __builtin_amdgcn_fractf(mid[x] * slow_turn[u]);
              const float sn = __builtin_amdgcn_sinf(ph), cs = __builtin_amdgcn_cosf(ph);
              v1[x] = __builtin_fmaf(cs, q1, -(sn * q2));
              v2[x] = __builtin_fmaf(cs, q2, sn * q1);
            }
            uint32_t* dst = reinterpret_cast<uint32_t*>(slow_q + (((u * Cfg::kParts0) * G + h) * 32 + pair) * kDkRows + r0);
            auto put = [&](bool rest) __attribute__((always_inline)) {   // (the next part, and what its rounding leaves over as another)
              const uint32_t p1 = pack_bf16(v1[0], v1[1]), p2 = pack_bf16(v2[0], v2[1]);
              dst[0] = p1;
              dst[16 * kDkRows / 2] = p2;
              dst += G * 32 * kDkRows / 2;
              if (!rest) return;
              dst[0] = pack_bf16(v1[0] - bf16_lo(p1), v1[1] - bf16_hi(p1));
              dst[16 * kDkRows / 2] = pack_bf16(v2[0] - bf16_lo(p2), v2[1] - bf16_hi(p2));
              dst += G * 32 * kDkRows / 2;
            };
            const float w = slow_turn[u] * (6.2831853f * kDkReach);
            auto times_iw = [&](float f) __attribute__((always_inline)) {
#pragma unroll
              for (int x = 0; x < 2; ++x) {
                const float a = v1[x];
                v1[x] = -(v2[x] * (w * f));
                v2[x] = a * (w * f);
              }
            };
            put(true);
            if constexpr (u == 0) {   // cos z ~ 1 - a2 z^2 + a4 z^4, sin z ~ z - z^3 / 6 + a5 z^5
              constexpr float Z2 = kDkLow0 * kDkLow0, a4 = 1.f / 24.f - 1.5f * Z2 / 720.f, a2 = 0.5f - 0.5625f * Z2 * Z2 / 720.f;
              constexpr float a5 = 1.f / 120.f - 0.8f * Z2 / 5040.f;
              times_iw(1.f);
              put(true);
              times_iw(a2);
              put(true);
              times_iw(1.f / (6.f * a2));
              put(kEltIsF16);
              times_iw(6.f * a4);
              put(false);
              times_iw(a5 / a4);
              put(false);
            } else {                  // cos z ~ 1 - z^2 / 2, sin z ~ a1 z
              constexpr float a1 = 1.f - kDkLow1 * kDkLow1 / 8.f;
              times_iw(a1);
              put(true);
              times_iw(0.5f / a1);
              put(false);
            }
          });
        }
        __syncthreads();
      }
      if (i0 < jw) continue;   // wave-uniform: all keys of this wave lie above the diagonal of the tile's rows
      // gate path: dk += W^T qL over the tile's 8 rows.  W enters as three bf16 parts (24 bits, any range), an fp16 query as two.
      {
        float hi[8], mid[8], lo[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          const float wij = tile[(x * MATS + 1) * kDkKeys + 32 * wave + col];
          hi[x] = bf16_to_f(f_to_bf16(wij));
          const float rest = wij - hi[x];
          mid[x] = bf16_to_f(f_to_bf16(rest));
          lo[x] = rest - mid[x];
        }
        u32x4 a1, a2;   // contraction slots of half 0: hi, then lo; of half 1: mid, then nothing
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const uint32_t h2 = pack_bf16(hi[2 * x], hi[2 * x + 1]), m2 = pack_bf16(mid[2 * x], mid[2 * x + 1]);
          const uint32_t l2 = pack_bf16(lo[2 * x], lo[2 * x + 1]);
          a1[x] = hf == 0 ? h2 : m2;
          a2[x] = hf == 0 ? l2 : 0u;
        }
#pragma unroll
        for (int cb = 0; cb < 2 * NP + LOW; ++cb) {
          const uint16_t* ql = qT + dk_slot<D>(cb < NP ? 32 * cb + col : cb < 2 * NP ? HALF + 32 * (cb - NP) + col : slow_column(cb - 2 * NP)) * 8;
          u32x4 b1, b2;
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const uint32_t q2 = ql[2 * x * D * 8] | (uint32_t)ql[(2 * x + 1) * D * 8] << 16;
            b1[x] = kEltIsF16 ? pack_bf16(elt_lo(q2), elt_hi(q2)) : q2;
            if constexpr (kEltIsF16) b2[x] = pack_bf16(elt_lo(q2) - bf16_lo(b1[x]), elt_hi(q2) - bf16_hi(b1[x]));
          }
          f32x16& acc = cb < NP ? dk1[cb % NP] : cb < 2 * NP ? dk2[cb % NP] : slow[cb - 2 * NP];
          if constexpr (kEltIsF16) {
            acc = mfma32_bf16(a2, b2, acc);
            acc = mfma32_bf16(a1, b2, acc);
          }
          acc = mfma32_bf16(a2, b1, acc);
          acc = mfma32_bf16(a1, b1, acc);
        }
      }
      if constexpr (LOW > 0) {
        // the slow pairs: A = dS y^n, lane = (key, two heads), registers = the tile's rows
        float y[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) y[x] = (tile[x * MATS * kDkKeys + 32 * wave + col] - mids[x]) * (1.f / kDkReach);
#pragma unroll
        for (int h0 = 0; h0 < G; h0 += 2) {
          const int h = min(h0 + hf, G - 1);
          float a[8];
#pragma unroll
          for (int x = 0; x < 8; ++x) a[x] = h0 + hf < G ? tile[(x * MATS + 2 + h) * kDkKeys + 32 * wave + col] : 0.f;
          const uint16_t* bp = slow_q + (h * 32 + col) * kDkRows;
          auto part = [&](int n) __attribute__((always_inline)) { return *reinterpret_cast<const u32x4*>(bp + n * G * 32 * kDkRows); };
          u32x4 hi, lo;
          auto split = [&]() __attribute__((always_inline)) {
            hi = u32x4{pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(a[4], a[5]), pack_bf16(a[6], a[7])};
#pragma unroll
            for (int x = 0; x < 4; ++x) lo[x] = pack_bf16(a[2 * x] - bf16_lo(hi[x]), a[2 * x + 1] - bf16_hi(hi[x]));
          };
          auto times_y = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < 8; ++x) a[x] *= y[x];
          };
          auto full = [&](int u, int n) __attribute__((always_inline)) {   // with parts n and n + 1 of the group
            const u32x4 b = part(n), rest = part(n + 1);
            slow[u] = mfma32_bf16(hi, rest, slow[u]);
            slow[u] = mfma32_bf16(lo, b, slow[u]);
            slow[u] = mfma32_bf16(hi, b, slow[u]);
          };
          constexpr int C1 = Cfg::kParts0, F = kEltIsF16 ? 1 : 0;
          split();
          full(0, 0);
          if constexpr (LOW > 1) full(1, C1);
          times_y();
          split();
          full(0, 2);
          if constexpr (LOW > 1) full(1, C1 + 2);
          times_y();
          split();
          full(0, 4);
          if constexpr (LOW > 1) slow[1] = mfma32_bf16(hi, part(C1 + 4), slow[1]);
          times_y();
          split();
          if constexpr (kEltIsF16) full(0, 6);
          else slow[0] = mfma32_bf16(hi, part(6), slow[0]);
#pragma unroll
          for (int n = 4; n < 6; ++n) {
            times_y();
            split();
            slow[0] = mfma32_bf16(hi, part(n + 3 + F), slow[0]);
          }
        }
      }
      const int n_rows = min(kDkRows, N - i0);
      // dS of a row is read from LDS under the row before: what begins a row is a chain from there through the conversion and the product
      float ds_next[G];
      auto read_ds = [&](int r) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < G; ++h) ds_next[h] = tile[(r * MATS + 2 + h) * kDkKeys + 32 * wave + col];
      };
      read_ds(0);
#pragma unroll 1
      for (int r = 0; r < n_rows; ++r) {
        const float* trow = tile + r * MATS * kDkKeys + 32 * wave;
        // A: (32 keys x 16 contraction slots): lane (key, half 0) holds dS^h for h = 0..7 rounded to bf16, half 1 what the
        // rounding left over (again as bf16); with the queries of heads 0..7 in both halves of B the product carries dS to
        // about 16 bits
        u32x4 aop;
        {
          float dsv[8];
#pragma unroll
          for (int h = 0; h < 8; ++h) {
            const float x = h < G ? ds_next[h < G ? h : 0] : 0.f;
            dsv[h] = hf == 0 ? x : x - elt_to_f(f_to_elt(x));
          }
          aop = u32x4{pack_elts(dsv[0], dsv[1]), pack_elts(dsv[2], dsv[3]), pack_elts(dsv[4], dsv[5]), pack_elts(dsv[6], dsv[7])};
        }
        read_ds(min(r + 1, kDkRows - 1));
        // delta of this lane's 16 keys: keys 8 n + 4 half + 0..3 for n = 0..3, as the accumulator rows are laid out
        f32x4 dl[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) dl[n] = *reinterpret_cast<const f32x4*>(trow + 8 * n + 4 * hf);
        // B: (heads x 32 columns) per column block.  One rotation pair per pass (columns 32 np + col and the same + D/2), so that only two product blocks are live.
        static_for<NP>([&](auto np_c) __attribute__((always_inline)) {
          constexpr int np = decltype(np_c)::value;
          const u32x4 bq1 = *reinterpret_cast<const u32x4*>(qT + (r * D + dk_slot<D>(32 * np + col)) * 8);
          const u32x4 bq2 = *reinterpret_cast<const u32x4*>(qT + (r * D + HALF + dk_slot<D>(32 * np + col)) * 8);
          const f32x16 u1 = mfma32(aop, bq1, f32x16{0}), u2 = mfma32(aop, bq2, f32x16{0});
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float delta = dl[e / 4][e % 4];
            const float x = corope_phase<(np < REDUCED)>(delta * w_turn[np]);
            const float sn = __builtin_amdgcn_sinf(x), cs = __builtin_amdgcn_cosf(x);
            dk1[np][e] = __builtin_fmaf(cs, u1[e], __builtin_fmaf(-sn, u2[e], dk1[np][e]));
            dk2[np][e] = __builtin_fmaf(cs, u2[e], __builtin_fmaf(sn, u1[e], dk2[np][e]));
          }
        });
#pragma unroll
        for (int h = 0; h < G; ++h) asm volatile("" : "+v"(ds_next[h]));   // (or the read sinks to its use)
      }
    }
    const bool whole = t == b0 && seg_end == b1;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int j = jw + acc_row(e, hf);
      if (j < N) {
        uint16_t* op = p.dk + ((int64_t)g * N + j) * D;
        float* pp = parts + (int64_t)g * group_floats + sh.slot(share, t == b0) * (kDkKeys * D) + (j - jb) * D;
#pragma unroll
        for (int np = 0; np < NP; ++np) {
          if (whole) {
            op[32 * np + col] = f_to_elt(dk1[np][e] * p.sm_scale);
            op[32 * np + col + HALF] = f_to_elt(dk2[np][e] * p.sm_scale);
          } else {
            pp[32 * np + col] = dk1[np][e];
            pp[32 * np + col + HALF] = dk2[np][e];
          }
        }
#pragma unroll
        for (int u = 0; u < LOW; ++u) {
          if (whole)
            op[slow_column(u)] = f_to_elt(slow[u][e] * p.sm_scale);
          else
            pp[slow_column(u)] = slow[u][e];
        }
      }
    }
    t = seg_end;
  }
}

// ---------------------------------------------------------------------------------------------------- host side
int64_t corope_gqa_bwd_workspace_floats(int B, int Hq, int Hkv, int N, int D) {
  return tri_row_start(N) * (2 * (int64_t)B * Hkv + 3 * (int64_t)B * Hq) + (int64_t)B * Hkv * N * D;
}

// Workgroups per group of the kernels that cut a group's list into equal shares: as many as give every compute unit its two
// workgroups once (a second, partly filled round would leave units idle), from 128 groups on, where that is too coarse, four
// rounds' worth; no more than the tiles, nor than two slots each in the space for the partial sums.
template <int ROWS>
static int corope_bwd_shares(int N, int n_groups_total, int64_t slots) {
  const int places = 2 * device_cu_count();
  const int64_t want = places / n_groups_total >= 4 ? places / n_groups_total : (4 * places + n_groups_total - 1) / n_groups_total;
  return (int)std::max<int64_t>(1, std::min({want, slots / 2, (int64_t)CoropeShares<ROWS>(N).total}));
}

// Rows per wave of the scores kernel: as many as fill the 16 columns where that leaves two waves per SIMD twice over; below that
// fewer rows per wave give more waves.  Decided on the whole call's groups, so a smaller workspace gives the same bits.
template <int D, int G, int REDUCED>
static void launch_corope_bwd_scores(const CoropeBwdParams& p, const CoropeBwdWs& ws, const CoropeBwdFreqs& fr, int n_groups_total,
                                     hipStream_t stream) {
  constexpr int kMost = G <= 4 ? 4 : 2;
  const int64_t rows = (int64_t)p.N * n_groups_total, simds = 4 * device_cu_count();
  const int n_groups = p.B * p.Hkv;
  auto blocks = [&](int R) { return dim3((unsigned)((p.N + R - 1) / R) * n_groups); };
  if (kMost > 2 && rows >= 4 * simds * kMost)
    hipLaunchKernelGGL((corope_bwd_scores_kernel<D, G, kMost, REDUCED>), blocks(kMost), dim3(kWave), 0, stream, p, ws, fr);
  else if (rows >= 8 * simds)
    hipLaunchKernelGGL((corope_bwd_scores_kernel<D, G, 2, REDUCED>), blocks(2), dim3(kWave), 0, stream, p, ws, fr);
  else
    hipLaunchKernelGGL((corope_bwd_scores_kernel<D, G, 1, REDUCED>), blocks(1), dim3(kWave), 0, stream, p, ws, fr);
}

template <int D, int G, int REDUCED, int LOW>
static hipError_t launch_corope_bwd_dk(const CoropeBwdParams& p, const CoropeBwdWs& ws, const CoropeBwdFreqs& fr, float* parts, int shares,
                                       hipStream_t stream) {
  constexpr int kLdsBytes = CoropeDkCfg<D, G, LOW>::kLdsBytes;
  auto kern = corope_bwd_dk_kernel<D, G, REDUCED, LOW>;
  static std::atomic<uint64_t> lds_ok{0};
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), kLdsBytes, lds_ok); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(shares, p.B * p.Hkv), dim3(kDkWaves * kWave), kLdsBytes, stream, p, ws, fr, parts, G * ws.NN);
  return hipSuccess;
}

template <int D, int G, int REDUCED>
static hipError_t launch_corope_bwd_cfg(const CoropeBwdParams& p, const CoropeBwdWs& ws, const CoropeBwdFreqs& fr, int n_groups_total,
                                        hipStream_t stream) {
  launch_corope_bwd_scores<D, G, REDUCED>(p, ws, fr, n_groups_total, stream);
  const int64_t group_floats = G * ws.NN, slots = ws.part_floats(G, p.N) / (kDkKeys * D);
  const int dv_shares = corope_bwd_shares<kDvRows>(p.N, n_groups_total, slots), dk_shares = corope_bwd_shares<kDkRows>(p.N, n_groups_total, slots);
  float* parts = ws.parts(0, G);
  const int n_groups = p.B * p.Hkv, n_blocks = (p.N + kDkKeys - 1) / kDkKeys;
  const unsigned leader_blocks = (unsigned)((p.N + kLeaderRows - 1) / kLeaderRows) * n_groups;
  hipLaunchKernelGGL((corope_bwd_dv_kernel<D, G>), dim3(leader_blocks + (unsigned)dv_shares * n_groups), dim3(4 * kWave), 0, stream, p, ws,
                     parts, group_floats, dv_shares);
  if (dv_shares > 1)
    hipLaunchKernelGGL((corope_bwd_sum_kernel<D, kDvRows>), dim3(n_blocks, n_groups, 8), dim3(256), 0, stream, parts, group_floats, p.dv,
                       p.N, dv_shares, 1.f);
  constexpr int kLow = D == 128 && CoropeDkCfg<D, G, 2>::kLdsBytes <= 80 * 1024 ? 2 : 0;   // (two workgroups a compute unit: up to five heads, fp16: four)
  const hipError_t e = corope_low_groups(fr.turns, D) >= 2 ? launch_corope_bwd_dk<D, G, std::min(REDUCED, D / 64 - kLow / 2), kLow>(p, ws, fr, parts, dk_shares, stream)
                                                           : launch_corope_bwd_dk<D, G, REDUCED, 0>(p, ws, fr, parts, dk_shares, stream);
  if (e != hipSuccess) return e;
  if (dk_shares > 1)
    hipLaunchKernelGGL((corope_bwd_sum_kernel<D, kDkRows>), dim3(n_blocks, n_groups, 8), dim3(256), 0, stream, parts, group_floats, p.dk,
                       p.N, dk_shares, p.sm_scale);
  return hipGetLastError();
}

template <int D, int REDUCED>
static hipError_t launch_corope_bwd_d(const CoropeBwdParams& p, const CoropeBwdWs& ws, const CoropeBwdFreqs& fr, int n_groups_total,
                                      hipStream_t stream) {
  switch (p.Hq / p.Hkv) {
    case 1: return launch_corope_bwd_cfg<D, 1, REDUCED>(p, ws, fr, n_groups_total, stream);
    case 2: return launch_corope_bwd_cfg<D, 2, REDUCED>(p, ws, fr, n_groups_total, stream);
    case 3: return launch_corope_bwd_cfg<D, 3, REDUCED>(p, ws, fr, n_groups_total, stream);
    case 4: return launch_corope_bwd_cfg<D, 4, REDUCED>(p, ws, fr, n_groups_total, stream);
    case 5: return launch_corope_bwd_cfg<D, 5, REDUCED>(p, ws, fr, n_groups_total, stream);
    case 6: return launch_corope_bwd_cfg<D, 6, REDUCED>(p, ws, fr, n_groups_total, stream);
    case 7: return launch_corope_bwd_cfg<D, 7, REDUCED>(p, ws, fr, n_groups_total, stream);
    case 8: return launch_corope_bwd_cfg<D, 8, REDUCED>(p, ws, fr, n_groups_total, stream);
    default: return hipErrorInvalidValue;
  }
}

// One pass of the launch sequence handles `gc` (batch, key/value head) groups with gc * (2 + 3 G) packed matrices; a
// workspace smaller than the whole problem's is walked in passes of as many groups as fit (every group is independent:
// its queries' heads, its key/value head, its slices of dq, dk, dv).
hipError_t launch_corope_gqa_bwd(const CoropeBwdParams& p, int D, float* workspace, int64_t workspace_floats,
                                 hipStream_t stream) {
  CoropeBwdFreqs fr{};
  // theta^(-2d/D) evaluated like the reference's torch expression (fp32 exponent, fp32 power), as in the forward
  for (int d = 0; d < D / 2; ++d) {
    const float e = (float)(2 * d) / (float)D;
    const float inv = 1.0f / powf(p.theta, e);
    fr.rad[d] = inv;
    fr.turns[d] = (float)((double)inv / 6.283185307179586);
  }
  const int G = p.Hq / p.Hkv, n_groups = p.B * p.Hkv;
  const int64_t per_group = corope_gqa_bwd_workspace_floats(1, G, 1, p.N, D);
  // (the dk and the sum launches have a group per step of the second grid axis, which ends at 65535)
  const int per_pass = (int)std::min<int64_t>(std::min(n_groups, 65535), workspace_floats / per_group);
  if (per_pass < 1) return hipErrorInvalidValue;
  for (int g0 = 0; g0 < n_groups; g0 += per_pass) {
    const int gc = std::min(per_pass, n_groups - g0);
    CoropeBwdParams c = p;
    const int64_t qoff = (int64_t)g0 * G * p.N * D, koff = (int64_t)g0 * p.N * D;
    c.q += qoff;
    c.d_o += qoff;
    c.dq += qoff;
    if (c.o != nullptr) c.o += qoff;
    c.k += koff;
    c.v += koff;
    c.dk += koff;
    c.dv += koff;
    c.B = 1;
    c.Hkv = gc;
    c.Hq = gc * G;
    CoropeBwdWs ws{workspace, tri_row_start(p.N), gc, gc * G};
    const int reduced = corope_reduced_blocks(fr.turns, D, p.N);
    const hipError_t e = D == 64 ? (reduced == 0 ? launch_corope_bwd_d<64, 0>(c, ws, fr, n_groups, stream) : launch_corope_bwd_d<64, 1>(c, ws, fr, n_groups, stream))
                         : reduced == 0 ? launch_corope_bwd_d<128, 0>(c, ws, fr, n_groups, stream)
                         : reduced == 1 ? launch_corope_bwd_d<128, 1>(c, ws, fr, n_groups, stream)
                                        : launch_corope_bwd_d<128, 2>(c, ws, fr, n_groups, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace COROPE_NS
