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
// Three restatements keep the work down.  (1) delta is a suffix sum that starts at the diagonal, so key chunks are
// swept right to left and delta accumulates directly: the reference's extra pass over all keys (:103-135) and the
// cancellation in a[i,i] - a[i,j] disappear (online softmax does not care about chunk order).  (2) The angle is
// shared by the whole group, so the key is rotated once per (i, j, d) - the only place sines and cosines are evaluated.
// (3) Everything that is a dot product with a key or value row runs on the matrix cores: the leader logits q_leader K^T (bf16 x
// bf16: exact products), the scores q^h Kt^T and O^T += V^T P^T.  The rotated keys are rounded to fp16, not bf16, and the score
// product runs in fp16 (the bf16 queries convert exactly): 11 significant bits keep the scores as accurate as the bf16 rounding of P
// afterwards, also at sm_scale = 1 where a bf16 key would cost several percent of a weight.
//
// Mapping: a wave owns R query rows of one (batch, kv head) group; four waves share a workgroup and the K and V tiles of 64 keys
// it stages in LDS, sweeping from the diagonal to key 0.  Everything is laid out for 16x16x32 MFMAs with the R x G (row, head)
// pairs as the 16 columns:
//   logits   A = leaders (row m of A is the leader of query row m R / 16), B = keys: lane (key % 16, row group) finds the logits
//            of its own rows in its own registers; gates and their suffix sums run along the 16 lanes of a DPP row and then over the
//            four 16-key blocks in registers; delta crosses the lanes once, through LDS.
//   rotation lane (key % 16, g) holds columns 8 g .. 8 g + 7 of every 32 of its key, both halves of each rotation pair, exactly as the
//            A operand of the score product wants them: the rotated keys never leave the registers.  Keys are unpacked once for all R rows.
//   scores   S^T = Kt Q^T per row: all 16 columns are multiplied, the row's own G are taken over.  The accumulators of the R rows
//            together are one full tile: lane = (row, head), registers = 16 keys of the chunk, so the softmax has no idle lane and its
//            row statistics are one register per lane.
//   O^T += V^T P^T  for all R rows at once; P is the B operand as the scores left it (the keys of a contraction step in accumulator
//            order, V read transposed in the same order).
// What bounds it: the vector units, 9 or 10 issue slots per (row, key, pair) -- one multiply, a range reduction where the phase can leave
// the sine unit's domain (REDUCED: in that many blocks of 32 pairs), sine and cosine at two slots each, two multiplies, two multiply-adds
// that round to fp16 -- of about 11.5 in all.  Measured at B2 Hq32 Hkv8 N4096 D128: 5.37 -> 3.20 ms (3.33 with every phase reduced; before, one wave per
// row, the rotated keys through LDS: 14 slots per pair, the keys four times through LDS and a softmax per head over the lanes),
// B1 Hq32 Hkv8 N1111 D128 fp16 224 -> 145 us (152 with every phase reduced), B2 Hq8 Hkv2 N512 D64 20.9 -> 18.4 us.
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
  static constexpr int kDeltaFloats = 4 * R * 16;                            // per wave: [16-key block][row][key % 16]
  static constexpr int kLdsBytes = 2 * kTileElems * 2 + kCoropeWaves * kDeltaFloats * 4;
  static_assert(2 * kLdsBytes <= 160 * 1024, "two workgroups per compute unit");
};

// (At D = 64 the registers allow more than two waves per SIMD: with several rows per wave that is 4 % faster, B2 Hq16 Hkv16 N2688
// 1458 -> 1397 us; with one, where the longest rows set the time, 7 % slower, B1 Hq2 Hkv1 N4096 173 -> 185 us.)
template <int D, int G, int R, int REDUCED>
__global__ __launch_bounds__(kCoropeWaves* kWave) __attribute__((amdgpu_waves_per_eu(2, R == 1 ? 2 : 8))) void corope_gqa_fwd_kernel(CoropeParams p,
                                                                                                       CoropeFreqs fr) {
  using Cfg = CoropeFwdCfg<D, R>;
  constexpr int KS = Cfg::kKStride, VS = Cfg::kVStride, NT = kCoropeWaves * kWave, PIECES = D / 8;
  constexpr int NKS = D / 32, HK = D / 64, NOB = D / 16, PER = kCoropeKeys * PIECES / NT;
  constexpr int ZR = R > 4 ? R / 4 : 1;     // query rows whose gates a lane holds
  static_assert(R * G <= 16 && 64 % (kCoropeWaves * R) == 0, "columns of a product; a workgroup's rows lie in one chunk");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int n = lane % 16, g = lane / 16;   // matrix-core identity: A row / B column, contraction group
  uint16_t* const tiles = reinterpret_cast<uint16_t*>(smem);
  float* const dbuf = reinterpret_cast<float*>(smem + 2 * Cfg::kTileElems * 2) + wave * Cfg::kDeltaFloats;

  const int n_groups = p.B * p.Hkv;
  const int grp = blockIdx.x % n_groups;
  const int i0 = (p.num_m_blocks - 1 - (int)(blockIdx.x / n_groups)) * (kCoropeWaves * R);   // longest rows first
  const int N = p.N, iw = i0 + wave * R;
  const int head0 = (grp / p.Hkv) * p.Hq + (grp % p.Hkv) * G;
  const uint16_t* kbase = p.k + (int64_t)grp * N * D;
  const uint16_t* vbase = p.v + (int64_t)grp * N * D;
  const int n_chunks = i0 / kCoropeKeys + 1;
  const float scale2 = p.sm_scale * 1.4426950408889634f;               // scores in the base-2 domain

  // column n of the score product: (query row, head) = (iw + n / G, n % G); columns from R G on are idle
  const int crow = n < R * G ? n / G : 0, chead = n < R * G ? n % G : 0;
  u32x4 qop[NKS], lop[NKS];   // B operand of the score product (fp16), A operand of the logit product (element type)
  {
    const uint16_t* qrow = p.q + ((int64_t)(head0 + chead) * N + min(iw + crow, N - 1)) * D + 8 * g;
    const uint16_t* lrow = p.q + ((int64_t)head0 * N + min(iw + n * R / 16, N - 1)) * D + 8 * g;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const u32x4 raw = *reinterpret_cast<const u32x4*>(qrow + 32 * ks);
#pragma unroll
      for (int e = 0; e < 4; ++e) qop[ks][e] = n < R * G ? pack_f16(elt_lo(raw[e]), elt_hi(raw[e])) : 0u;
      lop[ks] = *reinterpret_cast<const u32x4*>(lrow + 32 * ks);
    }
  }
  float turns[HK][8];         // w_d / 2 pi of this lane's columns d = 32 hk + 8 g + e
#pragma unroll
  for (int hk = 0; hk < HK; ++hk)
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(fr.w + 32 * hk + 8 * g + e);
#pragma unroll
      for (int x = 0; x < 4; ++x) turns[hk][e + x] = t[x];
    }

#pragma unroll
  for (int hk = 0; hk < HK; ++hk)
#pragma unroll
    for (int e = 0; e < 8; ++e) asm volatile("" ::"v"(turns[hk][e]));   // landed before the loop: left to their first use, the wait sits in it

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
  park(0);
  __syncthreads();
  int buf = 0;
#pragma unroll 1
  for (int c = n_chunks - 1; c >= 0; --c) {
    if (c > 0) fetch(c - 1, std::false_type{});
    const uint16_t* kt = tiles + buf * Cfg::kTileElems;
    const uint16_t* vt = kt + kCoropeKeys * KS;
    const bool diagonal = c == n_chunks - 1;   // wave-uniform

    // ---- leader logits, gates, delta: lane (key 16 b + n, query rows (4 g + e) R / 16) -------------------------------------
    {
      f32x4 lg[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        lg[b] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
          lg[b] = mfma16(lop[ks], *reinterpret_cast<const u32x4*>(kt + (16 * b + n) * KS + 32 * ks + 8 * g), lg[b]);
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
        carry[z] = right;
      }
    }
    lds_order();

    // ---- rotated keys and scores: 16 keys at a time ---------------------------------------------------------------------
    f32x4 sacc[4];
    static_for<4>([&](auto b_c) __attribute__((always_inline)) {
      constexpr int b = decltype(b_c)::value;
      float k1[HK][8], k2[HK][8];
#pragma unroll
      for (int hk = 0; hk < HK; ++hk) {
        const u32x4 x1 = *reinterpret_cast<const u32x4*>(kt + (16 * b + n) * KS + 32 * hk + 8 * g);
        const u32x4 x2 = *reinterpret_cast<const u32x4*>(kt + (16 * b + n) * KS + D / 2 + 32 * hk + 8 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          k1[hk][2 * e] = elt_lo(x1[e]);
          k1[hk][2 * e + 1] = elt_hi(x1[e]);
          k2[hk][2 * e] = elt_lo(x2[e]);
          k2[hk][2 * e + 1] = elt_hi(x2[e]);
        }
      }
      float delta = dbuf[b * R * 16 + n];
#pragma unroll 1
      for (int r = 0; r < R; ++r) {
        const float delta_r = delta;
        delta = dbuf[(b * R + min(r + 1, R - 1)) * 16 + n];
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
          acc = mfma16_f16(__builtin_bit_cast(u32x4, y1), qop[hk], acc);
          acc = mfma16_f16(__builtin_bit_cast(u32x4, y2), qop[HK + hk], acc);
        });
#pragma unroll
        for (int e = 0; e < 4; ++e) sacc[b][e] = crow == r ? acc[e] : sacc[b][e];
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

template <int D, int G, int R, int REDUCED>
static hipError_t launch_corope_rows(CoropeParams p, const CoropeFreqs& fr, hipStream_t stream) {
  using Cfg = CoropeFwdCfg<D, R>;
  auto kern = corope_gqa_fwd_kernel<D, G, R, REDUCED>;
  static std::atomic<uint64_t> lds_ok{0};
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes, lds_ok); e != hipSuccess) return e;
  p.num_m_blocks = (p.N + kCoropeWaves * R - 1) / (kCoropeWaves * R);
  hipLaunchKernelGGL(kern, dim3((unsigned)p.num_m_blocks * p.B * p.Hkv), dim3(kCoropeWaves * kWave), Cfg::kLdsBytes, stream, p, fr);
  return hipGetLastError();
}

template <int D, int G, int REDUCED>
static hipError_t launch_corope_cfg(const CoropeParams& p, const CoropeFreqs& fr, hipStream_t stream) {
  // Rows per wave: as many as fill the 16 columns where that leaves four waves per SIMD, of which two run at a time; below that
  // the longest rows, whose chunks follow one after the other, set the time, and fewer rows per wave shorten it.  us with four / two /
  // one row per wave at D = 128, fp16 B1 Hq32 Hkv8 N1111 171 / 143 / 179, bf16 B2 Hq16 Hkv4 N1024 152 / 122 / 153 and N2048 418 / 466 / 582;
  // at D = 64, B2 Hq8 Hkv2 N512 39 / 24 / 18.
  constexpr int kMost = G <= 2 ? 8 : G <= 4 ? 4 : 2;
  const int64_t rows = (int64_t)p.N * p.B * p.Hkv, simds = 4 * device_cu_count();
  if (rows >= 4 * simds * kMost) return launch_corope_rows<D, G, kMost, REDUCED>(p, fr, stream);
  if (kMost > 2 && rows >= 8 * simds) return launch_corope_rows<D, G, 2, REDUCED>(p, fr, stream);
  return launch_corope_rows<D, G, 1, REDUCED>(p, fr, stream);
}

template <int D, int REDUCED>
static hipError_t launch_corope_d(const CoropeParams& p, const CoropeFreqs& fr, hipStream_t stream) {
  switch (p.Hq / p.Hkv) {
    case 1: return launch_corope_cfg<D, 1, REDUCED>(p, fr, stream);
    case 2: return launch_corope_cfg<D, 2, REDUCED>(p, fr, stream);
    case 3: return launch_corope_cfg<D, 3, REDUCED>(p, fr, stream);
    case 4: return launch_corope_cfg<D, 4, REDUCED>(p, fr, stream);
    case 5: return launch_corope_cfg<D, 5, REDUCED>(p, fr, stream);
    case 6: return launch_corope_cfg<D, 6, REDUCED>(p, fr, stream);
    case 7: return launch_corope_cfg<D, 7, REDUCED>(p, fr, stream);
    case 8: return launch_corope_cfg<D, 8, REDUCED>(p, fr, stream);
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
  const int reduced = corope_reduced_blocks(fr.w, D, p.N);
  if (D == 64) return reduced == 0 ? launch_corope_d<64, 0>(p, fr, stream) : launch_corope_d<64, 1>(p, fr, stream);
  return reduced == 0   ? launch_corope_d<128, 0>(p, fr, stream)
         : reduced == 1 ? launch_corope_d<128, 1>(p, fr, stream)
                        : launch_corope_d<128, 2>(p, fr, stream);
}

}  // namespace COROPE_NS
