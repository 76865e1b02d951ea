// sdpa_stage.hip -- the staged attention over an MLX affine cache (2-, 4- or
// 8-bit codes) on the matrix cores, for 16-bit queries and equal key and value
// head dims of 64, 96, 128 or 256: same arguments and same masks as
// sdpa_gen_kernel, which keeps the other head dims and fp32 queries.
//
// Nothing is rounded below fp32 on the way. Codes minus 2^(bits-1) are exact
// 16-bit operands, so with k = (c - off) * s + b', b' = b + off * s,
//     score = sum_g s_g * (q . (c - off))_g + b'_g * (sum q)_g
// takes exact products into fp32 per quantization group g (q as given, the
// sums and the scaling in fp32); and with f = p * s_g in fp32 split into three
// bf16 terms (8 bits each: hi + mid + lo = f),
//     out = sum_t f (c - off) + sum_t p b'_g
// takes three MFMAs per operand pair and one fp32 FMA per weight and group.
//
// A workgroup of 4 waves owns 128 consecutive (position, head) rows of one
// (sequence, KV head), 32 per wave, and walks 32-token blocks of its context
// split. A block's codes are decoded once per workgroup into LDS (K in the
// query type, V in bf16, rows padded so that an operand read's 16 tokens start
// on distinct banks) next to its scales and offsets in fp32; two buffers, one
// barrier per block. Both products run in the transposed orientation
//     S^T (16 tokens x 16 rows) = K (16 x 32 dims) . Q^T
//     O^T (16 dims x 16 rows)  += V^T (16 x 32 tokens) . P^T
// so a row's weights, its maximum and its sums never leave its lane, and the
// weights are the second product's operand where the first one left them.
//
// What bounds it: the VALU (per weight: the exponential, per group the scaling
// and the split, 13 operations; ten VALU instructions per MFMA in all). Two
// waves per SIMD overlap the two (head dim 128 G64, L = 512 over N = 4096: waves
// issue 51% of their time, MFMAs are busy 24%); head dim 256 has registers for
// one wave per SIMD. Registers spill at head dim 128 G32 (35 to 41 a lane), 256
// G32 (64) and 256 G64 (6). Additive masks are read one value at a time and
// cost half as much again (108 -> 171 us; boolean ones 134). Us per call with
// the merge, against the vector kernel (one workgroup per query row, whose LDS
// reads bound it): 32/8 heads of 128, L = 512 over N = 4096 causal, 4-bit G64
// 7400 -> 108, 8-bit G32 10650 -> 165; 16/4 heads of 256, 8-bit G32 10520 -> 241;
// 12/4 heads of 96, L = 300 of N = 1000, 2-bit 476 -> 30; one query token with a
// boolean mask array over N = 4096 68 -> 16, 12/4 heads of 96 over N = 300 52 ->
// 14. Relative error of the fp32 output against float64: 2e-7 .. 8e-7 (vector
// kernel 5e-7 .. 1.2e-6).
#include <algorithm>
#include <cfloat>

#include "sdpa_common.h"
#include "sdpa_gen.h"

namespace sparkq {

namespace {

constexpr int kStageRows = 128;  // (position, head) rows per workgroup

template <int D, int G>
struct StageLds {
  static constexpr int NG = D / G;
  static constexpr int KROW = 2 * D + 16, VROW = 2 * D + 32;  // bytes per token row
  static constexpr int V = 32 * KROW;
  static constexpr int META = V + 32 * VROW;  // [4: ks, kb', vs, vb'][NG][32] fp32
  static constexpr int BUF = META + 4 * NG * 32 * 4;
  static constexpr int BYTES = 2 * BUF;
};

template <typename T>
__device__ __forceinline__ f32x4_t mfma_qk(u32x4_t a, u32x4_t b, f32x4_t c);
template <>
__device__ __forceinline__ f32x4_t mfma_qk<BF16>(u32x4_t a, u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4_t mfma_qk<F16>(u32x4_t a, u32x4_t b, f32x4_t c) {
  return mfma16x16x32_f16(a, b, c);
}

// The sixteen codes of a piece (bits/2 words) minus 2^(bits-1), as floats.
__device__ __forceinline__ void stage_codes(const uint32_t w[4], int bits, float f[16]) {
  if (bits == 8) {
#pragma unroll
    for (int i = 0; i < 16; ++i) f[i] = (float)((w[i >> 2] >> (8 * (i & 3))) & 255u) - 128.0f;
  } else if (bits == 4) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t m = ((i & 1) ? w[i >> 3] >> 4 : w[i >> 3]) & 0x0F0F0F0Fu;
      f[i] = (float)((m >> (8 * ((i & 7) >> 1))) & 255u) - 8.0f;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t m = (w[0] >> (2 * (i & 3))) & 0x03030303u;
      f[i] = (float)((m >> (8 * (i >> 2))) & 255u) - 2.0f;
    }
  }
}

// the high halves (bf16 by truncation) of a pair
__device__ __forceinline__ uint32_t hi_pair(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float bf16_trunc(float v) {
  return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u);
}

__device__ __forceinline__ float stage_max_rows4(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float stage_sum_rows4(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int D, int G, typename T>
__global__ __launch_bounds__(256, D <= 128 ? 2 : 1) void sdpa_stage_kernel(GenSdpaArgs a) {
  using LY = StageLds<D, G>;
  constexpr int NG = LY::NG;
  constexpr int NK = D / 32;                       // QK k chunks
  constexpr int KPG = G / 32;                      // of them per group
  constexpr int NJ = D / 16;                       // PV dim tiles
  constexpr int JPG = G / 16;                      // of them per group
  constexpr int PIECES = 2 * D;                    // 16-code pieces of a K (or V) block
  constexpr int PPT = (PIECES + 255) / 256;
  constexpr int NMETA = 32 * NG;                   // (token, group) pairs of a block
  __shared__ __attribute__((aligned(16))) unsigned char smem[LY::BYTES];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, grp = lane >> 4;
  int bx, by;
  xcd_grid_item(kXcdDealt, bx, by);
  const int b = by / a.Hkv, kh = by - b * a.Hkv;
  const int gqa = a.Hq / a.Hkv;
  const int R = a.L * gqa;
  const int S = a.S;
  const int xt = bx / S, split = bx - xt * S;
  const int ntiles = (R + kStageRows - 1) / kStageRows;
  const bool causal = a.mask_kind == kMaskCausal;
  const int tile = causal ? ntiles - 1 - xt : xt;  // the longest tiles first
  const int rw0 = tile * kStageRows;
  // Tokens this tile walks: all of them, or under the causal mask up to its
  // last row's last visible one, provided that every row sees a token (a row
  // that sees none averages all N values).
  int n_end = a.N;
  if (causal && a.N - a.L + rw0 / gqa >= 0)
    n_end = min(a.N, a.N - a.L + min(rw0 + kStageRows - 1, R - 1) / gqa + 1);
  const int nb_all = (n_end + 31) / 32;
  const int ib0 = (int)((int64_t)split * nb_all / S), ib1 = (int)((int64_t)(split + 1) * nb_all / S);

  // this lane's rows (rows past R repeat the last one and are not stored)
  u32x4_t qb[2][NK];
  float qsum[2][NG];
  int lim[2];
  int64_t mrow[2];
  const float off = (float)(1 << (a.bits - 1));
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int rr = min(rw0 + 32 * wave + 16 * rt + n16, R - 1);
    const int l = rr / gqa, h = kh * gqa + rr - l * gqa;
    lim[rt] = causal ? a.N - a.L + l : a.N - 1;
    mrow[rt] = b * a.m_b + h * a.m_h + l * a.m_l;
    const uint16_t* qrow =
        reinterpret_cast<const uint16_t*>(a.q) + (((int64_t)b * a.Hq + h) * a.L + l) * D;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
      qb[rt][kk] = *reinterpret_cast<const u32x4_t*>(qrow + 32 * kk + 8 * grp);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      float s = 0.0f;
#pragma unroll
      for (int kk = g * KPG; kk < (g + 1) * KPG; ++kk)
#pragma unroll
        for (int i = 0; i < 4; ++i) s += lo16<T>(qb[rt][kk][i]) + hi16<T>(qb[rt][kk][i]);
      qsum[rt][g] = stage_sum_rows4(s) * a.scale_log2;
    }
  }
  const bool wlive = rw0 + 32 * wave < R;

  // staging: piece p = tid + 256 i is token p / (D/16), codes 16 (p % (D/16))
  // .. +16; loads past n_end read zeros through the bounded descriptors
  const int esz = 2;
  const rsrc_t rk = make_rsrc(a.kp + b * a.kp_b + kh * a.kp_h,
                              (uint32_t)(((int64_t)(n_end - 1) * a.kp_t + D * a.bits / 32) * 4));
  const rsrc_t rv = make_rsrc(a.vp + b * a.vp_b + kh * a.vp_h,
                              (uint32_t)(((int64_t)(n_end - 1) * a.vp_t + D * a.bits / 32) * 4));
  const int64_t ksb = (b * a.ks_b + kh * a.ks_h) * esz, vsb = (b * a.vs_b + kh * a.vs_h) * esz;
  const uint32_t ksz = (uint32_t)(((int64_t)(n_end - 1) * a.ks_t + NG) * esz);
  const uint32_t vsz = (uint32_t)(((int64_t)(n_end - 1) * a.vs_t + NG) * esz);
  const rsrc_t rks = make_rsrc(reinterpret_cast<const unsigned char*>(a.ks) + ksb, ksz);
  const rsrc_t rkb = make_rsrc(reinterpret_cast<const unsigned char*>(a.kb) + ksb, ksz);
  const rsrc_t rvs = make_rsrc(reinterpret_cast<const unsigned char*>(a.vs) + vsb, vsz);
  const rsrc_t rvb = make_rsrc(reinterpret_cast<const unsigned char*>(a.vb) + vsb, vsz);
  const int kpt = (int)a.kp_t * 4, vpt = (int)a.vp_t * 4, kst = (int)a.ks_t, vst = (int)a.vs_t;
  u32x4_t kcr[PPT], vcr[PPT];
  uint32_t ksr, kbr, vsr, vbr;
  // the scales of (token, group) pair tid: NG <= 8, so one pair per thread
  const int mt = tid / NG, mg = tid - mt * NG;
  auto piece_load = [&](rsrc_t r, int o) -> u32x4_t {
    if (a.bits == 8) return buf_load16(r, (uint32_t)o);
    if (a.bits == 4) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0);
      return u32x4_t{(uint32_t)v[0], (uint32_t)v[1], 0u, 0u};
    }
    return u32x4_t{(uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0), 0u, 0u, 0u};
  };
  auto load = [&](int t0) {
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      const int p = tid + 256 * i, tk = p / (D / 16), jb = p % (D / 16);
      kcr[i] = piece_load(rk, (t0 + tk) * kpt + 2 * a.bits * jb);
      vcr[i] = piece_load(rv, (t0 + tk) * vpt + 2 * a.bits * jb);
    }
    // tokens past the block (idle threads) and past n_end read zeros
    const bool live = tid < NMETA;
    ksr = buf_load2(rks, live ? (uint32_t)(((t0 + mt) * kst + mg) * 2) : kOob);
    kbr = buf_load2(rkb, live ? (uint32_t)(((t0 + mt) * kst + mg) * 2) : kOob);
    vsr = buf_load2(rvs, live ? (uint32_t)(((t0 + mt) * vst + mg) * 2) : kOob);
    vbr = buf_load2(rvb, live ? (uint32_t)(((t0 + mt) * vst + mg) * 2) : kOob);
  };
  auto stage = [&](unsigned char* buf) {
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      const int p = tid + 256 * i, tk = p / (D / 16), jb = p % (D / 16);
      if (PIECES % 256 != 0 && p >= PIECES) break;
      float f[16];
      uint32_t o[8], w[4] = {kcr[i].x, kcr[i].y, kcr[i].z, kcr[i].w};
      stage_codes(w, a.bits, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = pack_round<T>(f[2 * e], f[2 * e + 1]);  // exact
      u32x4_t* kd = reinterpret_cast<u32x4_t*>(buf + tk * LY::KROW + 32 * jb);
      kd[0] = u32x4_t{o[0], o[1], o[2], o[3]};
      kd[1] = u32x4_t{o[4], o[5], o[6], o[7]};
      w[0] = vcr[i].x;
      w[1] = vcr[i].y;
      w[2] = vcr[i].z;
      w[3] = vcr[i].w;
      stage_codes(w, a.bits, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = hi_pair(f[2 * e], f[2 * e + 1]);  // exact
      u32x4_t* vd = reinterpret_cast<u32x4_t*>(buf + LY::V + tk * LY::VROW + 32 * jb);
      vd[0] = u32x4_t{o[0], o[1], o[2], o[3]};
      vd[1] = u32x4_t{o[4], o[5], o[6], o[7]};
    }
    if (tid < NMETA) {
      float* m = reinterpret_cast<float*>(buf + LY::META) + mg * 32 + mt;
      const float ks = T::to_f32((uint16_t)ksr), vs = T::to_f32((uint16_t)vsr);
      m[0] = ks * a.scale_log2;
      m[NG * 32] = fmaf(off, ks, T::to_f32((uint16_t)kbr));
      m[2 * NG * 32] = vs;
      m[3 * NG * 32] = fmaf(off, vs, T::to_f32((uint16_t)vbr));
    }
  };

  // operand addresses of this lane: K token n16 (+16), chunk 4 kk + grp; V
  // token 4 grp + n16/4 (+16), dims 16 j + 4 (n16 % 4) .. +4
  const int ka = n16 * LY::KROW + grp * 16;
  const int va = LY::V + (4 * grp + (n16 >> 2)) * LY::VROW + 8 * (n16 & 3);

  float mrun[2] = {kNegInf, kNegInf}, zl[2] = {0.0f, 0.0f};
  float pe[2][NG];
  f32x4_t acc[2][NJ];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
    for (int g = 0; g < NG; ++g) pe[rt][g] = 0.0f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[rt][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }

  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
  auto compute = [&](const unsigned char* buf, int t0) {
    const float* meta = reinterpret_cast<const float*>(buf + LY::META) + 4 * grp;
    float s[2][8];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int i = 0; i < 8; ++i) s[rt][i] = 0.0f;
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        f32x4_t sc[2] = {f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
        for (int kk = g * KPG; kk < (g + 1) * KPG; ++kk) {
          const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(buf + ka + 64 * kk + tt * 16 * LY::KROW);
          sc[0] = mfma_qk<T>(kf, qb[0][kk], sc[0]);
          sc[1] = mfma_qk<T>(kf, qb[1][kk], sc[1]);
        }
        const f32x4_t ks = *reinterpret_cast<const f32x4_t*>(meta + g * 32 + 16 * tt);
        const f32x4_t kb = *reinterpret_cast<const f32x4_t*>(meta + (NG + g) * 32 + 16 * tt);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            s[rt][4 * tt + r] = fmaf(ks[r], sc[rt][r], fmaf(kb[r], qsum[rt][g], s[rt][4 * tt + r]));
      }
    // masks; tokens past the tile's end weigh nothing
    if (a.mask_kind == kMaskBool) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        unsigned char mv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int n = min(t0 + 16 * (i >> 2) + 4 * grp + (i & 3), a.N - 1);
          mv[i] = reinterpret_cast<const unsigned char*>(a.mask)[mrow[rt] + n * a.m_n];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) s[rt][i] = mv[i] ? s[rt][i] : a.masked;
      }
    } else if (a.mask_kind == kMaskAdd) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int n = min(t0 + 16 * (i >> 2) + 4 * grp + (i & 3), a.N - 1);
          // a dtype-minimum mask stays finite (its product would overflow)
          s[rt][i] += fmaxf(load_in(a.mask, mrow[rt] + n * a.m_n, a.mask_dtype) * 1.4426950408889634f,
                            -FLT_MAX);
        }
    }
    // (a block that every row of the wave sees whole needs no comparison)
    const bool edge = t0 + 31 > min(lim[0], lim[1]) || t0 + 32 > n_end;
    if (__builtin_amdgcn_ballot_w64(edge) != 0) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int n = t0 + 16 * (i >> 2) + 4 * grp + (i & 3);
          s[rt][i] = n > lim[rt] ? a.masked : s[rt][i];
          s[rt][i] = n >= n_end ? kNegInf : s[rt][i];
        }
    }
    // The running maximum of a row moves when a block's maximum exceeds it by
    // more than 8 (log2 units): the weights stay below 2^8 and the
    // accumulators are rescaled (a wave-uniform branch) in few blocks.
    float p[2][8], alpha[2];
    bool up[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      float mb = fmaxf(fmaxf(fmaxf(s[rt][0], s[rt][1]), fmaxf(s[rt][2], s[rt][3])),
                       fmaxf(fmaxf(s[rt][4], s[rt][5]), fmaxf(s[rt][6], s[rt][7])));
      mb = stage_max_rows4(mb);
      up[rt] = mb > mrun[rt] + 8.0f;
      alpha[rt] = up[rt] ? exp2_guarded(mrun[rt] - mb, mrun[rt] != kNegInf) : 1.0f;
      mrun[rt] = up[rt] ? mb : mrun[rt];
      // nothing but -inf scores yet: their weights are 0, not 2^(-inf + inf)
      const float mu = mrun[rt] == kNegInf ? 0.0f : mrun[rt];
      float ps = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[rt][i] = __builtin_amdgcn_exp2f(s[rt][i] - mu);
        ps += p[rt][i];
      }
      zl[rt] = fmaf(zl[rt], alpha[rt], ps);
    }
    if (__builtin_amdgcn_ballot_w64(up[0] || up[1]) != 0) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[rt][j] *= alpha[rt];
#pragma unroll
        for (int g = 0; g < NG; ++g) pe[rt][g] *= alpha[rt];
      }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      u32x4_t ph[2], pm[2], pl[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const f32x4_t vs = *reinterpret_cast<const f32x4_t*>(meta + (2 * NG + g) * 32 + 16 * tt);
        const f32x4_t vb = *reinterpret_cast<const f32x4_t*>(meta + (3 * NG + g) * 32 + 16 * tt);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          float f[4], r1[4], r2[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float pr = p[rt][4 * tt + r];
            pe[rt][g] = fmaf(pr, vb[r], pe[rt][g]);
            f[r] = pr * vs[r];
            r1[r] = f[r] - bf16_trunc(f[r]);    // exact
            r2[r] = r1[r] - bf16_trunc(r1[r]);  // exact, at most 8 bits left
          }
          ph[rt][2 * tt] = hi_pair(f[0], f[1]);
          ph[rt][2 * tt + 1] = hi_pair(f[2], f[3]);
          pm[rt][2 * tt] = hi_pair(r1[0], r1[1]);
          pm[rt][2 * tt + 1] = hi_pair(r1[2], r1[3]);
          pl[rt][2 * tt] = hi_pair(r2[0], r2[1]);
          pl[rt][2 * tt + 1] = hi_pair(r2[2], r2[3]);
        }
      }
#pragma unroll
      for (int j = g * JPG; j < (g + 1) * JPG; ++j) {
        const unsigned char* vp = buf + va + 32 * j;
        const u32x2_t lo = __builtin_bit_cast(
            u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(vp)));
        const u32x2_t hi = __builtin_bit_cast(
            u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                         (__attribute__((address_space(3))) s16x4_t*)(vp + 16 * LY::VROW)));
        const u32x4_t vf = u32x4_t{lo.x, lo.y, hi.x, hi.y};
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          acc[rt][j] = mfma_qk<BF16>(vf, pl[rt], acc[rt][j]);
          acc[rt][j] = mfma_qk<BF16>(vf, pm[rt], acc[rt][j]);
          acc[rt][j] = mfma_qk<BF16>(vf, ph[rt], acc[rt][j]);
        }
      }
    }
  };

  if (ib0 < ib1) {
    load(32 * ib0);
    stage(smem);
    load(32 * ib0 + 32);
    __syncthreads();
    for (int ib = ib0; ib < ib1; ++ib) {
      const int t0 = 32 * ib, cur = (ib - ib0) & 1;
      if (wlive) compute(smem + cur * LY::BUF, t0);
      stage(smem + (cur ^ 1) * LY::BUF);
      load(t0 + 64);
      __syncthreads();
    }
  }

  // O^T lane (grp, n16): row n16, dims 16 j + 4 grp + r
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const float z = stage_sum_rows4(zl[rt]);
#pragma unroll
    for (int g = 0; g < NG; ++g) pe[rt][g] = stage_sum_rows4(pe[rt][g]);
    const int rr = rw0 + 32 * wave + 16 * rt + n16;
    if (rr >= R) continue;
    const int l = rr / gqa, h = kh * gqa + rr - l * gqa;
    const int64_t row = ((int64_t)b * a.Hq + h) * a.L + l;
    if (S > 1) {
      if (grp == 0) {
        a.pm[row * S + split] = mrun[rt];
        a.pz[row * S + split] = z;
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        *reinterpret_cast<f32x4_t*>(a.pacc + (row * S + split) * D + 16 * j + 4 * grp) =
            acc[rt][j] + pe[rt][j / JPG];
      continue;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      f32x4_t o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (acc[rt][j][r] + pe[rt][j / JPG]) / z;
      const int64_t idx = row * D + 16 * j + 4 * grp;
      if (a.out_dtype == SPARKQ_F32)
        *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(a.out) + idx) = o;
      else
        *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(a.out) + idx) =
            u32x2_t{pack_round<T>(o[0], o[1]), pack_round<T>(o[2], o[3])};
    }
  }
}

template <int D, int G>
void launch_stage_t(const GenSdpaArgs& a, dim3 grid, hipStream_t st) {
  if (a.q_dtype == SPARKQ_BF16)
    hipLaunchKernelGGL((sdpa_stage_kernel<D, G, BF16>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((sdpa_stage_kernel<D, G, F16>), grid, dim3(256), 0, st, a);
}
template <int D>
void launch_stage_g(const GenSdpaArgs& a, dim3 grid, hipStream_t st) {
  if (a.G == 32) {
    launch_stage_t<D, 32>(a, grid, st);
  } else if constexpr (D % 64 == 0) {
    if (a.G == 64) {
      launch_stage_t<D, 64>(a, grid, st);
    } else if constexpr (D % 128 == 0) {
      launch_stage_t<D, 128>(a, grid, st);
    }
  }
}

}  // namespace

// Context splits: two workgroups per CU over the row tiles (two waves per SIMD,
// so that one's softmax overlaps the other's products), at least two 32-token
// blocks each. Us for 256 / 512 / 768 workgroups: 32/8 heads of 128, L = 512
// over N = 4096 155 / 108 / 121. Head dim 256, where a CU holds one workgroup,
// takes two rounds of them: 16/4 heads, L = 512 over N = 2048 129 / 139 / 166, over
// 512 43 / 51 / 51, L = 100 over 4096 62 / 72 / 91.
int sdpa_stage_splits(int64_t B, int64_t Hq, int64_t Hkv, int64_t L, int64_t N) {
  const int64_t items = cdiv(L * (Hq / Hkv), kStageRows) * B * Hkv;
  const int64_t S = std::min<int64_t>(cdiv(512, items), std::max<int64_t>(N / 64, 1));
  return (int)std::min<int64_t>(S, 128);
}

// 16-bit queries and one head dim of 64/96/128/256
bool sdpa_stage_dims(int qdt, int64_t D, int64_t Dv) {
  return (qdt == SPARKQ_BF16 || qdt == SPARKQ_F16) && D == Dv &&
         (D == 64 || D == 96 || D == 128 || D == 256);
}

// ..., 16-byte aligned q and out and a context whose byte offsets fit 31 bits;
// groups that divide the head dim.
bool sdpa_stage_ok(const GenSdpaArgs& a) {
  if (!sdpa_stage_dims(a.q_dtype, a.D, a.Dv)) return false;
  if (!aligned(a.q, 16) || !aligned(a.out, 16)) return false;
  const int64_t lim = (int64_t)1 << 31;
  const int64_t n = (int64_t)a.N + 96;  // the loads run up to two blocks ahead
  if (n * a.kp_t * 4 >= lim || n * a.vp_t * 4 >= lim) return false;
  if (n * a.ks_t * 2 >= lim || n * a.vs_t * 2 >= lim) return false;
  return (int64_t)a.L * (a.Hq / a.Hkv) + kStageRows < lim;
}

int launch_sdpa_stage(const GenSdpaArgs& a, hipStream_t st) {
  const int64_t ntiles = cdiv((int64_t)a.L * (a.Hq / a.Hkv), kStageRows);
  const dim3 grid((unsigned)(ntiles * a.S), (unsigned)(a.B * a.Hkv));
  if (a.D == 64)
    launch_stage_g<64>(a, grid, st);
  else if (a.D == 96)
    launch_stage_g<96>(a, grid, st);
  else if (a.D == 128)
    launch_stage_g<128>(a, grid, st);
  else
    launch_stage_g<256>(a, grid, st);
  return check_launch("sdpa_stage_kernel");
}

}  // namespace sparkq
