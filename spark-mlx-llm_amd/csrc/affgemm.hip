// affgemm.hip -- matmul over groupwise affine weights whose scales do not fit
// into a 16-bit operand: 4-bit weights of float16 checkpoints (from 33 rows)
// and 8-bit weights with scales of any dtype (any number of rows). With the
// codes centred, c = q - 2^(bits-1) and b' = b + 2^(bits-1) s,
//   y[m,n] = sum_g s[n,g] * (sum_{k in g} x[m,k] c[n,k]) + b'[n,g] * X[m,g],
// X[m,g] the sum of x over group g. Nothing is rounded below fp32: centred
// codes are exact 16-bit operands, the products of a group accumulate in fp32
// on the 32x32x16 MFMA, each group's sum enters y with one fp32 FMA by its
// scale, and its bias part follows at once on the fp32 MFMA (32x32x1, two
// blocks). A running sum of the scale parts alone would reach hundreds of
// times the result before the bias parts cancel it. Relative error of the fp32
// output against float64, activations of mean 0 / mean 1: fp16 4-bit
// 512 x 3584 x 2560 G64 1.6e-7 / 1.7e-7, 333 x 2560 x 9728 G32 2.3e-7 / 2.3e-7,
// bf16 8-bit 512 x 3584 x 2560 G64 1.6e-7 / 1.7e-7 (uncentred codes, group by
// group 1.8e-7 / 5.9e-7; uncentred with all bias parts last 4.3e-7 / 1.0e-5).
//
// affine_prep_kernel turns scales and biases into fp32 [K/G][N] (a wave's 32
// columns in one 128-byte line; in [N][K/G] order each of them costs a line of
// its own at every group) and sums the activations to X[K/G][M].
//
// affine_gemm_kernel: a workgroup of 4 waves owns a 64 x 128 tile, each
// wave 64 rows x 32 columns, and walks K in units of 128, a whole number of
// groups, so that a weight row is read in runs of 64 (4-bit) or 128 (8-bit)
// bytes. Activations go through LDS (rows of 16 chunks of 16 bytes, chunk c of
// row r at c ^ (r & 15): operand reads of 16 rows touch every bank once), each
// wave loads its own codes into registers and decodes them there; the loads of
// unit u+2 go out in unit u. The compiler places them late in the unit, and
// the scales (of bf16 8-bit weights some codes too) move to other registers at
// the end of every second unit, which waits for loads just issued. Where the
// tiles do not fill the chip, pieces of K go to workgroups of their own and
// affine_sum_kernel adds their fp32 sums in order.
//
// What bounds it: the latency of the units' chain and the decode beside it: at
// one workgroup per CU (8-bit 512 x 3584 x 2560) a unit takes 1.7 us, waves wait
// 35% of the time, issue VALU 31%, and MFMAs are busy 12%; at two (4-bit 333 x
// 2560 x 9728) 1.8 us, 32%, 26% and 21%. Of the calls' time 8 to 14 us go to the
// prologue and the sum of the pieces. 64 columns per wave, which would halve
// the LDS reads, have no registers for it and measured 0-20% slower. 4-bit instances fit three workgroups on a CU, 8-bit
// ones two. Per call, against the kernels this replaced: fp16 4-bit 333 x 2560 x
// 9728 G128 234 -> 45 us, 512 x 3584 x 2560 G64 68 -> 34, 2048 x 19456 x 2560
// G64 371 -> 314 (650 TFLOP/s); bf16 8-bit 512 x 3584 x 2560 G64 104 -> 39,
// 700 x 19456 x 2560 G32 1258 -> 180.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace sparkq {

namespace {

struct AffPrepArgs {
  const uint16_t* x;   // [M][K]
  const void* sc;      // [N][ng] in the scale dtype
  const void* bi;
  float* st;           // [ngp][N]
  float* bt;           // [ngp][N]: b + centre * s
  float* xs;           // [ngp][M]
  int M, N, K, G, s_dtype;
  int ngp;             // groups of whole units; those past K are zeros
  float centre;        // of the codes: 8 or 128
  int wblocks;         // blocks of the weight half (dispatched first)
};

// Weight blocks: 64 rows x 32 groups through LDS, read along the groups and
// written along the rows. Activation blocks: 16-byte chunks in order, the G/8
// lanes of a group add their sums by a butterfly.
template <typename T>
__global__ __launch_bounds__(256) void affine_prep_kernel(AffPrepArgs a) {
  __shared__ float ts[32][65], tb[32][65];
  const int tid = threadIdx.x, ng = a.K / a.G;
  if ((int)blockIdx.x < a.wblocks) {
    const int gb = (a.ngp + 31) / 32;
    const int n0 = (int)blockIdx.x / gb * 64, g0 = (int)blockIdx.x % gb * 32;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int n = n0 + (tid >> 5) + 8 * i, g = g0 + (tid & 31);
      const bool live = n < a.N && g < ng;
      const int64_t at = live ? (int64_t)n * ng + g : 0;
      const float sc = load_in(a.sc, at, a.s_dtype), bi = load_in(a.bi, at, a.s_dtype);
      ts[tid & 31][(tid >> 5) + 8 * i] = live ? sc : 0.0f;
      tb[tid & 31][(tid >> 5) + 8 * i] = live ? fmaf(a.centre, sc, bi) : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int gl = (tid >> 6) + 4 * i, n = n0 + (tid & 63), g = g0 + gl;
      if (n < a.N && g < a.ngp) {
        a.st[(int64_t)g * a.N + n] = ts[gl][tid & 63];
        a.bt[(int64_t)g * a.N + n] = tb[gl][tid & 63];
      }
    }
    return;
  }
  // (a row holds whole groups, so the lanes of a group are active together)
  const int64_t c = (int64_t)((int)blockIdx.x - a.wblocks) * 256 + tid;
  const int nc = a.K / 8;
  if (c >= (int64_t)a.M * nc) return;
  const u32x4_t v = reinterpret_cast<const u32x4_t*>(a.x)[c];
  float f[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) f[e] = lo16<T>(v[e]) + hi16<T>(v[e]);
  float s = (f[0] + f[1]) + (f[2] + f[3]);
  const int cpg = a.G / 8;  // 4, 8 or 16 consecutive lanes
  for (int o = 1; o < cpg; o <<= 1) s += __shfl_xor(s, o);
  const int m = (int)(c / nc), cc = (int)(c - (int64_t)m * nc);
  if ((cc & (cpg - 1)) == 0) a.xs[(int64_t)(cc / cpg) * a.M + m] = s;
  if (cc == nc - 1)
    for (int g = ng; g < a.ngp; ++g) a.xs[(int64_t)g * a.M + m] = 0.0f;
}

struct AffGemmArgs {
  const uint16_t* x;   // [M][K]
  const uint32_t* w;   // [N][K*BITS/32]
  const float* st;     // [ngp][N]
  const float* bt;     // [ngp][N], b + centre * s
  const float* xs;     // [ngp][M]
  void* y;             // [M][N]
  float* part;         // [S][M][N] when S > 1
  int y_dtype, M, N, K, tiles_m, tiles_n, S;
};

typedef float f32x32_t __attribute__((ext_vector_type(32)));

constexpr int kAffBM = 64, kAffBN = 128, kAffBK = 128;

// a chunk's 8 codes minus 2^(BITS-1) as exact 16-bit values in k order
template <typename T, int BITS>
__device__ __forceinline__ u32x4_t aff_decode(const uint32_t* w, DecodeConsts dc) {
  u32x4_t r;
  if constexpr (BITS == 4) {
    static_assert(T::kExactDecode, "4-bit codes are decoded exactly for fp16 only");
    r = decode_w4<T, 8>(w[0], dc);
  } else if constexpr (T::code == SPARKQ_F16) {
#pragma unroll
    for (int i = 0; i < 4; ++i)  // bytes under fp16 1024, which an exact subtract removes
      r[i] = exact_f16_pair<128>(
          __builtin_amdgcn_perm(0x64646464u, w[i >> 1], (i & 1) ? 0x04030402u : 0x04010400u));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // c ^ 128 as a signed byte is c - 128
      const int v = (int)(w[i >> 1] ^ 0x80808080u) >> (16 * (i & 1));
      r[i] = pack_round<T>((float)(signed char)v, (float)(signed char)(v >> 8));
    }
  }
  return r;
}

template <typename T, int BITS, int G>
__global__ __launch_bounds__(256, BITS == 4 ? 3 : 2) void affine_gemm_kernel(AffGemmArgs a) {
  constexpr int WC = BITS / 4;          // words per chunk of 8 codes
  constexpr int WQ = 2 * WC;            // 16-byte code loads per unit and column
  constexpr int NGU = kAffBK / G;       // groups per unit
  constexpr int AL = kAffBM * kAffBK / 8 / 256;  // 16-byte A pieces per thread
  __shared__ __attribute__((aligned(16))) unsigned char As[2][kAffBM * kAffBK * 2];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane >> 5, l32 = lane & 31;
  const int K = a.K, N = a.N, M = a.M;
  // XCD-contiguous chunks of the (piece, tile) order, the tiles of a piece in
  // groups of 8 tile rows column by column: what an XCD runs together shares
  // activation rows and weight columns in its L2
  const int T_ = a.tiles_m * a.tiles_n, items = T_ * a.S;
  const int id = blockIdx.x;
  const int v0 = (items & 7) == 0 ? (id & 7) * (items >> 3) + (id >> 3) : id;
  const int piece = v0 / T_, v = v0 - piece * T_;
  const int width = 8 * a.tiles_n, grp8 = v / width, fm = 8 * grp8;
  const int gs = min(a.tiles_m - fm, 8), r8 = v - grp8 * width;
  const int m0 = (fm + r8 % gs) * kAffBM, n0 = (r8 / gs) * kAffBN;
  const int units = (K + kAffBK - 1) / kAffBK;
  const int u0 = (int)((int64_t)piece * units / a.S), u1 = (int)((int64_t)(piece + 1) * units / a.S);
  const int mrows = min(kAffBM, M - m0);
  const int wn0 = n0 + 32 * wave;
  const int ncols = __builtin_amdgcn_readfirstlane(max(0, min(32, N - wn0)));
  const uint32_t wrow = (uint32_t)K * BITS / 8;  // bytes of a weight row
  // rows past M and columns past N read zeros and are not stored
  const rsrc_t rx = make_rsrc(a.x + (int64_t)m0 * K, (uint32_t)mrows * (uint32_t)K * 2u);
  const rsrc_t rw = make_rsrc(reinterpret_cast<const unsigned char*>(a.w) + (int64_t)wn0 * wrow,
                              (uint32_t)ncols * wrow);
  const DecodeConsts dc = decode_consts<F16>();

  uint32_t xoff[AL], lds_w[AL];
  int xk[AL];
#pragma unroll
  for (int i = 0; i < AL; ++i) {
    const int p = tid + 256 * i, row = p >> 4, kc = p & 15;
    xk[i] = 8 * kc;
    xoff[i] = (uint32_t)(row * K + kc * 8) * 2u;
    lds_w[i] = (uint32_t)(row * 256 + ((kc ^ (row & 15)) << 4));
  }
  // A chunk of this lane in sub-step (h, ss): 8h + 4j + ss, or with two groups
  // per 64 k 8h + 2ss + j, so that no MFMA straddles a group
  constexpr bool NARROW = G == 32;
  const uint32_t lds_r = (uint32_t)(l32 * 256 + (((l32 & 15) ^ (NARROW ? j : 4 * j)) << 4));
  const uint32_t woff = (uint32_t)l32 * wrow + 16u * WC * j;
  const int col = min(wn0 + l32, N - 1), row = min(m0 + lane, M - 1);

  u32x4_t ra[2][AL], rb[2][WQ];
  float rs[2][NGU];
  auto load = [&](int u, int set) {
    const int k0 = u * kAffBK;
#pragma unroll
    for (int i = 0; i < AL; ++i)  // (k past K reads zeros, which no code matters to)
      ra[set][i] = buf_load16(rx, u < u1 && k0 + xk[i] < K ? xoff[i] + 2u * (uint32_t)k0 : kOob);
#pragma unroll
    for (int q = 0; q < WQ; ++q)  // half h = q / WC: 64 k, this lane's 32 of them
      rb[set][q] = buf_load16(
          rw, u < u1 ? woff + (uint32_t)(k0 * BITS / 8) + 32u * WC * (q / WC) + 16u * (q % WC) : kOob);
#pragma unroll
    for (int g = 0; g < NGU; ++g) {
      const int64_t gi = (int64_t)min(u, u1 - 1) * NGU + g;
      rs[set][g] = a.st[gi * N + col];
    }
  };

  f32x32_t acc = f32x32_t{};
  f32x16_t tmp[2];

  auto body = [&](int u, auto stc) {
    constexpr int st = decltype(stc)::value;
    __builtin_amdgcn_sched_barrier(0);
    uint32_t wc[4 * WQ];
    float sv[NGU], bv[NGU], xv[NGU];
#pragma unroll
    for (int q = 0; q < WQ; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) wc[4 * q + e] = rb[st][q][e];
#pragma unroll
    for (int g = 0; g < NGU; ++g) {
      sv[g] = rs[st][g];
      bv[g] = a.bt[(int64_t)(u * NGU + g) * N + col];
      xv[g] = a.xs[(int64_t)(u * NGU + g) * M + row];
    }
    // (the bias operands of this unit before the next loads: waits count in order)
    __builtin_amdgcn_sched_barrier(0);
    load(u + 2, st);
    if constexpr (NARROW) {
      // lane half j holds chunks 4j..4j+3 of each half; trade the upper half of
      // chunk 2i against the lower half of chunk 2i+1, after which register
      // 2i holds chunks (2i, 2i+1) of the first group and 2i+1 those of the
      // second: {0: 0|1, 1: 4|5, 2: 2|3, 3: 6|7}
#pragma unroll
      for (int c = 0; c < 8; c += 2)
#pragma unroll
        for (int e = 0; e < WC; ++e) {
          const auto r =
              __builtin_amdgcn_permlane32_swap(wc[c * WC + e], wc[(c + 1) * WC + e], false, false);
          wc[c * WC + e] = r[0];
          wc[(c + 1) * WC + e] = r[1];
        }
    }
    const unsigned char* as = As[st];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int ss = 0; ss < 4; ++ss) {
        // chunk register of sub-step ss (see the trade above)
        const int cr = 4 * h + (NARROW ? (ss & 1) * 2 + (ss >> 1) : ss);
        const u32x4_t bf = aff_decode<T, BITS>(&wc[cr * WC], dc);
        const int k = 64 * h + 16 * ss;  // (groups are whole sub-steps: 16 k each)
        const bool first = k % G == 0, last = (k + 16) % G == 0;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const u32x4_t af = *reinterpret_cast<const u32x4_t*>(
              as + ((lds_r ^ (uint32_t)((8 * h + (NARROW ? 2 * ss : ss)) << 4)) + x * 32 * 256));
          tmp[x] = mfma32x32x16<T>(af, bf, first ? f32x16_t{} : tmp[x]);
        }
        if (last) {
          const int g = k / G;
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[16 * x + e] = fmaf(sv[g], tmp[x][e], acc[16 * x + e]);
          // the group's bias part: two blocks of 32 rows, one k
          acc = __builtin_amdgcn_mfma_f32_32x32x1f32(xv[g], bv[g], acc, 0, 0, 0);
        }
      }
    // slot st^1 was last read in unit u-1, before the barrier that ended it
#pragma unroll
    for (int i = 0; i < AL; ++i) *reinterpret_cast<u32x4_t*>(&As[st ^ 1][lds_w[i]]) = ra[st ^ 1][i];
    __syncthreads();
  };

  load(u0, 0);
  __builtin_amdgcn_sched_barrier(0);
  load(u0 + 1, 1);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < AL; ++i) *reinterpret_cast<u32x4_t*>(&As[0][lds_w[i]]) = ra[0][i];
  __syncthreads();
  int u = u0;
  for (; u + 2 <= u1; u += 2) {
    body(u, std::integral_constant<int, 0>{});
    body(u + 1, std::integral_constant<int, 1>{});
  }
  if (u < u1) body(u, std::integral_constant<int, 0>{});

  const bool split = a.S > 1;
  float* part = a.part + (int64_t)piece * M * N;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int gm = m0 + 32 * x + mfma32_row(lane, e), gn = wn0 + l32;
      if (gm < M && gn < N) {
        const int64_t idx = (int64_t)gm * N + gn;
        if (split)
          part[idx] = acc[16 * x + e];
        else
          store_out(a.y, idx, acc[16 * x + e], a.y_dtype);
      }
    }
}

// y = the pieces' sums in order, four outputs per thread where total % 4 == 0
__global__ __launch_bounds__(256) void affine_sum_kernel(const float* __restrict__ part,
                                                         void* __restrict__ y, int y_dtype,
                                                         int64_t total, int S) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  if ((total & 3) == 0) {
    f32x4_t s = *reinterpret_cast<const f32x4_t*>(part + i);
    for (int p = 1; p < S; ++p) s += *reinterpret_cast<const f32x4_t*>(part + p * total + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) store_out(y, i + e, s[e], y_dtype);
    return;
  }
  for (int64_t k = i; k < std::min<int64_t>(i + 4, total); ++k) {
    float s = part[k];
    for (int p = 1; p < S; ++p) s += part[p * total + k];
    store_out(y, k, s, y_dtype);
  }
}

struct AffLayout {
  size_t st, bt, xs, part, bytes;
};
// Pieces of K, at most 8 and of at least three units: the number that
// minimises an estimate. Its unit times (1 in a workgroup that has a CU to
// itself, 1.5 where two share one) are below the traced ones (1.7 and 1.8 us),
// and order the pieces as measured beside what these cost, a launch and their
// partials' round trip. Us per call in 1, 2, 3, 4, 6, 8 pieces (its choice in
// brackets): fp16 4-bit 333 x 2560 x 9728 G128 79, 50, 48, [42], 43, 46; 512 x
// 3584 x 2560 G64 [33], 36, 36, 38, 42, 43; 2048 x 2560 x 9728 G128 157, 151, 161,
// [159], 167, 177; bf16 8-bit 333 x 2560 x 9728 G64 98, 59, 61, [51], 55, 57; 64 x
// 3584 x 2560 33, 23, 20, 19, 18, 19 [five: 18]; 1 x 2560 x 4096 G32 52, 33, 26, 22, 20, [18].
int aff_pieces(int64_t M, int64_t N, int64_t K) {
  const int64_t cus = device_cus(), units = cdiv(K, kAffBK);
  if (const int64_t s = env_int("SPARKQ_AFFG_S", 0); s > 0)
    return (int)std::min<int64_t>(s, units);
  const int64_t T = cdiv(M, kAffBM) * cdiv(N, kAffBN);
  int64_t S = 1;
  double cost = 0;
  for (int64_t s = 1; s <= std::min<int64_t>(8, std::max<int64_t>(units / 3, 1)); ++s) {
    const double chain = (double)(cdiv(T * s, 2 * cus) * cdiv(units, s)) * (T * s <= cus ? 1.0 : 1.5);
    const double c = chain + (s > 1 ? 5.0 + (double)s * (double)M * (double)N * 1.2e-6 : 0.0);
    if (s == 1 || c < cost) cost = c, S = s;
  }
  return (int)S;
}

AffLayout aff_layout(int64_t M, int64_t N, int64_t K, int G, int S) {
  const size_t ng = (size_t)cdiv(K, kAffBK) * (kAffBK / G);  // whole units
  AffLayout l;
  l.st = 0;
  l.bt = round_up(ng * N * 4, 256);
  l.xs = l.bt + round_up(ng * N * 4, 256);
  l.part = l.xs + round_up(ng * M * 4, 256);
  l.bytes = l.part + (S > 1 ? round_up((size_t)S * M * N * 4, 256) : 0);
  return l;
}

template <typename T, int BITS>
void launch_aff_g(int G, const AffGemmArgs& a, dim3 grid, hipStream_t st) {
  if (G == 32)
    hipLaunchKernelGGL((affine_gemm_kernel<T, BITS, 32>), grid, dim3(256), 0, st, a);
  else if (G == 64)
    hipLaunchKernelGGL((affine_gemm_kernel<T, BITS, 64>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((affine_gemm_kernel<T, BITS, 128>), grid, dim3(256), 0, st, a);
}

}  // namespace

size_t affine_gemm_workspace(int64_t M, int64_t N, int64_t K, int G) {
  return aff_layout(M, N, K, G, aff_pieces(M, N, K)).bytes;
}

// bits 4 takes fp16 activations only; a weight tile's rows (128 of them) and
// an activation tile's (64) must lie within one buffer descriptor's 2 GiB
int affine_gemm(const void* x, const uint32_t* w, const void* s, const void* b, void* y, int64_t M,
                int64_t N, int64_t K, int G, int bits, int xdt, int sdt, int ydt,
                unsigned char* ws, hipStream_t st) {
  const int S = aff_pieces(M, N, K);
  const AffLayout l = aff_layout(M, N, K, G, S);
  AffPrepArgs q{};
  q.x = (const uint16_t*)x;
  q.sc = s;
  q.bi = b;
  q.st = reinterpret_cast<float*>(ws + l.st);
  q.bt = reinterpret_cast<float*>(ws + l.bt);
  q.xs = reinterpret_cast<float*>(ws + l.xs);
  q.M = (int)M;
  q.N = (int)N;
  q.K = (int)K;
  q.G = G;
  q.s_dtype = sdt;
  q.ngp = (int)cdiv(K, kAffBK) * (kAffBK / G);
  q.centre = (float)(1 << (bits - 1));
  q.wblocks = (int)(cdiv(N, 64) * cdiv(q.ngp, 32));
  const dim3 pg((unsigned)(q.wblocks + cdiv(M * (K / 8), 256)));
  if (xdt == SPARKQ_BF16)
    hipLaunchKernelGGL(affine_prep_kernel<BF16>, pg, dim3(256), 0, st, q);
  else
    hipLaunchKernelGGL(affine_prep_kernel<F16>, pg, dim3(256), 0, st, q);
  if (int rc = check_launch("affine_prep_kernel")) return rc;
  AffGemmArgs a{};
  a.x = q.x;
  a.w = w;
  a.st = q.st;
  a.bt = q.bt;
  a.xs = q.xs;
  a.y = y;
  a.part = reinterpret_cast<float*>(ws + l.part);
  a.y_dtype = ydt;
  a.M = q.M;
  a.N = q.N;
  a.K = q.K;
  a.tiles_m = (int)cdiv(M, kAffBM);
  a.tiles_n = (int)cdiv(N, kAffBN);
  a.S = S;
  const dim3 grid((unsigned)((int64_t)a.tiles_m * a.tiles_n * S));
  if (bits == 4)
    launch_aff_g<F16, 4>(G, a, grid, st);
  else if (xdt == SPARKQ_BF16)
    launch_aff_g<BF16, 8>(G, a, grid, st);
  else
    launch_aff_g<F16, 8>(G, a, grid, st);
  if (int rc = check_launch("affine_gemm_kernel")) return rc;
  if (S > 1) {
    hipLaunchKernelGGL(affine_sum_kernel, dim3((unsigned)cdiv(M * N, 1024)), dim3(256), 0, st,
                       a.part, y, ydt, M * N, S);
    return check_launch("affine_sum_kernel");
  }
  return 0;
}

}  // namespace sparkq
