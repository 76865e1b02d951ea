// sdpa_gen.h -- argument block of the attention over an MLX affine cache of any
// width (sdpa_gen.hip: the vector kernel and the launcher; sdpa_stage.hip: the
// matrix-core kernel for 16-bit queries).
#pragma once

#include "common.h"

namespace sparkq {

struct GenSdpaArgs {
  const void* q;                  // [B,Hq,L,D] contiguous, q dtype
  const uint32_t* kp;             // packed codes, D*bits/32 words per token
  const void* ks;                 // scales [.., D/G], q dtype
  const void* kb;                 // biases, same strides as scales
  const uint32_t* vp;
  const void* vs;
  const void* vb;
  const void* mask;               // mask array or null
  void* out;                      // [B,Hq,L,Dv]
  float* pm;                      // split partials: max [rows][S]
  float* pz;                      //   sums [rows][S]
  float* pacc;                    //   outputs [rows][S][Dv]
  int64_t kp_b, kp_h, kp_t;       // strides in words
  int64_t ks_b, ks_h, ks_t;       // strides in elements (biases share them)
  int64_t vp_b, vp_h, vp_t;
  int64_t vs_b, vs_h, vs_t;
  int64_t m_b, m_h, m_l, m_n;     // mask strides in elements (0 to broadcast)
  int mask_kind;                  // kMask*
  int mask_dtype;                 // additive masks: SPARKQ_F32/F16/BF16
  int B, Hq, Hkv, L, N, D, Dv, G, bits;
  int q_dtype, out_dtype;
  int RC, nch;                    // query heads per workgroup, chunks per KV head
  int S, tps;                     // context splits, tokens per split
  int vt;                         // value tokens per LDS stage
  float scale_log2;               // softmax scale times log2(e)
  float masked;                   // score of a masked entry, in log2 units
};

constexpr int kMaskNone = 0, kMaskCausal = 1, kMaskBool = 2, kMaskAdd = 3;

// sdpa_stage.hip: whether the matrix-core kernel takes the types and head dims,
// and the call, its context splits and its launch
bool sdpa_stage_dims(int qdt, int64_t D, int64_t Dv);
bool sdpa_stage_ok(const GenSdpaArgs& a);
int sdpa_stage_splits(int64_t B, int64_t Hq, int64_t Hkv, int64_t L, int64_t N);
int launch_sdpa_stage(const GenSdpaArgs& a, hipStream_t st);

}  // namespace sparkq
