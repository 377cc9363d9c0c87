// The matrix-core step of the bandwidth decode kernels: one 16-token pool block of one KV head against its
// group of query heads, and the stripes that small launches cut a sequence into.
#pragma once

#include "mi_common.h"

namespace mi {
namespace {

constexpr int kHeadDim = 128;
constexpr int kBlockSize = 16;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kRescaleSlack = 8.0f;
constexpr int kStripes = 8;  // stripe v of a sequence: blocks v, v + kStripes, ...

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Reference rounding points: the bf16 matmul output, then the bf16 product with the
// scale (src/mini_infra/model/qwen3.py:243).  Returned in log2 units for exp2.
__device__ __forceinline__ float score_log2(float dot, float scale) {
  const float s = static_cast<float>(static_cast<__bf16>(static_cast<float>(static_cast<__bf16>(dot)) * scale));
  return s * kLog2e;
}

__device__ __forceinline__ void store_bf16x8(uint16_t* dst, const float* o, float inv) {
  uint4 v;
  v.x = pack_bf16x2(o[0] * inv, o[1] * inv);
  v.y = pack_bf16x2(o[2] * inv, o[3] * inv);
  v.z = pack_bf16x2(o[4] * inv, o[5] * inv);
  v.w = pack_bf16x2(o[6] * inv, o[7] * inv);
  *reinterpret_cast<uint4*>(dst) = v;
}

// ---- Matrix-core form (groups of up to 16 query heads).  Per 16-token block and wavefront:
//  * S^T = K Q^T with four v_mfma_f32_16x16x32_bf16 over the 128 dims: A = K (lane: token
//    lane % 16, dims 32 ks + 8 (lane / 16) .. +8), B = Q^T (lane: head lane % 16, zero past the
//    group), C: lane holds head lane % 16, tokens 4 (lane / 16) + i.  K is loaded in whole
//    256-byte token rows, as the dot-product form loads it, and restaged into the A layout
//    through 16 LDS rows per wavefront (A straight from the pool would read 64-byte pieces of 16
//    rows per instruction).
//  * That C layout is the A layout of v_mfma_f32_16x16x16_bf16 (row lane % 16, k = 4 (lane / 16)
//    + i), so the probabilities feed O = P V without moving.  V is loaded as token 4 (lane / 16) + i,
//    dims 8 (lane % 16) .. +8; output tile t takes dim 8 j + t as its column j, so B of tile t is
//    element t of the lane's four V pieces (two v_perm) and the lane ends up holding, for heads
//    4 (lane / 16) + i, dims 8 (lane % 16) .. +8: one 16-byte store per head.
//  * Softmax per head column: the running max m is shared by the column's four lanes (raised
//    lazily, with the column max, as in the dot-product form); each lane sums its own tokens.
struct MfmaState {
  float m;       // running max of head lane % 16 (log2 units), equal in the four lanes of its column
  float l;       // this lane's share of the head's sum
  f32x4 o[8];    // tile t: O[head 4 (lane / 16) + i][dim 8 (lane % 16) + t]
};

constexpr int kKStageRow = kHeadDim + 8;  // LDS row (elements) of a wavefront's K staging: 272 bytes

// kb: the lane's K pieces as the dot-product form loads them (token 4 i + lane / 16, dims
// 8 (lane % 16) .. +8: whole 256-byte rows per instruction); kst: the wavefront's 16-row K staging
// in LDS, through which they reach the MFMA A layout (token lane % 16, dims 32 ks + 8 (lane / 16)).
__device__ __forceinline__ void attend_block_mfma(MfmaState& st, const bf16x8 (&qf)[4], const u32x4 (&kb)[4],
                                                  const u32x4 (&vb)[4], uint16_t* kst, float scale,
                                                  int tok_base, int n, int lane) {
  const int dl = lane & 15, r = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(kst + (4 * i + r) * kKStageRow + 8 * dl) = kb[i];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(kst + dl * kKStageRow + 32 * ks + 8 * r),
                                                  qf[ks], acc, 0, 0, 0);
  // The next block's staging stores follow these reads in the wavefront's LDS order.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int tok0 = tok_base + 4 * (lane >> 4);
  float sc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) sc[i] = score_log2(acc[i], scale);
  if (tok_base + kBlockSize > n) {  // the sequence's last block (uniform branch)
#pragma unroll
    for (int i = 0; i < 4; ++i) sc[i] = tok0 + i < n ? sc[i] : -INFINITY;
  }
  const float mb = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
  if (__builtin_amdgcn_ballot_w64(mb > st.m + kRescaleSlack) != 0) {  // lazy rescale (wave-uniform)
    float cm = fmaxf(mb, __shfl_xor(mb, 16));
    cm = fmaxf(cm, __shfl_xor(cm, 32));
    const float nm = fmaxf(st.m, cm);
    const float al = (nm == -INFINITY) ? 1.0f : __builtin_amdgcn_exp2f(st.m - nm);
    st.m = nm;
    st.l *= al;
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // O rows are heads 4 (lane / 16) + i: lane h holds head h's factor
      const float ai = __shfl(al, 4 * (lane >> 4) + i);
#pragma unroll
      for (int t = 0; t < 8; ++t) st.o[t][i] *= ai;
    }
  }
  const float ref = st.m == -INFINITY ? 0.0f : st.m;
  float p[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_exp2f(sc[i] - ref);
  st.l += (p[0] + p[1]) + (p[2] + p[3]);
  const bf16x4 pa = __builtin_convertvector((f32x4){p[0], p[1], p[2], p[3]}, bf16x4);
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const uint32_t sel = (t & 1) ? 0x07060302u : 0x05040100u;
    const uint32_t w01 = __builtin_amdgcn_perm(vb[1][t >> 1], vb[0][t >> 1], sel);  // tokens 0, 1 at dim t
    const uint32_t w23 = __builtin_amdgcn_perm(vb[3][t >> 1], vb[2][t >> 1], sel);  // tokens 2, 3
    const bf16x4 vbf = __builtin_bit_cast(bf16x4, (u32x2){w01, w23});
    st.o[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pa, vbf, st.o[t], 0, 0, 0);
  }
}

// One head's 8 dims of the kStripes stripe states, joined in stripe order (log-sum-exp).
struct StripeMerge {
  float m[kStripes], l[kStripes];
  float4 x[kStripes], y[kStripes];
  __device__ __forceinline__ void store(uint16_t* dst) const {
    float M = -INFINITY;
#pragma unroll
    for (int v = 0; v < kStripes; ++v) M = fmaxf(M, m[v]);
    float L = 0.0f, o[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) o[d] = 0.0f;
#pragma unroll
    for (int v = 0; v < kStripes; ++v) {
      const float e = m[v] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m[v] - M);
      L += e * l[v];
      o[0] += e * x[v].x; o[1] += e * x[v].y; o[2] += e * x[v].z; o[3] += e * x[v].w;
      o[4] += e * y[v].x; o[5] += e * y[v].y; o[6] += e * y[v].z; o[7] += e * y[v].w;
    }
    store_bf16x8(dst, o, 1.0f / L);
  }
};

}  // namespace
}  // namespace mi
