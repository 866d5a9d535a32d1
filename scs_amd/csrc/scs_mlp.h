// Branching-score MLP (6 integer features -> 64 -> 64 -> 1), device side.
//
// The learned ordering replaces the connection score of selectUstar
// (src/helpers.cc:1104-1168) when a query runs with a model.  It only
// changes which vertex is branched on first; every rule and bound is the
// same, so the optimum is unchanged.
//
// Inference runs on the MFMA units: v_mfma_f32_16x16x16_bf16 with BF16
// weights/activations and FP32 accumulation, 16 candidates per tile.
// Operand layout of one 16x16x16 MFMA (lane l of 64, kb = l / 16):
//   A[m][k]: lane holds m = l % 16, k = 4*kb + i (i = 0..3)
//   B[k][n]: lane holds n = l % 16, k = 4*kb + i
//   D[m][n]: lane holds n = l % 16, m = 4*kb + i
#pragma once
#include "scs_internal.h"

#define MLP_IN 6
#define MLP_INP 16  // input padded to one MFMA K-step
#define MLP_H 64

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

// Packed inference model in device memory.
struct MlpDev {
  // bf16, [output unit][input]: a lane's four inputs of an MFMA step are one
  // 8-byte load
  u16 w1[MLP_H][MLP_INP];  // inputs >= MLP_IN are zero
  u16 w2[MLP_H][MLP_H];
  float b1[MLP_H];
  float b2[MLP_H];
  float w3[MLP_H];
  float b3;
  float mean[8];
  float scale[8];
  float pad[7];
};

__device__ __forceinline__ u16 f2bf(float f) {
  u32 x = __float_as_uint(f);
  x += 0x7fffu + ((x >> 16) & 1u);  // round to nearest even
  return (u16)(x >> 16);
}
__device__ __forceinline__ float bf2f(u16 b) { return __uint_as_float(((u32)b) << 16); }

// Raw features of a candidate v at the current node: four degrees/
// distances, the rule-1 slack and the plain connection score (in units).
struct MlpFeat {
  u32 dC, dR, dist, core;
  int slack;
  float cscore;
};

// The model as mlp_tile takes it.  MlpRegs: the wave's share in registers,
// loaded once and used for many tiles (stand-alone inference; 60 registers).
// MlpMem: read again for every tile, one group of 16 units at a time (the
// search kernel, whose own state leaves no room: held in registers there the
// model spilled 396 bytes per lane).
struct MlpMem {
  static constexpr int UNROLL = 1;
  const MlpDev* M;
  u32 row, kb;
  __device__ explicit MlpMem(const MlpDev* m)
      : M(m), row(threadIdx.x & 15u), kb((threadIdx.x & 63u) >> 4) {}
  __device__ bf16x4 w1(u32 j) const { return *(const bf16x4*)&M->w1[16 * j + row][4 * kb]; }
  __device__ bf16x4 w2(u32 j, u32 ks) const {
    return *(const bf16x4*)&M->w2[16 * j + row][16 * ks + 4 * kb];
  }
  __device__ float b1(u32 j) const { return M->b1[16 * j + row]; }
  __device__ float b2(u32 j) const { return M->b2[16 * j + row]; }
  __device__ float w3(u32 j) const { return M->w3[16 * j + row]; }
  __device__ float b3() const { return M->b3; }
  // of this lane's input 4*kb + i (0 beyond the sixth)
  __device__ float mean(u32 i) const { return 4 * kb + i < MLP_IN ? M->mean[4 * kb + i] : 0.f; }
  __device__ float scale(u32 i) const { return 4 * kb + i < MLP_IN ? M->scale[4 * kb + i] : 0.f; }
};
struct MlpRegs {
  static constexpr int UNROLL = 4;
  bf16x4 w1_[4], w2_[4][4];
  float b1_[4], b2_[4], w3_[4], b3_, mean_[4], scale_[4];
  __device__ explicit MlpRegs(const MlpMem& m) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      w1_[j] = m.w1(j);
#pragma unroll
      for (int ks = 0; ks < 4; ks++) w2_[j][ks] = m.w2(j, ks);
      b1_[j] = m.b1(j);
      b2_[j] = m.b2(j);
      w3_[j] = m.w3(j);
      mean_[j] = m.mean(j);
      scale_[j] = m.scale(j);
    }
    b3_ = m.b3();
  }
  __device__ bf16x4 w1(u32 j) const { return w1_[j]; }
  __device__ bf16x4 w2(u32 j, u32 ks) const { return w2_[j][ks]; }
  __device__ float b1(u32 j) const { return b1_[j]; }
  __device__ float b2(u32 j) const { return b2_[j]; }
  __device__ float w3(u32 j) const { return w3_[j]; }
  __device__ float b3() const { return b3_; }
  __device__ float mean(u32 i) const { return mean_[i]; }
  __device__ float scale(u32 i) const { return scale_[i]; }
};

// Scores the 16 candidates of one tile.  feat(row) gives the raw features
// of row (rows >= valid are ignored).  h1s: 16 x 64 bf16 LDS scratch.
// Returns the score of row (l % 16) on every lane (lanes with the same
// l % 16 hold the same value).
template <typename Model, typename FeatFn>
__device__ __forceinline__ float mlp_tile(const Model& R, FeatFn feat, u16* h1s) {
  const u32 l = threadIdx.x & 63u;
  const u32 row = l & 15u;
  const u32 kb = l >> 4;
  // layer 1 input: 16 rows x 16 k (features 0..5, rest zero)
  MlpFeat f = feat(row);
  float xin[8] = {(float)f.dC, (float)f.dR,    (float)f.dist, (float)f.core,
                  (float)f.slack, f.cscore, 0.f,          0.f};
  bf16x4 a1;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float x = kb == 0 ? xin[i] : (kb == 1 ? xin[4 + i] : 0.f);
    a1[i] = (short)f2bf((x - R.mean(i)) * R.scale(i));
  }
#pragma unroll Model::UNROLL
  for (u32 j = 0; j < 4; j++) {
    const float b1 = R.b1(j);
    f32x4 d = {0.f, 0.f, 0.f, 0.f};
    d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1, R.w1(j), d, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float z = d[i] + b1;
      h1s[(4 * kb + i) * MLP_H + 16 * j + row] = f2bf(z > 0.f ? z : 0.f);
    }
  }
  __syncthreads();
  // layer 2 (K = 64 in four steps) fused with the 64 -> 1 output layer
  bf16x4 a[4];
#pragma unroll
  for (u32 ks = 0; ks < 4; ks++) a[ks] = *(const bf16x4*)&h1s[row * MLP_H + 16 * ks + 4 * kb];
  float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll Model::UNROLL
  for (u32 j = 0; j < 4; j++) {
    bf16x4 wj[4];
#pragma unroll
    for (u32 ks = 0; ks < 4; ks++) wj[ks] = R.w2(j, ks);
    const float b2 = R.b2(j), w3 = R.w3(j);
    f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (u32 ks = 0; ks < 4; ks++)
      d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[ks], wj[ks], d, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float z = d[i] + b2;
      part[i] += (z > 0.f ? z : 0.f) * w3;
    }
  }
  // part[i] is row (4*kb + i)'s partial sum over this lane's 4 columns;
  // sum over the 16 lanes of the same kb
  for (int i = 0; i < 4; i++)
    for (int o = 8; o > 0; o >>= 1) part[i] += __shfl_xor(part[i], o, 16);
  // every lane of group kb now holds the sums of rows 4kb..4kb+3; lane l
  // needs row l % 16, held by group (l % 16) / 4 at index (l % 16) % 4
  const u32 src_kb = row >> 2, src_i = row & 3u;
  const float v0 = __shfl(part[0], 16 * src_kb), v1 = __shfl(part[1], 16 * src_kb);
  const float v2 = __shfl(part[2], 16 * src_kb), v3 = __shfl(part[3], 16 * src_kb);
  const float s = src_i == 0 ? v0 : src_i == 1 ? v1 : src_i == 2 ? v2 : v3;
  __syncthreads();
  return s + R.b3();
}
