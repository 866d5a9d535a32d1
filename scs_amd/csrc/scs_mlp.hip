// Training and stand-alone inference kernels of the branching MLP.
//
// Training runs in FP32: a mini-batch is one kernel for the forward and
// backward pass and the weight gradients, on the FP32 matrix units, and one for
// their sum and the Adam step.  Inference uses the same BF16 MFMA tile routine
// as the search engine (scs_mlp.h).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "scs_mlp.h"

// Flat parameter layout = scs_model (include/scs.h).
#define P_W1 0
#define P_B1 (P_W1 + 8 * MLP_H)
#define P_W2 (P_B1 + MLP_H)
#define P_B2 (P_W2 + MLP_H * MLP_H)
#define P_W3 (P_B2 + MLP_H)
#define P_B3 (P_W3 + MLP_H)
#define P_MEAN (P_B3 + 1)
#define P_SCALE (P_MEAN + 8)
#define P_TRAIN P_MEAN  // trainable parameters precede mean/scale
#define P_TOTAL (P_SCALE + 8 + 7)

static_assert(sizeof(scs_model) == P_TOTAL * sizeof(float), "scs_model layout");

// ---------------------------------------------------------------------------
// One gradient step.  A block takes MLP_S samples at a time through the
// forward and backward pass and keeps its share of every weight gradient in
// registers; the contractions (64 x 64 layers, both directions, and the
// weight gradients over the samples) run on the FP32 MFMA units with FP32
// accumulation.  Blocks leave partial gradients that a second kernel adds up
// in a fixed order, so a step gives the same bits each time.
//
// Wave w owns columns 16w .. 16w+15 of every 64-column matrix.  Operand
// layout of v_mfma_f32_16x16x4_f32 (lane l, n = l % 16, kb = l / 16): A[n][kb],
// B[kb][n], D[4*kb + i][n].  Where the summed index runs over a layer's 64
// units, step t of lane group kb takes unit 16*kb + t (any order that both
// operands share gives the sum), so a lane's operands are contiguous.
//
// Bound: launch and load latency; the arithmetic of a 2,048-sample step is
// 50 MFLOP.  A step took 630 us with one thread per sample and one serial sum
// over the batch per parameter (19 blocks), 20 us now, and its
// gradients are 3 to 80 times nearer to 64-bit ones (500 to 100,000 rows).
// ---------------------------------------------------------------------------
#define MLP_S 32           // samples per block and pass
#define MLP_LD 68          // LDS row stride (floats): 16-byte rows, shifted banks
#define MLP_MAXBLK 256     // blocks per step at most (each leaves P_TRAIN partial sums)

__device__ __forceinline__ f32x4 mlp_mfma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__global__ void __launch_bounds__(256) mlp_step(const float* __restrict__ P,
                                                const float* __restrict__ X,
                                                const float* __restrict__ Y,
                                                const u32* __restrict__ idx, u32 B, float posw,
                                                float* __restrict__ part,
                                                float* __restrict__ lossp) {
  __shared__ float xs[MLP_S][8];
  __shared__ __align__(16) float a1[MLP_S][MLP_LD], d2[MLP_S][MLP_LD], d1[MLP_S][MLP_LD];
  __shared__ float outp[4][MLP_S], gs[MLP_S];
  const u32 t = threadIdx.x, l = t & 63, w = t >> 6, n = l & 15, kb = l >> 4;
  const u32 col = 16 * w + n;
  // weights of this wave's columns, once per block
  float w1f[2], w2f[16], w2t[16];
#pragma unroll
  for (int k = 0; k < 2; k++) w1f[k] = P[P_W1 + (4 * k + kb) * MLP_H + col];
#pragma unroll
  for (int k = 0; k < 16; k++) w2f[k] = P[P_W2 + (16 * kb + k) * MLP_H + col];
#pragma unroll
  for (int k = 0; k < 16; k++) w2t[k] = P[P_W2 + col * MLP_H + 16 * kb + k];
  const float b1 = P[P_B1 + col], b2 = P[P_B2 + col], w3 = P[P_W3 + col], b3 = P[P_B3];
  f32x4 gW2[4], gW1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < 4; m++) gW2[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  float gb1 = 0.f, gb2 = 0.f, gw3 = 0.f, gb3 = 0.f, ls = 0.f;
  for (u32 s0 = blockIdx.x * MLP_S; s0 < B; s0 += gridDim.x * MLP_S) {
    {
      const u32 s = t >> 3, k = t & 7;  // 32 samples x 8 features
      float x = 0.f;
      if (s0 + s < B && k < MLP_IN) {
        const u64 r = idx[s0 + s];
        x = (X[r * MLP_IN + k] - P[P_MEAN + k]) * P[P_SCALE + k];
      }
      xs[s][k] = x;
    }
    float y = 0.f;
    if (t < MLP_S && s0 + t < B) y = Y[idx[s0 + t]];
    __syncthreads();
    f32x4 z2[2];
    u32 on1 = 0;  // bit 4r + i: hidden unit (row 16r + 4kb + i, col) is active
#pragma unroll
    for (int r = 0; r < 2; r++) {
      f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 2; k++) z = mlp_mfma(xs[16 * r + n][4 * k + kb], w1f[k], z);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float v = z[i] + b1;
        if (v > 0.f) on1 |= 1u << (4 * r + i);
        a1[16 * r + 4 * kb + i][col] = v > 0.f ? v : 0.f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; r++) {
      f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 16; k++) z = mlp_mfma(a1[16 * r + n][16 * kb + k], w2f[k], z);
      float o[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        z[i] += b2;
        o[i] = (z[i] > 0.f ? z[i] : 0.f) * w3;
      }
      z2[r] = z;
#pragma unroll
      for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int d = 8; d > 0; d >>= 1) o[i] += __shfl_xor(o[i], d, 16);
        if (n == 0) outp[w][16 * r + 4 * kb + i] = o[i];
      }
    }
    __syncthreads();
    if (t < MLP_S) {
      const float out = b3 + ((outp[0][t] + outp[1][t]) + (outp[2][t] + outp[3][t]));
      float g = 0.f;
      if (s0 + t < B) {
        // binary cross-entropy with logits, mean over the batch
        const float wt = y > 0.5f ? posw : 1.f;
        const float sp = out > 0.f ? out + log1pf(expf(-out)) : log1pf(expf(out));
        ls += wt * (sp - y * out) / (float)B;
        const float sig = 1.f / (1.f + expf(-out));
        g = wt * (sig - y) / (float)B;
      }
      gs[t] = g;
      gb3 += g;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float g = gs[16 * r + 4 * kb + i], z = z2[r][i];
        const float d = z > 0.f ? g * w3 : 0.f;
        gw3 += z > 0.f ? g * z : 0.f;
        gb2 += d;
        d2[16 * r + 4 * kb + i][col] = d;
      }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; r++) {
      f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 16; k++) z = mlp_mfma(d2[16 * r + n][16 * kb + k], w2t[k], z);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float d = (on1 >> (4 * r + i)) & 1u ? z[i] : 0.f;
        gb1 += d;
        d1[16 * r + 4 * kb + i][col] = d;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < MLP_S / 4; k++) {
      const u32 s = 4 * k + kb;
      const float dd = d2[s][col];
#pragma unroll
      for (int m = 0; m < 4; m++) gW2[m] = mlp_mfma(a1[s][16 * m + n], dd, gW2[m]);
      gW1 = mlp_mfma(n < 8 ? xs[s][n & 7] : 0.f, d1[s][col], gW1);
    }
    __syncthreads();
  }
  float* G = part + (u64)blockIdx.x * P_TRAIN;
#pragma unroll
  for (int m = 0; m < 4; m++)
#pragma unroll
    for (int i = 0; i < 4; i++) G[P_W2 + (16 * m + 4 * kb + i) * MLP_H + col] = gW2[m][i];
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (4 * kb + i < 8) G[P_W1 + (4 * kb + i) * MLP_H + col] = gW1[i];
  for (int d = 16; d < 64; d <<= 1) {
    gb1 += __shfl_xor(gb1, d);
    gb2 += __shfl_xor(gb2, d);
    gw3 += __shfl_xor(gw3, d);
  }
  if (kb == 0) {
    G[P_B1 + col] = gb1;
    G[P_B2 + col] = gb2;
    G[P_W3 + col] = gw3;
  }
  if (t < 64) {
    for (int d = 1; d < 64; d <<= 1) {
      gb3 += __shfl_xor(gb3, d);
      ls += __shfl_xor(ls, d);
    }
    if (t == 0) {
      G[P_B3] = gb3;
      lossp[blockIdx.x] = ls;
    }
  }
}

// Adds the blocks' partial gradients (four interleaved shares per parameter,
// then the shares) and takes the Adam step, or leaves the gradient in G when
// m is null.  Block 0 also leaves the step's loss.
__global__ void __launch_bounds__(256) mlp_update(const float* __restrict__ part,
                                                  const float* __restrict__ lossp, u32 nblk,
                                                  float* __restrict__ P, float* __restrict__ G,
                                                  float* __restrict__ m, float* __restrict__ v,
                                                  float lr, float b1t, float b2t,
                                                  float* __restrict__ loss) {
  __shared__ float sh[4][64];
  const u32 c = threadIdx.x & 63, q = threadIdx.x >> 6, p = blockIdx.x * 64 + c;
  float s = 0.f;
  if (p < P_TRAIN) {
    u32 b = q;
    for (; b + 12 < nblk; b += 16) {
      const float s0 = part[(u64)b * P_TRAIN + p], s1 = part[(u64)(b + 4) * P_TRAIN + p];
      const float s2 = part[(u64)(b + 8) * P_TRAIN + p], s3 = part[(u64)(b + 12) * P_TRAIN + p];
      s += (s0 + s1) + (s2 + s3);
    }
    for (; b < nblk; b += 4) s += part[(u64)b * P_TRAIN + p];
  }
  sh[q][c] = s;
  __syncthreads();
  if (blockIdx.x == 0 && q == 1) {
    float x = 0.f;
    for (u32 b = c; b < nblk; b += 64) x += lossp[b];
    for (int d = 1; d < 64; d <<= 1) x += __shfl_xor(x, d);
    if (c == 0) *loss = x;
  }
  if (q || p >= P_TRAIN) return;
  const float g = (sh[0][c] + sh[1][c]) + (sh[2][c] + sh[3][c]);
  if (!m) {
    G[p] = g;
    return;
  }
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float mm = b1 * m[p] + (1.f - b1) * g;
  const float vv = b2 * v[p] + (1.f - b2) * g * g;
  m[p] = mm;
  v[p] = vv;
  const float mh = mm / (1.f - b1t), vh = vv / (1.f - b2t);
  P[P_W1 + p] -= lr * mh / (sqrtf(vh) + eps);
}

// Stand-alone inference with the engine's MFMA tile routine: 16 rows per wave
// and pass, the weights held in registers over a wave's passes.
// X: n x 6 raw features.
__global__ void __launch_bounds__(64) mlp_infer_k(const MlpDev* M, const float* __restrict__ X,
                                                  u32 n, float* __restrict__ out) {
  __shared__ __align__(8) u16 h1s[16 * MLP_H];
  const MlpRegs R{MlpMem(M)};
  for (u64 base = (u64)blockIdx.x * 16; base < n; base += (u64)gridDim.x * 16) {
    auto feat = [&](u32 row) {
      MlpFeat f{0, 0, 0, 0, 0, 0.f};
      const u64 r = base + row;
      if (r < n) {
        f.dC = (u32)X[r * MLP_IN + 0];
        f.dR = (u32)X[r * MLP_IN + 1];
        f.dist = (u32)X[r * MLP_IN + 2];
        f.core = (u32)X[r * MLP_IN + 3];
        f.slack = (int)X[r * MLP_IN + 4];
        f.cscore = X[r * MLP_IN + 5];
      }
      return f;
    };
    const float s = mlp_tile(R, feat, h1s);
    const u32 row = threadIdx.x & 15u;
    if (threadIdx.x < 16 && base + row < n) out[base + row] = s;
  }
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
static u16 host_f2bf(float f) {
  u32 x;
  memcpy(&x, &f, 4);
  x += 0x7fffu + ((x >> 16) & 1u);
  return (u16)(x >> 16);
}

void scs_pack_model(const scs_model* m, MlpDev* d) {
  memset(d, 0, sizeof(*d));
  for (int k = 0; k < 8; k++)
    for (int j = 0; j < MLP_H; j++) d->w1[j][k] = k < MLP_IN ? host_f2bf(m->w1[k][j]) : 0;
  for (int i = 0; i < MLP_H; i++)
    for (int j = 0; j < MLP_H; j++) d->w2[j][i] = host_f2bf(m->w2[i][j]);
  for (int j = 0; j < MLP_H; j++) {
    d->b1[j] = m->b1[j];
    d->b2[j] = m->b2[j];
    d->w3[j] = m->w3[j];
  }
  d->b3 = m->b3;
  for (int k = 0; k < 8; k++) {
    d->mean[k] = m->mean[k];
    d->scale[k] = m->scale[k];
  }
}

#define HCK(x)                          \
  do {                                  \
    if ((x) != hipSuccess) return SCS_EHIP; \
  } while (0)

extern "C" int scs_model_init(scs_model* m, uint64_t seed) {
  if (!m) return SCS_EINVAL;
  memset(m, 0, sizeof(*m));
  std::mt19937_64 rng(seed);
  std::normal_distribution<float> nd(0.f, 1.f);
  for (int k = 0; k < MLP_IN; k++)
    for (int j = 0; j < MLP_H; j++) m->w1[k][j] = nd(rng) * sqrtf(2.f / MLP_IN);
  for (int i = 0; i < MLP_H; i++)
    for (int j = 0; j < MLP_H; j++) m->w2[i][j] = nd(rng) * sqrtf(2.f / MLP_H);
  for (int j = 0; j < MLP_H; j++) m->w3[j] = nd(rng) * sqrtf(1.f / MLP_H);
  for (int k = 0; k < 8; k++) m->scale[k] = 1.f;
  return SCS_OK;
}

namespace {
// One device allocation cut into the arrays of a call, freed with it.
struct DevBlock {
  char* base = nullptr;
  u64 used = 0;
  ~DevBlock() {
    if (base) (void)hipFree(base);
  }
  u64 add(u64 bytes) {
    const u64 o = used;
    used = (used + bytes + 255) & ~255ull;
    return o;
  }
  int alloc() { return hipMalloc((void**)&base, used) == hipSuccess ? SCS_OK : SCS_EHIP; }
};
struct TrainBufs : DevBlock {
  float *P, *G, *M, *V, *X, *Y, *part, *lossp, *loss;
  u32* idx;
  u32 nblk;
  // n rows, batches of B, losses of `steps` steps, `nidx` row numbers
  int init(u32 n, u32 B, u32 steps, u64 nidx) {
    nblk = (B + MLP_S - 1) / MLP_S < MLP_MAXBLK ? (B + MLP_S - 1) / MLP_S : MLP_MAXBLK;
    const u64 oP = add(sizeof(float) * P_TOTAL), oG = add(sizeof(float) * P_TOTAL);
    const u64 oM = add(sizeof(float) * P_TOTAL), oV = add(sizeof(float) * P_TOTAL);
    const u64 oX = add(sizeof(float) * MLP_IN * (u64)n), oY = add(sizeof(float) * (u64)n);
    const u64 opart = add(sizeof(float) * P_TRAIN * (u64)nblk), olp = add(sizeof(float) * nblk);
    const u64 ol = add(sizeof(float) * (u64)steps), oi = add(sizeof(u32) * nidx);
    if (alloc()) return SCS_EHIP;
    P = (float*)(base + oP);
    G = (float*)(base + oG);
    M = (float*)(base + oM);
    V = (float*)(base + oV);
    X = (float*)(base + oX);
    Y = (float*)(base + oY);
    part = (float*)(base + opart);
    lossp = (float*)(base + olp);
    loss = (float*)(base + ol);
    idx = (u32*)(base + oi);
    return SCS_OK;
  }
  // gradient of B rows (row numbers idx); with adam also the update of P
  int step(const u32* rows, u32 B, float posw, float* out_loss, bool adam, float lr, float b1t,
           float b2t) {
    mlp_step<<<nblk, 256>>>(P, X, Y, rows, B, posw, part, lossp);
    HCK(hipGetLastError());
    mlp_update<<<(P_TRAIN + 63) / 64, 256>>>(part, lossp, nblk, P, G, adam ? M : nullptr,
                                             adam ? V : nullptr, lr, b1t, b2t, out_loss);
    HCK(hipGetLastError());
    return SCS_OK;
  }
};
}  // namespace

// Gradient of the mean weighted BCE over rows 0..n-1 (for checks).
extern "C" int scs_mlp_grad(const scs_model* m, const float* X, const float* y, uint32_t n,
                            float pos_weight, scs_model* grad, float* loss) {
  if (!m || !X || !y || !grad || n == 0) return SCS_EINVAL;
  TrainBufs T;
  int rc = T.init(n, n, 1, n);
  if (rc) return rc;
  HCK(hipMemcpy(T.P, m, sizeof(float) * P_TOTAL, hipMemcpyHostToDevice));
  HCK(hipMemcpy(T.X, X, sizeof(float) * MLP_IN * (u64)n, hipMemcpyHostToDevice));
  HCK(hipMemcpy(T.Y, y, sizeof(float) * (u64)n, hipMemcpyHostToDevice));
  std::vector<u32> idx(n);
  for (u32 i = 0; i < n; i++) idx[i] = i;
  HCK(hipMemcpy(T.idx, idx.data(), sizeof(u32) * n, hipMemcpyHostToDevice));
  rc = T.step(T.idx, n, pos_weight, T.loss, false, 0.f, 0.f, 0.f);
  if (rc) return rc;
  memset(grad, 0, sizeof(*grad));
  HCK(hipMemcpy(grad, T.G, sizeof(float) * P_TRAIN, hipMemcpyDeviceToHost));
  if (loss) HCK(hipMemcpy(loss, T.loss, sizeof(float), hipMemcpyDeviceToHost));
  return SCS_OK;
}

// Mini-batch Adam on the GPU.  Input normalisation (mean/scale) is taken
// from the data before training starts.  An epoch's row order goes up in one
// copy (which waits for the epoch before) and its steps are launched without
// waiting, so the host draws the next order meanwhile; the last epoch's
// losses come back at the end.
extern "C" int scs_mlp_train(scs_model* m, const float* X, const float* y, uint32_t n,
                             uint32_t epochs, uint32_t batch, float lr, float pos_weight,
                             uint64_t seed, float* final_loss) {
  if (!m || !X || !y || n == 0 || batch == 0) return SCS_EINVAL;
  {
    // the six sums side by side, each in row order
    double s[MLP_IN] = {}, s2[MLP_IN] = {};
    for (u64 i = 0; i < n; i++)
      for (int k = 0; k < MLP_IN; k++) {
        const float x = X[i * MLP_IN + k];
        s[k] += x;
        s2[k] += (double)x * x;
      }
    for (int k = 0; k < MLP_IN; k++) {
      const double mu = s[k] / n, var = s2[k] / n - mu * mu;
      m->mean[k] = (float)mu;
      m->scale[k] = var > 1e-12 ? (float)(1.0 / sqrt(var)) : 1.f;
    }
  }
  const u32 B = std::min<u32>(batch, n), per = n / B;
  TrainBufs T;
  int rc = T.init(n, B, per, n);
  if (rc) return rc;
  HCK(hipMemcpy(T.P, m, sizeof(float) * P_TOTAL, hipMemcpyHostToDevice));
  HCK(hipMemset(T.M, 0, sizeof(float) * P_TOTAL));
  HCK(hipMemset(T.V, 0, sizeof(float) * P_TOTAL));
  HCK(hipMemcpy(T.X, X, sizeof(float) * MLP_IN * (u64)n, hipMemcpyHostToDevice));
  HCK(hipMemcpy(T.Y, y, sizeof(float) * (u64)n, hipMemcpyHostToDevice));
  std::mt19937_64 rng(seed);
  std::vector<u32> perm(n);
  for (u32 i = 0; i < n; i++) perm[i] = i;
  u64 t = 0;
  for (u32 ep = 0; ep < epochs; ep++) {
    std::shuffle(perm.begin(), perm.end(), rng);
    HCK(hipMemcpy(T.idx, perm.data(), sizeof(u32) * n, hipMemcpyHostToDevice));
    for (u32 b = 0; b < per; b++) {
      t++;
      rc = T.step(T.idx + (u64)b * B, B, pos_weight, T.loss + b, true, lr,
                  (float)pow(0.9, (double)t), (float)pow(0.999, (double)t));
      if (rc) return rc;
    }
  }
  std::vector<float> losses(per);
  if (epochs) HCK(hipMemcpy(losses.data(), T.loss, sizeof(float) * per, hipMemcpyDeviceToHost));
  HCK(hipMemcpy(m, T.P, sizeof(float) * P_TRAIN, hipMemcpyDeviceToHost));
  double sum = 0;
  for (float x : losses) sum += x;
  if (final_loss) *final_loss = epochs ? (float)(sum / per) : 0.f;
  return SCS_OK;
}

extern "C" int scs_mlp_infer(const scs_model* m, const float* X, uint32_t n, float* scores) {
  if (!m || !X || !scores || n == 0) return SCS_EINVAL;
  MlpDev h;
  scs_pack_model(m, &h);
  DevBlock D;
  const u64 om = D.add(sizeof(MlpDev)), ox = D.add(sizeof(float) * MLP_IN * (u64)n);
  const u64 oo = D.add(sizeof(float) * (u64)n);
  if (D.alloc()) return SCS_EHIP;
  HCK(hipMemcpy(D.base + om, &h, sizeof(MlpDev), hipMemcpyHostToDevice));
  HCK(hipMemcpy(D.base + ox, X, sizeof(float) * MLP_IN * (u64)n, hipMemcpyHostToDevice));
  // four waves per SIMD at most: more would only load the weights again
  const u32 tiles = (u32)(((u64)n + 15) / 16);
  mlp_infer_k<<<tiles < 4096 ? tiles : 4096, 64>>>((const MlpDev*)(D.base + om),
                                                   (const float*)(D.base + ox), n,
                                                   (float*)(D.base + oo));
  HCK(hipGetLastError());
  HCK(hipMemcpy(scores, D.base + oo, sizeof(float) * n, hipMemcpyDeviceToHost));
  return SCS_OK;
}
