// mlp.hip -- the learned warm-start network on gfx950: per-row MLP
// 24 -> 128 -> 128 -> 3 or 6 (ReLU) with BF16 weights and activations and FP32
// accumulation on the CDNA4 matrix cores (v_mfma_f32_16x16x32_bf16):
// hand-written forward, activation-gradient and split-K weight-gradient
// kernels, and Adam on the f32 master copy.
//
// The reference has no learned warm start; the network, its inputs and the
// fallback rule are this backend's own (avbd.h, learned.hip).
//
// MFMA 16x16x32 BF16 operand layouts (lane l of a wave64):
//   A (16 x 32, rows x k):  row l % 16, k = 8 (l / 16) + j, j = 0..7
//   B (32 x 16, k x cols):  col l % 16, k = 8 (l / 16) + j
//   D (16 x 16, f32):       col l % 16, row = 4 (l / 16) + i, i = 0..3
// so every operand fetch is one 16-byte load of 8 consecutive k.
//
// Rounding points (what a CPU restatement must reproduce): the inputs, the
// weights, the hidden activations h1 = bf16(relu(.)), h2 = bf16(relu(.)),
// and in the backward pass dY, dZ2 and dZ1 are rounded to bf16 (round to
// nearest even) before they feed a product; bias gradients use the f32 values.
#include "mlp.hpp"

namespace avbd {

typedef __bf16 bf16;
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kIn = kMlpIn, kInPad = kMlpInPad, kHid = kMlpHidden, kOutPad = kMlpOutPad;
// LDS row strides (bf16 elements): 80 B / 272 B rows put the 16 rows
// of one operand fetch on 16 distinct 4-bank groups
constexpr int kS1 = 40, kSH = 136, kSD = 40;

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x8 ld8(const bf16* p) { return *(const bf16x8*)p; }
__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int j = 0; j < 8; j++) z[j] = (bf16)0.0f;
  return z;
}
__device__ __forceinline__ f32x4 zero4() { return f32x4{0.0f, 0.0f, 0.0f, 0.0f}; }
// LDS writes of one lane visible to the other lanes of its wave
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Weights as the kernels read them (bf16; global arrays dense, LDS copies padded):
//   w1t [kHid][kInPad]   layer-1 B operand (output-major, inputs contiguous)
//   w2t [kHid][kHid]     layer-2 B operand (output-major)
//   w3t [kOutPad][kHid]  layer-3 B operand (output-major)
//   w2  [kHid][kHid]     backward B operand of dH1 = dZ2 W2^T (input-major)
//   w3  [kHid][kOutPad]  backward B operand of dH2 = dY W3^T (input-major)
struct LdsFwd {
  bf16 w1t[kHid * kS1];
  bf16 w2t[kHid * kSH];
  bf16 w3t[kOutPad * kSH];
};
// copy a dense [rows][cols] bf16 matrix into LDS rows of `stride` (16-byte chunks)
__device__ void stage(bf16* dst, const bf16* src, int rows, int cols, int stride) {
  const int chunks = cols / 8;
  for (int i = threadIdx.x; i < rows * chunks; i += blockDim.x) {
    int r = i / chunks, c = i % chunks;
    *(bf16x8*)(dst + r * stride + 8 * c) = *(const bf16x8*)(src + r * cols + 8 * c);
  }
}

__device__ void load_fwd(const MlpDevice& M, LdsFwd& L) {
  stage(L.w1t, M.w1t, kHid, kInPad, kS1);
  stage(L.w2t, M.w2t, kHid, kHid, kSH);
  stage(L.w3t, M.w3t, kOutPad, kHid, kSH);
}
// Forward of one 16-row tile by one wave.  h1, h2: the wave's [16][kSH] LDS
// rows, left holding the bf16 activations.  Returns the layer-3 accumulator
// (D layout) plus bias.
__device__ f32x4 tile_forward(const MlpDevice& M, const LdsFwd& W, const bf16* X, uint32_t rows, uint32_t r0,
                              bf16* h1, bf16* h2, uint32_t lane) {
  const uint32_t ar = lane & 15u, ak = 8u * (lane >> 4), dr = 4u * (lane >> 4);
  bf16x8 a1 = (r0 + ar < rows) ? ld8(X + (size_t)(r0 + ar) * kInPad + ak) : zero8();
#pragma unroll
  for (int nt = 0; nt < kHid / 16; nt++) {
    f32x4 acc = mfma(a1, ld8(W.w1t + (nt * 16 + ar) * kS1 + ak), zero4());
    const uint32_t col = nt * 16 + ar;
    const float b = M.b1[col];
#pragma unroll
    for (int i = 0; i < 4; i++) h1[(dr + i) * kSH + col] = (bf16)fmaxf(acc[i] + b, 0.0f);
  }
  wave_sync();
#pragma unroll
  for (int nt = 0; nt < kHid / 16; nt++) {
    f32x4 acc = zero4();
#pragma unroll
    for (int kt = 0; kt < kHid / 32; kt++)
      acc = mfma(ld8(h1 + ar * kSH + kt * 32 + ak), ld8(W.w2t + (nt * 16 + ar) * kSH + kt * 32 + ak), acc);
    const uint32_t col = nt * 16 + ar;
    const float b = M.b2[col];
#pragma unroll
    for (int i = 0; i < 4; i++) h2[(dr + i) * kSH + col] = (bf16)fmaxf(acc[i] + b, 0.0f);
  }
  wave_sync();
  f32x4 acc = zero4();
#pragma unroll
  for (int kt = 0; kt < kHid / 32; kt++)
    acc = mfma(ld8(h2 + ar * kSH + kt * 32 + ak), ld8(W.w3t + ar * kSH + kt * 32 + ak), acc);
  const float b3 = M.b3[ar];
#pragma unroll
  for (int i = 0; i < 4; i++) acc[i] += b3;
  return acc;
}

// one feature of 16 LDS rows, 32 contiguous bytes of its row in dst[f * P + r0 ..]
__device__ __forceinline__ void store_transposed(const bf16* h, int stride, uint32_t f, bf16* dst, size_t P,
                                                 uint32_t r0) {
  bf16x8 lo, hi;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    lo[j] = h[j * stride + f];
    hi[j] = h[(8 + j) * stride + f];
  }
  *(bf16x8*)(dst + (size_t)f * P + r0) = lo;
  *(bf16x8*)(dst + (size_t)f * P + r0 + 8) = hi;
}

}  // namespace

// ---------------------------------------------------------------------------
// inference: Y[r][0..nOut) = MLP(X[r]), X bf16 [rows][32], Y f32 [rows][nOut];
// 8 waves share one LDS copy of the weights
// ---------------------------------------------------------------------------
constexpr int kFwdWaves = 8;
__global__ void __launch_bounds__(64 * kFwdWaves) k_mlp_forward(MlpDevice M, const bf16* X, uint32_t rows, float* Y) {
  __shared__ LdsFwd W;
  __shared__ bf16 hbuf[kFwdWaves][2][16 * kSH];
  load_fwd(M, W);
  __syncthreads();
  const uint32_t wv = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  const uint32_t tiles = (rows + 15) / 16;
  for (uint32_t t = blockIdx.x * kFwdWaves + wv; t < tiles; t += gridDim.x * kFwdWaves) {
    const uint32_t r0 = t * 16;
    f32x4 y = tile_forward(M, W, X, rows, r0, hbuf[wv][0], hbuf[wv][1], lane);
    const uint32_t col = lane & 15u;
    if (col < M.nOut) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        uint32_t r = r0 + 4 * (lane >> 4) + i;
        if (r < rows) Y[(size_t)r * M.nOut + col] = y[i];
      }
    }
    wave_sync();  // the next tile overwrites h1 / h2
  }
}

// ---------------------------------------------------------------------------
// training, pass 1: forward + activation gradients of
// L = sum_r |y_r - t_r|^2 * lossScale over every 16-row tile of the padded
// batch (rows >= `rows` carry zero gradient; row r is dataset row perm[r], or
// r without perm); writes the feature-major operands of the weight-gradient
// GEMMs and the workgroup's parts of the bias gradients and of sum |y - t|^2.
//
// A workgroup owns a tile and each of its four waves two of the eight column
// tiles of every layer, so the weights a wave multiplies fit its registers:
// they are read once, all loads in flight together, straight from the L2.
// One wave per tile needs every weight, staged through 86 KB of LDS: at 4096
// rows that filled 64 CUs, was bound by the staging, and took 21 us (15 us
// with the bias sums added atomically, 11 us writing parts).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_mlp_act_grad(MlpDevice M, MlpTrain T, const bf16* X, const float* Tgt,
                                                      const uint32_t* perm, uint32_t rows, float lossScale) {
  __shared__ bf16 h1[16 * kSH], h2[16 * kSH], dz[16 * kSD];
  const uint32_t tid = threadIdx.x, wv = tid >> 6, lane = tid & 63u;
  const uint32_t ar = lane & 15u, ak = 8u * (lane >> 4), dr = 4u * (lane >> 4);
  constexpr int kN = 2, kK = kHid / 32;  // column tiles of a wave, k steps of a hidden layer
  bf16x8 w1[kN], w2[kN][kK], w3[kK], v3t[kN], v2[kN][kK];
  float b1[kN], b2[kN], db1[kN], db2[kN], db3 = 0.0f, loss = 0.0f;
#pragma unroll
  for (int c = 0; c < kN; c++) {
    const uint32_t col = (kN * wv + c) * 16 + ar;
    w1[c] = ld8(M.w1t + col * kInPad + ak);
    v3t[c] = lane < 32 ? ld8(M.w3 + col * kOutPad + ak) : zero8();  // k = outputs, zero beyond 16
#pragma unroll
    for (int kt = 0; kt < kK; kt++) {
      w2[c][kt] = ld8(M.w2t + col * kHid + kt * 32 + ak);
      v2[c][kt] = ld8(M.w2 + col * kHid + kt * 32 + ak);
    }
    b1[c] = M.b1[col];
    b2[c] = M.b2[col];
    db1[c] = db2[c] = 0.0f;
  }
#pragma unroll
  for (int kt = 0; kt < kK; kt++) w3[kt] = ld8(M.w3t + ar * kHid + kt * 32 + ak);
  const float b3 = M.b3[ar];
  const size_t P = T.rowsPad;
  const uint32_t tiles = T.rowsPad / 16;
  for (uint32_t t = blockIdx.x; t < tiles; t += gridDim.x) {
    const uint32_t r0 = t * 16, row = r0 + ar;
    const uint32_t src = row >= rows ? 0u : perm ? perm[row] : row;
    const bf16x8 a1 = row < rows ? ld8(X + (size_t)src * kInPad + ak) : zero8();
#pragma unroll
    for (int c = 0; c < kN; c++) {
      const f32x4 acc = mfma(a1, w1[c], zero4());
#pragma unroll
      for (int i = 0; i < 4; i++)
        h1[(dr + i) * kSH + (kN * wv + c) * 16 + ar] = (bf16)fmaxf(acc[i] + b1[c], 0.0f);
    }
    if (wv == 3u) {  // feature-major copy of X: a lane's operand is one row's 8 features
#pragma unroll
      for (int j = 0; j < 8; j++) T.xt[(size_t)(ak + j) * P + row] = a1[j];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kN; c++) {
      f32x4 acc = zero4();
#pragma unroll
      for (int kt = 0; kt < kK; kt++) acc = mfma(ld8(h1 + ar * kSH + kt * 32 + ak), w2[c][kt], acc);
#pragma unroll
      for (int i = 0; i < 4; i++)
        h2[(dr + i) * kSH + (kN * wv + c) * 16 + ar] = (bf16)fmaxf(acc[i] + b2[c], 0.0f);
    }
    __syncthreads();
    if (wv == 0u) {
      f32x4 y = zero4();
#pragma unroll
      for (int kt = 0; kt < kK; kt++) y = mfma(ld8(h2 + ar * kSH + kt * 32 + ak), w3[kt], y);
      // dY = 2 (y - t) lossScale (D layout; columns >= nOut and padded rows are zero)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t from = (uint32_t)__shfl((int)src, (int)(dr + i));
        float g = 0.0f;
        if (r0 + dr + i < rows && ar < M.nOut) {
          float e = y[i] + b3 - Tgt[(size_t)from * M.nOut + ar];
          loss += e * e;
          g = 2.0f * e * lossScale;
        }
        db3 += g;
        dz[(dr + i) * kSD + ar] = (bf16)g;
        dz[(dr + i) * kSD + 16 + ar] = (bf16)0.0f;
      }
    }
    if (tid < (uint32_t)kHid) store_transposed(h1, kSH, tid, T.h1t, P, r0);
    else store_transposed(h2, kSH, tid - kHid, T.h2t, P, r0);
    __syncthreads();  // dY is written, and the transposed reads of h2 precede its in-place update
    if (tid < (uint32_t)kOutPad) store_transposed(dz, kSD, tid, T.dyt, P, r0);
    // dH2 = dY W3^T; dZ2 = dH2 (h2 > 0) replaces h2 in place
    const bf16x8 ady = ld8(dz + ar * kSD + ak);
#pragma unroll
    for (int c = 0; c < kN; c++) {
      const f32x4 acc = mfma(ady, v3t[c], zero4());
#pragma unroll
      for (int i = 0; i < 4; i++) {
        bf16& h = h2[(dr + i) * kSH + (kN * wv + c) * 16 + ar];
        const float g = ((float)h > 0.0f && r0 + dr + i < rows) ? acc[i] : 0.0f;
        db2[c] += g;
        h = (bf16)g;  // each (row, col) is read and written by this lane only
      }
    }
    __syncthreads();
    if (tid < (uint32_t)kHid) store_transposed(h2, kSH, tid, T.dz2t, P, r0);
    // dH1 = dZ2 W2^T; dZ1 = dH1 (h1 > 0), then replaces h1
#pragma unroll
    for (int c = 0; c < kN; c++) {
      f32x4 acc = zero4();
#pragma unroll
      for (int kt = 0; kt < kK; kt++) acc = mfma(ld8(h2 + ar * kSH + kt * 32 + ak), v2[c][kt], acc);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        bf16& h = h1[(dr + i) * kSH + (kN * wv + c) * 16 + ar];
        const float g = ((float)h > 0.0f && r0 + dr + i < rows) ? acc[i] : 0.0f;
        db1[c] += g;
        h = (bf16)g;  // h1 is not an operand of this product
      }
    }
    __syncthreads();
    if (tid >= (uint32_t)kHid) store_transposed(h1, kSH, tid - kHid, T.dz1t, P, r0);
    __syncthreads();  // the next tile overwrites h1 / h2 / dz
  }
  // bias gradients: the four row groups of each column, then this workgroup's part
  float* part = T.gb + blockIdx.x;
  const uint32_t parts = gridDim.x;
#pragma unroll
  for (int c = 0; c < kN; c++) {
    float a = db1[c], b = db2[c];
    a += __shfl_xor(a, 16, 64);
    a += __shfl_xor(a, 32, 64);
    b += __shfl_xor(b, 16, 64);
    b += __shfl_xor(b, 32, 64);
    if (lane < 16) {
      const uint32_t col = (kN * wv + c) * 16 + lane;
      part[col * parts] = a;
      part[(kHid + col) * parts] = b;
    }
  }
  if (wv != 0u) return;
  db3 += __shfl_xor(db3, 16, 64);
  db3 += __shfl_xor(db3, 32, 64);
  if (lane < 16) part[(2 * kHid + lane) * parts] = db3;
  for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o, 64);
  if (lane == 0) part[(kMlpGb - 1u) * parts] = loss;
}

// ---------------------------------------------------------------------------
// training, pass 2: weight gradients as split-K GEMMs over the samples,
//   gW1 = Xt dZ1t^T (32 x 128), gW2 = H1t dZ2t^T (128 x 128), gW3 = H2t dYt^T (128 x 16);
// 88 output tiles of 16 x 16, one per wave (blockIdx.y: 22 groups of 4),
// blockIdx.x owns a range of samples (a multiple of 32) and writes part
// blockIdx.x of the sums
// ---------------------------------------------------------------------------
constexpr int kGradTiles = 2 * 8 + 8 * 8 + 8;
constexpr uint32_t kGw2 = kInPad * kHid, kGw3 = kGw2 + kHid * kHid;  // gW2 and gW3 in a part
__global__ void __launch_bounds__(256) k_mlp_wgrad(MlpTrain T, uint32_t samplesPerBlock) {
  const uint32_t wv = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  const uint32_t ar = lane & 15u, ak = 8u * (lane >> 4), dr = 4u * (lane >> 4);
  const size_t P = T.rowsPad;
  const uint32_t k0 = blockIdx.x * samplesPerBlock;
  const uint32_t k1 = min((uint32_t)P, k0 + samplesPerBlock);
  const int tile = blockIdx.y * 4 + wv;
  if (tile >= kGradTiles) return;
  const bf16 *At, *Bt;
  float* G = T.gw + (size_t)blockIdx.x * kMlpGw;
  uint32_t mt, nt, ldG;
  if (tile < 16) { At = T.xt; Bt = T.dz1t; mt = tile / 8; nt = tile % 8; ldG = kHid; }
  else if (tile < 80) { int q = tile - 16; At = T.h1t; Bt = T.dz2t; G += kGw2; mt = q / 8; nt = q % 8; ldG = kHid; }
  else { int q = tile - 80; At = T.h2t; Bt = T.dyt; G += kGw3; mt = q; nt = 0; ldG = kOutPad; }
  const bf16* ap = At + (size_t)(mt * 16 + ar) * P + ak;
  const bf16* bp = Bt + (size_t)(nt * 16 + ar) * P + ak;
  f32x4 acc = zero4();
  uint32_t k = k0;
  for (; k + 128 <= k1; k += 128) {  // eight loads in flight
    bf16x8 a[4], b[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a[j] = ld8(ap + k + 32 * j);
      b[j] = ld8(bp + k + 32 * j);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) acc = mfma(a[j], b[j], acc);
  }
  for (; k < k1; k += 32) acc = mfma(ld8(ap + k), ld8(bp + k), acc);
#pragma unroll
  for (int i = 0; i < 4; i++) G[(mt * 16 + dr + i) * ldG + nt * 16 + ar] = acc[i];
}

// The tail of a gradient: sums the parts of every gradient entry.  UPDATE: one
// training step's Adam (beta1 0.9, beta2 0.999, eps 1e-8) on the f32 master
// parameters, the bf16 operand layouts and f32 biases of the updated values,
// and the batch's share of the epoch's mean loss; otherwise the gradient in the
// master layout and the loss.
//
// The parts are added in the order of their workgroups, so a training run
// repeats bit for bit: float atomics added them as they arrived, and the
// thousand steps of an epoch of small batches amplified the last bits of the
// bias gradients to 6 percent of the parameters.  A thread owns a weight and a
// wave a bias (of up to kMlpRowParts parts, or the loss).  4096 rows (16 and 256
// parts) take 3.6 us, as an update of sums added atomically did (3.3 us): 20099
// parameters are nothing but a launch, and it replaces five of 2.3 to 4.2 us.
template <bool UPDATE>
__global__ void __launch_bounds__(256) k_mlp_sum(MlpDevice M, MlpTrain T, uint32_t weightParts, uint32_t rowParts,
                                                 uint32_t weightBlocks, float lr, float b1c, float b2c, float* lossDst,
                                                 float lossScale) {
  const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
  const uint32_t nOut = M.nOut, offB3 = (uint32_t)mlp_off_b3((int)nOut);
  uint32_t i;
  float g = 0.0f, m0 = 0.0f, v0 = 0.0f, p0 = 0.0f;
  auto fetch = [&]() {  // in flight beside the parts
    m0 = T.m[i];
    v0 = T.v[i];
    p0 = M.params[i];
  };
  if (blockIdx.x < weightBlocks) {
    constexpr uint32_t n1 = kIn * kHid, n2 = kHid * kHid;  // rows 0..23 of gW1 [32][128]
    const uint32_t w = blockIdx.x * 256u + threadIdx.x;
    if (w >= n1 + n2 + kHid * nOut) return;
    uint32_t q;
    if (w < n1) {
      i = q = w;
    } else if (w < n1 + n2) {
      i = kMlpOffW2 + (w - n1);
      q = kGw2 + (w - n1);
    } else {
      const uint32_t r = w - n1 - n2;
      i = kMlpOffW3 + r;
      q = kGw3 + r / nOut * kOutPad + r % nOut;
    }
    if (UPDATE) fetch();
    const float* p = T.gw + q;
#pragma unroll 8
    for (uint32_t k = 0; k < weightParts; k++) g += p[(size_t)k * kMlpGw];
  } else {
    const uint32_t c = (blockIdx.x - weightBlocks) * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (c > 2u * kHid + nOut) return;
    const bool isLoss = c == 2u * kHid + nOut;
    i = c < (uint32_t)kHid ? kMlpOffB1 + c : c < 2u * kHid ? kMlpOffB2 + (c - kHid) : offB3 + (c - 2u * kHid);
    if (UPDATE && !isLoss) fetch();
    const float* p = T.gb + (size_t)(isLoss ? kMlpGb - 1u : c) * rowParts;
#pragma unroll
    for (uint32_t k = 0; k < kMlpRowParts / 64u; k++)
      if (lane + 64u * k < rowParts) g += p[lane + 64u * k];
    for (int o = 32; o > 0; o >>= 1) g += __shfl_xor(g, o, 64);
    if (lane != 0u) return;
    if (isLoss) {
      if (UPDATE) lossDst[0] += g * lossScale;
      else T.loss[0] = g;
      return;
    }
  }
  if (!UPDATE) {
    T.grad[i] = g;
    return;
  }
  const float m = beta1 * m0 + (1.0f - beta1) * g;
  const float v = beta2 * v0 + (1.0f - beta2) * g * g;
  T.m[i] = m;
  T.v[i] = v;
  const float p = p0 - lr * (m / b1c) / (sqrtf(v / b2c) + eps);
  M.params[i] = p;
  // the padding of the operand layouts is zero since k_mlp_pack
  if (i < (uint32_t)kMlpOffB1) {
    M.w1t[(i % kHid) * kInPad + i / kHid] = (bf16)p;
  } else if (i < (uint32_t)kMlpOffW2) {
    M.b1[i - kMlpOffB1] = p;
  } else if (i < (uint32_t)kMlpOffB2) {
    const uint32_t q = i - kMlpOffW2;  // W2[in][out]
    M.w2[q] = (bf16)p;
    M.w2t[(q % kHid) * kHid + q / kHid] = (bf16)p;
  } else if (i < (uint32_t)kMlpOffW3) {
    M.b2[i - kMlpOffB2] = p;
  } else if (i < offB3) {
    const uint32_t a = (i - kMlpOffW3) / nOut, b = (i - kMlpOffW3) % nOut;
    M.w3[a * kOutPad + b] = (bf16)p;
    M.w3t[b * kHid + a] = (bf16)p;
  } else {
    M.b3[i - offB3] = p;
  }
}

// bf16 operand layouts and f32 biases from the f32 master parameters
__global__ void __launch_bounds__(256) k_mlp_pack(MlpDevice M) {
  const float* p = M.params;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < (uint32_t)(kHid * kHid); i += gridDim.x * blockDim.x) {
    const uint32_t a = i / kHid, b = i % kHid;
    const float w = p[kMlpOffW2 + a * kHid + b];  // W2[in a][out b]
    M.w2[a * kHid + b] = (bf16)w;
    M.w2t[b * kHid + a] = (bf16)w;
    if (a < (uint32_t)kInPad) {
      const float w1 = a < (uint32_t)kIn ? p[kMlpOffW1 + a * kHid + b] : 0.0f;  // W1[in a][out b]
      M.w1t[b * kInPad + a] = (bf16)w1;
    }
    if (b < (uint32_t)kOutPad) {
      const float w3 = b < M.nOut ? p[kMlpOffW3 + a * M.nOut + b] : 0.0f;  // W3[in a][out b]
      M.w3[a * kOutPad + b] = (bf16)w3;
      M.w3t[b * kHid + a] = (bf16)w3;
    }
    if (a == 0) {
      M.b1[b] = p[kMlpOffB1 + b];
      M.b2[b] = p[kMlpOffB2 + b];
      if (b < (uint32_t)kOutPad) M.b3[b] = b < M.nOut ? p[mlp_off_b3((int)M.nOut) + b] : 0.0f;
    }
  }
}

// f32 rows [n][24] -> bf16 rows [n][32]
__global__ void __launch_bounds__(256) k_mlp_pack_input(const float* Xf, uint32_t n, bf16* X) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n * (uint32_t)kInPad; i += gridDim.x * blockDim.x) {
    const uint32_t r = i / kInPad, c = i % kInPad;
    X[i] = (bf16)(c < (uint32_t)kIn ? Xf[(size_t)r * kIn + c] : 0.0f);
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static uint32_t grid_for(uint32_t work, uint32_t cap) {
  uint32_t b = (work + 255) / 256;
  return b == 0 ? 1 : (b > cap ? cap : b);
}

void launch_mlp_pack(hipStream_t st, const MlpDevice& M) {
  hipLaunchKernelGGL(k_mlp_pack, dim3(64), dim3(256), 0, st, M);
}
void launch_mlp_pack_input(hipStream_t st, const float* Xf, uint32_t n, void* X) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_mlp_pack_input, dim3(grid_for(n * kInPad, 2048)), dim3(256), 0, st, Xf, n, (bf16*)X);
}
void launch_mlp_forward(hipStream_t st, const MlpDevice& M, const void* X, uint32_t rows, float* Y, uint32_t cus) {
  if (rows == 0) return;
  const uint32_t tiles = (rows + 15) / 16;
  uint32_t blocks = (tiles + kFwdWaves - 1) / kFwdWaves;
  if (blocks > cus) blocks = cus;  // one 8-wave block per CU (LDS), tiles strided over the grid
  hipLaunchKernelGGL(k_mlp_forward, dim3(blocks), dim3(64 * kFwdWaves), 0, st, M, (const bf16*)X, rows, Y);
}
// parts of a batch: of its bias sums (workgroups of k_mlp_act_grad) and of its
// weight sums (ranges of samplesPerBlock).  4096 rows: the weight gradients take
// 6 us on 352 workgroups of 256 rows with eight loads in flight a wave (11 us
// on 88 of 1024 rows, two at a time)
static uint32_t row_parts(uint32_t rowsPad, uint32_t cus) {
  return std::min(rowsPad / 16u, std::min(2u * cus, kMlpRowParts));
}
static uint32_t weight_rows(uint32_t rowsPad) {
  const uint32_t spb = (rowsPad + kMlpWeightParts - 1) / kMlpWeightParts;
  return std::max(256u, (spb + 31u) / 32u * 32u);
}
static uint32_t weight_parts(uint32_t rowsPad) {
  return (rowsPad + weight_rows(rowsPad) - 1) / weight_rows(rowsPad);
}
void launch_mlp_backprop(hipStream_t st, const MlpDevice& M, const MlpTrain& T, const void* X, const float* Tgt,
                         const uint32_t* perm, uint32_t rows, uint32_t cus) {
  const float scale = 1.0f / ((float)M.nOut * (float)(rows > 0 ? rows : 1));
  hipLaunchKernelGGL(k_mlp_act_grad, dim3(row_parts(T.rowsPad, cus)), dim3(256), 0, st, M, T, (const bf16*)X, Tgt, perm,
                     rows, scale);
  hipLaunchKernelGGL(k_mlp_wgrad, dim3(weight_parts(T.rowsPad), (kGradTiles + 3) / 4), dim3(256), 0, st, T,
                     weight_rows(T.rowsPad));
}
template <bool UPDATE>
static void launch_sum(hipStream_t st, const MlpDevice& M, const MlpTrain& T, uint32_t cus, float lr, float b1c,
                       float b2c, float* lossDst, float lossScale) {
  const uint32_t weights = (kIn + kHid + M.nOut) * kHid, wb = (weights + 255) / 256;
  const uint32_t waves = 2 * kHid + M.nOut + 1;
  hipLaunchKernelGGL((k_mlp_sum<UPDATE>), dim3(wb + (waves + 3) / 4), dim3(256), 0, st, M, T, weight_parts(T.rowsPad),
                     row_parts(T.rowsPad, cus), wb, lr, b1c, b2c, lossDst, lossScale);
}
void launch_mlp_gather_grad(hipStream_t st, const MlpDevice& M, const MlpTrain& T, uint32_t cus) {
  launch_sum<false>(st, M, T, cus, 0.0f, 1.0f, 1.0f, nullptr, 0.0f);
}
void launch_mlp_update(hipStream_t st, const MlpDevice& M, const MlpTrain& T, uint32_t cus, float lr, int step,
                       float* lossDst, float lossScale) {
  const float b1c = 1.0f - powf(0.9f, (float)step), b2c = 1.0f - powf(0.999f, (float)step);
  launch_sum<true>(st, M, T, cus, lr, b1c, b2c, lossDst, lossScale);
}

}  // namespace avbd
