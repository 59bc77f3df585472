// Small MLP that scores SPR moves (32 features -> 128 -> 128 -> 1, GELU), with
// hand-written training and inference kernels: BF16-input / FP32-accumulate
// MFMA GEMMs (v_mfma_f32_16x16x32_bf16), FP32 master weights and Adam.
// The reference has no learned component; this serves the learned SPR
// proposal that re-ranks TreeNeighborhoods moves (lib/treeNeighborhoods.ml).
//
// Parameters (flat FP32): W1[n_in][H] b1[H] W2[H][H] b2[H] w3[H] b3[1].
// Loss: 0.5 * mean((y - t)^2).
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "rng.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct phy_mlp {
  phy_ctx* ctx = nullptr;
  int n_in = 32, H = 128;
  int64_t n_params = 0;
  float *params = nullptr, *grads = nullptr, *m1 = nullptr, *m2 = nullptr;
  int64_t step = 0;
  // activations for up to cap rows: Z1 H1 Z2 H2 [cap][H], y [cap], dy, dH [cap][H] x2
  float* act = nullptr;
  int64_t cap = 0;
  // partial results of the split-K weight-gradient GEMMs and column sums
  float* ws = nullptr;
  int64_t ws_floats = 0;
};

namespace {

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
  const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
  const float pdf = 0.3989422804014327f * expf(-0.5f * x * x);
  return cdf + x * pdf;
}

// C[M][N] (+)= op(A)[M][K] op(B)[K][N] (+ bias[n]), A at A[m*sam + k*sak],
// B at B[k*sbk + n*sbn], C row-major with ldc.  One wave per 16x16 tile;
// operands are rounded to BF16, accumulation is FP32.  Split K: workgroup z
// takes k in [z * kps, (z + 1) * kps) and writes its partial tile at
// Cm + z * c_split (the caller sums the splits).
__global__ __launch_bounds__(64) void k_gemm(const float* __restrict__ A, int64_t sam, int64_t sak,
                                             const float* __restrict__ B, int64_t sbk, int64_t sbn,
                                             float* __restrict__ Cm, int64_t ldc, int M, int N, int K,
                                             int accumulate, const float* __restrict__ bias,
                                             int kps = 1 << 30, int64_t c_split = 0) {
  const int l = threadIdx.x, q = l >> 4, r16 = l & 15;
  const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 16;
  const int am = m0 + r16, bn = n0 + r16;
  const int kb = (int)blockIdx.z * kps, ke = min(K, kb + kps);
  Cm += (int64_t)blockIdx.z * c_split;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = kb; k0 < ke; k0 += 32) {
    bf16x8 a, b;
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const int k = k0 + 8 * q + v;
      const bool ka = k < ke;
      a[v] = (__bf16)((ka && am < M) ? A[(int64_t)am * sam + (int64_t)k * sak] : 0.0f);
      b[v] = (__bf16)((ka && bn < N) ? B[(int64_t)k * sbk + (int64_t)bn * sbn] : 0.0f);
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
  }
  // lane l holds C[m0 + 4q + v][n0 + l%16]
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int m = m0 + 4 * q + v, n = n0 + r16;
    if (m < M && n < N) {
      float x = acc[v] + (bias ? bias[n] : 0.0f);
      float* c = Cm + (int64_t)m * ldc + n;
      *c = accumulate ? *c + x : x;
    }
  }
}

__global__ void k_gelu_fwd(const float* __restrict__ Z, float* __restrict__ Hh, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) Hh[i] = gelu(Z[i]);
}

// y[m] = H2[m] . w3 + b3  (FP32 dot product: the 128 -> 1 layer is a GEMV)
__global__ void k_out(const float* __restrict__ H2, const float* __restrict__ w3,
                      const float* __restrict__ b3, float* __restrict__ y, int64_t M, int H) {
  const int64_t m = (int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  const int l = threadIdx.x & 63;
  if (m >= M) return;
  float s = 0.f;
  for (int j = l; j < H; j += 64) s += H2[m * H + j] * w3[j];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (l == 0) y[m] = s + b3[0];
}

// dy = (y - t) / B; loss partials; dH2 = dy * w3; db3, dw3 accumulated later
__global__ void k_loss(const float* __restrict__ y, const float* __restrict__ t, float* __restrict__ dy,
                       double* __restrict__ loss, int64_t M) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double e = 0.0;
  if (m < M) {
    const float d = y[m] - t[m];
    dy[m] = d / (float)M;
    e = 0.5 * (double)d * (double)d / (double)M;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off, 64);
  if ((threadIdx.x & 63) == 0 && loss) atomicAdd(loss, e);
}

// dZ[m][j] = (dy[m] * w3[j] or dH[m][j]) * gelu'(Z[m][j])
__global__ void k_gelu_bwd(const float* __restrict__ dH, const float* __restrict__ dy,
                           const float* __restrict__ w3, const float* __restrict__ Z,
                           float* __restrict__ dZ, int64_t M, int H) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M * H) return;
  const int64_t m = i / H;
  const int j = (int)(i % H);
  const float g = dH ? dH[i] : dy[m] * w3[j];
  dZ[i] = g * gelu_grad(Z[i]);
}

// out[i] = sum over s < splits of part[s * n + i] (fixed order), written or
// added to out
__global__ void k_sum_splits(const float* __restrict__ part, int splits, int64_t n,
                             float* __restrict__ out, int accumulate) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
  for (int z = 0; z < splits; ++z) s += part[(int64_t)z * n + i];
  out[i] = accumulate ? out[i] + s : s;
}

// column sums by row chunks: part[c][j] = sum of X[m][j] over the rows of
// chunk c (threads over columns: coalesced rows)
__global__ void k_colsum_chunks(const float* __restrict__ X, int64_t M, int H, int64_t rows,
                                float* __restrict__ part) {
  const int64_t c = blockIdx.x;
  const int64_t m0 = c * rows, m1 = min(M, m0 + rows);
  for (int j = threadIdx.x; j < H; j += blockDim.x) {
    float s = 0.f;
    for (int64_t m = m0; m < m1; ++m) s += X[m * H + j];
    part[c * H + j] = s;
  }
}

__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1,
                       float* __restrict__ m2, int64_t n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.f - b1) * gi;
  const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  p[i] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// ---------------------------------------------------------------------------
// Fused pass for small networks (n_in <= 64, H = 64 or 128): forward, or
// forward + backward, of 32 rows of the batch at a time with every activation
// on chip.
//
// A block is H / 16 waves; wave w owns hidden units 16w .. 16w+15 of both
// layers and holds its slices of W1, W2^T and W2 as BF16 MFMA operands in
// registers for the whole launch.  Products are formed transposed (A = weights,
// B = activations), so a lane holds 4 units (16w + 4q + v) of one row (lane
// l: row l % 16 of each 16-row group, q = l / 16): GELU, its derivative, the
// loss and the bias / output-layer sums run in FP32 registers, and only the
// BF16 operands of the next product pass through LDS.  Weight gradients
// contract over the rows (one K = 32 MFMA step a tile) from unit-major copies,
// accumulate in registers over the block's tiles and leave as one partial
// per block, summed in a fixed order by k_mlp_sum.
//
// One wave per 16x16 tile with activations in memory (the k_gemm path below)
// spent 219 us on 65,536 rows forward and 1.25 ms backward, in strided 4-byte
// loads and 19 launches; here 20 us forward (one launch) and 89 us forward and
// backward (two launches); 1,024 rows forward and backward take 18 us.  The
// bound is the VALU: two erff a row and hidden unit (ocml's two branches, ~40
// instructions each) forward, two erff and two expf more backward.
// ---------------------------------------------------------------------------
constexpr int kMlpRows = 32;     // rows of a tile (the K of the weight gradients)
constexpr int kMlpMaxIn = 64;

struct MlpArgs {
  const float *X, *T, *W1, *b1, *W2, *b2, *w3, *b3;
  float* y;      // forward: outputs (backward: nullptr)
  float* part;   // backward: [blocks][n_params] gradient partials
  double* lpart; // backward: [blocks] loss partials
  int64_t B, n_params;
  int n_in, vec4;  // vec4: rows of X can be read 16 bytes at a time
};

__device__ __forceinline__ f32x4 mfma16(const bf16x8 a, const bf16x8 b, const f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// sum over the 16 lanes of a row (every lane gets it)
__device__ __forceinline__ float row16_sum(float v) {
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// W = waves per block = H / 16; KC = 32-feature chunks of the input
template <int W, int KC, bool BWD>
__global__ __launch_bounds__(64 * W) void k_mlp_fused(MlpArgs a) {
  constexpr int H = 16 * W, HC = H / 32, G = kMlpRows / 16;
  constexpr int RS = H + 8;         // row-major stride (bf16): 16-byte rows, staggered banks
  constexpr int US = kMlpRows + 8;  // unit-major stride
  __shared__ __attribute__((aligned(16))) __bf16 hr[kMlpRows * RS];  // H1, then dZ2, [row][unit]
  __shared__ float ys[W][kMlpRows];
  __shared__ __attribute__((aligned(16))) __bf16 ht[BWD ? H * US : 8];   // H1 [unit][row]
  __shared__ __attribute__((aligned(16))) __bf16 d2t[BWD ? H * US : 8];  // dZ2 [unit][row]
  __shared__ __attribute__((aligned(16))) __bf16 d1t[BWD ? H * US : 8];  // dZ1 [unit][row]
  __shared__ __attribute__((aligned(16))) __bf16 xt[BWD ? 32 * KC * US : 8];  // X [feature][row]
  const int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = l >> 4, c = l & 15;
  const int u0 = 16 * w + 4 * q;  // the lane's 4 units

  bf16x8 a1[KC], a2[HC], a2t[BWD ? HC : 1];
#pragma unroll
  for (int k = 0; k < KC; ++k)
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const int i = 32 * k + 8 * q + v;
      a1[k][v] = (__bf16)(i < a.n_in ? a.W1[(int64_t)i * H + 16 * w + c] : 0.0f);
    }
#pragma unroll
  for (int k = 0; k < HC; ++k)
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const int i = 32 * k + 8 * q + v;
      a2[k][v] = (__bf16)a.W2[i * H + 16 * w + c];
      if (BWD) a2t[k][v] = (__bf16)a.W2[(16 * w + c) * H + i];
    }
  float b1[4], b2[4], w3[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    b1[v] = a.b1[u0 + v];
    b2[v] = a.b2[u0 + v];
    w3[v] = a.w3[u0 + v];
  }
  const float b3 = a.b3[0];

  f32x4 gW2[BWD ? W : 1], gW1[BWD ? 2 * KC : 1];
  float gb1[4] = {0.f, 0.f, 0.f, 0.f}, gb2[4] = {0.f, 0.f, 0.f, 0.f}, gw3[4] = {0.f, 0.f, 0.f, 0.f}, gb3 = 0.f;
  double loss = 0.0;
#pragma unroll
  for (int j = 0; j < (BWD ? W : 1); ++j) gW2[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < (BWD ? 2 * KC : 1); ++j) gW1[j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int64_t tiles = (a.B + kMlpRows - 1) / kMlpRows;
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const int64_t row0 = tile * kMlpRows;
    // layer 1; the activations' derivatives stay in registers
    float g1[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int64_t row = row0 + 16 * g + c;
      const float* x = a.X + (row < a.B ? row : a.B - 1) * a.n_in;
      f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        const int i0 = 32 * k + 8 * q;
        float xv[8];
        if (a.vec4) {  // n_in is a multiple of 4 and the rows are 16-byte aligned
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            float4 t4 = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i0 + 4 * h < a.n_in) t4 = *reinterpret_cast<const float4*>(x + i0 + 4 * h);
            xv[4 * h] = t4.x;
            xv[4 * h + 1] = t4.y;
            xv[4 * h + 2] = t4.z;
            xv[4 * h + 3] = t4.w;
          }
        } else {
#pragma unroll
          for (int v = 0; v < 8; ++v) xv[v] = i0 + v < a.n_in ? x[i0 + v] : 0.0f;
        }
        bf16x8 b;
#pragma unroll
        for (int v = 0; v < 8; ++v) b[v] = (__bf16)xv[v];
        z = mfma16(a1[k], b, z);
        if (BWD && w == 0) {  // unit-major copy for dW1; rows past the batch meet dZ1 = 0
#pragma unroll
          for (int v = 0; v < 8; ++v) xt[(i0 + v) * US + 16 * g + c] = b[v];
        }
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float zv = z[v] + b1[v];
        const __bf16 h = (__bf16)gelu(zv);
        hr[(16 * g + c) * RS + u0 + v] = h;
        if (BWD) {
          ht[(u0 + v) * US + 16 * g + c] = h;
          g1[g][v] = gelu_grad(zv);
        }
      }
    }
    __syncthreads();
    // layer 2 and the output layer
    float z2[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < HC; ++k)
        z = mfma16(a2[k], *reinterpret_cast<const bf16x8*>(&hr[(16 * g + c) * RS + 32 * k + 8 * q]), z);
      float s = 0.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        z2[g][v] = z[v] + b2[v];
        s += gelu(z2[g][v]) * w3[v];
      }
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      if (q == 0) ys[w][16 * g + c] = s;
    }
    __syncthreads();
    if (!BWD) {
      // hr is rewritten only after this barrier (every wave has read it), ys
      // only after the next tile's first barrier
      if (threadIdx.x < kMlpRows && row0 + threadIdx.x < a.B) {
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < W; ++k) s += ys[k][threadIdx.x];
        a.y[row0 + threadIdx.x] = s + b3;
      }
      continue;
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int64_t row = row0 + 16 * g + c;
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < W; ++k) s += ys[k][16 * g + c];
      const float d = row < a.B ? (s + b3) - a.T[row] : 0.0f;
      const float dy = d / (float)a.B, dyb = (float)(__bf16)dy;
      if (w == 0 && q == 0) {
        loss += 0.5 * (double)d * (double)d / (double)a.B;
        gb3 += dy;
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float zv = z2[g][v];
        gw3[v] += (float)(__bf16)gelu(zv) * dyb;  // BF16 operands, as the GEMM path's
        const float dz = dy * w3[v] * gelu_grad(zv);
        gb2[v] += dz;
        const __bf16 h = (__bf16)dz;
        hr[(16 * g + c) * RS + u0 + v] = h;
        d2t[(u0 + v) * US + 16 * g + c] = h;
      }
    }
    __syncthreads();
    // dZ1 = (W2 dZ2) * gelu'(Z1)
#pragma unroll
    for (int g = 0; g < G; ++g) {
      f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < HC; ++k)
        z = mfma16(a2t[k], *reinterpret_cast<const bf16x8*>(&hr[(16 * g + c) * RS + 32 * k + 8 * q]), z);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float dz = z[v] * g1[g][v];
        gb1[v] += dz;
        d1t[(u0 + v) * US + 16 * g + c] = (__bf16)dz;
      }
    }
    // dW2 (units of layer 1 of this wave x every unit of layer 2)
    {
      const bf16x8 ah = *reinterpret_cast<const bf16x8*>(&ht[(16 * w + c) * US + 8 * q]);
#pragma unroll
      for (int j = 0; j < W; ++j)
        gW2[j] = mfma16(ah, *reinterpret_cast<const bf16x8*>(&d2t[(16 * j + c) * US + 8 * q]), gW2[j]);
    }
    __syncthreads();  // d1t written; hr, ht, d2t read
    // dW1 (every feature x the units of this wave)
    {
      const bf16x8 bd = *reinterpret_cast<const bf16x8*>(&d1t[(16 * w + c) * US + 8 * q]);
#pragma unroll
      for (int j = 0; j < 2 * KC; ++j)
        gW1[j] = mfma16(*reinterpret_cast<const bf16x8*>(&xt[(16 * j + c) * US + 8 * q]), bd, gW1[j]);
    }
    __syncthreads();  // xt read
  }
  if (!BWD) return;
  // the block's partial gradient, laid out as the parameters
  float* p = a.part + (int64_t)blockIdx.x * a.n_params;
#pragma unroll
  for (int j = 0; j < 2 * KC; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = 16 * j + 4 * q + v;
      if (i < a.n_in) p[(int64_t)i * H + 16 * w + c] = gW1[j][v];
    }
  p += (int64_t)a.n_in * H;
  float* pW2 = p + H;
#pragma unroll
  for (int j = 0; j < W; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v) pW2[(int64_t)(u0 + v) * H + 16 * j + c] = gW2[j][v];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float s1 = row16_sum(gb1[v]), s2 = row16_sum(gb2[v]), s3 = row16_sum(gw3[v]);
    if (c == 0) {
      p[u0 + v] = s1;
      pW2[(int64_t)H * H + u0 + v] = s2;
      pW2[(int64_t)H * H + H + u0 + v] = s3;
    }
  }
  if (w == 0) {
    const float s = row16_sum(q == 0 ? gb3 : 0.f);
    double e = q == 0 ? loss : 0.0;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) e += __shfl_xor(e, off, 64);
    if (l == 0) {
      pW2[(int64_t)H * H + 2 * H] = s;
      a.lpart[blockIdx.x] = e;
    }
  }
}

// Sums of the per-block partials in a fixed order: 64 parameters a block,
// the partials dealt to its 4 waves.  The last block of the grid sums the
// loss.  out2 (nullable) receives a second copy of the gradients.
__global__ __launch_bounds__(256) void k_mlp_sum(const float* __restrict__ part, int parts, int64_t n,
                                                 const double* __restrict__ lpart, float* __restrict__ out,
                                                 float* __restrict__ out2, double* __restrict__ loss) {
  __shared__ float sh[4][64];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (blockIdx.x == gridDim.x - 1) {
    if (threadIdx.x == 0 && loss) {
      double e = 0.0;
      for (int z = 0; z < parts; ++z) e += lpart[z];
      *loss = e;
    }
    return;
  }
  const int64_t i = (int64_t)blockIdx.x * 64 + l;
  float s = 0.f;
  if (i < n) {
#pragma unroll 8
    for (int z = w; z < parts; z += 4) s += part[(int64_t)z * n + i];
  }
  sh[w][l] = s;
  __syncthreads();
  if (w == 0 && i < n) {
    s = (sh[0][l] + sh[1][l]) + (sh[2][l] + sh[3][l]);
    out[i] = s;
    if (out2) out2[i] = s;
  }
}

struct Views {
  float *W1, *b1, *W2, *b2, *w3, *b3;
};
Views views(float* base, int n_in, int H) {
  Views v;
  v.W1 = base;
  v.b1 = v.W1 + (int64_t)n_in * H;
  v.W2 = v.b1 + H;
  v.b2 = v.W2 + (int64_t)H * H;
  v.w3 = v.b2 + H;
  v.b3 = v.w3 + H;
  return v;
}

// split-K plan of a weight gradient (reduction over K = the batch): enough
// workgroups to fill the chip, each a multiple of 32 rows long
struct SplitK {
  int splits, kps;
};
SplitK split_k(int64_t K, int tiles) {
  SplitK s;
  const int64_t want = std::max<int64_t>(1, std::min<int64_t>((4096 + tiles - 1) / tiles, (K + 255) / 256));
  s.kps = (int)((((K + want - 1) / want) + 31) / 32 * 32);
  s.splits = (int)((K + s.kps - 1) / s.kps);
  return s;
}

// grad (M x N, ldc = N) = A^T B over K rows, split over K into m->ws, then summed
int grad_gemm(phy_ctx* ctx, phy_mlp* m, const float* A, int64_t lda, const float* Bm, int64_t ldb,
              float* grad, int M, int N, int64_t K) {
  const dim3 t((unsigned)((N + 15) / 16), (unsigned)((M + 15) / 16));
  const SplitK s = split_k(K, (int)(t.x * t.y));
  const int64_t n = (int64_t)M * N;
  hipLaunchKernelGGL(k_gemm, dim3(t.x, t.y, (unsigned)s.splits), dim3(64), 0, ctx->stream, A, (int64_t)1,
                     lda, Bm, ldb, (int64_t)1, m->ws, (int64_t)N, M, N, (int)K, 0, (const float*)nullptr,
                     s.kps, n);
  hipLaunchKernelGGL(k_sum_splits, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, m->ws,
                     s.splits, n, grad, 0);
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

// out[j] = sum_m X[m][j], by row chunks into m->ws, then summed
int colsum(phy_ctx* ctx, phy_mlp* m, const float* X, int64_t M, int H, float* out) {
  const int64_t rows = std::max<int64_t>(64, (M + 1023) / 1024);
  const int64_t chunks = (M + rows - 1) / rows;
  hipLaunchKernelGGL(k_colsum_chunks, dim3((unsigned)chunks), dim3(std::min(H, 256)), 0, ctx->stream, X, M,
                     H, rows, m->ws);
  hipLaunchKernelGGL(k_sum_splits, dim3((unsigned)((H + 255) / 256)), dim3(256), 0, ctx->stream, m->ws,
                     (int)chunks, (int64_t)H, out, 0);
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

int ensure_cap(phy_mlp* m, int64_t B) {
  if (B <= m->cap) return PHY_OK;
  if (m->act) PHY_HIP(m->ctx, hipFree(m->act));
  m->act = nullptr;
  const int64_t cap = std::max<int64_t>(B, 1024);
  PHY_HIP(m->ctx, hipMalloc((void**)&m->act, sizeof(float) * (size_t)cap * (6 * m->H + 2)));
  m->cap = cap;
  return PHY_OK;
}

inline dim3 tiles(int M, int N) { return dim3((unsigned)((N + 15) / 16), (unsigned)((M + 15) / 16)); }

// forward; activations kept for backward
int forward(phy_ctx* ctx, phy_mlp* m, const float* X, int64_t B, float* y) {
  const int H = m->H, n_in = m->n_in;
  Views p = views(m->params, n_in, H);
  float* Z1 = m->act;
  float* H1 = Z1 + m->cap * H;
  float* Z2 = H1 + m->cap * H;
  float* H2 = Z2 + m->cap * H;
  const int Mi = (int)B;
  KernelSpan span(ctx, "mlp_forward");
  hipLaunchKernelGGL(k_gemm, tiles(Mi, H), dim3(64), 0, ctx->stream, X, (int64_t)n_in, (int64_t)1, p.W1,
                     (int64_t)H, (int64_t)1, Z1, (int64_t)H, Mi, H, n_in, 0, p.b1, 1 << 30, (int64_t)0);
  const int64_t nh = B * H;
  hipLaunchKernelGGL(k_gelu_fwd, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, ctx->stream, Z1, H1, nh);
  hipLaunchKernelGGL(k_gemm, tiles(Mi, H), dim3(64), 0, ctx->stream, H1, (int64_t)H, (int64_t)1, p.W2,
                     (int64_t)H, (int64_t)1, Z2, (int64_t)H, Mi, H, H, 0, p.b2, 1 << 30, (int64_t)0);
  hipLaunchKernelGGL(k_gelu_fwd, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, ctx->stream, Z2, H2, nh);
  hipLaunchKernelGGL(k_out, dim3((unsigned)((B + 3) / 4)), dim3(256), 0, ctx->stream, H2, p.w3, p.b3, y, B, H);
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

int backward(phy_ctx* ctx, phy_mlp* m, const float* X, const float* t, int64_t B, double* loss) {
  const int H = m->H, n_in = m->n_in;
  Views p = views(m->params, n_in, H);
  Views g = views(m->grads, n_in, H);
  float* Z1 = m->act;
  float* H1 = Z1 + m->cap * H;
  float* Z2 = H1 + m->cap * H;
  float* H2 = Z2 + m->cap * H;
  float* dZ2 = H2 + m->cap * H;
  float* dH1 = dZ2 + m->cap * H;  // reused as dZ1
  float* y = dH1 + m->cap * H;
  float* dy = y + m->cap;
  const int Mi = (int)B;
  int rc = forward(ctx, m, X, B, y);
  if (rc) return rc;
  KernelSpan span(ctx, "mlp_backward");
  hipLaunchKernelGGL(k_loss, dim3((unsigned)((B + 255) / 256)), dim3(256), 0, ctx->stream, y, t, dy, loss, B);
  // output layer: dw3 = H2^T dy (GEMM with N = 1), db3 = sum dy
  if ((rc = grad_gemm(ctx, m, H2, H, dy, 1, g.w3, H, 1, B))) return rc;
  if ((rc = colsum(ctx, m, dy, B, 1, g.b3))) return rc;
  const int64_t nh = B * H;
  hipLaunchKernelGGL(k_gelu_bwd, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, ctx->stream,
                     (const float*)nullptr, dy, p.w3, Z2, dZ2, B, H);
  // dW2 = H1^T dZ2 ; db2 = colsum dZ2 ; dH1 = dZ2 W2^T
  if ((rc = grad_gemm(ctx, m, H1, H, dZ2, H, g.W2, H, H, B))) return rc;
  if ((rc = colsum(ctx, m, dZ2, B, H, g.b2))) return rc;
  hipLaunchKernelGGL(k_gemm, tiles(Mi, H), dim3(64), 0, ctx->stream, dZ2, (int64_t)H, (int64_t)1, p.W2,
                     (int64_t)1, (int64_t)H, dH1, (int64_t)H, Mi, H, H, 0, (const float*)nullptr,
                     1 << 30, (int64_t)0);
  // dZ1 = dH1 * gelu'(Z1) (in place) ; dW1 = X^T dZ1 ; db1 = colsum dZ1
  hipLaunchKernelGGL(k_gelu_bwd, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, ctx->stream, dH1,
                     (const float*)nullptr, (const float*)nullptr, Z1, dH1, B, H);
  if ((rc = grad_gemm(ctx, m, X, n_in, dH1, H, g.W1, n_in, H, B))) return rc;
  if ((rc = colsum(ctx, m, dH1, B, H, g.b1))) return rc;
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

// The fused pass covers networks of up to 64 inputs with 64 or 128 hidden
// units (its weights fit a block's registers); other sizes take the GEMMs.
bool fused_fits(const phy_mlp* m) { return m->n_in <= kMlpMaxIn && (m->H == 64 || m->H == 128); }

// blocks of a fused launch, at most one per tile of rows: backward one a CU
// (each leaves a partial gradient, 84 KB at H = 128), forward three (what its
// registers keep resident; 65,536 rows: 28.5 / 22.1 / 20.3 / 22.4 us at
// 1 / 2 / 3 / 4 a CU)
int fused_blocks(const phy_ctx* ctx, int64_t B, bool bwd) {
  int n_cu = 256;
  (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, ctx->device);
  return (int)std::min<int64_t>((B + kMlpRows - 1) / kMlpRows, (int64_t)n_cu * (bwd ? 1 : 3));
}

MlpArgs fused_args(const phy_mlp* m, const float* X, const float* T, int64_t B) {
  const Views p = views(m->params, m->n_in, m->H);
  MlpArgs a{};
  a.X = X;
  a.T = T;
  a.W1 = p.W1;
  a.b1 = p.b1;
  a.W2 = p.W2;
  a.b2 = p.b2;
  a.w3 = p.w3;
  a.b3 = p.b3;
  a.B = B;
  a.n_params = m->n_params;
  a.n_in = m->n_in;
  a.vec4 = m->n_in % 4 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0;
  return a;
}

template <bool BWD>
void fused_launch(phy_ctx* ctx, const phy_mlp* m, int blocks, const MlpArgs& a) {
  const bool wide = m->n_in > 32;
  const dim3 g((unsigned)blocks), t((unsigned)(4 * m->H));
  if (m->H == 128) {
    if (wide)
      hipLaunchKernelGGL((k_mlp_fused<8, 2, BWD>), g, t, 0, ctx->stream, a);
    else
      hipLaunchKernelGGL((k_mlp_fused<8, 1, BWD>), g, t, 0, ctx->stream, a);
  } else {
    if (wide)
      hipLaunchKernelGGL((k_mlp_fused<4, 2, BWD>), g, t, 0, ctx->stream, a);
    else
      hipLaunchKernelGGL((k_mlp_fused<4, 1, BWD>), g, t, 0, ctx->stream, a);
  }
}

int ensure_ws(phy_ctx* ctx, phy_mlp* m, int64_t need) {
  if (m->ws_floats >= need) return PHY_OK;
  if (m->ws) PHY_HIP(ctx, hipFree(m->ws));
  m->ws = nullptr;
  m->ws_floats = 0;
  PHY_HIP(ctx, hipMalloc((void**)&m->ws, sizeof(float) * (size_t)need));
  m->ws_floats = need;
  return PHY_OK;
}

int fused_forward(phy_ctx* ctx, phy_mlp* m, const float* X, int64_t B, float* y) {
  MlpArgs a = fused_args(m, X, nullptr, B);
  a.y = y;
  KernelSpan span(ctx, "mlp_forward");
  fused_launch<false>(ctx, m, fused_blocks(ctx, B, false), a);
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

int fused_backward(phy_ctx* ctx, phy_mlp* m, const float* X, const float* T, int64_t B, float* d_grads,
                   double* d_loss) {
  const int blocks = fused_blocks(ctx, B, true);
  // loss partials (8-byte aligned) ahead of the gradient partials
  const int rc = ensure_ws(ctx, m, 2 * (int64_t)blocks + blocks * m->n_params);
  if (rc) return rc;
  MlpArgs a = fused_args(m, X, T, B);
  a.lpart = reinterpret_cast<double*>(m->ws);
  a.part = m->ws + 2 * (int64_t)blocks;
  KernelSpan span(ctx, "mlp_backward");
  fused_launch<true>(ctx, m, blocks, a);
  PHY_LAUNCHED(ctx);
  hipLaunchKernelGGL(k_mlp_sum, dim3((unsigned)((m->n_params + 63) / 64 + 1)), dim3(256), 0, ctx->stream, a.part,
                     blocks, m->n_params, a.lpart, m->grads, d_grads, d_loss);
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

}  // namespace

extern "C" {

int phy_mlp_create(phy_ctx* ctx, int32_t n_in, int32_t n_hidden, uint64_t seed, phy_mlp** out) {
  if (!ctx || !out) return PHY_EINVAL;
  *out = nullptr;
  if (n_in < 1 || n_in > 4096 || n_hidden < 16 || n_hidden > 4096 || n_hidden % 16)
    return set_err(ctx, PHY_EINVAL, "mlp: n_in in 1..4096, n_hidden a multiple of 16");
  phy_mlp* m = new phy_mlp();
  m->ctx = ctx;
  m->n_in = n_in;
  m->H = n_hidden;
  m->n_params = (int64_t)n_in * n_hidden + n_hidden + (int64_t)n_hidden * n_hidden + n_hidden + n_hidden + 1;
  // He-style initialisation on the host, deterministic in seed
  std::vector<float> p((size_t)m->n_params, 0.0f);
  phy::Rng r(seed, 17);
  Views v = views(p.data(), n_in, n_hidden);
  for (int64_t i = 0; i < (int64_t)n_in * n_hidden; ++i) v.W1[i] = (float)(r.normal() * std::sqrt(2.0 / n_in));
  for (int64_t i = 0; i < (int64_t)n_hidden * n_hidden; ++i) v.W2[i] = (float)(r.normal() * std::sqrt(2.0 / n_hidden));
  for (int i = 0; i < n_hidden; ++i) v.w3[i] = (float)(r.normal() * std::sqrt(1.0 / n_hidden));
  const size_t bytes = sizeof(float) * (size_t)m->n_params;
  hipError_t e = hipMalloc((void**)&m->params, bytes);
  if (e == hipSuccess) e = hipMalloc((void**)&m->grads, bytes);
  if (e == hipSuccess) e = hipMalloc((void**)&m->m1, bytes);
  if (e == hipSuccess) e = hipMalloc((void**)&m->m2, bytes);
  if (e == hipSuccess) e = hipMemcpy(m->params, p.data(), bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(m->m1, 0, bytes);
  if (e == hipSuccess) e = hipMemset(m->m2, 0, bytes);
  if (e == hipSuccess) e = hipMemset(m->grads, 0, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    phy_mlp_destroy(m);
    return set_err(ctx, PHY_ENOMEM, "mlp: device allocation failed");
  }
  *out = m;
  return PHY_OK;
}

void phy_mlp_destroy(phy_mlp* m) {
  if (!m) return;
  if (m->params) (void)hipFree(m->params);
  if (m->grads) (void)hipFree(m->grads);
  if (m->m1) (void)hipFree(m->m1);
  if (m->m2) (void)hipFree(m->m2);
  if (m->act) (void)hipFree(m->act);
  if (m->ws) (void)hipFree(m->ws);
  delete m;
}

int64_t phy_mlp_n_params(const phy_mlp* m) { return m ? m->n_params : 0; }

int phy_mlp_get_params(phy_ctx* ctx, const phy_mlp* m, float* h_out) {
  if (!ctx || !m || !h_out) return PHY_EINVAL;
  PHY_HIP(ctx, hipMemcpyAsync(h_out, m->params, sizeof(float) * m->n_params, hipMemcpyDeviceToHost, ctx->stream));
  PHY_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return PHY_OK;
}

int phy_mlp_set_params(phy_ctx* ctx, phy_mlp* m, const float* h_in) {
  if (!ctx || !m || !h_in) return PHY_EINVAL;
  PHY_HIP(ctx, hipMemcpyAsync(m->params, h_in, sizeof(float) * m->n_params, hipMemcpyHostToDevice, ctx->stream));
  PHY_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return PHY_OK;
}

int phy_mlp_forward(phy_ctx* ctx, phy_mlp* m, const float* d_x, int64_t B, float* d_y) {
  if (!ctx || !m || !d_x || !d_y || B < 0) return PHY_EINVAL;
  if (B == 0) return PHY_OK;
  if (B > (1 << 30)) return set_err(ctx, PHY_ERANGE, "mlp: batch too large");
  if (fused_fits(m)) return fused_forward(ctx, m, d_x, B, d_y);
  int rc = ensure_cap(m, B);
  if (rc) return rc;
  return forward(ctx, m, d_x, B, d_y);
}

int phy_mlp_backward(phy_ctx* ctx, phy_mlp* m, const float* d_x, const float* d_t, int64_t B,
                     float* d_grads, double* d_loss) {
  if (!ctx || !m || !d_x || !d_t || B < 1) return PHY_EINVAL;
  if (B > (1 << 30)) return set_err(ctx, PHY_ERANGE, "mlp: batch too large");
  if (fused_fits(m)) return fused_backward(ctx, m, d_x, d_t, B, d_grads, d_loss);
  int rc = ensure_cap(m, B);
  if (rc) return rc;
  {
    // split-K partials of the three weight gradients, and the column-sum chunks
    const int H = m->H;
    auto part = [&](int M, int N) {
      const SplitK s = split_k(B, ((N + 15) / 16) * ((M + 15) / 16));
      return (int64_t)s.splits * M * N;
    };
    const int64_t rows = std::max<int64_t>(64, (B + 1023) / 1024);
    const int64_t need = std::max({part(H, 1), part(H, H), part(m->n_in, H),
                                   ((B + rows - 1) / rows) * (int64_t)H});
    if ((rc = ensure_ws(ctx, m, need))) return rc;
  }
  if (d_loss && (rc = phy_zero_u64(ctx, reinterpret_cast<uint64_t*>(d_loss), 1))) return rc;
  rc = backward(ctx, m, d_x, d_t, B, d_loss);
  if (rc) return rc;
  if (d_grads)
    PHY_HIP(ctx, hipMemcpyAsync(d_grads, m->grads, sizeof(float) * m->n_params, hipMemcpyDeviceToDevice, ctx->stream));
  return PHY_OK;
}

int phy_mlp_step(phy_ctx* ctx, phy_mlp* m, const float* d_x, const float* d_t, int64_t B, float lr,
                 double* d_loss) {
  int rc = phy_mlp_backward(ctx, m, d_x, d_t, B, nullptr, d_loss);
  if (rc) return rc;
  m->step += 1;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - std::pow(b1, (float)m->step), c2 = 1.0f - std::pow(b2, (float)m->step);
  hipLaunchKernelGGL(k_adam, dim3((unsigned)((m->n_params + 255) / 256)), dim3(256), 0, ctx->stream,
                     m->params, m->grads, m->m1, m->m2, m->n_params, lr, b1, b2, 1e-8f, c1, c2);
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

}  // extern "C"
