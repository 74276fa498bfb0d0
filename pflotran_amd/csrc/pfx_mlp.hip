// Learned warm start of the batched reaction step (include/pfx_surrogate.h):
// a multilayer perceptron whose matrix products run on the gfx950 matrix
// cores (v_mfma_f32_16x16x32_bf16: BF16 operands, FP32 accumulation).
//
//  * training, layers up to CHAIN_WIDTH wide: three launches a step.  One
//    kernel takes 16 rows through every layer forward and back with the
//    activations in LDS, one forms all layers' weight and bias gradients over
//    slices of the batch, one adds the slices, applies Adam to the FP32 master
//    weights and rewrites their BF16 fragments;
//  * training, wider layers: a tiled BF16 GEMM (64x64 block tile, 2x2 MFMA
//    tiles per wavefront) with fused bias/GELU epilogue for the forward pass,
//    the same GEMM on transposed operands (split-K, atomic FP32 accumulation)
//    for the weight gradients, elementwise GELU backward, then the same Adam;
//  * inference: one fused kernel per 64 cells that computes the features,
//    keeps every activation in LDS (BF16, two ping-pong buffers), streams
//    the weights from L2 in the exact MFMA fragment order (pre-swizzled,
//    one 16-byte load per lane per fragment), and writes the FP64 Newton
//    guess.  Inference computes D = W x X^T: rows are output features and
//    columns are cells, so each lane ends with 4 consecutive features of
//    one cell and stores them as one 8-byte LDS write.
//
// MFMA 16x16x32 operand layout used throughout (lane l of 64):
//   A (16 x 32): row l%16, k = 8*(l/16) + 0..7
//   B (32 x 16): col l%16, k = 8*(l/16) + 0..7
//   D (16 x 16): col l%16, rows 4*(l/16) + 0..3
// (the k order inside a fragment only has to agree between A and B).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/pfx_surrogate.h"
#include "pfx_device.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define MLP_MAX_LAYERS 8

struct pfx_mlp {
  int nlayers;
  int dims[MLP_MAX_LAYERS + 1];
  float *W[MLP_MAX_LAYERS], *b[MLP_MAX_LAYERS];  // FP32 master, W[l]: [dims[l+1]][dims[l]]
  float *gW[MLP_MAX_LAYERS], *gb[MLP_MAX_LAYERS];
  float *mW[MLP_MAX_LAYERS], *vW[MLP_MAX_LAYERS], *mb[MLP_MAX_LAYERS], *vb[MLP_MAX_LAYERS];
  uint4 *Wsw[MLP_MAX_LAYERS];   // BF16 weights in MFMA fragment order
  uint4 *Wtsw[MLP_MAX_LAYERS];  // the same of W transposed (backward chain)
  float *in_shift, *in_scale, *out_shift, *out_scale;
  int bmax;
  float *Z[MLP_MAX_LAYERS];      // pre-activations (or gelu' there) [bmax][dims[l+1]]
  float *A[MLP_MAX_LAYERS + 1];  // activations; A[0] is the caller's input
  // layers up to CHAIN_WIDTH wide (Z, A and dZl rows padded to 4 floats)
  float *dZl[MLP_MAX_LAYERS];  // [bmax][dims[l+1]]
  float *part;                 // gradient slices [gsplit(bmax)][params]
  float *lpart;                // loss of each 16 rows
  // wider layers
  float *dA, *dZ;  // [bmax][max width]
  float *loss;
  int adam_step;
};

namespace {

#define MCHK(x)                                                               \
  do {                                                                        \
    hipError_t e_ = (x);                                                      \
    if (e_ != hipSuccess) {                                                   \
      fprintf(stderr, "pfx_mlp: %s failed: %s (%s:%d)\n", #x,                 \
              hipGetErrorString(e_), __FILE__, __LINE__);                     \
      return PFX_E_DEVICE;                                                    \
    }                                                                         \
  } while (0)

__host__ __device__ inline int roundup(int v, int m) { return (v + m - 1) / m * m; }

// FP32 -> BF16, round to nearest even (finite inputs)
__device__ __forceinline__ unsigned short f2bf(float f) {
  unsigned int u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// gelu for the fused inference, without branches: z Phi(z) with
// Phi(-t) = exp(-t^2/2) R(t) for t >= 0 and Phi(t) = 1 - Phi(-t), R a
// polynomial in s = 1/(1 + 0.32 t), fitted to erfcx(t/sqrt 2)/2 by reweighted
// least squares (3e-9 in Phi).  Against 64 bits over normal and uniform z in
// [-6, 6] the result is off by 3.8e-7 at most and 5.3e-8 rms, the form with erff by
// 4.5e-7 and 5.8e-8; about 25 issue slots where erff's two ranges took 80, which
// bounded the kernel (its 768 values a cell).  Training, and plain inference with
// its kernel, keep erff: the slope from the shared exponential would be off by
// 2.1e-7 (now 1.4e-7), and the GELUs are 2 of that kernel's 27 us.
__device__ __forceinline__ float gelu_tail(float z) {
  const float t = fabsf(z);
  const float s = __builtin_amdgcn_rcpf(fmaf(0.32f, t, 1.0f));
  const float e = __builtin_amdgcn_exp2f(z * z * -0.72134752f);
  float r = 0.04403404171357539f;
  r = fmaf(r, s, -0.23251810874648504f);
  r = fmaf(r, s, 0.39190461034610413f);
  r = fmaf(r, s, -0.14902075637082102f);
  r = fmaf(r, s, 0.20831288338966916f);
  r = fmaf(r, s, 0.10789852993782426f);
  r = fmaf(r, s, 0.12938879668537376f);
  const float q = r * s * e;
  return z * (z >= 0.0f ? 1.0f - q : q);
}

// two values rounded to BF16 by the conversion instruction (nearest even, as f2bf)
__device__ __forceinline__ unsigned int pack_bf(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(unsigned int, v);
}

// gelu and its derivative from one erf
__device__ __forceinline__ float gelu_both(float z, float &slope) {
  const float e = 1.0f + erff(z * 0.70710678118654752f);
  slope = 0.5f * e + z * 0.39894228040143268f * expf(-0.5f * z * z);
  return 0.5f * z * e;
}

__device__ __forceinline__ bf16x8 as_frag(uint4 u) { return __builtin_bit_cast(bf16x8, u); }

__device__ __forceinline__ float slog(double v) {
  const float s = log10f(1.0f + (float)fabs(v) * 1e12f);
  return v < 0.0 ? -s : s;
}

// ln of a previous free ion, held finite for a zero or broken entry
__device__ __forceinline__ double ln_prev(double m) { return log(fmin(fmax(m, 1e-300), 1e300)); }

// raw feature f of cell c (slots documented in pfx_surrogate.h)
__device__ __forceinline__ float feature_raw(int f, int64_t c, int N, int K, const double *total,
                                             const double *prev, const double *temp, const double *vf) {
  if (f < N) return slog(total[c * N + f]);
  if (f < 2 * N) return (float)ln_prev(prev[c * N + (f - N)]);
  if (f == 2 * N) return temp ? (float)temp[c] : 25.0f;
  if (f < 2 * N + 1 + K) return vf ? (float)vf[c * K + (f - 2 * N - 1)] : 0.0f;
  return 0.0f;
}

enum { EPI_STORE = 0, EPI_BIAS_GELU = 1, EPI_BIAS = 2, EPI_ATOMIC = 3 };

constexpr int BM = 64, BN = 64, BK = 32, LDSK = BK + 8;

// C[m][n] (op)= sum_k A(m,k) B(n,k) with A(m,k) = A[m*sam + k*sak] and
// B(n,k) = B[n*sbn + k*sbk] (FP32 in memory, rounded to BF16 when staged
// in LDS).  256 threads per 64x64 tile, wavefront w owns the 32x32 quarter
// (w/2, w%2) as 2x2 MFMA tiles.  blockIdx.z splits K (EPI_ATOMIC only).
template <int EPI>
__global__ __launch_bounds__(256) void k_gemm_bf16(int M, int N, int K, const float *__restrict__ A, long sam,
                                                   long sak, const float *__restrict__ B, long sbn, long sbk,
                                                   float *__restrict__ C, long ldc, const float *__restrict__ bias,
                                                   float *__restrict__ Zout, int ksplit) {
  __shared__ __attribute__((aligned(16))) unsigned short As[BM][LDSK];
  __shared__ __attribute__((aligned(16))) unsigned short Bs[BN][LDSK];
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int kchunk = roundup((K + ksplit - 1) / ksplit, BK);
  const int kbeg = blockIdx.z * kchunk;
  const int kend = min(K, kbeg + kchunk);
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int lr = t >> 2, lk = (t & 3) * 8;  // staging: row, first of 8 k
  for (int k0 = kbeg; k0 < kend; k0 += BK) {
    {
      const int m = m0 + lr, n = n0 + lr;
      unsigned short va[8], vb[8];
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const int k = k0 + lk + q;
        va[q] = f2bf((m < M && k < kend) ? A[(long)m * sam + (long)k * sak] : 0.0f);
        vb[q] = f2bf((n < N && k < kend) ? B[(long)n * sbn + (long)k * sbk] : 0.0f);
      }
      uint4 ua, ub;
      ua.x = va[0] | ((unsigned)va[1] << 16);
      ua.y = va[2] | ((unsigned)va[3] << 16);
      ua.z = va[4] | ((unsigned)va[5] << 16);
      ua.w = va[6] | ((unsigned)va[7] << 16);
      ub.x = vb[0] | ((unsigned)vb[1] << 16);
      ub.y = vb[2] | ((unsigned)vb[3] << 16);
      ub.z = vb[4] | ((unsigned)vb[5] << 16);
      ub.w = vb[6] | ((unsigned)vb[7] << 16);
      *(uint4 *)&As[lr][lk] = ua;
      *(uint4 *)&Bs[lr][lk] = ub;
    }
    __syncthreads();
    const int fr = lane & 15, fk = (lane >> 4) * 8;
    bf16x8 af[2], bfr[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      af[i] = as_frag(*(const uint4 *)&As[wm + 16 * i + fr][fk]);
      bfr[i] = as_frag(*(const uint4 *)&Bs[wn + 16 * i + fr][fk]);
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + q;
        const int n = n0 + wn + 16 * j + (lane & 15);
        if (m < M && n < N) {
          float v = acc[i][j][q];
          if (EPI == EPI_ATOMIC) {
            atomicAdd(&C[(long)m * ldc + n], v);
          } else if (EPI == EPI_STORE) {
            C[(long)m * ldc + n] = v;
          } else {
            v += bias[n];
            if (EPI == EPI_BIAS_GELU) {
              Zout[(long)m * ldc + n] = v;
              v = gelu(v);
            }
            C[(long)m * ldc + n] = v;
          }
        }
      }
}

__global__ void k_fill(float *p, long n, float v) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_gelu_back(const float *dA, const float *Z, float *dZ, long n) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i < n) dZ[i] = dA[i] * gelu_grad(Z[i]);
}

// dY = 2 (Y - T) / n and the loss sum((Y - T)^2) / n
__global__ void k_mse_grad(const float *Y, const float *T, float *dY, float *loss, long n, float inv) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  float l = 0.f;
  if (i < n) {
    const float d = Y[i] - T[i];
    dY[i] = 2.0f * d * inv;
    l = d * d * inv;
  }
  for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o);
  if ((threadIdx.x & 63) == 0) atomicAdd(loss, l);
}

// db[o] += sum over a slice of rows of dZ[b][o]: blockIdx.x covers 64
// columns, blockIdx.y a slice of rows (db zeroed beforehand)
constexpr int COLSUM_ROWS = 128;
__global__ __launch_bounds__(256) void k_colsum(const float *dZ, int B, int N, float *db) {
  __shared__ float red[4][64];
  const int o = blockIdx.x * 64 + (threadIdx.x & 63);
  const int w = threadIdx.x >> 6;
  const int b0 = blockIdx.y * COLSUM_ROWS, b1 = min(B, b0 + COLSUM_ROWS);
  float s = 0.f;
  if (o < N)
    for (int b = b0 + w; b < b1; b += 4) s += dZ[(long)b * N + o];
  red[w][threadIdx.x & 63] = s;
  __syncthreads();
  if (w == 0 && o < N)
    atomicAdd(&db[o], red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x]);
}

// Several tensors in one launch (training is launch-bound at these sizes):
// blockIdx.y picks the tensor, blockIdx.x strides over its elements.
constexpr int MT_MAX = 2 * MLP_MAX_LAYERS + 1;
struct mt_tensors {
  float *p[MT_MAX];
  long n[MT_MAX];
  int count;
};
struct mt_adam {
  float *w[MT_MAX], *g[MT_MAX], *m[MT_MAX], *v[MT_MAX];
  unsigned short *sw[MT_MAX], *swt[MT_MAX];  // BF16 fragments of a weight and of its transpose (or null)
  int K[MT_MAX];                             // row length of a weight
  long n[MT_MAX], off[MT_MAX];               // elements, first element in a gradient slice
  int count;
};

__global__ void k_fill_multi(const mt_tensors T, float v) {
  const int t = blockIdx.y;
  if (t >= T.count) return;
  float *p = T.p[t];
  const long n = T.n[t];
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

// element (r, c) of a matrix in MFMA fragment order (k_swizzle), kts
// fragments of 32 columns to a row tile
__device__ __forceinline__ long frag_at(int r, int c, int kts) {
  return (((long)(r >> 4) * kts + (c >> 5)) * 64 + (r & 15) + 2 * (c & 24)) * 8 + (c & 7);
}

// Gradients from their nsplit slices (0: they are there already), then Adam
// with bias correction over every weight and bias tensor (adam), which also
// rewrites the BF16 fragments that the products read.  blockIdx.y == count
// adds the rows' losses in a fixed order.  Bound by the slices' reads (9 MB at
// 145k parameters in 16 slices).  A fill, the atomics, Adam and the fragments'
// rewrite were four passes over the parameters.
__global__ __launch_bounds__(256) void k_update(const mt_adam T, int nsplit, const float *part, long stride,
                                                const float *lpart, int nlpart, float *loss, int adam, float lr,
                                                float b1, float b2, float c1, float c2, float eps) {
  const int t = blockIdx.y;
  if (t >= T.count) {
    if (blockIdx.x > 0) return;
    __shared__ float red[4];
    float l = 0.f;
    for (int i = threadIdx.x; i < nlpart; i += 256) l += lpart[i];
    for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) *loss = (red[0] + red[1]) + (red[2] + red[3]);
    return;
  }
  float *w = T.w[t], *g = T.g[t], *m = T.m[t], *v = T.v[t];
  const long n = T.n[t];
  const int K = T.K[t], N = (int)(n / K);
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    float gi;
    if (nsplit > 0) {
      const float *q = part + T.off[t] + i;
      gi = 0.f;
#pragma unroll 8
      for (int k = 0; k < nsplit; k++) gi += q[k * stride];
      g[i] = gi;
    } else {
      gi = g[i];
    }
    if (!adam) continue;
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    if (T.sw[t]) {
      const int r = (int)i / K, c = (int)i - r * K;
      const unsigned short h = f2bf(wi);
      T.sw[t][frag_at(r, c, (K + 31) / 32)] = h;
      if (T.swt[t]) T.swt[t][frag_at(c, r, (N + 31) / 32)] = h;
    }
  }
}

// grid x for a multi-tensor launch: the largest tensor in 256-element
// blocks, at most 1024 blocks (the rest by striding)
inline unsigned mt_blocks(const long *n, int count) {
  long mx = 1;
  for (int t = 0; t < count; t++) mx = n[t] > mx ? n[t] : mx;
  return (unsigned)std::min<long>(1024, (mx + 255) / 256);
}

// W(n, k) = W[n*sn + k*sk] FP32 -> BF16 fragments: uint4 index
// ((nt * Kp/32 + kt) * 64 + lane) holds W(nt*16 + lane%16,
// kt*32 + 8*(lane/16) + 0..7) (zero outside)
__global__ void k_swizzle(const float *W, int N, int K, long sn, long sk, int Np, int Kp, uint4 *out) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int kts = Kp / 32;
  const long total = (long)(Np / 16) * kts * 64;
  if (i >= total) return;
  const int lane = (int)(i & 63);
  const long f = i >> 6;
  const int kt = (int)(f % kts), nt = (int)(f / kts);
  const int n = nt * 16 + (lane & 15);
  const int k0 = kt * 32 + 8 * (lane >> 4);
  unsigned short v[8];
#pragma unroll
  for (int q = 0; q < 8; q++) v[q] = f2bf((n < N && k0 + q < K) ? W[n * sn + (k0 + q) * sk] : 0.0f);
  uint4 u;
  u.x = v[0] | ((unsigned)v[1] << 16);
  u.y = v[2] | ((unsigned)v[3] << 16);
  u.z = v[4] | ((unsigned)v[5] << 16);
  u.w = v[6] | ((unsigned)v[7] << 16);
  out[i] = u;
}

__global__ void k_features(int64_t ncells, int N, int K, const double *total, const double *prev,
                           const double *temp, const double *vf, int nfeat, const float *shift, const float *scale,
                           float *X) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= ncells * nfeat) return;
  const int64_t c = i / nfeat;
  const int f = (int)(i % nfeat);
  X[i] = (feature_raw(f, c, N, K, total, prev, temp, vf) - shift[f]) * scale[f];
}

// guess = previous free ion times exp(predicted change of ln m over the
// step); the change is held within +-30 (a factor of 1e13)
__device__ __forceinline__ double guess_of(float y, int j, const float *shift, const float *scale, double prev) {
  const double dlnm = (double)y / (double)scale[j] + (double)shift[j];
  return exp(fmin(fmax(ln_prev(prev) + fmin(fmax(dlnm, -30.0), 30.0), -700.0), 700.0));
}

__global__ void k_guess(const float *Y, int nout, const float *shift, const float *scale, const double *prev,
                        double *guess, int64_t n, int N) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= n * N) return;
  const long c = i / N;
  const int j = (int)(i % N);
  guess[i] = guess_of(Y[c * nout + j], j, shift, scale, prev[i]);
}

// ---------------------------------------------------------------------------
// fused inference
struct mlp_dev {
  int nlayers;
  int dims[MLP_MAX_LAYERS + 1];
  int kpad[MLP_MAX_LAYERS];  // input width of layer l rounded up to 32
  const uint4 *Wsw[MLP_MAX_LAYERS];
  const float *b[MLP_MAX_LAYERS];
  const float *in_shift, *in_scale, *out_shift, *out_scale;
};

// 1M cells of 40-256-256-256-15: 1.53 ms with erff, features cell by cell and
// two activation buffers (two workgroups on a CU); branch-free GELU 1.25,
// features a kind at a time 1.09, one buffer that a layer's outputs replace, and
// so three workgroups, 0.79 (366 TFLOP/s).  A register cap for a fourth spills
// and takes 0.80.
constexpr int SC = 64;      // cells per block
constexpr int ASTR = 264;   // LDS activation row stride (BF16 elements, 528 B)

__global__ __launch_bounds__(256, 3) void k_surrogate_guess(const mlp_dev D, int64_t ncells, int N, int K,
                                                         const double *__restrict__ total,
                                                         const double *__restrict__ prev,
                                                         const double *__restrict__ temp,
                                                         const double *__restrict__ vf, double *__restrict__ guess) {
  __shared__ __attribute__((aligned(16))) unsigned short act[SC * ASTR];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int64_t c0 = (int64_t)blockIdx.x * SC;
  // Features of the block's 64 cells, a kind at a time: consecutive threads
  // read consecutive words, all of a thread's loads are in flight together and no
  // wavefront runs both logarithms for every feature (four threads a cell, each
  // through its 16 features, took a round trip to memory a feature).
  {
    const int nf = D.dims[0];
    const unsigned inv = 65536u / N + 1;  // i / N for i < 4096
    const int64_t left = (ncells - c0) * N;
    const int count = (int)(left < SC * N ? left : SC * N);
    double v[4], u[4];                     // SC * 16 values over 256 threads
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int i = t + 256 * q;
      v[q] = i < count ? total[c0 * N + i] : 0.0;
      u[q] = i < count ? prev[c0 * N + i] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int i = t + 256 * q;
      if (i < SC * N) {
        const int cl = (int)((i * inv) >> 16), j = i - cl * N;
        const bool in = i < count;
        act[cl * ASTR + j] = f2bf(in ? (slog(v[q]) - D.in_shift[j]) * D.in_scale[j] : 0.0f);
        act[cl * ASTR + N + j] =
            f2bf(in ? ((float)ln_prev(u[q]) - D.in_shift[N + j]) * D.in_scale[N + j] : 0.0f);
      }
    }
    const int cl = t >> 2;
    const int64_t c = c0 + cl;
    for (int f = 2 * N + (t & 3); f < D.kpad[0]; f += 4) {
      float x = 0.0f;
      if (c < ncells && f < nf)
        x = (feature_raw(f, c, N, K, total, prev, temp, vf) - D.in_shift[f]) * D.in_scale[f];
      act[cl * ASTR + f] = f2bf(x);
    }
  }
  __syncthreads();
  const int col = lane & 15, kq = 8 * (lane >> 4), rq = 4 * (lane >> 4);
  for (int l = 0; l < D.nlayers - 1; l++) {
    const int kts = D.kpad[l] / 32;
    const int ntw = D.dims[l + 1] / 64;  // 16-row tiles per wavefront (1..4)
    const uint4 *Wl = D.Wsw[l];
    const unsigned short *in = act;
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // weight fragments of step kt + 1 are loaded while step kt's products
    // run: the fragments come from L2 and each block reuses them for only
    // 64 cells, so their latency, not the matrix cores, bounds the layer
    uint4 wa[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
      wa[i] = i < ntw ? Wl[((long)(w * ntw + i) * kts + 0) * 64 + lane] : make_uint4(0, 0, 0, 0);
    for (int kt = 0; kt < kts; kt++) {
      bf16x8 a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; i++) a[i] = as_frag(wa[i]);
      if (kt + 1 < kts) {
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (i < ntw) wa[i] = Wl[((long)(w * ntw + i) * kts + kt + 1) * 64 + lane];
      }
#pragma unroll
      for (int j = 0; j < 4; j++) b[j] = as_frag(*(const uint4 *)&in[(j * 16 + col) * ASTR + kt * 32 + kq]);
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (i < ntw)
#pragma unroll
          for (int j = 0; j < 4; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();  // every wavefront has read the layer's inputs: its outputs take their place
    unsigned short *out = act;
    const float *bl = D.b[l];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (i < ntw) {
        const int n0 = (w * ntw + i) * 16 + rq;
        const float4 bv = *(const float4 *)&bl[n0];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int cl = j * 16 + col;
          uint2 u;
          u.x = pack_bf(gelu_tail(acc[i][j][0] + bv.x), gelu_tail(acc[i][j][1] + bv.y));
          u.y = pack_bf(gelu_tail(acc[i][j][2] + bv.z), gelu_tail(acc[i][j][3] + bv.w));
          *(uint2 *)&out[cl * ASTR + n0] = u;
        }
      }
    }
    __syncthreads();
  }
  // output layer: one 16-row tile, wavefront w takes cells 16w..16w+15
  {
    const int l = D.nlayers - 1;
    const int kts = D.kpad[l] / 32;
    const uint4 *Wl = D.Wsw[l];
    const unsigned short *in = act;
    f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int64_t c = c0 + w * 16 + col;
    const int nout = D.dims[D.nlayers];
    double pm[4];
#pragma unroll
    for (int q = 0; q < 4; q++) pm[q] = c < ncells && rq + q < N ? prev[c * N + rq + q] : 1.0;
    for (int kt = 0; kt < kts; kt++) {
      const bf16x8 a = as_frag(Wl[(long)kt * 64 + lane]);
      const bf16x8 b = as_frag(*(const uint4 *)&in[(w * 16 + col) * ASTR + kt * 32 + kq]);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
    }
    if (c < ncells) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int j = rq + q;
        if (j < N && j < nout)
          guess[c * N + j] = guess_of(acc[q] + D.b[l][j], j, D.out_shift, D.out_scale, pm[q]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// training and plain inference of layers up to CHAIN_WIDTH wide
//
// With 16 rows to a workgroup, batches of some thousand rows fill the chip
// and one launch carries them through all layers: the weight fragments come
// from L2 (each workgroup reads all of them, 290 KB at 40-256-256-256-15), the
// activations stay in LDS as the BF16 operands they are rounded to anyway.
// One training step of 4096 rows at that shape took 23 launches and 231 us with
// the tiled products, whose scalar loads of transposed operands and passes
// between layers bound them; now 27 us (this kernel) + 19 (weight gradients) + 7
// (update).  What is left here is latency: 20 us remain with a single
// fragment a product, 25 without the GELUs.
// Widths (three equal hidden layers, 4096 rows, step / plain inference), tiled
// products -> this: 256: 231 -> 53 / 70 -> 12 us, 512: 399 -> 114 / 168 -> 24,
// 768: 720 -> 199 / 334 -> 39.  CHAIN_WIDTH is where the two buffers of 16 rows
// reach 64 KB of LDS.
constexpr int CHAIN_WIDTH = 960;
constexpr int CHAIN_ROWS = 16;
constexpr int CHAIN_THREADS = 512;  // inference: fewer for narrow networks (launch_chain)
constexpr int CHAIN_RESIDENT = 256 * 4 * CHAIN_ROWS;

struct mlp_chain {
  int nlayers, B, astr;  // astr: LDS row stride (BF16 elements)
  int dims[MLP_MAX_LAYERS + 1];
  const uint4 *Wsw[MLP_MAX_LAYERS], *Wtsw[MLP_MAX_LAYERS];
  const float *b[MLP_MAX_LAYERS];
  float *S[MLP_MAX_LAYERS], *A[MLP_MAX_LAYERS + 1], *dZ[MLP_MAX_LAYERS];  // gelu', activations
  const float *X, *T;
  float *Y, *lpart;
  float inv;
};

__host__ __device__ inline int ld4(int n) { return (n + 3) & ~3; }

// D = W x in^T for 16 rows: W in fragments (rt row tiles of kts fragments), in
// [16][astr] BF16 in LDS.  Each wavefront takes two row tiles at a time, the
// fragments of 8 steps of k in flight together (the loop waits on L2, not on the
// matrix cores).  Rows of D are walked up to the next multiple of 32, so that
// the next product's operand is padded with what epi writes there.
// pre(n0) loads four values ahead of the product, epi(n0, acc, those) takes
// rows n0..n0+3 of this lane's column (row lane % 16 of the batch tile).
template <int THREADS, class PRE, class EPI>
__device__ __forceinline__ void chain_product(const uint4 *__restrict__ W, int nrows, int kts,
                                              const unsigned short *in, int astr, PRE pre, EPI epi) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int rt = (nrows + 15) / 16, ft = (nrows + 31) / 32 * 2;
  const unsigned short *ap = in + (lane & 15) * astr + 8 * (lane >> 4);
  for (int nt = 2 * w; nt < ft; nt += 2 * (THREADS / 64)) {
    const uint4 *p0 = W + (long)min(nt, rt - 1) * kts * 64 + lane;
    const uint4 *p1 = W + (long)min(nt + 1, rt - 1) * kts * 64 + lane;
    const int n0 = nt * 16 + 4 * (lane >> 4);
    f32x4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = {0.f, 0.f, 0.f, 0.f};
    const f32x4 x0 = pre(n0), x1 = pre(n0 + 16);
    for (int k0 = 0; k0 < kts; k0 += 8) {
      uint4 f0[8], f1[8];
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const int kt = min(k0 + q, kts - 1);
        f0[q] = p0[kt * 64];
        f1[q] = p1[kt * 64];
      }
#pragma unroll
      for (int q = 0; q < 8; q++)
        if (k0 + q < kts) {
          const bf16x8 b = as_frag(*(const uint4 *)&ap[(k0 + q) * 32]);
          a0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(f0[q]), b, a0, 0, 0, 0);
          a1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(f1[q]), b, a1, 0, 0, 0);
        }
    }
    epi(n0, a0, x0);
    epi(n0 + 16, a1, x1);
  }
}

// Forward pass of 16 rows; TRAIN: also the loss and dZ of every layer,
// with the activations and gelu' kept for it and for the weight gradients.
template <bool TRAIN, int THREADS>
__global__ __launch_bounds__(THREADS) void k_chain(const mlp_chain D) {
  extern __shared__ __attribute__((aligned(16))) unsigned short chain_lds[];
  __shared__ float lred[THREADS / 64];
  const int t = threadIdx.x, lane = t & 63;
  const int r0 = blockIdx.x * CHAIN_ROWS;
  const long row = r0 + (lane & 15);
  const bool live = row < D.B;
  const int L = D.nlayers, astr = D.astr;
  unsigned short *in = chain_lds, *out = chain_lds + CHAIN_ROWS * astr;
  {
    const int K = D.dims[0], Kp = roundup(K, 32);
    for (int i = t; i < CHAIN_ROWS * Kp; i += THREADS) {
      const int r = i / Kp, k = i - r * Kp;
      in[r * astr + k] = f2bf((r0 + r < D.B && k < K) ? D.X[(long)(r0 + r) * K + k] : 0.0f);
    }
  }
  __syncthreads();
  auto put = [&](int n0, const f32x4 v) {
    uint2 u;
    u.x = f2bf(v[0]) | ((unsigned)f2bf(v[1]) << 16);
    u.y = f2bf(v[2]) | ((unsigned)f2bf(v[3]) << 16);
    *(uint2 *)&out[(lane & 15) * astr + n0] = u;
  };
  float loss = 0.f;
  for (int l = 0; l < L; l++) {
    const int K = D.dims[l], N = D.dims[l + 1], ld = ld4(N);
    const float *bl = D.b[l];
    const bool last = l == L - 1;
    auto bias = [&](int n0) {
      f32x4 v;
#pragma unroll
      for (int q = 0; q < 4; q++) v[q] = bl[min(n0 + q, N - 1)];
      return v;
    };
    if (!last) {
      float *Sl = D.S[l], *Al = D.A[l + 1];
      chain_product<THREADS>(D.Wsw[l], N, roundup(K, 32) / 32, in, astr, bias, [&](int n0, f32x4 acc, f32x4 bv) {
        f32x4 s, a;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const float z = n0 + q < N ? acc[q] + bv[q] : 0.0f;
          float slope = 0.f;
          a[q] = TRAIN ? gelu_both(z, slope) : gelu(z);
          s[q] = slope;
        }
        if (TRAIN && live && n0 < ld) {
          *(f32x4 *)&Sl[row * ld + n0] = s;
          *(f32x4 *)&Al[row * ld + n0] = a;
        }
        put(n0, a);
      });
    } else {
      chain_product<THREADS>(D.Wsw[l], N, roundup(K, 32) / 32, in, astr, bias, [&](int n0, f32x4 acc, f32x4 bv) {
        f32x4 dz = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (live && n0 + q < N) {
            const float y = acc[q] + bv[q];
            if (TRAIN) {
              const float d = y - D.T[row * N + n0 + q];
              dz[q] = 2.0f * d * D.inv;
              loss += d * d * D.inv;
            } else {
              D.Y[row * N + n0 + q] = y;
            }
          }
        if (TRAIN) {
          if (live && n0 < ld) *(f32x4 *)&D.dZ[l][row * ld + n0] = dz;
          put(n0, dz);
        }
      });
    }
    __syncthreads();
    unsigned short *x = in;
    in = out;
    out = x;
  }
  if (!TRAIN) return;
  for (int l = L - 1; l > 0; l--) {
    // dA = dZ W; dZ of layer l-1 = dA * gelu'(Z), the slopes as this thread wrote them
    const int K = D.dims[l], N = D.dims[l + 1], ld = ld4(K);
    const float *Sl = D.S[l - 1];
    float *dZl = D.dZ[l - 1];
    chain_product<THREADS>(
        D.Wtsw[l], K, roundup(N, 32) / 32, in, astr,
        [&](int n0) {
          return live && n0 < ld ? *(const f32x4 *)&Sl[row * ld + n0] : (f32x4){0.f, 0.f, 0.f, 0.f};
        },
        [&](int n0, f32x4 acc, f32x4 s) {
          f32x4 dz;
#pragma unroll
          for (int q = 0; q < 4; q++) dz[q] = live && n0 + q < K ? acc[q] * s[q] : 0.0f;
          if (live && n0 < ld) *(f32x4 *)&dZl[row * ld + n0] = dz;
          put(n0, dz);
        });
    __syncthreads();
    unsigned short *x = in;
    in = out;
    out = x;
  }
  for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o);
  if (lane == 0) lred[t >> 6] = loss;
  __syncthreads();
  if (t == 0) {
    float l = 0.f;
    for (int i = 0; i < THREADS / 64; i++) l += lred[i];
    D.lpart[blockIdx.x] = l;
  }
}

// dW[n][k] = sum_b dZ[b][n] A[b][k] and db[n] = sum_b dZ[b][n] of every layer
// in one launch: blockIdx.y is a 64x64 tile of some layer's dW, blockIdx.x a
// slice of the batch (so that the tiles that read the same rows share an
// XCD's L2 cache), whose sums go to a slice of their own.  Atomics into one
// copy took longer than the products (a step of 12.9 us a layer, most of it
// 16 additions to each address).
// The operands' contiguous side is n (k) and their product's is b, so a thread
// turns an 8 x 4 block in registers on its way to LDS; the loads of the next 128
// rows are in flight while the matrix cores work.
// Bound by the operands' reads (every row once for each of the other operand's
// tiles, 84 MB of which L2 keeps most): 32.5 us at 4096 rows of 40-256-256-256-15
// with the tile fastest over the grid, 30 with the slice fastest, 19 with
// four workgroups on a CU (128 registers) instead of two, whose 640 did not fit
// the chip at once.  Layer by layer with atomics: 99 us.
constexpr int GT = 64;            // tile of dW
constexpr int GB = 128;           // rows of the batch to a stage
constexpr int GSTR = GB + 8;      // LDS row stride (BF16 elements)

struct grad_layer {
  const float *dZ, *A;
  int N, K, ldz, lda, tk, tile0;
  long off;  // of dW in a slice, db behind it
  int avec;  // rows of A are 16-byte aligned
};
struct grad_args {
  grad_layer l[MLP_MAX_LAYERS];
  int nlayers, B, chunk;
  long params;
  float *part;
};

__device__ __forceinline__ void grad_load(f32x4 (&v)[8], const float *p, int ld, int n0, int n, bool vec, int b0,
                                          int b1) {
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const int b = b0 + q;
    v[q] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (b >= b1) continue;
    const float *r = p + (long)b * ld;
    if (vec) {
      if (n0 < ld) v[q] = *(const f32x4 *)&r[n0];
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (n0 + j < n) v[q][j] = r[n0 + j];
    }
  }
}

__device__ __forceinline__ void grad_stage(const f32x4 (&v)[8], unsigned short *s, int mg, int kg) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    uint4 u;
    u.x = f2bf(v[0][j]) | ((unsigned)f2bf(v[1][j]) << 16);
    u.y = f2bf(v[2][j]) | ((unsigned)f2bf(v[3][j]) << 16);
    u.z = f2bf(v[4][j]) | ((unsigned)f2bf(v[5][j]) << 16);
    u.w = f2bf(v[6][j]) | ((unsigned)f2bf(v[7][j]) << 16);
    *(uint4 *)&s[(4 * mg + j) * GSTR + 8 * kg] = u;
  }
}

__global__ __launch_bounds__(256, 4) void k_weight_grad(const grad_args G) {
  __shared__ __attribute__((aligned(16))) unsigned short Zs[GT * GSTR], As[GT * GSTR];
  __shared__ float red[16][GT];
  int li = 0;
  for (int l = 1; l < G.nlayers; l++)
    if ((int)blockIdx.y >= G.l[l].tile0) li = l;
  const grad_layer &P = G.l[li];
  const int tile = blockIdx.y - P.tile0;
  const int n0 = tile / P.tk * GT, k0 = tile % P.tk * GT;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int mg = t & 15, kg = t >> 4;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int beg = blockIdx.x * G.chunk, end = min(G.B, beg + G.chunk);
  const bool avec = P.avec != 0, want_db = k0 == 0;
  f32x4 acc[2][2], db = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  f32x4 vz[8], va[8];
  grad_load(vz, P.dZ, P.ldz, n0 + 4 * mg, P.N, true, beg + 8 * kg, end);
  grad_load(va, P.A, P.lda, k0 + 4 * mg, P.K, avec, beg + 8 * kg, end);
  for (int b = beg; b < end; b += GB) {
    if (b > beg) __syncthreads();
    grad_stage(vz, Zs, mg, kg);
    grad_stage(va, As, mg, kg);
    if (want_db) {
#pragma unroll
      for (int q = 0; q < 8; q++) db += vz[q];
    }
    __syncthreads();
    if (b + GB < end) {
      grad_load(vz, P.dZ, P.ldz, n0 + 4 * mg, P.N, true, b + GB + 8 * kg, end);
      grad_load(va, P.A, P.lda, k0 + 4 * mg, P.K, avec, b + GB + 8 * kg, end);
    }
    const int fr = lane & 15, fk = (lane >> 4) * 8;
#pragma unroll
    for (int kk = 0; kk < GB; kk += 32) {
      bf16x8 af[2], bfr[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        af[i] = as_frag(*(const uint4 *)&Zs[(wm + 16 * i + fr) * GSTR + kk + fk]);
        bfr[i] = as_frag(*(const uint4 *)&As[(wn + 16 * i + fr) * GSTR + kk + fk]);
      }
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
    }
  }
  float *out = G.part + blockIdx.x * G.params + P.off;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int n = n0 + wm + 16 * i + 4 * (lane >> 4) + q;
        const int k = k0 + wn + 16 * j + (lane & 15);
        if (n < P.N && k < P.K) out[(long)n * P.K + k] = acc[i][j][q];
      }
  if (want_db) {
    *(f32x4 *)&red[kg][4 * mg] = db;
    __syncthreads();
    if (t < GT && n0 + t < P.N) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 16; i++) s += red[i][t];
      out[(long)P.N * P.K + n0 + t] = s;
    }
  }
}

// ---------------------------------------------------------------------------
int launch_gemm(int epi, int M, int N, int K, const float *A, long sam, long sak, const float *B, long sbn,
                long sbk, float *C, long ldc, const float *bias, float *Zout, int ksplit, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  dim3 grid((M + BM - 1) / BM, (N + BN - 1) / BN, ksplit);
  switch (epi) {
    case EPI_STORE:
      hipLaunchKernelGGL(k_gemm_bf16<EPI_STORE>, grid, dim3(256), 0, s, M, N, K, A, sam, sak, B, sbn, sbk, C, ldc,
                         bias, Zout, ksplit);
      break;
    case EPI_BIAS_GELU:
      hipLaunchKernelGGL(k_gemm_bf16<EPI_BIAS_GELU>, grid, dim3(256), 0, s, M, N, K, A, sam, sak, B, sbn, sbk, C,
                         ldc, bias, Zout, ksplit);
      break;
    case EPI_BIAS:
      hipLaunchKernelGGL(k_gemm_bf16<EPI_BIAS>, grid, dim3(256), 0, s, M, N, K, A, sam, sak, B, sbn, sbk, C, ldc,
                         bias, Zout, ksplit);
      break;
    default:
      hipLaunchKernelGGL(k_gemm_bf16<EPI_ATOMIC>, grid, dim3(256), 0, s, M, N, K, A, sam, sak, B, sbn, sbk, C,
                         ldc, bias, Zout, ksplit);
  }
  MCHK(hipGetLastError());
  return 0;
}

int fill(float *p, long n, float v, hipStream_t s) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
  MCHK(hipGetLastError());
  return 0;
}

int max_width(const pfx_mlp *m) {
  int d = 0;
  for (int l = 0; l <= m->nlayers; l++) d = d > m->dims[l] ? d : m->dims[l];
  return d;
}

// forward pass of B <= bmax rows; the pre-activations go to Z (training) or
// to the dZ scratch (inference), the output to Y
int forward(pfx_mlp *m, const float *X, int B, float *Y, bool keep, hipStream_t s) {
  const float *in = X;
  for (int l = 0; l < m->nlayers; l++) {
    const int K = m->dims[l], N = m->dims[l + 1];
    const bool last = l == m->nlayers - 1;
    float *out = last ? Y : m->A[l + 1];
    float *z = keep ? m->Z[l] : m->dZ;
    int rc = launch_gemm(last ? EPI_BIAS : EPI_BIAS_GELU, B, N, K, in, K, 1, m->W[l], K, 1, out, N, m->b[l], z, 1,
                         s);
    if (rc) return rc;
    in = out;
  }
  return 0;
}

// The fragments of layer l from W[l].  They follow W wherever it changes: here
// once the caller has set it, in k_update with the step that moves it.  So every
// pass may read them as it reads W, on any stream and in a captured graph (a
// refresh ahead of the next pass would be enqueued on that pass's stream only,
// and not at all while one is captured or replayed).
int write_fragments(pfx_mlp *m, int l, hipStream_t s) {
  const int N = m->dims[l + 1], K = m->dims[l];
  const int Np = roundup(N, 16), Kp = roundup(K, 32);
  const long total = (long)(Np / 16) * (Kp / 32) * 64;
  hipLaunchKernelGGL(k_swizzle, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, m->W[l], N, K, (long)K, 1L,
                     Np, Kp, m->Wsw[l]);
  if (m->Wtsw[l]) {
    const int Nq = roundup(N, 32), Kq = roundup(K, 16);
    const long tt = (long)(Kq / 16) * (Nq / 32) * 64;
    hipLaunchKernelGGL(k_swizzle, dim3((unsigned)((tt + 255) / 256)), dim3(256), 0, s, m->W[l], K, N, 1L, (long)K,
                       Kq, Nq, m->Wtsw[l]);
  }
  MCHK(hipGetLastError());
  return 0;
}

bool chain_ok(const pfx_mlp *m) { return max_width(m) <= CHAIN_WIDTH; }

// batch rows B through all layers: Y (T null) or gradients' operands
int launch_chain(pfx_mlp *m, const float *X, const float *T, float *Y, int B, hipStream_t s) {
  mlp_chain D;
  memset(&D, 0, sizeof(D));
  D.nlayers = m->nlayers;
  D.B = B;
  D.astr = roundup(max_width(m), 32) + 8;
  for (int l = 0; l <= m->nlayers; l++) D.dims[l] = m->dims[l];
  for (int l = 0; l < m->nlayers; l++) {
    D.Wsw[l] = m->Wsw[l], D.Wtsw[l] = m->Wtsw[l], D.b[l] = m->b[l];
    D.S[l] = m->Z[l], D.A[l + 1] = m->A[l + 1], D.dZ[l] = m->dZl[l];
  }
  D.X = X, D.T = T, D.Y = Y, D.lpart = m->lpart;
  D.inv = 1.0f / (float)((long)B * m->dims[m->nlayers]);
  const unsigned grid = (unsigned)((B + CHAIN_ROWS - 1) / CHAIN_ROWS);
  const size_t lds = (size_t)2 * CHAIN_ROWS * D.astr * sizeof(unsigned short);
  // A wavefront takes 32 columns of a layer.  A batch too large to be resident at
  // once (CHAIN_RESIDENT rows, in workgroups of 8 wavefronts) gets no more
  // wavefronts in inference than the widest layer keeps busy: idle ones hold places
  // that other rows could have (262144 rows: 16-32-16 123 -> 52 us, 40-64-64-15 217
  // -> 113, 40-128-128-15 250 -> 180).  Below, 8 read the rows sooner (4096 rows of
  // 40-64-64-15 23.3 us, with two wavefronts 24.2).  Any split gives the same bits.
  // Training stays at 8: its weight gradients hide the difference.
  const int wide = T || B <= CHAIN_RESIDENT ? CHAIN_WIDTH : max_width(m);
  if (T) hipLaunchKernelGGL((k_chain<true, CHAIN_THREADS>), dim3(grid), dim3(CHAIN_THREADS), lds, s, D);
  else if (wide > 128) hipLaunchKernelGGL((k_chain<false, 512>), dim3(grid), dim3(512), lds, s, D);
  else if (wide > 64) hipLaunchKernelGGL((k_chain<false, 256>), dim3(grid), dim3(256), lds, s, D);
  else if (wide > 32) hipLaunchKernelGGL((k_chain<false, 128>), dim3(grid), dim3(128), lds, s, D);
  else hipLaunchKernelGGL((k_chain<false, 64>), dim3(grid), dim3(64), lds, s, D);
  MCHK(hipGetLastError());
  return 0;
}

long param_count(const pfx_mlp *m) {
  long n = 0;
  for (int l = 0; l < m->nlayers; l++) n += (long)m->dims[l + 1] * (m->dims[l] + 1);
  return n;
}

// Slices of the batch in the weight gradients: about 1024 workgroups (4 on a
// CU, as many as LDS and registers admit), of at least one stage of rows each
// and at most 16, beyond which the slices' traffic outweighs.
int grad_split(const pfx_mlp *m, int B) {
  int tiles = 0;
  for (int l = 0; l < m->nlayers; l++) tiles += ((m->dims[l + 1] + GT - 1) / GT) * ((m->dims[l] + GT - 1) / GT);
  return std::max(1, std::min({1024 / tiles, 16, (B + GB - 1) / GB}));
}

int launch_weight_grad(pfx_mlp *m, const float *X, int B, int nsplit, hipStream_t s) {
  grad_args G;
  memset(&G, 0, sizeof(G));
  G.nlayers = m->nlayers;
  G.B = B;
  G.chunk = roundup((B + nsplit - 1) / nsplit, 32);
  G.params = param_count(m);
  G.part = m->part;
  int tiles = 0;
  long off = 0;
  for (int l = 0; l < m->nlayers; l++) {
    grad_layer &P = G.l[l];
    P.N = m->dims[l + 1], P.K = m->dims[l];
    P.dZ = m->dZl[l], P.ldz = ld4(P.N);
    P.A = l ? m->A[l] : X, P.lda = l ? ld4(P.K) : P.K;
    P.avec = l > 0 || (P.K % 4 == 0 && (uintptr_t)X % 16 == 0);
    P.tk = (P.K + GT - 1) / GT;
    P.tile0 = tiles, P.off = off;
    tiles += P.tk * ((P.N + GT - 1) / GT);
    off += (long)P.N * (P.K + 1);
  }
  hipLaunchKernelGGL(k_weight_grad, dim3((unsigned)nsplit, (unsigned)tiles), dim3(256), 0, s, G);
  MCHK(hipGetLastError());
  return 0;
}

struct adam_rates {
  float lr, b1, b2, eps;
};

// gradients from nsplit slices (0: in place), loss from nlpart parts, and
// the Adam update if rates are given
int launch_update(pfx_mlp *m, int nsplit, int nlpart, const adam_rates *r, hipStream_t s) {
  mt_adam T{};
  long off = 0;
  for (int l = 0; l < m->nlayers; l++) {
    const int N = m->dims[l + 1], K = m->dims[l];
    T.w[T.count] = m->W[l], T.g[T.count] = m->gW[l], T.m[T.count] = m->mW[l], T.v[T.count] = m->vW[l];
    T.sw[T.count] = (unsigned short *)m->Wsw[l], T.swt[T.count] = (unsigned short *)m->Wtsw[l];
    T.K[T.count] = K, T.off[T.count] = off;
    T.n[T.count++] = (long)N * K;
    T.w[T.count] = m->b[l], T.g[T.count] = m->gb[l], T.m[T.count] = m->mb[l], T.v[T.count] = m->vb[l];
    T.K[T.count] = 1, T.off[T.count] = off + (long)N * K;
    T.n[T.count++] = N;
    off += (long)N * (K + 1);
  }
  float c1 = 1.f, c2 = 1.f;
  if (r) {
    m->adam_step++;
    c1 = 1.0f - powf(r->b1, (float)m->adam_step), c2 = 1.0f - powf(r->b2, (float)m->adam_step);
  }
  hipLaunchKernelGGL(k_update, dim3(mt_blocks(T.n, T.count), (unsigned)(T.count + (nlpart > 0))), dim3(256), 0, s, T,
                     nsplit, m->part, off, m->lpart, nlpart, m->loss, r ? 1 : 0, r ? r->lr : 0.f, r ? r->b1 : 0.f,
                     r ? r->b2 : 0.f, c1, c2, r ? r->eps : 0.f);
  MCHK(hipGetLastError());
  return 0;
}

// gradients by tiled products, layer by layer (layers wider than CHAIN_WIDTH)
int wide_gradients(pfx_mlp *m, const float *X, const float *T, int B, hipStream_t s) {
  const int L = m->nlayers;
  m->A[0] = (float *)X;
  int rc = forward(m, X, B, m->A[L], true, s);
  if (rc) return rc;
  const int no = m->dims[L];
  // every gradient buffer and the loss cleared in one launch (the weight
  // gradients and the loss accumulate with atomics)
  mt_tensors Zt{};
  for (int l = 0; l < L; l++) {
    Zt.p[Zt.count] = m->gW[l];
    Zt.n[Zt.count++] = (long)m->dims[l + 1] * m->dims[l];
    Zt.p[Zt.count] = m->gb[l];
    Zt.n[Zt.count++] = m->dims[l + 1];
  }
  Zt.p[Zt.count] = m->loss;
  Zt.n[Zt.count++] = 1;
  hipLaunchKernelGGL(k_fill_multi, dim3(mt_blocks(Zt.n, Zt.count), (unsigned)Zt.count), dim3(256), 0, s, Zt, 0.f);
  MCHK(hipGetLastError());
  const long nout = (long)B * no;
  hipLaunchKernelGGL(k_mse_grad, dim3((unsigned)((nout + 255) / 256)), dim3(256), 0, s, m->A[L], T, m->dZ, m->loss,
                     nout, 1.0f / (float)nout);
  MCHK(hipGetLastError());
  for (int l = L - 1; l >= 0; l--) {
    const int K = m->dims[l], N = m->dims[l + 1];
    // dW[n][k] = sum_b dZ[b][n] A[b][k], split over the batch
    const int ksplit = B >= 4096 ? 16 : (B >= 512 ? 4 : 1);
    if ((rc = launch_gemm(EPI_ATOMIC, N, K, B, m->dZ, 1, N, m->A[l], 1, K, m->gW[l], K, nullptr, nullptr, ksplit,
                          s)))
      return rc;
    hipLaunchKernelGGL(k_colsum, dim3((unsigned)((N + 63) / 64), (unsigned)((B + COLSUM_ROWS - 1) / COLSUM_ROWS)),
                       dim3(256), 0, s, m->dZ, B, N, m->gb[l]);
    MCHK(hipGetLastError());
    if (l > 0) {
      // dA[b][k] = sum_n dZ[b][n] W[n][k]; dZ of layer l-1 = dA * gelu'(Z)
      if ((rc = launch_gemm(EPI_STORE, B, K, N, m->dZ, N, 1, m->W[l], 1, K, m->dA, K, nullptr, nullptr, 1, s)))
        return rc;
      const long n = (long)B * K;
      hipLaunchKernelGGL(k_gelu_back, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, m->dA, m->Z[l - 1], m->dZ,
                         n);
      MCHK(hipGetLastError());
    }
  }
  return 0;
}

bool fused_shape_ok(const pfx_mlp *m, int N) {
  if (m->nlayers < 2 || m->dims[0] > 256) return false;
  for (int l = 1; l < m->nlayers; l++)
    if (m->dims[l] % 64 != 0 || m->dims[l] > 256) return false;
  const int nout = m->dims[m->nlayers];
  return nout >= 1 && nout <= 16 && N <= nout;
}

}  // namespace

// ---------------------------------------------------------------------------
extern "C" int pfx_mlp_create(int32_t nlayers, const int32_t *dims, int32_t batch_max, uint64_t seed,
                              pfx_mlp **out) {
  if (!out) return PFX_E_ARG;
  *out = nullptr;
  if (!dims || nlayers < 1 || nlayers > MLP_MAX_LAYERS || batch_max < 1) return PFX_E_ARG;
  for (int l = 0; l <= nlayers; l++)
    if (dims[l] < 1 || dims[l] > 4096) return PFX_E_ARG;
  pfx_mlp *m = new pfx_mlp();
  memset(m, 0, sizeof(*m));
  m->nlayers = nlayers;
  for (int l = 0; l <= nlayers; l++) m->dims[l] = dims[l];
  m->bmax = batch_max;
  // uniform(-a, a) initial weights, a = sqrt(3 / fan_in), from a seeded
  // splitmix64 stream on the host; zero biases
  uint64_t st = seed;
  auto next = [&]() {
    st += 0x9E3779B97F4A7C15ull;
    uint64_t z = st;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  };
  int rc = 0;
  const bool chain = chain_ok(m);
  for (int l = 0; l < nlayers && !rc; l++) {
    const long nw = (long)dims[l + 1] * dims[l];
    const int nb = dims[l + 1];
    std::vector<float> w(nw), bz(nb, 0.0f);
    const double a = std::sqrt(3.0 / dims[l]);
    for (long i = 0; i < nw; i++) w[i] = (float)(((double)(next() >> 11) * 0x1.0p-53 * 2.0 - 1.0) * a);
    const long nsw = (long)(roundup(dims[l + 1], 16) / 16) * (roundup(dims[l], 32) / 32) * 64;
    const long nswt = (long)(roundup(dims[l], 16) / 16) * (roundup(dims[l + 1], 32) / 32) * 64;
    if (hipMalloc(&m->W[l], nw * 4) != hipSuccess || hipMalloc(&m->b[l], nb * 4) != hipSuccess ||
        hipMalloc(&m->gW[l], nw * 4) != hipSuccess || hipMalloc(&m->gb[l], nb * 4) != hipSuccess ||
        hipMalloc(&m->mW[l], nw * 4) != hipSuccess || hipMalloc(&m->vW[l], nw * 4) != hipSuccess ||
        hipMalloc(&m->mb[l], nb * 4) != hipSuccess || hipMalloc(&m->vb[l], nb * 4) != hipSuccess ||
        hipMalloc(&m->Wsw[l], nsw * sizeof(uint4)) != hipSuccess ||
        hipMalloc(&m->Z[l], (long)batch_max * ld4(nb) * 4) != hipSuccess ||
        hipMalloc(&m->A[l + 1], (long)batch_max * ld4(nb) * 4) != hipSuccess ||
        (chain && (hipMalloc(&m->dZl[l], (long)batch_max * ld4(nb) * 4) != hipSuccess ||
                   hipMalloc(&m->Wtsw[l], nswt * sizeof(uint4)) != hipSuccess))) {
      rc = PFX_E_NOMEM;
      break;
    }
    if (hipMemcpy(m->W[l], w.data(), nw * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(m->b[l], bz.data(), nb * 4, hipMemcpyHostToDevice) != hipSuccess)
      rc = PFX_E_DEVICE;
    if (!rc) rc = fill(m->mW[l], nw, 0.f, 0);
    if (!rc) rc = fill(m->vW[l], nw, 0.f, 0);
    if (!rc) rc = fill(m->mb[l], nb, 0.f, 0);
    if (!rc) rc = fill(m->vb[l], nb, 0.f, 0);
    if (!rc) rc = fill(m->gW[l], nw, 0.f, 0);
    if (!rc) rc = fill(m->gb[l], nb, 0.f, 0);
    if (!rc) rc = write_fragments(m, l, 0);
  }
  const int md = max_width(m);
  if (!rc && chain &&
      (hipMalloc(&m->part, grad_split(m, batch_max) * param_count(m) * 4) != hipSuccess ||
       hipMalloc(&m->lpart, ((long)batch_max + CHAIN_ROWS - 1) / CHAIN_ROWS * 4) != hipSuccess))
    rc = PFX_E_NOMEM;
  if (!rc && !chain &&
      (hipMalloc(&m->dA, (long)batch_max * md * 4) != hipSuccess ||
       hipMalloc(&m->dZ, (long)batch_max * md * 4) != hipSuccess))
    rc = PFX_E_NOMEM;
  if (!rc && (hipMalloc(&m->loss, 4) != hipSuccess ||
              hipMalloc(&m->in_shift, dims[0] * 4) != hipSuccess ||
              hipMalloc(&m->in_scale, dims[0] * 4) != hipSuccess ||
              hipMalloc(&m->out_shift, dims[nlayers] * 4) != hipSuccess ||
              hipMalloc(&m->out_scale, dims[nlayers] * 4) != hipSuccess))
    rc = PFX_E_NOMEM;
  if (!rc) rc = fill(m->in_shift, dims[0], 0.f, 0);
  if (!rc) rc = fill(m->in_scale, dims[0], 1.f, 0);
  if (!rc) rc = fill(m->out_shift, dims[nlayers], 0.f, 0);
  if (!rc) rc = fill(m->out_scale, dims[nlayers], 1.f, 0);
  if (!rc && hipDeviceSynchronize() != hipSuccess) rc = PFX_E_DEVICE;
  if (rc) {
    pfx_mlp_destroy(m);
    return rc;
  }
  *out = m;
  return 0;
}

extern "C" int pfx_mlp_destroy(pfx_mlp *m) {
  if (!m) return PFX_E_ARG;
  for (int l = 0; l < m->nlayers; l++) {
    (void)hipFree(m->W[l]);
    (void)hipFree(m->b[l]);
    (void)hipFree(m->gW[l]);
    (void)hipFree(m->gb[l]);
    (void)hipFree(m->mW[l]);
    (void)hipFree(m->vW[l]);
    (void)hipFree(m->mb[l]);
    (void)hipFree(m->vb[l]);
    (void)hipFree(m->Wsw[l]);
    (void)hipFree(m->Wtsw[l]);
    (void)hipFree(m->dZl[l]);
    (void)hipFree(m->Z[l]);
    (void)hipFree(m->A[l + 1]);
  }
  (void)hipFree(m->part);
  (void)hipFree(m->lpart);
  (void)hipFree(m->dA);
  (void)hipFree(m->dZ);
  (void)hipFree(m->loss);
  (void)hipFree(m->in_shift);
  (void)hipFree(m->in_scale);
  (void)hipFree(m->out_shift);
  (void)hipFree(m->out_scale);
  delete m;
  return 0;
}

extern "C" int pfx_mlp_params(pfx_mlp *m, int32_t which, int32_t layer, float *host, int32_t to_device) {
  if (!m || !host) return PFX_E_ARG;
  if (which == 4) {
    const int ni = m->dims[0], no = m->dims[m->nlayers];
    float *dst[4] = {m->in_shift, m->in_scale, m->out_shift, m->out_scale};
    const int len[4] = {ni, ni, no, no};
    long off = 0;
    for (int q = 0; q < 4; q++) {
      if (to_device) MCHK(hipMemcpy(dst[q], host + off, len[q] * 4, hipMemcpyHostToDevice));
      else MCHK(hipMemcpy(host + off, dst[q], len[q] * 4, hipMemcpyDeviceToHost));
      off += len[q];
    }
    return 0;
  }
  if (layer < 0 || layer >= m->nlayers || which < 0 || which > 3) return PFX_E_ARG;
  float *p = which == 0 ? m->W[layer] : which == 1 ? m->b[layer] : which == 2 ? m->gW[layer] : m->gb[layer];
  const long n = (which == 0 || which == 2) ? (long)m->dims[layer + 1] * m->dims[layer] : m->dims[layer + 1];
  if (to_device) {
    MCHK(hipMemcpy(p, host, n * 4, hipMemcpyHostToDevice));
    if (which == 0) {
      int rc = write_fragments(m, layer, 0);
      if (rc) return rc;
      MCHK(hipStreamSynchronize(0));  // in place when the call returns, as W is
    }
  } else {
    MCHK(hipMemcpy(host, p, n * 4, hipMemcpyDeviceToHost));
  }
  return 0;
}

extern "C" int pfx_mlp_forward(pfx_mlp *m, const float *X, int64_t B, float *Y, void *stream) {
  if (!m || B < 0 || (B > 0 && (!X || !Y))) return PFX_E_ARG;
  hipStream_t s = (hipStream_t)stream;
  for (int64_t b0 = 0; b0 < B; b0 += m->bmax) {
    const int nb = (int)((B - b0) < m->bmax ? (B - b0) : m->bmax);
    const float *x = X + b0 * m->dims[0];
    float *y = Y + b0 * m->dims[m->nlayers];
    // One narrow layer over many rows is a plain product, whose tiles are 64 rows:
    // 262144 rows of 4-1 26 us (by rows of 16 70), of 256-16 169 (228).  The line
    // moves out with the inputs: 20000 rows of 16-16 20.6 us (22.2), of 256-16 37.6
    // (28.5), 65536 of 256-16 57.7 (60.5).
    const bool plain =
        m->nlayers == 1 && m->dims[1] <= 32 && nb > (long)CHAIN_RESIDENT * std::max(1, m->dims[0] / 64);
    int rc = chain_ok(m) && !plain ? launch_chain(m, x, nullptr, y, nb, s) : forward(m, x, nb, y, false, s);
    if (rc) return rc;
  }
  return 0;
}

// gradients of a batch, and the Adam update if rates are given
static int gradients(pfx_mlp *m, const float *X, const float *T, int32_t B, float *loss_out, const adam_rates *r,
                     hipStream_t s) {
  if (!m || !X || !T || B < 1 || B > m->bmax) return PFX_E_ARG;
  int rc;
  if (chain_ok(m)) {
    const int nsplit = grad_split(m, B);
    if ((rc = launch_chain(m, X, T, nullptr, B, s))) return rc;
    if ((rc = launch_weight_grad(m, X, B, nsplit, s))) return rc;
    if ((rc = launch_update(m, nsplit, (B + CHAIN_ROWS - 1) / CHAIN_ROWS, r, s))) return rc;
  } else {
    if ((rc = wide_gradients(m, X, T, B, s))) return rc;
    if (r && (rc = launch_update(m, 0, 0, r, s))) return rc;
  }
  if (loss_out) {
    MCHK(hipMemcpyAsync(loss_out, m->loss, 4, hipMemcpyDeviceToHost, s));
    MCHK(hipStreamSynchronize(s));
  }
  return 0;
}

extern "C" int pfx_mlp_gradients(pfx_mlp *m, const float *X, const float *T, int32_t B, float *loss_out,
                                 void *stream) {
  return gradients(m, X, T, B, loss_out, nullptr, (hipStream_t)stream);
}

extern "C" int pfx_mlp_adam(pfx_mlp *m, float lr, float beta1, float beta2, float eps, void *stream) {
  if (!m) return PFX_E_ARG;
  const adam_rates r = {lr, beta1, beta2, eps};
  return launch_update(m, 0, 0, &r, (hipStream_t)stream);
}

extern "C" int pfx_mlp_train_step(pfx_mlp *m, const float *X, const float *T, int32_t B, float lr, float *loss_out,
                                  void *stream) {
  const adam_rates r = {lr, 0.9f, 0.999f, 1e-8f};
  return gradients(m, X, T, B, loss_out, &r, (hipStream_t)stream);
}

extern "C" int pfx_surrogate_features(pfx_tables *tables, pfx_mlp *m, const pfx_cells *cells, float *X,
                                      void *stream) {
  if (!tables || !m || !cells || cells->ncells < 0) return PFX_E_ARG;
  int N, M, K, R;
  pfx_internal::table_sizes(tables, &N, &M, &K, &R);
  if (2 * N + 1 + K > m->dims[0]) return PFX_E_ARG;
  if (cells->ncells == 0) return 0;
  if (!X || !cells->total || !cells->pri_molal) return PFX_E_ARG;
  const long n = cells->ncells * (long)m->dims[0];
  hipLaunchKernelGGL(k_features, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     cells->ncells, N, K, cells->total, cells->pri_molal, cells->temperature,
                     cells->mnrl_volfrac, m->dims[0], m->in_shift, m->in_scale, X);
  MCHK(hipGetLastError());
  return 0;
}

extern "C" int pfx_surrogate_guess(pfx_tables *tables, pfx_mlp *m, pfx_cells *cells, void *stream) {
  if (!tables || !m || !cells || cells->ncells < 0) return PFX_E_ARG;
  int N, M, K, R;
  pfx_internal::table_sizes(tables, &N, &M, &K, &R);
  if (2 * N + 1 + K > m->dims[0]) return PFX_E_ARG;
  if (!fused_shape_ok(m, N)) return PFX_E_UNSUP;
  if (cells->ncells == 0) return 0;
  if (!cells->guess || !cells->total || !cells->pri_molal) return PFX_E_ARG;
  hipStream_t s = (hipStream_t)stream;
  mlp_dev D;
  memset(&D, 0, sizeof(D));
  D.nlayers = m->nlayers;
  for (int l = 0; l <= m->nlayers; l++) D.dims[l] = m->dims[l];
  for (int l = 0; l < m->nlayers; l++) {
    D.kpad[l] = roundup(m->dims[l], 32);
    D.Wsw[l] = m->Wsw[l];
    D.b[l] = m->b[l];
  }
  D.in_shift = m->in_shift;
  D.in_scale = m->in_scale;
  D.out_shift = m->out_shift;
  D.out_scale = m->out_scale;
  const unsigned blocks = (unsigned)((cells->ncells + SC - 1) / SC);
  hipLaunchKernelGGL(k_surrogate_guess, dim3(blocks), dim3(256), 0, s, D, cells->ncells, N, K, cells->total,
                     cells->pri_molal, cells->temperature, cells->mnrl_volfrac, (double *)cells->guess);
  MCHK(hipGetLastError());
  return 0;
}

extern "C" int pfx_surrogate_guess_from(pfx_mlp *m, const float *Y, int64_t ncells, int32_t naqcomp,
                                        const double *prev, double *guess, void *stream) {
  if (!m || ncells < 0 || naqcomp < 1 || naqcomp > m->dims[m->nlayers]) return PFX_E_ARG;
  if (ncells == 0) return 0;
  if (!Y || !prev || !guess) return PFX_E_ARG;
  const long n = ncells * naqcomp;
  hipLaunchKernelGGL(k_guess, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, Y,
                     m->dims[m->nlayers], m->out_shift, m->out_scale, prev, guess, ncells, naqcomp);
  MCHK(hipGetLastError());
  return 0;
}
