// mlp.hip -- BF16 MFMA perceptron for the chemistry surrogate: training (a pass
// over the rows, a pass over the weights, Adam) and fused all-layer inference.
//
// MFMA: v_mfma_f32_32x32x16_bf16 (gfx950).  Lane l of a wave holds
//   A fragment: A[row = l%32][k = 8*(l/32) + v], v = 0..7
//   B fragment: B[k = 8*(l/32) + v][col = l%32]
//   accumulator r = 0..15: C[row = 8*(r/4) + 4*(l/32) + r%4][col = l%32]
// Everything is padded so that GEMM dimensions are multiples of 32 (M, N)
// and 16 (K): the input to 32 features, the output to 32 columns; padded
// weights and biases are zero and stay zero under training (zero gradients).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <initializer_list>
#include <new>
#include <vector>

#include "../../include/nrg_mlp.h"
#include "mlp_internal.h"
#include "nrg_common.h"

namespace nrg {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int WAVE = 64;

__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c)
{
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// GELU, tanh form (Hendrycks & Gimpel 2016):
//   g(z) = z/2 (1 + tanh(u)),  u = sqrt(2/pi) (z + 0.044715 z^3)
// evaluated as z * sigma(2u) (1/2 (1 + tanh(u)) = 1 / (1 + e^(-2u))): one
// exp2 and one reciprocal, with -2 sqrt(2/pi) log2(e) folded into the cubic.
__device__ __forceinline__ float sigma2u(float z)
{
  const float a0 = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
  const float a1 = a0 * 0.044715f;
  const float e = __builtin_amdgcn_exp2f(z * __builtin_fmaf(z * z, a1, a0));
  return __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float gelu(float z) { return z * sigma2u(z); }
__device__ __forceinline__ float gelu_grad(float z)
{
  const float c = 0.7978845608028654f, a = 0.044715f;
  const float sg = sigma2u(z);
  const float dudz = c * (1.0f + 3.0f * a * z * z);
  return sg + 2.0f * z * sg * (1.0f - sg) * dudz;
}

// ---- training: one pass over the rows, one over the weights ----------------------
// A step was ~20 launches of a GEMM that loaded its operands by single strided
// bf16 values (689 us for 4096 rows of 256 x 4).  Two kernels do the work now:
//   train_rows_kernel  forward, loss and the chain of dZ for a block's rows, whose
//                      activations stay in LDS (one wave per 32 columns);
//   train_weights_kernel  all dW = H^T dZ and db, split over the rows.
// Between them H and dZ are kept as the second one's MFMA fragments: a lane's
// accumulator holds 16 rows of its column, and since the order of the rows inside
// a reduction over them is free, elements 0..7 and 8..15 are its 8 k-values of two
// k-blocks as they stand (rows 16 kb + 8 (v/4) + 4 hi + v%4), so that every operand
// of the reduction is one coalesced 16-byte load and nothing is transposed.
// What bounds the first is a block's way through the layers (9 products of 16
// dependent MFMAs, each with its GELUs and a barrier), the second the latency of
// its loads and the atomics that add up the ranges.  4096 rows of 256 x 4: 27 + 13
// us (before: 20 launches, 420 us).
struct TrainArgs {
  const float *x, *t, *w;      // n x n_in, n x n_out, n_out weights or NULL
  long long n;
  int n_in, n_out, layers;     // layers: hidden layers
  const bf16 *Wf[MLP_MAX_LAYERS];    // forward fragments of the weights (Wsw)
  const bf16 *Wb[MLP_MAX_LAYERS];    // backward fragments (frag_kernel)
  const float *bias[MLP_MAX_LAYERS];
  bf16 *Xf, *dYf;              // fragments of the input and of dL/dy
  bf16 *Hf[MLP_MAX_LAYERS], *dZf[MLP_MAX_LAYERS];   // of each hidden layer
  float *gz[MLP_MAX_LAYERS];   // gelu'(z), each lane's 16 values together
  float *y;                    // n x n_out, or NULL
  float *loss_part;            // a value per tile
  float *grad;                 // gradients, cleared here for train_weights_kernel
  long long n_grad;
};

// Barrier for what went through LDS.  (__syncthreads also waits for every global
// load and store under way, here the next product's weights and the fragments.)
__device__ __forceinline__ void lds_barrier()
{
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// row of its 32-row tile that element r of a lane's accumulator holds
__device__ __forceinline__ int acc_row(int r, int hi) { return 8 * (r / 4) + 4 * hi + r % 4; }

// A lane's first EL elements of an accumulator as bf16: its share of the fragments
// of EL / 8 k-blocks.
template <int EL>
__device__ __forceinline__ void store_frags(bf16 *f, const bf16 (&v)[EL], int l)
{
#pragma unroll
  for (int k = 0; k < EL / 8; ++k) {
    bf16x8 x;
#pragma unroll
    for (int r = 0; r < 8; ++r) x[r] = v[8 * k + r];
    reinterpret_cast<bf16x8 *>(f)[k * WAVE + l] = x;
  }
}

// Hidden width 32 NT (one wave per 32 columns), 2 EL rows per block (EL: the
// accumulator elements in use; with 8 the MFMAs see the 16 rows twice, but the
// epilogues, which cost more, are halved and twice the CUs work).
template <int NT, int EL>
__global__ void __launch_bounds__(NT * 64) train_rows_kernel(TrainArgs a)
{
  constexpr int HID = 32 * NT, KB = 2 * NT, LD = HID + 8, ROWS = 2 * EL, NTHR = NT * WAVE;
  constexpr int INLD = MLP_IN_PAD + 8;
  static_assert(EL == 8 || EL == 16, "one or two k-blocks of rows");
  __shared__ __align__(16) bf16 act[2][ROWS][LD];
  __shared__ __align__(16) bf16 io[ROWS][INLD];  // the input, later dL/dy
  const int w = threadIdx.x / WAVE, l = threadIdx.x & (WAVE - 1);
  const int r32 = l & 31, hi = l >> 5, col = 32 * w + r32;
  const int arow = r32 % ROWS;
  const long long row0 = (long long)blockIdx.x * ROWS;
  // the rows' fragments of columns 32 c.. of a matrix nt tiles wide
  auto frag = [&](bf16 *f, int nt, int c) {
    const long long kb = (long long)blockIdx.x * (ROWS / 16);   // first k-block
    return f + (((kb / 2) * nt + c) * 2 + kb % 2) * (WAVE * 8);
  };
  auto slope = [&](int layer) {                  // the lane's EL values of gelu'(z)
    return a.gz[layer] + (((long long)blockIdx.x * NT + w) * WAVE + l) * EL;
  };

  for (long long i = (long long)blockIdx.x * NTHR + threadIdx.x; i < a.n_grad; i += (long long)gridDim.x * NTHR)
    a.grad[i] = 0.0f;
  for (int i = threadIdx.x; i < ROWS * MLP_IN_PAD; i += NTHR) {
    const int row = i / MLP_IN_PAD, c = i % MLP_IN_PAD;
    io[row][c] = (bf16)(row0 + row < a.n && c < a.n_in ? a.x[(row0 + row) * a.n_in + c] : 0.0f);
  }
  bf16x8 b[KB];                                  // this wave's weights of a layer
  auto weights = [&](const bf16 *W, int kbs) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
      if (kb < kbs) b[kb] = reinterpret_cast<const bf16x8 *>(W)[(kb * NT + w) * WAVE + l];
  };
  f32x16 acc;
  auto product = [&](const bf16 *in, int ld, int kbs) {
    acc = f32x16{};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
      if (kb < kbs) acc = mfma(*reinterpret_cast<const bf16x8 *>(in + arow * ld + 16 * kb + 8 * hi), b[kb], acc);
  };
  weights(a.Wf[0], 2);
  lds_barrier();
  if (w == 0) {                                  // fragments of the input
    bf16 v[EL];
#pragma unroll
    for (int r = 0; r < EL; ++r) v[r] = io[acc_row(r, hi)][r32];
    store_frags<EL>(frag(a.Xf, 1, 0), v, l);
  }

  // forward through the hidden layers
  for (int layer = 0; layer < a.layers; ++layer) {
    if (layer == 0)
      product(&io[0][0], INLD, 2);
    else
      product(&act[(layer - 1) & 1][0][0], LD, KB);
    if (layer + 1 < a.layers) weights(a.Wf[layer + 1], KB);   // on their way during the epilogue
    const float bias = a.bias[layer][col];
    bf16 v[EL];
    float *gz = slope(layer);
#pragma unroll
    for (int r = 0; r < EL; ++r) {
      const float z = acc[r] + bias;
      gz[r] = gelu_grad(z);
      v[r] = (bf16)gelu(z);
      act[layer & 1][acc_row(r, hi)][col] = v[r];
    }
    store_frags<EL>(frag(a.Hf[layer], NT, w), v, l);
    lds_barrier();
  }

  // output, loss = sum_rows sum_c w_c (y - t)^2 / n and dY = 2 w_c (y - t) / n
  weights(a.Wb[a.layers], 2);
  if (w == 0) {
    const bf16 *in = &act[(a.layers - 1) & 1][arow][8 * hi];
    f32x16 o = {};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
      o = mfma(*reinterpret_cast<const bf16x8 *>(in + 16 * kb),
               reinterpret_cast<const bf16x8 *>(a.Wf[a.layers])[kb * WAVE + l], o);
    const float bias = a.bias[a.layers][r32], inv_n = 1.0f / (float)a.n;
    const float wc = a.w && r32 < a.n_out ? a.w[r32] : 1.0f;
    float s = 0.0f;
    bf16 v[EL];
#pragma unroll
    for (int r = 0; r < EL; ++r) {
      const long long row = row0 + acc_row(r, hi);
      float g = 0.0f;
      if (row < a.n && r32 < a.n_out) {
        const float y = o[r] + bias, d = y - a.t[row * a.n_out + r32];
        s += wc * d * d;
        g = 2.0f * wc * d * inv_n;
        if (a.y) a.y[row * a.n_out + r32] = y;
      }
      v[r] = (bf16)g;
      io[acc_row(r, hi)][r32] = v[r];
    }
    store_frags<EL>(frag(a.dYf, 1, 0), v, l);
    s *= inv_n;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (l == 0) a.loss_part[blockIdx.x] = s;
  }
  lds_barrier();

  // dZ of the hidden layers, last first: (dZ of the next W^T) * gelu'(z)
  for (int layer = a.layers - 1; layer >= 0; --layer) {
    float gz[EL];
#pragma unroll
    for (int r = 0; r < EL; ++r) gz[r] = slope(layer)[r];
    if (layer == a.layers - 1)
      product(&io[0][0], INLD, 2);
    else
      product(&act[layer & 1][0][0], LD, KB);
    if (layer > 0) weights(a.Wb[layer], KB);
    bf16 v[EL];
#pragma unroll
    for (int r = 0; r < EL; ++r) {
      v[r] = (bf16)(acc[r] * gz[r]);
      if (layer > 0) act[(layer - 1) & 1][acc_row(r, hi)][col] = v[r];
    }
    store_frags<EL>(frag(a.dZf[layer], NT, w), v, l);
    lds_barrier();
  }
}

// dW = H^T dZ and db = sum of dZ of every layer: a block takes 2 x 2 tiles of one
// layer's weights (a fragment then serves two products) and a range of the rows,
// which its four waves share; their sums meet in LDS and the ranges' in G.
struct WeightLayer {
  const bf16 *A, *B;           // fragments of H (the layer's input) and of dZ
  int MT, NT;                  // tiles of the weights
  int block0;                  // first block (x) of the layer
  int K, N;                    // extents kept of them, and the row pitch
  float *dW, *db;
};
struct WeightArgs {
  WeightLayer L[MLP_MAX_LAYERS];
  int layers;                  // weight matrices
  long long kblocks, kper;     // 16-row blocks, and those of one y-range
  const float *loss_part;
  long long n_part;
  float *loss;                 // or NULL
};

__global__ void __launch_bounds__(256) train_weights_kernel(WeightArgs a)
{
  __shared__ float red[4][4][16][WAVE];
  __shared__ float redb[4][2][32];
  const int w = threadIdx.x / WAVE, l = threadIdx.x & (WAVE - 1);
  const int r32 = l & 31, hi = l >> 5;
  int i = 0;
  while (i + 1 < a.layers && (int)blockIdx.x >= a.L[i + 1].block0) ++i;
  const WeightLayer &L = a.L[i];
  const int bn = (L.NT + 1) / 2, bid = (int)blockIdx.x - L.block0;
  const int mt = bid / bn * 2, nt = bid % bn * 2;
  const int m1 = mt + 1 < L.MT ? mt + 1 : mt, n1 = nt + 1 < L.NT ? nt + 1 : nt;   // a missing tile: twice the first
  const bf16x8 *A = reinterpret_cast<const bf16x8 *>(L.A) + l, *B = reinterpret_cast<const bf16x8 *>(L.B) + l;
  const long long k1 = min(a.kblocks, ((long long)blockIdx.y + 1) * a.kper);
  f32x16 c[2][2] = {};
  float s[2] = {0.0f, 0.0f};
  constexpr int AHEAD = 4;       // k-blocks loaded together
  for (long long k0 = (long long)blockIdx.y * a.kper + w; k0 < k1; k0 += 4 * AHEAD) {
    bf16x8 fa[AHEAD][2] = {}, fb[AHEAD][2] = {};
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) {
      const long long k = k0 + 4 * q;
      if (k < k1) {
        const long long ta = (k / 2) * L.MT, tb = (k / 2) * L.NT;
        const int h = (int)(k & 1);
        fa[q][0] = A[((ta + mt) * 2 + h) * WAVE];
        fa[q][1] = A[((ta + m1) * 2 + h) * WAVE];
        fb[q][0] = B[((tb + nt) * 2 + h) * WAVE];
        fb[q][1] = B[((tb + n1) * 2 + h) * WAVE];
      }
    }
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) {
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i / 2][i % 2] = mfma(fa[q][i / 2], fb[q][i % 2], c[i / 2][i % 2]);
      if (mt == 0) {
#pragma unroll
        for (int v = 0; v < 8; ++v) {
          s[0] += (float)fb[q][0][v];
          s[1] += (float)fb[q][1][v];
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[w][q][r][l] = c[q / 2][q % 2][r];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    s[j] += __shfl_xor(s[j], 32);
    if (hi == 0) redb[w][j][r32] = s[j];
  }
  __syncthreads();
  const int tm = mt + w / 2, tn = nt + w % 2;        // wave w adds up tile w
  if (tm < L.MT && tn < L.NT) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float v = ((red[0][w][r][l] + red[1][w][r][l]) + red[2][w][r][l]) + red[3][w][r][l];
      const int row = 32 * tm + acc_row(r, hi), col = 32 * tn + r32;
      if (row < L.K && col < L.N) atomicAdd(&L.dW[(long long)row * L.N + col], v);
    }
    if (mt == 0 && w < 2 && hi == 0 && 32 * tn + r32 < L.N)
      atomicAdd(&L.db[32 * tn + r32], ((redb[0][w][r32] + redb[1][w][r32]) + redb[2][w][r32]) + redb[3][w][r32]);
  }
  if (a.loss && blockIdx.x == 0 && blockIdx.y == 0 && w == 0) {
    float p = 0.0f;
    for (long long k = l; k < a.n_part; k += WAVE) p += a.loss_part[k];
    for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off);
    if (l == 0) *a.loss = p;
  }
}

// ---- small element-wise kernels ---------------------------------------------------

__global__ void fill_f32_kernel(float *p, long long n, float v)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void adam_kernel(float *P, bf16 *Pbf, const float *G, float *M1, float *M2, long long n,
                            float lr, float bc1, float bc2)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float g = G[i];
  const float m = b1 * M1[i] + (1.0f - b1) * g;
  const float v = b2 * M2[i] + (1.0f - b2) * g * g;
  M1[i] = m;
  M2[i] = v;
  const float w = P[i] - lr * (m / bc1) / (sqrtf(v / bc2) + eps);
  P[i] = w;
  Pbf[i] = (bf16)w;
}

__global__ void to_bf16_kernel(const float *P, bf16 *Pbf, long long n)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) Pbf[i] = (bf16)P[i];
}

// ---- fused inference -------------------------------------------------------------
// All layers in one kernel, computed transposed, Z^T = W^T H^T: the weights are the
// MFMA A operand (32 output features x 16 inputs) and the activations the B operand
// (16 inputs x 32 cells).  A wave owns 32 features of every hidden layer; its
// weights of a layer (up to 16 KB) come from L2 into registers and serve the two or
// four 32-cell tiles that a block works on, whose activations pass through LDS.  A
// lane's accumulator holds, for its cell, features 32 w + 8 q + 4 hi + i (q, i =
// 0..3, hi = lane/32): four stores of four.  Width 256 keeps a k-block's inputs in
// the order (8 hi + 4 (q%2) + i of block q/2) that its K rows have in WswT, and the
// bias as the accumulators' start; the others take the natural order and add it.
//
// What bounds it is the GELUs' VALU time (two of their seven operations are
// quarter-rate), which several waves per SIMD overlap with each other's MFMAs and
// loads.  The blocks share the tiles evenly.  Before, a wave took its cells through
// all features with the weights staged in LDS (at the narrower widths the
// activations): few cells left most of the chip idle for a long chain, and 70,001
// cells were a second, nearly empty round.
//
// At widths 128 and 256 nothing of a group of tiles waits for memory: the group's
// input is fetched while the one before goes through its layers and lies in its own
// LDS, the output layer's weights and bias come with the last GELUs, and the waves
// without an output tile go on with the next group, whose first layer writes the
// buffer that the output layer does not read (one barrier a layer).  Without that the
// ends of a group cost more than a layer: 256 x 1, 1,000,000 cells, 227 us with the
// loads where they are used, 169 with a wave per 32 cells, 140 so.
//
// Call times in turn (a wave per 32 cells -> loads where they are used -> this), width
// 256 x 4: 1000 cells 48 -> 22 -> 21 us, 16,384 49 -> 27 -> 26, 70,001 88 -> 62 -> 58,
// 262,144 180 -> 172 -> 157, 4,000,000 2401 -> 2388 -> 2095; 256 x 2, 1,000,000: 313 ->
// 340 -> 257; 128 x 1, 1,000,000: 144 -> 159 -> 93; 128 x 4, 262,144: 111 -> 89 -> 79;
// 64 x 4, 262,144: 71 -> 50 -> 49.
struct InferArgs {
  const bf16 *X;               // n x 32, or NULL:
  const float *x;              // n x n_in
  long long n;
  int n_in, n_out, layers;     // layers: hidden layers
  const bf16 *W[MLP_MAX_LAYERS];     // WswT (width 256) or Wsw
  const float *bias[MLP_MAX_LAYERS];
  float *Y;                    // n x n_out
};

// physical feature (output column of the previous layer) of logical K row kl
__host__ __device__ inline int t_phys(int kl)
{
  const int kb = kl / 16, hi = (kl / 8) % 2, v = kl % 8;
  const int r = 8 * (kb % 2) + v;
  return 32 * (kb / 2) + 8 * (r / 4) + 4 * hi + r % 4;
}

// MFMA fragments of every layer's weights W (K x N, row-major), 8 values a thread,
// so that a lane's fragment is one 16-byte load:
//   Wsw[((kb*N/32 + nt)*64 + lane)*8 + v] = W[16 kb + 8 (lane/32) + v][32 nt + lane%32]
//     (forward: kernels with the weights as B operand)
//   Wb[((kb*K/32 + nt)*64 + lane)*8 + v] = W[32 nt + lane%32][16 kb + 8 (lane/32) + v]
//     (backward: W^T as B operand)
//   WswT[((mt*K/16 + kb)*64 + lane)*8 + v] = W[k][32 mt + lane%32],
//     k = (layer > 0 ? t_phys : identity)(16 kb + 8 (lane/32) + v)
struct FragArgs {
  int K[MLP_MAX_LAYERS], N[MLP_MAX_LAYERS], layers;
  long long w_off[MLP_MAX_LAYERS], sw_off[MLP_MAX_LAYERS + 1];
  const bf16 *W;
  bf16 *Wsw, *Wb, *WswT;
};
__global__ void __launch_bounds__(256) frag_kernel(FragArgs a)
{
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= a.sw_off[a.layers]) return;
  int ly = 0;
  while (i >= a.sw_off[ly + 1]) ++ly;
  const int K = a.K[ly], N = a.N[ly];
  const bf16 *W = a.W + a.w_off[ly];
  const long long f = (i - a.sw_off[ly]) / 8;
  const int lane = (int)(f % WAVE), r32 = lane & 31, k8 = 8 * (lane >> 5);
  const int q = (int)(f / WAVE);
  bf16x8 fw, bw, tr;
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    fw[v] = W[(long long)(16 * (q / (N / 32)) + k8 + v) * N + 32 * (q % (N / 32)) + r32];
    bw[v] = W[(long long)(32 * (q % (K / 32)) + r32) * N + 16 * (q / (K / 32)) + k8 + v];
    const int kl = 16 * (q % (K / 16)) + k8 + v;
    tr[v] = W[(long long)(ly > 0 ? t_phys(kl) : kl) * N + 32 * (q / (K / 16)) + r32];
  }
  *reinterpret_cast<bf16x8 *>(a.Wsw + i) = fw;
  *reinterpret_cast<bf16x8 *>(a.Wb + i) = bw;
  *reinterpret_cast<bf16x8 *>(a.WswT + i) = tr;
}

// Resident waves per SIMD, and the 32-cell tiles a block takes through the layers
// together: two waves with up to 256 registers (a tile's fragments and a layer's
// weights in flight at once; before the inputs were fetched ahead 262,144 cells at
// width 256 took 186 us, 298 with four waves, which spill; at 128 99 and 104), but four
// at width 64 (50 us, 57 with two), where the blocks' LDS leaves no room for an input
// buffer of their own and the SIMD's other waves cover the loads.
constexpr int infer_waves(int nt) { return nt >= 4 ? 2 : 4; }
constexpr int infer_tiles(int nt) { return nt >= 4 ? 4 : 2; }
constexpr bool infer_ahead(int nt) { return nt >= 4; }

template <int NT>
__global__ void __launch_bounds__(NT * 64) __attribute__((amdgpu_waves_per_eu(infer_waves(NT), infer_waves(NT))))
mlp_infer_kernel(InferArgs a)
{
  constexpr bool PERM = NT == 8;
  constexpr int KB = 2 * NT, LD = 32 * NT + 8, TILES = infer_tiles(NT);
  constexpr bool AHEAD = infer_ahead(NT);
  constexpr int XBUF = !AHEAD ? 0 : NT == 8 ? 2 : 1, XLD = MLP_IN_PAD + 8, XV = 32 * TILES * MLP_IN_PAD / (NT * WAVE);
  static_assert(TILES <= NT, "a tile's output layer is one wave's work");
  __shared__ __align__(16) bf16 act[2][32 * TILES][LD];
  __shared__ __align__(16) bf16 xin[XBUF ? XBUF : 1][XBUF ? 32 * TILES : 1][XLD];
  const int w = threadIdx.x / WAVE, l = threadIdx.x & (WAVE - 1);
  const int r32 = l & 31, hi = l >> 5;
  const long long T = (a.n + 31) / 32;
  const long long t0 = T * blockIdx.x / gridDim.x, t1 = T * (blockIdx.x + 1) / gridDim.x;
  const int groups = (int)((t1 - t0 + TILES - 1) / TILES);
  // fragment kb of feature tile mt of a layer with nt feature tiles and kbs k-blocks
  auto weight = [&](int layer, int mt, int nt, int kb, int kbs) {
    return reinterpret_cast<const bf16x8 *>(a.W[layer])[(PERM ? mt * kbs + kb : kb * nt + mt) * WAVE + l];
  };
  bf16x8 W[KB];
  // this wave's weights of a layer (of the output layer: its one feature tile's)
  auto weights = [&](int layer) {
    const bool out = layer == a.layers;
    if (out && w >= TILES) return;
    const bf16x8 *p = reinterpret_cast<const bf16x8 *>(a.W[layer]) + (out ? 0 : PERM ? w * KB : w) * WAVE + l;
    const int step = out || PERM ? WAVE : NT * WAVE;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) W[kb] = p[kb * step];
  };
  auto biases = [&](int layer, int mt) {
    f32x16 b;
#pragma unroll
    for (int r = 0; r < 16; ++r) b[r] = a.bias[layer][32 * mt + acc_row(r, hi)];
    return b;
  };
  auto store = [&](int buf, int tile, const f32x16 &acc, const f32x16 &bias) {
    bf16 *d = &act[buf][32 * tile + r32][32 * w];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16)gelu(PERM ? acc[4 * q + i] : acc[4 * q + i] + bias[4 * q + i]);
      *reinterpret_cast<bf16x4 *>(d + (PERM ? 16 * (q / 2) + 8 * hi + 4 * (q % 2) : 8 * q + 4 * hi)) = v;
    }
  };
  // the input: packed in memory, or converted on its way through LDS: into its own
  // buffer while the group before is at work, or into the second one of activations
  auto tile_of = [&](int g) { return t0 + (t1 - t0) * g / groups; };
  const int xr = threadIdx.x / MLP_IN_PAD, xc = threadIdx.x % MLP_IN_PAD;
  float xv[XV];
  auto fetch = [&](int g) {
    const long long row0 = 32 * tile_of(g) + xr;
#pragma unroll
    for (int k = 0; k < XV; ++k) {
      const long long row = row0 + k * (NT * WAVE / MLP_IN_PAD), cell = row < a.n ? row : a.n - 1;
      xv[k] = xc < a.n_in ? a.x[cell * a.n_in + xc] : 0.0f;
    }
  };
  auto place = [&](int g) {
#pragma unroll
    for (int k = 0; k < XV; ++k) xin[g % (XBUF ? XBUF : 1)][xr + k * (NT * WAVE / MLP_IN_PAD)][xc] = (bf16)xv[k];
  };
  if (AHEAD && !a.X && groups > 0) {
    fetch(0);
    place(0);
    lds_barrier();
  }
  int first = 0;                                 // buffer of the first layer's output
  for (int g = 0; g < groups; ++g) {
    const long long tile = tile_of(g);
    const int nt = (int)(tile_of(g + 1) - tile);
    const bool more = AHEAD && !a.X && g + 1 < groups;
    if (more) fetch(g + 1);
    if (!AHEAD && !a.X) {
      for (int i = threadIdx.x; i < 32 * nt * MLP_IN_PAD; i += NT * WAVE) {
        const int row = i / MLP_IN_PAD, c = i % MLP_IN_PAD;
        const long long cell = 32 * tile + row < a.n ? 32 * tile + row : a.n - 1;
        act[1][row][c] = (bf16)(c < a.n_in ? a.x[cell * a.n_in + c] : 0.0f);
      }
    }
    f32x16 bias = biases(0, w);
    const bf16x8 W0[2] = {weight(0, w, NT, 0, 2), weight(0, w, NT, 1, 2)};
    if (!AHEAD && !a.X) lds_barrier();
    for (int t = 0; t < nt; ++t) {
      const long long cell = 32 * (tile + t) + r32 < a.n ? 32 * (tile + t) + r32 : a.n - 1;
      bf16x8 x[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        if (a.X)
          x[kb] = *reinterpret_cast<const bf16x8 *>(a.X + cell * MLP_IN_PAD + 16 * kb + 8 * hi);
        else if (AHEAD)
          x[kb] = *reinterpret_cast<const bf16x8 *>(&xin[g % (XBUF ? XBUF : 1)][32 * t + r32][16 * kb + 8 * hi]);
        else
          x[kb] = *reinterpret_cast<const bf16x8 *>(&act[1][32 * t + r32][16 * kb + 8 * hi]);
      f32x16 acc = PERM ? bias : f32x16{};
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) acc = mfma(W0[kb], x[kb], acc);
      if (t == nt - 1) weights(1);
      store(first, t, acc, bias);
    }
    for (int layer = 1; layer < a.layers; ++layer) {
      bias = biases(layer, w);
      lds_barrier();
      auto product = [&](int t) {
        const bf16 *in = &act[(first + layer - 1) & 1][32 * t + r32][8 * hi];
        f32x16 acc = PERM ? bias : f32x16{};
        if (NT >= 4) {                           // all loads ahead
          bf16x8 f[KB];
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) f[kb] = *reinterpret_cast<const bf16x8 *>(in + 16 * kb);
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) acc = mfma(W[kb], f[kb], acc);
        } else {
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) acc = mfma(W[kb], *reinterpret_cast<const bf16x8 *>(in + 16 * kb), acc);
        }
        return acc;
      };
      // a tile's product runs beside the GELUs of the one before, the next layer's
      // weights come during the last one's
      f32x16 cur = product(0);
#pragma unroll 1
      for (int t = 1; t < nt; ++t) {
        const f32x16 next = product(t);
        store((first + layer) & 1, t - 1, cur, bias);
        cur = next;
      }
      weights(layer + 1);
      store((first + layer) & 1, nt - 1, cur, bias);
    }
    bias = biases(a.layers, 0);
    if (more) {
      if (XBUF == 1 && a.layers == 1) lds_barrier();   // the first layer reads it to its end
      place(g + 1);
    }
    lds_barrier();
    if (w < nt) {                                // output layer: a tile to a wave
      const bf16 *in = &act[(first + a.layers - 1) & 1][32 * w + r32][8 * hi];
      f32x16 o = PERM ? bias : f32x16{};
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        o = mfma(W[kb], *reinterpret_cast<const bf16x8 *>(in + 16 * kb), o);
      const long long cell = 32 * (tile + w) + r32;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int f = acc_row(r, hi);
        if (cell < a.n && f < a.n_out) a.Y[cell * a.n_out + f] = PERM ? o[r] : o[r] + bias[r];
      }
    }
    // the next tiles' activations: in the buffer that nobody reads now, or in this one's place
    if (AHEAD) first = (first + a.layers) & 1;
    else lds_barrier();
  }
}

unsigned blocks_for(long long n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

// ---- handle ---------------------------------------------------------------------

struct MlpLayer {
  int K, N;                    // padded fan-in, fan-out
  int Kr, Nr;                  // real fan-in, fan-out
  long long w_off, b_off;      // offsets in the padded parameter arrays
  long long sw_off;            // offset in the swizzled bf16 array
};

}  // namespace nrg

struct nrg_mlp {
  int device = 0, num_cu = 0;
  hipStream_t stream = nullptr;
  int n_in = 0, hidden = 0, layers = 0, n_out = 0;
  std::vector<nrg::MlpLayer> L;            // layers + 1 entries
  long long n_pad = 0, n_packed = 0, n_sw = 0;
  float *P = nullptr, *G = nullptr, *M1 = nullptr, *M2 = nullptr;
  nrg::bf16 *Pbf = nullptr, *Wsw = nullptr, *Wb = nullptr, *WswT = nullptr;   // weights, and as fragments
  long long adam_t = 0;
  bool sw_dirty = true;                     // the fragments are older than the weights
  bool sw_synced = true;                    // written and waited for (other streams read them)
  // batch workspace
  long long train_cap = 0;
  nrg::bf16 *Xf = nullptr, *dYf = nullptr;  // training (TrainArgs)
  float *loss_part = nullptr;
  std::vector<nrg::bf16 *> Hf, dZf;         // per hidden layer
  std::vector<float *> gz;
};

namespace nrg {
namespace {

void free_all(std::initializer_list<void *> ps)
{
  for (void *p : ps)
    if (p) (void)hipFree(p);
}

void free_train(nrg_mlp_t *h)
{
  free_all({h->Xf, h->dYf, h->loss_part});
  for (auto p : h->Hf) free_all({p});
  for (auto p : h->dZf) free_all({p});
  for (auto p : h->gz) free_all({p});
  h->Xf = h->dYf = nullptr;
  h->loss_part = nullptr;
  h->Hf.assign(h->layers, nullptr);
  h->dZf.assign(h->layers, nullptr);
  h->gz.assign(h->layers, nullptr);
  h->train_cap = 0;
}

int ensure_train(nrg_mlp_t *h, long long n)
{
  if (n <= h->train_cap) return NRG_CHEM_OK;
  free_train(h);
  const long long m = ((n + 127) / 128) * 128;
  HIP_TRY(hipMalloc(&h->Xf, m * MLP_IN_PAD * sizeof(bf16)));
  HIP_TRY(hipMalloc(&h->dYf, m * MLP_OUT_PAD * sizeof(bf16)));
  HIP_TRY(hipMalloc(&h->loss_part, m / 16 * sizeof(float)));
  for (int i = 0; i < h->layers; ++i) {
    HIP_TRY(hipMalloc(&h->Hf[i], m * h->hidden * sizeof(bf16)));
    HIP_TRY(hipMalloc(&h->dZf[i], m * h->hidden * sizeof(bf16)));
    HIP_TRY(hipMalloc(&h->gz[i], m * h->hidden * sizeof(float)));
  }
  h->train_cap = m;
  return NRG_CHEM_OK;
}

// Bring the fragments up to date on the handle's stream; with `wait`, for other
// streams too (inference may run on the chemistry handle's).
int refresh_frags(nrg_mlp_t *h, bool wait)
{
  if (h->sw_dirty) {
    FragArgs f{};
    f.layers = (int)h->L.size();
    for (int i = 0; i < f.layers; ++i) {
      f.K[i] = h->L[i].K; f.N[i] = h->L[i].N;
      f.w_off[i] = h->L[i].w_off; f.sw_off[i] = h->L[i].sw_off;
    }
    f.sw_off[f.layers] = h->n_sw;
    f.W = h->Pbf; f.Wsw = h->Wsw; f.Wb = h->Wb; f.WswT = h->WswT;
    hipLaunchKernelGGL(frag_kernel, dim3(blocks_for(h->n_sw / 8, 256)), dim3(256), 0, h->stream, f);
    HIP_TRY(hipGetLastError());
    h->sw_dirty = false;
    h->sw_synced = false;
  }
  if (wait && !h->sw_synced) {
    HIP_TRY(hipStreamSynchronize(h->stream));
    h->sw_synced = true;
  }
  return NRG_CHEM_OK;
}

template <int NT>
void launch_rows(nrg_mlp_t *h, const TrainArgs &a, long long blocks, int rows)
{
  if (rows == 16)
    hipLaunchKernelGGL((train_rows_kernel<NT, 8>), dim3((unsigned)blocks), dim3(64 * NT), 0, h->stream, a);
  else
    hipLaunchKernelGGL((train_rows_kernel<NT, 16>), dim3((unsigned)blocks), dim3(64 * NT), 0, h->stream, a);
}

// Loss, predictions and the gradient: packed into `grad`, or padded into h->G.
int loss_and_grad(nrg_mlp_t *h, long long n, const float *x, const float *t, const float *w,
                  float *loss, float *y, float *grad)
{
  int rc = ensure_train(h, n);
  if (rc) return rc;
  if ((rc = refresh_frags(h, false))) return rc;
  // 16 rows to a block up to two blocks per CU, where a block's latency counts
  // (256 x 4: 4096 rows 50 us, 54 with 32; 128 x 4: 8192 rows 40, 44; 64 x 3: 4096 rows
  // 28, 31); above, the MFMAs' second half is worth having (256 x 4: 16384 rows 102, 109
  // with 16; 65536 340, 379; 128 x 4: 65536 157, 163; at 16384 the narrower widths are
  // 3 to 4 us faster with 16).
  const int rows = n <= 32ll * h->num_cu ? 16 : 32;
  const long long row_blocks = (n + rows - 1) / rows;
  TrainArgs a{};
  a.x = x; a.t = t; a.w = w; a.n = n;
  a.n_in = h->n_in; a.n_out = h->n_out; a.layers = h->layers;
  a.Xf = h->Xf; a.dYf = h->dYf; a.y = y; a.loss_part = h->loss_part;
  a.grad = grad ? grad : h->G;
  a.n_grad = grad ? h->n_packed : h->n_pad;
  WeightArgs g{};
  int blocks = 0;
  long long packed = 0;
  for (int i = 0; i <= h->layers; ++i) {
    const MlpLayer &ly = h->L[i];
    a.Wf[i] = h->Wsw + ly.sw_off;
    a.Wb[i] = h->Wb + ly.sw_off;
    a.bias[i] = h->P + ly.b_off;
    if (i < h->layers) {
      a.Hf[i] = h->Hf[i]; a.dZf[i] = h->dZf[i]; a.gz[i] = h->gz[i];
    }
    WeightLayer &q = g.L[i];
    q.A = i > 0 ? h->Hf[i - 1] : h->Xf;
    q.B = i < h->layers ? h->dZf[i] : h->dYf;
    q.MT = ly.K / 32; q.NT = ly.N / 32;
    q.block0 = blocks;
    blocks += ((q.MT + 1) / 2) * ((q.NT + 1) / 2);
    q.K = grad ? ly.Kr : ly.K; q.N = grad ? ly.Nr : ly.N;
    q.dW = a.grad + packed;
    q.db = q.dW + (long long)q.K * q.N;
    packed += (long long)q.K * q.N + q.N;
  }
  switch (h->hidden) {
    case 64: launch_rows<2>(h, a, row_blocks, rows); break;
    case 128: launch_rows<4>(h, a, row_blocks, rows); break;
    case 256: launch_rows<8>(h, a, row_blocks, rows); break;
    default: return set_error(NRG_CHEM_E_ARG, "hidden width %d has no training kernel", h->hidden);
  }
  g.layers = h->layers + 1;
  g.kblocks = row_blocks * (rows / 16);
  // Ranges of the rows: at least 512 rows each, and no more than fill the chip,
  // since every range adds its sums to G (256 x 4, 16384 rows: 103 us, 113 with all 32
  // ranges; 65536: 340, 371).
  const long long ksplit = std::max<long long>(1, std::min<long long>(n / 512, 2 * h->num_cu / blocks));
  g.kper = (g.kblocks + ksplit - 1) / ksplit;
  g.loss_part = h->loss_part; g.n_part = row_blocks; g.loss = loss;
  hipLaunchKernelGGL(train_weights_kernel, dim3((unsigned)blocks, (unsigned)((g.kblocks + g.kper - 1) / g.kper)),
                     dim3(256), 0, h->stream, g);
  HIP_TRY(hipGetLastError());
  return NRG_CHEM_OK;
}

}  // namespace

// X: n x 32 bf16, or NULL with x: n x n_in
static int launch_infer(nrg_mlp_t *h, long long n, const bf16 *X, const float *x, float *Y, hipStream_t stream)
{
  if (n <= 0) return NRG_CHEM_OK;
  int rc = refresh_frags(h, stream != h->stream);
  if (rc) return rc;
  InferArgs a{};
  a.X = X; a.x = x; a.n = n; a.n_in = h->n_in; a.n_out = h->n_out; a.layers = h->layers; a.Y = Y;
  for (int i = 0; i <= h->layers; ++i) {
    a.W[i] = (h->hidden == 256 ? h->WswT : h->Wsw) + h->L[i].sw_off;
    a.bias[i] = h->P + h->L[i].b_off;
  }
  const int nt = h->hidden / 32;
  const long long resident = (long long)h->num_cu * (4 * infer_waves(nt) / nt);
  const dim3 grid((unsigned)std::min<long long>((n + 31) / 32, resident)), block(2 * h->hidden);
  switch (h->hidden) {
    case 64: hipLaunchKernelGGL(mlp_infer_kernel<2>, grid, block, 0, stream, a); break;
    case 128: hipLaunchKernelGGL(mlp_infer_kernel<4>, grid, block, 0, stream, a); break;
    case 256: hipLaunchKernelGGL(mlp_infer_kernel<8>, grid, block, 0, stream, a); break;
    default: return set_error(NRG_CHEM_E_ARG, "hidden width %d has no inference kernel", h->hidden);
  }
  HIP_TRY(hipGetLastError());
  return NRG_CHEM_OK;
}

int mlp_infer_bf16(nrg_mlp_t *h, long long n, const bf16 *X, float *Y, hipStream_t stream)
{
  return launch_infer(h, n, X, nullptr, Y, stream);
}

namespace {

// The kernels write rows while other blocks still read theirs, so an input that an
// output overlaps is read from a copy (a caller may let the outputs take the
// inputs' place).
class Apart {
 public:
  explicit Apart(hipStream_t s) : stream(s) {}
  ~Apart() { free_all({copies[0], copies[1], copies[2]}); }   // (waits for the kernels that read them)
  void output(const float *p, long long n)
  {
    if (p) outs[n_outs++] = {p, p + n};
  }
  int input(const float *&p, long long n)
  {
    bool over = false;
    for (int i = 0; i < n_outs; ++i) over = over || (p < outs[i].end && outs[i].begin < p + n);
    if (!p || !over) return NRG_CHEM_OK;
    void *&c = copies[n_copies++];
    HIP_TRY(hipMalloc(&c, n * sizeof(float)));
    HIP_TRY(hipMemcpyAsync(c, p, n * sizeof(float), hipMemcpyDeviceToDevice, stream));
    p = (const float *)c;
    return NRG_CHEM_OK;
  }

 private:
  hipStream_t stream;
  struct Range {
    const float *begin, *end;
  } outs[3];
  void *copies[3] = {nullptr, nullptr, nullptr};
  int n_outs = 0, n_copies = 0;
};

}  // namespace

hipStream_t mlp_stream(nrg_mlp_t *h) { return h->stream; }
int mlp_n_out(const nrg_mlp_t *h) { return h->n_out; }
int mlp_n_in(const nrg_mlp_t *h) { return h->n_in; }

}  // namespace nrg

using namespace nrg;

extern "C" {

int nrg_mlp_create(int32_t n_in, int32_t n_hidden, int32_t n_layers, int32_t n_out, int32_t device,
                   nrg_mlp_t **out)
{
  if (!out) return set_error(NRG_CHEM_E_ARG, "out is NULL");
  *out = nullptr;
  if (n_in < 1 || n_in > MLP_IN_PAD || n_out < 1 || n_out > MLP_OUT_PAD || n_layers < 1 ||
      n_layers > MLP_MAX_LAYERS - 1 || !(n_hidden == 64 || n_hidden == 128 || n_hidden == 256))
    return set_error(NRG_CHEM_E_ARG, "unsupported network %d -> %d x %d -> %d", n_in, n_hidden,
                     n_layers, n_out);
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    return set_error(NRG_CHEM_E_NO_DEVICE, "no HIP device");
  if (device < 0 || device >= ndev) return set_error(NRG_CHEM_E_NO_DEVICE, "device %d out of range", device);
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return set_error(NRG_CHEM_E_NO_DEVICE, "device %d is %s, kernels are built for gfx950", device,
                     prop.gcnArchName);
  nrg_mlp_t *h = new (std::nothrow) nrg_mlp();
  if (!h) return set_error(NRG_CHEM_E_ARG, "out of host memory");
  h->device = device;
  h->num_cu = prop.multiProcessorCount;
  h->n_in = n_in; h->hidden = n_hidden; h->layers = n_layers; h->n_out = n_out;
  long long off = 0, sw = 0, packed = 0;
  for (int i = 0; i <= n_layers; ++i) {
    MlpLayer ly;
    ly.K = i == 0 ? MLP_IN_PAD : n_hidden;
    ly.N = i == n_layers ? MLP_OUT_PAD : n_hidden;
    ly.Kr = i == 0 ? n_in : n_hidden;
    ly.Nr = i == n_layers ? n_out : n_hidden;
    ly.w_off = off; off += (long long)ly.K * ly.N;
    ly.b_off = off; off += ly.N;
    ly.sw_off = sw; sw += (long long)ly.K * ly.N;
    packed += (long long)ly.Kr * ly.Nr + ly.Nr;
    h->L.push_back(ly);
  }
  h->n_pad = off; h->n_sw = sw; h->n_packed = packed;
  auto fail = [&](int rc) { nrg_mlp_destroy(h); return rc; };
  if (hipSetDevice(device) != hipSuccess) return fail(set_error(NRG_CHEM_E_HIP, "hipSetDevice"));
  if (hipStreamCreate(&h->stream) != hipSuccess) return fail(set_error(NRG_CHEM_E_HIP, "hipStreamCreate"));
  const size_t fb = h->n_pad * sizeof(float);
  if (hipMalloc(&h->P, fb) || hipMalloc(&h->G, fb) || hipMalloc(&h->M1, fb) || hipMalloc(&h->M2, fb) ||
      hipMalloc(&h->Pbf, h->n_pad * sizeof(bf16)) || hipMalloc(&h->Wsw, h->n_sw * sizeof(bf16)) ||
      hipMalloc(&h->Wb, h->n_sw * sizeof(bf16)) || hipMalloc(&h->WswT, h->n_sw * sizeof(bf16)))
    return fail(set_error(NRG_CHEM_E_HIP, "hipMalloc parameters"));
  std::vector<float> zero(h->n_packed, 0.0f);
  int rc = nrg_mlp_set_params(h, zero.data());
  if (rc) return fail(rc);
  *out = h;
  return NRG_CHEM_OK;
}

void nrg_mlp_destroy(nrg_mlp_t *h)
{
  if (!h) return;
  (void)hipSetDevice(h->device);
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  free_all({h->P, h->G, h->M1, h->M2, h->Pbf, h->Wsw, h->Wb, h->WswT});
  free_train(h);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
}

int64_t nrg_mlp_num_params(const nrg_mlp_t *h) { return h ? h->n_packed : 0; }

int nrg_mlp_set_params(nrg_mlp_t *h, const float *params)
{
  if (!h || !params) return set_error(NRG_CHEM_E_ARG, "NULL argument");
  HIP_TRY(hipSetDevice(h->device));
  std::vector<float> pad(h->n_pad, 0.0f);
  long long q = 0;
  for (const MlpLayer &ly : h->L) {
    for (int k = 0; k < ly.Kr; ++k)
      for (int n = 0; n < ly.Nr; ++n) pad[ly.w_off + (long long)k * ly.N + n] = params[q++];
    for (int n = 0; n < ly.Nr; ++n) pad[ly.b_off + n] = params[q++];
  }
  HIP_TRY(hipMemcpyAsync(h->P, pad.data(), h->n_pad * sizeof(float), hipMemcpyHostToDevice, h->stream));
  hipLaunchKernelGGL(fill_f32_kernel, dim3(blocks_for(h->n_pad, 256)), dim3(256), 0, h->stream,
                     h->M1, h->n_pad, 0.0f);
  hipLaunchKernelGGL(fill_f32_kernel, dim3(blocks_for(h->n_pad, 256)), dim3(256), 0, h->stream,
                     h->M2, h->n_pad, 0.0f);
  hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(h->n_pad, 256)), dim3(256), 0, h->stream,
                     h->P, h->Pbf, h->n_pad);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->adam_t = 0;
  h->sw_dirty = true;
  return NRG_CHEM_OK;
}

int nrg_mlp_get_params(nrg_mlp_t *h, float *params)
{
  if (!h || !params) return set_error(NRG_CHEM_E_ARG, "NULL argument");
  HIP_TRY(hipSetDevice(h->device));
  std::vector<float> pad(h->n_pad);
  HIP_TRY(hipMemcpyAsync(pad.data(), h->P, h->n_pad * sizeof(float), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  long long q = 0;
  for (const MlpLayer &ly : h->L) {
    for (int k = 0; k < ly.Kr; ++k)
      for (int n = 0; n < ly.Nr; ++n) params[q++] = pad[ly.w_off + (long long)k * ly.N + n];
    for (int n = 0; n < ly.Nr; ++n) params[q++] = pad[ly.b_off + n];
  }
  return NRG_CHEM_OK;
}

int nrg_mlp_forward_dev(nrg_mlp_t *h, int64_t n, const float *x, float *y)
{
  if (!h || (n > 0 && (!x || !y)) || n < 0) return set_error(NRG_CHEM_E_ARG, "bad argument");
  if (n == 0) return NRG_CHEM_OK;
  HIP_TRY(hipSetDevice(h->device));
  Apart apart(h->stream);
  apart.output(y, n * h->n_out);
  int rc = apart.input(x, n * h->n_in);
  if (!rc) rc = launch_infer(h, n, nullptr, x, y, h->stream);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(h->stream));
  return NRG_CHEM_OK;
}

int nrg_mlp_grad_dev(nrg_mlp_t *h, int64_t n, const float *x, const float *t, const float *w,
                     float *grad, float *loss, float *y_out)
{
  if (!h || n <= 0 || !x || !t || !grad) return set_error(NRG_CHEM_E_ARG, "bad argument");
  HIP_TRY(hipSetDevice(h->device));
  Apart apart(h->stream);
  apart.output(grad, h->n_packed);
  apart.output(loss, 1);
  apart.output(y_out, n * h->n_out);
  int rc = apart.input(x, n * h->n_in);
  if (!rc) rc = apart.input(t, n * h->n_out);
  if (!rc) rc = apart.input(w, h->n_out);
  if (!rc) rc = loss_and_grad(h, n, x, t, w, loss, y_out, grad);
  if (rc) return rc;
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(h->stream));
  return NRG_CHEM_OK;
}

int nrg_mlp_train_step_dev(nrg_mlp_t *h, int64_t n, const float *x, const float *t, const float *w,
                           float lr, float *loss)
{
  if (!h || n <= 0 || !x || !t) return set_error(NRG_CHEM_E_ARG, "bad argument");
  HIP_TRY(hipSetDevice(h->device));
  int rc = loss_and_grad(h, n, x, t, w, loss, nullptr, nullptr);
  if (rc) return rc;
  h->adam_t += 1;
  const float bc1 = 1.0f - std::pow(0.9f, (float)h->adam_t);
  const float bc2 = 1.0f - std::pow(0.999f, (float)h->adam_t);
  hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(h->n_pad, 256)), dim3(256), 0, h->stream, h->P,
                     h->Pbf, h->G, h->M1, h->M2, h->n_pad, lr, bc1, bc2);
  HIP_TRY(hipGetLastError());
  h->sw_dirty = true;
  HIP_TRY(hipStreamSynchronize(h->stream));
  return NRG_CHEM_OK;
}

void *nrg_mlp_stream(nrg_mlp_t *h) { return h ? (void *)h->stream : nullptr; }

}  // extern "C"
