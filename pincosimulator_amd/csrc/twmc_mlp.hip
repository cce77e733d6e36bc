// twmc_mlp.hip -- the warm start's network: a small fully connected MLP
// (inputs -> hidden layers with exact-erf GELU -> linear outputs) trained and
// evaluated by the kernels in this file, FP32 throughout, behind the C ABI
// twmc_mlp_* of include/twmc_hip.h.  No reference counterpart: the network
// maps drive / lattice parameters to a Gaussian steady-state estimate (mean
// field + radial k-space populations) that seeds TWMC_INIT_GAUSSIAN.
//
// Layout: activations row-major [rows][features]; layer l holds W_l
// [in_l][out_l] row-major followed by b_l [out_l] in one flat FP32 parameter
// vector, so Z_l = A_{l-1} W_l + b_l is a plain NN product.
//
// Networks of widths up to 256 (the warm start's has 256) take two launches per
// minibatch, or one for inference on few rows:
//   mlp_rows_kernel        four samples per workgroup through the whole network:
//                          forward, loss, and back to every layer's dZ
//   mlp_wgrad_kernel       weight and bias gradients as one product per layer,
//                          with the Adam update in its epilogue
//   mlp_pack_kernel        their copies of the weights, W and W^T of every layer
//                          with rows padded to 16 bytes, whenever parameters
//                          are set (the Adam update keeps both from then on)
// Kernels of wider networks and of inference on many rows (fused_forward), layer by layer:
//   mlp_gemm_kernel<MODE>  C[M x N] = op(A)[M x K] op(B)[K x N] with strided
//                          operands (covers NN forward, NT for dA = dZ W^T, TN
//                          for dW = A^T dZ), 64x64 tile per 256-thread
//                          workgroup, K staged through LDS 16 at a time, 4x4
//                          outputs per thread; epilogues: plain, +bias,
//                          +bias then GELU (keeping the pre-activation), and
//                          times GELU'(Z) for the backward pass
//   mlp_colsum_kernel      bias gradient, fixed summation order
//   mlp_loss_kernel        weighted MSE and its gradient, one workgroup,
//                          fixed-order FP64 reduction
//   mlp_adam_kernel        Adam update with bias correction
//   mlp_gather_kernel      minibatch rows by index
// Every reduction runs in a fixed order, so training is bitwise repeatable.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "../../include/twmc_hip.h"
#include "twmc_rng.h"

namespace twmc {
namespace {

constexpr int kTile = 64;
constexpr int kTileK = 16;
constexpr int kMaxLayers = 16;

enum { EPI_STORE = 0, EPI_BIAS = 1, EPI_BIAS_GELU = 2, EPI_GELU_BACK = 3 };

struct GemmArgs {
  int M, N, K;
  const float* A;
  long sam, sak;  // A(m, k) = A[m sam + k sak]
  const float* B;
  long sbk, sbn;  // B(k, n) = B[k sbk + n sbn]
  float* C;       // row-major M x N
  const float* bias;  // [N]
  float* Z;           // EPI_BIAS_GELU: pre-activation out, row-major M x N
  const float* Zin;   // EPI_GELU_BACK: pre-activation in
};

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float x) {
  // d/dx x Phi(x) = Phi(x) + x phi(x)
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

template <int MODE>
__global__ void __launch_bounds__(256) mlp_gemm_kernel(GemmArgs g) {
  __shared__ float As[kTileK][kTile + 4];
  __shared__ float Bs[kTileK][kTile + 4];
  const int m0 = blockIdx.y * kTile, n0 = blockIdx.x * kTile;
  const int tid = threadIdx.x;
  const int tm = tid >> 4, tn = tid & 15;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;

  for (int k0 = 0; k0 < g.K; k0 += kTileK) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int idx = tid + 256 * e;
      // A tile 64 (m) x 16 (k)
      const int mm = idx >> 4, kk = idx & 15;
      const int m = m0 + mm, k = k0 + kk;
      As[kk][mm] = (m < g.M && k < g.K) ? g.A[(long)m * g.sam + (long)k * g.sak] : 0.0f;
      // B tile 16 (k) x 64 (n)
      const int kb = idx >> 6, nb = idx & 63;
      const int k2 = k0 + kb, n = n0 + nb;
      Bs[kb][nb] = (k2 < g.K && n < g.N) ? g.B[(long)k2 * g.sbk + (long)n * g.sbn] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < kTileK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][tm * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tn * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + tm * 4 + i;
    if (m >= g.M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tn * 4 + j;
      if (n >= g.N) continue;
      const long o = (long)m * g.N + n;
      float v = acc[i][j];
      if (MODE == EPI_BIAS) {
        v += g.bias[n];
      } else if (MODE == EPI_BIAS_GELU) {
        v += g.bias[n];
        g.Z[o] = v;
        v = gelu(v);
      } else if (MODE == EPI_GELU_BACK) {
        v *= gelu_grad(g.Zin[o]);
      }
      g.C[o] = v;
    }
  }
}

// db[n] = sum_m dZ[m][n], summed in row order
__global__ void mlp_colsum_kernel(const float* dZ, int M, int N, float* db) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  float s = 0.0f;
  for (int m = 0; m < M; ++m) s += dZ[(long)m * N + n];
  db[n] = s;
}

// loss = sum_ij w_ij (y_ij - t_ij)^2 / rows ; dY = 2 w (y - t) / rows
__global__ void __launch_bounds__(256) mlp_loss_kernel(const float* Y, const float* T, const float* W, long count,
                                                       int rows, float* dY, double* loss_out) {
  __shared__ double red[256];
  double s = 0.0;
  const float inv = 1.0f / float(rows);
  for (long i = threadIdx.x; i < count; i += 256) {
    const float d = Y[i] - T[i];
    const float w = W ? W[i] : 1.0f;
    s += double(w) * double(d) * double(d);
    if (dY) dY[i] = 2.0f * w * d * inv;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0 && loss_out) *loss_out = red[0] / double(rows);
}

__global__ void mlp_adam_kernel(float* p, const float* g, float* m, float* v, long n, float lr, float b1, float b2,
                                float eps, float bc1, float bc2) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * bc1) / (sqrtf(vi * bc2) + eps);
  }
}

__global__ void mlp_gather_kernel(const float* src, int cols, const int* idx, int rows, float* dst) {
  const long total = (long)rows * cols;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const long r = e / cols, c = e - r * cols;
    dst[e] = src[(long)idx[r] * cols + c];
  }
}

// ---------------------------------------------------------------- narrow networks
constexpr int kMaxNarrow = 256;  // widest layer of the fused kernels
constexpr int kRowsBlock = 4;    // samples per workgroup
constexpr int kRowWaves = 16;    // waves per workgroup: each takes a sixteenth of the summed index
constexpr int kActLd = kMaxNarrow + 16;  // LDS row stride: the A operand's 4 rows x 16 columns in 64 banks

typedef float f32x4 __attribute__((ext_vector_type(4)));

// the network and one launch's rows; layer l = 1..n_layers maps width[l - 1] to width[l]
struct NetArgs {
  int n_layers, rows;
  int width[kMaxLayers + 1];
  int w_off[kMaxLayers], b_off[kMaxLayers];  // W, b in params
  int f_off[kMaxLayers], t_off[kMaxLayers];  // W [in][pad4(out)], W^T [out][pad4(in)] in packed
  const float* params;
  const float* packed;
  const float* x;     // samples, by idx[row] (idx null: by row)
  const float* t;     // targets and weights (weights null: all one); t null: forward only
  const float* w;
  const int* idx;
  float* act[kMaxLayers + 1];  // rows x width[l]: inputs of layer l + 1; act[n_layers]: outputs (forward only)
  float* dz[kMaxLayers + 1];   // rows x width[l]
  double* loss;                // [gridDim.x] partial sums of w (y - t)^2
};

__host__ __device__ constexpr int pad4(int n) { return (n + 3) / 4 * 4; }

// One product's share of a wave: weight rows k0 .. k0 + nk - 1 of the K, at the
// lane's four columns 4 lane + j.
struct RowTask {
  const float* W;
  int K, N, kc, k0, nk;
};

__device__ __forceinline__ RowTask row_task(const float* W, int K, int N, int wave) {
  RowTask t{W, K, N, (K + kRowWaves - 1) / kRowWaves, 0, 0};
  t.k0 = wave * t.kc;
  t.nk = min(t.kc, K - t.k0);
  return t;
}

// The loads carry no branch, so that all are in flight together: rows and
// columns past the end read the last one (their products are skipped or not
// stored).
template <int ROWS>
__device__ __forceinline__ void row_load_n(const RowTask& t, int lane, f32x4 (&wr)[16]) {
  const uint32_t c = (uint32_t)min(4 * lane, pad4(t.N) - 4);
#pragma unroll
  for (int kk = 0; kk < ROWS; ++kk) {
    const float* p = t.W + min(t.k0 + kk, t.K - 1) * pad4(t.N);  // wave-uniform
    wr[kk] = *reinterpret_cast<const f32x4*>(p + c);
  }
}

__device__ __forceinline__ void row_load(const RowTask& t, int lane, f32x4 (&wr)[16]) {
  if (t.nk <= 0) return;  // wave-uniform, as kc
  if (t.kc <= 4)
    row_load_n<4>(t, lane, wr);
  else
    row_load_n<16>(t, lane, wr);
}

// acc += the samples' values of k = kk (block kk of a, broadcast) times W's row
template <int KK>
__device__ __forceinline__ void row_mfma(float a, const f32x4 (&wr)[16], f32x4 (&acc)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, wr[KK][j], acc[j], 4, KK, 0);
}
template <int... KK>
__device__ __forceinline__ void row_product(int nk, float a, const f32x4 (&wr)[16], f32x4 (&acc)[4],
                                            std::integer_sequence<int, KK...>) {
  if (nk == 16)
    (row_mfma<KK>(a, wr, acc), ...);
  else
    ((KK < nk ? row_mfma<KK>(a, wr, acc) : void()), ...);
}

// A workgroup takes four samples through the whole network: products of 4 x K by
// K x N, N and K up to 256.  Bound by one CU's serial chain of layers, whatever
// the number of samples: per 256 x 256 layer 256 KB of weights through 64 B per
// clock (1.7 us), 0.9 us of products, then the partial sums and two barriers.
// Batches are small (64 in training), so few samples per workgroup spread them
// over more CUs.  Forward, loss and backward of 64 samples of the warm start's
// network: 26.6 us, 18.6 with the loads left out (before: ten launches, 250 us);
// other workgroups pulling the weights into the L2 ahead gave 1.5 us and were
// left out.  Each of the 16 waves holds a sixteenth of the weight rows in registers
// (16-byte loads, issued for the next layer as soon as this one's are used) and
// multiplies them on v_mfma_f32_4x4x1: its 16 blocks are 64 columns of W for
// one k, its A block the four samples' values at that k, one of 16 in a
// register, broadcast to all blocks -- 8 clocks for 256 FP32 multiply-adds
// against 16 on the VALU.  The waves' partial sums meet in LDS.
// Activations, pre-activations (for GELU') and dZ stay in LDS; act and dZ also
// go to memory for mlp_wgrad_kernel.
template <bool TRAIN>
__global__ void __launch_bounds__(64 * kRowWaves) mlp_rows_kernel(NetArgs g) {
  extern __shared__ __align__(16) unsigned char smem[];
  float(*part)[kRowsBlock][kMaxNarrow] = reinterpret_cast<float(*)[kRowsBlock][kMaxNarrow]>(smem);
  float* cur = reinterpret_cast<float*>(smem + sizeof(float) * kRowWaves * kRowsBlock * kMaxNarrow);
  float* zbuf = cur + kRowsBlock * kActLd;  // [hidden layer][row][column]
  __shared__ double red[kRowWaves];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = tid >> 8, o = tid & 255;  // this thread's output of a layer
  const long row = (long)blockIdx.x * kRowsBlock + r;
  const bool live = row < g.rows;
  const long src = live ? (g.idx ? (long)g.idx[row] : row) : 0;
  const int L = g.n_layers, n_out = g.width[L];

  f32x4 wr[16];
  RowTask task = row_task(g.packed + g.f_off[0], g.width[0], g.width[1], wave);
  row_load(task, lane, wr);
  if (o < g.width[0]) {
    const float v = live ? g.x[src * g.width[0] + o] : 0.f;
    cur[r * kActLd + o] = v;
    if (TRAIN && live) g.act[0][row * g.width[0] + o] = v;
  }
  float target = 0.f, weight = 1.f;
  if (TRAIN && live && o < n_out) {
    target = g.t[src * n_out + o];
    if (g.w) weight = g.w[src * n_out + o];
  }
  __syncthreads();

  // forward layers 1..L, then (TRAIN) the layers L..2 backward
  const int n_tasks = TRAIN ? 2 * L - 1 : L;
  for (int it = 0; it < n_tasks; ++it) {
    const bool fwd = it < L;
    const int l = fwd ? it + 1 : 2 * L - it;  // the layer whose weights are used
    // the samples' values of this wave's k: lane 4 b + i holds sample i, k0 + b
    float a = 0.f;
    if ((lane >> 2) < task.nk) a = cur[(lane & 3) * kActLd + task.k0 + (lane >> 2)];
    f32x4 acc[4] = {};
    row_product(task.nk, a, wr, acc, std::make_integer_sequence<int, 16>{});
    const int N = task.N, n_waves = (task.K + task.kc - 1) / task.kc;
    if (it + 1 < n_tasks) {
      // the next product's weights: forward layer l + 1, or W^T of the next one down
      const int nl = it + 1 < L ? it + 2 : 2 * L - it - 1;
      const bool nf = it + 1 < L;
      task = row_task(g.packed + (nf ? g.f_off[nl - 1] : g.t_off[nl - 1]), g.width[nf ? nl - 1 : nl],
                      g.width[nf ? nl : nl - 1], wave);
      row_load(task, lane, wr);
    }
    if (wave < n_waves && 4 * lane < N) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(&part[wave][i][4 * lane]) = f32x4{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
    }
    __syncthreads();
    float v = 0.f;
    if (o < N) {
      for (int u = 0; u < n_waves; ++u) v += part[u][r][o];
      if (fwd) {
        v += g.params[g.b_off[l - 1] + o];
        if (l < L) {
          if (TRAIN) zbuf[((l - 1) * kRowsBlock + r) * kMaxNarrow + o] = v;
          v = gelu(v);
          if (TRAIN && live) g.act[l][row * N + o] = v;
        } else if (!TRAIN) {
          if (live) g.act[L][row * N + o] = v;
        }
      } else {
        v = live ? v * gelu_grad(zbuf[((l - 2) * kRowsBlock + r) * kMaxNarrow + o]) : 0.f;
        if (live) g.dz[l - 1][row * N + o] = v;
      }
    }
    if (TRAIN && it == L - 1) {
      // loss and dZ of the outputs: dY = 2 w (y - t) / rows
      double s = 0.0;
      if (live && o < N) {
        const float d = v - target;
        s = double(weight) * double(d) * double(d);
        v = 2.0f * weight * d * (1.0f / float(g.rows));
        g.dz[L][row * N + o] = v;
      } else {
        v = 0.f;
      }
#pragma unroll
      for (int h = 32; h > 0; h >>= 1) s += __shfl_xor(s, h, 64);
      if (lane == 0) red[wave] = s;
    }
    if (o < N) cur[r * kActLd + o] = v;
    __syncthreads();
  }
  if (TRAIN && tid == 0) {
    double s = 0.0;
    for (int u = 0; u < kRowWaves; ++u) s += red[u];
    g.loss[blockIdx.x] = s;
  }
}

constexpr size_t rows_lds_bytes(int hidden_layers, bool train) {
  return sizeof(float) * (kRowWaves * kRowsBlock * kMaxNarrow + kRowsBlock * kActLd +
                          (train ? hidden_layers * kRowsBlock * kMaxNarrow : 0));
}

// Gradients of all layers: dW_l (and db_l, as the row of a constant input 1)
// = [A_{l-1}, 1]^T dZ_l, summed over the rows.  One wave per 16 x 16 tile on
// v_mfma_f32_16x16x4 (operands straight from memory, 64-byte segments: each is
// used by few tiles, and a batch of 64 rows is 16 products); ADAM applies the
// update to the tile's parameters and to their packed copies.
// Bound by latency: with 64 rows of the warm start's network, 6.9 us for the
// launch, a tile's loads, 16 dependent products and the update (before: the
// products on one to sixteen workgroups, a column sum that one thread ran through
// all rows and an update launch, 150 us).
struct GradArgs {
  NetArgs net;
  int tile0[kMaxLayers + 1];  // first tile of each layer
  int n_blocks_rows;          // partial losses
  double* loss_out;           // one value: sum of the partial losses / rows
  float* grads;               // !ADAM
  float *p, *packed, *m, *v;  // ADAM
  float lr, b1, b2, eps, bc1, bc2;
};

template <bool ADAM>
__global__ void __launch_bounds__(256) mlp_wgrad_kernel(GradArgs g) {
  __shared__ double red[256];
  const int tid = threadIdx.x, lane = tid & 63;
  if (blockIdx.x == 0) {
    // the minibatch's loss: the workgroups' partial sums in a fixed order
    double s = 0.0;
    for (int i = tid; i < g.n_blocks_rows; i += 256) s += g.net.loss[i];
    red[tid] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
      if (tid < h) red[tid] += red[tid + h];
      __syncthreads();
    }
    if (tid == 0) *g.loss_out = red[0] / double(g.net.rows);
  }
  const int tile = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (tid >> 6));
  if (tile >= g.tile0[g.net.n_layers]) return;
  int l = 1;
#pragma unroll
  for (int k = 1; k < kMaxLayers; ++k) l += k < g.net.n_layers && tile >= g.tile0[k];
  const int in = g.net.width[l - 1], out = g.net.width[l];
  const int cols = (out + 15) / 16, q = tile - g.tile0[l - 1];
  const int i0 = (q / cols) * 16, o0 = (q % cols) * 16;
  const int c = lane & 15, kq = lane >> 4;
  const int ia = i0 + c, ob = o0 + c;
  const float* A = g.net.act[l - 1];
  const float* Z = g.net.dz[l];
  const int rows = g.net.rows;
  // this lane's entries i0 + 4 kq + e of column ob (row `in` is the bias); the
  // update's operands are read now, beside the product's
  const long at0 = g.net.w_off[l - 1] + (long)(i0 + 4 * kq) * out + ob;
  const int n_e = ob < out ? min(4, in + 1 - (i0 + 4 * kq)) : 0;
  float p0[4], m0[4], v0[4];
  if (ADAM)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < n_e) {
        p0[e] = g.p[at0 + (long)e * out];
        m0[e] = g.m[at0 + (long)e * out];
        v0[e] = g.v[at0 + (long)e * out];
      }
  f32x4 acc = {};
  for (int b0 = 0; b0 < rows; b0 += 64) {
    float a[16], z[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int b = b0 + 4 * u + kq;
      a[u] = b < rows ? (ia < in ? A[(long)b * in + ia] : ia == in ? 1.f : 0.f) : 0.f;
      z[u] = b < rows && ob < out ? Z[(long)b * out + ob] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], z[u], acc, 0, 0, 0);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (e >= n_e) continue;
    const int i = i0 + 4 * kq + e;
    const long at = at0 + (long)e * out;
    const float gi = acc[e];
    if (!ADAM) {
      g.grads[at] = gi;
    } else {
      const float mi = g.b1 * m0[e] + (1.0f - g.b1) * gi;
      const float vi = g.b2 * v0[e] + (1.0f - g.b2) * gi * gi;
      g.m[at] = mi;
      g.v[at] = vi;
      const float pn = p0[e] - g.lr * (mi * g.bc1) / (sqrtf(vi * g.bc2) + g.eps);
      g.p[at] = pn;
      if (i < in) {
        g.packed[g.net.f_off[l - 1] + i * pad4(out) + ob] = pn;
        g.packed[g.net.t_off[l - 1] + ob * pad4(in) + i] = pn;
      }
    }
  }
}

// packed W [in][pad4(out)] and W^T [out][pad4(in)] of every layer (the padding
// is never used in a stored result)
__global__ void mlp_pack_kernel(NetArgs g, float* packed) {
  for (int l = 1; l <= g.n_layers; ++l) {
    const int in = g.width[l - 1], out = g.width[l];
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < in * out; e += gridDim.x * blockDim.x) {
      const int i = e / out, o = e - i * out;
      const float v = g.params[g.w_off[l - 1] + e];
      packed[g.f_off[l - 1] + i * pad4(out) + o] = v;
      packed[g.t_off[l - 1] + o * pad4(in) + i] = v;
    }
  }
}

struct Buf {
  void* p = nullptr;
  size_t bytes = 0;
  hipError_t ensure(size_t b) {
    if (b <= bytes) return hipSuccess;
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
    hipError_t e = hipMalloc(&p, std::max<size_t>(b, 256));
    if (e == hipSuccess) bytes = b;
    return e;
  }
  float* f() const { return static_cast<float*>(p); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
};

struct MlpCtx {
  int device = 0;
  hipStream_t stream = nullptr;
  int n_layers = 0;            // linear layers
  int width[kMaxLayers + 1];   // width[0] = inputs, width[n_layers] = outputs
  size_t w_off[kMaxLayers], b_off[kMaxLayers];
  size_t n_params = 0;
  uint64_t adam_t = 0;
  Buf params, grads, adam_m, adam_v;
  Buf act[kMaxLayers + 1];     // act[0] = input rows, act[l] = GELU(Z_l) or outputs
  Buf pre[kMaxLayers];         // Z_l of hidden layers
  Buf dA, dB;                  // backward ping-pong, rows x max width
  Buf data_x, data_t, data_w, bt, bw, idx, loss;
  // widths up to 256: the fused kernels' packed weights, dZ and partial losses
  bool narrow = false;
  Buf packed, dz[kMaxLayers + 1], loss_part;
  size_t f_off[kMaxLayers], t_off[kMaxLayers], n_packed = 0;
  int* perm[2] = {nullptr, nullptr};  // epoch orders, one computed while the other is used
  bool perm_pinned = false;
  hipEvent_t perm_ev[2] = {nullptr, nullptr};
  size_t perm_cap = 0;
  std::string err;
};

thread_local std::string g_mlp_err;

// (a HIP error is cleared: the next call's hipGetLastError would report it again)
int mlp_fail(MlpCtx* c, int code, const std::string& m) {
  if (code == TWMC_ERR_HIP) (void)hipGetLastError();
  if (c) c->err = m;
  g_mlp_err = m;
  return code;
}

#define MLPCHK(c, expr)                                                                      \
  do {                                                                                       \
    hipError_t e_ = (expr);                                                                  \
    if (e_ != hipSuccess) return mlp_fail(c, TWMC_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

hipError_t gemm(MlpCtx* c, int mode, const GemmArgs& a) {
  dim3 grid((unsigned)((a.N + kTile - 1) / kTile), (unsigned)((a.M + kTile - 1) / kTile));
  switch (mode) {
    case EPI_STORE: hipLaunchKernelGGL(mlp_gemm_kernel<EPI_STORE>, grid, dim3(256), 0, c->stream, a); break;
    case EPI_BIAS: hipLaunchKernelGGL(mlp_gemm_kernel<EPI_BIAS>, grid, dim3(256), 0, c->stream, a); break;
    case EPI_BIAS_GELU: hipLaunchKernelGGL(mlp_gemm_kernel<EPI_BIAS_GELU>, grid, dim3(256), 0, c->stream, a); break;
    default: hipLaunchKernelGGL(mlp_gemm_kernel<EPI_GELU_BACK>, grid, dim3(256), 0, c->stream, a); break;
  }
  return hipGetLastError();
}

int max_width(const MlpCtx* c) {
  int w = 0;
  for (int l = 0; l <= c->n_layers; ++l) w = std::max(w, c->width[l]);
  return w;
}

// each buffer by its own size: after an allocation that failed, no other one's size says
// that it is there
int ensure_rows(MlpCtx* c, int rows) {
  for (int l = 0; l <= c->n_layers; ++l) MLPCHK(c, c->act[l].ensure((size_t)rows * c->width[l] * 4));
  for (int l = 1; l < c->n_layers; ++l) MLPCHK(c, c->pre[l].ensure((size_t)rows * c->width[l] * 4));
  const size_t mw = (size_t)max_width(c);
  MLPCHK(c, c->dA.ensure((size_t)rows * mw * 4));
  MLPCHK(c, c->dB.ensure((size_t)rows * mw * 4));
  MLPCHK(c, c->bt.ensure((size_t)rows * c->width[c->n_layers] * 4));
  MLPCHK(c, c->bw.ensure((size_t)rows * c->width[c->n_layers] * 4));
  return TWMC_OK;
}

// the fused kernels' buffers for `rows` rows (only act[n_layers] without training)
int ensure_narrow(MlpCtx* c, int rows, bool train) {
  MLPCHK(c, c->act[c->n_layers].ensure((size_t)rows * c->width[c->n_layers] * 4));
  if (!train) return TWMC_OK;
  for (int l = 0; l < c->n_layers; ++l) MLPCHK(c, c->act[l].ensure((size_t)rows * c->width[l] * 4));
  for (int l = 1; l <= c->n_layers; ++l) MLPCHK(c, c->dz[l].ensure((size_t)rows * c->width[l] * 4));
  MLPCHK(c, c->loss_part.ensure((size_t)(rows + kRowsBlock - 1) / kRowsBlock * 8));
  return TWMC_OK;
}

NetArgs net_args(const MlpCtx* c, int rows, const float* x, const float* t, const float* w, const int* idx) {
  NetArgs a{};
  a.n_layers = c->n_layers;
  a.rows = rows;
  for (int l = 0; l <= c->n_layers; ++l) {
    a.width[l] = c->width[l];
    a.act[l] = c->act[l].f();
    a.dz[l] = c->dz[l].f();
  }
  for (int l = 0; l < c->n_layers; ++l) {
    a.w_off[l] = (int)c->w_off[l];
    a.b_off[l] = (int)c->b_off[l];
    a.f_off[l] = (int)c->f_off[l];
    a.t_off[l] = (int)c->t_off[l];
  }
  a.params = c->params.f();
  a.packed = c->packed.f();
  a.x = x;
  a.t = t;
  a.w = w;
  a.idx = idx;
  a.loss = static_cast<double*>(c->loss_part.p);
  return a;
}

hipError_t launch_rows(const MlpCtx* c, const NetArgs& a, bool train) {
  const size_t lds = rows_lds_bytes(c->n_layers - 1, train);
  const dim3 grid((unsigned)((a.rows + kRowsBlock - 1) / kRowsBlock)), block(64 * kRowWaves);
  if (train)
    hipLaunchKernelGGL(mlp_rows_kernel<true>, grid, block, lds, c->stream, a);
  else
    hipLaunchKernelGGL(mlp_rows_kernel<false>, grid, block, lds, c->stream, a);
  return hipGetLastError();
}

// the gradient launch after a training launch_rows over the same rows
GradArgs grad_args(const MlpCtx* c, const NetArgs& net, double* loss_out) {
  GradArgs a{};
  a.net = net;
  for (int l = 1; l <= c->n_layers; ++l)
    a.tile0[l] = a.tile0[l - 1] + ((c->width[l - 1] + 1 + 15) / 16) * ((c->width[l] + 15) / 16);
  a.n_blocks_rows = (net.rows + kRowsBlock - 1) / kRowsBlock;
  a.loss_out = loss_out;
  a.grads = c->grads.f();
  a.p = c->params.f();
  a.packed = c->packed.f();
  a.m = c->adam_m.f();
  a.v = c->adam_v.f();
  return a;
}

hipError_t launch_wgrad(const MlpCtx* c, const GradArgs& a, bool adam) {
  const dim3 grid((unsigned)((a.tile0[c->n_layers] + 3) / 4));
  if (adam)
    hipLaunchKernelGGL(mlp_wgrad_kernel<true>, grid, dim3(256), 0, c->stream, a);
  else
    hipLaunchKernelGGL(mlp_wgrad_kernel<false>, grid, dim3(256), 0, c->stream, a);
  return hipGetLastError();
}

// the fused path: every width at most kMaxNarrow.  Wider networks take the
// layer-by-layer products.
bool is_narrow(const MlpCtx* c) {
  // the pre-activations of all hidden layers (4 KB each) lie beside the 69 KB of partial
  // sums and activations in the LDS
  static_assert(rows_lds_bytes(kMaxLayers - 1, true) + 1024 <= 160 * 1024, "a network of kMaxLayers does not fit");
  for (int l = 0; l <= c->n_layers; ++l)
    if (c->width[l] > kMaxNarrow) return false;
  return true;
}

// Inference on the fused kernel: every four samples read all weights, so from some
// number of rows on the products of 64 samples at a time take less.  The whole call,
// fused / layer by layer, ms: 5-3x256-34 4096 rows 0.11 / 0.22, 8192 0.22 / 0.28, 16384
// 0.39 / 0.39, 65536 1.47 / 1.12; 64-4x128-64 8192 0.35 / 0.36, 16384 0.66 / 0.56; 3-8x32-2
// 8192 0.15 / 0.26, 16384 0.28 / 0.26; a few narrow layers: 5-2x64-8 4096 0.061 / 0.074,
// 8192 0.091 / 0.083, 5-1x16-4 4096 0.051 / 0.049, 8192 0.075 / 0.056.  (Training gains at
// any batch: the gradients of 65536 samples of 5-3x256-34 114 -> 3.4 ms.)
bool fused_forward(const MlpCtx* c, uint64_t rows) {
  return c->narrow && rows <= (max_width(c) <= 64 && c->n_layers <= 3 ? 4096u : 8192u);
}

// forward over act[0] (rows x inputs); outputs in act[n_layers]
int forward(MlpCtx* c, int rows) {
  for (int l = 1; l <= c->n_layers; ++l) {
    GemmArgs a{};
    a.M = rows;
    a.N = c->width[l];
    a.K = c->width[l - 1];
    a.A = c->act[l - 1].f();
    a.sam = a.K;
    a.sak = 1;
    a.B = c->params.f() + c->w_off[l - 1];
    a.sbk = a.N;
    a.sbn = 1;
    a.C = c->act[l].f();
    a.bias = c->params.f() + c->b_off[l - 1];
    const bool hidden = l < c->n_layers;
    if (hidden) a.Z = c->pre[l].f();
    MLPCHK(c, gemm(c, hidden ? EPI_BIAS_GELU : EPI_BIAS, a));
  }
  return TWMC_OK;
}

// backward from dY (in dA) to the parameter gradients
int backward(MlpCtx* c, int rows) {
  float* dcur = c->dA.f();
  float* dnext = c->dB.f();
  for (int l = c->n_layers; l >= 1; --l) {
    const int in = c->width[l - 1], out = c->width[l];
    // dW_l = A_{l-1}^T dZ_l : (in x rows) (rows x out)
    GemmArgs w{};
    w.M = in;
    w.N = out;
    w.K = rows;
    w.A = c->act[l - 1].f();
    w.sam = 1;
    w.sak = in;
    w.B = dcur;
    w.sbk = out;
    w.sbn = 1;
    w.C = c->grads.f() + c->w_off[l - 1];
    MLPCHK(c, gemm(c, EPI_STORE, w));
    hipLaunchKernelGGL(mlp_colsum_kernel, dim3((unsigned)((out + 255) / 256)), dim3(256), 0, c->stream,
                       (const float*)dcur, rows, out, c->grads.f() + c->b_off[l - 1]);
    MLPCHK(c, hipGetLastError());
    if (l > 1) {
      // dZ_{l-1} = (dZ_l W_l^T) . GELU'(Z_{l-1}) : (rows x out) (out x in)
      GemmArgs d{};
      d.M = rows;
      d.N = in;
      d.K = out;
      d.A = dcur;
      d.sam = out;
      d.sak = 1;
      d.B = c->params.f() + c->w_off[l - 1];
      d.sbk = 1;
      d.sbn = out;
      d.C = dnext;
      d.Zin = c->pre[l - 1].f();
      MLPCHK(c, gemm(c, EPI_GELU_BACK, d));
      std::swap(dcur, dnext);
    }
  }
  return TWMC_OK;
}

int loss_and_grad(MlpCtx* c, const float* T, const float* W, int rows, double* loss_dev) {
  const int out = c->width[c->n_layers];
  hipLaunchKernelGGL(mlp_loss_kernel, dim3(1), dim3(256), 0, c->stream, (const float*)c->act[c->n_layers].f(), T, W,
                     (long)rows * out, rows, c->dA.f(), loss_dev);
  MLPCHK(c, hipGetLastError());
  return backward(c, rows);
}

// splitmix64: host-side shuffles and initial weights
uint64_t splitmix(uint64_t& s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// the samples of a call on the device
int upload_data(MlpCtx* c, const float* x, const float* t, const float* w, uint64_t rows) {
  const size_t nin = (size_t)c->width[0], nout = (size_t)c->width[c->n_layers];
  MLPCHK(c, c->data_x.ensure(rows * nin * 4));
  MLPCHK(c, c->data_t.ensure(rows * nout * 4));
  if (w) MLPCHK(c, c->data_w.ensure(rows * nout * 4));
  MLPCHK(c, hipMemcpyAsync(c->data_x.p, x, rows * nin * 4, hipMemcpyHostToDevice, c->stream));
  MLPCHK(c, hipMemcpyAsync(c->data_t.p, t, rows * nout * 4, hipMemcpyHostToDevice, c->stream));
  if (w) MLPCHK(c, hipMemcpyAsync(c->data_w.p, w, rows * nout * 4, hipMemcpyHostToDevice, c->stream));
  return TWMC_OK;
}

void release_perm(MlpCtx* c) {
  for (int*& p : c->perm) {
    if (c->perm_pinned) (void)hipHostFree(p);
    else std::free(p);
    p = nullptr;
  }
  c->perm_cap = 0;
}

// two buffers for epoch orders of `rows` samples: pinned, or if there is no pinned
// memory to be had, pageable
int ensure_perm(MlpCtx* c, size_t rows) {
  for (int k = 0; k < 2; ++k)
    if (!c->perm_ev[k]) MLPCHK(c, hipEventCreateWithFlags(&c->perm_ev[k], hipEventDisableTiming));
  if (rows <= c->perm_cap) return TWMC_OK;
  release_perm(c);
  c->perm_pinned = true;
  for (int*& p : c->perm)
    if (hipHostMalloc(reinterpret_cast<void**>(&p), rows * sizeof(int), hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
      release_perm(c);
      c->perm_pinned = false;
      break;
    }
  if (!c->perm_pinned)
    for (int*& p : c->perm)
      if (!(p = static_cast<int*>(std::malloc(rows * sizeof(int)))))
        return mlp_fail(c, TWMC_ERR_NOMEM, "no memory for the epochs' orders");
  c->perm_cap = rows;
  return TWMC_OK;
}

// a shuffled epoch (Fisher-Yates)
void shuffle_epoch(int* perm, uint64_t rows, uint64_t& s) {
  for (uint64_t i = 0; i < rows; ++i) perm[i] = (int)i;
  for (uint64_t i = rows - 1; i > 0; --i) std::swap(perm[i], perm[splitmix(s) % (i + 1)]);
}

}  // namespace
}  // namespace twmc

using namespace twmc;

extern "C" {

const char* twmc_mlp_last_error(const twmc_mlp_ctx* ctx) {
  if (ctx) return reinterpret_cast<const MlpCtx*>(ctx)->err.c_str();
  return g_mlp_err.c_str();
}

int twmc_mlp_create(const twmc_mlp_config* cfg, int device, twmc_mlp_ctx** ctx_out) {
  if (!cfg || !ctx_out) return mlp_fail(nullptr, TWMC_ERR_INVALID, "null argument");
  *ctx_out = nullptr;
  if (cfg->n_in < 1 || cfg->n_out < 1 || cfg->n_hidden < 1 || cfg->n_hidden_layers < 0 ||
      cfg->n_hidden_layers + 1 > kMaxLayers || cfg->n_in > 65536 || cfg->n_out > 65536 || cfg->n_hidden > 65536)
    return mlp_fail(nullptr, TWMC_ERR_INVALID, "bad network shape");
  MlpCtx* c = new MlpCtx();
  c->device = device;
  c->n_layers = cfg->n_hidden_layers + 1;
  c->width[0] = cfg->n_in;
  for (int l = 1; l < c->n_layers; ++l) c->width[l] = cfg->n_hidden;
  c->width[c->n_layers] = cfg->n_out;
  size_t off = 0;
  for (int l = 0; l < c->n_layers; ++l) {
    c->w_off[l] = off;
    off += (size_t)c->width[l] * c->width[l + 1];
    c->b_off[l] = off;
    off += (size_t)c->width[l + 1];
  }
  c->n_params = off;
  for (int l = 0; l < c->n_layers; ++l) {
    c->f_off[l] = c->n_packed;
    c->n_packed += (size_t)c->width[l] * pad4(c->width[l + 1]);
    c->t_off[l] = c->n_packed;
    c->n_packed += (size_t)c->width[l + 1] * pad4(c->width[l]);
  }
  c->narrow = is_narrow(c);
  hipError_t e = hipSetDevice(device);
  if (e == hipSuccess && c->narrow)
    e = hipFuncSetAttribute((const void*)mlp_rows_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)rows_lds_bytes(kMaxLayers - 1, true));
  if (e == hipSuccess && c->narrow)
    e = hipFuncSetAttribute((const void*)mlp_rows_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)rows_lds_bytes(0, false));
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = c->params.ensure(off * 4);
  if (e == hipSuccess) e = c->grads.ensure(off * 4);
  if (e == hipSuccess) e = c->adam_m.ensure(off * 4);
  if (e == hipSuccess) e = c->adam_v.ensure(off * 4);
  if (e == hipSuccess && c->narrow) e = c->packed.ensure(c->n_packed * 4);
  if (e == hipSuccess && c->narrow) e = hipMemsetAsync(c->packed.p, 0, c->n_packed * 4, c->stream);  // the padding
  if (e != hipSuccess) {
    std::string m = std::string("twmc_mlp_create: ") + hipGetErrorString(e);
    twmc_mlp_destroy(reinterpret_cast<twmc_mlp_ctx*>(c));
    return mlp_fail(nullptr, TWMC_ERR_HIP, m);
  }
  // Glorot-uniform weights, zero biases, deterministic in cfg->seed
  std::vector<float> p(off, 0.0f);
  uint64_t s = cfg->seed;
  for (int l = 0; l < c->n_layers; ++l) {
    const double a = std::sqrt(6.0 / double(c->width[l] + c->width[l + 1]));
    const size_t n = (size_t)c->width[l] * c->width[l + 1];
    for (size_t i = 0; i < n; ++i) {
      const double u = double(splitmix(s) >> 11) * (1.0 / 9007199254740992.0);
      p[c->w_off[l] + i] = float((2.0 * u - 1.0) * a);
    }
  }
  *ctx_out = reinterpret_cast<twmc_mlp_ctx*>(c);
  int rc = twmc_mlp_set_params(*ctx_out, p.data());
  if (rc != TWMC_OK) {
    std::string m = c->err;
    twmc_mlp_destroy(reinterpret_cast<twmc_mlp_ctx*>(c));
    *ctx_out = nullptr;
    return mlp_fail(nullptr, rc, m);
  }
  return TWMC_OK;
}

void twmc_mlp_destroy(twmc_mlp_ctx* ctx) {
  if (!ctx) return;
  MlpCtx* c = reinterpret_cast<MlpCtx*>(ctx);
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  Buf* bufs[] = {&c->params, &c->grads, &c->adam_m, &c->adam_v, &c->dA, &c->dB, &c->data_x, &c->data_t,
                 &c->data_w, &c->bt, &c->bw, &c->idx, &c->loss, &c->packed, &c->loss_part};
  for (Buf* b : bufs) b->release();
  for (int l = 0; l <= kMaxLayers; ++l) {
    c->act[l].release();
    c->dz[l].release();
  }
  release_perm(c);
  for (hipEvent_t e : c->perm_ev)
    if (e) (void)hipEventDestroy(e);
  for (int l = 0; l < kMaxLayers; ++l) c->pre[l].release();
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

uint64_t twmc_mlp_n_params(const twmc_mlp_ctx* ctx) { return ctx ? reinterpret_cast<const MlpCtx*>(ctx)->n_params : 0; }

int twmc_mlp_get_params(twmc_mlp_ctx* ctx, float* out) {
  if (!ctx || !out) return mlp_fail(nullptr, TWMC_ERR_INVALID, "null argument");
  MlpCtx* c = reinterpret_cast<MlpCtx*>(ctx);
  MLPCHK(c, hipSetDevice(c->device));
  MLPCHK(c, hipStreamSynchronize(c->stream));
  MLPCHK(c, hipMemcpy(out, c->params.p, c->n_params * 4, hipMemcpyDeviceToHost));
  return TWMC_OK;
}

int twmc_mlp_set_params(twmc_mlp_ctx* ctx, const float* in) {
  if (!ctx || !in) return mlp_fail(nullptr, TWMC_ERR_INVALID, "null argument");
  MlpCtx* c = reinterpret_cast<MlpCtx*>(ctx);
  MLPCHK(c, hipSetDevice(c->device));
  MLPCHK(c, hipStreamSynchronize(c->stream));
  MLPCHK(c, hipMemcpy(c->params.p, in, c->n_params * 4, hipMemcpyHostToDevice));
  std::vector<float> zero(c->n_params, 0.0f);
  MLPCHK(c, hipMemcpy(c->adam_m.p, zero.data(), c->n_params * 4, hipMemcpyHostToDevice));
  MLPCHK(c, hipMemcpy(c->adam_v.p, zero.data(), c->n_params * 4, hipMemcpyHostToDevice));
  if (c->narrow) {
    hipLaunchKernelGGL(mlp_pack_kernel, dim3(256), dim3(256), 0, c->stream,
                       net_args(c, 0, nullptr, nullptr, nullptr, nullptr), c->packed.f());
    MLPCHK(c, hipGetLastError());
  }
  c->adam_t = 0;
  return TWMC_OK;
}

int twmc_mlp_forward(twmc_mlp_ctx* ctx, const float* x, uint64_t rows, float* y) {
  if (!ctx || !x || !y) return mlp_fail(nullptr, TWMC_ERR_INVALID, "null argument");
  MlpCtx* c = reinterpret_cast<MlpCtx*>(ctx);
  if (rows == 0 || rows > (1u << 24)) return mlp_fail(c, TWMC_ERR_INVALID, "rows out of range");
  MLPCHK(c, hipSetDevice(c->device));
  const bool fused = fused_forward(c, rows);
  int rc = fused ? ensure_narrow(c, (int)rows, false) : ensure_rows(c, (int)rows);
  if (rc != TWMC_OK) return rc;
  if (fused) {
    MLPCHK(c, c->data_x.ensure(rows * c->width[0] * 4));
    MLPCHK(c, hipMemcpyAsync(c->data_x.p, x, rows * c->width[0] * 4, hipMemcpyHostToDevice, c->stream));
    MLPCHK(c, launch_rows(c, net_args(c, (int)rows, c->data_x.f(), nullptr, nullptr, nullptr), false));
  } else {
    MLPCHK(c, hipMemcpyAsync(c->act[0].p, x, rows * c->width[0] * 4, hipMemcpyHostToDevice, c->stream));
    rc = forward(c, (int)rows);
    if (rc != TWMC_OK) return rc;
  }
  MLPCHK(c, hipMemcpyAsync(y, c->act[c->n_layers].p, rows * c->width[c->n_layers] * 4, hipMemcpyDeviceToHost,
                           c->stream));
  MLPCHK(c, hipStreamSynchronize(c->stream));
  return TWMC_OK;
}

int twmc_mlp_loss_grad(twmc_mlp_ctx* ctx, const float* x, const float* t, const float* w, uint64_t rows, double* loss,
                       float* grad) {
  if (!ctx || !x || !t) return mlp_fail(nullptr, TWMC_ERR_INVALID, "null argument");
  MlpCtx* c = reinterpret_cast<MlpCtx*>(ctx);
  if (rows == 0 || rows > (1u << 24)) return mlp_fail(c, TWMC_ERR_INVALID, "rows out of range");
  MLPCHK(c, hipSetDevice(c->device));
  int rc = c->narrow ? ensure_narrow(c, (int)rows, true) : ensure_rows(c, (int)rows);
  if (rc != TWMC_OK) return rc;
  const size_t out = (size_t)c->width[c->n_layers];
  MLPCHK(c, c->loss.ensure(sizeof(double)));
  if (c->narrow) {
    rc = upload_data(c, x, t, w, rows);
    if (rc != TWMC_OK) return rc;
    const NetArgs net = net_args(c, (int)rows, c->data_x.f(), c->data_t.f(), w ? c->data_w.f() : nullptr, nullptr);
    MLPCHK(c, launch_rows(c, net, true));
    MLPCHK(c, launch_wgrad(c, grad_args(c, net, static_cast<double*>(c->loss.p)), false));
  } else {
    MLPCHK(c, hipMemcpyAsync(c->act[0].p, x, rows * c->width[0] * 4, hipMemcpyHostToDevice, c->stream));
    MLPCHK(c, hipMemcpyAsync(c->bt.p, t, rows * out * 4, hipMemcpyHostToDevice, c->stream));
    if (w) MLPCHK(c, hipMemcpyAsync(c->bw.p, w, rows * out * 4, hipMemcpyHostToDevice, c->stream));
    rc = forward(c, (int)rows);
    if (rc == TWMC_OK)
      rc = loss_and_grad(c, c->bt.f(), w ? c->bw.f() : nullptr, (int)rows, static_cast<double*>(c->loss.p));
    if (rc != TWMC_OK) return rc;
  }
  double l = 0.0;
  MLPCHK(c, hipMemcpyAsync(&l, c->loss.p, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  if (grad) MLPCHK(c, hipMemcpyAsync(grad, c->grads.p, c->n_params * 4, hipMemcpyDeviceToHost, c->stream));
  MLPCHK(c, hipStreamSynchronize(c->stream));
  if (loss) *loss = l;
  return TWMC_OK;
}

int twmc_mlp_train(twmc_mlp_ctx* ctx, const float* x, const float* t, const float* w, uint64_t rows,
                   const twmc_mlp_train_opts* o, double* epoch_loss) {
  if (!ctx || !x || !t || !o) return mlp_fail(nullptr, TWMC_ERR_INVALID, "null argument");
  MlpCtx* c = reinterpret_cast<MlpCtx*>(ctx);
  if (rows == 0 || rows > (1u << 24)) return mlp_fail(c, TWMC_ERR_INVALID, "rows out of range");
  if (o->epochs < 0 || o->batch < 1 || !(o->lr > 0.0f) || !(o->beta1 >= 0.0f && o->beta1 < 1.0f) ||
      !(o->beta2 >= 0.0f && o->beta2 < 1.0f) || !(o->eps > 0.0f))
    return mlp_fail(c, TWMC_ERR_INVALID, "bad training options");
  MLPCHK(c, hipSetDevice(c->device));
  // after an error return, nothing of the call may still use its buffers
  std::vector<double> bl;
  struct Drain {
    hipStream_t s;
    ~Drain() { (void)hipStreamSynchronize(s); }
  } drain{c->stream};
  const int nin = c->width[0], nout = c->width[c->n_layers];
  const int batch = (int)std::min<uint64_t>((uint64_t)o->batch, rows);
  int rc = c->narrow ? ensure_narrow(c, batch, true) : ensure_rows(c, batch);
  if (rc == TWMC_OK) rc = ensure_perm(c, rows);
  if (rc != TWMC_OK) return rc;
  MLPCHK(c, c->idx.ensure(rows * 4));
  const uint64_t n_batches = rows / (uint64_t)batch;  // the remainder of a shuffled epoch is dropped
  // losses stay on the device for up to `keep` epochs
  const int keep = (int)std::max<uint64_t>(1, std::min<uint64_t>((uint64_t)std::max(o->epochs, 1), 65536 / n_batches));
  MLPCHK(c, c->loss.ensure((size_t)keep * n_batches * sizeof(double)));
  rc = upload_data(c, x, t, w, rows);
  if (rc != TWMC_OK) return rc;
  const float* wd = w ? c->data_w.f() : nullptr;
  bl.resize((size_t)keep * n_batches);
  uint64_t s = o->shuffle_seed;
  if (o->epochs > 0) shuffle_epoch(c->perm[0], rows, s);
  for (int ep = 0; ep < o->epochs; ++ep) {
    MLPCHK(c, hipMemcpyAsync(c->idx.p, c->perm[ep & 1], rows * 4, hipMemcpyHostToDevice, c->stream));
    MLPCHK(c, hipEventRecord(c->perm_ev[ep & 1], c->stream));
    double* loss = static_cast<double*>(c->loss.p) + (size_t)(ep % keep) * n_batches;
    for (uint64_t b = 0; b < n_batches; ++b) {
      const int* ib = static_cast<const int*>(c->idx.p) + b * batch;
      c->adam_t += 1;
      const double bc1 = 1.0 / (1.0 - std::pow((double)o->beta1, (double)c->adam_t));
      const double bc2 = 1.0 / (1.0 - std::pow((double)o->beta2, (double)c->adam_t));
      if (c->narrow) {
        const NetArgs net = net_args(c, batch, c->data_x.f(), c->data_t.f(), wd, ib);
        GradArgs ga = grad_args(c, net, loss + b);
        ga.lr = o->lr;
        ga.b1 = o->beta1;
        ga.b2 = o->beta2;
        ga.eps = o->eps;
        ga.bc1 = (float)bc1;
        ga.bc2 = (float)bc2;
        MLPCHK(c, launch_rows(c, net, true));
        MLPCHK(c, launch_wgrad(c, ga, true));
        continue;
      }
      const int gx = (int)std::min<int64_t>(((int64_t)batch * nout + 255) / 256, 4096);
      hipLaunchKernelGGL(mlp_gather_kernel, dim3((unsigned)gx), dim3(256), 0, c->stream, (const float*)c->data_x.f(),
                         nin, ib, batch, c->act[0].f());
      hipLaunchKernelGGL(mlp_gather_kernel, dim3((unsigned)gx), dim3(256), 0, c->stream, (const float*)c->data_t.f(),
                         nout, ib, batch, c->bt.f());
      if (w)
        hipLaunchKernelGGL(mlp_gather_kernel, dim3((unsigned)gx), dim3(256), 0, c->stream,
                           (const float*)c->data_w.f(), nout, ib, batch, c->bw.f());
      MLPCHK(c, hipGetLastError());
      rc = forward(c, batch);
      if (rc == TWMC_OK) rc = loss_and_grad(c, c->bt.f(), w ? c->bw.f() : nullptr, batch, loss + b);
      if (rc != TWMC_OK) return rc;
      const int ga = (int)std::min<size_t>((c->n_params + 255) / 256, 2048);
      hipLaunchKernelGGL(mlp_adam_kernel, dim3((unsigned)ga), dim3(256), 0, c->stream, c->params.f(),
                         (const float*)c->grads.f(), c->adam_m.f(), c->adam_v.f(), (long)c->n_params, o->lr,
                         o->beta1, o->beta2, o->eps, (float)bc1, (float)bc2);
      MLPCHK(c, hipGetLastError());
    }
    if (ep + 1 < o->epochs) {
      // the next epoch's order, while the device works; its buffer was last
      // read by the copy of the epoch before this one
      if (ep > 0) MLPCHK(c, hipEventSynchronize(c->perm_ev[(ep + 1) & 1]));
      shuffle_epoch(c->perm[(ep + 1) & 1], rows, s);
    }
    if ((ep + 1) % keep == 0 || ep + 1 == o->epochs) {
      const int n_ep = ep % keep + 1;
      MLPCHK(c, hipMemcpyAsync(bl.data(), c->loss.p, (size_t)n_ep * n_batches * 8, hipMemcpyDeviceToHost, c->stream));
      MLPCHK(c, hipStreamSynchronize(c->stream));
      for (int k = 0; epoch_loss && k < n_ep; ++k) {
        double m = 0.0;
        for (uint64_t b = 0; b < n_batches; ++b) m += bl[(size_t)k * n_batches + b];
        epoch_loss[ep - n_ep + 1 + k] = m / double(n_batches);
      }
    }
  }
  return TWMC_OK;
}

}  // extern "C"
