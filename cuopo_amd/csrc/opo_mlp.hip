// opo_mlp.hip -- the warm-start surrogate: a small MLP (n_in -> width x depth,
// GELU -> n_out) trained and evaluated on the GPU with BF16 weights and
// activations and FP32 accumulation.  Every matrix product (forward, weight
// gradient, input gradient) runs through one hand-written MFMA kernel
// (v_mfma_f32_16x16x16_bf16, 64x64 or 32x32 block tiles); bias/GELU/GELU' are
// fused into its epilogue and the bias gradients' column sums run beside the
// weight gradients.  FP32 master weights, Adam in FP32.  No reference
// counterpart: cuOPO has no learned component.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <random>
#include <string>
#include <vector>

#include "../../include/opo.h"

namespace opo {
void set_error(const std::string &msg);  // opo_api.cpp: message returned by opo_last_error()
}

namespace {

int mfail(int code, const std::string &m) {
  opo::set_error(m);
  return code;
}
#define MCHK(x)                                                                                 \
  do {                                                                                          \
    hipError_t e_ = (x);                                                                        \
    if (e_ != hipSuccess) return mfail(OPO_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)
#define MRCHK(x)                  \
  do {                            \
    int r_ = (x);                 \
    if (r_ != OPO_OK) return r_;  \
  } while (0)

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// float -> bf16 bits, round to nearest even (NaN kept quiet)
__host__ __device__ inline unsigned short f2bf(float f) {
  unsigned int u;
  std::memcpy(&u, &f, 4);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return (unsigned short)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ inline float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float x) {
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

enum Epi : int {
  EPI_STORE = 0,       // C = acc (fp32)
  EPI_BIAS = 1,        // C = acc + bias[n] (fp32), no activation (output layer)
  EPI_BIAS_GELU = 2,   // Z = acc + bias[n] (fp32, optional), H = gelu(Z) (bf16)
  EPI_GELU_GRAD = 3,   // C = acc * gelu'(Zprev[m, n]) (fp32)
};

// One operand of a product: R rows (A's m or B's n) of K values.  `kc`: the K
// values of a row are contiguous, element (r, k) at p[r * ld + k]; otherwise
// the rows are, at p[k * ld + r].
template <typename T> struct Operand {
  const T *p;
  long long ld;
  int R;
  int vec;  // rows (kc) or columns (!kc) start on a vector boundary: whole vectors load at once
};

struct GemmArgs {
  int M, N, K;
  long long ldc;         // C(m, n) = C[m*ldc + n]
  const float *bias;     // [N]
  const float *zprev;    // EPI_GELU_GRAD: Z of the layer below, same shape as C
  float *zout;           // EPI_BIAS_GELU: pre-activation out (may be null)
  unsigned short *hout;  // EPI_BIAS_GELU: bf16 activation out
  float *cout;           // fp32 out
  const float *col_in;   // column sums beside the product (bias gradient), or null
  float *col_out;        // col_out[c] = sum over r of col_in[r*cols + c], r < rows, in order
  int col_rows, col_cols;
};

// A block's stage of one operand: ROWS rows x KC values, read from memory into
// registers (fetch), then written to LDS as bf16 with K contiguous (put), so
// that the next stages' reads are in flight while this one is multiplied.  The
// registers hold the words as loaded: taking them apart in fetch would wait
// for the loads there (78 instead of 40 us for 256 x 256 over K = 4096).
template <typename T, bool KCONT, int ROWS, int KC> struct Stage {
  // K contiguous: vectors of 8 values of a row.  Rows contiguous: 4 rows x 2
  // values, so that pairs of K go to LDS as one word.
  static constexpr int kUnits = ROWS * KC / 8 / 256;
  static constexpr int kPer = 4 / sizeof(T);  // values per word
  static constexpr int kWords = 8 / kPer;
  static_assert(kUnits >= 1 && ROWS * KC % 2048 == 0, "whole units per thread");
  unsigned w[kUnits][kWords];

  // value j of a unit as bf16 bits
  __device__ __forceinline__ unsigned bits(int u, int j) const {
    if constexpr (kPer == 1) return f2bf(__builtin_bit_cast(float, w[u][j]));
    else return j & 1 ? w[u][j / 2] >> 16 : w[u][j / 2] & 0xffffu;
  }
  static __device__ __forceinline__ unsigned word(const T *q, bool on0, bool on1) {
    if constexpr (kPer == 1) return on0 ? __builtin_bit_cast(unsigned, (float)q[0]) : 0u;
    else return (on0 ? (unsigned)q[0] : 0u) | (on1 ? (unsigned)q[1] << 16 : 0u);
  }
  __device__ __forceinline__ void fetch(const Operand<T> &o, int r0, int k0, int K, int tid) {
    struct alignas(16) Vec { unsigned x[4]; };
    struct alignas(4 * sizeof(T)) Quad { unsigned x[4 / kPer]; };
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      const int id = tid + u * 256;
      if constexpr (KCONT) {
        const int r = r0 + id / (KC / 8), k = k0 + id % (KC / 8) * 8;
        const T *q = o.p + (long long)r * o.ld + k;
        if (o.vec && r < o.R && k + 8 <= K) {
#pragma unroll
          for (int j = 0; j < kWords; j += 4) {
            const Vec h = reinterpret_cast<const Vec *>(q)[j / 4];
#pragma unroll
            for (int i = 0; i < 4; ++i) w[u][j + i] = h.x[i];
          }
        } else {
#pragma unroll
          for (int j = 0; j < kWords; ++j)
            w[u][j] = word(q + j * kPer, r < o.R && k + j * kPer < K, r < o.R && k + j * kPer + 1 < K);
        }
      } else {
        const int r = r0 + id % (ROWS / 4) * 4, k = k0 + id / (ROWS / 4) * 2;
        constexpr int H = kWords / 2;  // words per k
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const T *q = o.p + (long long)(k + j) * o.ld + r;
          if (o.vec && r + 4 <= o.R && k + j < K) {
            const Quad h = *reinterpret_cast<const Quad *>(q);
#pragma unroll
            for (int i = 0; i < H; ++i) w[u][H * j + i] = h.x[i];
          } else {
#pragma unroll
            for (int i = 0; i < H; ++i)
              w[u][H * j + i] = word(q + i * kPer, k + j < K && r + i * kPer < o.R, k + j < K && r + i * kPer + 1 < o.R);
          }
        }
      }
    }
  }
  __device__ __forceinline__ void put(unsigned short (*lds)[KC + 8], int tid) const {
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      const int id = tid + u * 256;
      if constexpr (KCONT) {
        struct alignas(16) Oct { unsigned x[4]; } h;
#pragma unroll
        for (int j = 0; j < 4; ++j) h.x[j] = kPer == 2 ? w[u][j % kWords] : bits(u, 2 * j) | bits(u, 2 * j + 1) << 16;
        *reinterpret_cast<Oct *>(&lds[id / (KC / 8)][id % (KC / 8) * 8]) = h;
      } else {
        const int r = id % (ROWS / 4) * 4, k = id / (ROWS / 4) * 2;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *reinterpret_cast<unsigned *>(&lds[r + i][k]) = bits(u, i) | bits(u, 4 + i) << 16;
      }
    }
  }
};

// db[c] = sum over the batch, one column per thread, in batch order; 32 rows
// are read ahead of the sums.
__device__ __forceinline__ void column_sums(const GemmArgs &g, int block, int tid) {
  const int c = block * 256 + tid;
  if (c >= g.col_cols) return;
  float s = 0;
  for (int r = 0; r < g.col_rows; r += 32) {
    float z[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) z[j] = r + j < g.col_rows ? g.col_in[(long long)(r + j) * g.col_cols + c] : 0.f;
#pragma unroll
    for (int j = 0; j < 32; ++j)
      if (r + j < g.col_rows) s += z[j];
  }
  g.col_out[c] = s;
}

// C[M x N] = A B^T over K: 256 threads, TILE x TILE of C, each wave a quarter
// in 16 x 16 blocks of v_mfma_f32_16x16x16_bf16, K in stages of KC through two
// LDS buffers (one barrier per stage) with the next stage in registers.  The
// products are accumulated in K order, 16 at a time, whatever the tile, so a
// result depends on neither TILE nor KC.
// What bounds it: latency.  The network's products are 256 wide, so a launch
// is 64-256 blocks of a few stages, and the gradient through the output layer
// (K = 4096 for 256 x 256 results) one chain of stages per block.  Hence wide
// loads, a stage in flight, and small tiles where 64 x 64 would leave CUs idle.
// Measured at batch 256, width 256, 4096 outputs (us per launch), against
// single-value loads in stages of 16 and bias sums by themselves: hidden layer
// 27.7 -> 5.3, output layer 31.5 -> 7.5, its weight and bias gradient 34.6 +
// 59.7 -> 13.9, the seven other 256-wide gradient products of a training step
// 844 + 4 x 56.7 -> 90 in all, 40 of them the one over K = 4096.
// Operand lanes: lane l carries A(l%16, 4(l/16)+q) and B(l%16, 4(l/16)+q),
// q = 0..3; result register q holds C(4(l/16)+q, l%16).
template <int EPI, typename TA, bool AK, typename TB, bool BK, int TILE, int KC, int AHEAD>
__global__ __launch_bounds__(256) void gemm_bf16(Operand<TA> A, Operand<TB> B, GemmArgs g) {
  constexpr int W = TILE / 32;  // 16 x 16 blocks per wave and direction
  __shared__ __align__(16) unsigned short As[2][TILE][KC + 8], Bs[2][TILE][KC + 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int tiles = (g.N + TILE - 1) / TILE * ((g.M + TILE - 1) / TILE);
  if ((int)blockIdx.x >= tiles) {  // the blocks after the product's sum the columns
    column_sums(g, blockIdx.x - tiles, tid);
    return;
  }
  const int nt = (g.N + TILE - 1) / TILE;
  const int m_base = (int)blockIdx.x / nt * TILE, n_base = (int)blockIdx.x % nt * TILE;
  const int wm = (wave >> 1) * (TILE / 2), wn = (wave & 1) * (TILE / 2);
  Stage<TA, AK, TILE, KC> sa[AHEAD];
  Stage<TB, BK, TILE, KC> sb[AHEAD];
  f32x4 acc[W][W];
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < AHEAD; ++d) {
    if (d * KC < g.K) {
      sa[d].fetch(A, m_base, d * KC, g.K, tid);
      sb[d].fetch(B, n_base, d * KC, g.K, tid);
    }
  }
  int buf = 0;
  for (int kd = 0; kd < g.K; kd += AHEAD * KC) {
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) {  // (d is a constant: the stages stay in registers)
      const int k0 = kd + d * KC;
      if (k0 >= g.K) break;
      sa[d].put(As[buf], tid);
      sb[d].put(Bs[buf], tid);
      if (k0 + AHEAD * KC < g.K) {
        sa[d].fetch(A, m_base, k0 + AHEAD * KC, g.K, tid);
        sb[d].fetch(B, n_base, k0 + AHEAD * KC, g.K, tid);
      }
      __syncthreads();  // (the other buffer is rewritten only after the next stage's barrier)
#pragma unroll
      for (int kk = 0; kk < KC; kk += 16) {
        if (k0 + kk < g.K) {
          bf16x4 a[W], b[W];
#pragma unroll
          for (int i = 0; i < W; ++i)
            a[i] = *reinterpret_cast<const bf16x4 *>(&As[buf][wm + 16 * i + (lane & 15)][kk + 4 * (lane >> 4)]);
#pragma unroll
          for (int j = 0; j < W; ++j)
            b[j] = *reinterpret_cast<const bf16x4 *>(&Bs[buf][wn + 16 * j + (lane & 15)][kk + 4 * (lane >> 4)]);
#pragma unroll
          for (int i = 0; i < W; ++i)
#pragma unroll
            for (int j = 0; j < W; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
        }
      }
      buf ^= 1;
    }
  }
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = m_base + wm + 16 * i + 4 * (lane >> 4) + q;
        const int n = n_base + wn + 16 * j + (lane & 15);
        if (m >= g.M || n >= g.N) continue;
        const long long o = (long long)m * g.ldc + n;
        const float v = acc[i][j][q];
        if constexpr (EPI == EPI_STORE) {
          g.cout[o] = v;
        } else if constexpr (EPI == EPI_BIAS) {
          g.cout[o] = v + g.bias[n];
        } else if constexpr (EPI == EPI_BIAS_GELU) {
          const float z = v + g.bias[n];
          if (g.zout) g.zout[o] = z;
          g.hout[o] = f2bf(gelu(z));
        } else {
          g.cout[o] = v * gelu_grad(g.zprev[o]);
        }
      }
}

// dY = 2 (Y - T) / (B * n_out); per-block partial sums of (Y - T)^2
__global__ void mse_grad(const float *__restrict__ Y, const float *__restrict__ T, float *__restrict__ dY,
                         float *__restrict__ partial, long long n, float scale) {
  __shared__ float red[256];
  float s = 0;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const float d = Y[i] - T[i];
    dY[i] = 2.0f * d * scale;
    s += d * d;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void adam_step(float *w, unsigned short *wbf, const float *gr, float *m, float *v, long long n, float lr,
                          float b1, float b2, float eps, float c1, float c2) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const float g = gr[i];
    const float mi = b1 * m[i] + (1 - b1) * g;
    const float vi = b2 * v[i] + (1 - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    if (wbf) wbf[i] = f2bf(wi);
  }
}

__global__ void to_bf16(const float *x, unsigned short *y, long long n) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) y[i] = f2bf(x[i]);
}

}  // namespace

// ---------------------------------------------------------------- host side

struct opo_mlp {
  int n_in = 0, width = 0, depth = 0, n_out = 0, max_batch = 0, device = 0;
  int nl = 0;                                // layers = depth + 1
  std::vector<int> din, dout;                // per layer
  std::vector<size_t> woff, boff;            // offsets into the flat parameter vector
  size_t nparams = 0;
  float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // FP32 master, grads, Adam moments
  unsigned short *wbf = nullptr;             // BF16 copy of the flat vector
  unsigned short *x_bf = nullptr;            // input batch (bf16)
  std::vector<float *> Z;                    // pre-activations per hidden layer (fp32)
  std::vector<unsigned short *> H;           // activations per hidden layer (bf16)
  float *Y = nullptr, *Tt = nullptr, *dA = nullptr, *dB = nullptr, *partial = nullptr, *xf = nullptr;
  long long step = 0;
  hipStream_t stream = nullptr;
  std::vector<void *> allocs;
  ~opo_mlp() {
    for (void *p : allocs) (void)hipFree(p);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

int malloc_m(opo_mlp *M, void **p, size_t bytes) {
  if (hipMalloc(p, bytes) != hipSuccess) return mfail(OPO_ERR_NOMEM, "mlp allocation");
  M->allocs.push_back(*p);
  return OPO_OK;
}

// 16-byte vectors along K, or four rows at a time
template <typename T> Operand<T> operand(const T *p, long long ld, int rows, bool kcont) {
  const size_t step = kcont ? 16 : 4 * sizeof(T);
  return {p, ld, rows, reinterpret_cast<uintptr_t>(p) % step == 0 && (size_t)ld * sizeof(T) % step == 0};
}

// Tiles of 64 where they fill the 256 CUs, else of 32 (four times the blocks:
// the 256 x 256 products of the hidden layers are 64 blocks then, not 16).
template <int EPI, bool AK, bool BK, typename TA, typename TB>
int gemm(opo_mlp *M, const TA *A, long long lda, const TB *B, long long ldb, const GemmArgs &g) {
  if (g.M <= 0 || g.N <= 0 || g.K <= 0) return mfail(OPO_ERR_INVALID, "empty gemm");
  const Operand<TA> a = operand(A, lda, g.M, AK);
  const Operand<TB> b = operand(B, ldb, g.N, BK);
  const int cols = g.col_in ? (g.col_cols + 255) / 256 : 0;
  auto tiles = [&](int t) { return (g.M + t - 1) / t * ((g.N + t - 1) / t); };
  if (tiles(64) >= 256)
    hipLaunchKernelGGL((gemm_bf16<EPI, TA, AK, TB, BK, 64, 64, 1>), dim3(tiles(64) + cols), dim3(256), 0, M->stream, a, b, g);
  else
    hipLaunchKernelGGL((gemm_bf16<EPI, TA, AK, TB, BK, 32, 128, 2>), dim3(tiles(32) + cols), dim3(256), 0, M->stream, a, b, g);
  MCHK(hipGetLastError());
  return OPO_OK;
}

// forward pass for B rows already in M->x_bf; store_z keeps pre-activations for backward
int forward(opo_mlp *M, int Bn, bool store_z) {
  const unsigned short *in = M->x_bf;
  for (int l = 0; l < M->nl; ++l) {
    GemmArgs g{};
    g.M = Bn; g.N = M->dout[l]; g.K = M->din[l];  // activations [B x din], W [dout x din]
    g.ldc = M->dout[l];
    g.bias = M->w + M->boff[l];
    const unsigned short *W = M->wbf + M->woff[l];
    if (l < M->nl - 1) {
      g.zout = store_z ? M->Z[l] : nullptr;
      g.hout = M->H[l];
      MRCHK((gemm<EPI_BIAS_GELU, true, true>(M, in, M->din[l], W, M->din[l], g)));
      in = M->H[l];
    } else {
      g.cout = M->Y;
      MRCHK((gemm<EPI_BIAS, true, true>(M, in, M->din[l], W, M->din[l], g)));
    }
  }
  return OPO_OK;
}

// gradients of the MSE loss for the batch in x_bf / Tt; returns the loss
int backward(opo_mlp *M, int Bn, float *loss) {
  const long long ny = (long long)Bn * M->n_out;
  const int nb = 256;
  hipLaunchKernelGGL(mse_grad, dim3(nb), dim3(256), 0, M->stream, M->Y, M->Tt, M->dA, M->partial, ny,
                     1.0f / (float)ny);
  MCHK(hipGetLastError());
  float *dZ = M->dA, *dNext = M->dB;
  for (int l = M->nl - 1; l >= 0; --l) {
    const unsigned short *Hin = l == 0 ? M->x_bf : M->H[l - 1];
    // dW_l = dZ^T (B x dout -> dout x B) * Hin (B x din), and db_l beside it
    GemmArgs gw{};
    gw.M = M->dout[l]; gw.N = M->din[l]; gw.K = Bn;
    gw.ldc = M->din[l];
    gw.cout = M->g + M->woff[l];
    gw.col_in = dZ; gw.col_out = M->g + M->boff[l];
    gw.col_rows = Bn; gw.col_cols = M->dout[l];
    MRCHK((gemm<EPI_STORE, false, false>(M, dZ, M->dout[l], Hin, M->din[l], gw)));
    if (l == 0) break;
    // dZ_{l-1} = (dZ * W_l) .* gelu'(Z_{l-1});  dZ [B x dout], W [dout x din]
    GemmArgs gh{};
    gh.M = Bn; gh.N = M->din[l]; gh.K = M->dout[l];
    gh.ldc = M->din[l];
    gh.zprev = M->Z[l - 1];
    gh.cout = dNext;
    MRCHK((gemm<EPI_GELU_GRAD, true, false>(M, dZ, M->dout[l], M->wbf + M->woff[l], M->din[l], gh)));
    std::swap(dZ, dNext);
  }
  std::vector<float> part(nb);
  MCHK(hipMemcpyAsync(part.data(), M->partial, nb * sizeof(float), hipMemcpyDeviceToHost, M->stream));
  MCHK(hipStreamSynchronize(M->stream));
  double s = 0;
  for (float p : part) s += p;
  if (loss) *loss = (float)(s / (double)ny);
  return OPO_OK;
}

int upload_batch(opo_mlp *M, const float *x, const float *t, int Bn) {
  if (Bn < 1 || Bn > M->max_batch) return mfail(OPO_ERR_INVALID, "batch size out of range");
  MCHK(hipMemcpyAsync(M->xf, x, (size_t)Bn * M->n_in * sizeof(float), hipMemcpyHostToDevice, M->stream));
  hipLaunchKernelGGL(to_bf16, dim3(64), dim3(256), 0, M->stream, M->xf, M->x_bf, (long long)Bn * M->n_in);
  MCHK(hipGetLastError());
  if (t) MCHK(hipMemcpyAsync(M->Tt, t, (size_t)Bn * M->n_out * sizeof(float), hipMemcpyHostToDevice, M->stream));
  return OPO_OK;
}

}  // namespace

extern "C" {

int opo_mlp_create(int n_in, int width, int depth, int n_out, int max_batch, uint64_t seed, int device,
                   opo_mlp **out) {
  if (!out || n_in < 1 || width < 1 || depth < 1 || n_out < 1 || max_batch < 1)
    return mfail(OPO_ERR_INVALID, "bad MLP shape");
  *out = nullptr;
  std::unique_ptr<opo_mlp> M(new opo_mlp());
  M->n_in = n_in; M->width = width; M->depth = depth; M->n_out = n_out; M->max_batch = max_batch;
  M->device = device;
  MCHK(hipSetDevice(device));
  MCHK(hipStreamCreateWithFlags(&M->stream, hipStreamNonBlocking));
  M->nl = depth + 1;
  for (int l = 0; l < M->nl; ++l) {
    M->din.push_back(l == 0 ? n_in : width);
    M->dout.push_back(l == M->nl - 1 ? n_out : width);
  }
  size_t off = 0;
  for (int l = 0; l < M->nl; ++l) {
    M->woff.push_back(off); off += (size_t)M->din[l] * M->dout[l];
    M->boff.push_back(off); off += (size_t)M->dout[l];
  }
  M->nparams = off;
  const size_t np = M->nparams;
  MRCHK(malloc_m(M.get(), (void **)&M->w, np * 4));
  MRCHK(malloc_m(M.get(), (void **)&M->g, np * 4));
  MRCHK(malloc_m(M.get(), (void **)&M->m, np * 4));
  MRCHK(malloc_m(M.get(), (void **)&M->v, np * 4));
  MRCHK(malloc_m(M.get(), (void **)&M->wbf, np * 2));
  MRCHK(malloc_m(M.get(), (void **)&M->xf, (size_t)max_batch * n_in * 4));
  MRCHK(malloc_m(M.get(), (void **)&M->x_bf, (size_t)max_batch * n_in * 2));
  for (int l = 0; l < depth; ++l) {
    float *z; unsigned short *h;
    MRCHK(malloc_m(M.get(), (void **)&z, (size_t)max_batch * width * 4));
    MRCHK(malloc_m(M.get(), (void **)&h, (size_t)max_batch * width * 2));
    M->Z.push_back(z); M->H.push_back(h);
  }
  const size_t big = (size_t)max_batch * std::max(n_out, width);
  MRCHK(malloc_m(M.get(), (void **)&M->Y, (size_t)max_batch * n_out * 4));
  MRCHK(malloc_m(M.get(), (void **)&M->Tt, (size_t)max_batch * n_out * 4));
  MRCHK(malloc_m(M.get(), (void **)&M->dA, big * 4));
  MRCHK(malloc_m(M.get(), (void **)&M->dB, big * 4));
  MRCHK(malloc_m(M.get(), (void **)&M->partial, 256 * 4));
  // He-style initialisation from a seeded generator; zero biases
  std::vector<float> h(np, 0.f);
  std::mt19937_64 rng(seed);
  for (int l = 0; l < M->nl; ++l) {
    std::normal_distribution<float> nd(0.f, std::sqrt(2.0f / (float)M->din[l]));
    for (size_t i = 0; i < (size_t)M->din[l] * M->dout[l]; ++i) h[M->woff[l] + i] = nd(rng);
  }
  MCHK(hipMemcpy(M->w, h.data(), np * 4, hipMemcpyHostToDevice));
  MCHK(hipMemset(M->m, 0, np * 4));
  MCHK(hipMemset(M->v, 0, np * 4));
  hipLaunchKernelGGL(to_bf16, dim3(256), dim3(256), 0, M->stream, M->w, M->wbf, (long long)np);
  MCHK(hipGetLastError());
  MCHK(hipStreamSynchronize(M->stream));
  *out = M.release();
  return OPO_OK;
}

int opo_mlp_param_count(opo_mlp *M, size_t *n) {
  if (!M || !n) return mfail(OPO_ERR_INVALID, "null");
  *n = M->nparams;
  return OPO_OK;
}

int opo_mlp_set_weights(opo_mlp *M, const float *w, size_t n) {
  if (!M || !w || n != M->nparams) return mfail(OPO_ERR_INVALID, "weight count mismatch");
  MCHK(hipSetDevice(M->device));
  MCHK(hipMemcpyAsync(M->w, w, n * 4, hipMemcpyHostToDevice, M->stream));
  hipLaunchKernelGGL(to_bf16, dim3(256), dim3(256), 0, M->stream, M->w, M->wbf, (long long)n);
  MCHK(hipGetLastError());
  MCHK(hipMemsetAsync(M->m, 0, n * 4, M->stream));
  MCHK(hipMemsetAsync(M->v, 0, n * 4, M->stream));
  M->step = 0;
  MCHK(hipStreamSynchronize(M->stream));
  return OPO_OK;
}

int opo_mlp_get_weights(opo_mlp *M, float *w, size_t n) {
  if (!M || !w || n != M->nparams) return mfail(OPO_ERR_INVALID, "weight count mismatch");
  MCHK(hipMemcpy(w, M->w, n * 4, hipMemcpyDeviceToHost));
  return OPO_OK;
}

int opo_mlp_forward(opo_mlp *M, const float *x, int Bn, float *y) {
  if (!M || !x || !y) return mfail(OPO_ERR_INVALID, "null");
  MCHK(hipSetDevice(M->device));
  MRCHK(upload_batch(M, x, nullptr, Bn));
  MRCHK(forward(M, Bn, false));
  MCHK(hipMemcpyAsync(y, M->Y, (size_t)Bn * M->n_out * 4, hipMemcpyDeviceToHost, M->stream));
  MCHK(hipStreamSynchronize(M->stream));
  return OPO_OK;
}

int opo_mlp_gradients(opo_mlp *M, const float *x, const float *t, int Bn, float *grad, float *loss) {
  if (!M || !x || !t) return mfail(OPO_ERR_INVALID, "null");
  MCHK(hipSetDevice(M->device));
  MRCHK(upload_batch(M, x, t, Bn));
  MRCHK(forward(M, Bn, true));
  MRCHK(backward(M, Bn, loss));
  if (grad) MCHK(hipMemcpy(grad, M->g, M->nparams * 4, hipMemcpyDeviceToHost));
  return OPO_OK;
}

int opo_mlp_train_step(opo_mlp *M, const float *x, const float *t, int Bn, float lr, float *loss) {
  if (!M || !x || !t) return mfail(OPO_ERR_INVALID, "null");
  MCHK(hipSetDevice(M->device));
  MRCHK(upload_batch(M, x, t, Bn));
  MRCHK(forward(M, Bn, true));
  MRCHK(backward(M, Bn, loss));
  M->step += 1;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - std::pow(b1, (float)M->step), c2 = 1.0f - std::pow(b2, (float)M->step);
  hipLaunchKernelGGL(adam_step, dim3(512), dim3(256), 0, M->stream, M->w, M->wbf, M->g, M->m, M->v,
                     (long long)M->nparams, lr, b1, b2, 1e-8f, c1, c2);
  MCHK(hipGetLastError());
  MCHK(hipStreamSynchronize(M->stream));
  return OPO_OK;
}

int opo_mlp_destroy(opo_mlp *M) {
  delete M;
  return OPO_OK;
}

}  // extern "C"
