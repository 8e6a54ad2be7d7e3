// tsm_mlp.hip -- MLP surrogate of the Monte Carlo quantities of interest:
// BF16 weights and activations on MFMA (v_mfma_f32_32x32x16_bf16) with FP32
// accumulation, FP32 master weights, Adam.  No counterpart in the reference.
//
// Layers: z_l = x_l W_l^T + b_l (W_l: n_out x n_in, row-major), x_{l+1} =
// GELU(z_l) (exact, erf form) for hidden layers, y = z_last.  Activations are
// row-major [batch x features] in bf16; pre-activations z_l are kept in FP32
// for the backward pass.  Backward (loss = mean over batch and outputs of
// (y - t)^2):
//   dy = 2 (y - t) / (B n_out)            (fp32 -> bf16)
//   dW_l = dz_l^T x_l,  db_l = column sums of dz_l   (fp32)
//   dx_l = dz_l W_l,    dz_{l-1} = dx_l * GELU'(z_{l-1})   (-> bf16)
// Networks of layers up to FUSED_MAX wide (the surrogates are 64 to 256 wide) run
// in three kernels: k_rows (k_rows_reg up to 256 wide) takes eight rows of a minibatch through every layer and
// back, k_update forms each 32 x 32 tile of the weight gradients and applies Adam
// to it, k_infer takes rows through the layers only.  Wider ones take one launch
// of the tiled GEMM per product, the operands' transposes absorbed by the LDS
// staging.  Both form every sum in the same order (k ascending, 16 a product), so
// they give the same bits.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/tsm.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16;

__host__ __device__ inline u16 f2bf(float f) {  // round to nearest even
  uint32_t u;
  std::memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u16)((u >> 16) | 0x40);  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (u16)(u >> 16);
}
__host__ __device__ inline float bf2f(u16 h) {
  uint32_t u = (uint32_t)h << 16;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}

__device__ inline float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ inline float gelu_d(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) +
         z * 0.39894228040143268f * expf(-0.5f * z * z);
}

enum { EPI_F32 = 0, EPI_BIAS_GELU = 1, EPI_GELU_BWD = 2, EPI_BIAS_F32 = 3 };

constexpr int BM = 64, BN = 64, BK = 32, LDK = BK + 8;  // LDS rows padded by 16 bytes

// C[M x N] = A[M x K] * B[K x N].  AK: A stored M x K with k contiguous (else
// K x M with m contiguous); BK_: B stored N x K with k contiguous (else K x N
// with n contiguous).  256 threads = 4 waves, each wave one 32 x 32 MFMA tile
// of the 64 x 64 block tile.
template <bool AK, bool BKM, int EPI>
__global__ __launch_bounds__(256) void k_gemm(int M, int N, int K, const u16* __restrict__ A,
                                              int lda, const u16* __restrict__ B, int ldb,
                                              float* __restrict__ Cf, u16* __restrict__ Cb, int ldc,
                                              const float* __restrict__ bias,
                                              const float* __restrict__ Z, float* __restrict__ Zout) {
  __shared__ __attribute__((aligned(16))) u16 As[BM * LDK];
  __shared__ __attribute__((aligned(16))) u16 Bs[BN * LDK];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;

  for (int k0 = 0; k0 < K; k0 += BK) {
    // ---- stage A (64 x 32) and B (64 x 32) in LDS, k contiguous per row ----
    if (AK) {
      const int row = tid >> 2, ks = (tid & 3) * 8, gm = m0 + row, gk = k0 + ks;
      u16 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = (gm < M && gk + j < K) ? A[(size_t)gm * lda + gk + j] : (u16)0;
#pragma unroll
      for (int j = 0; j < 8; ++j) As[row * LDK + ks + j] = v[j];
    } else {
      const int kk = tid >> 3, ms = (tid & 7) * 8, gk = k0 + kk;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int gm = m0 + ms + j;
        As[(ms + j) * LDK + kk] = (gm < M && gk < K) ? A[(size_t)gk * lda + gm] : (u16)0;
      }
    }
    if (BKM) {
      const int row = tid >> 2, ks = (tid & 3) * 8, gn = n0 + row, gk = k0 + ks;
      u16 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = (gn < N && gk + j < K) ? B[(size_t)gn * ldb + gk + j] : (u16)0;
#pragma unroll
      for (int j = 0; j < 8; ++j) Bs[row * LDK + ks + j] = v[j];
    } else {
      const int kk = tid >> 3, ns = (tid & 7) * 8, gk = k0 + kk;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int gn = n0 + ns + j;
        Bs[(ns + j) * LDK + kk] = (gn < N && gk < K) ? B[(size_t)gk * ldb + gn] : (u16)0;
      }
    }
    __syncthreads();
    // ---- two MFMA 32x32x16 per k tile; lanes 0-31 take k 0-7, 32-63 k 8-15
    //      of each 16-slice (the same map for A and B, so the k order is moot)
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      const int ko = kk + (lane >> 5) * 8;
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(&As[(wm + (lane & 31)) * LDK + ko]);
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(&Bs[(wn + (lane & 31)) * LDK + ko]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    __syncthreads();
  }
  // ---- epilogue: acc[i] is C[row][col] with col = lane % 32 and
  //      row = 8 (i / 4) + 4 (lane / 32) + i % 4 within the wave tile
  const int gn = n0 + wn + (lane & 31);
  if (gn >= N) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int gm = m0 + wm + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
    if (gm >= M) continue;
    const size_t o = (size_t)gm * ldc + gn;
    float c = acc[i];
    if (EPI == EPI_F32) {
      Cf[o] = c;
    } else if (EPI == EPI_BIAS_F32) {
      Cf[o] = c + bias[gn];
    } else if (EPI == EPI_BIAS_GELU) {
      c += bias[gn];
      if (Zout) Zout[o] = c;
      Cb[o] = f2bf(gelu(c));
    } else {  // EPI_GELU_BWD
      Cb[o] = f2bf(c * gelu_d(Z[o]));
    }
  }
}

// Column sums of a [rows x cols] bf16 or fp32 matrix, fp32, fixed order.
__global__ void k_colsum_bf16(int rows, int cols, const u16* X, float* out) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= cols) return;
  float s = 0.0f;
  for (int r = 0; r < rows; ++r) s += bf2f(X[(size_t)r * cols + c]);
  out[c] = s;
}

// dy = 2 (y - t) / (B n), loss partials per block (sum of squares)
__global__ __launch_bounds__(256) void k_mse(int n, const float* y, const float* t, float scale,
                                             u16* dy, float* partial) {
  __shared__ float red[4];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  float e2 = 0.0f;
  if (i < n) {
    const float d = y[i] - t[i];
    e2 = d * d;
    dy[i] = f2bf(2.0f * d * scale);
  }
  for (int o = 32; o > 0; o >>= 1) e2 += __shfl_down(e2, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = e2;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// Adam on fp32 master weights; refreshes the bf16 copy.
__global__ void k_adam(int n, float* w, const float* g, float* m, float* v, u16* wb, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (wb) wb[i] = f2bf(wi);
}

__global__ void k_to_bf16(int n, const float* x, u16* y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

// rows of a [rows x cols] fp32 matrix picked by idx -> bf16 (inputs) or fp32 (targets)
__global__ void k_gather_rows(int rows, int cols, const int* idx, const float* src, u16* db,
                              float* df) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * cols) return;
  const int r = i / cols, c = i % cols;
  const float x = src[(size_t)idx[r] * cols + c];
  if (db) db[i] = f2bf(x);
  if (df) df[i] = x;
}

// ---------------------------------------------------------------------------
// fused kernels
// ---------------------------------------------------------------------------
constexpr int FUSED_MAX = 512, MAXL = 16, RT = 32;
inline int up(int n, int m) { return (n + m - 1) / m * m; }

// Weights twice in bf16, zero-padded: Wp[l] is up(n_out, 32) x up(n_in, 16) (the
// forward operand), Wt[l] its transpose, up(n_in, 32) x up(n_out, 16) (the
// backward one), both in the order the MFMA operand reads them (w_at): a wave's
// load of a 32 x 16 slice is one contiguous KB instead of 32 pieces of 32 bytes.
// Activations x_l and dz_l of a minibatch are kept transposed (XT, DT: feature
// x ldr rows, zero past the last row), which is how the weight gradients read
// them and how the MFMA result falls out (four rows per lane at a time).
struct Net {
  int L, ldr, lda;  // layers, row stride of XT/DT, LDS row stride
  int w[MAXL + 1];
  u16 *Wp[MAXL], *Wt[MAXL];
  float *P, *G, *Mo, *Vo;          // flat parameters, gradient, Adam moments
  int woff[MAXL], boff[MAXL];
  u16 *XT[MAXL], *DT[MAXL];
  float* Z[MAXL];
  float *Y, *T;
};
__host__ __device__ inline int upd(int n, int m) { return (n + m - 1) / m * m; }
// element (n, k) of a weight operand of padded depth Kp: slices of 32 n x 16 k,
// in a slice lane (k % 16 / 8) * 32 + n % 32 holds eight k one after another
__device__ __forceinline__ int w_at(int n, int k, int Kp) {
  return (n >> 5) * 32 * Kp + (k >> 4) * 512 + ((k >> 3) & 1) * 256 + (n & 31) * 8 + (k & 7);
}

// One layer's product for NT row tiles of 32: C (32 x 32 per tile, columns n0 ..)
// from LDS activations A (row stride lda) and weights W (padded depth Kp).
template <int NT>
__device__ __forceinline__ void tile_product(const u16* A, int lda, const u16* W, int Kp, int n0,
                                             f32x16* acc) {
  const int lane = threadIdx.x & 63, c = lane & 31, ko = (lane >> 5) * 8;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;
  const u16* wr = W + n0 * Kp + lane * 8;
  const u16* ar = A + c * lda + ko;
  int k0 = 0;
  for (; k0 + 128 <= Kp; k0 += 128) {  // eight slices in flight
    bf16x8 b[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) b[u] = *reinterpret_cast<const bf16x8*>(wr + 32 * (k0 + 16 * u));
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(ar + t * RT * lda + k0 + 16 * u);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[u], acc[t], 0, 0, 0);
      }
  }
  for (; k0 < Kp; k0 += 16) {
    const bf16x8 b = *reinterpret_cast<const bf16x8*>(wr + 32 * k0);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(ar + t * RT * lda + k0);
      acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[t], 0, 0, 0);
    }
  }
}
// row of result element i within a tile
__device__ __forceinline__ int c_row(int i) { return 8 * (i >> 2) + 4 * ((threadIdx.x & 63) >> 5) + (i & 3); }

// RB rows of a minibatch (rows idx[r], or r itself) forward, dy = 2 (y - t) / n,
// and back to dz_0; the transposed activations and dz of every layer go to XT/DT.
// Bound by the latency of its 2 L - 1 dependent products: eight waves, one or more
// 32-column tiles each.  Eight rows a block, though the MFMA tile has 32: the
// epilogues (an error function and an exponential per element) are most of the
// work, rows 0-7 of a tile are elements 0-3 of every lane, and a minibatch of 64
// then spreads over eight CUs instead of two.
constexpr int RB = 8;

// The product of a wave's tile with the weight slices in w (up to 16 of 16 deep),
// each slice's registers taking the next product's as soon as it is used.
struct WReg { bf16x8 b[16]; };
__device__ __forceinline__ void reg_load(WReg& w, const u16* W, int Kp) {
  const u16* p = W + (threadIdx.x & 63) * 8;
  const int last = (Kp >> 4) - 1;
#pragma unroll
  for (int u = 0; u < 16; ++u) w.b[u] = *reinterpret_cast<const bf16x8*>(p + 512 * min(u, last));
}
__device__ __forceinline__ f32x16 reg_product(const u16* A, int lda, WReg& w, int Kp, const u16* Wn,
                                              int Kpn) {
  const int lane = threadIdx.x & 63, lastn = (Kpn >> 4) - 1;
  const u16* ar = A + (lane & 31) * lda + (lane >> 5) * 8;
  const u16* p = Wn + lane * 8;
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    if (16 * u < Kp) {
      const bf16x8 x = *reinterpret_cast<const bf16x8*>(ar + 16 * u);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, w.b[u], acc, 0, 0, 0);
    }
    w.b[u] = *reinterpret_cast<const bf16x8*>(p + 512 * min(u, lastn));
  }
  return acc;
}

// For nets with no layer wider than 256: one tile per wave (waves beyond a layer's
// tiles repeat the last one, with the same results), its weights in registers.
// Nothing but the loss's row depends on a branch and pre-activations stay in LDS, so
// that a layer waits for its own weights only, which were asked for a product ago.
// At 64 rows of 6-256-256-256-66: 32 rows a block 56 us; eight, with the next
// weights asked for after a product, 36; weights in operand order 25; asked for
// before it 22; as now 18.
__global__ __launch_bounds__(512) void k_rows_reg(Net a, int nb, const int* idx, const float* Xin,
                                                  const float* Tin, float scale) {
  extern __shared__ __attribute__((aligned(16))) u16 sm[];
  u16 *cur = sm, *nxt = sm + RT * a.lda;
  float4* zs = reinterpret_cast<float4*>(sm + 2 * RT * a.lda);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r0 = blockIdx.x * RB, L = a.L;
  const int row0 = 4 * (lane >> 5);  // this lane's rows: row0 .. row0 + 3
  auto tile = [&](int n) { return min(32 * wave, upd(n, 32) - 32); };  // of a layer n wide
  auto fwd = [&](int l) { return a.Wp[l] + tile(a.w[l + 1]) * upd(a.w[l], 16); };
  auto bwd = [&](int l) { return a.Wt[l] + tile(a.w[l]) * upd(a.w[l + 1], 16); };
  auto bias = [&](int l) {
    return a.P[a.boff[l] + min(tile(a.w[l + 1]) + (lane & 31), a.w[l + 1] - 1)];
  };
  WReg w;
  reg_load(w, fwd(0), upd(a.w[0], 16));
  float bn = bias(0);
  const int no = a.w[L], ny = tile(no) + (lane & 31);
  float t[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = min(r0 + row0 + u, nb - 1);
    t[u] = Tin[(size_t)(idx ? idx[r] : r) * no + min(ny, no - 1)];
  }
  {
    const int K = a.w[0], Kp = upd(K, 16);
    for (int i = tid; i < RB * Kp; i += blockDim.x) {
      const int k = i / RB, r = i % RB;  // rows fastest: XT is written in order
      const bool in = k < K && r0 + r < nb;
      const u16 v = in ? f2bf(Xin[(size_t)(idx ? idx[r0 + r] : r0 + r) * K + k]) : (u16)0;
      cur[r * a.lda + k] = v;
      if (k < K) a.XT[0][(size_t)k * a.ldr + r0 + r] = v;
    }
  }
  __syncthreads();
  // four rows of column n to LDS and to the transposed operand
  auto put = [&](int n, const float* v, u16* out) {
    ushort4 q;
    u16* qv = reinterpret_cast<u16*>(&q);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      qv[u] = f2bf(v[u]);
      nxt[(row0 + u) * a.lda + n] = qv[u];
    }
    *reinterpret_cast<ushort4*>(out + (size_t)n * a.ldr + r0 + row0) = q;
  };
  float v[4];
  for (int l = 0; l + 1 < L; ++l) {
    const int n = tile(a.w[l + 1]) + (lane & 31);
    const f32x16 acc = reg_product(cur, a.lda, w, upd(a.w[l], 16), fwd(l + 1), upd(a.w[l + 1], 16));
    const float b0 = bn;
    bn = bias(l + 1);
    float4 z;
    float* zp = reinterpret_cast<float*>(&z);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      zp[u] = acc[u] + b0;
      const float g = gelu(zp[u]);
      v[u] = n < a.w[l + 1] && r0 + row0 + u < nb ? g : 0.0f;
    }
    zs[l * 512 + tid] = z;
    put(n, v, a.XT[l + 1]);
    __syncthreads();
    u16* x = cur; cur = nxt; nxt = x;
  }
  {
    const int l = L - 1;
    const f32x16 acc = reg_product(cur, a.lda, w, upd(a.w[l], 16), bwd(l), upd(no, 16));
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = r0 + row0 + u;
      const bool in = ny < no && r < nb;
      const float c = acc[u] + bn;
      if (in) a.Y[(size_t)r * no + ny] = c;
      v[u] = in ? 2.0f * (c - t[u]) * scale : 0.0f;
    }
    put(ny, v, a.DT[l]);
    __syncthreads();
    u16* x = cur; cur = nxt; nxt = x;
  }
  // dz_{l-1} = (dz_l W_l) * GELU'(z_{l-1}); z was kept by this very lane
  for (int l = L - 1; l > 0; --l) {
    const int k = tile(a.w[l]) + (lane & 31), ln = max(l - 1, 1);
    const f32x16 acc = reg_product(cur, a.lda, w, upd(a.w[l + 1], 16), bwd(ln), upd(a.w[ln + 1], 16));
    const float4 z = zs[(l - 1) * 512 + tid];
    const float* zp = reinterpret_cast<const float*>(&z);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float g = acc[u] * gelu_d(zp[u]);
      v[u] = k < a.w[l] && r0 + row0 + u < nb ? g : 0.0f;
    }
    put(k, v, a.DT[l - 1]);
    __syncthreads();
    u16* x = cur; cur = nxt; nxt = x;
  }
}

// ... and for wider ones, several tiles per wave and layer, pre-activations in Z
__global__ __launch_bounds__(512) void k_rows(Net a, int nb, const int* idx, const float* Xin,
                                              const float* Tin, float scale) {
  extern __shared__ __attribute__((aligned(16))) u16 sm[];
  u16 *cur = sm, *nxt = sm + RT * a.lda;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  const int r0 = blockIdx.x * RB, L = a.L;
  {
    const int K = a.w[0], Kp = upd(K, 16);
    for (int i = tid; i < RB * Kp; i += blockDim.x) {
      const int k = i / RB, r = i % RB;  // rows fastest: XT is written in order
      const bool in = k < K && r0 + r < nb;
      const u16 v = in ? f2bf(Xin[(size_t)(idx ? idx[r0 + r] : r0 + r) * K + k]) : (u16)0;
      cur[r * a.lda + k] = v;
      if (k < K) a.XT[0][(size_t)k * a.ldr + r0 + r] = v;
    }
  }
  const int row0 = 4 * (lane >> 5);  // this lane's rows: row0 .. row0 + 3
  int rows[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) rows[u] = (idx && r0 + row0 + u < nb) ? idx[r0 + row0 + u] : r0 + row0 + u;
  __syncthreads();
  f32x16 acc[1];
  for (int l = 0; l < L; ++l) {
    const int K = a.w[l], N = a.w[l + 1], Kp = upd(K, 16), Np = upd(N, 32);
    const bool last = l + 1 == L;
    const float* bias = a.P + a.boff[l];
    for (int n0 = 32 * wave; n0 < Np; n0 += 32 * nw) {
      const int n = n0 + (lane & 31);
      const bool col = n < N;
      const float bn = col ? bias[n] : 0.0f;
      float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (last && col)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (r0 + row0 + u < nb) t[u] = Tin[(size_t)rows[u] * N + n];
      tile_product<1>(cur, a.lda, a.Wp[l], Kp, n0, acc);
      ushort4 q;
      u16* qv = reinterpret_cast<u16*>(&q);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row = row0 + u, r = r0 + row;
        const bool in = col && r < nb;
        const float c = acc[0][u] + bn;
        u16 v = 0;
        if (in) {
          if (last) {
            a.Y[(size_t)r * N + n] = c;
            v = f2bf(2.0f * (c - t[u]) * scale);
          } else {
            a.Z[l][(size_t)r * N + n] = c;
            v = f2bf(gelu(c));
          }
        }
        qv[u] = v;
        nxt[row * a.lda + n] = v;
      }
      if (col) *reinterpret_cast<ushort4*>((last ? a.DT[l] : a.XT[l + 1]) + (size_t)n * a.ldr + r0 + row0) = q;
    }
    __syncthreads();
    u16* x = cur; cur = nxt; nxt = x;
  }
  // dz_{l-1} = (dz_l W_l) * GELU'(z_{l-1}); z was stored by this very lane
  for (int l = L - 1; l > 0; --l) {
    const int K = a.w[l], N = a.w[l + 1], Np = upd(N, 16), Kp = upd(K, 32);
    for (int k0 = 32 * wave; k0 < Kp; k0 += 32 * nw) {
      const int k = k0 + (lane & 31);
      const bool col = k < K;
      float z[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int r = r0 + row0 + u;
        z[u] = col && r < nb ? a.Z[l - 1][(size_t)r * K + k] : 0.0f;
      }
      tile_product<1>(cur, a.lda, a.Wt[l], Np, k0, acc);
      ushort4 q;
      u16* qv = reinterpret_cast<u16*>(&q);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const u16 v = col && r0 + row0 + u < nb ? f2bf(acc[0][u] * gelu_d(z[u])) : (u16)0;
        qv[u] = v;
        nxt[(row0 + u) * a.lda + k] = v;
      }
      if (col) *reinterpret_cast<ushort4*>(a.DT[l - 1] + (size_t)k * a.ldr + r0 + row0) = q;
    }
    __syncthreads();
    u16* x = cur; cur = nxt; nxt = x;
  }
}

// Adam on one parameter, as k_adam
struct Adam { float lr, b1, b2, eps, c1, c2; };
__device__ __forceinline__ float adam_step(const Adam& h, float gi, float p, float* m, float* v) {
  const float mi = h.b1 * *m + (1.0f - h.b1) * gi;
  const float vi = h.b2 * *v + (1.0f - h.b2) * gi * gi;
  *m = mi;
  *v = vi;
  return p - h.lr * (mi / h.c1) / (sqrtf(vi / h.c2) + h.eps);
}
// One job per wave: a 32 x 32 tile of a layer's weight gradient (MFMA over the
// rows), 64 bias gradients (sums in row order), or one 256-element part of the
// loss (the tree of k_mse).  TRAIN applies Adam at once and refreshes the bf16
// weights; else the gradient goes to G.  Bound by the latency of one pass over
// activations and moments (150 k parameters, 3.6 MB, 0.7 us at the copy rate):
// 13.9 us with each parameter's moments read in turn, 11.7 with all ahead.
template <bool TRAIN>
__global__ __launch_bounds__(256) void k_update(Net a, int nb, const int4* jobs, int n_jobs,
                                                const int* idx, const float* Tin, float* part, Adam h) {
  const int lane = threadIdx.x & 63;
  const int job = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int no = a.w[a.L], n_el = nb * no;
  if (job >= n_jobs) {
    const int b = job - n_jobs;
    if (256 * b >= n_el) return;
    float red[4];
    for (int w = 0; w < 4; ++w) {
      const int i = 256 * b + 64 * w + lane;
      float e2 = 0.0f;
      if (i < n_el) {
        const int r = i / no, c = i % no;
        const float d = a.Y[i] - Tin[(size_t)(idx ? idx[r] : r) * no + c];
        e2 = d * d;
      }
      for (int o = 32; o > 0; o >>= 1) e2 += __shfl_down(e2, o, 64);
      red[w] = e2;
    }
    if (lane == 0) part[b] = red[0] + red[1] + red[2] + red[3];
    return;
  }
  const int4 J = jobs[job];  // kind, layer, first output, first input
  const int l = J.y, K = a.w[l], N = a.w[l + 1];
  if (J.x == 1) {
    const int n = J.z + lane;
    if (n >= N) return;
    const u16* d = a.DT[l] + (size_t)n * a.ldr;
    float s = 0.0f;
    int r = 0;
    for (; r + 8 <= nb; r += 8) {
      u16 q[8];
      *reinterpret_cast<uint4*>(q) = *reinterpret_cast<const uint4*>(d + r);
#pragma unroll
      for (int u = 0; u < 8; ++u) s += bf2f(q[u]);
    }
    for (; r < nb; ++r) s += bf2f(d[r]);
    const int q = a.boff[l] + n;
    if (TRAIN) a.P[q] = adam_step(h, s, a.P[q], &a.Mo[q], &a.Vo[q]);
    else a.G[q] = s;
    return;
  }
  const int c = lane & 31, ko = (lane >> 5) * 8;
  const int nr = min(J.z + c, N - 1), kr = min(J.w + c, K - 1);  // rows past the layer: any, not stored
  const u16 *dr = a.DT[l] + (size_t)nr * a.ldr + ko, *xr = a.XT[l] + (size_t)kr * a.ldr + ko;
  const int k = J.w + c, Kp = upd(K, 16), Np = upd(N, 16);
  const bool in = k < K;
  // the moments and weights are asked for before the product: 48 loads in flight
  // instead of 16 waits for three
  float p[16], mo[16], vo[16];
  if (TRAIN) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int n = J.z + c_row(i), q = a.woff[l] + n * K + k;
      const bool ok = in && n < N;
      p[i] = ok ? a.P[q] : 0.0f;
      mo[i] = ok ? a.Mo[q] : 0.0f;
      vo[i] = ok ? a.Vo[q] : 0.0f;
    }
  }
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  for (int k0 = 0; k0 < nb; k0 += 16) {
    const bf16x8 A = *reinterpret_cast<const bf16x8*>(dr + k0);
    const bf16x8 B = *reinterpret_cast<const bf16x8*>(xr + k0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, B, acc, 0, 0, 0);
  }
  if (!in) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int n = J.z + c_row(i), q = a.woff[l] + n * K + k;
    if (n >= N) continue;
    if (TRAIN) {
      const float w = adam_step(h, acc[i], p[i], &mo[i], &vo[i]);
      a.Mo[q] = mo[i];
      a.Vo[q] = vo[i];
      a.P[q] = w;
      const u16 wb = f2bf(w);
      a.Wp[l][w_at(n, k, Kp)] = wb;
      a.Wt[l][w_at(k, n, Np)] = wb;
    } else {
      a.G[q] = acc[i];
    }
  }
}

// bf16 copies of the weights of layer l
__global__ void k_pack_weights(Net a, int l) {
  const int K = a.w[l], N = a.w[l + 1];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N * K) return;
  const int n = i / K, k = i % K;
  const u16 v = f2bf(a.P[a.woff[l] + i]);
  a.Wp[l][w_at(n, k, upd(K, 16))] = v;
  a.Wt[l][w_at(k, n, upd(N, 16))] = v;
}

// NT x 32 rows through the layers.  AFFINE: inputs (u - mu_x) / sd_x and outputs
// y sd_y + mu_y in FP64 (io: mu_x, sd_x, mu_y, sd_y one after another), else FP32
// rows in and out.  Two row tiles per wave share each weight load; at 65,536 rows
// the weights are read 1,024 times from L2 (0.3 GB) beside 20 GFLOP.
template <int NT, bool AFFINE>
__global__ __launch_bounds__(512) void k_infer(Net a, long rows, const void* in, const double* io,
                                               void* out) {
  extern __shared__ __attribute__((aligned(16))) u16 sm[];
  u16 *cur = sm, *nxt = sm + NT * RT * a.lda;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  const long r0 = (long)blockIdx.x * NT * RT;
  const int L = a.L, ni = a.w[0], no = a.w[L];
  {
    const int Kp = upd(ni, 16);
    for (int i = tid; i < NT * RT * Kp; i += blockDim.x) {
      const int r = i / Kp, k = i % Kp;
      u16 v = 0;
      if (k < ni && r0 + r < rows) {
        const size_t o = (size_t)(r0 + r) * ni + k;
        const float x = AFFINE ? (float)((static_cast<const double*>(in)[o] - io[k]) / io[ni + k])
                               : static_cast<const float*>(in)[o];
        v = f2bf(x);
      }
      cur[r * a.lda + k] = v;
    }
  }
  __syncthreads();
  f32x16 acc[NT];
  for (int l = 0; l < L; ++l) {
    const int N = a.w[l + 1], Kp = upd(a.w[l], 16), Np = upd(N, 32);
    const bool last = l + 1 == L;
    const float* bias = a.P + a.boff[l];
    for (int n0 = 32 * wave; n0 < Np; n0 += 32 * nw) {
      tile_product<NT>(cur, a.lda, a.Wp[l], Kp, n0, acc);
      const int n = n0 + (lane & 31);
      const bool col = n < N;
      const float bn = col ? bias[n] : 0.0f;
      const double sd = AFFINE && last && col ? io[2 * ni + no + n] : 1.0;
      const double mu = AFFINE && last && col ? io[2 * ni + n] : 0.0;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int row = t * RT + c_row(i);
          const float c = acc[t][i] + bn;
          if (!last) {
            nxt[row * a.lda + n] = col ? f2bf(gelu(c)) : (u16)0;
          } else if (col && r0 + row < rows) {
            const size_t o = (size_t)(r0 + row) * N + n;
            if (AFFINE) static_cast<double*>(out)[o] = (double)c * sd + mu;
            else static_cast<float*>(out)[o] = c;
          }
        }
    }
    __syncthreads();
    u16* x = cur; cur = nxt; nxt = x;
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct tsm_mlp {
  int L = 0, maxb = 0;
  std::vector<int> w;                 // widths, L + 1
  std::vector<size_t> woff, boff;     // offsets of W_l, b_l in the flat parameter vector
  size_t np = 0;
  bool fused = false;                 // no layer wider than FUSED_MAX
  float *P = nullptr, *G = nullptr, *Mo = nullptr, *Vo = nullptr;  // fp32 params, grads, Adam
  u16* Pb = nullptr;                  // bf16 copy of the parameters (not fused)
  std::vector<u16*> X;                // activations x_0..x_{L-1} (bf16), maxb x w_l (not fused)
  std::vector<float*> Z;              // pre-activations z_0..z_{L-1} (fp32)
  u16 *dA = nullptr, *dB = nullptr;   // backward ping-pong, maxb x max width (bf16; not fused)
  float *Y = nullptr, *T = nullptr, *part = nullptr;
  Net net{};                          // fused
  int4* jobs = nullptr;
  int n_jobs = 0;
  float *Xin = nullptr, *Tin = nullptr;  // staged training set
  int* idx = nullptr;
  size_t nin_cap = 0;
  float* parts = nullptr;             // loss parts of every minibatch of an epoch (fused)
  size_t parts_cap = 0;
  char* io = nullptr;                 // rows in and out of an evaluation (fused), INFER_BYTES at most
  size_t io_cap = 0;
  long adam_t = 0;
  hipStream_t st = nullptr;
  std::string err;
  std::vector<void*> allocs;
  template <class T>
  hipError_t al(T** p, size_t n) {
    hipError_t e = hipMalloc((void**)p, n * sizeof(T) + 16);
    if (e == hipSuccess) allocs.push_back((void*)*p);
    return e;
  }
  // replaces a buffer by a larger one once nothing on the stream uses it
  template <class T>
  hipError_t grow(T** p, size_t* cap, size_t n) {
    if (n <= *cap) return hipSuccess;
    hipError_t e = hipStreamSynchronize(st);
    if (e != hipSuccess) return e;
    if (*p) {
      allocs.erase(std::remove(allocs.begin(), allocs.end(), (void*)*p), allocs.end());
      (void)hipFree(*p);
      *p = nullptr;
      *cap = 0;
    }
    e = al(p, n);
    if (e == hipSuccess) *cap = n;
    return e;
  }
  ~tsm_mlp() {
    for (void* p : allocs) (void)hipFree(p);
    if (st) (void)hipStreamDestroy(st);
  }
};

namespace {
thread_local std::string g_mlp_err;
int mfail(int code, const std::string& m) {
  g_mlp_err = m;
  return code;
}
#define MLP_TRY(x)                                                     \
  do {                                                                 \
    hipError_t _e = (x);                                               \
    if (_e != hipSuccess) return mfail(TSM_E_HIP, hipGetErrorString(_e)); \
  } while (0)

template <bool AK, bool BKM, int EPI>
void gemm(hipStream_t st, int M, int N, int K, const u16* A, int lda, const u16* B, int ldb,
          float* Cf, u16* Cb, int ldc, const float* bias, const float* Z, float* Zout) {
  dim3 grid((M + BM - 1) / BM, (N + BN - 1) / BN);
  hipLaunchKernelGGL((k_gemm<AK, BKM, EPI>), grid, dim3(256), 0, st, M, N, K, A, lda, B, ldb, Cf,
                     Cb, ldc, bias, Z, Zout);
}

// forward of nb rows already in m->X[0]; output fp32 in m->Y (nb x w[L])
void forward(tsm_mlp* m, int nb, bool keep_z) {
  for (int l = 0; l < m->L; ++l) {
    const int K = m->w[l], N = m->w[l + 1];
    const u16* W = m->Pb + m->woff[l];
    const float* b = m->P + m->boff[l];
    if (l + 1 < m->L)
      gemm<true, true, EPI_BIAS_GELU>(m->st, nb, N, K, m->X[l], K, W, K, nullptr, m->X[l + 1], N, b,
                                      nullptr, keep_z ? m->Z[l] : nullptr);
    else
      gemm<true, true, EPI_BIAS_F32>(m->st, nb, N, K, m->X[l], K, W, K, m->Y, nullptr, N, b,
                                     nullptr, nullptr);
  }
}

// loss and gradient (into m->G) of nb rows in X[0] with targets in m->T
void backward(tsm_mlp* m, int nb) {
  const int L = m->L, no = m->w[L];
  const int n = nb * no;
  hipLaunchKernelGGL(k_mse, dim3((n + 255) / 256), dim3(256), 0, m->st, n, m->Y, m->T,
                     1.0f / (float)n, m->dA, m->part);
  u16 *dz = m->dA, *dx = m->dB;
  for (int l = L - 1; l >= 0; --l) {
    const int K = m->w[l], N = m->w[l + 1];
    // dW_l [N x K] = dz^T [N x nb] * x_l [nb x K]
    gemm<false, false, EPI_F32>(m->st, N, K, nb, dz, N, m->X[l], K, m->G + m->woff[l], nullptr, K,
                                nullptr, nullptr, nullptr);
    hipLaunchKernelGGL(k_colsum_bf16, dim3((N + 63) / 64), dim3(64), 0, m->st, nb, N, dz,
                       m->G + m->boff[l]);
    if (l > 0) {
      // dx_l [nb x K] = dz [nb x N] * W_l [N x K]; times GELU'(z_{l-1})
      gemm<true, false, EPI_GELU_BWD>(m->st, nb, K, N, dz, N, m->Pb + m->woff[l], K, nullptr, dx, K,
                                      nullptr, m->Z[l - 1], nullptr);
      std::swap(dz, dx);
    }
  }
}

// ---- fused nets ----
size_t rows_lds(const tsm_mlp* m) { return 2 * (size_t)RT * m->net.lda * sizeof(u16); }

// bf16 weights from the fp32 ones
void refresh_weights(tsm_mlp* m) {
  if (!m->fused) {
    hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((m->np + 255) / 256)), dim3(256), 0, m->st,
                       (int)m->np, m->P, m->Pb);
    return;
  }
  for (int l = 0; l < m->L; ++l)
    hipLaunchKernelGGL(k_pack_weights, dim3((m->w[l] * m->w[l + 1] + 255) / 256), dim3(256), 0, m->st,
                       m->net, l);
}

// one minibatch of nb rows: activations and dz, then the gradient (to G) or an
// Adam step, and the loss parts
void minibatch(tsm_mlp* m, int nb, const int* idx, const float* X, const float* T, float* part,
               const Adam* h) {
  const int no = m->w[m->L], n = nb * no;
  const size_t lds = rows_lds(m);
  // rows of XT/DT lie side by side for this minibatch (one stride of the largest
  // one a page apart would put every feature into the same cache sets)
  Net net = m->net;
  net.ldr = up(nb, RT);
  auto rows = [&](auto k, size_t lds) {
    if (lds > 48 * 1024)
      (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    // every row k_update reads (16 a product) is written, zero past the last
    hipLaunchKernelGGL(k, dim3(up(nb, 16) / RB), dim3(512), lds, m->st, net, nb, idx, X, T,
                       1.0f / (float)n);
  };
  if (net.lda <= 256 + 8) rows(k_rows_reg, lds + (size_t)(net.L - 1) * 512 * sizeof(float4));
  else rows(k_rows, lds);
  const int jobs = m->n_jobs + (n + 255) / 256;
  if (h)
    hipLaunchKernelGGL((k_update<true>), dim3((jobs + 3) / 4), dim3(256), 0, m->st, net, nb, m->jobs,
                       m->n_jobs, idx, T, part, *h);
  else
    hipLaunchKernelGGL((k_update<false>), dim3((jobs + 3) / 4), dim3(256), 0, m->st, net, nb, m->jobs,
                       m->n_jobs, idx, T, part, Adam{});
}

// Rows through the net in chunks whose staging stays under INFER_BYTES.  affine:
// FP64 rows with (mu_x, sd_x, mu_y, sd_y), else FP32 rows.
constexpr size_t INFER_BYTES = 64u << 20;
int infer(tsm_mlp* m, long n, const void* in, void* out, const double* affine) {
  const int ni = m->w[0], no = m->w[m->L];
  const size_t es = affine ? sizeof(double) : sizeof(float);
  const size_t na = affine ? 2 * (size_t)(ni + no) * sizeof(double) : 0;
  const long cap = std::max<long>(1024, (long)((INFER_BYTES - na) / (es * (ni + no))));
  const long rows = std::min(n, cap);
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t oi = al(na), oo = oi + al(es * ni * rows);
  MLP_TRY(m->grow(&m->io, &m->io_cap, oo + es * no * rows));
  if (affine) MLP_TRY(hipMemcpyAsync(m->io, affine, na, hipMemcpyHostToDevice, m->st));
  for (long r0 = 0; r0 < n; r0 += rows) {
    const long nr = std::min(rows, n - r0);
    MLP_TRY(hipMemcpyAsync(m->io + oi, static_cast<const char*>(in) + es * ni * r0, es * ni * nr,
                           hipMemcpyHostToDevice, m->st));
    // 64 rows per block once that still leaves two blocks per CU
    const int nt = nr >= 64 * 512 ? 2 : 1;
    const size_t lds = nt * rows_lds(m);
    auto go = [&](auto k) {
      if (lds > 48 * 1024)
        (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL(k, dim3((unsigned)((nr + RT * nt - 1) / (RT * nt))), dim3(512), lds, m->st,
                         m->net, nr, (const void*)(m->io + oi), (const double*)m->io,
                         (void*)(m->io + oo));
    };
    if (affine) { if (nt == 2) go(k_infer<2, true>); else go(k_infer<1, true>); }
    else { if (nt == 2) go(k_infer<2, false>); else go(k_infer<1, false>); }
    MLP_TRY(hipGetLastError());
    MLP_TRY(hipMemcpyAsync(static_cast<char*>(out) + es * no * r0, m->io + oo, es * no * nr,
                           hipMemcpyDeviceToHost, m->st));
    MLP_TRY(hipStreamSynchronize(m->st));
  }
  return TSM_OK;
}

int stage_rows(tsm_mlp* m, int rows, const float* x, const float* t) {
  const int ni = m->w[0], no = m->w[m->L];
  float* tmp = nullptr;
  MLP_TRY(hipMalloc(&tmp, (size_t)rows * ni * sizeof(float)));
  hipError_t e = hipMemcpyAsync(tmp, x, (size_t)rows * ni * sizeof(float), hipMemcpyHostToDevice, m->st);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_to_bf16, dim3((rows * ni + 255) / 256), dim3(256), 0, m->st, rows * ni, tmp,
                       m->X[0]);
    e = hipGetLastError();
  }
  if (e == hipSuccess && t)
    e = hipMemcpyAsync(m->T, t, (size_t)rows * no * sizeof(float), hipMemcpyHostToDevice, m->st);
  if (e == hipSuccess) e = hipStreamSynchronize(m->st);
  (void)hipFree(tmp);
  MLP_TRY(e);
  return TSM_OK;
}

}  // namespace

extern "C" const char* tsm_mlp_last_error(void) { return g_mlp_err.c_str(); }

extern "C" int tsm_mlp_create(int n_layers, const int* widths, int max_batch,
                              unsigned long long seed, tsm_mlp** out) {
  if (!out || n_layers < 1 || n_layers > 16 || !widths || max_batch < 1)
    return mfail(TSM_E_ARG, "bad argument");
  for (int l = 0; l <= n_layers; ++l)
    if (widths[l] < 1 || widths[l] > 4096) return mfail(TSM_E_ARG, "layer width out of range");
  tsm_mlp* m = new tsm_mlp();
  m->L = n_layers;
  m->maxb = max_batch;
  m->w.assign(widths, widths + n_layers + 1);
  int wmax = 0;
  for (int l = 0; l < n_layers; ++l) {
    m->woff.push_back(m->np);
    m->np += (size_t)m->w[l + 1] * m->w[l];
    m->boff.push_back(m->np);
    m->np += (size_t)m->w[l + 1];
  }
  for (int x : m->w) wmax = std::max(wmax, x);
  // He-style uniform init, variance 1/fan_in (splitmix64 stream)
  std::vector<float> h(m->np, 0.0f);
  uint64_t z = seed;
  auto next = [&]() {
    z += 0x9e3779b97f4a7c15ull;
    uint64_t q = z;
    q = (q ^ (q >> 30)) * 0xbf58476d1ce4e5b9ull;
    q = (q ^ (q >> 27)) * 0x94d049bb133111ebull;
    return (double)((q ^ (q >> 31)) >> 11) * 0x1p-53;
  };
  for (int l = 0; l < n_layers; ++l) {
    const double a = std::sqrt(3.0 / m->w[l]);
    for (size_t i = 0; i < (size_t)m->w[l + 1] * m->w[l]; ++i)
      h[m->woff[l] + i] = (float)(a * (2.0 * next() - 1.0));
  }
  m->fused = wmax <= FUSED_MAX;
  hipError_t e = hipStreamCreate(&m->st);
  m->X.assign(n_layers, nullptr);
  m->Z.assign(n_layers, nullptr);
  // one allocation for everything of a fixed size, cleared once (the padding of
  // the fused nets' operands stays zero)
  struct Piece { void** p; size_t bytes; };
  std::vector<Piece> pieces;
  auto want = [&](auto** p, size_t n) { pieces.push_back({(void**)p, n * sizeof(**p)}); };
  const int no = m->w[n_layers];
  want(&m->P, m->np); want(&m->G, m->np); want(&m->Mo, m->np); want(&m->Vo, m->np);
  for (int l = 0; l < n_layers; ++l) want(&m->Z[l], (size_t)max_batch * m->w[l + 1]);
  want(&m->Y, (size_t)max_batch * no);
  want(&m->T, (size_t)max_batch * no);
  want(&m->part, (size_t)max_batch * no / 256 + 2);
  Net& N = m->net;
  std::vector<int4> jobs;
  if (m->fused) {
    N.L = n_layers;
    N.ldr = up(max_batch, RT);
    for (int l = 0; l <= n_layers; ++l) {
      N.w[l] = m->w[l];
      N.lda = std::max(N.lda, up(m->w[l], 32) + 8);
    }
    for (int l = 0; l < n_layers; ++l) {
      const int ni = m->w[l], n1 = m->w[l + 1];
      want(&N.Wp[l], (size_t)up(n1, 32) * up(ni, 16));
      want(&N.Wt[l], (size_t)up(ni, 32) * up(n1, 16));
      want(&N.XT[l], (size_t)up(ni, 32) * N.ldr);
      want(&N.DT[l], (size_t)up(n1, 32) * N.ldr);
      N.woff[l] = (int)m->woff[l];
      N.boff[l] = (int)m->boff[l];
      for (int n = 0; n < n1; n += 32)
        for (int k = 0; k < ni; k += 32) jobs.push_back(int4{0, l, n, k});
      for (int n = 0; n < n1; n += 64) jobs.push_back(int4{1, l, n, 0});
    }
    m->n_jobs = (int)jobs.size();
    want(&m->jobs, jobs.size());
  } else {
    want(&m->Pb, m->np);
    for (int l = 0; l < n_layers; ++l) want(&m->X[l], (size_t)max_batch * m->w[l]);
    want(&m->dA, (size_t)max_batch * wmax);
    want(&m->dB, (size_t)max_batch * wmax);
  }
  size_t total = 0;
  for (auto& q : pieces) total += (q.bytes + 255) & ~(size_t)255;
  char* arena = nullptr;
  if (e == hipSuccess) e = m->al(&arena, total);
  if (e == hipSuccess) {
    size_t o = 0;
    for (auto& q : pieces) {
      *q.p = arena + o;
      o += (q.bytes + 255) & ~(size_t)255;
    }
    N.P = m->P; N.G = m->G; N.Mo = m->Mo; N.Vo = m->Vo; N.Y = m->Y; N.T = m->T;
    if (m->fused)
      for (int l = 0; l < n_layers; ++l) N.Z[l] = m->Z[l];
    e = hipMemsetAsync(arena, 0, total, m->st);
  }
  if (e == hipSuccess) e = hipMemcpyAsync(m->P, h.data(), m->np * sizeof(float), hipMemcpyHostToDevice, m->st);
  if (e == hipSuccess && m->fused)
    e = hipMemcpyAsync(m->jobs, jobs.data(), jobs.size() * sizeof(int4), hipMemcpyHostToDevice, m->st);
  if (e == hipSuccess) {
    refresh_weights(m);
    e = hipStreamSynchronize(m->st);
  }
  if (e != hipSuccess) {
    delete m;
    return mfail(TSM_E_HIP, hipGetErrorString(e));
  }
  *out = m;
  return TSM_OK;
}

extern "C" void tsm_mlp_destroy(tsm_mlp* m) { delete m; }

extern "C" long tsm_mlp_n_params(const tsm_mlp* m) { return m ? (long)m->np : -1; }

extern "C" int tsm_mlp_get_params(tsm_mlp* m, float* p) {
  if (!m || !p) return mfail(TSM_E_ARG, "bad argument");
  MLP_TRY(hipStreamSynchronize(m->st));
  MLP_TRY(hipMemcpy(p, m->P, m->np * sizeof(float), hipMemcpyDeviceToHost));
  return TSM_OK;
}

extern "C" int tsm_mlp_set_params(tsm_mlp* m, const float* p) {
  if (!m || !p) return mfail(TSM_E_ARG, "bad argument");
  MLP_TRY(hipStreamSynchronize(m->st));
  MLP_TRY(hipMemcpy(m->P, p, m->np * sizeof(float), hipMemcpyHostToDevice));
  refresh_weights(m);
  MLP_TRY(hipGetLastError());
  MLP_TRY(hipStreamSynchronize(m->st));
  return TSM_OK;
}

extern "C" int tsm_mlp_forward(tsm_mlp* m, long n, const float* x, float* y) {
  if (!m || n < 0 || (n > 0 && (!x || !y))) return mfail(TSM_E_ARG, "bad argument");
  if (m->fused) return n ? infer(m, n, x, y, nullptr) : TSM_OK;
  const int ni = m->w[0], no = m->w[m->L];
  for (long r0 = 0; r0 < n; r0 += m->maxb) {
    const int nb = (int)std::min<long>(m->maxb, n - r0);
    int rc = stage_rows(m, nb, x + (size_t)r0 * ni, nullptr);
    if (rc) return rc;
    forward(m, nb, false);
    MLP_TRY(hipGetLastError());
    MLP_TRY(hipMemcpyAsync(y + (size_t)r0 * no, m->Y, (size_t)nb * no * sizeof(float),
                           hipMemcpyDeviceToHost, m->st));
    MLP_TRY(hipStreamSynchronize(m->st));
  }
  return TSM_OK;
}

extern "C" int tsm_mlp_forward_affine(tsm_mlp* m, long n, const double* u, const double* mu_x,
                                      const double* sd_x, const double* mu_y, const double* sd_y,
                                      double* y) {
  if (!m || n < 0 || !mu_x || !sd_x || !mu_y || !sd_y || (n > 0 && (!u || !y)))
    return mfail(TSM_E_ARG, "bad argument");
  if (n == 0) return TSM_OK;
  const int ni = m->w[0], no = m->w[m->L];
  if (m->fused) {
    std::vector<double> a(mu_x, mu_x + ni);
    a.insert(a.end(), sd_x, sd_x + ni);
    a.insert(a.end(), mu_y, mu_y + no);
    a.insert(a.end(), sd_y, sd_y + no);
    return infer(m, n, u, y, a.data());
  }
  std::vector<float> x((size_t)n * ni), z((size_t)n * no);
  for (long r = 0; r < n; ++r)
    for (int k = 0; k < ni; ++k) x[(size_t)r * ni + k] = (float)((u[(size_t)r * ni + k] - mu_x[k]) / sd_x[k]);
  const int rc = tsm_mlp_forward(m, n, x.data(), z.data());
  if (rc) return rc;
  for (long r = 0; r < n; ++r)
    for (int k = 0; k < no; ++k) y[(size_t)r * no + k] = (double)z[(size_t)r * no + k] * sd_y[k] + mu_y[k];
  return TSM_OK;
}

extern "C" int tsm_mlp_gradient(tsm_mlp* m, int n, const float* x, const float* t, double* loss,
                                float* grad) {
  if (!m || n < 1 || n > m->maxb || !x || !t) return mfail(TSM_E_ARG, "bad argument");
  if (m->fused) {
    const size_t nx = (size_t)n * m->w[0], nt = (size_t)n * m->w[m->L];
    MLP_TRY(m->grow(&m->io, &m->io_cap, nx * sizeof(float)));
    MLP_TRY(hipMemcpyAsync(m->io, x, nx * sizeof(float), hipMemcpyHostToDevice, m->st));
    MLP_TRY(hipMemcpyAsync(m->T, t, nt * sizeof(float), hipMemcpyHostToDevice, m->st));
    minibatch(m, n, nullptr, reinterpret_cast<const float*>(m->io), m->T, m->part, nullptr);
  } else {
    int rc = stage_rows(m, n, x, t);
    if (rc) return rc;
    forward(m, n, true);
    backward(m, n);
  }
  MLP_TRY(hipGetLastError());
  const int nparts = (n * m->w[m->L] + 255) / 256;
  std::vector<float> part(nparts);
  MLP_TRY(hipMemcpyAsync(part.data(), m->part, nparts * sizeof(float), hipMemcpyDeviceToHost, m->st));
  if (grad) MLP_TRY(hipMemcpyAsync(grad, m->G, m->np * sizeof(float), hipMemcpyDeviceToHost, m->st));
  MLP_TRY(hipStreamSynchronize(m->st));
  double s = 0.0;
  for (float p : part) s += p;
  if (loss) *loss = s / ((double)n * m->w[m->L]);
  return TSM_OK;
}

extern "C" int tsm_mlp_train(tsm_mlp* m, long n, const float* x, const float* t, int epochs,
                             int batch, float lr, unsigned long long seed, double* epoch_loss) {
  if (!m || n < 1 || !x || !t || epochs < 0 || batch < 1 || batch > m->maxb)
    return mfail(TSM_E_ARG, "bad argument");
  const int ni = m->w[0], no = m->w[m->L];
  if ((size_t)n > m->nin_cap) {
    MLP_TRY(m->al(&m->Xin, (size_t)n * ni));
    MLP_TRY(m->al(&m->Tin, (size_t)n * no));
    MLP_TRY(m->al(&m->idx, (size_t)n));
    m->nin_cap = (size_t)n;
  }
  MLP_TRY(hipMemcpyAsync(m->Xin, x, (size_t)n * ni * sizeof(float), hipMemcpyHostToDevice, m->st));
  MLP_TRY(hipMemcpyAsync(m->Tin, t, (size_t)n * no * sizeof(float), hipMemcpyHostToDevice, m->st));
  std::vector<int> perm(n);
  for (long i = 0; i < n; ++i) perm[i] = (int)i;
  uint64_t z = seed ^ 0x5851f42d4c957f2dull;
  auto next = [&]() {
    z += 0x9e3779b97f4a7c15ull;
    uint64_t q = z;
    q = (q ^ (q >> 30)) * 0xbf58476d1ce4e5b9ull;
    q = (q ^ (q >> 27)) * 0x94d049bb133111ebull;
    return q ^ (q >> 31);
  };
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const int nmb = (int)((n + batch - 1) / batch);
  std::vector<float> part;
  const size_t mp = ((size_t)batch * no + 255) / 256;  // loss parts of a full minibatch
  if (m->fused) MLP_TRY(m->grow(&m->parts, &m->parts_cap, mp * nmb));
  for (int ep = 0; ep < epochs; ++ep) {
    for (long i = n - 1; i > 0; --i) std::swap(perm[i], perm[next() % (uint64_t)(i + 1)]);
    MLP_TRY(hipMemcpyAsync(m->idx, perm.data(), n * sizeof(int), hipMemcpyHostToDevice, m->st));
    MLP_TRY(hipStreamSynchronize(m->st));  // perm is reused by the next epoch
    double esum = 0.0;
    if (m->fused) {  // the loss parts stay on the device until the epoch has run
      for (int b = 0; b < nmb; ++b) {
        const int r0 = b * batch, nb = (int)std::min<long>(batch, n - r0);
        ++m->adam_t;
        const Adam h{lr, b1, b2, eps, 1.0f - std::pow(b1, (float)m->adam_t),
                     1.0f - std::pow(b2, (float)m->adam_t)};
        minibatch(m, nb, m->idx + r0, m->Xin, m->Tin, m->parts + mp * b, &h);
      }
      MLP_TRY(hipGetLastError());
      if (epoch_loss) {
        part.resize(mp * nmb);
        MLP_TRY(hipMemcpyAsync(part.data(), m->parts, part.size() * sizeof(float), hipMemcpyDeviceToHost,
                               m->st));
        MLP_TRY(hipStreamSynchronize(m->st));
        for (int b = 0; b < nmb; ++b) {
          const long nb = std::min<long>(batch, n - (long)b * batch);
          double s = 0.0;
          for (long k = 0; k < (nb * no + 255) / 256; ++k) s += part[mp * b + k];
          esum += s;
        }
        epoch_loss[ep] = esum / ((double)n * no);
      }
      continue;
    }
    for (int b = 0; b < nmb; ++b) {
      const int r0 = b * batch, nb = (int)std::min<long>(batch, n - r0);
      hipLaunchKernelGGL(k_gather_rows, dim3((nb * ni + 255) / 256), dim3(256), 0, m->st, nb, ni,
                         m->idx + r0, m->Xin, m->X[0], nullptr);
      hipLaunchKernelGGL(k_gather_rows, dim3((nb * no + 255) / 256), dim3(256), 0, m->st, nb, no,
                         m->idx + r0, m->Tin, nullptr, m->T);
      forward(m, nb, true);
      backward(m, nb);
      ++m->adam_t;
      const float c1 = 1.0f - std::pow(b1, (float)m->adam_t), c2 = 1.0f - std::pow(b2, (float)m->adam_t);
      hipLaunchKernelGGL(k_adam, dim3((unsigned)((m->np + 255) / 256)), dim3(256), 0, m->st,
                         (int)m->np, m->P, m->G, m->Mo, m->Vo, m->Pb, lr, b1, b2, eps, c1, c2);
      MLP_TRY(hipGetLastError());
      if (epoch_loss) {
        const int nparts = (nb * no + 255) / 256;
        part.resize(nparts);
        MLP_TRY(hipMemcpyAsync(part.data(), m->part, nparts * sizeof(float), hipMemcpyDeviceToHost,
                               m->st));
        MLP_TRY(hipStreamSynchronize(m->st));
        double s = 0.0;
        for (float p : part) s += p;
        esum += s;
      }
    }
    if (epoch_loss) epoch_loss[ep] = esum / ((double)n * no);
  }
  MLP_TRY(hipStreamSynchronize(m->st));
  return TSM_OK;
}

// Plain GEMM through the same kernel, for tests of the MFMA tiling:
// C[M x N] (fp32) = A * B with A, B given in bf16 bit patterns and the layout
// flags of the kernel (a_kmajor: A is M x K row-major, else K x M; b_kmajor: B
// is N x K row-major, else K x N).
extern "C" int tsm_mlp_gemm_test(int M, int N, int K, const unsigned short* A, int a_kmajor,
                                 const unsigned short* B, int b_kmajor, float* C) {
  if (M < 1 || N < 1 || K < 1 || !A || !B || !C) return mfail(TSM_E_ARG, "bad argument");
  u16 *dA = nullptr, *dB = nullptr;
  float* dC = nullptr;
  MLP_TRY(hipMalloc(&dA, (size_t)M * K * 2));
  hipError_t e = hipMalloc(&dB, (size_t)N * K * 2);
  if (e == hipSuccess) e = hipMalloc(&dC, (size_t)M * N * 4);
  if (e == hipSuccess) e = hipMemcpy(dA, A, (size_t)M * K * 2, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dB, B, (size_t)N * K * 2, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    const int lda = a_kmajor ? K : M, ldb = b_kmajor ? K : N;
    if (a_kmajor && b_kmajor) gemm<true, true, EPI_F32>(0, M, N, K, dA, lda, dB, ldb, dC, nullptr, N, nullptr, nullptr, nullptr);
    else if (a_kmajor) gemm<true, false, EPI_F32>(0, M, N, K, dA, lda, dB, ldb, dC, nullptr, N, nullptr, nullptr, nullptr);
    else if (b_kmajor) gemm<false, true, EPI_F32>(0, M, N, K, dA, lda, dB, ldb, dC, nullptr, N, nullptr, nullptr, nullptr);
    else gemm<false, false, EPI_F32>(0, M, N, K, dA, lda, dB, ldb, dC, nullptr, N, nullptr, nullptr, nullptr);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(C, dC, (size_t)M * N * 4, hipMemcpyDeviceToHost);
  (void)hipFree(dA); (void)hipFree(dB); (void)hipFree(dC);
  MLP_TRY(e);
  return TSM_OK;
}
