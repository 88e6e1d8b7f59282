// ekpnp_mlp.hip -- warm-start surrogate: BF16 MFMA multilayer perceptron with
// FP32 accumulation, FP32 master weights and Adam, all on the GPU.
//
// Layer l maps a_{l-1} [B][in_l] to z_l = a_{l-1} W_l^T + b_l [B][out_l];
// hidden layers store z_l (FP32, for GELU') and a_l = bf16(GELU(z_l)); the
// last layer is linear.  Backward (loss = mean (y - t)^2):
//   g_{L+1} = 2 (y - t) / (B n_out)
//   dW_l = g_l^T a_{l-1},  db_l = sum_b g_l,  g_{l-1} = (g_l W_l) * GELU'(z_{l-1})
// with g_l rounded to BF16 before it enters a product.  Every product is
// C[M][N] = sum_k A[m][k] B[n][k] with k contiguous in both operands
// (k_gemm, k_wgrad): the epilogues that write a_l and g_l also write their
// transposes, and the BF16 weight shadow is kept in both orders, so a lane
// loads its MFMA fragment (8 consecutive k of one row) straight from memory.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <algorithm>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/ekpnp_mlp.h"
#include "../../include/ekpnp_seed.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int TILE = 16;     // MFMA tile edge
constexpr int KSTEP = 32;    // k of one v_mfma_f32_16x16x32_bf16
constexpr int MLP_WG = 256;  // lanes of a work-group, four waves
constexpr int KGROUP = 8;    // k steps whose loads are in flight together

// round-to-nearest-even FP32 -> BF16 bits
__host__ __device__ inline uint16_t f2bf(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}


__device__ inline float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ inline float dgelu(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// Accumulates C(m0.., n0..) = sum_k A[m][k] B[n][k] of one 16 x 16 tile, k in
// steps of 32 from 0 up (K a multiple of 32, rows 16-byte aligned).
// Lane layout of v_mfma_f32_16x16x32_bf16: A / B row = lane % 16, k = 8 (lane /
// 16) + 0..7; C column = lane % 16, rows 4 (lane / 16) + 0..3.
__device__ __forceinline__ floatx4 tile_product(const uint16_t* __restrict__ A, long long lda,
                                                const uint16_t* __restrict__ B, long long ldb, int m0, int n0, int K) {
  const int lane = threadIdx.x & 63;
  const u16x8* pa = reinterpret_cast<const u16x8*>(A + (m0 + (lane & 15)) * lda) + (lane >> 4);
  const u16x8* pb = reinterpret_cast<const u16x8*>(B + (n0 + (lane & 15)) * ldb) + (lane >> 4);
  constexpr int STEP = KSTEP / 8;  // 16-byte values per k step and row
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  u16x8 va[KGROUP], vb[KGROUP];
  const int steps = K / KSTEP;
  for (int s0 = 0; s0 < steps; s0 += KGROUP) {
#pragma unroll
    for (int u = 0; u < KGROUP; ++u)
      if (s0 + u < steps) {
        va[u] = pa[(s0 + u) * STEP];
        vb[u] = pb[(s0 + u) * STEP];
      }
#pragma unroll
    for (int u = 0; u < KGROUP; ++u)
      if (s0 + u < steps)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, va[u]),
                                                      __builtin_bit_cast(bf16x8, vb[u]), acc, 0, 0, 0);
  }
  return acc;
}

enum Epi { EPI_HIDDEN = 0, EPI_OUT = 1, EPI_LOSS = 2, EPI_DGELU = 3 };

struct GemmArgs {
  const uint16_t* A;   // [rows][K], rows a multiple of 32
  const uint16_t* B;   // [N][K]
  int M, N, K;         // M: rows that count; the transposes hold 0 from row M up to the next multiple of 32
  const float* bias;   // [N]                       (HIDDEN, OUT, LOSS)
  float* z;            // pre-activation [M][N]: written (HIDDEN, OUT), read (DGELU)
  const float* t;      // targets [M][N]            (LOSS)
  float* g;            // FP32 gradient [M][N]      (LOSS, DGELU)
  uint16_t* c;         // BF16 a_l or g_l [rows][N] (HIDDEN, LOSS, DGELU)
  uint16_t* ct;        // its transpose [N][ldt]    (HIDDEN while training, LOSS, DGELU; may be null)
  long long ldt;
  double* partial;     // squared-error sum of each work-group (LOSS)
  float scale;         // 1 / (M N)                 (LOSS)
};

// One 16 x 16 tile per wave.  A layer of the warm-start network (256 x 256 at a
// batch of 256) is 256 waves, one per CU, each with all its loads in flight:
// latency bounds it.  64 x 64 tiles staged through LDS two bytes at a time put
// the same layer on 16 CUs (hidden layer 20.7 us, backward 49 us a launch; 4.0 and
// 4.5 - 12 us now).
template <int EPI>
__global__ __launch_bounds__(MLP_WG) void k_gemm(GemmArgs g) {
  __shared__ double red[MLP_WG / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * TILE, n0 = (blockIdx.x * (MLP_WG / 64) + wave) * TILE;
  // squared errors, summed in FP64: an FP32 sum over the work-group's 1024
  // loses the small ones beside a large one
  double e2 = 0.0;
  if (n0 < g.N) {
    const floatx4 acc = tile_product(g.A, g.K, g.B, g.K, m0, n0, g.K);
    const int n = n0 + (lane & 15), mr = m0 + (lane >> 4) * 4;
    uint16_t h[4] = {0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = mr + r;
      if (m >= g.M) continue;
      const long long o = (long long)m * g.N + n;
      float v = acc[r];
      if (EPI == EPI_HIDDEN) {
        v += g.bias[n];
        g.z[o] = v;
        h[r] = f2bf(gelu(v));
        g.c[o] = h[r];
      } else if (EPI == EPI_OUT) {
        g.z[o] = v + g.bias[n];
      } else if (EPI == EPI_LOSS) {
        // loss gradient 2 (y - t) / (M N)
        const float d = v + g.bias[n] - g.t[o];
        const float gv = 2.0f * d * g.scale;
        g.g[o] = gv;
        h[r] = f2bf(gv);
        g.c[o] = h[r];
        e2 += (double)d * (double)d;
      } else {
        v *= dgelu(g.z[o]);
        g.g[o] = v;
        h[r] = f2bf(v);
        g.c[o] = h[r];
      }
    }
    // four consecutive rows of one column: one 8-byte value of the transpose
    if (EPI != EPI_OUT && g.ct)
      *reinterpret_cast<u16x4*>(g.ct + (long long)n * g.ldt + mr) = u16x4{h[0], h[1], h[2], h[3]};
  }
  if (EPI == EPI_LOSS) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) e2 += __shfl_down(e2, off, 64);
    if (lane == 0) red[wave] = e2;
    __syncthreads();
    if (threadIdx.x == 0)
      g.partial[blockIdx.y * gridDim.x + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
  }
}

// One layer of the network as the weight kernels see it
struct Layer {
  const uint16_t* at;   // a_{l-1} transposed [in][ldt]
  const uint16_t* gt;   // g_l transposed [out][ldt]
  const float* g;       // g_l, FP32 [B][out]
  int in, out;
  long long off_w, off_b;  // in the parameter vector
  uint16_t* wt;         // W_l transposed [in][out], BF16 (null for the first layer)
  int wg_first;         // first k_wgrad work-group: weight tiles, then 16-column bias blocks
  int wg_bias;          // first of the bias blocks
  int up_first;         // first k_update work-group: 32 x 32 weight tiles, then the bias
};

// layer of work-group wg (first(l) ascending)
template <typename F>
__device__ __forceinline__ int find_layer(int n, int wg, F first) {
  int l = 0;
  while (l + 1 < n && wg >= first(l + 1)) ++l;
  return l;
}

// Weight and bias gradients of every layer in one launch:
//   dW_l[o][i] = sum_b g_l[b][o] a_{l-1}[b][i], one 16 x 16 tile per wave (K = the
//   batch rounded up to 32, zeros past it);
//   db_l[n] = sum_b g_l[b][n] in FP32, one row after the other: 16 columns per
//   work-group, 256 rows at a time through LDS (any other order would give
//   other last bits, which Adam's normalisation and the BF16 shadows amplify
//   over a training run).
// Five products of 26-30 us and five one-lane-per-column sums of 46-55 us
// before (a batch of 256): too few work-groups, and a serial chain of loads;
// 8.2 us now.  A training step of the 6 -> 4 x 256 -> 1024 network at a batch of
// 256, with its host copies: 840 -> 140 us, at 512 1309 -> 178 us.
constexpr int BIAS_ROWS = 256;
__global__ __launch_bounds__(MLP_WG) void k_wgrad(const Layer* __restrict__ layers, int n_layers, float* __restrict__ grad,
                                                  long long ldt, int B) {
  __shared__ float part[BIAS_ROWS][TILE + 1];
  const int wg = blockIdx.x;
  const Layer L = layers[find_layer(n_layers, wg, [&](int l) { return layers[l].wg_first; })];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wg < L.wg_bias) {
    const int tile = (wg - L.wg_first) * (MLP_WG / 64) + wave, nt = L.in / TILE;
    const int m0 = tile / nt * TILE, n0 = (tile - tile / nt * nt) * TILE;
    if (m0 >= L.out) return;
    const floatx4 acc = tile_product(L.gt, ldt, L.at, ldt, m0, n0, (B + KSTEP - 1) / KSTEP * KSTEP);
    float* o = grad + L.off_w + (long long)(m0 + (lane >> 4) * 4) * L.in + n0 + (lane & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) o[(long long)r * L.in] = acc[r];
    return;
  }
  const int n0 = (wg - L.wg_bias) * TILE, col = threadIdx.x & (TILE - 1), row = threadIdx.x / TILE;
  float s = 0.f;
  for (int b0 = 0; b0 < B; b0 += BIAS_ROWS) {
    float v[TILE];
#pragma unroll
    for (int c = 0; c < TILE; ++c) v[c] = L.g[(long long)min(b0 + row + c * (MLP_WG / TILE), B - 1) * L.out + n0 + col];
    __syncthreads();  // the previous rows have been added
#pragma unroll
    for (int c = 0; c < TILE; ++c) part[row + c * (MLP_WG / TILE)][col] = v[c];
    __syncthreads();
    if (row == 0)
#pragma unroll 16
      for (int k = 0; k < min(BIAS_ROWS, B - b0); ++k) s += part[k][col];
  }
  if (row == 0) grad[L.off_b + n0 + col] = s;
}

struct AdamArgs {
  float lr, b1, b2, eps, wd, c1, c2;
};

// Adam on the FP32 master parameters (UPDATE) and the BF16 shadows, as stored
// and transposed; one 32 x 32 weight tile per work-group, then 1024 biases
template <bool UPDATE>
__global__ __launch_bounds__(MLP_WG) void k_update(const Layer* __restrict__ layers, int n_layers, float* __restrict__ p,
                                                   const float* __restrict__ g, float* __restrict__ m,
                                                   float* __restrict__ v, uint16_t* __restrict__ pb, AdamArgs a) {
  __shared__ uint16_t tile[32][33];
  const int wg = blockIdx.x;
  const Layer L = layers[find_layer(n_layers, wg, [&](int l) { return layers[l].up_first; })];
  auto update = [&](long long i) {
    float pi = p[i];
    if (UPDATE) {
      // (the contractions are spelled out, so that they do not depend on what
      // surrounds this)
      const float gi = __builtin_fmaf(a.wd, pi, g[i]);
      const float mi = __builtin_fmaf(a.b1, m[i], (1.f - a.b1) * gi);
      const float vi = __builtin_fmaf(a.b2, v[i], (1.f - a.b2) * gi * gi);
      m[i] = mi;
      v[i] = vi;
      pi = pi - a.lr * (mi * a.c1) / (sqrtf(vi * a.c2) + a.eps);
      p[i] = pi;
    }
    const uint16_t h = f2bf(pi);
    pb[i] = h;
    return h;
  };
  const int nt = L.in / 32, t = wg - L.up_first, rt = t / nt;
  if (rt >= L.out / 32) {
    const int i0 = (t - nt * (L.out / 32)) * 1024;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int i = i0 + c * MLP_WG + (int)threadIdx.x;
      if (i < L.out) update(L.off_b + i);
    }
    return;
  }
  const int r0 = rt * 32, c0 = (t - rt * nt) * 32, x = threadIdx.x & 31, y = threadIdx.x >> 5;
#pragma unroll
  for (int c = 0; c < 4; ++c) tile[y + 8 * c][x] = update(L.off_w + (long long)(r0 + y + 8 * c) * L.in + c0 + x);
  if (!L.wt) return;
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 4; ++c) L.wt[(long long)(c0 + y + 8 * c) * L.out + r0 + x] = tile[x][y + 8 * c];
}

// x (FP32 [B][n_in]) -> BF16 [rows][in_pad] and its transpose, zeros past n_in
// and past B
__global__ void k_pack_input(const float* __restrict__ x, uint16_t* __restrict__ xb, uint16_t* __restrict__ xt,
                             long long ldt, int rows, int B, int n_in, int in_pad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * in_pad) return;
  const int b = i / in_pad, c = i - b * in_pad;
  const uint16_t h = (c < n_in && b < B) ? f2bf(x[(long long)b * n_in + c]) : (uint16_t)0;
  xb[i] = h;
  xt[(long long)c * ldt + b] = h;
}

}  // namespace

struct ekpnp_mlp {
  ekpnp_mlp_config cfg{};
  int in_pad = 32, L = 0;
  long long rows = 0;                      // max_batch rounded up to 32: rows of a and g, columns of their transposes
  std::vector<int> in_dim, out_dim;        // per layer 1..L+1 (index 0 unused)
  std::vector<long long> off_w, off_b;
  long long n_params = 0;
  float *p32 = nullptr, *m32 = nullptr, *v32 = nullptr, *g32 = nullptr;
  uint16_t* pbf = nullptr;
  std::vector<float*> z;       // [L+2], z[l] FP32 [B][out_l]
  std::vector<uint16_t*> a;    // [L+1], a[0] the packed input, a[l] BF16 [rows][out_l]
  std::vector<uint16_t*> at;   // [L+1], their transposes [out_l][rows]
  std::vector<float*> g;       // [L+2], g[l] FP32 [B][out_l]
  std::vector<uint16_t*> gb;   // [L+2], g[l] BF16 [rows][out_l]
  std::vector<uint16_t*> gt;   // [L+2], its transpose [out_l][rows]
  std::vector<uint16_t*> wt;   // [L+2], W_l transposed [in_l][out_l], l >= 2
  float* t = nullptr;          // targets
  float* xin = nullptr;        // FP32 input staging
  double* partial = nullptr;   // squared-error sums, written by the device into host memory
  Layer* layers = nullptr;     // layer table of the weight kernels, layers 1..L+1
  int n_wgrad = 0, n_update = 0;  // their work-groups
  std::vector<void*> bufs;     // every device allocation
  hipStream_t stream = nullptr;
  float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f, wd = 0.f;
  long long adam_t = 0;
  std::string err;
};

namespace {

int mfail(ekpnp_mlp* m, int code, const std::string& msg) {
  if (m) m->err = msg;
  return code;
}

#define MHIP(m, call)                                                                   \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess) return mfail((m), -2, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

void release(ekpnp_mlp* m) {
  for (void* p : m->bufs)
    if (p) (void)hipFree(p);
  if (m->partial) (void)hipHostFree(m->partial);
  if (m->stream) (void)hipStreamDestroy(m->stream);
}

int rows_of(int B) { return (B + KSTEP - 1) / KSTEP * KSTEP; }
int gemm_columns(int N) { return (N / TILE + MLP_WG / 64 - 1) / (MLP_WG / 64); }  // work-groups a row of tiles
// squared-error sums of a batch of rows (k_gemm<EPI_LOSS>)
size_t loss_partials(int N, int rows) { return (size_t)gemm_columns(N) * (rows / TILE); }

// k_gemm over rows (a multiple of 32) rows.  Row tiles lie on the grid's y, which
// holds 65536: a larger batch, above 1,048,560, takes several launches, each
// with its operands' first rows.  (The grid's z instead costs the launches of
// ordinary batches 0.3 us each: reading the grid's size, a bound to check.)
template <int EPI>
void launch_gemm(GemmArgs g, int rows, hipStream_t s) {
  constexpr int MOST = 65535 * TILE;
  const int gx = gemm_columns(g.N);
  for (;;) {
    const int n = std::min(rows, MOST);
    hipLaunchKernelGGL(k_gemm<EPI>, dim3(gx, n / TILE), dim3(MLP_WG), 0, s, g);
    rows -= n;
    if (rows == 0) return;
    const size_t o = (size_t)n * g.N;
    g.A += (size_t)n * g.K;
    g.M -= n;
    if (g.z) g.z += o;
    if (g.t) g.t += o;
    if (g.g) g.g += o;
    if (g.c) g.c += o;
    if (g.ct) g.ct += n;
    if (g.partial) g.partial += loss_partials(g.N, n);
  }
}

// layers 1 .. last of the forward pass (hidden layers, or with L + 1 the
// linear output too); train: the transposed activations are written as well
hipError_t forward(ekpnp_mlp* m, const float* x_host, int B, int last, bool train) {
  hipError_t e = hipMemcpyAsync(m->xin, x_host, (size_t)B * m->cfg.n_in * sizeof(float),
                                hipMemcpyHostToDevice, m->stream);
  if (e != hipSuccess) return e;
  const int rows = rows_of(B), n = rows * m->in_pad;
  hipLaunchKernelGGL(k_pack_input, dim3((n + 255) / 256), dim3(256), 0, m->stream, m->xin, m->a[0], m->at[0], m->rows,
                     rows, B, m->cfg.n_in, m->in_pad);
  for (int l = 1; l <= last; ++l) {
    GemmArgs g{};
    g.A = m->a[l - 1];
    g.B = m->pbf + m->off_w[l];
    g.M = B;
    g.N = m->out_dim[l];
    g.K = m->in_dim[l];
    g.bias = m->p32 + m->off_b[l];
    g.z = m->z[l];
    if (l <= m->L) {
      g.c = m->a[l];
      g.ct = train ? m->at[l] : nullptr;
      g.ldt = m->rows;
      launch_gemm<EPI_HIDDEN>(g, rows, m->stream);
    } else {
      launch_gemm<EPI_OUT>(g, rows, m->stream);
    }
  }
  return hipGetLastError();
}

// forward and backward pass: fills g32 with the gradient of the loss and
// leaves the work-groups' squared-error sums in partial (host memory, valid
// once the stream is synchronised; see loss_of)
int loss_grad(ekpnp_mlp* m, const float* x_host, const float* t_host, int B) {
  const int L = m->L, no = m->cfg.n_out, rows = rows_of(B);
  MHIP(m, forward(m, x_host, B, L, true));
  MHIP(m, hipMemcpyAsync(m->t, t_host, (size_t)B * no * sizeof(float), hipMemcpyHostToDevice, m->stream));
  for (int l = L + 1; l >= 1; --l) {
    GemmArgs g{};
    if (l == L + 1) {
      // output layer and the loss gradient g_{L+1}
      g.A = m->a[L];
      g.B = m->pbf + m->off_w[l];
      g.K = m->in_dim[l];
      g.bias = m->p32 + m->off_b[l];
      g.t = m->t;
      g.partial = m->partial;
      g.scale = 1.0f / (float)(B * no);
    } else {
      // g_l[b][i] = sum_o g_{l+1}[b][o] W_{l+1}[o][i] * GELU'(z_l[b][i])
      g.A = m->gb[l + 1];
      g.B = m->wt[l + 1];
      g.K = m->out_dim[l + 1];
      g.z = m->z[l];
    }
    g.M = B;
    g.N = m->out_dim[l];
    g.g = m->g[l];
    g.c = m->gb[l];
    g.ct = m->gt[l];
    g.ldt = m->rows;
    if (l == L + 1) launch_gemm<EPI_LOSS>(g, rows, m->stream);
    else launch_gemm<EPI_DGELU>(g, rows, m->stream);
  }
  hipLaunchKernelGGL(k_wgrad, dim3(m->n_wgrad), dim3(MLP_WG), 0, m->stream, m->layers, L + 1, m->g32, m->rows, B);
  MHIP(m, hipGetLastError());
  return 0;
}

float loss_of(const ekpnp_mlp* m, int B) {
  const int no = m->cfg.n_out;
  const size_t n = loss_partials(no, rows_of(B));
  double s = 0.0;
  for (size_t i = 0; i < n; ++i) s += m->partial[i];
  return (float)(s / (double)(B * no));
}

// BF16 shadows of the master parameters, and the Adam step before them
template <bool UPDATE>
hipError_t update(ekpnp_mlp* m, const AdamArgs& a) {
  hipLaunchKernelGGL(k_update<UPDATE>, dim3(m->n_update), dim3(MLP_WG), 0, m->stream, m->layers, m->L + 1, m->p32,
                     m->g32, m->m32, m->v32, m->pbf, a);
  return hipGetLastError();
}

}  // namespace

extern "C" {

int ekpnp_mlp_create(const ekpnp_mlp_config* cfg, ekpnp_mlp** out) {
  if (!cfg || !out) return -1;
  *out = nullptr;
  if (cfg->n_in < 1 || cfg->n_in > 32 || cfg->n_hidden < 32 || cfg->n_hidden % 32 || cfg->n_layers < 1 ||
      cfg->n_out < 32 || cfg->n_out % 32 || cfg->max_batch < 1)
    return -1;
  if (hipSetDevice(cfg->device) != hipSuccess) return -2;
  ekpnp_mlp* m = new ekpnp_mlp();
  m->cfg = *cfg;
  m->L = cfg->n_layers;
  const int L = m->L, H = cfg->n_hidden, B = cfg->max_batch;
  m->in_dim.assign(L + 2, 0);
  m->out_dim.assign(L + 2, 0);
  m->off_w.assign(L + 2, 0);
  m->off_b.assign(L + 2, 0);
  long long off = 0;
  for (int l = 1; l <= L + 1; ++l) {
    m->in_dim[l] = (l == 1) ? m->in_pad : H;
    m->out_dim[l] = (l <= L) ? H : cfg->n_out;
    m->off_w[l] = off;
    off += (long long)m->in_dim[l] * m->out_dim[l];
    m->off_b[l] = off;
    off += m->out_dim[l];
  }
  m->n_params = off;
  // He initialisation from the shared splitmix64 stream (Box-Muller)
  std::vector<float> p(off, 0.f);
  uint64_t st = ekpnp_stream_key(cfg->seed, 0x6d6c70ull, 0);
  for (int l = 1; l <= L + 1; ++l) {
    const int fan_in = (l == 1) ? cfg->n_in : H;
    const double sd = std::sqrt(2.0 / fan_in);
    for (int o = 0; o < m->out_dim[l]; ++o)
      for (int i = 0; i < m->in_dim[l]; ++i) {
        double u1 = ekpnp_uniform01(&st), u2 = ekpnp_uniform01(&st);
        double nrm = std::sqrt(-2.0 * std::log(1.0 - u1)) * std::cos(2.0 * M_PI * u2);
        if (l == 1 && i >= cfg->n_in) nrm = 0.0;  // padding columns
        p[m->off_w[l] + (long long)o * m->in_dim[l] + i] = (float)(sd * nrm);
      }
  }
  const long long R = m->rows = rows_of(B);
  hipError_t e = hipSuccess;
  auto A = [&](auto** ptr, size_t count) {
    if (e != hipSuccess) return;
    void* p = nullptr;
    e = hipMalloc(&p, std::max<size_t>(count * sizeof(**ptr), 16));
    if (e != hipSuccess) return;
    *ptr = static_cast<std::remove_reference_t<decltype(*ptr)>>(p);
    m->bufs.push_back(p);
  };
  A(&m->p32, off);
  A(&m->m32, off);
  A(&m->v32, off);
  A(&m->g32, off);
  A(&m->pbf, off);
  A(&m->xin, (size_t)B * cfg->n_in);
  A(&m->t, (size_t)B * cfg->n_out);
  A(&m->layers, L + 1);
  m->z.assign(L + 2, nullptr);
  m->g.assign(L + 2, nullptr);
  m->gb.assign(L + 2, nullptr);
  m->gt.assign(L + 2, nullptr);
  m->wt.assign(L + 2, nullptr);
  m->a.assign(L + 1, nullptr);
  m->at.assign(L + 1, nullptr);
  A(&m->a[0], R * m->in_pad);
  A(&m->at[0], R * m->in_pad);
  for (int l = 1; l <= L + 1; ++l) {
    const size_t n = (size_t)m->out_dim[l];
    A(&m->z[l], (size_t)B * n);
    A(&m->g[l], (size_t)B * n);
    A(&m->gb[l], R * n);
    A(&m->gt[l], R * n);
    if (l <= L) A(&m->a[l], R * n);
    if (l <= L) A(&m->at[l], R * n);
    if (l >= 2) A(&m->wt[l], n * m->in_dim[l]);
  }
  if (e == hipSuccess)
    e = hipHostMalloc((void**)&m->partial, loss_partials(cfg->n_out, (int)R) * sizeof(double), hipHostMallocDefault);
  std::vector<Layer> tab(L + 1);
  for (int l = 1; l <= L + 1; ++l) {
    Layer& d = tab[l - 1];
    d.at = m->at[l - 1];
    d.gt = m->gt[l];
    d.g = m->g[l];
    d.in = m->in_dim[l];
    d.out = m->out_dim[l];
    d.off_w = m->off_w[l];
    d.off_b = m->off_b[l];
    d.wt = m->wt[l];
    d.wg_first = m->n_wgrad;
    d.wg_bias = d.wg_first + (d.in / TILE * (d.out / TILE) + MLP_WG / 64 - 1) / (MLP_WG / 64);
    m->n_wgrad = d.wg_bias + d.out / TILE;
    d.up_first = m->n_update;
    m->n_update += d.in / 32 * (d.out / 32) + (d.out + 1023) / 1024;
  }
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipMemcpy(m->layers, tab.data(), tab.size() * sizeof(Layer), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(m->p32, p.data(), off * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(m->m32, 0, off * 4);
  if (e == hipSuccess) e = hipMemset(m->v32, 0, off * 4);
  if (e == hipSuccess) e = update<false>(m, AdamArgs{});
  if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
  if (e != hipSuccess) {
    release(m);
    delete m;
    return e == hipErrorOutOfMemory ? -3 : -2;
  }
  *out = m;
  return 0;
}

void ekpnp_mlp_destroy(ekpnp_mlp* m) {
  if (!m) return;
  (void)hipSetDevice(m->cfg.device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  release(m);
  delete m;
}

const char* ekpnp_mlp_last_error(const ekpnp_mlp* m) { return m ? m->err.c_str() : "null surrogate"; }

long long ekpnp_mlp_num_params(const ekpnp_mlp* m) { return m ? m->n_params : 0; }

int ekpnp_mlp_get_params(ekpnp_mlp* m, float* out) {
  if (!m || !out) return -1;
  MHIP(m, hipSetDevice(m->cfg.device));
  MHIP(m, hipStreamSynchronize(m->stream));
  MHIP(m, hipMemcpy(out, m->p32, m->n_params * 4, hipMemcpyDeviceToHost));
  return 0;
}

int ekpnp_mlp_set_params(ekpnp_mlp* m, const float* in) {
  if (!m || !in) return -1;
  MHIP(m, hipSetDevice(m->cfg.device));
  MHIP(m, hipStreamSynchronize(m->stream));
  MHIP(m, hipMemcpy(m->p32, in, m->n_params * 4, hipMemcpyHostToDevice));
  MHIP(m, hipMemset(m->m32, 0, m->n_params * 4));
  MHIP(m, hipMemset(m->v32, 0, m->n_params * 4));
  m->adam_t = 0;
  MHIP(m, update<false>(m, AdamArgs{}));
  MHIP(m, hipStreamSynchronize(m->stream));
  return 0;
}

int ekpnp_mlp_forward(ekpnp_mlp* m, const float* x, int batch, float* y) {
  if (!m || !x || !y) return -1;
  if (batch < 1 || batch > m->cfg.max_batch) return mfail(m, -1, "batch out of range");
  MHIP(m, hipSetDevice(m->cfg.device));
  MHIP(m, forward(m, x, batch, m->L + 1, false));
  MHIP(m, hipMemcpyAsync(y, m->z[m->L + 1], (size_t)batch * m->cfg.n_out * 4, hipMemcpyDeviceToHost, m->stream));
  MHIP(m, hipStreamSynchronize(m->stream));
  return 0;
}

int ekpnp_mlp_loss_grad(ekpnp_mlp* m, const float* x, const float* t, int batch, float* loss, float* grad) {
  if (!m || !x || !t) return -1;
  if (batch < 1 || batch > m->cfg.max_batch) return mfail(m, -1, "batch out of range");
  MHIP(m, hipSetDevice(m->cfg.device));
  int rc = loss_grad(m, x, t, batch);
  if (rc) return rc;
  MHIP(m, hipStreamSynchronize(m->stream));
  if (loss) *loss = loss_of(m, batch);
  if (grad) MHIP(m, hipMemcpy(grad, m->g32, m->n_params * 4, hipMemcpyDeviceToHost));
  return 0;
}

int ekpnp_mlp_set_adam(ekpnp_mlp* m, float beta1, float beta2, float eps, float weight_decay) {
  if (!m) return -1;
  m->b1 = beta1;
  m->b2 = beta2;
  m->eps = eps;
  m->wd = weight_decay;
  return 0;
}

int ekpnp_mlp_train_step(ekpnp_mlp* m, const float* x, const float* t, int batch, float lr, float* loss) {
  if (!m || !x || !t) return -1;
  if (batch < 1 || batch > m->cfg.max_batch) return mfail(m, -1, "batch out of range");
  MHIP(m, hipSetDevice(m->cfg.device));
  int rc = loss_grad(m, x, t, batch);
  if (rc) return rc;
  m->adam_t++;
  const float c1 = 1.0f / (1.0f - std::pow(m->b1, (float)m->adam_t));
  const float c2 = 1.0f / (1.0f - std::pow(m->b2, (float)m->adam_t));
  MHIP(m, update<true>(m, AdamArgs{lr, m->b1, m->b2, m->eps, m->wd, c1, c2}));
  MHIP(m, hipStreamSynchronize(m->stream));
  if (loss) *loss = loss_of(m, batch);
  return 0;
}

}  // extern "C"
