// Learned initial multipliers for SHAKE: inference of the 8 -> 64 -> 64 -> 1
// predictor over the per-constraint feature rows, the step log that
// collects (features, converged multiplier) rows from plain SHAKE, and the
// training kernels (per-block gradient partials of 64 samples, an ordered
// reduction with an Adam step).  The reference has no learned component;
// the model layout is documented beside HD_MLP_* in hd_kernels.h.
//
// Every sum runs in a fixed order (samples within a block, blocks within
// the reduction), so training is bit-reproducible run to run.
#include <hip/hip_runtime.h>

#include "hd_kernels.h"

namespace {

constexpr int F = HD_MLP_IN;
constexpr int H = HD_MLP_H;
constexpr int NS = HD_MLP_SAMPLES;
constexpr int HP = H + 1;  // padded LDS row pitch (conflict-free column reads)
constexpr int GW = 16;      // waves of a gradient block
constexpr int QS = NS / GW; // samples per wave
constexpr int RB = 64;      // partials a reduction thread has in flight

// nu1 columns (0..4) and rho (7) in units of the scale; the couplings
// (5, 6) are O(1) already
__device__ __forceinline__ float mlp_in(int f, float x, float si) {
  return (f == 5 || f == 6) ? x : x * si;
}

// Inference: lane j of a wave is hidden unit j (its rows of W1 and W2 in
// registers) and the wave walks PREDICT_ROWS feature rows: layer 1 per
// lane, layer 2 from layer 1 broadcast through LDS, the output as a
// butterfly sum over the lanes.
constexpr int PREDICT_ROWS = 8;

__global__ __launch_bounds__(256) void k_mlp_predict(const float* __restrict__ P,
                                                     const float* __restrict__ feat, unsigned n,
                                                     float* __restrict__ nu) {
  __shared__ float hsh[4][H];
  const unsigned lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
  float w1[F], w2[H];
#pragma unroll
  for (int f = 0; f < F; ++f) w1[f] = P[HD_MLP_W1 + lane * F + f];
  const float4* w2r = reinterpret_cast<const float4*>(P + HD_MLP_W2 + lane * H);
#pragma unroll
  for (int q = 0; q < H / 4; ++q) {
    float4 v = w2r[q];
    w2[4 * q] = v.x; w2[4 * q + 1] = v.y; w2[4 * q + 2] = v.z; w2[4 * q + 3] = v.w;
  }
  const float b1 = P[HD_MLP_B1 + lane], b2 = P[HD_MLP_B2 + lane], w3 = P[HD_MLP_W3 + lane];
  const float b3 = P[HD_MLP_B3], s = P[HD_MLP_SCALE];
  const float si = s > 0.f ? 1.0f / s : 0.f;
  const unsigned row0 = (blockIdx.x * 4u + wv) * PREDICT_ROWS;
  for (int q = 0; q < PREDICT_ROWS; ++q) {
    unsigned c = row0 + q;
    bool ok = c < n;  // uniform over the wave
    float x[F] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (ok) {
      const float4* xr = reinterpret_cast<const float4*>(feat + (size_t)c * F);
      float4 xa = xr[0], xb = xr[1];
      x[0] = xa.x; x[1] = xa.y; x[2] = xa.z; x[3] = xa.w;
      x[4] = xb.x; x[5] = xb.y; x[6] = xb.z; x[7] = xb.w;
    }
    float acc = b1;
#pragma unroll
    for (int f = 0; f < F; ++f) acc += w1[f] * mlp_in(f, x[f], si);
    hsh[wv][lane] = tanhf(acc);
    __syncthreads();
    acc = b2;
#pragma unroll
    for (int i = 0; i < H; ++i) acc += w2[i] * hsh[wv][i];
    float o = w3 * tanhf(acc);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) o += __shfl_xor(o, off);
    if (ok && lane == 0) nu[c] = x[0] + s * (o + b3);
    __syncthreads();
  }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One wave's 16 x 16 tile (wave / 4, wave % 4) of a 64 x 64 x 64 product in
// f32 on the matrix cores: a(row, k), b(k, col), c = the initial values.
// Lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16] of every step of
// four k and returns rows 16 (wave / 4) + 4 (l / 16) + r, column
// 16 (wave % 4) + l % 16.
template <class A, class B>
__device__ __forceinline__ f32x4 tile64(A a, B b, f32x4 c) {
  const unsigned lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
  const unsigned m = 16u * (wv >> 2) + (lane & 15u), n = 16u * (wv & 3u) + (lane & 15u);
#pragma unroll
  for (unsigned k0 = 0; k0 < (unsigned)H; k0 += 4u) {
    const unsigned k = k0 + (lane >> 4);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a(m, k), b(k, n), c, 0, 0, 0);
  }
  return c;
}
static_assert(NS == 64 && H == 64 && GW == 16, "tile64 covers 64 x 64 with 16 waves");

// One block = 64 samples, 1,024 threads (16 waves).  Forward activations stay
// in LDS and are overwritten in place by their gradients.  The three 64 x
// 64 x 64 products run on the matrix cores in f32: as multiply-adds of
// broadcast LDS reads they kept the LDS busy for 22 us with these 16 waves
// (27 with 4); now 13, a chain of short phases.
__global__ __launch_bounds__(1024) void k_mlp_grad(const float* __restrict__ P,
                                                  const float* __restrict__ X,
                                                  const float* __restrict__ T, uint64_t n,
                                                  uint64_t first, unsigned count, uint64_t mul,
                                                  uint64_t add, float inv_count,
                                                  float* __restrict__ part) {
  __shared__ float w[HD_MLP_NPARAM];
  __shared__ float w2t[H * HP];  // W2 transposed: w2t[i * HP + j] = W2[j][i]
  __shared__ float u[NS][F + 1];
  __shared__ float tgt[NS];      // scaled target, then dL/do
  __shared__ float sq[NS];       // squared residual
  __shared__ float h1[NS * HP];  // tanh of layer 1, then dL/d(pre-activation 1)
  __shared__ float h2[NS * HP];  // tanh of layer 2, then dL/d(pre-activation 2)
  __shared__ unsigned valid[NS];
  const unsigned t = threadIdx.x, lane = t & 63u, wv = t >> 6;
  // the lane's rows (row + r, r < 4) and column of the wave's tile
  const unsigned row = 16u * (wv >> 2) + 4u * (lane >> 4), col = 16u * (wv & 3u) + (lane & 15u);
  for (unsigned i = t; i < HD_MLP_NPARAM; i += 64 * GW) w[i] = P[i];
  for (unsigned e = t; e < H * H; e += 64 * GW) {
    unsigned j = e / H, i = e % H;
    w2t[i * HP + j] = P[HD_MLP_W2 + e];
  }
  const float s = P[HD_MLP_SCALE];
  const float si = s > 0.f ? 1.0f / s : 0.f;
  if (t < NS) {
    unsigned q = blockIdx.x * NS + t;
    unsigned ok = q < count ? 1u : 0u;
    float xr[F] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float tr = 0.f;
    if (ok) {
      uint64_t idx = (mul * (first + q) + add) % n;
      const float4* p4 = reinterpret_cast<const float4*>(X + idx * F);
      float4 xa = p4[0], xb = p4[1];
      xr[0] = xa.x; xr[1] = xa.y; xr[2] = xa.z; xr[3] = xa.w;
      xr[4] = xb.x; xr[5] = xb.y; xr[6] = xb.z; xr[7] = xb.w;
      tr = (T[idx] - xr[0]) * si;
    }
#pragma unroll
    for (int f = 0; f < F; ++f) u[t][f] = mlp_in(f, xr[f], si);
    tgt[t] = tr;
    valid[t] = ok;
  }
  __syncthreads();
  // layer 1: unit = lane, samples wv + 16 q
  {
    float wr[F];
#pragma unroll
    for (int f = 0; f < F; ++f) wr[f] = w[HD_MLP_W1 + lane * F + f];
    float b = w[HD_MLP_B1 + lane];
    for (int q = 0; q < QS; ++q) {
      unsigned sm = wv + (unsigned)GW * q;
      float acc = b;
#pragma unroll
      for (int f = 0; f < F; ++f) acc += wr[f] * u[sm][f];
      h1[sm * HP + lane] = tanhf(acc);
    }
  }
  __syncthreads();
  // layer 2: pre-activation [s][j] = b2[j] + sum_i h1[s][i] W2[j][i]
  {
    const float b = w[HD_MLP_B2 + col];
    const f32x4 d = tile64([&](unsigned s, unsigned i) { return h1[s * HP + i]; },
                           [&](unsigned i, unsigned j) { return w2t[i * HP + j]; },
                           f32x4{b, b, b, b});
#pragma unroll
    for (int r = 0; r < 4; ++r) h2[(row + r) * HP + col] = tanhf(d[r]);
  }
  __syncthreads();
  // output, residual, dL/do
  if (t < NS) {
    float o = w[HD_MLP_B3];
#pragma unroll 8
    for (int j = 0; j < H; ++j) o += w[HD_MLP_W3 + j] * h2[t * HP + j];
    float r = o - tgt[t];
    tgt[t] = valid[t] ? 2.0f * r * inv_count : 0.f;
    sq[t] = valid[t] ? r * r : 0.f;
  }
  __syncthreads();
  float* out = part + (size_t)blockIdx.x * HD_MLP_PSTRIDE;
  if (t < H) {
    float g = 0.f;
#pragma unroll 8
    for (int sm = 0; sm < NS; ++sm) g += tgt[sm] * h2[sm * HP + t];
    out[HD_MLP_W3 + t] = g;
  } else if (t == H) {
    float g = 0.f, l = 0.f;
#pragma unroll 8
    for (int sm = 0; sm < NS; ++sm) { g += tgt[sm]; l += sq[sm]; }
    out[HD_MLP_B3] = g;
    out[HD_MLP_NTRAIN] = l;
  }
  __syncthreads();
  // dL/d(pre-activation 2) in place of h2
  {
    float w3 = w[HD_MLP_W3 + lane];
    for (int q = 0; q < QS; ++q) {
      unsigned sm = wv + (unsigned)GW * q;
      float hv = h2[sm * HP + lane];
      h2[sm * HP + lane] = tgt[sm] * w3 * (1.0f - hv * hv);
    }
  }
  __syncthreads();
  // gW2[j][i] = sum_s D2[s][j] h1[s][i]
  {
    const f32x4 d = tile64([&](unsigned j, unsigned s) { return h2[s * HP + j]; },
                           [&](unsigned s, unsigned i) { return h1[s * HP + i]; },
                           f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int r = 0; r < 4; ++r) out[HD_MLP_W2 + (row + r) * H + col] = d[r];
    if (wv == 0) {
      float g = 0.f;
#pragma unroll 8
      for (int sm = 0; sm < NS; ++sm) g += h2[sm * HP + lane];
      out[HD_MLP_B2 + lane] = g;
    }
  }
  __syncthreads();
  // dL/d(pre-activation 1) in place of h1:
  // [s][i] = sum_j D2[s][j] W2[j][i] (1 - h1[s][i]^2)
  {
    const f32x4 d = tile64([&](unsigned s, unsigned j) { return h2[s * HP + j]; },
                           [&](unsigned j, unsigned i) { return w[HD_MLP_W2 + j * H + i]; },
                           f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float hv = h1[(row + r) * HP + col];
      h1[(row + r) * HP + col] = d[r] * (1.0f - hv * hv);
    }
  }
  __syncthreads();
  // gW1[i][f] = sum_s D1[s][i] u[s][f]: i = lane, f = wv; then gB1
  if (wv < (unsigned)F) {
    float g = 0.f;
#pragma unroll 8
    for (int sm = 0; sm < NS; ++sm) g += h1[sm * HP + lane] * u[sm][wv];
    out[HD_MLP_W1 + lane * F + wv] = g;
  } else if (wv == (unsigned)F) {
    float g = 0.f;
#pragma unroll 8
    for (int sm = 0; sm < NS; ++sm) g += h1[sm * HP + lane];
    out[HD_MLP_B1 + lane] = g;
  }
}

// One parameter per thread, its partials in block order, RB loads in flight
// (one at a time, 64 partials took 27 us of latency; now 6.9).
__global__ void k_mlp_reduce(const float* __restrict__ part, unsigned nb, float* __restrict__ P,
                             float* __restrict__ grad_out, HdAdam adam, int use_adam,
                             double* __restrict__ loss_acc) {
  unsigned p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < HD_MLP_NTRAIN) {
    float g = 0.f;
    unsigned b = 0;
    for (; b + RB <= nb; b += RB) {
      float v[RB];
#pragma unroll
      for (int k = 0; k < RB; ++k) v[k] = part[(size_t)(b + k) * HD_MLP_PSTRIDE + p];
#pragma unroll
      for (int k = 0; k < RB; ++k) g += v[k];
    }
    for (; b < nb; ++b) g += part[(size_t)b * HD_MLP_PSTRIDE + p];
    if (grad_out) grad_out[p] = g;
    if (use_adam) {
      float m = adam.b1 * adam.m[p] + (1.0f - adam.b1) * g;
      float v = adam.b2 * adam.v[p] + (1.0f - adam.b2) * g * g;
      adam.m[p] = m;
      adam.v[p] = v;
      P[p] -= adam.lr_t * m / (sqrtf(v) + adam.eps);
    }
  } else if (p == HD_MLP_NTRAIN && loss_acc) {
    double l = 0.0;
#pragma unroll 8
    for (unsigned b = 0; b < nb; ++b) l += (double)part[(size_t)b * HD_MLP_PSTRIDE + p];
    loss_acc[0] += l;
  }
}

__global__ __launch_bounds__(1024) void k_mlp_scale(const float* __restrict__ x, uint64_t n,
                                                    float* __restrict__ P) {
  __shared__ double red[1024];
  double acc = 0.0;
  uint64_t i = threadIdx.x;
  // 16 rows in flight per thread: 200,003 rows took 116 us one at a time
  for (; i + 15u * 1024u < n; i += 16u * 1024u) {
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = x[(i + 1024u * k) * F];
#pragma unroll
    for (int k = 0; k < 16; ++k) acc += (double)v[k] * (double)v[k];
  }
  for (; i < n; i += 1024) {
    double v = x[i * F];
    acc += v * v;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (unsigned h = 512; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double ms = n ? red[0] / (double)n : 0.0;
    P[HD_MLP_SCALE] = ms > 0.0 ? (float)sqrt(ms) : 1.0f;
  }
}

__global__ __launch_bounds__(1024) void k_shake_log(const float* __restrict__ feat,
                                                    const float* __restrict__ nu, unsigned n,
                                                    float* __restrict__ lx, float* __restrict__ lt,
                                                    unsigned long long* counter,
                                                    unsigned long long cap) {
  // the slot is claimed with a device-scope atomic, so the count never
  // depends on which XCD's cache served the previous step's value
  __shared__ unsigned long long claimed;
  if (threadIdx.x == 0) claimed = atomicAdd(counter, 1ull);
  __syncthreads();
  const unsigned long long slot = claimed;
  if (slot >= cap) return;  // uniform over the block
  const float4* src = reinterpret_cast<const float4*>(feat);
  float4* dst = reinterpret_cast<float4*>(lx + slot * (unsigned long long)n * F);
  for (unsigned i = threadIdx.x; i < n * (F / 4); i += 1024) dst[i] = src[i];
  float* dt = lt + slot * (unsigned long long)n;
  for (unsigned i = threadIdx.x; i < n; i += 1024) dt[i] = nu[i];
}

}  // namespace

void hd_launch_mlp_predict(hipStream_t st, const float* params, const float* feat, unsigned n,
                           float* nu) {
  if (n == 0) return;
  const unsigned rows_per_block = 4u * PREDICT_ROWS;
  hipLaunchKernelGGL(k_mlp_predict, dim3((n + rows_per_block - 1) / rows_per_block), dim3(256), 0,
                     st, params, feat, n, nu);
}

unsigned hd_launch_mlp_grad(hipStream_t st, const float* params, const float* x,
                            const float* t, uint64_t n, uint64_t first, unsigned count,
                            uint64_t mul, uint64_t add, float inv_count, float* partials) {
  unsigned nb = (count + NS - 1) / NS;
  if (nb == 0) return 0;
  hipLaunchKernelGGL(k_mlp_grad, dim3(nb), dim3(64 * GW), 0, st, params, x, t, n, first, count, mul,
                     add, inv_count, partials);
  return nb;
}

void hd_launch_mlp_reduce(hipStream_t st, const float* partials, unsigned nb, float* params,
                          float* grad_out, const HdAdam* adam, double* loss_acc) {
  HdAdam a{};
  if (adam) a = *adam;
  hipLaunchKernelGGL(k_mlp_reduce, dim3((HD_MLP_NTRAIN + 1 + 255) / 256), dim3(256), 0, st,
                     partials, nb, params, grad_out, a, adam ? 1 : 0, loss_acc);
}

void hd_launch_mlp_scale(hipStream_t st, const float* x, uint64_t n, float* params) {
  hipLaunchKernelGGL(k_mlp_scale, dim3(1), dim3(1024), 0, st, x, n, params);
}

void hd_launch_shake_log(hipStream_t st, const float* feat, const float* nu, unsigned n,
                         float* log_x, float* log_t, unsigned long long* counter,
                         unsigned long long cap) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_shake_log, dim3(1), dim3(1024), 0, st, feat, nu, n, log_x, log_t, counter,
                     cap);
}
