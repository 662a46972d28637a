// The learned seed scorer: a 10 -> 32 -> 32 -> 1 MLP with ReLU on BF16 MFMA (FP32 accumulation),
// trained on the seeds the plain search produces (no reference counterpart).
//
//   k_mlp_train        forward, binary cross-entropy and backward, 32 seeds per wave and pass;
//                      gradients accumulate in registers over the passes, one partial row per
//                      workgroup into partial[block][1441]
//   k_mlp_reduce_adam  sums the partial gradients (in an order fixed by the launch: deterministic)
//                      and applies one Adam step to the FP32 master parameters
//   k_mlp_score        forward only: the logit of each seed
//
// Arithmetic (the CPU restatement in oracle/mlp.py follows it step for step):
//   xb  = bf16(x)                      Z1 = xb W1b + b1 (FP32 accumulation)     W1b = bf16(W1)
//   A1b = bf16(relu(Z1))               Z2 = A1b W2b + b2                        W2b = bf16(W2)
//   A2  = relu(Z2)                     z3 = A2 . w3b + b3 (FP32)                w3b = bf16(w3)
//   dz3 = (sigmoid(z3) - y) / N        dZ2 = dz3 w3b * [Z2 > 0],  dZ2b = bf16(dZ2)
//   dW2 = A1b^T dZ2b, db2 = sum dZ2    dA1 = dZ2b W2b^T, dZ1 = dA1 * [Z1 > 0], dZ1b = bf16(dZ1)
//   dW1 = xb^T dZ1b, db1 = sum dZ1     dw3 = sum dz3 A2, db3 = sum dz3
// bf16() rounds FP32 to nearest even (v_cvt_pk_bf16_f32).
//
// Layout. A wave takes 32 seeds; lane l works on seed c = l % 32 and half h = l / 32 of the
// hidden units. The products run transposed (units x seeds) on v_mfma_f32_32x32x16_bf16, whose
// result element v of lane (c, h) is unit 8 (v / 4) + 4 h + v % 4 of seed c. Since the order of a
// contraction is free as long as both operands agree on it, the next product takes its operand
// from the same lane: k-step s (16 units) reads elements 8 s .. 8 s + 7. The forward pass and dA1
// therefore need no LDS and no exchange at all, the weights stay in registers for the life of
// the wave, and only the contractions over seeds (dW1, dW2) turn their operands through the
// wave's own LDS. Before, every operand element was a 2-byte LDS read (64 of them per product),
// the weights were converted again for every 64 seeds, and 1441 partial sums were written per
// 64 seeds and summed by one thread per parameter: 25 + 277 us for 65 536 seeds, 31 us to score
// 240 459.
#include "velo_common.cuh"
#include "velo_kernels.h"

namespace velo {
namespace mlp {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr unsigned rows_per_wave = 32, waves = rows_per_block / rows_per_wave, block_threads = waves * wave_size;

// Eight bf16 in four registers, packed two by two.
union Pack8 {
  uint32_t u[4];
  bf16x8 b;
};

__device__ __forceinline__ uint32_t pack2(float a, float b)
{
  const f32x2 f = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}
__device__ __forceinline__ float bf16_round(float a) { return __uint_as_float(pack2(a, 0.f) << 16); }

// Four consecutive floats, 4-byte aligned (the caller's pointers carry no wider promise).
struct F4 {
  float v[4];
};
__device__ __forceinline__ F4 load4(const float* p)
{
  F4 r;
  __builtin_memcpy(&r, p, sizeof(r));
  return r;
}

__device__ __forceinline__ f32x16 mma(const Pack8& a, const Pack8& b, f32x16 c)
{
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.b, b.b, c, 0, 0, 0);
}

__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A lane's share of the weights of the forward pass: the operands of its row c of W1^T and W2^T
// and the biases and w3 of the 16 units whose results it holds.
struct Forward {
  Pack8 w1, w2[2];
  f32x16 b1, b2;
  float w3[16];
  float b3;

  __device__ __forceinline__ void load(const float* p)
  {
    const unsigned c = lane_id() % 32, h = lane_id() / 32;
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) {
      const unsigned k = 8 * h + 2 * i;
      w1.u[i] = pack2(k < n_inputs ? p[param_w1 + 32 * k + c] : 0.f,
                      k + 1 < n_inputs ? p[param_w1 + 32 * (k + 1) + c] : 0.f);
    }
#pragma unroll
    for (unsigned s = 0; s < 2; ++s)
#pragma unroll
      for (unsigned i = 0; i < 4; ++i) {
        const unsigned k = 16 * s + 8 * (i / 2) + 4 * h + 2 * (i % 2);
        w2[s].u[i] = pack2(p[param_w2 + 32 * k + c], p[param_w2 + 32 * (k + 1) + c]);
      }
#pragma unroll
    for (unsigned q = 0; q < 4; ++q) {
      const unsigned u = 8 * q + 4 * h;
      const F4 x = load4(p + param_b1 + u), y = load4(p + param_b2 + u), z = load4(p + param_w3 + u);
#pragma unroll
      for (unsigned i = 0; i < 4; ++i) {
        b1[4 * q + i] = x.v[i];
        b2[4 * q + i] = y.v[i];
        w3[4 * q + i] = bf16_round(z.v[i]);
      }
    }
    b3 = p[param_b3];
  }
};

// Operand of the first product: features 8 h .. 8 h + 7 of the lane's seed (there are ten).
__device__ __forceinline__ Pack8 load_features(const float* x, size_t row, bool valid)
{
  Pack8 r;
  r.u[0] = r.u[1] = r.u[2] = r.u[3] = 0;
  if (!valid) return r;
  const float* f = x + row * n_inputs;
  if (lane_id() < 32) {
    const F4 a = load4(f), b = load4(f + 4);
    r.u[0] = pack2(a.v[0], a.v[1]);
    r.u[1] = pack2(a.v[2], a.v[3]);
    r.u[2] = pack2(b.v[0], b.v[1]);
    r.u[3] = pack2(b.v[2], b.v[3]);
  }
  else {
    float t[2];
    __builtin_memcpy(t, f + 8, sizeof(t));
    r.u[0] = pack2(t[0], t[1]);
  }
  return r;
}

__device__ __forceinline__ float relu(float z) { return z > 0.f ? z : 0.f; }

// Forward pass of the wave's 32 seeds: A1b (the second product's operands) and Z2 of the lane's
// units, and the logit of its seed (both halves return it).
__device__ __forceinline__ float forward(const Forward& w, const Pack8& xb, Pack8 (&a1)[2], f32x16& z2)
{
  const f32x16 z1 = mma(w.w1, xb, w.b1);
#pragma unroll
  for (unsigned s = 0; s < 2; ++s)
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) a1[s].u[i] = pack2(relu(z1[8 * s + 2 * i]), relu(z1[8 * s + 2 * i + 1]));
  z2 = mma(w.w2[1], a1[1], mma(w.w2[0], a1[0], w.b2));
  float part = 0.f;
#pragma unroll
  for (unsigned v = 0; v < 16; ++v) part += relu(z2[v]) * w.w3[v];
  return part + __shfl_xor(part, 32, wave_size) + w.b3;
}

// Sums a lane's 16 values over the 32 lanes of its half by halving exchanges: 16 exchanges for
// 16 sums. The sum of element v of half h ends in lanes c = 2 v and 2 v + 1 of that half.
__device__ __forceinline__ float half_sums(const float (&a)[16])
{
  float r[8];
  const unsigned c = lane_id() % 32;
  const bool b16 = c & 16, b8 = c & 8, b4 = c & 4, b2 = c & 2;
#pragma unroll
  for (unsigned i = 0; i < 8; ++i) {
    const float keep = b16 ? a[i + 8] : a[i], give = b16 ? a[i] : a[i + 8];
    r[i] = keep + __shfl_xor(give, 16, wave_size);
  }
#pragma unroll
  for (unsigned i = 0; i < 4; ++i) {
    const float keep = b8 ? r[i + 4] : r[i], give = b8 ? r[i] : r[i + 4];
    r[i] = keep + __shfl_xor(give, 8, wave_size);
  }
#pragma unroll
  for (unsigned i = 0; i < 2; ++i) {
    const float keep = b4 ? r[i + 2] : r[i], give = b4 ? r[i] : r[i + 2];
    r[i] = keep + __shfl_xor(give, 4, wave_size);
  }
  const float keep = b2 ? r[1] : r[0], give = b2 ? r[0] : r[1];
  const float s = keep + __shfl_xor(give, 2, wave_size);
  return s + __shfl_xor(s, 1, wave_size);
}

__device__ __forceinline__ unsigned unit(unsigned v) { return 8 * (v / 4) + 4 * (lane_id() / 32) + v % 4; }

// The operands of the contractions over seeds, turned in LDS: [unit or feature][seed]. The row
// stride keeps the 16-byte reads aligned and spreads the rows over the banks.
constexpr unsigned turn_stride = 40;
struct Turned {
  uint16_t x[16 * turn_stride];
  uint16_t a1[32 * turn_stride], dz2[32 * turn_stride], dz1[32 * turn_stride];
};

// Writes the lane's 16 packed values (elements 8 s + 2 i, + 1 of k-step s) to its seed's column.
__device__ __forceinline__ void turn(uint16_t* t, const Pack8 (&a)[2])
{
  const unsigned c = lane_id() % 32;
#pragma unroll
  for (unsigned s = 0; s < 2; ++s)
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) {
      const unsigned u = unit(8 * s + 2 * i);
      t[u * turn_stride + c] = static_cast<uint16_t>(a[s].u[i]);
      t[(u + 1) * turn_stride + c] = static_cast<uint16_t>(a[s].u[i] >> 16);
    }
}

// Operand of a contraction over seeds: seeds 16 s + 8 h .. + 7 of row `row`.
__device__ __forceinline__ Pack8 turned(const uint16_t* t, unsigned row, unsigned s)
{
  Pack8 r;
  const uint4 q = *reinterpret_cast<const uint4*>(t + row * turn_stride + 16 * s + 8 * (lane_id() / 32));
  r.u[0] = q.x;
  r.u[1] = q.y;
  r.u[2] = q.z;
  r.u[3] = q.w;
  return r;
}

} // namespace mlp

using namespace mlp;

// A workgroup of four waves takes 128 seeds per pass and as many passes as the grid leaves it.
// Bound by the latency of one pass (two chained products each way, two turns through LDS); the
// grid is capped at one workgroup per CU so that the partial rows to be summed stay few.
__global__ void __launch_bounds__(block_threads, 1) k_mlp_train(
  const float* features,
  const uint8_t* labels,
  unsigned n,
  float inv_norm,
  const float* params,
  float* partial,
  float* loss_partial)
{
  __shared__ union Lds {
    __align__(16) Turned turned[waves];
    float red[waves][n_params];
  } lds;
  __shared__ float s_loss[waves];
  const unsigned wave = threadIdx.x / wave_size, l = lane_id(), c = l % 32, h = l / 32;
  Turned& t = lds.turned[wave];
  Forward w;
  w.load(params);
  // The operand of dA1^T = W2 dZ2^T: row c of W2, units in the order of the results.
  Pack8 w2r[2];
#pragma unroll
  for (unsigned s = 0; s < 2; ++s)
#pragma unroll
    for (unsigned q = 0; q < 2; ++q) {
      const F4 f = load4(params + param_w2 + 32 * c + 16 * s + 8 * q + 4 * h);
      w2r[s].u[2 * q] = pack2(f.v[0], f.v[1]);
      w2r[s].u[2 * q + 1] = pack2(f.v[2], f.v[3]);
    }
  f32x16 zero;
  float db1[16], db2[16], dw3[16];
#pragma unroll
  for (unsigned v = 0; v < 16; ++v) zero[v] = db1[v] = db2[v] = dw3[v] = 0.f;
  f32x16 dw1 = zero, dw2 = zero;
  float db3 = 0.f, loss = 0.f;
  for (size_t base = (size_t) blockIdx.x * rows_per_block; base < n; base += (size_t) gridDim.x * rows_per_block) {
    const size_t row = base + wave * rows_per_wave + c;
    const bool valid = row < n;
    const Pack8 xb = load_features(features, row, valid);
    const float y = valid ? static_cast<float>(labels[row]) : 0.f;
    Pack8 a1[2], dz2b[2], dz1b[2];
    f32x16 z2;
    const float z3 = forward(w, xb, a1, z2);
    const float p = 1.f / (1.f + expf(-z3));
    const float dz3 = valid ? (p - y) * inv_norm : 0.f;
    // Loss of the row (binary cross-entropy from the logit, stable form), counted once per row.
    if (valid && h == 0) {
      loss += fmaxf(z3, 0.f) - z3 * y + log1pf(expf(-fabsf(z3)));
      db3 += dz3;
    }
    float dz2[16];
#pragma unroll
    for (unsigned v = 0; v < 16; ++v) {
      dz2[v] = z2[v] > 0.f ? dz3 * w.w3[v] : 0.f;
      db2[v] += dz2[v];
      dw3[v] += dz3 * relu(z2[v]);
    }
#pragma unroll
    for (unsigned s = 0; s < 2; ++s)
#pragma unroll
      for (unsigned i = 0; i < 4; ++i) dz2b[s].u[i] = pack2(dz2[8 * s + 2 * i], dz2[8 * s + 2 * i + 1]);
    const f32x16 da1 = mma(w2r[1], dz2b[1], mma(w2r[0], dz2b[0], zero));
    // [Z1 > 0] is [a1b != 0]: rounding a positive FP32 to bf16 gives zero only below its
    // smallest subnormal, where the product's own operand is zero as well.
#pragma unroll
    for (unsigned s = 0; s < 2; ++s)
#pragma unroll
      for (unsigned i = 0; i < 4; ++i) {
        const unsigned v = 8 * s + 2 * i;
        const float d0 = a1[s].u[i] & 0xFFFFu ? da1[v] : 0.f, d1 = a1[s].u[i] >> 16 ? da1[v + 1] : 0.f;
        db1[v] += d0;
        db1[v + 1] += d1;
        dz1b[s].u[i] = pack2(d0, d1);
      }
    wave_sync(); // the last pass's reads are done
    turn(t.a1, a1);
    turn(t.dz2, dz2b);
    turn(t.dz1, dz1b);
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) {
      t.x[(8 * h + 2 * i) * turn_stride + c] = static_cast<uint16_t>(xb.u[i]);
      t.x[(8 * h + 2 * i + 1) * turn_stride + c] = static_cast<uint16_t>(xb.u[i] >> 16);
    }
    wave_sync();
#pragma unroll
    for (unsigned s = 0; s < 2; ++s) {
      Pack8 xt = turned(t.x, c % 16, s);
      if (c >= 16) xt.u[0] = xt.u[1] = xt.u[2] = xt.u[3] = 0; // rows beyond the padded features
      dw2 = mma(turned(t.a1, c, s), turned(t.dz2, c, s), dw2);
      dw1 = mma(xt, turned(t.dz1, c, s), dw1);
    }
  }
  __syncthreads(); // every wave is done with its turned operands: the same LDS takes the sums
  float* g = lds.red[wave];
#pragma unroll
  for (unsigned v = 0; v < 16; ++v) {
    g[param_w2 + 32 * unit(v) + c] = dw2[v];
    if (unit(v) < n_inputs) g[param_w1 + 32 * unit(v) + c] = dw1[v];
  }
  const float s1 = half_sums(db1), s2 = half_sums(db2), s3 = half_sums(dw3);
  if (c % 2 == 0) {
    const unsigned u = unit(c / 2);
    g[param_b1 + u] = s1;
    g[param_b2 + u] = s2;
    g[param_w3 + u] = s3;
  }
#pragma unroll
  for (unsigned d = 32; d > 0; d >>= 1) {
    loss += __shfl_xor(loss, d, wave_size);
    db3 += __shfl_xor(db3, d, wave_size);
  }
  if (l == 0) {
    g[param_b3] = db3;
    s_loss[wave] = loss;
  }
  __syncthreads();
  // Sum of the waves in wave order.
  for (unsigned q = threadIdx.x; q < n_params; q += blockDim.x) {
    float s = lds.red[0][q];
#pragma unroll
    for (unsigned k = 1; k < waves; ++k) s += lds.red[k][q];
    partial[(size_t) blockIdx.x * n_params + q] = s;
  }
  if (threadIdx.x == 0) {
    float s = s_loss[0];
#pragma unroll
    for (unsigned k = 1; k < waves; ++k) s += s_loss[k];
    loss_partial[blockIdx.x] = s;
  }
}

// The gradient of 64 parameters per workgroup (the last workgroup takes the loss as well): lane q
// of wave k sums the partial rows k, k + 16, ... of its parameter, the waves' sums are added in
// wave order, and Adam with bias correction follows (step = 1-based count of this update; lr = 0:
// gradient only). 16 waves because a chain of up to 256 dependent adds behind one load each was
// what the step spent its time on.
constexpr unsigned reduce_waves = 16;
__global__ void __launch_bounds__(reduce_waves* wave_size) k_mlp_reduce_adam(
  const float* partial,
  const float* loss_partial,
  unsigned n_blocks,
  float* params,
  float* m,
  float* v,
  float* grad_out,
  float* loss_out,
  float lr,
  float beta1,
  float beta2,
  float eps,
  unsigned step)
{
  __shared__ float red[reduce_waves][wave_size];
  const unsigned k = threadIdx.x / wave_size, l = lane_id();
  const bool losses = blockIdx.x + 1 == gridDim.x;
  const unsigned q = blockIdx.x * wave_size + l;
  float s = 0.f;
  if (losses) {
    for (unsigned b = threadIdx.x; b < n_blocks; b += blockDim.x) s += loss_partial[b];
  }
  else if (q < n_params) {
#pragma unroll 8
    for (unsigned b = k; b < n_blocks; b += reduce_waves) s += partial[(size_t) b * n_params + q];
  }
  red[k][l] = s;
  __syncthreads();
  if (k != 0) return;
  float gsum = red[0][l];
#pragma unroll
  for (unsigned w = 1; w < reduce_waves; ++w) gsum += red[w][l];
  if (losses) {
#pragma unroll
    for (unsigned d = 32; d > 0; d >>= 1) gsum += __shfl_xor(gsum, d, wave_size);
    if (l == 0 && loss_out) *loss_out = gsum;
    return;
  }
  if (q >= n_params) return;
  if (grad_out) grad_out[q] = gsum;
  if (lr == 0.f) return;
  const float mq = beta1 * m[q] + (1.f - beta1) * gsum;
  const float vq = beta2 * v[q] + (1.f - beta2) * gsum * gsum;
  m[q] = mq;
  v[q] = vq;
  const float mh = mq / (1.f - powf(beta1, static_cast<float>(step)));
  const float vh = vq / (1.f - powf(beta2, static_cast<float>(step)));
  params[q] -= lr * mh / (sqrtf(vh) + eps);
}

// Waves walk over groups of 32 seeds; the weights are read once per wave.
__global__ void __launch_bounds__(block_threads) k_mlp_score(
  const float* features,
  unsigned n,
  const float* params,
  float* logits)
{
  Forward w;
  w.load(params);
  const unsigned c = lane_id() % 32;
  for (size_t base = (size_t) blockIdx.x * rows_per_block; base < n; base += (size_t) gridDim.x * rows_per_block) {
    const size_t row = base + threadIdx.x / wave_size * rows_per_wave + c;
    const bool valid = row < n;
    Pack8 a1[2];
    f32x16 z2;
    const float z3 = forward(w, load_features(features, row, valid), a1, z2);
    if (valid && lane_id() < 32) logits[row] = z3;
  }
}

hipError_t launch_mlp_train(
  const float* features,
  const uint8_t* labels,
  unsigned n,
  float inv_norm,
  const float* params,
  float* partial,
  float* loss_partial,
  hipStream_t s)
{
  if (!n) return hipSuccess;
  hipLaunchKernelGGL(
    k_mlp_train, dim3(mlp_blocks(n)), dim3(block_threads), 0, s, features, labels, n, inv_norm, params, partial,
    loss_partial);
  return hipGetLastError();
}

hipError_t launch_mlp_reduce_adam(
  const float* partial,
  const float* loss_partial,
  unsigned n_blocks,
  float* params,
  float* m,
  float* v,
  float* grad_out,
  float* loss_out,
  float lr,
  unsigned step,
  hipStream_t s)
{
  hipLaunchKernelGGL(
    k_mlp_reduce_adam, dim3((n_params + wave_size - 1) / wave_size + 1), dim3(reduce_waves * wave_size), 0, s, partial,
    loss_partial, n_blocks, params, m, v, grad_out, loss_out, lr, 0.9f, 0.999f, 1e-8f, step);
  return hipGetLastError();
}

hipError_t launch_mlp_score(const float* features, unsigned n, const float* params, float* logits, hipStream_t s)
{
  if (!n) return hipSuccess;
  // Up to four workgroups per CU: enough waves to hide the loads, and from there on each wave
  // reads the weights once for several groups.
  const unsigned grid = min((n - 1) / rows_per_block + 1, 4 * 256u);
  hipLaunchKernelGGL(k_mlp_score, dim3(grid), dim3(block_threads), 0, s, features, n, params, logits);
  return hipGetLastError();
}

} // namespace velo
