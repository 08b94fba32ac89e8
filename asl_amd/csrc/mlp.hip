// Training kernels of the closure network (7-32-32-1, ReLU; parameter
// layout and model in closure.hpp): forward + backward of a batch with
// deterministic per-workgroup gradient sums, and the reduction over
// workgroups with the Adam update.
//
// Loss: half the mean squared error over the batch.  Adam: Kingma & Ba,
// "Adam: A Method for Stochastic Optimization" (ICLR 2015), Algorithm 1.
// All FP32 except the sums over wavefronts and over workgroups (FP64, a workgroup's
// own sum stored as FP32 between the two).
#include <hip/hip_runtime.h>

#include "closure.hpp"
#include "mlp.hpp"

namespace aslhip {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

// splitmix64 finaliser (S. Vigna, public domain): sample indices of a batch.
__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__device__ __forceinline__ f32x16_t mfma(float a, float b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Rows of a tile in LDS: 32 values and 4 of padding (16-byte rows, other banks).
constexpr int LROW = 36;
constexpr int NWAVE = MLP_GRAD_BLOCK / 64;

// The row of D[row][lane % 32] that register r of v_mfma_f32_32x32x2f32's
// result holds in half h of the wavefront.
__device__ __forceinline__ constexpr int drow(int r, int h) { return 8 * (r / 4) + 4 * h + r % 4; }

// The hidden unit at row q of a layer's products: the rows are arranged so that
// register r in half h holds unit 2 r + h.
__device__ __forceinline__ int unit_at(int q) { return 2 * (4 * (q >> 3) + (q & 3)) + ((q >> 2) & 1); }

// The sample within the batch of a lane's column: 32-bit unsigned, since the last
// workgroup of a batch near 2^31 goes past it (as a signed number it would count as
// one before the first sample, and be read).
__device__ __host__ constexpr unsigned sample_of(unsigned block, int spw, int it, int w, int col) {
  return ((block * static_cast<unsigned>(spw) + static_cast<unsigned>(it)) * NWAVE + static_cast<unsigned>(w)) * 32u +
         static_cast<unsigned>(col);
}
constexpr unsigned MAX_BATCH = 0x7fffffffu;
static_assert(sample_of((MAX_BATCH - 1) / (64 * NWAVE), 2, 1, NWAVE - 1, 31) >= MAX_BATCH,
              "a lane past the largest batch must not count as one of its samples");

// Forward and backward on the FP32 matrix instructions: every wavefront takes
// 32 samples at a time, one per column, as six products
//   H1 = relu(W1 x + b1),   H2 = relu(W2 H1 + b2),   y = w3 H2 + b3,
//   dH1 = W2^T dH2 [H1 > 0],   gW2 += dH2 H1^T,   (gW1, gb1) += dH1 (x, 1)^T.
// v_mfma_f32_32x32x2f32 takes A[l % 32][l / 32] and B[l / 32][l % 32] from lane
// l; with the units in unit_at's order k-step r uses units 2 r and 2 r + 1, which
// is how the previous product left its result: layers chain without moving data.
// It also adds every sum over units up in index order, biases first, which are
// the bits of a chain of fma on the vector ALUs (1.6 million values of gradients
// of single samples: all equal).  In another order a unit whose input lies within
// a rounding of zero may switch sides (a third of the H2 differed in their last
// bit, and some training runs by 2e-6).
// The two gradients contract over samples; their operands go through LDS once,
// transposed.  g_b2, g_w3, g_b3 and the loss are sums per lane, added up at the
// end.  Sums of at most 64 samples (SPW blocks of 32) are kept in FP32, as few
// roundings as 64-sample blocks on the vector ALUs had; the four wavefronts' are
// added in FP64 and stored as the workgroup's FP32 sum, which k_mlp_reduce adds in
// FP64.
//
// Bound by latency: 16384 samples are 118 MFLOP (1 us of the matrix cores) in
// one block per wavefront, 84 matrix instructions of 64 cycles in a chain of 68 (gW2
// and gW1 are independent of each other); before, on
// the vector ALUs with the weight products summed from LDS one sample after the
// other, 91 us.  20 training steps of 16384 samples: 3370 -> 300 us with the
// reduction below (270 without the order of the sums).
template <int SPW>
__global__ __launch_bounds__(MLP_GRAD_BLOCK) void k_mlp_grad(const MlpGradArgs a) {
  __shared__ __attribute__((aligned(16))) float tile[NWAVE][3][CL_H * LROW];  // dH2, H1, dH1: [unit][sample]
  __shared__ __attribute__((aligned(16))) float xt[NWAVE][8 * LROW];          // x': [input][sample]
  const int w = static_cast<int>(threadIdx.x) >> 6, l = static_cast<int>(threadIdx.x) & 63;
  const int col = l & 31, half = l >> 5;
  float *dh2t = tile[w][0], *h1t = tile[w][1], *dh1t = tile[w][2], *x8 = xt[w];
  const float *p = a.p;

  // weights in operand order
  float w1[4], w2[16], w2t[16], b1[16], b2[16], w3[16];
  const int unit = unit_at(col);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int in = 2 * k + half;
    w1[k] = in < CL_NIN ? p[CL_W1 + unit * CL_NIN + in] : 0.f;
  }
  auto every_other = [&](const float *q, float (&d)[16]) {  // q[2 r + half]
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const f4 v = *reinterpret_cast<const f4 *>(q + 4 * i);
      d[2 * i] = half ? v[1] : v[0];
      d[2 * i + 1] = half ? v[3] : v[2];
    }
  };
  static_assert(CL_W2 % 4 == 0 && CL_B1 % 4 == 0 && CL_B2 % 4 == 0 && CL_W3 % 4 == 0, "16-byte loads");
  every_other(p + CL_W2 + unit * CL_H, w2);
  every_other(p + CL_B1, b1);
  every_other(p + CL_B2, b2);
  every_other(p + CL_W3, w3);
#pragma unroll
  for (int r = 0; r < 16; ++r) w2t[r] = p[CL_W2 + (2 * r + half) * CL_H + unit];
  const float b3 = p[CL_B3];

  f32x16_t gw2 = {}, gw1 = {};
  float gb2[16], gw3[16], gb3 = 0.f, loss = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) gb2[r] = gw3[r] = 0.f;

#pragma unroll 1
  for (int it = 0; it < SPW; ++it) {
    // this column's sample within the batch
    const unsigned k = sample_of(blockIdx.x, SPW, it, w, col);
    const bool live = k < static_cast<unsigned>(a.count);
    long long s = 0;
    if (live)
      s = a.seed ? static_cast<long long>(mix64(a.seed + (static_cast<unsigned long long>(k) + 1ull) *
                                                            0x9E3779B97F4A7C15ull) %
                                          static_cast<unsigned long long>(a.n))
                 : a.first + k;
    float x[4];  // inputs half, 2 + half, 4 + half, 6 + half (the eighth: 1)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int in = 2 * j + half;
      x[j] = in == CL_NIN ? 1.f : (live ? a.x[s * CL_NIN + in] : 0.f);
    }
    const float t = live ? a.t[s] : 0.f;

    f32x16_t h1;
#pragma unroll
    for (int r = 0; r < 16; ++r) h1[r] = b1[r];
#pragma unroll
    for (int j = 0; j < 4; ++j) h1 = mfma(w1[j], x[j], h1);
    float m1[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      m1[r] = h1[r] > 0.f ? 1.f : 0.f;
      h1[r] = h1[r] > 0.f ? h1[r] : 0.f;
    }
    f32x16_t h2;
#pragma unroll
    for (int r = 0; r < 16; ++r) h2[r] = b2[r];
#pragma unroll
    for (int r = 0; r < 16; ++r) h2 = mfma(w2[r], h1[r], h2);
    // y as row 0 and, for the upper half, row 4 of one more product
    f32x16_t yr;
#pragma unroll
    for (int r = 0; r < 16; ++r) yr[r] = b3;
#pragma unroll
    for (int r = 0; r < 16; ++r) yr = mfma((col & ~4) == 0 ? w3[r] : 0.f, h2[r] > 0.f ? h2[r] : 0.f, yr);
    const float y = yr[0];
    const float res = live ? y - t : 0.f;
    const float dy = res * a.inv_batch;
    f32x16_t d1 = {};
    float d2[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float v = h2[r] > 0.f ? h2[r] : 0.f;
      d2[r] = (h2[r] > 0.f ? 1.f : 0.f) * (dy * w3[r]);
      gw3[r] = __builtin_fmaf(dy, v, gw3[r]);
      gb2[r] += d2[r];
    }
    gb3 += dy;
    loss += 0.5f * res * res;
#pragma unroll
    for (int r = 0; r < 16; ++r) d1 = mfma(w2t[r], d2[r], d1);

    if (SPW > 1 && it) __syncthreads();  // the last block's operands have been read
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int o = (2 * r + half) * LROW + col;
      dh2t[o] = d2[r];
      h1t[o] = h1[r];
      dh1t[o] = d1[r] * m1[r];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) x8[(2 * j + half) * LROW + col] = live ? x[j] : 0.f;
    __syncthreads();
    // samples 16 half .. 16 half + 15 of unit (input) col; k-step i pairs samples i and 16 + i
    const f4 *ra = reinterpret_cast<const f4 *>(dh2t + col * LROW + 16 * half);
    const f4 *rb = reinterpret_cast<const f4 *>(h1t + col * LROW + 16 * half);
    const f4 *rc = reinterpret_cast<const f4 *>(dh1t + col * LROW + 16 * half);
    const f4 *rx = reinterpret_cast<const f4 *>(x8 + (col & 7) * LROW + 16 * half);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f4 va = ra[i], vb = rb[i], vc = rc[i];
      f4 vx = rx[i];
      if (col >= 8) vx = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        gw2 = mfma(va[j], vb[j], gw2);
        gw1 = mfma(vc[j], vx[j], gw1);
      }
    }
  }

  // sums over the lanes of a column block: transposed through LDS, each lane adds 16, then the two halves
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int o = (2 * r + half) * LROW + col;
    dh2t[o] = gb2[r];
    h1t[o] = gw3[r];
  }
  x8[col] = gb3;  // both halves hold the same sample's dy and loss
  x8[LROW + col] = loss;
  __syncthreads();
  float sb2 = 0.f, sw3 = 0.f, sl = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    sb2 += dh2t[col * LROW + 16 * half + i];
    sw3 += h1t[col * LROW + 16 * half + i];
    sl += x8[(col & 1) * LROW + 16 * half + i];
  }
  sb2 += __shfl_xor(sb2, 32);
  sw3 += __shfl_xor(sw3, 32);
  sl += __shfl_xor(sl, 32);
  __syncthreads();
  // this wavefront's sums in parameter order
  static_assert(3 * CL_H * LROW >= CL_NPARAM + 1, "the tiles hold one set of parameters");
  float *out = tile[w][0];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int o = drow(r, half);
    out[CL_W2 + o * CL_H + col] = gw2[r];
    if (col < CL_NIN) out[CL_W1 + o * CL_NIN + col] = gw1[r];
    if (col == CL_NIN) out[CL_B1 + o] = gw1[r];
  }
  if (half == 0) {
    out[CL_B2 + col] = sb2;
    out[CL_W3 + col] = sw3;
    if (col < 2) out[CL_B3 + col] = sl;  // g_b3, then the loss
  }
  __syncthreads();
  float *dst = a.partial + static_cast<long long>(blockIdx.x) * MLP_PSTRIDE;
  for (int q = static_cast<int>(threadIdx.x); q <= CL_NPARAM; q += MLP_GRAD_BLOCK) {
    double acc = 0.;
#pragma unroll
    for (int v = 0; v < NWAVE; ++v) acc += static_cast<double>(tile[v][0][q]);
    dst[q] = static_cast<float>(acc);
  }
}

// Parameters per workgroup of the reduction, and the slices that share the
// partial sums of one.
constexpr int RP = 32, RS = 256 / RP;

// grad[q] = sum over workgroups of partial[b][q] (FP64; slice s takes b = s,
// s + RS, ..., then the slices in order); the last entry is the loss
// (0.5 * sum r^2 / count).  ADAM: the parameter's update follows at once,
// which saves a launch per step.  Eight slices of 32 parameters per workgroup
// read whole 128-byte lines; with one thread per parameter, 16384 samples'
// partials took 61 us.
template <bool ADAM>
__global__ __launch_bounds__(256) void k_mlp_reduce(const float *partial, int nblocks, double inv_count, float *grad,
                                                    double *loss, float *p, float *m, float *v, AdamArgs a) {
  __shared__ double sh[RS][RP];
  const int i = static_cast<int>(threadIdx.x) % RP, s = static_cast<int>(threadIdx.x) / RP;
  const int q = static_cast<int>(blockIdx.x) * RP + i;
  double acc = 0.;
  if (q <= CL_NPARAM) {
#pragma unroll 8
    for (int b = s; b < nblocks; b += RS)
      acc += static_cast<double>(partial[static_cast<long long>(b) * MLP_PSTRIDE + q]);
  }
  sh[s][i] = acc;
  __syncthreads();
  if (s != 0 || q > CL_NPARAM) return;
#pragma unroll
  for (int k = 1; k < RS; ++k) acc += sh[k][i];
  if (q == CL_NPARAM) {
    *loss = acc * inv_count;
    return;
  }
  const float gq = static_cast<float>(acc);
  grad[q] = gq;
  if constexpr (ADAM) {
    const float mq = __builtin_fmaf(a.beta1, m[q], (1.f - a.beta1) * gq);
    const float vq = __builtin_fmaf(a.beta2, v[q], (1.f - a.beta2) * gq * gq);
    m[q] = mq;
    v[q] = vq;
    const float mhat = mq / a.bc1;
    const float vhat = vq / a.bc2;
    p[q] = p[q] - a.lr * mhat / (__builtin_sqrtf(vhat) + a.eps);
  }
}

}  // namespace

// One block of 32 samples per wavefront while that leaves CUs without work
// (256 workgroups of 128 samples), else two: half the partial sums.
int mlp_grad_blocks(int count) {
  const int per = count <= 256 * 32 * NWAVE ? 32 * NWAVE : 64 * NWAVE;
  return static_cast<int>((static_cast<long long>(count) + per - 1) / per);
}

hipError_t launch_mlp_grad(const MlpGradArgs &a, hipStream_t s) {
  const dim3 grid(mlp_grad_blocks(a.count)), block(MLP_GRAD_BLOCK);
  if (a.count <= 256 * 32 * NWAVE)
    hipLaunchKernelGGL(k_mlp_grad<1>, grid, block, 0, s, a);
  else
    hipLaunchKernelGGL(k_mlp_grad<2>, grid, block, 0, s, a);
  return hipGetLastError();
}

hipError_t launch_mlp_reduce(const float *partial, int nblocks, double inv_count, float *grad, double *loss,
                             hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_reduce<false>, dim3((CL_NPARAM + RP) / RP), dim3(256), 0, s, partial, nblocks, inv_count,
                     grad, loss, static_cast<float *>(nullptr), static_cast<float *>(nullptr),
                     static_cast<float *>(nullptr), AdamArgs{});
  return hipGetLastError();
}

hipError_t launch_mlp_reduce_adam(const float *partial, int nblocks, double inv_count, float *grad, double *loss,
                                  float *p, float *m, float *v, const AdamArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_reduce<true>, dim3((CL_NPARAM + RP) / RP), dim3(256), 0, s, partial, nblocks, inv_count,
                     grad, loss, p, m, v, a);
  return hipGetLastError();
}

}  // namespace aslhip
