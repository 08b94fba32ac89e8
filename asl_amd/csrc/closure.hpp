// Learned closure: per-cell relaxation-time correction from a small network.
//
// An extension with no counterpart in ASL.  Inputs (7 per cell): the
// non-equilibrium second moments of the pre-collision populations,
//   Pi_ab = sum_i w_i c_ia c_ib f_i - (rho/3 delta_ab + m_a m_b / rho),
// for ab = xx, yy, zz, xy, xz, yz, and rho - 1.  Network 7-32-32-1, ReLU
// after both hidden layers, BF16-rounded parameters evaluated in FP32:
//   xn = (x - mu) * sc,  h1 = relu(W1 xn + b1),  h2 = relu(W2 h1 + b2),
//   y = w3 . h2 + b3,    tau = max(tau0 + y * out, 1/2 + (tau0 - 1/2) / 2),  w = 1 / tau
// (the correction may lower the viscosity by at most half).
// Every sum is an fma chain in index order (the CPU oracle evaluates the same
// chain, so results agree bit for bit).
#pragma once

#include <cstddef>

#include "lattice_consts.hpp"

namespace aslhip {

constexpr int CL_NIN = 7, CL_H = 32, CL_NPARAM = 1345;
constexpr int CL_W1 = 0, CL_B1 = 224, CL_W2 = 256, CL_B2 = 1280, CL_W3 = 1312, CL_B3 = 1344;

// Closure parameters as the step kernel reads them (device memory).  The
// matrix-core path reads its operands pre-arranged in lane order (filled by
// pack_closure from p): one 8-byte load per BF16 A operand and 16-byte loads
// for the biases and output weights, instead of one load and one conversion
// per element.
struct ClosureParams {
  float p[CL_NPARAM];  // BF16-rounded weights and biases
  float mu[CL_NIN], sc[CL_NIN];
  float out;           // scale of the relaxation-time correction
  alignas(16) unsigned long long a1[64];  // lane l: W1'[l % 32][4 (l / 32) + j], j < 4 (BF16 x 4)
  unsigned long long a2[4][64];           // k-block kb, lane l: W2[l % 32][8 kb + 4 (l / 32) + j]
  alignas(16) float b2[2][16];            // half h, register r: b2[8 (r / 4) + 4 h + r % 4]
  alignas(16) float w3[2][16];            // half h, register r: w3[8 (r / 4) + 4 h + r % 4]
};

// The part of ClosureParams from p[CL_B3] on: what the matrix-core path reads,
// copied to LDS once per workgroup.
struct alignas(16) ClosureLds {
  float b3, mu[CL_NIN], sc[CL_NIN], out;
  unsigned long long a1[64], a2[4][64];
  float b2[2][16], w3[2][16];
};
static_assert(offsetof(ClosureParams, w3) + sizeof(ClosureParams::w3) == CL_B3 * sizeof(float) + sizeof(ClosureLds) &&
                  offsetof(ClosureParams, a1) == CL_B3 * sizeof(float) + offsetof(ClosureLds, a1),
              "ClosureLds mirrors the end of ClosureParams");

// BF16 bits of an already BF16-rounded float (the top half of its bits).
inline unsigned long long bf16x4_pack(const float *v) {
  unsigned long long r = 0;
  for (int j = 0; j < 4; ++j) {
    unsigned u;
    __builtin_memcpy(&u, &v[j], 4);
    r |= static_cast<unsigned long long>(u >> 16) << (16 * j);
  }
  return r;
}

// Arranges the matrix-core operands of c.p (already BF16-rounded).
inline void pack_closure(ClosureParams &c) {
  for (int l = 0; l < 64; ++l) {
    const int col = l & 31, half = l >> 5;
    float v[4];
    for (int j = 0; j < 4; ++j) {
      const int k = 4 * half + j;
      v[j] = k < CL_NIN ? c.p[CL_W1 + col * CL_NIN + k] : c.p[CL_B1 + col];
    }
    c.a1[l] = bf16x4_pack(v);
    for (int kb = 0; kb < 4; ++kb) {
      for (int j = 0; j < 4; ++j) v[j] = c.p[CL_W2 + col * CL_H + 8 * kb + 4 * half + j];
      c.a2[kb][l] = bf16x4_pack(v);
    }
  }
  for (int h = 0; h < 2; ++h)
    for (int r = 0; r < 16; ++r) {
      c.b2[h][r] = c.p[CL_B2 + 8 * (r / 4) + 4 * h + (r % 4)];
      c.w3[h][r] = c.p[CL_W3 + 8 * (r / 4) + 4 * h + (r % 4)];
    }
}

template <int Q>
__device__ __forceinline__ void closure_features(const float (&f)[Q], float r, const float (&m)[3], float (&x)[7]) {
  constexpr int A[6] = {0, 1, 2, 0, 0, 1}, B[6] = {0, 1, 2, 1, 2, 2};
  float mr[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) mr[d] = m[d] / r;
  const float third = 1.f / 3.f;
#pragma unroll
  for (int p = 0; p < 6; ++p) {
    float acc = 0.f;
    bool first = true;
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      const int cc = Lat<Q>::c[j][A[p]] * Lat<Q>::c[j][B[p]];
      if (cc == 0) continue;
      const float wcc = static_cast<float>(Lat<Q>::w(j) * cc);
      acc = first ? f[j] * wcc : __builtin_fmaf(f[j], wcc, acc);
      first = false;
    }
    const float t = A[p] == B[p] ? __builtin_fmaf(m[A[p]], mr[B[p]], r * third) : m[A[p]] * mr[B[p]];
    x[p] = acc - t;
  }
  x[6] = r - 1.f;
}

__device__ __forceinline__ float closure_relax(float y, float out, float tau0) {
  const float tau = tau0 + y * out;
  const float lo = 0.5f + 0.5f * (tau0 - 0.5f);
  return 1.f / (tau < lo ? lo : tau);
}

typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// Two values rounded to the nearest BF16 (ties to even), lo in the low half:
// one v_cvt_pk_bf16_f32.
__device__ __forceinline__ unsigned bf16_pair(float lo, float hi) {
  const f32x2_t f = {lo, hi};
  const bf16x2_t b = __builtin_convertvector(f, bf16x2_t);
  unsigned u;
  __builtin_memcpy(&u, &b, 4);
  return u;
}

// x > 0 ? x : 0 in one instruction: the median of x, 0 and inf (infinity, from
// a register: the compiler turns a known one into a maximum, which needs a
// second instruction to quiet signalling NaNs).  NaN gives the smaller of the
// others, 0, as the comparison does.
__device__ __forceinline__ float relu(float x, float inf) { return __builtin_amdgcn_fmed3f(x, 0.f, inf); }

// Exchanges the upper half-wavefront of a with the lower one of b.
__device__ __forceinline__ void swap_halves(unsigned &a, unsigned &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// The network on the matrix cores: every lane of the wavefront brings its own
// cell's inputs, all 64 lanes must be active.  Two column blocks of 32 cells
// (cells 0-31, 32-63 of the wavefront) go through
//   H1^T = relu(W1' xn')   one 32x32x8 BF16 MFMA (xn' = (xn, 1), W1' = (W1, b1)),
//   H2^T = relu(W2 H1^T + b2)   four 32x32x8 BF16 MFMAs, FP32 accumulation,
//   y = w3 . h2 + b3       FP32: each lane sums the 16 hidden units it holds,
//                          the two halves of the wavefront are added.
// v_mfma_f32_32x32x8bf16_1k operand layout (lane l): A[l % 32][4 (l / 32) + j],
// B[4 (l / 32) + j][l % 32], j < 4; result register r holds
// D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32] — the layout the next layer's B
// operand needs for k-block r / 4, so layers chain without shuffles.
//
// Beside the 10 MFMAs this is vector work (a wavefront instruction takes 4
// cycles) that has to stay in the shadow of the step's memory traffic: paired
// conversions, one instruction per relu, v_permlane32_swap for the exchange of
// halves.  The parameters come from LDS; loads of them from memory were waited
// for one layer after the other.  Even periodic step: 1003 -> 856 instructions
// with the rare paths, 66 -> 61 us for 128^3 FP32, and 52.5 (6.1 TB/s; the plain
// step 50) with the registers it asks for (97 to 103, 4 waves per SIMD):
// held to 96, it spilled 8.
__device__ __forceinline__ float closure_y_mfma(const float (&x)[7], const ClosureLds &c) {
  const int l = static_cast<int>(threadIdx.x) & 63;
  const int half = l >> 5;
  // own inputs as BF16 pairs: (x0, x1), (x2, x3), (x4, x5), (x6, 1.0 = the bias column of W1')
  float xn[8];
#pragma unroll
  for (int j = 0; j < 7; ++j) xn[j] = (x[j] - c.mu[j]) * c.sc[j];
  xn[7] = 1.f;
  // Column block cb holds cells 32 cb + col; a lane supplies inputs 4 half ..
  // 4 half + 3 of its column.  Inputs 0 .. 3 (in[cb = 0] before the exchange)
  // of the upper cells trade places with inputs 4 .. 7 of the lower ones.
  unsigned in[2][2];
#pragma unroll
  for (int p = 0; p < 4; ++p) in[p / 2][p % 2] = bf16_pair(xn[2 * p], xn[2 * p + 1]);
  swap_halves(in[0][0], in[1][0]);
  swap_halves(in[0][1], in[1][1]);
  bf16x4_t a1;
  __builtin_memcpy(&a1, &c.a1[l], 8);  // weights in lane order (pack_closure)
  float inf = __builtin_inff();
  asm("" : "+s"(inf));
  float part[2];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    bf16x4_t b1;
    __builtin_memcpy(&b1, in[cb], 8);
    f32x16_t d1 = {};
    d1 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a1, b1, d1, 0, 0, 0);
    // relu and BF16 rounding of the hidden layer first: d1 is dead before the second layer starts
    bf16x4_t hb[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const unsigned h[2] = {bf16_pair(relu(d1[4 * kb], inf), relu(d1[4 * kb + 1], inf)),
                             bf16_pair(relu(d1[4 * kb + 2], inf), relu(d1[4 * kb + 3], inf))};
      __builtin_memcpy(&hb[kb], h, 8);
    }
    f32x16_t d2;
    __builtin_memcpy(&d2, c.b2[half], 64);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      bf16x4_t a2;
      __builtin_memcpy(&a2, &c.a2[kb][l], 8);
      d2 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a2, hb[kb], d2, 0, 0, 0);
    }
    part[cb] = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) part[cb] = __builtin_fmaf(c.w3[half][r], relu(d2[r], inf), part[cb]);
  }
  // the lane's own cell: units of the lower half-wavefront + those of the upper one
  unsigned lo = __float_as_uint(part[0]), hi = __float_as_uint(part[1]);
  swap_halves(lo, hi);
  return (__uint_as_float(lo) + __uint_as_float(hi)) + c.b3;
}

// tau0: the plain relaxation time 3 nu + 1/2 (float).
__device__ __forceinline__ float closure_w(const float (&x)[7], const ClosureParams &c, float tau0) {
  float xn[7], h1[CL_H];
#pragma unroll
  for (int j = 0; j < 7; ++j) xn[j] = (x[j] - c.mu[j]) * c.sc[j];
#pragma unroll
  for (int o = 0; o < CL_H; ++o) {
    float a = c.p[CL_B1 + o];
#pragma unroll
    for (int j = 0; j < 7; ++j) a = __builtin_fmaf(c.p[CL_W1 + o * 7 + j], xn[j], a);
    h1[o] = a > 0.f ? a : 0.f;
  }
  float y = c.p[CL_B3];
#pragma unroll
  for (int o = 0; o < CL_H; ++o) {
    float a = c.p[CL_B2 + o];
#pragma unroll
    for (int j = 0; j < CL_H; ++j) a = __builtin_fmaf(c.p[CL_W2 + o * CL_H + j], h1[j], a);
    const float h2 = a > 0.f ? a : 0.f;
    y = __builtin_fmaf(c.p[CL_W3 + o], h2, y);
  }
  return closure_relax(y, c.out, tau0);
}

}  // namespace aslhip
