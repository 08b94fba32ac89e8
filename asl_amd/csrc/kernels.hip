// kernels.hip — hand-written gfx950 kernels of the LBGK hot path.
//
// One fused collide+stream pass per time step in the AA pattern: the
// populations live in one set of Q structure-of-arrays fields (ASL's
// ghost-inclusive, z-fastest layout per direction).  An even step reads and
// writes each cell's own slots (outgoing population i goes to slot inv(i));
// an odd step reads slot (x - c_i, inv i) and writes slot (x + c_i, i).  Both
// move Q reads + Q writes per cell and need no second copy of the lattice.
//
// Boundary conditions fold into the same pass.  ASL fills ghost links after
// the collision (src/num/aslLBGKBC.cxx); here every computation node resolves
// its incoming links when it reads them, through a packed one-byte cell-type
// map and, for the few cells next to a boundary, a 32-byte link pattern:
//   MODE_BOUNCE  f_k(x) = f*_kbar(x) [+ addend]: the cell's own outgoing kbar
//                population of the previous step, which the AA pattern left in
//                the other slot of the same link pair (the read simply uses
//                the other parity's address);
//   MODE_CONST   a constant population (pressure BCs);
//   MODE_LINK    written between steps by the boundary-link kernel
//                (velocity map BCs, whose value needs rho at the ghost node).
// Cells on the lattice's faces follow a rule on their coordinates instead.
// Both are wavefront-uniform branches: a wavefront without such cells runs the
// plain streaming path.
//
// The collision is ASL's LBGK::init0 (src/num/aslLBGK.cxx:187-235) in ASL's
// operation order; the library is compiled with -ffp-contract=off so each
// operation rounds once, as in the CPU oracle.
#include <hip/hip_runtime.h>

#include "../../include/aslhip.h"
#include "kernels.hpp"

namespace aslhip {
namespace {

constexpr int BLOCK = 256;

// The populations live in global memory; their pointers come from the
// argument block in device memory, so the compiler cannot tell the address
// space and would emit flat accesses.  These casts make them global ones.
template <class T>
__device__ __forceinline__ const __attribute__((address_space(1))) T *gload(const char *p) {
  return (const __attribute__((address_space(1))) T *)p;
}
template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T *gstore(char *p) {
  return (__attribute__((address_space(1))) T *)p;
}

// A wavefront-uniform address kept in scalar registers: without this the
// compiler adds the lane's offset first and carries one 64-bit vector address
// per direction (D3Q19: 90 instead of 64 VGPRs).
__device__ __forceinline__ char *scalar_base(char *p) {
  asm("" : "+s"(p));
  return p;
}

// ---------------------------------------------------------------------------
// Storage codecs: FP32, FP64, and BF16 / FP16 deviations f - 1 (ASL's
// weight-normalised populations are 1 at rest), all computed in FP32/FP64.
// ---------------------------------------------------------------------------
template <class S>
struct Codec;

// ld/st take a direction array base and a 32-bit byte offset, so loads use
// the scalar-base + 32-bit vector-offset addressing form.
template <>
struct Codec<float> {
  using C = float;
  using M = float;
  static __device__ __forceinline__ C ld(const char *b, unsigned o) { return *gload<float>(b + o); }
  static __device__ __forceinline__ void st(char *b, unsigned o, C v) { *gstore<float>(b + o) = v; }
  static __device__ __forceinline__ C dec(float s) { return s; }
  static __device__ __forceinline__ float enc(C v) { return v; }
};

template <>
struct Codec<double> {
  using C = double;
  using M = double;
  static __device__ __forceinline__ C ld(const char *b, unsigned o) { return *gload<double>(b + o); }
  static __device__ __forceinline__ void st(char *b, unsigned o, C v) { *gstore<double>(b + o) = v; }
  static __device__ __forceinline__ C dec(double s) { return s; }
  static __device__ __forceinline__ double enc(C v) { return v; }
};

// BF16 bit pattern of f - 1.
template <>
struct Codec<unsigned short> {
  using C = float;
  using M = float;
  static __device__ __forceinline__ C ld(const char *b, unsigned o) {
    return 1.0f + __uint_as_float(static_cast<unsigned>(*gload<unsigned short>(b + o)) << 16);
  }
  // round to nearest even in one instruction (v_cvt_pk_bf16_f32 on gfx950)
  static __device__ __forceinline__ void st(char *b, unsigned o, C v) {
    *gstore<unsigned short>(b + o) = __builtin_bit_cast(unsigned short, static_cast<__bf16>(v - 1.0f));
  }
  static __device__ __forceinline__ C dec(unsigned short s) { return 1.0f + __uint_as_float(static_cast<unsigned>(s) << 16); }
  static __device__ __forceinline__ unsigned short enc(C v) {
    return __builtin_bit_cast(unsigned short, static_cast<__bf16>(v - 1.0f));
  }
};

template <>
struct Codec<_Float16> {
  using C = float;
  using M = float;
  static __device__ __forceinline__ C ld(const char *b, unsigned o) {
    return 1.0f + static_cast<float>(*gload<_Float16>(b + o));
  }
  static __device__ __forceinline__ void st(char *b, unsigned o, C v) {
    *gstore<_Float16>(b + o) = static_cast<_Float16>(v - 1.0f);
  }
  static __device__ __forceinline__ C dec(_Float16 s) { return 1.0f + static_cast<float>(s); }
  static __device__ __forceinline__ _Float16 enc(C v) { return static_cast<_Float16>(v - 1.0f); }
};

__device__ __forceinline__ float fmaT(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmaT(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <int Q>
__device__ __forceinline__ constexpr int offc(int k, int sx, int sy) {
  return Lat<Q>::c[k][0] * sx + Lat<Q>::c[k][1] * sy + Lat<Q>::c[k][2];
}

// v . c_i with the zero terms left out (x + (+-0) == x for finite x).
template <int Q, class C>
__device__ __forceinline__ C dot_c(const C *u, int i) {
  C a = C(0);
  bool first = true;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int cd = Lat<Q>::c[i][d];
    if (cd == 0) continue;
    const C t = cd > 0 ? u[d] : -u[d];
    a = first ? t : a + t;
    first = false;
  }
  return a;
}

// computeMomentum / computeRho (src/num/aslLBGK.cxx:46-63): m = sum w_i c_i f_i
// and rho = sum w_i f_i, left-to-right fma chains without the zero terms.
template <int Q, class C>
__device__ __forceinline__ void moments(const C (&v)[Q], C &r, C (&m)[3]) {
  using LT = Lat<Q>;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    C acc = C(0);
    bool first = true;
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      if (LT::c[j][d] == 0) continue;
      const C cw = C(double(LT::c[j][d]) * LT::w(j));
      acc = first ? v[j] * cw : fmaT(v[j], cw, acc);
      first = false;
    }
    m[d] = acc;
  }
  r = v[0] * C(LT::w(0));
#pragma unroll
  for (int j = 1; j < Q; ++j) r = fmaT(v[j], C(LT::w(j)), r);
}

// x / r for many x and one r, the same bits as the IEEE division.
//
// y is the correctly rounded 1 / r and yl what it lacks, so that
// q = x y + x yl (one rounding) lies within one unit in the last place of
// x / r; for such a q the remainder x - r q is exact and fma(remainder, y, q)
// is the correctly rounded quotient (P. Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", IBM J. Res. Dev. 34,
// 1990).  Four full-rate instructions instead of the eleven of a division
// (one of them a quarter-rate reciprocal); a D3Q19 cell divides ten times by
// its density, with LBGKTurbulence twenty times.  us per step with divisions
// and with this, D3Q19: LBGKTurbulence 128^3 60.6 -> 53.8; FP16 box of
// 256 x 128 x 128 65.0 -> 62.3; FP32 boxes 64^3 9.9 -> 9.7, 16^3 4.6 -> 4.3.
// Nothing may overflow or underflow on the way: recip_safe.
template <class C>
struct Quotient {
  C r, y, yl;
  __device__ __forceinline__ explicit Quotient(C d) : r(d) {
    y = C(1.) / d;
    yl = fmaT(-d, y, C(1.)) * y;
  }
  __device__ __forceinline__ C operator()(C x) const {
    const C q = fmaT(x, y, x * yl);
    return fmaT(fmaT(-r, q, x), y, q);
  }
};

// The division itself, for cells outside recip_safe.
template <class C>
struct Division {
  C r;
  __device__ __forceinline__ explicit Division(C d) : r(d) {}
  __device__ __forceinline__ C operator()(C x) const { return x / r; }
};

// Whether Quotient(r) gives the terms of an equilibrium (4.5 a^2 / r and
// 1.5 m^2 / r = mm / r) as a division would.  r lies in [2^-16, 2^16] and x is at
// most 9 mm < 2^44 (4.5 a^2 of a corner direction, a^2 <= 3 m^2): no overflow (q <
// 2^60), and no underflow for x >= 2^-100 (q >= 2^-116, its
// remainder a multiple of 2^-146).  A smaller x may be off in its last bits,
// but then it is below 2^-84 and is added to or subtracted from a value of at
// least r / 2 >= 2^-17 (a < 2^-50 there), whose rounding it cannot reach.
// NaN and infinities fail the comparisons.
template <class C>
__device__ __forceinline__ bool recip_safe(C r, C mm) {
  return r >= C(0x1p-16) && r <= C(0x1p16) && mm <= C(0x1p40);
}

// 1.5 m . m
template <class C>
__device__ __forceinline__ C square15(const C (&m)[3]) {
  C mm = (C(1.5) * m[0]) * m[0];
  mm = fmaT(C(1.5) * m[1], m[1], mm);
  return fmaT(C(1.5) * m[2], m[2], mm);
}

// The equilibria of all directions of a cell, compressible or not
// (src/num/aslLBGK.cxx:220-231), handed to f0(feq_0) and f(i, j, feq_i,
// feq_j) for each pair of opposite directions.  Opposite directions share
// (4.5 a^2)/rho: a_inv(i) = -a_i exactly in IEEE arithmetic, so this is the
// same value ASL computes twice.
template <int Q, class C, class D, class F0, class F>
__device__ __forceinline__ void equilibria(bool compressible, C r, const C (&m)[3], C mm, const D &over_r, F0 f0,
                                           F f) {
  const C mmr = compressible ? over_r(mm) : mm;
  f0(r - mmr);
#pragma unroll
  for (int i = 1; i < Q; ++i) {
    const int j = inv_dir<Q>(i);
    if (j < i) continue;
    const C a = dot_c<Q>(m, i);
    if (compressible) {
      const C t = over_r(C(4.5) * (a * a));
      f(i, j, (fmaT(C(3.), a, r) + t) - mmr, (fmaT(C(3.), -a, r) + t) - mmr);
    } else {
      const C aa = a * a;
      f(i, j, fmaT(C(4.5), aa, fmaT(C(3.), a, r)) - mmr, fmaT(C(4.5), aa, fmaT(C(3.), -a, r)) - mmr);
    }
  }
}

// FP64 divides: its steps are bound by memory either way (D3Q19 128^3: 111 us
// per step with divisions and with quotients).
template <int Q, class C, class F0, class F>
__device__ __forceinline__ void equilibria_of(bool compressible, C r, const C (&m)[3], F0 f0, F f) {
  const C mm = square15<C>(m);
  if (sizeof(C) == 4 && compressible && __all(recip_safe(r, mm)))
    equilibria<Q, C>(true, r, m, mm, Quotient<C>(r), f0, f);
  else
    equilibria<Q, C>(compressible, r, m, mm, Division<C>(r), f0, f);
}

// LBGKTurbulence::init0 (src/num/aslLBGK.cxx:298-355): the relaxation of a
// cell from how far its populations are from equilibrium,
//   r = 4 |f - feq|^2 / |f|^2,   w = r > 1 ? 1 / (3 min(nu r, 1/2) + 1/2) : 1 / (3 nu + 1/2).
// ASL reads feq there before assigning it (undefined in its generated code);
// here feq is the equilibrium of the cell's own rho and momentum (before the
// rotating-frame term), the value that statement is evidently meant to use.
template <int Q, class C>
__device__ __forceinline__ C turbulence_w(const C (&v)[Q], const C (&e)[Q], C nu, C w0) {
  C d[Q];  // f - feq, summed in direction order
#pragma unroll
  for (int i = 0; i < Q; ++i) d[i] = v[i] - e[i];
  C fl2 = v[0] * v[0];
  C dl2 = d[0] * d[0];
#pragma unroll
  for (int i = 1; i < Q; ++i) {
    fl2 = fmaT(v[i], v[i], fl2);
    dl2 = fmaT(d[i], d[i], dl2);
  }
  const C rt = C(4.) * (dl2 / fl2);
  const C nr = nu * rt;
  const C lim = nr < C(.5) ? nr : C(.5);
  return rt > C(1.) ? C(1.) / (C(3.) * lim + C(.5)) : w0;
}

// The BGK collision of one cell: ASL's LBGK::init0 (src/num/aslLBGK.cxx:
// 187-235) with computeRho / computeMomentum / a_i_dot_v (:46-72).  Each
// x*y + z of ASL's expression tree is one fma (OpenCL's default FP_CONTRACT
// ON); the CPU oracle contracts the same sites.  On return v holds the
// post-collision populations, r the density and m the momentum.  CL: a
// per-cell relaxation replaces w: 1 LBGKTurbulence's, 2 the closure network's on
// the matrix cores, 3 the closure network's in FP32 on the vector ALUs
// (closures: D3Q19, FP32 collision).  Each is its own kernel, so that none holds
// the registers of another.  LBGKTurbulence apart from the FP32 network and with
// its equilibria formed once: 100 -> 64 VGPRs, FP16 box of 128^3 43.5 -> 34.6 us
// per step, FP32 box of 160 x 72 x 60 22.9 -> 21.1.
template <int Q, class C, int CL = 0>
__device__ __forceinline__ void collide(C (&v)[Q], C w, bool compressible, bool omega, const C (&om)[3], C &r_o,
                                        C (&m_o)[3], const ClosureParams *cl = nullptr, float tau0 = 0.f,
                                        C nu = C(0), const ClosureLds *lds = nullptr) {
  C m[3], r;
  moments<Q, C>(v, r, m);
  // LBGKTurbulence: the equilibria, in FP32 kept for the collision (a rotating
  // frame needs others); FP64 has no registers for them.
  constexpr bool KEEP = CL == 1 && sizeof(C) == 4;
  [[maybe_unused]] C e[Q];
  auto keep0 = [&](C x) { e[0] = x; };
  auto keep = [&](int i, int j, C xi, C xj) {
    e[i] = xi;
    e[j] = xj;
  };
  if constexpr (CL == 1) {
    equilibria_of<Q, C>(compressible, r, m, keep0, keep);
    w = turbulence_w<Q, C>(v, e, nu, w);
  }
  if constexpr (CL >= 2) {
    float x[7];
    closure_features<Q>(v, r, m, x);
    w = CL == 2 ? closure_relax(closure_y_mfma(x, *lds), lds->out, tau0) : closure_w(x, *cl, tau0);
  }
  // LBGK::setOmega (src/num/aslLBGK.cxx:207-208): momentum += (2/w) omega x
  // momentum, one component after the other, each seeing the ones before it
  // (ASL emits one statement per component).
  if (omega) {
    const C t = C(2.) / w;
    m[0] = fmaT(t, fmaT(om[1], m[2], -(om[2] * m[1])), m[0]);
    m[1] = fmaT(t, fmaT(om[2], m[0], -(om[0] * m[2])), m[1]);
    m[2] = fmaT(t, fmaT(om[0], m[1], -(om[1] * m[0])), m[2]);
    if constexpr (KEEP) equilibria_of<Q, C>(compressible, r, m, keep0, keep);
  }
  const C one_w = C(1.) - w;
  if constexpr (KEEP) {
#pragma unroll
    for (int i = 0; i < Q; ++i) v[i] = fmaT(v[i], one_w, w * e[i]);
  } else {
    equilibria_of<Q, C>(
        compressible, r, m, [&](C x) { v[0] = fmaT(v[0], one_w, w * x); },
        [&](int i, int j, C xi, C xj) {
          v[i] = fmaT(v[i], one_w, w * xi);
          v[j] = fmaT(v[j], one_w, w * xj);
        });
  }
  r_o = r;
#pragma unroll
  for (int d = 0; d < 3; ++d) m_o[d] = m[d];
}

// n / d for a divisor known to the host, M = floor(2^64 / d) + 1 (0: d = 1).
// n M / 2^64 lies above n / d by at most n / 2^64 < 1 / d, so the floor is
// exact for all 32-bit n and d.  Uniform operands: a few scalar instructions.
__device__ __forceinline__ unsigned udivm(unsigned n, unsigned long long M) {
  const unsigned long long lo = static_cast<unsigned long long>(n) * static_cast<unsigned>(M);
  const unsigned long long hi = static_cast<unsigned long long>(n) * static_cast<unsigned>(M >> 32);
  const unsigned q = static_cast<unsigned>((hi + (lo >> 32)) >> 32);
  return M == 0 ? n : q;
}

// n / d per lane for n < 2^21: (n + 1/2) / d is at least 1 / (2 d) from the
// next integer and its FP32 product with the rounded 1 / d is off by at most
// 2^-23 (n + 1/2) / d, so the truncation is exact.  Three full-rate
// instructions instead of a 64-bit multiplication's quarter-rate ones.
__device__ __forceinline__ unsigned lane_div(unsigned n, float inv) {
  return static_cast<unsigned>((static_cast<float>(n) + 0.5f) * inv);
}

// Workgroups are dispatched round-robin over the 8 XCDs (id % 8).  With a
// group size g > 1, each XCD takes runs of g consecutive chunks (workgroup b
// of a group of 8 g works on chunk  group * 8g + (b % 8) * g + (b % 8g) / 8),
// so that neighbouring chunks, which share cache lines at their edges, meet
// in the same L2; the last, partial group keeps the hardware order.
// m = floor(2^64 / 8g) + 1.
__device__ __forceinline__ int xcd_remap(int L, int n, int g, unsigned long long m) {
  const int span = 8 * g, grp = static_cast<int>(udivm(static_cast<unsigned>(L), m));
  const int r = L - grp * span;
  const int c = grp * span + (r & 7) * g + (r >> 3);
  return (grp + 1) * span > n ? L : c;
}

// Workgroup b of n taking the chunks in reverse order within its XCD's share:
// the chunks b' with b' % 8 == b % 8 are visited from the last to the first,
// so every chunk stays on the XCD (and in the L2) that processed it in the
// previous step.
__device__ __forceinline__ int xcd_reverse(int b, int n) {
  const int r = b & 7, nr = (n - r + 7) >> 3;
  return r + 8 * (nr - 1 - (b >> 3));
}

// The chunk of workgroup b in a launch of n.
template <bool ODD>
__device__ __forceinline__ int chunk_of(const StepHot &g, int b, int n) {
  if (ODD) b = xcd_reverse(b, n);
  return xcd_remap(b, n, g.remap, g.mspan);
}

__device__ __forceinline__ int wrap1(int v, int n) { return v < 1 ? n : (v > n ? 1 : v); }

// The item of work of one lane (StepHot).
struct Item {
  unsigned row;   // ghost-inclusive index of the row's cell z = 0
  int x, y, z;    // 1-based interior coordinates (runs of cells: z counts runs)
  bool act;       // false: past the end of the launch (stands in for the chunk's first item)
};

// No branches: each scalar load of g would sink into the branch that uses it
// and wait there, one memory latency after the other before the first load.
// Rows hold fewer than 2^20 cells (aslhip_lattice_create); only ny may be
// large, so rows are counted from the end of the plane the chunk starts in.
__device__ __forceinline__ Item item_of(const StepHot &g, int chunk) {
  // the chunk's first item, in scalar registers
  const unsigned rowi = static_cast<unsigned>(g.rowi), ny = static_cast<unsigned>(g.ny);
  const unsigned jb = g.first + static_cast<unsigned>(chunk) * static_cast<unsigned>(g.block);
  const unsigned row0 = udivm(jb, g.mrow), x0 = udivm(row0, g.mplane);
  const unsigned z0 = jb - row0 * rowi, y0 = row0 - x0 * ny, left = ny - y0;
  // (x, y, z) is cell x sx + y sy + z with sx = (ny + 2) sy: row r of the interior (r = (x - 1) ny + y - 1)
  // starts at (r + 2 (x - 1) + ny + 3) sy
  const unsigned base = (row0 + 2u * x0 + ny + 3u) * static_cast<unsigned>(g.sy);
  Item it;
  it.act = jb + threadIdx.x < g.first + g.count;
  const unsigned n = z0 + (it.act ? threadIdx.x : 0u);
  const unsigned dr = lane_div(n, g.inv_row);
  const bool next = dr >= left;  // past the plane of the first item
  const unsigned over = next ? dr - left : 0u, more = lane_div(over, g.inv_ny);
  const unsigned dx = next ? more + 1u : 0u;
  it.z = static_cast<int>(n - __umul24(dr, rowi)) + 1;
  it.y = static_cast<int>(next ? over - __umul24(more, ny) : y0 + dr) + 1;
  it.x = static_cast<int>(x0 + dx) + 1;
  it.row = base + __umul24(dr + 2u * dx, static_cast<unsigned>(g.sy));
  return it;
}

// Bit f: the cell lies on face f (X0 XE Y0 YE Z0 ZE).
__device__ __forceinline__ unsigned face_bits(const StepHot &g, int x, int y, int z) {
  return (x == 1 ? 1u : 0u) | (x == g.nx ? 2u : 0u) | (y == 1 ? 4u : 0u) | (y == g.ny ? 8u : 0u) |
         (z == 1 ? 16u : 0u) | (z == g.nz ? 32u : 0u);
}

// ~0 if the cell lies on the face of entry j of the face rule, else 0.
__device__ __forceinline__ unsigned on_entry(const StepHot &g, unsigned fb, int j) {
  return static_cast<unsigned>(__builtin_amdgcn_sbfe(static_cast<int>(fb), (g.fpos >> (4 * j)) & 15u, 1u));
}

// Bounce-back links of a cell on the faces fb: entry by entry, later ones over
// earlier ones.  Three vector instructions per entry, in place
// of a search over three faces per link that was about 800 instructions in
// every wavefront with a face cell, that is in nearly every wavefront where a
// row is not much longer than one.  us per step of a closed box before and
// after (256 x 128 x 128): D3Q19 FP32 126.2 -> 120.3, FP16 67.6 -> 62.4, FP64
// 230 -> 211, D3Q27 FP16 111 -> 91.5, FP64 382 -> 328; 64^3: D3Q19 FP32 12.1
// -> 9.6, FP16 10.8 -> 7.7.
__device__ __forceinline__ unsigned face_masks(const StepHot &g, unsigned fb) {
  unsigned bounce = 0u;
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const unsigned m = on_entry(g, fb, j) & g.flinks[j];
    bounce = (bounce & ~m) | ((g.fbounce >> j) & 1u ? m : 0u);
  }
  return bounce;
}

// Links that enter through face f.
template <int Q>
constexpr unsigned face_links(int f) {
  unsigned m = 0;
  for (int k = 1; k < Q; ++k)
    if (Lat<Q>::c[k][f / 2] == (f % 2 == 0 ? 1 : -1)) m |= 1u << k;
  return m;
}

// Adds (bounce-back) or sets (constant) the values of the faces that have
// some, each on the links it won.  Only wavefronts with a cell on such a face
// (an inlet, an outlet, a lid) get past the tests.  Faces and links are fixed
// at compile time: with the entries' order the links would be tested one by
// one, and the compiler threads those uniform branches into thousands of
// scalar instructions.
template <int Q, class C>
__device__ __forceinline__ void face_values(const StepHot &g, const StepArgs &a, unsigned fb, C (&v)[Q]) {
  if (g.fvalued == 0u) return;
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    if (!((g.fvalued >> f) & 1u)) continue;
    unsigned own = ((fb >> f) & 1u) ? face_links<Q>(f) : 0u;
    if (!__any(own != 0u)) continue;
    const unsigned beats = a.fbeats[f];
#pragma unroll
    for (int h = 0; h < 6; ++h)
      if (h / 2 != f / 2) own &= ((fb & beats) >> h) & 1u ? ~face_links<Q>(h) : ~0u;
    const bool bounce = (g.fbfaces >> f) & 1u;
#pragma unroll
    for (int k = 1; k < Q; ++k) {
      if (!((face_links<Q>(f) >> k) & 1u)) continue;
      const C val = sizeof(C) == 4 ? C(a.fval32[f][k]) : C(a.fval64[f][k]);
      const C nv = (bounce ? v[k] : C(0)) + val;
      v[k] = ((own >> k) & 1u) ? nv : v[k];
    }
  }
}

// One cell per lane of one step, chunk `chunk` of the launch g of the lattice
// described by a.  Every direction array is addressed by a base in scalar
// registers (array, shifted by the direction's offset on odd steps) plus the
// lane's 32-bit byte offset, so that a load or store of an interior wavefront
// takes no vector address arithmetic; an array stays below 4 GiB.
// WIDE: the arrays together exceed 4 GiB (only the links that choose between
// two slots are affected).
template <int Q, class S, bool ODD, bool PER, bool WIDE, int CL = 0>
__device__ __forceinline__ void step_body(const StepHot &g, const StepArgs &a, const int chunk) {
  using CD = Codec<S>;
  using C = typename CD::C;
  using M = typename CD::M;
  constexpr unsigned ES = sizeof(S);
  const Item it = item_of(g, chunk);
  // The matrix-core closure keeps every lane to the end (its network runs on
  // matrix instructions across the wavefront): a lane past the end works on a
  // stand-in cell and stores nothing.
  if constexpr (CL != 2) {
    if (!it.act) return;
  }
  const unsigned idx = it.row + static_cast<unsigned>(it.z), ib = idx * ES;
  char *const f = g.f;

  // The slot of link k that a cell shares with its neighbour x - c_k: array
  // inv k at x - c_k on odd steps, array k at x on even ones; outgoing k goes
  // to array k at x + c_k (odd) or array inv k at x (even).
  // Periodic lattices, odd steps: byte steps to the neighbours along each axis, wrapped.
  unsigned nx_[3], ny_[3], nz_[3];  // for c = -1, 0, 1
  if constexpr (PER && ODD) {
    const unsigned sxb = ES * static_cast<unsigned>(g.sx), syb = ES * static_cast<unsigned>(g.sy);
    nx_[0] = it.x == 1 ? (static_cast<unsigned>(g.nx) - 1u) * sxb : 0u - sxb;
    nx_[2] = it.x == g.nx ? (1u - static_cast<unsigned>(g.nx)) * sxb : sxb;
    ny_[0] = it.y == 1 ? (static_cast<unsigned>(g.ny) - 1u) * syb : 0u - syb;
    ny_[2] = it.y == g.ny ? (1u - static_cast<unsigned>(g.ny)) * syb : syb;
    nz_[0] = it.z == 1 ? (static_cast<unsigned>(g.nz) - 1u) * ES : 0u - ES;
    nz_[2] = it.z == g.nz ? (1u - static_cast<unsigned>(g.nz)) * ES : ES;
    nx_[1] = ny_[1] = nz_[1] = 0u;
  }
  // lane offset of x + sgn c_k (periodic odd steps); the base carries the shift otherwise
  auto lane = [&](int k, int sgn) -> unsigned {
    if constexpr (PER && ODD)
      return ib + nx_[1 + sgn * Lat<Q>::c[k][0]] + ny_[1 + sgn * Lat<Q>::c[k][1]] + nz_[1 + sgn * Lat<Q>::c[k][2]];
    else
      return ib;
  };
  // base of array j, shifted by sgn c_k on non-periodic lattices (sh: shifted at all)
  auto base = [&](int j, int k, int sgn, bool sh) -> char * {
    char *b = f + static_cast<unsigned long long>(j) * g.qs;
    if (!PER && sh) b += static_cast<long long>(sgn) * static_cast<long long>(ES) * offc<Q>(k, g.sx, g.sy);
    return scalar_base(b);
  };
  auto in_base = [&](int k) -> char * { return base(ODD ? inv_dir<Q>(k) : k, k, -1, ODD); };
  auto other_base = [&](int k) -> char * { return base(ODD ? k : inv_dir<Q>(k), k, -1, !ODD); };
  auto out_base = [&](int k) -> char * { return base(ODD ? k : inv_dir<Q>(k), k, 1, ODD); };
  // slot of link k, or the other slot of its pair where mask is ~0 (non-periodic)
  auto load_sel = [&](int k, unsigned mask) -> C {
    if constexpr (WIDE) {
      return CD::ld(mask ? other_base(k) : in_base(k), ib);
    } else {
      const unsigned on = static_cast<unsigned>(in_base(k) - f), op = static_cast<unsigned>(other_base(k) - f);
      return CD::ld(f, (ib + on) + (mask & (op - on)));
    }
  };

  // Faces of the lattice (face rule, see StepHot): a wavefront-uniform branch,
  // so interior wavefronts load plainly, and wavefronts whose face cells lie
  // on z faces only (all wavefronts, where rows are short) choose a slot for
  // the links through those only.
  const bool raw = (g.flags & STEP_F_RAW) != 0;
  unsigned fb = 0, bmask = 0;
  bool faces = false, xyfaces = false;
  if constexpr (!PER) {
    const bool bxy = (it.x == 1) | (it.x == g.nx) | (it.y == 1) | (it.y == g.ny);
    const bool bz = (it.z == 1) | (it.z == g.nz);
    xyfaces = __any(bxy & !raw);
    faces = __any((bxy | bz) & !raw);
    if (xyfaces) {
      fb = face_bits(g, it.x, it.y, it.z);
      bmask = face_masks(g, fb);
    } else if (faces) {
      fb = (it.z == 1 ? 16u : 0u) | (it.z == g.nz ? 32u : 0u);
    }
  }

  // One round of loads: the cell type and every population (bounce-back
  // links read the other slot of their link pair; the value read for a
  // constant link is replaced below).  All addresses lie inside the lattice
  // for interior cells.  Loads take no divergent branch (branches around
  // loads into the same register force the compiler to wait for memory inside
  // the branch).
  const unsigned char code = *gload<unsigned char>(reinterpret_cast<const char *>(g.code) + idx);
  C v[Q];
  if (!faces) {
#pragma unroll
    for (int k = 0; k < Q; ++k) v[k] = CD::ld(in_base(k), lane(k, -1));
  } else if (!xyfaces) {
    // z faces only (every wavefront that holds a row end): one choice for all
    // links that enter through a face.  The masks of all faces took an FP16
    // 128^3 box from 34.9 to 37.3 us a step, its matrix-core closure from 66.6 to 68.7.
    const unsigned lo = it.z == 1 && (g.fbfaces & 16u) ? ~0u : 0u, hi = it.z == g.nz && (g.fbfaces & 32u) ? ~0u : 0u;
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      if (Lat<Q>::c[k][2] != 0)
        v[k] = load_sel(k, Lat<Q>::c[k][2] > 0 ? lo : hi);
      else
        v[k] = CD::ld(in_base(k), ib);
    }
  } else {
    v[0] = CD::ld(in_base(0), ib);
#pragma unroll
    for (int k = 1; k < Q; ++k)
      v[k] = load_sel(k, static_cast<unsigned>(__builtin_amdgcn_sbfe(static_cast<int>(bmask), k, 1)));
  }
  // Keep the scheduler from hoisting the wait on the cell type above the
  // population loads.
  __builtin_amdgcn_sched_barrier(0);
  const ClosureLds *lds = nullptr;
  if constexpr (CL == 2) {  // the network's parameters: 2.9 KB from L2, waited for with the populations
    __shared__ ClosureLds sh;
    const char *src = reinterpret_cast<const char *>(a.cl) + CL_B3 * sizeof(float);
    for (unsigned i = threadIdx.x * 16u; i < sizeof(ClosureLds); i += static_cast<unsigned>(g.block) * 16u)
      *reinterpret_cast<u32x4_t *>(reinterpret_cast<char *>(&sh) + i) = *gload<u32x4_t>(src + i);
    __syncthreads();
    lds = &sh;
  }
  if (faces) face_values<Q, C>(g, a, fb, v);

  // Cells that are not computed run the collision on whatever they read and
  // store nothing; cells with a link pattern re-read their links from it.
  const bool live = code != CODE_SKIP;
  const bool bnd = live && code != CODE_FLUID;
  const bool general = !PER && __any(bnd);
  unsigned skipm = 0;
  if (general && bnd) {
    const LinkRec rec = a.rec[*gload<unsigned short>(reinterpret_cast<const char *>(a.pat) + 2u * idx)];
    skipm = rec.skip;
    const C *val = static_cast<const C *>(a.val);
#pragma unroll
    for (int k = 1; k < Q; ++k) {
      const int slot = raw ? 0 : rec.slot[k];
      const unsigned char md = slot ? a.mode[slot] : static_cast<unsigned char>(MODE_NONE);
      const C x = load_sel(k, md == MODE_BOUNCE ? ~0u : 0u);
      const C sv = val[slot * Q + k];
      v[k] = md == MODE_BOUNCE ? x + sv : (md == MODE_CONST ? sv : x);
    }
  }

  C r, m[3];
  const bool omega = (g.flags & STEP_F_OMEGA) != 0;
  C om[3] = {C(0), C(0), C(0)};
  if (omega) {
#pragma unroll
    for (int d = 0; d < 3; ++d) om[d] = sizeof(C) == 4 ? C(a.om32[d]) : C(a.om64[d]);
  }
  collide<Q, C, CL>(v, C(a.w), (g.flags & STEP_F_COMPRESSIBLE) != 0, omega, om, r, m, a.cl, a.cl_tau0,
                    sizeof(C) == 4 ? C(a.nu32) : C(a.nu64), lds);

  if (!live || !it.act) return;
  if constexpr (PER && ODD) {  // offsets formed again for the stores: 18 of them live across the collision cost waves
#pragma unroll
    for (int d = 0; d < 3; d += 2) asm("" : "+v"(nx_[d]), "+v"(ny_[d]), "+v"(nz_[d]));
  }
  if (general) {
#pragma unroll
    for (int k = 0; k < Q; ++k)
      if (!((skipm >> k) & 1u)) CD::st(out_base(k), lane(k, 1), v[k]);
  } else {
#pragma unroll
    for (int k = 0; k < Q; ++k) CD::st(out_base(k), lane(k, 1), v[k]);
  }
  if (g.flags & STEP_F_RHO) *gstore<M>(static_cast<char *>(a.rho) + sizeof(M) * idx) = M(r);
  if (g.flags & STEP_F_VEL) {
    const bool comp = (g.flags & STEP_F_COMPRESSIBLE) != 0;
    char *u = static_cast<char *>(a.u);
#pragma unroll
    for (int d = 0; d < 3; ++d)
      *gstore<M>(u + sizeof(M) * (static_cast<size_t>(d) * a.len + idx)) = M(comp ? m[d] / r : m[d]);
  }
}

// CPL consecutive cells along z in one lane (a vector of raw storage
// elements; only element alignment is assumed, gfx950 loads and stores such
// vectors as one access).
template <class S, int CPL>
struct RunVec {
  typedef S type __attribute__((ext_vector_type(CPL), aligned(sizeof(S))));
};

// One step of CPL consecutive cells z0 .. z0 + CPL - 1 of a row (lanes cover
// the interior only; nz is a multiple of CPL), non-periodic lattices under
// 4 GiB, plain or rotating-frame LBGK.  Same addresses, same collision and
// same link resolution per cell as step_body, so every cell ends bit for bit
// where step_body leaves it; each direction moves CPL elements per load and
// store.  Cells on a face layer or with a link pattern are fixed up after the
// vector loads (wavefront-uniform branches), and a run with a cell that is
// not computed, or that must not write some links, stores cell by cell.
template <int Q, class S, bool ODD, int CPL>
__device__ __forceinline__ void step_body_run(const StepHot &g, const StepArgs &a, const int chunk) {
  using CD = Codec<S>;
  using C = typename CD::C;
  using M = typename CD::M;
  using V = typename RunVec<S, CPL>::type;
  constexpr unsigned ES = sizeof(S);
  const Item it = item_of(g, chunk);
  if (!it.act) return;
  const int z0 = 1 + CPL * (it.z - 1);
  const int x = it.x, y = it.y;
  const unsigned idx = it.row + static_cast<unsigned>(z0);
  const unsigned ib = idx * ES;
  const char *f0 = g.f;

  // Face rule (as step_body), in one round of loads.  A run lies on an x or y
  // face with all its cells, so a bounce-back link there is a vector load of
  // the other slot of the link pair; only the first (z = 1) and the last
  // (z = nz) cell of a row lie on a z face, and their links with a z share
  // come from side loads of one element, issued with the vector loads.
  const bool raw_links = (g.flags & STEP_F_RAW) != 0;
  const unsigned fxy = raw_links ? 0u : face_bits(g, x, y, 0);
  const bool zlo = !raw_links && z0 == 1, zhi = !raw_links && z0 + CPL - 1 == g.nz;
  const bool xyf = __any(fxy != 0u), zf = __any(zlo || zhi);  // wavefront-uniform
  const unsigned bxy = xyf ? face_masks(g, fxy) : 0u;  // bounce-back links of the x and y faces
  // the other slot of link k's pair for the cell at byte offset ibc
  auto other = [&](int k, unsigned ibc) -> unsigned {
    const unsigned o = ES * static_cast<unsigned>(offc<Q>(k, g.sx, g.sy));
    return static_cast<unsigned>(ODD ? k : inv_dir<Q>(k)) * a.qs32 + (ODD ? ibc : ibc - o);
  };
  V raw[Q];
  C side[Q];  // links of the first (c_z > 0) or last (c_z < 0) cell: the other slot
#pragma unroll
  for (int k = 0; k < Q; ++k) {
    // normal slot: (x, k) (even) or (x - c_k, inv k) (odd)
    const unsigned o = ES * static_cast<unsigned>(offc<Q>(k, g.sx, g.sy));
    const unsigned on = static_cast<unsigned>(ODD ? inv_dir<Q>(k) : k) * a.qs32 + (ODD ? ib - o : ib);
    if (xyf) {
      const unsigned op = other(k, ib);
      raw[k] = *gload<V>(f0 + (((bxy >> k) & 1u) ? op : on));
    } else {
      raw[k] = *gload<V>(f0 + on);
    }
    if (zf && Lat<Q>::c[k][2] != 0) side[k] = CD::ld(f0, other(k, Lat<Q>::c[k][2] > 0 ? ib : ib + ES * (CPL - 1)));
  }
  unsigned codes = 0;  // CPL cell-type bytes
  const char *cb = reinterpret_cast<const char *>(g.code) + idx;
#pragma unroll
  for (int c = 0; c < CPL; ++c) codes |= static_cast<unsigned>(*gload<unsigned char>(cb + c)) << (8 * c);
  __builtin_amdgcn_sched_barrier(0);
  C v[CPL][Q];
#pragma unroll
  for (int c = 0; c < CPL; ++c)
#pragma unroll
    for (int k = 0; k < Q; ++k) v[c][k] = CD::dec(raw[k][c]);
  if (zf) {
    // bounce-back links with a z share of the end cells, whichever face they bounce at
    const unsigned blo = face_masks(g, fxy | (zlo ? 16u : 0u)), bhi = face_masks(g, fxy | (zhi ? 32u : 0u));
#pragma unroll
    for (int k = 1; k < Q; ++k) {
      const int cz = Lat<Q>::c[k][2];
      if (cz == 0) continue;
      const int c = cz > 0 ? 0 : CPL - 1;
      if (cz > 0 ? zlo && ((blo >> k) & 1u) : zhi && ((bhi >> k) & 1u)) v[c][k] = side[k];
    }
  }
  if (xyf || zf) {
#pragma unroll
    for (int c = 0; c < CPL; ++c)
      face_values<Q, C>(g, a, fxy | (c == 0 && zlo ? 16u : 0u) | (c == CPL - 1 && zhi ? 32u : 0u), v[c]);
  }

  // Cells with a link pattern re-read their links from it.
  bool live[CPL];
  bool bnd_any = false;
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    const unsigned char code = static_cast<unsigned char>(codes >> (8 * c));
    live[c] = code != CODE_SKIP;
    bnd_any |= live[c] && code != CODE_FLUID;
  }
  unsigned skipm[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) skipm[c] = 0u;
  const bool general = __any(bnd_any);
  if (general && bnd_any) {
    const C *val = static_cast<const C *>(a.val);
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const unsigned char code = static_cast<unsigned char>(codes >> (8 * c));
      if (!live[c] || code == CODE_FLUID) continue;
      const unsigned ibc = ib + ES * c;
      const LinkRec rec = a.rec[a.pat[idx + c]];
      skipm[c] = rec.skip;
#pragma unroll
      for (int k = 1; k < Q; ++k) {
        const int slot = raw_links ? 0 : rec.slot[k];
        const unsigned char md = slot ? a.mode[slot] : static_cast<unsigned char>(MODE_NONE);
        const unsigned o = ES * static_cast<unsigned>(offc<Q>(k, g.sx, g.sy));
        const unsigned on = static_cast<unsigned>(ODD ? inv_dir<Q>(k) : k) * a.qs32 + (ODD ? ibc - o : ibc);
        const unsigned op = static_cast<unsigned>(ODD ? k : inv_dir<Q>(k)) * a.qs32 + (ODD ? ibc : ibc - o);
        const C xk = CD::ld(f0, md == MODE_BOUNCE ? op : on);
        const C sv = val[slot * Q + k];
        v[c][k] = md == MODE_BOUNCE ? xk + sv : (md == MODE_CONST ? sv : xk);
      }
    }
  }

  const bool omega = (g.flags & STEP_F_OMEGA) != 0;
  const bool comp = (g.flags & STEP_F_COMPRESSIBLE) != 0;
  C om[3] = {C(0), C(0), C(0)};
  if (omega) {
#pragma unroll
    for (int d = 0; d < 3; ++d) om[d] = sizeof(C) == 4 ? C(a.om32[d]) : C(a.om64[d]);
  }
  C r[CPL], m[CPL][3];
#pragma unroll
  for (int c = 0; c < CPL; ++c) collide<Q, C>(v[c], C(a.w), comp, omega, om, r[c], m[c]);

  bool plain = true;
#pragma unroll
  for (int c = 0; c < CPL; ++c) plain = plain && live[c] && skipm[c] == 0u;
  char *fw = g.f;
#pragma unroll
  for (int k = 0; k < Q; ++k) {
    // even: slot (x, inv k); odd: slot (x + c_k, k)
    const unsigned o = ES * static_cast<unsigned>(offc<Q>(k, g.sx, g.sy));
    const unsigned ow = static_cast<unsigned>(ODD ? k : inv_dir<Q>(k)) * a.qs32 + (ODD ? ib + o : ib);
    if (plain) {
      V out;
#pragma unroll
      for (int c = 0; c < CPL; ++c) out[c] = CD::enc(v[c][k]);
      *gstore<V>(fw + ow) = out;
    } else {
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        if (live[c] && !((skipm[c] >> k) & 1u)) CD::st(fw, ow + ES * c, v[c][k]);
    }
  }
  if (g.flags & (STEP_F_RHO | STEP_F_VEL)) {
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      if (!live[c]) continue;
      if (g.flags & STEP_F_RHO) static_cast<M *>(a.rho)[idx + c] = M(r[c]);
      if (g.flags & STEP_F_VEL) {
        M *u = static_cast<M *>(a.u);
#pragma unroll
        for (int d = 0; d < 3; ++d) u[d * a.len + idx + c] = M(comp ? m[c][d] / r[c] : m[c][d]);
      }
    }
  }
}

// LDS slot of a raw storage element: the element itself, or its bits in a
// 32-bit word for 16-bit storage.
template <class S>
struct LdsSlot {
  using type = S;
  static __device__ __forceinline__ S put(S x) { return x; }
  static __device__ __forceinline__ S get(S x) { return x; }
};
template <>
struct LdsSlot<unsigned short> {
  using type = unsigned;
  static __device__ __forceinline__ unsigned put(unsigned short x) { return x; }
  static __device__ __forceinline__ unsigned short get(unsigned x) { return static_cast<unsigned short>(x); }
};
template <>
struct LdsSlot<_Float16> {
  using type = unsigned;
  static __device__ __forceinline__ unsigned put(_Float16 x) {
    unsigned short b;
    __builtin_memcpy(&b, &x, 2);
    return b;
  }
  static __device__ __forceinline__ _Float16 get(unsigned x) {
    const unsigned short b = static_cast<unsigned short>(x);
    _Float16 r;
    __builtin_memcpy(&r, &b, 2);
    return r;
  }
};

// Direction components packed two bits each ((c + 1) << 2k), so that the
// offset of a direction chosen at run time is a few scalar instructions.
template <int Q>
constexpr unsigned long long packed_dir(int d) {
  unsigned long long m = 0;
  for (int k = 0; k < Q; ++k) m |= static_cast<unsigned long long>(Lat<Q>::c[k][d] + 1) << (2 * k);
  return m;
}

// Offset of c_j in the layout for a direction j known at run time.
template <int Q>
__device__ __forceinline__ int offc_rt(int j, int sx, int sy) {
  constexpr unsigned long long PX = packed_dir<Q>(0), PY = packed_dir<Q>(1), PZ = packed_dir<Q>(2);
  const int cx = static_cast<int>((PX >> (2 * j)) & 3ull) - 1;
  const int cy = static_cast<int>((PY >> (2 * j)) & 3ull) - 1;
  const int cz = static_cast<int>((PZ >> (2 * j)) & 3ull) - 1;
  return cx * sx + cy * sy + cz;
}

// LDS-staged step: a workgroup of STEP_TILE lanes takes STEP_TILE consecutive
// cells of a plane (chunks as in step_body, ghost columns included; the last
// chunk of a plane is shorter).  In the AA pattern the slots the tile's cells
// use in direction array j form one contiguous range ("row" j): cells
// idx0 .. idx0 + n - 1 on even steps, shifted by the offset of c_j on odd
// steps.  So the kernel
//   1. loads every row into LDS with 16-byte loads,
//   2. lets each lane collide its own cell from LDS (one cell per lane, the
//      same link resolution and collision as step_body) and write its
//      outgoing populations into the rows in place, in its own column,
//   3. stores the rows back to the ranges they came from with 16-byte stores.
// Column t of the rows holds exactly the slots cell idx0 + t reads and
// writes: incoming k is row k (even) or row inv k (odd), outgoing k goes to
// row inv k (even) or row k (odd).  Each slot belongs to exactly one cell,
// so tiles never touch each other's slots, and cells that are not computed
// keep their slots as loaded.  A bounce-back link k reads the other slot of
// its pair (even: array inv k at x - c_k; odd: array k at x), which is the
// outgoing row of k at column t - (offset of c_k): from LDS if that column
// lies in the tile, else from global memory (read before the first barrier
// for face cells, after it for link-pattern cells; the slot belongs to a
// cell that is not computed, so its value does not change during the step).
template <int Q, class S, bool ODD>
__device__ __forceinline__ void step_body_tile(const StepHot &g, const StepArgs &a, const int L) {
  using CD = Codec<S>;
  using C = typename CD::C;
  using M = typename CD::M;
  constexpr int TB = STEP_TILE;
  constexpr int NW = TB / 64;             // wavefronts per workgroup
  constexpr int RPW = (Q + NW - 1) / NW;  // rows per wavefront, at most
  constexpr int EPL = TB / 64;            // row elements per lane
  constexpr unsigned ES = sizeof(S);
  static_assert(TB % 64 == 0 && (EPL & (EPL - 1)) == 0, "tile: a power-of-two multiple of 64 cells");
  // LDS slots hold the raw storage bits; 16-bit storage gets 32-bit slots
  // (sub-dword LDS writes from neighbouring lanes collide in a bank)
  using LS = typename LdsSlot<S>::type;
  typedef S V4 __attribute__((ext_vector_type(EPL), aligned(sizeof(S))));  // global: element alignment
  typedef LS L4 __attribute__((ext_vector_type(EPL)));                      // LDS: EPL slots aligned
  __shared__ __attribute__((aligned(16 * sizeof(LS)))) LS row[Q][TB];
  auto rd = [&](int j, int col) -> C { return CD::dec(LdsSlot<S>::get(row[j][col])); };
  const int t = static_cast<int>(threadIdx.x);
  const int plane = L / a.bpp;
  const int chunk = L - plane * a.bpp;
  const int c0 = chunk * TB;                // first cell of the tile in the plane's rows
  const int n = min(TB, g.ny * g.sy - c0);  // cells in the tile
  const long long idx0 = static_cast<long long>(plane + 1) * g.sx + g.sy + c0;
  const long long len = a.len;
  const char *f0 = g.f;
  // first cell of row j's range (j at run time: scalar arithmetic)
  auto row_base = [&](int j) -> long long { return ODD ? idx0 + offc_rt<Q>(j, g.sx, g.sy) : idx0; };
  auto in_row = [](int k) -> int { return ODD ? inv_dir<Q>(k) : k; };   // incoming k, column t
  auto out_row = [](int k) -> int { return ODD ? k : inv_dir<Q>(k); };  // outgoing k, column t

  // this lane's cell
  const bool in_tile = t < n;
  const unsigned off = static_cast<unsigned>(c0 + (in_tile ? t : 0));
  const unsigned rw = static_cast<unsigned>((static_cast<unsigned long long>(off) * a.zmagic) >> 40);
  const int zi = static_cast<int>(off - rw * static_cast<unsigned>(g.sy));
  const int x = plane + 1, y = static_cast<int>(rw) + 1;
  const unsigned idx = static_cast<unsigned>(idx0 + (in_tile ? t : 0));
  const bool column = in_tile && zi != 0 && zi != g.sy - 1;  // not a ghost column
  const unsigned char code = column ? *gload<unsigned char>(reinterpret_cast<const char *>(g.code) + idx) : CODE_SKIP;

  // 1. rows into LDS: wavefront w moves rows w, w + NW, w + 2 NW, ..., lane
  // t elements e .. e + EPL - 1 (e = EPL (t % 64)) of each; every load is issued
  // before the first wait.  A vector whose range leaves the lattice's cells
  // [0, len) (only at the two ends of the lattice) is loaded from cell 0 and
  // then replaced element by element; elements past the tile's n cells are
  // loaded but never used.
  const int e = EPL * (t & 63);
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  {
    V4 xr[RPW];
    bool vok[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int j = w + i * NW;
      const long long gp = j < Q ? row_base(j) + e : 0;
      vok[i] = gp >= 0 && gp + EPL <= len;
      const unsigned gi = vok[i] ? static_cast<unsigned>(gp) : 0u;
      if (j < Q) xr[i] = *gload<V4>(f0 + static_cast<unsigned>(j) * a.qs32 + gi * ES);
    }
    bool fix = false;
#pragma unroll
    for (int i = 0; i < RPW; ++i) fix = fix || (w + i * NW < Q && !vok[i]);
    if (fix) {
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
        const int j = w + i * NW;
        if (j >= Q || vok[i]) continue;
        const long long gp = row_base(j) + e;
#pragma unroll
        for (int q = 0; q < EPL; ++q)
          if (gp + q >= 0 && gp + q < len)
            xr[i][q] = *gload<S>(f0 + static_cast<unsigned>(j) * a.qs32 + static_cast<unsigned>(gp + q) * ES);
      }
    }
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int j = w + i * NW;
      if (j < Q) {
        L4 v4;
#pragma unroll
        for (int q = 0; q < EPL; ++q) v4[q] = LdsSlot<S>::put(xr[i][q]);
        *reinterpret_cast<L4 *>(&row[j][e]) = v4;
      }
    }
  }

  // face rule (as step_body)
  const bool raw = (g.flags & STEP_F_RAW) != 0;
  const unsigned fb = (!column || raw) ? 0u : face_bits(g, x, y, zi);
  const bool faces = __any(fb != 0u);
  const unsigned bmask = faces ? face_masks(g, fb) : 0u;
  // the other slot of link k's pair: the outgoing row of k at column t - (offset of c_k)
  auto other_col = [&](int k) -> int { return t - offc<Q>(k, g.sx, g.sy); };
  auto other_in_tile = [&](int k) -> bool {
    const int oc = other_col(k);
    return oc >= 0 && oc < n;
  };
  auto other_global = [&](int k) -> C {
    const int j = out_row(k);
    const long long gp = (ODD ? idx0 + offc<Q>(j, g.sx, g.sy) : idx0) + other_col(k);
    return CD::ld(f0, static_cast<unsigned>(j) * a.qs32 + static_cast<unsigned>(gp) * ES);
  };
  C side[Q];  // bounce-back values of face cells from outside the tile
  if (faces) {
#pragma unroll
    for (int k = 1; k < Q; ++k)
      if (((bmask >> k) & 1u) && !other_in_tile(k)) side[k] = other_global(k);
  }
  __syncthreads();

  // 2. collide this lane's cell from the rows
  const int tc = in_tile ? t : 0;
  C v[Q];
#pragma unroll
  for (int k = 0; k < Q; ++k) v[k] = rd(in_row(k), tc);
  if (faces) {
#pragma unroll
    for (int k = 1; k < Q; ++k)
      if ((bmask >> k) & 1u) v[k] = other_in_tile(k) ? rd(out_row(k), other_col(k)) : side[k];
    face_values<Q, C>(g, a, fb, v);
  }
  const bool live = code != CODE_SKIP;
  const bool bnd = live && code != CODE_FLUID;
  const bool general = __any(bnd);
  unsigned skipm = 0;
  if (general && bnd) {
    const LinkRec rec = a.rec[*gload<unsigned short>(reinterpret_cast<const char *>(a.pat) + 2u * idx)];
    skipm = rec.skip;
    const C *val = static_cast<const C *>(a.val);
#pragma unroll
    for (int k = 1; k < Q; ++k) {
      const int slot = raw ? 0 : rec.slot[k];
      const unsigned char md = slot ? a.mode[slot] : static_cast<unsigned char>(MODE_NONE);
      C xk = rd(in_row(k), t);
      if (md == MODE_BOUNCE)
        xk = other_in_tile(k) ? rd(out_row(k), other_col(k)) : other_global(k);
      const C sv = val[slot * Q + k];
      v[k] = md == MODE_BOUNCE ? xk + sv : (md == MODE_CONST ? sv : xk);
    }
  }
  // every lane has read what it needs from the rows before any lane writes them
  __syncthreads();
  C r, m[3];
  const bool omega = (g.flags & STEP_F_OMEGA) != 0;
  const bool comp = (g.flags & STEP_F_COMPRESSIBLE) != 0;
  C om[3] = {C(0), C(0), C(0)};
  if (omega) {
#pragma unroll
    for (int d = 0; d < 3; ++d) om[d] = sizeof(C) == 4 ? C(a.om32[d]) : C(a.om64[d]);
  }
  collide<Q, C>(v, C(a.w), comp, omega, om, r, m);
  if (live) {
#pragma unroll
    for (int k = 0; k < Q; ++k)
      if (!((skipm >> k) & 1u)) row[out_row(k)][t] = LdsSlot<S>::put(CD::enc(v[k]));
    if (g.flags & STEP_F_RHO) *gstore<M>(static_cast<char *>(a.rho) + sizeof(M) * idx) = M(r);
    if (g.flags & STEP_F_VEL) {
      char *u = static_cast<char *>(a.u);
#pragma unroll
      for (int d = 0; d < 3; ++d)
        *gstore<M>(u + sizeof(M) * (static_cast<size_t>(d) * a.len + idx)) = M(comp ? m[d] / r : m[d]);
    }
  }
  __syncthreads();

  // 3. rows back to their ranges
  {
    char *fw = g.f;
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int j = w + i * NW;
      if (j >= Q || e >= n) continue;
      const long long gp = row_base(j) + e;
      if (e + EPL <= n && gp >= 0 && gp + EPL <= len) {
        const L4 l4 = *reinterpret_cast<const L4 *>(&row[j][e]);
        V4 x4;
#pragma unroll
        for (int q = 0; q < EPL; ++q) x4[q] = LdsSlot<S>::get(l4[q]);
        *gstore<V4>(fw + static_cast<unsigned>(j) * a.qs32 + static_cast<unsigned>(gp) * ES) = x4;
      } else {
#pragma unroll
        for (int q = 0; q < EPL; ++q)
          if (e + q < n && gp + q >= 0 && gp + q < len)
            *gstore<S>(fw + static_cast<unsigned>(j) * a.qs32 + static_cast<unsigned>(gp + q) * ES) =
                LdsSlot<S>::get(row[j][e + q]);
      }
    }
  }
}

template <int Q, class S, bool ODD>
__global__ __launch_bounds__(STEP_TILE) void k_step_tile(const StepHot g, const StepArgs *args) {
  step_body_tile<Q, S, ODD>(g, *args, chunk_of<ODD>(g, static_cast<int>(blockIdx.x), g.nchunks));
}

// What a wavefront needs before its first load comes by value (StepHot); the
// rest lives in device memory, not in the kernel-argument segment: loads from
// that segment are invariant, the compiler hoists all of them (face values,
// link tables) into scalar registers, runs out of them and spills into vector
// registers.  Loads through a plain pointer stay where they are used.
//
// Odd steps take the chunks in reverse order (zig-zag over steps), each XCD
// over its own share (xcd_reverse): a step then starts where the previous
// one ended, on the populations written last, which its XCD's L2 still
// holds.  Every cell's reads and writes in one step are its own (AA
// pattern), so the order of the chunks does not change results.
template <int Q, class S, bool ODD, bool PER, bool WIDE, int CL>
__global__ __launch_bounds__(step_block(Q, sizeof(S))) void k_step(const StepHot g, const StepArgs *args) {
  step_body<Q, S, ODD, PER, WIDE, CL>(g, *args, chunk_of<ODD>(g, static_cast<int>(blockIdx.x), g.nchunks));
}

// The step with CPL cells per lane (step_body_run); same chunk order.  At
// most STEP_RUN_BLOCK lanes per workgroup: four cells per lane hold about
// 130 VGPRs, more than a 1024-lane workgroup allows without spilling.
template <int Q, class S, bool ODD, int CPL>
__global__ __launch_bounds__(STEP_RUN_BLOCK) void k_step_run(const StepHot g, const StepArgs *args) {
  step_body_run<Q, S, ODD, CPL>(g, *args, chunk_of<ODD>(g, static_cast<int>(blockIdx.x), g.nchunks));
}

// Cell idx + sgn c_i, wrapped into the interior for interior cells of periodic
// lattices.  sgn 1: the cell whose slot i holds population i of cell idx after
// an odd step.
template <int Q>
__device__ __forceinline__ int shifted(int idx, int i, int sgn, int sx, int sy, int per, int nx, int ny, int nz) {
  if (!per) return idx + sgn * offc<Q>(i, sx, sy);
  const int x = idx / sx, rem = idx - x * sx, y = rem / sy, z = rem - y * sy;
  if (x < 1 || x > nx || y < 1 || y > ny || z < 1 || z > nz) return idx + sgn * offc<Q>(i, sx, sy);
  return wrap1(x + sgn * Lat<Q>::c[i][0], nx) * sx + wrap1(y + sgn * Lat<Q>::c[i][1], ny) * sy +
         wrap1(z + sgn * Lat<Q>::c[i][2], nz);
}

// Population i of cell idx after the last step (ASL's view).  Slots outside
// the array (outer ghost layer) read as NaN.
template <int Q, class S>
__device__ __forceinline__ typename Codec<S>::C outgoing(const StepHot &g, int per, int len, int after_odd, int idx,
                                                         int i) {
  using CD = Codec<S>;
  if (!after_odd) return CD::ld(g.f + inv_dir<Q>(i) * g.qs, static_cast<unsigned>(idx) * sizeof(S));
  const int src = shifted<Q>(idx, i, 1, g.sx, g.sy, per, g.nx, g.ny, g.nz);
  if (src < 0 || src >= len) return typename CD::C(__builtin_nan(""));
  return CD::ld(g.f + i * g.qs, static_cast<unsigned>(src) * sizeof(S));
}

// Population k that cell idx receives in the next step, every BC resolved as
// step_body does (face rule, link patterns); 0 for cells that are not computed.
template <int Q, class S>
__device__ __forceinline__ typename Codec<S>::C incoming(const StepHot &g, const StepArgs &a, int per, int after_odd,
                                                         int idx, int k) {
  using CD = Codec<S>;
  using C = typename CD::C;
  const int x = idx / g.sx, rem = idx - x * g.sx, y = rem / g.sy, z = rem - y * g.sy;
  if (x < 1 || x > g.nx || y < 1 || y > g.ny || z < 1 || z > g.nz) return C(0);
  const unsigned char code = g.code[idx];
  if (code == CODE_SKIP) return C(0);
  bool bounce = false, cnst = false;
  C val = C(0);
  if (!per && code == CODE_FLUID) {
    const unsigned fb = face_bits(g, x, y, z) & a.fset;
    int f = -1;  // the face that claims the link, the one executed last
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int cd = Lat<Q>::c[k][d], c = 2 * d + (cd > 0 ? 0 : 1);
      if (cd != 0 && ((fb >> c) & 1u) && (f < 0 || ((a.fbeats[f] >> c) & 1u))) f = c;
    }
    if (f >= 0) {
      bounce = (g.fbfaces >> f) & 1u;
      cnst = !bounce;
      val = sizeof(C) == 4 ? C(a.fval32[f][k]) : C(a.fval64[f][k]);
    }
  } else if (!per) {
    const int slot = a.rec[a.pat[idx]].slot[k];
    const unsigned char md = slot ? a.mode[slot] : static_cast<unsigned char>(MODE_NONE);
    bounce = md == MODE_BOUNCE;
    cnst = md == MODE_CONST;
    val = static_cast<const C *>(a.val)[slot * Q + k];
  }
  if (cnst) return val;
  // array inv k at idx - c_k before an odd step, array k at idx before an even one; bounce-back: the other of the two
  const bool near = bounce == !after_odd;
  const int src = near ? idx : shifted<Q>(idx, k, -1, g.sx, g.sy, per, g.nx, g.ny, g.nz);
  const C v = CD::ld(g.f + (near ? k : inv_dir<Q>(k)) * g.qs, static_cast<unsigned>(src) * sizeof(S));
  return bounce ? v + val : v;
}

// asl::ComputeSurfaceForceMap / ComputeSurfaceFluxMap (src/num/aslLBGKBC.cxx:
// 623-736).  For a ghost cell x (map <= 0) next to a computation node y =
// x + c_i (map > 0), ASL's f_i(x) is the population i that y receives next
// (the value ASL's BCs leave at the ghost); for a computation node x next to a
// ghost y, ASL's f_inv(i)(y) is the population inv(i) that x receives.  Cells
// with |map| >= 0.9999 get 0 (ASL leaves them as they were); map reads outside
// the block are -0.9 (a ghost node), as in ASL.
//
// The populations are taken from the step kernel's slots, and only next to
// the surface: a read of the map and a write of the result for the other
// cells.  Full views of outgoing and incoming populations, as before, cost
// two copies of the lattice: 25 + 24 + 16 us and a clear of 11 on
// 160 x 72 x 60, D3Q19 FP32; 20 steps of LBGKTurbulence there with a force and
// a read of u 2461 -> 1696 us, allocations included.
template <int Q, class S>
__global__ __launch_bounds__(BLOCK) void k_surface(const SurfaceArgs s, const StepHot g, const StepArgs *args) {
  using C = typename Codec<S>::C;
  using M = typename Codec<S>::M;
  const int x = blockIdx.x * BLOCK + threadIdx.x;
  if (x >= s.len) return;
  M *out = static_cast<M *>(s.out);
  const float m0 = s.map[x];
  C acc[3] = {C(0), C(0), C(0)};
  if (__builtin_fabsf(m0) < .9999f) {
#pragma unroll
    for (int i = 1; i < Q; ++i) {
      const int kb = inv_dir<Q>(i);
      const long long y = static_cast<long long>(x) + offc<Q>(i, g.sx, g.sy);
      const float my = (y < 0 || y > s.len - 1) ? -.9f : s.map[y];
      const bool b0 = m0 <= 0.f && my > 0.f;  // isGhostNode(0) && isComputationNode(i)
      const bool bi = m0 > 0.f && my <= 0.f;  // isGhostNode(i) && isComputationNode(0)
      if (!b0 && !bi) continue;  // adds 0
      const int c = b0 ? static_cast<int>(y) : x;  // the computation node of the link
      const C in = incoming<Q, S>(g, *args, s.per, s.after_odd, c, b0 ? i : kb);
      const C post = outgoing<Q, S>(g, s.per, s.len, s.after_odd, c, b0 ? kb : i);
      const C f0 = b0 ? in : post, fI = b0 ? post : in;
      if (s.flux) {
        const C wi = C(Lat<Q>::w(i));
        acc[0] = acc[0] + (b0 ? (f0 - fI) * wi : (fI - f0) * wi);
      } else {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const C wc = C(Lat<Q>::w(i) * double(Lat<Q>::c[i][d]));
          acc[d] = acc[d] + (b0 ? ((f0 + fI) - C(2.)) * wc : ((-f0 - fI) + C(2.)) * wc);
        }
      }
    }
  }
  if (s.flux) {
    out[x] = M(acc[0]);
  } else {
#pragma unroll
    for (int d = 0; d < 3; ++d) out[static_cast<long long>(d) * s.len + x] = M(acc[d]);
  }
}

// Visualisation fills of rho / u (VisArgs).  Reads come only from cells with
// map > 0 and writes go only to cells with map <= 0, so the update in place
// is free of races.  The operations follow the CPU oracle's restatement of
// ASL's kernels (src/num/aslBasicBC.cxx:124-145, 167-227, 283-351) in its
// order, none contracted (the library is built with -ffp-contract=off):
//   NOSLIP_VEL: v += select(0 - v(x + c_i), b_i) * lc_i, n += select(lc_i, b_i),
//               v(x) = v / max(n, .01), over i = 1..Q-1, b_i = map(x + c_i) > 0;
//   NOSLIP_RHO: g_k = sum_i map(x + c_i) (gc_i c_i[k]) over c_i[k] != 0,
//               g /= |g|, p_i = g . c_i/|c_i|, d_i = (p_i + 1)^2,
//               n = max(sum_i select(d_i, b_i), .001),
//               r = sum_i select((rho(x + c_i) - p_i * 0) d_i, b_i),
//               rho(x) = r / n where n > 0.1;
//   VELOCITY:   u(x) = u0, or axis x (position - centre).
template <int Q, class S>
__global__ __launch_bounds__(BLOCK) void k_vis(const VisArgs a) {
  using M = typename Codec<S>::M;
  const int g = blockIdx.x * BLOCK + threadIdx.x;
  if (g >= a.len) return;
  const float mg = a.map[g];
  if (!(mg <= 0.f && mg > -.9999f)) return;
  M *rho = static_cast<M *>(a.rho), *u = static_cast<M *>(a.u);
  const long long len = a.len;
  auto mx = [&](long long y) { return (y < 0 || y > len - 1) ? -.9f : a.map[y]; };
  auto wrap = [&](long long y) { return (len + y) % len; };
  if (a.kind == ASLHIP_VIS_VELOCITY) {
    M uw[3] = {M(a.u0[0]), M(a.u0[1]), M(a.u0[2])};
    if (a.has_rot) {
      // Index2PositionACL over the ghost-inclusive block (src/math/aslIndex2Position.cxx:64-108)
      const int I0 = g / a.sx, rem = g - I0 * a.sx, I1 = rem / a.sy, I2 = rem - I1 * a.sy;
      const int I[3] = {I0, I1, I2};
      M pos[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) pos[d] = M(a.pos0[d] - a.dx) + M(a.dx) * M(I[d]);
      const M d0 = pos[0] - M(a.rot[3]), d1 = pos[1] - M(a.rot[4]), d2 = pos[2] - M(a.rot[5]);
      uw[0] = M(a.rot[1]) * d2 - M(a.rot[2]) * d1;
      uw[1] = M(a.rot[2]) * d0 - M(a.rot[0]) * d2;
      uw[2] = M(a.rot[0]) * d1 - M(a.rot[1]) * d0;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) u[c * len + g] = uw[c];
    return;
  }
  if constexpr (Q != 27) {
    using LT = Lat<Q>;
    if (a.kind == ASLHIP_VIS_NOSLIP_VEL) {
      M v[3] = {M(0), M(0), M(0)}, n = M(0);
#pragma unroll
      for (int i = 1; i < Q; ++i) {
        const long long y = g + offc<Q>(i, a.sx, a.sy);
        const bool b = mx(y) > 0.f;
        const M l = M(LT::lc(i));
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] = v[c] + (b ? M(0) - u[c * len + wrap(y)] : M(0)) * l;
        n = n + (b ? l : M(0));
      }
      const M den = n > M(.01) ? n : M(.01);
#pragma unroll
      for (int c = 0; c < 3; ++c) u[c * len + g] = v[c] / den;
    } else if (a.kind == ASLHIP_VIS_NOSLIP_RHO) {
      M mv[Q];
      bool bv[Q];
#pragma unroll
      for (int i = 1; i < Q; ++i) {
        const float m = mx(g + offc<Q>(i, a.sx, a.sy));
        mv[i] = M(m);
        bv[i] = m > 0.f;
      }
      M gn[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        M acc = M(0);
        bool first = true;
#pragma unroll
        for (int i = 1; i < Q; ++i) {
          if (LT::c[i][k] == 0) continue;
          const M t = mv[i] * M(LT::gc(i) * double(LT::c[i][k]));
          acc = first ? t : acc + t;
          first = false;
        }
        gn[k] = acc;
      }
      M l2 = gn[0] * gn[0];
      l2 = l2 + gn[1] * gn[1];
      l2 = l2 + gn[2] * gn[2];
      const M ln = sizeof(M) == 4 ? M(__builtin_sqrtf(float(l2))) : M(__builtin_sqrt(double(l2)));
#pragma unroll
      for (int k = 0; k < 3; ++k) gn[k] = gn[k] / ln;
      M pr[Q], dc[Q];
      M n = M(0);
#pragma unroll
      for (int i = 1; i < Q; ++i) {
        const double cl = __builtin_sqrt(double(LT::c[i][0] * LT::c[i][0] + LT::c[i][1] * LT::c[i][1] +
                                                LT::c[i][2] * LT::c[i][2]));
        M p = M(0);
        bool first = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          if (LT::c[i][d] == 0) continue;
          const M t = gn[d] * M(double(LT::c[i][d]) / cl);
          p = first ? t : p + t;
          first = false;
        }
        pr[i] = p;
        const M e = p + M(1.);
        dc[i] = e * e;
        n = n + (bv[i] ? dc[i] : M(0));
      }
      n = n > M(.001) ? n : M(.001);
      M r = M(0);
#pragma unroll
      for (int i = 1; i < Q; ++i) {
        const long long y = g + offc<Q>(i, a.sx, a.sy);
        r = r + (bv[i] ? (rho[wrap(y)] - pr[i] * M(0)) * dc[i] : M(0));
      }
      if (n > M(.1)) rho[g] = r / n;
    }
  }
}

// Many lattices in one launch: workgroup b works on chunk ent[b].y of
// lattice ent[b].x, whose descriptor lives in device memory.  One chunk per
// workgroup, with no loop around the body: a loop over several chunks kept
// values live across iterations and raised the kernel from 70 to 99 VGPRs,
// which cut the waves per SIMD from 7 to 4 at 256-lane workgroups.
// Odd steps take the entries in reverse order, as k_step does.
template <int Q, class S, bool ODD, bool PER, bool WIDE>
__global__ __launch_bounds__(step_block(Q, sizeof(S))) void k_step_batch(const StepArgs *desc, const uint2 *ent) {
  const int b = static_cast<int>(blockIdx.x);
  const uint2 e = ent[ODD ? xcd_reverse(b, static_cast<int>(gridDim.x)) : b];
  step_body<Q, S, ODD, PER, WIDE>(desc[e.x].g, desc[e.x], static_cast<int>(e.y));
}

// The same with LDS-staged tiles (entries are tiles of STEP_TILE cells).
template <int Q, class S, bool ODD>
__global__ __launch_bounds__(STEP_TILE) void k_step_batch_tile(const StepArgs *desc, const uint2 *ent) {
  const int b = static_cast<int>(blockIdx.x);
  const uint2 e = ent[ODD ? xcd_reverse(b, static_cast<int>(gridDim.x)) : b];
  step_body_tile<Q, S, ODD>(desc[e.x].g, desc[e.x], static_cast<int>(e.y));
}

// Closure features of every interior cell of a periodic D3Q19 lattice: the
// populations the next step would collide (AA addressing of that step's
// parity, periodic wrap), their moments as collide() forms them, and the 7
// inputs of the closure network, written to out[7 * cell + p] with cells in
// ASL order over the interior.
template <class S, bool ODD>
__global__ __launch_bounds__(256) void k_closure_features(const StepArgs *args, float *out) {
  using CD = Codec<S>;
  constexpr int Q = 19;
  constexpr unsigned ES = sizeof(S);
  const StepHot &a = args->g;
  const long long c = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (c >= static_cast<long long>(a.nx) * a.ny * a.nz) return;
  const int z = static_cast<int>(c % a.nz) + 1;
  const int y = static_cast<int>((c / a.nz) % a.ny) + 1;
  const int x = static_cast<int>(c / (static_cast<long long>(a.ny) * a.nz)) + 1;
  const unsigned idx = static_cast<unsigned>(x * a.sx + y * a.sy + z);
  float v[Q];
#pragma unroll
  for (int k = 0; k < Q; ++k) {
        if (ODD) {
      const unsigned src = static_cast<unsigned>(wrap1(x - Lat<Q>::c[k][0], a.nx) * a.sx +
                                                 wrap1(y - Lat<Q>::c[k][1], a.ny) * a.sy +
                                                 wrap1(z - Lat<Q>::c[k][2], a.nz));
      v[k] = CD::ld(a.f + inv_dir<Q>(k) * a.qs, ES * src);
    } else {
      v[k] = CD::ld(a.f + k * a.qs, ES * idx);
    }
  }
  float r, m[3], f7[7];
  moments<Q, float>(v, r, m);
  closure_features<Q>(v, r, m, f7);
#pragma unroll
  for (int p = 0; p < 7; ++p) out[7 * c + p] = f7[p];
}

// Boundary-link kernel: ASL's BCVelocityMap (src/num/aslLBGKBC.cxx:290-348).
// After a step, rho at ghost node g is estimated from the populations its
// computation-node neighbours sent towards it; the links g -> g+c_i are then
// written where the receivers read them in the next step.
template <int Q, class S>
__global__ __launch_bounds__(BLOCK) void k_vlinks(const VLinkArgs a) {
  using CD = Codec<S>;
  using C = typename CD::C;
  const int e = blockIdx.x * BLOCK + threadIdx.x;
  if (e >= a.nlinks) return;
  const VLink l = a.links[e];
  const VLinkBC bc = a.bc[l.slot];
  constexpr unsigned ES = sizeof(S);
  auto fk = [&](int k) -> char * { return a.f + k * a.qs_bytes; };
  C coef = C(0), r = C(0);
#pragma unroll
  for (int i = 1; i < Q; ++i) {
    if (!((l.comp >> i) & 1u)) continue;
    const int kb = inv_dir<Q>(i);
    const int p = l.g + offc<Q>(i, a.sx, a.sy);
    const C fi = a.after_odd ? CD::ld(fk(kb), ES * l.g) : CD::ld(fk(i), ES * p);
    coef = coef + C(Lat<Q>::w(i));
    r = r + fi * C(Lat<Q>::w(i));
  }
  r = r / coef;
  // Index2PositionACL over the ghost-inclusive block (src/math/aslIndex2Position.cxx:64-108)
  const int I0 = l.g / a.sx, rem = l.g - I0 * a.sx, I1 = rem / a.sy, I2 = rem - I1 * a.sy;
  const int I[3] = {I0, I1, I2};
  C pos[3], uw[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) pos[d] = C(a.pos0[d] - a.dx) + C(a.dx) * C(I[d]);
  if (bc.has_rot) {
    // PFRotationField: crossProduct(axis, pos - c)
    const C d0 = pos[0] - C(bc.centre[0]), d1 = pos[1] - C(bc.centre[1]), d2 = pos[2] - C(bc.centre[2]);
    uw[0] = C(bc.omega[1]) * d2 - C(bc.omega[2]) * d1;
    uw[1] = C(bc.omega[2]) * d0 - C(bc.omega[0]) * d2;
    uw[2] = C(bc.omega[0]) * d1 - C(bc.omega[1]) * d0;
  } else {
#pragma unroll
    for (int d = 0; d < 3; ++d) uw[d] = C(bc.u[d]);
  }
  const C mom[3] = {uw[0] * r, uw[1] * r, uw[2] * r};
#pragma unroll
  for (int i = 1; i < Q; ++i) {
    if (!((l.own >> i) & 1u)) continue;
    const int kb = inv_dir<Q>(i);
    const int p = l.g + offc<Q>(i, a.sx, a.sy);
    const C val = r + dot_c<Q>(mom, i) * C(3.);
    if (a.after_odd)
      CD::st(fk(i), ES * p, val);  // next step is even: p reads slot (p, i)
    else
      CD::st(fk(kb), ES * l.g, val);  // next step is odd: p reads slot (g, inv i)
  }
}

// LBGKUtilities::initF(rho, vel) (src/num/aslLBGK.cxx:262-275) into the state
// "after an even step": the outgoing population i of cell x in slot (x, inv i).
template <int Q, class S>
__global__ __launch_bounds__(BLOCK) void k_init(const InitArgs a) {
  using CD = Codec<S>;
  using C = typename CD::C;
  using M = typename CD::M;
  const int idx = blockIdx.x * BLOCK + threadIdx.x;
  if (idx >= a.len) return;
  C r, u[3];
  r = a.rho_in ? C(static_cast<const M *>(a.rho_in)[idx]) : C(a.rho0);
#pragma unroll
  for (int d = 0; d < 3; ++d) u[d] = a.u_in ? C(static_cast<const M *>(a.u_in)[d * a.len + idx]) : C(a.u0[d]);
  C uu = (C(1.5) * u[0]) * u[0];
  uu = fmaT(C(1.5) * u[1], u[1], uu);
  uu = fmaT(C(1.5) * u[2], u[2], uu);
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const C ai = i == 0 ? C(0) : dot_c<Q>(u, i);
    const C fi = fmaT(C(4.5), ai * ai, fmaT(C(3.), ai, C(1.))) - uu;
    CD::st(a.f + inv_dir<Q>(i) * a.qs_bytes, static_cast<unsigned>(idx) * sizeof(S), r * fi);
  }
  static_cast<M *>(a.rho)[idx] = M(r);
#pragma unroll
  for (int d = 0; d < 3; ++d) static_cast<M *>(a.u)[d * a.len + idx] = M(u[d]);
}

template <int Q, class S>
__global__ __launch_bounds__(BLOCK) void k_write_f(const WriteFArgs a) {
  using CD = Codec<S>;
  using C = typename CD::C;
  using M = typename CD::M;
  const int idx = blockIdx.x * BLOCK + threadIdx.x;
  if (idx >= a.len) return;
  const M *in = static_cast<const M *>(a.in);
  C v[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    v[i] = C(in[static_cast<long long>(i) * a.len + idx]);
    CD::st(a.f + inv_dir<Q>(i) * a.qs_bytes, static_cast<unsigned>(idx) * sizeof(S), v[i]);
  }
  C r, m[3];
  moments<Q, C>(v, r, m);
  static_cast<M *>(a.rho)[idx] = M(r);
#pragma unroll
  for (int d = 0; d < 3; ++d) static_cast<M *>(a.u)[d * a.len + idx] = M(a.compressible ? m[d] / r : m[d]);
}

// The post-collision populations in ASL's view (f_i of cell x), from the AA
// state.  Slots outside the array (outer ghost layer) read as NaN.
template <int Q, class S>
__global__ __launch_bounds__(BLOCK) void k_unpermute(const UnpermuteArgs a) {
  using CD = Codec<S>;
  using M = typename CD::M;
  const int c = blockIdx.x * BLOCK + threadIdx.x;
  if (c >= a.count) return;
  const int idx = a.first + c;
  M *out = static_cast<M *>(a.out);
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    M v;
    if (a.after_odd) {
      const int src = shifted<Q>(idx, i, 1, a.sx, a.sy, a.per, a.nx, a.ny, a.nz);
      v = (src >= 0 && src < a.len)
              ? M(CD::ld(a.f + i * a.qs_bytes, static_cast<unsigned>(src) * sizeof(S)))
              : M(__builtin_nan(""));
    } else {
      v = M(CD::ld(a.f + inv_dir<Q>(i) * a.qs_bytes, static_cast<unsigned>(idx) * sizeof(S)));
    }
    out[static_cast<long long>(i) * a.count + c] = v;
  }
}

// FP64 mass / momentum / kinetic energy over computation nodes: one read of
// the code map and of all populations, so bound by HBM.  Finding the cell's
// coordinates for the periodic wrap once per cell and not once per direction
// took the pass after an odd step from 671 to 243 us (224^3 D3Q27 FP32; 5.0
// TB/s) and from 105 to 49 us (128^3 D3Q19 FP32).
template <int Q, class S>
__global__ __launch_bounds__(BLOCK) void k_reduce(const ReduceArgs a) {
  using CD = Codec<S>;
  __shared__ double sh[5][BLOCK];
  double s[5] = {0., 0., 0., 0., 0.};
  for (int idx = blockIdx.x * BLOCK + threadIdx.x; idx < a.len; idx += gridDim.x * BLOCK) {
    const unsigned char c = a.code[idx];
    if (c != CODE_FLUID && c != CODE_FLUID_BC) continue;
    // after an odd step population i of a cell lies in slot i of idx + c_i:
    // steps to the neighbours along each axis, wrapped on periodic lattices
    // (the cell's coordinates are found once, not once per direction)
    int step[3][3] = {{-a.sx, 0, a.sx}, {-a.sy, 0, a.sy}, {-1, 0, 1}};
    if (a.per && a.after_odd) {
      const int x = idx / a.sx, rem = idx - x * a.sx, y = rem / a.sy, z = rem - y * a.sy;
      if (x == 1) step[0][0] = (a.nx - 1) * a.sx;
      if (x == a.nx) step[0][2] = (1 - a.nx) * a.sx;
      if (y == 1) step[1][0] = (a.ny - 1) * a.sy;
      if (y == a.ny) step[1][2] = (1 - a.ny) * a.sy;
      if (z == 1) step[2][0] = a.nz - 1;
      if (z == a.nz) step[2][2] = 1 - a.nz;
    }
    double r = 0., m[3] = {0., 0., 0.};
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const int slot = a.after_odd ? i : inv_dir<Q>(i);
      const int src = a.after_odd ? idx + step[0][1 + Lat<Q>::c[i][0]] + step[1][1 + Lat<Q>::c[i][1]] +
                                        step[2][1 + Lat<Q>::c[i][2]]
                                  : idx;
      double fi = double(CD::ld(a.f + slot * a.qs_bytes, static_cast<unsigned>(src) * sizeof(S)));
      fi *= Lat<Q>::w(i);
      r += fi;
#pragma unroll
      for (int d = 0; d < 3; ++d)
        if (Lat<Q>::c[i][d]) m[d] += Lat<Q>::c[i][d] > 0 ? fi : -fi;
    }
    s[0] += r;
    s[1] += m[0];
    s[2] += m[1];
    s[3] += m[2];
    s[4] += (m[0] * m[0] + m[1] * m[1] + m[2] * m[2]) / (2. * r);
  }
#pragma unroll
  for (int k = 0; k < 5; ++k) sh[k][threadIdx.x] = s[k];
  __syncthreads();
  for (int w = BLOCK / 2; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w)
#pragma unroll
      for (int k = 0; k < 5; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 5) a.partial[blockIdx.x * 5 + threadIdx.x] = sh[threadIdx.x][0];
}

__global__ __launch_bounds__(BLOCK) void k_reduce_final(const double *partial, int nblocks, double *out) {
  __shared__ double sh[5][BLOCK];
  double s[5] = {0., 0., 0., 0., 0.};
  for (int b = threadIdx.x; b < nblocks; b += BLOCK)
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] += partial[b * 5 + k];
#pragma unroll
  for (int k = 0; k < 5; ++k) sh[k][threadIdx.x] = s[k];
  __syncthreads();
  for (int w = BLOCK / 2; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w)
#pragma unroll
      for (int k = 0; k < 5; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 5) out[threadIdx.x] = sh[threadIdx.x][0];
}

template <int Q, class S, bool ODD, bool PER>
hipError_t step_w(bool wide, const StepLaunch &a, hipStream_t s) {
  const dim3 grid(a.hot.nchunks), block(a.hot.block);
  if (a.tile) {
    // the host sends only these: non-periodic, under 4 GiB, no per-cell relaxation, one cell per lane
    if (PER || wide || a.variant || a.cpl != 1 || a.hot.block != STEP_TILE) return hipErrorInvalidValue;
    if constexpr (!PER) hipLaunchKernelGGL((k_step_tile<Q, S, ODD>), grid, block, 0, s, a.hot, a.args);
    return hipGetLastError();
  }
  if (a.cpl > 1) {
    if (PER || wide || a.variant) return hipErrorInvalidValue;  // the host sends these one cell per lane
    if (a.cpl == 2)
      hipLaunchKernelGGL((k_step_run<Q, S, ODD, 2>), grid, block, 0, s, a.hot, a.args);
    else if (a.cpl == 4)
      hipLaunchKernelGGL((k_step_run<Q, S, ODD, 4>), grid, block, 0, s, a.hot, a.args);
    else
      return hipErrorInvalidValue;
    return hipGetLastError();
  }
  // (periodic lattices never choose between two slots: one addressing variant)
  if (a.variant >= 2) {  // the closure: D3Q19 with FP32 collision (checked by the host)
    if constexpr (Q == 19 && sizeof(typename Codec<S>::C) == 4) {
      if (wide && !PER && a.variant == 2)
        hipLaunchKernelGGL((k_step<Q, S, ODD, PER, !PER, 2>), grid, block, 0, s, a.hot, a.args);
      else if (a.variant == 2)
        hipLaunchKernelGGL((k_step<Q, S, ODD, PER, false, 2>), grid, block, 0, s, a.hot, a.args);
      else if (wide && !PER)
        hipLaunchKernelGGL((k_step<Q, S, ODD, PER, !PER, 3>), grid, block, 0, s, a.hot, a.args);
      else
        hipLaunchKernelGGL((k_step<Q, S, ODD, PER, false, 3>), grid, block, 0, s, a.hot, a.args);
      return hipGetLastError();
    } else {
      return hipErrorInvalidValue;
    }
  }
  if (a.variant == 1) {  // LBGKTurbulence
    if (wide && !PER)
      hipLaunchKernelGGL((k_step<Q, S, ODD, PER, !PER, 1>), grid, block, 0, s, a.hot, a.args);
    else
      hipLaunchKernelGGL((k_step<Q, S, ODD, PER, false, 1>), grid, block, 0, s, a.hot, a.args);
    return hipGetLastError();
  }
  if (wide && !PER)
    hipLaunchKernelGGL((k_step<Q, S, ODD, PER, !PER, 0>), grid, block, 0, s, a.hot, a.args);
  else
    hipLaunchKernelGGL((k_step<Q, S, ODD, PER, false, 0>), grid, block, 0, s, a.hot, a.args);
  return hipGetLastError();
}

template <int Q, class S, bool ODD, bool PER>
hipError_t batch_w(bool wide, const BatchLaunch &b, hipStream_t s) {
  const dim3 grid(b.nblocks), block(b.block);
  if (b.tile) {
    if (PER || wide || b.block != STEP_TILE) return hipErrorInvalidValue;  // the host sends only these
    if constexpr (!PER) hipLaunchKernelGGL((k_step_batch_tile<Q, S, ODD>), grid, block, 0, s, b.desc, b.ent);
    return hipGetLastError();
  }
  if (wide && !PER)
    hipLaunchKernelGGL((k_step_batch<Q, S, ODD, PER, !PER>), grid, block, 0, s, b.desc, b.ent);
  else
    hipLaunchKernelGGL((k_step_batch<Q, S, ODD, PER, false>), grid, block, 0, s, b.desc, b.ent);
  return hipGetLastError();
}

template <int Q, class S>
hipError_t step_q_s(bool odd, bool per, bool wide, const StepLaunch &a, hipStream_t s) {
  if (per) return odd ? step_w<Q, S, true, true>(wide, a, s) : step_w<Q, S, false, true>(wide, a, s);
  return odd ? step_w<Q, S, true, false>(wide, a, s) : step_w<Q, S, false, false>(wide, a, s);
}

// This object's template (the library holds one object per template).
template <template <int, class> class F, class... Args>
hipError_t dispatch(int dtype, Args &&...args) {
  switch (dtype) {
    case ASLHIP_F32: return F<ASLHIP_Q, float>::run(args...);
    case ASLHIP_F64: return F<ASLHIP_Q, double>::run(args...);
    case ASLHIP_BF16: return F<ASLHIP_Q, unsigned short>::run(args...);
    case ASLHIP_F16: return F<ASLHIP_Q, _Float16>::run(args...);
    default: return hipErrorInvalidValue;
  }
}

template <int Q, class S>
struct StepF {
  static hipError_t run(bool odd, bool per, bool wide, const StepLaunch &a, hipStream_t s) {
    return step_q_s<Q, S>(odd, per, wide, a, s);
  }
};
template <int Q, class S>
struct BatchF {
  static hipError_t run(bool odd, bool per, bool wide, const BatchLaunch &b, hipStream_t s) {
    if (per) return odd ? batch_w<Q, S, true, true>(wide, b, s) : batch_w<Q, S, false, true>(wide, b, s);
    return odd ? batch_w<Q, S, true, false>(wide, b, s) : batch_w<Q, S, false, false>(wide, b, s);
  }
};
template <int Q, class S>
struct VLinkF {
  static hipError_t run(const VLinkArgs &a, hipStream_t s) {
    if (a.nlinks == 0) return hipSuccess;
    hipLaunchKernelGGL((k_vlinks<Q, S>), dim3((a.nlinks + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, a);
    return hipGetLastError();
  }
};
template <int Q, class S>
struct InitF {
  static hipError_t run(const InitArgs &a, hipStream_t s) {
    hipLaunchKernelGGL((k_init<Q, S>), dim3((a.len + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, a);
    return hipGetLastError();
  }
};
template <int Q, class S>
struct SurfaceF {
  static hipError_t run(const SurfaceArgs &a, const StepHot &g, const StepArgs *args, hipStream_t s) {
    hipLaunchKernelGGL((k_surface<Q, S>), dim3((a.len + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, a, g, args);
    return hipGetLastError();
  }
};
template <int Q, class S>
struct VisF {
  static hipError_t run(const VisArgs &a, hipStream_t s) {
    if (Q == 27 && a.kind != ASLHIP_VIS_VELOCITY) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_vis<Q, S>), dim3((a.len + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, a);
    return hipGetLastError();
  }
};
template <int Q, class S>
struct WriteFF {
  static hipError_t run(const WriteFArgs &a, hipStream_t s) {
    hipLaunchKernelGGL((k_write_f<Q, S>), dim3((a.len + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, a);
    return hipGetLastError();
  }
};
template <int Q, class S>
struct UnpermuteF {
  static hipError_t run(const UnpermuteArgs &a, hipStream_t s) {
    if (a.first < 0 || a.count < 1 || a.first + a.count > a.len) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_unpermute<Q, S>), dim3((a.count + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, a);
    return hipGetLastError();
  }
};
template <int Q, class S>
struct ReduceF {
  static hipError_t run(const ReduceArgs &a, double *out, hipStream_t s) {
    const int nb = reduce_blocks(a.len);
    hipLaunchKernelGGL((k_reduce<Q, S>), dim3(nb), dim3(BLOCK), 0, s, a);
    hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(BLOCK), 0, s, a.partial, nb, out);
    return hipGetLastError();
  }
};

#if ASLHIP_Q == 19
template <class T>
void closure_features_w(bool odd, dim3 grid, const StepArgs *args, float *out, hipStream_t s) {
  if (odd)
    hipLaunchKernelGGL((k_closure_features<T, true>), grid, dim3(256), 0, s, args, out);
  else
    hipLaunchKernelGGL((k_closure_features<T, false>), grid, dim3(256), 0, s, args, out);
}
#endif

}  // namespace

#define ASLHIP_PASTE_(a, b) a##b
#define ASLHIP_PASTE(a, b) ASLHIP_PASTE_(a, b)
const KernelTable &ASLHIP_PASTE(kernels_q, ASLHIP_Q)() {
  static const KernelTable t = {
      [](int dt, bool odd, bool per, bool wide, const StepLaunch &a, hipStream_t s) {
        return dispatch<StepF>(dt, odd, per, wide, a, s);
      },
      [](int dt, bool odd, bool per, bool wide, const BatchLaunch &b, hipStream_t s) {
        return dispatch<BatchF>(dt, odd, per, wide, b, s);
      },
      [](int dt, const VLinkArgs &a, hipStream_t s) { return dispatch<VLinkF>(dt, a, s); },
      [](int dt, const InitArgs &a, hipStream_t s) { return dispatch<InitF>(dt, a, s); },
      [](int dt, const WriteFArgs &a, hipStream_t s) { return dispatch<WriteFF>(dt, a, s); },
      [](int dt, const SurfaceArgs &a, const StepHot &g, const StepArgs *args, hipStream_t s) {
        return dispatch<SurfaceF>(dt, a, g, args, s);
      },
      [](int dt, const VisArgs &a, hipStream_t s) { return dispatch<VisF>(dt, a, s); },
      [](int dt, const UnpermuteArgs &a, hipStream_t s) { return dispatch<UnpermuteF>(dt, a, s); },
      [](int dt, const ReduceArgs &a, double *out, hipStream_t s) { return dispatch<ReduceF>(dt, a, out, s); },
  };
  return t;
}

#if ASLHIP_Q == 19
hipError_t launch_closure_features(int dtype, bool odd, const StepArgs *args, long long ncell, float *out,
                                  hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((ncell + 255) / 256));
  switch (dtype) {
    case ASLHIP_F32: closure_features_w<float>(odd, grid, args, out, s); break;
    case ASLHIP_BF16: closure_features_w<unsigned short>(odd, grid, args, out, s); break;
    case ASLHIP_F16: closure_features_w<_Float16>(odd, grid, args, out, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
#endif

}  // namespace aslhip
