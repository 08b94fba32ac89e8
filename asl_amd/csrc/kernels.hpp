// kernels.hpp — argument blocks and launchers of the gfx950 LBGK kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "closure.hpp"
#include "lattice_consts.hpp"

namespace aslhip {

// Threads per workgroup of the step kernel (each thread one cell), at most;
// of its variant with runs of 2 or 4 cells per lane, at most; of its
// LDS-staged variant (one tile of STEP_TILE cells per workgroup), exactly.
constexpr int STEP_BLOCK = 1024;
constexpr int STEP_RUN_BLOCK = 512;
constexpr int STEP_TILE = 256;
// D3Q27 in FP64 holds 54 registers of populations alone: 1024 lanes per
// workgroup leave 128 registers and spill (periodic 128^3: 159 us per step),
// 512 leave it the 132 to 140 it takes (151 us).
constexpr int step_block(int q, int elem_bytes) { return q == 27 && elem_bytes == 8 ? 512 : STEP_BLOCK; }

// Step-kernel flags.
enum : unsigned {
  STEP_F_RHO = 1u,           // write rho of computed cells
  STEP_F_VEL = 2u,           // write u of computed cells
  STEP_F_RAW = 4u,           // read ghost links raw (no BC resolution)
  STEP_F_COMPRESSIBLE = 8u,  // compressible equilibrium (ASL default)
  STEP_F_OMEGA = 16u,        // rotating frame: momentum += (2/w) omega x momentum
  STEP_F_CLOSURE = 32u,      // per-cell relaxation time from the closure network
  STEP_F_CLOSURE_MFMA = 64u, // ... evaluated with BF16 matrix instructions
  STEP_F_TURB = 128u,        // LBGKTurbulence's relaxation limiter
};

// The part of a step's description that every wavefront reads before its
// first load: passed by value to the single-lattice kernels (scalar loads
// from the argument segment instead of a chain through device memory; with
// the face rule below 5.9 -> 4.6 us per step of a 16^3 box, D3Q19 FP32),
// read from StepArgs by the batch kernels.
//
// Work items are the interior cells j = (x ny + y) nz + z (0-based interior
// coordinates) in ASL's order, or runs of cpl of them; a chunk is `block`
// consecutive ones, so only the last chunk of a launch is partly empty,
// whatever the plane size.  A launch covers the interior planes that hold
// items first .. first + count - 1.  The LDS-staged tiles keep to the rows of
// one plane (chunks of STEP_TILE cells, ghost columns included).
//
// Face rule.  A link k into a cell is claimed by the faces the cell lies on
// whose inward direction e_f has c_k . e_f > 0; the BC executed last wins.
// Entry j (ascending execution slots; entries past the last one claim no
// links) names a face: fpos its bit, 4 bits per entry (0..5: X0 XE Y0 YE Z0
// ZE), flinks the links it claims, bit j of fbounce whether it bounces (else
// a constant); bit f of fvalued: face f has values to add or set, of fbfaces:
// its BC bounces.  Cells
// whose links this rule does not describe (next to map obstacles, computed
// ghost cells) carry CODE_FLUID_BC / CODE_GHOST and a link pattern instead.
struct StepHot {
  char *f;                    // first direction array
  const unsigned char *code;  // packed cell types
  unsigned long long qs;      // bytes between direction arrays
  unsigned long long mrow;    // floor(2^64 / row items) + 1 (0: one item per row): item -> row, see udivm
  unsigned long long mplane;  // floor(2^64 / ny) + 1 (0: one row): row -> plane
  unsigned long long mspan;   // floor(2^64 / (8 remap)) + 1: chunk -> group of 8 runs
  float inv_row, inv_ny;      // 1 / row items, 1 / ny (lane offsets, see lane_div)
  int sx, sy;                 // strides of the layout: Sy*Sz and Sz
  int nx, ny, nz;             // interior size
  int rowi;                   // items per row: nz (one cell per lane) or nz / cpl
  int block;                  // workgroup size (a multiple of 64, at most STEP_BLOCK)
  unsigned first, count;      // items of this launch
  int nchunks;                // workgroups of this launch
  int remap;                  // runs of that many chunks per XCD (see xcd_remap; 1: the hardware order)
  unsigned flags;             // STEP_F_*
  unsigned fpos;              // face of each entry of the face rule
  unsigned flinks[6];         // links each entry claims
  unsigned fbounce;           // bit j: entry j bounces
  unsigned fvalued, fbfaces;  // bit f: face f has values / bounces
};

// One fused collide+stream pass (AA pattern) over the ghost-inclusive block.
struct StepArgs {
  StepHot g;                  // one cell per lane over the whole lattice (runs of cells: cpl > 1)
  unsigned qs32;              // bytes between direction arrays (if all fit in 4 GiB)
  int len;                    // ghost-inclusive cell count
  int bpp;                    // LDS-staged tiles: chunks per plane
  unsigned long long zmagic;  // ceil(2^40 / sy): row = (off * zmagic) >> 40 (tiles)
  int cpl;                    // cells per lane along z
  int tile;                   // 1: LDS-staged tiles (block = STEP_TILE, cpl = 1)
  unsigned fset;              // bit f: face f has a BC
  unsigned fbeats[6];         // per face: the faces that own links they share with it (BC executed later, or the same BC)
  float fval32[6][28];        // per face and direction: addend / constant (FP32 lattices)
  double fval64[6][28];       // the same for FP64 lattices
  float om32[3];              // angular velocity of the frame (STEP_F_OMEGA)
  double om64[3];
  const ClosureParams *cl;    // closure network (STEP_F_CLOSURE)
  float cl_tau0;              // 3 nu + 1/2 in float
  float nu32;                 // viscosity (STEP_F_TURB)
  double nu64;
  const unsigned short *pat;  // link pattern of CODE_FLUID_BC / CODE_GHOST cells
  const LinkRec *rec;         // link patterns
  const unsigned char *mode;  // resolution mode of each BC slot
  const void *val;            // [slot][Q] addend or constant, compute type
  void *rho, *u;              // macroscopic outputs (ASL layout)
  double w;                   // relaxation rate (exact in the compute type)
};

// Several lattices advanced by one launch of the step kernel: desc[l] is
// lattice l's StepArgs (device memory), workgroup b works on lattice lat[b],
// chunk b - first[lat[b]].
struct BatchLaunch {
  const StepArgs *desc;
  const uint2 *ent;  // per workgroup: lattice, chunk
  int nblocks;
  int block;
  int tile;  // 1: LDS-staged tiles (block = STEP_TILE; non-periodic, under 4 GiB)
};

// Boundary-link kernel entries (velocity map BCs).
struct VLink {
  int g;              // ghost cell (linear index)
  unsigned comp;      // directions i whose neighbour g+c_i is a computation node
  unsigned own;       // links g -> g+c_i this BC resolves
  int slot;           // BC slot (parameters in VLinkArgs::bc)
};

struct VLinkBC {
  double u[3];
  double omega[3], centre[3];
  int has_rot;
};

struct VLinkArgs {
  char *f;
  long long qs_bytes;
  int sx, sy;
  const VLink *links;
  int nlinks;
  const VLinkBC *bc;  // indexed by slot
  double dx, pos0[3]; // position of ghost-inclusive index 0 is pos0 - dx
  int after_odd;      // state after an odd step (else after an even one / init)
};

struct InitArgs {
  char *f;
  long long qs_bytes;
  int len;
  double rho0, u0[3];       // constants (used when rho_in/u_in are null)
  const void *rho_in, *u_in;  // fields in the macroscopic type
  void *rho, *u;
};

// Surface force (3 x len) or flux (len) of a level-set map, in the macroscopic
// type, from the populations after the last step.
struct SurfaceArgs {
  const float *map;
  void *out;
  int len;
  int per;                // periodic lattice
  int after_odd;          // state after an odd step (else after an even one / init)
  int flux;               // 1: ComputeSurfaceFluxMap, 0: ComputeSurfaceForceMap
};

// Visualisation fill of a lattice's rho or u in place at the guarded boundary
// nodes of a map (map <= 0 and > -0.9999): ASLHIP_VIS_NOSLIP_VEL,
// ASLHIP_VIS_NOSLIP_RHO or ASLHIP_VIS_VELOCITY (include/aslhip.h).
struct VisArgs {
  const float *map;    // len values, ASL layout
  void *rho, *u;       // macroscopic type
  int kind;
  int len, sx, sy;
  double u0[3];        // ASLHIP_VIS_VELOCITY: the velocity (without rotation)
  double rot[6];       // ASLHIP_VIS_VELOCITY with has_rot: axis, centre
  int has_rot;
  double dx, pos0[3];  // position of ghost-inclusive index 0 is pos0 - dx
};

// Populations from a host view (Q x len, f_i of each cell) into the layout a
// step of odd parity reads (slot (x, inv(i))), with rho and u of each cell.
struct WriteFArgs {
  char *f;
  long long qs_bytes;
  int len;
  int compressible;
  const void *in;  // Q * len macroscopic type
  void *rho, *u;
};

// The cells first .. first + count - 1 (count = len: all of them) go to
// out[i * count + cell - first].  per: periodic lattice of interior size
// nx x ny x nz (after an odd step the populations of a face cell sit in the
// wrapped neighbour's slots).
struct UnpermuteArgs {
  const char *f;
  long long qs_bytes;
  int sx, sy, len;
  int per, nx, ny, nz;
  int after_odd;
  int first, count;
  void *out;  // Q * count macroscopic type
};

struct ReduceArgs {
  const char *f;
  long long qs_bytes;
  int sx, sy, len;
  int per, nx, ny, nz;
  int after_odd;
  const unsigned char *code;
  double *partial;  // 5 per block
};

// One step of one lattice: hot describes this launch, args points to the
// lattice's StepArgs in device memory.
struct StepLaunch {
  StepHot hot;
  const StepArgs *args;
  int variant;   // per-cell relaxation: 0 none, 1 LBGKTurbulence, 2 / 3 the closure on the matrix cores / in FP32
  int cpl;       // cells per lane (2 or 4: the run variant; non-periodic, under 4 GiB, no closure)
  int tile;      // 1: LDS-staged tiles of STEP_TILE cells (same restrictions, cpl 1, block STEP_TILE)
};

// The launchers of one template's object (kernels.hip compiled with ASLHIP_Q
// 15, 19 or 27); first argument: population type.
struct KernelTable {
  hipError_t (*step)(int, bool odd, bool periodic, bool wide, const StepLaunch &, hipStream_t);
  hipError_t (*batch)(int, bool odd, bool periodic, bool wide, const BatchLaunch &, hipStream_t);
  hipError_t (*vlinks)(int, const VLinkArgs &, hipStream_t);
  hipError_t (*init)(int, const InitArgs &, hipStream_t);
  hipError_t (*write_f)(int, const WriteFArgs &, hipStream_t);
  hipError_t (*surface)(int, const SurfaceArgs &, const StepHot &, const StepArgs *, hipStream_t);
  hipError_t (*vis)(int, const VisArgs &, hipStream_t);
  hipError_t (*unpermute)(int, const UnpermuteArgs &, hipStream_t);
  hipError_t (*reduce)(int, const ReduceArgs &, double *out, hipStream_t);
};
const KernelTable &kernels_q15();
const KernelTable &kernels_q19();
const KernelTable &kernels_q27();

// wide: the populations span more than 4 GiB (64-bit per-lane addresses).
hipError_t launch_step(int q, int dtype, bool odd, bool periodic, bool wide, const StepLaunch &a, hipStream_t s);
hipError_t launch_step_batch(int q, int dtype, bool odd, bool periodic, bool wide, const BatchLaunch &b,
                             hipStream_t s);
hipError_t launch_vlinks(int q, int dtype, const VLinkArgs &a, hipStream_t s);
// Closure features (7 floats per interior cell) of a periodic D3Q19 lattice
// with FP32 collision; args: the lattice's StepArgs in device memory.
hipError_t launch_closure_features(int dtype, bool odd, const StepArgs *args, long long ncell, float *out,
                                  hipStream_t s);
hipError_t launch_init(int q, int dtype, const InitArgs &a, hipStream_t s);
hipError_t launch_write_f(int q, int dtype, const WriteFArgs &a, hipStream_t s);
// g, args: the lattice's step description (args in device memory).
hipError_t launch_surface(int q, int dtype, const SurfaceArgs &a, const StepHot &g, const StepArgs *args,
                          hipStream_t s);
hipError_t launch_vis(int q, int dtype, const VisArgs &a, hipStream_t s);
hipError_t launch_unpermute(int q, int dtype, const UnpermuteArgs &a, hipStream_t s);
// The allocation-free staging array (ASLHIP_NOALLOC_SCRATCH_BYTES bytes of
// device memory in the library's code object, one per device): its address
// on the current device, looked up once per device.
hipError_t noalloc_scratch(void **ptr);
// partial must hold 5 * reduce_blocks(len) doubles; out: 5 doubles (device).
int reduce_blocks(int len);
hipError_t launch_reduce(int q, int dtype, const ReduceArgs &a, double *out, hipStream_t s);

}  // namespace aslhip
