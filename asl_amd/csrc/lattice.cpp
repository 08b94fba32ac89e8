// lattice.cpp — C ABI of the gfx950 LBGK library (include/aslhip.h).
//
// Host-side state of one lattice: device buffers, the boundary-condition
// list, the driver's execute order, and the finalize step that turns ASL's
// ghost-fill BCs into per-link resolution tables for the fused step kernel.
//
// How ASL's BC semantics map onto links.  ASL streams by pulling
// f_k(x) <- f_k(x - c_k) after the BCs have overwritten some ghost entries
// (g, k) (src/num/aslLBGK.cxx:237-250; src/num/aslLBGKBC.cxx).  So the value a
// computation node x receives along direction k is the BC value of entry
// (x - c_k, k) if some executed BC writes that entry (the last one executed
// wins), and otherwise the collided population of x - c_k.  finalize()
// resolves every incoming link of every computed cell that way, in the
// driver's execute order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/aslhip.h"
#include "kernels.hpp"
#include "lattice_consts.hpp"
#include "status.hpp"
#include "transfer.hpp"

using namespace aslhip;

namespace {
thread_local std::string g_err;
}  // namespace

int aslhip::fail(int code, const char *fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}

namespace {

// Round to the nearest BF16 value (ties to even), kept as a float.
float bf16_round(float x) {
  uint32_t u;
  std::memcpy(&u, &x, 4);
  if ((u & 0x7f800000u) == 0x7f800000u) return x;  // inf / nan unchanged
  u += 0x7fffu + ((u >> 16) & 1u);
  u &= 0xffff0000u;
  std::memcpy(&x, &u, 4);
  return x;
}

struct Templ {
  int Q;
  int c[27][3];
  double w[27];
  int inv[27];
};

template <int Q>
Templ make_templ_q() {
  Templ t;
  t.Q = Q;
  for (int i = 0; i < Q; ++i) {
    for (int d = 0; d < 3; ++d) t.c[i][d] = Lat<Q>::c[i][d];
    t.w[i] = Lat<Q>::w(i);
    t.inv[i] = inv_dir<Q>(i);
  }
  return t;
}

Templ make_templ(int q) {
  if (q == 15) return make_templ_q<15>();
  if (q == 27) return make_templ_q<27>();
  return make_templ_q<19>();
}

struct BCDesc {
  int kind = 0;
  unsigned faces = 0;
  double p = 0, u[3] = {0, 0, 0};
  bool has_rot = false;
  double rot[6] = {0, 0, 0, 0, 0, 0};
  std::vector<float> map, cd;
  bool is_map() const { return kind >= ASLHIP_BC_NOSLIP_MAP; }
};

// v . c_i with zero terms left out, in type C.
template <class C>
C dot_c(const Templ &t, const C *u, int i) {
  C a = C(0);
  bool first = true;
  for (int d = 0; d < 3; ++d) {
    if (t.c[i][d] == 0) continue;
    C v = t.c[i][d] > 0 ? u[d] : -u[d];
    a = first ? v : a + v;
    first = false;
  }
  return a;
}

}  // namespace

struct aslhip_lattice {
  int n[3] = {0, 0, 0};
  int S[3] = {0, 0, 0};
  int sx = 0, sy = 0, len = 0;
  int Q = 19, dtype = ASLHIP_F32;
  bool periodic = false;
  Templ t;
  size_t selem = 4, melem = 4, celem = 4;  // storage / macroscopic / compute element bytes
  long long qs_bytes = 0;
  hipStream_t stream = nullptr;
  int device = -1;  // the device current at creation (its memory and stream live there)
  // device buffers
  char *f = nullptr;
  void *rho = nullptr, *u = nullptr;
  unsigned char *code = nullptr;
  unsigned short *pat = nullptr;
  LinkRec *rec = nullptr;
  unsigned char *mode = nullptr;
  void *val = nullptr;
  VLink *vl = nullptr;
  VLinkBC *vlbc = nullptr;
  double *red_partial = nullptr, *red_out = nullptr;
  // step arguments of even and odd steps (they differ when only even steps run tiles)
  StepArgs *d_args = nullptr;
  std::vector<StepArgs> h_args;  // host copy of d_args (empty: not uploaded yet)
  StepHot h_direct;              // one cell per lane over the whole lattice (plane ranges are cut from it)
  // Captured runs of plain steps (the velocity-map link fills included):
  // full chunks of ASLHIP_GRAPH_CHUNK steps and the shorter remainders of
  // step counts that are not a multiple of it, each for a starting parity
  // and the step flags it was captured with; dropped after finalize.
  struct Graph {
    int n;
    bool odd;
    unsigned fl;
    hipGraphExec_t exec;
  };
  std::vector<Graph> graphs;
  int nvl = 0;
  // parameters
  double nu = 0.1;
  bool compressible = true, comp_rho = true, comp_vel = true;
  bool has_omega = false;
  double omega[3] = {0., 0., 0.};
  // learned closure (network parameters in device memory)
  bool has_closure = false;
  bool turbulence = false;   // LBGKTurbulence
  bool closure_mfma = true;  // evaluate the network with BF16 matrix instructions
  ClosureParams *d_cl = nullptr;
  float *d_feat = nullptr;  // closure features scratch (7 per interior cell)
  int queued = 0;   // step launches since the host last waited for the stream
  Scratch view;     // one view of the populations (read_f, write_f): Q len macroscopic values
  Scratch surface;  // surface force / flux: result (3 len macroscopic values), then the map (len floats)
  double dx = 1., pos0[3] = {0., 0., 0.};
  // a stream reading rho / u through aslhip_macro_device: the next work that
  // writes them waits for what it has queued by then
  hipStream_t consumer = nullptr;
  hipEvent_t ev_macro = nullptr, ev_consumer = nullptr;
  // visualisation fills (aslhip_vis_add): kind, device copy of the map, velocity
  struct Vis {
    int kind;
    float *map;
    double u[3];
    bool has_rot;
    double rot[6];
  };
  std::vector<Vis> vis;
  // BCs and order
  std::vector<BCDesc> bcs;
  std::vector<int> order, pending;
  bool dirty = true;
  bool initialized = false;
  bool fresh = false;        // no step since init
  bool bc_since_init = false;
  bool next_odd = true;
  // a step requested with ASLHIP_STEP_DEFER that has not run yet
  bool deferred = false;
  bool deferred_raw = false;
  bool deferred_first = false;
  // launch tuning
  int tune_block = 512;   // workgroup size (measured best with runs of 4 chunks per XCD)
  bool block_set = false; // tune_block was chosen by the user or the autotuner
  bool force_wide = false;  // 64-bit addressing on any size (ASLHIP_TUNE_WIDE)
  int tune_remap = 4;  // chunks per XCD run, where xcd_run does not choose
  bool remap_set = false;  // tune_remap was chosen by the user or the autotuner
  int tune_cpl = 0;    // cells per lane along z: 0 automatic, else 1, 2 or 4 (ASLHIP_TUNE_CPL)
  int tune_lds = -1;   // LDS-staged tiles: 0 off, 1 every step, 2 even steps, -1 automatic (ASLHIP_TUNE_LDS)
  int tune_sweep = -1; // sweeps: window in KiB, 0 off, -1 automatic (ASLHIP_TUNE_SWEEP_KB)
  bool vmap_skip_outer = false;  // velocity-map averages skip outer-layer neighbours (opt-in)
  // face rule: per face slot * 4 + mode of the winning slice BC, and values
  int fface[6] = {0, 0, 0, 0, 0, 0};
  float fval32[6][27] = {};
  double fval64[6][27] = {};
  // stats
  long long n_counted = 0, n_computed = 0, n_boundary = 0, n_patterns = 0;
  std::vector<unsigned char> h_code;

  int idx(int x, int y, int z) const { return x * sx + y * sy + z; }
};

namespace {

int check(aslhip_lattice *h) {
  if (!h) return fail(ASLHIP_EINVAL, "ASL ERROR: null lattice handle");
  return 0;
}

// Destroys the captured runs once the stream has finished any replay of them.
void drop_graphs(aslhip_lattice *h) {
  if (!h->graphs.empty() && h->stream) (void)hipStreamSynchronize(h->stream);
  for (auto &g : h->graphs) (void)hipGraphExecDestroy(g.exec);
  h->graphs.clear();
}

void free_all(aslhip_lattice *h) {
  drop_graphs(h);
  scratch_drop(h->view);
  scratch_drop(h->surface);
  void *ptrs[] = {h->f,  h->rho,  h->u,           h->code,         h->pat, h->rec, h->mode,
                  h->val, h->vl, h->vlbc, h->red_partial, h->red_out, h->d_args, h->d_cl, h->d_feat};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  for (auto &v : h->vis)
    if (v.map) (void)hipFree(v.map);
  if (h->ev_macro) (void)hipEventDestroy(h->ev_macro);
  if (h->ev_consumer) (void)hipEventDestroy(h->ev_consumer);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  transfer_drop();
}

// Work about to be queued on the lattice's stream may overwrite rho / u (and
// the populations): it first waits for whatever the consumer stream named in
// aslhip_macro_device has queued up to now.
int order_after_consumer(aslhip_lattice *h) {
  if (!h->consumer) return 0;
  HIPCHK(hipEventRecord(h->ev_consumer, h->consumer));
  HIPCHK(hipStreamWaitEvent(h->stream, h->ev_consumer, 0));
  h->consumer = nullptr;
  return 0;
}

// Relaxation rate w = 1/(3 nu + 1/2) in the compute type
// (src/num/aslLBGK.cxx:203).
// StepArgs::flags bits fixed by the lattice's parameters.
unsigned base_flags(const aslhip_lattice *h) {
  return (h->compressible ? STEP_F_COMPRESSIBLE : 0u) | (h->has_omega ? STEP_F_OMEGA : 0u) |
         (h->has_closure ? STEP_F_CLOSURE : 0u) | (h->has_closure && h->closure_mfma ? STEP_F_CLOSURE_MFMA : 0u) |
         (h->turbulence ? STEP_F_TURB : 0u);
}

double relaxation(const aslhip_lattice *h) {
  if (h->dtype == ASLHIP_F64) return 1. / (3. * h->nu + .5);
  const float nu = static_cast<float>(h->nu);
  return static_cast<double>(1.f / (3.f * nu + .5f));
}

// Slot values of one BC in the compute type C.
template <class C>
void bc_values(const aslhip_lattice *h, const BCDesc &b, unsigned char &md, C *val) {
  const Templ &t = h->t;
  const C u[3] = {C(b.u[0]), C(b.u[1]), C(b.u[2])};
  const C p = C(b.p);
  for (int k = 0; k < t.Q; ++k) val[k] = C(0);
  switch (b.kind) {
    case ASLHIP_BC_NOSLIP:
    case ASLHIP_BC_NOSLIP_MAP:
      md = MODE_BOUNCE;
      break;
    case ASLHIP_BC_CONSTANT_VELOCITY:  // f_kbar(p) + 6.*(velocity*c_k)
      md = MODE_BOUNCE;
      for (int k = 1; k < t.Q; ++k) val[k] = C(6.) * dot_c(t, u, k);
      break;
    case ASLHIP_BC_CONSTANT_PRESSURE:
      md = MODE_CONST;
      for (int k = 1; k < t.Q; ++k) val[k] = p;
      break;
    case ASLHIP_BC_CONSTANT_PRESSURE_VELOCITY:  // pressure + 3.*(velocity*c_k)
      md = MODE_CONST;
      for (int k = 1; k < t.Q; ++k) val[k] = p + C(3.) * dot_c(t, u, k);
      break;
    case ASLHIP_BC_PRESSURE_VELOCITY_MAP: {  // src/num/aslLBGKBC.cxx:400-415
      md = MODE_CONST;
      C uu = u[0] * u[0];
      uu = uu + u[1] * u[1];
      uu = uu + u[2] * u[2];
      for (int k = 1; k < t.Q; ++k) {
        const C a = dot_c(t, u, k);
        if (h->compressible) {
          val[k] = ((p + (C(3.) * p) * a) + ((C(4.5) * p) * a) * a) - (C(1.5) * p) * uu;
        } else {
          const C u3[3] = {C(3.) * u[0], C(3.) * u[1], C(3.) * u[2]};
          val[k] = ((p + dot_c(t, u3, k)) + (C(4.5) * a) * a) - C(1.5) * uu;
        }
      }
      break;
    }
    case ASLHIP_BC_VELOCITY_MAP:
      md = MODE_LINK;
      break;
    default:
      md = MODE_NONE;
  }
}

// Out-of-block-safe map read (src/acl/aclMath/aclMathAlg.cxx:84-94).
inline float map_safe(const std::vector<float> &m, long long i, long long len, float out) {
  return (i < 0 || i > len - 1) ? out : m[(size_t)i];
}

// isComputationNode (src/num/aslBCond.cxx:204-211): map > 0 [&& cdomain > 0].
inline bool comp_node(const BCDesc &b, long long i, long long len) {
  bool r = map_safe(b.map, i, len, -.9f) > 0.f;
  if (!b.cd.empty()) r = r && map_safe(b.cd, i, len, -1.f) > 0.f;
  return r;
}

struct PatHash {
  size_t operator()(const std::string &s) const { return std::hash<std::string>()(s); }
};

// allow_open: the next step reads ghost links raw (the first step after
// initF with no BC executed before it), so links no BC fills are allowed; the
// lattice is finalized again before any later step.
int finalize_impl(aslhip_lattice *h, bool allow_open = false) {
  drop_graphs(h);  // they hold the link tables replaced below
  const Templ &t = h->t;
  const int Q = t.Q, len = h->len;
  std::vector<unsigned char> code(len, CODE_SKIP);
  std::vector<unsigned short> pat(len, 0);
  std::vector<LinkRec> recs(1);
  std::memset(&recs[0], 0, sizeof(LinkRec));
  std::vector<VLink> vlinks;
  std::vector<VLinkBC> vlbc(256);
  const int nord = static_cast<int>(h->order.size());
  if (nord > 254) return fail(ASLHIP_EINVAL, "ASL ERROR: more than 254 boundary-condition executions per step");
  int off[27];
  for (int k = 0; k < Q; ++k) off[k] = t.c[k][0] * h->sx + t.c[k][1] * h->sy + t.c[k][2];
  auto interior = [&](int x, int y, int z) {
    return x >= 1 && x <= h->n[0] && y >= 1 && y <= h->n[1] && z >= 1 && z <= h->n[2];
  };

  h->n_counted = h->n_computed = h->n_boundary = 0;
  if (h->periodic) {
    if (nord > 0 || !h->bcs.empty())
      return fail(ASLHIP_EINVAL, "ASL ERROR: boundary conditions on a periodic lattice");
    for (int x = 1; x <= h->n[0]; ++x)
      for (int y = 1; y <= h->n[1]; ++y)
        for (int z = 1; z <= h->n[2]; ++z) code[h->idx(x, y, z)] = CODE_FLUID;
    h->n_counted = h->n_computed = (long long)h->n[0] * h->n[1] * h->n[2];
  } else {
    // BC of each order position; map BCs applied.
    std::vector<const BCDesc *> ob(nord);
    for (int o = 0; o < nord; ++o) ob[o] = &h->bcs[h->order[o]];
    std::vector<int> map_pos;
    for (int o = 0; o < nord; ++o)
      if (ob[o]->is_map()) map_pos.push_back(o);
    static const int face_dir[6] = {1, 4, 2, 5, 3, 6};  // X0 XE Y0 YE Z0 ZE: vectors[1..6]

    // Slot (order position + 1) of the last executed BC that writes entry
    // (x - c_k, k), for interior x; 0 if none.
    auto resolve = [&](int x, int y, int z, int k) -> int {
      const int i = h->idx(x, y, z);
      const int p[3] = {x, y, z};
      for (int o = nord - 1; o >= 0; --o) {
        const BCDesc &b = *ob[o];
        if (!b.is_map()) {
          // addSliceX0 ... addSliceZE (src/num/aslBCond.cxx:373-493)
          for (int fc = 0; fc < 6; ++fc) {
            if (!(b.faces & (1u << fc))) continue;
            const int axis = fc / 2;
            const int layer = (fc % 2 == 0) ? 1 : h->S[axis] - 2;
            const int *e = t.c[face_dir[fc]];
            if (p[axis] == layer && t.c[k][0] * e[0] + t.c[k][1] * e[1] + t.c[k][2] * e[2] > 0) return o + 1;
          }
        } else {
          // map guard and predicates (src/num/aslLBGKBC.cxx:235-251)
          const float mg = b.map[(size_t)(i - off[k])];
          if (mg <= 0.f && mg > -.9999f && comp_node(b, i, len)) return o + 1;
        }
      }
      return 0;
    };

    std::vector<unsigned char> computed(len, 0), counted(len, 0);
    for (int x = 1; x <= h->n[0]; ++x)
      for (int y = 1; y <= h->n[1]; ++y)
        for (int z = 1; z <= h->n[2]; ++z) {
          const int i = h->idx(x, y, z);
          bool solid = false;
          for (int o : map_pos)
            if (ob[o]->map[(size_t)i] <= 0.f) solid = true;
          computed[i] = counted[i] = solid ? 0 : 1;
        }
    // Closure: a cell that is not computed but sends an unresolved link into
    // a computed cell must be computed too (ASL collides every cell).
    for (bool changed = true; changed;) {
      changed = false;
      for (int x = 0; x < h->S[0]; ++x)
        for (int y = 0; y < h->S[1]; ++y)
          for (int z = 0; z < h->S[2]; ++z) {
            const int s = h->idx(x, y, z);
            if (computed[s]) continue;
            for (int k = 1; k < Q; ++k) {
              const int X = x + t.c[k][0], Y = y + t.c[k][1], Z = z + t.c[k][2];
              if (!interior(X, Y, Z)) continue;
              if (!computed[h->idx(X, Y, Z)] || resolve(X, Y, Z, k) != 0) continue;
              if (!interior(x, y, z)) {
                if (allow_open) continue;
                return fail(ASLHIP_EUNDEF,
                            "ASL ERROR: no boundary condition fills the ghost link (%d,%d,%d) -> (%d,%d,%d) "
                            "(ASL would stream uninitialised memory into the block)",
                            x - 1, y - 1, z - 1, X - 1, Y - 1, Z - 1);
              }
              computed[s] = 1;
              changed = true;
              break;
            }
          }
    }

    // Face rule: the last executed slice BC on each face claims the links
    // that enter through that face (see StepArgs).
    int fslot[6] = {0, 0, 0, 0, 0, 0};
    for (int o = 0; o < nord; ++o)
      if (!ob[o]->is_map())
        for (int fc = 0; fc < 6; ++fc)
          if (ob[o]->faces & (1u << fc)) fslot[fc] = o + 1;
    auto face_rule = [&](int x, int y, int z, int k) -> int {
      const int p[3] = {x, y, z};
      int best = 0;
      for (int d = 0; d < 3; ++d) {
        const int cd = t.c[k][d];
        if (cd == 0) continue;
        const int fc = 2 * d + (cd > 0 ? 0 : 1);
        const bool on = (fc % 2 == 0) ? p[d] == 1 : p[d] == h->n[d];
        if (on && fslot[fc] > best) best = fslot[fc];
      }
      return best;
    };
    for (int fc = 0; fc < 6; ++fc) {
      h->fface[fc] = 0;
      for (int k = 0; k < 27; ++k) {
        h->fval32[fc][k] = 0.f;
        h->fval64[fc][k] = 0.;
      }
      if (!fslot[fc]) continue;
      const BCDesc &b = *ob[fslot[fc] - 1];
      unsigned char md = MODE_NONE;
      double v64[27];
      float v32[27];
      bc_values<double>(h, b, md, v64);
      bc_values<float>(h, b, md, v32);
      h->fface[fc] = fslot[fc] * 4 + md;
      for (int k = 0; k < Q; ++k) {
        h->fval32[fc][k] = v32[k];
        h->fval64[fc][k] = v64[k];
      }
    }

    // Cells that some map BC treats as ghost nodes (map <= 0), any layer.
    std::vector<unsigned char> solid_any(len, 0);
    for (int o : map_pos)
      for (int i = 0; i < len; ++i)
        if (ob[o]->map[(size_t)i] <= 0.f) solid_any[i] = 1;
    std::unordered_map<std::string, int, PatHash> pid;
    for (int x = 1; x <= h->n[0]; ++x)
      for (int y = 1; y <= h->n[1]; ++y)
        for (int z = 1; z <= h->n[2]; ++z) {
          const int i = h->idx(x, y, z);
          if (!computed[i]) continue;
          LinkRec r;
          std::memset(&r, 0, sizeof r);
          bool any = false;
          // A link into x can only be BC-resolved if x is in a face layer or
          // its source x - c_k is a map ghost node.
          bool near = x == 1 || x == h->n[0] || y == 1 || y == h->n[1] || z == 1 || z == h->n[2];
          for (int k = 1; k < Q && !near && !map_pos.empty(); ++k) near = solid_any[i - off[k]] != 0;
          for (int k = 1; k < Q && near; ++k) {
            const int s = resolve(x, y, z, k);
            r.slot[k] = static_cast<unsigned char>(s);
            // the step kernel resolves this link itself unless the face
            // rule disagrees with the full resolution
            any = any || s != face_rule(x, y, z, k);
          }
          // Outgoing link k of a computed ghost cell: skip it if its receiver
          // resolves it (computation nodes are never the source of a BC entry).
          for (int k = 1; k < Q && !counted[i]; ++k) {
            const int X = x + t.c[k][0], Y = y + t.c[k][1], Z = z + t.c[k][2];
            if (interior(X, Y, Z) && computed[h->idx(X, Y, Z)] && resolve(X, Y, Z, k) != 0) {
              r.skip |= 1u << k;
              any = true;
            }
          }
          ++h->n_computed;
          if (counted[i]) ++h->n_counted;
          if (!any && counted[i]) {
            code[i] = CODE_FLUID;
            continue;
          }
          code[i] = counted[i] ? CODE_FLUID_BC : CODE_GHOST;
          if (counted[i]) ++h->n_boundary;
          std::string key(reinterpret_cast<const char *>(&r), sizeof r);
          auto it = pid.find(key);
          int id;
          if (it == pid.end()) {
            id = static_cast<int>(recs.size());
            if (id > 65535) return fail(ASLHIP_EINVAL, "ASL ERROR: more than 65535 distinct boundary link patterns");
            recs.push_back(r);
            pid.emplace(key, id);
          } else {
            id = it->second;
          }
          pat[i] = static_cast<unsigned short>(id);
        }

    // Boundary-link entries of velocity map BCs.
    for (int o = 0; o < nord; ++o) {
      const BCDesc &b = *ob[o];
      if (b.kind != ASLHIP_BC_VELOCITY_MAP) continue;
      VLinkBC &vb = vlbc[o + 1];
      for (int d = 0; d < 3; ++d) {
        vb.u[d] = b.u[d];
        vb.omega[d] = b.rot[d];
        vb.centre[d] = b.rot[3 + d];
      }
      vb.has_rot = b.has_rot ? 1 : 0;
      for (int g = 0; g < len; ++g) {
        const float mg = b.map[(size_t)g];
        if (!(mg <= 0.f && mg > -.9999f)) continue;
        VLink l{g, 0u, 0u, o + 1};
        const int gx = g / h->sx, gy = (g % h->sx) / h->sy, gz = g % h->sy;
        for (int i = 1; i < Q; ++i) {
          const long long p = (long long)g + off[i];
          if (!comp_node(b, p, len)) continue;
          l.comp |= 1u << i;
          const int X = gx + t.c[i][0], Y = gy + t.c[i][1], Z = gz + t.c[i][2];
          if (interior(X, Y, Z) && computed[h->idx(X, Y, Z)] && h->idx(X, Y, Z) == p &&
              resolve(X, Y, Z, i) == o + 1)
            l.own |= 1u << i;
        }
        if (!l.own) continue;
        for (int i = 1; i < Q; ++i) {
          if (!((l.comp >> i) & 1u)) continue;
          const int X = gx + t.c[i][0], Y = gy + t.c[i][1], Z = gz + t.c[i][2];
          if (!interior(X, Y, Z) && h->vmap_skip_outer) {
            l.comp &= ~(1u << i);  // left out of the density average (opt-in)
            continue;
          }
          if (!interior(X, Y, Z) || !computed[h->idx(X, Y, Z)])
            return fail(ASLHIP_EUNDEF,
                        "ASL ERROR: velocity map BC at ghost (%d,%d,%d) averages a neighbour that is not a "
                        "computed cell",
                        gx - 1, gy - 1, gz - 1);
        }
        vlinks.push_back(l);
      }
    }
  }
  h->n_patterns = static_cast<long long>(recs.size()) - 1;

  // Slot tables.
  std::vector<unsigned char> mode(256, MODE_NONE);
  std::vector<char> val(256 * (size_t)Q * h->celem, 0);
  for (int o = 0; o < nord; ++o) {
    const BCDesc &b = h->bcs[h->order[o]];
    if (h->celem == 8)
      bc_values<double>(h, b, mode[o + 1], reinterpret_cast<double *>(val.data()) + (size_t)(o + 1) * Q);
    else
      bc_values<float>(h, b, mode[o + 1], reinterpret_cast<float *>(val.data()) + (size_t)(o + 1) * Q);
  }

  // Upload.
  HIPCHK(hipMemcpyAsync(h->code, code.data(), len, hipMemcpyHostToDevice, h->stream));
  HIPCHK(hipMemcpyAsync(h->pat, pat.data(), (size_t)len * 2, hipMemcpyHostToDevice, h->stream));
  if (h->rec) HIPCHK(hipFree(h->rec));
  h->rec = nullptr;
  HIPCHK(device_alloc(&h->rec, recs.size() * sizeof(LinkRec)));
  HIPCHK(hipMemcpyAsync(h->rec, recs.data(), recs.size() * sizeof(LinkRec), hipMemcpyHostToDevice, h->stream));
  HIPCHK(hipMemcpyAsync(h->mode, mode.data(), 256, hipMemcpyHostToDevice, h->stream));
  HIPCHK(hipMemcpyAsync(h->val, val.data(), val.size(), hipMemcpyHostToDevice, h->stream));
  if (h->vl) HIPCHK(hipFree(h->vl));
  h->vl = nullptr;
  h->nvl = static_cast<int>(vlinks.size());
  if (h->nvl) {
    HIPCHK(device_alloc(&h->vl, vlinks.size() * sizeof(VLink)));
    HIPCHK(hipMemcpyAsync(h->vl, vlinks.data(), vlinks.size() * sizeof(VLink), hipMemcpyHostToDevice, h->stream));
  }
  HIPCHK(hipMemcpyAsync(h->vlbc, vlbc.data(), 256 * sizeof(VLinkBC), hipMemcpyHostToDevice, h->stream));
  HIPCHK(hipStreamSynchronize(h->stream));
  h->h_code.swap(code);
  h->dirty = allow_open;
  return 0;
}

int run_vlinks(aslhip_lattice *h, bool after_odd) {
  if (!h->nvl) return 0;
  VLinkArgs a;
  a.f = h->f;
  a.qs_bytes = h->qs_bytes;
  a.sx = h->sx;
  a.sy = h->sy;
  a.links = h->vl;
  a.nlinks = h->nvl;
  a.bc = h->vlbc;
  a.dx = h->dx;
  for (int d = 0; d < 3; ++d) a.pos0[d] = h->pos0[d];
  a.after_odd = after_odd ? 1 : 0;
  HIPCHK(launch_vlinks(h->Q, h->dtype, a, h->stream));
  return 0;
}

bool is_wide(const aslhip_lattice *h) { return h->force_wide || h->qs_bytes * h->Q > 0xffffffffLL; }

// Cells per lane the step kernel runs with: runs of 2 or 4 cells along z on
// non-periodic lattices under 4 GiB without a per-cell relaxation, when nz is
// a multiple of the run; else one cell per lane (the longest run that divides
// nz).  Automatic: one cell per lane.
// LDS-staged tiles apply to non-periodic lattices under 4 GiB without a
// per-cell relaxation unless runs of 2 or 4 cells per lane are asked for:
// 0 none, 1 every step, 2 even steps only (odd steps one cell per lane).
// Automatic: every step that is not part of a sweep (sweep_shape) for D3Q19
// FP32 lattices whose populations outgrow the 256 MiB Infinity Cache (box of 256 x 128 x 128, 331 MB: 116 us per step, 128
// direct); none for lattices the cache holds (64^3 box, 22 MB: 12.7 against
// 9.7 us), for the other templates (D3Q27 300 x 130 x 140: 226 against 224 us,
// and sweeps gain beside other lattices; D3Q15: 282 against 123 us) and for
// FP16 / BF16 / FP64 storage (the direct kernel is faster there).
constexpr long long CACHE_BYTES = 256LL << 20;  // the Infinity Cache
int effective_lds(const aslhip_lattice *h) {
  const bool big = h->qs_bytes * h->Q > CACHE_BYTES;
  const int mode = h->tune_lds < 0 ? (h->Q == 19 && h->dtype == ASLHIP_F32 && big ? 1 : 0) : h->tune_lds;
  return h->tune_cpl <= 1 && !(h->periodic || is_wide(h) || h->has_closure || h->turbulence) ? mode : 0;
}

int effective_cpl(const aslhip_lattice *h) {
  if (h->periodic || is_wide(h) || h->has_closure || h->turbulence || effective_lds(h)) return 1;
  int c = h->tune_cpl;
  if (c == 0) c = 1;
  while (c > 1 && h->n[2] % c) c /= 2;
  return c;
}

// Workgroup size of single steps whose direct kernel takes that many lanes (runs
// of cells: at most STEP_RUN_BLOCK; LDS-staged tiles on every step: STEP_TILE;
// tiles on even steps only: the odd steps' workgroup).
int step_workgroup(const aslhip_lattice *h, int lanes) {
  if (effective_lds(h) == 1) return STEP_TILE;
  const int most = step_block(h->Q, static_cast<int>(h->selem));
  return std::min(lanes, effective_cpl(h) > 1 ? std::min(most, STEP_RUN_BLOCK) : most);
}

// Lanes per workgroup of the direct kernel: tune_block, unless nobody chose it
// and the lattice is small.  A step of one workgroup per CU or less takes as
// long as one workgroup, and smaller ones start and end sooner: 16^3 D3Q19
// FP32 box in a graph 4.45 us (512 lanes), 3.84 (256), 3.69 (128); 16^3 D3Q27 FP64
// 7.14, 5.83, 5.37; 32^3 4.74, 4.15, 4.01; 40^3 5.19, 4.54, 5.08; 48^3 5.66, 5.60, 5.61.
// So the smallest of 128, 256 lanes that gives every CU at most one workgroup.
// (Above, 256 gain where they fill the last round of workgroups better, 56^3 8.0 ->
// 7.1, and are level elsewhere, 64^3 8.46 -> 8.34: not automatic.)  D3Q27 in FP64, of
// which a CU holds 12 wavefronts, takes 256 lanes, so that all 12 find room: 64^3
// periodic 18.5 (512) -> 17.8, 97^3 63.4 -> 61.4, beside two more 75.5 -> 73.9; in sweeps
// 200^3 631 -> 611, 300^3 2195 -> 2076.  Launches over a whole lattice that streams from
// HBM keep 512: 200^3 (1.8 GB) 671 (512), 675 (256), 120 x 400 x 300 1269, 1311, 300^3 2418,
// 2563.  The matrix-core closure kernel shares one copy of the weights per workgroup
// and keeps the large ones.
constexpr long long TALL_BYTES = 1536LL << 20;
int step_lanes(const aslhip_lattice *h, bool sweep) {
  const bool tall = step_block(h->Q, static_cast<int>(h->selem)) < STEP_BLOCK && (sweep || h->qs_bytes * h->Q <= TALL_BYTES);
  if (!h->block_set && !h->has_closure)
    for (int lanes : {128, 256})
      if ((tall && lanes == 256) || 1LL * h->n[0] * h->n[1] * h->n[2] <= 256LL * lanes)
        return std::min(lanes, h->tune_block);
  return h->tune_block;
}

// Consecutive chunks per XCD run of a launch of n chunks; at most an XCD's share.
// Unless somebody chose it, each XCD takes one slab of a lattice that the
// Infinity Cache holds, so that chunks whose cells exchange populations along x
// and y meet in one L2, within a step and from one step to the next.  us per
// step alone, runs of 4 -> slabs: D3Q19 FP32 48^3 6.5 -> 5.5, 64^3 9.5 -> 8.4,
// 96^3 24.9 -> 22.3, 112^3 38.7 -> 35.5, 128^3 52.0 -> 51.4; D3Q15 300 x 50 x 50
// 19.5 -> 16.2; D3Q19 FP64 64^3 14.8 -> 13.7; 97 x 61 x 83 14.9 -> 12.6; FP16 64^3
// 8.5 -> 7.5.  Four slabs per XCD over 150 MiB, which are level alone and better
// beside others; alone / beside two more, runs of 4, one slab, four: D3Q19 FP32
// 132^3 (175 MB) 59.5 / 69.0, 57.4 / 72.3, 57.9 / 68.6, 144^3 73.0 / 88.0, 70.5 /
// 89.4, 70.7 / 88.0; with 16-bit storage runs of 64 there, FP16 256 x 128 x 128 60.9
// / 69.3, one slab 59.6 / 75.7, four 62.1 / 72.4.  Larger lattices and tiles keep short runs: D3Q27 224^3 in sweeps 435
// (runs of 4), 447 (four slabs), 517 (one); tiles on 256 x 128 x 128 114, 121, 122.
constexpr long long SLAB_BYTES = 150LL << 20;
int xcd_run(const aslhip_lattice *h, int n, bool tile) {
  const int share = std::max(1, n / 8);
  const long long bytes = h->qs_bytes * h->Q;
  if (h->remap_set || tile || bytes > CACHE_BYTES) return std::min(std::max(1, h->tune_remap), share);
  if (bytes <= SLAB_BYTES) return share;
  return h->selem == 2 ? std::min(h->tune_remap, share) : std::max(1, share / 4);
}

// The divisor d of udivm (kernels.hip); 0 stands for d = 1.
unsigned long long udiv_magic(unsigned d) { return d <= 1 ? 0ULL : ~0ULL / d + 1ULL; }

// The face rule's entries (StepHot): the faces that have a slice BC, by the
// execution slot of the last one on them.
void face_entries(const aslhip_lattice *h, StepArgs &a) {
  std::vector<int> fc;
  for (int f = 0; f < 6; ++f)
    if (h->fface[f]) fc.push_back(f);
  std::stable_sort(fc.begin(), fc.end(), [h](int p, int q) { return h->fface[p] < h->fface[q]; });
  for (size_t j = 0; j < fc.size(); ++j) {
    const int f = fc[j], axis = f / 2, in = f % 2 == 0 ? 1 : -1;
    const bool bounce = (h->fface[f] & 3) == MODE_BOUNCE;
    bool valued = !bounce;
    for (int k = 0; k < h->Q; ++k) {
      a.fval32[f][k] = h->fval32[f][k];
      a.fval64[f][k] = h->fval64[f][k];
      valued = valued || (h->celem == 8 ? h->fval64[f][k] != 0. : h->fval32[f][k] != 0.f);
      if (h->t.c[k][axis] == in) a.g.flinks[j] |= 1u << k;
    }
    a.g.fpos |= static_cast<unsigned>(f) << (4 * j);
    if (bounce) a.g.fbounce |= 1u << j;
    a.fset |= 1u << f;
    if (bounce) a.g.fbfaces |= 1u << f;
    if (valued) a.g.fvalued |= 1u << f;
    for (int p : fc) {  // of faces with one BC the last one owns their common links: each link has one owner
      const int sp = h->fface[p] / 4, sf = h->fface[f] / 4;
      if (sp > sf || (sp == sf && p > f)) a.fbeats[f] |= 1u << p;
    }
  }
}

// That many lanes per workgroup, at most what the direct kernel takes.
int direct_block(const aslhip_lattice *h, int lanes) {
  return std::min(lanes, step_block(h->Q, static_cast<int>(h->selem)));
}

// Kernel arguments of one step of h over the whole lattice (STEP_F_* of the
// lattice's parameters).  With block and cpl 0 the lattice's own tuning for a
// step of that parity (LDS-staged tiles included), else one cell per lane in
// workgroups of that size, or tiles if asked for.
StepArgs step_args(const aslhip_lattice *h, int block = 0, int cpl = 0, bool odd = false, bool tiles = false) {
  StepArgs a;
  std::memset(static_cast<void *>(&a), 0, sizeof a);  // compared bytewise by upload_args
  StepHot &g = a.g;
  g.f = h->f;
  g.code = h->code;
  g.qs = static_cast<unsigned long long>(h->qs_bytes);
  a.qs32 = is_wide(h) ? 0u : static_cast<unsigned>(h->qs_bytes);
  face_entries(h, a);
  g.sx = h->sx;
  g.sy = h->sy;
  g.nx = h->n[0];
  g.ny = h->n[1];
  g.nz = h->n[2];
  a.len = h->len;
  a.cpl = cpl > 0 ? cpl : effective_cpl(h);
  g.block = block > 0 ? block : step_lanes(h, false);
  if (a.cpl > 1 && g.block > STEP_RUN_BLOCK) g.block = STEP_RUN_BLOCK;
  g.block = direct_block(h, g.block);
  const int lds = effective_lds(h);
  a.tile = tiles || (block <= 0 && cpl <= 0 && (lds == 1 || (lds == 2 && !odd))) ? 1 : 0;
  if (a.tile) g.block = STEP_TILE;

  g.rowi = h->n[2] / a.cpl;
  g.mrow = udiv_magic(static_cast<unsigned>(g.rowi));
  g.mplane = udiv_magic(static_cast<unsigned>(g.ny));
  g.inv_row = 1.f / static_cast<float>(g.rowi);
  g.inv_ny = 1.f / static_cast<float>(g.ny);
  g.first = 0;
  g.count = static_cast<unsigned>(g.nx) * static_cast<unsigned>(g.ny) * static_cast<unsigned>(g.rowi);
  a.bpp = (g.ny * g.sy + STEP_TILE - 1) / STEP_TILE;
  g.nchunks = a.tile ? a.bpp * g.nx : static_cast<int>((static_cast<long long>(g.count) + g.block - 1) / g.block);
  a.zmagic = ((1ULL << 40) + (unsigned long long)h->sy - 1) / (unsigned long long)h->sy;
  g.remap = xcd_run(h, g.nchunks, a.tile != 0);
  g.mspan = udiv_magic(8u * static_cast<unsigned>(g.remap));
  a.pat = h->pat;
  a.rec = h->rec;
  a.mode = h->mode;
  a.val = h->val;
  a.rho = h->rho;
  a.u = h->u;
  a.w = relaxation(h);
  for (int d = 0; d < 3; ++d) {
    a.om32[d] = static_cast<float>(h->omega[d]);
    a.om64[d] = h->omega[d];
  }
  a.cl = h->d_cl;
  a.cl_tau0 = 3.f * static_cast<float>(h->nu) + .5f;
  a.nu32 = static_cast<float>(h->nu);
  a.nu64 = h->nu;
  g.flags = base_flags(h);
  return a;
}

// Runs nsteps steps now.  raw_first: the first one reads ghost links raw
// (no BC executed before it since init); macro_last: the last one writes rho/u.
// The execute order of the BCs since the last step becomes the active one;
// the tables are rebuilt if anything changed.
int prepare(aslhip_lattice *h, bool allow_open) {
  if (!h->pending.empty()) {
    if (h->pending != h->order) {
      h->order = h->pending;
      h->dirty = true;
    }
    h->pending.clear();
  }
  return h->dirty ? finalize_impl(h, allow_open) : 0;
}

// Brings the device copies of the step arguments up to date; they change with
// the BC tables, viscosity, compressibility and tuning.  Captured runs carry
// the by-value part (StepHot) and are dropped when it changes.
int upload_args(aslhip_lattice *h) {
  const StepArgs base[2] = {step_args(h, 0, 0, false), step_args(h, 0, 0, true)};
  if (!h->h_args.empty()) {
    if (std::memcmp(base, h->h_args.data(), sizeof base) == 0) {
      // tiles and runs of cells do not show every change of the workgroup size that the sweeps take
      if (h->h_direct.block != direct_block(h, step_lanes(h, true))) h->h_direct = step_args(h, step_lanes(h, true), 1).g;
      return 0;
    }
    for (int p = 0; p < 2; ++p)
      if (std::memcmp(&base[p].g, &h->h_args[p].g, sizeof(StepHot)) != 0) drop_graphs(h);
    // the previous upload reads h_args: let it finish before overwriting
    HIPCHK(hipStreamSynchronize(h->stream));
  }
  h->h_args.assign(base, base + 2);
  h->h_direct = step_args(h, step_lanes(h, true), 1).g;
  // stream-ordered: steps queued before still see the previous arguments
  HIPCHK(hipMemcpyAsync(h->d_args, h->h_args.data(), sizeof base, hipMemcpyHostToDevice, h->stream));
  return 0;
}

// One launch of the step kernel: step args for parity odd, flags fl, the
// interior planes p0 .. p0 + np - 1 one cell per lane (np < 0: the whole
// lattice with its tuning).
int launch_planes(aslhip_lattice *h, bool odd, unsigned fl, int p0, int np) {
  StepLaunch a;
  const int p = odd ? 1 : 0;
  const StepArgs &A = h->h_args[p];
  a.hot = np < 0 ? A.g : h->h_direct;
  a.hot.flags = fl;
  a.args = h->d_args + p;
  // LBGKTurbulence takes precedence over a closure in the collision
  a.variant = h->turbulence ? 1 : (h->has_closure ? (h->closure_mfma ? 2 : 3) : 0);
  a.cpl = np < 0 ? A.cpl : 1;
  a.tile = np < 0 ? A.tile : 0;
  if (np >= 0) {
    const unsigned plane = static_cast<unsigned>(a.hot.ny) * static_cast<unsigned>(a.hot.nz);
    a.hot.first = static_cast<unsigned>(p0) * plane;
    a.hot.count = static_cast<unsigned>(np) * plane;
    a.hot.nchunks = static_cast<int>((static_cast<long long>(a.hot.count) + a.hot.block - 1) / a.hot.block);
    a.hot.remap = xcd_run(h, a.hot.nchunks, false);
    a.hot.mspan = udiv_magic(8u * static_cast<unsigned>(a.hot.remap));
  }
  ++h->queued;
  HIPCHK(launch_step(h->Q, h->dtype, odd, h->periodic, is_wide(h), a, h->stream));
  return 0;
}

// The shape of the sweeps (sweep_plan) of a run of n steps: g planes per launch,
// t steps per sweep; t = 0: one launch per step over the whole lattice.
// Automatic: for lattices that the 256 MiB Infinity Cache cannot hold, a window
// of 224 MiB (g + t planes) that takes up to 16 steps, so that most reads and
// writes of a step find their lines there.  us per step, alone / with two more
// lattices stepped beside it, before and after: D3Q27 FP32 224^3 periodic 463 /
// 518 -> 438 / 466, D3Q27 FP64 160^3 periodic 326 / 386 -> 317 / 309, D3Q19
// FP64 256 x 128 x 128 226 / 281 -> 215 / 222, D3Q15 BF16 300 x 200 x 200 161 /
// 161 -> 151 / 161.  192 MiB is 1 to 3 % slower, 64 MiB gains only beside other
// lattices.
// Runs of less than 4 steps read too much twice: 2 steps of the last two, 161
// -> 161 and 226 -> 244 us per step, 4 steps 159 -> 157 and 226 -> 224.
// D3Q19 FP32 lattices that run tiles sweep from 560 MiB and 6 steps on; tiles
// -> sweeps of 20 steps: 256 x 128 x 128 (346 MB) 113 / 119 -> 109 / 124, 300 x
// 128 x 128 137 / 141 -> 131 / 145, 192^3 194 / 203 -> 192 / 208; 320 x 160 x
// 160 (642 MB) 231 / 256 -> 223 / 256, 256 x 256 x 128 226 / 271 -> 219 / 242,
// 256^3 462 / 583 -> 447 / 482, 512 x 256 x 256 942 / 1211 -> 896 / 985; of 4
// steps 256 x 256 x 128 225 -> 227, of 6 steps 223 -> 223.
// FP64 lattices below 768 MiB, which lose 2 to 4 % alone and gain 4 to 19 % beside
// others, sweep from 8 steps on (156 x 153 x 150 D3Q19, 539 MB, alone, 4 steps: 190
// -> 197).
// Velocity-map links are filled after every step of the whole lattice: no
// sweeps.
constexpr long long SWEEP_WINDOW = 224LL << 20;
constexpr long long SWEEP_TILED_BYTES = 560LL << 20, SWEEP_F64_BYTES = 768LL << 20;
constexpr int SWEEP_STEPS = 16, SWEEP_MIN_STEPS = 4, SWEEP_TILED_MIN_STEPS = 6, SWEEP_F64_MIN_STEPS = 8;

// Whether a window of wp planes pays.  Every launch of a window costs some 5 us
// of its own and a sweep takes wp / 2 steps, so thick planes lose, more so in
// boxes (the direct kernel's own reuse, odd steps from the other end, is worth
// 256 MiB a step); the larger the lattice, the less.  us per step of 20 alone,
// launch per step -> sweeps: 16 planes and more at least level but for FP64
// (above).  Periodic: 12 planes, D3Q19 FP64 400 x 300: 20 planes 121 -> 132, 60 403 ->
// 396, 80 559 -> 531; 11, D3Q19 FP32 512 x 512: 24 165 -> 179, 80 604 -> 587; 8, D3Q27
// FP32 512 x 512: 40 439 -> 474, 200 2276 -> 2243; 10, FP16 750 x 750: 80 708 -> 720;
// 4, D3Q27 FP32 700 x 700: 300 6490 -> 6990, FP64 500 x 500: 20 408 -> 429, 60 1345 ->
// 1282, 200 4925 -> 4309; 5, D3Q19 FP64 512 x 512: 300 4937 -> 4528.  Boxes: 12 planes,
// D3Q19 FP64 400 x 300: 60 402 -> 408, 90 638 -> 648, 150 1059 -> 1024, 300 2150 -> 2055;
// 11, D3Q19 FP32 512 x 512: 40 292 -> 309, 150 1235 -> 1149, 300 2376 -> 2306; 8, D3Q27
// FP32 512 x 512: 200 2257 -> 2366, FP64 400 x 300: 40 392 -> 408, 120 1267 -> 1227; 10,
// FP16 750 x 750: 80 711 -> 753, 300 2730 -> 2876; 4, D3Q27 FP64 500 x 500: 60 1287 ->
// 1384, 200 4665 -> 4601; 5, D3Q19 FP64 512 x 512: 300 4685 -> 4837.
bool sweep_pays(const aslhip_lattice *h, long long wp, long long bytes) {
  constexpr long long MIB = 1LL << 20;
  const bool f64 = h->selem == 8;
  if (wp >= 16) return true;
  if (h->selem < 4) return false;
  if (wp >= 8)
    return h->periodic ? bytes >= 1536 * MIB : (wp >= 9 && bytes >= 2048 * MIB) || (f64 && bytes >= 2816 * MIB);
  return f64 && (h->periodic || h->Q == 27) && bytes >= (h->periodic && h->Q == 27 ? 3072 : 8192) * MIB;
}

void sweep_shape(const aslhip_lattice *h, int n, int &g, int &t) {
  g = t = 0;
  if (n < 2 || h->nvl || h->tune_sweep == 0) return;
  const long long plane = static_cast<long long>(h->Q) * h->selem * h->sx;
  if (h->tune_sweep < 0) {
    const long long bytes = h->qs_bytes * h->Q;
    if (bytes <= CACHE_BYTES || n < SWEEP_MIN_STEPS || !sweep_pays(h, SWEEP_WINDOW / plane, bytes)) return;
    if (h->selem == 8 && bytes < SWEEP_F64_BYTES && n < SWEEP_F64_MIN_STEPS) return;
    if (effective_lds(h) == 1 && (h->tune_lds == 1 || bytes <= SWEEP_TILED_BYTES || n < SWEEP_TILED_MIN_STEPS)) return;
  }
  const long long window = h->tune_sweep > 0 ? static_cast<long long>(h->tune_sweep) << 10 : SWEEP_WINDOW;
  const int wp = static_cast<int>(std::min<long long>(window / plane, h->n[0]));
  const int m = std::min(SWEEP_STEPS, wp / 2);
  if (m < 2 || wp >= h->n[0]) return;
  t = m;
  g = wp - m;
}

// Launches of a run of n steps, see sweep_plan.
struct SweepLaunch {
  int step;    // step of the run
  int p0, np;  // interior planes (x - 1) of this launch
};

// Orders n steps of a lattice of nx planes so that a window of planes takes
// several steps while it stays in the Infinity Cache.  A step of plane x
// needs planes x - 1, x, x + 1 one step earlier and nothing else (each slot of
// the AA pattern belongs to one cell in every step, and to a cell at most one
// plane away in the next), so blocks of g planes, shifted one plane back per
// step, can take t steps one block after the other: block b does planes
// [b g - s, (b + 1) g - s) in step s.  Periodic lattices: step s covers planes
// s .. nx + s - 1 (modulo nx), so that the first block starts from planes
// nobody needs yet and the last one closes the ring.
// Hands the launches to emit in order until it returns false.
template <class F>
void sweep_plan(long long nx, bool periodic, long long g, long long t, long long n, F emit) {
  for (long long s0 = 0; s0 < n; s0 += t) {
    const long long m = std::min(t, n - s0);
    const long long end = periodic ? nx + m - 1 : nx;  // planes of the last step end here
    for (long long b = 0; b * g - (m - 1) < end; ++b) {
      // the steps that have planes in this block
      const long long over = std::max(0LL, b * g - nx + 1), below = (b + 1) * g;
      const long long first = periodic ? (over + 1) / 2 : over, last = std::min(m, periodic ? (below + 1) / 2 : below);
      for (long long s = first; s < last; ++s) {
        const long long lo = std::max(b * g - s, periodic ? s : 0), hi = std::min((b + 1) * g - s, periodic ? nx + s : nx);
        if (lo < nx && !emit(SweepLaunch{static_cast<int>(s0 + s), static_cast<int>(lo), static_cast<int>(std::min(hi, nx) - lo)}))
          return;
        if (hi > nx && !emit(SweepLaunch{static_cast<int>(s0 + s), static_cast<int>(std::max(lo, nx) - nx),
                                         static_cast<int>(hi - std::max(lo, nx))}))
          return;
      }
    }
  }
}

int launch_one(aslhip_lattice *h, unsigned fl, std::vector<hipEvent_t> *ev, int s) {
  if (ev) HIPCHK(hipEventRecord((*ev)[2 * s], h->stream));
  if (int r = launch_planes(h, h->next_odd, fl, 0, -1)) return r;
  if (ev) HIPCHK(hipEventRecord((*ev)[2 * s + 1], h->stream));
  const bool was_odd = h->next_odd;
  h->next_odd = !h->next_odd;
  return run_vlinks(h, was_odd);
}

// n steps with the flags fl, the last one with last_fl.
int launch_run(aslhip_lattice *h, unsigned fl, unsigned last_fl, int n) {
  int g = 0, t = 0;
  sweep_shape(h, n, g, t);
  if (!t) {
    for (int s = 0; s < n; ++s)
      if (int r = launch_one(h, s == n - 1 ? last_fl : fl, nullptr, s)) return r;
    return 0;
  }
  for (int s = 0; s < n; s += t) {
    const int m = std::min(t, n - s);
    int r = 0;
    sweep_plan(h->n[0], h->periodic, g, t, m, [&](const SweepLaunch &l) {
      r = launch_planes(h, h->next_odd != ((l.step & 1) != 0), s + l.step == n - 1 ? last_fl : fl, l.p0, l.np);
      return r == 0;
    });
    if (r) return r;
    if (m & 1) h->next_odd = !h->next_odd;
  }
  return 0;
}

// At most this many captured remainders (runs shorter than a chunk) are kept.
constexpr size_t MAX_TAIL_GRAPHS = 6;

// The captured run of n plain steps starting at parity odd with the current
// step flags, captured now if there is none.
int get_graph(aslhip_lattice *h, int n, bool odd, hipGraphExec_t *out) {
  const unsigned fl = base_flags(h);
  for (const auto &g : h->graphs)
    if (g.n == n && g.odd == odd && g.fl == fl) {
      *out = g.exec;
      return 0;
    }
  // A run captured with other flags (frame, compressibility, relaxation
  // model) names the old kernel variant and flags, and the oldest
  // remainder makes room for a new one: destroyed once replays of them have
  // finished.
  auto drop = [h](size_t i) -> int {
    HIPCHK(hipStreamSynchronize(h->stream));
    (void)hipGraphExecDestroy(h->graphs[i].exec);
    h->graphs.erase(h->graphs.begin() + static_cast<long>(i));
    return 0;
  };
  for (size_t i = 0; i < h->graphs.size(); ++i)
    if (h->graphs[i].n == n && h->graphs[i].odd == odd) {
      if (int r = drop(i)) return r;
      break;
    }
  if (n != ASLHIP_GRAPH_CHUNK) {
    size_t tails = 0, oldest = 0;
    for (size_t i = h->graphs.size(); i-- > 0;)
      if (h->graphs[i].n != ASLHIP_GRAPH_CHUNK) {
        ++tails;
        oldest = i;
      }
    if (tails >= MAX_TAIL_GRAPHS)
      if (int r = drop(oldest)) return r;
  }
  const bool keep = h->next_odd;
  h->next_odd = odd;
  hipGraph_t graph = nullptr;
  HIPCHK(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
  int r = 0;
  r = launch_run(h, fl, fl, n);
  hipError_t e = hipStreamEndCapture(h->stream, &graph);
  h->next_odd = keep;
  if (r) {
    if (graph) (void)hipGraphDestroy(graph);
    return r;
  }
  if (e != hipSuccess) return fail(ASLHIP_EHIP, "ASL ERROR: graph capture: %s", hipGetErrorString(e));
  hipGraphExec_t g = nullptr;
  e = hipGraphInstantiate(&g, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) return fail(ASLHIP_EHIP, "ASL ERROR: graph instantiate: %s", hipGetErrorString(e));
  h->graphs.push_back({n, odd, fl, g});
  *out = g;
  return 0;
}

// graph: run whole chunks of plain steps (not the raw first one, not the
// one writing rho/u) as hipGraph replays, unless the lattice sweeps: its
// launches are long enough to hide the next one's submission, and a graph of
// several launches per step would have to be captured first.  consume: the BC executions
// recorded since the last step become the active order first (a deferred
// step runs with the order folded in when it was requested instead: the
// executions recorded since then belong to the step after it).
int run_steps(aslhip_lattice *h, int nsteps, bool first_after_init, bool raw_first, bool macro_last,
              std::vector<hipEvent_t> *ev, bool graph = false, bool consume = true) {
  if (nsteps <= 0) return 0;
  if (int r = order_after_consumer(h)) return r;
  const bool allow_open = raw_first && nsteps == 1;
  if (int r = consume ? prepare(h, allow_open) : (h->dirty ? finalize_impl(h, allow_open) : 0)) return r;
  if (first_after_init && !raw_first) {
    // the BCs were applied to the initial state: velocity-map links too
    int r = run_vlinks(h, false);
    if (r) return r;
  }
  if (int r = upload_args(h)) return r;
  for (int s = 0; s < nsteps;) {
    const bool raw = s == 0 && raw_first;
    const int plain = nsteps - s - (macro_last ? 1 : 0);  // plain steps left
    int sg = 0, st = 0;
    if (!raw && !ev) sweep_shape(h, nsteps - s, sg, st);
    if (graph && !ev && !raw && plain >= 1 && !st) {
      const int n = plain < ASLHIP_GRAPH_CHUNK ? plain : ASLHIP_GRAPH_CHUNK;
      hipGraphExec_t g = nullptr;
      if (int r = get_graph(h, n, h->next_odd, &g)) return r;
      HIPCHK(hipGraphLaunch(g, h->stream));
      s += n;
      if (n & 1) h->next_odd = !h->next_odd;
      continue;
    }
    unsigned fl = base_flags(h), last = fl;
    if (macro_last) {
      if (h->comp_rho) last |= STEP_F_RHO;
      if (h->comp_vel) last |= STEP_F_VEL;
    }
    if (raw || ev || (graph && !st)) {  // one step
      if (s == nsteps - 1) fl = last;
      if (raw) fl |= STEP_F_RAW;
      if (int r = launch_one(h, fl, ev, s)) return r;
      ++s;
    } else {
      if (int r = launch_run(h, fl, last, nsteps - s)) return r;
      s = nsteps;
    }
  }
  return 0;
}

// Runs a deferred step, writing rho and u (the host is about to look).  It
// uses the BC order folded in when it was requested.
int flush_deferred(aslhip_lattice *h) {
  if (!h->deferred) return 0;
  h->deferred = false;
  return run_steps(h, 1, h->deferred_first, h->deferred_raw, true, nullptr, false, false);
}

int step_impl(aslhip_lattice *h, int nsteps, unsigned flags, std::vector<hipEvent_t> *ev) {
  if (nsteps < 0) return fail(ASLHIP_EINVAL, "ASL ERROR: negative step count");
  if (!h->initialized) return fail(ASLHIP_ESTATE, "ASL ERROR: LBGK::execute before initF");
  if (h->deferred) {  // a newer step follows: no need for its rho/u
    h->deferred = false;
    int r = run_steps(h, 1, h->deferred_first, h->deferred_raw, false, nullptr, false, false);
    if (r) return r;
  }
  // the first step after initF reads raw ghost values unless a BC ran before it
  const bool first = h->fresh && nsteps > 0;
  const bool raw = first && !h->bc_since_init;
  if (nsteps > 0) h->fresh = false;
  const bool graph = (flags & ASLHIP_STEP_GRAPH) != 0;
  if ((flags & ASLHIP_STEP_DEFER) && nsteps > 0) {
    int r = run_steps(h, nsteps - 1, first, raw, false, ev, graph);
    if (r) return r;
    h->deferred_first = first && nsteps == 1;
    h->deferred_raw = raw && nsteps == 1;
    // the deferred step takes the BC executions recorded up to now; later
    // ones stay pending for the step after it
    if (int r2 = prepare(h, h->deferred_raw)) return r2;
    h->deferred = true;
    return 0;
  }
  return run_steps(h, nsteps, first, raw, (flags & ASLHIP_STEP_WRITE_MACRO) != 0, ev, graph);
}

int copy_out(aslhip_lattice *h, const void *dev, void *host, size_t bytes) {
  HIPCHK(to_host(host, dev, bytes, h->stream, &h->queued));
  return 0;
}

}  // namespace

int aslhip::read_f_through(aslhip_lattice *h, void *out, void *buf, size_t buf_bytes, bool staged) {
  if (int r = flush_deferred(h)) return r;
  const size_t cell_bytes = (size_t)h->Q * h->melem;  // one cell's Q values
  const size_t per = std::min(buf_bytes / cell_bytes, (size_t)h->len);
  if (per < 1) return fail(ASLHIP_EINVAL, "ASL ERROR: read_f: staging buffer smaller than one cell");
  UnpermuteArgs a;
  a.f = h->f;
  a.qs_bytes = h->qs_bytes;
  a.sx = h->sx;
  a.sy = h->sy;
  a.len = h->len;
  a.per = h->periodic ? 1 : 0;
  a.nx = h->n[0];
  a.ny = h->n[1];
  a.nz = h->n[2];
  a.after_odd = h->next_odd ? 0 : 1;
  a.out = buf;
  char *o = static_cast<char *>(out);
  for (size_t first = 0; first < (size_t)h->len; first += per) {
    const size_t count = std::min(per, (size_t)h->len - first);
    a.first = static_cast<int>(first);
    a.count = static_cast<int>(count);
    HIPCHK(launch_unpermute(h->Q, h->dtype, a, h->stream));
    if (staged && count == (size_t)h->len) return copy_out(h, buf, out, cell_bytes * count);  // one contiguous view
    HIPCHK(hipStreamSynchronize(h->stream));
    // piece i of the view: cells first .. first + count - 1 of direction i
    HIPCHK(hipMemcpy2D(o + first * h->melem, (size_t)h->len * h->melem, buf, count * h->melem, count * h->melem,
                       (size_t)h->Q, hipMemcpyDeviceToHost));
  }
  return 0;
}

extern "C" {

int aslhip_last_error(char *buf, size_t n) {
  if (buf && n) {
    std::strncpy(buf, g_err.c_str(), n - 1);
    buf[n - 1] = 0;
  }
  return static_cast<int>(g_err.size());
}

int aslhip_device_info(char *buf, size_t n, int *cu_count, double *hbm_bytes) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  hipDeviceProp_t p;
  HIPCHK(hipGetDeviceProperties(&p, dev));
  if (buf && n) {
    // some runtimes leave the marketing name empty: then the CU count names the part
    char name[256] = {0};
    if (p.name[0]) std::snprintf(name, sizeof name, "%s", p.name);
    else if (hipDeviceGetName(name, sizeof name, dev) != hipSuccess || !name[0])
      std::snprintf(name, sizeof name, "AMD GPU with %d CUs", p.multiProcessorCount);
    std::snprintf(buf, n, "%s (%s)", name, p.gcnArchName);
  }
  if (cu_count) *cu_count = p.multiProcessorCount;
  if (hbm_bytes) *hbm_bytes = static_cast<double>(p.totalGlobalMem);
  return 0;
}

int aslhip_lattice_create(aslhip_lattice **out, int nx, int ny, int nz, int q, int dtype, unsigned flags) {
  if (!out) return fail(ASLHIP_EINVAL, "ASL ERROR: null output handle");
  *out = nullptr;
  if (nx < 1 || ny < 1 || nz < 1) return fail(ASLHIP_EINVAL, "ASL ERROR: block size must be positive");
  if (q != 15 && q != 19 && q != 27) return fail(ASLHIP_EINVAL, "ASL ERROR: lattice template must be D3Q15, D3Q19 or D3Q27");
  if (dtype < ASLHIP_F32 || dtype > ASLHIP_F16) return fail(ASLHIP_EINVAL, "ASL ERROR: unknown population type %d", dtype);
  const unsigned per = flags & 7u;
  if (per != 0 && per != 7) return fail(ASLHIP_EINVAL, "ASL ERROR: periodic wrap must be on all three axes");
  const long long S0 = nx + 2LL, S1 = ny + 2LL, S2 = nz + 2LL;
  const long long len = S0 * S1 * S2;
  if (len > 0x7fffffffLL - 4096) return fail(ASLHIP_EINVAL, "ASL ERROR: block too large for one lattice");
  aslhip_lattice *h = new aslhip_lattice();
  transfer_hold();
  h->n[0] = nx;
  h->n[1] = ny;
  h->n[2] = nz;
  h->S[0] = (int)S0;
  h->S[1] = (int)S1;
  h->S[2] = (int)S2;
  h->sy = (int)S2;
  h->sx = (int)(S1 * S2);
  h->len = (int)len;
  h->Q = q;
  h->dtype = dtype;
  h->periodic = per == 7;
  h->t = make_templ(q);
  h->selem = dtype == ASLHIP_F64 ? 8 : (dtype == ASLHIP_F32 ? 4 : 2);
  // 16-bit storage: the run length reported until somebody chooses one
  if (h->selem == 2) h->tune_remap = 64;
  h->melem = h->celem = dtype == ASLHIP_F64 ? 8 : 4;
  // direction arrays 256-byte aligned
  const long long qs_elems = (len + 127) / 128 * 128;
  // The step kernel finds a cell's row as (off * ceil(2^40/Sz)) >> 40, exact
  // while (cells per plane) * Sz < 2^40.
  if ((double)S1 * S2 * S2 >= 1099511627776.0)
    return fail(ASLHIP_EINVAL, "ASL ERROR: block planes too large");
  if (qs_elems * (dtype == ASLHIP_F64 ? 8 : 4) > 0xffffffffLL)
    return fail(ASLHIP_EINVAL, "ASL ERROR: block too large: one direction array must stay below 4 GiB");
  h->qs_bytes = qs_elems * (long long)h->selem;
  hipError_t e = hipGetDevice(&h->device);
  if (e == hipSuccess) e = hipStreamCreate(&h->stream);
  if (e == hipSuccess) e = device_alloc(&h->f, (size_t)h->qs_bytes * q);
  if (e == hipSuccess) e = device_alloc(&h->rho, (size_t)len * h->melem);
  if (e == hipSuccess) e = device_alloc(&h->u, (size_t)len * 3 * h->melem);
  if (e == hipSuccess) e = device_alloc(&h->code, (size_t)len);
  if (e == hipSuccess) e = device_alloc(&h->pat, (size_t)len * 2);
  if (e == hipSuccess) e = device_alloc(&h->mode, 256);
  if (e == hipSuccess) e = device_alloc(&h->val, 256 * (size_t)q * h->celem);
  if (e == hipSuccess) e = device_alloc(&h->vlbc, 256 * sizeof(VLinkBC));
  if (e == hipSuccess) e = device_alloc(&h->d_args, 2 * sizeof(StepArgs));
  if (e == hipSuccess) e = device_alloc(&h->red_partial, (size_t)reduce_blocks((int)len) * 5 * sizeof(double));
  if (e == hipSuccess) e = device_alloc(&h->red_out, 5 * sizeof(double));
  if (e != hipSuccess) {
    free_all(h);
    delete h;
    return fail(e == hipErrorOutOfMemory ? ASLHIP_ENOMEM : ASLHIP_EHIP, "ASL ERROR: lattice allocation: %s",
                hipGetErrorString(e));
  }
  *out = h;
  return 0;
}

int aslhip_lattice_destroy(aslhip_lattice *h) {
  if (!h) return 0;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  free_all(h);
  delete h;
  return 0;
}

int aslhip_set_viscosity(aslhip_lattice *h, double nu) {
  if (int r = check(h)) return r;
  if (!(nu >= 0.) && !std::isinf(nu)) return fail(ASLHIP_EINVAL, "ASL ERROR: viscosity must be >= 0");
  if (int r = flush_deferred(h)) return r;  // a pending step runs with the old value
  h->nu = nu;
  return 0;
}

int aslhip_set_compressible(aslhip_lattice *h, int c) {
  if (int r = check(h)) return r;
  if (int r = flush_deferred(h)) return r;
  h->compressible = c != 0;
  h->dirty = true;  // pressure-velocity map values depend on it
  return 0;
}

int aslhip_set_omega(aslhip_lattice *h, const double omega[3]) {
  if (int r = check(h)) return r;
  if (omega && !(std::isfinite(omega[0]) && std::isfinite(omega[1]) && std::isfinite(omega[2])))
    return fail(ASLHIP_EINVAL, "ASL ERROR: setOmega: non-finite angular velocity");
  if (int r = flush_deferred(h)) return r;  // the pending step runs with the old frame
  h->has_omega = omega != nullptr;
  for (int d = 0; d < 3; ++d) h->omega[d] = omega ? omega[d] : 0.;
  return 0;
}

int aslhip_set_vmap_skip_outer(aslhip_lattice *h, int on) {
  if (int r = check(h)) return r;
  if (int r = flush_deferred(h)) return r;  // a pending step uses the current link tables
  if (h->vmap_skip_outer != (on != 0)) h->dirty = true;
  h->vmap_skip_outer = on != 0;
  return 0;
}

int aslhip_set_geometry(aslhip_lattice *h, double dx, const double position[3]) {
  if (int r = check(h)) return r;
  if (!position) return fail(ASLHIP_EINVAL, "ASL ERROR: set_geometry: null position");
  if (!(dx > 0.) || !std::isfinite(dx) ||
      !(std::isfinite(position[0]) && std::isfinite(position[1]) && std::isfinite(position[2])))
    return fail(ASLHIP_EINVAL, "ASL ERROR: set_geometry: bad dx or position");
  if (int r = flush_deferred(h)) return r;  // a pending step's BCs use the old positions
  h->dx = dx;
  for (int d = 0; d < 3; ++d) h->pos0[d] = position[d];
  h->dirty = true;  // captured graphs hold the velocity-link arguments by value
  return 0;
}

int aslhip_closure_set(aslhip_lattice *h, const float *params, const float mu[7], const float sc[7], float out_scale) {
  if (int r = check(h)) return r;
  if (params && (h->Q != 19 || h->dtype == ASLHIP_F64))
    return fail(ASLHIP_EINVAL, "ASL ERROR: the closure needs a D3Q19 lattice with FP32 collision");
  if (params && h->turbulence) return fail(ASLHIP_EINVAL, "ASL ERROR: LBGKTurbulence and the closure exclude each other");
  if (params && (!mu || !sc || !std::isfinite(out_scale) || out_scale < 0.f))
    return fail(ASLHIP_EINVAL, "ASL ERROR: closure_set: bad normalisation or output scale");
  if (int r = flush_deferred(h)) return r;  // a pending step runs with the old relaxation
  if (!params) {
    h->has_closure = false;
    return 0;
  }
  ClosureParams c;
  for (int i = 0; i < CL_NPARAM; ++i) {
    if (!std::isfinite(params[i])) return fail(ASLHIP_EINVAL, "ASL ERROR: closure_set: non-finite parameter %d", i);
    c.p[i] = bf16_round(params[i]);
  }
  for (int j = 0; j < CL_NIN; ++j) {
    c.mu[j] = mu[j];
    c.sc[j] = sc[j];
  }
  c.out = out_scale;
  pack_closure(c);
  if (!h->d_cl) HIPCHK(device_alloc(&h->d_cl, sizeof(ClosureParams)));
  HIPCHK(hipStreamSynchronize(h->stream));  // steps queued earlier read the old parameters
  HIPCHK(hipMemcpy(h->d_cl, &c, sizeof c, hipMemcpyHostToDevice));
  h->has_closure = true;
  return 0;
}

int aslhip_set_turbulence(aslhip_lattice *h, int on) {
  if (int r = check(h)) return r;
  if (on && h->has_closure) return fail(ASLHIP_EINVAL, "ASL ERROR: LBGKTurbulence and the closure exclude each other");
  if (int r = flush_deferred(h)) return r;
  h->turbulence = on != 0;
  return 0;
}

int aslhip_closure_set_mode(aslhip_lattice *h, int mode) {
  if (int r = check(h)) return r;
  if (mode != ASLHIP_CLOSURE_FP32 && mode != ASLHIP_CLOSURE_BF16_MFMA)
    return fail(ASLHIP_EINVAL, "ASL ERROR: unknown closure mode %d", mode);
  if (int r = flush_deferred(h)) return r;
  h->closure_mfma = mode == ASLHIP_CLOSURE_BF16_MFMA;
  return 0;
}

int aslhip_closure_features(aslhip_lattice *h, float *out) {
  if (int r = check(h)) return r;
  if (!out) return fail(ASLHIP_EINVAL, "ASL ERROR: closure_features needs an output buffer");
  if (h->Q != 19 || h->dtype == ASLHIP_F64 || !h->periodic)
    return fail(ASLHIP_EINVAL, "ASL ERROR: closure features need a periodic D3Q19 lattice with FP32 collision");
  if (!h->initialized) return fail(ASLHIP_ESTATE, "ASL ERROR: closure_features before initF");
  if (int r = flush_deferred(h)) return r;
  if (int r = prepare(h, false)) return r;
  if (int r = upload_args(h)) return r;
  const long long ncell = (long long)h->n[0] * h->n[1] * h->n[2];
  if (!h->d_feat) HIPCHK(device_alloc(&h->d_feat, (size_t)ncell * CL_NIN * sizeof(float)));
  HIPCHK(launch_closure_features(h->dtype, h->next_odd, h->d_args, ncell, h->d_feat, h->stream));
  return copy_out(h, h->d_feat, out, (size_t)ncell * CL_NIN * sizeof(float));
}

int aslhip_set_compute_macro(aslhip_lattice *h, int comp_rho, int comp_vel) {
  if (int r = check(h)) return r;
  h->comp_rho = comp_rho != 0;
  h->comp_vel = comp_vel != 0;
  return 0;
}

int aslhip_init_equilibrium(aslhip_lattice *h, double rho, const double u[3]) {
  if (int r = check(h)) return r;
  if (int r = flush_deferred(h)) return r;
  if (int r = order_after_consumer(h)) return r;
  InitArgs a;
  a.f = h->f;
  a.qs_bytes = h->qs_bytes;
  a.len = h->len;
  a.rho0 = rho;
  for (int d = 0; d < 3; ++d) a.u0[d] = u ? u[d] : 0.;
  a.rho_in = a.u_in = nullptr;
  a.rho = h->rho;
  a.u = h->u;
  HIPCHK(launch_init(h->Q, h->dtype, a, h->stream));
  h->initialized = true;
  h->fresh = true;
  h->bc_since_init = false;
  h->next_odd = true;
  h->pending.clear();
  return 0;
}

int aslhip_init_equilibrium_field(aslhip_lattice *h, const void *rho, const void *u) {
  if (int r = check(h)) return r;
  if (int r = flush_deferred(h)) return r;
  if (int r = order_after_consumer(h)) return r;
  if (!u) return fail(ASLHIP_EINVAL, "ASL ERROR: initF needs a velocity field");
  void *drho = nullptr, *du = nullptr;
  const size_t n = (size_t)h->len * h->melem;
  hipError_t e = device_alloc(&du, 3 * n);
  if (e == hipSuccess && rho) e = device_alloc(&drho, n);
  // the stream is waited for below, before the caller may change the fields
  if (e == hipSuccess) e = to_device(du, u, 3 * n, h->stream, false);
  if (e == hipSuccess && rho) e = to_device(drho, rho, n, h->stream, false);
  InitArgs a;
  a.f = h->f;
  a.qs_bytes = h->qs_bytes;
  a.len = h->len;
  a.rho0 = 1.;
  a.u0[0] = a.u0[1] = a.u0[2] = 0.;
  a.rho_in = drho;
  a.u_in = du;
  a.rho = h->rho;
  a.u = h->u;
  if (e == hipSuccess) e = launch_init(h->Q, h->dtype, a, h->stream);
  const hipError_t done = hipStreamSynchronize(h->stream);
  if (du) (void)hipFree(du);
  if (drho) (void)hipFree(drho);
  if (e != hipSuccess || done != hipSuccess)
    return fail(ASLHIP_EHIP, "ASL ERROR: initial fields: %s", hipGetErrorString(e != hipSuccess ? e : done));
  h->initialized = true;
  h->fresh = true;
  h->bc_since_init = false;
  h->next_odd = true;
  h->pending.clear();
  return 0;
}

int aslhip_template(int q, int *c, double *w, int *inv) {
  if (q != 15 && q != 19 && q != 27) return fail(ASLHIP_EINVAL, "ASL ERROR: no template with %d directions", q);
  const Templ t = make_templ(q);
  for (int i = 0; i < q; ++i) {
    for (int d = 0; d < 3; ++d)
      if (c) c[3 * i + d] = t.c[i][d];
    if (w) w[i] = t.w[i];
    if (inv) inv[i] = t.inv[i];
  }
  return 0;
}

int aslhip_write_f(aslhip_lattice *h, const void *f) {
  if (int r = check(h)) return r;
  if (!f) return fail(ASLHIP_EINVAL, "ASL ERROR: write_f needs populations");
  if (int r = flush_deferred(h)) return r;
  if (int r = order_after_consumer(h)) return r;
  void *d = nullptr;
  const size_t bytes = (size_t)h->len * h->Q * h->melem;
  HIPCHK(scratch_take(h->view, bytes, &d));
  hipError_t e = to_device(d, f, bytes, h->stream);
  WriteFArgs a;
  a.f = h->f;
  a.qs_bytes = h->qs_bytes;
  a.len = h->len;
  a.compressible = h->compressible ? 1 : 0;
  a.in = d;
  a.rho = h->rho;
  a.u = h->u;
  if (e == hipSuccess) e = launch_write_f(h->Q, h->dtype, a, h->stream);
  const hipError_t done = scratch_give(h->view, bytes, d, h->stream);
  HIPCHK(e != hipSuccess ? e : done);
  h->initialized = true;
  h->fresh = true;
  h->bc_since_init = false;
  h->next_odd = true;
  h->pending.clear();
  return 0;
}

int aslhip_bc_add_slice(aslhip_lattice *h, int kind, unsigned faces, double p, const double u[3], int *bc_id) {
  if (int r = check(h)) return r;
  if (h->periodic) return fail(ASLHIP_EINVAL, "ASL ERROR: slice BCs need a non-periodic lattice");
  if (kind < ASLHIP_BC_NOSLIP || kind > ASLHIP_BC_CONSTANT_PRESSURE_VELOCITY)
    return fail(ASLHIP_EINVAL, "ASL ERROR: %d is not a slice BC kind", kind);
  if (faces == 0 || faces > 63u) return fail(ASLHIP_EINVAL, "ASL ERROR: bad face mask %u", faces);
  BCDesc b;
  b.kind = kind;
  b.faces = faces;
  b.p = p;
  for (int d = 0; d < 3; ++d) b.u[d] = u ? u[d] : 0.;
  h->bcs.push_back(std::move(b));
  if (bc_id) *bc_id = static_cast<int>(h->bcs.size()) - 1;
  h->dirty = true;
  return 0;
}

int aslhip_bc_add_map(aslhip_lattice *h, int kind, const float *map, const float *cdomain, double p,
                      const double u[3], const double rot[6], int *bc_id) {
  if (int r = check(h)) return r;
  if (h->periodic) return fail(ASLHIP_EINVAL, "ASL ERROR: map BCs need a non-periodic lattice");
  if (kind < ASLHIP_BC_NOSLIP_MAP || kind > ASLHIP_BC_VELOCITY_MAP)
    return fail(ASLHIP_EINVAL, "ASL ERROR: %d is not a map BC kind", kind);
  if (!map) return fail(ASLHIP_EINVAL, "ASL ERROR: map BC without a map");
  BCDesc b;
  b.kind = kind;
  b.p = p;
  for (int d = 0; d < 3; ++d) b.u[d] = u ? u[d] : 0.;
  if (rot) {
    b.has_rot = true;
    for (int d = 0; d < 6; ++d) b.rot[d] = rot[d];
  }
  b.map.assign(map, map + h->len);
  if (cdomain) b.cd.assign(cdomain, cdomain + h->len);
  h->bcs.push_back(std::move(b));
  if (bc_id) *bc_id = static_cast<int>(h->bcs.size()) - 1;
  h->dirty = true;
  return 0;
}

int aslhip_vis_add(aslhip_lattice *h, int kind, const float *map, const double u[3], const double rot[6],
                   int *vis_id) {
  if (int r = check(h)) return r;
  if (kind < ASLHIP_VIS_NOSLIP_VEL || kind > ASLHIP_VIS_VELOCITY)
    return fail(ASLHIP_EINVAL, "ASL ERROR: %d is not a visualisation fill kind", kind);
  if (!map) return fail(ASLHIP_EINVAL, "ASL ERROR: visualisation fill without a map");
  if (h->Q == 27 && kind != ASLHIP_VIS_VELOCITY)
    return fail(ASLHIP_EINVAL, "ASL ERROR: d3q27 has no laplace / gradient coefficients for this fill");
  aslhip_lattice::Vis v{kind, nullptr, {0., 0., 0.}, rot != nullptr, {0., 0., 0., 0., 0., 0.}};
  for (int d = 0; d < 3; ++d) v.u[d] = u ? u[d] : 0.;
  if (rot)
    for (int d = 0; d < 6; ++d) v.rot[d] = rot[d];
  const size_t bytes = (size_t)h->len * sizeof(float);
  if (device_alloc(&v.map, bytes) != hipSuccess) return fail(ASLHIP_ENOMEM, "ASL ERROR: visualisation fill: out of memory");
  if (hipMemcpy(v.map, map, bytes, hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipFree(v.map);
    return fail(ASLHIP_EHIP, "ASL ERROR: visualisation fill: map upload failed");
  }
  h->vis.push_back(v);
  if (vis_id) *vis_id = static_cast<int>(h->vis.size()) - 1;
  return 0;
}

int aslhip_vis_execute(aslhip_lattice *h, int vis_id) {
  if (int r = check(h)) return r;
  if (vis_id < 0 || vis_id >= (int)h->vis.size())
    return fail(ASLHIP_EINVAL, "ASL ERROR: unknown visualisation fill id %d", vis_id);
  if (!h->initialized) return fail(ASLHIP_ESTATE, "ASL ERROR: visualisation fill before initF");
  // rho and u must hold the last step's values (a deferred step writes them)
  if (int r = flush_deferred(h)) return r;
  if (int r = order_after_consumer(h)) return r;
  const aslhip_lattice::Vis &v = h->vis[vis_id];
  VisArgs a;
  a.map = v.map;
  a.rho = h->rho;
  a.u = h->u;
  a.kind = v.kind;
  a.len = h->len;
  a.sx = h->sx;
  a.sy = h->sy;
  for (int d = 0; d < 3; ++d) a.u0[d] = v.u[d];
  for (int d = 0; d < 6; ++d) a.rot[d] = v.rot[d];
  a.has_rot = v.has_rot ? 1 : 0;
  a.dx = h->dx;
  for (int d = 0; d < 3; ++d) a.pos0[d] = h->pos0[d];
  HIPCHK(launch_vis(h->Q, h->dtype, a, h->stream));
  return 0;
}

int aslhip_bc_execute(aslhip_lattice *h, int bc_id) {
  if (int r = check(h)) return r;
  if (bc_id < 0 || bc_id >= (int)h->bcs.size()) return fail(ASLHIP_EINVAL, "ASL ERROR: unknown BC id %d", bc_id);
  // a BC executed twice in one cycle counts at its last position
  auto it = std::find(h->pending.begin(), h->pending.end(), bc_id);
  if (it != h->pending.end()) h->pending.erase(it);
  h->pending.push_back(bc_id);
  if (h->fresh) h->bc_since_init = true;
  return 0;
}

int aslhip_finalize(aslhip_lattice *h) {
  if (int r = check(h)) return r;
  // a deferred step keeps the order it was requested with
  if (int r = flush_deferred(h)) return r;
  if (!h->pending.empty()) {
    if (h->pending != h->order) {
      h->order = h->pending;
      h->dirty = true;
    }
    h->pending.clear();
  }
  return h->dirty ? finalize_impl(h) : 0;
}

int aslhip_step(aslhip_lattice *h, int nsteps, unsigned flags) {
  if (int r = check(h)) return r;
  return step_impl(h, nsteps, flags, nullptr);
}

int aslhip_synchronize(aslhip_lattice *h) {
  if (int r = check(h)) return r;
  if (int r = flush_deferred(h)) return r;
  HIPCHK(hipStreamSynchronize(h->stream));
  h->queued = 0;
  return 0;
}

int aslhip_read_rho(aslhip_lattice *h, void *out) {
  if (int r = check(h)) return r;
  if (int r = flush_deferred(h)) return r;
  return copy_out(h, h->rho, out, (size_t)h->len * h->melem);
}

int aslhip_read_velocity(aslhip_lattice *h, void *out) {
  if (int r = check(h)) return r;
  if (int r = flush_deferred(h)) return r;
  return copy_out(h, h->u, out, (size_t)h->len * 3 * h->melem);
}

int aslhip_macro_device(aslhip_lattice *h, void *stream, const void **rho, const void **u) {
  if (int r = check(h)) return r;
  if (!rho && !u) return fail(ASLHIP_EINVAL, "ASL ERROR: macro_device: no output address");
  if (int r = flush_deferred(h)) return r;
  if (!stream) {
    HIPCHK(hipStreamSynchronize(h->stream));  // readable from any stream until the next step
  } else {
    if (!h->ev_macro) HIPCHK(hipEventCreateWithFlags(&h->ev_macro, hipEventDisableTiming));
    if (!h->ev_consumer) HIPCHK(hipEventCreateWithFlags(&h->ev_consumer, hipEventDisableTiming));
    hipStream_t c = static_cast<hipStream_t>(stream);
    if (h->consumer && h->consumer != c) {
      // the earlier consumer's reads still come before the next step
      if (int r = order_after_consumer(h)) return r;
    }
    HIPCHK(hipEventRecord(h->ev_macro, h->stream));
    HIPCHK(hipStreamWaitEvent(c, h->ev_macro, 0));
    h->consumer = c;
  }
  if (rho) *rho = h->rho;
  if (u) *u = h->u;
  return 0;
}

int aslhip_read_f_noalloc(aslhip_lattice *h, void *out) {
  if (int r = check(h)) return r;
  if (!out) return fail(ASLHIP_EINVAL, "ASL ERROR: read_f_noalloc needs an output buffer");
  int dev = -1;
  HIPCHK(hipGetDevice(&dev));
  if (dev != h->device)
    return fail(ASLHIP_EINVAL, "ASL ERROR: read_f_noalloc: the lattice lives on device %d, device %d is current",
                h->device, dev);
  if ((size_t)h->Q * h->melem > ASLHIP_NOALLOC_SCRATCH_BYTES)
    return fail(ASLHIP_EINVAL, "ASL ERROR: read_f_noalloc: one cell's populations exceed the %u-byte staging array",
                ASLHIP_NOALLOC_SCRATCH_BYTES);
  if (h->deferred && (h->dirty || !h->pending.empty()))
    return fail(ASLHIP_ESTATE, "ASL ERROR: read_f_noalloc: the pending step needs its boundary tables rebuilt "
                               "(an allocation); call aslhip_finalize first");
  void *buf = nullptr;
  HIPCHK(noalloc_scratch(&buf));
  int r = aslhip::read_f_through(h, out, buf, ASLHIP_NOALLOC_SCRATCH_BYTES, false);
  (void)hipStreamSynchronize(h->stream);
  return r;
}

int aslhip_read_f(aslhip_lattice *h, void *out) {
  if (int r = check(h)) return r;
  if (!out) return fail(ASLHIP_EINVAL, "ASL ERROR: read_f needs an output buffer");
  if (int r = flush_deferred(h)) return r;
  void *d = nullptr;
  const size_t bytes = (size_t)h->len * h->Q * h->melem;
  HIPCHK(scratch_take(h->view, bytes, &d));
  int r = aslhip::read_f_through(h, out, d, bytes, true);
  (void)hipStreamSynchronize(h->stream);
  h->queued = 0;
  const hipError_t done = scratch_give(h->view, bytes, d);
  if (r) return r;
  HIPCHK(done);
  return 0;
}

}  // extern "C"

namespace {

// ComputeSurfaceForceMap / ComputeSurfaceFluxMap on the device.  The map and
// the result go through a kept buffer (allocating and freeing on each call took
// longer than the kernel).
int surface_impl(aslhip_lattice *h, const float *map, void *out, bool flux) {
  if (int r = check(h)) return r;
  if (!map || !out) return fail(ASLHIP_EINVAL, "ASL ERROR: surface force/flux needs a map and an output field");
  if (!h->initialized) return fail(ASLHIP_ESTATE, "ASL ERROR: surface force/flux before initF");
  if (is_wide(h)) return fail(ASLHIP_EINVAL, "ASL ERROR: surface force/flux on lattices over 4 GiB is not supported");
  if (int r = flush_deferred(h)) return r;
  if (int r = prepare(h, false)) return r;
  if (int r = upload_args(h)) return r;
  const size_t len = (size_t)h->len, outb = len * 3 * h->melem, mapb = len * sizeof(float);
  void *d = nullptr;
  if (scratch_take(h->surface, outb + mapb, &d) != hipSuccess)
    return fail(ASLHIP_EHIP, "ASL ERROR: surface force/flux: out of memory");
  SurfaceArgs s;
  s.out = d;
  float *dmap = reinterpret_cast<float *>(static_cast<char *>(d) + outb);
  s.map = dmap;
  s.len = h->len;
  s.per = h->periodic ? 1 : 0;
  s.after_odd = h->next_odd ? 0 : 1;
  s.flux = flux ? 1 : 0;
  hipError_t e = to_device(dmap, map, mapb, h->stream);
  if (e == hipSuccess) e = launch_surface(h->Q, h->dtype, s, h->h_direct, h->d_args, h->stream);
  const int r = e == hipSuccess ? copy_out(h, d, out, flux ? len * h->melem : outb) : 0;
  const hipError_t done = scratch_give(h->surface, outb + mapb, d, e == hipSuccess && r == 0 ? nullptr : h->stream);
  HIPCHK(e != hipSuccess ? e : done);
  return r;
}

}  // namespace

extern "C" {

int aslhip_surface_force(aslhip_lattice *h, const float *map, void *out) { return surface_impl(h, map, out, false); }

int aslhip_surface_flux(aslhip_lattice *h, const float *map, void *out) { return surface_impl(h, map, out, true); }

int aslhip_read_cell_types(aslhip_lattice *h, uint8_t *out) {
  if (int r = check(h)) return r;
  if (h->dirty) {
    int r = aslhip_finalize(h);
    if (r) return r;
  }
  return copy_out(h, h->code, out, (size_t)h->len);
}

int aslhip_reduce_conservation(aslhip_lattice *h, double out[5]) {
  if (int r = check(h)) return r;
  if (int r = flush_deferred(h)) return r;
  if (h->dirty) {
    int r = aslhip_finalize(h);
    if (r) return r;
  }
  ReduceArgs a;
  a.f = h->f;
  a.qs_bytes = h->qs_bytes;
  a.sx = h->sx;
  a.sy = h->sy;
  a.len = h->len;
  a.per = h->periodic ? 1 : 0;
  a.nx = h->n[0];
  a.ny = h->n[1];
  a.nz = h->n[2];
  a.after_odd = h->next_odd ? 0 : 1;
  a.code = h->code;
  a.partial = h->red_partial;
  HIPCHK(launch_reduce(h->Q, h->dtype, a, h->red_out, h->stream));
  return copy_out(h, h->red_out, out, 5 * sizeof(double));
}

int aslhip_stats(aslhip_lattice *h, int64_t out[4]) {
  if (int r = check(h)) return r;
  if (h->dirty) {
    int r = aslhip_finalize(h);
    if (r) return r;
  }
  out[0] = h->n_counted;
  out[1] = h->n_computed;
  out[2] = h->n_boundary;
  out[3] = h->n_patterns;
  return 0;
}

int aslhip_get_tuning(aslhip_lattice *h, int *block, int *remap) {
  if (int r = check(h)) return r;
  if (block) *block = step_workgroup(h, h->tune_block);
  if (remap) *remap = h->tune_remap;
  return 0;
}

int aslhip_set_tuning(aslhip_lattice *h, int knob, int value) {
  if (int r = check(h)) return r;
  if (knob == ASLHIP_TUNE_WIDE) {
    if (value != 0 && value != 1) return fail(ASLHIP_EINVAL, "ASL ERROR: ASLHIP_TUNE_WIDE takes 0 or 1");
    if (int r = flush_deferred(h)) return r;
    if ((value != 0) != h->force_wide) drop_graphs(h);  // captured launches name the variant
    h->force_wide = value != 0;
    return 0;
  }
  if (knob == ASLHIP_TUNE_XCD_REMAP) {
    if (value < 0 || value > 4096) return fail(ASLHIP_EINVAL, "ASL ERROR: XCD run length %d outside 0..4096", value);
    if (int r = flush_deferred(h)) return r;
    if (value != h->tune_remap || !h->remap_set) drop_graphs(h);  // captured launches carry the old order
    h->tune_remap = value;
    h->remap_set = true;
    return 0;
  }
  if (knob == ASLHIP_TUNE_CPL) {
    if (value != 0 && value != 1 && value != 2 && value != 4)
      return fail(ASLHIP_EINVAL, "ASL ERROR: cells per lane %d is not 0 (automatic), 1, 2 or 4", value);
    if (int r = flush_deferred(h)) return r;
    if (value != h->tune_cpl) drop_graphs(h);  // captured launches name the variant and grid
    h->tune_cpl = value;
    return 0;
  }
  if (knob == ASLHIP_TUNE_BLOCK) {
    if (value < 64 || value > STEP_BLOCK || value % 64)
      return fail(ASLHIP_EINVAL, "ASL ERROR: workgroup size %d is not a multiple of 64 in 64..%d", value, STEP_BLOCK);
    if (int r = flush_deferred(h)) return r;
    if (value != h->tune_block || !h->block_set) drop_graphs(h);  // captured launches carry the old grid
    h->tune_block = value;
    h->block_set = true;
    return 0;
  }
  if (knob == ASLHIP_TUNE_SWEEP_KB) {
    if (value < -1) return fail(ASLHIP_EINVAL, "ASL ERROR: ASLHIP_TUNE_SWEEP_KB takes a window in KiB, 0 or -1");
    if (int r = flush_deferred(h)) return r;
    h->tune_sweep = value;
    return 0;
  }
  if (knob == ASLHIP_TUNE_LDS) {
    if (value < 0 || value > 2) return fail(ASLHIP_EINVAL, "ASL ERROR: ASLHIP_TUNE_LDS takes 0, 1 or 2");
    if (int r = flush_deferred(h)) return r;
    if (value != h->tune_lds) drop_graphs(h);  // captured launches name the variant and grid
    h->tune_lds = value;
    return 0;
  }
  return fail(ASLHIP_EINVAL, "ASL ERROR: unknown tuning knob %d", knob);
}

int aslhip_sweep_plan(int nx, int periodic, int planes, int steps, int nsteps, int *out, int cap) {
  if (nx < 1 || planes < 1 || steps < 1 || nsteps < 0 || cap < 0 || (cap > 0 && !out) || (periodic && steps > nx))
    return fail(ASLHIP_EINVAL, "ASL ERROR: sweep_plan: bad arguments");
  // a step has at least one launch per block
  long long count = nsteps * ((static_cast<long long>(nx) + planes - 1) / planes);
  if (count > INT_MAX) return fail(ASLHIP_EINVAL, "ASL ERROR: sweep_plan: too many launches to count");
  count = 0;
  sweep_plan(nx, periodic != 0, planes, steps, nsteps, [&](const SweepLaunch &l) {
    if (count < cap) {
      out[3 * count] = l.step;
      out[3 * count + 1] = l.p0;
      out[3 * count + 2] = l.np;
    }
    return ++count <= INT_MAX;
  });
  if (count > INT_MAX) return fail(ASLHIP_EINVAL, "ASL ERROR: sweep_plan: too many launches to count");
  return static_cast<int>(count);
}

int aslhip_tuning_value(aslhip_lattice *h, int knob, int *value) {
  if (int r = check(h)) return r;
  if (!value) return fail(ASLHIP_EINVAL, "ASL ERROR: tuning_value needs an output");
  switch (knob) {
    case ASLHIP_TUNE_XCD_REMAP: *value = h->remap_set ? h->tune_remap : step_args(h).g.remap; return 0;
    case ASLHIP_TUNE_BLOCK: *value = step_workgroup(h, step_lanes(h, false)); return 0;
    case ASLHIP_TUNE_WIDE: *value = is_wide(h) ? 1 : 0; return 0;
    case ASLHIP_TUNE_CPL: *value = effective_cpl(h); return 0;
    case ASLHIP_TUNE_LDS: *value = effective_lds(h); return 0;
    case ASLHIP_TUNE_SWEEP_KB: *value = h->tune_sweep; return 0;
    default: return fail(ASLHIP_EINVAL, "ASL ERROR: unknown tuning knob %d", knob);
  }
}

}  // extern "C"

namespace {

// Times nsteps steps between two events; each: with events around every launch,
// one launch per step (no sweeps, no graphs).
int time_run(aslhip_lattice *h, int nsteps, unsigned flags, bool each, double *ms_total, double *ms_kernel,
             double *ms_each) {
  if (int r = flush_deferred(h)) return r;
  flags &= ~ASLHIP_STEP_DEFER;
  if (h->dirty || !h->pending.empty()) {
    int r = aslhip_finalize(h);
    if (r) return r;
  }
  std::vector<hipEvent_t> ev(each ? 2 * (size_t)nsteps : 0);
  for (auto &e : ev) HIPCHK(hipEventCreate(&e));
  hipEvent_t t0, t1;
  HIPCHK(hipEventCreate(&t0));
  HIPCHK(hipEventCreate(&t1));
  HIPCHK(hipEventRecord(t0, h->stream));
  int r = step_impl(h, nsteps, flags, each ? &ev : nullptr);
  HIPCHK(hipEventRecord(t1, h->stream));
  HIPCHK(hipEventSynchronize(t1));
  if (r == 0) {
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, t0, t1));
    if (ms_total) *ms_total = ms;
    double ksum = 0.;
    for (int s = 0; s < nsteps; ++s) {
      float k = 0.f;
      if (each) HIPCHK(hipEventElapsedTime(&k, ev[2 * s], ev[2 * s + 1]));
      ksum += k;
      if (ms_each) ms_each[s] = k;
    }
    if (ms_kernel) *ms_kernel = ksum;
  }
  for (auto &e : ev) (void)hipEventDestroy(e);
  (void)hipEventDestroy(t0);
  (void)hipEventDestroy(t1);
  return r;
}

}  // namespace

extern "C" {

int aslhip_autotune(aslhip_lattice *h, int nsteps, int *best_block, int *best_remap) {
  if (int r = check(h)) return r;
  if (nsteps < 1) return fail(ASLHIP_EINVAL, "ASL ERROR: autotune needs at least one step per candidate");
  nsteps += nsteps & 1;
  if (int r = flush_deferred(h)) return r;
  const int remaps[6] = {0, 2, 4, 8, 16, 64};
  // Direct kernel: these stand for the automatic order (xcd_run) and workgroup
  // (step_lanes), which small lattices and D3Q27 in FP64 run better with than with
  // any fixed value here.
  const int preset = h->selem == 2 ? 64 : 4, lanes = 512;
  struct Candidate {
    int lds, cpl, remap, block;
  };
  auto set = [&](const Candidate &c) {
    drop_graphs(h);
    h->tune_lds = c.lds;
    h->tune_cpl = c.cpl;
    h->tune_remap = c.remap;
    h->remap_set = c.remap != preset;
    h->tune_block = c.block;
    h->block_set = c.block != lanes;
  };
  const Candidate automatic = {-1, 0, preset, lanes};
  set(automatic);
  const int auto_lds = effective_lds(h);
  // Lattices whose runs of nsteps steps sweep, with the direct kernel at least:
  // candidates are compared by whole runs, as aslhip_step takes them, others by
  // the time of their launches.
  int g = 0, t = 0;
  set({0, 1, preset, lanes});
  sweep_shape(h, nsteps, g, t);
  const bool sweeping = t > 0;
  // the distinct cells-per-lane values this lattice can run (sweeps take one)
  std::vector<int> cpls;
  for (int c : {1, 2, 4}) {
    set({0, c, preset, lanes});
    if (effective_cpl(h) == c && (c == 1 || !sweeping)) cpls.push_back(c);
  }
  set({1, 0, preset, lanes});
  const bool tiles = effective_lds(h) != 0;
  std::vector<Candidate> all;
  if (sweeping) all.push_back(automatic);
  // LDS-staged tiles where the lattice can run them: on every step (fixed
  // workgroup), on even steps (workgroup of the odd steps' direct kernel; sweeps
  // of such a lattice are those of the direct kernel)
  if (tiles) {
    for (int remap : remaps) all.push_back({1, 0, remap, lanes});
    for (int remap : remaps)
      for (int blk : {256, 512, 1024})
        if (!sweeping) all.push_back({2, 0, remap, blk});
  }
  for (int cpl : cpls)
    for (int remap : remaps)
      for (int blk : {256, 512, 1024}) all.push_back({0, cpl, remap, blk});
  double best = 1e300, auto_ms = 1e300;
  Candidate win = automatic;
  for (Candidate c : all) {
    // what a lattice that does not sweep launches by itself
    const bool is_auto = c.lds < 0 || (!sweeping && c.lds == auto_lds && c.cpl <= 1 && c.remap == preset && c.block == lanes);
    if (is_auto) c = automatic;
    set(c);
    double tot = 0., ker = 0.;
    if (int r = time_run(h, nsteps, 0u, !sweeping, &tot, &ker, nullptr)) return r;
    const double ms = sweeping ? tot : ker;
    if (is_auto) auto_ms = ms;
    if (ms < best) {
      best = ms;
      win = c;
    }
  }
  if (best > 0.98 * auto_ms) win = automatic;  // a fixed setting has to be worth it
  set(win);
  if (best_block) *best_block = step_workgroup(h, h->tune_block);
  if (best_remap) *best_remap = win.remap;
  return 0;
}

int aslhip_time_steps(aslhip_lattice *h, int nsteps, unsigned flags, double *ms_total, double *ms_kernel,
                      double *ms_each) {
  if (int r = check(h)) return r;
  if (int r = flush_deferred(h)) return r;
  if (nsteps < 1) return fail(ASLHIP_EINVAL, "ASL ERROR: time_steps needs at least one step");
  // replayed graphs have no events between their launches
  return time_run(h, nsteps, flags, (flags & ASLHIP_STEP_GRAPH) == 0, ms_total, ms_kernel, ms_each);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Batches of lattices
// ---------------------------------------------------------------------------
struct aslhip_batch {
  std::vector<aslhip_lattice *> lat;
  int Q = 19, dtype = ASLHIP_F32;
  bool periodic = false, wide = false;
  hipStream_t stream = nullptr;
  hipEvent_t done = nullptr;
  StepArgs *desc = nullptr;  // [2][2][n]: launches of groups, of all; each plain steps, then steps writing rho/u
  uint2 *ent = nullptr;      // [2][all workgroups]: lattice, chunk; group by group, then for launches of all groups
  int block = STEP_BLOCK;    // workgroup size of all lattices of the batch (direct kernel)
  int tune_lds = -1;         // LDS-staged tiles: 1 on, 0 off, -1 by group (batch_tile)
  // Runs of several steps go group by group: each group of consecutive
  // lattices (at most group_mb MiB of populations; 0: one group; -1: automatic)
  // takes all the run's steps (a graph chunk, or the steps of an eager call)
  // before the next starts, so a group that fits the 256 MiB Infinity Cache is
  // stepped from cache.
  int group_mb = -1;
  // Measured on D3Q19 FP32 cavities, one group -> groups of 224 MiB: 16 of
  // 32^3..96^3 (330 MiB) 135 -> 123 us per step, 64 of 32^3..160^3 (4.1 GiB)
  // 1675 -> 1535; with 512 lanes 128 MiB 128.5 and 1633, 192 MiB 127.5 and 1621,
  // 224 MiB 127.0 and 1588.
  struct Range {  // workgroups of one launch: entries [first, end)
    int first, end;
    bool tile, all;
  };
  std::vector<Range> groups;  // one launch per step of each group
  Range all;                  // one launch per step of all lattices
  std::vector<char> tile;     // per lattice: its group's
  hipGraphExec_t graph[2] = {nullptr, nullptr};  // chunks starting with an even / odd step
  std::vector<StepArgs> hdesc;                    // host copy of desc (source of the async upload)
};

namespace {

// Tiles for the steps of a group of that many bytes: non-periodic batches under
// 4 GiB per lattice.  Automatic for D3Q19 FP32 groups that stream from HBM, as for
// single lattices: three of 220^3 1056 (direct) -> 1010 us per step, six of 166^3
// 969 -> 951; groups that step from the cache are faster with the direct kernel
// (the cavities of batch_group_bytes's figures: 127 against 136, 1621 against 1708).
bool batch_tile(const aslhip_batch *b, long long bytes) {
  if (b->periodic || b->wide) return false;
  return b->tune_lds < 0 ? b->Q == 19 && b->dtype == ASLHIP_F32 && bytes > CACHE_BYTES : b->tune_lds != 0;
}

// Steps from which an eager run goes group by group: a group's first step reads
// HBM in any case, and every group adds launches.  16 cavities of 32^3..96^3,
// one group -> groups, us per step: 2 steps 242 -> 285, 10 steps 178 -> 173,
// 100 steps 152 -> 145; 20 FP16 cavities of 96^3: 438 -> 496, 358 -> 336, 327 -> 294.
constexpr int BATCH_GROUP_STEPS = 8;

// Populations a group may hold, in bytes (0: all lattices form one group).
// Automatic: 224 MiB where the batch is larger than the Infinity Cache.
long long batch_group_bytes(const aslhip_batch *b) {
  if (b->group_mb >= 0) return static_cast<long long>(b->group_mb) << 20;
  long long bytes = 0;
  for (const aslhip_lattice *h : b->lat) bytes += h->qs_bytes * h->Q;
  return bytes > CACHE_BYTES ? SWEEP_WINDOW : 0;
}

// The group of each lattice, ascending from 0.  Lattices larger than the
// Infinity Cache stream from HBM in any case and share a group of their own (a
// launch per step for all of them); the others fill groups in order, split
// evenly so that no group is a small rest.
std::vector<int> batch_group_of(const aslhip_batch *b) {
  const long long budget = batch_group_bytes(b);
  std::vector<int> of(b->lat.size(), 0);
  if (!budget) return of;
  auto bytes = [&](size_t l) { return b->lat[l]->qs_bytes * b->lat[l]->Q; };
  long long rest = 0;
  int g = 0;
  for (size_t l = 0; l < of.size(); ++l)
    if (bytes(l) <= CACHE_BYTES)
      rest += bytes(l);
    else
      g = 1;
  const long long n = (rest + budget - 1) / budget, target = n ? (rest + n - 1) / n : 0;
  long long in = 0;
  for (size_t l = 0; l < of.size(); ++l) {
    if (bytes(l) > CACHE_BYTES) continue;
    if (in && (in >= target || in + bytes(l) > budget)) {
      ++g;
      in = 0;
    }
    in += bytes(l);
    of[l] = g;
  }
  return of;
}

// One lattice's step arguments in the batch's launch shape.
StepArgs batch_args(const aslhip_batch *b, const aslhip_lattice *h, bool tile) {
  return step_args(h, b->block, 1, false, tile);
}

void batch_free(aslhip_batch *b) {
  for (auto &g : b->graph)
    if (g) (void)hipGraphExecDestroy(g);
  void *ptrs[] = {b->desc, b->ent};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  if (b->done) (void)hipEventDestroy(b->done);
  if (b->stream) (void)hipStreamDestroy(b->stream);
}

// One step of the lattices whose workgroup entries are [e0, e1).
int batch_launch(aslhip_batch *b, bool odd, bool macro, const aslhip_batch::Range &e) {
  BatchLaunch L;
  L.desc = b->desc + ((e.all ? 2 : 0) + (macro ? 1 : 0)) * b->lat.size();
  L.ent = b->ent + e.first;
  L.nblocks = e.end - e.first;
  L.tile = e.tile ? 1 : 0;
  L.block = e.tile ? STEP_TILE : std::min(b->block, step_block(b->Q, static_cast<int>(b->lat[0]->selem)));
  HIPCHK(launch_step_batch(b->Q, b->dtype, odd, b->periodic, b->wide, L, b->stream));
  return 0;
}

// The workgroup table for the batch's settings (the lattices in order).  On
// failure the batch keeps the table it has.
int batch_tables(aslhip_batch *b) {
  const std::vector<int> of = batch_group_of(b);
  const int ng = *std::max_element(of.begin(), of.end()) + 1;
  std::vector<long long> bytes(ng, 0);
  for (size_t l = 0; l < of.size(); ++l) bytes[of[l]] += b->lat[l]->qs_bytes * b->lat[l]->Q;
  std::vector<char> tile(of.size());
  for (size_t l = 0; l < of.size(); ++l) tile[l] = batch_tile(b, bytes[of[l]]);
  std::vector<uint2> ent;
  auto add = [&](size_t l, bool t) {
    const StepArgs a = batch_args(b, b->lat[l], t);
    for (int c = 0; c < a.g.nchunks; ++c) ent.push_back(make_uint2(static_cast<unsigned>(l), static_cast<unsigned>(c)));
  };
  // Each XCD (workgroup id modulo 8) takes one run of the chunks of a group that
  // the Infinity Cache holds (see xcd_run), others the hardware order: the
  // cavities of batch_group_bytes's figures 123 -> 115 and 1535 -> 1437, 20 FP16
  // ones of 96^3 293 -> 272; streamed from HBM, 200^3 and three small D3Q27
  // lattices would take 362 instead of 344.
  std::vector<aslhip_batch::Range> groups;
  for (int g = 0; g < ng; ++g) {
    const size_t first = ent.size();
    for (size_t l = 0; l < of.size(); ++l)
      if (of[l] == g) add(l, tile[l] != 0);
    if (bytes[g] <= CACHE_BYTES) {
      const std::vector<uint2> plain(ent.begin() + first, ent.end());
      const size_t share = plain.size() / 8;
      for (size_t i = 0; i < 8 * share; ++i) ent[first + i] = plain[(i % 8) * share + i / 8];
    }
    groups.push_back({static_cast<int>(first), static_cast<int>(ent.size()), batch_tile(b, bytes[g]), false});
  }
  // all in one launch: streamed from HBM if there are several groups
  const bool t = batch_tile(b, std::accumulate(bytes.begin(), bytes.end(), 0LL));
  const size_t first = ent.size();
  for (int g = 0; g < ng; ++g)
    for (size_t l = 0; l < of.size(); ++l)
      if (of[l] == g) add(l, t);
  const aslhip_batch::Range all = {static_cast<int>(first), static_cast<int>(ent.size()), t, true};
  // replays in flight read the old tables and graphs: finish them first
  HIPCHK(hipStreamSynchronize(b->stream));
  uint2 *d = nullptr;
  HIPCHK(device_alloc(&d, ent.size() * sizeof(uint2)));
  if (hipError_t e = hipMemcpy(d, ent.data(), ent.size() * sizeof(uint2), hipMemcpyHostToDevice); e != hipSuccess) {
    (void)hipFree(d);
    return fail(ASLHIP_EHIP, "ASL ERROR: batch tables: %s", hipGetErrorString(e));
  }
  for (auto &g : b->graph)
    if (g) {
      (void)hipGraphExecDestroy(g);
      g = nullptr;
    }
  if (b->ent) (void)hipFree(b->ent);
  b->ent = d;
  b->groups = std::move(groups);
  b->all = all;
  b->tile = std::move(tile);
  return 0;
}

int batch_set(aslhip_batch *b, int *setting, int value) {
  const int old = *setting;
  if (value == old) return 0;
  *setting = value;
  const int r = batch_tables(b);
  if (r) *setting = old;  // the table of the old setting is still there
  return r;
}

int batch_graph(aslhip_batch *b, bool odd) {
  hipGraphExec_t &g = b->graph[odd ? 1 : 0];
  if (g) return 0;
  hipGraph_t graph = nullptr;
  HIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  int r = 0;
  for (const auto &g : b->groups) {
    bool o = odd;
    for (int s = 0; s < ASLHIP_GRAPH_CHUNK && !r; ++s, o = !o) r = batch_launch(b, o, false, g);
  }
  hipError_t e = hipStreamEndCapture(b->stream, &graph);
  if (r) {
    if (graph) (void)hipGraphDestroy(graph);
    return r;
  }
  if (e != hipSuccess) return fail(ASLHIP_EHIP, "ASL ERROR: graph capture: %s", hipGetErrorString(e));
  e = hipGraphInstantiate(&g, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) return fail(ASLHIP_EHIP, "ASL ERROR: graph instantiate: %s", hipGetErrorString(e));
  return 0;
}

int batch_step_impl(aslhip_batch *b, int nsteps, unsigned flags) {
  if (nsteps < 0) return fail(ASLHIP_EINVAL, "ASL ERROR: negative step count");
  if (nsteps == 0) return 0;
  // Lattices fresh from initF take their first step on their own (it may
  // read ghost links raw); all of them then share one parity.
  bool any_fresh = false;
  for (auto *h : b->lat) {
    if (!h->initialized) return fail(ASLHIP_ESTATE, "ASL ERROR: batch lattice without initF");
    if (int r = flush_deferred(h)) return r;
    any_fresh = any_fresh || h->fresh;
  }
  if (any_fresh) {
    for (auto *h : b->lat)
      if (int r = step_impl(h, 1, (nsteps == 1 && (flags & ASLHIP_STEP_WRITE_MACRO)) ? ASLHIP_STEP_WRITE_MACRO : 0u,
                            nullptr))
        return r;
    if (--nsteps == 0) return 0;
  }
  const size_t n = b->lat.size();
  // the previous upload may still be in flight from this buffer
  HIPCHK(hipStreamSynchronize(b->stream));
  std::vector<StepArgs> &desc = b->hdesc;
  desc.resize(4 * n);
  const bool odd = b->lat[0]->next_odd;
  // Whole graph chunks go group by group, and so do the steps left; fewer than
  // BATCH_GROUP_STEPS in one launch each for all lattices.
  const bool macro = (flags & ASLHIP_STEP_WRITE_MACRO) != 0;
  const int chunks = flags & ASLHIP_STEP_GRAPH ? (nsteps - (macro ? 1 : 0)) / ASLHIP_GRAPH_CHUNK : 0;
  const int left = nsteps - chunks * ASLHIP_GRAPH_CHUNK;
  const bool at_once = left < BATCH_GROUP_STEPS && b->groups.size() > 1;
  const int k0 = chunks || !at_once ? 0 : 1, k1 = at_once ? 1 : 0;  // the descriptions needed
  for (size_t l = 0; l < n; ++l) {
    aslhip_lattice *h = b->lat[l];
    if (int r = prepare(h, false)) return r;
    if (h->nvl) return fail(ASLHIP_EINVAL, "ASL ERROR: velocity map BCs are not supported in batches");
    if (h->has_closure || h->turbulence)
      return fail(ASLHIP_EINVAL, "ASL ERROR: per-cell relaxation (closure, turbulence) is not supported in batches");
    if (h->next_odd != odd) return fail(ASLHIP_ESTATE, "ASL ERROR: batch lattices are at different step parities");
    if (int r = order_after_consumer(h)) return r;
    for (int k = k0; k <= k1; ++k) {
      StepArgs &plain = desc[2 * k * n + l], &writing = desc[(2 * k + 1) * n + l];
      plain = batch_args(b, h, k ? b->all.tile : b->tile[l] != 0);
      writing = plain;
      if (h->comp_rho) writing.g.flags |= STEP_F_RHO;
      if (h->comp_vel) writing.g.flags |= STEP_F_VEL;
    }
    // work queued on the lattice's own stream comes first
    HIPCHK(hipEventRecord(b->done, h->stream));
    HIPCHK(hipStreamWaitEvent(b->stream, b->done, 0));
  }
  HIPCHK(hipMemcpyAsync(b->desc + 2 * k0 * n, desc.data() + 2 * k0 * n, 2 * (k1 - k0 + 1) * n * sizeof(StepArgs),
                        hipMemcpyHostToDevice, b->stream));
  for (int c = 0; c < chunks; ++c) {  // an even number of steps each: the parity is unchanged
    if (int r = batch_graph(b, odd)) return r;
    HIPCHK(hipGraphLaunch(b->graph[odd ? 1 : 0], b->stream));
  }
  const std::vector<aslhip_batch::Range> one = {b->all};
  for (const auto &g : at_once ? one : b->groups)
    for (int s = 0; s < left; ++s)
      if (int r = batch_launch(b, odd != ((s & 1) != 0), macro && s == left - 1, g)) return r;
  for (auto *h : b->lat) h->next_odd = (nsteps % 2) ? !odd : odd;
  // the lattices' own streams see the result in order
  HIPCHK(hipEventRecord(b->done, b->stream));
  for (auto *h : b->lat) HIPCHK(hipStreamWaitEvent(h->stream, b->done, 0));
  return 0;
}

}  // namespace

extern "C" {

int aslhip_batch_create(aslhip_batch **out, aslhip_lattice *const *lattices, int n) {
  if (!out || !lattices || n < 1) return fail(ASLHIP_EINVAL, "ASL ERROR: batch needs at least one lattice");
  *out = nullptr;
  if (n > 65535) return fail(ASLHIP_EINVAL, "ASL ERROR: at most 65535 lattices per batch");
  aslhip_batch *b = new aslhip_batch();
  b->lat.assign(lattices, lattices + n);
  b->Q = lattices[0]->Q;
  b->dtype = lattices[0]->dtype;
  b->periodic = lattices[0]->periodic;
  b->wide = is_wide(lattices[0]);
  // D3Q27 in FP64 (see step_lanes), 512 -> 256 lanes: 10 lattices of 40^3..70^3 in
  // groups 160 -> 153 us per step, 12 of 24^3 18.1 -> 16.3
  long long largest = 0;
  for (int l = 0; l < n; ++l)
    if (lattices[l]) largest = std::max(largest, lattices[l]->qs_bytes * lattices[l]->Q);
  if (step_block(b->Q, static_cast<int>(lattices[0]->selem)) < STEP_BLOCK && largest <= TALL_BYTES) b->block = 256;
  for (int l = 0; l < n; ++l) {
    aslhip_lattice *h = lattices[l];
    if (!h || h->Q != b->Q || h->dtype != b->dtype || h->periodic != b->periodic || is_wide(h) != b->wide) {
      delete b;
      return fail(ASLHIP_EINVAL, "ASL ERROR: batch lattices must share template, population type and periodicity");
    }
  }
  hipError_t e = hipStreamCreate(&b->stream);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&b->done, hipEventDisableTiming);
  if (e == hipSuccess) e = device_alloc(&b->desc, 4 * (size_t)n * sizeof(StepArgs));
  if (e != hipSuccess) {
    batch_free(b);
    delete b;
    return fail(ASLHIP_EHIP, "ASL ERROR: batch set-up: %s", hipGetErrorString(e));
  }
  if (int r = batch_tables(b)) {
    batch_free(b);
    delete b;
    return r;
  }
  *out = b;
  return 0;
}

int aslhip_batch_set_tuning(aslhip_batch *b, int knob, int value) {
  if (!b) return fail(ASLHIP_EINVAL, "ASL ERROR: null batch handle");
  int *setting = nullptr;
  if (knob == ASLHIP_TUNE_GROUP_MB) {
    if (value < 0 || value > (1 << 20)) return fail(ASLHIP_EINVAL, "ASL ERROR: group size %d MiB out of 0..2^20", value);
    setting = &b->group_mb;
  } else if (knob == ASLHIP_TUNE_LDS) {
    if (value != 0 && value != 1) return fail(ASLHIP_EINVAL, "ASL ERROR: batches take ASLHIP_TUNE_LDS 0 or 1");
    setting = &b->tune_lds;
  } else if (knob == ASLHIP_TUNE_BLOCK) {
    if (value < 64 || value > STEP_BLOCK || value % 64)
      return fail(ASLHIP_EINVAL, "ASL ERROR: workgroup size %d is not a multiple of 64 in 64..%d", value, STEP_BLOCK);
    setting = &b->block;
  } else {
    return fail(ASLHIP_EINVAL, "ASL ERROR: batches tune the workgroup size, the tiles and the group size only");
  }
  return batch_set(b, setting, value);
}

int aslhip_batch_autotune(aslhip_batch *b, int nsteps, int *best_block) {
  if (!b) return fail(ASLHIP_EINVAL, "ASL ERROR: null batch handle");
  if (nsteps < 1) return fail(ASLHIP_EINVAL, "ASL ERROR: autotune needs at least one step per candidate");
  nsteps += nsteps & 1;
  double best = 1e300;
  int bb = b->block, bl = b->tune_lds;
  auto trial = [&](int lds, int blk) -> int {
    if (int r = batch_set(b, &b->tune_lds, lds)) return r;
    if (int r = batch_set(b, &b->block, blk)) return r;
    double ms = 0.;
    if (int r = aslhip_batch_time_steps(b, nsteps, 0u, &ms)) return r;
    if (ms < best) {
      best = ms;
      bb = blk;
      bl = lds;
    }
    return 0;
  };
  if (!b->periodic && !b->wide)
    if (int r = trial(1, b->block)) return r;  // tiles: fixed workgroup
  for (int blk : {256, 512, 1024})
    if (int r = trial(-1, blk)) return r;  // tiles for groups that stream from HBM only
  if (int r = batch_set(b, &b->tune_lds, bl)) return r;
  if (int r = batch_set(b, &b->block, bb)) return r;
  if (best_block) *best_block = bl == 1 ? STEP_TILE : std::min(bb, step_block(b->Q, static_cast<int>(b->lat[0]->selem)));
  return 0;
}

int aslhip_batch_autotune_groups(aslhip_batch *b, int chunks, int *best_mb) {
  if (!b) return fail(ASLHIP_EINVAL, "ASL ERROR: null batch handle");
  if (chunks < 1) return fail(ASLHIP_EINVAL, "ASL ERROR: autotune needs at least one chunk per candidate");
  double best = 1e300;
  int bm = static_cast<int>(batch_group_bytes(b) >> 20);
  for (int mb : {0, 64, 128, 160, 192, 224, 256, 384}) {
    if (int r = aslhip_batch_set_tuning(b, ASLHIP_TUNE_GROUP_MB, mb)) return r;
    // the first chunk captures the graphs; the timed ones replay them
    if (int r = batch_step_impl(b, ASLHIP_GRAPH_CHUNK, ASLHIP_STEP_GRAPH)) return r;
    double ms = 0.;
    if (int r = aslhip_batch_time_steps(b, chunks * ASLHIP_GRAPH_CHUNK, ASLHIP_STEP_GRAPH, &ms)) return r;
    if (ms < best) {
      best = ms;
      bm = mb;
    }
  }
  if (int r = aslhip_batch_set_tuning(b, ASLHIP_TUNE_GROUP_MB, bm)) return r;
  if (best_mb) *best_mb = bm;
  return 0;
}

int aslhip_batch_destroy(aslhip_batch *b) {
  if (!b) return 0;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  batch_free(b);
  delete b;
  return 0;
}

int aslhip_batch_step(aslhip_batch *b, int nsteps, unsigned flags) {
  if (!b) return fail(ASLHIP_EINVAL, "ASL ERROR: null batch handle");
  return batch_step_impl(b, nsteps, flags);
}

int aslhip_batch_time_steps(aslhip_batch *b, int nsteps, unsigned flags, double *ms_total) {
  if (!b) return fail(ASLHIP_EINVAL, "ASL ERROR: null batch handle");
  hipEvent_t t0, t1;
  HIPCHK(hipEventCreate(&t0));
  HIPCHK(hipEventCreate(&t1));
  // start from an idle batch stream (previous work of the lattices included)
  for (auto *h : b->lat) {
    HIPCHK(hipEventRecord(b->done, h->stream));
    HIPCHK(hipStreamWaitEvent(b->stream, b->done, 0));
  }
  HIPCHK(hipEventRecord(t0, b->stream));
  int r = batch_step_impl(b, nsteps, flags);
  HIPCHK(hipEventRecord(t1, b->stream));
  HIPCHK(hipEventSynchronize(t1));
  float ms = 0.f;
  if (r == 0) HIPCHK(hipEventElapsedTime(&ms, t0, t1));
  if (ms_total) *ms_total = ms;
  (void)hipEventDestroy(t0);
  (void)hipEventDestroy(t1);
  return r;
}

}  // extern "C"
