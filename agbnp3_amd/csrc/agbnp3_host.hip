// Host side of libagbnp3: the agbnp3.h C API (instance registry, agbnp3_new /
// agbnp3_ener / agbnp3_delete), the Q4 spline tables, the static water-site
// topology, packs (the device arena of one or more systems, their work
// items and launch shapes), the per-call kernel pipeline on one stream,
// batches of instances with hipGraph replay, and the launch-shape autotuner.
#include <float.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <random>
#include <string>
#include <type_traits>
#include <vector>

#include "agb_common.h"
#include "agbnp3.h"
#include "agbnp3_amd.h"

using namespace agb;

// Per-call working state of agbnp3_ener_static: one array on every device the
// library runs on, held until the process ends.  Host code never uses this
// name as an address (it is a host-side stand-in): the device address comes
// from hipGetSymbolAddress, once per device (scratch_base).
static __device__ __align__(256) char scratch[AGBNP3_STATIC_SCRATCH_BYTES];

namespace {

void errprint(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vfprintf(stderr, fmt, ap);
  va_end(ap);
}

#define HIPCHK(expr)                                                                   \
  do {                                                                                 \
    hipError_t e_ = (expr);                                                            \
    if (e_ != hipSuccess) {                                                            \
      errprint("agbnp3: HIP error %s at %s:%d: %s\n", hipGetErrorString(e_), __FILE__, \
               __LINE__, #expr);                                                       \
      return AGBNP_ERR;                                                                \
    }                                                                                  \
  } while (0)

// ------------------------------------------------------------ Q4 tables
// The tables are model data; they are built with the reference's own mixed
// float/double arithmetic so every node is the reference's FP32 value:
// agbnp3_i4 (agbnp3.c:3886-3944), agbnp3_i4ov (agbnp3.c:3964-3975, both
// Gaussian exponents taken from Ri), agbnp3_create_ctablef4
// (agbnp3_utils.c:380-422: 511 nodes on [0, 20) at an accumulated spacing,
// y[511] = 0) and agbnp3_cspline_setup (agbnp3_utils.c:193-227, whose end
// condition divides by 2 dx).  The reference is C, where log/exp/pow of a
// float promote to double; the explicit casts keep that under C++ overloads.
float q4_integral(float rij, float Ri, float Rj, float *dr) {
  const float twopi = 2.0 * kPi;
  const float twothirds = 2.0 / 3.0;
  const float rij2 = rij * rij;
  float q;
  if (rij > (Ri + Rj)) {                         // no overlap
    float u1 = rij + Rj, u2 = rij - Rj, u3 = u1 * u2;
    float u4 = 0.5 * log((double)(u1 / u2));
    q = twopi * (Rj / u3 - u4 / rij);
    *dr = twopi * ((Rj / (rij * u3)) * (1. - 2. * rij2 / u3) + u4 / rij2);
    return q;
  }
  float u1 = Rj - Ri;
  if (rij2 > u1 * u1) {                          // partial overlap
    u1 = rij + Rj;
    float u2 = rij - Rj, u3 = u1 * u2;
    float u4 = 1. / u1, u4sq = u4 * u4;
    float u5 = 1. / Ri, u5sq = u5 * u5;
    float u6 = 0.5 * log((double)(u1 / Ri));
    q = twopi * (-(u4 - u5) + (0.25 * u3 * (u4sq - u5sq) - u6) / rij);
    *dr = twopi * (0.5 * (1. - 0.5 * u3 / rij2) * (u4sq - u5sq) + u6 / rij2);
    return q;
  }
  if (Ri > Rj) {                                 // i contains j
    *dr = 0.0f;
    return 0.0f;
  }
  u1 = rij + Rj;                                 // j contains i
  float u2 = Rj - rij, u3 = -u1 * u2;
  if (rij < .001 * Rj) {                         // series at the centre
    float a = rij / Rj, ad = a * a - 1;
    float u6 = (1. + twothirds * a * a) / Rj;
    q = twopi * (2. / Ri + Rj / u3 - u6);
    *dr = -(2. * twopi * a / (Rj * Rj)) * (1. / ad + twothirds);
  } else {
    float u6 = 0.5 * log((double)(u1 / u2));
    q = twopi * (2. / Ri + Rj / u3 - u6 / (rij));
    *dr = twopi * (-(Rj / u3) * (2. * rij / u3 - 1. / (rij)) + u6 / (rij2));
  }
  return q;
}

float q4_inflated(float rij, float Ri, float Rj, float *dr) {
  const float ai = kKFC / (Ri * Ri);
  const float pfc = kPFC;
  const float d2 = rij * rij;
  const float deltai = 1. / (ai + ai);
  const float p = pfc * pfc;
  const float kappa = exp((double)(-ai * ai * d2 * deltai));
  const float gvol = p * kappa * pow(kPi * deltai, 1.5);
  const float volj = 4. * kPi * Rj * Rj * Rj / 3.;
  const float newRj = pow((volj + 2. * gvol) / volj, 1. / 3.) * Rj;
  return q4_integral(rij, Ri, newRj, dr);
}

void spline_coeffs(float dx, int n, const float *y, float yp1, float ypn, float *y2) {
  std::vector<float> u(n);
  y2[0] = -0.5;
  u[0] = (3.0 / (dx)) * ((y[1] - y[0]) / (dx)-yp1);
  for (int i = 1; i < n - 1; i++) {
    const float sig = 0.5;
    const float p = sig * y2[i - 1] + 2.0;
    y2[i] = (sig - 1.0) / p;
    u[i] = (y[i + 1] - y[i]) / (dx) - (y[i] - y[i - 1]) / (dx);
    u[i] = (6.0 * u[i] / (2. * dx) - sig * u[i - 1]) / p;
  }
  const float qn = 0.5;
  const float un = (3.0 / (dx)) * (ypn - (y[n - 1] - y[n - 2]) / (2. * dx));
  y2[n - 1] = (un - qn * u[n - 2]) / (qn * y2[n - 2] + 1.0);
  for (int k = n - 2; k >= 0; k--) y2[k] = y2[k] * y2[k + 1] + u[k];
}

void build_table(float b, float *y, float *y2, float &dx, float &dxinv) {
  const int n = kTblN;
  const float amax = kTblAmax;
  const float da = amax / (n - 1);
  float a = 0.0f, dr = 0.0f, yp1 = 0.0f;
  for (int i = 0; i < n - 1; i++) {
    const float q = q4_inflated(a, b, 1.0f, &dr);
    if (i == 0) yp1 = dr;
    y[i] = q;
    a += da;
  }
  y[n - 1] = 0.0f;
  spline_coeffs(da, n, y, yp1, 0.0f, y2);
  dx = da;
  dxinv = 1. / da;
}

// The tables as per-interval cubics in the fraction u of the interval (the
// chain-rule kernel evaluates the value with 3 FMAs and derives the
// derivative from the same four numbers).  From the FP32 nodes y, y'' in
// FP64, with the spacing dx and dp2 = dx^2/6 in FP64 from the FP32 dx (as
// the FP64 oracle interpolates), then rounded once:
//   value (agbnp3_utils.c:266-295):  A y0 + u y1 + ((A^3 - A) z0 + (u^3 - u) z1) dp2, A = 1 - u
//     = c0 + c1 u + c2 u^2 + c3 u^3,  c0 = y0, c1 = y1 - y0 - dp2 (2 z0 + z1),
//       c2 = 3 dp2 z0, c3 = dp2 (z1 - z0).
// Interval 511 (past the last node) is zero.  Layout [ntab][512] float4.
void chain_tables(const std::vector<float> &ty, const std::vector<float> &ty2, int ntab, float tdx,
                  std::vector<float4> &out) {
  const double dx = tdx, dp2 = dx * (dx / 6.0);
  out.assign((size_t)ntab * kTblN, make_float4(0.f, 0.f, 0.f, 0.f));
  for (int t = 0; t < ntab; t++)
    for (int k = 0; k + 1 < kTblN; k++) {
      const size_t n = (size_t)t * kTblN + k;
      const double y0 = ty[n], y1 = ty[n + 1], z0 = ty2[n], z1 = ty2[n + 1];
      out[n] = make_float4((float)y0, (float)(y1 - y0 - dp2 * (2.0 * z0 + z1)), (float)(3.0 * dp2 * z0),
                           (float)(dp2 * (z1 - z0)));
    }
}

// ------------------------------------------------------------- model
// Host copy of one system's parameters, in internal order (heavy atoms first)
struct Model {
  int natoms = 0, nheavy = 0;
  int verbose = 0;
  int ws_error_atom = -1;              // TRIGONAL_OOP topology error (reported by ener)
  std::vector<int> int2ext, ext2int;
  std::vector<float> R, q, igamma, sgamma, ialpha, salpha, hbcorr, galpha;
  std::vector<int> hbtype, rtype;
  std::vector<double> vols;
  std::vector<int> cnne, coff, cnl;    // connection table, internal indices
  int ntypes = 0;
  std::vector<float> radii, ty, ty2;
  float tdx = 0, tdxinv = 0;
  float eps_in = 1, eps_out = 1;
  std::vector<WsDef> wsdef;
  std::vector<int> ws_stale0;          // per site; -1: no atom (spe 0)
  int nws = 0;
  // place of each atom along a space-filling curve through the coordinates
  // the instance was created with
  std::vector<unsigned> curve;
  float extent = 0;                    // longest edge of their box
};

// ------------------------------------------------------------- pack
// Device arena, work items and launch shapes of one or more systems that
// are evaluated together.
struct Pack {
  unsigned long long uid = 0;          // distinct for every pack built in the process
  int n = 0, nh = 0, nsys = 0, ntypes = 0;
  int options = 0;
  int cap = 128;                       // neighbour-list row capacity (64, 128, 256)
  float skin = 0.f;                    // neighbour-list reuse (0: rebuild every call)
  int reuse_every = 0;
  Tuning tune;
  std::vector<float> radii;            // radius types (union over the systems)
  std::vector<SysInfo> sinfo;
  std::vector<int> rtype;              // per atom
  std::vector<char> heavy;             // per atom
  std::vector<float> alpha_sum;        // per atom: ialpha + salpha
  std::vector<unsigned> curve;         // per atom: Model::curve
  hipStream_t stream = nullptr;
  // second stream (fork and join events, also inside a captured graph): in
  // large calls the water-site kernels, which need only the self volumes, run
  // there beside the descreening and pair kernels; later one tier of the
  // derivative pass beside the other
  hipStream_t side = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr, ev_fork2 = nullptr, ev_join2 = nullptr;
  std::vector<void *> allocs, item_allocs;
  Dev d{};
  int device = 0;                      // the device the pack lives on
  int ntile = 0;                       // GB tile-pair energy slots of all systems
  bool dt = false;                     // descreening by tiles (unless a surrogate is attached)
  long long ndpart = 0;                // its tile sums
  size_t call_ndpart() const { return dt ? (size_t)ndpart : 0; }
  bool split = false;                  // chain rule by row groups (unless a surrogate is attached)
  size_t call_nsplit() const { return split ? (size_t)d.nchain_items * kSplitSets * 2048 : 0; }
  // per-call working state (carve_call_state) and the host-API staging,
  // allocated by the first call that needs them (ensure_call_state), so an
  // instance evaluated only through agbnp3_ener_static never holds them
  void *call_block = nullptr;
  int call_nchain = 0;                 // chain-rule items the block's partial sums hold
  size_t call_split = 0;               // numbers of their sums by row groups
  size_t call_dpart = 0;               // descreening tile sums it holds
  double *dout = nullptr;                                  // outputs: 15n + 7 nsys
  // pinned host staging, which the first and last kernels of a host-API call
  // read and write themselves: outputs, coordinates, status and counters (5)
  double *hstage = nullptr;
  unsigned long long *hstat = nullptr; // pinned: status word and counters 0..3 of the last call
  std::vector<void *> pinned;          // what the two lie in
  bool host_status = false;            // the last call put its status there
  int routes = 0;                      // agbnp3_get_routes
  // timing mode: one event set per recorded call, averaged when read back
  std::vector<std::vector<hipEvent_t>> ev_sets;
  std::vector<std::string> ev_names;
  int ncalls_timed = 0;
  // captured pipeline and the device pointers it was captured with
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  const double *cap_in[3] = {nullptr, nullptr, nullptr};
  double *cap_out[8] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  // surrogate buffers (allocated on first attach)
  std::vector<void *> sg_allocs;
  int sg_model = -1;
};

// ------------------------------------------------------------ surrogate
// A trained (or training) Born-radius model: FP32 master parameters, Adam
// state, the bf16 copies the kernels read, the normalisation and the
// training window, and a training set on the device.
struct SgHost {
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr, *loss = nullptr;
  unsigned short *w1 = nullptr, *w2 = nullptr, *w3 = nullptr, *wt1 = nullptr, *wt2 = nullptr, *wt3 = nullptr;
  float *norm = nullptr;          // xmu, xsd_inv, xlo, xhi [4][kSgNFeat]
  float ymu = 0.f, ysd = 1.f;
  int step = 0;
  // training set
  int cap = 0, count = 0;
  float *F = nullptr, *target = nullptr;          // raw [cap][66], [cap]
  std::vector<unsigned long long> keys;           // per row: (pack uid << 32) | atom of the pack
  float *X = nullptr;                             // training rows, normalised [ntrain][96]
  float *y = nullptr;                             // normalised targets [ntrain]
  std::vector<int> order;                         // dataset row of each training row
  int ntrain = 0;
  float w_abs = 1.f, w_diff = 1.f;                // loss weights (w_diff per pair-difference variance)
  float dscale = 0.f;                             // 1 / mean squared normalised pair difference
  int bcap = 0;
  SgTrain tb{};
  std::vector<void *> allocs, tallocs;
  hipStream_t stream = nullptr;
  SgModel view() const {
    SgModel v{};
    v.w1 = w1; v.w2 = w2; v.w3 = w3; v.wt1 = wt1; v.wt2 = wt2; v.wt3 = wt3;
    v.b1 = p + kSgOffB1; v.b2 = p + kSgOffB2; v.b3 = p + kSgOffB3; v.w4 = p + kSgOffW4; v.b4 = p + kSgOffB4;
    v.xmu = norm; v.xsd_inv = norm + kSgNFeat; v.xlo = norm + 2 * kSgNFeat; v.xhi = norm + 3 * kSgNFeat;
    v.ymu = ymu;
    v.ysd = ysd;
    return v;
  }
};
std::vector<SgHost *> g_models;

void sg_free(SgHost *M) {
  if (M->stream) (void)hipStreamSynchronize(M->stream);
  for (void *q : M->allocs) (void)hipFree(q);
  for (void *q : M->tallocs) (void)hipFree(q);
  if (M->F) (void)hipFree(M->F);
  if (M->target) (void)hipFree(M->target);
  if (M->stream) (void)hipStreamDestroy(M->stream);
  delete M;
}

struct Instance {
  Model m;
  Pack p;
};

struct Batch {
  std::vector<int> tags;
  std::vector<int> ws_error;           // external atom of a TRIGONAL_OOP error per system, or -1
  Pack p;
};

std::mutex g_mutex;
bool g_initialized = false;

// device address of `scratch` per device (hipGetSymbolAddress with that
// device current), resolved by agbnp3_initialize for the current device and
// by the first agbnp3_ener_static call on any other
constexpr int kMaxDevices = 64;
char *g_scratch[kMaxDevices] = {};
std::mutex g_scratch_mutex;

int scratch_base(int dev, char **base) {
  if (dev < 0 || dev >= kMaxDevices) {
    errprint("agbnp3: device %d out of range\n", dev);
    return AGBNP_ERR;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mutex);
  if (!g_scratch[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      errprint("agbnp3: no address for the static scratch on device %d: %s\n", dev, hipGetErrorString(e));
      return AGBNP_ERR;
    }
    g_scratch[dev] = static_cast<char *>(ptr);
  }
  *base = g_scratch[dev];
  return AGBNP_OK;
}
std::vector<Instance *> g_slots;
std::vector<Batch *> g_batches;

Instance *get_instance(int tag, const char *who) {
  if (!g_initialized) {
    errprint("%s: agbnp library is not initialized.\n", who);
    return nullptr;
  }
  if (tag < 0 || tag >= (int)g_slots.size() || !g_slots[tag]) {
    errprint("%s: invalid tag %d.\n", who, tag);
    return nullptr;
  }
  return g_slots[tag];
}

Batch *get_batch(int id, const char *who) {
  if (!g_initialized) {
    errprint("%s: agbnp library is not initialized.\n", who);
    return nullptr;
  }
  if (id < 0 || id >= (int)g_batches.size() || !g_batches[id]) {
    errprint("%s: invalid batch %d.\n", who, id);
    return nullptr;
  }
  return g_batches[id];
}

// device allocation helpers: 0 on success, non-zero on failure
template <typename T>
int dalloc(std::vector<void *> &list, T **p, size_t count) {
  void *q = nullptr;
  if (count == 0) count = 1;
  hipError_t e = hipMalloc(&q, count * sizeof(T));
  if (e != hipSuccess) {
    errprint("agbnp3: device allocation of %zu bytes failed: %s\n", count * sizeof(T), hipGetErrorString(e));
    return 1;
  }
  list.push_back(q);
  *p = (T *)q;
  return 0;
}

template <typename T>
int upload(std::vector<void *> &list, const T **dst, const std::vector<T> &src) {
  T *p = nullptr;
  if (dalloc(list, &p, src.size())) return 1;
  if (!src.empty() && hipMemcpy(p, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess) {
    errprint("agbnp3: upload of %zu bytes failed\n", src.size() * sizeof(T));
    return 1;
  }
  *dst = p;
  return 0;
}

void drop_graph(Pack &P) {
  if (P.gexec) (void)hipGraphExecDestroy(P.gexec);
  if (P.graph) (void)hipGraphDestroy(P.graph);
  P.gexec = nullptr;
  P.graph = nullptr;
}

void free_pack(Pack &P) {
  if (P.stream) (void)hipStreamSynchronize(P.stream);
  drop_graph(P);
  for (void *p : P.allocs) (void)hipFree(p);
  for (void *p : P.item_allocs) (void)hipFree(p);
  for (void *p : P.sg_allocs) (void)hipFree(p);
  if (P.call_block) (void)hipFree(P.call_block);
  P.call_block = nullptr;
  P.allocs.clear();
  P.item_allocs.clear();
  P.sg_allocs.clear();
  for (void *p : P.pinned) (void)hipHostFree(p);
  P.pinned.clear();
  P.hstage = nullptr;
  P.hstat = nullptr;
  for (auto &set : P.ev_sets)
    for (hipEvent_t e : set) (void)hipEventDestroy(e);
  P.ev_sets.clear();
  if (P.stream) (void)hipStreamDestroy(P.stream);
  P.stream = nullptr;
  if (P.side) (void)hipStreamDestroy(P.side);
  P.side = nullptr;
  for (hipEvent_t e : {P.ev_fork, P.ev_join, P.ev_fork2, P.ev_join2})
    if (e) (void)hipEventDestroy(e);
  P.ev_fork = P.ev_join = P.ev_fork2 = P.ev_join2 = nullptr;
}

// static water-site topology: geometry per HB-active atom, following the
// dispatch of agbnp3_create_ws_ofatom (agbnp3.c:1920-2012); atoms whose
// topology does not fit get no sites, as in the reference
void build_water_sites(Model *I) {
  const int n = I->natoms, nh = I->nheavy;
  I->wsdef.clear();
  I->ws_stale0.clear();
  I->ws_error_atom = -1;
  int nsite = 0;
  auto nb = [&](int a, int k) { return I->cnl[I->coff[a] + k]; };
  for (int a = 0; a < n; a++) {
    const int t = I->hbtype[a], m = I->cnne[a];
    WsDef w{};
    w.atom = a;
    w.p[0] = a;
    int ns = 0;
    if (t == AGBNP_HB_POLARH) {
      int dd = -1;
      for (int k = 0; k < m; k++)
        if (nb(a, k) < nh) { dd = nb(a, k); break; }
      if (dd >= 0) { w.kind = WS_POLARH; w.p[1] = dd; ns = 1; }
    } else if (t == AGBNP_HB_TRIGONAL && m == 2) {
      w.kind = WS_TRIGONAL2; w.p[1] = nb(a, 0); w.p[2] = nb(a, 1); ns = 1;
    } else if ((t == AGBNP_HB_TRIGONAL || t == AGBNP_HB_TRIGONAL_S) && m == 1) {
      const int r = nb(a, 0);
      if (I->cnne[r] == 3) {
        int r1 = -1, r2 = -1;
        for (int k = 0; k < 3; k++) {
          const int c = nb(r, k);
          if (c == a) continue;
          if (r1 < 0) r1 = c;
          else if (r2 < 0 && c != r1) r2 = c;
        }
        if (r1 >= 0 && r2 >= 0) {
          w.kind = t == AGBNP_HB_TRIGONAL ? WS_TRIGONAL1 : WS_TRIGONAL_S;
          w.p[1] = r; w.p[2] = r1; w.p[3] = r2;
          ns = t == AGBNP_HB_TRIGONAL ? 2 : 4;
        }
      }
    } else if (t == AGBNP_HB_TRIGONAL_OOP) {
      if (m != 3) {
        if (I->ws_error_atom < 0) I->ws_error_atom = a;
      } else {
        w.kind = WS_TRIGONAL_OOP; w.p[1] = nb(a, 0); w.p[2] = nb(a, 1); w.p[3] = nb(a, 2); ns = 2;
      }
    } else if (t == AGBNP_HB_TETRAHEDRAL) {
      if (m == 2) {
        w.kind = WS_TETRAHEDRAL2; w.p[1] = nb(a, 0); w.p[2] = nb(a, 1); ns = 2;
      } else if (m == 3) {
        w.kind = WS_TETRAHEDRAL3; w.p[1] = nb(a, 0); w.p[2] = nb(a, 1); w.p[3] = nb(a, 2); ns = 1;
      } else if (m == 1) {
        const int r = nb(a, 0);
        if (I->cnne[r] == 4) {
          int c = 0;
          w.p[1] = r;
          for (int k = 0; k < 4 && c < 3; k++)
            if (nb(r, k) != a) w.p[2 + c++] = nb(r, k);
          if (c == 3) { w.kind = WS_TETRAHEDRAL1; ns = 3; }
        }
      }
    }
    if (ns == 0) continue;
    w.nsite = ns;
    w.first = nsite;
    I->wsdef.push_back(w);
    // last parent of each site: the stale index the next site starts from
    for (int s = 0; s < ns; s++) {
      int last;
      switch (w.kind) {
        case WS_POLARH: last = w.p[1]; break;
        case WS_TRIGONAL1: case WS_TRIGONAL_S: case WS_TRIGONAL_OOP: case WS_TETRAHEDRAL3: last = w.p[3]; break;
        case WS_TRIGONAL2: case WS_TETRAHEDRAL2: last = w.p[2]; break;
        default: last = w.p[2 + s]; break;      // tetrahedral1: (A, R, R_k)
      }
      I->ws_stale0.push_back(last);
    }
    nsite += ns;
  }
  // site s reads the last parent of site s-1 first; site 0 the index after
  // the heavy atoms (a hydrogen, spe = 0)
  std::vector<int> st(nsite);
  for (int s = 0; s < nsite; s++) st[s] = s == 0 ? (nh < n ? nh : -1) : I->ws_stale0[s - 1];
  I->ws_stale0 = st;
  I->nws = nsite;
}

// --------------------------------------------------------- work items
// Row blocks of one radius type and one system; descreening / chain items
// (row block x column range) and GB tile pairs, each list sorted by
// decreasing size so persistent blocks take the large items first.
int build_items(Pack &P) {
  for (void *p : P.item_allocs) (void)hipFree(p);
  P.item_allocs.clear();
  drop_graph(P);
  Dev &d = P.d;
  const int rows = P.tune.rows;
  std::vector<int> row_perm;
  std::vector<int4> rblk;
  for (int b = 0; b < P.nsys; b++) {
    const SysInfo &S = P.sinfo[b];
    for (int t = 0; t < P.ntypes; t++) {
      std::vector<int> r;
      for (int i = S.a0; i < S.a0 + S.n; i++)
        if (P.rtype[i] == t) r.push_back(i);
      // (a row's sum does not depend on the rows beside it: rows close in
      // space share a wave, so that it can pass over far columns)
      std::stable_sort(r.begin(), r.end(), [&](int a, int b) { return P.curve[a] < P.curve[b]; });
      for (size_t k = 0; k < r.size(); k += rows) {
        int allh = 1;
        for (int q = 0; q < rows; q++) {
          const int a = k + q < r.size() ? r[k + q] : -1;
          row_perm.push_back(a);
          if (a >= 0 && P.heavy[a]) allh = 0;
        }
        rblk.push_back(make_int4(t, b, allh, 0));
      }
    }
  }
  // column ranges
  auto chunked = [&](int chunk_param, bool chain) {
    std::vector<int4> items;
    double total = 0.0;
    for (size_t k = 0; k < rblk.size(); k++) {
      const SysInfo &S = P.sinfo[rblk[k].y];
      total += (double)rows * (chain ? (rblk[k].z ? S.nh : S.n) : S.nh);
    }
    int L = chunk_param;
    if (L <= 0) {       // about 2048 items in all, 512 to 2048 columns each
      // (the cap keeps an item short enough that a call needing a few row
      // blocks -- a surrogate call with out-of-range atoms -- spreads them
      // over many CUs)
      L = (int)std::ceil(total / (2048.0 * rows) / 256.0) * 256;
      L = std::min(std::max(L, 512), 2048);
    }
    for (size_t k = 0; k < rblk.size(); k++) {
      const SysInfo &S = P.sinfo[rblk[k].y];
      const int c0 = S.a0, c1 = S.a0 + (chain ? (rblk[k].z ? S.nh : S.n) : S.nh);
      for (int c = c0; c < c1; c += L) items.push_back(make_int4((int)k, c, std::min(c1, c + L), 0));
    }
    std::stable_sort(items.begin(), items.end(), [](const int4 &a, const int4 &b) { return a.z - a.y > b.z - b.y; });
    return std::make_pair(items, L);
  };
  const auto [desc, desc_cols] = chunked(P.tune.desc_chunk, false);
  // the same by tiles (k_desc_sites), where these fill the chip a few times
  // at most and the tables of every type fit in LDS
  std::vector<int4> dt;
  for (int k = 0; k < (int)rblk.size() && (int)dt.size() <= kDtItems; k++) {
    const SysInfo &S = P.sinfo[rblk[k].y];
    for (int c = 0, t = 0; c < S.nh; c += 256, t++)
      dt.push_back(make_int4(k, S.a0 + c, S.a0 + std::min(S.nh, c + 256), (int)(S.dp0 + (long long)t * S.n - S.a0)));
  }
  P.dt = P.tune.desc_chunk <= 0 && P.ntypes <= kLdsTypes && (int)dt.size() <= kDtItems;
  if (!P.dt) dt.clear();
  // chain rule: pairs (P <= Q) of 256-atom blocks of one radius type, inside
  // one system, not both hydrogen-only
  std::vector<int> cperm;
  std::vector<int4> cblk;
  std::vector<int> csize, novdw;    // novdw: every atom's ialpha + salpha is 0 (abrw = 0)
  std::vector<std::pair<int, int>> csys;             // first and end block of each system
  // types in order of radius: the blocks (and so which side of a tile pair an
  // atom is on) do not depend on how a pack numbers its radius types
  std::vector<int> by_radius(P.ntypes);
  for (int t = 0; t < P.ntypes; t++) by_radius[t] = t;
  std::stable_sort(by_radius.begin(), by_radius.end(), [&](int a, int b) { return P.radii[a] < P.radii[b]; });
  for (int b = 0; b < P.nsys; b++) {
    const SysInfo &S = P.sinfo[b];
    const int first = (int)cblk.size();
    for (int t : by_radius) {
      std::vector<int> r;
      for (int i = S.a0; i < S.a0 + S.n; i++)
        if (P.rtype[i] == t) r.push_back(i);
      for (size_t k = 0; k < r.size(); k += 256) {
        int allh = 1, allheavy = 1, cnt = 0, nv = 1;
        for (int q = 0; q < 256; q++) {
          const int a = k + q < r.size() ? r[k + q] : -1;
          cperm.push_back(a);
          if (a >= 0) {
            cnt++;
            if (P.heavy[a]) allh = 0; else allheavy = 0;
            if (P.alpha_sum[a] != 0.f) nv = 0;
          }
        }
        cblk.push_back(make_int4(t, b, allh, allheavy));
        csize.push_back(cnt);
        novdw.push_back(nv);
      }
    }
    csys.push_back({first, (int)cblk.size()});
  }
  // kinds (k_chain): both blocks heavy atoms only; hydrogen rows against heavy
  // columns (the hydrogen block is made the row block); anything else
  // (diagonal blocks, blocks mixing heavy atoms and hydrogens)
  std::vector<std::pair<int4, int>> cit;     // with its relative time
  for (const auto &fe : csys)
    for (int p = fe.first; p < fe.second; p++)
      for (int q = p; q < fe.second; q++) {
        if (cblk[p].z && cblk[q].z) continue;
        int4 it = make_int4(p, q, 0 /* general */, 0);
        if (p != q && cblk[p].w && cblk[q].w) it.z = 1;                          // heavy x heavy
        else if (p != q && cblk[p].z && cblk[q].w) it.z = 2;                     // hydrogens x heavy
        else if (p != q && cblk[p].w && cblk[q].z) it = make_int4(q, p, 2, 0);
        if (it.z == 2 && novdw[it.x]) it.z = 3;                                  // rows without vdW terms
        // columns in chunks of chain_chunk (64 or 128; 0: the whole block)
        const int step = P.tune.chain_chunk > 0 && P.tune.chain_chunk < 256 ? P.tune.chain_chunk / 64 : 4;
        const int ncol = csize[it.y], nch = (ncol + 63) / 64;
        // relative time of a pair by kind: general, heavy x heavy of two types or of one, hydrogen rows with and without vdW terms
        const int cost = it.z == 0 ? 9 : it.z == 1 ? (cblk[p].x == cblk[q].x ? 5 : 8) : (it.z == 2 ? 5 : 4);
        for (int c0 = 0; c0 < nch; c0 += step) {
          const int c1 = std::min(nch, c0 + step);
          int4 ci = it;
          ci.w = c0 | (c1 << 4);
          cit.push_back({ci, cost * (c1 - c0)});
        }
      }
  // longest first where the launch's end counts; in long launches only full
  // items before cut ones, so that those in flight together share their row blocks
  const bool by_time = cit.size() <= kChainByTime;
  std::stable_sort(cit.begin(), cit.end(), [&](const std::pair<int4, int> &a, const std::pair<int4, int> &b) {
    if (by_time) return a.second > b.second;
    return (a.first.w >> 4) - (a.first.w & 15) > (b.first.w >> 4) - (b.first.w & 15);
  });
  std::vector<int4> chain(cit.size());
  for (size_t k = 0; k < cit.size(); k++) chain[k] = cit[k].first;
  // the same by row groups, where the items are few and no shape was asked for
  // (whole blocks only: every chunk of an item's columns is then written)
  P.split = P.tune.chain_chunk == 0 && (int)chain.size() <= kSplitItems;
  std::vector<int> sub, sets;
  for (int k = 0; P.split && k < (int)chain.size(); k++) {
    const int4 &it = chain[k];
    const bool one_row = it.z == 0 || (it.z == 1 && cblk[it.x].x != cblk[it.y].x);     // rows per lane (k_chain)
    const int groups = (csize[it.x] + (one_row ? 63 : 127)) / (one_row ? 64 : 128), nch = it.w >> 4;
    const int parities = one_row || nch == 1 ? 1 : 2;
    for (int p = 0; p < parities; p++)
      for (int g = 0; g < groups; g++) sub.push_back(k << 2 | p << 1 | g);
    sets.push_back(groups | (parities == 2 ? 8 : 0));
  }
  // where each block's chain-rule sums are: (item, side) slots ordered by the
  // other block's place in its system, row side first, so that a batch member
  // adds its partial sums in the order its own instance does
  std::vector<std::vector<std::pair<long long, int>>> cl(cblk.size());
  std::vector<int> sys_first(P.nsys);
  for (int b = 0; b < P.nsys; b++) sys_first[b] = csys[b].first;
  for (size_t k = 0; k < chain.size(); k++) {
    const int r = chain[k].x, c = chain[k].y, c0 = chain[k].w & 15;
    const int f = sys_first[cblk[r].y];
    cl[r].push_back({((long long)(c - f) * 8 + c0) * 2, (int)k * 2});
    if (r != c) cl[c].push_back({((long long)(r - f) * 8 + c0) * 2 + 1, (int)k * 2 + 1});
  }
  // one list per summed quantity q (gb xyz, vdW xyz, U, V): hydrogen-row
  // items store only the quantities they can make nonzero (rows: gb, and vdW
  // when the rows have vdW terms; columns: all but the vdW ones and V when
  // they do not), so the lists leave out the (item, side) slots holding zeros
  auto stores = [&](int e, int q) {
    const int kind = chain[e >> 1].z, side = e & 1;
    if (kind == 3) return side == 0 ? q < 3 : (q < 3 || q == 6);
    if (kind == 2) return side == 0 ? q < 6 : true;
    return true;
  };
  const size_t nb1 = cblk.size() + 1;
  std::vector<int> ch_cstart(8 * nb1, 0), ch_contrib;
  for (size_t b = 0; b < cblk.size(); b++) std::sort(cl[b].begin(), cl[b].end());
  for (int q = 0; q < 8; q++) {
    for (size_t b = 0; b < cblk.size(); b++) {
      ch_cstart[q * nb1 + b] = (int)ch_contrib.size();
      for (const auto &e : cl[b])
        if (stores(e.second, q)) ch_contrib.push_back(e.second);
    }
    ch_cstart[q * nb1 + cblk.size()] = (int)ch_contrib.size();
  }
  // GB tile pairs of 256-atom tiles, I <= J
  std::vector<std::pair<int4, int>> gb;
  for (int b = 0; b < P.nsys; b++) {
    const SysInfo &S = P.sinfo[b];
    const int nb = (S.n + 255) / 256;
    int k = 0;
    for (int I = 0; I < nb; I++)
      for (int J = I; J < nb; J++, k++) {
        const int r0 = S.a0 + 256 * I, c0 = S.a0 + 256 * J;
        gb.push_back({make_int4(r0, std::min(S.a0 + S.n, r0 + 256), c0, std::min(S.a0 + S.n, c0 + 256)), S.tile0 + k});
      }
  }
  std::stable_sort(gb.begin(), gb.end(), [](const std::pair<int4, int> &a, const std::pair<int4, int> &b) {
    return (long long)(a.first.y - a.first.x) * (a.first.w - a.first.z) >
           (long long)(b.first.y - b.first.x) * (b.first.w - b.first.z);
  });
  std::vector<int4> gbi(gb.size());
  std::vector<int> gbs(gb.size());
  for (size_t k = 0; k < gb.size(); k++) {
    gbi[k] = gb[k].first;
    gbs[k] = gb[k].second;
  }
  if (upload(P.item_allocs, &d.row_perm, row_perm) || upload(P.item_allocs, &d.rblk, rblk) ||
      upload(P.item_allocs, &d.desc_items, desc) || upload(P.item_allocs, &d.dt_items, dt) || upload(P.item_allocs, &d.chain_items, chain) ||
      upload(P.item_allocs, &d.cperm, cperm) || upload(P.item_allocs, &d.cblk, cblk) ||
      upload(P.item_allocs, &d.ch_cstart, ch_cstart) || upload(P.item_allocs, &d.ch_contrib, ch_contrib) ||
      upload(P.item_allocs, &d.chain_sub, sub) || upload(P.item_allocs, &d.chain_sets, sets) ||
      upload(P.item_allocs, &d.gb_items, gbi) || upload(P.item_allocs, &d.gb_eslot, gbs))
    return AGBNP_ERR;
  d.rows = rows;
  d.nrow_blocks = (int)rblk.size();
  d.ndesc_items = (int)desc.size();
  d.ndt_items = (int)dt.size();
  d.dt_run = desc_cols / 256;
  d.nchain_items = (int)chain.size();
  d.nchain_sub = (int)sub.size();
  d.ncblk = (int)cblk.size();
  d.ngb_items = (int)gbi.size();
  return AGBNP_OK;
}

// Per-call working state: every buffer the kernels of one call write before
// they read it (the call's own coordinates, cell grids, neighbour list,
// scatter accumulators, per-atom factors, water sites, energy partials).
// Nothing in it carries over from one call to the next.  Each buffer starts
// on a 256-byte boundary of one block; with base == nullptr only the size is
// computed.  The neighbour-list rows are `cap` wide.
size_t carve_call_state(Dev &d, char *base, int n_, int nh_, int nsys, int nws_, int nablk, int ntile, int cap,
                        int nchain, size_t nsplit, size_t ndpart) {
  const size_t n = std::max(n_, 1), nh = std::max(nh_, 1), nws = std::max(nws_, 1);
  size_t off = 0;
  auto take = [&](auto *&ptr, size_t count) {
    using T = std::remove_reference_t<decltype(*ptr)>;
    off = (off + 255) & ~(size_t)255;
    ptr = base ? reinterpret_cast<T *>(base + off) : nullptr;
    off += std::max(count, (size_t)1) * sizeof(T);
  };
  take(d.pos, n);
  take(d.grid, (size_t)nsys);
  take(d.cell_start, (size_t)nsys * (kMaxCells + 1));
  take(d.cell_atoms, n);
  take(d.cell_tmp, n);
  take(d.nne, nh);
  take(d.nbr, nh * (size_t)cap);
  take(d.tree_ovf, 2 * nh);
  take(d.tree_tier, nh);
  take(d.acc_vol, n);
  take(d.acc_sa, n);
  take(d.acc_grad, n * TG_N);
  take(d.acc_hb, 3 * n);
  take(d.acc_derh, n);
  take(d.acc_beta, n);
  take(d.acc_gbA, n);
  take(d.acc_gbg, 3 * n);
  take(d.acc_ch, 8 * n);
  for (double **q : {&d.volumep_raw, &d.sa_raw, &d.sa_f, &d.sp, &d.spe, &d.psvol, &d.gammap, &d.beta, &d.br,
                     &d.brw, &d.swf, &d.A, &d.q2ab, &d.abrw, &d.deru, &d.derv, &d.derus, &d.dervs, &d.derh})
    take(*q, n);
  d.tree_cnt = reinterpret_cast<uint2 *>(d.A);
  for (float **q : {&d.sp_f, &d.spe_f, &d.br_f, &d.q2ab_f, &d.abrw_f, &d.deru_f, &d.derv_f, &d.derus_f,
                    &d.dervs_f, &d.derh_f, &d.gammap_f})
    take(*q, n);
  take(d.dcol, n);
  take(d.dcw, n);
  if (d.cull_chain) take(d.chbox, 8 * (size_t)std::max(d.ncblk, 1));
  take(d.gb_epart, (size_t)std::max(ntile, 1));
  const size_t ngbs = ntile <= kGbSplitItems ? ntile : 0;
  take(d.gbsplit, ngbs * kGbSets * 1024);
  take(d.gbener, ngbs * 4);
  take(d.ws_part, nws);
  take(d.ws_ovf, nws);
  take(d.epart, (size_t)EP_COUNT * std::max(nablk, 1));
  take(d.dpart, ndpart);
  take(d.chpart, (size_t)nchain * 2 * 8 * 256);
  // the descreening's boxes are read before the chain rule writes there
  const size_t nbox = d.cull_desc ? 2 * (size_t)std::max(nablk, 1) * (256 / kBoxCols) : 0;
  if (nbox * sizeof(float4) <= (size_t)nchain * 2 * 8 * 256 * sizeof(float)) d.cbox = reinterpret_cast<float4 *>(d.chpart);
  else take(d.cbox, nbox);
  take(d.chsplit, nsplit);
  take(d.ch_done, (size_t)nchain);
  take(d.ch_flag, 4 * (size_t)std::max(d.ncblk, 1));
  return (off + 255) & ~(size_t)255;
}

// the second stream and its events
int make_side(Pack &P) {
  HIPCHK(hipStreamCreateWithFlags(&P.side, hipStreamNonBlocking));
  // (the streams are one device's: no fence towards the host)
  for (hipEvent_t *e : {&P.ev_fork, &P.ev_join, &P.ev_fork2, &P.ev_join2})
    HIPCHK(hipEventCreateWithFlags(e, hipEventDisableTiming | hipEventDisableSystemFence));
  return AGBNP_OK;
}

// the pack's own per-call state and host-API staging, on first use (calls
// from agbnp3_ener_static use the library's static scratch instead)
constexpr size_t kHstatBytes = 256;    // (the staging behind it starts on a line)
int ensure_call_state(Pack &P, bool host_api = false) {
  Dev &d = P.d;
  // pinned memory: the call's status and counters, and the host API's staging
  // behind them (calls on device pointers do without those megabytes)
  if (host_api ? !P.hstage : !P.hstat) {
    const size_t stage = host_api ? (18 * (size_t)P.n + 7 * (size_t)P.nsys) * sizeof(double) : 0;
    char *blk = nullptr;
    HIPCHK(hipHostMalloc((void **)&blk, kHstatBytes + stage, hipHostMallocDefault));
    P.pinned.push_back(blk);
    memset(blk, 0, kHstatBytes);
    if (!P.hstat) P.hstat = reinterpret_cast<unsigned long long *>(blk);
    if (host_api) P.hstage = reinterpret_cast<double *>(blk + kHstatBytes);
  }
  d.hstat = P.hstat;
  if (P.call_block && d.nchain_items <= P.call_nchain && P.call_nsplit() <= P.call_split &&
      P.call_ndpart() <= P.call_dpart) return AGBNP_OK;
  if (P.call_block) {            // more items than the block holds (another launch shape)
    HIPCHK(hipStreamSynchronize(P.stream));
    if (P.side) HIPCHK(hipStreamSynchronize(P.side));
    (void)hipFree(P.call_block);
    P.call_block = nullptr;
  }
  const size_t bytes = carve_call_state(d, nullptr, P.n, P.nh, P.nsys, d.nws, d.nablk, P.ntile, 256, d.nchain_items, P.call_nsplit(),
                                       P.call_ndpart());
  const size_t nn = std::max(P.n, 1);
  const size_t outs = 15 * nn + 7 * (size_t)P.nsys;
  char *blk = nullptr;
  if (hipMalloc((void **)&blk, bytes + outs * sizeof(double)) != hipSuccess) {
    errprint("agbnp3: device allocation of %zu bytes failed\n", bytes + outs * sizeof(double));
    return AGBNP_ERR;
  }
  P.call_block = blk;
  P.call_nchain = d.nchain_items;
  P.call_split = P.call_nsplit();
  P.call_dpart = P.call_ndpart();
  carve_call_state(d, blk, P.n, P.nh, P.nsys, d.nws, d.nablk, P.ntile, 256, d.nchain_items, P.call_nsplit(),
                                       P.call_ndpart());
  P.dout = reinterpret_cast<double *>(blk + bytes);
  HIPCHK(hipMemset(d.ws_part, 0, sizeof(double) * std::max(d.nws, 1)));
  // (a pack that is only copied into a batch, or called through
  // agbnp3_ener_static, never comes here: no stream for it)
  if (!P.side && P.n >= kSideAtoms && make_side(P) != AGBNP_OK) return AGBNP_ERR;
  return AGBNP_OK;
}

void tune_apply_recorded(Pack &P);

// Pack the systems `ms` (internal order each) into one device arena.
int build_pack(Pack &P, const std::vector<const Model *> &ms, int options) {
  static unsigned long long next_uid = 1;
  P.uid = next_uid++;
  P.nsys = (int)ms.size();
  P.options = options;
  // radius types: union over the systems, by exact equality
  std::vector<std::vector<int>> lmap(P.nsys);
  for (int b = 0; b < P.nsys; b++)
    for (float r : ms[b]->radii) {
      int g = -1;
      for (int t = 0; t < (int)P.radii.size(); t++)
        if (fabsf(r - P.radii[t]) < FLT_MIN) { g = t; break; }
      if (g < 0) { g = (int)P.radii.size(); P.radii.push_back(r); }
      lmap[b].push_back(g);
    }
  P.ntypes = (int)P.radii.size();
  std::vector<int> ext2int, asys, hrow, ws_stale0;
  std::vector<float> R, q, galpha, igamma, sgamma, ialpha, salpha, hbcorr;
  std::vector<double> vols;
  std::vector<int2> ablk;
  std::vector<WsDef> wsdef;
  std::vector<int2> ws_site;
  int a0 = 0, h0 = 0, ws0 = 0, blk0 = 0, tile0 = 0;
  long long dp0 = 0;
  for (int b = 0; b < P.nsys; b++) {
    const Model &m = *ms[b];
    SysInfo S{};
    S.a0 = a0; S.n = m.natoms; S.nh = m.nheavy; S.h0 = h0;
    S.ws0 = ws0; S.nws = m.nws;
    S.blk0 = blk0; S.nblk = (m.natoms + 255) / 256;
    const int nb = (m.natoms + 255) / 256;
    S.tile0 = tile0; S.ntile = nb * (nb + 1) / 2;
    S.dp0 = (int)std::min(dp0, (long long)INT_MAX);      // (read only where all of them fit: build_items)
    S.df64 = -0.5 * (1.0 / (double)m.eps_in - 1.0 / (double)m.eps_out);
    S.df = (float)S.df64;
    float rmax = 0.f;
    for (int i = 0; i < m.nheavy; i++) rmax = std::max(rmax, m.R[i]);
    S.rmax_heavy = rmax;
    P.sinfo.push_back(S);
    for (int i = 0; i < m.natoms; i++) {
      ext2int.push_back(a0 + m.ext2int[i]);
      asys.push_back(b);
      P.rtype.push_back(lmap[b][m.rtype[i]]);
      P.heavy.push_back(i < m.nheavy);
      P.alpha_sum.push_back(m.ialpha[i] + m.salpha[i]);
      P.curve.push_back(m.curve[i]);
      R.push_back(m.R[i]); q.push_back(m.q[i]); galpha.push_back(m.galpha[i]);
      igamma.push_back(m.igamma[i]); sgamma.push_back(m.sgamma[i]);
      ialpha.push_back(m.ialpha[i]); salpha.push_back(m.salpha[i]);
      hbcorr.push_back(m.hbcorr[i]); vols.push_back(m.vols[i]);
    }
    for (int k = 0; k < m.nheavy; k++) hrow.push_back(a0 + k);
    for (int k = 0; k < S.nblk; k++) ablk.push_back(make_int2(a0 + 256 * k, std::min(a0 + m.natoms, a0 + 256 * k + 256)));
    for (WsDef w : m.wsdef) {
      w.atom += a0;
      for (int k = 0; k < 5; k++) w.p[k] += a0;
      w.first += ws0;
      for (int k = 0; k < w.nsite; k++) ws_site.push_back(make_int2((int)wsdef.size(), k));
      wsdef.push_back(w);
    }
    for (int s : m.ws_stale0) ws_stale0.push_back(s >= 0 && s < m.natoms ? a0 + s : -1);
    dp0 += (long long)m.natoms * ((m.nheavy + 255) / 256);
    a0 += m.natoms; h0 += m.nheavy; ws0 += m.nws; blk0 += S.nblk; tile0 += S.ntile;
  }
  P.n = a0;
  P.nh = h0;
  P.ndpart = dp0;
  Dev &d = P.d;
  d = Dev{};
  d.n = P.n;
  d.nh = P.nh;
  d.nsys = P.nsys;
  d.ntypes = P.ntypes;
  d.cap = P.cap;
  d.options = options;
  d.nws = ws0;
  d.nablk = blk0;
  // water-site candidates the first free-volume launch takes: 128, or fewer
  // from AGBNP3_WS_FIRST_CAP (1..128) so tests can route sites to the second
  d.ws_cap1 = 128;
  if (const char *e = getenv("AGBNP3_WS_FIRST_CAP")) {
    const int v = atoi(e);
    if (v >= 1 && v <= 128) d.ws_cap1 = v;
  }
  // likewise the nodes that the derivative pass's first tier takes, from
  // AGBNP3_TREE_DERIV_CAP, so a test can have a root outgrow it alone
  d.tree_cap_b = kLevelCap;
  if (const char *e = getenv("AGBNP3_TREE_DERIV_CAP")) {
    const int v = atoi(e);
    if (v >= 1 && v <= kLevelCap) d.tree_cap_b = v;
  }
  std::vector<float> ty((size_t)P.ntypes * P.ntypes * kTblN), ty2(ty.size());
  for (int a = 0; a < P.ntypes; a++)
    for (int b = 0; b < P.ntypes; b++) {
      const float c = kRadInc;
      const float ratio = (P.radii[a] - c) / P.radii[b];
      const size_t t = (size_t)(a * P.ntypes + b) * kTblN;
      build_table(ratio, &ty[t], &ty2[t], d.tdx, d.tdxinv);
    }
  std::vector<float2> tb(ty.size());
  for (size_t k = 0; k < tb.size(); k++) tb[k] = make_float2(ty[k], ty2[k]);
  std::vector<float4> ctab;
  chain_tables(ty, ty2, P.ntypes * P.ntypes, d.tdx, ctab);
  auto &L = P.allocs;
  if (upload(L, &d.sys, P.sinfo) || upload(L, &d.asys, asys) || upload(L, &d.hrow, hrow) ||
      upload(L, &d.ext2int, ext2int) || upload(L, &d.R, R) || upload(L, &d.q, q) || upload(L, &d.rtype, P.rtype) ||
      upload(L, &d.galpha, galpha) || upload(L, &d.igamma, igamma) || upload(L, &d.sgamma, sgamma) ||
      upload(L, &d.ialpha, ialpha) || upload(L, &d.salpha, salpha) || upload(L, &d.hbcorr_f, hbcorr) ||
      upload(L, &d.vols, vols) || upload(L, &d.tbl, tb) || upload(L, &d.ctab, ctab) || upload(L, &d.ablk, ablk) ||
      upload(L, &d.wsdef, wsdef) || upload(L, &d.ws_site, ws_site) || upload(L, &d.ws_stale0, ws_stale0))
    return AGBNP_ERR;
  P.ntile = tile0;
  float reaches = 0.f;                  // of the widest solute (as created; only a choice of kernels)
  for (int b = 0; b < P.nsys; b++)
    if (P.sinfo[b].nh) reaches = std::max(reaches, ms[b]->extent / (kTblAmax * P.sinfo[b].rmax_heavy));
  d.cull_desc = reaches > kCullDesc && P.ntypes <= kLdsTypes;
  d.cull_chain = reaches > kCullChain;
  // state that lives as long as the pack: status word, counters, queue heads
  if (dalloc(L, &d.status, 1) || dalloc(L, &d.queue, kQueueWords) || dalloc(L, &d.counters, kCounters))
    return AGBNP_ERR;
  HIPCHK(hipMemset(d.status, 0, sizeof(int)));
  HIPCHK(hipMemset(d.counters, 0, sizeof(unsigned long long) * kCounters));
  HIPCHK(hipGetDevice(&P.device));
  HIPCHK(hipStreamCreateWithFlags(&P.stream, hipStreamNonBlocking));
  if (P.n >= kForkAtoms && make_side(P) != AGBNP_OK) return AGBNP_ERR;
  HIPCHK(prepare_pairs(P.ntypes));
  HIPCHK(prepare_sites(P.ntypes));
  HIPCHK(prepare_tree());
  tune_apply_recorded(P);
  return build_items(P);
}

// ---------------------------------------------------------- the pipeline
// GB pairs by chunks, unless a grid is asked for
bool gb_by_chunks(const Dev &d) {
  return d.ngb_items <= kGbSplitItems && d.nchain_items <= kChainGroupItems && !d.sg_on;
}

// The kernels of one call on the pack's stream, with `d` the device view (the
// pack's own, or a copy whose per-call state lies in the static scratch).
// `capturing`: inside a graph capture (no timing events).
int run_pipeline_on(Pack &P, Dev &d, const double *x, const double *y, const double *z, double *sp, double *br,
                    double *sa, double *dgbdr, double *dvwdr, double *decav, double *dehb, double *energies,
                    bool capturing) {
  d.options = P.options;
  d.cap = P.cap;
  d.skin = P.skin;
  d.reuse_every = P.reuse_every;
  d.dt_on = P.dt && !d.sg_on;
  d.split_on = P.split && !d.sg_on;
  d.gbs_on = gb_by_chunks(d) && P.tune.gb_grid == 0;
  hipStream_t s = P.stream;
  const bool timed = !capturing && (P.options & AGBNP3_OPT_TIMING) != 0;
  int k = 0;
  std::vector<hipEvent_t> *set = nullptr;
  if (timed) {
    if ((size_t)P.ncalls_timed >= P.ev_sets.size()) P.ev_sets.emplace_back();
    set = &P.ev_sets[P.ncalls_timed++];
  }
  auto mark = [&](const char *name) {
    if (!timed) return;
    if ((size_t)k >= set->size()) {
      hipEvent_t e;
      (void)hipEventCreate(&e);
      set->push_back(e);
    }
    if ((size_t)k >= P.ev_names.size()) P.ev_names.push_back(name);
    P.ev_names[k] = name;
    (void)hipEventRecord((*set)[k], s);
    k++;
  };
  const Tuning &t = P.tune;
  mark("start");
  launch_ingest(d, x, y, z, s);
  mark("ingest");
  launch_cells(d, s);
  mark("cells");
  launch_nblist(d, s);
  mark("nblist");
  launch_tree(d, t, 0, s);
  mark("tree_volumes");
  launch_scale(d, s);
  mark("scale");
  // the water sites need only the self volumes: they share the tiled
  // descreening's launch, or run on the second stream beside the descreening
  // (with per-kernel timing every kernel stays on the one stream; below
  // kForkAtoms atoms the fork and join cost more than the overlap saves)
  const bool fork = !timed && P.side && d.nws > 0 && d.n >= kForkAtoms && !d.dt_on;
  if (fork) {
    HIPCHK(hipEventRecord(P.ev_fork, s));
    HIPCHK(hipStreamWaitEvent(P.side, P.ev_fork, 0));
    launch_ws_free(d, P.side);
    HIPCHK(hipEventRecord(P.ev_join, P.side));
  }
  launch_sg_front(d, s);
  mark("sg_front");
  if (d.dt_on) launch_desc_sites(d, s);
  else launch_descreen(d, t, s);
  mark("descreen");
  launch_born(d, s);
  mark("born");
  launch_gbpair(d, t, s);
  mark("gbpair");
  launch_q2ab(d, s);
  mark("q2ab");
  launch_sg_audit(d, s);
  if (fork) {
    HIPCHK(hipStreamWaitEvent(s, P.ev_join, 0));
  } else {
    if (!d.dt_on) launch_ws_free(d, s);
    mark("ws_free");                     // (every call has the same marks: pack_kernel_times)
  }
  launch_chain(d, t, s);
  mark("chain");
  launch_sg_grad(d, s);
  mark("sg_grad");
  launch_uv(d, s);
  mark("uv");
  // derivative pass: its second tier takes the roots pass A's first tier
  // queued, so it does not wait for the first tier and runs beside it on the
  // second stream (the largest trees start at once instead of after the rest)
  const bool fork2 = !timed && P.side;
  if (fork2) {
    HIPCHK(hipEventRecord(P.ev_fork2, s));
    HIPCHK(hipStreamWaitEvent(P.side, P.ev_fork2, 0));
    const int there = d.nh > kBigFirst && !capturing ? 0 : 1;    // the tier on the second stream
    launch_tree_tier(d, t, 1, there, P.side);
    HIPCHK(hipEventRecord(P.ev_join2, P.side));
    launch_tree_tier(d, t, 1, 1 - there, s);
    HIPCHK(hipStreamWaitEvent(s, P.ev_join2, 0));
  } else {
    launch_tree(d, t, 1, s);
  }
  mark("tree_derivs");
  launch_final(d, sp, br, sa, dgbdr, dvwdr, decav, dehb, energies, s);
  mark("final");
  if (!capturing) {
    P.host_status = d.hstat != nullptr;
    const bool group = d.nchain_items <= kChainGroupItems;
    P.routes = (d.dt_on ? 1 | (desc_sites_few(d) ? 2 : 0) : (d.cull_desc ? 4 : 0)) | (d.gbs_on ? 8 : 0) |
               (d.split_on ? 16 : (group ? 32 : (d.cull_chain ? 64 : 0)));
  }
  HIPCHK(hipGetLastError());
  return AGBNP_OK;
}

int run_pipeline(Pack &P, const double *x, const double *y, const double *z, double *sp, double *br, double *sa,
                 double *dgbdr, double *dvwdr, double *decav, double *dehb, double *energies, bool capturing) {
  if (!P.call_block) {
    if (capturing) {      // pack_capture allocates before the capture begins
      errprint("agbnp3: no per-call state to capture\n");
      return AGBNP_ERR;
    }
    if (ensure_call_state(P) != AGBNP_OK) return AGBNP_ERR;
  }
  return run_pipeline_on(P, P.d, x, y, z, sp, br, sa, dgbdr, dvwdr, decav, dehb, energies, capturing);
}

// status word and largest neighbour-list row of the last call (waits)
int read_status(Pack &P, int *status, int *maxrow) {
  if (P.host_status) {                  // k_final has written it to host memory
    HIPCHK(hipStreamSynchronize(P.stream));
    *status = (int)(P.d.hstat[0] & 0xffffffffull);
    if (maxrow) *maxrow = (int)P.d.hstat[1 + 3];
    return AGBNP_OK;
  }
  int st = 0;
  unsigned long long c[4] = {0, 0, 0, 0};
  HIPCHK(hipMemcpyAsync(&st, P.d.status, sizeof(int), hipMemcpyDeviceToHost, P.stream));
  HIPCHK(hipMemcpyAsync(c, P.d.counters, sizeof(c), hipMemcpyDeviceToHost, P.stream));
  HIPCHK(hipStreamSynchronize(P.stream));
  *status = st;
  if (maxrow) *maxrow = (int)c[3];
  return AGBNP_OK;
}

int pack_capture(Pack &P, const double *x, const double *y, const double *z, double *sp, double *br, double *sa,
                 double *dgbdr, double *dvwdr, double *decav, double *dehb, double *energies);

// Status of the last call (waits).  A neighbour-list row that outgrew the
// row capacity fails the call; the rows are widened for the next call (and a
// captured graph is captured again with the same pointers), so a device-API
// caller recovers as the host API does within its call.
int pack_sync(Pack &P, const char *who) {
  int st = 0;
  if (read_status(P, &st, nullptr) != AGBNP_OK) return AGBNP_ERR;
  if (st) {
    if ((st & ST_NBLIST_OVERFLOW) && P.cap < 256) {
      const bool had_graph = P.gexec != nullptr;
      P.cap = P.cap < 128 ? 128 : 256;
      drop_graph(P);
      errprint("%s: a neighbour-list row exceeded its capacity; rows are %d wide from the next call.\n", who,
               P.cap);
      if (had_graph)
        (void)pack_capture(P, P.cap_in[0], P.cap_in[1], P.cap_in[2], P.cap_out[0], P.cap_out[1], P.cap_out[2],
                           P.cap_out[3], P.cap_out[4], P.cap_out[5], P.cap_out[6], P.cap_out[7]);
      return AGBNP_ERR;
    }
    errprint("%s: device status 0x%x (capacity exceeded)\n", who, st);
    return AGBNP_ERR;
  }
  return AGBNP_OK;
}

// neighbour-list row capacity for the next call: the smallest variant that
// holds the longest row seen with a margin (smaller rows give the tree
// kernels more waves per CU)
void adapt_cap(Pack &P, int maxrow) {
  const int want = maxrow + 8 <= 64 ? 64 : (maxrow + 8 <= 128 ? 128 : 256);
  if (want != P.cap) {
    P.cap = want;
    drop_graph(P);
  }
}

// Evaluate with host arrays (caller order, concatenated over the systems):
// stage through pinned memory, retry once with wider rows when a row
// overflowed, copy the outputs back.
int pack_ener_host(Pack &P, const double *x, const double *y, const double *z, double *out /* 15n + 7 nsys */,
                   const char *who) {
  if (ensure_call_state(P, true) != AGBNP_OK) return AGBNP_ERR;
  const size_t n = P.n;
  double *h = P.hstage;
  double *hin = h + 15 * n + 7 * (size_t)P.nsys;
  memcpy(hin, x, n * sizeof(double));
  memcpy(hin + n, y, n * sizeof(double));
  memcpy(hin + 2 * n, z, n * sizeof(double));
  // the kernels read the coordinates and write outputs and status in place
  // (copies would be five launches of their own, 30 us of a small call): one
  // wait per call; the outputs of a call that overflowed are discarded and
  // the call re-run
  for (int attempt = 0; attempt < 3; attempt++) {
    if (run_pipeline(P, hin, hin + n, hin + 2 * n, h, h + n, h + 2 * n, h + 3 * n, h + 6 * n, h + 9 * n, h + 12 * n,
                     h + 15 * n, false) != AGBNP_OK)
      return AGBNP_ERR;
    HIPCHK(hipStreamSynchronize(P.stream));
    const unsigned long long *hst = P.d.hstat;
    const int st = (int)(hst[0] & 0xffffffffull), maxrow = (int)hst[1 + 3];
    if (st == 0) {
      adapt_cap(P, maxrow);
      break;
    }
    if ((st & ST_NBLIST_OVERFLOW) && P.cap < 256) {
      P.cap = P.cap < 128 ? 128 : 256;     // wider rows; re-run the call
      drop_graph(P);
      continue;
    }
    errprint("%s: device capacity exceeded (status 0x%x).\n", who, st);
    return AGBNP_ERR;
  }
  if (out != h) memcpy(out, h, (15 * n + 7 * (size_t)P.nsys) * sizeof(double));
  return AGBNP_OK;
}

// ------------------------------------------------------------- timing
int pack_kernel_times(Pack &P, float *ms, int nmax, char *names, int names_len) {
  HIPCHK(hipStreamSynchronize(P.stream));
  const int nk = P.ev_names.empty() ? 0 : (int)P.ev_names.size() - 1;
  const int k = std::min(nmax, nk);
  std::vector<double> acc(std::max(nk, 1), 0.0);
  for (int c = 0; c < P.ncalls_timed; c++) {
    const auto &set = P.ev_sets[c];
    for (int i = 0; i < nk && i + 1 < (int)set.size(); i++) {
      float t = 0.f;
      (void)hipEventElapsedTime(&t, set[i], set[i + 1]);
      acc[i] += t;
    }
  }
  std::string all;
  for (int i = 0; i < k; i++) {
    if (ms) ms[i] = P.ncalls_timed ? (float)(acc[i] / P.ncalls_timed) : 0.f;
    if (i) all += ";";
    all += P.ev_names[i + 1];
  }
  if (names && names_len > 0) {
    strncpy(names, all.c_str(), names_len - 1);
    names[names_len - 1] = 0;
  }
  P.ncalls_timed = 0;
  return k;
}

// ------------------------------------------------------------ autotuner
// Times the pipeline on the caller's coordinates for each candidate launch
// shape and keeps, kernel by kernel, the fastest: rows per spline block,
// column chunk of the descreening and chain items, persistent grid sizes.
// Coordinate descent; every trial is one warm-up call and `reps` timed calls.
enum : int { TUNE_ROWS = 0, TUNE_DESC_CHUNK, TUNE_CHAIN_CHUNK, TUNE_DESC_GRID, TUNE_GB_GRID, TUNE_CHAIN_GRID,
             TUNE_CAP, TUNE_TREE_GRID, TUNE_COUNT };

void tuning_to_params(const Pack &P, int *p) {
  p[TUNE_ROWS] = P.tune.rows;
  p[TUNE_DESC_CHUNK] = P.tune.desc_chunk;
  p[TUNE_CHAIN_CHUNK] = P.tune.chain_chunk;
  p[TUNE_DESC_GRID] = P.tune.desc_grid;
  p[TUNE_GB_GRID] = P.tune.gb_grid;
  p[TUNE_CHAIN_GRID] = P.tune.chain_grid;
  p[TUNE_CAP] = P.cap;
  p[TUNE_TREE_GRID] = P.tune.tree_grid;
}

int params_to_tuning(Pack &P, const int *p) {
  Tuning t;
  t.rows = p[TUNE_ROWS];
  t.desc_chunk = p[TUNE_DESC_CHUNK];
  t.chain_chunk = p[TUNE_CHAIN_CHUNK];
  t.desc_grid = p[TUNE_DESC_GRID];
  t.gb_grid = p[TUNE_GB_GRID];
  t.chain_grid = p[TUNE_CHAIN_GRID];
  t.tree_grid = p[TUNE_TREE_GRID];
  const int cap = p[TUNE_CAP];
  if ((t.rows != 64 && t.rows != 128 && t.rows != 256) || t.desc_chunk < 0 || t.desc_grid < 0 || t.gb_grid < 0 ||
      t.chain_grid < 0 || t.tree_grid < 0 || (cap != 64 && cap != 128 && cap != 256) || (t.desc_chunk % 256) ||
      (t.chain_chunk != 0 && t.chain_chunk != 64 && t.chain_chunk != 128 && t.chain_chunk != 256)) {
    errprint("agbnp3: invalid launch shape (rows %d, chunks %d/%d, grids %d/%d/%d/%d, cap %d)\n", t.rows,
             t.desc_chunk, t.chain_chunk, t.desc_grid, t.gb_grid, t.chain_grid, t.tree_grid, cap);
    return AGBNP_ERR;
  }
  const bool rebuild = t.rows != P.tune.rows || t.desc_chunk != P.tune.desc_chunk ||
                       t.chain_chunk != P.tune.chain_chunk;
  P.tune = t;
  P.cap = cap;
  drop_graph(P);
  if (!rebuild) return AGBNP_OK;
  if (build_items(P) != AGBNP_OK) return AGBNP_ERR;
  return P.call_block ? ensure_call_state(P) : AGBNP_OK;
}

// Launch shapes chosen by the tuner, per size class of a pack: the number of
// systems in octaves and the total atom count in half octaves.  Packs built
// later in a class start from its recorded shapes; the table can be written
// to and read from a text file (one class per line: the two class numbers,
// then the TUNE_COUNT parameters).
std::map<std::pair<int, int>, std::vector<int>> g_tune_table;
std::mutex g_tune_mutex;

std::pair<int, int> size_class(const Pack &P) {
  const int s = (int)std::ceil(std::log2((double)std::max(P.nsys, 1)));
  const int a = (int)std::lround(2.0 * std::log2((double)std::max(P.n, 1)));
  return {s, a};
}

void tune_record(const Pack &P) {
  std::vector<int> p(TUNE_COUNT);
  tuning_to_params(P, p.data());
  std::lock_guard<std::mutex> lk(g_tune_mutex);
  g_tune_table[size_class(P)] = p;
}

// shapes recorded for the pack's class, if any (before its items are built)
void tune_apply_recorded(Pack &P) {
  std::vector<int> p;
  {
    std::lock_guard<std::mutex> lk(g_tune_mutex);
    auto it = g_tune_table.find(size_class(P));
    if (it == g_tune_table.end()) return;
    p = it->second;
  }
  P.tune.rows = p[TUNE_ROWS];
  P.tune.desc_chunk = p[TUNE_DESC_CHUNK];
  P.tune.chain_chunk = p[TUNE_CHAIN_CHUNK];
  P.tune.desc_grid = p[TUNE_DESC_GRID];
  P.tune.gb_grid = p[TUNE_GB_GRID];
  P.tune.chain_grid = p[TUNE_CHAIN_GRID];
  P.tune.tree_grid = p[TUNE_TREE_GRID];
  P.cap = p[TUNE_CAP];
}

int pack_tune(Pack &P, const double *x, const double *y, const double *z, int reps, char *report, int report_len) {
  reps = std::max(1, reps);
  if (ensure_call_state(P) != AGBNP_OK) return AGBNP_ERR;
  const size_t n = P.n;
  // one call into the pack's own output buffers; P.dout is read at each call,
  // since a shape with more chain-rule items reallocates the per-call block
  auto call = [&]() {
    double *o = P.dout;
    return run_pipeline(P, x, y, z, o, o + n, o + 2 * n, o + 3 * n, o + 6 * n, o + 9 * n, o + 12 * n, o + 15 * n,
                        false);
  };
  const int saved_opts = P.options;
  std::string rep;
  char line[256];
  // one untimed call sizes the neighbour-list rows
  {
    P.options = saved_opts & ~AGBNP3_OPT_TIMING;
    if (call() != AGBNP_OK) return AGBNP_ERR;
    int st = 0, maxrow = 0;
    if (read_status(P, &st, &maxrow) != AGBNP_OK) return AGBNP_ERR;
    if (st & ST_NBLIST_OVERFLOW) {
      P.cap = 256;
    } else {
      adapt_cap(P, maxrow);
    }
  }
  // time one configuration: average ms per kernel name
  auto trial = [&](std::map<std::string, double> &out) -> int {
    P.options = (saved_opts & ~AGBNP3_OPT_TIMING);
    if (call() != AGBNP_OK) return AGBNP_ERR;
    P.options = saved_opts | AGBNP3_OPT_TIMING;
    pack_kernel_times(P, nullptr, 0, nullptr, 0);
    for (int r = 0; r < reps; r++)
      if (call() != AGBNP_OK) return AGBNP_ERR;
    int st = 0;
    if (read_status(P, &st, nullptr) != AGBNP_OK || st) return AGBNP_ERR;
    std::vector<float> ms(64);
    std::vector<char> names(2048);
    const int k = pack_kernel_times(P, ms.data(), 64, names.data(), (int)names.size());
    out.clear();
    std::string all(names.data());
    size_t pos = 0;
    for (int i = 0; i < k; i++) {
      const size_t e = all.find(';', pos);
      out[all.substr(pos, e == std::string::npos ? std::string::npos : e - pos)] = ms[i];
      pos = e == std::string::npos ? all.size() : e + 1;
    }
    return AGBNP_OK;
  };
  int p[TUNE_COUNT];
  tuning_to_params(P, p);
  std::map<std::string, double> t;
  int cu = 256;
  {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
      cu = prop.multiProcessorCount;
  }
  // each step: a parameter, its candidates, the kernels whose time decides.
  // Some candidates move work between kernels (the tiled descreening holds the
  // water sites, the GB pairs by chunks what k_q2ab does), so these count
  // together.  (The descreening by itself chose 1,024 columns at 61 atoms, on a
  // tie: 120 -> 136 us a call.)
  struct Axis {
    int param;
    std::vector<int> cand;
    std::vector<std::string> kernels;
  };
  const std::vector<Axis> axes = {
      {TUNE_ROWS, {64, 128, 256}, {"descreen", "ws_free"}},
      {TUNE_DESC_CHUNK, {0, 512, 1024, 2048, 4096}, {"descreen", "ws_free"}},
      {TUNE_DESC_GRID, {0, 2 * cu, 4 * cu, 8 * cu}, {"descreen", "ws_free"}},
      {TUNE_GB_GRID, {0, 2 * cu, 4 * cu, 8 * cu}, {"gbpair", "q2ab"}},
      {TUNE_CHAIN_CHUNK, {0, 128, 64}, {"chain"}},
      {TUNE_CHAIN_GRID, {0, 2 * cu, 4 * cu, 8 * cu}, {"chain"}},
      {TUNE_TREE_GRID, {0, 8 * cu, 32 * cu}, {"tree_volumes", "tree_derivs"}},
  };
  for (const Axis &ax : axes) {
    // grids of kernels that this pack's calls don't launch stay as they are, and
    // candidates that are what 0 stands for are left out: a choice among equals
    // would be recorded for the class's other packs, and may take another route
    // from them
    if (params_to_tuning(P, p) != AGBNP_OK) {
      P.options = saved_opts;
      return AGBNP_ERR;
    }
    if (!P.d.sg_on && ((ax.param == TUNE_DESC_GRID && P.dt) || (ax.param == TUNE_CHAIN_GRID && P.split))) continue;
    const Dev &d = P.d;
    int same = INT_MAX;                  // grids from here are a block per item
    if (ax.param == TUNE_DESC_GRID) same = d.ndesc_items;
    if (ax.param == TUNE_GB_GRID && !gb_by_chunks(d)) same = d.ngb_items;
    if (ax.param == TUNE_CHAIN_GRID) same = d.nchain_items;
    if (ax.param == TUNE_TREE_GRID) same = d.nh;
    // and the columns that 0 stands for (with tiles it is another kernel)
    const int cols = ax.param == TUNE_DESC_CHUNK && p[ax.param] == 0 && !(P.dt && !d.sg_on) ? 256 * d.dt_run : 0;
    int best = p[ax.param];
    double best_t = 1e30;
    for (int c : ax.cand) {
      if (c > 0 && (c >= same || c == cols)) continue;
      int q[TUNE_COUNT];
      memcpy(q, p, sizeof(q));
      q[ax.param] = c;
      if (params_to_tuning(P, q) != AGBNP_OK || trial(t) != AGBNP_OK) {
        P.options = saved_opts;
        return AGBNP_ERR;
      }
      double tt = 0.0;
      std::string counted;
      for (const auto &kname : ax.kernels) {
        tt += t[kname];
        counted += " " + kname;
      }
      snprintf(line, sizeof(line), "param %d = %d: %.4f ms (%s)\n", ax.param, c, tt, counted.c_str() + 1);
      rep += line;
      if (tt < best_t) { best_t = tt; best = c; }
    }
    p[ax.param] = best;
  }
  P.options = saved_opts;
  if (params_to_tuning(P, p) != AGBNP_OK) return AGBNP_ERR;
  tune_record(P);
  snprintf(line, sizeof(line),
           "chosen: rows %d desc_chunk %d chain_chunk %d desc_grid %d gb_grid %d chain_grid %d cap %d tree_grid %d\n",
           p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7]);
  rep += line;
  if (report && report_len > 0) {
    strncpy(report, rep.c_str(), report_len - 1);
    report[report_len - 1] = 0;
  }
  return AGBNP_OK;
}

// caller arrays of float_i as double: the caller's memory itself when
// float_i is double, else a converted copy in `tmp`
template <typename T>
const double *as_double(const T *p, size_t n, std::vector<double> &tmp) {
  if constexpr (std::is_same<T, double>::value) {
    return p;
  } else {
    tmp.assign(p, p + n);
    return tmp.data();
  }
}
template <typename T>
void store(T *dst, const double *src, size_t n) {
  if constexpr (std::is_same<T, double>::value) {
    memcpy(dst, src, n * sizeof(double));
  } else {
    for (size_t k = 0; k < n; k++) dst[k] = (T)src[k];
  }
}

int pack_capture(Pack &P, const double *x, const double *y, const double *z, double *sp, double *br, double *sa,
                 double *dgbdr, double *dvwdr, double *decav, double *dehb, double *energies) {
  drop_graph(P);
  if (ensure_call_state(P) != AGBNP_OK) return AGBNP_ERR;
  HIPCHK(hipStreamSynchronize(P.stream));
  HIPCHK(hipStreamBeginCapture(P.stream, hipStreamCaptureModeThreadLocal));
  const int rc = run_pipeline(P, x, y, z, sp, br, sa, dgbdr, dvwdr, decav, dehb, energies, true);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(P.stream, &g);
  if (rc != AGBNP_OK || e != hipSuccess) {
    errprint("agbnp3: graph capture failed: %s\n", hipGetErrorString(e));
    if (g) (void)hipGraphDestroy(g);
    return AGBNP_ERR;
  }
  P.graph = g;
  HIPCHK(hipGraphInstantiate(&P.gexec, P.graph, nullptr, nullptr, 0));
  P.cap_in[0] = x; P.cap_in[1] = y; P.cap_in[2] = z;
  double *outs[8] = {sp, br, sa, dgbdr, dvwdr, decav, dehb, energies};
  for (int k = 0; k < 8; k++) P.cap_out[k] = outs[k];
  return AGBNP_OK;
}

}  // namespace
// ======================================================================== API
extern "C" {

int agbnp3_initialize(void) {
  std::lock_guard<std::mutex> lk(g_mutex);
  if (g_initialized) return AGBNP_OK;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
    errprint("agbnp3_initialize(): no HIP device available.\n");
    return AGBNP_ERR;
  }
  int dev = 0;
  char *base = nullptr;
  if (hipGetDevice(&dev) != hipSuccess || scratch_base(dev, &base) != AGBNP_OK) {
    errprint("agbnp3_initialize(): static scratch unavailable.\n");
    return AGBNP_ERR;
  }
  g_initialized = true;
  return AGBNP_OK;
}

void agbnp3_terminate(void) {
  std::lock_guard<std::mutex> lk(g_mutex);
  if (!g_initialized) {
    errprint("agbnp3_terminate(): agbnp library is not initialized.\n");
    return;
  }
  for (auto &p : g_slots) {
    if (p) {
      free_pack(p->p);
      delete p;
    }
    p = nullptr;
  }
  g_slots.clear();
  for (auto &b : g_batches) {
    if (b) {
      free_pack(b->p);
      delete b;
    }
    b = nullptr;
  }
  g_batches.clear();
  for (auto &m : g_models) {
    if (m) sg_free(m);
    m = nullptr;
  }
  g_models.clear();
  g_initialized = false;
}

// Morton keys (10 bits per axis) of the coordinates; coordinates that are not
// finite (they are only meant to be replaced by ener) go to one end
static void curve_keys(int n, const float_i *x, const float_i *y, const float_i *z, const std::vector<int> &int2ext,
                       std::vector<unsigned> &key, float &extent) {
  const float_i *c[3] = {x, y, z};
  double lo[3] = {0, 0, 0}, ext = 0;
  for (int k = 0; k < 3; k++) {
    double a = INFINITY, b = -INFINITY;
    for (int i = 0; i < n; i++)
      if (std::isfinite((double)c[k][i])) {
        a = std::min(a, (double)c[k][i]);
        b = std::max(b, (double)c[k][i]);
      }
    if (a <= b) {
      lo[k] = a;
      ext = std::max(ext, b - a);
    }
  }
  extent = (float)ext;
  key.assign(n, 0u);
  for (int i = 0; i < n; i++)
    for (int k = 0; k < 3; k++) {
      const double u = ((double)c[k][int2ext[i]] - lo[k]) / ext * 1023.0;     // (NaN where every atom is in one place)
      const unsigned q = u >= 0.0 ? (unsigned)std::min(u, 1023.0) : 0u;
      for (int b = 0; b < 10; b++) key[i] |= ((q >> b) & 1u) << (3 * b + k);
    }
}

int agbnp3_new(int *tag, int natoms, float_i *x, float_i *y, float_i *z, float_i *r, float_i *charge,
               float_i dielectric_in, float_i dielectric_out, float_i *igamma, float_i *sgamma, float_i *ialpha,
               float_i *salpha, int *hbtype, float_i *hbcorr, int nhydrogen, int *ihydrogen, NeighList *conntbl,
               int verbose) {
  std::lock_guard<std::mutex> lk(g_mutex);
  if (!g_initialized) {
    errprint("agbnp3_new(): agbnp library is not initialized.\n");
    return AGBNP_ERR;
  }
  if (!conntbl) {
    errprint("agbnp3_new(): error: NULL connection table. AGBNP v.3 requires a connection table.\n");
    return AGBNP_ERR;
  }
  if (natoms <= 0 || nhydrogen < 0 || nhydrogen > natoms || !x || !y || !z || !r || !charge || !igamma ||
      !sgamma || !ialpha || !salpha || !hbtype || !hbcorr || (nhydrogen > 0 && !ihydrogen)) {
    errprint("agbnp3_new(): invalid arguments.\n");
    return AGBNP_ERR;
  }
  Instance *inst = new Instance();
  Model *I = &inst->m;
  const int n = natoms;
  I->natoms = n;
  I->verbose = verbose;
  // heavy atoms first, hydrogens last, both in caller order (agbnp3.c:739-779)
  std::vector<char> ish(n, 0);
  for (int k = 0; k < nhydrogen; k++) {
    if (ihydrogen[k] < 0 || ihydrogen[k] >= n) {
      errprint("agbnp3_new(): hydrogen index %d out of range.\n", ihydrogen[k]);
      delete inst;
      return AGBNP_ERR;
    }
    ish[ihydrogen[k]] = 1;
  }
  int nh_count = 0;
  for (int i = 0; i < n; i++) nh_count += ish[i];
  I->nheavy = n - nh_count;
  I->int2ext.resize(n);
  I->ext2int.resize(n);
  {
    int c = 0, h = I->nheavy;
    for (int i = 0; i < n; i++) {
      const int slot = ish[i] ? h++ : c++;
      I->int2ext[slot] = i;
      I->ext2int[i] = slot;
    }
  }
  curve_keys(n, x, y, z, I->int2ext, I->curve, I->extent);
  auto f = [](double v) { return (float)v; };
  I->R.resize(n); I->q.resize(n); I->igamma.resize(n); I->sgamma.resize(n); I->ialpha.resize(n);
  I->salpha.resize(n); I->hbcorr.resize(n); I->hbtype.resize(n); I->vols.resize(n); I->galpha.resize(n);
  for (int i = 0; i < n; i++) {
    const int e = I->int2ext[i];
    I->R[i] = f((double)r[e] + (double)kRadInc);     // radius + 0.5 in double, stored FP32 (agbnp3.c:210)
    if (!(I->R[i] > kRadInc)) {
      errprint("agbnp3_new(): atom %d has a non-positive radius.\n", e);
      delete inst;
      return AGBNP_ERR;
    }
    I->q[i] = f(charge[e]);
    I->igamma[i] = f(igamma[e]);
    I->sgamma[i] = f(sgamma[e]);
    I->ialpha[i] = f(ialpha[e]);
    I->salpha[i] = f(salpha[e]);
    I->hbcorr[i] = f(hbcorr[e]);
    I->hbtype[i] = hbtype[e];
    const double R = I->R[i];
    I->vols[i] = 4.0 * kPi / 3.0 * R * R * R;
    I->galpha[i] = kKFC / (I->R[i] * I->R[i]);
  }
  I->eps_in = f(dielectric_in);
  I->eps_out = f(dielectric_out);
  // connection table, remapped (agbnp3.c:296-317)
  if (conntbl->natoms < n) {
    errprint("agbnp3_new(): connection table has %d rows for %d atoms.\n", conntbl->natoms, n);
    delete inst;
    return AGBNP_ERR;
  }
  I->cnne.resize(n);
  I->coff.assign(n + 1, 0);
  for (int i = 0; i < n; i++) {
    I->cnne[i] = conntbl->nne[I->int2ext[i]];
    I->coff[i + 1] = I->coff[i] + I->cnne[i];
  }
  I->cnl.resize(I->coff[n]);
  for (int i = 0; i < n; i++) {
    const int e = I->int2ext[i];
    for (int k = 0; k < I->cnne[i]; k++) {
      const int nbr = conntbl->neighl[e][k];
      if (nbr < 0 || nbr >= n) {
        errprint("agbnp3_new(): connection table entry %d of atom %d out of range.\n", nbr, e);
        delete inst;
        return AGBNP_ERR;
      }
      I->cnl[I->coff[i] + k] = I->ext2int[nbr];
    }
  }
  // radius types by exact equality (agbnp3_utils.c:808-838) and one table per
  // ordered type pair (agbnp3_utils.c:840-883)
  I->rtype.resize(n);
  for (int i = 0; i < n; i++) {
    int found = -1;
    for (int t = 0; t < I->ntypes; t++)
      if (fabsf(I->R[i] - I->radii[t]) < FLT_MIN) { found = t; break; }
    if (found < 0) {
      found = I->ntypes++;
      I->radii.push_back(I->R[i]);
    }
    I->rtype[i] = found;
  }
  const int nt = I->ntypes;
  I->ty.assign((size_t)nt * nt * kTblN, 0.f);
  I->ty2.assign((size_t)nt * nt * kTblN, 0.f);
  for (int a = 0; a < nt; a++)
    for (int b = 0; b < nt; b++) {
      const float c = kRadInc;
      const float ratio = (I->radii[a] - c) / I->radii[b];
      const size_t t = (size_t)(a * nt + b) * kTblN;
      build_table(ratio, &I->ty[t], &I->ty2[t], I->tdx, I->tdxinv);
    }
  build_water_sites(I);
  if (build_pack(inst->p, {I}, 0) != AGBNP_OK) {
    free_pack(inst->p);
    delete inst;
    return AGBNP_ERR;
  }
  // lowest free slot (agbnp3.c:144-170)
  int slot = 0;
  while (slot < (int)g_slots.size() && g_slots[slot]) slot++;
  if (slot == (int)g_slots.size()) g_slots.push_back(nullptr);
  g_slots[slot] = inst;
  *tag = slot;
  return AGBNP_OK;
}

int agbnp3_delete(int tag) {
  std::lock_guard<std::mutex> lk(g_mutex);
  Instance *I = get_instance(tag, "agbnp3_delete()");
  if (!I) return AGBNP_ERR;
  free_pack(I->p);
  delete I;
  g_slots[tag] = nullptr;
  return AGBNP_OK;
}

int agbnp_initialize(void) { return agbnp3_initialize(); }
void agbnp_terminate(void) { agbnp3_terminate(); }
int agbnp_delete(int tag) { return agbnp3_delete(tag); }

int agbnp3_set_options(int tag, int options) {
  Instance *I = get_instance(tag, "agbnp3_set_options()");
  if (!I) return AGBNP_ERR;
  if ((I->p.options ^ options) & ~AGBNP3_OPT_TIMING) drop_graph(I->p);
  I->p.options = options;
  return AGBNP_OK;
}

int agbnp3_ener_device(int tag, const double *x, const double *y, const double *z, double *sp, double *br,
                       double *surf_area, double *dgbdr, double *dvwdr, double *decav, double *dehb,
                       double *energies) {
  Instance *I = get_instance(tag, "agbnp3_ener_device()");
  if (!I) return AGBNP_ERR;
  if (I->m.ws_error_atom >= 0) {
    errprint("agbnp3_create_ws_atoms(): error in agbnp3_create_ws_atoms_trigonal_oop(): atom %d needs 3 bonds.\n",
             I->m.int2ext[I->m.ws_error_atom]);
    errprint("agbnp3_ener(): error in agbnp3_total_energy().\n");
    return AGBNP_ERR;
  }
  return run_pipeline(I->p, x, y, z, sp, br, surf_area, dgbdr, dvwdr, decav, dehb, energies, false);
}

int agbnp3_ener_static(int tag, const double *x, const double *y, const double *z, double *sp, double *br,
                       double *surf_area, double *dgbdr, double *dvwdr, double *decav, double *dehb,
                       double *energies) {
  Instance *I = get_instance(tag, "agbnp3_ener_static()");
  if (!I) return AGBNP_ERR;
  if (I->m.ws_error_atom >= 0) {
    errprint("agbnp3_create_ws_atoms(): error in agbnp3_create_ws_atoms_trigonal_oop(): atom %d needs 3 bonds.\n",
             I->m.int2ext[I->m.ws_error_atom]);
    errprint("agbnp3_ener(): error in agbnp3_total_energy().\n");
    return AGBNP_ERR;
  }
  Pack &P = I->p;
  if (P.d.sg_on) {
    errprint("agbnp3_ener_static(): tag %d has a surrogate attached (its buffers are the instance's own; "
             "use agbnp3_ener_device).\n", tag);
    return AGBNP_ERR;
  }
  int dev = -1;
  HIPCHK(hipGetDevice(&dev));
  if (dev != P.device) {
    errprint("agbnp3_ener_static(): tag %d lives on device %d, the current device is %d.\n", tag, P.device, dev);
    return AGBNP_ERR;
  }
  char *base = nullptr;
  if (scratch_base(dev, &base) != AGBNP_OK) return AGBNP_ERR;
  Dev d = P.d;
  const size_t need = carve_call_state(d, nullptr, P.n, P.nh, P.nsys, d.nws, d.nablk, P.ntile, P.cap, d.nchain_items,
                                       P.call_nsplit(), P.call_ndpart());
  if (need > (size_t)AGBNP3_STATIC_SCRATCH_BYTES) {
    errprint("agbnp3_ener_static(): tag %d (%d atoms) needs %zu bytes of per-call state; the static scratch "
             "holds %zu (use agbnp3_ener_device).\n", tag, P.n, need, (size_t)AGBNP3_STATIC_SCRATCH_BYTES);
    return AGBNP_ERR;
  }
  carve_call_state(d, base, P.n, P.nh, P.nsys, d.nws, d.nablk, P.ntile, P.cap, d.nchain_items, P.call_nsplit(),
                                       P.call_ndpart());
  d.hstat = nullptr;
  // no per-kernel timing events here (creating them allocates)
  const int saved = P.options;
  P.options &= ~AGBNP3_OPT_TIMING;
  const int rc = run_pipeline_on(P, d, x, y, z, sp, br, surf_area, dgbdr, dvwdr, decav, dehb, energies, false);
  P.options = saved;
  return rc;
}

int agbnp3_sync(int tag) {
  Instance *I = get_instance(tag, "agbnp3_sync()");
  if (!I) return AGBNP_ERR;
  return pack_sync(I->p, "agbnp3_sync()");
}

void *agbnp3_stream(int tag) {
  Instance *I = get_instance(tag, "agbnp3_stream()");
  return I ? (void *)I->p.stream : nullptr;
}

int agbnp3_ener(int tag, int init, float_i *x, float_i *y, float_i *z, float_i *sp, float_i *br,
                float_i *mol_volume, float_i *surf_area, float_i *egb, float_i (*dgbdr)[3], float_i *evdw,
                float_i *ecorr_vdw, float_i (*dvwdr)[3], float_i *ecav, float_i *ecorr_cav, float_i (*decav)[3],
                float_i *ehb, float_i (*dehb)[3]) {
  (void)init;
  Instance *I = get_instance(tag, "agbnp3_agb_energy()");
  if (!I) return AGBNP_ERR;
  if (I->m.ws_error_atom >= 0) {
    errprint("agbnp3_create_ws_atoms(): error in agbnp3_create_ws_atoms_trigonal_oop(): atom %d needs 3 bonds.\n",
             I->m.int2ext[I->m.ws_error_atom]);
    errprint("agbnp3_ener(): error in agbnp3_total_energy().\n");
    return AGBNP_ERR;
  }
  const size_t n = I->m.natoms;
  // float_i is double, or float in the SINGLE_PREC_INTERFACE build of the
  // library (agbnp3.h); the engine's boundary arrays are double either way
  std::vector<double> xin, yin, zin;
  const double *xd = as_double(x, n, xin), *yd = as_double(y, n, yin), *zd = as_double(z, n, zin);
  if (ensure_call_state(I->p, true) != AGBNP_OK) return AGBNP_ERR;
  double *h = I->p.hstage;    // outputs land at the start of the staging area
  if (pack_ener_host(I->p, xd, yd, zd, h, "agbnp3_ener()") != AGBNP_OK) {
    errprint("agbnp3_ener(): error in agbnp3_total_energy().\n");
    return AGBNP_ERR;
  }
  store(sp, h, n);
  store(br, h + n, n);
  store(surf_area, h + 2 * n, n);
  store(&dgbdr[0][0], h + 3 * n, 3 * n);
  store(&dvwdr[0][0], h + 6 * n, 3 * n);
  store(&decav[0][0], h + 9 * n, 3 * n);
  store(&dehb[0][0], h + 12 * n, 3 * n);
  const double *e = h + 15 * n;
  *egb = e[0];
  *evdw = e[1];
  *ecorr_vdw = e[2];
  *ecav = e[3];
  *ecorr_cav = e[4];
  *ehb = e[5];
  *mol_volume = e[6];
  return AGBNP_OK;
}

int agbnp3_q4_tables(int ntypes, const float *radii, float *y, float *y2, float *dx) {
  if (ntypes <= 0 || !radii) return AGBNP_ERR;
  float tdx = 0.f, tdxinv = 0.f;
  for (int a = 0; a < ntypes; a++)
    for (int b = 0; b < ntypes; b++) {
      const float c = kRadInc;
      const float ratio = (radii[a] - c) / radii[b];
      const size_t t = (size_t)(a * ntypes + b) * kTblN;
      std::vector<float> ty(kTblN), ty2(kTblN);
      build_table(ratio, ty.data(), ty2.data(), tdx, tdxinv);
      if (y) memcpy(y + t, ty.data(), sizeof(float) * kTblN);
      if (y2) memcpy(y2 + t, ty2.data(), sizeof(float) * kTblN);
    }
  if (dx) { dx[0] = tdx; dx[1] = tdxinv; }
  return AGBNP_OK;
}

// ------------------------------------------------------------ introspection
int agbnp3_natoms(int tag, int *natoms, int *nheavy) {
  Instance *I = get_instance(tag, "agbnp3_natoms()");
  if (!I) return AGBNP_ERR;
  if (natoms) *natoms = I->m.natoms;
  if (nheavy) *nheavy = I->m.nheavy;
  return AGBNP_OK;
}

int agbnp3_get_int2ext(int tag, int *int2ext) {
  Instance *I = get_instance(tag, "agbnp3_get_int2ext()");
  if (!I) return AGBNP_ERR;
  memcpy(int2ext, I->m.int2ext.data(), sizeof(int) * I->m.natoms);
  return AGBNP_OK;
}

int agbnp3_get_near_list(int tag, int *nne, int *nbr, int cap) {
  Instance *I = get_instance(tag, "agbnp3_get_near_list()");
  if (!I) return AGBNP_ERR;
  if (!I->p.call_block) {
    errprint("agbnp3_get_near_list(): no evaluation of tag %d has run yet.\n", tag);
    return AGBNP_ERR;
  }
  const int nh = I->m.nheavy, dc = I->p.d.cap;
  std::vector<int> hn(std::max(nh, 1)), hb((size_t)std::max(nh, 1) * dc);
  HIPCHK(hipStreamSynchronize(I->p.stream));
  HIPCHK(hipMemcpy(hn.data(), I->p.d.nne, sizeof(int) * nh, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(hb.data(), I->p.d.nbr, sizeof(int) * (size_t)nh * dc, hipMemcpyDeviceToHost));
  for (int i = 0; i < nh; i++) {
    if (nne) nne[i] = hn[i];
    if (nbr)
      for (int k = 0; k < hn[i] && k < cap; k++) nbr[(size_t)i * cap + k] = hb[(size_t)i * dc + k];
  }
  return AGBNP_OK;
}

int agbnp3_get_tables(int tag, float *y, float *y2, float *radii) {
  Instance *I = get_instance(tag, "agbnp3_get_tables()");
  if (!I) return AGBNP_ERR;
  if (y) memcpy(y, I->m.ty.data(), sizeof(float) * I->m.ty.size());
  if (y2) memcpy(y2, I->m.ty2.data(), sizeof(float) * I->m.ty2.size());
  if (radii) memcpy(radii, I->m.radii.data(), sizeof(float) * I->m.ntypes);
  return I->m.ntypes;
}

int agbnp3_get_internal(int tag, const char *name, double *out) {
  Instance *I = get_instance(tag, "agbnp3_get_internal()");
  if (!I) return AGBNP_ERR;
  if (!I->p.call_block) {
    errprint("agbnp3_get_internal(): no evaluation of tag %d has run yet.\n", tag);
    return AGBNP_ERR;
  }
  const Dev &d = I->p.d;
  const double *src = nullptr;
  struct { const char *n; const double *p; } tab[] = {
      {"volumep_raw", d.volumep_raw}, {"sa_raw", d.sa_raw}, {"sa_f", d.sa_f}, {"sp", d.sp}, {"spe", d.spe},
      {"psvol", d.psvol}, {"gammap", d.gammap}, {"beta", d.beta}, {"br", d.br}, {"brw", d.brw}, {"swf", d.swf},
      {"A", d.A}, {"q2ab", d.q2ab}, {"abrw", d.abrw}, {"deru", d.deru}, {"derv", d.derv}, {"derus", d.derus},
      {"dervs", d.dervs}, {"derh", d.derh}};
  for (auto &e : tab)
    if (!strcmp(e.n, name)) src = e.p;
  if (!src) {
    errprint("agbnp3_get_internal(): unknown array '%s'\n", name);
    return AGBNP_ERR;
  }
  HIPCHK(hipStreamSynchronize(I->p.stream));
  HIPCHK(hipMemcpy(out, src, sizeof(double) * I->m.natoms, hipMemcpyDeviceToHost));
  return AGBNP_OK;
}

int agbnp3_get_counts(int tag, long long *counts) {
  Instance *I = get_instance(tag, "agbnp3_get_counts()");
  if (!I) return AGBNP_ERR;
  unsigned long long c[kCounters];
  HIPCHK(hipStreamSynchronize(I->p.stream));
  HIPCHK(hipMemcpy(c, I->p.d.counters, sizeof(c), hipMemcpyDeviceToHost));
  counts[0] = counts[1] = 0;
  for (int k = 0; k < kCountSlots; k++) {
    counts[0] += (long long)c[kCountBase + 8 * k];
    counts[1] += (long long)c[kCountBase + 8 * k + 1];
  }
  counts[2] = I->m.nws;
  counts[3] = (long long)c[2];
  counts[4] = (long long)c[3];
  counts[5] = (long long)(c[4] + c[6]);
  counts[6] = (long long)(c[4] + c[7]);
  return AGBNP_OK;
}

int agbnp3_get_routes(int tag, int *routes) {
  Instance *I = get_instance(tag, "agbnp3_get_routes()");
  if (!I) return AGBNP_ERR;
  *routes = I->p.routes;
  return AGBNP_OK;
}

int agbnp3_kernel_times(int tag, float *ms, int nmax, char *names, int names_len) {
  Instance *I = get_instance(tag, "agbnp3_kernel_times()");
  if (!I) return AGBNP_ERR;
  return pack_kernel_times(I->p, ms, nmax, names, names_len);
}

int agbnp3_get_tuning(int tag, int *params, int nparams) {
  Instance *I = get_instance(tag, "agbnp3_get_tuning()");
  if (!I || nparams < TUNE_COUNT) return AGBNP_ERR;
  tuning_to_params(I->p, params);
  return AGBNP_OK;
}

int agbnp3_set_tuning(int tag, const int *params, int nparams) {
  Instance *I = get_instance(tag, "agbnp3_set_tuning()");
  if (!I || nparams < TUNE_COUNT) return AGBNP_ERR;
  return params_to_tuning(I->p, params);
}

int agbnp3_tune(int tag, const double *x, const double *y, const double *z, int reps, char *report, int report_len) {
  Instance *I = get_instance(tag, "agbnp3_tune()");
  if (!I) return AGBNP_ERR;
  return pack_tune(I->p, x, y, z, reps, report, report_len);
}

int agbnp3_tune_table_save(const char *path) {
  FILE *f = path ? fopen(path, "w") : nullptr;
  if (!f) {
    errprint("agbnp3_tune_table_save(): cannot write %s\n", path ? path : "(null)");
    return AGBNP_ERR;
  }
  std::lock_guard<std::mutex> lk(g_tune_mutex);
  fprintf(f, "# agbnp3 launch shapes: systems class, atoms class, rows desc_chunk chain_chunk desc_grid gb_grid "
             "chain_grid cap tree_grid\n");
  for (const auto &e : g_tune_table) {
    fprintf(f, "%d %d", e.first.first, e.first.second);
    for (int v : e.second) fprintf(f, " %d", v);
    fprintf(f, "\n");
  }
  fclose(f);
  return AGBNP_OK;
}

int agbnp3_tune_table_load(const char *path) {
  FILE *f = path ? fopen(path, "r") : nullptr;
  if (!f) {
    errprint("agbnp3_tune_table_load(): cannot read %s\n", path ? path : "(null)");
    return AGBNP_ERR;
  }
  std::map<std::pair<int, int>, std::vector<int>> t;
  char line[512];
  int rc = AGBNP_OK;
  while (fgets(line, sizeof(line), f)) {
    if (line[0] == '#' || line[0] == '\n') continue;
    int v[2 + TUNE_COUNT];
    int k = 0, off = 0, used = 0;
    while (k < 2 + TUNE_COUNT && sscanf(line + off, "%d%n", &v[k], &used) == 1) {
      off += used;
      k++;
    }
    if (k != 2 + TUNE_COUNT) {
      rc = AGBNP_ERR;
      break;
    }
    std::vector<int> p(v + 2, v + 2 + TUNE_COUNT);
    const int cap = p[TUNE_CAP];
    if ((p[TUNE_ROWS] != 64 && p[TUNE_ROWS] != 128 && p[TUNE_ROWS] != 256) || (cap != 64 && cap != 128 && cap != 256) ||
        p[TUNE_DESC_CHUNK] < 0 || (p[TUNE_DESC_CHUNK] % 256) || p[TUNE_DESC_GRID] < 0 || p[TUNE_GB_GRID] < 0 ||
        p[TUNE_CHAIN_GRID] < 0 || p[TUNE_TREE_GRID] < 0 ||
        (p[TUNE_CHAIN_CHUNK] != 0 && p[TUNE_CHAIN_CHUNK] != 64 && p[TUNE_CHAIN_CHUNK] != 128 &&
         p[TUNE_CHAIN_CHUNK] != 256)) {
      rc = AGBNP_ERR;
      break;
    }
    t[{v[0], v[1]}] = p;
  }
  fclose(f);
  if (rc != AGBNP_OK) {
    errprint("agbnp3_tune_table_load(): malformed line in %s\n", path);
    return AGBNP_ERR;
  }
  std::lock_guard<std::mutex> lk(g_tune_mutex);
  for (const auto &e : t) g_tune_table[e.first] = e.second;
  return AGBNP_OK;
}

int agbnp3_tune_table_clear(void) {
  std::lock_guard<std::mutex> lk(g_tune_mutex);
  g_tune_table.clear();
  return AGBNP_OK;
}

// ------------------------------------------------------------------ batches
int agbnp3_batch_new(int *batch, int ntags, const int *tags) {
  std::lock_guard<std::mutex> lk(g_mutex);
  if (!g_initialized) {
    errprint("agbnp3_batch_new(): agbnp library is not initialized.\n");
    return AGBNP_ERR;
  }
  if (!batch || ntags <= 0 || !tags) {
    errprint("agbnp3_batch_new(): invalid arguments.\n");
    return AGBNP_ERR;
  }
  std::vector<const Model *> ms;
  Batch *B = new Batch();
  int options = -1;
  for (int k = 0; k < ntags; k++) {
    Instance *I = get_instance(tags[k], "agbnp3_batch_new()");
    if (!I) {
      delete B;
      return AGBNP_ERR;
    }
    const int o = I->p.options & ~AGBNP3_OPT_TIMING;
    if (options >= 0 && o != options) {
      errprint("agbnp3_batch_new(): instances %d and %d have different options.\n", tags[0], tags[k]);
      delete B;
      return AGBNP_ERR;
    }
    options = o;
    ms.push_back(&I->m);
    B->tags.push_back(tags[k]);
    B->ws_error.push_back(I->m.ws_error_atom >= 0 ? I->m.int2ext[I->m.ws_error_atom] : -1);
  }
  if (build_pack(B->p, ms, options) != AGBNP_OK) {
    free_pack(B->p);
    delete B;
    return AGBNP_ERR;
  }
  int slot = 0;
  while (slot < (int)g_batches.size() && g_batches[slot]) slot++;
  if (slot == (int)g_batches.size()) g_batches.push_back(nullptr);
  g_batches[slot] = B;
  *batch = slot;
  return AGBNP_OK;
}

int agbnp3_batch_delete(int batch) {
  std::lock_guard<std::mutex> lk(g_mutex);
  Batch *B = get_batch(batch, "agbnp3_batch_delete()");
  if (!B) return AGBNP_ERR;
  free_pack(B->p);
  delete B;
  g_batches[batch] = nullptr;
  return AGBNP_OK;
}

int agbnp3_batch_offsets(int batch, int *nsys, int *offsets) {
  Batch *B = get_batch(batch, "agbnp3_batch_offsets()");
  if (!B) return AGBNP_ERR;
  if (nsys) *nsys = B->p.nsys;
  if (offsets) {
    for (int b = 0; b < B->p.nsys; b++) offsets[b] = B->p.sinfo[b].a0;
    offsets[B->p.nsys] = B->p.n;
  }
  return AGBNP_OK;
}

int agbnp3_batch_set_options(int batch, int options) {
  Batch *B = get_batch(batch, "agbnp3_batch_set_options()");
  if (!B) return AGBNP_ERR;
  if ((B->p.options ^ options) & ~AGBNP3_OPT_TIMING) drop_graph(B->p);
  B->p.options = options;
  return AGBNP_OK;
}

static int set_reuse(Pack &P, float skin, int every, const char *who) {
  if (!(skin >= 0.f) || skin > 4.f || every < 0) {
    errprint("%s: invalid skin %g or rebuild period %d.\n", who, skin, every);
    return AGBNP_ERR;
  }
  HIPCHK(hipStreamSynchronize(P.stream));
  if (skin > 0.f && !P.d.nbl_state) {     // the kept candidates: allocated once reuse is asked for
    const size_t nn = std::max(P.n, 1), nhh = std::max(P.nh, 1);
    if (dalloc(P.allocs, &P.d.cand_nne, nhh) || dalloc(P.allocs, &P.d.cand_nbr, nhh * kCandCap) ||
        dalloc(P.allocs, &P.d.ref_pos, nn) || dalloc(P.allocs, &P.d.nbl_state, 8))
      return AGBNP_ERR;
  }
  if (P.d.nbl_state) HIPCHK(hipMemset(P.d.nbl_state, 0, sizeof(int) * 8));
  P.skin = skin;
  P.reuse_every = every;
  drop_graph(P);
  return AGBNP_OK;
}

int agbnp3_set_nblist_reuse(int tag, float skin, int every) {
  Instance *I = get_instance(tag, "agbnp3_set_nblist_reuse()");
  if (!I) return AGBNP_ERR;
  return set_reuse(I->p, skin, every, "agbnp3_set_nblist_reuse()");
}

int agbnp3_nblist_rebuilds(int tag, int *calls, int *rebuilds) {
  Instance *I = get_instance(tag, "agbnp3_nblist_rebuilds()");
  if (!I) return AGBNP_ERR;
  int st[4] = {0, 0, 0, 0};
  HIPCHK(hipStreamSynchronize(I->p.stream));
  if (I->p.d.nbl_state) HIPCHK(hipMemcpy(st, I->p.d.nbl_state, sizeof(st), hipMemcpyDeviceToHost));
  if (calls) *calls = st[1];
  if (rebuilds) *rebuilds = st[3];
  return AGBNP_OK;
}

int agbnp3_batch_set_nblist_reuse(int batch, float skin, int every) {
  Batch *B = get_batch(batch, "agbnp3_batch_set_nblist_reuse()");
  if (!B) return AGBNP_ERR;
  return set_reuse(B->p, skin, every, "agbnp3_batch_set_nblist_reuse()");
}

static int batch_topology_ok(Batch *B, const char *who) {
  for (size_t k = 0; k < B->ws_error.size(); k++)
    if (B->ws_error[k] >= 0) {
      errprint("%s: instance %d: water-site topology error at atom %d (TRIGONAL_OOP needs 3 bonds).\n", who,
               B->tags[k], B->ws_error[k]);
      return 0;
    }
  return 1;
}

int agbnp3_batch_ener_device(int batch, const double *x, const double *y, const double *z, double *sp, double *br,
                             double *surf_area, double *dgbdr, double *dvwdr, double *decav, double *dehb,
                             double *energies) {
  Batch *B = get_batch(batch, "agbnp3_batch_ener_device()");
  if (!B || !batch_topology_ok(B, "agbnp3_batch_ener_device()")) return AGBNP_ERR;
  return run_pipeline(B->p, x, y, z, sp, br, surf_area, dgbdr, dvwdr, decav, dehb, energies, false);
}

int agbnp3_batch_ener(int batch, const double *x, const double *y, const double *z, double *out) {
  Batch *B = get_batch(batch, "agbnp3_batch_ener()");
  if (!B || !batch_topology_ok(B, "agbnp3_batch_ener()")) return AGBNP_ERR;
  return pack_ener_host(B->p, x, y, z, out, "agbnp3_batch_ener()");
}

int agbnp3_batch_sync(int batch) {
  Batch *B = get_batch(batch, "agbnp3_batch_sync()");
  if (!B) return AGBNP_ERR;
  return pack_sync(B->p, "agbnp3_batch_sync()");
}

void *agbnp3_batch_stream(int batch) {
  Batch *B = get_batch(batch, "agbnp3_batch_stream()");
  return B ? (void *)B->p.stream : nullptr;
}

int agbnp3_batch_graph_capture(int batch, const double *x, const double *y, const double *z, double *sp, double *br,
                               double *surf_area, double *dgbdr, double *dvwdr, double *decav, double *dehb,
                               double *energies) {
  Batch *B = get_batch(batch, "agbnp3_batch_graph_capture()");
  if (!B || !batch_topology_ok(B, "agbnp3_batch_graph_capture()")) return AGBNP_ERR;
  return pack_capture(B->p, x, y, z, sp, br, surf_area, dgbdr, dvwdr, decav, dehb, energies);
}

int agbnp3_batch_graph_launch(int batch) {
  Batch *B = get_batch(batch, "agbnp3_batch_graph_launch()");
  if (!B) return AGBNP_ERR;
  if (!B->p.gexec) {
    errprint("agbnp3_batch_graph_launch(): no captured graph (capture again after a change of shape or options).\n");
    return AGBNP_ERR;
  }
  HIPCHK(hipGraphLaunch(B->p.gexec, B->p.stream));
  B->p.host_status = true;
  return AGBNP_OK;
}

int agbnp3_batch_kernel_times(int batch, float *ms, int nmax, char *names, int names_len) {
  Batch *B = get_batch(batch, "agbnp3_batch_kernel_times()");
  if (!B) return AGBNP_ERR;
  return pack_kernel_times(B->p, ms, nmax, names, names_len);
}

int agbnp3_batch_get_tuning(int batch, int *params, int nparams) {
  Batch *B = get_batch(batch, "agbnp3_batch_get_tuning()");
  if (!B || nparams < TUNE_COUNT) return AGBNP_ERR;
  tuning_to_params(B->p, params);
  return AGBNP_OK;
}

int agbnp3_batch_set_tuning(int batch, const int *params, int nparams) {
  Batch *B = get_batch(batch, "agbnp3_batch_set_tuning()");
  if (!B || nparams < TUNE_COUNT) return AGBNP_ERR;
  return params_to_tuning(B->p, params);
}

int agbnp3_batch_tune(int batch, const double *x, const double *y, const double *z, int reps, char *report,
                      int report_len) {
  Batch *B = get_batch(batch, "agbnp3_batch_tune()");
  if (!B || !batch_topology_ok(B, "agbnp3_batch_tune()")) return AGBNP_ERR;
  return pack_tune(B->p, x, y, z, reps, report, report_len);
}

// ---------------------------------------------------------------- surrogate
static SgHost *get_model(int id, const char *who) {
  if (id < 0 || id >= (int)g_models.size() || !g_models[id]) {
    errprint("%s: invalid surrogate model %d.\n", who, id);
    return nullptr;
  }
  return g_models[id];
}


static int sg_repack(SgHost *M) {
  launch_sg_pack(M->p, M->w1, M->w2, M->w3, M->wt1, M->wt2, M->wt3, M->stream);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(M->stream));
  return AGBNP_OK;
}

int agbnp3_sg_new(int *model, unsigned long long seed) {
  std::lock_guard<std::mutex> lk(g_mutex);
  if (!g_initialized) {
    errprint("agbnp3_sg_new(): agbnp library is not initialized.\n");
    return AGBNP_ERR;
  }
  if (prepare_surrogate() != hipSuccess) {
    errprint("agbnp3_sg_new(): the MLP kernels need %zu bytes of LDS per workgroup.\n", sg_mlp_lds());
    return AGBNP_ERR;
  }
  SgHost *M = new SgHost();
  auto &L = M->allocs;
  if (dalloc(L, &M->p, kSgNParam) || dalloc(L, &M->g, kSgNParam) || dalloc(L, &M->m, kSgNParam) ||
      dalloc(L, &M->v, kSgNParam) || dalloc(L, &M->loss, 1 << 16) || dalloc(L, &M->w1, kSgKPad * kSgHid) ||
      dalloc(L, &M->wt1, kSgKPad * kSgHid) || dalloc(L, &M->w2, kSgHid * kSgHid) ||
      dalloc(L, &M->wt2, kSgHid * kSgHid) || dalloc(L, &M->w3, kSgHid * kSgHid) ||
      dalloc(L, &M->wt3, kSgHid * kSgHid) || dalloc(L, &M->norm, 4 * kSgNFeat)) {
    sg_free(M);
    return AGBNP_ERR;
  }
  if (hipStreamCreateWithFlags(&M->stream, hipStreamNonBlocking) != hipSuccess) {
    sg_free(M);
    return AGBNP_ERR;
  }
  // Glorot-uniform weights, zero biases; identity normalisation, open window
  std::mt19937_64 rng(seed);
  std::vector<float> p(kSgNParam, 0.f);
  auto fill = [&](int off, int fin, int fout) {
    const float a = sqrtf(6.0f / (float)(fin + fout));
    std::uniform_real_distribution<float> u(-a, a);
    for (int k = 0; k < fin * fout; k++) p[off + k] = u(rng);
  };
  fill(kSgOffW1, kSgNFeat, kSgHid);
  fill(kSgOffW2, kSgHid, kSgHid);
  fill(kSgOffW3, kSgHid, kSgHid);
  fill(kSgOffW4, kSgHid, 1);
  std::vector<float> norm(4 * kSgNFeat);
  for (int k = 0; k < kSgNFeat; k++) {
    norm[k] = 0.f;
    norm[kSgNFeat + k] = 1.f;
    norm[2 * kSgNFeat + k] = -INFINITY;
    norm[3 * kSgNFeat + k] = INFINITY;
  }
  if (hipMemcpy(M->p, p.data(), sizeof(float) * kSgNParam, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(M->norm, norm.data(), sizeof(float) * norm.size(), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(M->m, 0, sizeof(float) * kSgNParam) != hipSuccess ||
      hipMemset(M->v, 0, sizeof(float) * kSgNParam) != hipSuccess || sg_repack(M) != AGBNP_OK) {
    sg_free(M);
    return AGBNP_ERR;
  }
  int slot = 0;
  while (slot < (int)g_models.size() && g_models[slot]) slot++;
  if (slot == (int)g_models.size()) g_models.push_back(nullptr);
  g_models[slot] = M;
  *model = slot;
  return AGBNP_OK;
}

int agbnp3_sg_delete(int model) {
  std::lock_guard<std::mutex> lk(g_mutex);
  SgHost *M = get_model(model, "agbnp3_sg_delete()");
  if (!M) return AGBNP_ERR;
  for (Instance *I : g_slots)
    if (I && I->p.sg_model == model) { I->p.d.sg_on = 0; I->p.sg_model = -1; drop_graph(I->p); }
  for (Batch *B : g_batches)
    if (B && B->p.sg_model == model) { B->p.d.sg_on = 0; B->p.sg_model = -1; drop_graph(B->p); }
  sg_free(M);
  g_models[model] = nullptr;
  return AGBNP_OK;
}

// export / import: params (kSgNParam), xmu, xsd_inv, xlo, xhi (kSgNFeat each), ymu, ysd
int agbnp3_sg_size(void) { return kSgNParam + 4 * kSgNFeat + 2; }

int agbnp3_sg_get_params(int model, float *out, int n) {
  SgHost *M = get_model(model, "agbnp3_sg_get_params()");
  if (!M || n < agbnp3_sg_size()) return AGBNP_ERR;
  HIPCHK(hipStreamSynchronize(M->stream));
  HIPCHK(hipMemcpy(out, M->p, sizeof(float) * kSgNParam, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(out + kSgNParam, M->norm, sizeof(float) * 4 * kSgNFeat, hipMemcpyDeviceToHost));
  out[kSgNParam + 4 * kSgNFeat] = M->ymu;
  out[kSgNParam + 4 * kSgNFeat + 1] = M->ysd;
  return AGBNP_OK;
}

static void sg_refresh_attached(int model) {
  SgHost *M = g_models[model];
  for (Instance *I : g_slots)
    if (I && I->p.sg_model == model) { I->p.d.sg = M->view(); drop_graph(I->p); }
  for (Batch *B : g_batches)
    if (B && B->p.sg_model == model) { B->p.d.sg = M->view(); drop_graph(B->p); }
}

int agbnp3_sg_set_params(int model, const float *in, int n) {
  SgHost *M = get_model(model, "agbnp3_sg_set_params()");
  if (!M || n < agbnp3_sg_size()) return AGBNP_ERR;
  HIPCHK(hipStreamSynchronize(M->stream));
  HIPCHK(hipMemcpy(M->p, in, sizeof(float) * kSgNParam, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(M->norm, in + kSgNParam, sizeof(float) * 4 * kSgNFeat, hipMemcpyHostToDevice));
  M->ymu = in[kSgNParam + 4 * kSgNFeat];
  M->ysd = in[kSgNParam + 4 * kSgNFeat + 1];
  if (sg_repack(M) != AGBNP_OK) return AGBNP_ERR;
  sg_refresh_attached(model);
  return AGBNP_OK;
}

// surrogate on a pack: every = anchor period (plain call every `every`
// calls, 1 = always plain), 0 detaches
static int pack_sg_attach(Pack &P, int model, int every) {
  HIPCHK(hipStreamSynchronize(P.stream));
  Dev &d = P.d;
  drop_graph(P);
  if (every <= 0) {
    d.sg_on = 0;
    P.sg_model = -1;
    return AGBNP_OK;
  }
  SgHost *M = get_model(model, "agbnp3_sg_attach()");
  if (!M) return AGBNP_ERR;
  HIPCHK(prepare_surrogate());
  if (P.sg_allocs.empty()) {
    const size_t nn = std::max(P.n, 1);
    std::vector<int> flags(P.nsys, 1);
    std::vector<int2> rows;
    for (const SysInfo &S : P.sinfo)
      for (int a = S.a0; a < S.a0 + S.n; a += kSgBlk) rows.push_back(make_int2(a, std::min(a + kSgBlk, S.a0 + S.n)));
    auto &L = P.sg_allocs;
    const size_t ns = std::max(P.nsys, 1);
    if (upload(L, &d.sys_sg, flags) || upload(L, &d.sg_rows, rows) || dalloc(L, &d.sg_state, 4 * ns) ||
        dalloc(L, &d.sg_any_plain, 1) || dalloc(L, &d.sg_F, 64 * nn) || dalloc(L, &d.sg_X, (size_t)kSgKPad * nn) ||
        dalloc(L, &d.sg_s, nn) || dalloc(L, &d.sg_dsdF, 4 * kSgRow * nn) || dalloc(L, &d.sg_target, nn) ||
        dalloc(L, &d.sg_c, nn) || dalloc(L, &d.sg_delta, nn) || dalloc(L, &d.sg_err, ns) ||
        dalloc(L, &d.sg_nbr, rows.size() * kSgNbrCap * kSgBlk) || dalloc(L, &d.sg_nn, nn) ||
        dalloc(L, &d.sg_ref, nn) || dalloc(L, &d.sg_nbl, 4 * ns) || dalloc(L, &d.sg_grid_p, ns) ||
        dalloc(L, &d.sg_cstart, ns * (kMaxCells + 1)) || dalloc(L, &d.sg_catoms, nn) || dalloc(L, &d.sg_ctmp, nn) ||
        dalloc(L, &d.sg_slot, nn) || dalloc(L, &d.sg_spos, nn) || dalloc(L, &d.sg_sgam, nn) || dalloc(L, &d.sg_sw, nn) ||
        dalloc(L, &d.sg_oor, nn) || dalloc(L, &d.sg_count, 4 * ns))
      return AGBNP_ERR;
    d.nsg_rows = (int)rows.size();
    // the descriptor lists depend on the coordinates only: they outlive a
    // change of model (the guard compares against the positions they were
    // built from)
    HIPCHK(hipMemset(d.sg_nbl, 0, sizeof(int) * 4 * ns));
    // the pads of the ds/dF rows stay zero (calls write the 16 shells only)
    HIPCHK(hipMemset(d.sg_dsdF, 0, sizeof(float) * 4 * kSgRow * nn));
    HIPCHK(hipMemset(d.sg_oor, 0, sizeof(int) * nn));
  }
  HIPCHK(hipMemset(d.sg_state, 0, sizeof(int) * 4 * P.nsys));
  HIPCHK(hipMemset(d.sg_count, 0, sizeof(int) * 4 * P.nsys));
  HIPCHK(hipMemset(d.sg_c, 0, sizeof(double) * std::max(P.n, 1)));
  HIPCHK(hipMemset(d.sg_err, 0, sizeof(double) * P.nsys));
  int dev = 0, cu = 256;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) cu = prop.multiProcessorCount;
  d.sg_on = 1;
  d.sg_every = every;
  d.sg_grid = cu;
  d.sg = M->view();
  P.sg_model = model;
  return AGBNP_OK;
}

int agbnp3_sg_attach(int tag, int model, int every) {
  Instance *I = get_instance(tag, "agbnp3_sg_attach()");
  if (!I) return AGBNP_ERR;
  return pack_sg_attach(I->p, model, every);
}

int agbnp3_batch_sg_attach(int batch, int model, int every) {
  Batch *B = get_batch(batch, "agbnp3_batch_sg_attach()");
  if (!B) return AGBNP_ERR;
  return pack_sg_attach(B->p, model, every);
}

static int pack_sg_stats(Pack &P, double *err, int *mode) {
  if (!P.d.sg_on) {
    errprint("agbnp3_sg_stats(): no surrogate attached.\n");
    return AGBNP_ERR;
  }
  HIPCHK(hipStreamSynchronize(P.stream));
  if (err) HIPCHK(hipMemcpy(err, P.d.sg_err, sizeof(double) * P.nsys, hipMemcpyDeviceToHost));
  if (mode) {
    std::vector<int> st(4 * P.nsys);
    HIPCHK(hipMemcpy(st.data(), P.d.sg_state, sizeof(int) * st.size(), hipMemcpyDeviceToHost));
    for (int b = 0; b < P.nsys; b++) mode[b] = st[4 * b + 2];
  }
  return AGBNP_OK;
}

int agbnp3_sg_stats(int tag, double *err, int *mode) {
  Instance *I = get_instance(tag, "agbnp3_sg_stats()");
  if (!I) return AGBNP_ERR;
  return pack_sg_stats(I->p, err, mode);
}

int agbnp3_batch_sg_stats(int batch, double *err, int *mode) {
  Batch *B = get_batch(batch, "agbnp3_batch_sg_stats()");
  if (!B) return AGBNP_ERR;
  return pack_sg_stats(B->p, err, mode);
}

static int pack_sg_lists(Pack &P, int *builds, int *overflow) {
  if (P.sg_allocs.empty()) {
    errprint("agbnp3_sg_lists(): no surrogate was attached.\n");
    return AGBNP_ERR;
  }
  HIPCHK(hipStreamSynchronize(P.stream));
  std::vector<int> st(4 * P.nsys);
  HIPCHK(hipMemcpy(st.data(), P.d.sg_nbl, sizeof(int) * st.size(), hipMemcpyDeviceToHost));
  for (int b = 0; b < P.nsys; b++) {
    if (builds) builds[b] = st[4 * b + 2];
    if (overflow) overflow[b] = st[4 * b + 3];
  }
  return AGBNP_OK;
}

// per system: calls in each mode (plain, surrogate, surrogate with plain
// out-of-window atoms) since the model was attached
static int pack_sg_modes(Pack &P, int *counts) {
  if (!P.d.sg_on) {
    errprint("agbnp3_sg_modes(): no surrogate attached.\n");
    return AGBNP_ERR;
  }
  HIPCHK(hipStreamSynchronize(P.stream));
  std::vector<int> c(4 * P.nsys);
  HIPCHK(hipMemcpy(c.data(), P.d.sg_count, sizeof(int) * c.size(), hipMemcpyDeviceToHost));
  for (int b = 0; b < P.nsys; b++)
    for (int m = 0; m < 3; m++) counts[3 * b + m] = c[4 * b + m];
  return AGBNP_OK;
}

int agbnp3_sg_modes(int tag, int *counts) {
  Instance *I = get_instance(tag, "agbnp3_sg_modes()");
  if (!I || !counts) return AGBNP_ERR;
  return pack_sg_modes(I->p, counts);
}

int agbnp3_batch_sg_modes(int batch, int *counts) {
  Batch *B = get_batch(batch, "agbnp3_batch_sg_modes()");
  if (!B || !counts) return AGBNP_ERR;
  return pack_sg_modes(B->p, counts);
}

int agbnp3_sg_lists(int tag, int *builds, int *overflow) {
  Instance *I = get_instance(tag, "agbnp3_sg_lists()");
  if (!I) return AGBNP_ERR;
  return pack_sg_lists(I->p, builds, overflow);
}

int agbnp3_batch_sg_lists(int batch, int *builds, int *overflow) {
  Batch *B = get_batch(batch, "agbnp3_batch_sg_lists()");
  if (!B) return AGBNP_ERR;
  return pack_sg_lists(B->p, builds, overflow);
}

// training set: plain evaluations of a batch at device coordinates x, y, z
int agbnp3_sg_reserve(int model, int natoms) {
  SgHost *M = get_model(model, "agbnp3_sg_reserve()");
  if (!M || natoms <= 0) return AGBNP_ERR;
  if (natoms <= M->cap) return AGBNP_OK;
  HIPCHK(hipStreamSynchronize(M->stream));
  float *F = nullptr, *t = nullptr;
  if (hipMalloc(&F, sizeof(float) * (size_t)natoms * kSgNFeat) != hipSuccess ||
      hipMalloc(&t, sizeof(float) * (size_t)natoms) != hipSuccess) {
    if (F) (void)hipFree(F);
    errprint("agbnp3_sg_reserve(): cannot allocate a training set of %d atoms.\n", natoms);
    return AGBNP_ERR;
  }
  if (M->count) {
    HIPCHK(hipMemcpy(F, M->F, sizeof(float) * (size_t)M->count * kSgNFeat, hipMemcpyDeviceToDevice));
    HIPCHK(hipMemcpy(t, M->target, sizeof(float) * (size_t)M->count, hipMemcpyDeviceToDevice));
  }
  if (M->F) { (void)hipFree(M->F); (void)hipFree(M->target); }
  M->F = F;
  M->target = t;
  M->cap = natoms;
  return AGBNP_OK;
}

int agbnp3_batch_sg_collect(int batch, int model, const double *x, const double *y, const double *z) {
  Batch *B = get_batch(batch, "agbnp3_batch_sg_collect()");
  SgHost *M = get_model(model, "agbnp3_batch_sg_collect()");
  if (!B || !M || !batch_topology_ok(B, "agbnp3_batch_sg_collect()")) return AGBNP_ERR;
  Pack &P = B->p;
  if (M->count + P.n > M->cap && agbnp3_sg_reserve(model, std::max(2 * M->cap, M->count + P.n)) != AGBNP_OK)
    return AGBNP_ERR;
  const int keep_model = P.sg_model, keep_every = P.d.sg_every, keep_on = P.d.sg_on;
  if (pack_sg_attach(P, model, 1) != AGBNP_OK) return AGBNP_ERR;      // plain calls with descriptors
  if (ensure_call_state(P) != AGBNP_OK) return AGBNP_ERR;
  const size_t n = P.n;
  double *o = P.dout;
  int rc = run_pipeline(P, x, y, z, o, o + n, o + 2 * n, o + 3 * n, o + 6 * n, o + 9 * n, o + 12 * n, o + 15 * n,
                        false);
  if (rc == AGBNP_OK) rc = pack_sync(P, "agbnp3_batch_sg_collect()");
  if (rc == AGBNP_OK) {
    std::vector<int> nbl(4 * P.nsys);
    HIPCHK(hipMemcpy(nbl.data(), P.d.sg_nbl, sizeof(int) * nbl.size(), hipMemcpyDeviceToHost));
    for (int b = 0; b < P.nsys && rc == AGBNP_OK; b++)
      if (nbl[4 * b + 3]) {
        errprint("agbnp3_batch_sg_collect(): system %d has atoms with more than %d neighbours within %.1f A.\n", b,
                 kSgNbrCap, (double)(kSgCut + kSgSkin));
        rc = AGBNP_ERR;
      }
  }
  if (rc == AGBNP_OK) {
    launch_sg_append(P.d, M->F, M->target, M->count, P.stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(P.stream));
    M->count += P.n;
    for (int a = 0; a < P.n; a++) M->keys.push_back((P.uid << 32) | (unsigned long long)a);
  }
  if (keep_on) pack_sg_attach(P, keep_model, keep_every);
  else pack_sg_attach(P, -1, 0);
  return rc;
}

int agbnp3_sg_dataset(int model, int *count, float *F, float *target) {
  SgHost *M = get_model(model, "agbnp3_sg_dataset()");
  if (!M) return AGBNP_ERR;
  if (count) *count = M->count;
  HIPCHK(hipStreamSynchronize(M->stream));
  if (F && M->count) HIPCHK(hipMemcpy(F, M->F, sizeof(float) * (size_t)M->count * kSgNFeat, hipMemcpyDeviceToHost));
  if (target && M->count) HIPCHK(hipMemcpy(target, M->target, sizeof(float) * M->count, hipMemcpyDeviceToHost));
  return AGBNP_OK;
}

// normalisation (mean / standard deviation per feature and of the target),
// the training window (observed range widened by `margin` of its width on
// each side), and the shuffled, normalised bf16 training matrix
int agbnp3_sg_fit(int model, float margin, unsigned long long seed) {
  SgHost *M = get_model(model, "agbnp3_sg_fit()");
  if (!M || M->count < 2) {
    errprint("agbnp3_sg_fit(): no training set.\n");
    return AGBNP_ERR;
  }
  const int N = M->count;
  std::vector<float> F((size_t)N * kSgNFeat), t(N);
  if (agbnp3_sg_dataset(model, nullptr, F.data(), t.data()) != AGBNP_OK) return AGBNP_ERR;
  std::vector<double> mu(kSgNFeat, 0.0), sd(kSgNFeat, 0.0);
  double ym = 0.0, ys = 0.0;
  for (int i = 0; i < N; i++) {
    for (int k = 0; k < kSgNFeat; k++) mu[k] += F[(size_t)i * kSgNFeat + k];
    ym += t[i];
  }
  for (int k = 0; k < kSgNFeat; k++) mu[k] /= N;
  ym /= N;
  for (int i = 0; i < N; i++) {
    for (int k = 0; k < kSgNFeat; k++) {
      const double e = F[(size_t)i * kSgNFeat + k] - mu[k];
      sd[k] += e * e;
    }
    ys += (t[i] - ym) * (t[i] - ym);
  }
  std::vector<float> norm(4 * kSgNFeat);
  for (int k = 0; k < kSgNFeat; k++) {
    const double s = std::max(sqrt(sd[k] / N), 1e-3);
    norm[k] = (float)mu[k];
    norm[kSgNFeat + k] = (float)(1.0 / s);
  }
  std::vector<float> lo(kSgNFeat, INFINITY), hi(kSgNFeat, -INFINITY);
  for (int i = 0; i < N; i++)
    for (int k = 0; k < kSgNFeat; k++) {
      const float v = (F[(size_t)i * kSgNFeat + k] - norm[k]) * norm[kSgNFeat + k];
      lo[k] = std::min(lo[k], v);
      hi[k] = std::max(hi[k], v);
    }
  // the window also keeps an absolute floor in raw units (half an atom in a
  // shell, 0.02 A of radius, 0.1 e of charge), so features that are rare in
  // the training set do not reject every small displacement
  for (int k = 0; k < kSgNFeat; k++) {
    const float floor_raw = k < 64 ? 0.5f : (k == 64 ? 0.02f : 0.1f);
    const float w = std::max(hi[k] - lo[k], 1e-3f);
    const float pad = margin * w + floor_raw * norm[kSgNFeat + k];
    norm[2 * kSgNFeat + k] = lo[k] - pad;
    norm[3 * kSgNFeat + k] = hi[k] + pad;
  }
  M->ymu = (float)ym;
  M->ysd = (float)std::max(sqrt(ys / N), 1e-6);
  // pairs: rows of the same atom of the same pack (collected from different
  // coordinates), taken in collection order two at a time; a row left over
  // pairs with the one before it, an atom seen once with itself
  std::vector<int> byk(N);
  for (int i = 0; i < N; i++) byk[i] = i;
  std::stable_sort(byk.begin(), byk.end(), [&](int a, int b) { return M->keys[a] < M->keys[b]; });
  std::vector<std::pair<int, int>> pairs;
  for (int g0 = 0; g0 < N;) {
    int g1 = g0 + 1;
    while (g1 < N && M->keys[byk[g1]] == M->keys[byk[g0]]) g1++;
    const int m = g1 - g0;
    for (int q = 0; q + 1 < m; q += 2) pairs.emplace_back(byk[g0 + q], byk[g0 + q + 1]);
    if (m % 2) pairs.emplace_back(byk[g1 - 1], m > 1 ? byk[g1 - 2] : byk[g1 - 1]);
    g0 = g1;
  }
  double dd = 0.0;
  long long nd = 0;
  for (const auto &pr : pairs)
    if (pr.first != pr.second) {
      const double e = (t[pr.first] - t[pr.second]) / M->ysd;
      dd += e * e;
      nd++;
    }
  M->dscale = nd && dd > 0.0 ? (float)(nd / dd) : 0.f;
  std::mt19937_64 rng(seed);
  if (nd) {
    std::shuffle(pairs.begin(), pairs.end(), rng);
    M->order.resize(2 * pairs.size());
    for (size_t q = 0; q < pairs.size(); q++) {
      M->order[2 * q] = pairs[q].first;
      M->order[2 * q + 1] = pairs[q].second;
    }
  } else {                            // every atom seen once: plain shuffled rows
    M->order.resize(N);
    for (int i = 0; i < N; i++) M->order[i] = i;
    std::shuffle(M->order.begin(), M->order.end(), rng);
  }
  const int NT = (int)M->order.size();
  std::vector<float> X((size_t)NT * kSgKPad, 0.f);
  std::vector<float> y(NT);
  for (int r = 0; r < NT; r++) {
    const int i = M->order[r];
    for (int k = 0; k < kSgNFeat; k++)
      X[(size_t)r * kSgKPad + k] = (F[(size_t)i * kSgNFeat + k] - norm[k]) * norm[kSgNFeat + k];
    y[r] = (float)((t[i] - ym) / M->ysd);
  }
  M->ntrain = NT;
  HIPCHK(hipStreamSynchronize(M->stream));
  for (void *q : M->tallocs) (void)hipFree(q);
  M->tallocs.clear();
  M->bcap = 0;
  if (upload(M->tallocs, (const float **)&M->X, X) || upload(M->tallocs, (const float **)&M->y, y))
    return AGBNP_ERR;
  HIPCHK(hipMemcpy(M->norm, norm.data(), sizeof(float) * norm.size(), hipMemcpyHostToDevice));
  sg_refresh_attached(model);
  return AGBNP_OK;
}

static int sg_batch_buffers(SgHost *M, int B) {
  if (B <= M->bcap) return AGBNP_OK;
  auto &L = M->tallocs;
  SgTrain &t = M->tb;
  if (dalloc(L, &t.A0, (size_t)kSgKPad * B) || dalloc(L, &t.A1, (size_t)kSgHid * B) ||
      dalloc(L, &t.A2, (size_t)kSgHid * B) || dalloc(L, &t.D1, (size_t)kSgHid * B) ||
      dalloc(L, &t.D2, (size_t)kSgHid * B) || dalloc(L, &t.D3, (size_t)kSgHid * B) ||
      dalloc(L, &t.A3, (size_t)kSgHid * B) || dalloc(L, &t.dy, (size_t)B) || dalloc(L, &t.err2, (size_t)B))
    return AGBNP_ERR;
  M->bcap = B;
  return AGBNP_OK;
}

// gradients of one batch of the shuffled training set (no update): tests
int agbnp3_sg_grads(int model, int r0, int B, float *grad, float *loss) {
  SgHost *M = get_model(model, "agbnp3_sg_grads()");
  if (!M || !M->X || B <= 0 || r0 < 0 || r0 % 2 || r0 + B > M->ntrain) return AGBNP_ERR;
  if (sg_batch_buffers(M, B) != AGBNP_OK) return AGBNP_ERR;
  M->tb.X = M->X;
  M->tb.y = M->y;
  M->tb.w_abs = M->w_abs;
  M->tb.w_diff = M->w_diff * M->dscale;
  launch_sg_train_step(M->view(), M->tb, r0, B, M->g, M->loss, 256, M->stream);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(M->stream));
  if (grad) HIPCHK(hipMemcpy(grad, M->g, sizeof(float) * kSgNParam, hipMemcpyDeviceToHost));
  if (loss) HIPCHK(hipMemcpy(loss, M->loss, sizeof(float), hipMemcpyDeviceToHost));
  return AGBNP_OK;
}

// Adam over `epochs` passes of mini-batches of B rows in a seeded random
// order; lr_e = lr decay^e; epoch_loss[e] = mean batch loss
int agbnp3_sg_train(int model, int epochs, int B, float lr, float decay, unsigned long long seed, float *epoch_loss) {
  SgHost *M = get_model(model, "agbnp3_sg_train()");
  if (!M || !M->X || B <= 0 || epochs <= 0) return AGBNP_ERR;
  const int nb = M->ntrain / B;
  if (nb <= 0 || nb > (1 << 16) || B % 2) {
    errprint("agbnp3_sg_train(): %d rows do not make batches of %d (an even number).\n", M->ntrain, B);
    return AGBNP_ERR;
  }
  if (sg_batch_buffers(M, B) != AGBNP_OK) return AGBNP_ERR;
  M->tb.X = M->X;
  M->tb.y = M->y;
  M->tb.w_abs = M->w_abs;
  M->tb.w_diff = M->w_diff * M->dscale;
  int dev = 0, cu = 256;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) cu = prop.multiProcessorCount;
  std::mt19937_64 rng(seed);
  std::vector<int> order(nb);
  std::vector<float> losses(nb);
  for (int e = 0; e < epochs; e++) {
    for (int b = 0; b < nb; b++) order[b] = b;
    std::shuffle(order.begin(), order.end(), rng);
    const float lre = lr * powf(decay, (float)e);
    for (int b = 0; b < nb; b++) {
      launch_sg_train_step(M->view(), M->tb, order[b] * B, B, M->g, M->loss + b, cu, M->stream);
      launch_sg_adam(M->p, M->g, M->m, M->v, lre, ++M->step, M->stream);
      launch_sg_pack(M->p, M->w1, M->w2, M->w3, M->wt1, M->wt2, M->wt3, M->stream);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(losses.data(), M->loss, sizeof(float) * nb, hipMemcpyDeviceToHost, M->stream));
    HIPCHK(hipStreamSynchronize(M->stream));
    double s = 0.0;
    for (float l : losses) s += l;
    if (epoch_loss) epoch_loss[e] = (float)(s / nb);
  }
  return AGBNP_OK;
}

int agbnp3_sg_set_loss(int model, float w_abs, float w_diff) {
  SgHost *M = get_model(model, "agbnp3_sg_set_loss()");
  if (!M || !(w_abs >= 0.f) || !(w_diff >= 0.f)) return AGBNP_ERR;
  M->w_abs = w_abs;
  M->w_diff = w_diff;
  return AGBNP_OK;
}

int agbnp3_sg_train_rows(int model, int *count, int *rows, float *diff_scale) {
  SgHost *M = get_model(model, "agbnp3_sg_train_rows()");
  if (!M) return AGBNP_ERR;
  if (count) *count = M->ntrain;
  if (rows) std::copy(M->order.begin(), M->order.end(), rows);
  if (diff_scale) *diff_scale = M->dscale;
  return AGBNP_OK;
}

// the MLP on raw descriptors F [n][66] (host): s [n], ds/dF [n][64]
int agbnp3_sg_infer(int model, const float *F, int n, float *s_out, float *dsdF) {
  SgHost *M = get_model(model, "agbnp3_sg_infer()");
  if (!M || n <= 0) return AGBNP_ERR;
  std::vector<float> norm(4 * kSgNFeat);
  HIPCHK(hipStreamSynchronize(M->stream));
  HIPCHK(hipMemcpy(norm.data(), M->norm, sizeof(float) * norm.size(), hipMemcpyDeviceToHost));
  std::vector<float> X((size_t)n * kSgKPad, 0.f);
  for (int i = 0; i < n; i++)
    for (int k = 0; k < kSgNFeat; k++)
      X[(size_t)i * kSgKPad + k] = (F[(size_t)i * kSgNFeat + k] - norm[k]) * norm[kSgNFeat + k];
  std::vector<void *> tmp;
  const float *dX = nullptr;
  float *ds = nullptr, *dd = nullptr;
  int rc = AGBNP_ERR;
  if (!upload(tmp, &dX, X) && !dalloc(tmp, &ds, (size_t)n) && !dalloc(tmp, &dd, (size_t)n * 64)) {
    launch_sg_infer(M->view(), dX, n, ds, dd, 256, M->stream);
    if (hipGetLastError() == hipSuccess && hipStreamSynchronize(M->stream) == hipSuccess &&
        hipMemcpy(s_out, ds, sizeof(float) * n, hipMemcpyDeviceToHost) == hipSuccess &&
        (!dsdF || hipMemcpy(dsdF, dd, sizeof(float) * (size_t)n * 64, hipMemcpyDeviceToHost) == hipSuccess))
      rc = AGBNP_OK;
  }
  for (void *q : tmp) (void)hipFree(q);
  return rc;
}

}  // extern "C"
