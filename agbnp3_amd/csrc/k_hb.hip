// Hydrogen-bond (water-site) term.
//
// One wavefront per site.  Its first lane places the site, a pseudo-atom of
// radius 1.4 A, and forms the Jacobians dpos[p][i][j] = d pos_i / d x_{parent
// p, j} of its geometry, one of the reference's eight (agbnp3.c:2014-3761),
// in the wave's LDS record.  Which atoms get which geometry is fixed by the
// topology and decided on the host when the instance is created.  (A launch
// of its own that wrote every site's 240-byte record to memory, one thread
// per HB-active atom, took 12 us at 2,000 atoms, its wave running all eight
// geometries in turn, and 16 us at 25,000.)
//
// Free volume: heavy atoms passing the FP32 test
// d2 < ((R + 1.4) * 1.6)^2 are collected from the cell grid and sorted by
// atom index; their Gaussian overlaps are evaluated lane-parallel, then taken
// in index order exactly as the reference does
// (agbnp3_ws_free_volumes_scalev_ps, kernels.c:2774-2934), every lane following
// the same walk: subtract spe * V' while the free volume exceeds 0.6 V_w.  By default the spe read is
// the previous overlap partner's (the reference's stale index, first one
// given by the previous site's last parent); AGBNP3_OPT_HB_FIXED uses the
// partner's own.  E_HB = sum khb s(V_free / V_w; 0.65, 1).
#include <float.h>

#include <type_traits>

#include "agb_common.h"
#include "agb_device.h"

namespace agb {

// --------------------------------------------------------------- 3-vectors
struct f3 {
  float x, y, z;
};
__device__ __forceinline__ f3 ld3(const float4 &p) { return {p.x, p.y, p.z}; }
__device__ __forceinline__ f3 operator-(f3 a, f3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ f3 operator+(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ f3 operator*(float s, f3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ float dot(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ f3 cross(f3 a, f3 b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float comp(f3 a, int k) { return k == 0 ? a.x : (k == 1 ? a.y : a.z); }
__device__ __forceinline__ f3 row3(const float M[3][3], int i) { return {M[i][0], M[i][1], M[i][2]}; }

// d u / d r of u = r/|r|: (I - u u^T)/|r|
__device__ __forceinline__ void unit_der(f3 u, float invr, float M[3][3]) {
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) M[i][j] = invr * ((i == j ? 1.f : 0.f) - comp(u, i) * comp(u, j));
}
__device__ __forceinline__ void mm3(const float A[3][3], const float B[3][3], float C[3][3]) {
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) C[i][j] = A[i][0] * B[0][j] + A[i][1] * B[1][j] + A[i][2] * B[2][j];
}
__device__ __forceinline__ f3 unit(f3 v, float &inv) {
  inv = 1.0f / sqrtf(dot(v, v));
  return inv * v;
}

__device__ __forceinline__ void site_init(WSite &w, f3 pos, float khb, int type, int np, int p0, int p1, int p2,
                                          int p3) {
  w.pos[0] = pos.x; w.pos[1] = pos.y; w.pos[2] = pos.z;
  w.khb = khb;
  w.type = type;
  w.nparents = np;
  w.parent[0] = p0; w.parent[1] = p1; w.parent[2] = p2; w.parent[3] = p3;
  for (int p = 0; p < 4; p++)
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) w.dpos[p][i][j] = 0.f;
}

// Site number `which` of HB-active atom `def`, into record w
__device__ void ws_place_site(const Dev &d, const WsDef &def, int which, WSite &w) {
  const float L = kHbLength;
  const int A = def.atom;
  const f3 xa = ld3(d.pos[A]);
  const float khb = d.hbcorr_f[A];
  switch (def.kind) {
    case WS_POLARH: {     // agbnp3_place_wat_hydrogen (agbnp3.c:2098-2150)
      const int D = def.p[1];
      const f3 xd = ld3(d.pos[D]);
      float inv;
      const f3 u = unit(xa - xd, inv);
      site_init(w, xd + L * u, khb, 1, 2, A, D, -1, -1);
      const float c = L * inv;
      for (int i = 0; i < 3; i++)
        for (int j = 0; j < 3; j++) {
          const float m = c * ((i == j ? 1.f : 0.f) - comp(u, i) * comp(u, j));
          w.dpos[0][i][j] = m;
          w.dpos[1][i][j] = (i == j ? 1.f : 0.f) - m;
        }
      break;
    }
    case WS_TRIGONAL1:
    case WS_TRIGONAL_S: {   // agbnp3_place_wat_trigonal1 (agbnp3.c:2295-2366)
      const int R = def.p[1], R1 = def.p[2], R2 = def.p[3];
      const f3 xr = ld3(d.pos[R]);
      const int type = def.kind == WS_TRIGONAL1 ? 11 : 30;
      if (which < 2) {
        const int s = which;
        float inv;
        const f3 u = unit(ld3(d.pos[s == 0 ? R1 : R2]) - xr, inv);
        site_init(w, xa - L * u, khb, type, 4, A, R, R1, R2);
        const float c = L * inv;
        for (int i = 0; i < 3; i++) {
          w.dpos[0][i][i] = 1.f;
          for (int j = 0; j < 3; j++) {
            const float m = c * ((i == j ? 1.f : 0.f) - comp(u, i) * comp(u, j));
            w.dpos[1][i][j] = m;
            w.dpos[2 + s][i][j] = -m;
          }
        }
      }
      if (which >= 2) {   // agbnp3_place_wat_trigonal_s (agbnp3.c:2590-2697)
        const float cs = 0.5f, sn = 0.866025f;
        const f3 dx0 = xa - xr, dx1 = ld3(d.pos[R1]) - xr;
        float d0i, d2i;
        const f3 uin = unit(dx0, d0i);
        const f3 uout = unit(cross(dx1, dx0), d2i);
        float Din[3][3], Dout[3][3], t1[3][3], t2[3][3];
        unit_der(uin, d0i, Din);
        unit_der(uout, d2i, Dout);
        for (int i = 0; i < 3; i++) {
          const f3 a = cross(dx1, row3(Dout, i)), b = cross(dx0, row3(Dout, i));
          t1[i][0] = a.x; t1[i][1] = a.y; t1[i][2] = a.z;
          t2[i][0] = b.x; t2[i][1] = b.y; t2[i][2] = b.z;
        }
        {
          const float sg = which == 2 ? 1.f : -1.f;
          site_init(w, xa + L * (cs * uin + (sg * sn) * uout), khb, 30, 4, A, R, R1, R2);
          for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++) {
              const float win = L * cs * Din[i][j];
              const float w1 = -L * sn * t1[i][j], w2 = L * sn * t2[i][j];
              w.dpos[0][i][j] = win + sg * w1 + (i == j ? 1.f : 0.f);
              w.dpos[1][i][j] = -win - sg * (w1 + w2);
              w.dpos[2][i][j] = sg * w2;
            }
        }
      }
      break;
    }
    case WS_TRIGONAL_OOP: {   // agbnp3_place_wat_trigonal_oop (agbnp3.c:2815-2942)
      const int R1 = def.p[1], R2 = def.p[2], R3 = def.p[3];
      const float dd = L + 0.2f;
      const f3 x1 = ld3(d.pos[R1]);
      const f3 v1 = ld3(d.pos[R2]) - x1, v2 = ld3(d.pos[R3]) - x1;
      const f3 nraw = cross(v2, v1);
      const float nun = sqrtf(dot(nraw, nraw));
      const f3 nu = (1.0f / nun) * nraw;
      const float J1[3][3] = {{0.f, -v2.z, v2.y}, {v2.z, 0.f, -v2.x}, {-v2.y, v2.x, 0.f}};
      const float J2[3][3] = {{0.f, v1.z, -v1.y}, {-v1.z, 0.f, v1.x}, {v1.y, -v1.x, 0.f}};
      float P[3][3], M1[3][3], M2[3][3];
      for (int i = 0; i < 3; i++)
        for (int j = 0; j < 3; j++) P[i][j] = (i == j ? 1.f : 0.f) - comp(nu, i) * comp(nu, j);
      mm3(P, J1, M1);
      mm3(P, J2, M2);
      const float dn = dd / nun;
      {
        const float sg = which == 0 ? 1.f : -1.f;
        site_init(w, xa + (sg * dd) * nu, khb, 13, 4, A, R1, R2, R3);
        for (int i = 0; i < 3; i++)
          for (int j = 0; j < 3; j++) {
            w.dpos[0][i][j] = i == j ? 1.f : 0.f;
            w.dpos[2][i][j] = sg * dn * M1[i][j];
            w.dpos[3][i][j] = sg * dn * M2[i][j];
            w.dpos[1][i][j] = -(w.dpos[2][i][j] + w.dpos[3][i][j]);
          }
      }
      break;
    }
    case WS_TRIGONAL2:
    case WS_TETRAHEDRAL3: {   // agbnp3_place_wat_trigonal2 / _tetrahedral3 (agbnp3.c:3024-3090, 3476-3556)
      const int nr = def.kind == WS_TRIGONAL2 ? 2 : 3;
      f3 dk[3];
      float inv[3];
      f3 sum = {0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 3; k++) {
        if (k >= nr) break;
        dk[k] = unit(ld3(d.pos[def.p[1 + k]]) - xa, inv[k]);
        sum = sum + dk[k];
      }
      float iw;
      const f3 dw = unit(sum, iw);
      site_init(w, xa - L * dw, khb, nr == 2 ? 12 : 23, nr + 1, A, def.p[1], def.p[2], nr == 3 ? def.p[3] : -1);
      float Dw[3][3];
      unit_der(dw, iw, Dw);
      for (int i = 0; i < 3; i++) w.dpos[0][i][i] = 1.f;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        if (k >= nr) break;
        float Dk[3][3], M[3][3];
        unit_der(dk[k], inv[k], Dk);
        mm3(Dw, Dk, M);
        for (int i = 0; i < 3; i++)
          for (int j = 0; j < 3; j++) {
            w.dpos[1 + k][i][j] = -L * M[i][j];
            w.dpos[0][i][j] += L * M[i][j];
          }
      }
      break;
    }
    case WS_TETRAHEDRAL2: {   // agbnp3_place_wat_tetrahedral2 (agbnp3.c:3266-3390)
      const float cs = -0.577350269f, sn = 0.816496581f;
      const int R1 = def.p[1], R2 = def.p[2];
      const f3 r1 = ld3(d.pos[R1]) - xa, r2 = ld3(d.pos[R2]) - xa;
      float i1, i2, iin, iout;
      const f3 d1 = unit(r1, i1), d2 = unit(r2, i2);
      const f3 pin = unit(d1 + d2, iin);
      const f3 out = unit(cross(r2, r1), iout);
      float Dp[3][3], D1[3][3], D2[3][3], P1[3][3], P2[3][3], Do[3][3], t1[3][3], t2[3][3];
      unit_der(pin, iin, Dp);
      unit_der(d1, i1, D1);
      unit_der(d2, i2, D2);
      mm3(Dp, D1, P1);
      mm3(Dp, D2, P2);
      unit_der(out, iout, Do);
      for (int i = 0; i < 3; i++) {
        const f3 a = cross(row3(Do, i), r2), b = cross(r1, row3(Do, i));
        t1[i][0] = a.x; t1[i][1] = a.y; t1[i][2] = a.z;
        t2[i][0] = b.x; t2[i][1] = b.y; t2[i][2] = b.z;
      }
      {
        const float sg = which == 0 ? 1.f : -1.f;
        site_init(w, xa + L * (cs * pin + (sg * sn) * out), khb, 22, 3, A, R1, R2, -1);
        for (int i = 0; i < 3; i++)
          for (int j = 0; j < 3; j++) {
            const float a1 = L * cs * P1[i][j], a2 = L * cs * P2[i][j];
            const float b1 = L * sn * t1[i][j], b2 = L * sn * t2[i][j];
            w.dpos[1][i][j] = a1 + sg * b1;
            w.dpos[2][i][j] = a2 + sg * b2;
            w.dpos[0][i][j] = -(a1 + a2) - sg * (b1 + b2) + (i == j ? 1.f : 0.f);
          }
      }
      break;
    }
    case WS_TETRAHEDRAL1: {   // agbnp3_place_wat_tetrahedral1_one (agbnp3.c:3689-3761)
      const int R = def.p[1];
      const f3 xr = ld3(d.pos[R]);
      {
        const int s = which;
        const int Rk = def.p[2 + s];
        float inv;
        const f3 u = unit(ld3(d.pos[Rk]) - xr, inv);
        site_init(w, xa - L * u, khb, 21, 3, A, R, Rk, -1);
        const float c = L * inv;
        for (int i = 0; i < 3; i++) {
          w.dpos[0][i][i] = 1.f;
          for (int j = 0; j < 3; j++) {
            const float m = c * ((i == j ? 1.f : 0.f) - comp(u, i) * comp(u, j));
            w.dpos[1][i][j] = m;
            w.dpos[2][i][j] = -m;
          }
        }
      }
      break;
    }
  }
}

// ------------------------------------------------------------ free volume
// One wave per site, WAVES sites per block, candidate buffers of CAP atoms.
// The first pass (4 x 128) leaves the sites with more candidates than it
// holds (up to d.ws_cap1, 128 unless lowered for tests) for a second
// (1 x 1024), which takes them one per wave; the per-site arithmetic is the
// same in both, so results do not depend on which pass took a site.  A
// site with more than 1024 candidates fails the call.
constexpr int kWsWaves = 4;
constexpr int kWsCap = 128, kWsCapBig = 1024;
constexpr int kWsAhead = 4;

template <int WAVES, int CAP>
struct WsLds {
  int cj[WAVES][CAP];
  int cs[WAVES][CAP];        // sorted candidate atoms
  float cvp[WAVES][CAP];
  float cgw[WAVES][CAP][3];
  double cspe[WAVES][CAP];   // spe of the sorted candidates
  unsigned long long keep[WAVES][CAP / 64];   // which of them the walk took
  WSite rec[WAVES];
};

// what becomes of a site with more candidates than CAP: listed for the second
// launch, a failed call, or returned to the caller
enum : int { WS_LIST = 0, WS_FAIL = 1, WS_RETURN = 2 };

// The free volume of one site and its derivatives by one wave with the LDS of
// slot w (every wave of the block calls it together: it holds block barriers;
// a wave without a site, site >= nws, touches no LDS).  True when the site had
// more candidates than this pass holds (it then adds nothing).
template <int WAVES, int CAP, int MORE>
__device__ bool ws_free_site(const Dev &d, WsLds<WAVES, CAP> &L, int site, int w) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const bool active = site < d.nws;
  if (active && lane == 0) {
    const int2 ds = d.ws_site[site];
    ws_place_site(d, d.wsdef[ds.x], ds.y, L.rec[w]);
  }
  __syncthreads();
  // the fields every lane uses, in registers; the parents and Jacobians are
  // read from the record only by the lanes that project onto them
  const WSite *Wg = &L.rec[w];
  float wpos[3] = {0.f, 0.f, 0.f};
  float wkhb = 0.f;
  int wstale0 = -1, wnparents = 0, sys = 0;
  if (active) {
    wpos[0] = Wg->pos[0]; wpos[1] = Wg->pos[1]; wpos[2] = Wg->pos[2];
    wkhb = Wg->khb;
    wnparents = Wg->nparents;
    wstale0 = d.ws_stale0[site];
    sys = d.asys[Wg->parent[0]];
  }
  const GridParams g = d.grid[sys];
  const int *cstart = d.cell_start + (size_t)sys * (kMaxCells + 1);
  const float aw = kKFC / (kHbRadius * kHbRadius);
  int cnt = 0;
  if (active) {
    int cx, cy, cz;
    cell_coords(g, wpos[0], wpos[1], wpos[2], cx, cy, cz);
    // the stencil's candidates, kWsAhead steps of 64 in flight; sorted by atom
    // index below
    int start[9], off[9];
    const int total = stencil_segments(g, cstart, cx, cy, cz, start, off);
    for (int base = 0; base < total; base += 64 * kWsAhead) {
      int j[kWsAhead];
      float4 pj[kWsAhead];
#pragma unroll
      for (int u = 0; u < kWsAhead; u++) j[u] = d.cell_atoms[stencil_slot(start, off, min(base + 64 * u + lane, total - 1))];
#pragma unroll
      for (int u = 0; u < kWsAhead; u++) pj[u] = d.pos[j[u]];
#pragma unroll
      for (int u = 0; u < kWsAhead; u++) {
        if (base + 64 * u >= total) break;             // wave-uniform
        bool pass = false;
        if (base + 64 * u + lane < total) {
          const float ex = __fsub_rn(pj[u].x, wpos[0]), ey = __fsub_rn(pj[u].y, wpos[1]), ez = __fsub_rn(pj[u].z, wpos[2]);
          const float d2 = __fadd_rn(__fadd_rn(__fmul_rn(ex, ex), __fmul_rn(ey, ey)), __fmul_rn(ez, ez));
          const float t = __fmul_rn(__fadd_rn(pj[u].w, kHbRadius), kNbOffset);
          pass = d2 < __fmul_rn(t, t);
        }
        const unsigned long long m = __ballot(pass);
        if (pass) {
          const int slot = cnt + __popcll(m & ((1ull << lane) - 1ull));
          if (slot < CAP) L.cj[w][slot] = j[u];
        }
        cnt += __popcll(m);
      }
    }
  }
  // a site past these buffers adds nothing here
  bool mine = active, more = false;
  if (cnt > (MORE == WS_FAIL ? CAP : min(CAP, d.ws_cap1))) {
    if (MORE == WS_FAIL && lane == 0) atomicOr(d.status, ST_WS_OVERFLOW);
    if (MORE == WS_LIST && lane == 0) {
      const unsigned q = atomicAdd(&d.counters[kCountWs], 1ull);
      d.ws_ovf[q] = site;
    }
    more = true;
    mine = false;
    cnt = 0;
  }
  __syncthreads();
  // sort by atom index, evaluate overlaps lane-parallel
  for (int e = lane; e < cnt; e += 64) {
    const int je = L.cj[w][e];
    int rank = 0;
#pragma unroll 8
    for (int f = 0; f < cnt; f++) rank += L.cj[w][f] < je;
    L.cs[w][rank] = je;
  }
  __syncthreads();
  for (int e = lane; e < cnt; e += 64) {
    const int k = L.cs[w][e];
    const float4 pk = d.pos[k];
    const float ak = d.galpha[k];
    const float ex = pk.x - wpos[0], ey = pk.y - wpos[1], ez = pk.z - wpos[2];
    const float d2 = ex * ex + ey * ey + ez * ez;
    const float a12 = aw + ak, dinv = 1.0f / a12;
    const float p12 = kPFC * kPFC * __expf(-aw * ak * d2 * dinv);
    const float u = kPiF * dinv;
    const float V = p12 * u * sqrtf(u);
    float s, sp, spp;
    vol_switch(V, s, sp, spp);
    const float fp = s + V * sp;
    // offsets from the overlap centre c = (aw w + ak x_k) / (aw + ak) written
    // with the site-atom difference e = x_k - w (w - c = -ak e / a12,
    // x_k - c = aw e / a12): the absolute centre would carry the rounding of
    // its tens-of-Angstrom position
    const float e3[3] = {ex, ey, ez};
    const float gsc = 2.f * aw * ak * V * fp * dinv;
    L.cvp[w][e] = s * V;
    L.cspe[w][e] = d.spe[k];
#pragma unroll
    for (int q = 0; q < 3; q++) L.cgw[w][e][q] = gsc * e3[q];   // site side; the atom side is its negative
  }
  __syncthreads();
  const double vw = 4.0 / 3.0 * kPi * (double)kHbRadius * (double)kHbRadius * (double)kHbRadius;
  if (!mine) return more;                // (no barrier follows)
  // The reference's sequential walk with early stop (kernels.c:2818-2860), 64
  // candidates at a time: the terms spe V' in parallel (by default the spe of
  // the candidate taken before, the site's stale partner's first), then one
  // subtraction after the other in index order, each term read from its lane
  // into every lane.  (Walked by one lane out of LDS, a site's ~50 candidates
  // cost it more than everything else together.)
  double freev = vw;
  {
    const bool fixed = (d.options & 1) != 0;
    const double cutoff = (double)kHbSwA0 * vw;
    double stale = wstale0 >= 0 ? d.spe[wstale0] : 0.0;
    for (int base = 0; base < cnt; base += 64) {
      const int e = base + lane;
      const float vp = e < cnt ? L.cvp[w][e] : 0.f;
      const double spk = e < cnt ? L.cspe[w][e] : 0.0;
      const unsigned long long taken = __ballot(vp > 0.f);      // (as far as the walk goes)
      const unsigned long long below = taken & ((1ull << lane) - 1ull);
      const double before = __shfl(spk, below ? 63 - __clzll(below) : 0, 64);
      const double term = (fixed ? spk : (below ? before : stale)) * (double)vp;
      unsigned long long todo = taken, keep = 0ull;
      while (todo != 0ull && __ballot(freev > cutoff) != 0ull) {  // (the same in every lane)
        const int b = __builtin_ctzll(todo);
        todo &= todo - 1ull;
        keep |= 1ull << b;
        freev -= lane_value(term, b);
      }
      if (lane == 0) L.keep[w][base / 64] = keep;
      if (taken != 0ull) stale = lane_value(spk, 63 - __clzll(taken));
    }
  }
  wave_sync();
  const double spw = freev / vw;
  double fp = 0.0, sw;
  {
    const double xa = kHbSwA, xb = kHbSwB;
    if (spw > xb) sw = 1.0;
    else if (spw < xa) sw = 0.0;
    else {
      const double dd = 1.0 / (xb - xa), uu = (spw - xa) * dd, u2 = uu * uu;
      sw = u2 * uu * (10.0 - 15.0 * uu + 6.0 * u2);
      fp = dd * 30.0 * u2 * (1.0 - 2.0 * uu + u2);
    }
  }
  const double dhw = (double)wkhb * fp / vw;
  if (lane == 0) d.ws_part[site] = (double)wkhb * sw;
  double jw[3] = {0.0, 0.0, 0.0};
  for (int e = lane; e < cnt; e += 64) {
    if (!((L.keep[w][e / 64] >> lane) & 1ull)) continue;
    const int k = L.cs[w][e];
    const double spk = L.cspe[w][e];
#pragma unroll
    for (int q = 0; q < 3; q++) {
      fix_add(&d.acc_hb[3 * (size_t)k + q], spk * dhw * (double)L.cgw[w][e][q]);
      jw[q] += -dhw * spk * (double)L.cgw[w][e][q];
    }
    fix_add(&d.acc_derh[k], dhw / d.vols[k] * (double)L.cvp[w][e]);
  }
#pragma unroll
  for (int q = 0; q < 3; q++) jw[q] = wave_sum(jw[q]);
  // project the site force onto its parents: dpos^T jw (agbnp3_rtvec)
  if (lane < 3 * wnparents) {
    const int p = lane / 3, j = lane - 3 * p;
    const double g = jw[0] * Wg->dpos[p][0][j] + jw[1] * Wg->dpos[p][1][j] + jw[2] * Wg->dpos[p][2][j];
    fix_add(&d.acc_hb[3 * (size_t)Wg->parent[p] + j], g);
  }
  return false;
}

template <int WAVES, int CAP, int MORE>
__global__ __launch_bounds__(64 * WAVES) void k_ws_free(Dev d) {
  __shared__ WsLds<WAVES, CAP> L;
  const int w = (int)(threadIdx.x >> 6);
  if (MORE == WS_LIST) {
    ws_free_site<WAVES, CAP, MORE>(d, L, (int)blockIdx.x * WAVES + w, w);
    return;
  }
  const int nlist = (int)d.counters[kCountWs];
  for (int item = blockIdx.x; item < nlist; item += gridDim.x) {
    ws_free_site<WAVES, CAP, MORE>(d, L, d.ws_ovf[item], w);
    __syncthreads();                     // the next listed site reuses the buffers
  }
}

void launch_ws_free(const Dev &d, hipStream_t s) {
  if (d.nws == 0) return;
  hipLaunchKernelGGL((k_ws_free<kWsWaves, kWsCap, WS_LIST>), dim3((d.nws + kWsWaves - 1) / kWsWaves),
                     dim3(64 * kWsWaves), 0, s, d);
  hipLaunchKernelGGL((k_ws_free<1, kWsCapBig, WS_FAIL>), dim3(std::min(d.nws, 64)), dim3(64), 0, s, d);
}

// ------------------------------------- descreening by tiles, beside the sites
// The descreening sums (k_descreen) of small and middle-sized calls, whose
// items are too few to fill the chip.  There a wave walks 512 columns, four
// behind each scalar load, a branch and an LDS wait per column: that one
// wave's latency, 100 us, is the launch's at 2,000 and at 8,000 atoms alike.
// Here an item is a row block against one 256-column tile; its columns and
// tables come to LDS in one round of vector loads, and the lookups of
// kDtUnroll columns are in flight together.  A row's FP32 sum runs over the tile's
// columns in the same order, with the same operations, as k_descreen's, and
// leaves as a plain store of the tile's sum (k_born adds the tiles).  The
// water sites' free volumes, which need only the self volumes too, take the
// launch's first blocks.
// Descreening and sites, before (three launches) and after: 61 atoms 30 -> 10
// us, 2,000 142 -> 22, 6,000 134 -> 35, 11,000 130 -> 72, 14,000 132 -> 98
// (bound there by LDS: two broadcast reads per column and wave beside the
// table's).  Past kDtItems items the plain kernel's scalar loads are the
// better form: 25,000 atoms 169 us against 239 here.
constexpr int kDtCols = 256, kDtUnroll = 4;
// most blocks, sites' and rows', for that: its LDS leaves a CU to each (1,500 atoms,
// call 206 -> 198 us; 2,000, 330 blocks, 208 either way; 4,000, 900 blocks, 258 -> 284)
constexpr int kDtFew = 320;
constexpr size_t dt_lds(int ntypes) {
  return (size_t)ntypes * kTblN * sizeof(float2) + kDtCols * (sizeof(float4) + sizeof(float2));
}

// one column's Q4 for a row at pi (q4_value without its branch)
__device__ __forceinline__ float desc_value(const float2 *tab, const float4 &pj, const float2 &cw, const float4 &pi) {
  const float ex = pj.x - pi.x, ey = pj.y - pi.y, ez = pj.z - pi.z;
  const float xh = __builtin_amdgcn_sqrtf(fmaf(ez, ez, fmaf(ex, ex, ey * ey))) * pj.w;
  const unsigned k = (unsigned)(int)xh;
  const float2 *n = tab + __float_as_int(cw.y) * kTblN + min(k, (unsigned)(kTblN - 2));
  const float2 n0 = n[0], n1 = n[1];
  const float B = __builtin_amdgcn_fractf(xh), A = 1.f - B;
  const float s = fmaf(B, n1.y, fmaf(A, n0.y, n0.y + n1.y));
  const float v = fmaf(-(A * B), s, fmaf(A, n0.x, B * n1.x));
  return k <= (unsigned)(kTblN - 2) ? v : 0.f;
}

__device__ __forceinline__ void desc_tile(const Dev &d, char *lds, int item) {
  float2 *tab = reinterpret_cast<float2 *>(lds);
  float4 *col = reinterpret_cast<float4 *>(tab + d.ntypes * kTblN);
  float2 *cwt = reinterpret_cast<float2 *>(col + kDtCols);
  const int4 it = d.dt_items[item];                 // row block, columns [y, z), place of the sums
  const int nc = it.z - it.y, nrow = d.rows;
  const int i = (int)threadIdx.x < nrow ? d.row_perm[it.x * nrow + threadIdx.x] : -1;
  const float dp2 = d.tdx * (d.tdx / 6.0f);         // the nodes carry dx^2 / 6 (as k_descreen's)
  const float2 *src = d.tbl + (size_t)d.rblk[it.x].x * d.ntypes * kTblN;
  float4 pi = make_float4(0.f, 0.f, 0.f, 0.f), pc = pi;
  float2 wc = make_float2(0.f, 0.f);
  if ((int)threadIdx.x < nc) {
    pc = d.dcol[it.y + threadIdx.x];
    wc = d.dcw[it.y + threadIdx.x];
  }
  if (i >= 0) pi = d.pos[i];
#pragma unroll 10
  for (int k = threadIdx.x; k < d.ntypes * kTblN; k += 256) {
    const float2 v = src[k];
    tab[k] = make_float2(v.x, v.y * dp2);
  }
  col[threadIdx.x] = pc;
  cwt[threadIdx.x] = wc;
  __syncthreads();
  if (__ballot(i >= 0) == 0ull) return;             // a wave of padding rows (no barrier follows)
  float acc = 0.f;
  auto tile = [&](auto self) {
    auto columns = [&](int c, auto count) {
      constexpr int N = decltype(count)::value;
      float q[N], w[N];
#pragma unroll
      for (int u = 0; u < N; u++) {
        const float2 cw = cwt[c + u];
        q[u] = desc_value(tab, col[c + u], cw, pi);
        w[u] = decltype(self)::value && it.y + c + u == i ? 0.f : cw.x;
      }
#pragma unroll
      for (int u = 0; u < N; u++) acc = fmaf(q[u], w[u], acc);      // in column order
    };
    int c = 0;
#pragma unroll 1
    for (; c + kDtUnroll <= nc; c += kDtUnroll) columns(c, std::integral_constant<int, kDtUnroll>{});
#pragma unroll 1
    for (; c < nc; c++) columns(c, std::integral_constant<int, 1>{});
  };
  if (__ballot(i >= it.y && i < it.z) != 0ull) tile(std::true_type{});
  else tile(std::false_type{});
  if (i >= 0) d.dpart[it.w + i] = acc;
}

// The same for calls of so few items that a wave's 256 columns are the launch:
// a block takes 64 of an item's rows, its four waves look up 64 columns each and
// leave the values in LDS, and one adds them up in column order.
// Bound: the sites beside it (12 us).  k_desc_sites at 613 atoms 22.1 -> 14.4 us.
__device__ __forceinline__ void desc_tile_few(const Dev &d, char *lds, int sub) {
  float2 *tab = reinterpret_cast<float2 *>(lds);
  float4 *col = reinterpret_cast<float4 *>(tab + d.ntypes * kTblN);
  float2 *cwt = reinterpret_cast<float2 *>(col + kDtCols);
  float4 *val = reinterpret_cast<float4 *>(cwt + kDtCols);       // [four columns][lane]
  const int groups = d.rows / 64, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int4 it = d.dt_items[sub / groups];
  const int nc = it.z - it.y;
  const int i = d.row_perm[it.x * d.rows + (sub % groups) * 64 + lane];
  if (__ballot(i >= 0) == 0ull) return;             // padding rows (the same in every wave)
  const float dp2 = d.tdx * (d.tdx / 6.0f);
  const float2 *src = d.tbl + (size_t)d.rblk[it.x].x * d.ntypes * kTblN;
  float4 pi = make_float4(0.f, 0.f, 0.f, 0.f), pc = pi;
  float2 wc = make_float2(0.f, 0.f);                // (columns past the range: no weight, tables of type 0)
  if ((int)threadIdx.x < nc) {
    pc = d.dcol[it.y + threadIdx.x];
    wc = d.dcw[it.y + threadIdx.x];
  }
  if (i >= 0) pi = d.pos[i];
#pragma unroll 10
  for (int k = threadIdx.x; k < d.ntypes * kTblN; k += 256) {
    const float2 v = src[k];
    tab[k] = make_float2(v.x, v.y * dp2);
  }
  col[threadIdx.x] = pc;
  cwt[threadIdx.x] = wc;
  __syncthreads();
#pragma unroll 2
  for (int c = 64 * w; c < min(64 * w + 64, nc); c += 4) {
    float q[4];
#pragma unroll
    for (int u = 0; u < 4; u++) q[u] = desc_value(tab, col[c + u], cwt[c + u], pi);
    val[c / 4 * 64 + lane] = make_float4(q[0], q[1], q[2], q[3]);
  }
  __syncthreads();
  if (w != 0) return;                               // (no barrier follows)
  float acc = 0.f;
#pragma unroll 4
  for (int c = 0; c < nc; c += 4) {
    const float4 v = val[c / 4 * 64 + lane];
    const float q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int u = 0; u < 4; u++) acc = fmaf(q[u], it.y + c + u == i ? 0.f : cwt[c + u].x, acc);
  }
  if (i >= 0) d.dpart[it.w + i] = acc;
}

template <bool FEW>
__global__ __launch_bounds__(256) void k_desc_sites(Dev d, int nsite_blocks) {
  extern __shared__ __align__(16) char lds[];
  if ((int)blockIdx.x >= nsite_blocks) {
    if constexpr (FEW) desc_tile_few(d, lds, (int)blockIdx.x - nsite_blocks);
    else desc_tile(d, lds, (int)blockIdx.x - nsite_blocks);
    return;
  }
  // four sites, then those with more candidates than 128 one by one
  __shared__ int more[kWsWaves];
  const int w = (int)(threadIdx.x >> 6), site = (int)blockIdx.x * kWsWaves + w;
  const bool again = ws_free_site<kWsWaves, kWsCap, WS_RETURN>(
      d, *reinterpret_cast<WsLds<kWsWaves, kWsCap> *>(lds), site, w);
  if ((threadIdx.x & 63) == 0) more[w] = again ? site : d.nws;
  __syncthreads();
  for (int k = 0; k < kWsWaves; k++) {
    const int s = more[k];
    if (s >= d.nws) continue;                       // block-uniform
    ws_free_site<1, kWsCapBig, WS_FAIL>(d, *reinterpret_cast<WsLds<1, kWsCapBig> *>(lds), w == 0 ? s : d.nws, 0);
    __syncthreads();
  }
}

static size_t desc_sites_lds(int ntypes, bool few) {
  const size_t tile = dt_lds(ntypes) + (few ? (size_t)kDtCols * 64 * sizeof(float) : 0);
  return std::max(tile, std::max(sizeof(WsLds<kWsWaves, kWsCap>), sizeof(WsLds<1, kWsCapBig>)));
}

hipError_t prepare_sites(int ntypes) {
  static int limit = 0;                             // raised to the largest any pack has needed
  const int t = std::min(ntypes, kLdsTypes);
  if (t <= limit) return hipSuccess;
  const auto set = [&](const void *f, bool few) {
    return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)desc_sites_lds(t, few));
  };
  hipError_t e = set((const void *)k_desc_sites<false>, false);
  if (e == hipSuccess) e = set((const void *)k_desc_sites<true>, true);
  if (e == hipSuccess) limit = t;
  return e;
}

// about a block per CU, which is what its LDS allows
bool desc_sites_few(const Dev &d) {
  return (d.nws + kWsWaves - 1) / kWsWaves + d.ndt_items * (d.rows / 64) <= kDtFew;
}

void launch_desc_sites(const Dev &d, hipStream_t s) {
  const int ns = (d.nws + kWsWaves - 1) / kWsWaves, subs = d.ndt_items * (d.rows / 64);
  const bool few = desc_sites_few(d);
  const int nb = ns + (few ? subs : d.ndt_items);
  if (nb)
    hipLaunchKernelGGL(few ? k_desc_sites<true> : k_desc_sites<false>, dim3(nb), dim3(256), desc_sites_lds(d.ntypes, few), s,
                       d, ns);
}

}  // namespace agb
