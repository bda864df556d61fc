// Gaussian-overlap tree: self volumes and surface areas (pass A) and their
// coordinate derivatives (pass B).
//
// Tree (reference agbnp3_self_volumes_rooti, agbnp3_cpu_simd_kernels.c:1064-1598):
// the order-2 overlaps of root i are (i, j) for j in i's neighbour list, in
// list order; the children of an overlap are formed with the last atom of
// each later sibling in its group; an overlap is kept when its switched
// volume exceeds FLT_MIN; orders 2..5.  Its inclusion-exclusion
// coefficient is (-1)^(n+1)/n for the volume and (-1)^(n+1) for the surface.
//
// GPU mapping: one workgroup per root (two waves; a second tier with 8
// waves and larger level buffers for the biggest trees).  Its neighbour row
// ("slots": 0 = the root, 1..m = list entries) is staged in LDS and the tree
// is built breadth first: every candidate of one order -- for each node, the
// last atoms of its later siblings -- is one thread-parallel pass (a few
// passes per order instead of one per sibling group), kept overlaps are
// compacted in candidate order with ballots and per-wave counts, so each
// node's children stay contiguous and in the order the reference forms
// them.  Every overlap of the root involves only slot atoms, so
// contributions are reduced per slot in LDS (64-bit fixed point, so the sum
// does not depend on which wave adds first) and scattered to atoms once per
// root with order-independent fixed-point atomics; the root, a member of
// every overlap, is summed in lane registers.  A root whose tree outgrows
// the LDS level buffers is queued for the next tier, and past the second
// tier walked depth first (one sibling group per pass), with one group per
// order held at a time.
//
// Root frame: a root's slot atoms are staged at their positions relative to
// the root (an FP32 difference of nearby coordinates, accurate to an ulp of
// the few-Angstrom result).  Every overlap centre and member offset of the
// root is then a small number; in absolute coordinates each centre would
// carry the rounding of its tens-of-Angstrom position (3.8e-6 A at 30 A from
// the origin), which shows up as relative errors of ~1e-5 in the surface
// area gradients of large solutes.  The model is translation invariant, so
// nothing else changes.
//
// Pass B re-walks the identical tree (same FP32 arithmetic, same pruning)
// instead of storing it, and applies in one place the derivatives of
// agbnp3_der_vp_rooti (kernels.c:1601-1956: self-volume changes through
// U_i, V_i, H_i) and agbnp3_cavity_dersgb_rooti (kernels.c:1959-2405:
// surface-area changes through gamma', dervs, derus).
#include <float.h>

#include <type_traits>

#include "agb_common.h"
#include "agb_device.h"

namespace agb {

template <int CAP, bool PB>
struct TreeLds {
  int idx[CAP + 1];
  float a[CAP + 1], x[CAP + 1], y[CAP + 1], z[CAP + 1], R[CAP + 1];
  // pass B per-slot coefficients: deru, derv, derh, gamma', dervs, derus
  float u[PB ? CAP + 1 : 1], v[PB ? CAP + 1 : 1], h[PB ? CAP + 1 : 1];
  float wc[PB ? CAP + 1 : 1], wv[PB ? CAP + 1 : 1], wg[PB ? CAP + 1 : 1];
  // sibling groups of depths 0..2 (overlap Gaussian + last slot)
  float ga[3][CAP], gp[3][CAP], gx[3][CAP], gy[3][CAP], gz[3][CAP];
  int gs[3][CAP];
  // per-slot FP64 accumulators: pass A (volume, surface), pass B 12 gradient terms
  double acc[PB ? TG_N : 2][CAP + 1];
};

// coefficients of an overlap of order n
__device__ __forceinline__ float ovl_sign(int n) { return (n & 1) ? 1.0f : -1.0f; }  // (-1)^(n+1)

struct Gauss {
  float a, p, x, y, z;
};

// FP32 Gaussian overlap of `par` with atom (ab, xb) (kernels.c:2418-2477).
// What an overlap is and passes on (V, exponent, prefactor, centre, and with
// vol_switch V') has its fused products written out and no others: this is
// inlined into every walk of both passes, and all of them have to keep the same
// overlaps (left to the compiler, a walk may fuse another product of a sum
// than the next one, and pass B keep an overlap that pass A dropped).
struct OvlOut {
  float V, Vp, fp, fpp, a, p, cx, cy, cz, dinv;
};
__device__ __forceinline__ OvlOut overlap(const Gauss &par, float ab, float xb, float yb, float zb) {
  OvlOut o;
  float s, sp, spp;
  {
#pragma clang fp contract(off)
    const float dx = xb - par.x, dy = yb - par.y, dz = zb - par.z;
    const float d2 = fmaf(dz, dz, fmaf(dx, dx, dy * dy));
    o.a = par.a + ab;
    o.dinv = __builtin_amdgcn_rcpf(o.a);                            // hardware reciprocal, exp, sqrt (1-2 ulp)
    o.p = par.p * kPFC * __expf(-par.a * ab * d2 * o.dinv);
    const float u = kPiF * o.dinv;
    o.V = o.p * u * __builtin_amdgcn_sqrtf(u);
    vol_switch(o.V, s, sp, spp);
    o.Vp = s * o.V;
    o.cx = o.dinv * fmaf(par.a, par.x, ab * xb);
    o.cy = o.dinv * fmaf(par.a, par.y, ab * yb);
    o.cz = o.dinv * fmaf(par.a, par.z, ab * zb);
  }
  o.fp = s + o.V * sp;
  o.fpp = 2.f * sp + o.V * spp;
  return o;
}

// pass-A contribution of one overlap to member (a, x, R): surface term
__device__ __forceinline__ float sa_term(const OvlOut &o, float sign, float a, float x, float y, float z, float R) {
  const float ex = x - o.cx, ey = y - o.cy, ez = z - o.cz;
  const float t = ex * ex + ey * ey + ez * ez;
  return sign * o.fp * a * o.V * (3.f * o.dinv + 2.f * t) * __builtin_amdgcn_rcpf(R);
}

// add to a per-slot accumulator: FP64 LDS atomics in the depth-first walk, one
// wave per root (the lanes' order is fixed), or 64-bit fixed point with integer
// atomics in the breadth-first ones with their several waves (the sum does not
// depend on their order; an LDS add of a zero costs less than testing for it)
__device__ __forceinline__ void slot_add(double *p, double v) { atomicAdd(p, v); }
__device__ __forceinline__ void slot_add(long long *p, double v) {
  atomicAdd((unsigned long long *)p, (unsigned long long)__double2ll_rn(v * kFix));
}
// The same for |v| < kSmall: at 1.5 x 2^20 a double's last place is 2^-32, so
// an addition there rounds v to the fixed point, and the sum's bits less the
// constant's are the integer: one addition and one subtraction instead of the
// conversion's seven FP64 instructions, 12 times per member of every overlap.
// 2,000 atoms: call 219 -> 216 us, 25,000 984 -> 977, 64 poses 800 -> 786.
constexpr float kSmall = 524288.f;
__device__ __forceinline__ void slot_add_small(long long *p, double v) {
  constexpr double c = 1572864.0;
  atomicAdd((unsigned long long *)p,
            (unsigned long long)(__builtin_bit_cast(long long, v + c) - __builtin_bit_cast(long long, c)));
}
// whether every active lane may add numbers of this sum of sizes as above
__device__ __forceinline__ bool all_small(float big) { return __builtin_expect(__ballot(!(big < kSmall)) == 0ull, 1); }

// Pass-B terms of one kept overlap of order N for each member k: the
// derivatives of its self-volume and surface contributions with respect to
// x_k (agbnp3_der_vp_rooti, kernels.c:1601-1956, through U, V, H;
// agbnp3_cavity_dersgb_rooti, kernels.c:1959-2405, through gamma', dervs,
// derus).  With g_k = dV/dx_k = -2 a_k V (x_k - c), the radius term
// G_k = a_k V (3/a + 2 |x_k - c|^2) / R_k, S1 = sum_k W_k G_k and
// S2 = sum_k W_k g_k / R_k per weight set W (sign folded in), member k gets
//   g_k (h3 S1 - 2 fp W_k / R_k [+ U or V coefficient]) + 2 fp a_k S2 / a
// for the GB, vdW and cavity terms and H g_k for the HB term; h3 = f'' +
// f'/V.  emit(k, out[TG_N]) receives them in member order.
template <int N, typename Emit>
__device__ __forceinline__ void member_derivs(const OvlOut &o, float cn, float df, const float (&A_)[N],
                                              const float (&X_)[N], const float (&Y_)[N], const float (&Z_)[N],
                                              const float (&R_)[N], const float (&WC)[N], const float (&WV)[N],
                                              const float (&WG)[N], float Us, float Vs, float Hs, Emit emit) {
  const float fourpi1 = 1.0f / (4.0f * kPiF);
  const float Uc = -df * fourpi1 * cn * Us * o.fp;
  const float Vc = -fourpi1 * cn * Vs * o.fp;
  const float Hc = -cn * Hs * o.fp;
  const float h3 = o.fpp + o.fp * __builtin_amdgcn_rcpf(o.V), h4 = 2.f * o.fp * o.dinv;
  const float c3 = 3.f * o.dinv, m2V = -2.f * o.V, m2fp = -2.f * o.fp;
  float g[N][3], iR[N];
  float S1c = 0.f, S1v = 0.f, S1g = 0.f;
  float S2c[3] = {0.f, 0.f, 0.f}, S2v[3] = {0.f, 0.f, 0.f}, S2g[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < N; k++) {
    const float ex = X_[k] - o.cx, ey = Y_[k] - o.cy, ez = Z_[k] - o.cz;
    const float av = A_[k] * o.V, mav = A_[k] * m2V;
    iR[k] = __builtin_amdgcn_rcpf(R_[k]);
    g[k][0] = mav * ex;
    g[k][1] = mav * ey;
    g[k][2] = mav * ez;
    const float GR = av * (c3 + 2.f * (ex * ex + ey * ey + ez * ez)) * iR[k];
    S1c += WC[k] * GR; S1v += WV[k] * GR; S1g += WG[k] * GR;
    const float wc = WC[k] * iR[k], wv = WV[k] * iR[k], wg = WG[k] * iR[k];
#pragma unroll
    for (int q = 0; q < 3; q++) {
      S2c[q] += wc * g[k][q];
      S2v[q] += wv * g[k][q];
      S2g[q] += wg * g[k][q];
    }
  }
  const float Kc = h3 * S1c, Kv = h3 * S1v + Vc, Kg = h3 * S1g + Uc;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const float t = m2fp * iR[k], ha = h4 * A_[k];
    const float kc = Kc + WC[k] * t, kv = Kv + WV[k] * t, kg = Kg + WG[k] * t;
    float out[TG_N];
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const float gq = g[k][q];
      out[TG_GB + q] = gq * kg + ha * S2g[q];
      out[TG_VW + q] = gq * kv + ha * S2v[q];
      out[TG_CAV + q] = gq * kc + ha * S2c[q];
      out[TG_HB + q] = Hc * gq;
    }
    emit(k, out);
  }
}

// Contributions of one kept overlap o of order N with members mem[0..N-1]
// (mem[0] = 0, the root) to the root's registers and the slot accumulators.
// The root's registers are per lane (RT: FP64 for the volume pass, FP32 for
// the derivative pass, where a lane adds a few terms per root before the
// FP64 wave sum).
template <int N, int CAP, bool PB, typename Lds, typename RT>
__device__ __forceinline__ void add_contrib(Lds &S, const OvlOut &o, const int (&mem)[N], RT (&root)[TG_N],
                                            float df) {
  const float sign = ovl_sign(N);
  const float cn = sign / (float)N;
  if (!PB) {
    const double wv = (double)cn * (double)o.Vp;
    root[0] += wv;
    const float4 p0 = S.p[0];
    root[1] += (double)sa_term(o, sign, p0.w, p0.x, p0.y, p0.z, S.r[0]);
    float sa[N];
#pragma unroll
    for (int k = 1; k < N; k++) {
      const float4 pk = S.p[mem[k]];
      sa[k] = sa_term(o, sign, pk.w, pk.x, pk.y, pk.z, S.r[mem[k]]);
    }
    float big = o.Vp;
#pragma unroll
    for (int k = 1; k < N; k++) big += fabsf(sa[k]);
    if (all_small(big)) {
#pragma unroll
      for (int k = 1; k < N; k++) {
        slot_add_small(&S.acc[0][mem[k]], wv);
        slot_add_small(&S.acc[1][mem[k]], (double)sa[k]);
      }
    } else {
#pragma unroll
      for (int k = 1; k < N; k++) {
        slot_add(&S.acc[0][mem[k]], wv);
        slot_add(&S.acc[1][mem[k]], (double)sa[k]);
      }
    }
  } else {
    float A_[N], X_[N], Y_[N], Z_[N], R_[N], WC[N], WV[N], WG[N];
    float Us = 0.f, Vs = 0.f, Hs = 0.f;
#pragma unroll
    for (int k = 0; k < N; k++) {
      const float4 pk = S.p[mem[k]], qk = S.q[mem[k]], wk = S.w[mem[k]];
      A_[k] = pk.w; X_[k] = pk.x; Y_[k] = pk.y; Z_[k] = pk.z; R_[k] = qk.x;
      WC[k] = sign * wk.x; WV[k] = sign * wk.y; WG[k] = sign * wk.z;
      Us += qk.y; Vs += qk.z; Hs += qk.w;
    }
    member_derivs<N>(o, cn, df, A_, X_, Y_, Z_, R_, WC, WV, WG, Us, Vs, Hs, [&](int k, const float (&out)[TG_N]) {
      if (k == 0) {
#pragma unroll
        for (int v = 0; v < TG_N; v++) root[v] += (RT)out[v];
      } else {
        float big = 0.f;
#pragma unroll
        for (int v = 0; v < TG_N; v++) big += fabsf(out[v]);
        if (all_small(big)) {
#pragma unroll
          for (int v = 0; v < TG_N; v++) slot_add_small(&S.acc[v][mem[k]], out[v]);
        } else {
#pragma unroll
          for (int v = 0; v < TG_N; v++) slot_add(&S.acc[v][mem[k]], out[v]);
        }
      }
    });
  }
}

// Evaluate the children of one tree node: lanes take candidate slots, keep
// overlaps above FLT_MIN, add their contributions, and (if STORE) compact
// them into group level L.  N = L + 2 is the order of the children; the
// members are the path slots path[0..L] and the candidate.
template <int L, int CAP, bool PB, bool STORE>
__device__ __forceinline__ int eval_children(TreeLds<CAP, PB> &S, const Gauss &par, const int *path,
                                             int ncand, const int *cand_slots_lds, int cand_base,
                                             double (&root)[TG_N], float df, unsigned &nkept, unsigned &neval) {
  constexpr int N = L + 2;
  const int lane = threadIdx.x & 63;
  const float sign = ovl_sign(N);
  const float cn = sign / (float)N;
  int cnt = 0;
  // path member data (wave-uniform broadcast reads)
  float ma[N - 1], mx[N - 1], my[N - 1], mz[N - 1], mR[N - 1];
#pragma unroll
  for (int k = 0; k < N - 1; k++) {
    const int s = path[k];
    ma[k] = S.a[s]; mx[k] = S.x[s]; my[k] = S.y[s]; mz[k] = S.z[s]; mR[k] = S.R[s];
  }
  float pU = 0.f, pV = 0.f, pH = 0.f;
  float mwc[N - 1], mwv[N - 1], mwg[N - 1];
  if (PB) {
#pragma unroll
    for (int k = 0; k < N - 1; k++) {
      const int s = path[k];
      pU += S.u[s]; pV += S.v[s]; pH += S.h[s];
      mwc[k] = sign * S.wc[s]; mwv[k] = sign * S.wv[s]; mwg[k] = sign * S.wg[s];
    }
  }
  for (int base = 0; base < ncand; base += 64) {
    const int c = base + lane;
    bool keep = false;
    int sb = 0;
    OvlOut o;
    if (c < ncand) {
      sb = cand_slots_lds ? cand_slots_lds[cand_base + c] : cand_base + c;
      o = overlap(par, S.a[sb], S.x[sb], S.y[sb], S.z[sb]);
      keep = o.Vp > FLT_MIN;
    }
    neval += (unsigned)__popcll(__ballot(c < ncand));
    const unsigned long long bal = __ballot(keep);
    if (keep) {
      const float ab = S.a[sb], xb = S.x[sb], yb = S.y[sb], zb = S.z[sb], Rb = S.R[sb];
      if (!PB) {
        const double wv = (double)cn * (double)o.Vp;
        root[0] += wv;
        root[1] += (double)sa_term(o, sign, ma[0], mx[0], my[0], mz[0], mR[0]);
#pragma unroll
        for (int k = 1; k < N - 1; k++) {
          slot_add(&S.acc[0][path[k]], wv);
          slot_add(&S.acc[1][path[k]], (double)sa_term(o, sign, ma[k], mx[k], my[k], mz[k], mR[k]));
        }
        slot_add(&S.acc[0][sb], wv);
        slot_add(&S.acc[1][sb], (double)sa_term(o, sign, ab, xb, yb, zb, Rb));
      } else {
        // members: path[0..N-2] then the candidate (index N-1)
        float A_[N], X_[N], Y_[N], Z_[N], R_[N], WC[N], WV[N], WG[N];
#pragma unroll
        for (int k = 0; k < N - 1; k++) {
          A_[k] = ma[k]; X_[k] = mx[k]; Y_[k] = my[k]; Z_[k] = mz[k]; R_[k] = mR[k];
          WC[k] = mwc[k]; WV[k] = mwv[k]; WG[k] = mwg[k];
        }
        A_[N - 1] = ab; X_[N - 1] = xb; Y_[N - 1] = yb; Z_[N - 1] = zb; R_[N - 1] = Rb;
        WC[N - 1] = sign * S.wc[sb]; WV[N - 1] = sign * S.wv[sb]; WG[N - 1] = sign * S.wg[sb];
        const float Us = pU + S.u[sb], Vs = pV + S.v[sb], Hs = pH + S.h[sb];
        member_derivs<N>(o, cn, df, A_, X_, Y_, Z_, R_, WC, WV, WG, Us, Vs, Hs,
                         [&](int k, const float (&out)[TG_N]) {
          if (k == 0) {
#pragma unroll
            for (int v = 0; v < TG_N; v++) root[v] += (double)out[v];
          } else {
            const int slot = k < N - 1 ? path[k] : sb;
#pragma unroll
            for (int v = 0; v < TG_N; v++) slot_add(&S.acc[v][slot], (double)out[v]);
          }
        });
      }
      if (STORE) {
        const int pos = cnt + __popcll(bal & ((1ull << lane) - 1ull));
        S.ga[L][pos] = o.a; S.gp[L][pos] = o.p;
        S.gx[L][pos] = o.cx; S.gy[L][pos] = o.cy; S.gz[L][pos] = o.cz;
        S.gs[L][pos] = sb;
      }
    }
    cnt += __popcll(bal);
  }
  nkept += (unsigned)cnt;
  wave_sync();
  return cnt;
}

// depth-first walk of one root by one wave (the other waves of its block are
// past their last access to the LDS it reuses, and take no part)
template <int CAP, bool PB>
__device__ void tree_dfs_root(const Dev &d, TreeLds<CAP, PB> &S, int h, unsigned long long &tk,
                              unsigned long long &te) {
  const int lane = threadIdx.x & 63;
  const int i = d.hrow[h];
  const int m = d.nne[h];
  // stage the slot atoms, positions relative to the root (root_frame)
  const float4 pr = d.pos[i];
  for (int s = lane; s <= m; s += 64) {
    const int at = s == 0 ? i : d.nbr[(size_t)h * d.cap + s - 1];
    const float4 p = d.pos[at];
    S.idx[s] = at;
    S.a[s] = d.galpha[at];
    S.x[s] = p.x - pr.x; S.y[s] = p.y - pr.y; S.z[s] = p.z - pr.z; S.R[s] = p.w;
    if (PB) {
      S.u[s] = d.deru_f[at]; S.v[s] = d.derv_f[at]; S.h[s] = d.derh_f[at];
      S.wc[s] = d.gammap_f[at]; S.wv[s] = d.dervs_f[at]; S.wg[s] = d.derus_f[at];
    }
#pragma unroll
    for (int v = 0; v < (PB ? TG_N : 2); v++) S.acc[v][s] = 0.0;
  }
  wave_sync();
  double root[TG_N];
#pragma unroll
  for (int v = 0; v < TG_N; v++) root[v] = 0.0;
  unsigned nkept = 0, neval = 0;
  const float df = d.sys[d.asys[i]].df;
  int path[4];
  path[0] = 0;
  const Gauss rg = {S.a[0], kPFC, S.x[0], S.y[0], S.z[0]};
  // order 2: (i, j) for every list entry
  const int n0 = eval_children<0, CAP, PB, true>(S, rg, path, m, nullptr, 1, root, df, nkept, neval);
  for (int i0 = 0; i0 + 1 < n0; i0++) {
    path[1] = S.gs[0][i0];
    const Gauss g0 = {S.ga[0][i0], S.gp[0][i0], S.gx[0][i0], S.gy[0][i0], S.gz[0][i0]};
    const int n1 = eval_children<1, CAP, PB, true>(S, g0, path, n0 - i0 - 1, &S.gs[0][0], i0 + 1, root, df, nkept,
                                                   neval);
    for (int i1 = 0; i1 + 1 < n1; i1++) {
      path[2] = S.gs[1][i1];
      const Gauss g1 = {S.ga[1][i1], S.gp[1][i1], S.gx[1][i1], S.gy[1][i1], S.gz[1][i1]};
      const int n2 = eval_children<2, CAP, PB, true>(S, g1, path, n1 - i1 - 1, &S.gs[1][0], i1 + 1, root, df,
                                                     nkept, neval);
      for (int i2 = 0; i2 + 1 < n2; i2++) {
        path[3] = S.gs[2][i2];
        const Gauss g2 = {S.ga[2][i2], S.gp[2][i2], S.gx[2][i2], S.gy[2][i2], S.gz[2][i2]};
        eval_children<3, CAP, PB, false>(S, g2, path, n2 - i2 - 1, &S.gs[2][0], i2 + 1, root, df, nkept, neval);
      }
    }
  }
  // the root's own sums, then every slot to its atom
#pragma unroll
  for (int v = 0; v < (PB ? TG_N : 2); v++) {
    const double r = wave_sum(root[v]);
    if (lane == 0) S.acc[v][0] += r;
  }
  wave_sync();
  for (int s = lane; s <= m; s += 64) {
    const int at = S.idx[s];
    if (!PB) {
      fix_add(&d.acc_vol[at], S.acc[0][s]);
      fix_add(&d.acc_sa[at], S.acc[1][s]);
    } else {
#pragma unroll
      for (int v = 0; v < TG_N; v++) fix_add(&d.acc_grad[(size_t)at * TG_N + v], S.acc[v][s]);
    }
  }
  tk += nkept;                          // wave-uniform; added to the counters once per block
  te += neval;
  wave_sync();
}

// ------------------------------------------------------ breadth-first tree
constexpr int kLevelCapBig = 512;       // second tier (dynamic LDS) for the largest trees

template <int CAP, bool PB, int LC, int W>
struct BfsLds {
  int idx[CAP + 1];
  // slot atoms, one 16-byte read per record: x, y, z, Gaussian exponent;
  // pass A radius; pass B (radius, deru, derv, derh), (gamma', dervs, derus)
  float4 p[CAP + 1];
  float r[PB ? 1 : CAP + 1];
  float4 q[PB ? CAP + 1 : 1], w[PB ? CAP + 1 : 1];
  long long acc[PB ? TG_N : 2][CAP + 1];
  // two node buffers: Gaussian, member slots (16 bits each, root excluded),
  // end of the node's sibling group, parent index in the previous order
  float ga[2][LC], gp[2][LC], gx[2][LC], gy[2][LC], gz[2][LC];
  // member slots packed 8 bits each while slots fit (CAP < 256), else 16;
  // node indices in 8 bits while levels hold fewer than 256 nodes
  using PathT = typename std::conditional<(CAP < 256), unsigned, unsigned long long>::type;
  using NodeT = typename std::conditional<(LC < 256), unsigned char, unsigned short>::type;
  static constexpr int kSlotBits = CAP < 256 ? 8 : 16;
  static constexpr PathT kSlotMask = (PathT)((1u << kSlotBits) - 1u);
  PathT path[2][LC];
  NodeT gend[2][LC], gpar[2][LC];
  int pref[LC + 1], cnt[LC];
  int wcnt[2][W];                       // kept candidates per wave of one pass
};

// Compaction of one pass over W*64 candidates (candidate = pass base +
// 64 * wave + lane): this lane's position among the pass's kept candidates,
// and their total (block-uniform).  wcnt alternates between two rows by
// pass parity, so one barrier per pass separates its writes from the reads
// of the pass before.
template <int W>
__device__ __forceinline__ int pass_compact(int (&wcnt)[2][W], int parity, unsigned long long bal, int &total) {
  const int lane = threadIdx.x & 63;
  const int below = __popcll(bal & ((1ull << lane) - 1ull));
  const int w = threadIdx.x >> 6;
  if (lane == 0) wcnt[parity][w] = __popcll(bal);
  __syncthreads();
  int off = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < W; k++) {
    const int c = wcnt[parity][k];
    off += k < w ? c : 0;
    tot += c;
  }
  total = tot;
  return off + below;
}

// per-atom fixed-point totals from the slot accumulators
__device__ __forceinline__ void scatter_add(long long *p, long long q) {
  if (q != 0) atomicAdd((unsigned long long *)p, (unsigned long long)q);
}

// exclusive scan of vals[0..n) into out[0..n], out[n] = total (one wave)
__device__ __forceinline__ int wave_exclusive_scan(const int *vals, int *out, int n) {
  const int lane = threadIdx.x & 63;
  int run = 0;
  for (int base = 0; base < n; base += 64) {
    const int k = base + lane;
    const int v = k < n ? vals[k] : 0;
    const int incl = wave_incl_scan(v);
    if (k < n) out[k] = run + incl - v;
    run += __shfl(incl, 63, 64);
  }
  if (lane == 0) out[n] = run;
  return run;
}

// children of order N: pairs (u, later sibling v) of the nodes of order N-1
// in buffer `cb` (n nodes), kept ones into buffer 1-cb; returns their count
// (LC + 1 on overflow).  W waves share the candidates; wave 0 runs the scans.
template <int N, int CAP, bool PB, int LC, int W, bool STORE, typename RT>
__device__ __forceinline__ int bfs_order(BfsLds<CAP, PB, LC, W> &S, int cb, int n, RT (&root)[TG_N], float df,
                                         unsigned &nkept, unsigned &neval) {
  constexpr int NT = 64 * W;
  const int tid = threadIdx.x;
  const int nb = 1 - cb;
  for (int k = tid; k < n; k += NT) {
    S.cnt[k] = S.gend[cb][k] - k - 1;     // later siblings of node k
  }
  __syncthreads();
  if (tid < 64) wave_exclusive_scan(S.cnt, S.pref, n);
  __syncthreads();
  const int P = S.pref[n];
  for (int k = tid; k < n; k += NT) S.cnt[k] = 0;
  __syncthreads();
  int nn = 0, parity = 0;
  for (int base = 0; base < P; base += NT, parity ^= 1) {
    const int q = base + tid;
    bool keep = false;
    int uu = 0, sb = 0;
    OvlOut o;
    if (q < P) {
      int lo = 0, hi = n - 1;              // last u with pref[u] <= q
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (S.pref[mid] <= q) lo = mid;
        else hi = mid - 1;
      }
      uu = lo;
      const int vv = uu + 1 + (q - S.pref[uu]);
      sb = (int)((S.path[cb][vv] >> (S.kSlotBits * (N - 3))) & S.kSlotMask);    // last atom of sibling v
      const Gauss par = {S.ga[cb][uu], S.gp[cb][uu], S.gx[cb][uu], S.gy[cb][uu], S.gz[cb][uu]};
      const float4 pb = S.p[sb];
      o = overlap(par, pb.w, pb.x, pb.y, pb.z);
      keep = o.Vp > FLT_MIN;
    }
    neval += (unsigned)__popcll(__ballot(q < P));
    int total;
    const int pos = nn + pass_compact<W>(S.wcnt, parity, __ballot(keep), total);
    if (keep) {
      const auto pu = S.path[cb][uu];
      int mem[N];
      mem[0] = 0;
#pragma unroll
      for (int k = 0; k < N - 2; k++) mem[1 + k] = (int)((pu >> (S.kSlotBits * k)) & S.kSlotMask);
      mem[N - 1] = sb;
      add_contrib<N, CAP, PB>(S, o, mem, root, df);
      if (STORE) {
        if (pos < LC) {
          S.ga[nb][pos] = o.a; S.gp[nb][pos] = o.p;
          S.gx[nb][pos] = o.cx; S.gy[nb][pos] = o.cy; S.gz[nb][pos] = o.cz;
          S.path[nb][pos] = pu | ((decltype(pu))sb << (S.kSlotBits * (N - 2)));
          S.gpar[nb][pos] = (std::remove_reference_t<decltype(S.gpar[0][0])>)uu;
        }
        atomicAdd(&S.cnt[uu], 1);
      }
    }
    nn += total;
  }
  nkept += (unsigned)nn;                // block-uniform
  __syncthreads();
  if (!STORE) return 0;
  if (nn > LC) return LC + 1;
  // a node's siblings are the kept children of its parent, contiguous
  if (tid < 64) wave_exclusive_scan(S.cnt, S.pref, n);
  __syncthreads();
  for (int k = tid; k < nn; k += NT) {
    const int par = S.gpar[nb][k];
    S.gend[nb][k] = (std::remove_reference_t<decltype(S.gend[0][0])>)(S.pref[par] + S.cnt[par]);
  }
  __syncthreads();
  return nn;
}

// one root of the breadth-first tree (the whole block); results scattered to
// the atoms, or the root queued for the next tier on overflow.  The block's
// waves split every order's candidates and the per-slot sums are fixed point,
// so the result does not depend on the waves' timing.
template <int CAP, bool PB, int LC, int W>
__device__ bool tree_bfs_root(const Dev &d, BfsLds<CAP, PB, LC, W> &S, int h, int list, unsigned long long &tk,
                              unsigned long long &te) {
  constexpr int NT = 64 * W;
  const int tid = threadIdx.x, lane = tid & 63;
  // pass B's first tier leaves the roots pass A queued to the second tier,
  // which takes pass A's list: both passes walk the same tree, so they
  // outgrow the same buffers
  // (its header and row are loaded together, and then all that hangs on them:
  // one by one, seven loads deep, they were a fifth of an average root's time)
  int i = d.hrow[h], m = d.nne[h], tier = PB && list == 0 ? d.tree_tier[h] : 0, nb = 0;
  if (tid > 0 && tid <= d.cap) nb = d.nbr[(size_t)h * d.cap + tid - 1];
  asm volatile("" : "+v"(i), "+v"(m), "+v"(tier), "+v"(nb));
  i = __builtin_amdgcn_readfirstlane(i);
  m = __builtin_amdgcn_readfirstlane(m);
  if (PB && list == 0 && __builtin_amdgcn_readfirstlane(tier)) return true;  // block-uniform
  // a root that outgrows these buffers: pass A's first tier queues it for the
  // second (and records that); past the second tier it is walked depth first,
  // in pass A by the caller, in pass B from a list.  None does in pass B's first
  // tier, which has the roots whose same walk fitted pass A's; one that did
  // would find nothing behind it that walks it, and fails the call.
  const int lc = PB && list == 0 ? d.tree_cap_b : LC;
  auto queue_next = [&]() {
    if (PB && list == 0) {
      if (tid == 0) atomicOr(d.status, ST_TREE_OVERFLOW);
    } else if (tid == 0) {
      const bool first = !PB && list == 0;
      const unsigned k = atomicAdd(&d.counters[first ? 4 : 6 + (PB ? 1 : 0)], 1ull);
      if (first || PB) d.tree_ovf[(PB ? (size_t)d.nh : 0) + k] = h;
      if (first) {
        d.tree_tier[h] = 1;
        d.tree_cnt[h] = make_uint2(0, 0);
      }
    }
    __syncthreads();
  };
  if (m > CAP) {                          // block-uniform: a row longer than these slot arrays, next tier
    queue_next();
    return false;
  }
  const float4 pr = d.pos[i];
  const int sys = PB ? d.asys[i] : 0;
  auto stage = [&](int s, int at) {
    const float4 p = d.pos[at];
    const float ga = d.galpha[at];
    float c[6];
    if (PB) {
      c[0] = d.deru_f[at]; c[1] = d.derv_f[at]; c[2] = d.derh_f[at];
      c[3] = d.gammap_f[at]; c[4] = d.dervs_f[at]; c[5] = d.derus_f[at];
    }
    S.idx[s] = at;
    S.p[s] = make_float4(p.x - pr.x, p.y - pr.y, p.z - pr.z, ga);   // root frame
    if (PB) {
      S.q[s] = make_float4(p.w, c[0], c[1], c[2]);
      S.w[s] = make_float4(c[3], c[4], c[5], 0.f);
    } else {
      S.r[s] = p.w;
    }
#pragma unroll
    for (int v = 0; v < (PB ? TG_N : 2); v++) S.acc[v][s] = 0;
  };
  if (tid <= m) stage(tid, tid == 0 ? i : nb);
  for (int s = tid + NT; s <= m; s += NT) stage(s, d.nbr[(size_t)h * d.cap + s - 1]);
  const float df = PB ? d.sys[sys].df : 0.f;
  __syncthreads();
  using RT = typename std::conditional<PB, float, double>::type;
  RT root[TG_N];
#pragma unroll
  for (int v = 0; v < TG_N; v++) root[v] = 0;
  unsigned nkept = 0, neval = 0;
  bool ovf = false;
  // order 2: the root with every list entry, one sibling group
  int n = 0;
  {
    const float4 p0 = S.p[0];
    const Gauss rg = {p0.w, kPFC, p0.x, p0.y, p0.z};
    int parity = 0;
    for (int base = 0; base < m; base += NT, parity ^= 1) {
      const int c = base + tid;
      bool keep = false;
      int sb = 0;
      OvlOut o;
      if (c < m) {
        sb = c + 1;
        const float4 pb = S.p[sb];
        o = overlap(rg, pb.w, pb.x, pb.y, pb.z);
        keep = o.Vp > FLT_MIN;
      }
      neval += (unsigned)__popcll(__ballot(c < m));
      int total;
      const int pos = n + pass_compact<W>(S.wcnt, parity, __ballot(keep), total);
      if (keep) {
        const int mem[2] = {0, sb};
        add_contrib<2, CAP, PB>(S, o, mem, root, df);
        if (pos < LC) {
          S.ga[0][pos] = o.a; S.gp[0][pos] = o.p;
          S.gx[0][pos] = o.cx; S.gy[0][pos] = o.cy; S.gz[0][pos] = o.cz;
          S.path[0][pos] = (std::remove_reference_t<decltype(S.path[0][0])>)sb;
        }
      }
      n += total;
    }
    nkept += (unsigned)n;
    if (n > lc) ovf = true;
    for (int k = tid; k < n && k < LC; k += NT) S.gend[0][k] = (std::remove_reference_t<decltype(S.gend[0][0])>)n;
    __syncthreads();
  }
  if (!ovf && n > 1) {
    n = bfs_order<3, CAP, PB, LC, W, true>(S, 0, n, root, df, nkept, neval);
    if (n > lc) ovf = true;
    else if (n > 1) {
      n = bfs_order<4, CAP, PB, LC, W, true>(S, 1, n, root, df, nkept, neval);
      if (n > lc) ovf = true;
      else if (n > 1) bfs_order<5, CAP, PB, LC, W, false>(S, 0, n, root, df, nkept, neval);
    }
  }
  if (ovf) {                              // block-uniform
    queue_next();
    return false;
  }
  if (!PB && list == 0 && tid == 0) d.tree_tier[h] = 0;
  // the root's own sums (slot 0 takes no member adds): each wave's
#pragma unroll
  for (int v = 0; v < (PB ? TG_N : 2); v++) {
    const double sum = wave_sum((double)root[v]);
    if (lane == 0) slot_add(&S.acc[v][0], sum);
  }
  if (lane == 0) S.wcnt[0][tid >> 6] = (int)neval;
  __syncthreads();
  if (!PB && list == 0 && tid == 0) {     // pass A's first tier: its counts, which k_scale adds up
    unsigned ev = 0;
#pragma unroll
    for (int w = 0; w < W; w++) ev += (unsigned)S.wcnt[0][w];
    d.tree_cnt[h] = make_uint2(nkept, ev);
  }
  for (int s = tid; s <= m; s += NT) {
    const int at = S.idx[s];
    if (!PB) {
      scatter_add(&d.acc_vol[at], S.acc[0][s]);
      scatter_add(&d.acc_sa[at], S.acc[1][s]);
    } else {
#pragma unroll
      for (int v = 0; v < TG_N; v++) scatter_add(&d.acc_grad[(size_t)at * TG_N + v], S.acc[v][s]);
    }
  }
  tk += nkept;                          // block-uniform: wave 0 reports it
  te += neval;                          // this wave's evaluations
  __syncthreads();                      // the next root restages the slots
  return true;
}

// overlaps kept (block totals) and evaluated (per wave) by one persistent
// block of pass A's second tier (the first stores them per root: three atomics
// of each block at exit cost it 1 % of a call)
__device__ __forceinline__ void add_tree_counts(const Dev &d, bool pass_b, unsigned long long tk,
                                                unsigned long long te) {
  if (pass_b || (threadIdx.x & 63) != 0) return;
  unsigned long long *c = d.counters + kCountBase + 8 * (blockIdx.x % kCountSlots);
  if (threadIdx.x == 0 && tk) atomicAdd(c, tk);
  if (te) atomicAdd(c + 1, te);
}


// A block per root (or, tuned, a persistent grid that takes roots from a
// queue): the dispatcher hands them out with less delay than a queue head, and
// evenly where the trees are not (11,000 atoms, call 445 -> 424 us, 90 ragged
// systems 1454 -> 1403, against 4,096 blocks that took two roots at a time).
// Overflowing roots go to the second tier's list.  Two waves per root share
// every order's candidates (slot sums in fixed point): at one wave per root
// the LDS of a root (13-27 KB) left a SIMD one or two waves to hide the
// walk's LDS and memory latency.
constexpr int kFirstWaves = 2;
// slot arrays of the first tier: 80 while rows are up to 128 wide (a root in
// 20 KB of LDS instead of 27 in pass B, so 8 roots per CU instead of 5; the
// few longer rows go to the second tier), else the rows' width.  At least 4
// waves per SIMD in pass B (at most 128 registers) and 7 in pass A (at most
// 72): LDS allows that many roots per CU.
constexpr int first_cap(int cap) { return cap == 128 ? 80 : cap; }
template <int CAP, bool PB>
__global__ __launch_bounds__(64 * kFirstWaves, PB ? 4 : 7) void k_tree_bfs(Dev d) {
  __shared__ BfsLds<CAP, PB, kLevelCap, kFirstWaves> S;
  __shared__ int slot;
  unsigned *head = queue_head(d.queue, PB ? Q_TREE_B : Q_TREE_A);
  // queue position k takes root (k * P) mod nh, P a prime that does not
  // divide nh: roots in flight together lie far apart in the atom order, so
  // their fixed-point scatters rarely meet on one atom
  const long long P = d.nh % 7919 ? 7919 : (d.nh % 7927 ? 7927 : 7933);
  unsigned long long tk = 0, te = 0;
  for (int k = first_item(); k < d.nh; k = next_item(head, &slot, d.nh))
    tree_bfs_root<CAP, PB, kLevelCap, kFirstWaves>(d, S, (int)(((long long)k * P) % d.nh), 0, tk, te);
}

// second tier: the roots pass A's first tier queued (in both passes), with
// 512-node levels in dynamic LDS shared by 8 waves, two blocks per CU (128
// registers).  The largest level of a 25,000-atom solute holds ~300 nodes;
// 1536-node levels with 16 waves per root (one block per CU) took 7 % longer
// on a batch of 50 6000-atom solutes, whose 3,200 queued roots keep every CU
// busy.  What still overflows is walked depth first: in pass A by the block's
// first wave in the same LDS (a launch of its own for those few roots cost
// 4.5 us on every call, mostly with nothing to walk), in pass B, whose walk
// would take this kernel past 128 registers (220 bytes of scratch per lane),
// by k_tree_dfs behind this kernel, beside the first tier.
constexpr int kBigWaves = 8;
template <int CAP, bool PB>
__global__ __launch_bounds__(64 * kBigWaves, 4) void k_tree_bfs_big(Dev d) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  using L = BfsLds<CAP, PB, kLevelCapBig, kBigWaves>;
  L &S = *reinterpret_cast<L *>(lds_raw);
  __shared__ int slot;
  const int count = (int)d.counters[4];
  unsigned *head = queue_head(d.queue, PB ? Q_TREE_BB : Q_TREE_BA);
  unsigned long long tk = 0, te = 0;
  for (int k = first_item(); k < count; k = next_item(head, &slot, count)) {
    const int h = d.tree_ovf[k];
    const bool done = tree_bfs_root<CAP, PB, kLevelCapBig, kBigWaves>(d, S, h, 1, tk, te);
    if constexpr (!PB) {
      if (!done && threadIdx.x < 64)
        tree_dfs_root<CAP, PB>(d, *reinterpret_cast<TreeLds<CAP, PB> *>(lds_raw), h, tk, te);
    }
  }
  add_tree_counts(d, PB, tk, te);
}

// pass B's depth-first walk of the roots its second tier listed: one wave each,
// as many at a time as the CUs hold, since a root here takes a millisecond or
// more where solutes are dense.  Calls of the synthetic solute, its coordinates
// scaled, with 64, 256 and 1,024 blocks: 6,000 atoms by 0.75 (824 roots here)
// 74.4, 30.4 and 21.7 ms, 25,000 by 0.8 (1,637 roots) 94.7, 33.5 and 21.5 ms.
// Blocks without a root cost nothing: 6,000 and 25,000 atoms as generated 299
// and 945 us with either number.
constexpr int kDfsBlocks = 1024;
template <int CAP>
__global__ __launch_bounds__(64) void k_tree_dfs(Dev d) {
  __shared__ TreeLds<CAP, true> S;
  const int count = (int)d.counters[7];
  unsigned long long tk = 0, te = 0;
  for (int k = blockIdx.x; k < count; k += gridDim.x) tree_dfs_root<CAP, true>(d, S, d.tree_ovf[d.nh + k], tk, te);
}

template <int CAP, bool PB>
static size_t big_lds() {
  return std::max(sizeof(BfsLds<CAP, PB, kLevelCapBig, kBigWaves>), PB ? 0 : sizeof(TreeLds<CAP, PB>));
}

hipError_t prepare_tree() {
  hipError_t e = hipSuccess;
  auto set = [&](const void *f, size_t bytes) {
    if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  };
  set((const void *)k_tree_bfs_big<64, false>, big_lds<64, false>());
  set((const void *)k_tree_bfs_big<64, true>, big_lds<64, true>());
  set((const void *)k_tree_bfs_big<128, false>, big_lds<128, false>());
  set((const void *)k_tree_bfs_big<128, true>, big_lds<128, true>());
  set((const void *)k_tree_bfs_big<256, false>, big_lds<256, false>());
  set((const void *)k_tree_bfs_big<256, true>, big_lds<256, true>());
  return e;
}

// the first tier a block per root unless a grid is asked for; the second a
// persistent grid of two blocks per CU
template <int CAP>
static void launch_tree_cap(const Dev &d, const Tuning &t, int pass, int tier, hipStream_t s) {
  const int g = std::min(d.nh, t.tree_grid > 0 ? t.tree_grid : d.nh), gf = std::min(d.nh, kDfsBlocks);
  const int gb = std::min(d.nh, 512);
  const size_t la = big_lds<CAP, false>(), lb = big_lds<CAP, true>();
  if (pass == 0) {
    if (tier == 0) hipLaunchKernelGGL((k_tree_bfs<first_cap(CAP), false>), dim3(g), dim3(64 * kFirstWaves), 0, s, d);
    if (tier == 1) hipLaunchKernelGGL((k_tree_bfs_big<CAP, false>), dim3(gb), dim3(64 * kBigWaves), la, s, d);
  } else {
    if (tier == 0) hipLaunchKernelGGL((k_tree_bfs<first_cap(CAP), true>), dim3(g), dim3(64 * kFirstWaves), 0, s, d);
    if (tier == 1) hipLaunchKernelGGL((k_tree_bfs_big<CAP, true>), dim3(gb), dim3(64 * kBigWaves), lb, s, d);
    if (tier == 1) hipLaunchKernelGGL((k_tree_dfs<CAP>), dim3(gf), dim3(64), 0, s, d);
  }
}

void launch_tree_tier(const Dev &d, const Tuning &t, int pass, int tier, hipStream_t s) {
  if (d.nh == 0) return;
  if (d.cap <= 64) launch_tree_cap<64>(d, t, pass, tier, s);
  else if (d.cap <= 128) launch_tree_cap<128>(d, t, pass, tier, s);
  else launch_tree_cap<256>(d, t, pass, tier, s);
}

void launch_tree(const Dev &d, const Tuning &t, int pass, hipStream_t s) {
  for (int tier = 0; tier < 2; tier++) launch_tree_tier(d, t, pass, tier, s);
}

}  // namespace agb
