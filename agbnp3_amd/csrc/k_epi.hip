// Per-atom epilogues in FP64: volume scaling factors and surface filter,
// Born radii, chain-rule factors, U/V coefficients, final gradient assembly
// (caller order) and the fixed-order energy reduction.
#include "agb_common.h"
#include "agb_device.h"

namespace agb {

constexpr int kEpi = 256;

// block sum of up to 4 doubles into epart[slot][blockIdx.x]; an atom block
// never spans two systems
__device__ void block_partials(const Dev &d, const int *slots, const double *v, int nv) {
  __shared__ double red[4][kEpi / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int k = 0; k < nv; k++) {
    const double s = wave_sum(v[k]);
    if (lane == 0) red[k][w] = s;
  }
  __syncthreads();
  if ((int)threadIdx.x < nv) {
    double s = 0.0;
    for (int q = 0; q < kEpi / 64; q++) s += red[threadIdx.x][q];
    d.epart[(size_t)slots[threadIdx.x] * d.nablk + blockIdx.x] = s;
  }
}

// near-pair total and longest row (counters 2, 3) and the first tree tier's
// counts: one add or max per block rather than per row (same-address atomics
// serialise in L2).  The grid has at least one block per 256 heavy rows.
__device__ __forceinline__ void row_counts(const Dev &d) {
  __shared__ unsigned red[4][kEpi / 64];
  const int h = blockIdx.x * kEpi + threadIdx.x;
  if (blockIdx.x * kEpi >= d.nh) return;             // block-uniform
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned v[4] = {0u, 0u, 0u, 0u};                  // pairs, longest row, overlaps kept, evaluated
  if (h < d.nh) {
    const uint2 c = d.tree_cnt[h];
    v[0] = v[1] = (unsigned)d.nne[h];
    v[2] = c.x;
    v[3] = c.y;
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const unsigned t = (unsigned)__shfl_xor((int)v[k], o, 64);
      v[k] = k == 1 ? max(v[k], t) : v[k] + t;
    }
    if (lane == 0) red[k][w] = v[k];
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    const int k = threadIdx.x;
    unsigned long long t = 0;
    for (int q = 0; q < kEpi / 64; q++) t = k == 1 ? max(t, (unsigned long long)red[k][q]) : t + red[k][q];
    unsigned long long *c = d.counters + kCountBase + 8 * (blockIdx.x % kCountSlots);
    if (k == 1) atomicMax(&d.counters[3], t);
    else if (t) atomicAdd(k == 0 ? &d.counters[2] : c + (k - 2), t);
  }
}

// ------------------------------------------------------- scaling factors
// agbnp3_scaling_factors (agbnp3_utils.c:524-613) with agbnp3_swf_area
// (agbnp3.c:1104-1117); E_cav, E_corr_cav, molecular volume
// (agbnp3.c:1390-1411)
__global__ __launch_bounds__(kEpi) void k_scale(Dev d) {
  row_counts(d);
  const int2 blk = d.ablk[blockIdx.x];
  const int i = blk.x + threadIdx.x;
  double ecav = 0.0, ecorr = 0.0, mv = 0.0;
  if (i < blk.y) {
    const SysInfo &S = d.sys[d.asys[i]];
    if (i < S.a0 + S.nh) {
      const double R = d.R[i];
      const double vraw = d.vols[i] + fix_get(d.acc_vol[i]);
      const double a = 4.0 * kPi * R * R + fix_get(d.acc_sa[i]);
      double f = 0.0, fp = 0.0;
      if (a >= 0.0) {
        const double t = a / (64.0 + a * a);
        f = a * t;
        fp = 2.0 * t * (1.0 - f);
      }
      const double saf = a * f;
      const double rv = (R - kRadInc) / R;
      const double pr = R * (1.0 - rv * rv * rv) / 3.0;
      const double vp = vraw - saf * pr;
      const double gp = ((double)d.igamma[i] + (double)d.sgamma[i]) * (f + a * fp);
      d.volumep_raw[i] = vraw;
      d.sa_raw[i] = a;
      d.sa_f[i] = saf;
      d.spe[i] = vraw / d.vols[i];
      d.psvol[i] = (fp * a + f) * pr;
      d.sp[i] = vp / d.vols[i];
      d.gammap[i] = gp;
      d.sp_f[i] = (float)d.sp[i];
      {                                 // the descreening's column record
        const float4 p = d.pos[i];
        const float iR = 1.0f / p.w;
        d.dcol[i] = make_float4(p.x, p.y, p.z, iR * d.tdxinv);   // d times .w: the table coordinate
        d.dcw[i] = make_float2(d.sp_f[i] * iR, __int_as_float(d.rtype[i]));
      }
      d.spe_f[i] = (float)d.spe[i];
      d.gammap_f[i] = (float)gp;
      ecav = (double)d.igamma[i] * saf;
      ecorr = (double)d.sgamma[i] * saf;
      mv = vp;
    } else {
      d.volumep_raw[i] = d.sa_raw[i] = d.sa_f[i] = d.spe[i] = d.psvol[i] = d.sp[i] = d.gammap[i] = 0.0;
      d.sp_f[i] = d.spe_f[i] = d.gammap_f[i] = 0.f;
    }
  }
  if (d.cull_desc) {                    // boxes of the descreening's column groups
    const bool col = i < blk.y && i < d.sys[d.asys[blk.x]].a0 + d.sys[d.asys[blk.x]].nh;
    float4 p = make_float4(0.f, 0.f, 0.f, 1.f);
    if (col) p = d.pos[i];
    Box b = box_of(col, p);
    float w = col ? 1.0f / p.w * d.tdxinv : INFINITY;
    box_union<kBoxCols>(b);
#pragma unroll
    for (int o = kBoxCols / 2; o > 0; o >>= 1) w = fminf(w, __shfl_xor(w, o, 64));
    if (threadIdx.x % kBoxCols == 0) {
      float4 *o = d.cbox + 2 * ((size_t)blockIdx.x * (kEpi / kBoxCols) + threadIdx.x / kBoxCols);
      o[0] = make_float4(b.lo[0], b.lo[1], b.lo[2], w);
      o[1] = make_float4(b.hi[0], b.hi[1], b.hi[2], 0.f);
    }
  }
  const int slots[3] = {EP_CAV, EP_CORR_CAV, EP_MOLVOL};
  const double v[3] = {ecav, ecorr, mv};
  block_partials(d, slots, v, 3);
}

void launch_scale(const Dev &d, hipStream_t s) {
  if (d.nablk) hipLaunchKernelGGL(k_scale, dim3(d.nablk), dim3(kEpi), 0, s, d);
}

// ------------------------------------------------------------ Born radii
// beta filter agbnp3_swf_invbr (agbnp3.c:1174-1188), agbnp3_born_radii
// (agbnp3_utils.c:615-670), E_vdW (agbnp3.c:1466-1487), GB self energy
__global__ __launch_bounds__(kEpi) void k_born(Dev d) {
  const int2 blk = d.ablk[blockIdx.x];
  const int i = blk.x + threadIdx.x;
  double evdw = 0.0, ecorr = 0.0, eself = 0.0;
  if (i < blk.y) {
    double s;
    if (d.dt_on) {
      // the tiles' FP32 sums, in runs of the columns that one of k_descreen's
      // items covers: added in FP64, rounded to the fixed point once per run
      const SysInfo &S = d.sys[d.asys[i]];
      const int nt = (S.nh + 255) / 256;
      const float *p = d.dpart + S.dp0 + (i - S.a0);
      // (eight tiles' loads in flight: 6,000 atoms 7.2 -> 5.2 us, 11,000, 21 tiles, 11.9 -> 6.5)
      long long sum = 0;
      double a = 0.0;
      int left = d.dt_run;                   // tiles of the run still to come
      for (int t0 = 0; t0 < nt; t0 += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = p[(size_t)min(t0 + u, nt - 1) * S.n];
        // (here, not each behind its test below)
        asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
#pragma unroll
        for (int u = 0; u < 8; u++) {
          if (t0 + u >= nt) break;
          a += (double)v[u];
          if (--left == 0 || t0 + u == nt - 1) {
            sum += __double2ll_rn(a * kFix);
            a = 0.0;
            left = d.dt_run;
          }
        }
      }
      s = fix_get(sum);
    } else {
      s = fix_get(d.acc_beta[i]);
    }
    if (d.sg_on && d.sys_sg[d.asys[i]]) {
      // surrogate call: the model's sum plus the correction of the last
      // anchor (an atom out of the training window keeps its descreening
      // sum); anchor call: record the surrogate's error and re-anchor
      const int mode = d.sg_state[4 * d.asys[i] + 2];
      const double sm = (double)d.sg_s[d.sg_slot[i]];      // the model's output is in slot order
      const double pred = sm + d.sg_c[i];
      if (mode == 1 || (mode == 2 && !d.sg_oor[i])) {
        s = pred;
      } else if (mode == 0) {
        d.sg_delta[i] = pred - s;
        d.sg_c[i] = s - sm;
        d.sg_target[i] = (float)s;
      }
    }
    const double beta = 1.0 / ((double)d.R[i] - kRadInc) - s / (4.0 * kPi);
    double bf, sw;
    if (beta < 0.0) {
      bf = 0.02;
      sw = 0.0;
    } else {
      bf = sqrt(0.02 * 0.02 + beta * beta);
      sw = beta / bf;
    }
    const double B = 1.0 / bf, t = B + kRwNp;
    d.beta[i] = beta;
    d.br[i] = B;
    d.br_f[i] = (float)B;
    d.swf[i] = sw;
    d.brw[i] = 3.0 * B * B / (t * t * t * t);
    const double a3 = 1.0 / (t * t * t);
    evdw = (double)d.ialpha[i] * a3;
    ecorr = (double)d.salpha[i] * a3;
    const double q = d.q[i];
    eself = d.sys[d.asys[i]].df64 * q * q / B;
  }
  const int slots[3] = {EP_VDW, EP_CORR_VDW, EP_SELF};
  const double v[3] = {evdw, ecorr, eself};
  block_partials(d, slots, v, 3);
}

void launch_born(const Dev &d, hipStream_t s) {
  if (d.nablk) hipLaunchKernelGGL(k_born, dim3(d.nablk), dim3(kEpi), 0, s, d);
}

// -------------------------------------------------- chain-rule factors
// (chain_factors), after the GB pairs
__global__ __launch_bounds__(kEpi) void k_q2ab(Dev d) {
  const int nblk = (d.n + kEpi - 1) / kEpi;
  if ((int)blockIdx.x >= nblk) {        // further blocks: the boxes of the chain rule's chunks
    const int slot = (blockIdx.x - nblk) * kEpi + threadIdx.x, a = d.cperm[slot];
    float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
    if (a >= 0) p = d.pos[a];
    Box b = box_of(a >= 0, p);
    box_union<64>(b);
    if ((threadIdx.x & 63) == 0) {
      d.chbox[2 * (slot >> 6)] = make_float4(b.lo[0], b.lo[1], b.lo[2], 0.f);
      d.chbox[2 * (slot >> 6) + 1] = make_float4(b.hi[0], b.hi[1], b.hi[2], 0.f);
    }
    return;
  }
  const int i = blockIdx.x * kEpi + threadIdx.x;
  if (i < d.n) chain_factors(d, i, fix_get(d.acc_gbA[i]));
}

void launch_q2ab(const Dev &d, hipStream_t s) {
  if (d.gbs_on) return;                 // (k_gb_sum's; no boxes at its sizes)
  const int boxes = d.cull_chain && d.nchain_items > kChainGroupItems ? d.ncblk : 0;
  hipLaunchKernelGGL(k_q2ab, dim3((d.n + kEpi - 1) / kEpi + boxes), dim3(kEpi), 0, s, d);
}

// ------------------------------------------------------ U, V coefficients
// for calls whose chain-rule sums k_chain_sum does not finish: a surrogate's
// gradient pass adds to them, or there are none (no heavy atoms)
__global__ __launch_bounds__(kEpi) void k_uv(Dev d) {
  const int i = blockIdx.x * kEpi + threadIdx.x;
  if (i >= d.n) return;
  const SysInfo &S = d.sys[d.asys[i]];
  for (int q = 0; q < 2; q++) uv_coeffs(d, i, S, q, d.acc_ch[8 * (size_t)i + 6 + q]);
}

void launch_uv(const Dev &d, hipStream_t s) {
  if (!d.sg_on && d.nchain_items) return;
  hipLaunchKernelGGL(k_uv, dim3((d.n + kEpi - 1) / kEpi), dim3(kEpi), 0, s, d);
}

// ---------------------------------------------------------------- energies
// fixed-order reduction of the per-block energy partials, GB tile pairs and
// site energies; one workgroup per system, energies[7 * system + k]; they need only the
// partials, so they run in the final launch beside the gradients
__device__ __forceinline__ void system_energies(const Dev &d, int sys, double *energies) {
  __shared__ double red[EP_COUNT][4];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const SysInfo S = d.sys[sys];
  double acc[EP_COUNT];
  for (int k = 0; k < EP_COUNT; k++) acc[k] = 0.0;
  // thread t sums partials t, t + 256, t + 512, ... in that order: a fixed
  // order that depends only on the system's own counts, with coalesced loads
  // (the loops unrolled so that several loads are in flight)
  for (int k = 0; k < EP_PAIR; k++)
#pragma unroll 8
    for (int b = t; b < S.nblk; b += 256) acc[k] += d.epart[(size_t)k * d.nablk + S.blk0 + b];
  // tile partials hold each unordered pair once; E_pair = 2 df sum_{i<j} q_i q_j / f
#pragma unroll 8
  for (int b = t; b < S.ntile; b += 256) acc[EP_PAIR] += 2.0 * S.df64 * d.gb_epart[S.tile0 + b];
#pragma unroll 8
  for (int b = t; b < S.nws; b += 256) acc[EP_HB] += d.ws_part[S.ws0 + b];
  for (int k = 0; k < EP_COUNT; k++) {
    const double s = wave_sum(acc[k]);
    if (lane == 0) red[k][w] = s;
  }
  __syncthreads();
  if (t == 0) {
    double e[EP_COUNT];
    for (int k = 0; k < EP_COUNT; k++) e[k] = red[k][0] + red[k][1] + red[k][2] + red[k][3];
    double *o = energies + 7 * (size_t)sys;
    o[0] = kTokcal * (e[EP_SELF] + e[EP_PAIR]);
    o[1] = e[EP_VDW];
    o[2] = e[EP_CORR_VDW];
    o[3] = e[EP_CAV];
    o[4] = e[EP_CORR_CAV];
    o[5] = e[EP_HB];
    o[6] = e[EP_MOLVOL];
  }
}

// ----------------------------------------------------------- final output
// gradients: GB = 332 (pair + chain + tree), vdW = chain + tree,
// cavity = tree, HB = direct + tree (agbnp3.c:1718-1786); caller order.  The
// outputs may lie in host memory, so a block's gradients go through LDS and
// leave as whole lines; the call's status goes there too (hstat), which saves
// the host three copies of their own launch and wait each.
__global__ __launch_bounds__(kEpi) void k_final(Dev d, double *sp, double *br, double *sa, double *dgbdr,
                                                double *dvwdr, double *decav, double *dehb, double *energies) {
  __shared__ double out[4][3 * kEpi];
  if ((int)blockIdx.x < d.nsys) {                    // the first blocks: a system's energies each
    if (blockIdx.x == 0 && d.hstat && threadIdx.x < 5)
      d.hstat[threadIdx.x] = threadIdx.x == 0 ? (unsigned long long)(unsigned)*d.status : d.counters[threadIdx.x - 1];
    system_energies(d, blockIdx.x, energies);
    return;
  }
  const int e0 = (blockIdx.x - d.nsys) * kEpi, e = e0 + threadIdx.x;
  if (e < d.n) {
    const int i = d.ext2int[e];
    const SysInfo &S = d.sys[d.asys[i]];
    const bool heavy = i < S.a0 + S.nh;
    const double df = S.df64;
    double g_gb[3], g_vw[3];
    const double f4 = 1.0 / (4.0 * kPi);
    for (int q = 0; q < 3; q++) {
      g_gb[q] = 2.0 * df * fix_get(d.acc_gbg[3 * (size_t)i + q]) + df * f4 * fix_get(d.acc_ch[8 * (size_t)i + q]);
      g_vw[q] = f4 * fix_get(d.acc_ch[8 * (size_t)i + 3 + q]);
    }
    double g_cav[3] = {0, 0, 0}, g_hb[3];
    for (int q = 0; q < 3; q++) g_hb[q] = fix_get(d.acc_hb[3 * (size_t)i + q]);
    if (heavy) {
      const long long *t = d.acc_grad + (size_t)i * TG_N;
      for (int q = 0; q < 3; q++) {
        g_gb[q] += fix_get(t[TG_GB + q]);
        g_vw[q] += fix_get(t[TG_VW + q]);
        g_cav[q] = fix_get(t[TG_CAV + q]);
        g_hb[q] += fix_get(t[TG_HB + q]);
      }
    }
    for (int q = 0; q < 3; q++) {
      out[0][3 * threadIdx.x + q] = kTokcal * g_gb[q];
      out[1][3 * threadIdx.x + q] = g_vw[q];
      out[2][3 * threadIdx.x + q] = g_cav[q];
      out[3][3 * threadIdx.x + q] = g_hb[q];
    }
    sp[e] = heavy ? d.sp[i] : 1.0;
    br[e] = d.br[i];
    sa[e] = heavy ? d.sa_f[i] : 0.0;
  }
  __syncthreads();
  double *const dst[4] = {dgbdr, dvwdr, decav, dehb};
  const int m = 3 * min(kEpi, d.n - e0);
#pragma unroll
  for (int k = 0; k < 4; k++)
    for (int q = threadIdx.x; q < m; q += kEpi) dst[k][3 * (size_t)e0 + q] = out[k][q];
}

void launch_final(const Dev &d, double *sp, double *br, double *sa, double *dgbdr, double *dvwdr, double *decav,
                  double *dehb, double *energies, hipStream_t s) {
  hipLaunchKernelGGL(k_final, dim3(d.nsys + (d.n + kEpi - 1) / kEpi), dim3(kEpi), 0, s, d, sp, br, sa, dgbdr, dvwdr,
                     decav, dehb, energies);
}

}  // namespace agb
