// Device helpers shared by the kernel translation units: wavefront (64-lane)
// reductions and scans, cell-grid indexing, order-independent fixed-point
// scatter, and the FP32 Gaussian-overlap / spline primitives of the model.
#pragma once
#include <hip/hip_runtime.h>

#include "agb_common.h"

namespace agb {

// ---------------------------------------------------------- wave collectives
// Sums and scans over the 64 lanes with DPP moves (no LDS round trips):
// row_shr:1, 2, 4, 8 with zero fill give every lane the inclusive prefix of
// its 16-lane row; row_bcast:15 into rows 1 and 3 and row_bcast:31 into
// rows 2 and 3 extend it over the wave, so lane 63 ends with the total.
// Every lane of the wave must be active.
namespace dpp {
constexpr int kShr1 = 0x111, kShr2 = 0x112, kShr4 = 0x114, kShr8 = 0x118, kBcast15 = 0x142, kBcast31 = 0x143;
// src moved by CTRL into the rows of ROWS; 0 where a row is masked out or the
// source lane lies outside the row
template <int CTRL, int ROWS>
__device__ __forceinline__ int mov(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, true); }
template <int CTRL, int ROWS>
__device__ __forceinline__ float mov(float v) { return __builtin_bit_cast(float, mov<CTRL, ROWS>(__builtin_bit_cast(int, v))); }
template <int CTRL, int ROWS>
__device__ __forceinline__ double mov(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = mov<CTRL, ROWS>((int)(b & 0xffffffffll)), hi = mov<CTRL, ROWS>((int)(b >> 32));
  return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
template <typename T>
__device__ __forceinline__ T incl_scan(T v) {
  v += mov<kShr1, 0xf>(v);
  v += mov<kShr2, 0xf>(v);
  v += mov<kShr4, 0xf>(v);
  v += mov<kShr8, 0xf>(v);
  v += mov<kBcast15, 0xa>(v);
  v += mov<kBcast31, 0xc>(v);
  return v;
}
__device__ __forceinline__ float lane63(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
}  // namespace dpp

// the value of one lane (wave-uniform index) in every lane
__device__ __forceinline__ double lane_value(double v, int lane) {
  const long long b = __builtin_bit_cast(long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}

// order the LDS accesses of one wave (its LDS instructions execute in program
// order; this keeps the compiler from moving them)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the wave's total, in every lane (a fixed order of additions)
__device__ __forceinline__ float wave_sum(float v) { return dpp::lane63(dpp::incl_scan(v)); }
__device__ __forceinline__ double wave_sum(double v) { return lane_value(dpp::incl_scan(v), 63); }
__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ int wave_incl_scan(int v) { return dpp::incl_scan(v); }

// --------------------------------------------------------------- far boxes
// The spline tables end in a zero interval (coordinate d / (R dx) >= kTblN - 1
// in FP32), so pairs past it add exact zeros and leave every sum as it is.
// Boxes of atoms decide it for many pairs at once: kFarCoord leaves 0.1 % for
// the rounding of boxes and coordinates.  A box with an atom that is not
// finite is the whole space, so its pairs are evaluated.
constexpr float kFarCoord = (float)(kTblN - 1) * 1.001f;
struct Box {
  float lo[3], hi[3];
};
__device__ __forceinline__ Box box_of(bool valid, const float4 &p) {
  Box b;
  const float v[3] = {p.x, p.y, p.z};
  const bool fin = fabsf(p.x) < INFINITY && fabsf(p.y) < INFINITY && fabsf(p.z) < INFINITY;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    b.lo[k] = !valid ? INFINITY : (fin ? v[k] : -INFINITY);
    b.hi[k] = !valid ? -INFINITY : (fin ? v[k] : INFINITY);
  }
  return b;
}
// the union over groups of W lanes, in every lane of the group
template <int W>
__device__ __forceinline__ void box_union(Box &b) {
#pragma unroll
  for (int o = W / 2; o > 0; o >>= 1)
#pragma unroll
    for (int k = 0; k < 3; k++) {
      b.lo[k] = fminf(b.lo[k], __shfl_xor(b.lo[k], o, 64));
      b.hi[k] = fmaxf(b.hi[k], __shfl_xor(b.hi[k], o, 64));
    }
}
// squared distance between two boxes (infinite when one is empty)
__device__ __forceinline__ float box_gap2(const Box &a, const float4 &lo, const float4 &hi) {
  const float x = fmaxf(0.f, fmaxf(a.lo[0] - hi.x, lo.x - a.hi[0]));
  const float y = fmaxf(0.f, fmaxf(a.lo[1] - hi.y, lo.y - a.hi[1]));
  const float z = fmaxf(0.f, fmaxf(a.lo[2] - hi.z, lo.z - a.hi[2]));
  return x * x + y * y + z * z;
}

// ------------------------------------------------------------ work queues
// Persistent blocks take work items from a queue head in memory; every block
// leaves once the head has passed the item count, so the grid always drains.
// A block's first item (or run of n items) is its own index: the whole grid
// starting at once would otherwise queue on the head's one address.  Later
// items come from the head, offset past those.  `slot` is block-shared
// scratch for the broadcast.
// The later items are spread over S = min(kQueueSpread, gridDim) heads
// (every head has a block): head x hands out items gridDim + S c + x
// (c = 0, 1, ...) to the blocks with blockIdx mod S = x.
__device__ __forceinline__ unsigned *queue_head(unsigned *queue, int which) {
  return queue + which * kQueueSpread * kQueueStride;
}
__device__ __forceinline__ int first_item() { return (int)blockIdx.x; }
// (A grid with a block per item asks no head: the answer, a microsecond away
// behind the block's own scatter, would only hold its place on the CU.)
__device__ __forceinline__ int next_item(unsigned *head, int *slot, int count) {
  if ((int)gridDim.x >= count) return count;
  __syncthreads();                       // the previous item is finished by all waves
  if (threadIdx.x == 0) {
    const unsigned S = min((unsigned)kQueueSpread, gridDim.x), x = blockIdx.x % S;
    *slot = (int)(gridDim.x + S * atomicAdd(head + x * kQueueStride, 1u) + x);
  }
  __syncthreads();
  return *slot;
}

// ------------------------------------------------------------------ cells
__device__ __forceinline__ void cell_coords(const GridParams &g, float x, float y, float z, int &cx, int &cy,
                                            int &cz) {
  cx = min(max((int)floorf((x - g.lo[0]) * g.inv_cs), 0), g.dim[0] - 1);
  cy = min(max((int)floorf((y - g.lo[1]) * g.inv_cs), 0), g.dim[1] - 1);
  cz = min(max((int)floorf((z - g.lo[2]) * g.inv_cs), 0), g.dim[2] - 1);
}
__device__ __forceinline__ int cell_index(const GridParams &g, float x, float y, float z) {
  int cx, cy, cz;
  cell_coords(g, x, y, z, cx, cy, cz);
  return (cz * g.dim[1] + cy) * g.dim[0] + cx;
}

// Bounding box of atoms [a0, a0 + count) by one 1024-thread block: lo[3],
// hi[3] valid in thread 0 (box is block-shared scratch [6][16]); empty
// ranges give lo = +inf, hi = -inf.
__device__ __forceinline__ void block_bbox(const float4 *pos, int a0, int count, float (*box)[16], float *lo,
                                           float *hi) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  float l[3] = {INFINITY, INFINITY, INFINITY}, h[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int k0 = t; k0 < count; k0 += 4 * 1024) {     // (four loads in flight; an atom met twice changes nothing)
    float4 p[4];
#pragma unroll
    for (int u = 0; u < 4; u++) p[u] = pos[a0 + min(k0 + 1024 * u, count - 1)];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      l[0] = fminf(l[0], p[u].x); l[1] = fminf(l[1], p[u].y); l[2] = fminf(l[2], p[u].z);
      h[0] = fmaxf(h[0], p[u].x); h[1] = fmaxf(h[1], p[u].y); h[2] = fmaxf(h[2], p[u].z);
    }
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float a = wave_min(l[k]), b = wave_max(h[k]);
    if (lane == 0) { box[k][w] = a; box[3 + k][w] = b; }
  }
  __syncthreads();
  if (t == 0)
    for (int k = 0; k < 3; k++) {
      lo[k] = box[k][0];
      hi[k] = box[3 + k][0];
      for (int q = 1; q < 16; q++) { lo[k] = fminf(lo[k], box[k][q]); hi[k] = fmaxf(hi[k], box[3 + k][q]); }
    }
}

// Grid over the box [lo, hi] with cells of at least `cs`, grown by 5 % steps
// until it has at most kMaxCells cells.
__device__ __forceinline__ GridParams make_grid(const float *lo_in, const float *hi_in, float cs) {
  GridParams g;
  float ext[3];
  for (int k = 0; k < 3; k++) {
    float lo = lo_in[k], hi = hi_in[k];
    if (!(hi >= lo)) { lo = 0.f; hi = 0.f; }    // no atoms
    g.lo[k] = lo - 1e-3f;
    ext[k] = hi - lo + 2e-3f;
    if (!(ext[k] < 1e7f)) ext[k] = 1e7f;          // non-finite input: keep the loop finite
  }
  for (;;) {
    long long nc = 1;
    for (int k = 0; k < 3; k++) {
      g.dim[k] = (int)floorf(ext[k] / cs) + 1;
      nc *= g.dim[k];
    }
    if (nc <= kMaxCells) { g.ncell = (int)nc; break; }
    cs *= 1.05f;
  }
  g.cs = cs;
  g.inv_cs = 1.0f / cs;
  return g;
}

// Counting sort of atoms [a0, a0 + count) into the cells of g by one
// 1024-thread block: start[c] is the first slot of cell c (start[ncell] =
// a0 + count) and out[start[c] ..] its atoms.  cnt (kMaxCells ints), wsum
// and wpre (16 ints) are block-shared scratch, cell_of[a0 ..] global scratch.
// The order inside a cell follows the arrival of the atomic adds; with
// `sorted` each cell is then put in atom order.
__device__ __forceinline__ void bin_atoms(const GridParams &g, const float4 *pos, int a0, int count, int *cell_of,
                                          int *start, int *out, int *cnt, int *wsum, int *wpre, bool sorted) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int ncell = g.ncell;
  for (int c = t; c < ncell; c += 1024) cnt[c] = 0;
  __syncthreads();
  for (int k0 = t; k0 < count; k0 += 4 * 1024) {     // four loads in flight
    float4 p[4];
#pragma unroll
    for (int u = 0; u < 4; u++) p[u] = pos[a0 + min(k0 + 1024 * u, count - 1)];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (k0 + 1024 * u < count) {
        const int c = cell_index(g, p[u].x, p[u].y, p[u].z);
        cell_of[a0 + k0 + 1024 * u] = c;
        atomicAdd(&cnt[c], 1);
      }
  }
  __syncthreads();
  // exclusive scan of cnt over the cells, contiguous cells per thread
  const int per = (ncell + 1023) / 1024;
  int local = 0;
  for (int k = 0; k < per; k++) {
    const int c = t * per + k;
    if (c < ncell) local += cnt[c];
  }
  const int incl = wave_incl_scan(local);
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  if (t < 16) {
    int s = 0;
    for (int q = 0; q < t; q++) s += wsum[q];
    wpre[t] = s;
  }
  __syncthreads();
  int run = a0 + incl - local + wpre[w];
  for (int k = 0; k < per; k++) {
    const int c = t * per + k;
    if (c < ncell) {
      const int v = cnt[c];
      start[c] = run;
      cnt[c] = run;                  // cursor
      run += v;
    }
  }
  if (t == 0) start[ncell] = a0 + count;
  __syncthreads();
  for (int k0 = t; k0 < count; k0 += 4 * 1024) {
    int c[4];
#pragma unroll
    for (int u = 0; u < 4; u++) c[u] = cell_of[a0 + min(k0 + 1024 * u, count - 1)];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (k0 + 1024 * u < count) out[atomicAdd(&cnt[c[u]], 1)] = a0 + k0 + 1024 * u;
  }
  if (!sorted) return;
  __syncthreads();
  for (int c = t; c < ncell; c += 1024) {     // insertion sort of each (short) cell
    const int b = start[c], e = start[c + 1];
    for (int k = b + 1; k < e; k++) {
      const int v = out[k];
      int q = k - 1;
      while (q >= b && out[q] > v) {
        out[q + 1] = out[q];
        q--;
      }
      out[q + 1] = v;
    }
  }
  __syncthreads();
}

// The 27-cell stencil around cell (cx, cy, cz) as 9 segments of the
// cell-sorted atoms (the three x-neighbour cells of one (y, z) are
// consecutive in the sort), their bounds loaded by lanes 0..8 at once.
// Candidate k (0 <= k < the returned total) of the stencil is atom slot
// stencil_slot(start, off, k); candidates come segment by segment.
__device__ __forceinline__ int stencil_segments(const GridParams &g, const int *cstart, int cx, int cy, int cz,
                                                int (&start)[9], int (&off)[9]) {
  const int lane = threadIdx.x & 63;
  int sbeg = 0, slen = 0;
  if (lane < 9) {
    const int zz = cz + lane / 3 - 1, yy = cy + lane % 3 - 1;
    if (zz >= 0 && zz < g.dim[2] && yy >= 0 && yy < g.dim[1]) {
      const int c0 = (zz * g.dim[1] + yy) * g.dim[0];
      sbeg = cstart[c0 + max(cx - 1, 0)];
      slen = cstart[c0 + min(cx + 1, g.dim[0] - 1) + 1] - sbeg;
    }
  }
  const int incl = wave_incl_scan(slen);
#pragma unroll
  for (int q = 0; q < 9; q++) {
    start[q] = __shfl(incl - slen, q, 64);
    off[q] = __shfl(sbeg, q, 64) - start[q];
  }
  return __shfl(incl, 8, 64);
}
__device__ __forceinline__ int stencil_slot(const int (&start)[9], const int (&off)[9], int k) {
  // off[q] for the last q with start[q] <= k (empty segments share the next
  // one's start), as a sum of steps: a select chain here is turned into an
  // indexed load of off[] from scratch memory
  int o = off[0];
#pragma unroll
  for (int q = 1; q < 9; q++) o += k >= start[q] ? off[q] - off[q - 1] : 0;
  return o + k;
}

// Block index remapped so that each XCD (blocks are dealt to the 8 XCDs in
// turn) works on one contiguous share of the index range, which keeps the
// data of neighbouring blocks in the same L2.
__device__ __forceinline__ int xcd_block(int b, int nb) {
  const int x = b & 7, l = b >> 3, q = nb >> 3, rem = nb & 7;
  return x * q + min(x, rem) + l;
}

// -------------------------------------------------- fixed-point scatter add
// Each contribution is rounded to 2^-32 once, so sums are exact and their
// value does not depend on the order in which waves arrive.
__device__ __forceinline__ void fix_add(long long *p, double v) {
  if (v != 0.0) atomicAdd((unsigned long long *)p, (unsigned long long)__double2ll_rn(v * kFix));
}
__device__ __forceinline__ double fix_get(long long v) { return (double)v * kFixInv; }

// ----------------------------------------------------- chain-rule factors
// q2ab = (q^2 + A B) swf', abrw = alpha brw swf' (kernels.c:433-450).  The
// FP32 copies are the chain rule's weights: on a surrogate call with
// out-of-range atoms (mode 2) only those atoms' radii come from the
// descreening, so every other atom's chain-rule weight is zero (the
// surrogate's gradient pass weighs them from the FP64 values)
__device__ __forceinline__ void chain_factors(const Dev &d, int i, double A) {
  const double q = d.q[i];
  const double q2ab = (q * q + A * d.br[i]) * d.swf[i];
  const double abrw = ((double)d.ialpha[i] + (double)d.salpha[i]) * d.brw[i] * d.swf[i];
  d.A[i] = A;
  d.q2ab[i] = q2ab;
  d.abrw[i] = abrw;
  const bool chain = !d.sg_on || d.sg_state[4 * d.asys[i] + 2] != 2 || d.sg_oor[i];
  d.q2ab_f[i] = chain ? (float)q2ab : 0.f;
  d.abrw_f[i] = chain ? (float)abrw : 0.f;
}

// ------------------------------------------------- U, V coefficients
// deru = U/V_i, derus = df/(4pi) psvol deru, dervs = psvol derv/(4pi)
// (kernels.c:861-875), from the chain rule's sums (which = 0: U, and H_i of
// the water sites with it; 1: V)
__device__ __forceinline__ void uv_coeffs(const Dev &d, int i, const SysInfo &S, int which, long long sum) {
  const bool heavy = i < S.a0 + S.nh;
  const double der = heavy ? fix_get(sum) / d.vols[i] : 0.0;
  const double f4 = 1.0 / (4.0 * kPi);
  if (which == 0) {
    const double ders = S.df64 * f4 * d.psvol[i] * der, h = heavy ? fix_get(d.acc_derh[i]) : 0.0;
    d.deru[i] = der;
    d.derus[i] = ders;
    d.derh[i] = h;
    d.deru_f[i] = (float)der;
    d.derus_f[i] = (float)ders;
    d.derh_f[i] = (float)h;
  } else {
    const double ders = f4 * d.psvol[i] * der;
    d.derv[i] = der;
    d.dervs[i] = ders;
    d.derv_f[i] = (float)der;
    d.dervs_f[i] = (float)ders;
  }
}

// ------------------------------------------------- overlap-volume switch
// quintic smoothstep of the raw overlap volume on [0.01, 0.1]
// (reference agbnp3_cpu_simd_kernels.c:2448-2471)
__device__ __forceinline__ void vol_switch(float v, float &s, float &sp, float &spp) {
  if (v > kVolMinB) { s = 1.f; sp = 0.f; spp = 0.f; return; }
  if (v < kVolMinA) { s = 0.f; sp = 0.f; spp = 0.f; return; }
  const float d = 1.0f / (kVolMinB - kVolMinA);
  const float u = (v - kVolMinA) * d, u2 = u * u;
  s = u2 * u * fmaf(6.f, u2, fmaf(-15.f, u, 10.f));     // (fused as written: overlap(), k_tree.hip)
  sp = d * 30.f * u2 * (1.f - 2.f * u + u2);
  spp = d * d * 60.f * u * (1.f - 3.f * u + 2.f * u2);
}

// --------------------------------------------------------- Q4 spline value
// Node pairs (y_k, z_k) of one table, z_k = y''_k dx^2 / 6 times zs (zs = 1
// for nodes staged with that factor applied, dx^2 / 6 for the pack's
// (y, y'') nodes); xh = d / (R_j dx), the coordinate on the table's grid of
// [0, 20) in d / R_j; k > 510 is the flat zero tail (agbnp3_utils.c:331-377,
// 266-295).  The cubic spline's value with B the fraction and A = 1 - B,
//   A y_k + B y_k+1 + (A^3 - A) z_k + (B^3 - B) z_k+1,
// is formed as A y_k + B y_k+1 - A B ((A + 1) z_k + (B + 1) z_k+1), since
// A^3 - A = A (A - 1)(A + 1) = -A B (A + 1) and likewise for B (fewer
// operations, and no cancellation in A^3 - A as B -> 0).
__device__ __forceinline__ float q4_value(const float2 *__restrict__ tab, float xh, float zs) {
  const int k = (int)xh;
  float q = 0.f;
  if (k >= 0 && k <= kTblN - 2) {
    const float2 n0 = tab[k], n1 = tab[k + 1];
    // xh >= 0 here, so its fraction is xh - k, exactly
    const float B = __builtin_amdgcn_fractf(xh), A = 1.f - B;
    const float z0 = n0.y * zs, z1 = n1.y * zs;
    const float c = fmaf(B, z1, fmaf(A, z0, z0 + z1));
    q = fmaf(-(A * B), c, fmaf(A, n0.x, B * n1.x));
  }
  return q;
}

}  // namespace agb
