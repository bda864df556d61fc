// All-pairs kernels: pairwise descreening (inverse Born radii), GB pair
// energy with A_i and the constant-B gradient, and the chain rule at
// constant self volumes fused with U_i / V_i.
//
// Work decomposition: each kernel has a list of work items, sorted by
// decreasing size, and a queue head; a grid of persistent blocks takes items
// until the list is exhausted, so systems of very different size (a batch)
// share one launch with balanced load.
//
// Descreening: an item is a block of rows of one radius type and one system
// against a range of that system's columns; the block stages the spline
// tables its rows can use in LDS, every lane reads the same column at the
// same step through scalar loads, and each row (one per thread) sums a
// 256-column tile in FP32.  GB pairs
// and the chain rule: an item is a pair of 256-atom tiles of one system.
// Their sums leave each item through order-independent fixed-point atomics
// (descreening, GB pairs) or as per-item partial sums that k_chain_sum adds
// in a fixed order (chain rule), so results are bitwise reproducible
// whatever the schedule.
#include <type_traits>

#include <climits>
#include "agb_common.h"
#include "agb_device.h"

namespace agb {

constexpr int kTile = 256;

// stage the spline tables [t][*] (ROW_FIRST) or [*][t] of row type t as
// (y, y'' zs) nodes
template <int ROWS>
__device__ __forceinline__ void stage_tables(const Dev &d, float2 *dst, int t, bool row_first, float zs) {
  const int nt = d.ntypes;
  for (int k = threadIdx.x; k < nt * kTblN; k += ROWS) {
    const int tj = k / kTblN, node = k - tj * kTblN;
    const int tab = row_first ? t * nt + tj : tj * nt + t;
    const float2 v = d.tbl[(size_t)tab * kTblN + node];
    dst[k] = make_float2(v.x, v.y * zs);
  }
}

// ------------------------------------------------------------ descreening
// beta_i = 1/(R_i - 0.5) - (1/4pi) sum_{j heavy, j != i} sp_j Q4(d_ij; i <- j)
// Q4 = f(d/R_j)/R_j from table [rtype_i][rtype_j]
// (reference agbnp3_inverse_born_radii_nolist_soa, kernels.c:500-678)
// GTAB: more radius types than kLdsTypes; the tables are read through the
// caches from the pack's table array instead of LDS.

// CULL (large solutes): columns are taken in groups of 16 whose boxes
// (k_scale) the wave's rows, close in space, may pass over as past the tables.
template <int ROWS, bool GTAB, bool CULL>
__global__ __launch_bounds__(ROWS) void k_descreen(Dev d, const float4 *__restrict__ ccol,
                                                  const float2 *__restrict__ cwt) {
  extern __shared__ float2 dyn_tab[];     // [ntypes][512]: tables [t_row][*]
  float2 (*tab)[kTblN] = reinterpret_cast<float2 (*)[kTblN]>(dyn_tab);
  __shared__ int slot;
  if (d.sg_on && !*d.sg_any_plain) return;   // every system on the surrogate this call (grid-uniform)
  const float dx_ = d.tdx, dp2 = dx_ * (dx_ / 6.0f);   // the spline's dx^2 / 6
  // a column is the same for every lane: its record (ccol, cwt: d.dcol and
  // d.dcw, written by k_scale) comes through scalar loads, its table base is
  // scalar arithmetic
  int staged = -1;
  for (int it0 = first_item(); it0 < d.ndesc_items;
       it0 = next_item(queue_head(d.queue, Q_DESC), &slot, d.ndesc_items)) {
    const int it = __builtin_amdgcn_readfirstlane(it0);
    const int4 item = d.desc_items[it];
    const int i = d.row_perm[item.x * ROWS + threadIdx.x];
    if (d.sg_on) {
      const int mode = d.sg_state[4 * d.rblk[item.x].y + 2];   // item-uniform
      if (mode == 1) continue;                                   // surrogate call for this system
      // surrogate call with the plain kernels for out-of-range atoms: only
      // row blocks holding one
      if (mode == 2 && !__syncthreads_or(i >= 0 && d.sg_oor[i] != 0)) continue;
    }
    const int t = d.rblk[item.x].x;
    if (!GTAB && t != staged) {        // uniform: every thread reads the same item
      stage_tables<ROWS>(d, dyn_tab, t, true, dp2);
      staged = t;
      __syncthreads();
    }
    const float2 *gtab = d.tbl + (size_t)t * d.ntypes * kTblN;   // tables [t][*] (GTAB)
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i >= 0) pi = d.pos[i];
    if (__ballot(i >= 0) == 0ull) continue;      // a wave of padding rows (the barriers are all in the queue and above)
    const int c0 = item.y, c1 = item.z;
    constexpr int kGroups = kTile / kBoxCols;
    const SysInfo &S = d.sys[d.rblk[item.x].y];
    Box rows{};
    if (CULL) {
      rows = box_of(i >= 0, pi);
      box_union<64>(rows);
    }
    unsigned long long near = ~0ull;     // column groups of the next four tiles that the wave's rows reach
    double acc = 0.0;
    for (int base = c0; base < c1; base += kTile, near >>= kGroups) {
      const int nc = min(kTile, c1 - base);
      if (CULL && ((base - c0) & (4 * kTile - 1)) == 0) {
        const float4 *box = d.cbox + 2 * (size_t)(S.blk0 * kGroups + (base - S.a0) / kBoxCols + (int)(threadIdx.x & 63));
        bool reach = false;
        if (base + (int)(threadIdx.x & 63) * kBoxCols < c1) {
          const float4 lo = box[0], hi = box[1];
          reach = !(box_gap2(rows, lo, hi) * (lo.w * lo.w) > kFarCoord * kFarCoord);
        }
        near = __ballot(reach);
      }
      unsigned groups = (unsigned)near & ((1u << kGroups) - 1u);
      if (CULL && groups == 0) continue;   // (its sum would be an exact zero)
      float tacc = 0.f;
      // every lane runs the loop (a padding row, i < 0, at the origin: its sum
      // is dropped), so the column index stays wave-uniform.  Only a tile
      // holding one of the wave's own rows among its columns tests for the
      // self pair.
      auto tile = [&](auto self) {
        auto column = [&](int j, const float4 &pj, const float2 &w) {
          const float ex = pj.x - pi.x, ey = pj.y - pi.y, ez = pj.z - pi.z;
          const float dist = __builtin_amdgcn_sqrtf(ex * ex + ey * ey + ez * ez);   // hardware square root (1 ulp)
          const float2 *row = GTAB ? gtab + (size_t)__float_as_int(w.y) * kTblN : tab[__float_as_int(w.y)];
          const float q = q4_value(row, dist * pj.w, GTAB ? dp2 : 1.f);   // LDS nodes carry dx^2 / 6
          // the same FMA either way: a pair's term does not depend on its tile's test
          tacc = fmaf(q, (decltype(self)::value && j == i) ? 0.f : w.x, tacc);
        };
        auto columns = [&](int c, int ce) {
          for (; c + 4 <= ce; c += 4) {                 // four columns' records in two scalar loads
            float4 pj[4];
            float2 w[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
              pj[u] = ccol[base + c + u];
              w[u] = cwt[base + c + u];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) column(base + c + u, pj[u], w[u]);   // sums stay in column order
          }
          for (; c < ce; c++) column(base + c, ccol[base + c], cwt[base + c]);
        };
        if (!CULL) columns(0, nc);
        else
          while (groups) {                              // runs of near groups, in column order
            const int g = __builtin_ctz(groups), run = __builtin_ctz(~(groups >> g));
            groups &= ~(((1u << run) - 1u) << g);
            columns(g * kBoxCols, min(nc, (g + run) * kBoxCols));
          }
      };
      if (__ballot(i >= base && i < base + nc) != 0ull) tile(std::true_type{});
      else tile(std::false_type{});
      acc += (double)tacc;
    }
    if (i >= 0) fix_add(&d.acc_beta[i], acc);
  }
}

void launch_descreen(const Dev &d, const Tuning &t, hipStream_t s) {
  if (!d.ndesc_items) return;
  const bool gtab = d.ntypes > kLdsTypes;
  const size_t lds = gtab ? 0 : (size_t)d.ntypes * kTblN * sizeof(float2);
  int grid = t.desc_grid > 0 ? std::min(t.desc_grid, d.ndesc_items) : d.ndesc_items;
  if (d.sg_on) grid = std::min(grid, kSgPersistentGrid);   // calls where every block leaves at once
  const float4 *ccol = d.dcol;
  const float2 *cwt = d.dcw;
  const int m = gtab ? 0 : (d.cull_desc ? 2 : 1);
  const auto pick = [&](auto g, auto plain, auto cull) { return m == 0 ? g : (m == 1 ? plain : cull); };
  const auto k = d.rows == 64 ? pick(k_descreen<64, true, false>, k_descreen<64, false, false>, k_descreen<64, false, true>)
               : d.rows == 128
                   ? pick(k_descreen<128, true, false>, k_descreen<128, false, false>, k_descreen<128, false, true>)
                   : pick(k_descreen<256, true, false>, k_descreen<256, false, false>, k_descreen<256, false, true>);
  hipLaunchKernelGGL(k, dim3(grid), dim3(d.rows), lds, s, d, ccol, cwt);
}

// ------------------------------------------------------------- GB pairs
// Each unordered pair once (agbnp3_gb_energy_inner_nolist_soa, kernels.c:66-151):
//   e   = q_i q_j / f,  f = sqrt(d2 + B_i B_j exp(-d2 / 4 B_i B_j))
//   g_i += q_i q_j (1 - e/4) / f^3 (x_j - x_i),  g_j -= same      (x 2 df later)
//   A_i, A_j += q_i q_j (B_i B_j + d2/4) exp(.) / f^3
// An item is a tile pair of up to 256 x 256 atoms of one system, its columns
// staged in LDS.  Wave w holds rows lane + 64 k, k = 0..3 -- every row of the
// tile, four per lane -- and sweeps the 64 columns of chunk w: at step s lane
// l reads column (l - s) mod 64 of the chunk, adds the four rows' terms to
// the column's partial sums, and those move on by one lane per step, so every
// lane meets every column once and the sums end where they started (one column
// read and one rotation per four pairs).  A row's
// sums over the four waves' chunks are added in wave order through LDS.
// Diagonal tiles see each pair twice and keep only the row side.
// Bound: VALU issue.  On this GPU two waves of a SIMD can each issue an FP32
// add, multiply or multiply-add in the same four cycles, but a DPP move and a
// transcendental stop both for about twenty; so the column sums rotate
// through the LDS crossbar (ds_bpermute; LDS is otherwise nearly idle here)
// instead of four DPP moves per step, and 98 registers, four waves per SIMD,
// are enough.  With that and without the mask's compare and select per pair
// off the diagonal: 25,000 atoms 0.262 -> 0.234 ms, 150,000 8.38 -> 7.95 ms
// (the clock falls to 2.0 GHz there), 24 x 6000 0.364 -> 0.357 ms.
__device__ __forceinline__ float wave_rot(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x13C, 0xF, 0xF, true));
}

// the same rotation through the LDS crossbar (rot_from: the byte address of
// the lane that lane l takes its value from)
__device__ __forceinline__ int rot_from(int lane) { return ((lane + 63) & 63) * 4; }
__device__ __forceinline__ float lds_rot(float v, int from) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, v)));
}

// one row's GB pair terms with one column
struct GbRow {
  float x, y, z, q, b, qib;     // position, charge, Born radius, -log2(e) / (4 B)
};
// its terms: q_i q_j and 1/f, x_j - x_i, the gradient's, and A's two factors.  MASK: the
// reference's mask (kernels.c:107), d2 > 0, which also drops the self pair;
// without it the smallest d2 is kept instead
struct GbTerm {
  float qq, fgb, ex, ey, ez, mw, h, bd;
};
template <bool MASK>
__device__ __forceinline__ void gb_term(const GbRow &r, const float4 &cp, const float2 &cb, float &d2min, GbTerm &g) {
  g.ex = cp.x - r.x; g.ey = cp.y - r.y; g.ez = cp.z - r.z;
  const float d2 = g.ex * g.ex + g.ey * g.ey + g.ez * g.ez;
  g.qq = r.q * cp.w;
  if (MASK) g.qq = d2 > 0.f ? g.qq : 0.f;
  else d2min = fminf(d2min, d2);
  const float bb = r.b * cb.x;
  const float et = __builtin_amdgcn_exp2f(d2 * (r.qib * cb.y));     // exp(-d2 / (4 B_i B_j))
  g.fgb = __builtin_amdgcn_rsqf(d2 + bb * et);
  const float qf3 = g.qq * g.fgb * g.fgb * g.fgb;
  g.h = qf3 * et;
  g.mw = fmaf(-0.25f, g.h, qf3);               // qf3 (1 - et/4)
  g.bd = fmaf(0.25f, d2, bb);                  // (A's term: qf3 et (bb + d2/4))
}
template <bool MASK>
__device__ __forceinline__ void gb_pair(const GbRow &r, const float4 &cp, const float2 &cb, float &d2min, float &re,
                                        float &rA, float &rx, float &ry, float &rz, float &cA, float &cgx, float &cgy,
                                        float &cgz) {
  GbTerm g;
  gb_term<MASK>(r, cp, cb, d2min, g);
  re += g.qq * g.fgb;
  rx += g.mw * g.ex; ry += g.mw * g.ey; rz += g.mw * g.ez;
  rA = fmaf(g.h, g.bd, rA);
  cA = fmaf(g.h, g.bd, cA);
  cgx = fmaf(g.mw, g.ex, cgx); cgy = fmaf(g.mw, g.ey, cgy); cgz = fmaf(g.mw, g.ez, cgz);     // (negated)
}

__global__ __launch_bounds__(256, 4) void k_gbpair(Dev d) {
  // tile columns per 64-column chunk, each chunk twice in a row so that
  // column (l - s) mod 64 sits at l + 64 - s: x, y, z, charge; Born radius,
  // its reciprocal
  __shared__ float4 cxq[4][128];
  __shared__ float2 cbr[4][128];
  __shared__ float rowacc[4][256];      // [A, gx, gy, gz][row]: the waves' row sums, added in wave order
  __shared__ double ered[4];
  __shared__ int slot;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;   // wave w: every row, column chunk w
  for (int it = first_item(); it < d.ngb_items; it = next_item(queue_head(d.queue, Q_GB), &slot, d.ngb_items)) {
    const int4 tp = d.gb_items[it];      // rows [x, y), columns [z, w)
    const bool diag = tp.x == tp.z;
    const int nch = (tp.w - tp.z + 63) >> 6;
    {
      const int j = tp.z + threadIdx.x;      // padding columns: far, no charge
      float4 c = make_float4(-1e6f - (float)threadIdx.x, 0.f, 0.f, 0.f);
      float2 b = make_float2(1.f, 1.f);
      if (j < tp.w) {
        const float4 p = d.pos[j];
        const float bj = d.br_f[j];
        c = make_float4(p.x, p.y, p.z, d.q[j]);
        b = make_float2(bj, __builtin_amdgcn_rcpf(bj));
      }
      cxq[w][lane] = c;
      cxq[w][lane + 64] = c;
      cbr[w][lane] = b;
      cbr[w][lane + 64] = b;
    }
    GbRow row[4];                          // the lane's rows lane + 64 k of the tile
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int i = tp.x + lane + 64 * k;
      row[k] = GbRow{1e6f + (float)(lane + 64 * k), 0.f, 0.f, 0.f, 1.f, 0.f};   // padding: far, no charge
      if (i < tp.y) {
        const float4 p = d.pos[i];
        row[k].x = p.x; row[k].y = p.y; row[k].z = p.z;
        row[k].q = d.q[i];
        row[k].b = d.br_f[i];
      }
      // exp(-d2 / (4 B_i B_j)) = exp2(d2 qib / B_j)
      row[k].qib = -0.25f * 1.44269504088896341f * __builtin_amdgcn_rcpf(row[k].b);
    }
    __syncthreads();
    float rA[4] = {0.f, 0.f, 0.f, 0.f}, rx[4] = {0.f, 0.f, 0.f, 0.f}, ry[4] = {0.f, 0.f, 0.f, 0.f},
          rz[4] = {0.f, 0.f, 0.f, 0.f}, re = 0.f;
    float cA = 0.f, cgx = 0.f, cgy = 0.f, cgz = 0.f;
    if (w < nch) {
      auto sweep = [&](auto mask) {
        constexpr bool M = decltype(mask)::value;
        const int from = rot_from(lane);
        float d2min = 1.f;
        re = cA = cgx = cgy = cgz = 0.f;
#pragma unroll
        for (int k = 0; k < 4; k++) rA[k] = rx[k] = ry[k] = rz[k] = 0.f;
        // the column whose partial sums this lane holds at step s: (lane - s) mod 64
        const float4 *cxc = &cxq[w][lane + 64];
        const float2 *cbc = &cbr[w][lane + 64];
#pragma unroll 1
        for (int s = 0; s < 64; s++) {
          const float4 cp = cxc[-s];
          const float2 cb = cbc[-s];
#pragma unroll
          for (int k = 0; k < 4; k++)
            gb_pair<M>(row[k], cp, cb, d2min, re, rA[k], rx[k], ry[k], rz[k], cA, cgx, cgy, cgz);
          cA = lds_rot(cA, from); cgx = lds_rot(cgx, from); cgy = lds_rot(cgy, from); cgz = lds_rot(cgz, from);
        }
        return __ballot(d2min == 0.f) != 0ull;
      };
      // without a self pair the mask only matters for two atoms in one place:
      // the sweep then runs again with it (a compare and a select per pair
      // less otherwise)
      if (diag || sweep(std::false_type{})) sweep(std::true_type{});
      // 64 rotations bring every column's sums back to its starting lane
    }
    const double e = wave_sum((double)re * (diag ? 0.5 : 1.0));
    if (lane == 0) ered[w] = e;
    const int j = tp.z + threadIdx.x;
    if (!diag && j < tp.w) {             // the columns' sums (this wave's chunk)
      fix_add(&d.acc_gbA[j], (double)cA);
      fix_add(&d.acc_gbg[3 * (size_t)j], -(double)cgx);
      fix_add(&d.acc_gbg[3 * (size_t)j + 1], -(double)cgy);
      fix_add(&d.acc_gbg[3 * (size_t)j + 2], -(double)cgz);
    }
    // the rows' sums over the four waves' column chunks in wave order
    for (int g = 0; g < 4; g++) {
      if (w == g) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int t = lane + 64 * k;
          rowacc[0][t] = g == 0 ? rA[k] : rowacc[0][t] + rA[k];
          rowacc[1][t] = g == 0 ? rx[k] : rowacc[1][t] + rx[k];
          rowacc[2][t] = g == 0 ? ry[k] : rowacc[2][t] + ry[k];
          rowacc[3][t] = g == 0 ? rz[k] : rowacc[3][t] + rz[k];
        }
      }
      __syncthreads();
    }
    const int i = tp.x + threadIdx.x;
    if (i < tp.y) {
      const int t = threadIdx.x;
      fix_add(&d.acc_gbA[i], (double)rowacc[0][t]);
      fix_add(&d.acc_gbg[3 * (size_t)i], (double)rowacc[1][t]);
      fix_add(&d.acc_gbg[3 * (size_t)i + 1], (double)rowacc[2][t]);
      fix_add(&d.acc_gbg[3 * (size_t)i + 2], (double)rowacc[3][t]);
    }
    if (threadIdx.x == 0) d.gb_epart[d.gb_eslot[it]] = ered[0] + ered[1] + ered[2] + ered[3];
  }
}

// ------------------------------------------- GB pairs of small calls
// The same sums (k_gbpair) where its items are fewer than the CUs and one
// wave's 64 steps of four rows are the launch.  A block takes one item's
// 64-column chunk, and six waves share the work of k_gbpair's one: four form
// the pairs' terms, each for 64 of the tile's rows with their sums, and pass
// them through LDS, batch by batch, to one that adds the column sums (its lanes
// are columns, so nothing rotates) and one that adds the energy, in the order
// k_gbpair's lanes do.  The sums leave apart; k_gb_sum adds them in k_gbpair's
// order, per atom, and does k_q2ab's work with them.
// Bound: the column wave's LDS reads, one batch of them per barrier.  Against
// k_gbpair (with k_q2ab): 61 atoms 21 + 4.2 -> 8.1 + 3.1 us, 613 22 + 4.3 ->
// 12.7 + 5.1, 2,000 22 + 4.7 -> 13.0 + 5.0.
constexpr int kGbSteps = 4;              // steps of a batch
constexpr int kGbWaves = 6;
__global__ __launch_bounds__(64 * kGbWaves) void k_gb_split(Dev d) {
  // columns and rows twice in a row (k_gbpair): x, y, z, charge; Born radius, its reciprocal
  __shared__ float4 cxq[128], rx4[4][128];
  __shared__ float2 cbr[128];
  __shared__ float4 grad[2][kGbSteps][4][64];              // the terms: gradient, A's factors
  __shared__ float2 ener[2][kGbSteps][4][64];              // charges, 1/f
  const int lane = threadIdx.x & 63, role = threadIdx.x >> 6;
  const int it = blockIdx.x >> 2, w = blockIdx.x & 3;
  const int4 tp = d.gb_items[it];        // rows [x, y), columns [z, w)
  if (w * 64 >= tp.w - tp.z) return;     // no such chunk (block-uniform)
  const bool diag = tp.x == tp.z;
  const int nrow = (tp.y - tp.x + 63) >> 6;                // row groups with an atom
  if (role == 4) {
    const int j = tp.z + 64 * w + lane;
    float4 c = make_float4(-1e6f - (float)(64 * w + lane), 0.f, 0.f, 0.f);
    float2 b = make_float2(1.f, 1.f);
    if (j < tp.w) {
      const float4 p = d.pos[j];
      const float bj = d.br_f[j];
      c = make_float4(p.x, p.y, p.z, d.q[j]);
      b = make_float2(bj, __builtin_amdgcn_rcpf(bj));
    }
    cxq[lane] = c;
    cxq[lane + 64] = c;
    cbr[lane] = b;
    cbr[lane + 64] = b;
  }
  GbRow row{1e6f + (float)(64 * role + lane), 0.f, 0.f, 0.f, 1.f, 0.f};
  if (role < 4) {
    const int i = tp.x + 64 * role + lane;
    if (i < tp.y) {
      const float4 p = d.pos[i];
      row.x = p.x; row.y = p.y; row.z = p.z;
      row.q = d.q[i];
      row.b = d.br_f[i];
    }
    row.qib = -0.25f * 1.44269504088896341f * __builtin_amdgcn_rcpf(row.b);
    rx4[role][lane] = rx4[role][lane + 64] = make_float4(row.x, row.y, row.z, 0.f);
  }
  __syncthreads();
  float rA = 0.f, rx = 0.f, ry = 0.f, rz = 0.f;            // a row's sums (the first four waves)
  float cA = 0.f, cgx = 0.f, cgy = 0.f, cgz = 0.f, re = 0.f;   // a column's (the fifth), the energy (the sixth)
  float d2min = 1.f;
  auto sweep = [&](auto rows) {
    constexpr int NROW = decltype(rows)::value;
#pragma unroll 1
    for (int t = 0; t <= 64 / kGbSteps; t++) {
      if (role < NROW) {
        if (t < 64 / kGbSteps) {
#pragma unroll
          for (int u = 0; u < kGbSteps; u++) {
            const int s = t * kGbSteps + u;
            GbTerm g;
            gb_term<true>(row, cxq[lane + 64 - s], cbr[lane + 64 - s], d2min, g);
            rx += g.mw * g.ex; ry += g.mw * g.ey; rz += g.mw * g.ez;
            rA = fmaf(g.h, g.bd, rA);
            grad[t & 1][u][role][lane] = make_float4(g.mw, g.h, g.bd, 0.f);
            ener[t & 1][u][role][lane] = make_float2(g.qq, g.fgb);
          }
        }
      } else if (t > 0 && role >= 4) {
        const int b = (t - 1) & 1, s0 = (t - 1) * kGbSteps;
        if (role == 5) {
          float2 e[kGbSteps][NROW];
#pragma unroll
          for (int u = 0; u < kGbSteps; u++)
#pragma unroll
            for (int k = 0; k < NROW; k++) e[u][k] = ener[b][u][k][lane];
#pragma unroll
          for (int u = 0; u < kGbSteps; u++)
#pragma unroll
            for (int k = 0; k < NROW; k++) re += e[u][k].x * e[u][k].y;
        } else if (!diag) {
          const float4 c = cxq[lane];
#pragma unroll
          for (int u = 0; u < kGbSteps; u++) {
            float4 g[NROW], r[NROW];
#pragma unroll
            for (int k = 0; k < NROW; k++) {
              g[k] = grad[b][u][k][(lane + s0 + u) & 63];
              r[k] = rx4[k][lane + s0 + u];
            }
#pragma unroll
            for (int k = 0; k < NROW; k++) {
              const float ex = c.x - r[k].x, ey = c.y - r[k].y, ez = c.z - r[k].z;
              cA = fmaf(g[k].y, g[k].z, cA);
              cgx = fmaf(g[k].x, ex, cgx); cgy = fmaf(g[k].x, ey, cgy); cgz = fmaf(g[k].x, ez, cgz);
            }
          }
        }
      }
      __syncthreads();
    }
  };
  // (row groups without an atom add nothing)
  if (nrow == 4) sweep(std::integral_constant<int, 4>{});
  else if (nrow == 3) sweep(std::integral_constant<int, 3>{});
  else if (nrow == 2) sweep(std::integral_constant<int, 2>{});
  else sweep(std::integral_constant<int, 1>{});
  // sets of 4 quantities x 256 atoms of the item's slot: 0..3 its rows by chunk, 4 its columns
  float *o = d.gbsplit + (size_t)d.gb_eslot[it] * kGbSets * 1024;
  if (role < 4) {
    float *p = o + w * 1024 + 64 * role + lane;
    p[0] = rA; p[256] = rx; p[512] = ry; p[768] = rz;
  } else if (role == 4) {
    float *p = o + 4 * 1024 + 64 * w + lane;
    p[0] = cA; p[256] = cgx; p[512] = cgy; p[768] = cgz;
  } else {
    const double e = wave_sum((double)re * (diag ? 0.5 : 1.0));
    if (lane == 0) d.gbener[4 * (size_t)d.gb_eslot[it] + w] = e;
  }
}

// one quantity (A, gradient x, y, z) of one tile's atoms from every item that
// holds the tile; A's threads form the chain-rule factors at once, and the
// first gradient's the items' energies.  Grid (tiles, 4).
__global__ __launch_bounds__(256) void k_gb_sum(Dev d) {
  const int b = blockIdx.x, q = blockIdx.y, t = threadIdx.x;
  const int2 blk = d.ablk[b];
  const SysInfo &S = d.sys[d.asys[blk.x]];
  const int T = b - S.blk0, nb = S.nblk;
  auto slot = [&](int I, int J) { return S.tile0 + I * nb - I * (I - 1) / 2 + J - I; };
  const int i = blk.x + t;
  if (q == 1)
    for (int J = T + t; J < nb; J += 256) {
      const int nch = (min(256, S.n - 256 * J) + 63) >> 6;
      const double *e = d.gbener + 4 * (size_t)slot(T, J);
      double v = e[0] + (nch > 1 ? e[1] : 0.0);
      v += nch > 2 ? e[2] : 0.0;
      v += nch > 3 ? e[3] : 0.0;
      d.gb_epart[slot(T, J)] = v;
    }
  if (i >= blk.y) return;
  const float *base = d.gbsplit + q * 256 + t;
  long long sum = 0;
#pragma unroll 2
  for (int J = T; J < nb; J++) {          // the tile as rows: by chunks, in FP32
    const int nch = (min(256, S.n - 256 * J) + 63) >> 6;
    const float *s = base + (size_t)slot(T, J) * kGbSets * 1024;
    const float v0 = s[0], v1 = s[1024], v2 = s[2048], v3 = s[3072];
    float v = v0 + (nch > 1 ? v1 : 0.f);
    v += nch > 2 ? v2 : 0.f;
    v += nch > 3 ? v3 : 0.f;
    sum += __double2ll_rn((double)v * kFix);
  }
#pragma unroll 4
  for (int I = 0; I < T; I++) {
    const double v = (double)base[(size_t)slot(I, T) * kGbSets * 1024 + 4 * 1024];
    sum += __double2ll_rn((q == 0 ? v : -v) * kFix);
  }
  if (q == 0) {
    d.acc_gbA[i] = sum;
    chain_factors(d, i, fix_get(sum));
  } else {
    d.acc_gbg[3 * (size_t)i + q - 1] = sum;
  }
}

void launch_gbpair(const Dev &d, const Tuning &t, hipStream_t s) {
  if (!d.ngb_items) return;
  if (d.gbs_on) {
    hipLaunchKernelGGL(k_gb_split, dim3(4 * d.ngb_items), dim3(64 * kGbWaves), 0, s, d);
    hipLaunchKernelGGL(k_gb_sum, dim3(d.nablk, 4), dim3(256), 0, s, d);
    return;
  }
  const int grid = t.gb_grid > 0 ? std::min(t.gb_grid, d.ngb_items) : d.ngb_items;
  hipLaunchKernelGGL(k_gbpair, dim3(grid), dim3(256), 0, s, d);
}

// -------------------------------------------- chain rule at constant sp
// For a pair (k, j) with at least one heavy atom, both directed descreening
// terms (reference agbnp3_gb_ders_constvp_nolist_ps kernels.c:681-805 and
// agbnp3_gb_deruv_nolist_ps kernels.c:809-904, without the q4cache):
//   k <- j (j heavy): Q4 from table [t_k][t_j] at d/R_j; weights q2ab_k sp_j
//   j <- k (k heavy): Q4 from table [t_j][t_k] at d/R_k; weights q2ab_j sp_k
// h = (sum of weight x dQ4) / d along (x_j - x_k), GB with q2ab and vdW with
// abrw (scaled by df/4pi and 1/4pi later); U_k += q2ab_j Q4(j <- k),
// V_k += abrw_j Q4(j <- k) and likewise U_j, V_j from Q4(k <- j).
//
// Items are pairs of 256-atom blocks of one radius type each (R, 1/R are
// block constants), so a block stages only the two tables it reads.  Each
// unordered pair is evaluated once: rows sit in lanes, the 256 columns are
// read from LDS at a lane-rotated index while their partial sums rotate one
// lane per step (DPP), as in the GB pair kernel; kinds whose registers allow
// it hold two rows per lane, so one column read and one rotation serve two
// pairs.  Item kinds (host-side):
//   CK_HH   both blocks heavy atoms only: both directions, no per-pair tests;
//   CK_HX   hydrogen rows, heavy columns: one direction (a hydrogen does not
//           descreen), no U/V of the rows;
//   CK_HX0  the same with rows whose vdW coefficients (ialpha + salpha) are
//           all zero, as hydrogens usually have: abrw = 0, no vdW terms;
//   CK_GEN  diagonal blocks and blocks that mix heavy atoms and hydrogens.
// A heavy x heavy item whose two blocks have one radius type runs as CK_HHS
// (chosen on the device): R_P = R_Q and the two tables are the same one, so
// both directions fall on one interval at one fraction (bitwise: the FP64
// branch squares the same differences) and one lookup serves both.
// The tables are read as per-interval cubics in the fraction u of the
// interval, c0 + c1 u + c2 u^2 + c3 u^3 (the host's chain-table builder;
// interval 511, past the last node, is zero), and the derivative is formed
// from the same four numbers (times 1/dx, folded into the weights):
//   the interpolant's own:   c1 + 2 c2 u + 3 c3 u^2;
//   the reference's (its sign of the y''_{k+1} term, agbnp3_utils.c:292-293):
//     (c1 + 2/3 c2 + 2 c3) + 2 c2 u - (2 c2 + 3 c3) u^2.
enum : int { CK_GEN = 0, CK_HH = 1, CK_HX = 2, CK_HX0 = 3, CK_HHS = 4 };

// Table coordinate of a chain-rule lookup, xh = (d / R) / dx, clamped at
// kTblN - 0.5: every coordinate past the last node lands in the zero
// interval kTblN - 1.  The reference's spline derivative jumps at the
// table nodes, so the interval a distance falls in decides the value and must
// be the one the FP64 arithmetic picks.  The FP32 xh is within 8e-7 xh of
// the exact value (rounding of the coordinate differences, d^2, the hardware
// reciprocal square root, c = 1 / (R dx) and the product); where that band
// reaches a node, xh is recomputed in FP64 from the FP32 coordinates as
// d / R * (1/dx) (a few lookups in 10^4: chain_fix).  u = xh - floor(xh) is
// exact (xh >= 0), as is the FP64 path's.
__device__ __forceinline__ void chain_coord(float &xh, int &k, float &u) {
  xh = fminf(xh, (float)kTblN - 0.5f);
  k = (int)xh;
  u = __builtin_amdgcn_fractf(xh);
}
__device__ __forceinline__ void chain_fix(float xh, const float4 &pa, const float4 &pb, float R, float dxinv, int &k,
                                          float &u) {
  constexpr float kLast = (float)kTblN - 0.5f;
  if (fabsf(u - 0.5f) > fmaf(-8e-7f, xh, 0.5f - 1e-6f)) {
    // the empty asm statements keep the FP64 conversions inside this rare
    // branch (hoisted, they cost three conversions on every pair), and keep
    // the squares rounded before they are added (no fused multiply-add)
    float ax = pa.x, ay = pa.y, az = pa.z, bx = pb.x, by = pb.y, bz = pb.z;
    asm volatile("" : "+v"(ax), "+v"(ay), "+v"(az), "+v"(bx), "+v"(by), "+v"(bz));
    const double ex = (double)bx - (double)ax, ey = (double)by - (double)ay, ez = (double)bz - (double)az;
    double sx = ex * ex, sy = ey * ey, sz = ez * ez;
    asm volatile("" : "+v"(sx), "+v"(sy), "+v"(sz));
    const double dd = sqrt((sx + sy) + sz);
    const double x64 = fmin(__dmul_rn(__ddiv_rn(dd, (double)R), (double)dxinv), (double)kLast);
    k = (int)x64;
    u = (float)(x64 - (double)k);
  }
}
// A group of lookups tests for the band together, against its widest
// (xh <= kTblN - 0.5): no lookup within |u - 0.5| <= kChainBand is in it.
constexpr float kChainBand = 0.49958f;    // < 0.5 - 1e-6 - 8e-7 (kTblN - 0.5)

// the derivative x dx of the interval record c as a quadratic in u,
// (e0, e1, e2): e0 + e1 u + e2 u^2
template <bool QUIRK>
__device__ __forceinline__ float4 chain_dpoly(const float4 &c) {
  const float m2 = c.z + c.z;
  if (QUIRK) return make_float4(fmaf(0.666666667f, c.z, fmaf(2.f, c.w, c.y)), m2, fmaf(-3.f, c.w, -m2), 0.f);
  return make_float4(c.y, m2, 3.f * c.w, 0.f);
}

// value and derivative x dx on the interval record c at fraction u
template <bool QUIRK>
__device__ __forceinline__ void chain_poly(const float4 &c, float u, float &q, float &dqx) {
  q = fmaf(fmaf(fmaf(c.w, u, c.z), u, c.y), u, c.x);
  const float4 e = chain_dpoly<QUIRK>(c);
  dqx = fmaf(fmaf(e.z, u, e.y), u, e.x);
}

// the same from the interval record and its staged derivative record
__device__ __forceinline__ void chain_poly(const float4 &c, const float4 &e, float u, float &q, float &dqx) {
  q = fmaf(fmaf(fmaf(c.w, u, c.z), u, c.y), u, c.x);
  dqx = fmaf(fmaf(e.z, u, e.y), u, e.x);
}

// one pair of a row atom k and a column atom j: x_j - x_k, 1 / d, and the table
// coordinates (as computed, interval, fraction) of k <- j and, with two
// lookups, j <- k
struct ChainPair {
  float ex, ey, ez, id, x1, x2, u1, u2;
  int k1, k2;
};
template <int KIND>
__device__ __forceinline__ ChainPair chain_meet(const float4 &pk, const float4 &pj, float cP, float cQ, bool pair) {
  ChainPair m;
  m.ex = pj.x - pk.x; m.ey = pj.y - pk.y; m.ez = pj.z - pk.z;
  const float d2 = m.ex * m.ex + m.ey * m.ey + m.ez * m.ez;
  m.id = __builtin_amdgcn_rsqf(d2);               // hardware reciprocal square root (1 ulp)
  float dist = d2 * m.id;
  if (KIND == CK_GEN) {
    m.id = pair ? m.id : 0.f;
    dist = pair ? dist : 1e6f;
  }
  m.x1 = dist * cQ;
  chain_coord(m.x1, m.k1, m.u1);
  if (KIND == CK_HH || KIND == CK_GEN) {
    m.x2 = dist * cP;
    chain_coord(m.x2, m.k2, m.u2);
  }
  return m;
}
// its terms: hgb and hvw (along x_j - x_k), Q4(k <- j) and Q4(j <- k), from
// the interval records c1 and c2 (one direction: c2 the derivative record)
template <int KIND, bool QUIRK>
__device__ __forceinline__ void chain_terms(const ChainPair &m, const float4 &pj, const float4 &pp, float wk, float q2k,
                                            float abk, bool kheavy, const float4 &c1, const float4 &c2, float &hgb,
                                            float &hvw, float &q1, float &q2) {
  float dq1, dq2;
  if (KIND == CK_HX || KIND == CK_HX0) {
    chain_poly(c1, c2, m.u1, q1, dq1);
    const float t1 = pj.w * dq1 * m.id;
    hgb = q2k * t1;
    hvw = KIND == CK_HX ? abk * t1 : 0.f;
    q2 = 0.f;
    return;
  }
  chain_poly<QUIRK>(c1, m.u1, q1, dq1);           // k <- j (weight 0 unless j heavy)
  if (KIND == CK_HH || KIND == CK_GEN) {
    chain_poly<QUIRK>(c2, m.u2, q2, dq2);         // j <- k
  } else {
    q2 = q1;
    dq2 = dq1;
  }
  if (KIND == CK_GEN) {
    q2 = kheavy ? q2 : 0.f;
    q1 = pp.z != 0.f ? q1 : 0.f;
  }
  const float t1 = pj.w * dq1 * m.id, t2 = wk * dq2 * m.id;
  hgb = fmaf(q2k, t1, pp.x * t2);
  hvw = fmaf(abk, t1, pp.y * t2);
}

enum : int { CM_PLAIN = 0, CM_GROUP = 1, CM_CULL = 2 };

// per 64-column chunk: the columns' records, and once every wave is past the
// chunk, in the same bytes, its column sums [gb xyz, vw xyz, U, V][column]
struct ChainChunk {
  union {
    struct {
      float4 pos[64];        // x, y, z, sp_j / (R_Q^2 dx) (0: hydrogen)
      float4 par[64];        // q2ab, abrw, 1 for a heavy atom (the general kind's per-pair test), 0
    } col;
    float acc[8][64];
  };
};

// CM_CULL (large solutes): a wave passes over the chunks past the tables' end.
// CM_GROUP: where a CU holds one item at a time (one wave per SIMD), the pairs of
// two column steps (four with one row per lane) are met first, tested for
// the band with one wave-uniform branch, and read the tables together: a
// divergent branch per lookup serialises the lookups' LDS reads (2,000 atoms:
// 76 -> 60 us; half as many steps 66, twice as many 64).  With several items per CU their waves fill those waits, and
// taking the lookups one by one is as fast or faster (150,000 atoms: 7.1 ms
// against 7.3).
template <int KIND, bool QUIRK, int MODE>
__device__ __forceinline__ void chain_item(const Dev &d, int it, const int4 &item, const float4 *__restrict__ tab_rc,
                                           const float4 *__restrict__ tab_cr, ChainChunk *ch) {
  // rows per lane: two where the registers allow 5 waves per SIMD (wave w
  // holds rows 128 (w & 1) + lane and + 64 and takes the chunks of parity
  // w >> 1), else one (wave w holds row 64 w + lane and takes every chunk)
  constexpr int NR = (KIND == CK_HH || KIND == CK_GEN) ? 1 : 2;
  constexpr int NW = 4 / NR;           // waves on one chunk
  constexpr int kUnroll = 3 - NR;      // column steps unrolled: 2 with one row, 1 with two
  constexpr bool GROUP = MODE == CM_GROUP;
  constexpr int NS = GROUP ? 2 * kUnroll : 1;              // column steps of a group
  constexpr bool kOne = KIND == CK_HX || KIND == CK_HX0;   // one direction: k (hydrogen) <- j
  constexpr bool kTwo = KIND == CK_HH || KIND == CK_GEN;   // two lookups (CK_HHS: one serves both directions)
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int rh = NR == 2 ? w & 1 : w, cp = NR == 2 ? w >> 1 : 0;   // row group, chunk parity
  const int4 bp = d.cblk[item.x];
  const bool diag = item.x == item.y;
  const float dxinv = d.tdxinv;
  const SysInfo &S = d.sys[bp.y];
  const int hend = S.a0 + S.nh;
  // block constants: the radii of the row (P) and column (Q) radius types
  const float RP = d.pos[d.cperm[item.x * 256]].w, RQ = d.pos[d.cperm[item.y * 256]].w;
  const float iRP = 1.0f / RP, iRQ = 1.0f / RQ;
  const float cP = iRP * dxinv, cQ = iRQ * dxinv;
  {
    const int j = d.cperm[item.y * 256 + threadIdx.x];
    float4 p = make_float4(1e6f, 1e6f, 1e6f, 0.f);
    float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
    if (j >= 0) {
      const float4 pj = d.pos[j];
      const float hv = j < hend ? 1.f : 0.f;
      p = make_float4(pj.x, pj.y, pj.z, hv != 0.f ? d.sp_f[j] * iRQ * iRQ * dxinv : 0.f);
      q = make_float4(d.q2ab_f[j], d.abrw_f[j], hv, 0.f);
    }
    ch[w].col.pos[lane] = p;
    ch[w].col.par[lane] = q;
  }
  // the lane's rows of block P
  int rr[NR];
  float4 pk[NR];
  float wk[NR], q2k[NR], abk[NR];
  bool kok[NR], kheavy[NR];
#pragma unroll
  for (int k = 0; k < NR; k++) {
    rr[k] = NR == 2 ? rh * 128 + lane + 64 * k : w * 64 + lane;
    const int kr = d.cperm[item.x * 256 + rr[k]];
    pk[k] = make_float4(-1e6f, -1e6f, -1e6f, 1.f);
    wk[k] = 0.f; q2k[k] = 0.f; abk[k] = 0.f;
    kok[k] = kr >= 0;
    kheavy[k] = false;
    if (kr >= 0) {
      pk[k] = d.pos[kr];
      q2k[k] = d.q2ab_f[kr];
      abk[k] = d.abrw_f[kr];
      kheavy[k] = kr < hend;
      wk[k] = kheavy[k] ? d.sp_f[kr] * iRP * iRP * dxinv : 0.f;
    }
  }
  __syncthreads();
  float rg[NR][3], rv[NR][3], rU[NR], rV[NR];
#pragma unroll
  for (int k = 0; k < NR; k++) {
    rg[k][0] = rg[k][1] = rg[k][2] = rv[k][0] = rv[k][1] = rv[k][2] = rU[k] = rV[k] = 0.f;
  }
  // pairs past the tables' end add nothing: a wave passes over the chunks whose
  // box lies that far from its rows'
  unsigned reach = 15u;
  // a wave of padding rows has none either (batches, whose blocks are often
  // cut short: 64 poses 102 -> 84 us, 24 x 6000 405 -> 375)
  if (__ballot(kok[0] || kok[NR - 1]) == 0ull) reach = 0u;
  if (MODE == CM_CULL && reach) {
    const float4 *b = d.chbox + 2 * (4 * item.x + (NR == 2 ? 2 * rh : rh)), *q = d.chbox + 2 * (4 * item.y + (lane & 3));
    Box rows{{b[0].x, b[0].y, b[0].z}, {b[1].x, b[1].y, b[1].z}};
    if (NR == 2) {
      rows.lo[0] = fminf(rows.lo[0], b[2].x); rows.lo[1] = fminf(rows.lo[1], b[2].y); rows.lo[2] = fminf(rows.lo[2], b[2].z);
      rows.hi[0] = fmaxf(rows.hi[0], b[3].x); rows.hi[1] = fmaxf(rows.hi[1], b[3].y); rows.hi[2] = fmaxf(rows.hi[2], b[3].z);
    }
    const float far = kFarCoord / fminf(cQ, kOne ? cQ : cP);
    reach = (unsigned)__ballot(!(box_gap2(rows, q[0], q[1]) > far * far)) & 15u;     // lane c: chunk c
  }
  // the item's 64-column chunks of block Q; waves of chunk parity cp take
  // chunks cbeg + cp, cbeg + cp + NR, ...
  const int cbeg = item.w & 15, cend = item.w >> 4;
  const int niter = (cend - cbeg + NR - 1) / NR;
  for (int ci = 0; ci < niter; ci++) {
    const int c = cbeg + cp + NR * ci;
    float ca[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (c < cend && ((reach >> c) & 1u)) {
      auto meet = [&](int k, int col, const float4 &pj, const float4 &pp) {
        // the self pair of a diagonal block, padding rows, hydrogen-hydrogen
        // pairs: no weight, and a distance past the tables (zero interval)
        const bool pair = KIND != CK_GEN || (kok[k] && (kheavy[k] || pp.z != 0.f) && !(diag && c * 64 + col == rr[k]));
        ChainPair m = chain_meet<KIND>(pk[k], pj, cP, cQ, pair);
        if (!GROUP) {
          chain_fix(m.x1, pk[k], pj, RQ, dxinv, m.k1, m.u1);
          if (kTwo) chain_fix(m.x2, pj, pk[k], RP, dxinv, m.k2, m.u2);
        }
        return m;
      };
      auto add = [&](int k, const ChainPair &m, const float4 &pj, const float4 &pp, const float4 &c1, const float4 &c2) {
        float hgb, hvw, q1, q2;
        chain_terms<KIND, QUIRK>(m, pj, pp, wk[k], q2k[k], abk[k], kheavy[k], c1, c2, hgb, hvw, q1, q2);
        if (kOne) {
          ca[6] = fmaf(q2k[k], q1, ca[6]);
          if (KIND == CK_HX) ca[7] = fmaf(abk[k], q1, ca[7]);
        } else {
          rU[k] = fmaf(pp.x, q2, rU[k]);
          rV[k] = fmaf(pp.y, q2, rV[k]);
          ca[6] = fmaf(q2k[k], q1, ca[6]);
          ca[7] = fmaf(abk[k], q1, ca[7]);
        }
        rg[k][0] = fmaf(hgb, m.ex, rg[k][0]); rg[k][1] = fmaf(hgb, m.ey, rg[k][1]); rg[k][2] = fmaf(hgb, m.ez, rg[k][2]);
        ca[0] = fmaf(-hgb, m.ex, ca[0]); ca[1] = fmaf(-hgb, m.ey, ca[1]); ca[2] = fmaf(-hgb, m.ez, ca[2]);
        if (KIND != CK_HX0) {
          rv[k][0] = fmaf(hvw, m.ex, rv[k][0]); rv[k][1] = fmaf(hvw, m.ey, rv[k][1]); rv[k][2] = fmaf(hvw, m.ez, rv[k][2]);
          ca[3] = fmaf(-hvw, m.ex, ca[3]); ca[4] = fmaf(-hvw, m.ey, ca[4]); ca[5] = fmaf(-hvw, m.ez, ca[5]);
        }
      };
      auto rotate = [&]() {
#pragma unroll
        for (int q = 0; q < 8; q++)
          if (KIND != CK_HX0 || q < 3 || q == 6) ca[q] = wave_rot(ca[q]);   // (the vdW sums stay zero)
      };
      if constexpr (GROUP) {
#pragma unroll 1
        for (int s = 0; s < 64; s += NS) {
          float4 pj[NS], pp[NS], c1[NS][NR], c2[NS][NR];
          ChainPair m[NS][NR];
          float band = 0.f;
#pragma unroll
          for (int t = 0; t < NS; t++) {
            const int col = (lane - s - t) & 63;          // the column whose sums this lane holds
            pj[t] = ch[c].col.pos[col];
            pp[t] = ch[c].col.par[col];
#pragma unroll
            for (int k = 0; k < NR; k++) {
              m[t][k] = meet(k, col, pj[t], pp[t]);
              band = fmaxf(band, fabsf(m[t][k].u1 - 0.5f));
              if (kTwo) band = fmaxf(band, fabsf(m[t][k].u2 - 0.5f));
            }
          }
          if (__builtin_expect(__ballot(band > kChainBand) != 0ull, 0)) {
#pragma unroll
            for (int t = 0; t < NS; t++)
#pragma unroll
              for (int k = 0; k < NR; k++) {
                chain_fix(m[t][k].x1, pk[k], pj[t], RQ, dxinv, m[t][k].k1, m[t][k].u1);
                if (kTwo) chain_fix(m[t][k].x2, pj[t], pk[k], RP, dxinv, m[t][k].k2, m[t][k].u2);
              }
          }
#pragma unroll
          for (int t = 0; t < NS; t++)
#pragma unroll
            for (int k = 0; k < NR; k++) {
              c1[t][k] = tab_rc[m[t][k].k1];
              if (kTwo || kOne) c2[t][k] = tab_cr[kTwo ? m[t][k].k2 : m[t][k].k1];
            }
#pragma unroll
          for (int t = 0; t < NS; t++) {
#pragma unroll
            for (int k = 0; k < NR; k++) add(k, m[t][k], pj[t], pp[t], c1[t][k], c2[t][k]);
            rotate();
          }
        }
      } else {
#pragma unroll kUnroll
        for (int s = 0; s < 64; s++) {
          const int col = (lane - s) & 63;
          const float4 pj = ch[c].col.pos[col], pp = ch[c].col.par[col];
#pragma unroll
          for (int k = 0; k < NR; k++) {
            const ChainPair m = meet(k, col, pj, pp);
            float4 c2;
            if (kTwo || kOne) c2 = tab_cr[kTwo ? m.k2 : m.k1];
            add(k, m, pj, pp, tab_rc[m.k1], c2);
          }
          rotate();
        }
      }
    }
    // chunk c's column sums over its waves' row groups in a fixed order
    // (0 + 1 + ...), over its column records once every wave is done with them
    __syncthreads();
    for (int g = 0; g < NW; g++) {
      if (c < cend && rh == g) {
#pragma unroll
        for (int q = 0; q < 8; q++) ch[c].acc[q][lane] = g == 0 ? ca[q] : ch[c].acc[q][lane] + ca[q];
      }
      __syncthreads();
    }
  }
  // the item's sums as plain stores (k_chain_sum adds them up per atom in a
  // fixed order); U, V are still to be scaled by 1/R of the block
  // (hydrogen-row items store only what they can make nonzero: k_chain_sum's
  // lists leave the other slots out)
  float *pr = d.chpart + (size_t)it * 2 * 8 * 256;
  if (!diag) {
    float *pc = pr + 8 * 256 + threadIdx.x;
    const bool mine = w >= cbeg && w < cend;            // column w * 64 + lane in the item's chunks
#pragma unroll
    for (int q = 0; q < 8; q++)
      if (KIND != CK_HX0 || q < 3 || q == 6) pc[q * 256] = mine ? ch[w].acc[q][lane] : 0.f;
  }
  // with two rows per lane, the rows' sums over the two chunk parities in a
  // fixed order (0 + 1), through the chunk records' bytes ([8][256] floats)
  float *xr = &ch[0].acc[0][0];
  const bool rowuv = KIND != CK_HX && KIND != CK_HX0;
  if (NR == 2) __syncthreads();
  if (NR == 2 && cp == 1) {
#pragma unroll
    for (int k = 0; k < NR; k++) {
      float *x = xr + rr[k];
      x[0 * 256] = rg[k][0]; x[1 * 256] = rg[k][1]; x[2 * 256] = rg[k][2];
      if (KIND != CK_HX0) {
        x[3 * 256] = rv[k][0]; x[4 * 256] = rv[k][1]; x[5 * 256] = rv[k][2];
      }
      if (rowuv) {
        x[6 * 256] = rU[k]; x[7 * 256] = rV[k];
      }
    }
  }
  if (NR == 2) __syncthreads();
  if (cp == 0) {
    // plus the other parity's sums (none with one row per lane)
    auto sum = [&](float v, int q, int r) {
      if constexpr (NR == 2) return v + xr[q * 256 + r];
      else return v;
    };
#pragma unroll
    for (int k = 0; k < NR; k++) {
      const int r = rr[k];
      float *o = pr + r;
      o[0 * 256] = sum(rg[k][0], 0, r); o[1 * 256] = sum(rg[k][1], 1, r); o[2 * 256] = sum(rg[k][2], 2, r);
      if (KIND != CK_HX0) {
        o[3 * 256] = sum(rv[k][0], 3, r); o[4 * 256] = sum(rv[k][1], 4, r); o[5 * 256] = sum(rv[k][2], 5, r);
      }
      if (rowuv) {
        o[6 * 256] = kheavy[k] ? sum(rU[k], 6, r) : 0.f;
        o[7 * 256] = kheavy[k] ? sum(rV[k], 7, r) : 0.f;
      }
    }
  }
}

// ------------------------------------- chain rule of small calls, by row groups
// The same sums (k_chain), where its items are about as few as the CUs and one
// wave's 256 steps through its 64 rows (or 128 steps of two rows) are the
// launch.  Those rows and the steps of a column through them fix the order of
// every sum, so they are not cut; the work on a pair is spread over waves
// instead.  A block takes one wave's share of an item: four waves (fronts) form
// the terms of a batch of pairs, EACH of them each, and pass them through LDS
// to four that add the GB and vdW sums of the rows and of the columns (lanes
// are columns there, so nothing rotates), one batch behind.  Column sums of an
// item's row groups, and row sums of its two chunk parities, leave apart and
// k_chain_sum adds them in the order k_chain does.
// Bound: a front's chain from the column's LDS read over the table reads to
// its terms, once per batch.  Against k_chain: 61 atoms 20 -> 13 us, 613 57 ->
// 24, 2,000 60 -> 26 (eight waves as fronts 30); with two waves instead of four
// behind the fronts no change there, but 5,000 atoms' call 267 -> 279 us.
constexpr int kSplitFronts = 4, kSplitWaves = kSplitFronts + 4;
template <int REC>
struct SplitLds {
  float4 cpos[256], cpar[256];           // the columns (ChainChunk's records)
  float4 rpos[2][64];                    // the rows: position,
  float rw[2][2][64], cw[2][256];        // [0] q2ab and [1] abrw of the rows and the columns
  float ring[2][REC][4][64];             // per pair: hgb, hvw, Q4(k <- j), Q4(j <- k)
};

template <int KIND, bool QUIRK, int EACH>
__device__ __forceinline__ void chain_split_item(const Dev &d, int it, int part, const int4 &item,
                                                 const float4 *__restrict__ tab_rc, const float4 *__restrict__ tab_cr,
                                                 SplitLds<kSplitFronts * EACH> &L) {
  constexpr int NR = (KIND == CK_HH || KIND == CK_GEN) ? 1 : 2;      // rows per lane, as k_chain has them
  constexpr bool kOne = KIND == CK_HX || KIND == CK_HX0;
  constexpr bool kTwo = KIND == CK_HH || KIND == CK_GEN;
  constexpr int kRec = kSplitFronts * EACH, kSteps = kRec / NR, kBatches = 64 / kSteps;     // of a batch, of a chunk
  const int lane = threadIdx.x & 63, role = threadIdx.x >> 6;
  const int rh = NR == 2 ? part & 1 : part, cp = NR == 2 ? part >> 1 : 0;
  const int4 bp = d.cblk[item.x];
  const bool diag = item.x == item.y;
  const float dxinv = d.tdxinv;
  const SysInfo &S = d.sys[bp.y];
  const int hend = S.a0 + S.nh;
  const float RP = d.pos[d.cperm[item.x * 256]].w, RQ = d.pos[d.cperm[item.y * 256]].w;
  const float iRP = 1.0f / RP, iRQ = 1.0f / RQ;
  const float cP = iRP * dxinv, cQ = iRQ * dxinv;
  if (threadIdx.x < 256) {
    const int j = d.cperm[item.y * 256 + threadIdx.x];
    float4 p = make_float4(1e6f, 1e6f, 1e6f, 0.f);
    float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
    if (j >= 0) {
      const float4 pj = d.pos[j];
      const float hv = j < hend ? 1.f : 0.f;
      p = make_float4(pj.x, pj.y, pj.z, hv != 0.f ? d.sp_f[j] * iRQ * iRQ * dxinv : 0.f);
      q = make_float4(d.q2ab_f[j], d.abrw_f[j], hv, 0.f);
    }
    L.cpos[threadIdx.x] = p;
    L.cpar[threadIdx.x] = q;
    L.cw[0][threadIdx.x] = q.x;
    L.cw[1][threadIdx.x] = q.y;
  }
  int rr[NR];
  float4 pk[NR];
  float wk[NR], q2k[NR], abk[NR];
  bool kok[NR], kheavy[NR];
#pragma unroll
  for (int k = 0; k < NR; k++) {
    rr[k] = NR == 2 ? rh * 128 + lane + 64 * k : rh * 64 + lane;
    const int kr = d.cperm[item.x * 256 + rr[k]];
    pk[k] = make_float4(-1e6f, -1e6f, -1e6f, 1.f);
    wk[k] = 0.f; q2k[k] = 0.f; abk[k] = 0.f;
    kok[k] = kr >= 0;
    kheavy[k] = false;
    if (kr >= 0) {
      pk[k] = d.pos[kr];
      q2k[k] = d.q2ab_f[kr];
      abk[k] = d.abrw_f[kr];
      kheavy[k] = kr < hend;
      wk[k] = kheavy[k] ? d.sp_f[kr] * iRP * iRP * dxinv : 0.f;
    }
    if (role == 0) {
      L.rpos[k][lane] = pk[k];
      L.rw[0][k][lane] = q2k[k];
      L.rw[1][k][lane] = abk[k];
    }
  }
  __syncthreads();
  const int cbeg = (item.w & 15) + cp, cend = item.w >> 4;
  const int nbatch = (cend - cbeg + NR - 1) / NR * kBatches;
  // of the four waves behind the fronts, two add the GB sums (x, y, z and U) and
  // two the vdW ones (and V); of each two, one the rows' and one the columns'
  const int part2 = (role - kSplitFronts) >> 1;
  const bool rows = ((role - kSplitFronts) & 1) == 0;
  float g[NR][3], uv[NR];
#pragma unroll
  for (int k = 0; k < NR; k++) g[k][0] = g[k][1] = g[k][2] = uv[k] = 0.f;
#pragma unroll 1
  for (int t = 0; t <= nbatch; t++) {
    if (role < kSplitFronts) {
      if (t < nbatch) {
        const int c = cbeg + NR * (t / kBatches), s0 = t % kBatches * kSteps;
        float4 pj[EACH], pp[EACH], c1[EACH], c2[EACH];
        ChainPair m[EACH];
        float band = 0.f;
#pragma unroll
        for (int r = 0; r < EACH; r++) {
          const int k = NR == 2 ? r & 1 : 0, col = (lane - s0 - (EACH * role + r) / NR) & 63;
          pj[r] = L.cpos[c * 64 + col];
          pp[r] = L.cpar[c * 64 + col];
          const bool pair = KIND != CK_GEN || (kok[k] && (kheavy[k] || pp[r].z != 0.f) && !(diag && c * 64 + col == rr[k]));
          m[r] = chain_meet<KIND>(pk[k], pj[r], cP, cQ, pair);
          band = fmaxf(band, fabsf(m[r].u1 - 0.5f));
          if (kTwo) band = fmaxf(band, fabsf(m[r].u2 - 0.5f));
        }
        if (__builtin_expect(__ballot(band > kChainBand) != 0ull, 0)) {
#pragma unroll
          for (int r = 0; r < EACH; r++) {
            const int k = NR == 2 ? r & 1 : 0;
            chain_fix(m[r].x1, pk[k], pj[r], RQ, dxinv, m[r].k1, m[r].u1);
            if (kTwo) chain_fix(m[r].x2, pj[r], pk[k], RP, dxinv, m[r].k2, m[r].u2);
          }
        }
#pragma unroll
        for (int r = 0; r < EACH; r++) {
          c1[r] = tab_rc[m[r].k1];
          if (kTwo || kOne) c2[r] = tab_cr[kTwo ? m[r].k2 : m[r].k1];
        }
#pragma unroll
        for (int r = 0; r < EACH; r++) {
          const int k = NR == 2 ? r & 1 : 0;
          float hgb, hvw, q1, q2;
          chain_terms<KIND, QUIRK>(m[r], pj[r], pp[r], wk[k], q2k[k], abk[k], kheavy[k], c1[r], c2[r], hgb, hvw, q1, q2);
          float (*rec)[64] = L.ring[t & 1][EACH * role + r];
          rec[0][lane] = hgb;
          if (KIND != CK_HX0) rec[1][lane] = hvw;
          rec[2][lane] = q1;
          if (!kOne) rec[3][lane] = q2;
        }
      }
    } else if (t > 0 && (KIND != CK_HX0 || part2 == 0)) {
      const int c = cbeg + NR * ((t - 1) / kBatches), s0 = (t - 1) % kBatches * kSteps;
      const float (*ring)[4][64] = L.ring[(t - 1) & 1];
      if (rows) {
#pragma unroll
        for (int r = 0; r < kRec; r++) {
          const int k = NR == 2 ? r & 1 : 0, col = (lane - s0 - r / NR) & 63;
          const float4 pj = L.cpos[c * 64 + col];
          const float h = ring[r][part2][lane];
          const float ex = pj.x - pk[k].x, ey = pj.y - pk[k].y, ez = pj.z - pk[k].z;
          g[k][0] = fmaf(h, ex, g[k][0]); g[k][1] = fmaf(h, ey, g[k][1]); g[k][2] = fmaf(h, ez, g[k][2]);
          if (!kOne) uv[k] = fmaf(L.cw[part2][c * 64 + col], ring[r][3][lane], uv[k]);
        }
      } else if (!diag) {
        const float4 pj = L.cpos[c * 64 + lane];
#pragma unroll
        for (int r = 0; r < kRec; r++) {
          const int k = NR == 2 ? r & 1 : 0, row = (lane + s0 + r / NR) & 63;
          const float4 pr = L.rpos[k][row];
          const float h = ring[r][part2][row];
          const float ex = pj.x - pr.x, ey = pj.y - pr.y, ez = pj.z - pr.z;
          g[0][0] = fmaf(-h, ex, g[0][0]); g[0][1] = fmaf(-h, ey, g[0][1]); g[0][2] = fmaf(-h, ez, g[0][2]);
          uv[0] = fmaf(L.rw[part2][k][row], ring[r][2][row], uv[0]);
        }
        if (t % kBatches == 0) {                          // the chunk's last batch
          float *o = d.chsplit + ((size_t)it * kSplitSets + rh) * 2048 + c * 64 + lane;
#pragma unroll
          for (int q = 0; q < 3; q++) {
            o[(3 * part2 + q) * 256] = g[0][q];
            g[0][q] = 0.f;
          }
          o[(6 + part2) * 256] = uv[0];
          uv[0] = 0.f;
        }
      }
    }
    __syncthreads();
  }
  if (role >= kSplitFronts && rows && (KIND != CK_HX0 || part2 == 0)) {
    float *pr = d.chsplit + ((size_t)it * kSplitSets + 4 + cp) * 2048;
#pragma unroll
    for (int k = 0; k < NR; k++) {
      float *o = pr + rr[k];
#pragma unroll
      for (int q = 0; q < 3; q++) o[(3 * part2 + q) * 256] = g[k][q];
      if (!kOne) o[(6 + part2) * 256] = kheavy[k] ? uv[k] : 0.f;
    }
  }
}

template <bool QUIRK, int EACH>
__global__ __launch_bounds__(64 * kSplitWaves) void k_chain_split(Dev d) {
  __shared__ float4 tab_rc[kTblN], tab_cr[kTblN];
  __shared__ SplitLds<kSplitFronts * EACH> L;
  const int sub = d.chain_sub[blockIdx.x], it = sub >> 2, part = sub & 3;
  const int4 item = d.chain_items[it];
  const int4 bp = d.cblk[item.x], bq = d.cblk[item.y];
  const int trc = bp.x * d.ntypes + bq.x, tcr = bq.x * d.ntypes + bp.x;
  const bool one = item.z == CK_HX || item.z == CK_HX0;
  for (int k = threadIdx.x; k < kTblN; k += 64 * kSplitWaves) {
    const float4 v = d.ctab[(size_t)trc * kTblN + k];
    tab_rc[k] = v;
    tab_cr[k] = one ? chain_dpoly<QUIRK>(v) : d.ctab[(size_t)tcr * kTblN + k];
  }
  if (item.z == CK_HH && bp.x == bq.x) chain_split_item<CK_HHS, QUIRK, EACH>(d, it, part, item, tab_rc, tab_cr, L);
  else if (item.z == CK_HH) chain_split_item<CK_HH, QUIRK, EACH>(d, it, part, item, tab_rc, tab_cr, L);
  else if (item.z == CK_HX0) chain_split_item<CK_HX0, QUIRK, EACH>(d, it, part, item, tab_rc, tab_cr, L);
  else if (item.z == CK_HX) chain_split_item<CK_HX, QUIRK, EACH>(d, it, part, item, tab_rc, tab_cr, L);
  else chain_split_item<CK_GEN, QUIRK, EACH>(d, it, part, item, tab_rc, tab_cr, L);
}

// Chain-rule sums per atom: the partial sums of every item holding its block,
// in the block's fixed slot order, added in FP64 and stored as the call's
// fixed-point accumulators (no atomics; systems on the surrogate this call
// keep what k_sg_grad adds to the values k_ingest cleared).  Grid (blocks, 8
// quantities), one thread per atom slot of a block; slots loaded four ahead
// of the sum.  Without a surrogate the sums of U and V are final here, and
// their threads form the derivative pass's coefficients (uv_coeffs) at once.
__global__ __launch_bounds__(256) void k_chain_sum(Dev d) {
  const int b = blockIdx.x, q = blockIdx.y;
  const int a = d.cperm[b * 256 + threadIdx.x];
  if (a < 0) return;
  const int4 blk = d.cblk[b];
  const int mode = d.sg_on ? d.sg_state[4 * blk.y + 2] : 0;
  if (mode == 1) return;
  const float *base = d.chpart + q * 256 + threadIdx.x;
  const int *cs = d.ch_cstart + (size_t)q * (d.ncblk + 1);     // the slots that hold quantity q
  const int c0 = cs[b], c1 = cs[b + 1];
  double acc = 0.0;
  if (d.split_on) {
    // an item's column sums by row groups and its row sums by chunk parities
    // first, in FP32 in k_chain's order
    const float *set = d.chsplit + q * 256 + threadIdx.x;
    for (int c = c0; c < c1; c += 4) {
      float v[4][4];
      int m[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int e = d.ch_contrib[min(c + u, c1 - 1)], it = e >> 1, col = e & 1, n = d.chain_sets[it];
        // sets 0 .. of a column, 4 and 5 of a row (the loads have no branches,
        // so that all are in flight; what is past the count is left out)
        const size_t at = ((size_t)it * kSplitSets + (col ? 0 : 4)) * 2048;
        m[u] = c + u < c1 ? (col ? n & 7 : 1 + (n >> 3)) : 0;
#pragma unroll
        for (int g = 0; g < 4; g++) v[u][g] = set[at + (g < 2 ? g : (col ? g : 1)) * 2048];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        float t = m[u] > 0 ? v[u][0] : 0.f;
#pragma unroll
        for (int g = 1; g < 4; g++) t += m[u] > g ? v[u][g] : 0.f;
        acc += (double)t;
      }
    }
  } else if (mode == 2) {
    // only the items k_chain evaluated this call (the others hold another
    // call's sums)
    for (int c = c0; c < c1; c++) {
      const int e = d.ch_contrib[c];
      if (d.ch_done[e >> 1]) acc += (double)base[(size_t)e * 8 * 256];
    }
  } else {
    int c = c0;
    for (; c + 4 <= c1; c += 4) {
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) v[u] = base[(size_t)d.ch_contrib[c + u] * 8 * 256];
#pragma unroll
      for (int u = 0; u < 4; u++) acc += (double)v[u];
    }
    for (; c < c1; c++) acc += (double)base[(size_t)d.ch_contrib[c] * 8 * 256];
  }
  if (q >= 6) acc *= (double)(1.0f / d.pos[d.cperm[b * 256]].w);   // U, V: 1/R of the block
  const long long fix = __double2ll_rn(acc * kFix);
  d.acc_ch[8 * (size_t)a + q] = fix;
  if (q >= 6 && !d.sg_on) uv_coeffs(d, a, d.sys[blk.y], q - 6, fix);
}

// surrogate calls with out-of-range atoms (mode 2): per 64-atom chunk of a
// chain-rule block, whether it holds such an atom (one wave per chunk)
__global__ __launch_bounds__(256) void k_chain_flags(Dev d) {
  const int slot = blockIdx.x * 256 + threadIdx.x;
  const int a = d.cperm[slot];
  const bool f = a >= 0 && d.sys_sg[d.asys[a]] && d.sg_state[4 * d.asys[a] + 2] == 2 && d.sg_oor[a] != 0;
  const unsigned long long m = __ballot(f);
  if ((threadIdx.x & 63) == 0) d.ch_flag[slot >> 6] = m != 0ull ? 1 : 0;
}

template <bool QUIRK, int MODE>
__global__ __launch_bounds__(256) void k_chain(Dev d) {
  // row <- column and column <- row interval cubics; for hydrogen rows (one
  // direction) the row <- column cubics and their derivative records
  __shared__ float4 tab_rc[kTblN], tab_cr[kTblN];
  __shared__ ChainChunk ch[4];
  __shared__ int slot;
  if (d.sg_on && !*d.sg_any_plain) return;   // every system on the surrogate this call (grid-uniform)
  int staged_rc = -1, staged_cr = INT_MIN;     // nothing staged (keys are tables >= 0 or -1 - table)
  for (int it = first_item(); it < d.nchain_items;
       it = next_item(queue_head(d.queue, Q_CHAIN), &slot, d.nchain_items)) {
    const int4 item = d.chain_items[it];
    const int4 bp = d.cblk[item.x], bq = d.cblk[item.y];
    if (d.sg_on) {
      const int mode = d.sg_state[4 * bp.y + 2];               // item-uniform
      if (mode == 1) continue;                                   // surrogate call: k_sg_grad instead
      if (mode == 2) {
        // only items with an out-of-range atom among their rows or their
        // columns (the chunks of block Q the item covers) carry weight
        const int *fp = d.ch_flag + 4 * item.x, *fq = d.ch_flag + 4 * item.y;
        int any = fp[0] | fp[1] | fp[2] | fp[3];
        for (int c = item.w & 15; c < (item.w >> 4); c++) any |= fq[c];
        if (threadIdx.x == 0) d.ch_done[it] = any;
        if (!any) continue;
      }
    }
    const int nt = d.ntypes;
    const int trc = bp.x * nt + bq.x, tcr = bq.x * nt + bp.x;
    // one direction (hydrogen rows): one table, and its derivative records
    // in the second slot (key -1 - table)
    const bool one = item.z == CK_HX || item.z == CK_HX0;
    const int kcr = one ? -1 - trc : tcr;
    if (trc != staged_rc || kcr != staged_cr) {   // uniform: one item per block
      for (int k = threadIdx.x; k < kTblN; k += 256) {
        const float4 v = d.ctab[(size_t)trc * kTblN + k];
        tab_rc[k] = v;
        tab_cr[k] = one ? chain_dpoly<QUIRK>(v) : d.ctab[(size_t)tcr * kTblN + k];
      }
      staged_rc = trc;
      staged_cr = kcr;
    }
    if (item.z == CK_HH && bp.x == bq.x) chain_item<CK_HHS, QUIRK, MODE>(d, it, item, tab_rc, tab_cr, ch);
    else if (item.z == CK_HH) chain_item<CK_HH, QUIRK, MODE>(d, it, item, tab_rc, tab_cr, ch);
    else if (item.z == CK_HX0) chain_item<CK_HX0, QUIRK, MODE>(d, it, item, tab_rc, tab_cr, ch);
    else if (item.z == CK_HX) chain_item<CK_HX, QUIRK, MODE>(d, it, item, tab_rc, tab_cr, ch);
    else chain_item<CK_GEN, QUIRK, MODE>(d, it, item, tab_rc, tab_cr, ch);
    __syncthreads();
  }
}

void launch_chain(const Dev &d, const Tuning &t, hipStream_t s) {
  if (!d.nchain_items) return;
  int grid = t.chain_grid > 0 ? std::min(t.chain_grid, d.nchain_items) : d.nchain_items;
  if (d.sg_on) {
    grid = std::min(grid, kSgPersistentGrid);
    if (d.ncblk) hipLaunchKernelGGL(k_chain_flags, dim3(d.ncblk), dim3(256), 0, s, d);
  }
  const bool fixed = (d.options & 2) != 0;
  if (d.split_on) {
    // four pairs per front while every block has a CU to itself (half
    // as many batches; 2,000 atoms, 190 blocks, call 224 -> 214 us; 4,000, 450 blocks, 268 -> 274)
    const auto k = d.nchain_sub <= kSplitFour ? (fixed ? k_chain_split<false, 4> : k_chain_split<true, 4>)
                                              : (fixed ? k_chain_split<false, 2> : k_chain_split<true, 2>);
    hipLaunchKernelGGL(k, dim3(d.nchain_sub), dim3(64 * kSplitWaves), 0, s, d);
    hipLaunchKernelGGL(k_chain_sum, dim3(d.ncblk, 8), dim3(256), 0, s, d);
    return;
  }
  auto k = fixed ? k_chain<false, CM_PLAIN> : k_chain<true, CM_PLAIN>;
  if (d.nchain_items <= kChainGroupItems) k = fixed ? k_chain<false, CM_GROUP> : k_chain<true, CM_GROUP>;
  else if (d.cull_chain) k = fixed ? k_chain<false, CM_CULL> : k_chain<true, CM_CULL>;
  hipLaunchKernelGGL(k, dim3(grid), dim3(256), 0, s, d);
  if (d.ncblk) hipLaunchKernelGGL(k_chain_sum, dim3(d.ncblk, 8), dim3(256), 0, s, d);
}

// The descreening kernel's dynamic LDS limit is a property of the kernel in
// the process: it is raised to the largest table set any pack has needed
// and never lowered (a pack with fewer types must not shrink it under
// another's launches).
hipError_t prepare_pairs(int ntypes) {
  static int limit = 0;
  const int d1 = std::min(ntypes, kLdsTypes) * kTblN * (int)sizeof(float2);
  if (d1 <= limit) return hipSuccess;
  hipError_t e = hipSuccess;
  auto set = [&](const void *f, int bytes) {
    if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  };
  set((const void *)k_descreen<64, false, false>, d1);
  set((const void *)k_descreen<128, false, false>, d1);
  set((const void *)k_descreen<256, false, false>, d1);
  set((const void *)k_descreen<64, false, true>, d1);
  set((const void *)k_descreen<128, false, true>, d1);
  set((const void *)k_descreen<256, false, true>, d1);
  if (e == hipSuccess) limit = d1;
  return e;
}

}  // namespace agb
