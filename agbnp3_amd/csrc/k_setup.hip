// Per-call setup kernels: coordinate ingest, per-system cell grids, heavy-atom
// neighbour list.
//
// The neighbour list must equal the reference's exactly (it fixes the shape
// of the overlap tree): heavy j > i with
//     d2 = (dx*dx + dy*dy) + dz*dz  <  ((R_i + R_j) * 1.6f)^2
// evaluated in FP32 without contraction, each row sorted by (d2, j)
// (reference agbnp3.c:4028-4066, agbnp3_fcompare agbnp3.c:3766-3784).
#include "agb_common.h"
#include "agb_device.h"

namespace agb {

// ---------------------------------------------------------------- ingest
// caller-order FP64 coordinates -> internal FP32 (x, y, z, R); clears the
// scatter accumulators and work-queue heads of the call.  A thread takes its
// caller's atom (the coordinates may lie in host memory, which is read in
// whole lines) and clears its internal one.
__global__ __launch_bounds__(256) void k_ingest(Dev d, const double *__restrict__ x,
                                                const double *__restrict__ y,
                                                const double *__restrict__ z) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (d.sg_on && i < d.nsys) d.sg_state[4 * i + 3] = 0;   // surrogate: out-of-range flag of the call
  if (d.sg_on && i == 0) *d.sg_any_plain = 0;
  if (i < d.n) {
    const int a = d.ext2int[i];
    d.pos[a] = make_float4((float)x[i], (float)y[i], (float)z[i], d.R[a]);
    const SysInfo &S = d.sys[d.asys[i]];
    if (i < S.a0 + S.nh) {
      d.acc_vol[i] = 0;
      d.acc_sa[i] = 0;
      d.acc_derh[i] = 0;
#pragma unroll
      for (int k = 0; k < TG_N; k++) d.acc_grad[(size_t)i * TG_N + k] = 0;
    }
    d.acc_gbA[i] = 0;
    d.acc_beta[i] = 0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      d.acc_hb[3 * (size_t)i + q] = 0;
      d.acc_gbg[3 * (size_t)i + q] = 0;
    }
    if (d.sg_on || !d.nchain_items)          // (else k_chain_sum stores every one)
#pragma unroll
      for (int q = 0; q < 8; q++) d.acc_ch[8 * (size_t)i + q] = 0;
  }
  if (i < Q_COUNT * kQueueSpread) d.queue[i * kQueueStride] = 0;
  if (i < kCountSlots) {
    d.counters[kCountBase + 8 * i] = 0;
    d.counters[kCountBase + 8 * i + 1] = 0;
  }
  if (i == 0) d.counters[kCountWs] = 0;
  if (i == 0) {
    *d.status = 0;
    for (int k = 0; k < 8; k++) d.counters[k] = 0;

    if (d.skin > 0.f) {       // neighbour-list reuse: forced rebuilds
      // [0] built, [1] calls, [2] rebuild this call, [3] rebuilds, [4] the
      // last build kept incomplete candidate rows (a row past kCandCap: that
      // call's own list was complete, the kept candidates are not, so every
      // call rebuilds until a build fits)
      const int calls = d.nbl_state[1] + 1;
      d.nbl_state[1] = calls;
      const bool rebuild =
          d.nbl_state[0] == 0 || d.nbl_state[4] != 0 || (d.reuse_every > 0 && calls % d.reuse_every == 0);
      d.nbl_state[2] = rebuild;
      if (rebuild) d.nbl_state[4] = 0;
    }
  }
}

void launch_ingest(const Dev &d, const double *x, const double *y, const double *z, hipStream_t s) {
  const int nblk = (d.n + 255) / 256;
  if (nblk) hipLaunchKernelGGL(k_ingest, dim3(nblk), dim3(256), 0, s, d, x, y, z);
}

// ------------------------------------------------------------ cell grid
// One workgroup per system: bounding box of its heavy atoms, grid sizing
// (cell edge >= largest heavy-heavy and site-heavy cutoff, so a 27-cell
// stencil is complete), counting sort of the heavy atoms into cells.
// kMaxCells bounds the LDS histogram; the edge grows until the grid fits.
__global__ __launch_bounds__(1024) void k_cells(Dev d) {
  __shared__ int cnt[kMaxCells];
  __shared__ int wsum[16], wpre[16];
  __shared__ float box[6][16];
  __shared__ GridParams g;
  const SysInfo S = d.sys[blockIdx.x];
  float lo[3], hi[3];
  block_bbox(d.pos, S.a0, S.nh, box, lo, hi);
  if (threadIdx.x == 0) {
    const float cs = fmaxf(kNbOffset * 2.0f * S.rmax_heavy, kNbOffset * (S.rmax_heavy + kHbRadius)) * 1.001f + 1e-3f;
    g = make_grid(lo, hi, cs);
    d.grid[blockIdx.x] = g;
  }
  __syncthreads();
  // the order inside a cell is irrelevant (rows are re-sorted)
  bin_atoms(g, d.pos, S.a0, S.nh, d.cell_tmp, d.cell_start + (size_t)blockIdx.x * (kMaxCells + 1), d.cell_atoms, cnt,
            wsum, wpre, false);
}

void launch_cells(const Dev &d, hipStream_t s) {
  if (d.nsys) hipLaunchKernelGGL(k_cells, dim3(d.nsys), dim3(1024), 0, s, d);
}

// ------------------------------------------------------- neighbour list
// one wavefront per heavy row; candidates from the 27-cell stencil are
// compacted into LDS with ballots, then rank-sorted by (d2, j).
//
// Reuse across calls (d.skin > 0): a rebuild also keeps, per row, every pair
// within the cutoff plus the skin, and the positions it was built from.
// While no heavy atom has moved more than skin/2 since, every pair inside the
// cutoff is among those candidates, so later calls re-test and re-sort just
// the candidates with the same FP32 arithmetic and get the same list as a
// full rebuild.  k_guard decides on the device (graph replays included).
// Bound: a row's chain of dependent loads (atom of a cell slot, its position)
// and, in the sort, of LDS reads.  Four steps' loads in flight and one 64-bit
// key per entry, its reads eight ahead: 2,000 atoms 12.2 -> 7.0 us, 6,000 21.0
// -> 9.2, 25,000 22.1 -> 15.1, 24 x 6000 89 -> 63.  (Positions kept in cell
// order by k_cells: 8.4 us at 6,000, but k_cells, one block, 7.8 -> 12.2.)
constexpr int kNbWaves = 4, kNbAhead = 4;

template <int CAP>
__global__ __launch_bounds__(64 * kNbWaves) void k_nblist(Dev d) {
#pragma clang fp contract(off)
  // a row's entries as one key: d2 >= 0, so its bits order as the number
  __shared__ unsigned long long key[kNbWaves][CAP];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int h = blockIdx.x * kNbWaves + w;
  if (h >= d.nh) return;                    // wave-uniform (no block barrier follows)
  const int i = d.hrow[h];
  const int sys = d.asys[i];
  const float4 pi = d.pos[i];
  const bool reuse = d.skin > 0.f;
  const bool rebuild = !reuse || d.nbl_state[2] != 0;
  int cnt = 0;
  // exact test of pair (i, j); the candidate test (reuse) on the same d2
  auto test = [&](const float4 &pj, bool want_cand, bool &pass, bool &cpass, float &d2) {
    const float ex = __fsub_rn(pj.x, pi.x), ey = __fsub_rn(pj.y, pi.y), ez = __fsub_rn(pj.z, pi.z);
    d2 = __fadd_rn(__fadd_rn(__fmul_rn(ex, ex), __fmul_rn(ey, ey)), __fmul_rn(ez, ez));
    const float u = __fmul_rn(__fadd_rn(pi.w, pj.w), kNbOffset);
    pass = d2 < __fmul_rn(u, u);
    if (want_cand) {
      const float uc = u + d.skin + 1e-3f;
      cpass = d2 < uc * uc;
    }
  };
  auto keep = [&](bool pass, int j, float d2) {
    const unsigned long long m = __ballot(pass);
    if (pass) {
      const int slot = cnt + __popcll(m & ((1ull << lane) - 1ull));
      if (slot < CAP) key[w][slot] = (unsigned long long)__float_as_uint(d2) << 32 | (unsigned)j;
    }
    cnt += __popcll(m);
  };
  if (rebuild) {
    const GridParams g = d.grid[sys];
    const int *cstart = d.cell_start + (size_t)sys * (kMaxCells + 1);
    int *cand = reuse ? d.cand_nbr + (size_t)h * kCandCap : nullptr;
    int ccnt = 0;
    int cx, cy, cz;
    cell_coords(g, pi.x, pi.y, pi.z, cx, cy, cz);
    // candidates over the whole stencil, kNbAhead steps of 64 in flight; the
    // (d2, j) sort below makes the list independent of the order of enumeration
    int start[9], off[9];
    const int total = stencil_segments(g, cstart, cx, cy, cz, start, off);
    for (int base = 0; base < total; base += 64 * kNbAhead) {
      int j[kNbAhead];
      float4 pj[kNbAhead];
#pragma unroll
      for (int u = 0; u < kNbAhead; u++) j[u] = d.cell_atoms[stencil_slot(start, off, min(base + 64 * u + lane, total - 1))];
#pragma unroll
      for (int u = 0; u < kNbAhead; u++) pj[u] = d.pos[j[u]];
#pragma unroll
      for (int u = 0; u < kNbAhead; u++) {
        if (base + 64 * u >= total) break;             // wave-uniform
        bool pass = false, cpass = false;
        float d2 = 0.f;
        if (base + 64 * u + lane < total && j[u] > i) test(pj[u], reuse, pass, cpass, d2);
        keep(pass, j[u], d2);
        if (reuse) {
          const unsigned long long mc = __ballot(cpass);
          if (cpass) {
            const int slot = ccnt + __popcll(mc & ((1ull << lane) - 1ull));
            if (slot < kCandCap) cand[slot] = j[u];
          }
          ccnt += __popcll(mc);
        }
      }
    }
    if (reuse && lane == 0) {
      if (ccnt > kCandCap) d.nbl_state[4] = 1;      // every writer stores the same 1
      d.cand_nne[h] = min(ccnt, kCandCap);
      d.ref_pos[i] = pi;
      if (h == 0) {
        d.nbl_state[0] = 1;
        d.nbl_state[3] += 1;       // rebuilds since reuse was set
      }
    }
  } else {
    const int nc = d.cand_nne[h];
    const int *cand = d.cand_nbr + (size_t)h * kCandCap;
    for (int base = 0; base < nc; base += 64) {
      const int k = base + lane;
      bool pass = false, cpass = false;
      int j = -1;
      float d2 = 0.f;
      if (k < nc) {
        j = cand[k];
        test(d.pos[j], false, pass, cpass, d2);
      }
      keep(pass, j, d2);
    }
  }
  int m = cnt;
  if (m > CAP) {
    if (lane == 0) atomicOr(d.status, ST_NBLIST_OVERFLOW);
    m = CAP;
  }
  wave_sync();
  for (int e = lane; e < m; e += 64) {
    const unsigned long long ke = key[w][e];
    int rank = 0;
#pragma unroll 8
    for (int f = 0; f < m; f++) rank += key[w][f] < ke;
    d.nbr[(size_t)h * d.cap + rank] = (int)(unsigned)ke;
  }
  if (lane == 0) d.nne[h] = m;
}

// rebuild decision of the neighbour-list reuse: any heavy atom farther than
// skin/2 from where the kept candidates were built
__global__ __launch_bounds__(256) void k_guard(Dev d) {
  const int h = blockIdx.x * 256 + threadIdx.x;
  if (h >= d.nh || d.nbl_state[0] == 0) return;
  const int i = d.hrow[h];
  const float4 p = d.pos[i], r = d.ref_pos[i];
  const float ex = p.x - r.x, ey = p.y - r.y, ez = p.z - r.z;
  const float half = 0.5f * d.skin;
  if (!(ex * ex + ey * ey + ez * ez <= half * half)) d.nbl_state[2] = 1;   // also for non-finite input
}

void launch_nblist(const Dev &d, hipStream_t s) {
  const int nblk = (d.nh + kNbWaves - 1) / kNbWaves;
  if (nblk == 0) return;
  if (d.skin > 0.f) hipLaunchKernelGGL(k_guard, dim3((d.nh + 255) / 256), dim3(256), 0, s, d);
  if (d.cap <= 64)
    hipLaunchKernelGGL(k_nblist<64>, dim3(nblk), dim3(64 * kNbWaves), 0, s, d);
  else if (d.cap <= 128)
    hipLaunchKernelGGL(k_nblist<128>, dim3(nblk), dim3(64 * kNbWaves), 0, s, d);
  else
    hipLaunchKernelGGL(k_nblist<256>, dim3(nblk), dim3(64 * kNbWaves), 0, s, d);
}

}  // namespace agb
