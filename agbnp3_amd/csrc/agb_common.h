// Shared definitions of the gfx950 AGBNP3 engine: model constants, the device
// view of a pack of systems passed by value to every kernel, and the launcher
// prototypes implemented by the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace agb {

// ---- model constants (reference agbnp3_private.h:57-137, agbnp3.c:1230-1236)
constexpr double kPi = 3.14159265359;   // the reference's pi
constexpr float kPiF = 3.14159265359f;
constexpr float kKFC = 2.5f;            // Gaussian exponent factor a = KFC / R^2
constexpr float kPFC = 2.97354f;        // Gaussian prefactor
constexpr float kRadInc = 0.5f;         // R = r + 0.5
constexpr float kNbOffset = 1.6f;       // neighbour test d < 1.6 (Ri + Rj)
constexpr float kVolMinA = 0.01f, kVolMinB = 0.1f;  // overlap-volume switch window
constexpr int kMaxOrder = 5;            // overlaps of order 2..5
constexpr double kTokcal = 332.0;
constexpr double kRwNp = 1.4;           // water radius in the vdW term
constexpr float kHbLength = 2.5f, kHbRadius = 1.4f;
constexpr float kHbSwA = 0.65f, kHbSwB = 1.0f, kHbSwA0 = 0.6f;
// atoms from which a call runs the water-site kernels on a second stream, and
// from which one tier of the derivative pass has that stream.  A process's
// streams share four hardware queues, so several instances in flight gain less
// by it (us a call, with the stream against without: one of 2,000 atoms 200
// against 210, four 97 to 103 against 113, eight 97 to 103 against 89 to 98; one
// of 11,003 419 against 427, four 259 against 290)
constexpr int kForkAtoms = 16384;
constexpr int kSideAtoms = 512;
// heavy atoms from which the derivative pass's second tier starts before the
// first: its blocks, two to a CU, otherwise find no room before that one ends
// (12 x 6000, 35,000 heavy atoms, call 1193 -> 1180 us, 64 systems of 2,000 1451
// -> 1431, 60,000 atoms 3700 -> 3661, 40,000, 19,000 heavy, 1933 -> 1922; 25,000
// and 34,000, 12,000 and 16,000 heavy, no change, 11,000 429 -> 437).  What the
// call's own stream is given starts at once, the second stream's 6 us later,
// behind its event; in a replayed graph the tier recorded first starts at once
// (both seen in a kernel trace), so a capture keeps the second tier, recorded
// first, on the side branch (the other way 24 x 6000 2230 -> 2272 us)
constexpr int kBigFirst = 16384;
// columns of a descreening group with a box of its own
constexpr int kBoxCols = 16;
// extents of a solute, in units of the longest table's reach (46 A for heavy
// atoms of up to 1.8 A), from which the descreening and the chain rule skip
// far columns by boxes.  Share of the pairs skipped and time, synthetic
// solutes: descreening 25,000 atoms (1.7 reaches across) 7 %, 169 -> 183 us;
// 40,000 (2.0) 19 %, 431 -> 391 us; 150,000 (3.1) 60 %, 3.66 -> 2.15 ms.
// Chain rule, whose sums fix the order of the atoms inside its blocks: 40,000
// 0.4 %, 567 -> 585 us; 150,000 14 %, 6.94 -> 6.64 ms.
constexpr float kCullDesc = 1.85f, kCullChain = 2.6f;
// most items of the descreening by tiles (measured: k_desc_sites)
constexpr int kDtItems = 2048;
// most items of a chain-rule launch whose lookups are grouped: four per CU
constexpr int kChainGroupItems = 1024;
// most chain-rule items of a launch that takes them longest first, by their
// kinds' times (k_chain at 25,000 atoms, 3,800 items for 1,280 places: 270 us
// by pair count alone, 237 by time; the order does not touch the sums).  At
// 40,000 atoms, 9,700 items, no difference is left to gain
constexpr size_t kChainByTime = 8192;
// most items of a chain rule by row groups (k_chain_split; calls of 4,000, 5,300
// and 6,000 atoms, 155, 250 and 300 items, 302 -> 264, 310 -> 277 and 309 ->
// 300 us; 6,600, 360 items, 323 -> 320), and most of its blocks for which a
// front takes four pairs at a time
constexpr int kSplitItems = 384, kSplitSets = 6, kSplitFour = 256;
// most items of the GB pairs by chunks (k_gb_split; a call of 2,000 atoms, 36
// items, 215 -> 208 us, of 2,700, 66 items, 233 -> 234, of 4,000, 136 items, 259 -> 271),
// and sets of 4 x 256 numbers that an item's sums take there
constexpr int kGbSplitItems = 48, kGbSets = 5;
// nodes of one order that the overlap tree's first tier holds in LDS
constexpr int kLevelCap = 128;
// per-call device counters: [0..7] scalars (see agbnp3_get_counts); the
// overlap-tree kept / evaluated totals spread over kCountSlots 64-byte lines
// (kCountBase + 8 s, + 1), so the blocks' adds at exit do not queue on one
// address
constexpr int kCountSlots = 32, kCountBase = 8;
// water sites with more candidates than the first free-volume launch holds
constexpr int kCountWs = kCountBase + 2;
constexpr int kCounters = kCountBase + 8 * kCountSlots;
constexpr int kTblN = 512;              // spline nodes per table (y[511] = 0)
constexpr float kTblAmax = 20.0f;

// fixed-point scale of the order-independent (deterministic) scatter sums
constexpr double kFix = 4294967296.0;   // 2^32
constexpr double kFixInv = 1.0 / 4294967296.0;

// status word bits (device side capacity / topology checks)
enum : int {
  ST_NBLIST_OVERFLOW = 1,   // a neighbour-list row exceeded the row capacity
  ST_TREE_OVERFLOW = 2,     // a root of pass B's first tier outgrew its buffers
  ST_WS_OVERFLOW = 4,       // a water site had more candidates than its buffer
  ST_GRID_OVERFLOW = 8,     // cell grid larger than allocated
};

// kept neighbour candidates per heavy row (neighbour-list reuse)
constexpr int kCandCap = 256;

// energy partial-sum slots (per block, reduced in a fixed order)
enum : int {
  EP_CAV = 0, EP_CORR_CAV, EP_MOLVOL, EP_VDW, EP_CORR_VDW, EP_SELF, EP_PAIR, EP_HB, EP_COUNT
};

// per-overlap-tree accumulator layout (int64 fixed point per heavy atom)
enum : int { TG_GB = 0, TG_VW = 3, TG_CAV = 6, TG_HB = 9, TG_N = 12 };

// a placed water site (one record per wave of the free-volume kernel, in LDS)
struct WSite {
  float pos[3];
  float khb;
  int parent[4];
  int nparents;
  int type;
  float dpos[4][3][3];   // d pos_i / d x_{parent p, j}
};

// static description of the water sites of one HB-active atom
struct WsDef {
  int atom;          // pack index of the acceptor / polar hydrogen
  int kind;          // placement geometry (WS_* below)
  int nsite;         // sites this atom creates
  int first;         // index of its first site
  int p[5];          // topology atoms used by the geometry
};
enum : int { WS_POLARH = 0, WS_TRIGONAL1, WS_TRIGONAL_S, WS_TRIGONAL_OOP, WS_TRIGONAL2,
             WS_TETRAHEDRAL2, WS_TETRAHEDRAL3, WS_TETRAHEDRAL1 };

struct GridParams {
  float lo[3];
  float cs, inv_cs;
  int dim[3];
  int ncell;
};

// radius types whose descreening tables a block holds in LDS
constexpr int kLdsTypes = 16;

// cells per system grid (LDS histogram of the binning kernel)
constexpr int kMaxCells = 8192;

// One system (an agbnp3 instance) inside a pack.  A pack concatenates the
// per-atom arrays of its systems; inside each system heavy atoms come first.
struct SysInfo {
  int a0, n, nh;        // atoms [a0, a0 + n), heavy atoms [a0, a0 + nh)
  int h0;               // its first heavy row (rows number the pack's heavy atoms)
  int ws0, nws;         // water sites [ws0, ws0 + nws)
  int blk0, nblk;       // atom blocks [blk0, blk0 + nblk) (energy partials)
  int tile0, ntile;     // GB tile-pair energy slots [tile0, tile0 + ntile)
  int dp0;              // its descreening tile sums (dt_on): tile t of atom a0 + k at dpart[dp0 + t n + k]
  float df;             // dielectric factor -0.5 (1/eps_in - 1/eps_out), FP32
  float rmax_heavy;     // largest heavy-atom R (cell size)
  double df64;          // same factor in FP64
};

// ---- Born-radius surrogate (MLP 66 -> 128 -> 128 -> 128 -> 1)
constexpr int kSgNShell = 16, kSgNFeat = 66, kSgKPad = 96, kSgHid = 128;
constexpr int kSgPad = 4, kSgRow = 24;   // padded ds/dF rows: zeros | 16 shells | zeros
constexpr int kSgBlk = 64;               // atoms per descriptor row block
constexpr int kSgNbrCap = 1536;          // neighbours per atom within kSgCut + kSgSkin
constexpr float kSgCut = 12.0f, kSgSkin = 1.5f;
// largest grid of the descreening and chain-rule kernels while a surrogate
// is attached (their items are then often all skipped)
constexpr int kSgPersistentGrid = 2048;
// FP32 master parameter layout: W1 [66][128], b1, W2 [128][128], b2, W3, b3, w4 [128], b4
constexpr int kSgOffW1 = 0;
constexpr int kSgOffB1 = kSgOffW1 + kSgNFeat * kSgHid;
constexpr int kSgOffW2 = kSgOffB1 + kSgHid;
constexpr int kSgOffB2 = kSgOffW2 + kSgHid * kSgHid;
constexpr int kSgOffW3 = kSgOffB2 + kSgHid;
constexpr int kSgOffB3 = kSgOffW3 + kSgHid * kSgHid;
constexpr int kSgOffW4 = kSgOffB3 + kSgHid;
constexpr int kSgOffB4 = kSgOffW4 + kSgHid;
constexpr int kSgNParam = kSgOffB4 + 1;

// device view of a model: bf16 weights row-major [in][out] (backward) and
// transposed [out][in] (forward, staged in LDS), FP32 biases / output layer
// (pointers into the master parameters), normalisation and training window
struct SgModel {
  const unsigned short *w1, *w2, *w3, *wt1, *wt2, *wt3;
  const float *b1, *b2, *b3, *w4, *b4;
  const float *xmu, *xsd_inv, *xlo, *xhi;   // per input feature (66)
  float ymu, ysd;
};

// training batch buffers (feature-major activations and deltas)
struct SgTrain {
  const float *X;            // normalised inputs [N][kSgKPad]
  const float *y;            // normalised targets [N]
  unsigned short *A0, *A1, *A2, *D1, *D2, *D3;   // [features][B] bf16
  float *A3, *dy, *err2;
  // loss per row w_abs e^2 + w_diff (e - e_partner)^2, rows 2k and 2k+1 a pair
  float w_abs, w_diff;
};

// work-queue heads (cleared by the ingest kernel of every call)
enum : int { Q_DESC = 0, Q_GB, Q_CHAIN, Q_TREE_A, Q_TREE_B, Q_TREE_BA, Q_TREE_BB, Q_COUNT };
// each queue has kQueueSpread heads, kQueueStride uints (64 bytes) apart: a
// block takes its later items from head blockIdx mod kQueueSpread
constexpr int kQueueSpread = 8, kQueueStride = 16;
constexpr int kQueueWords = Q_COUNT * kQueueSpread * kQueueStride;

// Device view of a pack of one or more systems, passed by value to every kernel.
struct Dev {
  int n, nh;             // atoms, heavy rows of the pack
  int nsys;
  int ntypes;            // radius types (union over the systems)
  int cap;               // neighbour-list row capacity
  int nws;               // water sites
  int options;
  const SysInfo *sys;
  const int *asys;       // system of each atom
  const int *hrow;       // atom of each heavy row
  // static inputs (pack order)
  const int *ext2int;    // caller order (concatenated per system) -> pack order
  const float *R;        // r + 0.5
  const float *q;
  const int *rtype;
  const float *galpha;   // KFC / R^2 (heavy)
  const float *igamma, *sgamma, *ialpha, *salpha, *hbcorr_f;
  const double *vols;    // 4/3 pi R^3
  const float2 *tbl;     // [ntypes*ntypes][512] (y, y2)
  // the same tables as per-interval cubics in the fraction u of the
  // interval, (c0, c1, c2, c3) [ntypes*ntypes][512]; interval 511 is zero
  const float4 *ctab;
  float tdx, tdxinv;
  // row blocks of the spline kernels: rows of one radius type and one system
  int rows;              // rows per block (64, 128 or 256)
  int nrow_blocks;
  const int *row_perm;   // [nrow_blocks][rows] pack atom or -1
  const int4 *rblk;      // per block: radius type, system, hydrogen rows only, -
  // descreening by tiles (dt_on; a call that few row blocks make up): items
  // of a row block x 256 columns (row block, column range, place of the sums
  // before adding the atom's number), and the tiles per run of k_born's sum
  int dt_on, ndt_items, dt_run;
  const int4 *dt_items;
  float *dpart;
  // work items, sorted by decreasing size, taken from the queues by
  // persistent blocks: descreening / chain (row block, column range), GB
  // tile pairs (row range, column range; diagonal when they start together)
  const int4 *desc_items, *chain_items, *gb_items;   // chain items: (row block, column block, kind, chunks c0 | c1 << 4)
  const int *cperm;      // chain-rule blocks: [ncblk][256] pack atom or -1
  // chain-rule partial sums: per item, its row side and column side, 8
  // quantities x 256 atoms (FP32 tile sums, [item][side][q][256]); per block
  // the (item, side) slots holding its atoms' sums, in a fixed order
  float *chpart;
  // the chain rule by row groups (split_on): blocks (item << 2 | row group, or
  // chunk parity << 1 | half of the rows), and per item kSplitSets sets of 8
  // quantities x 256 atoms: its column sums by row group, then (4, 5) its row
  // sums by parity; chain_sets: column sets, + 8 with a second parity
  int split_on, nchain_sub;
  const int *chain_sub, *chain_sets;
  float *chsplit;
  int *ch_done;          // [nchain]: item evaluated this call (hybrid surrogate calls skip items)
  int *ch_flag;          // [4 ncblk]: 64-atom chunk holds an out-of-range atom (hybrid calls)
  const int *ch_cstart;  // [8][ncblk + 1]: per summed quantity, each block's run of ch_contrib
  const int *ch_contrib; // item * 2 + side
  const int4 *cblk;      // per chain block: radius type, system, hydrogens only, heavy atoms only
  int ncblk;
  int ndesc_items, nchain_items, ngb_items;
  const int *gb_eslot;   // energy slot of each GB item
  unsigned *queue;       // [Q_COUNT][kQueueSpread][kQueueStride] (heads at stride 0)
  const int2 *ablk;      // atom blocks: [start, end) inside one system
  int nablk;
  const WsDef *wsdef;
  const int2 *ws_site;   // per site: its HB-active atom's entry of wsdef, its number there
  const int *ws_stale0;  // per site: atom whose spe the first subtraction reads (quirk Q3); -1: none (0)
  // per-call state
  float4 *pos;           // x, y, z, R
  GridParams *grid;      // [nsys]
  int *cell_start;       // [nsys][kMaxCells + 1]
  int *cell_atoms, *cell_tmp;          // [n]: heavy atoms by cell, per system range
  int *nne, *nbr;                      // [nh], [nh][cap]
  // neighbour-list reuse (skin > 0): candidates within cutoff + skin, the
  // heavy-atom positions they were built from, and [0] candidates valid,
  // [1] calls, [2] rebuild this call, [3] rebuilds so far, [4] the last
  // build's candidate rows incomplete (a row past kCandCap)
  float skin;
  int reuse_every;                     // forced rebuild every this many calls (0: guard only)
  int *cand_nne, *cand_nbr;            // [nh], [nh][kCandCap]
  float4 *ref_pos;                     // [n]
  int *nbl_state;
  int *status;
  long long *acc_vol, *acc_sa;         // tree pass A [n]
  long long *acc_grad;                 // tree pass B [n][TG_N]
  long long *acc_hb;                   // HB direct gradient [n][3]
  long long *acc_derh;                 // [n]
  long long *acc_beta;                 // descreening sums [n]
  long long *acc_gbA, *acc_gbg;        // GB pairs: A_i [n], gradient [n][3]
  long long *acc_ch;                   // chain rule [n][8]: gb xyz, vdw xyz, U, V
  unsigned long long *hstat;           // pinned host memory (may be null): the call's status word and counters 0..3
  unsigned long long *counters;        // [0] kept overlaps [1] evaluated [2] nbl entries [3] max row
                                       // [4] roots queued for the second breadth-first tier (pass A; pass B
                                       //     takes the same list), [5] unused
                                       // [6], [7] roots walked depth first (pass A, B)
  int *tree_ovf;                       // [2][nh] heavy rows of the roots queued for the second tier, for pass B's depth-first walk
  uint2 *tree_cnt;                     // [nh] overlaps kept and evaluated by pass A's first tier (in A's memory, until k_q2ab)
  int tree_cap_b;                      // nodes of one order pass B's first tier takes (kLevelCap; lower for tests)
  unsigned char *tree_tier;            // [nh] pass A's first tier: 0 walked there, 1 queued for the next
  double *volumep_raw, *sa_raw, *sa_f, *sp, *spe, *psvol, *gammap;   // [n]
  float *sp_f, *spe_f;                 // FP32 copies for pair kernels
  float4 *dcol;                        // heavy atoms as descreening columns: x, y, z, 1/(R dx)
  float2 *dcw;                         // and (sp / R, radius type as int bits)
  // boxes the spline kernels skip far columns by: per 16 descreening columns
  // ([nablk][16], a system's from blk0) low corner and smallest 1/(R dx),
  // high corner; per 64-atom chunk of a chain-rule block its corners
  int cull_desc, cull_chain;
  float4 *cbox;
  float4 *chbox;
  double *beta, *br, *brw, *swf;       // [n]
  float *br_f;
  int gbs_on;                          // GB pairs by chunks:
  float *gbsplit;                      // per GB energy slot its row sums by chunk and its column sums
  double *gbener;                      // and its energy by chunk
  double *gb_epart;                    // per GB energy slot: sum of q_i q_j / f
  double *A, *q2ab, *abrw;             // [n]
  float *q2ab_f, *abrw_f;
  double *deru, *derv, *derus, *dervs, *derh;   // [n]
  float *deru_f, *derv_f, *derus_f, *dervs_f, *derh_f, *gammap_f;
  int *ws_ovf;                         // [nws] sites for the second free-volume launch
  int ws_cap1;                         // candidates the first launch takes (128; lower for tests)
  double *ws_part;                     // per-site energy khb*s
  double *epart;                       // [EP_COUNT][nablk]
  // Born-radius surrogate (sg_on): per system [0] calls, [1] anchored,
  // [2] mode of this call (0: plain, 1: surrogate, 2: surrogate with the
  // plain kernels for the atoms whose descriptors are out of range), [3]
  // atoms out of range this call; sg_oor[i]: atom i out of range this call
  int sg_on, sg_every, sg_grid;
  int *sg_oor;
  int *sg_count;                       // per system: calls in mode 0, 1, 2 since sg_attach ([4 nsys])
  SgModel sg;
  const int *sys_sg;                   // per system: model attached
  int *sg_state;
  int *sg_any_plain;                   // [0]: some system of the pack runs the plain kernels this call
  const int2 *sg_rows;                 // kSgBlk-slot row blocks inside systems (slots of sg_catoms)
  int nsg_rows;
  // descriptor neighbour lists: every pair within kSgCut + kSgSkin, kept
  // while no atom of the system has moved more than kSgSkin / 2 since.  Rows
  // are the atoms in cell order (sg_catoms, from the same build); row r of
  // block b: neighbour k at sg_nbr[(b * kSgBlk + r) * kSgNbrCap + k],
  // heavy neighbours from k = 0, hydrogens (heavy rows only) down from
  // k = kSgNbrCap - 1; sg_nn[a] = (heavy, hydrogen) counts.
  int *sg_nbr;                         // neighbour slots (positions in sg_catoms)
  int2 *sg_nn;
  float4 *sg_ref;                      // [n] positions the lists were built from
  int *sg_slot;                        // [n] slot of each atom in sg_catoms
  // per call, in slot order: position and R, self-volume fraction (0 for
  // hydrogens), and (q2ab, abrw, self-volume fraction, 0) for the gradient
  // pass (one gather per neighbour); sg_F, sg_X, sg_s and sg_dsdF are also in
  // slot order
  float4 *sg_spos;
  float *sg_sgam;
  float4 *sg_sw;
  int *sg_nbl;                         // per system [0] built, [1] rebuild this call, [2] builds, [3] overflow
  GridParams *sg_grid_p;               // per system all-atom cell grid
  int *sg_cstart, *sg_catoms, *sg_ctmp;  // [nsys][kMaxCells + 1], [n], [n]
  float *sg_F;                         // raw shell descriptors [n][64] (slot order)
  float *sg_X;                         // normalised input [n][kSgKPad] (slot order)
  float *sg_s;                         // predicted s [n] (slot order)
  float *sg_dsdF;                      // ds/dF by channel: [4][n][kSgRow] (slot order): kSgPad zeros, the
                                       // 16 shells, zeros (any 4 consecutive shells of a B-spline one read)
  float *sg_target;                    // plain descreening sum of the call [n]
  double *sg_c, *sg_delta;             // anchor corrections, surrogate error at the anchor [n]
  double *sg_err;                      // per system: first-order Delta G error estimate
};

// launch shapes chosen per pack (the autotuner may change them)
struct Tuning {
  int rows = 256;          // rows per spline-kernel block
  int desc_chunk = 0;      // columns per descreening item (0: whole system)
  int chain_chunk = 0;     // columns per chain-rule item: 64, 128 or 256 of a block (0: 256)
  int desc_grid = 0;       // persistent blocks (0: one per item)
  int gb_grid = 0;
  int chain_grid = 0;
  int tree_grid = 0;       // persistent blocks of the first overlap-tree tier (0: one per root)
};

// ---- launchers (kernel translation units) ------------------------------
void launch_ingest(const Dev &d, const double *x, const double *y, const double *z, hipStream_t s);
void launch_cells(const Dev &d, hipStream_t s);
void launch_nblist(const Dev &d, hipStream_t s);
void launch_tree(const Dev &d, const Tuning &t, int pass, hipStream_t s);
// one tier of a pass: 0 breadth first, 1 breadth first with large levels (the
// roots pass A's first tier queued; past those levels, depth first)
void launch_tree_tier(const Dev &d, const Tuning &t, int pass, int tier, hipStream_t s);
hipError_t prepare_tree();
void launch_scale(const Dev &d, hipStream_t s);
void launch_descreen(const Dev &d, const Tuning &t, hipStream_t s);
void launch_born(const Dev &d, hipStream_t s);
void launch_gbpair(const Dev &d, const Tuning &t, hipStream_t s);
void launch_q2ab(const Dev &d, hipStream_t s);
void launch_chain(const Dev &d, const Tuning &t, hipStream_t s);
void launch_uv(const Dev &d, hipStream_t s);
hipError_t prepare_pairs(int ntypes);
void launch_ws_free(const Dev &d, hipStream_t s);
// descreening by tiles and the water sites' free volumes (dt_on)
void launch_desc_sites(const Dev &d, hipStream_t s);
bool desc_sites_few(const Dev &d);       // 64 rows per block there
hipError_t prepare_sites(int ntypes);
void launch_sg_front(const Dev &d, hipStream_t s);
void launch_sg_grad(const Dev &d, hipStream_t s);
void launch_sg_audit(const Dev &d, hipStream_t s);
hipError_t prepare_surrogate();
void launch_sg_append(const Dev &d, float *F, float *target, int at, hipStream_t s);
void launch_sg_infer(const SgModel &m, const float *X, int n, float *s_out, float *dsdF, int grid, hipStream_t s);
size_t sg_mlp_lds();
void launch_sg_train_step(const SgModel &m, const SgTrain &t, int r0, int B, float *grad, float *loss,
                          int grid, hipStream_t s);
void launch_sg_adam(float *p, const float *g, float *mom, float *vel, float lr, int step, hipStream_t s);
void launch_sg_pack(const float *p, unsigned short *w1, unsigned short *w2, unsigned short *w3, unsigned short *wt1,
                    unsigned short *wt2, unsigned short *wt3, hipStream_t s);
void launch_final(const Dev &d, double *sp, double *br, double *sa, double *dgbdr, double *dvwdr,
                  double *decav, double *dehb, double *energies, hipStream_t s);

}  // namespace agb
