/* Additive extensions of libagbnp3 (no counterpart in the reference API;
 * the reference entry points in agbnp3.h are unchanged).
 *
 * All functions return AGBNP_OK / AGBNP_ERR like the reference API and print
 * the reason on stderr.  Device pointers are plain hipMalloc'd addresses;
 * `stream` arguments are hipStream_t values passed as void*.
 */
#ifndef AGBNP3_AMD_H
#define AGBNP3_AMD_H
#include "agbnp3.h"
#ifdef __cplusplus
extern "C" {
#endif

/* ---- options (per instance; default 0 = reference behaviour) ---------- */
/* E_HB free volume subtracts spe of the current overlap partner instead of
   the reference's stale one (agbnp3_cpu_simd_kernels.c:2854, 2859) */
#define AGBNP3_OPT_HB_FIXED      1
/* spline derivative with the textbook sign of the y''(k+1) term instead of
   the reference's (agbnp3_utils.c:292-293, agbnp3_cpu_simd_kernels.c:964-965) */
#define AGBNP3_OPT_SPLINE_FIXED  2
/* record per-kernel HIP event times of every call (agbnp3_kernel_times) */
#define AGBNP3_OPT_TIMING        4
int agbnp3_set_options(int tag, int options);

/* ---- device-resident evaluation ---------------------------------------- */
/* Same computation as agbnp3_ener with every array in device memory (caller
   atom order): x, y, z [natoms]; sp, br, surf_area [natoms]; the four
   gradients [3*natoms], interleaved like float_i (*)[3]; energies[7] =
   egb, evdw, ecorr_vdw, ecav, ecorr_cav, ehb, mol_volume.  Enqueued on the
   instance stream and returns without waiting; call agbnp3_sync (or wait on
   agbnp3_stream) before reading outputs.  (From 512 atoms some of the
   kernels run on a second stream of the instance, joined into the instance
   stream before the call's last kernel: waiting on the instance stream
   covers them.)  Host-side errors (bad tag, HB
   topology) are reported immediately; device-side capacity errors by the
   next agbnp3_sync. */
int agbnp3_ener_device(int tag, const double *x, const double *y, const double *z,
                       double *sp, double *br, double *surf_area,
                       double *dgbdr, double *dvwdr, double *decav, double *dehb,
                       double *energies);
int agbnp3_sync(int tag);
void *agbnp3_stream(int tag);

/* ---- evaluation that allocates nothing ----------------------------------- */
/* No counterpart in the reference API.  For callers that cannot allocate
   device memory (code under hipGraph capture, tight serving loops, harnesses
   that forbid hipMalloc): the computation, arguments, stream and status of
   agbnp3_ener_device, with the call's working state (coordinates, cell
   grids, neighbour list, accumulators, per-atom factors, water sites) in a
   static device array of AGBNP3_STATIC_SCRATCH_BYTES per device instead of
   the instance's own.  The instance's per-call state is never allocated by
   this entry point (agbnp3_new allocates only parameters, tables, work items
   and a status word).  The working state grows with the number of
   chain-rule block pairs, so faster than the atom count: 15,000 atoms of a
   protein-like solute take 34 MiB, 20,000 take 54 MiB, 25,000 take 76 MiB,
   and the 96 MiB array holds such solutes up to about 28,000 atoms.  Instances whose working state does not fit
   and instances with a surrogate attached are rejected with AGBNP_ERR, and
   the message states the bytes the instance needs.  Every call on a device shares that device's array, which
   keeps the last call's contents: calls that overlap on one device (two
   instance streams, or two host threads) race; order them (agbnp3_sync, or
   one stream).  Results equal agbnp3_ener_device's bitwise. */
#define AGBNP3_STATIC_SCRATCH_BYTES (96u << 20)
int agbnp3_ener_static(int tag, const double *x, const double *y, const double *z,
                       double *sp, double *br, double *surf_area,
                       double *dgbdr, double *dvwdr, double *decav, double *dehb,
                       double *energies);

/* ---- neighbour-list reuse across calls ---------------------------------- */
/* The reference rebuilds the heavy-atom neighbour list on every call
   (agbnp3.c:3978-4115).  With skin > 0 (Angstrom, at most 4) a rebuild also
   keeps every pair within the cutoff plus `skin`; later calls re-test and
   re-sort only those candidates, which gives the identical list while no
   heavy atom has moved more than skin/2 since the rebuild.  A device-side
   guard checks that on every call and rebuilds when it fails; `every` > 0
   also forces a rebuild every `every` calls.  skin = 0 restores a rebuild on
   every call.  Results are bitwise those of the full rebuild. */
int agbnp3_set_nblist_reuse(int tag, float skin, int every);
/* calls and candidate rebuilds since the last agbnp3_set_nblist_reuse */
int agbnp3_nblist_rebuilds(int tag, int *calls, int *rebuilds);
int agbnp3_batch_set_nblist_reuse(int batch, float skin, int every);

/* ---- launch shapes and autotuner ----------------------------------------- */
/* params[8]: rows per descreening block (64, 128, 256); columns per
   descreening item (multiple of 256, 0 = automatic); columns per chain-rule
   item (64, 128 or 256 of a 256-atom block, 0 = 256); persistent grid of the
   descreening, GB-pair and chain-rule kernels (blocks, 0 = one per work
   item); neighbour-list row capacity (64, 128, 256); persistent grid of the
   first overlap-tree tier (blocks, 0 = one per heavy atom).  No counterpart in the
   reference. */
#define AGBNP3_TUNING_PARAMS 8
int agbnp3_get_tuning(int tag, int *params, int nparams);
int agbnp3_set_tuning(int tag, const int *params, int nparams);
/* times the pipeline on device coordinates x, y, z (caller order) for each
   candidate shape, `reps` timed calls per trial, keeps the fastest per
   kernel; a text report of the trials goes to `report` (may be NULL) */
int agbnp3_tune(int tag, const double *x, const double *y, const double *z, int reps, char *report,
                int report_len);
/* The shapes a tuning run chooses are recorded per size class (number of
   systems in octaves, total atoms in half octaves); instances and batches
   built later in a recorded class start from them.  The table persists
   through a text file: save writes every recorded class, load adds the
   file's classes (AGBNP_ERR on a malformed line, nothing loaded), clear
   empties it. */
int agbnp3_tune_table_save(const char *path);
int agbnp3_tune_table_load(const char *path);
int agbnp3_tune_table_clear(void);

/* ---- batches: many instances in one set of launches ---------------------- */
/* A batch packs existing instances (same options) into one device arena;
   every kernel of a call covers all of them, with per-system work items
   taken from work queues by persistent blocks.  The batch copies what it
   needs: the instances stay independent and may be deleted.  Arrays are the
   per-instance caller-order arrays concatenated in `tags` order (offsets
   from agbnp3_batch_offsets); energies are [ntags][7] as in
   agbnp3_ener_device. */
int agbnp3_batch_new(int *batch, int ntags, const int *tags);
int agbnp3_batch_delete(int batch);
/* nsys = ntags; offsets[ntags + 1]: first atom of each instance, total */
int agbnp3_batch_offsets(int batch, int *nsys, int *offsets);
int agbnp3_batch_set_options(int batch, int options);
int agbnp3_batch_ener_device(int batch, const double *x, const double *y, const double *z, double *sp,
                             double *br, double *surf_area, double *dgbdr, double *dvwdr, double *decav,
                             double *dehb, double *energies);
/* host arrays; out = sp, br, surf_area [n] each, dgbdr, dvwdr, decav, dehb
   [3n] each, energies [ntags][7] (15 n + 7 ntags doubles) */
int agbnp3_batch_ener(int batch, const double *x, const double *y, const double *z, double *out);
int agbnp3_batch_sync(int batch);
void *agbnp3_batch_stream(int batch);
/* capture one agbnp3_batch_ener_device call on these device buffers as a
   hipGraph; agbnp3_batch_graph_launch replays it on the batch stream (the
   caller rewrites x, y, z between replays).  A change of launch shape or
   options drops the graph. */
int agbnp3_batch_graph_capture(int batch, const double *x, const double *y, const double *z, double *sp,
                               double *br, double *surf_area, double *dgbdr, double *dvwdr, double *decav,
                               double *dehb, double *energies);
int agbnp3_batch_graph_launch(int batch);
int agbnp3_batch_kernel_times(int batch, float *ms, int nmax, char *names, int names_len);
int agbnp3_batch_get_tuning(int batch, int *params, int nparams);
int agbnp3_batch_set_tuning(int batch, const int *params, int nparams);
int agbnp3_batch_tune(int batch, const double *x, const double *y, const double *z, int reps, char *report,
                      int report_len);

/* ---- learned Born-radius surrogate --------------------------------------- */
/* A per-atom MLP (66 -> 128 -> 128 -> 128 -> 1, SiLU, bf16 on the matrix
   cores with FP32 accumulation) on local descriptors (4 heavy-atom channels
   x 16 radial shells to 12 A, R, q) predicts the descreening sum of the
   inverse Born radius.  Attached to an instance or batch with anchor period
   `every`, a system runs the plain kernels on its first call and every
   `every` calls ("anchor" calls); in between its descreening sum is the
   model's plus the correction the last anchor measured, with the model's
   gradient in place of the descreening chain rule.  Atoms whose descriptors
   leave the training window take the plain descreening and chain rule on
   such a call (the whole call is an anchor when they are more than one per
   2048 atoms).  On each anchor the first-order error of the
   solvation energy the surrogate would have made is recorded
   (agbnp3_*sg_stats).  No counterpart in the reference. */
int agbnp3_sg_new(int *model, unsigned long long seed);
int agbnp3_sg_delete(int model);
/* flat export: parameters, feature normalisation and window, target scale */
int agbnp3_sg_size(void);
int agbnp3_sg_get_params(int model, float *out, int n);
int agbnp3_sg_set_params(int model, const float *in, int n);
/* training set: descriptors and plain descreening sums of every atom of a
   batch evaluated (plain) at device coordinates x, y, z */
int agbnp3_sg_reserve(int model, int natoms);
int agbnp3_batch_sg_collect(int batch, int model, const double *x, const double *y, const double *z);
/* count, raw descriptors [count][66] and targets [count] (may be NULL) */
int agbnp3_sg_dataset(int model, int *count, float *F, float *target);
/* normalisation, training window (range widened by `margin` of its width
   plus half an atom per shell, 0.02 A of radius, 0.1 e of charge), and the
   training rows: pairs of rows of one atom of one batch collected at two
   coordinate sets (an atom collected once pairs with itself), in a shuffled
   pair order, rows 2k and 2k+1 a pair; without any such pair, the rows in a
   shuffled order */
int agbnp3_sg_fit(int model, float margin, unsigned long long seed);
/* loss per training row w_abs e^2 + w_diff c (e - e_pair)^2, e the error of
   the normalised output and c = 1 / (mean squared normalised difference of
   the pairs' targets); default w_abs = w_diff = 1 */
int agbnp3_sg_set_loss(int model, float w_abs, float w_diff);
/* training rows: count, dataset row of each (may be NULL), and c */
int agbnp3_sg_train_rows(int model, int *count, int *rows, float *diff_scale);
/* Adam, mini-batches of B rows (B even), lr decay^epoch; mean loss per epoch */
int agbnp3_sg_train(int model, int epochs, int B, float lr, float decay, unsigned long long seed,
                    float *epoch_loss);
/* gradients of the loss over training rows [r0, r0 + B), r0 even (no update) */
int agbnp3_sg_grads(int model, int r0, int B, float *grad, float *loss);
/* the model on raw descriptors F [n][66]: s [n], ds/dF [n][64] */
int agbnp3_sg_infer(int model, const float *F, int n, float *s, float *dsdF);
int agbnp3_sg_attach(int tag, int model, int every);
int agbnp3_batch_sg_attach(int batch, int model, int every);
/* per system: error estimate of the last audited anchor, mode of the last call
   (0 = plain/anchor, 1 = surrogate, 2 = surrogate with the plain descreening
   and chain rule for the few atoms whose descriptors left the training
   window: at most one per 2048 atoms of the system, else the call is plain) */
int agbnp3_sg_stats(int tag, double *err, int *mode);
int agbnp3_batch_sg_stats(int batch, double *err, int *mode);
/* per system: calls in mode 0, 1 and 2 (three ints per system) since the
   model was attached */
int agbnp3_sg_modes(int tag, int *counts);
int agbnp3_batch_sg_modes(int batch, int *counts);
/* per system: builds of the descriptor neighbour lists (pairs within 13.5 A,
   rebuilt after a move beyond 0.75 A) since a model was first attached, and
   1 if an atom had more than 1536 neighbours (the system then stays on the
   plain kernels) */
int agbnp3_sg_lists(int tag, int *builds, int *overflow);
int agbnp3_batch_sg_lists(int batch, int *builds, int *overflow);

/* ---- host-only helpers (no GPU needed) ------------------------------------ */
/* Q4 spline tables for radius types `radii` (R = r + 0.5): y, y2 sized
   ntypes*ntypes*512, table (i, j) at offset (i*ntypes + j)*512; dx[0..1] =
   node spacing and its inverse.  The same tables agbnp3_new builds. */
int agbnp3_q4_tables(int ntypes, const float *radii, float *y, float *y2, float *dx);

/* ---- introspection of the last evaluation (tests, profiling) ----------- */
int agbnp3_natoms(int tag, int *natoms, int *nheavy);
/* internal (heavy-first) order: int2ext[natoms] */
int agbnp3_get_int2ext(int tag, int *int2ext);
/* heavy-atom neighbour list: nne[nheavy], rows padded to `cap` */
int agbnp3_get_near_list(int tag, int *nne, int *nbr, int cap);
/* Q4 spline tables: returns ntypes; y, y2 [ntypes*ntypes*512], radii[ntypes]
   (any may be NULL) */
int agbnp3_get_tables(int tag, float *y, float *y2, float *radii);
/* per-atom internal array, internal order, natoms doubles: "volumep_raw",
   "sa_raw", "sa_f", "sp", "spe", "psvol", "gammap", "beta", "br", "brw",
   "swf", "A", "q2ab", "abrw", "deru", "derv", "derus", "dervs", "derh" */
int agbnp3_get_internal(int tag, const char *name, double *out);
/* counts[0] kept overlaps, [1] evaluated overlaps, [2] water sites,
   [3] neighbour-list entries, [4] max row length, [5] [6] overlap-tree roots
   that outgrew the breadth-first level buffers (volumes, derivatives) */
int agbnp3_get_counts(int tag, long long *counts);
/* which of the kernels that a rule on sizes chooses between the last call took
   (in agbnp3_ener_*, not a graph's replay): the sum of
   1 descreening by tiles, 2 with 64 rows per block of those, 4 descreening
   that passes over far columns, 8 GB pairs by chunks, 16 chain rule by row
   groups, 32 chain rule with its lookups in groups, 64 chain rule that passes over far
   columns; 0 before the first call */
int agbnp3_get_routes(int tag, int *routes);
/* per-kernel times (ms), averaged over the calls made since the previous
   read while AGBNP3_OPT_TIMING was set (HIP events on the instance stream);
   returns the number of kernels written; names joined by ';' */
int agbnp3_kernel_times(int tag, float *ms, int nmax, char *names, int names_len);

#ifdef __cplusplus
}
#endif
#endif
