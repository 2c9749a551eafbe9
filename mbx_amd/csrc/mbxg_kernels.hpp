// Kernel interfaces shared between the kernel translation units and the host runtime.
#pragma once

#include <hip/hip_runtime.h>

#include "mbxg_device.hpp"

namespace mbxg {

// Candidate grid of one configuration.  Cell of a position y (fractional coordinates under
// PBC, where the grid spans the slots' extended range [-1, 1]^3; Cartesian in the gas phase,
// over the bounding box): floor((y - lo) * inv_w) per dimension, clamped to [0, n).  Every cell
// is at least one cutoff wide, so a query's matches lie in the 27 cells around its own.
struct Grid {
    int n[3];
    int periodic;
    double lo[3];
    double inv_w[3];
};

// Per cloud point p (a monomer, or an image of one): its first atom in the working coordinates
// (not imaged) and its tag and kind, so the n-mer kernel reads a match's data with one load.
struct PtInfo {
    double x, y, z;
    int tag, kind;
};

// Everything an n-mer kernel needs to find a monomer's atoms.  Coordinates are the wrapped
// working copy (3 doubles per real atom, internal monomer order).  The box stays in device
// memory (read with scalar loads where needed) so it does not pin 48 SGPRs in the kernels.
struct NmerCtx {
    const double* xyz;
    const int* first_atom;
    const int* nat;
    const int* kind;
    const int* tag;
    const unsigned char* islocal;
    const int* members;  // cloud point -> monomer
    const Box* box;
    int periodic;
};

// Records the message returned by mbxg_last_error and returns code (api.hip).
int report_error(int code, const char* msg);

// Cell grids: at most kMaxCellsPerDim cells per dimension (the gas-phase grid is sized on the
// device; the cell buffers are allocated for the maximum).
constexpr int kMaxCellsPerDim = 64;
constexpr int kMaxCells = kMaxCellsPerDim * kMaxCellsPerDim * kMaxCellsPerDim;

__global__ void k_fix_monomers(const double* in, double* out, const int* first_atom, const int* nat, int nmon, Box B);
__global__ void k_grid_gas(const double* xyz, const int* first_atom, const int* members, const int* pt_off,
                           const int* cell_bound, double cut, Grid* grids);
__global__ void k_cloud(const double* xyz, const int* first_atom, const int* members, const int* tag, const int* kind,
                        int np, Box B, const Grid* grids, const int* pconf, const int* cell_base, double* cx,
                        double* cy, double* cz, int* cell, PtInfo* pinfo);
// cell_pos[s] receives slot s's place among its cell's slots (the count before its own).
__global__ void k_bin_count(const int* cell, int ns, int* cell_count, int* cell_pos);
// Up to four device ranges to zero in one launch (null pointers skipped).
struct ZeroJobs {
    double* p[4];
    size_t n[4];
};
// k_zero over every range of Z, grid-stride.
__global__ void k_zero_multi(ZeroJobs Z);
// k_fix_monomers, k_cloud and k_bin_count in one launch of max(nmon, 8 np) threads (eight per
// cloud point, one slot pattern each), which also zero the ranges of Z.
__global__ void k_cloud_fix(const double* in, double* xyz, const int* first_atom, const int* nat, int nmon,
                            const int* members, const int* tag, const int* kind, int np, Box B, const Grid* grids,
                            const int* pconf, const int* cell_base, double* cx, double* cy, double* cz, int* cell,
                            PtInfo* pinfo, int* cell_count, int* cell_pos, ZeroJobs Z);
__global__ void k_scan_cells(int* cell_count, int ncell, int* cell_start);
// The same over more than kCellsOneBlock cells: blocks of kCellChunk cells, sums[blocks] between them.
constexpr int kCellChunk = 4096, kCellsOneBlock = 8192;
__global__ void k_cell_sums(const int* cell_count, int ncell, int* sums);
__global__ void k_scan_cells_wide(int* cell_count, int ncell, const int* sums, int* cell_start);
__global__ void k_bin_fill(const int* cell, int ns, const int* cell_start, const int* cell_pos, const double* cx,
                           const double* cy, const double* cz, int* cell_slot, double* bx, double* by, double* bz);
__global__ void k_zero(double* p, size_t n);
__global__ void k_zero_int(int* p, size_t n);

// The n-mer kernel (lists.hip): one wavefront per query point; pass 0 counts, pass 1 writes.
// Points are grouped by configuration (pconf[p]); a configuration's cells start at
// cell_base[conf] and its grid is grids[conf], so lists never cross configurations.  Slots in
// cell order: cell_slot (slot index), bx/by/bz (coordinates), cell c holding
// [cell_start[c], cell_start[c+1]).
// Evaluated n-mer families (one evaluate list each): MB-pol 2B, MB-nrg CH4-H2O 2B, CH4-CH4 2B,
// MB-pol 3B, MB-nrg CH4-H2O-H2O 3B.
enum Family : int { FAM_MBPOL_2B = 0, FAM_CH4H2O_2B = 1, FAM_CH4CH4_2B = 2, FAM_MBPOL_3B = 3, FAM_CH4H2O2_3B = 4 };
constexpr int kFamilies = 5;
constexpr int family_order(int f) { return f < FAM_MBPOL_3B ? 2 : 3; }

// Wavefronts per query in the n-mer kernel; wpre / wpre_x hold each wavefront's prefix within
// its query (entry q * kQueryWaves + w), counts / offsets one entry per query.
constexpr int kQueryWaves = 4;

struct NmersArgs {
    const PtInfo* pinfo;
    const double* cx;
    const double* cy;
    const double* cz;
    const int* cell;
    const int* cell_start;
    const int* cell_slot;
    const double* bx;
    const double* by;
    const double* bz;
    const Grid* grids;
    const int* pconf;
    const int* cell_base;
    int np;
    double c2sq, c3sq;
    int4* counts;
    int4* counts_x;
    const int4* offsets;
    const int4* offsets_x;
    int4* wpre;
    int4* wpre_x;
    int* list2;
    int* list3;
    int* evals[kFamilies];
    int fam_mask;   // bit f: family f is evaluated (listed n-mers of a cleared family are not)
    // one-pass build (pass 2): wavefront w of query q stages its family-f n-mers at
    // stage[f] + (q * kQueryWaves + w) * scap[f] * order, at most scap[f] of them.  Every count
    // pass stores query q's largest per-wavefront counts in wmax[q] / wmax_x[q] (the layouts of
    // counts / counts_x; nullable)
    int* stage[kFamilies];
    int scap[kFamilies];
    int4* wmax;
    int4* wmax_x;
};

// One workgroup: the per-(query, wavefront) maxima of wmax / wmax_x into maxw[0..1] (skipped with wmax null) and
// the exclusive scans of counts and counts_x (.w maximised), totals at n, in one launch.
__global__ void k_scan_all(const int4* wmax, const int4* wmax_x, int4* maxw, const int4* counts, int4* offsets,
                           const int4* counts_x, int4* offsets_x, int n);
// The same over more than kScanOneBlock queries (the two launches take what one workgroup takes at 2048):
// blocks of kScanChunk queries, their shares between the launches.
constexpr int kScanChunk = 1024, kScanOneBlock = 2048;
struct ScanShare {
    int4 c, cx, m, mx;
};
__global__ void k_scan_shares(const int4* wmax, const int4* wmax_x, const int4* counts, const int4* counts_x, int n,
                              ScanShare* shares);
__global__ void k_scan_wide(const ScanShare* shares, const int4* counts, int4* offsets, const int4* counts_x,
                            int4* offsets_x, int4* maxw, int n);

// The staged n-mers of a one-pass build, moved to the evaluate lists: block q (striding),
// wavefront w copies its family-f n-mers to evals[f] at the family's offset of query q plus the
// wavefront's prefix, bounded by fcap[f] (the list capacity in n-mers) and scap[f].
// The per-family energy/virial records of one compute (null partials: family not evaluated).
struct FinishJobs {
    const double* partials[kFamilies];
    const int* n_dev[kFamilies];
    int cap[kFamilies];
};
// One workgroup of kFinishThreads: each family's partial records summed in a fixed order (zeros for the
// families not evaluated), then the per-order records of totals (2B = MB-pol + CH4-H2O + CH4-CH4, 3B =
// MB-pol + CH4-H2O-H2O) and the 4B record zeroed.  (The 1B record is a launch of its own before.)
// The last kernel of a compute also publishes what the host reads after every step (the totals and the
// list builder's counts and maxima) into pinned host memory, so that waiting for the stream is all the
// host does: three copies of a few bytes each cost 40 us a step.
struct Published {
    double totals[4 * kPartials];
    int4 tot, totx, maxw[2];
};
struct PublishJob {
    Published* host;
    const int4 *tot, *totx, *maxw;  // tot null: no lists were built
};
constexpr int kFinishThreads = 512;
__global__ void k_finish(FinishJobs J, double* totals, PublishJob P);

// By one workgroup, after its threads have written (and __syncthreads() has ordered) totals.
__device__ __forceinline__ void publish(const PublishJob& P, const double* totals) {
    const int t = threadIdx.x;
    if (t < 4 * kPartials) P.host->totals[t] = totals[t];
    const int4 zero = make_int4(0, 0, 0, 0);
    if (t == 0) P.host->tot = P.tot ? *P.tot : zero;
    if (t == 1) P.host->totx = P.tot ? *P.totx : zero;
    if (t < 2) P.host->maxw[t] = P.tot ? P.maxw[t] : zero;
}

struct CompactArgs {
    const int* stage[kFamilies];
    int scap[kFamilies];
    int* evals[kFamilies];
    int fcap[kFamilies];
};
__global__ void k_compact_evals(CompactArgs C, int np, const int4* counts, const int4* counts_x,
                                const int4* offsets, const int4* offsets_x, const int4* wpre, const int4* wpre_x);
// match_cap (a power of two) bounds the matches one query may hold.  With gscratch == nullptr
// they live in LDS (nmers_lds_bytes(match_cap) per block, one block per query); otherwise
// nblocks blocks stride over the queries, each with nmers_lds_bytes(match_cap) bytes of
// gscratch.
size_t nmers_lds_bytes(int match_cap);
hipError_t launch_nmers(const NmersArgs& A, const NmerCtx& N, int pass, int4 cap, int4 capx, int match_cap,
                        double* gscratch, int nblocks, hipStream_t st);

// Evaluation of the compacted "evaluate" lists (eval_mbpol2b.hip, eval_mbpol3b.hip): variable
// stage, polynomial stage (poly_mbpol2b.hip, poly_mbpol3b.hip), chain-rule stage.  One lane per
// n-mer.  The evaluated count n is read on the device from n_dev (clamped to cap): kernels are
// launched for cap n-mers and lanes past n retire at once, so the host never waits for the
// list builder.  e_out[t] receives n-mer t's energy and, when vir_out is not null,
// vir_out[q * ld + t] (q = xx xy xz yy yz zz, ld = cap rounded up to 64) its virial; partials
// one kPartials record per 64 n-mers (partials_records(cap) records); ws is a workspace of
// workspace_mbpolXb(cap) doubles.  ev (nullable) receives 4 events: before the variable stage, before the
// polynomial, before the chain-rule stage, after it.
inline size_t partials_records(int cap) { return ((size_t)cap + 127) / 128 * 2; }
size_t workspace_mbpol2b(int cap);
size_t workspace_mbpol3b(int cap);
hipError_t launch_mbpol2b(const int* list, const int* n_dev, int cap, const NmerCtx& N, const double* coef,
                          int do_grads, double* grad, double* e_out, double* vir_out, double* partials, double* ws,
                          int split, hipStream_t st, hipEvent_t* ev);
hipError_t launch_mbpol3b(const int* list, const int* n_dev, int cap, const NmerCtx& N, const double* coef,
                          int do_grads, double* grad, double* e_out, double* vir_out, double* partials, double* ws,
                          int split, hipStream_t st, hipEvent_t* ev);
// The variable and chain-rule stages alone (same workspace layout), and both MB-pol polynomial
// stages with gradients in one launch (poly_mbpol_pair.hip): the 3B blocks first, then the 2B
// ones, `split` wavefronts per 64 n-mers for both, so the short 2B blocks fill the machine while
// the last 3B blocks drain.
hipError_t launch_mbpol2b_vars(const int* list, const int* n_dev, int cap, const NmerCtx& N, double* ws,
                               hipStream_t st);
hipError_t launch_mbpol3b_vars(const int* list, const int* n_dev, int cap, const NmerCtx& N, double* ws,
                               hipStream_t st);
hipError_t launch_mbpol2b_chain(const int* list, const int* n_dev, int cap, const NmerCtx& N, int do_grads,
                                double* grad, double* e_out, double* vir_out, double* partials, double* ws,
                                hipStream_t st);
hipError_t launch_mbpol3b_chain(const int* list, const int* n_dev, int cap, const NmerCtx& N, int do_grads,
                                double* grad, double* e_out, double* vir_out, double* partials, double* ws,
                                hipStream_t st);
// 1B terms (eval_1b.hip): energies e_out[t] of monomers mons[0..n), and with g_out the gradient
// components of each (3 doubles per atom, written at its atoms) and vir_out[q * ld + t] (q = xx xy
// xz yy yz zz).  Water: MB-pol (Partridge-Schwenke); CH4: MB-nrg A1B4 with coefficients coef
// (ch4_1b_fit: the fitted ones).  k_reduce_1b sums n energies and virial rows into out[kPartials].
hipError_t launch_1b_ps(const double* xyz, const int* first_atom, const int* mons, int n, double* e_out,
                        double* g_out, double* vir_out, int ld, hipStream_t st);
hipError_t launch_1b_ch4(const double* xyz, const int* first_atom, const int* mons, int n, const double* coef,
                         double* e_out, double* g_out, double* vir_out, int ld, hipStream_t st);
const double* ch4_1b_fit(int* n);
// CO2 monomers (x1b_A1B2_v1x): the same outputs; co2_1b_fit: the fitted coefficients.
hipError_t launch_1b_co2(const double* xyz, const int* first_atom, const int* mons, int n, const double* coef,
                         double* e_out, double* g_out, double* vir_out, int ld, hipStream_t st);
const double* co2_1b_fit(int* n);
__global__ void k_reduce_1b(const double* e, const double* vir, int n, int ld, double* out);
hipError_t launch_poly_mbpol_pair(double* ws3, const int* n3_dev, int cap3, const double* coef3, double* ws2,
                                  const int* n2_dev, int cap2, const double* coef2, int split, hipStream_t st);
// launch_mbpol3b_vars and launch_mbpol2b_vars as one launch (workspaces as theirs).
hipError_t launch_mbpol_vars_pair(const int* list3, const int* n3_dev, int cap3, double* ws3, const int* list2,
                                  const int* n2_dev, int cap2, double* ws2, const NmerCtx& N, hipStream_t st);
// Both orders' whole evaluation with gradients in one launch (mbpol_fused.hip): energies e_out, gradient
// added to grad, virials vir_out (nullable, leading dimension ld), one partial record per 64 n-mers.  cap 0:
// that order is left out (n_dev is not read).
constexpr int kFusedSplit = 4;  // wavefronts per 64 n-mers
struct FusedJob {
    const int* list;
    const int* n_dev;
    int cap, ld;
    uint64_t coef_addr;
    double *grad, *e_out, *vir_out, *partials;
};
hipError_t launch_mbpol_fused(const FusedJob& trimers, const FusedJob& dimers, const NmerCtx& N, hipStream_t st);
// MB-nrg families (eval_nrg.hip): the same three stages for FAM_CH4H2O_2B, FAM_CH4CH4_2B and
// FAM_CH4H2O2_3B; list entries in emission order (the kernels order each n-mer's monomers
// for its holder).  `split` (1, 2, 4 or 8) is the wavefronts per 64 n-mers of the CH4-H2O-H2O
// polynomial; the 2B polynomials take poly_split's.
size_t workspace_nrg_family(int family, int cap);
hipError_t launch_nrg_family(int family, const int* list, const int* n_dev, int cap, const NmerCtx& N,
                             const double* coef, int do_grads, double* grad, double* e_out, double* vir_out,
                             double* partials, double* ws, int split, hipStream_t st, hipEvent_t* ev);

// Wavefronts per 64 n-mers for a polynomial kernel of `wpe` wavefronts per SIMD, from the n-mers'
// capacity.  Few groups of 64 leave the chip idle, so each is cut into more and shorter wavefronts; the
// cut costs a reduction and variables loaded again, so it stops once the chip is full.  Measured on
// MB-pol's polynomials as launches of their own (wpe 3; us at split 1 / 2 / 4 / 8).  3B, value and gradient: 72
// groups 66 / 41 / 26 / 25, 261 70 / 44 / 35 / 46, 1065 102 / 79 / 69 / 104, 2352 144 / 118 / 119 / 194, 3987
// 196 / 178 / 183 / 306, 11269 490 / 477 / 494 / 872; values alone: 72 46 / 28 / 18 / 14, 1065 65 / 44 / 40 / 39,
// 2352 84 / 75 / 65 / 69, 7286 181 / 162 / 162 / 180.  2B, value and gradient: 78 27 / 19 / 14 / 13, 518
// 37 / 28 / 24 / 34, 1711 49 / 46 / 43 / 68, 2657 63 / 61 / 60 / 102.
// poly_wpe: wavefronts per SIMD of a value + gradient kernel of nv variables (the generator's rule).
constexpr int poly_wpe(int nv) { return 512 / (4 * nv + 24) > 4 ? 4 : 512 / (4 * nv + 24) > 1 ? 512 / (4 * nv + 24) : 1; }
inline int poly_split(int cap, int wpe) {
    const int groups = (cap + 63) / 64;
    return groups <= 128 ? 8 : groups <= 800 * wpe ? 4 : 2;
}

// Polynomial stage alone: xs/gs variable-major with leading dimension ld (= cap rounded up
// to 64); ps values; n read from n_dev as above; `split` wavefronts (1, 2, 4 or 8) share each
// 64 n-mers (poly_kernel.hpp).
hipError_t launch_poly_mbpol2b(const double* xs, const int* n_dev, int cap, int ld, const double* coef, int do_grads,
                               double* gs, double* ps, int split, hipStream_t st);
hipError_t launch_poly_mbpol3b(const double* xs, const int* n_dev, int cap, int ld, const double* coef, int do_grads,
                               double* gs, double* ps, int split, hipStream_t st);
hipError_t launch_poly_ch4h2o2_3b(const double* xs, const int* n_dev, int cap, int ld, const double* coef,
                                  int do_grads, double* gs, double* ps, int split, hipStream_t st);

// Per-configuration totals in two fixed-order levels, all families in one launch each: block (c, s, f) of
// a (nconf, S, kFamilies) grid sums slice s of configuration c's evaluated n-mers of family f (null e_out:
// not evaluated), [offsets[pt_off[c]].comp, offsets[pt_off[c+1]].comp) clamped to cap, from e_out / vir_out
// (leading dimension cap rounded up to 64; zeros when vir_out is null) into part[f][c][s][kPartials]; comp
// selects the int4 component (0..3) holding the family's count.  k_reduce_slices adds the slices of the
// families of each order: out[2][nconf][kPartials].  k_sum_configs adds the configurations into the 2B and
// 3B records of totals, zeroes the 4B one and publishes.
struct ConfigJobs {
    const double* e_out[kFamilies];
    const double* vir_out[kFamilies];
    const int4* offsets[kFamilies];
    int comp[kFamilies], cap[kFamilies];
};
__global__ void k_reduce_configs(ConfigJobs J, const int* pt_off, double* part);
__global__ void k_reduce_slices(ConfigJobs J, const double* part, int nconf, int nsl, double* out);
__global__ void k_sum_configs(const double* conf, int nconf, double* totals, PublishJob P);

}  // namespace mbxg
