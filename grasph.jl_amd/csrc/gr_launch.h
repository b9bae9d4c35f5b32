// gr_launch.h — host-callable launchers of the device kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "gr_device.h"

namespace gr {

struct SweepArgs {
  const SysDesc *sd;
  const int *n;
  const Task *tasks;
  const SrcDesc *srcs;
  const Grid *grids;
  const CellArr *carr;
  const int *cells;
  const Blk *blk;
  int nblk;
  unsigned long long *pair_count;
  const LTask *lt = nullptr;  // non-null: use the neighbour lists
  const int *lcnt = nullptr;
  const int *lidx = nullptr;
  bool fluid_only = false;  // FORCE: every source's functor is FluidPfn / FluidSolidPfn
  int block = GR_BLOCK;     // targets per workgroup (the block table's step)
  bool inv = false;         // FP32 FluidPfn S = 2 stage whose records hold 1/ρ, p/ρ²
};

struct NlistArgs {
  const SysDesc *sd;
  const int *n;
  const LTask *lt;
  const SrcDesc *srcs;
  const Grid *grids;
  const CellArr *carr;
  const int *cells;
  const Blk *blk;
  int nblk;
  int *lcnt;
  int *lidx;
  const long long *bbmin = nullptr;  // per-system position bounds of this step
  const long long *bbmax = nullptr;  // (ordered int64, see ord_of)
  int win = 128;  // candidates staged in LDS per window (64, 128 or 256)
  int span = 2;   // lanes whose ranges start within span·(widest range) group
};

// Position bounds per system and dimension: replicas 1 .. GR_BB_REP of `rs`
// entries each take the bounds pass's atomics, replica 0 holds the folded
// bounds that every reader uses.  launch_key_minmax folds them itself when
// `fold`, launch_key_base and launch_key_sort always do.
#define GR_BB_REP 8
struct StepBounds {  // where the end of a step takes the bounds of the next
  const int *n_dev;
  long long *bbmin, *bbmax;
  int rs;
  int *flags;  // [0] is cleared
};
void launch_key_minmax(hipStream_t s, XP xs, const SysDesc *sd, const int *n, const Blk *blk,
                       int nblk, int D, long long *bbmin, long long *bbmax, int rs,
                       const int *list, int nlist, bool fold, int *flags = nullptr);
void launch_minmax_reset(hipStream_t s, const int *list, int nlist, long long *bbmin,
                         long long *bbmax, int rs);
void launch_key_base(hipStream_t s, const int *list, int nlist, int D, int pad, const int *n,
                     const StepSys *st, long long *bbmin, long long *bbmax, int rs, int *kmin,
                     int *kmax, unsigned *kbase, unsigned *krange, int *flags, int *sysfault);
void launch_key_write(hipStream_t s, XP xs, const SysDesc *sd, const int *n,
                      const StepSys *st, const Blk *blk, int nblk, const int *bbase, int D,
                      const int *kmin, const unsigned *krange, const unsigned *kbase,
                      unsigned *keys, int *vals, int *flags, unsigned *rscr);
// Stable radix sort of (keys, vals) by key, N entries.  `rscr` is the sort's
// scratch (radix_scratch_bytes(N), zeroed when allocated and left zeroed by
// every sort); launch_key_write counts the first pass into it and must run
// before it with the same scratch.  The sorted values end in vals when
// flags[3] is even and in vals2 when it is odd; the permutations take both.
// flags[1] bit 16: the counts did not place every key (not expected).
void launch_radix_sort(hipStream_t s, unsigned *keys, int *vals, unsigned *keys2, int *vals2,
                       unsigned *rscr, int N, int *flags);
size_t radix_scratch_bytes(int N);
// Interactions whose grids a step finds (from the bounds in replica 0) and the
// cell arrays it builds: cblk lists them 4·GR_BLOCK cells at a time, tflag holds
// a flag per that many cells of the pool (cell_tiles).
struct CellsArgs {
  int *cells, *tflag;
  const CellArr *carr;
  const Blk *cblk;
  int ncblk;
  const int *inter_list;
  int n_inter;
  const int2 *inter_sys;  // systems a and b (or -1) of an interaction
  const int2 *inter_carr;
  const double *cellsz;
  const long long *bbmin, *bbmax;
  const int *n_dev;
  Grid *grids;
  int D;
};
// The counting sort of a step (keys, table, placement) after the bounds pass:
// `table` of key_table_bytes(tiles) bytes, zeroed when allocated, of which this
// sort uses ntile <= tiles tiles: the listed systems' budgets of entries
// (key_budget) come to less than ntile·key_table_tile().  (The layout goes by
// `tiles`, as sorts of different sizes share the table.)  flags[0] must be clear;
// the permutations take the order by a KeyTable.  Replicas 1.. of the listed
// systems' bounds are reset, and `cells` prepared (as launch_cells_prep does).
size_t key_table_bytes(int64_t ntile);
int key_table_tile();
void launch_key_sort(hipStream_t s, XP xs, const SysDesc *sd, const int *n, const StepSys *st,
                     const Blk *blk, int nblk, const int *bbase, int D, const int *list, int nlist,
                     int N, long long *bbmin, long long *bbmax, int rs, int *kmin, int *kmax,
                     unsigned *krange, unsigned *kbase, int *kshift, unsigned *keys,
                     unsigned *full, unsigned *keys2, int *vals2, unsigned *rank,
                     int *flags, int *sysfault, int *run, unsigned *table, int tiles, int ntile,
                     const CellsArgs *cells = nullptr);
struct KeyTable {  // what the permutations read of the counting sort
  const unsigned *keys2, *start, *krange, *kbase;
  const int *kshift;     // log2 of a system's keys to an entry
  const unsigned *full;  // a particle's key in its system, where those are several
  const int *run;        // at the first slot of a run: its length (large cells)
};
template <typename R>
void launch_permute_real(hipStream_t s, const Pool<R> &A, const Pool<R> &B, const SysDesc *sd,
                         const Blk *blk, int nblk, const int *bbase, const int *vals,
                         const int *vals2, const int *flags, int vadj, int D,
                         const StepSys *st = nullptr, const int *halfsys = nullptr,
                         int pack = 0, const KeyTable *kt = nullptr);
// ghost generation: per-(boundary, source block) counts at gslot[g] + ...,
// then the scatter at the counts' exclusive scan (`scan` null: each workgroup
// adds up the counts itself); bbmin/bbmax: also the ghosts' bounds; flags: also
// clear the sort's flags
void launch_ghost_count(hipStream_t s, XP x, const SysDesc *sd, const Bnd *bnd,
                        const Blk *blk, int nblk, const int *gslot, int D, int *cnt,
                        int *flags = nullptr);
void launch_scan(hipStream_t s, const int *in, int *out, int *bsum, int N);
int scan_block_count(int N);
void launch_ghost_scatter(hipStream_t s, XP x, XPW gx, int *gidx,
                          int *gbnd, int *gnrm, const SysDesc *sd, const Bnd *bnd, const Blk *blk,
                          int nblk, const int *gslot, const int *cnt, const int *scan, int D,
                          int *n, long long *bbmin = nullptr, long long *bbmax = nullptr,
                          int rs = 0);
void launch_permute_ghost(hipStream_t s, XP gxs, const int *gidx_s,
                          const int *gbnd_s, XPW x, int *gidx, int *gbnd,
                          const SysDesc *sd, const int *n, const Blk *blk, int nblk,
                          const int *bbase, const int *vals, const int *vals2, const int *flags,
                          int D, const KeyTable *kt = nullptr);
template <typename R>
void launch_ghost_kin(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const Bnd *bnd,
                      const int *n, const Blk *blk, int nblk, int D);
template <typename R>
void launch_ghost_copy(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const Bnd *bnd,
                       const int *n, const Blk *blk, int nblk, const int2 *copy, int D);
int64_t cell_tiles(int64_t cells);
// The grids, and the arrays cleared: once the bounds are there.
void launch_cells_prep(hipStream_t s, const CellsArgs &A, int *flags, int *sysfault);
// The arrays, after that.
void launch_cells_build(hipStream_t s, XP x, const CellsArgs &A, const SysDesc *sd, const Blk *mblk,
                        int nmblk);
template <typename R>
void launch_halfstep(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                     const Blk *blk, int nblk, int D, double mult, int keep);
template <typename R>
void launch_rk4_acc(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                    const Blk *blk, int nblk, int D, double w, int first);
template <typename R>
void launch_rk4_apply(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                      const Blk *blk, int nblk, int D, int pos,
                     const StepBounds *bb = nullptr);
template <typename R>
void launch_fullstep(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                     const Blk *blk, int nblk, int D, int pos,
                     const StepBounds *bb = nullptr);
template <typename R>
void launch_xsph(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                 const int *n, const Blk *blk, int nblk, int D, int mode);
template <typename R>
// kinds: the set of updater kinds (bit GR_UPD_x) in ud; rec: the partner
// records written of every particle of blk after its updates, -1: none
void launch_updaters(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                     const Blk *blk, int nblk, const int2 *urange, const UpdDesc *ud, int D,
                     int kinds, int rec = -1);
template <typename R>
void launch_sweep(hipStream_t s, const Pool<R> &P, const SweepArgs &a, int D, int fam, bool cnt);
template <typename R>
void launch_virtual(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                    const int *n, const Blk *blk, int nblk, int mode, int D);
// Which partner records are written (FP64 pools: always RecA and RecB alone).
enum {
  GR_REC_C = 1,       // the compact records alone
  GR_REC_S = 2,       // the stress records
  GR_REC_INV = 4,     // compact records of 1/ρ and p/ρ²
  GR_REC_S_ONLY = 8,  // the stress records alone (the compact ones still hold)
};
// Records `mode` of the particles of blk, `gmode` of the ghosts of gblk; the
// latter after the kinematics (kin) and the copies of a stage (copy) if asked.
template <typename R>
void launch_pack(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const int *n, const Blk *blk,
                 int nblk, int mode, const Blk *gblk, int ngblk, int gmode, const Bnd *bnd,
                 const int2 *copy, bool kin, int D);
template <typename R>
void launch_nlist(hipStream_t s, const Pool<R> &P, const NlistArgs &a, int D);
// A field's arrays on the device (component k at k·cap): the field itself, and
// on the way in the shadows that follow it.
struct FieldSets {
  void *p[3];
  int esz[3];  // 8: double, 4: float
  int n;
};
// `count` elements between pinned host memory and the particles from `off` on
// (W: double, or float for a field held in 4 bytes).
template <typename W>
void launch_field(hipStream_t s, bool in, W *host, int64_t count, int nc, int64_t cap, int64_t off,
                  const FieldSets &F);
void launch_index(hipStream_t s, bool in, int *host, int64_t count, int *dev);
void launch_fill_i32(hipStream_t s, int *p, int v, long long n);
void launch_alias_check(hipStream_t s, const int *n, int ghost, int src_n, int *flags);
template <typename R>
void launch_probe_mirror(hipStream_t s, const Pool<R> &P, const SysDesc *sd, int probe, int src,
                         int64_t n_src, int D);
template <typename R>
void launch_probe_by_id(hipStream_t s, const Pool<R> &P, const SysDesc *sd, int probe, int64_t n,
                        double *scr, int mode, int D);

}  // namespace gr
