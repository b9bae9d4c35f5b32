// gr_kernels.hip — per-particle, sort, ghost and grid kernels for gfx950.
//
// Integer-deciding floating point (cell keys, CSR cells, ghost qualification,
// positions) is evaluated in FP64 in the order the reference writes it; the
// library is compiled with -ffp-contract=off so nothing is fused unless an
// explicit fma() is written (the reference's @fastmath scalar axpy).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/grasph_hip.h"
#include "gr_device.h"
#include "gr_launch.h"

namespace gr {

// ---------------------------------------------------------------------------
// Wave / block reductions (64-lane wavefronts)
// ---------------------------------------------------------------------------

// 64-bit wave-wide minimum / maximum (all 64 lanes active): DPP exchanges
// within each row of 16 lanes, then the four row results through readlane.
template <int CTRL>
__device__ __forceinline__ long long dpp_ll(long long v) {
  const int lo = __builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(v >> 32), (int)(v >> 32), CTRL, 0xF, 0xF, false);
  return (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ long long readlane_ll(long long v, int l) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)v, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), l);
  return (long long)(((unsigned long long)hi << 32) | lo);
}
template <bool MAX>
__device__ inline long long wave_red_ll(long long v) {
  auto op = [](long long x, long long y) { return MAX ? (x > y ? x : y) : (x < y ? x : y); };
  v = op(v, dpp_ll<0xB1>(v));   // quad_perm 1,0,3,2
  v = op(v, dpp_ll<0x4E>(v));   // quad_perm 2,3,0,1
  v = op(v, dpp_ll<0x141>(v));  // row_half_mirror
  v = op(v, dpp_ll<0x140>(v));  // row_mirror
  return op(op(readlane_ll(v, 0), readlane_ll(v, 16)), op(readlane_ll(v, 32), readlane_ll(v, 48)));
}
__device__ inline int wave_min_i(int v) {
  for (int o = 32; o > 0; o >>= 1) {
    int u = __shfl_xor(v, o, 64);
    v = u < v ? u : v;
  }
  return v;
}
__device__ inline int wave_max_i(int v) {
  for (int o = 32; o > 0; o >>= 1) {
    int u = __shfl_xor(v, o, 64);
    v = u > v ? u : v;
  }
  return v;
}

__device__ inline long long ord_d(double d) {
  long long i = __double_as_longlong(d);
  return i < 0 ? (i ^ 0x7FFFFFFFFFFFFFFFLL) : i;
}

// Coherent (device-scope, relaxed) read of a value other workgroups update
// with atomics.  Used to skip atomics that cannot change the value: a stale
// read only costs an atomic that turns out to be redundant.
template <typename T>
__device__ __forceinline__ T ld_dev(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// floor(Int, x / cutoff) (src/Sorting.jl:122-124), clamped to int32.
__device__ inline int key_comp(double x, double cutoff) {
  double f = floor(x / cutoff);
  if (!(f > -1.0e9)) f = -1.0e9;
  if (f > 1.0e9) f = 1.0e9;
  return (int)f;
}

// ---------------------------------------------------------------------------
// LSD radix sort, 8-bit digits, stable: two kernels per digit pass.
//
// The keys are cut into tiles of OS_TILE.  Each pass needs, for every tile
// and digit, the number of keys with that digit in the tiles before it.  The
// counts of pass p's tiles are taken by the kernel that writes pass p's
// input: k_key_write for pass 0, and pass p-1's scatter for pass p, which
// knows where each key lands and so which tile of the next pass holds it.
// Both count runs of equal (tile, digit) along a wavefront with one atomic
// per run (the keys are nearly in order: a wavefront holds few runs).
// k_radix_scan turns each digit's column of tile counts into exclusive
// prefixes and the digit's total; k_radix_scatter ranks its tile's keys per
// digit (stable), adds the prefixes and the digit starts, and scatters.
//
// Scratch (radix_scratch_bytes): digit totals [4][256], then two count
// arrays [tiles][256] used by alternate passes.  Every reader of a tile's
// row zeroes it, so the arrays are zero again after each sort (and are
// zeroed when allocated).
//
// Passes above the top bit of the largest key keep the order and are
// skipped; flags[3] is the number of passes that run, so the sorted pairs
// end in (keys2, vals2) when it is odd (radix_sorted_vals).  The whole sort
// is skipped when flags[0] == 0: the keys are already in order.
// ---------------------------------------------------------------------------

#ifndef OS_ITEMS
#define OS_ITEMS 16
#endif
#define OS_WAVE_KEYS (64 * OS_ITEMS)
#define OS_TILE (GR_BLOCK * OS_ITEMS)
#define RS_TOT 0      // words: digit totals [4][256]
#define RS_CNT 1024   // words: tile counts [2][tiles][256]

__device__ inline int radix_passes(unsigned bound) {
  // passes whose digit is not zero for some key below `bound`
  if (bound <= 1u) return 0;
  const int bits = 32 - __clz((int)(bound - 1u));
  return (bits + 7) >> 3;
}

// Add the lanes' bins to `cnt`: one atomic for each run of equal bins along
// the valid lanes, made by the run's first lane.
__device__ inline void radix_add_runs(unsigned bin, bool valid, unsigned *cnt) {
  const int lane = threadIdx.x & 63;
  const unsigned prev = __shfl_up(bin, 1, 64);
  const unsigned long long V = __ballot(valid);
  const bool prev_valid = lane > 0 && ((V >> (lane - 1)) & 1ull);
  const bool head = valid && (!prev_valid || prev != bin);
  const unsigned long long H = __ballot(head);
  if (head) {
    const unsigned long long ends = (H | ~V) & (lane == 63 ? 0ull : (~0ull << (lane + 1)));
    const int next = ends ? __ffsll((long long)ends) - 1 : 64;
    atomicAdd(&cnt[bin], (unsigned)(next - lane));
  }
}

// ---------------------------------------------------------------------------
// Keys: per-system key range and position bounding box
// ---------------------------------------------------------------------------

// Bounding box of the positions per dimension and system, as order-preserving
// integers (ord_d).  The cell keys' ranges follow from it (the key component
// is a monotone function of the position) and are derived in k_key_base.
// Each workgroup reduces PER consecutive entries of the block table in
// registers and flushes (workgroup reduction, then an atomic for each bound
// that improves on the current value) whenever the system changes and at the
// end.  The loads of all PER entries (table entry -> system descriptor ->
// positions) are issued before any is reduced, so their latencies overlap.
//
// The workgroups of a launch run concurrently, so they all see the initial
// bounds and most of them take their atomics; those atomics are spread over
// replicas 1 .. GR_BB_REP of the bounds (stride `rs`), one for the workgroups
// of each XCD, and folded into replica 0 afterwards (key_space, k_bb_fold).
// `flags`: also clear the sort's inversion flag for the key pass that follows.
//
// In small scenes the kernel that advances the positions takes their bounds
// for the next step instead (k_fullstep, k_rk4_apply with BB), which saves the
// launch (step_bounds).
template <int D>
__device__ inline void bb_flush(const long long *mn, const long long *mx, int s, long long *bbmin,
                                long long *bbmax) {
  __shared__ long long red[2][GR_BLOCK / 64][3];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const long long a = wave_red_ll<false>(mn[d]), bq = wave_red_ll<true>(mx[d]);
    if (lane == 0) {
      red[0][w][d] = a;
      red[1][w][d] = bq;
    }
  }
  __syncthreads();
  if (threadIdx.x < D) {
    const int d = threadIdx.x;
    long long a = LLONG_MAX, bq = LLONG_MIN;
    for (int q = 0; q < GR_BLOCK / 64; ++q) {
      a = red[0][q][d] < a ? red[0][q][d] : a;
      bq = red[1][q][d] > bq ? red[1][q][d] : bq;
    }
    // every workgroup of a system reduces into the same few words; only
    // a partial result that improves on the current value takes the atomic
    if (a != LLONG_MAX) {
      if (a < ld_dev(&bbmin[s * 3 + d])) atomicMin(&bbmin[s * 3 + d], a);
      if (bq > ld_dev(&bbmax[s * 3 + d])) atomicMax(&bbmax[s * 3 + d], bq);
    }
  }
  __syncthreads();
}
// Bounds of one workgroup's particles, all of system s, for the next step.
template <int D>
__device__ inline void bb_block(const double *x, bool live, int s, const StepBounds &B) {
  long long mn[D], mx[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    mn[d] = live ? ord_d(x[d]) : LLONG_MAX;
    mx[d] = live ? ord_d(x[d]) : LLONG_MIN;
  }
  const int r = (1 + blockIdx.x % GR_BB_REP) * B.rs;
  bb_flush<D>(mn, mx, s, B.bbmin + r, B.bbmax + r);
  if (blockIdx.x == 0 && threadIdx.x == 0) B.flags[0] = 0;  // for the next step's keys
}

template <int D, int PER>
__global__ void k_key_minmax(XP xs, const SysDesc *sd, const int *n_dev, const Blk *blk, int nblk,
                             long long *bbmin, long long *bbmax, int rs, int *flags) {
  if (flags && blockIdx.x == 0 && threadIdx.x == 0) flags[0] = 0;
  bbmin += (1 + blockIdx.x % GR_BB_REP) * rs;
  bbmax += (1 + blockIdx.x % GR_BB_REP) * rs;
  const int b0 = blockIdx.x * PER;
  int item[PER];
  bool live[PER];
  double xe[PER][D];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const Blk b = blk[b0 + k < nblk ? b0 + k : nblk - 1];
    item[k] = b.item;
    const int i = b.first + threadIdx.x;
    live[k] = b0 + k < nblk && i < n_dev[b.item];
    const int64_t gi = sd[b.item].off + i;
#pragma unroll
    for (int d = 0; d < D; ++d) xe[k][d] = live[k] ? xs[d][gi] : 0.0;
  }
  long long mn[D], mx[D];
  auto reset = [&]() {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      mn[d] = LLONG_MAX;
      mx[d] = LLONG_MIN;
    }
  };
  auto flush = [&](int s) { bb_flush<D>(mn, mx, s, bbmin, bbmax); };
  reset();
  int cur = item[0];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if (b0 + k >= nblk) break;  // uniform over the workgroup
    if (item[k] != cur) {       // uniform over the workgroup
      flush(cur);
      reset();
      cur = item[k];
    }
    if (live[k]) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const long long o = ord_d(xe[k][d]);
        mn[d] = o < mn[d] ? o : mn[d];
        mx[d] = o > mx[d] ? o : mx[d];
      }
    }
  }
  flush(cur);
}

// Reset the reduction slots of the listed systems.
__global__ void k_minmax_reset(const int *list, int nlist, long long *bbmin, long long *bbmax,
                               int rs) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nlist * 3 * GR_BB_REP) return;
  const int r = t / (nlist * 3);
  t -= r * nlist * 3;
  int s = list[t / 3], d = t % 3;
  bbmin[(r + 1) * rs + s * 3 + d] = LLONG_MAX;
  bbmax[(r + 1) * rs + s * 3 + d] = LLONG_MIN;
}

// The bounds of entry e over the replicas.
__device__ __forceinline__ void bb_fold(const long long *bbmin, const long long *bbmax, int rs,
                                        int e, long long &mn, long long &mx) {
  long long a = LLONG_MAX, b = LLONG_MIN;
#pragma unroll
  for (int r = 1; r <= GR_BB_REP; ++r) {
    const long long u = bbmin[r * rs + e], v = bbmax[r * rs + e];
    a = u < a ? u : a;
    b = v > b ? v : b;
  }
  mn = a;
  mx = b;
}
__global__ void k_bb_fold(const int *list, int nlist, long long *bbmin, long long *bbmax, int rs) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < nlist * 3) {
    const int e = list[t / 3] * 3 + t % 3;
    bb_fold(bbmin, bbmax, rs, e, bbmin[e], bbmax[e]);
  }
}

// Threads of k_key_base: one per listed system in each round.
#define KB_THREADS 1024
// Up to this many systems (a lane each) and workgroups, every workgroup of the
// counting sort's key pass finds the key bases itself, which saves a launch
// (2D dam break of 23k particles: sort 33 -> 30 us); with more workgroups the
// repeated work costs more (5700 workgroups: 145 us against 131).
#define KC_SYSTEMS 64
#define KC_BLOCKS 512

// Key space of each listed system: lexicographic linearisation of
// (k1 - kmin1, ..., kD - kminD), bases prefix-summed in list order.  Ghost
// systems reserve one extra key for padding slots.  flags[0] (the inversion
// flag) is cleared here; flags[1] records overflow.  kmin/kmax are the key
// components of the bounding box's corners: key_comp is monotone in the
// position, so they are the extremes of the particles' key components.  A
// NaN position leaves kmax below kmin or a range beyond 32 bits: overflow.
__device__ inline double unord_d(long long o) {
  return __longlong_as_double(o < 0 ? (o ^ 0x7FFFFFFFFFFFFFFFLL) : o);
}
struct KeySpace {
  int kmin[3], kmax[3];
  unsigned kr[3];        // cells per dimension; kr[0] == 0 marks a faulted system
  long long mn[3], mx[3];  // position bounds (ordered integers)
  int fault;             // GR_FAULT_*
};
// The key space of system s (n > 0 particles); returns its number of keys.
__device__ inline unsigned long long key_space(int D, double cutoff, const long long *bbmin,
                                               const long long *bbmax, int rs, int s,
                                               KeySpace &K) {
  unsigned long long range = 1;
  bool nonfinite = false;
  for (int d = 0; d < 3; ++d) {
    bb_fold(bbmin, bbmax, rs, s * 3 + d, K.mn[d], K.mx[d]);
    K.kmin[d] = K.kmax[d] = 0;
    K.kr[d] = 1u;
    if (d >= D) continue;
    const double lo = unord_d(K.mn[d]), hi = unord_d(K.mx[d]);
    const int ka = key_comp(lo, cutoff), kb = key_comp(hi, cutoff);
    K.kmin[d] = ka < kb ? ka : kb;
    K.kmax[d] = ka < kb ? kb : ka;
    long long r = (long long)K.kmax[d] - (long long)K.kmin[d] + 1;
    if (!(lo <= hi)) r = 1LL << 32;  // NaN
    K.kr[d] = (unsigned)r;
    // any product of 2^32 or more overflows the 32-bit keys: saturate there so
    // that neither this product nor the prefix sum wraps
    range = (range > 0xFFFFFFFFull || r > 0xFFFFFFFFLL) ? (1ull << 32)
                                                         : range * (unsigned long long)r;
    nonfinite = nonfinite || !(lo <= hi) || !isfinite(lo) || !isfinite(hi);
  }
  if (range > (1ull << 32)) range = 1ull << 32;
  // a system whose bounds are not finite, or whose own keys need 32 bits or
  // more, is faulted: all its keys become its base (the sort keeps its
  // order), so the systems after it keep their keys and the step goes on for
  // them
  K.fault = 0;
  if (nonfinite || range >= 0xFFFFFFFFull) {
    K.fault = nonfinite ? GR_FAULT_NONFINITE : GR_FAULT_DOMAIN;
    for (int d = 0; d < D; ++d) {
      K.kmin[d] = K.kmax[d] = 0;
      K.kr[d] = d == 0 ? 0u : 1u;
    }
    range = 1;
  }
  return range;
}
// Store what the later kernels read of a system's key space.
__device__ inline void key_space_store(const KeySpace &K, int s, bool live, long long *bbmin,
                                       long long *bbmax, int *kmin, int *kmax, unsigned *krange,
                                       int *flags, int *sysfault) {
  for (int d = 0; d < 3; ++d) {
    bbmin[s * 3 + d] = K.mn[d];
    bbmax[s * 3 + d] = K.mx[d];
    krange[s * 3 + d] = live ? K.kr[d] : 1u;
    if (live) {
      kmin[s * 3 + d] = K.kmin[d];
      kmax[s * 3 + d] = K.kmax[d];
    }
  }
  if (live && K.fault) {
    atomicOr(&sysfault[s], K.fault);
    atomicOr(&flags[1], 8);
  }
}
// Buckets of a system's `range` keys in the counting sort: a bucket is 2^sh keys,
// one where the system keeps to its budget.
__device__ inline unsigned key_buckets(unsigned long long range, unsigned budget, int &sh) {
  sh = 0;
  if (range == 0ull) return 0u;
  while (sh < 32 && ((range - 1ull) >> sh) >= (unsigned long long)budget) ++sh;
  return (unsigned)((range - 1ull) >> sh) + 1u;
}
// Flags of the whole key range: overflow, the bound of the keys and the radix
// passes below it.  The running base only grows, so overflowing at some system
// means the total overflows.
__device__ inline void key_flags(unsigned long long total, int *flags) {
  if (total >= 0xFFFFFFFFull) atomicOr(&flags[1], 1);
  flags[2] = (int)(unsigned)(total < 0xFFFFFFFFull ? total : 0xFFFFFFFFull);
  flags[3] = radix_passes((unsigned)flags[2]);
}

__global__ void __launch_bounds__(KB_THREADS)
    k_key_base(const int *list, int nlist, int D, int pad, const int *n_dev, const StepSys *st,
               long long *bbmin, long long *bbmax, int rs, int *kmin, int *kmax,
               unsigned *kbase, unsigned *krange, int *flags, int *sysfault,
               int *kshift) {
  // one workgroup: the systems' key ranges in parallel, KB_THREADS at a time,
  // and their exclusive prefix sum (each system's keys start after the ranges
  // of the systems listed before it, plus one padding key each when `pad`);
  // with `kshift`, for the counting sort, their buckets'
  __shared__ unsigned long long wsum[KB_THREADS / 64], wall[KB_THREADS / 64];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  unsigned long long carry = 0, all = 0;
  for (int q0 = 0; q0 < nlist; q0 += KB_THREADS) {
    const int q = q0 + t;
    unsigned long long range = 0, num = 0;
    int s = -1, sh = 0;
    if (q < nlist) {
      s = list[q];
      const unsigned most = st[s].key_budget;
      KeySpace K;
      const bool live = n_dev[s] > 0;
      range = key_space(D, st[s].sort_cutoff, bbmin, bbmax, rs, s, K);
      if (!live) range = 0;
      key_space_store(K, s, live, bbmin, bbmax, kmin, kmax, krange, flags, sysfault);
      range += pad ? 1 : 0;
      num = range;
      if (kshift) {
        num = key_buckets(range, most, sh);
        kshift[s] = sh;
      }
    }
    unsigned long long inc = num;
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned long long u = __shfl_up(inc, o, 64);
      if (lane >= o) inc += u;
    }
    unsigned long long sum = inc;  // of the ranges (at lane 63)
    if (__ballot(sh > 0) != 0ull) {
      sum = range;
      for (int o = 1; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
    }
    if (lane == 63) {
      wsum[w] = inc;
      wall[w] = sum;
    }
    __syncthreads();
    unsigned long long off = 0, tot = 0;
    for (int v = 0; v < KB_THREADS / 64; ++v) {
      off += v < w ? wsum[v] : 0ull;
      tot += wsum[v];
    }
    if (t == 0)
      for (int v = 0; v < KB_THREADS / 64; ++v) all += wall[v];
    if (q < nlist) kbase[s] = (unsigned)(carry + off + inc - num);
    carry += tot;
    __syncthreads();  // wsum is written again for the next systems
  }
  if (t == 0) {
    key_flags(all, flags);
    if (kshift)
      flags[2] = (int)(unsigned)carry;
    else
      flags[0] = 0;
  }
}

template <int D>
__device__ inline unsigned lin_key(XP xs, int64_t gi, double cutoff, const int *kmin,
                                   const unsigned *krange, int s) {
  unsigned k = 0;
  if (krange[s * 3] == 0u) return 0u;  // faulted system (k_key_base)
#pragma unroll
  for (int d = 0; d < D; ++d) {
    int c = key_comp(xs[d][gi], cutoff) - kmin[s * 3 + d];
    k = k * krange[s * 3 + d] + (unsigned)c;
  }
  return k;
}

// Write (key, pool index) at each particle's compact position and flag any
// key inversion inside a system (src/Sorting.jl:179-186).
template <int D>
__global__ void k_key_write(XP xs, const SysDesc *sd, const int *n_dev,
                            const StepSys *st, const Blk *blk, const int *bbase,
                            const int *kmin, const unsigned *krange, const unsigned *kbase,
                            unsigned *keys, int *vals, int *flags, unsigned *rscr) {
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int lane = threadIdx.x & 63;
  const int i = b.first + threadIdx.x;
  const int cap = sd[s].cap;
  const int n = n_dev[s];
  const int64_t gi = sd[s].off + i;
  const double cutoff = st[s].sort_cutoff;
  __shared__ unsigned kw[GR_BLOCK / 64];
  const int w = threadIdx.x >> 6;
  const bool last = threadIdx.x == GR_BLOCK - 1 && i + 1 < n;
  unsigned key, kn = 0u;
  if (i < n) {
    key = kbase[s] + lin_key<D>(xs, gi, cutoff, kmin, krange, s);
    // the key after the workgroup's last particle, the only neighbour key
    // that no thread of this workgroup computes for itself
    if (last) kn = kbase[s] + lin_key<D>(xs, gi + 1, cutoff, kmin, krange, s);
  } else {
    unsigned rng = 1;
    for (int d = 0; d < D; ++d) rng *= krange[s * 3 + d];
    key = kbase[s] + (n > 0 ? rng : 0u);
  }
  // the next particle's key: from the next lane, from the next wavefront's
  // first lane (through LDS) for lane 63, and kn for the workgroup's last
  // thread (every thread of the workgroup is active here)
  if (lane == 0) kw[w] = key;
  __syncthreads();
  unsigned k2 = __shfl_down(key, 1, 64);
  if (lane == 63) k2 = w + 1 < GR_BLOCK / 64 ? kw[w + 1] : kn;
  const bool inv = i + 1 < n && k2 < key;
  // most workgroups of a moving scene hold an inversion: one atomic per
  // workgroup at most, none once the flag reads as raised
  if (__syncthreads_or(inv) && threadIdx.x == 0 && ld_dev(&flags[0]) == 0) atomicOr(&flags[0], 1);
  if (i < cap) {
    const int p = bbase[s] + i;
    keys[p] = key;
    vals[p] = (int)gi;
  }
  // the radix sort's pass-0 tile counts (its entries are the slots below cap)
  if (flags[3] > 0) {
    const unsigned p = (unsigned)(bbase[s] + i);
    radix_add_runs((p / OS_TILE) * 256u + (key & 255u), i < cap, rscr + RS_CNT);
  }
}

// The radix sort's passes (described above the key kernels).
__device__ inline unsigned block_excl_scan256(unsigned v, unsigned *wsum) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  unsigned inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  unsigned off = 0;
  for (int q = 0; q < w; ++q) off += wsum[q];
  return off + inc - v;
}

// One workgroup per digit: the digit's tile counts become exclusive prefixes
// in place (each thread sums a run of consecutive tiles, a workgroup scan
// places the runs), and its total goes to the totals of the pass.
__global__ void __launch_bounds__(GR_BLOCK) k_radix_scan(int N, int pass, unsigned *scr,
                                                         const int *flags) {
  if (pass >= flags[3]) return;
  __shared__ unsigned wsum[GR_BLOCK / 64];
  const int ntile = (N + OS_TILE - 1) / OS_TILE;
  const int t = threadIdx.x, d = blockIdx.x;
  unsigned *cnt = scr + RS_CNT + (size_t)(pass & 1) * ntile * 256 + d;
  const int per = (ntile + GR_BLOCK - 1) / GR_BLOCK;
  const int j0 = t * per, j1 = j0 + per < ntile ? j0 + per : ntile;
  if (flags[0] == 0) {
    // keys already in order: nothing runs, so clear what k_key_write counted
    if (pass == 0)
      for (int j = j0; j < j1; ++j) cnt[(size_t)j * 256] = 0u;
    return;
  }
  unsigned sum = 0;
  for (int j = j0; j < j1; ++j) sum += cnt[(size_t)j * 256];
  unsigned run = block_excl_scan256(sum, wsum);
  for (int j = j0; j < j1; ++j) {
    const unsigned c = cnt[(size_t)j * 256];
    cnt[(size_t)j * 256] = run;
    run += c;
  }
  if (t == GR_BLOCK - 1) scr[RS_TOT + pass * 256 + d] = run;
}

// Stable scatter of one tile: wavefront w holds the tile's keys
// [w·OS_WAVE_KEYS, (w+1)·OS_WAVE_KEYS) in rounds of 64, and a key's rank
// among the wavefront's keys with its digit counts the earlier rounds, then
// the lower lanes.  A round whose digits never decrease along the lanes holds
// each digit as one run (the common case for keys nearly in order); other
// rounds match digits bit by bit with ballots.
__global__ void __launch_bounds__(GR_BLOCK)
    k_radix_scatter(const unsigned *__restrict__ kin, const int *__restrict__ vin,
                    unsigned *__restrict__ kout, int *__restrict__ vout, int N, int pass,
                    unsigned *scr, int *flags) {
  const int npass = flags[3];
  if (flags[0] == 0 || pass >= npass) return;
  const int shift = 8 * pass;
  // digit bits that vary: the top pass may use fewer than 8
  const int bits = 32 - __clz((int)((unsigned)flags[2] - 1u));
  const int nb = bits - shift < 8 ? bits - shift : 8;
  const int ntile = (N + OS_TILE - 1) / OS_TILE;
  __shared__ unsigned wcnt[GR_BLOCK / 64][256];
  __shared__ unsigned wsum[GR_BLOCK / 64];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const unsigned tile = blockIdx.x;
  const long long e0 = (long long)tile * OS_TILE + w * OS_WAVE_KEYS + lane;
  unsigned key[OS_ITEMS];
  int val[OS_ITEMS];
#pragma unroll
  for (int r = 0; r < OS_ITEMS; ++r) {
    const long long e = e0 + r * 64;
    key[r] = e < N ? kin[e] : 0u;
    val[r] = e < N ? vin[e] : 0;
  }
  // this tile's start within digit t; the row is left zeroed
  unsigned *row = scr + RS_CNT + (size_t)(pass & 1) * ntile * 256 + (size_t)tile * 256;
  const unsigned ex = row[t];
  row[t] = 0u;
#pragma unroll
  for (int q = 0; q < GR_BLOCK / 64; ++q) wcnt[q][t] = 0;
  // global start of digit t: totals of the digits below it
  const unsigned gstart = block_excl_scan256(scr[RS_TOT + pass * 256 + t], wsum);  // (synchronises)
  const unsigned long long lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const unsigned long long le_mask = (2ull << lane) - 1ull;
  unsigned rank[OS_ITEMS];
#pragma unroll
  for (int r = 0; r < OS_ITEMS; ++r) {
    const bool valid = e0 + r * 64 < N;
    const unsigned d = (key[r] >> shift) & 255u;
    const unsigned dp = __shfl_up(d, 1, 64);
    const unsigned long long V = __ballot(valid);
    unsigned rk, run;
    if (__ballot(valid && lane > 0 && d < dp) == 0ull) {
      // equal digits are adjacent: runs start where the digit changes
      const unsigned long long H = __ballot(valid && (lane == 0 || d != dp));
      const int head = 63 - __clzll((long long)(H & le_mask));
      const unsigned long long ends = (H | ~V) & ~le_mask;
      const int next = ends ? __ffsll((long long)ends) - 1 : 64;
      rk = (unsigned)(lane - head);
      run = (unsigned)(next - lane);
    } else {
      unsigned long long match = V;
      for (int b = 0; b < nb; ++b) {
        const unsigned long long bal = __ballot((d >> b) & 1u);
        match &= ((d >> b) & 1u) ? bal : ~bal;
      }
      rk = (unsigned)__popcll(match & lt_mask);
      run = (unsigned)__popcll(match);
    }
    const unsigned before = wcnt[w][d];
    rank[r] = before + rk;
    if (valid && rk == 0) wcnt[w][d] = before + run;
  }
  __syncthreads();
  // output start of (wavefront q, digit t)
  unsigned start = gstart + ex;
#pragma unroll
  for (int q = 0; q < GR_BLOCK / 64; ++q) {
    const unsigned c = wcnt[q][t];
    wcnt[q][t] = start;
    start += c;
  }
  __syncthreads();
  unsigned *cnext = scr + RS_CNT + (size_t)((pass + 1) & 1) * ntile * 256;
  const bool count_next = pass + 1 < npass;
  bool bad = false;
#pragma unroll
  for (int r = 0; r < OS_ITEMS; ++r) {
    const bool valid = e0 + r * 64 < N;
    const unsigned pos = wcnt[w][(key[r] >> shift) & 255u] + rank[r];
    // the counts place every key below N; a position beyond it is
    // reported, never written
    const bool ok = valid && pos < (unsigned)N;
    if (ok) {
      kout[pos] = key[r];
      vout[pos] = val[r];
    }
    bad = bad || (valid && !ok);
    // the next pass's tile counts
    if (count_next)
      radix_add_runs((pos / OS_TILE) * 256u + ((key[r] >> (shift + 8)) & 255u), ok, cnext);
  }
  if (bad) atomicOr(&flags[1], 16);
}

// The buffer that holds the sorted values (see the sort's header).
__device__ __forceinline__ const int *radix_sorted_vals(const int *vals, const int *vals2,
                                                        const int *flags) {
  return (flags[3] & 1) ? vals2 : vals;
}

// ---------------------------------------------------------------------------
// Grids of a step's interactions and its cleared cell arrays (CellsArgs)
// ---------------------------------------------------------------------------

// Cells of the pool per tile flag: k_cells_mark sets the flags of the tiles it
// writes to, so that k_cells_fill passes over empty regions a tile at a time.
#define CELL_TILE 1024
#define CELL_SHIFT 10
static_assert(CELL_TILE == 4 * GR_BLOCK && CELL_TILE == 1 << CELL_SHIFT, "cell tile");

// Grid of interaction `it` from the bounding boxes of its systems; cell arrays
// checked against their capacity.
__device__ inline void grid_of(const CellsArgs &A, int it, int *flags, int *sysfault) {
  const int2 ab = A.inter_sys[it];
  const double cutoff = A.cellsz[it];
  Grid G;
  double cells = 1.0;  // exact below 2^53, far beyond any capacity
  for (int d = 0; d < 3; ++d) {
    G.ming[d] = 0.0;
    G.ng[d] = 1;
    if (d >= A.D) continue;
    double mn = unord_d(A.bbmin[ab.x * 3 + d]), mx = unord_d(A.bbmax[ab.x * 3 + d]);
    if (ab.y >= 0 && A.n_dev[ab.y] > 0) {
      double mnb = unord_d(A.bbmin[ab.y * 3 + d]), mxb = unord_d(A.bbmax[ab.y * 3 + d]);
      mn = mnb < mn ? mnb : mn;
      mx = mxb > mx ? mxb : mx;
    }
    G.ming[d] = floor((mn - 2.0 * cutoff) / cutoff) * cutoff;  // _snap_to_grid :191
    double maxg = mx + 2.0 * cutoff;
    double ngd = floor((maxg - G.ming[d]) / cutoff) + 1.0;  // :179
    if (!(ngd >= 1.0) || ngd > 1.0e9) ngd = 1.0e9;
    G.ng[d] = (int)ngd;
    cells *= ngd;
  }
  const int2 ca = A.inter_carr[it];
  long long cap = A.carr[ca.x].cap;
  if (ca.y >= 0 && A.carr[ca.y].cap < cap) cap = A.carr[ca.y].cap;
  G.ok = cells + 1.0 <= (double)cap;
  if (!G.ok) {
    // an empty grid: the sweeps find no partner for these systems; the
    // systems are faulted, the other systems' grids are unaffected
    atomicOr(&flags[1], 2);
    atomicOr(&sysfault[ab.x], GR_FAULT_DOMAIN);
    if (ab.y >= 0) atomicOr(&sysfault[ab.y], GR_FAULT_DOMAIN);
  }
  G.ncells = G.ok ? (int)cells : 0;
  G.pad = 0;
  A.grids[it] = G;
}

// Workgroup k of cells_prep_blocks(A): the grids of GR_BLOCK interactions, or
// CELL_TILE cells cleared with the flags of the tiles they touch.
__device__ inline void cells_prep(const CellsArgs &A, int k, int *flags, int *sysfault) {
  const int ng = (A.n_inter + GR_BLOCK - 1) / GR_BLOCK, t = threadIdx.x;
  if (k < ng) {
    const int q = k * GR_BLOCK + t;
    if (q < A.n_inter) grid_of(A, A.inter_list[q], flags, sysfault);
    return;
  }
  const Blk b = A.cblk[k - ng];
  const CellArr C = A.carr[b.item];
  for (int c = b.first + t; c < C.cap && c < b.first + CELL_TILE; c += GR_BLOCK)
    A.cells[C.off + c] = 0;
  if (t < 2) {
    const int c = t == 0 ? b.first : min(b.first + CELL_TILE, C.cap) - 1;
    if (c >= 0) A.tflag[(C.off + c) >> CELL_SHIFT] = 0;
  }
}
__global__ void __launch_bounds__(GR_BLOCK) k_cells_prep(CellsArgs A, int *flags, int *sysfault) {
  cells_prep(A, blockIdx.x, flags, sysfault);
}

// ---------------------------------------------------------------------------
// Counting sort of the step: one table entry per key
//
// The keys of a step are cells, a few per 100 particles, so they are sorted by
// counting: k_key_count writes the keys and takes each particle a place in its
// cell (one atomic per run of equal keys along a wavefront), k_key_scan turns
// the counts into the cells' starts, k_key_place puts every particle into its
// cell, and the permutations order each cell by the particles' former places
// (the sort is stable): a particle's rank is the number of smaller former
// places in its cell, which holds a handful (of more than KT_BIG, the runs of
// former neighbours are counted instead, key_slot).  Against the radix sort's scan
// and scatter kernel per 8-bit digit (each 3 to 16 us, four of each launched
// whatever the key range) it takes two kernels.  Sort phase, radix before:
// 3D dam break of 1.4M particles 158 -> 140 us, 2D dam break of 23k 50 -> 30,
// 2D column of 12.8k 40 -> 28 (its ghosts, generated and sorted, 56 -> 28).
// Bound by the launches below 100k particles; at 1.4M by the atomics
// (k_key_count 33 us of the 140, the scan and the placement 9) and the moved
// bytes of the permutation (53 us).
//
// Table (key_table_bytes): counts, starts, tile sums, laid out for the tiles it
// was allocated with.  Every count and sum a sort raises is zero again when it
// has ended.  Each system has a budget of table entries.  One that has outgrown
// its budget since the plan was made has 2^sh keys to an entry until the plan is
// made anew (`kshift`), and its particles are ordered within an entry by their
// keys (`full`) first; the others do not notice.  Sort of 200k particles, 20 a cell
// (us), with a budget for all keys / 4 / 64 / 4096 keys to an entry: 2D 38 / 52 /
// 124 / 2260, 3D 40 / 40 / 65 / 480.
// ---------------------------------------------------------------------------

#define KT_TILE 1024  // keys per workgroup of the scan
#define KT_RANKS 8    // former places compared at a time in the rank within a cell
// Largest cell whose particles are compared one by one.  Beyond it the runs of
// equal keys along a wavefront, which the atomics of k_key_count place as one,
// are: their former places are consecutive.  Sort of a step (us), one by one /
// runs / radix kernels, 20k particles at 300 a cell 33 / 27 / 48, at 1024
// 60 / 33 / 51, all in one cell 655 / 108 / 48; 200k at 300 81 / 75 / 76, at
// 2048 181 / 87 / 66, in one cell 11500 / 1120 / 50.  (60k particles in one cell
// that interact with each other: 0.3 ms of a step's 14.5.)
#define KT_BIG 256
// Copies of each tile's sum: k_key_count's atomics are spread over them (a tile
// takes one from each of some 100 wavefronts; with one copy the kernel took
// 154 us instead of 40 in the 3D dam break of 1.4M particles).
#define KT_REP 16

// Lane's place among the valid lanes' run of equal `k` (valid lanes come
// first): lane of the run's head, and its length at the head.
__device__ inline int run_head(unsigned k, bool valid, int &len) {
  const int lane = threadIdx.x & 63;
  const unsigned prev = __shfl_up(k, 1, 64);
  const unsigned long long V = __ballot(valid);
  const unsigned long long H = __ballot(valid && (lane == 0 || prev != k));
  const unsigned long long le = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
  const unsigned long long ends = (H | ~V) & ~le;
  const int next = ends ? __ffsll((long long)ends) - 1 : 64;
  const int head = (H & le) ? 63 - __clzll((long long)(H & le)) : lane;
  len = next - lane;
  return head;
}

template <int D>
__global__ void __launch_bounds__(GR_BLOCK)
    k_key_count(XP xs, const SysDesc *sd, const int *n_dev, const StepSys *st, const Blk *blk,
                const int *bbase, const int *list, int nlist, long long *bbmin, long long *bbmax,
                int rs, int *kmin, int *kmax, unsigned *krange, unsigned *kbase, int *kshift,
                unsigned *keys, unsigned *full, unsigned *rank, int *flags, int *sysfault,
                unsigned *count, unsigned *tsum, int inl) {
  __shared__ int s_kmin[3], s_sh;
  __shared__ unsigned s_kr[3], s_base;
  __shared__ unsigned kw[GR_BLOCK / 64];
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = b.first + threadIdx.x;
  const int n = n_dev[s];
  const int64_t gi = sd[s].off + i;
  if (b.first >= n && blockIdx.x != 0) {  // beyond the live ghosts
    return;
  }
  const double cutoff = st[s].sort_cutoff;
  // (read early, though it is asked again below: the line is then at hand; 2D
  // cloud of 300k particles 14.6 -> 9.2 us)
  const int unsorted = threadIdx.x == 0 ? ld_dev(&flags[0]) : 0;
  double x[D];
#pragma unroll
  for (int d = 0; d < D; ++d) x[d] = i < n ? xs[d][gi] : 0.0;
  if (inl) {
    // the key bases, found by every workgroup for itself (the first stores them)
    if (w == 0) {
      unsigned long long range = 0;
      unsigned num = 0;
      int q = -1, sh = 0;
      KeySpace K;
      if (lane < nlist) {
        q = list[lane];
        const bool live = n_dev[q] > 0;
        range = key_space(D, st[q].sort_cutoff, bbmin, bbmax, rs, q, K);
        if (!live) range = 0;
        num = key_buckets(range, st[q].key_budget, sh);
        if (blockIdx.x == 0)
          key_space_store(K, q, live, bbmin, bbmax, kmin, kmax, krange, flags, sysfault);
      }
      unsigned inc = num;
      for (int o = 1; o < 64; o <<= 1) {
        const unsigned u = __shfl_up(inc, o, 64);
        if (lane >= o) inc += u;
      }
      if (blockIdx.x == 0) {
        if (q >= 0) {
          kbase[q] = inc - num;
          kshift[q] = sh;
        }
        for (int o = 1; o < 64; o <<= 1) range += __shfl_xor(range, o, 64);
        if (lane == 63) {
          key_flags(range, flags);
          flags[2] = (int)inc;
        }
      }
      if (q == s) {
        for (int d = 0; d < 3; ++d) {
          s_kmin[d] = K.kmin[d];
          s_kr[d] = K.kr[d];
        }
        s_base = inc - num;
        s_sh = sh;
      }
    }
  } else if (threadIdx.x == 0) {
    for (int d = 0; d < 3; ++d) {
      s_kmin[d] = kmin[s * 3 + d];
      s_kr[d] = krange[s * 3 + d];
    }
    s_base = kbase[s];
    s_sh = kshift[s];
  }
  __syncthreads();
  const bool faulted = s_kr[0] == 0u;
  const int sh = s_sh;
  auto key_of = [&](const double *p) {
    unsigned k = 0;
#pragma unroll
    for (int d = 0; d < D; ++d)
      k = k * s_kr[d] + (unsigned)(key_comp(p[d], cutoff) - s_kmin[d]);
    return faulted ? 0u : k;
  };
  unsigned key = 0xFFFFFFFFu, kn = 0u;
  if (i < n) {
    key = key_of(x);
    // the key after the workgroup's last particle, the only neighbour key
    // that no thread of this workgroup computes for itself
    if (threadIdx.x == GR_BLOCK - 1 && i + 1 < n) {
      double xn[D];
#pragma unroll
      for (int d = 0; d < D; ++d) xn[d] = xs[d][gi + 1];
      kn = key_of(xn);
    }
  }
  if (lane == 0) kw[w] = key;
  __syncthreads();
  unsigned k2 = __shfl_down(key, 1, 64);
  if (lane == 63) k2 = w + 1 < GR_BLOCK / 64 ? kw[w + 1] : kn;
  const bool inv = i + 1 < n && k2 < key;
  if (__syncthreads_or(inv) && threadIdx.x == 0 && unsorted == 0 && ld_dev(&flags[0]) == 0)
    atomicOr(&flags[0], 1);
  const bool valid = i < n;
  const int p = bbase[s] + i;
  const unsigned at = s_base + (key >> sh);  // the table's entry
  if (valid) {
    keys[p] = at;
    if (sh > 0) full[p] = key;
  }
  int len;
  int head = run_head(key, valid, len);
  unsigned r0 = 0;
  if (valid && head == lane) r0 = atomicAdd(&count[at], (unsigned)len);
  r0 = __shfl(r0, head, 64);
  if (valid) rank[p] = faulted ? (unsigned)i : r0 + (unsigned)(lane - head);
  head = run_head(at / KT_TILE, valid, len);
  if (valid && head == lane)
    atomicAdd(&tsum[at / KT_TILE * KT_REP + blockIdx.x % KT_REP], (unsigned)len);
}

// Starts of KT_TILE keys: the sums of the tiles before them, then a scan.
__global__ void __launch_bounds__(GR_BLOCK)
    k_key_scan(unsigned *count, const unsigned *tsum, unsigned *start, const int *flags) {
  const unsigned tile = blockIdx.x;
  if (tile * KT_TILE > (unsigned)flags[2]) return;
  __shared__ unsigned wsum[GR_BLOCK / 64], psum[GR_BLOCK / 64];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  uint4 *c4 = reinterpret_cast<uint4 *>(count + (size_t)tile * KT_TILE) + t;
  const uint4 c = *c4;
  *c4 = make_uint4(0u, 0u, 0u, 0u);
  if (flags[0] == 0) return;  // already in order: nothing reads the starts
  unsigned before = 0;
  for (unsigned k = t; k < tile * KT_REP; k += GR_BLOCK) before += tsum[k];
  const unsigned sum = c.x + c.y + c.z + c.w;
  unsigned inc = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
    before += __shfl_xor(before, o, 64);
  }
  if (lane == 63) {
    wsum[w] = inc;
    psum[w] = before;
  }
  __syncthreads();
  unsigned run = inc - sum;
  for (int q = 0; q < GR_BLOCK / 64; ++q) run += psum[q] + (q < w ? wsum[q] : 0u);
  reinterpret_cast<uint4 *>(start + (size_t)tile * KT_TILE)[t] =
      make_uint4(run, run + c.x, run + c.x + c.y, run + c.x + c.y + c.z);
}

// Every particle to its cell's slots (former place and key); also the tile
// sums and the listed systems' bounds back to their initial values.  The
// first nprep workgroups prepare the step's cell arrays (A): a longer chain of
// dependent loads than the others', so they start first.
__global__ void __launch_bounds__(GR_BLOCK)
    k_key_place(const SysDesc *sd, const int *n_dev, const Blk *blk, const int *bbase,
                const unsigned *keys, const unsigned *full, const int *kshift, unsigned *keys2,
                int *vals2, const unsigned *rank, const unsigned *start, unsigned *tsum, int ntile,
                int N, const int *list, int nlist, long long *bbmin, long long *bbmax, int rs,
                int *flags, int nprep, CellsArgs A, int *sysfault, int *run) {
  if ((int)blockIdx.x < nprep) {
    cells_prep(A, (int)blockIdx.x, flags, sysfault);
    return;
  }
  const int bid = (int)blockIdx.x - nprep;
  const int nthr = ((int)gridDim.x - nprep) * GR_BLOCK, me = bid * GR_BLOCK + threadIdx.x;
  for (int k = me; k < ntile * KT_REP; k += nthr) tsum[k] = 0u;
  for (int t = me; t < nlist * 3 * GR_BB_REP; t += nthr) {
    const int r = t / (nlist * 3), e = t % (nlist * 3);
    const int at = (r + 1) * rs + list[e / 3] * 3 + e % 3;
    bbmin[at] = LLONG_MAX;
    bbmax[at] = LLONG_MIN;
  }
  if (flags[0] == 0) return;
  const Blk b = blk[bid];
  const int s = b.item;
  const int i = b.first + threadIdx.x;
  if (i >= n_dev[s]) return;
  const int p = bbase[s] + i;
  const unsigned key = keys[p];
  const unsigned first = start[key];
  const unsigned slot = first + rank[p];
  const int sh = kshift[s];
  const bool big = sh > 0 || start[key + 1] - first > KT_BIG;
  if (__ballot(big) != 0ull) {  // the lengths of the runs, at their first slots
    int len;
    const int head = run_head(sh > 0 ? full[p] : key, true, len);
    if (big && head == (int)(threadIdx.x & 63) && slot < (unsigned)N) run[slot] = len;
  }
  // the counts place every particle below N; a slot beyond it is reported,
  // never written
  if (slot >= (unsigned)N) {
    atomicOr(&flags[1], 16);
    return;
  }
  keys2[slot] = key;
  vals2[slot] = (int)(sd[s].off + i);
}

// Slot p of the sorted order: the particle placed there (its pool index) and
// the slot its rank in the cell gives it.  sh: its system's kshift; rel: from a
// pool index of the system to its place in `full`.
__device__ __forceinline__ int key_slot(int p, const int *vals2, const KeyTable &kt, int sh,
                                        int64_t rel, int &slot) {
  const int v = vals2[p];
  const unsigned k = kt.keys2[p];
  const int a = (int)kt.start[k], e = (int)kt.start[k + 1];
  int r = 0;
  if (sh > 0 || e - a > KT_BIG) {
    const unsigned kv = sh > 0 ? kt.full[rel + v] : 0u;
    for (int j = a; j < e;) {
      const int u = vals2[j], len = kt.run[j] > 1 ? kt.run[j] : 1;
      const unsigned ku = sh > 0 ? kt.full[rel + u] : 0u;
      const int below = v - u;  // of the run's consecutive places
      r += ku < kv ? len : ku > kv || below <= 0 ? 0 : below < len ? below : len;
      j += len;
    }
    slot = a + r;
    return v;
  }
  for (int j = a; j < e; j += KT_RANKS) {
    int u[KT_RANKS];
#pragma unroll
    for (int q = 0; q < KT_RANKS; ++q) u[q] = vals2[j + q < e ? j + q : e - 1];
#pragma unroll
    for (int q = 0; q < KT_RANKS; ++q) r += j + q < e && u[q] < v ? 1 : 0;
  }
  slot = a + r;
  return v;
}

// ---------------------------------------------------------------------------
// Permutation of real systems (src/Sorting.jl:88-105): pool A → pool B for
// every real particle; identity where the system is not sorted this step.
// ---------------------------------------------------------------------------

__device__ inline double eos_p(int kind, double rho, double rho0, double gamma, double c);

// HALF: the leapfrog half step of the systems flagged in `halfsys` is done
// here, on the values as they are moved (the arithmetic of k_halfstep with
// mult ½): one pass over the particles instead of two.  PACK (FP32, with
// HALF): their compact partner records too, as k_pack writes them from the
// half-step state (1: ρ and p, 2: 1/ρ and p/ρ²).
// TAB: the order comes from the counting sort (each thread takes the particle
// of one slot to its place in the cell), else from the radix sort.
template <typename R, int D, bool HALF, int PACK = 0, bool TAB = false>
__global__ void k_permute_real(Pool<R> A, Pool<R> B, const SysDesc *sd, const Blk *blk,
                               const int *bbase, const int *vals, const int *vals2,
                               const int *flags, int vadj, const StepSys *st,
                               const int *halfsys, KeyTable kt) {
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int i = b.first + threadIdx.x;
  const SysDesc S = sd[s];
  if (i >= S.cap) return;
  int64_t dst = S.off + i;
  int64_t src = dst;
  if constexpr (TAB) {
    if (flags[0] != 0 && bbase[s] >= 0 && kt.krange[s * 3] != 0u) {  // not a faulted system
      int slot;
      src = key_slot(bbase[s] + i, vals2, kt, kt.kshift[s], bbase[s] - S.off, slot);
      dst = S.off + (slot - bbase[s]);
    }
  } else {
    if (flags[0] != 0 && bbase[s] >= 0) src = radix_sorted_vals(vals, vals2, flags)[bbase[s] + i];
  }
  const bool half = HALF && halfsys[s] != 0;
  // fields this step overwrites before reading them are not moved (only with
  // the half step, which has read the old rates here)
  const int skip = half ? st[s].perm_skip : 0;
  if (half) {
    const StepSys T = st[s];
    const double cf = 0.5 * T.dt;
    double xn[D];
    R vsn[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const double v = A.v[d][src];
      const R a = A.dvdt[d][src];
      xn[d] = A.x[d][src];
      vsn[d] = (R)(v + cf * (double)a);
      B.x[d][dst] = xn[d];
      B.v[d][dst] = v;
      B.vs[d][dst] = vsn[d];
      if (!(skip & 1)) B.dvdt[d][dst] = T.reset_force ? (R)S.sv[d] : a;
      if (vadj) B.vadj[d][dst] = A.vadj[d][src];
    }
    const double rho = A.rho[src];
    const R dr = A.drhodt[src];
    const double rh = fma(cf, (double)dr, rho);
    B.rho[dst] = rho;
    B.rho_h[dst] = rh;
    B.rhos[dst] = (R)rh;
    if (!(skip & 1)) B.drhodt[dst] = T.reset_force ? (R)S.srho : dr;
    R pn = (R)0;
    if (T.fuse_eos) {
      pn = (R)eos_p(T.fuse_eos, rh, T.eos_rho0, T.eos_gamma, S.c);
      B.p[dst] = pn;
    } else if (S.kind >= GR_SYS_FLUID) {
      pn = A.p[src];
      B.p[dst] = pn;
    } else {
      pn = B.p[dst];  // kept in place, as k_pack would read it
    }
    if constexpr (PACK > 0 && sizeof(R) == 4) {
      RecC cc;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        cc.xq[d] = d < D ? (int32_t)quant_of(xn[d], B.iqs) : 0;
        cc.v[d] = d < D ? (float)vsn[d] : 0.0f;
      }
      const float rs = (float)(R)rh;
      if constexpr (PACK == 2) {
        const float ir = __builtin_amdgcn_rcpf(rs);
        cc.rho = ir;
        cc.p = pn * (ir * ir);
      } else {
        cc.rho = rs;
        cc.p = pn;
      }
      B.rc[dst] = cc;
    }
  } else {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      B.x[d][dst] = A.x[d][src];
      B.v[d][dst] = A.v[d][src];
      B.dvdt[d][dst] = A.dvdt[d][src];
      if (vadj) B.vadj[d][dst] = A.vadj[d][src];
    }
    B.rho[dst] = A.rho[src];
    B.drhodt[dst] = A.drhodt[src];
    if (S.kind >= GR_SYS_FLUID) B.p[dst] = A.p[src];
  }
  B.id[dst] = A.id[src];
  if (S.kind >= GR_SYS_STRESS) {
#pragma unroll
    for (int k = 0; k < GR_MAXNS; ++k)
      if (k < S.ns) {
        const double sg = A.stress[k][src];
        B.stress[k][dst] = sg;
        B.stress_s[k][dst] = (R)sg;
        if (!(skip & 2)) B.sr[k][dst] = A.sr[k][src];
      }
  }
  if (S.kind == GR_SYS_EP) {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (k < S.nv && !(skip & 4)) B.vor[k][dst] = A.vor[k][src];
#pragma unroll
    for (int k = 0; k < GR_MAXNS; ++k)
      if (k < S.ns) {
        B.strain[k][dst] = A.strain[k][src];
        B.strainp[k][dst] = A.strainp[k][src];
      }
  }
}

// ---------------------------------------------------------------------------
// Ghosts (src/GhostParticles.jl:344-421)
// ---------------------------------------------------------------------------

// Ghost generation: candidate (boundary b, source particle i) qualifies when
// abs(da) <= cutoff && da > 0, and the ghosts follow boundary-major, then
// source order.  A thread takes one source particle and every boundary of its
// ghost system: k_ghost_count counts the qualifying candidates of each
// (boundary, block of GR_BLOCK source particles) slot, an exclusive scan of
// the slots gives each its first ghost, and k_ghost_scatter writes the ghosts
// there in source order.  Slots of ghost system g start at gslot[g],
// boundary-major.
template <int D>
__device__ inline bool ghost_qualifies(const double *xi, const Bnd &B, double gcut, double &da) {
  da = (xi[0] - B.p[0]) * B.n[0];
#pragma unroll
  for (int d = 1; d < D; ++d) da = da + (xi[d] - B.p[d]) * B.n[d];
  return fabs(da) <= gcut && da > 0.0;
}

template <int D>
__global__ void __launch_bounds__(GR_BLOCK)
    k_ghost_count(XP x, const SysDesc *sd, const Bnd *bnd, const Blk *blk, const int *gslot,
                  int *cnt, int *flags) {
  if (flags && blockIdx.x == 0 && threadIdx.x == 0) flags[0] = 0;  // for the ghosts' sort
  const Blk b = blk[blockIdx.x];
  const int g = b.item;
  const SysDesc G = sd[g];
  const SysDesc S = sd[G.src];
  const int i = b.first + threadIdx.x;
  const bool live = i < S.cap;
  const int64_t gi = S.off + (live ? i : 0);
  double xi[D];
#pragma unroll
  for (int d = 0; d < D; ++d) xi[d] = x[d][gi];
  const int nsb = (S.cap + GR_BLOCK - 1) / GR_BLOCK, sb = b.first / GR_BLOCK;
  for (int bi = 0; bi < G.nb; ++bi) {
    double da;
    const bool q = live && ghost_qualifies<D>(xi, bnd[G.bnd + bi], G.gcut, da);
    const int n = __syncthreads_count(q);
    if (threadIdx.x == 0) cnt[gslot[g] + bi * nsb + sb] = n;
  }
}

// Sum of v[0 .. n) by the workgroup.
__device__ inline int block_sum(const int *v, int n, int *wsum) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  int a = 0;
  for (int k = t; k < n; k += GR_BLOCK) a += v[k];
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
  if (lane == 0) wsum[w] = a;
  __syncthreads();
  int r = 0;
  for (int q = 0; q < GR_BLOCK / 64; ++q) r += wsum[q];
  __syncthreads();
  return r;
}

// Mirrored position, source index, boundary index, and the boundary whose
// normal slot k keeps (normals are not permuted by the ghost sort,
// src/Sorting.jl:33-40); also the ghosts' position bounds.  `scan`: the
// exclusive scan of the slots, or null: a workgroup that holds ghosts adds up
// the slots before its own (a ghost system has a few hundred).
template <int D>
__global__ void __launch_bounds__(GR_BLOCK)
    k_ghost_scatter(XP x, XPW gx, int *gidx, int *gbnd, int *gnrm, const SysDesc *sd,
                    const Bnd *bnd, const Blk *blk, const int *gslot, const int *cnt,
                    const int *scan, int *n_dev, long long *bbmin, long long *bbmax, int rs) {
  __shared__ int wc[GR_BLOCK / 64], wsum[GR_BLOCK / 64];
  const Blk b = blk[blockIdx.x];
  const int g = b.item;
  const SysDesc G = sd[g];
  const SysDesc S = sd[G.src];
  const int i = b.first + threadIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const bool live = i < S.cap;
  const int64_t gi = S.off + (live ? i : 0);
  double xi[D];
#pragma unroll
  for (int d = 0; d < D; ++d) xi[d] = x[d][gi];
  const int nsb = (S.cap + GR_BLOCK - 1) / GR_BLOCK, sb = b.first / GR_BLOCK;
  const int s0 = gslot[g];
  if (sb == 0) {
    const int tot = scan ? scan[s0 + G.nb * nsb] - scan[s0] : block_sum(cnt + s0, G.nb * nsb, wsum);
    if (threadIdx.x == 0) n_dev[g] = tot;
  }
  long long mn[D], mx[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    mn[d] = LLONG_MAX;
    mx[d] = LLONG_MIN;
  }
  bool any = false;
  for (int bi = 0; bi < G.nb; ++bi) {
    const Bnd B = bnd[G.bnd + bi];
    double da;
    const bool q = live && ghost_qualifies<D>(xi, B, G.gcut, da);
    const unsigned long long bal = __ballot(q);
    if (lane == 0) wc[w] = __popcll(bal);
    __syncthreads();
    int woff = 0, tot = 0;
    for (int v = 0; v < GR_BLOCK / 64; ++v) {
      woff += v < w ? wc[v] : 0;
      tot += wc[v];
    }
    __syncthreads();  // wc is written again for the next boundary
    if (tot == 0) continue;  // uniform over the workgroup
    any = true;
    const int k0 = scan ? scan[s0 + bi * nsb + sb] - scan[s0]
                        : block_sum(cnt + s0, bi * nsb + sb, wsum);
    if (q) {
      const int k = k0 + woff + __popcll(bal & ((1ull << lane) - 1ull));
      const int64_t go = G.off + k;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const double xm = xi[d] - (2.0 * da) * B.n[d];
        gx[d][go] = xm;
        const long long o = ord_d(xm);
        mn[d] = o < mn[d] ? o : mn[d];
        mx[d] = o > mx[d] ? o : mx[d];
      }
      gidx[go] = i;
      gbnd[go] = bi;
      gnrm[go] = bi;
    }
  }
  if (!bbmin || !any) return;
  bbmin += (1 + blockIdx.x % GR_BB_REP) * rs;
  bbmax += (1 + blockIdx.x % GR_BB_REP) * rs;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const long long a = wave_red_ll<false>(mn[d]), z = wave_red_ll<true>(mx[d]);
    if (lane == 0 && a != LLONG_MAX) {
      if (a < ld_dev(&bbmin[g * 3 + d])) atomicMin(&bbmin[g * 3 + d], a);
      if (z > ld_dev(&bbmax[g * 3 + d])) atomicMax(&bbmax[g * 3 + d], z);
    }
  }
}

// Ghost sort permutation: generation scratch → pool (x, idx_original,
// idx_boundary).
template <int D, bool TAB>
__global__ void k_permute_ghost(XP gxs, const int *gidx_s, const int *gbnd_s, XPW x, int *gidx,
                                int *gbnd, const SysDesc *sd, const int *n_dev, const Blk *blk,
                                const int *bbase, const int *vals, const int *vals2,
                                const int *flags, KeyTable kt) {
  const Blk b = blk[blockIdx.x];
  const int g = b.item;
  const int k = b.first + threadIdx.x;
  const SysDesc G = sd[g];
  if (k >= n_dev[g]) return;
  int64_t dst = G.off + k;
  int64_t src = dst;
  if constexpr (TAB) {
    if (flags[0] != 0 && kt.krange[g * 3] != 0u) {
      const int p0 = (int)kt.start[kt.kbase[g]];  // the live ghosts of the systems before
      int slot;
      src = key_slot(p0 + k, vals2, kt, kt.kshift[g], bbase[g] - G.off, slot);
      dst = G.off + (slot - p0);
    }
  } else {
    if (flags[0] != 0) src = radix_sorted_vals(vals, vals2, flags)[bbase[g] + k];
  }
#pragma unroll
  for (int d = 0; d < D; ++d) x[d][dst] = gxs[d][src];
  gidx[dst] = gidx_s[src];
  gbnd[dst] = gbnd_s[src];
}

// Partner records of a particle (positions, shadows of density and velocity,
// pressure, stress), read by the pair sweeps; which of them by GR_REC_* flags.
template <typename R>
struct Rec {
  double x[3];
  R v[3], rho, p;
  float s[8];
};
template <typename R>
__device__ inline void rec_load_stress(const Pool<R> &P, const SysDesc &S, int64_t g, Rec<R> &r) {
#pragma unroll
  for (int k = 0; k < 8; ++k) r.s[k] = 0.0f;
  if (S.kind >= GR_SYS_STRESS) {
#pragma unroll
    for (int k = 0; k < GR_MAXNS; ++k)
      if (k < S.ns) r.s[k] = (float)P.stress_s[k][g];
  }
}
template <typename R>
__device__ inline void rec_load(const Pool<R> &P, const SysDesc &S, int64_t g, int D, int mode,
                                Rec<R> &r) {
  if (!(mode & GR_REC_S_ONLY)) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      r.x[d] = d < D ? P.x[d][g] : 0.0;
      r.v[d] = d < D ? P.vs[d][g] : (R)0;
    }
    r.rho = P.rhos[g];
    r.p = P.p[g];
  }
  if (sizeof(R) == 4 && (mode & GR_REC_S)) rec_load_stress(P, S, g, r);
}
template <typename R>
__device__ inline void rec_store(const Pool<R> &P, int64_t g, int D, int mode, const Rec<R> &r) {
  if (!(mode & GR_REC_S_ONLY)) {
    if (sizeof(R) == 8 || !(mode & GR_REC_C)) {
      RecA<R> a;
      RecB<R> b;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        a.x[d] = r.x[d];
        b.v[d] = r.v[d];
      }
      a.rho = r.rho;
      if constexpr (sizeof(R) == 4) {
        a.p = r.p;
        b.pad = 0.0f;
      } else {
        b.p = r.p;
      }
      P.ra[g] = a;
      P.rb[g] = b;
    }
    if constexpr (sizeof(R) == 4) {
      RecC c;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        c.xq[d] = d < D ? (int32_t)quant_of(r.x[d], P.iqs) : 0;
        c.v[d] = r.v[d];
      }
      if (mode & GR_REC_INV) {  // 1/ρ and p/ρ² (the FluidPfn S = 2 force sweep)
        const float ir = __builtin_amdgcn_rcpf(r.rho);
        c.rho = ir;
        c.p = r.p * (ir * ir);
      } else {
        c.rho = r.rho;
        c.p = r.p;
      }
      P.rc[g] = c;
    }
  }
  if constexpr (sizeof(R) == 4) {
    if (mode & GR_REC_S) {  // stages with Cauchy sweeps
      // the whole record also in 2D, where the sweeps read only its first half:
      // writing half of every 32-byte record measured slower (partial lines)
      RecS q;
      q.a = make_float4(r.s[0], r.s[1], r.s[2], r.s[3]);
      q.b = make_float4(r.s[4], r.s[5], r.s[6], r.s[7]);
      P.rs[g] = q;
    }
  }
}

// update_ghost_kinematics! (:404-421): reflected half-step velocity of the
// source and its density, with the normal of the ghost's slot.
template <typename R>
__device__ inline void ghost_kin(const Pool<R> &P, int64_t si, int64_t go, const Bnd &B, int D,
                                 Rec<R> &r) {
  R vr[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) vr[d] = d < D ? P.vs[d][si] : (R)0;
  R dd = vr[0] * (R)B.n[0];
#pragma unroll
  for (int d = 1; d < 3; ++d)
    if (d < D) dd = dd + vr[d] * (R)B.n[d];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    r.v[d] = d < D ? vr[d] - (R)2 * dd * (R)B.n[d] : (R)0;
    if (d < D) P.vs[d][go] = r.v[d];
  }
  r.rho = P.rhos[si];
  P.rhos[go] = r.rho;
}
template <typename R>
__global__ void k_ghost_kin(Pool<R> P, const SysDesc *sd, const Bnd *bnd, const int *n_dev,
                            const Blk *blk, int D) {
  const Blk b = blk[blockIdx.x];
  const int g = b.item;
  const int k = b.first + threadIdx.x;
  const SysDesc G = sd[g];
  if (k >= n_dev[g]) return;
  const int64_t go = G.off + k;
  Rec<R> r;
  ghost_kin(P, sd[G.src].off + P.gidx[go], go, bnd[G.bnd + P.gnrm[go]], D, r);
}

// _apply_mode(σ, HouseholderReflect(), n̂) (:66-110) in FP64, one function
// per Voigt length so every index is static.
__device__ inline void householder3(double *s, const double *n) {
  const double nx = n[0], ny = n[1];
  const double tx = s[0] * nx + s[2] * ny, ty = s[2] * nx + s[1] * ny;
  const double q = tx * nx + ty * ny;
  const double o0 = s[0] - 4 * tx * nx + 4 * q * nx * nx;
  const double o1 = s[1] - 4 * ty * ny + 4 * q * ny * ny;
  const double o2 = s[2] - 2 * (tx * ny + nx * ty) + 4 * q * nx * ny;
  s[0] = o0;
  s[1] = o1;
  s[2] = o2;
}
__device__ inline void householder4(double *s, const double *n) {
  const double nx = n[0], ny = n[1];
  const double tx = s[0] * nx + s[3] * ny, ty = s[3] * nx + s[1] * ny;
  const double q = tx * nx + ty * ny;
  const double o0 = s[0] - 4 * tx * nx + 4 * q * nx * nx;
  const double o1 = s[1] - 4 * ty * ny + 4 * q * ny * ny;
  const double o3 = s[3] - 2 * (tx * ny + nx * ty) + 4 * q * nx * ny;
  s[0] = o0;
  s[1] = o1;
  s[3] = o3;
}
__device__ inline void householder6(double *s, const double *n) {
  const double nx = n[0], ny = n[1], nz = n[2];
  const double tx = s[0] * nx + s[3] * ny + s[4] * nz;
  const double ty = s[3] * nx + s[1] * ny + s[5] * nz;
  const double tz = s[4] * nx + s[5] * ny + s[2] * nz;
  const double q = tx * nx + ty * ny + tz * nz;
  const double o0 = s[0] - 4 * tx * nx + 4 * q * nx * nx;
  const double o1 = s[1] - 4 * ty * ny + 4 * q * ny * ny;
  const double o2 = s[2] - 4 * tz * nz + 4 * q * nz * nz;
  const double o3 = s[3] - 2 * (tx * ny + nx * ty) + 4 * q * nx * ny;
  const double o4 = s[4] - 2 * (tx * nz + nx * tz) + 4 * q * nx * nz;
  const double o5 = s[5] - 2 * (ty * nz + ny * tz) + 4 * q * ny * nz;
  s[0] = o0;
  s[1] = o1;
  s[2] = o2;
  s[3] = o3;
  s[4] = o4;
  s[5] = o5;
}

// GhostCopier of one stage (:112-129): copy p, copy or reflect stress.
// copy[g] = {copy_p, stress_mode (-1 none, 0 plain, 1 Householder)}.
template <typename R, int NS>
__device__ __forceinline__ void ghost_copy_stress(const Pool<R> &P, int64_t si, int64_t go, int mode,
                                                  const double *n, Rec<R> &r) {
  double s[NS];
#pragma unroll
  for (int q = 0; q < NS; ++q) s[q] = P.stress[q][si];
  if (mode == GR_COPY_HOUSEHOLDER) {
    if (NS == 3) householder3(s, n);
    if (NS == 4) householder4(s, n);
    if (NS == 6) householder6(s, n);
  }
#pragma unroll
  for (int q = 0; q < NS; ++q) {
    P.stress_s[q][go] = (R)s[q];
    r.s[q] = (float)(R)s[q];
  }
}
template <typename R>
__device__ inline void ghost_copy(const Pool<R> &P, const SysDesc &S, int64_t si, int64_t go,
                                  int2 cp, const Bnd &B, Rec<R> &r) {
  if (cp.x) {
    r.p = P.p[si];
    P.p[go] = r.p;
  }
  if (cp.y >= 0) {
    if (S.ns == 3) ghost_copy_stress<R, 3>(P, si, go, cp.y, B.n, r);
    if (S.ns == 4) ghost_copy_stress<R, 4>(P, si, go, cp.y, B.n, r);
    if (S.ns == 6) ghost_copy_stress<R, 6>(P, si, go, cp.y, B.n, r);
  }
}
template <typename R>
__global__ void k_ghost_copy(Pool<R> P, const SysDesc *sd, const Bnd *bnd, const int *n_dev,
                             const Blk *blk, const int2 *copy) {
  const Blk b = blk[blockIdx.x];
  const int g = b.item;
  const int k = b.first + threadIdx.x;
  const SysDesc G = sd[g];
  if (k >= n_dev[g]) return;
  const int64_t go = G.off + k;
  Rec<R> r;
  ghost_copy(P, sd[G.src], sd[G.src].off + P.gidx[go], go, copy[g], bnd[G.bnd + P.gnrm[go]], r);
}

// Partner records: of the particles of `blk` (mode < 0: none), then of the
// ghosts of `gblk`, with their kinematics and the stage's copies where asked.
// One launch for what took up to four (kinematics, copies, two packs), each 2.5
// to 4.5 us in a small scene and a chain of dependent loads: step of a 2D column
// of 13k particles 122 -> 118 us with it and the records written by the
// updaters, in FP64 of 2.3k 116 -> 110, 3D column of 179k 376 -> 371.
template <typename R>
__global__ void __launch_bounds__(GR_BLOCK)
    k_pack(Pool<R> P, const SysDesc *sd, const int *n_dev, const Blk *blk, int nblk, int mode,
           const Blk *gblk, int gmode, const Bnd *bnd, const int2 *copy, int kin, int D) {
  const bool ghost = (int)blockIdx.x >= nblk;
  const Blk b = ghost ? gblk[(int)blockIdx.x - nblk] : blk[blockIdx.x];
  const int i = b.first + threadIdx.x;
  if (i >= n_dev[b.item]) return;
  const SysDesc S = sd[b.item];
  const int64_t g = S.off + i;
  Rec<R> r;
  rec_load(P, S, g, D, ghost ? gmode : mode, r);
  if (ghost && (kin || copy)) {
    const SysDesc F = sd[S.src];
    const int64_t si = F.off + P.gidx[g];
    const Bnd B = bnd[S.bnd + P.gnrm[g]];
    if (kin) ghost_kin(P, si, g, B, D, r);
    if (copy) ghost_copy(P, F, si, g, copy[b.item], B, r);
  }
  rec_store(P, g, D, ghost ? gmode : mode, r);
}

// ---------------------------------------------------------------------------
// Device-wide exclusive scan of int32 (out has N + 1 entries, out[N] = total)
// ---------------------------------------------------------------------------

#define SCAN_TILE 1024

__global__ void k_scan_local(const int *in, int *out, int *bsum, int N) {
  __shared__ int s[SCAN_TILE];
  const int t = threadIdx.x;  // 256 threads × 4
  const int base = blockIdx.x * SCAN_TILE;
  int v[4], tot = 0;
  for (int q = 0; q < 4; ++q) {
    int e = base + t * 4 + q;
    v[q] = e < N ? in[e] : 0;
    tot += v[q];
  }
  s[t] = tot;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    int a = t >= o ? s[t - o] : 0;
    __syncthreads();
    s[t] += a;
    __syncthreads();
  }
  int run = t > 0 ? s[t - 1] : 0;
  for (int q = 0; q < 4; ++q) {
    int e = base + t * 4 + q;
    if (e < N) out[e] = run;
    run += v[q];
  }
  if (t == 255) bsum[blockIdx.x] = s[255];
}

__global__ void k_scan_blocks(int *bsum, int nb, int *out, int N) {
  __shared__ int part[1024];
  const int t = threadIdx.x;
  const int per = (nb + 1023) / 1024;
  const int b0 = t * per, b1 = min(nb, b0 + per);
  int s = 0;
  for (int k = b0; k < b1; ++k) s += bsum[k];
  part[t] = s;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    int v = t >= o ? part[t - o] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int run = t > 0 ? part[t - 1] : 0;
  for (int k = b0; k < b1; ++k) {
    int c = bsum[k];
    bsum[k] = run;
    run += c;
  }
  if (t == 1023) out[N] = part[1023];
}

__global__ void k_scan_add(int *out, const int *bsum, int N) {
  const int e = blockIdx.x * SCAN_TILE + threadIdx.x * 4;
  const int add = bsum[blockIdx.x];
  for (int q = 0; q < 4; ++q)
    if (e + q < N) out[e + q] += add;
}

// ---------------------------------------------------------------------------
// Grid / CSR (src/Interaction.jl:123-236)
// ---------------------------------------------------------------------------

template <int D>
__device__ inline int cell_flat0(XP x, int64_t gi, const Grid &G,
                                 double cell) {  // _cell_1idx − 1 (:197-206)
  long long flat = 0, stride = 1;
#pragma unroll
  for (int d = D - 1; d >= 0; --d) {
    long long cd = (long long)floor((x[d][gi] - G.ming[d]) / cell);
    flat += cd * stride;
    stride *= G.ng[d];
  }
  return (int)flat;
}

// Three launches, or two in a step, whose last sort prepares the cells
// (cells_prep): a launch costs 2.5 to 4 us in a scene of 20k particles whatever
// it does.  The five before them (grids, clearing, marks and two for the fill)
// took 13 us there and 43 at 1.4M particles; these two 5 to 7 and 24.

// First particle of each run of equal cells (forward pass :219-226); the
// last run of a cell wins, as the serial loop's last write does.
template <int D>
__global__ void __launch_bounds__(GR_BLOCK)
    k_cells_mark(XP x, int *cells, int *tflag, const CellArr *carr, const Grid *grids,
                 const double *cellsz, const SysDesc *sd, const int *n_dev, const Blk *blk) {
  const Blk b = blk[blockIdx.x];
  const CellArr C = carr[b.item];
  const int i = b.first + threadIdx.x;
  const int n = n_dev[C.sys];
  const Grid G = grids[C.grid];
  if (G.ncells <= 0) return;  // uniform over the block
  __shared__ int cw[GR_BLOCK / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const bool live = i < n;
  const double cell = cellsz[C.grid];
  const int64_t gi = sd[C.sys].off + i;
  const int c = live ? cell_flat0<D>(x, gi, G, cell) : -1;
  // the cell of particle i − 1: the previous lane's, the previous wavefront's
  // last lane's (through LDS), and for the workgroup's first thread its own
  // computation (the only one no other thread makes)
  const int c0 = (threadIdx.x == 0 && live && i > 0) ? cell_flat0<D>(x, gi - 1, G, cell) : -1;
  if (lane == 63) cw[w] = c;
  __syncthreads();
  int prev = __shfl_up(c, 1, 64);
  if (lane == 0) prev = w > 0 ? cw[w - 1] : c0;
  if (live && c != prev && c >= 0 && c < G.ncells) {
    atomicMax(&cells[C.off + c], i + 1);
    // (the first lane of a run of one tile: the flag's line is shared widely)
    const int64_t T = (C.off + c) >> CELL_SHIFT;
    if (lane == 0 || prev < 0 || (C.off + prev) >> CELL_SHIFT != T) tflag[T] = 1;
  }
}

// Backward pass (:231-235): every empty cell takes the first non-empty start
// to its right, the end of the array (the sentinel n + 1, :228) one after its
// last.  A workgroup fills its tile from the right; cells after its last start
// take the first start beyond the tile, which it finds for itself, whole tiles
// without a start passed over by their flags.  A cell that another workgroup
// has filled meanwhile holds that same start, so either reading is right.

__device__ inline int first_nz(int a, int b) { return a != 0 ? a : b; }

// First start at or after cell p of the pool, below `lim`; `end` if none.
__device__ inline int next_start(const int *cells, const int *tflag, int64_t p, int64_t lim,
                                 int end) {
  const int lane = threadIdx.x & 63;
  while (p < lim) {
    const int64_t last = (lim - 1) >> CELL_SHIFT;
    int64_t T = -1;
    for (int64_t k0 = p >> CELL_SHIFT; k0 <= last; k0 += 256) {
      int first = 4;
#pragma unroll
      for (int q = 3; q >= 0; --q) {
        const int64_t k = k0 + lane * 4 + q;
        if (k <= last && tflag[k] != 0) first = q;
      }
      const unsigned long long m = __ballot(first < 4);
      if (m != 0ull) {
        const int l = __ffsll((long long)m) - 1;
        T = k0 + l * 4 + __shfl(first, l, 64);
        break;
      }
    }
    if (T < 0) return end;
    const int64_t t0 = T << CELL_SHIFT;
    for (int64_t c0 = p > t0 ? p : t0; c0 < t0 + CELL_TILE; c0 += 256) {
      int v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t c = c0 + q * 64 + lane;
        v[q] = c < lim && c < t0 + CELL_TILE ? ld_dev(&cells[c]) : 0;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const unsigned long long m = __ballot(v[q] != 0);
        if (m != 0ull) return __shfl(v[q], __ffsll((long long)m) - 1, 64);
      }
    }
    p = t0 + CELL_TILE;
  }
  return end;
}

__global__ void __launch_bounds__(GR_BLOCK)
    k_cells_fill(int *cells, const int *tflag, const CellArr *carr, const Grid *grids,
                 const int *n_dev, const Blk *blk) {
  __shared__ int s[GR_BLOCK / 64], s_last, s_carry;
  const Blk b = blk[blockIdx.x];
  const CellArr C = carr[b.item];
  const int ncells = grids[C.grid].ncells;
  if (b.first > ncells) return;  // uniform: no cell of this block is in the grid
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int end = n_dev[C.sys] + 1;
  const int c0 = b.first + t * 4;
  int v[4];
  for (int q = 0; q < 4; ++q) {
    const int c = c0 + q;
    v[q] = c < ncells ? cells[C.off + c] : end;
  }
  if (t == GR_BLOCK - 1) s_last = v[3];
  // thread-local suffix, then the wavefront's (lanes lane..63) by shuffles
  for (int q = 2; q >= 0; --q) v[q] = first_nz(v[q], v[q + 1]);
  int a = v[0];
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_down(a, o, 64);
    if (lane + o < 64) a = first_nz(a, u);
  }
  if (lane == 0) s[w] = a;
  __syncthreads();
  int rw = 0;  // first start after this wavefront
  if (s_last == 0) {  // uniform over the workgroup
    if (w == 0) {
      const int u =
          next_start(cells, tflag, C.off + b.first + CELL_TILE, C.off + ncells, end);
      if (lane == 0) s_carry = u;
    }
    __syncthreads();
    rw = s_carry;
  }
  for (int q = GR_BLOCK / 64 - 1; q > w; --q) rw = first_nz(s[q], rw);
  const int nx = __shfl_down(a, 1, 64);
  const int right = first_nz(lane < 63 ? nx : 0, rw);
  for (int q = 0; q < 4; ++q) {
    const int c = c0 + q;
    if (c < C.cap && c <= ncells) cells[C.off + c] = first_nz(v[q], right);
  }
}

// ---------------------------------------------------------------------------
// Leapfrog per-particle kernels (src/TimeIntegration.jl:645-685)
// ---------------------------------------------------------------------------

// Julia ^(Float64, Integer) (compensated power by squaring, fused muladd).
__device__ inline double jl_pow_int(double x, long long n) {
  if (n == 0) return 1.0;
  double y = 1.0, xnlo = 0.0, ynlo = 0.0;
  if (n == 3) return x * x * x;
  if (n < 0) {
    double rx = 1.0 / x;
    if (n == -2) return rx * rx;
    if (isfinite(x)) xnlo = -fma(x, rx, -1.0) * rx;
    x = rx;
    n = -n;
  }
  while (n > 1) {
    if (n & 1) {
      double err = fma(y, xnlo, x * ynlo);
      double hi = x * y;
      double lo = fma(x, y, -hi);
      y = hi;
      ynlo = lo + err;
    }
    double err = x * 2 * xnlo;
    double hi = x * x;
    double lo = fma(x, x, -hi);
    x = hi;
    xnlo = lo + err;
    n >>= 1;
  }
  double err = fma(y, xnlo, x * ynlo);
  return (isfinite(x) && isfinite(err)) ? fma(x, y, err) : x * y;
}

// Julia ^(Float64, Float64) for the EOS exponent.
__device__ inline double jl_pow(double x, double y) {
  if (x == 1.0) return 1.0;
  double t = trunc(y);
  if (t == y && fabs(y) < 1.0e18) {
    long long yi = (long long)y;
    if (yi == 0) return 1.0;
    if (yi >= -4096 && yi <= 3 * 8192) return jl_pow_int(x, yi);
  }
  return pow(x, y);
}

__device__ inline double eos_p(int kind, double rho, double rho0, double gamma, double c) {
  if (kind == GR_UPD_TAIT) return rho0 * c * c / gamma * (jl_pow(rho / rho0, gamma) - 1.0);
  return c * c * (rho - rho0);
}

// _halfstep_ps! (:158-162) writing the half-step state to the sweep shadows
// (v and ρ keep their start-of-step values for the full step), the
// FP64 half-step density, the stage-1 EOS when fused, and the source reset.
template <typename R, int D>
__global__ void k_halfstep(Pool<R> P, const SysDesc *sd, const StepSys *st, const Blk *blk,
                           double mult, int keep) {
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int i = b.first + threadIdx.x;
  const SysDesc S = sd[s];
  if (i >= S.cap) return;
  const StepSys T = st[s];
  const int64_t g = S.off + i;
  // stage state q = q0 + (mult·dt)·dqdt: the leapfrog half step (mult ½) and
  // the RK4 stage advances (_rk4_advance_all!, src/TimeIntegration.jl:340-348;
  // keep: the first RK4 stage, q = q0)
  const double cf = mult * T.dt;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    double vh = keep ? P.v[d][g] : P.v[d][g] + cf * (double)P.dvdt[d][g];
    P.vs[d][g] = (R)vh;
  }
  const double rh = keep ? P.rho[g] : fma(cf, (double)P.drhodt[g], P.rho[g]);
  P.rho_h[g] = rh;
  P.rhos[g] = (R)rh;
  if (T.fuse_eos) P.p[g] = (R)eos_p(T.fuse_eos, rh, T.eos_rho0, T.eos_gamma, S.c);
  if (T.reset_force) {
#pragma unroll
    for (int d = 0; d < D; ++d) P.dvdt[d][g] = (R)S.sv[d];
    P.drhodt[g] = (R)S.srho;
  }
}

// RK4 (src/TimeIntegration.jl:350-362,801-811): damping of the stage rates,
// then acc += w·dqdt (vectors unfused, the density by the fused axpy).
template <typename R, int D>
__global__ void k_rk4_acc(Pool<R> P, const SysDesc *sd, const StepSys *st, const Blk *blk,
                          double w, int first) {
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int i = b.first + threadIdx.x;
  const SysDesc S = sd[s];
  if (i >= S.cap) return;
  const StepSys T = st[s];
  const int64_t g = S.off + i;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    double a = (double)P.dvdt[d][g];
    if (T.damping) {
      a = a - T.gdt * (double)P.vs[d][g];
      P.dvdt[d][g] = (R)a;
      a = (double)P.dvdt[d][g];
    }
    P.acc[d][g] = (first ? 0.0 : P.acc[d][g]) + w * a;
  }
  P.acc[3][g] = fma(w, (double)P.drhodt[g], first ? 0.0 : P.acc[3][g]);
}

// q = q0 + dt·acc, then x += dt·v (_apply_acc_all!, _update_positions_all!).
// BB: and the bounds of x for the next step's sort.
template <typename R, int D, bool BB>
__global__ void k_rk4_apply(Pool<R> P, const SysDesc *sd, const StepSys *st, const Blk *blk,
                            int pos, StepBounds B) {
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int i = b.first + threadIdx.x;
  const SysDesc S = sd[s];
  const bool live = i < S.cap;
  double x[D] = {};
  if (live) {
    const StepSys T = st[s];
    const int64_t g = S.off + i;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const double vn = P.v[d][g] + T.dt * P.acc[d][g];
      P.v[d][g] = vn;
      if (pos) {
        x[d] = P.x[d][g] + T.dt * vn;
        P.x[d][g] = x[d];
      }
    }
    P.rho[g] = fma(T.dt, P.acc[3][g], P.rho[g]);
  }
  if constexpr (BB) bb_block<D>(x, live && i < B.n_dev[s], s, B);
}

// _apply_damping_all! (:251-271), _fullstep_q_all! (:227-232),
// _update_positions_all! (:235-240).  v and x use separate products and sums
// (SVector arithmetic is outside @fastmath); ρ uses the fused axpy.
// BB: and the bounds of x for the next step's sort.
template <typename R, int D, bool BB>
__global__ void k_fullstep(Pool<R> P, const SysDesc *sd, const StepSys *st, const Blk *blk,
                           int pos, StepBounds B) {
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int i = b.first + threadIdx.x;
  const SysDesc S = sd[s];
  const bool live = i < S.cap;
  double x[D] = {};
  if (live) {
    const StepSys T = st[s];
    const int64_t g = S.off + i;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      double a = (double)P.dvdt[d][g];
      if (T.damping) {
        a = a - T.gdt * (double)P.vs[d][g];
        P.dvdt[d][g] = (R)a;
        a = (double)P.dvdt[d][g];
      }
      double vn = P.v[d][g] + T.dt * a;
      P.v[d][g] = vn;
      if (pos) {
        x[d] = P.x[d][g] + T.dt * vn;
        P.x[d][g] = x[d];
      }
    }
    P.rho[g] = fma(T.dt, (double)P.drhodt[g], P.rho[g]);
  }
  if constexpr (BB) bb_block<D>(x, live && i < B.n_dev[s], s, B);
}

// _xsph_correction! (src/TimeIntegration.jl:423-436) around the XSPH sweep.
// mode 0 (integrated systems): v ← v + (−1)·v_adjustment, v_adjustment ← 0,
//   and the sweep's view of v and ρ (the shadows) from the masters;
// mode 1 (virtual systems): shadows from the masters only;
// mode 2 (integrated systems): v ← v + 1·v_adjustment, then the position
//   update x ← x + dt·v (_update_positions_all!, :235-240).
template <typename R, int D>
__global__ void k_xsph(Pool<R> P, const SysDesc *sd, const StepSys *st, const int *n_dev,
                       const Blk *blk, int mode) {
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int i = b.first + threadIdx.x;
  if (i >= n_dev[s]) return;
  const int64_t g = sd[s].off + i;
  if (mode == 2) {
    const double dt = st[s].dt;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const double vn = P.v[d][g] + 1.0 * P.vadj[d][g];
      P.v[d][g] = vn;
      P.x[d][g] = P.x[d][g] + dt * vn;
    }
    return;
  }
#pragma unroll
  for (int d = 0; d < D; ++d) {
    double vn = P.v[d][g];
    if (mode == 0) {
      vn = vn + (-1.0) * P.vadj[d][g];
      P.v[d][g] = vn;
      P.vadj[d][g] = 0.0;
    }
    P.vs[d][g] = (R)vn;
  }
  P.rhos[g] = (R)P.rho[g];
}

// ---------------------------------------------------------------------------
// State updaters of one stage (src/StateUpdaters.jl)
// ---------------------------------------------------------------------------

// HookeLawStressUpdater (src/StateUpdaters.jl:366-405): elastic increment
// with the Jaumann correction; p = −(σxx + σyy + σzz)/3.
template <typename R>
__device__ __forceinline__ void hooke_update(Pool<R> P, int64_t g, double E, double nu, double dt) {
  const double sxx = P.stress[0][g], syy = P.stress[1][g], szz = P.stress[2][g],
               sxy = P.stress[3][g];
  const double dexx = (double)P.sr[0][g] * dt, deyy = (double)P.sr[1][g] * dt,
               dezz = (double)P.sr[2][g] * dt, dexy = (double)P.sr[3][g] * dt;
  const double D0 = E / ((1.0 + nu) * (1.0 - 2 * nu));
  double dsxx = D0 * ((1.0 - nu) * dexx + nu * deyy + nu * dezz);
  double dsyy = D0 * (nu * dexx + (1.0 - nu) * deyy + nu * dezz);
  const double dszz = D0 * (nu * dexx + nu * deyy + (1.0 - nu) * dezz);
  double dsxy = D0 * (1.0 - 2 * nu) * dexy;
  const double wdt = (double)P.vor[0][g] * dt;
  dsxx -= 2 * sxy * wdt;
  dsyy += 2 * sxy * wdt;
  dsxy += (sxx - syy) * wdt;
  const double n[4] = {sxx + dsxx, syy + dsyy, szz + dszz, sxy + dsxy};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    P.stress[k][g] = n[k];
    P.stress_s[k][g] = (R)n[k];
  }
  P.p[g] = (R)(-(n[0] + n[1] + n[2]) / 3.0);
}

// ElastoPlasticStressUpdater (:216-335), FP64.  prm = {E, nu, a_phi, k_c,
// a_psi} with the trigonometric constants evaluated on the host.
template <typename R>
__device__ __forceinline__ void ep_update(Pool<R> P, int64_t g, double E, double nu, double a_phi,
                                          double k_c, double a_psi, double dt) {
  double sxx = P.stress[0][g], syy = P.stress[1][g], szz = P.stress[2][g], sxy = P.stress[3][g];
  double dexx = (double)P.sr[0][g] * dt, deyy = (double)P.sr[1][g] * dt,
         dezz = (double)P.sr[2][g] * dt, dexy = (double)P.sr[3][g] * dt;
  double D0 = E / ((1.0 + nu) * (1.0 - 2 * nu));
  double dsxx = D0 * ((1.0 - nu) * dexx + nu * deyy + nu * dezz);
  double dsyy = D0 * (nu * dexx + (1.0 - nu) * deyy + nu * dezz);
  double dszz = D0 * (nu * dexx + nu * deyy + (1.0 - nu) * dezz);
  double dsxy = D0 * (1.0 - 2 * nu) * dexy;
  double wdt = (double)P.vor[0][g] * dt;
  dsxx -= 2 * sxy * wdt;
  dsyy += 2 * sxy * wdt;
  dsxy += (sxx - syy) * wdt;
  double txx = sxx + dsxx, tyy = syy + dsyy, tzz = szz + dszz, txy = sxy + dsxy;
  double I1 = txx + tyy + tzz;
  double p3 = I1 / 3;
  double s_xx = txx - p3, s_yy = tyy - p3, s_zz = tzz - p3, s_xy = txy;
  double J2 = 0.5 * (s_xx * s_xx + s_yy * s_yy + s_zz * s_zz + 2 * (s_xy * s_xy));
  double sqJ2 = sqrt(J2);
  double fy = a_phi * I1 + sqJ2 - k_c;
  double dpxx = 0, dpyy = 0, dpzz = 0, dpxy = 0;
  if (fy > 0.0) {
    double inv2 = 1.0 / (2 * sqJ2);
    double dfxx = a_phi + s_xx * inv2, dfyy = a_phi + s_yy * inv2, dfzz = a_phi + s_zz * inv2,
           dfxy = s_xy * inv2;
    double dgxx = a_psi + s_xx * inv2, dgyy = a_psi + s_yy * inv2, dgzz = a_psi + s_zz * inv2,
           dgxy = s_xy * inv2;
    double Dgxx = D0 * ((1.0 - nu) * dgxx + nu * dgyy + nu * dgzz);
    double Dgyy = D0 * (nu * dgxx + (1.0 - nu) * dgyy + nu * dgzz);
    double Dgzz = D0 * (nu * dgxx + nu * dgyy + (1.0 - nu) * dgzz);
    double Dgxy = D0 * (1.0 - 2 * nu) * dgxy;
    double denom = dfxx * Dgxx + dfyy * Dgyy + dfzz * Dgzz + 2 * dfxy * Dgxy;
    double dl = fy / denom;
    dpxx = dl * dgxx;
    dpyy = dl * dgyy;
    dpzz = dl * dgzz;
    dpxy = dl * dgxy;
    dsxx -= D0 * ((1.0 - nu) * dpxx + nu * dpyy + nu * dpzz);
    dsyy -= D0 * (nu * dpxx + (1.0 - nu) * dpyy + nu * dpzz);
    dszz -= D0 * (nu * dpxx + nu * dpyy + (1.0 - nu) * dpzz);
    dsxy -= D0 * (1.0 - 2 * nu) * dpxy;
  }
  double o0 = sxx + dsxx, o1 = syy + dsyy, o2 = szz + dszz, o3 = sxy + dsxy;
  if (sxx + dsxx + syy + dsyy + szz + dszz > k_c / a_phi) {
    double ap = k_c / a_phi / 3.0;
    o0 = ap;
    o1 = ap;
    o2 = ap;
    o3 = 0.0;
  }
  P.stress[0][g] = o0;
  P.stress[1][g] = o1;
  P.stress[2][g] = o2;
  P.stress[3][g] = o3;
  P.stress_s[0][g] = (R)o0;
  P.stress_s[1][g] = (R)o1;
  P.stress_s[2][g] = (R)o2;
  P.stress_s[3][g] = (R)o3;
  P.strain[0][g] += dexx;
  P.strain[1][g] += deyy;
  P.strain[2][g] += dezz;
  P.strain[3][g] += dexy;
  P.strainp[0][g] += dpxx;
  P.strainp[1][g] += dpyy;
  P.strainp[2][g] += dpzz;
  P.strainp[3][g] += dpxy;
}

// ViscoPlasticMCStressUpdater (:155-189).  prm = {eos_kind, rho0, gamma,
// tan(phi), cohesion}.
template <typename R>
__device__ __forceinline__ void vpmc_update(Pool<R> P, int64_t g, int NS, double p0, double p1,
                                            double p2, double p3, double p4, double c) {
  const double prm[5] = {p0, p1, p2, p3, p4};
  const double pval = eos_p((int)prm[0], P.rho_h[g], prm[1], prm[2], c);
  P.p[g] = (R)pval;
  double er[GR_MAXNS];
#pragma unroll
  for (int k = 0; k < GR_MAXNS; ++k) er[k] = k < NS ? (double)P.sr[k][g] : 0.0;
  double mag;
  if (NS == 3)
    mag = er[0] * er[0] + er[1] * er[1] + 2 * (er[2] * er[2]);
  else if (NS == 4)
    mag = er[0] * er[0] + er[1] * er[1] + 2 * (er[3] * er[3]);
  else
    mag = er[0] * er[0] + er[1] * er[1] + er[2] * er[2] +
          2 * (er[3] * er[3] + er[4] * er[4] + er[5] * er[5]);
  mag = sqrt(mag);
  if (!(mag >= 2.220446049250313e-16)) mag = isnan(mag) ? mag : 2.220446049250313e-16;
  const double sc = 2.0 * (prm[4] + pval * prm[3]);
  double sg[GR_MAXNS];
#pragma unroll
  for (int k = 0; k < GR_MAXNS; ++k) sg[k] = sc * er[k] / mag;
  bool zero;
  if (NS == 3) {
    sg[0] = sg[0] - pval;
    sg[1] = sg[1] - pval;
    sg[2] = sg[2] - 0.0;
    zero = sg[0] + sg[1] > 0.0;
  } else {
    sg[0] = sg[0] - pval;
    sg[1] = sg[1] - pval;
    sg[2] = sg[2] - pval;
#pragma unroll
    for (int k = 3; k < GR_MAXNS; ++k) sg[k] = sg[k] - 0.0;
    zero = sg[0] + sg[1] + sg[2] > 0.0;
  }
#pragma unroll
  for (int k = 0; k < GR_MAXNS; ++k)
    if (k < NS) {
      const double v = zero ? 0.0 : sg[k];
      P.stress[k][g] = v;
      P.stress_s[k][g] = (R)v;
    }
}

// The state updaters of one stage, in each system's order.  KM is the set of
// updater kinds (bit GR_UPD_x) the kernel handles: a stage is launched with
// the smallest instantiation that covers its kinds, so a stage of
// Drucker-Prager updaters does not carry the registers of the others.
template <typename R, int KM>
__global__ void k_updaters(Pool<R> P, const SysDesc *sd, const StepSys *st, const Blk *blk,
                           const int2 *urange, const UpdDesc *ud, int D, int rec) {
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int i = b.first + threadIdx.x;
  const SysDesc S = sd[s];
  if (i >= S.cap) return;
  const int64_t g0 = S.off + i;
  const int2 r = urange[s];
  const double dt = st[s].dt;
  for (int q = r.x; q < r.y; ++q) {
    const UpdDesc u = ud[q];
    // the element address of each of the ~40 arrays would otherwise be
    // hoisted out of the loop, two registers apiece (spilled): g is made
    // opaque per iteration (an empty asm statement, no instruction)
    int64_t g = g0;
    asm volatile("" : "+v"(g));
    switch (u.kind) {
      case GR_UPD_ZERO: if constexpr ((KM >> GR_UPD_ZERO) & 1) {
        const long long m = u.mask;
#pragma unroll
        for (int k = 0; k < GR_MAXNS; ++k) {
          if (k >= S.ns) continue;
          if (m & (1 << GR_F_STRAIN_RATE)) P.sr[k][g] = (R)0;
          if (m & (1 << GR_F_STRESS)) {
            P.stress[k][g] = 0.0;
            P.stress_s[k][g] = (R)0;
          }
          if (m & (1 << GR_F_STRAIN)) P.strain[k][g] = 0.0;
          if (m & (1 << GR_F_STRAIN_P)) P.strainp[k][g] = 0.0;
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          if ((m & (1 << GR_F_VORTICITY)) && k < S.nv) P.vor[k][g] = (R)0;
          if ((m & (1 << GR_F_DVDT)) && k < D) P.dvdt[k][g] = (R)0;
        }
        if (m & (1 << GR_F_DRHODT)) P.drhodt[g] = (R)0;
        if (m & (1 << GR_F_P)) P.p[g] = (R)0;
        break;
      }
      case GR_UPD_TAIT:
      case GR_UPD_LINEAR:
        if constexpr ((KM >> GR_UPD_TAIT) & 1)
          P.p[g] = (R)eos_p(u.kind, P.rho_h[g], u.prm[0], u.prm[1], S.c);
        break;
      case GR_UPD_EP:
        if constexpr ((KM >> GR_UPD_EP) & 1)
          ep_update(P, g, u.prm[0], u.prm[1], u.prm[2], u.prm[3], u.prm[4], dt);
        break;
      case GR_UPD_VPMC:
        if constexpr ((KM >> GR_UPD_VPMC) & 1)
          vpmc_update(P, g, S.ns, u.prm[0], u.prm[1], u.prm[2], u.prm[3], u.prm[4], S.c);
        break;
      case GR_UPD_HOOKE:
        if constexpr ((KM >> GR_UPD_HOOKE) & 1) hooke_update(P, g, u.prm[0], u.prm[1], dt);
        break;
      case GR_UPD_VNORM: if constexpr ((KM >> GR_UPD_VNORM) & 1) {  // VirtualNormUpdater (src/StateUpdaters.jl:74-84)
        const long long m = u.mask;
        const double w = P.wsum[g];
        const bool z = w == 0.0;
        if (m & (1 << GR_F_V)) {
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            if (d >= D) continue;
            const double val = z ? 0.0 : P.v[d][g] / w;
            const double nv = val * u.prm[d] + S.pv[d];
            P.v[d][g] = nv;
            P.vs[d][g] = (R)nv;
          }
        }
        if (m & (1 << GR_F_RHO)) {
          const double val = z ? 0.0 : P.rho[g] / w;
          P.rho[g] = val;
          P.rho_h[g] = val;
          P.rhos[g] = (R)val;
        }
        if (m & (1 << GR_F_P)) P.p[g] = (R)(z ? 0.0 : (double)P.p[g] / w);
        if (m & (1 << GR_F_STRESS)) {
#pragma unroll
          for (int k = 0; k < GR_MAXNS; ++k) {
            if (k >= S.ns) continue;
            const double val = z ? 0.0 : P.stress[k][g] / w;
            P.stress[k][g] = val;
            P.stress_s[k][g] = (R)val;
          }
        }
        break;
      }
      case GR_UPD_PRESCRIBED_V: if constexpr ((KM >> GR_UPD_PRESCRIBED_V) & 1) {
        // PrescribedVelocityUpdater (:88-92)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          if (d >= D) continue;
          const double nv = P.v[d][g] + S.pv[d];
          P.v[d][g] = nv;
          P.vs[d][g] = (R)nv;
        }
        break;
      }
      default:
        break;
    }
  }
  if (rec >= 0) {  // the partner records of the updated particle
    Rec<R> w;
    rec_load(P, S, g0, D, rec, w);
    rec_store(P, g0, D, rec, w);
  }
}

// Virtual systems: mode 0 refreshes the shadows of velocity and density
// after the sort, then clears w_sum and the zero fields before the stage
// loop (auto_zero_virtual!, src/Particles.jl:521-528); mode 1 advances the
// positions by prescribed_v·dt (_update_virtual_positions!,
// src/TimeIntegration.jl:389-397).
template <typename R, int D>
__global__ void k_virtual(Pool<R> P, const SysDesc *sd, const StepSys *st, const int *n_dev,
                          const Blk *blk, int mode) {
  const Blk b = blk[blockIdx.x];
  const int s = b.item;
  const int i = b.first + threadIdx.x;
  if (i >= n_dev[s]) return;
  const SysDesc S = sd[s];
  const int64_t g = S.off + i;
  if (mode == 1) {
    const double dt = st[s].dt;
#pragma unroll
    for (int d = 0; d < D; ++d) P.x[d][g] = P.x[d][g] + S.pv[d] * dt;
    return;
  }
  // the sort moved the masters; the single-copy shadows follow them
#pragma unroll
  for (int d = 0; d < D; ++d) P.vs[d][g] = (R)P.v[d][g];
  P.rhos[g] = (R)P.rho[g];
  P.rho_h[g] = P.rho[g];
  P.wsum[g] = 0.0;
  const long long m = S.zero_mask;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    if (m & (1 << GR_F_V)) {
      P.v[d][g] = 0.0;
      P.vs[d][g] = (R)0;
    }
    if (m & (1 << GR_F_DVDT)) P.dvdt[d][g] = (R)0;
  }
  if (m & (1 << GR_F_RHO)) {
    P.rho[g] = 0.0;
    P.rho_h[g] = 0.0;
    P.rhos[g] = (R)0;
  }
  if (m & (1 << GR_F_DRHODT)) P.drhodt[g] = (R)0;
  if (m & (1 << GR_F_P)) P.p[g] = (R)0;
  if (m & (1 << GR_F_COUNT)) P.pcnt[g] = 0.0;
#pragma unroll
  for (int k = 0; k < GR_MAXNS; ++k) {
    if (k >= S.ns) continue;
    if (m & (1 << GR_F_STRESS)) {
      P.stress[k][g] = 0.0;
      P.stress_s[k][g] = (R)0;
    }
    if (m & (1 << GR_F_STRAIN_RATE)) P.sr[k][g] = (R)0;
    if (m & (1 << GR_F_STRAIN)) P.strain[k][g] = 0.0;
    if (m & (1 << GR_F_STRAIN_P)) P.strainp[k][g] = 0.0;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if ((m & (1 << GR_F_VORTICITY)) && k < S.nv) P.vor[k][g] = (R)0;
}

// ---------------------------------------------------------------------------
// Small utilities
// ---------------------------------------------------------------------------

__global__ void k_fill_i32(int *p, int v, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Fields between the caller's layout (particle-major, staged in pinned host memory)
// and the pool's component arrays: element e of `host` is component e % nc of
// particle e / nc.  The kernels read and write the host memory over the bus
// themselves, so a transfer is one launch, in whole lines both ways.
template <typename W>
__global__ void __launch_bounds__(GR_BLOCK)
    k_field_in(const W *host, int64_t count, int nc, int64_t cap, int64_t off, FieldSets F) {
  const int64_t e = (int64_t)blockIdx.x * GR_BLOCK + threadIdx.x;
  if (e >= count) return;
  const W v = host[e];
  const int64_t at = (e % nc) * cap + off + e / nc;
  for (int q = 0; q < F.n; ++q) {
    if (F.esz[q] == 8)
      static_cast<double *>(F.p[q])[at] = v;
    else
      static_cast<float *>(F.p[q])[at] = (float)v;
  }
}
template <typename W>
__global__ void __launch_bounds__(GR_BLOCK)
    k_field_out(W *host, int64_t count, int nc, int64_t cap, int64_t off, FieldSets F) {
  const int64_t e = (int64_t)blockIdx.x * GR_BLOCK + threadIdx.x;
  if (e >= count) return;
  const int64_t at = (e % nc) * cap + off + e / nc;
  host[e] = F.esz[0] == 8 ? (W)static_cast<const double *>(F.p[0])[at]
                          : (W)static_cast<const float *>(F.p[0])[at];
}
__global__ void __launch_bounds__(GR_BLOCK) k_copy_i32(const int *src, int64_t count, int *dst) {
  const int64_t e = (int64_t)blockIdx.x * GR_BLOCK + threadIdx.x;
  if (e < count) dst[e] = src[e];
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------

static inline unsigned nb_of(long long n, int per) { return (unsigned)((n + per - 1) / per); }

void launch_key_minmax(hipStream_t s, XP xs, const SysDesc *sd, const int *n, const Blk *blk,
                       int nblk, int D, long long *bbmin, long long *bbmax, int rs,
                       const int *list, int nlist, bool fold, int *flags) {
  if (nblk > 0) {
    // 8 table entries (2048 particles) per workgroup: enough workgroups to
    // fill the chip, few enough that the per-system atomics stay cheap
    constexpr int per = 8;
    const unsigned g = nb_of(nblk, per);
    if (D == 2)
      k_key_minmax<2, per><<<g, GR_BLOCK, 0, s>>>(xs, sd, n, blk, nblk, bbmin, bbmax, rs, flags);
    else
      k_key_minmax<3, per><<<g, GR_BLOCK, 0, s>>>(xs, sd, n, blk, nblk, bbmin, bbmax, rs, flags);
  }
  if (fold && nlist > 0)
    k_bb_fold<<<nb_of(nlist * 3, GR_BLOCK), GR_BLOCK, 0, s>>>(list, nlist, bbmin, bbmax, rs);
}
void launch_minmax_reset(hipStream_t s, const int *list, int nlist, long long *bbmin,
                         long long *bbmax, int rs) {
  if (nlist > 0)
    k_minmax_reset<<<nb_of(nlist * 3 * GR_BB_REP, GR_BLOCK), GR_BLOCK, 0, s>>>(list, nlist, bbmin,
                                                                               bbmax, rs);
}
void launch_key_base(hipStream_t s, const int *list, int nlist, int D, int pad, const int *n,
                     const StepSys *st, long long *bbmin, long long *bbmax, int rs, int *kmin,
                     int *kmax, unsigned *kbase, unsigned *krange, int *flags, int *sysfault) {
  k_key_base<<<1, KB_THREADS, 0, s>>>(list, nlist, D, pad, n, st, bbmin, bbmax, rs, kmin, kmax,
                                      kbase, krange, flags, sysfault, nullptr);
}
static int cells_prep_blocks(const CellsArgs &A) { return nb_of(A.n_inter, GR_BLOCK) + A.ncblk; }
void launch_cells_prep(hipStream_t s, const CellsArgs &A, int *flags, int *sysfault) {
  if (A.n_inter > 0) k_cells_prep<<<cells_prep_blocks(A), GR_BLOCK, 0, s>>>(A, flags, sysfault);
}
size_t key_table_bytes(int64_t ntile) {
  return (size_t)ntile * (KT_TILE * 2 + KT_REP) * sizeof(unsigned);
}
int key_table_tile() { return KT_TILE; }
void launch_key_sort(hipStream_t s, XP xs, const SysDesc *sd, const int *n, const StepSys *st,
                     const Blk *blk, int nblk, const int *bbase, int D, const int *list, int nlist,
                     int N, long long *bbmin, long long *bbmax, int rs, int *kmin, int *kmax,
                     unsigned *krange, unsigned *kbase, int *kshift, unsigned *keys,
                     unsigned *full, unsigned *keys2, int *vals2, unsigned *rank,
                     int *flags, int *sysfault, int *run, unsigned *table, int tiles, int ntile,
                     const CellsArgs *cells) {
  if (nblk <= 0) {
    if (cells) launch_cells_prep(s, *cells, flags, sysfault);
    return;
  }
  unsigned *count = table, *start = table + (size_t)tiles * KT_TILE;
  unsigned *tsum = table + (size_t)tiles * KT_TILE * 2;
  const int inl = nlist <= KC_SYSTEMS && nblk <= KC_BLOCKS;
  if (!inl)
    k_key_base<<<1, KB_THREADS, 0, s>>>(list, nlist, D, 0, n, st, bbmin, bbmax, rs, kmin, kmax,
                                        kbase, krange, flags, sysfault, kshift);
  auto go = [&](auto dc) {
    k_key_count<decltype(dc)::value><<<nblk, GR_BLOCK, 0, s>>>(
        xs, sd, n, st, blk, bbase, list, nlist, bbmin, bbmax, rs, kmin, kmax, krange, kbase, kshift,
        keys, full, rank, flags, sysfault, count, tsum, inl);
  };
  if (D == 2)
    go(std::integral_constant<int, 2>{});
  else
    go(std::integral_constant<int, 3>{});
  k_key_scan<<<ntile, GR_BLOCK, 0, s>>>(count, tsum, start, flags);
  const CellsArgs A = cells ? *cells : CellsArgs{};
  const int nprep = cells_prep_blocks(A);
  k_key_place<<<nblk + nprep, GR_BLOCK, 0, s>>>(sd, n, blk, bbase, keys, full, kshift, keys2, vals2,
                                                rank, start, tsum, ntile, N, list, nlist, bbmin,
                                                bbmax, rs, flags, nprep, A, sysfault, run);
}
void launch_key_write(hipStream_t s, XP xs, const SysDesc *sd, const int *n, const StepSys *st,
                      const Blk *blk, int nblk, const int *bbase, int D, const int *kmin,
                      const unsigned *krange, const unsigned *kbase, unsigned *keys, int *vals,
                      int *flags, unsigned *rscr) {
  if (nblk <= 0) return;
  if (D == 2)
    k_key_write<2><<<nblk, GR_BLOCK, 0, s>>>(xs, sd, n, st, blk, bbase, kmin, krange, kbase, keys,
                                             vals, flags, rscr);
  else
    k_key_write<3><<<nblk, GR_BLOCK, 0, s>>>(xs, sd, n, st, blk, bbase, kmin, krange, kbase, keys,
                                             vals, flags, rscr);
}
void launch_radix_sort(hipStream_t s, unsigned *keys, int *vals, unsigned *keys2, int *vals2,
                       unsigned *rscr, int N, int *flags) {
  if (N <= 0) return;
  const unsigned ntile = nb_of(N, OS_TILE);
  for (int pass = 0; pass < 4; ++pass) {
    const bool even = (pass & 1) == 0;
    k_radix_scan<<<256, GR_BLOCK, 0, s>>>(N, pass, rscr, flags);
    k_radix_scatter<<<ntile, GR_BLOCK, 0, s>>>(even ? keys : keys2, even ? vals : vals2,
                                               even ? keys2 : keys, even ? vals2 : vals, N, pass,
                                               rscr, flags);
  }
}
size_t radix_scratch_bytes(int N) {
  const size_t ntile = nb_of(N > 0 ? N : 1, OS_TILE);
  return ((size_t)RS_CNT + 2 * ntile * 256) * 4;
}

template <typename R>
void launch_permute_real(hipStream_t s, const Pool<R> &A, const Pool<R> &B, const SysDesc *sd,
                         const Blk *blk, int nblk, const int *bbase, const int *vals,
                         const int *vals2, const int *flags, int vadj, int D, const StepSys *st,
                         const int *halfsys, int pack, const KeyTable *kt) {
  if (nblk <= 0) return;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  using P2 = std::integral_constant<int, 2>;
  auto go = [&](auto dc, auto pc, auto hc, auto tc) {
    constexpr int DD = decltype(dc)::value, PP = decltype(pc)::value;
    constexpr bool H = decltype(hc)::value, T = decltype(tc)::value;
    k_permute_real<R, DD, H, PP, T><<<nblk, GR_BLOCK, 0, s>>>(
        A, B, sd, blk, bbase, vals, vals2, flags, vadj, st, halfsys, kt ? *kt : KeyTable{});
  };
  auto tab = [&](auto dc, auto pc, auto hc) {
    if (kt)
      go(dc, pc, hc, std::true_type{});
    else
      go(dc, pc, hc, std::false_type{});
  };
  auto dim = [&](auto pc, auto hc) {
    if (D == 2)
      tab(I2{}, pc, hc);
    else
      tab(I3{}, pc, hc);
  };
  if (sizeof(R) != 4) pack = 0;
  if (!halfsys)
    dim(P0{}, std::false_type{});
  else if (pack == 2)
    dim(P2{}, std::true_type{});
  else if (pack == 1)
    dim(P1{}, std::true_type{});
  else
    dim(P0{}, std::true_type{});
}
template void launch_permute_real<float>(hipStream_t, const Pool<float> &, const Pool<float> &,
                                         const SysDesc *, const Blk *, int, const int *,
                                         const int *, const int *, const int *, int, int,
                                         const StepSys *, const int *, int, const KeyTable *);
template void launch_permute_real<double>(hipStream_t, const Pool<double> &,
                                          const Pool<double> &, const SysDesc *, const Blk *,
                                          int, const int *, const int *, const int *, const int *,
                                          int, int, const StepSys *, const int *, int,
                                          const KeyTable *);

void launch_ghost_count(hipStream_t s, XP x, const SysDesc *sd, const Bnd *bnd, const Blk *blk,
                        int nblk, const int *gslot, int D, int *cnt, int *flags) {
  if (nblk <= 0) return;
  if (D == 2)
    k_ghost_count<2><<<nblk, GR_BLOCK, 0, s>>>(x, sd, bnd, blk, gslot, cnt, flags);
  else
    k_ghost_count<3><<<nblk, GR_BLOCK, 0, s>>>(x, sd, bnd, blk, gslot, cnt, flags);
}
void launch_scan(hipStream_t s, const int *in, int *out, int *bsum, int N) {
  const int nb = (int)nb_of(N > 0 ? N : 1, SCAN_TILE);
  k_scan_local<<<nb, 256, 0, s>>>(in, out, bsum, N);
  k_scan_blocks<<<1, 1024, 0, s>>>(bsum, nb, out, N);
  k_scan_add<<<nb, 256, 0, s>>>(out, bsum, N);
}
int scan_block_count(int N) { return (int)nb_of(N > 0 ? N : 1, SCAN_TILE); }
void launch_ghost_scatter(hipStream_t s, XP x, XPW gx, int *gidx, int *gbnd, int *gnrm,
                          const SysDesc *sd, const Bnd *bnd, const Blk *blk, int nblk,
                          const int *gslot, const int *cnt, const int *scan, int D, int *n,
                          long long *bbmin, long long *bbmax, int rs) {
  if (nblk <= 0) return;
  if (D == 2)
    k_ghost_scatter<2><<<nblk, GR_BLOCK, 0, s>>>(x, gx, gidx, gbnd, gnrm, sd, bnd, blk, gslot,
                                                 cnt, scan, n, bbmin, bbmax, rs);
  else
    k_ghost_scatter<3><<<nblk, GR_BLOCK, 0, s>>>(x, gx, gidx, gbnd, gnrm, sd, bnd, blk, gslot,
                                                 cnt, scan, n, bbmin, bbmax, rs);
}
void launch_permute_ghost(hipStream_t s, XP gxs, const int *gidx_s, const int *gbnd_s, XPW x,
                          int *gidx, int *gbnd, const SysDesc *sd, const int *n, const Blk *blk,
                          int nblk, const int *bbase, const int *vals, const int *vals2,
                          const int *flags, int D, const KeyTable *kt) {
  if (nblk <= 0) return;
  auto go = [&](auto dc, auto tc) {
    k_permute_ghost<decltype(dc)::value, decltype(tc)::value><<<nblk, GR_BLOCK, 0, s>>>(
        gxs, gidx_s, gbnd_s, x, gidx, gbnd, sd, n, blk, bbase, vals, vals2, flags,
        kt ? *kt : KeyTable{});
  };
  auto dim = [&](auto tc) {
    if (D == 2)
      go(std::integral_constant<int, 2>{}, tc);
    else
      go(std::integral_constant<int, 3>{}, tc);
  };
  if (kt)
    dim(std::true_type{});
  else
    dim(std::false_type{});
}
template <typename R>
void launch_ghost_kin(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const Bnd *bnd,
                      const int *n, const Blk *blk, int nblk, int D) {
  if (nblk <= 0) return;
  k_ghost_kin<R><<<nblk, GR_BLOCK, 0, s>>>(P, sd, bnd, n, blk, D);
}
template void launch_ghost_kin<float>(hipStream_t, const Pool<float> &, const SysDesc *,
                                      const Bnd *, const int *, const Blk *, int, int);
template void launch_ghost_kin<double>(hipStream_t, const Pool<double> &, const SysDesc *,
                                       const Bnd *, const int *, const Blk *, int, int);
template <typename R>
void launch_ghost_copy(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const Bnd *bnd,
                       const int *n, const Blk *blk, int nblk, const int2 *copy, int D) {
  (void)D;
  if (nblk > 0) k_ghost_copy<R><<<nblk, GR_BLOCK, 0, s>>>(P, sd, bnd, n, blk, copy);
}
template void launch_ghost_copy<float>(hipStream_t, const Pool<float> &, const SysDesc *,
                                       const Bnd *, const int *, const Blk *, int, const int2 *,
                                       int);
template void launch_ghost_copy<double>(hipStream_t, const Pool<double> &, const SysDesc *,
                                        const Bnd *, const int *, const Blk *, int,
                                        const int2 *, int);

int64_t cell_tiles(int64_t cells) { return (cells + CELL_TILE - 1) / CELL_TILE; }
void launch_cells_build(hipStream_t s, XP x, const CellsArgs &A, const SysDesc *sd, const Blk *mblk,
                        int nmblk) {
  if (nmblk > 0) {
    if (A.D == 2)
      k_cells_mark<2><<<nmblk, GR_BLOCK, 0, s>>>(x, A.cells, A.tflag, A.carr, A.grids, A.cellsz, sd,
                                                 A.n_dev, mblk);
    else
      k_cells_mark<3><<<nmblk, GR_BLOCK, 0, s>>>(x, A.cells, A.tflag, A.carr, A.grids, A.cellsz, sd,
                                                 A.n_dev, mblk);
  }
  if (A.ncblk > 0)
    k_cells_fill<<<A.ncblk, GR_BLOCK, 0, s>>>(A.cells, A.tflag, A.carr, A.grids, A.n_dev, A.cblk);
}

template <typename R>
void launch_halfstep(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                     const Blk *blk, int nblk, int D, double mult, int keep) {
  if (nblk <= 0) return;
  if (D == 2)
    k_halfstep<R, 2><<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, blk, mult, keep);
  else
    k_halfstep<R, 3><<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, blk, mult, keep);
}
template <typename R>
void launch_rk4_acc(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                    const Blk *blk, int nblk, int D, double w, int first) {
  if (nblk <= 0) return;
  if (D == 2)
    k_rk4_acc<R, 2><<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, blk, w, first);
  else
    k_rk4_acc<R, 3><<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, blk, w, first);
}
template <typename F>
static void dispatch_bb(int D, bool bb, F go) {
  using T = std::true_type;
  using N = std::false_type;
  if (D == 2)
    bb ? go(std::integral_constant<int, 2>{}, T{}) : go(std::integral_constant<int, 2>{}, N{});
  else
    bb ? go(std::integral_constant<int, 3>{}, T{}) : go(std::integral_constant<int, 3>{}, N{});
}
template <typename R>
void launch_rk4_apply(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                      const Blk *blk, int nblk, int D, int pos, const StepBounds *bb) {
  if (nblk <= 0) return;
  const StepBounds B = bb ? *bb : StepBounds{};
  dispatch_bb(D, bb != nullptr, [&](auto d, auto q) {
    k_rk4_apply<R, decltype(d)::value, decltype(q)::value>
        <<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, blk, pos, B);
  });
}
template <typename R>
void launch_fullstep(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                     const Blk *blk, int nblk, int D, int pos, const StepBounds *bb) {
  if (nblk <= 0) return;
  const StepBounds B = bb ? *bb : StepBounds{};
  dispatch_bb(D, bb != nullptr, [&](auto d, auto q) {
    k_fullstep<R, decltype(d)::value, decltype(q)::value>
        <<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, blk, pos, B);
  });
}
template <typename R>
void launch_xsph(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                 const int *n, const Blk *blk, int nblk, int D, int mode) {
  if (nblk <= 0) return;
  if (D == 2)
    k_xsph<R, 2><<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, n, blk, mode);
  else
    k_xsph<R, 3><<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, n, blk, mode);
}
template <typename R>
void launch_updaters(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                     const Blk *blk, int nblk, const int2 *urange, const UpdDesc *ud, int D,
                     int kinds, int rec) {
  if (nblk <= 0) return;
  constexpr int Z = 1 << GR_UPD_ZERO | 1 << GR_UPD_NOTHING;
  constexpr int K_EP = Z | 1 << GR_UPD_EP, K_VPMC = Z | 1 << GR_UPD_VPMC,
                K_EOS = Z | 1 << GR_UPD_TAIT | 1 << GR_UPD_LINEAR, K_HOOKE = Z | 1 << GR_UPD_HOOKE;
  auto go = [&](auto km) {
    k_updaters<R, decltype(km)::value><<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, blk, urange, ud, D,
                                                              rec);
  };
  if ((kinds & ~K_EP) == 0)
    go(std::integral_constant<int, K_EP>{});
  else if ((kinds & ~K_VPMC) == 0)
    go(std::integral_constant<int, K_VPMC>{});
  else if ((kinds & ~K_EOS) == 0)
    go(std::integral_constant<int, K_EOS>{});
  else if ((kinds & ~K_HOOKE) == 0)
    go(std::integral_constant<int, K_HOOKE>{});
  else
    go(std::integral_constant<int, -1>{});
}
#define INST(R)                                                                                \
  template void launch_halfstep<R>(hipStream_t, const Pool<R> &, const SysDesc *,              \
                                   const StepSys *, const Blk *, int, int, double, int);       \
  template void launch_rk4_acc<R>(hipStream_t, const Pool<R> &, const SysDesc *,               \
                                  const StepSys *, const Blk *, int, int, double, int);        \
  template void launch_rk4_apply<R>(hipStream_t, const Pool<R> &, const SysDesc *,             \
                                    const StepSys *, const Blk *, int, int, int,               \
                                    const StepBounds *);                                       \
  template void launch_fullstep<R>(hipStream_t, const Pool<R> &, const SysDesc *,              \
                                   const StepSys *, const Blk *, int, int, int,                \
                                   const StepBounds *);                                        \
  template void launch_xsph<R>(hipStream_t, const Pool<R> &, const SysDesc *, const StepSys *, \
                               const int *, const Blk *, int, int, int);                       \
  template void launch_updaters<R>(hipStream_t, const Pool<R> &, const SysDesc *,              \
                                   const StepSys *, const Blk *, int, const int2 *,            \
                                   const UpdDesc *, int, int, int);
INST(float)
INST(double)
#undef INST

template <typename W>
void launch_field(hipStream_t s, bool in, W *host, int64_t count, int nc, int64_t cap, int64_t off,
                  const FieldSets &F) {
  if (count <= 0) return;
  if (in)
    k_field_in<W><<<nb_of(count, GR_BLOCK), GR_BLOCK, 0, s>>>(host, count, nc, cap, off, F);
  else
    k_field_out<W><<<nb_of(count, GR_BLOCK), GR_BLOCK, 0, s>>>(host, count, nc, cap, off, F);
}
template void launch_field<float>(hipStream_t, bool, float *, int64_t, int, int64_t, int64_t,
                                  const FieldSets &);
template void launch_field<double>(hipStream_t, bool, double *, int64_t, int, int64_t, int64_t,
                                   const FieldSets &);
void launch_index(hipStream_t s, bool in, int *host, int64_t count, int *dev) {
  if (count > 0)
    k_copy_i32<<<nb_of(count, GR_BLOCK), GR_BLOCK, 0, s>>>(in ? host : dev, count, in ? dev : host);
}

template <typename R>
void launch_virtual(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const StepSys *st,
                    const int *n, const Blk *blk, int nblk, int mode, int D) {
  if (nblk <= 0) return;
  if (D == 2)
    k_virtual<R, 2><<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, n, blk, mode);
  else
    k_virtual<R, 3><<<nblk, GR_BLOCK, 0, s>>>(P, sd, st, n, blk, mode);
}
template void launch_virtual<float>(hipStream_t, const Pool<float> &, const SysDesc *,
                                    const StepSys *, const int *, const Blk *, int, int, int);
template void launch_virtual<double>(hipStream_t, const Pool<double> &, const SysDesc *,
                                     const StepSys *, const int *, const Blk *, int, int, int);

template <typename R>
void launch_pack(hipStream_t s, const Pool<R> &P, const SysDesc *sd, const int *n, const Blk *blk,
                 int nblk, int mode, const Blk *gblk, int ngblk, int gmode, const Bnd *bnd,
                 const int2 *copy, bool kin, int D) {
  if (nblk + ngblk > 0)
    k_pack<R><<<nblk + ngblk, GR_BLOCK, 0, s>>>(P, sd, n, blk, nblk, mode, gblk, gmode, bnd, copy,
                                                kin ? 1 : 0, D);
}
template void launch_pack<float>(hipStream_t, const Pool<float> &, const SysDesc *, const int *,
                                 const Blk *, int, int, const Blk *, int, int, const Bnd *,
                                 const int2 *, bool, int);
template void launch_pack<double>(hipStream_t, const Pool<double> &, const SysDesc *, const int *,
                                  const Blk *, int, int, const Blk *, int, int, const Bnd *,
                                  const int2 *, bool, int);

// Probe slot id[i] − 1 takes the position of mirror particle i
// (_measure_probes!, src/TimeIntegration.jl:469-479).
template <typename R, int D>
__global__ void k_probe_mirror(Pool<R> P, const SysDesc *sd, int probe, int src) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const SysDesc Sp = sd[probe], Ss = sd[src];
  if (i >= Ss.cap) return;
  const int q = P.id[Ss.off + i] - 1;
  if (q < 0 || q >= Sp.cap) return;
#pragma unroll
  for (int d = 0; d < D; ++d) P.x[d][Sp.off + q] = P.x[d][Ss.off + i];
}

// _sort_probe_by_id! (src/ProbeParticles.jl:150-158): ids are 1..n, so the
// sort is the scatter slot i -> id[i] − 1, done through a scratch copy:
// mode 0 scatters the probe's fields into scr (ncol columns of n doubles),
// mode 1 copies them back and refreshes the shadows.
template <typename R, int D>
__global__ void k_probe_by_id(Pool<R> P, const SysDesc *sd, int probe, double *scr, int mode) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const SysDesc S = sd[probe];
  const int64_t n = S.cap;
  if (i >= n) return;
  const int64_t g = S.off + i;
  const int ns = S.kind >= GR_SYS_STRESS ? S.ns : 0;
  if (mode == 0) {
    const int64_t q = (int64_t)P.id[g] - 1;
    if (q < 0 || q >= n) return;
    int col = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) scr[(col++) * n + q] = P.x[d][g];
#pragma unroll
    for (int d = 0; d < D; ++d) scr[(col++) * n + q] = P.v[d][g];
    scr[(col++) * n + q] = P.rho[g];
    scr[(col++) * n + q] = P.wsum[g];
    scr[(col++) * n + q] = P.pcnt[g];
    scr[(col++) * n + q] = S.kind >= GR_SYS_FLUID ? (double)P.p[g] : 0.0;
    for (int k = 0; k < ns; ++k) scr[(col++) * n + q] = P.stress[k][g];
    return;
  }
  int col = 0;
#pragma unroll
  for (int d = 0; d < D; ++d) P.x[d][g] = scr[(col++) * n + i];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const double v = scr[(col++) * n + i];
    P.v[d][g] = v;
    P.vs[d][g] = (R)v;
  }
  const double rho = scr[(col++) * n + i];
  P.rho[g] = rho;
  P.rho_h[g] = rho;
  P.rhos[g] = (R)rho;
  P.wsum[g] = scr[(col++) * n + i];
  P.pcnt[g] = scr[(col++) * n + i];
  const double p = scr[(col++) * n + i];
  if (S.kind >= GR_SYS_FLUID) P.p[g] = (R)p;
  for (int k = 0; k < ns; ++k) {
    const double sg = scr[(col++) * n + i];
    P.stress[k][g] = sg;
    P.stress_s[k][g] = (R)sg;
  }
  P.id[g] = (int)(i + 1);
}

template <typename R>
void launch_probe_mirror(hipStream_t s, const Pool<R> &P, const SysDesc *sd, int probe, int src,
                         int64_t n_src, int D) {
  if (n_src <= 0) return;
  const unsigned nb = (unsigned)((n_src + GR_BLOCK - 1) / GR_BLOCK);
  if (D == 2)
    k_probe_mirror<R, 2><<<nb, GR_BLOCK, 0, s>>>(P, sd, probe, src);
  else
    k_probe_mirror<R, 3><<<nb, GR_BLOCK, 0, s>>>(P, sd, probe, src);
}
template <typename R>
void launch_probe_by_id(hipStream_t s, const Pool<R> &P, const SysDesc *sd, int probe, int64_t n,
                        double *scr, int mode, int D) {
  if (n <= 0) return;
  const unsigned nb = (unsigned)((n + GR_BLOCK - 1) / GR_BLOCK);
  if (D == 2)
    k_probe_by_id<R, 2><<<nb, GR_BLOCK, 0, s>>>(P, sd, probe, scr, mode);
  else
    k_probe_by_id<R, 3><<<nb, GR_BLOCK, 0, s>>>(P, sd, probe, scr, mode);
}
template void launch_probe_mirror<float>(hipStream_t, const Pool<float> &, const SysDesc *, int,
                                         int, int64_t, int);
template void launch_probe_mirror<double>(hipStream_t, const Pool<double> &, const SysDesc *, int,
                                          int, int64_t, int);
template void launch_probe_by_id<float>(hipStream_t, const Pool<float> &, const SysDesc *, int,
                                        int64_t, double *, int, int);
template void launch_probe_by_id<double>(hipStream_t, const Pool<double> &, const SysDesc *, int,
                                         int64_t, double *, int, int);

// A ghost-target XSPH task stores into its source's v_adjustment at the
// ghost's index: flag (bit 4 of flags[1]) a ghost count above the source's.
__global__ void k_alias_check(const int *n_dev, int ghost, int src_n, int *flags) {
  if (threadIdx.x == 0 && n_dev[ghost] > src_n) atomicOr(&flags[1], 4);
}
void launch_alias_check(hipStream_t s, const int *n, int ghost, int src_n, int *flags) {
  k_alias_check<<<1, 64, 0, s>>>(n, ghost, src_n, flags);
}

void launch_fill_i32(hipStream_t s, int *p, int v, long long n) {
  if (n > 0) k_fill_i32<<<nb_of(n, GR_BLOCK), GR_BLOCK, 0, s>>>(p, v, n);
}

}  // namespace gr
