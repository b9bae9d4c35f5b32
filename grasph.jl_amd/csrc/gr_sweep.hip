// gr_sweep.hip — neighbour search and fused pair-functor gather (gfx950).
//
// The reference visits each unordered pair once (half-shell colour sweep,
// src/Interaction.jl:393-541) and writes to both particles; the coupled sweep
// (:600-715) writes to system_a and, for two-sided functors, system_b.  Here
// every target particle instead gathers all its partners over the 3^D
// neighbour cells of each interaction it takes part in, evaluates the
// functor from its own side (which equals the reference's update of that
// particle: the pair formulas are antisymmetric/symmetric under i <-> j),
// accumulates in registers (FP64 sums of the pair terms) and writes once.  No
// atomics; the result is independent of scheduling.
//
// Two passes per step:
//  * k_nlist: neighbour search.  A wavefront stages the candidates of each
//    strip in LDS with coalesced loads and each lane keeps the candidates
//    in its own CSR ranges with r² < (2h)², evaluated in FP64 in the
//    reference's order, so the accepted pair set equals the reference's.
//  * k_sweep_list: the functors over each lane's accepted partners, once per
//    stage, so every lane does useful arithmetic on every iteration.  The
//    FP32 fluid-only force sweep reads 32-byte compact partner records
//    (fixed-point positions, see RecC) with two loads per pair.
// k_sweep walks the cells directly (fine-grained sweep! calls, and targets
// whose list overflowed).
#include <hip/hip_runtime.h>

#include "../../include/grasph_hip.h"
#include "gr_device.h"
#include "gr_launch.h"

namespace gr {

// Per-target sums of the pair terms, in FP64 whatever the arithmetic type of
// the terms: one conversion and one add per term (FP64 adds issue at the FP32
// rate), rounded to R once when stored.
template <typename R>
struct Acc {
  double s = 0;
  __device__ inline void add(R v) { s += (double)v; }
  __device__ inline R get() const { return (R)s; }
};
template <>
struct Acc<double> {
  double s = 0;
  __device__ inline void add(double v) { s += v; }
  __device__ inline double get() const { return s; }
};

// One pair's term instead of a sum (k_sweep_split adds the terms of several
// lanes in order).
template <typename R>
struct Term {
  R t = 0;
  __device__ inline void add(R v) { t = v; }
  __device__ inline R get() const { return t; }
};

// Julia's ^(Float64, Integer) for the LJ powers in FP64; plain products in FP32.
__device__ inline double pow_i(double x, int n) {
  double y = 1.0, xnlo = 0.0, ynlo = 0.0;
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
__device__ inline float pow_i(float x, int n) {
  float x2 = x * x, x3 = x2 * x, x6 = x3 * x3;
  if (n == 4) return x2 * x2;
  return n == 12 ? x6 * x6 : x6;
}

// kernel_dw_dq (src/Kernels.jl:79-81 cubic, :151-153 Wendland C2).
template <typename R>
__device__ inline R dwdq(int kk, R C, R q) {
  if (kk == GR_KERNEL_CUBIC) {
    R t2 = (R)2 - q, t1 = (R)1 - q;
    t2 = t2 > (R)0 ? t2 : (R)0;
    t1 = t1 > (R)0 ? t1 : (R)0;
    return C * ((R)-3 * ((R)0.25 * (t2 * t2) - t1 * t1));
  }
  R t = (R)2 - q;
  t = t > (R)0 ? t : (R)0;
  return ((-C * (R)10) * q) * (t * t * t);
}

// Reciprocals.  FP32 pair math uses the hardware reciprocal and reciprocal
// square root (1 ulp) and reuses each reciprocal within a pair; FP64 keeps
// correctly rounded division and square root.
template <typename R>
struct Fast;
template <>
struct Fast<float> {
  static constexpr bool on = true;
  __device__ static inline float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
  __device__ static inline float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
};
template <>
struct Fast<double> {
  static constexpr bool on = false;
  __device__ static inline double rcp(double x) { return 1.0 / x; }
  __device__ static inline double rsq(double x) { return 1.0 / sqrt(x); }
};

// kernel_w (src/Kernels.jl:70-72 cubic, :142-144 Wendland C2).
template <typename R>
__device__ inline R wq(int kk, R C, R q) {
  if (kk == GR_KERNEL_CUBIC) {
    R t2 = (R)2 - q, t1 = (R)1 - q;
    t2 = t2 > (R)0 ? t2 : (R)0;
    t1 = t1 > (R)0 ? t1 : (R)0;
    return C * ((R)0.25 * (t2 * t2 * t2) - t1 * t1 * t1);
  }
  R t = (R)2 - q;
  t = t > (R)0 ? t : (R)0;
  return (C * pow_i(t, 4)) * ((R)2 * q + (R)1);
}

template <typename R>
__device__ inline R jmin0(R v) {  // Julia min(v, 0)
  return v < (R)0 ? v : (isnan(v) ? v : (R)0);
}

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous run of logical blocks so neighbouring cells share an L2.
__device__ inline int xcd_block(int nblk) {
  const int b = blockIdx.x;
  const int full = (nblk / 8) * 8;
  if (b >= full) return b;
  return (b % 8) * (nblk / 8) + b / 8;
}

// Per-source constants in the arithmetic type.
template <typename R>
struct SrcK {
  R h, ih, norm, hf, alpha, beta, mc, h2, m_q, psi_coef, eps, ljcut, ljc2;
  int sigma, has_delta, has_eps;
  __device__ inline void load(const SrcDesc &Q) {
    h = (R)Q.h;
    ih = (R)(1.0 / Q.h);
    norm = (R)Q.norm;
    hf = (R)Q.hf;
    alpha = (R)Q.alpha;
    beta = (R)Q.beta;
    mc = (R)(0.5 * (Q.c_t_piv + Q.c_q_piv));
    h2 = (R)(Q.hf * Q.hf * 0.01);
    m_q = (R)Q.mass_q;
    psi_coef = (R)(2.0 * Q.delta * (0.5 * (Q.c_t_psi + Q.c_q_psi)) * Q.hf);
    eps = (R)Q.eps;
    ljcut = (R)Q.ljcut;
    ljc2 = (R)(0.01 * Q.c_t_piv * Q.c_t_piv);
    sigma = Q.sigma;
    has_delta = Q.has_delta;
    has_eps = Q.has_eps;
  }
};

// FORCE family specialised for stages whose force functors are all FluidPfn
// or FluidSolidPfn (no stress-based functor): the Cauchy branch and the
// target's stress are compiled out.  A template argument only, not a task
// family.
constexpr int FAM_FORCE_FLUID = NFAM + 1;
// The same for FluidPfn with S = 2, no δ-SPH and no surface tension, whose
// partner records hold 1/ρ and p/ρ² in place of ρ and p (k_pack INV): the
// reciprocal and the products the pair would compute are done once per
// particle, with the same FP32 operations, so the sums are unchanged.
constexpr int FAM_FORCE_FLUID_INV = NFAM + 2;

// Target particle: its state and its sums (A: Acc, or Term for one pair's).
template <int D, typename R, int FAM, typename A = Acc<R>>
struct Gather {
  static constexpr bool FORCE =
      FAM == FAM_FORCE || FAM == FAM_FORCE_FLUID || FAM == FAM_FORCE_FLUID_INV;
  static constexpr bool FLUID_ONLY = FAM == FAM_FORCE_FLUID || FAM == FAM_FORCE_FLUID_INV;
  static constexpr bool INV = FAM == FAM_FORCE_FLUID_INV;
  // FP32 fluid-only force sweeps read the compact records (RecC)
  static constexpr bool COMPACT = (FORCE || FAM == FAM_STRAIN) && sizeof(R) == 4;
  uint32_t xq[D];  // COMPACT: the target's fixed-point position
  double xi[D];
  R vi[D], ri, pi, iri;
  R si[GR_MAXNS];
  int NS;
  A adv[D], adr;
  A asr[GR_MAXNS], avo[3];

  __device__ inline void load(const Pool<R> P, const SysDesc &S, const Task &T, int64_t gi) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      xi[d] = P.x[d][gi];
      vi[d] = P.vs[d][gi];
    }
    if constexpr (COMPACT) {
#pragma unroll
      for (int d = 0; d < D; ++d) xq[d] = quant_of(xi[d], P.iqs);
    }
    ri = P.rhos[gi];
    iri = Fast<R>::rcp(ri);
    pi = 0;
    NS = T.ns;
    if (FORCE) {
      if (S.kind >= GR_SYS_FLUID) pi = P.p[gi];
      if (!FLUID_ONLY && T.has_stress) {
#pragma unroll
        for (int k = 0; k < GR_MAXNS; ++k) si[k] = k < NS ? P.stress_s[k][gi] : (R)0;
      }
    }
  }

  __device__ inline double da_of(const SrcDesc &Q) const {
    double da = (xi[0] - Q.wp[0]) * Q.wn[0];
#pragma unroll
    for (int d = 1; d < D; ++d) da = da + (xi[d] - Q.wp[d]) * Q.wn[d];
    return da;
  }

  // One accepted pair (target i, partner j at pool index gj), dx = x_i − x_j
  // and r² as evaluated by _pair_self!/_pair_coupled! (src/Interaction.jl:546-553).
  // DYN: 1 or 0 when the caller knows whether the source's partner is a
  // dynamic boundary (Q.pk == PK_DYNAMIC), -1 to test it here.
  template <int DYN = -1>
  __device__ __forceinline__ void pair(const Pool<R> P, const SrcDesc &Q, const SrcK<R> &K,
                                       int64_t gj, const RecA<R> &Aj, const RecB<R> &Bj,
                                       const RecC &Cj, const RecS &Sj, const double *dx,
                                       double r2, double da) {
    constexpr bool FA = Fast<R>::on;
    R dxr[D], gx[D];
    int32_t dq[D];  // COMPACT: x_i − x_j in quanta (exact)
    if constexpr (COMPACT) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        dq[d] = (int32_t)(xq[d] - (uint32_t)Cj.xq[d]);
        dxr[d] = (R)dq[d] * (R)P.qs;
      }
    } else {
#pragma unroll
      for (int d = 0; d < D; ++d) dxr[d] = (R)dx[d];
    }
    // in FP32 the squared distance is summed from the rounded components
    // (the FP64 r² has decided the acceptance already)
    R r2r;
    if constexpr (FA) {
      r2r = dxr[0] * dxr[0];
#pragma unroll
      for (int d = 1; d < D; ++d) r2r = fmaf(dxr[d], dxr[d], r2r);
    } else {
      r2r = (R)r2;
    }
    R r, g, ir = 0;
    if (FA) {
      ir = Fast<R>::rsq(r2r);
      r = r2r * ir;
      g = dwdq<R>(Q.kk, K.norm, r * K.ih) * (ir * K.ih);
    } else {
      r = sqrt(r2r);
      g = dwdq<R>(Q.kk, K.norm, r / K.h) / (r * K.h);
    }
#pragma unroll
    for (int d = 0; d < D; ++d) gx[d] = g * dxr[d];
    if (FAM == FAM_COUNT) {
      adv[0].add((R)1);
      adr.add((R)1);
      return;
    }
    if (FAM == FAM_INTERP && Q.pfn == GR_PFN_NCOUNT) {  // NeighborCountFn (:443-460)
      avo[2].add((R)1);
      return;
    }
    if (FAM == FAM_INTERP) {  // InterpolateFieldFn (src/PairwiseFunctors.jl:424-434)
      // W from the FP64 distance in every mode: an accepted pair (r < 2h in
      // FP64) must weigh W > 0 as in the reference, or a virtual particle
      // whose partners all sit at the edge of the support would get
      // w_sum = 0, zeroed fields and a zero density while still having
      // partners in the force sweeps
      const R w = (R)wq<double>(Q.kk, Q.norm, sqrt(r2) / Q.h);
      const R rj = Aj.rho;
      const R kw = FA ? w * (K.m_q * Fast<R>::rcp(rj)) : w * (K.m_q / rj);
      const int m = Q.sigma;
      if (m & (1 << GR_F_V)) {
#pragma unroll
        for (int d = 0; d < D; ++d) adv[d].add(kw * Bj.v[d]);
      }
      if (m & (1 << GR_F_RHO)) adr.add(kw * rj);
      if (m & (1 << GR_F_P)) avo[0].add(kw * rec_pres(Aj, Bj));
      if (m & (1 << GR_F_STRESS)) {
#pragma unroll
        for (int k = 0; k < GR_MAXNS; ++k)
          if (k < NS) asr[k].add(kw * P.stress_s[k][gj]);
      }
      if (K.alpha != (R)0) avo[1].add(kw);
      return;
    }
    if (FAM == FAM_XSPH) {  // XSPHPfn (src/PairwiseFunctors.jl:364-390)
      // du = −ε·(v_i − v_j)·w/(ρ_i + ρ_j) (src/PairwisePhysics.jl:268-270);
      // the target gains du·m_partner, which is the reference's update of
      // either particle of the pair (du flips sign exactly under i <-> j)
      const R w = wq<R>(Q.kk, K.norm, FA ? r * K.ih : r / K.h);
      const R rs = ri + Aj.rho;
      const R ne = -K.alpha;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const R t = (ne * (vi[d] - Bj.v[d])) * w;
        const R du = FA ? t * Fast<R>::rcp(rs) : t / rs;
        adv[d].add(du * K.m_q);
      }
      return;
    }
    R vj[D], rj, pj = (R)0;
    const R m = K.m_q;
    const bool dyn = DYN < 0 ? Q.pk == PK_DYNAMIC : DYN == 1;
    if (dyn) {  // DynamicBoundarySystem: mirrored velocity
      double db;
      if constexpr (COMPACT) {  // (x_j − p)·n = (x_i − p)·n − (x_i − x_j)·n
        db = da;
#pragma unroll
        for (int d = 0; d < D; ++d) db = db - ((double)dq[d] * P.qs) * Q.wn[d];
      } else {
        db = (Aj.x[0] - Q.wp[0]) * Q.wn[0];
#pragma unroll
        for (int d = 1; d < D; ++d) db = db + (Aj.x[d] - Q.wp[d]) * Q.wn[d];
      }
      const double rat = fabs(db / da);
      const double mn = isnan(rat) ? rat : (rat < Q.wbeta ? rat : Q.wbeta);
      const R fac = (R)(-mn);
#pragma unroll
      for (int d = 0; d < D; ++d) vj[d] = fac * vi[d];
      rj = ri;
      pj = pi;
    } else if constexpr (COMPACT) {
#pragma unroll
      for (int d = 0; d < D; ++d) vj[d] = Cj.v[d];
      rj = Cj.rho;
      pj = Cj.p;
    } else {
#pragma unroll
      for (int d = 0; d < D; ++d) vj[d] = Bj.v[d];
      rj = Aj.rho;
      pj = rec_pres(Aj, Bj);
    }
    R irj;
    if constexpr (INV)  // the record's 1/ρ (a dynamic partner mirrors the target)
      irj = dyn ? iri : rj;
    else  // a dynamic partner has rj = ri, so this is iri bit for bit (a select
          // of the two made the compiler keep them in scratch memory)
      irj = Fast<R>::rcp(rj);
    if (FAM == FAM_STRAIN) {  // strain_rate_tensor / vorticity_tensor
      R dv[D];
#pragma unroll
      for (int d = 0; d < D; ++d) dv[d] = vj[d] - vi[d];
      const R f = FA ? m * irj : m / rj;
      if (D == 2) {
        asr[0].add(dv[0] * gx[0] * f);
        asr[1].add(dv[1] * gx[1] * f);
        const R sh = (R)0.5 * (dv[0] * gx[1] + dv[1] * gx[0]) * f;
        if (NS == 4)
          asr[3].add(sh);
        else
          asr[2].add(sh);
      } else {
        asr[0].add(dv[0] * gx[0] * f);
        asr[1].add(dv[1] * gx[1] * f);
        asr[2].add(dv[D - 1] * gx[D - 1] * f);
        asr[3].add((R)0.5 * (dv[0] * gx[1] + dv[1] * gx[0]) * f);
        asr[4].add((R)0.5 * (dv[0] * gx[D - 1] + dv[D - 1] * gx[0]) * f);
        asr[5].add((R)0.5 * (dv[1] * gx[D - 1] + dv[D - 1] * gx[1]) * f);
      }
      if (Q.pfn == GR_PFN_SRV) {
        avo[0].add((R)0.5 * (dv[0] * gx[1] - dv[1] * gx[0]) * f);
        if (D == 3) {
          avo[1].add((R)0.5 * (dv[0] * gx[D - 1] - dv[D - 1] * gx[0]) * f);
          avo[2].add((R)0.5 * (dv[1] * gx[D - 1] - dv[D - 1] * gx[1]) * f);
        }
      }
      return;
    }
    // FAM_FORCE: FluidPfn / CauchyFluidPfn
    R dv[D];
#pragma unroll
    for (int d = 0; d < D; ++d) dv[d] = vi[d] - vj[d];
    R vr = dxr[0] * dv[0];
#pragma unroll
    for (int d = 1; d < D; ++d) vr = vr + dxr[d] * dv[d];
    vr = jmin0(vr);
    const R muv = FA ? K.hf * vr * Fast<R>::rcp(r2r + K.h2) : K.hf * vr / (r2r + K.h2);
    const R piv = FA ? (K.beta * muv - K.alpha * K.mc) * muv * ((R)2 * iri * irj)
                     : (K.beta * muv - K.alpha * K.mc) * muv / ((R)0.5 * ri * rj);
    if (Q.pk == PK_STATIC) {  // lennard_jones + artificial viscosity
      const R lr = FA ? K.ljcut * ir : K.ljcut / r;
      const R lj = (r < K.ljcut ? (R)1 : (R)0) * (pow_i(lr, 12) - pow_i(lr, 6));
      const R f = FA ? lj * (ir * ir) : lj / r2r;
      const R rf = K.ljc2 * f;
      const R t = -m * piv;
#pragma unroll
      for (int d = 0; d < D; ++d) adv[d].add(t * gx[d] + rf * dxr[d]);
      return;
    }
    R dr = dv[0] * gx[0];
#pragma unroll
    for (int d = 1; d < D; ++d) dr = dr + dv[d] * gx[d];
    R psi = (R)0;
    if (K.has_delta) {
      R dxg = dxr[0] * gx[0];
#pragma unroll
      for (int d = 1; d < D; ++d) dxg = dxg + dxr[d] * gx[d];
      psi = FA ? K.psi_coef * (ri - rj) * dxg * (ir * ir) : K.psi_coef * (ri - rj) * dxg / r2r;
    }
    if (FLUID_ONLY || Q.pfn == GR_PFN_FLUID || Q.pfn == GR_PFN_FLUIDSOLID) {
      // FluidSolidPfn: the fluid's pressure on both sides (the target's on
      // the fluid side, the partner's on the solid side)
      const R pa = Q.psel == 2 ? pj : pi, pb = Q.psel == 1 ? pi : pj;
      R dh;
      if constexpr (INV) {  // S = 2; the record's p/ρ² for a real partner
        dh = -(pa * (iri * iri) + (dyn ? pb * (irj * irj) : pj));
      } else if (FA) {
        if (K.sigma == 1)
          dh = -(pa + pb) * (iri * irj);
        else
          dh = -(pa * (iri * iri) + pb * (irj * irj));
      } else {
        if (K.sigma == 1)
          dh = -(pa + pb) / (ri * rj);
        else
          dh = -(pa / (ri * ri) + pb / (rj * rj));
      }
      if (Q.pk == PK_TWO_SIDED) {
        R ast = (R)0;
        if (K.has_eps)
          ast = FA ? K.eps * (-(fabs(pi) + fabs(pj)) * (iri * irj))
                   : K.eps * (-(fabs(pi) + fabs(pj)) / (ri * rj));
        const R t = dh + ast - piv;
#pragma unroll
        for (int d = 0; d < D; ++d) adv[d].add(m * (t * gx[d]));
      } else {
        const R t = m * (dh - piv);
#pragma unroll
        for (int d = 0; d < D; ++d) adv[d].add(t * gx[d]);
      }
      const R coef = (K.sigma == 1) ? (FA ? ri * irj : ri / rj) : (R)1;
      adr.add(m * (dr * coef + (FA ? psi * irj : psi / rj)));
    } else {  // cauchy_stress_force
      R sj[GR_MAXNS];
      if (dyn) {
#pragma unroll
        for (int k = 0; k < GR_MAXNS; ++k) sj[k] = si[k];
      } else {
#pragma unroll
        for (int k = 0; k < GR_MAXNS; ++k) {
          if constexpr (COMPACT) {
            const float sk = k < 4 ? (&Sj.a.x)[k] : (&Sj.b.x)[k - 4];
            sj[k] = k < NS ? (R)sk : (R)0;
          } else {
            sj[k] = k < NS ? P.stress_s[k][gj] : (R)0;
          }
        }
      }
      const R ci = FA ? iri * iri : (R)1 / (ri * ri), cj = FA ? irj * irj : (R)1 / (rj * rj);
      R hv[D];
      if (D == 2) {
        R a0, a1;
        if (NS == 3) {
          a0 = (si[0] * gx[0] + si[2] * gx[1]) * ci + (sj[0] * gx[0] + sj[2] * gx[1]) * cj;
          a1 = (si[2] * gx[0] + si[1] * gx[1]) * ci + (sj[2] * gx[0] + sj[1] * gx[1]) * cj;
        } else {
          a0 = (si[0] * gx[0] + si[3] * gx[1]) * ci + (sj[0] * gx[0] + sj[3] * gx[1]) * cj;
          a1 = (si[3] * gx[0] + si[1] * gx[1]) * ci + (sj[3] * gx[0] + sj[1] * gx[1]) * cj;
        }
        hv[0] = a0;
        hv[D - 1] = a1;
      } else {
        hv[0] = (si[0] * gx[0] + si[3] * gx[1] + si[4] * gx[D - 1]) * ci +
                (sj[0] * gx[0] + sj[3] * gx[1] + sj[4] * gx[D - 1]) * cj;
        hv[1] = (si[3] * gx[0] + si[1] * gx[1] + si[5] * gx[D - 1]) * ci +
                (sj[3] * gx[0] + sj[1] * gx[1] + sj[5] * gx[D - 1]) * cj;
        hv[D - 1] = (si[4] * gx[0] + si[5] * gx[1] + si[2] * gx[D - 1]) * ci +
                    (sj[4] * gx[0] + sj[5] * gx[1] + sj[2] * gx[D - 1]) * cj;
      }
#pragma unroll
      for (int d = 0; d < D; ++d) adv[d].add(m * (hv[d] - piv * gx[d]));
      adr.add(m * (dr + (FA ? psi * irj : psi / rj)));
    }
  }

  __device__ inline void store(const Pool<R> P, const SysDesc &S, const Task &T, int64_t gi) {
    if (FAM == FAM_INTERP) {  // += into the virtual system's fields (and shadows)
      const int m = T.imask;
      if (m & (1 << GR_F_V)) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
          const double nv = P.v[d][gi] + (double)adv[d].get();
          P.v[d][gi] = nv;
          P.vs[d][gi] = (R)nv;
        }
      }
      if (m & (1 << GR_F_RHO)) {
        const double nv = P.rho[gi] + (double)adr.get();
        P.rho[gi] = nv;
        P.rho_h[gi] = nv;
        P.rhos[gi] = (R)nv;
      }
      if (m & (1 << GR_F_P)) P.p[gi] = (R)((double)P.p[gi] + (double)avo[0].get());
      if (m & (1 << GR_F_STRESS)) {
#pragma unroll
        for (int k = 0; k < GR_MAXNS; ++k)
          if (k < NS) {
            const double nv = P.stress[k][gi] + (double)asr[k].get();
            P.stress[k][gi] = nv;
            P.stress_s[k][gi] = (R)nv;
          }
      }
      if (m & (1 << 30)) P.wsum[gi] += (double)avo[1].get();
      if (m & (1 << GR_F_COUNT)) P.pcnt[gi] += (double)avo[2].get();
      return;
    }
    if (FAM == FAM_XSPH) {
      int64_t gs = gi;
      if (T.alias >= 0) {
        const int64_t j = gi - S.off;
        if (j >= T.alias_cap) return;  // reported by k_alias_check
        gs = T.alias_off + j;
      }
#pragma unroll
      for (int d = 0; d < D; ++d) P.vadj[d][gs] = P.vadj[d][gs] + (double)adv[d].get();
      return;
    }
    if (FAM == FAM_STRAIN) {
#pragma unroll
      for (int k = 0; k < GR_MAXNS; ++k)
        if (k < NS) {
          const R v = asr[k].get();
          P.sr[k][gi] = T.assign ? v : P.sr[k][gi] + v;
        }
      if (T.write_vor) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
          if (k < T.nv) {
            const R v = avo[k].get();
            P.vor[k][gi] = T.assign ? v : P.vor[k][gi] + v;
          }
      }
      return;
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const R v = adv[d].get();
      P.dvdt[d][gi] = T.assign ? (R)S.sv[d] + v : P.dvdt[d][gi] + v;
    }
    const R v = adr.get();
    P.drhodt[gi] = T.assign ? (R)S.srho + v : P.drhodt[gi] + v;
  }
};

// Target cell in the grid of a source, clamped so every strip lies inside.
template <int D>
__device__ inline void target_cell(const double *xi, const Grid &G, double cell, int *c) {
#pragma unroll
  for (int d = 0; d < D; ++d) {
    int cd = (int)floor((xi[d] - G.ming[d]) / cell);
    cd = cd < 1 ? 1 : cd;
    cd = cd > G.ng[d] - 2 ? G.ng[d] - 2 : cd;
    c[d] = cd;
  }
}

// First cell of strip st (3 consecutive cells along the fastest dimension).
template <int D>
__device__ inline int strip_base(const int *c, const Grid &G, int st) {
  if (D == 3) {
    const int ddx = st / 3 - 1, ddy = st % 3 - 1;
    return ((c[0] + ddx) * G.ng[1] + (c[1] + ddy)) * G.ng[2] + (c[D - 1] - 1);
  }
  return (c[0] + st - 1) * G.ng[1] + (c[D - 1] - 1);
}

// Whether a pair of this family reads the partner's record B (velocity, and
// pressure in FP64): a dynamic boundary partner mirrors the target instead.
template <int FAM>
__device__ inline bool needs_b(const SrcDesc &Q) {
  if (FAM == FAM_COUNT) return false;
  if (FAM == FAM_INTERP) return Q.pfn != GR_PFN_NCOUNT;
  if (FAM == FAM_XSPH) return true;
  return Q.pk != PK_DYNAMIC;
}

// Whether a compact force pair reads the partner's stress record: Cauchy
// functors against a partner with its own stress (a dynamic boundary mirrors
// the target's).
template <int FAM>
__device__ inline bool needs_s(const SrcDesc &Q) {
  return FAM == FAM_FORCE && Q.pfn == GR_PFN_CAUCHY && Q.pk != PK_DYNAMIC;
}

// Direct cell walk of every source of the task (no list).
template <int D, typename R, int FAM>
__device__ void gather_direct(Gather<D, R, FAM> &Gt, const Pool<R> P, const SysDesc *sd,
                              const Task &T, const SrcDesc *srcs, const Grid *grids,
                              const CellArr *carr, const int *cells, int i,
                              unsigned long long &ns, unsigned long long &no) {
  for (int q = T.src_begin; q < T.src_end; ++q) {
    const SrcDesc Q = srcs[q];
    const Grid G = grids[Q.grid];
    if (G.ncells <= 0) continue;
    const int *cs = cells + carr[Q.carr].off;
    const int64_t poff = sd[Q.partner].off;
    SrcK<R> K;
    K.load(Q);
    int c[D];
    target_cell<D>(Gt.xi, G, Q.cell, c);
    const double da = (Q.pk == PK_DYNAMIC) ? Gt.da_of(Q) : 0.0;
    for (int st = 0; st < ((D == 3) ? 9 : 3); ++st) {
      const int base = strip_base<D>(c, G, st);
      const int j0 = cs[base] - 1, j1 = cs[base + 3] - 1;
      for (int j = j0; j < j1; ++j) {
        if (Q.pk == PK_SELF && j == i) continue;
        const int64_t gj = poff + j;
        constexpr bool CMP = Gather<D, R, FAM>::COMPACT;
        // compact sweeps read no RecA: the walk's FP64 test uses the positions
        RecA<R> Aj{};
        double dx[D];
        if constexpr (CMP) {
#pragma unroll
          for (int d = 0; d < D; ++d) dx[d] = Gt.xi[d] - P.x[d][gj];
        } else {
          Aj = P.ra[gj];
#pragma unroll
          for (int d = 0; d < D; ++d) dx[d] = Gt.xi[d] - Aj.x[d];
        }
        double r2 = dx[0] * dx[0];
#pragma unroll
        for (int d = 1; d < D; ++d) r2 = r2 + dx[d] * dx[d];
        if (!(r2 < Q.cutoff2)) continue;
        if (Q.pk == PK_SELF)
          ++ns;
        else
          ++no;
        Gt.pair(P, Q, K, gj, Aj, (!CMP && needs_b<FAM>(Q)) ? P.rb[gj] : RecB<R>{},
                CMP ? P.rc[gj] : RecC{}, (CMP && needs_s<FAM>(Q)) ? P.rs[gj] : RecS{}, dx,
                r2, da);
      }
    }
  }
}

template <bool CNT>
__device__ inline void count_pairs(unsigned long long *pc, unsigned long long a,
                                   unsigned long long o2) {
  if (!CNT) return;
  // [0]: ordered self pairs (each unordered pair seen from both sides),
  // [1]: coupled pairs seen from the gathering side.
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    o2 += __shfl_xor(o2, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    if (a) atomicAdd(&pc[0], a);
    if (o2) atomicAdd(&pc[1], o2);
  }
}

template <int D, typename R, int FAM, bool CNT>
__global__ void __launch_bounds__(GR_BLOCK)
    k_sweep(Pool<R> P, const SysDesc *__restrict__ sd, const int *__restrict__ n_dev,
            const Task *__restrict__ tasks, const SrcDesc *__restrict__ srcs,
            const Grid *__restrict__ grids, const CellArr *__restrict__ carr,
            const int *__restrict__ cells, const Blk *__restrict__ blk, int nblk,
            unsigned long long *pair_count) {
  const Blk b = blk[xcd_block(nblk)];
  const Task T = tasks[b.item];
  const int i = b.first + threadIdx.x;
  const SysDesc S = sd[T.sys];
  const bool live = i < n_dev[T.sys];
  const int64_t gi = S.off + (live ? i : 0);
  Gather<D, R, FAM> Gt;
  Gt.load(P, S, T, gi);
  unsigned long long ns = 0, no = 0;
  if (live) gather_direct<D, R, FAM>(Gt, P, sd, T, srcs, grids, carr, cells, i, ns, no);
  count_pairs<CNT>(pair_count, ns, no);
  if (live) Gt.store(P, S, T, gi);
}

// ---------------------------------------------------------------------------
// Neighbour lists
// ---------------------------------------------------------------------------

// Accepted partners of every target of a list task, per source, in the
// order the sources are listed, as acceptance masks: an entry, a 64-bit mask
// {lo, hi} and a base, says that candidates base + b of the source
// (source-local indices, b = 0..63) with bit b set are partners.  Entries
// follow the cell walk (strips in order, ascending candidates), so popping the
// bits in order visits the partners in the walk's order.  The masks and the
// bases are two arrays: entry e of target i has its mask at
// lidx[L.list_off + 2·(e·L.cap + i)] (an int2) and its base at
// lidx[L.list_off + 2·L.maxnb·L.cap + e·L.cap + i]; a lane writes one
// 12-byte entry per (strip, 64 candidates) that holds a partner, and a
// wavefront reads a row of entries as 512 and 256 contiguous bytes.
// lcnt[L.cnt_off + q·L.cap + i] holds the number of entries of source q.
// More than L.maxnb entries mean "overflow" (the physics pass then walks the
// cells directly).
//
// One wavefront per workgroup.  For each strip, lanes whose candidate ranges
// start within span·wmax of the lowest pending start form a group (targets
// in one cell column); the group's union of ranges is staged in LDS, WIN
// candidates at a time, with coalesced loads, and every lane walks its own
// range from LDS in ascending order and sets the bits of the candidates that
// pass the walk's test: no per-partner store.  The staged candidates are FP32
// offsets, on which all but the closest calls are decided exactly (Screen).
// The search is bound by its vector instructions (the loads of a strip hide
// behind the tests of the wavefronts next to it): testing all in FP64 took 8 FP64
// operations a candidate, a comparison and the bit's insertion, 307 us in the
// 3D dam break of 1.4M particles and 84 for 64 2D columns; the screen, 8 FP32
// operations in all, takes 214 and 74.
// WIN and span change only which lanes load together, never a lane's tests
// or their order: every choice gives the same lists.
// Wave-wide minimum / maximum (all 64 lanes active): DPP within each row of
// 16 lanes, then the four row results through scalar registers.
template <bool MAX>
__device__ inline int wave_red_dpp(int v) {
  auto op = [](int x, int y) { return MAX ? (x > y ? x : y) : (x < y ? x : y); };
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));   // quad_perm 1,0,3,2
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));   // quad_perm 2,3,0,1
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xF, 0xF, false));  // row_half_mirror
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xF, 0xF, false));  // row_mirror
  return op(op(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
            op(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// The walk's test r² < c² (FP64) screened in FP32: candidates and target as
// offsets from a point O near the wavefront's targets, r = Σ(x − x_j)² − c² by
// three subtractions and three FMAs, whose sign is the answer wherever |r|
// exceeds the FP32 error bound `tol`; the others are tested in FP64.
//
// Bound, with u = 2⁻²⁴, X the target's largest offset and c the cell (c² >=
// cutoff²).  A candidate of the cells around the target's differs from it by
// a <= 2c in each dimension: both offsets round by at most u(2X + 2c) together,
// their difference by ua, so r errs by 2Σa·u(2X + 4c) <= u(24cX + 48c²), and by
// 3u·12c² in the sums and uc² in c².  A candidate farther than 2c (of cells out
// of the sort's order) has r >= 3/4 a² and an error of u(12aX + 22a²), too
// small to change its sign while X <= 1e5 c; beyond that all are tested, and
// where c is so small or large that c² (or the tolerance's products) could
// leave FP32's normal range (`all`: cells outside 2^±40).
template <int D>
struct Screen {
  float xf[D], c2, tol;
  bool finite, all;
  __device__ inline void set(const double *xi, const double *O) {
    finite = true;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      xf[d] = (float)(xi[d] - O[d]);
      finite = finite && fabs(xi[d]) <= 1.7976931348623157e308;  // else it has no partner
    }
  }
  __device__ inline void source(double cutoff2, double cell) {
    float X = fabsf(xf[0]);
#pragma unroll
    for (int d = 1; d < D; ++d) X = fmaxf(X, fabsf(xf[d]));
    const float c = (float)cell;
    c2 = (float)cutoff2;
    tol = 6.1e-8f * (c * (24.0f * X + 96.0f * c));
    if (!(X <= 1.0e5f * c) || !(cutoff2 <= cell * cell * (1.0 + 1e-9))) tol = __builtin_inff();
    const unsigned e = (unsigned)((unsigned long long)__double_as_longlong(cell) >> 52);
    all = e - (1023u - 40u) > 80u;  // (by the exponent: scalar arithmetic)
  }
  // a staged coordinate; one beyond FP32's range (or not finite) is far from
  // every target of a cell whose candidates are screened
  static __device__ inline float stage(double x, double o) {
    const float f = (float)(x - o);
    return fabsf(f) < 3.0e38f ? f : 3.0e38f;
  }
};
// A point near the wavefront's targets (uniform): the first lane's.
template <int D>
__device__ inline void screen_origin(const double *xi, double *O) {
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(xi[d]);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    O[d] = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    if (!(fabs(O[d]) < 1.0e300)) O[d] = 0.0;
  }
}

// Screened signs of the four candidates staged at t, the first one's highest, in
// the low bits of `cur` (shifted up); returns the smallest |r| less `tol`.
template <int D, int W>
__device__ __forceinline__ float screen4(const Screen<D> &scr, const float (*sf)[W], int t,
                                         unsigned &cur) {
  float r[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float a0 = scr.xf[0] - sf[0][t + u];
    r[u] = fmaf(a0, a0, -scr.c2);
  }
#pragma unroll
  for (int k = 1; k < D; ++k)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float ak = scr.xf[k] - sf[k][t + u];
      r[u] = fmaf(ak, ak, r[u]);
    }
#pragma unroll
  for (int u = 0; u < 4; ++u) cur = __builtin_amdgcn_alignbit(cur, __float_as_uint(r[u]), 31);
  return fminf(fminf(fabsf(r[0]), fabsf(r[1])), fminf(fabsf(r[2]), fabsf(r[3]))) - scr.tol;
}
// The walk's own test of pool indices g .. g + 3 (none beyond `last` is read).
template <int D, typename R>
__device__ inline unsigned exact4(const Pool<R> &P, const double *xi, double c2, int64_t g,
                                  int64_t last) {
  unsigned ex = 0u;
#pragma unroll 1  // seldom run: registers count
  for (int u = 0; u < 4; ++u) {
    const int64_t j = g + u < last ? g + u : last;
    const double a0 = xi[0] - P.x[0][j];
    double r2 = a0 * a0;
#pragma unroll
    for (int k = 1; k < D; ++k) {
      const double ak = xi[k] - P.x[k][j];
      r2 = r2 + ak * ak;
    }
    ex = (ex << 1) | (unsigned)(r2 < c2);
  }
  return ex;
}

template <int D, typename R, int WIN>
__global__ void __launch_bounds__(64)
    k_nlist(Pool<R> P, const SysDesc *__restrict__ sd, const int *__restrict__ n_dev,
            const LTask *__restrict__ lt, const SrcDesc *__restrict__ srcs,
            const Grid *__restrict__ grids, const CellArr *__restrict__ carr,
            const int *__restrict__ cells, const Blk *__restrict__ blk, int nblk, int *lcnt,
            int *lidx, const long long *__restrict__ bbmin,
            const long long *__restrict__ bbmax, int span) {
  __shared__ float sf[D][WIN + 4];
  const Blk b = blk[xcd_block(nblk)];
  const LTask L = lt[b.item];
  const int lane = threadIdx.x;
  const int i = b.first + lane;
  const SysDesc S = sd[L.sys];
  const bool live = i < n_dev[L.sys];
  const int64_t gi = S.off + (live ? i : 0);
  double xi[D];
#pragma unroll
  for (int d = 0; d < D; ++d) xi[d] = P.x[d][gi];
  int2 *emask = reinterpret_cast<int2 *>(lidx + L.list_off) + i;
  int *ebase = lidx + L.list_off + 2 * (int64_t)L.maxnb * L.cap + i;
  double O[D];
  Screen<D> scr;
  screen_origin<D>(xi, O);
  scr.set(xi, O);
  int ne = 0;  // entries of this target
  int cq = 0;  // entries of the current source
  for (int q = L.src_begin; q < L.src_end; ++q) {
    const SrcDesc Q = srcs[q];
    const Grid G = grids[Q.grid];
    cq = 0;
    if (G.ncells > 0) {
      const int *cs = cells + carr[Q.carr].off;
      // the target itself (a self source) passes the distance test with
      // r² = 0; its bit is cleared when a mask is stored
      const int self_j = Q.pk == PK_SELF ? i : -1;
      const double c2 = Q.cutoff2;
      const int64_t poff = sd[Q.partner].off;
      // a dynamic boundary (a sorted real system, its bounds taken this
      // step) more than a cutoff from the target along some axis holds no
      // partner: the margin keeps every FP64 r² of such a pair above c2
      bool act = live && scr.finite;
      scr.source(c2, Q.cell);
      if (Q.pk == PK_DYNAMIC && bbmin) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
          const double mn = double_of(bbmin[Q.partner * 3 + d]);
          const double mx = double_of(bbmax[Q.partner * 3 + d]);
          const double gap = mn - xi[d] > xi[d] - mx ? mn - xi[d] : xi[d] - mx;
          act = act && !(gap > Q.cell * (1.0 + 1e-9));
        }
      }
      int c[D];
      target_cell<D>(xi, G, Q.cell, c);
      constexpr int NST = (D == 3) ? 9 : 3;
      // the next strip's range is loaded while the current strip is tested;
      // a lane past the system's end keeps the empty range [0, 0) (a
      // negative base would run its candidate loop)
      int n0 = 1, n1 = 1;
      if (act) {
        const int sb = strip_base<D>(c, G, 0);
        n0 = cs[sb];
        n1 = cs[sb + 3];
      }
      for (int st = 0; st < (__builtin_amdgcn_ballot_w64(act) != 0ull ? NST : 0); ++st) {
        const int j0 = n0 - 1, j1 = n1 - 1;
        if (act && st + 1 < NST) {
          const int sb = strip_base<D>(c, G, st + 1);
          n0 = cs[sb];
          n1 = cs[sb + 3];
        }
        bool pend = j0 < j1;
        if (__builtin_amdgcn_ballot_w64(pend) == 0ull) continue;
        // mask of candidates base .. base + 63 in two words; d = j − base
        int base = j0, d = 0;
        unsigned lo = 0u, hi = 0u;
        auto flush = [&]() {
          const unsigned sdl = (unsigned)(self_j - base);
          const unsigned sbit = 1u << (sdl & 31u);
          lo &= sdl < 32u ? ~sbit : ~0u;
          hi &= sdl - 32u < 32u ? ~sbit : ~0u;
          if (live && (lo | hi) != 0u) {
            if (ne < L.maxnb) {
              emask[(int64_t)ne * L.cap] = make_int2((int)lo, (int)hi);
              ebase[(int64_t)ne * L.cap] = base;
            }
            ++ne;
            ++cq;
          }
          lo = hi = 0u;
        };
        const int wmax = wave_red_dpp<true>(j1 - j0);
        while (true) {
          const int glo = wave_red_dpp<false>(pend ? j0 : INT_MAX);
          if (glo == INT_MAX) break;
          const bool mem = pend && j0 - glo <= span * wmax;
          const int ghi = wave_red_dpp<true>(mem ? j1 : INT_MIN);
          for (int w0 = glo; w0 < ghi; w0 += WIN) {
            const int w1 = ghi - w0 < WIN ? ghi : w0 + WIN;
            __syncthreads();  // the previous window has been read
            for (int t = lane; t < w1 - w0; t += 64) {
#pragma unroll
              for (int k = 0; k < D; ++k) sf[k][t] = scr.stage(P.x[k][poff + w0 + t], O[k]);
            }
            __syncthreads();
            // this lane's candidates in the window end before je; base + d is
            // the next one (where the previous window stopped)
            const int je = mem ? (j1 < w1 ? j1 : w1) : 0;
            while (base + d < je) {
              if (d == 64) {  // the mask is full: store it, move it on
                flush();
                base += 64;
                d = 0;
              }
              // a run of candidates within one 32-bit word of the mask
              const int wsel = d >> 5;
              const int lim = je - base, wend = (d & ~31) + 32;
              const int dend = lim < wend ? lim : wend;
              // four at a time, the last four beyond the run's end if need be
              // (read, never kept); nr has a bit for each four that hold one
              // too close to call
              const int n = dend - d, ng = (n + 3) >> 2, t0 = base - w0 + d;
              unsigned cur = 0u, nr = 0u;
              for (int t = t0; t < t0 + n; t += 4)
                nr = __builtin_amdgcn_alignbit(
                    nr, __float_as_uint(screen4<D>(scr, sf, t, cur)), 31);
              if (scr.all) nr = (1u << ng) - 1u;
              while (nr != 0u) {
                const int g = __builtin_ctz(nr);
                nr &= nr - 1u;
                cur &= ~(15u << (4 * g));
                cur |= exact4<D>(P, xi, c2, poff + base + d + 4 * (ng - 1 - g), poff + w1 - 1)
                       << (4 * g);
              }
              cur = (__brev(cur) >> (32 - 4 * ng)) & (~0u >> (32 - n));
              cur <<= d & 31;
              d = dend;
              // selects, not branches (here and when the target's own bit
              // is cleared): branches make the compiler index a pair
              // {lo, hi} kept in scratch memory
              lo |= wsel == 0 ? cur : 0u;
              hi |= wsel != 0 ? cur : 0u;
            }
          }
          if (mem) pend = false;
        }
        flush();
      }
    }
    if (live) lcnt[L.cnt_off + (int64_t)(q - L.src_begin) * L.cap + i] = cq;
  }
  if (live)
    lcnt[L.cnt_off + (int64_t)(L.src_end - L.src_begin) * L.cap + i] = ne > L.maxnb ? 1 : 0;
}

// OR over the quad of lanes (all four active).
__device__ __forceinline__ unsigned quad_or(unsigned v) {
  v |= (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xF, 0xF, false);
  v |= (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4E, 0xF, 0xF, false);
  return v;
}

// The search with S lanes per target (64 / S targets per wavefront, S
// wavefronts per entry of the block table): lane s of a target tests four of
// every 16 of its candidates, and the masks are the OR of the S lanes', so
// the lists are k_nlist's.  For launches of few targets, which latency bounds
// (nlist_split_blocks): S times the wavefronts, each with 1/S of the tests and
// about half the candidates to stage; a launch that fills the chip pays S
// times k_nlist's work per strip instead (3D dam break of 512k: 217 us against
// 132).
template <int D, typename R, int WIN, int S_>
__global__ void __launch_bounds__(64)
    k_nlist_split(Pool<R> P, const SysDesc *__restrict__ sd, const int *__restrict__ n_dev,
                  const LTask *__restrict__ lt, const SrcDesc *__restrict__ srcs,
                  const Grid *__restrict__ grids, const CellArr *__restrict__ carr,
                  const int *__restrict__ cells, const Blk *__restrict__ blk, int nblk, int *lcnt,
                  int *lidx, const long long *__restrict__ bbmin,
                  const long long *__restrict__ bbmax, int span) {
  static_assert(S_ == 4, "quad_or joins four lanes");
  __shared__ float sf[D][WIN + 4];
  const int lb = xcd_block(nblk * S_);
  const Blk b = blk[lb / S_];
  const LTask L = lt[b.item];
  const int lane = threadIdx.x, sl = lane % S_;
  const int i = b.first + (lb % S_) * (64 / S_) + lane / S_;
  const SysDesc S = sd[L.sys];
  const bool live = i < n_dev[L.sys];
  if (__builtin_amdgcn_ballot_w64(live) == 0ull) return;
  const int64_t gi = S.off + (live ? i : 0);
  double xi[D];
#pragma unroll
  for (int d = 0; d < D; ++d) xi[d] = P.x[d][gi];
  int2 *emask = reinterpret_cast<int2 *>(lidx + L.list_off) + i;
  int *ebase = lidx + L.list_off + 2 * (int64_t)L.maxnb * L.cap + i;
  double O[D];
  Screen<D> scr;
  screen_origin<D>(xi, O);
  scr.set(xi, O);
  int ne = 0;  // entries of this target
  int cq = 0;  // entries of the current source
  for (int q = L.src_begin; q < L.src_end; ++q) {
    const SrcDesc Q = srcs[q];
    const Grid G = grids[Q.grid];
    cq = 0;
    if (G.ncells > 0) {
      const int *cs = cells + carr[Q.carr].off;
      const int self_j = Q.pk == PK_SELF ? i : -1;
      const double c2 = Q.cutoff2;
      const int64_t poff = sd[Q.partner].off;
      bool act = live && scr.finite;  // as in k_nlist
      scr.source(c2, Q.cell);
      if (Q.pk == PK_DYNAMIC && bbmin) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
          const double mn = double_of(bbmin[Q.partner * 3 + d]);
          const double mx = double_of(bbmax[Q.partner * 3 + d]);
          const double gap = mn - xi[d] > xi[d] - mx ? mn - xi[d] : xi[d] - mx;
          act = act && !(gap > Q.cell * (1.0 + 1e-9));
        }
      }
      int c[D];
      target_cell<D>(xi, G, Q.cell, c);
      constexpr int NST = (D == 3) ? 9 : 3;
      if (__builtin_amdgcn_ballot_w64(act) != 0ull) {
        // every strip's range up front: one latency instead of one a strip
        int n0[NST], n1[NST];
#pragma unroll
        for (int st = 0; st < NST; ++st) {
          n0[st] = n1[st] = 1;
          if (act) {
            const int sb = strip_base<D>(c, G, st);
            n0[st] = cs[sb];
            n1[st] = cs[sb + 3];
          }
        }
#pragma unroll
        for (int st = 0; st < NST; ++st) {
          const int j0 = n0[st] - 1, j1 = n1[st] - 1;
          bool pend = j0 < j1;
          if (__builtin_amdgcn_ballot_w64(pend) == 0ull) continue;
          int base = j0;
          unsigned lo = 0u, hi = 0u;
          auto flush = [&]() {
            lo = quad_or(lo);
            hi = quad_or(hi);
            const unsigned sdl = (unsigned)(self_j - base);
            const unsigned sbit = 1u << (sdl & 31u);
            lo &= sdl < 32u ? ~sbit : ~0u;
            hi &= sdl - 32u < 32u ? ~sbit : ~0u;
            if (live && (lo | hi) != 0u) {
              if (ne < L.maxnb && sl == 0) {
                emask[(int64_t)ne * L.cap] = make_int2((int)lo, (int)hi);
                ebase[(int64_t)ne * L.cap] = base;
              }
              ++ne;
              ++cq;
            }
            lo = hi = 0u;
          };
          const int wmax = wave_red_dpp<true>(j1 - j0);
          while (true) {
            const int glo = wave_red_dpp<false>(pend ? j0 : INT_MAX);
            if (glo == INT_MAX) break;
            const bool mem = pend && j0 - glo <= span * wmax;
            const int ghi = wave_red_dpp<true>(mem ? j1 : INT_MIN);
            for (int w0 = glo; w0 < ghi; w0 += WIN) {
              const int w1 = ghi - w0 < WIN ? ghi : w0 + WIN;
              __syncthreads();  // the previous window has been read
              for (int t = lane; t < w1 - w0; t += 64) {
#pragma unroll
                for (int k = 0; k < D; ++k) sf[k][t] = scr.stage(P.x[k][poff + w0 + t], O[k]);
              }
              __syncthreads();
              // the target's candidates in the window, [js, je): the same for
              // its S lanes, so they store a full mask together
              const int js = j0 > w0 ? j0 : w0;
              const int je = mem ? (j1 < w1 ? j1 : w1) : 0;
              if (js < je) {
                if (js >= base + 64) {
                  flush();
                  base += 64;
                }
                while (true) {
                  const int ce = je < base + 64 ? je : base + 64;
                  const int jb = js > base ? js : base;
                  // the four lanes take four candidates each in turn: lane sl
                  // those at 4·sl of every 16
                  const int n = ce - jb;
                  unsigned part[4];
#pragma unroll
                  for (int m = 0; m < 4; ++m) {
                    const int o = 16 * m + 4 * sl;
                    unsigned sg = 0u;
                    if (o < n) {
                      if (screen4<D>(scr, sf, jb - w0 + o, sg) < 0.0f || scr.all)
                        sg = exact4<D>(P, xi, c2, poff + jb + o, poff + w1 - 1);
                      sg = __brev(sg) >> 28;
                    }
                    part[m] = sg << (4 * sl);
                  }
                  unsigned long long cur =
                      ((unsigned long long)(part[2] | part[3] << 16) << 32) |
                      (part[0] | part[1] << 16);
                  cur = (cur & (~0ull >> (64 - n))) << (jb - base);
                  lo |= (unsigned)cur;
                  hi |= (unsigned)(cur >> 32);
                  if (base + 64 >= je) break;
                  flush();
                  base += 64;
                }
              }
            }
            if (mem) pend = false;
          }
          flush();
        }
      }
    }
    if (live && sl == 0) lcnt[L.cnt_off + (int64_t)(q - L.src_begin) * L.cap + i] = cq;
  }
  if (live && sl == 0)
    lcnt[L.cnt_off + (int64_t)(L.src_end - L.src_begin) * L.cap + i] = ne > L.maxnb ? 1 : 0;
}

// k_nlist_split for launches smaller still (nlist_all_blocks): where the targets
// of a wavefront share a cell column, and so the unions of their ranges are
// short, all strips of a source are staged together, a memory latency or two
// instead of one a strip.  It takes 221 registers in 3D, so a SIMD holds two
// wavefronts.
template <int D, typename R, int WIN>
__global__ void __launch_bounds__(64)
    k_nlist_small(Pool<R> P, const SysDesc *__restrict__ sd, const int *__restrict__ n_dev,
                  const LTask *__restrict__ lt, const SrcDesc *__restrict__ srcs,
                  const Grid *__restrict__ grids, const CellArr *__restrict__ carr,
                  const int *__restrict__ cells, const Blk *__restrict__ blk, int nblk, int *lcnt,
                  int *lidx, const long long *__restrict__ bbmin,
                  const long long *__restrict__ bbmax, int span) {
  constexpr int S_ = 4;
  // one strip's window of candidates, or the short ones of all strips
  constexpr int NST = (D == 3) ? 9 : 3;
  constexpr int CAP = NST * 88 > WIN ? NST * 88 : WIN;
  __shared__ float sf[D][CAP + 4];
  const int lb = xcd_block(nblk * S_);
  const Blk b = blk[lb / S_];
  const LTask L = lt[b.item];
  const int lane = threadIdx.x, sl = lane % S_;
  const int i = b.first + (lb % S_) * (64 / S_) + lane / S_;
  const SysDesc S = sd[L.sys];
  const bool live = i < n_dev[L.sys];
  if (__builtin_amdgcn_ballot_w64(live) == 0ull) return;
  const int64_t gi = S.off + (live ? i : 0);
  double xi[D];
#pragma unroll
  for (int d = 0; d < D; ++d) xi[d] = P.x[d][gi];
  int2 *emask = reinterpret_cast<int2 *>(lidx + L.list_off) + i;
  int *ebase = lidx + L.list_off + 2 * (int64_t)L.maxnb * L.cap + i;
  double O[D];
  Screen<D> scr;
  screen_origin<D>(xi, O);
  scr.set(xi, O);
  int ne = 0;  // entries of this target
  int cq = 0;  // entries of the current source
  for (int q = L.src_begin; q < L.src_end; ++q) {
    const SrcDesc Q = srcs[q];
    const Grid G = grids[Q.grid];
    cq = 0;
    if (G.ncells > 0) {
      const int *cs = cells + carr[Q.carr].off;
      const int self_j = Q.pk == PK_SELF ? i : -1;
      const double c2 = Q.cutoff2;
      const int64_t poff = sd[Q.partner].off;
      bool act = live && scr.finite;  // as in k_nlist
      scr.source(c2, Q.cell);
      if (Q.pk == PK_DYNAMIC && bbmin) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
          const double mn = double_of(bbmin[Q.partner * 3 + d]);
          const double mx = double_of(bbmax[Q.partner * 3 + d]);
          const double gap = mn - xi[d] > xi[d] - mx ? mn - xi[d] : xi[d] - mx;
          act = act && !(gap > Q.cell * (1.0 + 1e-9));
        }
      }
      int c[D];
      target_cell<D>(xi, G, Q.cell, c);
      if (__builtin_amdgcn_ballot_w64(act) != 0ull) {
        // every strip's range up front: one latency instead of one a strip
        int n0[NST], n1[NST];
#pragma unroll
        for (int st = 0; st < NST; ++st) {
          n0[st] = n1[st] = 1;
          if (act) {
            const int sb = strip_base<D>(c, G, st);
            n0[st] = cs[sb];
            n1[st] = cs[sb + 3];
          }
        }
        int base = 0;
        unsigned lo = 0u, hi = 0u;
        auto flush = [&]() {
          lo = quad_or(lo);
          hi = quad_or(hi);
          const unsigned sdl = (unsigned)(self_j - base);
          const unsigned sbit = 1u << (sdl & 31u);
          lo &= sdl < 32u ? ~sbit : ~0u;
          hi &= sdl - 32u < 32u ? ~sbit : ~0u;
          if (live && (lo | hi) != 0u) {
            if (ne < L.maxnb && sl == 0) {
              emask[(int64_t)ne * L.cap] = make_int2((int)lo, (int)hi);
              ebase[(int64_t)ne * L.cap] = base;
            }
            ++ne;
            ++cq;
          }
          lo = hi = 0u;
        };
        // the target's candidates [js, je), staged from index js + o of sf on: the
        // same for its S lanes, so they store a full mask together
        auto walk = [&](int js, int je, int o, int64_t last) {
          if (js >= base + 64) {
            flush();
            base += 64;
          }
          while (true) {
            const int ce = je < base + 64 ? je : base + 64;
            const int jb = js > base ? js : base;
            // the four lanes take four candidates each in turn: lane sl those at
            // 4·sl of every 16
            const int n = ce - jb;
            unsigned part[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
              const int t = 16 * m + 4 * sl;
              unsigned sg = 0u;
              if (t < n) {
                if (screen4<D>(scr, sf, jb + o + t, sg) < 0.0f || scr.all)
                  sg = exact4<D>(P, xi, c2, poff + jb + t, last);
                sg = __brev(sg) >> 28;
              }
              part[m] = sg << (4 * sl);
            }
            unsigned long long cur =
                ((unsigned long long)(part[2] | part[3] << 16) << 32) | (part[0] | part[1] << 16);
            cur = (cur & (~0ull >> (64 - n))) << (jb - base);
            lo |= (unsigned)cur;
            hi |= (unsigned)(cur >> 32);
            if (base + 64 >= je) break;
            flush();
            base += 64;
          }
        };
        // where the strips' unions of ranges are short (the targets of a wavefront
        // in one cell column) all are staged together: a latency or two for the
        // source instead of one a strip
        int g0[NST], off[NST], tot = 0, most = 0;
        unsigned g1[NST];  // lengths
#pragma unroll
        for (int st = 0; st < NST; ++st) {
          const bool any = n0[st] < n1[st];
          g0[st] = wave_red_dpp<false>(any ? n0[st] - 1 : INT_MAX);
          const int e = wave_red_dpp<true>(any ? n1[st] - 1 : INT_MIN);
          g1[st] = e > g0[st] ? (unsigned)(e - g0[st]) : 0u;  // 0: no range
          off[st] = tot;
          tot = g1[st] < (unsigned)CAP ? tot + (int)g1[st] : CAP + 1;
          tot = tot < CAP ? tot : CAP + 1;
          most = (int)g1[st] > most ? (int)g1[st] : most;
        }
        if (tot <= CAP && most <= 128) {
          __syncthreads();  // the previous source's candidates have been read
#pragma unroll
          for (int h = 0; h < 128; h += 64) {
            if (h >= most) break;
            double x[NST][D];
#pragma unroll
            for (int st = 0; st < NST; ++st) {
              const int t = h + lane < (int)g1[st] ? h + lane : 0;
#pragma unroll
              for (int k = 0; k < D; ++k)
                x[st][k] = g1[st] != 0u ? P.x[k][poff + g0[st] + t] : 0.0;
            }
#pragma unroll
            for (int st = 0; st < NST; ++st)
              if (h + lane < (int)g1[st]) {
#pragma unroll
                for (int k = 0; k < D; ++k)
                  sf[k][off[st] + h + lane] = scr.stage(x[st][k], O[k]);
              }
          }
          __syncthreads();
#pragma unroll
          for (int st = 0; st < NST; ++st) {
            if (g1[st] == 0u) continue;  // uniform
            const int j0 = n0[st] - 1, j1 = n1[st] - 1;
            base = j0;
            if (j0 < j1) walk(j0, j1, off[st] - g0[st], poff + g0[st] + (int)g1[st] - 1);
            flush();
          }
        } else {
#pragma unroll
          for (int st = 0; st < NST; ++st) {
            const int j0 = n0[st] - 1, j1 = n1[st] - 1;
            bool pend = j0 < j1;
            if (__builtin_amdgcn_ballot_w64(pend) == 0ull) continue;
            base = j0;
            const int wmax = wave_red_dpp<true>(j1 - j0);
            while (true) {
              const int glo = wave_red_dpp<false>(pend ? j0 : INT_MAX);
              if (glo == INT_MAX) break;
              const bool mem = pend && j0 - glo <= span * wmax;
              const int ghi = wave_red_dpp<true>(mem ? j1 : INT_MIN);
              for (int w0 = glo; w0 < ghi; w0 += WIN) {
                const int w1 = ghi - w0 < WIN ? ghi : w0 + WIN;
                __syncthreads();  // the previous window has been read
                for (int t = lane; t < w1 - w0; t += 64) {
#pragma unroll
                  for (int k = 0; k < D; ++k) sf[k][t] = scr.stage(P.x[k][poff + w0 + t], O[k]);
                }
                __syncthreads();
                const int js = j0 > w0 ? j0 : w0;
                const int je = mem ? (j1 < w1 ? j1 : w1) : 0;
                if (js < je) walk(js, je, -w0, poff + w1 - 1);
              }
              if (mem) pend = false;
            }
            flush();
          }
        }
      }
    }
    if (live && sl == 0) lcnt[L.cnt_off + (int64_t)(q - L.src_begin) * L.cap + i] = cq;
  }
  if (live && sl == 0)
    lcnt[L.cnt_off + (int64_t)(L.src_end - L.src_begin) * L.cap + i] = ne > L.maxnb ? 1 : 0;
}

// Functors over the accepted partners of each target (one stage).
template <int D, typename R, int FAM, bool CNT>
__global__ void __launch_bounds__(GR_BLOCK)
    k_sweep_list(Pool<R> P, const SysDesc *__restrict__ sd, const int *__restrict__ n_dev,
                 const Task *__restrict__ tasks, const SrcDesc *__restrict__ srcs,
                 const Grid *__restrict__ grids, const CellArr *__restrict__ carr,
                 const int *__restrict__ cells, const Blk *__restrict__ blk, int nblk,
                 unsigned long long *pair_count, const LTask *__restrict__ lt,
                 const int *__restrict__ lcnt, const int *__restrict__ lidx) {
  const Blk b = blk[xcd_block(nblk)];
  const Task T = tasks[b.item];
  // a task without a list (ltask < 0) walks the cells
  const LTask L = lt[T.ltask >= 0 ? T.ltask : 0];
  const int i = b.first + threadIdx.x;
  const SysDesc S = sd[T.sys];
  const bool live = i < n_dev[T.sys];
  const int64_t gi = S.off + (live ? i : 0);
  Gather<D, R, FAM> Gt;
  Gt.load(P, S, T, gi);
  unsigned long long ns = 0, no = 0;
  const int nls = L.src_end - L.src_begin;
  const bool overflow =
      live && (T.ltask < 0 || lcnt[L.cnt_off + (int64_t)nls * L.cap + i] != 0);
  if (overflow) {
    gather_direct<D, R, FAM>(Gt, P, sd, T, srcs, grids, carr, cells, i, ns, no);
  } else if (live) {
    const int2 *emask = reinterpret_cast<const int2 *>(lidx + L.list_off) + i;
    const int *ebase = lidx + L.list_off + 2 * (int64_t)L.maxnb * L.cap + i;
    for (int q = T.src_begin; q < T.src_end; ++q) {
      const SrcDesc Q = srcs[q];
      const int64_t poff = sd[Q.partner].off;
      SrcK<R> K;
      K.load(Q);
      int e = 0;
      for (int l = 0; l < Q.lsrc; ++l) e += lcnt[L.cnt_off + (int64_t)l * L.cap + i];
      const int eend = e + lcnt[L.cnt_off + (int64_t)Q.lsrc * L.cap + i];
      const double da = (Q.pk == PK_DYNAMIC) ? Gt.da_of(Q) : 0.0;
      // the next entry is loaded while its predecessor is popped
      const bool nb = needs_b<FAM>(Q);
      unsigned long long m = 0ull;
      int base = 0;
      int2 mpre = make_int2(0, 0);
      int bpre = 0;
      if (e < eend) {
        mpre = emask[(int64_t)e * L.cap];
        bpre = ebase[(int64_t)e * L.cap];
      }
      auto next = [&](int &j) -> bool {
        if (m == 0ull) {  // next entry (entries hold at least one partner)
          if (e >= eend) return false;
          base = bpre;
          m = ((unsigned long long)(unsigned)mpre.y << 32) | (unsigned)mpre.x;
          ++e;
          if (e < eend) {
            mpre = emask[(int64_t)e * L.cap];
            bpre = ebase[(int64_t)e * L.cap];
          }
        }
        j = base + __builtin_ctzll(m);
        m &= m - 1ull;
        return true;
      };
      constexpr bool CMP = Gather<D, R, FAM>::COMPACT;
      // prefetching the next partner pays in 3D and for the fluid-only force
      // sweeps; the 2D strain-rate and Cauchy sweeps run faster without it
      // (measured: 3D dam break, 3D visco-plastic columns, 2D EP ensemble)
      constexpr bool PREFETCH =
          D == 3 || FAM == FAM_FORCE_FLUID || FAM == FAM_FORCE_FLUID_INV;
      // compact Cauchy sources also read the partner's stress (the second
      // half only for NS > 4)
      const bool ns_a = CMP && needs_s<FAM>(Q), ns_b = ns_a && Gt.NS > 4;
      int jn = 0;
      RecA<R> An{};
      RecB<R> Bn{};
      RecC Cn{};
      RecS Sn{};
      auto fetch = [&]() {
        if constexpr (CMP) {
          Cn = P.rc[poff + jn];
          if (ns_a) Sn.a = P.rs[poff + jn].a;
          if (ns_b) Sn.b = P.rs[poff + jn].b;
        } else {
          An = P.ra[poff + jn];
          if (nb) Bn = P.rb[poff + jn];
        }
      };
      auto one = [&](auto dk, int64_t gj, const RecA<R> &Aj, const RecB<R> &Bj, const RecC &Cj,
                     const RecS &Sj) {
        double dx[D] = {};
        double r2 = 0.0;
        if constexpr (!CMP) {
#pragma unroll
          for (int d = 0; d < D; ++d) dx[d] = Gt.xi[d] - Aj.x[d];
          r2 = dx[0] * dx[0];
#pragma unroll
          for (int d = 1; d < D; ++d) r2 = r2 + dx[d] * dx[d];
        }
        if (CNT) {
          if (Q.pk == PK_SELF)
            ++ns;
          else
            ++no;
        }
        Gt.template pair<decltype(dk)::value>(P, Q, K, gj, Aj, Bj, Cj, Sj, dx, r2, da);
      };
      auto run = [&](auto dk) {
        if constexpr (PREFETCH) {
          // the next partner's records are loaded while the current pair is
          // evaluated (the copy out of the prefetch registers costs a move per
          // word; two buffers used in turn measured no faster, the compiler
          // still copied one of them)
          bool have = next(jn);
          if (have) fetch();
          while (have) {
            const int64_t gj = poff + jn;
            const RecA<R> Aj = An;
            const RecB<R> Bj = Bn;
            const RecC Cj = Cn;
            const RecS Sj = Sn;
            // the next record is loaded whether or not there is a next
            // partner (jn then still names this one): a conditional load
            // would make the compiler keep a copy of the buffer for the path
            // without it
            have = next(jn);
            fetch();
            one(dk, gj, Aj, Bj, Cj, Sj);
          }
        } else {
          // loaded at the top of each iteration: the other wavefronts of the
          // SIMD hide the latency, and no registers are copied
          while (next(jn)) {
            fetch();
            one(dk, poff + jn, An, Bn, Cn, Sn);
          }
        }
      };
      // the prefetching pair loop is compiled once for sources whose partner
      // is a dynamic boundary and once for the others (dk), so that the
      // pair's selects on the partner kind leave the loop (measured: 1 % off
      // the 3D sweeps; the 2D sweeps without prefetch gained nothing)
      if constexpr (PREFETCH && (Gather<D, R, FAM>::FORCE || FAM == FAM_STRAIN)) {
        if (Q.pk == PK_DYNAMIC)
          run(std::integral_constant<int, 1>{});
        else
          run(std::integral_constant<int, 0>{});
      } else {
        run(std::integral_constant<int, -1>{});
      }
    }
  }
  count_pairs<CNT>(pair_count, ns, no);
  if (live) Gt.store(P, S, T, gi);
}

// ---------------------------------------------------------------------------
// Functors with four lanes per target
// ---------------------------------------------------------------------------

// DPP move within quads of lanes: CTRL a quad_perm.
template <int CTRL>
__device__ __forceinline__ int quad_mov(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xF, 0xF, false);
}
template <int CTRL>
__device__ __forceinline__ float quad_mov(float v) {
  return __int_as_float(quad_mov<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double quad_mov(double v) {
  return __hiloint2double(quad_mov<CTRL>(__double2hiint(v)), quad_mov<CTRL>(__double2loint(v)));
}
// Transpose in the quad: lane s gets the four lanes' x[s], in lane order.
template <typename R>
__device__ __forceinline__ void quad_transpose(R *x, int s) {
  const bool b0 = s & 1, b1 = s & 2;
  // z[r] = x[s ^ r], to be read by lane s ^ r
  const R u0 = b0 ? x[1] : x[0], u1 = b0 ? x[0] : x[1];
  const R u2 = b0 ? x[3] : x[2], u3 = b0 ? x[2] : x[3];
  const R z0 = b1 ? u2 : u0, z1 = b1 ? u3 : u1, z2 = b1 ? u0 : u2, z3 = b1 ? u1 : u3;
  const R y1 = quad_mov<0xB1>(z1), y2 = quad_mov<0x4E>(z2), y3 = quad_mov<0x1B>(z3);
  // the value from lane k is y[k ^ s]
  const R v0 = b0 ? y1 : z0, v1 = b0 ? z0 : y1, v2 = b0 ? y3 : y2, v3 = b0 ? y2 : y3;
  x[0] = b1 ? v2 : v0;
  x[1] = b1 ? v3 : v1;
  x[2] = b1 ? v0 : v2;
  x[3] = b1 ? v1 : v3;
}

// The terms of one pair as a list, and a target's sums from one.
template <int D, typename R, int FAM>
struct Terms {
  static constexpr bool STRAIN = FAM == FAM_STRAIN;
  static constexpr int N = STRAIN ? (D == 2 ? 4 : 9) : D + 1;
  static constexpr int NG = (N + 3) / 4;  // groups of four
  template <typename G>
  __device__ static inline void get(const G &g, R *t) {
    if constexpr (!STRAIN) {
#pragma unroll
      for (int d = 0; d < D; ++d) t[d] = g.adv[d].t;
      t[D] = g.adr.t;
    } else if constexpr (D == 2) {
      t[0] = g.asr[0].t;
      t[1] = g.asr[1].t;
      t[2] = g.NS == 4 ? g.asr[3].t : g.asr[2].t;
      t[3] = g.avo[0].t;
    } else {
#pragma unroll
      for (int k = 0; k < 6; ++k) t[k] = g.asr[k].t;
#pragma unroll
      for (int k = 0; k < 3; ++k) t[6 + k] = g.avo[k].t;
    }
  }
  template <typename G>
  __device__ static inline void set(G &g, const double *t) {
    if constexpr (!STRAIN) {
#pragma unroll
      for (int d = 0; d < D; ++d) g.adv[d].s = t[d];
      g.adr.s = t[D];
    } else if constexpr (D == 2) {
      g.asr[0].s = t[0];
      g.asr[1].s = t[1];
      if (g.NS == 4)
        g.asr[3].s = t[2];
      else
        g.asr[2].s = t[2];
      g.avo[0].s = t[3];
    } else {
#pragma unroll
      for (int k = 0; k < 6; ++k) g.asr[k].s = t[k];
#pragma unroll
      for (int k = 0; k < 3; ++k) g.avo[k].s = t[6 + k];
    }
  }
};

// k_sweep_list with the four lanes of a quad per target (16 targets per
// wavefront, four times the wavefronts): lane s evaluates the partners of rank
// 4r + s of each list entry, then lane c adds component c of the four lanes'
// terms in their order.  Every sum is the one k_sweep_list makes, addition by
// addition, so the results are the same bits.  For launches of few targets
// (sweep_split_targets): there a lane's chain of loads bounds the launch, 0.7
// to 1.1 us a partner, and this one walks a quarter of it.  Rounds end with
// their list entry and the terms are exchanged (19 moves a round), so a launch
// that fills the chip is slower with it (3D dam break of 1.4M: 456 us against
// 349).
// Entries of a target staged in LDS (a multiple of 4; the others are loaded as
// they come up), and sources whose counts are.
#define SPLIT_ENTRIES 24
#define SPLIT_SOURCES 8
// Where that pays: not in the 2D fluid sweeps, whose few entries (three strips a
// source) come and go behind the walls' short sources.  Measured, us with the
// entries loaded one ahead / staged: 2D column of 13k in FP32 25.2 / 13.8 (Cauchy
// force), 3D dam break of 224k 74 / 69, 3D column of 16k 50.8 / 49.4, 2D dam break
// of 13k in FP64 15.9 / 17.2.
template <int D, int FAM>
constexpr bool split_stages() {
  return D == 3 || (FAM != FAM_FORCE_FLUID && FAM != FAM_FORCE_FLUID_INV);
}

template <int D, typename R, int FAM, bool CNT>
__global__ void __launch_bounds__(64)
    k_sweep_split(Pool<R> P, const SysDesc *__restrict__ sd, const int *__restrict__ n_dev,
                  const Task *__restrict__ tasks, const SrcDesc *__restrict__ srcs,
                  const Grid *__restrict__ grids, const CellArr *__restrict__ carr,
                  const int *__restrict__ cells, const Blk *__restrict__ blk, int nblk,
                  unsigned long long *pair_count, const LTask *__restrict__ lt,
                  const int *__restrict__ lcnt, const int *__restrict__ lidx, int nsub) {
  // nsub workgroups of 16 targets take one entry of the block table
  const int lb = xcd_block(nblk * nsub);
  const Blk b = blk[lb / nsub];
  const Task T = tasks[b.item];
  const LTask L = lt[T.ltask >= 0 ? T.ltask : 0];
  const int sl = threadIdx.x & 3;
  const int i = b.first + (lb % nsub) * 16 + (threadIdx.x >> 2);
  const SysDesc S = sd[T.sys];
  const bool live = i < n_dev[T.sys];
  const int64_t gi = S.off + (live ? i : 0);
  Gather<D, R, FAM> Gt;
  Gt.load(P, S, T, gi);
  unsigned long long ns = 0, no = 0;
  const int nls = L.src_end - L.src_begin;
  const bool overflow =
      live && (T.ltask < 0 || lcnt[L.cnt_off + (int64_t)nls * L.cap + i] != 0);
  // the targets' entries come to LDS first, all loads in flight together: in
  // the pair loop an entry's load would hold up the records behind it, and the
  // search has just written the entries on other XCDs, so each is a miss of L2
  constexpr bool STAGE = split_stages<D, FAM>();
  constexpr int LE = STAGE ? SPLIT_ENTRIES : 4, LS = STAGE ? SPLIT_SOURCES : 1;
  __shared__ unsigned long long s_mask[LE][16];
  __shared__ int s_base[LE][16];
  __shared__ int s_cnt[LS][16];
  const int tg = threadIdx.x >> 2;
  if (STAGE && live && !overflow) {
    const unsigned long long *em =
        reinterpret_cast<const unsigned long long *>(lidx + L.list_off) + i;
    const int *eb = lidx + L.list_off + 2 * (int64_t)L.maxnb * L.cap + i;
    int cnt[LS], tot = 0;
#pragma unroll
    for (int l = 0; l < LS; ++l)
      cnt[l] = l < nls ? lcnt[L.cnt_off + (int64_t)l * L.cap + i] : 0;
#pragma unroll
    for (int l = 0; l < LS; ++l) {
      tot += cnt[l];
      if (sl == 0) s_cnt[l][tg] = cnt[l];
    }
    unsigned long long m[LE / 4];
    int bs[LE / 4];
#pragma unroll
    for (int k = 0; k < LE / 4; ++k) {
      const int e = 4 * k + sl;
      m[k] = e < tot ? em[(int64_t)e * L.cap] : 0ull;
      bs[k] = e < tot ? eb[(int64_t)e * L.cap] : 0;
    }
#pragma unroll
    for (int k = 0; k < LE / 4; ++k) {
      s_mask[4 * k + sl][tg] = m[k];
      s_base[4 * k + sl][tg] = bs[k];
    }
  }
  if (STAGE) __syncthreads();
  using TT = Terms<D, R, FAM>;
  double sum[TT::NG] = {};
  // OV: targets without a list (it overflowed, or there is none): the quad tests
  // the candidates of the cell walk itself, 16 of every 64 a lane, and takes the
  // partners of those as an entry's.  Sweep where every list overflows, with one
  // lane of the four walking alone / with the quad / with one lane per target (us,
  // 3D dam break functor in FP32, 400 particles a cell): 27k targets 4040 / 950 /
  // 4410, 110k 9010 / 2500 / 4510.
  auto sources = [&](auto ovc) {
    constexpr bool OV = decltype(ovc)::value;
    Gather<D, R, FAM, Term<R>> Gp;
    Gp.load(P, S, T, gi);
    constexpr bool CMP = Gather<D, R, FAM>::COMPACT;
    const unsigned long long *emask =
        reinterpret_cast<const unsigned long long *>(lidx + L.list_off) + i;
    const int *ebase = lidx + L.list_off + 2 * (int64_t)L.maxnb * L.cap + i;
    // -1 for each of the lanes before this one in the quad, as the addend
    // that drops a mask's lowest bit
    const unsigned c1 = sl > 0 ? ~0u : 0u, c2 = sl > 1 ? ~0u : 0u, c3 = sl > 2 ? ~0u : 0u;
    // entries staged: all up to SPLIT_ENTRIES, if the sources' counts were
    const int staged = STAGE && nls <= LS ? LE : 0;
    auto wide = [](unsigned c) { return ((unsigned long long)c << 32) | c; };
    for (int q = T.src_begin; q < T.src_end; ++q) {
      const SrcDesc Q = srcs[q];
      auto count = [&](int l) {
        return STAGE && l < LS ? s_cnt[l][tg] : lcnt[L.cnt_off + (int64_t)l * L.cap + i];
      };
      int e = 0, eend = 0;
      if constexpr (!OV) {
        for (int l = 0; l < Q.lsrc; ++l) e += count(l);
        eend = e + count(Q.lsrc);
        if (e >= eend) continue;
      }
      const int64_t poff = sd[Q.partner].off;
      SrcK<R> K;
      K.load(Q);
      const double da = (Q.pk == PK_DYNAMIC) ? Gp.da_of(Q) : 0.0;
      const bool nb = needs_b<FAM>(Q);
      const bool ns_a = CMP && needs_s<FAM>(Q), ns_b = ns_a && Gp.NS > 4;
      // a functor without vorticity leaves those terms as the last source's
      // pair left them
      if constexpr (FAM == FAM_STRAIN) {
#pragma unroll
        for (int k = 0; k < 3; ++k) Gp.avo[k].t = (R)0;
      }
      unsigned long long m = 0ull;
      int base = 0, jn = 0;
      bool vn = false;
      unsigned long long mpre = 0ull;
      int bpre = 0;
      if (!STAGE && !OV) {
        mpre = emask[(int64_t)e * L.cap];
        bpre = ebase[(int64_t)e * L.cap];
      }
      // OV: the mask of the 64 candidates from `base` on, below `wend`
      auto test = [&](int wend) {
        const int self_j = Q.pk == PK_SELF ? i : -1;
        unsigned h[2] = {0u, 0u};
#pragma unroll
        for (int w = 0; w < 2; ++w) {
#pragma unroll 1
          for (int b4 = 0; b4 < 32; b4 += 16) {
            // four loads in flight; beyond the range's end its last one again
            double r2[4];
#pragma unroll
            for (int d = 0; d < D; ++d) {
              double xj[4];
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const int j = base + 32 * w + b4 + 4 * u + sl;
                xj[u] = P.x[d][poff + (j < wend ? j : wend - 1)];
              }
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const double dx = Gp.xi[d] - xj[u];
                r2[u] = d == 0 ? dx * dx : r2[u] + dx * dx;
              }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const int j = base + 32 * w + b4 + 4 * u + sl;
              h[w] |= (unsigned)(r2[u] < Q.cutoff2 && j < wend && j != self_j)
                      << (b4 + 4 * u + sl);
            }
          }
          h[w] = quad_or(h[w]);
        }
        m = ((unsigned long long)h[1] << 32) | h[0];
      };
      // the quad's next (up to four) partners: whether there are any, and
      // this lane's (jn, vn)
      auto next = [&]() -> bool {
        if (m == 0ull) {
          if (OV || e >= eend) return false;
          if constexpr (STAGE) {
            if (e < staged) {
              m = s_mask[e][tg];
              base = s_base[e][tg];
            } else {
              m = emask[(int64_t)e * L.cap];
              base = ebase[(int64_t)e * L.cap];
            }
            ++e;
          } else {
            base = bpre;
            m = mpre;
            ++e;
            if (e < eend) {
              mpre = emask[(int64_t)e * L.cap];
              bpre = ebase[(int64_t)e * L.cap];
            }
          }
        }
        unsigned long long w = m;
        w &= w + wide(c1);
        w &= w + wide(c2);
        w &= w + wide(c3);
        vn = w != 0ull;
        if (vn) jn = base + __builtin_ctzll(w);
        w &= w - 1ull;
        if (!vn) w = 0ull;
        // the mask after the quad's last lane
        m = ((unsigned long long)(unsigned)quad_mov<0xFF>((int)(w >> 32)) << 32) |
            (unsigned)quad_mov<0xFF>((int)w);
        return true;
      };
      RecA<R> An{};
      RecB<R> Bn{};
      RecC Cn{};
      RecS Sn{};
      auto fetch = [&]() {
        if constexpr (CMP) {
          Cn = P.rc[poff + jn];
          if (ns_a) Sn.a = P.rs[poff + jn].a;
          if (ns_b) Sn.b = P.rs[poff + jn].b;
        } else {
          An = P.ra[poff + jn];
          if (nb) Bn = P.rb[poff + jn];
        }
      };
      auto run = [&](auto dk) {
        // a lane without a partner in the first round reads the entry's base
        bool have = next();
        if (!vn) jn = base;
        fetch();
        while (have) {
          const int64_t gj = poff + jn;
          const bool v = vn;
          const RecA<R> Aj = An;
          const RecB<R> Bj = Bn;
          const RecC Cj = Cn;
          const RecS Sj = Sn;
          have = next();
          fetch();
          R t[TT::NG * 4] = {};
          {
            double dx[D] = {};
            double r2 = 0.0;
            if constexpr (!CMP) {
#pragma unroll
              for (int d = 0; d < D; ++d) dx[d] = Gp.xi[d] - Aj.x[d];
              r2 = dx[0] * dx[0];
#pragma unroll
              for (int d = 1; d < D; ++d) r2 = r2 + dx[d] * dx[d];
            }
            if (CNT && v) {
              if (Q.pk == PK_SELF)
                ++ns;
              else
                ++no;
            }
            Gp.adr.t = (R)0;  // a static boundary pair adds no density term
            Gp.template pair<decltype(dk)::value>(P, Q, K, gj, Aj, Bj, Cj, Sj, dx, r2, da);
            TT::get(Gp, t);
          }
#pragma unroll
          for (int g = 0; g < TT::NG; ++g) {
            if (D == 3 && TT::STRAIN && g == 2 && !T.write_vor) continue;
#pragma unroll
            for (int k = 0; k < 4; ++k) t[4 * g + k] = v ? t[4 * g + k] : (R)0;
            quad_transpose(t + 4 * g, sl);
            // adding the zero of a lane without a partner changes nothing: no
            // sum is -0 (they start at +0)
#pragma unroll
            for (int k = 0; k < 4; ++k) sum[g] += (double)t[4 * g + k];
          }
        }
      };
      if constexpr (OV) {
        // (the quads of a wavefront test in step, then take their partners)
        const Grid G = grids[Q.grid];
        if (G.ncells <= 0) continue;
        const int *cs = cells + carr[Q.carr].off;
        int c[D];
        target_cell<D>(Gp.xi, G, Q.cell, c);
        for (int st = 0; st < (D == 3 ? 9 : 3); ++st) {
          const int sb = strip_base<D>(c, G, st);
          const int wend = cs[sb + 3] - 1;
          for (base = cs[sb] - 1; base < wend; base += 64) {
            test(wend);
            if (m != 0ull) run(std::integral_constant<int, -1>{});
          }
        }
      } else if (Q.pk == PK_DYNAMIC) {
        run(std::integral_constant<int, 1>{});
      } else {
        run(std::integral_constant<int, 0>{});
      }
    }
  };
  if (overflow)
    sources(std::true_type{});
  else if (live)
    sources(std::false_type{});
  // every lane of the quad takes all its components
  double tot[TT::NG * 4];
#pragma unroll
  for (int g = 0; g < TT::NG; ++g) {
    tot[4 * g] = quad_mov<0x00>(sum[g]);
    tot[4 * g + 1] = quad_mov<0x55>(sum[g]);
    tot[4 * g + 2] = quad_mov<0xAA>(sum[g]);
    tot[4 * g + 3] = quad_mov<0xFF>(sum[g]);
  }
  TT::set(Gt, tot);
  count_pairs<CNT>(pair_count, ns, no);
  if (live && sl == 0) Gt.store(P, S, T, gi);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

// Up to this many targets a launch of force or strain-rate sweeps takes four
// lanes per target (k_sweep_split).  Measured, us with one / four lanes (FP32; the
// columns both stages): 3D dam breaks of 22k targets 89 / 38, 69k 88 / 54, 125k
// 87 / 66, 157k 98 / 77; visco-plastic columns 72k 119 / 86, 144k 143 / 128, 216k
// 176 / 167; 2D dam breaks, whose entries are not staged, 20k 21 / 14, 80k 21 / 18,
// 99k 21 / 22, 163k 27 / 29; EP columns 13k 66 / 30, 97k 80 / 48, 157k 86 / 67, 259k
// 97 / 94.  FP64: 3D 69k 166 / 103, 125k 149 / 139, 216k 218 / 218, columns 144k
// 279 / 241; 2D 80k 36 / 31, 99k 34 / 35, EP 97k 96 / 80, 157k 116 / 113, 259k
// 149 / 166.
template <int D, int FAM>
constexpr int64_t sweep_split_targets() {
  return D == 3 ? 150000 : split_stages<D, FAM>() ? 115000 : 90000;
}

template <int D, typename R, int FAM>
static void launch_one(hipStream_t s, const Pool<R> &P, const SweepArgs &a, bool cnt) {
  if constexpr (FAM == FAM_FORCE || FAM == FAM_FORCE_FLUID || FAM == FAM_FORCE_FLUID_INV ||
                FAM == FAM_STRAIN) {
    if (a.lt && (int64_t)a.nblk * a.block <= sweep_split_targets<D, FAM>()) {
      const int nsub = a.block / 16;
      if (cnt)
        k_sweep_split<D, R, FAM, true><<<a.nblk * nsub, 64, 0, s>>>(
            P, a.sd, a.n, a.tasks, a.srcs, a.grids, a.carr, a.cells, a.blk, a.nblk, a.pair_count,
            a.lt, a.lcnt, a.lidx, nsub);
      else
        k_sweep_split<D, R, FAM, false><<<a.nblk * nsub, 64, 0, s>>>(
            P, a.sd, a.n, a.tasks, a.srcs, a.grids, a.carr, a.cells, a.blk, a.nblk, a.pair_count,
            a.lt, a.lcnt, a.lidx, nsub);
      return;
    }
  }
  if (a.lt) {
    // the block table steps by a.block targets (64, 128 or 256)
    if (cnt)
      k_sweep_list<D, R, FAM, true><<<a.nblk, a.block, 0, s>>>(
          P, a.sd, a.n, a.tasks, a.srcs, a.grids, a.carr, a.cells, a.blk, a.nblk, a.pair_count,
          a.lt, a.lcnt, a.lidx);
    else
      k_sweep_list<D, R, FAM, false><<<a.nblk, a.block, 0, s>>>(
          P, a.sd, a.n, a.tasks, a.srcs, a.grids, a.carr, a.cells, a.blk, a.nblk, a.pair_count,
          a.lt, a.lcnt, a.lidx);
    return;
  }
  if (cnt)
    k_sweep<D, R, FAM, true><<<a.nblk, a.block, 0, s>>>(P, a.sd, a.n, a.tasks, a.srcs, a.grids,
                                                         a.carr, a.cells, a.blk, a.nblk,
                                                         a.pair_count);
  else
    k_sweep<D, R, FAM, false><<<a.nblk, a.block, 0, s>>>(P, a.sd, a.n, a.tasks, a.srcs, a.grids,
                                                          a.carr, a.cells, a.blk, a.nblk,
                                                          a.pair_count);
}

template <typename R>
void launch_sweep(hipStream_t s, const Pool<R> &P, const SweepArgs &a, int D, int fam, bool cnt) {
  if (a.nblk <= 0) return;
  if (D == 2) {
    if (fam == FAM_FORCE && a.fluid_only && a.inv) launch_one<2, R, FAM_FORCE_FLUID_INV>(s, P, a, cnt);
    else if (fam == FAM_FORCE && a.fluid_only) launch_one<2, R, FAM_FORCE_FLUID>(s, P, a, cnt);
    else if (fam == FAM_FORCE) launch_one<2, R, FAM_FORCE>(s, P, a, cnt);
    else if (fam == FAM_STRAIN) launch_one<2, R, FAM_STRAIN>(s, P, a, cnt);
    else if (fam == FAM_INTERP) launch_one<2, R, FAM_INTERP>(s, P, a, cnt);
    else if (fam == FAM_XSPH) launch_one<2, R, FAM_XSPH>(s, P, a, cnt);
    else launch_one<2, R, FAM_COUNT>(s, P, a, cnt);
  } else {
    if (fam == FAM_FORCE && a.fluid_only && a.inv) launch_one<3, R, FAM_FORCE_FLUID_INV>(s, P, a, cnt);
    else if (fam == FAM_FORCE && a.fluid_only) launch_one<3, R, FAM_FORCE_FLUID>(s, P, a, cnt);
    else if (fam == FAM_FORCE) launch_one<3, R, FAM_FORCE>(s, P, a, cnt);
    else if (fam == FAM_STRAIN) launch_one<3, R, FAM_STRAIN>(s, P, a, cnt);
    else if (fam == FAM_INTERP) launch_one<3, R, FAM_INTERP>(s, P, a, cnt);
    else if (fam == FAM_XSPH) launch_one<3, R, FAM_XSPH>(s, P, a, cnt);
    else launch_one<3, R, FAM_COUNT>(s, P, a, cnt);
  }
}
template void launch_sweep<float>(hipStream_t, const Pool<float> &, const SweepArgs &, int, int,
                                  bool);
template void launch_sweep<double>(hipStream_t, const Pool<double> &, const SweepArgs &, int, int,
                                   bool);

// Up to this many blocks of 64 targets the search takes four lanes per target:
// with one, such a launch has at most about two wavefronts per SIMD, and a
// wavefront's own chain of loads and tests is the launch's time.  Measured, us
// with one / four lanes: 3D dam breaks of 422 blocks 80 / 50, 1000 77 / 52,
// 1954 81 / 82, 3375 88 / 110, 5593 122 / 167 (columns of 1500 blocks 73 / 65,
// 2250 78 / 81); 2D of 313 blocks 19 / 16, 1250 19.1 / 19.4, 2552 23 / 31 (EP
// columns of 1600 blocks 20 / 24).
template <int D>
constexpr int nlist_split_blocks() {
  return D == 3 ? 1950 : 1200;
}
// Up to this many blocks the strips are staged together.  Measured, us strip by
// strip / together: 2D dam breaks of 79 blocks 15.0 / 13.2, 640 16.2 / 14.0, 1155
// 19.3 / 19.9; 3D of 125 41 / 38, 422 50 / 46, 615 48 / 53, 1000 52 / 65 (columns
// of 500 blocks 40 / 34).
template <int D>
constexpr int nlist_all_blocks() {
  return D == 3 ? 500 : 1000;
}

template <int D, typename R, int WIN>
static void nlist_one(hipStream_t s, const Pool<R> &P, const NlistArgs &a) {
  if (a.nblk <= nlist_all_blocks<D>()) {
    k_nlist_small<D, R, WIN><<<a.nblk * 4, 64, 0, s>>>(P, a.sd, a.n, a.lt, a.srcs, a.grids, a.carr,
                                                       a.cells, a.blk, a.nblk, a.lcnt, a.lidx,
                                                       a.bbmin, a.bbmax, a.span);
    return;
  }
  if (a.nblk <= nlist_split_blocks<D>()) {
    k_nlist_split<D, R, WIN, 4><<<a.nblk * 4, 64, 0, s>>>(P, a.sd, a.n, a.lt, a.srcs, a.grids,
                                                          a.carr, a.cells, a.blk, a.nblk, a.lcnt,
                                                          a.lidx, a.bbmin, a.bbmax, a.span);
    return;
  }
  k_nlist<D, R, WIN><<<a.nblk, 64, 0, s>>>(P, a.sd, a.n, a.lt, a.srcs, a.grids, a.carr, a.cells,
                                           a.blk, a.nblk, a.lcnt, a.lidx, a.bbmin, a.bbmax,
                                           a.span);
}

template <typename R>
void launch_nlist(hipStream_t s, const Pool<R> &P, const NlistArgs &a, int D) {
  if (a.nblk <= 0) return;
  if (D == 2) {
    if (a.win == 64) nlist_one<2, R, 64>(s, P, a);
    else if (a.win == 256) nlist_one<2, R, 256>(s, P, a);
    else if (a.win == 512) nlist_one<2, R, 512>(s, P, a);
    else nlist_one<2, R, 128>(s, P, a);
  } else {
    if (a.win == 64) nlist_one<3, R, 64>(s, P, a);
    else if (a.win == 256) nlist_one<3, R, 256>(s, P, a);
    else if (a.win == 512) nlist_one<3, R, 512>(s, P, a);
    else nlist_one<3, R, 128>(s, P, a);
  }
}
template void launch_nlist<float>(hipStream_t, const Pool<float> &, const NlistArgs &, int);
template void launch_nlist<double>(hipStream_t, const Pool<double> &, const NlistArgs &, int);

}  // namespace gr
