// Euler tracer step with quasi-monotone limiters (EulerStepFunctorImpl.hpp
// and prim_advec_tracers_remap.cpp in the reference).
//
// Every kernel loops over all tracers of its points, so metric, dp and vstar
// are loaded once.  One remap interval's tracer step is
//   divdp_qmm  : divdp = div(vn0); stage-1 qmin/qmax
//   nbr_minmax
//   advect(1)
//   advect(2)  : gathers stage 1's exchange (extra field divdp_proj) and updates
//                qmin/qmax
//   dss_lap    : stage 2's exchange (extra field eta_dot_dpdn), stage-3
//                qmin/qmax, the first laplacian of the biharmonic
//   nbr_minmax
//   advect(3)  : gathers the laplacian's exchange, second laplacian
//   dss        : stage 3's exchange + SSP average (extra field omega_p)
// Limiter sums run over the 16 points in index order (slab_sum_serial) to
// round like the reference's serial reductions.
#include <type_traits>

#include "kernels.hpp"

namespace hx {

__device__ __forceinline__ bool slab_ie_k(size_t nslab_total, int nlev, size_t &slab, int &ie, int &k, int &pt) {
  const int b = xcd_block(blockIdx.x, gridDim.x);
  slab = (size_t)b * 16 + (threadIdx.x >> 4);
  pt = threadIdx.x & 15;
  if (slab >= nslab_total) return false;
  ie = (int)(slab / nlev);
  k = (int)(slab % nlev);
  return true;
}

// metric needed by divergence / weak laplacian only
__device__ __forceinline__ void load_elem_light(const MetricPtrs &m, int ie, int pt, ElemLane &e) {
  const size_t t = (size_t)ie * 64 + pt, s = (size_t)ie * 16 + pt;
#pragma unroll
  for (int j = 0; j < 4; ++j) e.Dinv[j] = m.Dinv[t + 16 * j];
  e.metdet = m.metdet[s];
  e.sph = m.spheremp[s];
  e.rsmp = m.rspheremp[s];
}

// --------------------------------------------------------------------------
// divdp = div(vn0), divdp_proj = divdp (EulerStepFunctorImpl.hpp:348-377) and
// the stage-1 compute_dp + compute_qmin_qmax (:406-485)
__global__ __launch_bounds__(256) void euler_divdp_qmm_kernel(EulerArgs a) {
  size_t slab;
  int ie, k, pt;
  if (!slab_ie_k((size_t)a.nelem * a.nlev, a.nlev, slab, ie, k, pt)) return;
  const int L = a.nlev, Q = a.qsize;
  ElemLane e;
  load_elem_light(a.m, ie, pt, e);
  DvvLane d;
  load_dvv(a.m.dvv, pt, d);
  const size_t s = slab * 16 + pt, v = slab * 32 + pt;
  const double dv = sph_div(e, d, a.vn0[v], a.vn0[v + 16]);
  a.divdp_w[s] = dv;
  a.divdp_proj_w[s] = dv;
  const double rhsmdt = a.rhs_multiplier * a.dt;
  const double dp = a.derived_dp[s] - rhsmdt * dv;
  const Recip rdp = recip(dp);  // Qdp / dp for every tracer
  // the Qdp of the next PD tracers is in flight during a tracer's
  // reductions: slot j of nx holds tracers j, j+PD, j+2PD, ..., refilled as
  // it is consumed (the loop body covers PD tracers, so no value moves
  // between registers: a move would wait for its load).  Every lane stores
  // the slab's bounds (the same value: measured faster here than a store
  // from one lane, whose branch makes the next wait cover the stores).
  if (Q <= 0) return;
  constexpr int PD = 4;
  const size_t q0i = ((size_t)ie * Q * L + k) * 16 + pt, qs = (size_t)L * 16;
  // (past the last tracer the last is reloaded: the loads stay unconditional)
  auto ld = [&](int q) { return a.qdp_n0[q0i + (size_t)(q < Q ? q : Q - 1) * qs]; };
  double nx[PD];
#pragma unroll
  for (int j = 0; j < PD; ++j) nx[j] = ld(j);
  auto tracer = [&](int q, double &slot) {
    const double x = div_r(slot, rdp);
    slot = ld(q + PD);
    const double mn = slab_min(x), mx = slab_max(x);
    double *ql = a.qlim + ((size_t)ie * Q + q) * ql_row(L);
    *(double2 *)(ql + ql_min(k)) = make_double2(mn, mx);
  };
  int q = 0;
  for (; q + PD <= Q; q += PD) {
#pragma unroll
    for (int j = 0; j < PD; ++j) tracer(q + j, nx[j]);
  }
#pragma unroll
  for (int j = 0; j < PD; ++j)
    if (q + j < Q) tracer(q + j, nx[j]);
}

// min/max of qlim over the element and its (up to 8) neighbours (:487-507).
// One thread per (tracer, element, level), tracer slowest, so a neighbour's
// qlim row is still in L2 when the next element row reads it.  The padding
// levels of a row get the last level's bounds: the advection works them like
// that level.  (Left unwritten, the limiter flattened them against the zeros of
// the allocation, 5 to 8 iterations instead of one, and their waves waited: at
// 3456 elements, 26 levels, 40 tracers the three stages took 2.47 ms, now 1.22;
// the bounds of the last level loaded by the stages instead: 1.30, and 2 to 3 %
// more at whole chunks.)
__global__ __launch_bounds__(256) void euler_nbr_minmax_kernel(EulerArgs a) {
  // XCD-aware block order: neighbouring elements' rows are read through one L2
  const size_t i = (size_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const int L = a.nlev, Q = a.qsize, Lp = (int)(ql_row(L) / 2);
  if (i >= (size_t)a.nelem * Q * Lp) return;
  const int k = (int)(i % Lp), kl = k < L ? k : L - 1;
  const int ie = (int)((i / Lp) % a.nelem);
  const int q = (int)(i / ((size_t)Lp * a.nelem));
  const size_t row = ((size_t)ie * Q + q) * ql_row(L);
  const double2 b = *(const double2 *)(a.qlim + row + ql_min(kl));
  double mn = b.x, mx = b.y;
  // an absent neighbour (-1) reads the element's own row, which leaves the
  // min and max unchanged: no branch, all loads in flight together
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int nb = a.nbr[ie * 8 + c];
    const size_t o = opaque_index(((size_t)(nb < 0 ? ie : nb) * Q + q) * ql_row(L) + ql_min(kl));
    const double2 n = *(const double2 *)(a.qlim + o);
    mx = vmax64(mx, n.y);
    mn = vmin64(mn, n.x);
  }
  *(double2 *)(a.qlim_new + row + ql_min(k)) = make_double2(mn, mx);
}

// ------------------------------------------------------------- lane mapping
// Advection, exchanges and laplacians: a wave is one element's 8-level chunk of
// the pre-exchange layout (lc_index), a lane one point at two levels k0, k0+1
// of it, for every tracer.  A wave then moves whole lines in 16-byte pieces,
// gathers its own points (no hand-off between lanes, no barrier), and two
// levels' chains run side by side.  Elements first, then chunks: the waves
// that run together on an XCD are neighbours at the same tracer, so neighbour
// copies come from its L2.  A last chunk that is not full costs a full one (its
// padding levels do the last level's work): 26 levels take the time of 32.
//
// What bounds them is HBM, if enough waves are in flight: a lane's two FP64
// chains take 100-130 registers, and the times follow the waves per SIMD which
// that leaves.  So the code is ordered to stay at four: bounds are loaded at the
// top of the tracer that uses them, the next tracer's gather once the
// laplacian's registers are free, and pin() keeps the two levels' chains apart.
// At 5400 elements, 72 levels, 40 tracers in FP64, ms:
//                one lane a level, an exchange of its own per stage  |  now
//   advect(1)                                        1.03            |  0.98
//   advect(2)    1.73 with its gather, 1.23 its exchange             |  1.26
//   dss_lap      0.96 bounds and laplacian                           |  1.57
//   advect(3)    1.43, 1.41 second laplacian and exchange            |  1.81
//   dss                                              1.23            |  1.19
//   in all                                           9.02            |  6.81
// dss, dss_lap and advect(3) move three tracer sets each (6.0 GB: 1.27 ms at the
// copy rate); FP64 arithmetic keeps advect(3) busy for 1.25 ms besides.  Capping
// registers with waves_per_eu spills (advect(3) 6.9 ms); two tracers' gathers
// ahead cost a wave (advect(3) 3.1, dss_lap 2.0 ms).
struct TLane {
  int ie, k0, pt;
  bool ok[2];  // the levels exist
  int lv[2];   // level, or the last one
};

__device__ __forceinline__ bool tracer_lane(int nelem, int nlev, TLane &t) {
  const long long w = (long long)xcd_block(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6);
  const int c = (int)(w / nelem);
  t.ie = __builtin_amdgcn_readfirstlane((int)(w % nelem));
  if (c * 8 >= nlev) return false;  // whole wave
  t.pt = threadIdx.x & 15;
  t.k0 = c * 8 + ((threadIdx.x >> 4) & 3) * 2;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    t.ok[j] = t.k0 + j < nlev;
    t.lv[j] = t.ok[j] ? t.k0 + j : nlev - 1;
  }
  return true;
}
static int tracer_blocks(const EulerArgs &a) {
  return (int)(((long long)a.nelem * ((a.nlev + 7) / 8) + 3) / 4);
}
// Small grids also split the tracers over blockIdx.y, up to TRACER_WAVES waves
// (two per SIMD): a wave's time is its chain of tracers there, and the setup
// that every share repeats (a fifth of a tracer's arithmetic, and loads that hit
// L2) runs on idle units.  96 elements, 26 levels, 4 tracers (384 waves):
// advect(3) 21.4 -> 12.0 us, advect(1) 17.9 -> 10.8, advect(2) 11.4 -> 7.5,
// dss_lap 9.2 -> 6.3.  Above it the repeated setup costs more: 3456 waves of 4
// tracers 23.3 -> 25.8 us for advect(3), 2904 of 7 tracers 20.3 -> 23.0 for
// dss_lap, in two shares.
constexpr long long TRACER_WAVES = 2048;
static dim3 tracer_grid(const EulerArgs &a) {
  const long long b = tracer_blocks(a);
  long long n = (TRACER_WAVES / 4 + b - 1) / b;
  n = n < a.qsize ? n : a.qsize;
  return dim3((unsigned)b, (unsigned)(n > 1 ? n : 1));
}
// this block's share [qa, qb) of the tracers
__device__ __forceinline__ bool tracer_share(int Q, int &qa, int &qb) {
  const int per = (Q + gridDim.y - 1) / gridDim.y;
  qa = blockIdx.y * per;
  qb = qa + per < Q ? qa + per : Q;
  return qa < qb;
}

// DSS gather of a lane's two levels from fields in the lc_index layout (element
// stride es).  load issues the loads of the field at offset off, masked to the
// lanes that have the source (the others read 0, which leaves a sum as it
// is), sum adds them in the reference's order.
template <typename T>
struct TGather {
  typedef typename vec2<T>::type V;
  gptr<T> p[4];
  bool edge, corner, third;
  V r[4];
  __device__ __forceinline__ TGather(const T *f0, size_t es, const TLane &t, const int *src) {
    const int *s = src + ((size_t)t.ie * 16 + t.pt) * 3;
    const int s0 = s[0], s1 = s[1], s2 = s[2];
    edge = s0 >= 0;
    corner = s1 >= 0;
    const gptr<T> f = (gptr<T>)f0 + lc_index(0, t.k0);
    p[0] = f + (size_t)t.ie * es + t.pt * 8;
    auto at = [&](int i) { return i >= 0 ? f + (size_t)(i >> 4) * es + (i & 15) * 8 : p[0]; };
    p[1] = at(s0);
    p[2] = at(s1);
    p[3] = at(s2);
    third = s2 >= 0;
  }
  __device__ __forceinline__ void load(size_t off) {
    r[0] = *(gptr<V>)(p[0] + off);
    r[1] = r[2] = r[3] = V{0, 0};
    if (edge) r[1] = *(gptr<V>)(p[1] + off);
    if (corner) {
      r[2] = *(gptr<V>)(p[2] + off);
      if (third) r[3] = *(gptr<V>)(p[3] + off);
    }
  }
  __device__ __forceinline__ double sum(int j) const {
    return (((double)r[0][j] + (double)r[1][j]) + (double)r[2][j]) + (double)r[3][j];
  }
};

// The weak divergence's columns of Dvv (TJ, TI) in LDS, a copy per wave: the
// laplacians read them for each tracer instead of holding 16 registers.
template <bool ON>
struct WkLds {
  d2_t *p;
  __device__ __forceinline__ WkLds() {
    __shared__ d2_t wk[ON ? 4 : 1][4][ON ? 64 : 1];
    p = &wk[ON ? threadIdx.x >> 6 : 0][0][ON ? threadIdx.x & 63 : 0];
  }
  __device__ __forceinline__ void put(const DvvLane &d) {
    p[0] = d2_t{d.TJ[0], d.TJ[1]};
    p[64] = d2_t{d.TJ[2], d.TJ[3]};
    p[128] = d2_t{d.TI[0], d.TI[1]};
    p[192] = d2_t{d.TI[2], d.TI[3]};
  }
  __device__ __forceinline__ void get(DvvLane &w) const {
    unsigned o = 0;
    asm volatile("" : "+v"(o));  // (read here: not hoisted out of the tracer loop)
    const d2_t w0 = p[o], w1 = p[o + 64], w2 = p[o + 128], w3 = p[o + 192];
    w.TJ[0] = w0[0], w.TJ[1] = w0[1], w.TJ[2] = w1[0], w.TJ[3] = w1[1];
    w.TI[0] = w2[0], w.TI[1] = w2[1], w.TI[2] = w3[0], w.TI[3] = w3[1];
  }
};

// ------------------------------------------------------------ limiters
// limiter_optim_iter_full (:767-823), one slab = one level of one tracer
__device__ __forceinline__ void limit8_slab(double mass, double minp, double maxp, double &x, double c) {
  const double tol_limiter = 5e-14;
  // (unrolled 15 times for two levels, it is 40 of a stage's 45 KB of code)
  for (int iter = 0; iter < NP2 - 1; ++iter) {
    double delta = 0;
    if (x > maxp) {
      delta = x - maxp;
      x = maxp;
    } else if (x < minp) {
      delta = x - minp;
      x = minp;
    }
    // (skipped when no slab of the wave clips; a slab that clips nothing
    // in a wave that does sums zeros: exactly 0, as if skipped)
    const double addmass = wave_any(delta != 0.0) ? slab_sum_serial(delta * c) : 0.0;
    if (fabs(addmass) <= tol_limiter * fabs(mass)) break;
    if (addmass > 0) {
      const double weightssum = slab_sum_serial(x < maxp ? c : 0.0);
      const double adw = addmass / weightssum;
      x += (x < maxp) ? adw : 0;
    } else {
      const double weightssum = slab_sum_serial(x > minp ? c : 0.0);
      const double adw = addmass / weightssum;
      x += (x > minp) ? adw : 0;
    }
  }
}

// limiter_clip_and_sum (:826-884)
__device__ __forceinline__ void limit9_slab(double minp, double maxp, double &x, double c) {
  double delta = 0;
  if (x > maxp) {
    delta = x - maxp;
    x = maxp;
  } else if (x < minp) {
    delta = x - minp;
    x = minp;
  }
  const double addmass = wave_any(delta != 0.0) ? slab_sum_serial(delta * c) : 0.0;
  if (addmass == 0) return;
  if (addmass > 0) {
    double fac = slab_sum_serial(c * (maxp - x));
    if (fac > 0) {
      fac = addmass / fac;
      x += fac * (maxp - x);
    }
  } else {
    double fac = slab_sum_serial(c * (x - minp));
    if (fac > 0) {
      fac = addmass / fac;
      x += fac * (x - minp);
    }
  }
}

// the bounds of a lane's two levels (equal in the lanes of a group), by the
// first two lanes of the group: one store of a whole line per wave (the padding
// levels' part of it too)
__device__ __forceinline__ void put_bounds(double *ql, const TLane &t, d2_t b0, d2_t b1) {
  if (t.pt < 2) *(d2_t *)(ql + 2 * t.pt) = t.pt ? b1 : b0;
}

// The assembled extra field of a lane's levels from its pre-exchange values
__device__ __forceinline__ void gather_extra(const EulerArgs &a, const double *pre, const TLane &t, double r,
                                             double (&x)[2]) {
  TGather<double> g(pre, lc_field(a.nlev), t, a.src);
  g.load(0);
#pragma unroll
  for (int j = 0; j < 2; ++j) x[j] = g.sum(j) * r;
}

// Setup phase (:585-626) + tracer phase (:571-687) for every tracer: div(vstar
// Qdp), the limiter, and the pre-exchange values of the stage.
// Stage 1 reads Qdp(n0).  Stage 2 gathers stage 1's exchange itself (the
// assembled stage-1 Qdp is never stored), and first updates the bounds with
// it (no neighbour exchange at this stage).  Stage 3 reads Qdp(np1) and
// gathers the exchange of the biharmonic's first laplacian; the second
// laplacian (:216-310) goes straight into the update.
// BIH: the biharmonic is 0 FP64, 1 the tensor form (FP64), 2 FP32 (mixed form).
template <bool MIXED, int STAGE, int BIH>
__global__ __launch_bounds__(256) void euler_advect_kernel(EulerArgs a) {
  TLane t;
  if (!tracer_lane(a.nelem, a.nlev, t)) return;
  const int L = a.nlev, Q = a.qsize, pt = t.pt;
  const size_t fs = lc_field(L), es = (size_t)Q * fs;
  // the tracer pre-exchange values are stored in FP32 in the mixed form (the
  // exchange sums them in FP64)
  using PreT = typename std::conditional<MIXED, float, double>::type;
  using LapT = typename std::conditional<BIH == 2, float, double>::type;
  using InT = typename std::conditional<STAGE == 3, LapT, PreT>::type;
  ElemLane e;
  load_elem_light(a.m, t.ie, pt, e);
  DvvLane d;
  load_dvv(a.m.dvv, pt, d);
  const double rhsmdt = (STAGE - 1) * a.dt;
  double dpproj[2], vs0[2], vs1[2], s1[2], fb[2];
  Recip rdp[2], rdpd[2];
  if (STAGE == 2) gather_extra(a, a.fdss_pre_in, t, e.rsmp, dpproj);
  const bool limit = a.limiter_option == 8 || a.limiter_option == 9;
  double fx[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const size_t s = ((size_t)t.ie * L + t.lv[j]) * 16 + pt, v = ((size_t)t.ie * L + t.lv[j]) * 32 + pt;
    if (STAGE == 2) {
      if (t.ok[j] && blockIdx.y == 0) a.divdp_proj_w[s] = dpproj[j];
    } else {
      dpproj[j] = a.divdp_proj[s];
    }
    const double dp = a.derived_dp[s] - rhsmdt * dpproj[j];
    vs0[j] = a.vn0[v] / dp;
    vs1[j] = a.vn0[v + 16] / dp;
    double dpdissk = dp - a.dt * a.divdp[s];
    if (STAGE == 3 && a.nu_p > 0) {
      const double diss_fac = -a.rhs_viss * a.dt * a.nu_q;
      dpdissk += diss_fac * a.dpdiss_bih[s] / e.sph;
    }
    fx[j] = a.fdss[s] * e.sph;
    // the divisors shared by the tracers: Qdp / dp (stage 2), ptens / dpdissk
    if (STAGE == 2) rdp[j] = recip(dp);
    rdpd[j] = recip(dpdissk);
    s1[j] = limit ? slab_sum_serial(e.sph * dpdissk) : 0.0;  // same for every tracer
    if (STAGE == 3) fb[j] = -a.rhs_viss * a.dt * a.nu_q * a.dp0[t.lv[j]];
  }
  if (blockIdx.y == 0) *(d2_t *)(a.fdss_pre + (size_t)t.ie * fs + lc_index(pt, t.k0)) = d2_t{fx[0], fx[1]};
  int qa, qb;
  if (!tracer_share(Q, qa, qb)) return;
  DvvLaneF df;
  float rmd = 0.f;
  if (MIXED) {
    load_dvvf(a.m.dvv, pt, df);
    rmd = (float)(1.0 / e.metdet * RREARTH);
  }
  ElemLaneF ef;
  if (STAGE == 3 && BIH == 2) load_elemf(a.m, t.ie, pt, ef);
  double tv[4], tvs[6];
  if (STAGE == 3 && BIH == 1) load_tensor(a.m, t.ie, pt, tv, tvs);
  const Recip rsph = recip(e.sph);
  constexpr bool TLDS = STAGE == 3 && BIH != 2;
  WkLds<TLDS> wk;
  if (TLDS) wk.put(d);
  // the element's parts of the arrays and the lane's offsets in them; tracer q
  // adds q uniform strides
  const size_t qs = (size_t)L * 16;
  const double *const qdpE = a.qdp_n0 + (size_t)t.ie * Q * qs;
  double *const qlE = a.qlim + (size_t)t.ie * Q * ql_row(L);
  PreT *const outE = (PreT *)a.qdp_pre + (size_t)t.ie * es;
  const unsigned qo0 = t.lv[0] * 16 + pt, qo1 = t.lv[1] * 16 + pt, lo = (unsigned)ql_min(t.k0),
                 oo = (unsigned)lc_index(pt, t.k0);
  TGather<InT> g((const InT *)(STAGE == 3 ? a.qbih_pre : a.qdp_pre_in), es, t, a.src);
  // tracer q+1's gather (stage 1: its Qdp) is loaded during tracer q's
  // arithmetic (past the last tracer the last is loaded again: the loads stay
  // unconditional)
  double nq0 = 0.0, nq1 = 0.0;
  auto fetch = [&](int q) {
    const size_t qq = q < qb ? q : qb - 1;
    if (STAGE == 1) {
      nq0 = (qdpE + qq * qs)[qo0];
      nq1 = (qdpE + qq * qs)[qo1];
    }
    if (STAGE != 1) g.load(qq * fs);
  };
  fetch(qa);
  for (int q = qa; q < qb; ++q) {
    double *const ql = qlE + (size_t)q * ql_row(L) + lo;
    const d2_t b0 = *(const d2_t *)ql, b1 = *(const d2_t *)(ql + 2);
    double minp[2] = {b0[0], b1[0]}, maxp[2] = {b0[1], b1[1]}, qd[2] = {nq0, nq1}, y[2];
    if (STAGE == 3) {
      qd[0] = (qdpE + q * qs)[qo0];
      qd[1] = (qdpE + q * qs)[qo1];
    }
    if (STAGE != 1) {
#pragma unroll
      for (int j = 0; j < 2; ++j) y[j] = g.sum(j) * e.rsmp;
    }
    double out[2], q0[2] = {0.0, 0.0};
    if (STAGE == 3) {
      DvvLane w = d;
      if (TLDS) wk.get(w);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        pin(y[j]);
        if constexpr (BIH == 2) q0[j] = (float)div_r(fb[j] * sph_laplacef(ef, df, (float)y[j]), rsph);
        else if constexpr (BIH == 1) q0[j] = div_r(fb[j] * sph_laplace_tensor(e, w, tv, y[j]), rsph);
        else q0[j] = div_r(fb[j] * sph_laplace(e, w, y[j]), rsph);
        pin(q0[j]);
      }
    }
    fetch(q + 1);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (STAGE == 2) qd[j] = y[j];
      pin(qd[j]);
      double ptens;
      if (MIXED) {
        // flux divergence in FP32 with compensated contractions; the update
        // qdp - dt*div + qbih stays FP64
        const double fa = vs0[j] * qd[j], fb2 = vs1[j] * qd[j];
        const float gv0 = (float)((e.Dinv[0] * fa + e.Dinv[2] * fb2) * e.metdet);
        const float gv1 = (float)((e.Dinv[1] * fa + e.Dinv[3] * fb2) * e.metdet);
        const float dv = (row_contractf(df.J, gv0) + col_contractf(df.I, gv1)) * rmd;
        ptens = (qd[j] + -a.dt * (double)dv + q0[j]);
      } else {
        ptens = sph_div_update(e, d, -a.dt, vs0[j], vs1[j], qd[j], q0[j]);
      }
      out[j] = ptens;
      pin(out[j]);
    }
    if (STAGE == 2) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const double xq = div_r(qd[j], rdp[j]);
        minp[j] = dmin(minp[j], slab_min(xq));
        maxp[j] = dmax(maxp[j], slab_max(xq));
        pin(minp[j]);
        pin(maxp[j]);
      }
    }
    bool moved = false;  // bounds of this lane's levels
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (!limit) continue;
      pin(out[j]);
      double x = div_r(out[j], rdpd[j]);
      const double cj = e.sph * rdpd[j].b;
      const double s0 = slab_sum_serial(x * cj);
      if (!(s1[j] <= 0)) {
        if (minp[j] < 0) {
          minp[j] = 0;
          moved = true;
        }
        if (s0 < minp[j] * s1[j]) {
          minp[j] = s0 / s1[j];
          moved = true;
        }
        if (s0 > maxp[j] * s1[j]) {
          maxp[j] = s0 / s1[j];
          moved = true;
        }
        if (a.limiter_option == 8) limit8_slab(s0, minp[j], maxp[j], x, cj);
        else limit9_slab(minp[j], maxp[j], x, cj);
        out[j] = x * rdpd[j].b;
      }
    }
    // stage 2 starts from stage 1's bounds; after it they are formed anew
    if (STAGE == 1 && moved)
      put_bounds(ql, t, d2_t{minp[0], maxp[0]}, d2_t{minp[1], maxp[1]});
    typedef typename vec2<PreT>::type V;
    *(V *)(outE + (size_t)q * fs + oo) = V{(PreT)(e.sph * out[0]), (PreT)(e.sph * out[1])};
  }
}

// The exchange of tracers and extra field, one wave an element's chunk: avg
// (stage 3) also forms the SSP average (Qdp(n0) + 2 Qdp(np1)) / 3 (:379-403).
template <bool F32>
__global__ __launch_bounds__(256) void euler_dss_kernel(EulerArgs a, int avg) {
  TLane t;
  if (!tracer_lane(a.nelem, a.nlev, t)) return;
  const int L = a.nlev, Q = a.qsize, pt = t.pt;
  const size_t fs = lc_field(L), es = (size_t)Q * fs, qs = (size_t)L * 16;
  const double r = a.m.rspheremp[(size_t)t.ie * 16 + pt];
  const unsigned qo[2] = {(unsigned)(t.lv[0] * 16 + pt), (unsigned)(t.lv[1] * 16 + pt)};
  if (blockIdx.y == 0) {
    double x[2];
    gather_extra(a, a.fdss_pre, t, r, x);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (t.ok[j]) st_stream(&(a.fdss + (size_t)t.ie * qs)[qo[j]], x[j]);
  }
  using PreT = typename std::conditional<F32, float, double>::type;
  const double *const avE = avg ? a.qdp_avg_n0 + (size_t)t.ie * Q * qs : nullptr;
  double *const outE = a.qdp_np1 + (size_t)t.ie * Q * qs;
  const TGather<PreT> g0((const PreT *)a.qdp_pre, es, t, a.src);
  // this launch's share of the tracers, QB in flight
  constexpr int QB = 4;
  int qa, qb;
  if (!tracer_share(Q, qa, qb)) return;
  for (int q = qa; q < qb; q += QB) {
    TGather<PreT> g[QB] = {g0, g0, g0, g0};
    double av[QB][2];
#pragma unroll
    for (int i = 0; i < QB; ++i) {
      const size_t qq = q + i < qb ? q + i : qb - 1;
      g[i].load(qq * fs);
      if (avg)
#pragma unroll
        for (int j = 0; j < 2; ++j) av[i][j] = (avE + qq * qs)[qo[j]];
    }
#pragma unroll
    for (int i = 0; i < QB; ++i) {
      if (q + i >= qb) break;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        double y = g[i].sum(j) * r;
        if (avg) y = div_c<3>(av[i][j] + (3.0 - 1) * y);
        if (t.ok[j]) st_stream(&(outE + (size_t)(q + i) * qs)[qo[j]], y);
      }
    }
  }
}

// The stage-2 exchange with what stage 3 starts from: the assembled Qdp(np1),
// its bounds (compute_dp + compute_qmin_qmax with rhs_multiplier 2, :406-485)
// and the first half of the tracer biharmonic, laplace(Q * dpdiss_ave / dp0)
// (:196-267).  LAP32: FP32 laplacian.
template <bool PRE32, bool LAP32>
__global__ __launch_bounds__(256) void euler_dss_lap_kernel(EulerArgs a) {
  TLane t;
  if (!tracer_lane(a.nelem, a.nlev, t)) return;
  const int L = a.nlev, Q = a.qsize, pt = t.pt;
  const size_t fs = lc_field(L), es = (size_t)Q * fs, qs = (size_t)L * 16;
  ElemLane e;
  load_elem_light(a.m, t.ie, pt, e);
  DvvLane d;
  ElemLaneF ef;
  DvvLaneF df;
  if (LAP32) {
    load_elemf(a.m, t.ie, pt, ef);
    load_dvvf(a.m.dvv, pt, df);
  } else {
    load_dvv(a.m.dvv, pt, d);
  }
  const unsigned qo[2] = {(unsigned)(t.lv[0] * 16 + pt), (unsigned)(t.lv[1] * 16 + pt)};
  double x[2], wdp[2];
  Recip rdp[2], rdp0[2];
  gather_extra(a, a.fdss_pre, t, e.rsmp, x);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const size_t s = (size_t)t.ie * qs + qo[j];
    if (t.ok[j] && blockIdx.y == 0) st_stream(&a.fdss[s], x[j]);
    rdp[j] = recip(a.derived_dp[s] - 2.0 * a.dt * a.divdp_proj[s]);
    rdp0[j] = recip(a.dp0[t.lv[j]]);
    wdp[j] = a.dpdiss_ave[s];
  }
  int qa, qb;
  if (!tracer_share(Q, qa, qb)) return;
  using PreT = typename std::conditional<PRE32, float, double>::type;
  using LapT = typename std::conditional<LAP32, float, double>::type;
  const bool scale = a.nu_p > 0;
  double *const outE = a.qdp_np1 + (size_t)t.ie * Q * qs;
  double *const qlE = a.qlim + (size_t)t.ie * Q * ql_row(L);
  LapT *const lapE = (LapT *)a.qbih_pre + (size_t)t.ie * es;
  const unsigned lo = (unsigned)ql_min(t.k0), oo = (unsigned)lc_index(pt, t.k0);
  TGather<PreT> g((const PreT *)a.qdp_pre, es, t, a.src);
  g.load((size_t)qa * fs);
  for (int q = qa; q < qb; ++q) {
    double y[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) y[j] = g.sum(j) * e.rsmp;
    g.load((size_t)(q + 1 < qb ? q + 1 : q) * fs);
    LapT lap[2];
    d2_t b[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      pin(y[j]);
      if (t.ok[j]) st_stream(&(outE + (size_t)q * qs)[qo[j]], y[j]);
      const double xq = div_r(y[j], rdp[j]);
      b[j] = d2_t{slab_min(xq), slab_max(xq)};
      const double yl = scale ? div_r(xq * wdp[j], rdp0[j]) : xq;
      if constexpr (LAP32) lap[j] = sph_laplacef(ef, df, (float)yl);
      else {
        lap[j] = sph_laplace(e, d, yl);
        pin(lap[j]);
      }
    }
    put_bounds(qlE + (size_t)q * ql_row(L) + lo, t, b[0], b[1]);
    typedef typename vec2<LapT>::type V;
    *(V *)(lapE + (size_t)q * fs + oo) = V{lap[0], lap[1]};
  }
}

static int slab_blocks(const EulerArgs &a) { return (int)(((size_t)a.nelem * a.nlev + 15) / 16); }

void launch_euler_divdp_qmm(hipStream_t st, const EulerArgs &a) {
  hipLaunchKernelGGL(euler_divdp_qmm_kernel, dim3(slab_blocks(a)), dim3(256), 0, st, a);
}

void launch_euler_nbr_minmax(hipStream_t st, const EulerArgs &a) {
  const size_t n = (size_t)a.nelem * a.qsize * (ql_row(a.nlev) / 2);
  hipLaunchKernelGGL(euler_nbr_minmax_kernel, dim3((n + 255) / 256), dim3(256), 0, st, a);
}

void launch_euler_advect(hipStream_t st, const EulerArgs &a, int stage) {
  const dim3 g = tracer_grid(a);
  auto go = [&](auto *kernel) { hipLaunchKernelGGL(kernel, g, dim3(256), 0, st, a); };
  if (stage == 1) go(a.mixed ? euler_advect_kernel<true, 1, 0> : euler_advect_kernel<false, 1, 0>);
  else if (stage == 2) go(a.mixed ? euler_advect_kernel<true, 2, 0> : euler_advect_kernel<false, 2, 0>);
  else if (a.bih32) go(euler_advect_kernel<true, 3, 2>);
  else if (a.mixed) go(a.consthv ? euler_advect_kernel<true, 3, 0> : euler_advect_kernel<true, 3, 1>);
  else go(a.consthv ? euler_advect_kernel<false, 3, 0> : euler_advect_kernel<false, 3, 1>);
}

void launch_euler_dss(hipStream_t st, const EulerArgs &a, int avg) {
  const dim3 g(tracer_blocks(a), (a.qsize + 7) / 8 < 1 ? 1 : (a.qsize + 7) / 8);
  if (a.mixed) hipLaunchKernelGGL(euler_dss_kernel<true>, g, dim3(256), 0, st, a, avg);
  else hipLaunchKernelGGL(euler_dss_kernel<false>, g, dim3(256), 0, st, a, avg);
}

void launch_euler_dss_lap(hipStream_t st, const EulerArgs &a) {
  const dim3 g = tracer_grid(a);
  auto go = [&](auto *kernel) { hipLaunchKernelGGL(kernel, g, dim3(256), 0, st, a); };
  if (a.bih32) go(euler_dss_lap_kernel<true, true>);
  else go(a.mixed ? euler_dss_lap_kernel<true, false> : euler_dss_lap_kernel<false, false>);
}

}  // namespace hx
