// Dynamics right-hand side and update for one RK stage (CAAR), plus the
// small element-wise kernels of the step (dp3d from ps).
//
// A block is one element; a lane holds GLL point pt at CL (2, 4 or 6) consecutive
// levels of it, so the 16 lanes of one group form a slab at each of its
// levels (cross-lane derivatives) and the whole column's state stays in
// registers over the phases:
//   in: the stage's state, read from the state arrays (stage 1) or gathered
//       and assembled from the previous stage's pre-exchange values, so no
//       exchange launch runs between stages
//   A: vdp, vn0 += w vdp, div(vdp); dp and div(vdp) -> LDS
//   scans: pressure and the sum of div(vdp) above, one lane per column each
//   B: omega/p, T, dp3d; Rgas*T_v*dp/(2p) -> LDS
//   scan: the sum of those terms below
//   D: energy gradient, vorticity, v
// The column scans stay serial recurrences in the reference's order
// (CaarFunctorImpl.hpp:621-650, 689-729, 854-889).
//
// Bound: the latency of a block's phases (about 10 us) against four resident
// blocks per CU; 702 MB move per stage at ne30 L72 (about 14 fields).  One
// lane per column and chunk, re-reading the state in every phase, moved 25
// fields per stage and needed an exchange launch between the stages: five
// stages with their exchanges and the RK combination took 1.85 ms at ne30 L72
// then and 1.13 ms now, 243 and 122 us at ne8.
//
// With rsplit == 0 phases B and D also carry the Eulerian vertical advection
// (eta_dot_dpdn from the column sums of div(v dp)); it reads neighbour levels
// of the state arrays, so its stages keep their exchange launches.
#include "kernels.hpp"

namespace hx {

// virtual temperature from the water vapour qv (as Qdp)
__device__ __forceinline__ double virtual_t(double qv, double t, double dp) {
  double qt = qv / dp;
  qt *= (RWATER_VAPOR / RGAS - 1.0);
  qt += 1.0;
  return t * qt;
}

// LDS rows: the lanes' levels, whole batches of eight (the lanes past the last
// level cover the rest: a wave is 4*CL levels)
template <int CL>
__host__ __device__ inline int caar_rows(int nlev) {
  return ((nlev + CL - 1) / CL * CL + 7) & ~7;
}

// GATHER: the input state is assembled from a.pre (else read from a.v, a.t,
// a.dp); BASE: the state the tendency is added to: 0 the input itself, 1
// a.bv, a.bt, a.bdp, 2 the combination (5 u1 - u0)/4 of a.u1* and a.b* (u0),
// which is also stored in a.w* (prim_advance_exp.cpp:139-156).
// Only the state stays in registers (u, w, t, dp: 122 VGPRs in all with four
// levels per lane, 138 with six); pressure, div(v dp) and the sums are read
// back from LDS, and pin keeps the levels of a lane apart (interleaved they
// held 206 VGPRs, two waves per SIMD).
template <int CL, bool RS0, bool GATHER, int BASE, bool MOIST, int MAXT>
__global__ __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(MAXT > 512 ? 4 : 3))) void caar_kernel(CaarArgs a) {
  extern __shared__ double xs[];
  const int L = a.nlev;
  const int pt = threadIdx.x & 15, ch = threadIdx.x >> 4;
  const int nch = (L + CL - 1) / CL;
  const int ie = xcd_block(blockIdx.x, gridDim.x);
  const int k0 = ch * CL;
  const bool on = ch < nch;
  // (rows past the last level: zero phi terms, otherwise unused)
  const int R = caar_rows<CL>(L);
  double *const sp = xs + pt;      // dp, then p   [R][16]
  double *const sd = sp + R * 16;  // div(v dp), then the phi terms
  double *const ss = sd + R * 16;  // sums of div(v dp) above, then of the phi terms below
  const double eta = a.eta_ave_w, dt = a.dt;
  // the element's part of the arrays (uniform), and the lane's offsets in it;
  // levels past the last are computed on the last one's values, or on the
  // padding of the pre-exchange layout, and not stored
  const size_t sE = (size_t)ie * L * 16, vE = 2 * sE;
  const size_t lf = sc_field<CL>(L);
  auto lv = [&](int j) { return k0 + j < L ? k0 + j : L - 1; };
  auto si = [&](int j) { return (unsigned)(lv(j) * 16 + pt); };
  auto vi = [&](int j) { return (unsigned)(lv(j) * 32 + pt); };

  // the base; the combination is formed and stored first and read back by the
  // lane that stored it (kept in registers it spilled)
  const double *bv_ = BASE == 2 ? a.wv : a.bv, *bt_ = BASE == 2 ? a.wt : a.bt, *bdp_ = BASE == 2 ? a.wdp : a.bdp;
  if (BASE == 2 && on) {
#pragma unroll
    for (int j = 0; j < CL; ++j) {
      if (k0 + j >= L) break;
      const double w0 = (5.0 * (a.u1v + vE)[vi(j)] - (a.bv + vE)[vi(j)]) / 4.0;
      const double w1 = (5.0 * (a.u1v + vE)[vi(j) + 16] - (a.bv + vE)[vi(j) + 16]) / 4.0;
      const double w2 = (5.0 * (a.u1t + sE)[si(j)] - (a.bt + sE)[si(j)]) / 4.0;
      const double w3 = (5.0 * (a.u1dp + sE)[si(j)] - (a.bdp + sE)[si(j)]) / 4.0;
      (a.wv + vE)[vi(j)] = w0;
      (a.wv + vE)[vi(j) + 16] = w1;
      (a.wt + sE)[si(j)] = w2;
      (a.wdp + sE)[si(j)] = w3;
    }
  }
  double u[CL], w[CL], t[CL], dp[CL];
  if (on) {
    if (GATHER) {
      const ScGather<double, CL> g(a.pre, 4 * lf, ie, pt, k0, a.src);
      const double r = a.m.rspheremp[(size_t)ie * 16 + pt];
      {
        double x[2][CL];
        g.sum({2 * lf, 3 * lf}, x);
#pragma unroll
        for (int j = 0; j < CL; ++j) {
          t[j] = x[0][j] * r;
          dp[j] = x[1][j] * r;
          pin(t[j]);
          pin(dp[j]);
        }
      }
      g.field(0, r, u);
      g.field(lf, r, w);
      if (a.out_v) {
#pragma unroll
        for (int j = 0; j < CL; ++j) {
          if (k0 + j >= L) break;
          (a.out_v + vE)[vi(j)] = u[j];
          (a.out_v + vE)[vi(j) + 16] = w[j];
          (a.out_t + sE)[si(j)] = t[j];
          (a.out_dp + sE)[si(j)] = dp[j];
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < CL; ++j) {
        u[j] = (a.v + vE)[vi(j)];
        w[j] = (a.v + vE)[vi(j) + 16];
        t[j] = (a.t + sE)[si(j)];
        dp[j] = (a.dp + sE)[si(j)];
      }
    }
  }
  // (the element's metric is loaded where a phase first needs it: held over
  // the scans it spilled)
  ElemLane e;
  const unsigned e4 = (unsigned)(ie * 64 + pt), e1 = (unsigned)(ie * 16 + pt);
#pragma unroll
  for (int k = 0; k < 4; ++k) e.Dinv[k] = a.m.Dinv[e4 + 16 * k];
  e.metdet = a.m.metdet[e1];
  DvvLane d;
  load_dvv(a.m.dvv, pt, d);
  double tv[CL];
  if (MOIST && on) {
    const double *qE = a.qdp_n0 + (size_t)ie * a.qsize * L * 16;
#pragma unroll
    for (int j = 0; j < CL; ++j) tv[j] = virtual_t(qE[si(j)], t[j], dp[j]);
  }
  // ---------------------------------------------------------------- A
  // (a stage of weight 0 leaves the accumulators alone; stages 2 to 4 have none)
  const bool acc = eta != 0.0;
  // the first stage of a step starts them and keeps its dp (a launch that cleared
  // them first cost 16 us of the step at 1536 elements L72, 73 at 5400, and as
  // many bytes again where they were read back)
  const bool start = BASE == 0 && a.derived_dp;
  if (on) {
    double q0[CL], q1[CL];
#pragma unroll
    for (int j = 0; j < CL; ++j) q0[j] = q1[j] = 0.0;
    if (acc && !start) {
#pragma unroll
      for (int j = 0; j < CL; ++j) {
        q0[j] = (a.vn0 + vE)[vi(j)];
        q1[j] = (a.vn0 + vE)[vi(j) + 16];
      }
    }
#pragma unroll
    for (int j = 0; j < CL; ++j) {
      pin(u[j]);
      pin(w[j]);
      pin(dp[j]);
      const double vdp0 = u[j] * dp[j], vdp1 = w[j] * dp[j];
      if (acc && k0 + j < L) {
        (a.vn0 + vE)[vi(j)] = q0[j] + eta * vdp0;
        (a.vn0 + vE)[vi(j) + 16] = q1[j] + eta * vdp1;
      }
      if (start && k0 + j < L) (a.derived_dp + sE)[si(j)] = dp[j];
      sp[(k0 + j) * 16] = dp[j];
      sd[(k0 + j) * 16] = sph_div(e, d, vdp0, vdp1);
    }
  }
  lds_barrier();
  // p(k) = p(k-1) + (dp(k-1) + dp(k))/2, and the sums of div(v dp) above k,
  // on the first lanes of two waves (of one in a block of one wave); the
  // total of the latter goes to the row past the last level
  {
    const int wave = threadIdx.x >> 6, second = blockDim.x > 64 ? 1 : 0;
    if ((threadIdx.x & 63) < 16) {
      if (wave == 0) {
        double p = a.p_top, prev = 0.0;
        column_scan<false>(sp, sp, R, [&](double x) {
          p = p + 0.5 * (prev + x);
          prev = x;
          return p;
        });
      }
      if (wave == second) {
        double s = 0.0;
        column_scan<false>(sd, ss, R, [&](double x) {
          const double above = s;
          s = s + x;
          return above;
        });
        if (RS0) {
          ss[R * 16] = ss[(L - 1) * 16] + sd[(L - 1) * 16];
        }
      }
    }
  }
  // the base of T and dp3d one level ahead (the first across the barrier)
  double bt[CL], bdp[CL];
  auto base_tdp = [&](int j) {
    if (BASE != 0 && j < CL && on) {
      bt[j] = (bt_ + sE)[si(j)];
      bdp[j] = (bdp_ + sE)[si(j)];
    }
  };
  base_tdp(0);
  lds_barrier();
  // ---------------------------------------------------------------- B
  e.sph = opaque_ptr(a.m.spheremp)[e1];
  // rsplit == 0: eta_dot_dpdn(k) = hybi(k) * S(L-1) - S(k-1), eta(0) = 0,
  // with S the serial column sums of div(v dp) (:264-301)
  const double stotal = RS0 ? ss[R * 16] : 0.0;
  auto eta_of = [&](int k, double s_below) {  // s_below = S(k-1)
    return k == 0 ? 0.0 : (k < L ? a.hybi[k] * stotal - s_below : 0.0);
  };
  // vertical advection of x at level k (preq_vertadv, :497-597)
  auto vadv = [&](double xm, double xk, double xp, int k, double dpk, double ek, double ek1) {
    if (k == 0) {
      const double facp = (0.5 * 1 / dpk) * ek1;
      return facp * (xp - xk);
    }
    if (k == L - 1) {
      const double facm = (0.5 * (1 / dpk)) * ek;
      return facm * (xk - xm);
    }
    const double facp = 0.5 * (1 / dpk) * ek1;
    const double facm = 0.5 * (1 / dpk) * ek;
    return facp * (xp - xk) + facm * (xk - xm);
  };
  // the levels next to the lane's (rsplit == 0 reads the state arrays)
  const int km = k0 > 0 ? k0 - 1 : 0, kp = k0 + CL < L ? k0 + CL : L - 1;
  double *const preE = a.pre_out + (size_t)ie * 4 * lf;
  const unsigned po = (unsigned)(k0 * 16 + pt * CL);
  double ek[CL + 1];
  if (on) {
    double tm = 0.0, tp = 0.0;
    if (RS0) {
      tm = (a.t + sE)[km * 16 + pt];
      tp = (a.t + sE)[kp * 16 + pt];
    }
    double ot[CL], odp[CL];
#pragma unroll
    for (int j = 0; j < CL; ++j) {
      const int k = k0 + j;
      pin(u[j]);
      pin(w[j]);
      pin(t[j]);
      base_tdp(j + 1);
      const double p = sp[k * 16], integ = ss[k * 16], dv = sd[k * 16];
      const double tvj = MOIST ? tv[j] : t[j];
      const double om0 = acc && !start ? (a.omega + sE)[si(j)] : 0.0;
      double tva = 0.0, ek1 = 0.0;
      if (RS0) {
        ek[j] = eta_of(k, integ);
        ek1 = eta_of(k + 1, integ + dv);
        ek[j + 1] = ek1;
        tva = vadv(j ? t[j - 1] : tm, t[j], j + 1 < CL && k + 1 < L ? t[j + 1] : tp, k, dp[j], ek[j], ek1);
        if (acc && k < L) (a.eta_acc + sE)[si(j)] = (start ? 0.0 : (a.eta_acc + sE)[si(j)]) + eta * ek[j];
      }
      double gp0, gp1;
      sph_grad(e, d, p, gp0, gp1);
      const double vgrad_p = u[j] * gp0 + w[j] * gp1;
      const double om = (vgrad_p - (integ + 0.5 * dv)) / p;
      if (acc && k < L) (a.omega + sE)[si(j)] = om0 + eta * om;
      double gt0, gt1;
      sph_grad(e, d, t[j], gt0, gt1);
      const double vgrad_t = u[j] * gt0 + w[j] * gt1;
      const double ttens = (RS0 ? -tva : 0) - vgrad_t + KAPPA * tvj * om;
      ot[j] = (ttens * dt + (BASE == 0 ? t[j] : bt[j])) * e.sph;
      double tmp = ek1;
      tmp += dv;
      tmp -= RS0 ? ek[j] : 0.0;
      tmp = (BASE == 0 ? dp[j] : bdp[j]) - tmp * dt;
      odp[j] = e.sph * tmp;
      sd[k * 16] = k < L ? RGAS * tvj * (dp[j] * 0.5 / p) : 0.0;
      pin(ot[j]);
      pin(odp[j]);
      if (j & 1) {
        *(d2_t *)(preE + 2 * lf + po + (j - 1)) = d2_t{ot[j - 1], ot[j]};
        *(d2_t *)(preE + 3 * lf + po + (j - 1)) = d2_t{odp[j - 1], odp[j]};
      }
    }
  }
  if (!on) {
#pragma unroll
    for (int j = 0; j < CL; ++j)
      if (k0 + j < R) sd[(k0 + j) * 16] = 0.0;
  }
  lds_barrier();
  // the sums of the phi terms below each level, from the bottom
  if (threadIdx.x < 16) {
    double s = 0.0;
    column_scan<true>(sd, ss, R, [&](double x) {
      const double below = s;
      s = s + x;
      return below;
    });
  }
  // ---------------------------------------------------------------- D
  // the base of v, likewise
  double b0[CL], b1[CL];
  auto base_v = [&](int j) {
    if (BASE != 0 && j < CL && on) {
      b0[j] = (bv_ + vE)[vi(j)];
      b1[j] = (bv_ + vE)[vi(j) + 16];
    }
  };
  base_v(0);
  lds_barrier();
  {
    const double *D = opaque_ptr(a.m.D);
#pragma unroll
    for (int k = 0; k < 4; ++k) e.D[k] = D[e4 + 16 * k];
    e.fcor = opaque_ptr(a.m.fcor)[e1];
    e.phis = opaque_ptr(a.m.phis)[e1];
  }
  if (on) {
    double um = 0.0, up = 0.0, wm = 0.0, wp = 0.0;
    if (RS0) {
      um = (a.v + vE)[km * 32 + pt];
      wm = (a.v + vE)[km * 32 + pt + 16];
      up = (a.v + vE)[kp * 32 + pt];
      wp = (a.v + vE)[kp * 32 + pt + 16];
    }
    double o0[CL], o1[CL];
#pragma unroll
    for (int j = 0; j < CL; ++j) {
      const int k = k0 + j;
      pin(u[j]);
      pin(w[j]);
      pin(t[j]);
      base_v(j + 1);
      const double p = sp[k * 16];
      const double phi = e.phis + 2.0 * ss[k * 16] + sd[k * 16];
      const double tvj = MOIST ? tv[j] : t[j];
      double gp0, gp1;
      sph_grad(e, d, p, gp0, gp1);
      double eg0 = RGAS * (tvj / p) * gp0;
      double eg1 = RGAS * (tvj / p) * gp1;
      const double ephi = 0.5 * (u[j] * u[j] + w[j] * w[j]) + phi;
      sph_grad_update(e, d, ephi, eg0, eg1);
      double vort = sph_vort(e, d, u[j], w[j]);
      vort += e.fcor;
      double va0 = 0.0, va1 = 0.0;
      if (RS0) {
        const bool in = j + 1 < CL && k + 1 < L;
        va0 = vadv(j ? u[j - 1] : um, u[j], in ? u[j + 1] : up, k, dp[j], ek[j], ek[j + 1]);
        va1 = vadv(j ? w[j - 1] : wm, w[j], in ? w[j + 1] : wp, k, dp[j], ek[j], ek[j + 1]);
      }
      eg0 *= -1;
      eg0 += (RS0 ? -va0 : 0) + w[j] * vort;
      eg1 *= -1;
      eg1 += (RS0 ? -va1 : 0) - u[j] * vort;
      const double base0 = BASE == 0 ? u[j] : b0[j], base1 = BASE == 0 ? w[j] : b1[j];
      eg0 *= dt;
      eg0 += base0;
      eg1 *= dt;
      eg1 += base1;
      o0[j] = e.sph * eg0;
      o1[j] = e.sph * eg1;
      pin(o0[j]);
      pin(o1[j]);
      if (j & 1) {
        *(d2_t *)(preE + po + (j - 1)) = d2_t{o0[j - 1], o0[j]};
        *(d2_t *)(preE + lf + po + (j - 1)) = d2_t{o1[j - 1], o1[j]};
      }
    }
  }
}

template <int CL, bool RS0, bool GATHER, int BASE>
static void launch_caar_as(hipStream_t st, const CaarArgs &a) {
  const int nch = (a.nlev + CL - 1) / CL;
  const dim3 threads((nch * 16 + 63) & ~63);  // at most 1024 (REMAP_MAX_NLEV levels)
  const size_t lds = ((size_t)3 * caar_rows<CL>(a.nlev) + (RS0 ? 1 : 0)) * 16 * sizeof(double);
  auto go = [&](auto *kernel) { hipLaunchKernelGGL(kernel, dim3(a.nelem), threads, lds, st, a); };
  // six levels per lane (up to 96 levels: 256 lanes) and rsplit == 0 hold more
  // (168 VGPRs), which blocks of up to 512 lanes may
  constexpr int T = RS0 || CL > 4 ? 512 : 1024;
  if constexpr (RS0 && CL > 2) {
    if (threads.x > T) {
      go(a.qdp_n0 ? caar_kernel<CL, RS0, GATHER, BASE, true, 1024> : caar_kernel<CL, RS0, GATHER, BASE, false, 1024>);
      return;
    }
  }
  go(a.qdp_n0 ? caar_kernel<CL, RS0, GATHER, BASE, true, T> : caar_kernel<CL, RS0, GATHER, BASE, false, T>);
}

template <int CL>
static void launch_caar_cl(hipStream_t st, const CaarArgs &a) {
  if (!a.pre) launch_caar_as<CL, false, false, 0>(st, a);
  else if (!a.wv) launch_caar_as<CL, false, true, 1>(st, a);
  else launch_caar_as<CL, false, true, 2>(st, a);
}

template <int CL>
static void launch_caar_rs0(hipStream_t st, const CaarArgs &a) {
  if (a.wv) launch_caar_as<CL, true, false, 2>(st, a);
  else if (a.bv) launch_caar_as<CL, true, false, 1>(st, a);
  else launch_caar_as<CL, true, false, 0>(st, a);
}

void launch_caar(hipStream_t st, const CaarArgs &a) {
  if (!a.rsplit0) {
    if (a.chunk == 6) launch_caar_cl<6>(st, a);
    else if (a.chunk == 2) launch_caar_cl<2>(st, a);
    else launch_caar_cl<4>(st, a);
  } else if (a.chunk == 2) launch_caar_rs0<2>(st, a);
  else launch_caar_rs0<4>(st, a);
}

// ------------------------------------------------------------------ small
__global__ void dp3d_from_ps_kernel(int nelem, int nlev, const double *__restrict__ hyai,
                                    const double *__restrict__ hybi, double ps0, const double *__restrict__ ps,
                                    double *__restrict__ dp) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t n = (size_t)nelem * nlev * 16;
  if (i >= n) return;
  const int pt = i & 15;
  const int k = (i >> 4) % nlev;
  const int ie = (int)((i >> 4) / nlev);
  const double da = hyai[k + 1] - hyai[k], db = hybi[k + 1] - hybi[k];
  dp[i] = da * ps0 + db * ps[(size_t)ie * 16 + pt];
}

void launch_dp3d_from_ps(hipStream_t st, int nelem, int nlev, const double *hyai, const double *hybi, double ps0,
                         const double *ps, double *dp) {
  const size_t n = (size_t)nelem * nlev * 16;
  hipLaunchKernelGGL(dp3d_from_ps_kernel, dim3((n + 255) / 256), dim3(256), 0, st, nelem, nlev, hyai, hybi, ps0, ps,
                     dp);
}

}  // namespace hx
