// Biharmonic hyperviscosity on the np1 state, one subcycle per call
// (HyperviscosityFunctorImpl.cpp:56-112, HyperviscosityFunctorImpl.hpp:71-257).
//   lap1      : weak laplacians of T, dp3d and the vector laplacian of v, formed
//               where the state is assembled: by the exchange of the last RK
//               stage (state_dss_kernel) and by the previous subcycle's update
//   lap2      : their exchange (gathered), second laplacians, dpdiss
//               accumulators, -nu scaling, the nu_top sponge on the top three
//               levels, dptens <- dp3d*sph + dt*dptens
//   update    : the exchange of those (gathered), inverse mass, v += ,
//               T += - heating/cp, dp3d = dptens*rsmp
// A lane holds one point's chunk of C levels (layout sc_field); the exchanged
// buffers go back and forth between a.lap and a.pre.  The mixed form forms the
// laplacians in FP32 and exchanges FP32 first laplacians (summed in FP64).
//
// The kernels finish one field before the next (pin), so that a field's C
// levels of gathers are in flight together and the metric is shared by them.
// Bound: memory, 30 fields per subcycle at 3.9 TB/s.  One lane per level on the
// [lev][pt] layout ran at 2.5 to 2.9 TB/s, because each neighbour's edge cost
// whole 128-byte lines of L2 traffic: three subcycles at ne30 L72 took 1.69 ms
// then and 1.16 ms now, and the exchange before them 275 and 183 us.  Caps of 3
// and 4 waves per SIMD spill: 1.58 and 2.41 ms.
#include "kernels.hpp"

namespace hx {

// ------------------------------------------------------------- operators
// the laplacians of the FP64 and the mixed form on a chunk of levels; P: the
// type the first laplacians are stored in
template <bool F32>
struct HvOps {
  typedef double P;
  ElemLane e;
  DvvLane d;
  __device__ __forceinline__ HvOps(const MetricPtrs &m, int ie, int pt) {
    load_elem(m, ie, pt, e);
    load_dvv(m.dvv, pt, d);
  }
  __device__ __forceinline__ double lap(double x) const { return sph_laplace(e, d, x); }
  __device__ __forceinline__ double lap_state(double x) const { return lap(x); }
  __device__ __forceinline__ double vlap(double ratio, double u, double w, double &l1) const {
    double l0;
    sph_vlaplace_contra(e, d, ratio, u, w, l0, l1);
    return l0;
  }
};
template <>
struct HvOps<true> {
  typedef float P;
  ElemLaneF e;
  DvvLaneF d;
  __device__ __forceinline__ HvOps(const MetricPtrs &m, int ie, int pt) {
    load_elemf(m, ie, pt, e);
    load_dvvf(m.dvv, pt, d);
  }
  __device__ __forceinline__ float lap(double x) const { return sph_laplacef(e, d, (float)x); }
  // of a state's T or dp3d: less its slab reference before rounding
  __device__ __forceinline__ float lap_state(double x) const { return lap(x - slab_ref(x)); }
  __device__ __forceinline__ float vlap(double ratio, double u, double w, float &l1) const {
    float l0;
    sph_vlaplace_contraf(e, d, (float)ratio, (float)u, (float)w, l0, l1);
    return l0;
  }
};

// the first laplacians of a chunk's levels into lap [ie][4][sc]
template <int C, bool F32>
__device__ __forceinline__ void lap1_scalar(const HvOps<F32> &o, const double (&x)[C], typename HvOps<F32>::P *lap) {
  typename HvOps<F32>::P l[C];
#pragma unroll
  for (int j = 0; j < C; ++j) l[j] = o.lap_state(x[j]);
  sc_store(lap, l);
}
template <int C, bool F32>
__device__ __forceinline__ void lap1_vector(const HvOps<F32> &o, double ratio, const double (&u)[C],
                                            const double (&w)[C], typename HvOps<F32>::P *lap, size_t lf) {
  typename HvOps<F32>::P l0[C], l1[C];
#pragma unroll
  for (int j = 0; j < C; ++j) l0[j] = o.vlap(ratio, u[j], w[j], l1[j]);
  sc_store(lap, l0);
  sc_store(lap + lf, l1);
}

// The exchange of an RK result (u, v, T, dp3d) into the state arrays.  LAP1:
// with the first laplacians of the assembled state, from registers.
template <int C, int LAP1>
__global__ __launch_bounds__(256) void state_dss_kernel(StateDssArgs a) {
  int ie, k0, pt;
  if (!sc_lane<C>(a.nelem, a.nlev, ie, k0, pt)) return;
  const size_t lf = sc_field<C>(a.nlev);
  const ScGather<double, C> g(a.pre, 4 * lf, ie, pt, k0, a.src);
  const double r = a.m.rspheremp[(size_t)ie * 16 + pt];
  const HvOps<LAP1 == 2> o(a.m, ie, pt);
  typedef typename HvOps<LAP1 == 2>::P P;
  P *const lap = (P *)a.lap + (size_t)ie * 4 * lf + (size_t)k0 * 16 + pt * C;
  double *const v = a.v + ((size_t)ie * a.nlev + k0) * 32 + pt;
  double *const t = a.t + ((size_t)ie * a.nlev + k0) * 16 + pt;
  double *const dp = a.dp + ((size_t)ie * a.nlev + k0) * 16 + pt;
  auto put = [&](double *out, int stride, const double (&x)[C]) {
#pragma unroll
    for (int j = 0; j < C; ++j)
      if (k0 + j < a.nlev) out[j * stride] = x[j];
  };
  double x[C], y[C];
  g.field(3 * lf, r, x);
  put(dp, 16, x);
  if (LAP1) lap1_scalar<C, LAP1 == 2>(o, x, lap + 3 * lf);
  g.field(2 * lf, r, x);
  put(t, 16, x);
  if (LAP1) lap1_scalar<C, LAP1 == 2>(o, x, lap + 2 * lf);
  g.field(0, r, x);
  g.field(lf, r, y);
  put(v, 32, x);
  put(v + 16, 32, y);
  if (LAP1) lap1_vector<C, LAP1 == 2>(o, a.nu_ratio1, x, y, lap, lf);
}

template <int C>
static void launch_state_dss_c(hipStream_t st, const StateDssArgs &a) {
  const dim3 g(sc_blocks<C>(a.nelem, a.nlev));
  if (a.lap1 == 2) hipLaunchKernelGGL((state_dss_kernel<C, 2>), g, dim3(256), 0, st, a);
  else if (a.lap1) hipLaunchKernelGGL((state_dss_kernel<C, 1>), g, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((state_dss_kernel<C, 0>), g, dim3(256), 0, st, a);
}

void launch_state_dss(hipStream_t st, const StateDssArgs &a) {
  if (a.chunk == 6) launch_state_dss_c<6>(st, a);
  else if (a.chunk == 2) launch_state_dss_c<2>(st, a);
  else launch_state_dss_c<4>(st, a);
}

// Second laplacians: constant coefficient, or (TENSOR) the tensor form
// (HyperviscosityFunctorImpl.hpp:88-128), and the pre-exchange scaling.  The
// sponge's laplacians of the state at the top three levels are the element's
// own first laplacians, read from a.lap; RATIO: except the vector one, where
// the first laplacian scales the divergence (nu_div != nu).
template <int C, bool F32, bool TENSOR, bool RATIO>
__global__ __launch_bounds__(256) void hv_lap2_kernel(HvArgs a) {
  int ie, k0, pt;
  if (!sc_lane<C>(a.nelem, a.nlev, ie, k0, pt)) return;
  typedef typename HvOps<F32>::P P;
  const int L = a.nlev;
  const size_t lf = sc_field<C>(L);
  const ScGather<P, C> g((const P *)a.lap, 4 * lf, ie, pt, k0, a.src);
  const double rs = a.m.rspheremp[(size_t)ie * 16 + pt];
  const double sph = a.m.spheremp[(size_t)ie * 16 + pt];
  const HvOps<F32> o(a.m, ie, pt);
  double tv[4], vs[6];
  if (TENSOR) load_tensor(a.m, ie, pt, tv, vs);
  auto lap2 = [&](double x) -> double {
    if constexpr (TENSOR) return sph_laplace_tensor(o.e, o.d, tv, x);
    else return o.lap(x);
  };
  const bool top = a.nu_top > 0 && k0 < 3;
  constexpr int TOP = C < 3 ? C : 3;
  auto top_level = [&](int j) { return C < 3 ? k0 + j : j; };  // (k0 is 0 in longer chunks)
  // the sponge adds sc(j) * (own first laplacian) at levels 0..2
  auto sponge = [&](size_t off, double (&x)[C]) {
    if (!top) return;
#pragma unroll
    for (int j = 0; j < TOP; ++j) {
      const int k = top_level(j);
      if (k < 3 && k < L) x[j] += (k == 0 ? 4.0 : k == 1 ? 2.0 : 1.0) * a.nu_top * (double)g.p[0][off + j];
    }
  };
  double *const out = a.pre + (size_t)ie * 4 * lf + (size_t)k0 * 16 + pt * C;
  double x[C], y[C];
  // ---------------------------------------------------------------- dp3d
  {
    double dpn[C], da[C], db[C];
    const size_t s = ((size_t)ie * L + k0) * 16 + pt;
    const bool acc = a.eta_ave_w != 0.0;
    auto at = [&](int j) { return s + (k0 + j < L ? j : L - 1 - k0) * 16; };
#pragma unroll
    for (int j = 0; j < C; ++j) {
      dpn[j] = a.dp[at(j)];
      if (acc && !a.first) {
        da[j] = a.dpdiss_ave[at(j)];
        db[j] = a.dpdiss_bih[at(j)];
      } else {
        da[j] = db[j] = 0.0;
      }
    }
    g.field(3 * lf, rs, x);
#pragma unroll
    for (int j = 0; j < C; ++j) {
      x[j] = lap2(x[j]);
      if (acc && k0 + j < L) {
        a.dpdiss_ave[s + j * 16] = da[j] + a.eta_ave_w * dpn[j] / a.nsub;
        a.dpdiss_bih[s + j * 16] = db[j] + a.eta_ave_w * x[j] / a.nsub;
      }
      x[j] *= -a.nu_p;
    }
    sponge(3 * lf, x);
#pragma unroll
    for (int j = 0; j < C; ++j) {
      x[j] *= a.dt;
      x[j] += dpn[j] * sph;
    }
    sc_store(out + 3 * lf, x);
  }
  // ------------------------------------------------------------------- T
  g.field(2 * lf, rs, x);
#pragma unroll
  for (int j = 0; j < C; ++j) x[j] = -a.nu_s * lap2(x[j]);
  sponge(2 * lf, x);
  sc_store(out + 2 * lf, x);
  // ------------------------------------------------------------------- v
  g.field(0, rs, x);
  g.field(lf, rs, y);
#pragma unroll
  for (int j = 0; j < C; ++j) {
    P l1;
    double l0, m1;
    if constexpr (TENSOR) {
      sph_vlaplace_cartesian(o.e, o.d, tv, vs, x[j], y[j], l0, m1);
    } else {
      l0 = o.vlap(a.nu_ratio2, x[j], y[j], l1);
      m1 = l1;
    }
    x[j] = l0 * -a.nu;
    y[j] = m1 * -a.nu;
  }
  if (!RATIO) {
    sponge(0, x);
    sponge(lf, y);
  } else if (top) {
    const size_t v = (size_t)ie * L * 32 + pt;
#pragma unroll
    for (int j = 0; j < TOP; ++j) {
      const int k = top_level(j);
      if (k >= 3 || k >= L) break;
      P l1;
      const double l0 = o.vlap(1.0, a.v[v + k * 32], a.v[v + k * 32 + 16], l1);
      const double sc = (k == 0 ? 4.0 : k == 1 ? 2.0 : 1.0) * a.nu_top;
      x[j] += sc * l0;
      y[j] += sc * (double)l1;
    }
  }
  sc_store(out, x);
  sc_store(out + lf, y);
}

// LAP1: with the first laplacians of the updated state for the next subcycle
// (1: FP64, 2: mixed form), from registers.
template <int C, int LAP1>
__global__ __launch_bounds__(256) void hv_update_kernel(HvArgs a) {
  int ie, k0, pt;
  if (!sc_lane<C>(a.nelem, a.nlev, ie, k0, pt)) return;
  const int L = a.nlev;
  const size_t lf = sc_field<C>(L);
  const ScGather<double, C> g(a.pre, 4 * lf, ie, pt, k0, a.src);
  const double r = a.m.rspheremp[(size_t)ie * 16 + pt];
  const HvOps<LAP1 == 2> o(a.m, ie, pt);
  typedef typename HvOps<LAP1 == 2>::P P;
  P *const lap = (P *)a.lap + (size_t)ie * 4 * lf + (size_t)k0 * 16 + pt * C;
  const size_t s = ((size_t)ie * L + k0) * 16 + pt, v = ((size_t)ie * L + k0) * 32 + pt;
  auto lv = [&](int j) { return k0 + j < L ? j : L - 1 - k0; };
  double x[C], y[C], heat[C];
  {
    double u[C], w[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      u[j] = a.v[v + lv(j) * 32];
      w[j] = a.v[v + lv(j) * 32 + 16];
    }
    g.field(0, 1.0, x);
    g.field(lf, 1.0, y);
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const double v0 = a.dt * x[j] * r, v1 = a.dt * y[j] * r;
      u[j] += v0;
      w[j] += v1;
      heat[j] = v0 * u[j] + v1 * w[j];
      if (k0 + j < L) {
        a.vo[v + j * 32] = u[j];
        a.vo[v + j * 32 + 16] = w[j];
      }
    }
    if (LAP1) lap1_vector<C, LAP1 == 2>(o, a.nu_ratio1, u, w, lap, lf);
  }
  {
    double t[C];
#pragma unroll
    for (int j = 0; j < C; ++j) t[j] = a.t[s + lv(j) * 16];
    g.field(2 * lf, 1.0, x);
#pragma unroll
    for (int j = 0; j < C; ++j) {
      t[j] = t[j] + a.dt * x[j] * r - heat[j] / CP;
      if (k0 + j < L) a.to[s + j * 16] = t[j];
    }
    if (LAP1) lap1_scalar<C, LAP1 == 2>(o, t, lap + 2 * lf);
  }
  g.field(3 * lf, r, x);
#pragma unroll
  for (int j = 0; j < C; ++j)
    if (k0 + j < L) a.dpo[s + j * 16] = x[j];
  if (LAP1) lap1_scalar<C, LAP1 == 2>(o, x, lap + 3 * lf);
}

template <int C>
static void launch_hv_cycle_c(hipStream_t st, const HvArgs &a, bool lap1_next) {
  const dim3 g(sc_blocks<C>(a.nelem, a.nlev));
  auto go = [&](auto *kernel) { hipLaunchKernelGGL(kernel, g, dim3(256), 0, st, a); };
  const bool ratio = a.nu_top > 0 && a.nu_ratio1 != 1.0;
  if (a.mixed) go(ratio ? hv_lap2_kernel<C, true, false, true> : hv_lap2_kernel<C, true, false, false>);
  else if (a.consthv) go(ratio ? hv_lap2_kernel<C, false, false, true> : hv_lap2_kernel<C, false, false, false>);
  else go(ratio ? hv_lap2_kernel<C, false, true, true> : hv_lap2_kernel<C, false, true, false>);
  if (!lap1_next) go(hv_update_kernel<C, 0>);
  else if (a.mixed) go(hv_update_kernel<C, 2>);
  else go(hv_update_kernel<C, 1>);
}

void launch_hv_cycle(hipStream_t st, const HvArgs &a, bool lap1_next) {
  if (a.chunk == 6) launch_hv_cycle_c<6>(st, a, lap1_next);
  else if (a.chunk == 2) launch_hv_cycle_c<2>(st, a, lap1_next);
  else launch_hv_cycle_c<4>(st, a, lap1_next);
}

}  // namespace hx
