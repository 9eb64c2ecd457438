// Host side of libhommexx_amd.so: the reference's iso_c_binding C-ABI
// (cxx_f90_interface.cpp, mpi/mpi_cxx_f90_interface.cpp, Hommexx_Session.cpp,
// prim_driver.cpp) over a device-resident context, plus hommexx_hip_*
// extensions for the test/benchmark harness.  Fortran passes scalars by
// reference and arrays as pointers to the flat elem_* arrays; time-level
// indices enter 1-based and leave prim_run_subcycle_c 0-based, exactly as in
// the reference.  Errors that the reference turns into MPI_Abort abort the
// process too unless hommexx_hip_set_abort_on_error(0) was called, in which
// case they are recorded for hommexx_hip_last_error().
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "kernels.hpp"
#include "../../include/hommexx_amd.h"

using namespace hx;

// the array behind scratch_pointer() (see there): 16 Mi doubles, 128 MiB per GPU
constexpr size_t ADJ_SCRATCH_DOUBLES = (size_t)16 << 20;
static __device__ __align__(256) double scratch[ADJ_SCRATCH_DOUBLES];

namespace {

struct Params {
  int remap_alg = 1, limiter_option = 8, rsplit = 1, qsplit = 1, time_step_type = 5, energy_fixer = 0;
  int qsize = 0, state_frequency = 1, hypervis_order = 2, hypervis_subcycle = 1, ftype = -1;
  double nu = 0, nu_p = 0, nu_q = 0, nu_s = 0, nu_div = 0, nu_top = 0, hypervis_scaling = 0;
  double nu_ratio1 = 1, nu_ratio2 = 1;
  bool prescribed_wind = false, moist = false, disable_diagnostics = true, use_cpstar = false, use_sl = false;
  bool set = false;
};

struct Timer {
  std::vector<std::pair<hipEvent_t, hipEvent_t>> pending;
  int count = 0;
  double total_ms = 0;
};

// pinned buffers of the copies to and from host arrays (HostCopy): two of a
// thread's, at most 16 MB in all, kept until the simulation ends
struct HostStage {
  static constexpr int W = 4;                       // threads
  static constexpr size_t PIECE = (size_t)1 << 18;  // doubles
  double *buf[2 * W] = {};
  hipEvent_t ev[2 * W] = {};
};

struct Ctx {
  // configuration
  bool session = false;
  // the reference's build-time PLEV and QSIZE_D (Makefile PREQX_PLEV, QSIZE_D)
  int nlev_cfg = HOMMEXX_PREQX_PLEV, qsize_d_cfg = HOMMEXX_QSIZE_D;
  bool abort_on_error = true;
  int last_error = 0;
  std::string msg;
  hipStream_t st = nullptr;
  // connectivity (host)
  int conn_nelem = -1;
  bool conn_final = false;
  std::vector<int> conn_rl, conn_rp;  // [ie*8 + pos] -> remote lid / pos (reference numbering)
  // params / dims
  Params p;
  double dvv[16] = {0};
  bool dvv_set = false;
  int nelem = 0, nlev = 0, qsize = 0, qsize_d = 0;
  bool elems_set = false, states_set = false, hv_set = false, be_set = false;
  // 2-D metric (device)
  double *D = nullptr, *Dinv = nullptr, *metinv = nullptr, *tensorvisc = nullptr, *vec_sph2cart = nullptr;
  double *fcor = nullptr, *mp = nullptr, *spheremp = nullptr, *rspheremp = nullptr, *metdet = nullptr,
         *phis = nullptr, *dvv_d = nullptr;
  bool consthv = true;
  int *dss_src = nullptr, *nbr = nullptr;
  // vertical coordinate
  double ps0 = 0, hyai0 = 0;
  std::vector<double> hyai, hybi;
  double *hyai_d = nullptr, *hybi_d = nullptr, *dp0_d = nullptr;
  // states
  double *v[3] = {}, *t[3] = {}, *dp[3] = {}, *ps[3] = {}, *qdp[2] = {}, *Q = nullptr;
  std::vector<double> qdp_tail;  // Qdp of tracers qsize..qsize_d-1 as received (never evolved)
  std::vector<double> fq_tail;   // FQ of tracers qsize..qsize_d-1 as received (never used)
  // derived
  double *omega = nullptr, *eta_dot = nullptr, *dpdiss_ave = nullptr, *dpdiss_bih = nullptr,
         *derived_dp = nullptr, *divdp = nullptr, *divdp_proj = nullptr, *vn0 = nullptr;
  // forcing
  double *ft = nullptr, *fm = nullptr, *fq = nullptr;
  // scratch
  double *pre[2] = {};   // pre-exchange states [ie][4][sc] (state_chunk)
  double *qdp_pre = nullptr, *qlim[2] = {}, *fdss_pre = nullptr;
  // stage-2 pre-exchange buffers: qdp_pre2 and an alias of
  // pre[0], which is free during the tracer step
  double *qdp_pre2 = nullptr, *fdss_pre2 = nullptr;
  int *err_d = nullptr;
  int *err_h = nullptr;
  HostStage stage;
  // diagnostics: the Fortran arrays of init_diagnostics_c (q, qvar, qmass,
  // q1mass, iener, iener_wet, kener, pener) and a device staging buffer
  double *dg[8] = {};
  bool dg_set = false;
  double *dg_dev = nullptr;
  // time levels (0-based)
  int nm1 = 0, n0 = 1, np1 = 2, nstep = 0, nstep0 = 0, n0_qdp = 0, np1_qdp = 1;
  // 0: FP64 step; 1: mixed form (FP32 sphere operators in hyperviscosity and
  // the tracer flux divergence / biharmonic)
  int form = 0;
  // debugging: stop prim_run_subcycle_c after a phase (0: never)
  int debug_stop = 0;
  bool stopped = false;
  // profiling
  bool prof = false;
  std::string prof_only;  // non-empty: time only the phase of this name
  std::map<std::string, Timer> timers;
  std::vector<void *> allocs;
};

Ctx *g = nullptr;

Ctx &C() {
  if (!g) g = new Ctx();
  return *g;
}

void fail(int code, const char *fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  Ctx &c = C();
  c.last_error = code;
  c.msg = buf;
  if (c.abort_on_error) {
    fprintf(stderr, "hommexx_amd error %d: %s\n", code, buf);
    fflush(stderr);
    abort();
  }
}

bool hipok(hipError_t e, const char *what) {
  if (e != hipSuccess) {
    fail(100, "%s: %s", what, hipGetErrorString(e));
    return false;
  }
  return true;
}

template <typename T>
T *dalloc(size_t n) {
  void *p = nullptr;
  if (n == 0) n = 1;
  if (!hipok(hipMalloc(&p, n * sizeof(T)), "hipMalloc")) return nullptr;
  // hipMemset runs on the null stream, which the library's non-blocking
  // stream does not wait for: finish it before any kernel can touch p
  hipMemset(p, 0, n * sizeof(T));
  if (!hipok(hipDeviceSynchronize(), "hipMemset")) return nullptr;
  C().allocs.push_back(p);
  return (T *)p;
}

void h2d(void *d, const void *h, size_t bytes) { hipok(hipMemcpy(d, h, bytes, hipMemcpyHostToDevice), "h2d"); }

void adj_reset();

void free_all() {
  Ctx &c = C();
  adj_reset();
  if (c.st) hipStreamSynchronize(c.st);
  for (void *p : c.allocs) hipFree(p);
  c.allocs.clear();
  for (auto &kv : c.timers)
    for (auto &e : kv.second.pending) {
      hipEventDestroy(e.first);
      hipEventDestroy(e.second);
    }
  c.timers.clear();
  if (c.err_h) hipHostFree(c.err_h);
  c.err_h = nullptr;
  for (int i = 0; i < 2 * HostStage::W; ++i) {
    if (c.stage.buf[i]) hipHostFree(c.stage.buf[i]);
    if (c.stage.ev[i]) hipEventDestroy(c.stage.ev[i]);
  }
  c.stage = HostStage();
  c.dg_dev = nullptr;
}

// ---------------------------------------------------------------- timing
struct Scope {
  const char *name;
  hipEvent_t a = nullptr, b = nullptr;
  explicit Scope(const char *n) : name(n) {
    Ctx &c = C();
    if (!c.prof || (!c.prof_only.empty() && c.prof_only != n)) return;
    hipEventCreate(&a);
    hipEventCreate(&b);
    hipEventRecord(a, c.st);
  }
  ~Scope() {
    Ctx &c = C();
    if (!c.prof || !a) return;
    hipEventRecord(b, c.st);
    c.timers[name].pending.push_back({a, b});
  }
};

void flush_timers() {
  Ctx &c = C();
  hipStreamSynchronize(c.st);
  for (auto &kv : c.timers) {
    for (auto &e : kv.second.pending) {
      float ms = 0;
      hipEventElapsedTime(&ms, e.first, e.second);
      kv.second.total_ms += ms;
      kv.second.count += 1;
      hipEventDestroy(e.first);
      hipEventDestroy(e.second);
    }
    kv.second.pending.clear();
  }
}

// ------------------------------------------------------ connectivity
// point lists of the 8 connections (ConnectivityHelpers.hpp), pt = igp*4+jgp
const int EDGE_FWD[4][4] = {{0, 1, 2, 3}, {12, 13, 14, 15}, {0, 4, 8, 12}, {3, 7, 11, 15}};
const int CORNER_PT[4] = {0, 3, 12, 15};
const int EDGE_DIR[4][4] = {{1, 0, 0, 1}, {0, 1, 1, 0}, {0, 1, 1, 0}, {1, 0, 0, 1}};

void build_dss_tables() {
  Ctx &c = C();
  const int ne = c.nelem;
  // slot (receiver elem, receiver pos)[k] <- (sender elem, sender point)
  std::vector<int> slot((size_t)ne * 8 * 4, -1);
  for (int a = 0; a < ne; ++a)
    for (int pa = 0; pa < 8; ++pa) {
      const int b = c.conn_rl[a * 8 + pa];
      if (b < 0) continue;
      const int pb = c.conn_rp[a * 8 + pa];
      if (pa < 4) {
        const int dir = EDGE_DIR[pa][pb];
        for (int k = 0; k < 4; ++k) {
          const int spt = EDGE_FWD[pa][dir ? 3 - k : k];
          slot[((size_t)b * 8 + pb) * 4 + k] = a * 16 + spt;
        }
      } else {
        slot[((size_t)b * 8 + pb) * 4 + 0] = a * 16 + CORNER_PT[pa - 4];
      }
    }
  std::vector<int> src((size_t)ne * 16 * 3, -1), cnt((size_t)ne * 16, 0);
  std::vector<int> nbr((size_t)ne * 8, -1);
  auto push = [&](int e, int pt, int s) {
    const size_t i = (size_t)e * 16 + pt;
    if (cnt[i] >= 3) {
      fail(10, "more than three neighbour copies at element %d point %d", e, pt);
      return;
    }
    src[i * 3 + cnt[i]++] = s;
  };
  for (int e = 0; e < ne; ++e) {
    for (int k = 0; k < 4; ++k)
      for (int ed = 0; ed < 4; ++ed) {
        const int s = slot[((size_t)e * 8 + ed) * 4 + k];
        if (s >= 0) push(e, EDGE_FWD[ed][k], s);
      }
    for (int cr = 0; cr < 4; ++cr) {
      const int s = slot[((size_t)e * 8 + 4 + cr) * 4];
      if (s >= 0) push(e, CORNER_PT[cr], s);
    }
    for (int pos = 0; pos < 8; ++pos) {
      const int s = slot[((size_t)e * 8 + pos) * 4];
      nbr[(size_t)e * 8 + pos] = s >= 0 ? s / 16 : -1;
    }
  }
  c.dss_src = dalloc<int>(src.size());
  c.nbr = dalloc<int>(nbr.size());
  h2d(c.dss_src, src.data(), src.size() * sizeof(int));
  h2d(c.nbr, nbr.data(), nbr.size() * sizeof(int));
}

MetricPtrs metric() {
  Ctx &c = C();
  MetricPtrs m;
  m.D = c.D;
  m.Dinv = c.Dinv;
  m.metinv = c.metinv;
  m.fcor = c.fcor;
  m.mp = c.mp;
  m.spheremp = c.spheremp;
  m.rspheremp = c.rspheremp;
  m.metdet = c.metdet;
  m.phis = c.phis;
  m.dvv = c.dvv_d;
  m.tensorvisc = c.tensorvisc;
  m.vec_sph2cart = c.vec_sph2cart;
  return m;
}

bool ready(const char *who) {
  Ctx &c = C();
  if (!(c.p.set && c.dvv_set && c.elems_set && c.states_set && c.hv_set && c.conn_final)) {
    fail(20, "%s: the library is not fully initialised (params %d, derivative %d, elements %d, states %d, hvcoord %d, "
             "connectivity %d)",
         who, c.p.set, c.dvv_set, c.elems_set, c.states_set, c.hv_set, c.conn_final);
    return false;
  }
  if (c.conn_nelem != c.nelem) {
    fail(21, "%s: connectivity has %d elements but the element data has %d", who, c.conn_nelem, c.nelem);
    return false;
  }
  return true;
}

void alloc_work() {
  Ctx &c = C();
  if (c.be_set) return;
  // pre-exchange buffers: whole 8-level chunks per element and field
  const size_t e3c = (size_t)c.nelem * lc_field(c.nlev), q3c = e3c * (c.qsize ? c.qsize : 1);
  const size_t sc = c.nelem * std::max(sc_field<4>(c.nlev), sc_field<6>(c.nlev));
  for (double *&p : c.pre) p = dalloc<double>(std::max(4 * sc, e3c));
  // Four 40-F3 tracer uses share two allocations (at Q = 40); no kernel
  // writes the allocation it gathers from:
  //   qdp_pre : stage-1 pre-exchange (-> stage 2), then the first laplacian of
  //             the biharmonic (-> stage 3)
  //   qdp_pre2: stage-2 pre-exchange (-> its exchange), then the stage-3
  //             pre-exchange (-> its exchange)
  c.qdp_pre = dalloc<double>(q3c);
  c.qdp_pre2 = dalloc<double>(q3c);
  c.qlim[0] = dalloc<double>((size_t)c.nelem * (c.qsize ? c.qsize : 1) * ql_row(c.nlev));
  c.qlim[1] = dalloc<double>((size_t)c.nelem * (c.qsize ? c.qsize : 1) * ql_row(c.nlev));
  c.fdss_pre = dalloc<double>(e3c);
  c.fdss_pre2 = c.pre[0];
  c.err_d = dalloc<int>(1);
  if (!c.err_h) hipHostMalloc((void **)&c.err_h, sizeof(int));
  c.be_set = true;
}

// ------------------------------------------------------ step phases
// one prognostic state: v [ie][lev][2][pt], T and dp3d [ie][lev][pt]
struct StateBuf {
  double *v, *t, *dp;
};

// The five RK stages (u3_5stage, prim_advance_exp.cpp:113-161).  The state of
// stage i+1 is u[i]; w = (5 u[1] - u[0])/4, out the result.  keep: u[2..4] are
// stored too (they may be one buffer otherwise; u[1] and w may be one).
struct RkBufs {
  StateBuf u[5], w, out;
  bool keep = false;
  bool start = false;  // the accumulators start here
};

StateBuf level(int tl) {
  Ctx &c = C();
  return {c.v[tl], c.t[tl], c.dp[tl]};
}

int chunk() {
  Ctx &c = C();
  return state_chunk(c.nlev, c.p.rsplit == 0);
}

// out = DSS_r(pre); lap1: also its first hyperviscosity laplacians
void state_dss(const double *pre, const StateBuf &out, bool lap1 = false) {
  Ctx &c = C();
  StateDssArgs x{};
  x.m = metric();
  x.src = c.dss_src;
  x.nelem = c.nelem;
  x.nlev = c.nlev;
  x.chunk = chunk();
  x.pre = pre;
  x.v = out.v;
  x.t = out.t;
  x.dp = out.dp;
  if (lap1) {
    x.lap1 = c.form == 1 && c.consthv ? 2 : 1;  // the mixed form's FP32 first laplacians
    x.lap = c.pre[1];
    x.nu_ratio1 = c.p.nu_ratio1;
  }
  Scope s("caar_dss");
  launch_state_dss(c.st, x);
}

bool stop_here(int phase) {
  Ctx &c = C();
  if (c.debug_stop == phase) c.stopped = true;
  return c.stopped;
}

void rk_stages(const RkBufs &r, double dt, double eta_ave_w) {
  Ctx &c = C();
  // rsplit > 0: each stage gathers the one before it; the vertical advection
  // of rsplit == 0 reads neighbour levels, so its stages read stored states
  const bool gather = c.p.rsplit > 0;
  const double h[5] = {dt / 5.0, dt / 5.0, dt / 3.0, 2.0 * dt / 3.0, 3.0 * dt / 4.0};
  const double eta[5] = {eta_ave_w / 4.0, 0.0, 0.0, 0.0, 3.0 * eta_ave_w / 4.0};
  for (int i = 0; i < 5; ++i) {
    CaarArgs a{};
    a.m = metric();
    a.src = c.dss_src;
    a.nelem = c.nelem;
    a.nlev = c.nlev;
    a.qsize = c.qsize;
    a.chunk = chunk();
    if (i > 0 && gather) {
      a.pre = c.pre[(i - 1) & 1];
      if (i == 1 || r.keep) {
        a.out_v = r.u[i].v;
        a.out_t = r.u[i].t;
        a.out_dp = r.u[i].dp;
      }
    } else {
      a.v = r.u[i].v;
      a.t = r.u[i].t;
      a.dp = r.u[i].dp;
    }
    if (i > 0) {
      a.bv = r.u[0].v;
      a.bt = r.u[0].t;
      a.bdp = r.u[0].dp;
    }
    if (i == 4) {
      a.u1v = r.u[1].v;
      a.u1t = r.u[1].t;
      a.u1dp = r.u[1].dp;
      a.wv = r.w.v;
      a.wt = r.w.t;
      a.wdp = r.w.dp;
    }
    a.qdp_n0 = (c.p.moist && c.qsize > 0) ? c.qdp[c.n0_qdp] : nullptr;
    a.vn0 = c.vn0;
    a.omega = c.omega;
    a.rsplit0 = c.p.rsplit == 0;
    a.hybi = c.hybi_d;
    a.eta_acc = c.eta_dot;
    a.pre_out = c.pre[i & 1];
    a.dt = h[i];
    a.eta_ave_w = eta[i];
    a.derived_dp = i == 0 && r.start ? c.derived_dp : nullptr;
    a.p_top = c.hyai0 * c.ps0;
    {
      Scope s("caar");
      launch_caar(c.st, a);
    }
    const bool stop = i == 0 && c.debug_stop == 1;
    if (i < 4 && (!gather || stop)) state_dss(a.pre_out, r.u[i + 1]);
    if (stop && stop_here(1)) return;
  }
  state_dss(c.pre[0], r.out, true);
}

void u3_5stage(int nm1, int n0, int np1, double dt, double eta_ave_w, bool start) {
  RkBufs r;
  r.start = start;
  r.u[0] = level(n0);
  r.u[1] = r.w = level(nm1);
  r.u[2] = r.u[3] = r.u[4] = r.out = level(np1);
  rk_stages(r, dt, eta_ave_w);
}

// one subcycle of hyperviscosity from the state x to o
HvArgs hv_args(const StateBuf &x, const StateBuf &o, double dt, double eta_ave_w) {
  Ctx &c = C();
  HvArgs a{};
  a.m = metric();
  a.src = c.dss_src;
  a.nelem = c.nelem;
  a.nlev = c.nlev;
  a.chunk = chunk();
  a.v = x.v;
  a.t = x.t;
  a.dp = x.dp;
  a.vo = o.v;
  a.to = o.t;
  a.dpo = o.dp;
  a.lap = c.pre[1];  // where state_dss leaves the first laplacians
  a.pre = c.pre[0];
  a.dpdiss_ave = c.dpdiss_ave;
  a.dpdiss_bih = c.dpdiss_bih;
  a.dt = dt / c.p.hypervis_subcycle;
  a.eta_ave_w = eta_ave_w;
  a.nu = c.p.nu;
  a.nu_s = c.p.nu_s;
  a.nu_p = c.p.nu_p;
  a.nu_top = c.p.nu_top;
  a.nu_ratio1 = c.p.nu_ratio1;
  a.nu_ratio2 = c.p.nu_ratio2;
  a.nsub = c.p.hypervis_subcycle;
  // the mixed form keeps the tensor form of hyperviscosity in FP64
  a.consthv = c.consthv;
  a.mixed = c.form == 1 && c.consthv;
  return a;
}

void hyperviscosity(int np1, double dt, double eta_ave_w, bool start) {
  Ctx &c = C();
  HvArgs a = hv_args(level(np1), level(np1), dt, eta_ave_w);
  const int nsub = c.p.hypervis_subcycle;
  for (int cyc = 0; cyc < nsub; ++cyc) {
    Scope s("hv_cycle");
    a.first = start && cyc == 0;
    launch_hv_cycle(c.st, a, cyc + 1 < nsub);
  }
}

void update_tracers_levels() {
  Ctx &c = C();
  const int it = c.nstep / c.p.qsplit;
  c.n0_qdp = it % 2 == 0 ? 0 : 1;
  c.np1_qdp = 1 - c.n0_qdp;
}

void leapfrog() {
  Ctx &c = C();
  const int tmp = c.np1;
  c.np1 = c.nm1;
  c.nm1 = c.n0;
  c.n0 = tmp;
  ++c.nstep;
}

void advec_tracers(double dt) {
  Ctx &c = C();
  update_tracers_levels();
  EulerArgs a{};
  a.m = metric();
  a.src = c.dss_src;
  a.nbr = c.nbr;
  a.nelem = c.nelem;
  a.nlev = c.nlev;
  a.qsize = c.qsize;
  a.derived_dp = c.derived_dp;
  a.divdp = c.divdp;
  a.divdp_proj = c.divdp_proj;
  a.divdp_w = c.divdp;
  a.divdp_proj_w = c.divdp_proj;
  a.vn0 = c.vn0;
  a.dpdiss_ave = c.dpdiss_ave;
  a.dpdiss_bih = c.dpdiss_bih;
  a.dp0 = c.dp0_d;
  a.fdss_pre = c.fdss_pre;
  a.nu_p = c.p.nu_p;
  a.nu_q = c.p.nu_q;
  a.limiter_option = c.p.limiter_option;
  a.mixed = c.form == 1;
  a.bih32 = c.form == 1 && c.consthv;
  a.consthv = c.consthv;
  a.rhs_viss = 0.0;
  const double dts = dt / 2.0;
  a.dt = dts;
  int cur = 0;
  // stage 1 bounds: divdp, then qmin/qmax of Qdp(n0_qdp) (rhs_multiplier 0)
  a.rhs_multiplier = 0.0;
  a.qdp_n0 = c.qdp[c.n0_qdp];
  a.qlim = c.qlim[cur];
  {
    Scope s("euler_divdp_qmm");
    launch_euler_divdp_qmm(c.st, a);
  }
  auto nbr_minmax = [&]() {
    a.qlim = c.qlim[cur];
    a.qlim_new = c.qlim[1 - cur];
    Scope s("euler_nbr_minmax");
    launch_euler_nbr_minmax(c.st, a);
    cur = 1 - cur;
    a.qlim = c.qlim[cur];
  };
  nbr_minmax();
  const double *qdp_n0 = c.qdp[c.n0_qdp];
  double *qdp_np1 = c.qdp[c.np1_qdp];
  a.qdp_np1 = qdp_np1;
  // stage 1: Qdp(n0) -> qdp_pre
  a.qdp_n0 = qdp_n0;
  a.fdss = c.divdp_proj;
  a.qdp_pre = c.qdp_pre;
  a.fdss_pre = c.fdss_pre;
  {
    Scope s("euler_advect");
    launch_euler_advect(c.st, a, 1);
  }
  if (c.debug_stop == 4) {
    launch_euler_dss(c.st, a, 0);
    stop_here(4);
    return;
  }
  // stage 2: gathers qdp_pre, -> qdp_pre2
  a.qdp_pre_in = c.qdp_pre;
  a.fdss_pre_in = c.fdss_pre;
  a.fdss = c.eta_dot;
  a.qdp_pre = c.qdp_pre2;
  a.fdss_pre = c.fdss_pre2;
  {
    Scope s("euler_advect");
    launch_euler_advect(c.st, a, 2);
  }
  // its exchange: gathers qdp_pre2, -> Qdp(np1), laplacian -> qdp_pre
  a.qbih_pre = c.qdp_pre;
  {
    Scope s("euler_dss_lap");
    launch_euler_dss_lap(c.st, a);
  }
  nbr_minmax();
  // stage 3: Qdp(np1), gathers qdp_pre, -> qdp_pre2, and its exchange
  a.qdp_n0 = qdp_np1;
  a.fdss = c.omega;
  a.fdss_pre = c.fdss_pre;
  a.rhs_viss = 3.0;
  {
    Scope s("euler_advect");
    launch_euler_advect(c.st, a, 3);
  }
  a.qdp_avg_n0 = qdp_n0;
  Scope s("euler_dss");
  launch_euler_dss(c.st, a, 1);
}

void prim_step(double dt) {
  Ctx &c = C();
  // The accumulators (vn0, omega, eta_dot, the dissipation) and the derived dp
  // start in the first dynamics step's first stage and first subcycle.  (With
  // rsplit > 0 nothing adds to eta_dot: it keeps the zeros it is allocated with.)
  for (int n = 0; n < c.p.qsplit; ++n) {
    if (n > 0) leapfrog();
    if (c.p.moist) update_tracers_levels();
    const double eta_ave_w = 1.0 / c.p.qsplit;
    u3_5stage(c.nm1, c.n0, c.np1, dt, eta_ave_w, n == 0);
    if (c.stopped || stop_here(2)) return;
    hyperviscosity(c.np1, dt, eta_ave_w, n == 0 && c.p.nu_p > 0);
    if (stop_here(3)) return;
  }
  if (c.qsize > 0) advec_tracers(dt * c.p.qsplit);
  stop_here(5);
}

void remap(double dt_remap) {
  Ctx &c = C();
  RemapArgs a{};
  a.nelem = c.nelem;
  a.nlev = c.nlev;
  a.qsize = c.qsize;
  a.nstates = c.p.rsplit > 0 ? 3 : 0;
  a.eta = c.eta_dot;
  a.src = c.pre[0];  // free at the remap
  a.dt = dt_remap;
  a.remap_alg = c.p.remap_alg;
  a.v = c.v[c.np1];
  a.t = c.t[c.np1];
  a.dp = c.dp[c.np1];
  a.ps = c.ps[c.np1];
  a.qdp = c.qsize ? c.qdp[c.np1_qdp] : nullptr;
  a.Q = c.Q;
  a.hyai = c.hyai_d;
  a.hybi = c.hybi_d;
  a.ps0 = c.ps0;
  a.hyai0 = c.hyai0;
  a.error = c.err_d;
  Scope s("remap");
  launch_remap(c.st, a);
}

// ------------------------------------------------------------ adjoint
// Reverse-mode derivative of one dry rsplit = 0 step (no tracers on the
// dynamics path).  The forward stage states are recomputed into private
// buffers first; the step's model state is not touched.
// The stage states of one dynamics step: CAAR stage inputs U0..U4, the
// combination w = (5 u1 - u0)/4 and the HV cycle states H0..Hnsub (U0 is the
// step's input, H[nsub] its output)
struct Stages {
  std::vector<StateBuf> U, H;
  StateBuf W{};
};

struct AdjBufs {
  size_t f3 = 0;  // doubles in one 3-D scalar
  int nsub = 0;
  int nd = 0;  // dynamics steps per prim_run_subcycle_c
  Stages cur;                  // the stage states of one dynamics step
  std::vector<StateBuf> X;     // input states of the nd dynamics steps
  StateBuf LX{}, L0{}, L1{}, LP{}, S{}, M{};
  double *div, *p, *cc, *stot, *pb, *phib, *etab, *ombp, *divb, *lv, *lt, *ldp;
  double *rscr = nullptr;  // remap adjoint scratch (rsplit > 0)
  double *base = nullptr;
};
AdjBufs *adjb = nullptr;

// hommexx_hip_adjoint_segment: the stage states of every dynamics step of a
// segment of calls, so the reverse sweep recomputes none of them
struct SegBufs {
  size_t f3 = 0;
  int nsub = 0, nsets = 0;
  std::vector<Stages> sets;
  StateBuf x{};  // the input of the next call (forward pass)
  double *ps = nullptr;
};
SegBufs *segb = nullptr;

void adj_reset() {
  delete adjb;
  adjb = nullptr;
  delete segb;
  segb = nullptr;
}

StateBuf carve_state(double *&q, size_t f3) {
  StateBuf s{q, q + 2 * f3, q + 3 * f3};
  q += 4 * f3;
  return s;
}

// Fixed device scratch of hommexx_hip_adjoint_step_noalloc: ADJ_SCRATCH_DOUBLES
// (128 MiB) per GPU, held until the process ends.  In host code `scratch`
// only names the symbol: its device address comes from hipGetSymbolAddress,
// once per device with that device current, and only that address goes to
// kernels and copies.
std::map<int, double *> scratch_ptrs;  // device -> the address of its copy of scratch

bool scratch_setup() {
  int dev = 0;
  if (!hipok(hipGetDevice(&dev), "hipGetDevice")) return false;
  if (scratch_ptrs.count(dev)) return true;
  void *p = nullptr;
  if (!hipok(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")) return false;
  scratch_ptrs[dev] = (double *)p;
  return true;
}

double *scratch_pointer() {
  int dev = 0;
  if (!hipok(hipGetDevice(&dev), "hipGetDevice")) return nullptr;
  if (!scratch_ptrs.count(dev) && !scratch_setup()) return nullptr;
  return scratch_ptrs[dev];
}

// doubles of the adjoint step's buffers for nd dynamics steps per call
size_t adj_total_doubles(int nd) {
  Ctx &c = C();
  const size_t f3 = (size_t)c.nelem * c.nlev * 16;
  const int nstates = 5 + 1 + (c.p.hypervis_subcycle + 1) + 6 + nd;  // U, W, H, LX L0 L1 LP S M, X
  return (size_t)nstates * 4 * f3 + 12 * f3 + (size_t)c.nelem * 16 + adj_remap_scratch(c.nelem, c.nlev);
}

// carve the adjoint step's buffers from base (adj_total_doubles(nd) doubles)
void adj_layout(AdjBufs &b, double *base, int nd) {
  Ctx &c = C();
  const size_t f3 = (size_t)c.nelem * c.nlev * 16;
  const int nsub = c.p.hypervis_subcycle;
  b.base = base;
  b.f3 = f3;
  b.nsub = nsub;
  b.nd = nd;
  double *q = b.base;
  b.cur.U.clear();
  b.cur.H.clear();
  b.X.clear();
  for (int i = 0; i < nd; ++i) b.X.push_back(carve_state(q, f3));
  for (int i = 0; i < 5; ++i) b.cur.U.push_back(carve_state(q, f3));
  b.cur.W = carve_state(q, f3);
  for (int i = 0; i <= nsub; ++i) b.cur.H.push_back(carve_state(q, f3));
  b.LX = carve_state(q, f3);
  b.L0 = carve_state(q, f3);
  b.L1 = carve_state(q, f3);
  b.LP = carve_state(q, f3);
  b.S = carve_state(q, f3);
  b.M = carve_state(q, f3);
  double **sc[] = {&b.div, &b.p, &b.cc, &b.pb, &b.phib, &b.etab, &b.ombp, &b.divb, &b.lt, &b.ldp};
  for (double **x : sc) {
    *x = q;
    q += f3;
  }
  b.lv = q;
  q += 2 * f3;
  b.stot = q;
  q += (size_t)c.nelem * 16;
  b.rscr = q;
}

bool adj_alloc(int nd) {
  Ctx &c = C();
  const size_t f3 = (size_t)c.nelem * c.nlev * 16;
  if (adjb && adjb->f3 == f3 && adjb->nsub == c.p.hypervis_subcycle && adjb->nd == nd) return true;
  if (!adjb) adjb = new AdjBufs();
  double *base = dalloc<double>(adj_total_doubles(nd));  // owned by the session (freed with it)
  if (!base) return false;
  adj_layout(*adjb, base, nd);
  return true;
}

void copy_state(const StateBuf &dst, const StateBuf &src, size_t f3) {
  Ctx &c = C();
  hipMemcpyAsync(dst.v, src.v, 4 * f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
}

// y = DSS_r(x) for the four fields of a state
void dss_state(const StateBuf &x, const StateBuf &y) {
  Ctx &c = C();
  DssArgs a{};
  a.nf = 4;
  a.nelem = c.nelem;
  a.nlev = c.nlev;
  a.src = c.dss_src;
  a.rsmp = c.rspheremp;
  const long long es = (long long)c.nlev * 16, ev = (long long)c.nlev * 32;
  a.f[0] = {x.v, y.v, ev, 32};
  a.f[1] = {x.v + 16, y.v + 16, ev, 32};
  a.f[2] = {x.t, y.t, es, 16};
  a.f[3] = {x.dp, y.dp, es, 16};
  launch_dss(c.st, a);
}

// adjoint of out = DSS_r(sph*(a + h*RHS(b))), lam = adjoint of out
// (b: the step's buffers, scratch included)
void caar_adjoint(AdjBufs &b, const StateBuf &xb, const StateBuf &lam, double h, const StateBuf &lb, bool b_acc,
                  const StateBuf &la1, double c1, const StateBuf *la2, double c2) {
  Ctx &c = C();
  dss_state(lam, b.LP);
  AdjCaarArgs a{};
  a.m = metric();
  a.nelem = c.nelem;
  a.nlev = c.nlev;
  a.v = xb.v;
  a.t = xb.t;
  a.dp = xb.dp;
  a.lp_v = b.LP.v;
  a.lp_t = b.LP.t;
  a.lp_dp = b.LP.dp;
  a.hybi = c.hybi_d;
  a.h = h;
  a.p_top = c.hyai0 * c.ps0;
  a.rsplit0 = c.p.rsplit == 0;
  a.div = b.div;
  a.p = b.p;
  a.c = b.cc;
  a.stot = b.stot;
  a.pb = b.pb;
  a.phib = b.phib;
  a.etab = b.etab;
  a.ombp = b.ombp;
  a.divb = b.divb;
  a.lv = b.lv;
  a.lt = b.lt;
  a.ldp = b.ldp;
  a.b_v = lb.v;
  a.b_t = lb.t;
  a.b_dp = lb.dp;
  a.b_acc = b_acc;
  a.a1_v = la1.v;
  a.a1_t = la1.t;
  a.a1_dp = la1.dp;
  a.c1 = c1;
  if (la2) {
    a.a2_v = la2->v;
    a.a2_t = la2->t;
    a.a2_dp = la2->dp;
    a.c2 = c2;
  }
  launch_adj_caar(c.st, a);
}

// adjoint of one hyperviscosity cycle x -> xo; lam (in place)
void hv_adjoint(AdjBufs &b, const StateBuf &x, const StateBuf &xo, const StateBuf &lam, double dt_cycle) {
  Ctx &c = C();
  AdjHvArgs a{};
  a.m = metric();
  a.nelem = c.nelem;
  a.nlev = c.nlev;
  a.x_v = x.v;
  a.xo_v = xo.v;
  a.l_v = lam.v;
  a.l_t = lam.t;
  a.l_dp = lam.dp;
  a.s_v = b.S.v;
  a.s_t = b.S.t;
  a.s_dp = b.S.dp;
  a.m_v = b.M.v;
  a.m_t = b.M.t;
  a.m_dp = b.M.dp;
  a.dt = dt_cycle;
  a.nu = c.p.nu;
  a.nu_s = c.p.nu_s;
  a.nu_p = c.p.nu_p;
  a.nu_top = c.p.nu_top;
  a.nu_ratio1 = c.p.nu_ratio1;
  a.nu_ratio2 = c.p.nu_ratio2;
  launch_adj_hv_pre(c.st, a);
  dss_state(b.S, b.M);
  launch_adj_hv_a(c.st, a);
  dss_state(b.S, b.M);
  launch_adj_hv_b(c.st, a);
}

// Copies between device arrays and rows of host arrays (rows of `row` doubles,
// `stride` apart on the host, adjacent on the device), made when the object goes
// out of scope (or MAX_ARRAYS are pending): nothing is left to do after that.
// They run in pieces through pinned buffers, on up to HostStage::W threads with
// two buffers each, the transfer of one piece beside the host's copy of others.
// A copy to or from pageable memory runs at 18 and 31-37 GB/s and needs a
// contiguous host copy first; a pinned one runs at 56 GB/s, one thread's copy
// between a buffer and the rows at 20-30.  A physics interval at 384 elements L72
// Q4 (141 MB both ways, six steps) took 17.7 ms with the former, 8.9 through one
// thread, 7.1 through four (7.6 two; pieces of 1 MB 8.3, of 4 MB 7.0).
// What fits one buffer goes through it side by side, with one wait for all: in
// pieces an array's transfer is waited for every second array.  Initial states and
// results of 24 elements, 26 levels, 1 tracer: 231 and 260 us in pieces, 194 and
// 239 from pageable memory, 154 and 217 so.
class HostCopy {
 public:
  explicit HostCopy(bool to_host) : c_(C()), to_host_(to_host), lock_(stage_mutex()) {}
  HostCopy(const HostCopy &) = delete;
  // [ie][blocks][block] on the host, one of the blocks on the device
  void levels(double *dev, const double *host, int blocks, int which, size_t block) {
    add(dev, host + (size_t)which * block, block, (size_t)blocks * block);
  }
  // [ie][tl][qsize_d][lev][pt] on the host, [ie][qsize][lev][pt] on the device
  void tracers(double *dev, const double *host, int ntl, int tl) {
    const size_t e3 = (size_t)c_.nlev * 16;
    add(dev, host + (size_t)tl * c_.qsize_d * e3, (size_t)c_.qsize * e3, (size_t)ntl * c_.qsize_d * e3);
  }
  ~HostCopy() { run(); }

 private:
  // what is pending, to its end
  void run() {
    if (!npieces_) return;
    copy();
    narrays_ = 0;
    npieces_ = total_ = 0;
    taken_ = 0;
    error_ = hipSuccess;
  }
  void copy() {
    // (a thread for every 8 MB)
    const size_t share = total_ / (4 * HostStage::PIECE);
    const int n = std::max(1, (int)std::min<size_t>({(size_t)HostStage::W, std::thread::hardware_concurrency(), share}));
    HostStage &s = c_.stage;
    auto pinned = [&](int i) {
      return s.buf[i] || hipok(hipHostMalloc((void **)&s.buf[i], HostStage::PIECE * sizeof(double)), "hipHostMalloc");
    };
    if (total_ <= HostStage::PIECE) {
      if (pinned(0)) copy_small(s.buf[0]);
      return;
    }
    int dev = 0;
    if (!hipok(hipGetDevice(&dev), "host copy")) return;
    for (int i = 0; i < 2 * n; ++i) {
      if (!pinned(i)) return;
      if (!s.ev[i] && !hipok(hipEventCreateWithFlags(&s.ev[i], hipEventDisableTiming), "hipEventCreate")) return;
    }
    std::thread helper[HostStage::W];
    for (int w = 1; w < n; ++w) {
      try {
        helper[w] = std::thread([this, w, dev] {
          if (hipSetDevice(dev) == hipSuccess) work(w);  // (else the others take its pieces)
        });
      } catch (...) {  // (no thread to be had: the others do its share)
        break;
      }
    }
    work(0);
    for (auto &t : helper)
      if (t.joinable()) t.join();
    hipError_t e = (hipError_t)error_.load();
    const hipError_t es = hipStreamSynchronize(c_.st);
    hipok(e != hipSuccess ? e : es, "host copy");
  }
  // all arrays through one buffer
  void copy_small(double *buf) {
    size_t at = 0;
    for (int k = 0; k < narrays_; at += arrays_[k++].n) {
      const Array &a = arrays_[k];
      if (!to_host_) host_copy(a, 0, a.n, buf + at);
      if (!good(to_host_ ? hipMemcpyAsync(buf + at, a.dev, a.n * sizeof(double), hipMemcpyDeviceToHost, c_.st)
                         : hipMemcpyAsync(a.dev, buf + at, a.n * sizeof(double), hipMemcpyHostToDevice, c_.st)))
        break;
    }
    const bool done = good(hipStreamSynchronize(c_.st));
    at = 0;
    for (int k = 0; k < narrays_ && to_host_ && done && error_.load() == hipSuccess; at += arrays_[k++].n)
      host_copy(arrays_[k], 0, arrays_[k].n, buf + at);
    hipok((hipError_t)error_.load(), "host copy");
  }
  static std::mutex &stage_mutex() {
    static std::mutex m;
    return m;
  }
  struct Array {
    double *dev, *host;
    size_t row, stride, n, first;  // first: the array's first piece
  };
  static constexpr int MAX_ARRAYS = 16;  // (cxx_push_results_to_f90 has 16)
  void add(double *dev, const double *host, size_t row, size_t stride) {
    const size_t n = (size_t)c_.nelem * row;
    if (!n) return;
    if (narrays_ == MAX_ARRAYS) run();
    // (the host's rows are written only where to_host_)
    arrays_[narrays_++] = Array{dev, const_cast<double *>(host), row, stride, n, npieces_};
    npieces_ += (n + HostStage::PIECE - 1) / HostStage::PIECE;
    total_ += n;
  }
  // between a buffer and the rows that doubles [off, off + n) of the array cover
  void host_copy(const Array &a, size_t off, size_t n, double *buf) const {
    for (size_t done = 0; done < n;) {
      const size_t o = off + done, r = o / a.row, k = o % a.row, m = std::min(a.row - k, n - done);
      double *h = a.host + r * a.stride + k;
      if (to_host_) memcpy(h, buf + done, m * sizeof(double));
      else memcpy(buf + done, h, m * sizeof(double));
      done += m;
    }
  }
  bool good(hipError_t e) {
    if (e == hipSuccess) return true;
    int none = hipSuccess;
    error_.compare_exchange_strong(none, (int)e);
    return false;
  }
  // one thread's share: buffers 2w and 2w + 1 in turn
  void work(int w) {
    struct Slot {
      const Array *a = nullptr;
      size_t off = 0, n = 0;
    } slot[2];
    auto retire = [&](int i) {
      if (!slot[i].a) return;
      if (good(hipEventSynchronize(c_.stage.ev[2 * w + i])) && to_host_)
        host_copy(*slot[i].a, slot[i].off, slot[i].n, c_.stage.buf[2 * w + i]);
      slot[i].a = nullptr;
    };
    int i = 0;
    for (;; i ^= 1) {
      retire(i);
      const size_t p = taken_.fetch_add(1);
      if (p >= npieces_ || error_.load() != hipSuccess) break;
      int k = narrays_ - 1;
      while (arrays_[k].first > p) --k;
      const Array &a = arrays_[k];
      const size_t off = (p - a.first) * HostStage::PIECE, n = std::min(HostStage::PIECE, a.n - off);
      double *buf = c_.stage.buf[2 * w + i];
      if (!to_host_) host_copy(a, off, n, buf);
      if (!good(to_host_ ? hipMemcpyAsync(buf, a.dev + off, n * sizeof(double), hipMemcpyDeviceToHost, c_.st)
                         : hipMemcpyAsync(a.dev + off, buf, n * sizeof(double), hipMemcpyHostToDevice, c_.st)) ||
          !good(hipEventRecord(c_.stage.ev[2 * w + i], c_.st)))
        break;
      slot[i] = Slot{&a, off, n};
    }
    retire(i ^ 1);
  }
  Ctx &c_;
  const bool to_host_;
  Array arrays_[MAX_ARRAYS];
  int narrays_ = 0;
  size_t npieces_ = 0, total_ = 0;
  std::atomic<size_t> taken_{0};
  std::atomic<int> error_{hipSuccess};
  std::lock_guard<std::mutex> lock_;
};

// Tracers::push_qdp (Tracers.cpp:46-51): both Qdp time levels of every tracer
// slot into the Fortran array (np,np,nlev,qsize_d,2,nelemd); the slots beyond
// qsize go back as they were received at init.
void push_qdp(HostCopy &h, double *Qdp) {
  Ctx &c = C();
  const size_t e3 = (size_t)c.nlev * 16;
  for (int tl = 0; tl < 2; ++tl) h.tracers(c.qdp[tl], Qdp, 2, tl);
  if (c.qsize_d > c.qsize && !c.qdp_tail.empty()) {
    const size_t tail = (size_t)(c.qsize_d - c.qsize) * e3;
    for (int ie = 0; ie < c.nelem; ++ie)
      for (int tl = 0; tl < 2; ++tl)
        memcpy(Qdp + (((size_t)ie * 2 + tl) * c.qsize_d + c.qsize) * e3, &c.qdp_tail[((size_t)ie * 2 + tl) * tail],
               tail * sizeof(double));
  }
}

// CAM forcing buffers FT, FM, FQ, allocated (zeroed, as the reference's
// views are) the first time a forcing run or a forcing push needs them
bool ensure_forcing() {
  Ctx &c = C();
  if (c.ft) return true;
  const size_t e3 = (size_t)c.nelem * c.nlev * 16;
  c.ft = dalloc<double>(e3);
  c.fm = dalloc<double>(2 * e3);
  c.fq = dalloc<double>(e3 * (c.qsize ? c.qsize : 1));
  return c.ft && c.fm && c.fq;
}

// ------------------------------------------------------------ diagnostics
// Diagnostics.cpp:37-185.  The device sums land in a staging buffer; slot
// ivar of each Fortran array is written with strided copies (the other slots
// keep their values, as in the reference).
double *diag_staging() {
  Ctx &c = C();
  if (!c.dg_dev) c.dg_dev = dalloc<double>((size_t)c.nelem * 16 * (4 + 2 * (size_t)c.qsize));
  return c.dg_dev;
}

// slot ivar of a Fortran array [ie][nslot][ncol] from a device array
// [ie][ncol] (ncol doubles per element, the first ncol of a row of width
// row_f doubles in the Fortran array)
void diag_copy(double *f90, int nslot, int ivar, size_t row_f, const double *dev, size_t ncol) {
  Ctx &c = C();
  hipMemcpy2DAsync(f90 + (size_t)ivar * row_f, (size_t)nslot * row_f * sizeof(double), dev, ncol * sizeof(double),
                   ncol * sizeof(double), c.nelem, hipMemcpyDeviceToHost, c.st);
}

DiagArgs diag_args(double *out) {
  Ctx &c = C();
  DiagArgs a{};
  a.nelem = c.nelem;
  a.nlev = c.nlev;
  a.qsize = c.qsize;
  a.use_cpstar = c.p.use_cpstar && c.qsize > 0;
  a.phis = c.phis;
  a.Q = c.Q;
  a.hyai = c.hyai_d;
  a.hybi = c.hybi_d;
  a.ps0 = c.ps0;
  a.out = out;
  return a;
}

// prim_diag_scalars (Diagnostics.cpp:37-88): Q to the Fortran Q array, then
// per column and tracer sum(Qdp*Q) -> qvar[slot], sum(Qdp) -> qmass[slot] and
// q1mass, at tracer level n0_qdp (before the advance) or np1_qdp (after)
void diag_scalars(bool before_advance, int ivar) {
  Ctx &c = C();
  if (!c.dg_set || c.p.time_step_type <= 0) return;
  double *out = diag_staging();
  const size_t e3 = (size_t)c.nlev * 16, nq = (size_t)c.nelem * c.qsize * 16;
  hipStreamSynchronize(c.st);
  HostCopy(true).tracers(c.Q, c.dg[0], 1, 0);
  for (int ie = 0; ie < c.nelem; ++ie)
    for (int q = c.qsize; q < c.qsize_d; ++q) memset(c.dg[0] + ((size_t)ie * c.qsize_d + q) * e3, 0, e3 * sizeof(double));
  if (c.qsize == 0) return;
  DiagArgs a = diag_args(out);
  a.qdp = c.qdp[before_advance ? c.n0_qdp : c.np1_qdp];
  launch_diag_scalars(c.st, a);
  const size_t row = (size_t)c.qsize_d * 16, ncol = (size_t)c.qsize * 16;
  diag_copy(c.dg[1], 4, ivar, row, out, ncol);       // qvar
  diag_copy(c.dg[2], 4, ivar, row, out + nq, ncol);  // qmass
  diag_copy(c.dg[3], 1, 0, row, out + nq, ncol);     // q1mass
  hipok(hipStreamSynchronize(c.st), "prim_diag_scalars");
}

// prim_energy_halftimes (Diagnostics.cpp:90-185) at dynamics level n0 (before
// the advance) or np1 (after): iener, kener, pener [slot] and iener_wet
void diag_energy(bool before_advance, int ivar) {
  Ctx &c = C();
  if (!c.dg_set) return;
  double *out = diag_staging();
  const size_t n = (size_t)c.nelem * 16;
  const int tl = before_advance ? c.n0 : c.np1;
  DiagArgs a = diag_args(out);
  a.v = c.v[tl];
  a.t = c.t[tl];
  a.ps = c.ps[tl];
  a.qdp = c.qdp[before_advance ? c.n0_qdp : c.np1_qdp];
  launch_diag_energy(c.st, a);
  diag_copy(c.dg[4], 4, ivar, 16, out, 16);          // iener
  diag_copy(c.dg[5], 1, 0, 16, out + n, 16);         // iener_wet
  diag_copy(c.dg[6], 4, ivar, 16, out + 2 * n, 16);  // kener
  diag_copy(c.dg[7], 4, ivar, 16, out + 3 * n, 16);  // pener
  hipok(hipStreamSynchronize(c.st), "prim_energy_halftimes");
}

// One dynamics step of the differentiable map from x into the stage states
// s, with the kernels of the forward step (no accumulators for the tracers)
void dyn_forward_stages(const StateBuf &x, Stages &s, double dt) {
  Ctx &c = C();
  const size_t f3 = (size_t)c.nelem * c.nlev * 16;
  const int nsub = c.p.hypervis_subcycle;
  std::vector<StateBuf> &U = s.U, &H = s.H;
  copy_state(U[0], x, f3);
  RkBufs r;
  for (int i = 0; i < 5; ++i) r.u[i] = U[i];
  r.w = s.W;
  r.out = H[0];
  r.keep = true;
  rk_stages(r, dt, 0.0);
  for (int cyc = 0; cyc < nsub; ++cyc) launch_hv_cycle(c.st, hv_args(H[cyc], H[cyc + 1], dt, 0.0), cyc + 1 < nsub);
}

void adj_dyn_forward(AdjBufs &b, int i, double dt) { dyn_forward_stages(b.X[i], b.cur, dt); }

// X[0] from (v, T, ps), then the nd dynamics steps of one
// prim_run_subcycle_c call; H[nsub] holds the last step's output
void adj_forward_steps(AdjBufs &b, int nd, double dt, const double *v, const double *T, const double *ps) {
  Ctx &c = C();
  const size_t f3 = b.f3;
  hipMemcpyAsync(b.X[0].v, v, 2 * f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  hipMemcpyAsync(b.X[0].t, T, f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  launch_dp3d_from_ps(c.st, c.nelem, c.nlev, c.hyai_d, c.hybi_d, c.ps0, ps, b.X[0].dp);
  for (int i = 0; i < nd; ++i) {
    adj_dyn_forward(b, i, dt);
    if (i + 1 < nd) copy_state(b.X[i + 1], b.cur.H[c.p.hypervis_subcycle], f3);
  }
}

// the configurations the differentiable form covers
bool adj_supported(const char *who) {
  Ctx &c = C();
  if (!ready(who)) return false;
  if (c.p.moist || !c.consthv || c.form != 0 || c.p.ftype != -1) {
    fail(70, "%s: needs a dry run, constant-coefficient hyperviscosity, no forcing and the FP64 form", who);
    return false;
  }
  if (!c.be_set) init_boundary_exchanges_c();
  return true;
}

// The reverse sweep of one prim_run_subcycle_c call: on entry lam_* hold
// the adjoint of the call's output (v, T, ps), on return that of its input.
// stages(i) returns the stage states of dynamics step i (recomputed or
// stored); the last step's are asked for first.
template <class F>
void adj_reverse_call(AdjBufs &b, int nd, double dt, F stages, double *lam_v, double *lam_T, double *lam_ps) {
  Ctx &c = C();
  const size_t f3 = b.f3;
  const int nsub = c.p.hypervis_subcycle;
  hipMemcpyAsync(b.LX.v, lam_v, 2 * f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  hipMemcpyAsync(b.LX.t, lam_T, f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  for (int i = nd - 1; i >= 0; --i) {
    const Stages &st = stages(i);
    const std::vector<StateBuf> &U = st.U, &H = st.H;
    if (i == nd - 1) {
      if (c.p.rsplit == 0) {
        launch_adj_fill_dp(c.st, c.nelem, c.nlev, lam_ps, b.LX.dp);  // ps = hyai(0) ps0 + sum_k dp3d
      } else {
        // linearised PPM remap of v and T from the thicknesses of the last step
        AdjRemapArgs r{};
        r.nelem = c.nelem;
        r.nlev = c.nlev;
        r.alg = c.p.remap_alg;
        r.v = H[nsub].v;
        r.t = H[nsub].t;
        r.dp = H[nsub].dp;
        r.l_v = b.LX.v;
        r.l_t = b.LX.t;
        r.l_dp = b.LX.dp;
        r.l_ps = lam_ps;
        r.hyai = c.hyai_d;
        r.hybi = c.hybi_d;
        r.ps0 = c.ps0;
        r.scr = b.rscr;
        launch_adj_remap(c.st, r);
      }
    } else {
      copy_state(b.LX, b.L0, f3);  // adjoint of its output = adjoint of the next step's input
    }
    for (int cyc = nsub - 1; cyc >= 0; --cyc) hv_adjoint(b, H[cyc], H[cyc + 1], b.LX, dt / nsub);
    launch_adj_zero(c.st, 4 * f3, b.L0.v);
    launch_adj_zero(c.st, 4 * f3, b.L1.v);
    // stage 5 from w = (5 u1 - u0)/4 and u4; then stages 4..1
    caar_adjoint(b, U[4], b.LX, 3.0 * dt / 4.0, b.LX, false, b.L1, 1.25, &b.L0, -0.25);
    caar_adjoint(b, U[3], b.LX, 2.0 * dt / 3.0, b.LX, false, b.L0, 1.0, nullptr, 0.0);
    caar_adjoint(b, U[2], b.LX, dt / 3.0, b.LX, false, b.L0, 1.0, nullptr, 0.0);
    caar_adjoint(b, U[1], b.LX, dt / 5.0, b.L1, true, b.L0, 1.0, nullptr, 0.0);
    caar_adjoint(b, U[0], b.L1, dt / 5.0, b.L0, true, b.L0, 1.0, nullptr, 0.0);
  }
  hipMemcpyAsync(lam_v, b.L0.v, 2 * f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  hipMemcpyAsync(lam_T, b.L0.t, f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  launch_adj_ps(c.st, c.nelem, c.nlev, c.hybi_d, b.L0.dp, lam_ps);  // dp3d = dhyai ps0 + dhybi ps
}

// The adjoint step on the buffers b (adj_layout for nd dynamics steps): the
// forward pass keeps each dynamics step's input and the last step's stage
// states; the reverse sweep recomputes the stage states of the others.
int adj_step_run(AdjBufs &b, int nd, double dt, const double *v, const double *T, const double *ps, double *lam_v,
                 double *lam_T, double *lam_ps, const char *who) {
  Ctx &c = C();
  {
    Scope s("adj_forward");
    adj_forward_steps(b, nd, dt, v, T, ps);
  }
  Scope s("adj_reverse");
  auto stages = [&](int i) -> const Stages & {
    if (i < nd - 1) adj_dyn_forward(b, i, dt);
    return b.cur;
  };
  adj_reverse_call(b, nd, dt, stages, lam_v, lam_T, lam_ps);
  return hipok(hipStreamSynchronize(c.st), who) ? 0 : 4;
}

// stage states for nsets dynamics steps (hommexx_hip_adjoint_segment)
bool seg_alloc(int nsets) {
  Ctx &c = C();
  const size_t f3 = (size_t)c.nelem * c.nlev * 16;
  const int nsub = c.p.hypervis_subcycle;
  if (segb && segb->f3 == f3 && segb->nsub == nsub && segb->nsets >= nsets) return true;
  delete segb;
  segb = new SegBufs();
  SegBufs &g = *segb;
  const int per = 5 + 1 + nsub + 1;
  double *q = dalloc<double>(((size_t)nsets * per + 1) * 4 * f3 + (size_t)c.nelem * 16);
  if (!q) {
    delete segb;
    segb = nullptr;
    return false;
  }
  g.f3 = f3;
  g.nsub = nsub;
  g.nsets = nsets;
  g.sets.resize(nsets);
  for (Stages &st : g.sets) {
    for (int i = 0; i < 5; ++i) st.U.push_back(carve_state(q, f3));
    st.W = carve_state(q, f3);
    for (int i = 0; i <= nsub; ++i) st.H.push_back(carve_state(q, f3));
  }
  g.x = carve_state(q, f3);
  g.ps = q;
  return true;
}

}  // namespace

// =================================================================== C-ABI
extern "C" {

// Hommexx_Session.cpp:35
void initialize_hommexx_session() {
  Ctx &c = C();
  if (c.session) return;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
    fail(1, "initialize_hommexx_session: no HIP device");
    return;
  }
  if (!hipok(hipStreamCreateWithFlags(&c.st, hipStreamNonBlocking), "hipStreamCreate")) return;
  if (!scratch_setup()) return;  // the no-allocation adjoint step's array on this device
  c.session = true;
}

// Hommexx_Session.cpp:75
void finalize_hommexx_session() {
  if (!g) return;
  free_all();
  if (g->st) hipStreamDestroy(g->st);
  const bool abort_flag = g->abort_on_error;
  delete g;
  g = nullptr;
  C().abort_on_error = abort_flag;
}

// mpi/mpi_cxx_f90_interface.cpp:20 (one rank: the communicator is recorded only)
void reset_cxx_comm(const int &f_comm) { (void)f_comm; }

// mpi/mpi_cxx_f90_interface.cpp:27
void init_connectivity(const int &num_local_elems) {
  Ctx &c = C();
  if (num_local_elems < 0) {
    fail(30, "init_connectivity: negative element count");
    return;
  }
  c.conn_nelem = num_local_elems;
  c.conn_final = false;
  c.conn_rl.assign((size_t)num_local_elems * 8, -1);
  c.conn_rp.assign((size_t)num_local_elems * 8, -1);
}

// mpi/mpi_cxx_f90_interface.cpp:34-55 (1-based ids, Fortran positions W,E,S,N,SW,SE,NW,NE)
void add_connection(const int &first_lid, const int &first_gid, const int &first_pos, const int &first_pid,
                    const int &second_lid, const int &second_gid, const int &second_pos, const int &second_pid) {
  Ctx &c = C();
  (void)first_gid;
  (void)second_gid;
  if (first_lid <= 0 || first_gid <= 0 || first_pos <= 0 || first_pid <= 0 || second_lid <= 0 || second_gid <= 0 ||
      second_pos <= 0 || second_pid <= 0) {
    fail(31, "add_connection: Fortran indices must start at 1");
    return;
  }
  if (first_pid != 1) return;  // only connections owned by this (single) rank are stored
  if (second_pid != 1) {
    fail(32, "add_connection: remote ranks are not supported on one GPU");
    return;
  }
  auto conv = [](int f) { return f <= 4 ? ((f - 1) + 2) % 4 : f - 1; };
  const int p1 = conv(first_pos), p2 = conv(second_pos);
  if (p1 > 7 || p2 > 7 || (p1 < 4) != (p2 < 4) || first_lid > c.conn_nelem || second_lid > c.conn_nelem) {
    fail(33, "add_connection: invalid connection (%d,%d)->(%d,%d)", first_lid, first_pos, second_lid, second_pos);
    return;
  }
  c.conn_rl[(size_t)(first_lid - 1) * 8 + p1] = second_lid - 1;
  c.conn_rp[(size_t)(first_lid - 1) * 8 + p1] = p2;
}

// mpi/mpi_cxx_f90_interface.cpp:57
void finalize_connectivity() {
  Ctx &c = C();
  for (int ie = 0; ie < c.conn_nelem; ++ie) {
    int missing = 0;
    for (int p = 0; p < 8; ++p) {
      if (c.conn_rl[(size_t)ie * 8 + p] < 0) {
        if (p < 4) {
          fail(34, "finalize_connectivity: element %d has no edge neighbour at position %d", ie + 1, p);
          return;
        }
        ++missing;
      }
    }
    if (missing > 1) {
      fail(35, "finalize_connectivity: element %d misses %d corner neighbours", ie + 1, missing);
      return;
    }
  }
  c.conn_final = true;
}

// cxx_f90_interface.cpp:207
void init_derivative_c(const double *const &dvv) {
  Ctx &c = C();
  memcpy(c.dvv, dvv, sizeof(c.dvv));
  c.dvv_set = true;
}

// cxx_f90_interface.cpp:33-117
void init_simulation_params_c(const int &remap_alg, const int &limiter_option, const int &rsplit, const int &qsplit,
                              const int &time_step_type, const int &energy_fixer, const int &qsize,
                              const int &state_frequency, const double &nu, const double &nu_p, const double &nu_q,
                              const double &nu_s, const double &nu_div, const double &nu_top,
                              const int &hypervis_order, const int &hypervis_subcycle, const double &hypervis_scaling,
                              const int &ftype, const bool &prescribed_wind, const bool &moisture,
                              const bool &disable_diagnostics, const bool &use_cpstar,
                              const bool &use_semi_lagrangian_transport) {
  Ctx &c = C();
  auto bad = [](const char *opt, const char *val) {
    fail(40, "init_simulation_params_c: unsupported option %s = %s", opt, val);
  };
  char buf[64];
  if (remap_alg != 1 && remap_alg != 2) return snprintf(buf, 64, "%d", remap_alg), bad("vert_remap_q_alg", buf);
  if (prescribed_wind) return bad("prescribed_wind", "true");
  if (hypervis_order != 2) return snprintf(buf, 64, "%d", hypervis_order), bad("hypervis_order", buf);
  if (use_semi_lagrangian_transport) return bad("use_semi_lagrangian_transport", "true");
  if (time_step_type != 5) return snprintf(buf, 64, "%d", time_step_type), bad("time_step_type", buf);
  if (limiter_option != 8 && limiter_option != 9)
    return snprintf(buf, 64, "%d", limiter_option), bad("limiter_option", buf);
  if (ftype != -1 && ftype != 0 && ftype != 2) return snprintf(buf, 64, "%d", ftype), bad("ftype", buf);
  if (!(nu_p > 0)) return snprintf(buf, 64, "%g", nu_p), bad("nu_p", buf);
  if (!(nu > 0)) return snprintf(buf, 64, "%g", nu), bad("nu", buf);
  if (!(nu_div > 0)) return snprintf(buf, 64, "%g", nu_div), bad("nu_div", buf);
  if (rsplit < 0) return snprintf(buf, 64, "%d", rsplit), bad("rsplit", buf);
  if (qsplit < 1 || hypervis_subcycle < 1 || qsize < 0)
    return bad("qsplit/hypervis_subcycle/qsize", "out of range");
  Params &p = c.p;
  p.remap_alg = remap_alg;
  p.limiter_option = limiter_option;
  p.rsplit = rsplit;
  p.qsplit = qsplit;
  p.time_step_type = time_step_type;
  p.energy_fixer = energy_fixer;
  p.qsize = qsize;
  p.state_frequency = state_frequency;
  p.nu = nu;
  p.nu_p = nu_p;
  p.nu_q = nu_q;
  p.nu_s = nu_s;
  p.nu_div = nu_div;
  p.nu_top = nu_top;
  p.hypervis_order = hypervis_order;
  p.hypervis_subcycle = hypervis_subcycle;
  p.hypervis_scaling = hypervis_scaling;
  p.ftype = ftype;
  p.prescribed_wind = prescribed_wind;
  p.moist = moisture;
  p.disable_diagnostics = disable_diagnostics;
  p.use_cpstar = use_cpstar;
  p.use_sl = use_semi_lagrangian_transport;
  if (p.nu != p.nu_div) {
    const double ratio = p.nu_div / p.nu;
    if (p.hypervis_scaling != 0.0) {
      p.nu_ratio1 = ratio * ratio;
      p.nu_ratio2 = 1.0;
    } else {
      p.nu_ratio1 = ratio;
      p.nu_ratio2 = ratio;
    }
  } else {
    p.nu_ratio1 = 1.0;
    p.nu_ratio2 = 1.0;
  }
  p.set = true;
}

// cxx_f90_interface.cpp:119 (hyam/hybm are accepted but unused, as in the reference)
void init_hvcoord_c(const double &ps0, const double *const &hybrid_am, const double *const &hybrid_ai,
                    const double *const &hybrid_bm, const double *const &hybrid_bi) {
  Ctx &c = C();
  (void)hybrid_am;
  (void)hybrid_bm;
  if (c.nlev <= 0) c.nlev = c.nlev_cfg;
  const int L = c.nlev;
  c.ps0 = ps0;
  c.hyai.assign(hybrid_ai, hybrid_ai + L + 1);
  c.hybi.assign(hybrid_bi, hybrid_bi + L + 1);
  c.hyai0 = hybrid_ai[0];
  std::vector<double> dp0(L);
  for (int k = 0; k < L; ++k) {
    const double da = c.hyai[k + 1] - c.hyai[k], db = c.hybi[k + 1] - c.hybi[k];
    dp0[k] = da * ps0 + db * ps0;
  }
  if (!c.hyai_d) {
    c.hyai_d = dalloc<double>(L + 1);
    c.hybi_d = dalloc<double>(L + 1);
    c.dp0_d = dalloc<double>(L);
  }
  h2d(c.hyai_d, c.hyai.data(), (L + 1) * sizeof(double));
  h2d(c.hybi_d, c.hybi.data(), (L + 1) * sizeof(double));
  h2d(c.dp0_d, dp0.data(), L * sizeof(double));
  c.hv_set = true;
}

// cxx_f90_interface.cpp:224-233
void init_elements_2d_c(const int &num_elems, const double *const &D, const double *const &Dinv,
                        const double *const &fcor, const double *const &mp, const double *const &spheremp,
                        const double *const &rspheremp, const double *const &metdet, const double *const &metinv,
                        const double *const &phis, const double *const &tensorvisc,
                        const double *const &vec_sph2cart, const bool &consthv) {
  Ctx &c = C();
  if (!c.session) initialize_hommexx_session();
  if (!c.p.set) {
    fail(50, "init_elements_2d_c: init_simulation_params_c must come first");
    return;
  }
  if (c.elems_set) {
    fail(51, "init_elements_2d_c: elements already initialised");
    return;
  }
  c.nelem = num_elems;
  c.nlev = c.nlev_cfg;
  c.qsize = c.p.qsize;
  c.qsize_d = c.qsize_d_cfg > 0 ? c.qsize_d_cfg : std::max(c.qsize, 1);
  if (c.qsize_d < c.qsize) {
    fail(52, "init_elements_2d_c: qsize %d exceeds qsize_d %d", c.qsize, c.qsize_d);
    return;
  }
  const size_t ne = num_elems;
  auto up = [&](double *&dst, const double *src, size_t n) {
    dst = dalloc<double>(n);
    if (src) h2d(dst, src, n * sizeof(double));
  };
  up(c.D, D, ne * 64);
  up(c.Dinv, Dinv, ne * 64);
  up(c.metinv, metinv, ne * 64);
  up(c.fcor, fcor, ne * 16);
  up(c.mp, mp, ne * 16);
  up(c.spheremp, spheremp, ne * 16);
  up(c.rspheremp, rspheremp, ne * 16);
  up(c.metdet, metdet, ne * 16);
  up(c.phis, phis, ne * 16);
  c.consthv = consthv;
  if (!consthv) {
    up(c.tensorvisc, tensorvisc, ne * 64);
    up(c.vec_sph2cart, vec_sph2cart, ne * 96);
  }
  c.dvv_d = dalloc<double>(16);
  h2d(c.dvv_d, c.dvv, sizeof(c.dvv));
  const size_t e3 = ne * c.nlev * 16;
  for (int tl = 0; tl < 3; ++tl) {
    c.v[tl] = dalloc<double>(2 * e3);
    c.t[tl] = dalloc<double>(e3);
    c.dp[tl] = dalloc<double>(e3);
    c.ps[tl] = dalloc<double>(ne * 16);
  }
  for (int tl = 0; tl < 2; ++tl) c.qdp[tl] = dalloc<double>(e3 * (c.qsize ? c.qsize : 1));
  c.Q = dalloc<double>(e3 * (c.qsize ? c.qsize : 1));
  c.omega = dalloc<double>(e3);
  c.eta_dot = dalloc<double>(e3);
  c.dpdiss_ave = dalloc<double>(e3);
  c.dpdiss_bih = dalloc<double>(e3);
  c.derived_dp = dalloc<double>(e3);
  c.divdp = dalloc<double>(e3);
  c.divdp_proj = dalloc<double>(e3);
  c.vn0 = dalloc<double>(2 * e3);
  c.ft = c.fm = c.fq = nullptr;  // CAM forcing buffers: on first use (ensure_forcing)
  c.elems_set = true;
}

// cxx_f90_interface.cpp:235-251
void init_elements_states_c(const double *const &v, const double *const &T, const double *const &dp3d,
                            const double *const &qdp, const double *const &ps_v) {
  Ctx &c = C();
  if (!c.elems_set) {
    fail(53, "init_elements_states_c: init_elements_2d_c must come first");
    return;
  }
  const size_t e3 = (size_t)c.nlev * 16;
  {
    HostCopy h(false);
    for (int tl = 0; tl < 3; ++tl) {
      h.levels(c.v[tl], v, 3, tl, 2 * e3);
      h.levels(c.t[tl], T, 3, tl, e3);
      h.levels(c.dp[tl], dp3d, 3, tl, e3);
      h.levels(c.ps[tl], ps_v, 3, tl, 16);
    }
    for (int tl = 0; tl < 2; ++tl) h.tracers(c.qdp[tl], qdp, 2, tl);
  }
  // tracers beyond qsize are carried unchanged (the reference keeps them in its qdp view)
  c.qdp_tail.clear();
  if (c.qsize_d > c.qsize) {
    const size_t tail = (size_t)(c.qsize_d - c.qsize) * e3;
    c.qdp_tail.resize((size_t)c.nelem * 2 * tail);
    for (int ie = 0; ie < c.nelem; ++ie)
      for (int tl = 0; tl < 2; ++tl)
        memcpy(&c.qdp_tail[((size_t)ie * 2 + tl) * tail], qdp + (((size_t)ie * 2 + tl) * c.qsize_d + c.qsize) * e3,
               tail * sizeof(double));
  }
  c.states_set = true;
}

// cxx_f90_interface.cpp:253-262, Diagnostics.cpp:17-35: the Fortran arrays
// prim_run_subcycle_c fills when diagnostics are enabled
void init_diagnostics_c(double *&q, double *&qvar, double *&qmass, double *&q1mass, double *&iener,
                        double *&iener_wet, double *&kener, double *&pener) {
  Ctx &c = C();
  double *p[8] = {q, qvar, qmass, q1mass, iener, iener_wet, kener, pener};
  bool all = true;
  for (int i = 0; i < 8; ++i) {
    c.dg[i] = p[i];
    all = all && p[i] != nullptr;
  }
  c.dg_set = all;
}

// cxx_f90_interface.cpp:264-280
void init_boundary_exchanges_c() {
  Ctx &c = C();
  if (!c.elems_set || !c.conn_final) {
    fail(54, "init_boundary_exchanges_c: elements and connectivity must be initialised first");
    return;
  }
  if (c.conn_nelem != c.nelem) {
    fail(21, "init_boundary_exchanges_c: connectivity has %d elements, element data %d", c.conn_nelem, c.nelem);
    return;
  }
  if (!c.dss_src) build_dss_tables();
  alloc_work();
}

// cxx_f90_interface.cpp:213-222 (1-based in)
void init_time_level_c(const int &nm1, const int &n0, const int &np1, const int &nstep, const int &nstep0) {
  Ctx &c = C();
  c.nm1 = nm1 - 1;
  c.n0 = n0 - 1;
  c.np1 = np1 - 1;
  c.nstep = nstep;
  c.nstep0 = nstep0;
}

// prim_driver.cpp:31-156: one remap interval.  Indices come back 0-based.
void prim_run_subcycle_c(const double &dt, int &nstep, int &nm1, int &n0, int &np1, const int &last_time_step) {
  Ctx &c = C();
  if (!ready("prim_run_subcycle_c")) return;
  if (!c.be_set) init_boundary_exchanges_c();
  const double dt_q = dt * c.p.qsplit;
  const double dt_remap = c.p.rsplit > 0 ? dt_q * c.p.rsplit : dt_q;
  // prim_driver.cpp:42-63: diagnostics at the state frequency, the first and
  // the last step, unless disabled (or no arrays were registered)
  const int nstep_end = c.nstep + c.p.qsplit * (c.p.rsplit > 0 ? c.p.rsplit : 1);
  const bool diag = !c.p.disable_diagnostics && c.dg_set &&
                    ((c.p.state_frequency > 0 && nstep_end % c.p.state_frequency == 0) || nstep_end == c.nstep0 ||
                     nstep_end >= last_time_step);
  update_tracers_levels();
  if (diag) {
    diag_scalars(true, 3);
    diag_energy(true, 2);
  }
  if ((c.p.ftype == 0 || c.p.ftype == 2) && !ensure_forcing()) return;
  if (c.p.ftype == 0) {
    Scope s("forcing");
    launch_state_forcing(c.st, c.nelem, c.nlev, dt_remap, c.ft, c.fm, c.t[c.n0], c.v[c.n0]);
    launch_tracer_forcing(c.st, c.nelem, c.nlev, c.qsize, c.p.moist, dt_remap, c.fq, c.qdp[c.n0_qdp], c.Q, c.hyai_d,
                          c.hybi_d, c.ps0, c.ps[c.n0]);
  } else if (c.p.ftype == 2) {
    Scope s("forcing");
    launch_state_forcing(c.st, c.nelem, c.nlev, dt_remap, c.ft, c.fm, c.t[c.n0], c.v[c.n0]);
  }
  if (diag) {
    diag_energy(true, 0);
    diag_scalars(true, 0);
  }
  {
    Scope s("dp3d_from_ps");
    launch_dp3d_from_ps(c.st, c.nelem, c.nlev, c.hyai_d, c.hybi_d, c.ps0, c.ps[c.n0], c.dp[c.n0]);
  }
  c.stopped = false;
  prim_step(dt);
  for (int r = 1; r < c.p.rsplit && !c.stopped; ++r) {
    leapfrog();
    prim_step(dt);
  }
  if (c.stopped) {
    hipStreamSynchronize(c.st);
    return;
  }
  update_tracers_levels();
  launch_zero_int(c.st, c.err_d);
  remap(dt_remap);
  if (diag) {
    diag_scalars(false, 1);
    diag_energy(false, 1);
  }
  leapfrog();
  nstep = c.nstep;
  nm1 = c.nm1;
  n0 = c.n0;
  np1 = c.np1;
  hipMemcpyAsync(c.err_h, c.err_d, sizeof(int), hipMemcpyDeviceToHost, c.st);
  if (!hipok(hipStreamSynchronize(c.st), "prim_run_subcycle_c")) return;
  if (*c.err_h & 1) fail(60, "Negative (or nan) layer thickness detected, aborting!");
  else if (*c.err_h & 2) fail(61, "vertical remap: Lagrangian levels deformed by more than one layer");
}

// cxx_f90_interface.cpp:126-154
void cxx_push_results_to_f90(double *&v, double *&T, double *&dp3d, double *&Qdp, double *&Q, double *&ps_v,
                             double *&omega_p) {
  Ctx &c = C();
  if (!c.states_set) {
    fail(55, "cxx_push_results_to_f90: no state");
    return;
  }
  hipStreamSynchronize(c.st);
  const size_t e3 = (size_t)c.nlev * 16;
  HostCopy h(true);
  for (int tl = 0; tl < 3; ++tl) {
    h.levels(c.v[tl], v, 3, tl, 2 * e3);
    h.levels(c.t[tl], T, 3, tl, e3);
    h.levels(c.dp[tl], dp3d, 3, tl, e3);
    h.levels(c.ps[tl], ps_v, 3, tl, 16);
  }
  push_qdp(h, Qdp);
  h.tracers(c.Q, Q, 1, 0);
  for (int ie = 0; ie < c.nelem; ++ie)
    for (int q = c.qsize; q < c.qsize_d; ++q) memset(Q + ((size_t)ie * c.qsize_d + q) * e3, 0, e3 * sizeof(double));
  h.levels(c.omega, omega_p, 1, 0, e3);
}

// cxx_f90_interface.cpp:157-178
void cxx_push_forcing_to_f90(double *FM, double *FT, double *FQ) {
  Ctx &c = C();
  if (!ensure_forcing()) return;
  hipStreamSynchronize(c.st);
  const size_t e3 = (size_t)c.nlev * 16;
  HostCopy h(true);
  h.levels(c.fm, FM, 1, 0, 2 * e3);
  h.levels(c.ft, FT, 1, 0, e3);
  if (c.p.ftype == 0 && FQ) {
    h.tracers(c.fq, FQ, 1, 0);
    // slots beyond qsize: what the last f90_push_forcing_to_cxx sent (zero
    // before any), as the reference's QSIZE_D-wide fq view holds them
    const size_t tail = (size_t)(c.qsize_d - c.qsize) * e3;
    for (int ie = 0; tail && ie < c.nelem; ++ie) {
      double *dst = FQ + ((size_t)ie * c.qsize_d + c.qsize) * e3;
      if (c.fq_tail.empty()) memset(dst, 0, tail * sizeof(double));
      else memcpy(dst, &c.fq_tail[(size_t)ie * tail], tail * sizeof(double));
    }
  }
}

// cxx_f90_interface.cpp:180-205.  FM, FT (and FQ with ftype 0) go to the
// device; Qdp goes the other way, as the reference's tracers.push_qdp does
// (:201): the Fortran array receives the device's Qdp.
void f90_push_forcing_to_cxx(double *FM, double *FT, double *FQ, double *Qdp) {
  Ctx &c = C();
  if (!ensure_forcing()) return;
  const size_t e3 = (size_t)c.nlev * 16;
  hipStreamSynchronize(c.st);
  {
    HostCopy h(false);
    h.levels(c.fm, FM, 1, 0, 2 * e3);
    h.levels(c.ft, FT, 1, 0, e3);
    if (c.p.ftype == 0 && FQ) h.tracers(c.fq, FQ, 1, 0);
  }
  if (c.p.ftype == 0 && FQ) {
    const size_t tail = (size_t)(c.qsize_d - c.qsize) * e3;
    c.fq_tail.resize((size_t)c.nelem * tail);
    for (int ie = 0; tail && ie < c.nelem; ++ie)
      memcpy(&c.fq_tail[(size_t)ie * tail], FQ + ((size_t)ie * c.qsize_d + c.qsize) * e3, tail * sizeof(double));
  }
  if (Qdp && c.states_set) {
    HostCopy h(true);
    push_qdp(h, Qdp);
  }
}

// ============================================================ extensions
// Dimensions the reference fixes at compile time (PLEV, QSIZE_D); call before
// init_elements_2d_c.  Defaults: the build's PREQX_PLEV and QSIZE_D; a
// qsize_d of 0 or less means qsize.  nlev is at most REMAP_MAX_NLEV: the
// remap keeps each element's target table in LDS.
int hommexx_hip_configure(int nlev, int qsize_d) {
  Ctx &c = C();
  if (c.elems_set) return 1;
  if (nlev < 3 || nlev > REMAP_MAX_NLEV) return 2;
  c.nlev_cfg = nlev;
  c.qsize_d_cfg = qsize_d;
  return 0;
}

void hommexx_hip_dimensions(int *nlev, int *qsize_d) {
  Ctx &c = C();
  *nlev = c.nlev_cfg;
  *qsize_d = c.qsize_d_cfg;
}

void hommexx_hip_set_abort_on_error(int on) { C().abort_on_error = on != 0; }

int hommexx_hip_set_form(int form) {
  if (form != 0 && form != 1) return 1;
  C().form = form;
  return 0;
}
// Debugging aid: make prim_run_subcycle_c return after phase n (1: first RK
// stage, 2: all RK stages, 3: hyperviscosity, 4: first tracer stage,
// 5: tracers); 0 disables.  Time levels are not rotated when it stops.
void hommexx_hip_debug_stop(int phase) { C().debug_stop = phase; }
int hommexx_hip_last_error() { return C().last_error; }
const char *hommexx_hip_error_message() { return C().msg.c_str(); }
void hommexx_hip_clear_error() {
  C().last_error = 0;
  C().msg.clear();
}
void hommexx_hip_synchronize() {
  if (C().st) hipStreamSynchronize(C().st);
}
void *hommexx_hip_stream() { return (void *)C().st; }

// Per-phase device timing with HIP events on the library's stream.
void hommexx_hip_profile(int enable) {
  Ctx &c = C();
  if (c.prof && !enable) flush_timers();
  c.prof = enable != 0;
}
void hommexx_hip_profile_only(const char *name) {
  Ctx &c = C();
  c.prof_only = name ? name : "";
}
void hommexx_hip_profile_reset() {
  Ctx &c = C();
  flush_timers();
  c.timers.clear();
}
int hommexx_hip_profile_get(const char *name, int *count, double *total_ms) {
  Ctx &c = C();
  flush_timers();
  auto it = c.timers.find(name);
  if (it == c.timers.end()) {
    *count = 0;
    *total_ms = 0;
    return 1;
  }
  *count = it->second.count;
  *total_ms = it->second.total_ms;
  return 0;
}
// names of the timed phases, '\n'-separated, into buf (returns needed length)
int hommexx_hip_profile_names(char *buf, int len) {
  Ctx &c = C();
  flush_timers();
  std::string s;
  for (auto &kv : c.timers) {
    s += kv.first;
    s += "\n";
  }
  if (buf && len > 0) {
    strncpy(buf, s.c_str(), len - 1);
    buf[len - 1] = 0;
  }
  return (int)s.size() + 1;
}

// ---------------------------------------------------------- differentiable form
// Device copies of the prognostic state at time level n0, in the library's
// layouts: v [ie][lev][2][pt], T [ie][lev][pt], ps [ie][pt].  Used by the
// checkpointing harness.
int hommexx_hip_get_state(double *v, double *T, double *ps) {
  Ctx &c = C();
  if (!c.states_set) {
    fail(55, "hommexx_hip_get_state: no state");
    return 1;
  }
  const size_t f3 = (size_t)c.nelem * c.nlev * 16;
  hipMemcpyAsync(v, c.v[c.n0], 2 * f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  hipMemcpyAsync(T, c.t[c.n0], f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  hipMemcpyAsync(ps, c.ps[c.n0], (size_t)c.nelem * 16 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  return hipok(hipStreamSynchronize(c.st), "hommexx_hip_get_state") ? 0 : 2;
}

// One field of the current state into device memory dst, library layout:
// which 0 = v [ie][lev][2][pt], 1 = T, 2 = dp3d [ie][lev][pt], 3 = ps_v
// [ie][pt] (time level n0), 4 = Qdp of tracer q [ie][lev][pt] (the tracer
// level the next step starts from, (nstep / qsplit) % 2), 5 = Q of tracer q.
int hommexx_hip_get_field(int which, int q, double *dst) {
  Ctx &c = C();
  if (!c.states_set) {
    fail(55, "hommexx_hip_get_field: no state");
    return 1;
  }
  if (which < 0 || which > 5 || (which >= 4 && (q < 0 || q >= c.qsize))) {
    fail(56, "hommexx_hip_get_field: no field %d (tracer %d)", which, q);
    return 1;
  }
  const size_t f3 = (size_t)c.nelem * c.nlev * 16, e3 = (size_t)c.nlev * 16;
  if (which <= 3) {
    const double *srcs[4] = {c.v[c.n0], c.t[c.n0], c.dp[c.n0], c.ps[c.n0]};
    const size_t n[4] = {2 * f3, f3, f3, (size_t)c.nelem * 16};
    hipMemcpyAsync(dst, srcs[which], n[which] * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  } else {
    const double *base = which == 4 ? c.qdp[(c.nstep / c.p.qsplit) % 2] : c.Q;
    hipMemcpy2DAsync(dst, e3 * sizeof(double), base + (size_t)q * e3, (size_t)c.qsize * e3 * sizeof(double),
                     e3 * sizeof(double), c.nelem, hipMemcpyDeviceToDevice, c.st);
  }
  return hipok(hipStreamSynchronize(c.st), "hommexx_hip_get_field") ? 0 : 2;
}

int hommexx_hip_set_state(const double *v, const double *T, const double *ps) {
  Ctx &c = C();
  if (!c.states_set || !c.hv_set) {
    fail(55, "hommexx_hip_set_state: no state");
    return 1;
  }
  const size_t f3 = (size_t)c.nelem * c.nlev * 16;
  hipMemcpyAsync(c.v[c.n0], v, 2 * f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  hipMemcpyAsync(c.t[c.n0], T, f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  hipMemcpyAsync(c.ps[c.n0], ps, (size_t)c.nelem * 16 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  launch_dp3d_from_ps(c.st, c.nelem, c.nlev, c.hyai_d, c.hybi_d, c.ps0, c.ps[c.n0], c.dp[c.n0]);
  return hipok(hipStreamSynchronize(c.st), "hommexx_hip_set_state") ? 0 : 2;
}

// Adjoint of one step of length dt (one prim_run_subcycle_c call) of a dry
// configuration (any rsplit and qsplit; constant-coefficient hyperviscosity;
// the FP64 form), taken at the step's input state (v, T, ps):
// on entry lam_* hold the adjoint of the step's output (v, T, ps), on return
// the adjoint of its input.  All pointers are device memory in the layouts of
// hommexx_hip_get_state.  The model state of the session is not changed.
int hommexx_hip_adjoint_step(double dt, const double *v, const double *T, const double *ps, double *lam_v,
                             double *lam_T, double *lam_ps) {
  Ctx &c = C();
  if (!adj_supported("hommexx_hip_adjoint_step")) return 2;
  // prim_run_subcycle_c: qsplit dynamics steps per prim_step, rsplit (at
  // least one) prim_steps, then the remap (prim_driver.cpp:115-130,
  // prim_step.cpp:57-80)
  const int nd = c.p.qsplit * (c.p.rsplit > 0 ? c.p.rsplit : 1);
  if (!adj_alloc(nd)) return 3;
  return adj_step_run(*adjb, nd, dt, v, T, ps, lam_v, lam_T, lam_ps, "hommexx_hip_adjoint_step");
}

// As hommexx_hip_adjoint_step, but every buffer of the step comes from the
// library's fixed device array `scratch` (ADJ_SCRATCH_DOUBLES doubles, one
// per GPU, held until the process ends) instead of device allocations: for
// callers that cannot allocate (graph capture, serving loops).  Larger
// configurations are rejected (error 71).  All calls on one GPU share its
// array, so calls that overlap on one GPU race.
int hommexx_hip_adjoint_step_noalloc(double dt, const double *v, const double *T, const double *ps, double *lam_v,
                                     double *lam_T, double *lam_ps) {
  Ctx &c = C();
  if (!ready("hommexx_hip_adjoint_step_noalloc")) return 2;
  if (!c.be_set) {
    fail(72, "hommexx_hip_adjoint_step_noalloc: init_boundary_exchanges_c has not run (it allocates)");
    return 2;
  }
  if (!adj_supported("hommexx_hip_adjoint_step_noalloc")) return 2;
  const int nd = c.p.qsplit * (c.p.rsplit > 0 ? c.p.rsplit : 1);
  const size_t need = adj_total_doubles(nd);
  if (need > ADJ_SCRATCH_DOUBLES) {
    fail(71, "hommexx_hip_adjoint_step_noalloc: needs %zu doubles of scratch, the library holds %zu", need,
         (size_t)ADJ_SCRATCH_DOUBLES);
    return 3;
  }
  double *base = scratch_pointer();
  if (!base) return 3;
  static AdjBufs nb;  // the layout is rebuilt only when the configuration changes
  if (nb.base != base || nb.f3 != (size_t)c.nelem * c.nlev * 16 || nb.nsub != c.p.hypervis_subcycle || nb.nd != nd)
    adj_layout(nb, base, nd);
  // the array keeps the last call's contents: start from zeros, as the
  // allocated buffers of hommexx_hip_adjoint_step do
  launch_adj_zero(c.st, need, base);
  return adj_step_run(nb, nd, dt, v, T, ps, lam_v, lam_T, lam_ps, "hommexx_hip_adjoint_step_noalloc");
}


// The adjoint of n consecutive prim_run_subcycle_c calls of length dt (a
// checkpointed segment), from the state (v, T, ps) before the first: the
// forward pass keeps the stage states of every dynamics step (40 F3 each at
// hypervis_subcycle 3), so the reverse sweep recomputes nothing.  lam_* as
// for hommexx_hip_adjoint_step (output adjoint in, input adjoint out).
int hommexx_hip_adjoint_segment(double dt, int n, const double *v, const double *T, const double *ps, double *lam_v,
                                double *lam_T, double *lam_ps) {
  Ctx &c = C();
  if (!adj_supported("hommexx_hip_adjoint_segment")) return 2;
  if (n < 1) {
    fail(73, "hommexx_hip_adjoint_segment: %d calls", n);
    return 2;
  }
  const int nd = c.p.qsplit * (c.p.rsplit > 0 ? c.p.rsplit : 1);
  if (!adj_alloc(nd) || !seg_alloc(n * nd)) return 3;
  AdjBufs &b = *adjb;
  SegBufs &g = *segb;
  const size_t f3 = b.f3;
  const int nsub = c.p.hypervis_subcycle;
  {
    Scope s("adj_forward");
    launch_zero_int(c.st, c.err_d);
    hipMemcpyAsync(g.x.v, v, 2 * f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
    hipMemcpyAsync(g.x.t, T, f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
    launch_dp3d_from_ps(c.st, c.nelem, c.nlev, c.hyai_d, c.hybi_d, c.ps0, ps, g.x.dp);
    for (int call = 0; call < n; ++call) {
      for (int i = 0; i < nd; ++i)
        dyn_forward_stages(i == 0 ? g.x : g.sets[call * nd + i - 1].H[nsub], g.sets[call * nd + i], dt);
      if (call + 1 == n) break;
      // the next call's input: remapped v, T (rsplit > 0), ps from the
      // thicknesses and dp3d from ps, as prim_run_subcycle_c leaves them
      copy_state(g.x, g.sets[call * nd + nd - 1].H[nsub], f3);
      if (c.p.rsplit > 0) {
        RemapArgs a{};
        a.nelem = c.nelem;
        a.nlev = c.nlev;
        a.qsize = 0;
        a.nstates = 3;
        a.remap_alg = c.p.remap_alg;
        a.v = g.x.v;
        a.t = g.x.t;
        a.dp = g.x.dp;
        a.ps = g.ps;
        a.hyai = c.hyai_d;
        a.hybi = c.hybi_d;
        a.ps0 = c.ps0;
        a.hyai0 = c.hyai0;
        a.error = c.err_d;
        launch_remap(c.st, a);
      } else {
        launch_ps_from_dp(c.st, c.nelem, c.nlev, c.hyai0, c.ps0, g.x.dp, g.ps);
      }
      launch_dp3d_from_ps(c.st, c.nelem, c.nlev, c.hyai_d, c.hybi_d, c.ps0, g.ps, g.x.dp);
    }
  }
  {
    Scope s("adj_reverse");
    for (int call = n - 1; call >= 0; --call) {
      auto stages = [&](int i) -> const Stages & { return g.sets[call * nd + i]; };
      adj_reverse_call(b, nd, dt, stages, lam_v, lam_T, lam_ps);
    }
  }
  hipMemcpyAsync(c.err_h, c.err_d, sizeof(int), hipMemcpyDeviceToHost, c.st);
  if (!hipok(hipStreamSynchronize(c.st), "hommexx_hip_adjoint_segment")) return 4;
  if (*c.err_h & 1) {
    fail(60, "Negative (or nan) layer thickness detected, aborting!");
    return 5;
  }
  return 0;
}

// The map hommexx_hip_adjoint_step differentiates, forward: (v, T, ps) is
// advanced in place by the dynamics steps of one prim_run_subcycle_c call and
// the remap of v and T (rsplit > 0), with no tracer step; for a dry run the
// result equals the (v, T, ps) that prim_run_subcycle_c produces.  The
// session's model state is not changed.
int hommexx_hip_dynamics_step(double dt, double *v, double *T, double *ps) {
  Ctx &c = C();
  if (!adj_supported("hommexx_hip_dynamics_step")) return 2;
  const int nd = c.p.qsplit * (c.p.rsplit > 0 ? c.p.rsplit : 1);
  if (!adj_alloc(nd)) return 3;
  AdjBufs &b = *adjb;
  const size_t f3 = b.f3;
  launch_zero_int(c.st, c.err_d);
  adj_forward_steps(b, nd, dt, v, T, ps);
  const StateBuf &o = b.cur.H[c.p.hypervis_subcycle];
  if (c.p.rsplit > 0) {
    RemapArgs a{};
    a.nelem = c.nelem;
    a.nlev = c.nlev;
    a.qsize = 0;
    a.nstates = 3;
    a.remap_alg = c.p.remap_alg;
    a.v = o.v;
    a.t = o.t;
    a.dp = o.dp;
    a.ps = ps;
    a.hyai = c.hyai_d;
    a.hybi = c.hybi_d;
    a.ps0 = c.ps0;
    a.hyai0 = c.hyai0;
    a.error = c.err_d;
    launch_remap(c.st, a);
  } else {
    launch_ps_from_dp(c.st, c.nelem, c.nlev, c.hyai0, c.ps0, o.dp, ps);
  }
  hipMemcpyAsync(v, o.v, 2 * f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  hipMemcpyAsync(T, o.t, f3 * sizeof(double), hipMemcpyDeviceToDevice, c.st);
  hipMemcpyAsync(c.err_h, c.err_d, sizeof(int), hipMemcpyDeviceToHost, c.st);
  if (!hipok(hipStreamSynchronize(c.st), "hommexx_hip_dynamics_step")) return 4;
  if (*c.err_h & 1) {
    fail(60, "Negative (or nan) layer thickness detected, aborting!");
    return 5;
  }
  return 0;
}

// Current time-level indices (0-based) and sizes.
void hommexx_hip_time_levels(int *nm1, int *n0, int *np1, int *nstep, int *n0_qdp, int *np1_qdp) {
  Ctx &c = C();
  *nm1 = c.nm1;
  *n0 = c.n0;
  *np1 = c.np1;
  *nstep = c.nstep;
  *n0_qdp = c.n0_qdp;
  *np1_qdp = c.np1_qdp;
}

}  // extern "C"
