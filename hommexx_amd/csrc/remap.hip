// Vertical remap of (v dp, T dp, Qdp) from the Lagrangian levels back to the
// reference hybrid levels with monotone PPM (RemapFunctor.hpp:226-331,
// PpmRemap.hpp:78-673 in the reference), plus update_q (prim_driver.cpp:171-206).
//
// The reference builds per-column arrays (pio, pin, ppmdx[10], kid, z2, ao,
// dma, ai, parabola coefficients) and then remaps; here one top-to-bottom
// sweep produces the same numbers with O(1) state: source cell j's parabola
// needs ai(j-1), ai(j), which need dma(j-1..j+1) and a, dx up to j+2, so a
// four-cell window suffices, and the target interface k+1 lies in source cell
// kid[k] >= k-1 (kid is found by the same forward search).  Every value is
// computed with the reference's expression and operand order; grid factors
// that depend on the thicknesses only (the reference's ppmdx rows) and the
// target table are evaluated once per column and shared through LDS by all
// the fields of the element's block.
#include <type_traits>

#include "kernels.hpp"

namespace hx {

// ps_v = sum(dp3d) + hyai0*ps0 and the thickness check (ComputeThicknessTag).
// rsplit == 0: the source thickness of the tracer remap is the target
// thickness plus dt*(eta_dot_dpdn(k+1) - eta_dot_dpdn(k)) (RemapFunctor.hpp:62-90).
__global__ __launch_bounds__(256) void remap_thickness_kernel(RemapArgs a) {
  const size_t col = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= (size_t)a.nelem * 16) return;
  const int ie = (int)(col >> 4), pt = (int)(col & 15);
  const double *dp = a.dp + (size_t)ie * a.nlev * 16 + pt;
  double s = 0.0;
  bool bad = false;
  for (int k = 0; k < a.nlev; ++k) {
    const double x = dp[(size_t)k * 16];
    s += x;
    if (a.nstates) bad |= isnan(x) || x < 0.0;
  }
  s += a.hyai0 * a.ps0;
  a.ps[col] = s;
  if (!a.nstates) {
    const double *eta = a.eta + (size_t)ie * a.nlev * 16 + pt;
    double *src = a.src + (size_t)ie * a.nlev * 16 + pt;
    for (int k = 0; k < a.nlev; ++k) {
      const double tgt = (a.hyai[k + 1] - a.hyai[k]) * a.ps0 + (a.hybi[k + 1] - a.hybi[k]) * s;
      const double en = k + 1 < a.nlev ? eta[(size_t)(k + 1) * 16] : 0;
      const double delta = en - eta[(size_t)k * 16];
      const double x = tgt + a.dt * delta;
      src[(size_t)k * 16] = x;
      bad |= isnan(x) || x < 0.0;
    }
  }
  if (bad) atomicOr(a.error, 1);
}

__device__ __forceinline__ double dmin3(double a, double b, double c) {
  const double bc = b < c ? b : c;
  return a < bc ? a : bc;
}

// (the divisions by 3 and 6 below are div_c: the same value, fewer operations)
__device__ __forceinline__ double integrate_parabola(double sq, double lin, double cst, double x1, double x2) {
  return (cst * (x2 - x1) + lin * (x2 * x2 - x1 * x1) / 2.0) + div_c<3>(sq * (x2 * x2 * x2 - x1 * x1 * x1));
}

// dma(j) from a(j-1..j+1) and the grid factors g0, g1, g2 of dx(j-1..j+1)
// (the reference's ppmdx rows 1-3)
__device__ __forceinline__ double ppm_dma_g(double am1, double a0, double a1, double g0, double g1, double g2) {
  if ((a1 - a0) * (a0 - am1) > 0.0) {
    const double da = g0 * (g1 * (a1 - a0) + g2 * (a0 - am1));
    return dmin3(fabs(da), 2.0 * fabs(a0 - am1), 2.0 * fabs(a1 - a0)) * copysign(1.0, da);
  }
  return 0.0;
}

// ai(j) from a(j), a(j+1), dma(j), dma(j+1) and the grid factors of
// dx(j-1..j+2): g3, g4, g56 = g5*(g6-g7), g8, g9 (the product associates
// left to right, so g5*(g6-g7)*(a1-a0) == g56*(a1-a0) exactly)
__device__ __forceinline__ double ppm_ai_g(double a0, double a1, double dma0, double dma1, const double *g) {
  return a0 + g[0] * (a1 - a0) + g[1] * (g[2] * (a1 - a0) - g[3] * dma1 + g[4] * dma0);
}

__device__ __forceinline__ void ppm_parabola(double al, double ar, double a, double &c0, double &c1, double &c2) {
  if ((ar - a) * (a - al) <= 0.) {
    al = a;
    ar = a;
  }
  // the two monotonicity tests share (ar - al) and (ar - al)^2 / 6 unless
  // the first one moves al (same operations and rounding as evaluating each
  // test in full)
  double d = ar - al, q = div_c<6>(d * d);
  if (d * (a - (al + ar) / 2.0) > q) {
    al = 3.0 * a - 2.0 * ar;
    d = ar - al;
    q = div_c<6>(d * d);
  }
  if (d * (a - (al + ar) / 2.0) < -q) ar = 3.0 * a - 2.0 * al;
  c0 = 1.5 * a - (al + ar) / 4.0;
  c1 = ar - al;
  c2 = 3.0 * (-2.0 * a + (al + ar));
}

// ------------------------------------------------------------ split columns
// Block = element; a wave remaps one field at a time: its four 16-lane groups
// hold the 16 columns' levels in four runs of n = ceil(nlev/4), so a field's
// levels are loaded at once into registers (before the first output
// overwrites them) and its sweep is nlev/4 + 4 steps long.  A group starts
// three cells early, for the slopes, edge values and parabola that its first
// target may need, and takes the mass of the cells above from the group above
// (the serial sum goes round the groups, in the reference's order).
//
// A step finishes the parabola of cell c and then target c-1, whose lower
// interface lies in cell c-2, c-1 or c: the three parabolas stay in registers
// and a select takes the right one, so the 16 columns store the same level
// together and no lane waits for another's second target.  If an interface of
// the element moved further (an upward shift by more than a layer), the block
// sweeps each field with one lane a column instead (remap_column).
//
// What depends on the column only is computed once per block and shared
// through LDS: the grid factors of every cell (the reference's ppmdx rows), the
// cell thicknesses and their reciprocals, and for each target level the source
// cell kid that holds its lower interface, the offset z2 in it and the
// reciprocal target thickness.  The thickness sums are serial scans by the
// first 16 lanes; each (target, column) then searches by itself, from the
// interface of its own level.  remap_kernel's search goes on from the last
// target's cell, which is the same unless a target interface lies above the one
// before (ps fell so far that the target thickness is negative): then the first
// 16 lanes take the cells down their columns again.
//
// Bound: the latency of a block's chain, about 8 us of tables and 10 us a round
// of fields (one block of 8 or 12 waves fills a CU's LDS).
constexpr int RG2 = 10;  // grid factors, thickness and its reciprocal, per cell
// the most levels whose tables fit the 160 KB of LDS (80 levels: 152 KB)
constexpr int REMAP_SPLIT_NLEV = 80;

__host__ __device__ inline int remap_run(int nlev) { return (nlev + 3) / 4; }
inline size_t remap_split_lds(int nlev) {
  const size_t lv = 4 * remap_run(nlev), rows = lv + 6;
  const size_t sums = 2 * ((nlev + 7) & ~7) + 4;
  return (rows * RG2 * 16 + sums * 16 + lv * (2 * 16 + 2) + 16) * 8 + lv * 16 * 2 + 16;
}

// f(0), ..., f(N-1) as straight code with constant arguments, so that register
// arrays stay in registers
template <int N, typename F>
__device__ __forceinline__ void unrolled(F &&f) {
  if constexpr (N > 0) {
    unrolled<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// (by value: a select of array elements would put the arrays in memory)
__device__ __forceinline__ double sel3(int i, double a, double b, double c) { return i == 0 ? a : i == 1 ? b : c; }

// One field of one column, top to bottom (fac: the row of Fortran cell -2).
// In place: when the targets of cell c (at most c+1) are written, the levels that
// later cells' parabolas need are in registers up to level c+2 (A2), read before.
// kid does not decrease, so each target is met.  Returns whether all were.
template <typename Put>
__device__ __forceinline__ bool remap_column(const double *fac, const double *zsh, const short *ksh, int L, int alg,
                                             const double *var, unsigned vs, bool state, Put put) {
  auto row = [&](int j) { return fac + (j + 2) * RG2 * 16; };
  auto mirror = [&](int r) { return r < 0 ? -r - 1 : r >= L ? 2 * L - 1 - r : r; };
  // (mass, mean) of Fortran cell j
  double below = 0.0;  // a(L+2) = a(L-1)
  auto mean = [&](int j, double &m) {
    const double *g = row(j);
    const double x = var[(unsigned)mirror(j - 1) * vs];
    m = state ? x * g[128] : x;
    return div_r(m, Recip{g[128], g[144]});
  };
  double m0 = 0.0, m1, m2, dma0, ai_prev = 0.0, prefix = 0.0, mass_prev = 0.0;
  double A0 = mean(0, m0), A1 = mean(1, m1), A2 = mean(2, m2), am1 = mean(-1, m0);
  dma0 = ppm_dma_g(am1, A0, A1, row(-1)[0], row(-1)[16], row(-1)[32]);
  int k = 0;
  for (int j = 0; j <= L; ++j) {
    const double *g = row(j);
    const double dma1 = ppm_dma_g(A0, A1, A2, g[0], g[16], g[32]);
    const double gai[5] = {g[48], g[64], g[80], g[96], g[112]};
    const double ai = ppm_ai_g(A0, A1, dma0, dma1, gai);
    if (j >= 1) {
      const int c = j - 1;
      double cc0, cc1, cc2;
      ppm_parabola(ai_prev, ai, A0, cc0, cc1, cc2);
      if (alg == 2 && (c <= 1 || c >= L - 2)) {
        cc0 = A0;
        cc1 = 0.0;
        cc2 = 0.0;
      }
      for (; k < L && ksh[k * 16] == c; ++k) {
        const double mass = prefix + integrate_parabola(cc2, cc1, cc0, -0.5, zsh[k * 16]) * g[128];
        put(k, k > 0 ? mass - mass_prev : mass);
        mass_prev = mass;
      }
      prefix += m0;
    }
    if (j == L - 2) below = A1;
    A0 = A1;
    A1 = A2;
    m0 = m1;
    m1 = m2;
    if (j + 3 <= L) A2 = mean(j + 3, m2);
    else A2 = j + 3 == L + 1 ? A1 : below;
    dma0 = dma1;
    ai_prev = ai;
  }
  return k == L;
}

template <int N, int FB>
__global__ __launch_bounds__(FB == 1 ? 768 : 512) void remap_split_kernel(RemapArgs a) {
  extern __shared__ double rsm[];
  const int L = a.nlev, n = remap_run(L), nt = blockDim.x;
  const int L4 = 4 * n;  // the groups' levels
  // row of Fortran cell j = -2..4n+3: j+2 (past the column: the mirrored cell)
  double *const fac = rsm;                              // [4n+6][RG2][16]
  double *const pio = fac + (L4 + 6) * RG2 * 16;        // source interfaces 0..L+1, rows for whole batches
  const int R = (L + 7) & ~7;
  double *const pin = pio + (R + 2) * 16;               // target interfaces 0..L
  double *const zsh = pin + (R + 2) * 16;               // z2 [L4][16]
  double *const rtk = zsh + L4 * 16;                    // 1 / target thickness [L4][16]
  double *const dab = rtk + L4 * 16;                    // hyai(k+1) - hyai(k), hybi(k+1) - hybi(k)  [L4][2]
  double *const pss = dab + L4 * 2;                     // ps [16]
  int *const deep = (int *)(pss + 16);                  // a target lies in none of its three cells
  int *const back = deep + 1;                           // a target interface lies above the one before
  short *const ksh = (short *)(deep + 4);               // kid [L4][16]
  double *const dxs = rtk;                              // first the source thicknesses
  const int ie = xcd_block(blockIdx.x, gridDim.x);
  const int tid = threadIdx.x;
  bool bad = false;
  {
    const double *s0 = (a.nstates ? a.dp : a.src) + (size_t)ie * L * 16;
    for (int i = tid; i < L * 16; i += nt) {
      const double x = s0[i];
      if (a.nstates) bad |= isnan(x) || x < 0.0;
      dxs[i] = x;
      pin[i] = x;
    }
    for (int i = L * 16 + tid; i < R * 16; i += nt) pin[i] = 0.0;
    for (int k = tid; k < L; k += nt) {
      dab[2 * k] = a.hyai[k + 1] - a.hyai[k];
      dab[2 * k + 1] = a.hybi[k + 1] - a.hybi[k];
    }
    for (int i = L * 16 + tid; i < L4 * 16; i += nt) {  // (levels past the last: any cell)
      ksh[i] = (short)(i >> 4);
      zsh[i] = 0.0;
    }
    if (tid == 0) *deep = *back = 0;
    if (bad) atomicOr(a.error, 1);
  }
  __syncthreads();
  auto target = [&](int k, double ps) { return dab[2 * k] * a.ps0 + dab[2 * k + 1] * ps; };
  // the mirrored ghosts are dx(0) = dx(1), dx(-1) = dx(2), dx(L+1) = dx(L),
  // dx(L+2) = dx(L-1) (cells further out only feed values nothing uses)
  auto mirror = [&](int r) {
    r = r < 0 ? -r - 1 : r;
    r = r >= L ? 2 * L - 1 - r : r;
    return r < 0 ? 0 : r;
  };
  if (tid < 64) {
    // the first wave: the source interfaces, ps = sum(dp3d) + hyai0*ps0
    // (rsplit == 0: formed with the source thicknesses), the target interfaces
    if (tid < 16) {
      // (the rows past the last, up to a batch of eight: zero thickness)
      double s = 0.0;
      pio[tid] = 0.0;
      column_scan<false>(pin + tid, pio + 16 + tid, R, [&](double x) { return s += x; });
      pio[(L + 1) * 16 + tid] = s + 1.0;
      double ps;
      if (a.nstates) {
        ps = s + a.hyai0 * a.ps0;
        a.ps[(size_t)ie * 16 + tid] = ps;
      } else {
        ps = a.ps[(size_t)ie * 16 + tid];
      }
      pss[tid] = ps;
      double t = 0.0;
      for (int b = 0; b < L; b += 8) {
        double r[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = target(b + i < L ? b + i : L - 1, ps);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          t += r[i];
          pin[(b + i + 1) * 16 + tid] = t;
        }
      }
      pin[L * 16 + tid] = s;
    }
  } else {
    // meanwhile the others: the grid factors
    for (int i = tid - 64; i < (L4 + 6) * 16; i += nt - 64) {
      const int j = (i >> 4) - 2, p = i & 15;
      // dma(j+1) factors from cells j..j+2, ai(j) factors from cells j-1..j+2
      auto dxf = [&](int m) { return dxs[mirror(m - 1) * 16 + p]; };
      const double Xm1 = dxf(j - 1), X0 = dxf(j), X1 = dxf(j + 1), X2 = dxf(j + 2);
      double *g = fac + (size_t)(j + 2) * RG2 * 16 + p;
      g[0] = X1 / (X0 + X1 + X2);
      g[16] = (2.0 * X0 + X1) / (X1 + X2);
      g[32] = (X1 + 2.0 * X2) / (X0 + X1);
      g[48] = X0 / (X0 + X1);
      g[64] = 1.0 / (Xm1 + X0 + X1 + X2);
      g[80] = (2.0 * X0 * X1) / (X0 + X1) * ((Xm1 + X0) / (2.0 * X0 + X1) - (X2 + X1) / (2.0 * X1 + X0));
      g[96] = X0 * (Xm1 + X0) / (2.0 * X0 + X1);
      g[112] = X1 * (X1 + X2) / (X0 + 2.0 * X1);
      g[128] = X0;
      g[144] = 1.0 / X0;
    }
  }
  __syncthreads();
  for (int i = tid; i < L * 16; i += nt) {
    const int k = i >> 4, p = i & 15;
    const double pk = pin[(k + 1) * 16 + p];
    int si = k;
    while (si <= L && pio[si * 16 + p] <= pk) ++si;
    if (si == L + 1) si = L;
    const int kid = si - 1;
    ksh[i] = (short)kid;
    zsh[i] = kid >= 0 ? (pk - (pio[kid * 16 + p] + pio[si * 16 + p]) * 0.5) / fac[((kid + 3) * RG2 + 8) * 16 + p] : 0.0;
    rtk[i] = 1.0 / target(k, pss[p]);
    if (kid > k + 1) *deep = 1;
    if (k > 0 && pk < pin[k * 16 + p]) *back = 1;
    if (kid < 0) atomicOr(a.error, 2);  // below the first interface: not a column the reference remaps
  }
  __syncthreads();
  if (*back) {
    if (tid < 16) {
      int last = 0;
      for (int k = 0; k < L; ++k) {
        const int i = k * 16 + tid, kid = ksh[i];
        if (kid >= last) {
          last = kid;
        } else if (k > 0) {
          ksh[i] = (short)last;
          zsh[i] = (pin[i + 16] - (pio[last * 16 + tid] + pio[(last + 1) * 16 + tid]) * 0.5) /
                   fac[((last + 3) * RG2 + 8) * 16 + tid];
          if (last > k + 1) *deep = 1;
        }
      }
    }
    __syncthreads();
  }

  // ------------------------------------------------------------ fields
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = nt >> 6;
  const int lane = tid & 63, pt = lane & 15, grp = lane >> 4;
  const int c0 = grp * n;
  const int nf = a.nstates + a.qsize, f0 = 3 - a.nstates;  // field 0,1: v components, 2: T, >= 3: tracers
  const double ps = pss[pt];
  const bool general = *deep;
  // the lane's rows of the tables: Fortran cell c0-2, target c0
  const double *const fg = fac + c0 * RG2 * 16 + pt;
  const double *const zg = zsh + c0 * 16 + pt, *const rg = rtk + c0 * 16 + pt, *const dg = dab + 2 * c0;
  const short *const kg = ksh + c0 * 16 + pt;
  // the value of the group above (garbage in group 0)
  auto above = [&](double x) {
    const int src = (lane - 16) * 4;
    return mk64(__builtin_amdgcn_ds_bpermute(src, hi32(x)), __builtin_amdgcn_ds_bpermute(src, lo32(x)));
  };
  for (int fi = wave * FB; fi < nf; fi += nw * FB) {
    // (a slot past the last field repeats the last one, without stores)
    bool state[FB], on[FB];
    unsigned vs[FB];
    double *var[FB], *Qout[FB];
#pragma unroll
    for (int b = 0; b < FB; ++b) {
      on[b] = fi + b < nf;
      const int f = f0 + (on[b] ? fi + b : nf - 1);
      state[b] = f < 3;
      vs[b] = f < 2 ? 32 : 16;
      var[b] = f < 2    ? a.v + (size_t)ie * L * 32 + f * 16
               : f == 2 ? a.t + (size_t)ie * L * 16
                        : a.qdp + ((size_t)ie * a.qsize + (f - 3)) * L * 16;
      Qout[b] = f >= 3 && a.Q ? a.Q + ((size_t)ie * a.qsize + (f - 3)) * L * 16 : nullptr;
    }
    const unsigned qo = (unsigned)c0 * 16 + pt;
    // target c0 + i of the lane
    auto put = [&](int b, int i, double out, const Recip &rt) {
      const unsigned vo = (unsigned)c0 * vs[b] + pt;
      double *const p = var[b] + i * (int)vs[b];
      if (state[b]) {
        p[vo] = div_r(out, rt);
      } else {
        p[vo] = out;
        if (Qout[b]) (Qout[b] + i * 16)[qo] = div_r(out, rt);
      }
    };
    auto thickness = [&](int i) { return Recip{dg[2 * i] * a.ps0 + dg[2 * i + 1] * ps, rg[i * 16]}; };
    if (general) {
#pragma unroll
      for (int b = 0; b < FB; ++b)
        if (grp == 0 && on[b] &&
            !remap_column(fg, zg, kg, L, a.remap_alg, var[b] + pt, vs[b], state[b],
                          [&](int i, double out) { put(b, i, out, thickness(i)); }))
          atomicOr(a.error, 2);
      continue;
    }
    // levels c0-3 .. c0+n+2, all in registers before the first store
    double v[FB][N + 6];
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
      for (int i = 0; i < N + 6; ++i) v[b][i] = var[b][(unsigned)mirror(c0 - 3 + i) * vs[b] + pt];
#pragma unroll
    for (int b = 0; b < FB; ++b) {
#pragma unroll
      for (int i = 0; i < N + 6; ++i) hx::pin(v[b][i]);
      if (state[b]) {
#pragma unroll
        for (int i = 0; i < N + 6; ++i)
          if (i < n + 6) v[b][i] *= fg[(i * RG2 + 8) * 16];
      }
    }
    // the mass above level c0-1: the sum over the levels, from each group to
    // the next (three rounds; all groups add, one more is final in each)
    double vtop[FB], prefix[FB] = {};  // vtop: level c0-1 as a cell (none above the column)
#pragma unroll
    for (int b = 0; b < FB; ++b) vtop[b] = grp ? v[b][2] : 0.0;
#pragma unroll 1
    for (int g = 1; g < 4; ++g) {
      double s[FB];
#pragma unroll
      for (int b = 0; b < FB; ++b) s[b] = prefix[b] + vtop[b];
#pragma unroll
      for (int i = 3; i < N + 2; ++i)
        if (i < n + 2)
#pragma unroll
          for (int b = 0; b < FB; ++b) s[b] += v[b][i];
#pragma unroll
      for (int b = 0; b < FB; ++b) {
        s[b] = above(s[b]);
        prefix[b] = grp ? s[b] : 0.0;
      }
    }
    double A0[FB], A1[FB], dma0[FB] = {}, ai_prev[FB] = {}, mass[FB] = {}, mfirst[FB] = {};
    {
      const Recip r0{fg[8 * 16], fg[9 * 16]}, r1{fg[(RG2 + 8) * 16], fg[(RG2 + 9) * 16]};
#pragma unroll
      for (int b = 0; b < FB; ++b) {
        A0[b] = div_r(v[b][0], r0);
        A1[b] = div_r(v[b][1], r1);
      }
    }
    // parabola and mass above of the last three cells
    double q0[FB][3] = {}, q1[FB][3] = {}, q2[FB][3] = {}, qp[FB][3] = {};
    unrolled<N + 4>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = ic;
      // (c and n are made anew in each step: hoisted out of the field loop, the
      // conditions on them filled the scalar registers)
      int nn = n, c = c0 + i - 3;  // c: the cell
      asm volatile("" : "+s"(nn));
      asm volatile("" : "+v"(c));
      if (i >= nn + 4) return;
      const double *g = fg + i * RG2 * 16;  // Fortran cell j = c0 - 2 + i
      const double h0 = g[0], h1 = g[16], h2 = g[32];
      const double gai[5] = {g[48], g[64], g[80], g[96], g[112]};
      const Recip r2{g[(2 * RG2 + 8) * 16], g[(2 * RG2 + 9) * 16]};
      constexpr int s = i % 3, s1 = (i + 2) % 3, s2 = (i + 1) % 3;  // its slot, and of cells c-1, c-2
      int up = 0;
      double z2 = 0.0, dx = 0.0;
      Recip rt{};
      if (i >= 4) {
        up = c - kg[(i - 4) * 16];  // 0, 1 or 2 cells above, for target c-1
        dx = g[8 * 16 - up * (RG2 * 16)];
        z2 = zg[(i - 4) * 16];
        rt = thickness(i - 4);
      }
#pragma unroll
      for (int b = 0; b < FB; ++b) {
        const double A2 = div_r(v[b][i + 2], r2);
        const double dma1 = ppm_dma_g(A0[b], A1[b], A2, h0, h1, h2);         // dma(j+1)
        const double ai = ppm_ai_g(A0[b], A1[b], dma0[b], dma1, gai);  // ai(j)
        if (i >= 2) {
          ppm_parabola(ai_prev[b], ai, A0[b], q0[b][s], q1[b][s], q2[b][s]);
          if (a.remap_alg == 2 && (c <= 1 || c >= L - 2)) {
            q0[b][s] = A0[b];
            q1[b][s] = 0.0;
            q2[b][s] = 0.0;
          }
          qp[b][s] = prefix[b];
          if (i >= 4) {
            const double p0 = sel3(up, q0[b][s], q0[b][s1], q0[b][s2]);
            const double p1 = sel3(up, q1[b][s], q1[b][s1], q1[b][s2]);
            const double p2 = sel3(up, q2[b][s], q2[b][s1], q2[b][s2]);
            const double pp = sel3(up, qp[b][s], qp[b][s1], qp[b][s2]);
            const double m = pp + integrate_parabola(p2, p1, p0, -0.5, z2) * dx;
            if (i == 4) mfirst[b] = m;
            else if (c - 1 < L && on[b]) put(b, i - 4, m - mass[b], rt);
            mass[b] = m;
          }
          prefix[b] += i == 2 ? vtop[b] : v[b][i];
        }
        A0[b] = A1[b];
        A1[b] = A2;
        dma0[b] = dma1;
        ai_prev[b] = ai;
      }
      // (a step's loads and arithmetic stay in it)
#pragma unroll
      for (int b = 0; b < FB; ++b) {
        hx::pin(A0[b]);
        hx::pin(A1[b]);
        hx::pin(dma0[b]);
        hx::pin(ai_prev[b]);
      }
    });
    // a group's first target takes the mass of the last one above it
#pragma unroll
    for (int b = 0; b < FB; ++b) {
      const double m = above(mass[b]);
      if (c0 < L && on[b]) put(b, 0, grp ? mfirst[b] - m : mfirst[b], thickness(0));
    }
  }
}

// ---------------------------------------------------------- one lane a column
// One block = one element (16 GLL columns) and up to 16*RFB fields; lane
// (row, pt) sweeps column pt for fields f0 + (16*blockIdx.y + row)*RFB + i
// (field 0,1: v components, 2: T, >= 3: tracer field-3).  What depends on
// the column only is computed once per block and shared through LDS:
// * the target table: for each target level k the source cell kid(k) that
//   holds its lower interface and the offset z2(k) in it (the reference's
//   kid and z2 arrays, the same forward search), found by the 16 lanes of
//   row 0 before the sweep;
// * the grid factors of RCH sweep iterations at a time (the reference's
//   ppmdx rows for dma(j+1) and ai(j), dx(j) and the incoming dx(j+3)),
//   iteration j0 + row computed by row row.
constexpr int RCH = 16;  // sweep iterations per grid chunk (rows 0..RCH-1 compute one each)
constexpr int RG = 11;   // shared grid values per (iteration, column)

size_t remap_lds_bytes(int nlev) { return (size_t)RCH * RG * 16 * 8 + (size_t)nlev * (16 * (8 + 8 + 2) + 2 * 8); }

template <int RFB>  // fields per lane
__global__ __launch_bounds__(256) void remap_kernel(RemapArgs a) {
  extern __shared__ double rsm[];
  const int L = a.nlev;
  double *gsh = rsm;                              // [RCH][RG][16]
  double *zsh = rsm + RCH * RG * 16;              // z2  [L][16]
  double *rtk = zsh + (size_t)L * 16;             // 1 / (target thickness)  [L][16]
  double *dab = rtk + (size_t)L * 16;             // hyai(k+1) - hyai(k), hybi(k+1) - hybi(k)  [L][2]
  short *ksh = (short *)(dab + (size_t)L * 2);    // kid [L][16]
  const int ie = xcd_block(blockIdx.x, gridDim.x);
  const int row = threadIdx.x >> 4, pt = threadIdx.x & 15;
  const int nf = 3 + a.qsize;    // in the field numbering above
  const int f0 = 3 - a.nstates;  // rsplit == 0: tracers only
  const int fb = f0 + (blockIdx.y * 16 + row) * RFB;
  const bool active = fb < nf;
  const size_t col = (size_t)ie * 16 + pt;
  const double *src = (a.nstates ? a.dp : a.src) + (size_t)ie * L * 16 + pt;
  const double ps = a.ps[col];
  // wait for that load on every path here (s_waitcnt vmcnt(0); expcnt and
  // lgkmcnt left at their maxima: 0x0F70 on gfx9): only row 0 uses ps before
  // the sweep, and without the wait the compiler's waits inside the sweep
  // assume it may still be in flight and also wait for the prefetched loads
  __builtin_amdgcn_s_waitcnt(0x0F70);
  // dx of Fortran cell m = 1..L with the mirrored ghosts dx(0) = dx(1),
  // dx(-1) = dx(2), dx(L+1) = dx(L), dx(L+2) = dx(L-1)
  auto dxf = [&](int m) {
    int c = m - 1;
    c = c < 0 ? -c - 1 : (c >= L ? 2 * L - 1 - c : c);
    return src[(size_t)c * 16];
  };

  // ------------------------------------------------------------ targets
  for (int k = threadIdx.x; k < L; k += blockDim.x) {
    dab[2 * k] = a.hyai[k + 1] - a.hyai[k];
    dab[2 * k + 1] = a.hybi[k + 1] - a.hybi[k];
  }
  // The element's source thicknesses go through LDS (the grid chunk's space,
  // free until the sweep) when they fit, so the serial search below waits on
  // LDS rather than on one global load per step.
  const bool lsrc = L <= RCH * RG;
  if (lsrc) {
    const double *s0 = (a.nstates ? a.dp : a.src) + (size_t)ie * L * 16;
    for (int i = threadIdx.x; i < L * 16; i += blockDim.x) gsh[i] = s0[i];
  }
  __syncthreads();
  auto search = [&](auto sat) {  // sat(c): thickness of source cell c of this column
    double pio_L = 0.0;  // pio(L): serial sum of the source thicknesses
    for (int c = 0; c < L; ++c) pio_L += sat(c);
    double pin_acc = 0.0, pio_si = 0.0, pio_m1 = 0.0, pio_m2 = 0.0;  // pio(si), pio(si-1), pio(si-2)
    int si = 0;
    auto advance_si = [&]() {
      pio_m2 = pio_m1;
      pio_m1 = pio_si;
      pio_si = si < L ? pio_si + sat(si) : pio_si + 1.0;  // pio(L+1) = pio(L) + 1
      ++si;
    };
    for (int k = 0; k < L; ++k) {
      double pin_k1;
      if (k + 1 < L) {
        pin_acc += dab[2 * k] * a.ps0 + dab[2 * k + 1] * ps;  // the target thickness of level k
        pin_k1 = pin_acc;
      } else {
        pin_k1 = pio_L;  // pin(L) = pio(L)
      }
      while (si < k) advance_si();  // the search for target k starts at interface k
      while (si <= L && pio_si <= pin_k1) advance_si();
      int kk = si;
      double plo = pio_m1, phi = pio_si;  // pio(kk-1), pio(kk)
      if (kk == L + 1) {
        kk = L;
        plo = pio_m2;
        phi = pio_m1;
      }
      const int kid = kk - 1;
      ksh[k * 16 + pt] = (short)kid;
      zsh[k * 16 + pt] = kid >= 0 ? (pin_k1 - (plo + phi) * 0.5) / sat(kid) : 0.0;
    }
  };
  if (row == 0) {
    if (lsrc) search([&](int c) { return gsh[c * 16 + pt]; });
    else search([&](int c) { return src[(size_t)c * 16]; });
  } else {
    // meanwhile the other rows form the reciprocals of the target
    // thicknesses (the outputs' divisor, shared by the fields)
    for (int k = row - 1; k < L; k += 15) rtk[k * 16 + pt] = 1.0 / (dab[2 * k] * a.ps0 + dab[2 * k + 1] * ps);
  }

  // ------------------------------------------------------------ fields
  // (pointers of absent fields stay valid device addresses, never null, so
  // every access compiles to a global, not a flat, instruction).  An absent
  // field slot of a lane (on[i] false: past the last tracer) is swept like
  // the others on its stand-in values and only its stores are skipped: the
  // sweep then has no per-field branches (1941 -> 1891 us at 43 fields)
  // (its loads read the first L*16 values of T, in bounds)
  double *var[RFB];
  double *Qout[RFB];
  size_t vs[RFB];
  bool on[RFB], state[RFB], qout[RFB];
#pragma unroll
  for (int i = 0; i < RFB; ++i) {
    const int f = fb + i;
    on[i] = f < nf;
    state[i] = f < 3;
    qout[i] = f >= 3 && f < nf && a.Q != nullptr;
    vs[i] = f < 2 ? 32 : 16;
    var[i] = a.t;
    Qout[i] = a.t;
    if (f < 2) var[i] = a.v + (size_t)ie * L * 32 + f * 16 + pt;
    else if (f == 2) var[i] = a.t + (size_t)ie * L * 16 + pt;
    else if (f < nf) {
      var[i] = a.qdp + (((size_t)ie * a.qsize + (f - 3)) * L) * 16 + pt;
      if (qout[i]) Qout[i] = a.Q + (((size_t)ie * a.qsize + (f - 3)) * L) * 16 + pt;
    }
  }
  const int alg = a.remap_alg;
  // Fortran-style cell indices j = 1..L.  Per field (A0..A2) = a(j..j+2),
  // V0..V2 = var(j..j+2)
  double A0[RFB], A1[RFB], A2[RFB], V0[RFB], V1[RFB], V2[RFB];
  double dma_j[RFB], ai_prev[RFB], var_prefix[RFB], mass_prev[RFB];
  double cc0[RFB], cc1[RFB], cc2[RFB];
  double pv[RFB], qv[RFB];  // field values of cells j+3, j+4 (loaded ahead)
  // unconditional loads (past the bottom the last cell is reloaded; an
  // absent field reads its stand-in pointer): with a branch here every later
  // wait would also cover the loads just issued
  auto fetch = [&](int m, double *v) {
    const size_t c = (size_t)((m <= L ? m : L) - 1);
#pragma unroll
    for (int i = 0; i < RFB; ++i) v[i] = var[i][c * vs[i]];
  };
  if (active) {
    const double s0 = src[0], s1 = src[16];
    // dma(0) factors: dx(-1), dx(0), dx(1) = s1, s0, s0
    const double g0 = s0 / (s1 + s0 + s0);
    const double g1 = (2.0 * s1 + s0) / (s0 + s0);
    const double g2 = (s0 + 2.0 * s0) / (s1 + s0);
#pragma unroll
    for (int i = 0; i < RFB; ++i) {
      const double x0 = var[i][0], x1 = var[i][vs[i]];
      const double v0 = state[i] ? x0 * s0 : x0, v1 = state[i] ? x1 * s1 : x1;
      const double a1 = v0 / s0, a2 = v1 / s1;
      A0[i] = a1;  // a(0) = a(1)
      A1[i] = a1;
      A2[i] = a2;
      V0[i] = 0.0;
      V1[i] = v0;
      V2[i] = v1;
      dma_j[i] = ppm_dma_g(a2, A0[i], A1[i], g0, g1, g2);  // dma(0), a(-1) = a(2)
      ai_prev[i] = 0.0;
      var_prefix[i] = 0.0;
      mass_prev[i] = 0.0;
    }
    fetch(3, pv);
    fetch(4, qv);
  }

  // ------------------------------------------------------------ sweep
  int k = 0;  // next target level
  bool live = active;
  for (int j0 = 0; j0 <= L; j0 += RCH) {
    __syncthreads();  // the previous chunk's grid values are consumed (and the target table is written)
    {
      const int j = j0 + row;
      if (row < RCH && j <= L) {
        // window dx(j-1..j+2): dma(j+1) factors use cells j..j+2, ai(j) factors cells j-1..j+2
        const double Xm1 = dxf(j - 1), X0 = dxf(j), X1 = dxf(j + 1), X2 = dxf(j + 2);
        double *g = gsh + row * RG * 16 + pt;
        g[0] = X1 / (X0 + X1 + X2);
        g[16] = (2.0 * X0 + X1) / (X1 + X2);
        g[32] = (X1 + 2.0 * X2) / (X0 + X1);
        g[48] = X0 / (X0 + X1);
        g[64] = 1.0 / (Xm1 + X0 + X1 + X2);
        g[80] = (2.0 * X0 * X1) / (X0 + X1) * ((Xm1 + X0) / (2.0 * X0 + X1) - (X2 + X1) / (2.0 * X1 + X0));
        g[96] = X0 * (Xm1 + X0) / (2.0 * X0 + X1);
        g[112] = X1 * (X1 + X2) / (X0 + 2.0 * X1);
        g[128] = X0;
        g[144] = dxf(j + 3);  // the cell entering the window (used for j + 3 <= L)
        g[160] = 1.0 / g[144];
      }
    }
    __syncthreads();
    if (!live) continue;
    const int jn = L + 1 - j0 < RCH ? L + 1 - j0 : RCH;
    // (unrolled by 3: the window's shift through A0..A2 and V0..V2 becomes
    // register renaming in two of three steps; 2030 -> 2004 us)
#pragma unroll 3
    for (int jj = 0; jj < jn; ++jj) {
      const int j = j0 + jj;
      double nv[RFB];
      fetch(j + 5, nv);
      const double *g = gsh + jj * RG * 16 + pt;
      const double h0 = g[0], h1 = g[16], h2 = g[32];
      const double gai[5] = {g[48], g[64], g[80], g[96], g[112]};
      const double X0 = g[128];
      double dma_j1[RFB], ai_j[RFB];
#pragma unroll
      for (int i = 0; i < RFB; ++i) {
        dma_j1[i] = ppm_dma_g(A0[i], A1[i], A2[i], h0, h1, h2);       // dma(j+1)
        ai_j[i] = ppm_ai_g(A0[i], A1[i], dma_j[i], dma_j1[i], gai);  // ai(j)
      }
      if (j >= 1) {
        const int c = j - 1;  // physical source cell, Fortran cell j
#pragma unroll
        for (int i = 0; i < RFB; ++i) {
          ppm_parabola(ai_prev[i], ai_j[i], A0[i], cc0[i], cc1[i], cc2[i]);
          if (alg == 2 && (c <= 1 || c >= L - 2)) {
            cc0[i] = A0[i];
            cc1[i] = 0.0;
            cc2[i] = 0.0;
          }
        }
        // kid is non-decreasing in k (each search continues from the last
        // interface reached, starting no lower than k), so every target is
        // finished while the sweep is at its own cell kid(k)
        while (k < L) {
          const int kid = ksh[k * 16 + pt];
          if (kid > c) break;
          if (kid < c) {
            atomicOr(a.error, 2);  // deformation beyond one layer: not supported
            live = false;
            break;
          }
          const double z2 = zsh[k * 16 + pt];
          const double tk = dab[2 * k] * a.ps0 + dab[2 * k + 1] * ps;  // the reference's (hyai(k+1)-hyai(k))*ps0 + ...
          const Recip rt{tk, rtk[k * 16 + pt]};
#pragma unroll
          for (int i = 0; i < RFB; ++i) {
            const double integral = integrate_parabola(cc2[i], cc1[i], cc0[i], -0.5, z2);
            const double mass = var_prefix[i] + integral * X0;
            const double out = k > 0 ? mass - mass_prev[i] : mass;
            mass_prev[i] = mass;
            if (!on[i]) continue;
            if (state[i]) {
              var[i][(size_t)k * vs[i]] = div_r(out, rt);
            } else {
              var[i][(size_t)k * vs[i]] = out;
              if (qout[i]) ((__attribute__((address_space(1))) double *)Qout[i])[(size_t)k * 16] = div_r(out, rt);
            }
          }
          ++k;
        }
        if (!live) break;
#pragma unroll
        for (int i = 0; i < RFB; ++i) var_prefix[i] += V0[i];
      }
      // shift: bring in cell j+3
      const int m = j + 3;
      const Recip rxn{g[144], g[160]};
#pragma unroll
      for (int i = 0; i < RFB; ++i) {
        double an, vn = 0.0;
        if (m <= L) {
          const double x = pv[i];
          vn = state[i] ? x * rxn.b : x;
          an = div_r(vn, rxn);
        } else if (m == L + 1) {
          an = A2[i];  // a(L+1) = a(L)
        } else {
          an = A0[i];  // a(L+2) = a(L-1)
        }
        A0[i] = A1[i]; A1[i] = A2[i]; A2[i] = an;
        V0[i] = V1[i]; V1[i] = V2[i]; V2[i] = vn;
        ai_prev[i] = ai_j[i];
        dma_j[i] = dma_j1[i];
        pv[i] = qv[i];
        qv[i] = nv[i];
      }
    }
  }
  if (live && k < L) atomicOr(a.error, 2);
}

__global__ void zero_int_kernel(int *p) { *p = 0; }

// a fill kernel rather than a memset node, so the step stays graph-capturable
void launch_zero_int(hipStream_t st, int *p) { hipLaunchKernelGGL(zero_int_kernel, dim3(1), dim3(1), 0, st, p); }

// ps_v = sum(dp3d) + hyai0*ps0, summed as remap_thickness_kernel does
__global__ __launch_bounds__(256) void ps_from_dp_kernel(int nelem, int nlev, double hyai0, double ps0,
                                                          const double *dp, double *ps) {
  const size_t col = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= (size_t)nelem * 16) return;
  const double *d = dp + (col >> 4) * nlev * 16 + (col & 15);
  double s = 0.0;
  for (int k = 0; k < nlev; ++k) s += d[(size_t)k * 16];
  ps[col] = s + hyai0 * ps0;
}

void launch_ps_from_dp(hipStream_t st, int nelem, int nlev, double hyai0, double ps0, const double *dp, double *ps) {
  const size_t ncol = (size_t)nelem * 16;
  hipLaunchKernelGGL(ps_from_dp_kernel, dim3((ncol + 255) / 256), dim3(256), 0, st, nelem, nlev, hyai0, ps0, dp, ps);
}

// Split columns are the shorter chain, one lane a column the fewer
// instructions a field (its lanes share a column's tables over up to 4 fields).
// Measured, us, split against one lane a column (with its thickness kernel):
//   few fields:    ne30 L72 3 fields 456/812, 7 fields L26 257/291, L40 385/435
//   long columns:  ne30 L72 15 fields 942/1137, 23 1276/1523, 27 1641/1583,
//                  43 2319/1981; L40 15 fields 624/545, L26 15 fields 440/365
//   few elements:  ne4 L26 7 fields 17/52, 43 51/76; ne8 L72 43 217/253, L26 43
//                  104/102; ne11 (726 elements) L26 43 157/129
// Below 20 levels the chain that is split is short, and a wave's slopes and
// tables ahead of its first target (4 + 4 steps whatever the run) weigh more:
//   3 to 8 levels: ne30 L3 8 fields 140/54, L6 162/82; ne16 L5 6 fields 48/29; ne8
//                  L6 8 fields 19/22, 15 fields 28/23; ne11 4 fields 15/21
//   12 levels:     ne16 6 fields 55/51, ne11 8 fields 32/37, ne30 4 fields 88/105
//   16, 17 levels: ne16 8 fields 61/76; ne24 8 fields L17 144/143; ne30 8 fields L17
//                  219/202, 4 fields 109/175
// (a block has four waves at least, so fewer fields cost it what four do).
constexpr int REMAP_SPLIT_ELEMS = 512;  // two blocks per CU
static bool remap_split(int nelem, int nlev, int nfld) {
  if (nlev > REMAP_SPLIT_NLEV || nfld == 0) return false;
  if (nlev < 20 && !(nfld <= 4 && nlev >= 8)) {
    const int waves = nlev >= 16 ? 28000 : nlev >= 12 ? 7000 : 4000;
    if ((long long)nelem * (nfld < 4 ? 4 : nfld) > waves) return false;
  }
  return nfld <= 8 || (nlev > 64 && nfld <= 24) || nelem <= REMAP_SPLIT_ELEMS;
}

void launch_remap(hipStream_t st, const RemapArgs &a) {
  const int nfld = a.nstates + a.qsize;
  const bool split = remap_split(a.nelem, a.nlev, nfld);
  // (the split kernel forms ps itself; the source thicknesses of rsplit == 0
  // need it first)
  if (!split || !a.nstates) {
    const size_t ncol = (size_t)a.nelem * 16;
    hipLaunchKernelGGL(remap_thickness_kernel, dim3((ncol + 255) / 256), dim3(256), 0, st, a);
  }
  if (nfld == 0) return;
  if (split) {
    const size_t lds = remap_split_lds(a.nlev);
    const int n = remap_run(a.nlev);
    // two fields a wave (eight waves, 256 VGPRs) where twelve waves of one
    // would need a second round: ne60 L72 13 fields 3.35 ms against 3.55
    const bool two = nfld > 12;
    // (where only one block fits a CU's LDS, spare waves help with the tables)
    const int waves = two ? 8 : lds > 80 * 1024 ? 12 : nfld < 4 ? 4 : nfld;
    auto go = [&](auto *kernel) { hipLaunchKernelGGL(kernel, dim3(a.nelem), dim3(64 * waves), lds, st, a); };
    if (n <= 8) go(two ? remap_split_kernel<8, 2> : remap_split_kernel<8, 1>);
    else if (n <= 18) go(two ? remap_split_kernel<18, 2> : remap_split_kernel<18, 1>);
    else go(two ? remap_split_kernel<20, 2> : remap_split_kernel<20, 1>);
    return;
  }
  // fields per lane: as few as fill the 16 rows (at most 4, then more
  // blocks per element)
  const int rfb = nfld <= 16 ? 1 : nfld <= 32 ? 2 : nfld <= 48 ? 3 : 4;
  const dim3 g(a.nelem, (nfld + 16 * rfb - 1) / (16 * rfb));
  const size_t lds = remap_lds_bytes(a.nlev);
  switch (rfb) {
    case 1: hipLaunchKernelGGL(remap_kernel<1>, g, dim3(256), lds, st, a); break;
    case 2: hipLaunchKernelGGL(remap_kernel<2>, g, dim3(256), lds, st, a); break;
    case 3: hipLaunchKernelGGL(remap_kernel<3>, g, dim3(256), lds, st, a); break;
    default: hipLaunchKernelGGL(remap_kernel<4>, g, dim3(256), lds, st, a); break;
  }
}

}  // namespace hx
