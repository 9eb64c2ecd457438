// Direct stiffness summation on one GPU (BoundaryExchange.cpp:285-618 in the
// reference, all connections LOCAL).  Instead of packing edge buffers, every
// output point gathers the neighbour copies it needs from the pre-exchange
// field.  The per-point source list (built on the host from the connection
// table) is already in the reference's accumulation order -- for k = 0..3
// the S, N, W, E edges, then the SW, SE, NW, NE corners -- so
//     out(p) = ((own(p) + c1) + c2) + c3     then  * rspheremp(p)
// rounds exactly like the reference's unpack.
#include "kernels.hpp"

namespace hx {

// One lane = one (element, level, point) for every field of the call: the
// source table is read once and all the fields' loads are issued before the
// first sum, so each lane has up to 4*nf independent loads in flight.
__global__ __launch_bounds__(256) void dss_kernel(DssArgs a) {
  int ie, k, pt;
  if (!group_slab(a.nelem, a.nlev, ie, k, pt)) return;
  const int *src = a.src + ((size_t)ie * 16 + pt) * 3;
  const int s0 = src[0], s1 = src[1], s2 = src[2];
  const double r0 = a.rsmp ? a.rsmp[(size_t)ie * 16 + pt] : 1.0;
  // all loads of all fields are issued before the first sum (gather_sum);
  // an absent source re-reads the own value
  auto at = [&](const DssField &F, int src, size_t own) {
    return opaque_index(src >= 0 ? (size_t)(src >> 4) * F.estride + (size_t)k * F.lstride + (src & 15) : own);
  };
  double r[DSS_MAX_FIELDS][4];
#pragma unroll
  for (int f = 0; f < DSS_MAX_FIELDS; ++f) {
    if (f < a.nf) {
      const DssField &F = a.f[f];
      const size_t own = (size_t)ie * F.estride + (size_t)k * F.lstride + pt;
      r[f][0] = F.in[own];
      r[f][1] = F.in[at(F, s0, own)];
      r[f][2] = F.in[at(F, s1, own)];
      r[f][3] = F.in[at(F, s2, own)];
    }
  }
#pragma unroll
  for (int f = 0; f < DSS_MAX_FIELDS; ++f) {
    if (f < a.nf) {
      const DssField &F = a.f[f];
      const double x = gather_sum(r[f], s0, s1, s2);
      F.out[(size_t)ie * F.estride + (size_t)k * F.lstride + pt] = a.rsmp ? x * r0 : x;
    }
  }
}

void launch_dss(hipStream_t st, const DssArgs &a) {
  if (a.nf <= 0) return;
  const dim3 g(group_blocks_x(a.nelem, a.nlev));
  hipLaunchKernelGGL(dss_kernel, g, dim3(256), 0, st, a);
}

}  // namespace hx
