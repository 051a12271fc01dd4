// Far field by direct summation over every surface node (zero at coincident
// points): u(t) = sum_j w_j (ubn_j / r - ub_j (x - y_j).n_j / r^3) / (4 pi).
//
// Reference: stellarator_grf_core_mod.f90:560-611
//
// Bound by the FP64 vector rate: 17 FP64 operations, one v_rsq_f64 and a select
// per (target, node), about 96 issue cycles per wave of 64 pairs; measured 102
// (200,000 targets x 513,000 nodes: 68 ms; one thread a target with the sources
// in LDS and IEEE divide and square root took 246 ms, and 102 ms at 50,000
// targets, now 17, because 196 workgroups left the chip idle).  Sources are packed once per call into one 64-byte record
// each (position, and the strengths with the quadrature weight, 1/(4 pi) and the
// normal multiplied in), which every wave reads with uniform addresses, so they
// come through the scalar cache and feed the arithmetic from scalar registers:
// no LDS traffic, and kFT targets per thread share each record.  The sources are
// split into chunks so that few targets still fill the chip; each chunk's sums
// go to part(chunk, target) and are added in chunk order, so the result does not
// depend on timing.
//
// Where the packed form could leave the FP64 range -- a position or strength beyond
// kFarHuge or not a number -- the sum is formed again term by term (far_plain): a source
// like that is packed with a strength that is not a number, which makes every sum one,
// and sums that are not finite, or whose target lies that far, are formed again.  The
// direct kernel itself tests nothing.
#include <algorithm>

#include "qol_kernels.h"

namespace qol {

namespace {

// below this no square of a coordinate difference and no product with a strength leaves
// the FP64 range
constexpr double kFarHuge = 1e150;

struct FarSources {
  const double *sx, *snx, *sw, *ub, *ubn;
};

// the sum over sources j0 .. j1 - 1 at x, term by term; a source whose r^2 is not above
// the coincidence threshold (or not a number) is left out, strength and all
__device__ double far_plain(const FarSources& S, int j0, int j1, const double* x) {
  const double pi4inv = 1.0 / (16.0 * atan(1.0));
  double acc = 0.0;
#pragma unroll 1
  for (int j = j0; j < j1; ++j) {
    const double *y = S.sx + 3 * (size_t)j, *n = S.snx + 3 * (size_t)j;
    const double dx = x[0] - y[0], dy = x[1] - y[1], dz = x[2] - y[2];
    const double rr = dx * dx + dy * dy + dz * dz;
    if (rr > 1.0e-28) {
      const double ri = 1.0 / sqrt(rr), w = pi4inv * S.sw[j];
      acc += w * S.ubn[j] * ri - w * S.ub[j] * (dx * n[0] + dy * n[1] + dz * n[2]) * ri * ri * ri;
    }
  }
  return acc;
}

}  // namespace

__global__ void __launch_bounds__(256) far_pack_kernel(int ns, FarSources S, double2* __restrict__ src) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= ns) return;
  const double pi4inv = 1.0 / (16.0 * atan(1.0));
  const double *y = S.sx + 3 * (size_t)j, *n = S.snx + 3 * (size_t)j;
  const double w = pi4inv * S.sw[j], d = w * S.ub[j];
  double v[7] = {y[0], y[1], y[2], w * S.ubn[j], d * n[0], d * n[1], d * n[2]};
  bool out = false;
#pragma unroll
  for (int c = 0; c < 7; ++c) out |= !(fabs(v[c]) < kFarHuge);
  if (out) v[3] = __builtin_nan("");
  double2* o = src + 4 * (size_t)j;
  o[0] = double2{v[0], v[1]};
  o[1] = double2{v[2], v[3]};
  o[2] = double2{v[4], v[5]};
  o[3] = double2{v[6], 0.0};
}

// one wave per tile of 64 kFT targets and chunk of sources
template <int kFT>
__global__ void __launch_bounds__(64) far_direct_kernel(int nt, const double* __restrict__ tx, int ns, int len,
                                                        const double* __restrict__ src, double* __restrict__ part) {
  const int t0 = blockIdx.x * 64 * kFT + threadIdx.x;
  double x[kFT][3], acc[kFT];
#pragma unroll
  for (int i = 0; i < kFT; ++i) {
    const size_t t = min(t0 + 64 * i, nt - 1);
    x[i][0] = tx[3 * t];
    x[i][1] = tx[3 * t + 1];
    x[i][2] = tx[3 * t + 2];
    acc[i] = 0.0;
  }
  const int j0 = blockIdx.y * len, j1 = min(ns, j0 + len);
#pragma unroll 2
  for (int j = j0; j < j1; ++j) {
    const double* s = src + 8 * (size_t)j;
    const double s0 = s[0], s1 = s[1], s2 = s[2], s3 = s[3], s4 = s[4], s5 = s[5], s6 = s[6];
#pragma unroll
    for (int i = 0; i < kFT; ++i) {
      const double dx = x[i][0] - s0, dy = x[i][1] - s1, dz = x[i][2] - s2;
      const double rr = fma(dz, dz, fma(dy, dy, dx * dx));
      const double ri = rr > 1.0e-28 ? rsqrt_h3(rr) : 0.0;
      const double dn = fma(dz, s6, fma(dy, s5, dx * s4));
      acc[i] = fma(ri, fma(-dn, ri * ri, s3), acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < kFT; ++i)
    if (t0 + 64 * i < nt) part[(size_t)blockIdx.y * nt + t0 + 64 * i] = acc[i];
}

// u(t) = sum of part(c, t): 64 targets per workgroup, each of the 4 waves adds
// every fourth chunk in order, then the four sums are added in order; the same four
// waves form a sum again
__global__ void __launch_bounds__(256) far_sum_kernel(int nt, int nchunk, int ns, FarSources S,
                                                      const double* __restrict__ tx, const double* __restrict__ part,
                                                      double* __restrict__ u) {
  __shared__ double s[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int t = blockIdx.x * 64 + lane;
  double acc = 0.0;
  if (t < nt)
#pragma unroll 8
    for (int c = wv; c < nchunk; c += 4) acc += part[(size_t)c * nt + t];
  s[wv][lane] = acc;
  __syncthreads();
  double v = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
  const size_t tc = min(t, nt - 1);
  const double x[3] = {tx[3 * tc], tx[3 * tc + 1], tx[3 * tc + 2]};
  const bool again = t < nt && !(isfinite(v) && fabs(x[0]) < kFarHuge && fabs(x[1]) < kFarHuge && fabs(x[2]) < kFarHuge);
  if (__syncthreads_or(again)) {
    const int per = (ns + 3) / 4;
    s[wv][lane] = again ? far_plain(S, wv * per, min(ns, (wv + 1) * per), x) : 0.0;
    __syncthreads();
    if (again) v = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
  }
  if (wv == 0 && t < nt) u[t] = v;
}

// Measured (targets x sources, billions of pairs a second): four targets a thread
// and 32,768 waves run 200,000 x 513,000 at 1,510 and 20,011 x 79,464 at 1,520;
// one target a thread at 1,420 and 1,380 (each record feeds a quarter of the
// arithmetic), 4,096 waves at 1,280 on the second (a few long waves end last).
// Below four tiles' worth of targets the shorter waves of one or two targets a
// thread win: 100 x 15,800 takes 8.7, 9.5 and 13.1 us at one, two and four.
FarPlan far_plan(int nt, int ns) {
  FarPlan P;
  P.per = nt > 256 ? 4 : (nt > 64 ? 2 : 1);
  const int tiles = (nt + 64 * P.per - 1) / (64 * P.per);
  // no chunk below 32 sources, and at most 512 sums a target to add up
  const int n = std::min({(32768 + tiles - 1) / tiles, (ns + 31) / 32, 512});
  P.len = (ns + n - 1) / n;
  P.nchunk = (ns + P.len - 1) / P.len;
  return P;
}

void launch_far(const FarPlan& P, int nt, const double* tx, int ns, const double* sx, const double* snx,
                const double* sw, const double* ub, const double* ubn, double* src, double* part, double* u,
                hipStream_t s) {
  const FarSources S{sx, snx, sw, ub, ubn};
  hipLaunchKernelGGL(far_pack_kernel, dim3((ns + 255) / 256), dim3(256), 0, s, ns, S, (double2*)src);
  const dim3 grid((nt + 64 * P.per - 1) / (64 * P.per), P.nchunk);
  switch (P.per) {
    case 1: hipLaunchKernelGGL(far_direct_kernel<1>, grid, dim3(64), 0, s, nt, tx, ns, P.len, src, part); break;
    case 2: hipLaunchKernelGGL(far_direct_kernel<2>, grid, dim3(64), 0, s, nt, tx, ns, P.len, src, part); break;
    default: hipLaunchKernelGGL(far_direct_kernel<4>, grid, dim3(64), 0, s, nt, tx, ns, P.len, src, part); break;
  }
  hipLaunchKernelGGL(far_sum_kernel, dim3((nt + 63) / 64), dim3(256), 0, s, nt, P.nchunk, ns, S, tx, part, u);
}

}  // namespace qol
