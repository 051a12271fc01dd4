// Recursive-reduction quadrature (RRQ) for the targets no refinement level can
// serve: per-panel set-up, the quaternion system and its weights operator, and
// the per-target boundary moments, recursion and weights.
//
// Reference: rrq_r64                       lap3d_close_mod.f90:622-881
//            build_closepanel_precomp_r64  lap3d_close_mod.f90:472-620
//            build_tc_chialpha_r64         lap3d_close_mod.f90:336-470
//            (SSQ weights, solid angle, omega moments: absent LQ/QA modules,
//             re-derived -- see the oracle header for the identities used)
// FP64 throughout.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <stdexcept>

#include "qol_kernels.h"

namespace qol {

// ---------------------------------------------------------------------------
// geometry polynomial x(u,v) = sum_k K_k(u,v) cx[c][k] and its uv derivatives,
// accumulated while the Koornwinder basis is generated (no h-sized arrays).
// The recurrence constants come from the per-order table kt (koorn_eval_table:
// no divisions or square roots here): kt[2am], kt[2am+1] scale the Legendre
// step to am, and term t (loop order am, bd) has its normalisation and Jacobi
// coefficients at kt[2N + 4t .. 2N + 4t + 3].
__device__ void geom_eval(const double* cx, const double* __restrict__ kt, int h, int korder, double u, double v,
                          double* x, double* xu, double* xv) {
  const int N = korder + 1;
  const double a = 2.0 * u + v - 1.0, b = 1.0 - v, bb = b * b;
  for (int c = 0; c < 3; ++c) { x[c] = 0.0; if (xu) { xu[c] = 0.0; xv[c] = 0.0; } }
  const double xx = 2.0 * v - 1.0;
  // Q_am(a, b) (scaled Legendre in a/b) and its u, v derivatives advance with am;
  // for each am, Jacobi P_bd^(2am+1,0)(xx) by its three-term recurrence in bd.
  // Basis index of (degree d = am + bd, bd) is d(d+1)/2 + bd.
  double Q = 1.0, Qu = 0.0, Qv = 0.0, Qm = 0.0, Qum = 0.0, Qvm = 0.0;
  const double* tt = kt + 2 * N;
  for (int am = 0; am < N; ++am) {
    if (am == 1) {
      Qm = Q; Qum = Qu; Qvm = Qv;
      Q = a; Qu = 2.0; Qv = 1.0;
    } else if (am >= 2) {
      const double e1 = kt[2 * am], e2 = kt[2 * am + 1];
      const double Qn = e1 * a * Q - e2 * bb * Qm;
      const double Qun = e1 * (2.0 * Q + a * Qu) - e2 * bb * Qum;
      const double Qvn = e1 * (Q + a * Qv) - e2 * (bb * Qvm - 2.0 * b * Qm);
      Qm = Q; Qum = Qu; Qvm = Qv;
      Q = Qn; Qu = Qun; Qv = Qvn;
    }
    const double al = 2.0 * am + 1.0;
    double p = 1.0, dp = 0.0, pm = 1.0, dpm = 0.0;
    for (int bd = 0; am + bd < N; ++bd, tt += 4) {
      if (bd == 1) {
        p = 0.5 * ((al + 2.0) * xx + al);
        dp = al + 2.0;
      } else if (bd >= 2) {
        const double w = tt[1] + tt[2] * xx;
        const double pn = w * p - tt[3] * pm;
        const double dpn = w * dp + 2.0 * tt[2] * p - tt[3] * dpm;
        pm = p; p = pn; dpm = dp; dp = dpn;
      }
      const int d = am + bd, idx = d * (d + 1) / 2 + bd;
      const double sc = tt[0];
      const double f = sc * Q * p;
      for (int c = 0; c < 3; ++c) x[c] += f * cx[c * h + idx];
      if (xu) {
        const double fu = sc * Qu * p, fv = sc * (Qv * p + Q * dp);
        for (int c = 0; c < 3; ++c) { xu[c] += fu * cx[c * h + idx]; xv[c] += fv * cx[c * h + idx]; }
      }
    }
  }
}

std::vector<double> koorn_eval_table(int N) {
  std::vector<double> t(2 * (size_t)N, 0.0);
  for (int am = 2; am < N; ++am) {
    const int m = am - 1;
    const double inv = 1.0 / (double)(m + 1);
    t[2 * am] = (2.0 * m + 1.0) * inv;
    t[2 * am + 1] = (double)m * inv;
  }
  for (int am = 0; am < N; ++am) {
    const double al = 2.0 * am + 1.0;
    for (int bd = 0; am + bd < N; ++bd) {
      const int d = am + bd;
      double ca = 0.0, cb = 0.0, cc = 0.0;
      if (bd >= 2) {
        const double dk = (double)(bd - 1);
        const double a1 = 2.0 * (dk + 1.0) * (dk + al + 1.0) * (2.0 * dk + al);
        const double a2 = (2.0 * dk + al + 1.0) * al * al;
        const double a3 = (2.0 * dk + al) * (2.0 * dk + al + 1.0) * (2.0 * dk + al + 2.0);
        const double a4 = 2.0 * (dk + al) * dk * (2.0 * dk + al + 2.0);
        ca = a2 / a1; cb = a3 / a1; cc = a4 / a1;
      }
      t.insert(t.end(), {std::sqrt((2.0 * am + 1.0) * 2.0 * (double)(d + 1)), ca, cb, cc});
    }
  }
  return t;
}

__device__ __forceinline__ void cross3(const double* a, const double* b, double* c) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}

// frame[] = R (rows e1,e2,e3), c, alpha, sigma, L
__device__ __forceinline__ void to_frame(const double* fr, const double* x, double* X) {
  const double d0 = x[0] - fr[9], d1 = x[1] - fr[10], d2 = x[2] - fr[11];
  for (int r = 0; r < 3; ++r) X[r] = fr[12] * (fr[3 * r] * d0 + fr[3 * r + 1] * d1 + fr[3 * r + 2] * d2);
}
__device__ __forceinline__ void rotate(const double* fr, const double* v, double* V) {
  for (int r = 0; r < 3; ++r) V[r] = fr[3 * r] * v[0] + fr[3 * r + 1] * v[1] + fr[3 * r + 2] * v[2];
}

// Im((-i)^m z)
__device__ __forceinline__ double imrot(int m, cd z) {
  switch (m & 3) {
    case 0: return z.im;
    case 1: return -z.re;
    case 2: return -z.im;
    default: return z.re;
  }
}

// ---------------------------------------------------------------------------
size_t rrq_frame_smem(int h, int nq) {
  const int nb = 3 * nq;
  return (size_t)(7 * h + 3 * h + 16 + 9 * nq + 6 * nb + h) * sizeof(double);
}
// complex values per boundary node in P.basis: H'_n^m (n < p, 0 <= m <= n), then
// T_n^m (n < p - 1, 0 <= m <= n + 1)
size_t rrq_basis_doubles(int p, int nq) {
  return (size_t)2 * 3 * nq * (p * (p + 1) / 2 + (p - 1) * (p + 2) / 2);
}

// One workgroup per panel (with RRQ pairs, or every panel when nrrq is null):
// Koornwinder coefficients, orientation, frame, boundary nodes and the edges'
// Legendre coefficients -- what the per-pair projection and edge kernels need.
__global__ void __launch_bounds__(256) rrq_panel_frame_kernel(RRQTables T, RRQPanels P, int npan,
                                                              const int* __restrict__ nrrq,
                                                              const double* __restrict__ sx,
                                                              const double* __restrict__ snx,
                                                              const double* __restrict__ sw, int ichart,
                                                              const double* __restrict__ sxbd_chart,
                                                              const double* __restrict__ rv_chart) {
  const int k = blockIdx.x;
  if (nrrq && nrrq[k] == 0) return;  // null: every panel
  extern __shared__ double sm[];
  const int h = T.h, nq = T.nq, p = T.p, nb = 3 * nq;
  double* ssx = sm;             // [3][h]
  double* ssn = ssx + 3 * h;    // [3][h]
  double* ssw = ssn + 3 * h;    // [h]
  double* scx = ssw + h;        // [3][h]
  double* fr = scx + 3 * h;     // 16
  double* ecf = fr + 16;        // [3 edges][3][nq]
  double* bx = ecf + 9 * nq;    // [nb][6]
  double* sg = bx + 6 * nb;     // [h] sigma contributions
  const size_t gk = (size_t)k * h;
  for (int i = threadIdx.x; i < h; i += blockDim.x) {
    for (int c = 0; c < 3; ++c) {
      ssx[c * h + i] = sx[3 * (gk + i) + c];
      ssn[c * h + i] = snx[3 * (gk + i) + c];
    }
    ssw[i] = sw[gk + i];
  }
  __syncthreads();
  // Koornwinder coefficients cx = umatr * sx
  for (int i = threadIdx.x; i < 3 * h; i += blockDim.x) {
    const int c = i / h, a = i % h;
    double s = 0.0;
    for (int q = 0; q < h; ++q) s += T.umatr[a + (size_t)h * q] * ssx[c * h + q];
    scx[c * h + a] = s;
    P.cx[(size_t)k * 3 * h + c * h + a] = s;
  }
  __syncthreads();
  // orientation: sigma = sign(sum (x_u x x_v) . snx) over the nodes
  for (int i = threadIdx.x; i < h; i += blockDim.x) {
    double x[3], xu[3], xv[3], n[3];
    geom_eval(scx, T.ktab, h, p - 1, T.uvn[2 * i], T.uvn[2 * i + 1], x, xu, xv);
    cross3(xu, xv, n);
    sg[i] = n[0] * ssn[i] + n[1] * ssn[h + i] + n[2] * ssn[2 * h + i];
  }
  // triangle vertices, one thread each (the patch at (0,0), (1,0), (0,1), or the chart's)
  __shared__ double srv[9];
  if (threadIdx.x < 3) {
    const int j = threadIdx.x;
    if (ichart == 1) {
      for (int c = 0; c < 3; ++c) srv[3 * j + c] = rv_chart[9 * (size_t)k + 3 * j + c];
    } else {
      double xv[3];
      geom_eval(scx, T.ktab, h, p - 1, j == 1 ? 1.0 : 0.0, j == 2 ? 1.0 : 0.0, xv, nullptr, nullptr);
      for (int c = 0; c < 3; ++c) srv[3 * j + c] = xv[c];
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double rv[9];
    for (int i = 0; i < 9; ++i) rv[i] = srv[i];
    double swsum = 0.0, acc = 0.0, mn[3] = {0, 0, 0};
    for (int i = 0; i < h; ++i) {
      swsum += ssw[i];
      acc += sg[i];
      for (int c = 0; c < 3; ++c) mn[c] += ssn[c * h + i];
    }
    const double alpha = 1.25 / sqrt(2.0 * swsum);
    double a[3], b[3], nrm[3], axb[3], t1[3], t2[3];
    for (int c = 0; c < 3; ++c) { a[c] = rv[3 + c] - rv[c]; b[c] = rv[6 + c] - rv[c]; }
    cross3(a, b, nrm);
    const double nn = sqrt(nrm[0] * nrm[0] + nrm[1] * nrm[1] + nrm[2] * nrm[2]);
    double e3[3] = {nrm[0] / nn, nrm[1] / nn, nrm[2] / nn};
    if (mn[0] * e3[0] + mn[1] * e3[1] + mn[2] * e3[2] < 0.0) for (int c = 0; c < 3; ++c) e3[c] = -e3[c];
    const double la = sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
    double e1[3] = {a[0] / la, a[1] / la, a[2] / la}, e2[3];
    cross3(e3, e1, e2);
    cross3(a, b, axb);
    const double aa = a[0] * a[0] + a[1] * a[1] + a[2] * a[2], bbv = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
    cross3(axb, a, t1);
    cross3(b, axb, t2);
    const double den = 2.0 * (axb[0] * axb[0] + axb[1] * axb[1] + axb[2] * axb[2]);
    double c0[3];
    for (int c = 0; c < 3; ++c) c0[c] = rv[c] + (bbv * t1[c] + aa * t2[c]) / den;
    for (int c = 0; c < 3; ++c) { fr[c] = e1[c]; fr[3 + c] = e2[c]; fr[6 + c] = e3[c]; fr[9 + c] = c0[c]; }
    fr[12] = alpha;
    double zmin = 1e300;
    for (int i = 0; i < h; ++i) {
      double x[3] = {ssx[i], ssx[h + i], ssx[2 * h + i]}, X[3];
      to_frame(fr, x, X);
      zmin = fmin(zmin, X[2]);
    }
    const double s3 = fmax(0.0, -zmin);
    for (int c = 0; c < 3; ++c) fr[9 + c] = c0[c] - (1.25 * s3 / alpha) * e3[c];
    fr[13] = acc >= 0.0 ? 1.0 : -1.0;
    double L = 0.0;
    for (int i = 0; i < 3; ++i)
      for (int j = i + 1; j < 3; ++j) {
        double d = 0.0;
        for (int c = 0; c < 3; ++c) d += (rv[3 * i + c] - rv[3 * j + c]) * (rv[3 * i + c] - rv[3 * j + c]);
        L = fmax(L, sqrt(d));
      }
    fr[14] = L;
    fr[15] = 0.0;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 16; i += blockDim.x) P.frame[(size_t)k * 16 + i] = fr[i];
  // boundary positions: edges (0,1)->(0,0), (0,0)->(1,0), (1,0)->(0,1)
  for (int ib = threadIdx.x; ib < nb; ib += blockDim.x) {
    const int e = ib / nq, i = ib % nq;
    double x[3];
    if (ichart == 1) {
      for (int c = 0; c < 3; ++c) x[c] = sxbd_chart[(size_t)k * 9 * nq + 3 * ib + c];
    } else {
      const double EA[3][2] = {{0, 1}, {0, 0}, {1, 0}}, EB[3][2] = {{0, 0}, {1, 0}, {0, 1}};
      const double s01 = 0.5 * (T.tgl[i] + 1.0);
      const double u = EA[e][0] + (EB[e][0] - EA[e][0]) * s01, v = EA[e][1] + (EB[e][1] - EA[e][1]) * s01;
      geom_eval(scx, T.ktab, h, p - 1, u, v, x, nullptr, nullptr);
    }
    to_frame(fr, x, bx + 6 * ib);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 9 * nq; i += blockDim.x) {
    const int e = i / (3 * nq), c = (i / nq) % 3, kk = i % nq;
    double s = 0.0;
    for (int q = 0; q < nq; ++q) s += T.Legmat[kk + (size_t)nq * q] * bx[6 * (e * nq + q) + c];
    ecf[i] = s;
  }
  __syncthreads();
  // the edges in the power basis for the per-pair kernels (Horner's rule costs
  // about half the Legendre recurrence per point): coefficient j of edge
  // component ec is sum_k ecf_k [s^j] P_k, over k = j, j+2, ...
  for (int i = threadIdx.x; i < 9 * nq; i += blockDim.x) {
    const int ec = i / nq, j = i % nq;
    double m = 0.0;
    for (int q = j; q < nq; q += 2) m += ecf[ec * nq + q] * T.leg2mon[(size_t)q * nq + j];
    P.edge[(size_t)k * 9 * nq + i] = m;
  }
  for (int ib = threadIdx.x; ib < nb; ib += blockDim.x) {
    const int e = ib / nq, i = ib % nq;
    for (int c = 0; c < 3; ++c) {
      double v, d;
      leg_eval_r(ecf + (e * 3 + c) * nq, nq, T.tgl[i], v, d);
      bx[6 * ib + 3 + c] = d;
    }
    for (int c = 0; c < 6; ++c) P.bX[((size_t)k * nb + ib) * 6 + c] = bx[6 * ib + c];
  }
  __syncthreads();
}

// Harmonics at a panel's boundary nodes (and their combinations with the edge
// tangent), and the quaternion matrix, Msl^T and Fn at its nodes, from the frame and
// boundary nodes written by rrq_panel_frame_kernel.
//
// One thread per node, panel nodes first, then (from the next wave on where that
// separates them) the boundary nodes: each keeps the previous degree's harmonics in
// registers.  Bound by its stores (1.24 GB for the 14,250 order-8 panels of the 48 x
// 120 workload): 0.31 ms; with the harmonics' degrees handed on through LDS, one
// thread a node and then one a matrix entry, it took 0.60 (0.48 before it also
// wrote the tangent combinations), without the gathering below 0.54.  1,580 panels
// of order 12: 0.60 -> 0.25.
template <int P>
struct SystemPlan {
  static constexpr int H = P * (P + 1) / 2, NB = 3 * (P + 2);
  static constexpr int B0 = H + NB <= 64 ? H : (H > 64 ? H : 64);  // first thread of the boundary nodes
  static constexpr int N = (B0 + NB + 63) / 64 * 64;
  // up to order 8 a panel's Fq and Msl^T (41 KB) are gathered in LDS and written in
  // order; rows of an odd number of doubles, so the nodes' lanes fall in different banks
  static constexpr bool GATHER = P <= 8;
  static constexpr int RF = 3 * H + 1 - (3 * H) % 2, RM = H + 1 - H % 2;
};

template <int P>
__global__ void __launch_bounds__(SystemPlan<P>::N) rrq_panel_system_kernel(RRQPanels pan, const double* __restrict__ sx,
                                                                            const double* __restrict__ snx) {
  using S = SystemPlan<P>;
  constexpr int H = S::H, NB = S::NB, NC1 = P * (P + 1) / 2, NCB = NC1 + (P - 1) * (P + 2) / 2;
  __shared__ double gq[S::GATHER ? H * S::RF : 1], gm[S::GATHER ? H * S::RM : 1];
  const int k = blockIdx.x, i = threadIdx.x;
  const bool node = i < H, bnd = i >= S::B0 && i < S::B0 + NB;
  const double* fr = pan.frame + (size_t)k * 16;
  double X[3] = {0.0, 0.0, 0.0}, N[3] = {0.0, 0.0, 0.0};  // position; normal at a panel node, tangent at a boundary node
  if (node) {
    const size_t g = (size_t)k * H + i;
    const double x[3] = {sx[3 * g], sx[3 * g + 1], sx[3 * g + 2]};
    const double n0[3] = {snx[3 * g], snx[3 * g + 1], snx[3 * g + 2]};
    to_frame(fr, x, X);
    rotate(fr, n0, N);
  } else if (bnd) {
    const double* bx = pan.bX + ((size_t)k * NB + i - S::B0) * 6;
    for (int c = 0; c < 3; ++c) {
      X[c] = bx[c];
      N[c] = bx[3 + c];
    }
  }
  // Fq(i,k) = grad F_k(y_i) as a pure quaternion, F_k = Im((-i)^m H'_n^m), n = 1..p,
  // m = 1..n; the real 4h x 4h matrix of the reference (Mmatrix with its first two
  // diagonal blocks zeroed, rrq_r64:851-858) is left multiplication by this h x h
  // quaternion matrix
  double *FQ0 = pan.Fq + (size_t)k * 3 * H * H, *MS0 = pan.Msl + (size_t)k * H * H;
  double* FQ = S::GATHER ? gq + i * S::RF : FQ0 + (size_t)i * 3 * H;
  double* MS = S::GATHER ? gm + i * S::RM : MS0 + (size_t)i * H;
  double* FN = pan.Fn + (size_t)k * H * H + i;
  cd* Ho = (cd*)pan.basis + ((size_t)k * NB + (i - S::B0)) * NCB;
  cd* To = Ho + NC1;
  const cd W = cmk(X[1], X[2]), dw = cmk(N[1], N[2]);
  cd E[P + 2];  // H'_{n-1}^m, zero past m = n - 1
#pragma unroll
  for (int m = 0; m < P + 2; ++m) E[m] = cmk(0.0, 0.0);
  E[0] = cmk(1.0, 0.0);
  int kk = 0, ih = 0, jt = 0;
#pragma unroll 1
  for (int n = 1; n <= P; ++n) {
    if (bnd) {
      // degree n - 1: H' and, below degree p - 1, T_n^m = dX_Z H'_n^m + i/2 (dW
      // H'_n^{m-1} + conj(dW) H'_n^{m+1})
      cd lo = cmk(-E[1].re, E[1].im);
#pragma unroll
      for (int m = 0; m <= P; ++m) {
        if (m < n) Ho[ih++] = E[m];
        if (m <= n && n < P)
          To[jt++] = cadd(cscale(E[m], N[0]), cscale(cmuli(cadd(cmul(dw, lo), cmul(cconj(dw), E[m + 1]))), 0.5));
        lo = E[m];
      }
    }
    const double dn = (double)n;
    cd lo = cmk(-E[1].re, E[1].im);
#pragma unroll
    for (int m = 0; m <= P; ++m) {
      if (m <= n) {
        const cd mid = E[m], hi = E[m + 1];
        const cd b = cadd(cmul(W, lo), cmul(cconj(W), hi));
        E[m] = cadd(cscale(mid, X[0]), cscale(cmuli(b), 0.5));
        if (node && m > 0) {
          // the gradient, from degree n - 1
          const double F1 = imrot(m, cscale(mid, dn)), F2 = imrot(m, cscale(cmuli(cadd(lo, hi)), 0.5 * dn)),
                       F3 = imrot(m, cscale(csub(hi, lo), 0.5 * dn));
          FN[(size_t)H * kk] = imrot(m, E[m]);
          MS[kk] = N[0] * F1 + N[1] * F2 + N[2] * F3;
          FQ[3 * kk] = F1;
          FQ[3 * kk + 1] = F2;
          FQ[3 * kk + 2] = F3;
          ++kk;
        }
        lo = mid;
      }
    }
  }
  if (S::GATHER) {
    __syncthreads();
    for (int e = i; e < 3 * H * H; e += S::N) FQ0[e] = gq[e / (3 * H) * S::RF + e % (3 * H)];
    for (int e = i; e < H * H; e += S::N) MS0[e] = gm[e / H * S::RM + e % H];
  }
}

void launch_rrq_system(int p, RRQPanels P, int npan, const double* sx, const double* snx, hipStream_t s) {
  switch (p) {
#define QOL_SYSTEM(P_)                                                                                                 \
  case P_:                                                                                                             \
    hipLaunchKernelGGL(rrq_panel_system_kernel<P_>, dim3(npan), dim3(SystemPlan<P_>::N), 0, s, P, sx, snx);            \
    break;
    QOL_SYSTEM(2) QOL_SYSTEM(3) QOL_SYSTEM(4) QOL_SYSTEM(5) QOL_SYSTEM(6) QOL_SYSTEM(7) QOL_SYSTEM(8) QOL_SYSTEM(9)
    QOL_SYSTEM(10) QOL_SYSTEM(11) QOL_SYSTEM(12)
#undef QOL_SYSTEM
    default: throw std::runtime_error("RRQ set-up: patch orders 2..12 only");
  }
}

// ---------------------------------------------------------------------------
// Weights operator of one panel by two Gauss-Jordan eliminations run in one loop:
//   [Fq | I] -> [I | X],  X = Fq^{-1}   (h x h pure-quaternion matrix, elements
//                                        combined by left multiplication), and
//   [Msl^T | I] -> [I | B]              (real).
// The matrices live in registers on a 16 x 16 thread grid, thread (ty, tx)
// holding rows ty+16a and columns tx+16b.  Partial pivoting without moving rows:
// step k picks the unused row with the largest |element| in column k (lowest
// index on ties), eliminates column k from every other row and normalises the
// pivot row, so row piv[k] ends as row k of the inverse.  Two barriers per step;
// LDS buffers alternate between steps.
//
// A pair's weights then are Ad = v / 4pi with v_j = sum_{k,q} (X_kj)_q rhs_qk, the
// solution of M^T w = rhs (first h components), and As = B (W + Fn^T v) / (4pi alpha)
// (rrq_weights_kernel).  Every solve kernel leaves the four components of X in P.X,
// (X_kj)_q at (q h + k) h + j, and B in P.Binv, transposed: B(j, r) at r h + j.
__device__ __forceinline__ void qmul_fma(const double* a, const double* b, double* c) {
  c[0] = fma(a[0], b[0], fma(-a[1], b[1], fma(-a[2], b[2], -a[3] * b[3])));
  c[1] = fma(a[0], b[1], fma(a[1], b[0], fma(a[2], b[3], -a[3] * b[2])));
  c[2] = fma(a[0], b[2], fma(-a[1], b[3], fma(a[2], b[0], a[3] * b[1])));
  c[3] = fma(a[0], b[3], fma(a[1], b[2], fma(-a[2], b[1], a[3] * b[0])));
}
// e -= a * b (quaternions)
__device__ __forceinline__ void qsub_mul(double* e, const double* a, const double* b) {
  e[0] = fma(-a[0], b[0], fma(a[1], b[1], fma(a[2], b[2], fma(a[3], b[3], e[0]))));
  e[1] = fma(-a[0], b[1], fma(-a[1], b[0], fma(-a[2], b[3], fma(a[3], b[2], e[1]))));
  e[2] = fma(-a[0], b[2], fma(a[1], b[3], fma(-a[2], b[0], fma(-a[3], b[1], e[2]))));
  e[3] = fma(-a[0], b[3], fma(-a[1], b[2], fma(a[2], b[1], fma(-a[3], b[0], e[3]))));
}

// lowest row not yet pivoted (bit clear in u[0..1]); the fallback pivot when
// NaN entries leave the search without a candidate
__device__ __forceinline__ int first_unused(const unsigned long long* u) {
  return u[0] != ~0ull ? __builtin_ctzll(~u[0]) : 64 + __builtin_ctzll(~u[1]);
}

template <int RPT, int CPT>
__global__ void __launch_bounds__(256) rrq_panel_solve_kernel(RRQTables T, RRQPanels P, int npan,
                                                              const int* __restrict__ nrrq) {
  const int k = blockIdx.x;
  if (nrrq && nrrq[k] == 0) return;  // null: every panel
  const int h = T.h, m = 2 * h;
  constexpr int NR = 16 * RPT, NC = 16 * CPT;
  __shared__ double colq[2][4 * NR], colr[2][NR], prq[2][4 * NC], prr[2][NC];
  __shared__ double cvq[2][4], cvr[2][4];
  __shared__ int ciq[2][4], cir[2][4];
  __shared__ int pivq[NR], pivr[NR];
  double *X = P.X + (size_t)k * 4 * h * h, *Bk = P.Binv + (size_t)k * h * h;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const double* FQ = P.Fq + (size_t)k * 3 * h * h;
  const double* MS = P.Msl + (size_t)k * h * h;
  double Aq[RPT][CPT][4], Ar[RPT][CPT];
#pragma unroll
  for (int a = 0; a < RPT; ++a)
#pragma unroll
    for (int b = 0; b < CPT; ++b) {
      const int r = ty + 16 * a, c = tx + 16 * b;
      double* e = Aq[a][b];
      e[0] = e[1] = e[2] = e[3] = 0.0;
      Ar[a][b] = 0.0;
      if (r < h && c < h) {
        const double* q = FQ + 3 * ((size_t)r * h + c);
        e[1] = q[0]; e[2] = q[1]; e[3] = q[2];
        Ar[a][b] = MS[r + (size_t)h * c];
      }
    }
  // rows already used as pivots (same in every thread)
  unsigned long long uq[2] = {0ull, 0ull}, ur[2] = {0ull, 0ull};
  const int wv = threadIdx.x >> 6;
  for (int kk = 0; kk < h; ++kk) {
    const int buf = kk & 1, kt = kk & 15, kb = kk >> 4;
    // column kk: its owners (tx == kt, four per wave) publish the multipliers and
    // their best unused row; the wave reduces the four candidates by shuffles
    double bq = -1.0, br = -1.0;
    int iq = NR, ir = NR;
    const bool own = tx == kt;
#pragma unroll
    for (int b = 0; b < CPT; ++b) {
      if (b != kb) continue;  // uniform
#pragma unroll
      for (int a = 0; a < RPT; ++a) {
        const int r = ty + 16 * a;
        if (own & (r < h)) {
          const double* e = Aq[a][b];
          for (int q = 0; q < 4; ++q) colq[buf][4 * r + q] = e[q];
          colr[buf][r] = Ar[a][b];
        }
        const bool ok = own & (r < h);
        const bool fq = (uq[r >> 6] >> (r & 63)) & 1ull, fr = (ur[r >> 6] >> (r & 63)) & 1ull;
        const double* e = Aq[a][b];
        const double vq = e[0] * e[0] + e[1] * e[1] + e[2] * e[2] + e[3] * e[3], vr = fabs(Ar[a][b]);
        const bool tq = ok & !fq & (vq > bq), tr = ok & !fr & (vr > br);
        bq = tq ? vq : bq; iq = tq ? r : iq;
        br = tr ? vr : br; ir = tr ? r : ir;
      }
    }
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
      const double oq = __shfl_xor(bq, off, 64), orr = __shfl_xor(br, off, 64);
      const int oiq = __shfl_xor(iq, off, 64), oir = __shfl_xor(ir, off, 64);
      const bool tq = (oq > bq) | ((oq == bq) & (oiq < iq)), tr = (orr > br) | ((orr == br) & (oir < ir));
      bq = tq ? oq : bq; iq = tq ? oiq : iq;
      br = tr ? orr : br; ir = tr ? oir : ir;
    }
    if ((threadIdx.x & 63) == kt) {
      cvq[buf][wv] = bq; ciq[buf][wv] = iq;
      cvr[buf][wv] = br; cir[buf][wv] = ir;
    }
    __syncthreads();
    int pq = NR, pr = NR;
    {
      double vbq = -1.0, vbr = -1.0;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const double vq = cvq[buf][t], vr = cvr[buf][t];
        const int i1 = ciq[buf][t], i2 = cir[buf][t];
        const bool tq = (vq > vbq) | ((vq == vbq) & (i1 < pq)), tr = (vr > vbr) | ((vr == vbr) & (i2 < pr));
        vbq = tq ? vq : vbq; pq = tq ? i1 : pq;
        vbr = tr ? vr : vbr; pr = tr ? i2 : pr;
      }
    }
    // identical in every lane: keep them in scalar registers
    pq = __builtin_amdgcn_readfirstlane(pq);
    pr = __builtin_amdgcn_readfirstlane(pr);
    if (pq >= h) pq = first_unused(uq);
    if (pr >= h) pr = first_unused(ur);
    uq[pq >> 6] |= 1ull << (pq & 63);
    ur[pr >> 6] |= 1ull << (pr & 63);
    if (threadIdx.x == 0) { pivq[kk] = pq; pivr[kk] = pr; }
    // pivot rows to LDS (row pq lives in slot a = pq/16 of the threads with ty =
    // pq%16); all 16*CPT columns are written (the buffers have room for them)
    // The right block is kept in pivot order: its column h+kk is the identity
    // column of the row pivoted at step kk, materialised now (1 in the pivot row,
    // 0 elsewhere, which is what every other row still holds there).
#pragma unroll
    for (int a = 0; a < RPT; ++a) {
      if (a == (pq >> 4) && ty == (pq & 15)) {
#pragma unroll
        for (int b = 0; b < CPT; ++b) {
          const bool unit = tx + 16 * b == h + kk;
#pragma unroll
          for (int q = 0; q < 4; ++q) prq[buf][4 * (tx + 16 * b) + q] = unit ? (q == 0 ? 1.0 : 0.0) : Aq[a][b][q];
        }
      }
      if (a == (pr >> 4) && ty == (pr & 15)) {
#pragma unroll
        for (int b = 0; b < CPT; ++b) prr[buf][tx + 16 * b] = tx + 16 * b == h + kk ? 1.0 : Ar[a][b];
      }
    }
    __syncthreads();
    // inverse of the pivots
    double iq4[4];
    {
      const double* e = prq[buf] + 4 * kk;
      const double n2 = e[0] * e[0] + e[1] * e[1] + e[2] * e[2] + e[3] * e[3];
      const double in2 = 1.0 / n2;
      iq4[0] = e[0] * in2; iq4[1] = -e[1] * in2; iq4[2] = -e[2] * in2; iq4[3] = -e[3] * in2;
    }
    const double irr = 1.0 / prr[buf][kk];
    // every row: A_r -= A_rk * (pivot^-1 * pivot row); the pivot row itself is
    // overwritten below.  Live columns are the window (kk, h+kk]: finished left
    // columns and right columns of rows not yet pivoted (still unit columns,
    // untouched by this step) get a zero normalised row, which leaves them
    // unchanged; chunks of 16 columns outside the window are skipped outright.
#pragma unroll
    for (int b = 0; b < CPT; ++b) {
      if (16 * b + 15 <= kk || 16 * b > h + kk) continue;  // uniform
      const int c = tx + 16 * b;
      const bool colok = (c > kk) & (c <= h + kk) & (c < m);
      const int cc = c < m ? c : m - 1;
      double nq[4];
      qmul_fma(iq4, prq[buf] + 4 * cc, nq);
#pragma unroll
      for (int q = 0; q < 4; ++q) nq[q] = colok ? nq[q] : 0.0;
      const double nr = colok ? irr * prr[buf][cc] : 0.0;
#pragma unroll
      for (int a = 0; a < RPT; ++a) {
        const int r = ty + 16 * a;
        const int rc = r < h ? r : h - 1;
        qsub_mul(Aq[a][b], colq[buf] + 4 * rc, nq);
        Ar[a][b] = fma(-colr[buf][rc], nr, Ar[a][b]);
      }
    }
#pragma unroll
    for (int a = 0; a < RPT; ++a) {
      if (a == (pq >> 4) && ty == (pq & 15)) {
#pragma unroll
        for (int b = 0; b < CPT; ++b) {
          const int c = tx + 16 * b, cc = c < m ? c : m - 1;
          double nq[4];
          qmul_fma(iq4, prq[buf] + 4 * cc, nq);
          // columns right of the window stay zero (unit columns of later pivots)
          const bool keep = c <= h + kk;
#pragma unroll
          for (int q = 0; q < 4; ++q) Aq[a][b][q] = keep ? nq[q] : 0.0;
        }
      }
      if (a == (pr >> 4) && ty == (pr & 15)) {
#pragma unroll
        for (int b = 0; b < CPT; ++b) {
          const int c = tx + 16 * b, cc = c < m ? c : m - 1;
          Ar[a][b] = c <= h + kk ? irr * prr[buf][cc] : 0.0;
        }
      }
    }
  }
  __syncthreads();
  // row piv[kk] holds row kk of the inverse: scatter by the inverse permutation
  __shared__ int posq[NR], posr[NR];
  for (int kk = threadIdx.x; kk < h; kk += blockDim.x) { posq[pivq[kk]] = kk; posr[pivr[kk]] = kk; }
  __syncthreads();
#pragma unroll
  for (int a = 0; a < RPT; ++a)
#pragma unroll
    for (int b = 0; b < CPT; ++b) {
      const int r = ty + 16 * a, c = tx + 16 * b;
      if (r < h && c >= h && c < m) {
        // row piv[k] holds row k of the inverse, column h+j' holds its column piv[j']
        const int jq = pivq[c - h], jr = pivr[c - h];
        const int kq = posq[r], kr = posr[r];
        for (int q = 0; q < 4; ++q) X[(size_t)(q * h + kq) * h + jq] = Aq[a][b][q];
        Bk[(size_t)jr * h + kr] = Ar[a][b];
      }
    }
}

// Entry (a, b) of the left-multiplication matrix of quaternion q (q*x = L(q) x):
// L[a][b] = +/- q[a ^ b], negative at (0,1) (0,2) (0,3) (1,2) (2,3) (3,1).
__device__ __forceinline__ double lmat(const double* q, int a, int b) {
  const unsigned neg = 0x0Eu | (0x4u << 4) | (0x8u << 8) | (0x2u << 12);
  const double v = q[a ^ b];
  return ((neg >> (a * 4 + b)) & 1u) ? -v : v;
}

__device__ __forceinline__ double qd4_get(const qd4& d, int i) {
  return i == 0 ? d[0] : (i == 1 ? d[1] : (i == 2 ? d[2] : d[3]));
}

// The same weights operator with the quaternion elimination on the FP64 matrix
// cores.  In real form the quaternion rank-1 update A_rc -= m_r n_c is
// A(4h x 2h) -= L(m)(4h x 4) N(4 x 2h): one v_mfma_f64_16x16x4 per 16x16 tile.
// A is held as accumulator tiles (row 4r + component, column c): wave w owns the
// row tiles w, w+4, ...; lane l holds rows 4i + l/16 (i = 0..3, i.e. quaternion
// 4*tile + i, component l/16) of column l%16.  The real Msl^T elimination stays
// on the 16 x 16 thread grid as in rrq_panel_solve_kernel; both share the step
// loop (implicit partial pivoting, pivot-ordered right block, column window).
template <int RT, int CT>
__global__ void __launch_bounds__(256) rrq_panel_solve_mfma_kernel(RRQTables T, RRQPanels P, int npan,
                                                                   const int* __restrict__ nrrq) {
  const int k = blockIdx.x;
  if (nrrq && nrrq[k] == 0) return;  // null: every panel
  const int h = T.h, m = 2 * h;
  constexpr int RTW = (RT + 3) / 4, NQR = 4 * RT, NC = 16 * CT;
  __shared__ double colq[2][4 * NQR], prq[2][4 * NC];
  __shared__ double cvq[2][4];
  __shared__ int ciq[2][4];
  __shared__ int pivq[NQR], posq[NQR];
  double* X = P.X + (size_t)k * 4 * h * h;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const double* FQ = P.Fq + (size_t)k * 3 * h * h;
  qd4 D[RTW][CT];
#pragma unroll
  for (int t = 0; t < RTW; ++t)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rt = wv + 4 * t, r = 4 * rt + i, c = 16 * ct + li;
        D[t][ct][i] = (rt < RT && r < h && c < h && lk > 0) ? FQ[3 * ((size_t)r * h + c) + lk - 1] : 0.0;
      }
  unsigned long long uq[2] = {0ull, 0ull};
  for (int kk = 0; kk < h; ++kk) {
    const int buf = kk & 1, kt = kk & 15, kb = kk >> 4;
    // ---- column kk: multipliers and pivot candidates
    {
      double bq = -1.0;
      int iq = NQR;
#pragma unroll
      for (int t = 0; t < RTW; ++t) {
        const int rt = wv + 4 * t;
        if (rt >= RT) continue;  // uniform
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          if (ct != kb) continue;  // uniform
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const double v = D[t][ct][i];
            double s2 = v * v;
            s2 += __shfl_xor(s2, 16, 64);
            s2 += __shfl_xor(s2, 32, 64);
            const int r = 4 * rt + i;
            const bool here = (li == kt) & (r < h);
            if (here) colq[buf][4 * r + lk] = v;
            const bool used = (uq[r >> 6] >> (r & 63)) & 1ull;
            const bool tq = here & !used & (s2 > bq);
            bq = tq ? s2 : bq;
            iq = tq ? r : iq;
          }
        }
      }
      if (lane == kt) { cvq[buf][wv] = bq; ciq[buf][wv] = iq; }
    }
    __syncthreads();
    int pq = NQR;
    {
      double vbq = -1.0;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const double vq = cvq[buf][t];
        const int i1 = ciq[buf][t];
        const bool tq = (vq > vbq) | ((vq == vbq) & (i1 < pq));
        vbq = tq ? vq : vbq; pq = tq ? i1 : pq;
      }
    }
    pq = __builtin_amdgcn_readfirstlane(pq);
    if (pq >= h) pq = first_unused(uq);
    uq[pq >> 6] |= 1ull << (pq & 63);
    if (threadIdx.x == 0) pivq[kk] = pq;
    const int rtp = pq >> 2, ip = pq & 3, wp = rtp & 3, tp = rtp >> 2;
    // pivot row to LDS; the right block is in pivot order, its column h+kk is the
    // unit column of the row pivoted now (materialised here)
    if (wv == wp) {
#pragma unroll
      for (int t = 0; t < RTW; ++t) {
        if (t != tp) continue;  // uniform
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const int c = 16 * ct + li;
          const double v = qd4_get(D[t][ct], ip);
          prq[buf][4 * c + lk] = c == h + kk ? (lk == 0 ? 1.0 : 0.0) : v;
        }
      }
    }
    __syncthreads();
    // ---- update
    double iq4[4];
    {
      const double* e = prq[buf] + 4 * kk;
      const double n2 = e[0] * e[0] + e[1] * e[1] + e[2] * e[2] + e[3] * e[3];
      const double in2 = 1.0 / n2;
      iq4[0] = e[0] * in2; iq4[1] = -e[1] * in2; iq4[2] = -e[2] * in2; iq4[3] = -e[3] * in2;
    }
    // B operand: component lk of the normalised pivot row at column 16ct + li
    // (zero outside the live window (kk, h+kk])
    double Bop[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int c = 16 * ct + li;
      const int cc = c < m ? c : m - 1;
      const double* x = prq[buf] + 4 * cc;
      double v = 0.0;
#pragma unroll
      for (int j = 0; j < 4; ++j) v = fma(lmat(iq4, lk, j), x[j], v);
      const bool colok = (c > kk) & (c <= h + kk) & (c < m);
      Bop[ct] = colok ? v : 0.0;
    }
    // A operand: -L(m_r)[comp][lk] for row 4r + comp = 16 rt + li; the pivot row
    // gets zero (it is overwritten below)
#pragma unroll
    for (int t = 0; t < RTW; ++t) {
      const int rt = wv + 4 * t;
      if (rt >= RT) continue;  // uniform
      const int r = 4 * rt + (li >> 2), comp = li & 3;
      const double mv = lmat(colq[buf] + 4 * r, comp, lk);
      const double aop = ((r < h) & (r != pq)) ? -mv : 0.0;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        if (16 * ct + 15 <= kk || 16 * ct > h + kk) continue;  // uniform: tile outside the window
        D[t][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(aop, Bop[ct], D[t][ct], 0, 0, 0);
      }
    }
    if (wv == wp) {
#pragma unroll
      for (int t = 0; t < RTW; ++t) {
        if (t != tp) continue;  // uniform
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int i = 0; i < 4; ++i) D[t][ct][i] = i == ip ? Bop[ct] : D[t][ct][i];
      }
    }
  }
  __syncthreads();
  for (int kk = threadIdx.x; kk < h; kk += blockDim.x) posq[pivq[kk]] = kk;
  __syncthreads();
  // row piv[k] holds row k of the inverse; column h+j' holds its column piv[j']
#pragma unroll
  for (int t = 0; t < RTW; ++t) {
    const int rt = wv + 4 * t;
    if (rt >= RT) continue;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 4 * rt + i, c = 16 * ct + li;
        if (r < h && c >= h && c < m) X[(size_t)(lk * h + posq[r]) * h + pivq[c - h]] = D[t][ct][i];
      }
  }
}

// B = (Msl^T)^{-1} (transposed, B(r,c) at c*h + r) by the same windowed
// Gauss-Jordan on the 16 x 16 thread grid; small enough to run many panels per CU.
template <int RPT, int CPT>
__global__ void __launch_bounds__(256) rrq_msl_inverse_kernel(RRQTables T, RRQPanels P, int npan,
                                                              const int* __restrict__ nrrq) {
  const int k = blockIdx.x;
  if (nrrq && nrrq[k] == 0) return;  // null: every panel
  const int h = T.h, m = 2 * h;
  constexpr int NR = 16 * RPT, NC = 16 * CPT;
  __shared__ double colr[2][NR], prr[2][NC], cvr[2][4];
  __shared__ int cir[2][4], pivr[NR], posr[NR];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const double* MS = P.Msl + (size_t)k * h * h;
  double Ar[RPT][CPT];
#pragma unroll
  for (int a = 0; a < RPT; ++a)
#pragma unroll
    for (int b = 0; b < CPT; ++b) {
      const int r = ty + 16 * a, c = tx + 16 * b;
      Ar[a][b] = (r < h && c < h) ? MS[r + (size_t)h * c] : 0.0;
    }
  unsigned long long ur[2] = {0ull, 0ull};
  for (int kk = 0; kk < h; ++kk) {
    const int buf = kk & 1, kt = kk & 15, kb = kk >> 4;
    double br = -1.0;
    int ir = NR;
    const bool own = tx == kt;
#pragma unroll
    for (int b = 0; b < CPT; ++b) {
      if (b != kb) continue;  // uniform
#pragma unroll
      for (int a = 0; a < RPT; ++a) {
        const int r = ty + 16 * a;
        if (own & (r < h)) colr[buf][r] = Ar[a][b];
        const bool fr = (ur[r >> 6] >> (r & 63)) & 1ull;
        const double vr = fabs(Ar[a][b]);
        const bool tr = own & (r < h) & !fr & (vr > br);
        br = tr ? vr : br;
        ir = tr ? r : ir;
      }
    }
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
      const double orr = __shfl_xor(br, off, 64);
      const int oir = __shfl_xor(ir, off, 64);
      const bool tr = (orr > br) | ((orr == br) & (oir < ir));
      br = tr ? orr : br;
      ir = tr ? oir : ir;
    }
    if (lane == kt) { cvr[buf][wv] = br; cir[buf][wv] = ir; }
    __syncthreads();
    int pr = NR;
    {
      double vbr = -1.0;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const double vr = cvr[buf][t];
        const int i2 = cir[buf][t];
        const bool tr = (vr > vbr) | ((vr == vbr) & (i2 < pr));
        vbr = tr ? vr : vbr; pr = tr ? i2 : pr;
      }
    }
    pr = __builtin_amdgcn_readfirstlane(pr);
    if (pr >= h) pr = first_unused(ur);
    ur[pr >> 6] |= 1ull << (pr & 63);
    if (threadIdx.x == 0) pivr[kk] = pr;
#pragma unroll
    for (int a = 0; a < RPT; ++a)
      if (a == (pr >> 4) && ty == (pr & 15)) {
#pragma unroll
        for (int b = 0; b < CPT; ++b) prr[buf][tx + 16 * b] = tx + 16 * b == h + kk ? 1.0 : Ar[a][b];
      }
    __syncthreads();
    const double irr = 1.0 / prr[buf][kk];
#pragma unroll
    for (int b = 0; b < CPT; ++b) {
      if (16 * b + 15 <= kk || 16 * b > h + kk) continue;  // uniform
      const int c = tx + 16 * b;
      const bool colok = (c > kk) & (c <= h + kk) & (c < m);
      const int cc = c < m ? c : m - 1;
      const double nr = colok ? irr * prr[buf][cc] : 0.0;
#pragma unroll
      for (int a = 0; a < RPT; ++a) {
        const int r = ty + 16 * a;
        const int rc = r < h ? r : h - 1;
        Ar[a][b] = fma(-colr[buf][rc], nr, Ar[a][b]);
      }
    }
#pragma unroll
    for (int a = 0; a < RPT; ++a)
      if (a == (pr >> 4) && ty == (pr & 15)) {
#pragma unroll
        for (int b = 0; b < CPT; ++b) {
          const int c = tx + 16 * b, cc = c < m ? c : m - 1;
          Ar[a][b] = c <= h + kk ? irr * prr[buf][cc] : 0.0;
        }
      }
  }
  __syncthreads();
  for (int kk = threadIdx.x; kk < h; kk += blockDim.x) posr[pivr[kk]] = kk;
  __syncthreads();
  double* Bk = P.Binv + (size_t)k * h * h;
#pragma unroll
  for (int a = 0; a < RPT; ++a)
#pragma unroll
    for (int b = 0; b < CPT; ++b) {
      const int r = ty + 16 * a, c = tx + 16 * b;
      if (r < h && c >= h && c < m) Bk[(size_t)pivr[c - h] * h + posr[r]] = Ar[a][b];
    }
}

// rows already pivoted by a register-resident Gauss-Jordan (h <= 128)
struct RowMask {
  unsigned long long lo = 0ull, hi = 0ull;
  __device__ __forceinline__ void add(int r) {
    if (r < 64) lo |= 1ull << r;
    else hi |= 1ull << (r & 63);
  }
  // lowest row not yet pivoted
  __device__ __forceinline__ int first_free() const { return ~lo ? __builtin_ctzll(~lo) : 64 + __builtin_ctzll(~hi); }
};

// largest of 64 lanes' values, in every lane
__device__ __forceinline__ unsigned wave_max(unsigned v) {
#define QOL_MAX_DPP(CTRL_, ROWS_) \
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL_, ROWS_, 0xf, false))
  QOL_MAX_DPP(0x111, 0xf);  // row_shr 1, 2, 4, 8: the last lane of each 16 holds theirs
  QOL_MAX_DPP(0x112, 0xf);
  QOL_MAX_DPP(0x114, 0xf);
  QOL_MAX_DPP(0x118, 0xf);
  QOL_MAX_DPP(0x142, 0xa);  // row_bcast 15, 31
  QOL_MAX_DPP(0x143, 0xc);
#undef QOL_MAX_DPP
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// The pivot: the unused row with the largest v, ties to the lower row; lane i holds
// rows i and, with TWO, i + 64 (v1).  Non-negative doubles compare like integers, so
// the high words' maximum decides, the low words' among the lanes it leaves.  No
// candidate is left only with NaN entries: then the lowest unused row, so that every
// row is pivoted once and every index stays in range.  second: the lane's row i + 64
// is the larger of its two.
template <bool TWO>
__device__ __forceinline__ int pivot_row(const RowMask& used, int h, int lane, double v0, double v1, bool& second) {
  const bool c0 = (lane < h) & !((used.lo >> lane) & 1ull) & (v0 >= 0.0);
  second = false;
  if constexpr (TWO) {
    const bool c1 = (lane + 64 < h) & !((used.hi >> lane) & 1ull) & (v1 >= 0.0);
    second = c1 & (!c0 | (v1 > v0));
  }
  const double v = second ? v1 : v0;
  const unsigned hi = c0 | second ? (unsigned)__double2hiint(v) + 1u : 0u;
  const unsigned m = wave_max(hi);
  if (m == 0u) return used.first_free();
  unsigned long long tied = __ballot(hi == m);
  if (tied & (tied - 1ull)) {  // uniform
    const unsigned lo = (unsigned)__double2loint(v);
    tied = __ballot((hi == m) & (lo == wave_max(hi == m ? lo : 0u)));
  }
  if constexpr (TWO) {
    const unsigned long long low = tied & __ballot(!second);
    return low ? __builtin_ctzll(low) : 64 + __builtin_ctzll(tied);
  }
  return __builtin_ctzll(tied);
}

// orders a wave's LDS stores before its later loads
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// X = Fq^{-1} for the h x h pure-quaternion matrix Fq by Gauss-Jordan, the
// matrix in registers of NW waves (one panel per workgroup).  Lane (ly, lx) of
// an RL x CL lane grid (RL*CL <= 64; lanes beyond it idle) owns rows ly + RL*a
// (a < RA) and column slots lx + CL*b for the wave's CB/NW slot groups b;
// RL*RA >= h and CL*CB >= h, the grid chosen per order to waste few registers.
// Slot s holds left column s until step s eliminates it and right column h+s
// afterwards (the unit column of the row pivoted at step s, zero in every other
// row until then), so h slots carry the live window (kk, h+kk] at every step.
// Pivoting is implicit (no row moves): the unused row with the largest |A_r,kk|
// wins, ties to the lower row.  Column kk lies in one wave: it publishes the column,
// reads it back a row per lane, finds the pivot and its inverse and puts -1 in the
// pivot row's place.  Each wave holds its part of the pivot row: it publishes that
// and clears it, so that the rank-1 update, the same in every lane, leaves
// 0 - (-1) (pivot^-1 row) there.  One workgroup barrier per step suffices (LDS
// double-buffered by step parity).
// Afterwards row piv[k] holds row k of X with slot s holding column piv[s].
//
// Bound by a step's chain (column, pivot, barrier, row, update) with two or three
// panels' waves a SIMD to hide it, and at order 8 a quarter by loads and scattered
// stores.  The pivot from shuffles among the column's own lanes, the inverse in every
// wave and a separate pass over the pivot row took 1.58 ms for 14,250 panels of order 8
// (206 VGPRs), this 0.95 (160); 1,600 of order 12: 1.90, now 1.27; the real inverses
// 0.33 and 0.54, now 0.17 and 0.29.
template <int RL, int RA, int CL, int CB, int NW>
__global__ void __launch_bounds__(64 * NW) rrq_quat_inverse_kernel(RRQTables T, RRQPanels P, int npan,
                                                                   const int* __restrict__ nrrq) {
  static_assert(RL * CL <= 64 && RL * RA <= 128 && CB % NW == 0, "lane grid");
  constexpr int CW = CB / NW;  // slot groups per wave
  const int k = blockIdx.x;
  if (nrrq && nrrq[k] == 0) return;  // null: every panel
  const int h = T.h;
  constexpr int NRW = RL * RA, NSL = CL * CB;
  __shared__ double colq[2][4 * NRW], rowq[2][4 * NSL], pinvs[2][4];
  __shared__ int pivs[2], piv[NRW], pos[NRW];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const bool act = lane < RL * CL;
  const int ly = lane / CL, lx = lane % CL;
  const double* FQ = P.Fq + (size_t)k * 3 * h * h;
  double A[RA][CW][4];
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < CW; ++b) {
      const int r = ly + RL * a, c = lx + CL * (wv * CW + b);
      double* e = A[a][b];
      e[0] = e[1] = e[2] = e[3] = 0.0;
      if (act & (r < h) & (c < h)) {
        const double* q = FQ + 3 * ((size_t)r * h + c);
        e[1] = q[0]; e[2] = q[1]; e[3] = q[2];
      }
    }
  const int lyr = act ? ly : -NRW - 1;  // lanes past the grid own no row
  RowMask used;
  for (int kk = 0; kk < h; ++kk) {
    const int buf = kk & 1, kt = kk % CL, kbg = kk / CL;
    const int ow = kbg / CW, kb = kbg % CW;  // wave and slot group holding column kk
    double* cq = colq[buf];
    double* rq = rowq[buf];
    if (wv == ow) {  // uniform
      // column kk by row, and slot kk turned into right column h+kk: zero, and 1 in
      // the pivot row, which goes straight into rq below
      if (act & (lx == kt)) {
#pragma unroll
        for (int b = 0; b < CW; ++b) {
          if (b != kb) continue;  // uniform
#pragma unroll
          for (int a = 0; a < RA; ++a)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              cq[4 * (ly + RL * a) + q] = A[a][b][q];
              A[a][b][q] = 0.0;
            }
        }
      }
      wave_lds_fence();
      double e[4], f[4], v1 = -1.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) e[q] = cq[4 * (lane < NRW ? lane : NRW - 1) + q];
      const double v0 = e[0] * e[0] + e[1] * e[1] + e[2] * e[2] + e[3] * e[3];
      if constexpr (NRW > 64) {
#pragma unroll
        for (int q = 0; q < 4; ++q) f[q] = cq[4 * (lane + 64 < NRW ? lane + 64 : NRW - 1) + q];
        v1 = f[0] * f[0] + f[1] * f[1] + f[2] * f[2] + f[3] * f[3];
      }
      bool second;
      const int p = pivot_row<(NRW > 64)>(used, h, lane, v0, v1, second);
      if constexpr (NRW > 64) {
#pragma unroll
        for (int q = 0; q < 4; ++q) e[q] = second ? f[q] : e[q];
      }
      const double in2 = 1.0 / (second ? v1 : v0);
      if (lane == (p & 63)) {
        double* c = cq + 4 * p;
        c[0] = -1.0;
        c[1] = c[2] = c[3] = 0.0;
        pinvs[buf][0] = e[0] * in2;
        pinvs[buf][1] = -e[1] * in2;
        pinvs[buf][2] = -e[2] * in2;
        pinvs[buf][3] = -e[3] * in2;
        pivs[buf] = p;
        piv[kk] = p;
      }
    }
    __syncthreads();
    const int p = pivs[buf];
    // this wave's part of the pivot row, by slot (wave-local exchange)
#pragma unroll
    for (int a = 0; a < RA; ++a)
      if (p - lyr == RL * a) {
#pragma unroll
        for (int b = 0; b < CW; ++b) {
          const int c = lx + CL * (wv * CW + b);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            rq[4 * c + q] = A[a][b][q];
            A[a][b][q] = 0.0;
          }
        }
      }
    if ((wv == ow) & (lane == 0)) rq[4 * kk] = 1.0;
    wave_lds_fence();
    double pinv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) pinv[q] = pinvs[buf][q];
    used.add(__builtin_amdgcn_readfirstlane(p));
    // every row: A_r -= A_r,kk * (pivot^-1 * pivot row); the normalised row entries of
    // this wave's slots first, then one column value per row
    double nq[CW][4];
#pragma unroll
    for (int b = 0; b < CW; ++b) qmul_fma(pinv, rq + 4 * (lx + CL * (wv * CW + b)), nq[b]);
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      const double* c = cq + 4 * (act ? ly + RL * a : 0);  // lanes past the grid idle
      const double cv[4] = {c[0], c[1], c[2], c[3]};
#pragma unroll
      for (int b = 0; b < CW; ++b) qsub_mul(A[a][b], cv, nq[b]);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < h; i += 64 * NW) pos[piv[i]] = i;
  __syncthreads();
  double* X = P.X + (size_t)k * 4 * h * h;
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < CW; ++b) {
      const int r = ly + RL * a, c = lx + CL * (wv * CW + b);
      if (act & (r < h) & (c < h)) {
        const int kx = pos[r], j = piv[c];
#pragma unroll
        for (int q = 0; q < 4; ++q) X[(size_t)(q * h + kx) * h + j] = A[a][b][q];
      }
    }
}

// B = (Msl^T)^{-1} by Gauss-Jordan in the registers of one wave per panel, the
// real counterpart of rrq_quat_inverse_kernel (same lane grid, slot reuse, implicit
// pivoting with ties to the lower row, -1 for the pivot row's column entry).
// The system matrix is A(r, c) = Msl[r + h*c]; output B transposed, B(kx, j) at
// Binv[j*h + kx].
template <int RL, int RA, int CL, int CB>
__global__ void __launch_bounds__(64) rrq_real_inverse_kernel(RRQTables T, RRQPanels P, int npan,
                                                              const int* __restrict__ nrrq) {
  static_assert(RL * CL <= 64 && RL * RA <= 128, "lane grid");
  const int k = blockIdx.x;
  if (nrrq && nrrq[k] == 0) return;  // null: every panel
  const int h = T.h;
  constexpr int NRW = RL * RA, NSL = CL * CB;
  __shared__ double colr[2][NRW], rowr[2][NSL], pivel[2];
  __shared__ int piv[NRW], pos[NRW];
  const int lane = threadIdx.x;
  const bool act = lane < RL * CL;
  const int ly = lane / CL, lx = lane % CL;
  const double* MS = P.Msl + (size_t)k * h * h;
  double A[RA][CB];
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int r = ly + RL * a, c = lx + CL * b;
      A[a][b] = (act & (r < h) & (c < h)) ? MS[r + (size_t)h * c] : 0.0;
    }
  const int lyr = act ? ly : -NRW - 1;  // lanes past the grid own no row
  RowMask used;
  for (int kk = 0; kk < h; ++kk) {
    const int buf = kk & 1, kt = kk % CL, kb = kk / CL;
    double* cr = colr[buf];
    double* rr = rowr[buf];
    if (act & (lx == kt)) {
#pragma unroll
      for (int b = 0; b < CB; ++b) {
        if (b != kb) continue;  // uniform
#pragma unroll
        for (int a = 0; a < RA; ++a) {
          cr[ly + RL * a] = A[a][b];
          A[a][b] = 0.0;
        }
      }
    }
    wave_lds_fence();
    const double e0 = cr[lane < NRW ? lane : NRW - 1];
    const double e1 = NRW > 64 ? cr[lane + 64 < NRW ? lane + 64 : NRW - 1] : 0.0;
    bool second;
    const int p = pivot_row<(NRW > 64)>(used, h, lane, fabs(e0), fabs(e1), second);
    used.add(p);
    if (lane == (p & 63)) {
      cr[p] = -1.0;
      pivel[buf] = 1.0 / (second ? e1 : e0);
      piv[kk] = p;
    }
#pragma unroll
    for (int a = 0; a < RA; ++a)
      if (p - lyr == RL * a) {
#pragma unroll
        for (int b = 0; b < CB; ++b) {
          rr[lx + CL * b] = A[a][b];
          A[a][b] = 0.0;
        }
      }
    if (lane == 0) rr[kk] = 1.0;
    wave_lds_fence();
    const double ip = pivel[buf];
    double nr[CB];
#pragma unroll
    for (int b = 0; b < CB; ++b) nr[b] = ip * rr[lx + CL * b];
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      const double c = cr[act ? ly + RL * a : 0];  // lanes past the grid idle
#pragma unroll
      for (int b = 0; b < CB; ++b) A[a][b] = fma(-c, nr[b], A[a][b]);
    }
  }
  __syncthreads();
  for (int i = lane; i < h; i += 64) pos[piv[i]] = i;
  __syncthreads();
  double* Bk = P.Binv + (size_t)k * h * h;
#pragma unroll
  for (int b = 0; b < CB; ++b)
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      const int r = ly + RL * a, c = lx + CL * b;
      if (act & (r < h) & (c < h)) Bk[(size_t)piv[c] * h + pos[r]] = A[a][b];
    }
}

// G of orders 11 and 12 (RRQPanels::G): G(j, q h + k) = sum_i C(j,i) (X_ki)_q / (4pi alpha)
// with C = B Fn^T.  One workgroup per panel, C in LDS; a wave forms 16 columns of G at a
// time from 16 rows of X, the order-12 panel's five tiles of 16 rows j as five independent
// chains over i that share every X value.
// Bound by memory (10h^2 doubles a panel in 165 us at order 12, 1,600 panels) and its latency:
// 0.31 ms there, where forming As, Ad and W blocks on the vector units took 0.70.
constexpr int kOpW = 8;  // waves
constexpr int kOpT = 5;  // tiles of 16 rows: 16 * 5 >= h

template <int P_>
__global__ void __launch_bounds__(64 * kOpW) rrq_operator_kernel(RRQPanels P, const int* __restrict__ nrrq) {
  const int k = blockIdx.x;
  if (nrrq && nrrq[k] == 0) return;
  constexpr int h = P_ * (P_ + 1) / 2, hp = 16 * kOpT + 4;
  static_assert(16 * kOpT >= h);
  __shared__ double Ct[h * hp];  // C(j, i) at i*hp + j, zero for j >= h
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const double *X = P.X + (size_t)k * 4 * h * h, *Fn = P.Fn + (size_t)k * h * h, *B = P.Binv + (size_t)k * h * h;
  double* G = P.G + (size_t)k * 4 * h * h;
  const double fac = 1.0 / (16.0 * atan(1.0)), fa = fac / P.frame[(size_t)k * 16 + 12];
  // D[4q + lk][li]: row i = i0 + 4q + lk, column j = j0 + li
  for (int tile = w; tile < kOpT * kOpT; tile += kOpW) {
    const int i0 = 16 * (tile / kOpT), j0 = 16 * (tile % kOpT);
    const int ic = min(i0 + li, h - 1), jc = min(j0 + li, h - 1);
    qd4 acc{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int r0 = 0; r0 < h; r0 += 4) {
      const int r = r0 + lk, rc = min(r, h - 1);
      const double f = r < h ? Fn[ic + (size_t)h * rc] : 0.0;
      const double b = j0 + li < h ? B[(size_t)rc * h + jc] : 0.0;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(f, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (i0 + 4 * q + lk < h) Ct[(i0 + 4 * q + lk) * hp + j0 + li] = acc[q];
  }
  __syncthreads();
  for (int c0 = 16 * w; c0 < 4 * h; c0 += 16 * kOpW) {
    const int cc = min(c0 + li, 4 * h - 1);
    qd4 acc[kOpT];
#pragma unroll
    for (int t = 0; t < kOpT; ++t) acc[t] = qd4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 5
    for (int i0 = 0; i0 < h; i0 += 4) {
      const int i = i0 + lk, ii = min(i, h - 1);
      const double x = i < h ? X[(size_t)cc * h + ii] : 0.0;
#pragma unroll
      for (int t = 0; t < kOpT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, Ct[ii * hp + 16 * t + li], acc[t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < kOpT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = c0 + 4 * q + lk, j = 16 * t + li;
        if ((c < 4 * h) & (j < h)) G[(size_t)c * h + j] = acc[t][q] * fa;
      }
  }
}

// Where the solve forms G for the weights rather than leave them X, Fn and B.  The
// two differ by how v's rounding passes through B Fn^T, which grows with the condition
// of X: against the weights by G the potentials of a 12 x 36 surface move by 1e-10
// (relative 2-norm, largest 7e-9) at order 10, 4e-10 (2e-8) at 11 and 2e-8 (1e-6) at
// 12, so that the two highest orders keep G, and with it the weights callers have had.
// Neither is the nearer one: by Green's identity the potentials at 6,000 targets of a 24 x
// 60 surface are off by 2.40e-10 (2-norm) with G and 2.42e-10 without at order 12, by
// 4.44e-10 with either at 11.  Up to order 10 the shorter product is the faster one.
bool rrq_forms_operator(int p) { return p >= 11; }

void launch_rrq_panel_solve(RRQTables T, RRQPanels P, int npan, const int* nrrq, hipStream_t s, int variant) {
  const int h = T.h;
  const int rpt = (h + 15) / 16, cpt = (2 * h + 15) / 16;
  // variant 2 (or QOL_SOLVE_MFMA=1) selects, for patch orders up to 8, the
  // matrix-core quaternion elimination (A as 4-wave accumulator tiles, B from a
  // separate real inverse), which is slower on the order-8 workload (4.2 ms for 14,250
  // panels, the fused kernel below 3.8, the register-resident inverses 1.1)
  const char* mf = std::getenv("QOL_SOLVE_MFMA");
  if (variant == 2 || (variant == 0 && mf && mf[0] == '1')) switch (T.p) {
#define QOL_SOLVE_MFMA(P_, RT_, CT_, RPT_)                                                                  \
  case P_:                                                                                                \
    hipLaunchKernelGGL((rrq_msl_inverse_kernel<RPT_, CT_>), dim3(npan), dim3(256), 0, s, T, P, npan, nrrq);  \
    hipLaunchKernelGGL((rrq_panel_solve_mfma_kernel<RT_, CT_>), dim3(npan), dim3(256), 0, s, T, P, npan,     \
                       nrrq);                                                                             \
    return;
    QOL_SOLVE_MFMA(2, 1, 1, 1)
    QOL_SOLVE_MFMA(3, 2, 1, 1)
    QOL_SOLVE_MFMA(4, 3, 2, 1)
    QOL_SOLVE_MFMA(5, 4, 2, 1)
    QOL_SOLVE_MFMA(6, 6, 3, 2)
    QOL_SOLVE_MFMA(7, 7, 4, 2)
    QOL_SOLVE_MFMA(8, 9, 5, 3)
    default: break;
  }
#undef QOL_SOLVE_MFMA
  // by default the real and the quaternion inverse with the matrix in registers;
  // variant 1 (or QOL_SOLVE_FUSED=1) selects the single fused kernel
  const char* fu = std::getenv("QOL_SOLVE_FUSED");
  const bool fused = variant == 1 || (variant == 0 && fu && fu[0] == '1');
  if (h <= 78 && !fused) {
    // lane grid per order (rows RL x RA, slots CL x CB) and waves.  Measured (us): order
    // 8, 14,250 panels, 2 waves 953 (4: 1078, 9 x 4 rows: 940-998); order 9 of 24 x 60, 3
    // waves 469 (2: 491, 6: 650); 10: 8 waves 862 (4: 943, 7: 884); 11: 4 waves of three
    // slot groups, so that two panels share a CU, 1440 (6: 2092); 12: 10 waves of 16 x 5
    // rows 1279 (8 of 12 x 7: 1318, 7: 1361)
#define QOL_QINV(RL_, RA_, CL_, CB_, NW_)                                                                \
  hipLaunchKernelGGL((rrq_real_inverse_kernel<RL_, RA_, CL_, CB_>), dim3(npan), dim3(64), 0, s, T, P, npan, nrrq); \
  hipLaunchKernelGGL((rrq_quat_inverse_kernel<RL_, RA_, CL_, CB_, NW_>), dim3(npan), dim3(64 * NW_), 0, s, T, P,   \
                     npan, nrrq)
    if (h <= 3) { QOL_QINV(3, 1, 3, 1, 1); }
    else if (h <= 6) { QOL_QINV(6, 1, 6, 1, 1); }
    else if (h <= 10) { QOL_QINV(5, 2, 10, 1, 1); }
    else if (h <= 15) { QOL_QINV(3, 5, 15, 1, 1); }
    else if (h <= 21) { QOL_QINV(3, 7, 21, 1, 1); }
    else if (h <= 28) { QOL_QINV(4, 7, 16, 2, 2); }
    else if (h <= 36) { QOL_QINV(6, 6, 10, 4, 2); }
    else if (h <= 45) { QOL_QINV(8, 6, 8, 6, 3); }
    else if (h <= 55) { QOL_QINV(9, 7, 7, 8, 8); }
    else if (h <= 66) { QOL_QINV(10, 7, 6, 12, 4); }
    else { QOL_QINV(16, 5, 4, 20, 10); }
#undef QOL_QINV
  } else if (rpt <= 3 && cpt <= 5) {
    hipLaunchKernelGGL((rrq_panel_solve_kernel<3, 5>), dim3(npan), dim3(256), 0, s, T, P, npan, nrrq);
  } else if (rpt <= 4 && cpt <= 7) {
    hipLaunchKernelGGL((rrq_panel_solve_kernel<4, 7>), dim3(npan), dim3(256), 0, s, T, P, npan, nrrq);
  } else if (rpt <= 5 && cpt <= 10) {
    hipLaunchKernelGGL((rrq_panel_solve_kernel<5, 10>), dim3(npan), dim3(256), 0, s, T, P, npan, nrrq);
  } else {
    throw std::runtime_error("RRQ solve supports patch orders up to 12");
  }
  if (rrq_forms_operator(T.p))
    hipLaunchKernelGGL(T.p == 11 ? rrq_operator_kernel<11> : rrq_operator_kernel<12>, dim3(npan), dim3(64 * kOpW), 0, s,
                       P, nrrq);
}

// ---------------------------------------------------------------------------
// per-target pieces

// Edge helpers, specialised on the number of edge nodes NQ so that every
// nq-sized array is a register array.  cf = 3 x NQ power-basis coefficients of
// one edge (cf[c * NQ + j] multiplies s^j): value and derivative of the three
// components by Horner's rule with fused multiply-adds
template <int NQ>
__device__ __forceinline__ void pow3_r(const double* cf, double s, double* val, double* der) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double v = cf[c * NQ + NQ - 1], d = 0.0;
#pragma unroll
    for (int k = NQ - 2; k >= 0; --k) {
      d = fma(d, s, v);
      v = fma(v, s, cf[c * NQ + k]);
    }
    val[c] = v;
    der[c] = d;
  }
}

// the same at complex s
template <int NQ>
__device__ __forceinline__ void pow3_c(const double* cf, cd s, cd* val, cd* der) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    cd v = cmk(cf[c * NQ + NQ - 1], 0.0), d = cmk(0.0, 0.0);
#pragma unroll
    for (int k = NQ - 2; k >= 0; --k) {
      // d = d s + v, v = v s + cf_k
      d = cmk(fma(d.re, s.re, fma(-d.im, s.im, v.re)), fma(d.re, s.im, fma(d.im, s.re, v.im)));
      v = cmk(fma(v.re, s.re, fma(-v.im, s.im, cf[c * NQ + k])), fma(v.re, s.im, v.im * s.re));
    }
    val[c] = v;
    der[c] = d;
  }
}

// complex root of |X_e(s) - x|^2 near [-1,1] by Newton from the chord's root
// s = (-C.D + i |C x D|) / D.D.  The imaginary part comes from the cross product:
// the equal form sqrt(|C|^2 |D|^2 - (C.D)^2) cancels for a target near the
// chord's line (near a vertex), can round to 0, and Newton from a real start
// stays on the real axis.
template <int NQ>
__device__ bool edge_root(const double* cf, const double* x, cd& s0) {
  double A[3], B[3], dA[3], dB[3], D[3], C[3];
  pow3_r<NQ>(cf, -1.0, A, dA);
  pow3_r<NQ>(cf, 1.0, B, dB);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    D[c] = 0.5 * (B[c] - A[c]);
    C[c] = 0.5 * (A[c] + B[c]) - x[c];
  }
  const double dd = D[0] * D[0] + D[1] * D[1] + D[2] * D[2];
  const double cdv = C[0] * D[0] + C[1] * D[1] + C[2] * D[2];
  double cxd[3];
  cross3(C, D, cxd);
  cd s = cmk(-cdv / dd, sqrt(cxd[0] * cxd[0] + cxd[1] * cxd[1] + cxd[2] * cxd[2]) / dd);
  for (int it = 0; it < 30; ++it) {
    cd v[3], d[3];
    pow3_c<NQ>(cf, s, v, d);
    cd f = cmk(0, 0), fp = cmk(0, 0);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      v[c].re -= x[c];
      f = cadd(f, cmul(v[c], v[c]));
      fp = cadd(fp, cscale(cmul(v[c], d[c]), 2.0));
    }
    const cd ds = cdiv(f, fp);
    s = csub(s, ds);
    if (cabs_(ds) < 1e-15 * (1.0 + cabs_(s))) { s0 = s; return isfinite(s.re) && isfinite(s.im); }
  }
  s0 = s;
  return false;
}

// singularity-swap weights for the 1/|X(s)-x| kernel on one edge; w applies to f_i/R_i
template <int NQ>
__device__ void ssq_w1(const double* cf, const double* tgl, const double* wgl, const double* x, double rho_thr,
                       double* w, cd* root, bool* rok) {
  cd s0;
  const bool ok = edge_root<NQ>(cf, x, s0);
  *root = s0;
  *rok = ok;
  if (!ok || bernstein_rho(s0) >= rho_thr) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) w[i] = wgl[i];
    return;
  }
  const double a = s0.re, b = fabs(s0.im), sg = 1.0 + fabs(a);
  const double x1 = 1.0 - a, x2 = -1.0 - a;
  const double r1 = sqrt(x1 * x1 + b * b), r2 = sqrt(x2 * x2 + b * b);
  double I[NQ];
  if (x2 >= 0.0) I[0] = log((x1 + r1) / (x2 + r2));
  else if (x1 <= 0.0) I[0] = log((r2 - x2) / (r1 - x1));
  else I[0] = log((x1 + r1) * (r2 - x2) / (b * b));
  if (NQ > 1) I[1] = r1 - r2;
  double p1 = x1, p2 = x2;
#pragma unroll
  for (int kk = 2; kk < NQ; ++kk) {
    const double dk = (double)kk;
    I[kk] = (p1 * r1 - p2 * r2 - (dk - 1.0) * b * b * I[kk - 2]) / dk;
    p1 *= x1;
    p2 *= x2;
  }
  double sc = 1.0;
#pragma unroll
  for (int kk = 0; kk < NQ; ++kk) { I[kk] *= sc; sc /= sg; }
  // dual Vandermonde system sum_i lam_i t_i^k = I_k (Bjorck-Pereyra), t_i = (s_i - a)/sg
  double t[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) t[i] = (tgl[i] - a) / sg;
  constexpr int N = NQ - 1;
#pragma unroll
  for (int kk = 0; kk < N; ++kk)
#pragma unroll
    for (int i = N; i > kk; --i) I[i] -= t[kk] * I[i - 1];
#pragma unroll
  for (int kk = N - 1; kk >= 0; --kk) {
#pragma unroll
    for (int i = kk + 1; i <= N; ++i) I[i] /= (t[i] - t[i - kk - 1]);
#pragma unroll
    for (int i = kk; i < N; ++i) I[i] -= I[i + 1];
  }
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const double ds = tgl[i] - a;
    w[i] = I[i] * sqrt(ds * ds + b * b);
  }
}

// Dirac-string line integral of one edge, adaptive march toward the near point.
// The march takes the largest interval [lo, hi], halving from twice the last one,
// whose Bernstein ellipse of parameter thr leaves the root s0 outside: with foci lo
// and hi that is |s0 - lo| + |s0 - hi| >= (thr + 1/thr) (hi - lo)/2, two square
// roots (hardware estimates do: which of two equally good intervals is taken when
// they tie changes the sum by the rule's own 1e-15) where the parameter itself
// takes a complex division, two complex square roots and three hypots.
// LW lanes share an item: lane i of them takes node i of every interval (LW = 1:
// all nodes); the caller adds the lanes' sums.
template <int NQ, int LW>
__device__ double solid_angle_edge(const double* cf, const double* tgl, const double* wgl, const double* x,
                                   const double* q, cd s0, bool ok, double ell, int i0) {
  double total = 0.0, lo = -1.0, len = 2.0;
  int guard = 0;
  const double im2 = s0.im * s0.im;
  while (lo < 1.0 && guard < 512) {
    ++guard;
    double hi = fmin(1.0, lo + len);
    if (ok) {
      const double dl = __builtin_amdgcn_sqrt(fma(s0.re - lo, s0.re - lo, im2));
      while (hi - lo > 1e-14) {
        const double dh = __builtin_amdgcn_sqrt(fma(s0.re - hi, s0.re - hi, im2));
        if (dl + dh >= ell * (hi - lo)) break;
        hi = lo + 0.5 * (hi - lo);
      }
    }
    const double c = 0.5 * (lo + hi), hh = 0.5 * (hi - lo);
#pragma unroll 2
    for (int i = i0; i < NQ; i += LW) {
      const double s = c + hh * tgl[i];
      double X[3], dX[3];
      pow3_r<NQ>(cf, s, X, dX);
      const double z[3] = {X[0] - x[0], X[1] - x[1], X[2] - x[2]};
      double zx[3];
      cross3(z, dX, zx);
      const double rz = sqrt(z[0] * z[0] + z[1] * z[1] + z[2] * z[2]);
      const double qz = q[0] * z[0] + q[1] * z[1] + q[2] * z[2];
      const double qzx = q[0] * zx[0] + q[1] * zx[1] + q[2] * zx[2];
      total += hh * wgl[i] * qzx * rcp_nr(rz * (rz + qz));
    }
    len = 2.0 * (hi - lo);
    lo = hi;
  }
  return total;
}

// Gauss-Newton projection of x (original coordinates) onto the patch, started
// at the nearest node (ssx: the panel's nodes, x(3,h)), in three pieces so the
// iterations can be split over two launches: the start, Gauss-Newton steps
// it0 <= it < it1 (true once a step is below 1e-15), and the end (the normal at
// the projection and the signed distance along it).
__device__ void project_start(const double* ssx, const double* uvn, int h, const double* x, double& u, double& v) {
  double best = 1e300;
  u = 1.0 / 3.0;
  v = 1.0 / 3.0;
  for (int i = 0; i < h; ++i) {
    const double d0 = ssx[3 * i] - x[0], d1 = ssx[3 * i + 1] - x[1], d2 = ssx[3 * i + 2] - x[2];
    const double d = d0 * d0 + d1 * d1 + d2 * d2;
    if (d < best) { best = d; u = uvn[2 * i]; v = uvn[2 * i + 1]; }
  }
}

// One Gauss-Newton update of (u, v) from the point y and its tangents, clamped
// to the triangle; true when the step |du| + |dv| (also returned in st) is below
// 1e-15 or below 8 eps |x| sqrt((a11 + a22) / det) (xn = |x|): eight times the
// step that rounding of the residual alone makes, since 1 / the Jacobian's
// smallest singular value is at most sqrt((a11 + a22) / det).  A fixed 1e-15 is
// below that floor on small panels, where the iteration would cycle to the cap.
__device__ __forceinline__ bool gn_step(const double* x, double xn, const double* y, const double* yu,
                                        const double* yv, double& u, double& v, double& st) {
  const double r[3] = {y[0] - x[0], y[1] - x[1], y[2] - x[2]};
  const double a11 = yu[0] * yu[0] + yu[1] * yu[1] + yu[2] * yu[2];
  const double a12 = yu[0] * yv[0] + yu[1] * yv[1] + yu[2] * yv[2];
  const double a22 = yv[0] * yv[0] + yv[1] * yv[1] + yv[2] * yv[2];
  const double b1 = -(yu[0] * r[0] + yu[1] * r[1] + yu[2] * r[2]);
  const double b2 = -(yv[0] * r[0] + yv[1] * r[1] + yv[2] * r[2]);
  const double det = a11 * a22 - a12 * a12;
  double un = u + (a22 * b1 - a12 * b2) / det, vn = v + (a11 * b2 - a12 * b1) / det;
  if (un < 0.0) un = 0.0;
  if (vn < 0.0) vn = 0.0;
  if (un + vn > 1.0) {
    const double ex = 0.5 * (un + vn - 1.0);
    un -= ex; vn -= ex;
    if (un < 0.0) { vn += un; un = 0.0; }
    if (vn < 0.0) { un += vn; vn = 0.0; }
  }
  st = fabs(un - u) + fabs(vn - v);
  u = un; v = vn;
  return st < fmax(1e-15, 8.0 * 2.220446049250313e-16 * xn * sqrt((a11 + a22) / det));
}

__device__ bool project_steps(const double* cx, const double* __restrict__ kt, int h, int korder, const double* x,
                              double& u, double& v, int it0, int it1) {
  const double xn = sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
  double y[3], yu[3], yv[3], st;
  for (int it = it0; it < it1; ++it) {
    geom_eval(cx, kt, h, korder, u, v, y, yu, yv);
    if (gn_step(x, xn, y, yu, yv, u, v, st)) return true;
  }
  return false;
}

// A projection that ends at the step cap: stat[0] counts them, the 8 bytes at
// stat + 2 hold the largest last step (a non-negative double's bits order as its
// value, so an unsigned maximum of the bits is the maximum of the values).
__device__ __forceinline__ void note_capped(int* stat, double st) {
  atomicAdd(stat, 1);
  atomicMax(reinterpret_cast<unsigned long long*>(stat + 2), (unsigned long long)__double_as_longlong(st));
}

__device__ double project_end(const double* cx, const double* __restrict__ kt, int h, int korder, const double* x,
                              double u, double v, double* nstar) {
  double y[3], yu[3], yv[3];
  geom_eval(cx, kt, h, korder, u, v, y, yu, yv);
  double nn[3];
  cross3(yu, yv, nn);
  const double l = sqrt(nn[0] * nn[0] + nn[1] * nn[1] + nn[2] * nn[2]);
  for (int c = 0; c < 3; ++c) nstar[c] = nn[c] / l;
  return (x[0] - y[0]) * nstar[0] + (x[1] - y[1]) * nstar[1] + (x[2] - y[2]) * nstar[2];
}

// ---------------------------------------------------------------------------
// Per-target work in three launches over the RRQ pair list (label 5, grouped by
// panel; r = position in that list):
//   rrq_project_kernel  one thread per pair: projection onto the patch, side,
//                       Dirac-string direction q (frame)            -> pq[r][4]
//   rrq_edge_kernel     one thread per (pair, edge): complex root, SSQ weights
//                       for the 1/r line kernel and the edge's solid-angle
//                       line integral                              -> w1[r][3nq], oe[r][3]
//   rrq_target_kernel   a panel's pairs in tiles: boundary moments, degree
//                       recursion, moment vectors                   -> vt

__device__ __forceinline__ int rrq_list_base(const int* ltot) { return ltot[0] + ltot[1] + ltot[2] + ltot[3]; }

__global__ void zero_ints_kernel(int* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Projection in two launches: every pair takes up to kPI Gauss-Newton steps;
// the few that have not converged (a list built with an atomic counter) continue
// in the second launch from the saved (u, v), so a wave no longer runs as long
// as its slowest pair.  The step sequence of every pair is the single loop's,
// so the results are the same.  A pair that has not met the stop test of
// gn_step after kPMax steps keeps its last iterate, as in the single loop, and is
// counted in `nfail` (with the largest such last step) so that the caller can
// see it.
constexpr int kPI = 8, kPMax = 40;

__device__ void project_write(RRQTables T, RRQPanels P, int k, const double* x, double u, double v, int exterior,
                              double side_tol, double* o) {
  const int h = T.h;
  const double* fr = P.frame + (size_t)k * 16;
  double ns[3];
  const double d = project_end(P.cx + (size_t)k * 3 * h, T.ktab, h, T.p - 1, x, u, v, ns);
  double side;
  if (fabs(d) > side_tol * fr[14]) side = d > 0.0 ? 1.0 : -1.0;
  else side = (exterior ? 1.0 : -1.0) * fr[13];
  const double qo[3] = {-side * ns[0], -side * ns[1], -side * ns[2]};
  double q[3];
  rotate(fr, qo, q);
  o[0] = q[0]; o[1] = q[1]; o[2] = q[2]; o[3] = side;
}

__global__ void __launch_bounds__(256) rrq_project_kernel(RRQTables T, RRQPanels P, const int* __restrict__ lpairs,
                                                          const int* __restrict__ ltot,
                                                          const int* __restrict__ ppanel,
                                                          const int* __restrict__ tidx,
                                                          const double* __restrict__ tx,
                                                          const double* __restrict__ sx, int exterior,
                                                          double side_tol, double* __restrict__ pq,
                                                          int* __restrict__ rest, int* __restrict__ nrest) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= ltot[4]) return;
  const int pair = lpairs[rrq_list_base(ltot) + r];
  const int k = ppanel[pair], h = T.h;
  const size_t g = (size_t)tidx[pair];
  const double x[3] = {tx[3 * g], tx[3 * g + 1], tx[3 * g + 2]};
  double u, v;
  project_start(sx + (size_t)k * 3 * h, T.uvn, h, x, u, v);
  double* o = pq + 4 * (size_t)r;
  if (project_steps(P.cx + (size_t)k * 3 * h, T.ktab, h, T.p - 1, x, u, v, 0, kPI)) {
    project_write(T, P, k, x, u, v, exterior, side_tol, o);
  } else {
    o[0] = u; o[1] = v;  // the state, for the second launch
    rest[atomicAdd(nrest, 1)] = r;
  }
}

__global__ void __launch_bounds__(256) rrq_project_rest_kernel(RRQTables T, RRQPanels P,
                                                               const int* __restrict__ lpairs,
                                                               const int* __restrict__ ltot,
                                                               const int* __restrict__ ppanel,
                                                               const int* __restrict__ tidx,
                                                               const double* __restrict__ tx, int exterior,
                                                               double side_tol, double* __restrict__ pq,
                                                               const int* __restrict__ rest,
                                                               const int* __restrict__ nrest,
                                                               int* __restrict__ nfail) {
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= *nrest) return;
  const int r = rest[gid];
  const int pair = lpairs[rrq_list_base(ltot) + r];
  const int k = ppanel[pair], h = T.h;
  const size_t g = (size_t)tidx[pair];
  const double x[3] = {tx[3 * g], tx[3 * g + 1], tx[3 * g + 2]};
  double* o = pq + 4 * (size_t)r;
  double u = o[0], v = o[1];
  const double* cx = P.cx + (size_t)k * 3 * h;
  const double xn = sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
  double y[3], yu[3], yv[3], st = 0.0;
  bool done = false;
  for (int it = kPI; it < kPMax && !done; ++it) {
    geom_eval(cx, T.ktab, h, T.p - 1, u, v, y, yu, yv);
    done = gn_step(x, xn, y, yu, yv, u, v, st);
  }
  if (!done) note_capped(nfail, st);
  project_write(T, P, k, x, u, v, exterior, side_tol, o);
}

// The second launch runs few pairs and so is bound by each step's latency: for
// the orders up to 8 it holds the panel's coefficients in registers and unrolls
// the evaluation (the same operations in the same order as geom_eval, so the
// same results).  In the first launch, which is bound by throughput, the same
// unrolled form measured slower (it needs more registers, so fewer waves).
template <int N>
__device__ __forceinline__ void geom_eval_reg(const double (&cr)[3][N * (N + 1) / 2], const double* __restrict__ kt,
                                              double u, double v, double* x, double* xu, double* xv) {
  const double a = 2.0 * u + v - 1.0, b = 1.0 - v, bb = b * b;
#pragma unroll
  for (int c = 0; c < 3; ++c) { x[c] = 0.0; xu[c] = 0.0; xv[c] = 0.0; }
  const double xx = 2.0 * v - 1.0;
  double Q = 1.0, Qu = 0.0, Qv = 0.0, Qm = 0.0, Qum = 0.0, Qvm = 0.0;
#pragma unroll
  for (int am = 0; am < N; ++am) {
    if (am == 1) {
      Qm = Q; Qum = Qu; Qvm = Qv;
      Q = a; Qu = 2.0; Qv = 1.0;
    } else if (am >= 2) {
      const double e1 = kt[2 * am], e2 = kt[2 * am + 1];
      const double Qn = e1 * a * Q - e2 * bb * Qm;
      const double Qun = e1 * (2.0 * Q + a * Qu) - e2 * bb * Qum;
      const double Qvn = e1 * (Q + a * Qv) - e2 * (bb * Qvm - 2.0 * b * Qm);
      Qm = Q; Qum = Qu; Qvm = Qv;
      Q = Qn; Qu = Qun; Qv = Qvn;
    }
    const double al = 2.0 * am + 1.0;
    double p = 1.0, dp = 0.0, pm = 1.0, dpm = 0.0;
#pragma unroll
    for (int bd = 0; am + bd < N; ++bd) {
      // table entry of (am, bd): terms are stored am-major after the 2N factors
      const double* tt = kt + 2 * N + 4 * (am * N - am * (am - 1) / 2 + bd);
      if (bd == 1) {
        p = 0.5 * ((al + 2.0) * xx + al);
        dp = al + 2.0;
      } else if (bd >= 2) {
        const double w = tt[1] + tt[2] * xx;
        const double pn = w * p - tt[3] * pm;
        const double dpn = w * dp + 2.0 * tt[2] * p - tt[3] * dpm;
        pm = p; p = pn; dpm = dp; dp = dpn;
      }
      const int d = am + bd, idx = d * (d + 1) / 2 + bd;
      const double sc = tt[0];
      const double f = sc * Q * p;
#pragma unroll
      for (int c = 0; c < 3; ++c) x[c] += f * cr[c][idx];
      const double fu = sc * Qu * p, fv = sc * (Qv * p + Q * dp);
#pragma unroll
      for (int c = 0; c < 3; ++c) { xu[c] += fu * cr[c][idx]; xv[c] += fv * cr[c][idx]; }
    }
  }
}

template <int N>
__global__ void __launch_bounds__(64) rrq_project_rest_reg_kernel(RRQTables T, RRQPanels P,
                                                                  const int* __restrict__ lpairs,
                                                                  const int* __restrict__ ltot,
                                                                  const int* __restrict__ ppanel,
                                                                  const int* __restrict__ tidx,
                                                                  const double* __restrict__ tx, int exterior,
                                                                  double side_tol, double* __restrict__ pq,
                                                                  const int* __restrict__ rest,
                                                                  const int* __restrict__ nrest,
                                                                  int* __restrict__ nfail) {
  constexpr int H = N * (N + 1) / 2;
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= *nrest) return;
  const int r = rest[gid];
  const int pair = lpairs[rrq_list_base(ltot) + r];
  const int k = ppanel[pair];
  const size_t g = (size_t)tidx[pair];
  const double x[3] = {tx[3 * g], tx[3 * g + 1], tx[3 * g + 2]};
  const double* cx = P.cx + (size_t)k * 3 * H;
  double cr[3][H];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int i = 0; i < H; ++i) cr[c][i] = cx[c * H + i];
  double* o = pq + 4 * (size_t)r;
  double u = o[0], v = o[1];
  const double xn = sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
  double y[3], yu[3], yv[3], st = 0.0;
  bool done = false;
  for (int it = kPI; it < kPMax && !done; ++it) {
    geom_eval_reg<N>(cr, T.ktab, u, v, y, yu, yv);
    done = gn_step(x, xn, y, yu, yv, u, v, st);
  }
  if (!done) note_capped(nfail, st);
  project_write(T, P, k, x, u, v, exterior, side_tol, o);
}

void launch_rrq_project(RRQTables T, RRQPanels P, const int* lpairs, const int* ltot, const int* ppanel,
                        const int* tidx, const double* tx, const double* sx, int exterior, double side_tol,
                        double* pq, int* order, int* nfail, int64_t nnz, hipStream_t s) {
  int* nrest = order;      // [1]
  int* rest = order + 1;   // [nnz]
  const dim3 grid((unsigned)((nnz + 255) / 256)), blk(256);
  hipLaunchKernelGGL(zero_ints_kernel, dim3(1), dim3(64), 0, s, nrest, 1);
  hipLaunchKernelGGL(zero_ints_kernel, dim3(1), dim3(64), 0, s, nfail, 4);
  hipLaunchKernelGGL(rrq_project_kernel, grid, blk, 0, s, T, P, lpairs, ltot, ppanel, tidx, tx, sx, exterior,
                     side_tol, pq, rest, nrest);
  const dim3 rgrid((unsigned)((nnz + 63) / 64)), rblk(64);
#define QOL_PROJ(NN)                                                                                            \
  case NN:                                                                                                      \
    hipLaunchKernelGGL(rrq_project_rest_reg_kernel<NN>, rgrid, rblk, 0, s, T, P, lpairs, ltot, ppanel, tidx, tx, \
                       exterior, side_tol, pq, (const int*)rest, (const int*)nrest, nfail);                      \
    break;
  switch (T.p) {
    QOL_PROJ(2) QOL_PROJ(3) QOL_PROJ(4) QOL_PROJ(5) QOL_PROJ(6) QOL_PROJ(7) QOL_PROJ(8)
    default:
      hipLaunchKernelGGL(rrq_project_rest_kernel, grid, blk, 0, s, T, P, lpairs, ltot, ppanel, tidx, tx, exterior,
                         side_tol, pq, (const int*)rest, (const int*)nrest, nfail);
  }
#undef QOL_PROJ
}

// per (pair, edge): complex root and SSQ weights -> w1[r][3NQ], root[r][3][3] (re, im, ok)
template <int NQ>
__global__ void __launch_bounds__(256) rrq_root_kernel(RRQTables T, RRQPanels P, const int* __restrict__ lpairs,
                                                       const int* __restrict__ ltot, const int* __restrict__ ppanel,
                                                       const int* __restrict__ tidx, const double* __restrict__ tx,
                                                       double* __restrict__ w1, double* __restrict__ root) {
  const int it = blockIdx.x * blockDim.x + threadIdx.x;
  if (it >= 3 * ltot[4]) return;
  const int r = it / 3, e = it % 3;
  const int pair = lpairs[rrq_list_base(ltot) + r];
  const int k = ppanel[pair];
  const double* fr = P.frame + (size_t)k * 16;
  const size_t g = (size_t)tidx[pair];
  const double x[3] = {tx[3 * g], tx[3 * g + 1], tx[3 * g + 2]};
  double X[3];
  to_frame(fr, x, X);
  const double* cf = P.edge + (size_t)k * 9 * NQ + e * 3 * NQ;
  const double rho_thr = pow(8.0, 8.0 / (double)NQ);
  cd s0;
  bool ok;
  ssq_w1<NQ>(cf, T.tgl, T.wgl, X, rho_thr, w1 + (size_t)r * 3 * NQ + e * NQ, &s0, &ok);
  double* o = root + 3 * (size_t)it;
  o[0] = s0.re; o[1] = s0.im; o[2] = ok ? 1.0 : 0.0;
}

// per (pair, edge): the edge's Dirac-string line integral of the solid angle -> oe[r][3].
// One thread an item when the items fill the chip (their march is up to 50 intervals,
// and the sort makes a wave's lengths alike); below that 8 or 16 lanes an item, one
// per node, since then one march's latency is all that counts.  The line lies where the
// two meet, which the lanes that have no node move: one thread and lanes take (us, on a
// stream of its own)
//   order 2   132,000 items 527, 394   195,000 549, 560
//   order 3   132,000       315, 227   195,000 317, 324
//   order 4   195,000       239, 206   291,000 272, 297
//   order 5   195,000       197, 182   291,000 225, 254
//   order 6   393,000       209, 191   480,000 239, 232   720,000 278, 333
//   order 7    72,000       143, 100   108,000 143, 140   132,000 145, 166
//   order 8    72,000       138, 101   108,000 142, 142   132,000 147, 166
//   order 9   132,000       164, 157   195,000 165, 223
//   order 10  108,000       131, 120   132,000 131, 141
//   order 11  132,000       155, 144   195,000 161, 201
//   order 12  132,000       156, 141   195,000 169, 198
// With the parameter test in solid_angle_edge and one thread an item 98,000 and 291,000
// items of order 6 took 239 and 319, the 60 items of one panel 148 (now 31), the 960,000
// of the 48 x 120 order-8 workload 480 (now 325, bound by the vector rate).
template <int NQ>
constexpr int solid_lanes() { return NQ <= 8 ? 8 : 16; }
template <int NQ>
constexpr int solid_wide() {
  return NQ <= 5 ? 180224 : (NQ <= 7 ? 229376 : (NQ == 8 ? 393216 : (NQ <= 10 ? 106496 : 131072)));
}

template <int NQ>
__global__ void __launch_bounds__(256) rrq_solid_kernel(RRQTables T, RRQPanels P, const int* __restrict__ lpairs,
                                                        const int* __restrict__ ltot, const int* __restrict__ ppanel,
                                                        const int* __restrict__ tidx, const double* __restrict__ tx,
                                                        const double* __restrict__ pq, const double* __restrict__ root,
                                                        const int* __restrict__ perm, double ell,
                                                        double* __restrict__ oe) {
  constexpr int LW = solid_lanes<NQ>();
  const int gid = blockIdx.x * blockDim.x + threadIdx.x, n = 3 * ltot[4];
  const bool wide = n <= solid_wide<NQ>();
  const int item = wide ? gid / LW : gid;
  if (item >= n) return;
  const int it = perm ? perm[item] : item;  // items in order of their cost bucket
  const int r = it / 3, e = it % 3;
  const int pair = lpairs[rrq_list_base(ltot) + r];
  const int k = ppanel[pair];
  const double* fr = P.frame + (size_t)k * 16;
  const size_t g = (size_t)tidx[pair];
  const double x[3] = {tx[3 * g], tx[3 * g + 1], tx[3 * g + 2]};
  double X[3];
  to_frame(fr, x, X);
  const double* cf = P.edge + (size_t)k * 9 * NQ + e * 3 * NQ;
  const double* rt = root + 3 * (size_t)it;
  const double q[3] = {pq[4 * (size_t)r], pq[4 * (size_t)r + 1], pq[4 * (size_t)r + 2]};
  const cd s0 = cmk(rt[0], rt[1]);
  const bool ok = rt[2] != 0.0;
  if (wide) {
    double v = solid_angle_edge<NQ, LW>(cf, T.tgl, T.wgl, X, q, s0, ok, ell, gid % LW);
#pragma unroll
    for (int o = LW / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (gid % LW == 0) oe[it] = v;
  } else {
    oe[it] = solid_angle_edge<NQ, 1>(cf, T.tgl, T.wgl, X, q, s0, ok, ell, 0);
  }
}

// The solid-angle march of a (pair, edge) item takes about 2 log2(1/d) intervals,
// d the distance of the edge's complex root from [-1, 1] (one interval without a
// root).  Items are grouped by that cost -- a counting sort into kSB buckets,
// costliest first -- so the lanes of a wave run similar marches.  Each item
// writes only its own result, so the order changes nothing but the time.
constexpr int kSB = 64;

__device__ __forceinline__ int solid_bucket(const double* rt) {
  if (rt[2] == 0.0) return 0;
  const double dx = fmax(fabs(rt[0]) - 1.0, 0.0), im = fabs(rt[1]);
  const double d = sqrt(dx * dx + im * im);
  if (!(d > 0.0)) return kSB - 1;  // on the segment, or not a number
  int e;
  (void)frexp(d, &e);  // d in [2^(e-1), 2^e)
  return min(max(2 - e, 0), kSB - 1);
}

// counts per bucket: a histogram per workgroup in LDS, then one global add per
// non-empty bucket (kSI items per thread)
constexpr int kSI = 4;
__global__ void __launch_bounds__(256) solid_count_kernel(const int* __restrict__ ltot, const double* __restrict__ root,
                                                          int* __restrict__ cnt, int* __restrict__ key) {
  __shared__ int lh[kSB];
  for (int b = threadIdx.x; b < kSB; b += blockDim.x) lh[b] = 0;
  __syncthreads();
  const int n = 3 * ltot[4];
  const int base = blockIdx.x * blockDim.x * kSI + threadIdx.x;
#pragma unroll
  for (int u = 0; u < kSI; ++u) {
    const int it = base + u * blockDim.x;
    if (it < n) {
      const int b = solid_bucket(root + 3 * (size_t)it);
      key[it] = b;
      atomicAdd(lh + b, 1);
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < kSB; b += blockDim.x)
    if (lh[b]) atomicAdd(cnt + b, lh[b]);
}

// bucket starts, costliest bucket first (one thread); cnt[kSB..2kSB) receive them
__global__ void solid_offsets_kernel(int* __restrict__ cnt) {
  if (threadIdx.x != 0) return;
  int s = 0;
  for (int b = kSB - 1; b >= 0; --b) {
    cnt[kSB + b] = s;
    s += cnt[b];
  }
}

// the permutation: ranks within the workgroup from LDS, one global range per
// non-empty bucket per workgroup
__global__ void __launch_bounds__(256) solid_scatter_kernel(const int* __restrict__ ltot, const int* __restrict__ key,
                                                            int* __restrict__ cnt, int* __restrict__ perm) {
  __shared__ int lh[kSB], lb[kSB];
  for (int b = threadIdx.x; b < kSB; b += blockDim.x) lh[b] = 0;
  __syncthreads();
  const int n = 3 * ltot[4];
  const int base = blockIdx.x * blockDim.x * kSI + threadIdx.x;
  int bk[kSI], rk[kSI];
#pragma unroll
  for (int u = 0; u < kSI; ++u) {
    const int it = base + u * blockDim.x;
    bk[u] = it < n ? key[it] : -1;
    rk[u] = bk[u] >= 0 ? atomicAdd(lh + bk[u], 1) : 0;
  }
  __syncthreads();
  for (int b = threadIdx.x; b < kSB; b += blockDim.x) lb[b] = lh[b] ? atomicAdd(cnt + kSB + b, lh[b]) : 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kSI; ++u)
    if (bk[u] >= 0) perm[lb[bk[u]] + rk[u]] = base + u * blockDim.x;
}

size_t rrq_edge_order_ints(int64_t nnz) { return (size_t)2 * kSB + (size_t)6 * nnz; }

void launch_rrq_edge(RRQTables T, RRQPanels P, const int* lpairs, const int* ltot, const int* ppanel,
                     const int* tidx, const double* tx, const double* pq, double* w1, double* root, double* oe,
                     int* order, int64_t nnz, hipStream_t s, hipEvent_t mid) {
  const dim3 grid((unsigned)((3 * nnz + 255) / 256)), blk(256);
  const dim3 gsort((unsigned)((3 * nnz + 256 * kSI - 1) / (256 * kSI)));
  int* cnt = order;                  // [2 kSB]: counts, then bucket starts
  int* key = order + 2 * kSB;        // [3 nnz]
  int* perm = key + 3 * nnz;         // [3 nnz]
  // so few items that all their waves run at once: their order does not matter, and
  // the sort's four launches (16 us) cost more than it saves
  const bool sort = 3 * nnz > 16384;
  const double thr = std::pow(8.0, 8.0 / (double)T.nq), ell = 0.5 * (thr + 1.0 / thr);
#define QOL_EDGE(NQ_)                                                                                      \
  case NQ_:                                                                                                \
    hipLaunchKernelGGL(rrq_root_kernel<NQ_>, grid, blk, 0, s, T, P, lpairs, ltot, ppanel, tidx, tx, w1, root); \
    if (mid) (void)hipEventRecord(mid, s);                                                                 \
    if (sort) {                                                                                           \
      hipLaunchKernelGGL(zero_ints_kernel, dim3(1), dim3(2 * kSB), 0, s, cnt, 2 * kSB);                    \
      hipLaunchKernelGGL(solid_count_kernel, gsort, blk, 0, s, ltot, (const double*)root, cnt, key);      \
      hipLaunchKernelGGL(solid_offsets_kernel, dim3(1), dim3(64), 0, s, cnt);                             \
      hipLaunchKernelGGL(solid_scatter_kernel, gsort, blk, 0, s, ltot, (const int*)key, cnt, perm);       \
    }                                                                                                     \
    hipLaunchKernelGGL(rrq_solid_kernel<NQ_>,                                                              \
                       dim3((unsigned)((std::max(3 * nnz, std::min<int64_t>(3 * nnz, solid_wide<NQ_>()) * solid_lanes<NQ_>()) + 255) / 256)), \
                       blk, 0, s, T, P, lpairs, ltot, ppanel, tidx, tx, pq, root, sort ? (const int*)perm : nullptr, ell, oe); \
    break;
  switch (T.nq) {
    QOL_EDGE(4) QOL_EDGE(5) QOL_EDGE(6) QOL_EDGE(7) QOL_EDGE(8) QOL_EDGE(9) QOL_EDGE(10) QOL_EDGE(11)
    QOL_EDGE(12) QOL_EDGE(13) QOL_EDGE(14)
    default: throw std::runtime_error("RRQ edge kernels: patch orders 2..12 only");
  }
#undef QOL_EDGE
}

// Boundary moments, degree recursion and moment vectors of a panel's RRQ pairs, in
// tiles of up to kRT = 16 pairs.
//
// With z = X_b - x, w = (SSQ weight)/|z| and dX the edge tangent at boundary node
// b, a pair needs chi_n^m = sum_b (w z x dX) . grad H'_n^m and the quaternion
// moments alpha_n^m = sum_b (w z) (x) V_n^m, V_n^m = n (dX_Z G + i/2 (dW G^{m-1} +
// conj(dW) G^{m+1})), G = grad H'_{n-1}^m.  Gradients are fixed combinations of
// harmonics one degree lower, and that step commutes with the combination over
// dX, so everything follows from six real node weights: R_c = sum_b (w z x dX)_c H'
// and S_c = sum_b (w z_c) T (T: rrq_panel_system_kernel),
//   chi  = n (R_0^m + i/2 (R_1^{m-1} + R_1^{m+1}) + 1/2 (R_2^{m+1} - R_2^{m-1}))
//   U_cd = n (n-1) (S_c^m, i/2 (S_c^{m-1} + S_c^{m+1}), 1/2 (S_c^{m+1} - S_c^{m-1}))_d
//   alpha = (-(U_00 + U_11 + U_22), U_12 - U_21, U_20 - U_02, U_01 - U_10)
// (twelve weights against H' alone, a general combination of 39 sums per
// coefficient and a barrier per degree took 2.6 ms on the 48 x 120 order-8
// workload, 320,000 pairs, of which the sums 0.9, the combination 0.5 and the
// degrees 0.75; now 0.96, of which the weights 0.15 and the sums about 0.4).
//
// The sums are a matrix product on the FP64 matrix cores: rows (pair, weight),
// columns the real and imaginary parts of the panel's H' or T, inner dimension
// the boundary nodes.  The rows of one tile share every harmonic loaded, the
// weights go through LDS once, and the results land in LDS for the recursion, one
// lane per (pair, component), which keeps its previous degree in registers and
// needs no barrier.
constexpr int kRT = 16;   // pairs a tile at most (12 and 10: 1.07 and 1.10 ms)
constexpr int kRW = 4;    // waves a workgroup: with 5, two workgroups a CU fit instead of three (1.6 ms)

template <int P>
struct MomentPlan {
  static constexpr int NB = 3 * (P + 2), KS = (NB + 3) / 4;            // nodes, in steps of 4
  static constexpr int CH = P * (P + 1), CT = (P - 1) * (P + 2);       // real columns of H' and T
  static constexpr int NH = (CH + 15) / 16, NN = NH + (CT + 15) / 16;  // 16-column tiles of H', of both
  static constexpr int RS = 3 * (CH + CT);                             // sums per pair
  static constexpr int rows(int t) { return 16 * ((3 * t + 15) / 16); }
  // the region holds the node weights (both sets, and w), then the sums
  static constexpr int region(int t) {
    const int w = 2 * 4 * KS * rows(t) + t * NB;
    return w > t * RS ? w : t * RS;
  }
  static constexpr size_t bytes(int t) { return 8 * (size_t)(region(t) + 6 * NB + 4 * kRT); }
  // three workgroups a CU up to order 8, two above (160 KB of LDS)
  static constexpr int tile() {
    int t = kRT;
    while (t > 1 && bytes(t) > (P <= 8 ? 54400 : 81600)) --t;
    return t;
  }
  static constexpr int T = tile(), MT = rows(T) / 16, TW = (NN + kRW - 1) / kRW;
};

template <int P>
__global__ void __launch_bounds__(64 * kRW, P <= 8 ? 3 : 2)
    rrq_target_kernel(RRQTables tab, RRQPanels pan, const int* __restrict__ lpairs, const int* __restrict__ lstart,
                      const int* __restrict__ ltot, int npan, const int* __restrict__ tidx,
                      const double* __restrict__ tx, const int* __restrict__ nrrq, const double* __restrict__ w1g,
                      const double* __restrict__ oeg, double* __restrict__ vt, double* __restrict__ omega_out,
                      double* __restrict__ ias_out) {
  using M = MomentPlan<P>;
  constexpr int NB = M::NB, KS = M::KS, T = M::T, H = P * (P + 1) / 2;
  const int k = blockIdx.x;
  const int nmine = nrrq[k];
  if ((int)blockIdx.y * T >= nmine) return;
  extern __shared__ double sm[];
  double* rg = sm;                 // the region
  double* bx = rg + M::region(T);  // [NB][6]
  double* lam = bx + 6 * NB;       // [kRT][4]: sum_b w dX
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const double* fr = pan.frame + (size_t)k * 16;
  for (int i = threadIdx.x; i < 6 * NB; i += blockDim.x) bx[i] = pan.bX[(size_t)k * NB * 6 + i];
  const double* basis = pan.basis + (size_t)k * NB * (M::CH + M::CT);
  const int r0 = lstart[4 * (size_t)npan + k];
  const int* mine = lpairs + rrq_list_base(ltot) + r0;
  for (int tile0 = blockIdx.y * T; tile0 < nmine; tile0 += gridDim.y * T) {
    const int nt = min(T, nmine - tile0), mt = (3 * nt + 15) / 16, rows = 16 * mt;
    double *Wa = rg, *Wz = Wa + 4 * KS * rows, *wl = Wz + 4 * KS * rows;
    __syncthreads();  // bx; the previous tile's sums are read
    // node weights, rows (pair, component); the rows of nodes past NB are zero
    for (int it = threadIdx.x; it < nt * 4 * KS; it += blockDim.x) {
      const int ib = it / nt, t = it % nt;  // neighbouring lanes: neighbouring rows
      double a[3] = {0.0, 0.0, 0.0}, zw[3] = {0.0, 0.0, 0.0};
      if (ib < NB) {
        const size_t g = (size_t)tidx[mine[tile0 + t]];
        const double x[3] = {tx[3 * g], tx[3 * g + 1], tx[3 * g + 2]};
        double X[3], zx[3];
        to_frame(fr, x, X);
        const double* Y = bx + 6 * ib;
        const double z[3] = {Y[0] - X[0], Y[1] - X[1], Y[2] - X[2]};
        const double zz = z[0] * z[0] + z[1] * z[1] + z[2] * z[2];
        const double wr = w1g[(size_t)(r0 + tile0 + t) * NB + ib] * (zz == HUGE_VAL ? 0.0 : rsqrt_h3(zz));
        wl[t * NB + ib] = wr;
        cross3(z, Y + 3, zx);
        for (int c = 0; c < 3; ++c) {
          a[c] = wr * zx[c];
          zw[c] = wr * z[c];
        }
      }
      for (int c = 0; c < 3; ++c) {
        Wa[ib * rows + 3 * t + c] = a[c];
        Wz[ib * rows + 3 * t + c] = zw[c];
      }
    }
    __syncthreads();
    // Lambda = sum w dX, by the last wave
    if (wv == kRW - 1 && lane < 3 * nt) {
      const int t = lane / 3, c = lane % 3;
      double l = 0.0;
      for (int ib = 0; ib < NB; ++ib) l = fma(wl[t * NB + ib], bx[6 * ib + 3 + c], l);
      lam[4 * t + c] = l;
    }
    // the sums: this wave's column tiles, all row tiles (lane numbers the compiler
    // cannot tell are the same for every tile: it would keep the addresses they
    // give in registers throughout, and spill)
    int li = lane & 15, lk = lane >> 4;
    asm volatile("" : "+v"(li), "+v"(lk));
    qd4 acc[M::TW][M::MT];
#pragma unroll
    for (int q = 0; q < M::TW; ++q) {
#pragma unroll
      for (int m = 0; m < M::MT; ++m) acc[q][m] = qd4{0.0, 0.0, 0.0, 0.0};
      const int tl = wv + kRW * q;
      if (tl < M::NN) {
        const bool tt = tl >= M::NH;
        const int col = tt ? M::CH + min(16 * (tl - M::NH) + li, M::CT - 1) : min(16 * tl + li, M::CH - 1);
        const double* W = tt ? Wz : Wa;
        double b[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s) b[s] = basis[(size_t)min(4 * s + lk, NB - 1) * (M::CH + M::CT) + col];
#pragma unroll
        for (int m = 0; m < M::MT; ++m)
          if (m < mt)
#pragma unroll
            for (int s = 0; s < KS; ++s)
              acc[q][m] = __builtin_amdgcn_mfma_f64_16x16x4f64(W[(4 * s + lk) * rows + 16 * m + li], b[s], acc[q][m],
                                                               0, 0, 0);
      }
    }
    __syncthreads();  // the weights are read: the sums take their place
#pragma unroll
    for (int q = 0; q < M::TW; ++q) {
      const int tl = wv + kRW * q;
      const bool tt = tl >= M::NH;
      const int col = 16 * (tt ? tl - M::NH : tl) + li;
      if (tl < M::NN && col < (tt ? M::CT : M::CH)) {
#pragma unroll
        for (int m = 0; m < M::MT; ++m)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int row = 16 * m + 4 * j + lk, t = row / 3, c = row % 3;
            if (t < nt) rg[t * M::RS + (tt ? 3 * M::CH + c * M::CT : c * M::CH) + col] = acc[q][m][j];
          }
      }
    }
    __syncthreads();
    // the recursion in degree, component c = 0 (chi) or 1..4 (alpha) of pair t:
    //   E_n^m = f1 base_n^m + f2 (x_Z E_{n-1}^m + i/2 (w E_{n-1}^{m-1} + conj(w) E_{n-1}^{m+1}))
    //   base  = s0 A^m + i h1 (B^{m-1} + B^{m+1}) + h2 (C^{m+1} - C^{m-1})
    // with (f1, f2) = (1, 1) for chi, (n, n / (n - 1)) for alpha, and A, B, C three
    // of the sums R (degree n - 1) or S (degree n - 2, one entry earlier)
    const int t = threadIdx.x % kRT, c = threadIdx.x / kRT;
    if (c < 5 && t < nt) {
      const int pair = mine[tile0 + t];
      const size_t g = (size_t)tidx[pair];
      const double x[3] = {tx[3 * g], tx[3 * g + 1], tx[3 * g + 2]};
      double X[3];
      to_frame(fr, x, X);
      const double* o = oeg + 3 * (size_t)(r0 + tile0 + t);
      const double om = o[0] + o[1] + o[2];
      const double l0 = lam[4 * t], l1 = lam[4 * t + 1], l2 = lam[4 * t + 2];
      const double sigma = fr[13], wr = 0.5 * X[1], wi = 0.5 * X[2], xz = X[0];
      // (A, B, C) by component: chi R0 R1 R2; alpha S0 S1 S2 negated; -, -S2, S1; S2, -, -S0; -S1, S0, -
      const double s0 = c == 0 ? 1.0 : (c == 2 ? 0.0 : (c == 3 ? 1.0 : -1.0));
      const double h1 = c == 0 || c == 4 ? 0.5 : (c == 3 ? 0.0 : -0.5);
      const double h2 = c == 0 || c == 2 ? 0.5 : (c == 4 ? 0.0 : -0.5);
      const cd* base = (const cd*)(rg + t * M::RS) + (c == 0 ? 0 : 3 * (M::CH / 2) - 1);
      const int ca = (c == 0 ? M::CH : M::CT) / 2;
      const cd *A = base + (c == 3 ? 2 : (c == 4 ? 1 : 0)) * ca;
      const cd *B = base + (c <= 1 ? 1 : (c == 2 ? 2 : 0)) * ca;
      const cd *C = base + (c <= 1 ? 2 : (c == 2 ? 1 : 0)) * ca;
      // slots of the moment vector: (x)-components -> h blocks 0..3, chi -> block 4
      const double sgn = c == 0 || c == 1 ? sigma : -sigma;
      double* v = vt + (size_t)r0 * 5 * H + tile0 + t + (size_t)(c == 0 ? 4 * H : (c - 1) * H) * nmine;
      double* om_row = omega_out && c > 0 ? omega_out + (size_t)pair * 4 * H + (c - 1) * H : nullptr;
      const double omf = 1.0 / (16.0 * atan(1.0)) / fr[12];
      cd E[P + 2];
#pragma unroll
      for (int m = 0; m < P + 2; ++m) E[m] = cmk(0.0, 0.0);
      if (c == 0) {
        E[0] = cmk(om, 0.0);
        if (ias_out) ias_out[pair] = sigma * om;
      }
      int i = 0;
#pragma unroll 1  // unrolled, its LDS reads are hoisted until the registers spill
      for (int n = 1; n <= P; ++n) {
        if (n == 1 && c > 0) {
          // seeds: Lambda (x) grad H'_1^m with Lambda = -omega + sum w dX
          E[0] = c == 1 ? cmk(-l0, 0.0) : (c == 2 ? cmk(-om, 0.0) : (c == 3 ? cmk(l2, 0.0) : cmk(-l1, 0.0)));
          E[1] = c == 1 ? cmk(0.5 * l2, -0.5 * l1)
                        : (c == 2 ? cmk(-0.5 * l1, -0.5 * l2) : (c == 3 ? cmk(0.5 * l0, -0.5 * om) : cmk(0.5 * om, 0.5 * l0)));
        } else {
          const double f1 = c == 0 ? 1.0 : (double)n, f2 = c == 0 ? 1.0 : (double)n / (double)(n - 1);
          const int b0 = hidx(n - 1, 0);
          cd bm = cmk(0.0, 0.0), cm = bm, bc = B[b0], cc = C[b0];  // entries m - 1 and m
          cd lo = cmk(-E[1].re, E[1].im);                         // E_{n-1}^{-1}
#pragma unroll
          for (int m = 0; m <= P; ++m) {
            if (m <= n) {
              const cd a = m < n ? A[b0 + m] : cmk(0.0, 0.0);
              const cd bp = m + 1 < n ? B[b0 + m + 1] : cmk(0.0, 0.0), cp = m + 1 < n ? C[b0 + m + 1] : cmk(0.0, 0.0);
              if (m == 0) {
                bm = cmk(-bp.re, bp.im);
                cm = cmk(-cp.re, cp.im);
              }
              const double br = fma(h2, cp.re - cm.re, fma(-h1, bm.im + bp.im, s0 * a.re));
              const double bi = fma(h2, cp.im - cm.im, fma(h1, bm.re + bp.re, s0 * a.im));
              const cd mid = E[m], hi = E[m + 1];
              const double sr = lo.re + hi.re, si = lo.im + hi.im, dr = lo.re - hi.re, di = lo.im - hi.im;
              const double gr = fma(-wi, dr, fma(-wr, si, xz * mid.re));
              const double gi = fma(-wi, di, fma(wr, sr, xz * mid.im));
              E[m] = cmk(fma(f1, br, f2 * gr), fma(f1, bi, f2 * gi));
              lo = mid;
              bm = bc; bc = bp;
              cm = cc; cc = cp;
            }
          }
        }
#pragma unroll
        for (int m = 1; m <= P; ++m)
          if (m <= n) {
            const double e = sgn * imrot(m, E[m]);
            v[(size_t)i * nmine] = e;
            if (om_row) om_row[i] = e * omf;
            ++i;
          }
      }
    }
  }
}

// Workgroups per panel: one when the panels alone fill the chip, else enough for
// 2,048 in all (a panel of 1,501 targets ran its 250 RRQ pairs on one workgroup
// in 470 us), at most one per tile.
void launch_rrq_target(RRQTables T, RRQPanels P, const int* lpairs, const int* lstart, const int* ltot, int npan,
                       const int* tidx, const double* tx, const int* nrrq, const double* w1g, const double* oeg,
                       double* vt, double* omega_out, double* ias_out, int64_t nnz, hipStream_t s) {
  switch (T.p) {
#define QOL_MOMENTS(P_)                                                                                             \
  case P_: {                                                                                                        \
    constexpr size_t lds = MomentPlan<P_>::bytes(MomentPlan<P_>::T);                                                \
    if (lds > 64 * 1024)                                                                                            \
      (void)hipFuncSetAttribute((const void*)rrq_target_kernel<P_>, hipFuncAttributeMaxDynamicSharedMemorySize,     \
                                (int)lds);                                                                          \
    const int64_t tiles = (nnz + MomentPlan<P_>::T - 1) / MomentPlan<P_>::T;                                        \
    const int split = (int)std::max<int64_t>(1, std::min<int64_t>((2048 + npan - 1) / npan, tiles));                \
    hipLaunchKernelGGL(rrq_target_kernel<P_>, dim3(npan, split), dim3(64 * kRW), lds, s, T, P, lpairs, lstart, ltot, \
                       npan, tidx, tx, nrrq, w1g, oeg, vt, omega_out, ias_out);                                      \
    break;                                                                                                          \
  }
    QOL_MOMENTS(2) QOL_MOMENTS(3) QOL_MOMENTS(4) QOL_MOMENTS(5) QOL_MOMENTS(6) QOL_MOMENTS(7) QOL_MOMENTS(8)
    QOL_MOMENTS(9) QOL_MOMENTS(10) QOL_MOMENTS(11) QOL_MOMENTS(12)
#undef QOL_MOMENTS
    default: throw std::runtime_error("RRQ moments: patch orders 2..12 only");
  }
}

// RRQ weights of a panel's pairs from their moment vectors (rhs_0 ... rhs_3, W), on
// the FP64 matrix cores: v = X^T rhs (4h terms), y = W + Fn^T v, Ad = v / 4pi and
// As = B y / (4pi alpha) (h terms each).  Rows: 32 pairs; columns: one wave per 16;
// v and y pass from one product to the next through LDS.
//
// Applying B and Fn here takes 4h^2 multiply-adds a pair, so that the solve need not
// multiply them into X (10h^3 a panel) and nothing but X, Fn and B goes through
// memory (6h^2 doubles a panel where the product took 10h^2, and 162 instead of 225
// matrix steps per 16 pairs at order 8).
// Bound by the matrix cores and, with few panels, by the chains of 4h/8 dependent steps;
// a panel's rounds are split over workgroups until there are 2048 of them.  Order 8,
// 200,000 targets: weights 0.55 to 0.45 ms and the solve 2.1 to 1.6 ms; order 6, 1,501
// targets of one panel: 44 to 13 us.
constexpr int kWT = 32;  // pairs a round

// acc0, acc1 = A (kWT rows, from at(row, k)) times the lane's column of M (col(k)), over
// k < n in steps of four: two row tiles share every column loaded, and even and odd
// steps are separate chains
template <class F, class M>
__device__ __forceinline__ void weights_product(F&& at, M&& col, int n, qd4& acc0, qd4& acc1) {
  const int li = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
  acc0 = acc1 = qd4{0.0, 0.0, 0.0, 0.0};
  qd4 acc2 = acc0, acc3 = acc0;
#pragma unroll 3
  for (int k0 = 0; k0 < n; k0 += 8) {
    const int ka = k0 + lk, kb = k0 + 4 + lk, ca = min(ka, n - 1), cb = min(kb, n - 1);
    const double ma = col(ca), mb = col(cb);
    const double a0 = ka < n ? at(li, ca) : 0.0, a1 = ka < n ? at(16 + li, ca) : 0.0;
    const double b0 = kb < n ? at(li, cb) : 0.0, b1 = kb < n ? at(16 + li, cb) : 0.0;
    acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, ma, acc0, 0, 0, 0);
    acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, ma, acc1, 0, 0, 0);
    acc2 = __builtin_amdgcn_mfma_f64_16x16x4f64(b0, mb, acc2, 0, 0, 0);
    acc3 = __builtin_amdgcn_mfma_f64_16x16x4f64(b1, mb, acc3, 0, 0, 0);
  }
  acc0 += acc2;
  acc1 += acc3;
}

__global__ void __launch_bounds__(320) rrq_weights_kernel(RRQTables T, RRQPanels P, const int* __restrict__ lpairs,
                                                          const int* __restrict__ lstart, const int* __restrict__ ltot,
                                                          int npan, const int* __restrict__ nrrq,
                                                          const double* __restrict__ vt, double* __restrict__ wout) {
  const int k = blockIdx.x;
  const int nm = nrrq[k];
  if ((int)blockIdx.y * kWT >= nm) return;
  extern __shared__ double sm[];
  const int h = T.h, hs = h + 1 - h % 2;  // rows of an odd number of doubles: a column's lanes in different banks
  double *vs = sm, *ys = vs + kWT * hs;
  const int li = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
  const int j = 16 * (threadIdx.x >> 6) + li, jc = min(j, h - 1);  // this lane's column
  const int r0 = lstart[4 * (size_t)npan + k];
  const int* mine = lpairs + rrq_list_base(ltot) + r0;
  const double *X = P.X + (size_t)k * 4 * h * h, *Fn = P.Fn + (size_t)k * h * h, *B = P.Binv + (size_t)k * h * h;
  const double* V = vt + (size_t)r0 * 5 * h;  // V(r, t) at r*nm + t
  const double fac = 1.0 / (16.0 * atan(1.0)), fa = fac / P.frame[(size_t)k * 16 + 12];
  for (int t0 = blockIdx.y * kWT; t0 < nm; t0 += kWT * gridDim.y) {
    const int nt = min(kWT, nm - t0);
    qd4 acc[2];
    // D[4q + lk][li]: pair 4q + lk of the row tile, column j
    auto each = [&](auto&& f) {
      if (j < h)
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int t = 16 * half + 4 * q + lk;
            f(t, acc[half][q]);
          }
    };
    weights_product([&](int t, int c) { return V[(size_t)c * nm + t0 + min(t, nt - 1)]; }, 
                    [&](int c) { return X[(size_t)c * h + jc]; }, 4 * h, acc[0], acc[1]);
    __syncthreads();  // the previous round has read vs and ys
    each([&](int t, double v) {
      vs[t * hs + j] = v;
      if (t < nt) wout[(size_t)mine[t0 + t] * 2 * h + h + j] = v * fac;
    });
    __syncthreads();
    weights_product([&](int t, int i) { return vs[t * hs + i]; }, [&](int i) { return Fn[(size_t)h * jc + i]; }, h, acc[0],
                    acc[1]);
    each([&](int t, double v) { ys[t * hs + j] = v + V[(size_t)(4 * h + j) * nm + t0 + min(t, nt - 1)]; });
    __syncthreads();
    weights_product([&](int t, int r) { return ys[t * hs + r]; }, [&](int r) { return B[(size_t)r * h + jc]; }, h, acc[0],
                    acc[1]);
    each([&](int t, double v) {
      if (t < nt) wout[(size_t)mine[t0 + t] * 2 * h + j] = v * fa;
    });
  }
}

// The same with G formed (orders 11 and 12): As = G rhs + B W / (4pi alpha), Ad = X^T rhs
// / 4pi with the factor in X, one wave per 16 columns of As and then of Ad (order 12,
// 30,000 targets: 0.42 ms, from 0.51 with five waves a panel and all of G in memory)
__global__ void __launch_bounds__(640) rrq_weights_formed_kernel(int h, RRQPanels P, const int* __restrict__ lpairs,
                                                                 const int* __restrict__ lstart,
                                                                 const int* __restrict__ ltot, int npan,
                                                                 const int* __restrict__ nrrq,
                                                                 const double* __restrict__ vt,
                                                                 double* __restrict__ wout) {
  const int nt16 = (h + 15) / 16;
  const int k = blockIdx.x;
  const int nm = nrrq[k];
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool ad = w >= nt16;
  const int j = 16 * (ad ? w - nt16 : w) + li, jc = min(j, h - 1);
  const int r0 = lstart[4 * (size_t)npan + k];
  const int* mine = lpairs + rrq_list_base(ltot) + r0;
  const double *X = P.X + (size_t)k * 4 * h * h + jc, *G = P.G + (size_t)k * 4 * h * h + jc;
  const double *B = P.Binv + (size_t)k * h * h + jc, *V = vt + (size_t)r0 * 5 * h;
  const double fac = 1.0 / (16.0 * atan(1.0)), fa = fac / P.frame[(size_t)k * 16 + 12];
  for (int t0 = blockIdx.y * kWT; t0 < nm; t0 += kWT * gridDim.y) {
    const int nt = min(kWT, nm - t0);
    qd4 acc[2];
    auto at = [&](int t, int c) { return V[(size_t)c * nm + t0 + min(t, nt - 1)]; };
    if (ad)
      weights_product(at, [&](int c) { return X[(size_t)c * h] * fac; }, 4 * h, acc[0], acc[1]);
    else
      weights_product(at, [&](int c) { return c < 4 * h ? G[(size_t)c * h] : B[(size_t)(c - 4 * h) * h] * fa; }, 5 * h, acc[0], acc[1]);
    if (j < h)
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int t = 16 * half + 4 * q + lk;
          if (t < nt) wout[(size_t)mine[t0 + t] * 2 * h + (ad ? h : 0) + j] = acc[half][q];
        }
  }
}

void launch_rrq_weights(RRQTables T, RRQPanels P, const int* lpairs, const int* lstart, const int* ltot, int npan,
                        const int* nrrq, const double* vt, double* wout, int64_t nnz, hipStream_t s) {
  const int64_t rounds = (nnz + kWT - 1) / kWT;
  const int split = (int)std::max<int64_t>(1, std::min<int64_t>((2048 + npan - 1) / npan, rounds));
  if (rrq_forms_operator(T.p)) {
    hipLaunchKernelGGL(rrq_weights_formed_kernel, dim3(npan, split), dim3(128 * ((T.h + 15) / 16)), 0, s, T.h, P, lpairs, lstart, ltot, npan, nrrq, vt, wout);
    return;
  }
  const int nw = (T.h + 15) / 16, hs = T.h + 1 - T.h % 2;
  hipLaunchKernelGGL(rrq_weights_kernel, dim3(npan, split), dim3(64 * nw), sizeof(double) * 2 * kWT * hs, s, T, P,
                     lpairs, lstart, ltot, npan, nrrq, vt, wout);
}

}  // namespace qol
