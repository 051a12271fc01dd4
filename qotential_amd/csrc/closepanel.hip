// Close DLP matrix of a tensor-product patch (the reference's
// Lap3dDLP_closepanel_r64, src/lap3d_close_mod.f90:135-270, behind
// qol_lap3ddlp_closepanel_mex, src/lap3d_close_mex.f90:2-15).
//
// For targets x_k near one patch given by its nodes s_x on a p x p
// Gauss-Legendre tensor grid (node ip = b p + a, a the fast first-parameter
// index), Ac(k, ip) = 1/(4 pi) int (x_k - y).(y_u x y_v)/|x_k - y|^3 L_ip(u,v) du dv
// over [-1,1]^2, y the tensor interpolant of s_x and L_ip its Lagrange basis,
// so that sum_ip Ac(k, ip) sigma(y_ip) is the double-layer potential of the
// interpolated density.  The reference forms it from boundary moments in its
// absent submodules; here the integrals are computed directly by adaptive
// quadrature: a quadtree on the parameter square whose cells are split while
// the target is within ETA diameters of the cell's centre image (depth at most
// MAXDEPTH), each leaf integrated with a q x q Gauss rule, q = 2p + 2 ref.
//
// A workgroup takes one target, or with few targets one of S parts of its leaves
// (the tree is cheap next to the leaves, so every part rebuilds it; the parts'
// sums are added in order).  It walks the tree level by level, one thread per
// (cell, test point), and integrates a level's leaves as soon as they are known,
// one wave per leaf, so no leaf list goes to memory.
//
// A leaf's q x q rule is a tensor product, and so are the interpolant and the
// basis: a lane sums the patch along u for its u-node once (kept in registers),
// then along v per node, and the kernel values are contracted with the basis one
// direction at a time.  At p = 8, q = 18 that is 49 thousand multiply-adds a leaf
// where summing p^2 terms per node took 320 thousand: 777 targets 1e-7 to 0.1 off
// the order-8 torus patch of the reference's smoke test took 99 ms a call, now 6.8
// (order 4: 2.4, order 10 with q = 24: 12, order 16: 90).  Bound by the FP64
// vector rate at two fifths of its issue slots: up to order 8 the registers are
// held to three waves per SIMD (7% over two; a few words of order 8 spill).
// Rules beyond kCpQU x kCpQV nodes go in equal blocks.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

#include "qol_engine.h"
#include "qol_host.h"
#include "qotential_hip.h"

namespace qol {
void set_status(int64_t s);
void set_error(const std::string& s);

namespace {

constexpr int kCpMaxP = 16;       // patch order limit (p^2 <= 256 basis functions)
constexpr int kCpCur = 256;       // cells per tree level
constexpr int kCpLeaves = 4096;   // leaves per target
constexpr int kCpQU = 32;         // quadrature nodes of one block along u (two or more per wave)
constexpr int kCpQV = 40;         // and along v
constexpr int kCpMaxDepth = 48;
constexpr double kCpEta = 2.5;

struct CpArgs {
  int p, q, m;
  int qu, qv;         // nodes a block along u and v
  const double* t;    // p GL nodes
  const double* wb;   // p barycentric weights
  const double* gq;   // q Gauss nodes
  const double* gw;   // q Gauss weights
  const double* sx;   // 3 p^2 patch nodes
  const double* tx;   // 3 m targets
  double* part;       // parts x p^2 x m; part 0 becomes Ac, column-major (m, p^2)
  int* flag;          // set when a target's tree passes the limits
};

// value and derivative of Lagrange polynomial j at u, by products (a call: inlined
// into every unrolled j, its node differences are hoisted into hundreds of registers)
__device__ __noinline__ double2 lagr_at_node(const double* t, int p, int j, double u) {
  double v = 1.0, d = 0.0;
  for (int k = 0; k < p; ++k)
    if (k != j) v *= (u - t[k]) / (t[j] - t[k]);
  for (int r = 0; r < p; ++r) {
    if (r == j) continue;
    double w = 1.0 / (t[j] - t[r]);
    for (int k = 0; k < p; ++k)
      if (k != j && k != r) w *= (u - t[k]) / (t[j] - t[k]);
    d += w;
  }
  return double2{v, d};
}

// Lagrange basis on the GL nodes at u and, with dl, its derivative (barycentric
// form; product form when u sits on a node).  Close to a node the derivative loses
// digits to cancellation, in the weights too; a product form would keep them, but
// callers hold weights of this one.
template <int P>
__device__ __forceinline__ void lagr(const CpArgs& A, double u, double* l, double* dl = nullptr) {
  int hit = -1;
#pragma unroll
  for (int j = 0; j < P; ++j)
    if (fabs(u - A.t[j]) < 1e-14) hit = j;
  if (hit < 0) {
    double S = 0.0, S2 = 0.0;
#pragma unroll
    for (int j = 0; j < P; ++j) {
      const double r = 1.0 / (u - A.t[j]);
      const double a = A.wb[j] * r;
      l[j] = a;
      S += a;
      if (dl) {
        dl[j] = r;
        S2 += a * r;
      }
    }
    const double iS = 1.0 / S, g = S2 * iS;
#pragma unroll
    for (int j = 0; j < P; ++j) {
      l[j] = l[j] * iS;
      if (dl) dl[j] = l[j] * (g - dl[j]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < P; ++j) {
      const double2 v = lagr_at_node(A.t, P, j, u);
      l[j] = v.x;
      if (dl) dl[j] = v.y;
    }
  }
}

// image of (u, v)
template <int P>
__device__ void cp_point(const CpArgs& A, const double* ssx, double u, double v, double* out) {
  double lu[P], lv[P], y[3] = {0.0, 0.0, 0.0};
  lagr<P>(A, u, lu);
  lagr<P>(A, v, lv);
#pragma unroll
  for (int b = 0; b < P; ++b)
#pragma unroll
    for (int a = 0; a < P; ++a) {
      const double* s = ssx + 3 * (b * P + a);
      const double f = lu[a] * lv[b];
      for (int c = 0; c < 3; ++c) y[c] += f * s[c];
    }
  for (int c = 0; c < 3; ++c) out[c] = y[c];
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// doubles of LDS per wave for blocks of nu x nv nodes: l_a at the u-nodes, l_b and
// l_b' at the v-nodes (rows of an odd number of doubles, so the lanes of a column
// fall in different banks), whose space each lane's v-contracted kernel values take
// over, and the v-weights
template <int P>
constexpr int cp_row() { return P + 1 - P % 2; }
template <int P>
__host__ __device__ constexpr int cp_wave_doubles(int nu, int nv) {
  return (nu + (2 * nv > 64 ? 2 * nv : 64)) * cp_row<P>() + nv;
}
constexpr int kCpBatch = 256 / 5;  // cells tested at a time

// one block of nu x nv nodes (u-nodes from ju0, v-nodes from jv0) of the leaf at
// (u0, v0) with half side hs, added into acc[i]: basis function lane + 64 i
template <int P>
__device__ __forceinline__ void cp_block(const CpArgs& A, double* W, const double* x, double u0, double v0, double hs,
                                         int ju0, int nu, int jv0, int nv, double* acc) {
  constexpr int R = cp_row<P>();
  const int lane = threadIdx.x & 63;
  double *wv = W, *lu = wv + A.qv, *lv = lu + A.qu * R, *dlv = lv + A.qv * R, *T = lv;
  // lanes (ju, g): the u-node's sums over a, against l_a (c < 3) and l_a', for
  // every b in registers.  The groups g repeat them: the patch's nodes then have
  // uniform addresses and come through the scalar cache, where dealing the (ju, b)
  // to the lanes cost more LDS reads than the arithmetic it saved
  const int G = 64 / nu, ju = lane % nu, g = lane / nu;
  double r[P][6], cw;
  // read-only address space: scalar loads at every order (left to its own analysis
  // the compiler makes them vector loads at orders 15 and 16, and spills)
  typedef const __attribute__((address_space(4))) double* const_ptr;
  const const_ptr nodes = (const_ptr)(uintptr_t)A.sx;
  {
    double l[P], dl[P];
    if (lane < nv) {
      lagr<P>(A, v0 + hs * (A.gq[jv0 + lane] + 1.0), l, dl);
#pragma unroll
      for (int b = 0; b < P; ++b) {
        lv[lane * R + b] = l[b];
        dlv[lane * R + b] = dl[b];
      }
      wv[lane] = hs * A.gw[jv0 + lane];
    }
    lagr<P>(A, u0 + hs * (A.gq[ju0 + ju] + 1.0), l, dl);
    cw = A.gw[ju0 + ju] * hs / (16.0 * atan(1.0));
    if (g == 0)
#pragma unroll
      for (int a = 0; a < P; ++a) lu[ju * R + a] = l[a];
#pragma unroll
    for (int b = 0; b < P; ++b) {
#pragma unroll
      for (int c = 0; c < 6; ++c) r[b][c] = 0.0;
#pragma unroll
      for (int a = 0; a < P; ++a)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const double n = nodes[3 * (b * P + a) + c];
          r[b][c] = fma(l[a], n, r[b][c]);
          r[b][3 + c] = fma(dl[a], n, r[b][3 + c]);
        }
    }
  }
  wave_sync();
  // v-nodes g, g + G, ...: the image and tangents, the kernel value, and its
  // contraction with l_b over this lane's v-nodes
  double tb[P];
#pragma unroll
  for (int b = 0; b < P; ++b) tb[b] = 0.0;
  if (g < G)
    for (int jv = g; jv < nv; jv += G) {
      double y[3] = {0.0, 0.0, 0.0}, yu[3] = {0.0, 0.0, 0.0}, yv[3] = {0.0, 0.0, 0.0}, l[P];
#pragma unroll
      for (int b = 0; b < P; ++b) {
        l[b] = lv[jv * R + b];
        const double d = dlv[jv * R + b];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          y[c] = fma(l[b], r[b][c], y[c]);
          yu[c] = fma(l[b], r[b][3 + c], yu[c]);
          yv[c] = fma(d, r[b][c], yv[c]);
        }
      }
      const double n0 = yu[1] * yv[2] - yu[2] * yv[1], n1 = yu[2] * yv[0] - yu[0] * yv[2],
                   n2 = yu[0] * yv[1] - yu[1] * yv[0];
      const double d0 = x[0] - y[0], d1 = x[1] - y[1], d2 = x[2] - y[2];
      // (held finite: beyond, 1/r^3 is 0 in either form)
      const double ri = rsqrt_h3(fmin(d0 * d0 + d1 * d1 + d2 * d2, 1e300));
      const double kv = cw * wv[jv] * (d0 * n0 + d1 * n1 + d2 * n2) * (ri * ri * ri);
#pragma unroll
      for (int b = 0; b < P; ++b) tb[b] = fma(kv, l[b], tb[b]);
    }
  wave_sync();
#pragma unroll
  for (int b = 0; b < P; ++b) T[lane * R + b] = tb[b];
  wave_sync();
  // the groups' sums, in order, into group 0's rows
  for (int e = lane; e < P * nu; e += 64) {
    const int b = e % P, i = e / P;
    double s = T[i * R + b];
    for (int j = 1; j < G; ++j) s += T[(j * nu + i) * R + b];
    T[i * R + b] = s;
  }
  wave_sync();
#pragma unroll
  for (int i = 0; i < (P * P + 63) / 64; ++i) {
    const int ip = lane + 64 * i;
    if (ip < P * P) {
      const int a = ip % P, b = ip / P;
      for (int j = 0; j < nu; ++j) acc[i] = fma(lu[j * R + a], T[j * R + b], acc[i]);
    }
  }
  wave_sync();
}

template <int P>
__global__ void __launch_bounds__(256, P <= 8 ? 3 : 1) closepanel_kernel(CpArgs A) {
  __shared__ double cur[kCpCur][2], leaf[kCpCur][2], pts[5 * kCpBatch][3];
  __shared__ int split[kCpCur], wcnt[4][2];
  extern __shared__ double sh[];
  double *ssx = sh, *W = ssx + 3 * P * P + (threadIdx.x >> 6) * cp_wave_doubles<P>(A.qu, A.qv);
  const int k = blockIdx.x, part = blockIdx.y, nparts = gridDim.y, q = A.q, qu = A.qu, qv = A.qv;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const double x[3] = {A.tx[3 * (size_t)k], A.tx[3 * (size_t)k + 1], A.tx[3 * (size_t)k + 2]};
  for (int i = tid; i < 3 * P * P; i += 256) ssx[i] = A.sx[i];
  if (tid == 0) cur[0][0] = cur[0][1] = -1.0;
  double acc[(P * P + 63) / 64] = {};
  int ncur = 1, nleaf = 0;
  bool bad = false;
  double s = 2.0;
  __syncthreads();
  for (int depth = 0; ncur > 0; ++depth, s *= 0.5) {
    // split while the target is within kCpEta diameters of the cell's centre image
    for (int base = 0; base < ncur; base += kCpBatch) {
      const int c = base + tid / 5, pt = tid % 5;  // points: the centre, then the corners
      if (tid < 5 * kCpBatch && c < ncur) {
        const double du = pt == 0 ? 0.5 * s : ((pt & 1) ? 0.0 : s), dv = pt == 0 ? 0.5 * s : (pt > 2 ? s : 0.0);
        cp_point<P>(A, ssx, cur[c][0] + du, cur[c][1] + dv, pts[tid]);
      }
      __syncthreads();
      if (tid < kCpBatch && base + tid < ncur) {
        const double(*y)[3] = pts + 5 * tid;
        double diam2 = 0.0;
        for (int i = 1; i < 5; ++i)
          for (int j = i + 1; j < 5; ++j) {
            const double d0 = y[i][0] - y[j][0], d1 = y[i][1] - y[j][1], d2 = y[i][2] - y[j][2];
            diam2 = fmax(diam2, d0 * d0 + d1 * d1 + d2 * d2);
          }
        const double e0 = x[0] - y[0][0], e1 = x[1] - y[0][1], e2 = x[2] - y[0][2];
        split[base + tid] =
            (depth < kCpMaxDepth && e0 * e0 + e1 * e1 + e2 * e2 < kCpEta * kCpEta * diam2) ? 1 : 0;
      }
      __syncthreads();
    }
    // the next level's cells, and this part's leaves of this level (every
    // nparts-th leaf of the tree), both in cell order
    const bool in = tid < ncur, sp = in && split[tid] != 0;
    const double u0 = in ? cur[tid][0] : 0.0, v0 = in ? cur[tid][1] : 0.0;
    const unsigned long long bs = __ballot(sp), bl = __ballot(in && !sp), below = (1ull << lane) - 1ull;
    if (lane == 0) {
      wcnt[wv][0] = __popcll(bs);
      wcnt[wv][1] = __popcll(bl);
    }
    __syncthreads();
    int ns = 0, nl = 0, rs = __popcll(bs & below), rl = __popcll(bl & below);
    for (int w = 0; w < 4; ++w) {
      if (w == wv) {
        rs += ns;
        rl += nl;
      }
      ns += wcnt[w][0];
      nl += wcnt[w][1];
    }
    const int first = ((part - nleaf) % nparts + nparts) % nparts;  // rank of this part's first leaf
    if (4 * ns > kCpCur || nleaf + nl > kCpLeaves) bad = true;
    const int room = min(nl, max(0, kCpLeaves - nleaf));
    if (sp && 4 * rs + 4 <= kCpCur) {
      const double h = 0.5 * s;
      for (int j = 0; j < 4; ++j) {
        cur[4 * rs + j][0] = u0 + ((j & 1) ? h : 0.0);
        cur[4 * rs + j][1] = v0 + ((j & 2) ? h : 0.0);
      }
    }
    if (in && !sp && rl < room && rl >= first && (rl - first) % nparts == 0) {
      leaf[(rl - first) / nparts][0] = u0;
      leaf[(rl - first) / nparts][1] = v0;
    }
    const int mine = room > first ? (room - first + nparts - 1) / nparts : 0;
    ncur = 4 * min(ns, kCpCur / 4);
    nleaf += room;
    __syncthreads();
    for (int i = wv; i < mine; i += 4)
      for (int iv = 0; iv < q; iv += qv)
        for (int iu = 0; iu < q; iu += qu)
          cp_block<P>(A, W, x, leaf[i][0], leaf[i][1], 0.5 * s, iu, min(qu, q - iu), iv, min(qv, q - iv), acc);
    __syncthreads();
  }
  if (tid == 0 && bad) atomicOr(A.flag, 1);
  // the four waves' sums, in order
  double* red = ssx + 3 * P * P;
#pragma unroll
  for (int i = 0; i < (P * P + 63) / 64; ++i)
    if (lane + 64 * i < P * P) red[wv * P * P + lane + 64 * i] = acc[i];
  __syncthreads();
  for (int ip = tid; ip < P * P; ip += 256)
    A.part[((size_t)part * P * P + ip) * A.m + k] =
        (red[ip] + red[P * P + ip]) + (red[2 * P * P + ip] + red[3 * P * P + ip]);
}

// parts 1.. added into part 0
__global__ void __launch_bounds__(256) closepanel_sum_kernel(size_t n, int nparts, double* part) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  double v = part[i];
  for (int s = 1; s < nparts; ++s) v += part[s * n + i];
  part[i] = v;
}

// Parts per target: about 2,048 workgroups, two rounds of what the chip holds, so
// that uneven targets even out; more parts only repeat the tree.  Measured at order
// 8 (20, 100, 300, 777, 2,000 targets) with one part 4.9, 5.0, 5.9, 8.2 and 15.8 ms a
// call, with the 10, 10, 7, 3 and 2 parts chosen here 1.04, 1.80, 3.4, 6.8 and 13.8, with
// 16 parts 0.99, 1.83, 4.1, 9.6 and 23.9.
int cp_parts(int64_t m) { return (int)std::min<int64_t>(10, (2048 + m - 1) / m); }

template <int P>
void cp_launch(const CpArgs& A, int nparts) {
  const size_t lds = sizeof(double) * (3 * P * P + 4 * std::max(cp_wave_doubles<P>(A.qu, A.qv), P * P));
  HIPCHK(hipFuncSetAttribute((const void*)closepanel_kernel<P>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(closepanel_kernel<P>, dim3((unsigned)A.m, nparts), dim3(256), lds, 0, A);
}

}  // namespace
}  // namespace qol

using namespace qol;

extern "C" void qol_lap3ddlp_closepanel_mex_(const int64_t* m_tgt, const double* t_x, const int64_t* npat,
                                             const double* s_x, const int64_t* order, const int64_t* ref,
                                             const double* if_adapt_d, double* Ac) {
  try {
    const int64_t p = *order, m = *m_tgt, h = p * p;
    if (p < 2 || p > kCpMaxP) throw std::runtime_error("qol_lap3ddlp_closepanel_mex_: order must be 2..16");
    if (*npat != h) throw std::runtime_error("qol_lap3ddlp_closepanel_mex_: npat must be order^2");
    // the reference implements the adaptive moments only (lap3d_close_mod.f90:234-245)
    if (*if_adapt_d == 0.0) throw std::runtime_error("qol_lap3ddlp_closepanel_mex_: if_adapt = false is not implemented "
                                                     "(as in the reference)");
    if (m < 0) throw std::runtime_error("qol_lap3ddlp_closepanel_mex_: m_tgt must be non-negative");
    if (m == 0) { set_status(0); return; }
    const int q = (int)(2 * p + 2 * (*ref > 0 ? *ref : 1));
    std::vector<double> t(p), w(p), wb(p), gq(q), gw(q);
    gl_nodes(p, t.data(), w.data(), nullptr);
    gl_nodes(q, gq.data(), gw.data(), nullptr);
    for (int64_t j = 0; j < p; ++j) {
      double pr = 1.0;
      for (int64_t k = 0; k < p; ++k)
        if (k != j) pr *= t[j] - t[k];
      wb[j] = 1.0 / pr;
    }
    const int parts = cp_parts(m);
    // one upload: nodes, weights, patch and targets
    std::vector<double> in;
    for (const std::vector<double>* v : {&t, &wb, &gq, &gw}) in.insert(in.end(), v->begin(), v->end());
    in.insert(in.end(), s_x, s_x + 3 * h);
    in.insert(in.end(), t_x, t_x + 3 * m);
    DevBuf d_in, d_part;
    d_in.alloc(sizeof(double) * (in.size() + 1));
    d_part.alloc(sizeof(double) * (size_t)parts * m * h);
    in.push_back(0.0);  // the flag
    HIPCHK(hipMemcpy(d_in.ptr, in.data(), sizeof(double) * in.size(), hipMemcpyHostToDevice));
    const double* di = (const double*)d_in.ptr;
    const int nbu = (q + kCpQU - 1) / kCpQU, nbv = (q + kCpQV - 1) / kCpQV;  // equal blocks
    CpArgs A{(int)p, q, (int)m, (q + nbu - 1) / nbu, (q + nbv - 1) / nbv, di, di + p, di + 2 * p, di + 2 * p + q, di + 2 * p + 2 * q,
             di + 2 * p + 2 * q + 3 * h, (double*)d_part.ptr, (int*)((double*)d_in.ptr + in.size() - 1)};
    switch (p) {
#define QOL_CP(P_) case P_: cp_launch<P_>(A, parts); break;
      QOL_CP(2) QOL_CP(3) QOL_CP(4) QOL_CP(5) QOL_CP(6) QOL_CP(7) QOL_CP(8) QOL_CP(9) QOL_CP(10) QOL_CP(11)
      QOL_CP(12) QOL_CP(13) QOL_CP(14) QOL_CP(15) QOL_CP(16)
#undef QOL_CP
    }
    if (parts > 1)
      hipLaunchKernelGGL(closepanel_sum_kernel, dim3((unsigned)(((size_t)m * h + 255) / 256)), dim3(256), 0, 0,
                         (size_t)m * h, parts, (double*)d_part.ptr);
    HIPCHK(hipGetLastError());
    int flag = 0;
    HIPCHK(hipMemcpy(&flag, A.flag, sizeof(int), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(Ac, d_part.ptr, sizeof(double) * (size_t)m * h, hipMemcpyDeviceToHost));
    if (flag) throw std::runtime_error("qol_lap3ddlp_closepanel_mex_: a target's quadrature tree passed its size limit");
    set_status(0);
  } catch (const std::exception& e) {
    set_error(e.what());
    set_status(1);
  }
}
