// Near-correction apply, deterministic scatter and COO triplets.
//
// Reference: naive block + apply   stellarator_grf_core_mod.f90:847-870
//            fixed-order scatter   stellarator_grf_core_mod.f90:895-899
//            COO triplets          lap3d_close_mod.f90:935-956
#include <algorithm>

#include "qol_kernels.h"

namespace qol {

// naive S and D entries of a target against one panel node (zero at coincident points)
__device__ __forceinline__ void naive_entries(double x0, double x1, double x2, const double* __restrict__ y,
                                              const double* __restrict__ n, double w, double pi4inv, double& an,
                                              double& dn) {
  const double dx = x0 - y[0], dy = x1 - y[1], dz = x2 - y[2];
  const double rr = dx * dx + dy * dy + dz * dz;
  an = 0.0;
  dn = 0.0;
  if (rr > 1.0e-28) {
    const double ir = rsqrt_nr(rr);
    an = pi4inv * w * ir;
    dn = an * (dx * n[0] + dy * n[1] + dz * n[2]) * (ir * ir);
  }
}

// val(pair) = sum_i (S - S_naive)_i ubn_i - (K - K_naive)_i ub_i over the panel's h
// nodes, for pairs pair_of(0 .. cnt-1), which come panel by panel: kAP pairs per
// workgroup, kAL lanes each (nodes part, part + kAL, ..., the parts summed in a fixed
// order).
//
// Bound by the loads of a node's nine values for every pair rather than by the weights
// (16 bytes a node): the panels' nodes are therefore gathered in LDS once per
// workgroup, as many as `slots`, and only pairs of further panels read them from
// memory.  Eight lanes read a row 64 bytes at a time.  1.62M level pairs of order 8 (0.93
// GB of weights): 0.45 to 0.33 ms; 30,000 targets of order 12: 158 to 100 us; all pairs
// of 50,000 targets of order 8: 121 to 81.  With four lanes and every node from memory,
// eight lanes alone gave 0.44, sixteen 0.51.
//
// Up to order 5 (15 nodes) eight lanes leave too many idle in their one or two rounds, and four
// take a pair: 1.97M pairs on 3,570 panels with eight and with four lanes take (with the
// targets' sums) 134 and 93 us at order 2, 137 and 121 at 3, 228 and 149 at 4, 237 and 189
// at 5; at order 6 253 and 274.
constexpr int kAT = 256, kRec = 10;  // doubles per node: x, n, w, ubn, ub, and one for the banks

struct ApplyArgs {
  const int *tidx, *ppanel;
  const double *tx, *sx, *snx, *sw, *ub, *ubn, *wout;
  double* val;
};

template <int kAL, class F>
__device__ __forceinline__ void apply_pairs(int cnt, int h, int slots, const ApplyArgs& A, F&& pair_of) {
  constexpr int kAP = kAT / kAL;
  static_assert(kAP <= 64, "one wave finds the workgroup's panels");
  extern __shared__ __align__(16) double rec[];  // [slots][h][kRec]
  __shared__ int pan[kAP], slot[kAP], npan;
  const int t0 = blockIdx.x * kAP;
  if (t0 >= cnt) return;
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x, k = A.ppanel[pair_of(min(t0 + (lane & (kAP - 1)), cnt - 1))];
    const int before = __shfl_up(k, 1, 64);
    const bool first = lane < kAP && (lane == 0 || k != before);
    const uint64_t m = __ballot(first);
    if (lane < kAP) slot[lane] = __popcll(m & ((2ull << lane) - 1ull)) - 1;
    if (first) pan[__popcll(m & ((1ull << lane) - 1ull))] = k;
    if (lane == 0) npan = __popcll(m);
  }
  __syncthreads();
  const int ns = min(npan, slots);
  for (int e = threadIdx.x; e < ns * h; e += kAT) {
    const size_t g = (size_t)pan[e / h] * h + e % h;
    double* r = rec + (size_t)kRec * e;
    for (int d = 0; d < 3; ++d) {
      r[d] = A.sx[3 * g + d];
      r[3 + d] = A.snx[3 * g + d];
    }
    r[6] = A.sw[g];
    r[7] = A.ubn[g];
    r[8] = A.ub[g];
  }
  __syncthreads();
  const int q = threadIdx.x / kAL, part = threadIdx.x % kAL;
  const bool live = t0 + q < cnt;
  const int j = pair_of(live ? t0 + q : cnt - 1), t = A.tidx[j];
  const double x0 = A.tx[3 * (size_t)t], x1 = A.tx[3 * (size_t)t + 1], x2 = A.tx[3 * (size_t)t + 2];
  const double* w = A.wout + (size_t)j * 2 * h;
  const double pi4inv = 1.0 / (16.0 * atan(1.0));
  double acc = 0.0, an, dn;
  if (slot[q] < ns) {
    const double* r = rec + (size_t)kRec * h * slot[q];
#pragma unroll 2
    for (int i = part; i < h; i += kAL) {
      const double* n = r + kRec * i;
      naive_entries(x0, x1, x2, n, n + 3, n[6], pi4inv, an, dn);
      acc = acc + (w[i] - an) * n[7] - (w[h + i] - dn) * n[8];
    }
  } else {
    const size_t k = (size_t)pan[slot[q]] * h;
    for (int i = part; i < h; i += kAL) {
      const size_t g = k + i;
      naive_entries(x0, x1, x2, A.sx + 3 * g, A.snx + 3 * g, A.sw[g], pi4inv, an, dn);
      acc = acc + (w[i] - an) * A.ubn[g] - (w[h + i] - dn) * A.ub[g];
    }
  }
#pragma unroll
  for (int o = 1; o < kAL; o <<= 1) acc = acc + __shfl_xor(acc, o, 64);
  if (live && part == 0) A.val[j] = acc;
}

// Weights of the pairs labelled 0 (the learned selector found the panel's own
// nodes accurate enough): the naive h-node entries themselves, formed exactly
// as the apply forms them, so each such pair's correction is exactly zero.
__global__ void __launch_bounds__(256) naive_fill_kernel(int nnz, int h, const int8_t* __restrict__ label,
                                                         const int* __restrict__ tidx, const int* __restrict__ ppanel,
                                                         const double* __restrict__ tx, const double* __restrict__ sx,
                                                         const double* __restrict__ snx,
                                                         const double* __restrict__ sw, double* __restrict__ wout,
                                                         double* __restrict__ val) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nnz || label[j] != 0) return;
  const double pi4inv = 1.0 / (16.0 * atan(1.0));
  const int t = tidx[j], k = ppanel[j];
  const double x0 = tx[3 * (size_t)t], x1 = tx[3 * (size_t)t + 1], x2 = tx[3 * (size_t)t + 2];
  double* w = wout + (size_t)j * 2 * h;
  for (int i = 0; i < h; ++i) {
    const size_t g = (size_t)k * h + i;
    naive_entries(x0, x1, x2, sx + 3 * g, snx + 3 * g, sw[g], pi4inv, w[i], w[h + i]);
  }
  if (val) val[j] = 0.0;
}

template <int kAL>
__global__ void __launch_bounds__(kAT) naive_apply_kernel(int nnz, int h, int slots, ApplyArgs A) {
  apply_pairs<kAL>(nnz, h, slots, A, [](int t) { return t; });
}

// The same for the pairs of the per-label lists first..last (lists concatenated in label
// order, lengths ltot), so each part can run as soon as its weights are in
template <int kAL>
__global__ void __launch_bounds__(kAT) naive_apply_list_kernel(const int* __restrict__ lpairs,
                                                               const int* __restrict__ ltot, int first, int last, int h,
                                                               int slots, ApplyArgs A) {
  int base = 0, cnt = 0;
  for (int q = 0; q <= last; ++q) {
    if (q < first) base += ltot[q];
    else cnt += ltot[q];
  }
  apply_pairs<kAL>(cnt, h, slots, A, [&](int t) { return lpairs[base + t]; });
}

// lanes per pair, pairs per workgroup, and the panels it gathers: 24 KB, so that six
// workgroups share a CU
struct ApplyPlan {
  int lanes, pairs, slots;
};
static ApplyPlan apply_plan(int h) {
  const int lanes = h <= 15 ? 4 : 8, pairs = kAT / lanes;
  return {lanes, pairs, std::max(1, std::min(pairs, 24 * 1024 / (kRec * 8 * h)))};
}

void launch_naive_apply(int64_t nnz, int h, const int* tidx, const int* ppanel, const double* tx, const double* sx,
                        const double* snx, const double* sw, const double* ub, const double* ubn, const double* wout,
                        double* val, hipStream_t s) {
  const ApplyPlan P = apply_plan(h);
  hipLaunchKernelGGL(P.lanes == 4 ? naive_apply_kernel<4> : naive_apply_kernel<8>,
                     dim3((unsigned)((nnz + P.pairs - 1) / P.pairs)), dim3(kAT), sizeof(double) * kRec * h * P.slots, s,
                     (int)nnz, h, P.slots, ApplyArgs{tidx, ppanel, tx, sx, snx, sw, ub, ubn, wout, val});
}

void launch_naive_apply_list(int64_t nnz, const int* lpairs, const int* ltot, int first, int last, int h, const int* tidx,
                             const int* ppanel, const double* tx, const double* sx, const double* snx, const double* sw,
                             const double* ub, const double* ubn, const double* wout, double* val, hipStream_t s) {
  const ApplyPlan P = apply_plan(h);
  hipLaunchKernelGGL(P.lanes == 4 ? naive_apply_list_kernel<4> : naive_apply_list_kernel<8>,
                     dim3((unsigned)((nnz + P.pairs - 1) / P.pairs)), dim3(kAT), sizeof(double) * kRec * h * P.slots, s,
                     lpairs, ltot, first, last, h, P.slots,
                     ApplyArgs{tidx, ppanel, tx, sx, snx, sw, ub, ubn, wout, val});
}

// The weights by column, out(j, c - c0) at (c - c0)*nnz + j for nc columns c from c0, from
// rows of m2 = 2h per pair: tiles of 32 x 32 through LDS, so that both sides move whole
// lines and the host, which looped over the rows before, copies finished blocks
__global__ void __launch_bounds__(256) weight_columns_kernel(int nnz, int m2, int c0, int nc,
                                                             const double* __restrict__ wout,
                                                             double* __restrict__ cols) {
  __shared__ double tile[32][33];
  const int j0 = blockIdx.x * 32, d0 = blockIdx.y * 32, x = threadIdx.x & 31, y = threadIdx.x >> 5;
  for (int r = y; r < 32; r += 8)
    if (j0 + r < nnz && d0 + x < nc) tile[r][x] = wout[(size_t)(j0 + r) * m2 + c0 + d0 + x];
  __syncthreads();
  for (int c = y; c < 32; c += 8)
    if (j0 + x < nnz && d0 + c < nc) cols[(size_t)(d0 + c) * nnz + j0 + x] = tile[x][c];
}

// COO triplets of getnearquad_lap_rrq: out = (tcxi(k)-1)*h + (j-1)*m + i (1-based)
__global__ void __launch_bounds__(256) triplet_kernel(int nnz, int h, const int* __restrict__ tidx,
                                                      const int* __restrict__ ppanel, const int* __restrict__ trow,
                                                      const int* __restrict__ offs, const double* __restrict__ tx,
                                                      const double* __restrict__ sx, const double* __restrict__ snx,
                                                      const double* __restrict__ sw, const double* __restrict__ wout,
                                                      int64_t* __restrict__ si, int64_t* __restrict__ sj,
                                                      double* __restrict__ vs, double* __restrict__ vd) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nnz) return;
  const double pi4inv = 1.0 / (16.0 * atan(1.0));
  const int t = tidx[j], k = ppanel[j];
  const int m = offs[k + 1] - offs[k], i = j - offs[k];
  const double x0 = tx[3 * (size_t)t], x1 = tx[3 * (size_t)t + 1], x2 = tx[3 * (size_t)t + 2];
  const double* w = wout + (size_t)j * 2 * h;
  const int row = trow[t];  // 1-based source index of the target, 0 if none
  for (int c = 0; c < h; ++c) {
    const size_t g = (size_t)k * h + c;
    const double dx = x0 - sx[3 * g], dy = x1 - sx[3 * g + 1], dz = x2 - sx[3 * g + 2];
    const double rr = dx * dx + dy * dy + dz * dz;
    double an = 0.0, dn = 0.0;
    if (rr > 1.0e-28) {
      const double r = sqrt(rr);
      an = pi4inv * sw[g] / r;
      dn = pi4inv * sw[g] * (dx * snx[3 * g] + dy * snx[3 * g + 1] + dz * snx[3 * g + 2]) / (r * rr);
    }
    if (row == (int)(g + 1)) { an = 0.0; dn = 0.0; }
    const size_t o = (size_t)offs[k] * h + (size_t)c * m + i;
    si[o] = row;
    sj[o] = (int64_t)g + 1;
    vs[o] = w[c] - an;
    vd[o] = w[h + c] - dn;
  }
}

// target-major pair lists (stable in pair order after the per-target sort)
__global__ void target_count_kernel(int nnz, const int* __restrict__ tidx, int* __restrict__ tcount) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < nnz) atomicAdd(&tcount[tidx[j]], 1);
}

__global__ void target_fill_kernel(int nnz, const int* __restrict__ tidx, const int* __restrict__ toffs,
                                   int* __restrict__ tcur, int* __restrict__ tpairs) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nnz) return;
  const int t = tidx[j];
  const int pos = atomicAdd(&tcur[t], 1);
  tpairs[toffs[t] + pos] = j;
}

// u(t) += val(pairs of t) in pair (= panel) order, starting from the far field
__global__ void target_sum_kernel(int nt, const int* __restrict__ toffs, int* __restrict__ tpairs,
                                  const double* __restrict__ val, double* __restrict__ u) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nt) return;
  const int a = toffs[t], b = toffs[t + 1];
  for (int i = a + 1; i < b; ++i) {  // insertion sort: lists are short
    const int v = tpairs[i];
    int j = i - 1;
    while (j >= a && tpairs[j] > v) { tpairs[j + 1] = tpairs[j]; --j; }
    tpairs[j + 1] = v;
  }
  double acc = u[t];
  for (int i = a; i < b; ++i) acc = acc + val[tpairs[i]];
  u[t] = acc;
}

// ---------------------------------------------------------------------------
// plain copy of n 16-byte words (each read once, written once): the reference
// workload for scaling the HBM byte counters
__global__ void __launch_bounds__(256) hbm_copy_kernel(size_t n, const double2* __restrict__ src,
                                                       double2* __restrict__ dst) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

}  // namespace qol
