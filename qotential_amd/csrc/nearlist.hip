// Near list by the reference's ball rule, CSR by panel with targets ascending.
//
// Reference: stellarator_grf_core_mod.f90:652-695 (count, then fill) and
// test/stellarator_bench.f90:88-94: ball centre = mean of the panel's nodes,
// radius 1.75*sqrt(sum sw), target kept when |x - c|^2 < r^2.  With a diameter
// factor f > 0 the radius is f h instead, h the largest distance between the
// corners of the panel's interpolant (the "radius 2h" near list, f = 2; h as the
// target generator defines the patch diameter).
// Brute force over (panel, target) like the reference, behind a test of groups of
// panels, and the fill keeps ascending target order with wavefront ballots so the
// CSR is bit-identical to the serial loop.
#include "qol_kernels.h"

namespace qol {

constexpr int kNearG = 4;  // groups of 16 panels a wave tests
constexpr int kNearB = 4;  // balls a wave tests between two loads

// ball[k] = (c0, c1, c2, r^2), summed in the reference's order; corner: the 3 x h
// rows interpolating a panel at its corners (used when diam > 0)
__global__ void nearlist_prep_kernel(int npan, int h, const double* __restrict__ sx, const double* __restrict__ sw,
                                     const double* __restrict__ corner, double diam, double* __restrict__ ball) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= npan) {  // up to whole sets of 64: nothing lies inside
    for (int d = 0; d < 4; ++d) ball[4 * k + d] = 0.0;
    return;
  }
  double q0 = 0.0, q1 = 0.0, q2 = 0.0, s = 0.0;
  for (int i = 0; i < h; ++i) {
    const size_t g = (size_t)k * h + i;
    q0 += sx[3 * g];
    q1 += sx[3 * g + 1];
    q2 += sx[3 * g + 2];
  }
  for (int i = 0; i < h; ++i) s += sw[(size_t)k * h + i];
  double qr = 1.75 * sqrt(s);
  if (diam > 0.0) {
    double v[3][3];
    for (int c = 0; c < 3; ++c)
      for (int d = 0; d < 3; ++d) {
        double a = 0.0;
        for (int i = 0; i < h; ++i) a += corner[c * h + i] * sx[3 * ((size_t)k * h + i) + d];
        v[c][d] = a;
      }
    double hd = 0.0;
    for (int a = 0; a < 3; ++a)
      for (int b = a + 1; b < 3; ++b) {
        const double e0 = v[a][0] - v[b][0], e1 = v[a][1] - v[b][1], e2 = v[a][2] - v[b][2];
        hd = fmax(hd, sqrt(e0 * e0 + e1 * e1 + e2 * e2));
      }
    qr = diam * hd;
  }
  ball[4 * k] = q0 / (double)h;
  ball[4 * k + 1] = q1 / (double)h;
  ball[4 * k + 2] = q2 / (double)h;
  ball[4 * k + 3] = qr * qr;
}

__device__ __forceinline__ bool in_ball(const double* b, double x0, double x1, double x2) {
  const double d0 = x0 - b[0], d1 = x1 - b[1], d2 = x2 - b[2];
  return d0 * d0 + d1 * d1 + d2 * d2 < b[3];
}

// One wave per 64 panels (lane = panel) and segment of `seg` targets: counts of the
// segment (part[segment][panel], and added to count), or with FILL the targets
// themselves from offs[panel] plus the counts of the earlier segments.
//
// Bound by the vector units (a test is 9 double operations; all pairs took 476 + 587 us
// for 14,250 panels x 50,000 targets), and most pairs are far apart.  So a target is
// first tested against a ball around the balls of 16 consecutive panels, widened beyond
// any rounding of either test, and targets inside wait in LDS until 64 of them fill the
// wave for the 16 panels' own tests: 1/16 of the tests plus those of the candidates, in
// the targets' order.  A not-a-number ball or target passes the first test and fails the
// second.  Segments and 64-thread workgroups because the fill's serial walk over all
// targets left most of the chip idle.  Panels in no spatial order leave their groups'
// balls so large that most targets are candidates: all pairs are tested then, so the
// tests themselves have to run at the vector rate, four balls at a time from scalar
// registers with one branch (ball by ball, each waiting for its own load, the kernel was
// slower on such panels than all pairs by the kernel before it).  14,250 panels x 50,000 targets: 52 +
// 63 us, panels in random order 292 + 320 (ball by ball 79 + 84 and 694 + 662); 2,400 x
// 20,011: 121 + 242 to 18 + 24.
template <bool FILL>
__global__ void __launch_bounds__(64) nearlist_kernel(int npan, int nt, int seg, const double* __restrict__ tx,
                                                      const double* __restrict__ ball, int* __restrict__ part,
                                                      int* __restrict__ count, const int* __restrict__ offs,
                                                      int* __restrict__ idx) {
  typedef const __attribute__((address_space(4))) double* const_ptr;  // scalar loads
  __shared__ int cand[kNearG][128];
  const int lane = threadIdx.x, k0 = blockIdx.x * 64, k = min(k0 + lane, npan - 1);
  const int t_lo = blockIdx.y * seg, t_hi = min(nt, t_lo + seg);
  // the ball around this lane's group of 16 (panels past the last repeat it)
  double bc[kNearG][4];
  {
    double c[3], m[3], r = sqrt(ball[4 * (size_t)k + 3]), d2 = 0.0;
    for (int d = 0; d < 3; ++d) m[d] = c[d] = ball[4 * (size_t)k + d];
    for (int o = 1; o < 16; o <<= 1)
      for (int d = 0; d < 3; ++d) m[d] += __shfl_xor(m[d], o);
    for (int d = 0; d < 3; ++d) {
      m[d] *= 1.0 / 16.0;
      d2 += (c[d] - m[d]) * (c[d] - m[d]);
    }
    r += sqrt(d2);
    for (int o = 1; o < 16; o <<= 1) {
      const double u = __shfl_xor(r, o);
      r = u > r || u != u ? u : r;  // not-a-number wins
    }
    for (int g = 0; g < kNearG; ++g) {
      for (int d = 0; d < 3; ++d) bc[g][d] = __shfl(m[d], 16 * g);
      const double rg = __shfl(r, 16 * g);
      bc[g][3] = rg * rg * (1.0 + 1e-9) + 1e-290;
    }
  }
  int held[kNearG] = {}, acc = 0;
  if (FILL) {
    acc = offs[k];
#pragma unroll 4
    for (int y = 0; y < (int)blockIdx.y; ++y) acc += part[(size_t)y * npan + k];
  }
  // the tests of group g's 16 panels on target t of the lanes in `on`, kNearB balls at a
  // time, the next ones' scalar loads under way meanwhile
  auto test_lanes = [&](int g, uint64_t on, int t, double x0, double x1, double x2) {
    const const_ptr B = (const_ptr)(uintptr_t)(ball + 4 * (size_t)(k0 + 16 * g));
    double c[4 * kNearB], next[4 * kNearB];
#pragma unroll
    for (int i = 0; i < 4 * kNearB; ++i) next[i] = B[i];
#pragma unroll 1
    for (int q0 = 0; q0 < 16; q0 += kNearB) {
#pragma unroll
      for (int i = 0; i < 4 * kNearB; ++i) {
        c[i] = next[i];
        next[i] = B[4 * min(q0 + kNearB, 16 - kNearB) + i];
      }
      uint64_t b[kNearB], any = 0;
#pragma unroll
      for (int u = 0; u < kNearB; ++u) {
        const double d0 = x0 - c[4 * u], d1 = x1 - c[4 * u + 1], d2 = x2 - c[4 * u + 2];
        b[u] = __ballot(d0 * d0 + d1 * d1 + d2 * d2 < c[4 * u + 3]) & on;
        any |= b[u];
      }
      if (any == 0) continue;
#pragma unroll
      for (int u = 0; u < kNearB; ++u) {
        const int to = 16 * g + q0 + u, base = __builtin_amdgcn_readlane(acc, to);
        if (FILL && (b[u] >> lane & 1ull)) idx[base + __popcll(b[u] & ((1ull << lane) - 1ull))] = t;
        acc += lane == to ? __popcll(b[u]) : 0;
      }
    }
  };
  // the same on its first n candidates
  auto test = [&](int g, int n) {
    const int t = cand[g][min(lane, n - 1)];
    const double* y = tx + 3 * (size_t)t;
    test_lanes(g, n < 64 ? (1ull << n) - 1ull : ~0ull, t, y[0], y[1], y[2]);
  };
  double x[3];
  auto load = [&](int t) {
    const size_t i = 3 * (size_t)min(t, nt - 1);
    for (int d = 0; d < 3; ++d) x[d] = tx[i + d];
  };
  load(t_lo + lane);
  for (int t0 = t_lo; t0 < t_hi; t0 += 64) {
    const int t = t0 + lane;
    const double x0 = x[0], x1 = x[1], x2 = x[2];
    load(t + 64);
#pragma unroll
    for (int g = 0; g < kNearG; ++g) {
      const double e0 = x0 - bc[g][0], e1 = x1 - bc[g][1], e2 = x2 - bc[g][2];
      const bool keep = t < t_hi && !(fma(e0, e0, fma(e1, e1, e2 * e2)) > bc[g][3]);
      const uint64_t b = __ballot(keep);
      if (b == 0) continue;
      if (keep) cand[g][held[g] + __popcll(b & ((1ull << lane) - 1ull))] = t;
      held[g] += __popcll(b);
      __syncthreads();
      if (held[g] < 64) continue;
      test(g, 64);
      held[g] -= 64;
      const int rest = cand[g][64 + lane];
      __syncthreads();
      cand[g][lane] = rest;
    }
  }
  __syncthreads();
  for (int g = 0; g < kNearG; ++g)
    if (held[g] > 0) test(g, held[g]);
  if (!FILL && k0 + lane < npan) {
    part[(size_t)blockIdx.y * npan + k] = acc;
    if (acc) atomicAdd(&count[k], acc);
  }
}

// targets of a segment: a multiple of 64, so that about 8,192 waves run
static int near_segment(int npan, int nt) {
  const int sets = (npan + 63) / 64, most = std::max(1, std::min(64, 8192 / sets));
  const int chunks = (nt + 63) / 64;
  return 64 * std::max(1, (chunks + most - 1) / most);
}

int nearlist_parts(int npan, int nt) { return nt > 0 ? (nt - 1) / near_segment(npan, nt) + 1 : 0; }

void launch_nearlist(bool fill, int npan, int nt, const double* tx, const double* ball, int* part, int* count,
                     const int* offs, int* idx, hipStream_t s) {
  const dim3 grid((npan + 63) / 64, nearlist_parts(npan, nt));
  hipLaunchKernelGGL(fill ? nearlist_kernel<true> : nearlist_kernel<false>, grid, dim3(64), 0, s, npan, nt,
                     near_segment(npan, nt), tx, ball, part, count, offs, idx);
}

// exclusive scan of n ints into out[0..n] with a single workgroup of 1024 threads,
// 4,096 at a time, the next ones loaded ahead of the scan (a thread's own run of n/1024
// took 87 us for 50,000, this 30)
__global__ void __launch_bounds__(1024) scan_kernel(const int* __restrict__ in, int n, int* __restrict__ out) {
  int v[4], carry = 0;
  auto load = [&](int i0) {
    for (int u = 0; u < 4; ++u) v[u] = i0 + u < n ? in[i0 + u] : 0;
  };
  load(4 * threadIdx.x);
  for (int base = 0; base < n; base += 4096) {
    const int i0 = base + 4 * threadIdx.x;
    int w[4], total;
    for (int u = 0; u < 4; ++u) w[u] = v[u];
    load(i0 + 4096);
    int acc = carry + block_scan_1024(w[0] + w[1] + w[2] + w[3], &total);
    for (int u = 0; u < 4; ++u) {
      if (i0 + u < n) out[i0 + u] = acc;
      acc += w[u];
    }
    carry += total;
    __syncthreads();  // the scan's shared sums are read
  }
  if (threadIdx.x == 0) out[n] = carry;
}


// ---------------------------------------------------------------------------
// The same near list through a uniform grid of cells no smaller than the
// largest panel ball (the spatial search the reference's MATLAB caller does
// with a k-d tree, test/torus_fmm3dbie_rrq_comparison.m:81-99): targets are
// binned by cell, each panel tests only the targets of the cells its ball's
// bounding box covers (at most 3 x 3 x 3), and each panel's list is sorted, so
// the CSR equals the brute-force one bit for bit (the same in_ball test).

__device__ __forceinline__ int grid_coord(double x, double lo, double inv_c, int n) {
  const double f = floor((x - lo) * inv_c);
  return f < 0.0 ? 0 : (f > (double)(n - 1) ? n - 1 : (int)f);
}

__global__ void grid_bin_kernel(int nt, const double* __restrict__ tx, GridArgs G, int* __restrict__ cell_of,
                                int* __restrict__ cell_count) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nt) return;
  const int i = grid_coord(tx[3 * (size_t)t], G.lo[0], G.inv_c, G.n[0]);
  const int j = grid_coord(tx[3 * (size_t)t + 1], G.lo[1], G.inv_c, G.n[1]);
  const int k = grid_coord(tx[3 * (size_t)t + 2], G.lo[2], G.inv_c, G.n[2]);
  const int c = (k * G.n[1] + j) * G.n[0] + i;
  cell_of[t] = c;
  atomicAdd(&cell_count[c], 1);
}

__global__ void grid_scatter_kernel(int nt, const int* __restrict__ cell_of, const int* __restrict__ cell_start,
                                    int* __restrict__ cursor, int* __restrict__ cell_targets) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nt) return;
  const int c = cell_of[t];
  cell_targets[cell_start[c] + atomicAdd(&cursor[c], 1)] = t;
}

// one wave per panel; fill == 0 counts, fill == 1 writes the hits (unordered)
__global__ void __launch_bounds__(64) grid_panel_kernel(int npan, const double* __restrict__ ball, GridArgs G,
                                                        const int* __restrict__ cell_start,
                                                        const int* __restrict__ cell_targets,
                                                        const double* __restrict__ tx, int fill,
                                                        int* __restrict__ count, const int* __restrict__ offs,
                                                        int* __restrict__ cursor, int* __restrict__ idx) {
  const int k = blockIdx.x;
  if (k >= npan) return;
  const double* b = ball + 4 * (size_t)k;
  const double r = sqrt(b[3]);
  int lo[3], hi[3];
  for (int d = 0; d < 3; ++d) {
    lo[d] = grid_coord(b[d] - r, G.lo[d], G.inv_c, G.n[d]);
    hi[d] = grid_coord(b[d] + r, G.lo[d], G.inv_c, G.n[d]);
  }
  int cnt = 0;
  for (int kk = lo[2]; kk <= hi[2]; ++kk)
    for (int jj = lo[1]; jj <= hi[1]; ++jj)
      for (int ii = lo[0]; ii <= hi[0]; ++ii) {
        const int c = (kk * G.n[1] + jj) * G.n[0] + ii;
        for (int s = cell_start[c] + threadIdx.x; s < cell_start[c + 1]; s += 64) {
          const int t = cell_targets[s];
          if (in_ball(b, tx[3 * (size_t)t], tx[3 * (size_t)t + 1], tx[3 * (size_t)t + 2])) {
            if (fill) idx[offs[k] + atomicAdd(&cursor[k], 1)] = t;
            else ++cnt;
          }
        }
      }
  if (!fill) {
    for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o);
    if (threadIdx.x == 0) count[k] = cnt;
  }
}

// each panel's list in ascending target order: bitonic sort in LDS up to
// kSortMax entries, one thread's insertion sort beyond
constexpr int kSortMax = 4096;
__global__ void __launch_bounds__(256) segment_sort_kernel(int npan, const int* __restrict__ offs, int* __restrict__ idx) {
  __shared__ int s[kSortMax];
  const int k = blockIdx.x;
  const int a = offs[k], n = offs[k + 1] - a;
  if (n <= 1) return;
  if (n > kSortMax) {
    if (threadIdx.x == 0)
      for (int i = a + 1; i < a + n; ++i) {
        const int v = idx[i];
        int j = i - 1;
        while (j >= a && idx[j] > v) { idx[j + 1] = idx[j]; --j; }
        idx[j + 1] = v;
      }
    return;
  }
  int m = 1;
  while (m < n) m <<= 1;
  for (int i = threadIdx.x; i < m; i += blockDim.x) s[i] = i < n ? idx[a + i] : 0x7fffffff;
  __syncthreads();
  for (int size = 2; size <= m; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < m; i += blockDim.x) {
        const int j = i ^ stride;
        if (j > i) {
          const bool up = (i & size) == 0;
          const int x = s[i], y = s[j];
          if ((x > y) == up) { s[i] = y; s[j] = x; }
        }
      }
      __syncthreads();
    }
  for (int i = threadIdx.x; i < n; i += blockDim.x) idx[a + i] = s[i];
}

}  // namespace qol
