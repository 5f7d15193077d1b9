// grad.hip -- gfx950 kernels of the projector's adjoint and of the gradients
// of L(x, s) = 1/2 |shift_s(radon(x)) - b|^2 + lambda TV_eps(x).
//
// adjoint_kernel is pixel-driven and deterministic: each thread owns one
// pixel and, per angle, tests the samples whose bilinear stencil can cover
// it.  Sample (jx, jy) of angle t sits at
//   xr = (c (jx-m) - s (jy-m)) + m,  yr = (s (jx-m) + c (jy-m)) + m
// (tomography/tv_hpc.F90:143-144) and covers the pixels x1..x1+1, y1..y1+1,
// x1 = floor(xr), y1 = floor(yr), when 2 <= x1,y1 <= N-1 (:145-150).  The
// samples covering pixel (px,py) therefore lie in the rotated 2x2 square
// around the inverse rotation q of (px,py); its bounding box holds at most
// 3 x 3 lattice points, and each is tested with the projector's own FP32
// expressions (contraction off), so the weights are exactly the projector's
// and the kernel is its transpose.
//
// The projector's weights (x1+1) - xr and xr - x1 are differences of floats
// within a factor of two of each other (x1 >= 2), hence exact (Sterbenz), and
// equal to 1 - |dx|, dx = xr - px, which is exact too; off the stencil 1 -
// |dx| <= 0.  So a candidate's weight is the product of two differences
// clamped to [0, 1] -- an output modifier, no comparison or select -- and
// the rays of an angle (rows jy) each add (sum of their three candidates'
// weights) x (their sinogram value).  That is 9 full-rate instructions per
// candidate.  The bounds test only bites on the image's rim: pixel 1 is in no
// valid cell, pixel 2 only in x1 = 2 (dx >= 0), pixel N only in x1 = N-1
// (dx < 0); tiles that hold such pixels, and angles at which a tile's samples
// reach jx < 1 or > N (or a window holds an infinity or NaN), take the same
// loop with those tests.  The sinogram
// values of a tile (a window of 32 rays per angle, zero off the detector) are
// staged in LDS for 32 angles at a time.
//
// Bound by VALU issue: about 115 instructions per pixel and angle, 90 of them
// the candidates' weights.  Those depend on the geometry alone, so a workgroup
// takes up to 8 slices of one geometry together (G, side by side in LDS): 3
// products and a sum more per slice.  On MI355X, 16 x 513^2 x 720: 6.7 ms by
// single slices (9.7 with comparisons per candidate and three global loads
// per angle), 2.2 by fours, 1.75 by eights; one 257^2 x 180 130 us (344).
#include "acu_grad.hpp"

#include <algorithm>
#include <map>

namespace acu {
namespace {

template <class Task, int Task::*Begin>
__device__ __forceinline__ int find_by(const Task* tasks, int ntasks, int gb) {
  int lo = 0, hi = ntasks - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tasks[mid].*Begin <= gb) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Sum of v over the workgroup (GR_THREADS), valid in thread 0.
__device__ double block_sum(double v, double* wsum) {
  v = wave_sum_d(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) wsum[wave] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0)
#pragma unroll
    for (int w = 0; w < GR_THREADS / 64; ++w) r += wsum[w];
  __syncthreads();
  return r;
}

static_assert(ADJ_AB == 32, "a bit of a mask per angle");
constexpr int ADJ_W = 32;  // rays staged per angle and tile: 15 (|c| + |s|) + 4 <= 25.3, and one of margin on each side

// One angle's contribution to one pixel.  (X, Y): the pixel relative to the
// midpoint; w: LDS offset (lds_units) of the angle's ray jy = m in P.  CHECK: the rim's and the sweep's bounds (xlo, xhi, ylo, yhi: dx, dy
// allowed in [lo, hi); u0, u1: jx - m allowed in [u0, u1]).
struct AdjPixel {
  float X, Y, px, py, xlo, xhi, ylo, yhi, u0, u1;
};
// one ray of each of G slices, side by side in LDS
template <int G>
struct __attribute__((aligned(G < 4 ? 4 * G : 16))) AdjRay {
  float v[G];
};
template <bool CHECK, int G>
__device__ __forceinline__ void adj_angle(const AdjPixel& g, float s, float c, float hw, float m, float w,
                                          const float* P, float (&blk)[G]) {
#pragma clang fp contract(off)
  // first candidate, relative to the midpoint (integer valued): the margin in
  // hw covers the rounding of this estimate and of the exact positions
  const float ua = ceilf(fmaf(c, g.X, fmaf(s, g.Y, -hw)));
  const float wa = ceilf(fmaf(c, g.Y, fmaf(-s, g.X, -hw)));
  const AdjRay<G>* r = (const AdjRay<G>*)((const char*)P + __float_as_uint(fmaf(wa, lds_units(4 * G), w)));
  const AdjRay<G> rv[3] = {r[0], r[1], r[2]};
  float cu[3], su[3];
  bool uok[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float u = a == 0 ? ua : ua + (float)a;
    cu[a] = c * u;
    su[a] = s * u;
    uok[a] = !CHECK || (u >= g.u0 && u <= g.u1);
  }
  float v[G];
#pragma unroll
  for (int k = 0; k < G; ++k) v[k] = 0.0f;
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    const float wb = b == 0 ? wa : wa + (float)b;
    const float sw = s * wb, cw = c * wb;
    float sum = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float dx = ((cu[a] - sw) + m) - g.px;
      const float dy = ((su[a] + cw) + m) - g.py;
      float wx = __builtin_amdgcn_fmed3f(1.0f - fabsf(dx), 0.0f, 1.0f);
      const float wy = __builtin_amdgcn_fmed3f(1.0f - fabsf(dy), 0.0f, 1.0f);
      if (CHECK) wx = uok[a] && dx >= g.xlo && dx < g.xhi && dy >= g.ylo && dy < g.yhi ? wx : 0.0f;
      sum = a == 0 ? wx * wy : fmaf(wx, wy, sum);
    }
    // CHECK: a ray of infinity or NaN stays out of the pixels it does not cover
#pragma unroll
    for (int k = 0; k < G; ++k) {
      if (!CHECK) v[k] = b == 0 ? rv[b].v[k] * sum : fmaf(rv[b].v[k], sum, v[k]);
      else v[k] = sum > 0.0f ? fmaf(rv[b].v[k], sum, v[k]) : v[k];
    }
  }
#pragma unroll
  for (int k = 0; k < G; ++k) blk[k] += v[k];
}

// One 16 x 16 tile of a task, its n <= G slices together.
template <int G>
__device__ __forceinline__ void adjoint_tile(const AdjTask& tk, int local, AdjRay<G>* __restrict__ P) {
  const int N = tk.N, T = tk.T;
  const float m = tk.mid;
  const int ty = local / tk.ntx, tx = local - ty * tk.ntx;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int px = tx * ADJ_T + tid % ADJ_T + 1;  // 1-based pixel; past the image in the last tiles (not stored)
  const int py = ty * ADJ_T + tid / ADJ_T + 1;
  AdjPixel g;
  g.px = (float)px;
  g.py = (float)py;
  g.X = g.px - m;
  g.Y = g.py - m;
  g.xlo = px == 1 ? 4.0f : px == 2 ? 0.0f : -4.0f;
  g.xhi = px >= N ? 0.0f : 4.0f;
  g.ylo = py == 1 ? 4.0f : py == 2 ? 0.0f : -4.0f;
  g.yhi = py >= N ? 0.0f : 4.0f;
  g.u0 = 1.0f - m;
  g.u1 = (float)N - m;
  const bool rim = tx == 0 || ty == 0 || (tx + 1) * ADJ_T >= N || (ty + 1) * ADJ_T >= N;  // uniform
  // tile corners relative to the midpoint
  const float X0 = (float)(tx * ADJ_T + 1) - m, X1 = X0 + (float)(ADJ_T - 1);
  const float Y0 = (float)(ty * ADJ_T + 1) - m, Y1 = Y0 + (float)(ADJ_T - 1);
  const float margin = 1e-3f + 3e-7f * (float)N;
  const ACU_GLOBAL float* __restrict__ sc = as_global((const float*)tk.sc);
  float acc[G];
#pragma unroll
  for (int k = 0; k < G; ++k) acc[k] = 0.0f;
  for (int t0 = 0; t0 < T; t0 += ADJ_AB) {
    const int na = min(ADJ_AB, T - t0);
    // lane l (mod 32) of every wave holds angle t0 + l: sine, cosine, first
    // ray of the tile's window, and whether a sample can leave 1 <= jx <= N
    const int t = min(t0 + (lane & (ADJ_AB - 1)), T - 1);
    const float hs = sc[2 * t], hc = sc[2 * t + 1];
    const float hh = fabsf(hc) + fabsf(hs) + margin;
    const float ymin = fminf(hc * Y0, hc * Y1) + fminf(-hs * X0, -hs * X1);
    const float xmin = fminf(hc * X0, hc * X1) + fminf(hs * Y0, hs * Y1);
    const float xmax = fmaxf(hc * X0, hc * X1) + fmaxf(hs * Y0, hs * Y1);
    const int lo = (int)floorf((ymin - hh) + m) - 1;
    const float hb = lds_base(4 * G * ((lane & (ADJ_AB - 1)) * ADJ_W + (int)m - lo));  // LDS offset of ray jy = m
    unsigned long long chk = rim ? ~0ull : __ballot(xmin - hh < g.u0 + 1.0f || xmax + hh > g.u1 - 1.0f);
    bool bad = false;
    {
      const int q = tid >> 3, j = tid & 7;  // 8 threads per angle
      const int jy0 = __shfl(lo, q) + j;
      AdjRay<G> v[ADJ_W / 8];
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const ACU_GLOBAL float* row = as_global(tk.sino[i]) + (size_t)min(t0 + q, T - 1) * N;
#pragma unroll
        for (int k = 0; k < ADJ_W / 8; ++k) v[k].v[i] = row[min(max(jy0 + 8 * k, 1), N) - 1];
      }
      if (t0 > 0) __syncthreads();  // the last block's rays are read
#pragma unroll
      for (int k = 0; k < ADJ_W / 8; ++k) {
        const bool on = jy0 + 8 * k >= 1 && jy0 + 8 * k <= N;
        AdjRay<G> u;
#pragma unroll
        for (int i = 0; i < G; ++i) {
          u.v[i] = on ? v[k].v[i] : 0.0f;
          bad = bad || !(fabsf(v[k].v[i]) <= 3.40282347e38f);
        }
        P[q * ADJ_W + j + 8 * k] = u;
      }
    }
    if (__syncthreads_or(bad)) chk = ~0ull;  // uniform
    float blk[G];  // FP32 sums over one block of angles, then into acc
#pragma unroll
    for (int k = 0; k < G; ++k) blk[k] = 0.0f;
    // an angle that is not finite covers no pixel (and has no window in LDS)
    for (unsigned live = (unsigned)__ballot(hh <= 4.0f) & (~0u >> (ADJ_AB - na)); live != 0; live &= live - 1) {
      const int a = __builtin_ctz(live);
      const float s = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hs), a));
      const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hc), a));
      const float hw = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hh), a));
      const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hb), a));
      if ((chk >> a) & 1) adj_angle<true, G>(g, s, c, hw, m, w, &P[0].v[0], blk);
      else adj_angle<false, G>(g, s, c, hw, m, w, &P[0].v[0], blk);
    }
#pragma unroll
    for (int k = 0; k < G; ++k) acc[k] += blk[k];
  }
  if (px <= N && py <= N)
#pragma unroll
    for (int k = 0; k < G; ++k)
      if (k < tk.n) tk.out[k][(size_t)(py - 1) * N + (px - 1)] = acc[k] / (float)N;
}

// W: the most slices of a task.  Each task runs at its own width, so a slice
// without a partner costs what it would in a launch of single slices: 5 equal
// and 20 different slices of 513^2 x 360 (loss and gradients) take 6.5 ms, 25
// different ones 6.95, with every task at the width of the widest 7.85.
// mixed: tasks whose tiles take unequal times, the longest first, go
// round-robin over the XCDs: with contiguous shares of the blocks the XCD of
// the wide tasks is the last (9 equal slices 1.62 ms instead of 1.50, eight
// sizes from 65^2 x 1000 to 600^2 x 90 1.48 instead of 1.19, the 25 slices
// above 6.9).  Others keep neighbouring tiles on one XCD (360^2 x 360 255 us,
// 286 round-robin; 16 different 65^2 x 48 400, 418; 513^2 x 360 397, 393).
template <int W>
__global__ __launch_bounds__(ADJ_T * ADJ_T) void adjoint_kernel(const AdjTask* __restrict__ tasks, int ntasks,
                                                                int nblocks, bool mixed) {
  __shared__ AdjRay<W> P[ADJ_AB * ADJ_W];
  const int gb = mixed ? (int)blockIdx.x : xcd_remap(blockIdx.x, gridDim.x);
  if (gb >= nblocks) return;  // uniform per workgroup
  const AdjTask& tk = tasks[find_by<AdjTask, &AdjTask::block_begin>(tasks, ntasks, gb)];
  const int local = gb - tk.block_begin;
  const int width = adj_width(tk.n);
  if (W == 1 || width == 1) return adjoint_tile<1>(tk, local, (AdjRay<1>*)P);
  if constexpr (W >= 2) if (width == 2) return adjoint_tile<2>(tk, local, (AdjRay<2>*)P);
  if constexpr (W >= 4) if (width == 4) return adjoint_tile<4>(tk, local, (AdjRay<4>*)P);
  if constexpr (W >= 8) adjoint_tile<8>(tk, local, (AdjRay<8>*)P);
}

__device__ __forceinline__ float at(const ACU_GLOBAL float* row, int N, int i) {
  return (i >= 1 && i <= N) ? row[i - 1] : 0.0f;
}

// detector shift of one row: out(d) = (1 - w) y(d + o) + w y(d + o + 1),
// o = floor(-s), w = -s - o (exact in FP32)
__device__ __forceinline__ void shift_weights(float s, int& o, float& w) {
  const float sg = -s;
  const float fl = floorf(sg);
  o = (int)fl;
  w = sg - fl;
}

__global__ __launch_bounds__(GR_THREADS) void shift_resid_kernel(const ResTask* __restrict__ tasks, int ntasks,
                                                                 int base, int nrows) {
#pragma clang fp contract(off)
  __shared__ double wsum[GR_THREADS / 64];
  const int lrow = xcd_remap(blockIdx.x, gridDim.x);
  if (lrow >= nrows) return;  // uniform per workgroup
  const int gr = base + lrow;
  const ResTask& tk = tasks[find_by<ResTask, &ResTask::row_begin>(tasks, ntasks, gr)];
  const int N = tk.N;
  const int t = gr - tk.row_begin;
  int o = 0;
  float w = 0.0f;
  if (tk.shift) shift_weights(tk.shift[t], o, w);
  const ACU_GLOBAL float* y = as_global(tk.y) + (size_t)t * N;
  const ACU_GLOBAL float* bm = as_global(tk.b) + (size_t)t * N;
  const float w1 = 1.0f - w;
  auto resid = [&](int d) -> float {  // r(d), zero off the detector
    if (d < 1 || d > N) return 0.0f;
    return (w1 * at(y, N, d + o) + w * at(y, N, d + o + 1)) - bm[d - 1];
  };
  double data = 0.0, g = 0.0, h = 0.0;
  for (int d = 1 + (int)threadIdx.x; d <= N; d += GR_THREADS) {
    const float ya = at(y, N, d + o), yb = at(y, N, d + o + 1);
    const float r = (w1 * ya + w * yb) - bm[d - 1];
    const double dy = (double)ya - (double)yb;
    data += 0.5 * (double)r * (double)r;
    g += (double)r * dy;
    h += dy * dy;
    // rs(k) = (1 - w) r(k - o) + w r(k - o - 1) at k = d
    tk.rs[(size_t)t * N + d - 1] = w1 * resid(d - o) + w * resid(d - o - 1);
  }
  data = block_sum(data, wsum);
  g = block_sum(g, wsum);
  h = block_sum(h, wsum);
  if (threadIdx.x == 0) {
    tk.part[t] = data;
    if (tk.gs) tk.gs[t] = (float)g;
    if (tk.hs) tk.hs[t] = (float)h;
  }
}

__global__ __launch_bounds__(GR_THREADS) void tvgrad_kernel(const TVGTask* __restrict__ tasks, int ntasks,
                                                            int base, int nblocks) {
  __shared__ double wsum[GR_THREADS / 64];
  const int lbk = xcd_remap(blockIdx.x, gridDim.x);
  if (lbk >= nblocks) return;  // uniform per workgroup
  const int gb = base + lbk;
  const TVGTask& tk = tasks[find_by<TVGTask, &TVGTask::block_begin>(tasks, ntasks, gb)];
  const int N = tk.N;
  const int lb = gb - tk.block_begin;
  const size_t i = (size_t)lb * GR_THREADS + threadIdx.x;
  double tv = 0.0;
  if (i < (size_t)N * N) {
    const int y = (int)(i / (size_t)N), x = (int)(i - (size_t)y * N);  // 0-based
    const int xp = x == N - 1 ? 0 : x + 1, xm = x == 0 ? N - 1 : x - 1;
    const int yp = y == N - 1 ? 0 : y + 1, ym = y == 0 ? N - 1 : y - 1;
    const ACU_GLOBAL float* u = as_global(tk.x);
    auto U = [&](int a, int b) { return u[(size_t)b * N + a]; };
    const float e2 = tk.eps * tk.eps;
    const float u0 = U(x, y);
    // difference vector and its norm at (x, y), at (x+1, y) and at (x, y+1)
    const float dx0 = U(xm, y) - u0, dy0 = U(x, ym) - u0;
    const float n0 = sqrtf(dx0 * dx0 + dy0 * dy0 + e2);
    tv = (double)n0;
    if (tk.gx) {
      const float u1 = U(xp, y);
      const float dx1 = u0 - u1, dy1 = U(xp, ym) - u1;
      const float n1 = sqrtf(dx1 * dx1 + dy1 * dy1 + e2);
      const float u2 = U(x, yp);
      const float dx2 = U(xm, yp) - u2, dy2 = u0 - u2;
      const float n2 = sqrtf(dx2 * dx2 + dy2 * dy2 + e2);
      const float gtv = (dx1 / n1 - dx0 / n0) + (dy2 / n2 - dy0 / n0);
      tk.gx[i] = tk.gx[i] + tk.lambda * gtv;
    }
  }
  tv = block_sum(tv, wsum);
  if (threadIdx.x == 0) tk.part[lb] = tv;
}

__global__ __launch_bounds__(GR_THREADS) void loss_finalize_kernel(const LossTask* __restrict__ tasks) {
  __shared__ double wsum[GR_THREADS / 64];
  const LossTask& tk = tasks[blockIdx.x];
  double a = 0.0, b = 0.0;
  for (int i = threadIdx.x; i < tk.nd; i += GR_THREADS) a += tk.pd[i];
  for (int i = threadIdx.x; i < tk.nt; i += GR_THREADS) b += tk.pt[i];
  a = block_sum(a, wsum);
  b = block_sum(b, wsum);
  if (threadIdx.x == 0) {
    tk.loss[0] = a + tk.lambda * b;
    tk.loss[1] = a;
    tk.loss[2] = b;
  }
}

}  // namespace

std::vector<std::vector<int>> adj_groups(const std::vector<int>& geo, const std::vector<int>& T, int most) {
  std::vector<std::vector<int>> g;
  std::map<int, size_t> open;  // geometry -> its last group
  for (int i = 0; i < (int)geo.size(); ++i) {
    const auto it = open.find(geo[i]);
    if (it != open.end() && (int)g[it->second].size() < most) {
      g[it->second].push_back(i);
      continue;
    }
    open[geo[i]] = g.size();
    g.push_back({i});
  }
  // a tile's time: us per tile and angle at widths 1, 2, 4 and 8 as 245, 283, 352 and 570
  auto time = [&](const std::vector<int>& v) {
    const int w = adj_width((int)v.size());
    return (double)T[v[0]] * (w == 1 ? 245 : w == 2 ? 283 : w == 4 ? 352 : 570);
  };
  std::stable_sort(g.begin(), g.end(), [&](const auto& a, const auto& b) { return time(a) > time(b); });
  return g;
}

void launch_adjoint(const AdjTask* d_tasks, const std::vector<AdjTask>& tasks, hipStream_t s) {
  int most = 1, blocks = 0;
  bool mixed = false;
  for (const AdjTask& t : tasks) {
    if (t.n < 1 || t.n > ADJ_GROUP || t.block_begin != blocks) throw Error("adjoint tasks do not match the launch");
    most = std::max(most, adj_width(t.n));
    mixed = mixed || t.T != tasks[0].T || adj_width(t.n) != adj_width(tasks[0].n);
    blocks += t.ntx * t.ntx;
  }
  if (blocks <= 0) return;
  const dim3 grid(xcd_grid(blocks)), wg(ADJ_T * ADJ_T);
  const int n = (int)tasks.size();
  switch (most) {
    case 1: hipLaunchKernelGGL(adjoint_kernel<1>, grid, wg, 0, s, d_tasks, n, blocks, mixed); break;
    case 2: hipLaunchKernelGGL(adjoint_kernel<2>, grid, wg, 0, s, d_tasks, n, blocks, mixed); break;
    case 4: hipLaunchKernelGGL(adjoint_kernel<4>, grid, wg, 0, s, d_tasks, n, blocks, mixed); break;
    default: hipLaunchKernelGGL(adjoint_kernel<8>, grid, wg, 0, s, d_tasks, n, blocks, mixed); break;
  }
}

void launch_shift_resid(const ResTask* d_tasks, int ntasks, int base, int rows, hipStream_t s) {
  if (rows <= 0) return;
  hipLaunchKernelGGL(shift_resid_kernel, dim3(xcd_grid(rows)), dim3(GR_THREADS), 0, s, d_tasks, ntasks, base,
                     rows);
}

void launch_tvgrad(const TVGTask* d_tasks, int ntasks, int base, int blocks, hipStream_t s) {
  if (blocks <= 0) return;
  hipLaunchKernelGGL(tvgrad_kernel, dim3(xcd_grid(blocks)), dim3(GR_THREADS), 0, s, d_tasks, ntasks, base,
                     blocks);
}

void launch_loss_finalize(const LossTask* d_tasks, int ntasks, hipStream_t s) {
  if (ntasks <= 0) return;
  hipLaunchKernelGGL(loss_finalize_kernel, dim3(ntasks), dim3(GR_THREADS), 0, s, d_tasks);
}

}  // namespace acu
