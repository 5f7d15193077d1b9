// prep.hip -- gfx950 kernels of the projection -> sinogram preprocessing
// (tomography/projections_to_sinogram_hpc.F90): 3x3x3 median filter,
// rotation / centre-of-rotation correction by clamped bilinear resampling
// written straight into the sinogram layout, and the mirror error that the
// centre-of-rotation search minimises.
//
// Layouts follow the reference (first index fastest): a projection is
// img(x, y), n x n (x = detector column, y = detector row = slice); the
// corrected projection row jy of projection `job` is sinogram row `job` of
// slice jy, Nw = n + add_Nx values long.
#include "acu_prep.hpp"
#include "median_net.hpp"

#include <algorithm>

namespace acu {
namespace {

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : v > hi ? hi : v; }
__device__ __forceinline__ float clampf(float v, float lo, float hi) { return fminf(fmaxf(v, lo), hi); }

// The 14th smallest of 27 values in registers: the compile-time network of
// median_net.hpp, fully unrolled (153 compare-exchanges).
__device__ __forceinline__ float median27(float (&v)[27]) {
#pragma unroll
  for (int i = 0; i < MEDIAN27_NET.n; ++i) {
    const float a = v[MEDIAN27_NET.lo[i]], b = v[MEDIAN27_NET.hi[i]];
    v[MEDIAN27_NET.lo[i]] = fminf(a, b);
    v[MEDIAN27_NET.hi[i]] = fmaxf(a, b);
  }
  return v[MEDIAN27_NET.out];
}

// the instructions themselves: fminf and fmaxf would quiet each operand first
struct Float3Ops {
  static __device__ __forceinline__ float min3(float a, float b, float c) {
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
  }
  static __device__ __forceinline__ float med3(float a, float b, float c) {
    float r;
    asm("v_med3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
  }
  static __device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
  }
};

// 3x3x3 median (:420-447): projections l, c, r; neighbours clamped into the
// image; the 14th of 27 in descending order = the 14th in ascending order.
// This is the median the reference's loop nest describes: its register
// slots 3*jxs+jys+2 (+9, +18) run from -2 to 24 in an array of 27 (:433-435
// against :134), so its own code writes 3 neighbours out of bounds and sorts
// 3 stale slots in their place; that undefined result is not reproduced.
// Values that compare equal but differ in bits (+0 and -0) or NaN are the
// exception: the reference's exchange sort is not stable, so which of them
// it leaves in the middle depends on its order of exchanges.
//
// A wave takes 62 x K pixels: a lane loads its column of the K + 2 rows of
// the three projections (all loads in flight, no LDS), gets its neighbours'
// values by DPP and, walking down, sorts the nine values of the next row once
// and selects the median of the last three sorted rows: 46 instructions a
// pixel (and 27 for each of the rows above and below its K) instead of the
// 306 of the network for 27 loose values.  That network stays for waves whose
// values hold a NaN, where the result depends on the order of comparisons.
// Bound by its traffic (three images in, one out: 67 MB, 12 us at the ingest
// kernels' rate) and its sorting (about 10 us of half-rate min, med and max
// issue), which a wave does one after the other. us per 2048^2 image: 19, 21
// with the rows staged in LDS, 57 with the network in every pixel.
constexpr int MED_X = 62;

__device__ __forceinline__ float lane_prev(float v) {  // wave_shr:1: lane i reads lane i - 1
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x138, 0xF, 0xF, false));
}
__device__ __forceinline__ float lane_next(float v) {  // wave_shl:1: lane i reads lane i + 1
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x130, 0xF, 0xF, false));
}

template <int K>
__global__ __launch_bounds__(256) void median27_kernel(int n, const float* __restrict__ l,
                                                       const float* __restrict__ c, const float* __restrict__ r,
                                                       float* __restrict__ out, int tiles_x) {
  const int bx = blockIdx.x % tiles_x, by = blockIdx.x / tiles_x;
  const int lane = threadIdx.x & 63;
  const int y = __builtin_amdgcn_readfirstlane((by * 4 + (int)(threadIdx.x >> 6)) * K);  // 0-based first row
  const int x = bx * MED_X + lane - 1;
  if (y >= n) return;  // the whole wave
  const unsigned gx = (unsigned)clampi(x, 0, n - 1);
  const bool own = lane >= 1 && lane <= MED_X && x < n;
  float raw[K + 2][3];
#pragma unroll
  for (int k = 0; k < K + 2; ++k) {
    const size_t o = (size_t)clampi(y + k - 1, 0, n - 1) * n;
    raw[k][0] = (l + o)[gx];
    raw[k][1] = (c + o)[gx];
    raw[k][2] = (r + o)[gx];
  }
  bool nan = false;
#pragma unroll
  for (int k = 0; k < K + 2; ++k)
#pragma unroll
    for (int p = 0; p < 3; ++p) nan = nan || raw[k][p] != raw[k][p];
  if (__ballot(nan)) {
    if (!own) return;
    for (int k = 0; k < K && y + k < n; ++k) {
      float v[27];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const float* img = p == 0 ? l : p == 1 ? c : r;
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
          for (int dx = 0; dx < 3; ++dx)
            v[p * 9 + dy * 3 + dx] =
                img[(size_t)clampi(y + k + dy - 1, 0, n - 1) * n + clampi(x + dx - 1, 0, n - 1)];
      }
      out[(size_t)(y + k) * n + x] = median27(v);
    }
    return;
  }
  auto row = [&](int k, float (&v)[9]) {
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      v[3 * p] = lane_prev(raw[k][p]);
      v[3 * p + 1] = raw[k][p];
      v[3 * p + 2] = lane_next(raw[k][p]);
    }
    sort9<Float3Ops>(v);
  };
  float v[3][9];
  row(0, v[0]);
  row(1, v[1]);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    row(k + 2, v[(k + 2) % 3]);
    const float med = median27_of_sorted<Float3Ops>(v[0], v[1], v[2]);
    if (own && y + k < n) out[(size_t)(y + k) * n + x] = med;
  }
}

// The resampling of :449-464 at output (jx, jy), 1-based, in the
// reference's FP32 order: u = (jx - mx) - S*shift, xr = clamp((c*u - s*(jy-my)) + mx),
// yr = clamp((s*u + c*(jy-my)) + my), taps clamped into the image; a tap
// pair clamped onto one pixel has both weights zero.
struct PrepTaps {
  size_t o11, o12, o21, o22;  // pixels (x1, y1), (x2, y1), (x1, y2), (x2, y2)
  float ax, bx, ay, by;
};
__device__ __forceinline__ PrepTaps prep_taps(const PrepGeom& g, int jx, int jy) {
#pragma clang fp contract(off)
  const int n = g.n;
  const float u = ((float)jx - g.mx) - g.S * g.shift;
  const float w = (float)jy - g.my;
  const float xr = clampf((g.c * u - g.s * w) + g.mx, 1.0f, (float)n);
  const float yr = clampf((g.s * u + g.c * w) + g.my, 1.0f, (float)n);
  const int y1 = clampi((int)floorf(yr), 1, n), y2 = clampi(y1 + 1, 1, n);
  const int x1 = clampi((int)floorf(xr), 1, n), x2 = clampi(x1 + 1, 1, n);
  PrepTaps q;
  q.ax = (float)x2 - xr;
  q.bx = xr - (float)x1;
  q.ay = (float)y2 - yr;
  q.by = yr - (float)y1;
  const size_t r1 = (size_t)(y1 - 1) * n, r2 = (size_t)(y2 - 1) * n;
  q.o11 = r1 + (x1 - 1);
  q.o12 = r1 + (x2 - 1);
  q.o21 = r2 + (x1 - 1);
  q.o22 = r2 + (x2 - 1);
  return q;
}
__device__ __forceinline__ float prep_lerp(const PrepTaps& q, const float* __restrict__ img) {
#pragma clang fp contract(off)
  float v = (img[q.o11] * q.ax) * q.ay;
  v = v + (img[q.o12] * q.bx) * q.ay;
  v = v + (img[q.o21] * q.ax) * q.by;
  v = v + (img[q.o22] * q.bx) * q.by;
  return v;
}
__device__ __forceinline__ float prep_sample(const PrepGeom& g, const float* __restrict__ img, int jx, int jy) {
  return prep_lerp(prep_taps(g, jx, jy), img);
}

// Corrected projections of a batch -> sinogram rows: projection k of the
// batch (global index job0 + k) fills row job0 + k of every slice's
// sinogram; sino is nslices(= n) x nfiles x Nw, slice-major.  Grid: x over
// the Nw output columns, y = the detector row jy - 1 - row0, z = groups of
// COR_K projections: the positions and weights are the same for every
// projection, so a thread forms them once for its group and has the group's
// gathers in flight together; the last group takes what is left.  Bound by
// its traffic: us at 2048^2 with 1, 2, 3, 4, 5 and 8 projections 10.9, 17.4,
// 24.4, 32.2, 41.4 and 62.5 (268 MB, 4.3 TB/s); with one projection a thread
// 10.9, 19.4, 27.9, 36.5, 44.9 and 70.6; with every group padded to four by its
// last projection 15.7, 17.0, 24.3, 32.4, 45.2 and 62.7.
constexpr int COR_K = 4;
template <int K>
__device__ __forceinline__ void correct_group(const PrepTaps& q, const float* __restrict__ img, size_t nn,
                                              float* __restrict__ o, int nw) {
  float v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = prep_lerp(q, img + (size_t)k * nn);
#pragma unroll
  for (int k = 0; k < K; ++k) o[(size_t)k * nw] = v[k];
}
// K: 1 for a launch over one projection, else COR_K
template <int K>
__global__ __launch_bounds__(256) void correct_kernel(PrepGeom g, const float* __restrict__ imgs, int count, int job0,
                                                      int nfiles, int row0, float* __restrict__ sino) {
  const int nw = g.n + g.add_nx;
  const int jx = (int)(blockIdx.x * blockDim.x + threadIdx.x) + 1;
  if (jx > nw) return;
  const int jy = row0 + (int)blockIdx.y + 1, k0 = (int)blockIdx.z * COR_K;
  const PrepTaps q = prep_taps(g, jx, jy);
  const size_t nn = (size_t)g.n * g.n;
  const float* img = imgs + (size_t)k0 * nn;
  float* o = sino + ((size_t)(jy - 1) * nfiles + (size_t)(job0 + k0)) * nw + (jx - 1);
  if constexpr (K < COR_K) return correct_group<K>(q, img, nn, o, nw);
  switch (min(count - k0, COR_K)) {  // uniform
    case 1: correct_group<1>(q, img, nn, o, nw); break;
    case 2: correct_group<2>(q, img, nn, o, nw); break;
    case 3: correct_group<3>(q, img, nn, o, nw); break;
    default: correct_group<COR_K>(q, img, nn, o, nw); break;
  }
}

// |V0(jx,jy) - V180(Nw-jx+1,jy)| summed per block in FP64 (:278-283).
__global__ __launch_bounds__(256) void mirror_kernel(PrepGeom g, const float* __restrict__ p0,
                                                     const float* __restrict__ p180, double* __restrict__ part) {
  __shared__ double ws[4];
  const int nw = g.n + g.add_nx;
  const size_t total = (size_t)nw * g.n;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  double e = 0.0;
  if (i < total) {
    const int jy = (int)(i / nw) + 1, jx = (int)(i - (size_t)(jy - 1) * nw) + 1;
    e = (double)fabsf(prep_sample(g, p0, jx, jy) - prep_sample(g, p180, nw - jx + 1, jy));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o);
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (ws[0] + ws[1]) + (ws[2] + ws[3]);
}

__global__ __launch_bounds__(256) void sum_kernel(const double* __restrict__ part, int n, double* __restrict__ out) {
  __shared__ double ws[4];
  double e = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) e += part[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o);
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) *out = (ws[0] + ws[1]) + (ws[2] + ws[3]);
}

}  // namespace

constexpr int MED_MIN = 512;  // workgroups of strips of 8 rows, two per CU: 1000^2 pixels

void launch_median27(int n, const float* l, const float* c, const float* r, float* out, hipStream_t s) {
  const int tx = (n + MED_X - 1) / MED_X;
  auto rows = [&](int k) { return (n + 4 * k - 1) / (4 * k); };
  // strips of 8 rows sort 10 rows for 8 pixels, of 2 rows 4 for 2, but keep
  // the GPU busier on small images: us of the kernel with 8 and with 2 rows, 3.6
  // and 2.6 at 65^2, 3.9 and 2.8 at 257^2, 4.0 and 3.2 at 512^2, 4.9 and 4.5 at
  // 700^2, 5.3 and 5.2 at 850^2, 6.5 and 6.5 at 1024^2, 18.9 and 21.0 at 2048^2
  if (tx * rows(8) >= MED_MIN)
    hipLaunchKernelGGL(median27_kernel<8>, dim3(tx * rows(8)), dim3(256), 0, s, n, l, c, r, out, tx);
  else
    hipLaunchKernelGGL(median27_kernel<2>, dim3(tx * rows(2)), dim3(256), 0, s, n, l, c, r, out, tx);
}

void launch_correct(const PrepGeom& g, const float* imgs, int count, int job0, int nfiles, float* sino,
                    hipStream_t s) {
  const unsigned gx = (unsigned)((g.n + g.add_nx + 255) / 256);
  for (int k0 = 0; k0 < count; k0 += 65535)  // the grid's y and z extents are at most 65535
    for (int r0 = 0; r0 < g.n; r0 += 65535) {
      const int cnt = std::min(65535, count - k0), rows = std::min(65535, g.n - r0);
      const dim3 grid(gx, (unsigned)rows, (unsigned)((cnt + COR_K - 1) / COR_K));
      const float* in = imgs + (size_t)k0 * g.n * g.n;
      // one projection by the groups' kernel: 11.9 us at 2048^2 instead of 10.9 (46 registers instead of 20)
      const auto kernel = cnt == 1 ? correct_kernel<1> : correct_kernel<COR_K>;
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, g, in, cnt, job0 + k0, nfiles, r0, sino);
    }
}

int mirror_blocks(const PrepGeom& g) { return (int)(((size_t)(g.n + g.add_nx) * g.n + 255) / 256); }

void launch_mirror(const PrepGeom& g, const float* p0, const float* p180, double* part, double* out,
                   hipStream_t s) {
  const int nb = mirror_blocks(g);
  hipLaunchKernelGGL(mirror_kernel, dim3(nb), dim3(256), 0, s, g, p0, p180, part);
  hipLaunchKernelGGL(sum_kernel, dim3(1), dim3(256), 0, s, part, nb, out);
}

PrepGeom prep_geom(int n, int add_nx, float theta, float shift) {
#pragma clang fp contract(off)
  PrepGeom g;
  g.n = n;
  g.add_nx = add_nx;
  const int nw = n + add_nx;
  g.mx = (float)(nw - 1) / 2.0f;
  g.my = (float)(n - 1) / 2.0f;
  g.S = (float)n;
  g.shift = shift;
  g.c = cosf(theta);
  g.s = sinf(theta);
  return g;
}

}  // namespace acu

// ---- FITS ingest normalisation (tomography/fits_to_hpc.F90:196-248) ----
//
// mean: one thread per pixel (VEC: four adjacent pixels, one 16-byte
// access) loops over the images in file order.
//
// normalize: -log(I / b), b = max(OB, 1).  The open beam is fixed per pixel
// across the projections, so its reciprocal y = RN(1/b) is formed once per
// pixel with the IEEE division and each quotient then costs one product and
// two FMAs:  q = RN(I y),  q' = RN(q + RN(I - b q) y).  With y correctly
// rounded and q within one ulp of I/b, the remainder I - b q is exact and q'
// is the correctly rounded quotient (P. Markstein, IBM J. Res. Dev. 34(1),
// 1990; Cornea-Hasegan, Golliver, Markstein, ARITH-14, 1999, Theorem 1),
// i.e. bit-identical to I / b, provided nothing underflows or overflows: for
// |I| < 2^-100, |q| < 2^-100, b = inf, or I not finite the kernel takes the
// IEEE division instead.  Each thread handles one pixel group of
// ING_CHUNK consecutive projections (grid: pixel groups x projection
// chunks); longer per-thread runs across images measured slower (the
// write streams lose DRAM locality).  VEC needs npix % 4 == 0 and 16-byte
// aligned pointers (checked on the host).
namespace acu {
namespace {

constexpr int ING_CHUNK = 2;

template <bool VEC> struct Px { typedef float type; };
template <> struct Px<true> { typedef float4 type; };

__device__ __forceinline__ float add_(float a, float b) { return a + b; }
__device__ __forceinline__ float4 add_(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
__device__ __forceinline__ float div_(float a, float c) { return a / c; }
__device__ __forceinline__ float4 div_(float4 a, float c) { return make_float4(a.x / c, a.y / c, a.z / c, a.w / c); }

struct BY { float b, y; };
__device__ __forceinline__ BY by_(float ob) {
  const float b = fmaxf(ob, 1.0f);
  return {b, 1.0f / b};
}
__device__ __forceinline__ float nlog_(float a, BY p) {
  float q = a * p.y;
  if (fabsf(a) >= 0x1p-100f && fabsf(a) <= 3.40282347e38f && fabsf(q) >= 0x1p-100f && p.b <= 3.40282347e38f)
    q = fmaf(fmaf(-p.b, q, a), p.y, q);
  else
    q = a / p.b;
  return -logf(q);
}

// out = (sum over images, in order, FP32) / count: the open-beam average of
// :203-215, accumulated one file at a time from bg = 0
template <bool VEC>
__global__ __launch_bounds__(256) void mean_kernel(const float* __restrict__ imgs, int count, size_t npix,
                                                   float* __restrict__ out) {
#pragma clang fp contract(off)
  typedef typename Px<VEC>::type P;
  const size_t n = VEC ? npix / 4 : npix;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const P* src = reinterpret_cast<const P*>(imgs);
  P s;
  if constexpr (VEC) s = make_float4(0.0f, 0.0f, 0.0f, 0.0f); else s = 0.0f;  // -0 + ... gives +0, as bg = 0
  for (int k = 0; k < count; ++k) s = add_(s, src[(size_t)k * n + i]);
  reinterpret_cast<P*>(out)[i] = div_(s, (float)count);
}

// projection = -log(image / max(open_beam, 1)) (:243); blockIdx.y = chunk
template <bool VEC>
__global__ __launch_bounds__(256) void normalize_kernel(const float* __restrict__ imgs, int count, size_t npix,
                                                        const float* __restrict__ ob, float* __restrict__ out) {
#pragma clang fp contract(off)
  const size_t n = VEC ? npix / 4 : npix;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int k0 = blockIdx.y * ING_CHUNK, k1 = min(count, k0 + ING_CHUNK);
  if constexpr (VEC) {
    const float4 o = reinterpret_cast<const float4*>(ob)[i];
    const BY p0 = by_(o.x), p1 = by_(o.y), p2 = by_(o.z), p3 = by_(o.w);
    const float4* src = reinterpret_cast<const float4*>(imgs);
    float4* dst = reinterpret_cast<float4*>(out);
    for (int k = k0; k < k1; ++k) {
      const float4 v = src[(size_t)k * n + i];
      dst[(size_t)k * n + i] = make_float4(nlog_(v.x, p0), nlog_(v.y, p1), nlog_(v.z, p2), nlog_(v.w, p3));
    }
  } else {
    const BY p = by_(ob[i]);
    for (int k = k0; k < k1; ++k) out[(size_t)k * n + i] = nlog_(imgs[(size_t)k * n + i], p);
  }
}

bool vec_ok(size_t npix, const void* a, const void* b, const void* c) {
  const uintptr_t m = (uintptr_t)a | (uintptr_t)b | (uintptr_t)c;
  return npix % 4 == 0 && (m & 15) == 0;
}

}  // namespace

void launch_mean(const float* imgs, int count, size_t npix, float* out, hipStream_t s) {
  if (vec_ok(npix, imgs, out, out))
    hipLaunchKernelGGL(mean_kernel<true>, dim3((unsigned)((npix / 4 + 255) / 256)), dim3(256), 0, s, imgs, count,
                       npix, out);
  else
    hipLaunchKernelGGL(mean_kernel<false>, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, s, imgs, count,
                       npix, out);
}

void launch_normalize(const float* imgs, int count, size_t npix, const float* ob, float* out, hipStream_t s) {
  const bool vec = vec_ok(npix, imgs, ob, out);
  const unsigned gx = (unsigned)(((vec ? npix / 4 : npix) + 255) / 256);
  constexpr int kMaxImages = 65535 * ING_CHUNK;  // gridDim.y limit
  for (int k = 0; k < count; k += kMaxImages) {
    const int c = std::min(kMaxImages, count - k);
    const dim3 grid(gx, (unsigned)((c + ING_CHUNK - 1) / ING_CHUNK));
    const float* in = imgs + (size_t)k * npix;
    float* o = out + (size_t)k * npix;
    if (vec)
      hipLaunchKernelGGL(normalize_kernel<true>, grid, dim3(256), 0, s, in, c, npix, ob, o);
    else
      hipLaunchKernelGGL(normalize_kernel<false>, grid, dim3(256), 0, s, in, c, npix, ob, o);
  }
}

}  // namespace acu
