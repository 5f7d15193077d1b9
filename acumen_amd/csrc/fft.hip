// fft.hip -- the ramp filter (tomography/tv_hpc.F90:93-105) by FFT
// convolution in FP64: RAMP_FP64 of slices up to N = 4097, and RAMP_FFT.
//
//   sinoCS(i, t) = sum_{j=0..N-1} g(i - j) sino(j, t),   g(m) = h[m + N],
//
// is a linear convolution with the symmetric kernel g on |m| <= N-1.  With
// L a power of two >= 2N-2 it equals the circular convolution of length L
// with gw(r) = sum_{m = r mod L} g(m), except when L = 2N-2, where m = N-1
// and m = -(N-1) share a residue: then outputs 0 and N-1 pick up one extra
// term each, g(N-1) s(N-1) and g(N-1) s(0), which are subtracted.  G =
// DFT(gw) is real and even (g is symmetric).
//
// A real row of L values is one complex transform of M = L/2 points z(n) =
// x(2n) + i x(2n+1), so rows never mix (a row of NaN or of huge values
// leaves its neighbours alone).  The spectrum X of the row, its product with
// G and the packing of the result back into M points are one pass over the
// pairs (k, M-k).
//
// gfx950 mapping: M/8 threads per row, rows packed into workgroups of NT =
// 64..512 threads (the largest row of the batch sets NT); the M points live
// in LDS, padded by one in eight against bank conflicts.  Forward: radix-8
// decimation in frequency, in place, the first pass straight from global
// memory, the last of radix 1, 2 or 4; the pair pass works on the
// digit-reversed order that leaves; the inverse runs the same passes
// backwards (decimation in time), the last one straight to global memory.
// A butterfly's twiddles are three table loads (w, w^2, w^4) and four
// products.  G and the twiddles come from the host in FP64 (the reference's
// FP32 taps).
//
// Bound by its LDS passes (about 16 of 16 bytes per point) and their
// barriers.  A 2049^2 x 1500 slice is 12.6 GFLOP as a Toeplitz product and
// 0.45 GFLOP this way.  The result is the exact one but for its rounding to
// FP32, as the Toeplitz product's on the FP64 matrix cores is (filter.hip):
// both are 2.5e-8 from FP64 on noise at N = 6..4097.  Kernel times on MI355X,
// us, this | the radix-2 FP32 transform of row pairs that it replaces | the
// product: 8 x 2049^2 x 1500 230 | 437 | 2285, 4 x 1025^2 x 720 35 | 54 | 208, 257^2 x
// 180 7 | 7 | 23.  The same passes in FP32 took 164 at 8 x 2049^2 x 1500 with
// products of FP32 twiddles, but 1.2x the error of that radix-2 transform;
// without the extra error they took 202, so there is no FP32 form.
#include "acu_internal.hpp"

#include <algorithm>
#include <cmath>
#include <complex>
#include <type_traits>
#include <vector>

namespace acu {
namespace {

constexpr double kPi = 3.14159265358979323846;

typedef double2 C;

__device__ __forceinline__ C mk(double x, double y) { return make_double2(x, y); }
__device__ __forceinline__ C cadd(C a, C b) { return mk(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ C csub(C a, C b) { return mk(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ C cmul(C a, C b) { return mk(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ __forceinline__ C cconj(C a) { return mk(a.x, -a.y); }
// a * (-i) (forward) or a * i (inverse)
template <bool INV> __device__ __forceinline__ C rot(C a) { return INV ? mk(-a.y, a.x) : mk(a.y, -a.x); }

template <bool INV>
__device__ __forceinline__ void dft4(C a0, C a1, C a2, C a3, C& y0, C& y1, C& y2, C& y3) {
  const C s02 = cadd(a0, a2), d02 = csub(a0, a2), s13 = cadd(a1, a3), r13 = rot<INV>(csub(a1, a3));
  y0 = cadd(s02, s13);
  y2 = csub(s02, s13);
  y1 = cadd(d02, r13);
  y3 = csub(d02, r13);
}

// x <- DFT of x (natural order both sides); INV: unnormalised inverse
template <int R, bool INV>
__device__ __forceinline__ void dft(C (&x)[R]) {
  if constexpr (R == 2) {
    const C a = x[0];
    x[0] = cadd(a, x[1]);
    x[1] = csub(a, x[1]);
  } else if constexpr (R == 4) {
    C y0, y1, y2, y3;
    dft4<INV>(x[0], x[1], x[2], x[3], y0, y1, y2, y3);
    x[0] = y0; x[1] = y1; x[2] = y2; x[3] = y3;
  } else {
    const double h = 0.70710678118654752440;
    const C e0 = cadd(x[0], x[4]), e1 = cadd(x[1], x[5]), e2 = cadd(x[2], x[6]), e3 = cadd(x[3], x[7]);
    const C o0 = csub(x[0], x[4]), d1 = csub(x[1], x[5]), d2 = csub(x[2], x[6]), d3 = csub(x[3], x[7]);
    // o_j = d_j exp(-+ i pi j / 4)
    const C r1 = rot<INV>(d1), r3 = rot<INV>(d3);
    const C o1 = mk((d1.x + r1.x) * h, (d1.y + r1.y) * h), o2 = rot<INV>(d2),
            o3 = mk((r3.x - d3.x) * h, (r3.y - d3.y) * h);
    dft4<INV>(e0, e1, e2, e3, x[0], x[2], x[4], x[6]);
    dft4<INV>(o0, o1, o2, o3, x[1], x[3], x[5], x[7]);
  }
}

__device__ __forceinline__ int pad(int i) { return i + (i >> 3); }

// the twiddles w^1..w^7 of one radix-8 butterfly, w = W_M^e (e < M/8); conj for the inverse
template <bool INV>
__device__ __forceinline__ void twiddles(const C* __restrict__ tw, int e, C (&w)[8]) {
  w[1] = tw[e];
  w[2] = tw[2 * e];
  w[4] = tw[4 * e];
  if (INV) { w[1] = cconj(w[1]); w[2] = cconj(w[2]); w[4] = cconj(w[4]); }
  w[3] = cmul(w[1], w[2]);
  w[5] = cmul(w[1], w[4]);
  w[6] = cmul(w[2], w[4]);
  w[7] = cmul(w[3], w[4]);
}

// position of frequency k after the forward passes: `q` base-8 digits of k
// from the top of the m-bit position down, the rest below
__device__ __forceinline__ int freq_pos(int k, int m, int q) {
  int pos = 0, sh = m;
  for (int i = 0; i < q; ++i) {
    sh -= 3;
    pos |= (k & 7) << sh;
    k >>= 3;
  }
  return pos | k;
}

__device__ __forceinline__ int find_task(const FFTTask* tasks, int ntasks, int gb) {
  int lo = 0, hi = ntasks - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tasks[mid].block_begin <= gb) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Outputs lt, lt + step, ... of one row of fewer than 8 points as the plain sum in FP64.
__device__ void direct_row(const float* __restrict__ h, const float* __restrict__ s, float* __restrict__ out, int N,
                           int lt, int step) {
  for (int i = lt; i < N; i += step) {
    double a = 0.0;
    for (int j = 0; j < N; ++j) a += (double)h[i - j + N] * (double)s[j];
    out[i] = (float)a;
  }
}

// A row that holds infinities or NaN: the plain sum's result follows from
// those values alone, as the finite terms cannot overflow FP64.  The tap at
// distance 0 is positive, every other one negative (tv_hpc.F90:53-56), and
// none is zero: a NaN makes every output NaN, and an infinity is an infinity
// of its own sign at its place and of the other sign everywhere else.  Each
// wave looks through the row itself (its rt threads, if fewer than 64 have
// the row).  A 2049^2 x 1500 sinogram with an infinity in every row, or of
// infinities only, takes 41 us (33 if finite; 2940 by the plain sum, 350 as a
// matrix product).
__device__ void nonfinite_row(const float* __restrict__ s, float* __restrict__ out, int N, int lt, int rt) {
  const float inf = __builtin_inff();
  const int g = min(rt, 64), lane = threadIdx.x & 63, first = lane & ~(g - 1);
  bool nan = false;
  int np = 0, nn = 0;
  for (int n = lane - first; n < N; n += g) {
    const float x = s[n];
    nan = nan || x != x;
    np += x == inf;
    nn += x == -inf;
  }
  const unsigned long long own = (g == 64 ? ~0ull : (1ull << g) - 1) << first;
  // infinities of each sign in the row: 0, 1, or 2 for more
  const int pos = (__ballot(np > 1) & own) ? 2 : min(2, __popcll(__ballot(np > 0) & own));
  const int neg = (__ballot(nn > 1) & own) ? 2 : min(2, __popcll(__ballot(nn > 0) & own));
  nan = (__ballot(nan) & own) != 0;
  for (int i = lt; i < N; i += rt) {
    const bool p = s[i] == inf, q = s[i] == -inf;
    const bool up = p || neg > (int)q, down = q || pos > (int)p;
    out[i] = nan || (up && down) ? __builtin_nanf("") : up ? inf : -inf;
  }
}

template <int NT>
__global__ __launch_bounds__(NT) void fft_ramp_kernel(const FFTTask* __restrict__ tasks, int ntasks, int base,
                                                      int nblocks) {
  __shared__ C lds[NT * 9];
  __shared__ unsigned long long bad_s[NT / 64];
  const int lbk = xcd_remap(blockIdx.x, gridDim.x);
  if (lbk >= nblocks) return;  // uniform per workgroup
  const int gb = base + lbk;
  const FFTTask& tk = tasks[find_task(tasks, ntasks, gb)];
  const int N = tk.N, m = tk.lg - 1, M = 1 << m;
  const int local = gb - tk.block_begin;
  const int tid = threadIdx.x;
  if (m < 3) {
    direct_row(tk.h, tk.sino + (size_t)local * N, tk.out + (size_t)local * N, N, tid, NT);
    return;
  }
  const int lt = tid & (M / 8 - 1), g = tid >> (m - 3);  // thread of its row, row of the workgroup
  const int row = local * (NT >> (m - 3)) + g;
  const bool act = row < tk.T;
  const float* __restrict__ s = tk.sino + (size_t)(act ? row : 0) * N;
  float* __restrict__ out = tk.out + (size_t)(act ? row : 0) * N;
  const C* __restrict__ tw = tk.tw;
  const C* __restrict__ twl = tw + M / 2;  // exp(-2 pi i k / L), k <= M/2
  const double* __restrict__ G = tk.G;
  C* X = lds + g * (M + M / 8);
  const int q = m / 3, tail = m - 3 * q;

  // forward pass 1 from global memory: points beyond the row are zero
  C x[8], w[8];
  bool bad = false;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int n = 2 * (lt + j * (M / 8));
    const float a = act && n < N ? s[n] : 0.0f, b = act && n + 1 < N ? s[n + 1] : 0.0f;
    bad = bad || !(fabsf(a) <= 3.40282347e38f) || !(fabsf(b) <= 3.40282347e38f);
    x[j] = mk((double)a, (double)b);
  }
  const float s0 = s[0], s1 = s[N - 1];  // for the alias correction
  const unsigned long long bm = __ballot(bad);
  if ((tid & 63) == 0) bad_s[tid >> 6] = bm;
  dft<8, false>(x);
  twiddles<false>(tw, lt, w);
  X[pad(lt)] = x[0];
#pragma unroll
  for (int j = 1; j < 8; ++j) X[pad(lt + j * (M / 8))] = cmul(x[j], w[j]);
  __syncthreads();
  const int rt = M / 8;  // does this thread's row hold an infinity or NaN
  if (rt >= 64) for (int v = 0; v < rt / 64; ++v) bad = bad || bad_s[g * (rt / 64) + v] != 0;
  else bad = ((bad_s[tid >> 6] >> ((tid & 63) & ~(rt - 1))) & ((1ull << rt) - 1)) != 0;
  for (int ls = m - 6; ls >= tail; ls -= 3) {  // sub-transforms of 8 << ls points
    const int p = lt & ((1 << ls) - 1), i0 = ((lt >> ls) << (ls + 3)) + p;
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = X[pad(i0 + (j << ls))];
    dft<8, false>(x);
    twiddles<false>(tw, p << (m - 3 - ls), w);
    X[pad(i0)] = x[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) X[pad(i0 + (j << ls))] = cmul(x[j], w[j]);
    __syncthreads();
  }
  auto small = [&](auto inv) {  // the tail: sub-transforms of 2 or 4 points, no twiddles
    constexpr bool INV = decltype(inv)::value;
    if (tail == 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i0 = 2 * (lt + j * (M / 8));
        C y[2] = {X[pad(i0)], X[pad(i0 + 1)]};
        dft<2, INV>(y);
        X[pad(i0)] = y[0];
        X[pad(i0 + 1)] = y[1];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int i0 = 4 * (lt + j * (M / 8));
        C y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = X[pad(i0 + v)];
        dft<4, INV>(y);
#pragma unroll
        for (int v = 0; v < 4; ++v) X[pad(i0 + v)] = y[v];
      }
    }
    __syncthreads();
  };
  if (tail) small(std::false_type{});

  // pairs (k, M-k): X_k = E + w^k O, conj(X_{M-k}) = E - w^k O from Z_k and
  // Z_{M-k}; times the real G; packed back (G carries the 1/M of the inverse)
  for (int k = lt; k <= M / 2; k += M / 8) {
    const int ia = pad(freq_pos(k, m, q));
    const C za = X[ia];
    if (k == 0) {
      const double a = G[0] * (za.x + za.y), b = G[M] * (za.x - za.y);
      X[ia] = mk(0.5 * (a + b), 0.5 * (a - b));
    } else if (k == M / 2) {
      X[ia] = mk(G[k] * za.x, G[k] * za.y);
    } else {
      const int ib = pad(freq_pos(M - k, m, q));
      const C zb = cconj(X[ib]);
      const C e = mk(0.5 * (za.x + zb.x), 0.5 * (za.y + zb.y));
      const C o = mk(0.5 * (za.y - zb.y), 0.5 * (zb.x - za.x));  // -i (za - zb) / 2
      const C wk = twl[k], t = cmul(wk, o);
      const double ga = G[k], gm = G[M - k];
      const C a = mk(ga * (e.x + t.x), ga * (e.y + t.y)), b = mk(gm * (e.x - t.x), gm * (e.y - t.y));
      const C e2 = mk(0.5 * (a.x + b.x), 0.5 * (a.y + b.y));
      const C o2 = cmul(cconj(wk), mk(0.5 * (a.x - b.x), 0.5 * (a.y - b.y)));
      X[ia] = mk(e2.x - o2.y, e2.y + o2.x);  // E' + i O'
      X[ib] = mk(e2.x + o2.y, o2.x - e2.y);  // conj(E' - i O')
    }
  }
  __syncthreads();

  if (tail) small(std::true_type{});
  for (int ls = tail; ls <= m - 6; ls += 3) {
    const int p = lt & ((1 << ls) - 1), i0 = ((lt >> ls) << (ls + 3)) + p;
    twiddles<true>(tw, p << (m - 3 - ls), w);
    x[0] = X[pad(i0)];
#pragma unroll
    for (int j = 1; j < 8; ++j) x[j] = cmul(X[pad(i0 + (j << ls))], w[j]);
    dft<8, true>(x);
#pragma unroll
    for (int j = 0; j < 8; ++j) X[pad(i0 + (j << ls))] = x[j];
    __syncthreads();
  }
  // inverse pass over all M points, to global memory (no barrier below)
  if (!act) return;
  if (bad) {
    nonfinite_row(s, out, N, lt, rt);
    return;
  }
  twiddles<true>(tw, lt, w);
  x[0] = X[pad(lt)];
#pragma unroll
  for (int j = 1; j < 8; ++j) x[j] = cmul(X[pad(lt + j * (M / 8))], w[j]);
  dft<8, true>(x);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int n = 2 * (lt + j * (M / 8));
    double a = x[j].x;
    if (tk.alias) {  // L = 2N-2: remove the wrapped term of the shared residue (N - 1 is even)
      if (n == 0) a -= (double)tk.g_edge * (double)s1;
      if (n == N - 1) a -= (double)tk.g_edge * (double)s0;
    }
    if (n < N) out[n] = (float)a;
    if (n + 1 < N) out[n + 1] = (float)x[j].y;
  }
}

void fft_host(std::vector<std::complex<double>>& a) {
  const size_t n = a.size();
  for (size_t i = 1, j = 0; i < n; ++i) {
    size_t bit = n >> 1;
    for (; j & bit; bit >>= 1) j ^= bit;
    j ^= bit;
    if (i < j) std::swap(a[i], a[j]);
  }
  for (size_t len = 2; len <= n; len <<= 1) {
    const double ang = -2.0 * kPi / (double)len;
    for (size_t i = 0; i < n; i += len)
      for (size_t k = 0; k < len / 2; ++k) {
        const std::complex<double> w(std::cos(ang * (double)k), std::sin(ang * (double)k));
        const std::complex<double> u = a[i + k], v = a[i + k + len / 2] * w;
        a[i + k] = u + v;
        a[i + k + len / 2] = u - v;
      }
  }
}

}  // namespace

int fft_len(int N) {
  int L = 1;
  while (L < 2 * N - 2) L <<= 1;
  return L;
}

bool fft_supported(int N) { return N >= 3 && fft_len(N) <= FFT_MAX_L; }

int fft_threads(int maxN) { return std::max(64, std::min(512, fft_len(maxN) / 16)); }

int fft_blocks(int N, int T, int threads) {
  const int rows = std::max(1, 16 * threads / std::max(16, fft_len(N)));
  return fft_len(N) < 16 ? T : (T + rows - 1) / rows;
}

void fft_tables(int N, const float* taps, double* G, double2* tw) {
  const int L = fft_len(N), M = L / 2;
  std::vector<std::complex<double>> a(L, 0.0);
  for (int m = -(N - 1); m <= N - 1; ++m) a[((m % L) + L) % L] += (double)taps[m + N];
  fft_host(a);
  for (int k = 0; k <= M; ++k) G[k] = a[k].real() / (double)M;
  auto unit = [](int k, int n) {
    const double ang = -2.0 * kPi * (double)k / (double)n;
    return make_double2(std::cos(ang), std::sin(ang));
  };
  for (int k = 0; k < M / 2; ++k) tw[k] = unit(k, M);
  for (int k = 0; k <= M / 2; ++k) tw[M / 2 + k] = unit(k, L);
}

void launch_ramp_fft(const FFTTask* d_tasks, int ntasks, int base, int blocks, int threads, hipStream_t s) {
  if (blocks <= 0) return;
  const dim3 g(xcd_grid(blocks)), t(threads);
  switch (threads) {
    case 64: hipLaunchKernelGGL(fft_ramp_kernel<64>, g, t, 0, s, d_tasks, ntasks, base, blocks); break;
    case 128: hipLaunchKernelGGL(fft_ramp_kernel<128>, g, t, 0, s, d_tasks, ntasks, base, blocks); break;
    case 256: hipLaunchKernelGGL(fft_ramp_kernel<256>, g, t, 0, s, d_tasks, ntasks, base, blocks); break;
    case 512: hipLaunchKernelGGL(fft_ramp_kernel<512>, g, t, 0, s, d_tasks, ntasks, base, blocks); break;
    default: throw Error("FFT ramp: workgroups of 64, 128, 256 or 512 threads");
  }
}

}  // namespace acu
