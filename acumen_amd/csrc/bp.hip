// bp.hip -- pixel-driven linear-interpolation backprojection on gfx950.
//
// Restates the second half of iradon (tomography/tv_hpc.F90:107-123):
//   yr  = sin(c)*(x-m) + cos(c)*(y-m) + m,   c = pi*(90-theta)/180
//   img(x,y) = cmask(x,y) * sum_t [S(y1,t)*(y2-yr) + S(y2,t)*(yr-y1)]
// with y1 = floor(yr), y2 = y1+1 and the taps used only when y1 > 1 and
// y2 < N+1.  Angles are summed in order, one pixel per accumulator.
//
// gfx950 mapping:
//  * one workgroup = a 64 (x) x TY (y) pixel tile, TY = 16, 32 or 64 (a
//    template parameter the autotuner picks per batch), one lane per x
//    column; 4 waves (8 for TY = 64) own 8 rows each (4 for TY = 16), so
//    one (sin, cos) pair and one LDS row serve that many updates per lane;
//  * angles are processed in blocks of 32; for each angle the tile only
//    touches a window of W detector bins (72 / 80 / 96), which is staged in
//    LDS as pairs P[t] = (S[lo+t], S[lo+t+1]-S[lo+t]) so an update is one
//    64-bit LDS read and one FMA:  S(y1) + frac*(S(y2)-S(y1));
//  * staging: 8 (16) threads per angle, each loading W/8 (W/16) pairs at
//    clamped (always in-image) positions with every load issued before the
//    first is used;
//  * a pair whose lower tap y1 violates the reference's bounds test is
//    staged as (0, 0), which reproduces the test exactly with no branch;
//  * positions (REFPOS, the default): the reference's own FP32 value,
//    yr = (s*(x-m) + c*(y-m)) + m with each product and sum rounded once and
//    no contraction, so every floor, weight and bounds decision is the
//    reference's.  Its rounding at magnitude N (~1e-4 px at N = 2049) is
//    what dominates the reference's distance from FP64 on noisy sinograms:
//    with these positions the FBP is ~1e-6 from the reference's FP32 FBP,
//    with exact positions ~2.7e-5 (noisy 2049^2 x 1500);
//  * positions (!REFPOS, ACUMEN_BP_POSITIONS=tile): relative to the tile
//    origin, yr - 1 - lo = s*xl + c*yl + K with xl < 64, yl < TY and
//    K = s*(x0+1-m) + c*(y0+1-m) + m-1-lo formed in FP64 once per angle and
//    tile, so a position is rounded at magnitude below ~100: closer to FP64,
//    farther from the reference, two VALU fewer per update;
//    in both, y1 = floor(yr) and the pair's LDS offset come from v_fract and
//    full-rate float arithmetic (lds_units) instead of v_cvt and
//    v_lshl_add: 551 against 575 us per 4 x 1025^2 x 720 launch, 6.23
//    against 6.34 ms per 8 x 2049^2 x 1500;
//  * REFPOS keeps scalar loads out of the loop over angles: the rows' terms,
//    the sine and the window's base come from LDS, which answers in order,
//    so the wait for one half of the rows' taps leaves the other half's and
//    the next angle's in flight (a scalar load outstanding turns every such
//    wait into a wait for all).  8 x 2049^2 x 1500 6.33 to 5.75 ms, 2 x
//    1025^2 x 720 at TY = 16 360 to 260 us;
//  * a pair of slices of one geometry (G = 2, REFPOS) shares positions,
//    weights and offsets: 4.2 VALU instructions an update instead of 7.  The
//    windows are two arrays read by two ds_read_b64 (2.2 clocks each; one
//    ds_read2st64_b64 takes 8, a b128 of interleaved pairs 5.9 with its bank
//    conflicts), staged 16 angles at a time so that 5 workgroups fit a CU.
//    8 x 2049^2 x 1500 5.75 to 5.0 ms, and 4.6 with five waves per SIMD instead
//    of four: 1.45 wave-instructions per CU and clock, LDS active 75% of the
//    cycles, at 1.83 GHz: the power limit is near as well;
//  * each 32-angle block is summed separately and then added;
//  * tiles whose mask is identically zero (by 64 x 16 sub-tiles) only store
//    zeros.
#include "acu_internal.hpp"

#include <algorithm>

namespace acu {
namespace {

constexpr int TX = BP_TX, AB = BP_AB;
constexpr int bp_waves(int ty) { return ty == 64 ? 8 : 4; }

// Detector bins staged per angle at tile height ty.  Over a 64 x ty tile the
// positions span at most hypot(63, ty-1) bins; the window starts at least
// one bin (less FP32 rounding) below the lowest position, and a sample at
// local position t reads pair t, so W >= hypot(63, ty-1) + 3.01 suffices
// (67.8, 73.2, 92.1); W is a multiple of the staging threads per angle.
constexpr int bp_window(int ty) { return ty == 16 ? 72 : ty == 32 ? 80 : 96; }

__device__ __forceinline__ int find_task(const BPTask* tasks, int ntasks, int gtile) {
  int lo = 0, hi = ntasks - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (tasks[mid].tile_begin <= gtile) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// LDS of a workgroup: AS angles' pairs (of two slices if G = 2), window starts,
// constants and row terms.
template <int TY, bool REFPOS, int G>
struct BPLds {
  static constexpr int AS = G == 2 ? 16 : AB;  // angles staged at a time (G = 1 with 16: 2% slower)
  static constexpr int W = (G == 2 && TY == 16) ? 80 : bp_window(TY);
  // second slice's window; not a multiple of 512 bytes, which would merge the reads
  static constexpr int P2 = AS * W + 1;
  float2 P[G == 2 ? P2 + AS * W : AS * W];
  float2 ab[REFPOS ? AS : 1];  // sine, LDS offset of P[a * W - 1 - lo] (lds_units)
  __attribute__((aligned(16))) float rt[REFPOS ? AS * TY : 1];  // row terms of the tile
  int lo[AS];
  float k[AS];  // K of the tile-local position (see above)
};

// Tile `local` of a task, its G slices together.
template <int TY, bool REFPOS, int G>
__device__ __forceinline__ void bp_tile(const BPTask& tk, int local, BPLds<TY, REFPOS, G>& lds) {
  typedef BPLds<TY, REFPOS, G> L;
  constexpr int NW = bp_waves(TY), NT = 64 * NW, PY = TY / NW, SUBS = TY / BP_SUB;
  constexpr int AS = L::AS, W = L::W, P2 = L::P2;
  constexpr int SPA = NT / AS, NST = W / SPA;  // staging threads per angle, pairs per thread
  static_assert(G == 1 || (G == 2 && REFPOS), "pairs have the reference's positions");
  static_assert(TY % BP_SUB == 0 && TY % NW == 0 && NT % AS == 0 && W % SPA == 0 && AB % AS == 0, "tile shape");
  float2* const P = lds.P;
  int* const lo_s = lds.lo;
  float* const k_s = lds.k;
  float* const rt_s = lds.rt;
  float2* const ab_s = lds.ab;
  const int N = tk.N, T = tk.T;
  const float m = tk.mid;
  const int tx = local % tk.ntx, tyi = local / tk.ntx;
  const int x0 = tx * TX, y0 = tyi * TY;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int x = x0 + lane;
  const int yb = y0 + wave * PY;

  bool active = false;
#pragma unroll
  for (int j = 0; j < SUBS; ++j) {
    const int r16 = tyi * SUBS + j;
    if (r16 < tk.nsub) active = active || tk.tile_active[r16 * tk.ntx + tx] != 0;
  }
  if (!active) {
    if (x < N) {
#pragma unroll
      for (int r = 0; r < PY; ++r)
        if (yb + r < N) {
          tk.img[(size_t)(yb + r) * N + x] = 0.0f;
          if (G == 2) tk.img2[(size_t)(yb + r) * N + x] = 0.0f;
        }
    }
    return;
  }

  // tile-local coordinates, exact in fp32
  const float xl = (float)lane;
  float yl[PY];
#pragma unroll
  for (int r = 0; r < PY; ++r) yl[r] = (float)(wave * PY + r);
  // the reference's jx - midpoint (1-based), exact in fp32
  const float ux = (float)(x + 1) - m;
  // tile corners (1-based) for the staging windows
  const float cx0 = (float)(x0 + 1) - m, cx1 = (float)(x0 + TX) - m;
  const float cy0 = (float)(y0 + 1) - m, cy1 = (float)(y0 + TY) - m;

  float acc[G][PY];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int r = 0; r < PY; ++r) acc[g][r] = 0.0f;

  const ACU_GLOBAL float* __restrict__ S[2] = {as_global(tk.sino), as_global(G == 2 ? tk.sino2 : tk.sino)};
  const float2* __restrict__ sc = tk.sc;
  const int sa = tid / SPA, sj = tid % SPA;  // staging: angle of the block, first bin

  float blk[G][PY];  // the 32-angle block's sums
  for (int a0 = 0; a0 < T; a0 += AS) {
    const int na = min(AS, T - a0);
    // window start per angle: lowest 0-based detector position over the tile, minus one bin
    if (tid < na) {
      const float2 v = const_f2(sc, a0 + tid);
      const float ex = fminf(v.x * cx0, v.x * cx1);
      const float ey = fminf(v.y * cy0, v.y * cy1);
      const int lo = (int)floorf(ex + ey + m - 1.0f) - 1;
      lo_s[tid] = lo;
      if (!REFPOS)
        k_s[tid] = (float)((double)v.x * (double)cx0 + (double)v.y * (double)cy0 + (double)m - 1.0 -
                         (double)lo);
      if (REFPOS) ab_s[tid] = make_float2(v.x, lds_base(8 * (tid * W - 1 - lo)));
    }
    if (REFPOS) {
#pragma unroll
      for (int i = 0; i < AS * TY; i += NT) {
        const int a = (i + tid) / TY, r = (i + tid) % TY;
        // rows past the image (not stored) as its last: positions in the window
        rt_s[i + tid] = as_global(tk.rowterm)[(size_t)min(a0 + a, T - 1) * N + min(y0 + r, N - 1)];
      }
    }
    __syncthreads();
    if (sa < na) {
      const int lo = lo_s[sa];
      float2 v[G][NST];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const ACU_GLOBAL float* row = S[g] + (size_t)(a0 + sa) * N;
#pragma unroll
        for (int k = 0; k < NST; ++k) {
          const int dc = min(max(lo + sj + SPA * k, 1), N - 2);  // N >= 3: row[dc + 1] is in the row
          v[g][k] = make_float2(row[dc], row[dc + 1]);
        }
      }
#pragma unroll
      for (int k = 0; k < NST; ++k) {
        const int d = lo + sj + SPA * k;
        const bool in = d >= 1 && d <= N - 2;
#pragma unroll
        for (int g = 0; g < G; ++g)
          P[g * P2 + sa * W + sj + SPA * k] = in ? make_float2(v[g][k].x, v[g][k].y - v[g][k].x) : make_float2(0.0f, 0.0f);
      }
    }
    __syncthreads();
    if (a0 % AB == 0) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int r = 0; r < PY; ++r) blk[g][r] = 0.0f;
    }
    if (REFPOS) {
#pragma clang fp contract(off)
      // the rows in two halves: one half's taps are in flight while the other
      // half's (of the angle before, at first) are added
      constexpr int H = PY / 2;
      float2 q[2][H][G];
      float fr[2][H];
#pragma unroll
      for (int h = 0; h < H; ++h) {
        fr[1][h] = 0.0f;
#pragma unroll
        for (int g = 0; g < G; ++g) q[1][h][g] = make_float2(0.0f, 0.0f);
      }
      const float* rts = rt_s + wave * PY;
      for (int a = 0; a < na; ++a) {
        const float2 ab = ab_s[a];
        float rv[PY];
#pragma unroll
        for (int r = 0; r < PY; ++r) rv[r] = rts[a * TY + r];
        const float A = ab.x * ux;  // sin(c)*(jx-midpoint), tv_hpc.F90:114
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
          for (int h = 0; h < H; ++h) {
            const float yr = (A + rv[u * H + h]) + m;  // (sin(c)*(jx-m) + cos(c)*(jy-m)) + m
            // yr - y1; y1 = floor(yr) = yr - fr, both exact
            fr[u][h] = __builtin_amdgcn_fractf(yr);
            const unsigned o = __float_as_uint(fmaf(yr - fr[u][h], lds_units(8), ab.y));
#pragma unroll
            for (int g = 0; g < G; ++g) q[u][h][g] = *(const float2*)((const char*)(P + g * P2) + o);
          }
#pragma unroll
          for (int h = 0; h < H; ++h)
#pragma unroll
            for (int g = 0; g < G; ++g)
              blk[g][(1 - u) * H + h] += fmaf(fr[1 - u][h], q[1 - u][h][g].y, q[1 - u][h][g].x);
        }
      }
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int g = 0; g < G; ++g) blk[g][H + h] += fmaf(fr[1][h], q[1][h][g].y, q[1][h][g].x);
    } else {
      for (int a = 0; a < na; ++a) {
        const float2 v = const_f2(sc, a0 + a);
        const float base = fmaf(v.x, xl, k_s[a]);
        const float Pa = lds_base(8 * a * W);
#pragma unroll
        for (int r = 0; r < PY; ++r) {
          const float yr = fmaf(v.y, yl[r], base);  // detector position - 1 - lo, in (0, W - 1)
          const float fr = __builtin_amdgcn_fractf(yr);
          const unsigned o = __float_as_uint(fmaf(yr - fr, lds_units(8), Pa));
          const float2 pv = *(const float2*)((const char*)P + o);
          blk[0][r] += fmaf(fr, pv.y, pv.x);
        }
      }
    }
    if (a0 % AB == AB - AS || a0 + AS >= T) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int r = 0; r < PY; ++r) acc[g][r] += blk[g][r];
    }
    __syncthreads();
  }

  if (x < N) {
#pragma unroll
    for (int r = 0; r < PY; ++r) {
      const int y = yb + r;
      if (y < N) {
        const size_t o = (size_t)y * N + x;
        const float cm = tk.cmask[o];
        tk.img[o] = cm * acc[0][r];
        if (G == 2) tk.img2[o] = cm * acc[G - 1][r];
      }
    }
  }
}

template <int TY, bool REFPOS, bool PAIRS>
constexpr int bp_lds() {
  const int a = sizeof(BPLds<TY, REFPOS, 1>), b = sizeof(BPLds<TY, REFPOS, PAIRS ? 2 : 1>);
  return a > b ? a : b;
}

// PAIRS: tasks of two slices (sino2) beside tasks of one, each at its own
// width.  Five waves per SIMD (96 registers instead of 101) for those.
template <int TY, bool REFPOS, bool PAIRS>
__global__ __launch_bounds__(64 * bp_waves(TY), PAIRS ? 5 : 1) void bp_kernel(const BPTask* __restrict__ tasks,
                                                                              int ntasks, int base, BPShares sh) {
  typedef BPLds<TY, REFPOS, 1> L1;
  typedef BPLds<TY, REFPOS, PAIRS ? 2 : 1> L2;
  __shared__ __attribute__((aligned(16))) char lds[bp_lds<TY, REFPOS, PAIRS>()];
  // XCD k (xcd_remap) runs the tiles of its share in order
  const int l = xcd_remap(blockIdx.x, gridDim.x);
  const int k = l / sh.C;
  const int lt = sh.b[k] + (l - k * sh.C);
  if (lt >= sh.b[k + 1]) return;
  const int gtile = base + lt;
  const BPTask& tk = tasks[find_task(tasks, ntasks, gtile)];
  const int local = gtile - tk.tile_begin;
  if constexpr (PAIRS) if (tk.sino2) return bp_tile<TY, REFPOS, 2>(tk, local, *(L2*)lds);
  bp_tile<TY, REFPOS, 1>(tk, local, *(L1*)lds);
}

// Backprojection of the smallest launches, with the reference's positions.  A
// tile of the kernel above walks its angles serially, so its time grows with
// T even where most CUs are idle (a 257^2 slice is 85 workgroups of 64 x 16).
// Here a workgroup of 8 waves takes a 64 x 8 tile and every wave another
// block of 32 angles: each stages its own window in its own part of LDS
// (BPS_AB angles at a time, no barrier), and the blocks' sums are then added
// in block order, so the result is the other kernel's bit for bit (but for
// the sign of the zeros it stores off the mask, as between that kernel's tile
// heights).  A staged pair serves 8 rows instead of 16 or more, so a fuller
// GPU is better off with the other kernel.
constexpr int BPS_WAVES = 8;  // waves of a workgroup, one angle block each
constexpr int BPS_AB = 8;     // angles staged at a time, 8 lanes each
constexpr int BPS_ROWS = 8;   // rows of a tile
constexpr int BPS_W = 72;     // window of 64 x 8 pixels: hypot(63, 7) + 3.01 = 66.4

__device__ __forceinline__ int find_split_task(const BPTask* tasks, int ntasks, int gtile) {
  int lo = 0, hi = ntasks - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (tasks[mid].split_begin <= gtile) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__global__ __launch_bounds__(64 * BPS_WAVES) void bp_split_kernel(const BPTask* __restrict__ tasks, int ntasks,
                                                                  int base, int ntiles) {
  constexpr int ROWS = BPS_ROWS, W = BPS_W, NST = W / 8, OWN = ROWS / BPS_WAVES;  // OWN: rows a wave adds up
  static_assert(AB % BPS_AB == 0 && W % 8 == 0 && ROWS % BPS_WAVES == 0 && ROWS <= BP_SUB, "tile shape");
  static_assert(ROWS * 64 <= 2 * BPS_AB * W, "a wave's block sums fit its pairs' space");
  __shared__ float2 Ps[BPS_WAVES][BPS_AB * W];
  const int l = xcd_remap(blockIdx.x, gridDim.x);
  if (l >= ntiles) return;  // uniform per workgroup
  const BPTask& tk = tasks[find_split_task(tasks, ntasks, base + l)];
  const int N = tk.N, T = tk.T;
  const float m = tk.mid;
  const int local = base + l - tk.split_begin;
  const int tx = local % tk.ntx, ty = local / tk.ntx;
  const int x0 = tx * TX, y0 = ty * ROWS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int x = x0 + lane, yo = y0 + wave * OWN;  // the pixels this thread stores: x, rows yo .. yo + OWN - 1
  // y0 / BP_SUB < nsub but for the tiles past the image's last rows, which store nothing
  if (y0 >= N) return;
  if (!tk.tile_active[(y0 / BP_SUB) * tk.ntx + tx]) {
#pragma unroll
    for (int r = 0; r < OWN; ++r)
      if (x < N && yo + r < N) tk.img[(size_t)(yo + r) * N + x] = 0.0f;
    return;
  }
  const float ux = (float)(x + 1) - m;
  const float cx0 = (float)(x0 + 1) - m, cx1 = (float)(x0 + TX) - m;
  const float cy0 = (float)(y0 + 1) - m, cy1 = (float)(y0 + ROWS) - m;
  float2* P = Ps[wave];
  float* part = (float*)P;  // the wave's 8 x 64 block sums, once its pairs are read
  const ACU_GLOBAL float* __restrict__ S = as_global(tk.sino);
  const ACU_GLOBAL float* __restrict__ sc = as_global((const float*)tk.sc);
  const int nblk = (T + AB - 1) / AB;

  float acc[OWN];
#pragma unroll
  for (int r = 0; r < OWN; ++r) acc[r] = 0.0f;
  for (int b0 = 0; b0 < nblk; b0 += BPS_WAVES) {
    const int b = b0 + wave;
    float blk[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) blk[r] = 0.0f;
    for (int a0 = b * AB; a0 < min(T, (b + 1) * AB); a0 += BPS_AB) {
      const int na = min(BPS_AB, T - a0);
      // lane l (mod BPS_AB) holds angle a0 + l: sine, cosine and window start
      const int t = min(a0 + (lane & (BPS_AB - 1)), T - 1);
      const float hs = sc[2 * t], hc = sc[2 * t + 1];
      const int hlo = (int)floorf(fminf(hs * cx0, hs * cx1) + fminf(hc * cy0, hc * cy1) + m - 1.0f) - 1;
      // staging: 8 lanes per angle, their loads issued before the first is used
      const int q = lane >> 3, j = lane & 7, lo = __shfl(hlo, q) + j;
      const ACU_GLOBAL float* row = S + (size_t)min(a0 + q, T - 1) * N;
      float2 v[NST];
#pragma unroll
      for (int k = 0; k < NST; ++k) {
        const int dc = min(max(lo + 8 * k, 1), N - 2);  // N >= 3: row[dc + 1] is in the row
        v[k] = make_float2(row[dc], row[dc + 1]);
      }
#pragma unroll
      for (int k = 0; k < NST; ++k) {
        const int d = lo + 8 * k;
        P[q * W + j + 8 * k] = (d >= 1 && d <= N - 2) ? make_float2(v[k].x, v[k].y - v[k].x) : make_float2(0.0f, 0.0f);
      }
      __builtin_amdgcn_wave_barrier();  // one wave: its LDS operations are in order
      for (int a = 0; a < na; ++a) {
#pragma clang fp contract(off)
        const float sn = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hs), a));
        const float cs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hc), a));
        const float A = sn * ux;
        const float ob = lds_base(8 * (a * W - 1 - __builtin_amdgcn_readlane(hlo, a)));
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
          const float yr = (A + cs * ((float)(y0 + r + 1) - m)) + m;
          const float fr = __builtin_amdgcn_fractf(yr);
          const unsigned o = __float_as_uint(fmaf(yr - fr, lds_units(8), ob));
          const float2 pv = *(const float2*)((const char*)P + o);
          blk[r] += fmaf(fr, pv.y, pv.x);
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) part[r * 64 + lane] = blk[r];
    __syncthreads();
    for (int k = 0; k < min(BPS_WAVES, nblk - b0); ++k)
#pragma unroll
      for (int r = 0; r < OWN; ++r) acc[r] += ((const float*)Ps[k])[(wave * OWN + r) * 64 + lane];
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < OWN; ++r)
    if (x < N && yo + r < N) {
      const size_t o = (size_t)(yo + r) * N + x;
      tk.img[o] = tk.cmask[o] * acc[r];
    }
}

}  // namespace

int bp_split_tiles(int N) { return bp_tiles_x(N) * ((N + 15) / 16) * 2; }

// us per FBP (host call and ramp included), MI355X: this kernel | 64 x 16 |
// 64 x 32 tiles of bp_kernel, by the launch's 64 x 8 tiles:
//   20 (65^2) x 48 19 | 16 | 21, x 100 19 | 24 | 33, x 180 21 | 34 | 50;
//   54 (129^2) x 64 20 | 19 | 25, x 90 20 | 23 | 31;
//   170 (257^2) x 60 19 | 18 | 24, x 180 21 | 35 | 51;
//   594 (513^2) x 360 58 | 61 | 93;      680 (4 x 257^2) x 180 34 | 35 | 51;
//   1274 (769^2) x 600 133 | 111 | 150;  2720 (16 x 257^2) x 180 74 | 54 | 66
// and 64 x 16 | 64 x 32 | 64 x 64 tiles of bp_kernel:
//   2210 (1025^2) x 720 176 | 223 | 245; 4752 (8 x 513^2) x 720 251 | 330 | 371;
//   4850 (1537^2) x 900 344 | 394 | 418; 5096 (4 x 769^2) x 600 215 | 287 | 316.
// From about there on taller tiles win in part, so the height is as set (the
// autotuner's to choose): 6630 (3 x 1025^2) x 720 335 | 372 | 344; 8514 (2049^2) x
// 1500 832 | 892 | 927; 8840 (4 x 1025^2) x 720 414 | 396 | 373
bool bp_use_split(int tiles, int T) { return tiles <= 640 && T > 64; }
int bp_launch_height(int tiles, int ty) { return tiles <= 5200 ? 16 : ty; }
// us per FBP without | with pairs, by the launch's 64 x 8 tiles (heights 16 up
// to 5200, then 32): 1188 (2 x 513^2) x 360 70 | 90; 1360 (8 x 257^2) x 180 40 |
// 51; 2376 (4 x 513^2) x 360 95 | 104; 2548 (2 x 769^2) x 600 153 | 152; 3456 (64 x
// 129^2) x 90 35 | 37; 4080 (24 x 257^2) x 180 69 | 63; 5096 (4 x 769^2) x 600
// 251 | 215; 8840 (4 x 1025^2) x 720 478 | 393; 68112 (8 x 2049^2) x 1500 6250 |
// 4790.  A pair's tile takes 1.54 times as long, so a few pairs among single
// slices lengthen the launch's end more than they shorten the rest: by share
// of the tiles in pairs 0.2% (2 x 65^2 x 1500 + 3 x 2049^2 x 300) 475 | 552, 10%
// (2 equal of 20 x 1025^2 x 720) 1891 | 1890, 20% (2 equal of 10 x 513^2 x 720) 376
// | 386, 57% (4 equal of 7 x 1025^2 x 720) 713 | 663, 80% (16 of 20) 1890 | 1607;
// and where a slice is left over in launches of few tiles: 6370 (5 x 769^2 x 600)
// 318 | 331, 6534 (11 x 513^2 x 360) 197 | 204, 8918 (7 x 769^2 x 600) 411 | 389,
// 25542 (3 x 2049^2 x 1500) 2299 | 2005.  Pairs and singles share a launch: in one
// of each kind, the first's end waits for nobody (990 for the 0.2%, 5 x 2049^2 x
// 1500 3450 instead of 3190).
bool bp_use_pairs(int tiles, int paired) { return tiles >= (paired < tiles ? 8500 : 3500) && 2 * (long)paired >= tiles; }

void launch_backproject_split(const BPTask* d_tasks, int ntasks, int base, int tiles, hipStream_t s) {
  if (tiles <= 0) return;
  hipLaunchKernelGGL(bp_split_kernel, dim3(xcd_grid(tiles)), dim3(64 * BPS_WAVES), 0, s, d_tasks, ntasks, base, tiles);
}

__global__ __launch_bounds__(256) void rowterm_kernel(const float2* __restrict__ sc, int N, int T, float mid,
                                                      float* __restrict__ out) {
#pragma clang fp contract(off)
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)N * T + BP_ROWTERM_PAD) return;
  const int t = (int)(i / N), y = (int)(i - (size_t)t * N);
  out[i] = t < T ? sc[t].y * ((float)(y + 1) - mid) : 0.0f;
}

void launch_bp_rowterm(const float2* sc, int N, int T, float mid, float* rowterm, hipStream_t s) {
  const size_t n = (size_t)N * T + BP_ROWTERM_PAD;
  hipLaunchKernelGGL(rowterm_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, sc, N, T, mid, rowterm);
}

int bp_tiles_x(int N) { return (N + TX - 1) / TX; }
int bp_tiles_y(int N, int ty) { return (N + ty - 1) / ty; }

// LDS to ask for on top of a kernel's `own`, so that an XCD whose `share` of
// workgroups (of those that do not only store zeros) fits its 32 CUs at once
// spreads them evenly: no CU has room for more than its part.  Without it some
// CUs fill up and the launch waits for those: us per FBP without | with, 4 x
// 1025^2 x 720 444 | 393, 8 x 769^2 x 600 396 | 355, 16 x 513^2 x 360 238 | 210, 4
// x 769^2 x 600 (16 rows) 244 | 215.  No fewer than 3 to a CU (64 x 129^2 x 90 37
// with more, 52 with 2).
int bp_pad(int share, int own) {
  constexpr int CUS = 32, LDS = 160 << 10, GRAIN = 1280;
  if (share <= 0) return 0;
  const int k = std::max(3, (share + CUS - 1) / CUS);
  const int total = LDS / k - GRAIN;  // k fit, k + 1 do not
  return total > own ? total - own : 0;
}

template <int TY, bool REFPOS, bool PAIRS>
void launch_bp_ty(const BPTask* d_tasks, int ntasks, int base, const BPShares& sh, int share, hipStream_t s) {
  int pad = 0;
  if (PAIRS) pad = bp_pad(share, bp_lds<TY, REFPOS, PAIRS>());
  hipLaunchKernelGGL((bp_kernel<TY, REFPOS, PAIRS>), dim3((unsigned)(XCDS * sh.C)), dim3(64 * bp_waves(TY)), pad, s, d_tasks,
                     ntasks, base, sh);
}
template <bool REFPOS, bool PAIRS>
void launch_bp(const BPTask* d_tasks, int ntasks, int base, int ty, const BPShares& sh, int share, hipStream_t s) {
  switch (ty) {
    case 16: launch_bp_ty<16, REFPOS, PAIRS>(d_tasks, ntasks, base, sh, share, s); break;
    case 32: launch_bp_ty<32, REFPOS, PAIRS>(d_tasks, ntasks, base, sh, share, s); break;
    case 64: launch_bp_ty<64, REFPOS, PAIRS>(d_tasks, ntasks, base, sh, share, s); break;
    default: throw Error("backprojection tile height must be 16, 32 or 64");
  }
}

void check_bp_launch(const BPTask* d_tasks, int ntasks, int tiles, const BPShares& sh) {
  if (!d_tasks || ntasks < 1 || sh.b[0] != 0 || sh.b[XCDS] != tiles || sh.C < 1) throw Error("backprojection tasks or shares do not match the launch");
}

void launch_backproject(const BPTask* d_tasks, int ntasks, int base, int tiles, int ty, bool refpos,
                        const BPShares& sh, hipStream_t s) {
  if (tiles <= 0) return;
  check_bp_launch(d_tasks, ntasks, tiles, sh);
  if (refpos) launch_bp<true, false>(d_tasks, ntasks, base, ty, sh, 0, s);
  else launch_bp<false, false>(d_tasks, ntasks, base, ty, sh, 0, s);
}

void launch_backproject_pairs(const BPTask* d_tasks, int ntasks, int tiles, int share, int ty, const BPShares& sh,
                              hipStream_t s) {
  if (tiles <= 0) return;
  check_bp_launch(d_tasks, ntasks, tiles, sh);
  launch_bp<true, true>(d_tasks, ntasks, 0, ty, sh, share, s);
}

// Cut points at k/XCDS of the total estimated work (a tile starts the next
// share once the work before it reaches the share's target), so the shares
// are contiguous runs of the launch's tiles with about equal work; with 8
// equal slices each XCD gets one slice.
BPShares bp_xcd_shares(const std::vector<float>& w) {
  BPShares sh{};
  const int n = (int)w.size();
  double tot = 0.0;
  for (float v : w) tot += v;
  int k = 1;
  double acc = 0.0;
  for (int i = 0; i < n && k < XCDS; ++i) {
    while (k < XCDS && acc >= tot * k / XCDS - 1e-9 * tot) sh.b[k++] = i;
    acc += w[i];
  }
  while (k < XCDS) sh.b[k++] = n;
  sh.b[0] = 0;
  sh.b[XCDS] = n;
  sh.C = 1;
  for (int j = 0; j < XCDS; ++j) sh.C = std::max(sh.C, sh.b[j + 1] - sh.b[j]);
  return sh;
}

}  // namespace acu
