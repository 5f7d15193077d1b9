// median_net.hpp -- a comparator network that selects the 14th smallest of
// 27 values (the median of a 3x3x3 neighbourhood), built at compile time by
// forgetful selection:
//   keep a working set of (27 + 3) / 2 = 15 values; while values remain
//   unseen, move the set's minimum and maximum out of it with
//   compare-exchanges (pair the set up, then a minimum tournament over the
//   pairs' smaller and a maximum tournament over their larger elements) --
//   with 15 values in the set the minimum has 14 larger and the maximum 14
//   smaller values, so neither is the median, and the median of the rest
//   is the median of the whole -- and bring the next value in; the last
//   three values' median is the answer.
// 153 compare-exchanges (306 min/max), against 240 for a 32-value bitonic
// sort.
//
// Neighbouring pixels share work: sort9 sorts the nine values of one image
// row of the neighbourhood once for the three pixels that see it, and
// median27_of_sorted selects the median of three sorted rows.  Of the
// rank-wise sorted triples (min3, med3, max3 of the rows' i-th values) only
// 13 values can be the median, and five 3-element operations leave it; the
// two steps were found by search over 0-1 inputs.  27 + 19 instructions.
//
// Plain C++ (no HIP), so that a host program can check both exhaustively by
// the 0-1 principle.  O supplies min3, med3 and max3 of a totally ordered V.
#pragma once

namespace acu {

struct MedianNet {
  int n = 0;                   // compare-exchanges
  unsigned char lo[160] = {};  // after exchange i: slot lo[i] holds the smaller value,
  unsigned char hi[160] = {};  // slot hi[i] the larger
  int out = 0;                 // slot of the median at the end
};

constexpr MedianNet make_median27_net() {
  MedianNet net;
  int set[27] = {};
  int size = 15, next = 15;
  for (int i = 0; i < size; ++i) set[i] = i;
  auto ce = [&net](int a, int b) {
    net.lo[net.n] = (unsigned char)a;
    net.hi[net.n] = (unsigned char)b;
    ++net.n;
  };
  while (!(size == 3 && next == 27)) {
    int lo[8] = {}, hi[8] = {}, nl = 0, nh = 0;
    for (int i = 0; i + 1 < size; i += 2) {
      ce(set[i], set[i + 1]);
      lo[nl++] = set[i];
      hi[nh++] = set[i + 1];
    }
    if (size % 2) {
      lo[nl++] = set[size - 1];
      hi[nh++] = set[size - 1];
    }
    const int mn = lo[0];
    for (int i = 1; i < nl; ++i) ce(mn, lo[i]);  // mn keeps the smallest
    const int mx = hi[0];
    for (int i = 1; i < nh; ++i)
      if (hi[i] != mn) ce(hi[i], mx);           // mx keeps the largest
    int k = 0;
    for (int i = 0; i < size; ++i)
      if (set[i] != mn && set[i] != mx) set[k++] = set[i];
    set[k++] = next++;
    size = k;
  }
  ce(set[0], set[1]);
  ce(set[1], set[2]);
  ce(set[0], set[1]);
  net.out = set[1];
  return net;
}

constexpr MedianNet MEDIAN27_NET = make_median27_net();
static_assert(MEDIAN27_NET.n == 153, "forgetful selection of the median of 27");

#ifdef __HIPCC__
#define ACU_HD __host__ __device__ __forceinline__
#else
#define ACU_HD inline
#endif

template <class O, class V>
ACU_HD void sort3(V& a, V& b, V& c) {
  const V lo = O::min3(a, b, c), mid = O::med3(a, b, c), hi = O::max3(a, b, c);
  a = lo;
  b = mid;
  c = hi;
}

// v ascending, nine 3-sorts: rows and columns of a 3 x 3 matrix, then its
// antidiagonal and the two triples that this leaves out of order
template <class O, class V>
ACU_HD void sort9(V (&v)[9]) {
  sort3<O>(v[0], v[1], v[2]);
  sort3<O>(v[3], v[4], v[5]);
  sort3<O>(v[6], v[7], v[8]);
  sort3<O>(v[0], v[3], v[6]);
  sort3<O>(v[1], v[4], v[7]);
  sort3<O>(v[2], v[5], v[8]);
  sort3<O>(v[6], v[4], v[2]);
  sort3<O>(v[3], v[6], v[1]);
  sort3<O>(v[7], v[2], v[5]);
  // ascending: 0 3 6 1 4 7 2 5 8
  V t = v[1]; v[1] = v[3]; v[3] = t;
  t = v[2]; v[2] = v[6]; v[6] = t;
  t = v[5]; v[5] = v[7]; v[7] = t;
}

// the 14th smallest of 27 in three ascending nines
template <class O, class V>
ACU_HD V median27_of_sorted(const V (&a)[9], const V (&b)[9], const V (&c)[9]) {
  auto mn = [&](int i) { return O::min3(a[i], b[i], c[i]); };
  auto md = [&](int i) { return O::med3(a[i], b[i], c[i]); };
  auto mx = [&](int i) { return O::max3(a[i], b[i], c[i]); };
  const V u = O::max3(mx(1), md(2), mn(5));
  const V w = O::min3(mx(3), md(6), mn(7));
  const V x = O::med3(mx(0), md(5), w);
  const V y = O::med3(md(3), mn(8), u);
  const V z = O::med3(mx(2), md(4), mn(6));
  return O::med3(x, y, z);
}

}  // namespace acu
