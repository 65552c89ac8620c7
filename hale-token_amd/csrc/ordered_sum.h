// ordered_sum.h -- a sequential f32 sum of non-negative values, by many lanes.
//
// acc = acc + v[0], acc = acc + v[1], ... rounds at every step, so its bits
// depend on the order.  As one chain it costs about 10 cycles per value
// (8.5 us for 2048 of them).  While acc stays inside one binade, though,
// every step rounds to the same unit (ulp), and what a step adds to acc
// depends on acc through one bit only: a value that ends half-way between
// two multiples of the ulp goes to the even one, so the parity of acc in
// ulps decides.  A run of K values is then a function of that parity: "d0
// ulps if acc is even, d1 if it is odd".  Two real f32 chains over the K
// values, from 2^e and from 2^e + ulp, give d0 and d1, and such functions
// compose (associatively), so 64 lanes form their K-value functions side by
// side and a wave scan joins them.
//
// Which binade a lane's values meet is known beforehand: a tree sum of the
// values up to the lane differs from the sequential sum by less than
// (values + 64) * 2^-24 of it, and the sequential sum of non-negative
// values never lies below the largest of them.  A lane whose bounds share
// one exponent is clean; the others (where the sum enters a new binade, a
// dozen lanes for a thousand values; infinities, NaN and subnormal sums)
// are walked in order, each with K real additions from the exact acc that
// reaches it.
#pragma once

#include "hale_device.h"

namespace hale {

// values one call may take (the margin below covers their rounding errors)
constexpr int ORDERED_MAX = 8192;
// LDS floats team_sum_in_order needs per team of nw waves
constexpr int ordered_lds(int nw) { return 2 * nw + 1; }

// DPP moves towards higher lanes: `id` where there is no source lane
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_up(int id, int x) {
  return __builtin_amdgcn_update_dpp(id, x, CTRL, ROWS, 0xF, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_up(float id, float x) {
  return __int_as_float(dpp_up<CTRL, ROWS>(__float_as_int(id), __float_as_int(x)));
}
// a scan step of every distance: 1, 2, 4, 8 within a row of 16 lanes, then
// the ends of rows 0 and 2, then the end of row 1
#define HALE_SCAN_STEPS(STEP) \
  STEP(0x111, 0xF) STEP(0x112, 0xF) STEP(0x114, 0xF) STEP(0x118, 0xF) STEP(0x142, 0xA) STEP(0x143, 0xC)

// acc + v_0 + v_1 + ... in order over the `nw` waves of a team, lane l of
// wave w holding the K values from (64 w + l) K on (0 past the end, at most
// ORDERED_MAX in all, each >= +0, infinite or NaN).  acc >= +0 is the sum so
// far.  Every thread of the work-group calls it together (it synchronizes
// 1 + nw times); waves from nw on add nothing, and every thread gets the sum.
template <int K>
__device__ __forceinline__ float team_sum_in_order(const float (&v)[K], float acc, int w, int nw,
                                                   float* lds) {
  // tree sums and maxima of the lanes up to this one
  float part[K];
#pragma unroll
  for (int k = 0; k < K; k++) part[k] = v[k];
#pragma unroll
  for (int s = 1; s < K; s *= 2)
#pragma unroll
    for (int k = 0; k + s < K; k += 2 * s) part[k] = part[k] + part[k + s];
  float vmax = v[0];
#pragma unroll
  for (int k = 1; k < K; k++) vmax = fmaxf(vmax, v[k]);
  const float own = part[0];
  float incl = own, top = vmax;
#define HALE_STEP(C, R)                       \
  incl = incl + dpp_up<C, R>(0.0f, incl);     \
  top = fmaxf(top, dpp_up<C, R>(0.0f, top));
  HALE_SCAN_STEPS(HALE_STEP)
#undef HALE_STEP
  if (w < nw && __lane_id() == 63) {
    lds[w] = incl;
    lds[nw + w] = top;
  }
  __syncthreads();
  float base = acc, floor_ = acc;
  for (int i = 0; i < min(w, nw); i++) {
    base = base + lds[i];
    floor_ = fmaxf(floor_, lds[nw + i]);
  }
  constexpr float MARGIN = 0x1p-10f;  // above (ORDERED_MAX + 64) * 2^-24, twice
  const float before = base + dpp_up<0x138, 0xF>(0.0f, incl);  // the lane's left neighbour
  const float least = fmaxf(before * (1.0f - MARGIN), fmaxf(floor_, dpp_up<0x138, 0xF>(0.0f, top)));
  const float most = (base + incl) * (1.0f + MARGIN);
  const int e = __float_as_int(least) & 0x7f800000;
  const bool zero = own == 0.0f;  // nothing to add, in any binade
  const bool clean = zero || (e == (__float_as_int(most) & 0x7f800000) && e != 0 && e != 0x7f800000);

  // the lane's function: what even and odd acc gain, in ulps
  float even = __int_as_float(e), odd = __int_as_float(e + 1);
#pragma unroll
  for (int k = 0; k < K; k++) {
    even = even + v[k];
    odd = odd + v[k];
  }
  int d0 = __float_as_int(even) - e, d1 = __float_as_int(odd) - (e + 1);
  if (!clean || zero) d0 = d1 = 0;
  int walk = clean ? 0 : 1;
  const unsigned long long dirty = __ballot(walk);
  // scanned from the last walked lane on (a walked lane ends its run)
#define HALE_STEP(C, R)                                                  \
  {                                                                      \
    const int l0 = dpp_up<C, R>(0, d0), l1 = dpp_up<C, R>(0, d1);        \
    const int lw = dpp_up<C, R>(0, walk);                                \
    const int j0 = l0 + (l0 & 1 ? d1 : d0), j1 = l1 + (l1 & 1 ? d0 : d1); \
    d0 = walk ? d0 : j0;                                                 \
    d1 = walk ? d1 : j1;                                                 \
    walk |= lw;                                                          \
  }
  HALE_SCAN_STEPS(HALE_STEP)
#undef HALE_STEP

  // the waves' turns, in order
  for (int turn = 0; turn < nw; turn++) {
    if (w == turn) {
      float s = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(turn ? lds[2 * nw] : acc)));
      auto run = [&](int lane) {  // the clean lanes up to `lane`
        const int b = __float_as_int(s);
        const int g0 = __builtin_amdgcn_readlane(d0, lane), g1 = __builtin_amdgcn_readlane(d1, lane);
        s = __int_as_float(b + (b & 1 ? g1 : g0));
      };
      unsigned long long m = dirty;
      while (m) {
        const int lane = __builtin_ctzll(m);
        m &= m - 1;
        if (lane) run(lane - 1);
        float t = s;
#pragma unroll
        for (int k = 0; k < K; k++) t = t + v[k];
        s = lane_value(t, lane);
      }
      run(63);
      if (__lane_id() == 0) lds[2 * nw] = s;
    }
    __syncthreads();
  }
  return lds[2 * nw];
}

}  // namespace hale
