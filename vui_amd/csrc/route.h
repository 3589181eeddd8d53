// The choice of experts of one row, shared by the routing launches and the row kernel.
#pragma once
#include "lm.h"

__device__ __forceinline__ void route_choose(const RouteArgs& p, int m, int c, int e) {
  p.choice[(size_t)m * p.top + c] = e;
}
// One wave; z: the row's logits.  Up to 64 experts: a maximum over the wave per choice, a logit per lane (2.1 us for 4 of 32 when every lane
// ranked its own among all); more: picks in order of falling logits, so that "behind the last pick" needs no
// list of what was taken.  A NaN is never chosen; what is missing then is expert 0 with the weight of -inf.
__device__ __forceinline__ void route_row(const RouteArgs& p, int m, const float* z) {
  const int lane = threadIdx.x & 63;
  if (p.E <= 64) {
    const float v = lane < p.E ? z[lane] : 0.f;
    uint64_t left = __builtin_amdgcn_ballot_w64(lane < p.E && v == v);
    float vmax = -INFINITY, w = 0.f, none = 0.f, sum = 0.f, mine = 0.f;
    for (int c = 0; c < p.top; ++c) {
      const float mx = wave_max(left >> lane & 1 ? v : -INFINITY);
      const uint64_t who = __builtin_amdgcn_ballot_w64(v == mx) & left;
      const int e = who ? __builtin_ctzll(who) : 0;
      left &= ~(1ull << e);
      if (c == 0) {
        if (who) vmax = mx;
        w = expf(v - vmax); none = expf(-INFINITY - vmax);
      }
      const float wc = who ? lane_f(w, e) : none;
      sum += wc;
      if (lane == c) { mine = wc; route_choose(p, m, c, e); }
    }
    if (lane < p.top) p.share[(size_t)m * p.top + lane] = mine / sum;
    return;
  }
  float last = INFINITY, vmax = 0.f, sum = 0.f, mine = 0.f;
  int last_e = -1;
  for (int c = 0; c < p.top; ++c) {
    float bv = -INFINITY;
    int be = 0x7fffffff;
    for (int e = lane; e < p.E; e += 64) {
      const float v = z[e];
      if ((v < last || (v == last && e > last_e)) && (v > bv || be == 0x7fffffff)) { bv = v; be = e; }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const float ov = __shfl_xor(bv, o);
      const int oe = __shfl_xor(be, o);
      if (oe != 0x7fffffff && (be == 0x7fffffff || ov > bv || (ov == bv && oe < be))) { bv = ov; be = oe; }
    }
    if (c == 0) vmax = bv;
    const float w = expf(bv - vmax);
    sum += w;
    if (lane == c) mine = w;
    if (lane == 0) route_choose(p, m, c, be < p.E ? be : 0);
    last = bv;
    last_e = be;
  }
  if (lane < p.top) p.share[(size_t)m * p.top + lane] = mine / sum;
}
