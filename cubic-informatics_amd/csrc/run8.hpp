// run8.hpp -- passes along one axis with the radius at run time, eight outputs at a time: each
// input is read once per group of eight, and the taps that all eight share are taken together.
// next() gives the inputs c - r, c - r + 1, ... c + 7 + r in order; R > 0 fixes the radius, for
// windows shorter than the group (r <= 3), R = 0 takes r >= 4 at run time.  A work-group of
// four waves walks its lines, or the rows of a strip of 64 columns, with the last 2r + 32
// positions in LDS.
#ifndef HDOG_RUN8_HPP
#define HDOG_RUN8_HPP
#include "hdog_internal.hpp"

namespace hdog {
namespace {

constexpr int OK = 8;
constexpr int kRunRadius = 24;

// acc[o] = 0 + input o + input o + 1 ... + input o + 2r, in that order
template <int R, typename F>
__device__ __forceinline__ void sum8(F&& next, int r, float (&acc)[OK]) {
#pragma unroll
  for (int o = 0; o < OK; ++o) acc[o] = 0.0f;
  if constexpr (R > 0) {
    float v[2 * R + OK];
#pragma unroll
    for (int i = 0; i < 2 * R + OK; ++i) v[i] = next();
#pragma unroll
    for (int i = 0; i < 2 * R + OK; ++i)
#pragma unroll
      for (int o = 0; o < OK; ++o)
        if (i - o >= 0 && i - o <= 2 * R) acc[o] += v[i];
  } else {
    float h[OK - 1], v[4], e[OK - 1];
#pragma unroll
    for (int i = 0; i < OK - 1; ++i) h[i] = next();
#pragma unroll
    for (int q = 0; q < 2; ++q) v[q] = next();
#pragma unroll
    for (int i = 0; i < OK - 1; ++i)
#pragma unroll
      for (int o = 0; o <= i; ++o) acc[o] += h[i];
    // inputs 7 .. 2r meet all eight (an even number), two always read ahead
    int i = OK - 1;
#pragma unroll 1
    for (; i + 3 <= 2 * r; i += 2) {
#pragma unroll
      for (int q = 2; q < 4; ++q) v[q] = next();
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int o = 0; o < OK; ++o) acc[o] += v[q];
      v[0] = v[2];
      v[1] = v[3];
    }
#pragma unroll
    for (int q = 0; q < OK - 1; ++q) e[q] = next();
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int o = 0; o < OK; ++o) acc[o] += v[q];
#pragma unroll
    for (int u = 1; u < OK; ++u)
#pragma unroll
      for (int o = u; o < OK; ++o) acc[o] += e[u - 1];
  }
}

// Where a work-group of four waves stands on its lines: 64 x-adjacent lines, eight positions
// per wave and step of 32.
struct RunAt {
  int l, wave, x0, s0, s1;
  i64 base;
};
__device__ __forceinline__ RunAt run_at(int L, i64 so, unsigned nxb, unsigned no, int len) {
  RunAt a;
  a.l = (int)(threadIdx.x & 63);
  a.wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  a.x0 = (int)(t % nxb) * 64;
  a.base = (i64)(t / nxb % no) * so;
  a.s0 = (int)(t / nxb / no) * len;
  a.s1 = min(L, a.s0 + len);
  return a;
}

// f with the radius fixed for windows shorter than a group of outputs, else 0
template <typename F>
hipError_t dispatch_short(int r, F&& f) {
  static_assert(OK == 8, "2 * 3 + 1 < 8");
  switch (r) {
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    default: return f(std::integral_constant<int, 0>{});
  }
}
// grid of a walk over 64-line strips by work-groups of four waves
LineGrid run_grid(int W, int L, i64 n_other, int halo) {
  LineGrid g;
  g.nxb = (unsigned)((W + 63) / 64);
  g.no = (unsigned)n_other;
  int nseg;
  line_segments(L, (i64)g.nxb * n_other * 4, 1024.0, 2.0, false, halo, &nseg, &g.len);
  g.blocks = (unsigned)((i64)g.nxb * n_other * nseg);
  return g;
}

}  // namespace
}  // namespace hdog
#endif
