// normalize.hip -- local contrast normalization on gfx950.
//
// Reference semantics: src/3D/NormalizeFilter.cu:53-654.
//   E = box_mean(min_filter(I)), D = box_mean(max_filter(I)), both with clamp-to-edge
//   borders and the same radius for the min/max window and the box;
//   norm = I >= min_intensity ? (I - E) / (D - E) : 0.
//
// MI355X design:
//   * Erosion and dilation run together: each voxel is packed into one 32-bit word
//     (v, 65535 - v) so a single v_pk_min_u16 advances both filters (max(v) =
//     65535 - min(65535 - v)).
//   * Min/max over a clamped box is separable and exact in any order, so the y and z
//     passes run first (in one z walk for radius 10, k_minmax_zy_walk, and for most others,
//     k_minmax_zy_run; else z then y) and the x pass is fused with the box filter along x (sums
//     of integers, exact in any order, so a sliding sum is used) and y.  The y and z box passes
//     sum FP32 values and keep the reference's sequential order (c-r .. c+r); the z pass is
//     fused with the normalization.
//   * Radius 10 has column walkers along z (one thread per line, a compile-time-sized register
//     ring, every input read once, no LDS) and a row walker along x and y.  Other radii up to
//     kRunRadius, and stacks too small for the row walker, have walks with the radius at run time
//     and their history in LDS; lines of a few positions are a thread's registers, and planes
//     of a few rows have their x and y passes apart.  Larger radii take LDS tiles, min/max by
//     van Herk / Gil-Werman (3 packed mins per output).
#include "run8.hpp"

namespace hdog {
namespace {

constexpr int NT = 256;
// slices of raw input in flight per thread in the fused y / z min/max walk (a divisor of
// the z window 2 RZ + 1)
#ifndef HDOG_ZY_PF
#define HDOG_ZY_PF 3
#endif
typedef unsigned short us2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pkmin(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(us2, a),
                                                                __builtin_bit_cast(us2, b)));
}

// min of w[3 .. 2R] (the window middle shared by four window minima) in four independent
// chains: consecutive dependent packed 16-bit ops need a wait state between them on
// gfx950, interleaved chains do not (min is exact, so the order is free)
template <int R>
__device__ __forceinline__ uint32_t mid_min(const uint32_t* w) {
  static_assert(2 * R >= 6, "four chains");
  uint32_t m[4] = {w[3], w[4], w[5], w[6]};
#pragma unroll
  for (int t = 7; t <= 2 * R; ++t) m[(t - 3) & 3] = pkmin(m[(t - 3) & 3], w[t]);
  return pkmin(pkmin(m[0], m[1]), pkmin(m[2], m[3]));
}
__device__ __forceinline__ uint32_t pack(uint32_t v) { return v | ((65535u - v) << 16); }

// van Herk prefix (P) / suffix (in place over A) minima over blocks of w along one LDS
// line whose consecutive elements are `stride` words apart.
__device__ __forceinline__ void vh_block(uint32_t* A, uint32_t* P, int p0, int p1, int stride) {
  uint32_t m = A[p0 * stride];
  P[p0 * stride] = m;
#pragma unroll 4
  for (int p = p0 + 1; p < p1; ++p) {
    m = pkmin(m, A[p * stride]);
    P[p * stride] = m;
  }
  m = A[(p1 - 1) * stride];
#pragma unroll 4
  for (int p = p1 - 2; p >= p0; --p) {
    m = pkmin(m, A[p * stride]);
    A[p * stride] = m;
  }
}

// 1-D packed min/max along y (sa = W) or z (sa = W*H).  Work-group tile: XW consecutive
// x positions times C consecutive outputs along the axis, at one coordinate of the
// remaining axis (stride so).  LDS holds the clamped input span (C + 2r) x XW twice:
// A (input, then suffix minima in place) and P (prefix minima).
template <int XW, bool FROM_U16>
__global__ __launch_bounds__(NT) void k_minmax_line(const void* __restrict__ src,
                                                    uint32_t* __restrict__ dst, int W, int L,
                                                    i64 sa, i64 so, int r, int C, int nxt,
                                                    int nct) {
  extern __shared__ uint32_t smem[];
  const int span = C + 2 * r;
  uint32_t* A = smem;
  uint32_t* P = smem + span * XW;
  unsigned b = blockIdx.x;
  const int xt = b % nxt; b /= nxt;
  const int ct = b % nct; b /= nct;
  const i64 base = (i64)b * so;
  const int x0 = xt * XW, c0 = ct * C;
  stage_tile<8, NT, uint32_t>(
      span * XW,
      [&](int e) -> uint32_t {
        const int p = e / XW, x = x0 + e % XW;
        if (x >= W) return 0u;
        const i64 idx = base + (i64)clampi(c0 - r + p, 0, L - 1) * sa + x;
        return FROM_U16 ? pack(((const uint16_t*)src)[idx]) : ((const uint32_t*)src)[idx];
      },
      [&](int e, uint32_t v) { A[e] = v; });
  __syncthreads();
  const int w = 2 * r + 1;
  const int nb = (span + w - 1) / w;
  for (int t = threadIdx.x; t < nb * XW; t += NT) {
    const int blk = t / XW, xl = t % XW;
    const int p0 = blk * w;
    vh_block(A + xl, P + xl, p0, min(p0 + w, span), XW);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < C * XW; e += NT) {
    const int i = e / XW, xl = e % XW, c = c0 + i, x = x0 + xl;
    if (c < L && x < W)
      dst[base + (i64)c * sa + x] = pkmin(A[i * XW + xl], P[(i + 2 * r) * XW + xl]);
  }
}

// x pass of min/max (packed) fused with the x pass of the box filter.  One wave per row
// (4 rows per work-group), C = 64 * RUN outputs per row tile.  The min/max result is
// needed on [c0-r, c0+C+r) clamped to [0, W) because the box pass clamps to the edge of
// the *filtered* row.  Phase 1 stages the clamped packed input of the row in LDS; phase 2
// gives each lane 4 consecutive window minima (the window middle, shared by all four,
// plus short prefix / suffix runs: about (2r + 12) / 4 packed mins per output); phase 3
// gives each lane RUN consecutive box sums by sliding (integers: exact in any order).
// Output: float2 (E_x, D_x) = (sum(min) * k, sum(max) * k).  For r above kRunRadius.
template <int RUN>
__global__ __launch_bounds__(NT) void k_minmax_x_box(const uint32_t* __restrict__ src,
                                                     float2* __restrict__ dst, int W, i64 nrows,
                                                     int r, int nct, float k) {
  static_assert(RUN == 4, "four outputs per lane");
  constexpr int C = 64 * RUN;
  extern __shared__ __align__(16) uint32_t smem_x[];
  const int spanmax = C + 4 * r + 4;  // a multiple of 4: both rows stay 16-byte aligned
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint32_t* A = smem_x + wave * 2 * spanmax;  // clamped packed input of the row
  uint32_t* B = A + spanmax;                  // window minima
  const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
  const int ct = tile % nct;
  const i64 row = (i64)(tile / nct) * (NT / 64) + wave;
  const bool live = row < nrows;  // wave-uniform
  const int c0 = ct * C;
  const int qa = max(0, c0 - r), qb = min(W, c0 + C + r);
  const int nq = qb - qa, span = nq + 2 * r;
  const uint32_t* srow = src + (live ? row : 0) * W;
  if (live)
    for (int p = lane; p < span; p += 64) A[p] = srow[clampi(qa - r + p, 0, W - 1)];
  __syncthreads();
  // window minima B[j] = min(A[j .. j + 2r]), j in [0, nq), four per lane: the window
  // middle A[j0+3 .. j0+2r] is shared by all four, plus short prefix / suffix runs
  for (int j0 = lane * 4; live && j0 < nq; j0 += 256) {
    uint32_t o[4];
    uint32_t mid = A[j0 + 3];
    for (int t = 4; t <= 2 * r; ++t) mid = pkmin(mid, A[j0 + t]);
    const uint32_t l2 = A[j0 + 2], l1 = pkmin(A[j0 + 1], l2), l0 = pkmin(A[j0], l1);
    const uint32_t r1 = A[j0 + 2 * r + 1], r2 = pkmin(r1, A[j0 + 2 * r + 2]),
                   r3 = pkmin(r2, A[j0 + 2 * r + 3]);
    o[0] = pkmin(mid, l0);
    o[1] = pkmin(pkmin(mid, l1), r1);
    o[2] = pkmin(pkmin(mid, l2), r2);
    o[3] = pkmin(mid, r3);
    *reinterpret_cast<uint4*>(B + j0) = make_uint4(o[0], o[1], o[2], o[3]);
  }
  __syncthreads();
  const int xs = c0 + lane * RUN;
  if (!live || xs >= W) return;
  const uint32_t full = (uint32_t)(2 * r + 1) * 65535u;
  float2 out[RUN];
  const uint32_t* m = B - qa;  // m[x]: window minimum at x, x in [qa, qb)
  auto at = [&](int x) { return m[clampi(x, 0, W - 1)]; };
  uint32_t se = 0, sdn = 0;
  for (int j = -r; j <= r; ++j) {
    const uint32_t v = at(xs + j);
    se += v & 0xFFFFu;
    sdn += v >> 16;
  }
#pragma unroll
  for (int q = 0; q < RUN; ++q) {
    if (q > 0) {
      const int x = xs + q;
      const uint32_t vin = at(x + r), vout = at(x - r - 1);
      se += (vin & 0xFFFFu) - (vout & 0xFFFFu);
      sdn += (vin >> 16) - (vout >> 16);
    }
    out[q] = make_float2((float)se * k, (float)(full - sdn) * k);
  }
  float2* drow = dst + row * W;
  // 16-byte stores (a wave writes 1 KB in two instructions) where the row start allows
  if (xs + RUN <= W && ((row * W) & 1) == 0) {
#pragma unroll
    for (int q = 0; q < RUN; q += 2)
      *reinterpret_cast<float4*>(drow + xs + q) =
          make_float4(out[q].x, out[q].y, out[q + 1].x, out[q + 1].y);
  } else {
#pragma unroll
    for (int q = 0; q < RUN; ++q)
      if (xs + q < W) drow[xs + q] = out[q];
  }
}

// With NORM the z pass also normalizes against img.
template <int XW, bool NORM, typename TS>
__global__ __launch_bounds__(NT) void k_box_line(const float2* __restrict__ src,
                                                 float2* __restrict__ dst, TS* __restrict__ norm,
                                                 const uint16_t* __restrict__ img, float min_int,
                                                 int W, int L, i64 sa, i64 so, int r, int C,
                                                 int nxt, int nct, float k) {
  extern __shared__ float2 smem2[];
  const int span = C + 2 * r;
  unsigned b = blockIdx.x;
  const int xt = b % nxt; b /= nxt;
  const int ct = b % nct; b /= nct;
  const i64 base = (i64)b * so;
  const int x0 = xt * XW, c0 = ct * C;
  stage_tile<8, NT, float2>(
      span * XW,
      [&](int e) -> float2 {
        const int p = e / XW, x = x0 + e % XW;
        if (x >= W) return make_float2(0.0f, 0.0f);
        return src[base + (i64)clampi(c0 - r + p, 0, L - 1) * sa + x];
      },
      [&](int e, float2 v) { smem2[e] = v; });
  __syncthreads();
  for (int e = threadIdx.x; e < C * XW; e += NT) {
    const int i = e / XW, xl = e % XW, c = c0 + i, x = x0 + xl;
    if (c >= L || x >= W) continue;
    float ve = 0.0f, vd = 0.0f;
#pragma unroll 4
    for (int j = 0; j <= 2 * r; ++j) {
      const float2 t = smem2[(i + j) * XW + xl];
      ve += t.x;
      vd += t.y;
    }
    ve *= k;
    vd *= k;
    const i64 idx = base + (i64)c * sa + x;
    if (NORM) {
      const float I = (float)img[idx];
      norm[idx] = cvt<TS>((I >= min_int) ? (I - ve) / (vd - ve) : 0.0f);
    } else {
      dst[idx] = make_float2(ve, vd);
    }
  }
}

// ---- column walkers (compile-time radius) ------------------------------------------
// One thread owns one line along the axis (x-consecutive threads -> coalesced rows) and
// walks it front to back, so every input is read once and no LDS is needed.
//
// Min / max: van Herk blocks of w = 2R+1 over the clamp-extended line g[k] = f[c(k-R)].
// With S = suffix minima of the previous block and P = prefix minima of the current
// one, output c = (b-1)w + j is S[0] for j = 0 and min(S[j], P[j-1]) otherwise.
template <int R, bool FROM_U16>
__global__ __launch_bounds__(NT) void k_minmax_walk(const void* __restrict__ src,
                                                    uint32_t* __restrict__ dst, int W, int L,
                                                    i64 sa, i64 so, unsigned nxb, unsigned no,
                                                    int len) {
  constexpr int WB = 2 * R + 1;
  const LineAt la = line_at_block(nxb, no, len, L);
  const int x = la.x;
  if (x >= W) return;
  const i64 base = (i64)la.other * so + x;
  const int s0 = la.c0;
  const int n = la.c1 - s0;  // outputs of the segment; below, positions count from s0
  auto load = [&](int k) -> uint32_t {
    const i64 idx = base + (i64)clampi(s0 + k - R, 0, L - 1) * sa;
    return FROM_U16 ? pack(((const uint16_t*)src)[idx]) : ((const uint32_t*)src)[idx];
  };
  uint32_t S[WB], cur[WB];
#pragma unroll
  for (int j = 0; j < WB; ++j) cur[j] = load(j);
  S[WB - 1] = cur[WB - 1];
#pragma unroll
  for (int j = WB - 2; j >= 0; --j) S[j] = pkmin(cur[j], S[j + 1]);
  const int nb = (n + WB - 1) / WB;
  for (int b = 1; b <= nb; ++b) {
#pragma unroll
    for (int j = 0; j < WB; ++j) cur[j] = load(b * WB + j);
    const int c0 = (b - 1) * WB;
    uint32_t p = cur[0];
#pragma unroll
    for (int j = 0; j < WB; ++j) {
      if (j > 0) {
        if (c0 + j < n) st_nt(dst + base + (i64)(s0 + c0 + j) * sa, pkmin(S[j], p));
        p = pkmin(p, cur[j]);
      } else if (c0 < n) {
        st_nt(dst + base + (i64)(s0 + c0) * sa, S[0]);
      }
    }
    S[WB - 1] = cur[WB - 1];
#pragma unroll
    for (int j = WB - 2; j >= 0; --j) S[j] = pkmin(cur[j], S[j + 1]);
  }
}

// Min / max along y and z in one pass: a work-group of 16 waves owns a 64-column x 32-row
// tile of every plane and walks z.  Per slice:
//   1. the packed rows y0-RY .. y0+31+RY of the slice (clamped to the plane; raw u16
//      loaded PF slices ahead) enter an LDS buffer (two buffers, alternating: the next
//      slice is stored while this one is read, one barrier per slice);
//   2. each thread (lane = column, wave = row pair) forms the y window minima of its two
//      rows from the 2RY+2 values of its column: a shared window middle plus one end value
//      each;
//   3. these enter the thread's z walk: van Herk blocks of WB = 2RZ+1 slices over the
//      clamp-extended line g[k] = slice(clamp(k - RZ)), held in place in a register array:
//      slot j holds the suffix minimum S[j] of the previous block until slice j of the
//      current block takes it, and a running prefix minimum P covers the current block,
//      so output c = min(S[j+1], P) leaves when g[c + 2RZ] arrives; at a block's end its
//      suffix minima replace it in place and give the output c = k - 2RZ as S[0].
// Min is exact, so y then z equals the z then y of the unfused passes bit for bit.  The
// z-min/maxed volume between them (8 B/voxel of traffic) is never stored.  Slices beyond the
// volume are not walked: 32 x 2160 x 2560 took 401 us with its 20 copies of the first and last
// slice, 301 without (96 slices: 858, 754).
template <int RZ, int RY, int PF>
__global__ __launch_bounds__(1024) void k_minmax_zy_walk(const uint16_t* __restrict__ img,
                                                        uint32_t* __restrict__ dst, int W, int H,
                                                        int D, unsigned nyt, unsigned nxt,
                                                        int zlen) {
  constexpr int TY = 32, KR = 2, NWV = TY / KR;  // rows per tile, rows per thread, waves
  constexpr int SR = TY + 2 * RY;                 // staged rows per slice
  constexpr int NLD = (SR + NWV - 1) / NWV;       // row loads per lane and slice
  constexpr int SRP = NLD * NWV;  // rows of an LDS buffer: every wave loads and stores NLD
                                  // rows (rows past SR repeat a clamped row, unused)
  constexpr int WB = 2 * RZ + 1;
  constexpr int NW = 2 * RY + KR;                 // window values per thread
  static_assert(WB % PF == 0, "queue slots must be static in the unrolled block");
  static_assert(RY >= 2, "shared window middle");
  __shared__ uint32_t S[2][SRP * 64];
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int yt = (int)(t % nyt), xt = (int)(t / nyt % nxt);
  // outputs z0 .. z1-1 of one of the segments of the volume; below, k and c count from z0
  const int z0 = (int)(t / nyt / nxt) * zlen, z1 = min(D, z0 + zlen);
  const int lane = (int)(threadIdx.x & 63);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // wave-uniform
  const int x = xt * 64 + lane, y0 = yt * TY;
  const int xc = min(x, W - 1);
  const size_t WH = (size_t)W * (size_t)H;
  // staged row wv + NWV j of every slice: its offset in the slice (rows clamped); no
  // load or LDS store is under a condition
  uint32_t off[NLD];
#pragma unroll
  for (int j = 0; j < NLD; ++j)
    off[j] = (uint32_t)clampi(y0 - RY + wv + NWV * j, 0, H - 1) * (uint32_t)W + (uint32_t)xc;
  // loads and stores go through a buffer descriptor of the slice (scalar) with 32-bit
  // lane offsets: with 64-bit lane addresses the compiler kept one per unrolled step
  uint32_t q[PF][NLD];  // raw values of slice k wait in slot k % PF
  auto fetch = [&](int k, int slot) {
    const __amdgpu_buffer_rsrc_t r =
        buf_rsrc(img + (size_t)clampi(z0 + k - RZ, 0, D - 1) * WH, (uint32_t)(WH * 2));
#pragma unroll
    for (int j = 0; j < NLD; ++j)
      q[slot][j] = __builtin_amdgcn_raw_buffer_load_b16(r, (int)(off[j] * 2u), 0, 0);
  };
  // slice k's packed rows into buffer k & 1, the loads of slice k + PF into the freed slot.
  // Step k stores slice k + 1 and reads slice k's rows, then one barrier: every wave's
  // stores of slice k + 1 are then done before step k + 1 reads them, and its reads of
  // slice k before step k + 1 stores slice k + 2 over them (one wait per slice, not two).
  auto stage = [&](int k, int slot) {
    uint32_t* Sb = S[k & 1];
#pragma unroll
    for (int j = 0; j < NLD; ++j)
      Sb[(wv + NWV * j) * 64 + lane] = pack(q[slot][j]);
    fetch(k + PF, slot);
  };
  const int ty = KR * wv;  // first output row of this thread in the tile
  // y window minima of rows ty, ty + 1: staged rows ty .. ty + 2RY + 1 of column lane
  auto ymin = [&](const uint32_t* Sb, uint32_t o[KR]) {
    uint32_t w[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) w[i] = Sb[(ty + i) * 64 + lane];
    // middle w[1 .. 2RY], shared by both windows, in four interleaved chains
    uint32_t m[4] = {w[1], w[2], w[3], w[4]};
#pragma unroll
    for (int i = 5; i <= 2 * RY; ++i) m[(i - 1) & 3] = pkmin(m[(i - 1) & 3], w[i]);
    const uint32_t mid = pkmin(pkmin(m[0], m[1]), pkmin(m[2], m[3]));
    o[0] = pkmin(mid, w[0]);
    o[1] = pkmin(mid, w[2 * RY + 1]);
  };
  // byte offsets of the thread's outputs in a slice; outside the plane past the slice
  // descriptor's record count, so those stores are dropped
  uint32_t ro[KR];
#pragma unroll
  for (int i = 0; i < KR; ++i)
    ro[i] = x < W && y0 + ty + i < H ? ((uint32_t)(y0 + ty + i) * (uint32_t)W + (uint32_t)x) * 4u
                                     : 0xFFFFFFF0u;
  auto put = [&](int c, const uint32_t v[KR]) {
    const __amdgpu_buffer_rsrc_t r = buf_rsrc(dst + (size_t)(z0 + c) * WH, (uint32_t)(WH * 4));
#pragma unroll
    for (int i = 0; i < KR; ++i)  // streaming (nontemporal) stores
      __builtin_amdgcn_raw_buffer_store_b32(v[i], r, (int)ro[i], 0, kCachePolicyNT);
  };
  uint32_t zs[KR][WB], P[KR];
  auto suffix = [&]() {
#pragma unroll
    for (int i = 0; i < KR; ++i)
#pragma unroll
      for (int j = WB - 2; j >= 0; --j) zs[i][j] = pkmin(zs[i][j], zs[i][j + 1]);
  };
  // block 0 (slices k = 0 .. WB-1) only fills the slots; its suffix minimum S[0] is
  // output 0.  Slices before the volume repeat slice 0, which the window holds anyway:
  // they take the minimum's identity and are not walked.
  auto fill = [&](auto first) {
    constexpr int F = decltype(first)::value;
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int i = 0; i < KR; ++i) zs[i][j] = 0xFFFFFFFFu;
#pragma unroll
    for (int k = F; k < F + PF; ++k) fetch(k, k % PF);
    stage(F, F % PF);
    __syncthreads();
#pragma unroll
    for (int j = F; j < WB; ++j) {
      stage(j + 1, (j + 1) % PF);
      uint32_t v[KR];
      ymin(S[j & 1], v);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < KR; ++i) zs[i][j] = v[i];
    }
  };
  if (z0 == 0)
    fill(std::integral_constant<int, RZ>());
  else
    fill(std::integral_constant<int, 0>());
  suffix();
  {
    uint32_t v[KR];
#pragma unroll
    for (int i = 0; i < KR; ++i) v[i] = zs[i][0];
    put(0, v);
  }
  // output c leaves when slice k = c + 2RZ has arrived; the last is z1 - 1.  Slices past the
  // volume repeat the last one: as before it, they are not walked.  The walk's end leaves
  // the loop (uniform over the work-group: every wave has the same k).
  const int kend = z1 - z0 + 2 * RZ, kreal = D - z0 + RZ;
  const int klim = kreal >= WB ? min(kend, kreal) : kend;
  auto walk = [&] {
    for (int k0 = WB;; k0 += WB) {
#pragma unroll
      for (int j = 0; j < WB; ++j) {
        const int k = k0 + j;
        if (k >= klim) return;
        stage(k + 1, (j + 1) % PF);  // (k0 + j) % PF == j % PF
        uint32_t v[KR], o[KR];
        ymin(S[k & 1], v);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < KR; ++i) {
          P[i] = j == 0 ? v[i] : pkmin(P[i], v[i]);
          if (j < WB - 1) o[i] = pkmin(zs[i][j + 1], P[i]);
          zs[i][j] = v[i];
        }
        if (j < WB - 1) {
          put(k - 2 * RZ, o);
        } else {
          suffix();
#pragma unroll
          for (int i = 0; i < KR; ++i) o[i] = zs[i][0];
          put(k - 2 * RZ, o);
        }
      }
    }
  };
  walk();
  // the outputs whose windows end past the volume (RZ at most): the block's other slots take
  // the identity, as does the prefix of a block that holds no slice
  int k = klim;
  const int jt = k % WB;
#pragma unroll
  for (int i = 0; i < KR; ++i) P[i] = jt == 0 ? 0xFFFFFFFFu : P[i];
#pragma unroll
  for (int j = 0; j < WB - 1; ++j)
    if (j >= jt) {  // uniform
      uint32_t o[KR];
#pragma unroll
      for (int i = 0; i < KR; ++i) {
        o[i] = pkmin(zs[i][j + 1], P[i]);
        zs[i][j] = 0xFFFFFFFFu;
      }
      if (k < kend) put(k - 2 * RZ, o);
      ++k;
    }
#pragma unroll
  for (int i = 0; i < KR; ++i) zs[i][WB - 1] = 0xFFFFFFFFu;
  suffix();
#pragma unroll
  for (int j = 0; j < RZ; ++j) {
    uint32_t o[KR];
#pragma unroll
    for (int i = 0; i < KR; ++i) o[i] = zs[i][j];
    if (k < kend) put(k - 2 * RZ, o);
    ++k;
  }
}

// Box mean: a register ring of the last 2R+1 inputs (clamp), unrolled by the ring period
// so every index is static; each output sums its window in the reference order.  Ring
// refills are loaded PF steps before they enter the ring (PF divides the ring period, so
// every queue slot is static too), and the walk leaves the kernel at the line's end
// instead of skipping the remaining unrolled steps, so no merged control path makes the
// compiler wait for the whole queue.
template <int R, bool NORM, typename TS>
__global__ __launch_bounds__(NT) void k_box_walk(const float2* __restrict__ src,
                                                 float2* __restrict__ dst, TS* __restrict__ norm,
                                                 const uint16_t* __restrict__ img, float min_int,
                                                 int W, int L, i64 sa, i64 so, unsigned nxb,
                                                 unsigned no, int len, float k) {
  constexpr int WB = 2 * R + 1;
  constexpr int PF = WB % 3 == 0 ? 3 : WB % 5 == 0 ? 5 : WB % 7 == 0 ? 7 : 1;
  const LineAt la = line_at_block(nxb, no, len, L);
  const int x = la.x, s0 = la.c0, s1 = la.c1;
  if (x >= W) return;
  const i64 base = (i64)la.other * so + x;
  auto at = [&](int p) { return src[base + (i64)clampi(p, 0, L - 1) * sa]; };
  float2 ring[WB];  // position p lives in ring[(p - s0 + R) % WB]
#pragma unroll
  for (int q = 0; q < WB; ++q) ring[q] = at(s0 + q - R);
  float2 pf[PF];  // the refill of step c (position c + R + 1) waits in slot (c - s0) % PF
#pragma unroll
  for (int j = 0; j < PF; ++j) pf[j] = at(s0 + R + 1 + j);
  for (int c0 = s0;; c0 += WB) {
    // with the normalization fused, the raw intensities of this block's WB outputs are
    // loaded up front: loading each one at its output made every output wait for all
    // outstanding loads, the ring refills included
    float iv[WB];
    if (NORM) {
#pragma unroll
      for (int q = 0; q < WB; ++q)
        iv[q] = (float)img[base + (i64)min(c0 + q, L - 1) * sa];
    }
#pragma unroll
    for (int q = 0; q < WB; ++q) {
      const int c = c0 + q;
      if (c >= s1) return;
      float ve = 0.0f, vd = 0.0f;
#pragma unroll
      for (int j = 0; j <= 2 * R; ++j) {  // position c - R + j -> ring[(q + j) % WB]
        ve += ring[(q + j) % WB].x;
        vd += ring[(q + j) % WB].y;
      }
      ve *= k;
      vd *= k;
      const i64 idx = base + (i64)c * sa;
      if (NORM) {
        const float I = iv[q];
        st_nt(norm + idx, (I >= min_int) ? (I - ve) / (vd - ve) : 0.0f);
      } else {
        st_nt(dst + idx, make_float2(ve, vd));
      }
      // slot of position c - R is reused for position c + R + 1
      ring[q] = pf[q % PF];
      pf[q % PF] = at(c + R + 1 + PF);
    }
  }
}

// min/max along x, box along x and box along y fused.  A one-wave work-group walks the
// rows of one plane of the y-min/maxed (packed) volume for a strip of CW = 128 columns,
// two per lane.  Per row:
//   1. the clamped packed row segment x0-2R .. x0+CW-1+2R enters an LDS line A;
//   2. window minima B[b] = min(A[b .. b+2R]) (the min/max at x = x0-R+b) are formed four
//      per task (a shared window middle plus short prefix / suffix runs); on a strip at
//      the plane's edge, positions outside [0, W) then take the value at the edge, since
//      the box pass clamps to the edge of the filtered row;
//   3. each lane sums B over its two windows (integers, exact in any order) -> (E_x, D_x)
//      of its columns; B keeps the min channel and the 65535 - max channel in two 16-bit
//      arrays, so one v_dot2 with (1, 1) adds two window positions;
//   4. these enter a register ring of the last 2R+1 rows (rows clamped), and each output
//      row sums its window in the reference order, as the y pass walker does.
// The (E_x, D_x) volume of the unfused passes is never stored.  Rows are fetched PF rows
// ahead of their use; the plane's end leaves the kernel (see the DoG row walker).
template <int R>
__global__ __launch_bounds__(64) void k_norm_xy_walk(const uint32_t* __restrict__ src,
                                                     float4* __restrict__ dst, int W, int H,
                                                     int nxs, int nys, int rows, float k) {
  constexpr int WB = 2 * R + 1;
  constexpr int CW = 128;                    // output columns per wave
  constexpr int HX = (2 * R + 3) / 4 * 4;    // line halo: 16-byte aligned task reads
  constexpr int NB = CW + 2 * R;             // window minima per row
  constexpr int NTASK = (NB + 3) / 4;        // four minima per task
  constexpr int LW = 64 * ((4 * NTASK + 2 * R + 4 + 63) / 64);  // line, whole lane loads
  constexpr int NLD = LW / 64;               // loads per lane per row
  constexpr int PF = WB % 3 == 0 ? 3 : WB % 5 == 0 ? 5 : WB % 7 == 0 ? 7 : 1;
  static_assert(HX == 2 * R, "task windows assume a halo of exactly 2R");
  static_assert(4 * NTASK + 2 * R + 4 <= LW, "task reads stay inside the line");
  __shared__ __align__(16) uint32_t A[LW];
  // B[b] = window minimum b: its min channel in Bm, its 65535 - max channel in Bx, as
  // 16-bit entries, positions 2i and 2i + 1 in word i
  __shared__ __align__(16) uint32_t Bm[2 * NTASK];
  __shared__ __align__(16) uint32_t Bx[2 * NTASK];
  // work-group = one strip of one plane over the rows [y0, y1) of one of the nys segments
  // of the plane (rows: a multiple of WB)
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int y0 = (int)(t % nys) * rows, y1 = min(H, y0 + rows);
  const unsigned tile = t / nys;
  const int l = threadIdx.x;
  const int x0 = (int)(tile % nxs) * CW;
  const uint32_t* plane = src + (i64)(tile / nxs) * H * W;
  int xl[NLD];  // clamped column of each line position this lane loads
#pragma unroll
  for (int j = 0; j < NLD; ++j) xl[j] = clampi(x0 - HX + 64 * j + l, 0, W - 1);
  uint32_t qv[PF][NLD];  // row y is held in slot y % PF
  auto fetch = [&](int y, int s) {
    const uint32_t* row = plane + (i64)min(y, H - 1) * W;
#pragma unroll
    for (int j = 0; j < NLD; ++j) qv[s][j] = row[xl[j]];
  };
  // row y waits in queue slot y % PF (y0 is a multiple of WB, so of PF)
  if (y0 == 0) {
#pragma unroll
    for (int s = 0; s < PF; ++s) fetch(s, s);
  } else {
#pragma unroll
    for (int s = 0; s < PF; ++s) fetch(y0 - R + s, ((s - R) % PF + PF) % PF);
  }
  const bool edge = x0 - R < 0 || x0 + CW + R > W;  // wave-uniform
  const int blo = R - x0, bhi = W - 1 - x0 + R;     // B index of x = 0 and x = W - 1
  const uint32_t full = (uint32_t)WB * 65535u;
  const us2 lo1 = {1, 0}, hi1 = {0, 1}, one = {1, 1};
  // (E_x, D_x) of the lane's two columns for row y (slot s); fetches row y + PF into s
  auto xrow = [&](int y, int s) -> float4 {
#pragma unroll
    for (int j = 0; j < NLD; ++j) A[64 * j + l] = qv[s][j];
    fetch(y + PF, s);
    wave_lds_sync();
    if (l < NTASK) {
      constexpr int NV = (2 * R + 4) / 4;
      uint32_t w[4 * NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const uint4 q = *reinterpret_cast<const uint4*>(A + 4 * l + 4 * v);
        w[4 * v] = q.x; w[4 * v + 1] = q.y; w[4 * v + 2] = q.z; w[4 * v + 3] = q.w;
      }
      const uint32_t mid = mid_min<R>(w);
      const uint32_t l2 = w[2], l1 = pkmin(w[1], l2), l0 = pkmin(w[0], l1);
      const uint32_t r1 = w[2 * R + 1], r2 = pkmin(r1, w[2 * R + 2]), r3 = pkmin(r2, w[2 * R + 3]);
      const uint32_t b0 = pkmin(mid, l0), b1 = pkmin(pkmin(mid, l1), r1),
                     b2 = pkmin(pkmin(mid, l2), r2), b3 = pkmin(mid, r3);
      // v_perm_b32: perm(b1, b0, 0x05040100) = lo16(b0) | lo16(b1) << 16,
      //             perm(b1, b0, 0x07060302) = hi16(b0) | hi16(b1) << 16
      *reinterpret_cast<uint2*>(Bm + 2 * l) =
          make_uint2(__builtin_amdgcn_perm(b1, b0, 0x05040100u),
                     __builtin_amdgcn_perm(b3, b2, 0x05040100u));
      *reinterpret_cast<uint2*>(Bx + 2 * l) =
          make_uint2(__builtin_amdgcn_perm(b1, b0, 0x07060302u),
                     __builtin_amdgcn_perm(b3, b2, 0x07060302u));
    }
    wave_lds_sync();
    if (edge) {  // positions outside the plane take the edge value
      constexpr int NF = (4 * NTASK + 63) / 64;
      uint16_t* bm = reinterpret_cast<uint16_t*>(Bm);
      uint16_t* bx = reinterpret_cast<uint16_t*>(Bx);
      uint16_t fm[NF], fx[NF];
#pragma unroll
      for (int j = 0; j < NF; ++j) {
        const int b = 64 * j + l;
        const int c = clampi(b, blo, bhi);
        fm[j] = b < 4 * NTASK ? bm[c] : (uint16_t)0;
        fx[j] = b < 4 * NTASK ? bx[c] : (uint16_t)0;
      }
      wave_lds_sync();
#pragma unroll
      for (int j = 0; j < NF; ++j)
        if (64 * j + l < 4 * NTASK) {
          bm[64 * j + l] = fm[j];
          bx[64 * j + l] = fx[j];
        }
      wave_lds_sync();
    }
    // column x0 + 2l sums positions 2l .. 2l + 2R: words l .. l + R - 1 and the low half
    // of word l + R; column x0 + 2l + 1 sums 2l + 1 .. 2l + 2R + 1: the high half of word
    // l and words l + 1 .. l + R
    uint32_t m[R + 1], x[R + 1];
#pragma unroll
    for (int t = 0; t <= R; ++t) {
      m[t] = Bm[l + t];
      x[t] = Bx[l + t];
    }
    uint32_t sm = 0, sx = 0;
#pragma unroll
    for (int t = 1; t < R; ++t) {
      sm = __builtin_amdgcn_udot2(__builtin_bit_cast(us2, m[t]), one, sm, false);
      sx = __builtin_amdgcn_udot2(__builtin_bit_cast(us2, x[t]), one, sx, false);
    }
    const us2 m0 = __builtin_bit_cast(us2, m[0]), mr = __builtin_bit_cast(us2, m[R]);
    const us2 x0w = __builtin_bit_cast(us2, x[0]), xr = __builtin_bit_cast(us2, x[R]);
    const uint32_t se = __builtin_amdgcn_udot2(m0, one, __builtin_amdgcn_udot2(mr, lo1, sm, false), false);
    const uint32_t se1 = __builtin_amdgcn_udot2(m0, hi1, __builtin_amdgcn_udot2(mr, one, sm, false), false);
    const uint32_t sdn = __builtin_amdgcn_udot2(x0w, one, __builtin_amdgcn_udot2(xr, lo1, sx, false), false);
    const uint32_t sdn1 = __builtin_amdgcn_udot2(x0w, hi1, __builtin_amdgcn_udot2(xr, one, sx, false), false);
    float4 o = make_float4((float)se * k, (float)(full - sdn) * k, (float)se1 * k,
                           (float)(full - sdn1) * k);
    // pin the row's outputs here (see the DoG row walker)
    asm volatile("" : "+v"(o.x), "+v"(o.y), "+v"(o.z), "+v"(o.w));
    return o;
  };
  const int xc = x0 + 2 * l;
  const bool st2 = xc + 1 < W && (W & 1) == 0, st1 = xc < W;
  float4* dq = dst + ((tile / nxs) * (i64)H * W + xc) / 2;  // valid when st2
  float2* dp = reinterpret_cast<float2*>(dst) + (tile / nxs) * (i64)H * W + xc;
  float4 ring[WB];  // row p lives in ring[(p + R) % WB]; rows clamp to [0, H)
  if (y0 == 0) {
    ring[R] = xrow(0, 0);
#pragma unroll
    for (int q = 0; q < R; ++q) ring[q] = ring[R];
#pragma unroll
    for (int q = R + 1; q < WB; ++q) ring[q] = xrow(min(q - R, H - 1), (q - R) % PF);
  } else {  // a later segment starts from the R rows above it
#pragma unroll
    for (int q = 0; q < WB; ++q) ring[q] = xrow(y0 - R + q, ((q - R) % PF + PF) % PF);
  }
  for (int c0 = y0;; c0 += WB) {
#pragma unroll
    for (int q = 0; q < WB; ++q) {
      const int c = c0 + q;
      if (c >= y1) return;
      float e0 = 0.0f, d0 = 0.0f, e1 = 0.0f, d1 = 0.0f;
#pragma unroll
      for (int j = 0; j <= 2 * R; ++j) {  // row c - R + j -> ring[(q + j) % WB]
        const float4 t = ring[(q + j) % WB];
        e0 += t.x;
        d0 += t.y;
        e1 += t.z;
        d1 += t.w;
      }
      const float4 o = make_float4(e0 * k, d0 * k, e1 * k, d1 * k);
      if (st2) {
        st_nt(dq + (i64)c * W / 2, o);
      } else if (st1) {
        dp[(i64)c * W] = make_float2(o.x, o.y);
        if (xc + 1 < W) dp[(i64)c * W + 1] = make_float2(o.z, o.w);
      }
      ring[q] = xrow(min(c + R + 1, H - 1), (q + R + 1) % PF);  // replaces row c - R
    }
  }
}

// ---- radii without a kernel of their own, up to kRunRadius ---------------------------
// The same passes with the radius at run time, eight outputs at a time (run8.hpp).

// out[o] = packed minimum of inputs o .. o + 2r
template <int R, typename F>
__device__ __forceinline__ void min8(F&& next, int r, uint32_t (&out)[OK]) {
  if constexpr (R > 0) {
    uint32_t v[2 * R + OK];
#pragma unroll
    for (int i = 0; i < 2 * R + OK; ++i) v[i] = next();
#pragma unroll
    for (int o = 0; o < OK; ++o) {
      out[o] = v[o];
#pragma unroll
      for (int i = 1; i <= 2 * R; ++i) out[o] = pkmin(out[o], v[o + i]);
    }
  } else {
    uint32_t h[OK - 1], m[4], t;
#pragma unroll
    for (int i = 0; i < OK - 1; ++i) h[i] = next();
    m[0] = next();  // input 7; inputs 7 .. 2r are in every window (2r - 6 of them, odd)
#pragma unroll
    for (int q = 1; q < 4; ++q) m[q] = m[0];
    int i = OK;
#pragma unroll 1
    for (; i + 3 <= 2 * r; i += 4)
#pragma unroll
      for (int q = 0; q < 4; ++q) m[q] = pkmin(m[q], next());  // four chains (see mid_min)
    for (; i <= 2 * r; ++i) m[1] = pkmin(m[1], next());
    const uint32_t mid = pkmin(pkmin(m[0], m[1]), pkmin(m[2], m[3]));
    uint32_t e[OK - 1];
#pragma unroll
    for (int q = 0; q < OK - 1; ++q) e[q] = next();
    t = mid;
    out[OK - 1] = mid;
#pragma unroll
    for (int o = OK - 2; o >= 0; --o) out[o] = t = pkmin(t, h[o]);  // inputs o .. 2r
    t = e[0];
#pragma unroll
    for (int o = 1; o < OK; ++o) {
      if (o > 1) t = pkmin(t, e[o - 1]);
      out[o] = pkmin(out[o], t);
    }
  }
}

// integer sums over inputs o .. o + 2r of the two 16-bit channels
template <int R, typename F>
__device__ __forceinline__ void sum8_u16(F&& next, int r, uint32_t (&lo)[OK], uint32_t (&hi)[OK]) {
  const us2 l1 = {1, 0}, h1 = {0, 1};
  auto add = [&](uint32_t v, uint32_t& a, uint32_t& b) {
    a = __builtin_amdgcn_udot2(__builtin_bit_cast(us2, v), l1, a, false);
    b = __builtin_amdgcn_udot2(__builtin_bit_cast(us2, v), h1, b, false);
  };
  uint32_t a = 0u, b = 0u;
  if constexpr (R > 0) {
    uint32_t v[2 * R + OK];
#pragma unroll
    for (int i = 0; i < 2 * R + OK; ++i) v[i] = next();
#pragma unroll
    for (int i = 0; i <= 2 * R; ++i) add(v[i], a, b);
    lo[0] = a;
    hi[0] = b;
#pragma unroll
    for (int o = 1; o < OK; ++o) {
      lo[o] = lo[o - 1] + (v[2 * R + o] & 0xFFFFu) - (v[o - 1] & 0xFFFFu);
      hi[o] = hi[o - 1] + (v[2 * R + o] >> 16) - (v[o - 1] >> 16);
    }
  } else {
    uint32_t h[OK - 1], e[OK - 1];
#pragma unroll
    for (int i = 0; i < OK - 1; ++i) h[i] = next();
    int i = OK - 1;
#pragma unroll 1
    for (; i <= 2 * r; i += 2) {  // 2r - 6 of them, even
      const uint32_t v0 = next(), v1 = next();
      add(v0, a, b);
      add(v1, a, b);
    }
#pragma unroll
    for (int q = 0; q < OK - 1; ++q) e[q] = next();
#pragma unroll
    for (int q = 0; q < OK - 1; ++q) add(h[q], a, b);
    lo[0] = a;
    hi[0] = b;
#pragma unroll
    for (int o = 1; o < OK; ++o) {
      lo[o] = lo[o - 1] + (e[o - 1] & 0xFFFFu) - (h[o - 1] & 0xFFFFu);
      hi[o] = hi[o - 1] + (e[o - 1] >> 16) - (h[o - 1] >> 16);
    }
  }
}

// Packed min / max along y or z: a work-group walks a segment of 64 lines through an LDS plane
// of the last 2r + 32 positions (clamped to the line).  Bound by its 6 (from raw) or 8 bytes
// per voxel: 130 and 180 us for 70 x 1080 x 1280 at radii 4 and 8 (4.5 and 4.3 TB/s); van Herk
// blocks on LDS tiles of 64 outputs and their halo, a serial chain each, took 533 and 209.
template <int R, bool FROM_U16>
__global__ __launch_bounds__(256) void k_minmax_run(const void* __restrict__ src,
                                                    uint32_t* __restrict__ dst, int W, int L,
                                                    i64 sa, i64 so, int r, unsigned nxb,
                                                    unsigned no, int len) {
  extern __shared__ uint32_t sm_mm[];
  constexpr int STEP = 4 * OK;
  const int hist = 2 * r;
  const RunAt a = run_at(L, so, nxb, no, len);
  const int xc = min(a.x0 + a.l, W - 1);
  uint32_t q[OK];
  auto fetch = [&](int p) {
#pragma unroll
    for (int k = 0; k < OK; ++k) {
      const i64 at = a.base + (i64)clampi(p + k, 0, L - 1) * sa + xc;
      q[k] = FROM_U16 ? (uint32_t)((const uint16_t*)src)[at] : ((const uint32_t*)src)[at];
    }
  };
  auto put = [&](int row) {
#pragma unroll
    for (int k = 0; k < OK; ++k) sm_mm[(row + k) * 64 + a.l] = FROM_U16 ? pack(q[k]) : q[k];
  };
  for (int g = a.wave; OK * g < hist; g += 4) {  // (the last may reach into the step's rows)
    fetch(a.s0 - r + OK * g);
    put(OK * g);
  }
  if (a.s0 + OK * a.wave < a.s1) fetch(a.s0 + r + OK * a.wave);
  __syncthreads();
  for (int c0 = a.s0; c0 < a.s1; c0 += STEP) {
    const int c = c0 + OK * a.wave;
    if (c < a.s1) put(hist + OK * a.wave);
    if (c + STEP < a.s1) fetch(c + STEP + r);
    __syncthreads();
    if (c < a.s1) {
      const uint32_t* p = sm_mm + OK * a.wave * 64 + a.l;
      uint32_t o[OK];
      min8<R>([&] { const uint32_t v = *p; p += 64; return v; }, r, o);
      if (a.x0 + a.l < W) {
#pragma unroll
        for (int k = 0; k < OK; ++k)
          if (c + k < a.s1) st_nt(dst + a.base + (i64)(c + k) * sa + a.x0 + a.l, o[k]);
      }
    }
    if (c0 + STEP >= a.s1) break;  // uniform
    __syncthreads();
    shift_rows<256, STEP, 64>(sm_mm, hist);
    __syncthreads();
  }
}

// The same for lines of at most kShallow positions.
template <bool FROM_U16>
__global__ __launch_bounds__(NT) void k_minmax_shallow(const void* __restrict__ src,
                                                       uint32_t* __restrict__ dst, int W, int L,
                                                       i64 sa, i64 so, int r, unsigned nxb,
                                                       unsigned no) {
  const LineAt la = line_at_block(nxb, no, L, L);
  if (la.x >= W) return;
  const i64 base = (i64)la.other * so + la.x;
  uint32_t v[kShallow];
#pragma unroll
  for (int i = 0; i < kShallow; ++i)
    if (i < L)  // uniform, as all that follow
      v[i] = FROM_U16 ? pack(((const uint16_t*)src)[base + i * sa]) : ((const uint32_t*)src)[base + i * sa];
#pragma unroll
  for (int c = 0; c < kShallow; ++c) {
    if (c >= L) break;
    uint32_t m = v[c];
#pragma unroll
    for (int i = 0; i < kShallow; ++i)
      if (i != c && i < L && i - c <= r && c - i <= r) m = pkmin(m, v[i]);
    st_nt(dst + base + c * sa, m);
  }
}

// out[o] = packed minimum of v[o] .. v[o + 2 R], in registers
template <int R, int N>
__device__ __forceinline__ void min8_regs(const uint32_t (&v)[N], uint32_t (&out)[OK]) {
  static_assert(2 * R >= OK && 2 * R + OK <= N, "inputs that all eight share");
  uint32_t m[4] = {v[OK - 1], v[OK - 1], v[OK - 1], v[OK - 1]};
#pragma unroll
  for (int i = OK; i <= 2 * R; ++i) m[i & 3] = pkmin(m[i & 3], v[i]);
  uint32_t t = pkmin(pkmin(m[0], m[1]), pkmin(m[2], m[3]));
  out[OK - 1] = t;
#pragma unroll
  for (int o = OK - 2; o >= 0; --o) out[o] = t = pkmin(t, v[o]);
  t = v[2 * R + 1];
#pragma unroll
  for (int o = 1; o < OK; ++o) {
    if (o > 1) t = pkmin(t, v[2 * R + o]);
    out[o] = pkmin(out[o], t);
  }
}

// Packed min / max along y and z in one pass (k_minmax_zy_walk for other radii, at least 4): a
// work-group of eight waves walks z for a tile of 64 columns x 8 rows, eight slices per step.
//   1. wave w holds the 8 + 2 ry rows of slice w, loaded a step ahead (clamped; a lane a
//      column), and forms the eight y windows in registers, whose number NQ fits four radii,
//      told apart by a uniform switch; they enter an LDS block of the last 2 rz + 8 slices;
//   2. wave w forms the eight z windows of row w.
// The halo rows come from L2 (three rows read per row written at ry = 8).  70 x 1080 x 1280 at
// radii 8 / 4: 171 us, in two passes 137 + 181.
constexpr int kZyRadiusZ = 12;  // 64 KB of LDS
// Above, a wave holds too many rows in flight (70 x 1080 x 1280, in two passes in brackets:
// 171 us (318) at 8 / 4, 198 (317) at 4 / 12, 287 (327) at 16 / 12, 348 (317) at 20 / 4).
constexpr int kZyRadiusY = 16;
template <int NQ>
__global__ __launch_bounds__(512) void k_minmax_zy_run(const uint16_t* __restrict__ img,
                                                       uint32_t* __restrict__ dst, int W, int H,
                                                       int D, int ry, int rz, unsigned nyt,
                                                       unsigned nxt, int len) {
  extern __shared__ uint32_t sm_zy[];
  constexpr int TY = OK, PL = TY * 64, RM = (NQ - OK) / 2;  // the largest radius
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int y0 = (int)(t % nyt) * TY, x0 = (int)(t / nyt % nxt) * 64;
  const int s0 = (int)(t / nyt / nxt) * len, s1 = min(D, s0 + len);
  const int l = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int xc = min(x0 + l, W - 1), hist = 2 * rz;
  uint32_t q[NQ];
  auto fetch = [&](int s) {
    const uint16_t* slice = img + (i64)clampi(s, 0, D - 1) * H * W;
#pragma unroll
    for (int i = 0; i < NQ; ++i) q[i] = slice[(i64)clampi(y0 - ry + i, 0, H - 1) * W + xc];
  };
  auto ymin = [&](int plane, int ahead, bool more) {
    uint32_t v[NQ], o[OK];
#pragma unroll
    for (int i = 0; i < NQ; ++i) v[i] = pack(q[i]);
    if (ry == RM) min8_regs<RM>(v, o);
    if constexpr (RM > 4) {
      if (ry == RM - 1) min8_regs<RM - 1>(v, o);
      if (ry == RM - 2) min8_regs<RM - 2>(v, o);
      if (ry == RM - 3) min8_regs<RM - 3>(v, o);
    }
    if (more) fetch(ahead);
#pragma unroll
    for (int i = 0; i < OK; ++i) sm_zy[plane * PL + i * 64 + l] = o[i];
  };
  fetch(s0 - rz + wave);
  for (int g = wave; g < hist; g += 8)
    ymin(g, g + 8 < hist ? s0 - rz + g + 8 : s0 + rz + wave, g + 8 < hist || s0 + wave < s1);
  const int y = y0 + wave;
  const bool out = x0 + l < W && y < H;
  const i64 WH = (i64)W * H;
  uint32_t* d = dst + (i64)y * W + x0 + l;
  for (int c = s0; c < s1; c += OK) {
    if (c + wave < s1) ymin(hist + wave, c + OK + rz + wave, c + OK + wave < s1);
    __syncthreads();
    const uint32_t* p = sm_zy + wave * 64 + l;
    uint32_t o[OK];
    min8<0>([&] { const uint32_t v = *p; p += PL; return v; }, rz, o);
    if (out) {
#pragma unroll
      for (int k = 0; k < OK; ++k)
        if (c + k < s1) st_nt(d + (i64)(c + k) * WH, o[k]);
    }
    if (c + OK >= s1) break;  // uniform
    __syncthreads();
    shift_rows<512, OK, PL>(sm_zy, hist);
    __syncthreads();
  }
}

// Clamped box mean of (E, D) pairs along y or z, with NORM fused with the normalization; ero
// and dil (optional) receive E and D.  Bound by its 14 (16) bytes per voxel: 275 us for
// 70 x 1080 x 1280 at radius 4 (4.9 TB/s), 568 with an LDS tile per 64 outputs.
template <int R, bool NORM, typename TS>
__global__ __launch_bounds__(256) void k_box_run(const float2* __restrict__ src,
                                                 float2* __restrict__ dst, TS* __restrict__ norm,
                                                 const uint16_t* __restrict__ img,
                                                 float* __restrict__ ero, float* __restrict__ dil,
                                                 float min_int, int W, int L, i64 sa, i64 so,
                                                 int r, unsigned nxb, unsigned no, int len,
                                                 float k) {
  extern __shared__ float sm_box[];
  constexpr int STEP = 4 * OK;
  const int hist = 2 * r;
  float* B1 = sm_box;
  float* B2 = B1 + (hist + STEP) * 64;
  const RunAt a = run_at(L, so, nxb, no, len);
  const int xc = min(a.x0 + a.l, W - 1);
  float2 q[OK];
  uint16_t iq[OK];
  auto fetch = [&](int p) {
#pragma unroll
    for (int j = 0; j < OK; ++j) q[j] = src[a.base + (i64)clampi(p + j, 0, L - 1) * sa + xc];
  };
  auto put = [&](int row) {
#pragma unroll
    for (int j = 0; j < OK; ++j) {
      B1[(row + j) * 64 + a.l] = q[j].x;
      B2[(row + j) * 64 + a.l] = q[j].y;
    }
  };
  for (int g = a.wave; OK * g < hist; g += 4) {
    fetch(a.s0 - r + OK * g);
    put(OK * g);
  }
  if (a.s0 + OK * a.wave < a.s1) fetch(a.s0 + r + OK * a.wave);
  __syncthreads();
  for (int c0 = a.s0; c0 < a.s1; c0 += STEP) {
    const int c = c0 + OK * a.wave;
    if (c < a.s1) {
      put(hist + OK * a.wave);
      if (NORM) {
#pragma unroll
        for (int j = 0; j < OK; ++j) iq[j] = img[a.base + (i64)min(c + j, L - 1) * sa + xc];
      }
    }
    if (c + STEP < a.s1) fetch(c + STEP + r);
    __syncthreads();
    if (c < a.s1) {
      float e[OK], d[OK];
      const float* p = B1 + OK * a.wave * 64 + a.l;
      sum8<R>([&] { const float v = *p; p += 64; return v; }, r, e);
      p = B2 + OK * a.wave * 64 + a.l;
      sum8<R>([&] { const float v = *p; p += 64; return v; }, r, d);
      if (a.x0 + a.l < W) {
#pragma unroll
        for (int j = 0; j < OK; ++j) {
          if (c + j >= a.s1) continue;
          const i64 idx = a.base + (i64)(c + j) * sa + a.x0 + a.l;
          const float ve = e[j] * k, vd = d[j] * k;
          if (NORM) {
            const float I = (float)iq[j];
            st_nt(norm + idx, (I >= min_int) ? (I - ve) / (vd - ve) : 0.0f);
            if (ero) {  // uniform
              st_nt(ero + idx, ve);
              st_nt(dil + idx, vd);
            }
          } else {
            st_nt(dst + idx, make_float2(ve, vd));
          }
        }
      }
    }
    if (c0 + STEP >= a.s1) break;  // uniform
    __syncthreads();
    shift_rows<256, STEP, 64>(B1, hist);
    shift_rows<256, STEP, 64>(B2, hist);
    __syncthreads();
  }
}

// The same for lines of at most kShallow positions: the positions that repeat at the line's ends
// are added as often as the window holds them, in its order.
template <bool NORM, typename TS>
__global__ __launch_bounds__(NT) void k_box_shallow(const float2* __restrict__ src,
                                                    float2* __restrict__ dst,
                                                    TS* __restrict__ norm,
                                                    const uint16_t* __restrict__ img,
                                                    float* __restrict__ ero,
                                                    float* __restrict__ dil, float min_int, int W,
                                                    int L, i64 sa, i64 so, int r, unsigned nxb,
                                                    unsigned no, float k) {
  const LineAt la = line_at_block(nxb, no, L, L);
  if (la.x >= W) return;
  const i64 base = (i64)la.other * so + la.x;
  float2 v[kShallow], last = make_float2(0.0f, 0.0f);
  uint16_t iv[kShallow];
#pragma unroll
  for (int i = 0; i < kShallow; ++i)
    if (i < L) {  // uniform, as all that follow
      v[i] = src[base + i * sa];
      if (NORM) iv[i] = img[base + i * sa];
      last = v[i];
    }
#pragma unroll
  for (int c = 0; c < kShallow; ++c) {
    if (c >= L) break;
    float e = 0.0f, d = 0.0f;
    // taps at or before the first position (all of them on a line of one), and after the last
    const int first = L == 1 ? 2 * r + 1 : r - c + 1, beyond = L == 1 ? 0 : c + r - (L - 2);
    for (int t = 0; t < first; ++t) {
      e += v[0].x;
      d += v[0].y;
    }
#pragma unroll
    for (int i = 1; i < kShallow - 1; ++i)
      if (i < L - 1 && i - c <= r && c - i <= r) {
        e += v[i].x;
        d += v[i].y;
      }
    for (int t = 0; t < beyond; ++t) {
      e += last.x;
      d += last.y;
    }
    const i64 idx = base + c * sa;
    const float ve = e * k, vd = d * k;
    if (NORM) {
      const float I = (float)iv[c];
      st_nt(norm + idx, (I >= min_int) ? (I - ve) / (vd - ve) : 0.0f);
      if (ero) {
        st_nt(ero + idx, ve);
        st_nt(dil + idx, vd);
      }
    } else {
      st_nt(dst + idx, make_float2(ve, vd));
    }
  }
}

// min/max along x, box along x and box along y fused (k_norm_xy_walk for other radii): four
// waves walk the rows of one plane of the y-min/maxed volume for a strip of 64 columns, eight
// rows per wave and step.
//   1. a wave's rows, columns x0-2r .. x0+63+2r clamped to the plane, enter its lines A;
//   2. lane (row l % 8, columns 8 (l / 8) ..) forms the window minima, two groups of eight at
//      most, which replace the lines; positions outside the plane take the edge's value;
//   3. the same lane sums them for its eight columns -> two planes B of the last 2r + 32 rows;
//   4. lane l sums eight rows of column x0 + l along y, in the reference order.
// (padded pitches: the lanes of every access fall on different banks.)  Near its 12 bytes per
// voxel at small radii (70 x 1080 x 1280: 314 us at radius 8, 3.7 TB/s), bound by instruction
// issue above (478 us at 16); the x pass and the y pass it replaces, one output per thread,
// took 698 us at 8.
template <int R, int NC>
__global__ __launch_bounds__(256) void k_norm_xy_run(const uint32_t* __restrict__ src,
                                                     float2* __restrict__ dst, int W, int H, int r,
                                                     int nxs, int nys, int rows, float k) {
  extern __shared__ uint32_t sm_xy[];
  constexpr int BP = 65, STEP = 4 * OK;
  const int hist = 2 * r, span = 64 + 4 * r, AP = (span + 7) / 8 * 8 + 9;
  const int l = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  uint32_t* A = sm_xy + wave * (OK * AP);
  float* B1 = reinterpret_cast<float*>(sm_xy + 4 * (OK * AP));
  float* B2 = B1 + (hist + STEP) * BP;
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int y0 = (int)(t % (unsigned)nys) * rows, y1 = min(H, y0 + rows);
  const unsigned tile = t / (unsigned)nys;
  const int x0 = (int)(tile % (unsigned)nxs) * 64;
  const i64 pbase = (i64)(tile / (unsigned)nxs) * H * W;
  int xl[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) xl[j] = clampi(x0 - 2 * r + 64 * j + l, 0, W - 1);
  uint32_t q[OK][NC];
  auto fetch = [&](int y) {
#pragma unroll
    for (int i = 0; i < OK; ++i) {
      const uint32_t* row = src + pbase + (i64)clampi(y + i, 0, H - 1) * W;
#pragma unroll
      for (int j = 0; j < NC; ++j) q[i][j] = row[xl[j]];
    }
  };
  const bool edge = x0 - r < 0 || x0 + 64 + r > W;  // uniform
  const int blo = r - x0, bhi = W - 1 - x0 + r;     // minima positions of x = 0 and W - 1
  const int nm = 64 + 2 * r;                        // minima per row
  const int xr = l % OK, xg = l / OK;
  const uint32_t full = (uint32_t)(2 * r + 1) * 65535u;
  auto xpass = [&](int row, int ahead) {
#pragma unroll
    for (int i = 0; i < OK; ++i)
#pragma unroll
      for (int j = 0; j < NC; ++j)
        if (64 * j + l < span) A[i * AP + 64 * j + l] = q[i][j];
    fetch(ahead);
    wave_lds_sync();
    uint32_t* line = A + xr * AP;
    uint32_t m[2][OK];
    {
      const uint32_t* p = line + OK * xg;
      min8<R>([&] { return *p++; }, r, m[0]);
    }
    const bool two = OK * (xg + 8) < nm;
    if (two) {
      const uint32_t* p = line + OK * (xg + 8);
      min8<R>([&] { return *p++; }, r, m[1]);
    }
    wave_lds_sync();
#pragma unroll
    for (int o = 0; o < OK; ++o) line[OK * xg + o] = m[0][o];
    if (two) {
#pragma unroll
      for (int o = 0; o < OK; ++o) line[OK * (xg + 8) + o] = m[1][o];
    }
    wave_lds_sync();
    if (edge) {  // each lane its row: positions outside the plane take the edge value
      const uint32_t lo = line[clampi(blo, 0, nm - 1)], hi = line[clampi(bhi, 0, nm - 1)];
      wave_lds_sync();
      for (int j = xg; j < nm; j += 8) {
        if (j < blo) line[j] = lo;
        if (j > bhi) line[j] = hi;
      }
      wave_lds_sync();
    }
    uint32_t se[OK], sd[OK];
    {
      const uint32_t* p = line + OK * xg;
      sum8_u16<R>([&] { return *p++; }, r, se, sd);
    }
    const int b = (row + xr) * BP + xg * OK;
#pragma unroll
    for (int o = 0; o < OK; ++o) {
      B1[b + o] = (float)se[o] * k;
      B2[b + o] = (float)(full - sd[o]) * k;
    }
    wave_lds_sync();
  };
  const int main0 = y0 + r + OK * wave;
  if (OK * wave < hist) {
    fetch(y0 - r + OK * wave);
    for (int g = wave; OK * g < hist; g += 4)
      xpass(OK * g, OK * (g + 4) < hist ? y0 - r + OK * (g + 4) : main0);
  } else {
    fetch(main0);
  }
  __syncthreads();
  const bool out = x0 + l < W;
  float2* dcol = dst + pbase + x0 + l;
  for (int c0 = y0; c0 < y1; c0 += STEP) {
    xpass(hist + OK * wave, c0 + STEP + r + OK * wave);
    __syncthreads();
    const int c = c0 + OK * wave;
    if (c < y1) {
      float e[OK], d[OK];
      const float* p = B1 + OK * wave * BP + l;
      sum8<R>([&] { const float v = *p; p += BP; return v; }, r, e);
      p = B2 + OK * wave * BP + l;
      sum8<R>([&] { const float v = *p; p += BP; return v; }, r, d);
      if (out) {
#pragma unroll
        for (int o = 0; o < OK; ++o)
          if (c + o < y1) st_nt(dcol + (i64)(c + o) * W, make_float2(e[o] * k, d[o] * k));
      }
    }
    if (c0 + STEP >= y1) break;  // uniform
    __syncthreads();
    shift_rows<256, STEP, BP>(B1, hist);
    shift_rows<256, STEP, BP>(B2, hist);
    __syncthreads();
  }
}

template <typename TS>
__global__ __launch_bounds__(NT) void k_copy_norm(const uint16_t* __restrict__ img,
                                                  TS* __restrict__ norm, float min_int, i64 N) {
  for (i64 i = (i64)blockIdx.x * NT + threadIdx.x; i < N; i += (i64)gridDim.x * NT) {
    const float v = (float)img[i];
    norm[i] = cvt<TS>((v >= min_int) ? v : 0.0f);
  }
}

struct LineCfg { int XW, C; };
LineCfg line_cfg(int r, int L, size_t elem_bytes, int arrays) {
  LineCfg c{64, 64};
  if (r > 24) c.XW = 32;
  if ((size_t)arrays * (c.C + 2 * r) * c.XW * elem_bytes > 60 * 1024) c.XW = 16;
  if (L < c.C) c.C = L;
  return c;
}

template <typename F>
hipError_t dispatch_xw(int XW, F&& f) {
  if (XW == 64) return f(std::integral_constant<int, 64>{});
  if (XW == 32) return f(std::integral_constant<int, 32>{});
  return f(std::integral_constant<int, 16>{});
}

template <int R>
hipError_t minmax_walk(const void* src, bool from_u16, uint32_t* dst, int W, int L, i64 sa, i64 so,
                       i64 n_other, hipStream_t s) {
  const LineGrid g = line_grid(W, L, n_other, 2 * R);
  if (from_u16)
    hipLaunchKernelGGL((k_minmax_walk<R, true>), dim3(g.blocks), dim3(NT), 0, s, src, dst, W, L, sa,
                       so, g.nxb, g.no, g.len);
  else
    hipLaunchKernelGGL((k_minmax_walk<R, false>), dim3(g.blocks), dim3(NT), 0, s, src, dst, W, L,
                       sa, so, g.nxb, g.no, g.len);
  return hipGetLastError();
}

hipError_t minmax_line(const void* src, bool from_u16, uint32_t* dst, int W, int L, i64 sa,
                       i64 so, i64 n_other, int r, hipStream_t s) {
  if (L <= kShallow) {
    const unsigned nxb = (unsigned)((W + NT - 1) / NT);
    const dim3 grid((unsigned)(nxb * n_other));
    if (from_u16)
      hipLaunchKernelGGL((k_minmax_shallow<true>), grid, dim3(NT), 0, s, src, dst, W, L, sa, so, r,
                         nxb, (unsigned)n_other);
    else
      hipLaunchKernelGGL((k_minmax_shallow<false>), grid, dim3(NT), 0, s, src, dst, W, L, sa, so, r,
                         nxb, (unsigned)n_other);
    return hipGetLastError();
  }
  // the configured radius has a walk with its window in registers (70 x 1080 x 1280 along y:
  // 166 us; the walk of any radius 180 at 8, 182 at 12; at 3 and 5 the two take the same)
  if (r == 10) return minmax_walk<10>(src, from_u16, dst, W, L, sa, so, n_other, s);
  if (r <= kRunRadius) {
    const LineGrid g = run_grid(W, L, n_other, 2 * r);
    const size_t lds = (size_t)(2 * r + 32) * 64 * 4;
    return dispatch_short(r, [&](auto rs) {
      constexpr int R = decltype(rs)::value;
      if (from_u16)
        hipLaunchKernelGGL((k_minmax_run<R, true>), dim3(g.blocks), dim3(256), lds, s, src, dst, W,
                           L, sa, so, r, g.nxb, g.no, g.len);
      else
        hipLaunchKernelGGL((k_minmax_run<R, false>), dim3(g.blocks), dim3(256), lds, s, src, dst, W,
                           L, sa, so, r, g.nxb, g.no, g.len);
      return hipGetLastError();
    });
  }
  const LineCfg c = line_cfg(r, L, 4, 2);
  const int nxt = (W + c.XW - 1) / c.XW, nct = (L + c.C - 1) / c.C;
  const i64 nblk = (i64)nxt * nct * n_other;
  const size_t lds = 2 * (size_t)(c.C + 2 * r) * c.XW * 4;
  return dispatch_xw(c.XW, [&](auto xw) {
    constexpr int XW = decltype(xw)::value;
    if (from_u16)
      hipLaunchKernelGGL((k_minmax_line<XW, true>), dim3((unsigned)nblk), dim3(NT), lds, s, src,
                         dst, W, L, sa, so, r, c.C, nxt, nct);
    else
      hipLaunchKernelGGL((k_minmax_line<XW, false>), dim3((unsigned)nblk), dim3(NT), lds, s,
                         src, dst, W, L, sa, so, r, c.C, nxt, nct);
    return hipGetLastError();
  });
}

template <int R, bool NORM, typename TS>
hipError_t box_line_fast(const float2* src, float2* dst, TS* norm, const uint16_t* img,
                         float min_int, int W, int L, i64 sa, i64 so, i64 n_other, float k,
                         hipStream_t s) {
  const LineGrid g = line_grid(W, L, n_other, 2 * R);
  hipLaunchKernelGGL((k_box_walk<R, NORM, TS>), dim3(g.blocks), dim3(NT), 0, s, src, dst, norm, img,
                     min_int, W, L, sa, so, g.nxb, g.no, g.len, k);
  return hipGetLastError();
}

template <bool NORM, typename TS>
hipError_t box_line(const float2* src, float2* dst, TS* norm, const uint16_t* img, float min_int,
                    int W, int L, i64 sa, i64 so, i64 n_other, int r, hipStream_t s,
                    float* ero = nullptr, float* dil = nullptr) {
  const float k = 1.0f / (float)(2 * r + 1);
  const bool ed = NORM && ero && dil;  // the walks of any radius write them
  if (L <= kShallow) {
    const unsigned nxb = (unsigned)((W + NT - 1) / NT);
    hipLaunchKernelGGL((k_box_shallow<NORM, TS>), dim3((unsigned)(nxb * n_other)), dim3(NT), 0, s,
                       src, dst, norm, img, ed ? ero : nullptr, ed ? dil : nullptr, min_int, W, L,
                       sa, so, r, nxb, (unsigned)n_other, k);
    return hipGetLastError();
  }
  // (70 x 1080 x 1280, fused with the normalization: 267 us; the walk of any radius 275 at 4,
  // 277 at 6)
  if (r == 10 && !ed)
    return box_line_fast<10, NORM, TS>(src, dst, norm, img, min_int, W, L, sa, so, n_other, k, s);
  if (r <= kRunRadius) {
    const LineGrid g = run_grid(W, L, n_other, 2 * r);
    const size_t lds = 2 * (size_t)(2 * r + 32) * 64 * 4;
    return dispatch_short(r, [&](auto rs) {
      constexpr int R = decltype(rs)::value;
      hipLaunchKernelGGL((k_box_run<R, NORM, TS>), dim3(g.blocks), dim3(256), lds, s, src, dst,
                         norm, img, ed ? ero : nullptr, ed ? dil : nullptr, min_int, W, L, sa, so,
                         r, g.nxb, g.no, g.len, k);
      return hipGetLastError();
    });
  }
  const LineCfg c = line_cfg(r, L, 8, 1);
  const int nxt = (W + c.XW - 1) / c.XW, nct = (L + c.C - 1) / c.C;
  const i64 nblk = (i64)nxt * nct * n_other;
  const size_t lds = (size_t)(c.C + 2 * r) * c.XW * 8;
  return dispatch_xw(c.XW, [&](auto xw) {
    constexpr int XW = decltype(xw)::value;
    hipLaunchKernelGGL((k_box_line<XW, NORM, TS>), dim3((unsigned)nblk), dim3(NT), lds, s, src,
                       dst, norm, img, min_int, W, L, sa, so, r, c.C, nxt, nct, k);
    return hipGetLastError();
  });
}

__global__ __launch_bounds__(NT) void k_split_ed(const float2* __restrict__ ed,
                                                 float* __restrict__ ero, float* __restrict__ dil,
                                                 i64 N) {
  for (i64 i = (i64)blockIdx.x * NT + threadIdx.x; i < N; i += (i64)gridDim.x * NT) {
    const float2 v = ed[i];
    ero[i] = v.x;
    dil[i] = v.y;
  }
}

}  // namespace

hipError_t launch_box_pair(const float2* src, float2* dst, int W, int L, i64 sa, i64 so,
                           i64 n_other, int r, hipStream_t s) {
  return box_line<false, float>(src, dst, nullptr, nullptr, 0.0f, W, L, sa, so, n_other, r, s);
}

// The row walker with its window in registers (radius 10) takes a wave per strip of 128
// columns.  Too few strips leave the chip idle or are cut into segments that each walk 20 rows
// more; the walk of any radius puts four waves on a strip of 64 (x min/max and x/y boxes,
// strips: its us / the walker's): 24 x 96 x 112, 24: 12 / 28; 128 x 256 x 256, 256: 51 / 67;
// 64 x 512 x 512, 256: 83 / 99; 96 x 512 x 512, 384: 120 / 121; 128 x 512 x 512, 512: 149 / 140;
// 300 x 200 x 200, 600: 85 / 68; 32 x 2160 x 2560, 640: 655 / 558.
static bool norm_row_walker(int rxy, int W, int D) {
  return rxy == 10 && (i64)((W + 127) / 128) * D > 384;
}

WalkShape norm_walk_shape(int rxy, int W, int D) {
  if (norm_row_walker(rxy, W, D)) return {(i64)((W + 127) / 128) * D, 21, 20};
  return {(i64)((W + 63) / 64) * D * 4, 32, 2 * rxy};
}

template <typename TS>
hipError_t launch_normalize(const uint16_t* img, TS* norm, void* tmp1, void* tmp2,
                            float min_intensity, int W, int H, int D, int rxy, int rz,
                            hipStream_t s, float* ero, float* dil, int segments) {
  const i64 WH = (i64)W * H, N = WH * D;
  if (rxy == 0 || rz == 0) {
    const i64 nb = std::min<i64>((N + NT - 1) / NT, 1 << 20);
    hipLaunchKernelGGL((k_copy_norm<TS>), dim3((unsigned)nb), dim3(NT), 0, s, img, norm,
                       min_intensity, N);
    mark("normalize/copy", s);
    return hipGetLastError();
  }
  hipError_t e;
  const ZColumns zc = z_columns(W, H);
  uint32_t* p1 = (uint32_t*)tmp1;
  uint32_t* p2 = (uint32_t*)tmp2;
  // The z walk of radius 10 keeps its window in registers and goes slice by slice, a barrier
  // each; the walk of other radii goes eight slices at a time, which is sooner done where there
  // are few (slices of 64 x 32 tiles: its us / the walk's): 24 x 96 x 112, 144: 10 / 18;
  // 40 x 160 x 160, 600: 13 / 23; 64 x 200 x 200, 1792: 22 / 24; 128 x 256 x 256, 4096: 32 / 30;
  // 20 x 1080 x 1280, 13600: 92 / 59.
  const unsigned nxt = (W + 63) / 64, nyt = (H + 31) / 32;
  if (rxy == 10 && rz == 10 && (i64)nxt * nyt * D > 2048 && WH * 4 < 0xFFFFFFF0ll) {
    // min/max along y and z in one z walk over 64 x 32 tiles (slices addressed by buffer
    // descriptors with 32-bit byte offsets)
    int nzs, zlen;
    // one 1024-thread work-group per CU: whole rounds of 256 (128 x 256 x 256, 32 work-groups
    // per segment: 93 us whole, 28 in eight segments, 43 in twelve)
    line_segments(D, (i64)nxt * nyt, 256.0, 1.0, true, 24, &nzs, &zlen);
    hipLaunchKernelGGL((k_minmax_zy_walk<10, 10, HDOG_ZY_PF>),
                       dim3((unsigned)((i64)nxt * nyt * nzs)), dim3(1024), 0, s, img, p2, W, H, D,
                       nyt, nxt, zlen);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    mark("normalize/minmax_zy", s);
    } else if (rxy >= 4 && rxy <= kZyRadiusY && rz >= 4 && rz <= kZyRadiusZ) {
    const unsigned nyg = (H + OK - 1) / OK;
    int nzs, zlen;
    line_segments(D, (i64)nxt * nyg * 8, 1024.0, 2.0, false, 2 * rz, &nzs, &zlen);
    const dim3 grid((unsigned)((i64)nxt * nyg * nzs));
    const size_t lds = (size_t)(2 * rz + OK) * OK * 64 * 4;
#define X(NQ)                                                                                   \
  if (2 * rxy + OK <= NQ && 2 * rxy > NQ - 2 * OK)                                                 \
    hipLaunchKernelGGL((k_minmax_zy_run<NQ>), grid, dim3(512), lds, s, img, p2, W, H, D, rxy, rz, \
                       nyg, nxt, zlen);
    X(16) X(24) X(32) X(40)
#undef X
    static_assert(2 * kZyRadiusY + OK == 40, "the largest");
    if ((e = hipGetLastError()) != hipSuccess) return e;
    mark("normalize/minmax_zy", s);
  } else {
    // min/max along z (lines over x, y fixed per work-group), then along y
    if ((e = minmax_line(img, true, p1, zc.n, D, WH, W, zc.rows, rz, s)) != hipSuccess) return e;
    mark("normalize/minmax_z", s);
    if ((e = minmax_line(p1, false, p2, W, H, W, WH, D, rxy, s)) != hipSuccess) return e;
    mark("normalize/minmax_y", s);
  }
  // min/max along x, box along x and box along y in one row walker -> (E, D) in tmp1
  const float2* exy = (const float2*)tmp1;
  const float k = 1.0f / (float)(2 * rxy + 1);
  if (norm_row_walker(rxy, W, D)) {
    constexpr int CW = 128;
    const int nxs = (W + CW - 1) / CW;
    int nys, rows;
    walk_segments(H, norm_walk_shape(rxy, W, D), &nys, &rows, segments);
    const i64 nblk = (i64)nxs * D * nys;
    hipLaunchKernelGGL((k_norm_xy_walk<10>), dim3((unsigned)nblk), dim3(64), 0, s, p2,
                       (float4*)tmp1, W, H, nxs, nys, rows, k);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    mark("normalize/minmax_x_box_xy", s);
  } else if (rxy <= kRunRadius && 2 * H >= 3 * rxy) {
    // (a walk forms the x windows of 2 rxy rows above and below a plane's own; on planes of fewer
    // rows than half of those, the two passes below are sooner done: 300 x 5 x 2000 at radius 8
    // 75 us, the walk 104; x 8 at 16: 98, 161; x 33 at 23: 351, 557.  300 x 15 x 300 at 8: 38, 35;
    // 100 x 30 x 300 at 16: 38, 32)
    const int nxs = (W + 63) / 64;
    int nys, rows;
    walk_segments(H, norm_walk_shape(rxy, W, D), &nys, &rows, segments);
    const dim3 grid((unsigned)((i64)nxs * D * nys));
    const int ap = (64 + 4 * rxy + 7) / 8 * 8 + 9;  // the kernel's line pitch
    const size_t lds = (size_t)(4 * OK * ap + 2 * (2 * rxy + 32) * 65) * 4;
    e = dispatch_short(rxy, [&](auto rs) {
      constexpr int R = decltype(rs)::value;
      if (rxy <= 16)
        hipLaunchKernelGGL((k_norm_xy_run<R, 2>), grid, dim3(256), lds, s, p2, (float2*)tmp1, W, H,
                           rxy, nxs, nys, rows, k);
      else
        hipLaunchKernelGGL((k_norm_xy_run<0, 3>), grid, dim3(256), lds, s, p2, (float2*)tmp1, W, H,
                           rxy, nxs, nys, rows, k);
      return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    mark("normalize/minmax_x_box_xy", s);
  } else {
    // min/max along x fused with the box x pass -> float2 (E, D) in tmp1, then box along y
    constexpr int RUN = 4, C = 64 * RUN, ROWS = NT / 64;
    const int nct = (W + C - 1) / C;
    const i64 nrows = (i64)H * D;
    const i64 nblk = ((nrows + ROWS - 1) / ROWS) * nct;
    const size_t lds = (size_t)ROWS * 2 * (C + 4 * rxy + 4) * 4;
    hipLaunchKernelGGL((k_minmax_x_box<RUN>), dim3((unsigned)nblk), dim3(NT), lds, s, p2,
                       (float2*)tmp1, W, nrows, rxy, nct, k);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    mark("normalize/minmax_x_box_x", s);
    if ((e = box_line<false, float>((const float2*)tmp1, (float2*)tmp2, nullptr, nullptr, 0.0f, W, H,
                                 W, WH, D, rxy, s)) != hipSuccess)
      return e;
    mark("normalize/box_y", s);
    exy = (const float2*)tmp2;
  }
  // box along z fused with the normalization
  if (ero && dil && rz > kRunRadius) {  // E and D by a z pass of their own, then split
    float2* ed = exy == (const float2*)tmp1 ? (float2*)tmp2 : (float2*)tmp1;
    if ((e = box_line<false, float>(exy, ed, nullptr, nullptr, 0.0f, zc.n, D, WH, W, zc.rows, rz, s)) !=
        hipSuccess)
      return e;
    const i64 nb = std::min<i64>((N + NT - 1) / NT, 1 << 20);
    hipLaunchKernelGGL(k_split_ed, dim3((unsigned)nb), dim3(NT), 0, s, (const float2*)ed, ero, dil,
                       N);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  e = box_line<true, TS>(exy, nullptr, norm, img, min_intensity, zc.n, D, WH, W, zc.rows, rz, s,
                         rz <= kRunRadius ? ero : nullptr, dil);
  mark("normalize/box_z_norm", s);
  return e;
}

template hipError_t launch_normalize<float>(const uint16_t*, float*, void*, void*, float, int,
                                            int, int, int, int, hipStream_t, float*, float*, int);
template hipError_t launch_normalize<__half>(const uint16_t*, __half*, void*, void*, float, int,
                                             int, int, int, int, hipStream_t, float*, float*, int);
template hipError_t launch_normalize<__hip_bfloat16>(const uint16_t*, __hip_bfloat16*, void*,
                                                     void*, float, int, int, int, int, int,
                                                     hipStream_t, float*, float*, int);

}  // namespace hdog
