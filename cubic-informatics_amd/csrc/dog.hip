// dog.hip -- separable anisotropic difference of Gaussians on gfx950.
//
// Reference semantics: src/3D/DoG3DFilter.cu:70-437.  Each Gaussian is x -> y (xy
// weights) -> z (z weights) with zero padding; every output is the FMA chain
// sum = fmaf(w[r-j], s[c+j], sum), j = -r..r, from 0.  dog = (G1 - G2) * normalizer.
//
// MI355X design: both Gaussians are evaluated from one read of `norm`.  The x and y passes are
// one walk over the rows of a plane, which writes the pair (G1, G2) as float2, and the z pass
// forms the difference of the pair directly, so the reference's intermediate volumes become
// one interleaved stream.  Intermediates stay FP32 whatever the storage type of norm / dog.
//
// Radius pairs (r1, r2) that occur in practice have compile-time kernels: a row walker along x
// and y, and along z a column walker (one thread per line, a register ring, every input read
// once, no LDS).  Other radii, and the smallest stacks along x and y, have walks with their
// history in LDS that form eight outputs at a time; along z up to eight slices of those radii
// are a thread's registers.
#include "hdog_internal.hpp"

namespace hdog {
namespace {

constexpr int NT = 256;

// ------------------------------------------------------------------- any radii
// Sums of eight consecutive outputs of one Gaussian of radius r: every input is read once and
// meets its outputs' accumulators in turn, so each output is the chain over ascending inputs,
// and no tap outside the window is formed (a zero weight would still turn an infinite or NaN
// input into NaN).  next() gives inputs c - r, c - r + 1, ... c + 7 + r.  The weights are
// symmetric (both halves are set from one value); the lanes of `wv` hold them, w[j] in lane j
// or, for more than 64 (WIDE), w[r + j], and a tap's weight is read from there into a scalar
// register, an operand of its FMAs; loaded from memory, every four inputs waited for their
// weights, and with them for all LDS reads.
constexpr int GK = 8;
constexpr int kLaneRadius = 31;  // 2r + 1 weights fit a wave's lanes
template <bool WIDE>
__device__ __forceinline__ float gauss_lanes(const float* w, int r) {
  const int l = (int)(threadIdx.x & 63);
  return WIDE ? w[r + min(l, r)] : w[min(l, 2 * r)];
}
template <bool WIDE>
__device__ __forceinline__ float gauss_tap(float wv, int t, int r) {  // weight of tap t
  const int l = WIDE ? abs(t - r) : t;
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(wv), l));
}
template <bool WIDE, int R, typename F>
__device__ __forceinline__ void gauss8_short(F&& next, float wv, float (&acc)[GK]) {
  float v[2 * R + GK];
#pragma unroll
  for (int i = 0; i < 2 * R + GK; ++i) v[i] = next();
#pragma unroll
  for (int i = 0; i < 2 * R + GK; ++i)
#pragma unroll
    for (int o = 0; o < GK; ++o)
      if (i - o >= 0 && i - o <= 2 * R) acc[o] = fmaf(gauss_tap<WIDE>(wv, i - o, R), v[i], acc[o]);
}
template <bool WIDE, typename F>
__device__ __forceinline__ void gauss8(F&& next, float wv, int r, float (&acc)[GK]) {
#pragma unroll
  for (int o = 0; o < GK; ++o) acc[o] = 0.0f;
  if (r < 3) {  // uniform: fewer taps than outputs
    if (r == 0) gauss8_short<WIDE, 0>(next, wv, acc);
    if (r == 1) gauss8_short<WIDE, 1>(next, wv, acc);
    if (r == 2) gauss8_short<WIDE, 2>(next, wv, acc);
    return;
  }
  // inputs 0 .. 6 start the outputs, 7 .. 2r meet all eight, 2r + 1 .. 2r + 7 end them;
  // four inputs are always read ahead of their use
  float h[GK - 1], v[4], e[GK - 1];
  float t[GK + 3];  // weights of taps i - 7 .. i + 3 at input i
#pragma unroll
  for (int i = 0; i < GK - 1; ++i) h[i] = next();
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = next();
#pragma unroll
  for (int i = 0; i < GK - 1; ++i) e[i] = t[i] = gauss_tap<WIDE>(wv, i, r);
#pragma unroll
  for (int i = 0; i < GK - 1; ++i)
#pragma unroll
    for (int o = 0; o <= i; ++o) acc[o] = fmaf(e[i - o], h[i], acc[o]);
  int i = GK - 1;
#pragma unroll 1
  for (; i + 3 <= 2 * r; i += 4) {
    float n[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) n[q] = next();
#pragma unroll
    for (int q = 0; q < 4; ++q) t[GK - 1 + q] = gauss_tap<WIDE>(wv, i + q, r);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int o = 0; o < GK; ++o) acc[o] = fmaf(t[GK - 1 + q - o], v[q], acc[o]);
#pragma unroll
    for (int q = 0; q < GK - 1; ++q) t[q] = t[q + 4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = n[q];
  }
  // the end: tap 2r + u - o of input 2r + u, whose weight is that of tap o - u
  auto end = [&](const float* z) {
#pragma unroll
    for (int u = 1; u < GK; ++u)
#pragma unroll
      for (int o = u; o < GK; ++o) acc[o] = fmaf(e[o - u], z[u - 1], acc[o]);
  };
  if (i <= 2 * r) {  // two inputs left before it (2r - 6 is even)
    float z[GK + 1] = {v[0], v[1], v[2], v[3]};
#pragma unroll
    for (int q = 4; q < GK + 1; ++q) z[q] = next();
#pragma unroll
    for (int q = 0; q < 2; ++q) t[GK - 1 + q] = gauss_tap<WIDE>(wv, i + q, r);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int o = 0; o < GK; ++o) acc[o] = fmaf(t[GK - 1 + q - o], z[q], acc[o]);
    end(z + 2);
  } else {
    float z[GK - 1] = {v[0], v[1], v[2], v[3]};
#pragma unroll
    for (int q = 4; q < GK - 1; ++q) z[q] = next();
    end(z);
  }
}

// x and y passes of both Gaussians for any radii.  A work-group of NW waves walks the rows of
// one plane for a strip of 64 columns, eight rows per wave and step:
//   1. a wave's eight rows x0-RX .. x0+63+RX, loaded a step ahead through row descriptors
//      (zero outside the plane), enter its LDS lines A;
//   2. lane (row l % 8, columns 8 (l / 8) ..) forms eight x outputs of each Gaussian, which
//      enter two LDS planes B below the 2RY rows before them (padded pitches: the lanes of
//      both accesses fall on different banks);
//   3. lane l forms eight y outputs of column x0 + l; then the last 2RY rows of B move up.
// The (G1_x, G2_x) volume between the passes is never stored.  Bound by instruction issue
// (2 (rx1 + rx2 + ry1 + ry2 + 2) FMAs per voxel): the LDS leaves three waves per SIMD at
// radius 14, and four waves sharing B keep it at that; one wave with B as a ring of its own
// left one or two, whose ring arithmetic then cost as much as the FMAs (606 us, below).  One
// output per thread with a read per tap, in two passes through memory, took 1360 us for
// 61 x 900 x 1111 at radii 9 / 14; this takes 356 us.
template <typename TS, int NC, int NW>
__global__ __launch_bounds__(64 * NW) void k_gauss_xy_run(
    const TS* __restrict__ src, float2* __restrict__ dst, const float* __restrict__ wx1,
    const float* __restrict__ wx2, const float* __restrict__ wy1, const float* __restrict__ wy2,
    int rx1, int rx2, int ry1, int ry2, int W, int H, int nxs, int nys, int rows) {
  extern __shared__ float sm_xy[];
  constexpr bool WIDE = NC > 2;
  constexpr int BP = 65, STEP = GK * NW;  // pitch of B, rows per step
  const int RX = max(rx1, rx2), RY = max(ry1, ry2), hist = 2 * RY;
  const int AP = (64 + 2 * RX + 7) / 8 * 8 + 1, NRB = hist + STEP;
  const int l = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  float* A = sm_xy + wave * (GK * AP);
  float* B1 = sm_xy + NW * (GK * AP);
  float* B2 = B1 + NRB * BP;
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int y0 = (int)(t % (unsigned)nys) * rows, y1 = min(H, y0 + rows);
  const unsigned tile = t / (unsigned)nys;
  const int x0 = (int)(tile % (unsigned)nxs) * 64;
  const i64 pbase = (i64)(tile / (unsigned)nxs) * H * W;
  typedef typename StoredBits<TS>::type Bits;
  Bits q[GK][NC];
  const uint32_t row_bytes = (uint32_t)W * (uint32_t)sizeof(TS);
  // column x0 - RX + 64 k + l; left of the row the offset wraps past the record count
  uint32_t off[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = 64 * k + l;
    off[k] = c < 64 + 2 * RX ? (uint32_t)(x0 - RX + c) * (uint32_t)sizeof(TS) : 0xFFFFFFF0u;
  }
  auto fetch = [&](int y) {
#pragma unroll
    for (int r = 0; r < GK; ++r) {
      const bool in = y + r >= 0 && y + r < H;
      const __amdgpu_buffer_rsrc_t rs =
          buf_rsrc(src + pbase + (i64)(in ? y + r : 0) * W, in ? row_bytes : 0u);
#pragma unroll
      for (int k = 0; k < NC; ++k) q[r][k] = buf_load<TS>(rs, off[k]);
    }
  };
  const float vx1 = gauss_lanes<WIDE>(wx1, rx1), vx2 = gauss_lanes<WIDE>(wx2, rx2),
              vy1 = gauss_lanes<WIDE>(wy1, ry1), vy2 = gauss_lanes<WIDE>(wy2, ry2);
  const int xr = l % GK, xg = l / GK;
  // x outputs of the eight fetched rows into rows `row` .. of B, fetching rows `ahead` ..
  auto xpass = [&](int row, int ahead) {
#pragma unroll
    for (int r = 0; r < GK; ++r)
#pragma unroll
      for (int k = 0; k < NC; ++k)
        if (64 * k + l < 64 + 2 * RX) A[r * AP + 64 * k + l] = from_bits<TS>(q[r][k]);
    fetch(ahead);
    wave_lds_sync();
#pragma unroll 1
    for (int g = 0; g < 2; ++g) {  // one copy of the sums for both Gaussians
      const int r = g ? rx2 : rx1;
      const float* p = A + xr * AP + xg * GK + (RX - r);
      float acc[GK];
      gauss8<WIDE>([&] { return *p++; }, g ? vx2 : vx1, r, acc);
      float* b = (g ? B2 : B1) + (row + xr) * BP + xg * GK;
#pragma unroll
      for (int o = 0; o < GK; ++o) b[o] = acc[o];
    }
    wave_lds_sync();
  };
  // the rows above the segment (the last eight may reach into the first step's rows, which
  // are written again after the barrier)
  const int main0 = y0 + RY + GK * wave;
  if (GK * wave < hist) {
    fetch(y0 - RY + GK * wave);
    for (int g = wave; GK * g < hist; g += NW)
      xpass(GK * g, GK * (g + NW) < hist ? y0 - RY + GK * (g + NW) : main0);
  } else {
    fetch(main0);
  }
  __syncthreads();
  const bool out = x0 + l < W;
  float2* dcol = dst + pbase + x0 + l;
  for (int c0 = y0; c0 < y1; c0 += STEP) {
    xpass(hist + GK * wave, c0 + STEP + RY + GK * wave);
    __syncthreads();
    const int c = c0 + GK * wave;
    if (c < y1) {
      float a1[GK], a2[GK];
#pragma unroll 1
      for (int g = 0; g < 2; ++g) {
        const int r = g ? ry2 : ry1;
        const float* p = (g ? B2 : B1) + (GK * wave + RY - r) * BP + l;
        float acc[GK];
        gauss8<WIDE>([&] { const float v = *p; p += BP; return v; }, g ? vy2 : vy1, r, acc);
#pragma unroll
        for (int o = 0; o < GK; ++o) {
          if (g == 0) a1[o] = acc[o];
          a2[o] = acc[o];
        }
      }
      if (out) {
#pragma unroll
        for (int o = 0; o < GK; ++o)
          if (c + o < y1) st_nt(dcol + (i64)(c + o) * W, make_float2(a1[o], a2[o]));
      }
    }
    if (c0 + STEP >= y1) break;  // uniform
    __syncthreads();
    shift_rows<64 * NW, STEP, BP>(B1, hist);
    shift_rows<64 * NW, STEP, BP>(B2, hist);
    __syncthreads();
  }
}

// The z pass (sa = W H) for any radii: a work-group of four waves walks a
// segment of 64 x-adjacent lines, eight positions per wave and step, through two LDS planes of
// the last 2R + 32 positions (zero outside the line).  Bound by its 12 or 16 bytes per voxel
// for short windows (61 x 900 x 1111 along z at radii 4 / 7: 377 us with one output per thread
// and a read per tap, 198 us now).
template <bool DOT, bool WIDE, typename TS>
__global__ __launch_bounds__(256) void k_gauss_line_run(const float2* __restrict__ src,
                                                        TS* __restrict__ dog,
                                                        const float* __restrict__ a,
                                                        double* __restrict__ dots,
                                                        const float* __restrict__ w1,
                                                        const float* __restrict__ w2, int r1,
                                                        int r2, float nz, int W, int L, i64 sa,
                                                        i64 so, unsigned nxb, unsigned no,
                                                        int len) {
  extern __shared__ float sm_line[];
  constexpr int NW = 4, STEP = GK * NW;
  const int R = max(r1, r2), hist = 2 * R;
  float* B1 = sm_line;
  float* B2 = B1 + (hist + STEP) * 64;
  const int l = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int x0 = (int)(t % nxb) * 64;
  const i64 base = (i64)(t / nxb % no) * so + x0;
  const int s0 = (int)(t / nxb / no) * len, s1 = min(L, s0 + len);
  const uint32_t nrec = (uint32_t)min(64, W - x0) * (uint32_t)sizeof(float2);
  float2 q[GK];
  auto fetch = [&](int p) {
#pragma unroll
    for (int r = 0; r < GK; ++r) {
      const bool in = p + r >= 0 && p + r < L;
      const __amdgpu_buffer_rsrc_t rs =
          buf_rsrc(src + base + (i64)(in ? p + r : 0) * sa, in ? nrec : 0u);
      q[r] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(
                                            rs, l * (int)sizeof(float2), 0, 0));
    }
  };
  auto put = [&](int row) {
#pragma unroll
    for (int r = 0; r < GK; ++r) {
      B1[(row + r) * 64 + l] = q[r].x;
      B2[(row + r) * 64 + l] = q[r].y;
    }
  };
  const float v1 = gauss_lanes<WIDE>(w1, r1), v2 = gauss_lanes<WIDE>(w2, r2);
  for (int g = wave; GK * g < hist; g += NW) {
    fetch(s0 - R + GK * g);
    put(GK * g);
  }
  if (s0 + GK * wave < s1) fetch(s0 + R + GK * wave);
  __syncthreads();
  const bool out = x0 + l < W;
  double d[2] = {0.0, 0.0};
  for (int c0 = s0; c0 < s1; c0 += STEP) {
    const int c = c0 + GK * wave;
    if (c < s1) put(hist + GK * wave);
    if (c + STEP < s1) fetch(c + STEP + R);
    __syncthreads();
    if (c < s1) {
      float a1[GK], a2[GK];
      const float* p = B1 + (GK * wave + R - r1) * 64 + l;
      gauss8<WIDE>([&] { const float v = *p; p += 64; return v; }, v1, r1, a1);
      p = B2 + (GK * wave + R - r2) * 64 + l;
      gauss8<WIDE>([&] { const float v = *p; p += 64; return v; }, v2, r2, a2);
      if (out) {
#pragma unroll
        for (int o = 0; o < GK; ++o) {
          if (c + o >= s1) continue;
          const i64 idx = base + (i64)(c + o) * sa + l;
          if (DOT) {
            const double v = a[idx];
            d[0] += v * a1[o];
            d[1] += v * a2[o];
          } else {
            dog[idx] = cvt<TS>((a1[o] - a2[o]) * nz);
          }
        }
      }
    }
    if (c0 + STEP >= s1) break;  // uniform
    __syncthreads();
    shift_rows<256, STEP, 64>(B1, hist);
    shift_rows<256, STEP, 64>(B2, hist);
    __syncthreads();
  }
  if (DOT) group_add<256>(d, dots);
}

// The z pass for lines of at most kShallow positions.  Taps past the line meet zeros and change
// nothing but the sign of a sum that rounded to -0: one of them stands for all.
template <bool DOT, typename TS>
__global__ __launch_bounds__(NT) void k_gauss_shallow(const float2* __restrict__ src,
                                                      TS* __restrict__ dog,
                                                      const float* __restrict__ a,
                                                      double* __restrict__ dots,
                                                      const float* __restrict__ w1,
                                                      const float* __restrict__ w2, int r1, int r2,
                                                      float nz, int W, int L, i64 sa, i64 so,
                                                      unsigned nxb, unsigned no) {
  const LineAt la = line_at_block(nxb, no, L, L);
  double sum[2] = {0.0, 0.0};
  if (la.x < W) {
    const i64 base = (i64)la.other * so + la.x;
    float2 v[kShallow];
#pragma unroll
    for (int i = 0; i < kShallow; ++i)
      if (i < L) v[i] = src[base + i * sa];  // uniform, as all that follow
#pragma unroll
    for (int c = 0; c < kShallow; ++c) {
      if (c >= L) break;
      float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
      for (int i = 0; i < kShallow; ++i) {
        if (i < L && i - c <= r1 && c - i <= r1) s1 = fmaf(w1[r1 + c - i], v[i].x, s1);
        if (i < L && i - c <= r2 && c - i <= r2) s2 = fmaf(w2[r2 + c - i], v[i].y, s2);
      }
      if (c + r1 >= L) s1 = fmaf(w1[r1 + c - L], 0.0f, s1);
      if (c + r2 >= L) s2 = fmaf(w2[r2 + c - L], 0.0f, s2);
      const i64 idx = base + c * sa;
      if (DOT) {
        const double u = a[idx];
        sum[0] += u * s1;
        sum[1] += u * s2;
      } else {
        dog[idx] = cvt<TS>((s1 - s2) * nz);
      }
    }
  }
  if (DOT) group_add<NT>(sum, dots);
}

// ------------------------------------------------------------- compile-time radii
// z pass as a column walker: one thread per line, a register ring of the last 2R+1
// (G1, G2) pairs (zero outside the line), unrolled by the ring period so every index is
// static; every input is read once and no LDS is used.  Ring refills are loaded PF steps
// before they enter the ring (PF divides the ring period: static queue slots), and the
// walk ends at the line's end so no merged control path makes the compiler wait for the
// whole queue.  DOT: the outputs meet the volume `a` in FP64 sums instead of leaving (as a
// pair volume and a pass of its own over it: 97 + 85 us at 128 x 512 x 512, here 87).
template <int R1, int R2, bool DOT, typename TS>
__global__ __launch_bounds__(NT) void k_gauss_walk(const float2* __restrict__ src,
                                                   TS* __restrict__ dog,
                                                   const float* __restrict__ a,
                                                   double* __restrict__ dots,
                                                   const float* __restrict__ w1,
                                                   const float* __restrict__ w2, float nz, int W,
                                                   int L, i64 sa, i64 so, unsigned nxb,
                                                   unsigned no, int len) {
  constexpr int R = R1 > R2 ? R1 : R2;
  constexpr int WB = 2 * R + 1;
  constexpr int PF = WB % 3 == 0 ? 3 : WB % 5 == 0 ? 5 : WB % 7 == 0 ? 7 : 1;
  const LineAt la = line_at_block(nxb, no, len, L);
  const int x = la.x, b0 = la.c0, b1 = la.c1;
  double d[2] = {0.0, 0.0};
  auto walk = [&] {
    const i64 base = (i64)la.other * so + x;
    // zero padding in the load itself: position p is read through a buffer descriptor of
    // the wave's 64 columns at p (a uniform base), whose record count is 0 outside the
    // line, so those loads return zeros and no value is tested (or waited for) when it
    // enters the ring
    const int lane = (int)(threadIdx.x & 63);
    const int xw = __builtin_amdgcn_readfirstlane(x - lane);  // the wave's first column
    const i64 bw = (i64)la.other * so + xw;
    const int nrec = min(64, W - xw) * (int)sizeof(float2);
    auto load = [&](const float2* line, bool in) -> float2 {
      const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float2*>(line), 0, in ? nrec : 0, kBufferWord3);
      return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(
                                            r, lane * (int)sizeof(float2), 0, 0));
    };
    float2 ring[WB];  // position p lives in ring[(p - b0 + R) % WB]
#pragma unroll
    for (int q = 0; q < WB; ++q) {
      const int p = b0 - R + q;
      ring[q] = load(src + bw + (i64)p * sa, (unsigned)p < (unsigned)L);
    }
    // the refills are read front to back: a pointer and the positions left on the line
    const float2* line = src + bw + (i64)(b0 + R + 1) * sa;
    const float* aline = a + bw + (i64)b0 * sa;
    int left = L - (b0 + R + 1), aleft = L - b0;
    auto refill = [&]() -> float2 {
      const float2 v = load(line, left > 0);
      line += sa;
      --left;
      return v;
    };
    auto next_a = [&]() -> float {
      const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float*>(aline), 0, aleft > 0 ? nrec / 2 : 0, kBufferWord3);
      aline += sa;
      --aleft;
      return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, lane * 4, 0, 0));
    };
    // what step c needs (position c + R + 1, and a at c) waits in slot (c - b0) % PF
    float2 pf[PF];
    float pa[PF];
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      pf[j] = refill();
      if (DOT) pa[j] = next_a();
    }
    i64 idx = base + (i64)b0 * sa;
    for (int n = b1 - b0;; n -= WB) {  // outputs left
#pragma unroll
      for (int q = 0; q < WB; ++q) {
        if (q >= n) return;
        float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int j = -R1; j <= R1; ++j) s1 = fmaf(w1[R1 - j], ring[(q + j + R) % WB].x, s1);
#pragma unroll
        for (int j = -R2; j <= R2; ++j) s2 = fmaf(w2[R2 - j], ring[(q + j + R) % WB].y, s2);
        if (DOT) {
          const double v = pa[q % PF];
          d[0] += v * s1;
          d[1] += v * s2;
          pa[q % PF] = next_a();
        } else {
          dog[idx] = cvt<TS>((s1 - s2) * nz);
          idx += sa;
        }
        ring[q] = pf[q % PF];  // position c + R + 1 replaces position c - R
        pf[q % PF] = refill();
      }
    }
  };
  if (x < W) walk();
  if (DOT) group_add<NT>(d, dots);
}

// x and y passes fused: a one-wave work-group walks the rows of one plane for a strip of
// 64 columns.  Each row's window x0-16 .. x0+79 goes through an LDS line (two lines,
// alternating; the wave's own LDS order needs no barrier); lane l forms the x outputs
// (G1_x, G2_x) of column x0+l, which enter the register ring of the last 2R+1 rows
// exactly as in the column walker, and the y outputs leave as float2.  The (G1_x, G2_x)
// volume of the unfused passes is never stored.  Rows are fetched PF rows ahead of their
// use.  The Gaussian weights are symmetric (set pairwise from one value,
// w[r - i] == w[r + i]), so tap j reads w[r + |j|]: r + 1 distinct values per Gaussian,
// held in registers for the whole walk.
// AXES: weights of their own along y (wy1, wy2), else those along x.
template <int R1, int R2, bool AXES, typename TS>
__global__ __launch_bounds__(64) void k_gauss_xy_walk(const TS* __restrict__ src,
                                                      float2* __restrict__ dst,
                                                      const float* __restrict__ w1,
                                                      const float* __restrict__ w2,
                                                      const float* __restrict__ wy1,
                                                      const float* __restrict__ wy2, int W, int H,
                                                      int nxs, int nys, int rows) {
  constexpr int R = R1 > R2 ? R1 : R2;
  constexpr int WB = 2 * R + 1;
  // rows fetched ahead: a divisor of WB, so the queue slot of every row is static in
  // the loop unrolled by WB
  constexpr int PF = WB % 3 == 0 ? 3 : WB % 5 == 0 ? 5 : WB <= 13 ? WB : 1;
  constexpr int HX = 16, LW = 128;  // line positions 96 .. 127 stay unused (zero)
  static_assert(R <= HX, "x window exceeds the LDS line");
  __shared__ float line[2][LW];
  // work-group = one 64-column strip of one plane over the rows [y0, y1) of one of the nys
  // segments of the plane (rows: a multiple of WB)
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int y0 = (int)(t % nys) * rows, y1 = min(H, y0 + rows);
  const unsigned tile = t / nys;
  const int l = threadIdx.x;
  const int x0 = (int)(tile % nxs) * 64;
  const i64 pbase = (i64)(tile / nxs) * H * W;
  const int xa = x0 - HX + l, xb = x0 + 64 - HX + l;  // line positions l and 64 + l
  const bool va = xa >= 0 && xa < W, vb = l < 2 * HX && xb < W;
  const int xac = min(max(xa, 0), W - 1), xbc = min(xb, W - 1);
  // branch-free: every lane loads an in-bounds element (row and column clamped); zero is
  // selected outside the plane when the row is consumed, so no load sits under an exec
  // mask and none is waited for before its use
  float qa[PF], qb[PF];  // row y is held in slot y % PF
  auto fetch = [&](int y, int k) {
    const i64 rb = pbase + (i64)min(y, H - 1) * W;
    qa[k] = ld(src, rb + xac);
    qb[k] = ld(src, rb + xbc);
  };
  // the distinct weights in vector registers for the whole walk: in scalar registers the
  // unrolled walk ran out of them and reloaded the weights row after row, and every such
  // scalar load shares its wait counter with the LDS reads
  float v1[R1 + 1], v2[R2 + 1];
#pragma unroll
  for (int i = 0; i <= R1; ++i) {
    v1[i] = w1[R1 + i];
    asm volatile("" : "+v"(v1[i]));
  }
#pragma unroll
  for (int i = 0; i <= R2; ++i) {
    v2[i] = w2[R2 + i];
    asm volatile("" : "+v"(v2[i]));
  }
  float u1[R1 + 1], u2[R2 + 1];  // along y
#pragma unroll
  for (int i = 0; i <= R1; ++i) {
    u1[i] = AXES ? wy1[R1 + i] : v1[i];
    if (AXES) asm volatile("" : "+v"(u1[i]));
  }
#pragma unroll
  for (int i = 0; i <= R2; ++i) {
    u2[i] = AXES ? wy2[R2 + i] : v2[i];
    if (AXES) asm volatile("" : "+v"(u2[i]));
  }
  // row y waits in queue slot y % PF (y0 is a multiple of WB, so of PF): every slot index
  // below is a compile-time constant
  if (y0 == 0) {
#pragma unroll
    for (int k = 0; k < PF; ++k) fetch(k, k);
  } else {
#pragma unroll
    for (int k = 0; k < PF; ++k) fetch(y0 - R + k, ((k - R) % PF + PF) % PF);
  }
  // x outputs of row y, whose slot is k; fetches row y + PF into the freed slot.  Past
  // the plane the line holds zeros, so the outputs are +0 as the y pass's zero padding
  // requires.
  auto xrow = [&](int y, int k) -> float2 {
    const float a = (va && y < H) ? qa[k] : 0.0f, b = (vb && y < H) ? qb[k] : 0.0f;
    fetch(y + PF, k);
    float* ln = line[y & 1];
    ln[l] = a;
    ln[64 + l] = b;
    wave_lds_sync();
    const float* t = ln + l + HX;
    float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int j = -R1; j <= R1; ++j) s1 = fmaf(v1[j < 0 ? -j : j], t[j], s1);
#pragma unroll
    for (int j = -R2; j <= R2; ++j) s2 = fmaf(v2[j < 0 ? -j : j], t[j], s2);
    // pin the row's outputs here: otherwise the compiler sinks the FMA chains towards
    // their uses and keeps many rows' LDS windows live at once
    asm volatile("" : "+v"(s1), "+v"(s2));
    return make_float2(s1, s2);
  };
  const bool out = x0 + l < W;
  float2* dcol = dst + pbase + x0 + l;
  float2 ring[WB];  // row p lives in ring[(p + R) % WB]; rows < 0 are zero
  if (y0 == 0) {
#pragma unroll
    for (int q = 0; q < R; ++q) ring[q] = make_float2(0.0f, 0.0f);
#pragma unroll
    for (int q = R; q < WB; ++q) ring[q] = xrow(q - R, (q - R) % PF);
  } else {  // a later segment starts from the R rows above it
#pragma unroll
    for (int q = 0; q < WB; ++q) ring[q] = xrow(y0 - R + q, ((q - R) % PF + PF) % PF);
  }
  // The segment's end leaves the kernel (a wave-uniform return) instead of skipping the
  // remaining unrolled rows: no path that skips a row's loads merges back into the loop,
  // so the compiler's memory-wait counts keep the PF rows in flight.
  for (int c0 = y0;; c0 += WB) {
#pragma unroll
    for (int q = 0; q < WB; ++q) {
      const int c = c0 + q;
      if (c >= y1) return;
      float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
      for (int j = -R1; j <= R1; ++j) s1 = fmaf(u1[j < 0 ? -j : j], ring[(q + j + R) % WB].x, s1);
#pragma unroll
      for (int j = -R2; j <= R2; ++j) s2 = fmaf(u2[j < 0 ? -j : j], ring[(q + j + R) % WB].y, s2);
      if (out) st_nt(dcol + (i64)c * W, make_float2(s1, s2));
      ring[q] = xrow(c + R + 1, (q + R + 1) % PF);  // row c + R + 1 replaces row c - R
    }
  }
}

// (r1, r2) pairs with compile-time kernels: truncation 4 and 2 of the benchmark sigmas
// (2.0 / 3.2, 1.6 / 2.56) and of the reference's example sigmas (4.0 / 6.0, 1.8 / 2.7).
#define HDOG_GAUSS_PAIRS(X) X(8, 13) X(6, 10) X(4, 6) X(3, 5) X(8, 12) X(4, 5) X(7, 11)

bool has_pair(int r1, int r2) {
#define X(A, B) if (r1 == A && r2 == B) return true;
  HDOG_GAUSS_PAIRS(X)
#undef X
  return false;
}

// Waves per work-group of the walker for any radii: four where their LDS stays within the
// 64 KB of a launch and the weights fit the lanes (radii up to 28), else two.
size_t xy_run_lds(int RX, int RY, int nw) {
  return ((size_t)nw * GK * ((64 + 2 * RX + 7) / 8 * 8 + 1) + 2 * (size_t)(2 * RY + GK * nw) * 65) * 4;
}
int xy_run_waves(int RX, int RY) {
  return xy_run_lds(RX, RY, 4) <= 64 * 1024 && std::max(RX, RY) <= kLaneRadius ? 4 : 2;
}

WalkShape xy_run_shape(int RX, int RY, int W, int D) {
  return {(i64)((W + 63) / 64) * D * xy_run_waves(RX, RY), GK * 4, 2 * RY};
}

// x and y passes of any radii, each axis with its own
template <typename TS>
hipError_t gauss_xy_run(const TS* src, float2* dst, const float* wx1, const float* wx2,
                        const float* wy1, const float* wy2, int rx1, int rx2, int ry1, int ry2,
                        int W, int H, int D, hipStream_t s, int segments) {
  // taps past a plane of few rows meet zeros: one of them stands for all (k_gauss_shallow)
  wy1 += ry1 - std::min(ry1, H);
  wy2 += ry2 - std::min(ry2, H);
  ry1 = std::min(ry1, H);
  ry2 = std::min(ry2, H);
  const int RX = std::max(rx1, rx2), RY = std::max(ry1, ry2);
  const int nxs = (W + 63) / 64;
  const int nw = xy_run_waves(RX, RY);
  int nys, rows;
  walk_segments(H, xy_run_shape(RX, RY, W, D), &nys, &rows, segments);
  const dim3 grid((unsigned)((i64)nxs * D * nys));
  const size_t lds = xy_run_lds(RX, RY, nw);
  if (nw == 4)
    hipLaunchKernelGGL((k_gauss_xy_run<TS, 2, 4>), grid, dim3(256), lds, s, src, dst, wx1, wx2, wy1,
                       wy2, rx1, rx2, ry1, ry2, W, H, nxs, nys, rows);
  else
    hipLaunchKernelGGL((k_gauss_xy_run<TS, 3, 2>), grid, dim3(128), lds, s, src, dst, wx1, wx2, wy1,
                       wy2, rx1, rx2, ry1, ry2, W, H, nxs, nys, rows);
  return hipGetLastError();
}

// The compile-time walkers take a wave per strip of 64 columns.  On the smallest stacks, where
// a wave would walk hardly more rows than its window, the walk of any radii with four waves on
// a strip is the faster one (radii 8 / 13, rows of all strips: its us / the walker's):
// 24 x 96 x 112, 4608: 13 / 20; 40 x 160 x 160, 19200: 18 / 23; 48 x 192 x 192, 27648: 22 / 24;
// 20 x 256 x 400, 35840: 26 / 25; 64 x 200 x 200, 51200: 35 / 27.  Windows of radius 6 and less
// gain nothing (radii 4 / 6 at 40 x 160 x 160: 13 / 12).
bool gauss_row_walker(int r1, int r2, int W, int H, int D) {
  return has_pair(r1, r2) &&
         (std::max(r1, r2) < 8 || (i64)((W + 63) / 64) * D * H > 28 * 1024);
}

// Fused x + y passes of radii r1, r2 on both axes; AXES: with their own weights along y
template <bool AXES, typename TS>
hipError_t gauss_xy(const TS* src, float2* dst, const float* w1, const float* w2, const float* wy1,
                    const float* wy2, int r1, int r2, int W, int H, int D, hipStream_t s,
                    int segments) {
  if (!gauss_row_walker(r1, r2, W, H, D))
    return gauss_xy_run<TS>(src, dst, w1, w2, wy1, wy2, r1, r2, r1, r2, W, H, D, s, segments);
#define X(A, B)                                                                              \
  if (r1 == A && r2 == B) {                                                                  \
    const int nxs = (W + 63) / 64;                                                           \
    int nys, rows;                                                                           \
    walk_segments(H, gauss_walk_shape(A, B, W, H, D), &nys, &rows, segments);                   \
    const i64 nblk = (i64)nxs * D * nys;                                                     \
    hipLaunchKernelGGL((k_gauss_xy_walk<A, B, AXES, TS>), dim3((unsigned)nblk), dim3(64), 0, \
                       s, src, dst, w1, w2, wy1, wy2, W, H, nxs, nys, rows);                 \
    return hipGetLastError();                                                                \
  }
  HDOG_GAUSS_PAIRS(X)
#undef X
  return hipErrorInvalidValue;
}

// z pass: the difference (dog), or with DOT the sums of both with a.  (The difference leaves by
// plain stores: streaming ones are slower where the planes do not start on whole lines, 217 us
// for 93 x 777 x 1001 and 166 plain, and no faster where they do: 195 and 194 for
// 64 x 1080 x 1280.)
template <bool DOT, typename TS>
hipError_t gauss_z(const float2* src, TS* dog, const float* a, double* dots, const float* w1,
                   const float* w2, int r1, int r2, float nz, int W, int H, int D, hipStream_t s) {
  const i64 WH = (i64)W * H;
  const ZColumns z = z_columns(W, H);
  const int n = z.n, m = z.rows;
#define X(A, B)                                                                              \
  if (r1 == A && r2 == B) {                                                                  \
    const LineGrid g = line_grid(n, D, m, 2 * (A > B ? A : B));                              \
    hipLaunchKernelGGL((k_gauss_walk<A, B, DOT, TS>), dim3(g.blocks), dim3(NT), 0, s, src,   \
                       dog, a, dots, w1, w2, nz, n, D, WH, (i64)W, g.nxb, g.no, g.len);      \
    return hipGetLastError();                                                                \
  }
  HDOG_GAUSS_PAIRS(X)
#undef X
  if (D <= kShallow) {
    const unsigned nxs = (unsigned)((n + NT - 1) / NT);
    hipLaunchKernelGGL((k_gauss_shallow<DOT, TS>), dim3((unsigned)((i64)nxs * m)), dim3(NT), 0, s,
                       src, dog, a, dots, w1, w2, r1, r2, nz, n, D, WH, (i64)W, nxs, (unsigned)m);
    return hipGetLastError();
  }
  const int R = std::max(r1, r2);
  const i64 nxb = (n + 63) / 64;
  int nseg, len;
  line_segments(D, nxb * m * 4, 1024.0, 2.0, false, 2 * R, &nseg, &len);
  const dim3 grid((unsigned)(nxb * m * nseg));
  const size_t lds = 2 * (size_t)(2 * R + 4 * GK) * 64 * 4;
  if (R <= kLaneRadius)
    hipLaunchKernelGGL((k_gauss_line_run<DOT, false, TS>), grid, dim3(256), lds, s, src, dog, a,
                       dots, w1, w2, r1, r2, nz, n, D, WH, (i64)W, (unsigned)nxb, (unsigned)m, len);
  else
    hipLaunchKernelGGL((k_gauss_line_run<DOT, true, TS>), grid, dim3(256), lds, s, src, dog, a,
                       dots, w1, w2, r1, r2, nz, n, D, WH, (i64)W, (unsigned)nxb, (unsigned)m, len);
  return hipGetLastError();
}

}  // namespace

WalkShape gauss_walk_shape(int r1, int r2, int W, int H, int D) {
  const int R = std::max(r1, r2);
  if (!gauss_row_walker(r1, r2, W, H, D)) return xy_run_shape(R, std::min(R, H), W, D);
  return {(i64)((W + 63) / 64) * D, 2 * R + 1, 2 * R};
}

template <typename TN, typename TD>
hipError_t launch_dog(const TN* norm, TD* dog, void* tmp1, const float* weights,
                      const int r[4], float normalizer, int W, int H, int D, hipStream_t s,
                      int segments) {
  const float* wxy1 = weights;
  const float* wz1 = weights + kMaxTaps;
  const float* wxy2 = weights + 2 * kMaxTaps;
  const float* wz2 = weights + 3 * kMaxTaps;
  hipError_t e = gauss_xy<false, TN>(norm, (float2*)tmp1, wxy1, wxy2, wxy1, wxy2, r[0], r[2], W, H,
                                     D, s, segments);
  if (e != hipSuccess) return e;
  mark("dog/gauss_xy", s);
  e = gauss_z<false, TD>((const float2*)tmp1, dog, nullptr, nullptr, wz1, wz2, r[1], r[3],
                         normalizer, W, H, D, s);
  mark("dog/gauss_z_dog", s);
  return e;
}

// The differentiable form's pair: weights of their own per axis (anisotropic sigmas and their
// derivatives).  x and y fused as in the detector (in two passes over the pair volume: 118 +
// 140 us at radii 8 / 13 and 128 x 512 x 512, here 148).
static hipError_t gauss_xy_axes(const float* src, void* tmp1, const float* const w[6],
                                const int r[6], int W, int H, int D, hipStream_t s) {
  if (r[0] == r[1] && r[3] == r[4])
    return gauss_xy<true, float>(src, (float2*)tmp1, w[0], w[3], w[1], w[4], r[0], r[3], W, H, D, s,
                                 0);
  return gauss_xy_run<float>(src, (float2*)tmp1, w[0], w[3], w[1], w[4], r[0], r[3], r[1], r[4], W,
                             H, D, s, 0);
}

hipError_t launch_gauss_dog(const float* src, void* tmp1, const float* const w[6], const int r[6],
                            float nz, float* dog, int W, int H, int D, hipStream_t s) {
  const hipError_t e = gauss_xy_axes(src, tmp1, w, r, W, H, D, s);
  if (e != hipSuccess) return e;
  return gauss_z<false, float>((const float2*)tmp1, dog, nullptr, nullptr, w[2], w[5], r[2], r[5],
                               nz, W, H, D, s);
}

hipError_t launch_gauss_dots(const float* src, void* tmp1, const float* const w[6], const int r[6],
                             const float* a, double* out, int W, int H, int D, hipStream_t s) {
  const hipError_t e = gauss_xy_axes(src, tmp1, w, r, W, H, D, s);
  if (e != hipSuccess) return e;
  return gauss_z<true, float>((const float2*)tmp1, nullptr, a, out, w[2], w[5], r[2], r[5], 0.0f, W,
                              H, D, s);
}

#define HDOG_INST_DOG(TN, TD)                                                                \
  template hipError_t launch_dog<TN, TD>(const TN*, TD*, void*, const float*, const int*, float, \
                                         int, int, int, hipStream_t, int);
HDOG_INST_DOG(float, float)
HDOG_INST_DOG(__half, __half)
HDOG_INST_DOG(__hip_bfloat16, __hip_bfloat16)
HDOG_INST_DOG(__half, float)
HDOG_INST_DOG(__hip_bfloat16, float)
#undef HDOG_INST_DOG

}  // namespace hdog
