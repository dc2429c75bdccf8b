// soft.hip -- kernels of the differentiable blob response (no counterpart in the
// reference, which only thresholds the Hessian).
//
//   dog  = s * (G_s1 v - G_s2 v),  s = (sx1 * sy1 * sz1)^gamma, anisotropic sigmas, fixed radii
//   H    = Hessian of dog (the same zero-padded central differences as the detector)
//   M    = candidate mask (all leading minors of H negative), held constant
//   u    = -det(H) / tau,  loss = mean over M of BCE(sigmoid(u), target)
//
// Backward pass (hand-written adjoints):
//   dL/du   = (sigmoid(u) - t) / |M|                    (pointwise, FP64)
//   dL/dH_k = dL/du * (-1/tau) * d det / d H_k           (cofactors)
//   dL/ddog = sum_k A_k^T dL/dH_k, with A_k the pair of first differences producing H_k; the
//             zero-padded central difference g satisfies g^T = -g, so A_k^T applies the same
//             two differences in reverse order:  g_x(P_x) + g_y(P_y) + g_z(P_z) with
//             P_x = g_x Gxx + g_y Gxy + g_z Gxz, P_y = g_y Gyy + g_z Gyz, P_z = g_z Gzz.
//   dL/dv   = s * (G_s1 - G_s2) dL/ddog (a symmetric zero-padded Gaussian is self-adjoint)
//   dL/dsigma: one separable pass with the weight derivative along one axis, dotted with
//             dL/ddog, plus the normalizer term (gamma / sigma_a1) <dL/ddog, dog>.
//
// Local-contrast normalization in front of the DoG (src/3D/NormalizeFilter.cu:53-654 on a
// float volume v): E = box(min3(v)), D = box(max3(v)) with clamp-to-edge windows of
// radius (rxy, rxy, rz) for both the min / max and the box, n = v >= m ? (v - E)/(D - E)
// : 0.  Its adjoint, given dL/dn:
//   dL/dv  = [v >= m] dL/dn / (D - E)                          (direct term)
//          + route(argmin, box^T(dL/dE)) + route(argmax, box^T(dL/dD))
//   dL/dE  = [v >= m] dL/dn (v - D) / (D - E)^2,  dL/dD = -[v >= m] dL/dn (v - E) / (D - E)^2
// box^T is the transpose of the clamped box mean (the clamped border positions collect
// the weight of every window tap that clamps onto them); the min filter is taken by its
// subgradient: each output's gradient goes to the voxel that attains the window minimum
// (the lowest linear index among equal minima), likewise for the max.  The argmin / argmax
// of the 3-D window are found by separable passes over (value, index) pairs, which is exact
// because the order "smaller value, then smaller index" is total.
#include "run8.hpp"

namespace hdog {
namespace {

constexpr int NT = 256;

__device__ __forceinline__ double det3(double xx, double xy, double xz, double yy, double yz,
                                       double zz) {
  return xx * yy * zz + 2 * xy * yz * xz - xx * yz * yz - yy * xz * xz - zz * xy * xy;
}

__device__ __forceinline__ double softplus(double u) {
  return u > 0 ? u + log1p(exp(-u)) : log1p(exp(u));
}

// The records of the masked voxels (launch_hessian_records): per Hessian tile a count and
// the voxels' positions and six elements, so the FP64 work below runs on full waves and
// touches nothing else.  A pass over the dense volumes and mask instead spent 282 us on the
// loss and 326 on the gradient at 128 x 512 x 512 with 7 % masked (now 34 and 34).
struct TileOf {
  int x0, y0, z0;
};
__device__ __forceinline__ TileOf tile_of(unsigned tile, unsigned nbx, unsigned nby) {
  const unsigned r = tile / nbx;
  return {(int)(tile - r * nbx) * kHessTX, (int)(r % nby) * kHessTY, (int)(r / nby) * kHessTZ};
}

// sums[0] += sum over M of softplus(u) - t*u ; sums[1] += |M|
__global__ __launch_bounds__(NT) void k_soft_loss(const float* __restrict__ cand,
                                                  const uint32_t* __restrict__ cand_cnt,
                                                  const uint8_t* __restrict__ target,
                                                  unsigned ntiles, unsigned nbx, unsigned nby,
                                                  int W, int H, int D, double inv_tau,
                                                  double* sums) {
  double ls = 0.0, cnt = 0.0;
  for (unsigned tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const uint32_t n = cand_cnt[tile];
    const TileOf T = tile_of(tile, nbx, nby);
    const RecBlock b = rec_block(T.x0, T.y0, T.z0, W, H, D);
    const float* rec = cand + b.first * 7;
    const float* el = rec + b.slots;
    for (uint32_t i = threadIdx.x; i < n; i += NT) {
      const uint32_t v = __float_as_uint(rec[i]);
      const size_t at = ((size_t)(T.z0 + (int)(v / (kHessTX * kHessTY))) * H +
                         (T.y0 + (int)(v / kHessTX % kHessTY))) * W + T.x0 + (int)(v % kHessTX);
      float e[6];
      rec_elements(el, i, e);
      const double u = -det3(e[0], e[1], e[2], e[3], e[4], e[5]) * inv_tau;
      ls += softplus(u) - (target[at] ? u : 0.0);
      cnt += 1.0;
    }
  }
  double a[2] = {ls, cnt};
  group_add<NT>(a, sums);
}

// the records' elements are overwritten by dL/dH; sums[0] += dL/dtau contributions
__global__ __launch_bounds__(NT) void k_soft_grad_h(float* __restrict__ cand,
                                                    const uint32_t* __restrict__ cand_cnt,
                                                    const uint8_t* __restrict__ target,
                                                    unsigned ntiles, unsigned nbx, unsigned nby,
                                                    int W, int H, int D, double inv_tau,
                                                    double inv_count, double* sums) {
  double gt = 0.0;
  for (unsigned tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const uint32_t n = cand_cnt[tile];
    const TileOf T = tile_of(tile, nbx, nby);
    const RecBlock b = rec_block(T.x0, T.y0, T.z0, W, H, D);
    float* rec = cand + b.first * 7;
    float* el = rec + b.slots;
    for (uint32_t i = threadIdx.x; i < n; i += NT) {
      const uint32_t v = __float_as_uint(rec[i]);
      const size_t at = ((size_t)(T.z0 + (int)(v / (kHessTX * kHessTY))) * H +
                         (T.y0 + (int)(v / kHessTX % kHessTY))) * W + T.x0 + (int)(v % kHessTX);
      float h[6];
      rec_elements(el, i, h);
      const double xx = h[0], xy = h[1], xz = h[2], yy = h[3], yz = h[4], zz = h[5];
      const double d = det3(xx, xy, xz, yy, yz, zz);
      const double u = -d * inv_tau;
      const double p = 1.0 / (1.0 + exp(-u));
      const double gu = (p - (target[at] ? 1.0 : 0.0)) * inv_count;  // dL/du
      gt += gu * d * inv_tau * inv_tau;                               // du/dtau = det / tau^2
      const double gd = -gu * inv_tau;                                // dL/ddet
      rec_store(el, i, 0, {(float)(gd * 2.0 * (xz * yz - zz * xy)), (float)(gd * (xx * zz - xz * xz)),
                           (float)(gd * 2.0 * (xy * xz - xx * yz))});
      rec_store(el, i, 1, {(float)(gd * (yy * zz - yz * yz)),
                           (float)(gd * 2.0 * (xy * yz - yy * xz)), (float)(gd * (xx * yy - xy * xy))});
    }
  }
  double a[1] = {gt};
  group_add<NT>(a, sums);
}

// dL/ddog from the records of dL/dH, and *dot += <dL/ddog, dog>:
//   P_x = g_x Gxx + g_y Gxy + g_z Gxz, P_y = g_y Gyy + g_z Gyz, P_z = g_z Gzz,
//   dL/ddog = g_x P_x + g_y P_y + g_z P_z,
// g the zero-padded central difference, P zero outside the volume.  A wave owns kAdjX columns
// of AR rows and marches over the slices of a segment: its lanes hold the columns and two more
// on either side, so the differences along x are lane shifts, those along y differences of its
// own registers, and those along z of the ones it kept.  A row of a slice is laid out straight
// from the records: its bits (from the two tiles that the 64 lanes touch) say which lanes hold
// one and which one; a lane without one reads past the end of the buffer, which gives 0 without
// touching memory.  Nothing dense but the result leaves the chip.  Bound by instruction issue
// (seven row lookups and ten loads for three output rows).  As dense volumes dL/dH went out and back
// in two passes: 262 + 132 us at 128 x 512 x 512 with 7 % masked, and 76 for the dot product
// (154 here; with tiles of 64 x 8 x 8 in LDS, one element at a time, 820).
// Rows of outputs of a wave: with more the registers leave fewer waves, with fewer more rows
// are laid out twice (us at 128 x 512 x 512, each row's block looked up for itself: 2: 199, 3: 172,
// 4: 221, 6: 215, 8: 290; looked up once per slice and side, 3: 154).
constexpr int AR = 3;
constexpr int kAdjX = 60;   // columns of outputs: lanes 2 .. 61
constexpr int AI = AR + 4;  // rows of inputs, two beyond either side
typedef float F3 __attribute__((ext_vector_type(3)));
__device__ __forceinline__ float lane_up(float v) {  // the value of lane - 1
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_down(float v) {  // the value of lane + 1
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, false));
}
__device__ __forceinline__ uint32_t read_lane(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__global__ __launch_bounds__(NT, 4) void k_hessian_adjoint(const float* __restrict__ cand,
                                                           const TileRow* __restrict__ rows,
                                                           const float* __restrict__ dog,
                                                           float* __restrict__ out, int nsx,
                                                           int nsy, int nbx, int len, int W, int H,
                                                           int D, double* dot) {
  const int lane = (int)(threadIdx.x & 63);
  const int strip = __builtin_amdgcn_readfirstlane(
      (int)blockIdx.x * (NT / 64) + (int)(threadIdx.x >> 6));  // x fastest, then y, then z
  const int c0 = strip % nsx * kAdjX - 2, y0 = strip / nsx % nsy * AR,
            z0 = strip / nsx / nsy * len, z1 = min(z0 + len, D);
  double acc = 0.0;
  if (z0 < D) {
    const int col = c0 + lane;
    const bool colin = col >= 0 && col < W, writes = colin && lane >= 2 && lane < 2 + kAdjX;
    // the tile of column c0 covers the lanes below `split`, the next one the others
    const int tl = (c0 + 64) / 64 - 1, sh = (c0 + 64) % 64, split = 64 - sh;
    const bool right = lane >= split;
    // lane j < AI looks up row y0 - 2 + j, of the left tile, lane AI + j of the right one
    const int lt = lane >= AI ? tl + 1 : tl, ly = y0 - 2 + (lane >= AI ? lane - AI : lane);
    const bool look = lane < 2 * AI && lt >= 0 && lt < nbx && ly >= 0 && ly < H;
    const i64 rowbase = look ? (i64)ly * nbx + lt : 0;
    auto find = [&](int z) -> TileRow {
      TileRow r = {0ull, 0ull};
      if (look && z >= 0 && z < D) r = rows[rowbase + (i64)z * H * nbx];
      return r;
    };
    // bytes from the left tile's block to the elements of the lane's tile, per slice of theirs
    const int exl = min(kHessTX, W - tl * kHessTX), exr = min(kHessTX, W - (tl + 1) * kHessTX);
    const uint32_t head =
        look ? (uint32_t)((lane < AI ? exl * 4 : exl * 28 + exr * 4) *
                          min(kHessTY, H - ly / kHessTY * kHessTY)) : 0u;
    // the rows lie in KT tile rows at most, the first from row yu on; where the left block of
    // each starts in its layer of tiles, per slice of theirs
    constexpr int KT = (AI + kHessTY - 2) / kHessTY + 1;
    const int yu = max(y0 - 2, 0) / kHessTY * kHessTY;
    i64 start[KT];
#pragma unroll
    for (int k = 0; k < KT; ++k) {
      const int yk = yu + k * kHessTY;
      start[k] = (i64)yk * W + (i64)min(kHessTY, H - yk) * (tl * kHessTX);
    }
    auto half = [](float hi, float lo) { return (hi - lo) * 0.5f; };
    // [z & 1]: the values of two slices ago until this one's replace them
    float xz[2][AR] = {}, yz[2][AR + 2] = {}, zz[2][AR] = {}, pz[2][AR] = {};
    float ax[AR] = {}, ay[AR + 2] = {}, o[AR] = {};
    TileRow next = find(z0 - 2);
    auto slice = [&](int z, auto par) {
      constexpr int q = decltype(par)::value;
      const TileRow cur = next;
      next = find(z + 1);
      const int zo = z - 2;  // the slice that leaves
      const bool leaves = zo >= z0 && writes;
      const i64 at = ((i64)zo * H + y0) * W + col;
      float gxx[AR] = {}, gxy[AR + 2] = {}, gyy[AI] = {}, nxz[AR] = {}, nyz[AR + 2] = {}, nzz[AR] = {};
      // bits of the lanes' columns and, per side, the slot of the first record among them
      const unsigned long long own = lane < AI ? cur.bits >> sh : sh ? cur.bits << split : 0ull;
      const int zt = max(z, 0) / kHessTZ * kHessTZ, ez = min(kHessTZ, D - zt);
      const uint32_t first = ((uint32_t)cur.first +
          (lane < AI && sh ? (uint32_t)__popcll(cur.bits << split) : 0u)) * 24u +
          head * (uint32_t)ez;  // in bytes
      if (__ballot(own != 0ull)) {
        const uint32_t olo = (uint32_t)own, ohi = (uint32_t)(own >> 32);
        const float* layer = cand + (i64)zt * W * H * 7;
        const float* block[KT];
#pragma unroll
        for (int k = 0; k < KT; ++k) block[k] = layer + start[k] * ez * 7;
#pragma unroll
        for (int j = 0; j < AI; ++j) {
          const unsigned long long mlo = read_lane(olo, j), mhi = read_lane(ohi, j);
          const unsigned long long ml = mhi << 32 | mlo;
          const unsigned long long m = ml | (unsigned long long)read_lane(ohi, AI + j) << 32 |
                                       read_lane(olo, AI + j);
          const uint32_t fl = read_lane(first, j);
          const uint32_t fr = read_lane(first, AI + j) - (uint32_t)__popcll(ml) * 24u;
          // two tiles' records, never used beyond the last tile's (no bits there)
          const float* at_block = block[0];
#pragma unroll
          for (int k = 1; k < KT; ++k)
            if (y0 - 2 + j >= yu + k * kHessTY) at_block = block[k];  // uniform
          const __amdgpu_buffer_rsrc_t r = buf_rsrc(at_block, (uint32_t)kCandTile * 7u * 8u);
          const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
              (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
          const uint32_t slot = rank * 24u + (right ? fr : fl);  // in bytes
          const int off = (int)((m >> lane) & 1ull ? slot : 0xF0000000u);
          const F3 u = __builtin_bit_cast(
              F3, __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, 0));
          gyy[j] = u[kRecYY];
          if (j >= 1 && j <= AR + 2) {
            gxy[j - 1] = u[kRecXY];
            nyz[j - 1] = u[kRecYZ];
          }
          if (j >= 2 && j <= AR + 1) {
            const F3 v = __builtin_bit_cast(
                F3, __builtin_amdgcn_raw_buffer_load_b96(r, off + 12, 0, 0));
            gxx[j - 2] = v[kRecXX - 3];
            nxz[j - 2] = v[kRecXZ - 3];
            nzz[j - 2] = v[kRecZZ - 3];
          }
        }
      }
      // z - 2 leaves: g_z P_z
      const bool zin = z >= 1 && z <= D;  // slice z - 1
#pragma unroll
      for (int j = 0; j < AR; ++j) {
        const float p = zin ? half(nzz[j], zz[q][j]) : 0.0f;  // P_z(z - 1)
        const float v = o[j] + half(p, pz[1 - q][j]);  // P_z(z - 3)
        if (leaves && y0 + j < H) {
          out[at + (i64)j * W] = v;
          acc += (double)v * dog[at + (i64)j * W];
        }
        pz[1 - q][j] = p;
        zz[q][j] = nzz[j];
      }
      // z - 1 is completed but for P_z
#pragma unroll
      for (int j = 0; j < AR; ++j) {
        const float p = colin ? ax[j] + half(nxz[j], xz[q][j]) : 0.0f;
        o[j] = half(lane_down(p), lane_up(p));
        xz[q][j] = nxz[j];
      }
      float py[AR + 2];
#pragma unroll
      for (int j = 0; j < AR + 2; ++j) {
        const int y = y0 - 1 + j;
        py[j] = y >= 0 && y < H ? ay[j] + half(nyz[j], yz[q][j]) : 0.0f;
        yz[q][j] = nyz[j];
      }
#pragma unroll
      for (int j = 0; j < AR; ++j) o[j] += half(py[j + 2], py[j]);
      // z
#pragma unroll
      for (int j = 0; j < AR; ++j)
        ax[j] = half(lane_down(gxx[j]), lane_up(gxx[j])) + half(gxy[j + 2], gxy[j]);
#pragma unroll
      for (int j = 0; j < AR + 2; ++j) ay[j] = half(gyy[j + 2], gyy[j]);
    };
    for (int z = z0 - 2; z < z1 + 2; z += 2) {
      slice(z, std::integral_constant<int, 0>());
      if (z + 1 < z1 + 2) slice(z + 1, std::integral_constant<int, 1>());
    }
  }
  double a[1] = {acc};
  group_add<NT>(a, dot);
}

// Line kernels run one element per thread on a grid of nxb x-blocks per row (y + H z):
// x, y, z come from the thread and the block with 32-bit arithmetic, not from divisions
// of a 64-bit linear index.
struct Pos {
  int x, y, z;
  i64 i;  // linear index
};
__device__ __forceinline__ bool pos_of(int W, int H, unsigned nxb, Pos& p) {
  const unsigned row = blockIdx.x / nxb;
  p.x = (int)(blockIdx.x - row * nxb) * NT + (int)threadIdx.x;
  p.y = (int)(row % (unsigned)H);
  p.z = (int)(row / (unsigned)H);
  p.i = (i64)row * W + p.x;
  return p.x < W;
}
unsigned xblocks(int W) { return (unsigned)((W + NT - 1) / NT); }
unsigned grid_rows(int W, int H, int D) { return xblocks(W) * (unsigned)H * (unsigned)D; }

__global__ __launch_bounds__(NT) void k_pack_pair(const float* __restrict__ a,
                                                  const float* __restrict__ b,
                                                  float2* __restrict__ out, i64 N) {
  for (i64 i = (i64)blockIdx.x * NT + threadIdx.x; i < N; i += (i64)gridDim.x * NT)
    out[i] = make_float2(a[i], b[i]);
}

__global__ void k_zero_f64(double* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0.0;
}

unsigned grid_for(i64 N) { return (unsigned)std::min<i64>((N + NT - 1) / NT, 1 << 16); }
struct Line {  // the line through a voxel along one axis
  i64 base, stride;
  int c, L;
};
__device__ __forceinline__ Line line_at(const Pos& p, int axis, int W, int H, int D) {
  Line l;
  if (axis == 0) { l.c = p.x; l.L = W; l.stride = 1; }
  else if (axis == 1) { l.c = p.y; l.L = H; l.stride = W; }
  else { l.c = p.z; l.L = D; l.stride = (i64)W * H; }
  l.base = p.i - (i64)l.c * l.stride;
  return l;
}

// ---- radii up to kArgRadius: eight outputs at a time (run8.hpp) ------------------------
// Window extremes with their positions.  A value travels as a 32-bit key that orders as the
// floats do (-0 taken as +0, as == takes them), one for the minimum, kx = kn + 1 for the
// maximum: a NaN, which no window picks, is the largest kn and the smallest kx.  Windows are
// joined front to back and the earlier one wins a tie, so with x, then y, then z a window's
// extreme is the one of the lowest linear index.  Its position travels as its taps (0 .. 2r)
// along the axes so far, eight bits each.
struct Arg {
  uint32_t kn, kx, cn, cx;  // keys, taps
};
__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t b = __float_as_uint(v + 0.0f);
  const uint32_t k = b ^ ((uint32_t)((int)b >> 31) | 0x80000000u);
  return v != v ? 0xFFFFFFFFu : k;
}
__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float(k & 0x80000000u ? k ^ 0x80000000u : ~k);
}
__device__ __forceinline__ Arg arg_join(const Arg& a, const Arg& b) {  // b comes after a
  Arg o;
  o.cn = b.kn < a.kn ? b.cn : a.cn;
  o.kn = min(a.kn, b.kn);
  o.cx = b.kx > a.kx ? b.cx : a.cx;
  o.kx = max(a.kx, b.kx);
  return o;
}
// out[o] = extremes of inputs o .. o + 2r; next(i) gives input i, i = 0, 1, ... 2r + 7
template <int R, typename F>
__device__ __forceinline__ void arg8(F&& next, int r, Arg (&out)[OK]) {
  if constexpr (R > 0) {
    Arg v[2 * R + OK];
#pragma unroll
    for (int i = 0; i < 2 * R + OK; ++i) v[i] = next(i);
#pragma unroll
    for (int o = 0; o < OK; ++o) {
      out[o] = v[o];
#pragma unroll
      for (int i = 1; i <= 2 * R; ++i) out[o] = arg_join(out[o], v[o + i]);
    }
  } else {
    Arg h[OK - 1];
#pragma unroll
    for (int i = 0; i < OK - 1; ++i) h[i] = next(i);
    // inputs 7 .. 2r are in every window (an even number, 2r - 6), two always read ahead
    Arg mid = next(OK - 1), v = next(OK);
#pragma unroll 1
    for (int i = OK + 1; i < 2 * r; i += 2) {
      const Arg n0 = next(i), n1 = next(i + 1);
      mid = arg_join(arg_join(mid, v), n0);
      v = n1;
    }
    mid = arg_join(mid, v);
    Arg e[OK - 1];
#pragma unroll
    for (int q = 0; q < OK - 1; ++q) e[q] = next(2 * r + 1 + q);
    Arg t = mid;
    out[OK - 1] = mid;
#pragma unroll
    for (int o = OK - 2; o >= 0; --o) out[o] = t = arg_join(h[o], t);  // inputs o .. 2r
    t = e[0];
#pragma unroll
    for (int o = 1; o < OK; ++o) {
      if (o > 1) t = arg_join(t, e[o - 1]);
      out[o] = arg_join(out[o], t);
    }
  }
}

constexpr int kArgRadius = 23;  // the work-group's LDS below stays within 64 KB
constexpr int kStep = 4 * OK;   // positions per step of a work-group
constexpr int arg_line_pitch(int r) { return (64 + 2 * r + 7) / 8 * 8 + 1; }
constexpr size_t arg_xy_lds(int r) {
  return (size_t)4 * OK * arg_line_pitch(r) * 4 + (size_t)(2 * r + kStep) * (65 * 8 + 66 * 2);
}
static_assert(arg_xy_lds(kArgRadius) <= 64 * 1024, "LDS of a launch");  // the largest
constexpr size_t box_xy_lds(int r) {
  return ((size_t)4 * OK * arg_line_pitch(r) + 2 * (size_t)(2 * r + kStep) * 65) * 4;
}
struct XyRun {  // grid of a walk over the rows of 64-column strips
  int nxs, nys, rows;
  unsigned blocks;
};
XyRun xy_run(int W, int H, int D, int r) {
  XyRun x;
  x.nxs = (W + 63) / 64;
  walk_segments(H, WalkShape{(i64)x.nxs * D * 4, kStep, 2 * r}, &x.nys, &x.rows);
  x.blocks = (unsigned)((i64)x.nxs * D * x.nys);
  return x;
}

// First and second pass (x, y) of the window extremes: four waves walk the rows of one plane
// for a strip of 64 columns, eight rows per wave and step.
//   1. a wave's rows (clamped to the plane, loaded a step ahead) enter its LDS lines as keys;
//   2. lane (row l % 8, columns 8 (l / 8) ..) forms eight x windows -> three LDS planes of the
//      last 2r + 32 rows: both keys, and both taps;
//   3. lane l forms eight y windows of column x0 + l, which leave as keys and taps.
// 4 bytes in and 12 out per voxel and nothing between the passes: 153 us at 128 x 512 x 512,
// radius 10 (a kernel per axis, 16 bytes per voxel and side between them, a tap each along x
// and van Herk blocks along y: 383 + 281).
template <int R>
__global__ __launch_bounds__(256) void k_soft_arg_xy(const float* __restrict__ v,
                                                     uint32_t* __restrict__ pkn,
                                                     uint32_t* __restrict__ pkx,
                                                     uint32_t* __restrict__ ptap, int W, int H,
                                                     int r, int nxs, int nys, int rows) {
  extern __shared__ uint32_t sm_arg[];
  constexpr int BP = 65, TP = 66;
  const int hist = 2 * r, span = 64 + 2 * r, AP = arg_line_pitch(r);
  const int l = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  uint32_t* A = sm_arg + wave * (OK * AP);
  uint32_t* Bn = sm_arg + 4 * (OK * AP);
  uint32_t* Bx = Bn + (hist + kStep) * BP;
  uint16_t* Bt = reinterpret_cast<uint16_t*>(Bx + (hist + kStep) * BP);
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int y0 = (int)(t % (unsigned)nys) * rows, y1 = min(H, y0 + rows);
  const unsigned tile = t / (unsigned)nys;
  const int x0 = (int)(tile % (unsigned)nxs) * 64;
  const i64 pbase = (i64)(tile / (unsigned)nxs) * H * W;
  int xl[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) xl[j] = clampi(x0 - r + 64 * j + l, 0, W - 1);
  float q[OK][2];
  auto fetch = [&](int y) {
#pragma unroll
    for (int i = 0; i < OK; ++i) {
      const float* row = v + pbase + (i64)clampi(y + i, 0, H - 1) * W;
#pragma unroll
      for (int j = 0; j < 2; ++j) q[i][j] = row[xl[j]];
    }
  };
  const int xr = l % OK, xg = l / OK;
  auto xpass = [&](int row, int ahead) {
#pragma unroll
    for (int i = 0; i < OK; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (64 * j + l < span) A[i * AP + 64 * j + l] = order_key(q[i][j]);
    fetch(ahead);
    wave_lds_sync();
    const uint32_t* p = A + xr * AP + OK * xg;
    Arg o[OK];
    arg8<R>([&](int i) -> Arg {
      const uint32_t k = *p++;
      return {k, k + 1u, (uint32_t)i, (uint32_t)i};
    }, r, o);
    const int at = row + xr;
#pragma unroll
    for (int k = 0; k < OK; ++k) {
      Bn[at * BP + OK * xg + k] = o[k].kn;
      Bx[at * BP + OK * xg + k] = o[k].kx;
      Bt[at * TP + OK * xg + k] = (uint16_t)((o[k].cn - k) | (o[k].cx - k) << 8);
    }
    wave_lds_sync();
  };
  // the rows above the segment (the last eight may reach into the first step's rows, which
  // are written again after the barrier)
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
  for (int c0 = y0; c0 < y1; c0 += kStep) {
    xpass(hist + OK * wave, c0 + kStep + r + OK * wave);
    __syncthreads();
    const int c = c0 + OK * wave;
    if (c < y1) {
      const uint32_t* pn = Bn + OK * wave * BP + l;
      const uint32_t* px = Bx + OK * wave * BP + l;
      const uint16_t* pt = Bt + OK * wave * TP + l;
      Arg o[OK];
      arg8<R>([&](int i) -> Arg {
        const uint32_t tp = *pt;
        const Arg a = {*pn, *px, (tp & 0xFFu) | (uint32_t)i << 8, tp >> 8 | (uint32_t)i << 8};
        pn += BP;
        px += BP;
        pt += TP;
        return a;
      }, r, o);
      if (out) {
#pragma unroll
        for (int k = 0; k < OK; ++k)
          if (c + k < y1) {
            const i64 at = pbase + (i64)(c + k) * W + x0 + l;
            st_nt(pkn + at, o[k].kn);
            st_nt(pkx + at, o[k].kx);
            st_nt(ptap + at, (o[k].cn - (k << 8)) | (o[k].cx - (k << 8)) << 16);
          }
      }
    }
    if (c0 + kStep >= y1) break;  // uniform
    __syncthreads();
    shift_rows<256, kStep, BP>(Bn, hist);
    shift_rows<256, kStep, BP>(Bx, hist);
    shift_rows<256, kStep, TP>(Bt, hist);
    __syncthreads();
  }
}

// Third pass (z): the extremes leave as (min, max) pairs and linear indices (none: an index of
// all ones).  Bound by its 28 bytes per voxel: 207 us at 128 x 512 x 512 (van Herk blocks over
// 16 bytes per voxel, two copies and a pass that paired the values: 226 + 107 + 94).
template <int R>
__global__ __launch_bounds__(256) void k_soft_arg_z(const uint32_t* __restrict__ pkn,
                                                    const uint32_t* __restrict__ pkx,
                                                    const uint32_t* __restrict__ ptap,
                                                    float2* __restrict__ pair,
                                                    uint32_t* __restrict__ amn,
                                                    uint32_t* __restrict__ amx, int n, int W,
                                                    int H, int D, int rxy, int r, unsigned nxb,
                                                    unsigned no, int len) {
  extern __shared__ uint32_t sm_argz[];
  const int hist = 2 * r;
  const i64 sa = (i64)W * H;
  uint32_t* Bn = sm_argz;
  uint32_t* Bx = Bn + (hist + kStep) * 64;
  uint32_t* Bt = Bx + (hist + kStep) * 64;
  const RunAt a = run_at(D, W, nxb, no, len);
  const int xn = a.x0 + a.l, xc = min(xn, n - 1);  // column of the plane, or of the row
  const int x = xn % W, y = (int)(a.base / W) + xn / W;
  uint32_t qn[OK], qx[OK], qt[OK];
  auto fetch = [&](int p) {
#pragma unroll
    for (int k = 0; k < OK; ++k) {
      const i64 at = a.base + (i64)clampi(p + k, 0, D - 1) * sa + xc;
      qn[k] = pkn[at];
      qx[k] = pkx[at];
      qt[k] = ptap[at];
    }
  };
  auto put = [&](int row) {
#pragma unroll
    for (int k = 0; k < OK; ++k) {
      Bn[(row + k) * 64 + a.l] = qn[k];
      Bx[(row + k) * 64 + a.l] = qx[k];
      Bt[(row + k) * 64 + a.l] = qt[k];
    }
  };
  for (int g = a.wave; OK * g < hist; g += 4) {  // (the last may reach into the step's rows)
    fetch(a.s0 - r + OK * g);
    put(OK * g);
  }
  if (a.s0 + OK * a.wave < a.s1) fetch(a.s0 + r + OK * a.wave);
  __syncthreads();
  for (int c0 = a.s0; c0 < a.s1; c0 += kStep) {
    const int c = c0 + OK * a.wave;
    if (c < a.s1) put(hist + OK * a.wave);
    if (c + kStep < a.s1) fetch(c + kStep + r);
    __syncthreads();
    if (c < a.s1) {
      const uint32_t* p = Bn + OK * a.wave * 64 + a.l;
      const int plane = (hist + kStep) * 64;
      Arg o[OK];
      arg8<R>([&](int i) -> Arg {
        const uint32_t tp = p[2 * plane];
        const Arg b = {p[0], p[plane], (tp & 0xFFFFu) | (uint32_t)i << 16,
                       tp >> 16 | (uint32_t)i << 16};
        p += 64;
        return b;
      }, r, o);
      if (xn < n) {
#pragma unroll
        for (int k = 0; k < OK; ++k) {
          const int z = c + k;
          if (z >= a.s1) continue;
          auto index = [&](uint32_t tap) -> uint32_t {
            const int jx = clampi(x - rxy + (int)(tap & 0xFFu), 0, W - 1),
                      jy = clampi(y - rxy + (int)(tap >> 8 & 0xFFu), 0, H - 1),
                      jz = clampi(z - r + (int)(tap >> 16) - k, 0, D - 1);
            return ((uint32_t)jz * (uint32_t)H + (uint32_t)jy) * (uint32_t)W + (uint32_t)jx;
          };
          const i64 at = a.base + (i64)z * sa + xn;
          const bool none = o[k].kn == 0xFFFFFFFFu;  // NaN only: then kx is 0
          st_nt(pair + at, make_float2(none ? INFINITY : key_value(o[k].kn),
                                       none ? -INFINITY : key_value(o[k].kx - 1u)));
          st_nt(amn + at, none ? 0xFFFFFFFFu : index(o[k].cn));
          st_nt(amx + at, none ? 0xFFFFFFFFu : index(o[k].cx));
        }
      }
    }
    if (c0 + kStep >= a.s1) break;  // uniform
    __syncthreads();
    shift_rows<256, kStep, 64>(Bn, hist);
    shift_rows<256, kStep, 64>(Bx, hist);
    shift_rows<256, kStep, 64>(Bt, hist);
    __syncthreads();
  }
}

// Clamped box means of the pairs along x and y, sums in window order: as k_soft_arg_xy, with
// the two channels one after the other through the wave's lines.  128 us at 128 x 512 x 512,
// radius 10 (a pass each, 8 bytes per voxel out and back between them: 156 + 185).
template <int R>
__global__ __launch_bounds__(256) void k_soft_box_xy(const float2* __restrict__ src,
                                                     float2* __restrict__ dst, int W, int H, int r,
                                                     int nxs, int nys, int rows, float k) {
  extern __shared__ float sm_bxy[];
  constexpr int BP = 65;
  const int hist = 2 * r, span = 64 + 2 * r, AP = arg_line_pitch(r);
  const int l = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  float* A = sm_bxy + wave * (OK * AP);
  float* B1 = sm_bxy + 4 * (OK * AP);
  float* B2 = B1 + (hist + kStep) * BP;
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int y0 = (int)(t % (unsigned)nys) * rows, y1 = min(H, y0 + rows);
  const unsigned tile = t / (unsigned)nys;
  const int x0 = (int)(tile % (unsigned)nxs) * 64;
  const i64 pbase = (i64)(tile / (unsigned)nxs) * H * W;
  int xl[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) xl[j] = clampi(x0 - r + 64 * j + l, 0, W - 1);
  float2 q[OK][2];
  auto fetch = [&](int y) {
#pragma unroll
    for (int i = 0; i < OK; ++i) {
      const float2* row = src + pbase + (i64)clampi(y + i, 0, H - 1) * W;
#pragma unroll
      for (int j = 0; j < 2; ++j) q[i][j] = row[xl[j]];
    }
  };
  const int xr = l % OK, xg = l / OK;
  auto xsum = [&](float* b) {
    wave_lds_sync();
    const float* p = A + xr * AP + OK * xg;
    float o[OK];
    sum8<R>([&] { return *p++; }, r, o);
#pragma unroll
    for (int i = 0; i < OK; ++i) b[i] = o[i] * k;
    wave_lds_sync();
  };
  auto xpass = [&](int row, int ahead) {
    const int b = (row + xr) * BP + OK * xg;
#pragma unroll
    for (int i = 0; i < OK; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (64 * j + l < span) A[i * AP + 64 * j + l] = q[i][j].x;
    xsum(B1 + b);
#pragma unroll
    for (int i = 0; i < OK; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (64 * j + l < span) A[i * AP + 64 * j + l] = q[i][j].y;
    fetch(ahead);
    xsum(B2 + b);
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
  for (int c0 = y0; c0 < y1; c0 += kStep) {
    xpass(hist + OK * wave, c0 + kStep + r + OK * wave);
    __syncthreads();
    const int c = c0 + OK * wave;
    if (c < y1) {
      float e[OK], d[OK];
      const float* p = B1 + OK * wave * BP + l;
      sum8<R>([&] { const float u = *p; p += BP; return u; }, r, e);
      p = B2 + OK * wave * BP + l;
      sum8<R>([&] { const float u = *p; p += BP; return u; }, r, d);
      if (out) {
#pragma unroll
        for (int o = 0; o < OK; ++o)
          if (c + o < y1) st_nt(dcol + (i64)(c + o) * W, make_float2(e[o] * k, d[o] * k));
      }
    }
    if (c0 + kStep >= y1) break;  // uniform
    __syncthreads();
    shift_rows<256, kStep, BP>(B1, hist);
    shift_rows<256, kStep, BP>(B2, hist);
    __syncthreads();
  }
}

// Clamped box means along z -> (E, D), and the normalization.  Bound by its 24 bytes per
// voxel: 164 us at 128 x 512 x 512 (in two passes, 104 + 109).
template <int R>
__global__ __launch_bounds__(256) void k_soft_box_norm(const float2* __restrict__ src,
                                                       const float* __restrict__ v,
                                                       float2* __restrict__ ed,
                                                       float* __restrict__ norm, float min_int,
                                                       int W, int D, i64 sa, int r, unsigned nxb,
                                                       unsigned no, int len, float k) {
  extern __shared__ float sm_bz[];
  const int hist = 2 * r;
  float* B1 = sm_bz;
  float* B2 = B1 + (hist + kStep) * 64;
  const RunAt a = run_at(D, W, nxb, no, len);
  const int xc = min(a.x0 + a.l, W - 1);
  float2 q[OK];
  float vq[OK];
  auto fetch = [&](int p) {
#pragma unroll
    for (int j = 0; j < OK; ++j) q[j] = src[a.base + (i64)clampi(p + j, 0, D - 1) * sa + xc];
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
  for (int c0 = a.s0; c0 < a.s1; c0 += kStep) {
    const int c = c0 + OK * a.wave;
    if (c < a.s1) {
      put(hist + OK * a.wave);
#pragma unroll
      for (int j = 0; j < OK; ++j) vq[j] = v[a.base + (i64)min(c + j, D - 1) * sa + xc];
    }
    if (c + kStep < a.s1) fetch(c + kStep + r);
    __syncthreads();
    if (c < a.s1) {
      float e[OK], d[OK];
      const float* p = B1 + OK * a.wave * 64 + a.l;
      sum8<R>([&] { const float u = *p; p += 64; return u; }, r, e);
      p = B2 + OK * a.wave * 64 + a.l;
      sum8<R>([&] { const float u = *p; p += 64; return u; }, r, d);
      if (a.x0 + a.l < W) {
#pragma unroll
        for (int j = 0; j < OK; ++j) {
          if (c + j >= a.s1) continue;
          const i64 idx = a.base + (i64)(c + j) * sa + a.x0 + a.l;
          const float ve = e[j] * k, vd = d[j] * k;
          st_nt(ed + idx, make_float2(ve, vd));
          st_nt(norm + idx, vq[j] >= min_int ? (vq[j] - ve) / (vd - ve) : 0.0f);
        }
      }
    }
    if (c0 + kStep >= a.s1) break;  // uniform
    __syncthreads();
    shift_rows<256, kStep, 64>(B1, hist);
    shift_rows<256, kStep, 64>(B2, hist);
    __syncthreads();
  }
}

// one separable pass of the windowed (value, index) minimum and maximum, clamp-to-edge;
// first pass: indices are the voxels' own (imn == NULL)
__global__ __launch_bounds__(NT) void k_soft_argminmax(const float* __restrict__ vmn,
                                                       const uint32_t* __restrict__ imn,
                                                       const float* __restrict__ vmx,
                                                       const uint32_t* __restrict__ imx,
                                                       float* __restrict__ omn, uint32_t* __restrict__ oimn,
                                                       float* __restrict__ omx, uint32_t* __restrict__ oimx,
                                                       int W, int H, int D, int axis, int r,
                                                       unsigned nxb) {
  Pos q;
  if (!pos_of(W, H, nxb, q)) return;
  const i64 i = q.i;
  {
    const Line l = line_at(q, axis, W, H, D);
    float bmn = INFINITY, bmx = -INFINITY;
    uint32_t jmn = 0xFFFFFFFFu, jmx = 0xFFFFFFFFu;
    for (int t = -r; t <= r; ++t) {
      const i64 p = l.base + (i64)clampi(l.c + t, 0, l.L - 1) * l.stride;
      const float a = vmn[p], b = vmx[p];
      const uint32_t ja = imn ? imn[p] : (uint32_t)p, jb = imx ? imx[p] : (uint32_t)p;
      if (a < bmn || (a == bmn && ja < jmn)) { bmn = a; jmn = ja; }
      if (b > bmx || (b == bmx && jb < jmx)) { bmx = b; jmx = jb; }
    }
    omn[i] = bmn; oimn[i] = jmn;
    omx[i] = bmx; oimx[i] = jmx;
  }
}

// The x passes with the work-group's row segment x0 - r .. x0 + NT - 1 + r staged in LDS
// (clamped to the row): the same taps, in the same order, as the line kernels, each read
// from LDS instead of global memory.  For radii up to kXR; others use the line kernels.
constexpr int kXR = 64;

// stages the clamped row segment of the work-group; returns the row's linear base, x0
template <typename T>
__device__ __forceinline__ i64 stage_row(const T* __restrict__ in, T* sv, int W, int r,
                                         unsigned nxb, int& x0) {
  const unsigned row = blockIdx.x / nxb;
  x0 = (int)(blockIdx.x - row * nxb) * NT;
  const i64 base = (i64)row * W;
  for (int e = (int)threadIdx.x; e < NT + 2 * r; e += NT) sv[e] = in[base + clampi(x0 - r + e, 0, W - 1)];
  __syncthreads();
  return base;
}

// first (x) pass of the windowed (value, index) minimum and maximum: value v[p], index p
__global__ __launch_bounds__(NT) void k_soft_argminmax_x(const float* __restrict__ v,
                                                         float* __restrict__ omn,
                                                         uint32_t* __restrict__ oimn,
                                                         float* __restrict__ omx,
                                                         uint32_t* __restrict__ oimx, int W,
                                                         int r, unsigned nxb) {
  __shared__ float sv[NT + 2 * kXR];
  int x0;
  const i64 base = stage_row(v, sv, W, r, nxb, x0);
  const int x = x0 + (int)threadIdx.x;
  if (x >= W) return;
  float bmn = INFINITY, bmx = -INFINITY;
  uint32_t jmn = 0xFFFFFFFFu, jmx = 0xFFFFFFFFu;
  for (int t = -r; t <= r; ++t) {
    const int c = clampi(x + t, 0, W - 1);
    const float a = sv[x + t - x0 + r];  // the value at c
    const uint32_t j = (uint32_t)(base + c);
    if (a < bmn || (a == bmn && j < jmn)) { bmn = a; jmn = j; }
    if (a > bmx || (a == bmx && j < jmx)) { bmx = a; jmx = j; }
  }
  omn[base + x] = bmn; oimn[base + x] = jmn;
  omx[base + x] = bmx; oimx[base + x] = jmx;
}

// clamped box mean of the (E, D) pair along x (FP32 sums in window order)
__global__ __launch_bounds__(NT) void k_soft_box_x(const float2* __restrict__ in,
                                                   float2* __restrict__ out, int W, int r,
                                                   unsigned nxb) {
  __shared__ float2 sv[NT + 2 * kXR];
  const float k = 1.0f / (float)(2 * r + 1);
  int x0;
  const i64 base = stage_row(in, sv, W, r, nxb, x0);
  const int x = x0 + (int)threadIdx.x;
  if (x >= W) return;
  float se = 0.0f, sd = 0.0f;
  for (int t = -r; t <= r; ++t) {
    const float2 v = sv[x + t - x0 + r];
    se += v.x;
    sd += v.y;
  }
  out[base + x] = make_float2(se * k, sd * k);
}

// transpose of the clamped box mean along x (k_soft_box_adj's sums, from LDS)
__global__ __launch_bounds__(NT) void k_soft_box_adj_x(const float2* __restrict__ in,
                                                       float2* __restrict__ out, int W, int r,
                                                       unsigned nxb) {
  __shared__ float2 sv[NT + 2 * kXR];
  const float k = 1.0f / (float)(2 * r + 1);
  int x0;
  const i64 base = stage_row(in, sv, W, r, nxb, x0);
  const int p = x0 + (int)threadIdx.x, L = W;
  if (p >= W) return;
  const int o = r - x0;  // LDS slot of position c: c + o
  float se = 0.0f, sd = 0.0f;
  for (int c = max(0, p - r); c <= min(L - 1, p + r); ++c) {
    const float2 v = sv[c + o];
    se += v.x;
    sd += v.y;
  }
  if (p == 0)
    for (int c = 0; c <= min(L - 1, r - 1); ++c) {
      const float2 v = sv[c + o];
      se += v.x * (float)(r - c);
      sd += v.y * (float)(r - c);
    }
  if (p == L - 1)
    for (int c = max(0, L - r); c <= L - 1; ++c) {
      const float2 v = sv[c + o];
      se += v.x * (float)(c + r - L + 1);
      sd += v.y * (float)(c + r - L + 1);
    }
  out[base + p] = make_float2(se * k, sd * k);
}

// Transpose of the clamped box mean over eight positions c .. c + 7 of a line of L (radius r):
// acc holds the window sums over the line (zero outside it); the border positions also
// receive the taps that clamp onto them.  B: position `first` of the line, `pitch` apart.
__device__ __forceinline__ void add_clamped(const float* B, int pitch, int first, int c, int L,
                                            int r, float (&acc)[OK]) {
  if (c == 0)  // taps c - r + j < 0 of the windows of c < r
    for (int i = 0; i <= min(L - 1, r - 1); ++i) acc[0] += B[(i - first) * pitch] * (float)(r - i);
  if (c <= L - 1 && L - 1 < c + OK) {  // taps beyond L - 1 of the windows of c > L - 1 - r
    float t = 0.0f;
    for (int i = max(0, L - r); i <= L - 1; ++i)
      t += B[(i - first) * pitch] * (float)(i + r - L + 1);
#pragma unroll
    for (int o = 0; o < OK; ++o)
      if (c + o == L - 1) acc[o] += t;
  }
}

// Adjoint of the normalization and, transposed, of its z boxes: the direct term into gv, (dL/dE,
// dL/dD) summed along z into dst.  Bound by its 28 bytes per voxel: 184 us at 128 x 512 x 512,
// radius 10 (in two passes, 152 + 112).  rbox: the boxes' radius; r: that of the sums, which
// need no more than the line's length, being zero past its ends.
template <int R>
__global__ __launch_bounds__(256) void k_soft_adj_z(const float* __restrict__ v,
                                                    const float2* __restrict__ ed,
                                                    const float* __restrict__ gn,
                                                    float* __restrict__ gv,
                                                    float2* __restrict__ dst, float min_int, int W,
                                                    int D, i64 sa, int r, int rbox, unsigned nxb,
                                                    unsigned no, int len, float k) {
  extern __shared__ float sm_adjz[];
  const int hist = 2 * r;
  float* B1 = sm_adjz;
  float* B2 = B1 + (hist + kStep) * 64;
  const RunAt a = run_at(D, W, nxb, no, len);
  const bool out = a.x0 + a.l < W;
  const int xc = min(a.x0 + a.l, W - 1);
  float qv[OK], qg[OK];
  float2 qe[OK];
  auto fetch = [&](int p) {
#pragma unroll
    for (int j = 0; j < OK; ++j) {
      const i64 at = a.base + (i64)clampi(p + j, 0, D - 1) * sa + xc;
      qv[j] = v[at];
      qe[j] = ed[at];
      qg[j] = gn[at];
    }
  };
  auto put = [&](int row, int p) {  // the fetched positions p .. p + 7
#pragma unroll
    for (int j = 0; j < OK; ++j) {
      const bool in = p + j >= 0 && p + j < D;
      const float I = qv[j], g = I >= min_int ? qg[j] : 0.0f;
      const float inv = 1.0f / (qe[j].y - qe[j].x);
      B1[(row + j) * 64 + a.l] = in ? g * (I - qe[j].y) * inv * inv : 0.0f;
      B2[(row + j) * 64 + a.l] = in ? -g * (I - qe[j].x) * inv * inv : 0.0f;
      if (out && p + j >= a.s0 && p + j < a.s1)
        gv[a.base + (i64)(p + j) * sa + a.x0 + a.l] = g * inv;
    }
  };
  for (int g = a.wave; OK * g < hist; g += 4) {  // (the last may reach into the step's rows)
    fetch(a.s0 - r + OK * g);
    put(OK * g, a.s0 - r + OK * g);
  }
  if (a.s0 + OK * a.wave < a.s1) fetch(a.s0 + r + OK * a.wave);
  __syncthreads();
  for (int c0 = a.s0; c0 < a.s1; c0 += kStep) {
    const int c = c0 + OK * a.wave;
    if (c < a.s1) put(hist + OK * a.wave, c + r);
    if (c + kStep < a.s1) fetch(c + kStep + r);
    __syncthreads();
    if (c < a.s1) {
      float e[OK], d[OK];
      const float* p = B1 + OK * a.wave * 64 + a.l;
      sum8<R>([&] { const float u = *p; p += 64; return u; }, r, e);
      p = B2 + OK * a.wave * 64 + a.l;
      sum8<R>([&] { const float u = *p; p += 64; return u; }, r, d);
      add_clamped(B1 + a.l, 64, c0 - r, c, D, rbox, e);
      add_clamped(B2 + a.l, 64, c0 - r, c, D, rbox, d);
      if (out) {
#pragma unroll
        for (int j = 0; j < OK; ++j)
          if (c + j < a.s1)
            st_nt(dst + a.base + (i64)(c + j) * sa + a.x0 + a.l, make_float2(e[j] * k, d[j] * k));
      }
    }
    if (c0 + kStep >= a.s1) break;  // uniform
    __syncthreads();
    shift_rows<256, kStep, 64>(B1, hist);
    shift_rows<256, kStep, 64>(B2, hist);
    __syncthreads();
  }
}

// Sum of v over the run of equal consecutive keys (lanes of one wave) that starts at each
// run's first lane, where *head is set; every lane of the wave must be active.  A segmented
// suffix sum by lane shifts: after the step of offset o each lane holds the sum over
// [lane, lane + 2o) within its run.
__device__ __forceinline__ float run_sum(uint32_t key, float v, bool* head) {
  const int lane = (int)(threadIdx.x & 63);
  const uint32_t prev = __shfl_up(key, 1, 64);
  *head = lane == 0 || prev != key;
  const unsigned long long heads = __ballot(*head);
  const unsigned long long after = lane == 63 ? 0ull : heads & (~0ull << (lane + 1));
  const int tail = after ? __builtin_ctzll(after) - 1 : 63;  // last lane of the run
  for (int o = 1; o < 64; o <<= 1) {
    const float w = __shfl_down(v, o, 64);
    if (lane + o <= tail) v += w;
  }
  return v;
}

// Sums per target of the values that a work-group routes in a step, in LDS: windows of a patch
// share a few dozen extremes.  A target that finds no slot in kProbes (plateaus, where every
// window has its own extreme) goes to memory, where it is then not contended.
constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr int kRouteSlots = 512, kProbes = 4;
struct RouteTable {
  uint32_t* key;
  float* sum;
  __device__ __forceinline__ void add(uint32_t k, float s, float* gv) const {
    uint32_t slot = k * 2654435761u >> 23;
    static_assert(kRouteSlots == 1 << 9, "hash bits");
    for (int p = 0; p < kProbes; ++p, slot = (slot + 1) & (kRouteSlots - 1)) {
      // (a key, once set, stays until the flush; other lanes may be setting it)
      uint32_t cur = __atomic_load_n(&key[slot], __ATOMIC_RELAXED);
      if (cur == kNone) {
        cur = atomicCAS(&key[slot], kNone, k);
        if (cur == kNone) cur = k;
      }
      if (cur == k) {
        __hip_atomic_fetch_add(&sum[slot], s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return;
      }
    }
    atomicAdd(gv + k, s);
  }
  // whole work-group, between barriers: the sums leave (to memory, unless clearing only)
  __device__ __forceinline__ void flush(float* gv) const {
    for (int i = (int)threadIdx.x; i < kRouteSlots; i += 256) {
      const uint32_t k = key[i];
      if (gv && k != kNone) atomicAdd(gv + k, sum[i]);
      key[i] = kNone;
      sum[i] = 0.0f;
    }
  }
};
// A lane's eight rows of one column: mostly one or two targets, summed before they go to the
// table, and once more over runs of equal targets in neighbouring columns (LDS adds to one
// address take turns: 392 us for the whole pass below without, 208 with no routing at all).
// Rows without a target have key kNone and value 0.
__device__ __forceinline__ void route8(const uint32_t (&key)[OK], const float (&val)[OK],
                                       const RouteTable& t, float* gv) {
  uint32_t k1 = key[0], k2 = kNone;
  float s1 = val[0], s2 = 0.0f;
#pragma unroll
  for (int o = 1; o < OK; ++o) {
    const uint32_t k = key[o];
    const bool m1 = k == k1, m2 = !m1 && (k == k2 || k2 == kNone);
    s1 += m1 ? val[o] : 0.0f;
    s2 += m2 ? val[o] : 0.0f;
    k2 = m2 ? k : k2;
    if (!m1 && !m2 && k != kNone) t.add(k, val[o], gv);
  }
  bool h1, h2;
  s1 = run_sum(k1, s1, &h1);
  s2 = run_sum(k2, s2, &h2);
  if (h1 && k1 != kNone) t.add(k1, s1, gv);
  if (h2 && k2 != kNone) t.add(k2, s2, gv);
}

// The transposed x and y boxes (walked as k_soft_box_xy, zero outside the plane), and the
// routing of their sums by subgradient: gv[argmin(i)] += dL/dmin(i), gv[argmax(i)] +=
// dL/dmax(i).  The sums never leave the chip.  355 us at 128 x 512 x 512, radius 10 (the two
// boxes and a routing pass with one atomic per run of equal targets in a row of 64: 308 + 183 +
// 490), of which the routing takes 147: short runs in the maximum's plateaus.
template <int R>
__global__ __launch_bounds__(256) void k_soft_adj_xy(const float2* __restrict__ src,
                                                     const uint32_t* __restrict__ amn,
                                                     const uint32_t* __restrict__ amx,
                                                     float* __restrict__ gv, int W, int H, int r,
                                                     int nxs, int nys, int rows, float k) {
  extern __shared__ float sm_axy[];
  constexpr int BP = 65;
  const int hist = 2 * r, span = 64 + 2 * r, AP = arg_line_pitch(r);
  const int l = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  float* A = sm_axy + wave * (OK * AP);
  float* B1 = sm_axy + 4 * (OK * AP);
  float* B2 = B1 + (hist + kStep) * BP;
  const RouteTable table = {reinterpret_cast<uint32_t*>(B2 + (hist + kStep) * BP),
                            B2 + (hist + kStep) * BP + kRouteSlots};
  table.flush(nullptr);  // (cleared; barriers follow)
  const unsigned t = xcd_tile(blockIdx.x, gridDim.x);
  const int y0 = (int)(t % (unsigned)nys) * rows, y1 = min(H, y0 + rows);
  const unsigned tile = t / (unsigned)nys;
  const int x0 = (int)(tile % (unsigned)nxs) * 64;
  const i64 pbase = (i64)(tile / (unsigned)nxs) * H * W;
  int xl[2];
  bool xin[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int x = x0 - r + 64 * j + l;
    xl[j] = clampi(x, 0, W - 1);
    xin[j] = x >= 0 && x < W;
  }
  float2 q[OK][2];
  auto fetch = [&](int y) {
#pragma unroll
    for (int i = 0; i < OK; ++i) {
      const float2* row = src + pbase + (i64)clampi(y + i, 0, H - 1) * W;
#pragma unroll
      for (int j = 0; j < 2; ++j) q[i][j] = row[xl[j]];
    }
  };
  const int xr = l % OK, xg = l / OK;
  auto xsum = [&](float* b) {
    wave_lds_sync();
    const float* line = A + xr * AP;
    const float* p = line + OK * xg;
    float o[OK];
    sum8<R>([&] { return *p++; }, r, o);
    add_clamped(line, 1, x0 - r, x0 + OK * xg, W, r, o);
#pragma unroll
    for (int i = 0; i < OK; ++i) b[i] = o[i] * k;
    wave_lds_sync();
  };
  auto xpass = [&](int row, int y, int ahead) {  // the fetched rows y .. y + 7
    const int b = (row + xr) * BP + OK * xg;
#pragma unroll
    for (int i = 0; i < OK; ++i) {
      const bool in = y + i >= 0 && y + i < H;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (64 * j + l < span) A[i * AP + 64 * j + l] = in && xin[j] ? q[i][j].x : 0.0f;
    }
    xsum(B1 + b);
#pragma unroll
    for (int i = 0; i < OK; ++i) {
      const bool in = y + i >= 0 && y + i < H;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (64 * j + l < span) A[i * AP + 64 * j + l] = in && xin[j] ? q[i][j].y : 0.0f;
    }
    fetch(ahead);
    xsum(B2 + b);
  };
  const int main0 = y0 + r + OK * wave;
  if (OK * wave < hist) {
    fetch(y0 - r + OK * wave);
    for (int g = wave; OK * g < hist; g += 4)
      xpass(OK * g, y0 - r + OK * g, OK * (g + 4) < hist ? y0 - r + OK * (g + 4) : main0);
  } else {
    fetch(main0);
  }
  __syncthreads();
  const int xc = min(x0 + l, W - 1);
  const bool out = x0 + l < W;
  for (int c0 = y0; c0 < y1; c0 += kStep) {
    const int c = c0 + OK * wave;
    xpass(hist + OK * wave, c + r, c + kStep + r);
    uint32_t kn[OK], kx[OK];
#pragma unroll
    for (int o = 0; o < OK; ++o) {
      const i64 at = pbase + (i64)min(c + o, H - 1) * W + xc;
      kn[o] = amn[at];
      kx[o] = amx[at];
    }
    __syncthreads();
    if (c < y1) {
      auto channel = [&](const float* B, uint32_t (&key)[OK]) {
        float acc[OK];
        const float* p = B + OK * wave * BP + l;
        sum8<R>([&] { const float u = *p; p += BP; return u; }, r, acc);
        add_clamped(B + l, BP, c0 - r, c, H, r, acc);
#pragma unroll
        for (int o = 0; o < OK; ++o) {
          acc[o] *= k;
          if (!out || c + o >= y1 || acc[o] == 0.0f) key[o] = kNone;
          if (key[o] == kNone) acc[o] = 0.0f;
        }
        route8(key, acc, table, gv);
      };
      channel(B1, kn);
      channel(B2, kx);
    }
    __syncthreads();
    table.flush(gv);
    if (c0 + kStep >= y1) break;  // uniform
    shift_rows<256, kStep, BP>(B1, hist);
    shift_rows<256, kStep, BP>(B2, hist);
    __syncthreads();
  }
}

// ---- any radius ------------------------------------------------------------------------
// clamped box mean of the (E, D) pair along one axis (FP32 sums in window order)
__global__ __launch_bounds__(NT) void k_soft_box(const float2* __restrict__ in,
                                                 float2* __restrict__ out, int W, int H, int D,
                                                 int axis, int r, unsigned nxb) {
  const float k = 1.0f / (float)(2 * r + 1);
  Pos q;
  if (!pos_of(W, H, nxb, q)) return;
  const i64 i = q.i;
  {
    const Line l = line_at(q, axis, W, H, D);
    float se = 0.0f, sd = 0.0f;
    for (int t = -r; t <= r; ++t) {
      const float2 v = in[l.base + (i64)clampi(l.c + t, 0, l.L - 1) * l.stride];
      se += v.x;
      sd += v.y;
    }
    out[i] = make_float2(se * k, sd * k);
  }
}

// transpose of the clamped box mean along one axis: position p receives every window tap
// that lands on it, border positions also the taps that clamp onto them
__global__ __launch_bounds__(NT) void k_soft_box_adj(const float2* __restrict__ in,
                                                     float2* __restrict__ out, int W, int H,
                                                     int D, int axis, int r, unsigned nxb) {
  const float k = 1.0f / (float)(2 * r + 1);
  Pos q;
  if (!pos_of(W, H, nxb, q)) return;
  const i64 i = q.i;
  {
    const Line l = line_at(q, axis, W, H, D);
    const int p = l.c, L = l.L;
    float se = 0.0f, sd = 0.0f;
    for (int c = max(0, p - r); c <= min(L - 1, p + r); ++c) {
      const float2 v = in[l.base + (i64)c * l.stride];
      se += v.x;
      sd += v.y;
    }
    if (p == 0)  // taps c - r + j < 0 of the windows of c < r clamp onto 0
      for (int c = 0; c <= min(L - 1, r - 1); ++c) {
        const float2 v = in[l.base + (i64)c * l.stride];
        se += v.x * (float)(r - c);
        sd += v.y * (float)(r - c);
      }
    if (p == L - 1)  // taps c - r + j > L - 1 of the windows of c > L - 1 - r clamp onto L - 1
      for (int c = max(0, L - r); c <= L - 1; ++c) {
        const float2 v = in[l.base + (i64)c * l.stride];
        se += v.x * (float)(c + r - L + 1);
        sd += v.y * (float)(c + r - L + 1);
      }
    out[i] = make_float2(se * k, sd * k);
  }
}

__global__ __launch_bounds__(NT) void k_soft_norm(const float* __restrict__ v,
                                                  const float2* __restrict__ ed,
                                                  float* __restrict__ norm, float min_int, i64 N) {
  for (i64 i = (i64)blockIdx.x * NT + threadIdx.x; i < N; i += (i64)gridDim.x * NT) {
    const float I = v[i];
    const float2 e = ed[i];
    norm[i] = I >= min_int ? (I - e.x) / (e.y - e.x) : 0.0f;
  }
}

// direct term into gv; (dL/dE, dL/dD) into g_ed
__global__ __launch_bounds__(NT) void k_soft_norm_adj(const float* __restrict__ v,
                                                      const float2* __restrict__ ed,
                                                      const float* __restrict__ gn,
                                                      float* __restrict__ gv,
                                                      float2* __restrict__ g_ed, float min_int,
                                                      i64 N) {
  for (i64 i = (i64)blockIdx.x * NT + threadIdx.x; i < N; i += (i64)gridDim.x * NT) {
    const float I = v[i];
    const float2 e = ed[i];
    const float g = I >= min_int ? gn[i] : 0.0f;
    const float inv = 1.0f / (e.y - e.x);
    gv[i] = g * inv;
    g_ed[i] = make_float2(g * (I - e.y) * inv * inv, -g * (I - e.x) * inv * inv);
  }
}

// subgradient routing: gv[argmin(i)] += dL/dmin(i), gv[argmax(i)] += dL/dmax(i).  Windows
// of neighbouring voxels mostly share their extreme, so a wave first sums its lanes' values
// per run of equal targets and adds each run with one atomic (one atomic per voxel made the
// contended targets serialize).
__global__ __launch_bounds__(NT) void k_soft_route(const float2* __restrict__ g,
                                                   const uint32_t* __restrict__ amn,
                                                   const uint32_t* __restrict__ amx,
                                                   float* __restrict__ gv, i64 N) {
  const int lane = (int)(threadIdx.x & 63);
  for (i64 b = (i64)blockIdx.x * NT + (threadIdx.x - lane); b < N; b += (i64)gridDim.x * NT) {
    const i64 i = b + lane;  // the whole wave iterates together
    const bool ok = i < N;
    const float2 q = ok ? g[i] : make_float2(0.0f, 0.0f);
    const uint32_t kmn = ok ? amn[i] : kNone, kmx = ok ? amx[i] : kNone;
    bool hmn, hmx;
    const float smn = run_sum(kmn, q.x, &hmn);
    const float smx = run_sum(kmx, q.y, &hmx);
    if (hmn && kmn != kNone && smn != 0.0f) atomicAdd(gv + kmn, smn);
    if (hmx && kmx != kNone && smx != 0.0f) atomicAdd(gv + kmx, smx);
  }
}

}  // namespace

// norm, and for the backward pass ed (E, D pairs) and arg (argmin N, then argmax N);
// scratch: 8 N words (radii up to kArgRadius: 5 N, one more for an odd N)
hipError_t launch_soft_normalize(const float* v, float* norm, float2* ed, uint32_t* arg,
                                 void* scratch, float min_int, int W, int H, int D, int rxy,
                                 int rz, hipStream_t s) {
  const i64 N = (i64)W * H * D, WH = (i64)W * H;
  if (rxy <= kArgRadius && rz <= kArgRadius) {
    uint32_t* pk = (uint32_t*)scratch;       // keys and taps, 3 N words
    float2* pair = (float2*)(pk + (3 * N + 1) / 2 * 2);  // 2 N words, on whole pairs
    float2* exy = (float2*)scratch;          // in the place of the keys
    const XyRun x = xy_run(W, H, D, rxy);
    const ZColumns c = z_columns(W, H);
    const LineGrid g = run_grid(c.n, D, c.rows, 2 * rz);
    const float kxy = 1.0f / (float)(2 * rxy + 1), kz = 1.0f / (float)(2 * rz + 1);
    // the extremes of a window past both ends of its line are those of one that reaches them
    const int mz = std::min(rz, std::max(1, D - 1));
    const LineGrid m = run_grid(c.n, D, c.rows, 2 * mz);
    const size_t zrows = (size_t)(2 * rz + kStep) * 64 * 4, mrows = (size_t)(2 * mz + kStep) * 64 * 4;
    hipError_t e = dispatch_short(rxy, [&](auto rs) {
      constexpr int R = decltype(rs)::value;
      hipLaunchKernelGGL((k_soft_arg_xy<R>), dim3(x.blocks), dim3(256), arg_xy_lds(rxy), s, v, pk, pk + N,
                         pk + 2 * N, W, H, rxy, x.nxs, x.nys, x.rows);
      return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    e = dispatch_short(mz, [&](auto rs) {
      constexpr int R = decltype(rs)::value;
      hipLaunchKernelGGL((k_soft_arg_z<R>), dim3(m.blocks), dim3(256), 3 * mrows, s, pk, pk + N,
                         pk + 2 * N, pair, arg, arg + N, c.n, W, H, D, rxy, mz, m.nxb, m.no, m.len);
      return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    e = dispatch_short(rxy, [&](auto rs) {
      constexpr int R = decltype(rs)::value;
      hipLaunchKernelGGL((k_soft_box_xy<R>), dim3(x.blocks), dim3(256), box_xy_lds(rxy), s, pair,
                         exy, W, H, rxy, x.nxs, x.nys, x.rows, kxy);
      return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    if (D <= kShallow) {
      e = launch_box_pair(exy, ed, c.n, D, WH, W, c.rows, rz, s);
      if (e != hipSuccess) return e;
      hipLaunchKernelGGL(k_soft_norm, dim3(grid_for(N)), dim3(NT), 0, s, v, ed, norm, min_int, N);
      return hipGetLastError();
    }
    return dispatch_short(rz, [&](auto rs) {
      constexpr int R = decltype(rs)::value;
      hipLaunchKernelGGL((k_soft_box_norm<R>), dim3(g.blocks), dim3(256), 2 * zrows, s, exy, v, ed,
                         norm, min_int, c.n, D, WH, rz, g.nxb, g.no, g.len, kz);
      return hipGetLastError();
    });
  }
  float* a = (float*)scratch;  // ping-pong (value, index) min / max planes
  float* fmn[2] = {a, a + 4 * N};
  const unsigned g = grid_for(N);
  const int rad[3] = {rxy, rxy, rz};
  for (int axis = 0; axis < 3; ++axis) {
    float* src = fmn[(axis + 1) & 1];
    float* dst = fmn[axis & 1];
    const float* vmn = axis ? src : v;
    const float* vmx = axis ? src + 2 * N : v;
    const uint32_t* imn = axis ? (const uint32_t*)(src + N) : nullptr;
    const uint32_t* imx = axis ? (const uint32_t*)(src + 3 * N) : nullptr;
    if (axis == 0 && rad[0] <= kXR) {  // x, the first pass: indices are positions
      hipLaunchKernelGGL(k_soft_argminmax_x, dim3(grid_rows(W, H, D)), dim3(NT), 0, s, v, dst,
                         (uint32_t*)(dst + N), dst + 2 * N, (uint32_t*)(dst + 3 * N), W, rad[0],
                         xblocks(W));
    } else {
      hipLaunchKernelGGL(k_soft_argminmax, dim3(grid_rows(W, H, D)), dim3(NT), 0, s, vmn, imn,
                         vmx, imx, dst, (uint32_t*)(dst + N), dst + 2 * N,
                         (uint32_t*)(dst + 3 * N), W, H, D, axis, rad[axis], xblocks(W));
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const float* res = fmn[0];  // axis 2 wrote plane set 0
  hipError_t e = hipMemcpyAsync(arg, res + N, N * 4, hipMemcpyDeviceToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(arg + N, res + 3 * N, N * 4, hipMemcpyDeviceToDevice, s);
  if (e != hipSuccess) return e;
  // (min, max) pairs -> box along x, y, z -> (E, D)
  float2* p0 = (float2*)fmn[1];
  float2* p1 = ed;
  hipLaunchKernelGGL(k_pack_pair, dim3(g), dim3(NT), 0, s, res, res + 2 * N, p0, N);
  float2* bufs[2] = {p0, p1};
  for (int axis = 0; axis < 3; ++axis) {
    // x: p0 -> ed, y: ed -> p0, z: p0 -> ed; y and z by the normalization's box passes
    if (axis == 0 && rad[0] <= kXR) {
      hipLaunchKernelGGL(k_soft_box_x, dim3(grid_rows(W, H, D)), dim3(NT), 0, s, bufs[0],
                         bufs[1], W, rad[0], xblocks(W));
    } else if (axis == 0) {
      hipLaunchKernelGGL(k_soft_box, dim3(grid_rows(W, H, D)), dim3(NT), 0, s, bufs[0], bufs[1],
                         W, H, D, axis, rad[axis], xblocks(W));
    } else {
      e = launch_box_pair(bufs[axis & 1], bufs[(axis + 1) & 1], W, axis == 1 ? H : D,
                          axis == 1 ? W : WH, axis == 1 ? WH : W, axis == 1 ? D : H, rad[axis], s);
      if (e != hipSuccess) return e;
    }
  }
  hipLaunchKernelGGL(k_soft_norm, dim3(g), dim3(NT), 0, s, v, ed, norm, min_int, N);
  return hipGetLastError();
}

hipError_t launch_soft_normalize_adjoint(const float* v, const float2* ed, const uint32_t* arg,
                                         const float* gn, float* gv, void* scratch,
                                         float min_int, int W, int H, int D, int rxy, int rz,
                                         hipStream_t s) {
  const i64 N = (i64)W * H * D, WH = (i64)W * H;
  float2* q0 = (float2*)scratch;
  if (rxy <= kArgRadius && rz <= kArgRadius) {
    const ZColumns c = z_columns(W, H);
    const int sz = std::min(rz, D);
    const LineGrid g = run_grid(c.n, D, c.rows, 2 * sz);
    hipError_t e = dispatch_short(sz, [&](auto rs) {
      constexpr int R = decltype(rs)::value;
      hipLaunchKernelGGL((k_soft_adj_z<R>), dim3(g.blocks), dim3(256),
                         2 * (size_t)(2 * sz + kStep) * 64 * 4, s, v, ed, gn, gv, q0, min_int,
                         c.n, D, WH, sz, rz, g.nxb, g.no, g.len, 1.0f / (float)(2 * rz + 1));
      return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    const XyRun x = xy_run(W, H, D, rxy);
    return dispatch_short(rxy, [&](auto rs) {
      constexpr int R = decltype(rs)::value;
      hipLaunchKernelGGL((k_soft_adj_xy<R>), dim3(x.blocks), dim3(256),
                         box_xy_lds(rxy) + kRouteSlots * 8, s, q0, arg, arg + N, gv, W, H, rxy,
                         x.nxs, x.nys, x.rows, 1.0f / (float)(2 * rxy + 1));
      return hipGetLastError();
    });
  }
  float2* q1 = q0 + N;
  const unsigned g = grid_for(N);
  const int rad[3] = {rxy, rxy, rz};
  hipLaunchKernelGGL(k_soft_norm_adj, dim3(g), dim3(NT), 0, s, v, ed, gn, gv, q0, min_int, N);
  // the box was applied x, y, z: its transpose runs z, y, x
  float2* bufs[2] = {q0, q1};
  for (int k = 0; k < 3; ++k) {
    const int axis = 2 - k;
    if (axis == 0 && rad[0] <= kXR)
      hipLaunchKernelGGL(k_soft_box_adj_x, dim3(grid_rows(W, H, D)), dim3(NT), 0, s,
                         bufs[k & 1], bufs[(k + 1) & 1], W, rad[0], xblocks(W));
    else
      hipLaunchKernelGGL(k_soft_box_adj, dim3(grid_rows(W, H, D)), dim3(NT), 0, s, bufs[k & 1],
                         bufs[(k + 1) & 1], W, H, D, axis, rad[axis], xblocks(W));
  }
  hipLaunchKernelGGL(k_soft_route, dim3(g), dim3(NT), 0, s, bufs[1], arg, arg + N, gv, N);
  return hipGetLastError();
}

// grid of a pass over tiles that ends in a reduction
static unsigned grid_tiles(i64 ntiles) { return (unsigned)std::min<i64>(ntiles, kReduceGroups); }

hipError_t launch_soft_loss(const float* cand, const uint32_t* cand_cnt, const uint8_t* target,
                            int W, int H, int D, double inv_tau, double* sums, hipStream_t s) {
  const i64 nt = hessian_tiles(W, H, D);
  const unsigned nbx = (unsigned)((W + kHessTX - 1) / kHessTX),
                 nby = (unsigned)((H + kHessTY - 1) / kHessTY);
  hipLaunchKernelGGL(k_zero_f64, dim3(1), dim3(64), 0, s, sums, 2);
  hipLaunchKernelGGL(k_soft_loss, dim3(grid_tiles(nt)), dim3(NT), 0, s, cand, cand_cnt, target,
                     (unsigned)nt, nbx, nby, W, H, D, inv_tau, sums);
  return hipGetLastError();
}

hipError_t launch_soft_grad_h(float* cand, const uint32_t* cand_cnt, const uint8_t* target, int W,
                              int H, int D, double inv_tau, double inv_count, double* sums,
                              hipStream_t s) {
  const i64 nt = hessian_tiles(W, H, D);
  const unsigned nbx = (unsigned)((W + kHessTX - 1) / kHessTX),
                 nby = (unsigned)((H + kHessTY - 1) / kHessTY);
  hipLaunchKernelGGL(k_soft_grad_h, dim3(grid_tiles(nt)), dim3(NT), 0, s, cand, cand_cnt, target,
                     (unsigned)nt, nbx, nby, W, H, D, inv_tau, inv_count, sums);
  return hipGetLastError();
}

hipError_t launch_hessian_adjoint(const float* cand, const TileRow* rows, const float* dog,
                                  float* out, int W, int H, int D, double* dot, hipStream_t s) {
  const int nsx = (W + kAdjX - 1) / kAdjX, nsy = (H + AR - 1) / AR;
  const i64 groups = ((i64)nsx * nsy + NT / 64 - 1) / (NT / 64);
  int nseg, len;
  line_segments(D, groups, 1024.0, 1.0, false, 4, &nseg, &len);
  const i64 waves = (i64)nsx * nsy * nseg;
  hipLaunchKernelGGL(k_hessian_adjoint, dim3((unsigned)((waves + NT / 64 - 1) / (NT / 64))),
                     dim3(NT), 0, s, cand, rows, dog, out, nsx, nsy, row_pieces(W), len, W, H, D,
                     dot);
  return hipGetLastError();
}

hipError_t launch_zero_f64(double* p, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_zero_f64, dim3(1), dim3(64), 0, s, p, n);
  return hipGetLastError();
}

}  // namespace hdog
