// regions.hip -- per-region features without sorting.
//
// Reference semantics (src/3D/RegionalFeatures.cu:65-329, src/3D/Eigenvalues.cu:18-112):
// regions are the distinct labels in ascending order (region 0 = background), each with
// the six Hessian sums, max (or, in ave mode, sum) of normalized intensity, the voxel
// count as u16 (wrapping modulo 65536), the centroid sum(coord) / (float)size and the
// eigen-features of the summed Hessian in FP64.  The reference gets there with CUB radix
// sorts of (label, value) pairs and reduce-by-key, about 1 KB of traffic per voxel.
//
// MI355X design: the labels already are the component minima, so a region's id is the
// rank of its root among all roots in linear order -- root counts at three levels, then an
// assign pass that preserves the reference's ascending order.  Each work-group folds its voxels
// into an LDS table of partial sums (packed integer sums, FP64 Hessian and
// intensity-float sums, ordered-integer max for the float max); each table entry then
// ends in the region's 128-byte accumulator line, stored when the work-group holds the
// whole region, else added with hardware atomics (u64 counts and coordinate / intensity
// sums, exact; FP64 sums).  A finalize kernel turns the sums into the reference's output
// arrays.
#include "hdog_internal.hpp"

namespace hdog {
namespace {

constexpr int NT = 256;
constexpr int ITEMS = 16;
constexpr i64 BLK = (i64)NT * ITEMS;  // voxels per numbering block
static_assert(BLK == kRootBlock, "numbering block");

__device__ __forceinline__ int wave_sum_int(int v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;  // lane 0 holds the sum
}

// Per block of BLK voxels: the positions of the roots (L[i] == i, i > 0) as a bitmask
// (masks[64 b + 4 k + wave] bit lane <-> voxel b*BLK + k*NT + 64 wave + lane, so bit order is
// linear order).  Clears the chunk counts for the counting kernel.
__global__ __launch_bounds__(NT) void k_root_bits(const uint32_t* __restrict__ L, i64 N,
                                                  unsigned long long* __restrict__ masks,
                                                  uint32_t* __restrict__ chunk_counts,
                                                  int chunks) {
  if (blockIdx.x == 0)
    for (int i = (int)threadIdx.x; i < chunks; i += NT) chunk_counts[i] = 0u;
  const i64 base = (i64)blockIdx.x * BLK;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t v[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const i64 i = base + (i64)k * NT + threadIdx.x;
    v[k] = i < N ? L[i] : 0u;
  }
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const i64 i = base + (i64)k * NT + threadIdx.x;
    const unsigned long long m = __ballot(i > 0 && i < N && v[k] == (uint32_t)i);
    if (lane == 0) masks[(size_t)blockIdx.x * (BLK / 64) + k * (NT / 64) + wave] = m;
  }
}

// Roots per block, per group of 64 blocks (one work-group) and per chunk of 64 groups (added;
// cleared before) from the root bit mask, whose 512 bytes per block bound it.  A wave takes 16
// blocks, all their words in flight, and folds the 16 sums together: after the exchange over
// lane bits 5 .. 2 a lane holds a quarter of one block's count.  (With the exchange as a loop
// over its distance the sums were indexed at run time, by chains of compares, and the loads
// under their bounds: 22 us for the 22 MB of 32 x 2160 x 2560, now 15; 13 for the smallest
// stacks, now 6.)
__global__ __launch_bounds__(NT) void k_mask_counts(const unsigned long long* __restrict__ masks,
                                                    i64 nb, uint32_t* __restrict__ cnt,
                                                    uint32_t* __restrict__ groups,
                                                    uint32_t* __restrict__ chunks) {
  __shared__ uint32_t part[NT / 64];
  const int lane = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int n = (int)nb, b0 = (int)blockIdx.x * 64 + wave * 16;
  uint32_t v[16];
  unsigned long long w[16];
#pragma unroll
  for (int j = 0; j < 16; ++j)
    w[j] = (masks + (i64)min(b0 + j, n - 1) * (BLK / 64))[lane];  // (no load under a condition)
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = b0 + j < n ? (uint32_t)__popcll(w[j]) : 0u;
  auto exchange = [&](auto kc) {  // lane bit 4 k picks the upper half of the blocks
    constexpr int k = decltype(kc)::value;
    const bool up = (lane & (4 * k)) != 0;
#pragma unroll
    for (int j = 0; j < k; ++j) {
      const uint32_t keep = up ? v[j + k] : v[j], give = up ? v[j] : v[j + k];
      v[j] = keep + __shfl_xor(give, 4 * k, 64);
    }
  };
  exchange(std::integral_constant<int, 8>());
  exchange(std::integral_constant<int, 4>());
  exchange(std::integral_constant<int, 2>());
  exchange(std::integral_constant<int, 1>());
  uint32_t t = v[0];
  t += __shfl_xor(t, 1, 64);
  t += __shfl_xor(t, 2, 64);
  const int blk = b0 + (lane >> 2);  // bits 5 .. 2 of the lane: its block's bits 3 .. 0
  if ((lane & 3) == 0 && blk < n) cnt[blk] = t;
#pragma unroll
  for (int o = 4; o < 64; o <<= 1) t += __shfl_xor(t, o, 64);
  if (lane == 0) part[wave] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t g = part[0] + part[1] + part[2] + part[3];
    groups[blockIdx.x] = g;
    atomicAdd(chunks + blockIdx.x / 64, g);
  }
}

// rid[root] = 1 + rank of the root in linear order; acc[rid] = zero sums with .root = root (a
// whole 128-byte line per region, which also clears the accumulator; acc[0], the background's,
// is cleared too); *d_R and *h_R = 1 + number of roots.  One wave per block of BLK voxels: its
// first rank is the sum of the chunks, groups and blocks before it, a few words per lane, so
// no scan runs before; lane m takes root mask m of the block, a wave scan of the mask
// popcounts gives each mask's rank, and only the (few) roots are visited: each round takes one
// root per lane and writes their lines with eight lanes per line.
__global__ __launch_bounds__(NT) void k_assign_ids(const unsigned long long* __restrict__ masks,
                                                   const uint32_t* __restrict__ cnt,
                                                   const uint32_t* __restrict__ groups,
                                                   const uint32_t* __restrict__ chunks,
                                                   int n_chunks, i64 nb, uint32_t* __restrict__ rid,
                                                   RegionAcc* __restrict__ acc, i64 cap,
                                                   uint32_t* d_R, uint32_t* h_R) {
  static_assert(BLK / 64 == 64, "one mask per lane");
  static_assert(sizeof(RegionAcc) == 128 && offsetof(RegionAcc, root) == 100, "line layout");
  __shared__ uint2 ent[NT / 64][64];
  const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
  const i64 blk = (i64)blockIdx.x * (NT / 64) + wave;
  if (blk >= nb) return;  // whole waves
  if (blk == 0) {
    uint32_t t = 0u;
    for (int i = lane; i < n_chunks; i += 64) t += chunks[i];
    t = 1u + (uint32_t)wave_sum_int((int)t);
    if (lane == 0) {
      *d_R = t;
      if (h_R) *h_R = t;
      if (cap > 0) acc[0] = RegionAcc{};
    }
  }
  unsigned long long m = masks[blk * (BLK / 64) + lane];
  const i64 g = blk / 64, c = g / 64;
  uint32_t before = 0u;
  for (int i = lane; i < (int)c; i += 64) before += chunks[i];
  if (lane < (int)(g % 64)) before += groups[c * 64 + lane];
  if (lane < (int)(blk % 64)) before += cnt[g * 64 + lane];
  if (!__ballot(m != 0ull)) return;  // uniform over the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) before += __shfl_xor(before, o, 64);
  const uint32_t n = (uint32_t)__popcll(m);
  uint32_t incl = n;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  uint32_t r = 1u + before + (incl - n);
  const i64 base = blk * BLK + 64 * lane;
  const unsigned long long below = (1ull << lane) - 1ull;
  while (true) {
    const unsigned long long on = __ballot(m != 0ull);
    if (!on) break;
    if (m) {
      const uint32_t i = (uint32_t)(base + __builtin_ctzll(m));
      m &= m - 1;
      rid[i] = r;
      ent[wave][__popcll(on & below)] = make_uint2(i, r);
      ++r;
    }
    wave_lds_sync();
    const int ne = __popcll(on);
    for (int e = lane >> 3; e < ne; e += 8) {
      const uint2 v = ent[wave][e];
      if ((i64)v.y < cap)
        reinterpret_cast<uint4*>(acc + v.y)[lane & 7] =
            make_uint4(0u, (lane & 7) == 6 ? v.x : 0u, 0u, 0u);
    }
    wave_lds_sync();
  }
}

__device__ __forceinline__ uint32_t fkey(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float fdecode(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

constexpr uint32_t EMPTY = 0xFFFFFFFFu;

// Partial sums of one region, then one set of global atomics per region and work-group.
struct RunSums {
  uint32_t cnt, imax, nkey;
  unsigned long long sx, sy, sz, isum;
  double h[6], ns;
};

template <bool AVE>
__device__ __forceinline__ void flush_global(RegionAcc* a, const RunSums& v, bool has_img) {
  atomicAdd(&a->cnt, v.cnt);
  atomicAdd(&a->sx, v.sx);
  atomicAdd(&a->sy, v.sy);
  atomicAdd(&a->sz, v.sz);
#pragma unroll
  for (int k = 0; k < 6; ++k) unsafeAtomicAdd(&a->h[k], v.h[k]);
  if (AVE)
    unsafeAtomicAdd(&a->nsum, v.ns);
  else
    atomicMax(&a->nmax_key, v.nkey);
  if (has_img) {
    atomicAdd(&a->isum, v.isum);
    atomicMax(&a->imax, v.imax);
  }
}

// A region whose voxels all lie in one work-group's tiles: its sums are final after the
// work-group's fold and are stored, not added (the accumulator is zeroed beforehand).
__device__ __forceinline__ void store_final(RegionAcc* a, const RunSums& v) {
  a->sx = v.sx;
  a->sy = v.sy;
  a->sz = v.sz;
  a->isum = v.isum;
#pragma unroll
  for (int k = 0; k < 6; ++k) a->h[k] = v.h[k];
  a->nsum = v.ns;
  a->cnt = v.cnt;
  a->nmax_key = v.nkey;
  a->imax = v.imax;
}

// Per-work-group hash table in LDS keyed by region id (open addressing, LDS atomics, FP64
// for the Hessian and normalized sums).  Each occupied slot ends as one set of global
// atomics, so a region pays one set per work-group that touches it instead of one per
// voxel; a region that finds no slot in kProbes tries goes straight to the global atomics.  A
// slot whose region the caller marks `owned` (no other work-group holds any of its voxels) is
// stored instead.  (Slots are never freed, so a region that once found its kProbes slots taken
// always does: all its voxels are in the table or none.)
// Coordinates are summed relative to the work-group's origin (ox, oy, oz), with the count
// and the x and y sums packed in one 64-bit word (count: bits 0-15, x: 16-39, y: 40-63)
// and the z sums with the raw intensity sums in another (z: bits 0-23, intensity: 24-63):
// two LDS atomics instead of five.  For the < 2^16 voxels of a work-group whose offsets
// stay below 256 in x, y and z the fields cannot carry into each other.
// AVE: the normalized value's sum in place of its maximum.
template <int S, bool AVE>
struct LdsTable {
  static constexpr int kProbes = S < 32 ? S : 32;
  static constexpr uint32_t kOwn = 1u << 16;
  uint32_t key[S];
  unsigned long long cxy[S], zis[S];
  uint32_t im[S];  // maximum raw intensity; kOwn: an owned region
  typename std::conditional<AVE, double, uint32_t>::type nv[S];  // sum, or maximum key
  double h[6][S];
  uint32_t ox, oy, oz;

  __device__ void init(uint32_t x0, uint32_t y0, uint32_t z0) {
    if (threadIdx.x == 0) {
      ox = x0;
      oy = y0;
      oz = z0;
    }
    for (int t = threadIdx.x; t < S; t += blockDim.x) {
      key[t] = EMPTY;
      cxy[t] = zis[t] = 0ull;
      im[t] = 0u;
      nv[t] = 0;
#pragma unroll
      for (int k = 0; k < 6; ++k) h[k][t] = 0.0;
    }
  }

  // sums of some voxels of one region: count, coordinate offsets from the origin, raw
  // intensity sum and max, max key (or sum) of the normalized value, Hessian sums
  struct Part {
    uint32_t cnt, dx, dy, dz, isum, imax, nkey;
    double ns, h[6];
  };

  __device__ void add_part(RegionAcc* acc, uint32_t r, const Part& q, bool has_img, bool owned) {
    uint32_t slot = (r * 2654435761u) >> (32 - __builtin_ctz(S));
    bool placed = false;
    for (int probes = 0; probes < kProbes; ++probes) {
      // a key, once set, never changes: a plain read finds the region's slot, and only an
      // empty slot needs the compare-and-swap
      uint32_t k0 = __atomic_load_n(&key[slot], __ATOMIC_RELAXED);
      if (k0 == EMPTY) k0 = atomicCAS(&key[slot], EMPTY, r);
      if (k0 == EMPTY || k0 == r) { placed = true; break; }
      slot = (slot + 1) & (S - 1);
    }
    if (!placed) {
      RunSums v;
      v.cnt = q.cnt;
      v.sx = q.dx + (unsigned long long)q.cnt * ox;
      v.sy = q.dy + (unsigned long long)q.cnt * oy;
      v.sz = q.dz + (unsigned long long)q.cnt * oz;
      v.isum = q.isum;
      v.imax = q.imax;
      v.nkey = q.nkey;
      v.ns = q.ns;
#pragma unroll
      for (int k = 0; k < 6; ++k) v.h[k] = q.h[k];
      flush_global<AVE>(acc + r, v, has_img);
      return;
    }
    atomicAdd(&cxy[slot], (unsigned long long)q.cnt | ((unsigned long long)q.dx << 16) |
                              ((unsigned long long)q.dy << 40));
    atomicAdd(&zis[slot], (unsigned long long)q.dz | ((unsigned long long)q.isum << 24));
#pragma unroll
    for (int k = 0; k < 6; ++k) unsafeAtomicAdd(&h[k][slot], q.h[k]);
    if constexpr (AVE)
      unsafeAtomicAdd(&nv[slot], q.ns);
    else
      atomicMax(&nv[slot], q.nkey);
    // (owned is the same for every voxel of a region)
    atomicMax(&im[slot], q.imax | (owned ? kOwn : 0u));
  }

  __device__ void flush(RegionAcc* acc, bool has_img) {
    for (int t = threadIdx.x; t < S; t += blockDim.x) {
      const uint32_t rr = key[t];
      if (rr == EMPTY) continue;
      RunSums v;
      const unsigned long long p = cxy[t];
      v.cnt = (uint32_t)(p & 0xFFFFull);
      v.sx = ((p >> 16) & 0xFFFFFFull) + (unsigned long long)v.cnt * ox;
      v.sy = (p >> 40) + (unsigned long long)v.cnt * oy;
      const unsigned long long q = zis[t];
      v.sz = (q & 0xFFFFFFull) + (unsigned long long)v.cnt * oz;
      v.isum = q >> 24;
      v.imax = im[t] & (kOwn - 1u);
      v.nkey = 0u;
      v.ns = 0.0;
      if constexpr (AVE)
        v.ns = nv[t];
      else
        v.nkey = nv[t];
#pragma unroll
      for (int k = 0; k < 6; ++k) v.h[k] = h[k][t];
      if (im[t] & kOwn)
        store_final(acc + rr, v);
      else
        flush_global<AVE>(acc + rr, v, has_img);
    }
  }
};

// v of lane i + 1 (lane 63 keeps its own) and of lane i - 1 (lane 0 keeps its own); one
// DPP move each.  The whole wave must be active.
__device__ __forceinline__ uint32_t lane_next(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x130, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t lane_prev(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x138, 0xf, 0xf, false);
}

// Adds one voxel per lane (those with ok) to the table; the whole wave calls it together.
// hv: the six elements, nv: the normalized value, iv: the raw intensity.
template <int S, bool AVE>
__device__ __forceinline__ void fold_wave(LdsTable<S, AVE>& tab, RegionAcc* acc, uint32_t cap, bool ok,
                                          bool owned, uint32_t r, uint32_t x, uint32_t y,
                                          uint32_t z, const float* hv, float nv, uint32_t iv,
                                          bool has_img) {
  const int lane = (int)(threadIdx.x & 63);
  // Consecutive records are mostly x-neighbours in one row of one region.  Runs of
  // lanes with the same region are cut into groups of at most four; the first lane of
  // a group adds the group's sums, so the table sees one set of atomics per group.
  // (the shifts run in every lane, outside any condition: a lane whose source lane is
  // inactive would get its own value back)
  const uint32_t r_prev = lane_prev(r);
  const uint32_t ok_prev = lane_prev(ok ? 1u : 0u);
  const bool run_head = (lane == 0) | !ok | (ok_prev == 0u) | (r_prev != r);
  const unsigned long long heads = __ballot(run_head);
  const unsigned long long upto = lane == 63 ? ~0ull : (2ull << lane) - 1ull;
  const int start = 63 - __builtin_clzll(heads & upto);  // first lane of the run
  const unsigned long long later = heads & ~upto;
  const int next = later ? __builtin_ctzll(later) : 64;  // first lane of the next run
  const int last = min(next - 1, lane + 3);  // last lane of a group that starts here
  typename LdsTable<S, AVE>::Part g;
  g.cnt = 1u;
  g.dx = x - tab.ox;
  g.dy = y - tab.oy;
  g.dz = z - tab.oz;
  g.isum = g.imax = iv;
  g.nkey = AVE ? 0u : fkey(nv);
  g.ns = AVE ? (double)nv : 0.0;
#pragma unroll
  for (int k = 0; k < 6; ++k) g.h[k] = (double)hv[k];
  // the values of lanes +1, +2, +3 arrive by one-lane shifts; those past `last` are
  // left out (a shift keeps lane 63's own value, which is never inside its group)
  uint32_t sdx = g.dx, sdy = g.dy, sdz = g.dz, siv = iv, snk = g.nkey;
  float snv = nv, sh[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) sh[k] = hv[k];
#pragma unroll
  for (int o = 1; o <= 3; ++o) {
    sdx = lane_next(sdx);
    sdy = lane_next(sdy);
    sdz = lane_next(sdz);
    siv = lane_next(siv);
    if (AVE)
      snv = __uint_as_float(lane_next(__float_as_uint(snv)));
    else
      snk = lane_next(snk);
#pragma unroll
    for (int k = 0; k < 6; ++k) sh[k] = __uint_as_float(lane_next(__float_as_uint(sh[k])));
    if (lane + o <= last) {
      g.cnt += 1u;
      g.dx += sdx;
      g.dy += sdy;
      g.dz += sdz;
      g.isum += siv;
      g.imax = max(g.imax, siv);
      if (AVE)
        g.ns += (double)snv;
      else
        g.nkey = max(g.nkey, snk);
#pragma unroll
      for (int k = 0; k < 6; ++k) g.h[k] += (double)sh[k];
    }
  }
  const bool head = ((lane - start) & 3) == 0;
  if (ok && head && r < cap) tab.add_part(acc, r, g, has_img, owned);
}

// Region sums from the materialized Hessian (the per-stage interface).  A work-group takes
// one 64 x 8 x 16 tile: it reads the tile's labels (a row of 64 per wave, eight rows in
// flight), lists the positions of the labelled voxels in LDS, row by row in lane order, and
// then folds the list with full waves, as the record form below does.  Bound by its gathers:
// the label again (from L2), region id, six elements, normalized and raw intensity of the
// labelled voxels.  Voxel by voxel without the list, on 64 x 4 x 4 bricks, a wave of 64
// voxels folded about four, with one set of table atomics each and three bricks' global
// atomics per region: 783 us for 48 x 1080 x 1280 with 6 % labelled, 296 us with the list.
template <typename TH, typename TN, bool AVE>
__global__ __launch_bounds__(NT) void k_accum(const uint32_t* __restrict__ L,
                                              const uint32_t* __restrict__ rid,
                                              const TH* __restrict__ hess,
                                              const TN* __restrict__ norm,
                                              const uint16_t* __restrict__ img, RegionAcc* acc,
                                              uint32_t cap, int W, int H, int D, i64 N, int nbx,
                                              int nby) {
  constexpr int ROWS = kHessTY * kHessTZ, NWV = NT / 64, PF = 8;  // rows, waves, loads in flight
  static_assert(ROWS % (NWV * PF) == 0 && kCandTile <= 65536, "whole batches of rows");
  __shared__ LdsTable<128, AVE> tab;
  __shared__ uint16_t list[kCandTile];
  __shared__ uint32_t n_list;
  unsigned b = xcd_tile(blockIdx.x, gridDim.x);
  const int x0 = (int)(b % (unsigned)nbx) * kHessTX; b /= (unsigned)nbx;
  const int y0 = (int)(b % (unsigned)nby) * kHessTY; b /= (unsigned)nby;
  const int z0 = (int)b * kHessTZ;
  const int lane = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const i64 WH = (i64)W * H;
  const bool has_img = img != nullptr;
  if (threadIdx.x == 0) n_list = 0u;
  tab.init((uint32_t)x0, (uint32_t)y0, (uint32_t)z0);
  __syncthreads();
  for (int r0 = wave; r0 < ROWS; r0 += NWV * PF) {
    uint32_t l[PF];
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int row = r0 + NWV * j, y = y0 + row % kHessTY, z = z0 + row / kHessTY;
      l[j] = (x0 + lane < W && y < H && z < D) ? L[(i64)z * WH + (i64)y * W + x0 + lane] : 0u;
    }
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const unsigned long long on = __ballot(l[j] != 0u);
      if (!on) continue;  // uniform over the wave
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(&n_list, (uint32_t)__popcll(on));
      base = __builtin_amdgcn_readfirstlane(base);
      if (l[j] != 0u)
        list[base + (uint32_t)__popcll(on & ((1ull << lane) - 1ull))] =
            (uint16_t)(lane + kHessTX * (r0 + NWV * j));
    }
  }
  __syncthreads();
  const uint32_t n = n_list;
  if (n == 0u) return;  // uniform over the work-group
  for (uint32_t k0 = threadIdx.x - lane; k0 < n; k0 += NT) {
    const bool ok = k0 + lane < n;
    uint32_t r = 0u, x = 0u, y = 0u, z = 0u, iv = 0u;
    float hv[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, nv = 0.0f;
    if (ok) {
      const uint32_t v = list[k0 + lane];
      x = (uint32_t)x0 + v % kHessTX;
      y = (uint32_t)y0 + v / kHessTX % kHessTY;
      z = (uint32_t)z0 + v / (kHessTX * kHessTY);
      const i64 i = (i64)z * WH + (i64)y * W + x;
#pragma unroll
      for (int k = 0; k < 6; ++k) hv[k] = ld(hess, (i64)k * N + i);
      nv = ld(norm, i);
      iv = has_img ? (uint32_t)img[i] : 0u;
      r = rid[L[i]];
    }
    fold_wave(tab, acc, cap, ok, false, r, x, y, z, hv, nv, iv, has_img);
  }
  __syncthreads();
  tab.flush(acc, has_img);
}

// Region sums from the candidate records of the Hessian kernel: one work-group per
// kAccGY x kAccGZ Hessian tiles folds their records (voxel position + six elements) into
// the table, gathering the label, normalized and raw intensity of each candidate voxel; no
// pass over the non-candidate voxels.
static_assert(kAccGY * kAccGZ * kCandTile < (1 << 16) && kHessTX <= 256 &&
                  kAccGY * kHessTY <= 256 && kAccGZ * kHessTZ <= 256,
              "packed table sums: count below 2^16, offsets below 256");
// S: table slots.  G: groups of four waves; a tile's records are folded by one group, so with
// G = 4 four tiles of a work-group go side by side.
constexpr int kTileGroups = kAccGY * kAccGZ < 4 ? kAccGY * kAccGZ : 4;
static_assert(NT * kTileGroups <= 1024, "threads of a work-group");
template <typename TN, bool AVE, int S, int G>
__global__ __launch_bounds__(NT * G) void k_accum_cand(const float* __restrict__ cand,
                                                   const uint32_t* __restrict__ cand_cnt,
                                                   const uint32_t* __restrict__ rlab,
                                                   const unsigned long long* __restrict__ multi,
                                                   const uint32_t* __restrict__ rid,
                                                   const TN* __restrict__ norm,
                                                   const uint16_t* __restrict__ img,
                                                   RegionAcc* acc, uint32_t cap, uint32_t W,
                                                   uint32_t WH, unsigned nbx, unsigned nby,
                                                   unsigned nbz) {
  // work-group p takes the tiles (bx, kAccGY gy + a, kAccGZ gz + b) of the Hessian tiling;
  // a region within them is final here, others pay one set of global atomics
  constexpr int TPW = kAccGY * kAccGZ;
  const int lane = (int)(threadIdx.x & 63);
  const unsigned p = xcd_tile(blockIdx.x, gridDim.x);
  const unsigned ngy = (nby + kAccGY - 1) / kAccGY;
  const unsigned bx = p % nbx, gy = (p / nbx) % ngy, gz = p / nbx / ngy;
  uint32_t n[TPW];
  unsigned tiles[TPW], tby[TPW], tbz[TPW];
  uint32_t any = 0;
#pragma unroll
  for (int q = 0; q < TPW; ++q) {
    const unsigned by = gy * kAccGY + q % kAccGY, bz = gz * kAccGZ + q / kAccGY;
    tiles[q] = (bz * nby + by) * nbx + bx;
    tby[q] = by;
    tbz[q] = bz;
    n[q] = (by < nby && bz < nbz) ? cand_cnt[tiles[q]] : 0u;
    any |= n[q];
  }
  if (any == 0) return;  // uniform over the work-group
  __shared__ LdsTable<S, AVE> tab;
  tab.init(bx * kHessTX, gy * kAccGY * kHessTY, gz * kAccGZ * kHessTZ);
  const bool has_img = img != nullptr;
  __syncthreads();
  const int group = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / NT));
#pragma unroll
  for (int q = 0; q < TPW; ++q) {
    if (G > 1 && q % G != group) continue;  // uniform over the wave
    const float* t = cand + (size_t)tiles[q] * kCandTile * 7;
    const uint32_t* rl = rlab + (size_t)tiles[q] * kCandTile;  // each record's root label
    // tile origin: records hold the voxel's position in the tile
    const uint32_t tx0 = bx * kHessTX, ty0 = tby[q] * kHessTY, tz0 = tbz[q] * kHessTZ;
    // the whole wave walks the records together (the group sums below move values across
    // lanes); lanes past the tile's records load nothing and add nothing
    for (uint32_t b = threadIdx.x % NT - lane; b < n[q]; b += NT) {
      const uint32_t i = b + lane;
      const bool ok = i < n[q];
      uint32_t r = 0u, x = 0u, y = 0u, z = 0u, iv = 0u;
      float hv[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, nv = 0.0f;
      bool owned = false;
      if (ok) {
        const uint32_t v = __float_as_uint(t[i]);
        x = tx0 + (v % kHessTX);
        y = ty0 + (v / kHessTX) % kHessTY;
        z = tz0 + v / (kHessTX * kHessTY);
        const uint32_t idx = z * WH + y * W + x;
        rec_elements(t + kCandTile, i, hv);
        const uint32_t root = rl[i];
        r = rid[root];
        // the labeling marks every region that reaches beyond one work-group's tiles
        owned = !((multi[root >> 6] >> (root & 63)) & 1ull);
        nv = ld(norm, (i64)idx);
        iv = has_img ? (uint32_t)img[idx] : 0u;
      }
      fold_wave(tab, acc, cap, ok, owned, r, x, y, z, hv, nv, iv, has_img);
    }
  }
  __syncthreads();
  tab.flush(acc, has_img);
}

// src/3D/Eigenvalues.cu:32-94 (Eberly's closed form, FP64)
__device__ void eigen_features(const float h6[6], float* st, float* bl) {
  const double xx = h6[0], xy = h6[1], xz = h6[2], yy = h6[3], yz = h6[4], zz = h6[5];
  const double m = fmax(fmax(fmax(fabs(xx), fabs(xy)), fmax(fabs(xz), fabs(yy))),
                        fmax(fabs(yz), fabs(zz)));
  if (m < 1e-30) { *st = 0.0f; *bl = 0.0f; return; }
  const double nrm = xy * xy + xz * xz + yz * yz;
  double e0, e1, e2;
  if (nrm > 1e-30) {
    const double t = (xx + yy + zz) / 3.0;
    const double b00 = xx - t, b11 = yy - t, b22 = zz - t;
    const double den = sqrt((b00 * b00 + b11 * b11 + b22 * b22 + nrm * 2.0) / 6.0);
    const double c00 = b11 * b22 - yz * yz;
    const double c01 = xy * b22 - yz * xz;
    const double c02 = xy * yz - b11 * xz;
    double half = (b00 * c00 - xy * c01 + xz * c02) / (den * den * den) * 0.5;
    half = fmin(fmax(half, -1.0), 1.0);
    const double ang = acos(half) / 3.0;
    const double beta2 = cos(ang) * 2.0;
    const double beta0 = cos(ang + 2.094395102393195) * 2.0;
    const double beta1 = -(beta0 + beta2);
    e0 = t + den * beta0;
    e1 = t + den * beta1;
    e2 = t + den * beta2;
  } else {
    e0 = xx; e1 = yy; e2 = zz;
  }
  *st = (float)(e0 * e0 + e1 * e1 + e2 * e2);
  *bl = (float)(e2 * e2 / (e0 * e1));
}

__global__ __launch_bounds__(NT) void k_finalize(const RegionAcc* __restrict__ acc,
                                                 const uint32_t* __restrict__ d_R, i64 cap,
                                                 int is_ave, RegionOut o, i64 pitch,
                                                 const TileOut* __restrict__ tile) {
  i64 base = 0, first = 0, R = min((i64)*d_R, cap);
  if (tile) {
    if (tile->overflow) return;
    R = (i64)tile->count + 1;
    base = (i64)tile->offset - 1;  // region r >= 1 goes to slot offset + r - 1
    first = 1;
  }
  for (i64 r = (i64)blockIdx.x * NT + threadIdx.x + first; r < R; r += (i64)gridDim.x * NT) {
    if (r == 0) {
      if (o.label) o.label[0] = 0;
      if (o.size) o.size[0] = 0;
      if (o.voxels) o.voxels[0] = 0;
      if (o.cx) { o.cx[0] = 0; o.cy[0] = 0; o.cz[0] = 0; }
      if (o.st) { o.st[0] = 0; o.bl[0] = 0; }
      if (o.nrm) o.nrm[0] = 0;
      if (o.hess) for (int k = 0; k < 6; ++k) o.hess[k * pitch] = 0;
      if (o.isum) o.isum[0] = 0;
      if (o.imax) o.imax[0] = 0;
      continue;
    }
    const RegionAcc& a = acc[r];
    const i64 q = base + r;
    const uint16_t s16 = (uint16_t)a.cnt;
    const float fs = (float)s16;
    if (o.label) o.label[q] = a.root;
    if (o.size) o.size[q] = s16;
    if (o.voxels) o.voxels[q] = a.cnt;
    if (o.cx) {
      o.cx[q] = (float)a.sx / fs;
      o.cy[q] = (float)a.sy / fs;
      o.cz[q] = (float)a.sz / fs;
    }
    float h6[6];
    for (int k = 0; k < 6; ++k) h6[k] = (float)a.h[k];
    if (o.hess) for (int k = 0; k < 6; ++k) o.hess[k * pitch + q] = h6[k];
    if (o.st) eigen_features(h6, o.st + q, o.bl + q);
    if (o.nrm) o.nrm[q] = is_ave ? (float)a.nsum : fdecode(a.nmax_key);
    if (o.isum) o.isum[q] = a.isum;
    if (o.imax) o.imax[q] = (uint16_t)a.imax;
  }
}

// The arena counter is advanced by compare-and-swap: stacks of a batch may reserve their
// ranges concurrently (the branches of a batch graph).
__global__ void k_tile_reserve(const uint32_t* __restrict__ d_R, i64 acc_cap, i64 arena_cap,
                               u64* running, TileOut* t) {
  if (threadIdx.x != 0) return;
  const i64 R = (i64)*d_R;
  u64 off = __hip_atomic_load(running, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  bool over;
  for (;;) {
    over = R > acc_cap || (i64)off + (R - 1) > arena_cap;
    if (over) break;
    const u64 seen = atomicCAS((unsigned long long*)running, (unsigned long long)off,
                               (unsigned long long)(off + (u64)(R - 1)));
    if (seen == off) break;
    off = seen;  // another stack reserved first: retry from its end
  }
  t->offset = off;
  t->count = over ? 0 : (u64)(R - 1);
  t->overflow = over ? 1u : 0u;
  t->found = (uint32_t)(R - 1);
}

template <typename V>
__device__ __forceinline__ void copy_as(const void* s, void* d, u64 bytes) {
  const u64 n = bytes / sizeof(V), step = (u64)gridDim.x * NT;
  u64 i = (u64)blockIdx.x * NT + threadIdx.x;
  for (; i + 3 * step < n; i += 4 * step) {
    V v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = ((const V*)s)[i + k * step];
#pragma unroll
    for (int k = 0; k < 4; ++k) ((V*)d)[i + k * step] = v[k];
  }
  for (; i < n; i += step) ((V*)d)[i] = ((const V*)s)[i];
  if (blockIdx.x == 0 && threadIdx.x < bytes % sizeof(V)) {
    const u64 t = n * sizeof(V) + threadIdx.x;
    ((uint8_t*)d)[t] = ((const uint8_t*)s)[t];
  }
}

// gridDim.y arrays, each with the widest access its two addresses allow.  One launch in place
// of one copy per array: the copies of a short list are launches (17 of them 75 us of a
// 24 x 96 x 112 stack's 214), a long one is bound by the host link either way.
__global__ __launch_bounds__(NT) void k_copy_list(CopyList l) {
  const void* s = l.src[blockIdx.y];
  void* d = l.dst[blockIdx.y];
  const u64 bytes = l.bytes[blockIdx.y], at = (u64)s | (u64)d;
  if (at % 16 == 0)
    copy_as<uint4>(s, d, bytes);
  else if (at % 4 == 0)
    copy_as<uint32_t>(s, d, bytes);
  else if (at % 2 == 0)
    copy_as<uint16_t>(s, d, bytes);
  else
    copy_as<uint8_t>(s, d, bytes);
}

__global__ __launch_bounds__(NT) void k_fill_u64(u64* p, i64 n, u64 v) {
  for (i64 i = (i64)blockIdx.x * NT + threadIdx.x; i < n; i += (i64)gridDim.x * NT) p[i] = v;
}

}  // namespace

hipError_t launch_region_count_masks(const unsigned long long* masks, uint32_t* counts, i64 N,
                                     hipStream_t s) {
  const CountLayout c = count_layout(N);
  hipLaunchKernelGGL(k_mask_counts, dim3((unsigned)c.groups), dim3(NT), 0, s, masks, c.nb, counts,
                     counts + c.groups_off, counts + c.chunks_off);
  mark("regions/count_root_bits", s);
  return hipGetLastError();
}

hipError_t launch_region_ids(const uint32_t* labels, uint32_t* counts, unsigned long long* masks,
                             i64 N, hipStream_t s) {
  const CountLayout c = count_layout(N);
  hipLaunchKernelGGL(k_root_bits, dim3((unsigned)c.nb), dim3(NT), 0, s, labels, N, masks,
                     counts + c.chunks_off, (int)c.chunks);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  mark("regions/root_bits", s);
  return launch_region_count_masks(masks, counts, N, s);
}

hipError_t launch_region_assign(const unsigned long long* masks, const uint32_t* counts,
                                uint32_t* rid, RegionAcc* acc, i64 cap, i64 N, uint32_t* d_R,
                                uint32_t* h_R, hipStream_t s) {
  const CountLayout c = count_layout(N);
  hipLaunchKernelGGL(k_assign_ids, dim3((unsigned)((c.nb + NT / 64 - 1) / (NT / 64))), dim3(NT), 0,
                     s, masks, counts, counts + c.groups_off, counts + c.chunks_off, (int)c.chunks,
                     c.nb, rid, acc, cap, d_R, h_R);
  mark("regions/assign_ids", s);
  return hipGetLastError();
}

template <typename TH, typename TN>
hipError_t launch_region_accum(const uint32_t* labels, const uint32_t* rid, const TH* hess,
                               const TN* norm, const uint16_t* img, RegionAcc* acc, i64 cap,
                               int W, int H, int D, int is_ave, hipStream_t s) {
  const int nbx = (W + kHessTX - 1) / kHessTX, nby = (H + kHessTY - 1) / kHessTY;
  const i64 nblk = hessian_tiles(W, H, D);
  const i64 N = (i64)W * H * D;
  auto go = [&](auto ave) {
    hipLaunchKernelGGL((k_accum<TH, TN, decltype(ave)::value>), dim3((unsigned)nblk), dim3(NT), 0, s,
                       labels, rid, hess, norm, img, acc,
                       (uint32_t)std::min<i64>(cap, 0xFFFFFFFFll), W, H, D, N, nbx, nby);
  };
  if (is_ave)
    go(std::true_type{});
  else
    go(std::false_type{});
  mark("regions/accum", s);
  return hipGetLastError();
}

template <typename TN>
hipError_t launch_region_accum_cand(const float* cand, const uint32_t* cand_cnt, i64 ntiles,
                                    const uint32_t* rlab, const unsigned long long* multi,
                                    const uint32_t* rid, const TN* norm, const uint16_t* img,
                                    RegionAcc* acc, i64 cap, int W, int H, int is_ave, float blob,
                                    hipStream_t s) {
  const unsigned nbx = (unsigned)((W + kHessTX - 1) / kHessTX),
                 nby = (unsigned)((H + kHessTY - 1) / kHessTY);
  const unsigned nbz = (unsigned)(ntiles / ((i64)nbx * nby));
  const i64 ngroups =
      (i64)nbx * ((nby + kAccGY - 1) / kAccGY) * ((nbz + kAccGZ - 1) / kAccGZ);
  // Noise and blobs give a region per about 70 sxy^2 sz voxels of the narrow Gaussian, so a
  // work-group's 32768 voxels hold 470 / (sxy^2 sz) regions.  256 slots leave room for twice
  // the waves: 2111 us for 256 x 2160 x 2560 at 74 regions, 2225 with 512 slots.  Past about
  // 150 they fill up and regions pay global atomics per voxel: 61 x 900 x 1111 at 270 regions
  // takes 362 us with 256 slots, 222 with 512.
  const bool many = blob < 3.2f;
  // One group of four waves per work-group, or, where the work-groups leave the chip idle, one
  // per tile (24 x 96 x 112, 12 work-groups: 21 us with one, 16 with four;
  // 128 x 256 x 256, 256: 31, 24; 128 x 512 x 512, 1024: 65, 62; 32 x 2160 x 2560, 5400: 227, 243).
  auto go = [&](auto ave, auto slots) {
    auto launch = [&](auto groups) {
      constexpr int G = decltype(groups)::value;
      hipLaunchKernelGGL((k_accum_cand<TN, decltype(ave)::value, decltype(slots)::value, G>),
                         dim3((unsigned)ngroups), dim3(NT * G), 0, s, cand, cand_cnt, rlab, multi,
                         rid, norm, img, acc, (uint32_t)std::min<i64>(cap, 0xFFFFFFFFll),
                         (uint32_t)W, (uint32_t)((i64)W * H), nbx, nby, nbz);
    };
    if (ngroups <= 1024)
      launch(std::integral_constant<int, kTileGroups>{});
    else
      launch(std::integral_constant<int, 1>{});
  };
  using S256 = std::integral_constant<int, 256>;
  using S512 = std::integral_constant<int, 512>;
  if (is_ave)
    many ? go(std::true_type{}, S512{}) : go(std::true_type{}, S256{});
  else
    many ? go(std::false_type{}, S512{}) : go(std::false_type{}, S256{});
  mark("regions/accum_candidates", s);
  return hipGetLastError();
}

#define HDOG_INST_ACC(TH, TN)                                                                  \
  template hipError_t launch_region_accum<TH, TN>(const uint32_t*, const uint32_t*, const TH*, \
                                                  const TN*, const uint16_t*, RegionAcc*, i64,  \
                                                  int, int, int, int, hipStream_t);
HDOG_INST_ACC(float, float)
HDOG_INST_ACC(__half, __half)
HDOG_INST_ACC(__hip_bfloat16, __hip_bfloat16)
#undef HDOG_INST_ACC
#define HDOG_INST_ACCC(TN)                                                                  \
  template hipError_t launch_region_accum_cand<TN>(                                         \
      const float*, const uint32_t*, i64, const uint32_t*, const unsigned long long*,         \
      const uint32_t*, const TN*, const uint16_t*, RegionAcc*, i64, int, int, int, float,     \
      hipStream_t);
HDOG_INST_ACCC(float)
HDOG_INST_ACCC(__half)
HDOG_INST_ACCC(__hip_bfloat16)
#undef HDOG_INST_ACCC

hipError_t launch_region_finalize(const RegionAcc* acc, const uint32_t* d_R, i64 cap, i64 expect,
                                  int is_ave, RegionOut o, i64 pitch, hipStream_t s,
                                  const TileOut* t) {
  const i64 nb = std::max<i64>(1, std::min<i64>((expect + NT - 1) / NT, 1 << 16));
  hipLaunchKernelGGL(k_finalize, dim3((unsigned)nb), dim3(NT), 0, s, acc, d_R, cap, is_ave, o,
                     pitch, t);
  mark("regions/finalize", s);
  return hipGetLastError();
}

hipError_t launch_tile_reserve(const uint32_t* d_R, i64 acc_cap, i64 arena_cap, u64* running,
                               TileOut* t, hipStream_t s) {
  hipLaunchKernelGGL(k_tile_reserve, dim3(1), dim3(64), 0, s, d_R, acc_cap, arena_cap, running, t);
  return hipGetLastError();
}

hipError_t launch_copy_list(const CopyList& l, hipStream_t s) {
  if (l.n == 0) return hipSuccess;
  u64 most = 0;
  for (int k = 0; k < l.n; ++k) most = std::max(most, l.bytes[k]);
  const u64 nb = std::max<u64>(1, std::min<u64>((most + NT * 16 - 1) / (NT * 16), 64));
  hipLaunchKernelGGL(k_copy_list, dim3((unsigned)nb, (unsigned)l.n), dim3(NT), 0, s, l);
  return hipGetLastError();
}

hipError_t launch_fill_u64(u64* p, i64 n, u64 value, hipStream_t s) {
  const i64 nb = std::max<i64>(1, std::min<i64>((n + NT - 1) / NT, 1 << 16));
  hipLaunchKernelGGL(k_fill_u64, dim3((unsigned)nb), dim3(NT), 0, s, p, n, value);
  return hipGetLastError();
}

}  // namespace hdog
