// hdog_internal.hpp -- shared declarations of the HIP kernels' launchers and the
// context object behind include/hdog.h.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>
#include <algorithm>
#include <cstdint>
#include <string>

typedef int64_t i64;
typedef uint64_t u64;

namespace hdog {

constexpr int kMaxGaussRadius = 40;            // 2r+1 <= 81 taps per axis
constexpr int kMaxTaps = 2 * kMaxGaussRadius + 1;
constexpr int kMaxNormRadius = 200;
constexpr int kRootBlock = 4096;  // voxels per root-numbering block (64 mask words)
// Root counts of a volume of N voxels: per numbering block, per group of 64 blocks, per chunk
// of 64 groups (one 32-bit word each, the levels at 64-word boundaries).
struct CountLayout {
  i64 nb, groups_off, groups, chunks_off, chunks, words;
};
inline CountLayout count_layout(i64 N) {
  CountLayout c;
  c.nb = (N + kRootBlock - 1) / kRootBlock;
  c.groups = (c.nb + 63) / 64;
  c.chunks = (c.groups + 63) / 64;
  c.groups_off = (c.nb + 63) / 64 * 64;
  c.chunks_off = c.groups_off + (c.groups + 63) / 64 * 64;
  c.words = c.chunks_off + c.chunks;
  return c;
}
// word 3 of a raw buffer descriptor on gfx9-family GPUs (32-bit data format; no swizzle)
constexpr int kBufferWord3 = 0x00020000;
// cache-policy operand of a buffer store: nontemporal (streaming), as a nontemporal global
// store is compiled on gfx950
constexpr int kCachePolicyNT = 2;
// Hessian tiles: 64 x 8 outputs per work-group over 16 slices.  Candidate records are kept
// per tile in a block of kCandTile slots x 7 words: the positions, then per slot six elements.
// The tile height and the region pass's tile group are build-time choices (-DHDOG_HESS_TY,
// -DHDOG_ACC_GY / GZ; static_asserts guard the limits); 8 and 2 x 2 measured fastest.
#ifndef HDOG_HESS_TY
#define HDOG_HESS_TY 8
#endif
constexpr int kHessTX = 64, kHessTY = HDOG_HESS_TY, kHessTZ = 16;
constexpr int kCandTile = kHessTX * kHessTY * kHessTZ;
// Element words of slot i: kCandTile + 6 i (the functions below take the address of slot 0's), in
// this order (two groups of three: one 12-byte access each; the adjoint's halo rows need only
// the first).  As six planes, a row with a few
// candidates took seven stores of a few lanes each instead of three: 393 us instead of
// 366 for the Hessian pass of 32 x 2160 x 2560.
enum RecWord { kRecXY, kRecYY, kRecYZ, kRecXX, kRecXZ, kRecZZ };
struct RecHalf {
  float a, b, c;
};
__device__ __forceinline__ RecHalf rec_load(const float* el, uint32_t slot, int half) {
  return *reinterpret_cast<const RecHalf*>(el + 6 * (size_t)slot + 3 * half);
}
__device__ __forceinline__ void rec_store(float* el, uint32_t slot, int half, RecHalf v) {
  *reinterpret_cast<RecHalf*>(el + 6 * (size_t)slot + 3 * half) = v;
}
// xx, xy, xz, yy, yz, zz of a slot
__device__ __forceinline__ void rec_elements(const float* el, uint32_t slot, float (&h)[6]) {
  const RecHalf u = rec_load(el, slot, 0), v = rec_load(el, slot, 1);
  h[0] = v.a;
  h[1] = u.a;
  h[2] = v.b;
  h[3] = u.b;
  h[4] = u.c;
  h[5] = v.c;
}
// reduced-precision forms: default FP64 re-evaluation band of the leading minors (relative
// to the sum of the magnitudes of their terms)
constexpr float kDefaultMinorBand = 1e-5f;
inline i64 hessian_tiles(int W, int H, int D) {
  return (i64)((W + kHessTX - 1) / kHessTX) * ((H + kHessTY - 1) / kHessTY) *
         ((D + kHessTZ - 1) / kHessTZ);
}
// words of the candidate bit mask: one per (z, y) row of each Hessian tile, tile-major
inline i64 fg_words(int W, int H, int D) { return hessian_tiles(W, H, D) * kHessTY * kHessTZ; }
// The differentiable form keeps no blocks of kCandTile slots: the block of the tile at
// (x0, y0, z0) has a slot per voxel that the tile holds of the volume, and the blocks follow one
// another, 28 bytes per voxel for any shape.  (Whole tiles would be 16 times that for a
// single plane, more than the card has for 30000 x 30000.)
struct RecBlock {
  i64 first;  // slots before the block; its words start at 7 first
  int slots;
};
__host__ __device__ inline RecBlock rec_block(int x0, int y0, int z0, int W, int H, int D) {
  const int ex = W - x0 < kHessTX ? W - x0 : kHessTX, ey = H - y0 < kHessTY ? H - y0 : kHessTY,
            ez = D - z0 < kHessTZ ? D - z0 : kHessTZ;
  return {(i64)z0 * W * H + ez * ((i64)y0 * W + ey * (i64)x0), ex * ey * ez};
}
// Region sums from candidate records: one work-group folds kAccGY x kAccGZ Hessian tiles
// (y, z); a region inside one such group is summed by that work-group alone.
#ifndef HDOG_ACC_GY
#define HDOG_ACC_GY 2
#endif
#ifndef HDOG_ACC_GZ
#define HDOG_ACC_GZ 2
#endif
constexpr int kAccGY = HDOG_ACC_GY, kAccGZ = HDOG_ACC_GZ;

// ---- storage types of float intermediates --------------------------------------
template <typename T> __device__ __forceinline__ float ld(const T* p, i64 i);
template <> __device__ __forceinline__ float ld<float>(const float* p, i64 i) { return p[i]; }
template <> __device__ __forceinline__ float ld<__half>(const __half* p, i64 i) {
  return __half2float(p[i]);
}
template <> __device__ __forceinline__ float ld<__hip_bfloat16>(const __hip_bfloat16* p, i64 i) {
  return __bfloat162float(p[i]);
}
template <typename T> __device__ __forceinline__ T cvt(float v);
template <> __device__ __forceinline__ float cvt<float>(float v) { return v; }
template <> __device__ __forceinline__ __half cvt<__half>(float v) { return __float2half_rn(v); }
template <> __device__ __forceinline__ __hip_bfloat16 cvt<__hip_bfloat16>(float v) {
  return __float2bfloat16(v);
}

// LDS stores before, LDS loads after, in a work-group of one wave: the LDS instructions of
// all waves execute in one total order, the order in which each wave issues them, so a
// load issued after a store sees it without a wait or a barrier instruction; the fence
// only keeps the compiler from moving the accesses across it.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// Raw buffer loads of one stored element (the bits, converted by from_bits): a load whose
// byte offset lies at or beyond the descriptor's record count returns zero.
template <typename T> struct StoredBits { typedef uint16_t type; };
template <> struct StoredBits<float> { typedef uint32_t type; };
template <typename T>
__device__ __forceinline__ typename StoredBits<T>::type buf_load(__amdgpu_buffer_rsrc_t r,
                                                                 uint32_t off) {
  if constexpr (sizeof(T) == 4)
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
  else
    return __builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0);
}
template <typename T> __device__ __forceinline__ float from_bits(typename StoredBits<T>::type b);
template <> __device__ __forceinline__ float from_bits<float>(uint32_t b) {
  return __uint_as_float(b);
}
template <> __device__ __forceinline__ float from_bits<__half>(uint16_t b) {
  return __half2float(__builtin_bit_cast(__half, b));
}
template <> __device__ __forceinline__ float from_bits<__hip_bfloat16>(uint16_t b) {
  return __bfloat162float(__builtin_bit_cast(__hip_bfloat16, b));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, kBufferWord3);
}

__host__ __device__ __forceinline__ int clampi(int v, int lo, int hi) {
  return v < lo ? lo : (v > hi ? hi : v);
}

// ---- streaming (nontemporal) stores of volumes written once, read by a later kernel ----
__device__ __forceinline__ void st_nt(float* p, float v) { __builtin_nontemporal_store(v, p); }
__device__ __forceinline__ void st_nt(uint32_t* p, uint32_t v) { __builtin_nontemporal_store(v, p); }
__device__ __forceinline__ void st_nt(float2* p, float2 v) {
  __builtin_nontemporal_store(v.x, &p->x);
  __builtin_nontemporal_store(v.y, &p->y);
}
__device__ __forceinline__ void st_nt(float4* p, float4 v) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 t = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(t, reinterpret_cast<f4*>(p));
}
template <typename T> __device__ __forceinline__ void st_nt(T* p, float v) { *p = cvt<T>(v); }

// rows `bytes` apart start on whole lines (half of them)
__host__ __device__ inline bool whole_lines(i64 bytes) { return bytes % 64 == 0; }

// The lines along z as rows of n columns: a plane's columns as one row where they can be
// counted, so that no lanes idle at the rows' ends and odd rows do not shift each row's lines.
// (box_z_norm 357 -> 287 us for 64 x 1080 x 1279, 266 -> 213 for 93 x 777 x 1001; the Gaussians'
// z pass 274 -> 216 and 246 -> 178.)
struct ZColumns {
  int n, rows;
};
inline ZColumns z_columns(int W, int H) {
  const i64 WH = (i64)W * H;
  return WH < (1ll << 31) - 256 ? ZColumns{(int)WH, 1} : ZColumns{W, H};
}

// Lines of at most this many positions have passes with a thread per line that holds it in
// registers (k_minmax_shallow, k_box_shallow, k_gauss_shallow): a walk's work-group, its history
// and its barriers would serve a step of which a line fills a part.  Along z, 4000 x 5000 columns
// of one slice / 3000 x 3001 of eight, the walk and this: minima of radius 3, 344 and 61 us / 205
// and 134; box of radius 5 with the normalization, 546 and 85 / 350 and 205; Gaussians of radius 1,
// 482 and 110 / 258 and 181.  (The Gaussians' compiled walks stay: 190 us at radii 6 / 10 and
// 8 x 1500 x 2001, 220 so.)
constexpr int kShallow = 8;

// ---- tile staging -----------------------------------------------------------------
// Copies n elements global -> LDS with B independent loads in flight per lane before the
// first LDS store (a plain strided loop waits for each load in turn).
template <int B, int NTH, typename T, typename LD, typename ST>
__device__ __forceinline__ void stage_tile(int n, LD&& ldf, ST&& stf) {
  for (int base = (int)threadIdx.x; base < n; base += B * NTH) {
    T v[B];
#pragma unroll
    for (int k = 0; k < B; ++k) {
      const int e = base + k * NTH;
      if (e < n) v[k] = ldf(e);
    }
#pragma unroll
    for (int k = 0; k < B; ++k) {
      const int e = base + k * NTH;
      if (e < n) stf(e, v[k]);
    }
  }
}

// Moves rows STEP .. STEP + hist - 1 of an LDS plane to rows 0 .. hist - 1 (whole work-group;
// a barrier before and after is the caller's): the history of a walk of STEP rows per step.
template <int NTH, int STEP, int PITCH, typename T>
__device__ __forceinline__ void shift_rows(T* B, int hist) {
  for (int r0 = 0; r0 < hist; r0 += STEP) {  // source and target of one part are disjoint
    if (r0) __syncthreads();                 // the part before was read from this target
    const int n = min(STEP, hist - r0) * PITCH;
    for (int e = (int)threadIdx.x; e < n; e += NTH) B[r0 * PITCH + e] = B[(r0 + STEP) * PITCH + e];
  }
}

// ---- per-region accumulator (one 128-byte line per region) -----------------------
struct alignas(128) RegionAcc {
  unsigned long long sx, sy, sz, isum;
  double h[6];
  double nsum;
  unsigned int cnt, nmax_key, imax, root;
  unsigned int pad[2];
};

// ---- optional per-kernel event marks (profiling mode of the C-ABI) ----------------
// A launcher calls mark(name, s) after each kernel it enqueues; with profiling on the
// context points tl_prof at its event pool for the duration of the call.  A mark with
// name nullptr only starts a new interval (after a host synchronization).
struct Prof {
  static constexpr int kMax = 64;
  hipEvent_t ev[kMax];
  const char* name[kMax];
  int n = 0;
};
extern thread_local Prof* tl_prof;
inline void mark(const char* name, hipStream_t s) {
  Prof* p = tl_prof;
  if (p && p->n < Prof::kMax) {
    (void)hipEventRecord(p->ev[p->n], s);
    p->name[p->n++] = name;
  }
}

// ---- how long walks are split -------------------------------------------------------
// A walker (one wave or work-group per strip, walking an axis) may be split along its axis;
// every later segment starts with the positions of context its window needs.  Its time goes
// with (x + t) * (steps per segment), x its waves per SIMD: t is what a launch loses to waves
// that run alone (latency) and to its last, part-empty round.  The splits below take the
// segment count with the least such time; t is fitted to sweeps of 1 .. 16 segments on
// stacks from 24 x 96 x 112 to 256 x 1080 x 1280.

// Row segments of a row walker.
// t = 1.3 gives both walkers' sweeps within 10 %: norm_xy, 32 x 2160 x 2560: 914 us with two
// segments, 543 with eight, 528 with sixteen; 128 x 256 x 256: 165 us with one, 54 with seven,
// 60 with thirteen; gauss_xy there 102, 46 and 51 us with one, five and ten; on a full tile
// 2 to 4 segments are within 2 %.  A tuned launch shape `want` (1 .. 4) takes want / 2 of the
// built-in count; a negative one is a number of segments.
struct WalkShape {
  i64 strips;        // waves per segment, all planes
  int period, halo;  // segment length: a multiple of period; rows of context
};
inline void walk_segments(int H, const WalkShape& w, int* nys, int* rows, int want = 0) {
  const int wb = w.period;
  auto shape = [&](int n, int* k, int* r) {
    const int per = (H + n - 1) / n;
    *r = (per + wb - 1) / wb * wb;
    *k = (H + *r - 1) / *r;
  };
  const int most = (H + wb - 1) / wb;
  int best = 1;
  double best_cost = 0.0;
  for (int n = 1; n <= most && n <= 64; ++n) {
    int k, r;
    shape(n, &k, &r);
    const double cost = ((double)w.strips * k / 1024.0 + 1.3) * (std::min(r, H) + w.halo);
    if (n == 1 || cost < best_cost) {
      best_cost = cost;
      best = n;
    }
  }
  const int n = want > 0 ? (best * want + 1) / 2 : want < 0 ? -want : best;
  shape(std::max(1, std::min(most, n)), nys, rows);
}

// Segments of a line of L positions, each reading `halo` positions more than it writes.
// The column walkers (one thread per line) stream: two waves per SIMD already saturate the
// memory, fewer leave it idle (box_z_norm, 128 x 256 x 256, one wave per SIMD: 39 us whole,
// 29 in two segments; 64 x 512 x 512, four waves per SIMD: 47 us whole, 51 in two).  So the
// load of a launch counts as at least `alone`.  groups: launch units per segment, on `slots`
// of the chip at a time, in whole rounds when `whole` (long work-groups, one per CU).
inline void line_segments(int L, i64 groups, double slots, double alone, bool whole, int halo,
                          int* nseg, int* len) {
  int best = 1;
  double best_cost = 0.0;
  for (int n = 1; n <= 32 && n <= L; ++n) {
    const int l = (L + n - 1) / n;
    double x = (double)groups * ((L + l - 1) / l) / slots;
    if (whole) x = (double)(i64)(x + 0.9999);
    const double cost = (x > alone ? x : alone) * (l + halo);
    if (n == 1 || cost < best_cost) {
      best_cost = cost;
      best = n;
    }
  }
  *len = (L + best - 1) / best;
  *nseg = (L + *len - 1) / *len;
}

// Grid of a column walker with work-groups of 256 lines: x blocks, then the n_other lines
// of the remaining axis, then the segments.
struct LineGrid {
  unsigned blocks, nxb, no;
  int len;
};
inline LineGrid line_grid(int W, int L, i64 n_other, int halo) {
  LineGrid g;
  g.nxb = (unsigned)((W + 255) / 256);
  g.no = (unsigned)n_other;
  int nseg;
  line_segments(L, (i64)g.nxb * n_other * 4, 1024.0, 2.0, false, halo, &nseg, &g.len);
  g.blocks = (unsigned)((i64)g.nxb * n_other * nseg);
  return g;
}
struct LineAt {
  int x, other, c0, c1;  // outputs c0 .. c1-1 of the line (x, other)
};
__device__ __forceinline__ LineAt line_at_block(unsigned nxb, unsigned no, int len, int L) {
  LineAt a;
  const unsigned r = blockIdx.x / nxb;
  a.x = (int)(blockIdx.x - r * nxb) * 256 + (int)threadIdx.x;
  a.other = (int)(r % no);
  a.c0 = (int)(r / no) * len;
  a.c1 = min(L, a.c0 + len);
  return a;
}

// Work-group b of n runs on XCD b % 8 (the dispatcher deals work-groups to the 8 XCDs in
// turn, each XCD with its own L2).  Returns the logical tile for b such that every XCD
// walks one contiguous range of tiles in order: tiles that share cache lines (halo rows,
// 128-byte lines split between narrow tiles) then meet in the same L2.  A bijection of
// [0, n) for any n.
__device__ __forceinline__ unsigned xcd_tile(unsigned b, unsigned n) {
  constexpr unsigned X = 8;
  const unsigned q = n / X, r = n % X, j = b % X;
  return j * q + min(j, r) + b / X;
}

// Adds the sums of a[k] over a work-group of NT threads to out[k] (K <= 2) with one FP64
// atomic each: a handful of atomics meet at one address (one per wave over a grid sized for
// the volume serialized hundreds of thousands of them there).
constexpr int kReduceGroups = 1024;  // work-groups of a pass that is a reduction only
template <int NT, int K>
__device__ __forceinline__ void group_add(double (&a)[K], double* out) {
  __shared__ double part[NT / 64][K];
#pragma unroll
  for (int k = 0; k < K; ++k)
    for (int o = 32; o > 0; o >>= 1) a[k] += __shfl_down(a[k], o, 64);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < K; ++k) part[threadIdx.x >> 6][k] = a[k];
  __syncthreads();
  if (threadIdx.x < K) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) t += part[w][threadIdx.x];
    unsafeAtomicAdd(out + threadIdx.x, t);
  }
}

// One zero-padded central difference ((0 + hi) - lo) * 0.5 in the reference's order; the
// Hessian kernel and the region pass that recomputes the Hessian share it.
__device__ __forceinline__ float cdiff_half(float hi, float lo) {
  float s = 0.0f;
  s += hi;
  s -= lo;
  s *= 0.5f;
  return s;
}

// v rounded to the storage type T and widened back
template <typename T> __device__ __forceinline__ float round_to(float v) {
  const T t = cvt<T>(v);
  return ld(&t, 0);
}

// ---- launchers (return hipSuccess or the launch error) ----------------------------
// normalize stage; tmp1/tmp2 each hold >= 8*N bytes.  ero / dil (optional): the box means
// of the min and max filters, E and D, as separate float volumes.
// segments: row segments of the row walker (0: walk_segments' default).
template <typename TS>
hipError_t launch_normalize(const uint16_t* img, TS* norm, void* tmp1, void* tmp2,
                            float min_intensity, int W, int H, int D, int rxy, int rz,
                            hipStream_t s, float* ero = nullptr, float* dil = nullptr,
                            int segments = 0);
// Clamped box mean of float2 pairs along y (sa = W, so = W*H, n_other = D) or z (sa = W*H,
// so = W, n_other = H): the sequential sums c-r .. c+r times 1/(2r+1) of the normalization's
// y and z passes.
hipError_t launch_box_pair(const float2* src, float2* dst, int W, int L, i64 sa, i64 so,
                           i64 n_other, int r, hipStream_t s);
// DoG stage; weights: device array [4][kMaxTaps] (xy1, z1, xy2, z2); tmp1 >= 8*N bytes;
// segments as for launch_normalize
template <typename TN, typename TD>
hipError_t launch_dog(const TN* norm, TD* dog, void* tmp1, const float* weights, const int r[4], float normalizer, int W, int H, int D, hipStream_t s,
                      int segments = 0);
// how the xy walkers of the two stages split planes of W columns (and H rows), D of them
WalkShape norm_walk_shape(int rxy, int W, int D);
WalkShape gauss_walk_shape(int r1, int r2, int W, int H, int D);
// Differentiable form: separable pair of Gaussians, weights w[0..2] = x, y, z of the first and
// w[3..5] of the second, each symmetric, radii r[6]; tmp1 >= 8*N bytes.  launch_gauss_dog:
// dog = (G1 - G2) * nz; launch_gauss_dots: out[0] += <a, G1>, out[1] += <a, G2>.
hipError_t launch_gauss_dog(const float* src, void* tmp1, const float* const w[6], const int r[6],
                            float nz, float* dog, int W, int H, int D, hipStream_t s);
hipError_t launch_gauss_dots(const float* src, void* tmp1, const float* const w[6], const int r[6],
                             const float* a, double* out, int W, int H, int D, hipStream_t s);
template <typename TD, typename TH>
// hess and pd may be NULL (not written).  cand / cand_cnt (optional): per Hessian tile
// (kHessTX x kHessTY x kHessTZ, tiles x-fastest), the number of candidate voxels and their
// records: the voxel's position in the tile, lx + kHessTX (ly + kHessTY lz), then the six
// elements rounded to TH, as described at kCandTile; cand holds hessian_tiles() *
// kCandTile * 7 words.  Voxel 0 never has a record (its label is 0 whatever its mask).
// band: the FP64 re-evaluation band of the leading minors when TD or TH is a 2-byte type.
hipError_t launch_hessian(const TD* dog, TH* hess, uint8_t* pd, int W, int H, int D,
                          hipStream_t s, float* cand = nullptr, uint32_t* cand_cnt = nullptr,
                          float band = kDefaultMinorBand);
// Region numbering.  Root counts of a label volume (launch_region_ids, which also writes the
// root bit mask) or of a root bit mask whose chunk counts the labeling has cleared
// (launch_region_count_masks), in the layout of count_layout(N).
hipError_t launch_region_ids(const uint32_t* labels, uint32_t* counts, unsigned long long* masks,
                             i64 N, hipStream_t s);
hipError_t launch_region_count_masks(const unsigned long long* masks, uint32_t* counts, i64 N,
                                     hipStream_t s);
// Region ids from the root bits and the counts: rid at every root, a cleared accumulator line
// (with the root) for every id below cap, and the number of regions, 1 + the number of roots,
// in *d_R and, if given, *h_R (page-locked host memory).  Ids >= cap are skipped: the host may
// launch this and what follows before it has seen the count.
hipError_t launch_region_assign(const unsigned long long* masks, const uint32_t* counts,
                                uint32_t* rid, RegionAcc* acc, i64 cap, i64 N, uint32_t* d_R,
                                uint32_t* h_R, hipStream_t s);
template <typename TH, typename TN>
hipError_t launch_region_accum(const uint32_t* labels, const uint32_t* rid, const TH* hess,
                               const TN* norm, const uint16_t* img, RegionAcc* acc, i64 cap,
                               int W, int H, int D, int is_ave, hipStream_t s);
// Region sums from the candidate records of launch_hessian (ntiles = hessian_tiles()).
// rlab and multi come from launch_ccl_candidates: each record's root, and the roots of
// regions reaching beyond one work-group's tiles (all others are summed by one work-group
// and stored without atomics).  blob: sxy^2 sz of the narrow Gaussian, which sets how many
// regions to expect.
template <typename TN>
hipError_t launch_region_accum_cand(const float* cand, const uint32_t* cand_cnt, i64 ntiles,
                                    const uint32_t* rlab, const unsigned long long* multi,
                                    const uint32_t* rid, const TN* norm, const uint16_t* img,
                                    RegionAcc* acc, i64 cap, int W, int H, int is_ave, float blob,
                                    hipStream_t s);
struct RegionOut {
  uint32_t* label; uint16_t* size; u64* voxels; float* cx; float* cy; float* cz;
  float* st; float* bl; float* nrm; float* hess; u64* isum; uint16_t* imax;
};
// Placement of one stack's regions in a batch's region arena (device memory): regions
// 1..count of the stack occupy arena slots offset .. offset + count - 1.
struct TileOut {
  u64 offset, count;
  uint32_t overflow, found;  // found: regions of the stack, also when they did not fit
};
// With t == nullptr: region r goes to slot r, r < min(*d_R, cap).  With t: regions
// 1..t->count go to slots t->offset + r - 1 (nothing when t->overflow).  `expect`: sizes the
// grid.
hipError_t launch_region_finalize(const RegionAcc* acc, const uint32_t* d_R, i64 cap, i64 expect,
                                  int is_ave, RegionOut o, i64 pitch, hipStream_t s,
                                  const TileOut* t = nullptr);
// t->offset = *running, t->count = *d_R - 1, *running += t->count; overflow (count 0) when
// *d_R > acc_cap or the arena of arena_cap slots would overflow
hipError_t launch_tile_reserve(const uint32_t* d_R, i64 acc_cap, i64 arena_cap, u64* running,
                               TileOut* t, hipStream_t s);
hipError_t launch_fill_u64(u64* p, i64 n, u64 value, hipStream_t s);
// Copies of a region list's arrays in one launch (device memory to page-locked host memory).
struct CopyList {
  static constexpr int kMax = 18;
  const void* src[kMax];
  void* dst[kMax];
  u64 bytes[kMax];
  int n = 0;
  void add(void* d, const void* s, size_t b) {
    src[n] = s;
    dst[n] = d;
    bytes[n++] = b;
  }
};
hipError_t launch_copy_list(const CopyList& l, hipStream_t s);
// Labeling of the candidates the Hessian pass recorded (cand / cand_cnt, see
// launch_hessian): fgbits (fg_words() words) receives the candidate bit mask; P is a
// volume-sized parent array written and read at candidate voxels only; rlab (slot-aligned
// with the records) receives each record's label, the component's minimum linear index;
// roots (root_words 64-bit words, cleared here) receives the root bit of every component,
// in linear order, and multi (same size, cleared here) the root bit of every component
// with voxels outside the kAccGY x kAccGZ tile group of its root (both NULL: not wanted).
// dense: P becomes the full label volume (0 for the background).  chunk_counts (optional,
// chunks words) is cleared for launch_region_count_masks.
// rec_words: 32-bit words per record slot block (7: the Hessian pass's records; 1: the
// positions of launch_mask_records).
hipError_t launch_ccl_candidates(const float* cand, const uint32_t* cand_cnt, i64 ntiles,
                                 unsigned long long* fgbits, uint32_t* P, uint32_t* rlab,
                                 unsigned long long* roots, unsigned long long* multi,
                                 i64 root_words, bool dense, int W, int H, int D, hipStream_t s,
                                 int rec_words = 7, uint32_t* chunk_counts = nullptr,
                                 int chunks = 0);
// The candidate positions of a byte mask (pd != 0, voxel 0 excluded) in the Hessian pass's
// record layout with one word per slot (pos: hessian_tiles() * kCandTile words).
hipError_t launch_mask_records(const uint8_t* pd, float* pos, uint32_t* cand_cnt, int W, int H,
                               int D, hipStream_t s);
// differentiable blob response (soft.hip)
// 64 voxels of a row, x0 .. x0 + 63 for x0 a multiple of 64: the masked ones, and where in the
// tile's records theirs start (consecutive, in x order).  Row y of slice z has its pieces at
// ((z H + y) + 0, 1, ...) * row_pieces(W).
struct TileRow {
  unsigned long long bits;
  unsigned long long first;
};
inline int row_pieces(int W) { return (W + kHessTX - 1) / kHessTX; }
// The records of the masked voxels of a DoG volume, voxel 0 included, in blocks as rec_block
// says (7 words per voxel); the mask volume is written, or, with `rows` (one per piece of a row,
// written), decides.
hipError_t launch_hessian_records(const float* dog, uint8_t* mask, TileRow* rows, int W, int H,
                                  int D, float* cand, uint32_t* cand_cnt, hipStream_t s);
// sums[0] = loss sum, sums[1] = |M| over the records
hipError_t launch_soft_loss(const float* cand, const uint32_t* cand_cnt, const uint8_t* target,
                            int W, int H, int D, double inv_tau, double* sums, hipStream_t s);
// the records' elements become dL/dH; *sums += dL/dtau
hipError_t launch_soft_grad_h(float* cand, const uint32_t* cand_cnt, const uint8_t* target, int W,
                              int H, int D, double inv_tau, double inv_count, double* sums,
                              hipStream_t s);
// dL/ddog from those records; *dot += <dL/ddog, dog>
hipError_t launch_hessian_adjoint(const float* cand, const TileRow* rows, const float* dog,
                                  float* out, int W, int H, int D, double* dot, hipStream_t s);
hipError_t launch_zero_f64(double* p, int n, hipStream_t s);
// Differentiable form, local-contrast normalization of a float volume (clamped min / max
// and box of radius (rxy, rxy, rz)): norm, the (E, D) pairs and the window argmin / argmax
// (N each) for the backward pass; scratch 8 N words.
hipError_t launch_soft_normalize(const float* v, float* norm, float2* ed, uint32_t* arg,
                                 void* scratch, float min_int, int W, int H, int D, int rxy,
                                 int rz, hipStream_t s);
// Its adjoint: gv = dL/dv from gn = dL/dnorm (min / max by their subgradient); scratch 4 N
// words.
hipError_t launch_soft_normalize_adjoint(const float* v, const float2* ed, const uint32_t* arg,
                                         const float* gn, float* gv, void* scratch,
                                         float min_int, int W, int H, int D, int rxy, int rz,
                                         hipStream_t s);
hipError_t launch_synth(uint16_t* img, float* scratch, int W, int H, int D, u64 seed,
                        double mean0, double mean1, double sd, const double* d_blobs,
                        i64 n_blobs, hipStream_t s);

}  // namespace hdog
