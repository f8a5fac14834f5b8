// Declarations shared by the kernels of the binned backward (dfa3d_backward_binned.hip, dfa3d_backward_cells.hip):
// the bin plan and workspace the binning kernels leave behind, the work queues of the tile workgroups, and the
// small wavefront / LDS helpers they use.
#pragma once

#include "dfa3d_device.h"
#include "dfa3d_launch.h"

namespace dfa3d {

constexpr int kClasses = 8;         // work queues: one per XCD (workgroup id % 8 with round-robin placement)
constexpr int kQueueStride = 16;    // ints between queue counters: one 64-byte line each
constexpr int kQueueInts = kClasses * kQueueStride + 32;   // + room for the optional phase timers
constexpr int kBinQueries = 32;     // bin_points_in_order: queries of one (batch, head) per block step, at least
constexpr int kHistCap = 8192;      // bins of one (batch, head) that fit the LDS histogram

struct BinPlan {
  int H[DFA3D_MAX_LEVELS], W[DFA3D_MAX_LEVELS], Dd[DFA3D_MAX_LEVELS], start[DFA3D_MAX_LEVELS];
  int tiles_x[DFA3D_MAX_LEVELS], level_base[DFA3D_MAX_LEVELS];
  int bins_per_bm;     // tiles over all levels of one (batch, head); 0: see backward_without_bins
  int total_bins;      // slots * bins_per_bm
  int bins_per_class;  // total_bins / kClasses
  int class_start[kClasses + 1];   // first work item of each head class (written by the scan)
  int ty, tx;          // tile edge in pixels
  int chunk;           // points of a bin per work item that the caller asked for, 0: chunk_of() decides
  int total_chunks;    // work items (written by the scan)
  int disjoint;        // no key belongs to two levels
};

// Bins are numbered slot * bins_per_bm + tile, where the slot of (batch b, head m) puts the heads with the
// same m % 8 next to each other: class c = m % 8 owns the slots [c, c + 1) * head_groups(M) * B.  The
// binning blocks and the tile workgroups of class c run on XCD c, so everything written and read for one
// head (records, gradients per point, tiles) goes through one L2.
__host__ __device__ inline int head_groups(int M) { return (M + kClasses - 1) / kClasses; }
__host__ __device__ inline int slot_count(int B, int M) { return kClasses * head_groups(M) * B; }
__device__ __forceinline__ int slot_of(int b, int m, int B, int M) {
  return ((m % kClasses) * head_groups(M) + m / kClasses) * B + b;
}
__device__ __forceinline__ void slot_decode(int slot, int B, int M, int &b, int &m) {
  b = slot % B;
  const int hm = slot / B, G = head_groups(M);
  m = (hm % G) * kClasses + hm / G;
}

// Division of n < 2^31 by a number the host knows: multiply by ceil(2^(32 + shift) / d) - 2^32, add, shift (T. Granlund and
// P. Montgomery, Division by invariant integers using multiplication, 1994).
struct FastDiv {
  uint32_t mul, shift;
  explicit FastDiv(uint32_t d) {
    shift = 0;
    while ((1ull << shift) < d) ++shift;
    mul = (uint32_t)((((1ull << shift) - d) << 32) / d + 1);
  }
  __device__ __forceinline__ uint32_t div(uint32_t n) const { return (__umulhi(mul, n) + n) >> shift; }
};

// pixel (y, x) lies inside an H x W map (a tile's first row and column may be pixel -1)
__device__ __forceinline__ bool in_map(int y, int x, int H, int W) { return (unsigned)y < (unsigned)H && (unsigned)x < (unsigned)W; }

// Workgroup barrier that orders LDS accesses only.  __syncthreads() also waits for every global load and store the
// wavefront has in flight (one counter covers both on this part); the tile workgroups hand work to each other
// through LDS alone, so their loads may stay in flight across a barrier and their stores may drain behind it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 16 bytes per lane from a buffer to consecutive LDS addresses (`lds`: the wavefront's first byte).  Written out because
// behind the builtin the compiler waits for the data before the next LDS read of any kind; here the kernel
// waits for itself, as late as it can.  (The compiler does not count these loads: where it waits for an older one, it waits for more
// than it has to, never for less.)
__device__ __forceinline__ void load_to_lds16(rsrc_t r, const void *lds, uint32_t off) {
#ifdef __HIP_DEVICE_COMPILE__
  const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)lds);
  uint32_t kept;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
               : "=&s"(kept) : "s"(at), "v"(off), "s"(r) : "memory");
#endif
}

struct BinWorkspace {      // device pointers into the caller's workspace
  BinPlan *plan;
  int *queues;             // kClasses counters, kQueueStride ints apart; beside each, a part of the number of points counted
  int *counts;             // points per bin
  int *cursor;             // begin of each bin's segment after the scan, end after the fill
  int4 *items;             // work items: (bin, begin of its points, number of points, 1 = writes its tile alone: see bin_scan_kernel)
  int4 *geom;              // the items' bins decoded: (batch, head_level(), pixel row, pixel column of the tile's row 0)
  uint32_t *entries;       // point indices grouped by bin
  float4 *recs;            // (x, y, z, attention weight) of the same points, same order; without bins: in point order
};

// Head and level of an item in one word (a batch element's slice below 2^30 bytes leaves room for them); the batch has one
// of its own.
__device__ __forceinline__ int head_level(int m, int l) { return m * DFA3D_MAX_LEVELS + l; }
__device__ __forceinline__ int head_of(int word) { return word / DFA3D_MAX_LEVELS; }
__device__ __forceinline__ int level_of(int word) { return word % DFA3D_MAX_LEVELS; }

// Inclusive prefix sum over the 64 lanes with DPP moves: shifts by 1, 2, 4, 8 inside rows of 16 lanes, then
// lane 15 of a row to the next row, then lane 31 to the upper half.
__device__ __forceinline__ int wave_inclusive_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);   // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);   // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);   // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);   // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);   // row_bcast:15 into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);   // row_bcast:31 into rows 2 and 3
  return x;
}

// Points of a bin per work item.  Small items balance the workgroups, but the items of one bin add to its gradients
// with atomics, which the memory takes at one 64-byte piece per 50 ps (a split bin of 96 channels and depth bins:
// 20 ns per item), where a bin of one item stores them.  So: about 4096 items if that leaves large ones, else down to
// 1024 items of up to kMidChunk points, none under 256 points.  0.34 M points in 240 bins: 88 us with 4096 points per item,
// 44 with these; 0.58 M of plain attention: 230 and 60; 15.4 M: no difference.  kMidChunk, which decides from 1.3 to 5.2 M
// points, is five passes, in the middle of a flat range: the training step on two levels from 60 x 100, 3 x 10000
// queries (3.8 M points), takes 635 / 590 / 600 / 622 / 730 us with 512 / 1024 / 1280 / 2048 / 4096 points per item at
// clustered locations and 621 / 537 / 533 / 530 / 548 at uniform ones, on one level of 29 x 50 at coherent ones (2.6 M)
// 384 / 333 / 350 / 325 / 335.
constexpr int kMaxChunk = 4096, kMidChunk = 1280;
__device__ __forceinline__ int chunk_of(const BinWorkspace &ws, const BinPlan &p) {
  if (p.chunk > 0) return p.chunk;
  int n = 0;
  for (int c = 0; c < kClasses; ++c) n += ws.queues[c * kQueueStride + 1];
  return min(max(max(n >> 12, min(n >> 10, kMidChunk)), 256), kMaxChunk);
}
// Work items of a bin with c points, of equal shares (most bins have one, which saves the division); item t of k starts
// at point share_begin(c, k, t) of the bin.
__device__ __forceinline__ int items_of_bin(int c, int ch) { return c <= ch ? (c > 0 ? 1 : 0) : (c + ch - 1) / ch; }
__device__ __forceinline__ int share_begin(int c, int k, int t) { const int q = c / k; return t * q + min(t, c - q * k); }

// Optional phase clocks of the tile kernels (development builds only, -DDFA3D_TILE_TIMING).  A wavefront or two of every
// workgroup count shader-clock ticks per phase and add them to 64-bit counters that live in the padding behind the queue
// counters.  The clock is a scalar and the sums are in LDS, so that the kernel keeps the registers that it has without them.
#ifdef DFA3D_TILE_TIMING
#define TICKS_DECL(n) __shared__ unsigned long long s_ticks[n]; for (int i = threadIdx.x; i < (n); i += blockDim.x) s_ticks[i] = 0; __syncthreads(); unsigned long long ticks_last = clock64();
#define TICKS_MARK(mine, slot) do { if (mine) { const unsigned long long ticks_now = clock64(); if (threadIdx.x % kWave == 0) atomicAdd(&s_ticks[slot], ticks_now - ticks_last); ticks_last = ticks_now; } } while (0)
#define TICKS_FLUSH(mine, first, n) do { if ((mine) && threadIdx.x % kWave < (n)) atomicAdd(reinterpret_cast<unsigned long long *>(ws.queues + kClasses * kQueueStride) + (first) + threadIdx.x % kWave, s_ticks[(first) + threadIdx.x % kWave]); } while (0)
#define TT_MINE (__builtin_amdgcn_readfirstlane(threadIdx.x / kWave) == 0)
#define TT_DECL TICKS_DECL(10)
#define TT_MARK(i) TICKS_MARK(TT_MINE, i)
#define TT_FLUSH() TICKS_FLUSH(TT_MINE, 0, 10)
#else
#define TT_DECL
#define TT_MARK(i) do { } while (0)
#define TT_FLUSH() do { } while (0)
#endif

// Workgroups of this launch whose home is class c.
__device__ __forceinline__ int workgroups_of_class(int c) { return ((int)gridDim.x - c + kClasses - 1) / kClasses; }

// Thread 0 of a tile workgroup: next work item, from the queue of the workgroup's own class first and
// from the other classes once that is empty; -1 when every queue is drained.  `dealt`: items per workgroup of the class
// that are not taken from the queue.
__device__ __forceinline__ int pop_item(const BinWorkspace &ws, const BinPlan &p, int home, int &classes_done, int dealt = 0) {
  while (classes_done < kClasses) {
    const int c = (home + classes_done) % kClasses;
    const int lo = p.class_start[c], hi = p.class_start[c + 1] - dealt * workgroups_of_class(c);
    if (lo < hi) {
      // from the end: the bins of the coarsest level, which hold the most points, come last in a (batch, head)
      // and should not be what the kernel's last workgroups are left with
      const int w = hi - 1 - atomicAdd(&ws.queues[c * kQueueStride], 1);
      if (w >= lo) return w;
    }
    ++classes_done;
  }
  return -1;
}

// Thread 0's pipeline of work items: the item taken now was popped two items ago and its record requested
// one item ago, so neither the queue atomic nor the record's load is waited for.
struct ItemFetch {
  int classes_done, w_next;
  int4 rec;
  __device__ __forceinline__ int4 load(const BinWorkspace &ws, int w) const {
    return w >= 0 ? ws.items[w] : make_int4(-1, 0, 0, 0);
  }
  __device__ __forceinline__ void start(const BinWorkspace &ws, const BinPlan &p, int home) {
    classes_done = 0;
    const int w = pop_item(ws, p, home, classes_done);
    rec = load(ws, w);
    w_next = w >= 0 ? pop_item(ws, p, home, classes_done) : -1;
  }
  __device__ __forceinline__ void advance(const BinWorkspace &ws, const BinPlan &p, int home, int4 *out) {
    *out = rec;
    rec = load(ws, w_next);
    w_next = w_next >= 0 ? pop_item(ws, p, home, classes_done) : -1;
  }
};

__device__ __forceinline__ float dpp_xadd(float x, int pick) {
  const int xi = __float_as_int(x);
  int r;
  switch (pick) {
    case 0: r = __builtin_amdgcn_mov_dpp(xi, 0xB1, 0xF, 0xF, true); break;    // quad_perm [1,0,3,2]
    case 1: r = __builtin_amdgcn_mov_dpp(xi, 0x4E, 0xF, 0xF, true); break;    // quad_perm [2,3,0,1]
    case 2: r = __builtin_amdgcn_mov_dpp(xi, 0x141, 0xF, 0xF, true); break;   // row_half_mirror
    default: r = __builtin_amdgcn_mov_dpp(xi, 0x140, 0xF, 0xF, true); break;  // row_mirror
  }
  return x + __int_as_float(r);
}
template <int LPR> __device__ __forceinline__ float row_sum_f(float x) {
  if (LPR >= 2) x = dpp_xadd(x, 0);
  if (LPR >= 4) x = dpp_xadd(x, 1);
  if (LPR >= 8) x = dpp_xadd(x, 2);
  if (LPR >= 16) x = dpp_xadd(x, 3);
  if (LPR >= 32) x += __shfl_xor(x, 16, kWave);
  if (LPR >= 64) x += __shfl_xor(x, 32, kWave);
  return x;
}

// VEC consecutive floats of an LDS row, moved with one instruction (the address is VEC-float
// aligned: rows start on 16-byte boundaries and a lane's first channel is a multiple of VEC)
template <int VEC> struct LdsVec;
template <> struct LdsVec<1> {
  static __device__ __forceinline__ void ld(const float *p, float (&v)[1]) { v[0] = p[0]; }
  static __device__ __forceinline__ void st(float *p, const float (&v)[1]) { p[0] = v[0]; }
};
template <> struct LdsVec<2> {
  static __device__ __forceinline__ void ld(const float *p, float (&v)[2]) {
    const float2 t = *reinterpret_cast<const float2 *>(p);
    v[0] = t.x; v[1] = t.y;
  }
  static __device__ __forceinline__ void st(float *p, const float (&v)[2]) {
    *reinterpret_cast<float2 *>(p) = make_float2(v[0], v[1]);
  }
};
template <> struct LdsVec<4> {
  static __device__ __forceinline__ void ld(const float *p, float (&v)[4]) {
    const float4 t = *reinterpret_cast<const float4 *>(p);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
  }
  static __device__ __forceinline__ void st(float *p, const float (&v)[4]) {
    *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
  }
};
template <> struct LdsVec<8> {
  static __device__ __forceinline__ void ld(const float *p, float (&v)[8]) {
    const float4 t0 = reinterpret_cast<const float4 *>(p)[0], t1 = reinterpret_cast<const float4 *>(p)[1];
    v[0] = t0.x; v[1] = t0.y; v[2] = t0.z; v[3] = t0.w; v[4] = t1.x; v[5] = t1.y; v[6] = t1.z; v[7] = t1.w;
  }
  static __device__ __forceinline__ void st(float *p, const float (&v)[8]) {
    reinterpret_cast<float4 *>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4 *>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
  }
};
template <int VEC> __device__ __forceinline__ void lds_ld(const float *p, float (&v)[VEC]) { LdsVec<VEC>::ld(p, v); }

// The eight depth taps of a point added to an LDS tile of floats: read, add, compare-and-swap, all eight in flight
// together; a tap that met another one tries again with what it found, and after a few rounds (many points on one pixel
// and depth) the float atomic ends it.  The LDS float atomic alone retires 0.33 lanes per clock and CU, this 2.9.
// A further round swaps at all eight words again, so that all are in flight together: where a tap is done, a value that was
// found there is replaced by itself.  With a branch around each of them the round waited for one after the other: tile
// kernel 1185 -> 1153 us at the base shape, 4366 -> 4251 us dense, 117.3 -> 112.6 us small.
// Such a round costs the wavefront 60 vector instructions and eight swaps by all lanes.  The float atomic's time goes with the lanes that
// take part, so it comes at once where few are left (none, 8, 20, 40 of the active ones: tile kernel 1104, 1094, 1081, 1087 us at the base shape,
// 4092, 4052, 3981, 3987 dense, 106.6, 104.9, 103, 104.8 small), and nothing is looked at again where none is.
constexpr int kFewLanes = 32;
__device__ __forceinline__ void lds_add_taps(float *tile, const int (&at)[8], const float (&tv)[8]) {
  uint32_t *words = reinterpret_cast<uint32_t *>(tile);
  uint32_t old[8], got[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) old[j] = words[at[j]];
#pragma unroll
  for (int j = 0; j < 8; ++j) got[j] = atomicCAS(words + at[j], old[j], __float_as_uint(__uint_as_float(old[j]) + tv[j]));
  unsigned again = 0;                         // bit j: tap j is still to be added
#pragma unroll
  for (int j = 0; j < 8; ++j) again |= got[j] != old[j] ? 1u << j : 0u;
  for (int round = 0; __popcll(__ballot(again != 0)) > kFewLanes && round < 4; ++round) {      // uniform over the active lanes
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      old[j] = got[j];
      got[j] = atomicCAS(words + at[j], old[j], (again >> j & 1) ? __float_as_uint(__uint_as_float(old[j]) + tv[j]) : old[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) again &= got[j] == old[j] ? ~(1u << j) : ~0u;
  }
  if (again == 0) return;
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (again >> j & 1) atomicAdd(tile + at[j], tv[j]);
}

// The rim of a tile of (ty + 1) x (tx + 1) pixels, numbered: row 0, row ty, then the first and last pixel of the rows between.
__host__ __device__ inline int rim_pixels(int ty, int tx) { return 2 * (tx + 1) + 2 * (ty - 1); }
__device__ __forceinline__ int rim_index(int row, int col, int ty, int tx) {
  return row == 0 ? col : row == ty ? tx + 1 + col : 2 * (tx + 1) + 2 * (row - 1) + (col == 0 ? 0 : 1);
}
__device__ __forceinline__ void rim_decode(int i, int ty, int tx, int &row, int &col) {
  const int s = i - 2 * (tx + 1);
  row = s >= 0 ? 1 + (s >> 1) : i <= tx ? 0 : ty;
  col = s >= 0 ? ((s & 1) ? tx : 0) : i <= tx ? i : i - (tx + 1);
}

// What the tile kernels do when the plan has no bins: no level of the table is usable (every point is then skipped), or the
// levels have more tiles than the host sized the counters for, which takes many levels that share keys.  Every thread takes
// points of its own and adds to device memory; rare enough that only being right counts.  value == nullptr: stage 1 alone
// (grad_score_in is the scores' gradient); !FUSED: stage 2 alone.
template <typename T, bool FUSED>
__device__ __forceinline__ void backward_without_bins(
    const BinWorkspace &ws, const T *value, const T *dist, const T *score_in, const T *grad_out, const T *grad_score_in,
    void *grad_value, void *grad_dist, float *grad_loc, int gl_stride, float *grad_attn, float *grad_score_out,
    const float *grad_wu, int Md, int Mg, int B, int S, int M, int C, int D, int L, int Q, int P, int grad16) {
  const BinPlan &p = *ws.plan;
  const uint32_t LP = (uint32_t)L * P, n = (uint32_t)B * Q * M * LP;             // below 2^31
  auto add = [](void *base, bool is16, size_t e, float x) {      // a bfloat16 element: in its pair, the other one gets zero
    if (is16) atomic_add_bf16x2(static_cast<char *>(base) + (e & ~(size_t)1) * 2, (e & 1) ? 0.f : x, (e & 1) ? x : 0.f);
    else atomicAdd(static_cast<float *>(base) + e, x);
  };
  for (uint32_t gp = blockIdx.x * blockDim.x + threadIdx.x; gp < n; gp += gridDim.x * blockDim.x) {
    const float4 rec = ws.recs[gp];
    const uint32_t unit = gp / LP;
    const int l = (int)((gp - unit * LP) / P), m = (int)(unit % M), b = (int)(unit / M / Q), md = Md == 1 ? 0 : m, mg = Mg == 1 ? 0 : m;
    const Point2D<float> g = locate_2d<float>(rec.x, rec.y, p.H[l], p.W[l], p.start[l]);
    const DepthTap<float> tap = locate_depth<float>(rec.z, p.Dd[l]);
    const float a = g.inside ? rec.w : 0.f;
    float sc[4], lo[4] = {0, 0, 0, 0}, hi[4] = {0, 0, 0, 0}, s[4], gs[4], ga = 0;
    if (FUSED) {
      corner_scores<T, float>(make_rsrc(dist + (size_t)b * S * Md * D, (size_t)S * Md * D * sizeof(T)), g.key, tap, md, Md, D, sc, lo, hi);
    } else {
      for (int k = 0; k < 4; ++k) sc[k] = score_in != nullptr ? Elem<T>::ld(score_in + (size_t)gp * 4 + k) : 1.f;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool on = g.key[k] >= 0;
      const float bk = g.bil(k), w = bk * sc[k] * a;
      float dot = 0;
      if (on && value != nullptr) {
        const size_t row = (((size_t)b * S + g.key[k]) * M + m) * C;
        for (int c = 0; c < C; ++c) {
          const float go = Elem<T>::ld(grad_out + (size_t)unit * C + c);
          dot += Elem<T>::ld(value + row + c) * go;
          if (w != 0) add(grad_value, (grad16 & 1) != 0, row + c, w * go);
        }
      }
      s[k] = on ? sc[k] * dot : 0.f;
      gs[k] = on ? bk * a * dot : 0.f;
      ga += bk * s[k];
    }
    float *gl = grad_loc + (size_t)gp * gl_stride;
    gl[0] = (float)p.W[l] * a * (g.hh * (s[1] - s[0]) + g.lh * (s[2] - s[3]));
    gl[1] = (float)p.H[l] * a * (g.hw * (s[3] - s[0]) + g.lw * (s[2] - s[1]));
    if (FUSED) {
      const float gw = grad_wu != nullptr ? grad_wu[unit] * 0.25f : 0.f;
      float gz = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (g.key[k] < 0) continue;
        ga += gw * sc[k];
        gs[k] += gw * a + (grad_score_in != nullptr ? Elem<T>::ld(grad_score_in + (size_t)gp * 4 + k) : 0.f);
        if (!tap.inside) continue;
        const size_t row = (((size_t)b * S + g.key[k]) * Mg + mg) * D + tap.d0;
        if (tap.lo_ok) add(grad_dist, (grad16 & 2) != 0, row, tap.hd * gs[k]);
        if (tap.hi_ok) add(grad_dist, (grad16 & 2) != 0, row + 1, tap.ld * gs[k]);
        gz += gs[k] * (hi[k] - lo[k]);
      }
      gl[2] = gz * (float)p.Dd[l];
    } else if (grad_score_out != nullptr) {
      for (int k = 0; k < 4; ++k) grad_score_out[(size_t)gp * 4 + k] = gs[k];
    }
    if (grad_attn != nullptr) grad_attn[gp] = ga;
  }
}

// The cell-owned tile kernel (dfa3d_backward_cells.hip): rows of up to 64 channels, tiles 8 pixels wide.
constexpr int kCellTX = 8;
int cell_max_ty(int C);                // the most tile rows its walkers own
bool cell_kernel_applies(int C, int ty, int tx);
int cell_kernel_pass(int C);           // points per pass
int cell_kernel_block(int C);          // threads per workgroup
size_t cell_kernel_lds_bytes(int ty, int C, int D, int elem);
size_t cell_kernel_half_cu_lds();      // the most dynamic LDS with which two of its workgroups fit a CU
const void *cell_kernel_symbol(const BwdArgs &a, int dtype);
hipError_t launch_cell_kernel(const BwdArgs &a, int dtype, const BinWorkspace &ws, size_t lds, int grid, float *gd_heads,
                              hipStream_t stream);

}  // namespace dfa3d
