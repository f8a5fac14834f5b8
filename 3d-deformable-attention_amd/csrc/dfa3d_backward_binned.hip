// Binned backward of the fused DFA3D operator for gfx950: no floating-point atomics on device
// memory in the hot loop.
//
// Why: device-memory atomics retire at roughly 10^10 cache-line requests per second on this part,
// and the straightforward backward (bwd_attention_kernel) needs 4 row updates of grad_value and 8
// scalar updates of grad_dist per sampling point.  So the points are first binned by the image tile they
// fall in, and one workgroup per tile accumulates that tile of grad_value and grad_dist in registers and LDS and
// writes it out once: grad_value without any atomics (a lane group owns a cell, or a tile row), grad_dist taps with
// plain LDS updates made exclusive by integer operations (compare-and-swap, or tickets; LDS floating-point atomics
// only for the few taps that meet others at their address).
//
//   plan_and_clear_kernel       validates the level table, lays out the tiles (bins), clears counters
//   bin_count_kernel            points per bin (LDS histogram per block, one atomic per touched bin)
//   bin_scan_kernel             exclusive prefix over bins, work items (bin, chunk of its points); its further
//                               blocks clear gradient rows for callers that did not zero them (options.clear)
//   bin_fill_sorted_kernel      writes each point's index and record into its bin's segment, a block's points
//                               sorted by bin in LDS first so that runs of records leave together; zero
//                               gradients for points the operator skips
//                               (both turn to bin_points_in_order for more than 2048 tiles per (batch, head) or
//                               more than 2048 points per unit: every record straight to its slot)
//   cell_backward_kernel        persistent workgroups pull work items from per-XCD queues: rows of up to 64
//                               channels in whole groups of four (dfa3d_backward_cells.hip)
//   tile_backward_kernel        the same for all other rows; per item: LDS tiles of (TY+1) x (TX+1) pixels
//                               (one-pixel halo to the right/bottom, so all four corners of a point of this
//                               bin land in the tile), the phases described above the kernel, then one
//                               flush of the tile.  FUSED=false (of both): stage 2 alone
//   tile_depth_backward_kernel  stage 1 alone on the same bins
//   head_sum_kernel             a distribution shared by the heads: grad_dist per head, then summed
//   round_rows_kernel           bfloat16 gradients whose sums were formed in float (sums_in_float)
//
// A point belongs to the tile that holds its base pixel (h0, w0) = floor of its pixel coordinates, -1 <= h0 < H,
// -1 <= w0 < W; the tiles are laid over that range, so the first tile of a level starts at pixel -1.
// Semantics are those of bwd_attention_kernel (see dfa3d_backward.hip for the formulas and the
// reference lines they restate).
#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

#include "dfa3d_binned.h"

namespace dfa3d {

#ifdef DFA3D_TILE_SYNCTHREADS
#define TILE_BARRIER() __syncthreads()
#else
#define TILE_BARRIER() lds_barrier()
#endif


// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void plan_and_clear_kernel(
    BinWorkspace ws, const int64_t *__restrict__ shapes, int shape_stride, const int64_t *__restrict__ level_start, int L,
    int S, int D,
    int B, int M, int ty, int tx, int chunk, int max_bins_per_bm) {
  if (blockIdx.x == 0) {      // a lane per level, a lane per pair of levels: one after the other they took most of the launch
    static_assert(DFA3D_MAX_LEVELS * DFA3D_MAX_LEVELS == 256, "one thread per pair of levels");
    __shared__ BinPlan p;
    __shared__ int s_tiles[DFA3D_MAX_LEVELS];
    const int t = threadIdx.x;
    if (t < DFA3D_MAX_LEVELS) {
      int64_t H = 0, W = 0, Dd = 0, st = 0;
      bool ok = false;
      if (t < L) {
        H = shapes[t * shape_stride]; W = shapes[t * shape_stride + 1];
        Dd = (shape_stride > 2 && D > 0) ? shapes[t * shape_stride + 2] : 1; st = level_start[t];
        ok = H > 0 && W > 0 && st >= 0 && H <= S && W <= S && st + H * W <= (int64_t)S && Dd > 0 &&
             (D <= 0 || Dd <= D);
      }
      p.H[t] = ok ? (int)H : 0; p.W[t] = ok ? (int)W : 0; p.Dd[t] = ok ? (int)Dd : 0; p.start[t] = ok ? (int)st : 0;
      // tiles are laid over the base pixels of the points, which run from -1 (a location within half a pixel of
      // the map's upper / left edge) to H - 1 / W - 1: the first tile starts at pixel -1
      const int nx = ok ? ((int)W + tx) / tx : 0, ny = ok ? ((int)H + ty) / ty : 0;
      p.tiles_x[t] = nx;
      s_tiles[t] = nx * ny;
    }
    if (t <= kClasses) p.class_start[t] = 0;
    if (t == 0) p.disjoint = 1;
    __syncthreads();
    const int l = t / DFA3D_MAX_LEVELS, k = t % DFA3D_MAX_LEVELS;
    if (k < l && l < L && p.start[l] < p.start[k] + p.H[k] * p.W[k] && p.start[k] < p.start[l] + p.H[l] * p.W[l]) p.disjoint = 0;
    if (t == 0) {
      int base = 0;
      for (int i = 0; i < DFA3D_MAX_LEVELS; ++i) {
        p.level_base[i] = base;
        base += s_tiles[i];
      }
      // the host sized the counters for levels that share no keys: no bins (backward_without_bins) for more tiles than that
      if (base > max_bins_per_bm) base = 0;
      p.bins_per_bm = base;
      p.total_bins = base * slot_count(B, M);
      p.bins_per_class = base * head_groups(M) * B;
      p.ty = ty; p.tx = tx;
      p.chunk = chunk; p.total_chunks = 0;
    }
    __syncthreads();
    for (int i = t; i < (int)(sizeof(BinPlan) / 4); i += 256) reinterpret_cast<int *>(ws.plan)[i] = reinterpret_cast<const int *>(&p)[i];
  }
  const size_t n = (size_t)max_bins_per_bm * slot_count(B, M);
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    ws.counts[i] = 0;
    ws.cursor[i] = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x < kQueueInts) ws.queues[threadIdx.x] = 0;    // the counters and their padding
}

// bin (within one (batch, head)) of a point that the operator does not skip: the tile that holds its base pixel
// (h0, w0), -1 <= h0 < H, -1 <= w0 < W; tile (i, j) covers base pixels [i ty - 1, (i + 1) ty - 1) x [j tx - 1, ...)
__device__ __forceinline__ int bin_of(const BinPlan &p, int l, const Point2D<float> &g) {
  return p.level_base[l] + ((g.h0 + 1) / p.ty) * p.tiles_x[l] + (g.w0 + 1) / p.tx;
}

// The bins of the work items decoded (batch, head, level, pixel of the tile's row 0), so that the tile workgroups
// need no divisions to find their tile: block `block` of `n_blocks` of a fill launch takes its share of the items.
__device__ __forceinline__ void decode_items(const BinWorkspace &ws, int B, int M, int L, int block, int n_blocks) {
  const BinPlan &p = *ws.plan;
  const int n = p.total_chunks;
  for (int w = block * (int)blockDim.x + (int)threadIdx.x; w < n; w += n_blocks * (int)blockDim.x) {
    const int bin = ws.items[w].x;
    const int bm = bin / p.bins_per_bm, local = bin - bm * p.bins_per_bm;
    int b, m, l = 0;
    slot_decode(bm, B, M, b, m);
    while (l + 1 < L && local >= p.level_base[l + 1]) ++l;
    const int tile = local - p.level_base[l];
    ws.geom[w] = make_int4(b, head_level(m, l), (tile / p.tiles_x[l]) * p.ty - 1, (tile % p.tiles_x[l]) * p.tx - 1);
  }
}

// Count and fill come in two forms, of which the plan's number of bins decides.  The sorted one (few enough bins and points per
// unit): a block sorts its kStage points by bin in LDS and writes each bin's run of records to consecutive addresses, so a
// wavefront's store touches a handful of lines instead of 64.  bin_points_in_order: every point's record goes straight to
// its slot.  Both live in one launch each of count and fill: as launches of their own that stepped aside the others took
// 4.6 us each (2 x 40000 queries of plain attention: 9 of 418 us a training step).
constexpr int kSortedBins = 2048;   // bins of one (batch, head) the sorted fill holds counters for
constexpr int kStage = 2048;        // points a block of the sorted fill stages (1024: 0.39 ms, 4096: 0.36 ms against 0.32 ms)
constexpr int kFillThreads = 1024;  // 256 / 512 threads: 0.49 / 0.38 ms
__host__ __device__ inline bool sorted_fill_applies(int bins_per_bm, int LP) { return bins_per_bm <= kSortedBins && LP <= kStage; }
constexpr size_t kSortedFillLds = (size_t)kStage * (16 + 4 + 2) + (size_t)(3 * kSortedBins + 1) * 4;

// this block's part of the total that chunk_of() reads
__device__ __forceinline__ int *counted_points(const BinWorkspace &ws) { return &ws.queues[(blockIdx.x % kClasses) * kQueueStride + 1]; }

// a fill launch's share of the records when there are no bins
__device__ __forceinline__ void fill_in_point_order(const BinWorkspace &ws, const float *loc, int loc_stride, const float *attn, size_t n) {
  for (size_t gp = (size_t)blockIdx.x * blockDim.x + threadIdx.x; gp < n; gp += (size_t)gridDim.x * blockDim.x) {
    const float *at = loc + gp * loc_stride;
    ws.recs[gp] = make_float4(at[0], at[1], loc_stride > 2 ? at[2] : 0.f, attn != nullptr ? attn[gp] : 0.f);
  }
}

// MODE 0: count.  MODE 1: fill (needs the scanned cursor).  For 1 to hist_cap bins s_hist holds [0, nb): counts, then for
// MODE 1 [nb, 2 nb): segment bases.
template <int MODE>
__device__ __forceinline__ void bin_points_in_order(
    const BinWorkspace &ws, const float *__restrict__ loc, int loc_stride, const float *__restrict__ attn,
    float *__restrict__ grad_loc, int gl_stride, float *__restrict__ grad_attn, float *__restrict__ grad_score,
    int B, int M, int L, int Q, int P, int hist_cap, int *s_hist) {
  const BinPlan &p = *ws.plan;
  const int nb = p.bins_per_bm;
  if (nb == 0) {
    if (MODE == 1) fill_in_point_order(ws, loc, loc_stride, attn, (size_t)B * Q * M * L * P);
    return;
  }
  const bool use_lds = nb <= hist_cap;
  if (MODE == 1) decode_items(ws, B, M, L, blockIdx.x, gridDim.x);
  // Blocks of work: a thread a point, kBinQueries queries at least.  head = block % M: with the round-robin placement of
  // workgroups on the 8 XCDs and a grid that is a multiple of 8, the records of one (batch, head) are written through one
  // XCD's L2.
  const int q_block = max(kBinQueries, kFillThreads / (L * P)), q_blocks = (Q + q_block - 1) / q_block, n_blocks = B * M * q_blocks;
  int counted = 0;
  for (int blk = blockIdx.x; blk < n_blocks; blk += gridDim.x) {
  __syncthreads();                          // the previous block's LDS histogram is no longer in use
  const int m = blk % M, rest = blk / M;
  const int qb = rest % q_blocks, b = rest / q_blocks;
  const int bm = slot_of(b, m, B, M);
  const int LP = L * P;
  const int q0 = qb * q_block, nq = min(q_block, Q - q0);
  const int npts = nq * LP;
  int *gcount = ws.counts + (size_t)bm * nb;
  int *gcursor = ws.cursor + (size_t)bm * nb;

  if (use_lds) {
    for (int i = threadIdx.x; i < nb * (MODE == 1 ? 2 : 1); i += blockDim.x) s_hist[i] = 0;
    __syncthreads();
  }
  // pass 1: histogram of this block's points; the fill keeps the bins of its first kKept rounds in registers
  constexpr int kKept = 4;
  int kept[kKept];
#pragma unroll
  for (int k = 0; k < kKept; ++k) kept[k] = -1;
  int round = 0;
  for (int i = threadIdx.x; i < npts; i += blockDim.x, ++round) {
    const int qi = i / LP, lp = i - qi * LP, l = lp / P;
    const size_t gp = ((size_t)(b * (size_t)Q + q0 + qi) * M + m) * LP + lp;
    const Point2D<float> g = locate_2d<float>(loc[gp * loc_stride], loc[gp * loc_stride + 1], p.H[l], p.W[l], p.start[l]);
    if (g.inside && p.tiles_x[l] > 0) {
      const int bin = bin_of(p, l, g);
      if (MODE == 1) {
#pragma unroll
        for (int k = 0; k < kKept; ++k) kept[k] = round == k ? bin : kept[k];
      }
      ++counted;
      if (use_lds) atomicAdd(&s_hist[bin], 1);
      else if (MODE == 0) atomicAdd(&gcount[bin], 1);
    } else if (MODE == 1) {
      // skipped by the operator: all its gradients are zero, and no tile will visit it
      for (int i = 0; i < gl_stride; ++i) grad_loc[gp * gl_stride + i] = 0;
      if (grad_attn != nullptr) grad_attn[gp] = 0;
      if (grad_score != nullptr) {
        for (int k = 0; k < 4; ++k) grad_score[gp * 4 + k] = 0;
      }
    }
  }
  if (use_lds) {
    __syncthreads();
    for (int i = threadIdx.x; i < nb; i += blockDim.x) {
      const int c = s_hist[i];
      if (c > 0) {
        if (MODE == 0) atomicAdd(&gcount[i], c);
        else s_hist[nb + i] = atomicAdd(&gcursor[i], c);     // reserve a run of the bin's segment
      }
      if (MODE == 1) s_hist[i] = 0;                          // reused as the running rank
    }
    __syncthreads();
  }
  if (MODE == 1) {
    // pass 2: place the points
    round = 0;
    for (int i = threadIdx.x; i < npts; i += blockDim.x, ++round) {
      const int qi = i / LP, lp = i - qi * LP, l = lp / P;
      const size_t gp = ((size_t)(b * (size_t)Q + q0 + qi) * M + m) * LP + lp;
      int bin = -1;
      if (round < kKept) {
#pragma unroll
        for (int k = 0; k < kKept; ++k) bin = round == k ? kept[k] : bin;
      } else {
        const Point2D<float> g = locate_2d<float>(loc[gp * loc_stride], loc[gp * loc_stride + 1], p.H[l], p.W[l], p.start[l]);
        if (g.inside && p.tiles_x[l] > 0) bin = bin_of(p, l, g);
      }
      if (bin >= 0) {
        const int slot = use_lds ? s_hist[nb + bin] + atomicAdd(&s_hist[bin], 1) : atomicAdd(&gcursor[bin], 1);
        ws.entries[slot] = (uint32_t)gp;
        ws.recs[slot] = make_float4(loc[gp * loc_stride], loc[gp * loc_stride + 1],
                                    loc_stride > 2 ? loc[gp * loc_stride + 2] : 0.f, attn != nullptr ? attn[gp] : 0.f);
      }
    }
  }
  }
  if (MODE == 0) {
    counted = wave_inclusive_scan(counted);
    if (threadIdx.x % kWave == kWave - 1) atomicAdd(counted_points(ws), counted);
  }
}

// What the count and the sorted fill divide by, per point: points of a unit and of a level, tile edges.
struct BinDivs { FastDiv lp, p, ty, tx; };
// The plan's tables in LDS: the bin of a point otherwise takes a chain of three reads of device memory after its location has
// come, and four divisions by numbers the compiler does not know.  15.36 M points: count 89 -> 52 us, fill 195 -> 153 us.
// Both kernels then had a block per turn, which waited for its points, then for its reservations.  As many blocks as the
// chip holds, with the next turn's points on their way while they work on one: count 52 -> 36 us (184 MB read, 5.1 TB/s), fill
// 153 -> 144 us, and 141 since it waits for its reservations only when it has staged the points (553 MB moved, 3.9 TB/s, where a
// copy reaches 4.7); 61 M clustered points count 281 -> 134 us, fill 595 -> 575.
struct BinTable {
  int H[DFA3D_MAX_LEVELS], W[DFA3D_MAX_LEVELS], base[DFA3D_MAX_LEVELS], tiles_x[DFA3D_MAX_LEVELS];
  __device__ __forceinline__ void load(const BinPlan &p) {     // the caller's barrier
    const int l = threadIdx.x;
    if (l < DFA3D_MAX_LEVELS) { H[l] = p.H[l]; W[l] = p.W[l]; base[l] = p.level_base[l]; tiles_x[l] = p.tiles_x[l]; }
  }
  // bin of a location on level l, or -1 when the operator skips it (see bin_of)
  __device__ __forceinline__ int bin(int l, float x, float y, const BinDivs &d) const {
    const Point2D<float> g = locate_2d<float>(x, y, H[l], W[l], 0);
    const int across = tiles_x[l];
    if (!g.inside || across <= 0) return -1;
    return base[l] + (int)d.ty.div(g.h0 + 1) * across + (int)d.tx.div(g.w0 + 1);
  }
};

// Count: turns of kStage points, as many blocks per (batch, head) as the chip holds, each with one set of counters for all its
// turns: an atomic per bin that it touched.  (Tried: runs of consecutive turns per block, 39 us and slow where the locations
// come from memory; counters for all heads and turns of consecutive points, 41 us, and too many blocks that meet on the
// counters of a batch element, 5 -> 10 us for 0.3 M points.)
__global__ __launch_bounds__(kFillThreads, 8) void bin_count_kernel(
    BinWorkspace ws, const float *__restrict__ loc, int loc_stride, int B, int M, int L, int Q, int P, int q_turn,
    int parts, int hist_cap, BinDivs divs) {
  __shared__ int s_cnt[kSortedBins], s_inside;
  __shared__ BinTable tab;
  extern __shared__ int s_hist[];                                // hist_cap counters, where the host cannot rule them out
  const BinPlan &p = *ws.plan;
  const int nb = p.bins_per_bm;
  const int LP = L * P;
  if (nb == 0) return;
  if (!sorted_fill_applies(nb, LP)) {
    bin_points_in_order<0>(ws, loc, loc_stride, nullptr, nullptr, 0, nullptr, nullptr, B, M, L, Q, P, hist_cap, s_hist);
    return;
  }
  const int tid = threadIdx.x;
  const int m = blockIdx.x % M, rest = blockIdx.x / M;
  const int part = rest % parts, b = rest / parts;
  constexpr int kPer = kStage / kFillThreads;
  // a thread's points keep their place within the unit from turn to turn
  int qi[kPer], lp[kPer], lv[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const int i = tid + kFillThreads * r;
    qi[r] = divs.lp.div(i); lp[r] = i - qi[r] * LP; lv[r] = divs.p.div(lp[r]);
  }
  float x[kPer], y[kPer];
  auto ask = [&](int q0) {                                       // always asked for, so that the waits can be counted
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const int q = min(q0 + qi[r], Q - 1);
      const float *at = loc + (((size_t)b * Q + q) * M + m) * LP * loc_stride + (size_t)lp[r] * loc_stride;
      x[r] = at[0]; y[r] = at[1];
    }
  };
  ask(part * q_turn);
  for (int i = tid; i < nb; i += kFillThreads) s_cnt[i] = 0;
  if (tid == 0) s_inside = 0;
  tab.load(p);
  __syncthreads();
  int counted = 0;                                               // of this wavefront
  auto tally = [&](int q0, const float (&tx)[kPer], const float (&ty)[kPer]) {
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const int bin = qi[r] < q_turn && q0 + qi[r] < Q ? tab.bin(lv[r], tx[r], ty[r], divs) : -1;
      if (bin >= 0) atomicAdd(&s_cnt[bin], 1);
      counted += __popcll(__ballot(bin >= 0));
    }
  };
  int q0 = part * q_turn;
  for (; q0 + parts * q_turn < Q; q0 += parts * q_turn) {
    float tx[kPer], ty[kPer];
#pragma unroll
    for (int r = 0; r < kPer; ++r) { tx[r] = x[r]; ty[r] = y[r]; }
    ask(q0 + parts * q_turn);
    tally(q0, tx, ty);
  }
  tally(q0, x, y);
  if (tid % kWave == 0) atomicAdd(&s_inside, counted);
  __syncthreads();
  if (tid == 0) atomicAdd(counted_points(ws), s_inside);
  int *gcount = ws.counts + (size_t)slot_of(b, m, B, M) * nb;
  for (int i = tid; i < nb; i += kFillThreads) {
    const int c = s_cnt[i];
    if (c > 0) atomicAdd(&gcount[i], c);
  }
}

__global__ __launch_bounds__(kFillThreads, 8) void bin_fill_sorted_kernel(
    BinWorkspace ws, const float *__restrict__ loc, int loc_stride, const float *__restrict__ attn,
    float *__restrict__ grad_loc, int gl_stride, float *__restrict__ grad_attn, float *__restrict__ grad_score,
    int B, int M, int L, int Q, int P, int q_blocks, int hist_cap, BinDivs divs) {
  extern __shared__ __align__(16) unsigned char s_raw[];        // kSortedFillLds bytes
  __shared__ BinTable tab;
  uint4 *s_rec = reinterpret_cast<uint4 *>(s_raw);               // staged records, grouped by bin
  uint32_t *s_gp = reinterpret_cast<uint32_t *>(s_rec + kStage);
  uint16_t *s_bin = reinterpret_cast<uint16_t *>(s_gp + kStage);
  int *s_cnt = reinterpret_cast<int *>(s_bin + kStage);                                   // points of this block per bin
  int *s_lofs = s_cnt + kSortedBins;                             // first staged slot of each bin; [kSortedBins]: total
  int *s_shift = s_lofs + kSortedBins + 1;                       // from a staged slot to the record's place, by bin
  __shared__ int s_wave[kFillThreads / kWave];
  const BinPlan &p = *ws.plan;
  const int nb = p.bins_per_bm;
  const int LP = L * P;
  if (nb == 0 || !sorted_fill_applies(nb, LP)) {
    bin_points_in_order<1>(ws, loc, loc_stride, attn, grad_loc, gl_stride, grad_attn, grad_score, B, M, L, Q, P, hist_cap, reinterpret_cast<int *>(s_raw));
    return;
  }
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  constexpr int kPer = kStage / kFillThreads;                             // points per thread
  // A turn takes every q_blocks-th query, not a run of consecutive ones.  Consecutive queries of a model look at
  // neighbouring places (BEV pillars in raster order), so a run of them would put a compact patch of points into a
  // bin, the tile kernel's passes (consecutive points of a bin) would each hit a few tile rows only, and its rows
  // phase, which takes as long as the longest row's list, would slow down (measured: 1.74 -> 2.25 ms).  Spread
  // over the whole query range a turn's points cover each bin's area evenly, whatever the order of the queries.
  int qi[kPer], level[kPer];                                       // a thread's points keep their place within the turn
  uint32_t from[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const int i = tid + kFillThreads * r;
    qi[r] = (int)divs.lp.div(i) * q_blocks;
    const int lp = i - (int)divs.lp.div(i) * LP;
    level[r] = divs.p.div(lp);
    from[r] = (uint32_t)qi[r] * (uint32_t)M * (uint32_t)LP + (uint32_t)lp;
  }
  struct Turn { int b, m, qb; };
  auto turn_of = [&](unsigned blk) {                                  // head = block % M, as in bin_points_in_order
    Turn t;
    t.m = blk % M;
    const unsigned rest = blk / M;
    t.qb = rest % q_blocks; t.b = rest / q_blocks;
    return t;
  };
  uint4 rec[kPer];
  auto first_of = [&](const Turn &t) { return (uint32_t)(((size_t)t.b * Q + t.qb) * M + t.m) * LP; };
  auto ask = [&](const Turn &t) {                                // always asked for, so that the waits can be counted
    const uint32_t first = first_of(t);
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const uint32_t gp = t.qb + qi[r] < Q ? first + from[r] : first;
      const float *at = loc + (size_t)gp * loc_stride;
      rec[r] = make_uint4(__float_as_uint(at[0]), __float_as_uint(at[1]), loc_stride > 2 ? __float_as_uint(at[2]) : 0u,
                          attn != nullptr ? __float_as_uint(attn[gp]) : 0u);
    }
  };
  const unsigned n_turns = (unsigned)(B * M * q_blocks);
  if (blockIdx.x < n_turns) ask(turn_of(blockIdx.x));
  for (int i = tid; i < nb; i += kFillThreads) s_cnt[i] = 0;
  tab.load(p);
  decode_items(ws, B, M, L, blockIdx.x, gridDim.x);
  __syncthreads();
  auto turn = [&](unsigned blk, auto more) {                     // more: another one follows
    const Turn t = turn_of(blk);
    int *gcursor = ws.cursor + (size_t)slot_of(t.b, t.m, B, M) * nb;
    // 1. every point: its bin and its rank among this turn's points of that bin
    int bin[kPer], rank[kPer];
    uint4 mine[kPer];
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      mine[r] = rec[r];
      bin[r] = -1; rank[r] = 0;
      if (t.qb + qi[r] >= Q) continue;
      bin[r] = tab.bin(level[r], __uint_as_float(mine[r].x), __uint_as_float(mine[r].y), divs);
      if (bin[r] >= 0) {
        rank[r] = atomicAdd(&s_cnt[bin[r]], 1);
      } else {
        // skipped by the operator: all its gradients are zero, and no tile will visit it
        const size_t at = first_of(t) + from[r];
        for (int c = 0; c < gl_stride; ++c) grad_loc[at * gl_stride + c] = 0;
        if (grad_attn != nullptr) grad_attn[at] = 0;
        if (grad_score != nullptr) {
          for (int k = 0; k < 4; ++k) grad_score[at * 4 + k] = 0;
        }
      }
    }
    lds_barrier();
    int base[kSortedBins / kFillThreads];
    // 2. runs: reserve this turn's run in every touched bin's segment; staged order = bins in order (exclusive scan).
    // The next turn's points are asked for behind the reservations, and have come when this turn's are written out.
    {
      constexpr int kBinsPer = kSortedBins / kFillThreads;                  // consecutive bins per thread
      int c[kBinsPer], sum = 0;
#pragma unroll
      for (int j = 0; j < kBinsPer; ++j) {
        const int i = tid * kBinsPer + j;
        c[j] = i < nb ? s_cnt[i] : 0;
        s_cnt[i] = 0;
        sum += c[j];
        base[j] = 0;
        if (c[j] > 0) base[j] = atomicAdd(&gcursor[i], c[j]);
      }
      if constexpr (decltype(more)::value) ask(turn_of(blk + gridDim.x));
      const int inc = wave_inclusive_scan(sum);
      if (lane == kWave - 1) s_wave[wave] = inc;
      lds_barrier();
      int run = inc - sum;
      for (int w = 0; w < wave; ++w) run += s_wave[w];
#pragma unroll
      for (int j = 0; j < kBinsPer; ++j) {
        const int i = tid * kBinsPer + j;
        s_lofs[i] = run;
        run += c[j];
      }
      if (tid == kFillThreads - 1) s_lofs[kSortedBins] = run;                   // number of staged points
    }
    lds_barrier();
    // 3. stage
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      if (bin[r] >= 0) {
        const int pos = s_lofs[bin[r]] + rank[r];
        s_rec[pos] = mine[r];
        s_gp[pos] = first_of(t) + from[r];
        s_bin[pos] = (uint16_t)bin[r];
      }
    }
    // the reservations are only now waited for
#pragma unroll
    for (int j = 0; j < kSortedBins / kFillThreads; ++j) {
      const int i = tid * (kSortedBins / kFillThreads) + j;
      s_shift[i] = base[j] - s_lofs[i];
    }
#pragma unroll
    for (int r = 0; r < kPer && decltype(more)::value; ++r) asm volatile("" : "+v"(rec[r].x), "+v"(rec[r].y), "+v"(rec[r].z), "+v"(rec[r].w));      // waits for them here: behind the stores it would wait for those too
    lds_barrier();
    // 4. write out: consecutive staged slots of one bin go to consecutive addresses
    const int total = s_lofs[kSortedBins];
    for (int i = tid; i < total; i += kFillThreads) {
      const int dst = s_shift[s_bin[i]] + i;
      ws.recs[dst] = *reinterpret_cast<const float4 *>(&s_rec[i]);
      ws.entries[dst] = s_gp[i];
    }
  };
  unsigned blk = blockIdx.x;
  for (; blk + gridDim.x < n_turns; blk += gridDim.x) turn(blk, std::true_type());
  if (blk < n_turns) turn(blk, std::false_type());
}

// What the tile kernel adds to instead of storing, cleared for a caller that did not zero grad_value / grad_dist
// (options.clear).  The tile kernel stores the rows of the pixels that lie inside a tile (not on its first row or
// column, which are the halo of its upper and left neighbours) when that tile's points fit one work item, no key belongs
// to two levels and the kernel stores rows of that length (ClearArgs::stores); every other row of the two tensors only
// ever receives atomic adds, or nothing: pixels on tile rims, pixels of tiles without points or with several work items,
// keys outside every level.
// A lane decides for one (batch, key, head) row; the wavefront then clears its rows together, 16 bytes per lane on
// consecutive addresses (the heads of a key share their fate, so whole lines go out).  Every division but that by the
// map's width is by a number the host knows (FastDiv; a batch element has fewer than 2^28 rows): with the compiler's, in 64 bits
// for the row and one per 16 bytes cleared, the vector units were what bound the launch.  The launch with the scan: base shape (1.48 M
// rows of 128 and 256 bytes, 0.13 GB cleared) 40 -> 25 us; 3 levels from 37 x 67, 59 k rows of 80 and 236 bytes, 17 -> 7 us.
struct ClearRows {                  // one tensor's rows
  char *base;                       // nullptr: not this one
  int row_bytes, pieces;            // a row in pieces of 16 bytes, or of 4 where rows are not made of those
  FastDiv div_pieces;
  ClearRows(void *at, int bytes) : base(static_cast<char *>(at)), row_bytes(bytes), pieces((bytes & 15) ? bytes >> 2 : bytes >> 4), div_pieces((uint32_t)(pieces > 0 ? pieces : 1)) {}
  __device__ __forceinline__ void clear(size_t first_row, int rows, uint64_t which, int lane) const {
    char *dst = base + first_row * row_bytes;
    const bool wide = (row_bytes & 15) == 0;                 // uniform
#pragma unroll 1
    for (int c = lane; c < rows * pieces; c += kWave) {
      if (!(which >> div_pieces.div(c) & 1)) continue;
      if (wide) *reinterpret_cast<uint4 *>(dst + (size_t)c * 16) = make_uint4(0, 0, 0, 0);
      else *reinterpret_cast<uint32_t *>(dst + (size_t)c * 4) = 0;
    }
  }
};
struct ClearArgs {
  ClearRows value, dist;
  int B, M, L;
  int stores;                       // the tile kernel stores what its item alone writes (else it adds everything)
  int rows_of_b, rows_of_wave;      // rows of a batch element (S M); rows a wavefront takes at a time: 64, or 16 where that leaves CUs idle
  FastDiv div_waves, div_m, div_ty, div_tx;      // by a batch element's turns of a wavefront; heads; tile edges
};
__device__ __forceinline__ void clear_unstored(const BinWorkspace &ws, const ClearArgs &ca, unsigned block, unsigned n_blocks) {
  __shared__ int4 s_level[DFA3D_MAX_LEVELS];                 // first key, keys, width, tiles across
  __shared__ int s_base[DFA3D_MAX_LEVELS];
  const BinPlan &p = *ws.plan;
  if (threadIdx.x < DFA3D_MAX_LEVELS) {
    const int l = threadIdx.x;
    s_level[l] = make_int4(p.start[l], p.H[l] * p.W[l], p.W[l], p.tiles_x[l]);
    s_base[l] = p.level_base[l];
  }
  __syncthreads();
  const int nb = p.bins_per_bm, TY = p.ty, TX = p.tx, ch = chunk_of(ws, p);
  const bool decide = ca.stores != 0 && nb > 0 && p.disjoint != 0;
  const int lane = threadIdx.x % kWave;
  const unsigned waves_of_b = (unsigned)((ca.rows_of_b + ca.rows_of_wave - 1) / ca.rows_of_wave);
  const unsigned step = n_blocks * (blockDim.x / kWave), n = waves_of_b * (unsigned)ca.B;
  for (unsigned w = block * (blockDim.x / kWave) + threadIdx.x / kWave; w < n; w += step) {
    const unsigned b = ca.div_waves.div(w);
    const int first = (int)(w - b * waves_of_b) * ca.rows_of_wave, i = first + lane;
    bool mine = lane < ca.rows_of_wave && i < ca.rows_of_b;
    if (mine && decide) {
      const int s = (int)ca.div_m.div(i), m = i - s * ca.M;
      for (int l = 0; l < ca.L; ++l) {
        const int4 lv = s_level[l];
        const int local = s - lv.x;
        if (local >= 0 && local < lv.y) {
          const int y = (int)((unsigned)local / (unsigned)lv.z), x = local - y * lv.z;
          const int ty = (int)ca.div_ty.div(y + 1), tx = (int)ca.div_tx.div(x + 1);      // the first tile starts at pixel -1
          if (ty * TY != y + 1 && tx * TX != x + 1) {
            const int c = ws.counts[slot_of((int)b, m, ca.B, ca.M) * nb + s_base[l] + ty * lv.w + tx];
            mine = items_of_bin(c, ch) != 1;                // exactly one work item stores this row
          }
          break;
        }
      }
    }
    const uint64_t which = __ballot(mine);
    const size_t row = (size_t)b * ca.rows_of_b + first;
    if (ca.value.base != nullptr) ca.value.clear(row, ca.rows_of_wave, which, lane);
    if (ca.dist.base != nullptr) ca.dist.clear(row, ca.rows_of_wave, which, lane);
  }
}

// The first `scan_blocks` blocks scan, 1024 bins each (in turns if there are more bins than that).  A block needs no
// word from the blocks before it: it adds up the counts of all bins before its own (16 bytes a load, a few loads per
// thread for tens of thousands of bins), which is cheaper than one workgroup walking all bins and writing every work item from
// one CU.  Further blocks, if any, clear the gradient rows that need it meanwhile (both kinds only read the counts);
// the kernel is held to 64 registers so that two such workgroups fit a CU.
// An item's last word says whether it alone writes the pixels inside its tile, which the tile kernels then store: it holds
// all the points of its bin, and no key belongs to two levels (a level table may give one map to several levels; their
// tiles then meet on the same rows, and all of them add).
__global__ __launch_bounds__(1024, 8) void bin_scan_kernel(BinWorkspace ws, ClearArgs ca, int scan_blocks) {
  if ((int)blockIdx.x >= scan_blocks) {
    clear_unstored(ws, ca, blockIdx.x - scan_blocks, gridDim.x - scan_blocks);
    return;
  }
  __shared__ int s_pts[16], s_chk[16], s_bp[16], s_bc[16];
  const int n = ws.plan->total_bins, ch = chunk_of(ws, *ws.plan), per_class = ws.plan->bins_per_class;
  const int sole = ws.plan->disjoint;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  for (int base = (int)blockIdx.x * 1024; base < n; base += scan_blocks * 1024) {
    // points and work items of the bins before this block's: every thread its share, summed over the wavefront
    int bp = 0, bc = 0;
    const int4 *quads = reinterpret_cast<const int4 *>(ws.counts);      // base is a multiple of 1024
#pragma unroll 4
    for (int i = threadIdx.x; i < base / 4; i += 1024) {
      const int4 c = quads[i];
      bp += c.x + c.y + c.z + c.w;
      bc += items_of_bin(c.x, ch) + items_of_bin(c.y, ch) + items_of_bin(c.z, ch) + items_of_bin(c.w, ch);
    }
    bp = __builtin_amdgcn_readlane(wave_inclusive_scan(bp), kWave - 1);
    bc = __builtin_amdgcn_readlane(wave_inclusive_scan(bc), kWave - 1);
    const int i = base + (int)threadIdx.x;
    const int c = i < n ? ws.counts[i] : 0, k = items_of_bin(c, ch);
    const int ip = wave_inclusive_scan(c), ic = wave_inclusive_scan(k);      // inclusive scans within the wavefront
    __syncthreads();                                         // the tables of the turn before have been read
    if (lane == kWave - 1) { s_pts[wave] = ip; s_chk[wave] = ic; }
    if (lane == 0) { s_bp[wave] = bp; s_bc[wave] = bc; }
    __syncthreads();
    int run_p = ip - c, run_c = ic - k;
#pragma unroll 4
    for (int w = 0; w < 16; ++w) {
      run_p += s_bp[w] + (w < wave ? s_pts[w] : 0);
      run_c += s_bc[w] + (w < wave ? s_chk[w] : 0);
    }
    if (i < n) {
      if (i % per_class == 0) ws.plan->class_start[i / per_class] = run_c;
      ws.cursor[i] = run_p;
      if (k == 1) ws.items[run_c] = make_int4(i, run_p, c, sole);
      for (int t = 0, begin = 0; k > 1 && t < k; ++t) {
        const int end = share_begin(c, k, t + 1);
        ws.items[run_c + t] = make_int4(i, run_p + begin, end - begin, 0);
        begin = end;
      }
      if (i == n - 1) {
        ws.plan->total_chunks = run_c + k;
        ws.plan->class_start[kClasses] = run_c + k;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------
// Tile workgroups.
//
// A work item is one bin (image tile of one batch element, head and level) and up to `chunk` of
// its points.  The points are taken PP (128 or 256) at a time, one per thread:
//   phase A  thread = point: geometry, depth taps, corner weights; every corner becomes a task
//            (tile row, weight, point slot); the point's grad_out row is staged in LDS
//   sort     tasks are grouped by tile row (counting sort in LDS, integer counters)
//   rows     a group of LPR lanes owns a tile row: it loads the value row once, then for each of the
//            row's tasks takes the staged grad_out row, leaves the dot product for phase C and
//            accumulates weight * grad_out in registers; the row sum is added to the LDS tile with a
//            plain read-modify-write (nobody else touches that row during the pass)
//   phase C  thread = point: per-point gradients from the four dots; the 8 grad_dist taps of a point go
//            to the LDS tile (first taker of an address: plain update, later ones: atomics)
// After the item's last pass the tile is flushed to memory once: stores for the inner rows of an item that
// writes its tile alone, atomic adds for the rest (the chunks of one bin overlap, the rims of neighbouring bins do, and
// so do the tiles of levels that share keys).
// ---------------------------------------------------------------------------------------


struct TileLds {      // offsets (in 4-byte words) into the dynamic LDS block
  int gv, gd, gstage, tasks, dots, cnt, offs, goff, total;
};
__host__ __device__ inline TileLds tile_lds_layout(int ty, int tx, int C, int D, int PP) {
  TileLds o;
  const int R = (ty + 1) * (tx + 1);
  o.gv = 0;
  o.gd = o.gv + R * C;
  o.gstage = (o.gd + R * D + 3) & ~3;              // 16-byte aligned rows
  o.tasks = (o.gstage + (PP + 1) * C + 1) & ~1;    // PP staged rows and one row of zeros; 8-byte records
  o.dots = o.tasks + PP * 4 * 2;
  o.cnt = o.dots + PP * 4 + kWave;                 // + one scrap word per lane
  o.offs = o.cnt + R;
  o.goff = o.offs + R + 1;
  o.total = o.goff + PP;
  return o;
}


struct RowTask { float w; uint32_t who; };   // who = point slot * 4 + corner: the index of the task's dot


// FUSED: both stages (depth scores recomputed from dist, grad_dist and the z gradient produced).
// !FUSED: stage 2 alone: scores read from score_in, their gradient written to grad_score_out, no
// depth tile (the launcher passes D = 0), grad_loc has gl_stride components of which x, y are written.
template <typename T, int VEC, int LPR, bool FUSED>
__global__ __launch_bounds__(512, 4) void tile_backward_kernel(
    BinWorkspace ws, const T *__restrict__ value, const T *__restrict__ dist, const T *__restrict__ score_in,
    const T *__restrict__ grad_out, const T *__restrict__ grad_score_in,
    void *__restrict__ grad_value, void *__restrict__ grad_dist, float *__restrict__ grad_loc, int gl_stride,
    float *__restrict__ grad_attn, float *__restrict__ grad_score_out, const float *__restrict__ grad_wu, int Md,
    int Mg, int B, int S, int M, int C, int D, int L, int Q, int P, int PP, int grad16) {
  // grad16: bit 0 = grad_value is bfloat16, bit 1 = grad_dist is bfloat16 (else float)
  // Md: heads stored in dist (M, or 1 = shared by all heads); Mg: heads of the grad_dist buffer written here
  constexpr int RPI = kWave / LPR;                  // row groups per wavefront
  extern __shared__ __align__(16) float smem[];
  __shared__ int4 s_item;

  const BinPlan &p = *ws.plan;
  const int nb = p.bins_per_bm;
  if (__builtin_expect(nb == 0, 0)) {
    backward_without_bins<T, FUSED>(ws, value, dist, score_in, grad_out, grad_score_in, grad_value, grad_dist, grad_loc, gl_stride,
                                    grad_attn, grad_score_out, grad_wu, Md, Mg, B, S, M, C, D, L, Q, P, grad16);
    return;
  }
  const int TY = p.ty, TX = p.tx, TW = TX + 1, R = (TY + 1) * TW;
  const TileLds lay = tile_lds_layout(TY, TX, C, D, PP);
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int n_thr = blockDim.x, n_waves = n_thr / kWave;
  const int kGroups = n_waves * RPI;                   // row groups in the workgroup
  const int stage_per_wave = PP / n_waves;             // grad_out rows each wavefront stages
  float *gv = smem + lay.gv, *gd = smem + lay.gd, *gstage = smem + lay.gstage, *dots = smem + lay.dots;
  RowTask *tasks = reinterpret_cast<RowTask *>(smem + lay.tasks);
  int *cnt = reinterpret_cast<int *>(smem + lay.cnt), *offs = reinterpret_cast<int *>(smem + lay.offs);
  uint32_t *goff = reinterpret_cast<uint32_t *>(smem + lay.goff);
  const int group = wave * RPI + lane / LPR, cl = lane % LPR;
  const int passes = (C + VEC * LPR - 1) / (VEC * LPR);
  const int LP = L * P;
  const int my_set = tid / PP, slot = tid % PP;         // the workgroup has at least 2 PP threads; halves 0 and 1
                                                        // own alternate passes, further threads none

  for (int i = tid; i < R * (C + D); i += n_thr) smem[i] = 0;   // gv and gd are adjacent
  for (int i = tid; i < C; i += n_thr) gstage[PP * C + i] = 0;  // the row that idle lanes of the rows phase read
  TT_DECL

  ItemFetch fetch;
  if (tid == 0) fetch.start(ws, p, blockIdx.x % kClasses);
  int pass_tag = 0x5EED0000;                               // changes with every pass of this workgroup
  for (;;) {
    // ---- next work item: (bin, chunk of its points), in bin order
    TILE_BARRIER();
    if (tid == 0) fetch.advance(ws, p, blockIdx.x % kClasses, &s_item);
    TILE_BARRIER();
    const int4 item = s_item;
    const int bin = item.x, seg = item.y, n_item = item.z;
    if (bin < 0) break;                                   // queues drained: every wave leaves
    TT_MARK(0);
    const int bm = bin / nb, local = bin - bm * nb;
    int b, m;
    slot_decode(bm, B, M, b, m);
    int l = 0;
    while (l + 1 < L && local >= p.level_base[l + 1]) ++l;
    const int tile = local - p.level_base[l];
    const int H = p.H[l], W = p.W[l], Dd = p.Dd[l], start = p.start[l];
    const int y0 = (tile / p.tiles_x[l]) * TY - 1, x0 = (tile % p.tiles_x[l]) * TX - 1;      // pixel of the tile's row 0

    const rsrc_t value_r = make_rsrc(value + (size_t)b * S * M * C, (size_t)S * M * C * sizeof(T));
    const int md = Md == 1 ? 0 : m;
    const rsrc_t dist_r = make_rsrc(FUSED ? dist + (size_t)b * S * Md * D : nullptr, FUSED ? (size_t)S * Md * D * sizeof(T) : 0);
    const rsrc_t go_r = make_rsrc(grad_out + (size_t)b * Q * M * C, (size_t)Q * M * C * sizeof(T));

    // Per-point state of the pass a thread owns.  With twice as many threads as points per pass the two halves
    // of the workgroup own alternate passes: while one half runs phase C of pass i, the other runs phase A of
    // pass i + 1 (two dependent memory round trips), which then costs no time of its own.
    // What phase C needs of a point, kept small: it stays in registers through the rows phase, where every
    // register counts.  Complements (1 - lh, ...) are formed again where they are used.
    uint32_t st_gp = 0;                                 // index of the point
    float st_a = 0, sc[4], hl[4];                       // weight; corner scores; upper minus lower depth tap per corner
    float st_lh = 0, st_lw = 0, st_ld = 0;              // fractional parts along h, w, depth
    int st_d0 = 0;                                      // lower depth bin
    uint32_t st_tr01 = 0xFFFFFFFFu, st_tr23 = 0xFFFFFFFFu;   // tile rows of the corners, 16 bits each, 0xFFFF = none
    unsigned st_bits = 0;            // bit k: corner k inside the map; 4: depth inside; 5, 6: lower, upper tap exists; 7: live
    // ---------------- phase A: one thread per point ----------------
    auto phase_a = [&](int base, int (&tr)[4], float (&wk)[4]) {
      for (int i = slot; i < R; i += PP) cnt[i] = 0;
      const bool live = slot < n_item - base;
      Point2D<float> g;
      DepthTap<float> tap;
      size_t gp = 0;
      float a = 0;
      unsigned on_bits = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) { sc[k] = 0; hl[k] = 0; g.key[k] = -1; }
      g.inside = false; g.lh = g.lw = g.hh = g.hw = 0; g.h0 = g.w0 = 0;
      tap.inside = tap.lo_ok = tap.hi_ok = false; tap.d0 = 0; tap.ld = tap.hd = 0;
      uint32_t my_goff = kNoRow;
      if (live) {
        gp = ws.entries[seg + base + slot];
        const float4 rec = ws.recs[seg + base + slot];
        const size_t unit = gp / LP;
        a = rec.w;
        g = locate_2d<float>(rec.x, rec.y, H, W, start);
        if (FUSED) {
          tap = locate_depth<float>(rec.z, Dd);
          {
            float lo[4], hi[4];
            corner_scores<T, float, true>(dist_r, g.key, tap, md, Md, D, sc, lo, hi);
#pragma unroll
            for (int k = 0; k < 4; ++k) hl[k] = hi[k] - lo[k];
          }
        } else {
          const T *si = score_in + gp * 4;
#pragma unroll
          for (int k = 0; k < 4; ++k) sc[k] = score_in != nullptr ? Elem<T>::ld(si + k) : 1.f;
        }
        my_goff = (uint32_t)((unit - (size_t)b * Q * M) * C * sizeof(T));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (g.key[k] >= 0) {
            on_bits |= 1u << k;
            const int ry = g.h0 + (k >= 2 ? 1 : 0) - y0, rx = g.w0 + ((k == 1 || k == 2) ? 1 : 0) - x0;
            if (ry >= 0 && ry <= TY && rx >= 0 && rx <= TX) {
              tr[k] = ry * TW + rx;
              wk[k] = g.bil(k) * sc[k] * a;
            }
          }
        }
      }
      goff[slot] = my_goff;
      st_gp = (uint32_t)gp; st_a = a; st_lh = g.lh; st_lw = g.lw; st_ld = tap.ld; st_d0 = tap.d0;
      st_tr01 = ((uint32_t)tr[0] & 0xFFFFu) | ((uint32_t)tr[1] << 16);
      st_tr23 = ((uint32_t)tr[2] & 0xFFFFu) | ((uint32_t)tr[3] << 16);
      st_bits = on_bits | (tap.inside ? 16u : 0u) | (tap.lo_ok ? 32u : 0u) | (tap.hi_ok ? 64u : 0u) | (live ? 128u : 0u);
    };
    // The loop is rotated: a turn runs phase C of the previous pass on the half that owns it and, meanwhile,
    // phase A of this pass on the other half; then sort and rows of this pass on everybody.  One extra turn
    // finishes the last pass.
    for (int pass_idx = 0;; ++pass_idx) {                        // uniform over the workgroup
      const int base = pass_idx * PP;
      const bool has = base < n_item;
      const bool mine = has && my_set == (pass_idx & 1);         // this thread's half owns the pass
      const bool prev_mine = pass_idx > 0 && my_set == ((pass_idx - 1) & 1);
      int tr[4] = {-1, -1, -1, -1};                               // of this pass: used until its tasks are placed
      float wk[4] = {0, 0, 0, 0};
      if (mine) phase_a(base, tr, wk);

      // ---------------- phase C: per-point gradients, grad_dist taps into the LDS tile ----------------
      // LDS floating-point atomics retire about 0.3 lanes per clock per CU on this part, integer ones more
      // than twenty times as many.  So every tap first swaps this pass's tag into a word that belongs to its
      // tile address (the words live where the grad_out rows were staged: the rows phase is over).  Whoever
      // gets something else than the tag back is the first at that address and adds at once with a plain
      // read-modify-write: nobody else touches the address before the barrier below.  Only the others (under
      // a fifth of the taps at 256 points per pass) use the floating-point atomic, after that barrier.  Stale
      // words cannot do harm: one that happens to equal the tag just sends its address's taps to the atomics.
      int *tickets = reinterpret_cast<int *>(gstage);
      const bool ticketed = FUSED && R * D <= PP * C;         // uniform over the workgroup
      ++pass_tag;
      // the previous pass's points as phase A left them
      Point2D<float> g;
      DepthTap<float> tap;
      g.lh = st_lh; g.lw = st_lw; g.hh = 1 - st_lh; g.hw = 1 - st_lw;
      tap.inside = (st_bits & 16u) != 0; tap.lo_ok = (st_bits & 32u) != 0; tap.hi_ok = (st_bits & 64u) != 0;
      tap.d0 = st_d0; tap.ld = st_ld; tap.hd = tap.inside ? 1 - st_ld : 0.f;
      int trc[4] = {(int)(int16_t)(st_tr01 & 0xFFFFu), (int)(int16_t)(st_tr01 >> 16),
                    (int)(int16_t)(st_tr23 & 0xFFFFu), (int)(int16_t)(st_tr23 >> 16)};
      const unsigned on_bits = st_bits & 15u;
      const bool live = (st_bits & 128u) != 0;
      const float a = st_a;
      const size_t gp = st_gp;
      float gs[4] = {0, 0, 0, 0};
      unsigned first_mask = 0;              // bit 2k / 2k+1: this thread took the first ticket of corner k's lower / upper tap
      if (prev_mine && live) {
        float s[4], ga = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float dk = dots[slot * 4 + k];
          const bool on = on_bits >> k & 1;
          const float bk = g.bil(k);
          gs[k] = on ? bk * a * dk : 0.f;
          s[k] = on ? sc[k] * dk : 0.f;
          ga += bk * s[k];
        }
        const float gx = (float)W * a * (g.hh * (s[1] - s[0]) + g.lh * (s[2] - s[3]));
        const float gy = (float)H * a * (g.hw * (s[3] - s[0]) + g.lw * (s[2] - s[1]));
        float *gl = grad_loc + gp * gl_stride;
        if (!FUSED) { gl[0] = gx; gl[1] = gy; }
        if (FUSED) {
          if (grad_score_in != nullptr) {
            const T *gi = grad_score_in + gp * 4;
#pragma unroll
            for (int k = 0; k < 4; ++k) gs[k] += Elem<T>::ld(gi + k);
          }
          if (grad_wu != nullptr) {       // weight_update = sum over points of attn * mean corner score
            const float gw = grad_wu[gp / LP] * 0.25f;
            ga += gw * (sc[0] + sc[1] + sc[2] + sc[3]);
#pragma unroll
            for (int k = 0; k < 4; ++k) gs[k] += gw * a;
          }
          float gz = 0;
          int at8[8];                               // tile address of each of the eight taps, -1 = no tap
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const bool taps = trc[k] >= 0 && tap.inside && gs[k] != 0;
            const int at = trc[k] * D + tap.d0;
            at8[2 * k] = (taps && tap.lo_ok) ? at : -1;
            at8[2 * k + 1] = (taps && tap.hi_ok) ? at + 1 : -1;
            if (!taps) {
              gs[k] = ((on_bits >> k & 1) && tap.inside) ? gs[k] : 0.f;      // no taps below for this corner
              if (!(trc[k] >= 0 && tap.inside)) trc[k] = -1;
            }
            gz += ((on_bits >> k & 1) && tap.inside) ? gs[k] * hl[k] : 0.f;
          }
          gl[0] = gx; gl[1] = gy; gl[2] = gz * (float)Dd;      // one 12-byte store
          grad_attn[gp] = ga;                       // all stores before the tile updates: they complete slowly
          if (ticketed) {
            // the eight swaps back to back, then the reads of the first takers, then their writes: one LDS
            // round trip each instead of one per tap (a thread's eight addresses are all different)
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (at8[j] >= 0 && atomicExch(&tickets[at8[j]], pass_tag) != pass_tag) first_mask |= 1u << j;
            float cur8[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) cur8[j] = (first_mask >> j & 1) ? gd[at8[j]] : 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (first_mask >> j & 1) gd[at8[j]] = cur8[j] + ((j & 1) ? tap.ld : tap.hd) * gs[j >> 1];
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (at8[j] >= 0) atomicAdd(gd + at8[j], ((j & 1) ? tap.ld : tap.hd) * gs[j >> 1]);
          }
        } else if (grad_score_out != nullptr) {
          float *go4 = grad_score_out + gp * 4;
#pragma unroll
          for (int k = 0; k < 4; ++k) go4[k] = gs[k];
          grad_attn[gp] = ga;
        } else {
          grad_attn[gp] = ga;
        }
      }
      if (ticketed && pass_idx > 0) {
        TILE_BARRIER();                                 // plain updates done before the atomic ones start
        if (prev_mine && live) {
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            if (trc[k] >= 0 && gs[k] != 0) {
              float *dst = gd + trc[k] * D + tap.d0;
              if (tap.lo_ok && !(first_mask & (1u << (2 * k)))) atomicAdd(dst, tap.hd * gs[k]);
              if (tap.hi_ok && !(first_mask & (2u << (2 * k)))) atomicAdd(dst + 1, tap.ld * gs[k]);
            }
          }
        }
      }
      TT_MARK(5);
      if (!has) break;
      TILE_BARRIER();                                   // counters cleared, goff visible
      TT_MARK(1);
      int rank[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) rank[k] = (mine && tr[k] >= 0) ? atomicAdd(&cnt[tr[k]], 1) : 0;
      // stage the grad_out rows of this wavefront's 64 points (lanes over channels)
      for (int pass = 0; pass < passes; ++pass) {
        const int chan = (pass * LPR + cl) * VEC;
        const uint32_t chan_off = chan < C ? (uint32_t)(chan * sizeof(T)) : kNoChan;
#pragma unroll 4
        for (int j = 0; j < stage_per_wave; j += RPI) {
          // a wavefront with fewer rows to stage than row groups (short passes, few lanes per row) leaves the
          // groups beyond its share idle: their slots belong to the next wavefront, or lie past the last one
          const int sub = j + lane / LPR;
          const bool slot_ok = sub < stage_per_wave;
          const int slot = wave * stage_per_wave + min(sub, stage_per_wave - 1);
          float gg[VEC];
          RowVec<T, float, VEC>::ld(go_r, goff[slot] + chan_off, gg);
          if (slot_ok && chan < C) LdsVec<VEC>::st(gstage + slot * C + chan, gg);
        }
      }
      TILE_BARRIER();                                   // counts complete
      TT_MARK(2);
      // Exclusive prefix of the row counters.  Every wavefront that places tasks computes it, two rows per
      // lane and 128 rows per step, and writes the same numbers: it can go on with its own copy without
      // waiting for the others.
      if (mine) {                                        // whole wavefronts
        int run = 0;
        for (int r0 = 0; r0 < R; r0 += 2 * kWave) {
          const int r = r0 + 2 * lane;
          const int c0 = r < R ? cnt[r] : 0, c1 = r + 1 < R ? cnt[r + 1] : 0;
          const int inc = wave_inclusive_scan(c0 + c1);
          if (r < R) offs[r] = run + inc - c0 - c1;
          if (r + 1 < R) offs[r + 1] = run + inc - c1;
          run += __builtin_amdgcn_readlane(inc, kWave - 1);
        }
        if (lane == 0) offs[R] = run;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (!mine) {
        } else if (tr[k] >= 0) {
          RowTask t;
          t.w = wk[k];
          t.who = (uint32_t)(slot * 4 + k);
          tasks[offs[tr[k]] + rank[k]] = t;
        } else {
          dots[slot * 4 + k] = 0;                        // no row will write this dot
        }
      }
      TILE_BARRIER();                                   // tasks grouped by row, grad_out rows staged
      TT_MARK(3);

      // ---------------- rows: one group of LPR lanes per tile row ----------------
      for (int pass = 0; pass < passes; ++pass) {
        const int chan = (pass * LPR + cl) * VEC;
        const bool chan_ok = chan < C;
        const uint32_t chan_off = chan_ok ? (uint32_t)(chan * sizeof(T)) : kNoChan;
        float v_next[VEC];
        {
          const int r = group;
          const int y = y0 + r / TW, x = x0 + r % TW;
          const bool ld_ok = r < R && offs[min(r, R - 1) + 1] > offs[min(r, R - 1)] && in_map(y, x, H, W);
          RowVec<T, float, VEC>::ld(value_r, (ld_ok ? (uint32_t)(((start + y * W + x) * M + m) * C * (int)sizeof(T)) : kNoRow) + chan_off, v_next);
        }
        for (int r0 = 0; r0 < R; r0 += kGroups) {        // uniform over the workgroup
          const int r = r0 + group;
          const bool row_ok = r < R;
          const int beg = row_ok ? offs[r] : 0;
          const int n_r = row_ok ? offs[r + 1] - beg : 0;
          int n_max = n_r;                               // longest list among this wavefront's groups
#pragma unroll
          for (int off = LPR; off < kWave; off <<= 1) n_max = max(n_max, __shfl_xor(n_max, off, kWave));
          const int y = y0 + r / TW, x = x0 + r % TW;
          const bool pix_ok = row_ok && n_r > 0 && in_map(y, x, H, W);
          float v[VEC], acc[VEC];
#pragma unroll
          for (int i = 0; i < VEC; ++i) { v[i] = v_next[i]; acc[i] = 0; }
          {                                              // value row of this group's next round
            const int rn = r + kGroups;
            const int yn = y0 + rn / TW, xn = x0 + rn % TW;
            const bool ld_ok = rn < R && offs[min(rn, R - 1) + 1] > offs[min(rn, R - 1)] && in_map(yn, xn, H, W);
            RowVec<T, float, VEC>::ld(value_r, (ld_ok ? (uint32_t)(((start + yn * W + xn) * M + m) * C * (int)sizeof(T)) : kNoRow) + chan_off, v_next);
          }
          if (n_max == 0) continue;                      // wave-uniform
          // tasks in flight per group: registers decide (measured: 4 with four channels per lane, 1 with eight;
          // one more costs 1 % .. 10 % of the kernel's time)
          constexpr int UT = VEC >= 8 ? 1 : 4;
          const RowTask *row_tasks = tasks + beg;
          const int last_task = PP * 4 - 1 - beg;         // reads past a short list stay inside the array
          const float *g_lane = gstage + (chan_ok ? chan : 0);
          const int dummy = PP * 4 + lane;                // private scrap word for lanes with nothing to report
          for (int t0 = 0; t0 < n_max; t0 += UT) {
            RowTask tk[UT];
            float gg[UT][VEC], part[UT];
            // A group whose list is shorter than the wavefront's longest one idles on a task of weight zero that
            // points at the row of zeros: nothing another point staged (a non-finite gradient, say) and no
            // stale word is ever multiplied in.
#pragma unroll
            for (int j = 0; j < UT; ++j) {
              const RowTask t = row_tasks[min(t0 + j, last_task)];
              const bool on = t0 + j < n_r;
              tk[j].w = on ? t.w : 0.f;
              tk[j].who = on ? t.who : (uint32_t)(PP * 4);
            }
#pragma unroll
            for (int j = 0; j < UT; ++j) lds_ld<VEC>(g_lane + (tk[j].who >> 2) * C, gg[j]);
#pragma unroll
            for (int j = 0; j < UT; ++j) {
              part[j] = 0;
#pragma unroll
              for (int i = 0; i < VEC; ++i) part[j] += v[i] * gg[j][i];
            }
#pragma unroll
            for (int j = 0; j < UT; ++j) part[j] = row_sum_f<LPR>(part[j]);
#pragma unroll
            for (int j = 0; j < UT; ++j) {
#pragma unroll
              for (int i = 0; i < VEC; ++i) acc[i] += tk[j].w * gg[j][i];
              const int di = cl == 0 ? (int)tk[j].who : dummy;     // an idle task's dot lands in the scrap words
              if (pass == 0) dots[di] = part[j];          // uniform branch
              else dots[di] += part[j];
            }
          }
          if (pix_ok && chan_ok) {
            float *dst = gv + r * C + chan;
            float cur[VEC];
            LdsVec<VEC>::ld(dst, cur);
#pragma unroll
            for (int i = 0; i < VEC; ++i) cur[i] += acc[i];
            LdsVec<VEC>::st(dst, cur);
          }
        }
      }
      TILE_BARRIER();                                   // dots complete
      TT_MARK(4);
    }
    TILE_BARRIER();                                     // the tile is complete

    // ---------------- flush the tile (and leave it zeroed for the next item) ----------------
    const bool gv16 = (grad16 & 1) != 0, gd16 = (grad16 & 2) != 0;          // uniform
    const int mg = Mg == 1 ? 0 : m;
    char *gvalue_b = static_cast<char *>(grad_value) + (size_t)b * S * M * C * (gv16 ? 2 : 4);
    char *gdist_b = FUSED ? static_cast<char *>(grad_dist) + (size_t)b * S * Mg * D * (gd16 ? 2 : 4) : nullptr;
    const rsrc_t gvalue_r = make_rsrc(gvalue_b, (size_t)S * M * C * sizeof(float));
    const rsrc_t gdist_r = make_rsrc(gdist_b, FUSED ? (size_t)S * Mg * D * sizeof(float) : 0);
    // Rows 1..TY-1 x 1..TX-1 of the tile belong to no neighbour's halo; when this item writes its tile alone
    // nobody else adds to them, so they are stored instead of added atomically (grad_value and grad_dist are
    // zero on entry).
    const bool sole = item.w != 0;
    const bool sole_d = sole && Mg == M;                 // a gradient shared by the heads collects from all of them
    // four consecutive elements at element index `e` of a batch slice: stored, or added atomically
    auto put4 = [&](char *base, rsrc_t r, bool is16, uint32_t e, const float4 &val, bool store, bool every) {
      if (!is16) {
        float *fb = reinterpret_cast<float *>(base);
        if (store) {
          *reinterpret_cast<float4 *>(fb + e) = val;                              // zeros too: full lines
        } else {
          if (every || val.x != 0) scatter_add(r, fb, e * 4, val.x);
          if (every || val.y != 0) scatter_add(r, fb, e * 4 + 4, val.y);
          if (every || val.z != 0) scatter_add(r, fb, e * 4 + 8, val.z);
          if (every || val.w != 0) scatter_add(r, fb, e * 4 + 12, val.w);
        }
      } else {
        char *dst = base + (size_t)e * 2;
        if (store) {
          *reinterpret_cast<uint2 *>(dst) = make_uint2(pack_bf16x2(val.x, val.y), pack_bf16x2(val.z, val.w));
        } else {
          if (val.x != 0 || val.y != 0) atomic_add_bf16x2(dst, val.x, val.y);
          if (val.z != 0 || val.w != 0) atomic_add_bf16x2(dst + 4, val.z, val.w);
        }
      }
    };
    if (((C | D) & 3) == 0) {
      // four floats per lane: whole 128-byte lines leave each row group at once
      const int c4n = C >> 2, d4n = D >> 2;
      for (int i = tid; i < R * c4n; i += n_thr) {
        const int r = i / c4n, c = (i - r * c4n) << 2;
        float4 val = *reinterpret_cast<float4 *>(gv + r * C + c);
        const bool nz = val.x != 0 || val.y != 0 || val.z != 0 || val.w != 0;
        if (nz) *reinterpret_cast<float4 *>(gv + r * C + c) = make_float4(0, 0, 0, 0);
        const int ry = r / TW, rx = r - ry * TW;
        const int y = y0 + ry, x = x0 + rx;
        if (in_map(y, x, H, W)) {
          const uint32_t e = (uint32_t)(((start + y * W + x) * M + m) * C + c);
          const bool store = sole && ry >= 1 && ry < TY && rx >= 1 && rx < TX;
          if (store || nz) put4(gvalue_b, gvalue_r, gv16, e, val, store, true);
        }
      }
      for (int i = tid; i < R * d4n; i += n_thr) {
        const int r = i / d4n, d = (i - r * d4n) << 2;
        float4 val = *reinterpret_cast<float4 *>(gd + r * D + d);
        const bool nz = val.x != 0 || val.y != 0 || val.z != 0 || val.w != 0;
        if (nz) *reinterpret_cast<float4 *>(gd + r * D + d) = make_float4(0, 0, 0, 0);
        const int ry = r / TW, rx = r - ry * TW;
        const int y = y0 + ry, x = x0 + rx;
        if (in_map(y, x, H, W)) {
          const uint32_t e = (uint32_t)(((start + y * W + x) * Mg + mg) * D + d);
          const bool store = sole_d && ry >= 1 && ry < TY && rx >= 1 && rx < TX;
          if (store || nz) put4(gdist_b, gdist_r, gd16, e, val, store, false);
        }
      }
    } else {                                                    // float gradients only (the launcher sees to it)
      float *gvalue_f = reinterpret_cast<float *>(gvalue_b), *gdist_f = reinterpret_cast<float *>(gdist_b);
      for (int i = tid; i < R * C; i += n_thr) {
        const float val = gv[i];
        if (val != 0) {
          gv[i] = 0;
          const int r = i / C, c = i - r * C;
          const int ry = r / TW, rx = r % TW;
          const int y = y0 + ry, x = x0 + rx;
          if (in_map(y, x, H, W))
            scatter_add(gvalue_r, gvalue_f, (uint32_t)((((start + y * W + x) * M + m) * C + c) * 4), val);
        }
      }
      for (int i = tid; i < R * D; i += n_thr) {
        const float val = gd[i];
        if (val != 0) {
          gd[i] = 0;
          const int r = i / D, d = i - r * D;
          const int ry = r / TW, rx = r % TW;
          const int y = y0 + ry, x = x0 + rx;
          if (in_map(y, x, H, W))
            scatter_add(gdist_r, gdist_f, (uint32_t)((((start + y * W + x) * Mg + mg) * D + d) * 4), val);
        }
      }
    }
    TT_MARK(6);
  }
  TT_MARK(7);
  TT_FLUSH();
}

// ---------------------------------------------------------------------------------------
// Stage-1 backward alone on the same bins: the gradient with respect to the four depth scores of
// each point is given; grad_dist is accumulated in an LDS tile, the z gradient written per point.
//
// What bounds it is the random access of each point (its score gradient, its z gradient, four pairs of bins) and the
// tile's way out, so the kernel keeps both going at once: no barrier between the points of an item (taps go to LDS by
// compare-and-swap, so nobody waits for anybody), the next round's records asked for one round ahead and the next item's
// before the tile is flushed.  The bins come from the caches as long as few tiles are worked on at a time: with 16
// wavefronts per CU either way, one workgroup of 1024 threads beats four of 256 where tiles have the points for it (BLOCK:
// tile_config_of).  For a caller whose buffer may hold anything, a pixel that only this item can touch (no neighbour's halo, all
// the points of its bin, levels that share no keys) is stored 16 bytes per lane; everything else is added atomically, one
// float per lane on consecutive addresses.
// 6 x 9502 queries, 4 levels from 116 x 200, 8 points, 112 bins (14.6 M points): 1.19 ms with a ticket per tap and three
// barriers per 256 points, 1.01 ms without them, 0.85 ms with 1024 threads per tile.  With parts cut out of the 1.01 ms form, the z
// gradients' scattered stores were 0.27 of it, the tiles' way out 0.2, the taps 0.10, the score gradients' gathers 0.09.
// The stored pixels leave the L2 first (non-temporal: nobody reads them again, and the z gradients' lines need the room to fill
// up): the call 1061 -> 1039 us, 1030 with the z gradients stored behind the taps; 2 x 1000 queries on the same maps 144 -> 128.
// ---------------------------------------------------------------------------------------
constexpr int kNonTemporal = 2;       // cache policy of a buffer store on gfx950: the NT bit
// The fetching thread's state: the queue is asked for an item's number when another item is begun, the answer is looked
// at when that one's points are done, and the records asked for then are handed over with the next item.
struct DepthFetch {
  int classes_done, asked;        // asked: what the home queue's counter held, or -1: that queue is empty
  int4 rec, geo;
  __device__ __forceinline__ void load(const BinWorkspace &ws, int w) {
    rec = w >= 0 ? ws.items[w] : make_int4(-1, 0, 0, 0);
    geo = w >= 0 ? ws.geom[w] : make_int4(0, 0, 0, 0);
  }
  __device__ __forceinline__ void ask(const BinWorkspace &ws, int home) {
    unsigned at = home * kQueueStride;
    asm volatile("" : "+v"(at));      // a lane's own address: the compiler would combine lanes, and wait for the answer to do it
    if (classes_done == 0) asked = atomicAdd(&ws.queues[at], 1);
  }
  __device__ __forceinline__ void answer(const BinWorkspace &ws, const BinPlan &p, int home) {
    int w = -1;
    if (classes_done == 0) {
      w = p.class_start[home + 1] - 1 - asked;               // from the end, as pop_item does
      if (w < p.class_start[home]) { w = -1; classes_done = 1; }
    }
    load(ws, w >= 0 ? w : pop_item(ws, p, home, classes_done));
  }
};
template <typename T, int BLOCK>
__global__ __launch_bounds__(BLOCK, 4) void tile_depth_backward_kernel(
    BinWorkspace ws, const T *__restrict__ dist, const T *__restrict__ grad_score, float *__restrict__ grad_dist,
    float *__restrict__ grad_loc3, int B, int S, int M, int D, int L, int Q, int P, int stores) {
  // stores: the binning launches cleared what is added to here and nothing else (clear_unstored), else everything is added
  extern __shared__ __align__(16) float smem[];
  __shared__ int4 s_item[2], s_geo[2];
  __shared__ int s_lv[4][DFA3D_MAX_LEVELS];              // H, W, Dd, first key
  const BinPlan &p = *ws.plan;
  if (__builtin_expect(p.bins_per_bm == 0, 0)) {
    backward_without_bins<T, true>(ws, nullptr, dist, nullptr, nullptr, grad_score, nullptr, grad_dist, grad_loc3, 3, nullptr,
                                   nullptr, nullptr, M, M, B, S, M, 0, D, L, Q, P, 0);
    return;
  }
  const int TY = p.ty, TX = p.tx, TW = TX + 1, R = (TY + 1) * TW;
  const int tid = threadIdx.x;
  float *gd = smem;
  for (int i = tid; i < R * D; i += BLOCK) gd[i] = 0;
  if (tid < DFA3D_MAX_LEVELS) {
    s_lv[0][tid] = p.H[tid]; s_lv[1][tid] = p.W[tid]; s_lv[2][tid] = p.Dd[tid]; s_lv[3][tid] = p.start[tid];
  }
  const int home = blockIdx.x % kClasses;
  DepthFetch fetch;
  if (tid == 0) {
    fetch.classes_done = 0;
    fetch.ask(ws, home); fetch.answer(ws, p, home);
    s_item[0] = fetch.rec; s_geo[0] = fetch.geo;
    fetch.ask(ws, home); fetch.answer(ws, p, home);
  }
  __syncthreads();
  uint32_t next_gp = 0;
  float4 next_rec = make_float4(0, 0, 0, 0);
  auto ask_record = [&](int seg, int n, int i) {           // n > 0; lanes beyond the last point take that one's
    const int at = seg + min(i, n - 1);
    next_gp = ws.entries[at];
    next_rec = ws.recs[at];
  };
  if (s_item[0].x >= 0) ask_record(s_item[0].y, s_item[0].z, tid);
  for (int which = 0;; which ^= 1) {
    const int bin = __builtin_amdgcn_readfirstlane(s_item[which].x), seg = __builtin_amdgcn_readfirstlane(s_item[which].y);
    const int n_item = __builtin_amdgcn_readfirstlane(s_item[which].z);
    const bool sole = stores != 0 && __builtin_amdgcn_readfirstlane(s_item[which].w) != 0;
    if (bin < 0) break;                                   // queues drained: every wave leaves
    if (tid == 0) {
      s_item[which ^ 1] = fetch.rec; s_geo[which ^ 1] = fetch.geo;
      fetch.ask(ws, home);
    }
    const int b = __builtin_amdgcn_readfirstlane(s_geo[which].x), ml = __builtin_amdgcn_readfirstlane(s_geo[which].y);
    const int y0 = __builtin_amdgcn_readfirstlane(s_geo[which].z), x0 = __builtin_amdgcn_readfirstlane(s_geo[which].w);
    const int m = head_of(ml), l = level_of(ml);
    const int H = __builtin_amdgcn_readfirstlane(s_lv[0][l]), W = __builtin_amdgcn_readfirstlane(s_lv[1][l]);
    const int Dd = __builtin_amdgcn_readfirstlane(s_lv[2][l]), start = __builtin_amdgcn_readfirstlane(s_lv[3][l]);
    const rsrc_t dist_r = make_rsrc(dist + (size_t)b * S * M * D, (size_t)S * M * D * sizeof(T));

    for (int base = 0; base < n_item; base += BLOCK) {       // uniform over the workgroup
      const bool live = base + tid < n_item;
      const uint32_t gp = next_gp;
      const float4 rec = next_rec;
      if (base + BLOCK < n_item) ask_record(seg, n_item, base + BLOCK + tid);
      if (live) {
        const T *gi = grad_score + (size_t)gp * 4;
        float g4[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) g4[k] = Elem<T>::ld(gi + k);
        const Point2D<float> g = locate_2d<float>(rec.x, rec.y, H, W, start);
        const DepthTap<float> tap = locate_depth<float>(rec.z, Dd);
        float sc[4], lo[4], hi[4];
        corner_scores<T, float, true>(dist_r, g.key, tap, m, M, D, sc, lo, hi);
        // the base pixel lies in the tile (the binning put the point into this tile by it), so all four do
        const int cy = min(max(g.h0 - y0, 0), TY - 1), cx = min(max(g.w0 - x0, 0), TX - 1);
        const int row0 = (cy * TW + cx) * D, lo_at = max(tap.d0, 0), hi_at = min(tap.d0 + 1, D - 1);
        int at[8];
        float tv[8], gz = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool on = g.key[k] >= 0 && tap.inside;
          const int row = row0 + (k == 0 ? 0 : k == 1 ? D : k == 2 ? (TW + 1) * D : TW * D);
          at[2 * k] = row + lo_at; at[2 * k + 1] = row + hi_at;
          tv[2 * k] = on && tap.lo_ok ? tap.hd * g4[k] : 0.f;
          tv[2 * k + 1] = on && tap.hi_ok ? tap.ld * g4[k] : 0.f;
          gz += on ? g4[k] * (hi[k] - lo[k]) : 0.f;
        }
        lds_add_taps(gd, at, tv);
        float *gl = grad_loc3 + (size_t)gp * 3;
        gl[0] = 0; gl[1] = 0; gl[2] = gz * (float)Dd;
      }
    }
    if (tid == 0) fetch.answer(ws, p, home);
    lds_barrier();                                        // every tap is in the tile; the next item's record is there
    const int next_bin = s_item[which ^ 1].x;
    if (next_bin >= 0) ask_record(s_item[which ^ 1].y, s_item[which ^ 1].z, tid);

    float *gdist_b = grad_dist + (size_t)b * S * M * D;
    const rsrc_t gdist_r = make_rsrc(gdist_b, (size_t)S * M * D * sizeof(float));
    auto lanes_log2 = [](int n) { return n > 32 ? 6 : n > 16 ? 5 : n > 8 ? 4 : n > 4 ? 3 : 2; };
    if (sole) {
      const int n = D >> 2, sh = lanes_log2(n), inner = (TY - 1) * (TX - 1);
      for (int i = tid >> sh; i < inner; i += BLOCK >> sh) {
        const int ry = i / (TX - 1) + 1, rx = i % (TX - 1) + 1, y = y0 + ry, x = x0 + rx;
        const uint32_t e0 = (uint32_t)((((start + y * W + x) * M + m) * D) * 4);
        for (int c = tid & ((1 << sh) - 1); c < n; c += 1 << sh) {
          float4 *from = reinterpret_cast<float4 *>(gd + (ry * TW + rx) * D) + c;
          const float4 v = *from;
          *from = make_float4(0, 0, 0, 0);
          const u32x4 o = {__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)};
          __builtin_amdgcn_raw_buffer_store_b128(o, gdist_r, y < H && x < W ? e0 + 16 * c : kNoRow, 0, kNonTemporal);
        }
      }
    }
    const int sh = lanes_log2(D), rows = sole ? rim_pixels(TY, TX) : R;
    for (int i = tid >> sh; i < rows; i += BLOCK >> sh) {
      int ry, rx;
      if (sole) {
        rim_decode(i, TY, TX, ry, rx);
      } else {
        ry = i / TW; rx = i % TW;
      }
      const int r = ry * TW + rx, y = y0 + ry, x = x0 + rx;
      const bool out = in_map(y, x, H, W);
      const uint32_t e0 = (uint32_t)((((start + y * W + x) * M + m) * D) * 4);
      for (int c = tid & ((1 << sh) - 1); c < D; c += 1 << sh) {
        const float val = gd[r * D + c];
        if (val != 0) {
          gd[r * D + c] = 0;
          if (out) scatter_add(gdist_r, gdist_b, e0 + 4 * c, val);
        }
      }
    }
    lds_barrier();                                        // the tile is zero again
  }
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------
static int max_bins_per_bm(int S, int L, int ty, int tx) {
  // tiles of a level = ((H + ty) / ty) ((W + tx) / tx) <= (H/ty + 1) (W/tx + 1) <= HW/(ty tx) + H/ty + W/tx + 1
  // and H + W <= HW + 1
  const int e = ty < tx ? ty : tx;
  const long long v = (long long)S / (ty * tx) + ((long long)S + L) / e + 2LL * L + 1;
  return (int)v;
}

constexpr int kMinChunk = 64;        // smallest accepted points-per-item
// only the fused entry point sets dist_heads
static bool shared_dist(const BwdArgs &a) { return a.dist_heads == 1 && a.M > 1; }

// Up to two buffers: the direct kernels' two gradients of a small call took as long to clear as two empty launches.
__global__ __launch_bounds__(256) void fill_zero_kernel(float4 *__restrict__ dst, size_t n4, float4 *__restrict__ other, size_t other4) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4 + other4; i += (size_t)gridDim.x * 256)
    (i < n4 ? dst[i] : other[i - n4]) = make_float4(0, 0, 0, 0);
}
__global__ __launch_bounds__(64) void fill_zero_words_kernel(uint32_t *__restrict__ dst, size_t n) {
  for (size_t i = threadIdx.x; i < n; i += 64) dst[i] = 0;
}

hipError_t launch_zero_fill(void *dst, size_t bytes, hipStream_t stream) {
  if (dst == nullptr || (bytes & 3) != 0 || ((uintptr_t)dst & 3) != 0) return hipErrorInvalidValue;
  char *p = static_cast<char *>(dst);
  const size_t head = ((uintptr_t)p & 15) ? 16 - ((uintptr_t)p & 15) : 0;        // bytes before the first 16-byte boundary
  const size_t lead = head < bytes ? head : bytes, body = (bytes - lead) & ~(size_t)15, tail = bytes - lead - body;
  if (lead) hipLaunchKernelGGL(fill_zero_words_kernel, dim3(1), dim3(64), 0, stream, reinterpret_cast<uint32_t *>(p), lead / 4);
  if (body) hipLaunchKernelGGL(fill_zero_kernel, dim3(2048), dim3(256), 0, stream, reinterpret_cast<float4 *>(p + lead), body / 16, (float4 *)nullptr, (size_t)0);
  if (tail) hipLaunchKernelGGL(fill_zero_words_kernel, dim3(1), dim3(64), 0, stream, reinterpret_cast<uint32_t *>(p + lead + body), tail / 4);
  return hipGetLastError();
}

hipError_t launch_zero_fill(void *dst, size_t bytes, void *other, size_t other_bytes, hipStream_t stream) {
  if (((uintptr_t)dst & 15) == 0 && ((uintptr_t)other & 15) == 0 && (bytes & 15) == 0 && (other_bytes & 15) == 0 && dst != nullptr && other != nullptr) {
    hipLaunchKernelGGL(fill_zero_kernel, dim3(2048), dim3(256), 0, stream, static_cast<float4 *>(dst), bytes / 16, static_cast<float4 *>(other), other_bytes / 16);
    return hipGetLastError();
  }
  if (hipError_t e = launch_zero_fill(dst, bytes, stream)) return e;
  return launch_zero_fill(other, other_bytes, stream);
}

// dst[r, :] = sum over heads m of src[r, m, :], rows of D floats, heads in order; dst is float, or bfloat16
// when dst16 is set (then D is a multiple of 4)
__global__ __launch_bounds__(256) void head_sum_kernel(const float *__restrict__ src, void *__restrict__ dst,
                                                       size_t rows, int M, int D, int dst16) {
  if ((D & 3) == 0) {
    const int d4 = D >> 2;
    const size_t n = rows * d4;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
      const size_t r = i / d4;
      const int d = (int)(i - r * d4) << 2;
      float4 acc = make_float4(0, 0, 0, 0);
      for (int m = 0; m < M; ++m) {
        const float4 t = *reinterpret_cast<const float4 *>(src + (r * M + m) * D + d);
        acc.x += t.x; acc.y += t.y; acc.z += t.z; acc.w += t.w;
      }
      if (dst16)
        *reinterpret_cast<uint2 *>(static_cast<char *>(dst) + (r * D + d) * 2) =
            make_uint2(pack_bf16x2(acc.x, acc.y), pack_bf16x2(acc.z, acc.w));
      else
        *reinterpret_cast<float4 *>(static_cast<float *>(dst) + r * D + d) = acc;
    }
  } else {
    const size_t n = rows * D;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
      const size_t r = i / D;
      const int d = (int)(i - r * D);
      float acc = 0;
      for (int m = 0; m < M; ++m) acc += src[(r * M + m) * D + d];
      static_cast<float *>(dst)[i] = acc;
    }
  }
}
// bfloat16 gradients from float sums: everything rounded once, after the tile kernel
__global__ __launch_bounds__(256) void round_rows_kernel(const float4 *__restrict__ value_sums, uint2 *__restrict__ grad_value, size_t nv4,
                                                         const float4 *__restrict__ dist_sums, uint2 *__restrict__ grad_dist, size_t nd4) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < nv4 + nd4; i += (size_t)gridDim.x * 256) {
    const float4 f = i < nv4 ? value_sums[i] : dist_sums[i - nv4];
    *(i < nv4 ? grad_value + i : grad_dist + (i - nv4)) = make_uint2(pack_bf16x2(f.x, f.y), pack_bf16x2(f.z, f.w));
  }
}

// gd_heads: grad_dist per head (shared_dist); value_sums, dist_sums: see sums_in_float; without them the workspace ends at `least`
struct BinLayout { size_t plan, queues, counts, cursor, items, geom, entries, recs, gd_heads, value_sums, dist_sums, least, total; };
static BinLayout bin_layout(const BwdArgs &a, int ty, int tx, bool float_sums) {
  BinLayout o;
  const size_t nbins = (size_t)max_bins_per_bm(a.S, a.L, ty, tx) * slot_count(a.B, a.M);
  const size_t npts = (size_t)a.B * a.Q * a.M * a.L * a.P;
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  o.plan = 0;
  o.queues = up(o.plan + sizeof(BinPlan));
  o.counts = up(o.queues + kQueueInts * sizeof(int));
  o.cursor = up(o.counts + nbins * sizeof(int));
  // work items: at most one partial chunk per bin plus the full chunks
  o.items = up(o.cursor + nbins * sizeof(int));
  o.geom = up(o.items + (nbins + npts / kMinChunk + 1) * sizeof(int4));
  o.entries = up(o.geom + (nbins + npts / kMinChunk + 1) * sizeof(int4));
  o.recs = up(o.entries + npts * sizeof(uint32_t));
  // a distribution shared by the heads: grad_dist per head first (stores, as with a distribution per head),
  // summed over the heads afterwards; eight XCDs adding atomically into one shared tile cost twice as much
  o.gd_heads = up(o.recs + npts * sizeof(float4));
  const size_t per_head = shared_dist(a) ? (size_t)a.B * a.S * a.M * a.D * sizeof(float) : 0;
  o.least = o.total = up(o.gd_heads + per_head);
  o.value_sums = o.dist_sums = o.total;
  if (float_sums) {
    o.dist_sums = up(o.value_sums + (size_t)a.B * a.S * a.M * a.C * sizeof(float));
    o.total = up(o.dist_sums + (shared_dist(a) ? 0 : (size_t)a.B * a.S * a.M * a.D * sizeof(float)));
  }
  return o;
}

#ifdef DFA3D_TILE_TIMING
// development builds: where in a workspace the tile kernels' phase clocks live (sixteen 64-bit counters)
size_t tile_timer_offset() {
  return ((sizeof(BinPlan) + 255) & ~(size_t)255) + (size_t)kClasses * kQueueStride * sizeof(int);
}
#endif

// Launch shape of the tile kernels: tile edge, threads per workgroup, points per pass.
struct TileConfig { int ty, tx, block, pp; size_t lds; bool cells; };      // cells: the cell-owned kernel takes the launch

// kind 0: both stages, 1: stage 2 alone (no depth tile), 2: stage 1 alone (depth tile only)
static size_t tile_lds_bytes(int kind, int ty, int tx, int C, int D, int pp) {
  if (kind == 2) return (((size_t)(ty + 1) * (tx + 1) * D + 3) & ~(size_t)3) * 4;      // the depth tile
  return (size_t)tile_lds_layout(ty, tx, C, kind == 1 ? 0 : D, pp).total * 4;
}

// Defaults: 512 threads; the tile and the points per pass (pp) follow from what fits in LDS, in an order of
// preference taken from measurements on rows of 32 .. 256 channels and 64 .. 256 depth bins:
//   * two workgroups per CU (79 KB each) beat one, and one per CU on a 4x8 tile beats tiles under 4x4 pixels by
//     far (256 channels: 3.2 ms against 11.9 ms);
//   * tiles above 8x16 pixels lose (the rows phase needs several rounds); passes of 64 points lose to 128 and 256;
//   * an 8x8 tile at pp 128 beats a 4x8 tile at pp 256 (128 bins: 0.68 against 0.74 ms for 2.56 M points) unless
//     most tiles take several passes (`dense`: the dense BEV workload, 41 points per pixel, 7.0 against 8.9 ms).
static TileConfig pick_tile_config(int kind, int C, int D, int elem, int tile_hint, int block_hint, int pass_hint, bool dense,
                                   bool cells_wanted, int depth_block, bool depth_small) {
  TileConfig c;
  c.cells = false;
  if (cells_wanted && kind != 2 && C <= 64 && (block_hint == 0 || block_hint == cell_kernel_block(C)) &&
      (pass_hint == 0 || pass_hint == cell_kernel_pass(C))) {
    // The cell-owned kernel: the tallest tile whose depth tile leaves room for two workgroups per CU (half of the 160 KB
    // less the kernel's static LDS: 8x8 pixels up to 112 bins, 7x8 with 128), else for one.
    const int hy = tile_hint / 100, hx = tile_hint % 100, Dk = kind == 1 ? 0 : D;
    for (size_t budget : {cell_kernel_half_cu_lds(), (size_t)150 * 1024}) {
      for (int ty = tile_hint > 0 ? hy : cell_max_ty(C); ty >= 1; --ty) {
        if (cell_kernel_applies(C, ty, tile_hint > 0 ? hx : kCellTX) && cell_kernel_lds_bytes(ty, C, Dk, elem) <= budget) {
          c.cells = true; c.block = cell_kernel_block(C); c.pp = cell_kernel_pass(C); c.ty = ty; c.tx = kCellTX;
          c.lds = cell_kernel_lds_bytes(ty, C, Dk, elem);
          return c;
        }
        if (tile_hint > 0) break;
      }
    }
  }
  c.block = kind == 2 ? depth_block : (block_hint == 256 ? 256 : 512);
  const int pp_max = kind == 2 ? c.block : c.block / 2;      // the fused tile kernel wants two halves of pp threads
  auto clamp_pp = [&](int pp) { return pp > pp_max ? pp_max : pp; };
  const size_t two_per_cu = kind == 2 && depth_block == 256 ? 40 * 1024 : 79 * 1024, one_per_cu = 150 * 1024;
  const int hy = tile_hint / 100, hx = tile_hint % 100;
  const bool tile_given = tile_hint > 0 && hy >= 1 && hx >= 1 && hy <= 64 && hx <= 64;
  const bool pass_given = pass_hint == 64 || pass_hint == 128 || pass_hint == 256;
  auto fits = [&](int ty, int tx, int pp, size_t budget) { return tile_lds_bytes(kind, ty, tx, C, D, clamp_pp(pp)) <= budget; };
  auto done = [&](int ty, int tx, int pp) {
    c.ty = ty; c.tx = tx; c.pp = clamp_pp(pp);
    c.lds = tile_lds_bytes(kind, c.ty, c.tx, C, D, c.pp);
    return c;
  };
  struct Pref { int ty, tx, pp; };
  static const Pref sparse_order[] = {{8, 16, 256}, {8, 8, 256}, {8, 8, 128}, {4, 8, 256}, {4, 8, 128}, {4, 4, 256},
                                      {4, 4, 128}, {8, 8, 64}, {4, 8, 64}, {4, 4, 64}};
  static const Pref dense_order[] = {{8, 16, 256}, {8, 8, 256}, {4, 8, 256}, {4, 4, 256}, {8, 8, 128}, {4, 8, 128},
                                     {4, 4, 128}, {8, 8, 64}, {4, 8, 64}, {4, 4, 64}};
  const Pref *order = dense ? dense_order : sparse_order;
  if (kind == 2 && depth_small && !tile_given && fits(8, 8, 256, two_per_cu)) return done(8, 8, 256);
  for (size_t budget : {two_per_cu, one_per_cu}) {
    for (int i = 0; i < 10; ++i) {
      const int ty = tile_given ? hy : order[i].ty, tx = tile_given ? hx : order[i].tx;
      const int pp = pass_given ? pass_hint : order[i].pp;
      if (fits(ty, tx, pp, budget)) return done(ty, tx, pp);
    }
  }
  // nothing of at least 4x4 pixels fits: whatever the caller fixed, else the largest small tile with short passes
  const int pp = pass_given ? pass_hint : 64;
  if (tile_given) return done(hy, hx, pp);
  const int small[][2] = {{2, 4}, {2, 2}, {1, 1}};
  for (auto &t : small)
    if (fits(t[0], t[1], pp, one_per_cu)) return done(t[0], t[1], pp);
  return done(1, 1, pp);
}

static int bwd_kind(const BwdArgs &a) { return a.dist != nullptr ? 0 : 1; }
static TileConfig tile_config_of(const BwdArgs &a, int kind, int dtype) {
  const double per_pixel = (double)a.Q * a.L * a.P / (a.S > 0 ? a.S : 1);      // sampling points per pixel of a (batch, head)
  // a caller that names the channels per lane asks for the row-owned kernel, whose tiling that is
  // (its per-point gradients are buffer-addressed per batch element: below 2^31 bytes of 16 per point)
  const bool cells = a.vec_hint == 0 && (size_t)a.Q * a.M * a.L * a.P * 16 < (size_t)kNoRow;
  // Stage 1 alone: threads per tile by the points it can expect, and 8 x 8 tiles instead of 8 x 16 where those would give
  // a CU only a few.  The call, four levels from 116 x 200 unless said, 256 / 512 / 1024 threads:
  //   6 x 9502 queries, 32 points each (10 per pixel), 112 bins 1224 / 1154 / 1065 us, 64 bins 1109 / 950 / 872, 16 bins 930 / 750 / 717
  //   6 x 4000 queries, 16 points (2 per pixel), 64 bins 387 / 367 / 404; 6 x 2000 281 / 284 / 336
  //   4 x 1000 queries, 16 points (0.5 per pixel), 48 bins 161 / 174 / 212
  //   8 x 8 for 8 x 16 tiles, 1024 threads: 6 x 4000 queries, 8 points, 23 x 40, 112 bins (345 tiles) 144 -> 122; 2 x 9502 queries,
  //   32 points, 4 heads, 80 bins (1927 tiles) 230 -> 222; 6 x 9502 queries, 112 bins (11559 tiles) 1065 -> 1097
  const int depth_block = per_pixel < 0.75 ? 256 : per_pixel < 3.0 ? 512 : 1024;
  const bool depth_small = depth_block == 1024 && (double)a.S * a.B * a.M / 128 < 4096;
  return pick_tile_config(kind, a.C, a.D, dtype == DFA3D_F32 ? 4 : 2, a.tile_hint, a.block_hint, a.pass_hint, per_pixel >= 16.0, cells,
                          depth_block, depth_small);
}

// Whether bfloat16 gradients are summed in float in the workspace and rounded once at the end.  A bfloat16 buffer rounds at
// every add to a pixel that several tiles share, so the share of such pixels decides the error, and the cell-owned kernel's
// tiles are smaller than what LDS allows where its walkers own fewer rows (over 32 channels: 4 x 8 pixels, 34 % of them on
// the rim) or where rows and bins are short (8 x 8: 23 %; 8 x 16: 18 %).  There the sums are formed in float.  2 x 20000
// queries, 8 heads, 60 x 100 map, relative error of grad_value against float: 64 channels, 16 bins 1.97e-3 with 4 x 8
// tiles and bfloat16 adds, 1.86e-3 with the row-owned kernel's 8 x 8, 1.66e-3 this way (a single rounding); backward
// 231 / 354 / 248 us.  16 channels, 16 bins: 1.87e-3, 1.82e-3, 1.66e-3; 134 / 242 / 137 us.
// Rows of 32 channels keep 8 x 8 tiles and bfloat16 adds (1.86e-3), also up to 22 bins, where LDS would hold 8 x 16
// (1.81e-3): they have had them since there are 8 x 8 tiles, and float sums would cost them 145 -> 153 us on the 60 x 100
// map and 776 -> 865 us with 6 x 20000 queries of 8 points on 116 x 200.
static bool sums_in_float(const BwdArgs &a, int kind, int dtype, const TileConfig &c) {
  if (!a.grad_bf16 || kind != 0 || !c.cells || a.tile_hint != 0 || a.C == 32) return false;
  BwdArgs rows = a;
  rows.vec_hint = 1;                                                           // asks for the row-owned kernel's tile
  const TileConfig r = tile_config_of(rows, kind, dtype);
  return r.ty * r.tx >= 2 * c.ty * c.tx;
}

static size_t workspace_bytes_for(const BwdArgs &a, int kind, int dtype, bool least = false) {
  if (dtype == DFA3D_F64) return 0;
  if ((size_t)a.B * a.Q * a.M * a.L * a.P >= (1ull << 31)) return 0;          // point indices and segment offsets are 32-bit
  if (kind != 2 && (size_t)a.Q * a.M * a.C * 4 >= (size_t)kMaxSliceBytes) return 0;   // grad_out rows are buffer-addressed per batch element
  if (a.grad_bf16 && (kind != 0 || ((a.C | a.D) & 3) != 0)) return 0;          // bfloat16 gradients: whole 8-byte groups
  const TileConfig c = tile_config_of(a, kind, dtype);
  if (c.lds > 150 * 1024) return 0;                                            // rows too long for LDS tiles
  if ((size_t)max_bins_per_bm(a.S, a.L, c.ty, c.tx) * slot_count(1, a.M) * a.B >= (1ull << 31)) return 0;      // so are bin numbers
  const BinLayout lay = bin_layout(a, c.ty, c.tx, sums_in_float(a, kind, dtype, c));
  return least ? lay.least : lay.total;
}

// kind as in tile_lds_bytes; `a.dist != nullptr` is not consulted here, so dimension-only queries work
size_t binned_backward_workspace_bytes(const BwdArgs &a, int kind, int dtype) { return workspace_bytes_for(a, kind, dtype); }
size_t binned_backward_least_workspace_bytes(const BwdArgs &a, int kind, int dtype) { return workspace_bytes_for(a, kind, dtype, true); }

// A backward on the tile kernels is five launches (six for a distribution shared by the heads), of which each takes its 5 us however
// few points there are, and visits every tile that has one.  The direct kernels are two launches, whose time is the clearing and one
// atomic per 64-byte piece of what a point adds to, 20 G of which the L2 executes a second where points are spread; adds to the same
// few lines wait for one another, some 40 ns each.  So the direct kernels take calls
//   * whose atomics, as of spread points, cost less than launches and tiles do: lines drawn where neither points all over the map, nor
//     around the query, nor clustered (a normal distribution about the middle, 0.15 of the map) lose more than some percent;
//   * with at most 8000 (stage 1: 4000) points of a batch element, head and level, ten of a row, three of a line of a shared
//     distribution: they may lie closer together;
//   * with float sums of 80 MB at most, where those are formed for bfloat16 gradients alone: the tile kernels add bfloat16 in place (384
//     points, 6 x 116 x 200, 66 us; 222 for the direct kernels, whatever the points.  For a shared distribution 240 us and more).
// The call's kernels alone (captured in a graph), 8 heads of 32 channels, 64 bins, float32, at the line, thousands of points: tile kernels,
// direct; all over, around the query, clustered | normal, 0.02 of the map | all in one cell:
//   1 x 20 x 30, 32 bins          33: 33, 28   34, 26   36, 41 | 69, 156 | 87, 192
//   2 x 40 x 60 and 20 x 30       47: 46, 39   46, 38   46, 45 | 67, 94 | 91, 125
//     16 channels, 64 channels    69: 44, 39   45, 37   47, 43 | 67, 111 | 93, 168             30: 57, 42   57, 41   55, 42 | 71, 68 | 90, 99
//   2 x 80 x 120, 3 levels        97: 100, 76   100, 75   91, 84 | 83, 159 | 129, 268
//   2 x 116 x 200, 128 bins       128: 192, 140   192, 136   158, 135 | 98, 155 | 150, 462
//   2 x 116 x 200, 4 levels       193: 182, 156   183, 152   152, 164 | 133, 335 | 195, 448
//   6 x 116 x 200, 4 levels       283: 434, 306   415, 301   318, 311 | 221, 416 | 336, 566
//     (beyond the line              500: 451, 424   452, 413   352, 431 | 288, 712 | 491, 1057)
//   one distribution for all heads, 2 x 40 x 60   53: 54, 42   54, 40   56, 49 | 73, 165 | 96, 268
//     6 x 116 x 200, 4 levels     554: 536, 372   536, 359   443, 408 | 392, 881 | 624, 1182
//   plain, 2 x 40 x 60            63: 36, 34   36, 33   39, 35 | 48, 67 | 84, 138
//     6 x 116 x 200, 4 levels     412: 306, 203   304, 203   226, 211 | 152, 347 | 273, 545
//   stage 1 alone, 2 x 40 x 60    64: 48, 22   49, 20   53, 22 | 53, 36 | 66, 170
//     (beyond the line            177: 59, 46   61, 41   55, 46 | 61, 91 | 86, 528)
//     6 x 116 x 200, 4 levels     151: 159, 141   154, 122   158, 148 | 141, 137 | 156, 135
//   bfloat16, 2 x 40 x 60         36: 42, 39   42, 38   43, 44 | 137, 85 | 264, 93
//     2 x 80 x 120, 3 levels      52: 93, 66   90, 66   81, 70 | 167, 100 | 312, 159
//     sums of 95 MB               0.5: 41, 49   37: 101, 64   100, 63   81, 63 | 115, 111 | 329, 145
//     of 189 MB                   25: 129, 99   108, 97   94, 97 | 69, 108 | 140, 122
//     one distribution for all heads, 6 x 116 x 200, 4 levels   207: 510, 236   488, 233   390, 247 | 363, 363 | 482, 486
//   beyond ten of a row: plain, 15 x 21                            51: 38, 31   40, 31   48, 61 | 72, 255 | 96, 265
//   beyond three of a line: 4 x 45 x 70, 4 levels, 16 bins         84: 78, 70   79, 63   74, 109
bool few_points(const BwdArgs &a, int kind, int dtype) {
  if (dtype == DFA3D_F64) return true;                       // (no tile kernels)
  const double points = (double)a.B * a.Q * a.M * a.L * a.P, rows = (double)a.B * a.S * a.M;
  if ((double)a.Q * a.P > (kind == 2 ? 4000 : 8000) || points > 10 * rows) return false;
  const int pieces = (kind == 2 ? 0 : 4 * ((a.C * 4 + 63) / 64)) + (kind == 1 ? 0 : 4);        // that a point adds to
  double atomics_us = points * pieces * 0.05e-3;
  if (kind == 2) return atomics_us < std::max(40 - rows * 0.01e-3, 10.0);
  if (kind == 1) return atomics_us < std::min(20 + rows * 0.14e-3, 165.0);
  // float sums that the tile kernels would not form are cleared, written, read and rounded besides
  if (a.grad_bf16 && !sums_in_float(a, kind, dtype, tile_config_of(a, kind, dtype))) {
    const double sums = 4 * rows * a.C + 4 * (double)a.B * a.S * (shared_dist(a) ? 1 : a.M) * a.D;
    if (sums > 80e6 && !shared_dist(a)) return false;
    atomics_us += sums * 0.35e-6;
  }
  if (shared_dist(a)) return points < 3.0 * a.B * a.S * ((a.D * 4 + 63) / 64) && atomics_us < 22 + rows * 0.21e-3;
  return atomics_us < std::min(19 + rows * (0.10e-3 + 0.001e-3 * (a.C + a.D)), 170.0);
}

static size_t few_points_value_bytes(const BwdArgs &a) { return ((size_t)a.B * a.S * a.M * a.C * sizeof(float) + 255) & ~(size_t)255; }
static size_t few_points_dist_rows(const BwdArgs &a) { return (size_t)a.B * a.S * (a.dist_heads == 1 ? 1 : a.M); }
size_t few_points_workspace_bytes(const BwdArgs &a) {
  if (((a.C | a.D) & 3) != 0) return 0;                      // bfloat16 gradients: whole 8-byte groups
  return few_points_value_bytes(a) + few_points_dist_rows(a) * a.D * sizeof(float);
}

// Per-device facts and per-kernel attributes are looked up once and remembered (a launch then costs no
// runtime queries).
static std::mutex g_launch_mutex;
static int g_cu_count[64];                                           // 0 = not asked yet
static std::map<std::pair<const void *, int>, size_t> g_lds_allowed;  // (kernel, device) -> dynamic LDS bytes granted

static int current_device() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  return dev;
}

int cu_count() {
  const int dev = current_device();
  std::lock_guard<std::mutex> lock(g_launch_mutex);
  if (g_cu_count[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    g_cu_count[dev] = n;
  }
  return g_cu_count[dev];
}

static int tile_grid(size_t lds, int block) {
  const size_t per_cu = lds > 0 ? (160 * 1024) / lds : 8;
  int wg_per_cu = (int)(per_cu < 1 ? 1 : per_cu > 8 ? 8 : per_cu);
  const int by_waves = 32 / (block / kWave);
  if (wg_per_cu > by_waves) wg_per_cu = by_waves < 1 ? 1 : by_waves;
  return cu_count() * wg_per_cu;
}

hipError_t allow_lds(const void *fn, size_t lds) {
  if (lds <= 64 * 1024) return hipSuccess;
  const std::pair<const void *, int> key(fn, current_device());
  std::lock_guard<std::mutex> lock(g_launch_mutex);
  auto it = g_lds_allowed.find(key);
  if (it != g_lds_allowed.end() && it->second >= lds) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e == hipSuccess) g_lds_allowed[key] = lds;
  return e;
}
template <typename K> static hipError_t allow_lds(K kern, size_t lds) {
  return allow_lds(reinterpret_cast<const void *>(kern), lds);
}

template <typename T, int VEC, int LPR>
static hipError_t launch_tile_cfg(const BwdArgs &a, const BinWorkspace &ws, const TileConfig &c, float *gd_heads,
                                  hipStream_t stream) {
  // gd_heads != nullptr: the kernel writes grad_dist per head there instead of into a.grad_dist
  const int grid = tile_grid(c.lds, c.block);
  if (a.dist != nullptr) {
    auto kern = tile_backward_kernel<T, VEC, LPR, true>;
    if (hipError_t e = allow_lds(kern, c.lds)) return e;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(c.block), c.lds, stream, ws, (const T *)a.value, (const T *)a.dist,
                       (const T *)nullptr, (const T *)a.grad_out, (const T *)a.grad_score_in, a.grad_value,
                       gd_heads != nullptr ? (void *)gd_heads : a.grad_dist, (float *)a.grad_loc, a.grad_loc_stride, (float *)a.grad_attn,
                       (float *)nullptr, (const float *)a.grad_weight_update, a.dist_heads == 1 ? 1 : a.M,
                       (a.dist_heads == 1 && gd_heads == nullptr) ? 1 : a.M, a.B, a.S, a.M, a.C, a.D, a.L, a.Q, a.P, c.pp,
                       (a.grad_bf16 ? 1 : 0) | ((a.grad_bf16 && gd_heads == nullptr) ? 2 : 0));
  } else {
    auto kern = tile_backward_kernel<T, VEC, LPR, false>;
    if (hipError_t e = allow_lds(kern, c.lds)) return e;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(c.block), c.lds, stream, ws, (const T *)a.value, (const T *)nullptr,
                       (const T *)a.score_in, (const T *)a.grad_out, (const T *)nullptr, a.grad_value,
                       (void *)nullptr, (float *)a.grad_loc, a.grad_loc_stride, (float *)a.grad_attn,
                       (float *)a.grad_score_out, (const float *)nullptr, a.M, a.M, a.B, a.S, a.M, a.C, 0, a.L, a.Q,
                       a.P, c.pp, 0);
  }
  return hipGetLastError();
}


template <typename T>
static hipError_t launch_tile_typed(const BwdArgs &a, const BinWorkspace &ws, const TileConfig &c, float *gd_heads,
                                    hipStream_t stream) {
  if (c.cells) {
    const int dtype = sizeof(T) == 4 ? DFA3D_F32 : DFA3D_BF16;
    if (hipError_t e = allow_lds(cell_kernel_symbol(a, dtype), c.lds)) return e;
    // two workgroups per CU at most (its registers): a workgroup that had to wait for a place would sit on dealt items
    return launch_cell_kernel(a, dtype, ws, c.lds, tile_grid(c.lds < 80 * 1024 ? 80 * 1024 : c.lds, c.block), gd_heads, stream);
  }
  // Eight channels per lane when the tile has more rows than four-channel row groups (a 9x9 tile against 64
  // groups of 8 lanes): 128 groups of 4 lanes then cover it in one round with fewer instructions per corner
  // task.  Smaller tiles would leave most of those groups idle.
  const int groups4 = (c.block / 64) * 8;
  if (((a.vec_hint == 0 && (c.ty + 1) * (c.tx + 1) > groups4) || a.vec_hint == 8) && sizeof(T) <= 4) {
    if (a.C == 32) return launch_tile_cfg<T, 8, 4>(a, ws, c, gd_heads, stream);
    if (a.C == 64) return launch_tile_cfg<T, 8, 8>(a, ws, c, gd_heads, stream);
  }
  const RowTiling rt = pick_row_tiling(a.C, (int)sizeof(T), a.vec_hint);
#define DFA3D_CASE(V, R) \
  if (rt.vec == V && rt.lpr == R) return launch_tile_cfg<T, V, R>(a, ws, c, gd_heads, stream);
  DFA3D_ROW_TILINGS(DFA3D_CASE)
#undef DFA3D_CASE
  return hipErrorInvalidValue;
}

static BinWorkspace carve_workspace(void *workspace, const BinLayout &lay) {
  char *base = static_cast<char *>(workspace);
  BinWorkspace ws;
  ws.plan = reinterpret_cast<BinPlan *>(base + lay.plan);
  ws.queues = reinterpret_cast<int *>(base + lay.queues);
  ws.counts = reinterpret_cast<int *>(base + lay.counts);
  ws.cursor = reinterpret_cast<int *>(base + lay.cursor);
  ws.items = reinterpret_cast<int4 *>(base + lay.items);
  ws.geom = reinterpret_cast<int4 *>(base + lay.geom);
  ws.entries = reinterpret_cast<uint32_t *>(base + lay.entries);
  ws.recs = reinterpret_cast<float4 *>(base + lay.recs);
  return ws;
}

// plan, count, scan, fill.  `a` supplies dimensions, shapes, locations and the per-point gradient
// buffers that receive zeros for points the operator skips.
static hipError_t run_binning(const BwdArgs &a, const BinWorkspace &ws, const TileConfig &cfg, float *gd_heads, hipStream_t stream) {
  // gradients stored in bfloat16 are rounded at every atomic add: their bins are split no more than they have to be
  const int chunk = a.chunk_hint > 0 ? a.chunk_hint : a.grad_bf16 ? kMaxChunk : 0;
  const int ty = cfg.ty, tx = cfg.tx;
  const int mb = max_bins_per_bm(a.S, a.L, ty, tx);
  hipLaunchKernelGGL(plan_and_clear_kernel, dim3(64), dim3(256), 0, stream, ws, a.shapes, a.shape_stride, a.level_start,
                     a.L, a.S, (a.dist != nullptr || a.C == 0) ? a.D : 0, a.B, a.M, ty, tx, chunk, mb);
  const int LP = a.L * a.P;
  const bool sorted_maybe = LP <= kStage, sorted_surely = sorted_maybe && mb <= kSortedBins;
  const int q_turn = sorted_maybe ? kStage / LP : 1;             // (bin_points_in_order makes its own of it)
  const int q_blocks = (a.Q + q_turn - 1) / q_turn;
  const long long blocks = (long long)a.B * a.M * q_blocks;
  if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
  const int held = tile_grid(kSortedFillLds, kFillThreads);       // blocks of kFillThreads that the chip holds
  const unsigned grid = blocks < held ? (unsigned)blocks : (unsigned)held;
  const int hist_cap = sorted_surely ? 0 : mb < kHistCap ? mb : kHistCap;
  static_assert((size_t)kHistCap * 8 <= kSortedFillLds, "bin_points_in_order's counters lie in the sorted fill's LDS");
  const BinDivs divs{FastDiv((uint32_t)LP), FastDiv((uint32_t)a.P), FastDiv((uint32_t)ty), FastDiv((uint32_t)tx)};
  // blocks of the count per (batch, head): what the chip holds, all with as many turns
  const int parts_held = std::max(1, held / std::min(held, a.B * a.M)), turns = (q_blocks + parts_held - 1) / parts_held;
  const int parts = (q_blocks + turns - 1) / turns;
  hipLaunchKernelGGL(bin_count_kernel, dim3((unsigned)(a.B * a.M * parts)), dim3(kFillThreads), (size_t)hist_cap * 4, stream, ws,
                     (const float *)a.loc, a.loc_stride, a.B, a.M, a.L, a.Q, a.P, q_turn, parts, hist_cap, divs);
  // What further blocks of the scan's launch clear meanwhile: for a caller that did not zero them (options.clear),
  // the rows of grad_value / grad_dist that the tile kernel adds to rather than stores; and always, for a
  // distribution shared by the heads, those rows of the per-head grad_dist in the workspace (the head sum then
  // writes all of the caller's grad_dist).
  const int ge = a.grad_bf16 ? 2 : 4;
  const bool writes_dist = a.dist != nullptr || a.C == 0;
  const size_t rows_of_b = (size_t)a.S * a.M, rows = rows_of_b * a.B;
  // 64 rows a turn are four wavefronts per SIMD from 2^18 rows on; fewer would leave CUs idle (59 k rows: 12.1 us against 7.4 in turns of 16)
  const int rows_of_wave = rows >= (size_t)256 * 1024 ? kWave : 16;
  const ClearRows value_rows(a.clear_grads && a.C > 0 ? a.grad_value : nullptr, a.C * ge);
  const ClearRows dist_rows = gd_heads != nullptr ? ClearRows(gd_heads, a.D * 4) : ClearRows(a.clear_grads && writes_dist ? a.grad_dist : nullptr, a.D * ge);
  const ClearArgs ca = {value_rows, dist_rows, a.B, a.M, a.L,
                        cfg.cells || ((a.C | (writes_dist ? a.D : 0)) & 3) == 0 ? 1 : 0,        // the tile kernel's own condition
                        (int)rows_of_b, rows_of_wave, FastDiv((uint32_t)((rows_of_b + rows_of_wave - 1) / rows_of_wave)),
                        FastDiv((uint32_t)a.M), FastDiv((uint32_t)ty), FastDiv((uint32_t)tx)};
  unsigned clear_blocks = 0;
  if (a.clear_grads || gd_heads != nullptr) {            // launch_backward_binned has checked that this applies
    const size_t turns = (rows_of_b + rows_of_wave - 1) / rows_of_wave * a.B, per_block = 1024 / kWave;
    clear_blocks = (unsigned)((turns + per_block - 1) / per_block < 4096 ? (turns + per_block - 1) / per_block : 4096);
  }
  // scanning blocks for the most bins there can be (the plan kernel knows how many there are), 64 at most
  const size_t max_bins = (size_t)mb * slot_count(a.B, a.M);
  const unsigned scan_blocks = (max_bins + 1023) / 1024 < 64 ? (unsigned)((max_bins + 1023) / 1024) : 64u;
  hipLaunchKernelGGL(bin_scan_kernel, dim3(scan_blocks + clear_blocks), dim3(1024), 0, stream, ws, ca, (int)scan_blocks);
  if (hipError_t e = allow_lds(bin_fill_sorted_kernel, kSortedFillLds)) return e;
  hipLaunchKernelGGL(bin_fill_sorted_kernel, dim3(grid), dim3(kFillThreads), kSortedFillLds, stream, ws, (const float *)a.loc,
                     a.loc_stride, (const float *)a.attn, (float *)a.grad_loc, a.grad_loc_stride, (float *)a.grad_attn,
                     (float *)a.grad_score_out, a.B, a.M, a.L, a.Q, a.P, q_blocks, hist_cap, divs);
  return hipGetLastError();
}

// Binned backward of both stages (a.dist given) or of stage 2 alone (a.dist == nullptr, a.score_in /
// a.grad_score_out given).  Returns hipErrorNotSupported when the binned path does not apply and the
// caller should use launch_backward instead.
hipError_t launch_backward_binned(const BwdArgs &args, int dtype, void *workspace, size_t workspace_bytes,
                                  hipStream_t stream) {
  BwdArgs a = args;
  const int kind = bwd_kind(a);
  if (dtype == DFA3D_F64) return hipErrorNotSupported;
  if (kind == 0 && (a.loc_stride != 3 || a.grad_loc_stride != 3 || a.shape_stride != 3)) return hipErrorNotSupported;
  const size_t need = workspace_bytes_for(a, kind, dtype, true);
  if (need == 0 || workspace == nullptr || workspace_bytes < need || ((uintptr_t)workspace & 255) != 0)
    return hipErrorNotSupported;
  if (a.grad_bf16 && dtype != DFA3D_BF16) return hipErrorInvalidValue;
  if (a.clear_grads) {
    // clear_unstored writes 16-byte groups where a row is made of them: buffers on 16-byte boundaries,
    // or the direct kernels (which clear everything) take the call
    if ((((uintptr_t)a.grad_value | (uintptr_t)a.grad_dist) & 15) != 0) return hipErrorNotSupported;
  }
  const TileConfig cfg = tile_config_of(a, kind, dtype);
  BinLayout lay = bin_layout(a, cfg.ty, cfg.tx, sums_in_float(a, kind, dtype, cfg));
  if (lay.total > workspace_bytes) lay = bin_layout(a, cfg.ty, cfg.tx, false);      // no room for them
  const BinWorkspace ws = carve_workspace(workspace, lay);
  const bool float_sums = lay.total > lay.least;
  if (float_sums) {            // the kernels below see float gradients, which hold anything on entry
    a.grad_bf16 = 0; a.clear_grads = 1;
    a.grad_value = static_cast<char *>(workspace) + lay.value_sums;
    if (!shared_dist(a)) a.grad_dist = static_cast<char *>(workspace) + lay.dist_sums;
  }
  float *gd_heads = shared_dist(a) ? reinterpret_cast<float *>(static_cast<char *>(workspace) + lay.gd_heads) : nullptr;
  if (hipError_t e = run_binning(a, ws, cfg, gd_heads, stream)) return e;
  if (a.event_binned != nullptr) {
    if (hipError_t e = hipEventRecord((hipEvent_t)a.event_binned, stream)) return e;
  }
  const hipError_t e = dtype == DFA3D_F32 ? launch_tile_typed<float>(a, ws, cfg, gd_heads, stream)
                                          : launch_tile_typed<__hip_bfloat16>(a, ws, cfg, gd_heads, stream);
  if (e != hipSuccess) return e;
  if (gd_heads != nullptr)
    hipLaunchKernelGGL(head_sum_kernel, dim3(2048), dim3(256), 0, stream, gd_heads, args.grad_dist,
                       (size_t)a.B * a.S, a.M, a.D, args.grad_bf16 ? 1 : 0);
  if (float_sums) {
    const size_t rows = (size_t)a.B * a.S * a.M;
    hipLaunchKernelGGL(round_rows_kernel, dim3(2048), dim3(256), 0, stream, (const float4 *)a.grad_value, (uint2 *)args.grad_value,
                       rows * a.C / 4, (const float4 *)a.grad_dist, (uint2 *)args.grad_dist, gd_heads != nullptr ? 0 : rows * a.D / 4);
  }
  return hipGetLastError();
}

hipError_t launch_few_points_rounded(const BwdArgs &args, int dtype, void *workspace, size_t workspace_bytes, hipStream_t stream) {
  const size_t need = few_points_workspace_bytes(args);
  if (dtype != DFA3D_BF16 || need == 0 || workspace_bytes < need || ((uintptr_t)workspace & 15) != 0 ||
      (((uintptr_t)args.grad_value | (uintptr_t)args.grad_dist) & 7) != 0)
    return hipErrorNotSupported;
  BwdArgs a = args;
  a.grad_bf16 = 0;
  a.grad_value = workspace;
  a.grad_dist = static_cast<char *>(workspace) + few_points_value_bytes(a);
  const size_t value_elems = (size_t)a.B * a.S * a.M * a.C, dist_elems = few_points_dist_rows(a) * a.D;
  if (hipError_t e = launch_zero_fill(a.grad_value, value_elems * sizeof(float), a.grad_dist, dist_elems * sizeof(float), stream)) return e;
  if (hipError_t e = launch_backward(a, dtype, stream)) return e;
  hipLaunchKernelGGL(round_rows_kernel, dim3(2048), dim3(256), 0, stream, (const float4 *)a.grad_value, (uint2 *)args.grad_value, value_elems / 4,
                     (const float4 *)a.grad_dist, (uint2 *)args.grad_dist, dist_elems / 4);
  return hipGetLastError();
}

// Binned backward of stage 1 alone.
size_t binned_depth_score_backward_workspace_bytes(const DepthScoreBwdArgs &d, int dtype, int tile_hint) {
  BwdArgs a{};
  a.B = d.B; a.S = d.S; a.M = d.M; a.C = 0; a.D = d.D; a.L = d.L; a.Q = d.Q; a.P = d.P; a.tile_hint = tile_hint;
  return workspace_bytes_for(a, 2, dtype);
}

template <typename T>
static hipError_t launch_depth_tiles(const DepthScoreBwdArgs &d, const BinWorkspace &ws, const TileConfig &cfg, int stores, hipStream_t stream) {
  auto launch = [&](auto kern) -> hipError_t {
    if (hipError_t e = allow_lds(kern, cfg.lds)) return e;
    hipLaunchKernelGGL(kern, dim3(tile_grid(cfg.lds, cfg.block)), dim3(cfg.block), cfg.lds, stream, ws, (const T *)d.dist, (const T *)d.grad_score,
                       (float *)d.grad_dist, (float *)d.grad_loc3, d.B, d.S, d.M, d.D, d.L, d.Q, d.P, stores);
    return hipGetLastError();
  };
  if (cfg.block == 1024) return launch(tile_depth_backward_kernel<T, 1024>);
  if (cfg.block == 512) return launch(tile_depth_backward_kernel<T, 512>);
  return launch(tile_depth_backward_kernel<T, 256>);
}

hipError_t launch_depth_score_backward_binned(const DepthScoreBwdArgs &d, int dtype, void *workspace,
                                              size_t workspace_bytes, int tile_hint, int chunk_hint,
                                              void *event_binned, hipStream_t stream) {
  if (dtype == DFA3D_F64) return hipErrorNotSupported;
  BwdArgs a{};
  a.B = d.B; a.S = d.S; a.M = d.M; a.C = 0; a.D = d.D; a.L = d.L; a.Q = d.Q; a.P = d.P;
  a.shapes = d.shapes3; a.shape_stride = 3; a.level_start = d.level_start; a.loc = d.loc3; a.loc_stride = 3;
  a.attn = nullptr; a.grad_loc = d.grad_loc3; a.grad_loc_stride = 3; a.grad_attn = nullptr; a.grad_score_out = nullptr;
  a.tile_hint = tile_hint; a.chunk_hint = chunk_hint;
  a.grad_dist = d.grad_dist; a.clear_grads = d.clear;
  if (d.clear && ((uintptr_t)d.grad_dist & 15) != 0) return hipErrorNotSupported;      // as in launch_backward_binned
  const int stores = d.clear && (d.D & 3) == 0 ? 1 : 0;
  const size_t need = workspace_bytes_for(a, 2, dtype);
  if (need == 0 || workspace == nullptr || workspace_bytes < need || ((uintptr_t)workspace & 255) != 0)
    return hipErrorNotSupported;
  const TileConfig cfg = tile_config_of(a, 2, dtype);
  const BinWorkspace ws = carve_workspace(workspace, bin_layout(a, cfg.ty, cfg.tx, false));
  if (hipError_t e = run_binning(a, ws, cfg, nullptr, stream)) return e;
  if (event_binned != nullptr) {
    if (hipError_t e = hipEventRecord((hipEvent_t)event_binned, stream)) return e;
  }
  return dtype == DFA3D_F32 ? launch_depth_tiles<float>(d, ws, cfg, stores, stream) : launch_depth_tiles<__hip_bfloat16>(d, ws, cfg, stores, stream);
}

}  // namespace dfa3d
