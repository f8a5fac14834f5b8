// Forward kernels of the DFA3D operator for gfx950.
//
//   fwd_attention_kernel<..., FUSED=true>   depth-score sampling + weighted attention in one pass
//                                           (the reference runs two kernels and two slice copies:
//                                           multi_scale_3ddeformable_attn_function.py:279-303)
//   fwd_attention_kernel<..., FUSED=false>  stage 2 alone, scores given
//                                           (wms_deform_attn_cuda_kernel.cuh:240-303)
//   depth_score_kernel                      stage 1 alone
//                                           (ms_depth_score_sample_cuda_kernel.cuh:94-148)
#include <algorithm>
#include <type_traits>

#include "dfa3d_device.h"
#include "dfa3d_launch.h"

namespace dfa3d {

// How the wavefronts share the units: `upw` units of L * P points each, a power of two, or three times one, so that the
// row slots of phase B can be dealt to them evenly; `chunks` rounds of 64 points where one unit has more.
struct FwdShape { int LP, upw, chunks; };
__host__ __device__ inline FwdShape fwd_shape(int L, int P, int upw) {
  return FwdShape{L * P, upw, upw > 1 ? 1 : (L * P + kWave - 1) / kWave};
}
constexpr int kMaxUnitsPerWave = 16;
constexpr int kLdsRowsBlock = 1024;    // threads of a workgroup that holds its (batch, head)'s value rows in LDS
constexpr int kTasksPerWave = kWave * 4 + 32;      // room for its tasks, padding included (task_run)
// Places that a row slot's run of a unit's tasks takes.  Two runs are read at 16 bytes each at a time, so they start 16 bytes apart on the LDS banks
// (two places more than a multiple of four), but for 21 points a unit on eight slots, for which there is no room.
__device__ __forceinline__ int task_run(int longest, int runs) {
  const int padded = ((longest + 1) & ~3) + 2;
  return runs * padded <= kTasksPerWave ? padded : longest;
}

// Phase B of the forward pass: acc += sum of w * row over a row slot's tasks.  LPR lanes of VEC channels take a row; the
// wavefront's 64/LPR row slots may share a unit, each with its tasks, `step` apart, or work on units of their own.  `all` tasks every slot
// of the unit has, `most` the longest run (both uniform), `mine` this slot's.  Eight rows per lane are in flight, whatever the length
// of the list: a unit of 8 points has 32 tasks, and walking it one row at a time waited for memory once per row.  A batch is summed in
// two chains and added to acc as a whole, which keeps the longest chain of additions of a unit at about what a tree over the
// row slots has.  `rows` reads this lane's channels of the row at a byte offset; `none` is the offset of a row of zeros.
template <typename A, int VEC, typename Rows>
__device__ __forceinline__ void gather_rows(const Rows &rows, uint32_t none, const Task<A> *tasks, int step, int all, int most,
                                            int mine, A (&acc)[VEC]) {
  constexpr int U = 8, UT = 4;
  int t = 0;                                             // uniform
  for (; t + U <= all; t += U) {
    Task<A> e[U];
#pragma unroll
    for (int j = 0; j < U; ++j) e[j] = tasks[(t + j) * step];
    A v[U][VEC];
#pragma unroll
    for (int j = 0; j < U; ++j) rows(e[j].off, v[j]);
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      A s0 = e[0].w * v[0][i], s1 = e[1].w * v[1][i];
#pragma unroll
      for (int j = 2; j < U; j += 2) { s0 += e[j].w * v[j][i]; s1 += e[j + 1].w * v[j + 1][i]; }
      acc[i] += s0 + s1;
    }
  }
  for (; t < most; t += UT) {                            // the rest: no load is issued that no slot has a row for
    Task<A> e[UT];
    A v[UT][VEC];
#pragma unroll
    for (int j = 0; j < UT; ++j) {
      e[j].off = none; e[j].w = 0;
#pragma unroll
      for (int i = 0; i < VEC; ++i) v[j][i] = 0;
      if (t + j < most) {                                // uniform
        const bool has = t + j < mine;
        e[j] = tasks[has ? (t + j) * step : 0];
        if (!has) { e[j].off = none; e[j].w = 0; }
        rows(e[j].off, v[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < UT; ++j) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] += e[j].w * v[j][i];
    }
  }
}
// x summed over the lanes that differ in the bits FROM, 2 FROM, ... below `to` (uniform) of their number
template <int FROM, int VEC> __device__ __forceinline__ void sum_over_slots(int to, float (&x)[VEC]) {
  if constexpr (FROM < kWave) {
    if (FROM < to) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const int v = __float_as_int(x[i]);
        if constexpr (FROM == 8) {
          x[i] += __int_as_float(__builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true));              // row_ror:8
        } else if constexpr (FROM == 16) {
          const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
          x[i] = __int_as_float(r[0]) + __int_as_float(r[1]);
        } else if constexpr (FROM == 32) {
          const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
          x[i] = __int_as_float(r[0]) + __int_as_float(r[1]);
        } else {
          x[i] += __shfl_xor(x[i], FROM, kWave);
        }
      }
      sum_over_slots<2 * FROM, VEC>(to, x);
    }
  }
}
template <int FROM, int VEC> __device__ __forceinline__ void sum_over_slots(int to, double (&x)[VEC]) {
  for (int off = FROM; off < to; off <<= 1) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) x[i] += __shfl_xor(x[i], off, kWave);
  }
}

// ---------------------------------------------------------------------------------------
// Fused / stage-2 forward.
// grid: M * B * ceil(Q / queries_per_block) blocks; block id % M = head, so that with the
// round-robin placement of workgroups on the 8 XCDs each XCD's L2 serves one head (M = 8).
//
// Bound by the rate at which a CU's front end turns gathered lines around, and by the L2 misses of the finest level, once
// enough rows are in flight.  In phase B the row slots are dealt to the wavefront's units (8 units of 8 points: one slot
// each), so that lists of any length keep eight rows per lane in flight and a unit's sum crosses lanes only where
// it has several slots.  Before, the whole wavefront walked one unit after the other, and short units one row at a time:
//   6 x 10000 queries, 4 levels from 116 x 200, points around the query   664 -> 617 us
//   6 x 4000 queries, one level of 8 points (training step)               261 -> 239 us
//   2 x 40000 queries, plain attention, 4 points (training step)          461 -> 427 us
//
// A CU's L1 answers in the order in which it was asked, and has 256 lines: 256 lines in flight divided by the latency of the farthest
// is all that it brings, whichever lines the caches hold.  So where a (batch, head)'s value rows fit in LDS (IN_LDS: small
// maps), a workgroup of 16 wavefronts brings them there once and walks through a share of the queries: four of a point's eight lines
// less.  6 x 4000 queries, one level of 23 x 40, 8 points: 53.4 -> 41.0 us (uniform), 41.0 -> 36.4 (points around the query), bfloat16
// 56.6 -> 51.8, one distribution for all heads 49.1 -> 40.3, plain attention 36.3 -> 28.7; 64 channels, 4 x 4000, 15 x 24: 52.2 -> 32.5.
// On larger maps the coarser levels' rows: 6 x 10000 queries, four levels from 116 x 200, 8 points (one level in LDS): 915 -> 864 us (884 on
// another card), points around the query 605 -> 571; bfloat16 (two levels) 842 -> 787, 572 -> 505; plain attention 297 -> 261.  Groups are taken,
// not dealt: dealt, a workgroup's slowest wavefront held up the CU (883, 614).  Tried with it and not kept: two workgroups of 8, 10 or 12
// wavefronts per CU (908, 870, 1031; 596, 625, 706), 16 gathers in flight (880, 623), the next group's locations asked for ahead (850, 581;
// bfloat16 951) or brought to the L2 by scalar loads (874, 587); the same workgroups without rows in LDS: 942, 603.
//
// A quarter of the instructions found places: divisions by the points of a unit and of a level, 64-bit indexes, a product per corner.  What a
// lane's point has from its place in the group and its level is kept from group to group (IN_LDS), the group's part is in scalars, corners
// are a row and a column apart, and a slot's tasks lie side by side (656 -> 498 vector instructions per 64 points).  And the wavefronts of a SIMD,
// which meet at the L1, go by what they hold: one that gathers value rows comes before one that looks for its points' corners, and that before one
// that begins a group (s_setprio 2, 1, 0; the other way round 3120 us for the 3047 of two steps and 3000 of three, 24 planes and 128 bins).
// Together, one card, us:
//   6 x 10000 queries, 4 levels from 116 x 200, 8 points: 885 -> 872, around the query 574 -> 571 (bfloat16 483 -> 476), plain attention 436 -> 389;
//   6 x 40000 clustered, 128 bins: 3067 -> 3000; the two separate stages without gradients, 112 bins: 1013 -> 936; one level of 23 x 40: 39.7 -> 38.0;
// Where a workgroup has one group (not IN_LDS) there are none: plain attention, 4 points, 2 x 40000 queries on 200 x 200 gained from them (103 -> 96),
// 4 x 10000 on 116 x 197 lost (59.5 -> 63.7).
//
// Six wavefronts a SIMD (kFwdWaves: 80 vector registers, none of which is spilled; of the scalars 64 are with depth taps, 84 with EARLY, to vector
// lanes) where five were: plain attention, 3 x 3 points 33.5 -> 30.1; one distribution for all heads, packed, four levels of 8 points, around the
// query 125 -> 118.5, anywhere 150 -> 144, 9000 queries, 116 x 197 326 -> 315; other calls with runs +- 0.5 %.  Seven spill (118.5 -> 141).
// --------------------------------------------------------------------------------------- wavefronts a SIMD that the registers have to leave room
// for (1: as the compiler likes)
template <typename T, int VEC, bool IN_LDS> constexpr int kFwdWaves = !IN_LDS && sizeof(T) == 4 && VEC == 4 ? 6 : 1;
// SCALAR: the first by_scalar points of a unit take their depth taps by scalar loads (points_by_scalar)
template <typename T, typename A, int VEC, int LPR, bool FUSED, bool IN_LDS, bool IN_TURN, bool EARLY, bool SCALAR = false>
__global__ __launch_bounds__(IN_LDS ? kLdsRowsBlock : kBlock, (kFwdWaves<T, VEC, IN_LDS>)) void fwd_attention_kernel(
    const T *__restrict__ value, const T *__restrict__ dist, const int64_t *__restrict__ shapes, int shape_stride,
    const int64_t *__restrict__ level_start, const A *__restrict__ loc, int loc_stride,
    const A *__restrict__ attn, const T *__restrict__ score_in, T *__restrict__ out, T *__restrict__ score_out,
    A *__restrict__ weight_update, const T *__restrict__ packed_arg, int Md, int B, int S, int M, int C, int D, int L,
    int Q, int P, int upw, int iters, int q_blocks, int once, int lds_rows, int by_scalar) {
  // packed: the head-shared distribution as dfa3d_pack_dist lays it out (D >= 2), or nullptr
  __shared__ LevelTable tab;
  constexpr int WAVES = (IN_LDS ? kLdsRowsBlock : kBlock) / kWave;
  __shared__ __align__(16) Task<A> s_tasks[WAVES][kTasksPerWave];
  __shared__ int s_next;                                      // IN_LDS: the workgroup's next group of units
  extern __shared__ __align__(16) unsigned char s_rows[];    // IN_LDS: value rows [key0, S) of (b, m), then a row of zeros

  const FwdShape ws = fwd_shape(L, P, upw);
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int m = blockIdx.x % M;
  const int rest = blockIdx.x / M;
  const int qb = rest % q_blocks, b = rest / q_blocks;
  const int row_slot = lane / LPR, cl = lane % LPR;
  const int passes = (C + VEC * LPR - 1) / (VEC * LPR);
  Task<A> *tasks = s_tasks[wave];
  const int q_per_iter = WAVES * ws.upw;
  // This lane's point of chunk `chunk` of a group: unit and point within the unit, and the point's number counted from the group's
  // first unit's first point.  The same for all groups (of one chunk): what a group adds is in scalars.
  struct Place { int ul, lp; uint32_t idx; };
  auto place = [&](int chunk) {
    const int pt = chunk * kWave + lane, ul = pt / ws.LP, lp = pt - ul * ws.LP;
    return Place{ul, lp, (uint32_t)ul * (uint32_t)(M * ws.LP) + (uint32_t)lp};
  };
  auto first_point = [&](int q0) { return ((size_t)(b * (size_t)Q + q0) * M + m) * ws.LP; };      // of the group that begins with query q0
  struct Operands { A x, y, z, a; };
  auto fetch = [&](int q0, const Place &pl) {
    Operands o{0, 0, 0, 0};
    if (pl.ul < min(ws.upw, Q - q0)) {
      const size_t first = first_point(q0);
      const A *pt = reinterpret_cast<const A *>(reinterpret_cast<const char *>(loc + first * loc_stride) + pl.idx * (uint32_t)(loc_stride * (int)sizeof(A)));
      const A *pa = reinterpret_cast<const A *>(reinterpret_cast<const char *>(attn + first) + pl.idx * (uint32_t)sizeof(A));
      if (!IN_LDS && (once & 1) != 0) {                         // uniform
        asm volatile("");                                       // (or the compiler merges the branches into plain loads)
        o.x = __builtin_nontemporal_load(pt); o.y = __builtin_nontemporal_load(pt + 1);
        if (FUSED) o.z = __builtin_nontemporal_load(pt + 2);
        asm volatile("");
      } else {
        o.x = pt[0]; o.y = pt[1];
        if (FUSED) o.z = pt[2];
      }
      if (!IN_LDS && (once & 2) != 0) {
        asm volatile("");
        o.a = __builtin_nontemporal_load(pa);
        asm volatile("");
      } else {
        o.a = *pa;
      }
    }
    return o;
  };
  // EARLY, no depth taps: the first group's are on their way while the level table is (launch_fwd_cfg)
  constexpr bool kAhead = EARLY && !FUSED;
  Place pl = place(0);
  const Operands first = kAhead ? fetch((qb * iters * WAVES + wave) * ws.upw, pl) : Operands{0, 0, 0, 0};
  // phase B: `par` units at a time, `spu` row slots each
  constexpr int RPI = kWave / LPR;
  const int par = min(ws.upw & -ws.upw, RPI), spu = RPI / par, spu_log2 = 31 - __builtin_clz(spu);
  // Task i of a unit belongs to its slot i % spu.  A slot's tasks lie side by side, so that a batch of them is read from one address.
  const int unit_points = ws.upw == 1 ? min(kWave, ws.LP) : ws.LP;                 // of a chunk
  const int run = task_run((unit_points * 4 + spu - 1) >> spu_log2, ws.upw * spu);
  const int my_point = ws.upw == 1 ? lane : pl.lp, my_unit = ws.upw == 1 ? 0 : pl.ul;
  const bool my_tasks = my_point < unit_points && my_unit < ws.upw;
  // IN_TURN: as they come instead, a unit's side by side.
  const int unit_room = unit_points * 4 + (ws.upw == 1 ? 0 : 2);
  Task<A> *const to = tasks + (IN_TURN ? my_unit * unit_room + my_point * 4
                                       : (my_unit * spu + ((my_point * 4) & (spu - 1))) * run + ((my_point * 4) >> spu_log2));
  const int to1 = !IN_TURN && spu > 1 ? run : 1, to2 = !IN_TURN && spu > 2 ? 2 * run : !IN_TURN && spu == 2 ? 1 : 2;
  const int to3 = !IN_TURN && spu == 2 ? run + 1 : to1 + to2;
  const int part = row_slot % spu;

  // EARLY, depth taps: no level table, each wavefront reads the levels' sizes as scalars (launch_fwd_cfg)
  constexpr bool kOwnLevels = EARLY && FUSED;
  int cells = 0;
  if constexpr (!kOwnLevels) {
    load_level_table(tab, shapes, shape_stride, level_start, L, S, FUSED ? D : 0);
    if (FUSED && packed_arg != nullptr) {                              // uniform
      load_cell_starts(tab, L);
      cells = tab.cell[L];
    }
  } else if (packed_arg != nullptr) {
    for_each_level(shapes, shape_stride, level_start, L, S, D, [&](int, const LevelSize &z) { cells += (z.H + 1) * (z.W + 1); });
  }
  // The packed table was sized on the host for levels that share no keys (at most 2 S + 2 L cells).  A level
  // table whose levels overlap can ask for more: then the table is not used (nor was it written) and the taps
  // come from dist itself.
  const T *packed = (FUSED && packed_arg != nullptr && cells <= packed_cell_capacity(S, L)) ? packed_arg : nullptr;

  const rsrc_t value_r = make_rsrc(value + (size_t)b * S * M * C, (size_t)S * M * C * sizeof(T));
  const rsrc_t dist_r = make_rsrc(FUSED ? dist + (size_t)b * S * Md * D : nullptr,
                                  FUSED ? (size_t)S * Md * D * sizeof(T) : 0);
  const int md = Md == 1 ? 0 : m;                                    // head whose distribution this head reads
  const size_t packed_slice = (FUSED && packed != nullptr) ? (size_t)cells * D * 4 : 0;   // elements per batch element
  const rsrc_t packed_r = make_rsrc(packed_slice ? packed + (size_t)b * packed_slice : nullptr, packed_slice * sizeof(T));
  // IN_LDS: levels l0, l0 + 1, ... , whose keys are among the last lds_rows ones
  int l0 = IN_LDS ? L : 0, key0 = S;
  if constexpr (IN_LDS) {
    if (threadIdx.x == 0) s_next = 0;
    while (l0 > 0 && tab.start[l0 - 1] >= S - lds_rows) { --l0; key0 = min(key0, tab.start[l0]); }
    const int n_rows = S - key0;
    // LPR lanes per row as in phase B
    for (int pass = 0; pass < passes; ++pass) {
      const int chan = (pass * LPR + cl) * VEC;
      if (chan >= C) break;
      for (int s0 = wave * RPI + row_slot; s0 <= n_rows; s0 += 4 * WAVES * RPI) {
        RawPiece<VEC * sizeof(T)> piece[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int s = s0 + j * WAVES * RPI;
          piece[j].ld(value_r, s < n_rows ? (uint32_t)((((key0 + s) * M + m) * C + chan) * (int)sizeof(T)) : kNoRow);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int s = s0 + j * WAVES * RPI;
          if (s <= n_rows) *reinterpret_cast<decltype(piece[j].w) *>(s_rows + (s * C + chan) * (int)sizeof(T)) = piece[j].w;
        }
      }
    }
    __syncthreads();
  }
  const uint32_t zero_row = (uint32_t)((S - key0) * C * (int)sizeof(T));
  // What the geometry of a lane's point takes from its level: sizes, and byte offsets (modulo 2^32) of value rows and distributions, those of
  // a map's pixel (y, x) being base + y * row + x * col.  Kept from group to group, like the lane's place.
  struct Level { int H, W, Dd, cell; uint32_t v_col, v_row, v_base, d_row, d_base; bool in_lds; };
  const uint32_t d_col = (uint32_t)(Md * D * (int)sizeof(T));
  const bool whole_words = (S * Md * D & 1) == 0 && ((uintptr_t)dist & 3) == 0;      // 2-byte elements: what each batch element has of dist
  auto level = [&](const Place &at) {
    const int l = min(at.lp / P, L - 1);
    Level v{};
    int start = 0;
    if constexpr (kOwnLevels) {
      int cell = 0;
      for_each_level(shapes, shape_stride, level_start, L, S, D, [&](int i, const LevelSize &z) {
        const bool here = i == l;
        v.H = here ? z.H : v.H; v.W = here ? z.W : v.W; v.Dd = here ? z.Dd : v.Dd; v.cell = here ? cell : v.cell;
        start = here ? z.start : start;
        cell += (z.H + 1) * (z.W + 1);
      });
    } else {
      v.H = tab.H[l]; v.W = tab.W[l]; v.Dd = tab.Dd[l]; start = tab.start[l];
      v.cell = FUSED && packed != nullptr ? tab.cell[l] : 0;
    }
    v.in_lds = IN_LDS && l >= l0;
    v.v_col = (uint32_t)((v.in_lds ? C : M * C) * (int)sizeof(T));
    v.v_row = (uint32_t)v.W * v.v_col;
    v.v_base = v.in_lds ? (uint32_t)((start - key0) * C * (int)sizeof(T)) : (uint32_t)((start * M + m) * C * (int)sizeof(T));
    v.d_row = (uint32_t)v.W * d_col;
    v.d_base = (uint32_t)((start * Md + md) * D * (int)sizeof(T));
    return v;
  };
  Level lv{};
  if (IN_LDS) lv = level(pl);                                // (else worked out where it is needed: most workgroups have one group, and registers are wavefronts)

  // Groups of units, WAVES to a round; rounds are dealt to the workgroups of a (batch, head) in turn, so that what they gather at a
  // time lies together.  IN_LDS: a workgroup's wavefronts take its next group each.
  for (int it = 0; IN_LDS || it < iters; ++it) {
    int round = qb * iters + it, slot = wave;
    if constexpr (IN_LDS) {
      int n = 0;
      if (lane == 0) n = atomicAdd(&s_next, 1);
      n = __builtin_amdgcn_readfirstlane(n);
      if (n >= iters * WAVES) break;
      round = n / WAVES * q_blocks + qb;
      slot = n % WAVES;
    }
    const int q0 = round * q_per_iter + slot * ws.upw;               // first query of this wave's group
    if (q0 >= Q) {                                                   // wave-uniform
      if (IN_LDS) continue;
      break;
    }
    A wu_unit = 0;                                                   // upw == 1: the unit's sum over its chunks
    for (int pass = 0; pass < passes; ++pass) {
      const int chan = (pass * LPR + cl) * VEC;
      const bool chan_ok = chan < C;
      const uint32_t chan_off = chan_ok ? (uint32_t)(chan * sizeof(T)) : kNoChan, lds_chan = chan_ok ? chan_off : 0u;
      auto rows = [&](uint32_t off, A (&v)[VEC]) { RowVec<T, A, VEC>::ld(value_r, off + chan_off, v); };
      auto rows_in_lds = [&](uint32_t off, A (&v)[VEC]) { lds_row<T, A, VEC>(s_rows + off + lds_chan, v); };
      A acc[VEC];
#pragma unroll
      for (int v = 0; v < VEC; ++v) acc[v] = 0;

      for (int chunk = 0; chunk < ws.chunks; ++chunk) {
        if (IN_LDS) __builtin_amdgcn_s_setprio(0);                       // a group begins
        // ---------------- phase A: one lane per sampling point ----------------
        if (ws.chunks > 1) pl = place(chunk);                // uniform
        const int ul = pl.ul, lp = pl.lp, q = q0 + ul;       // unit within group, point within unit
        const bool live = ul < min(ws.upw, Q - q0);
        Operands in = first;
        if (!kAhead || it > 0 || pass > 0 || chunk > 0) in = fetch(q0, pl);      // uniform
        if (!IN_LDS || ws.chunks > 1) lv = level(pl);
        Task<A> t4[4];
        A wu = 0;
        const uint32_t none = lv.in_lds ? zero_row : kNoRow;
#pragma unroll
        for (int k = 0; k < 4; ++k) { t4[k].off = none; t4[k].w = 0; }
        if (live) {
          const A a = in.a;
          if (IN_LDS) __builtin_amdgcn_s_setprio(1);
          const Grid2D<A> g = locate_grid<A>(in.x, in.y, lv.H, lv.W);
          A sc[4];
          if (FUSED) {
            const DepthTap<A> tap = locate_depth<A>(in.z, lv.Dd);
            if (packed != nullptr) {                                // uniform: all eight taps from one line
              const DepthPair<A> pair(tap, D);
              const int cell = lv.cell + (g.h0 + 1) * (lv.W + 1) + g.w0 + 1;
              A x4[4], y4[4];
              PackedTap<T>::ld(packed_r, (g.inside && tap.inside) ? (uint32_t)((cell * D + pair.db) * 4 * (int)sizeof(T)) : kNoRow,
                               x4, y4);
#pragma unroll
              for (int k = 0; k < 4; ++k) sc[k] = pair.score(x4[k], y4[k]);
            } else {
              grid_scores<T, A, SCALAR>(dist_r, g, tap, lv.d_base, lv.d_row, d_col, D, whole_words, sc, dist + (size_t)b * S * Md * D,
                                         (uint32_t)(S * Md * D * (int)sizeof(T)) - 8, lp < by_scalar);
            }
            if (score_out != nullptr && pass == 0) {
              T *so = reinterpret_cast<T *>(reinterpret_cast<char *>(score_out + first_point(q0) * 4) + pl.idx * (uint32_t)(4 * sizeof(T)));
              if constexpr (sizeof(T) == 4) {                     // one 16-byte store
                typedef float f4 __attribute__((ext_vector_type(4)));
                f4 v4 = {(float)sc[0], (float)sc[1], (float)sc[2], (float)sc[3]};
                __builtin_nontemporal_store(v4, reinterpret_cast<f4 *>(so));
              } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) Elem<T>::st(so + k, sc[k]);
              }
            }
            wu = a * ((sc[0] + sc[1] + sc[2] + sc[3]) * (A)0.25);
          } else {
            // no scores given: plain deformable attention
#pragma unroll
            for (int k = 0; k < 4; ++k) sc[k] = (A)1;
            if (score_in != nullptr) {                              // uniform
              const T *si = reinterpret_cast<const T *>(reinterpret_cast<const char *>(score_in + first_point(q0) * 4) + pl.idx * (uint32_t)(4 * sizeof(T)));
#pragma unroll
              for (int k = 0; k < 4; ++k) sc[k] = Elem<T>::ld(si + k);
            }
          }
          const uint32_t at = (uint32_t)g.h0 * lv.v_row + (uint32_t)g.w0 * lv.v_col + lv.v_base;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t off = at + (k >= 2 ? lv.v_row : 0) + (k == 1 || k == 2 ? lv.v_col : 0);
            const A w = g.bil(k) * sc[k] * a;
            t4[k].off = g.on(k) ? off : none;
            t4[k].w = g.on(k) ? w : (A)0;
          }
        }
        if (FUSED && weight_update != nullptr && pass == 0) {      // wave-uniform
          // sum over the lanes of each unit: lane i gathers lanes [i, i + 2^k) of its own unit
          const int seg = ws.upw == 1 ? kWave : ws.LP, pos = ws.upw == 1 ? lane : lp;
          for (int off = 1; off < seg; off <<= 1) {
            const A up = __shfl_down(wu, off, kWave);
            if (pos + off < seg) wu += up;
          }
          if (ws.upw == 1) {
            wu_unit += wu;                                         // lane 0 holds the chunk's sum
            if (chunk == ws.chunks - 1 && lane == 0) weight_update[((size_t)b * Q + q0) * M + m] = wu_unit;
          } else if (live && lp == 0) {
            weight_update[((size_t)b * Q + q) * M + m] = wu;
          }
        }
        wave_lds_handover();     // previous phase B has consumed the task list
        if (my_tasks) {
          to[0] = t4[0]; to[to1] = t4[1]; to[to2] = t4[2]; to[to3] = t4[3];
        }
        wave_lds_handover();

        if (IN_LDS) __builtin_amdgcn_s_setprio(2);
        // ---------------- phase B: lanes over channels ----------------
        for (int u0 = 0; u0 < ws.upw; u0 += par) {              // one round, or three (one where a unit takes several chunks)
          const int u = u0 + row_slot / spu;
          const int n = (ws.upw == 1 ? min(kWave, ws.LP - chunk * kWave) : ws.LP) * 4;
          const int far = IN_LDS ? min(max((l0 * P - chunk * kWave) * 4, 0), n) : n;
          const int n_far = (far + spu - 1 - part) >> spu_log2;
          const Task<A> *mine = tasks + (IN_TURN ? u * unit_room + part : (u0 * spu + row_slot) * run);
          gather_rows<A, VEC>(rows, kNoRow, mine, IN_TURN ? spu : 1, far >> spu_log2, (far + spu - 1) >> spu_log2, n_far, acc);
          if constexpr (IN_LDS)
            gather_rows<A, VEC>(rows_in_lds, zero_row, mine + n_far, 1, (n - far) >> spu_log2, (n - far + spu - 1) >> spu_log2,
                                ((n + spu - 1 - part) >> spu_log2) - n_far, acc);
          if (chunk == ws.chunks - 1) {
            if (IN_LDS) __builtin_amdgcn_s_setprio(1);
            sum_over_slots<LPR, VEC>(spu * LPR, acc);
            if (part == 0 && chan_ok && q0 + u < Q) {
              T *group_out = out + ((size_t)(b * (size_t)Q + q0) * M + m) * C;
              RowVec<T, A, VEC>::st(reinterpret_cast<T *>(reinterpret_cast<char *>(group_out) + ((uint32_t)u * (uint32_t)(M * C) + (uint32_t)chan) * (uint32_t)sizeof(T)), acc);
            }
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc[i] = 0;
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------------
// Stage 1 alone: one lane per sampling point.  Block id -> (head, block of queries, group of levels, batch) with head =
// block % M, as in the attention kernels: the distributions one XCD's L2 sees are those of one head.
//
// Bound by the gathers, a cache line for each of a point's four pairs of bins.  So a group is one level: what an XCD reads at a time
// is then one head's distributions of one level, which the L2 holds but for the finest, where all levels together (13.8 MB
// with 112 bins) pushed one another out.  And a lane takes four points at a time, sixteen gathers in flight, where a block has
// them; it has where the launch would be more than 4096 blocks of 1024 points.  6 x 9502 queries, four levels from
// 116 x 200, 8 points (14.6 M points), 112 bins 536 -> 496 us level by level, 470 with four points at a time; 64 bins 514 / 440 /
// 403, 16 bins 439 / 372 / 331, bfloat16 446 / 432 / 402.  As it stands, with
// non-temporal stores of the scores: 468, 407, 272 and bfloat16 404.  Below four points per level a level's locations and scores
// are less than half a line each: all levels together (2 points: 53 against 55 us for 1.3 M points).
// ---------------------------------------------------------------------------------------
struct DepthScoreShape { int levels, points; };          // levels per group, points per block at most
__host__ __device__ inline DepthScoreShape depth_score_shape(int B, int M, int L, int Q, int P) {
  return DepthScoreShape{P >= 4 ? 1 : L, (long long)B * M * L * Q * P > 4096LL * 1024 ? 1024 : 256};
}
__host__ __device__ inline int depth_score_queries(const DepthScoreShape &s, int P) { return s.points > s.levels * P ? s.points / (s.levels * P) : 1; }
template <typename T, typename A>
__global__ __launch_bounds__(kBlock) void depth_score_kernel(
    const T *__restrict__ dist, const int64_t *__restrict__ shapes3, const int64_t *__restrict__ level_start,
    const A *__restrict__ loc3, T *__restrict__ score, int B, int S, int M, int D, int L, int Q, int P) {
  __shared__ LevelTable tab;
  load_level_table(tab, shapes3, 3, level_start, L, S, D);
  const DepthScoreShape shape = depth_score_shape(B, M, L, Q, P);
  const int queries = depth_score_queries(shape, P), q_blocks = (Q + queries - 1) / queries, groups = L / shape.levels;
  const int m = blockIdx.x % M;
  int rest = blockIdx.x / M;
  const int q0 = rest % q_blocks * queries;
  rest /= q_blocks;
  const int l0 = rest % groups * shape.levels, b = rest / groups;
  const int per_query = shape.levels * P, n = min(queries, Q - q0) * per_query;
  const rsrc_t dist_r = make_rsrc(dist + (size_t)b * S * M * D, (size_t)S * M * D * sizeof(T));
  // points i, i + kBlock, ... N of them
  auto points = [&](int i, auto count) {
    constexpr int N = decltype(count)::value;
    A x[N], y[N], z[N];
    size_t gp[N];
    int l[N];
#pragma unroll
    for (int r = 0; r < N; ++r) {
      const int ql = (i + r * kBlock) / per_query, lp = i + r * kBlock - ql * per_query;
      l[r] = shape.levels == 1 ? l0 : lp / P;
      gp[r] = (((size_t)b * Q + q0 + ql) * M + m) * ((size_t)L * P) + l0 * P + lp;
      const A *pl = loc3 + gp[r] * 3;
      x[r] = pl[0]; y[r] = pl[1]; z[r] = pl[2];
    }
    A sc[N][4];
#pragma unroll
    for (int r = 0; r < N; ++r) {
      const Point2D<A> g = locate_2d<A>(x[r], y[r], tab.H[l[r]], tab.W[l[r]], tab.start[l[r]]);
      const DepthTap<A> tap = locate_depth<A>(z[r], tab.Dd[l[r]]);
      A lo[4], hi[4];
      corner_scores<T, A>(dist_r, g.key, tap, m, M, D, sc[r], lo, hi);
    }
#pragma unroll
    for (int r = 0; r < N; ++r) {
      T *so = score + gp[r] * 4;
      // non-temporal: the scores leave the L2 to the distributions
      if constexpr (std::is_same<T, float>::value) {
        typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
        __builtin_nontemporal_store((f4){sc[r][0], sc[r][1], sc[r][2], sc[r][3]}, reinterpret_cast<f4 *>(so));
      } else if constexpr (std::is_same<T, __hip_bfloat16>::value) {
        typedef uint32_t u2 __attribute__((ext_vector_type(2), aligned(2)));
        __builtin_nontemporal_store((u2){pack_bf16x2(sc[r][0], sc[r][1]), pack_bf16x2(sc[r][2], sc[r][3])}, reinterpret_cast<u2 *>(so));
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) Elem<T>::st(so + k, sc[r][k]);
      }
    }
  };
  int i = threadIdx.x;
  for (; i - (int)threadIdx.x + 4 * kBlock <= n; i += 4 * kBlock) points(i, std::integral_constant<int, 4>());      // uniform
  for (; i < n; i += kBlock) points(i, std::integral_constant<int, 1>());
}

// ---------------------------------------------------------------------------------------
// Packs a head-shared distribution (B,S,1,D) for the forward's depth taps: see load_cell_starts for the layout.
// One thread per (cell, bin): four gathered values, one 16-byte (bfloat16: 8-byte) store; consecutive threads
// write consecutive addresses.
// ---------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void pack_dist_kernel(
    const T *__restrict__ dist, const int64_t *__restrict__ shapes3, const int64_t *__restrict__ level_start,
    T *__restrict__ packed, int B, int S, int D, int L) {
  __shared__ LevelTable tab;
  load_level_table(tab, shapes3, 3, level_start, L, S, D);
  load_cell_starts(tab, L);
  if (tab.cell[L] > packed_cell_capacity(S, L)) return;       // overlapping levels: more cells than the table holds; the forward then ignores it
  const size_t cells = (size_t)tab.cell[L];
  const size_t n = (size_t)B * cells * D;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int d = (int)(i % D);
    const size_t bc = i / D;
    const int cell = (int)(bc % cells), b = (int)(bc / cells);
    int l = 0;
    while (l + 1 < L && cell >= tab.cell[l + 1]) ++l;
    const int H = tab.H[l], W = tab.W[l], local = cell - tab.cell[l];
    const int h0 = local / (W + 1) - 1, w0 = local % (W + 1) - 1;
    const T *lvl = dist + ((size_t)b * S + tab.start[l]) * D + d;
    T v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int h = h0 + (k >= 2 ? 1 : 0), w = w0 + ((k == 1 || k == 2) ? 1 : 0);      // slots LT, RT, RB, LB
      const bool in = h >= 0 && h < H && w >= 0 && w < W;
      v[k] = in ? lvl[(size_t)(h * W + w) * D] : T(0.f);
    }
    T *dst = packed + i * 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[k] = v[k];
  }
}

template <typename T>
static hipError_t launch_pack_typed(const void *dist, const int64_t *shapes3, const int64_t *level_start, void *packed,
                                    int B, int S, int D, int L, hipStream_t stream) {
  hipLaunchKernelGGL((pack_dist_kernel<T>), dim3(256 * 16), dim3(256), 0, stream, (const T *)dist, shapes3, level_start,
                     (T *)packed, B, S, D, L);
  return hipGetLastError();
}

hipError_t launch_pack_dist(const void *dist, const int64_t *shapes3, const int64_t *level_start, void *packed, int B,
                            int S, int D, int L, int dtype, hipStream_t stream) {
  switch (dtype) {
    case DFA3D_F32: return launch_pack_typed<float>(dist, shapes3, level_start, packed, B, S, D, L, stream);
    case DFA3D_BF16: return launch_pack_typed<__hip_bfloat16>(dist, shapes3, level_start, packed, B, S, D, L, stream);
  }
  return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------
// Whether value rows are brought to LDS: those of the last `rows` keys as far as they are whole levels, by `parts` workgroups per (batch, head),
// one per CU; parts = 0: all rows are gathered from memory.  For rows of whole groups of four channels, up to 64, of 4- or 2-byte elements.
//   * The whole map fits: the workgroups of all (batch, head) run at once, where each has at least as many points as it brings
//     rows.  Kernel, us, memory and LDS, 920 rows of 32 channels, points per workgroup 500: 8.6, 11.0   640: 11.6, 12.9   800: 11.9, 12.9
//     1000: 13.3, 12.6   1600: 19.6, 17.2   6400: 53.4, 41.0; 504 rows, 720 points: 10.7, 10.1; 384 rows, 800 points: 10.9, 10.6.
//   * The coarser levels of a pyramid fit (the level sizes are on the device; each is taken for a quarter of the one before): one
//     (batch, head) at a time on an XCD, as its L2 holds no more, so M has to divide 8 or be a multiple of it.  What a workgroup spends on
//     its start, its end and fewer wavefronts is worth some thousand points; LDS saves half of the lines of a point on a level that it holds
//     (plain attention all), which cost less where rows are bfloat16.  Memory over LDS, maps from 58 x 100, 80 x 128 and 116 x 200 in
//     three or four levels, locations anywhere and around the query, operands that change from call to call, lowest and highest:
//       points per workgroup, share of the levels in LDS   2500 x 1/2    3500 x 1/2    5000 x 1/4    5000 x 1/3    5000 x 1/2    8000 x 1/2
//       float32, one stage                                 0.94 - 1.01   0.96 - 1.02   0.99 - 1.05   0.96 - 1.10   1.07 - 1.12   1.06 - 1.15
//       scores given                                       0.99 - 1.14   0.99 - 1.14   1.03 - 1.09   1.02 - 1.05   1.13 - 1.19   1.21 - 1.24
//       plain attention                                    0.97 - 1.11   0.94 - 1.08   1.03 - 1.04   1.02 - 1.03   1.05 - 1.12   1.10 - 1.17
//       bfloat16, one stage                                0.87 - 0.92   0.87 - 0.93                 0.93 - 0.97   0.99 - 1.02   0.99 - 1.07
//       scores given                                       0.90 - 1.01   0.89 - 0.99                 0.95 - 0.99   0.98 - 1.08   1.04 - 1.13
//       plain attention                                    0.87 - 1.04   0.89 - 1.02                 1.01 - 1.06   1.05 - 1.14   1.10 - 1.19
//     (12000 x 1/2: bfloat16, one stage 1.03 - 1.09; float32, scores given, below 1000 points on levels in LDS 0.84 - 1.05.)  On the same operands again
//     and again, part of which the Infinity Cache then holds: plain attention, 6 x 10000 queries on base maps, 4 points 265, 250 (the same ones 237, 241),
//     8 points 457, 438 (415, 434).  So: from 5000 points (bfloat16 in one stage 8000; float32 with scores fewer) of which 1200 (bfloat16 2400)
//     are on levels in LDS.
//     Levels that are no such pyramid (equal ones, or coarse to fine) may have none that fits; such a call takes 1 to 12 % longer than from memory.
//     Not with packed distributions, which a cross-attention layer uses: its points share a pillar's few pixels, whose rows the L1 has
//     (200 x 200 queries, base maps 412, 432; 120 x 120, 30 x 48 226, 239).
template <typename T, int VEC, int LPR> constexpr bool kLdsRowsTiling = sizeof(T) <= 4 && VEC == 4 && LPR <= 16;
struct LdsRows { int parts, rows; };
template <typename T, typename A> static LdsRows lds_rows_plan(const FwdArgs &a) {
  constexpr size_t kStatic = (kLdsRowsBlock / kWave) * sizeof(Task<A>) * kTasksPerWave + sizeof(LevelTable) + 64;
  const LdsRows none{0, 0};
  const long long room = (long long)((160 * 1024 - kStatic) / (a.C * sizeof(T))) - 1, points = (long long)a.Q * a.L * a.P;
  if (a.iters > 1 || room < 1) return none;
  const long long cus = cu_count(), pairs = (long long)a.M * a.B;
  if (room >= a.S) {
    const long long parts = cus / pairs;
    if (4 * pairs * parts < 3 * cus || points < parts * a.S) return none;      // idle CUs; too few points
    return LdsRows{(int)parts, a.S};
  }
  const long long parts = cus / a.M;
  if (parts < 1 || (8 % a.M != 0 && a.M % 8 != 0) || a.packed_dist != nullptr) return none;
  long long all = 1, some = 1;                              // pixels of the pyramid, and of its coarsest levels, in the coarsest one's
  int in_lds = 0;
  for (int l = 1; l < a.L; ++l) all = 4 * all + 1;          // (at most 16 levels)
  for (; in_lds + 1 < a.L && 1.1 * a.S * some <= (double)room * all; ++in_lds) some = 4 * some + 1;
  constexpr bool k16 = sizeof(T) == 2;
  const long long least = a.dist != nullptr ? (k16 ? 8000 : 5000) : (!k16 && a.score_in != nullptr) ? 0 : 5000;
  if (points < parts * least || points * in_lds < parts * (k16 ? 2400 : 1200) * a.L) return none;
  return LdsRows{(int)parts, (int)room};
}

// How many of a unit's points, the first ones, take their depth taps by scalar loads, where a (batch, head) has this much of values and
// distributions:
//   rows from memory                  an eighth above 3.5 MB (one point at least), three sixteenths above 6 MB
//     one distribution for all heads  an eighth above 8 MB
//     bfloat16                        three sixteenths above 5 MB
//   the coarser levels in LDS         an eighth above 5.5 MB; bfloat16, or a map that is in LDS whole (3 to 20 % slower): none
//   a packed distribution             none: with one line a point instead of four, 4 % either way
// The vector path's front end is what bounds the gathers, a scattered line in 2 to 10 clocks; the scalar path answers a load in 10 to 14,
// side by side.  But neighbouring points find each other's lines in the L1 where maps are small, and the scalar path has nothing of the
// kind: so the lines lie where points around the query stop losing.  Kernel, us, points around the query, anywhere, clustered, 6 batch
// elements, 32 channels and four levels of 8 points unless noted.
//   Rows from memory, 4000 queries, none / an eighth / three sixteenths:
//     58 x 100, 16 bins          1.4 MB   159, 228, 226   164, 231, 228   169, 231, 224
//     80 x 128, 16 bins          2.5 MB   185, 264, 268   181, 266, 262   193, 266, 258
//     46 x 80, 128 bins, 3 x 8   3.0 MB   153, 225, 231   159, 222, 222   171, 217, 216
//     100 x 170, 16 bins, 1 x 4  3.1 MB   106, 125, 121   106, 123, 116   106, 123, 116
//     58 x 100, 80 bins          3.3 MB   197, 300, 293   193, 294, 281   200, 284, 270
//     80 x 128, 64 bins, 1 x 8   3.8 MB   123, 144, 150   117, 140, 142   120, 136, 140
//     58 x 100, 112 bins, 3 x 4  4.2 MB   156, 213, 203   150, 206, 194   159, 195, 183
//     70 x 119, 112 bins         6.1 MB   240, 367, 335   226, 354, 317   232, 340, 303
//     116 x 200, 16 channels     9.4 MB   244, 375, 338   225, 358, 320   230, 344, 310
//     116 x 200, 64 bins        11.3 MB   283, 415, 376   263, 401, 360   268, 389, 354   (a quarter 292, 385, 343)
//   Units of few points, for which one or two are a larger part, none / by the rule:
//     3 points   100 x 170, 32 bins  4.2 MB   84, 90, 69   77, 82, 63         116 x 200, 64 bins  8.5 MB   87, 91, 74   87, 90, 71
//                three levels of 1 from 58 x 100, 112 bins  4.2 MB   61, 70, 47   58, 63, 44
//     4 points   80 x 128, 64 bins   3.8 MB   74, 78, 68   73, 77, 65         70 x 119, 112 bins  4.6 MB   76, 84, 69   74, 83, 65
//                116 x 200, 16 bins  4.2 MB   80, 89, 73   82, 89, 72         116 x 200, 64 bins  8.5 MB   99, 106, 86   98, 103, 82
//                two levels of 2 from 80 x 128  4.7 MB   73, 83, 71   72, 81, 68   from 116 x 200  10.6 MB   97, 104, 87   96, 102, 84
//     5 and 7    116 x 200, 64 bins  8.5 MB   116, 129, 107   113, 124, 102   and   141, 159, 134   135, 152, 126
//     6 points   three levels of 2 from 116 x 200  11.2 MB   112, 130, 116   113, 128, 112   two of 3, 40 bins  8.0 MB   116, 135, 114   117, 132, 111
//   One distribution for all heads (not packed: few points), none / an eighth:
//     65 x 116, 128 bins, 2 x 8, 2000 queries  6.0 MB   18.1, 18.2 around the query     116 x 200, 64 bins  11.3 MB   232, 357, 328   224, 347, 318
//   The coarser levels in LDS, 10000 queries, none / an eighth:
//     58 x 100, 16 bins          1.5 MB   323, 499, 517   359, 478, 483
//     80 x 128, 16 bins          2.6 MB   359, 565, 564   382, 530, 515
//     58 x 100, 64 bins          3.0 MB   367, 533, 565   384, 510, 520
//     70 x 119, 64 bins          4.2 MB   403, 610, 605   408, 577, 554
//     80 x 128, 64 bins, 3 x 8   5.2 MB   680, 1027, 965   697, 998, 925
//     116 x 200, 16 bins         5.9 MB   487, 769, 721   474, 737, 675   (three sixteenths 515, 749, 680)
//     16 channels, 64 bins       9.9 MB   488, 759, 691   454, 721, 640
//     64 bins                   11.8 MB   571, 869, 803   538, 839, 766   (three sixteenths 578, 825, 752)
//   Bfloat16, rows from memory, 4000 queries, none / three sixteenths:
//     70 x 119, 112 bins         3.1 MB   190, 299, 263   213, 282, 241   (an eighth 194, 290, 250)
//     116 x 200, 59 bins         5.6 MB   231, 355, 327   228, 335, 302
//     64 bins                    5.9 MB   250, 379, 351   229, 341, 302
//   Bfloat16, the coarser levels in LDS, 10000 queries, none / a sixteenth / an eighth:
//     64 bins   475, 795, 738   482, 760, 684   486, 738, 663     128 bins   498, 763, 697   505, 748, 676   515, 733, 665
template <typename T> static int points_by_scalar(const FwdArgs &a, const LdsRows &lds) {
  const int LP = a.L * a.P;
  if (sizeof(T) > 4 || a.dist == nullptr || a.packed_dist != nullptr || a.D < 2 || LP < 3 || (lds.parts > 0 && lds.rows == a.S)) return 0;
  const long long bytes = (long long)(a.C + a.D) * a.S * (long long)sizeof(T);
  const int eighth = LP / 8, three_sixteenths = (3 * LP + 15) / 16;
  if (sizeof(T) == 2) return lds.parts == 0 && bytes > (5LL << 20) ? three_sixteenths : 0;
  if (lds.parts > 0) return bytes > (11LL << 19) ? eighth : 0;
  if (a.dist_heads == 1) return bytes > (8LL << 20) ? eighth : 0;
  return bytes > (6LL << 20) ? three_sixteenths : bytes > (7LL << 19) ? std::max(eighth, 1) : 0;
}

template <typename T, typename A, int VEC, int LPR>
static hipError_t launch_fwd_cfg(const FwdArgs &a, hipStream_t stream) {
  // Units per wavefront: as many as its 64 lanes have points for.  A call with few units is spread over more wavefronts
  // instead, down to one unit each, while that leaves fewer than kFewWaves of them (four per CU): its time is the
  // length of one wavefront's chain of loads, which is proportional to the units.
  constexpr long long kFewWaves = 1024;
  int upw = 1;
  while (upw < kMaxUnitsPerWave && 2 * upw * a.L * a.P <= kWave) upw *= 2;
  if (upw > 1 && upw < kMaxUnitsPerWave && upw / 2 * 3 * a.L * a.P <= kWave) upw = upw / 2 * 3;    // 20 points: 60 lanes, not 40
  while (upw > 1 && (long long)a.M * a.B * ((a.Q + upw - 1) / upw) < kFewWaves) upw /= 2;
  // (the kernel counts bytes from a group's first point, and from its first output row, in 32 bits)
  while (upw > 1 && (long long)upw * a.M * std::max((long long)a.L * a.P * std::max<int>(a.loc_stride * sizeof(A), 4 * sizeof(T)), (long long)a.C * (long long)sizeof(T)) > 0x7FFFFFFFLL) upw /= 2;
  const FwdShape ws = fwd_shape(a.L, a.P, upw);
  const LdsRows lds = kLdsRowsTiling<T, VEC, LPR> ? lds_rows_plan<T, A>(a) : LdsRows{0, 0};
  const int parts = lds.parts, by_scalar = points_by_scalar<T>(a, lds);
  const int q_per_iter = (parts > 0 ? kLdsRowsBlock / kWave : kWavesPerBlock) * ws.upw, groups = (a.Q + q_per_iter - 1) / q_per_iter;
  const int iters = parts > 0 ? (groups + parts - 1) / parts : a.iters > 0 ? a.iters : 1;
  const int q_blocks = (groups + iters - 1) / iters;
  const long long blocks = (long long)a.M * a.B * q_blocks;
  if (blocks <= 0 || blocks > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
  const bool fused = a.dist != nullptr;
  // Locations and weights pass through once.  Non-temporal loads keep them out of the way of the rows and distributions, but a line that
  // workgroups on several XCDs share (neighbouring heads, where a unit's points are no whole lines) is then fetched from memory
  // by each.  6 batch elements, four levels from 80 x 128, 8 points (whole lines), non-temporal and plain, us: 610, 618; bfloat16 556, 572; plain
  // attention, maps from 116 x 185 360, 380; with 2, 3 or 4 points per level 212, 202; 211, 203; 346, 341; one level of 58 x 92, 4 points
  // 137, 112; three of 58 x 92 226, 208.  Small operands come from the caches either way (37 x 59, 20 MB, whole lines: 48, 43).
  // (Plain attention, four levels of 4 points, whose locations are whole lines and whose weights are not: both non-temporal, neither, the
  // locations alone 272, 269, 267; on the same operands again and again, which the Infinity Cache then holds in part, 230, 258, 238.)
  const bool large = (long long)a.B * a.Q * a.M * a.L * a.P * (a.loc_stride + 1) * (long long)sizeof(A) > (48LL << 20);
  const int once = !large ? 0 : (a.L * a.P * a.loc_stride * sizeof(A) % 128 == 0 ? 1 : 0) | (a.L * a.P * sizeof(A) % 128 == 0 ? 2 : 0);
  // How a unit's tasks lie in LDS where several row slots share it: in the order of its points, or a run for each slot, which takes half the
  // instructions to read.  Runs where the XCD's L2 does not hold a (batch, head)'s value rows well: half of it, 2 MB.  In turn and runs, us, 4 x 4000
  // queries, 8 points on four levels, value rows of 1 MB: 110.7, 113; plain attention 81.4, 89 and with 4 points 45.5, 49.7; 12 points, 16 channels
  // 33.7, 35.8.  3.9 MB, 3000 queries 159.5, 151; 2.3 MB, 4 points a level 116, 111; their second stage alone 133, 129.  A packed float32
  // distribution, 1 MB: 160.6, 144 (3.9 MB: 167, 155); bfloat16 141, 143.
  const int par = std::min(upw & -upw, kWave / LPR);
  const long long map_bytes = (long long)a.S * a.C * (long long)sizeof(T);                  // a (batch, head)'s value rows
  const bool in_turn = kWave / LPR > par && map_bytes <= (2LL << 20) && !(fused && a.packed_dist != nullptr && sizeof(T) == 4);
  // Early: plain attention asks for the first group's locations and weights before the level table, depth taps read the levels' sizes by
  // scalar loads instead of the table.  Float32 on maps above 1.5 MB: units of four points with rows of whole lines, and a packed distribution.
  // A wavefront of one group then waits once, not twice, but all of them gather rows the sooner together, which costs more where
  // caches serve them (a barrier in the table's place changes nothing, a table for each wavefront is slower).
  //   Plain attention, 4 x 31250 queries of 4 points, around the query and anywhere, us, table first and early:
  //     32 channels  1.1 MB 110, 110 and 106, 107    2.2 MB 136, 133 and 137, 139    8.7 MB 206, 204 and 269, 268    2 x 2 points, 2.7 MB 137, 134
  //       and 155, 156
  //     64 channels  2.1 MB 203, 196 and 189, 186    4.4 MB 238, 229 and 269, 271    16 channels  4.4 MB 143, 145 and 220, 219
  //     20 channels  5.4 MB 189, 202 and 308, 307    2 points a unit, 2.2 MB 120, 122 and 127, 130
  //     early over table first, 32 channels, four sizes of map: 8 to 64 points 1.00 - 1.12 (20 points 0.96 - 1.01), bfloat16 0.99 - 1.07 (15 and 20 points
  //     0.95 - 1.02), float64 up to 1.08
  //   Packed distribution, around the query and anywhere, us, table and own sizes, 4 levels of 8 points:
  //     4 x 9000 queries on 116 x 197, 112 bins 300, 284 and 424, 405    4 x 3906 on 100 x 170 117, 114 and 169, 162    64 channels 191, 188 and 258, 251
  //     on 70 x 119 (1.4 MB) 96, 100 and 132, 129    16 channels 80, 93 and 117, 113    3 levels of 4 points 119, 122 and 150, 145, 16 channels
  //       95, 113 and 129, 125
  //     bfloat16, 60 x 102, 3 levels of 4 points 62, 69 and 73, 74    4 levels of 8, 16 channels 80, 96 and 102, 105    116 x 197 244, 251 and 349, 351
  //   A distribution per head, 60 x 102, 111, 111 and 157, 162 (bfloat16 106, 107 and 160, 167); other shapes 0.98 - 1.06 and 0.99 - 1.02, own over table.
  const bool early = sizeof(T) == 4 && !in_turn && 2 * map_bytes > (3LL << 20) &&
                     (fused ? a.packed_dist != nullptr : a.score_in == nullptr && a.L * a.P == 4 && a.C >= 32);
  auto launch = [&](auto kernel, int threads, size_t bytes) -> hipError_t {
    if (hipError_t e = allow_lds(reinterpret_cast<const void *>(kernel), bytes)) return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(threads), bytes, stream, (const T *)a.value, (const T *)a.dist, a.shapes,
                       a.shape_stride, a.level_start, (const A *)a.loc, a.loc_stride, (const A *)a.attn,
                       fused ? nullptr : (const T *)a.score_in, (T *)a.out, fused ? (T *)a.score_out : nullptr,
                       fused ? (A *)a.weight_update : nullptr, fused ? (const T *)a.packed_dist : nullptr,
                       fused && a.dist_heads == 1 ? 1 : a.M, a.B, a.S, a.M, a.C, fused ? a.D : 0, a.L, a.Q, a.P, upw, iters, q_blocks, once, lds.rows, by_scalar);
    return hipGetLastError();
  };
  if constexpr (kLdsRowsTiling<T, VEC, LPR>) {
    if (parts > 0) {
      const size_t bytes = ((size_t)lds.rows + 1) * a.C * sizeof(T);
      if constexpr (sizeof(T) == 4) {
        if (by_scalar > 0) return launch(fwd_attention_kernel<T, A, VEC, LPR, true, true, false, false, true>, kLdsRowsBlock, bytes);
      }
      return fused ? launch(fwd_attention_kernel<T, A, VEC, LPR, true, true, false, false>, kLdsRowsBlock, bytes)
                   : launch(fwd_attention_kernel<T, A, VEC, LPR, false, true, false, false>, kLdsRowsBlock, bytes);
    }
  }
  if constexpr (std::is_same<T, float>::value) {
    if (early)
      return fused ? launch(fwd_attention_kernel<T, A, VEC, LPR, true, false, false, true>, kBlock, 0)
                   : launch(fwd_attention_kernel<T, A, VEC, LPR, false, false, false, true>, kBlock, 0);
  }
  if constexpr (sizeof(T) <= 4) {
    if (by_scalar > 0)
      return in_turn ? launch(fwd_attention_kernel<T, A, VEC, LPR, true, false, true, false, true>, kBlock, 0)
                     : launch(fwd_attention_kernel<T, A, VEC, LPR, true, false, false, false, true>, kBlock, 0);
  }
  if (in_turn)
    return fused ? launch(fwd_attention_kernel<T, A, VEC, LPR, true, false, true, false>, kBlock, 0)
                 : launch(fwd_attention_kernel<T, A, VEC, LPR, false, false, true, false>, kBlock, 0);
  return fused ? launch(fwd_attention_kernel<T, A, VEC, LPR, true, false, false, false>, kBlock, 0)
               : launch(fwd_attention_kernel<T, A, VEC, LPR, false, false, false, false>, kBlock, 0);
}

template <typename T, typename A>
static hipError_t launch_fwd_typed(const FwdArgs &a, hipStream_t stream) {
  const RowTiling rt = pick_gather_tiling(a.C, (int)sizeof(T), a.vec_hint);
#define DFA3D_CASE(V, R) \
  if (rt.vec == V && rt.lpr == R) return launch_fwd_cfg<T, A, V, R>(a, stream);
  DFA3D_GATHER_TILINGS(DFA3D_CASE)
#undef DFA3D_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_forward(const FwdArgs &a, int dtype, hipStream_t stream) {
  switch (dtype) {
    case DFA3D_F32: return launch_fwd_typed<float, float>(a, stream);
    case DFA3D_F64: return launch_fwd_typed<double, double>(a, stream);
    case DFA3D_BF16: return launch_fwd_typed<__hip_bfloat16, float>(a, stream);
  }
  return hipErrorInvalidValue;
}

template <typename T, typename A>
static hipError_t launch_ds_typed(const DepthScoreArgs &a, hipStream_t stream) {
  const DepthScoreShape shape = depth_score_shape(a.B, a.M, a.L, a.Q, a.P);
  const int queries = depth_score_queries(shape, a.P);
  const long long blocks = (long long)a.M * a.B * (a.L / shape.levels) * ((a.Q + queries - 1) / queries);
  if (blocks <= 0 || blocks > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((depth_score_kernel<T, A>), dim3((unsigned)blocks), dim3(kBlock), 0, stream, (const T *)a.dist,
                     a.shapes3, a.level_start, (const A *)a.loc3, (T *)a.score, a.B, a.S, a.M, a.D, a.L, a.Q, a.P);
  return hipGetLastError();
}

hipError_t launch_depth_score(const DepthScoreArgs &a, int dtype, hipStream_t stream) {
  switch (dtype) {
    case DFA3D_F32: return launch_ds_typed<float, float>(a, stream);
    case DFA3D_F64: return launch_ds_typed<double, double>(a, stream);
    case DFA3D_BF16: return launch_ds_typed<__hip_bfloat16, float>(a, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace dfa3d
