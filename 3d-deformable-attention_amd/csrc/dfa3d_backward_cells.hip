// Tile kernel of the binned backward for rows of up to 64 channels: cell-owned lane groups and two kinds of wavefronts.
//
// The bins, work items and queues are those of dfa3d_backward_binned.hip; only the work inside a tile differs.
// A tile of TY x 8 pixels is seen as its "cells": the points whose base pixel (upper left of the four pixels around
// the location) is that pixel.  All points of a cell touch the same four value rows, so
//   * a group of LPR lanes (VEC channels each) owns a cell for the whole work item: the four value rows and the four
//     accumulators of weight * grad_out live in its registers, every point's grad_out row is read from LDS once, the
//     four dot products and the four weighted sums are formed from it, and nothing is added to an LDS tile during the
//     passes.  The weighted sums are outer products (4 corners x channels, one point deep) of 4-lane blocks: one
//     v_mfma_f32_4x4x1 per channel of a lane does what four FMAs per lane would, on the matrix pipe; with 2-byte
//     elements, unless points are sparse, the dot products are matrix instructions too, four points at a time (walk_fours);
//   * a pass sorts its points (256, or 128 with long rows) by cell: one integer LDS atomic per point.
// (Base pixels run from -1, for a location within half a pixel of the map's upper or left edge, to H - 1 / W - 1;
// the tiles are laid over that range, so a cell's upper or left pixels may lie outside the map like its lower or
// right ones: such corners carry weight zero, their value rows read as zero and their sums are never written.)
//
// The 8 wavefronts of a workgroup have two roles.  "Walkers" (wavefronts 0-3, one or two tile rows of 8 cells each)
// walk the cells' lists; "pointers" (wavefronts 4-7, one point of the pass per thread) do everything that is per point:
// geometry, depth taps, corner weights, the sort, and afterwards the point's gradients and its grad_dist taps into the
// LDS depth tile.  The roles meet at two barriers per turn and otherwise overlap.  Turns follow one another without a gap, whatever item their
// passes belong to (pass t: one of the item's passes), so that an item of a single pass costs a single turn:
//   phase X(t):  walkers: walk(t-1)        pointers: scores and corner weights of t, prepare(t+1)
//   phase Y(t):  walkers: stage(t)         pointers: place(t) (scan + sorted slots), finish(t-1)
// and where pass t-1 was its item's last:
//   Y(t):    walkers put the old item's corner sums together in registers (neighbouring cells are neighbouring lane groups;
//            sums that cross into the next wavefront's rows, and the rim's, go through a few rows of LDS) and ask for the
//            value rows of the item of pass t
//   X(t+1):  walkers send the old item's last rows and its rim before they walk; pointers write the depth tile out and leave
//            it zeroed, before the first finish of the next item in Y(t+1)
// grad_dist taps go to the LDS tile by compare-and-swap on the word's bits: the LDS float atomic retires 0.33 lanes per
// clock and CU, read + compare-and-swap 2.9 (and a tap is complete when its phase ends, which the flush relies on).
//
// Semantics are those of bwd_attention_kernel (dfa3d_backward.hip holds the formulas and the reference lines).
#include <type_traits>

#include "dfa3d_binned.h"

namespace dfa3d {

constexpr int kWalkers = 256;         // threads of the walker wavefronts 0-3; the wavefronts after them own the points

#ifdef DFA3D_TILE_TIMING
// wavefront 0 (walkers) clocks slots 0-7, wavefront 4 (pointers) slots 8-15
#define CT_DECL TICKS_DECL(16)
#define CT_MARK(i) TICKS_MARK((wave & 3) == 0, (i) + 2 * wave)
#define CT_FLUSH() TICKS_FLUSH((wave & 3) == 0, 2 * wave, 8)
constexpr size_t kTicksLds = 16 * sizeof(unsigned long long);
#else
#define CT_DECL
#define CT_MARK(i) do { } while (0)
#define CT_FLUSH() do { } while (0)
constexpr size_t kTicksLds = 0;
#endif

// Lane groups by row length: LPR lanes of VEC channels per row, 64 / LPR cells per wavefront; points per pass, one per
// pointer thread (256 staged rows of 64 channels would leave room for one workgroup per CU only).
struct CellShape { int vec, lpr, pass; };
__host__ __device__ constexpr int cell_pass(int lpr) { return lpr == 4 ? 256 : 128; }
__host__ __device__ inline CellShape cell_shape(int C) {
  return C <= 16 ? CellShape{4, 4, cell_pass(4)} : C <= 32 ? CellShape{8, 4, cell_pass(4)} : CellShape{8, 8, cell_pass(8)};
}
// the most tile rows of 8 cells that four walker wavefronts own
int cell_max_ty(int C) { return 4 * (kWave / cell_shape(C).lpr) / kCellTX; }

struct CellLds {      // offsets (in 4-byte words) into the dynamic LDS block
  int gd, gstage, dots, sslot, cnt, offs, goff, cross, rim, total;
};
__host__ __device__ inline CellLds cell_lds_layout(int ty, int row, int cells, int pass, int D, int elem) {
  CellLds o;
  const int R = (ty + 1) * (kCellTX + 1);
  o.gd = 0;
  o.gstage = (o.gd + R * D + 3) & ~3;                        // 16-byte aligned rows
  o.dots = o.gstage + (pass + 1) * row * elem / 4;           // the staged rows, as they lie in memory, and a row of zeros
  o.sslot = o.dots + (pass + 1) * 4;                    // corner weights, then dot products; four zeros at the end
  o.cnt = o.sslot + (pass + 2) / 2;                     // 16-bit point slots; the one at the end names the row of zeros
  o.offs = o.cnt + 3 * cells;
  o.goff = o.offs + cells + 1;
  o.cross = (o.goff + 2 * pass + 3) & ~3;                   // sums that cross into the next wavefront's tile rows
  o.rim = o.cross + 3 * (kCellTX + 1) * row;                 // sums of the tile's rim pixels, on their way out
  o.total = o.rim + rim_pixels(ty, kCellTX) * row;
  return o;
}

int cell_kernel_pass(int C) { return cell_shape(C).pass; }
int cell_kernel_block(int C) { return kWalkers + cell_shape(C).pass; }
size_t cell_kernel_lds_bytes(int ty, int C, int D, int elem) {
  const CellShape s = cell_shape(C);
  return (size_t)cell_lds_layout(ty, s.vec * s.lpr, 4 * kWave / s.lpr, s.pass, D, elem).total * 4;
}

// what a pointer thread keeps of its point between the phases
struct PointState {
  uint32_t gp;                // index of the point
  float a, sc[4], hl[4];      // attention weight; corner scores; upper minus lower depth tap per corner
  float lh, lw, ld;           // fractional parts along h, w, depth
  unsigned bits;              // bit k: corner k inside the map; 4: depth inside; 5, 6: lower, upper tap exists; 7: live;
                              // 8-13: the point's cell; 16-31: lower depth bin + 1
};
// Queue state of the thread that fetches the work items: the item taken now was popped two items ago and its two
// records asked for one item ago, so neither the queue atomic nor the loads are waited for.  A workgroup's first
// kDealt items are dealt, not popped (its number among the workgroups of its class says which), so that a workgroup
// starts after one round trip to memory instead of one for each item it looks ahead.
constexpr int kDealt = 4;
struct CellFetch {
  int classes_done, w_next;
  int4 rec, geo;
  __device__ __forceinline__ void load(const BinWorkspace &ws, int w) {
    rec = w >= 0 ? ws.items[w] : make_int4(-1, 0, 0, 0);
    geo = w >= 0 ? ws.geom[w] : make_int4(0, 0, 0, 0);
  }
  __device__ __forceinline__ int pop(const BinWorkspace &ws, const BinPlan &p) {
    return pop_item(ws, p, blockIdx.x % kClasses, classes_done, kDealt);
  }
  __device__ __forceinline__ void start(const BinWorkspace &ws, const BinPlan &p, int4 (&r)[kDealt - 1], int4 (&g)[kDealt - 1]) {
    const int c = blockIdx.x % kClasses, lo = p.class_start[c], hi = p.class_start[c + 1], n_wg = workgroups_of_class(c);
    int w[kDealt];
    classes_done = 0;
    for (int k = 0; k < kDealt; ++k) w[k] = hi - 1 - ((int)blockIdx.x / kClasses + k * n_wg);
    for (int k = 0; k < kDealt; ++k)
      if (w[k] < lo) w[k] = pop(ws, p);                     // the class has no more: another one's
    for (int k = 0; k < kDealt - 1; ++k) {
      load(ws, w[k]);
      r[k] = rec; g[k] = geo;
    }
    load(ws, w[kDealt - 1]);
    w_next = w[kDealt - 1] >= 0 ? pop(ws, p) : -1;
  }
  __device__ __forceinline__ void advance(const BinWorkspace &ws, const BinPlan &p, int4 *r, int4 *g) {
    *r = rec; *g = geo;
    load(ws, w_next);
    w_next = w_next >= 0 ? pop(ws, p) : -1;
  }
};
// a work item, decoded
struct ItemGeom { int bin, seg, n_item, sole, b, m, H, W, Dd, start, y0, x0; };      // sole: see bin_scan_kernel
constexpr int kItemSlots = 8;      // a power of two; in use: the item before (finish, flush), this one and the next three
__device__ __forceinline__ int slot_of_item(int it) { return it & (kItemSlots - 1); }
// what the kernel declares as static LDS (level tables, the fetching thread's state, item records): the dynamic
// block of each of two workgroups on a CU may be half of the CU's 160 KB less this
constexpr size_t kCellStaticLds = 4 * DFA3D_MAX_LEVELS * sizeof(int) + sizeof(CellFetch) + kItemSlots * sizeof(ItemGeom) + kTicksLds;
size_t cell_kernel_half_cu_lds() { return 80 * 1024 - kCellStaticLds; }
// an item record read from LDS is the same in every lane: keep it in scalar registers
__device__ __forceinline__ ItemGeom uniform(const ItemGeom &g) {
  ItemGeom u;
  u.bin = __builtin_amdgcn_readfirstlane(g.bin); u.seg = __builtin_amdgcn_readfirstlane(g.seg);
  u.n_item = __builtin_amdgcn_readfirstlane(g.n_item); u.sole = __builtin_amdgcn_readfirstlane(g.sole);
  u.b = __builtin_amdgcn_readfirstlane(g.b); u.m = __builtin_amdgcn_readfirstlane(g.m);
  u.H = __builtin_amdgcn_readfirstlane(g.H); u.W = __builtin_amdgcn_readfirstlane(g.W);
  u.Dd = __builtin_amdgcn_readfirstlane(g.Dd); u.start = __builtin_amdgcn_readfirstlane(g.start);
  u.y0 = __builtin_amdgcn_readfirstlane(g.y0); u.x0 = __builtin_amdgcn_readfirstlane(g.x0);
  return u;
}

// Four partial sums per lane (one per corner) over the four lanes of a quad: lane c gets the whole sum of corner c.
// Two exchange steps in which every lane passes on the two (then one) partial sums its partner collects.
__device__ __forceinline__ float quad_corner_sum(float d0, float d1, float d2, float d3, bool odd, bool upper) {
  const float keep_a = odd ? d1 : d0, send_a = odd ? d0 : d1, keep_b = odd ? d3 : d2, send_b = odd ? d2 : d3;
  const float a = keep_a + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(send_a), 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
  const float b = keep_b + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(send_b), 0xB1, 0xF, 0xF, true));
  const float keep = upper ? b : a, send = upper ? a : b;
  return keep + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(send), 0x4E, 0xF, 0xF, true));               // quad_perm [2,3,0,1]
}

// Where the 16-byte piece `piece` of staged row `row` lies, in bytes.  Of 2-byte elements the pieces of a row lie in an order that
// depends on the row, so that the same piece of eight neighbouring rows falls on different banks: a lane that takes a whole row
// (WholeRow) reads them one after the other, as its neighbours do with theirs.
template <typename T, int ROWB> __device__ __forceinline__ constexpr int piece_at(int row, int piece) {
  if constexpr (sizeof(T) == 2) {
    constexpr int N = ROWB / 16, SH = ROWB >= 128 ? 0 : ROWB == 64 ? 1 : 2;
    piece ^= (row >> SH) & (N - 1);
  }
  return row * ROWB + 16 * piece;
}

// The channels of one lane of a row of C elements, in NG groups of four.  Rows of 4-byte elements: group g covers
// channels 4 (LPR g + cl) .. + 3, so that the lanes of a row read whole 64-byte pieces together; 2-byte elements: VEC
// consecutive channels.  A group beyond C reads as zero and is never written.
template <typename T, int VEC, int LPR> struct LaneChannels {
  static constexpr int NG = VEC / 4;
  int first[NG];            // first channel of each group
  uint32_t off[NG];         // its byte offset inside a row, kNoChan beyond the last channel
  bool c8;
  __device__ __forceinline__ LaneChannels(int cl, int C) : c8((C & 7) == 0) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      first[g] = sizeof(T) == 4 ? 4 * (LPR * g + cl) : VEC * cl + 4 * g;
      off[g] = first[g] < C ? (uint32_t)(first[g] * (int)sizeof(T)) : kNoChan;
    }
  }
  // the lane's elements as they lie in memory
  struct Raw { uint32_t w[VEC * (int)sizeof(T) / 4]; };
  __device__ __forceinline__ void load(rsrc_t r, uint32_t row, Raw &o) const {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, row + off[g], 0, 0);
        o.w[4 * g] = t.x; o.w[4 * g + 1] = t.y; o.w[4 * g + 2] = t.z; o.w[4 * g + 3] = t.w;
      }
    } else {
      if (VEC == 8 && c8) {                                  // uniform
        const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, row + off[0], 0, 0);
        o.w[0] = t.x; o.w[1] = t.y;
        if constexpr (VEC == 8) { o.w[2] = t.z; o.w[3] = t.w; }
      } else {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          const u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(r, row + off[g], 0, 0);
          o.w[2 * g] = t.x; o.w[2 * g + 1] = t.y;
        }
      }
    }
  }
  static __device__ __forceinline__ void to_float(const Raw &r, float (&v)[VEC]) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      if constexpr (sizeof(T) == 4) v[i] = __uint_as_float(r.w[i]);
      else v[i] = __uint_as_float((i & 1) ? r.w[i / 2] & 0xFFFF0000u : r.w[i / 2] << 16);
    }
  }
  // the same lane's place in a row staged in LDS
  static constexpr int ROWB = VEC * LPR * (int)sizeof(T);
  __device__ __forceinline__ void put(unsigned char *rows, int row, int cl, const Raw &r) const {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int g = 0; g < NG; ++g)
        *reinterpret_cast<uint4 *>(rows + piece_at<T, ROWB>(row, LPR * g + cl)) = make_uint4(r.w[4 * g], r.w[4 * g + 1], r.w[4 * g + 2], r.w[4 * g + 3]);
    } else if constexpr (VEC == 8) {
      *reinterpret_cast<uint4 *>(rows + piece_at<T, ROWB>(row, cl)) = make_uint4(r.w[0], r.w[1], r.w[2], r.w[3]);
    } else {
      *reinterpret_cast<uint2 *>(rows + piece_at<T, ROWB>(row, cl >> 1) + 8 * (cl & 1)) = make_uint2(r.w[0], r.w[1]);
    }
  }
  __device__ __forceinline__ void get(const unsigned char *rows, int row, int cl, Raw &r) const {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const uint4 t = *reinterpret_cast<const uint4 *>(rows + piece_at<T, ROWB>(row, LPR * g + cl));
        r.w[4 * g] = t.x; r.w[4 * g + 1] = t.y; r.w[4 * g + 2] = t.z; r.w[4 * g + 3] = t.w;
      }
    } else if constexpr (VEC == 8) {
      const uint4 t = *reinterpret_cast<const uint4 *>(rows + piece_at<T, ROWB>(row, cl));
      r.w[0] = t.x; r.w[1] = t.y; r.w[2] = t.z; r.w[3] = t.w;
    } else {
      const uint2 t = *reinterpret_cast<const uint2 *>(rows + piece_at<T, ROWB>(row, cl >> 1) + 8 * (cl & 1));
      r.w[0] = t.x; r.w[1] = t.y;
    }
  }
};

// The other way to hold rows, of 2-byte elements: each lane of four takes all that the four hold of one row (with eight lanes to
// a row: of their half of it), in the order of the four lanes' Raw words.
template <typename T, int VEC, int LPR> struct WholeRow {
  static constexpr int W = VEC * 2, ROWB = VEC * LPR * 2;      // words; bytes of a row
  uint32_t w[W];
  __device__ __forceinline__ void get(const unsigned char *rows, int row, int half) {
#pragma unroll
    for (int i = 0; i < W / 4; ++i) {
      const uint4 t = *reinterpret_cast<const uint4 *>(rows + piece_at<T, ROWB>(row, 4 * half + i));
      w[4 * i] = t.x; w[4 * i + 1] = t.y; w[4 * i + 2] = t.z; w[4 * i + 3] = t.w;
    }
  }
};
// x[k] of lane b of four becomes x[b] of lane k
__device__ __forceinline__ void quad_transpose(uint32_t (&x)[4], bool odd, bool upper) {
#pragma unroll
  for (int k = 0; k < 4; k += 2) {
    const uint32_t got = __builtin_amdgcn_mov_dpp(odd ? x[k] : x[k + 1], 0xB1, 0xF, 0xF, true);      // quad_perm [1,0,3,2]
    x[k] = odd ? got : x[k];
    x[k + 1] = odd ? x[k + 1] : got;
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t got = __builtin_amdgcn_mov_dpp(upper ? x[k] : x[k + 2], 0x4E, 0xF, 0xF, true);    // quad_perm [2,3,0,1]
    x[k] = upper ? got : x[k];
    x[k + 2] = upper ? x[k + 2] : got;
  }
}
// the four corners' rows, as the lanes of a group hold them, to one corner's row per lane
template <typename T, int VEC, int LPR>
__device__ __forceinline__ void whole_rows(const typename LaneChannels<T, VEC, LPR>::Raw (&r)[4], int cl, WholeRow<T, VEC, LPR> &o) {
#pragma unroll
  for (int e = 0; e < VEC / 2; ++e) {
    uint32_t x[4] = {r[0].w[e], r[1].w[e], r[2].w[e], r[3].w[e]};
    quad_transpose(x, (cl & 1) != 0, (cl & 2) != 0);
#pragma unroll
    for (int b = 0; b < 4; ++b) o.w[VEC / 2 * b + e] = x[b];
  }
}
typedef float f4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
// Dot products of the four corners' rows (a corner per lane of four) with four points' rows (a point per lane): lane j gets those
// of point j.  Products of bfloat16 numbers are exact in float; up to four chains of sums, added in pairs.
template <typename T, int VEC, int LPR>
__device__ __forceinline__ f4 corner_dots(const WholeRow<T, VEC, LPR> &v, const WholeRow<T, VEC, LPR> &g) {
  constexpr int W = WholeRow<T, VEC, LPR>::W;
  f4 half[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    f4 d[2] = {(f4){0, 0, 0, 0}, (f4){0, 0, 0, 0}};
#pragma unroll
    for (int i = 0; i < W / 4; ++i) {
      const int k = h * (W / 2) + 2 * i;
      const u32x2 a = {v.w[k], v.w[k + 1]}, b = {g.w[k], g.w[k + 1]};
      d[i & 1] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), d[i & 1], 0, 0, 0);
    }
    half[h] = d[0] + d[1];
  }
  return half[0] + half[1];
}

// The two taps (bins db, db + 1) of each of a point's four corners, asked for one phase before they are looked at.
// The choice between the two ways of 2-byte elements is made once for all four corners: made per corner, each load was followed
// by a wait for the one before, because the two ways' registers meet after it (six cameras, 30825 rows, 8 x 32 channels, bf16: 990 us for the
// kernel, now 951).
template <typename T> struct TapsInFlight {
  u32x2 t[4];
  // off: byte offset of bin db of each corner's distribution, kNoRow where there is nothing to fetch
  __device__ __forceinline__ void ask(rsrc_t r, const uint32_t (&off)[4], int D) {
    if (sizeof(T) == 4 || (D & 1) == 0) {                    // uniform; 2-byte elements: BufPair<__hip_bfloat16>::ld_word_aligned
#pragma unroll
      for (int k = 0; k < 4; ++k)
        t[k] = __builtin_amdgcn_raw_buffer_load_b64(r, sizeof(T) == 4 || off[k] == kNoRow ? off[k] : (off[k] & ~3u), 0, 0);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        t[k].x = __builtin_amdgcn_raw_buffer_load_b16(r, off[k], 0, 0);
        t[k].y = __builtin_amdgcn_raw_buffer_load_b16(r, off[k] == kNoRow ? kNoRow : off[k] + 2, 0, 0);
      }
    }
  }
  __device__ __forceinline__ void get(int k, int db, int D, float &x, float &y) const {
    if constexpr (sizeof(T) == 4) {
      x = __uint_as_float(t[k].x); y = __uint_as_float(t[k].y);
    } else if ((D & 1) == 0) {                               // rows start on words: the pair's place depends on the bin alone
      const uint32_t lo = t[k].x, hi = t[k].y;
      x = (db & 1) ? __uint_as_float(lo & 0xFFFF0000u) : __uint_as_float(lo << 16);
      y = (db & 1) ? __uint_as_float(hi << 16) : __uint_as_float(lo & 0xFFFF0000u);
    } else {
      x = bf16_bits_to_float(t[k].x); y = bf16_bits_to_float(t[k].y);
    }
  }
};

__device__ __forceinline__ void wait_for_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }           // vmcnt(0)

// The kernel's arguments.  There are more of them, and of the numbers that follow from them, than scalar registers.
template <typename T> struct CellArgs {
  BinWorkspace ws;
  const T *value, *dist, *score_in, *grad_out, *grad_score_in;
  void *grad_value, *grad_dist;
  float *grad_loc, *grad_attn, *grad_score_out;
  const float *grad_wu;
  int gl_stride;
  int Md, Mg;                 // heads stored in dist (M, or 1 = shared by all heads); heads of the grad_dist buffer written here
  int B, S, M, C, D, L, Q, P;
  FastDiv div_lp;
  int grad16;                 // bit 0 = grad_value is bfloat16, bit 1 = grad_dist is bfloat16 (else float)
};
// Where a kernel has them from:
//   anew     read from the constant segment in every phase; what a lane owns is worked out anew as well (Owner)
//   pointer  read there where the compiler wants to
//   value    kept from the start, as parameters
// What is kept and does not fit goes to lanes of vector registers and comes back one instruction each (both stages, float: 80 to 100 by
// value, 40 to 66 by pointer, none anew); what is read is waited for, which counts where phases are short because points are sparse.  Tile
// kernel, us, anew against what is taken: both stages, float, 32 channels, base shape 1133 -> 1113 (by value 1127), the same maps with
// 6 x 300 queries 429 -> 417, 400 x 400 at 0.1 points a pixel 254 -> 252; 16 channels 1013 -> 1007, 423 -> 408, 232 -> 222.  Stage 2 alone, 400 x 400
// at 0.1 and 200 x 200 at 4 (coherent): 32 channels 239 -> 227, 213 -> 209, bfloat16 231 -> 219, 198 -> 189; 16 channels 181 -> 167, 160 -> 153; 64
// channels 436 -> 419, 381 -> 371.  Both stages in bfloat16 lose with either (base shape 1104 -> 1138, 1124); float rows of over 32 channels
// gain on the base maps what they lose on others (982 -> 965, 400 x 400 446 -> 453).
enum class ArgsFrom { anew, pointer, value };
template <typename T, int LPR, bool FUSED> constexpr ArgsFrom args_from() {
  return !FUSED ? ArgsFrom::value : sizeof(T) == 4 && LPR == 4 ? ArgsFrom::pointer : ArgsFrom::anew;
}
#ifdef __HIP_DEVICE_COMPILE__
template <typename T, ArgsFrom FROM> __device__ __forceinline__ auto args(const CellArgs<T> &param) {
  if constexpr (FROM == ArgsFrom::value) {
    return &param;
  } else {
    auto a = (const __attribute__((address_space(4))) CellArgs<T> *)__builtin_amdgcn_kernarg_segment_ptr();
    if (FROM == ArgsFrom::anew) asm volatile("" : "+s"(a));
    return a;
  }
}
#else
template <typename T, ArgsFrom FROM> __device__ const CellArgs<T> *args(const CellArgs<T> &);
#endif

// FUSED: both stages (depth scores recomputed from dist, grad_dist and the z gradient produced).
// !FUSED: stage 2 alone: scores read from score_in, their gradient written to grad_score_out, no depth tile
// (the launcher passes D = 0), grad_loc has gl_stride components of which x, y are written.
// FOURS: the walkers take the points of a cell four at a time (see walks_fours() below).  Both walks in one kernel, chosen pass by
// pass, do not fit its registers: base shape, bfloat16, 32 channels 580 -> 742 us for half of its cameras, 64 channels 830 -> 1706.
template <typename T, int VEC, int LPR, bool FUSED, bool FOURS>
__global__ __launch_bounds__(kWalkers + cell_pass(LPR), 4) void cell_backward_kernel(const CellArgs<T> param) {
  constexpr int PP = cell_pass(LPR), BLOCK = kWalkers + PP, TX = kCellTX, TW = TX + 1, ROW = VEC * LPR;
  constexpr int GPW = kWave / LPR, CELLS = 4 * GPW, ROWS = GPW / TX;      // cells and tile rows per walker wavefront
  extern __shared__ __align__(16) float smem[];
  __shared__ int s_lv[4][DFA3D_MAX_LEVELS];              // the plan's level tables: H, W, Dd, first key
  __shared__ CellFetch s_fetch;                           // the fetching thread's queue state, between its turns
  __shared__ ItemGeom s_geom[kItemSlots];                // items, decoded by the thread that fetches them

  constexpr ArgsFrom ARGS = args_from<T, LPR, FUSED>();
  const auto arg = [&]() { return args<T, ARGS>(param); };
  const auto a0 = arg();
  const BinWorkspace ws = a0->ws;
  const BinPlan &p = *ws.plan;
  if (__builtin_expect(p.bins_per_bm == 0, 0)) {
    const auto a1 = args<T, ArgsFrom::anew>(param);
    backward_without_bins<T, FUSED>(a1->ws, a1->value, a1->dist, a1->score_in, a1->grad_out, a1->grad_score_in, a1->grad_value, a1->grad_dist,
                                    a1->grad_loc, a1->gl_stride, a1->grad_attn, a1->grad_score_out, a1->grad_wu, a1->Md, a1->Mg,
                                    a1->B, a1->S, a1->M, a1->C, a1->D, a1->L, a1->Q, a1->P, a1->grad16);
    return;
  }
  const int TY = p.ty, R = (TY + 1) * TW;
  const CellLds lay = cell_lds_layout(TY, ROW, CELLS, PP, a0->D, (int)sizeof(T));
  const int tid = threadIdx.x, lane = tid % kWave;
  // The role is decided by a scalar, so that the compiler branches on it uniformly: a wavefront must never run
  // through the other role's code with all lanes switched off, because barriers count wavefronts, not lanes.
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const bool walker = wave < 4;
  unsigned char *gstage = reinterpret_cast<unsigned char *>(smem + lay.gstage);
  float *gd = smem + lay.gd, *dots = smem + lay.dots, *cross = smem + lay.cross, *rim = smem + lay.rim;
  uint16_t *s_slot = reinterpret_cast<uint16_t *>(smem + lay.sslot);
  int *cnt = reinterpret_cast<int *>(smem + lay.cnt), *offs = reinterpret_cast<int *>(smem + lay.offs);
  uint32_t *goff = reinterpret_cast<uint32_t *>(smem + lay.goff);

  for (int i = tid; i < lay.gstage; i += BLOCK) smem[i] = 0;                   // depth tile
  for (int i = tid; i < 3 * CELLS; i += BLOCK) cnt[i] = 0;
  // What a group without a point reads; and rows shorter than their lane group once whole, as nothing need be written beyond their
  // channels.
  for (int i = tid + (a0->C == ROW ? PP * ROW * (int)sizeof(T) / 4 : 0); i < (PP + 1) * ROW * (int)sizeof(T) / 4; i += BLOCK) smem[lay.gstage + i] = 0;
  if (tid < 4) dots[PP * 4 + tid] = 0;
  if (tid == 0) s_slot[PP] = (uint16_t)PP;
  if (tid < DFA3D_MAX_LEVELS) {      // decoding an item then costs no dependent loads from device memory
    s_lv[0][tid] = p.H[tid]; s_lv[1][tid] = p.W[tid]; s_lv[2][tid] = p.Dd[tid]; s_lv[3][tid] = p.start[tid];
  }
  __syncthreads();
  CT_DECL

  // Gradient rows leave in two ways: stored, or added atomically.  The L2 executes about 20 G (instruction, 64-byte piece)
  // pairs of float atomics per second on the whole part, whatever the number of floats in a pair: added rows go out
  // one float (bfloat16: one pair) per lane on consecutive addresses, 16 to a pair (four floats per lane took four times
  // the pairs: this kernel's flushes alone were worth 1 ms at the BEVFormer-base shape).

  // The depth tile of the item in slot `which` goes out and is left zeroed, by `threads` threads of which this one is
  // number `first`, in the phase in which nobody adds to the tile.  A tile row (one pixel) takes 2^sh threads.  Pixels
  // 1..TY-1 x 1..7 belong to no neighbour's halo: when the item writes its tile alone they are stored, the others are added.
  // What bounds it are the vector instructions that find a pixel's place, so what is the same for a wavefront stays in scalars: the tile row
  // that it takes of the inner pixels, the pixel that it takes of the rim where that is all its lanes have room for.  (With a pixel's number
  // divided into row and column by every lane, tile kernel, one card: base shape 1210 us for 1110, bfloat16 1090 for 1025, dense 4349 for 4100, 59
  // bins and 20 channels 124.7 for 117.5, one level of 23 x 40 113.6 for 107.  Several pixels of a lane read at once instead: registers spill, + 9 %.)
  auto flush_gd = [&](int which, int first, int threads) {
    const auto a = arg();
    const int D = a->D, S = a->S, M = a->M, Mg = a->Mg;
    void *grad_dist = a->grad_dist;
    const bool gd16 = (a->grad16 & 2) != 0;                // uniform
    const ItemGeom q = uniform(s_geom[which]);
    const int mg = Mg == 1 ? 0 : q.m;
    char *gdist_b = static_cast<char *>(grad_dist) + (size_t)q.b * S * Mg * D * (gd16 ? 2 : 4);
    float *gdist_f = reinterpret_cast<float *>(gdist_b);
    const rsrc_t gdist_r = make_rsrc(gdist_b, (size_t)S * Mg * D * sizeof(float));
    const bool sole_d = q.sole != 0 && Mg == M;       // a gradient shared by the heads collects from all of them
    const bool d4 = (D & 3) == 0;
    auto lanes_log2 = [](int n) { return n > 32 ? 6 : n > 16 ? 5 : n > 8 ? 4 : n > 4 ? 3 : 2; };
    const uint32_t col_step = (uint32_t)(Mg * D), row_step = (uint32_t)q.W * col_step;
    const uint32_t e_tile = (uint32_t)(q.start + q.y0 * q.W + q.x0) * col_step + (uint32_t)(mg * D);      // of the tile's pixel (0, 0), where that exists
    if (sole_d) {
      // a wavefront takes as many pixels of a tile row as it has lanes for; the row is a scalar
      const int n = d4 ? D >> 2 : D, sh = lanes_log2(n), at_once = 6 - sh, parts = sh >= 3 ? sh - 3 : 0;   // pixels at once, parts of a row (log2)
      const int lane_px = (first & (kWave - 1)) >> sh, c0 = first & ((1 << sh) - 1);
      const int waves = threads / kWave, wave0 = __builtin_amdgcn_readfirstlane(first / kWave);
      for (int k = wave0; k < (TY - 1) << parts; k += waves) {                // uniform
        const int ry = 1 + (k >> parts), rx = 1 + ((k & ((1 << parts) - 1)) << at_once) + lane_px;
        const bool in_row = rx < TX, out = q.y0 + ry < q.H && q.x0 + rx < q.W;
        float *row = gd + (ry * TW + rx) * D;
        const uint32_t e0 = e_tile + (uint32_t)ry * row_step + (uint32_t)rx * col_step;
        if (in_row) {
          for (int c = c0; c < n; c += 1 << sh) {
            if (d4) {
              float4 *at = reinterpret_cast<float4 *>(row) + c;
              const float4 val = *at;
              *at = make_float4(0, 0, 0, 0);
              if (out) {
                if (gd16) *reinterpret_cast<uint2 *>(gdist_b + (size_t)(e0 + 4 * c) * 2) = make_uint2(pack_bf16x2(val.x, val.y), pack_bf16x2(val.z, val.w));
                else *reinterpret_cast<float4 *>(gdist_f + e0 + 4 * c) = val;
              }
            } else {                                        // float gradients only (the launcher sees to it)
              const float val = row[c];
              row[c] = 0;
              if (out) gdist_f[e0 + c] = val;
            }
          }
        }
      }
    }
    const int n = gd16 ? D >> 1 : D, sh = lanes_log2(n);
    const int rows = sole_d ? rim_pixels(TY, TX) : R;
    auto add_pixel = [&](int i) {
      int ry, rx;
      if (sole_d) {
        rim_decode(i, TY, TX, ry, rx);
      } else {
        ry = i / TW; rx = i % TW;
      }
      float *row = gd + (ry * TW + rx) * D;
      const bool out = in_map(q.y0 + ry, q.x0 + rx, q.H, q.W);
      const uint32_t e0 = e_tile + (uint32_t)ry * row_step + (uint32_t)rx * col_step;
      for (int c = first & ((1 << sh) - 1); c < n; c += 1 << sh) {
        if (gd16) {
          float2 *at = reinterpret_cast<float2 *>(row) + c;
          const float2 val = *at;
          if (val.x != 0 || val.y != 0) {
            *at = make_float2(0, 0);
            if (out) atomic_add_bf16x2(gdist_b + (size_t)(e0 + 2 * c) * 2, val.x, val.y);
          }
        } else {
          const float val = row[c];
          if (val != 0) {
            row[c] = 0;
            if (out) scatter_add(gdist_r, gdist_f, (e0 + c) * 4, val);
          }
        }
      }
    };
    if (sh == 6) {                                          // a pixel per wavefront: its place is a scalar
      for (int i = __builtin_amdgcn_readfirstlane(first / kWave); i < rows; i += threads / kWave) add_pixel(i);
    } else {
      for (int i = first >> sh; i < rows; i += threads >> sh) add_pixel(i);
    }
  };

  // Both roles run the same sequence of turns and barriers, each in a loop of its own: what a role keeps in registers
  // from turn to turn then never competes with the other role's registers.
  //   pass t: points [base, base + PP) of item `it` (g, valid); pass t - 1: item it1 (valid1, last1: its item's last
  //   pass); last2, it2: the same of pass t - 2
  if (walker) {
    // =========================== walkers ===========================
    // What a lane owns.  With ArgsFrom::anew it is worked out anew in every block that needs it (from a copy of the lane number that
    // the compiler does not see through): kept from turn to turn it would cost the registers that the value rows and sums need.
    struct Owner {
      int lane, cl, group, crow, ccol;                       // lane of the wavefront, of its group; the group's cell
      LaneChannels<T, VEC, LPR> ch;
      __device__ __forceinline__ Owner(unsigned lane, int wave, int C)
          : lane(lane), cl(lane % LPR), group(lane / LPR), crow(wave * ROWS + lane / LPR / TX), ccol(lane / LPR % TX), ch(lane % LPR, C) {}
      // x of the lane `back` lanes before this one
      __device__ __forceinline__ float from_before(float x, int back) const {
        return __int_as_float(__builtin_amdgcn_ds_bpermute((lane - back) << 2, __float_as_int(x)));
      }
    };
    auto owner = [&](auto a) {
      unsigned l = lane;
      if (ARGS == ArgsFrom::anew) asm volatile("" : "+v"(l));
      return Owner(l, wave, a->C);
    };
    auto decode = [&](const int4 &item, const int4 &geo) {
      ItemGeom g;
      g.bin = item.x; g.seg = item.y; g.n_item = item.z; g.sole = item.w;
      g.b = geo.x; g.m = head_of(geo.y);
      const int l = level_of(geo.y);
      g.H = s_lv[0][l]; g.W = s_lv[1][l]; g.Dd = s_lv[2][l]; g.start = s_lv[3][l];
      g.y0 = geo.z; g.x0 = geo.w;                            // pixel of the tile's row 0
      return g;
    };
    if (tid == 0) {
      CellFetch fetch;
      int4 rec[kDealt - 1], geo[kDealt - 1];
      fetch.start(ws, p, rec, geo);
      for (int k = 0; k < kDealt - 1; ++k) s_geom[k] = decode(rec[k], geo[k]);
      s_fetch = fetch;
    }
    __syncthreads();                                        // the first item's record is there

    auto put_lds = [&](const Owner &o, float *row, const float (&val)[VEC]) {
#pragma unroll
      for (int gi = 0; gi < VEC / 4; ++gi)
        *reinterpret_cast<float4 *>(row + o.ch.first[gi]) = make_float4(val[4 * gi], val[4 * gi + 1], val[4 * gi + 2], val[4 * gi + 3]);
    };
    // The sums of tile pixel (crow, ccol) of item q are complete in u.  Pixels 1..TY-1 x 1..7 belong to no neighbour's
    // halo: when the item writes its tile alone they are stored (grad_value is zero on entry, or the binning launches
    // cleared what is added to), else added.  Rim pixels go to their place in LDS, to be added by put_rim.
    auto put_pixel = [&](auto a, const Owner &o, const ItemGeom &q, const float (&u)[VEC], bool active) {
      const int S = a->S, M = a->M, C = a->C;
      const bool gv16 = (a->grad16 & 1) != 0;               // uniform
      void *grad_value = a->grad_value;
      const int y = q.y0 + o.crow, x = q.x0 + o.ccol;
      if (active && (o.crow == 0 || o.ccol == 0)) put_lds(o, rim + rim_index(o.crow, o.ccol, TY, TX) * ROW, u);
      if (active && o.crow > 0 && o.ccol > 0 && y < q.H && x < q.W) {
        char *gvalue_b = static_cast<char *>(grad_value) + (size_t)q.b * S * M * C * (gv16 ? 2 : 4);
        float *gvalue_f = reinterpret_cast<float *>(gvalue_b);
        const rsrc_t gvalue_r = make_rsrc(gvalue_b, (size_t)S * M * C * sizeof(float));
        const uint32_t e = (uint32_t)(((q.start + y * q.W + x) * M + q.m) * C);
#pragma unroll
        for (int gi = 0; gi < VEC / 4; ++gi) {
          const uint32_t at = e + o.ch.first[gi];
          const float4 f = make_float4(u[4 * gi], u[4 * gi + 1], u[4 * gi + 2], u[4 * gi + 3]);
          if (o.ch.first[gi] < C) {
            if (q.sole != 0) {                              // uniform
              if (gv16) *reinterpret_cast<uint2 *>(gvalue_b + (size_t)at * 2) = make_uint2(pack_bf16x2(f.x, f.y), pack_bf16x2(f.z, f.w));
              else *reinterpret_cast<float4 *>(gvalue_f + at) = f;
            } else if (gv16) {
              atomic_add_bf16x2(gvalue_b + (size_t)at * 2, f.x, f.y);
              atomic_add_bf16x2(gvalue_b + (size_t)at * 2 + 4, f.z, f.w);
            } else {
              scatter_add(gvalue_r, gvalue_f, at * 4, f.x); scatter_add(gvalue_r, gvalue_f, at * 4 + 4, f.y);
              scatter_add(gvalue_r, gvalue_f, at * 4 + 8, f.z); scatter_add(gvalue_r, gvalue_f, at * 4 + 12, f.w);
            }
          }
        }
      }
    };
    // Rim pixels of tile row `ry` of item q, whose sums this wavefront left in LDS: the whole row where it is the tile's first or last, else its
    // first and last pixel.  What is the same for the row is in scalars.
    auto put_rim = [&](auto a, const ItemGeom &q, int ry) {
      if ((unsigned)(q.y0 + ry) >= (unsigned)q.H) return;   // uniform
      const int S = a->S, M = a->M, C = a->C;
      const bool gv16 = (a->grad16 & 1) != 0, whole = ry == 0 || ry == TY;      // uniform
      void *grad_value = a->grad_value;
      char *gvalue_b = static_cast<char *>(grad_value) + (size_t)q.b * S * M * C * (gv16 ? 2 : 4);
      float *gvalue_f = reinterpret_cast<float *>(gvalue_b);
      const rsrc_t gvalue_r = make_rsrc(gvalue_b, (size_t)S * M * C * sizeof(float));
      constexpr int kRowLog2 = ROW == 64 ? 6 : ROW == 32 ? 5 : 4;
      const int sh = gv16 ? kRowLog2 - 1 : kRowLog2;        // lanes per pixel: a float, or a pair of bfloat16 (log2)
      const int c = (lane & ((1 << sh) - 1)) * (gv16 ? 2 : 1), pixels = whole ? TW : 2, apart = whole ? 1 : TX;
      const uint32_t col_step = (uint32_t)(M * C), e_row = (uint32_t)(q.start + (q.y0 + ry) * q.W + q.x0) * col_step + (uint32_t)(q.m * C);
      const float *row = rim + rim_index(ry, 0, TY, TX) * ROW + c;
#pragma unroll 1
      for (int i = lane >> sh; i < pixels; i += kWave >> sh) {
        const int rx = i * apart;
        const float f0 = row[i * ROW], f1 = gv16 ? row[i * ROW + 1] : 0.f;
        if (c < C && (unsigned)(q.x0 + rx) < (unsigned)q.W && (f0 != 0 || f1 != 0)) {
          const uint32_t e = e_row + (uint32_t)rx * col_step + (uint32_t)c;
          if (gv16) atomic_add_bf16x2(gvalue_b + (size_t)e * 2, f0, f1);
          else scatter_add(gvalue_r, gvalue_f, e * 4, f0);
        }
      }
    };

    int turn = 0, it = 0;                                    // of phase X; the item being walked
    ItemGeom g = uniform(s_geom[0]);
    constexpr int kRows = PP / 4, IN_FLIGHT = kRows / GPW < 4 ? kRows / GPW : 4;   // rows per walker wavefront; loads asked for at once

    // Always true, which the compiler cannot know: keeps the walk in a block of its own.  Scheduled together with what
    // surrounds it, it spills registers, and every reload waits for all of the wavefront's memory accesses.
    auto apart = []() {
      int yes = 1;
      asm volatile("" : "+s"(yes));
      return yes != 0;
    };
    // phase X: the counters of the pass sorted in the phase Y before this turn's
    auto clear_counts = [&]() {
      unsigned i = tid;
      asm volatile("" : "+v"(i));
      if (i < (unsigned)CELLS) cnt[(turn + 2) % 3 * CELLS + i] = 0;
    };
    // phase Y: the grad_out rows of the pass come to LDS; they must be there before the phase ends (wait_for_loads()).  (The
    // pointers, whose work in phase Y is the longer one, brought them before: tile kernel 1158 -> 1121 us at the base shape,
    // bfloat16 1045 -> 1022, dense 4245 -> 4160, small 111 -> 106.)
    // Rows of whole 16-byte pieces go straight there, a piece per lane, without a register in between.  Where a row is shorter than
    // its lane group, a lane beyond its channels asks beyond the buffer.  (Brought by registers, whose wait came before the value rows
    // were asked for, rows of 40 channels took 737 us in bfloat16, 714 in float, and straight 706 and 685: tile kernel, 4 x 4000 queries,
    // four levels from 116 x 200, 32 points a query; on a sparse map, 400 x 400 with 8000 queries of 4 points, 554 -> 514 and 514 -> 471,
    // 20 channels in float 277 -> 258.)
    const bool straight = sizeof(T) == 4 || (arg()->C & 7) == 0;         // uniform
    auto stage_straight = [&](int n) {
      const auto a = arg();
      const int Q = a->Q, M = a->M, C = a->C;
      const T *grad_out = a->grad_out;
      // Instructions take turns over the wavefronts and stop where the pass's points do: an item of a few dozen points
      // asks for its rows in one or two of each (6 x 2000 queries, four levels from 116 x 200, 32 points a query: tile kernel
      // 535 -> 526 us).
      constexpr int RL = ROW * (int)sizeof(T) / 16, RPI = kWave / RL, N = kRows / RPI, NB = N < 2 ? N : 2;      // lanes per row, rows per instruction
      const rsrc_t go_r = make_rsrc(grad_out + (size_t)g.b * Q * M * C, (size_t)Q * M * C * sizeof(T));
      unsigned l = lane;
      asm volatile("" : "+v"(l));                            // (not worth registers from turn to turn)
      const int r0 = wave * RPI, at = r0 + (int)(l / RL);
      // this lane's piece, the same in every instruction: the order of a row's pieces repeats within the rows of one
      static_assert(piece_at<T, RL * 16>(4 * RPI, 0) % (RL * 16) == 0, "");
      const uint32_t piece = piece_at<T, RL * 16>(at, l % RL) % (RL * 16), from = piece < (uint32_t)C * (uint32_t)sizeof(T) ? piece : kNoChan;
#pragma unroll
      for (int j0 = 0; j0 < N; j0 += NB) {
        if (j0 > 0 && r0 + j0 * 4 * RPI >= n) break;         // uniform
        uint32_t row[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) row[j] = goff[(turn & 1) * PP + (j0 + j) * 4 * RPI + at];
#pragma unroll
        for (int j = 0; j < NB; ++j) load_to_lds16(go_r, gstage + (r0 + (j0 + j) * 4 * RPI) * RL * 16, row[j] + from);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // Rows that end within a piece (2-byte elements, an odd number of groups of four).  The loads end in registers that are put
    // into LDS: what else the phase asks for comes first, so that there is one wait (44 channels: 749 -> 729 us, sparse 567 -> 536).
    auto stage_by_registers = [&]() {
      const auto a = arg();
      const int Q = a->Q, M = a->M, C = a->C;
      const T *grad_out = a->grad_out;
      const Owner o = owner(a);
      const rsrc_t go_r = make_rsrc(grad_out + (size_t)g.b * Q * M * C, (size_t)Q * M * C * sizeof(T));
      const uint32_t *offs_of = goff + (turn & 1) * PP + wave * kRows;
#pragma unroll
      for (int j0 = 0; j0 < kRows / GPW; j0 += IN_FLIGHT) {
        typename LaneChannels<T, VEC, LPR>::Raw gg[IN_FLIGHT];
#pragma unroll
        for (int j = 0; j < IN_FLIGHT; ++j) o.ch.load(go_r, offs_of[(j0 + j) * GPW + o.group], gg[j]);
#pragma unroll
        for (int j = 0; j < IN_FLIGHT; ++j) o.ch.put(gstage, wave * kRows + (j0 + j) * GPW + o.group, o.cl, gg[j]);
      }
    };
    // phase X: walk the lists of the staged pass.  A group whose list has ended goes on with the row of zeros and weight zero
    // (the matrix instructions ignore the execution mask).
    // 2-byte elements: four points per step and group.  Each lane of four takes the row of one of them for the dots, which are
    // products of matrices then (v_mfma_f32_4x4x4, four channels deep), and all four take all of them for the sums.
    // The step takes a third of the vector instructions that four steps of one point do, for two and a half times the reads
    // from LDS, and does the work of four also where a cell has one point (walks_fours()): base shape 1061 -> 1040 us.  With 4-byte elements, where
    // a matrix instruction is one channel deep and a row twice as long, it lost: plain attention 209 -> 227 us, base shape 1194 -> 1277.
    auto walk_fours = [&](const auto &v, f4 (&acc)[VEC]) {
      const Owner o = owner(arg());
      const int corner = o.cl & 3, cell = o.crow * TX + o.ccol;
      const bool cell_ok = o.crow < TY;
      const int beg = cell_ok ? offs[cell] : 0, n = cell_ok ? offs[cell + 1] - beg : 0;
      int mine = s_slot[corner < n ? beg + corner : PP];
      for (int t = 0; __any(t < n); t += 4) {
        WholeRow<T, VEC, LPR> g;
        g.get(gstage, mine, o.cl >> 2);
        int s[4];
        float w[4];
        s[0] = __builtin_amdgcn_mov_dpp(mine, 0x00, 0xF, 0xF, true);      // quad_perm [k,k,k,k]
        s[1] = __builtin_amdgcn_mov_dpp(mine, 0x55, 0xF, 0xF, true);
        s[2] = __builtin_amdgcn_mov_dpp(mine, 0xAA, 0xF, 0xF, true);
        s[3] = __builtin_amdgcn_mov_dpp(mine, 0xFF, 0xF, 0xF, true);
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = dots[s[k] * 4 + corner];
        const int ahead = s_slot[t + 4 + corner < n ? beg + t + 4 + corner : PP];
        f4 d = corner_dots<T, VEC, LPR>(v, g);
        __builtin_amdgcn_sched_barrier(0);                  // (the whole rows' registers are free)
        typedef typename LaneChannels<T, VEC, LPR>::Raw Raw;
        if (LPR == 8) {                                     // the other half of the channels
#pragma unroll
          for (int k = 0; k < 4; ++k) d[k] += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(d[k]), 0x104, 0xF, 0xF, true));   // row_shl:4
        }
#pragma unroll
        for (int k0 = 0; k0 < 4; k0 += 2) {
          Raw r[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) o.ch.get(gstage, s[k0 + k], o.cl, r[k]);
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            float gk[VEC];
            LaneChannels<T, VEC, LPR>::to_float(r[k], gk);
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc[i] = __builtin_amdgcn_mfma_f32_4x4x1f32(w[k0 + k], gk[i], acc[i], 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        wave_lds_handover();                                // the weights have been read: the dots take their place
        if (t + corner < n && o.cl < 4) *reinterpret_cast<float4 *>(dots + mine * 4) = make_float4(d[0], d[1], d[2], d[3]);
        mine = ahead;
      }
    };

    // One point per step and group; the next step's row and weights and the slot after that are asked for while
    // this step's sums are formed, so that no LDS round trip is waited for with nothing to do.  Two steps to a turn of the loop,
    // which leaves what was read ahead in its registers (a copy of row and weights each step: tile kernel, base shape 1077 us for 1064, dense 3940
    // for 3865, in the 200 x 200 layer 1129 for 1084).
    auto walk_ones = [&](const auto &v, f4 (&acc)[VEC]) {
      const Owner o = owner(arg());
      const int corner = o.cl & 3, cell = o.crow * TX + o.ccol;
      const bool cell_ok = o.crow < TY;
      const int beg = cell_ok ? offs[cell] : 0, n = cell_ok ? offs[cell + 1] - beg : 0;
      const uint16_t *p = s_slot + beg, *const end = p + n, *const none = s_slot + PP;
      auto slot_at = [&](const uint16_t *q) { return (int)*(q < end ? q : none); };
      struct Ahead {
        typename LaneChannels<T, VEC, LPR>::Raw row;
        float w, *at;                                        // the corner's weight, and where it lies: the dot product takes its place
      };
      auto read = [&](int s, Ahead &a) {
        a.at = dots + s * 4 + corner;
        o.ch.get(gstage, s, o.cl, a.row);
        a.w = *a.at;
      };
      auto step = [&](const uint16_t *q, const Ahead &now, int &s, Ahead &next) {
        const int after = slot_at(q + 2);
        read(s, next);
        s = after;
        float d[4], g0[VEC];
        LaneChannels<T, VEC, LPR>::to_float(now.row, g0);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          d[k] = v[k][0] * g0[0];
#pragma unroll
          for (int i = 1; i < VEC; ++i) d[k] += v[k][i] * g0[i];
        }
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] = __builtin_amdgcn_mfma_f32_4x4x1f32(now.w, g0[i], acc[i], 0, 0, 0);
        float dot = quad_corner_sum(d[0], d[1], d[2], d[3], (o.cl & 1) != 0, (o.cl & 2) != 0);      // lane c: corner c
        if (LPR == 8) dot += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(dot), 0x104, 0xF, 0xF, true));   // row_shl:4
        if (q < end && o.cl < 4) *now.at = dot;
      };
      Ahead a, b;
      read(slot_at(p), a);
      int s = slot_at(p + 1);
      for (; __any(p < end); p += 2) {
        step(p, a, s, b);
        if (!__any(p + 1 < end)) break;
        step(p + 1, b, s, a);
      }
    };

    auto walk = [&](const auto &v, f4 (&acc)[VEC]) {
      if constexpr (FOURS) walk_fours(v, acc);
      else walk_ones(v, acc);
    };

    if (g.bin >= 0) {
      CT_MARK(0);
      lds_barrier();                                         // X(0): nothing to walk yet
      bool have_prev = false;
      f4 acc[VEC];                                           // acc[channel][corner] of the item before, then of this one
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] = (f4){0, 0, 0, 0};
      for (;;) {                                             // items: from the phase Y of one's first pass to the next one's
        const bool done = g.bin < 0;
        const int r0 = wave * ROWS;                          // this wavefront's first tile row
        float u[VEC];                                        // sums of this group's pixel, on their way out
#pragma unroll
        for (int i = 0; i < VEC; ++i) u[i] = 0;
        CT_MARK(0);
        const auto now = arg();                              // read once for all of the change of items (C = 64, 1.28 M points on 400 x 400: 583 -> 574 us)
        // The record of the item three on, first of all: what thread 0 waits for was asked for an item ago.
        if (tid == 0 && !done) {
          CellFetch fetch = s_fetch;
          int4 rec, geo;
          const BinWorkspace w = args<T, ArgsFrom::anew>(param)->ws;
          fetch.advance(w, *w.plan, &rec, &geo);
          s_geom[slot_of_item(it + 3)] = decode(rec, geo);
          s_fetch = fetch;
        }
        if (have_prev) {
          // The item before is over.  Tile pixel (r, c) collects corner 0 of cell (r, c), corner 1 of (r, c - 1), corner 2
          // of (r - 1, c - 1) and corner 3 of (r - 1, c): the cell to the left is the lane group to the left, the row
          // above the lower half of this wavefront, or the wavefront before it.
          const Owner o = owner(now);
          float dn[VEC], ux[VEC], dx[VEC];                   // for the row below; the same of the ninth pixel (last cell)
#pragma unroll
          for (int i = 0; i < VEC; ++i) {
            const float l1 = o.from_before(acc[i][1], LPR), l2 = o.from_before(acc[i][2], LPR);
            u[i] = acc[i][0] + (o.ccol > 0 ? l1 : 0.f);
            dn[i] = acc[i][3] + (o.ccol > 0 ? l2 : 0.f);
            ux[i] = acc[i][1];
            dx[i] = acc[i][2];
            if (ROWS == 2) {
              const float up = o.from_before(dn[i], kWave / 2), upx = o.from_before(dx[i], kWave / 2);
              if (o.group >= TX) { u[i] += up; ux[i] += upx; }
            }
          }
          if (o.crow < TY) {
            if (o.ccol == TX - 1) put_lds(o, rim + rim_index(o.crow, TX, TY, TX) * ROW, ux);
            if (o.crow + 1 == TY) {
              put_lds(o, rim + rim_index(TY, o.ccol, TY, TX) * ROW, dn);
              if (o.ccol == TX - 1) put_lds(o, rim + rim_index(TY, TX, TY, TX) * ROW, dx);
            } else if (o.group >= (ROWS - 1) * TX) {         // for the wavefront below
              put_lds(o, cross + (wave * TW + o.ccol) * ROW, dn);
              if (o.ccol == TX - 1) put_lds(o, cross + (wave * TW + TX) * ROW, dx);
            }
          }
          if (ROWS == 2) put_pixel(now, o, uniform(s_geom[slot_of_item(it - 1)]), u, o.crow < TY && o.group >= TX);   // the second row is complete
        }
        CT_MARK(3);
        if (!done && straight) stage_straight(g.n_item);
        typename LaneChannels<T, VEC, LPR>::Raw vr[4];
        {
          // the four value rows of this group's cell (zero outside the map, when the cell is not part of the tile, or when
          // there is no item)
          const int S = now->S, M = now->M, C = now->C;
          const T *value = now->value;
          const Owner o = owner(now);
          const rsrc_t value_r = make_rsrc(value + (size_t)g.b * S * M * C, (size_t)S * M * C * sizeof(T));
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int y = g.y0 + o.crow + (k >= 2 ? 1 : 0), x = g.x0 + o.ccol + ((k == 1 || k == 2) ? 1 : 0);
            const bool ok = !done && o.crow < TY && in_map(y, x, g.H, g.W);
            o.ch.load(value_r, ok ? (uint32_t)(((g.start + y * g.W + x) * M + g.m) * C * (int)sizeof(T)) : kNoRow, vr[k]);
          }
        }
        if (!done && !straight) stage_by_registers();
        wait_for_loads();
        CT_MARK(6);
        lds_barrier();
        CT_MARK(4);
        // ---------------- phase X of the first pass ----------------
        ++turn;
        clear_counts();
        if (have_prev && r0 < TY) {                          // uniform
          // The first tile row of this wavefront collects what the wavefront before it left for it; then the rim goes out.
          const ItemGeom q = uniform(s_geom[slot_of_item(it - 1)]);
          const Owner o = owner(now);
          const bool mine = o.crow < TY && o.group < TX;
          if (wave > 0 && mine) {
            const float *from = cross + ((wave - 1) * TW + o.ccol) * ROW;
#pragma unroll
            for (int gi = 0; gi < VEC / 4; ++gi) {
              const float4 a = *reinterpret_cast<const float4 *>(from + o.ch.first[gi]);
              u[4 * gi] += a.x; u[4 * gi + 1] += a.y; u[4 * gi + 2] += a.z; u[4 * gi + 3] += a.w;
              if (o.ccol == TX - 1) {
                float4 *at = reinterpret_cast<float4 *>(rim + rim_index(o.crow, TX, TY, TX) * ROW + o.ch.first[gi]);
                const float4 b = *reinterpret_cast<const float4 *>(from + ROW + o.ch.first[gi]), c = *at;
                *at = make_float4(c.x + b.x, c.y + b.y, c.z + b.z, c.w + b.w);
              }
            }
          }
          put_pixel(now, o, q, u, mine);
          wave_lds_handover();
#pragma unroll 1
          for (int ry = r0; ry < min(r0 + ROWS, TY); ++ry) put_rim(now, q, ry);      // uniform
          if (r0 + ROWS >= TY) put_rim(now, q, TY);
        }
        if (done) break;
        typename std::conditional<FOURS, WholeRow<T, VEC, LPR>, float[4][VEC]>::type v;      // the four value rows
        if constexpr (FOURS) {
          whole_rows<T, VEC, LPR>(vr, owner(now).cl, v);
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k) LaneChannels<T, VEC, LPR>::to_float(vr[k], v[k]);
        }
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] = (f4){0, 0, 0, 0};
        CT_MARK(5);
        if (apart()) walk(v, acc);
        CT_MARK(1);
        lds_barrier();
        CT_MARK(2);
        for (int base = PP; base < g.n_item; base += PP) {   // the item's further passes
          if (straight) stage_straight(g.n_item - base);
          else stage_by_registers();
          wait_for_loads();
          CT_MARK(6);
          lds_barrier();
          CT_MARK(4);
          ++turn;
          clear_counts();
          if (apart()) walk(v, acc);
          CT_MARK(1);
          lds_barrier();
          CT_MARK(2);
        }
        have_prev = true;
        ++it;
        g = uniform(s_geom[slot_of_item(it)]);
      }
    }
  } else {
    // =========================== pointers ===========================
    // What a point needs from memory is asked for ahead of time: its record two turns, its depth taps one phase before
    // they are used.  Loads and stores that are always issued (inactive lanes with offsets beyond the buffer) let the
    // waits be counted: a wait for a load does not have to include the stores issued after it.
    const int pslot = tid - kWalkers;                        // the point slot of this thread
    PointState cur, nxt;                                     // of pass t - 1 and of pass t
    TapsInFlight<T> taps;                                    // of the pass prepared last
    u32x4 given = {0, 0, 0, 0};                              // (stage 2 alone) its given scores
    int rank = 0;                                            // place of its point among the points of its cell
    cur.bits = 0; nxt.bits = 0;
    cur.gp = nxt.gp = 0; cur.a = nxt.a = 0; cur.lh = cur.lw = cur.ld = nxt.lh = nxt.lw = nxt.ld = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) { cur.sc[k] = cur.hl[k] = nxt.sc[k] = nxt.hl[k] = 0; taps.t[k] = (u32x2){0, 0}; }
    __syncthreads();                                        // the first items' records are there

    ItemGeom g = uniform(s_geom[0]);                         // pass A (the one prepared last): points [base, base + PP) of item `it`
    int it = 0, base = 0;
    int rec_it = 0, rec_base = 0, rec_bin = g.bin, rec_seg = g.seg, rec_n = g.n_item;      // the pass whose records were asked for last
    uint32_t pre_gp = 0;
    float4 pre_rec = make_float4(0, 0, 0, 0);
    auto ask_records = [&]() {
      const int at = rec_bin >= 0 ? rec_seg + rec_base + min(pslot, rec_n - rec_base - 1) : 0;
      const auto a = arg();
      pre_gp = a->ws.entries[at];
      pre_rec = a->ws.recs[at];
    };
    auto next_records = [&]() {
      if (rec_bin >= 0) {
        rec_base += PP;
        if (rec_base >= rec_n) {
          ++rec_it;
          rec_base = 0;
          const ItemGeom &q = s_geom[slot_of_item(rec_it)];
          rec_bin = __builtin_amdgcn_readfirstlane(q.bin); rec_seg = __builtin_amdgcn_readfirstlane(q.seg);
          rec_n = __builtin_amdgcn_readfirstlane(q.n_item);
        }
      }
    };
    // geometry of this thread's point of pass A, its place in the sort, its grad_out row for the walkers; its taps are asked for
    auto prepare = [&](int pass, const f4 &rec, uint32_t index) {
      const auto ar = arg();
      const int D = ar->D, S = ar->S, M = ar->M, Md = ar->Md, Q = ar->Q, C = ar->C;
      const T *dist = ar->dist, *score_in = ar->score_in;
      const FastDiv div_lp = ar->div_lp;
      const bool live = g.bin >= 0 && pslot < g.n_item - base;
      const uint32_t gp = live ? index : 0u;
      const uint32_t unit = div_lp.div(gp);
      goff[(pass & 1) * PP + pslot] = live ? (unit - (uint32_t)g.b * (uint32_t)Q * (uint32_t)M) * (uint32_t)(C * (int)sizeof(T)) : kNoRow;
      const Point2D<float> pg = locate_2d<float>(rec.x, rec.y, g.H, g.W, g.start);
      const bool in = live && pg.inside;
      DepthTap<float> tap;
      tap.inside = tap.lo_ok = tap.hi_ok = false; tap.d0 = 0; tap.ld = tap.hd = 0;
      unsigned on_bits = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) on_bits |= (in && pg.key[k] >= 0) ? 1u << k : 0u;
      if (FUSED) {
        tap = locate_depth<float>(rec.z, g.Dd);
        const int md = Md == 1 ? 0 : g.m, db = min(max(tap.d0, 0), max(D - 2, 0));
        const rsrc_t dist_r = make_rsrc(dist + (size_t)g.b * S * Md * D, (size_t)S * Md * D * sizeof(T));
        uint32_t off[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          off[k] = ((on_bits >> k & 1) && tap.inside) ? (uint32_t)(((pg.key[k] * Md + md) * D + db) * (int)sizeof(T)) : kNoRow;
        taps.ask(dist_r, off, D);
      } else if (score_in != nullptr) {                      // uniform
        const T *si = score_in + (size_t)gp * 4;
        if constexpr (sizeof(T) == 4) {
#pragma unroll
          for (int k = 0; k < 4; ++k) given[k] = __float_as_uint(si[k]);
        } else {
          const uint16_t *sh = reinterpret_cast<const uint16_t *>(si);
#pragma unroll
          for (int k = 0; k < 4; ++k) given[k] = (uint32_t)sh[k] << 16;
        }
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) given[k] = __float_as_uint(1.f);
      }
      // the cell: the base pixel within the tile (the binning put the point into this tile by it)
      const int cy = min(max(pg.h0 - g.y0, 0), TY - 1), cx = min(max(pg.w0 - g.x0, 0), TX - 1), cell = cy * TX + cx;
      if (in) rank = atomicAdd(cnt + pass % 3 * CELLS + cell, 1);
      nxt.gp = gp; nxt.a = rec.w; nxt.lh = pg.lh; nxt.lw = pg.lw; nxt.ld = tap.ld;
      nxt.bits = on_bits | (tap.inside ? 16u : 0u) | (tap.lo_ok ? 32u : 0u) | (tap.hi_ok ? 64u : 0u) | (in ? 128u : 0u) |
                 ((unsigned)(in ? cell : 0) << 8) | ((unsigned)(tap.d0 + 1) << 16);
    };
    // The record asked for last.  All of it at once, whether a pass follows or not: a part that the compiler moves elsewhere
    // before is waited for where the turn before ends, and that turn's stores with it; one that is still on its way where its
    // register is needed is waited for behind the depth taps.  Six cameras, 30825 rows, 8 x 32 channels, 32 + 8 points: 1065
    // -> 1057 us; 100 bins, 24 planes of 58 x 100: 3862 -> 3840.
    auto take_record = [&](f4 &rec, uint32_t &index) {
      rec = (f4){pre_rec.x, pre_rec.y, pre_rec.z, pre_rec.w};
      index = pre_gp;
      asm volatile("" : "+v"(rec), "+v"(index));
    };
    f4 rec;
    uint32_t index;
    ask_records();
    take_record(rec, index);
    prepare(0, rec, index);
    next_records();
    ask_records();

    int it1 = 0, it2 = 0;
    bool valid1 = false, last1 = false, last2 = false;
    for (int turn = 0;; ++turn) {                            // uniform over the workgroup
      const bool valid = g.bin >= 0, last = valid && base + PP >= g.n_item;
      const int it_now = it;
      CT_MARK(0);
      // ---------------- phase X: scores and corner weights of pass t, prepare pass t + 1 ----------------
      float4 pw = make_float4(0, 0, 0, 0);                  // corner weights of this thread's point
      if (valid) {
        const int D = arg()->D;
        const float hh = 1 - nxt.lh, hw = 1 - nxt.lw;
        const int d0 = (int)(nxt.bits >> 16) - 1, db = min(max(d0, 0), max(D - 2, 0));
        const bool lo_ok = (nxt.bits & 32u) != 0, hi_ok = (nxt.bits & 64u) != 0;
        const float hd = (nxt.bits & 16u) != 0 ? 1 - nxt.ld : 0.f;
        float wk[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (FUSED) {
            float x, y;
            taps.get(k, db, D, x, y);
            const float lo = (lo_ok && d0 == db) ? x : (lo_ok && d0 == db + 1) ? y : 0.f;
            const float hi = (hi_ok && d0 + 1 == db) ? x : (hi_ok && d0 == db) ? y : 0.f;
            nxt.sc[k] = depth_lerp(lo, hi, hd, nxt.ld);
            nxt.hl[k] = hi - lo;
          } else {
            nxt.sc[k] = __uint_as_float(given[k]);
          }
          const float bk = k == 0 ? hh * hw : k == 1 ? hh * nxt.lw : k == 2 ? nxt.lh * nxt.lw : nxt.lh * hw;
          wk[k] = (nxt.bits >> k & 1) ? bk * nxt.sc[k] * nxt.a : 0.f;
        }
        pw = make_float4(wk[0], wk[1], wk[2], wk[3]);
      }
      const PointState now = nxt;                            // of pass t
      const int rank_now = rank;
      base += PP;
      if (last) { ++it; base = 0; g = uniform(s_geom[slot_of_item(it)]); }
      nxt.bits = 0;
      take_record(rec, index);
      if (g.bin >= 0) prepare(turn + 1, rec, index);
      next_records();
      ask_records();
      CT_MARK(1);
      if (FUSED && last2) flush_gd(slot_of_item(it2), pslot, PP);
      if (!valid && !valid1) break;
      CT_MARK(2);
      lds_barrier();
      CT_MARK(3);
      // ---------------- phase Y: place pass t, finish pass t - 1 ----------------
      const auto ar = arg();
      const int D = ar->D, gl_stride = ar->gl_stride;
      const T *grad_score_in = ar->grad_score_in;
      float *grad_loc = ar->grad_loc, *grad_attn = ar->grad_attn, *grad_score_out = ar->grad_score_out;
      const float *grad_wu = ar->grad_wu;
      const uint32_t slice = (uint32_t)ar->Q * (uint32_t)ar->M * (uint32_t)(ar->L * ar->P);      // points of a batch element
      const float4 d4 = *reinterpret_cast<const float4 *>(dots + pslot * 4);       // of pass t - 1, before its place is taken
      if (valid) {
        // exclusive prefix of the cell counters; every pointer wavefront computes it and writes the same numbers,
        // so it can go on with its own copy without waiting for the others
        const int c = lane < CELLS ? cnt[turn % 3 * CELLS + lane] : 0;
        const int inc = wave_inclusive_scan(c);
        if (lane < CELLS) offs[lane] = inc - c;
        if (lane == kWave - 1) offs[CELLS] = inc;
        *reinterpret_cast<float4 *>(dots + pslot * 4) = pw;
        if (now.bits & 128u) s_slot[offs[(now.bits >> 8) & 63] + rank_now] = (uint16_t)pslot;
      }
      CT_MARK(4);
      if (valid1) {
        const ItemGeom &q = s_geom[slot_of_item(it1)];
        const int gH = __builtin_amdgcn_readfirstlane(q.H), gW = __builtin_amdgcn_readfirstlane(q.W), gDd = __builtin_amdgcn_readfirstlane(q.Dd);
        const int gb = __builtin_amdgcn_readfirstlane(q.b);
        const bool live = (cur.bits & 128u) != 0;
        Point2D<float> pg;
        DepthTap<float> tap;
        pg.lh = cur.lh; pg.lw = cur.lw; pg.hh = 1 - cur.lh; pg.hw = 1 - cur.lw;
        tap.inside = (cur.bits & 16u) != 0; tap.lo_ok = (cur.bits & 32u) != 0; tap.hi_ok = (cur.bits & 64u) != 0;
        tap.d0 = (int)(cur.bits >> 16) - 1; tap.ld = cur.ld; tap.hd = tap.inside ? 1 - cur.ld : 0.f;
        const unsigned on_bits = cur.bits & 15u;
        const int ccell = (cur.bits >> 8) & 63, ccy = ccell / TX, ccx = ccell % TX;
        const float a = cur.a;
        const float dc[4] = {d4.x, d4.y, d4.z, d4.w};
        float gs[4], sk[4], ga = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool on = on_bits >> k & 1;
          const float bk = pg.bil(k);
          gs[k] = on ? bk * a * dc[k] : 0.f;
          sk[k] = on ? cur.sc[k] * dc[k] : 0.f;
          ga += bk * sk[k];
        }
        const float gx = (float)gW * a * (pg.hh * (sk[1] - sk[0]) + pg.lh * (sk[2] - sk[3]));
        const float gy = (float)gH * a * (pg.hw * (sk[3] - sk[0]) + pg.lw * (sk[2] - sk[1]));
        // where the point's gradients go, relative to its batch element
        const uint32_t at = live ? cur.gp - (uint32_t)gb * slice : 0u;
        const rsrc_t gl_r = make_rsrc(grad_loc + (size_t)gb * slice * gl_stride, (size_t)slice * gl_stride * 4);
        const rsrc_t ga_r = make_rsrc(grad_attn + (size_t)gb * slice, (size_t)slice * 4);
        const uint32_t gl_off = live ? at * (uint32_t)(gl_stride * 4) : kNoRow, ga_off = live ? at * 4 : kNoRow;
        if (FUSED) {
          if (grad_score_in != nullptr) {
            const T *gi = grad_score_in + (size_t)cur.gp * 4;
#pragma unroll
            for (int k = 0; k < 4; ++k) gs[k] += Elem<T>::ld(gi + k);
          }
          if (grad_wu != nullptr) {       // weight_update = sum over points of attn * mean corner score
            const float gw = grad_wu[ar->div_lp.div(cur.gp)] * 0.25f;
            ga += gw * (cur.sc[0] + cur.sc[1] + cur.sc[2] + cur.sc[3]);
#pragma unroll
            for (int k = 0; k < 4; ++k) gs[k] += gw * a;
          }
          float gz = 0;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            if (!tap.inside) gs[k] = 0.f;              // (a corner outside the map has none already)
            gz += gs[k] * cur.hl[k];
          }
          const u32x3 g3 = {__float_as_uint(gx), __float_as_uint(gy), __float_as_uint(gz * (float)gDd)};
          __builtin_amdgcn_raw_buffer_store_b96(g3, gl_r, gl_off, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ga), ga_r, ga_off, 0, 0);
          // The taps.  One that does not exist adds zero to a word nearby: the four pixels always lie in the tile, the bins
          // are clamped.
          if (live) {
            const int row0 = (ccy * TW + ccx) * D, lo_at = max(tap.d0, 0), hi_at = min(tap.d0 + 1, D - 1);
            const float w_lo = tap.lo_ok ? tap.hd : 0.f, w_hi = tap.hi_ok ? tap.ld : 0.f;
            int at[8];
            float tv[8];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const int row = row0 + (k == 0 ? 0 : k == 1 ? D : k == 2 ? (TW + 1) * D : TW * D);
              at[2 * k] = row + lo_at; at[2 * k + 1] = row + hi_at;
              tv[2 * k] = tap.lo_ok ? w_lo * gs[k] : 0.f; tv[2 * k + 1] = tap.hi_ok ? w_hi * gs[k] : 0.f;
            }
            lds_add_taps(gd, at, tv);
          }
        } else {
          const u32x2 g2 = {__float_as_uint(gx), __float_as_uint(gy)};
          __builtin_amdgcn_raw_buffer_store_b64(g2, gl_r, gl_off, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ga), ga_r, ga_off, 0, 0);
          if (grad_score_out != nullptr) {                   // uniform
            const rsrc_t gs_r = make_rsrc(grad_score_out + (size_t)gb * slice * 4, (size_t)slice * 16);
            const u32x4 g4 = {__float_as_uint(gs[0]), __float_as_uint(gs[1]), __float_as_uint(gs[2]), __float_as_uint(gs[3])};
            __builtin_amdgcn_raw_buffer_store_b128(g4, gs_r, live ? at * 16 : kNoRow, 0, 0);
          }
        }
      }
      cur = now;
      CT_MARK(5);
      lds_barrier();
      CT_MARK(6);
      it2 = it1; last2 = last1; it1 = it_now; valid1 = valid; last1 = last;
    }
  }
  CT_FLUSH();
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------
// The kernel takes rows of up to 64 channels, whole groups of four, on tiles 8 pixels wide of at most as many rows as
// its walkers own.  The row-owned tile kernel keeps the rest.
bool cell_kernel_applies(int C, int ty, int tx) { return C <= 64 && (C & 3) == 0 && tx == kCellTX && ty >= 1 && ty <= cell_max_ty(C); }

// Whether the walkers take the points of a cell four at a time.  Never with 4-byte elements (walk_fours).  With 2-byte elements a step of
// four costs about as much as three of one and is wasted on shorter lists, so it is taken from three quarters of a point per
// pixel on.  Tile kernel, one at a time against four, by points per pixel (uniform locations; the sign turns at 0.5 where they
// are clustered, + 1.5 % at 0.75):
//   32 channels, stage 2 on 400 x 400   0.15: 237, 256 us   0.5: 260, 271   0.75: 274, 281   1: 287, 289   1.5: 309, 310   3: 387, 383
//   32 channels, 16 bins, 232 x 400     0.15: 160, 165      0.5: 168, 171   0.75: 172, 174   1: 179, 180   1.5: 198, 196   3: 257, 254
//   64 channels, 16 bins, 232 x 400     0.15: 294, 306      0.5: 318, 331   0.75: 332, 339   1: 342, 348   1.5: 363, 363   3: 423, 421
// Rows of up to 16 channels, whose steps are short, gain at most 1 % below a third of a point, and lose from a half on.
static bool walks_fours(const BwdArgs &a, int dtype) {
  return dtype == DFA3D_BF16 && (cell_shape(a.C).vec == 4 || 4LL * a.Q * a.L * a.P >= 3LL * a.S);
}

template <typename T, int VEC, int LPR, bool FOURS>
static hipError_t launch_cell_cfg(const BwdArgs &a, const BinWorkspace &ws, size_t lds, int grid, float *gd_heads,
                                  hipStream_t stream) {
  const bool fused = a.dist != nullptr, one = a.dist_heads == 1;
  const CellArgs<T> c = {ws, (const T *)a.value, (const T *)a.dist, fused ? nullptr : (const T *)a.score_in, (const T *)a.grad_out,
                         fused ? (const T *)a.grad_score_in : nullptr, a.grad_value, gd_heads != nullptr ? (void *)gd_heads : a.grad_dist,
                         (float *)a.grad_loc, (float *)a.grad_attn, fused ? nullptr : (float *)a.grad_score_out,
                         fused ? (const float *)a.grad_weight_update : nullptr, a.grad_loc_stride,
                         fused && one ? 1 : a.M, fused && one && gd_heads == nullptr ? 1 : a.M,
                         a.B, a.S, a.M, a.C, fused ? a.D : 0, a.L, a.Q, a.P, FastDiv((uint32_t)(a.L * a.P)),
                         !fused ? 0 : (a.grad_bf16 ? 1 : 0) | (a.grad_bf16 && gd_heads == nullptr ? 2 : 0)};
  const dim3 block(kWalkers + cell_pass(LPR));
  if (fused) hipLaunchKernelGGL((cell_backward_kernel<T, VEC, LPR, true, FOURS>), dim3(grid), block, lds, stream, c);
  else hipLaunchKernelGGL((cell_backward_kernel<T, VEC, LPR, false, FOURS>), dim3(grid), block, lds, stream, c);
  return hipGetLastError();
}

template <typename T, int VEC, int LPR, bool FOURS> static const void *symbol_of(bool fused) {
  return fused ? reinterpret_cast<const void *>(cell_backward_kernel<T, VEC, LPR, true, FOURS>)
               : reinterpret_cast<const void *>(cell_backward_kernel<T, VEC, LPR, false, FOURS>);
}

#define DFA3D_CELL_DISPATCH(dtype, a, CALL)                                  \
  do {                                                                       \
    const CellShape s = cell_shape((a).C);                                   \
    const bool fours = walks_fours(a, dtype);                                \
    if (dtype == DFA3D_F32) {                                                \
      if (s.lpr == 8) return CALL(float, 8, 8, false);                       \
      if (s.vec == 8) return CALL(float, 8, 4, false);                       \
      return CALL(float, 4, 4, false);                                       \
    }                                                                        \
    if (s.lpr == 8 && fours) return CALL(__hip_bfloat16, 8, 8, true);        \
    if (s.lpr == 8) return CALL(__hip_bfloat16, 8, 8, false);                \
    if (s.vec == 8 && fours) return CALL(__hip_bfloat16, 8, 4, true);        \
    if (s.vec == 8) return CALL(__hip_bfloat16, 8, 4, false);                \
    return CALL(__hip_bfloat16, 4, 4, true);                                 \
  } while (0)

const void *cell_kernel_symbol(const BwdArgs &a, int dtype) {
#define DFA3D_CELL_SYMBOL(T, V, R, F) (symbol_of<T, V, R, F>(a.dist != nullptr))
  DFA3D_CELL_DISPATCH(dtype, a, DFA3D_CELL_SYMBOL);
#undef DFA3D_CELL_SYMBOL
}

hipError_t launch_cell_kernel(const BwdArgs &a, int dtype, const BinWorkspace &ws, size_t lds, int grid, float *gd_heads,
                              hipStream_t stream) {
#define DFA3D_CELL_LAUNCH(T, V, R, F) (launch_cell_cfg<T, V, R, F>(a, ws, lds, grid, gd_heads, stream))
  DFA3D_CELL_DISPATCH(dtype, a, DFA3D_CELL_LAUNCH);
#undef DFA3D_CELL_LAUNCH
}

}  // namespace dfa3d
