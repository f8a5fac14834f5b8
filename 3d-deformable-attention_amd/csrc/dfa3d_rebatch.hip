// Camera re-batching around the DFA3D operator for gfx950.
//
// DFA3D-BEVFormer's spatial cross-attention lets every camera attend only with the BEV queries that
// project into it: it copies those queries (and their reference points) into a per-camera batch
// before the operator and adds the per-camera results back into the BEV slots afterwards, in python
// loops over batch x cameras with one indexing kernel each
// (BEVFormer_DFA3D/projects/mmdet3d_plugin/bevformer/modules/spatial_cross_attention.py:716-722 and
// :741-748).  Here each direction is one kernel, and neither uses atomics:
//
//   rebatch_gather_kernel   dst[j, i, k, :] = scale[j, q] * src[i, j, q, :]   with q = index[i, k]
//                           (`pad`, usually zero, where index[i, k] < 0); also the backward of the combine
//   rebatch_queries_kernel  the gather of the queries, with what is added to each (their positions), and of the reference points
//   rebatch_combine_kernel  dst[j, q, :] = scale[j, q] * sum over cameras i with pos[i, q] >= 0 of
//                           src[j, i, pos[i, q], :]; also the backward of the gather
//
//   camera_hits_kernel      which cameras see a query, and one over how many do
//   camera_count_kernel, camera_index_kernel   the queries of each camera in ascending order, and the inverse
//                           (:704-707 is a nonzero call per camera)
//
// index (cams, max_len) lists the queries of each camera, pos (cams, Nq) is its inverse
// (position of query q in camera i's list, or -1).  Rows are E contiguous elements; a lane moves
// 16 bytes when the row length allows it.  Pure streaming: bound by HBM bandwidth.
#include "../../include/dfa3d.h"
#include "dfa3d_binned.h"
#include "dfa3d_launch.h"

namespace dfa3d {

constexpr int kRebatchBlock = 256;

template <typename T, int VEC> struct Pack { T v[VEC]; };

template <typename T, int VEC>
__device__ __forceinline__ Pack<T, VEC> load_pack(const T *p) {
  Pack<T, VEC> r;
  if (VEC * sizeof(T) == 16) {
    const uint4 t = *reinterpret_cast<const uint4 *>(p);
    __builtin_memcpy(&r, &t, 16);
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) r.v[i] = p[i];
  }
  return r;
}
template <typename T, int VEC>
__device__ __forceinline__ void store_pack(T *p, const Pack<T, VEC> &r) {
  if (VEC * sizeof(T) == 16) {
    uint4 t;
    __builtin_memcpy(&t, &r, 16);
    *reinterpret_cast<uint4 *>(p) = t;
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) p[i] = r.v[i];
  }
}

// Pieces of a row: piece number to row and piece, without a division in 64 bits where there are few enough.
struct Pieces {
  FastDiv by;
  int per;
  bool few;                            // fewer than 2^31 of them
  explicit Pieces(long long rows, int per) : by((uint32_t)per), per(per), few(rows * per < (1LL << 31)) {}
  __device__ __forceinline__ void place(long long u, long long &row, int &piece) const {
    row = few ? (long long)by.div((uint32_t)u) : u / per;    // uniform
    piece = (int)(u - row * per);
  }
};

// One thread per VEC elements of a destination row of one batch element and camera (blockIdx.y).
template <typename T, int VEC>
__global__ __launch_bounds__(kRebatchBlock) void rebatch_gather_kernel(
    const T *__restrict__ src, long long cam_stride, long long batch_stride, const int *__restrict__ index,
    const T *__restrict__ scale, T *__restrict__ dst, int bs, int cams, int max_len, int Nq, int E, T pad, Pieces pieces) {
  const long long total = (long long)max_len * pieces.per;
  for (int ji = blockIdx.y; ji < bs * cams; ji += gridDim.y) {
    const int j = ji / cams, i = ji - j * cams;
    for (long long t = (long long)blockIdx.x * kRebatchBlock + threadIdx.x; t < total; t += (long long)gridDim.x * kRebatchBlock) {
      long long k;
      int piece;
      pieces.place(t, k, piece);
      const int q = index[(long long)i * max_len + k], e = piece * VEC;
      Pack<T, VEC> r;
#pragma unroll
      for (int c = 0; c < VEC; ++c) r.v[c] = pad;
      if (q >= 0 && q < Nq) {
        r = load_pack<T, VEC>(src + i * cam_stride + j * batch_stride + (long long)q * E + e);
        if (scale != nullptr) {
          const T s = scale[(long long)j * Nq + q];
#pragma unroll
          for (int c = 0; c < VEC; ++c) r.v[c] *= s;
        }
      }
      store_pack<T, VEC>(dst + ((long long)ji * max_len + k) * E + e, r);
    }
  }
}

// One thread per VEC elements of a destination row of one batch element (blockIdx.y).  A query's places in four cameras' lists are asked for at once, then
// its rows: one after the other, each waits for the last one's place and row in turn (22500 queries of 256 in six cameras, a fifth in each, 14.3 us
// for 12.0 now; 40000 22.5, 18.0).
constexpr int kCamsAtOnce = 4;
template <typename T, int VEC>
__global__ __launch_bounds__(kRebatchBlock) void rebatch_combine_kernel(
    const T *__restrict__ src, const int *__restrict__ pos, const T *__restrict__ scale, T *__restrict__ dst,
    int bs, int cams, int max_len, int Nq, int E, Pieces pieces) {
  const long long total = (long long)Nq * pieces.per;
  for (int j = blockIdx.y; j < bs; j += gridDim.y) {
    for (long long t = (long long)blockIdx.x * kRebatchBlock + threadIdx.x; t < total; t += (long long)gridDim.x * kRebatchBlock) {
      long long q;
      int piece;
      pieces.place(t, q, piece);
      const int e = piece * VEC;
      Pack<T, VEC> acc;
#pragma unroll
      for (int c = 0; c < VEC; ++c) acc.v[c] = 0;
      for (int i0 = 0; i0 < cams; i0 += kCamsAtOnce) {       // cameras in order: a fixed summation order
        int k[kCamsAtOnce];
        Pack<T, VEC> r[kCamsAtOnce];
#pragma unroll
        for (int n = 0; n < kCamsAtOnce; ++n) k[n] = pos[(long long)min(i0 + n, cams - 1) * Nq + q];
#pragma unroll
        for (int n = 0; n < kCamsAtOnce; ++n) {
#pragma unroll
          for (int c = 0; c < VEC; ++c) r[n].v[c] = 0;       // (adds nothing: the sum is no negative zero)
          if (i0 + n < cams && k[n] >= 0 && k[n] < max_len) r[n] = load_pack<T, VEC>(src + (((long long)j * cams + i0 + n) * max_len + k[n]) * E + e);
        }
#pragma unroll
        for (int n = 0; n < kCamsAtOnce; ++n)
#pragma unroll
          for (int c = 0; c < VEC; ++c) acc.v[c] += r[n].v[c];
      }
      if (scale != nullptr) {
        const T s = scale[(long long)j * Nq + q];
#pragma unroll
        for (int c = 0; c < VEC; ++c) acc.v[c] *= s;
      }
      store_pack<T, VEC>(dst + ((long long)j * Nq + q) * E + e, acc);
    }
  }
}

// The layer's gather in one launch: dst[j, i, k, :] = src[j, q, :] + plus[j, q, :] (`plus` may be null), zero in the padding, and
// ref_dst[j, i, k, :] = ref[i, j, q, :], `ref_pad` in the padding, q = index[i, k].  One thread per VEC elements of a row of dst, then one per
// VEC_REF of a row of ref_dst.  Bound by what is read and written; the queries alone are summed as they are read and the sum not written out and
// read again: 22500 queries of 256 and their positions, a fifth in each of six cameras, 14.5 us for 10.9 (sum), 10.5 and 2.7 (gathers); 40000 24.0
// for 18.1, 16.7 and 3.0 (a copy of the result 9 and 15).
template <typename T, int VEC, int VEC_REF>
__global__ __launch_bounds__(kRebatchBlock) void rebatch_queries_kernel(
    const T *__restrict__ src, const T *__restrict__ plus, const T *__restrict__ ref, const int *__restrict__ index, T *__restrict__ dst,
    T *__restrict__ ref_dst, int bs, int cams, int max_len, int Nq, int E, int R, T ref_pad, Pieces pieces, Pieces ref_pieces) {
  const long long queries = (long long)max_len * pieces.per, total = queries + (long long)max_len * ref_pieces.per;
  for (int ji = blockIdx.y; ji < bs * cams; ji += gridDim.y) {
    const int j = ji / cams, i = ji - j * cams;
    for (long long t = (long long)blockIdx.x * kRebatchBlock + threadIdx.x; t < total; t += (long long)gridDim.x * kRebatchBlock) {
      const bool is_ref = t >= queries;
      long long k;
      int piece;
      if (is_ref) ref_pieces.place(t - queries, k, piece);
      else pieces.place(t, k, piece);
      const int q = index[(long long)i * max_len + k];
      const bool there = q >= 0 && q < Nq;
      const long long to = (long long)ji * max_len + k;
      if (is_ref) {
        Pack<T, VEC_REF> r;
#pragma unroll
        for (int c = 0; c < VEC_REF; ++c) r.v[c] = ref_pad;
        if (there) r = load_pack<T, VEC_REF>(ref + (((long long)i * bs + j) * Nq + q) * R + piece * VEC_REF);
        store_pack<T, VEC_REF>(ref_dst + to * R + piece * VEC_REF, r);
      } else {
        const long long from = ((long long)j * Nq + q) * E + piece * VEC;
        Pack<T, VEC> r;
#pragma unroll
        for (int c = 0; c < VEC; ++c) r.v[c] = 0;
        if (there) {
          r = load_pack<T, VEC>(src + from);
          if (plus != nullptr) {                             // uniform
            const Pack<T, VEC> a = load_pack<T, VEC>(plus + from);
#pragma unroll
            for (int c = 0; c < VEC; ++c) r.v[c] += a.v[c];
          }
        }
        store_pack<T, VEC>(dst + to * E + piece * VEC, r);
      }
    }
  }
}

static unsigned rebatch_grid(long long threads) {
  long long blocks = (threads + kRebatchBlock - 1) / kRebatchBlock;
  if (blocks < 1) blocks = 1;
  if (blocks > (1 << 20)) blocks = 1 << 20;
  return (unsigned)blocks;
}
// `threads` for each of `rows` batch elements (and cameras)
static dim3 rebatch_grid(long long threads, long long rows) { return dim3(rebatch_grid(threads), (unsigned)(rows < 1024 ? rows : 1024)); }

template <typename T, int VEC>
static hipError_t gather_cfg(const void *src, long long cam_stride, long long batch_stride, const int *index, const void *scale, void *dst, int bs,
                             int cams, int max_len, int Nq, int E, double pad, hipStream_t stream) {
  const Pieces pieces(max_len, E / VEC);
  hipLaunchKernelGGL((rebatch_gather_kernel<T, VEC>), rebatch_grid((long long)max_len * pieces.per, (long long)bs * cams), dim3(kRebatchBlock), 0, stream,
                     (const T *)src, cam_stride, batch_stride, index, (const T *)scale, (T *)dst, bs, cams, max_len, Nq, E, (T)pad, pieces);
  return hipGetLastError();
}
template <typename T>
static hipError_t gather_typed(const void *src, long long cam_stride, long long batch_stride, const int *index,
                               const void *scale, void *dst, int bs, int cams, int max_len, int Nq, int E,
                               double pad, bool aligned, hipStream_t stream) {
  constexpr int W = 16 / (int)sizeof(T);
  return aligned && E % W == 0 && cam_stride % W == 0 && batch_stride % W == 0
             ? gather_cfg<T, W>(src, cam_stride, batch_stride, index, scale, dst, bs, cams, max_len, Nq, E, pad, stream)
             : gather_cfg<T, 1>(src, cam_stride, batch_stride, index, scale, dst, bs, cams, max_len, Nq, E, pad, stream);
}

template <typename T, int VEC>
static hipError_t combine_cfg(const void *src, const int *pos, const void *scale, void *dst, int bs, int cams, int max_len, int Nq, int E,
                              hipStream_t stream) {
  const Pieces pieces(Nq, E / VEC);
  hipLaunchKernelGGL((rebatch_combine_kernel<T, VEC>), rebatch_grid((long long)Nq * pieces.per, bs), dim3(kRebatchBlock), 0, stream, (const T *)src, pos,
                     (const T *)scale, (T *)dst, bs, cams, max_len, Nq, E, pieces);
  return hipGetLastError();
}
template <typename T>
static hipError_t combine_typed(const void *src, const int *pos, const void *scale, void *dst, int bs, int cams,
                                int max_len, int Nq, int E, bool aligned, hipStream_t stream) {
  constexpr int W = 16 / (int)sizeof(T);
  return aligned && E % W == 0 ? combine_cfg<T, W>(src, pos, scale, dst, bs, cams, max_len, Nq, E, stream)
                               : combine_cfg<T, 1>(src, pos, scale, dst, bs, cams, max_len, Nq, E, stream);
}

hipError_t launch_rebatch_gather(const void *src, long long cam_stride, long long batch_stride, const int *index,
                                 const void *scale, void *dst, int bs, int cams, int max_len, int Nq, int E,
                                 int dtype, double pad, hipStream_t stream) {
  const bool aligned = (((uintptr_t)src | (uintptr_t)dst) & 15) == 0;
  if (dtype == DFA3D_F32)
    return gather_typed<float>(src, cam_stride, batch_stride, index, scale, dst, bs, cams, max_len, Nq, E, pad, aligned, stream);
  if (dtype == DFA3D_F64)
    return gather_typed<double>(src, cam_stride, batch_stride, index, scale, dst, bs, cams, max_len, Nq, E, pad, aligned, stream);
  return hipErrorInvalidValue;
}

hipError_t launch_rebatch_combine(const void *src, const int *pos, const void *scale, void *dst, int bs, int cams,
                                  int max_len, int Nq, int E, int dtype, hipStream_t stream) {
  const bool aligned = (((uintptr_t)src | (uintptr_t)dst) & 15) == 0;
  if (dtype == DFA3D_F32) return combine_typed<float>(src, pos, scale, dst, bs, cams, max_len, Nq, E, aligned, stream);
  if (dtype == DFA3D_F64) return combine_typed<double>(src, pos, scale, dst, bs, cams, max_len, Nq, E, aligned, stream);
  return hipErrorInvalidValue;
}

template <typename T>
static hipError_t queries_typed(const RebatchQueries &a, hipStream_t stream) {
  constexpr int W = 16 / (int)sizeof(T);
  const bool wide = a.E % W == 0 && (((uintptr_t)a.src | (uintptr_t)a.plus | (uintptr_t)a.dst) & 15) == 0;
  const bool wide_ref = a.R % W == 0 && (((uintptr_t)a.ref | (uintptr_t)a.ref_dst) & 15) == 0;
  auto launch = [&](auto kernel, int vec, int vec_ref) {
    const Pieces pieces(a.max_len, a.E / vec), ref_pieces(a.max_len, a.R / vec_ref);
    hipLaunchKernelGGL(kernel, rebatch_grid((long long)a.max_len * (pieces.per + ref_pieces.per), (long long)a.bs * a.cams), dim3(kRebatchBlock), 0, stream,
                       (const T *)a.src, (const T *)a.plus, (const T *)a.ref, a.index, (T *)a.dst, (T *)a.ref_dst, a.bs, a.cams, a.max_len, a.Nq, a.E, a.R,
                       (T)a.ref_pad, pieces, ref_pieces);
    return hipGetLastError();
  };
  if (wide) return wide_ref ? launch(rebatch_queries_kernel<T, W, W>, W, W) : launch(rebatch_queries_kernel<T, W, 1>, W, 1);
  return wide_ref ? launch(rebatch_queries_kernel<T, 1, W>, 1, W) : launch(rebatch_queries_kernel<T, 1, 1>, 1, 1);
}
hipError_t launch_rebatch_queries(const RebatchQueries &a, int dtype, hipStream_t stream) {
  if (dtype == DFA3D_F32) return queries_typed<float>(a, stream);
  if (dtype == DFA3D_F64) return queries_typed<double>(a, stream);
  return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------------------
// From the mask of the anchors to index and pos.  All of it is a few hundred kilobytes: what it costs is launches and
// dependent passes, of which plain tensor operations take about twenty (a running sum along 40 000 queries alone
// 93 us: one workgroup per camera walks them); these are two launches (three for many queries), with the one copy of the counts to the host, which has to
// size the batch, before the last.
// ---------------------------------------------------------------------------------------
constexpr int kIndexBlock = 1024;
constexpr int kHitsBlock = 1024, kHitsCams = 1024;

// mask (cams, bs, Nq, Z) bytes: hit[i, q] = any anchor of query q of the first batch element falls into camera i;
// scale[j, q] = 1 / max(number of cameras with any anchor of query q of batch element j, 1)
__global__ __launch_bounds__(256) void camera_hits_kernel(const uint8_t *__restrict__ mask, uint8_t *__restrict__ hit,
                                                          float *__restrict__ scale, int cams, int bs, int Nq, int Z) {
  const long long n = (long long)bs * Nq;
  for (long long t = (long long)blockIdx.x * 256 + threadIdx.x; t < n; t += (long long)gridDim.x * 256) {
    int seen = 0;
    for (int i = 0; i < cams; ++i) {
      const uint8_t *p = mask + ((long long)i * n + t) * Z;
      int any = 0;
      if (Z == 4 && ((uintptr_t)mask & 3) == 0) {            // uniform
        any = *reinterpret_cast<const uint32_t *>(p) != 0;
      } else {
        for (int z = 0; z < Z; ++z) any |= p[z] != 0;
      }
      seen += any;
      if (t < Nq) hit[(long long)i * Nq + t] = (uint8_t)any;
    }
    scale[t] = 1.0f / (float)max(seen, 1);
  }
}

// The same, and how many queries of each camera each workgroup hit: counts (cams, gridDim.x), which the host adds up.  A pass over `hit` by one
// workgroup per camera and its launch are saved: 22500 queries, six cameras 4.3 us for 3.1 and 4.6, 40000 4.3 for 3.1 and 6.6; with lists, copy and
// host 36.7 for 40.1, 37.6 for 47.4.
__global__ __launch_bounds__(kHitsBlock) void camera_hits_counted_kernel(const uint8_t *__restrict__ mask, uint8_t *__restrict__ hit, float *__restrict__ scale,
                                                                         int *__restrict__ counts, int cams, int bs, int Nq, int Z) {
  __shared__ int s_count[kHitsCams];
  const long long n = (long long)bs * Nq, step = (long long)gridDim.x * kHitsBlock;
  for (int i = threadIdx.x; i < cams; i += kHitsBlock) s_count[i] = 0;
  __syncthreads();
  const bool words = Z == 4 && ((uintptr_t)mask & 3) == 0;   // uniform
  for (long long t = (long long)blockIdx.x * kHitsBlock + threadIdx.x; t - threadIdx.x < n; t += step) {       // uniform over the workgroup
    const bool there = t < n, first = t < Nq;
    int seen = 0;
    for (int i = 0; i < cams; ++i) {
      int any = 0;
      if (there) {
        const uint8_t *p = mask + ((long long)i * n + t) * Z;
        if (words) {
          any = *reinterpret_cast<const uint32_t *>(p) != 0;
        } else {
          for (int z = 0; z < Z; ++z) any |= p[z] != 0;
        }
      }
      seen += any;
      if (first) hit[(long long)i * Nq + t] = (uint8_t)any;
      const unsigned long long lanes = __ballot(first && any != 0);
      if (threadIdx.x % 64 == 0 && lanes != 0) atomicAdd(&s_count[i], __popcll(lanes));
    }
    if (there) scale[t] = 1.0f / (float)max(seen, 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < cams; i += kHitsBlock) counts[(size_t)i * gridDim.x + blockIdx.x] = s_count[i];
}

// the block's sum of a number per thread, in every thread
__device__ __forceinline__ int block_sum(int x, int *s_part) {
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = x;
  __syncthreads();
  int sum = 0;
  for (int w = 0; w < kIndexBlock / 64; ++w) sum += s_part[w];
  return sum;
}

__global__ __launch_bounds__(kIndexBlock) void camera_count_kernel(const uint8_t *__restrict__ hit, int *__restrict__ totals, int Nq) {
  __shared__ int s_part[kIndexBlock / 64];
  const uint8_t *mine = hit + (long long)blockIdx.x * Nq;
  int n = 0;
  for (int q = threadIdx.x; q < Nq; q += kIndexBlock) n += mine[q] != 0;
  n = block_sum(n, s_part);
  if (threadIdx.x == 0) totals[blockIdx.x] = n;
}

// This thread's share of the number of bytes among hit[0 .. n) that are not zero: whole words, and the bytes before and after them.  (Byte by
// byte, lists of six cameras, 22500 queries 5.6 us for 3.6, 40000 7.8 for 4.0, 160000 37 for 11.)
__device__ __forceinline__ int hits_before(const uint8_t *__restrict__ hit, int n) {
  const int head = min((int)(-(uintptr_t)hit & 3), n), words = (n - head) / 4, rest = n - 4 * words;      // rest: the bytes that are in no word
  const uint32_t *__restrict__ const word = reinterpret_cast<const uint32_t *>(hit + head);
  int sum = 0;
#pragma unroll 4
  for (int k = threadIdx.x; k < words; k += kIndexBlock) {
    const uint32_t w = word[k];
    sum += __popc((((w & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | w) & 0x80808080u);
  }
  const int t = threadIdx.x;
  if (t < rest) sum += hit[t < head ? t : t + 4 * words] != 0;
  return sum;
}

// A block ranks kIndexBlock queries of one camera; it counts the hits before them itself instead of waiting for the
// blocks that rank those.  pos is written whole, index from 0 to max_len: ranks, then the padding, in which a query that is no hit takes the place from
// the end that it has among those.
__global__ __launch_bounds__(kIndexBlock) void camera_index_kernel(const uint8_t *__restrict__ hit, int *__restrict__ index, int *__restrict__ pos,
                                                                   int Nq, int max_len) {
  __shared__ int s_part[kIndexBlock / 64];
  const int cam = blockIdx.y, first = blockIdx.x * kIndexBlock, q = first + threadIdx.x;
  const uint8_t *mine = hit + (long long)cam * Nq;
  int *index_row = index + (long long)cam * max_len;
  const int before = block_sum(hits_before(mine, first), s_part);
  const bool on = q < Nq && mine[q] != 0;
  const unsigned long long lanes = __ballot(on);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) s_part[wave] = __popcll(lanes);
  __syncthreads();
  int rank = before + __popcll(lanes & ((1ull << lane) - 1));
  for (int w = 0; w < wave; ++w) rank += s_part[w];
  if (q >= Nq) return;
  pos[(long long)cam * Nq + q] = on ? rank : -1;
  const int place = on ? rank : Nq - 1 - (q - rank);          // each of 0 to Nq - 1 once
  if (place < max_len) index_row[place] = on ? q : -1;
}

hipError_t launch_camera_hits(const uint8_t *mask, uint8_t *hit, float *scale, int cams, int bs, int Nq, int Z, hipStream_t stream) {
  hipLaunchKernelGGL(camera_hits_kernel, dim3(rebatch_grid((long long)bs * Nq)), dim3(256), 0, stream, mask, hit, scale, cams,
                     bs, Nq, Z);
  return hipGetLastError();
}
hipError_t launch_camera_count(const uint8_t *hit, int *totals, int cams, int Nq, hipStream_t stream) {
  hipLaunchKernelGGL(camera_count_kernel, dim3(cams), dim3(kIndexBlock), 0, stream, hit, totals, Nq);
  return hipGetLastError();
}
hipError_t launch_camera_hits_counted(const uint8_t *mask, uint8_t *hit, float *scale, int *counts, int parts, int cams, int bs, int Nq, int Z,
                                      hipStream_t stream) {
  if (cams > kHitsCams) return hipErrorInvalidValue;
  hipLaunchKernelGGL(camera_hits_counted_kernel, dim3(parts), dim3(kHitsBlock), 0, stream, mask, hit, scale, counts, cams, bs, Nq, Z);
  return hipGetLastError();
}
hipError_t launch_camera_index(const uint8_t *hit, int *index, int *pos, int cams, int Nq, int max_len, hipStream_t stream) {
  hipLaunchKernelGGL(camera_index_kernel, dim3((Nq + kIndexBlock - 1) / kIndexBlock, cams), dim3(kIndexBlock), 0, stream, hit,
                     index, pos, Nq, max_len);
  return hipGetLastError();
}

}  // namespace dfa3d
