// Sampling locations from what the layer predicts (BEVFormer_DFA3D/projects/mmdet3d_plugin/bevformer/modules/
// spatial_cross_attention.py:498-537): for row n (a query of a camera), head m, level l, point p
//
//   loc[n, m, l, p] = (u / W_l, v / H_l, d / D_l) + ref[n, p % Z]
//
// with (u, v) = uv[n, m, l, p] and d = dz[n, m, l, p]; and the gradients of uv and dz.  With them, where a head's points are a power of two up to a
// wavefront's lanes, the softmax over those of what the layer predicts as their weights, and its gradient.  Pure streaming, 24 bytes read or
// written per point and direction (with the weights 32, back 36), where tensor operations took three passes each way (softmax: one, back two).  A
// thread keeps its place in the row and walks down the block's rows, as many at once as 256 threads have room for, so that the place is decoded
// once and neighbouring lanes are neighbouring points; a head's points are neighbouring lanes.  Locations and softmax by themselves (with 16 rows a
// block, one at once) and in one kernel, us: 50000 rows of 8 heads, 32 points each 74 and 26, 77; back 55 and 46, 84; 27500 rows of 8 points each
// 12 and 5, 12; 9 and 10, 12; 3300 rows of 16 6 and 3, 5.6; 5 and 5, 4.9.
#include <algorithm>
#include <type_traits>

#include "../../include/dfa3d.h"
#include "dfa3d_device.h"
#include "dfa3d_launch.h"

namespace dfa3d {

constexpr int kLocThreads = 256;

struct LocPlace { float w, h, d; int z; };
__device__ __forceinline__ LocPlace loc_place(int r, const int64_t *__restrict__ shapes3, int L, int P, int Z) {
  const int l = (r / P) % L;
  return LocPlace{(float)shapes3[l * 3 + 1], (float)shapes3[l * 3], (float)shapes3[l * 3 + 2], (r % P) % Z};
}
// the threads' places: `at_once` rows side by side
struct LocRows {
  int at_once, row, first;
  bool on;
  __device__ __forceinline__ explicit LocRows(int MLP) {
    at_once = max(kLocThreads / MLP, 1);
    row = at_once > 1 ? (int)threadIdx.x / MLP : 0;
    first = (int)threadIdx.x - row * MLP;
    on = row < at_once;
  }
};
// over the lanes that differ in the bits below LANES (a power of two) of their number
template <int LANES> __device__ __forceinline__ float lanes_sum(float x) {
#pragma unroll
  for (int off = 1; off < LANES; off <<= 1) x += __shfl_xor(x, off, kWave);
  return x;
}
template <int LANES> __device__ __forceinline__ float lanes_max(float x) {
#pragma unroll
  for (int off = 1; off < LANES; off <<= 1) x = fmaxf(x, __shfl_xor(x, off, kWave));
  return x;
}

// LANES: the points of a head, or 0 without weights
template <int LANES>
__global__ __launch_bounds__(kLocThreads) void locations_kernel(const float *__restrict__ uv, const float *__restrict__ dz, const float *__restrict__ logits,
                                                                const float *__restrict__ ref, const int64_t *__restrict__ shapes3,
                                                                float *__restrict__ loc, float *__restrict__ attn, long long rows, int per_block, int MLP, int L, int P, int Z) {
  const long long n0 = (long long)blockIdx.x * per_block, n1 = min(n0 + per_block, rows);
  const LocRows at_row(MLP);
  if (!at_row.on) return;
  for (int r = at_row.first; r < MLP; r += kLocThreads) {
    const LocPlace at = loc_place(r, shapes3, L, P, Z);
#pragma unroll 4
    for (long long n = n0 + at_row.row; n < n1; n += at_row.at_once) {
      const long long i = n * MLP + r;
      const float *a = ref + (n * Z + at.z) * 3;
      const float u = uv[2 * i], v = uv[2 * i + 1], d = dz[i];
      float *o = loc + 3 * i;
      o[0] = u / at.w + a[0]; o[1] = v / at.h + a[1]; o[2] = d / at.d + a[2];
      if (LANES > 0) {
        const float x = logits[i], e = expf(x - lanes_max<LANES>(x));
        attn[i] = e / lanes_sum<LANES>(e);
      }
    }
  }
}

template <int LANES>
__global__ __launch_bounds__(kLocThreads) void locations_grad_kernel(const float *__restrict__ grad_loc, const float *__restrict__ grad_attn,
                                                                     const float *__restrict__ attn, const int64_t *__restrict__ shapes3,
                                                                     float *__restrict__ grad_uv, float *__restrict__ grad_dz,
                                                                     float *__restrict__ grad_logits, long long rows, int per_block, int MLP, int L, int P) {
  const long long n0 = (long long)blockIdx.x * per_block, n1 = min(n0 + per_block, rows);
  const LocRows at_row(MLP);
  if (!at_row.on) return;
  for (int r = at_row.first; r < MLP; r += kLocThreads) {
    const LocPlace at = loc_place(r, shapes3, L, P, 1);
#pragma unroll 4
    for (long long n = n0 + at_row.row; n < n1; n += at_row.at_once) {
      const long long i = n * MLP + r;
      const float *g = grad_loc + 3 * i;
      const float gx = g[0], gy = g[1], gz = g[2];
      grad_uv[2 * i] = gx / at.w; grad_uv[2 * i + 1] = gy / at.h;
      grad_dz[i] = gz / at.d;
      if (LANES > 0) {
        const float y = attn[i], weighted = grad_attn[i] * y;
        grad_logits[i] = weighted - y * lanes_sum<LANES>(weighted);
      }
    }
  }
}

__global__ __launch_bounds__(64) void level_table_kernel(const int64_t *__restrict__ shapes, int64_t *__restrict__ shapes3, int L, int D) {
  for (int i = threadIdx.x; i < 3 * L; i += 64) shapes3[i] = i % 3 == 2 ? D : shapes[i / 3 * 2 + i % 3];
}

hipError_t launch_level_table(const int64_t *shapes, int64_t *shapes3, int L, int D, hipStream_t stream) {
  hipLaunchKernelGGL(level_table_kernel, dim3(1), dim3(64), 0, stream, shapes, shapes3, L, D);
  return hipGetLastError();
}
// Rows of a block: four times those that it takes at once, fewer where that leaves fewer than 1024 blocks.  50000 rows of 256 points, 4, 8 and 16
// rows a block, there and back 77 and 84, 79 and 87, 84 and 93 us; 27500 rows of 64, 6 and 13 rows (four at once) 15 and 13, 12 and 12; 3300 rows
// of 128, 2, 3 and 16 rows 5.8 and 5.0, 5.6 and 4.9, 9.4 and 6.9.
static int rows_per_block(long long rows, int MLP) {
  const long long at_once = MLP < kLocThreads ? kLocThreads / MLP : 1, share = rows / 1024;
  return (int)std::max(at_once, std::min(share, 4 * at_once));
}
static dim3 loc_grid(long long rows, int per_block) { return dim3((unsigned)((rows + per_block - 1) / per_block)); }
template <typename Launch> static hipError_t with_lanes(int lanes, const Launch &launch) {
  switch (lanes) {
    case 0: launch(std::integral_constant<int, 0>()); break;
    case 1: launch(std::integral_constant<int, 1>()); break;
    case 2: launch(std::integral_constant<int, 2>()); break;
    case 4: launch(std::integral_constant<int, 4>()); break;
    case 8: launch(std::integral_constant<int, 8>()); break;
    case 16: launch(std::integral_constant<int, 16>()); break;
    case 32: launch(std::integral_constant<int, 32>()); break;
    case 64: launch(std::integral_constant<int, 64>()); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
// logits and attn, or neither
hipError_t launch_locations(const float *uv, const float *dz, const float *logits, const float *ref, const int64_t *shapes3, float *loc, float *attn,
                            long long rows, int M, int L, int P, int Z, hipStream_t stream) {
  const int per_block = rows_per_block(rows, M * L * P);
  return with_lanes(attn != nullptr ? L * P : 0, [&](auto lanes) {
    hipLaunchKernelGGL(locations_kernel<decltype(lanes)::value>, loc_grid(rows, per_block), dim3(kLocThreads), 0, stream, uv, dz, logits, ref, shapes3, loc, attn, rows,
                       per_block, M * L * P, L, P, Z);
  });
}
hipError_t launch_locations_grad(const float *grad_loc, const float *grad_attn, const float *attn, const int64_t *shapes3, float *grad_uv, float *grad_dz,
                                 float *grad_logits, long long rows, int M, int L, int P, hipStream_t stream) {
  const int per_block = rows_per_block(rows, M * L * P);
  return with_lanes(attn != nullptr ? L * P : 0, [&](auto lanes) {
    hipLaunchKernelGGL(locations_grad_kernel<decltype(lanes)::value>, loc_grid(rows, per_block), dim3(kLocThreads), 0, stream, grad_loc, grad_attn, attn, shapes3, grad_uv,
                       grad_dz, grad_logits, rows, per_block, M * L * P, L, P);
  });
}

}  // namespace dfa3d
