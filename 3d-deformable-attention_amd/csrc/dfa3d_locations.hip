// Sampling locations from what the layer predicts (BEVFormer_DFA3D/projects/mmdet3d_plugin/bevformer/modules/
// spatial_cross_attention.py:498-537): for row n (a query of a camera), head m, level l, point p
//
//   loc[n, m, l, p] = (u / W_l, v / H_l, d / D_l) + ref[n, p % Z]
//
// with (u, v) = uv[n, m, l, p] and d = dz[n, m, l, p]; and the gradients of uv and dz.  Pure streaming, 24 bytes read or
// written per point and direction, where a concatenation, a division and an addition (backwards: a division and two strided
// copies) took three passes each way.  A thread keeps its place in the row and walks down the block's rows, so that the
// place is decoded once and neighbouring lanes are neighbouring points.  200 x 200 queries in six cameras, 256 points each:
// 65 us and 48 us back (about 4.5 TB/s); the tensor operations took about 0.25 and 0.2 ms.
#include "../../include/dfa3d.h"
#include "dfa3d_device.h"
#include "dfa3d_launch.h"

namespace dfa3d {

constexpr int kLocRows = 16;           // rows per block

struct LocPlace { float w, h, d; int z; };
__device__ __forceinline__ LocPlace loc_place(int r, const int64_t *__restrict__ shapes3, int L, int P, int Z) {
  const int l = (r / P) % L;
  return LocPlace{(float)shapes3[l * 3 + 1], (float)shapes3[l * 3], (float)shapes3[l * 3 + 2], (r % P) % Z};
}

__global__ __launch_bounds__(256) void locations_kernel(const float *__restrict__ uv, const float *__restrict__ dz,
                                                        const float *__restrict__ ref, const int64_t *__restrict__ shapes3,
                                                        float *__restrict__ loc, long long rows, int MLP, int L, int P, int Z) {
  const long long n0 = (long long)blockIdx.x * kLocRows, n1 = min(n0 + kLocRows, rows);
  for (int r = threadIdx.x; r < MLP; r += 256) {
    const LocPlace at = loc_place(r, shapes3, L, P, Z);
#pragma unroll 4
    for (long long n = n0; n < n1; ++n) {
      const long long i = n * MLP + r;
      const float *a = ref + (n * Z + at.z) * 3;
      const float u = uv[2 * i], v = uv[2 * i + 1], d = dz[i];
      float *o = loc + 3 * i;
      o[0] = u / at.w + a[0]; o[1] = v / at.h + a[1]; o[2] = d / at.d + a[2];
    }
  }
}

__global__ __launch_bounds__(256) void locations_grad_kernel(const float *__restrict__ grad_loc, const int64_t *__restrict__ shapes3,
                                                             float *__restrict__ grad_uv, float *__restrict__ grad_dz,
                                                             long long rows, int MLP, int L, int P) {
  const long long n0 = (long long)blockIdx.x * kLocRows, n1 = min(n0 + kLocRows, rows);
  for (int r = threadIdx.x; r < MLP; r += 256) {
    const LocPlace at = loc_place(r, shapes3, L, P, 1);
#pragma unroll 4
    for (long long n = n0; n < n1; ++n) {
      const long long i = n * MLP + r;
      const float *g = grad_loc + 3 * i;
      const float gx = g[0], gy = g[1], gz = g[2];
      grad_uv[2 * i] = gx / at.w; grad_uv[2 * i + 1] = gy / at.h;
      grad_dz[i] = gz / at.d;
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
hipError_t launch_locations(const float *uv, const float *dz, const float *ref, const int64_t *shapes3, float *loc, long long rows,
                            int M, int L, int P, int Z, hipStream_t stream) {
  hipLaunchKernelGGL(locations_kernel, dim3((unsigned)((rows + kLocRows - 1) / kLocRows)), dim3(256), 0, stream, uv, dz, ref,
                     shapes3, loc, rows, M * L * P, L, P, Z);
  return hipGetLastError();
}
hipError_t launch_locations_grad(const float *grad_loc, const int64_t *shapes3, float *grad_uv, float *grad_dz, long long rows,
                                 int M, int L, int P, hipStream_t stream) {
  hipLaunchKernelGGL(locations_grad_kernel, dim3((unsigned)((rows + kLocRows - 1) / kLocRows)), dim3(256), 0, stream, grad_loc,
                     shapes3, grad_uv, grad_dz, rows, M * L * P, L, P);
  return hipGetLastError();
}

}  // namespace dfa3d
