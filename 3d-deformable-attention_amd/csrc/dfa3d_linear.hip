// Weight and bias gradients of the projections around the operator (the value, offset, weight and output layers of the
// cross-attention module) for gfx950:
//
//   grad_weight (O, K) = grad_out (N, O)^T  input (N, K)      grad_bias (O) = column sums of grad_out
//
// in float32.  N is the number of rows (pixels of all cameras, or queries: 10^4 to 10^6), O and K are embedding widths
// (64 to 1024): a contraction over a very long dimension with a small result.  What bounds it is the float32 matrix
// rate, and what it needs is parallelism that the 4 to 16 result tiles do not have: the rows are cut into parts, a
// workgroup forms one 128 x 128 tile of one part's product, and a second kernel adds the parts up in a fixed order.
//
//   * v_mfma_f32_32x32x2: a lane holds one element of row n of grad_out and one of input; both operands are read along
//     their rows, so nothing is transposed and nothing goes through LDS.  A lane reads two neighbouring columns (8 bytes)
//     and gives them to two tiles (even and odd columns), so a wavefront's load covers whole 256-byte pieces of two rows
//     and feeds a 64 x 64 tile with four matrix instructions per row pair.
//   * the loads of the next 16 rows are in flight while the current 16 are multiplied.
//   * workgroups of one part differ by multiples of the number of parts (a multiple of 8), so they run on one XCD and
//     share its L2.
//   * rows beyond a part's end and columns beyond O or K read as zero (buffer range check).
//
// Measured with the library's product and column sum for comparison, us: 184950 rows of 256 x 256 248 (98 TFLOP/s; float32
// matrix peak 157) against 608; 48000 of 256 x 512 123 against 562; 9000 of 256 x 64 23 against 77; 5000 of 128 x 96 21
// against 40.  The relative error of grad_weight against float64 is 3e-7 to 1e-6 where the library's is 1e-6 to 5e-6
// (random signs), that of grad_bias 1e-7 to 3e-7 where it is 1e-7 to 4e-7: the parts shorten the chain of additions.
#include "../../include/dfa3d.h"
#include "dfa3d_device.h"
#include "dfa3d_launch.h"

namespace dfa3d {

typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kPairs = 8;              // row pairs loaded at once

struct LinearTiles { int o, k, parts, rows; };      // result tiles along O and K; parts of the rows, rows of a part
static LinearTiles linear_tiles(long long N, int O, int K) {
  LinearTiles t;
  t.o = (O + 127) / 128; t.k = (K + 127) / 128;
  // two workgroups per CU over all tiles, at least 256 rows each
  long long parts = (512 + t.o * t.k - 1) / (t.o * t.k), most = (N + 255) / 256;
  parts = parts < most ? parts : most;
  parts = (parts + 7) / 8 * 8;
  const long long widest = O > K ? O : K, cap = (kMaxSliceBytes / 2) / (widest * 4);     // a part's rows stay below 2^30 bytes
  long long rows = (N + parts - 1) / parts;
  if (rows > cap) { rows = cap; parts = ((N + rows - 1) / rows + 7) / 8 * 8; }
  t.parts = (int)parts; t.rows = (int)rows;
  return t;
}

__global__ __launch_bounds__(256, 2) void linear_grad_part_kernel(
    const float *__restrict__ x, const float *__restrict__ g, float *__restrict__ partial, long long N, int O, int K,
    int parts, int rows, int o_tiles, int want_bias) {
  const int part = blockIdx.x % parts, tile = blockIdx.x / parts;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int half = lane / 32, col = lane % 32;
  const int o0 = (tile % o_tiles) * 128 + (wave & 1) * 64, k0 = (tile / o_tiles) * 128 + (wave >> 1) * 64;
  if (o0 >= O || k0 >= K) return;                          // uniform per wavefront; no barriers below
  const long long n0 = (long long)part * rows;
  const int n_rows = n0 < N ? (int)(N - n0 < rows ? N - n0 : rows) : 0;
  const rsrc_t g_r = make_rsrc(g + (n_rows > 0 ? n0 * O : 0), (size_t)n_rows * O * 4);
  const rsrc_t x_r = make_rsrc(x + (n_rows > 0 ? n0 * K : 0), (size_t)n_rows * K * 4);
  const int go = o0 + 2 * col, xk = k0 + 2 * col;
  uint32_t g_off = go < O ? (uint32_t)(half * O + go) * 4 : kNoRow, x_off = xk < K ? (uint32_t)(half * K + xk) * 4 : kNoRow;
  const uint32_t g_step = 2u * O * 4, x_step = 2u * K * 4;

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
  float bias0 = 0, bias1 = 0;
  u32x2 ga[kPairs], xa[kPairs], gb[kPairs], xb[kPairs];
  auto load = [&](u32x2 (&gv)[kPairs], u32x2 (&xv)[kPairs]) {
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
      gv[j] = __builtin_amdgcn_raw_buffer_load_b64(g_r, g_off + j * g_step, 0, 0);
      xv[j] = __builtin_amdgcn_raw_buffer_load_b64(x_r, x_off + j * x_step, 0, 0);
    }
    g_off += kPairs * g_step; x_off += kPairs * x_step;
  };
  auto multiply = [&](const u32x2 (&gv)[kPairs], const u32x2 (&xv)[kPairs]) {
    static_assert(kPairs == 8, "the sums below");
    auto sum8 = [&](auto of) { return ((of(0) + of(1)) + (of(2) + of(3))) + ((of(4) + of(5)) + (of(6) + of(7))); };
    bias0 += sum8([&](int j) { return __uint_as_float(gv[j].x); });      // a tree per batch: a chain of rows would round more
    bias1 += sum8([&](int j) { return __uint_as_float(gv[j].y); });
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
      const float a0 = __uint_as_float(gv[j].x), a1 = __uint_as_float(gv[j].y);
      const float b0 = __uint_as_float(xv[j].x), b1 = __uint_as_float(xv[j].y);
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc[1][1], 0, 0, 0);
    }
  };
  load(ga, xa);
  for (int n = 0; n < n_rows; n += 4 * kPairs) {            // uniform; what lies beyond the part's rows reads as zero
    load(gb, xb);
    multiply(ga, xa);
    load(ga, xa);
    multiply(gb, xb);
  }
  float *mine = partial + (size_t)part * ((size_t)O * K + O);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int o = o0 + 2 * (8 * (r / 4) + 4 * half + r % 4) + i, k = k0 + 2 * col;
      if (o < O && k < K) *reinterpret_cast<float2 *>(mine + (size_t)o * K + k) = make_float2(acc[i][0][r], acc[i][1][r]);
    }
  }
  if (want_bias && k0 == 0) {
    bias0 += __shfl_xor(bias0, 32, kWave);
    bias1 += __shfl_xor(bias1, 32, kWave);
    if (half == 0 && go < O) *reinterpret_cast<float2 *>(mine + (size_t)O * K + go) = make_float2(bias0, bias1);
  }
}

// One result element per thread of a group of 64; the block's four groups take a quarter of the parts each.
__global__ __launch_bounds__(256) void linear_grad_sum_kernel(const float *__restrict__ partial, float *__restrict__ grad_weight,
                                                              float *__restrict__ grad_bias, int parts, int weights, int n) {
  __shared__ float s_sum[4][64];
  const int c = threadIdx.x % 64, q = threadIdx.x / 64;
  const int i = blockIdx.x * 64 + c;
  const size_t stride = (size_t)n;
  float sum = 0;
  if (i < n && (i < weights || grad_bias != nullptr)) {
    const int per = parts / 4;                               // parts: a multiple of 8
    const float *p = partial + (size_t)q * per * stride + i;
#pragma unroll 8
    for (int k = 0; k < per; ++k) sum += p[k * stride];
  }
  s_sum[q][c] = sum;
  __syncthreads();
  if (q == 0 && i < n) {
    const float s = (s_sum[0][c] + s_sum[1][c]) + (s_sum[2][c] + s_sum[3][c]);
    if (i < weights) grad_weight[i] = s;
    else if (grad_bias != nullptr) grad_bias[i - weights] = s;
  }
}

size_t linear_grad_workspace_bytes(long long N, int O, int K) {
  return (size_t)linear_tiles(N, O, K).parts * ((size_t)O * K + O) * sizeof(float);
}

hipError_t launch_linear_grad(const float *x, const float *g, float *grad_weight, float *grad_bias, float *workspace,
                              long long N, int O, int K, hipStream_t stream) {
  const LinearTiles t = linear_tiles(N, O, K);
  const long long blocks = (long long)t.parts * t.o * t.k;
  if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(linear_grad_part_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, x, g, workspace, N, O, K, t.parts,
                     t.rows, t.o, grad_bias != nullptr ? 1 : 0);
  const int n = O * K + O;
  hipLaunchKernelGGL(linear_grad_sum_kernel, dim3((n + 63) / 64), dim3(256), 0, stream, workspace, grad_weight, grad_bias,
                     t.parts, O * K, n);
  return hipGetLastError();
}

}  // namespace dfa3d
