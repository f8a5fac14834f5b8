// The projections around the operator (the value, offset, weight and output layers of the cross-attention module) in float32, for gfx950:
//
//   y (N, O) = x (N, K) weight (O, K)^T + bias          grad_x (N, K) = grad_out (N, O) weight (O, K)
//   grad_weight (O, K) = grad_out (N, O)^T x (N, K)     grad_bias (O) = column sums of grad_out
//
// N is the number of rows (pixels of all cameras, or queries: 10^4 to 10^6), O and K are embedding widths (64 to 1024).  Float32
// matrix instructions have a sixteenth of bfloat16's rate, and bounded these products.  So each float32 is split into three bfloat16 whose
// sum it is, and a product is six of bfloat16 parts, summed in float32: those whose size is 2^-25 of the whole or less are left out.  What
// bounds it now is what goes on beside the matrix unit, which is busy for a third of the time: the splitting (one third as many
// vector cycles as matrix cycles), LDS, rows that come and go.
//
//   * A workgroup of four wavefronts forms a tile of the result, 16 contraction steps at a time: the next step's operands are split into
//     LDS and the one after is asked for while this one's parts are multiplied, with one barrier per step.  Steps of 32 with one buffer
//     and two barriers took as long or longer (184950 rows of 256 x 256, 64 x 128 tiles: 195 us for 184; weight gradient 197 for 193).
//   * 64 x 128 tiles: 128 x 256, 128 x 128, 64 x 128, 64 x 64 take 210, 199, 184, 206 us for 184950 rows of 256 x 256, 43, 31, 26, 27 for 22500, 35, 21,
//     13, 12 for 5520; smaller tiles have more workgroups per CU, which wait in turn.
//   * The result of a weight gradient is small and its contraction long: the rows are cut into parts, a workgroup forms one 128 x 128 tile of
//     one part's product, and a second kernel adds the parts up in a fixed order.  Workgroups of one part differ by multiples of the
//     number of parts (a multiple of 8), so they run on one XCD and share its L2.
//   * The gradient of rows that several layers share is formed in one launch; its sums are added up by the vector unit every 128 steps, as they
//     run over all layers: 58000 rows of 256 from 512, 256 and 256 columns 200 us for three products and 48 for their sums, 185 together.
//   * Rows beyond the end and columns beyond O or K read as zero (buffer range check).
//
// Library (forward and grad_x) or the float32 matrix instructions before (weight gradient), and now, us, between other kernels: 184950 rows of
// 256 x 256 229, 177 (forward), 220, 171 (grad_x), 227, 147 (weight gradient); 58000 of 256 x 256 80, 56; 22500 45, 26; 5520 20, 12; 6600 of 256 x
// 64 19, 9.  Relative error against float64 (2-norm), the same: forward 2.0e-7, 1.7e-7 (5520 to 10^6 rows); grad_x 2.9e-7, 2.4e-7; weight gradient
// 184950 rows 6.9e-7, 4.4e-7, 10^6 rows 1.6e-6, 9.6e-7, all positive 6.7e-8, 4.8e-8; grad_bias 2.1e-7, 2.1e-7.  Library's and these, forward and
// grad_x alike, random signs (all positive): sums of 256 2.9e-7, 2.4e-7 (2.2e-7, 1.8e-7), 512 4.1e-7, 3.4e-7 (3.1e-7, 2.4e-7), 1024 5.7e-7, 4.9e-7
// (4.3e-7, 2.9e-7), 2048 8.1e-7, 7.0e-7 (6.0e-7, 3.8e-7), 4096 1.2e-6, 1.0e-6 (8.5e-7, 5.3e-7).  Of few rows (linear_few_kernel): sums of 256
// 2.9e-7, 1.2e-7 (2.4e-7, 0.6e-7), of 512, 256 and 256 terms of three layers 3.5e-7, 1.3e-7 (2.0e-7, 0.4e-7).
#include <algorithm>

#include "../../include/dfa3d.h"
#include "dfa3d_binned.h"
#include "dfa3d_device.h"
#include "dfa3d_launch.h"

namespace dfa3d {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
constexpr int kStep = 16;              // contraction steps staged at once: of one matrix instruction

// x = p1 + p2 + p3, each rounded to nearest: 24 bits and more, so nothing of a float32 of 2^-108 or more is lost, and of a smaller one
// 2^-133 at most (odd_sums).  put(i, p): the numbers' parts i, two to a word, before the next ones are formed.  `most`: the largest size that came by.
template <int N, typename Put> __device__ __forceinline__ void split_parts(const float (&v)[N], float &most, const Put &put) {
  float rest[N];
#pragma unroll
  for (int j = 0; j < N; ++j) rest[j] = v[j];
#pragma unroll
  for (int j = 0; j < N; j += 2) asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most) : "v"(rest[j]), "v"(rest[j + 1]));
#pragma unroll
  for (int plane = 0; plane < 3; ++plane) {
    uint32_t p[N / 2];
#pragma unroll
    for (int j = 0; j < N / 2; ++j) {
      uint32_t two = pack_bf16x2(rest[2 * j], rest[2 * j + 1]);
      asm("" : "+v"(two));                                     // (or each half is rounded once more for its difference)
      p[j] = two;
      if (plane < 2) {
        rest[2 * j] -= __uint_as_float(two << 16);
        rest[2 * j + 1] -= __uint_as_float(two & 0xFFFF0000u);
      }
    }
    put(plane, p);
  }
}
// the six products of parts, smallest first: part of the one operand, part of the other
constexpr int kProducts[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};

// One operand of a product as its tile of R rows and kStep contraction steps comes through registers into LDS.  Element (row, k) lies at
// row * ld + k, or (ACROSS) at k * ld + row.  In LDS: three planes of bfloat16, each in two pieces of eight contraction steps, 16 bytes per
// row and piece; the 64 bytes between the pieces keep writes and reads off each other's banks.
template <int R, bool ACROSS> struct SplitOperand {
  static constexpr int kPiece = R * 16 + 64, kPlane = 2 * kPiece, kBytes = 3 * kPlane;
  static constexpr int kRun = ACROSS ? 8 : 4;                                  // contraction steps of a thread's unit
  static constexpr int kUnits = (R * kStep / kRun + 255) / 256;
  float v[kUnits][kRun];

  // r: begins at the tile's first row, or (ACROSS) at the first contraction step, and ends with the last valid one.  `row0` and `rows`: ACROSS,
  // the tile's first row and how many there are in all.  What lies beyond reads as zero.
  __device__ __forceinline__ void load(rsrc_t r, int ld, int row0, int rows, int k0, int depth) {
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      const int idx = (int)threadIdx.x + 256 * u;
      if constexpr (ACROSS) {
        const int row = row0 + idx % R, k = k0 + 8 * (idx / R);
        const uint32_t off = (row < rows && idx < 2 * R) ? (uint32_t)(k * ld + row) * 4 : kNoRow;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[u][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off + (uint32_t)(j * ld) * 4, 0, 0));
      } else {
        const int row = idx / 4, k = k0 + 4 * (idx % 4);
        const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, k < depth ? (uint32_t)(row * ld + k) * 4 : kNoRow, 0, 0);
        v[u][0] = __uint_as_float(t.x); v[u][1] = __uint_as_float(t.y);
        v[u][2] = __uint_as_float(t.z); v[u][3] = __uint_as_float(t.w);
      }
    }
  }

  __device__ __forceinline__ void to_lds(unsigned char *lds, float &most) const {
    typedef unsigned int words __attribute__((ext_vector_type(kRun / 2)));
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      const int idx = (int)threadIdx.x + 256 * u;
      if (2 * R % 256 != 0 && ACROSS && idx >= 2 * R) break;
      unsigned char *at = lds + (ACROSS ? idx / R * kPiece + idx % R * 16 : idx % 4 / 2 * kPiece + idx / 4 * 16 + idx % 2 * 8);
      split_parts(v[u], most, [&](int plane, const uint32_t (&p)[kRun / 2]) {
        words w;
#pragma unroll
        for (int j = 0; j < kRun / 2; ++j) w[j] = p[j];
        *reinterpret_cast<words *>(at + plane * kPlane) = w;
      });
    }
  }
  // this lane's part of a matrix instruction's operand
  static __device__ __forceinline__ bf16x8 part(const unsigned char *lds, int plane, int half, int row) {
    return *reinterpret_cast<const bf16x8 *>(lds + plane * kPlane + half * kPiece + row * 16);
  }
};

template <int MT, int NT> __device__ __forceinline__ void zero_sums(f32x16 (&x)[MT][NT]) {
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) x[i][j][r] = 0;
}

// acc += sum over depth contraction steps of A(m, k) B(n, k) for a TM x TN tile by four wavefronts, 2 x 2; `seen` is called with A's registers
// once per kStep steps.  FLUSH: an instruction cuts off what lies about 2^-24 below the largest of its terms instead of rounding it (16 products of
// 2^-27 on a sum of 1 leave 1, 16 of -2^-27 leave 1 - 2^-23; one of 3 2^-25 is rounded up), which a chain over thousands of rows of a weight
// gradient feels; its sums start from zero every FLUSH steps and the vector unit adds them up.  Without, up to 4096 terms: see above.  `most`: the
// largest size among the operands that this thread brought.
template <int TM, int TN, bool A_ACROSS, bool B_ACROSS, int FLUSH, typename Seen>
__device__ __forceinline__ void split_product(unsigned char *lds, rsrc_t a_r, int lda, int a_row0, int a_rows, rsrc_t b_r, int ldb, int b_row0,
                                              int b_rows, int depth, f32x16 (&acc)[TM / 64][TN / 64], float &most, const Seen &seen) {
  constexpr int MT = TM / 64, NT = TN / 64;
  using OpA = SplitOperand<TM, A_ACROSS>;
  using OpB = SplitOperand<TN, B_ACROSS>;
  constexpr int kBuffer = OpA::kBytes + OpB::kBytes;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int half = lane / 32, row_a = (wave & 1) * MT * 32 + lane % 32, row_b = (wave >> 1) * NT * 32 + lane % 32;
  f32x16 since[MT][NT];                                       // FLUSH: since the last time
  f32x16(&sum)[MT][NT] = *(FLUSH ? &since : &acc);
  if (FLUSH) zero_sums(since);
  OpA a;
  OpB b;
  a.load(a_r, lda, a_row0, a_rows, 0, depth);
  b.load(b_r, ldb, b_row0, b_rows, 0, depth);
  a.to_lds(lds, most);
  b.to_lds(lds + OpA::kBytes, most);
  seen(a);
  a.load(a_r, lda, a_row0, a_rows, kStep, depth);
  b.load(b_r, ldb, b_row0, b_rows, kStep, depth);
  for (int k0 = 0, at = 0; k0 < depth; k0 += kStep, at ^= kBuffer) {          // uniform
    lds_barrier();                                            // this step's parts are there, and nobody reads the last one's any more
    const unsigned char *const mine = lds + at;
    unsigned char *const next = lds + (at ^ kBuffer);
    bf16x8 pa[MT][3], pb[NT][3];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < MT; ++i) pa[i][p] = OpA::part(mine, p, half, row_a + 32 * i);
#pragma unroll
      for (int j = 0; j < NT; ++j) pb[j][p] = OpB::part(mine + OpA::kBytes, p, half, row_b + 32 * j);
    }
    a.to_lds(next, most);                                           // (beyond depth: zeros that nobody reads)
    b.to_lds(next + OpA::kBytes, most);
    seen(a);
    a.load(a_r, lda, a_row0, a_rows, k0 + 2 * kStep, depth);
    b.load(b_r, ldb, b_row0, b_rows, k0 + 2 * kStep, depth);
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pa[i][kProducts[t][0]], pb[j][kProducts[t][1]], sum[i][j], 0, 0, 0);
    if (FLUSH && (k0 + kStep) % (FLUSH ? FLUSH : 1) == 0) {   // uniform
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] += since[i][j][r];
      zero_sums(since);
    }
  }
  if (FLUSH) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] += since[i][j][r];
  }
}

// Whether the wavefront has a sum among its own that parts give no number for, or too coarse a one; it is then formed again without parts.
//   * A float32 infinity, or a number next to the largest, is no bfloat16 number, and an infinity times a lower part of zero is none either:
//     a sum that is no finite number.
//   * The lowest part of an operand below 2^-108 is denormal, and 2^-133 of it may be lost, times its partner.  Where all partners are 2^32 or
//     less, 4096 such products lose 2^-89: 2^-25 of a sum of 2^-64 or more.  So: a smaller sum than that (not zero: it may be 2^-89 in
//     truth), or a larger operand in the workgroup's tile (`large`).
template <int MT, int NT> __device__ __forceinline__ bool odd_sums(const f32x16 (&acc)[MT][NT], bool large) {
  uint32_t least = 0xFFFFFFFFu, most = 0;                     // of the sizes' bits, twice; least: without zeros, less one
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t twice = __float_as_uint(acc[i][j][r]) << 1;
        least = min(least, twice - 1);
        most = max(most, twice);
      }
  const bool odd = large || most >= 0xFF000000u || least < (__float_as_uint(0x1p-64f) << 1) - 1;
  return __builtin_amdgcn_ballot_w64(odd) != 0;
}

__device__ __forceinline__ bool odd_sum(float sum) {           // of one, but for `large`
  const uint32_t twice = __float_as_uint(sum) << 1;
  return twice >= 0xFF000000u || twice - 1 < (__float_as_uint(0x1p-64f) << 1) - 1;
}

// Whether a thread of the workgroup brought an operand beyond 2^32.  flag: zero since before the last barrier but this one.
__device__ __forceinline__ bool any_large(float most, int *flag) {
  if (!(most <= 0x1p32f)) *flag = 1;
  lds_barrier();
  return __builtin_amdgcn_readfirstlane(*flag) != 0;
}

// This lane's four of eight contraction steps from k0 on of one row, for float32 matrix instructions; arguments as of SplitOperand::load.
template <bool ACROSS> __device__ __forceinline__ void load_whole(rsrc_t r, int ld, int row0, int rows, int row, int k0, int depth, float (&v)[4]) {
  const int k = k0 + 4 * ((int)threadIdx.x % kWave / 32);
  if constexpr (ACROSS) {
    const uint32_t off = row0 + row < rows ? (uint32_t)(k * ld + row0 + row) * 4 : kNoRow;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off + (uint32_t)(j * ld) * 4, 0, 0));
  } else {
    const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, k < depth ? (uint32_t)(row * ld + k) * 4 : kNoRow, 0, 0);
    v[0] = __uint_as_float(t.x); v[1] = __uint_as_float(t.y);
    v[2] = __uint_as_float(t.z); v[3] = __uint_as_float(t.w);
  }
}

// acc += the wavefront's part of the tile by float32 matrix instructions, straight from memory: what split_product forms, for sums that
// parts give no number for; row_a, row_b: this lane's first rows within the tile.  Gradients of a loss that is no number are all of that kind, and
// cost a few times the usual, not a walk over the rows per element: weight gradient of 58000 rows of 256 x 256 56 us, all NaN 119 (by one lane per
// element 10000); grad_x 59, 124 (3280); with one NaN row in a thousand 125 (6400) and 70 (173).
template <int MT, int NT, bool A_ACROSS, bool B_ACROSS>
__device__ __forceinline__ void whole_product(rsrc_t a_r, int lda, int a_row0, int a_rows, rsrc_t b_r, int ldb, int b_row0, int b_rows, int depth,
                                              int row_a, int row_b, f32x16 (&acc)[MT][NT]) {
  for (int k0 = 0; k0 < depth; k0 += 8) {                     // uniform
    float a[MT][4], b[NT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i) load_whole<A_ACROSS>(a_r, lda, a_row0, a_rows, row_a + 32 * i, k0, depth, a[i]);
#pragma unroll
    for (int j = 0; j < NT; ++j) load_whole<B_ACROSS>(b_r, ldb, b_row0, b_rows, row_b + 32 * j, k0, depth, b[j]);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][k], b[j][k], acc[i][j], 0, 0, 0);
  }
}

// the same for the tiles of split_product
template <int TM, int TN, bool A_ACROSS, bool B_ACROSS>
__device__ __forceinline__ void whole_tile(rsrc_t a_r, int lda, int a_row0, int a_rows, rsrc_t b_r, int ldb, int b_row0, int b_rows, int depth,
                                           f32x16 (&acc)[TM / 64][TN / 64]) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  whole_product<TM / 64, TN / 64, A_ACROSS, B_ACROSS>(a_r, lda, a_row0, a_rows, b_r, ldb, b_row0, b_rows, depth,
                                                      (wave & 1) * (TM / 2) + lane % 32, (wave >> 1) * (TN / 2) + lane % 32, acc);
}

// c (TM x TN tile of `ms` x `ns` valid elements, row length ldc) = acc + bias, + addend (as c) where there is one, asked for
// 16 elements at a time (one by one, each between two stores, 2500 rows of 256 x 256 14.5 us; product 8.5, product and sum 12.3, so 9.6; 22500 of
// 128 x 128 17.4; 11.0, 19.3, 11.5; 40000 of 512 x 512 178; 134, 168, 143).
template <int TM, int TN>
__device__ __forceinline__ void store_product(const f32x16 (&acc)[TM / 64][TN / 64], float *__restrict__ c, int ldc, int ms, int ns,
                                              const float *__restrict__ bias, const float *__restrict__ addend = nullptr) {
  constexpr int MT = TM / 64, NT = TN / 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int first_m = (wave & 1) * MT * 32 + 4 * (lane / 32), first_n = (wave >> 1) * NT * 32 + lane % 32;
  const rsrc_t from = make_rsrc(addend, addend != nullptr ? ((size_t)(ms - 1) * ldc + ns) * 4 : 0);      // (none: zeros)
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = first_n + 32 * j;
    const float add = (bias != nullptr && n < ns) ? bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m0 = first_m + 32 * i;
      float sum[16], plus[16];
      if (addend != nullptr) {                               // uniform
#pragma unroll
        for (int r = 0; r < 16; ++r)
          plus[r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, n < ns ? (uint32_t)((m0 + 8 * (r / 4) + r % 4) * ldc + n) * 4 : kNoRow, 0, 0));
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[r] = acc[i][j][r] + add + plus[r];
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[r] = acc[i][j][r] + add;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + 8 * (r / 4) + r % 4;
        if (m < ms && n < ns) c[(size_t)m * ldc + n] = sum[r];
      }
    }
  }
}

// y (N, O) = x (N, K) w (O, K)^T + bias + addend.  TM rows of one tile of TN columns per workgroup; those of the same rows run on one XCD.
template <int TM, int TN>
__global__ __launch_bounds__(256, 3) void linear_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
                                                        const float *__restrict__ addend, float *__restrict__ y, long long N, int O, int K, int tiles) {
  __shared__ __align__(16) unsigned char lds[2 * (SplitOperand<TM, false>::kBytes + SplitOperand<TN, false>::kBytes)];
  __shared__ int large;
  const long long n0 = (blockIdx.x / (8 * tiles) * 8 + blockIdx.x % 8) * (long long)TM;
  if (n0 >= N) return;                                        // uniform
  const int o0 = blockIdx.x % (8 * tiles) / 8 * TN, ms = N - n0 < TM ? (int)(N - n0) : TM, ns = O - o0 < TN ? O - o0 : TN;
  const rsrc_t x_r = make_rsrc(x + n0 * K, (size_t)ms * K * 4), w_r = make_rsrc(w + (size_t)o0 * K, (size_t)ns * K * 4);
  f32x16 acc[TM / 64][TN / 64];
  zero_sums(acc);
  float most = 0;
  if (threadIdx.x == 0) large = 0;
  split_product<TM, TN, false, false, 0>(lds, x_r, K, 0, 0, w_r, K, 0, 0, K, acc, most, [](const auto &) {});
  if (odd_sums(acc, any_large(most, &large))) {                                        // uniform
    zero_sums(acc);
    whole_tile<TM, TN, false, false>(x_r, K, 0, 0, w_r, K, 0, 0, K, acc);
  }
  store_product<TM, TN>(acc, y + n0 * O + o0, O, ms, ns, bias != nullptr ? bias + o0 : nullptr,
                        addend != nullptr ? addend + n0 * O + o0 : nullptr);
}

// y (N, K) = sum of rows (N, width) weight (width, K) over the sets: the gradient of the rows that several layers share.  FLUSH: 0 for one set.
template <int TM, int TN, int FLUSH>
__global__ __launch_bounds__(256, 3) void linear_sum_kernel(LinearSets sets, float *__restrict__ y, long long N, int K, int tiles) {
  __shared__ __align__(16) unsigned char lds[2 * (SplitOperand<TM, false>::kBytes + SplitOperand<TN, true>::kBytes)];
  __shared__ int large;
  const long long n0 = (blockIdx.x / (8 * tiles) * 8 + blockIdx.x % 8) * (long long)TM;
  if (n0 >= N) return;                                        // uniform
  const int k0 = blockIdx.x % (8 * tiles) / 8 * TN, ms = N - n0 < TM ? (int)(N - n0) : TM;
  f32x16 acc[TM / 64][TN / 64];
  zero_sums(acc);
  float most = 0;
  if (threadIdx.x == 0) large = 0;
  auto rows = [&](const LinearSet &s) { return make_rsrc(s.rows + n0 * s.width, (size_t)ms * s.width * 4); };
  auto weight = [&](const LinearSet &s) { return make_rsrc(s.weight, (size_t)s.width * K * 4); };
  for (int i = 0; i < sets.n; ++i) {                          // uniform
    const LinearSet &s = sets.set[i];
    if (i > 0) lds_barrier();                                 // nobody reads the last set's parts any more
    split_product<TM, TN, false, true, FLUSH>(lds, rows(s), s.width, 0, 0, weight(s), K, k0, K, s.width, acc, most, [](const auto &) {});
  }
  if (odd_sums(acc, any_large(most, &large))) {              // uniform
    zero_sums(acc);
    for (int i = 0; i < sets.n; ++i) {
      const LinearSet &s = sets.set[i];
      whole_tile<TM, TN, false, true>(rows(s), s.width, 0, 0, weight(s), K, k0, K, s.width, acc);
    }
  }
  store_product<TM, TN>(acc, y + n0 * K + k0, K, ms, K - k0 < TN ? K - k0 : TN, nullptr);
}

// eight contraction steps of one row or column, as a matrix instruction takes them from a lane, and their parts
__device__ __forceinline__ void column_parts(const float (&v)[8], bf16x8 (&parts)[3], float &most) {
  split_parts(v, most, [&](int i, const uint32_t (&p)[4]) {
    const u32x4 words = {p[0], p[1], p[2], p[3]};
    parts[i] = __builtin_bit_cast(bf16x8, words);
  });
}
// Element (row, k) lies at row * ld + k, or (ACROSS) at k * ld + row; `r` begins with both and ends with the last valid one.
template <bool ACROSS> __device__ __forceinline__ void load_eight(rsrc_t r, int ld, int row, int rows, int k, int depth, float (&v)[8]) {
  if constexpr (ACROSS) {
    const uint32_t off = row < rows ? (uint32_t)(k * ld + row) * 4 : kNoRow;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off + (uint32_t)(j * ld) * 4, 0, 0));
  } else {
#pragma unroll
    for (int j = 0; j < 8; j += 4) {
      const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, k + j < depth ? (uint32_t)(row * ld + k + j) * 4 : kNoRow, 0, 0);
      v[j] = __uint_as_float(t.x); v[j + 1] = __uint_as_float(t.y); v[j + 2] = __uint_as_float(t.z); v[j + 3] = __uint_as_float(t.w);
    }
  }
}

// The same products and sums where the tiles of the two kernels above are few: y (N, cols) = sum over the sets of rows (N, width) weight (cols,
// width)^T, or (ACROSS) weight (width, cols), + bias + addend.  A workgroup forms 32 x 32, and its four wavefronts take every fourth 16 steps each,
// straight from memory into registers, four of their steps at a time: a chain a sixteenth as long as those kernels', on up to four times as many
// workgroups. Sums start from zero every four steps (split_product, FLUSH) and the vector unit adds them up; those of the wavefronts meet in LDS.
constexpr int kFewTile = 32, kFewSteps = 4;
template <bool ACROSS>
__global__ __launch_bounds__(256, 2) void linear_few_kernel(LinearSets sets, const float *__restrict__ bias, const float *__restrict__ addend,
                                                            float *__restrict__ y, long long N, int cols, int tiles) {
  __shared__ float s_sum[4][16][kWave];
  __shared__ int large, any_odd;
  const long long n0 = (blockIdx.x / (8 * tiles) * 8 + blockIdx.x % 8) * (long long)kFewTile;
  if (n0 >= N) return;                                        // uniform
  const int c0 = blockIdx.x % (8 * tiles) / 8 * kFewTile, ms = N - n0 < kFewTile ? (int)(N - n0) : kFewTile;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, half = lane / 32, at = lane % 32;
  if (threadIdx.x == 0) { large = 0; any_odd = 0; }
  lds_barrier();
  auto rows = [&](const LinearSet &s) { return make_rsrc(s.rows + n0 * s.width, (size_t)ms * s.width * 4); };
  auto weight = [&](const LinearSet &s) {
    return ACROSS ? make_rsrc(s.weight, (size_t)s.width * cols * 4)
                  : make_rsrc(s.weight + (size_t)c0 * s.width, (size_t)min(cols - c0, kFewTile) * s.width * 4);
  };
  f32x16 acc[1][1], since;
  zero_sums(acc);
  float most = 0;
  for (int i = 0; i < sets.n; ++i) {                          // uniform
    const LinearSet &s = sets.set[i];
    const rsrc_t a_r = rows(s), b_r = weight(s);
    for (int k0 = kStep * wave; k0 < s.width; k0 += 4 * kFewSteps * kStep) {         // uniform
      float a[kFewSteps][8], b[kFewSteps][8];
#pragma unroll
      for (int u = 0; u < kFewSteps; ++u) {
        const int k = k0 + 4 * u * kStep + 8 * half;
        load_eight<false>(a_r, s.width, at, kFewTile, k, s.width, a[u]);
        load_eight<ACROSS>(b_r, ACROSS ? cols : s.width, ACROSS ? c0 + at : at, ACROSS ? cols : kFewTile, k, s.width, b[u]);
      }
      __builtin_amdgcn_sched_barrier(0);                       // (all of them under way before the first is waited for)
#pragma unroll
      for (int r = 0; r < 16; ++r) since[r] = 0;
#pragma unroll
      for (int u = 0; u < kFewSteps; ++u) {
        bf16x8 pa[3], pb[3];
        column_parts(a[u], pa, most);
        column_parts(b[u], pb, most);
#pragma unroll
        for (int t = 0; t < 6; ++t) since = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pa[kProducts[t][0]], pb[kProducts[t][1]], since, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][0][r] += since[r];
    }
  }
  // this thread's four sums: of rows 8 * wave + 4 * half and the three below, column `at`
  float sum[4];
  auto meet = [&]() {
#pragma unroll
    for (int r = 0; r < 16; ++r) s_sum[wave][r][lane] = acc[0][0][r];
    lds_barrier();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = 4 * wave + r;
      sum[r] = (s_sum[0][e][lane] + s_sum[1][e][lane]) + (s_sum[2][e][lane] + s_sum[3][e][lane]);
    }
  };
  if (!(most <= 0x1p32f)) large = 1;
  meet();
  bool odd = large != 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) odd |= odd_sum(sum[r]);
  if (odd) any_odd = 1;
  lds_barrier();
  if (__builtin_amdgcn_readfirstlane(any_odd) != 0) {         // uniform over the workgroup
    zero_sums(acc);
    for (int i = 0; i < sets.n; ++i) {
      const LinearSet &s = sets.set[i];
      const rsrc_t a_r = rows(s), b_r = weight(s);
      for (int k0 = 8 * wave; k0 < s.width; k0 += 32) {
        float a[4], b[4];
        load_whole<false>(a_r, s.width, 0, 0, at, k0, s.width, a);
        load_whole<ACROSS>(b_r, ACROSS ? cols : s.width, ACROSS ? c0 : 0, cols, at, k0, s.width, b);
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[k], b[k], acc[0][0], 0, 0, 0);
      }
    }
    meet();
  }
  const int col = c0 + at, row = 8 * wave + 4 * half;
  if (col >= cols) return;
  const float add = bias != nullptr ? bias[col] : 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (row + r < ms) {
      const size_t to = (size_t)(n0 + row + r) * cols + col;
      y[to] = addend != nullptr ? sum[r] + add + addend[to] : sum[r] + add;
    }
}

// y (N, cols) = x (N, depth) times the weight of one layer, whose parts for 32 columns and all of the depth (up to KS * 16 steps) a wavefront keeps in
// registers: 192 of its 256 (the others are taken too; one or two are spilled, outside of the loop).  A workgroup (8 wavefronts, one per CU) splits
// its 256 columns once and walks through tiles of 32 rows; what is left of a tile is its rows: straight to LDS two tiles ahead (a thread's own 16
// bytes each, so no register holds them and no barrier is needed), split once, read by all eight.  Power bounds it: 32x32x16 products of random
// numbers alone run at 1.8 of 2.4 GHz, so every split, access to LDS and load that is left out counts, not only those that something waits for.  Same
// products and sums in the same order as by linear_kernel and linear_sum_kernel, to the bit but where odd sums are formed again (here for 32 rows and
// columns at a time, there for a wavefront's part of a tile).  With those, and with this one, us, new operands each time: 184950 rows of 256 x 256
// 200, 151 (x W^T), 178, 130 (g W); 49536 60, 44 and 58, 43; 40000 47, 33 and 45, 33; 22500 28, 22 and 27, 23; 58000 of 256 x 512 117, 92.
constexpr int kRowTile = 32, kRowThreads = 512, kRowCols = 256;
constexpr int kOddTiles = 256;         // a wavefront's tiles with odd sums, a bit each; of more tiles, several share one
template <int KS> struct RowTile {
  static constexpr int kPiece = kRowTile * 16 + 16, kPlane = 2 * KS * kPiece, kParts = 3 * kPlane;      // (pieces begin on other banks)
  static constexpr int kQuads = 4 * KS, kUnits = kRowTile * kQuads / kRowThreads, kRaw = kRowTile * kQuads * 16;
  static constexpr int kLds = 2 * kParts + kRaw;
  // unit u of the rows straight to this thread's place in LDS; beyond the depth or the last row: zeros
  static __device__ __forceinline__ void ask(int u, unsigned char *raw, rsrc_t r, int depth) {
    int idx = (int)threadIdx.x;
    asm volatile("" : "+v"(idx));                              // (not worth registers from tile to tile)
    idx += kRowThreads * u;
    const int row = idx / kQuads, k = 4 * (idx % kQuads);
    load_to_lds16(r, raw + (kRowThreads * u + (int)threadIdx.x / kWave * kWave) * 16, k < depth ? (uint32_t)(row * depth + k) * 4 : kNoRow);
  }
  static __device__ __forceinline__ void split(int u, const unsigned char *raw, unsigned char *parts, float &most) {
    const int idx = (int)threadIdx.x + kRowThreads * u, row = idx / kQuads, quad = idx % kQuads;
    const float4 t = *reinterpret_cast<const float4 *>(raw + idx * 16);
    const float v[4] = {t.x, t.y, t.z, t.w};
    split_parts(v, most, [&](int plane, const uint32_t (&p)[2]) {
      *reinterpret_cast<uint2 *>(parts + plane * kPlane + quad / 2 * kPiece + row * 16 + quad % 2 * 8) = make_uint2(p[0], p[1]);
    });
  }
  static __device__ __forceinline__ bf16x8 part(const unsigned char *parts, int plane, int step, int half, int row) {
    return *reinterpret_cast<const bf16x8 *>(parts + plane * kPlane + (2 * step + half) * kPiece + row * 16);
  }
};
// waits until at most N of the wavefront's loads and stores are under way: those before them have arrived
template <int N> __device__ __forceinline__ void wait_until_left() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// waits for the wavefront's accesses to LDS
__device__ __forceinline__ void wave_lds_read() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// The parts of a wavefront's 32 columns of a weight, eight contraction steps of one column to a lane and step.
template <int KS> using ColumnParts = bf16x8[KS][3];
// Element (column, k) lies at k * ld + column: 32 lanes take a whole line at a time.
template <int KS> __device__ __forceinline__ void load_columns_across(rsrc_t r, int ld, int col, int cols, ColumnParts<KS> &parts, float &most) {
  float v[KS][8];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const uint32_t off = col < cols ? (uint32_t)((16 * s + 8 * ((int)threadIdx.x % kWave / 32)) * ld + col) * 4 : kNoRow;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[s][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off + (uint32_t)(j * ld) * 4, 0, 0));
  }
  __builtin_amdgcn_sched_barrier(0);                           // (all of them under way before the first is waited for)
#pragma unroll
  for (int s = 0; s < KS; ++s) column_parts(v[s], parts[s], most);
}
// Element (column, k) lies at column * depth + k: a lane per column would take 64 pieces of 16 bytes with an instruction, which cost 7 us
// for 256 x 256.  So they come through LDS, whole lines of 32 steps of each column, three such rounds of 4 KB (`ring`: the wavefront's) under way.
constexpr int kRing = 3, kRound = 32 * 32 * 4;
template <int KS> __device__ __forceinline__ void load_columns(rsrc_t r, int col0, int cols, int depth, unsigned char *ring, ColumnParts<KS> &parts, float &most) {
  const int lane = threadIdx.x % kWave;
  constexpr int kRounds = KS / 2;
  auto ask = [&](int round) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {                              // eight columns each; a column's pieces in an order that depends on it
      const int c = 8 * i + lane / 8, k = 32 * round + 4 * (lane % 8 ^ c / 2 % 8);
      load_to_lds16(r, ring + round % kRing * kRound + i * 1024, col0 + c < cols && k < depth ? (uint32_t)((col0 + c) * depth + k) * 4 : kNoRow);
    }
  };
  auto wait = [&](int rounds_left) {                           // rounds asked for after the one that is waited for
    if (rounds_left >= 2) wait_until_left<8>();
    else if (rounds_left == 1) wait_until_left<4>();
    else wait_until_left<0>();
  };
#pragma unroll
  for (int round = 0; round < kRing; ++round) ask(round);
#pragma unroll
  for (int round = 0; round < kRounds; ++round) {
    wait(kRounds - 1 - round);
    float v[2][8];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int c = lane % 32, piece = 4 * (h / 2) + 2 * (lane / 32) + h % 2;
      const float4 t = *reinterpret_cast<const float4 *>(ring + round % kRing * kRound + c * 128 + 16 * (piece ^ c / 2 % 8));
      v[h / 2][4 * (h % 2)] = t.x; v[h / 2][4 * (h % 2) + 1] = t.y; v[h / 2][4 * (h % 2) + 2] = t.z; v[h / 2][4 * (h % 2) + 3] = t.w;
    }
    wave_lds_read();                                           // they are read: their place is free
    if (round + kRing < kRounds) ask(round + kRing);
    column_parts(v[0], parts[2 * round], most);
    column_parts(v[1], parts[2 * round + 1], most);
  }
}

// ADD: `addend` (N, cols) is added to the result: its elements are asked for when the tile's last product is under way (there are no registers to
// hold them before), and what their way takes per tile is less than a pass over the result: product, product and sum, and both in one, 22500 rows
// of 256 x 256 23.2, 37.6 and 29.6 us; 40000 34.2, 56.5, 45.7; 80000 67, 101, 82.
template <int KS, bool ACROSS, bool ADD>
__global__ __launch_bounds__(kRowThreads, 2) void linear_rows_kernel(const float *__restrict__ x, const float *__restrict__ weight,
                                                                     const float *__restrict__ bias, const float *__restrict__ addend,
                                                                     float *__restrict__ y, long long N, int cols, int depth) {
  using Tile = RowTile<KS>;
  constexpr int kStores = 16;
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ int s_large[3];                                   // an operand beyond 2^32 in this tile, the next, the one before
  __shared__ uint32_t s_odd[kRowThreads / kWave][kOddTiles / 32];
  unsigned char *const raw = lds + 2 * Tile::kParts;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, half = lane / 32;
  const int c0 = blockIdx.y * kRowCols, col = wave * 32 + lane % 32, ldw = ACROSS ? cols : depth;
  const rsrc_t w_r = ACROSS ? make_rsrc(weight + c0, ((size_t)depth * cols - c0) * 4) : make_rsrc(weight + (size_t)c0 * depth, (size_t)(cols - c0) * depth * 4);
  const int tiles = (int)((N + kRowTile - 1) / kRowTile), stride = gridDim.x;
  auto rows_of = [&](int t) {
    const long long n0 = (long long)t * kRowTile, left = N - n0;
    return make_rsrc(x + (left > 0 ? n0 * depth : 0), left > 0 ? (size_t)(left < kRowTile ? left : kRowTile) * depth * 4 : 0);
  };
  auto result_in = [&](const float *in, int t) {
    const long long n0 = (long long)t * kRowTile, left = N - n0;
    return make_rsrc(in + n0 * cols, (size_t)(left < kRowTile ? left : kRowTile) * cols * 4);
  };
  const uint32_t y_off = c0 + col < cols ? (uint32_t)(4 * half * cols + c0 + col) * 4 : kNoRow;
  const float add = bias != nullptr && c0 + col < cols ? bias[c0 + col] : 0.f;
  // always the same number of stores, as their number is part of what is waited for
  auto put = [&](f32x16 &acc, int t, uint32_t off) {
    const rsrc_t r = result_in(y, t);
    asm volatile("" : "+v"(off));
    if constexpr (ADD) {
      const rsrc_t from = result_in(addend, t);
      float plus[kStores];
      uint32_t at = off;
#pragma unroll
      for (int i = 0; i < kStores; ++i) {
        plus[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, at, 0, 0));
        at += (uint32_t)(i % 4 == 3 ? 5 : 1) * cols * 4;
      }
#pragma unroll
      for (int i = 0; i < kStores; ++i) acc[i] = acc[i] + add + plus[i];
    }
#pragma unroll
    for (int i = 0; i < kStores; ++i) {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ADD ? acc[i] : acc[i] + add), r, off, 0, 2);      // 2: non-temporal
      off += (uint32_t)(i % 4 == 3 ? 5 : 1) * cols * 4;
    }
  };

  int t = blockIdx.x;
#pragma unroll
  for (int u = 0; u < Tile::kUnits; ++u) Tile::ask(u, raw, rows_of(t), depth);
  if (threadIdx.x < 3) s_large[threadIdx.x] = 0;
  for (int i = lane; i < kOddTiles / 32; i += kWave) s_odd[wave][i] = 0;
  ColumnParts<KS> w;
  bool large_weight;
  {
    float most = 0;
    if constexpr (ACROSS) load_columns_across<KS>(w_r, ldw, col, cols - c0, w, most);
    else load_columns<KS>(w_r, wave * 32, cols - c0, depth, lds + wave * kRing * kRound, w, most);
    large_weight = __builtin_amdgcn_ballot_w64(!(most <= 0x1p32f)) != 0;
  }
  static_assert(kRowThreads / kWave * kRing * kRound <= 2 * Tile::kParts, "");
  lds_barrier();                                               // s_large is zero, and nobody uses a ring any more
  float most = 0;
  wait_until_left<0>();
#pragma unroll
  for (int u = 0; u < Tile::kUnits; ++u) Tile::split(u, raw, lds, most);
  if (!(most <= 0x1p32f)) s_large[0] = 1;
#pragma unroll
  for (int u = 0; u < Tile::kUnits; ++u) Tile::ask(u, raw, rows_of(t + stride), depth);

  bool any_odd = false;
  int i = 0, at = 0, now = 0;                                  // number of the tile; its parts; i % 3
  for (; t < tiles; t += stride, ++i, at ^= Tile::kParts) {
    lds_barrier();                                             // this tile's parts are there, and nobody reads the last one's any more
    const unsigned char *const mine = lds + at;
    unsigned char *const next = lds + (at ^ Tile::kParts);
    const int after = now == 2 ? 0 : now + 1;
    if (threadIdx.x == 0) s_large[after == 2 ? 0 : after + 1] = 0;
    const rsrc_t ahead = rows_of(t + 2 * stride);
    f32x16 acc[1][1];
    zero_sums(acc);
    most = 0;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      bf16x8 px[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) px[p] = Tile::part(mine, p, s, half, lane % 32);
      constexpr int kEvery = KS / Tile::kUnits;
      if (s % kEvery == kEvery - 1) {
        // the next tile's rows of this unit, asked for a tile ago: after them the other units' and the stores
        if (i == 0) wait_until_left<Tile::kUnits - 1>();       // uniform
        else wait_until_left<Tile::kUnits - 1 + kStores>();
        Tile::split(s / kEvery, raw, next, most);
        Tile::ask(s / kEvery, raw, ahead, depth);
      }
#pragma unroll
      for (int q = 0; q < 6; ++q) acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(px[kProducts[q][0]], w[s][kProducts[q][1]], acc[0][0], 0, 0, 0);
    }
    if (!(most <= 0x1p32f)) s_large[after] = 1;
    const bool odd = odd_sums(acc, large_weight || __builtin_amdgcn_readfirstlane(s_large[now]) != 0);
    if (odd) {                                                 // uniform over the wavefront
      any_odd = true;
      if (lane == 0) s_odd[wave][i % kOddTiles / 32] |= 1u << (i % 32);
    }
    put(acc[0][0], t, odd ? kNoRow : y_off);
    now = after;
  }
  wait_until_left<0>();                                        // nothing is on its way to LDS when the workgroup ends
  if (any_odd) {                                               // uniform over the wavefront
    wave_lds_handover();
    for (t = blockIdx.x, i = 0; t < tiles; t += stride, ++i) {
      if (!(__builtin_amdgcn_readfirstlane(s_odd[wave][i % kOddTiles / 32]) >> (i % 32) & 1)) continue;
      f32x16 acc[1][1];
      zero_sums(acc);
      whole_product<1, 1, false, ACROSS>(rows_of(t), depth, 0, 0, w_r, ldw, 0, cols - c0, depth, lane % 32, col, acc);
      put(acc[0][0], t, y_off);
    }
  }
}

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

// What the kernels are told of the layers: of layer i the workgroups from first[i] on in the first launch and from first_sum[i] on in the second.
// Each layer's parts and tiles are those that it would have alone, so its results are too, to the bit.
struct GradLayers {
  LinearGradSet set[DFA3D_MAX_LINEAR_SETS];
  LinearTiles tiles[DFA3D_MAX_LINEAR_SETS];
  float *partial[DFA3D_MAX_LINEAR_SETS];
  uint32_t first[DFA3D_MAX_LINEAR_SETS], first_sum[DFA3D_MAX_LINEAR_SETS];
  int n;
};
__device__ __forceinline__ int layer_of(const uint32_t (&first)[DFA3D_MAX_LINEAR_SETS], int n) {
  int i = 0;
  for (int k = 1; k < n; ++k) i += blockIdx.x >= first[k];    // uniform
  return i;
}

__global__ __launch_bounds__(256, 2) void linear_grad_part_kernel(const float *__restrict__ x, const GradLayers layers, long long N, int K) {
  using OpG = SplitOperand<128, true>;
  __shared__ __align__(16) unsigned char lds[4 * OpG::kBytes];
  __shared__ int large;
  const int layer = layer_of(layers.first, layers.n);
  const LinearTiles &t = layers.tiles[layer];
  const int O = layers.set[layer].width, parts = t.parts, rows = t.rows, o_tiles = t.o;
  const float *const g = layers.set[layer].rows;
  const bool want_bias = layers.set[layer].grad_bias != nullptr;
  const int block = blockIdx.x - layers.first[layer], part = block % parts, tile = block / parts;
  const int o0 = (tile % o_tiles) * 128, k0 = (tile / o_tiles) * 128;
  const long long n0 = (long long)part * rows;
  const int n_rows = n0 < N ? (int)(N - n0 < rows ? N - n0 : rows) : 0;
  const rsrc_t g_r = make_rsrc(g + (n_rows > 0 ? n0 * O : 0), (size_t)n_rows * O * 4);
  const rsrc_t x_r = make_rsrc(x + (n_rows > 0 ? n0 * K : 0), (size_t)n_rows * K * 4);
  f32x16 acc[2][2];
  zero_sums(acc);
  float most = 0;
  if (threadIdx.x == 0) large = 0;
  float bias_sum = 0;                                       // of this thread's column and every other eight rows
  split_product<128, 128, true, true, 64>(lds, g_r, O, o0, O, x_r, K, k0, K, n_rows, acc, most, [&](const OpG &a) {
    const float *v = a.v[0];                                // a tree per batch: a chain of rows would round more
    bias_sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  });
  float *const mine = layers.partial[layer] + (size_t)part * ((size_t)O * K + O);
  if (odd_sums(acc, any_large(most, &large))) {             // uniform
    zero_sums(acc);
    whole_tile<128, 128, true, true>(g_r, O, o0, O, x_r, K, k0, K, n_rows, acc);
  }
  store_product<128, 128>(acc, mine + (size_t)o0 * K + k0, K, O - o0, K - k0, nullptr);
  if (want_bias && k0 == 0) {                               // uniform
    float *s_bias = reinterpret_cast<float *>(lds);
    lds_barrier();
    s_bias[threadIdx.x] = bias_sum;
    lds_barrier();
    const int col = threadIdx.x;
    if (col < 128 && o0 + col < O) mine[(size_t)O * K + o0 + col] = s_bias[col] + s_bias[128 + col];
  }
}

// One result element per thread of a group of 64; the block's four groups take a quarter of the parts each.
__global__ __launch_bounds__(256) void linear_grad_sum_kernel(const GradLayers layers, int K) {
  __shared__ float s_sum[4][64];
  const int c = threadIdx.x % 64, q = threadIdx.x / 64;
  const int layer = layer_of(layers.first_sum, layers.n);
  const LinearGradSet &set = layers.set[layer];
  const float *__restrict__ const partial = layers.partial[layer];
  float *__restrict__ const grad_weight = set.grad_weight, *__restrict__ const grad_bias = set.grad_bias;
  const int parts = layers.tiles[layer].parts, weights = set.width * K, n = weights + set.width;
  const int i = (int)(blockIdx.x - layers.first_sum[layer]) * 64 + c;
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

// Workgroups of TM x TN tiles, rows in groups of eight (one per XCD), or 0 where they are too many for a launch; `tiles`: of one row of them.
template <int TM, int TN> static unsigned linear_blocks(long long N, int tiles) {
  const long long blocks = ((N + TM - 1) / TM + 7) / 8 * 8 * tiles;
  return blocks <= 0x7FFFFFFFLL ? (unsigned)blocks : 0u;
}
// 64 x 128 tiles where there are two of them per CU: 4096 rows of 256 x 256 (128) 14 us with them, 10 with 256 smaller ones; 22500 (704) 26, 27
static bool wide_tiles(long long N, int width) { return width > 64 && (N + 63) / 64 * ((width + 127) / 128) >= 512; }

template <int TM, int TN>
static hipError_t launch_linear_cfg(const float *x, const float *w, const float *bias, const float *addend, float *y, long long N, int O, int K, hipStream_t stream) {
  const int tiles = (O + TN - 1) / TN;
  const unsigned blocks = linear_blocks<TM, TN>(N, tiles);
  if (blocks == 0) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((linear_kernel<TM, TN>), dim3(blocks), dim3(256), 0, stream, x, w, bias, addend, y, N, O, K, tiles);
  return hipGetLastError();
}

// Where linear_rows_kernel takes a product.  A workgroup multiplies by 256 columns and 256 steps whether they are there or not and begins with 5 us of
// weights, more where they lie along the depth; the other kernels' tiles end where a multiple of 64 columns does.  So the share of the products that the
// others would form too, in sixteenths, has to be the larger the fewer row tiles a CU gets and the more blocks of columns there are.  Time over
// that of the others, 4928 to 185000 rows, depths 196 to 256, 130 to 1024 columns, lowest and highest where this kernel is taken and where not:
//   row tiles per CU        0.6 - 1                    1.5 - 2                    2 - 4                      4 - 8                      8 and more
//   256 columns or fewer    x W^T from 15, g W 12      from 14                    from 10                    all                        all
//     taken, not            0.77 - 1.01, 0.93 - 1.35   0.81 - 0.97, 0.89 - 1.19   0.83 - 1.02, 0.93 - 1.06   0.77 - 0.96                0.67 - 0.88
//   more                    none                       none                       512 from 14 (more: below)  from 12                    from 9
//     taken, not                                       0.95 - 1.54                0.87 - 1.05, 0.88 - 1.44   0.80 - 1.06, 0.89 - 1.23   0.72 - 0.93
// More than 512 columns gain from three tiles per CU on if they are whole blocks (25000 rows, 768 columns 0.88, 1024 0.96; 16500 rows 1.02, 1.08).
// In us, the others and this one: 4928 rows of 256 x 256 10.7, 10.8 (x W^T), 13.0, 11.1 (g W); 12500 17.8, 15.2 and 18.5, 15.2; 12500 of 258
// columns 22.5, 27.6 and 21.8, 29.5; 25000 of 320 38.7, 42.5; 58000 of 320 77.5, 78.5; 58000 of 512 108, 89; of 128 columns 27850 21.1, 25.1.
// (16-byte loads to LDS want their addresses whole.)
static bool rows_kernel_applies(const float *x, const float *weight, long long N, int cols, int depth, bool across) {
  if (cols <= 128 || depth <= 192 || depth > 256 || (depth & 3) != 0 || (((uintptr_t)x | (uintptr_t)weight) & 15) != 0) return false;
  const long long tiles = (N + kRowTile - 1) / kRowTile, cus = cu_count(), blocks = (cols + kRowCols - 1) / kRowCols;
  const long long sixteenth = blocks * kRowCols * 256 / 16, share = (cols + 63) / 64 * 64 * (long long)depth;
  if (tiles >= 8 * cus) return share >= 9 * sixteenth;
  if (tiles >= 4 * cus) return blocks == 1 || share >= 12 * sixteenth;
  if (tiles >= 2 * cus) return share >= (blocks == 1 ? 10 : blocks == 2 ? 14 : 16) * sixteenth && (blocks <= 2 || tiles >= 3 * cus);
  if (blocks > 1) return false;
  if (2 * tiles >= 3 * cus) return share >= 14 * sixteenth;
  return tiles <= cus && 5 * tiles >= 3 * cus && share >= (across ? 12 : 15) * sixteenth;
}
template <int KS, bool ACROSS, bool ADD>
static hipError_t launch_linear_rows(const float *x, const float *w, const float *bias, const float *addend, float *y, long long N, int cols, int depth,
                                     hipStream_t stream) {
  const auto kernel = linear_rows_kernel<KS, ACROSS, ADD>;
  if (const hipError_t e = allow_lds(reinterpret_cast<const void *>(kernel), RowTile<KS>::kLds); e != hipSuccess) return e;
  const long long tiles = (N + kRowTile - 1) / kRowTile;
  const int cus = cu_count();
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles < cus ? tiles : cus), (cols + kRowCols - 1) / kRowCols), dim3(kRowThreads), RowTile<KS>::kLds, stream,
                     x, w, bias, addend, y, N, cols, depth);
  return hipGetLastError();
}

// Where linear_few_kernel takes a product: few 64 x 64 tiles for the depth of the sums, as its own 32 x 32 read operands twice as often.  On the
// device alone (captured in a graph), the other kernels and this one, us:
//   x W^T, 256 columns of 256 terms   100 rows 8.0, 5.9   625 (40 tiles) 8.1, 6.2   1500 (96) 8.3, 8.1   2500 (160) 8.7, 10.3
//     64 columns                      6600 rows (104) 8.4, 8.2
//     128 columns of 128 terms        625 (20) 5.9, 5.5   1500 (48) 5.9, 5.5   2500 (80) 6.0, 6.8     256 of 64 terms 100 (8) 4.7, 5.0
//   sums of 512, 256 and 256 terms    16 rows 35.6, 9.1   1000 (64) 37.1, 12.0   4000 (252) 43.0, 27.8   5500 (344) 47.0, 36.8   8000 (500) 50.3, 52.2
//     of 256, 128 and 128             1000 20.5, 8.3   4000 (252) 22.7, 20.9   5500 (344) 25.7, 26.8
//     of 128, 64 and 64               2000 (128) 13.2, 12.1   4000 13.9, 18.8
//     of 64, 32 and 32                1000 (64) 9.0, 7.9   2000 (128) 9.2, 10.8
static bool few_rows(long long N, int cols, int depth, bool across) {
  const long long tiles = (N + 63) / 64 * ((cols + 63) / 64);
  return across ? tiles <= std::min(depth / 2, 384) : depth >= 128 && tiles <= std::min(depth * 3 / 8, 96);
}
template <bool ACROSS>
static hipError_t launch_linear_few(const LinearSets &sets, const float *bias, const float *addend, float *y, long long N, int cols, hipStream_t stream) {
  const int tiles = (cols + kFewTile - 1) / kFewTile;
  const unsigned blocks = linear_blocks<kFewTile, kFewTile>(N, tiles);
  if (blocks == 0) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(linear_few_kernel<ACROSS>, dim3(blocks), dim3(256), 0, stream, sets, bias, addend, y, N, cols, tiles);
  return hipGetLastError();
}

hipError_t launch_linear(const float *x, const float *w, const float *bias, const float *addend, float *y, long long N, int O, int K, hipStream_t stream) {
  if (few_rows(N, O, K, false)) {
    const LinearSets one = {{{w, x, K}}, 1};
    return launch_linear_few<false>(one, bias, addend, y, N, O, stream);
  }
  if (rows_kernel_applies(x, w, N, O, K, false))
    return addend != nullptr ? launch_linear_rows<16, false, true>(x, w, bias, addend, y, N, O, K, stream)
                             : launch_linear_rows<16, false, false>(x, w, bias, nullptr, y, N, O, K, stream);
  return wide_tiles(N, O) ? launch_linear_cfg<64, 128>(x, w, bias, addend, y, N, O, K, stream)
                          : launch_linear_cfg<64, 64>(x, w, bias, addend, y, N, O, K, stream);
}

template <int TM, int TN, int FLUSH> static hipError_t launch_linear_sum_cfg(const LinearSets &sets, float *y, long long N, int K, hipStream_t stream) {
  const int tiles = (K + TN - 1) / TN;
  const unsigned blocks = linear_blocks<TM, TN>(N, tiles);
  if (blocks == 0) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((linear_sum_kernel<TM, TN, FLUSH>), dim3(blocks), dim3(256), 0, stream, sets, y, N, K, tiles);
  return hipGetLastError();
}

hipError_t launch_linear_sum(const LinearSets &sets, float *y, long long N, int K, hipStream_t stream) {
  int depth = 0;
  for (int i = 0; i < sets.n; ++i) depth += sets.set[i].width;
  if (few_rows(N, K, depth, true)) return launch_linear_few<true>(sets, nullptr, nullptr, y, N, K, stream);
  const LinearSet &s = sets.set[0];
  if (sets.n == 1 && rows_kernel_applies(s.rows, s.weight, N, K, s.width, true)) return launch_linear_rows<16, true, false>(s.rows, s.weight, nullptr, nullptr, y, N, K, s.width, stream);
  const bool wide = wide_tiles(N, K);
  if (sets.n == 1) return wide ? launch_linear_sum_cfg<64, 128, 0>(sets, y, N, K, stream) : launch_linear_sum_cfg<64, 64, 0>(sets, y, N, K, stream);
  return wide ? launch_linear_sum_cfg<64, 128, 128>(sets, y, N, K, stream) : launch_linear_sum_cfg<64, 64, 128>(sets, y, N, K, stream);
}

size_t linear_grad_workspace_bytes(long long N, int O, int K) {
  return (size_t)linear_tiles(N, O, K).parts * ((size_t)O * K + O) * sizeof(float);
}

// Several layers in two launches, whose workgroups fill the device together where one layer has few parts: 512, 256 and 256 columns on rows of 256,
// three pairs of launches and these, 1000 rows 45 us, 21; 7700 78, 42; 58000 231, 208; 256, 128 and 128 columns 7700 rows 70, 29.
hipError_t launch_linear_grads(const float *x, const LinearGradSets &sets, float *workspace, long long N, int K, hipStream_t stream) {
  GradLayers layers{};
  layers.n = sets.n;
  long long blocks = 0, sum_blocks = 0;
  for (int i = 0; i < sets.n; ++i) {
    const LinearGradSet &s = layers.set[i] = sets.set[i];
    const LinearTiles &t = layers.tiles[i] = linear_tiles(N, s.width, K);
    layers.partial[i] = workspace;
    layers.first[i] = (uint32_t)blocks;
    layers.first_sum[i] = (uint32_t)sum_blocks;
    workspace += linear_grad_workspace_bytes(N, s.width, K) / sizeof(float);
    blocks += (long long)t.parts * t.o * t.k;
    sum_blocks += (s.width * K + s.width + 63) / 64;
    if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
  }
  hipLaunchKernelGGL(linear_grad_part_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, x, layers, N, K);
  hipLaunchKernelGGL(linear_grad_sum_kernel, dim3((unsigned)sum_blocks), dim3(256), 0, stream, layers, K);
  return hipGetLastError();
}

}  // namespace dfa3d
