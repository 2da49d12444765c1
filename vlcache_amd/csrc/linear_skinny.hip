// Linear layers of a few rows, for decode steps: out[m][n] = bf16(sum_k x[m][k] w[n][k] + bias[n]).
//
// In a decode step the projections of the decoder (models/qwen3.py: QKV, output, gate/up
// and down projections, and the LM head) multiply a handful of token rows by the whole
// weight matrix, so the work is streaming the weights from HBM once.
//
// A wave multiplies a 16-row tile of weights with 16 columns of x on the matrix pipe,
// v_mfma_f32_16x16x32_bf16, 64 bytes of a weight row per instruction and row.  Few rows of
// x leave most of the 16 columns empty, so the tile's 16 x 16 products are used as Z
// diagonal blocks of 16 / Z features x 16 / Z rows, each block summing its own 32 of 32 Z
// consecutive k: the tile then reads 64 Z contiguous bytes of each weight row (1 KB of two
// rows for Z = 8) and there are Z times as many tiles to spread over the chip, which is
// what shapes with few features lack.  TF tiles of features share each x operand, RB row
// blocks each weight operand, KS waves of a workgroup split K; the partial products meet
// in LDS in a fixed order, the bias is added in fp32 and the sum rounded to bf16 once.
// The cost beside the weights is x, which every tile reads again from L2: 16 / (Z TF)
// times fewer bytes per row for a larger tile.
//
// Measured, us, cold weights, calls of distinct weights in one graph, K x N; before is a
// tile of Z = 1, TF = 1 with K split four or eight ways:
//   rows                     3584 x 4608  3584^2  3584 x 37888  18944 x 3584  2048 x 22016  11008 x 2048
//   1, Z 8 TF 1 (before)                                                      15.7 (19.6)   10.3 (20.7)
//   4, Z 4 TF 2, 4 (before)  11.1 (12.9)  8.1 (8.5)  49.6 (54.3)  27.6 (28.6)  18.8 (20.5)   12.3 (20.7)
//   8, Z 2 (Z 1)             12.4 (12.9)  8.9 (9.0)  52.5 (62)    30.0 (33)    20.6 (23)     13.7 (18)
//   16, Z 1, or Z 2 RB 2     14.2         9.9        57.6 (75.8)  36.9         22.6 (25.3)   17.8
// and, one row, 2048 x 2560 4.1 (5.2), 2048^2 3.7 (5.0), 2048 x 151936 95.9 (104.8).
#include <type_traits>

#include "common.h"

namespace vlc {
namespace {

constexpr int kMaxRows = 16;       // vlc_linear_skinny
constexpr int kMaxSplitRows = 64;  // vlc_linear_split
constexpr int kPad = 17;           // floats per row of a 16 x 16 partial tile in LDS

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 ld16(const char* p) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4v*>(p));
}

struct Args {
  const char* x;
  int64_t x_stride_b;
  int rows, k_steps, tiles;
  const char* w;
  int64_t w_stride_b;
  const uint16_t* bias;
  uint16_t* out;
  int64_t out_stride;
  float* partial;  // gridDim.y > 1: [gridDim.y][rows][out_features]
  int out_features;
};

// SiLU-and-multiply as vlc_silu_mul computes it, of a gate and an up value rounded to bf16.
__device__ __forceinline__ float silu_mul(float gate, float up) {
  const float g = static_cast<float>(static_cast<__bf16>(gate)), u = static_cast<float>(static_cast<__bf16>(up));
  return g / (1.0f + expf(-g)) * u;
}

// U: k steps in flight; KS waves of the workgroup's W split K; gridDim.y splits it further.
// kSilu: the second half of a tile's TF feature groups are the up rows (out_features further) of the
// gate rows in the first half, and the output is silu(gate) * up: a decode step then has one launch
// less per layer (four layers of the 3B model, one row: 333.6 -> 326.5 us with the logits).
template <int U, int KS, int Z, int TF, int RB, int W, bool kSilu = false>
__global__ __launch_bounds__(64 * W) void linear_skinny_kernel(const Args p) {
  constexpr int kTiles = W / KS;  // tiles of a workgroup
  constexpr int F = 16 / Z;       // features, and rows, of a diagonal block
  constexpr int kStepB = 64 * Z;  // bytes of a row per k step
  constexpr int TO = kSilu ? TF / 2 : TF;  // feature groups of the output
  static_assert(!kSilu || TF % 2 == 0, "gate and up halves");
  __shared__ float part[W][TF][RB][16 * kPad];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int z = r / F, f = r % F;  // diagonal block; feature (A) or row of x (B) within it
  const int t = blockIdx.x * kTiles + wave / KS;
  const bool live = t < p.tiles;   // the last workgroup's tiles past N do no work
  const char* wp = p.w + (int64_t)((live ? t : 0) * (F * TO) + f) * p.w_stride_b + z * 64 + g * 16;
  const char* xp[RB];
  bool xr[RB];
#pragma unroll
  for (int q = 0; q < RB; ++q) {
    const int m = f + F * q;
    xr[q] = m < p.rows;  // other rows read as zero
    xp[q] = p.x + (int64_t)(xr[q] ? m : 0) * p.x_stride_b + z * 64 + g * 16;
  }
  const int splits = KS * (int)gridDim.y, split = (int)blockIdx.y * KS + wave % KS;
  int s = live ? (int)((int64_t)p.k_steps * split / splits) : 0;
  const int s1 = live ? (int)((int64_t)p.k_steps * (split + 1) / splits) : 0;
  const bf16x8 zero = __builtin_bit_cast(bf16x8, u32x4v{0u, 0u, 0u, 0u});
  f32x4 acc[TF][RB] = {};
  auto steps = [&](auto depth, int s0) __attribute__((always_inline)) {
    constexpr int D = decltype(depth)::value;
    bf16x8 a[D][TF], b[D][RB];
#pragma unroll
    for (int u = 0; u < D; ++u) {
#pragma unroll
      for (int j = 0; j < TF; ++j)
        a[u][j] = ld16(wp + (int64_t)(j % TO * F + (j >= TO ? p.out_features : 0)) * p.w_stride_b +
                       (int64_t)(s0 + u) * kStepB);
#pragma unroll
      for (int q = 0; q < RB; ++q) b[u][q] = xr[q] ? ld16(xp[q] + (int64_t)(s0 + u) * kStepB) : zero;
    }
#pragma unroll
    for (int u = 0; u < D; ++u)
#pragma unroll
      for (int j = 0; j < TF; ++j)
#pragma unroll
        for (int q = 0; q < RB; ++q)
          acc[j][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][j], b[u][q], acc[j][q], 0, 0, 0);
  };
  for (; s + U <= s1; s += U) steps(std::integral_constant<int, U>{}, s);
  for (; s < s1; ++s) steps(std::integral_constant<int, 1>{}, s);

  // lane holds C[row 4 g + e][column r] of its tiles
#pragma unroll
  for (int j = 0; j < TF; ++j)
#pragma unroll
    for (int q = 0; q < RB; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[wave][j][q][(4 * g + e) * kPad + r] = acc[j][q][e];
  __syncthreads();
  // output (tile, row block, row, feature) = sum over the waves of the tile and the diagonal blocks
  constexpr int kOut = kTiles * RB * F * TO * F;
  for (int i = threadIdx.x; i < kOut; i += 64 * W) {
    const int ff = i % F, j = i / F % TO, m = i / (F * TO) % F, q = i / (F * TO * F) % RB, tt = i / (F * TO * F * RB);
    const int row = m + F * q, tile = blockIdx.x * kTiles + tt;
    if (row >= p.rows || tile >= p.tiles) continue;
    auto sum = [&](int jj) __attribute__((always_inline)) {
      float y = 0.f;
#pragma unroll
      for (int v = 0; v < KS; ++v)
#pragma unroll
        for (int zz = 0; zz < Z; ++zz) y += part[tt * KS + v][jj][q][(zz * F + ff) * kPad + zz * F + m];
      return y;
    };
    const float y = sum(j);
    const int n = (tile * TO + j) * F + ff;
    if constexpr (kSilu)
      p.out[row * p.out_stride + n] = (uint16_t)f32_to_bf16_bits(silu_mul(y, sum(j + TO)));
    else if (gridDim.y == 1)
      p.out[row * p.out_stride + n] =
          (uint16_t)f32_to_bf16_bits(p.bias ? y + bf16_bits_to_f32(p.bias[n]) : y);
    else
      p.partial[((int64_t)blockIdx.y * p.rows + row) * p.out_features + n] = y;
  }
}

// Sum of the K splits in order, bias, one rounding: four features per lane.
__global__ __launch_bounds__(256) void linear_reduce_kernel(const float* __restrict__ partial, int splits, int rows,
                                                            int n, const uint16_t* __restrict__ bias,
                                                            uint16_t* __restrict__ out, int64_t out_stride) {
  const int i = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= rows * n) return;
  const int row = i / n, f = i - row * n;
  f32x4 y = *reinterpret_cast<const f32x4*>(partial + i);
  for (int s = 1; s < splits; ++s) y += *reinterpret_cast<const f32x4*>(partial + (int64_t)s * rows * n + i);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (bias) y[e] += bf16_bits_to_f32(bias[f + e]);
    out[row * out_stride + f + e] = (uint16_t)f32_to_bf16_bits(y[e]);
  }
}

template <int U, int KS, int Z, int TF, int RB, int W, bool kSilu = false>
void launch(Args a, int64_t in_features, int splits, hipStream_t st) {
  constexpr int kTiles = W / KS;
  a.tiles = a.out_features / (16 / Z * (kSilu ? TF / 2 : TF));
  a.k_steps = (int)(in_features / (32 * Z));
  hipLaunchKernelGGL((linear_skinny_kernel<U, KS, Z, TF, RB, W, kSilu>),
                     dim3((unsigned)((a.tiles + kTiles - 1) / kTiles), (unsigned)splits), dim3(64 * W), 0, st, a);
}

// vlc_linear_split's tile and K splits across workgroups: about one workgroup a CU.  Two or four feature
// groups a wave re-read x less, two diagonal blocks read 128 contiguous bytes of a weight row.  us, 18944 x 3584
// and 11008 x 2048, in brackets the library: 32 rows 38.2 (110), 18.2 (27), with tiles of 32 features and
// one diagonal block 43.0 and 20.1; 64 rows 54.8 (91), 25.2 (31), with tiles of 32 features 63.0 and 26.9.
int split_tile(int64_t rows, int64_t k, int64_t n) {
  if (rows > 16 && rows <= 32 && k % 64 == 0) return n % 64 == 0 && n >= 64 * 48 ? 64 : 32;
  return rows > 32 && n % 64 == 0 ? 64 : 32;
}
int num_splits(int64_t tiles) {
  const int64_t s = 256 / tiles;
  return (int)(s < 1 ? 1 : s > 8 ? 8 : s);
}

int check(const void* x, int64_t xs, int64_t rows, int64_t max_rows, int64_t k, const void* w, int64_t ws, int64_t n,
          const void* bias, const void* out, int64_t os) {
  if (rows < 0 || rows > max_rows || k <= 0 || n <= 0) return VLC_ERR_INVALID;
  if (k % 32 != 0 || n % 16 != 0) return VLC_ERR_UNSUPPORTED;
  if (xs < k || ws < k || os < n) return VLC_ERR_INVALID;
  if (rows == 0) return VLC_OK;
  if (!x || !w || !out) return VLC_ERR_INVALID;
  if (!aligned16(x) || !aligned16(w) || (xs % 8) || (ws % 8) || (reinterpret_cast<uintptr_t>(out) & 7) || (os % 4) ||
      (bias && (reinterpret_cast<uintptr_t>(bias) & 7)))
    return VLC_ERR_UNSUPPORTED;
  if (n / 16 >= ((int64_t)1 << 26)) return VLC_ERR_UNSUPPORTED;
  return VLC_OK;
}

}  // namespace
}  // namespace vlc

VLC_API int vlc_linear_skinny(const void* x, int64_t x_row_stride, int64_t rows, int64_t in_features,
                              const void* weight, int64_t w_row_stride, int64_t out_features, const void* bias,
                              void* out, int64_t out_row_stride, void* stream) {
  using namespace vlc;
  const int bad = check(x, x_row_stride, rows, kMaxRows, in_features, weight, w_row_stride, out_features, bias, out,
                        out_row_stride);
  if (bad != VLC_OK || rows == 0) return bad;
  const Args a = {static_cast<const char*>(x), x_row_stride * 2, (int)rows, 0, 0, static_cast<const char*>(weight),
                  w_row_stride * 2, static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(out), out_row_stride,
                  nullptr, (int)out_features};
  hipStream_t st = as_stream(stream);
  const int64_t k = in_features, n = out_features;
  // Z as large as the rows leave diagonal blocks free (and K divides); then as many tiles
  // per x operand as leave about 200 workgroups (the figures at the head of the file).
  if (rows <= 2 && k % 256 == 0)
    launch<2, 4, 8, 1, 1, 4>(a, k, 1, st);
  else if (rows <= 4 && k % 128 == 0) {
    if (n >= 16 * 200)
      launch<2, 8, 4, 4, 1, 8>(a, k, 1, st);
    else
      launch<2, 8, 4, 2, 1, 8>(a, k, 1, st);
  } else if (rows <= 8 && k % 64 == 0) {
    if (n >= 32 * 400 && n % 32 == 0)
      launch<2, 4, 2, 4, 1, 4>(a, k, 1, st);
    else if (n >= 16 * 200)
      launch<2, 8, 2, 2, 1, 8>(a, k, 1, st);
    else
      launch<2, 8, 2, 1, 1, 8>(a, k, 1, st);
  } else if (n >= 32 * 140 && n % 32 == 0 && k % 64 == 0) {
    launch<2, 4, 2, 4, 2, 4>(a, k, 1, st);
  } else {
    launch<2, 8, 1, 1, 1, 8>(a, k, 1, st);
  }
  return launch_status();
}

VLC_API int vlc_linear_skinny_silu(const void* x, int64_t x_row_stride, int64_t rows, int64_t in_features,
                                   const void* weight, int64_t w_row_stride, int64_t inter, void* out,
                                   int64_t out_row_stride, void* stream) {
  using namespace vlc;
  const int bad = check(x, x_row_stride, rows, kMaxRows, in_features, weight, w_row_stride, inter, nullptr, out,
                        out_row_stride);
  if (bad != VLC_OK || rows == 0) return bad;
  const Args a = {static_cast<const char*>(x), x_row_stride * 2, (int)rows, 0, 0, static_cast<const char*>(weight),
                  w_row_stride * 2, nullptr, static_cast<uint16_t*>(out), out_row_stride, nullptr, (int)inter};
  hipStream_t st = as_stream(stream);
  const int64_t k = in_features;
  // as vlc_linear_skinny chooses for many features, with an even number of feature groups
  if (rows <= 2 && k % 256 == 0)
    launch<2, 4, 8, 2, 1, 4, true>(a, k, 1, st);
  else if (rows <= 4 && k % 128 == 0)
    launch<2, 8, 4, 4, 1, 8, true>(a, k, 1, st);
  else if (rows <= 8 && k % 64 == 0)
    launch<2, 4, 2, 4, 1, 4, true>(a, k, 1, st);
  else if (k % 64 == 0)
    launch<2, 4, 2, 4, 2, 4, true>(a, k, 1, st);
  else
    launch<2, 8, 1, 2, 1, 8, true>(a, k, 1, st);
  return launch_status();
}

VLC_API int64_t vlc_linear_split_workspace(int64_t rows, int64_t in_features, int64_t out_features) {
  using namespace vlc;
  if (rows <= 0 || rows > kMaxSplitRows || out_features < 32 || out_features >= ((int64_t)1 << 24)) return 0;
  return num_splits(out_features / split_tile(rows, in_features, out_features)) * rows * out_features * 4;
}

VLC_API int vlc_linear_split(const void* x, int64_t x_row_stride, int64_t rows, int64_t in_features,
                             const void* weight, int64_t w_row_stride, int64_t out_features, const void* bias,
                             void* out, int64_t out_row_stride, void* workspace, int64_t workspace_bytes,
                             void* stream) {
  using namespace vlc;
  const int bad = check(x, x_row_stride, rows, kMaxSplitRows, in_features, weight, w_row_stride, out_features, bias,
                        out, out_row_stride);
  if (bad != VLC_OK || rows == 0) return bad;
  if (out_features % 32 || out_features >= ((int64_t)1 << 24)) return VLC_ERR_UNSUPPORTED;
  const int tile = split_tile(rows, in_features, out_features), splits = num_splits(out_features / tile);
  if (splits > 1 && (!workspace || !aligned16(workspace) ||
                     workspace_bytes < vlc_linear_split_workspace(rows, in_features, out_features)))
    return VLC_ERR_WORKSPACE;
  const Args a = {static_cast<const char*>(x), x_row_stride * 2, (int)rows, 0, 0, static_cast<const char*>(weight),
                  w_row_stride * 2, static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(out), out_row_stride,
                  static_cast<float*>(workspace), (int)out_features};
  hipStream_t st = as_stream(stream);
  if (rows <= 16)
    launch<2, 4, 1, 2, 1, 4>(a, in_features, splits, st);
  else if (rows <= 32 && in_features % 64 == 0) {
    if (tile == 64)
      launch<2, 4, 2, 8, 4, 4>(a, in_features, splits, st);
    else
      launch<1, 8, 2, 4, 4, 8>(a, in_features, splits, st);
  } else if (rows <= 32)
    launch<2, 4, 1, 2, 2, 4>(a, in_features, splits, st);
  else if (rows <= 48) {
    if (tile == 64)
      launch<2, 4, 1, 4, 3, 4>(a, in_features, splits, st);
    else
      launch<2, 4, 1, 2, 3, 4>(a, in_features, splits, st);
  } else {
    if (tile == 64)
      launch<2, 4, 1, 4, 4, 4>(a, in_features, splits, st);
    else
      launch<2, 4, 1, 2, 4, 4>(a, in_features, splits, st);
  }
  const int st1 = launch_status();
  if (st1 != VLC_OK || splits == 1) return st1;
  const int64_t lanes = rows * out_features / 4;
  hipLaunchKernelGGL(linear_reduce_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, st, a.partial, splits,
                     (int)rows, (int)out_features, a.bias, a.out, out_row_stride);
  return launch_status();
}
