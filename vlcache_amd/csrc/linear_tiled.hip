// Linear layers of some hundred to a few thousand rows and a long K (the decoder's down projections in a
// prefill): out[m][n] = bf16(sum_k x[m][k] w[n][k] + bias[n]), K split across workgroups.
//
// Few features and rows give few tiles: 1247 x 11008 -> 2048 has 160 of 128 x 128 for 256 CUs, each walking
// 172 steps of K, and the library takes 90 us for 56 GFLOP.  The loop is gemm_tile.h's; tiles of 256 x 256 or
// 128 x 128 and 1 to 8 splits of K are chosen so that the launch fills the CUs (choose()).  Each split
// stores fp32 partial sums; a second kernel adds them in order, adds the bias and rounds once.
//
// Measured, us, cold weights, in brackets the library, rows x K -> N:
//   11008 -> 2048: 65 rows 21 (29), 256 27 (41), 640 55 (64), 1000 71 (77), 1247 72 (87), 2500 114 (124)
//   18944 -> 3584: 65 rows 34 (96), 256 65 (125), 640 100 (145), 1247 169 (227), 1600 245 (225), 2500 367 (525)
// On shapes with K at most 2 N the partial sums cost what the splits gain (3584 -> 3584, 1247 rows: 52 against 45).
#include "gemm_tile.h"

namespace vlc {
namespace {

using namespace gemm;

constexpr int kMaxSplits = 8;

struct Args {
  const char* x;
  int64_t x_stride_b;
  const char* w;
  int64_t w_stride_b;
  float* partial;  // [splits][m][n]
  int m, n, k_tiles, splits;
  int m_tiles, n_tiles;
};

template <typename T>
__global__ __launch_bounds__(64 * T::W, 2) void linear_tiled_kernel(const Args p) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[T::S * T::STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // the splits of a tile are neighbours: its rows are shared by none, its tile's neighbours by all
  const int id = xcd_range(blockIdx.x, p.m_tiles * p.n_tiles * p.splits);
  const int split = id % p.splits;
  int mt, nt;
  band_tile(id / p.splits, p.m_tiles, p.n_tiles, mt, nt);
  const int n0 = nt * T::BN, m0 = mt * T::BM;
  const int k0 = (int)((int64_t)p.k_tiles * split / p.splits), k1 = (int)((int64_t)p.k_tiles * (split + 1) / p.splits);

  // rows past the operand's end read its last row (their results are not stored)
  const char* base[T::D];
  uint32_t voff[T::D];
#pragma unroll
  for (int j = 0; j < T::D; ++j) {
    const int row = T::dma_row(wave, j, lane);
    const bool is_x = T::dma_row0(wave, j) < T::BM;
    const int64_t st = is_x ? p.x_stride_b : p.w_stride_b;
    base[j] = (is_x ? p.x + (int64_t)m0 * st : p.w + (int64_t)n0 * st) + (int64_t)k0 * kRowB;
    voff[j] = (uint32_t)(is_x ? min(row, p.m - 1 - m0) : min(row - T::BM, p.n - 1 - n0)) * (uint32_t)st +
              T::dma_chunk(row, lane);
  }
  f32x4 acc[T::FN][T::FM] = {};
  T::run(lds, wave, lane, base, voff, k1 - k0, acc);

  const int r = lane & 15, g = lane >> 4, wm = wave / T::WN, wn = wave % T::WN;
#pragma unroll
  for (int j = 0; j < T::FM; ++j) {
    const int m = m0 + wm * 16 * T::FM + 16 * j + r;
    if (m >= p.m) continue;
#pragma unroll
    for (int i = 0; i < T::FN; ++i) {
      const int n = n0 + wn * 16 * T::FN + 16 * i + 4 * g;
      if (n < p.n) *reinterpret_cast<f32x4*>(p.partial + ((int64_t)split * p.m + m) * p.n + n) = acc[i][j];
    }
  }
}

// Sum of the splits in order, bias, one rounding: four features per lane.
__global__ __launch_bounds__(256) void tiled_reduce_kernel(const float* __restrict__ partial, int splits, int64_t total,
                                                           int n, const uint16_t* __restrict__ bias,
                                                           uint16_t* __restrict__ out, int64_t out_stride) {
  const uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  f32x4 y = *reinterpret_cast<const f32x4*>(partial + i);
  for (int s = 1; s < splits; ++s) y += *reinterpret_cast<const f32x4*>(partial + s * total + i);
  const uint32_t row = i / (uint32_t)n, f = i - row * n;
  if (bias) {
    const uint2 b = *reinterpret_cast<const uint2*>(bias + f);
    y[0] += bf16_bits_to_f32(b.x & 0xffffu), y[1] += bf16_bits_to_f32(b.x >> 16);
    y[2] += bf16_bits_to_f32(b.y & 0xffffu), y[3] += bf16_bits_to_f32(b.y >> 16);
  }
  *reinterpret_cast<uint2*>(out + row * out_stride + f) = uint2{pack2(y[0], y[1]), pack2(y[2], y[3])};
}

// Tile kind and splits by the time they take: rounds of the launch over the CUs, steps of K per workgroup at the
// us measured per step (256 x 256: 1.8; 128 x 128: 0.66 alone on a CU, 1.1 with two), and the partial
// sums' way out and back at 5 TB/s: the fastest or next to it of the 22 combinations on most of those calls.
enum Kind { kBig, kDeep, kPair };
struct Choice {
  Kind kind;
  int splits;
};
Choice choose(int64_t rows, int64_t k, int64_t n) {
  Choice best = {kBig, 1};
  double best_us = 1e30;
  for (const Kind kind : {kBig, kDeep, kPair}) {
    const int64_t side = kind == kBig ? 256 : 128, tiles = ((rows + side - 1) / side) * ((n + side - 1) / side);
    const int64_t slots = kind == kPair ? 512 : 256;
    const double step_us = kind == kBig ? 1.8 : kind == kDeep ? 0.66 : 1.1;
    for (int splits = 1; splits <= kMaxSplits && splits * 4 <= k / kStepK; ++splits) {
      const double us = (double)((tiles * splits + slots - 1) / slots) * ((double)k / kStepK / splits) * step_us +
                        (double)splits * rows * n * 8 / 5e6;
      if (us < best_us) best_us = us, best = {kind, splits};
    }
  }
  return best;
}

template <typename T>
int launch_tiled(Args a, hipStream_t st) {
  a.m_tiles = (a.m + T::BM - 1) / T::BM;
  a.n_tiles = (a.n + T::BN - 1) / T::BN;
  hipLaunchKernelGGL(linear_tiled_kernel<T>, dim3((unsigned)(a.m_tiles * a.n_tiles * a.splits)), dim3(64 * T::W), 0, st, a);
  return launch_status();
}

bool sizes_ok(int64_t rows, int64_t k, int64_t n) {
  return rows > 0 && k > 0 && n > 0 && k % kStepK == 0 && n % 4 == 0 && rows < (1 << 24) && n < (1 << 24) &&
         rows * n < ((int64_t)1 << 31) && k < ((int64_t)1 << 30);
}

}  // namespace
}  // namespace vlc

VLC_API int64_t vlc_linear_tiled_workspace(int64_t rows, int64_t in_features, int64_t out_features) {
  using namespace vlc;
  if (!sizes_ok(rows, in_features, out_features)) return 0;
  return choose(rows, in_features, out_features).splits * rows * out_features * 4;
}

VLC_API int vlc_linear_tiled(const void* x, int64_t x_row_stride, int64_t rows, int64_t in_features,
                             const void* weight, int64_t w_row_stride, int64_t out_features, const void* bias,
                             void* out, int64_t out_row_stride, void* workspace, int64_t workspace_bytes,
                             void* stream) {
  using namespace vlc;
  if (rows < 0 || in_features <= 0 || out_features <= 0) return VLC_ERR_INVALID;
  if (x_row_stride < in_features || w_row_stride < in_features || out_row_stride < out_features)
    return VLC_ERR_INVALID;
  if (rows == 0) return VLC_OK;
  if (!x || !weight || !out) return VLC_ERR_INVALID;
  if (!sizes_ok(rows, in_features, out_features) || !aligned16(x) || !aligned16(weight) || (x_row_stride % 8) ||
      (w_row_stride % 8) || (reinterpret_cast<uintptr_t>(out) & 7) || (out_row_stride % 4) ||
      (bias && (reinterpret_cast<uintptr_t>(bias) & 7)))
    return VLC_ERR_UNSUPPORTED;
  // a lane's offset within a tile's 256 rows is 32 bits wide
  if (x_row_stride >= (1 << 22) || w_row_stride >= (1 << 22)) return VLC_ERR_UNSUPPORTED;
  const Choice c = choose(rows, in_features, out_features);
  if (!workspace || !aligned16(workspace) || workspace_bytes < c.splits * rows * out_features * 4)
    return VLC_ERR_WORKSPACE;
  const Args a = {static_cast<const char*>(x), x_row_stride * 2, static_cast<const char*>(weight), w_row_stride * 2,
                  static_cast<float*>(workspace), (int)rows, (int)out_features, (int)(in_features / kStepK), c.splits,
                  0, 0};
  hipStream_t st = as_stream(stream);
  const int bad = c.kind == kBig    ? launch_tiled<Tile<8, 4, 2, 4, 2>>(a, st)
                  : c.kind == kDeep ? launch_tiled<Tile<4, 2, 2, 4, 4>>(a, st)
                                    : launch_tiled<Tile<4, 2, 2, 4, 2>>(a, st);
  if (bad != VLC_OK) return bad;
  const int64_t total = rows * out_features;
  hipLaunchKernelGGL(tiled_reduce_kernel, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, st, a.partial,
                     c.splits, total, (int)out_features, static_cast<const uint16_t*>(bias),
                     static_cast<uint16_t*>(out), out_row_stride);
  return launch_status();
}
