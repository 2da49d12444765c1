// The gate/up projection of an MLP with SiLU-and-multiply in its epilogue, for many rows:
// out = bf16(silu(bf16(x . wg^T + bg)) * bf16(x . wu^T + bu)).
//
// A workgroup of eight waves computes 256 tokens x (128 gate + 128 up features) with the loop of
// gemm_tile.h: a wave's 64 features are 32 gate features and their up features.
//
// Bound by the matrix cores (the loop without the epilogue: 8192^3 at 1400 TFLOP/s, the library's
// best 1392); the epilogue's exponentials run when the products of a tile are done.  Measured, us,
// in brackets the library's product and the SiLU kernel, rows x K -> 2 * inter: 1247 x 2048 ->
// 22016 111 (114), 2500 217 (236), 10741 800 (902); 1247 x 3584 -> 37888 278 (396), 2500 556 (671).
// 32 x 32 MFMAs, four waves of 128 x 128 and 128 x 128 tiles were slower.
#include "gemm_tile.h"

namespace vlc {
namespace {

using namespace gemm;

__device__ __forceinline__ float round_bf16(float f) { return static_cast<float>(static_cast<__bf16>(f)); }

// g / (1 + exp(-g)) in fp32: exp2 of -g log2(e), the rounding error of that product carried
// into the result, so that 1 + exp(-g) has about 2 ulps; the reciprocal 1 ulp.  0 where exp(-g)
// overflows, NaN for NaN.
__device__ __forceinline__ float silu(float g) {
  constexpr float kL = 1.44269502f, kLLo = 1.92596303e-8f, kLn2 = 0.693147182f;
  const float c = __builtin_amdgcn_fmed3f(g, -88.72f, 88.72f);
  const float t = c * -kL;
  const float lo = __builtin_fmaf(c, -kLLo, __builtin_fmaf(c, -kL, -t));
  const float e0 = __builtin_amdgcn_exp2f(t);
  const float r = __builtin_amdgcn_rcpf(1.0f + __builtin_fmaf(e0, lo * kLn2, e0));
  return g * (g < -88.72f ? 0.0f : r);
}

struct Args {
  const char* x;
  int64_t x_stride_b;
  const char* w;
  int64_t w_stride_b;
  const uint16_t* bias;
  uint16_t* out;
  int64_t out_stride;
  int m, n, width, k_tiles;  // n: gate features; columns n .. width - 1 of out are zero
  int m_tiles, n_tiles;
};

typedef Tile<8, 4, 2, 4, 2> T;
constexpr int FM = T::FM, FN = T::FN, BM = T::BM, D = T::D;
constexpr int kOutN = T::BN / 2, kOutF = FN / 2;

__global__ __launch_bounds__(64 * T::W, 2) void linear_silu_kernel(const Args p) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[T::S * T::STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  int mt, nt;
  band_tile(xcd_range(blockIdx.x, p.m_tiles * p.n_tiles), p.m_tiles, p.n_tiles, mt, nt);
  const int n0 = nt * kOutN, m0 = mt * BM;

  // DMA sources: instruction j of the wave fills rows row0 .. row0 + 7 of a stage, lane i slot i % 8 of
  // row i / 8; rows past the operand's end read its last row (their results are not stored)
  const char* base[D];
  uint32_t voff[D];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const int row0 = T::dma_row0(wave, j), row = T::dma_row(wave, j, lane);
    const uint32_t chunk = T::dma_chunk(row, lane);
    if (row0 < BM) {
      base[j] = p.x + (int64_t)m0 * p.x_stride_b;
      voff[j] = (uint32_t)min(row, p.m - 1 - m0) * (uint32_t)p.x_stride_b + chunk;
    } else {  // 16 FN rows per wave column: its gate features, then its up features (rows n .. 2 n - 1 of w)
      const int col = (row - BM) / (16 * FN), f = (row - BM) % (16 * FN);
      const bool up = (row0 - BM) % (16 * FN) >= 8 * FN;
      base[j] = p.w + ((int64_t)n0 + (up ? p.n : 0)) * p.w_stride_b;
      voff[j] = (uint32_t)min(col * 8 * FN + (up ? f - 8 * FN : f), p.n - 1 - n0) * (uint32_t)p.w_stride_b + chunk;
    }
  }
  f32x4 acc[FN][FM] = {};
  T::run(lds, wave, lane, base, voff, p.k_tiles, acc);
  const int wm = wave / T::WN, wn = wave % T::WN;

  // lane holds gate features 16 i + 4 g .. + 3 of token 16 j + r in acc[i][j], their up features in
  // acc[i + kOutF][j]; both round to bf16 as the separate product's output does
#pragma unroll
  for (int i = 0; i < kOutF; ++i) {
    const int n = n0 + wn * 16 * kOutF + 16 * i + 4 * g;
    if (n >= p.width) continue;
    float bg[4] = {}, bu[4] = {};
    if (p.bias && n < p.n) {
      const uint2 a = *reinterpret_cast<const uint2*>(p.bias + n), b = *reinterpret_cast<const uint2*>(p.bias + p.n + n);
      bg[0] = bf16_bits_to_f32(a.x & 0xffffu), bg[1] = bf16_bits_to_f32(a.x >> 16);
      bg[2] = bf16_bits_to_f32(a.y & 0xffffu), bg[3] = bf16_bits_to_f32(a.y >> 16);
      bu[0] = bf16_bits_to_f32(b.x & 0xffffu), bu[1] = bf16_bits_to_f32(b.x >> 16);
      bu[2] = bf16_bits_to_f32(b.y & 0xffffu), bu[3] = bf16_bits_to_f32(b.y >> 16);
    }
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + wm * 16 * FM + 16 * j + r;
      if (m >= p.m) continue;
      uint2 o = {0u, 0u};
      if (n < p.n) {
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          y[e] = silu(round_bf16(acc[i][j][e] + bg[e])) * round_bf16(acc[i + kOutF][j][e] + bu[e]);
        o = uint2{pack2(y[0], y[1]), pack2(y[2], y[3])};
      }
      *reinterpret_cast<uint2*>(p.out + (int64_t)m * p.out_stride + n) = o;
    }
  }
}

}  // namespace
}  // namespace vlc

VLC_API int vlc_linear_silu(const void* x, int64_t x_row_stride, int64_t rows, int64_t in_features,
                            const void* weight, int64_t w_row_stride, int64_t inter, const void* bias, void* out,
                            int64_t out_row_stride, int64_t out_width, void* stream) {
  using namespace vlc;
  if (rows < 0 || in_features <= 0 || inter <= 0 || out_width < inter) return VLC_ERR_INVALID;
  if (in_features % kStepK || inter % 4 || out_width % 4) return VLC_ERR_UNSUPPORTED;
  if (x_row_stride < in_features || w_row_stride < in_features || out_row_stride < out_width) return VLC_ERR_INVALID;
  if (rows == 0) return VLC_OK;
  if (!x || !weight || !out) return VLC_ERR_INVALID;
  if (!aligned16(x) || !aligned16(weight) || (x_row_stride % 8) || (w_row_stride % 8) ||
      (reinterpret_cast<uintptr_t>(out) & 7) || (out_row_stride % 4) || (bias && (reinterpret_cast<uintptr_t>(bias) & 7)))
    return VLC_ERR_UNSUPPORTED;
  // a lane's offset within a tile's 256 rows is 32 bits wide
  if (x_row_stride >= (1 << 22) || w_row_stride >= (1 << 22) || rows >= (1 << 30) || out_width >= (1 << 29))
    return VLC_ERR_UNSUPPORTED;
  const int64_t m_tiles = (rows + BM - 1) / BM, n_tiles = (inter + kOutN - 1) / kOutN;
  // the last feature tile writes the padding too
  if (out_width > n_tiles * kOutN || m_tiles * n_tiles >= ((int64_t)1 << 27)) return VLC_ERR_UNSUPPORTED;
  const Args a = {static_cast<const char*>(x), x_row_stride * 2, static_cast<const char*>(weight), w_row_stride * 2,
                  static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(out), out_row_stride, (int)rows,
                  (int)inter, (int)out_width, (int)(in_features / kStepK), (int)m_tiles, (int)n_tiles};
  hipLaunchKernelGGL(linear_silu_kernel, dim3((unsigned)(m_tiles * n_tiles)), dim3(64 * T::W), 0, as_stream(stream), a);
  return launch_status();
}
