// The gate/up projection of an MLP with SiLU-and-multiply in its epilogue, for many rows:
// out = bf16(silu(bf16(x . wg^T + bg)) * bf16(x . wu^T + bu)).
//
// A workgroup of eight waves computes 256 tokens x (128 gate + 128 up features).  K runs in
// steps of 64: the step's 512 rows of 128 bytes (whole cache lines: rows of 64 bytes moved at
// 10 TB/s from L2 and gave 1257 TFLOP/s at 8192^3, against 1400) go global -> LDS by DMA into a
// ring of two stages, 16-byte chunks XOR-swizzled by the row so that the 16 rows of a
// ds_read_b128 fall into distinct banks.  Each wave multiplies its 128 x (32 + 32) part with
// v_mfma_f32_16x16x32_bf16, weights as the A operand, so that a lane ends with four
// consecutive gate features of a token and their up features.  The operands of one 32-wide
// half step are read while the other half's products run, so the one barrier of a step (tile
// t + 1 has landed, tile t is read: its stage is refilled with t + 2) finds every wave with
// products to issue.  Workgroups are handed out in ranges per XCD, in bands of eight token
// tiles, so that the tiles in flight on an XCD share rows in its L2.
//
// Bound by the matrix cores (the loop without the epilogue: 8192^3 at 1400 TFLOP/s, the library's
// best 1392); the epilogue's exponentials run when the products of a tile are done.  Measured, us,
// in brackets the library's product and the SiLU kernel, rows x K -> 2 * inter: 1247 x 2048 ->
// 22016 111 (114), 2500 217 (236), 10741 800 (902); 1247 x 3584 -> 37888 278 (396), 2500 556 (671).
// 32 x 32 MFMAs, four waves of 128 x 128 and 128 x 128 tiles were slower.
#include <type_traits>

#include "common.h"

namespace vlc {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kStepK = 64;
constexpr int kRowB = kStepK * 2;  // LDS bytes of a row
constexpr int kBand = 8;           // token tiles of a band

__device__ __forceinline__ uint32_t lds_u32(const void* p) { return (uint32_t)(uintptr_t)(const lds_void*)p; }

// Uniform base + per-lane offset -> LDS, 16 bytes a lane.  Inline assembly: the compiler would
// drain every LDS read wait for a DMA in flight.  The loads are counted in vmcnt; no register
// is written.
__device__ __forceinline__ void dma16(const void* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(voff), "s"(base) : "m0");
}
// All but the last N loads of this wave have landed, its LDS reads are done, then the barrier.
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  const bf16x2 v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, v);
}
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

constexpr int FM = 8, FN = 4, WM = 2, WN = 4;  // wave (wm, wn) owns 16 FM tokens x 16 FN features, half gate, half up
constexpr int W = WM * WN, BM = 16 * FM * WM, BN = 16 * FN * WN, ROWS = BM + BN, S = 2, STAGE = ROWS * kRowB;
constexpr int D = ROWS / 8 / W;  // DMA instructions (8 rows each) per wave and step
constexpr int kOutN = BN / 2, kOutF = FN / 2;

__global__ __launch_bounds__(64 * W, 2) void linear_silu_kernel(const Args p) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[S * STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;

  // the workgroup's tile: XCD x = id % 8 takes a contiguous range of tiles
  const int total = p.m_tiles * p.n_tiles, xcd = blockIdx.x & 7;
  const int id = xcd * (total / 8) + min(xcd, total % 8) + (int)(blockIdx.x >> 3);
  const int band = id / (kBand * p.n_tiles), in = id - band * kBand * p.n_tiles;
  const int band_m = min(kBand, p.m_tiles - band * kBand);
  const int n0 = in / band_m * kOutN, m0 = (band * kBand + in % band_m) * BM;

  // DMA sources: instruction j of the wave fills rows row0 .. row0 + 7 of a stage, lane i slot i % 8 of
  // row i / 8; rows past the operand's end read its last row (their results are not stored)
  const char* base[D];
  uint32_t voff[D];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const int row0 = (wave * D + j) * 8, row = row0 + (lane >> 3);
    const uint32_t chunk = (lane & 7) ^ ((row >> 1) & 7);
    if (row0 < BM) {
      base[j] = p.x + (int64_t)m0 * p.x_stride_b;
      voff[j] = (uint32_t)min(row, p.m - 1 - m0) * (uint32_t)p.x_stride_b + chunk * 16;
    } else {  // 16 FN rows per wave column: its gate features, then its up features (rows n .. 2 n - 1 of w)
      const int col = (row - BM) / (16 * FN), f = (row - BM) % (16 * FN);
      const bool up = (row0 - BM) % (16 * FN) >= 8 * FN;
      base[j] = p.w + ((int64_t)n0 + (up ? p.n : 0)) * p.w_stride_b;
      voff[j] = (uint32_t)min(col * 8 * FN + (up ? f - 8 * FN : f), p.n - 1 - n0) * (uint32_t)p.w_stride_b + chunk * 16;
    }
  }
  const uint32_t lds0 = lds_u32(lds) + wave * D * 1024;
  auto dma = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < D; ++j)
      dma16(base[j] + (int64_t)t * kRowB, voff[j], lds0 + j * 1024 + (uint32_t)(t % S) * STAGE);
  };

  // operand reads: row r of a 16-row fragment, chunk 4 half + g (the swizzle has the same value in every fragment)
  const int wm = wave / WN, wn = wave % WN;
  const uint32_t slot = (g ^ ((r >> 1) & 7)) * 16;
  const uint32_t xo = (wm * 16 * FM + r) * kRowB + slot, wo = (BM + wn * 16 * FN + r) * kRowB + slot;
  f32x4 acc[FN][FM] = {};
  bf16x8 xf[2][FM], wf[2][FN];
  auto read = [&](int t, auto half) __attribute__((always_inline)) {
    constexpr int h = decltype(half)::value;
    const uint8_t* s = lds + (t % S) * STAGE;
#pragma unroll
    for (int i = 0; i < FN; ++i) wf[h][i] = *reinterpret_cast<const bf16x8*>(s + (wo ^ (h * 64)) + i * 16 * kRowB);
#pragma unroll
    for (int i = 0; i < FM; ++i) xf[h][i] = *reinterpret_cast<const bf16x8*>(s + (xo ^ (h * 64)) + i * 16 * kRowB);
  };
  auto products = [&](auto half) __attribute__((always_inline)) {
    constexpr int h = decltype(half)::value;
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int i = 0; i < FN; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][i], xf[h][j], acc[i][j], 0, 0, 0);
  };
  // operand reads (0x100) spread over the products (0x008)
  auto interleave = [&]() __attribute__((always_inline)) {
    constexpr int R = FM + FN, per = FM * FN / R > 0 ? FM * FN / R : 1;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, per, 0);
    }
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  auto step = [&](auto refill, int t) __attribute__((always_inline)) {
    read(t, H1{});
    products(H0{});
    interleave();
    __builtin_amdgcn_sched_barrier(0);
    wait_barrier<(S - 2) * D>();
    if constexpr (decltype(refill)::value) dma(t + S);
    __builtin_amdgcn_sched_barrier(0);
    read(t + 1, H0{});
    products(H1{});
    interleave();
    __builtin_amdgcn_sched_barrier(0);
  };

  const int nk = p.k_tiles;
#pragma unroll
  for (int i = 0; i < S; ++i)
    if (i < nk) dma(i);
  if (nk >= S)
    wait_barrier<(S - 1) * D>();
  else
    wait_barrier<0>();
  read(0, H0{});
  int t = 0;
  for (; t + S < nk; ++t) step(std::true_type{}, t);
  for (; t + 1 < nk; ++t) step(std::false_type{}, t);
  read(t, H1{});
  products(H0{});
  interleave();
  products(H1{});

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
  hipLaunchKernelGGL(linear_silu_kernel, dim3((unsigned)(m_tiles * n_tiles)), dim3(64 * W), 0, as_stream(stream), a);
  return launch_status();
}
