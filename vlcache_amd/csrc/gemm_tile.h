// The main loop of the tiled products (linear_silu.hip, linear_tiled.hip): a workgroup's BM tokens x BN
// features over a range of K.
//
// K runs in steps of 64: the step's BM + BN rows of 128 bytes (whole cache lines: rows of 64 bytes moved
// at 10 TB/s from L2 and gave 1257 TFLOP/s at 8192^3, against 1400) go global -> LDS by DMA into a ring
// of S stages, 16-byte chunks XOR-swizzled by the row so that the 16 rows of a ds_read_b128 fall into
// distinct banks.  Wave (wm, wn) of WM x WN multiplies its 16 FM tokens x 16 FN features with
// v_mfma_f32_16x16x32_bf16, weights as the A operand, so that a lane ends with four consecutive features
// of a token: acc[i][j][e] is feature 16 i + 4 (lane / 16) + e of token 16 j + lane % 16.  The operands of one 32-wide
// half step are read while the other half's products run, so the one barrier of a step (stage t + 1 has
// landed, stage t is read and is refilled with t + S) finds every wave with products to issue.
#pragma once

#include <type_traits>

#include "common.h"

namespace vlc {
namespace gemm {

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

// The tile of workgroup `block` of `total`: XCD block % 8 takes a contiguous range of tiles, so that the
// tiles in flight on an XCD share rows in its L2.
__device__ __forceinline__ int xcd_range(int block, int total) {
  const int xcd = block & 7;
  return xcd * (total / 8) + min(xcd, total % 8) + (block >> 3);
}
// (token tile, feature tile) of tile id: bands of kBand token tiles, tokens first.
__device__ __forceinline__ void band_tile(int id, int m_tiles, int n_tiles, int& mt, int& nt) {
  const int band = id / (kBand * n_tiles), in = id - band * kBand * n_tiles;
  const int band_m = min(kBand, m_tiles - band * kBand);
  nt = in / band_m;
  mt = band * kBand + in % band_m;
}

template <int FM_, int FN_, int WM_, int WN_, int S_>
struct Tile {
  static constexpr int FM = FM_, FN = FN_, WM = WM_, WN = WN_, S = S_;
  static constexpr int W = WM * WN, BM = 16 * FM * WM, BN = 16 * FN * WN, ROWS = BM + BN, STAGE = ROWS * kRowB;
  static constexpr int D = ROWS / 8 / W;  // DMA instructions (8 rows each) per wave and step
  static_assert(ROWS % (8 * W) == 0 && BM % 8 == 0 && S >= 2, "whole DMA instructions");

  // Row of a stage (tokens, then features) that DMA instruction j of a wave starts at, and a lane's row and the
  // byte of its chunk within a 128-byte step.
  static __device__ __forceinline__ int dma_row0(int wave, int j) { return (wave * D + j) * 8; }
  static __device__ __forceinline__ int dma_row(int wave, int j, int lane) { return dma_row0(wave, j) + (lane >> 3); }
  static __device__ __forceinline__ uint32_t dma_chunk(int row, int lane) {
    return (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16;
  }

  // acc += the products of nk steps; base[j] + voff[j] is the first step's source of DMA instruction j.
  static __device__ __forceinline__ void run(uint8_t* lds, int wave, int lane, const char* (&base)[D],
                                             const uint32_t (&voff)[D], int nk, f32x4 (&acc)[FN][FM]) {
    const int r = lane & 15, g = lane >> 4;
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
      wait_barrier<decltype(refill)::value ? (S - 2) * D : 0>();  // without refills fewer are behind stage t + 1
      if constexpr (decltype(refill)::value) dma(t + S);
      __builtin_amdgcn_sched_barrier(0);
      read(t + 1, H0{});
      products(H1{});
      interleave();
      __builtin_amdgcn_sched_barrier(0);
    };

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
  }
};

}  // namespace gemm
}  // namespace vlc
