// Window attention of the vision tower, from the QKV projection's rows to the output
// projection's input in one launch: the 2-D rotary of q and k, the attention within each
// window and the head layout of the result (models/qwen2_5_vl.py:176-212 of the reference,
// for the blocks that attend within windows of at most 64 patches).
//
// What bounds it: memory.  A 4K image's block reads 324 MB of q, k, v and writes 108 MB;
// its 1.4e10 multiply-adds are nothing beside that.  As three passes (rotary into padded
// heads, attention of padded heads, unpadding copy) it moved 842 + 1037 + 280 MB.
//
// Split: a window of at most 64 patches is one 64 x 64 score tile, so a wave owns one
// (window, head) and the four waves of a workgroup take four neighbouring heads (640
// contiguous bytes of each token row).  Waves share nothing and never wait for each other.
//
// A lane's share of a q or k row is what the rotation pairs up: half-wave h holds dims
// [20h, 20h + 20) and [40 + 20h, 60 + 20h) of its row, whose angles all belong to one
// axis (h = 0 rows, h = 1 columns).  The rotated 40 values are the lane's five operands of
// v_mfma_f32_32x32x16_bf16: the products sum over dims, so q and k may hold them in any
// common order.  S^T = K Q^T leaves a lane one query column and 16 keys of each 32-key
// block; the probabilities are then the B operand of O^T += V^T P^T, with V read
// transposed from LDS (ds_read_b64_tr_b16).
//
// Measured, two window blocks of a 4K image (42196 patches, 16 heads): 4908 us for the tower
// against 5474 us with the three passes (rotary into padded heads 160 us, attention of padded
// heads 173 us, unpadding copy 46 us a block); eight blocks of a 64 x 64 image 2315 against 2524.
// The kernel itself takes 102 us for the 432 MB (4.25 TB/s).  Larger windows are rotated in place
// (vlc_vision_rope) and attend through vlc_vision_attn.
#include "common.h"

namespace vlc {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kHd = 80;                // head dim
constexpr int kMaxWin = 64;            // patches of a window
constexpr int kQuarter = kHd / 4;      // angles per axis
constexpr int kRowChunks = kHd / 8;    // 16-byte chunks of a head row
constexpr int kVRow = 192;             // LDS bytes of a V row: 4 rows x 64 bytes of a half-wave's
                                       // transpose read fall into distinct banks
constexpr int kORow = 168;             // LDS bytes of an output row while it is transposed: 42 words,
                                       // so 32 rows' 8-byte writes fall into distinct banks

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4a8 __attribute__((ext_vector_type(4), aligned(8)));  // head rows start at 8-byte steps

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  const bf16x2 v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float lo16(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi16(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// 40 bytes (20 bf16) from an 8-byte aligned address.
__device__ __forceinline__ void ld40(const char* p, uint32_t (&w)[10]) {
  const u32x4a8 a = *reinterpret_cast<const u32x4a8*>(p), b = *reinterpret_cast<const u32x4a8*>(p + 16);
  const u32x2v c = *reinterpret_cast<const u32x2v*>(p + 32);
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = a[i], w[4 + i] = b[i];
  w[8] = c[0], w[9] = c[1];
}

// max over lanes l and l ^ 32 (the swap builtin's two results are folded into one by the
// compiler, hence the assembly; the s_nop covers the VALU-write hazard it does not track).
__device__ __forceinline__ float half_wave_max(float x) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return fmaxf(a, b);
}

// One head row's share of a lane: the 20 low and 20 high dims of its rotation pairs, each
// product and the sum rounded to bf16 as the published model's bf16 tensor arithmetic does.
struct Row {
  uint32_t lo[10], hi[10];
};
__device__ __forceinline__ void rotate(const Row& x, const uint32_t (&c)[10], const uint32_t (&s)[10],
                                       bf16x8 (&frag)[5]) {
  uint32_t y[20];
#pragma unroll
  for (int i = 0; i < 10; ++i) {
    const float c0 = lo16(c[i]), c1 = hi16(c[i]), s0 = lo16(s[i]), s1 = hi16(s[i]);
    const float a0 = lo16(x.lo[i]), a1 = hi16(x.lo[i]), b0 = lo16(x.hi[i]), b1 = hi16(x.hi[i]);
    const uint32_t ac = pack2(a0 * c0, a1 * c1), bs = pack2(-b0 * s0, -b1 * s1);
    const uint32_t bc = pack2(b0 * c0, b1 * c1), as = pack2(a0 * s0, a1 * s1);
    y[i] = pack2(lo16(ac) + lo16(bs), hi16(ac) + hi16(bs));
    y[10 + i] = pack2(lo16(bc) + lo16(as), hi16(bc) + hi16(as));
  }
#pragma unroll
  for (int kk = 0; kk < 5; ++kk)
    frag[kk] = __builtin_bit_cast(bf16x8, u32x4v{y[4 * kk], y[4 * kk + 1], y[4 * kk + 2], y[4 * kk + 3]});
}

__global__ __launch_bounds__(kThreads, 2) void vision_window_attn_kernel(
    const char* __restrict__ qkv, int64_t qkv_stride_b, const int32_t* __restrict__ pos_hw,
    const char* __restrict__ cos_tab, const char* __restrict__ sin_tab, int max_pos,
    const int32_t* __restrict__ cu, int num_tokens, int num_heads, int head_groups, float scale_log2,
    char* __restrict__ out, int64_t out_stride_b) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[kWaves][kMaxWin * kVRow];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lc = lane & 31, hf = lane >> 5;
  const int win = blockIdx.x / head_groups;
  const int head = (blockIdx.x - win * head_groups) * kWaves + wave;
  if (head >= num_heads) return;
  // Boundaries are checked on the host; a device copy that disagrees must not reach past the rows.
  const int start = min(max(cu[win], 0), num_tokens);
  const int n = min(min(cu[win + 1], num_tokens) - start, kMaxWin);
  if (n <= 0) return;
  uint8_t* const my = lds[wave];

  // ---- loads: q and k of rows lc and lc + 32, the rows' angles, V in 16-byte chunks; rows past
  // the window read its last row (their keys are masked, their queries are not stored) ----------
  Row xq[2], xk[2];
  int pos[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int tok = start + min(lc + 32 * b, n - 1);
    pos[b] = pos_hw[2 * (int64_t)tok + hf];
    const char* row = qkv + tok * qkv_stride_b + head * (kHd * 2) + hf * (kQuarter * 2);
    ld40(row, xq[b].lo);
    ld40(row + kHd, xq[b].hi);
    ld40(row + num_heads * (kHd * 2), xk[b].lo);
    ld40(row + num_heads * (kHd * 2) + kHd, xk[b].hi);
  }
  u32x4v vv[kRowChunks];
#pragma unroll
  for (int i = 0; i < kRowChunks; ++i) {
    const int x = lane + 64 * i, r = x / kRowChunks, c = x - r * kRowChunks;
    vv[i] = *reinterpret_cast<const u32x4v*>(qkv + (start + min(r, n - 1)) * qkv_stride_b +
                                             (2 * num_heads + head) * (kHd * 2) + c * 16);
  }
  bf16x8 fq[2][5], fk[2][5];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int p = min(max(pos[b], 0), max_pos - 1);
    uint32_t c[10], s[10];
    ld40(cos_tab + (int64_t)p * (kQuarter * 2), c);
    ld40(sin_tab + (int64_t)p * (kQuarter * 2), s);
    rotate(xq[b], c, s, fq[b]);
    rotate(xk[b], c, s, fk[b]);
  }

  // ---- S^T = K Q^T: [key block][query block] --------------------------------------------------
  f32x16 S[2][2] = {};
#pragma unroll
  for (int kk = 0; kk < 5; ++kk)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        S[kb][qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fk[kb][kk], fq[qb][kk], S[kb][qb], 0, 0, 0);

#pragma unroll
  for (int i = 0; i < kRowChunks; ++i) {
    const int x = lane + 64 * i, r = x / kRowChunks, c = x - r * kRowChunks;
    *reinterpret_cast<u32x4v*>(my + r * kVRow + c * 16) = vv[i];
  }

  // ---- softmax over the keys of each query column: element e of key block kb is key
  // 32 kb + 8 (e / 4) + 4 hf + e % 4 ------------------------------------------------------------
  float inv[2];
  bf16x8 P[2][2][2];  // [query block][key block][16-key chunk]
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        if (32 * kb + 8 * (e >> 2) + 4 * hf + (e & 3) >= n) S[kb][qb][e] = -INFINITY;
        mx = fmaxf(mx, S[kb][qb][e]);
      }
    mx = half_wave_max(mx) * scale_log2;
    const float base = mx == -INFINITY ? 0.f : mx;
    float l = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int ch = 0; ch < 2; ++ch) {
        u32x4v w;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(S[kb][qb][8 * ch + 2 * u], scale_log2, -base));
          const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(S[kb][qb][8 * ch + 2 * u + 1], scale_log2, -base));
          l += p0;
          l += p1;
          w[u] = pack2(p0, p1);
        }
        P[qb][kb][ch] = __builtin_bit_cast(bf16x8, w);
      }
    l += __shfl_xor(l, 32);
    inv[qb] = l > 0.f ? 1.f / l : 0.f;
  }

  // ---- O^T += V^T P^T.  In each 16-lane group lane 4f + r reads dims 4r .. 4r + 3 of key row f
  // and the transposing read hands lane j the four keys of dim j; a wave's LDS accesses run in
  // order, so V's writes above need no wait (the clobber keeps the compiler from reordering).
  // Dims 80..95 read what the row's padding holds; those output rows are not stored. ------------
  asm volatile("" ::: "memory");
  f32x16 O[2][3] = {};
  const int s = lane & 15, lg = lane >> 4;
  const uint8_t* vbase = my + (4 * (lg >> 1) + (s >> 2)) * kVRow + (lg & 1) * 32 + (s & 3) * 8;
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int ch = 0; ch < 2; ++ch)
#pragma unroll
      for (int mb = 0; mb < 3; ++mb) {
        const uint8_t* vp = vbase + (32 * kb + 16 * ch) * kVRow + mb * 64;
        const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)vp);
        const s16x4 b =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vp + 8 * kVRow));
        const s16x8 w = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
          O[qb][mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), P[qb][kb][ch],
                                                              O[qb][mb], 0, 0, 0);
      }
  asm volatile("" ::: "memory");

  // ---- output: lane holds O^T[dim 32 mb + 8 i + 4 hf + j][query 32 qb + lc] in O[qb][mb][4 i + j];
  // through LDS to whole rows, 16 bytes per lane ------------------------------------------------
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int mb = 0; mb < 3; ++mb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (32 * mb + 8 * i < kHd) {
          const u32x2v w = {pack2(O[qb][mb][4 * i] * inv[qb], O[qb][mb][4 * i + 1] * inv[qb]),
                            pack2(O[qb][mb][4 * i + 2] * inv[qb], O[qb][mb][4 * i + 3] * inv[qb])};
          *reinterpret_cast<u32x2v*>(my + (32 * qb + lc) * kORow + (32 * mb + 8 * i + 4 * hf) * 2) = w;
        }
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < kRowChunks; ++i) {
    const int x = lane + 64 * i, r = x / kRowChunks, c = x - r * kRowChunks;
    const u32x2v a = *reinterpret_cast<const u32x2v*>(my + r * kORow + c * 16);
    const u32x2v b = *reinterpret_cast<const u32x2v*>(my + r * kORow + c * 16 + 8);
    if (r < n)
      *reinterpret_cast<u32x4v*>(out + (start + r) * out_stride_b + head * (kHd * 2) + c * 16) =
          u32x4v{a[0], a[1], b[0], b[1]};
  }
}

}  // namespace
}  // namespace vlc

VLC_API int vlc_vision_window_attn(const void* qkv, int64_t qkv_row_stride, const int32_t* pos_hw,
                                   const void* cos_table, const void* sin_table, int64_t max_pos,
                                   const int32_t* cu_host, const int32_t* cu_dev, int num_windows,
                                   int64_t num_tokens, int num_heads, int head_dim, float softmax_scale,
                                   void* out, int64_t out_row_stride, void* stream) {
  using namespace vlc;
  if (head_dim != kHd) return VLC_ERR_UNSUPPORTED;
  if (num_tokens < 0 || num_windows < 0 || num_heads <= 0 || max_pos <= 0 || max_pos >= (1 << 24) ||
      num_tokens >= ((int64_t)1 << 30) || !(softmax_scale > 0.f))
    return VLC_ERR_INVALID;
  if (num_windows == 0 || num_tokens == 0) return VLC_OK;
  if (!qkv || !pos_hw || !cos_table || !sin_table || !cu_host || !cu_dev || !out) return VLC_ERR_INVALID;
  const int64_t width = (int64_t)num_heads * kHd;
  if (qkv_row_stride < 3 * width || out_row_stride < width) return VLC_ERR_INVALID;
  if (!aligned16(qkv) || !aligned16(out) || qkv_row_stride % 8 || out_row_stride % 8 ||
      (reinterpret_cast<uintptr_t>(cos_table) & 7) || (reinterpret_cast<uintptr_t>(sin_table) & 7))
    return VLC_ERR_UNSUPPORTED;
  if (cu_host[0] < 0 || cu_host[num_windows] > num_tokens) return VLC_ERR_INVALID;
  for (int i = 0; i < num_windows; ++i) {
    if (cu_host[i + 1] < cu_host[i]) return VLC_ERR_INVALID;
    if (cu_host[i + 1] - cu_host[i] > kMaxWin) return VLC_ERR_UNSUPPORTED;
  }
  const int64_t groups = (num_heads + kWaves - 1) / kWaves;
  if (groups * num_windows >= ((int64_t)1 << 31)) return VLC_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(vision_window_attn_kernel, dim3((unsigned)(groups * num_windows)), dim3(kThreads), 0,
                     as_stream(stream), static_cast<const char*>(qkv), qkv_row_stride * 2, pos_hw,
                     static_cast<const char*>(cos_table), static_cast<const char*>(sin_table), (int)max_pos, cu_dev,
                     (int)num_tokens, num_heads, (int)groups, softmax_scale * 1.4426950408889634f,
                     static_cast<char*>(out), out_row_stride * 2);
  return launch_status();
}
