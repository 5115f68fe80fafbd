// Interface between the single-token GEMV entry points and the small-batch MFMA kernel.
#pragma once

#include <mutex>

#include "common.cuh"

namespace mui {

enum { WF_16BIT = 0, WF_I8_CHANNEL = 1, WF_U8_GROUP = 2 };
enum { SK_LINEAR = 0, SK_GATEUP = 1 };

struct SkinnyParams {
  const void* w0;       // linear: matrix; gate/up: gate rows
  const void* w1;       // gate/up: up rows
  long pitch;           // row pitch in weight elements
  const uint16_t* s0;   // I8_CHANNEL: scale of row n at s0[n*s_pitch]; U8_GROUP: pairs at s0 + n*s_pitch + 2g
  const uint16_t* s1;
  long s_pitch;
  int group_shift;
  const uint16_t* x;    // [tokens, k], token rows x_pitch elements apart (0: k)
  long x_pitch;         // honoured by the 1..4-token kernels (their K-segment calls); others need 0
  const uint16_t* gamma;
  const uint16_t* mul_bias;  // gate/up: the up rows' bias (both biases or none)
  const uint16_t* add_bias;  // gate/up: the gate rows' bias
  const uint16_t* residual;  // [tokens, n]
  uint16_t* y;               // [tokens, n]
  int n;       // outputs (weight rows, or gate/up pairs)
  int k;
  int tokens;  // 1..16
  float eps;
  void* workspace;         // optional scratch of the prompt GEMM (mui_linear_ws), zeroed once by the caller
  size_t workspace_bytes;
};

// Operands of the prompt GEMM (gemm_prefill.hip)
struct PrefillGemmParams {
  const uint8_t* w0;      // linear: matrix; gate/up: gate rows
  const uint8_t* w1;      // gate/up: up rows
  long pitch;             // weight row pitch in bytes
  const uint16_t* s0;     // per-channel int8: scale of row n at s0[n * s_pitch]; group format: (scale, min) pairs of row n at s0 + n * s_pitch + 2 g
  const uint16_t* s1;
  long s_pitch;
  int group_shift;        // group format: log2 of the codes per (scale, min) pair
  const uint16_t* x;      // [tokens, k] dense
  const uint16_t* gamma;
  const uint16_t* mul_bias;
  const uint16_t* add_bias;
  const uint16_t* residual;  // [tokens, n] dense
  uint16_t* y;               // [tokens, n]: row pitch y_pitch elements (n unless the launch covers a band of the outputs)
  long y_pitch;              // (the residual has the same pitch)
  int n;        // outputs (weight rows; gate/up pairs)
  int k;
  int tokens;
  float eps;
  int n_tiles;  // row tiles
  int t_tiles;  // token tiles
  // K split over workgroups (prefill_gemm_kernel<..., XS = true>): partial tiles and arrival counters
  int k_splits;
  int row_split;          // the XCDs divide the tile grid row_split ways by rows, 8 / row_split ways by tokens
  int row_group;          // row tiles per panel of an XCD's tile walk
  int total_blocks;       // software-pipelined tiles: tiles of the launch (slots of an XCD, times 8)
  int slots;              // tiles that each XCD takes (0: all of its share)
  int first_slot;         // sub_rows > 0: the launch takes what another one's larger tiles left, from this slot on, every tile of it as
  int sub_rows, sub_toks; // sub_rows x sub_toks smaller ones; n_tiles to row_group are the other launch's
  float* part;            // [tiles * k_splits] partial tiles in fp32
  unsigned* part_count;   // [tiles], zero between launches
};

// SiLU(g) * u of the gate/up epilogues, the product rounded to fp32 before it is rounded to the 16-bit
// type. Left alone the compiler merges the product and the conversion into one mixed-precision
// instruction (v_fma_mixlo_f16) for some outputs and not for others, depending on the code around
// them, and the instruction does not round like the pair it replaces: two kernels of the same tile
// then differ in the last place of a few outputs in a hundred thousand. The empty asm keeps the
// product a value of its own.
__device__ __forceinline__ float gateup_f32(float g, float u) {
  float r = silu_f32(g) * u;
  asm volatile("" : "+v"(r));
  return r;
}

// B operand of one k-chunk: gamma * x rounded to the 16-bit type, sum of squares on the side.
// fp16: packed multiply (one rounding, same result as the fp32 product rounded once) and a
// packed dot for the squares.
template <typename T, bool NORM>
__device__ __forceinline__ u32x4 make_b(const u32x4 xv, const u32x4 gv, float& ss) {
  if constexpr (!NORM) {
    return xv;
  } else if constexpr (T::kDtype == MUI_DTYPE_F16) {
    const uint32_t xw[4] = {xv.x, xv.y, xv.z, xv.w};
    const uint32_t gw[4] = {gv.x, gv.y, gv.z, gv.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f16x2 xx = __builtin_bit_cast(f16x2, xw[i]);
      ss = __builtin_amdgcn_fdot2(xx, xx, ss, false);
      o[i] = __builtin_bit_cast(uint32_t, xx * __builtin_bit_cast(f16x2, gw[i]));
    }
    u32x4 b = {o[0], o[1], o[2], o[3]};
    return b;
  } else {
    float xf[8], gf[8], o[8];
    unpack8<T>(xv, xf);
    unpack8<T>(gv, gf);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      ss = fmaf(xf[i], xf[i], ss);
      o[i] = xf[i] * gf[i];
    }
    return pack8<T>(o);
  }
}

// v_mfma_f32_16x16x32: A = 16 rows x 32 k, B = 32 k x 16 columns; lane l supplies 8 k-values
// (k-chunk l / 16 of the step) of row / column l % 16
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <typename T>
__device__ __forceinline__ f32x4 mfma16x16x32(u32x4 a, u32x4 b, f32x4 c);
template <>
__device__ __forceinline__ f32x4 mfma16x16x32<F16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma16x16x32<BF16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// 8 int8/uint8 weights (two dwords) -> the 16-bit MFMA operand.
//   per-channel: exact integers (the row scale is applied in the epilogue). For fp16 the bytes
//   are dropped into the mantissa of 1024.0 (0x6400 | b = 1024 + b) with two byte permutes and
//   the offset is removed with a packed subtract: 5 VALU ops per dword instead of a convert
//   and a pack per weight.
//   group format: u8 * scale + min, rounded once to the 16-bit type.
template <typename T, int WF>
__device__ __forceinline__ u32x4 convert_a(uint32_t w0, uint32_t w1, const uint16_t* srow, int elem, int group_shift) {
  const uint32_t v[2] = {w0, w1};
  if constexpr (WF == WF_I8_CHANNEL && T::kDtype == MUI_DTYPE_F16) {
    u32x4 out;
    const f16x2 off = {(_Float16)1152.f, (_Float16)1152.f};  // 1024 + 128 (sign bit flipped below)
    uint32_t o[4];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const uint32_t u = v[m] ^ 0x80808080u;
      const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
      const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
      o[2 * m + 0] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, lo) - off);
      o[2 * m + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, hi) - off);
    }
    out.x = o[0]; out.y = o[1]; out.z = o[2]; out.w = o[3];
    return out;
  } else {
    float f[8];
    if constexpr (WF == WF_I8_CHANNEL) {
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int b = 0; b < 4; ++b) f[4 * m + b] = (float)(int)(int8_t)((v[m] >> (8 * b)) & 0xffu);
    } else {
      const uint32_t pr = ld4(srow + 2 * (elem >> group_shift));
      const float sc = T::lo(pr), mn = T::hi(pr);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int b = 0; b < 4; ++b) f[4 * m + b] = fmaf((float)((v[m] >> (8 * b)) & 0xffu), sc, mn);
    }
    return pack8<T>(f);
  }
}

// group format with the (scale, min) pair already in a register: u8 * scale + min, rounded once
template <typename T>
__device__ __forceinline__ u32x4 convert_a_pair(uint32_t w0, uint32_t w1, uint32_t pair) {
  const uint32_t v[2] = {w0, w1};
  const float sc = T::lo(pair), mn = T::hi(pair);
  float f[8];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int b = 0; b < 4; ++b) f[4 * m + b] = fmaf((float)((v[m] >> (8 * b)) & 0xffu), sc, mn);
  return pack8<T>(f);
}

// the same for fp16 in packed arithmetic: 1024 + u8 by byte permutes, 1024 off again (exact), one fused multiply-add whose
// single rounding is the one to fp16
__device__ __forceinline__ u32x4 convert_a_pair_f16(uint32_t w0, uint32_t w1, uint32_t pair) {
  const uint32_t v[2] = {w0, w1};
  const f16x2 pr = __builtin_bit_cast(f16x2, pair), sc = {pr.x, pr.x}, mn = {pr.y, pr.y};
  const f16x2 off = {(_Float16)1024.f, (_Float16)1024.f};
  uint32_t o[4];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, v[m], 0x04010400u);
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, v[m], 0x04030402u);
    o[2 * m + 0] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, lo) - off, sc, mn));
    o[2 * m + 1] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, hi) - off, sc, mn));
  }
  return u32x4{o[0], o[1], o[2], o[3]};
}

// A linear that shares K writes its scratch in one launch and reads it in the next. Threads may issue linears on one stream, and with it on one scratch: whoever holds this has both
// launches in the stream before another thread's calls. (20 ns; none: without scratch)
inline std::unique_lock<std::recursive_mutex> scratch_turn(const void* scratch) {
  static std::recursive_mutex turns[16];
  if (!scratch) return {};
  return std::unique_lock<std::recursive_mutex>(turns[((uintptr_t)scratch >> 20) % 16]);
}
// tiled matrix-core GEMM for prompts (gemm_prefill.hip): any token count, 16-bit weights or int8 codes of either format
int launch_prefill_gemm(hipStream_t s, int dtype, int weight_format, int epilogue, const SkinnyParams& p);
size_t prefill_workspace_bytes();  // what SkinnyParams::workspace must hold for the prompt GEMM to use it
size_t prefill_workspace_best();   // beyond, more of it is no use
// more than 128 tokens (codes: 64), n % 4 == 0: fp32 partial outputs [*shares][tokens][n] of shares of K, where they are worth it, and what adds them up behind
int launch_prefill_parts(hipStream_t s, int dtype, int weight_format, const SkinnyParams& p, float* part, size_t part_bytes, int* shares);
// what mui_int8_linear_ws (group_shift 0) and mui_int8_group_linear_ws ask of their operands (int8.hip)
int check_int8_linear(int dtype, const void* codes, long pitch, const void* scales, int group_shift, const void* x, int n, int k, int tokens);
int launch_codes_norm(hipStream_t s, int dtype, int weight_format, const SkinnyParams& p, const void* next_gain, float eps, void* h);  // (linear_join.hip)
int launch_parts_add(hipStream_t s, int dtype, const SkinnyParams& p, float* part, int shares);
size_t prefill_counter_bytes();    // of that, at its start: counters that stay zero
// 17..128 tokens: 16 weight rows per workgroup, K split over its waves, token columns in up to 8 MFMA tiles (gemm_wide.hip)
int launch_gemm_wide(hipStream_t s, int dtype, int weight_format, int epilogue, const SkinnyParams& p);
// 17..128 tokens, 16-bit weights, k % 256 == 0, n % 8 == 0, no fused norm: bands of weight rows streamed through LDS stages that
// the workgroup shares; part (part_bytes, may be none): fp32 partial outputs where shares of K are worth it (gemm_stream.hip). MUI_ERR_UNSUPPORTED
// for everything else and for what the tiled GEMM does faster
float gemm_stream_time(int dtype, int weight_format, int epilogue, const SkinnyParams& p, size_t part_bytes);  // of the next two, in us; negative: they decline
int launch_gemm_stream(hipStream_t s, int dtype, int epilogue, const SkinnyParams& p, float* part, size_t part_bytes);
int launch_gemm_stream_int8(hipStream_t s, int dtype, int weight_format, int epilogue, const SkinnyParams& p);  // codes, 17..64 tokens
int launch_gemm_stream_parts(hipStream_t s, int dtype, const SkinnyParams& p, float* part, size_t part_bytes, int* splits);
// launches gemm_skinny_kernel<dtype, weight format, epilogue>; returns a MUI_* status
int launch_skinny(hipStream_t s, int dtype, int weight_format, int epilogue, const SkinnyParams& p);
// experiments: 0 disables the B-stationary persistent variant
void skinny_set_bstat(int on);
void skinny_set_lt(int on);  // 0: operands loaded straight from HBM in MFMA order (older kernels)

// The boundary between two sublayers (residual_norm.hip) in front of a product of one token
struct BoundaryInFront {
  const float* stream;
  const uint16_t *post_gain, *next_gain;  // or null
  float branch_scale, next_scale;
  float* stream_out;  // not stream: other workgroups still read that
  uint16_t* h;        // the product's input
};
// What a workgroup of 256 threads reads of it, thread t having values 8 (t + 256 j) .. + 7; values and order of sums are residual_norm.hip's
template <typename T, int CH>
struct FrontOperands {
  f32x4 stream[CH][2];
  u32x4 post[CH], next[CH];
  // y: the sublayer's output (read where a gain is not there)
  __device__ __forceinline__ void request(const BoundaryInFront& f, const uint16_t* y, const int (&at)[CH]) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      stream[j][0] = *(const f32x4*)(f.stream + at[j]);
      stream[j][1] = *(const f32x4*)(f.stream + at[j] + 4);
      post[j] = ld16((f.post_gain ? f.post_gain : y) + at[j]);
      next[j] = ld16((f.next_gain ? f.next_gain : y) + at[j]);
    }
  }
  // x: the sublayer's output on the way in, the next one's input on the way out (zeros past the end)
  __device__ __forceinline__ void finish(const BoundaryInFront& f, u32x4 (&x)[CH], const bool (&valid)[CH], const int (&at)[CH], int k, float eps, float (&red)[2][4], bool writes) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    auto block_sum = [&](float v, float (&meet)[4]) {
      v = wave_sum(v);
      if (lane == 0) meet[wave] = v;
      __syncthreads();
      return (meet[0] + meet[1]) + (meet[2] + meet[3]);
    };
    float xs[CH][8], ys[CH][8], g[8], sq = 0.f;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      unpack8<T>(x[j], ys[j]);
#pragma unroll
      for (int i = 0; i < 8; ++i) xs[j][i] = stream[j][i >> 2][i & 3];
    }
    if (f.post_gain) {
#pragma unroll
      for (int j = 0; j < CH; ++j)
        if (valid[j])
#pragma unroll
          for (int i = 0; i < 8; ++i) sq = fmaf(ys[j][i], ys[j][i], sq);
      const float rs = rsqrtf(block_sum(sq, red[0]) / (float)k + eps);
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        unpack8<T>(post[j], g);
#pragma unroll
        for (int i = 0; i < 8; ++i) xs[j][i] = fmaf(g[i] * f.branch_scale, ys[j][i] * rs, xs[j][i]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < CH; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) xs[j][i] += ys[j][i];
    }
    float rs = f.next_scale;
    if (f.next_gain) {
      sq = 0.f;
#pragma unroll
      for (int j = 0; j < CH; ++j)
        if (valid[j])
#pragma unroll
          for (int i = 0; i < 8; ++i) sq = fmaf(xs[j][i], xs[j][i], sq);
      rs = rsqrtf(block_sum(sq, red[1]) / (float)k + eps) * f.next_scale;
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      unpack8<T>(next[j], g);
      float o[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = (f.next_gain ? g[i] : 1.f) * (xs[j][i] * rs);
      const u32x4 b = pack8<T>(o), zero = {0u, 0u, 0u, 0u};
      if (writes && valid[j]) {
        *(f32x4*)(f.stream_out + at[j]) = f32x4{xs[j][0], xs[j][1], xs[j][2], xs[j][3]};
        *(f32x4*)(f.stream_out + at[j] + 4) = f32x4{xs[j][4], xs[j][5], xs[j][6], xs[j][7]};
        *(u32x4*)(f.h + at[j]) = b;
      }
      x[j] = valid[j] ? b : zero;
    }
  }
};
int launch_gemv_join(hipStream_t s, int dtype, int epilogue, const SkinnyParams& p, const BoundaryInFront& front);
// 1..8 tokens, 16-bit weights: the single-token GEMV structure with the token operands packed
// in registers (gemv_multi.hip); returns MUI_ERR_UNSUPPORTED for shapes it does not cover
int launch_gemv_multi(hipStream_t s, int dtype, int epilogue, const SkinnyParams& p);
void gemv_multi_set_two(int min_passes);  // fewest row groups per workgroup for its two-set variant (0: never)
// MFMA skinny GEMM whose weight rows are read as contiguous runs and turned into operands
// through wave-private LDS (gemm_skinny_lt.hip); MUI_ERR_UNSUPPORTED for shapes it does not cover
int launch_skinny_lt(hipStream_t s, int dtype, int weight_format, int epilogue, const SkinnyParams& p);
int int8_tuned_wgs_per_cu();  // mui_tune_int8's workgroups-per-CU override (0 = built-in)
int int8_tuned_rows();        // mui_tune_int8's rows-per-group override (0 = built-in)
int gemv_tuned_wgs_per_cu();  // mui_tune_gemv's workgroups-per-CU override (0 = built-in)
// 2..4 tokens, int8 weights, fp16 activations (int8_multi.hip); same contract
int launch_int8_multi(hipStream_t s, int dtype, int weight_format, int epilogue, const SkinnyParams& p);
void skinny_set_int8_multi(int on);
// 1..4 tokens, int8 weights, fp16 activations on the 4 x 4 x 4 matrix instruction (int8_quad.hip); same contract
int launch_int8_quad(hipStream_t s, int dtype, int weight_format, int epilogue, const SkinnyParams& p);
void int8_set_packed_dot(bool on);  // int8.hip: single fp16 token through int8_multi.hip

}  // namespace mui
