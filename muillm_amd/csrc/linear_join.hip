// A linear layer together with what follows it at the boundary between two sublayers:
//   fp32 residual stream    y = W x + bias;  r <- r + branch_scale * post_gain * y * rsqrt(mean(y^2) + eps);
//                           h = next_scale * next_gain * r * rsqrt(mean(r^2) + eps)          (mui_residual_norm behind mui_linear)
//   16-bit residual stream  y = W x + bias + r;  h = next_gain * y * rsqrt(mean(y^2) + eps)  (mui_rmsnorm behind mui_linear)
//
// The linear divides its K between workgroups wherever that is worth a launch that adds the fp32 partial outputs up: with 17 to 128 tokens in gemm_stream.hip,
// with more of them, and codes from 65 on, in gemm_prefill.hip. That launch and the norm's are one here: one workgroup per token adds the token's row up and has it in registers for
// the norms. Neither is bound by its bytes (a few hundred KB per row at most); each is a launch, a chain of cold loads and one or two sums over the
// workgroup, so one of them is what is saved. Everything else runs as the two calls it stands for, and K is divided as without the norm: the bits are those of the two
// calls. (Dividing it also where only the adding launch spoke against it gave 14.8 -> 12.5 us for 4096 x 4096 at 32 tokens, and other sums than a model whose boundaries are not
// taken along.) us in bf16 as captured, two calls -> one, at 32 / 128 tokens: with an fp32 stream 4096 x 4096 (K undivided / divided) 14.8 -> 14.6 / 22.6 -> 19.9,
// 4096 x 14336 28.5 -> 25.1 / 39.4 -> 36.8, 2048 x 2048 (undivided) 9.7 -> 9.7 / 14.4 -> 14.4, 2048 x 8192 14.4 -> 12.1 / 22.2 -> 19.7; with a 16-bit one 4096 x 4096
// 13.7 -> 13.5 / 21.5 -> 19.4, 4096 x 14336 27.5 -> 25.4 / 38.6 -> 36.4, 2048 x 8192 13.8 -> 11.8 / 22.1 -> 19.3.
#include "skinny.cuh"

namespace mui {

struct JoinRow {
  const float* part;  // [splits][tokens][n]
  int splits, n, tokens;
  const uint16_t* add_bias;   // [n] or null
  const float* r32;           // [tokens, n], fp32 residual (or null: 0)
  const uint16_t* r16;        // [tokens, n], 16-bit residual
  const uint16_t *post_gain, *next_gain;  // [n] or null
  float branch_scale, next_scale, eps;
  uint16_t* y;
  float* r_out;
  uint16_t* h;
};

constexpr int kJoinThreads = 256;

__device__ __forceinline__ float join_sum(float v, float* red) {
  v = wave_sum(v);
  __syncthreads();  // the previous use of red is over
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// One token per workgroup; thread t has outputs 8 (t + 256 j) .. + 7 (n <= 2048 CH). Sums are taken in the order of the kernels that this one stands for
// (gemm_stream_add, rmsnorm, residual_norm): the results are theirs, bit for bit.
template <typename T, bool F32, int CH>
__global__ void __launch_bounds__(kJoinThreads) linear_join_kernel(const JoinRow p) {
  __shared__ float red[kJoinThreads / kWave];
  int at_c[CH];
  bool in[CH];
  const long row = (long)blockIdx.x * p.n, all = (long)p.tokens * p.n;
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int c = (threadIdx.x + kJoinThreads * j) * 8;
    in[j] = c < p.n;
    at_c[j] = in[j] ? c : 0;
  }
  // everything is requested before anything is used; four shares at a time, added in order
  u32x4 gp[CH], gn[CH], rh[CH], bias[CH];
  f32x4 r[CH][2], a[CH][2], v[CH][4][2];
  auto request = [&](int s0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float* src = p.part + (s0 + u < p.splits ? s0 + u : p.splits - 1) * all + row;
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        v[j][u][0] = *(const f32x4*)(src + at_c[j]);
        v[j][u][1] = *(const f32x4*)(src + at_c[j] + 4);
      }
    }
  };
  request(0);
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    if constexpr (F32) {
      r[j][0] = r[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (p.r32) {
        r[j][0] = *(const f32x4*)(p.r32 + row + at_c[j]);
        r[j][1] = *(const f32x4*)(p.r32 + row + at_c[j] + 4);
      }
      if (p.post_gain) gp[j] = ld16(p.post_gain + at_c[j]);
    } else {
      rh[j] = ld16(p.r16 + row + at_c[j]);
    }
    if (p.next_gain) gn[j] = ld16(p.next_gain + at_c[j]);
    if (p.add_bias) bias[j] = ld16(p.add_bias + at_c[j]);
  }
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    a[j][0] = v[j][0][0];
    a[j][1] = v[j][0][1];
  }
  auto add = [&](int u, int s) {
    if (s < p.splits)
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        a[j][0] += v[j][u][0];
        a[j][1] += v[j][u][1];
      }
  };
#pragma unroll
  for (int u = 1; u < 4; ++u) add(u, u);
  if (p.splits > 4) {
    request(4);
#pragma unroll
    for (int u = 0; u < 4; ++u) add(u, 4 + u);
  }
  float y[CH][8], f[8];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < CH; ++j) {
#pragma unroll
    for (int i = 0; i < 8; ++i) y[j][i] = a[j][i >> 2][i & 3];
    if (p.add_bias) {
      unpack8<T>(bias[j], f);
#pragma unroll
      for (int i = 0; i < 8; ++i) y[j][i] += f[i];
    }
    if constexpr (!F32) {
      unpack8<T>(rh[j], f);
#pragma unroll
      for (int i = 0; i < 8; ++i) y[j][i] += f[i];
    }
    // the norms see y as it is stored
    const u32x4 packed = pack8<T>(y[j]);
    if (in[j]) *(u32x4*)(p.y + row + at_c[j]) = packed;
    unpack8<T>(packed, y[j]);
  }
  if constexpr (F32) {
    if (p.post_gain) {
#pragma unroll
      for (int j = 0; j < CH; ++j)
        if (in[j])
#pragma unroll
          for (int i = 0; i < 8; ++i) ss = fmaf(y[j][i], y[j][i], ss);
      const float rs = rsqrtf(join_sum(ss, red) / (float)p.n + p.eps);
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        unpack8<T>(gp[j], f);
#pragma unroll
        for (int i = 0; i < 8; ++i) y[j][i] = fmaf(f[i] * p.branch_scale, y[j][i] * rs, r[j][i >> 2][i & 3]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < CH; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) y[j][i] += r[j][i >> 2][i & 3];
    }
#pragma unroll
    for (int j = 0; j < CH; ++j)
      if (in[j]) {
        *(f32x4*)(p.r_out + row + at_c[j]) = f32x4{y[j][0], y[j][1], y[j][2], y[j][3]};
        *(f32x4*)(p.r_out + row + at_c[j] + 4) = f32x4{y[j][4], y[j][5], y[j][6], y[j][7]};
      }
  }
  float rs = p.next_scale;
  if (p.next_gain) {
    ss = 0.f;
#pragma unroll
    for (int j = 0; j < CH; ++j)
      if (in[j])
#pragma unroll
        for (int i = 0; i < 8; ++i) ss = fmaf(y[j][i], y[j][i], ss);
    rs = rsqrtf(join_sum(ss, red) / (float)p.n + p.eps) * p.next_scale;
  }
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    if (p.next_gain) {
      unpack8<T>(gn[j], f);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = 1.f;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) y[j][i] = f[i] * (y[j][i] * rs);
    if (in[j]) *(u32x4*)(p.h + row + at_c[j]) = pack8<T>(y[j]);
  }
}

template <typename T, bool F32>
static int launch_join(hipStream_t s, const JoinRow& p) {
  const dim3 grid(p.tokens), block(kJoinThreads);
  const int ch = ceil_div(p.n, 8 * kJoinThreads);
  if (ch <= 1) hipLaunchKernelGGL((linear_join_kernel<T, F32, 1>), grid, block, 0, s, p);
  else if (ch <= 2) hipLaunchKernelGGL((linear_join_kernel<T, F32, 2>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((linear_join_kernel<T, F32, 4>), grid, block, 0, s, p);
  return launch_status();
}
constexpr int kJoinMost = 8192;  // outputs

// q: the product, without what its end applies. MUI_ERR_UNSUPPORTED: not a case for it, nothing has been launched
static int linear_join(hipStream_t s, int dtype, int wf, SkinnyParams q, JoinRow p, bool f32, void* workspace, size_t workspace_bytes) {
  // (rows are read and written eight values at a time; what leaves the shares of K asks for four only)
  if (p.tokens <= MUI_MAX_TOKENS || p.n > kJoinMost || p.n % 8 || !p.h || !workspace || ((uintptr_t)workspace & 255u) || workspace_bytes < prefill_workspace_bytes()) return MUI_ERR_UNSUPPORTED;
  const void* ptrs[] = {q.w0, q.x, p.add_bias, p.r32, p.r16, p.post_gain, p.next_gain, p.y, p.r_out, p.h};
  for (const void* at : ptrs)
    if (!aligned16(at)) return MUI_ERR_UNSUPPORTED;
  q.y = p.y; q.n = p.n; q.tokens = p.tokens;
  const auto turn = scratch_turn(workspace);
  float* part = (float*)((char*)workspace + prefill_counter_bytes());
  // (K is divided only where it is without the norm, too: whether the boundary was taken along, a hook was listening or all layers came in one call does not show in the bits)
  const size_t part_bytes = workspace_bytes - prefill_counter_bytes();
  const int st = wf == WF_16BIT && p.tokens <= 128 ? launch_gemm_stream_parts(s, dtype, q, part, part_bytes, &p.splits)
                                                   : launch_prefill_parts(s, dtype, wf, q, part, part_bytes, &p.splits);
  if (st != MUI_OK) return st;
  p.part = part;
  if (dtype == MUI_DTYPE_F16) return f32 ? launch_join<F16, true>(s, p) : launch_join<F16, false>(s, p);
  return f32 ? launch_join<BF16, true>(s, p) : launch_join<BF16, false>(s, p);
}

static SkinnyParams product(const void* weights, long w_pitch, const void* x, int k) {
  SkinnyParams q = {};
  q.w0 = weights; q.pitch = w_pitch; q.x = (const uint16_t*)x; q.k = k;
  return q;
}

// int8 codes (dense pairs) with the residual and the norm behind, where K is shared between workgroups; MUI_ERR_UNSUPPORTED: it is not, nothing has been launched
int launch_codes_norm(hipStream_t s, int dtype, int wf, const SkinnyParams& q, const void* next_gain, float eps, void* h) {
  if (q.gamma || q.mul_bias) return MUI_ERR_UNSUPPORTED;
  const int st = check_int8_linear(dtype, q.w0, q.pitch, q.s0, wf == WF_U8_GROUP ? q.group_shift : 0, q.x, q.n, q.k, q.tokens);
  if (st != MUI_OK) return st;
  JoinRow p = {};
  p.n = q.n; p.tokens = q.tokens; p.add_bias = q.add_bias; p.r16 = q.residual; p.next_gain = (const uint16_t*)next_gain;
  p.next_scale = 1.f; p.eps = eps; p.y = q.y; p.h = (uint16_t*)h;
  SkinnyParams a = q;
  a.add_bias = a.residual = nullptr;
  a.s_pitch = wf == WF_U8_GROUP ? 2L * (q.k >> q.group_shift) : 1;
  return linear_join(s, dtype, wf, a, p, false, q.workspace, q.workspace_bytes);
}

static bool linear_args(int dtype, const void* weights, long w_pitch, const void* x, const void* y, int n, int k, int tokens) {
  return weights && x && y && n > 0 && k > 0 && tokens > 0 && w_pitch >= k && (dtype == MUI_DTYPE_F16 || dtype == MUI_DTYPE_BF16);
}

}  // namespace mui

using namespace mui;

extern "C" int mui_linear_residual_norm(mui_stream_t stream, int dtype, const void* weights, long w_pitch, const void* x, const void* add_bias,
                                        const float* residual_in, const void* post_gain, float branch_scale, const void* next_gain,
                                        float next_scale, float epsilon, void* y, float* residual_out, void* h, int n_out, int k_in, int tokens,
                                        void* workspace, size_t workspace_bytes) {
  MUI_CHECK_ARG(linear_args(dtype, weights, w_pitch, x, y, n_out, k_in, tokens));
  MUI_CHECK_ARG(residual_out && (h || !next_gain) && (workspace || workspace_bytes == 0));
  {
    JoinRow p = {};
    p.n = n_out; p.tokens = tokens; p.add_bias = (const uint16_t*)add_bias; p.r32 = residual_in; p.post_gain = (const uint16_t*)post_gain;
    p.next_gain = (const uint16_t*)next_gain; p.branch_scale = branch_scale; p.next_scale = next_scale; p.eps = epsilon;
    p.y = (uint16_t*)y; p.r_out = residual_out; p.h = (uint16_t*)h;
    const int st = linear_join((hipStream_t)stream, dtype, WF_16BIT, product(weights, w_pitch, x, k_in), p, true, workspace, workspace_bytes);
    if (st != MUI_ERR_UNSUPPORTED) return st;
  }
  const int st = mui_linear_ws(stream, dtype, weights, w_pitch, x, nullptr, 0.f, nullptr, add_bias, nullptr, y, n_out, k_in, tokens, workspace, workspace_bytes);
  if (st != MUI_OK) return st;
  return mui_residual_norm(stream, dtype, residual_in, y, 1.f, post_gain, branch_scale, next_gain, next_scale, epsilon, residual_out, h, tokens, n_out);
}

extern "C" int mui_linear_norm(mui_stream_t stream, int dtype, const void* weights, long w_pitch, const void* x, const void* add_bias, const void* residual,
                               const void* next_gain, float epsilon, void* y, void* h, int n_out, int k_in, int tokens, void* workspace,
                               size_t workspace_bytes) {
  MUI_CHECK_ARG(linear_args(dtype, weights, w_pitch, x, y, n_out, k_in, tokens));
  MUI_CHECK_ARG(residual && next_gain && h && (workspace || workspace_bytes == 0));
  {
    JoinRow p = {};
    p.n = n_out; p.tokens = tokens; p.add_bias = (const uint16_t*)add_bias; p.r16 = (const uint16_t*)residual; p.next_gain = (const uint16_t*)next_gain;
    p.next_scale = 1.f; p.eps = epsilon; p.y = (uint16_t*)y; p.h = (uint16_t*)h;
    const int st = linear_join((hipStream_t)stream, dtype, WF_16BIT, product(weights, w_pitch, x, k_in), p, false, workspace, workspace_bytes);
    if (st != MUI_ERR_UNSUPPORTED) return st;
  }
  const int st = mui_linear_ws(stream, dtype, weights, w_pitch, x, nullptr, 0.f, nullptr, add_bias, residual, y, n_out, k_in, tokens, workspace, workspace_bytes);
  if (st != MUI_OK) return st;
  return mui_rmsnorm(stream, dtype, next_gain, y, epsilon, h, tokens, n_out);
}
