// The boundary between two sublayers (mui_residual_norm) together with the product behind it: a linear, gate and up with their activation, or a linear with
// fp32 outputs. Of a single token it is one launch, in which every workgroup computes the boundary while its first weights are on their way (gemv_multi.hip, moe.hip);
// everything else, and what those decline, runs as the two calls it stands for. The bits are those of the two calls.
#include "skinny.cuh"

namespace mui {

int launch_linear_f32_join(hipStream_t s, int dtype, const void* w, const void* x, const void* bias, float* y, int n, int k, float eps, const BoundaryInFront& front);

struct Bytes { const void* at; size_t n; };
static bool apart(Bytes a, Bytes b) {
  const uintptr_t x = (uintptr_t)a.at, y = (uintptr_t)b.at;
  return !a.at || !b.at || x + a.n <= y || y + b.n <= x;
}

// Operands and sizes that the kernels' loads cannot take. Every workgroup reads the boundary's inputs while others are writing: no output may lie on one of them, nor on another output,
// where the two calls, one after the other, allow it.
static bool joins(int dtype, int tokens, int k, const BoundaryInFront& f, const void* y, Bytes out) {
  const void* ptrs[] = {y, f.stream, f.post_gain, f.next_gain, f.stream_out, f.h};
  bool ok = tokens == 1 && k % 8 == 0 && f.stream && (dtype == MUI_DTYPE_F16 || dtype == MUI_DTYPE_BF16);
  for (const void* p : ptrs) ok = ok && aligned16(p);
  const size_t row = (size_t)k * 2;
  const Bytes in[] = {{f.stream, 2 * row}, {y, row}, {f.post_gain, row}, {f.next_gain, row}}, outs[] = {{f.stream_out, 2 * row}, {f.h, row}, out};
  for (int i = 0; i < 3; ++i) {
    for (const Bytes& b : in) ok = ok && apart(outs[i], b);
    for (int j = 0; j < i; ++j) ok = ok && apart(outs[i], outs[j]);
  }
  return ok;
}

static BoundaryInFront boundary(const float* stream, const void* post_gain, float branch_scale, const void* next_gain, float next_scale, float* stream_out, void* h) {
  return {stream, (const uint16_t*)post_gain, (const uint16_t*)next_gain, branch_scale, next_scale, stream_out, (uint16_t*)h};
}

}  // namespace mui

using namespace mui;

extern "C" int mui_joined_linear(mui_stream_t stream, int dtype, const float* residual_in, const void* y, const void* post_gain, float branch_scale, const void* next_gain,
                                 float next_scale, float epsilon, float* residual_out, void* h, const void* weights, long w_pitch, const void* add_bias, void* out,
                                 int n_out, int k_in, int tokens, void* workspace, size_t workspace_bytes) {
  MUI_CHECK_ARG(y && residual_out && h && weights && out && n_out > 0 && k_in > 0 && tokens > 0 && w_pitch >= k_in && (workspace || workspace_bytes == 0));
  const BoundaryInFront front = boundary(residual_in, post_gain, branch_scale, next_gain, next_scale, residual_out, h);
  if (joins(dtype, tokens, k_in, front, y, {out, (size_t)n_out * 2}) && aligned16(weights) && w_pitch % 8 == 0) {
    SkinnyParams p = {};
    p.w0 = weights; p.pitch = w_pitch; p.x = (const uint16_t*)y; p.add_bias = (const uint16_t*)add_bias; p.y = (uint16_t*)out; p.n = n_out; p.k = k_in; p.tokens = 1;
    p.eps = epsilon;
    const int st = launch_gemv_join((hipStream_t)stream, dtype, SK_LINEAR, p, front);
    if (st != MUI_ERR_UNSUPPORTED) return st;
  }
  const int st = mui_residual_norm(stream, dtype, residual_in, y, 1.f, post_gain, branch_scale, next_gain, next_scale, epsilon, residual_out, h, tokens, k_in);
  if (st != MUI_OK) return st;
  return mui_linear_ws(stream, dtype, weights, w_pitch, h, nullptr, 0.f, nullptr, add_bias, nullptr, out, n_out, k_in, tokens, workspace, workspace_bytes);
}

extern "C" int mui_joined_gateup_silu(mui_stream_t stream, int dtype, const float* residual_in, const void* y, const void* post_gain, float branch_scale,
                                      const void* next_gain, float next_scale, float epsilon, float* residual_out, void* h, const void* gate, const void* up,
                                      long gu_pitch, const void* gate_bias, const void* up_bias, void* out, int n_inter, int k_in, int tokens) {
  MUI_CHECK_ARG(y && residual_out && h && gate && up && out && n_inter > 0 && k_in > 0 && tokens > 0 && gu_pitch >= k_in && (gate_bias == nullptr) == (up_bias == nullptr));
  const BoundaryInFront front = boundary(residual_in, post_gain, branch_scale, next_gain, next_scale, residual_out, h);
  if (joins(dtype, tokens, k_in, front, y, {out, (size_t)n_inter * 2}) && aligned16(gate) && aligned16(up) && gu_pitch % 8 == 0) {
    SkinnyParams p = {};
    p.w0 = gate; p.w1 = up; p.pitch = gu_pitch; p.x = (const uint16_t*)y; p.add_bias = (const uint16_t*)gate_bias; p.mul_bias = (const uint16_t*)up_bias;
    p.y = (uint16_t*)out; p.n = n_inter; p.k = k_in; p.tokens = 1; p.eps = epsilon;
    const int st = launch_gemv_join((hipStream_t)stream, dtype, SK_GATEUP, p, front);
    if (st != MUI_ERR_UNSUPPORTED) return st;
  }
  const int st = mui_residual_norm(stream, dtype, residual_in, y, 1.f, post_gain, branch_scale, next_gain, next_scale, epsilon, residual_out, h, tokens, k_in);
  if (st != MUI_OK) return st;
  return mui_gateup_silu_bias(stream, dtype, gate, up, gu_pitch, h, nullptr, 0.f, gate_bias, up_bias, out, n_inter, k_in, tokens);
}

extern "C" int mui_joined_linear_f32(mui_stream_t stream, int dtype, const float* residual_in, const void* y, const void* post_gain, float branch_scale,
                                     const void* next_gain, float next_scale, float epsilon, float* residual_out, void* h, const void* weights, const void* bias,
                                     float* out, int n_out, int k_in, int tokens) {
  MUI_CHECK_ARG(y && residual_out && h && weights && out && n_out > 0 && k_in > 0 && tokens > 0);
  const BoundaryInFront front = boundary(residual_in, post_gain, branch_scale, next_gain, next_scale, residual_out, h);
  if (joins(dtype, tokens, k_in, front, y, {out, (size_t)n_out * 4}) && aligned16(weights)) {
    const int st = launch_linear_f32_join((hipStream_t)stream, dtype, weights, y, bias, out, n_out, k_in, epsilon, front);
    if (st != MUI_ERR_UNSUPPORTED) return st;
  }
  const int st = mui_residual_norm(stream, dtype, residual_in, y, 1.f, post_gain, branch_scale, next_gain, next_scale, epsilon, residual_out, h, tokens, k_in);
  if (st != MUI_OK) return st;
  return mui_linear_f32(stream, dtype, weights, h, bias, out, n_out, k_in, tokens);
}
