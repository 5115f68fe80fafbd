// Latent attention of one new token per row in one launch: what latent_attention.hip does in four (prepare, absorb, decode, output), for caches that are
// short. One workgroup per head and row:
//   q' = Wuk_h^T q_h,  score_s = (q' . c_s + rot(q_h) . r_s) scale,  out_h = Wuv_h (sum_s softmax_s c_s)
// all in fp32 but for the stored rows. The new token's latent row and rotated key part come from the down projection's output where the layer keeps its own: every workgroup makes
// them for itself (they are one of its keys), the first head's writes them to the cache.
//
// Eight waves; a lane owns eight of the kv_rank columns, so that a row of Wuk, Wuv or the cache is one load instruction of a wave, 1 KB: wave w takes rows w, w + 8, ..
// of the matrices and keys w, w + 8, .. . Both matrices (256 KB at rank 512 and 128 + 128 rows) and the first keys are requested before anything is used: what bounds it is what a CU takes in
// (about 45 KB a microsecond), and so the keys' part ends where their rows weigh as much as the matrices (256 keys of 1.1 KB): longer caches are split over workgroups by the launches apart,
// whose other three are 3 to 4 us each whatever they do. Nor are there more workgroups than CUs: a second round would repeat the first one's wait. us in bf16 as captured, latent rank
// 512, heads of 128 + 64 and 128; apart (attention + prepare) / here:
//              61 keys                      256 keys
//   1 row      16 heads 19.6 / 12.5         16 heads 20.0 / 17.9, 32 heads 21.4 / 18.0
//   8 rows     32 heads 25.9 / 12.5         32 heads 26.3 / 18.0 (16 heads, 156 keys: 23.2 / 15.9)
// (attention alone; with what is around it, and at other ranks, MuiLatentAttention has the line.)
// A sum per key over the wave and an exponential in every lane made 256 keys 19.5: the eight keys of a batch are reduced together, a key per two lanes.
#include "hybrid.cuh"

namespace mui {

struct LatentStep {
  const uint16_t* w_uv;
  const uint16_t* kv;  // [rows, kv_pitch]: latent row | key part to rotate, as projected; null: the caches hold the new token
  long kv_pitch;
  const uint16_t* kv_gain;
  const double* inv_freq;
  uint16_t *c_cache, *r_cache;
  long c_batch, r_batch;
  uint16_t* out;  // [rows, heads * vdim]
  int heads, dim, rot, vdim, kv_rank, window, max_cache_len;
  float scale, eps;
};

constexpr int kLsThreads = 512, kLsWaves = 8, kLsRank = 512, kLsRows = 128, kLsRot = 64, kLsKeys = 256;
constexpr int kLsPer = kLsRows / kLsWaves, kLsBatch = 8;  // matrix rows of a wave; keys of a wave at a time

// q: [rows, heads * (dim + rot)], not rotated
template <typename T>
__global__ void __launch_bounds__(kLsThreads, 1) latent_step_kernel(const int64_t* cache_position, const int64_t* row_start, const uint16_t* q, const uint16_t* w_uk,
                                                                    const LatentStep p) {
  __shared__ float qs[kLsRows + kLsRot], cs[2][kLsRot / 2];     // the head's query, its last part rotated below; cosines, sines
  __shared__ __align__(16) float part[kLsWaves][kLsRank], row[kLsRank];  // partial rows of the waves; their sum
  __shared__ float ml[kLsWaves][2];
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int h = blockIdx.x, b = blockIdx.y, hd = p.dim + p.rot, half = p.rot >> 1;
  const long pos = cache_position[0], first = row_start ? row_start[b] : 0;
  const int c0 = lane * 8, col = c0 < p.kv_rank ? c0 : 0;  // this lane's columns (past the end: the first ones, met by zeros)
  const bool there = c0 < p.kv_rank;

  // ---- requests, in the order of use
  const float qv = T::one(q[((long)b * p.heads + h) * hd + (t < hd ? t : 0)]);
  const double freq = p.inv_freq[t < half ? t : 0];
  u32x4 nc = {0u, 0u, 0u, 0u}, ng = nc, nu = nc, nw = nc;  // the new token's latent row, its gain, the two halves of its key part
  const bool own = p.kv != nullptr;
  const int j0 = (lane & 7) * 8, i0 = j0 < half ? j0 : (j0 < p.rot ? j0 - half : 0);
  if (own) {
    const uint16_t* kv = p.kv + (long)b * p.kv_pitch;
    nc = ld16(kv + col);
    ng = ld16(p.kv_gain + col);
    nu = ld16(kv + p.kv_rank + i0);
    nw = ld16(kv + p.kv_rank + half + i0);
  }
  const uint16_t* wk = w_uk + (long)h * p.dim * p.kv_rank + col;
  u32x4 uk[kLsPer], uv[kLsPer];
#pragma unroll
  for (int i = 0; i < kLsPer; ++i) {
    const int d = wave + kLsWaves * i;
    uk[i] = ld16_stream(wk + (long)(d < p.dim ? d : 0) * p.kv_rank);
  }
  // visible slots lo .. hi; key n of this wave is slot lo + wave + 8 n
  long hi = pos < p.max_cache_len ? pos : p.max_cache_len - 1, lo = p.window > 0 ? hi - p.window + 1 : 0;
  lo = lo > first ? lo : first;
  lo = lo > 0 ? lo : 0;
  const int keys = hi >= lo ? (int)(hi - lo) + 1 : 0;
  const long stored = own && hi == pos ? hi - 1 : hi;  // the last one that is read from the cache
  const uint16_t *cc = p.c_cache + b * p.c_batch + col, *rc = p.r_cache + b * p.r_batch;
  struct Keys { u32x4 c[kLsBatch], r; } ks;  // r: lane 8 j + i has chunk i of key j
  auto slot_of = [&](int n) {
    long s = lo + wave + kLsWaves * n;
    s = s < stored ? s : stored;
    return s > 0 ? s : 0;
  };
  auto request = [&](int n0) {
    Keys k;
#pragma unroll
    for (int j = 0; j < kLsBatch; ++j) k.c[j] = ld16(cc + slot_of(n0 + j) * p.kv_rank);
    k.r = ld16(rc + slot_of(n0 + (lane >> 3)) * p.rot + (j0 < p.rot ? j0 : 0));
    return k;
  };
  ks = request(0);
  const uint16_t* wv = p.w_uv + (long)h * p.vdim * p.kv_rank + col;
#pragma unroll
  for (int i = 0; i < kLsPer; ++i) {
    const int v = wave + kLsWaves * i;
    uv[i] = ld16_stream(wv + (long)(v < p.vdim ? v : 0) * p.kv_rank);
  }
  asm volatile("" ::: "memory");  // (nothing is asked for later)

  // ---- the query, the angles
  if (t < kLsRows + kLsRot) qs[t] = t < hd ? qv : 0.f;
  if (t < half) {
    const long at = pos - first;
    rope_angle((double)(at > 0 ? at : 0), freq, cs[0][t], cs[1][t]);
  }
  __syncthreads();
  // this lane's chunk of the rotated query and of the new key (both rounded as they are stored), chunk lane % 8
  float qr[8], kr[8], f[8], g[8];
  auto turned = [&](const float (&u)[8], const float (&w)[8], float (&o)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float co = cs[0][i0 + e], si = cs[1][i0 + e];
      o[e] = j0 < half ? u[e] * co - w[e] * si : w[e] * co + u[e] * si;
    }
    const u32x4 rounded = pack8<T>(o);
    unpack8<T>(rounded, o);
    return rounded;
  };
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    f[e] = qs[p.dim + i0 + e];
    g[e] = qs[p.dim + half + i0 + e];
  }
  turned(f, g, qr);
  unpack8<T>(nu, f);
  unpack8<T>(nw, g);
  const u32x4 new_r = turned(f, g, kr);
  // the new latent row: normed by every wave for itself, rounded as it is stored
  u32x4 new_c = {0u, 0u, 0u, 0u};
  if (own) {
    unpack8<T>(nc, f);
    unpack8<T>(ng, g);
    float sq = 0.f;
    if (there)
#pragma unroll
      for (int e = 0; e < 8; ++e) sq = fmaf(f[e], f[e], sq);
    const float rs = rsqrtf(wave_sum(sq) / (float)p.kv_rank + p.eps);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] *= f[e] * rs;
    new_c = pack8<T>(g);
    if (h == 0 && wave == 0 && pos >= 0 && pos < p.max_cache_len) {
      if (there) *(u32x4*)(p.c_cache + b * p.c_batch + pos * p.kv_rank + c0) = new_c;
      if (lane < 8 && j0 < p.rot) *(u32x4*)(p.r_cache + b * p.r_batch + pos * p.rot + j0) = new_r;
    }
  }

  // ---- q' = Wuk^T q
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
#pragma unroll
  for (int i = 0; i < kLsPer; ++i) {
    const int d = wave + kLsWaves * i;
    const float qd = d < p.dim ? qs[d] : 0.f;
    unpack8<T>(uk[i], f);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = fmaf(f[e], qd, acc[e]);
  }
  auto meet = [&]() {  // part: the waves' rows
    *(f32x4*)&part[wave][c0] = f32x4{acc[0], acc[1], acc[2], acc[3]};
    *(f32x4*)&part[wave][c0 + 4] = f32x4{acc[4], acc[5], acc[6], acc[7]};
  };
  meet();
  __syncthreads();
  {
    float a = part[0][t];
#pragma unroll
    for (int w = 1; w < kLsWaves; ++w) a += part[w][t];
    row[t] = t < p.kv_rank ? a * (p.scale * 1.4426950408889634f) : 0.f;
  }
  __syncthreads();
  float qa[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    qa[e] = row[c0 + e];
    qr[e] *= p.scale * 1.4426950408889634f;
    acc[e] = 0.f;
  }

  // ---- this wave's keys, eight at a time, with a running maximum
  float m = -1e30f, l = 0.f;
  const int newest = own && hi == pos ? keys - 1 : -1;  // (key of the wave newest % 8)
  for (int n0 = 0; wave + kLsWaves * n0 < keys; n0 += kLsBatch) {  // uniform for the wave
    Keys k = ks;
    if (wave + kLsWaves * (n0 + kLsBatch) < keys) ks = request(n0 + kLsBatch);
    // the rotated part: eight keys at once, eight lanes each
    unpack8<T>(k.r, f);
    if (wave + kLsWaves * (n0 + (lane >> 3)) == newest)
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = kr[e];
    float rr = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) rr = fmaf(f[e], qr[e], rr);
    rr = j0 < p.rot ? rr : 0.f;
    rr += dpp_f32<kDppXor1>(rr);
    rr += dpp_f32<kDppXor2>(rr);
    rr += dpp_f32<kDppHalfMirror>(rr);
    // the latent parts: every row of sixteen lanes sums key (lane % 16) / 2 over its columns
    float s[kLsBatch];
#pragma unroll
    for (int j = 0; j < kLsBatch; ++j) {
      const int n = wave + kLsWaves * (n0 + j);
      if (n == newest) k.c[j] = new_c;
      else if (n >= keys) k.c[j] = u32x4{0u, 0u, 0u, 0u};  // (a slot that nobody has written may hold anything)
      unpack8<T>(k.c[j], f);
      float a = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) a = fmaf(f[e], qa[e], a);
      s[j] = there ? a : 0.f;
    }
    static_assert(kLsBatch == 8, "a key per two lanes of sixteen");
    row16_reduce_scatter<8>(s, lane);
    const int mine = (lane & 15) >> 1;
    float sc = s[0] + __shfl_xor(s[0], 16);
    sc += __shfl_xor(sc, 32);
    sc += __shfl(rr, 8 * mine);
    sc = wave + kLsWaves * (n0 + mine) < keys ? sc : -INFINITY;
    const float mn = fmaxf(m, readlane_f32(row16_max(sc), 0)), keep = exp2f(m - mn), pm = exp2f(sc - mn);
    l = fmaf(l, keep, pm);  // (lane by lane, every key in two of them)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= keep;
#pragma unroll
    for (int j = 0; j < kLsBatch; ++j) {
      const float pj = readlane_f32(pm, 2 * j);
      unpack8<T>(k.c[j], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(pj, f[e], acc[e]);
    }
    m = mn;
  }
  l = 0.5f * row16_sum(l);
  meet();
  if (lane == 0) {
    ml[wave][0] = m;
    ml[wave][1] = l;
  }
  __syncthreads();
  {
    float mm = ml[0][0], ll = 0.f, a = 0.f;
#pragma unroll
    for (int w = 1; w < kLsWaves; ++w) mm = fmaxf(mm, ml[w][0]);
#pragma unroll
    for (int w = 0; w < kLsWaves; ++w) {
      const float e = ml[w][1] > 0.f ? exp2f(ml[w][0] - mm) : 0.f;  // (a wave without keys)
      ll = fmaf(e, ml[w][1], ll);
      a = fmaf(e, part[w][t], a);
    }
    row[t] = ll > 0.f && t < p.kv_rank ? a / ll : 0.f;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 8; ++e) qa[e] = row[c0 + e];

  // ---- out = Wuv (..)
  float o[kLsPer];
#pragma unroll
  for (int i = 0; i < kLsPer; ++i) {
    unpack8<T>(uv[i], f);
    o[i] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[i] = fmaf(f[e], qa[e], o[i]);
  }
  static_assert(kLsPer == 16, "a value per lane of sixteen");
  row16_reduce_scatter<16>(o, lane);  // lane i of sixteen: value i over its sixteen lanes
  float v = o[0];
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  const int vr = wave + kLsWaves * (lane & 15);
  if (lane < 16 && vr < p.vdim) p.out[((long)b * p.heads + h) * p.vdim + vr] = T::pack(v);
}

static bool latent_step_serves(int dtype, int batch, int heads, int dim, int rot, int vdim, int kv_rank, int span) {
  if (dtype != MUI_DTYPE_F16 && dtype != MUI_DTYPE_BF16) return false;
  if (batch < 1 || heads < 1 || dim < 1 || vdim < 1 || kv_rank < 8 || span < 1) return false;
  return dim <= kLsRows && vdim <= kLsRows && kv_rank <= kLsRank && kv_rank % 8 == 0 && rot >= 16 && rot <= kLsRot && rot % 16 == 0 && span <= kLsKeys &&
         (long)batch * heads <= device_cus();
}

}  // namespace mui

using namespace mui;

extern "C" int mui_latent_step_serves(int dtype, int batch, int heads, int dim, int rot_dim, int vdim, int kv_rank, int window, int max_cache_len) {
  return latent_step_serves(dtype, batch, heads, dim, rot_dim, vdim, kv_rank, window > 0 && window < max_cache_len ? window : max_cache_len);
}

extern "C" int mui_latent_step(mui_stream_t stream, int dtype, const void* q, const void* w_uk, const void* w_uv, const void* kv, long kv_pitch, const void* kv_gain, float epsilon,
                               const double* inv_freq, void* c_cache, long c_batch_stride, void* r_cache, long r_batch_stride, const int64_t* cache_position,
                               const int64_t* row_start, float scale, int window, void* out, int batch, int heads, int dim, int rot_dim, int vdim, int kv_rank, int max_cache_len) {
  MUI_CHECK_ARG(q && w_uk && w_uv && c_cache && r_cache && cache_position && out && max_cache_len > 0 && (!kv || kv_gain) && inv_freq);
  MUI_CHECK_ARG(!kv || kv_pitch >= kv_rank + rot_dim);
  if (!mui_latent_step_serves(dtype, batch, heads, dim, rot_dim, vdim, kv_rank, window, max_cache_len)) return MUI_ERR_UNSUPPORTED;
  if (!aligned16(w_uk) || !aligned16(w_uv) || !aligned16(c_cache) || !aligned16(r_cache) || c_batch_stride % 8 || r_batch_stride % 8) return MUI_ERR_ALIGNMENT;
  if (kv && (!aligned16(kv) || !aligned16(kv_gain) || kv_pitch % 8)) return MUI_ERR_ALIGNMENT;
  LatentStep p = {};
  p.w_uv = (const uint16_t*)w_uv; p.kv = (const uint16_t*)kv; p.kv_pitch = kv_pitch; p.kv_gain = (const uint16_t*)kv_gain; p.inv_freq = inv_freq;
  p.c_cache = (uint16_t*)c_cache; p.r_cache = (uint16_t*)r_cache; p.c_batch = c_batch_stride; p.r_batch = r_batch_stride; p.out = (uint16_t*)out;
  p.heads = heads; p.dim = dim; p.rot = rot_dim; p.vdim = vdim; p.kv_rank = kv_rank; p.window = window; p.max_cache_len = max_cache_len; p.scale = scale; p.eps = epsilon;
  const dim3 grid(heads, batch), block(kLsThreads);
  if (dtype == MUI_DTYPE_F16)
    hipLaunchKernelGGL((latent_step_kernel<F16>), grid, block, 0, (hipStream_t)stream, cache_position, row_start, (const uint16_t*)q, (const uint16_t*)w_uk, p);
  else
    hipLaunchKernelGGL((latent_step_kernel<BF16>), grid, block, 0, (hipStream_t)stream, cache_position, row_start, (const uint16_t*)q, (const uint16_t*)w_uk, p);
  return launch_status();
}
