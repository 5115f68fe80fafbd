// Mixture-of-experts feed-forward: routing, grouping of the chosen (token, expert) pairs by expert, and
// the experts' two matrix products over the groups.
//
//   logits   fp32 [tokens, outputs]  (linear_f32 below; also the gates of recurrent layers)
//   route    s = softmax(logits); the `top` outputs with the largest s + correction are chosen, weighted
//            by their s. Outputs >= n_experts are identity experts: they take part in the choice and are
//            added by mui_moe_residual_norm, no product is computed for them.
//   group    pairs sorted by expert, cut into tiles of at most `tile_pairs` pairs of ONE expert
//   gateup   act[pair] = a(G_e x, U_e x), a(g, u) = g' sigmoid(1.702 g') (u' + 1) with g' = min(g, limit),
//            u' = clamp(u, -limit, limit)
//   down     out[pair] = D_e act[pair]
//
// Everything stays on the device (no counts travel to the host): the grids cover the largest possible
// number of tiles and workgroups without one leave at once, so a captured decode step replays whatever
// the routing does.
//
// Products, wave64 v_mfma_f32_16x16x32 (weights = A rows, pairs = B columns):
//   tile 16   up to 16 pairs of an expert: 16 gate + 16 up rows (or 32 rows) at a time by a workgroup, K dealt out to
//             its four waves, rows in runs of 256 bytes through LDS. Decode and short
//             prompts: every chosen expert's weights are streamed once.
//   tile 128 / 256   as many pairs x as many rows, both operands through swizzled LDS stages filled by
//             LDS-direct loads; waves of 64 x 64, or of 128 x 64 with operands read a half step ahead.
// fp32 models and sizes that are no multiple of 8 take a plain one-wave-per-output kernel.
#include "skinny.cuh"

namespace mui {

enum { MOE_GATEUP = 0, MOE_DOWN = 1, MOE_F32 = 2 };

struct MoeTile { int expert, first, count, pad; };

__device__ __forceinline__ float moe_act(float g, float u, float limit) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.0f + __expf(-1.702f * g)) * (u + 1.0f);
}

template <typename T>
__device__ __forceinline__ float moe_dot2(uint32_t a, uint32_t b, float c);
template <>
__device__ __forceinline__ float moe_dot2<F16>(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
}
typedef __bf16 bf16x2_moe __attribute__((ext_vector_type(2)));
template <>
__device__ __forceinline__ float moe_dot2<BF16>(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_moe, a), __builtin_bit_cast(bf16x2_moe, b), c, false);
}

// ---------------------------------------------------------------------------------------
// fp32 outputs of a small matrix: y[t, n] = W[n, :] . x[t, :] + bias[n], one workgroup per row
// ---------------------------------------------------------------------------------------
template <typename T, bool VEC, int TB>  // TB tokens per pass over a row
__global__ void __launch_bounds__(256) linear_f32_rows_kernel(const typename T::storage* w, const typename T::storage* x,
                                                              const typename T::storage* bias, float* y, int n, int k,
                                                              int tokens) {
  __shared__ float red[4][TB];
  const int t = threadIdx.x, row = blockIdx.x;
  const typename T::storage* wr = w + (long)row * k;
  const float add = bias ? T::one(bias[row]) : 0.f;
  for (int t0 = blockIdx.y * TB; t0 < tokens; t0 += gridDim.y * TB) {
    float acc[TB];
#pragma unroll
    for (int j = 0; j < TB; ++j) acc[j] = 0.f;
    if constexpr (VEC) {
#pragma unroll 2
      for (int c = t * 8; c < k; c += 256 * 8) {
        float wf[8];
        load8<T>(wr + c, wf);
#pragma unroll
        for (int j = 0; j < TB; ++j) {
          const int tk = t0 + j < tokens ? t0 + j : tokens - 1;
          float xf[8];
          load8<T>(x + (long)tk * k + c, xf);
#pragma unroll
          for (int i = 0; i < 8; ++i) acc[j] = fmaf(wf[i], xf[i], acc[j]);
        }
      }
    } else {
      for (int c = t; c < k; c += 256) {
        const float wf = T::one(wr[c]);
#pragma unroll
        for (int j = 0; j < TB; ++j) {
          const int tk = t0 + j < tokens ? t0 + j : tokens - 1;
          acc[j] = fmaf(wf, T::one(x[(long)tk * k + c]), acc[j]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < TB; ++j) {
      const float s = wave_sum(acc[j]);
      if ((t & 63) == 0) red[t >> 6][j] = s;
    }
    __syncthreads();
    if (t < TB && t0 + t < tokens)
      y[(long)(t0 + t) * n + row] = ((red[0][t] + red[1][t]) + (red[2][t] + red[3][t])) + add;
    __syncthreads();
  }
}

// One token, with the boundary in front (gemv_join.hip): every row's workgroup computes that for itself; x is the sublayer's output
template <typename T, int CH>
__global__ void __launch_bounds__(256) linear_f32_join_kernel(const uint16_t* x, const uint16_t* w, const uint16_t* bias, float* y, int k, float eps, const BoundaryInFront front) {
  __shared__ float red[4], red_join[2][4];
  const int t = threadIdx.x, row = blockIdx.x;
  int at[CH];
  bool valid[CH];
  u32x4 xq[CH], wq[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int c = (t + 256 * j) * 8;
    valid[j] = c < k;
    at[j] = valid[j] ? c : 0;
    xq[j] = ld16(x + at[j]);
  }
  FrontOperands<T, CH> ahead;
  ahead.request(front, x, at);
#pragma unroll
  for (int j = 0; j < CH; ++j) wq[j] = ld16(w + (long)row * k + at[j]);
  ahead.finish(front, xq, valid, at, k, eps, red_join, row == 0);
  float acc = 0.f;
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    float wf[8], xf[8];
    unpack8<T>(wq[j], wf);
    unpack8<T>(xq[j], xf);
    if (valid[j])
#pragma unroll
      for (int i = 0; i < 8; ++i) acc = fmaf(wf[i], xf[i], acc);
  }
  acc = wave_sum(acc);
  if ((t & 63) == 0) red[t >> 6] = acc;
  __syncthreads();
  if (t == 0) y[row] = ((red[0] + red[1]) + (red[2] + red[3])) + (bias ? T::one(bias[row]) : 0.f);
}

template <typename T>
static int launch_linear_f32_join_t(hipStream_t s, const void* w, const void* x, const void* bias, float* y, int n, int k, float eps, const BoundaryInFront& front) {
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(n), dim3(256), 0, s, (const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, y, k, eps, front);
    return launch_status();
  };
  // every row repeats the boundary, 24 KB from L2 at 4096: for as many as fill the chip once
  if (n > device_cus() || k > 4 * 256 * 8) return MUI_ERR_UNSUPPORTED;
  if (k <= 256 * 8) return launch(linear_f32_join_kernel<T, 1>);
  if (k <= 2 * 256 * 8) return launch(linear_f32_join_kernel<T, 2>);
  return launch(linear_f32_join_kernel<T, 4>);
}
int launch_linear_f32_join(hipStream_t s, int dtype, const void* w, const void* x, const void* bias, float* y, int n, int k, float eps, const BoundaryInFront& front) {
  if (dtype == MUI_DTYPE_F16) return launch_linear_f32_join_t<F16>(s, w, x, bias, y, n, k, eps, front);
  if (dtype == MUI_DTYPE_BF16) return launch_linear_f32_join_t<BF16>(s, w, x, bias, y, n, k, eps, front);
  return MUI_ERR_UNSUPPORTED;
}

// ---------------------------------------------------------------------------------------
// routing
// ---------------------------------------------------------------------------------------
constexpr int kMaxRouter = 1024;   // router outputs
constexpr int kRouteThreads = 1024;  // at most; few tokens take fewer
constexpr int kRouterPerLane = kMaxRouter / kWave;

// one token by one wave
template <typename T>
__device__ __forceinline__ void route_token(const float* lg, const typename T::storage* corr, int n_out, int top,
                                            int lane, int32_t* expert, float* weight, int* expert_lds = nullptr) {
  float s[kRouterPerLane], choice[kRouterPerLane], add[kRouterPerLane];  // add: requested with the logits
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < kRouterPerLane; ++i) {
    const int e = lane + kWave * i;
    s[i] = e < n_out ? lg[e] : -INFINITY;
    add[i] = corr && e < n_out ? T::one(corr[e]) : 0.f;
    mx = fmaxf(mx, s[i]);
    if (kWave * (i + 1) >= n_out) break;
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kRouterPerLane; ++i) {
    s[i] = expf(s[i] - mx);
    sum += s[i];
    if (kWave * (i + 1) >= n_out) break;
  }
  sum = wave_sum(sum);
#pragma unroll
  for (int i = 0; i < kRouterPerLane; ++i) {
    const int e = lane + kWave * i;
    s[i] = s[i] / sum;
    choice[i] = e < n_out ? s[i] + add[i] : -INFINITY;
    if (kWave * (i + 1) >= n_out) break;
  }
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY, bs = 0.f;
    int bi = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < kRouterPerLane; ++i) {
      const int e = lane + kWave * i;
      if (choice[i] > best) { best = choice[i]; bi = e; bs = s[i]; }
      if (kWave * (i + 1) >= n_out) break;
    }
    // the wave's largest, the lowest index where several lanes hold it
    const float top_v = wave_max(best);
    uint64_t holders = __ballot(best == top_v && bi < n_out);
    int win = 0x7fffffff;
    float win_s = 0.f;
    while (holders) {
      const int l = __ffsll((unsigned long long)holders) - 1;
      const int li = __builtin_amdgcn_readlane(bi, l);
      if (li < win) {
        win = li;
        win_s = readlane_f32(bs, l);
      }
      holders &= holders - 1;
    }
    bi = win < n_out ? win : 0;  // nothing left to choose (NaN logits): stays in range
    bs = win_s;
#pragma unroll
    for (int i = 0; i < kRouterPerLane; ++i) {
      if (lane + kWave * i == bi) choice[i] = -INFINITY;
      if (kWave * (i + 1) >= n_out) break;
    }
    if (lane == 0) {
      expert[j] = bi;
      weight[j] = bs;
      if (expert_lds) expert_lds[j] = bi;
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256) moe_route_kernel(const float* logits, const typename T::storage* corr, int n_out,
                                                        int top, int tokens, int32_t* expert, float* weight) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t < tokens)
    route_token<T>(logits + (long)t * n_out, corr, n_out, top, threadIdx.x & (kWave - 1), expert + (long)t * top,
                   weight + (long)t * top);
}

// One workgroup: (ROUTE: the routing of all tokens, then) count per expert, cut into tiles, scatter.
// tiles[0].count = number of tiles, tiles[0].pad: some expert has several; tiles[1 + i] the i-th tile, unused entries up to max_tiles get count 0.
constexpr int kChosen = 1024;
template <typename T, bool ROUTE>
__global__ void __launch_bounds__(kRouteThreads) moe_group_kernel(const float* logits, const typename T::storage* corr,
                                                                  int n_out, int n_experts, int top, int tokens,
                                                                  int tile_pairs, int max_tiles, int32_t* expert,
                                                                  float* weight, int32_t* pairs, MoeTile* tiles) {
  __shared__ int count[kMaxRouter], cursor[kMaxRouter], first_tile[kMaxRouter];
  __shared__ int n_tiles_s;
  __shared__ int chosen[ROUTE ? kChosen : 1];  // the routing's result without the way through memory
  const int t = threadIdx.x, nt_threads = blockDim.x;
  const int n_pairs = tokens * top;
  for (int e = t; e < n_experts; e += nt_threads) count[e] = 0;
  if constexpr (ROUTE) {
    for (int tk = t >> 6; tk < tokens; tk += nt_threads / kWave)
      route_token<T>(logits + (long)tk * n_out, corr, n_out, top, t & (kWave - 1), expert + (long)tk * top,
                     weight + (long)tk * top, n_pairs <= kChosen ? chosen + tk * top : nullptr);
    __threadfence_block();
  }
  auto expert_of = [&](int i) {
    if constexpr (ROUTE) return n_pairs <= kChosen ? chosen[i] : expert[i];
    else return expert[i];
  };
  __syncthreads();
  for (int i = t; i < n_pairs; i += nt_threads) {
    const int e = expert_of(i);
    if (e < n_experts) atomicAdd(&count[e], 1);
  }
  __syncthreads();
  if (t < kWave) {  // exclusive sums over experts: 64 at a time by one wave
    int pair_base = 0, tile_base = 0;
    for (int e0 = 0; e0 < n_experts; e0 += kWave) {
      const int e = e0 + t;
      const int c = e < n_experts ? count[e] : 0;
      const int nt = (c + tile_pairs - 1) / tile_pairs;
      int sc = c, st = nt;
#pragma unroll
      for (int d = 1; d < kWave; d <<= 1) {
        const int oc = __shfl_up(sc, d), ot = __shfl_up(st, d);
        if (t >= d) { sc += oc; st += ot; }
      }
      if (e < n_experts) {
        cursor[e] = pair_base + sc - c;
        first_tile[e] = tile_base + st - nt;
      }
      pair_base += __shfl(sc, kWave - 1);
      tile_base += __shfl(st, kWave - 1);
    }
    if (t == 0) n_tiles_s = tile_base < max_tiles ? tile_base : max_tiles;
  }
  // whether an expert has several tiles
  int several = 0;
  for (int e = t; e < n_experts; e += nt_threads) several |= count[e] > tile_pairs;
  several = __syncthreads_or(several);
  const int n_tiles = n_tiles_s;
  for (int e = t; e < n_experts; e += nt_threads) {
    const int c = count[e], base = cursor[e], ft = first_tile[e];
    for (int i = 0; i * tile_pairs < c && ft + i < max_tiles; ++i) {
      const int left = c - i * tile_pairs;
      tiles[1 + ft + i] = MoeTile{e, base + i * tile_pairs, left < tile_pairs ? left : tile_pairs, 0};
    }
  }
  for (int i = n_tiles + t; i < max_tiles; i += nt_threads) tiles[1 + i] = MoeTile{0, 0, 0, 0};
  if (t == 0) tiles[0] = MoeTile{0, 0, n_tiles, several != 0};
  __syncthreads();  // cursors are read above before they move
  for (int i = t; i < n_pairs; i += nt_threads) {
    const int e = expert_of(i);
    if (e < n_experts) pairs[atomicAdd(&cursor[e], 1)] = i;
  }
}

// ---------------------------------------------------------------------------------------
// products
// ---------------------------------------------------------------------------------------
struct MoeGemmParams {
  const uint16_t* w0;   // gate / down / matrix: [experts, n, k]
  const uint16_t* w1;   // up
  long expert_stride;   // elements between experts (w0 and w1)
  const uint16_t* x;    // gateup, f32: [tokens, k]; down: [pairs, k]
  const uint16_t* bias; // f32: [n] or null
  void* y;              // gateup: [pairs, n] 16-bit; down: [pairs, n] 16-bit; f32: [tokens, n] fp32
  const int32_t* pairs; // sorted pairs, null: pair i is i (f32)
  const MoeTile* tiles;
  int n, k, top, tokens;
  float limit;
  int max_tiles;
  bool once;            // gate and up of the layer are too large to be found in the memory-side cache at the next call
};

__device__ __forceinline__ MoeTile moe_tile_at(const MoeGemmParams& p, int i, int tile_pairs) {
  if (p.tiles) return p.tiles[1 + i];
  const int first = i * tile_pairs, left = p.tokens - first;
  return MoeTile{0, first, left < 0 ? 0 : (left < tile_pairs ? left : tile_pairs), 0};
}

// Weight rows reach LDS (a private area per wave, two stages) in runs of 256 bytes by LDS-direct loads and are
// read back as operands: 16 rows x 128 k-values per tile and stage, rows of 256 bytes whose 16-byte chunk c
// lives at chunk c ^ row. Loaded straight in operand order (64 bytes of 16 rows per instruction) the same
// bytes arrive at about two thirds of the rate.
// What a workgroup needs first stands in front of p as scalars: the first 16 dwords of a kernel's scalar arguments are in registers when a wave starts (the compiler's
// kernarg preload, which a struct does not get), the rest comes with a load of its own.
constexpr int kT16Seg = 128;
template <typename T, int EPI>
__global__ void __launch_bounds__(256, 2) moe_tile16_kernel(const MoeTile* tiles, const uint16_t* w0, const uint16_t* w1, long expert_stride, int n, int k, int max_tiles,
                                                            int once, const int32_t* pairs, const uint16_t* x, MoeGemmParams p) {
  p.tiles = tiles; p.w0 = w0; p.w1 = w1; p.expert_stride = expert_stride; p.n = n; p.k = k; p.max_tiles = max_tiles; p.once = once; p.pairs = pairs; p.x = x;
  constexpr int ROWS = EPI == MOE_GATEUP ? 16 : 32;  // outputs per workgroup
  // [wave][tile]; the stages are arrays of their own, so that the compiler can tell which loads a read waits for
  __shared__ __align__(16) uint16_t wl0[4][2][16 * kT16Seg], wl1[4][2][16 * kT16Seg];
  __shared__ int prow[16];
  MoeTile tile;
  // Gate and up rows that only this tile reads, in this call and the next, are requested non-temporally: 38.6 -> 36.8 us for 1 token, 8 of 64 experts of
  // 1792 x 4096 (the down product gained nothing here). An expert's further tiles find the rows in L2 only if they are requested
  // ordinarily: 95 tokens that favour 20 of the experts 180 us, 225 with all rows non-temporal.
  bool alone = false;
  if constexpr (EPI == MOE_GATEUP) {
    // (entries requested together: tile i is entry i + 1, entry 0 holds their count)
    const int i = (int)blockIdx.y, count = p.tiles[0].count, before = p.tiles[i].expert, behind = p.tiles[i + 1 < p.max_tiles ? i + 2 : i + 1].expert;
    tile = p.tiles[1 + i];
    alone = p.once & ((i == 0) | (before != tile.expert)) & ((i + 1 >= count) | (behind != tile.expert));
  } else {
    tile = moe_tile_at(p, blockIdx.y, 16);
  }
  if (tile.count <= 0) return;
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int o0 = blockIdx.x * ROWS;
  if (t < 16) {
    const int i = tile.first + (t < tile.count ? t : 0);
    prow[t] = p.pairs ? p.pairs[i] : i;
  }
  const int mine = tile.first + (r16 < tile.count ? r16 : 0);
  const int pair = p.pairs ? p.pairs[mine] : mine;
  const uint16_t* xr = p.x + (long)(EPI == MOE_GATEUP ? pair / p.top : pair) * p.k;
  const long eb = (long)tile.expert * p.expert_stride;
  // load instruction q of a tile: rows 4 q + lane / 16, this lane's logical chunk of the row
  const uint16_t* src[2][4];
  int chunk[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = 4 * q + g;
    chunk[q] = (r16 ^ r) * 8;
    const int ra = o0 + r < p.n ? o0 + r : p.n - 1;
    const int rb = EPI == MOE_GATEUP ? ra : (o0 + 16 + r < p.n ? o0 + 16 + r : p.n - 1);
    src[0][q] = p.w0 + eb + (long)ra * p.k;
    src[1][q] = (EPI == MOE_GATEUP ? p.w1 : p.w0) + eb + (long)rb * p.k;
  }
  f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  const int segs = (p.k + kT16Seg - 1) / kT16Seg;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  // segment s into a stage (past the last one: the first again, into a stage nobody reads); chunks past
  // the end of a row read its start and meet x = 0
  auto issue = [&](auto stream, int s, uint16_t (&wl)[4][2][16 * kT16Seg], u32x4 (&x)[4]) {
    const int k0 = s < segs ? s * kT16Seg : 0;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int kk = k0 + chunk[q];
        const uint16_t* from = src[j][q] + (kk < p.k ? kk : 0);
        if constexpr (decltype(stream)::value) load_lds16_stream(from, &wl[wave][j][q * 4 * kT16Seg]);
        else load_lds16(from, &wl[wave][j][q * 4 * kT16Seg]);
      }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int kk = k0 + 32 * u + 8 * g;
      x[u] = ld16(xr + (kk < p.k ? kk : 0));
    }
  };
  auto multiply = [&](int s, const uint16_t (&wl)[4][2][16 * kT16Seg], const u32x4 (&x)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const u32x4 xv = s * kT16Seg + 32 * u + 8 * g < p.k ? x[u] : zero;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[j] = mfma16x16x32<T>(*(const u32x4*)&wl[wave][j][r16 * kT16Seg + ((4 * u + g) ^ r16) * 8], xv, acc[j]);
    }
  };
  u32x4 x0[4], x1[4];
  auto run = [&](auto stream) {
    issue(stream, wave, wl0, x0);
    for (int s = wave; s < segs; s += 8) {
      issue(stream, s + 4, wl1, x1);
      wait_loads<12>();  // everything but the newest segment has landed
      multiply(s, wl0, x0);
      if (s + 4 >= segs) break;
      issue(stream, s + 8, wl0, x0);
      wait_loads<12>();
      multiply(s + 4, wl1, x1);
    }
  };
  if (wave < segs) {
    if (EPI == MOE_GATEUP && alone) run(std::integral_constant<bool, EPI == MOE_GATEUP>());
    else run(std::false_type());
  }
  wait_loads<0>();  // (no load is still on its way into LDS)
  __syncthreads();
  float(*red)[2][16][17] = (float(*)[2][16][17])wl0;
  static_assert(sizeof(wl0) >= sizeof(float) * 4 * 2 * 16 * 17, "the partial tiles fit where the weights were");
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    red[wave][0][4 * g + r][r16] = acc[0][r];
    red[wave][1][4 * g + r][r16] = acc[1][r];
  }
  __syncthreads();
  const int row = t & 15, col = t >> 4;
  float v0 = 0.f, v1 = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) { v0 += red[w][0][row][col]; v1 += red[w][1][row][col]; }
  if (col >= tile.count) return;
  const long out = (long)prow[col] * p.n;
  if constexpr (EPI == MOE_GATEUP) {
    if (o0 + row < p.n) ((uint16_t*)p.y)[out + o0 + row] = T::pack(moe_act(v0, v1, p.limit));
  } else if constexpr (EPI == MOE_DOWN) {
    if (o0 + row < p.n) ((uint16_t*)p.y)[out + o0 + row] = T::pack(v0);
    if (o0 + 16 + row < p.n) ((uint16_t*)p.y)[out + o0 + 16 + row] = T::pack(v1);
  } else {
    const int n0 = o0 + row, n1 = o0 + 16 + row;
    if (n0 < p.n) ((float*)p.y)[out + n0] = v0 + (p.bias ? T::one(p.bias[n0]) : 0.f);
    if (n1 < p.n) ((float*)p.y)[out + n1] = v1 + (p.bias ? T::one(p.bias[n1]) : 0.f);
  }
}

// The same tiles for K in whole segments (four at least), by a round of workgroups, two per CU, that take the units (tile, block of rows) blockIdx, blockIdx + grid, ..
// The segments run on across units: while a unit's partial tiles meet in LDS, the next one's first segment is on its way, and tiles that are not there cost nothing.
// A wave takes every fourth segment of its workgroup's units, counted through (so it has some of every unit): which of a unit's four runs of segments that is moves on from unit to
// unit where their number is no multiple of four. Partial tiles are kept by run and added in the order of the runs: a row's sums don't depend on where its tile stands. Rows go through registers to LDS: of a
// wave that has loads into LDS and loads into registers (the pairs' operands) under way the compiler waits for ALL where it needs one of the latter, and
// every second segment drained the wave.
// Bound by the weight stream (7.1 TB/s at best). Rows that only one unit reads, in this call and the next, are requested non-temporally, of down too: ordinarily
// 4096 x 1792, 8 / 50 tokens of 8 experts, 96 / 158 us, non-temporally 85 / 143. An expert's further tiles find the rows in L2 only if they are requested ordinarily; where
// there are any it is decided by unit (the branch costs 1 to 2 % of gate and up). us of gate and up / down, a workgroup per tile and block before -> now, 64
// experts: 4096 x 1792, 8 of them per token, 1 token 41.2 / 23.9 -> 39.2 / 20.6, 8 tokens 176.7 / 94.1 -> 169.8 / 85.4, 50 tokens 287 / 156 -> 273 / 143;
// 2048 x 1408, 6 per token, 1 token 17.1 / 10.3 -> 15.4 / 9.7, 8 tokens 67.8 / 36.7 -> 62.0 / 31.4, 50 tokens 125.9 / 66.5 -> 120 / 57.6. Three workgroups per CU: the same to 5 % more.
template <typename T, int EPI>
__global__ void __launch_bounds__(256, 2) moe_units_kernel(const MoeTile* tiles, const uint16_t* w0, const uint16_t* w1, long expert_stride, const int32_t* pairs, int n, int k,
                                                           const uint16_t* x, int top, int blocks, int max_tiles, int once, float limit, uint16_t* y) {
  constexpr int ROWS = EPI == MOE_GATEUP ? 16 : 32;  // outputs per unit
  __shared__ __align__(16) uint16_t wl[4][2][16 * kT16Seg];
  __shared__ float red[4][2][16][17];  // by run of segments
  typedef const __attribute__((address_space(4))) MoeTile ConstTile;
  ConstTile* list = (ConstTile*)(uintptr_t)tiles;
  const int grid = gridDim.x, units = list[0].count * blocks;
  if ((int)blockIdx.x >= units) return;
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int segs = k / kT16Seg;
  // how rows are requested: 0 ordinarily, 1 non-temporally, 2 by unit
  auto run = [&](auto how) {
    constexpr int HOW = decltype(how)::value;

    // a unit as the loads need it
    struct Unit { int id, o0, count, first; bool alone; const uint8_t *b0, *b1; };
    auto unit_at = [&](int id) {
      Unit u;
      u.id = id < units ? id : units - 1;  // (past the last: one that is there; what comes of it is not used)
      const int ti = u.id / blocks;
      u.o0 = (u.id - ti * blocks) * ROWS;
      const int expert = list[1 + ti].expert;
      u.first = list[1 + ti].first;
      u.count = list[1 + ti].count;
      if constexpr (HOW == 2) {
        const int before = list[ti].expert, behind = list[ti + 1 < max_tiles ? ti + 2 : ti + 1].expert;
        u.alone = (ti == 0 || before != expert) && (u.id + blocks >= units || behind != expert);
      } else {
        u.alone = HOW == 1;
      }
      const long at = (long)expert * expert_stride + (long)u.o0 * k;
      u.b0 = (const uint8_t*)(w0 + at);
      u.b1 = EPI == MOE_GATEUP ? (const uint8_t*)(w1 + at) : u.b0;
      return u;
    };
    auto pair_of = [&](const Unit& u) { return pairs + u.first + (r16 < u.count ? r16 : 0); };
    Unit lu = unit_at(blockIdx.x), nu = unit_at(blockIdx.x + grid);  // the unit that is loaded, and the one after it
    int lpair = *pair_of(lu), npair = *pair_of(nu);
    int ls = wave;
    unsigned woff[2][4], xoff;
    auto place = [&]() {  // this lane's rows of the unit: load instruction q of a tile takes rows 4 q + lane / 16, 256 bytes each
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = 4 * q + g, last = n - 1 - lu.o0, chunk = (r16 ^ r) * 8;
        woff[0][q] = (unsigned)((r < last ? r : last) * k + chunk) * 2u;
        if constexpr (EPI != MOE_GATEUP) woff[1][q] = (unsigned)((16 + r < last ? 16 + r : last) * k + chunk) * 2u;
        else woff[1][q] = woff[0][q];
      }
      xoff = (unsigned)((EPI == MOE_GATEUP ? lpair / top : lpair) * k + 8 * g) * 2u;
    };
    place();
    struct Segment { u32x4 w[2][4], x[4]; } s0, s1;
    // the next segment of this wave
    auto issue = [&](Segment& sg) {
      if (ls >= segs) {
        ls -= segs;
        lu = nu;
        lpair = npair;
        nu = unit_at(lu.id + grid);
        place();
      }
      npair = *pair_of(nu);  // (again with every segment: a value that is loaded only sometimes has to be waited for where the ways meet)
      const int kb = ls * (kT16Seg * 2);
      auto rows = [&](auto stream) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            unsigned off = woff[j][q];
            asm volatile("" : "+v"(off));  // (kept a 32-bit lane offset from a scalar base)
            sg.w[j][q] = ld16_sel<decltype(stream)::value>((j ? lu.b1 : lu.b0) + kb + off);
          }
      };
      if constexpr (HOW == 2) {
        if (lu.alone) rows(std::true_type());
        else rows(std::false_type());
      } else {
        rows(std::integral_constant<bool, HOW == 1>());
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) sg.x[u] = ld16((const uint16_t*)((const uint8_t*)x + kb + 64 * u + xoff));
      ls += 4;
      asm volatile("" ::: "memory");  // the loads stay in front of what follows
    };
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    int cid = lu.id, cs = wave, run_of = wave, ccount = lu.count, co0 = lu.o0, cpair = lpair;  // the unit that is multiplied
    // true at the end of the last unit
    auto step = [&](const Segment& sg) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) *(u32x4*)&wl[wave][j][q * 4 * kT16Seg + lane * 8] = sg.w[j][q];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = mfma16x16x32<T>(*(const u32x4*)&wl[wave][j][r16 * kT16Seg + ((4 * u + g) ^ r16) * 8], sg.x[u], acc[j]);
      cs += 4;
      if (cs < segs) return false;
      cs -= segs;
      // ---- end of a unit; these barriers do not wait for the loads on their way
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();  // the unit before has been read
      asm volatile("" ::: "memory");
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        red[run_of][0][4 * g + r][r16] = acc[0][r];
        red[run_of][1][4 * g + r][r16] = acc[1][r];
      }
      run_of = cs;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const int row = t & 15, col = t >> 4;
      float v0 = 0.f, v1 = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) { v0 += red[w][0][row][col]; v1 += red[w][1][row][col]; }
      const long out = (long)__shfl(cpair, col) * n;
      if (col < ccount) {
        if constexpr (EPI == MOE_GATEUP) {
          if (co0 + row < n) y[out + co0 + row] = T::pack(moe_act(v0, v1, limit));
        } else {
          if (co0 + row < n) y[out + co0 + row] = T::pack(v0);
          if (co0 + 16 + row < n) y[out + co0 + 16 + row] = T::pack(v1);
        }
      }
      acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
      // (the segment requested last is this wave's first of the next unit)
      cid += grid;
      ccount = lu.count;
      co0 = lu.o0;
      cpair = lpair;
      return cid >= units;
    };
    issue(s0);
    while (true) {
      issue(s1);
      if (step(s0)) break;
      issue(s0);
      if (step(s1)) break;
    }
  };
  if (!once) run(std::integral_constant<int, 0>());
  else if (!list[0].pad) run(std::integral_constant<int, 1>());
  else run(std::integral_constant<int, 2>());
}

// NWR x NWT waves of 64 rows x 64 pairs each (gate/up: a wave's rows are 32 gate rows and the 32 up rows of the
// same outputs), 64 k-values per step. LDS rows are 128 bytes; 16-byte chunk c of row r lives at chunk
// c ^ ((r >> 1) & 7). DMA (k % 64 == 0): LDS-direct loads, lane i of a wave instruction fills slot i of eight
// consecutive rows, the swizzle applied to the source chunk. Otherwise the chunks go through registers and
// those past the end of a row are zeroed.
constexpr int kMgK = 64;
extern __shared__ __align__(16) unsigned char moe_smem[];

template <typename T, int EPI, bool DMA, int NWR, int NWT>
__global__ void __launch_bounds__(64 * NWR * NWT, NWR * NWT == 4 ? 2 : 1) moe_tile_kernel(const MoeGemmParams p) {
  constexpr int NW = NWR * NWT, ROWS = 64 * NWR, PAIRS = 64 * NWT, OUT = EPI == MOE_GATEUP ? ROWS / 2 : ROWS;
  constexpr int WQ = 8 / NWT, XQ = 8 / NWR;  // load instructions (eight rows each) per wave and step
  typedef uint16_t WStage[ROWS * kMgK];
  typedef uint16_t XStage[PAIRS * kMgK];
  WStage* w_lds = (WStage*)moe_smem;
  XStage* x_lds = (XStage*)(moe_smem + 2 * sizeof(WStage));
  __shared__ int prow[PAIRS];

  // tile order: a few pair tiles (of one expert, mostly) fastest, then row tiles, so that the workgroups
  // an XCD runs at a time share weight rows and token rows; the tiles are dealt to the XCDs in
  // contiguous shares of what there really is
  constexpr int SUP = PAIRS == 128 ? 4 : 2;
  const int n_tiles = p.tiles[0].count;
  const int r_tiles = (p.n + OUT - 1) / OUT;
  const int total = ((n_tiles + SUP - 1) / SUP) * SUP * r_tiles;
  const int share = (total + 7) / 8;
  const int slot = blockIdx.x >> 3, id = (blockIdx.x & 7) * share + slot;
  if (slot >= share || id >= total) return;
  const int sup = id / (SUP * r_tiles), in_sup = id - sup * SUP * r_tiles;
  const int ti = sup * SUP + in_sup % SUP;
  if (ti >= n_tiles) return;
  const MoeTile tile = p.tiles[1 + ti];
  const int o0 = (in_sup / SUP) * OUT;

  const int t = threadIdx.x, lane = t & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wr = wave / NWT, wt = wave % NWT;
  if (t < PAIRS) prow[t] = p.pairs[tile.first + (t < tile.count ? t : 0)];
  __syncthreads();
  const long eb = (long)tile.expert * p.expert_stride;
  // tile row r -> weight row
  auto wrow = [&](int r) -> const uint16_t* {
    if constexpr (EPI == MOE_GATEUP) {
      const int h = r >> 6, in = r & 63;
      int o = o0 + h * 32 + (in & 31);
      o = o < p.n ? o : p.n - 1;
      return (in >= 32 ? p.w1 : p.w0) + eb + (long)o * p.k;
    } else {
      int o = o0 + r;
      o = o < p.n ? o : p.n - 1;
      return p.w0 + eb + (long)o * p.k;
    }
  };
  // instruction q of this wave covers tile rows (q NW + wave) * 8 ..; the swizzled chunk of a row depends on
  // the lane (and the wave's parity) only
  const int sr = lane >> 3, sc = lane & 7;
  const int chunk = (sc ^ (((wave * 8 + sr) >> 1) & 7)) * 8;
  static_assert(NW % 2 == 0, "rows q NW * 8 apart share their swizzle");
  const uint16_t *wsrc[WQ], *xsrc[XQ];
#pragma unroll
  for (int q = 0; q < WQ; ++q) wsrc[q] = wrow((q * NW + wave) * 8 + sr) + chunk;
#pragma unroll
  for (int q = 0; q < XQ; ++q) {
    const int pr = prow[(q * NW + wave) * 8 + sr];
    xsrc[q] = p.x + (long)(EPI == MOE_GATEUP ? pr / p.top : pr) * p.k + chunk;
  }
  const int steps = (p.k + kMgK - 1) / kMgK;
  // Tiles start at different k-steps, those of an expert's rows at the same: rows are whole multiples of the memory channels' interleave apart, and tiles that walk K in step ask
  // the same channels. Pairs that are not there are not loaded. Weights that no other tile reads, in this call and the next, are requested non-temporally, of gate and up where the tile
  // is a few pairs. us in bf16, 64 experts, before / now, 1408 x 2048, 6 per token, 130 / 400 / 732 /
  // 1100 tokens gate and up 152 / 114, 165 / 127, 169 / 141, 177 / 150, down 68 / 60, 74 / 65, 82 / 72, 90 / 81; 1792 x 4096, 8 per token, 120 / 300 / 600 346 / 297, 344 / 312, 358 / 352 and 164 / 150,
  // 175 / 168, 197 / 190; 16 of 1024 x 2048, 4 per token, 200 tokens 37 / 35, 20 / 18. (From 400 tokens of 1408 x 2048 on, 141 us at 732, gate and up are slower non-temporally, 144. A third stage of weights, or
  // weights of two steps requested together, changes nothing.)
  const int turn = DMA ? (int)((unsigned)(in_sup / SUP + 8 * tile.expert) % (unsigned)steps) : 0;
  const bool alone = p.once && (ti == 0 || p.tiles[ti].expert != tile.expert) && (ti + 1 >= n_tiles || p.tiles[ti + 2].expert != tile.expert) &&
                     (EPI == MOE_DOWN || tile.count <= 32);
  auto dma = [&](int s, int buf) {
    s = s + turn < steps ? s + turn : s + turn - steps;
    if (alone) {
#pragma unroll
      for (int q = 0; q < WQ; ++q) load_lds16_stream(wsrc[q] + s * kMgK, &w_lds[buf][(q * NW + wave) * 8 * kMgK]);
    } else {
#pragma unroll
      for (int q = 0; q < WQ; ++q) load_lds16(wsrc[q] + s * kMgK, &w_lds[buf][(q * NW + wave) * 8 * kMgK]);
    }
#pragma unroll
    for (int q = 0; q < XQ; ++q)
      if ((q * NW + wave) * 8 < tile.count) load_lds16(xsrc[q] + s * kMgK, &x_lds[buf][(q * NW + wave) * 8 * kMgK]);
  };
  u32x4 rw[WQ], rx[XQ];
  auto fetch = [&](int s) {
    const u32x4 zero = {0u, 0u, 0u, 0u};
    const bool live = s * kMgK + chunk < p.k;
    const int off = live ? s * kMgK : -chunk;
#pragma unroll
    for (int q = 0; q < WQ; ++q) { rw[q] = ld16(wsrc[q] + off); rw[q] = live ? rw[q] : zero; }
#pragma unroll
    for (int q = 0; q < XQ; ++q) { rx[q] = ld16(xsrc[q] + off); rx[q] = live ? rx[q] : zero; }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int q = 0; q < WQ; ++q) *(u32x4*)&w_lds[buf][(q * NW + wave) * 8 * kMgK + lane * 8] = rw[q];
#pragma unroll
    for (int q = 0; q < XQ; ++q) *(u32x4*)&x_lds[buf][(q * NW + wave) * 8 * kMgK + lane * 8] = rx[q];
  };
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, lg = lane >> 4, lsw = (r16 >> 1) & 7;
  const int a_base = (wr * 64 + r16) * kMgK, b_base = (wt * 64 + r16) * kMgK;

  if constexpr (DMA) {
    dma(0, 0);
  } else {
    fetch(0);
    put(0);
  }
  for (int s = 0; s < steps; ++s) {
    const int buf = s & 1;
    const bool more = s + 1 < steps;
    if constexpr (DMA) wait_loads<0>();  // this wave's blocks of step s have landed
    __syncthreads();  // ... and everybody's; everybody is done with the other stage
    if (more) {
      if constexpr (DMA) dma(s + 1, buf ^ 1);
      else fetch(s + 1);
    }
    if (wt * 64 < tile.count) {  // (a wave whose pairs are not there only loads)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        u32x4 a[4], b[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = *(const u32x4*)&x_lds[buf][b_base + j * 16 * kMgK + (((kk * 4 + lg) ^ lsw) * 8)];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = *(const u32x4*)&w_lds[buf][a_base + i * 16 * kMgK + (((kk * 4 + lg) ^ lsw) * 8)];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] = mfma16x16x32<T>(a[i], b[j], acc[i][j]);
      }
    }
    if constexpr (!DMA) {
      if (more) put(buf ^ 1);
    }
  }
  // lane: pair column r16, rows 4 lg + r of every 16-row tile
  const bool n4 = (p.n & 3) == 0;
  auto store4 = [&](uint16_t* yr, int o, const float (&v)[4]) {
    if (n4 && o + 4 <= p.n) {
      *(u32x2*)&yr[o] = u32x2{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (o + r < p.n) yr[o + r] = T::pack(v[r]);
    }
  };
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = wt * 64 + j * 16 + r16;
    if (c >= tile.count) continue;
    uint16_t* yr = (uint16_t*)p.y + (long)prow[c] * p.n;
    float v[4];
    if constexpr (EPI == MOE_GATEUP) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = moe_act(acc[i][j][r], acc[i + 2][j][r], p.limit);
        store4(yr, o0 + wr * 32 + i * 16 + 4 * lg, v);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = acc[i][j][r];
        store4(yr, o0 + wr * 64 + i * 16 + 4 * lg, v);
      }
    }
  }
}

// 256 rows x up to 256 pairs on eight waves of 128 x up to 64 (a quarter less LDS traffic per product than waves of 64 x 64,
// which is what bounds those), k a multiple of 64. A wave holds two sets of operands: the LDS reads of one
// half of a k-step are in flight while the other half is multiplied, and the one barrier per step has a
// half's multiplications behind it. An expert's weights come from HBM, mostly once: they have three stages and are
// requested two and a half steps ahead, the tokens (L2) two stages; 160 KB in all, so pairs are read again from memory where
// they are needed. The pairs that there are, in strips of 32, are split evenly over the SIMDs. Gate and up, us, 64 experts,
// with two stages and pairs in strips of 64 -> now: width 4096 x 1792, 2000 tokens of 8 experts 508 -> 470, 1200 tokens 452 -> 397;
// 2048 x 1408, 2000 tokens of 6 experts 206 -> 180. Down 300 -> 286, 243 -> 225, 110 -> 104. The weights at 4 to 5 TB/s and
// the matrix instructions at 0.9 PFLOP/s share the bound; a last round of workgroups that is half empty takes the rest.
// Waiting for all the first loads before the first step looks idle, but it keeps the workgroups that share rows in step:
// without it they miss in L2 (470 -> 500).
template <typename T, int EPI>
__global__ void __launch_bounds__(512) moe_pipe_kernel(const MoeGemmParams p) {
  constexpr int NW = 8, TILE = 256, OUT = EPI == MOE_GATEUP ? TILE / 2 : TILE, WR = 8;
  typedef uint16_t Stage[TILE * kMgK];
  Stage* w_lds = (Stage*)moe_smem;
  Stage* x_lds = (Stage*)(moe_smem + 3 * sizeof(Stage));
  constexpr int SUP = 2;
  const int n_tiles = p.tiles[0].count;
  const int r_tiles = (p.n + OUT - 1) / OUT;
  const int total = ((n_tiles + SUP - 1) / SUP) * SUP * r_tiles;
  const int share = (total + 7) / 8;
  const int slot = blockIdx.x >> 3, id = (blockIdx.x & 7) * share + slot;
  if (slot >= share || id >= total) return;
  const int sup = id / (SUP * r_tiles), in_sup = id - sup * SUP * r_tiles;
  const int ti = sup * SUP + in_sup % SUP;
  if (ti >= n_tiles) return;
  const MoeTile tile = p.tiles[1 + ti];
  const int o0 = (in_sup / SUP) * OUT;

  const int t = threadIdx.x, lane = t & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // SIMD i runs waves i and i + 4: the pairs are dealt out in strips of 32, the odd one to waves 0 .. 3
  const int wr = wave & 1, wt = wave >> 1, strips = (tile.count + 31) >> 5;
  const int cols = 16 * (wt < 2 ? (strips + 1) >> 1 : strips >> 1);  // pairs of this wave, 0 .. 64
  const int col0 = wt < 2 ? wt * cols : 32 * ((strips + 1) >> 1) + (wt - 2) * cols;
  auto pair_at = [&](int c) { return p.pairs[tile.first + (c < tile.count ? c : 0)]; };
  // wave instruction q covers tile rows (q NW + wave) * 8 ..: 32-bit offsets from bases that are the same for
  // the wave (gate and up rows change at multiples of 64)
  const int sr = lane >> 3, sc = lane & 7;
  const int chunk = (sc ^ (((wave * 8 + sr) >> 1) & 7)) * 8;
  const int steps = p.k / kMgK;
  int pr[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) pr[q] = pair_at((q * NW + wave) * 8 + sr);
  const uint16_t* wbase[4];
  unsigned woff[4], xoff[4];
  const long eb = (long)tile.expert * p.expert_stride;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r0 = (q * NW + wave) * 8, r = r0 + sr;
    int o;
    if constexpr (EPI == MOE_GATEUP) {  // a wave's 128 rows: 64 gate rows, the 64 up rows of the same outputs
      o = o0 + (r >> 7) * 64 + (r & 63);
      wbase[q] = ((r0 & 64) ? p.w1 : p.w0) + eb;
    } else {
      o = o0 + r;
      wbase[q] = p.w0 + eb;
    }
    o = o < p.n ? o : p.n - 1;
    woff[q] = (unsigned)o * (unsigned)p.k + chunk;
  }
  auto load_x = [&](int s) {
    const uint16_t* base = p.x + (s < steps ? s : steps - 1) * kMgK;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      unsigned off = xoff[q];
      asm volatile("" : "+v"(off));  // (kept as a 32-bit offset from a scalar base)
      load_lds16(base + off, &x_lds[s & 1][(q * NW + wave) * 8 * kMgK]);
    }
  };
  auto load_w = [&](int s, int stage) {
    s = s < steps ? s : steps - 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      unsigned off = woff[q];
      asm volatile("" : "+v"(off));
      load_lds16(wbase[q] + s * kMgK + off, &w_lds[stage][(q * NW + wave) * 8 * kMgK]);
    }
  };
  const int r16 = lane & 15, lg = lane >> 4, lsw = (r16 >> 1) & 7;
  const int a_base = (wr * 128 + r16) * kMgK, b_base = (col0 + r16) * kMgK;
  load_w(0, 0);
#pragma unroll
  for (int q = 0; q < 4; ++q) xoff[q] = (unsigned)(EPI == MOE_GATEUP ? pr[q] / p.top : pr[q]) * (unsigned)p.k + chunk;
  load_x(0);
  load_x(1);
  load_w(1, 1);
  load_w(2, 2);
  wait_loads<12>();
  __syncthreads();
  const bool n4 = (p.n & 3) == 0;
  auto store4 = [&](uint16_t* yr, int o, const float (&v)[4]) {
    if (n4 && o + 4 <= p.n) {
      *(u32x2*)&yr[o] = u32x2{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (o + r < p.n) yr[o + r] = T::pack(v[r]);
    }
  };
  // Loads past the last step repeat it, into a stage nobody reads any more: no branches in the loop. Every wave
  // meets the same barriers, whatever its width.
  auto run = [&](auto width) {
    constexpr int WT = decltype(width)::value;
    constexpr int MF = WT > 2 ? 2 : 1;  // matrix instructions between two LDS reads
    f32x4 acc[WR][WT];
#pragma unroll
    for (int i = 0; i < WR; ++i)
#pragma unroll
      for (int j = 0; j < WT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 a[2][WR], b[2][WT];
    auto read = [&](int buf, int stage, int kk, int set) {
      const int c = ((kk * 4 + lg) ^ lsw) * 8;
#pragma unroll
      for (int j = 0; j < WT; ++j) b[set][j] = *(const u32x4*)&x_lds[buf][b_base + j * 16 * kMgK + c];
#pragma unroll
      for (int i = 0; i < WR; ++i) a[set][i] = *(const u32x4*)&w_lds[stage][a_base + i * 16 * kMgK + c];
    };
    auto multiply = [&](int set) {
#pragma unroll
      for (int i = 0; i < WR; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) acc[i][j] = mfma16x16x32<T>(a[set][i], b[set][j], acc[i][j]);
    };
    read(0, 0, 0, 0);
    for (int s = 0, stage = 0; s < steps; ++s) {
      const int buf = s & 1, next = stage < 2 ? stage + 1 : 0;
      read(buf, stage, 1, 1);
      multiply(0);
      // issue order of the half: matrix instructions, an LDS read, ...
#pragma unroll
      for (int i = 0; i < WR + WT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, MF, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      if constexpr (WR * WT > MF * (WR + WT)) __builtin_amdgcn_sched_group_barrier(0x008, WR * WT - MF * (WR + WT), 0);
      wait_loads<4>();  // step s + 1 has landed, the weights of step s + 2 may be on their way
      __syncthreads();  // ... for everybody, and everybody has read step s
      load_x(s + 2);
      load_w(s + 3, stage);
      read(buf ^ 1, next, 0, 0);
      multiply(1);
      stage = next;
      // ... a matrix instruction and a load, eight times, then matrix instructions and a read
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
      }
#pragma unroll
      for (int i = 0; i < WR + WT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, WT > 3 ? 2 : 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
    wait_loads<0>();  // no load is still on its way into LDS when the workgroup ends
    int out[WT];
#pragma unroll
    for (int j = 0; j < WT; ++j) out[j] = pair_at(col0 + j * 16 + r16);
#pragma unroll
    for (int j = 0; j < WT; ++j) {
      const int c = col0 + j * 16 + r16;
      if (c >= tile.count) continue;
      uint16_t* yr = (uint16_t*)p.y + (long)out[j] * p.n;
      float v[4];
      if constexpr (EPI == MOE_GATEUP) {
#pragma unroll
        for (int i = 0; i < WR / 2; ++i) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = moe_act(acc[i][j][r], acc[i + WR / 2][j][r], p.limit);
          store4(yr, o0 + wr * 64 + i * 16 + 4 * lg, v);
        }
      } else {
#pragma unroll
        for (int i = 0; i < WR; ++i) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = acc[i][j][r];
          store4(yr, o0 + wr * 128 + i * 16 + 4 * lg, v);
        }
      }
    }
  };
  if (cols == 64) run(std::integral_constant<int, 4>());
  else if (cols == 48) run(std::integral_constant<int, 3>());
  else if (cols == 32) run(std::integral_constant<int, 2>());
  else if (cols == 16) run(std::integral_constant<int, 1>());
  else {  // no pairs for this wave: it only keeps the loads going
    for (int s = 0, stage = 0; s < steps; ++s) {
      wait_loads<4>();
      __syncthreads();
      load_x(s + 2);
      load_w(s + 3, stage);
      stage = stage < 2 ? stage + 1 : 0;
    }
    wait_loads<0>();
  }
}

// One token: routing, gate and up in one launch. Every workgroup chooses the experts by itself: a thread per output counts those that are ahead of its own (top rounds of
// a maximum over a wave took 3 us longer), about a microsecond behind the logits, where a launch for it is five. Then the chosen experts' rows are one long list for the
// single-token GEMV structure of gemv_multi.hip: gate and up rows of two outputs at a time, thread t has chunks t, t + 256 of every row, the next rows are requested before
// the sums meet. A matrix instruction has no use for fifteen of its sixteen columns here, and weights go from memory to registers to the ALU without LDS between. Workgroup
// 0 writes down what was chosen, and the tiles of one pair that the down product reads. us of routing, gate and up in bf16 as captured, two launches / this: 64 experts of 1792 x 4096, 8 / 7 / 6 of them
// 46.8 / 39.3, 44.6 / 35.5, 36.9 / 30.9 (their bytes take 33.1, 28.9, 24.8); of 1408 x 2048, 6 / 5 21.6 / 16.1, 18.8 / 14.3 (9.7, 8.1).
constexpr int kMoeOneOutputs = 256, kMoeOneTop = 8;
template <typename T, int CH, bool STREAM>
__global__ void __launch_bounds__(256) moe_one_gateup_kernel(const float* logits, const uint16_t* corr, const uint16_t* x, int n_out, int k, const uint16_t* w0,
                                                             const uint16_t* w1, int n_experts, int top, long expert_stride, int n, float limit, uint16_t* act,
                                                             int32_t* expert, float* weight, int32_t* pairs, MoeTile* tiles, int max_tiles) {
  constexpr int R = 4, OUT = R / 2;
  __shared__ float red[2][16][R];  // [buffer][16-lane row of the workgroup][row]
  __shared__ float meet[2][4];
  __shared__ __align__(16) float value[kMoeOneOutputs];
  __shared__ int list[kMoeOneTop][2];  // of the chosen with matrices: which it is, its place in the choice
  __shared__ int real_s;
  const int t = threadIdx.x, lane = t & (kWave - 1), kc = k >> 3;
  const bool there = t < n_out;
  float lg = logits[there ? t : 0], add = T::one(*(corr ? corr + (there ? t : 0) : x));
  int coff[CH];
  u32x4 xq[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int c = t + 256 * j;
    coff[j] = c < kc ? c << 3 : 0;
    xq[j] = ld16(x + coff[j]);
  }
  lg = there ? lg : -INFINITY;
  const float wave_mx = wave_max(lg);
  if (lane == 0) meet[0][t >> 6] = wave_mx;
  if (t == 0) real_s = 0;
  if (t < 2 * kMoeOneTop) list[t >> 1][t & 1] = 0;
  __syncthreads();
  const float ex = expf(lg - fmaxf(fmaxf(meet[0][0], meet[0][1]), fmaxf(meet[0][2], meet[0][3])));
  const float wave_ex = wave_sum(ex);
  if (lane == 0) meet[1][t >> 6] = wave_ex;
  __syncthreads();
  const float share = ex / ((meet[1][0] + meet[1][1]) + (meet[1][2] + meet[1][3]));
  float choice = share + (corr ? add : 0.f);
  choice = there & (choice == choice) ? choice : -INFINITY;
  value[t] = choice;
  __syncthreads();
  if (there) {
    // how many outputs are ahead of this one, and how many of them have matrices (those past the last one are behind all)
    int ahead = 0, ahead_real = 0;
#pragma unroll 2
    for (int i = 0; i < n_out; i += 8) {
      const f32x4 v0 = *(const f32x4*)&value[i], v1 = *(const f32x4*)&value[(i + 4) & (kMoeOneOutputs - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float v = u < 4 ? v0[u & 3] : v1[u & 3];
        const int before = (int)(v > choice) | ((int)(v == choice) & (int)(i + u < t));
        ahead += before;
        ahead_real += i + u < n_experts ? before : 0;
      }
    }
    if (ahead < top) {
      if (t < n_experts) {
        list[ahead_real][0] = t;
        list[ahead_real][1] = ahead;
        atomicAdd(&real_s, 1);
      }
      if (blockIdx.x == 0) {
        expert[ahead] = t;
        weight[ahead] = share;
      }
    }
  }
  __syncthreads();
  const int real = __builtin_amdgcn_readfirstlane(real_s);
#pragma unroll
  for (int j = 0; j < CH; ++j)
    if (t + 256 * j >= kc) xq[j] = u32x4{0u, 0u, 0u, 0u};
  if (blockIdx.x == 0) {
    if (t == 0) tiles[0] = MoeTile{0, 0, real, 0};
    if (t < max_tiles) {
      tiles[1 + t] = t < real ? MoeTile{list[t][0], t, 1, 0} : MoeTile{0, 0, 0, 0};
      if (t < real) pairs[t] = list[t][1];
    }
  }
  const int groups = real * (n / OUT);  // (n is even)
  struct Place { int slot, row, expert, place; } now = {0, (int)blockIdx.x * OUT, 0, 0}, next;
  auto settle = [&](Place& p) {  // the row's expert
    while (p.row >= n && p.slot + 1 < kMoeOneTop) {
      p.row -= n;
      ++p.slot;
    }
    p.expert = __builtin_amdgcn_readfirstlane(list[p.slot][0]);
    p.place = __builtin_amdgcn_readfirstlane(list[p.slot][1]);
  };
  u32x4 w[R][CH];
  auto request = [&](const Place& p) {
    const long base = (long)p.expert * expert_stride + (long)p.row * k;
    const uint16_t *gate = w0 + base, *up = w1 + base;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int j = 0; j < CH; ++j) w[r][j] = ld16_sel<STREAM>(((r & 1) ? up : gate) + (long)(r >> 1) * k + coff[j]);
  };
  int buf = 0;
  if ((int)blockIdx.x >= groups) return;  // uniform for the workgroup
  settle(now);
  request(now);
  for (int g = blockIdx.x; g < groups; g += gridDim.x) {
    next = now;
    next.row += (int)gridDim.x * OUT;
    settle(next);
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float a = 0.f;
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        a = moe_dot2<T>(w[r][j].x, xq[j].x, a);
        a = moe_dot2<T>(w[r][j].y, xq[j].y, a);
        a = moe_dot2<T>(w[r][j].z, xq[j].z, a);
        a = moe_dot2<T>(w[r][j].w, xq[j].w, a);
      }
      acc[r] = a;
    }
    if (g + (int)gridDim.x < groups) request(next);
    row16_reduce_scatter<R>(acc, lane);
    if ((lane & (16 / R - 1)) == 0) red[buf][t >> 4][(lane & 15) / (16 / R)] = acc[0];
    __syncthreads();
    if (t < 16 * OUT) {  // sixteen lanes per output
      const int part = t & 15, o = t >> 4;
      const float v0 = row16_sum(red[buf][part][2 * o]), v1 = row16_sum(red[buf][part][2 * o + 1]);
      if (part == 0) act[(long)now.place * n + now.row + o] = T::pack(moe_act(v0, v1, limit));
    }
    buf ^= 1;
    now = next;
  }
}

// One token's down product, built like gate and up above: R rows of one chosen expert at a time, thread t has chunks t, t + 256 of every row, the next rows are on their
// way before the sums meet. The chosen are read by lane; a pair's activations are requested with its rows. Bound by the rows' bytes and a cold chain of two loads. us in
// bf16 as captured, 16-pair tiles / this (at 7.1 TB/s): 64 experts of 1792 x 4096, 8 / 7 / 5 with matrices 19.7 / 19.0 (16.5), 18.6 / 17.4 (14.5), 14.3 / 12.6 (10.3); of
// 1408 x 2048 10.8 / 9.8 (6.5), 10.3 / 8.6 (5.7), 9.1 / 6.7 (4.1); 32 of 4096 x 1024, 8 / 2 15.0 / 12.8 (9.5), 8.4 / 4.8 (2.4); 16 of 768 x 2048, 8 / 5 7.9 / 7.6, 7.0 / 5.3; 8 of
// 1024 x 512, 8 4.2 / 3.4. Rows of 512 keep a quarter of the threads: 64 of 512 x 4096, 8 9.0 / 11.7, so shorter rows than 768 stay with the tiles, and those below 1280 where there
// are 32768 of them and more: 64 of 768 x 4096, 4 / 8 / 32 8.1 / 7.9, 11.1 / 13.1, 32.5 / 38.6; of 1024 x 4096, 4 / 16 8.9 / 8.3, 22.4 / 23.8 (of 1408 x 4096, 8 16.6 / 16.3).
template <typename T, int CH, int R, bool STREAM>
__global__ void __launch_bounds__(256) moe_one_down_kernel(const int32_t* expert, const uint16_t* act, int top, int n_experts, int n, int k, const uint16_t* w0,
                                                           long expert_stride, uint16_t* y) {
  __shared__ float red[2][16][R];  // [buffer][16-lane row of the workgroup][row]
  const int t = threadIdx.x, lane = t & (kWave - 1), kc = k >> 3;
  const int mine = lane < top ? expert[lane] : n_experts;
  int coff[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) coff[j] = t + 256 * j < kc ? (t + 256 * j) << 3 : 0;
  uint64_t real = __ballot(mine < n_experts);  // places of the chosen with matrices, those behind `row`'s taken out
  const int groups = __popcll(real) * (n / R);
  if ((int)blockIdx.x >= groups) return;  // uniform for the workgroup
  int row = (int)blockIdx.x * R, place = 0;
  u32x4 w[R][CH], xq[CH], xn[CH];
  auto request = [&]() {
    while (row >= n) {
      row -= n;
      real &= real - 1;
    }
    place = __ffsll((unsigned long long)real) - 1;
    const uint16_t* base = w0 + (long)__builtin_amdgcn_readlane(mine, place) * expert_stride + (long)row * k;
#pragma unroll
    for (int j = 0; j < CH; ++j) xn[j] = ld16(act + (long)place * k + coff[j]);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int j = 0; j < CH; ++j) w[r][j] = ld16_sel<STREAM>(base + (long)r * k + coff[j]);
  };
  request();
  int buf = 0;
  for (int g = blockIdx.x; g < groups; g += gridDim.x) {
    const int out_place = place, out_row = row;
#pragma unroll
    for (int j = 0; j < CH; ++j) xq[j] = t + 256 * j < kc ? xn[j] : u32x4{0u, 0u, 0u, 0u};
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float a = 0.f;
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        a = moe_dot2<T>(w[r][j].x, xq[j].x, a);
        a = moe_dot2<T>(w[r][j].y, xq[j].y, a);
        a = moe_dot2<T>(w[r][j].z, xq[j].z, a);
        a = moe_dot2<T>(w[r][j].w, xq[j].w, a);
      }
      acc[r] = a;
    }
    if (g + (int)gridDim.x < groups) {
      row += (int)gridDim.x * R;
      request();
    }
    row16_reduce_scatter<R>(acc, lane);
    if ((lane & (16 / R - 1)) == 0) red[buf][t >> 4][(lane & 15) / (16 / R)] = acc[0];
    __syncthreads();
    if (t < 16 * R) {  // sixteen lanes per output
      const int part = t & 15, o = t >> 4;
      const float v = row16_sum(red[buf][part][o]);
      if (part == 0) y[(long)out_place * n + out_row + o] = T::pack(v);
    }
    buf ^= 1;
  }
}

// one wave per output of a pair: fp32 storage, and sizes that are no multiple of 8
template <typename T, int EPI>
__global__ void __launch_bounds__(256) moe_rows_kernel(const typename T::storage* w0, const typename T::storage* w1,
                                                       long expert_stride, const typename T::storage* x,
                                                       typename T::storage* y, const int32_t* expert, int n_experts,
                                                       int n, int k, int top, float limit) {
  const int lane = threadIdx.x & (kWave - 1);
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const long pair = blockIdx.y;
  if (row >= n) return;
  const int e = expert[pair];
  if (e >= n_experts) return;
  const typename T::storage* xr = x + (EPI == MOE_GATEUP ? pair / top : pair) * k;
  const typename T::storage* a = w0 + e * expert_stride + (long)row * k;
  float s0 = 0.f, s1 = 0.f;
  for (int c = lane; c < k; c += kWave) {
    const float xv = T::one(xr[c]);
    s0 = fmaf(T::one(a[c]), xv, s0);
    if constexpr (EPI == MOE_GATEUP) s1 = fmaf(T::one(w1[e * expert_stride + (long)row * k + c]), xv, s1);
  }
  s0 = wave_sum(s0);
  if constexpr (EPI == MOE_GATEUP) {
    s1 = wave_sum(s1);
    s0 = moe_act(s0, s1, limit);
  }
  if (lane == 0) y[pair * n + row] = T::pack(s0);
}

template <typename T, int EPI>
static void launch_moe_tile16(hipStream_t s, dim3 grid, const MoeGemmParams& p) {
  hipLaunchKernelGGL((moe_tile16_kernel<T, EPI>), grid, dim3(256), 0, s, p.tiles, p.w0, p.w1, p.expert_stride, p.n, p.k, p.max_tiles, (int)p.once, p.pairs, p.x, p);
}

template <typename T, int EPI, int NWR, int NWT>
static int launch_moe_tile(hipStream_t s, const MoeGemmParams& p) {
  constexpr int OUT = (EPI == MOE_GATEUP ? 32 : 64) * NWR, SUP = NWT == 2 ? 4 : 2;
  const long total = (long)ceil_div(p.max_tiles, SUP) * SUP * ceil_div(p.n, OUT);
  if (total > (1L << 30)) return MUI_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)((total + 7) / 8 * 8)), block(64 * NWR * NWT);
  const size_t lds = (size_t)2 * 64 * (NWR + NWT) * kMgK * 2;
  if (p.k % kMgK == 0) return launch_with_lds(moe_tile_kernel<T, EPI, true, NWR, NWT>, grid, block, lds, s, p);
  return launch_with_lds(moe_tile_kernel<T, EPI, false, NWR, NWT>, grid, block, lds, s, p);
}

template <typename T, int EPI>
static int launch_moe_product(hipStream_t s, const MoeGemmParams& p, const int32_t* expert, int n_experts, int n_pairs,
                              int tile_pairs) {
  typedef typename T::storage S;
  bool rows = T::kDtype == MUI_DTYPE_F32 || p.k % 8 != 0 || tile_pairs == 0;
  rows = rows || !aligned16(p.w0) || (p.w1 && !aligned16(p.w1)) || !aligned16(p.x) || p.expert_stride % 8 != 0;
  if (rows) {
    // pairs are one dimension of the grid: whole tokens' worth of them per launch
    const int step = 65535 / p.top * p.top;
    if (step < 1) return MUI_ERR_UNSUPPORTED;
    for (int first = 0; first < n_pairs; first += step) {
      const int cnt = n_pairs - first < step ? n_pairs - first : step;
      const long xrow = EPI == MOE_GATEUP ? first / p.top : first;
      hipLaunchKernelGGL((moe_rows_kernel<T, EPI>), dim3(ceil_div(p.n, 4), cnt), dim3(256), 0, s, (const S*)p.w0,
                         (const S*)p.w1, p.expert_stride, (const S*)p.x + xrow * p.k, (S*)p.y + (long)first * p.n,
                         expert + first, n_experts, p.n, p.k, p.top, p.limit);
    }
    return launch_status();
  }
  if constexpr (T::kDtype != MUI_DTYPE_F32) {
    if (tile_pairs == 16) {
      if (p.max_tiles > 65535) return MUI_ERR_UNSUPPORTED;
      const int blocks = ceil_div(p.n, EPI == MOE_GATEUP ? 16 : 32);
      const long units = (long)blocks * p.max_tiles, xrows = EPI == MOE_GATEUP ? p.tokens : (long)p.tokens * p.top;
      if (p.tiles && p.k % kT16Seg == 0 && p.k >= 4 * kT16Seg && (long)p.n * p.k < (1L << 30) && xrows * p.k < (1L << 30) && units < (1L << 30)) {
        const long round = 2L * device_cus();
        hipLaunchKernelGGL((moe_units_kernel<T, EPI>), dim3((unsigned)(units < round ? units : round)), dim3(256), 0, s, p.tiles, p.w0, p.w1, p.expert_stride,
                           p.pairs, p.n, p.k, p.x, p.top, blocks, p.max_tiles, (int)p.once, p.limit, (uint16_t*)p.y);
        return launch_status();
      }
      launch_moe_tile16<T, EPI>(s, dim3(blocks, p.max_tiles), p);
      return launch_status();
    }
    if (((uintptr_t)p.y & 7) != 0) return MUI_ERR_ALIGNMENT;
    if (tile_pairs == 128) return launch_moe_tile<T, EPI, 2, 2>(s, p);
    if (tile_pairs == 256) {
      const long xrows = EPI == MOE_GATEUP ? p.tokens : (long)p.tokens * p.top;
      if (p.k % kMgK == 0 && (long)p.n * p.k < (1L << 30) && xrows * p.k < (1L << 30)) {
        const long total = (long)ceil_div(p.max_tiles, 2) * 2 * ceil_div(p.n, EPI == MOE_GATEUP ? 128 : 256);
        if (total > (1L << 30)) return MUI_ERR_UNSUPPORTED;
        return launch_with_lds(moe_pipe_kernel<T, EPI>, dim3((unsigned)((total + 7) / 8 * 8)), dim3(512),
                               (size_t)5 * 256 * kMgK * 2, s, p);
      }
      return launch_moe_tile<T, EPI, 4, 4>(s, p);
    }
    return MUI_ERR_INVALID_ARG;
  }
  return MUI_ERR_UNSUPPORTED;
}

template <typename T>
static int launch_linear_f32(hipStream_t s, const void* w, const void* x, const void* bias, float* y, int n, int k,
                             int tokens) {
  typedef typename T::storage S;
  const bool vec = k % 8 == 0 && aligned16(w) && aligned16(x);
  if constexpr (T::kDtype != MUI_DTYPE_F32) {
    if (vec && tokens > MUI_MAX_TOKENS) {
      MoeGemmParams p = {};
      p.w0 = (const uint16_t*)w; p.x = (const uint16_t*)x; p.bias = (const uint16_t*)bias; p.y = y; p.n = n; p.k = k;
      p.top = 1; p.tokens = tokens;
      const int tiles = ceil_div(tokens, 16);
      if (tiles > 65535) return MUI_ERR_UNSUPPORTED;
      launch_moe_tile16<T, MOE_F32>(s, dim3(ceil_div(n, 32), tiles), p);
      return launch_status();
    }
  }
  auto launch = [&](auto kernel, int tb) {
    int ty = ceil_div(tokens, tb);
    if (ty > 4096) ty = 4096;
    hipLaunchKernelGGL(kernel, dim3(n, ty), dim3(256), 0, s, (const S*)w, (const S*)x, (const S*)bias, y, n, k, tokens);
    return launch_status();
  };
  if (!vec) return launch(linear_f32_rows_kernel<T, false, 4>, 4);
  if (tokens == 1) return launch(linear_f32_rows_kernel<T, true, 1>, 1);
  return launch(linear_f32_rows_kernel<T, true, 4>, 4);
}

template <typename T>
static int launch_route(hipStream_t s, const float* logits, const void* corr, int n_out, int n_experts, int top,
                        int tokens, int tile_pairs, int max_tiles, int32_t* expert, float* weight, int32_t* pairs,
                        MoeTile* tiles) {
  typedef typename T::storage S;
  // One launch of one workgroup, whose waves route a token each, or another workgroup per four tokens in front: us, one launch / two, 64 experts, 8 chosen: 8 tokens 6.7 / 7.6,
  // 12 7.1 / 7.2, 16 8.0 / 7.6, 20 9.7 / 7.6, 32 12.6 / 7.6, 64 22.0 / 7.6; 6 chosen 6.0 / 6.9, 6.3 / 6.7, 7.2 / 6.9, 8.3 / 6.9, 10.9 / 6.9, 18.7 / 6.9; 4 chosen 12 5.8 / 6.1,
  // 16 6.1 / 6.2, 20 6.8 / 6.1; 1 chosen 12 4.7 / 5.3, 16 5.1 / 5.3, 24 5.5 / 5.4
  const bool one = tokens <= (top <= 4 ? 16 : 12) && tile_pairs;
  if (!one)
    hipLaunchKernelGGL((moe_route_kernel<T>), dim3(ceil_div(tokens, 4)), dim3(256), 0, s, logits, (const S*)corr, n_out,
                       top, tokens, expert, weight);
  if (!tile_pairs) return launch_status();
  if (one)
    hipLaunchKernelGGL((moe_group_kernel<T, true>), dim3(1), dim3(tokens <= 4 ? 256 : kRouteThreads), 0, s, logits, (const S*)corr, n_out,
                       n_experts, top, tokens, tile_pairs, max_tiles, expert, weight, pairs, tiles);
  else
    hipLaunchKernelGGL((moe_group_kernel<T, false>), dim3(1), dim3(kRouteThreads), 0, s, logits, (const S*)corr, n_out,
                       n_experts, top, tokens, tile_pairs, max_tiles, expert, weight, pairs, tiles);
  return launch_status();
}

}  // namespace mui

using namespace mui;

#define MUI_BY_DTYPE(call)                                  \
  do {                                                      \
    if (dtype == MUI_DTYPE_F16) { typedef F16 TT; return call; }   \
    if (dtype == MUI_DTYPE_BF16) { typedef BF16 TT; return call; } \
    if (dtype == MUI_DTYPE_F32) { typedef F32 TT; return call; }   \
    return MUI_ERR_INVALID_ARG;                             \
  } while (0)

extern "C" int mui_linear_f32(mui_stream_t stream, int dtype, const void* weights, const void* x, const void* bias,
                              float* y, int n_out, int k_in, int tokens) {
  MUI_CHECK_ARG(weights && x && y && n_out > 0 && k_in > 0 && tokens > 0);
  MUI_BY_DTYPE((launch_linear_f32<TT>((hipStream_t)stream, weights, x, bias, y, n_out, k_in, tokens)));
}

extern "C" int mui_moe_tile_pairs(int dtype, int tokens, int top, int n_experts, int width, int ff) {
  if (dtype == MUI_DTYPE_F32 || width % 8 || ff % 8 || n_experts < 1) return 0;
  // 16-pair tiles stream an expert's weights once per tile; from about a dozen pairs per expert on a wide tile
  // is cheaper even half empty. 256-pair tiles of the pipelined kernel cost what their pairs cost, where there are
  // enough of them for the chip (one tile per expert, gate and up in tiles of 128 rows and down of 256). 128-pair tiles take what an expert has beyond 128 pairs in a tile
  // of its own, which the mean foretells the better the more experts there are. us of both products, 128 / 256 pairs, at 97, 104, 112 and 120 pairs per expert,
  // tokens spread evenly (two figures: with and without experts beyond 128):
  //   gate and up on less than three quarters of the CUs: 8 of 1792 x 4096 97 / 109, 16 of 768 x 2048 52 / 62
  //   down on less than half: 16 of 2048 x 1024 51 / 58, 52 / 59, 60 / 60, 52 and 62 / 60; 16 of 4096 x 1024 123 / 139 to 152, 124 / 139 to 153, 125 / 140 to 154, 141 / 142 to 155
  //   down on half: 32 of 1024 x 1024 44 / 49, 44 / 49, 44 and 57 / 50, 57 / 51; 32 of 2048 x 1024 108 / 114, 111 and 124 / 116, 112 and 124 / 116, 130 / 117; 16 of
  //   2048 x 2048 98 / 104, 100 / 105, 101 and 136 / 106, 136 / 107; 64 of 512 x 512 29 / 34, 37 / 35, 38 / 35, 37 / 36; 8 of 4096 x 4096, 125 pairs, 232 to 261 / 194 to 206
  //   down on three quarters: 24 of 1408 x 2048 123 / 129, 122 / 130, 126 / 132, 128 / 133; 32 of 1024 x 2048 92 to 108 / 99 to 110, 92 to 138 / 100 to 112,
  //   126 to 139 / 95 to 112, 128 to 135 / 95 to 113; 64 of 1408 x 2048 260 / 261, 265 to 294 / 265 to 280, 291 to 306 / 264 to 282, 303 to 320 / 261 to 279; 128 of 768 x 2048
  //   274 / 286, 304 / 293, 316 / 297, 328 / 299; and a long K makes up for more: 64 of 1792 x 4096 597 / 591, 609 / 598, 635 / 603, 690 / 611; 16 of it 163 / 164,
  //   162 / 160, 179 and 216 / 157, 217 / 160.
  // Those of the other kernel (k no multiple of 64), rarely full, cost about 1.3 times as much as a 128-pair one.
  const long per = (long)tokens * top / n_experts;
  if (per < 12) return 16;
  if (width % kMgK == 0 && ff % kMgK == 0) {
    const long cus = device_cus(), gateup = (long)n_experts * ceil_div(ff, 128), down = (long)n_experts * ceil_div(width, 256);
    const int line = gateup * 4 < cus * 3 || down * 2 < cus ? 129 : down * 4 < cus * 3 ? 108 : width >= 4096 ? 96 : n_experts >= 32 ? 104 : 120;
    return per < line ? 128 : 256;
  }
  return 13 * ((per + 255) / 256) < 10 * ((per + 127) / 128) ? 256 : 128;
}

extern "C" int mui_moe_max_tiles(int tokens, int top, int n_experts, int tile_pairs) {
  if (tile_pairs < 1) return 0;
  const long pairs = (long)tokens * top;
  return (int)(pairs / tile_pairs + (pairs < n_experts ? pairs : n_experts));
}

extern "C" int mui_moe_route(mui_stream_t stream, int dtype, const float* logits, const void* correction, int n_experts,
                             int n_identity, int top, int tokens, int tile_pairs, int32_t* expert, float* weight,
                             int32_t* pairs, void* tiles) {
  MUI_CHECK_ARG(logits && expert && weight && tokens > 0 && n_experts >= 0 && n_identity >= 0);
  const int n_out = n_experts + n_identity;
  MUI_CHECK_ARG(n_out > 0 && top > 0 && top <= n_out);
  MUI_CHECK_ARG(tile_pairs == 0 || tile_pairs == 16 || tile_pairs == 128 || tile_pairs == 256);
  MUI_CHECK_ARG(tile_pairs == 0 || (pairs && tiles));
  if (n_out > kMaxRouter || (long)tokens * top > (1L << 30)) return MUI_ERR_UNSUPPORTED;
  const int mt = mui_moe_max_tiles(tokens, top, n_experts, tile_pairs);
  MUI_BY_DTYPE((launch_route<TT>((hipStream_t)stream, logits, correction, n_out, n_experts, top, tokens, tile_pairs, mt,
                                 expert, weight, pairs, (MoeTile*)tiles)));
}

// Whether a layer's experts (n x k each) are too large to be found in the memory-side cache at the next call:
// that cache holds 256 MB: the experts of eight layers and more of 32 MB don't stay there. Below (8 experts of 512 x 1024, 17 MB) a model may stay:
// 4 tokens 4.7 us ordinary, 5.1 non-temporal while it does, 5.5 either way when it does not
// Rows that are no whole cache lines share one at their ends and where two runs meet: non-temporal it came twice (64 experts of 1000 x 2000, 1 token each
// for 32 of them 16.1 us ordinary, 17.8 non-temporal, 100 tokens of 2 137 and 148).
static bool read_once(int n_experts, int n, int k, const void* a, const void* b) {
  return (long)n_experts * n * k * 4 > (32L << 20) && k % 64 == 0 && (((uintptr_t)a | (uintptr_t)b) & 127) == 0;
}

extern "C" int mui_moe_gateup(mui_stream_t stream, int dtype, const void* gate, const void* up, long expert_stride,
                              const void* x, float limit, const int32_t* expert, const int32_t* pairs,
                              const void* tiles, int tile_pairs, void* act, int n_experts, int n_inter, int k_in,
                              int top, int tokens) {
  MUI_CHECK_ARG(gate && up && x && expert && act && n_experts > 0 && n_inter > 0 && k_in > 0 && top > 0 && tokens > 0);
  MUI_CHECK_ARG(tile_pairs == 0 || (pairs && tiles));
  MoeGemmParams p = {};
  p.w0 = (const uint16_t*)gate; p.w1 = (const uint16_t*)up; p.expert_stride = expert_stride; p.x = (const uint16_t*)x;
  p.y = act; p.pairs = pairs; p.tiles = (const MoeTile*)tiles; p.n = n_inter; p.k = k_in; p.top = top; p.tokens = tokens;
  p.limit = limit; p.max_tiles = mui_moe_max_tiles(tokens, top, n_experts, tile_pairs);
  p.once = read_once(n_experts, n_inter, k_in, gate, up);
  MUI_BY_DTYPE((launch_moe_product<TT, MOE_GATEUP>((hipStream_t)stream, p, expert, n_experts, tokens * top, tile_pairs)));
}

namespace mui {
// Microseconds: what counting who is ahead takes, outputs after outputs in every workgroup, the more of them on a CU the longer, and what rounds of rows too short for 256 threads lose
// against the tiles' (long ones gain), against the launch in front. Of 1530 sizes (8 to 256 outputs, 1 to 8 chosen, 256 to 4096 activations of rows of 256 to 4096, cold weights) it is taken
// for 783, 25 % faster, six of them 2 to 8 % slower; taken wherever the kernel could, 554 were slower: us, two launches / one, 128 outputs, 4 of 1024 x 256 9.1 / 11.1; 248, 2 of 1024 x 512
// 9.4 / 14.7; 64, 8 of 4096 x 512 18.5 / 26.4.
static bool one_launch_is_faster(int n_out, int top, int n, int k, int grid) {
  const int per_cu = ceil_div(grid, device_cus()), rounds = ceil_div(top * (n / 2), grid);
  return (float)n_out * (0.022f + 0.008f * (float)per_cu) + (k < 768 ? 0.5f : k < 1536 ? 0.2f : -0.2f) * (float)rounds < 5.f;
}

// One token and sizes that moe_one_gateup_kernel covers, else MUI_ERR_UNSUPPORTED (nothing launched)
template <typename T>
static int launch_moe_one(hipStream_t s, const MoeGemmParams& p, const float* logits, const void* corr, int n_out, int n_experts, int32_t* expert, float* weight,
                          int32_t* pairs, MoeTile* tiles) {
  if constexpr (T::kDtype == MUI_DTYPE_F32) {
    return MUI_ERR_UNSUPPORTED;
  } else {
    if (p.tokens != 1 || n_out > kMoeOneOutputs || p.top > kMoeOneTop || p.n % 2 || p.k % 8 || p.k > 2 * 256 * 8 || p.expert_stride % 8) return MUI_ERR_UNSUPPORTED;
    if (!aligned16(p.w0) || !aligned16(p.w1) || !aligned16(p.x) || (long)p.top * p.n >= (1L << 30)) return MUI_ERR_UNSUPPORTED;
    const dim3 grid(balanced_grid(p.top * (p.n / 2), 3)), block(256);
    if (!one_launch_is_faster(n_out, p.top, p.n, p.k, (int)grid.x)) return MUI_ERR_UNSUPPORTED;
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, block, 0, s, logits, (const uint16_t*)corr, p.x, n_out, p.k, p.w0, p.w1, n_experts, p.top, p.expert_stride, p.n, p.limit,
                         (uint16_t*)p.y, expert, weight, pairs, tiles, p.max_tiles);
      return launch_status();
    };
    if (p.k <= 256 * 8) return p.once ? launch(moe_one_gateup_kernel<T, 1, true>) : launch(moe_one_gateup_kernel<T, 1, false>);
    return p.once ? launch(moe_one_gateup_kernel<T, 2, true>) : launch(moe_one_gateup_kernel<T, 2, false>);
  }
}

}  // namespace mui

extern "C" int mui_moe_route_gateup(mui_stream_t stream, int dtype, const float* logits, const void* correction, int n_identity, const void* gate, const void* up,
                                    long expert_stride, const void* x, float limit, int tile_pairs, int32_t* expert, float* weight, int32_t* pairs, void* tiles,
                                    void* act, int n_experts, int n_inter, int k_in, int top, int tokens) {
  if (tile_pairs == 16 && tokens == 1) {
    MUI_CHECK_ARG(logits && gate && up && x && act && expert && weight && pairs && tiles && n_experts > 0 && n_identity >= 0 && n_inter > 0 && k_in > 0);
    MUI_CHECK_ARG(top > 0 && top <= n_experts + n_identity);
    MoeGemmParams p = {};
    p.w0 = (const uint16_t*)gate; p.w1 = (const uint16_t*)up; p.expert_stride = expert_stride; p.x = (const uint16_t*)x; p.y = act;
    p.n = n_inter; p.k = k_in; p.top = top; p.tokens = 1; p.limit = limit;
    p.max_tiles = mui_moe_max_tiles(1, top, n_experts, 16);
    p.once = read_once(n_experts, n_inter, k_in, gate, up);
    auto one = [&](auto t) {
      return launch_moe_one<decltype(t)>((hipStream_t)stream, p, logits, correction, n_experts + n_identity, n_experts, expert, weight, pairs, (MoeTile*)tiles);
    };
    const int st = dtype == MUI_DTYPE_F16 ? one(F16{}) : dtype == MUI_DTYPE_BF16 ? one(BF16{}) : MUI_ERR_UNSUPPORTED;
    if (st != MUI_ERR_UNSUPPORTED) return st;
  }
  const int st = mui_moe_route(stream, dtype, logits, correction, n_experts, n_identity, top, tokens, tile_pairs, expert, weight, pairs, tiles);
  if (st != MUI_OK) return st;
  return mui_moe_gateup(stream, dtype, gate, up, expert_stride, x, limit, expert, pairs, tiles, tile_pairs, act, n_experts, n_inter, k_in, top, tokens);
}

extern "C" int mui_moe_down(mui_stream_t stream, int dtype, const void* down, long expert_stride, const void* act,
                            const int32_t* expert, const int32_t* pairs, const void* tiles, int tile_pairs, void* out,
                            int n_experts, int n_out, int k_in, int top, int tokens) {
  MUI_CHECK_ARG(down && act && expert && out && n_experts > 0 && n_out > 0 && k_in > 0 && top > 0 && tokens > 0);
  MUI_CHECK_ARG(tile_pairs == 0 || (pairs && tiles));
  MoeGemmParams p = {};
  p.w0 = (const uint16_t*)down; p.expert_stride = expert_stride; p.x = (const uint16_t*)act; p.y = out; p.pairs = pairs;
  p.tiles = (const MoeTile*)tiles; p.n = n_out; p.k = k_in; p.top = top; p.tokens = tokens;
  p.max_tiles = mui_moe_max_tiles(tokens, top, n_experts, tile_pairs);
  p.once = read_once(n_experts, n_out, k_in, down, down);
  MUI_BY_DTYPE((launch_moe_product<TT, MOE_DOWN>((hipStream_t)stream, p, expert, n_experts, tokens * top, tile_pairs)));
}

namespace mui {
// Sizes that moe_one_down_kernel covers, else MUI_ERR_UNSUPPORTED (nothing launched)
template <typename T>
static int launch_moe_one_down(hipStream_t s, const MoeGemmParams& p, const int32_t* expert, int n_experts) {
  if (p.tokens != 1 || p.top > kWave || p.n % 8 || p.k % 8 || p.k < 768 || p.k > 2 * 256 * 8 || p.expert_stride % 8) return MUI_ERR_UNSUPPORTED;
  if (p.k < 1280 && (long)p.top * p.n >= 32768) return MUI_ERR_UNSUPPORTED;
  if (!aligned16(p.w0) || !aligned16(p.x) || (long)p.top * p.n >= (1L << 30)) return MUI_ERR_UNSUPPORTED;
  auto launch = [&](auto kernel, int rows) {
    hipLaunchKernelGGL(kernel, dim3(balanced_grid(p.top * (p.n / rows), 3)), dim3(256), 0, s, expert, p.x, p.top, n_experts, p.n, p.k, p.w0, p.expert_stride, (uint16_t*)p.y);
    return launch_status();
  };
  if (p.k <= 256 * 8) return p.once ? launch(moe_one_down_kernel<T, 1, 8, true>, 8) : launch(moe_one_down_kernel<T, 1, 8, false>, 8);
  return p.once ? launch(moe_one_down_kernel<T, 2, 4, true>, 4) : launch(moe_one_down_kernel<T, 2, 4, false>, 4);
}
}  // namespace mui

extern "C" int mui_moe_one_down(mui_stream_t stream, int dtype, const void* down, long expert_stride, const void* act, const int32_t* expert, const int32_t* pairs,
                                const void* tiles, int tile_pairs, void* out, int n_experts, int n_out, int k_in, int top) {
  if (tile_pairs == 16) {
    MUI_CHECK_ARG(down && act && expert && out && pairs && tiles && n_experts > 0 && n_out > 0 && k_in > 0 && top > 0);
    MoeGemmParams p = {};
    p.w0 = (const uint16_t*)down; p.expert_stride = expert_stride; p.x = (const uint16_t*)act; p.y = out; p.n = n_out; p.k = k_in; p.top = top; p.tokens = 1;
    p.once = read_once(n_experts, n_out, k_in, down, down);
    const int st = dtype == MUI_DTYPE_F16 ? launch_moe_one_down<F16>((hipStream_t)stream, p, expert, n_experts)
                   : dtype == MUI_DTYPE_BF16 ? launch_moe_one_down<BF16>((hipStream_t)stream, p, expert, n_experts) : MUI_ERR_UNSUPPORTED;
    if (st != MUI_ERR_UNSUPPORTED) return st;
  }
  return mui_moe_down(stream, dtype, down, expert_stride, act, expert, pairs, tiles, tile_pairs, out, n_experts, n_out, k_in, top, 1);
}
