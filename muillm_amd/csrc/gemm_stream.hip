// Linear layers for 17..128 tokens (batched decoding beyond 16 rows, short prompts); of int8 codes for 17..64.
//
// Bound by the weight stream, and by the tokens: a matrix is read once, but every workgroup reads all token rows again from L2.
// A CU's vector cache returns data in the order of the requests, whichever wave made them, and holds a few tens of KB of them:
// weights arrive at 27.5 KB per microsecond and CU (7 TB/s in all), token rows at 105, and the two times ADD UP, however far ahead
// either is requested and however the waves divide the loads (measured on 4096 x 14336 with one, the other and both; waves that
// load only weights beside waves that load only tokens change nothing). So a unit of work is wide in rows -- what it reads of the
// tokens, it reads for ROWS weight rows --, and where the matrix has too few rows to give every CU a wide unit, K is divided
// between workgroups: their fp32 partial outputs go through a workspace and a second kernel adds them in order (about 3 us
// and the bytes; down 4096 x 14336 at 32 tokens, 64 rows x a quarter of K instead of 16 rows x all of K).
//
// A step of 256 or 128 k-values of ROWS weight rows and all tokens is a stage of LDS (global_load_lds_dwordx4, rows of 512 or 256 bytes
// contiguous); three to eight stages, all but one of them on their way. One barrier per step: the loads of a step go into the
// stage that the barrier has freed. The waves divide a step by shares of 64 k-values, token tiles and (few tokens) row
// tiles; the shares' partial tiles meet in LDS at the end of a unit and are added in order. A workgroup takes the units blockIdx,
// blockIdx + grid, ...; the stages run on across units, so the next unit is on its way while the last one is added up.
//
// int8 codes lie in the stages as they are, half the bytes; a lane reads sixteen of a row at a time (their k-values are two of a token's chunks) and converts them for two
// matrix instructions. A scale per row is applied to the sums; the pairs of the group format, one per row and share, are part of the stage, and the weight is rounded to 16 bits.
//
// us at 32 tokens in bf16, tiled GEMM or 16-rows-per-workgroup kernel -> here: 6144 x 4096 20.7 -> 12.7, 4096 x 4096 15.0 -> 10.9,
// gate/up 14336 x 4096 42.6 -> 37.4, 4096 x 14336 47 -> 24.2, 2048 x 8192 25.8 -> 11.7, 128256 x 4096 226 -> 167; at 101
// tokens 24.3 -> 20.6, 19.6 -> 17.2, 49.3 -> 33.9, 33.2 -> 18.6, gate/up 8192 x 2048 (80 tokens) 22.9 -> 18.4.
#include "skinny.cuh"

namespace mui {

constexpr int kStreamWaves = 8;
constexpr int kStreamThreads = kStreamWaves * kWave;

struct StreamParams {
  const uint8_t* w0; const uint8_t* w1; long pitch;  // bytes
  const uint16_t* s0; const uint16_t* s1; long s_pitch; int group_shift;  // codes: as in SkinnyParams
  const uint16_t* x;
  const uint16_t* mul_bias; const uint16_t* add_bias; const uint16_t* residual;
  uint16_t* y;
  float* part;     // [k_splits][tokens][n] where K is divided between workgroups
  bool add;        // a launch behind this one adds the partial outputs up (else the caller's does)
  int n, k, tokens;
  int n_units;     // bands of ROWS weight rows (gate/up: gate and up rows together)
  int k_splits;    // more than one (16-bit weights): every workgroup has one unit, a share of K of one band
};

// Geometry for ROWS weight rows x NT token tiles of 16 per unit
template <int ROWS, int NT, int WF>
struct StreamShape {
  static constexpr bool W8 = WF != WF_16BIT;  // codes
  static constexpr int KS = W8 || ROWS + 16 * NT <= 96 ? 256 : 128;  // k-values per step: at least three stages fit
  static constexpr int KSH = KS / 64;                              // shares of a step
  static constexpr int RT = (ROWS + 15) / 16;
  static constexpr int GROUPS = kStreamWaves / KSH;
  // groups of token tiles (six tiles: two waves only load). Codes are converted by every group, so there is one where there are row tiles to deal out
  static constexpr int GT = W8 && RT > 1 ? 1 : NT == 2 ? 2 : NT == 6 ? 3 : GROUPS;
  static constexpr int GR = GROUPS / GT;                           // groups of row tiles
  static constexpr int TW = NT / GT, RW = (RT + GR - 1) / GR;      // token and row tiles per wave
  static constexpr int RPI = 512 / KS, WRPI = W8 ? 2 * RPI : RPI;  // token and weight rows per load instruction (1 KB)
  static constexpr int W_INSTR = ROWS / WRPI, X_INSTR = 16 * NT / RPI, P_INSTR = WF == WF_U8_GROUP ? RT : 0, INSTR = W_INSTR + X_INSTR + P_INSTR;
  static constexpr int ROW_BYTES = KS * 2, WROW_BYTES = W8 ? KS : KS * 2;
  static constexpr int Q = (INSTR + kStreamWaves - 1) / kStreamWaves;  // load instructions per wave and step (at most)
  static constexpr int FULL = INSTR - (Q - 1) * kStreamWaves;      // waves that have Q of them, the others Q - 1
  static constexpr int PAIRS = ROWS * WROW_BYTES + 16 * NT * ROW_BYTES;  // where a stage's (scale, min) pairs are: one per row and share
  static constexpr int STAGE = PAIRS + P_INSTR * 256;
  static constexpr int MOST_MEET = WF == WF_U8_GROUP && NT == 4 ? 3 : 16 / KSH;  // (three stages and what meets have to fit)
  static constexpr int MEET = RT * NT < MOST_MEET ? RT * NT : MOST_MEET;  // tiles that meet at a time (KSH KB each)
  static constexpr int FIT = (160 * 1024 - MEET * KSH * 1024) / STAGE;
  static constexpr int S = FIT < 8 ? FIT : 8;
  static constexpr int LDS = S * STAGE + MEET * KSH * 1024;
  // row tiles read past the weights' rows (a half tile's other half, a last row group's spare tile) read token rows of the stage
  static_assert(GR * RW * 16 * WROW_BYTES <= STAGE, "a wave's rows lie in its stage");
  static_assert(S >= 3 && (S - 2) * Q <= 63 && ROWS % 8 == 0 && TW * GT == NT && GR >= 1, "shape");
};

extern __shared__ __align__(16) unsigned char st_smem[];

template <int AUX>
__device__ __forceinline__ void stream_load16(const uint8_t* base, unsigned off, unsigned char* dst) {
  asm volatile("" : "+v"(off));  // (kept a 32-bit lane offset from a scalar base)
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + off),
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, AUX);
}

// wait until at most `steps` steps' loads (Q each) are outstanding; steps beyond MOST count as MOST
template <int MOST, int Q>
__device__ __forceinline__ void stream_wait_steps(int steps) {
  if constexpr (MOST > 0) {
    if (steps >= MOST) wait_loads<MOST * Q>();
    else stream_wait_steps<MOST - 1, Q>(steps);
  } else {
    wait_loads<0>();
  }
}

template <typename T, int EPI, int ROWS, int NT, int WF>
__global__ void __launch_bounds__(kStreamThreads, 2) gemm_stream_kernel(const StreamParams p) {
  using G = StreamShape<ROWS, NT, WF>;
  constexpr bool W8 = G::W8;
  constexpr int KS = G::KS, KSH = G::KSH, RT = G::RT, TW = G::TW, RW = G::RW, RPI = G::RPI, WRPI = G::WRPI, S = G::S, MEET = G::MEET;
  constexpr int CPR = KS / 8, WCPR = W8 ? KS / 16 : CPR;  // 16-byte chunks per row of a stage
  constexpr int ROW_BYTES = G::ROW_BYTES, WROW_BYTES = G::WROW_BYTES;
  const int t = threadIdx.x, lane = t & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  f32x4* meet = (f32x4*)(st_smem + S * G::STAGE);

  // this lane's place in a load instruction: row lr of RPI, chunk ls. Chunk c of row r lives in slot c ^ (r % 16) (16 rows
  // read at one chunk fall into 16 different bank groups); the row's upper bits come with the instruction.
  const int lr = lane / CPR, ls = (lane % CPR) ^ lr;
  const int wlr = W8 ? lane / WCPR : lr, wls = W8 ? (lane % WCPR) ^ wlr : ls;

  const int all_steps = p.k / KS;
  const int k_splits = W8 ? 1 : p.k_splits;
  const int share_k = k_splits > 1 ? (int)(blockIdx.x % (unsigned)k_splits) : 0;
  const int first_unit = k_splits > 1 ? (int)(blockIdx.x / (unsigned)k_splits) : (int)blockIdx.x;
  const int sb = (int)((long)all_steps * share_k / k_splits);
  const int unit_steps = (int)((long)all_steps * (share_k + 1) / k_splits) - sb;
  const int units = k_splits > 1 ? 1 : (p.n_units - first_unit + (int)gridDim.x - 1) / (int)gridDim.x;
  const int steps = unit_steps * units;
  // workgroups start at different steps: their rows are whole multiples of the memory channels' interleave apart, so
  // workgroups that walked K in step would all ask the same channels (reads of a matrix 6.0 -> 6.9 TB/s)
  const int turn = (int)((blockIdx.x >> 3) % (unsigned)unit_steps);

  // the step that is loaded next
  int lu = first_unit, lc = 0, lslot = 0;
  auto load_next = [&]() {
    const int turned = lc + turn < unit_steps ? lc + turn : lc + turn - unit_steps;
    const long kb = (long)(sb + turned) * ROW_BYTES, kbw = W8 ? kb / 2 : kb;
    const int row0 = lu * ROWS;
    unsigned char* stage = st_smem + lslot * G::STAGE;
#pragma unroll
    for (int q = 0; q < G::Q; ++q) {
      const int i = q * kStreamWaves + wave;
      if (q == G::Q - 1 && G::FULL < kStreamWaves && wave >= G::FULL) continue;
      if (i < G::W_INSTR) {
        const int r = i * WRPI;  // weight rows r .. r + WRPI of the stage
        const uint8_t* base;
        if constexpr (EPI == SK_GATEUP) {  // a tile of 16 rows: eight gate rows, then the up rows of the same outputs
          int o = (row0 >> 1) + (r >> 4) * 8 + (r & 7);
          o = o < p.n - WRPI ? o : p.n - WRPI;  // (past the matrix: rows that are there, never stored)
          base = ((r & 8) ? p.w1 : p.w0) + (long)o * p.pitch;
        } else {
          const int o = row0 + r < p.n - WRPI ? row0 + r : p.n - WRPI;
          base = p.w0 + (long)o * p.pitch;
        }
        stream_load16<2>(base + kbw, (unsigned)(wlr * (unsigned)p.pitch) + (unsigned)((wls ^ (r & 15)) * 16), stage + r * WROW_BYTES);  // non-temporal
      } else if (G::P_INSTR > 0 && i >= G::W_INSTR + G::X_INSTR) {
        // pairs of a tile of 16 rows: lane 4 row + share
        const int tile = i - G::W_INSTR - G::X_INSTR, tr = lane >> 2;
        int o;
        if constexpr (EPI == SK_GATEUP) o = (row0 >> 1) + tile * 8 + (tr & 7);
        else o = row0 + tile * 16 + tr;
        o = o < p.n ? o : p.n - 1;
        const long at = (long)o * p.s_pitch + 2 * (((sb + turned) * KS + (lane & 3) * 64) >> p.group_shift);
        const uint16_t* pair = (EPI == SK_GATEUP && (tr & 8) ? p.s1 : p.s0) + at;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)pair,
                                         (__attribute__((address_space(3))) void*)(stage + G::PAIRS + tile * 256), 4, 0, 0);
      } else {
        const int tr = (i - G::W_INSTR) * RPI;  // tokens past the end read the last one
        const int rb = tr < p.tokens ? tr : p.tokens - 1, most = p.tokens - 1 - rb;
        const int tk = lr < most ? lr : most;
        stream_load16<0>((const uint8_t*)p.x + (long)rb * p.k * 2 + kb, (unsigned)(tk * p.k * 2) + (unsigned)((ls ^ (tr & 15)) * 16),
                         stage + ROWS * WROW_BYTES + tr * ROW_BYTES);
      }
    }
    lslot = lslot + 1 == S ? 0 : lslot + 1;
    if (++lc == unit_steps) { lc = 0; lu += (int)gridDim.x; }
  };

  // operand reads: lane l takes row l % 16 of a tile, chunk 8 share + l / 16 (+ 4); int8: the 16 codes of chunk 4 share + l / 16 and the tokens' two chunks of the
  // same k-values
  const int share = wave % KSH, group = wave / KSH;
  const int gt = group % G::GT, gr = group / G::GT;
  const int rr = lane & 15, rc = share * 8 + (W8 ? 2 * (lane >> 4) : lane >> 4);
  const int ro0 = rr * ROW_BYTES + ((rc ^ rr) * 16), ro1 = rr * ROW_BYTES + (((rc + (W8 ? 1 : 4)) ^ rr) * 16);
  const int wo = rr * WROW_BYTES + (((share * 4 + (lane >> 4)) ^ rr) * 16);
  const bool multiplies = gr < G::GR;

  f32x4 acc[RW][TW];
#pragma unroll
  for (int i = 0; i < RW; ++i)
#pragma unroll
    for (int j = 0; j < TW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int s = 0; s < S - 1 && s < steps; ++s) load_next();
  int slot = 0, c = 0, u = first_unit;
  for (int s = 0; s < steps; ++s) {
    const int left = steps - s;
    // this wave's part of step s has landed: what is outstanding belongs to the steps behind it
    if (G::FULL == kStreamWaves || wave < G::FULL) stream_wait_steps<S - 2, G::Q>(left - 1);
    else stream_wait_steps<S - 2, G::Q - 1>(left - 1);
    __builtin_amdgcn_s_barrier();  // ... and everybody's, and everybody has read step s - 1: its stage is free
    asm volatile("" ::: "memory");
    if (S - 1 < left) load_next();
    if (multiplies) {
      const unsigned char* ws = st_smem + slot * G::STAGE + gr * RW * 16 * WROW_BYTES;
      const unsigned char* xs = st_smem + slot * G::STAGE + ROWS * WROW_BYTES + gt * TW * 16 * ROW_BYTES;
      u32x4 b[TW][2];
#pragma unroll
      for (int j = 0; j < TW; ++j) {
        b[j][0] = *(const u32x4*)(xs + j * 16 * ROW_BYTES + ro0);
        b[j][1] = *(const u32x4*)(xs + j * 16 * ROW_BYTES + ro1);
      }
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        u32x4 a0, a1;
        if constexpr (W8) {
          const u32x4 codes = *(const u32x4*)(ws + i * 16 * WROW_BYTES + wo);
          if constexpr (WF == WF_U8_GROUP) {
            const uint32_t pair = *(const uint32_t*)(st_smem + slot * G::STAGE + G::PAIRS + ((gr * RW + i) * 16 + rr) * 16 + share * 4);
            if constexpr (T::kDtype == MUI_DTYPE_F16) {
              a0 = convert_a_pair_f16(codes.x, codes.y, pair);
              a1 = convert_a_pair_f16(codes.z, codes.w, pair);
            } else {
              a0 = convert_a_pair<T>(codes.x, codes.y, pair);
              a1 = convert_a_pair<T>(codes.z, codes.w, pair);
            }
          } else {
            a0 = convert_a<T, WF_I8_CHANNEL>(codes.x, codes.y, nullptr, 0, 0);
            a1 = convert_a<T, WF_I8_CHANNEL>(codes.z, codes.w, nullptr, 0, 0);
          }
        } else {
          a0 = *(const u32x4*)(ws + i * 16 * ROW_BYTES + ro0);
          a1 = *(const u32x4*)(ws + i * 16 * ROW_BYTES + ro1);
        }
#pragma unroll
        for (int j = 0; j < TW; ++j) {
          acc[i][j] = mfma16x16x32<T>(a0, b[j][0], acc[i][j]);
          acc[i][j] = mfma16x16x32<T>(a1, b[j][1], acc[i][j]);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    slot = slot + 1 == S ? 0 : slot + 1;
    if (++c < unit_steps) continue;
    // ---- end of a unit: the shares' partial tiles meet, MEET tiles at a time; wave w finishes tile w of a round
    const int row0 = u * ROWS;
    c = 0;
    u += (int)gridDim.x;
#pragma unroll
    for (int r0 = 0; r0 < RT * NT; r0 += MEET) {
      if (r0 > 0) {
        __builtin_amdgcn_s_barrier();  // the round before has been read
        asm volatile("" ::: "memory");
      }
      if (multiplies) {
#pragma unroll
        for (int i = 0; i < RW; ++i)
#pragma unroll
          for (int j = 0; j < TW; ++j) {
            const int id = (gr * RW + i) * NT + gt * TW + j;
            if (id >= r0 && id < r0 + MEET && gr * RW + i < RT) meet[((id - r0) * KSH + share) * 64 + lane] = acc[i][j];
          }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const int id = r0 + wave;
      if (wave < MEET && id < RT * NT) {
        const int i = id / NT, j = id % NT;
        const f32x4* in = meet + wave * KSH * 64;
        const int tok = 16 * j + (lane & 15), sub = lane >> 4;  // acc[e]: row 4 sub + e of the tile
        if constexpr (EPI == SK_GATEUP) {
          // rows 0-7 of a tile are gate rows, 8-15 the up rows of the same outputs
          const int o = (row0 >> 1) + 8 * i + 4 * (sub & 1);
          f32x4 g = in[lane & 31], h = in[(lane & 31) + 32];
#pragma unroll
          for (int w = 1; w < KSH; ++w) {
            g += in[w * 64 + (lane & 31)];
            h += in[w * 64 + (lane & 31) + 32];
          }
          if (lane < 32 && tok < p.tokens && o < p.n && 16 * i < ROWS) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float gv = g[e], uv = h[e];
              if constexpr (WF == WF_I8_CHANNEL) {
                gv *= T::one(p.s0[(o + e) * p.s_pitch]);
                uv *= T::one(p.s1[(o + e) * p.s_pitch]);
              }
              if (p.add_bias) {
                gv += T::one(p.add_bias[o + e]);
                uv += T::one(p.mul_bias[o + e]);
              }
              v[e] = gateup_f32(gv, uv);
            }
            u32x2 pk;
            pk.x = (uint32_t)T::pack(v[0]) | ((uint32_t)T::pack(v[1]) << 16);
            pk.y = (uint32_t)T::pack(v[2]) | ((uint32_t)T::pack(v[3]) << 16);
            *(u32x2*)(p.y + (long)tok * p.n + o) = pk;
          }
        } else {
          const int o = row0 + 16 * i + 4 * sub;
          f32x4 a = in[lane];
#pragma unroll
          for (int w = 1; w < KSH; ++w) a += in[w * 64 + lane];
          if (tok < p.tokens && o < p.n && 16 * i + 4 * sub < ROWS) {
            if constexpr (WF == WF_I8_CHANNEL) {
#pragma unroll
              for (int e = 0; e < 4; ++e) a[e] *= T::one(p.s0[(o + e) * p.s_pitch]);
            }
            if (k_splits > 1) {
              *(f32x4*)(p.part + ((long)share_k * p.tokens + tok) * p.n + o) = a;
            } else {
              float res[4] = {0.f, 0.f, 0.f, 0.f};
              if (p.residual) {
                const u32x2 q = ld8(p.residual + (long)tok * p.n + o);
                res[0] = T::one((uint16_t)(q.x & 0xffffu)); res[1] = T::one((uint16_t)(q.x >> 16));
                res[2] = T::one((uint16_t)(q.y & 0xffffu)); res[3] = T::one((uint16_t)(q.y >> 16));
              }
              float v[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                v[e] = a[e];
                if (p.mul_bias) v[e] *= T::one(p.mul_bias[o + e]);
                if (p.add_bias) v[e] += T::one(p.add_bias[o + e]);
                if (p.residual) v[e] += res[e];
              }
              u32x2 pk;
              pk.x = (uint32_t)T::pack(v[0]) | ((uint32_t)T::pack(v[1]) << 16);
              pk.y = (uint32_t)T::pack(v[2]) | ((uint32_t)T::pack(v[3]) << 16);
              *(u32x2*)(p.y + (long)tok * p.n + o) = pk;
            }
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
#pragma unroll
    for (int i = 0; i < RW; ++i)
#pragma unroll
      for (int j = 0; j < TW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// adds the partial outputs of the shares of K in order and applies what a linear's end applies; four outputs per thread
template <typename T>
__global__ void __launch_bounds__(256) gemm_stream_add_kernel(const StreamParams p) {
  const long at = ((long)blockIdx.x * 256 + threadIdx.x) * 4, all = (long)p.tokens * p.n;
  if (at >= all) return;
  f32x4 a = *(const f32x4*)(p.part + at);
  for (int s = 1; s < p.k_splits; ++s) a += *(const f32x4*)(p.part + s * all + at);
  const int o = (int)(at % p.n);
  float v[4] = {a.x, a.y, a.z, a.w};
  u32x2 q = {0u, 0u};
  if (p.residual) q = ld8(p.residual + at);
  const uint32_t q0 = q.x, q1 = q.y;
  const float res[4] = {T::lo(q0), T::hi(q0), T::lo(q1), T::hi(q1)};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (p.mul_bias) v[e] *= T::one(p.mul_bias[o + e]);
    if (p.add_bias) v[e] += T::one(p.add_bias[o + e]);
    if (p.residual) v[e] += res[e];
  }
  u32x2 pk;
  pk.x = (uint32_t)T::pack(v[0]) | ((uint32_t)T::pack(v[1]) << 16);
  pk.y = (uint32_t)T::pack(v[2]) | ((uint32_t)T::pack(v[3]) << 16);
  *(u32x2*)(p.y + at) = pk;
}

static unsigned add_blocks(int tokens, int n) { return (unsigned)(((long)tokens * n / 4 + 255) / 256); }

template <typename T, int EPI, int ROWS, int NT, int WF>
static int launch_stream_cfg(hipStream_t s, const StreamParams& p) {
  using G = StreamShape<ROWS, NT, WF>;
  static_assert(G::LDS <= 160 * 1024, "LDS of a workgroup");
  const int cus = device_cus(), wgs = p.n_units * p.k_splits;
  const int st = launch_with_lds(gemm_stream_kernel<T, EPI, ROWS, NT, WF>, dim3(wgs < cus ? wgs : cus), dim3(kStreamThreads), G::LDS, s, p);
  if (WF != WF_16BIT || st != MUI_OK || p.k_splits == 1 || !p.add) return st;
  hipLaunchKernelGGL(gemm_stream_add_kernel<T>, dim3(add_blocks(p.tokens, p.n)), dim3(256), 0, s, p);
  return launch_status();
}

// token tiles of 16 per unit
static int stream_token_tiles(int tokens) { return tokens <= 32 ? 2 : tokens <= 64 ? 4 : tokens <= 96 ? 6 : 8; }
constexpr int stream_widest(int nt) { return 192 - 16 * nt < 128 ? 192 - 16 * nt : 128; }  // rows with three stages of 128 k-values
template <int EPI, int WF>
constexpr bool stream_built(int rows, int nt) {
  if (WF != WF_16BIT) return nt == 2 ? rows <= 112 : nt == 4 && rows <= 64;  // (three stages of 256 k-values)
  return rows <= stream_widest(nt) && (EPI == SK_LINEAR || nt <= 4 || rows == 48 || rows == 64);
}

template <typename T, int EPI, int ROWS, int WF>
static int launch_stream_rows(hipStream_t s, const StreamParams& p) {
  switch (stream_token_tiles(p.tokens)) {
    case 2: if constexpr (stream_built<EPI, WF>(ROWS, 2)) return launch_stream_cfg<T, EPI, ROWS, 2, WF>(s, p); break;
    case 4: if constexpr (stream_built<EPI, WF>(ROWS, 4)) return launch_stream_cfg<T, EPI, ROWS, 4, WF>(s, p); break;
    case 6: if constexpr (stream_built<EPI, WF>(ROWS, 6)) return launch_stream_cfg<T, EPI, ROWS, 6, WF>(s, p); break;
    default: if constexpr (stream_built<EPI, WF>(ROWS, 8)) return launch_stream_cfg<T, EPI, ROWS, 8, WF>(s, p); break;
  }
  return MUI_ERR_UNSUPPORTED;
}

// Whether the tiled GEMM of longer prompts is faster than linear units of `width` rows x all of K: from 65 tokens on a narrow unit takes longer for its
// token rows than for its weights, and the tiles read tokens less often. The tiles' time over this kernel's on 250 matrices, 17 to 128 tokens:
// up to 64 tokens 1.04 to 2, one round of units of 40 rows or more 1.02 to 1.4, and else, by K:
//   8, 16 rows      65 tokens 1.17 at 1024, 1.0 at 14336; 96 tokens 1.10 at 1024, 1.0 at 4096, 0.93 at 14336; 97 .. 128 tokens 1.03 at 2048, 0.95 at 3072, 0.85 at 28672
//   24, 32 rows     up to 104 tokens 1.0 to 1.4; 128 tokens 1.2 at 1024, 1.0 at 4096, 0.91 at 28672
//   several rounds  65 .. 96 tokens 0.86 to 1.05 (28672, 32000 rows), 97 .. 128 tokens 0.81 to 1.05 (28672 to 50304 rows)
// Of several rounds those stay whose rows are whole multiples of 4 KB apart, which slows the tiles, with a last round that is nearly full: 1.0 to 1.25 where the units
// are as wide as they can be (40960 to 151936 rows) or the rows a multiple of 8192.
static bool tiles_are_faster(int tokens, int rows, int k, int width, int rounds) {
  if (tokens <= 64) return false;
  const bool most = tokens > 96;
  if (rounds > 1) {
    const long full = (long)rounds * device_cus() * width;
    if (k % 2048 || k > 8192 || width < 64) return true;
    return most ? rows % 8192 || rounds > 4 || rows * 20L < full * 19 : (width < 96 && rows % 8192) || rows * 5L < full * 4;
  }
  if (width <= 16) return most ? k > 2560 : (long)(tokens - 56) * k > 130000;
  return width <= 32 && tokens > 104 && (long)(tokens - 80) * k > 240000;
}

// Whether the 16-rows-per-workgroup kernel (gemm_wide.hip, one round of workgroups, up to 40 tokens) is faster than linear units: a ring of stages pays from a few
// steps on. Its time over this kernel's, up to 4096 rows: K 256 0.79 to 1.01; K 512 17 to 24 tokens 0.82 to 0.98 up to 2048 rows and 0.94 to 1.05 at 4096, 25 to 32
// tokens 0.95 to 1.02 and 1.02 to 1.08, 33 tokens 0.99 to 1.10; K 768 and more 0.98 to 1.4.
static bool wide_is_faster(int tokens, int rows, int k) {
  if (tokens > 40 || ceil_div(rows, 16) > device_cus()) return false;
  return k <= 256 || (k <= 512 && tokens <= 32 && rows <= 8 * device_cus());
}

// And the tiled GEMM against units of gate and up rows. Both take matrices in rounds, units 112 rows per CU at most, tiles 128. Where units need a round more they
// are slower beyond 32 tokens, but for rows that are whole multiples of 4 KB apart, which slows the tiles (us at 33 to 64 tokens, tiles / units: 14400 to 15600 outputs, K 512 12.5 to 14.1 / 12.6 to 14.2, 1024
// 17.5 to 18.9 / 18.0 to 20.0, 2048 28.8 to 35 / 29 to 31, 4096 48 to 59 / 48 to 55, 5120 57 to 60 / 63 to 69, 8192 87 to 117 / 98 to 106; 30000 outputs, K 512 23 to 24 / 22 to 23, 4096
// 93 to 114 / 96 to 105, 5120 111 to 125 / 124 to 144, 8192 183 to 222 / 182 to 189); elsewhere units take 0.63 to 1.02 of the tiles' time.
// Beyond 64 tokens units have 48 or 64 rows (what three stages leave room for): one round of those up to 16384 rows, us, tiles / units at 65 / 96 / 128 tokens: 8192 x 2048
// 20.5 / 17.5, 22.4 / 19.4, 22.3 / 21.1, 8192 x 4096 33.7 / 28.7, 34.7 / 30.5, 36.7 / 34.3, 6144 x 4096 31.1 / 25.4, 32.1 / 26.7, 33.9 / 30.2, 4096 x 2048 29.4 / 14.9, 30.3 /
// 15.6, 31.3 / 17.4. Two rounds read the tokens twice: 14336 x 4096 at 128 tokens 64 us, tiles 55.
static bool gateup_tiles_are_faster(int tokens, int rows, int k, int units) {
  const int cus = device_cus();
  if (tokens > 64) return units > cus;
  return tokens > 32 && k > 512 && k % 2048 && ceil_div(rows, 112 * cus) > ceil_div(rows, 128 * cus);
}

// Codes: what the other int8 kernels keep. Up to 32 tokens with a scale per row the 16-rows-per-workgroup kernel where it takes the matrix in one round and K is short for the
// number of tokens (us, that / bands: 4096 x 4096 at 20 / 24 / 32 tokens 10.0 / 10.8, 10.7 / 10.9, 12.2 / 11.2; 2048 x 8192 16.4 / 17.4, 17.7 / 17.5, 20.3 / 17.9; 3072 x 2048
// at 32 7.2 / 7.6; 4096 x 14336 at 17 / 24 26.1 / 26.9, 29.5 / 26.7; 4096 x 256 and x 512
// at 33 3.8 / 4.1, 4.8 / 4.8, 2048 x 1024 6.3 / 5.8); beyond 32 tokens several rounds (gate/up 14336 x 4096 at 64 tokens 41 / 44); groups in
// bf16 bands of 112 rows (14336 x 4096 at 32 41.8 / 42.8: a pair for every 64 codes is as many cache lines as the codes). Everywhere else the bands: per row,
// 6144 x 4096 at 17 / 32 / 64 tokens 21.5 / 12.0, 21.7 / 12.4, 21.9 / 15.4, 4096 x 14336 at 32 / 33 / 64 33.8 / 27.2, 54.0 / 31.8, 58.8 / 34.6, gate/up 14336 x 4096 at 32 40.3 / 27.2,
// 8192 x 2048 21.3 / 11.8 and at 64 21.2 / 16.4; groups of 128, 6144 x 4096 at 32 22.5 / 13.5, 4096 x 14336 62.8 / 33.0, 2048 x 2048 13.6 / 8.4, gate/up 8192 x 2048 21.7 / 15.8.
static bool codes_are_faster_elsewhere(bool groups, bool bf16, int epi, int tokens, int rows, int k, int width, int units) {
  const int cus = device_cus();
  const bool wide = !groups && epi == SK_LINEAR && ceil_div(rows, 16) <= cus;
  if (tokens > 32) return units > cus || (wide && tokens <= 40 && k <= 512);
  return groups ? bf16 && width == 112 : wide && (long)(tokens - 16) * k < 49152;
}

static int g_stream_rows = 0, g_stream_shares = 0;  // mui_tune_stream

// (forced units that do not exist are an error, but where the kernel has none for the call at all)
template <int EPI, int WF>
static bool stream_forced_must_exist(int tokens) { return WF == WF_16BIT && (EPI == SK_LINEAR || stream_token_tiles(tokens) <= 4); }

// The time of the units that it chooses in us, or a negative number where another kernel is faster or, with forced units, none exist (*width 0 then)
template <typename T, int EPI, int WF>
static float plan_stream(StreamParams& p, size_t part_bytes, int* chosen) {
  constexpr bool W8 = WF != WF_16BIT;
  // Rows per unit and shares of K by the least time: what a CU takes in (27.5 KB of weights, 105 KB of token rows per microsecond, 82 in
  // steps of 128 k-values), a barrier per step, a fixed part per round of workgroups; for shares of K the second launch and the
  // partial outputs, written and read. Measured against every other pair at 17 to 128 tokens on matrices from 2048 x 2048 to 128256 x 4096 it
  // is within 5 % of the best: 4096 x 4096 takes 16 rows x all of K (10.9 us at 32 tokens; 64 rows x a quarter 12.1), 4096 x 14336 64 x a
  // quarter (24.2; 16 rows x all 32.3), 2048 x 8192 32 x a quarter (11.6; 8 x all 16.3).
  constexpr int kLinear[] = {128, 96, 64, 56, 48, 40, 32, 24, 16, 8}, kGateup[] = {112, 96, 64, 48, 32, 16};
  const int rows = EPI == SK_GATEUP ? 2 * p.n : p.n, cus = device_cus(), nt = stream_token_tiles(p.tokens);
  const int tried = EPI == SK_GATEUP ? 6 : 10;
  float best = 0.f;
  int width = 0;
  for (int c = 0; c < tried; ++c) {
    const int r = EPI == SK_GATEUP ? kGateup[c] : kLinear[c];
    if (!stream_built<EPI, WF>(r, nt) || (g_stream_rows && r != g_stream_rows)) continue;
    const int units = ceil_div(rows, r);
    for (int k = 1; k <= 8; ++k) {
      if (k > 1 && (W8 || (long)units * k > cus || (size_t)k * p.tokens * p.n * 4 > part_bytes || p.k / 256 < 2 * k)) break;
      if (g_stream_shares && k != g_stream_shares) continue;
      const float one = (float)p.k / k * 2.f * ((float)r / (W8 ? 55e3f : 27.5e3f) + 16.f * nt / (nt > 4 ? 82e3f : 105e3f));
      const float barriers = (float)p.k / k / (W8 || r + 16 * nt <= 96 ? 256 : 128) * 0.08f;
      const float cost = ceil_div(units, cus) * (one + barriers + 1.f) + (k > 1 ? 2.5f + 0.3f * k + (float)k * p.tokens * p.n * 8.f / 4e6f : 0.f);
      if (width == 0 || cost < best) { best = cost; width = r; p.n_units = units; p.k_splits = k; }
    }
  }
  *chosen = width;
  const bool forced = g_stream_rows || g_stream_shares;
  if ((!p.add && p.k_splits == 1) || !width) return -1.f;
  if (forced) return best;
  if constexpr (W8) {
    if (codes_are_faster_elsewhere(WF == WF_U8_GROUP, T::kDtype == MUI_DTYPE_BF16, EPI, p.tokens, rows, p.k, width, p.n_units)) return -1.f;
  } else if constexpr (EPI == SK_GATEUP) {
    if (gateup_tiles_are_faster(p.tokens, rows, p.k, p.n_units)) return -1.f;
  } else {
    if (wide_is_faster(p.tokens, rows, p.k)) return -1.f;
    if (p.k_splits == 1 && tiles_are_faster(p.tokens, rows, p.k, width, ceil_div(p.n_units, cus))) return -1.f;
  }
  return best;
}

template <typename T, int EPI, int WF = WF_16BIT>
static int launch_stream_t(hipStream_t s, StreamParams p, size_t part_bytes, int* splits = nullptr) {
  int width = 0;
  const float us = plan_stream<T, EPI, WF>(p, part_bytes, &width);
  if (splits) *splits = p.k_splits;
  if (us < 0.f) return (g_stream_rows || g_stream_shares) && p.add && !width && stream_forced_must_exist<EPI, WF>(p.tokens) ? MUI_ERR_INVALID_ARG : MUI_ERR_UNSUPPORTED;
  switch (width) {
    case 16: return launch_stream_rows<T, EPI, 16, WF>(s, p);
    case 32: return launch_stream_rows<T, EPI, 32, WF>(s, p);
    case 48: return launch_stream_rows<T, EPI, 48, WF>(s, p);
    case 64: return launch_stream_rows<T, EPI, 64, WF>(s, p);
    case 96: return launch_stream_rows<T, EPI, 96, WF>(s, p);
  }
  if constexpr (EPI == SK_LINEAR) {
    switch (width) {
      case 8: return launch_stream_rows<T, EPI, 8, WF>(s, p);
      case 24: return launch_stream_rows<T, EPI, 24, WF>(s, p);
      case 40: return launch_stream_rows<T, EPI, 40, WF>(s, p);
      case 56: return launch_stream_rows<T, EPI, 56, WF>(s, p);
      case 128: return launch_stream_rows<T, EPI, 128, WF>(s, p);
    }
  } else if (width == 112) {
    return launch_stream_rows<T, EPI, 112, WF>(s, p);
  }
  return MUI_ERR_UNSUPPORTED;
}

// what the loads cannot serve
static bool stream_serves(const SkinnyParams& q, int most, bool w8 = false) {
  if (q.tokens < 1 || q.tokens > most || q.gamma || (q.x_pitch != 0 && q.x_pitch != q.k)) return false;
  if (q.k % 256 || q.n % 8 || q.n < 8 || q.pitch % (w8 ? 16 : 8) || q.pitch > (1L << 26)) return false;
  return !((((uintptr_t)q.w0 | (uintptr_t)q.w1 | (uintptr_t)q.x) & 15) || (((uintptr_t)q.y | (uintptr_t)q.residual) & 7));
}

static StreamParams stream_params(const SkinnyParams& q, float* part, bool add, bool w8 = false) {
  StreamParams p = {};
  p.w0 = (const uint8_t*)q.w0; p.w1 = (const uint8_t*)q.w1; p.pitch = q.pitch * (w8 ? 1 : 2);
  p.s0 = q.s0; p.s1 = q.s1; p.s_pitch = q.s_pitch; p.group_shift = q.group_shift;
  p.x = q.x; p.mul_bias = q.mul_bias; p.add_bias = q.add_bias; p.residual = q.residual; p.y = q.y;
  p.n = q.n; p.k = q.k; p.tokens = q.tokens; p.part = part; p.k_splits = 1; p.add = add;
  return p;
}

// (pairs are read in fours of bytes)
static bool stream_serves_codes(const SkinnyParams& q, int wf) {
  if (!stream_serves(q, 64, true)) return false;
  if (wf == WF_I8_CHANNEL) return true;
  return wf == WF_U8_GROUP && q.group_shift >= 6 && q.k % (1 << q.group_shift) == 0 && q.s_pitch % 2 == 0 && (((uintptr_t)q.s0 | (uintptr_t)q.s1) & 3) == 0;
}

template <typename T, int WF>
static float stream_time_t(int epilogue, StreamParams p, size_t part_bytes) {
  int width = 0;
  return epilogue == SK_GATEUP ? plan_stream<T, SK_GATEUP, WF>(p, 0, &width) : plan_stream<T, SK_LINEAR, WF>(p, part_bytes, &width);
}

// What the launches below take in us, by the plan that chooses their units, or a negative number for what they decline
float gemm_stream_time(int dtype, int wf, int epilogue, const SkinnyParams& q, size_t part_bytes) {
  if (!(wf == WF_16BIT ? stream_serves(q, 128) : stream_serves_codes(q, wf))) return -1.f;
  const StreamParams p = stream_params(q, nullptr, true, wf != WF_16BIT);
  auto of = [&](auto t) {
    using T = decltype(t);
    return wf == WF_16BIT ? stream_time_t<T, WF_16BIT>(epilogue, p, part_bytes)
           : wf == WF_I8_CHANNEL ? stream_time_t<T, WF_I8_CHANNEL>(epilogue, p, 0) : stream_time_t<T, WF_U8_GROUP>(epilogue, p, 0);
  };
  return dtype == MUI_DTYPE_F16 ? of(F16{}) : dtype == MUI_DTYPE_BF16 ? of(BF16{}) : -1.f;
}

// 17..128 tokens, 16-bit weights, no fused norm, x / residual / y dense; MUI_ERR_UNSUPPORTED for what the loads cannot serve and for
// what another kernel does faster
int launch_gemm_stream(hipStream_t s, int dtype, int epilogue, const SkinnyParams& q, float* part, size_t part_bytes) {
  if (!stream_serves(q, 128)) return MUI_ERR_UNSUPPORTED;
  const StreamParams p = stream_params(q, part, true);
  if (dtype == MUI_DTYPE_F16) return epilogue == SK_GATEUP ? launch_stream_t<F16, SK_GATEUP>(s, p, 0) : launch_stream_t<F16, SK_LINEAR>(s, p, part_bytes);
  if (dtype == MUI_DTYPE_BF16) return epilogue == SK_GATEUP ? launch_stream_t<BF16, SK_GATEUP>(s, p, 0) : launch_stream_t<BF16, SK_LINEAR>(s, p, part_bytes);
  return MUI_ERR_UNSUPPORTED;
}

template <int WF>
static int launch_stream_codes(hipStream_t s, int dtype, int epilogue, const StreamParams& p) {
  if (dtype == MUI_DTYPE_F16) return epilogue == SK_GATEUP ? launch_stream_t<F16, SK_GATEUP, WF>(s, p, 0) : launch_stream_t<F16, SK_LINEAR, WF>(s, p, 0);
  if (dtype == MUI_DTYPE_BF16) return epilogue == SK_GATEUP ? launch_stream_t<BF16, SK_GATEUP, WF>(s, p, 0) : launch_stream_t<BF16, SK_LINEAR, WF>(s, p, 0);
  return MUI_ERR_UNSUPPORTED;
}

// The same for int8 codes, 17 to 64 tokens; groups of 64 or more. (K is never divided here: from 65 tokens on launch_prefill_parts does so.)
int launch_gemm_stream_int8(hipStream_t s, int dtype, int wf, int epilogue, const SkinnyParams& q) {
  if (!stream_serves_codes(q, wf)) return MUI_ERR_UNSUPPORTED;
  const StreamParams p = stream_params(q, nullptr, true, true);
  if (wf == WF_I8_CHANNEL) return launch_stream_codes<WF_I8_CHANNEL>(s, dtype, epilogue, p);
  return launch_stream_codes<WF_U8_GROUP>(s, dtype, epilogue, p);
}

// The same for a caller whose next launch adds the partial outputs up itself: part [*splits][tokens][n] gets the products, nothing else is applied.
// K is divided as by launch_gemm_stream; MUI_ERR_UNSUPPORTED also where it is left undivided.
int launch_gemm_stream_parts(hipStream_t s, int dtype, const SkinnyParams& q, float* part, size_t part_bytes, int* splits) {
  if (!part || !stream_serves(q, 128)) return MUI_ERR_UNSUPPORTED;
  const StreamParams p = stream_params(q, part, false);
  if (dtype == MUI_DTYPE_F16) return launch_stream_t<F16, SK_LINEAR>(s, p, part_bytes, splits);
  if (dtype == MUI_DTYPE_BF16) return launch_stream_t<BF16, SK_LINEAR>(s, p, part_bytes, splits);
  return MUI_ERR_UNSUPPORTED;
}

// The launch that adds up what launch_prefill_parts has left
int launch_parts_add(hipStream_t s, int dtype, const SkinnyParams& q, float* part, int shares) {
  StreamParams p = stream_params(q, part, true);
  p.k_splits = shares;
  if (dtype == MUI_DTYPE_F16) hipLaunchKernelGGL(gemm_stream_add_kernel<F16>, dim3(add_blocks(p.tokens, p.n)), dim3(256), 0, s, p);
  else if (dtype == MUI_DTYPE_BF16) hipLaunchKernelGGL(gemm_stream_add_kernel<BF16>, dim3(add_blocks(p.tokens, p.n)), dim3(256), 0, s, p);
  else return MUI_ERR_UNSUPPORTED;
  return launch_status();
}

}  // namespace mui

extern "C" int mui_tune_stream(int rows_per_unit, int shares) {
  MUI_TUNE_GUARD();
  if (rows_per_unit < 0 || rows_per_unit > 128 || shares < 0 || shares > 8) return MUI_ERR_INVALID_ARG;
  mui::g_stream_rows = rows_per_unit;
  mui::g_stream_shares = shares;
  return MUI_OK;
}
