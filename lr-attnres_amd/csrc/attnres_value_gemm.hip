// Value-derived LR keys with their projection on the matrix cores
// (LRIDSourceKeyProjection with its value norm, model.py:391-428):
//   keys[s] = rnd(rnd(inv v[s]) W^T),  inv = 1 / sqrt(<v, v> / D + eps)
//   dv[s]   = rnd(inv (gk W) - v inv^2 <gk, key> / D)
//   dW      = rnd(sum_{s, t} rnd(inv gk)^T v)
// The normed rows, which were written once and read three times around library
// GEMMs, exist only in registers.  In the backward the norm's 1/rms, a factor of a
// whole row, multiplies the fp32 product or the short gradient row (rounded
// where the long one was), and <gk W, v> = <gk, v W^T> = <gk, key> / inv, so that
// the rms-norm's backward needs no second pass over the row either.
//
// Bound by memory: the forward reads the rows from HBM once (and once more from
// the last-level cache, the norm first); the backward reads them once for dv (and
// writes it) and once for dW.  rank is 32, 64 or 128: about 128 flops per
// byte of a row, well below the matrix cores' rate at these bytes.
//
// Layout.  MFMA 32x32x16: A and B hold 8 values of k per lane (k = 8 (lane / 32) +
// j), row / column lane % 32; C holds for column lane % 32 the rows
// 8 (i / 4) + 4 (lane / 32) + i % 4.  k may be permuted as long as A and B agree.
//   forward  C = keys^T: A = W (from LDS, 64 columns of D at a time, double
//            buffered), B = 32 rows of v straight from memory, 64 bytes of a row
//            per lane and step, so a row's norm and its 1/rms stay in its lane.
//   dv       C = (gk W)^T: A = W^T (LDS, 64 columns of D at a time), its rows
//            permuted so that a lane's two tiles are 8 consecutive columns of one
//            row; B = 32 gradient rows, held throughout.
//   dW       C = dW: k runs over tokens, so both operands are rows transposed:
//            a lane reads 8 rows of a column pair (and of rank / 32 gradient
//            columns) from LDS and pairs their halves with v_perm.  A wave holds
//            all rank x 64 sums; workgroups split the tokens, and a second kernel
//            adds their partial sums in a fixed order.
//
// Measured with 17 sources of 16384 rows, D = 2048, rank 128, bf16 (one MI355X):
// forward 388 us (was 357 for the norm and 287 for the GEMM), dv 585 (350 for the
// GEMM and 591 for the norm's backward), dW 262 with its reduction 10 and the
// gradient rows' preparation 38 (703 and 50 for stacking them): 1.29 ms of kernels
// against 2.34.  dv is at 78% of a copy's rate; the forward at the last-level
// cache's for its second reading.
#include "attnres_device.h"
#include "attnres_launch.h"
#include "attnres_params.h"

namespace attnres {

typedef __bf16 vk_b8 __attribute__((ext_vector_type(8)));
typedef float vk_f16 __attribute__((ext_vector_type(16)));

using DT = BF16;  // the only type (an fp16 rnd(inv gk) could overflow)

__device__ __forceinline__ vk_f16 vk_mfma(const u32x4& a, const u32x4& b, const vk_f16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(vk_b8, a), __builtin_bit_cast(vk_b8, b), c, 0, 0, 0);
}

constexpr int kVkRows = 128;   // rows of a workgroup (32 a wave) in the forward and dv
constexpr int kVkCols = 64;    // columns of D per step

// A wave's tile of 32 rows x 64 columns.  Memory side: lane i holds in piece q the
// 16-byte chunk i % 8 of row 8 q + i / 8 (whole 128-byte lines per access; the
// operand layout straight from memory touched 32 lines for 16 or 32 bytes each:
// dv 789 us with cached accesses, 1528 with streaming ones).  Operand side: lane l
// reads any chunk of row l % 32.  Between them 4 KB of LDS of the wave's own, the
// chunks of row r swapped by r % 8 so that neither side meets bank conflicts.
struct VkTile {
  int64_t row[4];  // this lane's rows (clamped to the last one)
  int chunk;       // and its chunk
  char* lds;
  char* mem_side;
  int l32;
  __device__ __forceinline__ VkTile(char* stage, int lane, int64_t row0, int64_t n_tok) {
    chunk = lane & 7;
    lds = stage;
    mem_side = stage + (lane >> 3) * 128 + ((chunk ^ (lane >> 3)) * 16);
    l32 = lane & 31;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t r = row0 + 8 * q + (lane >> 3);
      row[q] = r < n_tok ? r : n_tok - 1;
    }
  }
  __device__ __forceinline__ void put(const u32x4 (&x)[4]) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) *(u32x4*)(mem_side + q * 1024) = x[q];
  }
  __device__ __forceinline__ void get(u32x4 (&x)[4]) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = *(const u32x4*)(mem_side + q * 1024);
  }
  __device__ __forceinline__ u32x4* chunk_of(int c) const { return (u32x4*)(lds + l32 * 128 + ((c ^ (l32 & 7)) * 16)); }
};

// ---------------------------------------------------------------- forward
template <int RT>  // rank = 32 RT
__global__ void __launch_bounds__(256) value_keys_fwd_kernel(const ValueKeysParams p) {
  using S = typename DT::S;
  constexpr int R = 32 * RT, PITCH = kVkCols * 2 + 16;  // bytes of an LDS row (padded against bank conflicts)
  __shared__ __align__(16) char s_w[2][R * PITCH];
  __shared__ __align__(16) char s_v[4][4096];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid / 64;
  const int l32 = lane & 31, h = lane >> 5;
  const int s = blockIdx.y, D = p.D;
  const int64_t row0 = (int64_t)blockIdx.x * kVkRows + wave * 32, row = row0 + l32;
  const VkTile tile(s_v[wave], lane, row0, p.n_tok);
  const S* vp[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) vp[q] = (const S*)p.val[s] + tile.row[q] * (int64_t)p.vstride[s] + tile.chunk * 8;
  const S* wp = (const S*)p.weight + (int64_t)(tid / 8) * D + (tid & 7) * 8;  // rows tid / 8 + 32 i of W
  const int wdst = (tid / 8) * PITCH + (tid & 7) * 16;

  vk_f16 acc[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  // the rows' norms first: the second reading finds them in the last-level cache
  // (128 rows a workgroup, at most 3 workgroups a CU)
  float inv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < D; k += kVkCols) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u32x4 x = *(const u32x4*)(vp[q] + k);
#pragma unroll
      for (int i = 0; i < 4; ++i) inv[q] = dot2<DT>(x[i], x[i], inv[q]);
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    inv[q] = 1.0f / sqrtf(group_sum(inv[q], 8) / (float)D + p.eps);
    const int64_t r = row0 + 8 * q + (lane >> 3);
    if (tile.chunk == 0 && r < p.n_tok && p.inv) p.inv[(int64_t)s * p.n_tok + r] = inv[q];
  }
  u32x4 vn[4], wn[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) wn[i] = *(const u32x4*)(wp + (int64_t)i * 32 * D);
#pragma unroll
  for (int q = 0; q < 4; ++q) vn[q] = __builtin_nontemporal_load((const u32x4*)vp[q]);
#pragma unroll
  for (int i = 0; i < RT; ++i) *(u32x4*)(s_w[0] + wdst + i * 32 * PITCH) = wn[i];
  const int steps = D / kVkCols;
  for (int k = 0; k < steps; ++k) {
    // rnd(v / rms), to the operand side
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        vn[q][i] = pack2<DT>(__uint_as_float(vn[q][i] << 16) * inv[q], __uint_as_float(vn[q][i] & 0xffff0000u) * inv[q]);
    tile.put(vn);
    const int nx = (k + 1 < steps ? k + 1 : k) * kVkCols;  // (the last step re-reads its own columns)
#pragma unroll
    for (int i = 0; i < RT; ++i) wn[i] = *(const u32x4*)(wp + (int64_t)i * 32 * D + nx);
#pragma unroll
    for (int q = 0; q < 4; ++q) vn[q] = __builtin_nontemporal_load((const u32x4*)(vp[q] + nx));
    __syncthreads();
    const char* w = s_w[k & 1] + l32 * PITCH + h * 64;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x4 x = *tile.chunk_of(4 * h + j);
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[t] = vk_mfma(*(const u32x4*)(w + t * 32 * PITCH + j * 16), x, acc[t]);
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) *(u32x4*)(s_w[(k + 1) & 1] + wdst + i * 32 * PITCH) = wn[i];
    wave_sync();  // the tile is read before the next step writes it
  }
  if (row >= p.n_tok) return;
  const int64_t at = (int64_t)s * p.n_tok + row;
  S* kp = (S*)p.keys + at * R + h * 4;
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      u32x2 o = {pack2<DT>(acc[t][4 * a], acc[t][4 * a + 1]),
                 pack2<DT>(acc[t][4 * a + 2], acc[t][4 * a + 3])};
      *(u32x2*)(kp + t * 32 + a * 8) = o;
    }
}

// ---------------------------------------------------------------- backward
// W^T, and per row: gs = rnd(inv gk), c = inv^2 <gk, key> / D
__global__ void __launch_bounds__(256) value_keys_transpose_kernel(const ValueKeysParams p) {
  using S = typename DT::S;
  __shared__ S t[32][33];
  const int x = threadIdx.x & 31, y = threadIdx.x / 32, d0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const S* w = (const S*)p.weight;
  S* o = (S*)p.wt;
#pragma unroll
  for (int i = 0; i < 32; i += 8) t[y + i][x] = w[(int64_t)(r0 + y + i) * p.D + d0 + x];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 32; i += 8) o[(int64_t)(d0 + y + i) * p.R + r0 + x] = t[x][y + i];
}

__global__ void __launch_bounds__(256) value_keys_prep_kernel(const ValueKeysParams p) {
  using S = typename DT::S;
  const int s = blockIdx.y, lanes = p.R / 8;  // 4, 8 or 16 lanes a row
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, n = p.n_tok * lanes;
  const int64_t ic = i < n ? i : n - 1, row = ic / lanes;
  const int64_t at = (int64_t)s * p.n_tok + row;
  const S* g = (const S*)p.gkey[s];
  float gk[8], k[8], m = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) gk[e] = 0.f;
  if (g) load_vec<DT, 8, true>(g + ic * 8, gk);
  load_vec<DT, 8, true>((const S*)p.keys + at * p.R + (ic - row * lanes) * 8, k);
  const float inv = p.inv[at];
#pragma unroll
  for (int e = 0; e < 8; ++e) m += gk[e] * k[e];
  m = group_sum(m, lanes);
  if (i >= n) return;
  if (ic - row * lanes == 0) p.c[at] = inv * inv * (m / (float)p.D);
#pragma unroll
  for (int e = 0; e < 8; ++e) gk[e] *= inv;
  store_vec<DT, 8>((S*)p.gs + at * p.R + (ic - row * lanes) * 8, gk);
}

template <int RT>
__global__ void __launch_bounds__(256) value_keys_dv_kernel(const ValueKeysParams p) {
  using S = typename DT::S;
  constexpr int R = 32 * RT, KK = 2 * RT, PITCH = R * 2 + 16, CH = RT;  // 16-byte chunks of a step per thread
  __shared__ __align__(16) char s_w[2][kVkCols * PITCH];
  __shared__ __align__(16) char s_v[4][4096];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid / 64;
  const int l32 = lane & 31, h = lane >> 5;
  const int s = blockIdx.y, D = p.D;
  const int64_t row0 = (int64_t)blockIdx.x * kVkRows + wave * 32, row = row0 + l32;
  const int64_t rowc = row < p.n_tok ? row : p.n_tok - 1, at = (int64_t)s * p.n_tok + rowc;
  const VkTile tile(s_v[wave], lane, row0, p.n_tok);
  const S* vp[4];
  S* dp[4];
  bool in[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    vp[q] = (const S*)p.val[s] + tile.row[q] * (int64_t)p.vstride[s] + tile.chunk * 8;
    dp[q] = (S*)p.dval[s] + tile.row[q] * (int64_t)D + tile.chunk * 8;
    in[q] = row0 + 8 * q + (lane >> 3) < p.n_tok;
  }
  const float inv = p.inv[at], c = p.c[at];
  u32x4 b[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    const u32x4 zero = {0u, 0u, 0u, 0u};
    b[kk] = p.gkey[s] ? *(const u32x4*)((const S*)p.gkey[s] + rowc * R + kk * 16 + h * 8) : zero;
  }
  // column of A's row m of tile T: 16 (m / 8) + 8 (m / 4 % 2) + 4 T + m % 4
  const int col = 16 * (l32 / 8) + 8 * ((l32 / 4) & 1) + (l32 & 3);
  constexpr int RC = R / 8;  // chunks of a W^T row
  const u32x4* wp = (const u32x4*)p.wt;
  u32x4 wn[CH], vn[4];
  auto wload = [&](int d0) {
#pragma unroll
    for (int i = 0; i < CH; ++i) wn[i] = wp[(int64_t)d0 * RC + tid + 256 * i];
  };
  auto wstore = [&](char* dst) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int x = tid + 256 * i;
      *(u32x4*)(dst + (x / RC) * PITCH + (x % RC) * 16) = wn[i];
    }
  };
  wload(0);
#pragma unroll
  for (int q = 0; q < 4; ++q) vn[q] = __builtin_nontemporal_load((const u32x4*)vp[q]);
  wstore(s_w[0]);
  const int steps = D / kVkCols;
  for (int k = 0; k < steps; ++k) {
    tile.put(vn);
    const int nx = (k + 1 < steps ? k + 1 : k) * kVkCols;
    wload(nx);
#pragma unroll
    for (int q = 0; q < 4; ++q) vn[q] = __builtin_nontemporal_load((const u32x4*)(vp[q] + nx));
    __syncthreads();
    vk_f16 acc[2];
#pragma unroll
    for (int T = 0; T < 2; ++T)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[T][i] = 0.f;
    const char* w = s_w[k & 1] + col * PITCH + h * 16;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int T = 0; T < 2; ++T)
        acc[T] = vk_mfma(*(const u32x4*)(w + T * 4 * PITCH + kk * 32), b[kk], acc[T]);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      u32x4* at_v = tile.chunk_of(2 * a + h);
      const u32x4 x = *at_v;
      Raw<DT, 8> r;
      float v[8], d[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) r.w[i] = x[i];
      unpack<DT, 8>(r, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) d[e] = inv * acc[e / 4][4 * a + (e & 3)] - v[e] * c;
      const u32x4 o = {pack2<DT>(d[0], d[1]), pack2<DT>(d[2], d[3]), pack2<DT>(d[4], d[5]), pack2<DT>(d[6], d[7])};
      *at_v = o;
    }
    wstore(s_w[(k + 1) & 1]);
    wave_sync();
    u32x4 o[4];
    tile.get(o);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (in[q]) __builtin_nontemporal_store(o[q], (u32x4*)(dp[q] + k * kVkCols));
    wave_sync();  // the tile is read before the next step writes it
  }
}

// partial dW of workgroup (column group x, token part y): tokens [t0, t1) of one source.
// Stages of 32 rows x 256 columns and their gradient rows go straight from memory to
// LDS (16 bytes a lane), two stages ahead of the one in use: 4.5 TB/s of rows, where
// loads of a lane's own column pair into registers (4 bytes of a row a lane, 16 a
// step, all that fit in flight) reached 2.9 (17 sources of 16384 rows, D = 2048, rank
// 128: 262 us against 390; one source, D = 1024, rank 64: 10.8 against 16.7; cached
// instead of streaming rows: 269).
constexpr int kDwTok = 32, kDwStages = 3;
constexpr int kDwRow = 512;  // bytes of a row in a stage
template <int RT>
constexpr int dw_stage_bytes() { return kDwTok * (kDwRow + 64 * RT); }

template <int RT>
__global__ void __launch_bounds__(256) value_keys_dw_kernel(const ValueKeysParams p) {
  using S = typename DT::S;
  constexpr int R = 32 * RT, GW = RT == 1 ? 1 : RT / 2;  // words of a lane's gradient columns (RT == 1: half of one)
  constexpr int GI = RT == 4 ? 2 : 1;                    // a wave's gradient pieces of 1 KB (RT == 1: waves 2, 3 as 0, 1)
  constexpr int kLoads = 4 + GI, kStage = dw_stage_bytes<RT>();
  __shared__ __align__(16) char s_dw[kDwStages * kStage];  // [stages][rows' 256 columns | their gradient rows]
  const int lane = threadIdx.x & 63, wave = uniform_i32(threadIdx.x / 64);
  const int l32 = lane & 31, h = lane >> 5;
  const int s = blockIdx.y / p.parts, part = blockIdx.y - s * p.parts, D = p.D;
  const int cb = (blockIdx.x * 4 + wave) * 64;
  const int64_t per = (p.n_tok + p.parts - 1) / p.parts;
  const int64_t t0 = part * per, t1 = t0 + per < p.n_tok ? t0 + per : p.n_tok;
  const int col = min((int)blockIdx.x * 256 + 8 * l32, D - 8);  // the last group may be short: any column in its place
  const char* vp = (const char*)((const S*)p.val[s] + col);
  const char* gp = (const char*)((const S*)p.gs + (int64_t)s * p.n_tok * R);
  const int64_t vst = (int64_t)p.vstride[s] * 2;

  vk_f16 acc[RT][2];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int T = 0; T < 2; ++T)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][T][i] = 0.f;
  // stage k: rows t = t0 + 32 k ... (past the part's end: its last row)
  const int64_t v_lane = (8 * wave + h) * vst;
  auto load = [&](int k, char* to) {
    const int64_t t = t0 + (int64_t)k * kDwTok;
    const bool whole = t + kDwTok <= t1;  // wave-uniform
    const char* vt = vp + t * vst + v_lane;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const char* src = vt + 2 * q * vst;
      if (!whole) {
        const int64_t r = t + 8 * wave + 2 * q + h;
        src = vp + (r < t1 ? r : t1 - 1) * vst;
      }
      stage16<true>(src, to + (8 * wave + 2 * q) * kDwRow);
    }
#pragma unroll
    for (int i = 0; i < GI; ++i) {
      const int piece = RT == 1 ? (wave & 1) : wave * GI + i, at = piece * 1024 + lane * 16;
      const char* src = gp + t * (2 * R) + at;
      if (!whole) {
        const int64_t r = t + at / (2 * R);
        src = gp + (r < t1 ? r : t1 - 1) * (2 * R) + at % (2 * R);
      }
      stage16(src, to + kDwTok * kDwRow + piece * 1024);
    }
  };
  const int v_at = 8 * h * kDwRow + wave * 128 + 4 * l32, g_at = kDwTok * kDwRow + 8 * h * (2 * R) + 2 * RT * l32;
  // 16 rows of a stage: row 8 h + j of this lane's columns
  auto step = [&](const char* from, int64_t t, int row0) {
    uint32_t v[8], g[8][GW];
    const char* vl = from + v_at;
    const char* gl = from + g_at;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = *(const uint32_t*)(vl + (row0 + j) * kDwRow);
      const char* gr = gl + (row0 + j) * (2 * R);
      if constexpr (RT == 4) {
        const u32x2 x = *(const u32x2*)gr;
        g[j][0] = x.x;
        g[j][GW - 1] = x.y;
      } else if constexpr (RT == 2) {
        g[j][0] = *(const uint32_t*)gr;
      } else {
        g[j][0] = *(const uint16_t*)gr;
      }
    }
    if (t + row0 + 16 > t1) {  // wave-uniform: rows past the part's end count as zero
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool ok = t + row0 + 8 * h + j < t1;
        v[j] = ok ? v[j] : 0u;
#pragma unroll
        for (int i = 0; i < GW; ++i) g[j][i] = ok ? g[j][i] : 0u;
      }
    }
    u32x4 a[RT], b[2];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      b[0][q] = lo_pair(v[2 * q], v[2 * q + 1]);
      b[1][q] = hi_pair(v[2 * q], v[2 * q + 1]);
#pragma unroll
      for (int r = 0; r < RT; ++r)
        a[r][q] = (r & 1) ? hi_pair(g[2 * q][r / 2], g[2 * q + 1][r / 2]) : lo_pair(g[2 * q][r / 2], g[2 * q + 1][r / 2]);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int T = 0; T < 2; ++T) acc[r][T] = vk_mfma(a[r], b[T], acc[r][T]);
  };
  const int n = t0 < t1 ? (int)((t1 - t0 + kDwTok - 1) / kDwTok) : 0;
  for (int k = 0; k < kDwStages - 1 && k < n; ++k) load(k, s_dw + k * kStage);
  int buf = 0;
  for (int k = 0; k < n; ++k) {
    // this wave's part of stage k has arrived (the next stage's loads may still run) ...
    if (k + 1 < n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kLoads * (kDwStages - 2)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // ... every wave's has, and none reads stage k - 1 any more
    asm volatile("" ::: "memory");
    const int ahead = buf == 0 ? kDwStages - 1 : buf - 1;
    if (k + kDwStages - 1 < n) load(k + kDwStages - 1, s_dw + ahead * kStage);
    const int64_t t = t0 + (int64_t)k * kDwTok;
    step(s_dw + buf * kStage, t, 0);
    step(s_dw + buf * kStage, t, 16);
    buf = buf + 1 == kDwStages ? 0 : buf + 1;
  }
  if (cb >= D) return;
  float* out = p.partials + (int64_t)blockIdx.y * R * D + cb + 2 * l32;
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = 8 * (i / 4) + 4 * h + (i & 3);
      *(float2*)(out + (int64_t)(RT * m + r) * D) = make_float2(acc[r][0][i], acc[r][1][i]);
    }
}

// dW = rnd(sum of the parts, in order): four columns a thread
__global__ void __launch_bounds__(256) value_keys_dw_reduce_kernel(const ValueKeysParams p, int n_parts) {
  using S = typename DT::S;
  const int64_t n = (int64_t)p.R * p.D, i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int k = 0; k < n_parts; ++k) {
    const float4 x = *(const float4*)(p.partials + (int64_t)k * n + i);
    a[0] += x.x;
    a[1] += x.y;
    a[2] += x.z;
    a[3] += x.w;
  }
  store_vec<DT, 4>((S*)p.dweight + i, a);
}

template <int RT>
static hipError_t value_keys_rt(const ValueKeysParams& p, bool bwd, hipStream_t st) {
  const dim3 rows((unsigned)((p.n_tok + kVkRows - 1) / kVkRows), p.n_src);
  if (!bwd) {
    hipLaunchKernelGGL((value_keys_fwd_kernel<RT>), rows, dim3(256), 0, st, p);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(value_keys_prep_kernel, dim3((unsigned)((p.n_tok * (p.R / 8) + 255) / 256), p.n_src), dim3(256), 0, st, p);
  if (p.want_dv) {
    hipLaunchKernelGGL(value_keys_transpose_kernel, dim3(p.D / 32, p.R / 32), dim3(256), 0, st, p);
    hipLaunchKernelGGL((value_keys_dv_kernel<RT>), rows, dim3(256), 0, st, p);
  }
  if (p.dweight) {
    hipLaunchKernelGGL((value_keys_dw_kernel<RT>), dim3((p.D + 255) / 256, p.n_src * p.parts), dim3(256), 0, st, p);
    hipLaunchKernelGGL(value_keys_dw_reduce_kernel, dim3((unsigned)(((int64_t)p.R * p.D / 4 + 255) / 256)), dim3(256), 0, st,
                       p, p.n_src * p.parts);
  }
  return hipGetLastError();
}

hipError_t launch_value_keys(bool bwd, const ValueKeysParams& p, hipStream_t st) {
  switch (p.R) {
    case 32: return value_keys_rt<1>(p, bwd, st);
    case 64: return value_keys_rt<2>(p, bwd, st);
    case 128: return value_keys_rt<4>(p, bwd, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace attnres
