// Phase 1 from a query bank in one pass each way (attention_residual_phase1,
// attnres_ops.py:3862-3907; eager form _attnres_phase1_read_torch :2620-2627):
//   key[s]       = rnd(rms_norm(v[s]))          (or v[s] without key_norm)
//   logit[q, s]  = rnd(<bank[q], key[s]>)
//   w = softmax_s(logit), lse[q] = logsumexp,   out[q] = rnd(sum_s rnd(w[q, s]) v[s])
// and the backward of the composition, rounded where its parts are rounded:
//   dW[q, s] = rnd(<g[q], v[s]>),  dl = rnd(rnd(w (dW - <w, dW>)) + rnd(w glse))
//   dkey[s]  = rnd(sum_q dl[q, s] bank[q])
//   dv[s]    = rnd(rnd(sum_q rnd(w) g[q]) + rnd(inv (dkey - v inv mr))),  mr = <dkey, v> inv / D
//   dbank[q] = rnd(sum_{s, t} dl[q, s] key[s])
//
// Bound by HBM: forward S rows in and Q out per token, backward S + Q in and S
// out.  Scoring the bank in kernels of its own (attnres_keyed_logits.hip, one
// element per lane, the bank re-read for every row) and composing them with
// phase 1 read the values four times, wrote their gradients twice and added
// them in a pass per source.
//
// Layout: one workgroup per token at a time, a wave per 256 columns (four
// elements per lane), so that S value rows, Q upstream rows, the bank (loop
// invariant, in registers) and the backward's bank-gradient sums (Q x 4 per
// lane, written once per workgroup) fit: the backward at 2 sources and sites /
// 6 and 4 / 12 and 12 takes 62 / 111 / 228 registers in bf16, 60 / 119 / 256 in
// fp16 and 74 / 149 / 256 in fp32, where 12 and 12 spills 109 words (8 and 12
// under 20), still four times faster than the two kernel families (d768, 4096
// tokens, forward and backward: 440 us against 2363).  Row sums are folded per wave
// (wave_sums) and added over the waves through LDS in a fixed order: two
// barriers per token, the buffers alternating between tokens.  The (site,
// source) pairs -- lane = q * np + s, np a power of two, 64 pairs at a time --
// are worked out by every wave for itself, so nothing else is exchanged.
// 16-bit contractions are v_dot2 on packed words (source or site pairs).
// Workgroups walk tokens in XCD-major order: logits and lse are token-minor.
//
// Measured with 6 sources, 4 sites, D = 768, 16384 tokens, bf16 (one MI355X):
// forward 64 us (250 MB, 3.9 TB/s), backward 118 us (400 MB, 3.4 TB/s) and the
// bank's reduction 5 us, against 1033 + 40 and 1625 + 368 + 75 us of the two
// kernel families and 110 us of gradient adds before.  What is left is
// instructions: about 760 vector and 280 scalar ones per token and wave in the
// backward, against 910 slots in the token's bytes at the copy rate; loading a
// token ahead changed nothing.
#include "attnres_device.h"
#include "attnres_launch.h"
#include "attnres_params.h"

namespace attnres {

constexpr int kBankWaves = 8;  // at most: D <= 2048

template <class DT>
constexpr bool kIs16 = sizeof(typename DT::S) == 2;

// a . b over a lane's four elements
template <class DT>
__device__ __forceinline__ float dot4(const Raw<DT, 4>& a, const Raw<DT, 4>& b, float c) {
  if constexpr (kIs16<DT>) {
    c = dot2<DT>(a.w[0], b.w[0], c);
    return dot2<DT>(a.w[1], b.w[1], c);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) c += __uint_as_float(a.w[i]) * __uint_as_float(b.w[i]);
    return c;
  }
}

// words of rows 2k, 2k + 1 interleaved in place: element e of both rows in one word
template <class DT, int NR>
__device__ __forceinline__ void pair_rows(Raw<DT, 4> (&r)[NR]) {
  if constexpr (kIs16<DT>) {
#pragma unroll
    for (int k = 0; k < NR / 2; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t a = r[2 * k].w[i], b = r[2 * k + 1].w[i];
        r[2 * k].w[i] = lo_pair(a, b);
        r[2 * k + 1].w[i] = hi_pair(a, b);
      }
  }
}

// sum_i c[i] * row[i] over NR rows paired by pair_rows, coefficients in LDS:
// 16-bit types packed by pairs (coef points at NR / 2 words), fp32 plain
// (slots without a row hold zeros, so they need no guard: 0 * 0)
template <class DT, int NR>
__device__ __forceinline__ void combine_rows(const Raw<DT, 4> (&r)[NR], const uint32_t* coef, float (&acc)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = 0.f;
  if constexpr (kIs16<DT>) {
#pragma unroll
    for (int k = 0; k < NR / 2; ++k) {
      const uint32_t c = coef[k];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        acc[2 * i] = dot2<DT>(r[2 * k].w[i], c, acc[2 * i]);
        acc[2 * i + 1] = dot2<DT>(r[2 * k + 1].w[i], c, acc[2 * i + 1]);
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const float c = __uint_as_float(coef[k]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += c * __uint_as_float(r[k].w[i]);
    }
  }
}

// coefficient i of a table that combine_rows reads
template <class DT>
__device__ __forceinline__ void put_coef(uint32_t* tab, int i, float x) {
  if constexpr (kIs16<DT>) ((uint16_t*)tab)[i] = (uint16_t)bits16<DT>(x);
  else tab[i] = __float_as_uint(x);
}

// wave sums of x[0..V), V a multiple of 4, left in dst[0..V)
template <int V>
__device__ __forceinline__ void sums_to_lds(const float (&x)[V], float* dst, int lane) {
  float z[V / 4];
  wave_sums<V>(x, z);
  if ((lane & 15) == 0) {
    const int r = lane >> 4, j = r == 1 ? 2 : r == 2 ? 1 : r;
#pragma unroll
    for (int k = 0; k < V / 4; ++k) dst[4 * k + j] = z[k];
  }
}

// Slot counts are instantiated for the counts just below them, so only the
// last slots can be without a row (host: phase1_bank_plan).
__host__ __device__ constexpr int bank_slot_floor(int slots) { return slots <= 8 ? slots - 1 : 9; }

// rows (or lanes past the row's end) that count as zero
template <class DT, int NR>
__device__ __forceinline__ void zero_rows(Raw<DT, 4> (&r)[NR], int n, bool in) {
#pragma unroll
  for (int s = 0; s < NR; ++s) {
    const bool keep = in && (s < bank_slot_floor(NR) || s < n);
#pragma unroll
    for (int i = 0; i < Vec<DT, 4>::kWords; ++i) r[s].w[i] = keep ? r[s].w[i] : 0u;
  }
}

template <class DT, int NR>
__device__ __forceinline__ void load_rows(const Phase1BankParams& p, int64_t tok, int col, Raw<DT, 4> (&vr)[NR]) {
  using S = typename DT::S;
#pragma unroll
  for (int s = 0; s < NR; ++s) {
    const int j = s < bank_slot_floor(NR) ? s : min(s, p.n_src - 1);
    load_raw<DT, 4, true>((const S*)p.val[j] + tok * (int64_t)p.vstride[j] + col, vr[s]);
  }
}

template <class DT, int NR>
__device__ __forceinline__ void load_bank(const Phase1BankParams& p, int col, bool in, Raw<DT, 4> (&bank)[NR]) {
  using S = typename DT::S;
#pragma unroll
  for (int q = 0; q < NR; ++q) load_raw<DT, 4>((const S*)p.queries + (int64_t)min(q, p.n_q - 1) * p.D + col, bank[q]);
  zero_rows<DT, NR>(bank, p.n_q, in);
}

// sum over the workgroup's waves of part[wave * stride], in wave order, four reads at a time
__device__ __forceinline__ float waves_sum(const float* part, int stride, int nw) {
  float t = 0.f;
#pragma unroll 1
  for (int w = 0; w < nw; w += 4) {
    float x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = part[min(w + u, nw - 1) * stride];
#pragma unroll
    for (int u = 0; u < 4; ++u) t += w + u < nw ? x[u] : 0.f;
  }
  return t;
}

// packed rnd(x[0..4))
template <class DT>
__device__ __forceinline__ Raw<DT, 4> pack4(const float (&x)[4]) {
  Raw<DT, 4> r;
  if constexpr (kIs16<DT>) {
    r.w[0] = pack2<DT>(x[0], x[1]);
    r.w[1] = pack2<DT>(x[2], x[3]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) r.w[i] = __float_as_uint(x[i]);
  }
  return r;
}

// rnd(a) + rnd(b), not rounded (16-bit types: one pack and one v_dot2 with (1, 1))
template <class DT>
__device__ __forceinline__ float add_rounded(float a, float b) {
  if constexpr (kIs16<DT>) return dot2<DT>(pack2<DT>(a, b), DT::kCode == 1 ? 0x3f803f80u : 0x3c003c00u, 0.f);
  else return a + b;
}

template <class DT, int QB, int SB>
__global__ void __launch_bounds__(512) phase1_bank_fwd_kernel(const Phase1BankParams p) {
  using S = typename DT::S;
  constexpr int V = QB * SB, VG = V % 16 == 0 ? 16 : V % 12 == 0 ? 12 : V % 8 == 0 ? 8 : 4;
  constexpr int SV = (SB + 3) / 4 * 4;
  __shared__ float s_ss[2][kBankWaves][SV];
  __shared__ float s_dot[2][kBankWaves][V];
  __shared__ __align__(4) uint32_t s_w[kBankWaves][kIs16<DT> ? V / 2 : V];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = uniform_i32(threadIdx.x / kWave), nw = blockDim.x / kWave;
  const int N = p.n_src, Q = p.n_q, D = p.D, np = p.np;
  const bool in = wave * 256 + lane * 4 < D;
  const int col = in ? wave * 256 + lane * 4 : 0;
  Raw<DT, 4> bank[QB];
  load_bank<DT, QB>(p, col, in, bank);
  // weights of source slots past N stay zero
  for (int i = lane; i < (int)(sizeof(s_w[0]) / 4); i += kWave) s_w[wave][i] = 0u;
  wave_sync();

  int par = 0;
  for (int64_t tok = xcd_block(blockIdx.x, gridDim.x); tok < p.n_tok; tok += gridDim.x, par ^= 1) {
    Raw<DT, 4> vr[SB];
    load_rows<DT, SB>(p, tok, col, vr);
    zero_rows<DT, SB>(vr, N, in);
    float inv_l = 1.f;
    if (p.key_norm) {
      float ss[SV];
#pragma unroll
      for (int s = 0; s < SV; ++s) ss[s] = s < SB ? dot4<DT>(vr[s < SB ? s : 0], vr[s < SB ? s : 0], 0.f) : 0.f;
      sums_to_lds<SV>(ss, s_ss[par][wave], lane);
      __syncthreads();
      inv_l = 1.0f / sqrtf(waves_sum(&s_ss[par][0][min(lane, SB - 1)], SV, nw) / (float)D + p.eps);
      if (p.inv && wave == 0 && lane < N) p.inv[(int64_t)lane * p.n_tok + tok] = inv_l;
    }
    Raw<DT, 4> kr[SB];
#pragma unroll
    for (int s = 0; s < SB; ++s) {
      kr[s] = vr[s];
      if (p.key_norm) {
        const float inv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv_l), s));
        float x[4];
        unpack<DT, 4>(vr[s], x);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] *= inv;
        kr[s] = pack4<DT>(x);
      }
    }
#pragma unroll
    for (int b = 0; b < V; b += VG) {
      if (b / SB < bank_slot_floor(QB) || b / SB < Q) {
        float x[VG];
#pragma unroll
        for (int m = 0; m < VG; ++m) x[m] = dot4<DT>(bank[(b + m) / SB], kr[(b + m) % SB], 0.f);
        sums_to_lds<VG>(x, &s_dot[par][wave][b], lane);
      }
    }
    __syncthreads();
    // ---- softmax rows: pairs (q, s), 64 lanes at a time
    for (int b = 0; b < Q * np; b += kWave) {
      const int q = (b + lane) / np, s = (b + lane) & (np - 1);
      const bool own = q < Q && s < N;
      const int at = own ? q * SB + s : 0;
      const float l = own ? DT::rnd(waves_sum(&s_dot[par][0][at], V, nw)) : -INFINITY;
      const float lm = group_max(l, np);
      const float ex = own ? expf(l - lm) : 0.f;
      const float z = group_sum(ex, np);
      if (own) {
        put_coef<DT>(s_w[wave], at, DT::rnd(ex / z));
        if (wave == 0) {
          if (p.logits) DT::store1((S*)p.logits + ((int64_t)q * N + s) * p.n_tok + tok, l);
          if (s == 0) p.lse[(int64_t)q * p.n_tok + tok] = lm + logf(z);
        }
      }
    }
    wave_sync();
    // ---- mix
    pair_rows<DT, SB>(vr);
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      if (q < bank_slot_floor(QB) || q < Q) {
        float acc[4];
        combine_rows<DT, SB>(vr, &s_w[wave][kIs16<DT> ? q * SB / 2 : q * SB], acc);
        if (in) store_vec<DT, 4, true>((S*)p.out + ((int64_t)q * p.n_tok + tok) * D + col, acc);
      }
    }
    wave_sync();  // the weights are read before the next token writes them
  }
}

template <class DT, int QB, int SB>
__global__ void __launch_bounds__(512) phase1_bank_bwd_kernel(const Phase1BankParams p) {
  using S = typename DT::S;
  constexpr int V = QB * SB, VG = V % 16 == 0 ? 16 : V % 12 == 0 ? 12 : V % 8 == 0 ? 8 : 4;
  constexpr int SV = (SB + 3) / 4 * 4;
  constexpr int TW = kIs16<DT> ? V / 2 : V;  // words of a coefficient table
  __shared__ float s_m[2][kBankWaves][SV];
  __shared__ float s_dot[2][kBankWaves][V];
  // per wave: weights and logit gradients by [s][q], logit gradients by [q][s]
  __shared__ __align__(4) uint32_t s_wq[kBankWaves][TW], s_lq[kBankWaves][TW], s_ls[kBankWaves][TW];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = uniform_i32(threadIdx.x / kWave), nw = blockDim.x / kWave;
  const int N = p.n_src, Q = p.n_q, D = p.D, np = p.np;
  const bool in = wave * 256 + lane * 4 < D;
  const int col = in ? wave * 256 + lane * 4 : 0;
  Raw<DT, 4> bank[QB];
  load_bank<DT, QB>(p, col, in, bank);
  pair_rows<DT, QB>(bank);
  float qacc[QB][4];
#pragma unroll
  for (int q = 0; q < QB; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) qacc[q][i] = 0.f;
  for (int i = lane; i < TW; i += kWave) s_wq[wave][i] = s_lq[wave][i] = s_ls[wave][i] = 0u;
  wave_sync();

  int par = 0;
  for (int64_t tok = xcd_block(blockIdx.x, gridDim.x); tok < p.n_tok; tok += gridDim.x, par ^= 1) {
    Raw<DT, 4> gr[QB], vr[SB];
#pragma unroll
    for (int q = 0; q < QB; ++q)
      load_raw<DT, 4, true>((const S*)p.gout + ((int64_t)min(q, Q - 1) * p.n_tok + tok) * D + col, gr[q]);
    load_rows<DT, SB>(p, tok, col, vr);
    zero_rows<DT, QB>(gr, Q, in);
    zero_rows<DT, SB>(vr, N, true);  // (past the row's end the upstream rows and the bank are zero)
    const float inv_l = p.key_norm ? p.inv[(int64_t)min(lane, N - 1) * p.n_tok + tok] : 1.f;
    // ---- dW[q, s] = <g[q], v[s]>
#pragma unroll
    for (int b = 0; b < V; b += VG) {
      if (b / SB < bank_slot_floor(QB) || b / SB < Q) {
        float x[VG];
#pragma unroll
        for (int m = 0; m < VG; ++m) x[m] = dot4<DT>(gr[(b + m) / SB], vr[(b + m) % SB], 0.f);
        sums_to_lds<VG>(x, &s_dot[par][wave][b], lane);
      }
    }
    __syncthreads();
    for (int b = 0; b < Q * np; b += kWave) {
      const int q = (b + lane) / np, s = (b + lane) & (np - 1);
      const bool own = q < Q && s < N;
      const float l = own ? DT::load1((const S*)p.logits + ((int64_t)q * N + s) * p.n_tok + tok) : -INFINITY;
      const float gl = own && p.glse ? p.glse[(int64_t)q * p.n_tok + tok] : 0.f;
      const float dw = own ? DT::rnd(waves_sum(&s_dot[par][0][q * SB + s], V, nw)) : 0.f;
      const float lm = group_max(l, np);  // (in every lane: not inside the selects)
      const float ex = own ? expf(l - lm) : 0.f;
      const float w = ex / group_sum(ex, np);
      const float inner = group_sum(own ? w * dw : 0.f, np);
      const float dl = DT::rnd(DT::rnd(w * (dw - inner)) + DT::rnd(gl * w));
      if (own) {
        put_coef<DT>(s_wq[wave], s * QB + q, DT::rnd(w));
        put_coef<DT>(s_lq[wave], s * QB + q, dl);
        put_coef<DT>(s_ls[wave], q * SB + s, dl);
      }
    }
    wave_sync();
    // ---- dkey, and mr of every source
    Raw<DT, 4> dk[SB];
#pragma unroll
    for (int s = 0; s < SB; ++s) {
      float a[4];
      combine_rows<DT, QB>(bank, &s_lq[wave][kIs16<DT> ? s * QB / 2 : s * QB], a);
      dk[s] = pack4<DT>(a);
    }
    float mr_l = 0.f;
    if (p.key_norm) {
      float m[SV];
#pragma unroll
      for (int s = 0; s < SV; ++s) m[s] = s < SB ? dot4<DT>(dk[s < SB ? s : 0], vr[s < SB ? s : 0], 0.f) : 0.f;
      sums_to_lds<SV>(m, s_m[par][wave], lane);
      __syncthreads();
      mr_l = waves_sum(&s_m[par][0][min(lane, SB - 1)], SV, nw) * inv_l / (float)D;
    }
    // ---- dv; the value rows become the keys
    pair_rows<DT, QB>(gr);
#pragma unroll
    for (int s = 0; s < SB; ++s) {
      if (s < bank_slot_floor(SB) || s < N) {
        const float inv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv_l), s));
        const float mr = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mr_l), s));
        float mix[4], k[4], v[4];
        combine_rows<DT, QB>(gr, &s_wq[wave][kIs16<DT> ? s * QB / 2 : s * QB], mix);
        unpack<DT, 4>(dk[s], k);
        unpack<DT, 4>(vr[s], v);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (p.key_norm) {
            v[i] *= inv;
            k[i] = inv * (k[i] - v[i] * mr);
          }
          mix[i] = add_rounded<DT>(mix[i], k[i]);  // rounded by the store
        }
        if (in) store_vec<DT, 4, true>((S*)p.dval[s] + tok * (int64_t)D + col, mix);
        if (p.key_norm) vr[s] = pack4<DT>(v);
      }
    }
    // ---- dbank += sum_s dl[q, s] key[s]
    pair_rows<DT, SB>(vr);
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      float a[4];
      combine_rows<DT, SB>(vr, &s_ls[wave][kIs16<DT> ? q * SB / 2 : q * SB], a);
#pragma unroll
      for (int i = 0; i < 4; ++i) qacc[q][i] += a[i];
    }
    wave_sync();  // the tables are read before the next token writes them
  }
  if (!p.partials || !in) return;
#pragma unroll
  for (int q = 0; q < QB; ++q)
    if (q < Q)  // four consecutive slots of one 16-slot tile
      *(float4*)&p.partials[part_index(kPartTiled, blockIdx.x, q * D + col, gridDim.x, 0)] =
          make_float4(qacc[q][0], qacc[q][1], qacc[q][2], qacc[q][3]);
}

// L.wpt = waves per token, L.nmax = source slots, L.teams = site slots
template <class DT, bool BWD>
static hipError_t phase1_bank_dt(const Phase1BankParams& p, const Launch& L, hipStream_t st) {
  const dim3 g(L.grid), b(L.wpt * kWave);
#define ATTNRES_P1B(QB, SB)                                                                              \
  case QB * 100 + SB:                                                                                    \
    if constexpr (BWD) hipLaunchKernelGGL((phase1_bank_bwd_kernel<DT, QB, SB>), g, b, 0, st, p);         \
    else hipLaunchKernelGGL((phase1_bank_fwd_kernel<DT, QB, SB>), g, b, 0, st, p);                       \
    break;
#define ATTNRES_P1B_S(QB) \
  ATTNRES_P1B(QB, 2) ATTNRES_P1B(QB, 4) ATTNRES_P1B(QB, 6) ATTNRES_P1B(QB, 8) ATTNRES_P1B(QB, 12)
  switch (L.teams * 100 + L.nmax) {
    ATTNRES_P1B_S(2)
    ATTNRES_P1B_S(4)
    ATTNRES_P1B_S(6)
    ATTNRES_P1B_S(8)
    ATTNRES_P1B_S(12)
    default: return hipErrorInvalidValue;
  }
#undef ATTNRES_P1B_S
#undef ATTNRES_P1B
  return hipGetLastError();
}

hipError_t launch_phase1_bank_forward(int dtype, const Phase1BankParams& p, const Launch& L, hipStream_t st) {
  switch (dtype) {
    case ATTNRES_DTYPE_F32: return phase1_bank_dt<F32, false>(p, L, st);
    case ATTNRES_DTYPE_BF16: return phase1_bank_dt<BF16, false>(p, L, st);
    default: return phase1_bank_dt<F16, false>(p, L, st);
  }
}
hipError_t launch_phase1_bank_backward(int dtype, const Phase1BankParams& p, const Launch& L, hipStream_t st) {
  switch (dtype) {
    case ATTNRES_DTYPE_F32: return phase1_bank_dt<F32, true>(p, L, st);
    case ATTNRES_DTYPE_BF16: return phase1_bank_dt<BF16, true>(p, L, st);
    default: return phase1_bank_dt<F16, true>(p, L, st);
  }
}

}  // namespace attnres
