// Base AttnRes read with a token's row split over the waves of one workgroup:
// more than 16 sources (a read site deep in a model whose every sublayer output
// is a source), the output norm, and the row widths and types that
// attnres_base_fast.h does not cover.  Semantics and rounding points are those
// of attnres_base.hip.
//
// Bound by HBM.  A key is the rms norm of the whole row and the mix needs every
// logit first, so each row is used twice (three times in the backward); with
// more than 16 rows a wave cannot hold a token, and the streaming kernels read
// them again from memory for every use.  Split by columns, a wave holds 64
// lane vectors of all N rows (2 or 4 VGPRs a source) and the rows are read
// once: row sums are folded per wave (wave_sums), added over the waves through
// LDS, and lane s of every wave carries source s's scalars.  Two barriers per
// token (forward: the norms, the logits; backward: dW with the norms, the key
// gradients' means), one more with the output norm, buffers alternating between
// tokens.
//
// Measured (one MI355X, bf16, d1024): 25 sources, 8192 tokens, forward 80 us
// (427 MB, 5.3 TB/s), backward 203 us (862 MB, 4.2 TB/s); with the rows
// streamed twice 174 and 414.  9 sources, output norm, 8192 tokens, forward
// 35 us (168 MB) against 67 of the resident step-by-step kernel.  The backward
// is near its instructions: about 2700 vector ones per token and wave at 26
// slots against 3000 in the time of its bytes at the copy rate (3300 before
// sources were taken in pairs: 254 us).
#pragma once

#include "attnres_device.h"
#include "attnres_launch.h"
#include "attnres_lr_fast.h"
#include "attnres_lr_split.h"
#include "attnres_params.h"

namespace attnres {

// sums over the wave of val(i), i < NB, in groups of at most 16: dst[i]
template <int NB, class F>
__device__ __forceinline__ void base_split_sums(float* dst, int lane, F val) {
  constexpr int G = NB % 16 == 0 ? 16 : NB % 12 == 0 ? 12 : NB % 8 == 0 ? 8 : 4;
  constexpr int NP = (NB + G - 1) / G * G;
#pragma unroll
  for (int b = 0; b < NP; b += G) {
    float x[G], z[G / 4];
#pragma unroll
    for (int i = 0; i < G; ++i) x[i] = b + i < NB ? val(b + i < NB ? b + i : 0) : 0.f;
    wave_sums<G>(x, z);
    if ((lane & 15) == 0) {
      const int r = lane >> 4, j = r == 1 ? 2 : r == 2 ? 1 : r;
#pragma unroll
      for (int k = 0; k < G / 4; ++k) dst[b + 4 * k + j] = z[k];
    }
  }
}
__host__ __device__ constexpr int base_split_row(int nb) { return (nb + 15) / 16 * 16; }  // floats of one wave's sums

// sum over the workgroup's waves, four reads at a time
__device__ __forceinline__ float base_split_total(const float* part, int stride, int nw) {
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

__device__ __forceinline__ float lane_value(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// <a, b> of a lane's vectors
template <class DT, int E>
__device__ __forceinline__ float vec_dot(const Raw<DT, E>& a, const Raw<DT, E>& b) {
  float d = 0.f;
  if constexpr (sizeof(typename DT::S) == 2) {
#pragma unroll
    for (int i = 0; i < E / 2; ++i) d = dot2<DT>(a.w[i], b.w[i], d);
  } else {
#pragma unroll
    for (int i = 0; i < E; ++i) d += __uint_as_float(a.w[i]) * __uint_as_float(b.w[i]);
  }
  return d;
}

// <rnd(a * c), b>
template <class DT, int E>
__device__ __forceinline__ float scaled_dot(const Raw<DT, E>& a, float c, const Raw<DT, E>& b) {
  float x[E], d = 0.f;
  unpack<DT, E>(a, x);
  if constexpr (sizeof(typename DT::S) == 2) {
#pragma unroll
    for (int i = 0; i < E / 2; ++i) d = dot2<DT>(pack2<DT>(x[2 * i] * c, x[2 * i + 1] * c), b.w[i], d);
  } else {
#pragma unroll
    for (int i = 0; i < E; ++i) d += x[i] * c * __uint_as_float(b.w[i]);
  }
  return d;
}

template <class DT, int E, int NB>
__device__ __forceinline__ void base_split_load(const SrcTab* tab, int N, int64_t tok, int eoff, bool ok, bool part,
                                                Raw<DT, E> (&vr)[NB]) {
  lr_split_load<DT, E, NB>(tab, N, tok, eoff, vr);
  if (part)  // the row ends inside this wave (wave-uniform)
#pragma unroll
    for (int s = 0; s < NB; ++s)
#pragma unroll
      for (int i = 0; i < Vec<DT, E>::kWords; ++i) vr[s].w[i] = ok ? vr[s].w[i] : 0u;
}

template <class DT, int VB, int NB>
__global__ void __launch_bounds__(512) base_split_fwd_kernel(const ReadParams p) {
  using S = typename DT::S;
  constexpr int E = VB / (int)sizeof(S), F = lr_split_floor(NB), ROW = base_split_row(NB);
  constexpr int NP = NB <= 4 ? 4 : NB <= 8 ? 8 : NB <= 16 ? 16 : NB <= 32 ? 32 : 64;
  __shared__ SrcTab s_tab;
  __shared__ float s_ss[2][8][ROW], s_lg[2][8][ROW], s_red[2][8];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = uniform_i32(threadIdx.x / kWave), nw = blockDim.x / kWave;
  const int N = p.n_src, D = p.D;
  for (int i = threadIdx.x; i < N; i += blockDim.x) {
    s_tab.vptr[i] = (uint64_t)p.val[i];
    s_tab.vstrb[i] = (uint32_t)p.vstride[i] * (uint32_t)sizeof(S);
  }
  __syncthreads();
  const bool ok = (wave * kWave + lane) * E < D, part = (wave + 1) * kWave * E > D;
  const int eoff = ok ? (wave * kWave + lane) * E : 0;
  Raw<DT, E> qr;
  load_raw<DT, E>((const S*)p.q_static + eoff, qr);
  const float bias = p.bias && lane < N ? p.bias[lane] : 0.f;
  const int at = min(lane, NB - 1);

  int par = 0;
  for (int64_t tok = blockIdx.x; tok < p.n_tok; tok += gridDim.x, par ^= 1) {
    Raw<DT, E> vr[NB];
    base_split_load<DT, E, NB>(&s_tab, N, tok, eoff, ok, part, vr);
    float inv_l = 1.f;
    if (p.key_norm) {
      base_split_sums<NB>(s_ss[par][wave], lane, [&](int s) { return vec_dot<DT, E>(vr[s], vr[s]); });
      __syncthreads();
      inv_l = 1.0f / sqrtf(base_split_total(&s_ss[par][0][at], ROW, nw) / (float)D + p.eps);
    }
    base_split_sums<NB>(s_lg[par][wave], lane, [&](int s) {
      return p.key_norm ? scaled_dot<DT, E>(vr[s], lane_value(inv_l, s), qr) : vec_dot<DT, E>(vr[s], qr);
    });
    __syncthreads();
    // ---- softmax, lane s for source s
    const float lg = lane < N ? DT::rnd(base_split_total(&s_lg[par][0][at], ROW, nw)) + bias : -INFINITY;
    const float mx = group_max(lg, NP);
    const float ex = lane < N ? expf(lg - mx) : 0.f;
    const float pw = ex / group_sum(ex, NP);
    if (wave == 0 && lane < N && p.weights) p.weights[tok * N + lane] = pw;
    // ---- mix (an odd last source is paired with zeros)
    float acc[E];
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] = 0.f;
    if constexpr (sizeof(S) == 2) {
      const uint32_t wb = lane < N ? bits16<DT>(DT::rnd(pw)) : 0u;
      const uint32_t wn = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)wb, kDppXor1, 0xF, 0xF, true);
      const uint32_t w2 = wb | (wn << 16);  // even lanes: sources lane, lane + 1
#pragma unroll
      for (int s = 0; s < NB; s += 2) {
        if (s < F || s < N) {
          const uint32_t wp = (uint32_t)__builtin_amdgcn_readlane((int)w2, s);
          const bool two = s + 1 < F || s + 1 < N;
#pragma unroll
          for (int i = 0; i < E / 2; ++i) {
            const uint32_t a = vr[s].w[i], c = two ? vr[s + 1].w[i] : 0u;
            acc[2 * i] = dot2<DT>(lo_pair(a, c), wp, acc[2 * i]);
            acc[2 * i + 1] = dot2<DT>(hi_pair(a, c), wp, acc[2 * i + 1]);
          }
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < NB; ++s)
        if (s < F || s < N) {
          const float w = lane_value(pw, s);
#pragma unroll
          for (int e = 0; e < E; ++e) acc[e] += w * __uint_as_float(vr[s].w[e]);
        }
    }
    if (p.norm_out) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        acc[e] = DT::rnd(acc[e]);
        ss += acc[e] * acc[e];
      }
      if (p.out_prenorm && ok)
        store_vec<DT, E, true>(global_ptr<S>((uint64_t)p.out_prenorm) + tok * (int64_t)D + eoff, acc);
      ss = wave_sum(ss);  // (zero past the row's end)
      if (lane == 0) s_red[par][wave] = ss;
      __syncthreads();
      const float inv = 1.0f / sqrtf(base_split_total(s_red[par], 1, nw) / (float)D + p.eps);
#pragma unroll
      for (int e = 0; e < E; ++e) acc[e] *= inv;
      if (threadIdx.x == 0 && p.out_inv_rms) p.out_inv_rms[tok] = inv;
    }
    if (ok) store_vec<DT, E, true>(global_ptr<S>((uint64_t)p.out) + tok * (int64_t)D + eoff, acc);
  }
}

template <class DT, int VB, int NB>
__global__ void __launch_bounds__(512) base_split_bwd_kernel(const ReadBwdParams bp) {
  using S = typename DT::S;
  constexpr int E = VB / (int)sizeof(S), F = lr_split_floor(NB), ROW = base_split_row(NB);
  constexpr int NP = NB <= 4 ? 4 : NB <= 8 ? 8 : NB <= 16 ? 16 : NB <= 32 ? 32 : 64;
  const ReadParams& p = bp.f;
  __shared__ SrcTab s_tab;
  __shared__ float s_dw[2][8][ROW], s_ss[2][8][ROW], s_m[2][8][ROW], s_red[2][8];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = uniform_i32(threadIdx.x / kWave), nw = blockDim.x / kWave;
  const int N = p.n_src, D = p.D;
  for (int i = threadIdx.x; i < N; i += blockDim.x) {
    s_tab.vptr[i] = (uint64_t)p.val[i];
    s_tab.vstrb[i] = (uint32_t)p.vstride[i] * (uint32_t)sizeof(S);
    s_tab.dvptr[i] = (uint64_t)bp.dval[i];
  }
  __syncthreads();
  const uint32_t rowb = (uint32_t)D * (uint32_t)sizeof(S);
  const bool ok = (wave * kWave + lane) * E < D, part = (wave + 1) * kWave * E > D;
  const int eoff = ok ? (wave * kWave + lane) * E : 0;
  const int at = min(lane, NB - 1);
  float q[E], qacc[E], bacc = 0.f;
  load_vec<DT, E>((const S*)p.q_static + eoff, q);
#pragma unroll
  for (int e = 0; e < E; ++e) qacc[e] = 0.f;

  int par = 0;
  for (int64_t tok = blockIdx.x; tok < p.n_tok; tok += gridDim.x, par ^= 1) {
    const float pw = lane < N ? bp.saved_w[tok * N + min(lane, N - 1)] : 0.f;
    Raw<DT, E> gr, xr, vr[NB];
    load_raw<DT, E, true>(global_ptr<const S>((uint64_t)bp.gout) + tok * (int64_t)D + eoff, gr);
    // (without an output norm the upstream row stands in: a cache hit, no branch)
    load_raw<DT, E, true>(global_ptr<const S>((uint64_t)(p.norm_out ? p.out_prenorm : bp.gout)) + tok * (int64_t)D + eoff, xr);
    base_split_load<DT, E, NB>(&s_tab, N, tok, eoff, ok, part, vr);
    float g[E];
    unpack<DT, E>(gr, g);
    if (p.norm_out) {
      float x[E], dot = 0.f;
      unpack<DT, E>(xr, x);
#pragma unroll
      for (int e = 0; e < E; ++e) dot += ok ? g[e] * x[e] : 0.f;
      dot = wave_sum(dot);
      if (lane == 0) s_red[par][wave] = dot;
      __syncthreads();
      const float inv = bp.saved_inv[tok];
      const float k3 = inv * inv * inv * (base_split_total(s_red[par], 1, nw) / (float)D);
#pragma unroll
      for (int e = 0; e < E; ++e) g[e] = DT::rnd(inv * g[e] - x[e] * k3);
      if constexpr (sizeof(S) == 2) {
#pragma unroll
        for (int i = 0; i < E / 2; ++i) gr.w[i] = pack2<DT>(g[2 * i], g[2 * i + 1]);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) gr.w[e] = __float_as_uint(g[e]);
      }
    }
    // ---- dW = <g, v> and <v, v> of every source (v is zero past the row's end)
    base_split_sums<NB>(s_dw[par][wave], lane, [&](int s) { return vec_dot<DT, E>(gr, vr[s]); });
    if (p.key_norm) base_split_sums<NB>(s_ss[par][wave], lane, [&](int s) { return vec_dot<DT, E>(vr[s], vr[s]); });
    __syncthreads();
    const float dw = DT::rnd(base_split_total(&s_dw[par][0][at], ROW, nw));
    const float inner = group_sum(lane < N ? pw * dw : 0.f, NP);
    const float dl = lane < N ? pw * (dw - inner) : 0.f;
    bacc += dl;
    const float w_l = DT::rnd(pw);
    float ge_l = DT::rnd(dl);
    float inv_l = 1.f, mr_l = 0.f;
    // ---- key norm: mr = <rnd(ge q), v> inv / D
    if (p.key_norm) {
      inv_l = 1.0f / sqrtf(base_split_total(&s_ss[par][0][at], ROW, nw) / (float)D + p.eps);
      Raw<DT, E> qr;
      if constexpr (sizeof(S) == 2) {
#pragma unroll
        for (int i = 0; i < E / 2; ++i) qr.w[i] = pack2<DT>(q[2 * i], q[2 * i + 1]);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) qr.w[e] = __float_as_uint(q[e]);
      }
      base_split_sums<NB>(s_m[par][wave], lane,
                          [&](int s) { return scaled_dot<DT, E>(qr, lane_value(ge_l, s), vr[s]); });
      __syncthreads();
      mr_l = base_split_total(&s_m[par][0][at], ROW, nw) * inv_l / (float)D;
    }
    // ---- dv = rnd(rnd(w g) + rnd(inv (rnd(ge q) - v inv mr))), dq += ge rnd(v inv),
    // two sources at a time: the packings and the query's products then serve
    // both.  ge q is worked out again rather than kept from the sums above (a
    // register per element and source): the empty asm hides that it is the same.
    asm volatile("" : "+v"(ge_l));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < NB; s += 2) {
      if (s < F || s < N) {
        const bool two = s + 1 < F || s + 1 < N;  // an odd last source is paired with zeros
        const float ge0 = lane_value(ge_l, s), ge1 = two ? lane_value(ge_l, s + 1) : 0.f;
        const float w0 = lane_value(w_l, s), w1 = lane_value(w_l, s + 1);
        const float i0 = lane_value(inv_l, s), i1 = two ? lane_value(inv_l, s + 1) : 0.f;
        const float m0 = lane_value(mr_l, s), m1 = lane_value(mr_l, s + 1);
        float v0[E], v1[E], d0[E], d1[E];
        unpack<DT, E>(vr[s], v0);
        Raw<DT, E> r1 = vr[s + 1];
#pragma unroll
        for (int i = 0; i < Vec<DT, E>::kWords; ++i) r1.w[i] = two ? r1.w[i] : 0u;
        unpack<DT, E>(r1, v1);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          if constexpr (sizeof(S) == 2) {
            const uint32_t one2 = DT::kCode == 1 ? 0x3f803f80u : 0x3c003c00u;
            Raw<DT, 2> kk;
            kk.w[0] = pack2<DT>(ge0 * q[e], ge1 * q[e]);
            float k[2];
            unpack<DT, 2>(kk, k);
            if (p.key_norm) {
              v0[e] *= i0;
              v1[e] *= i1;
              k[0] = i0 * (k[0] - v0[e] * m0);
              k[1] = i1 * (k[1] - v1[e] * m1);
            }
            // rnd(a) + rnd(b): one pack and one v_dot2 with (1, 1)
            d0[e] = dot2<DT>(pack2<DT>(w0 * g[e], k[0]), one2, 0.f);
            d1[e] = dot2<DT>(pack2<DT>(w1 * g[e], k[1]), one2, 0.f);
            qacc[e] = dot2<DT>(pack2<DT>(v0[e], v1[e]), bits16<DT>(ge0) | (bits16<DT>(ge1) << 16), qacc[e]);
          } else {
            float k0 = ge0 * q[e], k1 = ge1 * q[e];
            if (p.key_norm) {
              v0[e] *= i0;
              v1[e] *= i1;
              k0 = i0 * (k0 - v0[e] * m0);
              k1 = i1 * (k1 - v1[e] * m1);
            }
            d0[e] = w0 * g[e] + k0;
            d1[e] = w1 * g[e] + k1;
            qacc[e] += ge0 * v0[e] + ge1 * v1[e];
          }
        }
        if (ok) {
          store_vec<DT, E, true>(global_ptr<S>(row_addr(uniform_u64(s_tab.dvptr[s]), tok, rowb)) + eoff, d0);
          if (two)
            store_vec<DT, E, true>(global_ptr<S>(row_addr(uniform_u64(s_tab.dvptr[s + 1]), tok, rowb)) + eoff, d1);
        }
      }
    }
  }
  if (!bp.partials) return;
  if (bp.part_q >= 0 && ok) {
#pragma unroll
    for (int e = 0; e < E; ++e)
      bp.partials[part_index(bp.part_layout, blockIdx.x, bp.part_q + eoff + e, gridDim.x, bp.n_part)] = qacc[e];
  }
  if (bp.part_bias >= 0 && wave == 0 && lane < N)
    bp.partials[part_index(bp.part_layout, blockIdx.x, bp.part_bias + lane, gridDim.x, bp.n_part)] = bacc;
}

}  // namespace attnres
