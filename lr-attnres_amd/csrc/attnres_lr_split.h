// LR AttnRes read with a token's row split over the waves of one workgroup:
// the head widths that attnres_lr_fast.h cannot give to a single wave (one
// head of 768, 1024 with many sources, 2048; heads of 192, 384, 640 ...), up
// to 64 sources, a static query, any of key norm, bias and output norm.
// Semantics and rounding points are those of attnres_lr.hip.
//
// Bound by HBM like every read here.  The step-by-step kernels gave one
// (head, source) pair to a lane, which walked its key slice alone while the
// value rows waited behind workgroup barriers (13 lanes of a wave busy with one
// head), in groups of eight sources.  Here:
//   * a wave owns 64 lane vectors of the row (256 or 512 columns) and has all
//     N of its value vectors in flight at once, every load of the token
//     issued before the first use;
//   * a key slice is spread over its 16-byte chunks, one per lane (kch lanes a
//     pair, a power of two), the norm and the dot product folded by DPP;
//   * forward: each wave scores the heads of its own columns for itself, so
//     that nothing crosses waves (the output norm adds one barrier);
//   * backward: dW partials of each 16-lane row go to LDS (head widths are
//     whole rows of 16 lanes), one barrier per token (two with the output
//     norm), buffers alternating between tokens; the pairs' key gradients are
//     spread over the waves, a wave taking pairs of its own columns' heads, so
//     the saved weights it loaded serve both.  The static query's gradient stays
//     in registers per (pair, chunk) and is folded over the sources once per
//     workgroup.
//
// Measured (one MI355X, bf16, one head of d768, 13 sources, rank 64, output
// norm, 16384 tokens): forward 85 us (420 MB, 4.9 TB/s), backward 154 us
// (765 MB, 5.0 TB/s); step by step 181 and 526.  One token, 9 sources of d1024,
// rank 32: 8.0 us against 15.1.
#pragma once

#include "attnres_device.h"
#include "attnres_launch.h"
#include "attnres_lr_fast.h"
#include "attnres_params.h"

namespace attnres {

// Source slots: instantiated counts, and the smallest source count each holds
// (slots below it need no guard).
__host__ __device__ constexpr int lr_split_slots(int n) {
  return n <= 4 ? 4 : n <= 32 ? (n + 1) / 2 * 2 : (n + 3) / 4 * 4;
}
__host__ __device__ constexpr int lr_split_floor(int nb) {
  return nb <= 4 ? 1 : nb <= 32 ? nb - 1 : nb - 3;
}

// Per-wave column ownership and the workgroup's LDS carve-up, shared by both
// directions.  floats: tables | query (raw) | pair table | per wave [2][nh * np] | tail
struct LrSplitLds {
  SrcTab* tab;
  char* q;         // [R] raw elements
  uint16_t* pair;  // [H * N]: head << 8 | source
  float* wave;     // this wave's 2 * nh * np floats
  float* tail;
};
__host__ __device__ inline size_t lr_split_lds_head(int R, int es, int HN, int wpt, int nh, int np) {
  return sizeof(SrcTab) + ((size_t)R * es + 15) / 16 * 16 + ((size_t)HN * 2 + 15) / 16 * 16 +
         (size_t)wpt * 2 * nh * np * sizeof(float);
}
__device__ __forceinline__ LrSplitLds lr_split_lds(float* base, const ReadParams& p, int es, int wpt, int wave) {
  LrSplitLds l;
  l.tab = (SrcTab*)base;
  l.q = (char*)base + sizeof(SrcTab);
  l.pair = (uint16_t*)(l.q + (p.R * es + 15) / 16 * 16);
  float* w = (float*)((char*)l.pair + (p.H * p.n_src * 2 + 15) / 16 * 16);
  l.wave = w + wave * 2 * p.nh * p.np;
  l.tail = w + wpt * 2 * p.nh * p.np;
  return l;
}

template <class DT>
__device__ __forceinline__ void lr_split_tables(const ReadParams& p, const LrSplitLds& l) {
  using S = typename DT::S;
  for (int i = threadIdx.x; i < p.n_src; i += blockDim.x) {
    l.tab->vptr[i] = (uint64_t)p.val[i];
    l.tab->vstrb[i] = (uint32_t)p.vstride[i] * (uint32_t)sizeof(S);
    l.tab->kptr[i] = (uint64_t)p.key[i];
    l.tab->kstrb[i] = (uint32_t)p.kstride[i] * (uint32_t)sizeof(S);
  }
  for (int i = threadIdx.x; i < p.R; i += blockDim.x) ((S*)l.q)[i] = ((const S*)p.q_static)[i];
  for (int i = threadIdx.x; i < p.H * p.n_src; i += blockDim.x) {
    const int h = i / p.n_src;
    l.pair[i] = (uint16_t)(h << 8 | (i - h * p.n_src));
  }
}

// the token's value vectors of this lane (slots past N re-read the last source)
template <class DT, int E, int NB>
__device__ __forceinline__ void lr_split_load(const SrcTab* tab, int N, int64_t tok, int eoff, Raw<DT, E> (&vr)[NB]) {
  using S = typename DT::S;
  constexpr int F = lr_split_floor(NB);
#pragma unroll
  for (int s = 0; s < NB; ++s)
    load_raw<DT, E, true>(global_ptr<const S>(row_base(tab, s < F ? s : min(s, N - 1), tok)) + eoff, vr[s]);
}

// one 16-byte chunk of a key: khat (rnd(k / rms) with key norm) and 1/rms, the
// slice's kch lanes together
template <class DT, int KV>
__device__ __forceinline__ float lr_split_key(const float (&k)[KV], bool key_norm, int kch, int rh, float eps,
                                              float (&kh)[KV]) {
  float inv = 1.f;
  if (key_norm) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < KV; ++i) ss += k[i] * k[i];
    inv = 1.0f / sqrtf(group_sum(ss, kch) / (float)rh + eps);
  }
#pragma unroll
  for (int i = 0; i < KV; ++i) kh[i] = key_norm ? DT::rnd(k[i] * inv) : k[i];
  return inv;
}

template <class DT, int VB, int NB>
__global__ void __launch_bounds__(512) lr_split_fwd_kernel(const ReadParams p) {
  using S = typename DT::S;
  constexpr int E = VB / (int)sizeof(S), KV = 16 / (int)sizeof(S);
  constexpr int F = lr_split_floor(NB);
  constexpr int KF = NB <= 16 ? 2 : 4;  // key chunks loaded ahead of the value rows
  extern __shared__ float lds_base[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = uniform_i32(threadIdx.x / kWave), wpt = blockDim.x / kWave;
  const int N = p.n_src, D = p.D, dh = p.dh, rh = p.rh, np = p.np, kch = p.kch;
  const LrSplitLds l = lr_split_lds(lds_base, p, (int)sizeof(S), wpt, wave);
  float* s_lg = l.wave;
  uint32_t* s_w = (uint32_t*)(l.wave + p.nh * np);
  lr_split_tables<DT>(p, l);
  __syncthreads();

  const int c0 = wave * kWave * E;
  const int h_lo = c0 / dh, nh = min(c0 + kWave * E - 1, D - 1) / dh - h_lo + 1;
  const bool ok = c0 + lane * E < D;
  const int eoff = ok ? c0 + lane * E : 0;
  const int hd = ok ? eoff / dh - h_lo : 0;
  const int pairs = nh * N, lk = __ffs(kch) - 1, ppi = kWave >> lk;
  const int chunk = lane & (kch - 1), pl = lane >> lk;

  int par = 0;
  for (int64_t tok = blockIdx.x; tok < p.n_tok; tok += gridDim.x, par ^= 1) {
    auto key_load = [&](int it, Raw<DT, KV>& r) {
      const int hs = l.pair[h_lo * N + min(it * ppi + pl, pairs - 1)], s = hs & 255;
      const uint64_t a = row_addr(l.tab->kptr[s], tok, l.tab->kstrb[s]);
      load_raw<DT, KV>(global_ptr<const S>(a) + (hs >> 8) * rh + chunk * KV, r);
    };
    auto score = [&](int it, const Raw<DT, KV>& r) {
      const int pi = min(it * ppi + pl, pairs - 1), hs = l.pair[h_lo * N + pi];
      float k[KV], kh[KV], q[KV];
      unpack<DT, KV>(r, k);
      lr_split_key<DT, KV>(k, p.key_norm, kch, rh, p.eps, kh);
      load_vec<DT, KV>((const S*)l.q + (hs >> 8) * rh + chunk * KV, q);
      float d = 0.f;
#pragma unroll
      for (int i = 0; i < KV; ++i) d += kh[i] * q[i];
      d = group_sum(d, kch);
      const float lg = DT::rnd(DT::rnd(d) * p.scale) + (p.bias ? p.bias[hs & 255] : 0.f);
      if (chunk == 0 && it * ppi + pl < pairs) s_lg[pi] = lg;
    };
    Raw<DT, KV> kr[KF];
#pragma unroll
    for (int i = 0; i < KF; ++i) key_load(i, kr[i]);
    Raw<DT, E> vr[NB];
    lr_split_load<DT, E, NB>(l.tab, N, tok, eoff, vr);
#pragma unroll
    for (int i = 0; i < KF; ++i)
      if (i * ppi < pairs) score(i, kr[i]);
    for (int i = KF; i * ppi < pairs; ++i) {
      key_load(i, kr[0]);
      score(i, kr[0]);
    }
    wave_sync();
    // ---- softmax: (head, source) lanes, np lanes a head
    for (int b = 0; b < nh * np; b += kWave) {
      const int hh = (b + lane) / np, s = (b + lane) & (np - 1);
      const bool own = hh < nh && s < N;
      const float lg = own ? s_lg[hh * N + s] : -INFINITY;
      const float lm = group_max(lg, np);
      const float ex = own ? expf(lg - lm) : 0.f;
      const float pw = ex / group_sum(ex, np);
      if (hh < nh) {
        const float w = own ? DT::rnd(pw) : 0.f;
        if constexpr (sizeof(S) == 2) ((uint16_t*)s_w)[b + lane] = (uint16_t)bits16<DT>(w);
        else s_w[b + lane] = __float_as_uint(w);
        // a head is written by the wave that holds its first column
        if (own && p.weights && (h_lo + hh) * dh >= c0) p.weights[(tok * p.H + h_lo + hh) * N + s] = pw;
      }
    }
    wave_sync();
    // ---- mix
    float acc[E];
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] = 0.f;
    if constexpr (sizeof(S) == 2) {
#pragma unroll
      for (int s = 0; s < NB; s += 2) {
        if (s < F || s < N) {
          const uint32_t wp = s_w[(hd * np + s) >> 1];
          const bool two = s + 1 < F || s + 1 < N;  // an odd last source is paired with zeros
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
          const float w = __uint_as_float(s_w[hd * np + s]);
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
      ss = wave_sum(ok ? ss : 0.f);
      float* s_red = l.tail + par * 8;
      if (lane == 0) s_red[wave] = ss;
      __syncthreads();
      ss = 0.f;
      for (int w = 0; w < wpt; ++w) ss += s_red[w];
      const float inv = 1.0f / sqrtf(ss / (float)D + p.eps);
#pragma unroll
      for (int e = 0; e < E; ++e) acc[e] *= inv;
      if (threadIdx.x == 0 && p.out_inv_rms) p.out_inv_rms[tok] = inv;
    }
    if (ok) store_vec<DT, E, true>(global_ptr<S>((uint64_t)p.out) + tok * (int64_t)D + eoff, acc);
    wave_sync();  // this token's weights are read before the next one writes them
  }
}

// KI: (pair, chunk) items of the key gradients per lane
template <class DT, int VB, int NB, int KI>
__global__ void __launch_bounds__(512) lr_split_bwd_kernel(const ReadBwdParams bp) {
  using S = typename DT::S;
  constexpr int E = VB / (int)sizeof(S), KV = 16 / (int)sizeof(S), RE = 16 * E;
  constexpr int F = lr_split_floor(NB);
  const ReadParams& p = bp.f;
  extern __shared__ float lds_base[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = uniform_i32(threadIdx.x / kWave), wpt = blockDim.x / kWave;
  const int N = p.n_src, D = p.D, H = p.H, R = p.R, dh = p.dh, rh = p.rh, np = p.np, kch = p.kch;
  const LrSplitLds l = lr_split_lds(lds_base, p, (int)sizeof(S), wpt, wave);
  float* s_p = l.wave;            // saved weights [nh][np]
  float* s_dl = l.wave + p.nh * np;
  float* s_red = l.tail;          // [2][8]
  float* s_dw = l.tail + 16;      // [2][4 * wpt][N]: dW partials of each 16-lane row
  lr_split_tables<DT>(p, l);
  for (int i = threadIdx.x; i < N; i += blockDim.x) {
    l.tab->dvptr[i] = (uint64_t)bp.dval[i];
    l.tab->dkptr[i] = (uint64_t)bp.dkey[i];
  }
  __syncthreads();

  const int c0 = wave * kWave * E, c1 = min(c0 + kWave * E, D);
  const int h_lo = c0 / dh, nh = (c1 - 1) / dh - h_lo + 1;
  const bool ok = c0 + lane * E < D;
  const int eoff = ok ? c0 + lane * E : 0;
  const int hd = ok ? eoff / dh - h_lo : 0;
  // this wave's pairs: a share of H * N by its columns, so heads of its columns
  const int p0 = (int)((int64_t)H * N * c0 / D), p1 = (int)((int64_t)H * N * c1 / D);
  const int lk = __ffs(kch) - 1, ppi = kWave >> lk, chunk = lane & (kch - 1), pl = lane >> lk;
  const uint32_t rowb = (uint32_t)D * (uint32_t)sizeof(S);
  int hs[KI];
  bool item[KI];
  float qacc[KI][KV], bacc[KI];
#pragma unroll
  for (int i = 0; i < KI; ++i) {
    item[i] = p0 + i * ppi + pl < p1;
    hs[i] = l.pair[item[i] ? p0 + i * ppi + pl : p0 < H * N ? p0 : 0];
    bacc[i] = 0.f;
#pragma unroll
    for (int j = 0; j < KV; ++j) qacc[i][j] = 0.f;
  }

  int par = 0;
  for (int64_t tok = blockIdx.x; tok < p.n_tok; tok += gridDim.x, par ^= 1) {
    // ---- every load of the token
    float w0;
    {
      const int hh = min(lane / np, nh - 1), s = min(lane & (np - 1), N - 1);
      w0 = bp.saved_w[(tok * H + h_lo + hh) * N + s];
    }
    Raw<DT, KV> kr[KI];
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int s = hs[i] & 255;
      const uint64_t a = row_addr(l.tab->kptr[s], tok, l.tab->kstrb[s]);
      load_raw<DT, KV>(global_ptr<const S>(a) + (hs[i] >> 8) * rh + chunk * KV, kr[i]);
    }
    Raw<DT, E> gr, xr, vr[NB];
    load_raw<DT, E, true>(global_ptr<const S>((uint64_t)bp.gout) + tok * (int64_t)D + eoff, gr);
    // (without an output norm the upstream row stands in: a cache hit, no branch)
    load_raw<DT, E, true>(global_ptr<const S>((uint64_t)(p.norm_out ? p.out_prenorm : bp.gout)) + tok * (int64_t)D + eoff, xr);
    lr_split_load<DT, E, NB>(l.tab, N, tok, eoff, vr);
    float g[E];
    unpack<DT, E>(gr, g);
#pragma unroll
    for (int e = 0; e < E; ++e) g[e] = ok ? g[e] : 0.f;
    if (p.norm_out) {
      float x[E], dot = 0.f;
      unpack<DT, E>(xr, x);
#pragma unroll
      for (int e = 0; e < E; ++e) dot += g[e] * x[e];
      dot = wave_sum(dot);
      if (lane == 0) s_red[par * 8 + wave] = dot;
      __syncthreads();
      dot = 0.f;
      for (int w = 0; w < wpt; ++w) dot += s_red[par * 8 + w];
      const float inv = bp.saved_inv[tok];
      const float k3 = inv * inv * inv * (dot / (float)D);
#pragma unroll
      for (int e = 0; e < E; ++e) g[e] = ok ? DT::rnd(inv * g[e] - x[e] * k3) : 0.f;
    }
    // saved weights of this wave's heads, np lanes a head
    if (lane < nh * np) s_p[lane] = w0;
    for (int b = kWave; b < nh * np; b += kWave) {
      const int hh = min((b + lane) / np, nh - 1), s = min((b + lane) & (np - 1), N - 1);
      if (b + lane < nh * np) s_p[b + lane] = bp.saved_w[(tok * H + h_lo + hh) * N + s];
    }
    wave_sync();
    // ---- dW partials of each 16-lane row
    uint32_t gp[E];
    if constexpr (sizeof(S) == 2) {
#pragma unroll
      for (int i = 0; i < E / 2; ++i) gp[i] = pack2<DT>(g[2 * i], g[2 * i + 1]);
    }
    float* dwr = s_dw + (par * 4 * wpt + wave * 4 + (lane >> 4)) * N;
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      if (s < F || s < N) {
        float d = 0.f;
        if constexpr (sizeof(S) == 2) {
#pragma unroll
          for (int i = 0; i < E / 2; ++i) d = dot2<DT>(gp[i], vr[s].w[i], d);
        } else {
#pragma unroll
          for (int e = 0; e < E; ++e) d += g[e] * __uint_as_float(vr[s].w[e]);
        }
        d += dpp_f32<kDppXor1>(d);
        d += dpp_f32<kDppXor2>(d);
        d += dpp_f32<kDppHalfMirror>(d);
        d += dpp_f32<kDppMirror>(d);
        if ((lane & 15) == 0) dwr[s] = d;
      }
    }
    // ---- dv = rnd(w) g (the store rounds)
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      if (s < F || s < N) {
        const float w = DT::rnd(s_p[hd * np + s]);
        float dv[E];
#pragma unroll
        for (int e = 0; e < E; ++e) dv[e] = w * g[e];
        if (ok)
          store_vec<DT, E, true>(global_ptr<S>(row_addr(uniform_u64(l.tab->dvptr[s]), tok, rowb)) + eoff, dv);
      }
    }
    __syncthreads();
    // ---- softmax backward of this wave's heads
    for (int b = 0; b < nh * np; b += kWave) {
      const int hh = (b + lane) / np, s = (b + lane) & (np - 1);
      const bool own = hh < nh && s < N;
      float dw = 0.f;
      const int rows = dh / RE;
      const float* src = s_dw + (par * 4 * wpt + (h_lo + min(hh, nh - 1)) * rows) * N + min(s, N - 1);
      for (int r = 0; r < rows; r += 4) {
        float x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = src[min(r + u, rows - 1) * N];
#pragma unroll
        for (int u = 0; u < 4; ++u) dw += r + u < rows ? x[u] : 0.f;
      }
      dw = DT::rnd(dw);
      const float pw = own ? s_p[b + lane] : 0.f;
      const float inner = group_sum(own ? pw * dw : 0.f, np);
      if (own) s_dl[b + lane] = pw * (dw - inner);
    }
    wave_sync();
    // ---- key gradients and the query's, a 16-byte chunk per lane
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      if (i > 0 && p0 + i * ppi >= p1) continue;  // wave-uniform
      const int h = hs[i] >> 8, s = hs[i] & 255;
      const float dl = item[i] ? s_dl[(h - h_lo) * np + s] : 0.f;
      const float ge = DT::rnd(DT::rnd(dl) * p.scale);
      float k[KV], kh[KV], q[KV], t[KV];
      unpack<DT, KV>(kr[i], k);
      const float inv = lr_split_key<DT, KV>(k, p.key_norm, kch, rh, p.eps, kh);
      load_vec<DT, KV>((const S*)l.q + h * rh + chunk * KV, q);
      float m = 0.f;
#pragma unroll
      for (int j = 0; j < KV; ++j) {
        t[j] = DT::rnd(ge * q[j]);
        m += t[j] * (k[j] * inv);
      }
      const float mr = group_sum(m, kch) / (float)rh;
#pragma unroll
      for (int j = 0; j < KV; ++j) {
        qacc[i][j] += ge * kh[j];
        if (p.key_norm) t[j] = inv * (t[j] - k[j] * inv * mr);
      }
      if (item[i]) {
        bacc[i] += dl;
        store_vec<DT, KV>(global_ptr<S>(l.tab->dkptr[s]) + tok * (int64_t)R + h * rh + chunk * KV, t);
      }
    }
    wave_sync();  // this token's tables are read before the next one writes them
  }

  // ---- fold the items over the sources into this workgroup's partial row
  if (!bp.partials) return;
  __syncthreads();
  float* s_c = s_dw;  // [H * N][rh + 1]: the query's slots, the bias in the last
#pragma unroll
  for (int i = 0; i < KI; ++i)
    if (item[i]) {
      float* row = s_c + ((hs[i] >> 8) * N + (hs[i] & 255)) * (rh + 1);
#pragma unroll
      for (int j = 0; j < KV; ++j) row[chunk * KV + j] = qacc[i][j];
      if (chunk == 0) row[rh] = bacc[i];
    }
  __syncthreads();
  for (int i = threadIdx.x; i < bp.n_part; i += blockDim.x) {
    float a = 0.f;
    if (bp.part_q >= 0 && i >= bp.part_q && i < bp.part_q + R) {
      const int h = (i - bp.part_q) / rh, j = (i - bp.part_q) - h * rh;
      for (int s = 0; s < N; ++s) a += s_c[(h * N + s) * (rh + 1) + j];
    } else {
      for (int h = 0; h < H; ++h) a += s_c[(h * N + i - bp.part_bias) * (rh + 1) + rh];
    }
    bp.partials[(int64_t)i * gridDim.x + blockIdx.x] = a;  // slot-major
  }
}

// launch switch: L.nmax = source slots, L.vb = vector bytes (8 / 16); 16-byte
// vectors hold up to 32 sources
#define ATTNRES_LR_SPLIT_NB8(CASE) CASE(36) CASE(40) CASE(44) CASE(48) CASE(52) CASE(56) CASE(60) CASE(64)
#define ATTNRES_LR_SPLIT_NB(CASE) \
  CASE(4) CASE(6) CASE(8) CASE(10) CASE(12) CASE(14) CASE(16) CASE(18) CASE(20) CASE(22) CASE(24) CASE(26) CASE(28) \
  CASE(30) CASE(32)

}  // namespace attnres
