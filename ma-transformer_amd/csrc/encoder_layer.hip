// encoder_layer.hip -- the reference encoder layer's eval-mode forward in one
// kernel (C-ABI in include/ma_encoder.h).
//
// Reference: CustomTransformerEncoderLayer.forward (src/model.py:42-53) with
// its SparseAttention (src/layers/sparse_attention.py:49-86: one head over
// [B, S, d_model], window w, keys [i-w, i+w]) and torch's LayerNorm / Linear.
//
// One workgroup (4 waves) per 16 consecutive tokens of [B*S, d_model]:
//   1. attention (16 lanes per token, d_model/16 values per lane): the row's
//      keys are its sequence's rows [i-w, i+w] (K = V = src), an online
//      softmax in registers; h = src + attn; LayerNorm1 -> LDS.
//   2. linear1 + bias + ReLU on fp32 MFMA (16x16x4): wave v computes hidden
//      units [v*d, (v+1)*d) of the 16 tokens -> LDS.
//   3. linear2 on fp32 MFMA: wave v contracts hidden units [v*d, (v+1)*d)
//      for every output column; the four partial sums meet in LDS and are
//      added in a fixed order.
//   4. residual, bias, LayerNorm2; each token's row stored once.
// MFMA operands: for 4 consecutive 16x16x4 steps, lane group g (lane/16)
// feeds contraction indices 16t + 4g + {0..3}, so each lane fetches its four
// A values (LDS) and four B values (the weight row, from L2) as one 16-byte
// read each.  The contraction order therefore differs from torch's; the
// arithmetic is float32 throughout.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>

#include "../../include/ma_encoder.h"
#include "device_common.h"
#include "host_common.h"

namespace {

using ma_dev::f32x4;
using ma_dev::mfma_f32;

constexpr int kTokens = 16;  // tokens per workgroup

struct EncArgs {
  const float* src;
  const float* attn;  // null: computed here
  float* out;
  const float *g1, *be1, *w1, *bi1, *w2, *bi2, *g2, *be2;
  int64_t rows;  // batch * seq_len
  int32_t seq_len;
  int32_t window;  // clipped to [-1, seq_len]
  float scale;
  float eps;
};

template <int D>
struct EncGeom {
  static constexpr int F = 4 * D;       // hidden units
  static constexpr int EPT = D / 16;    // values per lane in the row passes (16 lanes per token)
  static constexpr int XS = D + 4;      // LDS row stride (floats) of LayerNorm1's output
  static constexpr int ZS = F + 4;      // of relu(linear1)
  static constexpr int PS = D + 4;      // of linear2's per-wave partial sums
  static constexpr int ZBUF = 16 * ZS > 64 * PS ? 16 * ZS : 64 * PS;
};

template <int N>
__device__ __forceinline__ void load_row(const float* p, float (&x)[N]) {
  if constexpr (N % 4 == 0) {
#pragma unroll
    for (int e = 0; e < N; e += 4) {
      const float4 v = *reinterpret_cast<const float4*>(p + e);
      x[e] = v.x;
      x[e + 1] = v.y;
      x[e + 2] = v.z;
      x[e + 3] = v.w;
    }
  } else if constexpr (N == 2) {
    const float2 v = *reinterpret_cast<const float2*>(p);
    x[0] = v.x;
    x[1] = v.y;
  } else {
    x[0] = p[0];
  }
}

template <int N>
__device__ __forceinline__ void store_row(float* p, const float (&x)[N]) {
  if constexpr (N % 4 == 0) {
#pragma unroll
    for (int e = 0; e < N; e += 4) *reinterpret_cast<float4*>(p + e) = make_float4(x[e], x[e + 1], x[e + 2], x[e + 3]);
  } else if constexpr (N == 2) {
    *reinterpret_cast<float2*>(p) = make_float2(x[0], x[1]);
  } else {
    p[0] = x[0];
  }
}

// Sum over the 16 lanes of a token (lanes 16k .. 16k+15 of a wave).
__device__ __forceinline__ float sum16(float x) {
#pragma unroll
  for (int m = 8; m >= 1; m >>= 1) x += __shfl_xor(x, m, 64);
  return x;
}

// LayerNorm of a 16-lane-distributed row: (x - mean) / sqrt(var + eps) * g + b,
// biased variance, as torch.nn.LayerNorm.
template <int N, int D>
__device__ __forceinline__ void layer_norm(float (&x)[N], const float (&gw)[N], const float (&bw)[N], float eps) {
  float s = 0.0f;
#pragma unroll
  for (int e = 0; e < N; ++e) s += x[e];
  const float mean = sum16(s) / (float)D;
  float q = 0.0f;
#pragma unroll
  for (int e = 0; e < N; ++e) {
    const float c = x[e] - mean;
    q = fmaf(c, c, q);
  }
  const float rstd = 1.0f / sqrtf(sum16(q) / (float)D + eps);
#pragma unroll
  for (int e = 0; e < N; ++e) x[e] = (x[e] - mean) * rstd * gw[e] + bw[e];
}

template <int D>
__global__ __launch_bounds__(256) void encoder_layer_kernel(EncArgs a) {
  using G = EncGeom<D>;
  constexpr int F = G::F, EPT = G::EPT, NT = D / 16;  // NT: 16-wide column tiles (and 16-deep k groups) per wave
  __shared__ __attribute__((aligned(16))) float xs[kTokens * G::XS];
  __shared__ __attribute__((aligned(16))) float zs[G::ZBUF];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wv = tid >> 6;
  const int r = tid >> 4, u = tid & 15;  // token of the tile, lane within the token
  const int d0 = u * EPT;
  const int64_t m = (int64_t)blockIdx.x * kTokens + r;
  const bool live = m < a.rows;

  // ---- 1. attention, residual, LayerNorm1
  float x[EPT], h[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) x[e] = 0.0f;
  if (live) load_row<EPT>(a.src + m * D + d0, x);
  // the lane's slices of both norms' affine parameters and linear2's bias,
  // loaded up front so their round trip overlaps the attention
  float g1[EPT], be1[EPT], g2[EPT], be2[EPT], b2[EPT];
  load_row<EPT>(a.g1 + d0, g1);
  load_row<EPT>(a.be1 + d0, be1);
  load_row<EPT>(a.g2 + d0, g2);
  load_row<EPT>(a.be2 + d0, be2);
  load_row<EPT>(a.bi2 + d0, b2);
  if (a.attn) {
    float at[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) at[e] = 0.0f;
    if (live) load_row<EPT>(a.attn + m * D + d0, at);
#pragma unroll
    for (int e = 0; e < EPT; ++e) h[e] = x[e] + at[e];
  } else {
    const int64_t i = live ? m % a.seq_len : 0;
    const int64_t base = m - i;  // the sequence's first token
    const int64_t jlo = live ? (i - a.window > 0 ? i - a.window : 0) : 1;
    const int64_t jhi = live ? (i + a.window < a.seq_len - 1 ? i + a.window : a.seq_len - 1) : 0;
    float mx = -INFINITY, l = 0.0f, acc[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) acc[e] = 0.0f;
    // keys in batches of kKB: the batch's rows are loaded together (one
    // round trip), rows past the window's end re-read its last row and get
    // no weight; the loop bounds are uniform across the token's 16 lanes
    constexpr int kKB = 8;  // the reference window (w = 3, 7 keys) in one batch
    for (int64_t j = jlo; j <= jhi; j += kKB) {
      float kv[kKB][EPT], s[kKB];
#pragma unroll
      for (int c = 0; c < kKB; ++c) {
        const int64_t jj = j + c <= jhi ? j + c : jhi;
        load_row<EPT>(a.src + (base + jj) * D + d0, kv[c]);
      }
#pragma unroll
      for (int c = 0; c < kKB; ++c) {
        float t = 0.0f;
#pragma unroll
        for (int e = 0; e < EPT; ++e) t = fmaf(x[e], kv[c][e], t);
        s[c] = t;
      }
      float mn = mx;
#pragma unroll
      for (int c = 0; c < kKB; ++c) {
        const float t = sum16(s[c]) * a.scale;
        s[c] = j + c <= jhi ? t : -INFINITY;
        mn = fmaxf(mn, s[c]);
      }
      const float cf = expf(mx - mn);
      l *= cf;
#pragma unroll
      for (int e = 0; e < EPT; ++e) acc[e] *= cf;
#pragma unroll
      for (int c = 0; c < kKB; ++c) {
        const float p = expf(s[c] - mn);  // 0 for the batch's padding
        l += p;
#pragma unroll
        for (int e = 0; e < EPT; ++e) acc[e] = fmaf(p, kv[c][e], acc[e]);
      }
      mx = mn;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int e = 0; e < EPT; ++e) h[e] = x[e] + acc[e] * inv;
  }
  layer_norm<EPT, D>(h, g1, be1, a.eps);
  store_row<EPT>(xs + r * G::XS + d0, h);
  __syncthreads();

  const int lr = lane & 15, lg = lane >> 4;

  // ---- 2. linear1 + bias + ReLU: wave wv, hidden units [wv*D, (wv+1)*D)
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) {
    const int col = wv * D + ct * 16 + lr;
    const float* wrow = a.w1 + (int64_t)col * D;
    float4 bv[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) bv[t] = *reinterpret_cast<const float4*>(wrow + 16 * t + 4 * lg);
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float4 av = *reinterpret_cast<const float4*>(xs + lr * G::XS + 16 * t + 4 * lg);
      acc = mfma_f32(av.x, bv[t].x, acc);
      acc = mfma_f32(av.y, bv[t].y, acc);
      acc = mfma_f32(av.z, bv[t].z, acc);
      acc = mfma_f32(av.w, bv[t].w, acc);
    }
    const float bias = a.bi1[col];
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) zs[(4 * lg + jj) * G::ZS + col] = fmaxf(acc[jj] + bias, 0.0f);
  }
  __syncthreads();

  // ---- 3. linear2: wave wv contracts hidden units [wv*D, (wv+1)*D) for every column
  f32x4 part[NT];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) {
    const int col = ct * 16 + lr;
    const float* wrow = a.w2 + (int64_t)col * F + wv * D;
    float4 bv[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) bv[t] = *reinterpret_cast<const float4*>(wrow + 16 * t + 4 * lg);
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float4 av = *reinterpret_cast<const float4*>(zs + lr * G::ZS + wv * D + 16 * t + 4 * lg);
      acc = mfma_f32(av.x, bv[t].x, acc);
      acc = mfma_f32(av.y, bv[t].y, acc);
      acc = mfma_f32(av.z, bv[t].z, acc);
      acc = mfma_f32(av.w, bv[t].w, acc);
    }
    part[ct] = acc;
  }
  __syncthreads();  // every wave is done reading zs: its space takes the partial sums
  float* ps = zs;
#pragma unroll
  for (int ct = 0; ct < NT; ++ct)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) ps[(wv * 16 + 4 * lg + jj) * G::PS + ct * 16 + lr] = part[ct][jj];
  __syncthreads();

  // ---- 4. residual + bias, LayerNorm2, store
  float y[EPT], p0[EPT], p1[EPT], p2[EPT], p3[EPT];
  load_row<EPT>(ps + (0 * 16 + r) * G::PS + d0, p0);
  load_row<EPT>(ps + (1 * 16 + r) * G::PS + d0, p1);
  load_row<EPT>(ps + (2 * 16 + r) * G::PS + d0, p2);
  load_row<EPT>(ps + (3 * 16 + r) * G::PS + d0, p3);
#pragma unroll
  for (int e = 0; e < EPT; ++e) y[e] = h[e] + ((((p0[e] + p1[e]) + p2[e]) + p3[e]) + b2[e]);
  layer_norm<EPT, D>(y, g2, be2, a.eps);
  if (live) store_row<EPT>(a.out + m * D + d0, y);
}

// ------------------------------------------------------------------ whole model
//
// encoder_model_kernel: TransformerModel.forward (reference src/model.py:74-92)
// in one launch.  Sequences are independent, so a workgroup (8 waves) carries
// whole sequences (one, or several short ones of a batch above one per CU)
// through every layer in LDS: no activation touches memory between the input
// and the prediction, and the layers cost no launches.  Bound
// by latency: per layer two weight reads from L2 (a wave's share of linear1 is
// requested before the attention, of linear2 before linear1's products) and a
// chain of five barriers.  The work of a layer is the encoder_layer_kernel's:
//   attention, residual, LayerNorm1 (16 lanes per token; keys in LDS) -> hs
//   linear1 + ReLU: wave w takes hidden tiles w, w + 8, ...            -> zs
//   linear2: wave w takes column tile w % NT and part w / NT of the
//   hidden units; the parts are added in a fixed order                 -> ps
//   residual, LayerNorm2                                               -> xs
// With one sequence, the last layer computes only the 16-token tile of the
// last token, which is all the decoder reads.  The reference's configuration
// (batch 64, sequence 10, d_model 64, 4 layers): 29 us a call, against 129 us as
// four layer launches and the torch operations around them.
struct ModelLayer {
  const float *g1, *be1, *w1, *bi1, *w2, *bi2, *g2, *be2;
  int32_t window;
  float eps;
};
struct ModelArgs {
  const float *src, *we, *bie, *pos, *wd, *bid;
  float* out;
  int32_t S, in, layers;
  int32_t batch, per_wg;  // sequences, and of them per workgroup
  float scale, root;  // softmax scale, sqrt(d_model)
  ModelLayer layer[MA_ENCODER_MAX_LAYERS];
};

template <int D>
struct ModelGeom {
  static constexpr int F = 4 * D, EPT = D / 16, XS = D + 4, ZS = F + 4, NT = D / 16;
  static constexpr int KS = 8 / NT < F / 16 ? 8 / NT : F / 16;  // parts of linear2's contraction
  // linear2's partial sums take xs's place when there is one part (each lane
  // reads what it then overwrites)
  static constexpr int lds(int mt) { return 16 * mt * (2 * XS + ZS + (KS > 1 ? KS * XS : 0)) * 4; }
  static constexpr int max_tiles() {
    int m = 4;
    while (lds(m) > 160 * 1024) --m;
    return m;
  }
};

template <int D, int MT>
__global__ __launch_bounds__(512) void encoder_model_kernel(ModelArgs a) {
  using G = ModelGeom<D>;
  constexpr int F = G::F, EPT = G::EPT, XS = G::XS, ZS = G::ZS, NT = G::NT, KS = G::KS, T = 16 * MT;
  constexpr int N1 = (F / 16 + 7) / 8;    // linear1 hidden tiles per wave
  constexpr int NC = N1 < 2 ? N1 : 2;     // of them in registers at a time
  constexpr int K2 = F / KS / 16;         // linear2 16-deep groups per wave
  constexpr int KC = K2 < 8 ? K2 : 8;     // of them in registers at a time
  extern __shared__ __attribute__((aligned(16))) float sm[];
  float* xs = sm;
  float* hs = xs + T * XS;
  float* zs = hs + T * XS;
  float* ps = KS > 1 ? zs + T * ZS : xs;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = tid >> 4, u = tid & 15, d0 = u * EPT;
  const int lr = lane & 15, lg = lane >> 4;
  const int S = a.S;
  const int b0 = blockIdx.x * a.per_wg;                 // first sequence
  const int V = min(a.per_wg, a.batch - b0) * S;        // tokens in use

  // ---- input projection and position
  for (int t = r; t < T; t += 32) {
    float x[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) x[e] = 0.0f;
    if (t < V) {
      const float* in = a.src + ((int64_t)b0 * S + t) * a.in;
      for (int i = 0; i < a.in; ++i) {
        const float v = in[i];
#pragma unroll
        for (int e = 0; e < EPT; ++e) x[e] = fmaf(v, a.we[(int64_t)(d0 + e) * a.in + i], x[e]);
      }
      float bi[EPT], po[EPT];
      load_row<EPT>(a.bie + d0, bi);
      load_row<EPT>(a.pos + (int64_t)(b0 + t / S) * D + d0, po);
#pragma unroll
      for (int e = 0; e < EPT; ++e) x[e] = (x[e] + bi[e]) * a.root + po[e];
    }
    store_row<EPT>(xs + t * XS + d0, x);
  }
  __syncthreads();

  for (int l = 0; l < a.layers; ++l) {
    const ModelLayer& p = a.layer[l];
    // first 16-token tile this layer computes
    const int mt0 = l + 1 == a.layers && V == S ? (S - 1) / 16 : 0;
    // this wave's first hidden tiles of linear1, in flight during the attention
    float4 w1[NC][NT];
    auto load_w1 = [&](int n0) __attribute__((always_inline)) {
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        const int nt = wv + 8 * (n0 + n);
#pragma unroll
        for (int t = 0; t < NT; ++t)
          w1[n][t] = nt < F / 16
                         ? *reinterpret_cast<const float4*>(p.w1 + (int64_t)(16 * nt + lr) * D + 16 * t + 4 * lg)
                         : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
    };
    load_w1(0);
    // ---- attention, residual, LayerNorm1
    float g1[EPT], be1[EPT];
    load_row<EPT>(p.g1 + d0, g1);
    load_row<EPT>(p.be1 + d0, be1);
    for (int t = 16 * mt0 + r; t < T; t += 32) {  // uniform across a token's 16 lanes
      float x[EPT], h[EPT];
      load_row<EPT>(xs + t * XS + d0, x);
#pragma unroll
      for (int e = 0; e < EPT; ++e) h[e] = 0.0f;
      if (t < V) {
        const int s0 = t - t % S;  // the token's sequence
        const int jlo = max(t - p.window, s0), jhi = min(t + p.window, s0 + S - 1);
        float mx = -INFINITY, sum = 0.0f, acc[EPT];
#pragma unroll
        for (int e = 0; e < EPT; ++e) acc[e] = 0.0f;
        constexpr int kKB = 8;  // the reference window (w = 3, 7 keys) in one batch
        for (int j = jlo; j <= jhi; j += kKB) {
          float kv[kKB][EPT], s[kKB], mn = mx;
#pragma unroll
          for (int c = 0; c < kKB; ++c) load_row<EPT>(xs + min(j + c, jhi) * XS + d0, kv[c]);
#pragma unroll
          for (int c = 0; c < kKB; ++c) {
            float v = 0.0f;
#pragma unroll
            for (int e = 0; e < EPT; ++e) v = fmaf(x[e], kv[c][e], v);
            v = sum16(v) * a.scale;
            s[c] = j + c <= jhi ? v : -INFINITY;
            mn = fmaxf(mn, s[c]);
          }
          const float cf = expf(mx - mn);
          sum *= cf;
#pragma unroll
          for (int e = 0; e < EPT; ++e) acc[e] *= cf;
#pragma unroll
          for (int c = 0; c < kKB; ++c) {
            const float q = expf(s[c] - mn);  // 0 for the batch's padding
            sum += q;
#pragma unroll
            for (int e = 0; e < EPT; ++e) acc[e] = fmaf(q, kv[c][e], acc[e]);
          }
          mx = mn;
        }
        const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
#pragma unroll
        for (int e = 0; e < EPT; ++e) h[e] = x[e] + acc[e] * inv;
        layer_norm<EPT, D>(h, g1, be1, p.eps);
      }
      store_row<EPT>(hs + t * XS + d0, h);
    }
    __syncthreads();

    // linear2's first weights, in flight during linear1
    const int ct = wv % NT, kp = min(wv / NT, KS - 1);
    const bool has2 = wv < NT * KS;  // wave-uniform
    const float* w2row = p.w2 + (int64_t)(16 * ct + lr) * F + kp * (F / KS) + 4 * lg;
    float4 w2[KC];
#pragma unroll
    for (int t = 0; t < KC; ++t) w2[t] = *reinterpret_cast<const float4*>(w2row + 16 * t);

    // ---- linear1 + bias + ReLU
#pragma unroll
    for (int n0 = 0; n0 < N1; n0 += NC) {
      if (n0 > 0) load_w1(n0);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        if (m < mt0) continue;
        f32x4 acc[NC];
#pragma unroll
        for (int n = 0; n < NC; ++n) acc[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const float4 av = *reinterpret_cast<const float4*>(hs + (16 * m + lr) * XS + 16 * t + 4 * lg);
#pragma unroll
          for (int n = 0; n < NC; ++n) acc[n] = mfma_f32(av.x, w1[n][t].x, acc[n]);
#pragma unroll
          for (int n = 0; n < NC; ++n) acc[n] = mfma_f32(av.y, w1[n][t].y, acc[n]);
#pragma unroll
          for (int n = 0; n < NC; ++n) acc[n] = mfma_f32(av.z, w1[n][t].z, acc[n]);
#pragma unroll
          for (int n = 0; n < NC; ++n) acc[n] = mfma_f32(av.w, w1[n][t].w, acc[n]);
        }
#pragma unroll
        for (int n = 0; n < NC; ++n) {
          const int col = 16 * (wv + 8 * (n0 + n)) + lr;
          if (wv + 8 * (n0 + n) < F / 16) {
            const float bias = p.bi1[col];
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) zs[(16 * m + 4 * lg + jj) * ZS + col] = fmaxf(acc[n][jj] + bias, 0.0f);
          }
        }
      }
    }
    __syncthreads();

    // ---- linear2, this wave's column tile and part of the hidden units
    if (has2) {
      f32x4 acc[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int t0 = 0; t0 < K2; t0 += KC) {
        if (t0 > 0) {
#pragma unroll
          for (int t = 0; t < KC; ++t) w2[t] = *reinterpret_cast<const float4*>(w2row + 16 * (t0 + t));
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          if (m < mt0) continue;
#pragma unroll
          for (int t = 0; t < KC; ++t) {
            const float4 av = *reinterpret_cast<const float4*>(zs + (16 * m + lr) * ZS + kp * (F / KS) +
                                                               16 * (t0 + t) + 4 * lg);
            acc[m] = mfma_f32(av.x, w2[t].x, acc[m]);
            acc[m] = mfma_f32(av.y, w2[t].y, acc[m]);
            acc[m] = mfma_f32(av.z, w2[t].z, acc[m]);
            acc[m] = mfma_f32(av.w, w2[t].w, acc[m]);
          }
        }
      }
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (m >= mt0) {
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) ps[(kp * T + 16 * m + 4 * lg + jj) * XS + 16 * ct + lr] = acc[m][jj];
        }
    }
    __syncthreads();

    // ---- residual + bias, LayerNorm2
    float g2[EPT], be2[EPT], b2[EPT];
    load_row<EPT>(p.g2 + d0, g2);
    load_row<EPT>(p.be2 + d0, be2);
    load_row<EPT>(p.bi2 + d0, b2);
    for (int t = 16 * mt0 + r; t < T; t += 32) {
      float y[EPT], h[EPT];
      load_row<EPT>(ps + t * XS + d0, y);
#pragma unroll
      for (int k = 1; k < KS; ++k) {
        float q[EPT];
        load_row<EPT>(ps + (k * T + t) * XS + d0, q);
#pragma unroll
        for (int e = 0; e < EPT; ++e) y[e] += q[e];
      }
      load_row<EPT>(hs + t * XS + d0, h);
#pragma unroll
      for (int e = 0; e < EPT; ++e) y[e] = h[e] + (y[e] + b2[e]);
      layer_norm<EPT, D>(y, g2, be2, p.eps);
      store_row<EPT>(xs + t * XS + d0, y);
    }
    __syncthreads();
  }

  // ---- decoder on each sequence's last token
  for (int q = r; q * S < V; q += 32) {  // uniform across a token's 16 lanes
    float x[EPT], w[EPT], s = 0.0f;
    load_row<EPT>(xs + (q * S + S - 1) * XS + d0, x);
    load_row<EPT>(a.wd + d0, w);
#pragma unroll
    for (int e = 0; e < EPT; ++e) s = fmaf(x[e], w[e], s);
    s = sum16(s);
    if (u == 0) a.out[b0 + q] = s + a.bid[0];
  }
}

template <int D, int MT>
int launch_model(const ModelArgs& a, hipStream_t st) {
  if constexpr (MT <= ModelGeom<D>::max_tiles()) {
    constexpr size_t shm = ModelGeom<D>::lds(MT);
    auto kern = &encoder_model_kernel<D, MT>;
    if (ma_host::reserve_lds(reinterpret_cast<const void*>(kern), shm, st)) return 1;
    hipLaunchKernelGGL(kern, dim3((unsigned)((a.batch + a.per_wg - 1) / a.per_wg)), dim3(512), (uint32_t)shm, st, a);
    return 0;
  } else {
    return ma_host::set_error("ma_encoder_model_forward: sequence too long");
  }
}

// Sequences per workgroup: one until the batch passes one workgroup per CU
// (latency), then as many as keep one per CU and fit the longest tile.
template <int D>
int launch_model_d(ModelArgs a, hipStream_t st) {
  const int fit = 16 * ModelGeom<D>::max_tiles() / a.S, want = (a.batch + 255) / 256;
  a.per_wg = want < fit ? want : fit;
  switch ((a.per_wg * a.S + 15) / 16) {
    case 1: return launch_model<D, 1>(a, st);
    case 2: return launch_model<D, 2>(a, st);
    case 3: return launch_model<D, 3>(a, st);
    default: return launch_model<D, 4>(a, st);
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

bool overlaps(const void* a, const void* b, size_t bytes) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return x < y + bytes && y < x + bytes;
}

int fail(const char* fmt, long long v = 0) {
  char buf[256];
  snprintf(buf, sizeof(buf), fmt, v);
  return ma_host::set_error(buf);
}

}  // namespace

extern "C" int ma_encoder_layer_forward(const ma_encoder_layer* L, const float* src, const float* attn, float* out,
                                        void* stream) {
  ma_host::clear_error();
  if (!L) return fail("ma_encoder_layer_forward: null layer");
  const int64_t D = L->d_model;
  if (D != 16 && D != 32 && D != 64 && D != 128)
    return fail("ma_encoder_layer_forward: d_model %lld unsupported (16, 32, 64 or 128)", (long long)D);
  if (L->d_ff != 4 * D) return fail("ma_encoder_layer_forward: d_ff must be 4 * d_model (got %lld)", (long long)L->d_ff);
  if (L->batch < 0 || L->seq_len < 0) return fail("ma_encoder_layer_forward: negative batch or seq_len");
  if (L->seq_len > (int64_t)INT32_MAX) return fail("ma_encoder_layer_forward: seq_len exceeds int32 range");
  if (!(L->ln_eps > 0.0f) || std::isinf(L->ln_eps)) return fail("ma_encoder_layer_forward: ln_eps must be finite and > 0");
  const int64_t rows = L->batch * L->seq_len;
  if (rows == 0) return 0;
  const int64_t wgs = (rows + kTokens - 1) / kTokens;
  if (wgs > (int64_t)INT32_MAX) return fail("ma_encoder_layer_forward: too many tokens for one launch");
  const void* ptrs[] = {src, out, L->norm1_weight, L->norm1_bias, L->linear1_weight, L->linear1_bias,
                        L->linear2_weight, L->linear2_bias, L->norm2_weight, L->norm2_bias};
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return fail("ma_encoder_layer_forward: null or non-16-byte-aligned pointer");
  if (attn && !aligned16(attn)) return fail("ma_encoder_layer_forward: attn is not 16-byte aligned");
  const size_t bytes = (size_t)rows * (size_t)D * sizeof(float);
  if (overlaps(out, src, bytes) || (attn && overlaps(out, attn, bytes)))
    return fail("ma_encoder_layer_forward: out overlaps src or attn");
  EncArgs a;
  a.src = src;
  a.attn = attn;
  a.out = out;
  a.g1 = L->norm1_weight;
  a.be1 = L->norm1_bias;
  a.w1 = L->linear1_weight;
  a.bi1 = L->linear1_bias;
  a.w2 = L->linear2_weight;
  a.bi2 = L->linear2_bias;
  a.g2 = L->norm2_weight;
  a.be2 = L->norm2_bias;
  a.rows = rows;
  a.seq_len = (int32_t)L->seq_len;
  a.window = (int32_t)(L->window < 0 ? -1 : (L->window > L->seq_len ? L->seq_len : L->window));
  a.scale = 1.0f / std::sqrt(static_cast<float>(D));  // as src/csrc/ma_core.cpp:188 for head_dim = d_model
  a.eps = L->ln_eps;
  hipStream_t st = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  const dim3 grid((unsigned)wgs), block(256);
  switch (D) {
    case 16: hipLaunchKernelGGL(encoder_layer_kernel<16>, grid, block, 0, st, a); break;
    case 32: hipLaunchKernelGGL(encoder_layer_kernel<32>, grid, block, 0, st, a); break;
    case 64: hipLaunchKernelGGL(encoder_layer_kernel<64>, grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL(encoder_layer_kernel<128>, grid, block, 0, st, a); break;
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ma_host::set_error(hipGetErrorString(e));
  return 0;
}

extern "C" int64_t ma_encoder_model_max_seq(int64_t d_model) {
  switch (d_model) {
    case 16: return 16 * ModelGeom<16>::max_tiles();
    case 32: return 16 * ModelGeom<32>::max_tiles();
    case 64: return 16 * ModelGeom<64>::max_tiles();
    case 128: return 16 * ModelGeom<128>::max_tiles();
    default: return 0;
  }
}

extern "C" int ma_encoder_model_forward(const ma_encoder_model* M, const float* src, float* out, void* stream) {
  ma_host::clear_error();
  if (!M) return fail("ma_encoder_model_forward: null model");
  const int64_t D = M->d_model, max_seq = ma_encoder_model_max_seq(D);
  if (max_seq == 0) return fail("ma_encoder_model_forward: d_model %lld unsupported (16, 32, 64 or 128)", (long long)D);
  if (M->batch < 0 || M->batch > (1LL << 30)) return fail("ma_encoder_model_forward: bad batch");
  if (M->seq_len < 1 || M->seq_len > max_seq)
    return fail("ma_encoder_model_forward: seq_len must be in [1, %lld]", (long long)max_seq);
  if (M->input_dim < 1 || M->input_dim > (1 << 16)) return fail("ma_encoder_model_forward: bad input_dim");
  if (M->num_layers < 1 || M->num_layers > MA_ENCODER_MAX_LAYERS)
    return fail("ma_encoder_model_forward: 1 to %lld layers", (long long)MA_ENCODER_MAX_LAYERS);
  if (M->batch == 0) return 0;
  if (!M->layers || !src || !out || !M->encoder_weight || !M->decoder_bias)
    return fail("ma_encoder_model_forward: null pointer");
  const void* ptrs[] = {M->encoder_bias, M->pos, M->decoder_weight};
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return fail("ma_encoder_model_forward: null or non-16-byte-aligned pointer");
  const uintptr_t s0 = reinterpret_cast<uintptr_t>(src), o0 = reinterpret_cast<uintptr_t>(out);
  const uintptr_t sb = (uintptr_t)(M->batch * M->seq_len * M->input_dim) * sizeof(float);
  if (s0 < o0 + (uintptr_t)M->batch * sizeof(float) && o0 < s0 + sb)
    return fail("ma_encoder_model_forward: out overlaps src");
  ModelArgs a{};
  a.src = src;
  a.we = M->encoder_weight;
  a.bie = M->encoder_bias;
  a.pos = M->pos;
  a.wd = M->decoder_weight;
  a.bid = M->decoder_bias;
  a.out = out;
  a.S = (int32_t)M->seq_len;
  a.batch = (int32_t)M->batch;
  a.in = (int32_t)M->input_dim;
  a.layers = (int32_t)M->num_layers;
  a.scale = 1.0f / std::sqrt(static_cast<float>(D));  // as src/csrc/ma_core.cpp:188 for head_dim = d_model
  a.root = static_cast<float>(std::sqrt(static_cast<double>(D)));
  for (int l = 0; l < a.layers; ++l) {
    const ma_encoder_layer& L = M->layers[l];
    if (L.d_model != D || L.d_ff != 4 * D) return fail("ma_encoder_model_forward: layer %lld has another width", l);
    if (!(L.ln_eps > 0.0f) || std::isinf(L.ln_eps))
      return fail("ma_encoder_model_forward: ln_eps must be finite and > 0");
    const void* lp[] = {L.norm1_weight, L.norm1_bias, L.linear1_weight, L.linear1_bias,
                        L.linear2_weight, L.linear2_bias, L.norm2_weight, L.norm2_bias};
    for (const void* p : lp)
      if (!p || !aligned16(p)) return fail("ma_encoder_model_forward: null or non-16-byte-aligned pointer");
    a.layer[l] = ModelLayer{L.norm1_weight, L.norm1_bias, L.linear1_weight, L.linear1_bias, L.linear2_weight,
                            L.linear2_bias, L.norm2_weight, L.norm2_bias,
                            (int32_t)(L.window < 0 ? -1 : (L.window > a.S ? a.S : L.window)), L.ln_eps};
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  int rc;
  switch (D) {
    case 16: rc = launch_model_d<16>(a, st); break;
    case 32: rc = launch_model_d<32>(a, st); break;
    case 64: rc = launch_model_d<64>(a, st); break;
    default: rc = launch_model_d<128>(a, st); break;
  }
  if (rc) return rc;
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ma_host::set_error(hipGetErrorString(e));
  return 0;
}
