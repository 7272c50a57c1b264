// gfx950 kernels of the decoder's other layer steps, behind the reference's
// lab_gpu_enc_* encoders (lib/src/gpu.dart:179-312; semantics of the Metal
// layer, src/metal/lab_metal.m:321-579): RMSNorm, the per-head norm + RoPE,
// the gated short convolution, causal attention over a KV cache, the
// residual add and copy, and the control-vector steer. All fp32, HBM- or
// latency-bound; none is on the quantized linear layer's path.
//
// Reductions run as a wave butterfly (all lanes end with the total) and then
// a fixed-order sum of the waves' totals, so every result is deterministic.
// Their order differs from the Metal layer's SIMD-group sums, so results
// agree with it (and with the CPU oracle) to fp32 rounding, not bit for bit.
// Built with -ffp-contract=off: no multiply-add is fused unless written as
// fmaf.

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "f6_panel.h"
#include "dnx_kernels.h"
#include "prefill_split.h"

#include <math.h>

using namespace dnx;

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

DNX_DEV float wave_sum(float v) { return wave_sum_xor(v); }


DNX_DEV float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

// Sum over the workgroup: each wave's butterfly, then the waves' totals in
// wave order. `scratch` holds kWaves floats; every thread gets the total.
DNX_DEV float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  __syncthreads();  // scratch may still be read from a previous call
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = scratch[0];
#pragma unroll
  for (int w = 1; w < kWaves; w++) t += scratch[w];
  return t;
}

DNX_DEV float block_max(float v, float* scratch) {
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = scratch[0];
#pragma unroll
  for (int w = 1; w < kWaves; w++) t = fmaxf(t, scratch[w]);
  return t;
}

// Row-wise RMS normalisation, semantics of lab_metal.m:327-347. Each
// workgroup owns one row: its threads stride over the row for the sum of
// squares, one block-wide reduction gives the inverse root of (mean square +
// eps), and a second pass writes w[j] * (x[j] * r) with the inner product
// rounded before the weight multiplies it. The `accumulate` flag turns the
// store into out += value, which is how a norm applied after a block feeds
// the residual stream without a separate add launch.
__global__ void __launch_bounds__(kThreads)
rms_norm_kernel(const float* __restrict__ x, const float* __restrict__ w, float* out,
                int cols, float eps, int accumulate) {
  __shared__ float scratch[kWaves];
  const float* xr = x + (size_t)blockIdx.x * cols;
  float* yr = out + (size_t)blockIdx.x * cols;
  float sum = 0.0f;
  for (int j = threadIdx.x; j < cols; j += kThreads) sum += xr[j] * xr[j];
  sum = block_sum(sum, scratch);
  const float r = 1.0f / sqrtf(sum / (float)cols + eps);
  for (int j = threadIdx.x; j < cols; j += kThreads) {
    const float v = w[j] * (xr[j] * r);
    yr[j] = accumulate ? yr[j] + v : v;
  }
}

// The same RMSNorm with a row held in registers (V float4 per thread, rows
// of up to 1024 V floats, 16-byte aligned operands): every load of x, w and
// (accumulating) out is issued at the start, so the row costs one memory
// round trip instead of a dependent walk over it. The decode step's norms
// (one row of the hidden size) are latency, not bandwidth: 6.6 -> ~3 us.
//
// kAdd: the residual add before the norm in the same pass (x += m, as
// add_kernel rounds it, stored back to x, then the norm of the new x): the
// pair dnx_add + dnx_rms_norm in one launch.
// kPanel: also the fp6 GEMMs' activation panel of the normed rows (for the
// prefill matmuls that read them), as dnx_quantize_q8_f6panel would make it
// from out: the row goes through LDS (cols floats, dynamic) to four lanes
// per 32-value block (panel4_lane); row blockIdx.x is token blockIdx.x.
template <int V, bool kAdd = false, bool kPanel = false>
__global__ void __launch_bounds__(kThreads)
rms_norm_vec_kernel(const float* x_in, const float* __restrict__ w, float* out, int cols,
                    float eps, int accumulate, const float* __restrict__ m, float* x_out,
                    uint8_t* __restrict__ panel) {
  __shared__ float scratch[kWaves];
  const int q = cols / 4;
  const float4* xr = (const float4*)(x_in + (size_t)blockIdx.x * cols);
  const float4* mr = (const float4*)(m + (size_t)blockIdx.x * cols);
  float4* xw = (float4*)(x_out + (size_t)blockIdx.x * cols);
  const float4* wr = (const float4*)w;
  float4* yr = (float4*)(out + (size_t)blockIdx.x * cols);
  float4 xv[V], wv[V], ov[V], mv[V];
  const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int e = 0; e < V; e++) {
    const int i = e * kThreads + threadIdx.x;
    const bool ok = i < q;
    xv[e] = ok ? xr[i] : z;
    wv[e] = ok ? wr[i] : z;
    ov[e] = (ok && accumulate) ? yr[i] : z;
    mv[e] = (ok && kAdd) ? mr[i] : z;
  }
  if (kAdd) {
#pragma unroll
    for (int e = 0; e < V; e++) {
      const int i = e * kThreads + threadIdx.x;
      xv[e].x = xv[e].x + mv[e].x;
      xv[e].y = xv[e].y + mv[e].y;
      xv[e].z = xv[e].z + mv[e].z;
      xv[e].w = xv[e].w + mv[e].w;
      if (i < q) xw[i] = xv[e];
    }
  }
  float sum = 0.0f;
#pragma unroll
  for (int e = 0; e < V; e++) {
    sum += xv[e].x * xv[e].x;
    sum += xv[e].y * xv[e].y;
    sum += xv[e].z * xv[e].z;
    sum += xv[e].w * xv[e].w;
  }
  sum = norm_row_sum(sum, scratch);
  const float r = 1.0f / sqrtf(sum / (float)cols + eps);
#pragma unroll
  for (int e = 0; e < V; e++) {
    const int i = e * kThreads + threadIdx.x;
    if (i >= q) break;
    float4 v;
    v.x = wv[e].x * (xv[e].x * r);
    v.y = wv[e].y * (xv[e].y * r);
    v.z = wv[e].z * (xv[e].z * r);
    v.w = wv[e].w * (xv[e].w * r);
    if (accumulate) {
      v.x = ov[e].x + v.x;
      v.y = ov[e].y + v.y;
      v.z = ov[e].z + v.z;
      v.w = ov[e].w + v.w;
    }
    yr[i] = v;
    if constexpr (kPanel) {
      extern __shared__ float4 row_lds[];
      row_lds[i] = v;
    }
  }
  if constexpr (kPanel) {
    extern __shared__ float4 row_lds[];
    __syncthreads();
    const int B = cols / kBlock;
    const int tok = blockIdx.x, r = tok % kTokens;
    uint8_t* recs = panel + (size_t)(tok / kTokens) * B * kRec;
    // Whole quads of lanes (kThreads and 4 B are multiples of 4): the quad
    // reductions inside panel4_lane see their four lanes.
    for (int idx = threadIdx.x; idx < 4 * B; idx += kThreads) {
      const int j = idx & 3, b = idx >> 2;
      const float4 v0 = row_lds[b * 8 + 2 * j], v1 = row_lds[b * 8 + 2 * j + 1];
      panel4_lane(v0, v1, j, r, recs + (size_t)b * kRec);
    }
  }
}

// Per (head, token), one wave (lab_metal.m:357-380): RMSNorm over head_dim
// with weight w, then the half-split RoPE rotation pairing j with
// j + hd / 2, from the token's tables [cos(hd / 2), sin(hd / 2)]. In place;
// each lane reads its pairs before the reduction and writes only them.
//
// Two operands may share a launch (a decode step's q and k heads, one rope
// table): workgroups with blockIdx.x below heads0 take (x, x_stride, w) and
// the rest (xb, xb_stride, wb), head blockIdx.x - heads0.
// One head's RMSNorm over hd with weight w, then the half-split RoPE
// rotation pairing j with j + hd / 2 from the table row [cos(hd / 2),
// sin(hd / 2)], by one wave (lane j holds the pairs j + 64 e, e < P):
// rope_row_load requests a lane's operands, rope_row_finish computes and
// writes dst (which may be src: every lane reads its pairs before it writes
// them). Shared by head_norm_rope_kernel and the attention that folds it in,
// so both give the same bits (pairs past hd / 2 would only add +0 to the
// sum, so any P covering hd / 2 gives the same result).
template <int P>
struct RopeRow {
  float x1[P], x2[P], w1[P], w2[P], c[P], s[P];
};

template <int P>
DNX_DEV RopeRow<P> rope_row_load(const float* src, const float* __restrict__ w,
                                 const float* __restrict__ table, int hd, int lane) {
  const int pair = hd / 2;
  RopeRow<P> r;
#pragma unroll
  for (int e = 0; e < P; e++) {
    const int j = lane + 64 * e;
    const bool ok = j < pair;
    r.x1[e] = ok ? src[j] : 0.0f;
    r.x2[e] = ok ? src[j + pair] : 0.0f;
    r.w1[e] = ok ? w[j] : 0.0f;
    r.w2[e] = ok ? w[j + pair] : 0.0f;
    r.c[e] = ok ? table[j] : 0.0f;
    r.s[e] = ok ? table[pair + j] : 0.0f;
  }
  return r;
}

template <int P>
DNX_DEV void rope_row_finish(const RopeRow<P>& r, int hd, float eps, float* dst, int lane) {
  const int pair = hd / 2;
  float sum = 0.0f;
#pragma unroll
  for (int e = 0; e < P; e++) sum += r.x1[e] * r.x1[e] + r.x2[e] * r.x2[e];
  sum = wave_sum(sum);
  const float rr = 1.0f / sqrtf(sum / (float)hd + eps);
#pragma unroll
  for (int e = 0; e < P; e++) {
    const int j = lane + 64 * e;
    if (j >= pair) break;
    const float n1 = r.w1[e] * (r.x1[e] * rr), n2 = r.w2[e] * (r.x2[e] * rr);
    dst[j] = n1 * r.c[e] - n2 * r.s[e];
    dst[j + pair] = n2 * r.c[e] + n1 * r.s[e];
  }
}

DNX_DEV void head_norm_rope_row(float* x, const float* __restrict__ w,
                                const float* __restrict__ table, int hd, float eps, int lane) {
  constexpr int kPairs = 4;  // hd <= 512
  rope_row_finish<kPairs>(rope_row_load<kPairs>(x, w, table, hd, lane), hd, eps, x, lane);
}

__global__ void __launch_bounds__(64)
head_norm_rope_kernel(float* x, int x_stride, const float* __restrict__ w,
                      const float* __restrict__ rope, int rope_stride, int hd, float eps,
                      int heads0, float* xb, int xb_stride, const float* __restrict__ wb) {
  const int lane = threadIdx.x;
  const bool second = (int)blockIdx.x >= heads0;
  if (second) {
    x = xb;
    x_stride = xb_stride;
    w = wb;
  }
  const int head = second ? (int)blockIdx.x - heads0 : (int)blockIdx.x;
  float* xh = x + (size_t)blockIdx.y * x_stride + (size_t)head * hd;
  const float* table = rope + (size_t)blockIdx.y * rope_stride;
  head_norm_rope_row(xh, w, table, hd, eps, lane);
}

constexpr int kMaxConvK = 16;
constexpr int kConvCh = 64;   // channels per workgroup (one wave's lanes)
constexpr int kConvT = 16;    // tokens per workgroup tile (>= kMaxConvK - 1)

// Gated short convolution (LFM2's conv block; semantics of lab_metal.m:383-412),
// token-parallel. Per channel c the input sequence is z_j = B_j[c] * X_j[c]
// for tokens j >= 0, and the carried state for j < 0: history row k - 1 + j
// (rows oldest first). Output y_t[c] = C_t[c] * a_t with
//   a_t = w[k-1] z_t + w[k-2] z_{t-1} + ... + w[0] z_{t-k+1},
// each product rounded, summed left to right from the newest term. Afterwards
// history row r holds z_{n-k+1+r}.
//
// Workgroup (slab, tile) owns kConvCh consecutive channels and kConvT
// consecutive tokens. It stages z for its tokens and the k - 1 before them in
// LDS (one product per value, coalesced along channels), then each thread
// forms whole outputs from the staged window: no token waits on another.
// Only tile 0 reaches back into the carried state, so tile 0 alone rewrites
// it: every old row it needs is already in its LDS copy, and no other
// workgroup reads the state, so the in-place update cannot race.
__global__ void __launch_bounds__(kThreads)
conv_kernel(const float* __restrict__ bcx, const float* __restrict__ weight, float* history,
            float* __restrict__ y, int width, int k, int n) {
  __shared__ float zs[kConvT + kMaxConvK - 1][kConvCh];
  const int lane = threadIdx.x % kConvCh, part = threadIdx.x / kConvCh;
  constexpr int kParts = kThreads / kConvCh;
  const int c = blockIdx.x * kConvCh + lane;
  const bool live = c < width;
  const int t0 = blockIdx.y * kConvT;
  const int tn = min(kConvT, n - t0);
  const int span = tn + k - 1;  // staged rows: tokens t0 - (k - 1) .. t0 + tn - 1
  const size_t row3 = (size_t)3 * width;

  constexpr int kStageIters = (kConvT + kMaxConvK - 1 + kParts - 1) / kParts;
#pragma unroll
  for (int m = 0; m < kStageIters; m++) {  // all loads of a thread in flight together
    const int i = part + m * kParts;
    if (i < span) {
      const int j = t0 - (k - 1) + i;
      float z = 0.0f;
      if (live) {
        z = j >= 0 ? bcx[(size_t)j * row3 + c] * bcx[(size_t)j * row3 + 2 * (size_t)width + c]
                   : history[(size_t)(k - 1 + j) * width + c];
      }
      zs[i][lane] = z;
    }
  }
  __syncthreads();
  if (!live) return;

  // Taps by lag: wl[s] weights z_{t-s} (register indices stay constant).
  float wl[kMaxConvK];
#pragma unroll
  for (int s = 0; s < kMaxConvK; s++) wl[s] = s < k ? weight[(size_t)c * k + (k - 1 - s)] : 0.0f;
#pragma unroll
  for (int m = 0; m < kConvT / kParts; m++) {
    const int i = part + m * kParts;
    if (i >= tn) break;
    const int t = t0 + i;
    // Row of z_t in the staged window is i + k - 1; z_{t-s} sits s rows up.
    float a = wl[0] * zs[i + k - 1][lane];
#pragma unroll
    for (int s = 1; s < kMaxConvK; s++) {
      if (s < k) a += wl[s] * zs[i + k - 1 - s][lane];
    }
    y[(size_t)t * width + c] = bcx[(size_t)t * row3 + width + c] * a;
  }

  if (blockIdx.y == 0) {
    // New state row r = z_{n-k+1+r}: from the staged window when that token
    // is in it (or is an old state row), else a product of the last tokens.
    for (int r = part; r + 1 < k; r += kParts) {
      const int j = n - (k - 1) + r;
      float z;
      if (j < tn) {
        z = zs[j + k - 1][lane];
      } else {
        z = bcx[(size_t)j * row3 + c] * bcx[(size_t)j * row3 + 2 * (size_t)width + c];
      }
      history[(size_t)r * width + c] = z;
    }
  }
}

// Causal attention of n tokens at positions position.. over their cached
// keys and values (lab_metal.m:414-521), one workgroup per (head, token):
// scores q.k / sqrt(hd) against the keys the token may see (window 0:
// every earlier position; else the last `window`, its own included), a
// softmax, the weighted sum of values, and the per-head output gate
// sigmoid(gate) when `gate` is not null. GQA: query head h reads KV head
// h / (heads / kv_heads). Scores live in LDS (dynamic, sized by the launch
// for the last token's keys). Each thread takes whole keys for the dots
// (one key row per lane: 16-byte loads), and the value sum splits the keys
// over 256 / hd thread groups added in group order.
__global__ void __launch_bounds__(kThreads)
attention_kernel(const float* __restrict__ q, const float* __restrict__ keys,
                 const float* __restrict__ values, const float* __restrict__ gate,
                 float* __restrict__ out, int position, int heads, int kv_dim, int group,
                 int hd, int window, float scale) {
  extern __shared__ __align__(16) float lds[];
  __shared__ float scratch[kWaves];
  const int head = blockIdx.x, token = blockIdx.y, tid = threadIdx.x;
  const int pos = position + token;
  const int start = window > 0 && pos >= window ? pos - window + 1 : 0;
  const int count = pos - start + 1;
  const size_t qo = ((size_t)token * heads + head) * hd;
  const int kvo = head / group * hd;
  float* qs = lds;                      // [hd]
  float* scores = lds + hd;             // [count]
  float* part = scores + ((count + 3) & ~3);   // [groups][hd] value partials
  for (int d = tid; d < hd; d += kThreads) qs[d] = q[qo + d];
  __syncthreads();

  const int hd4 = hd / 4;
  for (int i = tid; i < count; i += kThreads) {
    const float4* k4 = (const float4*)(keys + (size_t)(start + i) * kv_dim + kvo);
    float d = 0.0f;
    for (int c = 0; c < hd4; c++) {
      const float4 kc = k4[c];
      const float4 qc = *(const float4*)(qs + 4 * c);
      d += qc.x * kc.x + qc.y * kc.y + qc.z * kc.z + qc.w * kc.w;
    }
    scores[i] = d * scale;
  }
  __syncthreads();
  float m = -INFINITY;
  for (int i = tid; i < count; i += kThreads) m = fmaxf(m, scores[i]);
  m = block_max(m, scratch);
  float sum = 0.0f;
  for (int i = tid; i < count; i += kThreads) {
    const float e = expf(scores[i] - m);
    scores[i] = e;
    sum += e;
  }
  sum = block_sum(sum, scratch);  // its barriers also publish the exponentials
  const int groups = kThreads / hd;  // >= 1: hd <= 256
  const int gi = tid / hd, d = tid - gi * hd;
  if (gi < groups) {
    const float* v = values + (size_t)start * kv_dim + kvo + d;
    float acc = 0.0f;
    int i = gi;
    for (; i + 3 * groups < count; i += 4 * groups) {  // 4 keys' loads together
      const float v0 = v[(size_t)i * kv_dim], v1 = v[(size_t)(i + groups) * kv_dim];
      const float v2 = v[(size_t)(i + 2 * groups) * kv_dim];
      const float v3 = v[(size_t)(i + 3 * groups) * kv_dim];
      acc += scores[i] * v0;
      acc += scores[i + groups] * v1;
      acc += scores[i + 2 * groups] * v2;
      acc += scores[i + 3 * groups] * v3;
    }
    for (; i < count; i += groups) acc += scores[i] * v[(size_t)i * kv_dim];
    part[gi * hd + d] = acc;
  }
  __syncthreads();
  if (gi == 0) {
    float acc = part[d];
    for (int g2 = 1; g2 < groups; g2++) acc += part[g2 * hd + d];
    if (gate != nullptr) {
      const float g = 1.0f / (1.0f + expf(-gate[(size_t)token * heads + head]));
      out[qo + d] = (acc / sum) * g;
    } else {
      out[qo + d] = acc / sum;
    }
  }
}

// Long contexts with few (head, token) pairs (decode) split the keys: each
// workgroup of attention_split_kernel takes split_keys(hd) keys of one
// token for G query heads that share one KV head, and writes for each head
// its max m, its exponentials' sum l (relative to m) and its unnormalised
// value sums o[hd] (a row of hd + 4 floats: m, l, two unused, o, so o is
// 16-byte aligned); attention_combine_kernel rescales the splits to their
// common max and adds them in split order (deterministic):
// O = sum_s o_s e^(m_s - M) / sum_s l_s e^(m_s - M). The same softmax as
// attention_kernel, summed in another order.
// A split puts hd / 4 lanes on a key row (one 16-byte piece each,
// coalesced), 256 / (hd / 4) keys per workgroup step, and kSplitSteps
// steps: every key and value load of the split is issued at its start, so
// it waits for memory once, and each row is read once for the G heads
// (GQA). Eight steps (64 keys at hd 128: 512 workgroups at 4096 positions
// of 8 KV heads) read faster than 16 with half the workgroups (Qwen3-1.7B
// at position 4095: 9.0 against 11.0 us; a pure read of the same bytes in
// the two patterns: 7.2 against 8.1-9.5 us).
// Dots end in a butterfly over the key's lanes; wave w takes the softmax
// statistics of heads w, w + 4, ...; value sums go to per-lane float4
// partials added in a fixed order.
constexpr int kSplitSteps = 8;
constexpr int kSplitMaxKeys = 256;

int split_keys(int hd) {
  const int step = kThreads / (hd / 4);   // keys per workgroup step
  const int k = kSplitSteps * step;
  return k < kSplitMaxKeys ? k : kSplitMaxKeys;
}

// Sum over aligned groups of LT lanes (a power of two up to 32); every lane
// of a group gets the group's sum. DPP moves up to 16 lanes (no LDS round
// trip), a swizzle for 32.
template <int LT>
DNX_DEV float group_sum(float v) {
  if constexpr (LT >= 2) v += dppf<kQuadXor1>(v);
  if constexpr (LT >= 4) v += dppf<kQuadXor2>(v);
  if constexpr (LT >= 8) v += dppf<kHalfRowMirror>(v);
  if constexpr (LT >= 16) v += dppf<kRowMirror>(v);
  if constexpr (LT >= 32) v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401F));
  static_assert(LT <= 32, "group_sum: at most 32 lanes");
  return v;
}

// G query heads per workgroup; LT lanes per key when fixed at compile time
// (hd = 4 * LT), 0 for any hd.
// The q and k head norms + RoPE of a decode step folded into its attention
// (one token): the table row of the token, the two norm weights, eps, and
// the cache's keys (written: the new key row, normed in place).
struct RopeArgs {
  const float* table;
  const float* qw;
  const float* kw;
  float* keys;
  float eps;
};
constexpr int kRopeMaxHd = 256;

template <int G, int LT, int STEPS = kSplitSteps, bool kRope = false>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 2)))
attention_split_kernel(const float* __restrict__ q, const float* keys,
                       const float* __restrict__ values, float* __restrict__ ws, int position,
                       int heads, int kv_dim, int group, int hd, int window, float scale,
                       int splits, int keys_per_split, RopeArgs rp) {
  __shared__ float scores[G][kSplitMaxKeys];
  __shared__ float4 part[G][kThreads];
  __shared__ float stat[G][2];
  const int h0 = blockIdx.x * G, token = blockIdx.y, split = blockIdx.z, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int pos = position + token;
  const int start = window > 0 && pos >= window ? pos - window + 1 : 0;
  const int count = pos - start + 1;
  const int k0 = split * keys_per_split;
  const int nk = max(0, min(keys_per_split, count - k0));   // this split's keys
  const int kvo = h0 / group * hd;
  const int L = LT > 0 ? LT : hd / 4;                      // lanes per key
  const int per = 64 / L, step = kWaves * per;               // keys per wave, per step
  const int c = lane % L, kb = wave * per + lane / L;       // this lane's first key
  float4 qr[G];
  if constexpr (!kRope) {
#pragma unroll
    for (int g = 0; g < G; g++)
      qr[g] = *(const float4*)(q + ((size_t)token * heads + h0 + g) * hd + 4 * c);
  }
  // Resources over this split's nk key rows: a row past them lies wholly
  // beyond the range (its offset is at least nk rows) and reads zeros.
  const size_t first = (size_t)(start + k0) * kv_dim + kvo;
  const uint32_t range = (uint32_t)nk * (uint32_t)kv_dim * 4u;
  const i32x4 krs = buffer_rsrc(keys + first, range);
  const i32x4 vrs = buffer_rsrc(values + first, range);
  const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  // Folded head norms (one token): wave w norms and rotates q heads h0 + w,
  // h0 + w + 4, ..., and in the split that holds the token's own key, the
  // wave after the last q head its key row (as stored). Their operands are
  // requested before the keys and values, which return in order after them.
  const int cur = count - 1 - k0;                // the token's key within the split
  const bool has_cur = kRope && cur >= 0 && cur < nk;
  constexpr int kRP = kRopeMaxHd / 128;          // pairs per lane
  constexpr int kRows = kRope ? (G + kWaves) / kWaves : 1;
  RopeRow<kRP> rrow[kRows];
  float dcur[G];  // the token's own key's dots (folded norms)
  if constexpr (kRope) {
#pragma unroll
    for (int r = 0; r < kRows; r++) {
      // Rows a wave does not norm load q's first head (always valid), unused.
      const int g = wave + r * kWaves;
      const bool is_k = g == G && has_cur;
      const float* src = g < G ? q + ((size_t)h0 + g) * hd
                         : is_k ? keys + (size_t)pos * kv_dim + kvo : q + (size_t)h0 * hd;
      rrow[r] = rope_row_load<kRP>(src, is_k ? rp.kw : rp.qw, rp.table, hd, lane);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  float4 kv[STEPS], vv[STEPS];
#pragma unroll
  for (int j = 0; j < STEPS; j++)
    kv[j] = buffer_load_f4(krs, (kb + j * step) * kv_dim * 4 + 16 * c);
#pragma unroll
  for (int j = 0; j < STEPS; j++)
    vv[j] = buffer_load_f4(vrs, (kb + j * step) * kv_dim * 4 + 16 * c);
  // The folded norms' results go through LDS to the lanes that need them;
  // the keys and values are in flight meanwhile.
  if constexpr (kRope) {
    __shared__ float qn[G][kRopeMaxHd];
    __shared__ float kn[kRopeMaxHd];
#pragma unroll
    for (int r = 0; r < kRows; r++) {
      const int g = wave + r * kWaves;
      if (g < G) {
        rope_row_finish<kRP>(rrow[r], hd, rp.eps, qn[g], lane);
      } else if (g == G && has_cur) {
        rope_row_finish<kRP>(rrow[r], hd, rp.eps, kn, lane);
      }
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; g++) qr[g] = *(const float4*)(qn[g] + 4 * c);
    if (has_cur) {
      // The token's own key scores against its normed row (every key group
      // holds all dims, so every lane computes the same dot, reduced as the
      // other keys' dots are); its loaded copy is not used.
      const float4 k4 = *(const float4*)(kn + 4 * c);
#pragma unroll
      for (int g = 0; g < G; g++) {
        float d = qr[g].x * k4.x + qr[g].y * k4.y + qr[g].z * k4.z + qr[g].w * k4.w;
        if constexpr (LT > 0) {
          d = group_sum<LT>(d);
        } else {
          for (int o = L / 2; o > 0; o >>= 1) d += __shfl_xor(d, o);
        }
        dcur[g] = d;
      }
      // The normed key row back into the cache (only this workgroup reads it).
      if (tid < hd / 4) {
        *(float4*)(rp.keys + (size_t)pos * kv_dim + kvo + 4 * tid) = *(const float4*)(kn + 4 * tid);
      }
    }
  }
  // Dots in batches of kBatch steps x G heads: each butterfly stage issues
  // the batch's lane exchanges together and waits once (L is a run-time
  // count, so per-dot loops would wait on every exchange).
  constexpr int kBatch = 4;
#pragma unroll
  for (int j0 = 0; j0 < STEPS; j0 += kBatch) {
    float d[kBatch][G];
#pragma unroll
    for (int u = 0; u < kBatch; u++)
#pragma unroll
      for (int g = 0; g < G; g++) {
        const float4 k4 = kv[j0 + u];
        d[u][g] = qr[g].x * k4.x + qr[g].y * k4.y + qr[g].z * k4.z + qr[g].w * k4.w;
      }
    if constexpr (LT > 0) {
#pragma unroll
      for (int u = 0; u < kBatch; u++)
#pragma unroll
        for (int g = 0; g < G; g++) d[u][g] = group_sum<LT>(d[u][g]);
    } else {
      for (int o = L / 2; o > 0; o >>= 1) {
#pragma unroll
        for (int u = 0; u < kBatch; u++)
#pragma unroll
          for (int g = 0; g < G; g++) d[u][g] += __shfl_xor(d[u][g], o);
      }
    }
#pragma unroll
    for (int u = 0; u < kBatch; u++) {
      const int i = kb + (j0 + u) * step;
      if (i < nk && c == 0) {
#pragma unroll
        for (int g = 0; g < G; g++) scores[g][i] = (has_cur && i == cur ? dcur[g] : d[u][g]) * scale;
      }
    }
  }
  __syncthreads();
  for (int g = wave; g < G; g += kWaves) {  // one wave per head: no block barrier
    constexpr int kPerLane = kSplitMaxKeys / 64;
    float v[kPerLane];
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < kPerLane; u++) {
      const int i = u * 64 + lane;
      v[u] = i < nk ? scores[g][i] : -INFINITY;
      mx = fmaxf(mx, v[u]);
    }
    mx = wave_max_dpp(mx);
    float sum = 0.0f;
#pragma unroll
    for (int u = 0; u < kPerLane; u++) {
      const int i = u * 64 + lane;
      if (i < nk) {
        const float e = expf(v[u] - mx);
        scores[g][i] = e;
        sum += e;
      }
    }
    sum = wave_sum_dpp(sum);
    if (lane == 0) {
      stat[g][0] = mx;   // -inf for a split past the token's keys (l = 0, o = 0)
      stat[g][1] = sum;
    }
  }
  __syncthreads();
  float4 acc[G];
#pragma unroll
  for (int g = 0; g < G; g++) acc[g] = zero;
#pragma unroll
  for (int j = 0; j < STEPS; j++) {
    const int i = kb + j * step;
#pragma unroll
    for (int g = 0; g < G; g++) {
      const float p = i < nk ? scores[g][i] : 0.0f;
      acc[g].x += p * vv[j].x;
      acc[g].y += p * vv[j].y;
      acc[g].z += p * vv[j].z;
      acc[g].w += p * vv[j].w;
    }
  }
#pragma unroll
  for (int g = 0; g < G; g++) part[g][tid] = acc[g];
  __syncthreads();
  for (int e = tid; e < G * L; e += kThreads) {
    // Head g, dimensions 4cc..4cc+3: the (wave, key-in-step) partials in order.
    const int g = e / L, cc = e - g * L;
    float4 t = zero;
    for (int w = 0; w < kWaves; w++)
      for (int s2 = 0; s2 < per; s2++) {
        const float4 p4 = part[g][w * 64 + s2 * L + cc];
        t.x += p4.x;
        t.y += p4.y;
        t.z += p4.z;
        t.w += p4.w;
      }
    float* out = ws + (((size_t)token * heads + h0 + g) * splits + split) * (hd + 4);
    *(float4*)(out + 4 + 4 * cc) = t;
    if (cc == 0) {
      out[0] = stat[g][0];
      out[1] = stat[g][1];
    }
  }
}

template <int G, bool kRope = false>
void launch_split(dim3 grid, hipStream_t stream, const float* q, const float* keys,
                  const float* values, float* ws, int position, int heads, int kv_dim, int group,
                  int hd, int window, float scale, int splits, int kps, RopeArgs rp = {}) {
  auto kernel = hd == 128 ? attention_split_kernel<G, 32, kSplitSteps, kRope>
              : hd == 64  ? attention_split_kernel<G, 16, kSplitSteps, kRope>
                          : attention_split_kernel<G, 0, kSplitSteps, kRope>;
  hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, q, keys, values, ws, position,
                     heads, kv_dim, group, hd, window, scale, splits, kps, rp);
}

// The splits of one (head, token). Thread t takes dimension t % hd of the
// splits s = t / hd + P j (P = 256 / hd threads per dimension). Its first
// kChunk value loads and the split statistics are issued together, so a
// short context waits for memory once; the rescaling factors e^(m_s - M)
// go through LDS (dynamic: `splits` floats), and the P partial sums of a
// dimension are added in a fixed order.
// More than 64 splits: each thread takes splits s0, s0 + 256, ...; the max
// and l over the workgroup (the block reductions' barriers also publish fs).
DNX_DEV float combine_stats(const float* w, int splits, int row, int s0, float m0, float l0,
                            float* fs, float* scratch) {
  float mx = s0 < splits ? m0 : -INFINITY;
  for (int s = s0 + kThreads; s < splits; s += kThreads) mx = fmaxf(mx, w[(size_t)s * row]);
  mx = block_max(mx, scratch);
  float lp = 0.0f;
  if (s0 < splits) {
    const float f = m0 != -INFINITY ? expf(m0 - mx) : 0.0f;
    fs[s0] = f;
    lp = l0 * f;
  }
  for (int s = s0 + kThreads; s < splits; s += kThreads) {
    const float ms = w[(size_t)s * row];
    const float f = ms != -INFINITY ? expf(ms - mx) : 0.0f;
    fs[s] = f;
    lp += w[(size_t)s * row + 1] * f;
  }
  return block_sum(lp, scratch);
}

template <bool kRope = false>
__global__ void __launch_bounds__(kThreads)
attention_combine_kernel(const float* __restrict__ ws, const float* __restrict__ gate,
                         float* __restrict__ out, int heads, int hd, int splits,
                         float* qio = nullptr, RopeArgs rp = {}) {
  extern __shared__ float fs[];   // [splits] e^(m_s - M), 0 for empty splits
  __shared__ float scratch[kWaves];
  __shared__ float red[kThreads];
  constexpr int kChunk = 32;
  const int head = blockIdx.x, token = blockIdx.y, tid = threadIdx.x;
  const int row = hd + 4;
  const float* w = ws + ((size_t)token * heads + head) * splits * row;
  // Every offset past the (head, token)'s rows reads zero.
  const i32x4 rs = buffer_rsrc(w, (uint32_t)splits * (uint32_t)row * 4u);
  const int P = kThreads / hd, d = tid % hd, part = tid / hd;
  float v[kChunk];
#pragma unroll
  for (int u = 0; u < kChunk; u++) {
    const int sp = part + u * P;
    v[u] = __int_as_float(dnx_raw_buffer_load_i32(rs, (sp * row + 4 + d) * 4, 0, 0));
  }
  const int s0 = tid;   // the first split whose statistics this thread reads
  const float m0 = __int_as_float(dnx_raw_buffer_load_i32(rs, s0 * row * 4, 0, 0));
  const float l0 = __int_as_float(dnx_raw_buffer_load_i32(rs, (s0 * row + 1) * 4, 0, 0));
  if constexpr (kRope) {
    // The folded q norm of this head, in place (one token): the split
    // kernel normed its own copies; every split has finished reading q.
    // Wave 1, while wave 0 reduces the split statistics.
    if (tid >= 64 && tid < 128) {
      head_norm_rope_row(qio + (size_t)head * hd, rp.qw, rp.table, hd, rp.eps, tid - 64);
    }
  }
  float l;
  if (splits <= 64) {
    // One wave holds every split's statistics (lane s): the max, the
    // factors and l without a block reduction; one barrier publishes them.
    if (tid < 64) {
      const bool live = s0 < splits;
      const float m = live ? m0 : -INFINITY;
      const float mx = wave_max_dpp(m);
      const float f = live && m != -INFINITY ? expf(m - mx) : 0.0f;
      if (live) fs[s0] = f;
      const float lsum = wave_sum_dpp(live ? l0 * f : 0.0f);
      if (tid == 0) scratch[0] = lsum;
    }
    __syncthreads();
    l = scratch[0];
  } else {
    l = combine_stats(w, splits, row, s0, m0, l0, fs, scratch);
  }
  float acc = 0.0f;
#pragma unroll
  for (int u = 0; u < kChunk; u++) {
    const int sp = part + u * P;
    if (sp < splits) acc += v[u] * fs[sp];
  }
  for (int sp = part + kChunk * P; sp < splits; sp += P) acc += w[(size_t)sp * row + 4 + d] * fs[sp];
  red[tid] = acc;
  __syncthreads();
  if (part == 0) {
    float t = red[d];
    for (int p2 = 1; p2 < P; p2++) t += red[p2 * hd + d];
    const size_t qo = ((size_t)token * heads + head) * hd;
    const float g =
        gate != nullptr ? 1.0f / (1.0f + expf(-gate[(size_t)token * heads + head])) : 1.0f;
    out[qo + d] = gate != nullptr ? (t / l) * g : t / l;
  }
}

// Attention of many tokens (prefill) on the bf16 matrix cores, float32 in and
// out. A float32 operand of 2^-110 or more is the exact sum of three bf16
// pieces (8 significant bits each; below that the last piece is a bf16
// subnormal or lost: 2e-7 of the operand at 2^-112, 2e-3 at 2^-125); of the
// nine piece products of a q.k or p.v term the six with i + j <= 2 are formed,
// the others lie below 2^-26 of the term, and the sums are float32. Six bf16 MFMAs cost less than half of the float32
// ones they replace (v_mfma_f32_16x16x4f32: 32 multiply-adds a clock and
// SIMD, 16x16x32_bf16: 512).
//
// A wave takes 16 queries of one head, a workgroup 4 waves sharing one KV
// head (GW heads of a GQA group x 4 / GW query blocks); it walks its keys in
// tiles of KT, split into their pieces once per workgroup on the way into
// LDS (the next tile's values are in registers meanwhile). Per tile and wave:
// * S^T = K Q^T: A = 16 keys x 32 dims (LDS), B = 32 dims x 16 queries (the
//   pieces of Q, held in registers); lane l ends with the scores of query
//   l % 16 for keys 4 (l / 16) + 0..3 of each 16, so the online softmax
//   needs two lane exchanges for the max and two for the sum;
// * O^T += V^T P^T: the lane's probabilities, split in registers, are the B
//   operand as they are if k slot j of lane group g stands for key 4 g + j
//   (j < 4) or 16 + 4 g + j - 4; V^T is staged in that order.
// A tile's products start from zero and join the running sums in one
// multiply-add, so a long run rounds once a tile; within a tile the products
// of first pieces have a sum of their own (mfma_pieces). Error against 64
// bits, relative 2-norm, with the float32 MFMAs -> so: 64 tokens after 256
// (16 / 8 heads, hd 128) 2.8e-7 -> 1.7e-7 (3.0e-7 with all six products in one
// sum), 512 from 0 (32 / 8) 2.5e-7 -> 1.2e-7, 1000 after 1000 (16 / 8) 6.0e-7
// -> 2.1e-7, 8 after 4000 (8 / 2, hd 64) 3.0e-7 -> 2.3e-7.
// A wave whose queries see no key of a tile skips it; only tiles at the edge
// of the causal or window range are masked.
//
// An infinity or NaN has no pieces (nor has a float that rounds to an infinity
// as bf16), and finite terms may overflow with either sign: what they meet
// comes out as NaN. A wave that ends with an infinity or NaN in its sums forms
// them anew from memory (prefill_special).
//
// With `splits` > 1 a workgroup takes a run of tiles_per_split tiles and
// writes per (token, head) the partial (m, l, o) rows that
// attention_combine_rows_kernel adds; one whose run lies past its queries'
// keys writes nothing (live_splits). Otherwise it writes the output, gated.
// m is in units of log2: exponentials use the hardware exp2 of a fused
// multiply-add, one rounding before it.
//
// What bounds it: at prompt chunks the latency of one pass (launch, first
// loads, splitting, two barriers: at hd 128 6.6 us with one tile, 2.3 us for
// each more), at long prompts the MFMAs (six times the product's 2 flops, 215
// of 400 us at the 1.6 PFLOP/s a large bf16 product reaches) and the splitting
// and softmax they do not cover. Measured with the combine (us, graph-timed,
// against the float32 MFMAs; heads / KV heads, hd): 64 tokens after 256,
// 16 / 8, 128: 15.0 -> 12.2; 37 after 500, 8 / 8, 64: 11.6 -> 8.6; 512 from
// 0, 32 / 8, 128: 41.7 -> 33.6; 1000 after 1000, 16 / 8, 128: 170 -> 99;
// 1024 after 4000, 8 / 4, 64: 119 -> 78. 32 queries a wave (32x32x16 MFMAs,
// half the LDS reads) gained 8% on the longest but needed 256 registers, and
// was 4 us slower with one tile.
constexpr int kPQ = 16;   // queries per wave

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

template <int HD, int KT_>
struct PrefillTile {
  static constexpr int KT = KT_;                // keys per tile: 32 or 64
  static constexpr int KS = KT * 16 + 16;       // K: one 8-dim group of all keys, + pad
  static constexpr int VS = HD * 16;            // V^T: 8 keys of all dims
  static constexpr int kK = 3 * (HD / 8) * KS;  // [piece][dim group][key][16 B]
  static constexpr int kV = 3 * (KT / 8) * VS;  // [piece][key group][dim][16 B]
};

// The tiles of a workgroup's queries (tokens first .. last): the range of
// its keys, and how many splits of tps tiles they fill.
struct KeyRange {
  int start, end;
};
DNX_DEV KeyRange key_range(int position, int first, int last, int window) {
  return {window > 0 ? max(0, position + first - window + 1) : 0, position + last + 1};
}
DNX_DEV int live_splits(KeyRange r, int kt, int tps) {
  return ((r.end - r.start + kt - 1) / kt + tps - 1) / tps;
}

// Max / sum over lanes i, i ^ 16, i ^ 32 and i ^ 48 (lane i % 16 of the four
// 16-lane rows), every lane getting the result, on gfx950's VALU lane swaps:
// with both operands v, permlane16_swap pairs each lane with lane ^ 16 and
// permlane32_swap with lane ^ 32. No LDS round trip.
DNX_DEV float rows4_max(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

DNX_DEV float rows4_sum(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Eight floats as three bf16 fragments (piece i of value j in element j),
// each piece the rest rounded to nearest: the terms that are not formed are
// then as often too small as too large. An infinity, a NaN and a float that
// rounds to an infinity have NaN among their pieces.
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
DNX_DEV void split_pieces(const float* x, uint4* p) {
  uint32_t w[3][4];
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    f32x2 v = {x[j], x[j + 1]};
#pragma unroll
    for (int i = 0; i < 3; i++) {
      w[i][j / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf2));
      if (i == 2) break;
      v.x -= __uint_as_float(w[i][j / 2] << 16);
      v.y -= __uint_as_float(w[i][j / 2] & 0xffff0000u);
    }
  }
#pragma unroll
  for (int i = 0; i < 3; i++) p[i] = make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]);
}

// big += A0 B0 and low += the five other piece products, the smallest first.
// Each product rounds its sum: low rounds at 2^-8 of big or less, where all
// six in one sum rounded it six times a step at its full size.
DNX_DEV void mfma_pieces(const uint4* a, const uint4* b, v4f& big, v4f& low) {
  auto product = [&](int i, int j, v4f acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a[i]),
                                                   __builtin_bit_cast(bf8, b[j]), acc, 0, 0, 0);
  };
  big = product(0, 0, big);
  low = product(2, 0, low);
  low = product(1, 1, low);
  low = product(0, 2, low);
  low = product(1, 0, low);
  low = product(0, 1, low);
}

// The sums (m, l, o) of a wave's 16 queries over keys k_lo .. k_hi - 1 where
// an operand has no pieces: the same products on the float32 matrix cores,
// straight from memory, in the layout of the kernel below (see_lo and see_n:
// the keys that the lane's query sees). Hidden keys count for nothing,
// whatever they hold: an infinity or NaN among the values is zero in the
// products, and a code for it (1: +inf, 128: -inf, 129: NaN) is summed over
// the keys that are seen, times 1 where p > 0 and 2^14 where p is zero (zero
// times an infinity is NaN; 32 codes stay below 2^14). Once every sum l is
// NaN, so is every output, and the rest of the keys is left out.
//
// One wave alone walks its keys, so a step's latency is what it costs: 32
// keys a step in two chains, the next step's keys and this step's values
// requested before the scores are formed (1000 tokens after 1000, 16 / 8
// heads, hd 128, us; the finite call takes 116: one infinity among the values
// 202, 236 with 16 keys a step and nothing ahead, and 4270 as a query at a time
// in plain loads; every value infinite 371, 424 and 7060; a NaN among the keys
// 115 to 145, every operand NaN 124. The float32 matrix cores alone, with the
// keys shared in LDS, took 170 to 180 whatever the values).
template <int HD>
DNX_DEV void prefill_special(const float* qp, const float* keys, const float* values, int kv_dim,
                             float sl, int k_lo, int k_hi, uint32_t see_lo, uint32_t see_n,
                             int lane, float& m, float& l, v4f* o) {
  constexpr int NE = HD / 16, ND = HD / 16, NU = 2;   // NU times 16 keys a step
  const int l16 = lane & 15, g4 = lane >> 4;
  m = -INFINITY;
  l = 0.0f;
#pragma unroll
  for (int e = 0; e < NE; e++) o[e] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  float4 qr[ND], kr[NU][ND];
#pragma unroll
  for (int d = 0; d < ND; d++) qr[d] = *(const float4*)(qp + 16 * d + 4 * g4);
  auto load_keys = [&](int k0) {   // those past the last: the last
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const float* kp = keys + (size_t)min(k0 + 16 * u + l16, k_hi - 1) * kv_dim + 4 * g4;
#pragma unroll
      for (int d = 0; d < ND; d++) kr[u][d] = *(const float4*)(kp + 16 * d);
    }
  };
  if (k_lo < k_hi) load_keys(k_lo);
#pragma unroll 1
  for (int k0 = k_lo; k0 < k_hi; k0 += 16 * NU) {
    float x[NU][NE][4];
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const float* vp = values + (size_t)min(k0 + 16 * u + 4 * g4 + v, k_hi - 1) * kv_dim + l16;
#pragma unroll
        for (int e = 0; e < NE; e++) x[u][e][v] = vp[16 * e];
      }
    v4f s[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) s[u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
      for (int c = 0; c < 4; c++)
#pragma unroll
        for (int u = 0; u < NU; u++)
          s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32((&kr[u][d].x)[c], (&qr[d].x)[c], s[u], 0, 0, 0);
    if (k0 + 16 * NU < k_hi) load_keys(k0 + 16 * NU);
    float mt = -INFINITY, weight[NU][4];
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const uint32_t key = k0 + 16 * u + 4 * g4 + v;
        weight[u][v] = (int)key < k_hi && key - see_lo < see_n ? 1.0f : 0.0f;
        if (weight[u][v] == 0.0f) s[u][v] = -INFINITY;
        mt = fmaxf(mt, s[u][v]);
      }
    const float m_new = fmaxf(m, rows4_max(mt) * sl), ref = m_new == -INFINITY ? 0.0f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m - ref);
    float ps = 0.0f;
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        s[u][v] = __builtin_amdgcn_exp2f(fmaf(s[u][v], sl, -ref));
        ps += s[u][v];
        if (s[u][v] == 0.0f) weight[u][v] *= 16384.0f;
      }
    l = l * alpha + rows4_sum(ps);
    m = m_new;
    if (!__any(l == l)) return;
#pragma unroll
    for (int e = 0; e < NE; e++) {
      bool finite = true;
#pragma unroll
      for (int u = 0; u < NU; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) finite &= fabsf(x[u][e][v]) < INFINITY;
      v4f d = {0.0f, 0.0f, 0.0f, 0.0f};
      if (__any(!finite)) {
        v4f codes = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
          for (int v = 0; v < 4; v++) {
            const float xv = x[u][e][v];
            const float code = xv == INFINITY ? 1.0f : xv == -INFINITY ? 128.0f
                               : xv != xv ? 129.0f : 0.0f;
            codes = __builtin_amdgcn_mfma_f32_16x16x4f32(code, weight[u][v], codes, 0, 0, 0);
            x[u][e][v] = code == 0.0f ? xv : 0.0f;
          }
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const float minus = floorf(codes[v] * (1.0f / 128.0f));
          const float up = codes[v] - 128.0f * minus > 0.0f ? INFINITY : 0.0f;
          const float down = minus > 0.0f ? INFINITY : 0.0f;
          d[v] = codes[v] >= 16384.0f ? NAN : up - down;
        }
      }
#pragma unroll
      for (int u = 0; u < NU; u++)
#pragma unroll
        for (int v = 0; v < 4; v++)
          d = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u][e][v], s[u][v], d, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 4; v++) o[e][v] = fmaf(o[e][v], alpha, d[v]);
    }
  }
}

template <int HD, int GW, int KT_>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 3)))
attention_prefill_kernel(const float* __restrict__ q, const float* __restrict__ keys,
                         const float* __restrict__ values, const float* __restrict__ gate,
                         float* __restrict__ out, float* __restrict__ ws, int position, int n,
                         int heads, int kv_dim, int group, int window, float scale, int splits,
                         int tiles_per_split) {
  using T = PrefillTile<HD, KT_>;
  constexpr int KT = T::KT, NS = KT / 16, NE = HD / 16;
  constexpr int QW = 4 / GW;                     // query blocks of a workgroup
  __shared__ __align__(16) uint8_t lds[T::kK + T::kV];
  uint8_t* Kp = lds;
  uint8_t* Vp = lds + T::kK;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g4 = lane >> 4;
  const int head = blockIdx.x * GW + wave % GW;
  const int split = blockIdx.z;
  // The last query blocks have the most keys: they start first.
  const int yb = gridDim.y - 1 - blockIdx.y;
  const int t0 = (yb * QW + wave / GW) * kPQ;   // the wave's first token
  const int wq_first = yb * QW * kPQ;
  const int wq_last = min(n, wq_first + QW * kPQ) - 1;
  const KeyRange kr = key_range(position, wq_first, wq_last, window);
  const int ntiles = (kr.end - kr.start + KT - 1) / KT;
  const int tile_lo = split * tiles_per_split;
  const int tile_hi = min(ntiles, tile_lo + tiles_per_split);
  if (tile_lo >= tile_hi) return;   // the whole workgroup
  const size_t kvo = (size_t)(blockIdx.x * GW / group) * HD;
  const float sl = scale * 1.44269504088896341f;   // scores in units of log2

  // Staging: the first half of the workgroup carries V (thread: NV dims of the
  // 8 keys of a key group), the second K (thread: NV times 8 dims of a key).
  constexpr int NV = KT * HD / 1024;             // 4, or 2 where KT * HD is 2048
  const bool v_half = wave < 2;
  const int su = tid & 127;
  const int vd = su % (HD / NV), vg = su / (HD / NV);   // V: dims NV vd.., key group vg
  // As loaded, whole vectors: taken apart here they would be waited for where
  // they are loaded (1000 tokens after 1000: 97 -> 114 us).
  float4 raw[2 * NV];
  // A resource per row of a thread's eight loads, so that one offset serves
  // them all; rows past the keys read zeros.
  const int v_off = (32 * (vg >> 2) + 4 * (vg & 3)) * kv_dim * 4 + vd * NV * 4;
  const int k_off = su / (HD / 8) * kv_dim * 4 + su % (HD / 8) * 32;
  auto load_tile = [&](int t) {
    const int kt = kr.start + t * KT, rows = min(KT, kr.end - kt);
    const size_t at = (size_t)kt * kv_dim + kvo;
    auto row = [&](const float* base, int r) {
      return buffer_rsrc(base + at + (size_t)r * kv_dim,
                         (uint32_t)max(0, rows - r) * (uint32_t)kv_dim * 4u);
    };
    if (v_half) {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const i32x4 r = row(values, 16 * (j >> 2) + (j & 3));
        if constexpr (NV == 4) {
          raw[j] = buffer_load_f4(r, v_off);
        } else {
          const i32x2 x = dnx_raw_buffer_load_v2i32(r, v_off, 0, 0);
          (&raw[j >> 1].x)[2 * (j & 1)] = __int_as_float(x.x);
          (&raw[j >> 1].x)[2 * (j & 1) + 1] = __int_as_float(x.y);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < NV; j++) {
        const i32x4 r = row(keys, j * (128 / (HD / 8)));
        raw[2 * j] = buffer_load_f4(r, k_off);
        raw[2 * j + 1] = buffer_load_f4(r, k_off + 16);
      }
    }
  };
  auto store_tile = [&] {
    uint4 p[3];
    if (v_half) {
#pragma unroll
      for (int d = 0; d < NV; d++) {
        float x[8];   // dim d of the eight keys
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = (&raw[j * NV / 4].x)[j * NV % 4 + d];
        split_pieces(x, p);
        // Rows of four dims, 64 bytes, would meet in the same banks for
        // threads two apart: the row's place is turned by bits 3, 4 of the dim.
        const int dim = NV * vd + d, slot = dim ^ ((dim >> 3) & 3);
#pragma unroll
        for (int i = 0; i < 3; i++)
          *(uint4*)(Vp + (i * (KT / 8) + vg) * T::VS + slot * 16) = p[i];
      }
    } else {
#pragma unroll
      for (int j = 0; j < NV; j++) {
        const int u = j * 128 + su, key = u / (HD / 8), g = u % (HD / 8);
        const float4 a = raw[2 * j], b = raw[2 * j + 1];
        const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        split_pieces(x, p);
#pragma unroll
        for (int i = 0; i < 3; i++)
          *(uint4*)(Kp + (i * (HD / 8) + g) * T::KS + key * 16) = p[i];
      }
    }
  };

  // B operand of S^T: the lane's query, dims 32 s + 8 g4 + 0..7, in pieces.
  const int tq = t0 + l16;
  const int qpos = position + tq;
  float4 qv[HD / 16];
  {
    const float* qp = q + ((size_t)min(tq, n - 1) * heads + head) * HD + 8 * g4;
#pragma unroll
    for (int s = 0; s < HD / 32; s++) {
      qv[2 * s] = *(const float4*)(qp + 32 * s);
      qv[2 * s + 1] = *(const float4*)(qp + 32 * s + 4);
    }
  }
  load_tile(tile_lo);
  uint4 qf[HD / 32][3];
#pragma unroll
  for (int s = 0; s < HD / 32; s++) {
    const float4 a = qv[2 * s], b = qv[2 * s + 1];
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    split_pieces(x, qf[s]);
  }
  // The keys that the lane's query sees: see_lo .. see_lo + see_n - 1.
  const uint32_t see_lo = window > 0 ? max(0, qpos - window + 1) : 0;
  const uint32_t see_n = min(kr.end - 1, qpos) + 1 - see_lo;
  float m_run = -INFINITY, l_run = 0.0f;
  v4f o[NE];
#pragma unroll
  for (int e = 0; e < NE; e++) o[e] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

  for (int t = tile_lo; t < tile_hi; t++) {
    __syncthreads();  // every wave is done with the previous tile
    store_tile();
    __syncthreads();
    if (t + 1 < tile_hi) load_tile(t + 1);  // in flight during this tile's math
    const int kt = kr.start + t * KT;
    const int q_hi = position + min(t0 + kPQ, n) - 1;   // the wave's last query's place
    if (t0 >= n || kt > q_hi) continue;                 // no query of the wave sees a key

    // Scores of keys kt + 16 u + 4 g4 + v.
    v4f s[NS], low[NS];
#pragma unroll
    for (int u = 0; u < NS; u++) s[u] = low[u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < HD / 32; d++) {
#pragma unroll
      for (int u = 0; u < NS; u++) {
        uint4 kf[3];
#pragma unroll
        for (int i = 0; i < 3; i++)
          kf[i] = *(const uint4*)(Kp + (i * (HD / 8) + 4 * d + g4) * T::KS + (16 * u + l16) * 16);
        mfma_pieces(kf, qf[d], s[u], low[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < NS; u++) s[u] += low[u];
    const bool edge = kt + KT > position + t0 + 1 || kt + KT > kr.end ||
                      (window > 0 && kt <= q_hi - window);
    float mt = -INFINITY;
#pragma unroll
    for (int u = 0; u < NS; u++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        if (edge) {
          const uint32_t key = kt + 16 * u + 4 * g4 + v;
          s[u][v] = key - see_lo < see_n ? s[u][v] : -INFINITY;
        }
        mt = fmaxf(mt, s[u][v]);
      }
    mt = rows4_max(mt) * sl;
    const float m_new = fmaxf(m_run, mt);
    const float m_ref = m_new == -INFINITY ? 0.0f : m_new;   // nothing seen yet: all p are 0
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_ref);
    float ps = 0.0f;
#pragma unroll
    for (int u = 0; u < NS; u++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        s[u][v] = __builtin_amdgcn_exp2f(fmaf(s[u][v], sl, -m_ref));
        ps += s[u][v];
      }
    l_run = l_run * alpha + rows4_sum(ps);
    m_run = m_new;
    uint4 pf[KT / 32][3];
#pragma unroll
    for (int h = 0; h < KT / 32; h++) {   // 32 keys
      float x[8];
#pragma unroll
      for (int j = 0; j < 8; j++) x[j] = s[2 * h + (j >> 2)][j & 3];
      split_pieces(x, pf[h]);
    }
    // A tile's sums start from zero and join the running ones in one
    // multiply-add (with the rescale): one rounding a tile of a long run.
#pragma unroll
    for (int e = 0; e < NE; e++) {
      v4f d = {0.0f, 0.0f, 0.0f, 0.0f}, low = d;
#pragma unroll
      for (int h = 0; h < KT / 32; h++) {
        uint4 vf[3];
        const int slot = e * 16 + (l16 ^ ((2 * e + (l16 >> 3)) & 3));
#pragma unroll
        for (int i = 0; i < 3; i++)
          vf[i] = *(const uint4*)(Vp + (i * (KT / 8) + 4 * h + g4) * T::VS + slot * 16);
        mfma_pieces(vf, pf[h], d, low);
      }
      d += low;
#pragma unroll
      for (int v = 0; v < 4; v++) o[e][v] = fmaf(o[e][v], alpha, d[v]);
    }
  }
  // NaN if a sum is (an infinity or NaN in Q or K, or a score that overflowed,
  // makes l NaN), or if one is infinite.
  float check = l_run - l_run;
#pragma unroll
  for (int e = 0; e < NE; e++)
#pragma unroll
    for (int v = 0; v < 4; v++) check += o[e][v] - o[e][v];
  if (__builtin_expect(__any(check != check), 0)) {
    const int first = window > 0 ? max(0, position + t0 - window + 1) : 0;
    prefill_special<HD>(q + ((size_t)min(tq, n - 1) * heads + head) * HD, keys + kvo,
                        values + kvo, kv_dim, sl, max(first, kr.start + tile_lo * KT),
                        min(min(kr.end, position + min(t0 + kPQ, n)), kr.start + tile_hi * KT),
                        see_lo, see_n, lane, m_run, l_run, o);
  }
  // The lane's query, dims 16 e + 4 g4 + 0..3: 64 bytes of a row per store
  // and query. Lanes past the last token divide with the others and only
  // store nothing: with them out before, where 4 or 8 lanes were left (one or
  // two tokens), the divisions took 0.4 to 0.8 us longer (65 tokens, 16 / 4
  // heads, hd 64: 8.5 -> 7.7 us).
  const bool own = tq < n;
  const size_t th = (size_t)min(tq, n - 1) * heads + head;
  if (splits > 1) {
    float* w = ws + (th * splits + split) * (HD + 4);
#pragma unroll
    for (int e = 0; e < NE; e++)
      if (own) *(float4*)(w + 4 + e * 16 + 4 * g4) = make_float4(o[e][0], o[e][1], o[e][2], o[e][3]);
    if (g4 == 0 && own) {
      w[0] = m_run;
      w[1] = l_run;
    }
  } else {
    const float g = gate != nullptr ? 1.0f / (1.0f + expf(-gate[th])) : 1.0f;
#pragma unroll
    for (int e = 0; e < NE; e++) {
      float4 y = make_float4(o[e][0] / l_run, o[e][1] / l_run, o[e][2] / l_run, o[e][3] / l_run);
      if (gate != nullptr) y = make_float4(y.x * g, y.y * g, y.z * g, y.w * g);
      if (own) *(float4*)(out + th * HD + e * 16 + 4 * g4) = y;
    }
  }
}

// How the prefill kernel dealt a row's keys: workgroups of `queries` tokens,
// tiles of kt keys, tps tiles to a split. A row's last splits may be empty
// (its keys end before them): they were not written and are not read.
struct RowSplits {
  int position, n, window, queries, kt, tps;
};

// The combine of the prefill kernel's partial rows (at most 64 splits, hd 64
// or 128): one wave per row, four rows per workgroup, no barrier. Lane s
// holds split s's statistics, reduced by DPP; lane i sums dims ND i .. ND i +
// ND - 1 in split order, C splits' loads in flight (the fewest of 2, 4, 8
// covering the splits), the first C requested with the statistics, so that a
// row of up to C splits waits for memory once. Splits past the row's last
// read zeros (the resource ends there).
//
// With `panel`, each row's values also go into the fp6 activation panel of
// out ([tokens][heads * hd]) for the matmul that reads it (a prefill chunk's
// o projection): the row through the wave's LDS, then four lanes per 32-value
// block (panel4_lane, the panel quantizer's bytes). Records of tokens past
// the last row are not written.
template <int C, int ND>  // splits per load batch: 2, 4 or 8; hd / 64
__global__ void __launch_bounds__(kThreads)
attention_combine_rows_kernel(const float* __restrict__ ws, const float* __restrict__ gate,
                              float* __restrict__ out, int heads, int max_splits, int rows,
                              uint8_t* __restrict__ panel, RowSplits rsp) {
  constexpr int hd = 64 * ND, row = hd + 4;
  __shared__ __align__(16) float row_lds[kWaves][hd];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = blockIdx.x * kWaves + wave;   // token * heads + head
  if (r >= rows) return;
  const int token = r / heads;
  const int first = token / rsp.queries * rsp.queries;
  const int splits = live_splits(
      key_range(rsp.position, first, min(rsp.n, first + rsp.queries) - 1, rsp.window), rsp.kt,
      rsp.tps);
  const i32x4 rs = buffer_rsrc(ws + (size_t)r * max_splits * row, (uint32_t)splits * row * 4u);
  const i32x2 ml = dnx_raw_buffer_load_v2i32(rs, lane * row * 4, 0, 0);
  float v[C][ND];
  auto load = [&](int s0) {
#pragma unroll
    for (int u = 0; u < C; u++) {
      const int off = ((s0 + u) * row + 4 + ND * lane) * 4;
      if constexpr (ND == 2) {
        const i32x2 x = dnx_raw_buffer_load_v2i32(rs, off, 0, 0);
        v[u][0] = __int_as_float(x.x);
        v[u][1] = __int_as_float(x.y);
      } else {
        v[u][0] = __int_as_float(dnx_raw_buffer_load_i32(rs, off, 0, 0));
      }
    }
  };
  load(0);
  const float m = lane < splits ? __int_as_float(ml.x) : -INFINITY;
  const float mx = wave_max_dpp(m);
  const float f = m == -INFINITY ? 0.0f : exp2f(m - mx);   // m in units of log2
  const float l = wave_sum_dpp(__int_as_float(ml.y) * f);
  float acc[ND] = {};
  for (int s0 = 0; s0 < splits; s0 += C) {
    if (s0 > 0) load(s0);
#pragma unroll
    for (int u = 0; u < C; u++) {
      const float fs = lane_value(f, s0 + u);   // 0 past the last split
#pragma unroll
      for (int i = 0; i < ND; i++) acc[i] += v[u][i] * fs;
    }
  }
  const float g = gate != nullptr ? 1.0f / (1.0f + expf(-gate[r])) : 1.0f;
#pragma unroll
  for (int i = 0; i < ND; i++) acc[i] = gate != nullptr ? (acc[i] / l) * g : acc[i] / l;
  float* mine = row_lds[wave];
  float* y = out + (size_t)r * hd + ND * lane;
  if constexpr (ND == 2) {
    *(float2*)y = make_float2(acc[0], acc[1]);
    *(float2*)(mine + 2 * lane) = make_float2(acc[0], acc[1]);
  } else {
    *y = acc[0];
    mine[lane] = acc[0];
  }
  if (panel == nullptr) return;
  // LDS operations of one wave execute in order; the fence keeps the
  // compiler from moving the reads above the writes.
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (lane < hd / 8) {
    const int head = r - token * heads;
    const int B = heads * hd / kBlock;
    const int b = head * (hd / kBlock) + (lane >> 2);
    const float4 v0 = *(const float4*)(mine + lane * 8);
    const float4 v1 = *(const float4*)(mine + lane * 8 + 4);
    panel4_lane(v0, v1, lane & 3, token % kTokens,
                panel + ((size_t)(token / kTokens) * B + b) * kRec);
  }
}

template <int HD>
void launch_combine_rows(const float* ws, const float* gate, float* out, int64_t heads, int splits,
                         int64_t rows, uint8_t* panel, RowSplits rsp, hipStream_t st) {
  constexpr int ND = HD / 64;
  auto k = splits <= 2 ? attention_combine_rows_kernel<2, ND>
         : splits <= 4 ? attention_combine_rows_kernel<4, ND> : attention_combine_rows_kernel<8, ND>;
  hipLaunchKernelGGL(k, dim3((unsigned)((rows + kWaves - 1) / kWaves)), dim3(kThreads), 0, st, ws,
                     gate, out, (int)heads, splits, (int)rows, panel, rsp);
}

template <int HD, int KT>
void launch_prefill(int gw, dim3 grid, hipStream_t st, const float* q, const float* keys,
                    const float* values, const float* gate, float* out, float* ws, int position,
                    int n, int heads, int kv_dim, int group, int window, float scale, int splits,
                    int tps) {
  auto k = gw == 4 ? attention_prefill_kernel<HD, 4, KT>
         : gw == 2 ? attention_prefill_kernel<HD, 2, KT> : attention_prefill_kernel<HD, 1, KT>;
  hipLaunchKernelGGL(k, grid, dim3(kThreads), 0, st, q, keys, values, gate, out, ws, position, n,
                     heads, kv_dim, group, window, scale, splits, tps);
}

// Library-owned workspace of the split attention, grown on demand: a call
// with more (head, token, split) entries than any before allocates, so such
// a call must not be the first inside a graph capture.
float* gAttnWs = nullptr;
size_t gAttnWsBytes = 0;

float* attention_workspace(size_t bytes) {
  if (bytes <= gAttnWsBytes) return gAttnWs;
  if (gAttnWs != nullptr) {
    if (hipDeviceSynchronize() != hipSuccess) return nullptr;
    (void)hipFree(gAttnWs);
    gAttnWs = nullptr;
    gAttnWsBytes = 0;
  }
  if (hipMalloc(&gAttnWs, bytes) != hipSuccess) return nullptr;
  gAttnWsBytes = bytes;
  return gAttnWs;
}

// dst += src (lab_metal.m:560-566) and dst = src (:567-572), element-wise.
__global__ void __launch_bounds__(kThreads)
add_kernel(const float* __restrict__ src, float* __restrict__ dst, int64_t count) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < count;
       i += (int64_t)gridDim.x * kThreads) {
    dst[i] = dst[i] + src[i];
  }
}

__global__ void __launch_bounds__(kThreads)
copy_kernel(const float* __restrict__ src, float* __restrict__ dst, int64_t count) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < count;
       i += (int64_t)gridDim.x * kThreads) {
    dst[i] = src[i];
  }
}

// Activation steering in place, semantics of lab_metal.m:531-557. Each
// workgroup rewrites one row. Mode 0 shifts the row by the vector. Mode 1
// projects out the vector's direction, scaled: the block reduces the row's
// dot product with v (v is expected to have unit length), then every
// element drops (scale * dot) * v[j].
__global__ void __launch_bounds__(kThreads)
steer_kernel(float* x, const float* __restrict__ v, int cols, int mode, float scale) {
  __shared__ float scratch[kWaves];
  float* xr = x + (size_t)blockIdx.x * cols;
  if (mode == 0) {
    for (int j = threadIdx.x; j < cols; j += kThreads) xr[j] = xr[j] + v[j];
    return;
  }
  float along = 0.0f;
  for (int j = threadIdx.x; j < cols; j += kThreads) along += xr[j] * v[j];
  along = block_sum(along, scratch);
  const float c = scale * along;
  for (int j = threadIdx.x; j < cols; j += kThreads) xr[j] = xr[j] - c * v[j];
}

int grid_for(int64_t items) {
  const int64_t g = (items + kThreads - 1) / kThreads;
  return (int)(g < 1 ? 1 : g > 65536 ? 65536 : g);
}

// The split-key attention (few (head, token) pairs, many keys): the split
// kernel, then the combine. DNX_EINVAL when it does not apply (nothing
// launched). rp: the q and k head norms folded in (one token, one
// workgroup per KV head and split), or null.
int attention_split(const float* q, const float* keys, const float* values, const float* gate,
                    float* out, int64_t position, int64_t n, int64_t heads, int64_t kv_heads,
                    int64_t hd, int64_t window, float scale, dnx_stream_t stream,
                    const RopeArgs* rp) {
  const int64_t last = position + n - 1;
  const int64_t keys_of_last = window > 0 && last >= window ? window : last + 1;
  const int kps = split_keys((int)hd);
  const int64_t splits = (keys_of_last + kps - 1) / kps;
  // (Also when the keys exceed the one-workgroup kernel's LDS.) The split
  // kernel's buffer offsets reach 4096 key rows: 32-bit up to 2^17 floats
  // per row.
  const size_t ws_bytes = (size_t)heads * n * splits * (hd + 4) * 4;
  if (!(splits > 1 && (heads * n < 256 || keys_of_last > dnx_attention_max_keys(hd)) &&
        splits <= 16000 && ws_bytes <= ((size_t)1 << 30) && kv_heads * hd <= (1 << 17))) {
    return DNX_EINVAL;
  }
  // G query heads per workgroup: the largest of 8, 4, 2, 1 dividing the
  // heads per KV head.
  const int group = (int)(heads / kv_heads);
  const int G = group % 8 == 0 ? 8 : group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
  if (rp != nullptr && (n != 1 || G != group || hd > kRopeMaxHd)) return DNX_EINVAL;
  float* ws = attention_workspace(ws_bytes);
  if (ws == nullptr) return DNX_ENOMEM;
  const dim3 grid((unsigned)(heads / G), (unsigned)n, (unsigned)splits);
  const hipStream_t st = (hipStream_t)stream;
  const int kv_dim = (int)(kv_heads * hd);
  const RopeArgs ra = rp != nullptr ? *rp : RopeArgs{};
  auto split = [&](auto g_tag, auto rope_tag) {
    constexpr int kG = decltype(g_tag)::value;
    constexpr bool kR = decltype(rope_tag)::value;
    launch_split<kG, kR>(grid, st, q, keys, values, ws, (int)position, (int)heads, kv_dim, group,
                         (int)hd, (int)window, scale, (int)splits, kps, ra);
  };
  auto by_g = [&](auto rope_tag) {
    switch (G) {
      case 8: split(std::integral_constant<int, 8>{}, rope_tag); break;
      case 4: split(std::integral_constant<int, 4>{}, rope_tag); break;
      case 2: split(std::integral_constant<int, 2>{}, rope_tag); break;
      default: split(std::integral_constant<int, 1>{}, rope_tag); break;
    }
  };
  if (rp != nullptr) {
    by_g(std::true_type{});
  } else {
    by_g(std::false_type{});
  }
  if (hipGetLastError() != hipSuccess) return DNX_ELAUNCH;
  if (rp != nullptr) {
    hipLaunchKernelGGL(attention_combine_kernel<true>, dim3((unsigned)heads, (unsigned)n),
                       dim3(kThreads), (size_t)splits * 4, st, ws, gate, out, (int)heads,
                       (int)hd, (int)splits, const_cast<float*>(q), ra);
  } else {
    hipLaunchKernelGGL(attention_combine_kernel<false>, dim3((unsigned)heads, (unsigned)n),
                       dim3(kThreads), (size_t)splits * 4, st, ws, gate, out, (int)heads,
                       (int)hd, (int)splits, (float*)nullptr, RopeArgs{});
  }
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

// The vector norm with the activation panel of its output (kPanel), with
// or without the residual add before it (kAdd): V float4 per thread as the
// row needs, the row in dynamic LDS.
template <bool kAdd>
int launch_norm_panel(const float* x_in, const float* w, float* out, int64_t rows, int64_t cols,
                      float eps, const float* m, float* x_out, uint8_t* panel, hipStream_t s) {
  const int64_t per = (cols / 4 + kThreads - 1) / kThreads;  // float4 per thread
  const size_t lds = (size_t)cols * 4;
  const dim3 grid((unsigned)rows);
  if (per <= 1) {
    hipLaunchKernelGGL((rms_norm_vec_kernel<1, kAdd, true>), grid, dim3(kThreads), lds, s, x_in, w,
                       out, (int)cols, eps, 0, m, x_out, panel);
  } else if (per <= 2) {
    hipLaunchKernelGGL((rms_norm_vec_kernel<2, kAdd, true>), grid, dim3(kThreads), lds, s, x_in, w,
                       out, (int)cols, eps, 0, m, x_out, panel);
  } else if (per <= 4) {
    hipLaunchKernelGGL((rms_norm_vec_kernel<4, kAdd, true>), grid, dim3(kThreads), lds, s, x_in, w,
                       out, (int)cols, eps, 0, m, x_out, panel);
  } else {
    hipLaunchKernelGGL((rms_norm_vec_kernel<8, kAdd, true>), grid, dim3(kThreads), lds, s, x_in, w,
                       out, (int)cols, eps, 0, m, x_out, panel);
  }
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

bool norm_panel_ok(int64_t rows, int64_t cols, uintptr_t ptrs) {
  return rows > 0 && rows <= 256 && cols > 0 && cols % kBlock == 0 && cols <= 8192 &&
         (ptrs & 15) == 0 && f6_panel_bytes(rows, cols) < (1ll << 31);
}

}  // namespace

extern "C" {

int dnx_rms_norm_f6panel(const float* x, const float* w, float* out, void* panel, int64_t rows,
                         int64_t cols, float eps, dnx_stream_t stream) {
  if (!norm_panel_ok(rows, cols, (uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)panel)) {
    return DNX_EINVAL;
  }
  return launch_norm_panel<false>(x, w, out, rows, cols, eps, nullptr, nullptr, (uint8_t*)panel,
                                  (hipStream_t)stream);
}

int dnx_add_rms_norm_f6panel(const float* m, float* x, const float* w, float* out, void* panel,
                             int64_t rows, int64_t cols, float eps, dnx_stream_t stream) {
  if (!norm_panel_ok(rows, cols, (uintptr_t)m | (uintptr_t)x | (uintptr_t)w | (uintptr_t)out |
                                     (uintptr_t)panel)) {
    return DNX_EINVAL;
  }
  return launch_norm_panel<true>(x, w, out, rows, cols, eps, m, x, (uint8_t*)panel,
                                 (hipStream_t)stream);
}

int dnx_rms_norm(const float* x, const float* w, float* out, int64_t rows, int64_t cols,
                 float eps, int accumulate, dnx_stream_t stream) {
  if (rows < 0 || cols <= 0 || cols > (1 << 30) || rows > 0x7fffffff) return DNX_EINVAL;
  if (rows == 0) return DNX_OK;
  // Register rows for the latency-bound case (no more rows than CUs, as in a
  // decode step); at prefill sizes the streaming loop keeps more rows in
  // flight (4096 x 2048: 14 against 21 us).
  const bool vec = rows <= 256 && cols % 4 == 0 && cols <= 16 * 4 * kThreads &&
                   (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0;
  const unsigned grid = (unsigned)rows;
  const hipStream_t s = (hipStream_t)stream;
  if (vec) {
    const int64_t per = (cols / 4 + kThreads - 1) / kThreads;  // float4 per thread
    if (per <= 1) {
      hipLaunchKernelGGL(rms_norm_vec_kernel<1>, dim3(grid), dim3(kThreads), 0, s, x, w, out,
                         (int)cols, eps, accumulate, nullptr, nullptr, nullptr);
    } else if (per <= 2) {
      hipLaunchKernelGGL(rms_norm_vec_kernel<2>, dim3(grid), dim3(kThreads), 0, s, x, w, out,
                         (int)cols, eps, accumulate, nullptr, nullptr, nullptr);
    } else if (per <= 4) {
      hipLaunchKernelGGL(rms_norm_vec_kernel<4>, dim3(grid), dim3(kThreads), 0, s, x, w, out,
                         (int)cols, eps, accumulate, nullptr, nullptr, nullptr);
    } else if (per <= 8) {
      hipLaunchKernelGGL(rms_norm_vec_kernel<8>, dim3(grid), dim3(kThreads), 0, s, x, w, out,
                         (int)cols, eps, accumulate, nullptr, nullptr, nullptr);
    } else {
      hipLaunchKernelGGL(rms_norm_vec_kernel<16>, dim3(grid), dim3(kThreads), 0, s, x, w, out,
                         (int)cols, eps, accumulate, nullptr, nullptr, nullptr);
    }
  } else {
    hipLaunchKernelGGL(rms_norm_kernel, dim3(grid), dim3(kThreads), 0, s, x, w, out, (int)cols,
                       eps, accumulate);
  }
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

int dnx_add_rms_norm(const float* m, float* x, const float* w, float* out, int64_t rows,
                     int64_t cols, float eps, dnx_stream_t stream) {
  if (rows < 0 || cols <= 0 || rows > 256 || cols % 4 != 0 || cols > 16 * 4 * kThreads ||
      (((uintptr_t)m | (uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) != 0) {
    return DNX_EINVAL;
  }
  if (rows == 0) return DNX_OK;
  const unsigned grid = (unsigned)rows;
  const hipStream_t s = (hipStream_t)stream;
  const int64_t per = (cols / 4 + kThreads - 1) / kThreads;  // float4 per thread
  if (per <= 1) {
    hipLaunchKernelGGL((rms_norm_vec_kernel<1, true>), dim3(grid), dim3(kThreads), 0, s, x, w,
                       out, (int)cols, eps, 0, m, x, nullptr);
  } else if (per <= 2) {
    hipLaunchKernelGGL((rms_norm_vec_kernel<2, true>), dim3(grid), dim3(kThreads), 0, s, x, w,
                       out, (int)cols, eps, 0, m, x, nullptr);
  } else if (per <= 4) {
    hipLaunchKernelGGL((rms_norm_vec_kernel<4, true>), dim3(grid), dim3(kThreads), 0, s, x, w,
                       out, (int)cols, eps, 0, m, x, nullptr);
  } else if (per <= 8) {
    hipLaunchKernelGGL((rms_norm_vec_kernel<8, true>), dim3(grid), dim3(kThreads), 0, s, x, w,
                       out, (int)cols, eps, 0, m, x, nullptr);
  } else {
    hipLaunchKernelGGL((rms_norm_vec_kernel<16, true>), dim3(grid), dim3(kThreads), 0, s, x, w,
                       out, (int)cols, eps, 0, m, x, nullptr);
  }
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

int dnx_head_norm_rope(float* x, int64_t x_stride, const float* w, const float* rope,
                       int64_t rope_stride, int64_t heads, int64_t hd, int64_t n, float eps,
                       dnx_stream_t stream) {
  if (heads <= 0 || n < 0 || hd <= 0 || hd % 2 != 0 || hd > 512 || x_stride < heads * hd ||
      rope_stride < hd || x_stride > 0x7fffffff || rope_stride > 0x7fffffff ||
      heads > 65535 || n > 65535) {
    return DNX_EINVAL;
  }
  if (n == 0) return DNX_OK;
  hipLaunchKernelGGL(head_norm_rope_kernel, dim3((unsigned)heads, (unsigned)n), dim3(64), 0,
                     (hipStream_t)stream, x, (int)x_stride, w, rope, (int)rope_stride, (int)hd,
                     eps, (int)heads, x, (int)x_stride, w);
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

int dnx_head_norm_rope2(float* x0, int64_t x0_stride, const float* w0, int64_t heads0,
                        float* x1, int64_t x1_stride, const float* w1, int64_t heads1,
                        const float* rope, int64_t rope_stride, int64_t hd, int64_t n, float eps,
                        dnx_stream_t stream) {
  if (heads0 <= 0 || heads1 <= 0 || n < 0 || hd <= 0 || hd % 2 != 0 || hd > 512 ||
      x0_stride < heads0 * hd || x1_stride < heads1 * hd || rope_stride < hd ||
      x0_stride > 0x7fffffff || x1_stride > 0x7fffffff || rope_stride > 0x7fffffff ||
      heads0 + heads1 > 65535 || n > 65535) {
    return DNX_EINVAL;
  }
  if (n == 0) return DNX_OK;
  hipLaunchKernelGGL(head_norm_rope_kernel, dim3((unsigned)(heads0 + heads1), (unsigned)n),
                     dim3(64), 0, (hipStream_t)stream, x0, (int)x0_stride, w0, rope,
                     (int)rope_stride, (int)hd, eps, (int)heads0, x1, (int)x1_stride, w1);
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

int dnx_short_conv(const float* bcx, const float* weight, float* history, float* y,
                   int64_t width, int64_t k, int64_t n, dnx_stream_t stream) {
  if (width <= 0 || k < 1 || k > kMaxConvK || n < 0 || width > 0x7fffffff ||
      n > 0x7fffffff) {
    return DNX_EINVAL;
  }
  if (n == 0) return DNX_OK;
  const int64_t slabs = (width + kConvCh - 1) / kConvCh, tiles = (n + kConvT - 1) / kConvT;
  if (slabs > 0x7fffffff || tiles > 65535) return DNX_EINVAL;
  hipLaunchKernelGGL(conv_kernel, dim3((unsigned)slabs, (unsigned)tiles), dim3(kThreads), 0,
                     (hipStream_t)stream, bcx, weight, history, y, (int)width, (int)k, (int)n);
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

int dnx_attention_rope(float* q, float* keys, const float* values, const float* gate, float* out,
                       int64_t position, int64_t heads, int64_t kv_heads, int64_t hd,
                       int64_t window, const float* q_norm, const float* k_norm,
                       const float* rope, float eps, dnx_stream_t stream) {
  if (position < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || hd <= 0 ||
      hd % 4 != 0 || hd > kRopeMaxHd || kThreads % hd != 0 || window < 0 || heads > 65535 ||
      position + 1 > 0x7fffffff || ((uintptr_t)keys & 15) || ((uintptr_t)q & 15) ||
      q_norm == nullptr || k_norm == nullptr || rope == nullptr) {
    return DNX_EINVAL;
  }
  const RopeArgs rp{rope, q_norm, k_norm, keys, eps};
  return attention_split(q, keys, values, gate, out, position, 1, heads, kv_heads, hd, window,
                         (float)(1.0 / sqrt((double)hd)), stream, &rp);
}

int64_t dnx_attention_max_keys(int64_t hd) {
  if (hd <= 0 || hd > 256 || kThreads % hd != 0) return -1;
  // LDS: q (hd) + scores (rounded up to 4) + value partials ((256 / hd) x
  // hd) + the kernel's 4-float reduction scratch, within 64 KB.
  return (64 * 1024 / 4) - hd - kThreads - 4 - kWaves;
}

// The attention, and with `panel` the fp6 activation panel of out too (only
// where the split matrix-core path and its row combine run; else DNX_EINVAL
// before anything is launched).
static int attention_impl(const float* q, const float* keys, const float* values,
                          const float* gate, float* out, uint8_t* panel, int64_t position,
                          int64_t n, int64_t heads, int64_t kv_heads, int64_t hd, int64_t window,
                          dnx_stream_t stream) {
  if (n < 0 || position < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 ||
      hd <= 0 || hd % 4 != 0 || hd > 256 || kThreads % hd != 0 || window < 0 ||
      heads > 65535 || n > 65535 || position + n > 0x7fffffff || ((uintptr_t)keys & 15) ||
      ((uintptr_t)q & 15)) {
    return DNX_EINVAL;
  }
  if (panel != nullptr && (hd % kBlock != 0 || ((uintptr_t)panel & 15) || n == 0)) {
    return DNX_EINVAL;
  }
  if (n == 0) return DNX_OK;
  const int64_t last = position + n - 1;
  const int64_t keys_of_last = window > 0 && last >= window ? window : last + 1;
  const float scale = (float)(1.0 / sqrt((double)hd));
  // 8+ tokens at hd 64 or 128: the matrix-core kernel.
  if ((hd == 64 || hd == 128) && n >= 8 && kv_heads * hd <= (1 << 20) &&
      ((uintptr_t)out & 15) == 0) {
    const int64_t group = heads / kv_heads;
    const int gw = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    const PrefillSplit sp = prefill_split(position, n, heads, hd, window, gw);
    if (panel != nullptr && !sp.panel) return DNX_EINVAL;
    float* ws = nullptr;
    if (sp.splits > 1) {
      const size_t need = (size_t)n * heads * sp.splits * (hd + 4) * 4;
      ws = attention_workspace(std::max(need, kPrefillWorkspace));
      if (ws == nullptr) return DNX_ENOMEM;
    }
    const int64_t qb = kPQ * (4 / gw);
    const dim3 grid((unsigned)(heads / gw), (unsigned)((n + qb - 1) / qb), (unsigned)sp.splits);
    const hipStream_t st = (hipStream_t)stream;
    auto launch = hd == 128 ? launch_prefill<128, 32>
                : sp.kt == 32 ? launch_prefill<64, 32> : launch_prefill<64, 64>;
    launch(gw, grid, st, q, keys, values, gate, out, ws, (int)position, (int)n, (int)heads,
           (int)(kv_heads * hd), (int)group, (int)window, scale, sp.splits, sp.tps);
    if (hipGetLastError() != hipSuccess) return DNX_ELAUNCH;
    if (sp.splits > 1) {
      const RowSplits rsp{(int)position, (int)n, (int)window, (int)qb, sp.kt, sp.tps};
      if (hd == 128) {
        launch_combine_rows<128>(ws, gate, out, heads, sp.splits, n * heads, panel, rsp, st);
      } else {
        launch_combine_rows<64>(ws, gate, out, heads, sp.splits, n * heads, panel, rsp, st);
      }
    }
    return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
  }
  if (panel != nullptr) return DNX_EINVAL;
  // Few (head, token) workgroups for many keys: split the keys.
  const int rc = attention_split(q, keys, values, gate, out, position, n, heads, kv_heads, hd,
                                 window, scale, stream, nullptr);
  if (rc != DNX_EINVAL) return rc;
  if (keys_of_last > dnx_attention_max_keys(hd)) return DNX_EINVAL;
  const size_t lds = (size_t)(hd + ((keys_of_last + 3) & ~3ll) + kThreads) * 4;
  hipLaunchKernelGGL(attention_kernel, dim3((unsigned)heads, (unsigned)n), dim3(kThreads), lds,
                     (hipStream_t)stream, q, keys, values, gate, out, (int)position,
                     (int)heads, (int)(kv_heads * hd), (int)(heads / kv_heads), (int)hd,
                     (int)window, scale);
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

int dnx_attention(const float* q, const float* keys, const float* values, const float* gate,
                  float* out, int64_t position, int64_t n, int64_t heads, int64_t kv_heads,
                  int64_t hd, int64_t window, dnx_stream_t stream) {
  return attention_impl(q, keys, values, gate, out, nullptr, position, n, heads, kv_heads, hd,
                        window, stream);
}

int dnx_attention_f6panel(const float* q, const float* keys, const float* values,
                          const float* gate, float* out, void* panel, int64_t position, int64_t n,
                          int64_t heads, int64_t kv_heads, int64_t hd, int64_t window,
                          dnx_stream_t stream) {
  if (panel == nullptr) return DNX_EINVAL;
  return attention_impl(q, keys, values, gate, out, (uint8_t*)panel, position, n, heads,
                        kv_heads, hd, window, stream);
}

int dnx_add(const float* src, float* dst, int64_t count, dnx_stream_t stream) {
  if (count < 0) return DNX_EINVAL;
  if (count == 0) return DNX_OK;
  hipLaunchKernelGGL(add_kernel, dim3(grid_for(count)), dim3(kThreads), 0, (hipStream_t)stream,
                     src, dst, count);
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

int dnx_copy(const float* src, float* dst, int64_t count, dnx_stream_t stream) {
  if (count < 0) return DNX_EINVAL;
  if (count == 0) return DNX_OK;
  hipLaunchKernelGGL(copy_kernel, dim3(grid_for(count)), dim3(kThreads), 0, (hipStream_t)stream,
                     src, dst, count);
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

int dnx_steer(float* x, const float* v, int64_t rows, int64_t cols, int64_t mode, float scale,
              dnx_stream_t stream) {
  if (rows < 0 || cols <= 0 || (mode != 0 && mode != 1) || rows > 0x7fffffff ||
      cols > (1 << 30)) {
    return DNX_EINVAL;
  }
  if (rows == 0) return DNX_OK;
  hipLaunchKernelGGL(steer_kernel, dim3((unsigned)rows), dim3(kThreads), 0, (hipStream_t)stream,
                     x, v, (int)cols, (int)mode, scale);
  return hipGetLastError() == hipSuccess ? DNX_OK : DNX_ELAUNCH;
}

}  // extern "C"
