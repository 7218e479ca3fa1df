/*
 * aoship_model.hip — the parts of a decoder step around the adapter-augmented projections, as in
 * the MLX fused forward (mlx_model_forward_with_cache_and_lora,
 * crates/adapteros-lora-mlx-ffi/src/mlx_cpp_wrapper_real.cpp:3339-3527):
 *
 *   embedding lookup          take(embed, ids) with 4-bit rows dequantised (…real.cpp:3421-3432)
 *   residual add + RMSNorm    x * (w / sqrt(mean(x^2) + eps)) (…real.cpp:3384-3390), float32, the
 *                             residual stream kept in float32 (MLX promotes to float32 after RoPE)
 *   RoPE + bias + KV cache    the fused forward's rotation (…real.cpp:3249-3279): halves
 *                             [x1, x2] -> [x1 cos - x2 sin, x1 sin + x2 cos] with
 *                             inv_freq_i = 1 / theta^(-2i / hd), angle = position * inv_freq_i;
 *                             K and V appended to a bf16 cache laid out [kv head][position][hd]
 *   attention                 causal scaled dot-product attention over the cache, GQA by head
 *                             group (…real.cpp:3282-3327), with an online softmax in float32:
 *                             decode and short prompts by one wave per (split of positions, head,
 *                             token) and a fixed-order merge of the splits; prompts by 128-token
 *                             tiles on the matrix cores
 *
 * Every reduction has a fixed order, so results are bit-identical run to run.
 */
#include "aoship_device.h"
#include "aoship_internal.h"
#include <hip/hip_ext.h>

namespace {

/* ---- embedding -------------------------------------------------------------------------------- */

/* One thread per 8 elements of a row (one packed word, or 16 bytes of bfloat16), so every load of
 * the launch is in flight at once. */
__global__ void __launch_bounds__(256) aos_embed_kernel(aos_embed_params p) {
  const int t = blockIdx.y, g = blockIdx.x * 256 + threadIdx.x;
  if (t == 0 && g == 0 && p.clear) *p.clear = 0u;
  if (8 * g >= p.H) return;
  const int id = p.ids[t];
  float4 *dst = (float4 *)(p.hidden + (size_t)t * p.H + 8 * g);
  if (id < 0 || id >= p.vocab) {
    dst[0] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    dst[1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (g == 0 && p.status) p.status[0] = 1;
    return;
  }
  float v[8];
  if (p.q4) {
    const uint32_t w = p.q4[(size_t)id * (p.H / 8) + g];
    const size_t gi = (size_t)id * (p.H / 64) + (g >> 3);
    const float s = aos_f16_to_f32(p.s16[gi]);
    const float b = p.b16 ? aos_f16_to_f32(p.b16[gi]) : 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = s * (float)((w >> (4 * e)) & 15u) + b; /* low nibble first */
  } else {
    const u32x4 r = *(const u32x4 *)(p.bf16 + (size_t)id * p.H + 8 * g);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[2 * e] = __builtin_bit_cast(float, w[e] << 16);
      v[2 * e + 1] = __builtin_bit_cast(float, w[e] & 0xffff0000u);
    }
  }
  dst[0] = make_float4(v[0], v[1], v[2], v[3]);
  dst[1] = make_float4(v[4], v[5], v[6], v[7]);
}

/* ---- residual add + RMSNorm ------------------------------------------------------------------- */

/* One workgroup of 1024 threads per token; each thread holds up to NORM_J runs of 4 elements
 * (H <= 16384), loaded together before any arithmetic. The sum of squares is formed per thread
 * in element order, across each wave by a butterfly and across the 16 waves in wave order. */
constexpr int NORM_J = 4;

__global__ void __launch_bounds__(1024) aos_norm_kernel(aos_norm_params p) {
  __shared__ float red[16];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, H = p.H;
  float *x = p.hidden + (size_t)t * H;
  const uint16_t *a = p.add ? p.add + (size_t)t * H : nullptr;
  float4 xv[NORM_J], wv[NORM_J];
  u32x2 av[NORM_J];
#pragma unroll
  for (int j = 0; j < NORM_J; ++j) {
    const int e = 4 * (tid + 1024 * j);
    if (e < H) {
      xv[j] = *(const float4 *)(x + e);
      wv[j] = *(const float4 *)(p.w + e);
      if (a) av[j] = *(const u32x2 *)(a + e);
    }
  }
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < NORM_J; ++j) {
    const int e = 4 * (tid + 1024 * j);
    if (e < H) {
      if (a) {
        xv[j].x = xv[j].x + __builtin_bit_cast(float, av[j].x << 16);
        xv[j].y = xv[j].y + __builtin_bit_cast(float, av[j].x & 0xffff0000u);
        xv[j].z = xv[j].z + __builtin_bit_cast(float, av[j].y << 16);
        xv[j].w = xv[j].w + __builtin_bit_cast(float, av[j].y & 0xffff0000u);
        *(float4 *)(x + e) = xv[j];
      }
      ss += xv[j].x * xv[j].x;
      ss += xv[j].y * xv[j].y;
      ss += xv[j].z * xv[j].z;
      ss += xv[j].w * xv[j].w;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) ss = ss + aos_shfl_f(ss, lane ^ o);
  if (lane == 0) red[tid >> 6] = ss;
  __syncthreads();
  float tot = 0.0f;
#pragma unroll
  for (int w = 0; w < 16; ++w) tot += red[w];
  const float mean = tot / (float)H;
  const float d = sqrtf(mean + p.eps);
  uint16_t *o = p.out + (size_t)t * H;
#pragma unroll
  for (int j = 0; j < NORM_J; ++j) {
    const int e = 4 * (tid + 1024 * j);
    if (e < H) {
      u32x2 r;
      r.x = (uint32_t)aos_f32_to_bf16(xv[j].x * (wv[j].x / d)) | ((uint32_t)aos_f32_to_bf16(xv[j].y * (wv[j].y / d)) << 16);
      r.y = (uint32_t)aos_f32_to_bf16(xv[j].z * (wv[j].z / d)) | ((uint32_t)aos_f32_to_bf16(xv[j].w * (wv[j].w / d)) << 16);
      *(u32x2 *)(o + e) = r;
    }
  }
}

/* ---- RoPE, biases, KV cache append ---------------------------------------------------------- */

/* A bfloat16 infinity or NaN. */
__device__ __forceinline__ bool bf16_nonfinite(uint32_t b) { return (b & 0x7f80u) == 0x7f80u; }

/* Workgroup (part, token): items w = 256 part + thread, then every gridDim.x * 256 further; an item is a
 * rotated pair of q or k, or an element of v. The token's cosines and sines are formed once per workgroup
 * in LDS: formed per item, the same angle's for every head, they made the launch arithmetic-bound (1900
 * tokens of 28 + 4 heads of 128: 32 us, now 17). */
__global__ void __launch_bounds__(256) aos_rope_kernel(aos_rope_params p) {
  __shared__ float cs[AOS_ATTN_MAX_HD / 2], sn[AOS_ATTN_MAX_HD / 2];
  const int t = blockIdx.y, half = p.hd / 2;
  const int pos = p.offset + t;
  const float fpos = (float)pos;
  const int nq = p.nh * half, nk = p.nkv * half, nv = p.nkv * p.hd;
  for (int i = threadIdx.x; i < half; i += 256) {
    const float ang = fpos * p.inv_freq[i];
    cs[i] = cosf(ang);
    sn[i] = sinf(ang);
  }
  __syncthreads();
  for (int w = blockIdx.x * 256 + threadIdx.x; w < nq + nk + nv; w += gridDim.x * 256) {
    if (w < nq + nk) {
      const bool isq = w < nq;
      const int idx = isq ? w : w - nq;
      const int h = idx / half, i = idx - h * half;
      const int width = (isq ? p.nh : p.nkv) * p.hd;
      const uint16_t *src = (isq ? p.q : p.k) + (size_t)t * width + (size_t)h * p.hd;
      const float *bias = isq ? p.bq : p.bk;
      float x1 = aos_bf16_to_f32(src[i]), x2 = aos_bf16_to_f32(src[i + half]);
      if (bias) {
        x1 = x1 + bias[h * p.hd + i];
        x2 = x2 + bias[h * p.hd + i + half];
      }
      const float c = cs[i], s = sn[i];
      const float r1 = x1 * c - x2 * s, r2 = x1 * s + x2 * c;
      if (isq) {
        float *dst = p.qr + ((size_t)t * p.nh + h) * p.hd;
        dst[i] = r1;
        dst[i + half] = r2;
      } else {
        uint16_t *dst = p.kc + ((size_t)h * p.max_seq + pos) * p.hd;
        const uint16_t b1 = aos_f32_to_bf16(r1), b2 = aos_f32_to_bf16(r2);
        dst[i] = b1;
        dst[i + half] = b2;
        if (bf16_nonfinite(b1) || bf16_nonfinite(b2)) *p.nonfinite = 1u;
      }
    } else {
      const int idx = w - nq - nk;
      const int h = idx / p.hd, d = idx - h * p.hd;
      float v = aos_bf16_to_f32(p.v[(size_t)t * nv + idx]);
      if (p.bv) v = v + p.bv[idx];
      const uint16_t b = aos_f32_to_bf16(v);
      p.vc[((size_t)h * p.max_seq + pos) * p.hd + d] = b;
      if (bf16_nonfinite(b)) *p.nonfinite = 1u;
    }
  }
}

/* ---- attention ---------------------------------------------------------------------------------- */

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, aos_shfl_f(v, (int)(threadIdx.x ^ o)));
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = v + aos_shfl_f(v, (int)(threadIdx.x ^ o));
  return v;
}

/* One wave (attn_wave): positions [split * chunk, min(+chunk, visible)) of token t for head h, in blocks of
 * 64. Phase 1 puts one position on each lane: its key row (hd <= 64 * DPL) is loaded whole, then
 * the score q . k is formed in order over d. Phase 2 puts one or two 32-bit words of the value row
 * (two dimensions each) on each lane and adds p . v over the block's positions in order. A
 * block's key rows and its first PB value rows are loaded before anything waits on memory (the
 * query is staged into LDS behind them), so a block costs about one memory round trip. */
constexpr int ATTN_MAX_SPLITS = 1024;
constexpr int MERGE_B = 16;

/* RoPE of one pair (x1, x2) = (x[i], x[i + hd/2]) at position pos, as the separate RoPE kernel
 * computes it. */
__device__ __forceinline__ void rope_pair(float x1, float x2, float fpos, float invf, float &r1, float &r2) {
  const float ang = fpos * invf;
  const float c = cosf(ang), s = sinf(ang);
  r1 = x1 * c - x2 * s;
  r2 = x1 * s + x2 * c;
}

template <int DPL>
__device__ void attn_merge(const aos_attn_params &p, int h, int t, int lane, float *fs, float *lf);

/* qs [hd] and ps [64]: the wave's LDS; kcur, vcur [hd / 2]: the current key (bf16 pairs) and value, with
 * rope_fused. WHOLE: all visible positions, no splits, queries rotated already (p.chunk and p.splits are
 * not read). */
template <int DPL, bool WHOLE>
__device__ __forceinline__ void attn_wave(const aos_attn_params &p, int split, int h, int t, int lane, float *qs,
                                          float *ps, uint32_t *kcur, uint32_t *vcur) {
  constexpr int NC = 8 * DPL;            /* 16-byte chunks of the longest key row */
  constexpr int NW = (DPL + 1) / 2;      /* value words per lane */
  constexpr int PB = DPL > 2 ? 32 : 64;  /* value rows loaded per batch */
  const int hd = p.hd, hw = hd / 2, kvh = h / (p.nh / p.nkv);
  const int visible = p.offset + t + 1;
  const int beg = WHOLE ? 0 : split * p.chunk;
  const int end = WHOLE ? visible : min(beg + p.chunk, visible);
  const float *q = p.q + ((size_t)t * p.nh + h) * hd;
  /* rope_fused: this token's own key and value are formed here, not read from the cache */
  const bool rope_fused = !WHOLE && p.rope_fused;
  const int cur = p.offset + t;
  const bool has_cur = rope_fused && beg <= cur && cur < end;
  const uint16_t *kbase = p.kc + (size_t)kvh * p.max_seq * hd;
  const uint32_t *vbase = (const uint32_t *)(p.vc + (size_t)kvh * p.max_seq * hd);
  float m = -__builtin_inff(), l = 0.0f, acc[2 * NW];
#pragma unroll
  for (int j = 0; j < 2 * NW; ++j) acc[j] = 0.0f;
  int wi[NW];
#pragma unroll
  for (int jw = 0; jw < NW; ++jw) {
    const int w = lane + 64 * jw;
    wi[jw] = w < hw ? w : 0;
  }
  /* rope_fused: the token's query pairs (and, in the split holding its position, its key pairs
   * and value words) with their biases and frequencies are loaded first, so that they share the
   * memory round trip of the first block's key and value rows; pair w = lane + 64 jw */
  float cq1[NW], cq2[NW], cf[NW], ck1[NW], ck2[NW], cv0[NW], cv1[NW];
  if (rope_fused) {
    const uint16_t *qb = p.qb + (size_t)h * hd;
    const uint16_t *kb = p.kb + (size_t)kvh * hd;
    const uint32_t *vb = (const uint32_t *)(p.vb + (size_t)kvh * hd);
#pragma unroll
    for (int jw = 0; jw < NW; ++jw) {
      const int w = wi[jw];
      cq1[jw] = aos_bf16_to_f32(qb[w]);
      cq2[jw] = aos_bf16_to_f32(qb[w + hw]);
      if (p.bq) {
        cq1[jw] = cq1[jw] + p.bq[h * hd + w];
        cq2[jw] = cq2[jw] + p.bq[h * hd + w + hw];
      }
      cf[jw] = p.inv_freq[w];
      ck1[jw] = ck2[jw] = cv0[jw] = cv1[jw] = 0.0f;
      if (has_cur) {
        ck1[jw] = aos_bf16_to_f32(kb[w]);
        ck2[jw] = aos_bf16_to_f32(kb[w + hw]);
        if (p.bk) {
          ck1[jw] = ck1[jw] + p.bk[kvh * hd + w];
          ck2[jw] = ck2[jw] + p.bk[kvh * hd + w + hw];
        }
        const uint32_t pr = vb[w];
        cv0[jw] = __builtin_bit_cast(float, pr << 16);
        cv1[jw] = __builtin_bit_cast(float, pr & 0xffff0000u);
        if (p.bv) {
          cv0[jw] = cv0[jw] + p.bv[kvh * hd + 2 * w];
          cv1[jw] = cv1[jw] + p.bv[kvh * hd + 2 * w + 1];
        }
      }
    }
  }
  for (int base = beg; base < end; base += 64) {
    const int pos = base + lane;
    const bool valid = pos < end;
    const int n = min(64, end - base);
    u32x4 kv[NC];
    {
      const u32x4 *kr = (const u32x4 *)(kbase + (size_t)(valid ? pos : base) * hd);
#pragma unroll
      for (int c = 0; c < NC; ++c) kv[c] = c < hd / 8 ? kr[c] : kv[0];
    }
    uint32_t vv[PB][NW];
#pragma unroll
    for (int u = 0; u < PB; ++u) {
      const int jj = u < n ? u : n - 1;
#pragma unroll
      for (int jw = 0; jw < NW; ++jw) vv[u][jw] = vbase[(size_t)(base + jj) * hw + wi[jw]];
    }
    if (base == beg) {
      if (rope_fused) {
        const float fpos = (float)cur;
        /* the key and value as the cache holds them (bf16); the first head of the group
         * appends them */
        const bool writer = has_cur && h % (p.nh / p.nkv) == 0;
        uint16_t *kdst = p.kc + ((size_t)kvh * p.max_seq + cur) * hd;
        uint32_t *vdst = (uint32_t *)(p.vc + ((size_t)kvh * p.max_seq + cur) * hd);
#pragma unroll
        for (int jw = 0; jw < NW; ++jw) {
          const int i = lane + 64 * jw;
          if (i < hw) {
            rope_pair(cq1[jw], cq2[jw], fpos, cf[jw], qs[i], qs[i + hw]);
            if (has_cur) {
              float r1, r2;
              rope_pair(ck1[jw], ck2[jw], fpos, cf[jw], r1, r2);
              const uint16_t b1 = aos_f32_to_bf16(r1), b2 = aos_f32_to_bf16(r2);
              ((uint16_t *)kcur)[i] = b1;
              ((uint16_t *)kcur)[i + hw] = b2;
              const uint32_t o = (uint32_t)aos_f32_to_bf16(cv0[jw]) | ((uint32_t)aos_f32_to_bf16(cv1[jw]) << 16);
              vcur[i] = o;
              if (writer) {
                kdst[i] = b1;
                kdst[i + hw] = b2;
                vdst[i] = o;
              }
            }
          }
        }
      } else {
        for (int d = lane; d < hd; d += 64) qs[d] = q[d];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    }
    if (has_cur && pos == cur) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (c < hd / 8) kv[c] = ((const u32x4 *)kcur)[c];
    }
    float s = -__builtin_inff();
    {
      float dot = 0.0f;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if (c < hd / 8) {
          const uint32_t wv[4] = {kv[c].x, kv[c].y, kv[c].z, kv[c].w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            dot = dot + qs[8 * c + 2 * e] * __builtin_bit_cast(float, wv[e] << 16);
            dot = dot + qs[8 * c + 2 * e + 1] * __builtin_bit_cast(float, wv[e] & 0xffff0000u);
          }
        }
      }
      if (valid) s = dot * p.scale;
    }
    const float mc = wave_max(s);
    const float mn = fmaxf(m, mc);
    const float alpha = expf(m - mn);
    const float pv = valid ? expf(s - mn) : 0.0f;
    l = l * alpha + wave_sum(pv);
    ps[lane] = pv;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
#pragma unroll
    for (int j = 0; j < 2 * NW; ++j) acc[j] = acc[j] * alpha;
    for (int j0 = 0; j0 < n; j0 += PB) {
      if (j0 > 0) {
#pragma unroll
        for (int u = 0; u < PB; ++u) {
          const int jj = j0 + u < n ? j0 + u : n - 1;
#pragma unroll
          for (int jw = 0; jw < NW; ++jw) vv[u][jw] = vbase[(size_t)(base + jj) * hw + wi[jw]];
        }
      }
      if (has_cur && cur >= base + j0 && cur < base + j0 + PB) { /* uniform */
        const int uc = cur - base - j0;
#pragma unroll
        for (int u = 0; u < PB; ++u)
          if (u == uc) {
#pragma unroll
            for (int jw = 0; jw < NW; ++jw) vv[u][jw] = vcur[wi[jw]];
          }
      }
#pragma unroll
      for (int u = 0; u < PB; ++u) {
        if (j0 + u < n) {
          const float pj = ps[j0 + u];
#pragma unroll
          for (int jw = 0; jw < NW; ++jw) {
            acc[2 * jw] = acc[2 * jw] + pj * __builtin_bit_cast(float, vv[u][jw] << 16);
            acc[2 * jw + 1] = acc[2 * jw + 1] + pj * __builtin_bit_cast(float, vv[u][jw] & 0xffff0000u);
          }
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    m = mn;
  }
  /* an infinity or NaN that this token appended: read back from LDS here, after the loop, whose schedule the
   * check in place cost 0.4 to 0.7 us (28 heads of 128, 220 positions: 10.7 us without it, 10.8 here, 11.1 and
   * 11.4 us there) */
  if constexpr (!WHOLE) {
    if (has_cur && h % (p.nh / p.nkv) == 0) {
      for (int i = lane; i < hd; i += 64) {
        const uint32_t w = i < hw ? kcur[i] : vcur[i - hw];
        if (bf16_nonfinite(w) || bf16_nonfinite(w >> 16)) *p.nonfinite = 1u;
      }
    }
  }
  if (WHOLE || p.splits == 1) {
    uint32_t *o = (uint32_t *)(p.out + (size_t)t * p.nh * hd + (size_t)h * hd);
#pragma unroll
    for (int jw = 0; jw < NW; ++jw) {
      const int w = lane + 64 * jw;
      if (w < hw)
        o[w] = (uint32_t)aos_f32_to_bf16(acc[2 * jw] / l) | ((uint32_t)aos_f32_to_bf16(acc[2 * jw + 1] / l) << 16);
    }
    return;
  }
  if constexpr (!WHOLE) {
    float *pp = p.part + (((size_t)t * p.nh + h) * p.splits + split) * (hd + 2);
    if (!p.counters) {
#pragma unroll
      for (int jw = 0; jw < NW; ++jw) {
        const int w = lane + 64 * jw;
        if (w < hw) {
          pp[2 * w] = acc[2 * jw];
          pp[2 * w + 1] = acc[2 * jw + 1];
        }
      }
      if (lane == 0) {
        pp[hd] = m;
        pp[hd + 1] = l;
      }
      return;
    }
    /* device-scope stores, then the arrival count; the last split of (token, head) merges */
#pragma unroll
    for (int jw = 0; jw < NW; ++jw) {
      const int w = lane + 64 * jw;
      if (w < hw) {
        aos_publish(pp + 2 * w, acc[2 * jw]);
        aos_publish(pp + 2 * w + 1, acc[2 * jw + 1]);
      }
    }
    if (lane == 0) {
      aos_publish(pp + hd, m);
      aos_publish(pp + hd + 1, l);
    }
    uint32_t *ctr = p.counters + (size_t)t * p.nh + h;
    uint32_t old = 0;
    if (lane == 0) old = aos_arrive(ctr);
    old = aos_shfl(old, 0);
    if (old != (uint32_t)p.splits - 1u) return;
    if (lane == 0) aos_reset(ctr);
    __shared__ float fs[1024], lf[1024];
    attn_merge<DPL>(p, h, t, lane, fs, lf);
  }
}

template <int DPL>
__global__ void __launch_bounds__(64) aos_attn_kernel(aos_attn_params p) {
  __shared__ float qs[AOS_ATTN_MAX_HD];
  __shared__ float ps[64];
  __shared__ __attribute__((aligned(16))) uint32_t kcur[AOS_ATTN_MAX_HD / 2];
  __shared__ uint32_t vcur[AOS_ATTN_MAX_HD / 2];
  attn_wave<DPL, false>(p, blockIdx.x, blockIdx.y, blockIdx.z, threadIdx.x, qs, ps, kcur, vcur);
}

/* Merge of the splits of (head, token), in split order. A split past the visible positions has
 * max -inf and sum 0 and adds nothing. The splits' maxima and sums are read one split per lane;
 * the partial outputs 16 splits at a time. */

template <int DPL>
__device__ void attn_merge(const aos_attn_params &p, int h, int t, int lane, float *fs, float *lf) {
  const int hd = p.hd, S = p.splits;
  const bool co = p.counters != nullptr; /* partials of this launch: device-scope loads */
  auto ld = [&](const float *a) { return co ? aos_collect(a) : *a; };
  const float *pp = p.part + ((size_t)t * p.nh + h) * S * (hd + 2);
  float mloc = -__builtin_inff();
  for (int s = lane; s < S; s += 64) mloc = fmaxf(mloc, ld(pp + (size_t)s * (hd + 2) + hd));
  const float M = wave_max(mloc);
  for (int s = lane; s < S; s += 64) {
    const float ms = ld(pp + (size_t)s * (hd + 2) + hd), ls = ld(pp + (size_t)s * (hd + 2) + hd + 1);
    const bool live = ls > 0.0f;
    const float f = live ? expf(ms - M) : 0.0f;
    fs[s] = f;
    lf[s] = live ? ls * f : 0.0f;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  float L = 0.0f, acc[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) acc[j] = 0.0f;
  int di[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) {
    const int d = lane + 64 * j;
    di[j] = d < hd ? d : 0;
  }
  for (int s0 = 0; s0 < S; s0 += MERGE_B) {
    float qv[MERGE_B][DPL];
#pragma unroll
    for (int u = 0; u < MERGE_B; ++u) {
      const int s = s0 + u < S ? s0 + u : S - 1;
#pragma unroll
      for (int j = 0; j < DPL; ++j) qv[u][j] = ld(pp + (size_t)s * (hd + 2) + di[j]);
    }
#pragma unroll
    for (int u = 0; u < MERGE_B; ++u) {
      if (s0 + u < S && fs[s0 + u] != 0.0f) {
        const float f = fs[s0 + u];
        L = L + lf[s0 + u];
#pragma unroll
        for (int j = 0; j < DPL; ++j) acc[j] = acc[j] + qv[u][j] * f;
      }
    }
  }
  uint16_t *o = p.out + (size_t)t * p.nh * hd + (size_t)h * hd;
#pragma unroll
  for (int j = 0; j < DPL; ++j) {
    const int d = lane + 64 * j;
    if (d < hd) o[d] = aos_f32_to_bf16(acc[j] / L);
  }
}

template <int DPL>
__global__ void __launch_bounds__(64) aos_attn_merge_kernel(aos_attn_params p) {
  __shared__ float fs[ATTN_MAX_SPLITS], lf[ATTN_MAX_SPLITS];
  attn_merge<DPL>(p, blockIdx.x, blockIdx.y, threadIdx.x, fs, lf);
}

/* ---- attention of a prompt on the matrix cores ------------------------------------------------ */

/* Four waves cover 128 tokens of one head, each wave 32 (one per MFMA column); the keys and values of
 * the causal range go by in tiles of 64 positions, straight from memory to a two-stage LDS ring the
 * waves share (64 KB: two workgroups per CU, so one's softmax runs under the other's MFMAs).
 *
 * Scores: S^T[key][token] = K . Q^T. The keys are bfloat16; the float32 query is held as three
 * bfloat16 pieces (the top 8, the next 8 and the last 8 bits of its significand, by truncation: the
 * split is exact), so three MFMAs give the float32 products, summed in float32. The row of K on MFMA
 * row r is key swap23(r) (bits 2 and 3 exchanged), which puts on lane (token, half c), register
 * 8 s + e, the score of key 16 s + 8 c + e: the B operand layout of the second product, so the
 * probabilities never cross lanes.
 *
 * Output: O^T[d][token] = V^T . P^T, the float32 probabilities split the same way (three MFMAs, P
 * exact); V^T fragments come from the row-major value tile through ds_read_b64_tr_b16 (a 16-lane
 * group reads 4 keys x 16 dimensions, lane l receiving column l of the 4 rows). Online softmax in
 * float32, one token per lane pair; the output is rescaled only where a maximum grew.
 *
 * LDS chunks (16 bytes) are swizzled so that neither read conflicts: key rows by their row, value rows
 * by the two row bits a transposed read spans.
 *
 * Bound by the matrix cores (three MFMAs for each of the plain bfloat16 products) and the float32
 * exponentials and splits between them. One layer of 1900 tokens, 28 heads of 128, 4 key/value heads: 128 us
 * (26 GFLOP of products over the causal half; 82 GFLOP executed, with the pieces and the masked parts of the
 * edge tiles: 640 TFLOP/s) against 2452 us for the wave per (token, head), which reads every visible key and
 * value row once per token. */
constexpr int PA_BQ = 128; /* tokens per workgroup */
constexpr int PA_BK = 64;  /* positions per tile */

/* float32 pair -> its top 8, next 8 and last 8 significand bits as packed bfloat16 pairs */
__device__ __forceinline__ void split3(float a, float b, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
  const uint32_t ua = __builtin_bit_cast(uint32_t, a), ub = __builtin_bit_cast(uint32_t, b);
  hi = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
  const float ra = a - __builtin_bit_cast(float, ua & 0xffff0000u);
  const float rb = b - __builtin_bit_cast(float, ub & 0xffff0000u);
  const uint32_t va = __builtin_bit_cast(uint32_t, ra), vb = __builtin_bit_cast(uint32_t, rb);
  mid = __builtin_amdgcn_perm(vb, va, 0x07060302u);
  const float sa = ra - __builtin_bit_cast(float, va & 0xffff0000u);
  const float sb = rb - __builtin_bit_cast(float, vb & 0xffff0000u);
  lo = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, sb), __builtin_bit_cast(uint32_t, sa), 0x07060302u);
}

/* e^x for x <= 0 through the hardware's 2^t: t = x log2(e) rounded, its rounding error and the
 * constant's low part put back to first order. x below -200 (and -infinity) gives 0; NaN stays NaN. */
__device__ __forceinline__ float exp_neg(float x) {
  const float L2E = 1.44269502f, L2E_LO = 1.92596303e-8f, LN2 = 0.693147182f;
  x = x < -200.0f ? -200.0f : x;
  const float t = x * L2E;
  const float r = fmaf(x, L2E_LO, fmaf(x, L2E, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, r * LN2, e);
}

/* Group of DMA loads of a tile: LDS bytes base + 1024 b + 16 lane of blocks b = 4 k + wave; v[k] is the
 * lane's byte offset in the first tile. Positions past the resource's end read as zeros. */
template <int N>
__device__ __forceinline__ void pa_dma(const uint16_t *src, int bytes, unsigned char *dst, int wave, const int *v,
                                       int tile_bytes) {
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)src, (short)0, bytes, 0x00020000);
#pragma unroll
  for (int k = 0; k < N; ++k)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rs, (__attribute__((address_space(3))) void *)(dst + (4 * k + wave) * 1024), 16, v[k], tile_bytes, 0, 0);
}

/* A cache that holds an infinity or a NaN takes the wave per (token, head) instead (attn_wave): products of
 * such a value with the zero pieces of a split would be NaN where the float32 product is not. The rows, the
 * longest first, are dealt over the waves of pa_min_wgs workgroups, which every grid has: the 256 CUs times
 * the workgroups that fit on one, as many waves as the registers of aos_attn_kernel allow too. Those past the
 * token tiles end at once when the cache is finite. 28 heads of 128, 1900 tokens: 2372 us, against 2303 us as
 * aos_attn_kernel; 74 tokens after 2000 positions 373 against 344 us. */
constexpr int pa_min_wgs(int hd) { return 256 * (hd == 64 ? 3 : 2); }

template <int HD>
__global__ void __launch_bounds__(256, 2) aos_attn_prefill_kernel(aos_attn_params p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  constexpr int KS = HD / 16, DB = HD / 32, ROWB = HD * 2, TB = PA_BK * ROWB, NB = TB / 1024 / 4, CPR = HD / 8;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 31, c = lane >> 5;
  const int h = blockIdx.x, kvh = h / (p.nh / p.nkv);
  if (*p.nonfinite) { /* uniform */
    constexpr int NWG = pa_min_wgs(HD); /* (more would wait for these, and then work alone) */
    const int wg = (int)(blockIdx.y * gridDim.x + blockIdx.x), rows = p.T * p.nh;
    if (wg >= NWG) return;
    float *ws = (float *)smem + wave * (HD + 64);
    for (int r = wg * 4 + wave; r < rows; r += 4 * NWG)
      attn_wave<HD / 64, true>(p, 0, r % p.nh, p.T - 1 - r / p.nh, lane, ws, ws + HD, nullptr, nullptr);
    return;
  }
  const int q0 = ((p.T - 1) / PA_BQ - (int)blockIdx.y) * PA_BQ; /* the longest ranges first */
  if (q0 < 0) return;
  const int row = q0 + 32 * wave + i;
  const int first = p.offset + q0 + 32 * wave; /* the wave's first position */
  const int kend = p.offset + (q0 + PA_BQ < p.T ? q0 + PA_BQ : p.T);
  const int ntiles = (kend + PA_BK - 1) / PA_BK;
  const uint16_t *kb = p.kc + (size_t)kvh * p.max_seq * HD;
  const uint16_t *vb = p.vc + (size_t)kvh * p.max_seq * HD;

  /* LDS chunk slot of (row, chunk): keys slot = chunk ^ kx(row), values slot = chunk ^ vx(row) */
  auto kx = [](int r) { return HD == 128 ? (r & 15) : ((r >> 1) & 7); };
  auto vx = [](int r) {
    return HD == 128 ? 2 * ((r & 3) | (((r >> 3) & 1) << 2)) : 2 * (((r >> 1) & 1) | (((r >> 3) & 1) << 1));
  };
  int kv_off[NB], vv_off[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    const int slot = (4 * k + wave) * 64 + lane, r = slot / CPR, sl = slot % CPR;
    kv_off[k] = r * ROWB + ((sl ^ kx(r)) << 4);
    vv_off[k] = r * ROWB + ((sl ^ vx(r)) << 4);
  }
  auto dma = [&](int kt) {
    unsigned char *st = smem + (kt & 1) * 2 * TB;
    pa_dma<NB>(kb, kend * ROWB, st, wave, kv_off, kt * TB);
    pa_dma<NB>(vb, kend * ROWB, st + TB, wave, vv_off, kt * TB);
  };
  dma(0);

  /* the token's query pieces: B operand, K elements 16 ks + 8 c .. +7 */
  u32x4 qf[KS][3];
  {
    const float *q = p.q + ((size_t)(row < p.T ? row : p.T - 1) * p.nh + h) * HD + 8 * c;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float4 a = *(const float4 *)(q + 16 * ks), b = *(const float4 *)(q + 16 * ks + 4);
      const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t hi, mid, lo;
        split3(v[2 * e], v[2 * e + 1], hi, mid, lo);
        qf[ks][0][e] = hi;
        qf[ks][1][e] = mid;
        qf[ks][2][e] = lo;
      }
    }
  }
  /* A operand row i of a 32-key block is key swap23(i) */
  const int krow = (i & ~12) | ((i & 4) << 1) | ((i & 8) >> 1);
  const int kbase = krow * ROWB + ((c ^ kx(krow)) << 4); /* chunk 2 ks + c: ^ (ks << 5) */
  /* transposed value reads: 16-lane group (c, g) takes rows 8 c + 4 qq + w / 4 of a 16-key step,
   * bytes 64 db + 32 g + 8 (w % 4) of the row */
  const int w = lane & 15, g = (lane >> 4) & 1;
  int vbase[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    const int r = 8 * c + (w >> 2);
    vbase[db] = TB + r * ROWB + (((4 * db + 2 * g + ((w & 3) >> 1)) ^ vx(r)) << 4) + 8 * (w & 1);
  }

  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = f32x16{};
  float m = -__builtin_inff(), l = 0.0f; /* l: this lane's half of the token's sum */
  for (int kt = 0; kt < ntiles; ++kt) {
    aos_mem_wait(); /* tile kt, issued a tile ago */
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); /* and every wave is past tile kt - 1 */
    if (kt + 1 < ntiles) dma(kt + 1);
    const int k0 = kt * PA_BK;
    if (k0 > first + 31) continue; /* uniform: every key is later than the wave's tokens */
    const unsigned char *st = smem + (kt & 1) * 2 * TB;
    f32x16 s[2] = {f32x16{}, f32x16{}};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 a0 = *(const u32x4 *)(st + (kbase ^ (ks << 5)));
      const u32x4 a1 = *(const u32x4 *)(st + (kbase ^ (ks << 5)) + 32 * ROWB);
#pragma unroll
      for (int pc = 2; pc >= 0; --pc) {
        s[0] = aos_mfma32(a0, qf[ks][pc], s[0]);
        s[1] = aos_mfma32(a1, qf[ks][pc], s[1]);
      }
    }
    const bool edge = k0 + PA_BK - 1 > first; /* uniform */
    const int last = p.offset + row;          /* the token's own position */
    float mx = m;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        float x = s[b][v] * p.scale;
        if (edge && k0 + 32 * b + 16 * (v >> 3) + 8 * c + (v & 7) > last) x = -__builtin_inff();
        s[b][v] = x;
        mx = fmaxf(mx, x);
      }
    mx = fmaxf(mx, aos_shfl_f(mx, lane ^ 32));
    if (__ballot(mx > m)) {
      const float alpha = m == mx ? 1.0f : exp_neg(m - mx);
      l = l * alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[db][v] = o[db][v] * alpha;
      m = mx;
    }
#pragma unroll
    for (int sp = 0; sp < 4; ++sp) {
      u32x4 pf[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float pa = exp_neg(s[sp >> 1][8 * (sp & 1) + 2 * e] - m);
        const float pb = exp_neg(s[sp >> 1][8 * (sp & 1) + 2 * e + 1] - m);
        l = l + pa;
        l = l + pb;
        uint32_t hi, mid, lo;
        split3(pa, pb, hi, mid, lo);
        pf[0][e] = hi;
        pf[1][e] = mid;
        pf[2][e] = lo;
      }
      u32x4 a[DB];
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const __attribute__((address_space(3))) unsigned char *vt =
            (const __attribute__((address_space(3))) unsigned char *)(st + vbase[db] + 16 * sp * ROWB);
        const s16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)vt);
        const s16x4 x1 =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(vt + 4 * ROWB));
        const u32x2 y0 = __builtin_bit_cast(u32x2, x0), y1 = __builtin_bit_cast(u32x2, x1);
        a[db] = u32x4{y0.x, y0.y, y1.x, y1.y};
      }
#pragma unroll
      for (int pc = 2; pc >= 0; --pc)
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] = aos_mfma32(a[db], pf[pc], o[db]);
    }
  }
  aos_mem_wait();
  if (row >= p.T) return;
  l = l + aos_shfl_f(l, lane ^ 32);
  uint16_t *out = p.out + ((size_t)row * p.nh + h) * HD;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      u32x2 r;
      r.x = (uint32_t)aos_f32_to_bf16(o[db][4 * q] / l) | ((uint32_t)aos_f32_to_bf16(o[db][4 * q + 1] / l) << 16);
      r.y = (uint32_t)aos_f32_to_bf16(o[db][4 * q + 2] / l) | ((uint32_t)aos_f32_to_bf16(o[db][4 * q + 3] / l) << 16);
      *(u32x2 *)(out + 32 * db + 8 * q + 4 * c) = r;
    }
}

template <int HD>
int launch_attn_prefill(const aos_attn_params *p, const aos_launch_ctx *ctx) {
  const int tiles = (p->T + PA_BQ - 1) / PA_BQ, least = (pa_min_wgs(HD) + p->nh - 1) / p->nh;
  AOS_LAUNCH(ctx, aos_attn_prefill_kernel<HD>, dim3(p->nh, tiles > least ? tiles : least), dim3(256),
             4 * PA_BK * HD * 2, *p);
  return (int)hipGetLastError();
}

template <int DPL>
int launch_attn(const aos_attn_params *p, const aos_launch_ctx *ctx) {
  AOS_LAUNCH(ctx, aos_attn_kernel<DPL>, dim3(p->splits, p->nh, p->T), dim3(64), 0, *p);
  if (p->splits > 1 && !p->counters) AOS_LAUNCH(ctx, aos_attn_merge_kernel<DPL>, dim3(p->nh, p->T), dim3(64), 0, *p);
  return (int)hipGetLastError();
}

}  // namespace

extern "C" int aos_launch_embed(const aos_embed_params *p, const aos_launch_ctx *ctx) {
  if (p->H % 64) return (int)hipErrorInvalidValue;
  AOS_LAUNCH(ctx, aos_embed_kernel, dim3((p->H / 8 + 255) / 256, p->T), dim3(256), 0, *p);
  return (int)hipGetLastError();
}

extern "C" int aos_launch_norm(const aos_norm_params *p, const aos_launch_ctx *ctx) {
  if (p->H % 64 || p->H > 4 * 1024 * NORM_J) return (int)hipErrorInvalidValue;
  AOS_LAUNCH(ctx, aos_norm_kernel, dim3(p->T), dim3(1024), 0, *p);
  return (int)hipGetLastError();
}

extern "C" int aos_launch_rope(const aos_rope_params *p, const aos_launch_ctx *ctx) {
  if (!p->nonfinite || p->hd > AOS_ATTN_MAX_HD) return (int)hipErrorInvalidValue;
  const int items = p->nh * (p->hd / 2) + p->nkv * (p->hd / 2) + p->nkv * p->hd;
  /* parts of a token: as many as about 1024 workgroups allow (few tokens), so that none loops long */
  int parts = p->T < 1024 ? 1024 / p->T : 1;
  if (parts > (items + 255) / 256) parts = (items + 255) / 256;
  AOS_LAUNCH(ctx, aos_rope_kernel, dim3(parts, p->T), dim3(256), 0, *p);
  return (int)hipGetLastError();
}

/* The prompt kernel's shapes: its head_dims, and a head's cache within a 32-bit byte offset (a tile past
 * the end included). */
extern "C" int aos_attn_prefill_fits(int hd, int max_seq) {
  return (hd == 64 || hd == 128) && ((long long)max_seq + 2 * PA_BK) * hd * 2 < (1ll << 31);
}

extern "C" int aos_launch_attention(const aos_attn_params *p, const aos_launch_ctx *ctx) {
  if (p->hd % 8 || p->hd > AOS_ATTN_MAX_HD || p->splits < 1 || p->splits > ATTN_MAX_SPLITS || p->chunk % 64)
    return (int)hipErrorInvalidValue;
  if (!p->nonfinite) return (int)hipErrorInvalidValue;
  if (p->prefill) {
    if (p->rope_fused || !aos_attn_prefill_fits(p->hd, p->max_seq)) return (int)hipErrorInvalidValue;
    return p->hd == 64 ? launch_attn_prefill<64>(p, ctx) : launch_attn_prefill<128>(p, ctx);
  }
  if (p->rope_fused && (p->T != 1 || !p->qb || !p->kb || !p->vb || !p->inv_freq)) return (int)hipErrorInvalidValue;
  if (p->hd <= 64) return launch_attn<1>(p, ctx);
  if (p->hd <= 128) return launch_attn<2>(p, ctx);
  return launch_attn<4>(p, ctx);
}

AOS_DEFINE_SPIN_SETTER(aos_spin_setter_model)
