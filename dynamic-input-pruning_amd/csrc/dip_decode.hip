// dip_decode.hip — the one-token decode steps of a Qwen3 decoder layer around
// the DIP MLP: residual add + RMSNorm, q/k RMSNorm + rotary embedding + key /
// value cache write, and grouped-query attention of the token over the cache.
//
// The reference runs these steps through transformers' Qwen3 modules with
// PyTorch ops (the model its loader builds, dip_stream_predispatch.py:218-289;
// transformers' modeling_qwen3: Qwen3RMSNorm.forward, apply_rotary_pos_emb,
// Qwen3Attention.forward, Qwen3DecoderLayer.forward).  Where those modules
// round to bf16 these kernels round at the same points:
//   RMSNorm   y = bf16(w * bf16(x * rsqrt(mean(x^2) + eps)))  (fp32 mean)
//   residual  h = bf16(h + a)
//   rotary    q' = bf16(bf16(q * cos) + bf16(rotate_half(q) * sin))
// The attention keeps scores, softmax and the weighted value sum in fp32 and
// rounds its output once (torch's fused attention kernels round in between,
// so the two agree to bf16 rounding, not bit for bit).
//
// Every kernel here is latency-bound (a few KB per token, except attention
// over a long cache); each is one launch of a handful of workgroups.
#include "dip_common.h"
#include "dip_internal.h"

namespace dip {
namespace {

constexpr int kNormThreads = 256;
constexpr int kNormVecs = 4;              // 16-byte vectors per thread: n <= 8192
constexpr int kHeadDim = 128;
constexpr int kAttnChunk = 32;            // cache positions a wave takes at a time
constexpr int kPartFloats = 2 + kHeadDim; // m, l, acc[128] per (kv head, chunk, query head)

// Wave-wide reductions on DPP / permlane exchanges (no LDS round trips).
DIP_DEV float wave_sum(float v) { return group_sum<64>(v); }
DIP_DEV float wave_max(float v) { return group_max<64>(v); }

DIP_DEV float round_bf16(float v) { return bf16_to_f32(f32_to_bf16(v)); }

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

DIP_DEV bf16x8_t as_bf16x8(const uint4& v) {
  return __builtin_bit_cast(bf16x8_t, u32x4_t{v.x, v.y, v.z, v.w});
}

// h = bf16(h + add) when add is given; out = RMSNorm(h) * w.  One workgroup
// per row of n values (a decode step has one, a prompt one per token: 200 rows of
// 4096 values 4.7 us, where the module's six launches took about 30);
// thread t owns the 16-byte vectors t, t + 256, ... (8 values each), all
// loaded before anything is stored.
__global__ __launch_bounds__(kNormThreads) void add_rmsnorm_kernel(
    uint16_t* __restrict__ h, const uint16_t* __restrict__ add, const uint16_t* __restrict__ w,
    uint16_t* __restrict__ out, int n, float eps) {
  __shared__ float part[kNormThreads / 64];
  const int nv = n / 8;
  const size_t row = (size_t)blockIdx.x * n;
  h += row;
  out += row;
  if (add) add += row;
  uint4 hv[kNormVecs], av[kNormVecs], wv[kNormVecs];
#pragma unroll
  for (int j = 0; j < kNormVecs; ++j) {
    const int c = threadIdx.x + j * kNormThreads;
    hv[j] = av[j] = wv[j] = make_uint4(0, 0, 0, 0);
    if (c < nv) {
      hv[j] = reinterpret_cast<const uint4*>(h)[c];
      av[j] = add ? reinterpret_cast<const uint4*>(add)[c] : make_uint4(0, 0, 0, 0);
      wv[j] = reinterpret_cast<const uint4*>(w)[c];
    }
  }
  float x[kNormVecs][8];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < kNormVecs; ++j) {
    const int c = threadIdx.x + j * kNormThreads;
    const uint32_t hw[4] = {hv[j].x, hv[j].y, hv[j].z, hv[j].w};
    const uint32_t aw[4] = {av[j].x, av[j].y, av[j].z, av[j].w};
    uint32_t nw[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float lo = bf16_to_f32(hw[e] & 0xFFFFu), hi = bf16_to_f32(hw[e] >> 16);
      if (add) {
        lo = round_bf16(lo + bf16_to_f32(aw[e] & 0xFFFFu));
        hi = round_bf16(hi + bf16_to_f32(aw[e] >> 16));
      }
      nw[e] = f32_to_bf16(lo) | (f32_to_bf16(hi) << 16);
      x[j][2 * e] = lo;
      x[j][2 * e + 1] = hi;
      if (c < nv) ss += lo * lo + hi * hi;
    }
    if (add && c < nv) reinterpret_cast<uint4*>(h)[c] = make_uint4(nw[0], nw[1], nw[2], nw[3]);
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < kNormThreads / 64; ++i) tot += part[i];
  const float r = rsqrtf(tot * (1.0f / (float)n) + eps);
#pragma unroll
  for (int j = 0; j < kNormVecs; ++j) {
    const int c = threadIdx.x + j * kNormThreads;
    if (c >= nv) continue;
    const uint32_t ww[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
    uint32_t ow[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t lo = f32_to_bf16(bf16_to_f32(ww[e] & 0xFFFFu) * round_bf16(x[j][2 * e] * r));
      const uint32_t hi =
          f32_to_bf16(bf16_to_f32(ww[e] >> 16) * round_bf16(x[j][2 * e + 1] * r));
      ow[e] = lo | (hi << 16);
    }
    reinterpret_cast<uint4*>(out)[c] = make_uint4(ow[0], ow[1], ow[2], ow[3]);
  }
}

// One wave per token and head of the fused q|k|v projection output, four heads
// to a workgroup (token t, at position *pos + t, or t where pos is null):
// q heads [0, nh) and k heads [nh, nh + nkv) get RMSNorm over the head and
// the rotary embedding at `pos`; q goes to q_out, k to the key cache; v heads
// [nh + nkv, nh + 2 nkv) are copied to the value cache.  Lane l holds
// dimensions 2l and 2l + 1; rotate_half pairs dimension d with d +- 64, which
// lives in lane l ^ 32.  Cache writes happen only for 0 <= pos < max_len.  200
// tokens, 32 / 8 heads 4.5 us (as module ops about 25 launches of 3 to 7 us).
constexpr int kRopeHeads = 4;

__global__ __launch_bounds__(64 * kRopeHeads) void qk_rope_cache_kernel(
    const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ q_w,
    const uint16_t* __restrict__ k_w, const uint16_t* __restrict__ cos_t,
    const uint16_t* __restrict__ sin_t, const int64_t* __restrict__ pos_p,
    uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_cache,
    uint16_t* __restrict__ v_cache, int nh, int nkv, int max_len, float eps) {
  const int head = blockIdx.y * kRopeHeads + (threadIdx.x >> 6);
  const int l = threadIdx.x & 63;
  if (head >= nh + 2 * nkv) return;
  const int64_t pos = (pos_p ? *pos_p : 0) + blockIdx.x;
  const bool pos_ok = pos >= 0 && pos < max_len;
  const uint32_t pair = reinterpret_cast<const uint32_t*>(
      qkv)[((size_t)blockIdx.x * (nh + 2 * nkv) + head) * 64 + l];
  if (head >= nh + nkv) {
    if (pos_ok)
      reinterpret_cast<uint32_t*>(v_cache)[((size_t)(head - nh - nkv) * max_len + pos) * 64 + l] =
          pair;
    return;
  }
  const bool is_q = head < nh;
  const uint32_t wp = reinterpret_cast<const uint32_t*>(is_q ? q_w : k_w)[l];
  const float x0 = bf16_to_f32(pair & 0xFFFFu), x1 = bf16_to_f32(pair >> 16);
  const float ss = wave_sum(x0 * x0 + x1 * x1);
  const float r = rsqrtf(ss * (1.0f / (float)kHeadDim) + eps);
  const uint32_t y0 = f32_to_bf16(bf16_to_f32(wp & 0xFFFFu) * round_bf16(x0 * r));
  const uint32_t y1 = f32_to_bf16(bf16_to_f32(wp >> 16) * round_bf16(x1 * r));
  // rotate_half: dims [0, 64) take -y[d + 64], dims [64, 128) take y[d - 64]
  float r0 = bf16_to_f32(__shfl_xor(y0, 32, 64));
  float r1 = bf16_to_f32(__shfl_xor(y1, 32, 64));
  if (l < 32) {
    r0 = -r0;
    r1 = -r1;
  }
  const size_t trow = (size_t)(pos_ok ? pos : 0) * 64 + l;
  const uint32_t cs = reinterpret_cast<const uint32_t*>(cos_t)[trow];
  const uint32_t sn = reinterpret_cast<const uint32_t*>(sin_t)[trow];
  const uint32_t o0 = f32_to_bf16(round_bf16(bf16_to_f32(y0) * bf16_to_f32(cs & 0xFFFFu)) +
                                  round_bf16(r0 * bf16_to_f32(sn & 0xFFFFu)));
  const uint32_t o1 = f32_to_bf16(round_bf16(bf16_to_f32(y1) * bf16_to_f32(cs >> 16)) +
                                  round_bf16(r1 * bf16_to_f32(sn >> 16)));
  const uint32_t o = o0 | (o1 << 16);
  if (is_q)
    reinterpret_cast<uint32_t*>(q_out)[((size_t)blockIdx.x * nh + head) * 64 + l] = o;
  else if (pos_ok)
    reinterpret_cast<uint32_t*>(k_cache)[((size_t)(head - nh) * max_len + pos) * 64 + l] = o;
}

// Attention over a long cache, pass 1.  The rows 0 .. pos are cut into
// attn_rows_per_wave rows per wave, 4 waves to a workgroup (split) and
// attn_splits splits per kv head at most, from pos itself: a cache that is
// mostly empty still spreads over the chip.  A wave walks its rows 32 at a
// time with a running (max, sum, value sum) per query head of the group:
//   * scores on bf16 MFMA (A = 16 cache rows, B = the q heads, exact products,
//     fp32 sums), both operands in memory order (slice j: lane quarter kb holds
//     dims 32 j + 8 kb ..), so one load covers 64 contiguous bytes of a row;
//   * softmax in fp32; the weights reach the value lanes through LDS;
//   * values in fp32 on the VALU: lane l holds dims 8 (l % 16) .. + 7 of rows
//     4 i + l / 16, a 128-bit load per four rows' worth of a wave.
// At the end the four lane groups and the four waves are merged in a fixed
// order and the split stores per query head its max, sum of exp and
// unnormalised value sum.  Bound by HBM: 64 query / 8 kv heads, 20011 rows
// (82 MB) 23 us, and 4.5 us for the merge of 63 splits.  (One wave and one
// partial per 32 rows: 26 us, and 60 us to merge 626 of them in series.)
constexpr int kAttnWaves = 4;
constexpr int kAttnMaxSplits = 256;

// Splits per kv head that fill the chip about twice over.
inline int attn_splits(int nkv, int max_len) {
  const int want = (2 * device_cus() + nkv - 1) / nkv;
  const int most = (max_len + kAttnChunk * kAttnWaves - 1) / (kAttnChunk * kAttnWaves);
  return max(1, min(min(want, most), kAttnMaxSplits));
}

// Cache rows attended at position pos: 0 .. pos, none before the first.
DIP_DEV int attn_rows(int64_t pos, int max_len) {
  return pos < 0 ? 0 : (pos < (int64_t)max_len ? (int)pos + 1 : max_len);
}

// Rows a wave takes of `rows`, never fewer than one chunk.
DIP_DEV int attn_rows_per_wave(int rows, int splits) {
  return max(kAttnChunk, (rows + splits * kAttnWaves - 1) / (splits * kAttnWaves));
}

template <int G>
__global__ __launch_bounds__(kAttnWaves * 64) void attn_partial_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache,
    const uint16_t* __restrict__ v_cache, const int64_t* __restrict__ pos_p,
    float* __restrict__ part, int max_len, int splits, float scale) {
  static_assert(G <= 16, "one MFMA column per query head");
  constexpr int GP = G <= 2 ? G : (G + 3) / 4 * 4;  // LDS row of weights
  __shared__ __align__(16) float ps[kAttnWaves][kAttnChunk][GP];
  __shared__ __align__(16) float fac[kAttnWaves][GP];
  __shared__ float wm[kAttnWaves][G], wl[kAttnWaves][G];
  __shared__ __align__(16) float wacc[kAttnWaves][G][kHeadDim];
  const int split = blockIdx.x, kvh = blockIdx.y;
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int l16 = l & 15, kb = l >> 4;
  const int64_t pos = *pos_p;
  const int rows = attn_rows(pos, max_len);
  const int rpw = attn_rows_per_wave(rows, splits);
  if (rows <= 0 || split >= (rows + kAttnWaves * rpw - 1) / (kAttnWaves * rpw)) return;
  const int r0 = min((split * kAttnWaves + wave) * rpw, rows), r1 = min(r0 + rpw, rows);
  const uint16_t* kbase = k_cache + (size_t)kvh * max_len * kHeadDim;
  const uint16_t* vbase = v_cache + (size_t)kvh * max_len * kHeadDim;

  uint4 bq[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    bq[j] = l16 < G ? reinterpret_cast<const uint4*>(q + (size_t)(kvh * G + l16) * kHeadDim)[4 * j + kb]
                    : make_uint4(0, 0, 0, 0);
  float acc[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[g][d] = 0.f;
  float m = -INFINITY, den = 0.f;  // of head l16

  for (int start = r0; start < r1; start += kAttnChunk) {
    const int npos = min(r1 - start, kAttnChunk);
    uint4 ka[2][4], vv[8];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ka[t][j] = make_uint4(0, 0, 0, 0);
        if (16 * t + l16 < npos)
          ka[t][j] = ldg_nt(reinterpret_cast<const uint4*>(
                                kbase + (size_t)(start + 16 * t + l16) * kHeadDim) + 4 * j + kb);
      }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      vv[i] = make_uint4(0, 0, 0, 0);
      if (4 * i + kb < npos)
        vv[i] = ldg_nt(reinterpret_cast<const uint4*>(
                           vbase + (size_t)(start + 4 * i + kb) * kHeadDim) + l16);
    }
    float sc[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      floatx4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(ka[t][j]), as_bf16x8(bq[j]), d, 0, 0,
                                                    0);
#pragma unroll
      for (int r = 0; r < 4; ++r) sc[t][r] = 16 * t + 4 * kb + r < npos ? d[r] * scale : -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[t][r]);
    mx = fmaxf(m, row_pair_max32(row_pair_max16(mx)));
    const float f = m == -INFINITY ? 0.f : expf(m - mx);  // what the sums so far are worth
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = sc[t][r] == -INFINITY ? 0.f : expf(sc[t][r] - mx);
        sum += e;
        if (l16 < G) ps[wave][16 * t + 4 * kb + r][l16] = e;
      }
    if (kb == 0 && l16 < G) fac[wave][l16] = f;
    den = den * f + row_pair_sum32(row_pair_sum16(sum));
    m = mx;
    // the wave's own LDS writes before its reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float fg = fac[wave][g];
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[g][d] *= fg;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t w[4] = {vv[i].x, vv[i].y, vv[i].z, vv[i].w};
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[2 * e] = bf16_to_f32(w[e] & 0xFFFFu);
        v[2 * e + 1] = __uint_as_float(w[e] & 0xFFFF0000u);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float pg = ps[wave][4 * i + kb][g];
#pragma unroll
        for (int d = 0; d < 8; ++d) acc[g][d] = fmaf(pg, v[d], acc[g][d]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }

  if (kb == 0 && l16 < G) {
    wm[wave][l16] = m;
    wl[wave][l16] = den;
  }
#pragma unroll
  for (int g = 0; g < G; ++g) {
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[g][d] = row_pair_sum32(row_pair_sum16(acc[g][d]));
    if (kb == (g & 3)) {
      float4* o = reinterpret_cast<float4*>(&wacc[wave][g][8 * l16]);
      o[0] = make_float4(acc[g][0], acc[g][1], acc[g][2], acc[g][3]);
      o[1] = make_float4(acc[g][4], acc[g][5], acc[g][6], acc[g][7]);
    }
  }
  __syncthreads();
  float* out = part + ((size_t)kvh * splits + split) * G * kPartFloats;
  for (int e = threadIdx.x; e < G * kHeadDim; e += kAttnWaves * 64) {
    const int g = e / kHeadDim, d = e % kHeadDim;
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) mx = fmaxf(mx, wm[w][g]);
    float s = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
      const float f = wl[w][g] > 0.f ? expf(wm[w][g] - mx) : 0.f;
      s = fmaf(f, wl[w][g], s);
      o = fmaf(f, wacc[w][g][d], o);
    }
    if (d == 0) {
      out[g * kPartFloats] = mx;
      out[g * kPartFloats + 1] = s;
    }
    out[g * kPartFloats + 2 + d] = o;
  }
}

// Attention, pass 2: one workgroup per query head.  The splits' weights first
// (one thread per split), then dimension d on the threads d, d + 128, ...,
// which sum every fourth split; the four sums are added in order.
__global__ __launch_bounds__(4 * kHeadDim) void attn_combine_kernel(
    const float* __restrict__ part, const int64_t* __restrict__ pos_p, uint16_t* __restrict__ out,
    int G, int max_len, int splits) {
  __shared__ float wgt[kAttnMaxSplits];
  __shared__ float red[8][2];
  __shared__ float so[4][kHeadDim];
  const int qh = blockIdx.x, kvh = qh / G, g = qh % G, tid = threadIdx.x;
  const int64_t pos = *pos_p;
  const int rows = attn_rows(pos, max_len);
  const int rpw = attn_rows_per_wave(max(rows, 1), splits);
  const int ns = rows <= 0 ? 0 : (rows + kAttnWaves * rpw - 1) / (kAttnWaves * rpw);
  const size_t stride = (size_t)G * kPartFloats;
  const float* base = part + (size_t)kvh * splits * stride + (size_t)g * kPartFloats;
  const int d = tid % kHeadDim, p = tid / kHeadDim;
  const float ms = tid < ns ? base[tid * stride] : -INFINITY;
  const float ls = tid < ns ? base[tid * stride + 1] : 0.f;
  float mx = wave_max(ms);
  if ((tid & 63) == 0) red[tid >> 6][0] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 8; ++w) mx = fmaxf(mx, red[w][0]);
  const float f = ls > 0.f ? expf(ms - mx) : 0.f;
  if (tid < kAttnMaxSplits) wgt[tid] = f;
  const float dsum = wave_sum(f * ls);
  if ((tid & 63) == 0) red[tid >> 6][1] = dsum;
  __syncthreads();
  float den = 0.f;
#pragma unroll
  for (int w = 0; w < 8; ++w) den += red[w][1];
  float o = 0.f;
  for (int s0 = p; s0 < ns; s0 += 32) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = base[min(s0 + 4 * u, ns - 1) * stride + 2 + d];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + 4 * u < ns) o = fmaf(wgt[s0 + 4 * u], v[u], o);
  }
  so[p][d] = o;
  __syncthreads();
  if (tid < kHeadDim / 2) {
    float r[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int c = 2 * tid + e;
      r[e] = ((so[0][c] + so[1][c]) + so[2][c]) + so[3][c];
    }
    reinterpret_cast<uint32_t*>(out)[(size_t)qh * 64 + tid] =
        f32_to_bf16(r[0] / den) | (f32_to_bf16(r[1] / den) << 16);
  }
}

// Norm + rotary + cache write + attention in one launch, for caches of at
// most kFusedMaxLen rows (4 waves up to 128 rows, 8 beyond, which walk the
// 32-row chunks 8 at a time): workgroup = HPW consecutive query heads of one kv
// head (group = nh / nkv query heads share it).  Every workgroup of a group
// normalises and rotates the group's k itself; only the group's first
// workgroup writes k and v to cache row pos (the others take this token's
// row from their own LDS copy, never from the cache).  One query head per
// workgroup spreads a layer over nh workgroups instead of nkv, which takes
// the per-head norm, rotary, softmax and value sums off one serial chain.
//   0. every load that does not need this token's k and v is issued first:
//      the q heads, k and v, the norm weights and the cos / sin rows into
//      LDS, each wave's first 32-row chunk of the cache into registers;
//   1. RMSNorm + rotary as qk_rope_cache_kernel; q into LDS as bf16, this
//      token's k and v into LDS (and into cache row pos);
//   2. wave w of NW takes the chunks w, w + NW, ...: the scores on bf16 MFMA
//      (v_mfma_f32_16x16x32_bf16, A = 16 cache rows, B = the q heads, exact
//      products, fp32 sums; row pos from LDS, not read back), softmax in
//      fp32, the value sum in fp32 on the VALU, merged into a running (max,
//      sum, value sum) per query head.  Keys and values come by 128-bit loads
//      that cover 64 (256) contiguous bytes of a row, the next chunk's while
//      this one is worked on;
//   3. the NW waves' partials are merged through LDS in a fixed order.
// Bound by what one CU can fetch: one workgroup per query head occupies 32 or
// 64 CUs of the chip, and each reads its kv head's rows.  64 / 8 heads, us in a graph: 121 rows of 128 7.1 -> 5.5, 101
// rows of 1024 7.3 -> 5.5, 501 rows 11.8 -> 10.0, 701 rows 15.3 -> 11.9, 1021
// rows 18.5 -> 14.7 (before: 16 waves without room for a chunk ahead, 16-byte
// pieces of 64 lines per key load, 4-byte value loads; two chunks ahead on 8
// waves 13.2 at 701 rows, 12 waves 12.5).  The split path takes 14.1 at 501 and
// 14.5 at 1021 rows, so one launch serves caches of up to 1024 rows.
constexpr int kFusedMaxLen = 1024;

template <int HPW, int NW>
__global__ __launch_bounds__(NW * 64) void attn_fused_kernel(
    const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ q_w,
    const uint16_t* __restrict__ k_w, const uint16_t* __restrict__ cos_t,
    const uint16_t* __restrict__ sin_t, const int64_t* __restrict__ pos_p,
    uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache, uint16_t* __restrict__ out,
    int nh, int nkv, int max_len, float eps, float scale) {
  static_assert(HPW <= 16, "one MFMA column per query head");
  static_assert(NW >= 4 && NW <= 16, "waves");
  constexpr int kThreads = NW * 64;
  const int group = nh / nkv;           // query heads per kv head
  const int h0 = blockIdx.x * HPW;      // this workgroup's first query head
  const bool writer = h0 % group == 0;  // the group's first workgroup writes the cache
  __shared__ __align__(16) uint32_t qb[16][64 + 4];   // q as bf16 pairs; heads >= HPW are 0
  __shared__ __align__(16) uint32_t kv_new[2][64];
  __shared__ uint32_t heads[HPW + 2][64];  // raw q heads | k | v
  __shared__ uint32_t tabs[4][64];         // q_w, k_w, cos row, sin row
  __shared__ float ps[NW][HPW][kAttnChunk];
  __shared__ float cm[NW][HPW], cl[NW][HPW];
  __shared__ float wm[NW][HPW], wl[NW][HPW];
  __shared__ __align__(16) float wacc[NW][HPW][kHeadDim];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kvh = h0 / group, l = threadIdx.x & 63;
  const int l16 = l & 15, kb = l >> 4;
  const int64_t pos = *pos_p;
  const bool pos_ok = pos >= 0 && pos < max_len;
  const int last = attn_rows(pos, max_len) - 1;  // the last attended row
  const int own = pos_ok ? (int)pos : -1;        // this token's row

  // 0. loads
  for (int i = threadIdx.x; i < (HPW + 2) * 64; i += kThreads) {
    const int hi = i >> 6;
    const int head = hi < HPW ? h0 + hi : (hi == HPW ? nh + kvh : nh + nkv + kvh);
    heads[hi][i & 63] = reinterpret_cast<const uint32_t*>(qkv)[(size_t)head * 64 + (i & 63)];
  }
  for (int i = threadIdx.x + HPW * 64; i < 16 * 64; i += kThreads) qb[i >> 6][i & 63] = 0u;
  if (wave < 4) {
    const size_t trow = (size_t)(pos_ok ? pos : 0) * 64 + l;
    const uint32_t* src = wave == 0 ? reinterpret_cast<const uint32_t*>(q_w) + l
                        : wave == 1 ? reinterpret_cast<const uint32_t*>(k_w) + l
                        : wave == 2 ? reinterpret_cast<const uint32_t*>(cos_t) + trow
                                    : reinterpret_cast<const uint32_t*>(sin_t) + trow;
    tabs[wave][l] = *src;
  }
  int start = wave * kAttnChunk;
  const char* kbase = reinterpret_cast<const char*>(k_cache + (size_t)kvh * max_len * kHeadDim);
  const char* vbase = reinterpret_cast<const char*>(v_cache + (size_t)kvh * max_len * kHeadDim);
  uint4 ka[2][4];  // A operand: cache rows st + 16 t + l16, slice j: dims 32 j + 8 kb .. + 7
  uint4 vv[8];     // values: rows st + 4 i + kb, dims 8 l16 .. + 7
  auto load_k = [&](int st) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = st + 16 * t + l16;
        ka[t][j] = make_uint4(0, 0, 0, 0);
        if (row <= last)
          ka[t][j] = *reinterpret_cast<const uint4*>(kbase + (uint32_t)(row * 256 + 64 * j + 16 * kb));
      }
  };
  auto load_v = [&](int st) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = st + 4 * i + kb;
      vv[i] = make_uint4(0, 0, 0, 0);
      if (row <= last)
        vv[i] = *reinterpret_cast<const uint4*>(vbase + (uint32_t)(row * 256 + 16 * l16));
    }
  };
  if (start <= last) {
    load_k(start);
    load_v(start);
  }
  __syncthreads();

  // 1. RMSNorm + rotary of the q heads and the k head; v and k to the cache
  for (int hi = wave; hi < HPW + 2; hi += NW) {
    const uint32_t pair = heads[hi][l];
    if (hi == HPW + 1) {
      kv_new[1][l] = pair;
      if (pos_ok && writer)
        reinterpret_cast<uint32_t*>(v_cache)[((size_t)kvh * max_len + pos) * 64 + l] = pair;
      continue;
    }
    const uint32_t wp = tabs[hi < HPW ? 0 : 1][l];
    const float x0 = bf16_to_f32(pair & 0xFFFFu), x1 = bf16_to_f32(pair >> 16);
    const float ss = wave_sum(x0 * x0 + x1 * x1);
    const float r = rsqrtf(ss * (1.0f / (float)kHeadDim) + eps);
    const uint32_t y0 = f32_to_bf16(bf16_to_f32(wp & 0xFFFFu) * round_bf16(x0 * r));
    const uint32_t y1 = f32_to_bf16(bf16_to_f32(wp >> 16) * round_bf16(x1 * r));
    float r0 = bf16_to_f32(__shfl_xor(y0, 32, 64));
    float r1 = bf16_to_f32(__shfl_xor(y1, 32, 64));
    if (l < 32) {
      r0 = -r0;
      r1 = -r1;
    }
    const uint32_t cs = tabs[2][l], sn = tabs[3][l];
    const uint32_t o0 = f32_to_bf16(round_bf16(bf16_to_f32(y0) * bf16_to_f32(cs & 0xFFFFu)) +
                                    round_bf16(r0 * bf16_to_f32(sn & 0xFFFFu)));
    const uint32_t o1 = f32_to_bf16(round_bf16(bf16_to_f32(y1) * bf16_to_f32(cs >> 16)) +
                                    round_bf16(r1 * bf16_to_f32(sn >> 16)));
    if (hi < HPW) {
      qb[hi][l] = o0 | (o1 << 16);
    } else {
      kv_new[0][l] = o0 | (o1 << 16);
      if (pos_ok && writer)
        reinterpret_cast<uint32_t*>(k_cache)[((size_t)kvh * max_len + pos) * 64 + l] =
            o0 | (o1 << 16);
    }
  }
  __syncthreads();

  // 2. B operand (q head l16, the same dims per slice) once; then the chunks
  uint4 bq[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) bq[j] = *reinterpret_cast<const uint4*>(&qb[l16][16 * j + 4 * kb]);
  float m[HPW], lsum[HPW], acc[HPW][8];
#pragma unroll
  for (int g = 0; g < HPW; ++g) {
    m[g] = -INFINITY;
    lsum[g] = 0.f;
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[g][d] = 0.f;
  }
  for (; start <= last; start += NW * kAttnChunk) {
    const int npos = min(last - start + 1, kAttnChunk);
    const int next = start + NW * kAttnChunk;
    const bool more = next <= last;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (start + 16 * t + l16 == own) {  // this token's row from LDS
#pragma unroll
        for (int j = 0; j < 4; ++j)
          ka[t][j] = *reinterpret_cast<const uint4*>(&kv_new[0][16 * j + 4 * kb]);
      }
    }
    // scores: lane (head l16, rows 4 kb + r of tile t)
    float sc[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      floatx4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(ka[t][j]), as_bf16x8(bq[j]), d, 0,
                                                    0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool ok = 16 * t + 4 * kb + r < npos;
        sc[t][r] = ok ? d[r] * scale : -INFINITY;
      }
    }
    // the next chunk's keys while this one's softmax and values run, and its
    // values behind them
    if (more) load_k(next);
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[t][r]);
    mx = row_pair_max32(row_pair_max16(mx));  // over the lanes of head l16
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = sc[t][r] == -INFINITY ? 0.f : expf(sc[t][r] - mx);
        sum += e;
        if (l16 < HPW) ps[wave][l16][16 * t + 4 * kb + r] = e;
      }
    sum = row_pair_sum32(row_pair_sum16(sum));
    if (kb == 0 && l16 < HPW) {
      cm[wave][l16] = mx;
      cl[wave][l16] = sum;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");

    // values: lane dims 8 l16 .. + 7 of every fourth row
    float c[HPW][8];
#pragma unroll
    for (int g = 0; g < HPW; ++g)
#pragma unroll
      for (int d = 0; d < 8; ++d) c[g][d] = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (start + 4 * i + kb == own)  // this token's row from LDS
        vv[i] = *reinterpret_cast<const uint4*>(&kv_new[1][4 * l16]);
      const uint32_t vw[4] = {vv[i].x, vv[i].y, vv[i].z, vv[i].w};
#pragma unroll
      for (int g = 0; g < HPW; ++g) {
        const float pg = ps[wave][g][4 * i + kb];  // 0 for rows past the end
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          c[g][2 * e] = fmaf(pg, bf16_to_f32(vw[e] & 0xFFFFu), c[g][2 * e]);
          c[g][2 * e + 1] = fmaf(pg, __uint_as_float(vw[e] & 0xFFFF0000u), c[g][2 * e + 1]);
        }
      }
    }
    if (more) load_v(next);
#pragma unroll
    for (int g = 0; g < HPW; ++g) {
      const float mc = cm[wave][g], lc = cl[wave][g];
      const float mn = fmaxf(m[g], mc);
      const float fo = expf(m[g] - mn), fn = expf(mc - mn);
      lsum[g] = lsum[g] * fo + lc * fn;
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[g][d] = acc[g][d] * fo + c[g][d] * fn;
      m[g] = mn;
    }
    __builtin_amdgcn_wave_barrier();
  }

  // 3. merge the waves in a fixed order
#pragma unroll
  for (int g = 0; g < HPW; ++g) {
    if (l == 0) {
      wm[wave][g] = m[g];
      wl[wave][g] = lsum[g];
    }
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[g][d] = row_pair_sum32(row_pair_sum16(acc[g][d]));
    if (kb == 0) {
      float4* o = reinterpret_cast<float4*>(&wacc[wave][g][8 * l16]);
      o[0] = make_float4(acc[g][0], acc[g][1], acc[g][2], acc[g][3]);
      o[1] = make_float4(acc[g][4], acc[g][5], acc[g][6], acc[g][7]);
    }
  }
  __syncthreads();
  for (int g = wave; g < HPW; g += NW) {
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) mx = fmaxf(mx, wm[w][g]);
    float den = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = wl[w][g] > 0.f ? expf(wm[w][g] - mx) : 0.f;
      den = fmaf(f, wl[w][g], den);
      o0 = fmaf(f, wacc[w][g][2 * l], o0);
      o1 = fmaf(f, wacc[w][g][2 * l + 1], o1);
    }
    reinterpret_cast<uint32_t*>(out)[((size_t)h0 + g) * 64 + l] =
        f32_to_bf16(o0 / den) | (f32_to_bf16(o1 / den) << 16);
  }
}

template <int G>
void launch_attention(const uint16_t* q, const uint16_t* kc, const uint16_t* vc, const int64_t* pos,
                      uint16_t* out, int nkv, int max_len, float scale, float* part,
                      hipStream_t stream) {
  const int splits = attn_splits(nkv, max_len);
  hipLaunchKernelGGL((attn_partial_kernel<G>), dim3(splits, nkv), dim3(kAttnWaves * 64), 0, stream,
                     q, kc, vc, pos, part, max_len, splits, scale);
  hipLaunchKernelGGL(attn_combine_kernel, dim3(nkv * G), dim3(4 * kHeadDim), 0, stream, part, pos,
                     out, G, max_len, splits);
}

}  // namespace
}  // namespace dip

using namespace dip;

extern "C" int dip_add_rmsnorm_rows(uint16_t* h, const uint16_t* add, const uint16_t* weight,
                                    uint16_t* out, int64_t rows, int64_t n, float eps,
                                    void* stream) {
  if (!h || !weight || !out) return DIP_ERR_NULL;
  if (n <= 0 || n % 8 != 0 || n > (int64_t)kNormThreads * kNormVecs * 8 || rows < 0 ||
      rows > INT32_MAX)
    return DIP_ERR_SHAPE;
  if (!(eps >= 0.f)) return DIP_ERR_ARG;
  if (!aligned16(h) || !aligned16(weight) || !aligned16(out) || (add && !aligned16(add)))
    return DIP_ERR_ALIGN;
  if (rows == 0) return DIP_OK;
  hipLaunchKernelGGL(add_rmsnorm_kernel, dim3((unsigned)rows), dim3(kNormThreads), 0,
                     (hipStream_t)stream, h, add, weight, out, (int)n, eps);
  return hip_status(hipGetLastError());
}

extern "C" int dip_add_rmsnorm(uint16_t* h, const uint16_t* add, const uint16_t* weight,
                               uint16_t* out, int64_t n, float eps, void* stream) {
  return dip_add_rmsnorm_rows(h, add, weight, out, 1, n, eps, stream);
}

namespace {
int launch_qk_rope_cache(const uint16_t* qkv, const uint16_t* q_norm_w, const uint16_t* k_norm_w,
                         const uint16_t* cos_table, const uint16_t* sin_table, const int64_t* pos,
                         uint16_t* q_out, uint16_t* k_cache, uint16_t* v_cache, int64_t tokens,
                         int64_t n_heads, int64_t n_kv_heads, int64_t head_dim, int64_t max_len,
                         float eps, void* stream) {
  if (!qkv || !q_norm_w || !k_norm_w || !cos_table || !sin_table || !q_out || !k_cache || !v_cache)
    return DIP_ERR_NULL;
  if (head_dim != kHeadDim) return DIP_ERR_UNSUPPORTED;
  if (n_heads <= 0 || n_kv_heads <= 0 || n_heads > 4096 || n_kv_heads > 4096 || max_len <= 0 ||
      max_len > INT32_MAX / kHeadDim || tokens < 0 || tokens > max_len)
    return DIP_ERR_SHAPE;
  if (!(eps >= 0.f)) return DIP_ERR_ARG;
  if (!aligned16(qkv) || !aligned16(q_out) || !aligned16(k_cache) || !aligned16(v_cache) ||
      !aligned16(cos_table) || !aligned16(sin_table) || !aligned16(q_norm_w) ||
      !aligned16(k_norm_w))
    return DIP_ERR_ALIGN;
  if (tokens == 0) return DIP_OK;
  const unsigned groups = (unsigned)((n_heads + 2 * n_kv_heads + kRopeHeads - 1) / kRopeHeads);
  hipLaunchKernelGGL(qk_rope_cache_kernel, dim3((unsigned)tokens, groups), dim3(64 * kRopeHeads), 0,
                     (hipStream_t)stream, qkv, q_norm_w, k_norm_w, cos_table, sin_table, pos,
                     q_out, k_cache, v_cache, (int)n_heads, (int)n_kv_heads, (int)max_len, eps);
  return hip_status(hipGetLastError());
}
}  // namespace

extern "C" int dip_qk_norm_rope_cache(const uint16_t* qkv, const uint16_t* q_norm_w,
                                      const uint16_t* k_norm_w, const uint16_t* cos_table,
                                      const uint16_t* sin_table, const int64_t* pos,
                                      uint16_t* q_out, uint16_t* k_cache, uint16_t* v_cache,
                                      int64_t n_heads, int64_t n_kv_heads, int64_t head_dim,
                                      int64_t max_len, float eps, void* stream) {
  if (!pos) return DIP_ERR_NULL;
  return launch_qk_rope_cache(qkv, q_norm_w, k_norm_w, cos_table, sin_table, pos, q_out, k_cache,
                              v_cache, 1, n_heads, n_kv_heads, head_dim, max_len, eps, stream);
}

extern "C" int dip_qk_norm_rope_cache_rows(const uint16_t* qkv, const uint16_t* q_norm_w,
                                           const uint16_t* k_norm_w, const uint16_t* cos_table,
                                           const uint16_t* sin_table, uint16_t* q_out,
                                           uint16_t* k_cache, uint16_t* v_cache, int64_t tokens,
                                           int64_t n_heads, int64_t n_kv_heads, int64_t head_dim,
                                           int64_t max_len, float eps, void* stream) {
  return launch_qk_rope_cache(qkv, q_norm_w, k_norm_w, cos_table, sin_table, nullptr, q_out,
                              k_cache, v_cache, tokens, n_heads, n_kv_heads, head_dim, max_len,
                              eps, stream);
}

extern "C" int64_t dip_decode_attention_fused_max_len(void) { return kFusedMaxLen; }

extern "C" int dip_decode_attention_fused(const uint16_t* qkv, const uint16_t* q_norm_w,
                                          const uint16_t* k_norm_w, const uint16_t* cos_table,
                                          const uint16_t* sin_table, const int64_t* pos,
                                          uint16_t* k_cache, uint16_t* v_cache, uint16_t* out,
                                          int64_t n_heads, int64_t n_kv_heads, int64_t head_dim,
                                          int64_t max_len, float eps, float scale, void* stream) {
  if (!qkv || !q_norm_w || !k_norm_w || !cos_table || !sin_table || !pos || !k_cache ||
      !v_cache || !out)
    return DIP_ERR_NULL;
  if (head_dim != kHeadDim) return DIP_ERR_UNSUPPORTED;
  if (n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads != 0 || n_heads > 4096 ||
      max_len <= 0 || max_len > kFusedMaxLen)
    return DIP_ERR_SHAPE;
  if (!(eps >= 0.f)) return DIP_ERR_ARG;
  if (!aligned16(qkv) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out) ||
      !aligned16(cos_table) || !aligned16(sin_table) || !aligned16(q_norm_w) ||
      !aligned16(k_norm_w))
    return DIP_ERR_ALIGN;
  const int nh = (int)n_heads, nkv = (int)n_kv_heads, ml = (int)max_len;
  hipStream_t s = (hipStream_t)stream;
  // one query head per workgroup; 8 waves (chunks 8 at a time) for caches of
  // more than 128 rows
  if (ml <= 128)
    hipLaunchKernelGGL((attn_fused_kernel<1, 4>), dim3(nh), dim3(256), 0, s, qkv, q_norm_w,
                       k_norm_w, cos_table, sin_table, pos, k_cache, v_cache, out, nh, nkv, ml,
                       eps, scale);
  else
    hipLaunchKernelGGL((attn_fused_kernel<1, 8>), dim3(nh), dim3(512), 0, s, qkv, q_norm_w,
                       k_norm_w, cos_table, sin_table, pos, k_cache, v_cache, out, nh, nkv, ml,
                       eps, scale);
  return hip_status(hipGetLastError());
}

extern "C" size_t dip_decode_attention_workspace_size(int64_t n_heads, int64_t head_dim,
                                                      int64_t max_len) {
  if (n_heads <= 0 || head_dim != kHeadDim || max_len <= 0) return 0;
  const size_t nchunks = (size_t)((max_len + kAttnChunk - 1) / kAttnChunk);
  return nchunks * (size_t)n_heads * kPartFloats * sizeof(float);
}

extern "C" int dip_decode_attention(const uint16_t* q, const uint16_t* k_cache,
                                    const uint16_t* v_cache, const int64_t* pos, uint16_t* out,
                                    int64_t n_heads, int64_t n_kv_heads, int64_t head_dim,
                                    int64_t max_len, float scale, void* workspace,
                                    size_t ws_bytes, void* stream) {
  if (!q || !k_cache || !v_cache || !pos || !out) return DIP_ERR_NULL;
  if (head_dim != kHeadDim) return DIP_ERR_UNSUPPORTED;
  if (n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads != 0 || n_heads > 4096 ||
      max_len <= 0 || max_len > INT32_MAX / kHeadDim)
    return DIP_ERR_SHAPE;
  if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out))
    return DIP_ERR_ALIGN;
  if (!workspace || ws_bytes < dip_decode_attention_workspace_size(n_heads, head_dim, max_len))
    return DIP_ERR_WORKSPACE;
  if (!aligned16(workspace)) return DIP_ERR_ALIGN;
  const int nkv = (int)n_kv_heads;
  const int G = (int)(n_heads / n_kv_heads);
  float* part = static_cast<float*>(workspace);
  hipStream_t s = (hipStream_t)stream;
  const int ml = (int)max_len;
  switch (G) {
    case 1: launch_attention<1>(q, k_cache, v_cache, pos, out, nkv, ml, scale, part, s); break;
    case 2: launch_attention<2>(q, k_cache, v_cache, pos, out, nkv, ml, scale, part, s); break;
    case 4: launch_attention<4>(q, k_cache, v_cache, pos, out, nkv, ml, scale, part, s); break;
    case 5: launch_attention<5>(q, k_cache, v_cache, pos, out, nkv, ml, scale, part, s); break;
    case 8: launch_attention<8>(q, k_cache, v_cache, pos, out, nkv, ml, scale, part, s); break;
    case 16: launch_attention<16>(q, k_cache, v_cache, pos, out, nkv, ml, scale, part, s); break;
    default: return DIP_ERR_UNSUPPORTED;
  }
  return hip_status(hipGetLastError());
}
