// dip_quantize.hip — the int4 g128 format conversions on the GPU, bit-exact
// with the reference's CPU torch code:
//   * quantize (scripts/quantize.py:32-64): per group of 128 columns,
//     s = max(max|w| / 7, 1e-8) in fp32, q = clamp(rint(w / s), -8, 7) with
//     the fp32 s, stored scale = bf16(s);
//   * down transpose (dip_stream_predispatch.py:100-120): down [out, inter]
//     int4 -> bf16(q*s) -> transpose -> fp32 -> quantize along `out`.
// Divisions are IEEE correctly rounded (hipcc's default for fp32 '/'), and
// rintf rounds half to even, matching torch.round.
#include <algorithm>

#include "dip_common.h"
#include "dip_internal.h"

namespace dip {

namespace {

constexpr float kRoundMagic = 12582912.0f;  // 1.5 * 2^23: adding it rounds to an integer (half even)
constexpr float kSureDist = 0.49999f;

DIP_DEV uint32_t quantize_one(float v, float s) {
  const float q = fminf(fmaxf(rintf(v / s), -8.0f), 7.0f);
  return (uint32_t)(int)q & 0xFu;
}

// clamp(rint(v / s), -8, 7) of 8 values as 8 nibbles, first value lowest,
// where s is the group's scale (|v| <= 7 s up to rounding, or s = 1e-8 >
// |v| / 7, so the clamp never acts on finite values).  An IEEE division costs
// over ten instructions a value, so the quotient is v * rcp(s), at most 2^-21
// from the exact one here: its rounding is the quotient's unless it lies
// within 1e-5 of a half-integer, and then (or with an infinite or NaN value
// or scale) the lane divides.
DIP_DEV uint32_t quantize8(const float v[8], float s) {
  const float inv = __builtin_amdgcn_rcpf(s);
  bool sure = s < 1e30f;
  uint32_t packed = 0;
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const float t = fmaf(v[p], inv, kRoundMagic);  // low bits: the integer, two's complement
    const float r = t - kRoundMagic;
    sure = sure && fabsf(fmaf(v[p], inv, -r)) < kSureDist;
    packed = __builtin_amdgcn_alignbit(__float_as_uint(t), packed, 4);
  }
  if (!sure) {
    packed = 0;
#pragma unroll
    for (int p = 0; p < 8; ++p) packed |= quantize_one(v[p], s) << (4 * p);
  }
  return packed;
}

// The scale of a group whose 128 values sit 8 to a lane on 16 lanes (NaN
// values do not count, as fmaxf has it).
DIP_DEV float group_scale(const float v[8]) {
  float m = fabsf(v[0]);
#pragma unroll
  for (int p = 1; p < 8; ++p) m = fmaxf(m, fabsf(v[p]));
  const float s = group_max<16>(m) / 7.0f;
  return s < 1e-8f ? 1e-8f : s;
}

// A dword to a byte pointer that need not be aligned.
DIP_DEV void store_dword(int8_t* p, uint32_t v, bool aligned4) {
  if (aligned4) {
    *reinterpret_cast<uint32_t*>(p) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = (int8_t)(v >> (8 * i));
  }
}

}  // namespace

// 16 lanes per (row, group), 8 consecutive values per lane: one 128-bit load
// (bf16; two for fp32), one packed dword out.  The matrix is one flat run of
// groups.  Bound by HBM: 25600 x 5120 bf16 (331 MB in and out) 87 us, 3.8 TB/s; with one
// wave per group (4 bytes a lane) and a division per value 208 us.
template <bool BF16, bool ALIGN16>
__global__ __launch_bounds__(256) void quantize_kernel(const void* __restrict__ w,
                                                       int8_t* __restrict__ qw,
                                                       uint16_t* __restrict__ sc, long long total,
                                                       bool q_aligned4) {
  const int j = threadIdx.x & 15;
  for (long long g = ((long long)blockIdx.x * 256 + threadIdx.x) >> 4; g < total;
       g += (long long)gridDim.x * 16) {
    const size_t e = (size_t)g * kGroupSize + 8 * j;
    float v[8];
    if constexpr (BF16) {
      const uint16_t* p = reinterpret_cast<const uint16_t*>(w) + e;
      uint4 u;
      if constexpr (ALIGN16) {
        u = ldg_nt(reinterpret_cast<const uint4*>(p));
      } else {
        const uint2 a = reinterpret_cast<const uint2*>(p)[0], b = reinterpret_cast<const uint2*>(p)[1];
        u = make_uint4(a.x, a.y, b.x, b.y);
      }
      const uint32_t d[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[2 * i] = bf16_to_f32(d[i] & 0xFFFFu);
        v[2 * i + 1] = bf16_to_f32(d[i] >> 16);
      }
    } else {
      const float* p = reinterpret_cast<const float*>(w) + e;
#pragma unroll
      for (int i = 0; i < 8; i += 4) {
        if constexpr (ALIGN16) {
          const uint4 u = ldg_nt(reinterpret_cast<const uint4*>(p + i));
          v[i] = __uint_as_float(u.x);
          v[i + 1] = __uint_as_float(u.y);
          v[i + 2] = __uint_as_float(u.z);
          v[i + 3] = __uint_as_float(u.w);
        } else {
          const float2 a = reinterpret_cast<const float2*>(p + i)[0];
          const float2 b = reinterpret_cast<const float2*>(p + i)[1];
          v[i] = a.x;
          v[i + 1] = a.y;
          v[i + 2] = b.x;
          v[i + 3] = b.y;
        }
      }
    }
    const float s = group_scale(v);
    store_dword(qw + (size_t)g * 64 + 4 * j, quantize8(v, s), q_aligned4);
    if (j == 0) sc[g] = (uint16_t)f32_to_bf16(s);
  }
}

// Tile: 128 `out` rows (one output group of down_t) x 256 `inter` columns of
// down, its nibbles staged in LDS by 128-byte row segments.  Lane j of a
// 16-lane group then takes rows 8 j .. 8 j + 7 of 8 neighbouring columns (one
// dword of each row) and requantizes column after column: 16 lanes hold a
// column's 128 values, 8 to a lane, as in quantize_kernel, and write its 64
// packed bytes.  Row 8 j + i sits at LDS row 16 i + j, 36 dwords apart: the
// lanes of a read then spread over all banks.  VALU-bound: 5120 x 25600 took
// 189 us with byte accesses and a division per value, 104 us in this form.
constexpr int kTileCols = 256;
constexpr int kTileStride = kTileCols / 8 + 4;  // dwords

__global__ __launch_bounds__(256) void transpose_down_kernel(
    const int8_t* __restrict__ dqw, const uint16_t* __restrict__ dsc, int8_t* __restrict__ tqw,
    uint16_t* __restrict__ tsc, int out_f, int inter, bool in_aligned16, bool out_aligned4) {
  __shared__ __align__(16) uint32_t tile[128 * kTileStride];
  __shared__ float tscale[2][128];  // scale / 16 of (column group of the tile, LDS row)
  const int n_ctiles = (inter + kTileCols - 1) / kTileCols;
  const int g = blockIdx.x / n_ctiles;  // output group (128 out rows)
  const int c0 = (blockIdx.x % n_ctiles) * kTileCols;
  const int tid = threadIdx.x;
  const size_t in_half = (size_t)(inter / 2);
  const int in_groups = inter / kGroupSize;
#pragma unroll
  for (int e = tid; e < 128 * (kTileCols / 32); e += 256) {
    const int o = e / (kTileCols / 32), q = e % (kTileCols / 32);
    uint4 v = make_uint4(0, 0, 0, 0);
    if (c0 + 32 * q < inter) {  // inter is a multiple of 128
      const int8_t* p = dqw + (size_t)(g * 128 + o) * in_half + c0 / 2 + 16 * q;
      if (in_aligned16) v = *reinterpret_cast<const uint4*>(p);
      else __builtin_memcpy(&v, p, 16);
    }
    *reinterpret_cast<uint4*>(&tile[((o & 7) * 16 + (o >> 3)) * kTileStride + 4 * q]) = v;
  }
  {
    const int h = tid >> 7, o = tid & 127;
    const int cg = min(c0 / kGroupSize + h, in_groups - 1);
    tscale[h][(o & 7) * 16 + (o >> 3)] =
        bf16_to_f32(dsc[(size_t)(g * 128 + o) * in_groups + cg]) * 0.0625f;
  }
  __syncthreads();
  const int lane = tid & 63, wave = tid >> 6;
  const int j = lane & 15;
  const int out_groups = out_f / kGroupSize;
#pragma unroll 1
  for (int it = 0; it < 2; ++it) {
    const int d = wave * 8 + it * 4 + (lane >> 4);  // dword column: columns c0 + 8 d + p
    if (c0 + 8 * d >= inter) continue;  // uniform over the wave: inter is a multiple of 128
    uint32_t lo[8], hi[8];
    float s16[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t w = tile[(i * 16 + j) * kTileStride + d];
      lo[i] = (w << 4) & 0xF0F0F0F0u;
      hi[i] = w & 0xF0F0F0F0u;
      s16[i] = tscale[d >> 4][i * 16 + j];
    }
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        const uint32_t a = p & 1 ? hi[i] : lo[i], b = p & 1 ? hi[i + 1] : lo[i + 1];
        const float fa = p < 2 ? cvt_sbyte<0>(a) : p < 4 ? cvt_sbyte<1>(a) : p < 6 ? cvt_sbyte<2>(a) : cvt_sbyte<3>(a);
        const float fb = p < 2 ? cvt_sbyte<0>(b) : p < 4 ? cvt_sbyte<1>(b) : p < 6 ? cvt_sbyte<2>(b) : cvt_sbyte<3>(b);
        // qlinear.dequantize rounds q*s to bf16 before the transpose
        const uint32_t r = f32x2_to_bf16x2_nan(fa * s16[i], fb * s16[i + 1]);
        v[i] = bf16_to_f32(r & 0xFFFFu);
        v[i + 1] = __uint_as_float(r & 0xFFFF0000u);
      }
      const float s = group_scale(v);
      const size_t c = (size_t)(c0 + 8 * d + p);
      store_dword(tqw + c * (out_f / 2) + (size_t)g * 64 + 4 * j, quantize8(v, s), out_aligned4);
      if (j == 0) tsc[c * out_groups + g] = (uint16_t)f32_to_bf16(s);
    }
  }
}

// sc_gm[g][r] = sc[r][g]: 64 x 64 tiles through LDS, both sides coalesced.
__global__ __launch_bounds__(256) void scales_group_major_kernel(
    const uint16_t* __restrict__ sc, uint16_t* __restrict__ gm, int rows, int groups) {
  __shared__ uint16_t tile[64][65];
  const int r0 = blockIdx.x * 64, g0 = blockIdx.y * 64;
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int r = e / 64, g = e % 64;
    if (r0 + r < rows && g0 + g < groups) tile[r][g] = sc[(size_t)(r0 + r) * groups + g0 + g];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int g = e / 64, r = e % 64;
    if (r0 + r < rows && g0 + g < groups) gm[(size_t)(g0 + g) * rows + r0 + r] = tile[r][g];
  }
}

}  // namespace dip

using namespace dip;

extern "C" int dip_scales_group_major(const uint16_t* scales, uint16_t* scales_gm, int64_t rows,
                                      int64_t groups, void* stream) {
  if (!scales || !scales_gm) return DIP_ERR_NULL;
  if (rows < 0 || groups <= 0 || rows > INT32_MAX || groups > 65536 ||
      (rows + 63) / 64 > INT32_MAX)
    return DIP_ERR_SHAPE;
  if (rows == 0) return DIP_OK;
  const dim3 grid((unsigned)((rows + 63) / 64), (unsigned)((groups + 63) / 64));
  hipLaunchKernelGGL(scales_group_major_kernel, grid, dim3(256), 0, (hipStream_t)stream, scales,
                     scales_gm, (int)rows, (int)groups);
  return hip_status(hipGetLastError());
}

extern "C" int dip_quantize_int4(const void* w, int w_is_bf16, int8_t* qweight, uint16_t* scales,
                                 int64_t rows, int64_t cols, void* stream) {
  if (!w || !qweight || !scales) return DIP_ERR_NULL;
  if (rows < 0 || cols <= 0 || cols % kGroupSize != 0 || rows > INT32_MAX || cols > (1 << 24))
    return DIP_ERR_SHAPE;
  if ((reinterpret_cast<uintptr_t>(w) & 7u) != 0) return DIP_ERR_ALIGN;
  if (rows == 0) return DIP_OK;
  const long long groups = rows * (cols / kGroupSize);
  const dim3 grid((unsigned)std::min<long long>((groups + 15) / 16, 1 << 20));
  const bool a16 = aligned16(w), q4 = (reinterpret_cast<uintptr_t>(qweight) & 3u) == 0;
  hipStream_t s = (hipStream_t)stream;
  if (w_is_bf16 && a16)
    hipLaunchKernelGGL((quantize_kernel<true, true>), grid, dim3(256), 0, s, w, qweight, scales, groups, q4);
  else if (w_is_bf16)
    hipLaunchKernelGGL((quantize_kernel<true, false>), grid, dim3(256), 0, s, w, qweight, scales, groups, q4);
  else if (a16)
    hipLaunchKernelGGL((quantize_kernel<false, true>), grid, dim3(256), 0, s, w, qweight, scales, groups, q4);
  else
    hipLaunchKernelGGL((quantize_kernel<false, false>), grid, dim3(256), 0, s, w, qweight, scales, groups, q4);
  return hip_status(hipGetLastError());
}

extern "C" int dip_transpose_down_int4(const int8_t* down_qw, const uint16_t* down_sc,
                                       int8_t* down_t_qw, uint16_t* down_t_sc,
                                       int64_t out_features, int64_t inter, void* stream) {
  if (!down_qw || !down_sc || !down_t_qw || !down_t_sc) return DIP_ERR_NULL;
  if (out_features <= 0 || inter <= 0 || out_features % kGroupSize || inter % kGroupSize ||
      out_features > INT32_MAX || inter > INT32_MAX)
    return DIP_ERR_SHAPE;
  const long long blocks = (out_features / kGroupSize) * ((inter + kTileCols - 1) / kTileCols);
  if (blocks > INT32_MAX) return DIP_ERR_SHAPE;
  hipLaunchKernelGGL(transpose_down_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     (hipStream_t)stream, down_qw, down_sc, down_t_qw, down_t_sc,
                     (int)out_features, (int)inter, aligned16(down_qw),
                     (reinterpret_cast<uintptr_t>(down_t_qw) & 3u) == 0);
  return hip_status(hipGetLastError());
}
