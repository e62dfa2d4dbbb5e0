// dip_gemm.hip — int4 g128 GEMM for prompts (more than one token) on bf16
// MFMA: out[M, N] = bf16( x[M, K] . W[N, K]^T ), W in the reference's Linear
// layout (qweight int8 [N, K/2], scales bf16 [N, K/128]).
//
// The reference computes this as dequantize + F.linear (qlinear.py:86-88,
// dip_stream_predispatch.py:206-215 for gate and up): it writes a bf16 copy
// of W and reads it back in a GEMM.  Here each weight is read once, as
// packed nibbles, and turned into an MFMA operand in registers:
//   * a nibble u (two's complement q) in mantissa bits 3..6 of bf16 16.0, its
//     top bit flipped, is 24 + q exactly; nibbles j and j + 4 of a dword sit
//     16 bits apart, so two weights cost a shift and one v_bitop3;
//   * x is paired the same way, (x[c + j], x[c + j + 4]), on its way into LDS;
//   * v_mfma_f32_16x16x32_bf16 sums (24 + q) * x over one 128-column group in
//     fp32, starting from -24 * sum(x) of the group, which the same MFMA gives
//     with a constant operand: the result is sum(q * x), scaled by the group's
//     scale into the fp32 total.  (Tokens that leave fp32's range on the way
//     are computed from plain q * s: plain_dot.)
// So the weights enter exactly as q * s in fp32 (the reference rounds q * s
// to bf16 first); the output is rounded to bf16 once.
#include <algorithm>

#include "dip_common.h"
#include "dip_internal.h"

namespace dip {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr uint32_t kPair24 = 0x41C041C0u;    // bf16 16.0 twice, the nibbles' top bits flipped
constexpr uint32_t kMinus24 = 0xC1C0C1C0u;   // bf16 -24.0, twice

DIP_DEV bf16x8_t as_bf16x8(const uint4& v) {
  return __builtin_bit_cast(bf16x8_t, u32x4_t{v.x, v.y, v.z, v.w});
}

// 8 nibbles -> 24 + q as bf16, in the order 0, 4, 1, 5, 2, 6, 3, 7.
DIP_DEV bf16x8_t weights24(uint32_t w) {
  return __builtin_bit_cast(
      bf16x8_t, u32x4_t{((w << 3) & kPairMask) ^ kPair24, ((w >> 1) & kPairMask) ^ kPair24,
                        ((w >> 5) & kPairMask) ^ kPair24, ((w >> 9) & kPairMask) ^ kPair24});
}

constexpr size_t kGemmLds = 160 * 1024;
constexpr int kXcds = 8;  // workgroups go to the 8 XCDs round-robin

// ---------------------------------------------------------------------------
// Few tokens (or few rows): K split over a workgroup's waves.  16 TM tokens and
// RW tiles of 16 weight rows per workgroup, whose KS waves take the K groups ks,
// ks + KS, ... and add their sums through LDS at the end, in a fixed order.
// Bound by HBM, or by the launch.  Per group a wave
//   * has its RW x 16 rows' nibbles in flight D groups ahead (lane: row l16,
//     columns 32 kb ..: 16 bytes, so 64 contiguous bytes of each row; cached,
//     since the next wave reads the other half of the same lines: with
//     streaming loads 25600 x 5120 took 30 us instead of 25);
//   * stages its own x tile in LDS, loaded a group ahead by whole 256-byte token
//     rows (read as operands from memory, 16 bytes of 64 different lines per
//     load, x bounds the kernel), chunk c of token t at slot c ^ (t % 16), which
//     is free of bank conflicts on both sides; nothing is shared, so the loop
//     has no barrier;
//   * works on UB row tiles at a time, UB * TM independent chains of MFMAs (one
//     chain at a time left the matrix cores waiting: 20.6 us of 25 us).
// 25600 x 5120: 2 tokens 27.8 -> 22 us, 32 tokens 45.5 -> 30 us; 10240 x 5120,
// 7 tokens 17.1 -> 12 us; 5120 x 8192, 32 tokens 24.5 -> 16 us (before: RW
// tiles and K parts by the matrix alone, x and 16-bit scales from memory).
// Tokens are the MFMA's rows, so that a lane's 4 sums belong to one weight row
// and share its scale.  The scales of the workgroup's rows are one contiguous
// run, staged in LDS once (SCL) unless K is too long for that or they are not
// 4-byte aligned.
// ---------------------------------------------------------------------------
constexpr int kScaleRegs = 5;  // scale dwords a thread holds before the first barrier

// Between LDS accesses of one wave's lanes that depend on each other: the LDS
// keeps a wave's order by itself, this holds the compiler to it.
DIP_DEV void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// A workgroup's scales, staged in LDS by dwords: the run of its n values of one
// matrix or (GU) of the gate, and at `stride` (even) that of up.
template <bool GU>
struct ScaleRun {
  const uint16_t *sc, *sc_up;
  int n, stride;
  DIP_DEV int values() const { return GU ? stride + n : n; }
  DIP_DEV int at(int up) const { return GU && up ? stride : 0; }
  // values e and e + 1, e even
  DIP_DEV uint32_t dword(int e) const {
    const uint16_t* p = sc;
    if (GU && e >= stride) {
      p = sc_up;
      e -= stride;
    }
    // an odd count's last value is loaded alone: it may end the matrix
    return e + 1 < n ? *reinterpret_cast<const uint32_t*>(p + e) : e < n ? p[e] : 0u;
  }
};

// An output from plain q * s, by one lane: for tokens that 24 * sum(x) takes out
// of fp32's range (an infinite x, or values near the largest), whose sums above
// are not finite and stay so whatever follows.  A kernel's last step watches its
// sums with one instruction each (gate and up of 12288 x 4096, 333 tokens 108.9 ->
// 109.1 us; with a class compare and its mask 109.6), and the lanes that hold such
// a one come here for their outputs that are not finite, so other tokens keep
// their bits.  A sum that is NaN ends the walk (512 tokens through 25600 x 5120:
// 190 us, one of them infinite 570, all NaN 510, an infinity in each 13 ms).
DIP_DEV float plain_dot(const int8_t* qw, const uint16_t* sc, const uint16_t* x, int row, int tok,
                        int K) {
  const int ngroups = K >> 7;
  const uint32_t* w = reinterpret_cast<const uint32_t*>(qw + (size_t)row * (K >> 1));
  const uint4* xv = reinterpret_cast<const uint4*>(x + (size_t)tok * K);
  float acc = 0.f;
  for (int g = 0; g < ngroups && acc == acc; ++g) {
    const float s = bf16_to_f32(sc[(size_t)row * ngroups + g]);
    float v = 0.f;
#pragma unroll 2
    for (int d = 0; d < 16; ++d) {
      const uint32_t q = w[16 * g + d];
      const uint4 p = xv[16 * g + d];
      const uint32_t px[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v = fmaf((float)(int)__builtin_amdgcn_sbfe(q, 4 * i, 4) * s,
                 bf16_to_f32(i & 1 ? px[i / 2] >> 16 : px[i / 2] & 0xFFFFu), v);
    }
    acc += v;
  }
  return acc;
}

DIP_DEV bool not_finite(float v) { return __builtin_amdgcn_classf(v, 0x207); }  // NaN, inf
// 0 while every v so far was finite, then NaN.
DIP_DEV void watch(float& seen, float v) { seen = fmaf(v, 0.f, seen); }

// The output of (tok, row) again from plain q * s if the stored one, this lane's
// own, is not finite.  (With gate and up: whichever of the two was not finite, the
// stored product is not either, silu(-inf) being NaN.)
template <bool GU>
DIP_DEV void redo_output(const int8_t* qw, const uint16_t* sc, const int8_t* qw_up,
                         const uint16_t* sc_up, const uint16_t* x, uint16_t* out, int N, int K,
                         int row, int tok) {
  uint16_t* o = out + (size_t)tok * N + row;
  if (!not_finite(bf16_to_f32(*o))) return;
  uint32_t v = f32_to_bf16(plain_dot(qw, sc, x, row, tok, K));
  if constexpr (GU) v = swiglu_bf16(v, f32_to_bf16(plain_dot(qw_up, sc_up, x, row, tok, K)));
  *o = (uint16_t)v;
}

template <int TM, int RW, int KS, int D, bool SCL, bool GU>
__global__ __launch_bounds__(KS * 64, 2) void int4_gemm_split_kernel(
    const int8_t* __restrict__ qw, const uint16_t* __restrict__ sc, const int8_t* __restrict__ qw_up,
    const uint16_t* __restrict__ sc_up, const uint16_t* __restrict__ x, uint16_t* __restrict__ out,
    int M, int N, int K, int row_blocks) {
  static_assert(!GU || RW % 2 == 0, "tiles in pairs");
  extern __shared__ __align__(16) uint4 gemm_lds[];
  constexpr int kThreads = KS * 64;
  constexpr int XT = TM * 256;         // 16-byte chunks of a wave's x tile
  constexpr int UB = TM == 1 ? 4 : 2;  // row tiles worked on together
  const int ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int kb = lane >> 4, l16 = lane & 15;
  // Row tile u starts at a row that leaves it 16 rows (a matrix of fewer than
  // 16: its lanes past the last row repeat it); tiles that overlap compute and
  // store the same values.
  // GU: tile 2 p is rows of the gate, tile 2 p + 1 the same rows of up.
  constexpr int kRows = GU ? 8 * RW : 16 * RW;  // of a matrix, per workgroup
  const int row0 = max(0, min((int)(blockIdx.x % row_blocks) * kRows, N - 16));
  auto tile_row = [&](int u) { return max(0, min(row0 + 16 * (GU ? u / 2 : u), N - 16)); };
  const int lrow = min(l16, N - 1);
  const int tok0 = (int)(blockIdx.x / row_blocks) * (16 * TM);
  const int ngroups = K >> 7;
  const int ng = ngroups > ks ? (ngroups - ks + KS - 1) / KS : 0;
  const int glast = ks + (ng - 1) * KS;  // loads past the end repeat the last group
  uint4* xt = gemm_lds + ks * XT;
  uint32_t* ssc = reinterpret_cast<uint32_t*>(gemm_lds + KS * XT);

  [[maybe_unused]] uint32_t sreg[kScaleRegs];
  const ScaleRun<GU> run{sc + (size_t)row0 * ngroups, GU ? sc_up + (size_t)row0 * ngroups : nullptr,
                         min(kRows, N - row0) * ngroups, kRows * ngroups};
  const int n_sc = run.values();  // this workgroup's scales
  if constexpr (SCL) {
#pragma unroll
    for (int i = 0; i < kScaleRegs; ++i) sreg[i] = run.dword(2 * (i * kThreads + (int)threadIdx.x));
  }
  const uint32_t woff = (uint32_t)lrow * (uint32_t)(K >> 1) + 16u * kb;
  const char* xbase = reinterpret_cast<const char*>(x + (size_t)tok0 * K);
  const int tlast = M - 1 - tok0;
  uint4 xr[TM * 4], w[D][RW];
  [[maybe_unused]] uint32_t s[D][RW];
  auto load_x = [&](int g) {
#pragma unroll
    for (int i = 0; i < TM * 4; ++i)
      xr[i] = *reinterpret_cast<const uint4*>(
          xbase + (size_t)g * 256 +
          ((uint32_t)min(4 * i + kb, tlast) * (uint32_t)(2 * K) + (uint32_t)(16 * l16)));
  };
  auto stage_x = [&] {
#pragma unroll
    for (int i = 0; i < TM * 4; ++i) {
      const int t = 4 * i + kb;
      uint32_t p[4];
      make_xpairs(xr[i].x, xr[i].y, xr[i].z, xr[i].w, p);
      xt[t * 16 + (l16 ^ (t & 15))] = make_uint4(p[0], p[1], p[2], p[3]);
    }
  };
  auto load_w = [&](int d, int u, int g) {
    const int8_t* p = (GU && u % 2 ? qw_up : qw) + (size_t)tile_row(u) * (K >> 1) + (size_t)g * 64;
    w[d][u] = *reinterpret_cast<const uint4*>(p + woff);
    if constexpr (!SCL)
      s[d][u] = (GU && u % 2 ? sc_up : sc)[(size_t)(tile_row(u) + lrow) * ngroups + g];
  };
  floatx4 acc[RW][TM];
#pragma unroll
  for (int u = 0; u < RW; ++u)
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[u][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (ng > 0) {
    load_x(ks);
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int u = 0; u < RW; ++u) load_w(d, u, min(ks + d * KS, glast));
    stage_x();
    wave_lds_order();
  }
  if constexpr (SCL) {
#pragma unroll
    for (int i = 0; i < kScaleRegs; ++i) {
      const int e = i * kThreads + (int)threadIdx.x;
      if (2 * e < n_sc) ssc[e] = sreg[i];
    }
    for (int e = kScaleRegs * kThreads + (int)threadIdx.x; 2 * e < n_sc; e += kThreads)
      ssc[e] = run.dword(2 * e);
    __syncthreads();
  }

  const bf16x8_t m24 = __builtin_bit_cast(bf16x8_t, u32x4_t{kMinus24, kMinus24, kMinus24, kMinus24});
  for (int i0 = 0; i0 < ng; i0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int i = i0 + d;
      if (i < ng) {
        const int g = ks + i * KS;
        load_x(min(g + KS, glast));
        bf16x8_t xa[TM][4];
        floatx4 c[TM];  // -24 * (the group's sum of x) per token
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < TM; ++t) {
            xa[t][j] = as_bf16x8(xt[(16 * t + l16) * 16 + ((4 * kb + j) ^ l16)]);
            c[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                xa[t][j], m24, j ? c[t] : floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
          }
#pragma unroll
        for (int u0 = 0; u0 < RW; u0 += UB) {
          float sf[UB];
          bf16x8_t b[UB][4];
          floatx4 v[UB][TM];
#pragma unroll
          for (int q = 0; q < UB; ++q) {
            const int u = u0 + q;
            if (u < RW) {
              if constexpr (SCL)
                sf[q] = bf16_to_f32(
                    reinterpret_cast<const uint16_t*>(ssc)[run.at(u % 2) + (tile_row(u) - row0 + lrow) * ngroups + g]);
              else
                sf[q] = bf16_to_f32(s[d][u]);
              b[q][0] = weights24(w[d][u].x);
              b[q][1] = weights24(w[d][u].y);
              b[q][2] = weights24(w[d][u].z);
              b[q][3] = weights24(w[d][u].w);
              load_w(d, u, min(g + D * KS, glast));
            }
          }
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < UB; ++q)
#pragma unroll
              for (int t = 0; t < TM; ++t)
                if (u0 + q < RW)
                  v[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                      xa[t][j], b[q][j], j ? v[q][t] : c[t], 0, 0, 0);
          if (u0 + UB >= RW) {  // the next group's tile over this one's
            wave_lds_order();
            stage_x();
            wave_lds_order();
          }
#pragma unroll
          for (int q = 0; q < UB; ++q)
#pragma unroll
            for (int t = 0; t < TM; ++t)
              if (u0 + q < RW)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  acc[u0 + q][t][r] = fmaf(sf[q], v[q][t][r], acc[u0 + q][t][r]);
        }
      }
    }
  }

  // the waves' sums, in wave order; wave k takes every KS-th of the values
  constexpr int F = RW * TM * 4;
  float* red = reinterpret_cast<float*>(gemm_lds) + lane;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < RW; ++u)
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[(ks * F + (u * TM + t) * 4 + r) * 64] = acc[u][t][r];
  __syncthreads();
  float seen = 0.f;
  auto sum = [&](int f) {
    float v = red[f * 64];
#pragma unroll
    for (int k = 1; k < KS; ++k) v += red[(k * F + f) * 64];
    watch(seen, v);
    return f32_to_bf16(v);
  };
  for (int f = ks; f < (GU ? F / 2 : F); f += KS) {
    const int r = f & 3, t = (f >> 2) % TM, u = (f >> 2) / TM * (GU ? 2 : 1);
    const int tok = tok0 + 16 * t + 4 * kb + r;
    const int fu = (u * TM + t) * 4 + r;
    const uint32_t v = GU ? swiglu_bf16(sum(fu), sum(fu + 4 * TM)) : sum(fu);
    if (tok < M && l16 < N) out[(size_t)tok * N + tile_row(u) + l16] = (uint16_t)v;
  }
  if (seen != 0.f && l16 < N)
    for (int f = ks; f < (GU ? F / 2 : F); f += KS) {
      const int r = f & 3, t = (f >> 2) % TM, u = (f >> 2) / TM * (GU ? 2 : 1);
      const int tok = tok0 + 16 * t + 4 * kb + r;
      if (tok < M)
        redo_output<GU>(qw, sc, qw_up, sc_up, x, out, N, K, tile_row(u) + l16, tok);
    }
}

constexpr size_t split_lds_bytes(int tm, int rw, int ks, int scale_groups) {
  const size_t x = (size_t)ks * tm * 4096 + (size_t)16 * rw * scale_groups * 2;
  const size_t red = (size_t)ks * rw * tm * 4 * 256;
  return x > red ? x : red;
}

// A product's operands; qw_up null: out = x . W^T alone, else gate and up.
struct GemmArgs {
  const int8_t* qw;
  const uint16_t* sc;
  const int8_t* qw_up;
  const uint16_t* sc_up;
  const uint16_t* x;
  uint16_t* out;
  int M, N, K;
  long long rows() const { return qw_up ? 2LL * N : N; }  // of weights
};

template <int TM, int RW, int KS, int D, bool SCL, bool GU>
int launch_split(const GemmArgs& a, hipStream_t s) {
  static std::atomic<uint64_t> granted{0};
  if (const int st = allow_lds(
          granted, reinterpret_cast<const void*>(&int4_gemm_split_kernel<TM, RW, KS, D, SCL, GU>),
          (int)kGemmLds))
    return st;
  constexpr int kRows = GU ? 8 * RW : 16 * RW;
  const int row_blocks = (a.N + kRows - 1) / kRows;
  const unsigned grid = (unsigned)row_blocks * (unsigned)((a.M + 16 * TM - 1) / (16 * TM));
  hipLaunchKernelGGL((int4_gemm_split_kernel<TM, RW, KS, D, SCL, GU>), dim3(grid), dim3(KS * 64),
                     split_lds_bytes(TM, RW, KS, SCL ? a.K / kGroupSize : 0), s, a.qw, a.sc, a.qw_up,
                     a.sc_up, a.x, a.out, a.M, a.N, a.K, row_blocks);
  return hip_status(hipGetLastError());
}

// Row tiles per workgroup: the count that leaves the busiest CU the least to
// do, with 0.6 of a row tile as a workgroup's own share (its x tile).  Gate and
// up have them in pairs: two pairs once that still gives more than 1.5
// workgroups per CU (us, one pair / two, 32 tokens: 25600 x 5120, 800
// workgroups of two, 64.8 / 56.7; 14336 x 4096, 448, 31.4 / 24.4; 9728 x 2560,
// 304, 17.1 / 17.4; 3072 x 1024, 96, 6.6 / 8.1).
int split_row_tiles(const GemmArgs& a, int token_blocks) {
  const long long tiles = (a.N + 15) / 16;
  const int cus = device_cus();
  if (a.qw_up) return 2 * ((tiles + 1) / 2 * token_blocks) > 3LL * cus ? 4 : 2;
  int best = 1;
  long long cost = 0;
  for (int rw = 1; rw <= 4; ++rw) {
    const long long wgs = (tiles + rw - 1) / rw * token_blocks;
    const long long c = (wgs + cus - 1) / cus * (10 * rw + 6);
    if (rw == 1 || c <= cost) {
      best = rw;
      cost = c;
    }
  }
  return best;
}

// Scale runs are staged by dwords, so they start at even values.
bool scales_by_dword(const GemmArgs& a) {
  return ((reinterpret_cast<uintptr_t>(a.sc) | reinterpret_cast<uintptr_t>(a.sc_up)) & 3u) == 0 &&
         (a.K / kGroupSize % 2 == 0 || a.N % 2 == 0);
}

template <int TM, bool GU>
int launch_split_tokens(const GemmArgs& a, hipStream_t s) {
  const int blocks = (a.M + 16 * TM - 1) / (16 * TM);
  const int rw = split_row_tiles(a, blocks);
  // at most one workgroup per CU: twice the waves, on half as many groups each
  const bool few = ((a.N + 15) / 16 * (GU ? 2LL : 1LL) + rw - 1) / rw * blocks <= device_cus();
  if (!scales_by_dword(a) ||
      split_lds_bytes(TM, rw, few ? 8 : 4, a.K / kGroupSize) > kGemmLds / (few ? 1 : 2))
    return launch_split<TM, 2, 4, 1, false, GU>(a, s);
  // two pairs of gate and up tiles come with more than 1.5 workgroups per CU
  if constexpr (GU) {
    if (rw == 4) return launch_split<TM, 4, 4, 2, true, GU>(a, s);
    return few ? launch_split<TM, 2, 8, 2, true, GU>(a, s) : launch_split<TM, 2, 4, 2, true, GU>(a, s);
  } else {
#define DIP_SPLIT(R)                                                    \
  if (rw == (R))                                                        \
    return few ? launch_split<TM, R, 8, 2, true, GU>(a, s)              \
               : launch_split<TM, R, 4, 2, true, GU>(a, s);
    DIP_SPLIT(2) DIP_SPLIT(3) DIP_SPLIT(4)
#undef DIP_SPLIT
    // one block of tokens has a single tile a workgroup only while those are few:
    // beyond one to a CU two tiles or more cost less
    if constexpr (TM == 1) return launch_split<TM, 1, 8, 2, true, GU>(a, s);
    else return few ? launch_split<TM, 1, 8, 2, true, GU>(a, s) : launch_split<TM, 1, 4, 2, true, GU>(a, s);
  }
}

// ---------------------------------------------------------------------------
// Enough tokens and rows to fill the chip: 64 RW weight rows and 64 tokens per
// workgroup, 4 waves side by side with RW tiles of 16 rows each, times KS parts
// of K (part ks takes groups ks, ks + KS, ...) whose sums are added through LDS
// at the end, in a fixed order.  Per group (one step, one barrier):
//   * a part's 4 waves stage its x tile in LDS, P steps ahead in registers, as
//     above, and each token's -24 * sum(x) beside it;
//   * a wave has its rows' nibbles in flight P steps ahead and turns each into
//     an operand once for all 64 tokens;
//   * per 32-column slice, 4 operands from LDS feed 4 RW independent MFMAs.
// Bound by instruction issue (RW 4: 64 MFMAs and 283 other vector instructions
// a step, half of them the nibbles) and below about 500 workgroups by a step's
// latency: 25600 x 5120, 64 tokens 68 -> 35 us, 100 tokens 57 us (dequantize
// and the library's product: 119), 333 tokens 132 us (159), 512 tokens 180 us
// (191); 2048 tokens 639 us, 840 TFLOP/s (540).  The token blocks of a row block run on one XCD, whose
// L2 then reads the rows once.
// ---------------------------------------------------------------------------
// x pairs of 8 values, and their sum.
DIP_DEV uint4 pair8(const uint4& v, float& sum) {
  uint32_t p[4];
  make_xpairs(v.x, v.y, v.z, v.w, p);
  sum = dot2_bf16(v.x, 0x3F803F80u, 0.f);
  sum = dot2_bf16(v.y, 0x3F803F80u, sum);
  sum = dot2_bf16(v.z, 0x3F803F80u, sum);
  sum = dot2_bf16(v.w, 0x3F803F80u, sum);
  return make_uint4(p[0], p[1], p[2], p[3]);
}

constexpr int kTileTokens = 64;

template <int RW, int KS, bool GU>
__global__ __launch_bounds__(KS * 256, 2) void int4_gemm_kernel(
    const int8_t* __restrict__ qw, const uint16_t* __restrict__ sc, const int8_t* __restrict__ qw_up,
    const uint16_t* __restrict__ sc_up, const uint16_t* __restrict__ x, uint16_t* __restrict__ out,
    int M, int N, int K, int row_blocks, int token_blocks) {
  extern __shared__ __align__(16) uint4 gemm_lds[];
  constexpr int TM = kTileTokens / 16;
  constexpr int P = RW == 4 ? 1 : 2;
  constexpr int XT = TM * 256;  // 16-byte chunks of an x tile
  const int bi = blockIdx.x / kXcds;
  const int rb = blockIdx.x % kXcds + kXcds * (bi / token_blocks);
  if (rb >= row_blocks) return;
  const int tok0 = (bi % token_blocks) * kTileTokens;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int ks = wave >> 2, wr = wave & 3;
  const int kb = lane >> 4, l16 = lane & 15;
  // row tiles at the end of the matrix overlap, and GU pairs them, as in the
  // kernel above
  constexpr int kRows = GU ? 32 * RW : 64 * RW;
  const int row0 = max(0, min(rb * kRows, N - 16));
  auto tile_row = [&](int u) {
    return max(0, min(row0 + 16 * (GU ? (RW * wr + u) / 2 : RW * wr + u), N - 16));
  };
  const int lrow = min(l16, N - 1);
  const int ngroups = K >> 7;
  const int steps = (ngroups + KS - 1) / KS;
  uint4* xt = gemm_lds + ks * 2 * XT;  // two buffers
  float* xs = reinterpret_cast<float*>(gemm_lds + KS * 2 * XT) + ks * 2 * kTileTokens;
  uint32_t* ssc = reinterpret_cast<uint32_t*>(gemm_lds + KS * 2 * (XT + kTileTokens / 4));

  const int xtok = (threadIdx.x & 255) >> 4;  // the thread's token of every 16
  const char* xbase = reinterpret_cast<const char*>(x + (size_t)tok0 * K);
  uint32_t xoff[TM];
#pragma unroll
  for (int e = 0; e < TM; ++e)
    xoff[e] = (uint32_t)min(16 * e + xtok, M - 1 - tok0) * (uint32_t)(2 * K) + (uint32_t)(16 * l16);
  const uint32_t woff = (uint32_t)lrow * (uint32_t)(K >> 1) + 16u * kb;
  uint4 xr[P][TM], w[P][RW];
  auto group = [&](int i) { return min(ks + i * KS, ngroups - 1); };  // past the end: the last again
  auto load_x = [&](int p, int i) {
    const char* b = xbase + (size_t)group(i) * 256;
#pragma unroll
    for (int e = 0; e < TM; ++e) xr[p][e] = *reinterpret_cast<const uint4*>(b + xoff[e]);
  };
  auto stage_x = [&](int p, int buf) {
#pragma unroll
    for (int e = 0; e < TM; ++e) {
      const int t = 16 * e + xtok;
      float sum;
      xt[buf * XT + t * 16 + (l16 ^ (t & 15))] = pair8(xr[p][e], sum);
      sum = group_sum<16>(sum);
      if (l16 == 0) xs[buf * kTileTokens + t] = -24.0f * sum;
    }
  };
  auto load_w = [&](int p, int u, int i) {
    const int8_t* q =
        (GU && u % 2 ? qw_up : qw) + (size_t)tile_row(u) * (K >> 1) + (size_t)group(i) * 64;
    w[p][u] = *reinterpret_cast<const uint4*>(q + woff);
  };
  load_x(0, 0);
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int u = 0; u < RW; ++u) load_w(p, u, p);
  const ScaleRun<GU> run{sc + (size_t)row0 * ngroups, GU ? sc_up + (size_t)row0 * ngroups : nullptr,
                         min(kRows, N - row0) * ngroups, kRows * ngroups};
  for (int e0 = threadIdx.x; 2 * e0 < run.values(); e0 += 8 * KS * 256) {
    uint32_t r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = run.dword(2 * (e0 + i * KS * 256));
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (2 * (e0 + i * KS * 256) < run.values()) ssc[e0 + i * KS * 256] = r[i];
  }
  stage_x(0, 0);
#pragma unroll
  for (int p = 0; p < P; ++p) load_x((p + 1) % P, p + 1);
  __syncthreads();

  floatx4 acc[RW][TM];
#pragma unroll
  for (int u = 0; u < RW; ++u)
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[u][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  // two steps per turn: the register slots and the buffers are constants
  for (int i0 = 0; i0 < steps; i0 += 2) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int i = i0 + e;
      if (i < steps) {
        const int p = e % P;
        // the next step's x into the other buffer, which every wave has left
        stage_x((e + 1) % P, e ^ 1);
        load_x((e + 1) % P, i + 1 + P);
        if (ks + i * KS < ngroups) {
          float sf[RW];
#pragma unroll
          for (int u = 0; u < RW; ++u)
            sf[u] = bf16_to_f32(reinterpret_cast<const uint16_t*>(
                ssc)[run.at(u % 2) + (tile_row(u) - row0 + lrow) * ngroups + ks + i * KS]);
          floatx4 v[RW][TM];
#pragma unroll
          for (int t = 0; t < TM; ++t) {
            const floatx4 c = *reinterpret_cast<const floatx4*>(&xs[e * kTileTokens + 16 * t + 4 * kb]);
#pragma unroll
            for (int u = 0; u < RW; ++u) v[u][t] = c;
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            bf16x8_t xa[TM], b[RW];
#pragma unroll
            for (int t = 0; t < TM; ++t)
              xa[t] = as_bf16x8(xt[e * XT + (16 * t + l16) * 16 + ((4 * kb + j) ^ l16)]);
#pragma unroll
            for (int u = 0; u < RW; ++u)
              b[u] = weights24(j == 0 ? w[p][u].x : j == 1 ? w[p][u].y : j == 2 ? w[p][u].z : w[p][u].w);
#pragma unroll
            for (int u = 0; u < RW; ++u)
#pragma unroll
              for (int t = 0; t < TM; ++t)
                v[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[t], b[u], v[u][t], 0, 0, 0);
          }
#pragma unroll
          for (int u = 0; u < RW; ++u) load_w(p, u, i + P);
#pragma unroll
          for (int u = 0; u < RW; ++u)
#pragma unroll
            for (int t = 0; t < TM; ++t)
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[u][t][r] = fmaf(sf[u], v[u][t][r], acc[u][t][r]);
        }
        __syncthreads();
      }
    }
  }

  // the K parts' sums, in order, on part 0
  if constexpr (KS > 1) {
    constexpr int F = RW * TM * 4;
    float* red = reinterpret_cast<float*>(gemm_lds) + lane;
    if (ks > 0) {
#pragma unroll
      for (int u = 0; u < RW; ++u)
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            red[((wave - 4) * F + (u * TM + t) * 4 + r) * 64] = acc[u][t][r];
    }
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int k = 1; k < KS; ++k)
#pragma unroll
      for (int u = 0; u < RW; ++u)
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[u][t][r] += red[((4 * (k - 1) + wr) * F + (u * TM + t) * 4 + r) * 64];
  }
  float seen[RW] = {};
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int u = 0; u < RW; ++u) watch(seen[u], acc[u][t][r]);
#pragma unroll
  for (int u = 1; u < RW; ++u) seen[0] += seen[u];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tok = tok0 + 16 * t + 4 * kb + r;
      if (tok < M && l16 < N) {
#pragma unroll
        for (int u = 0; u < RW; u += GU ? 2 : 1) {
          uint32_t v = f32_to_bf16(acc[u][t][r]);
          if constexpr (GU) v = swiglu_bf16(v, f32_to_bf16(acc[u + 1][t][r]));
          out[(size_t)tok * N + tile_row(u) + l16] = (uint16_t)v;
        }
      }
    }
  if (seen[0] != 0.f && l16 < N)
    for (int e = 0; e < TM * 4 * RW; e += GU ? 2 : 1) {
      const int u = e % RW, tr = e / RW;
      const int tok = tok0 + 16 * (tr >> 2) + 4 * kb + (tr & 3);
      if (tok < M)
        redo_output<GU>(qw, sc, qw_up, sc_up, x, out, N, K, tile_row(u) + l16, tok);
    }
}

constexpr size_t gemm_lds_bytes(int rw, int ks, int ngroups) {
  const size_t x = (size_t)ks * 2 * kTileTokens * (256 + 4) + (size_t)64 * rw * ngroups * 2;
  const size_t red = (size_t)(ks - 1) * 4 * rw * kTileTokens * 64;
  return x > red ? x : red;
}

template <int RW, int KS, bool GU>
int launch_gemm(const GemmArgs& a, hipStream_t s) {
  static std::atomic<uint64_t> granted{0};
  if (const int st = allow_lds(
          granted, reinterpret_cast<const void*>(&int4_gemm_kernel<RW, KS, GU>), (int)kGemmLds))
    return st;
  constexpr int kRows = GU ? 32 * RW : 64 * RW;
  const int rbs = (a.N + kRows - 1) / kRows, tbs = (a.M + kTileTokens - 1) / kTileTokens;
  const unsigned grid = (unsigned)((rbs + kXcds - 1) / kXcds * kXcds) * (unsigned)tbs;
  hipLaunchKernelGGL((int4_gemm_kernel<RW, KS, GU>), dim3(grid), dim3(KS * 256),
                     gemm_lds_bytes(RW, KS, a.K / kGroupSize), s, a.qw, a.sc, a.qw_up, a.sc_up, a.x,
                     a.out, a.M, a.N, a.K, rbs, tbs);
  return hip_status(hipGetLastError());
}

// The kernel for a product (us measured on both sides of each line): up to 32
// tokens the split kernel.  Beyond, the tiled one once 128-row blocks give 160
// workgroups (12288 x 4096: 96 workgroups 28 against 19 split, 192 28 against
// 32): with two K parts, 8 waves a workgroup, while every CU gets at most one
// (25600 x 5120, 64 tokens, 200 workgroups: 35, with one part 41), else with one
// (100 tokens, 400 workgroups: 57, with two parts 63; 5120 x 8192, 400 tokens,
// 280 workgroups: two parts 93), and with four row tiles per wave from 1024
// workgroups of them (25600 x 5120: 333 tokens, 600 of them, 148 against 132
// with two; 2048 tokens, 3200 of them, 639 against 718).
// Gate and up with the SwiGLU between them (GU) follow the same lines with
// their rows counted together; us against the two products and dip_swiglu:
// 25600 x 5120, 7 tokens 50 -> 44, 32 64 -> 57, 64 75 -> 61, 333 274 -> 240;
// 12288 x 4096, 200 tokens 97 -> 70, 333 131 -> 106; 3072 x 1024, 16 tokens 12
// -> 5.
template <bool GU>
int launch_int4_gemm(const GemmArgs& a, hipStream_t s) {
  if (a.M <= 16) return launch_split_tokens<1, GU>(a, s);
  const long long tbs = (a.M + kTileTokens - 1) / kTileTokens;
  const long long wgs2 = (a.rows() + 127) / 128 * tbs, wgs4 = (a.rows() + 255) / 256 * tbs;
  const int cus = device_cus(), ngroups = a.K / kGroupSize;
  if (a.M <= 32 || 8 * wgs2 < 5 * cus || !scales_by_dword(a) ||
      gemm_lds_bytes(2, 2, ngroups) > kGemmLds)
    return launch_split_tokens<2, GU>(a, s);
  if (wgs4 >= 4 * cus && gemm_lds_bytes(4, 1, ngroups) <= kGemmLds / 2)
    return launch_gemm<4, 1, GU>(a, s);
  if (wgs2 > cus) return launch_gemm<2, 1, GU>(a, s);
  return launch_gemm<2, 2, GU>(a, s);
}

// ---------------------------------------------------------------------------
// Transposed layout: out[M, N] = bf16( x[M, K] . W[K, N] ) with W stored as
// rows of K (qweight int8 [K, N/2], scales bf16 [K, N/128]): the transposed
// down matrix down_t of the dense route's h @ down_t
// (dip_stream_predispatch.py:213-215).  The scale varies along k here, so
// each weight becomes the reference's bf16(q * s) (qlinear.dequantize's
// rounding, exact to it) in registers:
//   * a wave owns 128 columns (one scale group), lane l16 the 8 columns 8 l16 ..:
//     a dword of each row.  An MFMA slice is 32 rows; the lane quarter kb loads
//     rows 8 kb .. + 7 (64 contiguous bytes of each row), and column c of the
//     16 lanes' 8 is one 16-column operand whose k pairs are two rows' values
//     rounded by one v_cvt_pk_bf16_f32: the transposition costs nothing;
//   * q * s: a nibble in the low mantissa bits of an fp16 1024.0 is 1032 + q (or
//     1152 + 16 q, four bits higher), read as fp16 by v_fma_mix_f32, which
//     multiplies by s and takes 1032 s (72 s) away with one rounding of an
//     exactly representable result: 17 instructions per 8 weights.  Scales of
//     2^118 or more, infinite or NaN, take plain products instead;
//   * x comes from memory as operands, 64 contiguous bytes of each token, so
//     nothing is staged and the loop has no barrier;
//   * a row's four factors are read from LDS, 256 rows of them prepared at a
//     time by the wave itself.
// A workgroup is 2 such column blocks (whole 128-byte lines) times 4 parts of
// K, added through LDS; blockIdx.z splits K further, its fp32 partials added in
// a fixed order by int4_gemm_t_reduce_kernel.  Bound by instruction issue (136
// vector instructions to 8 TM MFMAs a slice).  25600 x 5120: 2 tokens 63 -> 32
// us, 32 tokens 112 -> 39 us, 64 tokens 201 -> 49 us (before: values transposed
// through LDS a barrier at a time, 64 columns a workgroup), 333 tokens 143 us
// (dequantize and the library's product: 233), 768 tokens 263 us (363), 900
// tokens 515 us (408).
// ---------------------------------------------------------------------------
constexpr int kGemmTThreads = 512;
constexpr int kGemmTCols = 256;  // columns of a workgroup
constexpr int kGemmTParts = 4;   // K parts of a workgroup
constexpr int kChunkSlices = 8;  // slices per round of prepared factors

// fp16 half H of v times a plus c, in fp32.
template <int H>
DIP_DEV float fma_mix(uint32_t v, float a, float c) {
  float r;
  if (H == 0)
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[1,0,0]"
        : "=v"(r) : "v"(v), "v"(a), "v"(c));
  else
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "=v"(r) : "v"(v), "v"(a), "v"(c));
  return r;
}

// The 8 columns' q * s of one row; f = (s, s / 16, -1032 s, -72 s).
template <bool PLAIN>
DIP_DEV void row_values(uint32_t w, const float4& f, float v[8]) {
  if constexpr (PLAIN) {
#pragma unroll
    for (int p = 0; p < 8; ++p) v[p] = (float)(int)__builtin_amdgcn_sbfe(w, 4 * p, 4) * f.x;
    return;
  }
  const uint32_t t = w >> 8;
  const uint32_t a = (w & 0x000F000Fu) ^ 0x64086408u, b = (w & 0x00F000F0u) ^ 0x64806480u;
  const uint32_t c = (t & 0x000F000Fu) ^ 0x64086408u, d = (t & 0x00F000F0u) ^ 0x64806480u;
  v[0] = fma_mix<0>(a, f.x, f.z);
  v[4] = fma_mix<1>(a, f.x, f.z);
  v[1] = fma_mix<0>(b, f.y, f.w);
  v[5] = fma_mix<1>(b, f.y, f.w);
  v[2] = fma_mix<0>(c, f.x, f.z);
  v[6] = fma_mix<1>(c, f.x, f.z);
  v[3] = fma_mix<0>(d, f.y, f.w);
  v[7] = fma_mix<1>(d, f.y, f.w);
}

// A lane's 8 rows x 8 columns as 8 operands.
template <bool PLAIN>
DIP_DEV void slice_operands(const uint32_t w[8], const float4* f, bf16x8_t b[8]) {
  uint32_t r[8][4];
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    float v0[8], v1[8];
    row_values<PLAIN>(w[i], f[i], v0);
    row_values<PLAIN>(w[i + 1], f[i + 1], v1);
#pragma unroll
    for (int c = 0; c < 8; ++c) r[c][i / 2] = f32x2_to_bf16x2_nan(v0[c], v1[c]);
  }
#pragma unroll
  for (int c = 0; c < 8; ++c)
    b[c] = __builtin_bit_cast(bf16x8_t, u32x4_t{r[c][0], r[c][1], r[c][2], r[c][3]});
}

template <int TM>
__global__ __launch_bounds__(kGemmTThreads, 2) void int4_gemm_t_kernel(
    const int8_t* __restrict__ qw, const uint16_t* __restrict__ sc, const uint16_t* __restrict__ x,
    uint16_t* __restrict__ out, float* __restrict__ part, int M, int N, int K, int part_slices) {
  constexpr int D = TM == 4 ? 2 : 4;  // slices of weights in flight
  constexpr int DX = 2;               // slices of x in flight
  constexpr int F = 8 * TM * 4;       // sums of a lane
  extern __shared__ __align__(16) float4 gemmt_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int kb = lane >> 4, l16 = lane & 15;
  const int col0 = blockIdx.x * kGemmTCols + (wave & 1) * 128;
  const int kp = wave >> 1;
  const int tok0 = blockIdx.y * (16 * TM);
  const int slices = (K + 31) / 32;
  const int s0 = min(((int)blockIdx.z * kGemmTParts + kp) * part_slices, slices);
  const int s1 = col0 < N ? min(s0 + part_slices, slices) : s0;
  const size_t row_bytes = (size_t)(N >> 1);
  const int ngroups_n = N >> 7;
  float4* fac = gemmt_lds + wave * (32 * kChunkSlices);

  // K is a multiple of 8, so a lane's 8 rows are all inside or all past the end
  const int tail8 = K - 32 * (slices - 1);  // rows of the last slice
  const bool in_tail = 8 * kb < tail8;
  const uint32_t off_full = 8u * kb * (uint32_t)row_bytes + 4u * l16;
  const uint32_t off_tail = (in_tail ? 8u * kb : 0u) * (uint32_t)row_bytes + 4u * l16;
  const int8_t* wbase = qw + (col0 >> 1);
  const char* xp[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t)
    xp[t] = reinterpret_cast<const char*>(x + (size_t)min(tok0 + 16 * t + l16, M - 1) * K + 8 * kb);
  uint32_t w[D][8], sreg[4];
  uint4 xr[DX][TM];
  auto load_w = [&](int d, int s) {
    const int8_t* b = wbase + (size_t)s * 32 * row_bytes;
    const uint32_t o = s == slices - 1 ? off_tail : off_full;
#pragma unroll
    for (int i = 0; i < 8; ++i) w[d][i] = *reinterpret_cast<const uint32_t*>(b + i * row_bytes + o);
  };
  auto load_x = [&](int d, int s) {
    const bool in = s < slices - 1 || in_tail;
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      xr[d][t] = make_uint4(0, 0, 0, 0);
      if (in) xr[d][t] = *reinterpret_cast<const uint4*>(xp[t] + (size_t)s * 64);
    }
  };
  auto load_s = [&](int s) {  // the factors' scales of rows 32 s .. + 255
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = min(32 * s + 64 * e + lane, K - 1);
      sreg[e] = sc[(size_t)row * ngroups_n + (col0 >> 7)];
    }
  };
  floatx4 acc[8][TM];
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[c][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  if (s0 < s1) {
    load_s(s0);
#pragma unroll
    for (int d = 0; d < DX; ++d) load_x(d, min(s0 + d, s1 - 1));
#pragma unroll
    for (int d = 0; d < D; ++d) load_w(d, min(s0 + d, s1 - 1));
  }
  for (int sb = s0; sb < s1; sb += kChunkSlices) {
    bool plain = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 32 * sb + 64 * e + lane;
      const float f = row < K ? bf16_to_f32(sreg[e]) : 0.f;  // rows past the end weigh nothing
      plain |= row < K && (sreg[e] & 0x7FFFu) >= 0x7A80u;
      fac[64 * e + lane] = make_float4(f, f * 0.0625f, f * -1032.0f, f * -72.0f);
    }
    plain = __any(plain);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    load_s(min(sb + kChunkSlices, slices - 1));
    for (int q0 = 0; q0 < kChunkSlices; q0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int s = sb + q0 + d;
        if (s < s1) {
          bf16x8_t b[8];
          const float4* fr = fac + 32 * (q0 + d) + 8 * kb;
          if (plain) slice_operands<true>(w[d], fr, b);
          else slice_operands<false>(w[d], fr, b);
          load_w(d, min(s + D, s1 - 1));
          bf16x8_t xa[TM];
#pragma unroll
          for (int t = 0; t < TM; ++t) xa[t] = as_bf16x8(xr[d % DX][t]);
#pragma unroll
          for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int t = 0; t < TM; ++t)
              acc[c][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[t], b[c], acc[c][t], 0, 0, 0);
          load_x(d % DX, min(s + DX, s1 - 1));
        }
      }
    }
    // this round's reads of the factors before the next round's writes
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }

  // (part 0 + part 2) + (part 1 + part 3)
  float* red = reinterpret_cast<float*>(gemmt_lds);
#pragma unroll
  for (int h = kGemmTParts / 2; h >= 1; h /= 2) {
    __syncthreads();
    if (kp >= h && kp < 2 * h) {
#pragma unroll
      for (int c = 0; c < 8; ++c)
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            red[((wave - 2 * h) * F + (c * TM + t) * 4 + r) * 64 + lane] = acc[c][t][r];
    }
    __syncthreads();
    if (kp < h) {
#pragma unroll
      for (int c = 0; c < 8; ++c)
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[c][t][r] += red[(wave * F + (c * TM + t) * 4 + r) * 64 + lane];
    }
  }
  if (kp > 0 || col0 >= N) return;
  const bool wide = (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tok = tok0 + 16 * t + 4 * kb + r;
      if (tok >= M) continue;
      if (part) {
        float4* o = reinterpret_cast<float4*>(part + ((size_t)blockIdx.z * M + tok) * N + col0 + 8 * l16);
        o[0] = make_float4(acc[0][t][r], acc[1][t][r], acc[2][t][r], acc[3][t][r]);
        o[1] = make_float4(acc[4][t][r], acc[5][t][r], acc[6][t][r], acc[7][t][r]);
      } else {
        uint16_t* o = out + (size_t)tok * N + col0 + 8 * l16;
        uint32_t v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = f32x2_to_bf16x2(acc[2 * c][t][r], acc[2 * c + 1][t][r]);
        if (wide) {
          *reinterpret_cast<uint4*>(o) = make_uint4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
          for (int c = 0; c < 8; ++c) o[c] = (uint16_t)(v[c / 2] >> (16 * (c & 1)));
        }
      }
    }
}

constexpr size_t gemm_t_lds_bytes(int tm) {
  const size_t red = (size_t)4 * 8 * tm * 4 * 256, fac = (size_t)8 * 32 * kChunkSlices * 16;
  return red > fac ? red : fac;
}

// Sum of the K split's fp32 partials in split order, rounded to bf16: four
// values a thread (M * N is a multiple of 128).
__global__ __launch_bounds__(256) void int4_gemm_t_reduce_kernel(const float* __restrict__ part,
                                                                 uint16_t* __restrict__ out,
                                                                 size_t mn, int splits) {
  const bool wide = (reinterpret_cast<uintptr_t>(out) & 7u) == 0;
  for (size_t e = 4 * ((size_t)blockIdx.x * 256 + threadIdx.x); e < mn; e += 4 * (size_t)gridDim.x * 256) {
    float4 v = *reinterpret_cast<const float4*>(part + e);
#pragma unroll 4
    for (int z = 1; z < splits; ++z) {
      const float4 p = *reinterpret_cast<const float4*>(part + (size_t)z * mn + e);
      v.x += p.x;
      v.y += p.y;
      v.z += p.z;
      v.w += p.w;
    }
    const uint32_t lo = f32x2_to_bf16x2(v.x, v.y), hi = f32x2_to_bf16x2(v.z, v.w);
    if (wide) {
      *reinterpret_cast<uint2*>(out + e) = make_uint2(lo, hi);
    } else {
      out[e] = (uint16_t)lo;
      out[e + 1] = (uint16_t)(lo >> 16);
      out[e + 2] = (uint16_t)hi;
      out[e + 3] = (uint16_t)(hi >> 16);
    }
  }
}

template <int TM>
int launch_gemm_t(const int8_t* qw, const uint16_t* sc, const uint16_t* x, uint16_t* out, float* part,
                  int M, int N, int K, int splits, int part_slices, hipStream_t s) {
  static std::atomic<uint64_t> granted{0};
  if (const int st = allow_lds(
          granted, reinterpret_cast<const void*>(&int4_gemm_t_kernel<TM>), (int)kGemmLds))
    return st;
  const dim3 grid((unsigned)((N + kGemmTCols - 1) / kGemmTCols), (unsigned)((M + 16 * TM - 1) / (16 * TM)),
                  (unsigned)splits);
  hipLaunchKernelGGL(int4_gemm_t_kernel<TM>, grid, dim3(kGemmTThreads), gemm_t_lds_bytes(TM), s, qw, sc,
                     x, out, part, M, N, K, part_slices);
  return hip_status(hipGetLastError());
}

}  // namespace
}  // namespace dip

using namespace dip;

extern "C" int dip_int4_gemm(const int8_t* qweight, const uint16_t* scales, const uint16_t* x,
                             uint16_t* out, int64_t m, int64_t out_features,
                             int64_t in_features, void* stream) {
  if (!qweight || !scales) return DIP_ERR_NULL;
  if (m < 0 || out_features <= 0 || in_features <= 0 || in_features % kGroupSize != 0 ||
      out_features > INT32_MAX || in_features > (1 << 20) || m > 64 * 65535 ||
      m * out_features > ((int64_t)1 << 40))
    return DIP_ERR_SHAPE;
  if (m == 0) return DIP_OK;  // x and out may be NULL then
  if (!x || !out) return DIP_ERR_NULL;
  if (!aligned16(qweight) || !aligned16(x)) return DIP_ERR_ALIGN;
  return launch_int4_gemm<false>(GemmArgs{qweight, scales, nullptr, nullptr, x, out, (int)m,
                                          (int)out_features, (int)in_features},
                                 (hipStream_t)stream);
}

extern "C" int dip_int4_gemm_swiglu(const int8_t* gate_qw, const uint16_t* gate_sc,
                                    const int8_t* up_qw, const uint16_t* up_sc, const uint16_t* x,
                                    uint16_t* out, int64_t m, int64_t inter, int64_t hidden,
                                    void* stream) {
  if (!gate_qw || !gate_sc || !up_qw || !up_sc) return DIP_ERR_NULL;
  if (m < 0 || inter <= 0 || hidden <= 0 || hidden % kGroupSize != 0 || inter > INT32_MAX ||
      hidden > (1 << 20) || m > 64 * 65535 || m * inter > ((int64_t)1 << 39))
    return DIP_ERR_SHAPE;
  if (m == 0) return DIP_OK;
  if (!x || !out) return DIP_ERR_NULL;
  if (!aligned16(gate_qw) || !aligned16(up_qw) || !aligned16(x)) return DIP_ERR_ALIGN;
  return launch_int4_gemm<true>(
      GemmArgs{gate_qw, gate_sc, up_qw, up_sc, x, out, (int)m, (int)inter, (int)hidden},
      (hipStream_t)stream);
}

namespace {
int gemm_t_token_tiles(int64_t m) { return m <= 16 ? 1 : (m <= 32 ? 2 : 4); }

// K split of dip_int4_gemm_t over blockIdx.z: as many as give every CU one
// workgroup (8 waves fill it; us for 25600 x 5120: 64 tokens, 20 workgroups a
// split, 12 splits 49, 10: 53, 16: 72; 200 tokens 3 splits 103, 4: 146; 333
// tokens 2 splits 143, 3: 188).  Where one round of workgroups would leave a
// third of the chip idle and two rounds would not, two (512 tokens, 160
// workgroups: one split 279, three 210).
int gemm_t_splits(int64_t m, int64_t n, int64_t k) {
  const int64_t tm = gemm_t_token_tiles(m);
  const int64_t tiles = ((n + kGemmTCols - 1) / kGemmTCols) * ((m + 16 * tm - 1) / (16 * tm));
  const int64_t most = std::min<int64_t>(16, (k + 32 * kGemmTParts - 1) / (32 * kGemmTParts));
  const int64_t cus = device_cus(), two = 2 * cus / tiles;
  int64_t z = std::max<int64_t>(1, cus / tiles);
  if (3 * z * tiles < 2 * cus && 20 * two * tiles >= 17 * 2 * cus) z = two;
  return (int)std::max<int64_t>(1, std::min(z, most));
}
}  // namespace

extern "C" size_t dip_int4_gemm_t_workspace_size(int64_t m, int64_t out_features,
                                                 int64_t in_features) {
  if (m <= 0 || out_features <= 0 || in_features <= 0) return 0;
  const int splits = gemm_t_splits(m, out_features, in_features);
  return splits > 1 ? (size_t)splits * (size_t)m * (size_t)out_features * sizeof(float) : 0;
}

extern "C" int dip_int4_gemm_t(const int8_t* qweight_t, const uint16_t* scales_t,
                               const uint16_t* x, uint16_t* out, int64_t m, int64_t out_features,
                               int64_t in_features, void* workspace, size_t ws_bytes,
                               void* stream) {
  if (!qweight_t || !scales_t) return DIP_ERR_NULL;
  if (m < 0 || out_features <= 0 || in_features <= 0 || out_features % kGroupSize != 0 ||
      in_features % 8 != 0 || out_features > (1 << 20) || in_features > INT32_MAX / 2 ||
      m > 64 * 65535 || m * out_features > ((int64_t)1 << 40))
    return DIP_ERR_SHAPE;
  if (m == 0) return DIP_OK;
  if (!x || !out) return DIP_ERR_NULL;
  if (!aligned16(qweight_t) || !aligned16(x)) return DIP_ERR_ALIGN;
  const int M = (int)m, N = (int)out_features, K = (int)in_features;
  int splits = gemm_t_splits(m, out_features, in_features);
  const size_t need = splits > 1 ? (size_t)splits * (size_t)M * (size_t)N * sizeof(float) : 0;
  if (need > 0 && (!workspace || ws_bytes < need)) return DIP_ERR_WORKSPACE;
  if (splits > 1 && !aligned16(workspace)) return DIP_ERR_ALIGN;
  const int slices = (K + 31) / 32;
  const int part_slices = (slices + splits * kGemmTParts - 1) / (splits * kGemmTParts);
  float* part = splits > 1 ? static_cast<float*>(workspace) : nullptr;
  hipStream_t s = (hipStream_t)stream;
  const int tm = gemm_t_token_tiles(m);
  const int st =
      tm == 1 ? launch_gemm_t<1>(qweight_t, scales_t, x, out, part, M, N, K, splits, part_slices, s)
      : tm == 2 ? launch_gemm_t<2>(qweight_t, scales_t, x, out, part, M, N, K, splits, part_slices, s)
                : launch_gemm_t<4>(qweight_t, scales_t, x, out, part, M, N, K, splits, part_slices, s);
  if (st) return st;
  if (splits > 1) {
    const size_t mn = (size_t)M * N;
    const unsigned blocks = (unsigned)std::min<size_t>((mn / 4 + 255) / 256, 4096);
    hipLaunchKernelGGL(int4_gemm_t_reduce_kernel, dim3(blocks), dim3(256), 0, s, part, out, mn,
                       splits);
  }
  return hip_status(hipGetLastError());
}
