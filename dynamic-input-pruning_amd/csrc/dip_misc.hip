// dip_misc.hip — cache-aware hit/miss assembly and miss stream, SwiGLU, row dequantisation, the
// host-side miss gather, the one-call resident MLP decode step and the
// library's status helpers.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include "dip_common.h"
#include "dip_host_pool.h"
#include "dip_internal.h"

namespace dip {

// ---------------------------------------------------------------------------
// Cache-aware assembly (dip_ca.py:137-171).  One workgroup, whose time is its
// chains of dependent loads (idx, then the slot): each wave owns a contiguous
// run of idx, 64 channels a step and kAsmUnroll steps in flight, counts its
// hits by ballots, and a scan over the waves gives every element its place in
// [hits in idx order, misses in idx order].  7373 channels: 20.9 us with a run
// of single loads per thread, 8.4 us so.
// ---------------------------------------------------------------------------
namespace {
constexpr int kAsmThreads = 1024;
constexpr int kAsmWaves = kAsmThreads / 64;
constexpr int kAsmUnroll = 8;

// The channels at j0 + 64 u of a wave's run [.., end) and their slots, -1
// where not resident.
DIP_DEV void asm_load(const int64_t* id2slot, const int32_t* idx, int inter, uint32_t j0,
                      uint32_t end, int c[kAsmUnroll], int slot[kAsmUnroll]) {
#pragma unroll
  for (int u = 0; u < kAsmUnroll; ++u) {
    const uint32_t j = j0 + 64 * u;
    c[u] = j < end ? idx[j] : -1;
  }
#pragma unroll
  for (int u = 0; u < kAsmUnroll; ++u)
    slot[u] = (unsigned)c[u] < (unsigned)inter ? (int)max(id2slot[c[u]], (int64_t)-1) : -1;
}
}  // namespace

__global__ __launch_bounds__(kAsmThreads) void ca_assemble_kernel(
    const int64_t* __restrict__ id2slot, const int32_t* __restrict__ idx, int inter, int k,
    int32_t* __restrict__ combined, int32_t* __restrict__ src, int32_t* __restrict__ row,
    int32_t* __restrict__ miss_ids, int32_t* __restrict__ counts) {
  __shared__ int wave_hits[kAsmWaves];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  // (unsigned: a step past the last of 2^31 - 1 channels does not wrap)
  const uint32_t steps = ((uint32_t)k + kAsmThreads - 1) / kAsmThreads;  // 64 channels each
  const uint32_t beg = min((uint32_t)k, wave * steps * 64);
  const uint32_t end = min((uint32_t)k, beg + steps * 64);
  int c[kAsmUnroll], slot[kAsmUnroll];

  int hits = 0;
  for (uint32_t s = 0; s < steps; s += kAsmUnroll) {
    asm_load(id2slot, idx, inter, beg + s * 64 + lane, end, c, slot);
#pragma unroll
    for (int u = 0; u < kAsmUnroll; ++u) hits += __popcll(__ballot(slot[u] >= 0));
  }
  if (lane == 0) wave_hits[wave] = hits;
  __syncthreads();
  int n_hit = 0, hit_pos = 0;  // of all waves; of the waves before this one
#pragma unroll
  for (int w = 0; w < kAsmWaves; ++w) {
    const int v = wave_hits[w];
    n_hit += v;
    hit_pos += w < wave ? v : 0;
  }
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  for (uint32_t s = 0; s < steps; s += kAsmUnroll) {
    const uint32_t j0 = beg + s * 64 + lane;
    // (a run of one pass is still in the registers)
    if (steps > kAsmUnroll) asm_load(id2slot, idx, inter, j0, end, c, slot);
#pragma unroll
    for (int u = 0; u < kAsmUnroll; ++u) {
      const uint32_t j = j0 + 64 * u;
      const uint64_t m = __ballot(slot[u] >= 0);
      const int before = hit_pos + __popcll(m & below);  // hits before j
      hit_pos += __popcll(m);
      if (j >= end) continue;
      if (slot[u] >= 0) {
        combined[before] = c[u];
        src[before] = 0;
        row[before] = slot[u];
      } else {
        const int miss_rank = (int)j - before;
        combined[n_hit + miss_rank] = c[u];
        src[n_hit + miss_rank] = 1;
        row[n_hit + miss_rank] = miss_rank;
        miss_ids[miss_rank] = c[u];
      }
    }
  }
  if (threadIdx.x == 0) {
    counts[0] = n_hit;
    counts[1] = k - n_hit;
  }
}

// ---------------------------------------------------------------------------
// Miss rows straight from pinned host memory (the index_select and copies of
// dip_ca.py:146-156 as one kernel).  Bound by the host link: the rows of all
// pieces are one run of vectors (a channel's up row, up scales, down row and
// down scales behind each other), dealt to the grid in order, so that
// neighbouring lanes ask the link for neighbouring bytes, and the device's
// own count ends the run: the host learns it only afterwards.  5161 rows of
// 4224 bytes 420 us, 52 GB/s, the rate of a plain copy over the link (64 to
// 1024 blocks and 1 to 8 vectors a lane are within 4 %).  A layer's whole
// token, 12288 x 4096, 5161 misses: 759 us with host threads gathering into
// staging for DMA copies, 487 us so.
// ---------------------------------------------------------------------------
constexpr int kStreamPieces = 8;
constexpr int kStreamBlocks = 256;
constexpr int kStreamUnroll = 4;

struct StreamArgs {
  const char* src[kStreamPieces];
  char* dst[kStreamPieces];
  uint32_t row_bytes[kStreamPieces];
  uint32_t end[kStreamPieces];    // vectors of the pieces up to this one, in a row
  uint32_t shift[kStreamPieces];  // log2 of the piece's vector bytes
  int npieces;
  uint32_t per_row;               // vectors of all pieces in a row
};

__global__ __launch_bounds__(256) void stream_rows_kernel(StreamArgs a,
                                                          const int32_t* __restrict__ ids,
                                                          const int32_t* __restrict__ count,
                                                          uint32_t max_rows, uint32_t src_rows) {
  const uint32_t n = (uint32_t)min(max(*count, 0), (int)max_rows);
  const uint32_t total = n * a.per_row;
  const uint32_t step = gridDim.x * blockDim.x;
  for (uint32_t e0 = blockIdx.x * blockDim.x + threadIdx.x; e0 < total;
       e0 += kStreamUnroll * step) {
    uint4 v[kStreamUnroll];
    char* to[kStreamUnroll];
    uint32_t sh[kStreamUnroll];
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u) {
      const uint32_t e = e0 + u * step;
      to[u] = nullptr;
      v[u] = make_uint4(0, 0, 0, 0);
      if (e >= total) continue;
      const uint32_t i = e / a.per_row, o = e - i * a.per_row;
      int p = 0;
      while (o >= a.end[p]) ++p;
      const uint32_t off = (o - (p ? a.end[p - 1] : 0u)) << a.shift[p];
      const uint32_t id = (uint32_t)ids[i];
      sh[u] = a.shift[p];
      to[u] = a.dst[p] + (size_t)i * a.row_bytes[p] + off;
      // an id past the matrix leaves a row of zeros
      if (id >= src_rows) continue;
      const char* from = a.src[p] + (size_t)id * a.row_bytes[p] + off;
      switch (sh[u]) {
        case 4: v[u] = *reinterpret_cast<const uint4*>(from); break;
        case 3: *reinterpret_cast<uint2*>(&v[u]) = *reinterpret_cast<const uint2*>(from); break;
        case 2: v[u].x = *reinterpret_cast<const uint32_t*>(from); break;
        case 1: v[u].x = *reinterpret_cast<const uint16_t*>(from); break;
        default: v[u].x = *reinterpret_cast<const uint8_t*>(from);
      }
    }
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u) {
      if (!to[u]) continue;
      switch (sh[u]) {
        case 4: *reinterpret_cast<uint4*>(to[u]) = v[u]; break;
        case 3: *reinterpret_cast<uint2*>(to[u]) = make_uint2(v[u].x, v[u].y); break;
        case 2: *reinterpret_cast<uint32_t*>(to[u]) = v[u].x; break;
        case 1: *reinterpret_cast<uint16_t*>(to[u]) = (uint16_t)v[u].x; break;
        default: *reinterpret_cast<uint8_t*>(to[u]) = (uint8_t)v[u].x;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Row dequantisation.  Bound by the stores (bf16: 4 bytes out for each byte
// in).  A thread turns one dword (8 columns) into one or two 128-bit stores,
// kDqUnroll dwords apart by a block, so that a wave stores whole kilobytes and
// has its loads in flight together; each value is one SDWA convert and one
// multiply.  Rows in order are one flat run (the scale of dword e is e / 16).
// 25600 x 5120 to bf16 (332 MB): 174 us with one byte per thread and two
// 16-bit stores; 50 us in this form, 23 us for 5120 x 8192.
// ---------------------------------------------------------------------------
constexpr int kDqUnroll = 4;

// 8 nibbles of w (each converted as 16 times itself) times the scale s16 / 16.
DIP_DEV void dequant8(uint32_t w, float s16, float v[8]) {
  const uint32_t lo = (w << 4) & 0xF0F0F0F0u, hi = w & 0xF0F0F0F0u;
  v[0] = cvt_sbyte<0>(lo) * s16;
  v[1] = cvt_sbyte<0>(hi) * s16;
  v[2] = cvt_sbyte<1>(lo) * s16;
  v[3] = cvt_sbyte<1>(hi) * s16;
  v[4] = cvt_sbyte<2>(lo) * s16;
  v[5] = cvt_sbyte<2>(hi) * s16;
  v[6] = cvt_sbyte<3>(lo) * s16;
  v[7] = cvt_sbyte<3>(hi) * s16;
}

template <int MODE>
DIP_DEV void store_dequant8(uint32_t w, uint32_t s, bool bad, void* out, size_t dword) {
  float v[8];
  dequant8(w, bf16_to_f32(s) * 0.0625f, v);
  if (bad) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __builtin_nanf("");
  }
  if constexpr (MODE == 0) {
    float4* o = reinterpret_cast<float4*>(out) + 2 * dword;
    o[0] = make_float4(v[0], v[1], v[2], v[3]);
    o[1] = make_float4(v[4], v[5], v[6], v[7]);
  } else {
    reinterpret_cast<uint4*>(out)[dword] =
        make_uint4(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]),
                   f32x2_to_bf16x2(v[4], v[5]), f32x2_to_bf16x2(v[6], v[7]));
  }
}

template <int MODE>
__global__ __launch_bounds__(256) void dequant_flat_kernel(const uint32_t* __restrict__ qw,
                                                           const uint16_t* __restrict__ sc,
                                                           void* __restrict__ out, size_t ndwords) {
  constexpr size_t kSpan = 256 * kDqUnroll;
  for (size_t b = (size_t)blockIdx.x * kSpan; b < ndwords; b += (size_t)gridDim.x * kSpan) {
    uint32_t w[kDqUnroll], s[kDqUnroll];
#pragma unroll
    for (int u = 0; u < kDqUnroll; ++u) {
      const size_t e = b + threadIdx.x + 256 * u, c = e < ndwords ? e : ndwords - 1;
      w[u] = qw[c];
      s[u] = sc[c >> 4];
    }
#pragma unroll
    for (int u = 0; u < kDqUnroll; ++u) {
      const size_t e = b + threadIdx.x + 256 * u;
      if (e < ndwords) store_dequant8<MODE>(w[u], s[u], false, out, e);
    }
  }
}

// Rows through an id list: workgroup y takes rows y, y + gridDim.y, ...
template <int MODE>
__global__ __launch_bounds__(256) void dequant_gather_kernel(const uint32_t* __restrict__ qw,
                                                             const uint16_t* __restrict__ sc,
                                                             const int32_t* __restrict__ indices,
                                                             void* __restrict__ out, int n_out_rows,
                                                             int rows, int row_dwords) {
  for (int i = blockIdx.y; i < n_out_rows; i += gridDim.y) {
    const int id = indices[i];
    const bool bad = (unsigned)id >= (unsigned)rows;
    if (bad && rows == 0) {
      for (int c = blockIdx.x * 256 + threadIdx.x; c < row_dwords; c += gridDim.x * 256)
        store_dequant8<MODE>(0u, 0u, true, out, (size_t)i * row_dwords + c);
      continue;
    }
    const size_t r0 = (size_t)(bad ? 0 : id) * row_dwords;
    for (int c = blockIdx.x * 256 + threadIdx.x; c < row_dwords; c += gridDim.x * 256)
      store_dequant8<MODE>(qw[r0 + c], sc[(r0 + c) >> 4], bad, out, (size_t)i * row_dwords + c);
  }
}

// One byte per thread: buffers that are not aligned for the vector forms.
__global__ __launch_bounds__(256) void dequant_rows_kernel(
    const int8_t* __restrict__ qw, const uint16_t* __restrict__ sc,
    const int32_t* __restrict__ indices, void* __restrict__ out, int n_out_rows, int rows,
    int cols, int mode) {
  const int half = cols >> 1;
  const int ngroups = cols >> 7;
  const size_t total = (size_t)n_out_rows * half;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total;
       e += (size_t)gridDim.x * 256) {
    const int i = (int)(e / half);
    const int b = (int)(e % half);
    const int r = indices ? indices[i] : i;
    float v0, v1;
    if ((unsigned)r < (unsigned)rows) {
      const uint32_t byte = (uint8_t)qw[(size_t)r * half + b];
      const int q0 = (int)(byte & 0xFu) - (int)((byte & 0x8u) << 1);
      const int q1 = (int)(byte >> 4) - (int)((byte & 0x80u) >> 3);
      const float s = bf16_to_f32(sc[(size_t)r * ngroups + (2 * b) / kGroupSize]);
      v0 = (float)q0 * s;
      v1 = (float)q1 * s;
    } else {
      v0 = v1 = __builtin_nanf("");
    }
    const size_t o = (size_t)i * cols + 2 * (size_t)b;
    if (mode == 0) {
      reinterpret_cast<float*>(out)[o] = v0;
      reinterpret_cast<float*>(out)[o + 1] = v1;
    } else {
      reinterpret_cast<uint16_t*>(out)[o] = (uint16_t)f32_to_bf16(v0);
      reinterpret_cast<uint16_t*>(out)[o + 1] = (uint16_t)f32_to_bf16(v1);
    }
  }
}

}  // namespace dip

using namespace dip;

extern "C" const char* dip_status_string(int status) {
  switch (status) {
    case DIP_OK: return "ok";
    case DIP_ERR_NULL: return "a required pointer is NULL";
    case DIP_ERR_SHAPE: return "invalid or unsupported size";
    case DIP_ERR_ALIGN: return "pointer is not 16-byte aligned";
    case DIP_ERR_UNSUPPORTED: return "no kernel instantiation for this shape";
    case DIP_ERR_WORKSPACE: return "workspace missing or too small";
    case DIP_ERR_ARG: return "invalid argument";
    case DIP_ERR_SCRATCH: return "the shape needs more workspace than the no-alloc scratch holds";
    default: break;
  }
  if (status > 0) return hipGetErrorString((hipError_t)status);
  return "unknown status";
}

extern "C" int dip_version(void) { return DIP_VERSION; }

extern "C" int dip_timeline_read(int kernel, dip_wg_stamps* dst) {
  if (!dst) return DIP_ERR_NULL;
  if (kernel < DIP_STAMP_GATE || kernel > DIP_STAMP_REDUCE) return DIP_ERR_ARG;
#ifdef DIP_WG_STAMPS
  if (hipDeviceSynchronize() != hipSuccess) return hip_status(hipGetLastError());
#endif
  switch (kernel) {
    case DIP_STAMP_GATE: return timeline_read_rowdot(dst);
    case DIP_STAMP_TOPK: return timeline_read_topk(dst);
    case DIP_STAMP_DOWN: return timeline_read_down(0, dst);
    default: return timeline_read_down(1, dst);
  }
}

// ---------------------------------------------------------------------------
// Tuning table and device facts.
// ---------------------------------------------------------------------------
namespace {
int g_tune[DIP_TUNE_COUNT] = {0, 0, 8, 0, 1};  // [3]: not a knob
}  // namespace

int dip::tuning(int knob) { return g_tune[knob]; }

int dip::device_cus() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cache[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    cache[dev] = n;
  }
  return cache[dev];
}

extern "C" int dip_set_tuning(int knob, int value) {
  switch (knob) {
    case DIP_TUNE_ROWDOT_WGS_PER_CU:
      if (value < 0 || value > 16) return DIP_ERR_ARG;
      break;
    case DIP_TUNE_TOPK_STAMPS:
      if (value != 0 && value != 1) return DIP_ERR_ARG;
      break;
    case DIP_TUNE_SPEC_MARGIN:
      if (value < 0 || value > 1024) return DIP_ERR_ARG;
      break;
    case DIP_TUNE_ROW_TIERS:
      if (value != 0 && value != 1) return DIP_ERR_ARG;
      break;
    default:
      return DIP_ERR_ARG;
  }
  g_tune[knob] = value;
  return DIP_OK;
}

extern "C" int dip_get_tuning(int knob) {
  if (knob < 0 || knob >= DIP_TUNE_COUNT || knob == 3) return DIP_ERR_ARG;
  return g_tune[knob];
}

extern "C" int dip_ca_assemble(const int64_t* id2slot, const int32_t* idx, int32_t* combined,
                               int32_t* src, int32_t* row, int32_t* miss_ids, int32_t* counts,
                               int64_t inter, int64_t k, void* stream) {
  if (inter < 0 || k < 0 || inter > INT32_MAX || k > INT32_MAX) return DIP_ERR_SHAPE;
  if (!counts || !id2slot) return DIP_ERR_NULL;
  if (k > 0 && (!idx || !combined || !src || !row || !miss_ids)) return DIP_ERR_NULL;
  hipLaunchKernelGGL(ca_assemble_kernel, dim3(1), dim3(kAsmThreads), 0, (hipStream_t)stream,
                     id2slot, idx, (int)inter, (int)k, combined, src, row, miss_ids, counts);
  return hip_status(hipGetLastError());
}

extern "C" int dip_stream_rows(const void* const* src, void* const* dst, const int64_t* row_bytes,
                               int64_t npieces, const int32_t* ids, const int32_t* count,
                               int64_t max_rows, int64_t src_rows, void* stream) {
  if (npieces < 0 || npieces > kStreamPieces || max_rows < 0 || src_rows < 0 ||
      max_rows > INT32_MAX || src_rows > INT32_MAX)
    return DIP_ERR_SHAPE;
  if (npieces == 0 || max_rows == 0) return DIP_OK;
  if (!src || !dst || !row_bytes || !ids || !count) return DIP_ERR_NULL;
  StreamArgs a{};
  uint64_t per_row = 0;
  for (int p = 0; p < (int)npieces; ++p) {
    if (row_bytes[p] < 0 || row_bytes[p] > INT32_MAX) return DIP_ERR_SHAPE;
    if (row_bytes[p] == 0) continue;
    if (!src[p] || !dst[p]) return DIP_ERR_NULL;
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, src[p]) != hipSuccess) {
      (void)hipGetLastError();
      return DIP_ERR_UNSUPPORTED;
    }
    // (only pinned memory has both; a kernel may read no other)
    if (at.type != hipMemoryTypeHost || !at.devicePointer) return DIP_ERR_UNSUPPORTED;
    const void* from = at.devicePointer;
    // the widest vector that rows and both bases allow
    const uint64_t al = reinterpret_cast<uintptr_t>(from) | reinterpret_cast<uintptr_t>(dst[p]) |
                        (uint64_t)row_bytes[p] | 16u;
    const int q = a.npieces++;
    a.src[q] = static_cast<const char*>(from);
    a.dst[q] = static_cast<char*>(dst[p]);
    a.row_bytes[q] = (uint32_t)row_bytes[p];
    a.shift[q] = (uint32_t)__builtin_ctzll(al);
    per_row += (uint64_t)row_bytes[p] >> a.shift[q];
    a.end[q] = (uint32_t)per_row;
  }
  if (a.npieces == 0) return DIP_OK;
  // vector numbers, also those a stride past the last, stay within 32 bits
  const uint64_t slack = (uint64_t)kStreamUnroll * kStreamBlocks * 256;
  if (per_row > INT32_MAX || per_row * (uint64_t)max_rows + 2 * slack > UINT32_MAX)
    return DIP_ERR_SHAPE;
  a.per_row = (uint32_t)per_row;
  hipLaunchKernelGGL(stream_rows_kernel, dim3(kStreamBlocks), dim3(256), 0, (hipStream_t)stream, a,
                     ids, count, (uint32_t)max_rows, (uint32_t)src_rows);
  return hip_status(hipGetLastError());
}

// ---------------------------------------------------------------------------
// SwiGLU of a prompt's gate and up products, h = bf16(bf16(silu(g)) * u), with
// the roundings of the two torch ops it takes the place of.  Bound by memory
// beside expf and a division per value.  A block takes kSwigluUnroll runs of
// 256 vectors, all loaded first.  2048 x 25600 values 64 us (4.9 TB/s; the two
// ops 95), 333 x 12288 8.6 us (12.1).
// ---------------------------------------------------------------------------
namespace {
constexpr int kSwigluUnroll = 2;

DIP_DEV uint32_t swiglu2(uint32_t g, uint32_t u) {
  return swiglu_bf16(g & 0xFFFFu, u & 0xFFFFu) | (swiglu_bf16(g >> 16, u >> 16) << 16);
}

__global__ __launch_bounds__(256) void swiglu_kernel(const uint16_t* __restrict__ g,
                                                     const uint16_t* __restrict__ u,
                                                     uint16_t* __restrict__ out, size_t n) {
  const size_t nv = n / 8;
  const size_t v0 = (size_t)blockIdx.x * (256 * kSwigluUnroll) + threadIdx.x;
  uint4 a[kSwigluUnroll], b[kSwigluUnroll];
#pragma unroll
  for (int i = 0; i < kSwigluUnroll; ++i) {
    const size_t v = v0 + 256 * i;
    if (v < nv) {
      a[i] = reinterpret_cast<const uint4*>(g)[v];
      b[i] = reinterpret_cast<const uint4*>(u)[v];
    }
  }
#pragma unroll
  for (int i = 0; i < kSwigluUnroll; ++i) {
    const size_t v = v0 + 256 * i;
    if (v < nv)
      reinterpret_cast<uint4*>(out)[v] =
          make_uint4(swiglu2(a[i].x, b[i].x), swiglu2(a[i].y, b[i].y), swiglu2(a[i].z, b[i].z),
                     swiglu2(a[i].w, b[i].w));
  }
  // the values past the last vector
  if (blockIdx.x == 0 && threadIdx.x < (n & 7)) {
    const size_t e = 8 * nv + threadIdx.x;
    out[e] = (uint16_t)swiglu2(g[e], u[e]);
  }
}

}  // namespace

extern "C" int dip_swiglu(const uint16_t* g, const uint16_t* u, uint16_t* out, int64_t n,
                          void* stream) {
  if (n < 0) return DIP_ERR_SHAPE;
  if (n == 0) return DIP_OK;
  if (!g || !u || !out) return DIP_ERR_NULL;
  if (!aligned16(g) || !aligned16(u) || !aligned16(out)) return DIP_ERR_ALIGN;
  const size_t blocks = ((size_t)n / 8 + 256 * kSwigluUnroll - 1) / (256 * kSwigluUnroll);
  if (blocks > INT32_MAX) return DIP_ERR_SHAPE;
  hipLaunchKernelGGL(swiglu_kernel, dim3((unsigned)std::max<size_t>(blocks, 1)), dim3(256), 0,
                     (hipStream_t)stream, g, u, out, (size_t)n);
  return hip_status(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Dequantisation to the transpose, out[c][r] = bf16(q * s)[r][c]: the layout the
// library's products are fastest on (2048 tokens through 25600 x 5120: 433 us,
// with the rows as they are 582).  Bound by the stores, so a wave owns 32 columns of
// 128 rows: lane l loads 16 bytes of rows 2 l and 2 l + 1, packs each column's
// pair into one dword of LDS (64 lanes, 64 banks), and the wave stores each
// column as 256 contiguous bytes.  A workgroup's waves sit side by side, so the
// loads cover whole lines of the rows.  25600 x 5120 71 us (the rows as they
// are 50), 12288 x 4096 22 us (either order of the tiles within 2 %).
// ---------------------------------------------------------------------------
namespace {
constexpr int kDqtWaves = 8;   // 256 columns
constexpr int kDqtRows = 128;

__global__ __launch_bounds__(64 * kDqtWaves) void dequant_t_kernel(const int8_t* __restrict__ qw,
                                                                   const uint16_t* __restrict__ sc,
                                                                   uint16_t* __restrict__ out,
                                                                   int rows, int cols) {
  __shared__ __align__(16) uint32_t tile[kDqtWaves][32][kDqtRows / 2];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // waves past the last column repeat it (the same values, stored once more)
  const int c0 = min(((int)blockIdx.x * kDqtWaves + wave) * 32, cols - 32);
  const int r0 = (int)blockIdx.y * kDqtRows;
  uint4 w[2];
  uint32_t s[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const size_t r = (size_t)min(r0 + 2 * lane + i, rows - 1);
    w[i] = *reinterpret_cast<const uint4*>(qw + r * (size_t)(cols / 2) + c0 / 2);
    s[i] = sc[r * (size_t)(cols / kGroupSize) + c0 / kGroupSize];
  }
  const float s0 = bf16_to_f32(s[0]) * 0.0625f, s1 = bf16_to_f32(s[1]) * 0.0625f;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    float a[8], b[8];
    dequant8(d == 0 ? w[0].x : d == 1 ? w[0].y : d == 2 ? w[0].z : w[0].w, s0, a);
    dequant8(d == 0 ? w[1].x : d == 1 ? w[1].y : d == 2 ? w[1].z : w[1].w, s1, b);
#pragma unroll
    for (int i = 0; i < 8; ++i) tile[wave][8 * d + i][lane] = f32x2_to_bf16x2(a[i], b[i]);
  }
  __syncthreads();
  const int r = r0 + 8 * (lane & 15);  // rows is a multiple of 8
  if (r < rows) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int c = 4 * i + (lane >> 4);
      *reinterpret_cast<uint4*>(out + (size_t)(c0 + c) * rows + r) =
          *reinterpret_cast<const uint4*>(&tile[wave][c][4 * (lane & 15)]);
    }
  }
}
}  // namespace

extern "C" int dip_dequant_t(const int8_t* qweight, const uint16_t* scales, uint16_t* out,
                             int64_t rows, int64_t cols, void* stream) {
  if (!qweight || !scales || !out) return DIP_ERR_NULL;
  if (rows < 0 || cols <= 0 || cols % kGroupSize != 0 || rows > INT32_MAX - kDqtRows ||
      cols > INT32_MAX - 32 * kDqtWaves)
    return DIP_ERR_SHAPE;
  if (!aligned16(qweight) || !aligned16(out)) return DIP_ERR_ALIGN;
  const int64_t blocks_r = (rows + kDqtRows - 1) / kDqtRows;
  if (rows % 8 != 0 || blocks_r > 65535) return DIP_ERR_UNSUPPORTED;
  if (rows == 0) return DIP_OK;
  const unsigned blocks_c = (unsigned)((cols + 32 * kDqtWaves - 1) / (32 * kDqtWaves));
  hipLaunchKernelGGL(dequant_t_kernel, dim3(blocks_c, (unsigned)blocks_r), dim3(64 * kDqtWaves), 0,
                     (hipStream_t)stream, qweight, scales, out, (int)rows, (int)cols);
  return hip_status(hipGetLastError());
}

extern "C" int dip_dequant_rows(const int8_t* qweight, const uint16_t* scales,
                                const int32_t* indices, void* out, int64_t n_out_rows,
                                int64_t rows, int64_t cols, int mode, void* stream) {
  if (!qweight || !scales || !out) return DIP_ERR_NULL;
  if (cols <= 0 || cols % kGroupSize != 0 || rows < 0 || n_out_rows < 0 ||
      rows > INT32_MAX || n_out_rows > INT32_MAX)
    return DIP_ERR_SHAPE;
  if (!indices && n_out_rows > rows) return DIP_ERR_SHAPE;
  if (mode != 0 && mode != 1) return DIP_ERR_ARG;
  if (n_out_rows == 0) return DIP_OK;
  // The vector forms load dwords and store 128 bits; a caller's buffers need
  // not be aligned for that.
  const bool vec = (reinterpret_cast<uintptr_t>(qweight) & 3u) == 0 && aligned16(out);
  hipStream_t s = (hipStream_t)stream;
  if (vec && !indices) {
    const size_t n = (size_t)n_out_rows * (size_t)(cols / 8);
    const unsigned blocks = (unsigned)std::min<size_t>((n + 256 * kDqUnroll - 1) / (256 * kDqUnroll), 1u << 20);
    const uint32_t* q = reinterpret_cast<const uint32_t*>(qweight);
    if (mode == 0)
      hipLaunchKernelGGL(dequant_flat_kernel<0>, dim3(blocks), dim3(256), 0, s, q, scales, out, n);
    else
      hipLaunchKernelGGL(dequant_flat_kernel<1>, dim3(blocks), dim3(256), 0, s, q, scales, out, n);
  } else if (vec) {
    const int rd = (int)(cols / 8);
    const dim3 grid((unsigned)((rd + 255) / 256), (unsigned)std::min<int64_t>(n_out_rows, 65535));
    const uint32_t* q = reinterpret_cast<const uint32_t*>(qweight);
    if (mode == 0)
      hipLaunchKernelGGL(dequant_gather_kernel<0>, grid, dim3(256), 0, s, q, scales, indices, out,
                         (int)n_out_rows, (int)rows, rd);
    else
      hipLaunchKernelGGL(dequant_gather_kernel<1>, grid, dim3(256), 0, s, q, scales, indices, out,
                         (int)n_out_rows, (int)rows, rd);
  } else {
    const size_t total = (size_t)n_out_rows * (size_t)(cols / 2);
    const unsigned blocks = (unsigned)std::min<size_t>((total + 255) / 256, 4096);
    hipLaunchKernelGGL(dequant_rows_kernel, dim3(blocks), dim3(256), 0, s, qweight, scales, indices,
                       out, (int)n_out_rows, (int)rows, (int)cols, mode);
  }
  return hip_status(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Host-side miss gather (the pinned index_select of dip_ca.py:148-153) on the
// persistent host thread pool of dip_host_pool.h.
// ---------------------------------------------------------------------------
namespace {

int check_pieces(int npieces, const void* const* src, void* const* dst, const int64_t* row_bytes,
                 const int32_t* ids, int64_t n, int64_t src_rows) {
  if (n < 0 || src_rows < 0 || npieces < 0 || npieces > 64) return DIP_ERR_SHAPE;
  if (n == 0 || npieces == 0) return DIP_OK;
  if (!ids || !src || !dst || !row_bytes) return DIP_ERR_NULL;
  for (int p = 0; p < npieces; ++p) {
    if (row_bytes[p] < 0) return DIP_ERR_SHAPE;
    if (row_bytes[p] > 0 && (!src[p] || !dst[p])) return DIP_ERR_NULL;
  }
  for (int64_t i = 0; i < n; ++i)
    if (ids[i] < 0 || ids[i] >= src_rows) return DIP_ERR_SHAPE;
  return DIP_OK;
}

// dst_p[i] = src_p[ids[i]] for every piece p and i in [b, e).
void copy_rows(int npieces, const void* const* src, void* const* dst, const int64_t* row_bytes,
               const int32_t* ids, int64_t b, int64_t e) {
  for (int p = 0; p < npieces; ++p) {
    const int64_t rb = row_bytes[p];
    const char* s = static_cast<const char*>(src[p]);
    char* d = static_cast<char*>(dst[p]);
    for (int64_t i = b; i < e; ++i) std::memcpy(d + i * rb, s + (int64_t)ids[i] * rb, (size_t)rb);
  }
}

int pool_threads(int threads, int64_t n) {
  int nt = std::max(1, std::min(threads, 64));
  return (int)std::min<int64_t>(nt, n);
}

int gather_rows(int npieces, const void* const* src, void* const* dst, const int64_t* row_bytes,
                const int32_t* ids, int64_t n, int64_t src_rows, int threads) {
  const int st = check_pieces(npieces, src, dst, row_bytes, ids, n, src_rows);
  if (st || n == 0 || npieces == 0) return st;
  const int nt = pool_threads(threads, n);
  const int64_t per = (n + nt - 1) / nt;
  auto work = [&](int t) {
    copy_rows(npieces, src, dst, row_bytes, ids, std::min(n, t * per), std::min(n, (t + 1) * per));
  };
  if (nt == 1)
    work(0);
  else
    HostPool::get().run(nt, work);
  return DIP_OK;
}

}  // namespace

extern "C" int dip_host_gather_rows(const void* src, const int32_t* ids, void* dst, int64_t n,
                                    int64_t row_bytes, int64_t src_rows, int threads) {
  return gather_rows(1, &src, &dst, &row_bytes, ids, n, src_rows, threads);
}

extern "C" int dip_host_gather_rows_multi(const void* const* src, void* const* dst,
                                          const int64_t* row_bytes, int64_t npieces,
                                          const int32_t* ids, int64_t n, int64_t src_rows,
                                          int threads) {
  if (npieces < 0 || npieces > 64) return DIP_ERR_SHAPE;
  return gather_rows((int)npieces, src, dst, row_bytes, ids, n, src_rows, threads);
}

namespace {

// The miss stream's second copy stream on the current device and the events
// that fork it from and join it to the caller's stream (created on first
// use, kept for the life of the process; default priority).
struct SideStream {
  hipStream_t stream = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};

int side_stream(SideStream** out) {
  static SideStream table[64];
  static std::mutex mu;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= 64) return DIP_ERR_ARG;
  std::lock_guard<std::mutex> lock(mu);
  SideStream& t = table[dev];
  if (!t.stream) {
    e = hipStreamCreateWithFlags(&t.stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&t.fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&t.join, hipEventDisableTiming);
    if (e != hipSuccess) {
      if (t.fork) (void)hipEventDestroy(t.fork);
      if (t.stream) (void)hipStreamDestroy(t.stream);
      t = SideStream{};
      return (int)e;
    }
  }
  *out = &t;
  return DIP_OK;
}

}  // namespace

extern "C" int dip_host_stream_rows(const void* const* src, void* const* pinned,
                                    void* const* dst, const int64_t* row_bytes, int64_t npieces,
                                    const int32_t* ids, int64_t n, int64_t src_rows,
                                    int64_t chunk_rows, int threads, void* stream,
                                    float* copy_ms) {
  if (copy_ms) *copy_ms = 0.f;
  if (chunk_rows <= 0) return DIP_ERR_ARG;
  int st = check_pieces((int)npieces, src, pinned, row_bytes, ids, n, src_rows);
  if (st) return st;
  st = check_pieces((int)npieces, pinned, dst, row_bytes, ids, n, src_rows);
  if (st || n == 0 || npieces == 0) return st;
  const int np = (int)npieces;
  // Chunk c covers rows [cut[c], cut[c + 1]).  The first chunks ramp up from
  // chunk_rows / 8, doubling, so the first copy starts after a short gather
  // instead of a whole chunk's; the rest are chunk_rows.
  std::vector<int64_t> cut{0};
  for (int64_t c = std::max<int64_t>(chunk_rows / 8, 1); cut.back() < n;
       c = std::min(chunk_rows, 2 * c))
    cut.push_back(std::min(n, cut.back() + c));
  const int64_t nchunks = (int64_t)cut.size() - 1;
  const int nt = std::min(pool_threads(threads, chunk_rows), HostPool::max_async_jobs());
  hipStream_t s = (hipStream_t)stream;
  // Pieces [0, np/2) are copied on the caller's stream, the rest on a side
  // stream, so two DMA engines share each chunk; the caller's stream waits
  // for the side stream before the call returns.
  // (without it, as without a device, the gather still runs to the end and
  // the call returns the error, as for a failed copy)
  SideStream* side = nullptr;
  const int st_side = side_stream(&side);
  hipStream_t ss = side ? side->stream : nullptr;
  const int np0 = np / 2 > 0 ? np / 2 : np;  // one piece: the caller's stream alone
  std::vector<hipEvent_t> ev;
  if (copy_ms && st_side == DIP_OK) {
    ev.assign(4 * nchunks, nullptr);
    for (auto& e : ev)
      if (hipEventCreate(&e) != hipSuccess) {
        for (auto& e2 : ev)
          if (e2) (void)hipEventDestroy(e2);
        return hip_status(hipGetLastError());
      }
  }
  // The pool's threads only gather (left[c]: their slices of chunk c not yet
  // gathered); this thread queues each chunk's copies as soon as it is
  // complete, so every HIP call stays on the caller's thread.
  std::vector<std::atomic<int>> left(nchunks);
  for (auto& l : left) l.store(nt, std::memory_order_relaxed);
  // a named std::function: the workers call it until pool.finish() returns
  const std::function<void(int)> work = [&](int t) {
    for (int64_t c = 0; c < nchunks; ++c) {
      const int64_t c0 = cut[c], c1 = cut[c + 1];
      const int64_t per = (c1 - c0 + nt - 1) / nt;
      copy_rows(np, src, pinned, row_bytes, ids, std::min(c1, c0 + t * per),
                std::min(c1, c0 + (t + 1) * per));
      left[c].fetch_sub(1, std::memory_order_release);
    }
  };
  const bool copies = st_side == DIP_OK;
  hipError_t e = hipSuccess;
  HostPool& pool = HostPool::get();
  // Callers run one at a time from start() to finish(), so the side stream
  // and its two events serve one call at a time.
  pool.start(nt, &work);
  // the side stream starts after the work already queued on the caller's
  if (copies) {
    e = hipEventRecord(side->fork, s);
    if (e == hipSuccess) e = hipStreamWaitEvent(ss, side->fork, 0);
  }
  for (int64_t c = 0; c < nchunks; ++c) {
    while (left[c].load(std::memory_order_acquire) != 0) std::this_thread::yield();
    // let the gather finish; report the first error
    if (!copies || e != hipSuccess) continue;
    const int64_t c0 = cut[c], c1 = cut[c + 1];
    if (copy_ms) e = hipEventRecord(ev[4 * c], s);
    if (copy_ms && e == hipSuccess) e = hipEventRecord(ev[4 * c + 2], ss);
    for (int p = 0; p < np && e == hipSuccess; ++p) {
      const int64_t rb = row_bytes[p];
      if (rb == 0) continue;
      e = hipMemcpyAsync(static_cast<char*>(dst[p]) + c0 * rb,
                         static_cast<const char*>(pinned[p]) + c0 * rb,
                         (size_t)((c1 - c0) * rb), hipMemcpyHostToDevice, p < np0 ? s : ss);
    }
    if (copy_ms && e == hipSuccess) e = hipEventRecord(ev[4 * c + 1], s);
    if (copy_ms && e == hipSuccess) e = hipEventRecord(ev[4 * c + 3], ss);
  }
  if (copies && e == hipSuccess) e = hipEventRecord(side->join, ss);
  if (copies && e == hipSuccess) e = hipStreamWaitEvent(s, side->join, 0);
  pool.finish();
  st = !copies ? st_side : (e == hipSuccess ? DIP_OK : (int)e);
  if (copy_ms && copies) {
    // a chunk's copy time: the longer of its two streams' spans
    float total = 0.f;
    if (!st) {
      for (int64_t c = 0; c < nchunks && !st; ++c) {
        float ms[2] = {0.f, 0.f};
        for (int k = 0; k < 2 && !st; ++k) {
          hipError_t e2 = hipEventSynchronize(ev[4 * c + 2 * k + 1]);
          if (e2 == hipSuccess) e2 = hipEventElapsedTime(&ms[k], ev[4 * c + 2 * k],
                                                         ev[4 * c + 2 * k + 1]);
          if (e2 != hipSuccess) st = (int)e2;
        }
        total += std::max(ms[0], ms[1]);
      }
    }
    for (auto& ev1 : ev) (void)hipEventDestroy(ev1);
    *copy_ms = total;
  }
  return st;
}

// ---------------------------------------------------------------------------
// One resident DIP MLP decode step.
//   workspace: [0, 512) top-k state | the down workspace (the XCD-local
//   reduce's counters at a fixed offset, then the partials) | h by channel
//   [inter] bf16
// ---------------------------------------------------------------------------
namespace {
constexpr size_t kMlpTopkBytes = 512;
static_assert(kTopkWorkspace <= kMlpTopkBytes, "top-k state");
size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }
}  // namespace

extern "C" size_t dip_mlp_workspace_size(int64_t hidden, int64_t inter, int64_t k) {
  const size_t hfull = inter > 0 ? align256((size_t)inter * sizeof(uint16_t)) : 0;
  return kMlpTopkBytes + align256(down_workspace_bytes(k, hidden)) + hfull;
}

extern "C" int dip_mlp_decode_rmsnorm(const int8_t* gate_qw, const uint16_t* gate_sc,
                                      const int8_t* up_qw, const uint16_t* up_sc,
                                      const int8_t* down_t_qw, const uint16_t* down_t_sc,
                                      const uint16_t* down_t_sc_gm, const uint16_t* h,
                                      const uint16_t* add, const uint16_t* norm_w, float eps, uint16_t* h_res_out,
                                      uint16_t* x_out, uint16_t* y, uint16_t* g_out,
                                      int32_t* idx_out, uint16_t* h_out, int64_t hidden,
                                      int64_t inter, int64_t k, void* workspace, size_t ws_bytes,
                                      void* layer_state, void* stream) {
  if (!gate_qw || !gate_sc || !up_qw || !up_sc || !h || !norm_w || !x_out || !g_out || !y)
    return DIP_ERR_NULL;
  if (k < 0 || k > inter || inter <= 0 || inter > INT32_MAX) return DIP_ERR_SHAPE;
  if (k > 0 && (!idx_out || !h_out)) return DIP_ERR_NULL;
  if (!rowdot_norm_supported(hidden)) return DIP_ERR_UNSUPPORTED;
  if (!(eps >= 0.f)) return DIP_ERR_ARG;
  if (!aligned16(gate_qw) || !aligned16(up_qw) || !aligned16(h) || !aligned16(norm_w) ||
      !aligned16(x_out) || !aligned16(g_out) || (add && !aligned16(add)) ||
      (h_res_out && !aligned16(h_res_out)))
    return DIP_ERR_ALIGN;
  // every workgroup of the gate reads h and add while workgroup 0 writes
  // the residual and x
  if (x_out == h || x_out == add || (h_res_out && (h_res_out == h || h_res_out == add)))
    return DIP_ERR_ARG;
  if (!workspace || ws_bytes < dip_mlp_workspace_size(hidden, inter, k)) return DIP_ERR_WORKSPACE;
  if (!aligned16(workspace)) return DIP_ERR_ALIGN;
  char* ws = static_cast<char*>(workspace);
  char* down_ws = ws + kMlpTopkBytes;
  const size_t down_bytes = align256(down_workspace_bytes(k, hidden));
  uint16_t* h_full = reinterpret_cast<uint16_t*>(down_ws + down_bytes);
  hipStream_t s = (hipStream_t)stream;
  RowdotArgs a{};
  a.qw_a = gate_qw;
  a.sc_a = gate_sc;
  a.qw_safe = gate_qw;
  a.sc_safe = gate_sc;
  a.x = h;
  a.out = g_out;
  a.nrows = (int)inter;
  a.in_features = (int)hidden;
  a.rows_a = (int)inter;
  a.norm_w = norm_w;
  a.norm_add = add;
  a.norm_h_out = h_res_out;
  a.norm_x_out = x_out;
  a.norm_eps = eps;
  const bool spec = layer_state && k > 0 && topk_spec_supported(hidden) && inter <= kTopkMaxN;
  if (spec) {
    if (reinterpret_cast<uintptr_t>(layer_state) & 3u) return DIP_ERR_ALIGN;
    a.rotate = static_cast<uint32_t*>(layer_state);
    int st = launch_rowdot_norm(kSilu, a, s);
    if (st) return st;
    st = launch_spec_after_gate(g_out, inter, hidden, k, idx_out, h_full, up_qw, up_sc, x_out, ws,
                                layer_state, s);
    if (st) return st;
    return dip_int4_gather_down_by_channel(down_t_qw, down_t_sc, down_t_sc_gm, h_full, idx_out,
                                           y, h_out, inter, hidden, k, down_ws, down_bytes,
                                           stream);
  }
  int st = launch_rowdot_norm(kSilu, a, s);
  if (st) return st;
  st = dip_topk_select(g_out, idx_out, inter, k, ws, kMlpTopkBytes, stream);
  if (st) return st;
  if (k > 0) {
    st = dip_up_gather_h(up_qw, up_sc, x_out, idx_out, g_out, h_out, inter, hidden, k, stream);
    if (st) return st;
  }
  return run_down(kGather, down_t_qw, down_t_sc, inter, nullptr, nullptr, 0, h_out, idx_out,
                  nullptr, k, hidden, y, down_ws, down_bytes, (hipStream_t)stream, 0, nullptr,
                  down_t_sc_gm);
}

extern "C" int dip_mlp_decode(const int8_t* gate_qw, const uint16_t* gate_sc,
                              const int8_t* up_qw, const uint16_t* up_sc,
                              const int8_t* down_t_qw, const uint16_t* down_t_sc,
                              const uint16_t* down_t_sc_gm, const uint16_t* x, uint16_t* y,
                              uint16_t* g_out, int32_t* idx_out, uint16_t* h_out, int64_t hidden, int64_t inter, int64_t k,
                              void* workspace, size_t ws_bytes, void* layer_state,
                              void* stream) {
  if (!g_out || !y || !x) return DIP_ERR_NULL;
  if (k < 0 || k > inter) return DIP_ERR_SHAPE;
  if (k > 0 && (!idx_out || !h_out)) return DIP_ERR_NULL;
  if (!workspace || ws_bytes < dip_mlp_workspace_size(hidden, inter, k)) return DIP_ERR_WORKSPACE;
  char* ws = static_cast<char*>(workspace);
  char* down_ws = ws + kMlpTopkBytes;
  const size_t down_bytes = align256(down_workspace_bytes(k, hidden));
  uint16_t* h_full = reinterpret_cast<uint16_t*>(down_ws + down_bytes);
  if (layer_state && k > 0 && topk_spec_supported(hidden) && inter <= kTopkMaxN) {
    int st = dip_gate_silu_topk_spec(gate_qw, gate_sc, up_qw, up_sc, x, g_out, idx_out, h_full,
                                     inter, hidden, k, ws, kMlpTopkBytes, layer_state, stream);
    if (st) return st;
    return dip_int4_gather_down_by_channel(down_t_qw, down_t_sc, down_t_sc_gm, h_full, idx_out,
                                           y, h_out, inter, hidden, k, down_ws, down_bytes,
                                           stream);
  }
  int st = dip_gate_silu_topk(gate_qw, gate_sc, x, g_out, idx_out, inter, hidden, k, ws,
                              kMlpTopkBytes, stream);
  if (st) return st;
  if (k > 0) {
    st = dip_up_gather_h(up_qw, up_sc, x, idx_out, g_out, h_out, inter, hidden, k, stream);
    if (st) return st;
  }
  return run_down(kGather, down_t_qw, down_t_sc, inter, nullptr, nullptr, 0, h_out, idx_out,
                  nullptr, k, hidden, y, down_ws, down_bytes, (hipStream_t)stream, 0, nullptr,
                  down_t_sc_gm);
}
