// Bit packing, Lloyd-Max quantize/dequantize and the library's error plumbing.
//
// Layout follows src/turboquant_pytorch/kernels/bit_ops.py:243-326: code i of a
// row occupies bits [i*b, i*b+b), LSB first.  Each thread owns one output byte
// (pack / quantize) or one output code (unpack / dequantize), so no atomics are
// needed (the reference's Triton kernels OR into shared bytes,
// bit_ops.py:94-109, quantize.py:124-143).
//
// Contiguous rows of a multiple of 8 codes (every head dim here) are one stream of 8-code groups,
// b bytes each: a thread of the stream kernels takes a group, 16-byte loads and stores on the wide
// side, and a block's packed bytes cross LDS so that they move as whole dwords.  Both sides then
// run near memory speed: 65536 x 128 codes of 3 bits (33.6 MB of f32 / int32, 16.8 of f16) quantise in
// 8.5, pack in 7.1, unpack in 10.6 and dequantise in 7.3 us, where the byte- and code-per-thread
// kernels, which serve every other layout, take 25, 15, 20 and 24.
#include <cstdarg>
#include <cstdio>

#include "tq_common.h"

namespace tq {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

int launch_status(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: HIP launch failed: %s", what, hipGetErrorString(e));
    return TQ_EHIP;
  }
  return TQ_OK;
}

// One thread per output byte p of row r: OR the (masked) codes whose bits
// overlap [8p, 8p+8).
__global__ void pack_bits_kernel(const int32_t* __restrict__ idx, int64_t n, int d, int64_t ld_idx,
                                 int b, uint8_t* __restrict__ out, int64_t ld_out, int oc) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n * oc) return;
  const int64_t r = t / oc;
  const int p = static_cast<int>(t - r * oc);
  const uint32_t mask = (1u << b) - 1u;
  const int lo_bit = 8 * p;
  const int c0 = lo_bit / b;
  int c1 = (lo_bit + 7) / b;
  if (c1 > d - 1) c1 = d - 1;
  const int32_t* row = idx + r * ld_idx;
  uint32_t acc = 0;
  for (int c = c0; c <= c1; ++c) {
    const uint32_t v = static_cast<uint32_t>(row[c]) & mask;
    const int sh = c * b - lo_bit;
    acc |= (sh >= 0) ? (v << sh) : (v >> (-sh));
  }
  out[r * ld_out + p] = static_cast<uint8_t>(acc & 0xffu);
}

__global__ void unpack_bits_kernel(const uint8_t* __restrict__ packed, int64_t n, int d,
                                   int64_t ld_in, int b, int32_t* __restrict__ out,
                                   int64_t ld_out) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n * d) return;
  const int64_t r = t / d;
  const int i = static_cast<int>(t - r * d);
  out[r * ld_out + i] = static_cast<int32_t>(read_code(packed + r * ld_in, i, b));
}

// searchsorted-left codes of y, packed; the boundary table sits in LDS.
__global__ void quantize_pack_kernel(const float* __restrict__ y, int64_t n, int d, int64_t ld_y,
                                     const float* __restrict__ bounds, int b,
                                     uint8_t* __restrict__ out, int64_t ld_out, int oc) {
  __shared__ float sb[255];
  const int nb = (1 << b) - 1;
  for (int j = threadIdx.x; j < nb; j += blockDim.x) sb[j] = bounds[j];
  __syncthreads();
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n * oc) return;
  const int64_t r = t / oc;
  const int p = static_cast<int>(t - r * oc);
  const int lo_bit = 8 * p;
  const int c0 = lo_bit / b;
  int c1 = (lo_bit + 7) / b;
  if (c1 > d - 1) c1 = d - 1;
  const float* row = y + r * ld_y;
  uint32_t acc = 0;
  for (int c = c0; c <= c1; ++c) {
    const uint32_t v = searchsorted_left(row[c], sb, nb);
    const int sh = c * b - lo_bit;
    acc |= (sh >= 0) ? (v << sh) : (v >> (-sh));
  }
  out[r * ld_out + p] = static_cast<uint8_t>(acc & 0xffu);
}

__global__ void dequantize_kernel(const uint8_t* __restrict__ packed, int64_t n, int d,
                                  int64_t ld_in, const uint16_t* __restrict__ cent, int b,
                                  uint16_t* __restrict__ out, int64_t ld_out) {
  __shared__ uint16_t sc[256];
  for (int j = threadIdx.x; j < (1 << b); j += blockDim.x) sc[j] = cent[j];
  __syncthreads();
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n * d) return;
  const int64_t r = t / d;
  const int i = static_cast<int>(t - r * d);
  out[r * ld_out + i] = sc[read_code(packed + r * ld_in, i, b)];
}

// ---------------------------------------------------------------- 8-code groups
constexpr int kGroupThreads = 256;
typedef int int4v __attribute__((ext_vector_type(4)));

// low b bytes of `bits` to this thread's place in the block's staging, then the block's bytes to
// out[first * b ..): whole dwords, the last partial one as bytes
__device__ __forceinline__ void store_groups(uint64_t bits, int b, int64_t first, int64_t groups, uint8_t* stage,
                                             uint8_t* __restrict__ out) {
  const int tid = threadIdx.x;
  for (int k = 0; k < b; ++k) stage[tid * b + k] = static_cast<uint8_t>(bits >> (8 * k));
  __syncthreads();
  const int64_t left = groups - first;
  const int bytes = static_cast<int>(left < kGroupThreads ? left : kGroupThreads) * b;
  uint8_t* dst = out + first * b;
  for (int i = tid; i < bytes / 4; i += kGroupThreads)
    reinterpret_cast<uint32_t*>(dst)[i] = reinterpret_cast<const uint32_t*>(stage)[i];
  for (int i = (bytes & ~3) + tid; i < bytes; i += kGroupThreads) dst[i] = stage[i];
}
// the reverse: this thread's b bytes of packed[first * b ..)
__device__ __forceinline__ uint64_t load_groups(const uint8_t* __restrict__ packed, int b, int64_t first, int64_t groups,
                                                uint8_t* stage) {
  const int tid = threadIdx.x;
  const int64_t left = groups - first;
  const int bytes = static_cast<int>(left < kGroupThreads ? left : kGroupThreads) * b;
  const uint8_t* src = packed + first * b;
  for (int i = tid; i < bytes / 4; i += kGroupThreads)
    reinterpret_cast<uint32_t*>(stage)[i] = reinterpret_cast<const uint32_t*>(src)[i];
  for (int i = (bytes & ~3) + tid; i < bytes; i += kGroupThreads) stage[i] = src[i];
  __syncthreads();
  uint64_t v = 0;
  for (int k = 0; k < b; ++k) v |= static_cast<uint64_t>(stage[tid * b + k]) << (8 * k);
  return v;
}

__global__ void __launch_bounds__(kGroupThreads) pack_groups_kernel(const int32_t* __restrict__ idx, int64_t groups, int b,
                                                                    uint8_t* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) uint8_t stage[kGroupThreads * 8];
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kGroupThreads, g = first + threadIdx.x;
  uint64_t v = 0;
  if (g < groups) {
    const int4v x = reinterpret_cast<const int4v*>(idx)[2 * g], y = reinterpret_cast<const int4v*>(idx)[2 * g + 1];
    const uint32_t mask = (1u << b) - 1u;
#pragma unroll
    for (int e = 0; e < 8; ++e) v |= static_cast<uint64_t>(static_cast<uint32_t>(e < 4 ? x[e] : y[e - 4]) & mask) << (b * e);
  }
  store_groups(v, b, first, groups, stage, out);
}

__global__ void __launch_bounds__(kGroupThreads) unpack_groups_kernel(const uint8_t* __restrict__ packed, int64_t groups,
                                                                      int b, int32_t* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) uint8_t stage[kGroupThreads * 8];
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kGroupThreads, g = first + threadIdx.x;
  const uint64_t v = load_groups(packed, b, first, groups, stage);
  if (g >= groups) return;
  const uint32_t mask = (1u << b) - 1u;
  int4v x, y;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[e] = static_cast<int>(static_cast<uint32_t>(v >> (b * e)) & mask);
    y[e] = static_cast<int>(static_cast<uint32_t>(v >> (b * (e + 4))) & mask);
  }
  reinterpret_cast<int4v*>(out)[2 * g] = x;
  reinterpret_cast<int4v*>(out)[2 * g + 1] = y;
}

// up to 4 bits: the boundaries in scalar registers, counted as searchsorted_left does
template <int B>
__global__ void __launch_bounds__(kGroupThreads) quantize_groups_kernel(const float* __restrict__ y, int64_t groups,
                                                                        const float* __restrict__ bounds,
                                                                        uint8_t* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) uint8_t stage[kGroupThreads * 8];
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kGroupThreads, g = first + threadIdx.x;
  uint32_t v = 0;
  if (g < groups) {
    const float4v p = reinterpret_cast<const float4v*>(y)[2 * g], q = reinterpret_cast<const float4v*>(y)[2 * g + 1];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x = e < 4 ? p[e] : q[e - 4];
      uint32_t c = 0;
#pragma unroll
      for (int j = 0; j < (1 << B) - 1; ++j) c += (bounds[j] < x) ? 1u : 0u;
      v |= c << (B * e);
    }
  }
  store_groups(v, B, first, groups, stage, out);
}

__global__ void __launch_bounds__(kGroupThreads) dequantize_groups_kernel(const uint8_t* __restrict__ packed, int64_t groups,
                                                                          const uint16_t* __restrict__ cent, int b,
                                                                          uint16_t* __restrict__ out) {
  __shared__ uint16_t sc[256];
  __shared__ __attribute__((aligned(16))) uint8_t stage[kGroupThreads * 8];
  for (int j = threadIdx.x; j < (1 << b); j += blockDim.x) sc[j] = cent[j];
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kGroupThreads, g = first + threadIdx.x;
  const uint64_t v = load_groups(packed, b, first, groups, stage);  // its barrier covers sc
  if (g >= groups) return;
  const uint32_t mask = (1u << b) - 1u;
  int4v o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = sc[static_cast<uint32_t>(v >> (b * 2 * e)) & mask];
    const uint32_t hi = sc[static_cast<uint32_t>(v >> (b * (2 * e + 1))) & mask];
    o[e] = static_cast<int>(lo | (hi << 16));
  }
  reinterpret_cast<int4v*>(out)[g] = o;
}

// contiguous rows of whole 8-code groups, 16-byte aligned on the wide side and dword aligned on the
// packed side (a block's bytes start at a multiple of 256 b)
static bool group_stream(int64_t ld_wide, int64_t ld_packed, int d, int b, const void* wide, const void* packed) {
  return d % 8 == 0 && ld_wide == d && ld_packed == static_cast<int64_t>(d) / 8 * b &&
         reinterpret_cast<uintptr_t>(wide) % 16 == 0 && reinterpret_cast<uintptr_t>(packed) % 4 == 0;
}

static inline unsigned grid_for(int64_t work, int threads) {
  return static_cast<unsigned>((work + threads - 1) / threads);
}

}  // namespace tq

using namespace tq;

extern "C" {

int tq_version(void) { return 100; }

const char* tq_last_error(void) { return g_err; }

int64_t tq_out_cols(int64_t d, int32_t b) { return out_cols(d, b); }

int tq_pack_bits(const int32_t* idx, int64_t n, int32_t d, int64_t ld_idx, int32_t b,
                 uint8_t* out, int64_t ld_out, void* stream) {
  TQ_REQUIRE(b >= 1 && b <= 8, "tq_pack_bits: b must be between 1 and 8, got %d", b);
  TQ_REQUIRE(n >= 0 && d >= 1, "tq_pack_bits: bad shape n=%lld d=%d", (long long)n, d);
  const int oc = static_cast<int>(out_cols(d, b));
  TQ_REQUIRE(ld_idx >= d && ld_out >= oc, "tq_pack_bits: row strides too small");
  if (n == 0) return TQ_OK;
  TQ_REQUIRE(idx && out, "tq_pack_bits: null pointer");
  if (group_stream(ld_idx, ld_out, d, b, idx, out)) {
    const int64_t groups = n * (d / 8);
    pack_groups_kernel<<<grid_for(groups, kGroupThreads), kGroupThreads, 0, as_stream(stream)>>>(idx, groups, b, out);
    return launch_status("tq_pack_bits");
  }
  const int64_t work = n * oc;
  pack_bits_kernel<<<grid_for(work, 256), 256, 0, as_stream(stream)>>>(idx, n, d, ld_idx, b, out,
                                                                        ld_out, oc);
  return launch_status("tq_pack_bits");
}

int tq_unpack_bits(const uint8_t* packed, int64_t n, int32_t d, int64_t ld_in, int32_t b,
                   int32_t* out, int64_t ld_out, void* stream) {
  TQ_REQUIRE(b >= 1 && b <= 8, "tq_unpack_bits: b must be between 1 and 8, got %d", b);
  TQ_REQUIRE(n >= 0 && d >= 1, "tq_unpack_bits: bad shape");
  TQ_REQUIRE(ld_in >= out_cols(d, b) && ld_out >= d, "tq_unpack_bits: row strides too small");
  if (n == 0) return TQ_OK;
  TQ_REQUIRE(packed && out, "tq_unpack_bits: null pointer");
  if (group_stream(ld_out, ld_in, d, b, out, packed)) {
    const int64_t groups = n * (d / 8);
    unpack_groups_kernel<<<grid_for(groups, kGroupThreads), kGroupThreads, 0, as_stream(stream)>>>(packed, groups, b, out);
    return launch_status("tq_unpack_bits");
  }
  unpack_bits_kernel<<<grid_for(n * d, 256), 256, 0, as_stream(stream)>>>(packed, n, d, ld_in, b,
                                                                         out, ld_out);
  return launch_status("tq_unpack_bits");
}

int tq_quantize_pack(const float* y, int64_t n, int32_t d, int64_t ld_y, const float* bounds,
                     int32_t b_eff, uint8_t* out, int64_t ld_out, void* stream) {
  TQ_REQUIRE(b_eff >= 1 && b_eff <= 8, "tq_quantize_pack: b_eff must be between 1 and 8, got %d",
             b_eff);
  TQ_REQUIRE(n >= 0 && d >= 1, "tq_quantize_pack: bad shape");
  const int oc = static_cast<int>(out_cols(d, b_eff));
  TQ_REQUIRE(ld_y >= d && ld_out >= oc, "tq_quantize_pack: row strides too small");
  if (n == 0) return TQ_OK;
  TQ_REQUIRE(y && bounds && out, "tq_quantize_pack: null pointer");
  if (b_eff <= 4 && group_stream(ld_y, ld_out, d, b_eff, y, out)) {
    const int64_t groups = n * (d / 8);
    const unsigned grid = grid_for(groups, kGroupThreads);
    hipStream_t s = as_stream(stream);
    if (b_eff == 1) quantize_groups_kernel<1><<<grid, kGroupThreads, 0, s>>>(y, groups, bounds, out);
    else if (b_eff == 2) quantize_groups_kernel<2><<<grid, kGroupThreads, 0, s>>>(y, groups, bounds, out);
    else if (b_eff == 3) quantize_groups_kernel<3><<<grid, kGroupThreads, 0, s>>>(y, groups, bounds, out);
    else quantize_groups_kernel<4><<<grid, kGroupThreads, 0, s>>>(y, groups, bounds, out);
    return launch_status("tq_quantize_pack");
  }
  quantize_pack_kernel<<<grid_for(n * oc, 256), 256, 0, as_stream(stream)>>>(
      y, n, d, ld_y, bounds, b_eff, out, ld_out, oc);
  return launch_status("tq_quantize_pack");
}

int tq_dequantize(const uint8_t* packed, int64_t n, int32_t d, int64_t ld_in,
                  const uint16_t* centroids_f16, int32_t b, uint16_t* out_f16, int64_t ld_out,
                  void* stream) {
  TQ_REQUIRE(b >= 1 && b <= 8, "tq_dequantize: b must be between 1 and 8, got %d", b);
  TQ_REQUIRE(n >= 0 && d >= 1, "tq_dequantize: bad shape");
  TQ_REQUIRE(ld_in >= out_cols(d, b) && ld_out >= d, "tq_dequantize: row strides too small");
  if (n == 0) return TQ_OK;
  TQ_REQUIRE(packed && centroids_f16 && out_f16, "tq_dequantize: null pointer");
  if (group_stream(ld_out, ld_in, d, b, out_f16, packed)) {
    const int64_t groups = n * (d / 8);
    dequantize_groups_kernel<<<grid_for(groups, kGroupThreads), kGroupThreads, 0, as_stream(stream)>>>(
        packed, groups, centroids_f16, b, out_f16);
    return launch_status("tq_dequantize");
  }
  dequantize_kernel<<<grid_for(n * d, 256), 256, 0, as_stream(stream)>>>(
      packed, n, d, ld_in, centroids_f16, b, out_f16, ld_out);
  return launch_status("tq_dequantize");
}

}  // extern "C"
