// Compressed-domain attention for many query rows through expanded tiles.
//
// The asymmetric estimator of one key is linear in the rotated query: with S_eff the QJL
// matrix the query projection uses (q_proj = q_rot S_eff^T),
//   vn <q_rot, C[codes]> + coeff rn <q_proj, s>  =  <q_rot, k^>,
//   k^ = vn C[codes] + coeff rn S_eff^T s        (s the +-1 sign row).
// A prefill meets every key with thousands of query rows, so k^ is formed once per key
// (one d x d product per key: dense_expand_kernel) and the attention kernel scores with one
// d-long product instead of two, needs no q_proj, no decoding and no per-key factors in its
// loop.  k^ is kept at f32 grade as f16 (hi, lo) parts, both multiplied with the f16 q_rot
// (2 MFMA passes; the term-by-term form takes 3: codes, and q_proj's hi and lo against the
// signs).  V^ = f16(C_v[codes] vn), as in the term-by-term kernels.
//
// Tiles.  32 keys of one (batch, kv head) make a record of 3 DP/16 fragments of 1 KiB (DP: d
// rounded up to a multiple of 32, zero padded): k^ hi, k^ lo, V^.  A fragment is one
// v_mfma_f32_32x32x16_f16 A operand in lane order (16 bytes per lane), so that the attention
// kernel copies records into LDS as they are and reads fragments at lane * 16: contiguous in
// memory, free of bank conflicts, no address arithmetic.  k^ carries a power of two per tile
// (from a bound on the tile's largest |k^|), whose inverse the score scaling takes: hi stays finite
// and lo a normal f16 for keys down to kMixed of that bound.  A tile with a smaller key, or with a
// norm that is not finite, is a mixed tile: its keys carry factors of their own, one for the hi and
// one for the lo product, and the kernels take its scores over a separate, slower branch.
//
// Bound and measurements (bits 3, 32 / 8 heads, head_dim 128, against tq_query_prep and the
// term-by-term prefill kernel, one MI355X): 8192 causal rows 1154-1364 -> 830-887 us for the whole layer,
// the attention kernel 760-865 of them, 0.97-1.1 PFLOP/s on the matrix cores where a large library
// product reaches 1.23 (both hold the clock below 2 GHz); 512 rows over 16k cached keys 734 -> 241-258
// us (blocks split the keys, the term-by-term kernel ran 128 blocks); head_dim 80, 1531 rows, 32
// heads: 247 -> 80 us without the compressions.  A tile takes a compute unit 0.90 us with two
// waves per SIMD (its matrix work alone 0.64 at 2.4 GHz); the rest is the chain scores -> softmax ->
// P.V and the barrier.  The expansion writes 6 bytes per element at about 2.7 TB/s (131k keys x 128: 37
// us; a copy of as much runs at 5.1): see dense_expand_kernel.
#include "tq_common.h"
#include "tq_stream.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace tq {

typedef float float16v __attribute__((ext_vector_type(16)));

// v_mfma_f32_32x32x16_f16.  Lane l holds A[m = l%32][k = 8*(l/32) + 0..7],
// B[k = 8*(l/32) + 0..7][n = l%32]; register i of the accumulator holds
// D[m = 8*(i/4) + 4*(l/32) + i%4][n = l%32].
__device__ __forceinline__ float16v mfma32x32x16(half8 a, half8 b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float16v zero16() {
  return float16v{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
}
// Row m of a 32-row A operand holds dim perm32(m) (bits 2 and 3 exchanged): accumulator
// registers 8s..8s+7 of lane (n, h) are then dims 16s + 8h + 0..7, eight consecutive ones, which
// is also the B operand layout of a following product's k-step s.
__device__ __forceinline__ int perm32(int m) { return (m & 19) | ((m & 4) << 1) | ((m & 8) >> 1); }

// 8 halves of row i, columns j .. j + 7, of a d x d matrix; zero outside it.  The address is clamped
// instead of the load skipped: a branch around each load would make every one its own round trip.
__device__ __forceinline__ half8 mat8(const uint16_t* m, int i, int j, int d) {
  const bool real = i < d && j < d;  // d % 8 == 0: the 8 columns are all real or all padding
  const half8 v = *reinterpret_cast<const half8*>(m + (real ? i * d + j : 0));
  return real ? v : half8{};
}

constexpr int kDenseKeys = 32;  // keys per tile
constexpr float kMixed = 0x1p-11f;  // keys below this part of their tile's bound make it a mixed tile
constexpr int kKeyFac = 2 * kDenseKeys;  // floats of a mixed tile's factors: (hi, lo) per key
template <int DP, bool VALS = true>
constexpr int dense_rec() { return (VALS ? 3 : 2) * DP * 64; }  // bytes of a tile record; keys only without VALS

// ---------------------------------------------------------------- query rotation
// q_rot = f16(q Pi^T) of q[B, Hq, Sq, d] (element strides), rows in (b, h, s) order.
struct RotArgs {
  const void* q;
  int64_t n, sqb, sqh, sqs;
  int Hq, Sq, d, vec, blocks;  // blocks along x that rotate; the ones after them lay S_eff out
  const uint16_t* pi;    // split Pi [2][d][d]
  const uint16_t* seff;  // f16 S_eff [d][d]
  uint16_t *q_rot, *seff_frag;
};

// Output blocks (32 dims) whose weights a block holds in LDS (16 KiB each at head_dim 128)
template <int DP>
constexpr int rot_blocks() { return DP <= 192 ? DP / 32 : 4; }

// A wave owns 32 rows (MFMA columns) and computes every output dim of its block's weight planes,
// which sit in LDS as fragments in lane order.  bf16 / f16 rows are exact f16 operands under a
// power-of-two row scale: the weight's hi and lo parts against one operand, 2 passes; f32 rows are
// split too, 3 passes.  Blocks past a.blocks write S_eff^T as the expansion's A fragments (32-dim
// block w, k-step s: row m is dim 32 w + perm32(m), k-slot e is S_eff row 16 s + 8 h + e), so that
// it reads them 16 bytes per lane instead of as single halves of S_eff's columns.
// A few thousand rows leave the chip half idle (256 rows a block: 128 blocks for 32k rows), every block
// staging its weights first: 10 us for 8 MB of rows.  f32 rows keep both parts of a row and spill from
// head_dim 128 on (18 VGPRs there, 44 at 192, 104 at 224, 217 at 256; bf16 at 256: 10).
template <int DP, int DT>
__global__ void __launch_bounds__(512) dense_rotate_kernel(RotArgs a) {
  constexpr int KS = DP / 16, NOB = rot_blocks<DP>(), NF = NOB * KS;
  constexpr bool EXACT = DT != TQ_F32;
  __shared__ __attribute__((aligned(16))) half8 wsm[2 * NF * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5, d = a.d, ob0 = blockIdx.y * NOB;
  if (static_cast<int>(blockIdx.x) >= a.blocks) {
    if (blockIdx.y) return;
    for (int f = (static_cast<int>(blockIdx.x) - a.blocks) * 8 + wave; f < KS * (DP / 32);
         f += (static_cast<int>(gridDim.x) - a.blocks) * 8) {
      const int j = 32 * (f / KS) + perm32(n);
      half8 v = half8{};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int i = 16 * (f % KS) + 8 * h + e;
        if (i < d && j < d) v[e] = __builtin_bit_cast(_Float16, a.seff[i * d + j]);
      }
      reinterpret_cast<half8*>(a.seff_frag)[f * 64 + lane] = v;
    }
    return;
  }
  for (int f = wave; f < 2 * NF; f += 8) {
    const int pl = f / NF, r = f - pl * NF, i = 32 * (ob0 + r / KS) + perm32(n), j = 16 * (r % KS) + 8 * h;
    wsm[f * 64 + lane] = mat8(a.pi + static_cast<int64_t>(pl) * d * d, i, j, d);
  }
  const int64_t nt = (a.n + 31) / 32, step = static_cast<int64_t>(a.blocks) * 8;
  constexpr int RW = EXACT ? 1 : 2;
  u32x4 raw[KS][RW];  // this lane's elements 16 ks + 8 h + 0..7 of its row
  auto fetch = [&](int64_t t) __attribute__((always_inline)) {
    const int64_t g = min(t * 32 + n, a.n - 1);
    const int64_t bh = g / a.Sq, s = g - bh * a.Sq, b = bh / a.Hq, hq = bh - b * a.Hq;
    constexpr int ES = EXACT ? 2 : 4;
    // a half past a row's end (h = 1 of a head dim of 8 mod 16) reads the row's start instead
    const uint8_t* p = static_cast<const uint8_t*>(a.q) + (b * a.sqb + hq * a.sqh + s * a.sqs + (8 * h < d ? 8 * h : 0)) * ES;
    if (a.vec) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bool real = 16 * ks + 8 * h < d;
#pragma unroll
        for (int r = 0; r < RW; ++r) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(p + (real ? 16 * ks * ES + 16 * r : 0));
          raw[ks][r] = real ? v : u32x4{0u, 0u, 0u, 0u};
        }
      }
      return;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        const bool real = 16 * ks + 8 * h < d;
        const uint8_t* pp = p + (real ? 16 * ks * ES + 16 * r : 0);
        u32x4 v;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if constexpr (EXACT)
            v[w] = static_cast<uint32_t>(reinterpret_cast<const uint16_t*>(pp)[2 * w]) |
                   (static_cast<uint32_t>(reinterpret_cast<const uint16_t*>(pp)[2 * w + 1]) << 16);
          else v[w] = reinterpret_cast<const uint32_t*>(pp)[w];
        }
        raw[ks][r] = real ? v : u32x4{0u, 0u, 0u, 0u};
      }
  };
  auto at = [&](int ks, int e) __attribute__((always_inline)) {
    if constexpr (!EXACT) {
      return __uint_as_float(raw[ks][e >> 2][e & 3]);
    } else {
      const uint32_t u = raw[ks][0][e >> 1];
      const uint16_t v = static_cast<uint16_t>((e & 1) ? (u >> 16) : (u & 0xffffu));
      return DT == TQ_F16 ? h2f(v) : bf16_to_f32(v);
    }
  };
  int64_t t = static_cast<int64_t>(blockIdx.x) * 8 + wave;
  if (t < nt) fetch(t);
  __syncthreads();
  for (; t < nt; t += step) {
    float mx = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(at(ks, e)));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    int e2;
    frexpf(mx, &e2);
    e2 = e2 < -100 ? -100 : e2;  // tiny rows: the scale stays finite
    constexpr int SX = EXACT ? 15 : 10;
    const float sc = ldexpf(1.f, SX - e2), inv = ldexpf(1.f / kSplit, e2 - SX);
    half8 xh[KS], xl[EXACT ? 1 : KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (EXACT) {
          xh[ks][e] = static_cast<_Float16>(at(ks, e) * sc);
        } else {
          _Float16 vh, vl;
          split_f16(at(ks, e) * sc, vh, vl);
          xh[ks][e] = vh;
          xl[ks][e] = vl;
        }
      }
    if (t + step < nt) fetch(t + step);  // in flight during the products
    const int64_t gr = t * 32 + n;
    uint16_t* out = a.q_rot + gr * d;
#pragma unroll 1
    for (int ob = 0; ob < NOB; ++ob) {
      const half8* w = wsm + ob * KS * 64 + lane;
      float16v f = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        f = mfma32x32x16(w[ks * 64], xh[ks], f);
        f = mfma32x32x16(w[(NF + ks) * 64], xh[ks], f);
        if constexpr (!EXACT) f = mfma32x32x16(w[ks * 64], xl[ks], f);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int d0 = 32 * (ob0 + ob) + 16 * q + 8 * h;
        half8 r;
#pragma unroll
        for (int e = 0; e < 8; ++e) r[e] = static_cast<_Float16>(f[8 * q + e] * inv);
        if (gr < a.n && d0 < d) *reinterpret_cast<half8*>(out + d0) = r;
      }
    }
  }
}

// ---------------------------------------------------------------- expansion
struct ExpandArgs {
  const uint8_t *kcodes, *ksigns, *vcodes;
  const uint16_t *krn, *kvn, *vvn, *kcent, *seff_frag;
  const float* vcent;
  int Sk, d, kb, vb, ntile;  // ntile: tiles per (batch, kv head)
  int64_t ldk, bh0, total;   // total: tiles of this launch
  float coeff;
  uint8_t* tiles;
  float *tfac, *kfac;  // factor of each tile (0: a mixed tile); key factors of mixed tiles
};

// A row's bits of 32 dims, b <= 4 bits each, as dwords (dims past d read as code 0)
struct Field32 {
  uint32_t w[4];
  // codes of dims 8 g .. 8 g + 7 in the low 8 b bits
  __device__ __forceinline__ uint32_t codes8(int g, int b) const {
    const int bit = 8 * b * g;
    const uint32_t lo = (bit >> 5) == 0 ? w[0] : (bit >> 5) == 1 ? w[1] : (bit >> 5) == 2 ? w[2] : w[3];
    const uint32_t hi = (bit >> 5) == 0 ? w[1] : (bit >> 5) == 1 ? w[2] : w[3];
    return __builtin_amdgcn_alignbit(hi, lo, bit & 31);
  }
};
// W: bytes per load.  Rows are whole dwords at head dims that are multiples of 32, whole 16-bit
// words at other multiples of 16 (head_dim 80, 32 x 1531 keys: the expansion takes 18.3 us, by single
// bytes 21.4), single bytes otherwise
template <int W>
__device__ __forceinline__ Field32 load_field(const uint8_t* row, int blk, int b, int d) {
  Field32 f;
#pragma unroll
  for (int i = 0; i < 4; ++i) f.w[i] = 0;
  if constexpr (W == 4) {
    const uint32_t* p = reinterpret_cast<const uint32_t*>(row) + blk * b;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < b) f.w[i] = p[i];
  } else {
    const int n = min(32, d - 32 * blk) * b / 8;  // real bytes of the field
    const uint8_t* p = row + 4 * blk * b;
#pragma unroll
    for (int i = 0; i < 16 / W; ++i)
      if (W * i < n) {
        const uint32_t v = W == 2 ? reinterpret_cast<const uint16_t*>(p)[i] : p[i];
        f.w[W * i >> 2] |= v << (8 * (W * i & 3));
      }
  }
  return f;
}

// One wave per 32-dim block; blocks walk the tiles.  Lane (key n, half h) of wave w ends with
// dims 32w + 16s + 8h + 0..7 (s = 0, 1) of its key: exactly its 16 bytes of k^ fragments 2w + s.
// V^ is transposed through a wave-private LDS tile.
template <int DP, int W, bool VALS>
__global__ void __launch_bounds__(2 * DP) dense_expand_kernel(ExpandArgs a) {
  constexpr int KS = DP / 16, NW = DP / 32;
  constexpr int VP = 36;  // halves per row of the V^ transposition tile
  __shared__ float s_kc[8], s_vc[16];
  __shared__ float s_bound[NW];
  __shared__ __attribute__((aligned(16))) _Float16 s_v[VALS ? NW : 1][32 * VP];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5, d = a.d;
  if (tid < 8) s_kc[tid] = tid < (1 << a.kb) ? h2f(a.kcent[tid]) : 0.f;
  if (VALS && tid >= 16 && tid < 32) s_vc[tid - 16] = tid - 16 < (1 << a.vb) ? a.vcent[tid - 16] : 0.f;

  half8 sf[KS];      // S_eff^T rows of this wave's dims
  float asum = 0.f;  // sum over S_eff's rows of |S_eff[., dim]|: bounds |S_eff^T s|
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    sf[s] = reinterpret_cast<const half8*>(a.seff_frag)[(w * KS + s) * 64 + lane];
#pragma unroll
    for (int e = 0; e < 8; ++e) asum += fabsf(static_cast<float>(sf[s][e]));
  }
  asum += __shfl_xor(asum, 32, 64);
  asum = wave_max(asum);
  if (lane == 0) s_bound[w] = asum;
  __syncthreads();
  float smax = 0.f, cmax = 0.f;  // |S_eff^T s| and |C| of any key
#pragma unroll
  for (int i = 0; i < NW; ++i) smax = fmaxf(smax, s_bound[i]);
#pragma unroll
  for (int i = 0; i < 8; ++i) cmax = fmaxf(cmax, fabsf(s_kc[i]));

  const int kc = d * a.kb / 8, sc = d / 8, vc = d * a.vb / 8;
  const uint32_t km = (1u << a.kb) - 1u, vm = (1u << a.vb) - 1u;
  // A tile's packed bytes of this lane's key, requested one tile ahead.  codes8 picks words by the
  // lane's half, so the compiler keeps the record in scratch (48 to 76 bytes a lane) and the wait before
  // each read back covers the request as well: the fetch is not hidden, and this chain, not the 6 bytes
  // written per element, bounds the kernel.
  struct Raw {
    uint32_t sw[NW];
    Field32 kf, vf;
    uint16_t vn, rn, vvn;
    bool ok;
  };
  auto fetch = [&](int64_t T) __attribute__((always_inline)) {
    const int64_t bh = T / a.ntile;
    const int k0 = static_cast<int>(T - bh * a.ntile) * kDenseKeys;
    const int64_t row = (a.bh0 + bh) * a.ldk + min(k0 + n, a.Sk - 1);
    Raw r;
    r.ok = k0 + n < a.Sk;
#pragma unroll
    for (int i = 0; i < NW; ++i) r.sw[i] = load_field<W>(a.ksigns + row * sc, i, 1, d).w[0];
    r.kf = load_field<W>(a.kcodes + row * kc, w, a.kb, d);
    if constexpr (VALS) r.vf = load_field<W>(a.vcodes + row * vc, w, a.vb, d);
    r.vn = a.kvn[row];
    r.rn = a.krn[row];
    if constexpr (VALS) r.vvn = a.vvn[row];
    return r;
  };
  Raw nx;
  if (blockIdx.x < a.total) nx = fetch(blockIdx.x);
  for (int64_t T = blockIdx.x; T < a.total; T += gridDim.x) {
    const Raw r = nx;
    if (T + gridDim.x < a.total) nx = fetch(T + gridDim.x);
    // keys past Sk have zero norms: k^ and V^ zero
    const float vn = r.ok ? h2f(r.vn) : 0.f, rn = r.ok ? a.coeff * h2f(r.rn) : 0.f;
    const Field32& kf = r.kf;
    // S_eff^T s: the sign bits as +-1 halves (a clear bit sets the half's sign bit).  Of a byte's
    // clear bits, y holds the even ones from bit 9 and the odd ones from bit 25 on, so that one
    // shift brings each pair to bits 15 and 31
    float16v acc = zero16();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint32_t nb = ~(r.sw[s >> 1] >> (16 * (s & 1) + 8 * h));
      const uint32_t y = (nb & 0x55u) << 9 | (nb & 0xAAu) << 24;
      u32x4 p;
#pragma unroll
      for (int q = 0; q < 4; ++q) p[q] = ((y << (6 - 2 * q)) & 0x80008000u) | 0x3C003C00u;
      acc = mfma32x32x16(sf[s], __builtin_bit_cast(half8, p), acc);
    }
    // power-of-two tile scale: the bound vn cmax + |coeff| rn smax of the tile's largest |k^| lands
    // in [2^13, 2^14)
    const float bound = wave_max(fabsf(vn)) * cmax + wave_max(fabsf(rn)) * smax;
    const float own = fabsf(vn) * cmax + fabsf(rn) * smax;  // this key's bound
    const bool finite = own <= 3.0e38f;
    const bool mixed = __any(own != 0.f && !(finite && own >= bound * kMixed));  // the same for every wave
    float up = qproj_split_scale(bound);
    if (tid == 0) a.tfac[T] = mixed ? 0.f : 1.f / up;
    uint8_t* rec = a.tiles + T * dense_rec<DP, VALS>();
    if (mixed) {  // a key of finite norms takes a power of two of its own
      asm volatile("; mixed tile" ::: "memory");
      int e;
      frexpf(own, &e);
      up = finite && own > 0.f ? ldexpf(1.f, 14 - e) : 1.f;
      if (tid < kDenseKeys) {  // lanes (key tid, h 0) of wave 0
        float* f = a.kfac + T * kKeyFac + 2 * tid;
        f[0] = finite ? 1.f / up : vn;
        f[1] = finite ? 1.f / up : rn;
      }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bool real = 32 * w + 16 * s + 8 * h < d;  // this lane's 8 dims
      half8 hi, lo;
      const uint32_t c = kf.codes8(2 * s + h, a.kb);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = real ? fmaf(rn, acc[8 * s + e], vn * s_kc[(c >> (a.kb * e)) & km]) * up : 0.f;
        _Float16 vh, vl;
        split_f16(v, vh, vl);
        hi[e] = vh;
        lo[e] = vl;
      }
      *reinterpret_cast<half8*>(rec + (2 * w + s) * 1024 + lane * 16) = hi;
      *reinterpret_cast<half8*>(rec + (KS + 2 * w + s) * 1024 + lane * 16) = lo;
    }
    if (mixed && !finite) {
      // infinite (or NaN) norms: the two terms apart, C in hi and S_eff^T s (one f16: only its sign
      // matters) in lo.  The norms are the key's factors and enter with the scores, as the packed kernels
      // have it: a score of +-inf
      asm volatile("; norms not finite" ::: "memory");
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bool real = 32 * w + 16 * s + 8 * h < d;
        half8 hi, lo;
        const uint32_t c = kf.codes8(2 * s + h, a.kb);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          hi[e] = static_cast<_Float16>(real ? s_kc[(c >> (a.kb * e)) & km] : 0.f);
          lo[e] = static_cast<_Float16>(real ? acc[8 * s + e] : 0.f);
        }
        *reinterpret_cast<half8*>(rec + (2 * w + s) * 1024 + lane * 16) = hi;
        *reinterpret_cast<half8*>(rec + (KS + 2 * w + s) * 1024 + lane * 16) = lo;
      }
    }
    if constexpr (VALS) {
      // V^ into row perm32 of the block
      const float vvn = r.ok ? h2f(r.vvn) : 0.f;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bool real = 32 * w + 16 * s + 8 * h < d;
        const uint32_t cv = r.vf.codes8(2 * s + h, a.vb);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float v = real ? s_vc[(cv >> (a.vb * e)) & vm] * vvn : 0.f;
          s_v[w][perm32(16 * s + 8 * h + e) * VP + n] = static_cast<_Float16>(v);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // fragment 2w + s of V^: row n, keys 16s + 4h + 0..3 and 16s + 8 + 4h + 0..3, the key order
      // of the accumulator registers 8s..8s+7 that become the P operand
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const _Float16* p = &s_v[w][n * VP + 16 * s + 4 * h];
        const half4 x = *reinterpret_cast<const half4*>(p), y = *reinterpret_cast<const half4*>(p + 8);
        *reinterpret_cast<half8*>(rec + (2 * KS + 2 * w + s) * 1024 + lane * 16) =
            half8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
}

// ---------------------------------------------------------------- attention
struct DenseArgs {
  const uint16_t* q_rot;
  const uint8_t* tiles;
  const float *tfac, *kfac;
  const uint16_t* vpit;  // split Pi_v^T (hi, lo), [2][d][d]
  int Hq, Hkv, Sq, Sk, d, G, QT, nqb, nbh, ntile;
  int64_t bh0;
  float scale;
  int causal;
  const void* mask;  // f32, f16 or bf16 (mask_dtype)
  int mask_dtype;
  int64_t smb, smh, smq, smk;
  void* out;  // contiguous [B, Sq, Hq, d]
  int out_dtype;
  // keys split over blocks: split s takes tiles [s * cpt, (s + 1) * cpt) of its query block
  float *part_o, *part_ml;
  int nsplit, cpt;
};

// 4 or 8 waves of 32 columns; up to head_dim 128 two or three waves per SIMD (at most 256 VGPRs each),
// above one.
// RES: blocks that share a compute unit's LDS (4-wave blocks; a lone one takes a deeper ring: the
// copies' latency is longer than one wave per SIMD takes for a tile).
template <int DP, int NW, bool MASK, int RES>
struct DenseCfg {
  static constexpr int KS = DP / 16, DB = DP / 32, REC = dense_rec<DP>();
  static constexpr int CPW = (REC / 1024 + NW - 1) / NW;  // 1 KiB copies per wave and tile
  static constexpr int KIB = 160 / RES;                   // LDS of one block
  static constexpr bool MDMA = MASK && 3 * REC + NW * 8192 <= KIB * 1024;  // mask values through LDS
  static constexpr int MB = MDMA ? NW * 8192 : 16;
  // ring slots: the tile being finished, the one being scored, the others in flight
  static constexpr int FIT = (KIB * 1024 - MB) / REC;
  static constexpr int NS = FIT >= 6 ? 6 : FIT;
  static constexpr int WPE = NW == 8 ? 2 : RES;  // waves per SIMD
  // six slots allow one block barrier per two tiles, with copies NS - 2 tiles ahead instead of NS - 1
  // (a tile of 256 columns at head_dim 128: 0.94 -> 0.90 us; of 128 at head_dim 64: 0.45 -> 0.43)
  static constexpr bool PAIR = NS == 6 && !MASK;
  static constexpr int LEAD = PAIR ? NS - 2 : NS - 1;
  static_assert(NS >= 3 && (LEAD - 2) * CPW < 64, "ring");
};

// Block -> work: query blocks heavy first across every (batch, kv head); consecutive blocks are
// different (batch, kv head)s, so each XCD (blocks dealt round-robin) keeps to a fixed set of them
struct DenseBlock {
  int qblk, split, bhi;
};
__device__ __forceinline__ DenseBlock dense_block(const DenseArgs& a, int id) {
  const int r = id / a.nbh;
  return {a.nqb - 1 - r / a.nsplit, r % a.nsplit, id % a.nbh};
}
// tiles that query block `qblk` attends
__device__ __forceinline__ int dense_tiles(const DenseArgs& a, int qblk) {
  int kend = a.Sk;
  if (a.causal) kend = min(a.Sk, min(qblk * a.QT + a.QT - 1, a.Sq - 1) + (a.Sk - a.Sq) + 1);
  return (kend + kDenseKeys - 1) / kDenseKeys;
}

struct DenseCol {
  int qi, hq;
  bool ok;
};
__device__ __forceinline__ DenseCol dense_col(const DenseArgs& a, int qblk, int hkv, int r) {
  const int ql = static_cast<int>(static_cast<uint32_t>(r) / static_cast<uint32_t>(a.G)), gi = r - ql * a.G;
  DenseCol c;
  c.qi = qblk * a.QT + ql;
  c.hq = hkv * a.G + gi;
  c.ok = ql < a.QT && c.qi < a.Sq;
  return c;
}

__device__ __forceinline__ void store8(void* p, int64_t i, int dtype, const float (&v)[8]) {
  if (dtype == TQ_F32) {
    float* o = static_cast<float*>(p) + i;
    *reinterpret_cast<float4v*>(o) = float4v{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<float4v*>(o + 4) = float4v{v[4], v[5], v[6], v[7]};
    return;
  }
  u32x4 w;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t lo = dtype == TQ_F16 ? f2h(v[2 * q]) : f32_to_bf16(v[2 * q]);
    const uint32_t hi = dtype == TQ_F16 ? f2h(v[2 * q + 1]) : f32_to_bf16(v[2 * q + 1]);
    w[q] = lo | (hi << 16);
  }
  *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(p) + i) = w;
}

// out = (O^T / l)^T Pi_v for this lane's column: O^T registers 8s..8s+7 of block db are dims
// 32 db + 16 s + 8 h + 0..7 (perm32), i.e. the B operand of k-step 2 db + s; Pi_v^T rows as split-f16
// A operands in the same row order, so a lane ends with runs of 8 output dims.  Pi_v^T's fragments
// are copied into the block's idle ring where they fit (RING bytes), all in flight during the
// normalisation: read from memory block by block they cost a round trip per 32 output dims, 10 us
// of a block's life at head_dim 128.  Every wave of the block calls this (block barriers).
template <int DP, int NW, int RING>
__device__ __forceinline__ void dense_finish(const DenseArgs& a, float16v (&o)[DP / 32], float l, const DenseCol& c,
                                             int64_t b, int lane, int wave, uint8_t* ring) {
  constexpr int KS = DP / 16, DB = DP / 32, NF = 2 * DB * KS;  // fragments: [hi, lo][block][k-step]
  constexpr bool LDS = NF * 1024 <= RING;
  const int n = lane & 31, h = lane >> 5, d = a.d;
  if constexpr (LDS) {
    wait_lds();
    __builtin_amdgcn_s_barrier();  // every wave is done with the ring
    asm volatile("" ::: "memory");
    const uint64_t p = reinterpret_cast<uint64_t>(a.vpit);
    const i32x4 r{static_cast<int>(static_cast<uint32_t>(p)), static_cast<int>(static_cast<uint32_t>(p >> 32) & 0xffffu),
                  4 * d * d, 0x00020000};
    const uint32_t dst = lds_offset(ring);
#pragma unroll
    for (int u = 0; u < (NF + NW - 1) / NW; ++u) {
      const int f = NF % NW == 0 ? wave + NW * u : min(wave + NW * u, NF - 1);
      const int pl = f / (DB * KS), ib = f % (DB * KS) / KS, ks = f % KS;
      const int i = 32 * ib + perm32(n), j = 16 * ks + 8 * h;
      dma16_cached(r, dst + f * 1024, i < d && j < d ? static_cast<uint32_t>(((pl * d + i) * d + j) * 2) : kOutOfRange);
    }
  }
  l += __shfl_xor(l, 32, 64);
  const float inv_l = l > 0.f ? 1.f / l : 0.f;
  float mx = 0.f;
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    o[db] *= inv_l;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, fabsf(o[db][i]));
  }
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  int ex;
  frexpf(mx, &ex);
  const float up = ldexpf(kSplit, -ex), down = ldexpf(kUnsplit2, ex);
  half8 oh[KS], ol[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      _Float16 vh, vl;
      split_f16(o[ks >> 1][8 * (ks & 1) + e] * up, vh, vl);
      oh[ks][e] = vh;
      ol[ks][e] = vl;
    }
  if constexpr (LDS) {
    wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  const uint16_t* ph = a.vpit;
  const uint16_t* pl = a.vpit + static_cast<int64_t>(d) * d;
  const int64_t orow = ((b * a.Sq + c.qi) * a.Hq + c.hq) * static_cast<int64_t>(d);
#pragma unroll 1
  for (int ib = 0; ib < DB; ++ib) {
    float16v f = zero16();
    half8 ah[KS], al[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if constexpr (LDS) {
        ah[ks] = *reinterpret_cast<const half8*>(ring + (ib * KS + ks) * 1024 + lane * 16);
        al[ks] = *reinterpret_cast<const half8*>(ring + ((DB + ib) * KS + ks) * 1024 + lane * 16);
      } else {
        const int i = 32 * ib + perm32(n);
        ah[ks] = mat8(ph, i, 16 * ks + 8 * h, d);
        al[ks] = mat8(pl, i, 16 * ks + 8 * h, d);
      }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      f = mfma32x32x16(ah[ks], oh[ks], f);
      f = mfma32x32x16(al[ks], oh[ks], f);
      f = mfma32x32x16(ah[ks], ol[ks], f);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int d0 = 32 * ib + 16 * s + 8 * h;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = f[8 * s + e] * down;
      if (c.ok && d0 < d) store8(a.out, orow + d0, a.out_dtype, v);
    }
  }
}

// A block owns 32 NW (query row, query head) columns of one (batch, kv head) and walks its
// tiles; S^T = K^ Q_rot^T (keys are MFMA rows), online softmax down the rows, O^T += V^T P^T with
// P = f16(2^(s - m)) straight from S^T's registers.  The scores of tile t + 1 are issued with the
// softmax of tile t, so that a wave's matrix and vector work overlap.  Records are copied into an
// LDS ring with direct-to-LDS loads, LEAD tiles ahead; one block barrier per tile, or per two tiles
// (PAIR) while no tile needs masking.
template <int DP, int NW, bool MASK, bool PLO, int RES>
__global__ void __launch_bounds__(64 * NW)
__attribute__((amdgpu_waves_per_eu(DenseCfg<DP, NW, MASK, RES>::WPE)))
dense_attn_kernel(DenseArgs a) {
  using C = DenseCfg<DP, NW, MASK, RES>;
  constexpr bool MDMA = C::MDMA;
  constexpr int KS = C::KS, DB = C::DB, REC = C::REC, NS = C::NS, CPW = C::CPW, NF = REC / 1024, LEAD = C::LEAD;
  constexpr float LOG2E = 1.4426950408889634f;
  constexpr float TAU = 8.0f;  // lazy-rescale headroom (log2 units)
  __shared__ __attribute__((aligned(16))) uint8_t ring[NS * REC];
  // mask values of two tiles, per wave: 32 columns x 32 keys
  __shared__ __attribute__((aligned(16))) uint8_t smask[C::MB];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const DenseBlock blk = dense_block(a, blockIdx.x);
  const int qblk = blk.qblk, split = blk.split;
  const uint32_t bh = static_cast<uint32_t>(a.bh0 + blk.bhi);  // < 2^31 (host check)
  const int hkv = static_cast<int>(bh % static_cast<uint32_t>(a.Hkv));
  const int64_t b = bh / static_cast<uint32_t>(a.Hkv);
  // tiles [tb, te) of this block
  const int tb = split * a.cpt;
  const int te = min(dense_tiles(a, qblk), tb + a.cpt);
  if (a.nsplit > 1 && tb >= te) return;

  // ---- this lane's column
  const DenseCol c = dense_col(a, qblk, hkv, wave * 32 + n);
  const int off = a.Sk - a.Sq;
  const int lim = a.causal ? min(c.qi + off, a.Sk - 1) : a.Sk - 1;  // last key this column attends
  half8 qf[KS];
  {
    const uint16_t* q = a.q_rot + ((b * a.Hq + (c.ok ? c.hq : 0)) * a.Sq + (c.ok ? c.qi : 0)) * static_cast<int64_t>(a.d);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d0 = 16 * ks + 8 * h;
      const bool real = c.ok && d0 < a.d;
      const half8 v = *reinterpret_cast<const half8*>(q + (real ? d0 : 0));
      qf[ks] = real ? v : half8{};
    }
  }
  // this wave's tiles end at tw (its last row's last key); tiles from tf on need masking, tiles before
  // tfb in no wave of the block.  A wave without columns (tw = tb) only copies
  int tw = te, tf = te;
  int tfb = min(te, (a.causal ? min(qblk * a.QT + off + 1, a.Sk) : a.Sk) / kDenseKeys);
  {
    const int ql0 = wave * 32 / a.G, ql1 = min((wave * 32 + 31) / a.G, a.QT - 1);
    const int i0 = qblk * a.QT + ql0, i1 = min(qblk * a.QT + ql1, a.Sq - 1);
    const int l1 = a.causal ? min(i1 + off, a.Sk - 1) : a.Sk - 1;
    const int l0 = a.causal ? min(i0 + off, a.Sk - 1) : a.Sk - 1;
    tw = (ql0 >= a.QT || i0 >= a.Sq) ? tb : max(tb, min(te, l1 / kDenseKeys + 1));
    tf = max(tb, min(tw, (l0 + 1) / kDenseKeys));
  }
  // The mask reaches a lane through LDS: a tile's 32 columns x 32 keys as whole row segments
  // (64 or 128 bytes per column, copied one tile ahead) instead of 8- or 16-byte pieces of 32 rows
  // per load.  Rows must be whole dwords from a dword on and contiguous in keys (a 16-bit row of an odd
  // key count ends inside a dword: its copy would read past the mask or drop the last key); others are
  // read directly.
  // Segment c of column r sits at chunk c ^ (r's bits that pick its banks): conflict-free reads.
  [[maybe_unused]] const uint8_t* mrow = nullptr;
  [[maybe_unused]] const uint8_t* mbase = nullptr;
  [[maybe_unused]] bool mdma = false, m32 = false;
  [[maybe_unused]] uint32_t moff[MASK ? 4 : 1];
  if constexpr (MASK) {
    m32 = a.mask_dtype == TQ_F32;
    const int es = m32 ? 4 : 2;
    const int64_t bq = b * a.smb + static_cast<int64_t>(hkv) * a.G * a.smh + static_cast<int64_t>(qblk) * a.QT * a.smq;
    mbase = static_cast<const uint8_t*>(a.mask) + bq * es;
    auto at = [&](const DenseCol& k) {  // element offset of a column's row from mbase
      return k.ok ? (k.hq - hkv * a.G) * a.smh + (k.qi - qblk * a.QT) * a.smq : int64_t{0};
    };
    mrow = mbase + at(c) * es;
    const int64_t far = (a.G - 1) * (a.smh < 0 ? -a.smh : a.smh) + a.QT * (a.smq < 0 ? -a.smq : a.smq) + a.Sk;
    mdma = MDMA && a.smk == 1 && a.smh >= 0 && a.smq >= 0 && far * es < (int64_t(1) << 31) &&
           (reinterpret_cast<uintptr_t>(a.mask) & 3) == 0 && ((a.smb | a.smh | a.smq | a.Sk) * es & 3) == 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = m32 ? 8 * i + (lane >> 3) : 16 * (i & 1) + (lane >> 2);
      const int seg = m32 ? (lane & 7) ^ (r & 7) : (lane & 3) ^ ((r >> 1) & 3);
      moff[i] = static_cast<uint32_t>(at(dense_col(a, qblk, hkv, wave * 32 + r)) * es + seg * 16);
    }
  }

  // ---- ring
  const uint8_t* recs = a.tiles + static_cast<int64_t>(blk.bhi) * a.ntile * REC;
  const float* tfac = a.tfac + static_cast<int64_t>(blk.bhi) * a.ntile;
  const float* kfac = a.kfac + static_cast<int64_t>(blk.bhi) * a.ntile * kKeyFac;
  const uint32_t ring_lds = lds_offset(ring);
  // copy the next tile's record into the ring; past the last tile the last one again (into a free
  // slot), so that every iteration has the same number of copies in flight.  The descriptor and the
  // slot advance by one record per call
  uint64_t src = reinterpret_cast<uint64_t>(recs) + static_cast<uint64_t>(tb) * REC;
  int left = te - tb;  // tiles not yet copied
  uint32_t dst = ring_lds;
  auto issue = [&]() __attribute__((always_inline)) {
    const i32x4 r{static_cast<int>(static_cast<uint32_t>(src)), static_cast<int>(static_cast<uint32_t>(src >> 32) & 0xffffu),
                  REC, 0x00020000};
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
      const int f = NF % NW == 0 ? wave + NW * i : min(wave + NW * i, NF - 1);  // surplus: the last fragment again
      dma16_cached(r, dst + f * 1024, f * 1024 + lane * 16);
    }
    if (--left > 0) src += REC;
    dst = dst + REC == ring_lds + NS * REC ? ring_lds : dst + REC;
  };
  // the record issued LEAD - 2 calls before the latest one has landed (this wave's copies)
  auto landed = [&]() __attribute__((always_inline)) {
    // mask copies of a tile are issued one iteration ahead, before that iteration's record
    if constexpr (MASK) wait_vm<(NS > 3 ? CPW : 0)>();
    else wait_vm<(LEAD - 2) * CPW>();
  };
  auto block_sync = [&]() __attribute__((always_inline)) {
    wait_lds();  // this wave's fragment reads are done: their slot may be overwritten
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  float mref = 0.f, thr = -INFINITY, l_run = 0.f;
  float16v o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = zero16();
  float sc[16];                      // scores of the tile at hand relative to mref, log2 units
  const float fa = a.scale * LOG2E;
  float fv = 0.f;                    // tile factors of 64 tiles, one per lane
  auto factors = [&](int t) __attribute__((always_inline)) {  // of tiles t .. t + 63
    fv = tfac[min(t + lane, te - 1)];
    wait_vm0_visible();
  };
  auto factor = [&](int t) __attribute__((always_inline)) {
    return fa * __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, fv), (t - tb) & 63));
  };
  auto mixed_tile = [&](int t) __attribute__((always_inline)) {
    return __builtin_amdgcn_readlane(__builtin_bit_cast(int, fv), (t - tb) & 63) == 0;
  };
  bool mixed = false;  // the block meets a mixed tile
  auto frag = [&](const uint8_t* rec, int f) __attribute__((always_inline)) {  // rec: record + lane * 16
    return *reinterpret_cast<const half8*>(rec + f * 1024);
  };
  // fragment of score step i: k^ hi, then k^ lo of k-step i / 2
  constexpr auto kfrag = [](int i) { return (i & 1) * KS + (i >> 1); };

  // mask values of tile t: keys 32t + 8g + 4h + 0..3
  [[maybe_unused]] float4v mk[4];
  [[maybe_unused]] auto load_mask = [&](int t) __attribute__((always_inline)) {
    if (MDMA && mdma) {
      const uint8_t* p = smask + (wave * 2 + (t & 1)) * 4096;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (m32) {
          mk[g] = *reinterpret_cast<const float4v*>(p + n * 128 + (((2 * g + h) ^ (n & 7)) << 4));
        } else {
          const u32x2 u = *reinterpret_cast<const u32x2*>(p + n * 64 + ((g ^ ((n >> 1) & 3)) << 4) + 8 * h);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint16_t v = static_cast<uint16_t>((e & 1) ? (u[e >> 1] >> 16) : (u[e >> 1] & 0xffffu));
            mk[g][e] = a.mask_dtype == TQ_F16 ? h2f(v) : bf16_to_f32(v);
          }
        }
      }
      return;
    }
    const int kb = t * kDenseKeys + 4 * h;
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = kb + 8 * g + e;
        const int64_t at = static_cast<int64_t>(k) * a.smk;
        if (k >= a.Sk) mk[g][e] = 0.f;
        else if (a.mask_dtype == TQ_F32) mk[g][e] = load_act<TQ_F32>(mrow, at);
        else if (a.mask_dtype == TQ_F16) mk[g][e] = load_act<TQ_F16>(mrow, at);
        else mk[g][e] = load_act<TQ_BF16>(mrow, at);
      }
  };
  // copy this wave's mask values of tile t.  The range check ends at the last byte that any of the
  // block's rows may hold for a key below Sk: nothing past the mask is read
  [[maybe_unused]] auto issue_mask = [&](int t) __attribute__((always_inline)) {
    if (!MDMA || !mdma || t >= tw) return;
    const int es = m32 ? 4 : 2;
    const int rows = min(a.QT, a.Sq - qblk * a.QT);
    const int64_t end = ((a.G - 1) * a.smh + (rows - 1) * a.smq + a.Sk) * es;
    const int64_t base = static_cast<int64_t>(t) * kDenseKeys * es;
    const uint64_t p = reinterpret_cast<uint64_t>(mbase) + base;
    const i32x4 r{static_cast<int>(static_cast<uint32_t>(p)), static_cast<int>(static_cast<uint32_t>(p >> 32) & 0xffffu),
                  static_cast<int>(end - base), 0x00020000};
    const uint32_t dst = lds_offset(smask) + (wave * 2 + (t & 1)) * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (m32 || i < 2) dma16_cached(r, dst + i * 1024, moff[i]);
  };
  // score i of a tile from its product: relative to mref, or absolute under a mask (a first tile
  // of finfo.min would otherwise leave no bits of the real scores in s - m)
  auto score_at = [&](float v, int i, float f) __attribute__((always_inline)) {
    if constexpr (MASK) return fmaf(v, f, fmaxf(mk[i >> 2][i & 3] * LOG2E, -3.0e38f));
    else return fmaf(v, f, -mref);
  };
  auto clip_edge = [&](int t) __attribute__((always_inline)) {
    const int kb = t * kDenseKeys + 4 * h;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (kb + 8 * (i >> 2) + (i & 3) > lim) sc[i] = -INFINITY;
  };
  // The column's reference maximum moves only when a score exceeds it by more than TAU: each lane
  // tests its own scores (lmax); the exact maxima and the rescale run in the rare branch.
  auto settle = [&](float lmax) __attribute__((always_inline)) {
    if (__any((MASK ? lmax - mref : lmax) > thr)) {
      asm volatile("; rescale");
      const float tmax = fmaxf(lmax, __shfl_xor(lmax, 32, 64));
      const bool grow = (MASK ? tmax - mref : tmax) > thr;
      const float m_new = grow ? (MASK ? tmax : tmax + mref) : mref;
      const float alpha = (grow && thr != -INFINITY) ? __builtin_amdgcn_exp2f(mref - m_new) : 1.f;
      if constexpr (!MASK) {
        const float shift = m_new - mref;
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] -= shift;
      }
      mref = m_new;
      thr = grow ? TAU : thr;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] *= alpha;
    }
    if constexpr (MASK) {
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[i] -= mref;
    }
  };
  auto max16 = [&]() __attribute__((always_inline)) {
    return max_raw(max8_raw(sc[0], sc[1], sc[2], sc[3], sc[4], sc[5], sc[6], sc[7]),
                   max8_raw(sc[8], sc[9], sc[10], sc[11], sc[12], sc[13], sc[14], sc[15]));
  };
  // scores of a mixed tile t (landed at `rec`): hi and lo products under their keys' own factors
  auto mixed_scores = [&](int t, const uint8_t* rec) __attribute__((always_inline)) {
    asm volatile("; mixed tile" ::: "memory");  // fragments are read anew: none is kept for this branch
    float16v sh = zero16(), sl = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      sh = mfma32x32x16(frag(rec, ks), qf[ks], sh);
      sl = mfma32x32x16(frag(rec, KS + ks), qf[ks], sl);
    }
    const float* kf = kfac + static_cast<int64_t>(t) * kKeyFac + 8 * h;
#pragma unroll
    for (int i = 0; i < 16; i += 2) {  // keys 8 (i / 4) + 4 h + i % 4, + 1
      const float4v k2 = *reinterpret_cast<const float4v*>(kf + 16 * (i >> 2) + 2 * (i & 3));
      sc[i] = score_at(fmaf(sl[i], k2[1], sh[i] * k2[0]), i, fa);
      sc[i + 1] = score_at(fmaf(sl[i + 1], k2[3], sh[i + 1] * k2[2]), i + 1, fa);
    }
  };
  // scores of tile t (landed at `rec`) with nothing to overlap: the first tile
  auto first_scores = [&](int t, const uint8_t* rec) __attribute__((always_inline)) {
    float16v s = zero16();
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) s = mfma32x32x16(frag(rec, kfrag(i)), qf[i >> 1], s);
    if constexpr (MASK) load_mask(t);
    const float f = factor(t);
#pragma unroll
    for (int i = 0; i < 16; ++i) sc[i] = score_at(s[i], i, f);
    if (mixed && mixed_tile(t)) mixed_scores(t, rec);
    if (t >= tf) clip_edge(t);
    settle(max16());
  };
  const half2v one2 = {static_cast<_Float16>(1.f), static_cast<_Float16>(1.f)};
  // One tile: P and P.V of tile t (scores in sc, values at `cur`), with the scores of tile
  // t + 1 (at `nxt`) when `more`.  The order is written out: 2 KS score MFMAs with the
  // exponentials of tile t between them, then the P.V MFMAs with the score scaling of tile t + 1
  // between them, fragments read PF steps ahead.
  auto tile = [&](int t, const uint8_t* cur, const uint8_t* nxt, auto more) __attribute__((always_inline)) {
    constexpr bool MORE = decltype(more)::value;
    constexpr int PF = 4, NQK = 2 * KS, NPV = 2 * DB, NST = (MORE ? NQK : 0) + NPV;
    [[maybe_unused]] half8 pl[2];  // lo parts of P (PLO)
    half8 fr[PF];
    // fragment of step i of the whole sequence: score steps, then P.V steps (dim block db,
    // 16-key half k): value fragments 2 db + k, visited with k outermost
    auto step_frag = [&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      if constexpr (MORE && i < NQK) return frag(nxt, kfrag(i));
      else {
        constexpr int j = i - (MORE ? NQK : 0);
        return frag(cur, 2 * KS + 2 * (j % DB) + j / DB);
      }
    };
    half8 pb[2];
    auto exp_pair = [&](int q) __attribute__((always_inline)) {  // P of registers 2q, 2q + 1
      const float p0 = __builtin_amdgcn_exp2f(sc[2 * q]), p1 = __builtin_amdgcn_exp2f(sc[2 * q + 1]);
      const half2v p = {static_cast<_Float16>(p0), static_cast<_Float16>(p1)};
      pb[q >> 2][2 * (q & 3)] = p[0];
      pb[q >> 2][2 * (q & 3) + 1] = p[1];
      if constexpr (PLO) {
        pl[q >> 2][2 * (q & 3)] = static_cast<_Float16>(p0 - static_cast<float>(p[0]));
        pl[q >> 2][2 * (q & 3) + 1] = static_cast<_Float16>(p1 - static_cast<float>(p[1]));
        l_run += p0 + p1;
      } else {
        l_run = __builtin_amdgcn_fdot2(p, one2, l_run, false);
      }
    };
    if constexpr (MORE && MASK) load_mask(t + 1);
    static_for<PF>([&](auto I) __attribute__((always_inline)) { fr[decltype(I)::value] = step_frag(I); });
    float16v s = zero16();
    if constexpr (MORE) {
      static_for<NQK>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        s = mfma32x32x16(fr[i % PF], qf[i >> 1], s);
        if constexpr (i + PF < NST) fr[i % PF] = step_frag(std::integral_constant<int, i + PF>{});
        // the 8 pairs of exponentials spread over the score steps
#pragma unroll
        for (int q = i * 8 / NQK; q < (i + 1) * 8 / NQK; ++q) exp_pair(q);
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) exp_pair(q);
    }
    const float f = MORE ? factor(t + 1) : 0.f;
    static_for<NPV>([&](auto J) __attribute__((always_inline)) {
      constexpr int j = decltype(J)::value, i = j + (MORE ? NQK : 0);
      o[j % DB] = mfma32x32x16(fr[i % PF], pb[j / DB], o[j % DB]);
      if constexpr (PLO) o[j % DB] = mfma32x32x16(fr[i % PF], pl[j / DB], o[j % DB]);
      if constexpr (i + PF < NST) fr[i % PF] = step_frag(std::integral_constant<int, i + PF>{});
      if constexpr (MORE) {
#pragma unroll
        for (int q = j * 16 / NPV; q < (j + 1) * 16 / NPV; ++q) sc[q] = score_at(s[q], q, f);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // A block with a mixed tile takes every tile as one that needs masking: the loops before that one know
  // nothing of mixed tiles.  (A tile's factor is 1/6000 of its record.)
  fv = tfac[min(tb + lane, te - 1)];
  float least = fv;
#pragma unroll 4
  for (int t = tb + 64; t < te; t += 64) least = fminf(least, tfac[min(t + lane, te - 1)]);
  mixed = __any(least == 0.f);
  if (mixed) tf = tfb = tb;
  wait_vm0_visible();  // q and the factors have landed: the ring's waits count copies only
  if (te > tb) {
#pragma unroll
    for (int i = 0; i < LEAD; ++i) {
      issue();
      if (i == 0) {
        if constexpr (MASK) issue_mask(tb);
      }
    }
    wait_vm<MASK ? 0 : (LEAD - 1) * CPW>();
    if constexpr (MASK) {
      issue_mask(tb + 1);
      if (NS > 3) wait_vm<0>();  // the first advance() leaves CPW copies in flight, not these
    }
    block_sync();
    const uint8_t* const ring0 = ring + lane * 16;
    const uint8_t* const ring1 = ring0 + NS * REC;
    const uint8_t* cur = ring0;  // tile t's record
    if (tb < tw) first_scores(tb, cur);
    auto next = [&](const uint8_t* p) { return p + REC == ring1 ? ring0 : p + REC; };
    // tile t + 1 landed for every wave, every wave done with tile t - 1: the slot of tile t + LEAD is free
    auto advance = [&](int t) __attribute__((always_inline)) {
      if (((t + 1 - tb) & 63) == 0) factors(t + 1);
      landed();
      block_sync();
      if constexpr (MASK) issue_mask(t + 2);
      issue();
    };
    int t = tb;
    if constexpr (C::PAIR) {
      // two tiles per barrier while the block's tiles need no masking (tfb: the same for its waves):
      // tiles t + 1 and t + 2 have landed, every wave is done with t - 1, so the slots of t - 2 and t - 1
      // take t + 4 and t + 5
      // (t - tb is even here: a new 64 tiles of factors can begin at t + 2 only)
      for (; t + 2 < tfb; t += 2) {
        wait_vm<(LEAD - 3) * CPW>();
        block_sync();
        issue();
        issue();
        const uint8_t* nxt = next(cur);
        if (tb < tw) {
          tile(t, cur, nxt, std::true_type{});
          settle(max16());
        }
        if (((t + 2 - tb) & 63) == 0) factors(t + 2);
        cur = next(nxt);
        if (tb < tw) {
          tile(t + 1, nxt, cur, std::true_type{});
          settle(max16());
        }
      }
    }
    for (; t + 1 < tf; ++t) {  // the next tile needs no masking
      advance(t);
      const uint8_t* nxt = next(cur);
      tile(t, cur, nxt, std::true_type{});
      settle(max16());
      cur = nxt;
    }
    for (; t + 1 < te; ++t) {
      advance(t);
      const uint8_t* nxt = next(cur);
      if (t + 1 < tw) {
        tile(t, cur, nxt, std::true_type{});
        if (mixed && mixed_tile(t + 1)) mixed_scores(t + 1, nxt);
        clip_edge(t + 1);
        settle(max16());
      } else if (t < tw) {
        tile(t, cur, nxt, std::false_type{});
      }
      cur = nxt;
    }
    if (t < tw) tile(t, cur, cur, std::false_type{});
    wait_vm<0>();  // no copy outlives the block
  }

  if (a.nsplit > 1) {
    // partial O^T in register order (coalesced), the reference its weights are relative to (-inf
    // while the column has none) and this wave's sums
    const int64_t rec = (static_cast<int64_t>(blk.bhi * a.nqb + qblk) * a.nsplit + split) * NW + wave;
    float* po = a.part_o + rec * (DB * 1024) + lane * 4;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4v*>(po + (4 * db + g) * 256) =
            float4v{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
    const float l = l_run + __shfl_xor(l_run, 32, 64);
    if (h == 0) {
      a.part_ml[(rec * 32 + n) * 2] = thr == -INFINITY ? -INFINITY : mref;
      a.part_ml[(rec * 32 + n) * 2 + 1] = l;
    }
    return;
  }
  dense_finish<DP, NW, NS * REC>(a, o, l_run, c, b, lane, wave, ring);
}

// Combines the splits of 32 columns (one wave's record), normalises and applies Pi_v.  Wave w of
// the block combines dims 32w..32w+31, all waves exchange their (hi, lo) operands through LDS, and
// wave w forms output dims 32w..32w+31; its Pi_v^T fragments are loaded before the partials.
template <int DP>
__global__ void __launch_bounds__(2 * DP) dense_merge_kernel(DenseArgs a, int nw) {
  constexpr int KS = DP / 16, DB = DP / 32, U = 4;  // splits loaded together
  __shared__ __attribute__((aligned(16))) half8 s_b[2][KS][64];
  __shared__ float s_mx[DB][32];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5, d = a.d;
  const int wave = blockIdx.x % nw, id = blockIdx.x / nw;
  const int qblk = id % a.nqb, bhi = id / a.nqb;
  const int64_t bh = a.bh0 + bhi, b = bh / a.Hkv;
  const DenseCol c = dense_col(a, qblk, static_cast<int>(bh % a.Hkv), wave * 32 + n);
  const int ns = min(a.nsplit, (dense_tiles(a, qblk) + a.cpt - 1) / a.cpt);
  const int64_t rec0 = static_cast<int64_t>(id) * a.nsplit * nw + wave;
  const uint16_t* ph = a.vpit;
  const uint16_t* pl = a.vpit + static_cast<int64_t>(d) * d;
  half8 ah[KS], al[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    ah[ks] = mat8(ph, 32 * w + perm32(n), 16 * ks + 8 * h, d);
    al[ks] = mat8(pl, 32 * w + perm32(n), 16 * ks + 8 * h, d);
  }
  const float* ml = a.part_ml + (rec0 * 32 + n) * 2;
  const int64_t mstep = static_cast<int64_t>(nw) * 64;
  float mx = -INFINITY;
  for (int s = 0; s < ns; ++s) mx = fmaxf(mx, ml[s * mstep]);
  float16v o = zero16();
  float l = 0.f;
  const float* po = a.part_o + rec0 * (DB * 1024) + w * 1024 + lane * 4;
  const int64_t pstep = static_cast<int64_t>(nw) * (DB * 1024);
  for (int s0 = 0; s0 < ns; s0 += U) {
    float4v v[U][4];
    float m[U], ls[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = min(s0 + u, ns - 1);  // the last batch repeats a split with weight 0
      m[u] = s0 + u < ns ? ml[s * mstep] : -INFINITY;
      ls[u] = ml[s * mstep + 1];
#pragma unroll
      for (int g = 0; g < 4; ++g) v[u][g] = *reinterpret_cast<const float4v*>(po + s * pstep + g * 256);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float wt = m[u] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[u] - mx);
      l = fmaf(wt, ls[u], l);
#pragma unroll
      for (int i = 0; i < 16; ++i) o[i] = fmaf(wt, v[u][i >> 2][i & 3], o[i]);
    }
  }
  const float inv_l = l > 0.f ? 1.f / l : 0.f;
  float om = 0.f;
  o *= inv_l;
#pragma unroll
  for (int i = 0; i < 16; ++i) om = fmaxf(om, fabsf(o[i]));
  om = fmaxf(om, __shfl_xor(om, 32, 64));
  if (h == 0) s_mx[w][n] = om;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < DB; ++i) om = fmaxf(om, s_mx[i][n]);
  int ex;
  frexpf(om, &ex);
  const float up = ldexpf(kSplit, -ex), down = ldexpf(kUnsplit2, ex);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    half8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      _Float16 vh, vl;
      split_f16(o[8 * s + e] * up, vh, vl);
      hi[e] = vh;
      lo[e] = vl;
    }
    s_b[0][2 * w + s][lane] = hi;
    s_b[1][2 * w + s][lane] = lo;
  }
  __syncthreads();
  float16v f = zero16();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const half8 bh8 = s_b[0][ks][lane];
    f = mfma32x32x16(ah[ks], bh8, f);
    f = mfma32x32x16(al[ks], bh8, f);
    f = mfma32x32x16(ah[ks], s_b[1][ks][lane], f);
  }
  const int64_t orow = ((b * a.Sq + c.qi) * a.Hq + c.hq) * static_cast<int64_t>(d);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int d0 = 32 * w + 16 * s + 8 * h;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = f[8 * s + e] * down;
    if (c.ok && d0 < d) store8(a.out, orow + d0, a.out_dtype, v);
  }
}

// ---------------------------------------------------------------- materialised scores
struct DenseScoreArgs {
  const uint16_t* q_rot;
  const uint8_t* tiles;  // keys only
  const float *tfac, *kfac;
  int Hq, Hkv, Sq, Sk, d, G, rchunks, nbh, ntile, nblk, cpt;  // rchunks: 32-row chunks of a head
  int64_t bh0;
  float* out;  // [B, Hq, Sq, Sk]
};

// A wave owns 32 query rows of one head (MFMA rows) and walks its block's key tiles (MFMA columns):
// accumulator register i of lane (key n, h) is row 8 (i / 4) + 4 h + i % 4, so that every store
// writes 32 consecutive keys of two rows, whole 128-byte lines.  Blocks of 4 waves take
// consecutive (head, row chunk)s of one kv head and a range of its tiles; records (16 KiB at
// head_dim 128) reach LDS as in dense_attn_kernel.  Bound by the 4 bytes written per score: 32 heads
// x 2048 x 2048 take 129 us (4.2 TB/s written; the tiled kernel took 322).  LINES: output rows are
// whole 128-byte lines, stored past the L2; rows that are not (Sk not a multiple of 32) leave half
// lines for the L2 to join (32 x 1000 x 1000, whole call: 113 us past it, 76 through it).
template <int DP, bool LINES>
__global__ void __launch_bounds__(256) dense_scores_kernel(DenseScoreArgs a) {
  constexpr int KS = DP / 16, REC = dense_rec<DP, false>(), NF = REC / 1024, CPW = (NF + 3) / 4;
  constexpr int NS = 3;  // 48 KiB at head_dim 128: three blocks per compute unit
  __shared__ __attribute__((aligned(16))) uint8_t ring[NS * REC];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const uint32_t bid = blockIdx.x / static_cast<uint32_t>(a.nbh);
  const int bhi = static_cast<int>(blockIdx.x - bid * a.nbh);
  const int rb = static_cast<int>(bid % static_cast<uint32_t>(a.nblk)), split = static_cast<int>(bid / static_cast<uint32_t>(a.nblk));
  const uint32_t bh = static_cast<uint32_t>(a.bh0 + bhi);
  const int hkv = static_cast<int>(bh % static_cast<uint32_t>(a.Hkv));
  const int64_t b = bh / static_cast<uint32_t>(a.Hkv);
  const int tb = split * a.cpt, te = min(a.ntile, tb + a.cpt);
  if (tb >= te) return;
  const int task = rb * 4 + wave;  // (head of the group, row chunk)
  const bool live = task < a.G * a.rchunks;
  const int gi = live ? task / a.rchunks : 0, r0 = live ? (task - gi * a.rchunks) * 32 : 0;
  const int hq = hkv * a.G + gi, rows = min(32, a.Sq - r0);
  const int64_t row0 = (b * a.Hq + hq) * a.Sq + r0;
  half8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d0 = 16 * ks + 8 * h;
    const bool real = n < rows && d0 < a.d;
    const half8 v = *reinterpret_cast<const half8*>(a.q_rot + (row0 + (n < rows ? n : 0)) * a.d + (real ? d0 : 0));
    qf[ks] = real ? v : half8{};
  }
  // rows past the head's end are dropped by the store's range check
  const rsrc_t ro = make_rsrc(a.out + row0 * a.Sk, live ? static_cast<uint32_t>(rows) * a.Sk * 4 : 0);
  const float* tfac = a.tfac + static_cast<int64_t>(bhi) * a.ntile;
  const float* kfac = a.kfac + static_cast<int64_t>(bhi) * a.ntile * kKeyFac;
  float fv = 0.f;
  auto factors = [&](int t) __attribute__((always_inline)) {  // of tiles t .. t + 63
    fv = tfac[min(t + lane, te - 1)];
    wait_vm0_visible();
  };
  uint64_t src = reinterpret_cast<uint64_t>(a.tiles) + (static_cast<uint64_t>(bhi) * a.ntile + tb) * REC;
  int left = te - tb;
  const uint32_t ring_lds = lds_offset(ring);
  uint32_t dst = ring_lds;
  auto issue = [&]() __attribute__((always_inline)) {
    const i32x4 r{static_cast<int>(static_cast<uint32_t>(src)), static_cast<int>(static_cast<uint32_t>(src >> 32) & 0xffffu),
                  REC, 0x00020000};
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
      const int f = NF % 4 == 0 ? wave + 4 * i : min(wave + 4 * i, NF - 1);
      dma16_cached(r, dst + f * 1024, f * 1024 + lane * 16);
    }
    if (--left > 0) src += REC;
    dst = dst + REC == ring_lds + NS * REC ? ring_lds : dst + REC;
  };
  factors(tb);  // and waits for q
#pragma unroll
  for (int i = 0; i < NS - 1; ++i) issue();
  const uint8_t* rec = ring + lane * 16;
  for (int t = tb; t < te; ++t) {
    if (t != tb && ((t - tb) & 63) == 0) factors(t);
    // tile t's copies have landed: after them come NS - 2 records and, once the ring has gone round,
    // the 16 stores of each of the last NS - 1 tiles, which need not be waited for
    if (t - tb >= NS - 1) wait_vm<(NS - 2) * CPW + 16 * (NS - 1)>();
    else wait_vm<(NS - 2) * CPW>();
    wait_lds();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue();
    float16v s = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = mfma32x32x16(qf[ks], *reinterpret_cast<const half8*>(rec + ks * 1024), s);
      s = mfma32x32x16(qf[ks], *reinterpret_cast<const half8*>(rec + (KS + ks) * 1024), s);
    }
    float f = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, fv), (t - tb) & 63));
    if (__builtin_expect(f == 0.f, 0)) {  // a mixed tile: hi and lo apart, under this lane's key's factors
      asm volatile("; mixed tile" ::: "memory");  // fragments read anew: none is kept for this branch
      float16v sl = zero16();
      s = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        s = mfma32x32x16(qf[ks], *reinterpret_cast<const half8*>(rec + ks * 1024), s);
        sl = mfma32x32x16(qf[ks], *reinterpret_cast<const half8*>(rec + (KS + ks) * 1024), sl);
      }
      const float* kf = kfac + static_cast<int64_t>(t) * kKeyFac + 2 * n;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = fmaf(sl[i], kf[1], s[i] * kf[0]);
      f = 1.f;
    }
    const int key = t * kDenseKeys + n;
    // the range check covers the lane offset: it carries the row, and keys past Sk start out of range
    // (Sk < 2^24: neither wraps)
    const uint32_t at = key < a.Sk ? static_cast<uint32_t>(4 * h * a.Sk + key) * 4 : kOutOfRange;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, s[i] * f), ro,
                                            at + static_cast<uint32_t>((8 * (i >> 2) + (i & 3)) * a.Sk) * 4, 0,
                                            LINES ? kStream : 0);
    rec = rec + REC == ring + NS * REC + lane * 16 ? ring + lane * 16 : rec + REC;
  }
  wait_vm<0>();  // no copy outlives the block
}

// ---------------------------------------------------------------- host
struct DensePlan {
  int NW = 0, QT = 0, nqb = 0, ntile = 0, nsplit = 1, cpt = 0;
  int res = 1;  // blocks that share a compute unit
  int64_t group_bytes = 0;  // workspace of one (batch, kv head)
};

static int device_cus() {
  static int cache[16] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) dev = 0;
  if (cache[dev] == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
    cache[dev] = cus;
  }
  return cache[dev];
}

// Blocks that fit a compute unit together (LDS, and 256 VGPRs a wave up to head_dim 128)
constexpr int dense_resident(int DP, int NW, bool masked) {
  if (NW == 8) return 1;
  return masked ? (DP <= 64 ? 2 : 1) : (DP <= 64 ? 3 : DP <= 128 ? 2 : 1);
}
// Head dims with an 8-wave form
constexpr bool dense_wide(int DP) { return DP == 96 || DP == 128; }
// Block size and key splits for the smallest estimated time.  Unit: the time a compute unit takes for
// one tile of 256 columns (two waves per SIMD; a lone 4-wave block takes kLone of it, two of them
// kNarrow, kUnfilled where they leave some units to one).  A block adds
// kBlock (query fragments, first copies, output rotation), a split its partial sums through memory
// and the merge launch.
constexpr double kLone = 0.7, kBlock = 4.0, kMergeLaunch = 4.0, kPart = 0.04, kNarrow = 1.02, kUnfilled = 0.95;

static DensePlan dense_plan(int64_t groups, int G, int Sq, int Sk, int d, bool causal, bool masked, int cus) {
  const int DP = pad_dim(d);
  DensePlan best;
  double best_t = 0;
  const int ntile = (Sk + kDenseKeys - 1) / kDenseKeys;
  for (int NW = 8; NW >= 4; NW -= 4) {
    if (NW == 8 && !dense_wide(DP)) continue;
    DensePlan p;
    p.ntile = ntile;
    p.NW = NW;
    p.QT = 32 * NW / G;
    p.nqb = (Sq + p.QT - 1) / p.QT;
    auto tiles = [&](int q) {
      int kend = Sk;
      if (causal) kend = std::min(Sk, std::min(q * p.QT + p.QT - 1, Sq - 1) + (Sk - Sq) + 1);
      return (kend + kDenseKeys - 1) / kDenseKeys;
    };
    const int longest = tiles(p.nqb - 1);
    const int resident = dense_resident(DP, NW, masked);  // blocks per compute unit
    constexpr int kSample = 16;                                      // query blocks looked at
    const int ns_q = std::min(p.nqb, kSample);
    for (int ns = 1; ns <= 32; ns = ns < 4 ? ns + 1 : ns * 3 / 2) {
      const int cpt = (longest + ns - 1) / ns;
      if (ns > 1 && cpt < 4) break;
      double mean = 0, pieces = 0;
      for (int i = 0; i < ns_q; ++i) {
        const int t = tiles(static_cast<int>((2LL * i + 1) * p.nqb / (2 * ns_q)));
        mean += t;
        pieces += (t + cpt - 1) / cpt;
      }
      const double scale = static_cast<double>(groups) * p.nqb / ns_q;
      const double work = mean * scale, blocks = pieces * scale;
      const double per_cu = std::min<double>(resident, std::ceil(blocks / cus));
      // time of one tile of one block: `per_cu` blocks of NW waves share the compute unit
      const double tile = NW == 8 ? 1.0 : per_cu > 1 ? 0.5 * per_cu * (blocks < cus * per_cu ? kUnfilled : kNarrow) : kLone;
      const double slots = cus * per_cu;
      const double even = (work + kBlock * blocks) / slots * tile;
      const double rounds = std::ceil(blocks / slots - 0.02);
      // at least the longest block; whole rounds where all blocks are alike
      const bool alike = ns > 1 || !causal;
      double t = std::max({even, (cpt + kBlock) * tile, alike ? rounds * (cpt + kBlock) * tile : 0.0});
      if (ns > 1) t += kMergeLaunch * 128 / DP + kPart * blocks * NW / 8;
      if (best.NW == 0 || t < best_t) {
        best_t = t;
        best = p;
        best.cpt = cpt;
        best.res = static_cast<int>(per_cu);
        best.nsplit = (longest + cpt - 1) / cpt;
      }
    }
  }
  const int64_t recs = static_cast<int64_t>(best.nqb) * best.nsplit * best.NW;
  best.group_bytes = (static_cast<int64_t>(ntile) * 4 + 15) / 16 * 16 +
                     static_cast<int64_t>(ntile) * (3 * DP * 64 + kKeyFac * 4) +
                     (best.nsplit > 1 ? recs * (DP * 32 + 64) * 4 : 0);
  return best;
}

// tq_attn.hip
bool weights_are_f16(int B, int Hq, int Hkv, int Sq, int Sk, int d, int bits, int val_bits, bool masked);

}  // namespace tq

using namespace tq;

// Workspace: whole (batch, kv head)s; calls with more of them than fit kDenseWorkspace run in
// several rounds over the same memory.
static constexpr int64_t kDenseWorkspace = int64_t(1) << 30;
static constexpr int kDenseMaxGroup = 128;  // query heads per kv head that fit a block's columns

// the start of the workspace: S_eff's fragments and q_rot
static int64_t dense_q_bytes(int B, int Hq, int Sq, int d) {
  const int64_t DP = pad_dim(d);
  return 2 * DP * DP + (static_cast<int64_t>(B) * Hq * Sq * d * 2 + 255) / 256 * 256;
}

// workspace of one (batch, kv head)'s expanded keys and factors
static int64_t score_group_bytes(int Sk, int d) {
  const int64_t nt = (Sk + kDenseKeys - 1) / kDenseKeys;
  return nt * (2 * pad_dim(d) * 64 + kKeyFac * 4) + (nt * 4 + 15) / 16 * 16;
}

// Bytes per load that every packed row (d / 8 bytes per code bit) and plane base allows the expansion
static int row_width(int d, uintptr_t bases) {
  return d % 32 == 0 && bases % 4 == 0 ? 4 : d % 16 == 0 && bases % 2 == 0 ? 2 : 1;
}

// q_rot, and S_eff's fragments for the expansion
static void launch_rotate(const void* q, int dtype, int B, int Hq, int Sq, int d, int64_t sqb, int64_t sqh, int64_t sqs,
                          const uint16_t* key_pi_split, const uint16_t* key_s_eff_f16, uint16_t* q_rot,
                          uint16_t* seff_frag, int cus, hipStream_t s) {
  const int DP = pad_dim(d);
  RotArgs r{};
  r.q = q; r.n = static_cast<int64_t>(B) * Hq * Sq; r.sqb = sqb; r.sqh = sqh; r.sqs = sqs;
  r.Hq = Hq; r.Sq = Sq; r.d = d; r.pi = key_pi_split; r.seff = key_s_eff_f16;
  r.q_rot = q_rot; r.seff_frag = seff_frag;
  const int64_t es = dtype == TQ_F32 ? 4 : 2;
  r.vec = reinterpret_cast<uintptr_t>(q) % 16 == 0 && (sqb * es) % 16 == 0 && (sqh * es) % 16 == 0 &&
          (sqs * es) % 16 == 0;
  r.blocks = static_cast<int>(std::min<int64_t>((r.n + 255) / 256, 2LL * cus));
  const unsigned gx = r.blocks + 4;
#define TQ_ROT_CASE(DD)                                                                     \
  case DD: {                                                                                \
    const dim3 g(gx, (DD / 32 + rot_blocks<DD>() - 1) / rot_blocks<DD>());                  \
    if (dtype == TQ_F32) dense_rotate_kernel<DD, TQ_F32><<<g, 512, 0, s>>>(r);              \
    else if (dtype == TQ_F16) dense_rotate_kernel<DD, TQ_F16><<<g, 512, 0, s>>>(r);         \
    else dense_rotate_kernel<DD, TQ_BF16><<<g, 512, 0, s>>>(r);                             \
  } break;
  switch (DP) {
    TQ_ROT_CASE(32)
    TQ_ROT_CASE(64)
    TQ_ROT_CASE(96)
    TQ_ROT_CASE(128)
    TQ_ROT_CASE(160)
    TQ_ROT_CASE(192)
    TQ_ROT_CASE(224)
    TQ_ROT_CASE(256)
  }
#undef TQ_ROT_CASE
}

extern "C" {

int64_t tq_prefill_workspace_size(int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Sk, int32_t d,
                                  int32_t causal, int32_t masked) {
  if (!supported_dim(d) || B <= 0 || Hkv <= 0 || Hq <= 0 || Hq % Hkv || Sq <= 0 || Sk <= 0) return 0;
  const int G = Hq / Hkv;
  if (G > kDenseMaxGroup) return 0;
  const int64_t groups = static_cast<int64_t>(B) * Hkv;
  const DensePlan p = dense_plan(groups, G, Sq, Sk, d, causal != 0, masked != 0, device_cus());
  const int64_t fit = std::max<int64_t>(1, kDenseWorkspace / p.group_bytes);
  return dense_q_bytes(B, Hq, Sq, d) + std::min(groups, fit) * p.group_bytes;
}

int tq_prefill_attention(const void* q, int32_t dtype, int64_t sqb, int64_t sqh, int64_t sqs,
                         const uint16_t* key_pi_split, const uint16_t* key_s_eff_f16, const uint8_t* key_codes,
                         const uint8_t* key_signs, const uint16_t* key_rn, const uint16_t* key_vn,
                         const uint16_t* key_centroids_f16, int32_t bits, const uint8_t* val_codes,
                         const uint16_t* val_vn, const float* val_centroids, int32_t val_bits,
                         const uint16_t* val_pit_split, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Sk,
                         int64_t kv_stride, int32_t d, float coeff, float scale, int32_t causal, const void* mask,
                         int32_t mask_dtype, int64_t smb, int64_t smh, int64_t smq, int64_t smk, void* out,
                         int32_t out_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  const char* what = "tq_prefill_attention";
  if (!supported_dim(d)) {
    set_error("%s: head_dim %d not supported (multiples of 8 from 8 to 256)", what, (int)d);
    return TQ_EUNSUPPORTED;
  }
  TQ_REQUIRE(bits >= 2 && bits <= 4, "%s: key bits must be in [2, 4], got %d", what, (int)bits);
  TQ_REQUIRE(val_bits >= 1 && val_bits <= 4, "%s: value bits must be in [1, 4], got %d", what, (int)val_bits);
  TQ_REQUIRE(B >= 0 && Hq >= 0 && Hkv >= 1 && Sq >= 0 && Sk >= 1 && Hq % Hkv == 0, "%s: bad shape", what);
  const int64_t ldk = kv_stride > 0 ? kv_stride : Sk;
  TQ_REQUIRE(ldk >= Sk, "%s: kv_stride %lld < Sk %d", what, (long long)kv_stride, (int)Sk);
  TQ_REQUIRE(dtype == TQ_F32 || dtype == TQ_F16 || dtype == TQ_BF16, "%s: unknown dtype %d", what, (int)dtype);
  TQ_REQUIRE(out_dtype == TQ_F32 || out_dtype == TQ_F16 || out_dtype == TQ_BF16, "%s: unknown out dtype %d", what,
             (int)out_dtype);
  TQ_REQUIRE(!mask || mask_dtype == TQ_F32 || mask_dtype == TQ_F16 || mask_dtype == TQ_BF16,
             "%s: unknown mask dtype %d", what, (int)mask_dtype);
  TQ_REQUIRE(!causal || Sk >= Sq, "%s: causal needs Sk >= Sq", what);
  if (static_cast<int64_t>(B) * Hq * Sq == 0) return TQ_OK;
  const int G = Hq / Hkv;
  TQ_REQUIRE(G <= kDenseMaxGroup, "%s: group size %d exceeds %d", what, G, kDenseMaxGroup);
  TQ_REQUIRE(q && key_pi_split && key_s_eff_f16 && key_codes && key_signs && key_rn && key_vn && key_centroids_f16 &&
                 val_codes && val_vn && val_centroids && val_pit_split && out && workspace,
             "%s: null pointer", what);
  TQ_REQUIRE(((reinterpret_cast<uintptr_t>(key_pi_split) | reinterpret_cast<uintptr_t>(val_pit_split) |
               reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(workspace)) & 15) == 0,
             "%s: key_pi_split, val_pit_split, out and workspace must be 16-byte aligned", what);
  const int cus = device_cus();
  const int64_t groups = static_cast<int64_t>(B) * Hkv;
  const DensePlan p = dense_plan(groups, G, Sq, Sk, d, causal != 0, mask != nullptr, cus);
  const int64_t qbytes = dense_q_bytes(B, Hq, Sq, d);
  const int64_t per = std::min(groups, (workspace_bytes - qbytes) / p.group_bytes);
  TQ_REQUIRE(workspace_bytes >= qbytes && per >= 1, "%s: %lld workspace bytes, at least %lld needed", what,
             (long long)workspace_bytes, (long long)(qbytes + p.group_bytes));
  const int DP = pad_dim(d);
  const int64_t recs = static_cast<int64_t>(p.nqb) * p.nsplit * p.NW;
  TQ_REQUIRE(per * recs < (int64_t(1) << 31) && groups < (int64_t(1) << 31), "%s: too many blocks", what);
  hipStream_t s = as_stream(stream);

  uint16_t* seff_frag = static_cast<uint16_t*>(workspace);
  uint16_t* q_rot = seff_frag + static_cast<int64_t>(DP) * DP;
  launch_rotate(q, dtype, B, Hq, Sq, d, sqb, sqh, sqs, key_pi_split, key_s_eff_f16, q_rot, seff_frag, cus, s);
  // P as f16 (hi, lo) where the term-by-term path keeps it so (its tiled kernel, split over keys or
  // not); one f16 where the kernel it would run for this shape rounds it (the prefill kernel)
  const bool plo = !weights_are_f16(B, Hq, Hkv, Sq, Sk, d, bits, val_bits, mask != nullptr);
  const int width = row_width(d, reinterpret_cast<uintptr_t>(key_codes) | reinterpret_cast<uintptr_t>(key_signs) |
                                     reinterpret_cast<uintptr_t>(val_codes));
  uint8_t* tiles = static_cast<uint8_t*>(workspace) + qbytes;
  float* part_o = reinterpret_cast<float*>(tiles + per * p.ntile * (3 * DP * 64));
  float* part_ml = part_o + (p.nsplit > 1 ? per * recs * DP * 32 : 0);
  float* kfac = part_ml + (p.nsplit > 1 ? per * recs * 64 : 0);
  float* tfac = kfac + per * p.ntile * kKeyFac;
  for (int64_t g0 = 0; g0 < groups; g0 += per) {
    const int nbh = static_cast<int>(std::min(per, groups - g0));
    ExpandArgs e{};
    e.kcodes = key_codes; e.ksigns = key_signs; e.vcodes = val_codes;
    e.krn = key_rn; e.kvn = key_vn; e.vvn = val_vn; e.kcent = key_centroids_f16; e.seff_frag = seff_frag;
    e.vcent = val_centroids;
    e.Sk = Sk; e.d = d; e.kb = bits - 1; e.vb = val_bits; e.ntile = p.ntile;
    e.ldk = ldk; e.bh0 = g0; e.total = static_cast<int64_t>(nbh) * p.ntile;
    e.coeff = coeff; e.tiles = tiles; e.tfac = tfac; e.kfac = kfac;
    DenseArgs a{};
    a.q_rot = q_rot; a.tiles = tiles; a.tfac = tfac; a.kfac = kfac; a.vpit = val_pit_split;
    a.Hq = Hq; a.Hkv = Hkv; a.Sq = Sq; a.Sk = Sk; a.d = d; a.G = G; a.QT = p.QT; a.nqb = p.nqb; a.nbh = nbh;
    a.ntile = p.ntile; a.bh0 = g0; a.scale = scale; a.causal = causal;
    a.mask = mask; a.mask_dtype = mask_dtype; a.smb = smb; a.smh = smh; a.smq = smq; a.smk = smk;
    a.out = out; a.out_dtype = out_dtype;
    a.part_o = part_o; a.part_ml = part_ml; a.nsplit = p.nsplit; a.cpt = p.cpt;
    const unsigned egrid = static_cast<unsigned>(std::min<int64_t>(e.total, 8LL * cus));
    const unsigned grid = static_cast<unsigned>(nbh) * p.nqb * p.nsplit;
    const unsigned mgrid = static_cast<unsigned>(nbh) * p.nqb * p.NW;
#define TQ_DENSE_R(DD, NN, MM, PL)                                                             \
  if (p.res > 1) dense_attn_kernel<DD, NN, MM, PL, dense_resident(DD, NN, MM)><<<grid, 64 * NN, 0, s>>>(a); \
  else dense_attn_kernel<DD, NN, MM, PL, 1><<<grid, 64 * NN, 0, s>>>(a);
#define TQ_DENSE_P(DD, NN, PL)                                                                 \
  if (mask) { TQ_DENSE_R(DD, NN, true, PL) } else { TQ_DENSE_R(DD, NN, false, PL) }
#define TQ_DENSE(DD, NN)                                                                       \
  if constexpr (DD == 64 || DD == 128) {                                                       \
    if (plo) { TQ_DENSE_P(DD, NN, true) } else { TQ_DENSE_P(DD, NN, false) }                   \
  } else { TQ_DENSE_P(DD, NN, true) }
#define TQ_DENSE_CASE(DD)                                                                      \
  case DD:                                                                                     \
    if (width == 4) dense_expand_kernel<DD, 4, true><<<egrid, 2 * DD, 0, s>>>(e);              \
    else if (width == 2) dense_expand_kernel<DD, 2, true><<<egrid, 2 * DD, 0, s>>>(e);         \
    else dense_expand_kernel<DD, 1, true><<<egrid, 2 * DD, 0, s>>>(e);                         \
    if (p.NW == 8) { if constexpr (dense_wide(DD)) { TQ_DENSE(DD, 8) } }                            \
    else { TQ_DENSE(DD, 4) }                                                                   \
    if (p.nsplit > 1) dense_merge_kernel<DD><<<mgrid, 2 * DD, 0, s>>>(a, p.NW);                \
    break;
    switch (DP) {
      TQ_DENSE_CASE(32)
      TQ_DENSE_CASE(64)
      TQ_DENSE_CASE(96)
      TQ_DENSE_CASE(128)
      TQ_DENSE_CASE(160)
      TQ_DENSE_CASE(192)
      TQ_DENSE_CASE(224)
      TQ_DENSE_CASE(256)
    }
#undef TQ_DENSE_CASE
#undef TQ_DENSE
#undef TQ_DENSE_P
#undef TQ_DENSE_R
    const int st = launch_status(what);
    if (st != TQ_OK) return st;
  }
  return TQ_OK;
}

int64_t tq_prefill_scores_workspace_size(int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq, int32_t Sk, int32_t d) {
  if (!supported_dim(d) || B <= 0 || Hkv <= 0 || Hq <= 0 || Hq % Hkv || Sq <= 0 || Sk <= 0 || Sk >= (1 << 24)) return 0;
  const int64_t groups = static_cast<int64_t>(B) * Hkv, group = score_group_bytes(Sk, d);
  return dense_q_bytes(B, Hq, Sq, d) + std::min(groups, std::max<int64_t>(1, kDenseWorkspace / group)) * group;
}

int tq_prefill_scores(const void* q, int32_t dtype, int64_t sqb, int64_t sqh, int64_t sqs,
                      const uint16_t* key_pi_split, const uint16_t* key_s_eff_f16, const uint8_t* key_codes,
                      const uint8_t* key_signs, const uint16_t* key_rn, const uint16_t* key_vn,
                      const uint16_t* key_centroids_f16, int32_t bits, int32_t B, int32_t Hq, int32_t Hkv, int32_t Sq,
                      int32_t Sk, int64_t kv_stride, int32_t d, float coeff, float* out, void* workspace,
                      int64_t workspace_bytes, void* stream) {
  const char* what = "tq_prefill_scores";
  if (!supported_dim(d)) {
    set_error("%s: head_dim %d not supported (multiples of 8 from 8 to 256)", what, (int)d);
    return TQ_EUNSUPPORTED;
  }
  TQ_REQUIRE(bits >= 2 && bits <= 4, "%s: key bits must be in [2, 4], got %d", what, (int)bits);
  TQ_REQUIRE(B >= 0 && Hq >= 0 && Hkv >= 1 && Sq >= 0 && Sk >= 0 && Hq % Hkv == 0, "%s: bad shape", what);
  const int64_t ldk = kv_stride > 0 ? kv_stride : Sk;
  TQ_REQUIRE(ldk >= Sk, "%s: kv_stride %lld < Sk %d", what, (long long)kv_stride, (int)Sk);
  TQ_REQUIRE(dtype == TQ_F32 || dtype == TQ_F16 || dtype == TQ_BF16, "%s: unknown dtype %d", what, (int)dtype);
  if (static_cast<int64_t>(B) * Hq * Sq * Sk == 0) return TQ_OK;
  TQ_REQUIRE(Sk < (1 << 24), "%s: %d keys, fewer than 2^24 wanted", what, (int)Sk);
  TQ_REQUIRE(q && key_pi_split && key_s_eff_f16 && key_codes && key_signs && key_rn && key_vn && key_centroids_f16 &&
                 out && workspace,
             "%s: null pointer", what);
  TQ_REQUIRE(((reinterpret_cast<uintptr_t>(key_pi_split) | reinterpret_cast<uintptr_t>(workspace)) & 15) == 0,
             "%s: key_pi_split and workspace must be 16-byte aligned", what);
  const int cus = device_cus(), G = Hq / Hkv, DP = pad_dim(d);
  const int64_t groups = static_cast<int64_t>(B) * Hkv, group = score_group_bytes(Sk, d);
  const int64_t qbytes = dense_q_bytes(B, Hq, Sq, d);
  const int64_t per = std::min(groups, (workspace_bytes - qbytes) / group);
  TQ_REQUIRE(workspace_bytes >= qbytes && per >= 1, "%s: %lld workspace bytes, at least %lld needed", what,
             (long long)workspace_bytes, (long long)(qbytes + group));
  hipStream_t s = as_stream(stream);
  uint16_t* seff_frag = static_cast<uint16_t*>(workspace);
  uint16_t* q_rot = seff_frag + static_cast<int64_t>(DP) * DP;
  launch_rotate(q, dtype, B, Hq, Sq, d, sqb, sqh, sqs, key_pi_split, key_s_eff_f16, q_rot, seff_frag, cus, s);
  const int width = row_width(d, reinterpret_cast<uintptr_t>(key_codes) | reinterpret_cast<uintptr_t>(key_signs));
  const bool lines = Sk % 32 == 0 && reinterpret_cast<uintptr_t>(out) % 128 == 0;
  uint8_t* tiles = static_cast<uint8_t*>(workspace) + qbytes;
  DenseScoreArgs a{};
  a.q_rot = q_rot; a.tiles = tiles;
  a.Hq = Hq; a.Hkv = Hkv; a.Sq = Sq; a.Sk = Sk; a.d = d; a.G = G;
  a.rchunks = (Sq + 31) / 32;
  a.ntile = (Sk + kDenseKeys - 1) / kDenseKeys;
  a.out = out;
  TQ_REQUIRE(static_cast<int64_t>(G) * a.rchunks < (int64_t(1) << 31) && groups < (int64_t(1) << 31), "%s: too many rows",
             what);
  a.nblk = (G * a.rchunks + 3) / 4;
  float* kfac = reinterpret_cast<float*>(tiles + per * a.ntile * static_cast<int64_t>(2 * DP * 64));
  float* tfac = kfac + per * a.ntile * kKeyFac;
  a.kfac = kfac; a.tfac = tfac;
  // about eight blocks per compute unit, of at least four tiles
  const int64_t blocks = std::min(per, groups) * a.nblk;
  a.cpt = static_cast<int>(std::min<int64_t>(a.ntile, std::max<int64_t>(4, blocks * a.ntile / (8LL * cus))));
  const int nsplit = (a.ntile + a.cpt - 1) / a.cpt;
  TQ_REQUIRE(blocks * nsplit < (int64_t(1) << 31), "%s: too many blocks", what);
  for (int64_t g0 = 0; g0 < groups; g0 += per) {
    a.nbh = static_cast<int>(std::min(per, groups - g0));
    a.bh0 = g0;
    ExpandArgs e{};
    e.kcodes = key_codes; e.ksigns = key_signs; e.krn = key_rn; e.kvn = key_vn; e.kcent = key_centroids_f16;
    e.seff_frag = seff_frag; e.Sk = Sk; e.d = d; e.kb = bits - 1; e.vb = 1; e.ntile = a.ntile;
    e.ldk = ldk; e.bh0 = g0; e.total = static_cast<int64_t>(a.nbh) * a.ntile;
    e.coeff = coeff; e.tiles = tiles; e.tfac = tfac; e.kfac = kfac;
    const unsigned egrid = static_cast<unsigned>(std::min<int64_t>(e.total, 8LL * cus));
    const unsigned grid = static_cast<unsigned>(a.nbh) * a.nblk * nsplit;
#define TQ_SCORES_CASE(DD)                                                                     \
  case DD:                                                                                     \
    if (width == 4) dense_expand_kernel<DD, 4, false><<<egrid, 2 * DD, 0, s>>>(e);             \
    else if (width == 2) dense_expand_kernel<DD, 2, false><<<egrid, 2 * DD, 0, s>>>(e);        \
    else dense_expand_kernel<DD, 1, false><<<egrid, 2 * DD, 0, s>>>(e);                        \
    if (lines) dense_scores_kernel<DD, true><<<grid, 256, 0, s>>>(a);                          \
    else dense_scores_kernel<DD, false><<<grid, 256, 0, s>>>(a);                               \
    break;
    switch (DP) {
      TQ_SCORES_CASE(32)
      TQ_SCORES_CASE(64)
      TQ_SCORES_CASE(96)
      TQ_SCORES_CASE(128)
      TQ_SCORES_CASE(160)
      TQ_SCORES_CASE(192)
      TQ_SCORES_CASE(224)
      TQ_SCORES_CASE(256)
    }
#undef TQ_SCORES_CASE
    const int st = launch_status(what);
    if (st != TQ_OK) return st;
  }
  return TQ_OK;
}

}  // extern "C"
