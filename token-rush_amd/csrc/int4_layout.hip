// Conversions between the engine's int4 packing, the quad layout (int4_layout.h) and dense weights:
// tr_pack_int4 / tr_unpack_int4 (the role of marlin.pack / marlin.unpack, tokenrush/marlin.py:73-118),
// tr_dequant_int4 (tokenrush/quant.py:47-53) and tr_dequant_packed (the same from the quad layout).
//
// All are bound by HBM. One wave converts one quad (16 rows x 512 k): its four 1 KiB code blocks move as
// one 16-byte access per lane, and a lane holds four words of one row (j = 0..3 at k = 32 j + 8 (lane / 16)).
// The engine's row order wants the lanes' words transposed: lane row o (lanes 16 o ..) takes the words
// j = o of all four lane rows, 16 consecutive bytes of its row. Four permlane swaps do that 4 x 4
// transpose in registers. One thread per output word, as before, spent its time on 64-bit divisions,
// 4-byte accesses and (dequant) one byte of codes per thread. 34816 x 5120, bf16 parameters, us:
// pack 93 -> 42, unpack 74 -> 33, dense from engine codes 200 -> 121, dense from the quad
// layout (unpack + dequant before) 260 -> 85.
#include "int4_layout.h"

namespace tr {

// Engine tensors may start at any byte (a view of a byte buffer): unaligned 16-byte accesses.
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u32x2_u __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32x4_w __attribute__((ext_vector_type(4), aligned(4)));

// Engine row of packed row i (0..15) of strip `strip`: identity, or for the gate/up pair layout
// (F = N / 2 > 0) gate row 8 strip + i for i < 8 and up row F + 8 strip + i - 8 otherwise.
__device__ __forceinline__ size_t src_row(int strip, int i, int F) {
  return F > 0 ? (i < 8 ? (size_t)8 * strip + i : (size_t)F + 8 * (size_t)strip + (i - 8)) : (size_t)16 * strip + i;
}

// r[j] of lane row o (lanes 16 o .. 16 o + 15) <-> r[o] of lane row j: its own inverse.
__device__ __forceinline__ void transpose_rows(uint32_t (&r)[4]) {
  const auto a = __builtin_amdgcn_permlane32_swap(r[0], r[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(r[1], r[3], false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  r[0] = c[0];
  r[1] = c[1];
  r[2] = d[0];
  r[3] = d[1];
}

// Eight codes in engine order (byte p = codes 2p | 2p + 1 << 4) <-> the quad layout's word (code 2p in
// nibble p, code 2p + 1 in nibble p + 4).
__device__ __forceinline__ uint32_t gather_nibbles(uint32_t x) {  // low nibble of each byte -> low 16 bits
  x &= 0x0F0F0F0Fu;
  x = (x | (x >> 4)) & 0x00FF00FFu;
  return (x | (x >> 8)) & 0xFFFFu;
}
__device__ __forceinline__ uint32_t spread_nibbles(uint32_t x) {  // its inverse
  x = (x | (x << 8)) & 0x00FF00FFu;
  return (x | (x << 4)) & 0x0F0F0F0Fu;
}
__device__ __forceinline__ uint32_t to_quad_word(uint32_t e) { return gather_nibbles(e) | (gather_nibbles(e >> 4) << 16); }
__device__ __forceinline__ uint32_t to_engine_word(uint32_t w) {
  return spread_nibbles(w & 0xFFFFu) | (spread_nibbles(w >> 16) << 4);
}

// The wave's quads: quad index, its strip and first group.
struct QuadWalk {
  uint32_t quad, total, step;
  int nq;
  __device__ __forceinline__ QuadWalk(int N, int nq_) : nq(nq_) {
    quad = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    step = gridDim.x * (blockDim.x >> 6);
    total = (uint32_t)(N / 16) * nq_;
  }
};

__global__ __launch_bounds__(256) void pack_kernel(const uint8_t* __restrict__ q, const uint16_t* __restrict__ scale,
                                                   const uint16_t* __restrict__ mn, uint8_t* __restrict__ packed, int N,
                                                   int K, int F) {
  const int G = K / kGroup, lane = threadIdx.x & 63, o = lane >> 4;
  for (QuadWalk w(N, padded_groups(K) / kQuad); w.quad < w.total; w.quad += w.step) {
    const int strip = w.quad / w.nq, g0 = (int)(w.quad - (uint32_t)strip * w.nq) * kQuad;
    uint8_t* dst = packed + (size_t)w.quad * kQuadBytes;
    const uint8_t* src = q + src_row(strip, lane & 15, F) * (K / 2) + 16 * o;
    u32x4 v[kQuad];
#pragma unroll
    for (int t = 0; t < kQuad; ++t)
      v[t] = g0 + t < G ? (u32x4)__builtin_nontemporal_load((const u32x4_u*)(src + (size_t)(g0 + t) * 64)) : u32x4{0, 0, 0, 0};
    // parameters: lane l holds row l / 4, group l % 4
    const int pg = g0 + (lane & 3);
    const size_t pi = src_row(strip, lane >> 2, F) * G + pg;
    const uint32_t sm = pg < G ? (uint32_t)scale[pi] | ((uint32_t)mn[pi] << 16) : 0u;
#pragma unroll
    for (int t = 0; t < kQuad; ++t) {
      uint32_t r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = to_quad_word(v[t][i]);
      transpose_rows(r);
      *(u32x4_w*)(dst + t * kCodeBytes + 16 * lane) = u32x4_w{r[0], r[1], r[2], r[3]};
    }
    *(uint32_t*)(dst + kSmOff + 4 * lane) = sm;
  }
}

__global__ __launch_bounds__(256) void unpack_kernel(const uint8_t* __restrict__ packed, uint8_t* __restrict__ q,
                                                     uint16_t* __restrict__ scale, uint16_t* __restrict__ mn, int N,
                                                     int K, int F) {
  const int G = K / kGroup, lane = threadIdx.x & 63, o = lane >> 4;
  for (QuadWalk w(N, padded_groups(K) / kQuad); w.quad < w.total; w.quad += w.step) {
    const int strip = w.quad / w.nq, g0 = (int)(w.quad - (uint32_t)strip * w.nq) * kQuad;
    const uint8_t* src = packed + (size_t)w.quad * kQuadBytes;
    u32x4 v[kQuad];
#pragma unroll
    for (int t = 0; t < kQuad; ++t) v[t] = __builtin_nontemporal_load((const u32x4_w*)(src + t * kCodeBytes + 16 * lane));
    const uint32_t sm = *(const uint32_t*)(src + kSmOff + 4 * lane);
    uint8_t* dst = q + src_row(strip, lane & 15, F) * (K / 2) + 16 * o;
#pragma unroll
    for (int t = 0; t < kQuad; ++t) {
      uint32_t r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = to_engine_word(v[t][i]);
      transpose_rows(r);
      if (g0 + t < G) *(u32x4_u*)(dst + (size_t)(g0 + t) * 64) = u32x4_u{r[0], r[1], r[2], r[3]};
    }
    const int pg = g0 + (lane & 3);
    if (pg < G) {
      const size_t pi = src_row(strip, lane >> 2, F) * G + pg;
      scale[pi] = (uint16_t)(sm & 0xFFFF);
      mn[pi] = (uint16_t)(sm >> 16);
    }
  }
}

// round(round(c * s) + m) of two codes, as a pair of 16-bit values (tokenrush/quant.py:47-53): bf16
// parameters round in bf16, fp16 ones (the benchmark format) in fp16. AS_BF16 rounds fp16 results
// once more to bf16 (what a .to(bfloat16) of the dense weight does).
template <bool F16S, bool AS_BF16>
__device__ __forceinline__ uint32_t dequant2(float c0, float c1, float s, float m) {
  if (F16S) {
    const _Float16 a = (_Float16)((float)(_Float16)(c0 * s) + m), b = (_Float16)((float)(_Float16)(c1 * s) + m);
    if (AS_BF16) return f32x2_to_bf16x2_bits((float)a, (float)b);
    return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
  }
  const uint32_t t = f32x2_to_bf16x2_bits(c0 * s, c1 * s);
  return f32x2_to_bf16x2_bits(__uint_as_float(t << 16) + m, __uint_as_float(t & 0xFFFF0000u) + m);
}

// The quad layout -> dense [N, K]. Lanes l and l ^ 8 (rows i and i + 8) trade words j and j + 1 first, so
// that each store covers whole 128-byte lines: 64 consecutive values of eight rows. Storing a lane's own
// words (16 rows x 64 bytes) took 106 us where this takes 85 us (450 MB, 5.3 TB/s).
template <bool F16S, bool AS_BF16>
__global__ __launch_bounds__(256) void dequant_packed_kernel(const uint8_t* __restrict__ packed,
                                                             uint16_t* __restrict__ out, int N, int K, int F) {
  const int G = K / kGroup, lane = threadIdx.x & 63, o = lane >> 4, i = lane & 15;
  const bool up = i >= 8;
  for (QuadWalk w(N, padded_groups(K) / kQuad); w.quad < w.total; w.quad += w.step) {
    const int strip = w.quad / w.nq, g0 = (int)(w.quad - (uint32_t)strip * w.nq) * kQuad;
    const uint8_t* src = packed + (size_t)w.quad * kQuadBytes;
    const u32x4 smA = *(const u32x4_w*)(src + kSmOff + 16 * (i & 7)), smB = *(const u32x4_w*)(src + kSmOff + 16 * (i | 8));
    u32x4 v[kQuad];
#pragma unroll
    for (int t = 0; t < kQuad; ++t) v[t] = __builtin_nontemporal_load((const u32x4_w*)(src + t * kCodeBytes + 16 * lane));
    const size_t col = (size_t)g0 * kGroup + 8 * o + (up ? 32 : 0);
    uint16_t* dA = out + src_row(strip, i & 7, F) * K + col;
    uint16_t* dB = out + src_row(strip, i | 8, F) * K + col;
#pragma unroll
    for (int t = 0; t < kQuad; ++t) {
      if (g0 + t >= G) break;
      const float sA = sm_scale<F16S>(smA[t]), mA = sm_min<F16S>(smA[t]);
      const float sB = sm_scale<F16S>(smB[t]), mB = sm_min<F16S>(smB[t]);
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const uint32_t give = up ? v[t][j] : v[t][j + 1];
        const uint32_t got = __builtin_amdgcn_update_dpp(0, give, 0x128 /* row_ror:8 */, 0xF, 0xF, false);
        const uint32_t cA = up ? got : v[t][j], cB = up ? v[t][j + 1] : got;
        u32x4_w a, b;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint32_t x = cA >> (4 * p), y = cB >> (4 * p);
          a[p] = dequant2<F16S, AS_BF16>((float)(x & 0xF), (float)((x >> 16) & 0xF), sA, mA);
          b[p] = dequant2<F16S, AS_BF16>((float)(y & 0xF), (float)((y >> 16) & 0xF), sB, mB);
        }
        *(u32x4_w*)(dA + t * kGroup + 32 * j) = a;
        *(u32x4_w*)(dB + t * kGroup + 32 * j) = b;
      }
    }
  }
}

// The engine packing -> dense [N, K]: a wave takes a row, a lane 16 codes (8 bytes, one group) at a time.
template <bool F16S>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ q, const uint16_t* __restrict__ scale,
                                                      const uint16_t* __restrict__ mn, uint16_t* __restrict__ out,
                                                      int N, int K) {
  const int G = K / kGroup, segs = K / 16;
  for (int n = blockIdx.x * 4 + (threadIdx.x >> 6); n < N; n += gridDim.x * 4) {
#pragma unroll 4
    for (int i = threadIdx.x & 63; i < segs; i += 64) {
      const size_t gi = (size_t)n * G + (i >> 3);
      const float s = F16S ? f16_bits_to_f32(scale[gi]) : bf16_bits_to_f32(scale[gi]);
      const float m = F16S ? f16_bits_to_f32(mn[gi]) : bf16_bits_to_f32(mn[gi]);
      const u32x2 v = __builtin_nontemporal_load((const u32x2_u*)(q + (size_t)n * (K / 2) + 8 * (size_t)i));
      u32x4_w* dst = (u32x4_w*)(out + (size_t)n * K + 16 * (size_t)i);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4_w d;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint32_t c = v[h] >> (8 * p);
          d[p] = dequant2<F16S, false>((float)(c & 0xF), (float)((c >> 4) & 0xF), s, m);
        }
        dst[h] = d;
      }
    }
  }
}

}  // namespace tr

using namespace tr;

namespace {

// One wave per quad, four to a workgroup; the kernels stride over the rest beyond this many workgroups.
int quad_grid(int N, int K) {
  const size_t wgs = ((size_t)N / 16 * (padded_groups(K) / kQuad) + 3) / 4;
  return (int)(wgs < 65536 ? wgs : 65536);
}

int pack_impl(const void* qweight, const void* scale, const void* mn, void* packed, int N, int K, int F, void* stream) {
  if (!qweight || !scale || !mn || !packed) return TR_ERR_ARG;
  if (!shape_ok(N, K) || (F && N % 32)) return TR_ERR_SHAPE;
  hipLaunchKernelGGL(pack_kernel, dim3(quad_grid(N, K)), dim3(256), 0, (hipStream_t)stream, (const uint8_t*)qweight,
                     (const uint16_t*)scale, (const uint16_t*)mn, (uint8_t*)packed, N, K, F);
  return hipGetLastError() == hipSuccess ? TR_OK : TR_ERR_LAUNCH;
}

int unpack_impl(const void* packed, void* qweight, void* scale, void* mn, int N, int K, int F, void* stream) {
  if (!qweight || !packed || !scale || !mn) return TR_ERR_ARG;
  if (!shape_ok(N, K) || (F && N % 32)) return TR_ERR_SHAPE;
  hipLaunchKernelGGL(unpack_kernel, dim3(quad_grid(N, K)), dim3(256), 0, (hipStream_t)stream, (const uint8_t*)packed,
                     (uint8_t*)qweight, (uint16_t*)scale, (uint16_t*)mn, N, K, F);
  return hipGetLastError() == hipSuccess ? TR_OK : TR_ERR_LAUNCH;
}

}  // namespace

extern "C" {

size_t tr_packed_bytes(int N, int K) { return shape_ok(N, K) ? packed_bytes(N, K) : 0; }

int tr_pack_int4(const void* qweight, const void* scale, const void* mn, void* packed, int N, int K, void* stream) {
  return pack_impl(qweight, scale, mn, packed, N, K, 0, stream);
}

int tr_unpack_int4(const void* packed, void* qweight, void* scale, void* mn, int N, int K, void* stream) {
  return unpack_impl(packed, qweight, scale, mn, N, K, 0, stream);
}

int tr_pack_int4_pairs(const void* qweight, const void* scale, const void* mn, void* packed, int N, int K,
                       void* stream) {
  return pack_impl(qweight, scale, mn, packed, N, K, N / 2, stream);
}

int tr_unpack_int4_pairs(const void* packed, void* qweight, void* scale, void* mn, int N, int K, void* stream) {
  return unpack_impl(packed, qweight, scale, mn, N, K, N / 2, stream);
}

int tr_dequant_int4(const void* qweight, const void* scale, const void* mn, void* out, int N, int K, int group,
                    int scale_dtype, void* stream) {
  if (!qweight || !scale || !mn || !out) return TR_ERR_ARG;
  if (group != kGroup) return TR_ERR_CONFIG;
  if (N <= 0 || K <= 0 || K % kGroup) return TR_ERR_SHAPE;
  const int rows4 = (N + 3) / 4;
  const dim3 grid(rows4 < 65536 ? rows4 : 65536);
  if (scale_dtype == 1)
    hipLaunchKernelGGL(dequant_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, (const uint8_t*)qweight,
                       (const uint16_t*)scale, (const uint16_t*)mn, (uint16_t*)out, N, K);
  else if (scale_dtype == 0)
    hipLaunchKernelGGL(dequant_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, (const uint8_t*)qweight,
                       (const uint16_t*)scale, (const uint16_t*)mn, (uint16_t*)out, N, K);
  else
    return TR_ERR_ARG;
  return hipGetLastError() == hipSuccess ? TR_OK : TR_ERR_LAUNCH;
}

int tr_dequant_packed(const void* packed, void* out, int N, int K, int scale_dtype, int pairs, int as_bf16,
                      void* stream) {
  if (!packed || !out) return TR_ERR_ARG;
  if (!shape_ok(N, K) || (pairs && N % 32)) return TR_ERR_SHAPE;
  if (scale_dtype != 0 && scale_dtype != 1) return TR_ERR_ARG;
  const dim3 grid(quad_grid(N, K)), block(256);
  const int F = pairs ? N / 2 : 0;
  if (scale_dtype == 0)
    hipLaunchKernelGGL((dequant_packed_kernel<false, false>), grid, block, 0, (hipStream_t)stream,
                       (const uint8_t*)packed, (uint16_t*)out, N, K, F);
  else if (as_bf16)
    hipLaunchKernelGGL((dequant_packed_kernel<true, true>), grid, block, 0, (hipStream_t)stream,
                       (const uint8_t*)packed, (uint16_t*)out, N, K, F);
  else
    hipLaunchKernelGGL((dequant_packed_kernel<true, false>), grid, block, 0, (hipStream_t)stream,
                       (const uint8_t*)packed, (uint16_t*)out, N, K, F);
  return hipGetLastError() == hipSuccess ? TR_OK : TR_ERR_LAUNCH;
}

}  // extern "C"
