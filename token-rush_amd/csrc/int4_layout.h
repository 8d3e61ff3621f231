// The int4 weight layout ("quad layout") shared by the GEMMs and the conversion kernels.
//
// Weight layout ("quad layout", made once at load time by tr_pack_int4): the K/128 groups of a
// 16-row strip are padded to a multiple of four (padding groups have zero codes, scale and min,
// so they contribute exactly 0) and stored as quads of four groups, 4352 bytes each
// (34 cache lines of 128 B, so no line is shared by two loads):
//   packed[N/16][Gp/4][4352]
//   bytes [1024 t, 1024 t + 1024): the codes of group 4 q + t. Lane l's 16 bytes at 16 l hold
//     row l % 16 of the group as four 32-bit words; word j covers k0 = 32 j + 8 (l/16) .. k0 + 7
//     (so MFMA j contracts k in [32 j, 32 j + 32) and the matching activations of one row are 64
//     contiguous bytes) with code k0 + 2p in nibble p and k0 + 2p + 1 in
//     nibble p + 4 (p = 0..3), so (w >> 4p) & 0x000F000F is the bf16 pair (k0 + 2p, k0 + 2p + 1)
//     once the exponent is set.
//   bytes [4096, 4352): row i's scale (low 16 bits) and min (high 16 bits) of group 4 q + t at
//     4096 + 16 i + 4 t, so one 16-byte load gives a lane its row's parameters for all four groups.
#pragma once
#include "tr_common.h"

namespace tr {

constexpr int kGroup = 128;
constexpr int kQuad = 4;                          // groups per quad
constexpr int kCodeBytes = 1024;                  // one group's codes for 16 rows
constexpr int kSmOff = kQuad * kCodeBytes;        // parameters of the quad's groups
constexpr int kQuadBytes = kSmOff + 16 * kQuad * 4;  // 4352 = 34 x 128 B

// Groups of a K-long row after padding to whole quads.
__host__ __device__ __forceinline__ int padded_groups(int K) { return (K / kGroup + kQuad - 1) / kQuad * kQuad; }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Scale of a (scale | min << 16) word, fp32.
template <bool F16S>
__device__ __forceinline__ float sm_scale(uint32_t sm) {
  return F16S ? f16_bits_to_f32(sm & 0xFFFFu) : __uint_as_float(sm << 16);
}
template <bool F16S>
__device__ __forceinline__ float sm_min(uint32_t sm) {
  return F16S ? f16_bits_to_f32(sm >> 16) : __uint_as_float(sm & 0xFFFF0000u);
}

// Bytes of the quad layout of an N x K weight.
inline size_t packed_bytes(int N, int K) { return (size_t)N / 16 * (padded_groups(K) / kQuad) * kQuadBytes; }

// Shapes the kernels take: whole 16-row strips and 128-wide groups, and a packed weight that
// 32-bit buffer offsets address.
inline bool shape_ok(int N, int K) {
  return N > 0 && K > 0 && N % 16 == 0 && K % kGroup == 0 && packed_bytes(N, K) < ((size_t)1 << 31);
}

}  // namespace tr
