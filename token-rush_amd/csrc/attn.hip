// Full-attention verify step for gfx950 over an FP8 (e4m3fn) KV cache with per-(head, position)
// fp32 scales: the prep of the M new tokens (q/k RMSNorm, partial rope, cache write) and
// flash-decoding (split over the live keys, then a reduce with the sigmoid output gate).
//
// Follows the reference's Triton kernels (tokenrush/fused.py:247-325 _attn_prep_kernel and
// attn_prep, :355-470 _attn_split_kernel, _attn_reduce_kernel and attn_decode_fused):
//   prep (heads 0..HQ-1 from the q part of qkv [HQ (q | gate) 2D | HKV D | HKV D], heads HQ..
//   for k): xn = bf16(x * rsqrt(mean(x^2) + eps) * (1 + w)); on the first RD dims, with halves
//   x1, x2 and the position's cos/sin: o1 = bf16(bf16(x1 c) + bf16(-x2 s)),
//   o2 = bf16(bf16(x2 c) + bf16(x1 s)). q is written bf16; k and the raw v go to cache row
//   pos + t as fp8(x / sc) with sc = max(amax(x), 1e-6) / 448.
//   attention: query t of head h sees cache rows <= pos + t; scores q . bf16(k8 * ksc) / sqrt(D);
//   online softmax in fp32 (base 2 on the device: maxima and exponents in log2 units) with l
//   summed before the value scale, P = bf16(p * vsc), acc += P v8;
//   splits combined by their maxima; o = bf16(acc / l) * bf16(sigmoid(gate)), bf16 out.
//
// MI355X layout of the split kernel: one workgroup of four waves per (kv head, split, group of up to 48 of
// the G M query rows of the kv head, G = HQ / HKV). The waves take alternate 32-key blocks and each runs all
// of the group's rows on its own block, straight from the cache rows in registers: no LDS and no barrier
// between the blocks.
//   S^T = K8 Q^T (v_mfma_f32_16x16x32_bf16): a lane's 16-byte load of a key row is the A operand of two MFMAs
//   (fp8 is exact in bf16; the k index may run over the dims in any order that Q^T, held in LDS, shares); the
//   key's scale multiplies the fp32 score. The lane then holds eight keys' scores of one query row, which is
//   the B operand of O^T = V^T P^T for those keys. V: a lane loads 16 dims of its eight keys; byte e of the
//   eight is the A operand of O^T tile e (dims 16 i + e), so V is transposed in registers, by v_perm_b32.
//   Row maxima need two permlane swaps, row sums are made after the loop. After the last block the waves'
//   (m, l, O^T) meet in LDS.
// A split of one or two rounds of four blocks does not merge O^T: the waves' P^T meet in LDS instead, and each
// wave makes a quarter of the dims over all of a round's blocks (attn_split_kernel's `shared`). That alone
// took 1.5 us off 8 tokens over 1k rows; with the last round's empty prefetches gone and O^T transposed over the
// octets, so that its stores are 64 contiguous bytes a row, split + combine over 1k rows went, us: 1 token 9.5 -> 8.5,
// 8 tokens 15.0 -> 12.9, a 32-node tree 20.5 -> 17.8. What is left of the split at 8 tokens over 8100 rows (9.1 us
// from entry): 4.4 until K, V and Q are there (17 MB), 2.7 for scores, probabilities and O^T, 1.9 for 12.6 MB of
// partials.
// Each wave otherwise keeps O^T for up to 48 rows x 256 d in 192 AGPRs, one workgroup per CU, so the launch takes as
// many splits as leave one workgroup per CU.
//
// Before, four waves converted each block into LDS together (two barriers and a transposed write per block)
// and then held 16 query rows each: 2.4 us per 32 keys of a CU, whatever the rows. Split + combine, us
// (24 / 4 heads): 1 token over 100k rows 87 -> 42, 4 tokens 90 -> 46 (208 MB, 4.9 TB/s in the split kernel),
// 8 tokens 93 -> 54; over 8k rows 15.7 -> 12.6, 19.0 -> 16.2, 22.6 -> 20.2; a 32-node tree over 8k 37 -> 29.
// Measured and not kept: a second block of K and V in flight in registers (M = 8 over 8k 22.3 us, 100k 61.6;
// the copies cost more than the wait); key splits not rounded to four blocks (22.9 us at 8k); partial rows
// stored whole through a transposing LDS read (22.6 us; the merge of a 16-row tile costs 2.3 us either way).
#include "accept_common.h"

#include <atomic>

namespace tr {

constexpr int kAttnD = 256;      // head dim
constexpr int kAttnBlk = 32;     // keys per block
constexpr int kAttnMaxM = 8;     // query tokens per chain step
constexpr int kAttnMaxTree = 32; // query tokens (nodes) per draft-tree step: one bit each in a mask word
constexpr int kAttnWaves = 4;
constexpr int kAttnTiles = 3;    // 16-row query tiles per workgroup, at most
constexpr int kAttnCUs = 256;
constexpr float kFp8Max = 448.f;
constexpr float kLog2e = 1.4426950408889634f;  // scores are kept in log2 units: p = 2^(s - m)
constexpr int kMaxSplit = 256;  // key-range splits of one flash-decoding call
static_assert(kMaxSplit <= kAttnD, "the combine kernel gives each split one thread");

// ------------------------------------------------------------------ fp8 e4m3fn (OCP) helpers

// fp32 -> fp8 e4m3fn bits, round to nearest even; magnitudes past the largest finite value
// (448) saturate to it (the writers keep |x| <= 448 up to rounding).
__device__ __forceinline__ uint32_t f32_to_fp8(float x) {
  const uint32_t u = __float_as_uint(x);
  const uint32_t sign = (u >> 24) & 0x80;
  const float a = fabsf(x);
  uint32_t code;
  if (a < 0x1p-6f) {
    code = (uint32_t)__builtin_rintf(a * 512.f);  // subnormal steps of 2^-9; 8 becomes 2^-6
  } else {
    uint32_t v = __float_as_uint(a);
    v += 0x7FFFFu + ((v >> 20) & 1u);            // round the mantissa to 3 bits
    const int e = (int)(v >> 23) - 120;
    const uint32_t m = (v >> 20) & 7;
    code = (e > 15 || (e == 15 && m == 7)) ? 0x7Eu : ((uint32_t)e << 3) | m;
  }
  return sign | code;
}

__device__ __forceinline__ float bf16r_a(float v) { return bf16_bits_to_f32(f32_to_bf16_bits(v)); }

typedef uint32_t u32x4a __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
// Two fp32 -> packed bf16 (round to nearest even, v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pk_bf16(float x, float y) {
  const bf16x2v r = {(__bf16)x, (__bf16)y};
  return __builtin_bit_cast(uint32_t, r);
}
// Eight fp8 bytes -> bf16, exact (scale 1).
__device__ __forceinline__ bf16x8 fp8x8_to_bf16(uint32_t lo, uint32_t hi) {
  const uint4 v = make_uint4(__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, false)),
                             __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, true)),
                             __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, false)),
                             __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, true)));
  return __builtin_bit_cast(bf16x8, v);
}
__device__ __forceinline__ float max_x16(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_x32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Lane (i, o) with elements r -> lane (i, r) with elements o: four by four over a wave's rows of 16 lanes.
__device__ __forceinline__ f32x4 transpose_octets(f32x4 v) {
  uint32_t x[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const float f = v[n];
    x[n] = __float_as_uint(f);
  }
  const auto a = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(x[2], x[3], false, false);
  const auto c = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
  return f32x4{__uint_as_float(c[0]), __uint_as_float(d[0]), __uint_as_float(c[1]), __uint_as_float(d[1])};
}

// ------------------------------------------------------------------ prep

struct AttnPrepArgs {
  const uint16_t* qkv;   // [M, QKV] bf16
  const uint16_t* qn_w;  // [D] bf16
  const uint16_t* kn_w;  // [D] bf16
  const uint16_t* cos;   // [max_pos, RD] bf16
  const uint16_t* sin;
  const int64_t* pos;
  uint8_t* k_cache;      // [HKV, maxlen, D] fp8
  uint8_t* v_cache;
  float* k_scale;        // [HKV, maxlen]
  float* v_scale;
  uint16_t* q_out;       // [M, HQ, D] bf16
  const int32_t* parent; // [M] draft-tree parents, or null for a chain
  int HQ, HKV, RD, maxlen, ld;
  float eps;
};

// Parent of node t of a draft tree (parent[t] < t; node 0 is the root). A parent outside
// 0..t-1 reads as the root, so every walk up the tree ends within t steps.
__device__ __forceinline__ int attn_tree_parent(const int32_t* parent, int t) {
  const int p = parent[t];
  return (p >= 0 && p < t) ? p : 0;
}

// One wave per (head, token); lane l holds dims 4 l .. 4 l + 3. Token t is written to cache row
// pos + t and roped at position pos + t, or, for node t of a draft tree, at pos + depth(t): the
// position it takes once its root path is committed.
__global__ __launch_bounds__(64) void attn_prep_kernel(AttnPrepArgs a) {
  const int head = blockIdx.x, t = blockIdx.y, lane = threadIdx.x;
  int dep = t;
  if (a.parent) {
    // the depth by walking the parents held one per lane (one load for the wave, then shuffles:
    // a walk of dependent memory loads waited for each)
    const int pl = lane > 0 && lane < (int)gridDim.y ? attn_tree_parent(a.parent, lane) : 0;
    dep = 0;
    for (int j = t; j > 0 && dep < kAttnMaxTree; ++dep) j = __shfl(pl, j);
  }
  // Positions past the cache's end: the rope table (maxlen rows) is read at the last row and no
  // cache row is written (the split kernel reads at most maxlen rows), so nothing outside the
  // cache is touched whatever the device position holds.
  const int64_t p_raw = *a.pos + t, r_raw = *a.pos + dep;
  const bool in_cache = p_raw >= 0 && p_raw < a.maxlen;
  const int64_t p = in_cache ? p_raw : (p_raw < 0 ? 0 : a.maxlen - 1);
  const int64_t pr = r_raw < 0 ? 0 : (r_raw >= a.maxlen ? a.maxlen - 1 : r_raw);
  const bool isq = head < a.HQ;
  const int j = head - a.HQ;
  const uint16_t* row = a.qkv + (size_t)t * a.ld;
  const uint16_t* src = isq ? row + (size_t)head * 2 * kAttnD : row + (size_t)a.HQ * 2 * kAttnD + (size_t)j * kAttnD;
  const uint16_t* w = isq ? a.qn_w : a.kn_w;
  const int d0 = 4 * lane;
  uint16_t cs_raw[4], sn_raw[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = (d0 + i) % (a.RD / 2);
    cs_raw[i] = a.cos[(size_t)pr * a.RD + r];
    sn_raw[i] = a.sin[(size_t)pr * a.RD + r];
  }
  float x[4], wv[4];
  {
    const uint2 xu = *(const uint2*)(src + d0), wu = *(const uint2*)(w + d0);
    x[0] = bf16_bits_to_f32(xu.x & 0xFFFFu);
    x[1] = bf16_bits_to_f32(xu.x >> 16);
    x[2] = bf16_bits_to_f32(xu.y & 0xFFFFu);
    x[3] = bf16_bits_to_f32(xu.y >> 16);
    wv[0] = bf16_bits_to_f32(wu.x & 0xFFFFu);
    wv[1] = bf16_bits_to_f32(wu.x >> 16);
    wv[2] = bf16_bits_to_f32(wu.y & 0xFFFFu);
    wv[3] = bf16_bits_to_f32(wu.y >> 16);
  }
  float ss = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  const float inv = 1.f / sqrtf(ss / (float)kAttnD + a.eps);
  float xn[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) xn[i] = bf16r_a(x[i] * inv * (1.f + wv[i]));
  // partial rope on dims < RD: dim r pairs with r + RD / 2 (a lane RD / 8 lanes away). The
  // table entries were loaded with x (in-range indices for every dim, used where d < RD).
  const int half = a.RD / 2;
  float out[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float other = __shfl_xor(xn[i], half / 4);
    const int d = d0 + i;
    out[i] = xn[i];
    if (d < a.RD) {
      const float c = bf16_bits_to_f32(cs_raw[i]), s = bf16_bits_to_f32(sn_raw[i]);
      out[i] = d < half ? bf16r_a(bf16r_a(xn[i] * c) + bf16r_a(-other * s))
                        : bf16r_a(bf16r_a(xn[i] * c) + bf16r_a(other * s));
    }
  }
  if (isq) {
    uint16_t* qo = a.q_out + ((size_t)t * a.HQ + head) * kAttnD + d0;
    uint2 st;
    st.x = (uint32_t)f32_to_bf16_bits(out[0]) | ((uint32_t)f32_to_bf16_bits(out[1]) << 16);
    st.y = (uint32_t)f32_to_bf16_bits(out[2]) | ((uint32_t)f32_to_bf16_bits(out[3]) << 16);
    *(uint2*)qo = st;
    return;
  }
  if (!in_cache) return;
  // key: fp8 with one scale per (head, position)
  float am = fmaxf(fmaxf(fabsf(out[0]), fabsf(out[1])), fmaxf(fabsf(out[2]), fabsf(out[3])));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o));
  const float sc = fmaxf(am, 1e-6f) / kFp8Max;
  const size_t crow = ((size_t)j * a.maxlen + p);
  uint32_t kb = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) kb |= f32_to_fp8(out[i] / sc) << (8 * i);
  *(uint32_t*)(a.k_cache + crow * kAttnD + d0) = kb;
  // value: raw bf16 from qkv
  const uint2 vu = *(const uint2*)(row + (size_t)a.HQ * 2 * kAttnD + (size_t)(a.HKV + j) * kAttnD + d0);
  const float v[4] = {bf16_bits_to_f32(vu.x & 0xFFFFu), bf16_bits_to_f32(vu.x >> 16), bf16_bits_to_f32(vu.y & 0xFFFFu),
                      bf16_bits_to_f32(vu.y >> 16)};
  float vm = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) vm = fmaxf(vm, __shfl_xor(vm, o));
  const float sv = fmaxf(vm, 1e-6f) / kFp8Max;
  uint32_t vb = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) vb |= f32_to_fp8(v[i] / sv) << (8 * i);
  *(uint32_t*)(a.v_cache + crow * kAttnD + d0) = vb;
  if (lane == 0) {
    a.k_scale[crow] = sc;
    a.v_scale[crow] = sv;
  }
}

// ------------------------------------------------------------------ split (flash-decoding)

struct AttnSplitArgs {
  const uint16_t* q;       // [M, HQ, D] bf16
  const uint8_t* k_cache;  // [HKV, maxlen, D] fp8
  const uint8_t* v_cache;
  const float* k_scale;    // [HKV, maxlen]
  const float* v_scale;
  const int64_t* pos;
  float* m_part;           // [M HQ, NSPLIT]
  float* l_part;
  float* acc_part;         // [M HQ, NSPLIT, D]
  const int32_t* parent;   // [M] draft-tree parents, or null for a chain
  int HQ, HKV, M, maxlen, nsplit;
  float scale;
};

// Splits that hold keys: split s takes blocks s per .. of the nblk live blocks, per a multiple of the four
// waves (a wave alone on a last block takes as long as four, and fewer splits mean fewer partials to combine).
struct AttnRange {
  int nblk, per;
  __device__ __forceinline__ AttnRange(int64_t L, int nsplit) {
    nblk = (int)((L + kAttnBlk - 1) / kAttnBlk);
    per = ((nblk + nsplit - 1) / nsplit + kAttnWaves - 1) / kAttnWaves * kAttnWaves;
  }
  // split 0 always counts: it writes the empty partials of a call without live rows
  __device__ __forceinline__ int used(int nsplit) const { return per > 0 ? max(1, min(nsplit, (nblk + per - 1) / per)) : 1; }
};

// T 16-row query tiles per workgroup; its four waves take alternate key blocks of the split.
template <int T>
__global__ __launch_bounds__(64 * kAttnWaves, 1) void attn_split_kernel(AttnSplitArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];  // Q operands; after the loop each wave's O^T tile, then its (m, l)
  const int j = blockIdx.x / a.nsplit, s = blockIdx.x % a.nsplit;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, o = lane >> 4;
  const int G = a.HQ / a.HKV, rows = G * a.M;
  const int tile0 = (int)blockIdx.y * T;
  const int64_t pos = *a.pos;
  const int64_t L = pos + a.M;
  const AttnRange range(L, a.nsplit);
  const int b0 = s * range.per, b1 = min(b0 + range.per, range.nblk);
  if (s >= range.used(a.nsplit)) return;

  // Cache reads go through buffer resources sized to the L live rows: rows past them, and the
  // prefetch past the split's last block, read zeros with no memory access and no branch.
  const int liveL = (int)min(max(L, (int64_t)0), (int64_t)a.maxlen);   // never past the cache
  const auto krs = __builtin_amdgcn_make_buffer_rsrc((void*)(a.k_cache + (size_t)j * a.maxlen * kAttnD), (short)0,
                                                     liveL * kAttnD, 0x00020000);
  const auto vrs = __builtin_amdgcn_make_buffer_rsrc((void*)(a.v_cache + (size_t)j * a.maxlen * kAttnD), (short)0,
                                                     liveL * kAttnD, 0x00020000);
  const auto ksr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.k_scale + (size_t)j * a.maxlen), (short)0, liveL * 4,
                                                     0x00020000);
  const auto vsr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.v_scale + (size_t)j * a.maxlen), (short)0, liveL * 4,
                                                     0x00020000);
  constexpr uint32_t kOob = 0x7FFF0000u;
  constexpr int kNt = 2;  // the cache rows are read once per step: non-temporal, as the GEMM streams its weights
  // K: lane (i, o) loads key 16 kt + i, dims 64 c + 16 o .. + 15; V: keys 16 kt + 4 o + r, dims 16 i .. + 15;
  // the scales of keys 16 kt + 4 o .. + 3
  u32x4a kraw[2][4], vraw[2][4], ksv[2], vsv[2];
  auto fetch_k = [&](int blk) {
    const uint32_t base = blk < b1 ? (uint32_t)blk * kAttnBlk : kOob / kAttnD;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        kraw[kt][c] = __builtin_amdgcn_raw_buffer_load_b128(krs, (base + 16 * kt + i) * kAttnD + 16 * o + 64 * c, 0, kNt);
      ksv[kt] = __builtin_amdgcn_raw_buffer_load_b128(ksr, (base + 16 * kt + 4 * o) * 4, 0, kNt);
    }
  };
  auto fetch_v = [&](int blk) {
    const uint32_t base = blk < b1 ? (uint32_t)blk * kAttnBlk : kOob / kAttnD;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        vraw[kt][r] = __builtin_amdgcn_raw_buffer_load_b128(vrs, (base + 16 * kt + 4 * o + r) * kAttnD + 16 * i, 0, kNt);
      vsv[kt] = __builtin_amdgcn_raw_buffer_load_b128(vsr, (base + 16 * kt + 4 * o) * 4, 0, kNt);
    }
  };
  // A round of the short ranges: the wave's quarter of the dims of the round's four blocks (lane (i, o): dims
  // 64 wave + 4 i .. + 3 of keys 16 kt + 4 o + r), and the scales of its own block
  uint32_t vq[kAttnWaves][8];
  auto fetch_vq = [&](int blk0) {
#pragma unroll
    for (int b = 0; b < kAttnWaves; ++b) {
      const uint32_t base = blk0 + b < b1 ? (uint32_t)(blk0 + b) * kAttnBlk : kOob / kAttnD;
#pragma unroll
      for (int n = 0; n < 8; ++n)
        vq[b][n] = __builtin_amdgcn_raw_buffer_load_b32(vrs, (base + 16 * (n / 4) + 4 * o + n % 4) * kAttnD + 64 * wave + 4 * i,
                                                        0, kNt);
    }
  };
  auto fetch_vs = [&](int blk) {
    const uint32_t base = blk < b1 ? (uint32_t)blk * kAttnBlk : kOob / kAttnD;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) vsv[kt] = __builtin_amdgcn_raw_buffer_load_b128(vsr, (base + 16 * kt + 4 * o) * 4, 0, kNt);
  };
  // One round always, two from two query tiles up (8 tokens over 8192 rows, 257 blocks: 20.2 us against 20.9;
  // 1 token 13.4 / 12.7); at three rounds and more the barriers cost what the merge does (16-node tree over 8k
  // 25.3 / 25.2) and at eight more (8 tokens over 32k 35.0 / 30.5). The same for every split.
  const bool shared = range.per <= (T > 1 ? 2 : 1) * kAttnWaves;
  fetch_k(b0 + wave);
  if (shared) {
    fetch_vs(b0 + wave);
    fetch_vq(b0);
  } else {
    fetch_v(b0 + wave);
  }

  // Q^T operand of MFMA (c, h): lane (i, o) holds row i of the tile, dims 64 c + 16 o + 8 h .. + 7. They sit
  // in LDS in lane order: in registers they and O^T did not fit beside the block in flight.
  char* const qs = (char*)lds + lane * 16;
  size_t head[T];    // the lane's row as (token, query head)
  uint32_t vis[T];   // the new keys it sees, bit r for row pos + r: i <= its token, or its tree ancestors
  bool rvalid[T];
  const int pl = a.parent && lane > 0 && lane < a.M ? attn_tree_parent(a.parent, lane) : 0;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int row = 16 * (tile0 + t) + i;
    rvalid[t] = row < rows;
    const int qrow = rvalid[t] ? row : 0, qi = qrow / G;  // padding rows repeat row 0 and are not stored
    head[t] = (size_t)qi * a.HQ + j * G + (qrow - qi * G);
    u32x4a q[2];  // wave w brings c = w
#pragma unroll
    for (int h = 0; h < 2; ++h) q[h] = *(const u32x4a*)(a.q + head[t] * kAttnD + 64 * wave + 16 * o + 8 * h);
#pragma unroll
    for (int h = 0; h < 2; ++h) *(u32x4a*)(qs + ((t * 4 + wave) * 2 + h) * 1024) = q[h];
    vis[t] = qi >= 31 ? ~0u : (2u << qi) - 1u;  // (no bit at or past M: qi < M)
    if (a.parent) {
      // the parents one per lane (one load for the wave), then the walk by shuffles
      vis[t] = 1u;  // the root: every node sees it
      int jn = qi;
      for (int d = 0; d < kAttnMaxTree; ++d) {
        vis[t] |= 1u << jn;
        jn = __shfl(pl, jn);  // the root's entry is 0
        if (__all(jn == 0)) break;
      }
    }
  }
  lds_barrier();

  const float sl2 = a.scale * kLog2e;
  // Masked scores of block blk in log2 units, its V scales, and the K prefetch of the wave's next block
  auto scores = [&](int blk, float (&sc)[T][8], float (&vf)[8], bool more) {
    // S^T = K8 Q^T for the block's two 16-key tiles (fp8 is exact in bf16): lane (i, o) gets keys
    // 16 kt + 4 o + r of row i; the key's scale multiplies the fp32 score
    f32x4 st[T][2];
#pragma unroll
    for (int t = 0; t < T; ++t) st[t][0] = st[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 qc[T][2];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) qc[t][h] = *(const bf16x8*)(qs + (t * 8 + h) * 1024);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      bf16x8 qn[T][2];  // the next c's Q, read ahead of this one's MFMAs
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) qn[t][h] = *(const bf16x8*)(qs + ((t * 4 + (c < 3 ? c + 1 : c)) * 2 + h) * 1024);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bf16x8 k0 = fp8x8_to_bf16(kraw[0][c][2 * h], kraw[0][c][2 * h + 1]);
        const bf16x8 k1 = fp8x8_to_bf16(kraw[1][c][2 * h], kraw[1][c][2 * h + 1]);
#pragma unroll
        for (int t = 0; t < T; ++t) {
          st[t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qc[t][h], st[t][0], 0, 0, 0);
          st[t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qc[t][h], st[t][1], 0, 0, 0);
        }
      }
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) qc[t][h] = qn[t][h];
      __builtin_amdgcn_sched_barrier(0);  // bounds the operands made ahead
    }
    float kf[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      kf[n] = __uint_as_float(ksv[n / 4][n % 4]) * sl2;
      vf[n] = __uint_as_float(vsv[n / 4][n % 4]);
    }
    if (more) fetch_k(blk + kAttnWaves);
    const int64_t key0 = (int64_t)blk * kAttnBlk;
    const bool committed = key0 + kAttnBlk <= pos;  // uniform: no new key in the block, nothing to mask
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int n = 0; n < 8; ++n) sc[t][n] = st[t][n / 4][n % 4] * kf[n];
    if (!committed) {
      // bit 32 + r of a row's 64-bit word: key pos + r visible; committed keys (r < 0) always are. This lane's
      // keys sit at bits 0-3 and 16-19 once the word is shifted to its first key.
      const int sh = (int)(key0 - pos) + 4 * o + 32;  // 1 .. 75
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const uint64_t word = ((uint64_t)vis[t] << 32) | 0xFFFFFFFFu;
        const uint32_t seen = sh < 64 ? (uint32_t)(word >> (sh & 63)) : 0u;
#pragma unroll
        for (int n = 0; n < 8; ++n) sc[t][n] = (seen >> (16 * (n / 4) + n % 4)) & 1u ? sc[t][n] : -INFINITY;
      }
    }
  };
  constexpr float kLazyMax = 48.f;

  if (shared) {
    // Rounds of four blocks, scores of one block to each wave; P^T meets in LDS at the row's common maximum and
    // each wave makes its quarter of O^T over all four blocks, so nothing is left to merge.
    char* const ps = (char*)lds + T * 8192;
    float* const mw = (float*)(ps + kAttnWaves * T * 1024);
    f32x4 oq[T][4];  // tile e: dims 64 wave + 4 i' + e; lane (i, o): row i, dims 64 wave + 16 o + 4 r + e
    float m_r[T], l_r[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
#pragma unroll
      for (int e = 0; e < 4; ++e) oq[t][e] = f32x4{0.f, 0.f, 0.f, 0.f};
      m_r[t] = -INFINITY;
      l_r[t] = 0.f;
    }
    // `more` is a constant at both uses: the last round issues no loads for a next one (one load instruction of a
    // wave holds the CU's address unit for 16 cycles whether its lanes fetch or not)
    auto round = [&](int blk0, bool more) {
      float sc[T][8], vf[8];
      scores(blk0 + wave, sc, vf, more);
      if (more) fetch_vs(blk0 + kAttnWaves + wave);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const float mx = fmaxf(fmaxf(fmaxf(sc[t][0], sc[t][1]), fmaxf(sc[t][2], sc[t][3])),
                               fmaxf(fmaxf(sc[t][4], sc[t][5]), fmaxf(sc[t][6], sc[t][7])));
        const float mr = max_x32(max_x16(mx));
        if (o == 0) mw[(t * 16 + i) * kAttnWaves + wave] = mr;
      }
      lds_barrier();
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const float4 mv = *(const float4*)(mw + (t * 16 + i) * kAttnWaves);
        const float mx = fmaxf(fmaxf(mv.x, mv.y), fmaxf(mv.z, mv.w));
        if (mx > m_r[t] + kLazyMax) {  // the reference maximum and its restart: see below
          m_r[t] = mx;
          l_r[t] = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) oq[t][e] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const float m_safe = m_r[t] == -INFINITY ? 0.f : m_r[t];
        uint32_t w[4];
#pragma unroll
        for (int n = 0; n < 8; n += 2) {
          const float p0 = __builtin_amdgcn_exp2f(sc[t][n] - m_safe), p1 = __builtin_amdgcn_exp2f(sc[t][n + 1] - m_safe);
          l_r[t] += p0 + p1;
          w[n / 2] = pk_bf16(p0 * vf[n], p1 * vf[n + 1]);
        }
        *(uint4*)(ps + (wave * T + t) * 1024 + lane * 16) = make_uint4(w[0], w[1], w[2], w[3]);
      }
      lds_barrier();
#pragma unroll
      for (int b = 0; b < kAttnWaves; ++b) {
        bf16x8 pb[T];
#pragma unroll
        for (int t = 0; t < T; ++t) pb[t] = *(const bf16x8*)(ps + (b * T + t) * 1024 + lane * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t sel = 0x0C0C0000u | ((4u + e) << 8) | (uint32_t)e;
          uint32_t w[4];
#pragma unroll
          for (int n = 0; n < 4; ++n)
            w[n] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                                                    __builtin_amdgcn_perm(vq[b][2 * n + 1], vq[b][2 * n], sel), 1.f, false));
          const bf16x8 va = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
#pragma unroll
          for (int t = 0; t < T; ++t) oq[t][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pb[t], oq[t][e], 0, 0, 0);
        }
      }
      if (more) fetch_vq(blk0 + kAttnWaves);
    };
    int blk0 = b0;
    for (; blk0 + kAttnWaves < b1; blk0 += kAttnWaves) round(blk0, true);
    if (blk0 < b1) round(blk0, false);
    // row sums over the octets, then over the waves (mw's reads are behind the last barrier)
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const float l = sum_x32(sum_x16(l_r[t]));
      if (o == 0) mw[(t * 16 + i) * kAttnWaves + wave] = l;
      // registers r <-> octets o transposed, so that a row's four lanes store 64 contiguous bytes
      f32x4 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = transpose_octets(oq[t][e]);
      if (rvalid[t]) {
        float* const part = a.acc_part + (head[t] * a.nsplit + s) * kAttnD + 64 * wave + 4 * o;
#pragma unroll
        for (int k = 0; k < 4; ++k) *(float4*)(part + 16 * k) = make_float4(v[0][k], v[1][k], v[2][k], v[3][k]);
      }
    }
    lds_barrier();
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if (wave != 0 || o != 0 || !rvalid[t]) continue;
      const float4 lv = *(const float4*)(mw + (t * 16 + i) * kAttnWaves);
      a.m_part[head[t] * a.nsplit + s] = m_r[t];
      a.l_part[head[t] * a.nsplit + s] = ((lv.x + lv.y) + lv.z) + lv.w;
    }
    return;
  }

  f32x4 acc[T][16];  // O^T tile e: dims 16 i' + e; lane (i, o), register r: row i, dim 64 o + 16 r + e
  float m_i[T], l_i[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[t][e] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_i[t] = -INFINITY;
    l_i[t] = 0.f;
  }
  for (int blk = b0 + wave; blk < b1; blk += kAttnWaves) {
    float sc[T][8], vf[8];
    scores(blk, sc, vf, true);
    // online softmax in log2 units: p = 2^(s - m) by v_exp_f32
    // Rows keep the maximum of their first block as the reference m (p, l and O^T are floats: any common scale
    // will do) until a key passes it by more than 2^kLazyMax. That key outweighs everything before it: 2^20
    // keys at the old maximum are 2^-28 of it, below fp32's last bit, so the row's sums restart from zero.
    // (Rescaling instead put O^T, which lives in AGPRs, through VGPRs and spilled.)
#pragma unroll
    for (int t = 0; t < T; ++t) {
      float mx = fmaxf(fmaxf(fmaxf(sc[t][0], sc[t][1]), fmaxf(sc[t][2], sc[t][3])),
                       fmaxf(fmaxf(sc[t][4], sc[t][5]), fmaxf(sc[t][6], sc[t][7])));
      mx = max_x32(max_x16(mx));
      if (mx > m_i[t] + kLazyMax) {  // a first finite maximum always passes -inf
        m_i[t] = mx;
        l_i[t] = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][e] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    bf16x8 pb[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const float m_safe = m_i[t] == -INFINITY ? 0.f : m_i[t];
      uint32_t w[4];
#pragma unroll
      for (int n = 0; n < 8; n += 2) {
        const float p0 = __builtin_amdgcn_exp2f(sc[t][n] - m_safe), p1 = __builtin_amdgcn_exp2f(sc[t][n + 1] - m_safe);
        l_i[t] += p0 + p1;  // this lane's keys; the octets' sums meet after the loop
        w[n / 2] = pk_bf16(p0 * vf[n], p1 * vf[n + 1]);
      }
      pb[t] = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
    }
    // O^T += V^T P^T: tile e takes byte e of the lane's eight keys (k-index 4 kt + r <-> key 16 kt + 4 o + r),
    // one v_perm_b32 and one conversion (scale 1: exact) per pair
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const uint32_t sel = 0x0C0C0000u | ((4u + (e & 3)) << 8) | (uint32_t)(e & 3);  // byte 0 = second[e], byte 1 = first[e]
      uint32_t w[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const uint32_t b = __builtin_amdgcn_perm(vraw[n / 2][2 * (n & 1) + 1][e / 4], vraw[n / 2][2 * (n & 1)][e / 4], sel);
        w[n] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, false));
      }
      const bf16x8 va = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
#pragma unroll
      for (int t = 0; t < T; ++t) acc[t][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pb[t], acc[t][e], 0, 0, 0);
      if (e % 2) __builtin_amdgcn_sched_barrier(0);
    }
    fetch_v(blk + kAttnWaves);
  }
#pragma unroll
  for (int t = 0; t < T; ++t) l_i[t] = sum_x32(sum_x16(l_i[t]));

  // The waves meet in LDS, one query tile at a time: each puts its (m, l) and O^T there and
  // sums its share of the O^T tiles over the waves, in wave order, at the common maximum.
  constexpr int EP = 16 / kAttnWaves;
  float* const ml = lds + (size_t)kAttnWaves * 4096;
  float* const mine = lds + (size_t)wave * 4096 + lane * 4;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    lds_barrier();  // the loop's Q reads, or the previous tile's, are done
    if (o == 0) *(float2*)(ml + (wave * 16 + i) * 2) = make_float2(m_i[t], l_i[t]);
#pragma unroll
    for (int e = 0; e < 16; ++e) *(f32x4*)(mine + e * 256) = acc[t][e];
    lds_barrier();
    float2 p[kAttnWaves];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int k = 0; k < kAttnWaves; ++k) {
      p[k] = *(const float2*)(ml + (k * 16 + i) * 2);
      m = fmaxf(m, p[k].x);
    }
    const float m_safe = m == -INFINITY ? 0.f : m;
    f32x4 v[EP];
#pragma unroll
    for (int e = 0; e < EP; ++e) v[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kAttnWaves; ++k) {
      const float f = __builtin_amdgcn_exp2f(p[k].x - m_safe);
      l += p[k].y * f;
      const float* const from = lds + (size_t)k * 4096 + (EP * wave) * 256 + lane * 4;
#pragma unroll
      for (int e = 0; e < EP; ++e) v[e] = v[e] + *(const f32x4*)(from + e * 256) * f;
    }
    if (!rvalid[t]) continue;
    float* const part = a.acc_part + (head[t] * a.nsplit + s) * kAttnD + 64 * o;
    if (o == 0 && wave == 0) {
      a.m_part[head[t] * a.nsplit + s] = m;
      a.l_part[head[t] * a.nsplit + s] = l;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int e = 0; e < EP; e += 4)
        *(float4*)(part + EP * wave + 16 * r + e) = make_float4(v[e][r], v[e + 1][r], v[e + 2][r], v[e + 3][r]);
  }
}

// ------------------------------------------------------------------ reduce + output gate

struct AttnReduceArgs {
  const float* m_part;
  const float* l_part;
  const float* acc_part;
  const uint16_t* qkv;  // [M, QKV] for the gates
  const int64_t* pos;
  uint16_t* out;        // [M, HQ D]
  int HQ, M, nsplit, ld;
};

// One workgroup of D threads per (token, query head). Every load is issued up front: the split
// accumulators of this thread's dimension in batches of 64 (clamped indices past nsplit, weight
// 0), one split's (m, l) per thread, and the gate; the split maximum and the weighted total are
// block reductions.
__global__ __launch_bounds__(kAttnD) void attn_reduce_kernel(AttnReduceArgs a) {
  constexpr int kB = 64;
  __shared__ float wsh[kMaxSplit], red[kAttnD / 64];
  const int h = blockIdx.x, d = threadIdx.x, lane = d & 63, wave = d >> 6;
  const int ns = AttnRange(*a.pos + a.M, a.nsplit).used(a.nsplit);  // the splits that hold keys
  const int t = h / a.HQ, hh = h % a.HQ;
  const uint16_t graw = a.qkv[(size_t)t * a.ld + (size_t)hh * 2 * kAttnD + kAttnD + d];
  const float* ap = a.acc_part + (size_t)h * a.nsplit * kAttnD + d;
  float v[kB];
#pragma unroll
  for (int i = 0; i < kB; ++i) v[i] = ap[(size_t)min(i, ns - 1) * kAttnD];
  const int sc = min(d, ns - 1);
  const float m_s = a.m_part[(size_t)h * a.nsplit + sc], l_s = a.l_part[(size_t)h * a.nsplit + sc];
  const bool mine = d < ns;  // ns <= kMaxSplit == kAttnD
  // maximum over the splits
  float mm = mine ? m_s : -INFINITY;
  mm = fmaxf(mm, __shfl_xor(mm, 32));
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) mm = fmaxf(mm, __shfl_xor(mm, o));
  if (lane == 0) red[wave] = mm;
  __syncthreads();
  mm = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float w = mine && m_s != -INFINITY ? __builtin_amdgcn_exp2f(m_s - mm) : 0.f;  // maxima in log2 units
  if (mine) wsh[d] = w;
  // total weight sum_s w_s l_s
  float lt = sum_wave(w * l_s);
  __syncthreads();  // red[] reads done, wsh[] written
  if (lane == 0) red[wave] = lt;
  __syncthreads();
  lt = ((red[0] + red[1]) + red[2]) + red[3];
  float o = 0.f;
#pragma unroll
  for (int i = 0; i < kB; ++i)
    if (i < ns) o += wsh[i] * v[i];
  for (int s0 = kB; s0 < ns; s0 += kB) {  // nsplit > 64: further batches
#pragma unroll
    for (int i = 0; i < kB; ++i) v[i] = ap[(size_t)min(s0 + i, ns - 1) * kAttnD];
#pragma unroll
    for (int i = 0; i < kB; ++i)
      if (s0 + i < ns) o += wsh[s0 + i] * v[i];
  }
  o = bf16r_a(o / lt);
  const float gate = bf16_bits_to_f32(graw);
  const float g = bf16r_a(1.f / (1.f + expf(-gate)));
  a.out[(size_t)h * kAttnD + d] = f32_to_bf16_bits(o * g);
}

}  // namespace tr

using namespace tr;

extern "C" {

size_t tr_attn_workspace_bytes(int M, int HQ, int nsplit) {
  if (M < 1 || M > kAttnMaxTree || HQ < 1 || nsplit < 1) return 0;
  const size_t rows = (size_t)M * HQ * nsplit;
  return rows * (2 + kAttnD) * sizeof(float);
}

}  // extern "C"

namespace {

int attn_prep_launch(const void* qkv, int ld, const void* q_norm_w, const void* k_norm_w, const void* cos,
                     const void* sin, int rotary_dim, const int64_t* pos, void* k_cache, void* v_cache, float* k_scale,
                     float* v_scale, int maxlen, void* q_out, int M, int HQ, int HKV, int D, float eps,
                     const int32_t* parent, void* stream) {
  // rotary_dim: a power of two (its two halves are then an xor-shuffle apart) in [8, D]
  if (D != kAttnD || HQ < 1 || HKV < 1 || HQ % HKV || (rotary_dim & (rotary_dim - 1)) || rotary_dim < 8 ||
      rotary_dim > D || maxlen < M)
    return TR_ERR_SHAPE;
  if (!qkv || !q_norm_w || !k_norm_w || !cos || !sin || !pos || !k_cache || !v_cache || !k_scale || !v_scale || !q_out)
    return TR_ERR_ARG;
  if (ld < 2 * HQ * D + 2 * HKV * D) return TR_ERR_ARG;
  AttnPrepArgs a;
  a.qkv = (const uint16_t*)qkv;
  a.qn_w = (const uint16_t*)q_norm_w;
  a.kn_w = (const uint16_t*)k_norm_w;
  a.cos = (const uint16_t*)cos;
  a.sin = (const uint16_t*)sin;
  a.pos = pos;
  a.k_cache = (uint8_t*)k_cache;
  a.v_cache = (uint8_t*)v_cache;
  a.k_scale = k_scale;
  a.v_scale = v_scale;
  a.q_out = (uint16_t*)q_out;
  a.parent = parent;
  a.HQ = HQ;
  a.HKV = HKV;
  a.RD = rotary_dim;
  a.maxlen = maxlen;
  a.ld = ld;
  a.eps = eps;
  hipLaunchKernelGGL(attn_prep_kernel, dim3(HQ + HKV, M), dim3(64), 0, (hipStream_t)stream, a);
  return hipGetLastError() == hipSuccess ? TR_OK : TR_ERR_LAUNCH;
}

template <int T>
hipError_t split_launch(const AttnSplitArgs& s, int wgs, int groups, hipStream_t stream) {
  // the Q operands; after the loop each wave's O^T tile, then its (m, l) per row
  constexpr size_t kLds = (size_t)kAttnWaves * (16384 + 16 * 8);
  static_assert(T * 8192 <= kLds, "Q operands");
  static std::atomic<uint64_t> raised{0};  // devices on which the kernel's LDS limit is raised
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  if (!(raised.load(std::memory_order_relaxed) & bit)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_split_kernel<T>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
    if (e != hipSuccess) return e;
    raised.fetch_or(bit, std::memory_order_relaxed);
  }
  hipLaunchKernelGGL((attn_split_kernel<T>), dim3(wgs, groups), dim3(64 * kAttnWaves), kLds, stream, s);
  return hipGetLastError();
}

int attn_decode_launch(const void* q, const void* qkv, int ld, const void* k_cache, const void* v_cache,
                       const float* k_scale, const float* v_scale, int maxlen, const int64_t* pos, void* out,
                       void* workspace, size_t workspace_bytes, int M, int HQ, int HKV, int D, int nsplit,
                       const int32_t* parent, void* stream) {
  if (D != kAttnD || HQ < 1 || HKV < 1 || HQ % HKV || nsplit < 1 || nsplit > kMaxSplit || maxlen < M)
    return TR_ERR_SHAPE;
  if (!q || !qkv || !k_cache || !v_cache || !k_scale || !v_scale || !pos || !out || !workspace) return TR_ERR_ARG;
  if (ld < 2 * HQ * D + 2 * HKV * D || workspace_bytes < tr_attn_workspace_bytes(M, HQ, nsplit)) return TR_ERR_ARG;
  const size_t rows = (size_t)M * HQ * nsplit;
  AttnSplitArgs s;
  s.q = (const uint16_t*)q;
  s.k_cache = (const uint8_t*)k_cache;
  s.v_cache = (const uint8_t*)v_cache;
  s.k_scale = k_scale;
  s.v_scale = v_scale;
  s.pos = pos;
  s.m_part = (float*)workspace;
  s.l_part = s.m_part + rows;
  s.acc_part = s.l_part + rows;
  s.parent = parent;
  s.HQ = HQ;
  s.HKV = HKV;
  s.M = M;
  s.maxlen = maxlen;
  s.nsplit = nsplit;
  s.scale = 1.f / sqrtf((float)D);
  // The G M query rows of a kv head in groups of up to three 16-row tiles, and as many key splits (nsplit at
  // most) as leave one workgroup per CU: a CU holds one of them (see the kernel's registers), and every split
  // costs its partials.
  const int tiles = ((HQ / HKV) * M + 15) / 16, groups = (tiles + kAttnTiles - 1) / kAttnTiles;
  const int fit = kAttnCUs / (HKV * groups);
  s.nsplit = nsplit < fit ? nsplit : fit > 1 ? fit : 1;
  const hipStream_t st = (hipStream_t)stream;
  const int T = (tiles + groups - 1) / groups, wgs = HKV * s.nsplit;
  const hipError_t e = T == 1 ? split_launch<1>(s, wgs, groups, st)
                       : T == 2 ? split_launch<2>(s, wgs, groups, st) : split_launch<3>(s, wgs, groups, st);
  if (e != hipSuccess) return TR_ERR_LAUNCH;
  AttnReduceArgs r;
  r.m_part = s.m_part;
  r.l_part = s.l_part;
  r.acc_part = s.acc_part;
  r.qkv = (const uint16_t*)qkv;
  r.out = (uint16_t*)out;
  r.pos = pos;
  r.HQ = HQ;
  r.M = M;
  r.nsplit = s.nsplit;
  r.ld = ld;
  hipLaunchKernelGGL(attn_reduce_kernel, dim3(M * HQ), dim3(kAttnD), 0, (hipStream_t)stream, r);
  return hipGetLastError() == hipSuccess ? TR_OK : TR_ERR_LAUNCH;
}

}  // namespace

extern "C" {

int tr_attn_prep(const void* qkv, int ld, const void* q_norm_w, const void* k_norm_w, const void* cos,
                 const void* sin, int rotary_dim, const int64_t* pos, void* k_cache, void* v_cache, float* k_scale,
                 float* v_scale, int maxlen, void* q_out, int M, int HQ, int HKV, int D, float eps, void* stream) {
  if (M == 0) return TR_OK;
  if (M < 0 || M > kAttnMaxM) return TR_ERR_SHAPE;
  return attn_prep_launch(qkv, ld, q_norm_w, k_norm_w, cos, sin, rotary_dim, pos, k_cache, v_cache, k_scale, v_scale,
                          maxlen, q_out, M, HQ, HKV, D, eps, nullptr, stream);
}

int tr_attn_decode(const void* q, const void* qkv, int ld, const void* k_cache, const void* v_cache,
                   const float* k_scale, const float* v_scale, int maxlen, const int64_t* pos, void* out,
                   void* workspace, size_t workspace_bytes, int M, int HQ, int HKV, int D, int nsplit, void* stream) {
  if (M == 0) return TR_OK;
  // a chain's query rows of one kv head fit one workgroup's four 16-row tiles
  if (M < 0 || M > kAttnMaxM || HQ < 1 || HKV < 1 || (HQ / HKV) * M > 16 * kAttnWaves) return TR_ERR_SHAPE;
  return attn_decode_launch(q, qkv, ld, k_cache, v_cache, k_scale, v_scale, maxlen, pos, out, workspace,
                            workspace_bytes, M, HQ, HKV, D, nsplit, nullptr, stream);
}

int tr_attn_prep_tree(const void* qkv, int ld, const void* q_norm_w, const void* k_norm_w, const void* cos,
                      const void* sin, int rotary_dim, const int64_t* pos, const int32_t* parent, void* k_cache,
                      void* v_cache, float* k_scale, float* v_scale, int maxlen, void* q_out, int M, int HQ, int HKV,
                      int D, float eps, void* stream) {
  if (M == 0) return TR_OK;
  if (M < 0 || M > kAttnMaxTree) return TR_ERR_SHAPE;
  if (!parent) return TR_ERR_ARG;
  return attn_prep_launch(qkv, ld, q_norm_w, k_norm_w, cos, sin, rotary_dim, pos, k_cache, v_cache, k_scale, v_scale,
                          maxlen, q_out, M, HQ, HKV, D, eps, parent, stream);
}

int tr_attn_decode_tree(const void* q, const void* qkv, int ld, const void* k_cache, const void* v_cache,
                        const float* k_scale, const float* v_scale, int maxlen, const int64_t* pos,
                        const int32_t* parent, void* out, void* workspace, size_t workspace_bytes, int M, int HQ,
                        int HKV, int D, int nsplit, void* stream) {
  if (M == 0) return TR_OK;
  if (M < 0 || M > kAttnMaxTree) return TR_ERR_SHAPE;
  if (!parent) return TR_ERR_ARG;
  return attn_decode_launch(q, qkv, ld, k_cache, v_cache, k_scale, v_scale, maxlen, pos, out, workspace,
                            workspace_bytes, M, HQ, HKV, D, nsplit, parent, stream);
}

}  // extern "C"
