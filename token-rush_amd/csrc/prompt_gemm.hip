// int4 group-128 GEMM for prompts: T > 32 activation rows, y[t, n] = sum_k x[t, k] (q[n, k] s + mn).
//
// The reference dequantizes the weight and calls a dense matmul here (tokenrush/quant.py:373-374). For a few
// hundred rows that is mostly the dense copy (2 N K bytes written and read back), so this kernel feeds the
// codes to the matrix cores as the verify GEMM does (int4_gemm.hip): a code becomes the bf16 value 128 + q
// with one v_and_or_b32, E = sum x (128 + q) per group on v_mfma_f32_32x32x16_bf16, acc += s E in fp32, and
// the (mn - 128 s) sum(x) term comes from two v_mfma_f32_32x32x2_f32 per four groups, with the sums of x made
// once per call by group_sums_kernel. No weight is rounded to bf16.
//
// Work split: a workgroup of eight waves owns 32 MB activation rows (MB = 2..4) and eight 16-row weight
// strips. Waves w and w + 4 hold the same two strips and the two halves of the workgroup's K range: each
// 32 x 16 activation operand read from LDS meets 32 weight rows, and two waves share each SIMD, so one's
// dequantization can run under the other's MFMAs. Per step each half's next group of x (32 MB x 256 bytes)
// goes through registers into the other of two LDS buffers (rows of sixteen 16-byte chunks, chunk c in
// slot c ^ row % 16, so the 16 rows of an operand read fall in different banks); weights arrive two to four
// steps ahead, straight in the B-operand layout. The halves add their sums through LDS at the end.
//
// Whole rounds of 256 workgroups take the full K. The blocks left over (all of them for small N) split K
// over S workgroups, so that they fill the chip too; those write fp32 partials and a second kernel adds
// the slots in order.
//
// What bounds it: the step. At 64 rows of 34816 x 5120 a step of two groups takes 2.2 us where its MFMAs take
// 0.4 (rocprofv3: MFMA busy 22%, 44% of wave cycles in s_waitcnt, 30% waiting to issue, no bank conflicts):
// the x tile's L2 latency and the barrier are paid per step. Measured, us, against the dense path (bf16 copy
// and library matmul): 34816 x 5120 53 / 178 at 64 rows, 67 / 183 at 96, 89 / 189 at 128, 150 / 200 at 256;
// 5120 x 17408 32 / 126, 38 / 135, 50 / 148, 81 / 214. The same tile on v_mfma_f32_16x16x32_bf16 measured
// the same within 5% (58, 72, 91, 151); loads left to the scheduler, which moves them down to the barrier
// that waits for them, 56, 72, 98, 163.
#include "int4_layout.h"

#include <atomic>

namespace tr {

constexpr int kPromptStrips = 8;  // strips per workgroup

enum { PROMPT_ROWS = 0, PROMPT_PAIRS = 1, PROMPT_SILU = 2 };

struct PromptArgs {
  const uint16_t* x;      // bf16 [T, K]
  const uint8_t* packed;  // quad layout
  const float* xsum;      // fp32 [T, Gp]: sums of x over each group
  uint16_t* out;          // bf16 [T, N], or [T, N / 2] (silu)
  float* part;            // fp32 [S, T, tail_n]: the split blocks' partials
  int T, N, K, nq, quad_stride, wbytes;
  int nfull, S, Ty, tail_n, mode;
};

// xsum[t, g] = sum of x over group g (0 for padding groups). One wave per row and four groups.
__global__ __launch_bounds__(256) void group_sums_kernel(const uint16_t* __restrict__ x, float* __restrict__ xsum,
                                                         int K, int Gp) {
  const int lane = threadIdx.x & 63, t = blockIdx.y;
  const int g = 4 * (blockIdx.x * 4 + (threadIdx.x >> 6)) + (lane >> 4);
  if (g >= Gp) return;
  float v[8], s = 0.f;
  unpack8(g < K / kGroup ? *(const uint4*)(x + (size_t)t * K + g * kGroup + 8 * (lane & 15)) : make_uint4(0, 0, 0, 0), v);
#pragma unroll
  for (int e = 0; e < 8; ++e) s += v[e];
  s += dpp_mov<0xB1>(s);
  s += dpp_mov<0x4E>(s);
  s += dpp_mov<0x124>(s);
  s = sum_x8(s);
  if ((lane & 15) == 0) xsum[(size_t)t * Gp + g] = s;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int MB, bool F16S>
__global__ __launch_bounds__(512) void prompt_gemm_kernel(PromptArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];  // [2 buffers][2 halves][32 MB rows][256 bytes]
  constexpr int kRows = 32 * MB, kHalf = kRows * 256, kBuf = 2 * kHalf, kLoads = 2 * MB;
  constexpr int kAhead = MB <= 2 ? 4 : 2;  // steps between a weight load and its use
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int kp = wave >> 2, nw = wave & 3, i = lane & 15, up = lane >> 5;

  // Workgroup -> (block, row tile, K slot). Row tiles of one block sit eight workgroups apart, on one XCD,
  // whose L2 then serves the block's weights to all of them.
  int block, y, slot = 0, S = 1;
  {
    int id = blockIdx.x, first = 0, blocks = a.nfull;
    if (id >= a.nfull * a.Ty) {
      id -= a.nfull * a.Ty;
      first = a.nfull;
      blocks = (a.N / 16 + kPromptStrips - 1) / kPromptStrips - a.nfull;
      S = a.S;
      slot = id / (blocks * a.Ty);
      id -= slot * blocks * a.Ty;
    }
    const int band = id / (8 * a.Ty), width = min(8, blocks - 8 * band), r = id - band * 8 * a.Ty;
    y = r / width;
    block = first + 8 * band + (r - y * width);
  }
  const int row0 = y * kRows;
  // this half's quads, and the steps the workgroup runs (both halves stage together)
  const int p0 = 2 * slot + kp, q0 = p0 * a.nq / (2 * S), q1 = (p0 + 1) * a.nq / (2 * S);
  const int pa = 2 * slot * a.nq / (2 * S), pb = (2 * slot + 1) * a.nq / (2 * S), pc = (2 * slot + 2) * a.nq / (2 * S);
  const int Lq = max(pb - pa, pc - pb);

  const auto xrs = __builtin_amdgcn_make_buffer_rsrc((void*)(a.x + (size_t)row0 * a.K), (short)0, (a.T - row0) * a.K * 2,
                                                     0x00020000);  // rows past T read as zeros
  const auto wrs = __builtin_amdgcn_make_buffer_rsrc((void*)a.packed, (short)0, a.wbytes, 0x00020000);
  const int G = a.K / kGroup;
  const int srow = (threadIdx.x & 255) >> 4, schunk = threadIdx.x & 15;
  const int svoff = srow * a.K * 2 + schunk * 16;
  char* const sdst = lds + kp * kHalf + srow * 256 + ((schunk ^ srow) & 15) * 16;
  const char* const xsrc = lds + kp * kHalf + (lane & 31) * 256;

  u32x4 xv[kLoads];
  auto stage_load = [&](int step) {
    const int g = min(4 * q0 + step, G - 1);
#pragma unroll
    for (int m = 0; m < kLoads; ++m) xv[m] = __builtin_amdgcn_raw_buffer_load_b128(xrs, svoff + m * 32 * a.K, g * 256, 0);
  };
  auto stage_store = [&](int buf) {
#pragma unroll
    for (int m = 0; m < kLoads; ++m) *(u32x4*)(sdst + buf * kBuf + m * 4096) = xv[m];
  };
  const int strip0 = block * kPromptStrips + 2 * nw, nstrips = a.N / 16;
  // strips and quads past the range load from offset wbytes, beyond the resource: zeros, no memory access
  // (never from further on: the range check subtracts the scalar offset from the size)
  const uint32_t oob = a.wbytes;
  const uint32_t sbase[2] = {strip0 < nstrips ? (uint32_t)strip0 * a.quad_stride : oob,
                             strip0 + 1 < nstrips ? (uint32_t)(strip0 + 1) * a.quad_stride : oob};
  auto quad_off = [&](int s, int q) { return (int)(q < q1 ? min(sbase[s] + (uint32_t)q * kQuadBytes, oob) : oob); };
  u32x4 w[kAhead][2], sm, smn;
  auto weight_load = [&](u32x4 (&d)[2], int step) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
      d[s] = __builtin_amdgcn_raw_buffer_load_b128(wrs, 16 * lane + (step & 3) * kCodeBytes, quad_off(s, q0 + (step >> 2)), 2);
  };
  // a lane's column is row i of strip (lane / 16) % 2; the last block's second strip may not exist
  const int pstep = (lane & 16) ? (strip0 + 1 < nstrips ? a.quad_stride : a.wbytes) : 0;
  auto param_load = [&](int q) {
    return __builtin_amdgcn_raw_buffer_load_b128(wrs, kSmOff + 16 * i + pstep, quad_off(0, q), 2);
  };

  f32x16 acc[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) acc[m] = f32x16{};
  const uint32_t kExp128 = vgpr_const(0x43004300u), kMask = 0x000F000Fu;

  stage_load(0);
  sm = param_load(q0);
#pragma unroll
  for (int t = 0; t < kAhead; ++t) weight_load(w[t], t);
  stage_store(0);
  lds_barrier();
  for (int qi = 0; qi < Lq; ++qi) {
    float xa[MB][2];  // A operands of the min term: row lane % 32, groups up and 2 + up of the quad
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int step = 4 * qi + t;
      stage_load(step + 1);
      if (t == 2) {
        smn = param_load(q0 + qi + 1);
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          const float* xs = a.xsum + (size_t)min(row0 + 32 * m + (lane & 31), a.T - 1) * (a.nq * kQuad) +
                            4 * min(q0 + qi, a.nq - 1) + up;
          xa[m][0] = xs[0];
          xa[m][1] = xs[2];
        }
      }
      // Without this the scheduler moves the loads down to their first use, right before the barrier that
      // waits for them.
      __builtin_amdgcn_sched_barrier(0);
      // The two strips' words with odd lane rows of one and even lane rows of the other exchanged are the
      // 32-column B operand: columns 0-15 strip 0, 16-31 strip 1, k octets 0 and 2 (then 1 and 3) of 32 j.
      bf16x8 b[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const auto r = __builtin_amdgcn_permlane16_swap(w[t % kAhead][0][j], w[t % kAhead][1][j], false, false);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t c = r[h];
          b[2 * j + h] = __builtin_bit_cast(bf16x8, u32x4{(c & kMask) | kExp128, ((c >> 4) & kMask) | kExp128,
                                                          ((c >> 8) & kMask) | kExp128, ((c >> 12) & kMask) | kExp128});
        }
      }
      const float sf = sm_scale<F16S>(sm[t]);
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        f32x16 E = {};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int chunk = 4 * (q >> 1) + (q & 1) + 2 * up;
          const bf16x8 xo = *(const bf16x8*)(xsrc + (t & 1) * kBuf + m * 8192 + ((chunk ^ i) & 15) * 16);
          E = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xo, b[q], E, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][r] = fmaf(sf, E[r], acc[m][r]);
      }
      if (t == 3) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t p = up ? sm[2 * h + 1] : sm[2 * h];
          const float c1 = fmaf(-128.f, sm_scale<F16S>(p), sm_min<F16S>(p));  // mn - 128 s: removes the code offset
#pragma unroll
          for (int m = 0; m < MB; ++m) acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[m][h], c1, acc[m], 0, 0, 0);
        }
      }
      weight_load(w[t % kAhead], step + kAhead);
      stage_store((t + 1) & 1);  // read two steps ago, before the last barrier
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
    sm = smn;
  }

  // The halves trade: of every 32-row block the wave of half kp finishes registers 8 kp .. 8 kp + 7 (rows
  // 16 kp ..) with its partner's sums of them, half 0's first.
  char* const xch = lds + wave * MB * 2048 + lane * 16;
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = kp ? acc[m][4 * h + r] : acc[m][8 + 4 * h + r];
      *(f32x4*)(xch + (2 * m + h) * 1024) = v;
    }
  lds_barrier();
  const char* const peer = lds + (wave ^ 4) * MB * 2048 + lane * 16;
  const int strip = strip0 + ((lane >> 4) & 1);
  if (strip >= nstrips) return;
  const int F = a.N / 2;
#pragma unroll
  for (int m = 0; m < MB; ++m) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 theirs = *(const f32x4*)(peer + (2 * m + h) * 1024);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = kp ? theirs[r] + acc[m][8 + 4 * h + r] : acc[m][4 * h + r] + theirs[r];
        const int row = row0 + 32 * m + 16 * kp + 8 * h + 4 * up + r;
        const bool live = row < a.T;
        if (S > 1) {
          if (live) a.part[((size_t)slot * a.T + row) * a.tail_n + 16 * strip + i - 16 * kPromptStrips * a.nfull] = v;
        } else if (a.mode == PROMPT_SILU) {
          const float vb = bf16_bits_to_f32(f32_to_bf16_bits(v)), u = dpp_mov<0x128>(vb);  // lane i ^ 8: the up row
          if (live && i < 8) a.out[(size_t)row * F + 8 * strip + i] = f32_to_bf16_bits(silu_mul_f32(vb, u));
        } else {
          const int col = a.mode == PROMPT_ROWS ? 16 * strip + i : i < 8 ? 8 * strip + i : F + 8 * strip + i - 8;
          if (live) a.out[(size_t)row * a.N + col] = f32_to_bf16_bits(v);
        }
      }
    }
  }
}

// The split blocks' slots in order: four columns per thread (silu: four outputs from two fours).
__global__ __launch_bounds__(256) void prompt_sum_kernel(const float* __restrict__ part, uint16_t* __restrict__ out, int S,
                                                         int T, int N, int n0, int tail_n, int mode) {
  const int per = mode == PROMPT_SILU ? tail_n / 8 : tail_n / 4;  // fours per row
  const int q = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
  if (q >= per) return;
  // silu: four q holds outputs 4 q .. of this tail: strip q / 2, gate columns 4 (q % 2) ..
  const int c = mode == PROMPT_SILU ? 16 * (q >> 1) + 4 * (q & 1) : 4 * q;
  const float* p = part + (size_t)t * tail_n + c;
  float4 g = make_float4(0.f, 0.f, 0.f, 0.f), u = g;
  for (int s = 0; s < S; ++s, p += (size_t)T * tail_n) {
    const float4 v = *(const float4*)p;
    g.x += v.x; g.y += v.y; g.z += v.z; g.w += v.w;
    if (mode == PROMPT_SILU) {
      const float4 z = *(const float4*)(p + 8);
      u.x += z.x; u.y += z.y; u.z += z.z; u.w += z.w;
    }
  }
  uint32_t lo = f32x2_to_bf16x2_bits(g.x, g.y), hi = f32x2_to_bf16x2_bits(g.z, g.w);
  const int F = N / 2, n = n0 + c;
  size_t at = (size_t)t * N + n;
  if (mode != PROMPT_ROWS) {
    const int strip = n >> 4, j = n & 15;
    at = mode == PROMPT_SILU ? (size_t)t * F + 8 * strip + j : (size_t)t * N + (j < 8 ? 8 * strip + j : F + 8 * strip + j - 8);
  }
  if (mode == PROMPT_SILU) {
    const uint32_t ul = f32x2_to_bf16x2_bits(u.x, u.y), uh = f32x2_to_bf16x2_bits(u.z, u.w);
    auto act = [](uint32_t gb, uint32_t ub) { return silu_mul_f32(bf16_bits_to_f32(gb & 0xFFFFu), bf16_bits_to_f32(ub & 0xFFFFu)); };
    lo = f32x2_to_bf16x2_bits(act(lo, ul), act(lo >> 16, ul >> 16));
    hi = f32x2_to_bf16x2_bits(act(hi, uh), act(hi >> 16, uh >> 16));
  }
  *(uint2*)(out + at) = make_uint2(lo, hi);
}

}  // namespace tr

using namespace tr;

namespace {

constexpr int kPromptCUs = 256, kPromptMaxS = 16;

struct PromptPlan {
  int MB, Ty, blocks, nfull, S, tail_n;
  size_t sums, part;  // workspace bytes
};

bool prompt_plan(int T, int N, int K, PromptPlan* p) {
  // 32-bit buffer offsets into x
  if (!shape_ok(N, K) || T < 33 || (size_t)T * K * 2 >= ((size_t)1 << 31) || T > 65535) return false;
  const int nq = padded_groups(K) / kQuad;
  p->Ty = (T + 127) / 128;
  p->MB = ((T + p->Ty - 1) / p->Ty + 31) / 32;
  p->Ty = (T + 32 * p->MB - 1) / (32 * p->MB);
  p->blocks = (N / 16 + kPromptStrips - 1) / kPromptStrips;
  // whole rounds of one workgroup per CU, then the rest split over K (two halves per workgroup, each at
  // least one quad) to fill the chip
  p->nfull = p->blocks * p->Ty / kPromptCUs * kPromptCUs / p->Ty;
  const int tail = p->blocks - p->nfull;
  p->S = 1;
  if (tail > 0) {
    int S = kPromptCUs / (tail * p->Ty);
    if (S > kPromptMaxS) S = kPromptMaxS;
    if (S > nq / 2) S = nq / 2;
    if (S > 1) {
      const int L = (nq + 2 * S - 1) / (2 * S);
      p->S = (nq + 2 * L - 1) / (2 * L);
    }
  }
  if (p->S == 1) p->nfull = p->blocks;
  p->tail_n = N - p->nfull * 16 * kPromptStrips;
  p->sums = ((size_t)T * nq * kQuad * sizeof(float) + 255) / 256 * 256;
  p->part = p->S > 1 ? (size_t)p->S * T * p->tail_n * sizeof(float) : 0;
  return true;
}

template <int MB, bool F16S>
hipError_t prompt_launch(const PromptArgs& a, int grid, hipStream_t stream) {
  constexpr int kLds = 2 * 2 * 32 * MB * 256;
  static std::atomic<uint64_t> raised{0};  // devices on which the kernel's LDS limit is raised
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  if (!(raised.load(std::memory_order_relaxed) & bit)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prompt_gemm_kernel<MB, F16S>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) return e;
    raised.fetch_or(bit, std::memory_order_relaxed);
  }
  hipLaunchKernelGGL((prompt_gemm_kernel<MB, F16S>), dim3(grid), dim3(512), kLds, stream, a);
  return hipGetLastError();
}

template <bool F16S>
hipError_t prompt_launch_mb(int MB, const PromptArgs& a, int grid, hipStream_t stream) {
  if (MB == 2) return prompt_launch<2, F16S>(a, grid, stream);
  if (MB == 3) return prompt_launch<3, F16S>(a, grid, stream);
  return prompt_launch<4, F16S>(a, grid, stream);
}

}  // namespace

extern "C" {

size_t tr_prompt_workspace_bytes(int T, int N, int K) {
  PromptPlan p;
  return prompt_plan(T, N, K, &p) ? p.sums + p.part : 0;
}

int tr_int4_gemm_prompt(const void* x, const void* packed, void* out, void* workspace, size_t workspace_bytes, int T,
                        int N, int K, int group, int scale_dtype, int mode, void* stream) {
  if (group != kGroup) return TR_ERR_CONFIG;
  PromptPlan p;
  if (!prompt_plan(T, N, K, &p) || (mode != PROMPT_ROWS && N % 32)) return TR_ERR_SHAPE;
  if (!x || !packed || !out || !workspace || workspace_bytes < p.sums + p.part) return TR_ERR_ARG;
  if ((scale_dtype != 0 && scale_dtype != 1) || mode < PROMPT_ROWS || mode > PROMPT_SILU) return TR_ERR_ARG;
  if ((uintptr_t)x % 16 || (uintptr_t)workspace % 16 || (uintptr_t)out % 8) return TR_ERR_ARG;
  const int Gp = padded_groups(K);
  PromptArgs a;
  a.x = (const uint16_t*)x;
  a.packed = (const uint8_t*)packed;
  a.xsum = (const float*)workspace;
  a.out = (uint16_t*)out;
  a.part = (float*)((char*)workspace + p.sums);
  a.T = T;
  a.N = N;
  a.K = K;
  a.nq = Gp / kQuad;
  a.quad_stride = a.nq * kQuadBytes;
  a.wbytes = (int)packed_bytes(N, K);
  a.nfull = p.nfull;
  a.S = p.S;
  a.Ty = p.Ty;
  a.tail_n = p.tail_n;
  a.mode = mode;
  const hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(group_sums_kernel, dim3((a.nq + 3) / 4, T), dim3(256), 0, st, a.x, (float*)workspace, K, Gp);
  if (hipGetLastError() != hipSuccess) return TR_ERR_LAUNCH;
  const int grid = (p.nfull + (p.blocks - p.nfull) * p.S) * p.Ty;
  const hipError_t e = scale_dtype == 1 ? prompt_launch_mb<true>(p.MB, a, grid, st) : prompt_launch_mb<false>(p.MB, a, grid, st);
  if (e != hipSuccess) return TR_ERR_LAUNCH;
  if (p.S > 1) {
    const int per = mode == PROMPT_SILU ? p.tail_n / 8 : p.tail_n / 4;
    hipLaunchKernelGGL(prompt_sum_kernel, dim3((per + 255) / 256, T), dim3(256), 0, st, a.part, a.out, p.S, T, N,
                       N - p.tail_n, p.tail_n, mode);
    if (hipGetLastError() != hipSuccess) return TR_ERR_LAUNCH;
  }
  return TR_OK;
}

}  // extern "C"
