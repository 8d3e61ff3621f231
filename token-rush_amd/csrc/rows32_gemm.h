// The verify GEMM for 17 to 32 rows (a draft tree) and 24 < K / 128 <= 40: int4_gemm.hip includes this after
// tile_mac and GemmArgs.
//
// The work split of int4_gemm_kernel at two row tiles, sized so that these K need no second K slot: a wave holds
// GW = 4 or 5 groups of x for all 32 rows (128 or 160 VGPRs), eight waves (two per SIMD, 256 VGPRs each) cover
// 40 groups, and one strip's tiles are in flight, each group's refilled for the next strip as soon as it is
// dequantized. int4_gemm_kernel's 12 waves of two groups cover 24, so K = 5120 took two slots there: half the
// groups per workgroup and twice the strips, each batch of strips with its barrier and sum, then the slots'
// fp32 partials written, read and added. Bound as that kernel is, by the instructions and waits of a strip (MFMA
// and VALU of a SIMD's waves hardly overlap), not by memory. M = 32, us (graph of launches), before -> now:
// gate/up 34816 x 5120 with silu 36.0 -> 28.6, 14336 x 5120 18.1 -> 16.1, 16384 x 5120 19.9 -> 17.0, 7168 x 5120
// 12.4 -> 11.9, 248320 x 5120 218 -> 170; 16384 x 4096 (GW = 4) 17.3 -> 13.7, with GW = 5 15.6.
// Not taken outside the range: at K <= 3072 int4_gemm_kernel already has one slot and more waves (8192 x 2048
// 7.1 against 8.2-9.2, 12288 x 3072 10.0 / 10.7-12.5), and callers of partials want the slots (5120 x 6144 9.5
// at 3 slots against 9.9-11.1, 5120 x 17408 17.5 / 18.1-18.2). Also measured and not kept: x staged in LDS step
// by step and the waves spread over strips instead of K (40 us for gate/up: an operand read per MFMA, the
// staging and a barrier per step).
#pragma once

namespace tr {

constexpr int kWideWaves = 8;  // waves of a workgroup, at most, and of a CU

template <int GW, bool F16S>
__global__ __launch_bounds__(64 * kWideWaves) void rows32_gemm_kernel(GemmArgs a) {
  constexpr int MT = 2;
  extern __shared__ __attribute__((aligned(16))) float red[];  // [2][RB][W][MT][64][4]; first 8 KiB per wave: x staging
  const int G = a.K / kGroup, Gp = padded_groups(a.K);
  const int W = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, i = lane & 15, o = lane >> 4;
  const int rbi = blockIdx.x;  // takes strips rbi, rbi + gn, ..
  const int nr = rbi < a.rfull ? a.R : a.R - 1;
  const int gbase = wave * GW;  // every wave has a block: W = ceil(G / GW)
  const uint32_t kExp128 = vgpr_const(0x43004300u);

  // Groups past the packed row and strips past the range load from offset wbytes, beyond the resource: zeros.
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a.packed, (short)0, a.wbytes, 0x00020000);
  u32x4 w[GW];
  uint32_t sm[GW];
  auto load_tile = [&](int gw, int r) {
    const int g = gbase + gw, q = (g >> 2) * kQuadBytes;
    const bool on = r < nr && g < Gp;
    const int base = (rbi + r * a.gn) * a.quad_stride + q;
    sm[gw] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, kSmOff + 16 * i, on ? base + 4 * (g & 3) : a.wbytes, 2 /* nt */);
    w[gw] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, 16 * lane, on ? base + kCodeBytes * (g & 3) : a.wbytes, 2);
  };

  // x: per group eight loads of four rows (lane: row lane / 16, 16-byte chunk lane % 16), all issued before any
  // weight, then group by group through this wave's 8 KiB of LDS into the operand layout (row r's chunk c in
  // slot c ^ r % 16). Rows >= M load zeros; groups past K repeat the last one and meet zero parameters.
  const auto xrs = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, (short)0, a.M * a.K * 2, 0x00020000);
  u32x4 xv[GW][8];
#pragma unroll
  for (int gw = 0; gw < GW; ++gw) {
    const int g = min(gbase + gw, G - 1);
#pragma unroll
    for (int m = 0; m < 8; ++m)
      xv[gw][m] = __builtin_amdgcn_raw_buffer_load_b128(xrs, (4 * m + o) * a.K * 2 + 16 * i, g * 256, 0);
  }
  __builtin_amdgcn_s_barrier();  // every wave's x requests ahead of any wave's weights
#pragma unroll
  for (int gw = 0; gw < GW; ++gw) load_tile(gw, 0);
  __builtin_amdgcn_sched_barrier(0);
  uint4 xa[GW][MT][4];
  char* const stage = (char*)red + wave * 8192;
#pragma unroll
  for (int gw = 0; gw < GW; ++gw) {
#pragma unroll
    for (int m = 0; m < 8; ++m)
      *(u32x4*)(stage + (4 * m + o) * 256 + ((i ^ (4 * m + o)) & 15) * 16) = xv[gw][m];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j) xa[gw][mt][j] = *(const uint4*)(stage + (16 * mt + i) * 256 + (((4 * j + o) ^ i) & 15) * 16);
    __builtin_amdgcn_sched_barrier(0);
  }
  lds_barrier();  // every wave's staging reads before any ring write

  // Group sums of x in the A-operand layout of the min term's 16 x 16 x 4 MFMAs (int4_gemm_kernel's selector
  // MFMAs): groups 0-3 in the four k slots, group 4 in slot 0 of a second one.
  float Xa[MT], Xb[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    f32x4 D[GW];
#pragma unroll
    for (int gw = 0; gw < GW; ++gw) {
      const uint32_t one = (i >> 2) == (gw & 3) ? 0x3F803F80u : 0u;
      const bf16x8 A = __builtin_bit_cast(bf16x8, make_uint4(one, one, one, one));
      D[gw] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        D[gw] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, __builtin_bit_cast(bf16x8, xa[gw][mt][j]), D[gw], 0, 0, 0);
    }
    Xa[mt] = D[0][0];
#pragma unroll
    for (int gw = 1; gw < (GW < 4 ? GW : 4); ++gw) Xa[mt] += D[gw][0];
    Xb[mt] = D[GW - 1][0];
  }
  const StripWalk walk16(threadIdx.x, 4, blockDim.x, a.M, a.magicM), walk8(threadIdx.x, 3, blockDim.x, a.M, a.magicM);
  auto c1_of = [&](uint32_t p) { return fmaf(-128.f, sm_scale<F16S>(p), sm_min<F16S>(p)); };

  const int RB = a.RB;
  int sib = 0, half = 0;  // position in the current batch, ring half (wave-uniform)
  for (int r = 0; r < nr; ++r) {
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint32_t pa = 0, pb = 0;  // the parameters of this lane's group slot o, and of group 4
#pragma unroll
    for (int gw = 0; gw < GW; ++gw) {
      tile_mac<MT, F16S>(make_uint4(w[gw].x, w[gw].y, w[gw].z, w[gw].w), sm[gw], xa[gw], acc, kExp128);
      if (gw < 4) pa = o == gw ? sm[gw] : pa;
      else pb = sm[gw];
      load_tile(gw, r + 1);
    }
    const float ca = c1_of(pa), cb = GW > 4 && o == 0 ? c1_of(pb) : 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(Xa[mt], ca, acc[mt], 0, 0, 0);
      if (GW > 4) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(Xb[mt], cb, acc[mt], 0, 0, 0);
    }
    float* ring = red + (size_t)half * RB * W * MT * 256;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) *(f32x4*)(ring + ((size_t)(sib * W + wave) * MT + mt) * 256 + lane * 4) = acc[mt];
    if (sib < RB - 1 && r < nr - 1) {
      ++sib;
      continue;
    }
    lds_barrier();
    const int ns = sib + 1, r_first = r - sib;
    // Sum over the waves' partial tiles, in wave order, of output (m, n16) of strip r_first + sidx.
    auto wave_sum = [&](int sidx, int m, int n16) {
      const int mt = m >> 4, mm = m & 15;
      const float* src = ring + ((size_t)sidx * W * MT + mt) * 256 + (16 * (mm >> 2) + n16) * 4 + (mm & 3);
      float part[kWideWaves];
#pragma unroll
      for (int k = 0; k < kWideWaves; ++k) part[k] = k < W ? src[(size_t)k * MT * 256] : 0.f;
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < kWideWaves; ++k)
        if (k < W) v += part[k];
      return v;
    };
    if (a.silu) {
      // pair layout: rows 0..7 of a strip are gate rows, 8..15 the matching up rows
      const int F = a.N / 2, j = threadIdx.x & 7;
      for (StripWalk wk = walk8; wk.s < ns; wk.next()) {
        const float g = bf16_bits_to_f32(f32_to_bf16_bits(wave_sum(wk.s, wk.m, j)));
        const float u = bf16_bits_to_f32(f32_to_bf16_bits(wave_sum(wk.s, wk.m, j + 8)));
        ((uint16_t*)a.out)[(size_t)wk.m * F + 8 * (rbi + (r_first + wk.s) * a.gn) + j] = f32_to_bf16_bits(silu_mul_f32(g, u));
      }
    } else {
      const int n16 = threadIdx.x & 15;
      for (StripWalk wk = walk16; wk.s < ns; wk.next()) {
        const float v = wave_sum(wk.s, wk.m, n16);
        const int n = 16 * (rbi + (r_first + wk.s) * a.gn) + n16;
        ((uint16_t*)a.out)[(size_t)wk.m * a.N + n] = f32_to_bf16_bits(v);
      }
    }
    sib = 0;
    half ^= 1;
  }
}

}  // namespace tr
