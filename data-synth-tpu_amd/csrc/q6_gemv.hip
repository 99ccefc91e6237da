// Decode-fused skinny GEMM for packed Q6_K projections: y = x @ decode(W)^T.
//
// Replaces the Pallas kernel packed_q6_k_projection (kaggle/packed_q6/kernel.py:65-148).
// Each wave decodes a 16-row x 256-K unit of the SoA tile straight into MFMA
// A operands (no LDS round trip, no materialised weights) and multiplies it
// with up to 16*NT tokens on v_mfma_f32_16x16x32_bf16 (FP32 accumulation).
// The K blocks of a 16-row group are spread over the waves of one workgroup
// and reduced through LDS in a fixed wave order, so results are deterministic.
#include "moe_tile.h"
#include "q6moe_api.h"
#include "q6moe_device.h"

namespace q6moe {

// Eight BF16 x values for lane (token row ``xr``) at element ``col`` of a row,
// zero beyond ``k`` (the reference zero-pads x to whole 256-blocks).
__device__ __forceinline__ u32x4 load_x8(const uint16_t* xr, int col, int k, int vec) {
  if (vec && col + 8 <= k) return *reinterpret_cast<const u32x4*>(xr + col);
  u32x4 v = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t e = (col + i < k) ? (uint32_t)xr[col + i] : 0u;
    v[i >> 1] |= e << (16 * (i & 1));
  }
  return v;
}

template <int NT>
__global__ void __launch_bounds__(512) q6_skinny_kernel(const uint16_t* __restrict__ x, int m, int k,
                                                        int64_t ldx, int xvec,
                                                        const uint8_t* __restrict__ data,
                                                        const uint8_t* __restrict__ scales, int n,
                                                        int kb_count, int kw, void* __restrict__ y,
                                                        int ybf16, int64_t ldy) {
  __shared__ float red[8][NT][256];
  const int rgg = blockIdx.x;
  const int tile = rgg >> 2, rg = rgg & 3;
  const int m0 = blockIdx.y * 16 * NT;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int jA = lane >> 4, j = lane & 15;
  const int row = rg * 16 + j;

  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int kb = wave; kb < kb_count; kb += kw) {
    const int64_t t = (int64_t)tile * kb_count + kb;
    Q6Raw raw;
    q6_load(raw, data + t * kTileBytes, scales + t * 128, row, jA);
    u32x4 xf[NT][8];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int gm = m0 + nt * 16 + j;
#pragma unroll
      for (int f = 0; f < 8; ++f) {
        xf[nt][f] = gm < m ? load_x8(x + (int64_t)gm * ldx, kb * kQK + q6_xfrag_offset(f, jA), k, xvec)
                           : u32x4{0u, 0u, 0u, 0u};
      }
    }
    u32x4 a[8];
    q6_decode_unit(raw, jA, a);
#pragma unroll
    for (int f = 0; f < 8; ++f) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma16(a[f], xf[nt][f], acc[nt]);
    }
  }

#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][nt][lane * 4 + i] = acc[nt][i];
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < NT * 256; idx += blockDim.x) {
    const int nt = idx >> 8, e = idx & 255;
    float s = 0.f;
    for (int w = 0; w < kw; ++w) s += red[w][nt][e];
    const int ln = e >> 2, i = e & 3;
    const int gn = tile * kTileRows + rg * 16 + 4 * (ln >> 4) + i;
    const int gm = m0 + nt * 16 + (ln & 15);
    if (gn < n && gm < m) {
      if (ybf16)
        reinterpret_cast<uint16_t*>(y)[(int64_t)gm * ldy + gn] = bf16_bits(s);
      else
        reinterpret_cast<float*>(y)[(int64_t)gm * ldy + gn] = s;
    }
  }
}

// ---------------------------------------------------------------------------
// Many tokens: 64 tokens x 64 rows (one SoA row tile) per workgroup. The skinny
// kernel above reads a unit's 64 token rows again from L2 for every 16 output
// rows (32 KB per 3.3 KB of weights), which bounds it; here the four row groups
// of a tile share them through LDS. A workgroup is KS sets of 4 waves that split
// the K blocks; wave (set, rg) decodes row group rg's units straight into MFMA
// operands, its next K block's bytes in flight in a second register set. Each
// set's token rows of a K half (64 x 128 BF16, XOR-swizzled so that an operand
// read touches every bank once) are double-buffered in LDS by buffer->LDS DMA;
// columns past K and rows past m arrive as zeros (their lanes address past the
// buffer's end; m > 16, so that the wave-uniform part of an address, at most one
// row and 12 rows on, stays inside). The sets' sums meet in LDS in set order.
// Bound by waiting, with about one workgroup per CU: 777 tokens, 2560 -> 1280 (260
// workgroups), the vector ALU issues in 38 % of a SIMD's cycles (232 instructions
// of decode per unit and 64 tokens), the matrix cores work in 15 %, and a wave
// spends 49 % of its time waiting, mostly for a half's DMA and the next weights,
// issued one step before. 49.0 -> 20.3 us (251 TFLOP/s); 1024 tokens, 4096 -> 4096:
// 294 -> 67.6 us (508 TFLOP/s).
// ---------------------------------------------------------------------------
namespace pj {

constexpr int kTok = 64;                      // tokens per workgroup
constexpr int kCg = kTok / 16;
constexpr int kHalf = kTok * 128 * 2;         // LDS bytes of a K half of the token tile
constexpr int kNoRow = (int)0x80000000u;      // a buffer offset past any x taken here

struct Raw {
  u32x4 ql[2], qh[2], sc;
  uint32_t d;
  __device__ __forceinline__ void load(const uint8_t* tile, const uint8_t* dplane, int row, int jA) {
    const uint8_t* l = tile + kQlOff + row * 128 + 16 * jA;
    const uint8_t* h = tile + kQhOff + row * 64 + 16 * (jA & 1);
    ql[0] = *reinterpret_cast<const u32x4*>(l);
    ql[1] = *reinterpret_cast<const u32x4*>(l + 64);
    qh[0] = *reinterpret_cast<const u32x4*>(h);
    qh[1] = *reinterpret_cast<const u32x4*>(h + 32);
    sc = *reinterpret_cast<const u32x4*>(tile + kScOff + row * 16);
    d = *reinterpret_cast<const uint16_t*>(dplane + row * 2);
  }
  // A fragment 2g + e of K half h (q6_decode_unit's fragment 4h + 2g + e):
  // columns 64g + 16jA + 8e + [0, 8) of the half
  __device__ __forceinline__ u32x4 frag(int h, int g, int e, int jA) const {
    const int sh = 2 * (jA >> 1);
    const float ds = half_bits_to_float(d) * (float)(int)(int8_t)((sc[2 * h + g] >> (8 * jA)) & 0xff);
    const uint32_t h0 = qh[h][2 * e] >> sh, h1 = qh[h][2 * e + 1] >> sh;
    const uint32_t l0 = ql[h][2 * e], l1 = ql[h][2 * e + 1];
    return g ? q6_frag_mix(q6_codes_hi(l0, h0), q6_codes_hi(l1, h1), ds, -1056.f * ds)
             : q6_frag_mix(q6_codes_lo(l0, h0), q6_codes_lo(l1, h1), ds, -1056.f * ds);
  }
};

}  // namespace pj

template <int KS>
__global__ void __launch_bounds__(256 * KS, 4) q6_tile_kernel(const uint16_t* __restrict__ x, int m, int k, int64_t ldx,
                                                           const uint8_t* __restrict__ data,
                                                           const uint8_t* __restrict__ scales, int n, int kbs,
                                                           void* __restrict__ y, int ybf16, int64_t ldy) {
  using namespace pj;
  using namespace pf;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int wave = wave_id(), lane = threadIdx.x & 63;
  const int ks = wave >> 2, rg = wave & 3;  // K set, row group (and quarter of the set's token DMA)
  const int j = lane & 15, jA = lane >> 4;
  const int64_t tile = blockIdx.x;
  const int m0 = blockIdx.y * kTok;
  const int kb0 = ks * kbs / KS, kb1 = (ks + 1) * kbs / KS;
  const int halves = (k + 127) >> 7, hend = 2 * kb1 < halves ? 2 * kb1 : halves;
  const int steps = 2 * ((kbs + KS - 1) / KS);  // of the longest set: every wave passes as many barriers
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(x), (short)0, (int)(uint32_t)((((int64_t)m - 1) * ldx + k) * 2), 0x00020000);
  uint8_t* const stages = smem + ks * 2 * kHalf;
  // DMA instruction i of this wave fills granules (rg*4 + i)*64 + lane: token
  // t = that/16, column granule (lane % 16) ^ (t % 16) = (j ^ jA) ^ 4i. Rows past
  // m lie past the buffer's end.
  const uint32_t row0 = opaque((uint32_t)(m0 + rg * 16 + jA) * (uint32_t)ldx * 2u);
  const uint32_t gran0 = opaque((uint32_t)((j ^ jA) * 16));
  auto dma = [&](int hs, int slot) {
    if (hs >= hend) return;
    const bool part = (hs + 1) * 128 > k;
#pragma unroll
    for (int i = 0; i < kCg; ++i) {
      const uint32_t gr = gran0 ^ (64u * i);
      uint32_t vo = row0 + gr;
      if (part && hs * 128 + (int)(gr >> 1) >= k) vo = (uint32_t)kNoRow;
      bdma16(xr, vo, (uint32_t)hs * 256u + (uint32_t)(8 * i) * (uint32_t)ldx,
             stages + slot * kHalf + (rg * kCg + i) * 1024);
    }
  };
  Raw w[2];
  auto load_w = [&](Raw& r, int kb) {
    const int64_t t = tile * kbs + kb;
    r.load(data + t * kTileBytes, scales + t * 128, rg * 16 + j, jA);
  };
  // a K block's sum is formed apart and then added to the running one, so that
  // no chain of FP32 additions is longer than the skinny kernel's
  f32x4 acc[kCg], sum[kCg];
#pragma unroll
  for (int t = 0; t < kCg; ++t) sum[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int s, auto slot_c, auto set_c) {
    constexpr int slot = decltype(slot_c)::value, set = decltype(set_c)::value;
    const int hs = 2 * kb0 + s;
    wait_vm<0>();                         // this step's share of the token tile, and its weights
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's reads of the other stage
    wg_barrier();
    dma(hs + 1, 1 - slot);
    if constexpr (slot == 0) {
      if (kb0 + (s >> 1) + 1 < kb1) load_w(w[1 - set], kb0 + (s >> 1) + 1);
    }
    if (hs < hend) {
      if constexpr (slot == 0) {
#pragma unroll
        for (int t = 0; t < kCg; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const u32x4 a = w[set].frag(slot, f >> 1, f & 1, jA);
#pragma unroll
        for (int tg = 0; tg < kCg; ++tg) {
          const u32x4 xv = *reinterpret_cast<const u32x4*>(
              stages + slot * kHalf + xgran(tg * 16 + j, 8 * (f >> 1) + 2 * jA + (f & 1)));
          acc[tg] = mfma16(a, xv, acc[tg]);
        }
      }
      if (slot == 1 || hs + 1 >= hend) {
#pragma unroll
        for (int t = 0; t < kCg; ++t) sum[t] += acc[t];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if (kb0 < kb1) load_w(w[0], kb0);
  dma(2 * kb0, 0);
  for (int s = 0; s < steps; s += 4) {
    step(s, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
    step(s + 1, std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{});
    if (s + 2 < steps) {
      step(s + 2, std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
      step(s + 3, std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
    }
  }
  __syncthreads();
  if (ks > 0) {
#pragma unroll
    for (int tg = 0; tg < kCg; ++tg)
      *reinterpret_cast<f32x4*>(smem + (((ks - 1) * 4 + rg) * kCg + tg) * 1024 + lane * 16) = sum[tg];
  }
  __syncthreads();
  if (ks > 0) return;
  const int gn = (int)tile * kTileRows + rg * 16 + 4 * jA;
  const bool vec = ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0 && gn + 4 <= n;
#pragma unroll
  for (int tg = 0; tg < kCg; ++tg) {
#pragma unroll
    for (int o = 0; o < KS - 1; ++o)
      sum[tg] += *reinterpret_cast<const f32x4*>(smem + ((o * 4 + rg) * kCg + tg) * 1024 + lane * 16);
    const int gm = m0 + tg * 16 + j;
    if (gm >= m) continue;
    const int64_t at = gm * ldy + gn;
    if (vec && ybf16) {
      *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(y) + at) =
          u32x2{pack_bf16x2(sum[tg][0], sum[tg][1]), pack_bf16x2(sum[tg][2], sum[tg][3])};
    } else if (vec) {
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(y) + at) = sum[tg];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (gn + i < n) {
          if (ybf16)
            reinterpret_cast<uint16_t*>(y)[at + i] = bf16_bits(sum[tg][i]);
          else
            reinterpret_cast<float*>(y)[at + i] = sum[tg][i];
        }
    }
  }
}

template <int KS>
static void launch_tile(const uint16_t* x, int m, int k, int64_t ldx, const uint8_t* data, const uint8_t* scales, int n,
                        int kb, void* y, int ybf16, int64_t ldy, hipStream_t s) {
  constexpr int lds = KS * 2 * pj::kHalf;
  static std::atomic<uint64_t> attr_done{0};
  once_per_device(attr_done, [] {
    (void)hipFuncSetAttribute((const void*)q6_tile_kernel<KS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  });
  hipLaunchKernelGGL(q6_tile_kernel<KS>, dim3((unsigned)cdiv(n, kTileRows), (unsigned)cdiv(m, pj::kTok)),
                     dim3(256 * KS), lds, s, x, m, k, ldx, data, scales, n, kb, y, ybf16, ldy);
}

}  // namespace q6moe

using namespace q6moe;

extern "C" int q6moe_q6_matmul(const uint16_t* x, int64_t m, int64_t k, int64_t ldx,
                               const uint8_t* data, const uint8_t* scales, int64_t n, void* y,
                               int y_dtype, int64_t ldy, void* stream) {
  Q6MOE_REQUIRE(x && data && scales && y, "q6_matmul: null pointer");
  Q6MOE_REQUIRE(m >= 1 && k >= 1 && n >= 1, "q6_matmul: x must be a nonempty [M,K] array");
  Q6MOE_REQUIRE(ldx >= k && ldy >= n, "q6_matmul: leading dimensions too small");
  Q6MOE_REQUIRE(m <= (1 << 30) && k <= (1 << 30) && n <= (1 << 30), "q6_matmul: dimension too large");
  Q6MOE_REQUIRE(y_dtype == Q6MOE_F32 || y_dtype == Q6MOE_BF16, "q6_matmul: y dtype must be F32 or BF16");
  Q6MOE_REQUIRE(aligned(data, 16) && aligned(scales, 2) && aligned(x, 2),
                "q6_matmul: data must be 16-byte aligned");
  const int kb = (int)cdiv(k, kQK);
  const int rowgroups = (int)cdiv(n, kTileRows) * 4;
  const int kw = kb < 8 ? kb : 8;
  const int xvec = (ldx % 8 == 0) && aligned(x, 16);
  const int ybf16 = y_dtype == Q6MOE_BF16;
  hipStream_t s = (hipStream_t)stream;
  // The tiled kernel from 64 tokens on, and above 16 for up to five 128-wide halves
  // of K: its halves pass one after another in each set (~0.6 us each with few
  // workgroups), the skinny kernel's blocks all at once. Skinny and tiled (us),
  // 17 and 48 tokens: 1280 x 256 6.4 and 4.7, 6.8 and 5.0; x 512 5.5 and 5.2, 5.9
  // and 5.5; x 640 7.4 and 6.3, 8.6 and 6.5; x 736 6.6 and 7.0, 7.5 and 7.2; x 768
  // 5.5 and 6.9, 6.5 and 7.2, with 63 tokens 7.2 and 7.3; 1280 x 2560, 48 tokens 11.0
  // and 12.7, 64 tokens 13.0 and 12.8, 777 tokens 49.0 and 20.3. It needs whole
  // 16-byte groups of x and 32-bit offsets into it.
  const bool tiled = (m >= 64 || (m > 16 && k <= 640)) && xvec && k % 8 == 0 && (m + 63) * ldx * 2 < (1ll << 31);
  if (tiled) {
    // four K sets where the workgroups leave CUs idle (1280 x 2560, 256 tokens:
    // 13.0 us against 13.9 with two; 777 tokens, 260 workgroups: 26.4 against 20.3)
    if (kb >= 6 && cdiv(n, kTileRows) * cdiv(m, pj::kTok) <= 256)
      launch_tile<4>(x, (int)m, (int)k, ldx, data, scales, (int)n, kb, y, ybf16, ldy, s);
    else
      launch_tile<2>(x, (int)m, (int)k, ldx, data, scales, (int)n, kb, y, ybf16, ldy, s);
  } else if (m <= 16) {
    hipLaunchKernelGGL(q6_skinny_kernel<1>, dim3(rowgroups, 1), dim3(64 * kw), 0, s, x, (int)m,
                       (int)k, ldx, xvec, data, scales, (int)n, kb, kw, y, ybf16, ldy);
  } else {
    hipLaunchKernelGGL(q6_skinny_kernel<4>, dim3(rowgroups, (unsigned)cdiv(m, 64)), dim3(64 * kw), 0,
                       s, x, (int)m, (int)k, ldx, xvec, data, scales, (int)n, kb, kw, y, ybf16, ldy);
  }
  return check_launch("q6_skinny_kernel");
}
