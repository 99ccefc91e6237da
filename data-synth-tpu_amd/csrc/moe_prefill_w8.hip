// W8A8 policy of Q8_0 projections on the INT8 matrix cores, tiled: the rows of
// kaggle/qwen38_tpu/compute.py:20-34 (q8_matmul) for routed tiles of tokens.
// Per 32-value group one v_mfma_i32_16x16x32_i8 gives exact INT32 dot products
// p; a 256-wide K block's sum is fma(f32(p) * s_x, d_w) over its groups, in
// order, in FP32, and the result is the sum of the K blocks, in order, rounded to
// BF16: the order of moe_w8_kernel's waves (one block each up to 2048 inputs), so
// that the number of tokens does not show, and no chain is longer than its own.
//
// Bound by the vector ALU first: each partial product takes a conversion, a
// multiply by the token's scale and a fused multiply-add by the row's
// (v_fma_mix_f32, the FP16 scale as it lies in the unit), 12 instructions per MFMA,
// which issue in 66 % (gate/up) and 57 % (down) of a SIMD's cycles at the step
// below; a wave waits 27 % of its time, for a K block's weights and DMA. One
// workgroup of 4 waves takes up to 64 routes of a tile against 64 rows of gate
// and up, or 128 rows of down; each wave owns 2 units (16 weight rows x one
// 256-wide K block) per K block, whose codes and scales it loads straight into
// registers in MFMA layout; the routes' codes (16 KB per K block, XOR-swizzled
// so that an operand read touches every bank once) and scales are
// double-buffered in LDS by direct buffer->LDS DMA. The running and the K block's
// sums take 64 registers, so two waves share a SIMD (212 registers; held to 168
// for a third, the kernel spills and takes 295-570 us for the step below that
// takes 291): four groups' MFMAs go first, then their conversions, products and
// sums, eight independent instructions at a time, since with two waves nothing
// else covers a dependent one's wait (306 -> 291 us). 128-expert top-8 layer,
// H 2048, I 768, 1024 tokens, cold weights: gate/up 1473 us by the kernel of 16
// tokens per weight pass (moe_w8_kernel), 189 us here, down 1075 and 108 (one
// chain over K at three waves per SIMD: 175 and 98 us).
#include "moe_tile.h"
#include "q6moe_api.h"

namespace q6moe {

namespace pf {

constexpr int kW8Groups = 4;                          // 16-route column groups per item
constexpr int kW8Routes = 16 * kW8Groups;
constexpr int kW8Subs = kM / kW8Routes;               // items per tile and column block
constexpr int kW8Codes = kW8Routes * 256;             // LDS bytes of a K block's codes
constexpr int kW8Stage = kW8Codes + kW8Routes * 32;   // and of its 8 scales per route
constexpr int kW8Lds = 2 * kW8Stage;

// A unit's weights for the INT8 MFMA: lane (row j = lane % 16, k-group kq =
// lane / 16) feeds codes 8kq..8kq+7 of group G = 2g + h (row j's Q8_0 block G),
// at 1024g + 16(16(2h + kq/2) + j) + 8(kq % 2) of the unit, and scales the four
// rows 4kq + i of its results: the FP16 scale of row 4kq + i's block 2g + h is
// half 4h + g of the 16 bytes at 4096 + 16(4kq + i).
struct W8Unit {
  uint64_t c[8];
  u32x4 s[4];
  __device__ __forceinline__ void load_codes(const uint8_t* u, int quad, int lane) {
    const int kq = lane >> 4, j = lane & 15;
    const uint8_t* v = u + 16 * (16 * (kq >> 1) + j) + 8 * (kq & 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int G = 4 * quad + q;
      c[G] = *reinterpret_cast<const uint64_t*>(v + 1024 * (G >> 1) + 512 * (G & 1));
    }
  }
  __device__ __forceinline__ void load_scales(const uint8_t* u, int lane) {
    const uint8_t* v = u + 4096 + 64 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = *reinterpret_cast<const u32x4*>(v + 16 * i);
  }
  __device__ __forceinline__ float scale(int i, int G) const {
    const uint32_t w = s[i][2 * (G & 1) + (G >> 2)];
    return (G >> 1) & 1 ? h16_hi(w) : h16_lo(w);
  }
};

__device__ __forceinline__ i32x4 mfma_i8z(uint64_t a, uint64_t b) {
  return __builtin_amdgcn_mfma_i32_16x16x32_i8((long)a, (long)b, i32x4{0, 0, 0, 0}, 0, 0, 0);
}

// acc[u][tg] += unit u's 16 rows x the routes of column group tg, over all of K
// (a multiple of 128). ``row_of(t)`` is the activation row of the item's route t.
template <int NCG, typename RowOf>
__device__ __forceinline__ void w8_stream(uint8_t* smem, const uint8_t* const (&units)[kUnits], int kbs, const W8Src& a,
                                          int a_rows, RowOf row_of, f32x4 (&acc)[kUnits][NCG]) {
  const int wave = wave_id(), lane = threadIdx.x & 63;
  const int j = lane & 15, kq = lane >> 4;
  const int groups = a.k / 32;
  const __amdgpu_buffer_rsrc_t cr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t*>(a.codes), (short)0, (int)((uint32_t)a_rows * (uint32_t)a.k), 0x00020000);
  const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.scales), (short)0, (int)((uint32_t)a_rows * (uint32_t)groups * 4u), 0x00020000);
  // DMA of a K block: NCG instructions per wave for the codes (granule
  // (wave*NCG + i)*64 + lane), one for the scales of 32 routes on the first
  // ceil(NCG / 2) waves. Past the last whole K block the granules hold the
  // next row's values (zeros past the buffer); their groups are skipped.
  int rows[NCG], srow;
  {
    const int t = 32 * wave + (lane >> 1);
#pragma unroll
    for (int i = 0; i < NCG; ++i) rows[i] = row_of(((wave * NCG + i) * 64 + lane) >> 4);
    srow = row_of(t < 16 * NCG ? t : 16 * NCG - 1);
  }
  W8Unit w[kUnits];
#pragma unroll
  for (int u = 0; u < kUnits; ++u) {
    w[u].load_codes(units[u], 0, lane);
    w[u].load_scales(units[u], lane);
    w[u].load_codes(units[u], 1, lane);
  }
  asm volatile("" ::: "memory");  // every load above issues before the offsets wait on the rows
  uint32_t xoff[NCG];
#pragma unroll
  for (int i = 0; i < NCG; ++i) {
    const int p = (wave * NCG + i) * 64 + lane;
    xoff[i] = opaque((uint32_t)(rows[i] * a.k + ((p & 15) ^ ((p >> 4) & 15)) * 16));
  }
  const uint32_t soff = opaque((uint32_t)(srow * groups * 4 + 16 * (lane & 1)));
  const bool scale_wave = 2 * wave < NCG;
  auto dma = [&](int kb) {
    uint8_t* st = smem + (kb & 1) * kW8Stage;
#pragma unroll
    for (int i = 0; i < NCG; ++i) bdma16(cr, xoff[i], (uint32_t)kb * 256u, st + (wave * NCG + i) * 1024);
    if (scale_wave) bdma16(sr, soff, (uint32_t)kb * 32u, st + kW8Codes + wave * 1024);
  };
  dma(0);
  for (int kb = 0; kb < kbs; ++kb) {
    // this block's DMA and weights have arrived; with every wave past the
    // barrier the tile is whole and the other stage's readers are done
    wait_vm<0>();
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's reads of the other stage
    wg_barrier();
    const bool more = kb + 1 < kbs;
    if (more) dma(kb + 1);
    const uint8_t* st = smem + (kb & 1) * kW8Stage;
    const int ng = groups - 8 * kb;
    f32x4 blk[kUnits][NCG];
#pragma unroll
    for (int u = 0; u < kUnits; ++u)
#pragma unroll
      for (int t = 0; t < NCG; ++t) blk[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    static_for<0, 2>([&](auto qc) {
      constexpr int quad = decltype(qc)::value;
      if (4 * quad < ng) {  // false only in the second half of a last, half K block
#pragma unroll
        for (int tg = 0; tg < NCG; ++tg) {
          const f32x4 sa = *reinterpret_cast<const f32x4*>(st + kW8Codes + (tg * 16 + j) * 32 + 16 * quad);
          // this column group's 8 MFMAs first, then their conversions, so that none waits for its product
          i32x4 p[4][kUnits];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int G = 4 * quad + q;
            const uint64_t b = *reinterpret_cast<const uint64_t*>(st + xgran(tg * 16 + j, 2 * G + (kq >> 1)) + 8 * (kq & 1));
#pragma unroll
            for (int u = 0; u < kUnits; ++u) p[q][u] = mfma_i8z(w[u].c[G], b);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float v[kUnits][4];
#pragma unroll
            for (int u = 0; u < kUnits; ++u)
#pragma unroll
              for (int i = 0; i < 4; ++i) v[u][i] = (float)p[q][u][i];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < kUnits; ++u)
#pragma unroll
              for (int i = 0; i < 4; ++i) v[u][i] *= sa[q];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < kUnits; ++u)
#pragma unroll
              for (int i = 0; i < 4; ++i) blk[u][tg][i] = __builtin_fmaf(v[u][i], w[u].scale(i, 4 * quad + q), blk[u][tg][i]);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      // the next block's weights, each into the registers just used up
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
          const uint8_t* un = units[u] + (int64_t)(kb + 1) * kQ8Unit;
          w[u].load_codes(un, quad, lane);
          if (quad == 1) w[u].load_scales(un, lane);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
#pragma unroll
    for (int u = 0; u < kUnits; ++u)
#pragma unroll
      for (int t = 0; t < NCG; ++t) acc[u][t] += blk[u][t];
  }
}

}  // namespace pf

// PAIR: gate p0 and up p1 of a row block of 64, with the SwiGLU epilogue
// a = RNE(RNE(g*sigmoid(g)) * u); otherwise 128 rows of p0, RNE. Items as in
// the BF16 tiled kernels, each tile in kW8Subs parts of 64 routes. Activation
// row of a route: its token (gate/up) or its position (``route_rows``, down);
// dense items (D.tiles > 0, p0 only): the token.
template <bool PAIR>
__global__ void __launch_bounds__(64 * pf::kWaves, 2)
    moe_pf_w8_kernel(Proj p0, Proj p1, MoeWs ws, int route_rows, W8Src a, int a_rows, uint16_t* __restrict__ out,
                     int ncol, PfDense D) {
  using namespace pf;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  Tile T;
  bool dense;
  int tile, col;
  if (!pf_item<!PAIR>(ws, ncol, D, dense, tile, col)) return;
  const int ncb = (dense ? D.ncol : ncol) / kW8Subs, sub = col / ncb;
  col -= sub * ncb;
  item_tile(ws, D, dense, tile, T);
  T.r0 += sub * kW8Routes;
  T.nv -= sub * kW8Routes;
  if (T.nv <= 0) return;
  if (T.nv > kW8Routes) T.nv = kW8Routes;
  const int wave = wave_id(), lane = threadIdx.x & 63;
  const int j = lane & 15, kq = lane >> 4;
  const int rg0 = PAIR ? col * kWaves + wave : (col * kWaves + wave) * 2;  // this wave's first row group
  const uint8_t* units[kUnits] = {unit_ptr<FMT_Q8>(p0, T.expert, rg0, 0),
                                  PAIR ? unit_ptr<FMT_Q8>(p1, T.expert, rg0, 0)
                                       : unit_ptr<FMT_Q8>(p0, T.expert, rg0 + 1, 0)};
  const bool direct = dense || route_rows;
  auto run = [&](auto ncg_c) {
    constexpr int NCG = decltype(ncg_c)::value;
    f32x4 acc[kUnits][NCG];
#pragma unroll
    for (int u = 0; u < kUnits; ++u)
#pragma unroll
      for (int t = 0; t < NCG; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto row_of = [&](int t) {
      const int r = T.r0 + (t < T.nv ? t : T.nv - 1);
      return direct ? r : ws.route_tok[r];
    };
    w8_stream<NCG>(smem, units, p0.kb, a, a_rows, row_of, acc);
#pragma unroll
    for (int tg = 0; tg < NCG; ++tg) {
      const int q = tg * 16 + j;
      if (q >= T.nv) continue;
      uint16_t* o = out + (int64_t)(T.r0 + q) * p0.rows + rg0 * 16 + 4 * kq;
      if constexpr (PAIR) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float g = bf16_round(acc[0][tg][i]), u = bf16_round(acc[1][tg][i]);
          v[i] = bf16_round(g * sigmoid_acc(g)) * u;
        }
        *reinterpret_cast<u32x2*>(o) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      } else {
#pragma unroll
        for (int u = 0; u < kUnits; ++u)
          *reinterpret_cast<u32x2*>(o + 16 * u) =
              u32x2{pack_bf16x2(acc[u][tg][0], acc[u][tg][1]), pack_bf16x2(acc[u][tg][2], acc[u][tg][3])};
      }
    }
  };
  switch ((T.nv + 15) >> 4) {
    case 1: run(std::integral_constant<int, 1>{}); break;
    case 2: run(std::integral_constant<int, 2>{}); break;
    case 3: run(std::integral_constant<int, 3>{}); break;
    default: run(std::integral_constant<int, 4>{}); break;
  }
}

bool pf_w8_supported(bool pair, int64_t rows, int64_t k) {
  return k % 128 == 0 && rows % (pair ? 16 * pf::kWaves : 32 * pf::kWaves) == 0;
}

template <bool PAIR>
static void pf_launch_w8(const Proj& p0, const Proj& p1, const MoeWs& ws, int max_tiles, int route_rows,
                         const W8Src& a, int a_rows, uint16_t* out, PfDense D, hipStream_t s) {
  static std::atomic<uint64_t> attr_done{0};
  once_per_device(attr_done, [] {
    (void)hipFuncSetAttribute((const void*)moe_pf_w8_kernel<PAIR>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              pf::kW8Lds);
  });
  const int per = pf::kW8Subs * (p0.rows / (PAIR ? 16 * pf::kWaves : 32 * pf::kWaves));
  const int ncol = max_tiles ? per : 0;
  D.ncol = per;
  const int64_t routed = ((int64_t)ncol * max_tiles + 7) / 8, dense = ((int64_t)D.tiles * D.ncol + 7) / 8;
  hipLaunchKernelGGL(moe_pf_w8_kernel<PAIR>, dim3((unsigned)(8 * (routed + dense))), dim3(64 * pf::kWaves), pf::kW8Lds,
                     s, p0, p1, ws, route_rows, a, a_rows, out, ncol, D);
}

void launch_moe_prefill_w8(bool pair, const Proj& p0, const Proj& p1, const MoeWs& ws, int max_tiles, int route_rows,
                           const W8Src& a, int a_rows, uint16_t* out, hipStream_t s) {
  if (pair)
    pf_launch_w8<true>(p0, p1, ws, max_tiles, route_rows, a, a_rows, out, PfDense{}, s);
  else
    pf_launch_w8<false>(p0, p1, ws, max_tiles, route_rows, a, a_rows, out, PfDense{}, s);
}

void launch_prefill_w8_dense(const Proj& p, const W8Src& a, int tokens, uint16_t* out, hipStream_t s) {
  PfDense D{};
  D.tokens = tokens;
  D.tiles = (tokens + pf::kM - 1) / pf::kM;
  pf_launch_w8<false>(p, p, MoeWs{}, 0, 1, a, tokens, out, D, s);
}

}  // namespace q6moe
