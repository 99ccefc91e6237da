// Building blocks of the tiled grouped-GEMM kernels: direct buffer->LDS DMA,
// waits, the LDS layout of a token tile and the mapping of workgroups to
// (tile, column block) items.
#pragma once
#include <type_traits>

#include "moe_common.h"

#define LDS_PTR(p) ((__attribute__((address_space(3))) void*)(uint32_t)(uintptr_t)(p))

namespace q6moe {

namespace pf {

constexpr int kWaves = 4;
constexpr int kM = 128;            // routes per tile (MFMA column groups of 16)
constexpr int kUnits = 2;          // units per wave per K block

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// Wave index as a wave-uniform (SGPR) value, so that row groups and the
// weight addresses derived from it stay in scalar registers.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

__device__ __forceinline__ uint32_t opaque(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}
// Direct buffer->LDS DMA of 16 bytes per lane: byte offset voff (per lane)
// plus soff (wave-uniform) into the buffer r, no address arithmetic in VGPRs;
// an offset past the buffer's end reads zeros.
__device__ __forceinline__ void bdma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, void* lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, LDS_PTR(lds), 16, voff, soff, 0, 0);
}
// Workgroup barrier without the memory fence of __syncthreads (whose release
// would wait for every outstanding DMA, including the ones prefetching the
// next stage). LDS visibility comes from each wave's own vmcnt wait before it.
__device__ __forceinline__ void wg_barrier() { asm volatile("s_barrier" ::: "memory"); }

template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// LDS byte offset of token-tile granule (token t, 8-column granule c) of a K half.
__device__ __forceinline__ int xgran(int t, int c) { return (t * 16 + (c ^ (t & 15))) * 16; }

struct Tile {
  int64_t expert;
  int r0, nv;  // first route position, valid routes (<= kM)
};

// Work item of workgroup blockIdx.x. Workgroup i runs on XCD i % 8
// (round-robin dispatch), so the items are split into eight contiguous runs,
// one per XCD, each walked in dispatch order.
// The dense expert's items (D.ncol column blocks x D.tiles token tiles) come
// first, an eighth on each XCD, since they are full tiles over the longest K;
// token tile fastest: the workgroups that share a block of its weights run on
// one XCD at the same time and share its L2 (every XCD reads the tokens, which
// are the smaller side).
// Routed items are (tile, column block), column block fastest: those that
// share a token tile (its column blocks) or an expert's weights (its tiles)
// run together. ncol 0: no routed items. Returns false past the last item.
// kDense false: a launch without dense items, compiled apart (the choice per
// item cost the routed-only 4096-token step 0.6 %).
template <bool kDense>
__device__ __forceinline__ bool pf_item(const MoeWs& ws, int ncol, const PfDense& D, bool& dense, int& tile, int& col) {
  const int xcd = blockIdx.x & 7;
  int k = blockIdx.x >> 3;
  dense = false;
  if constexpr (kDense) {
    const int nd = D.tiles * D.ncol, rd = (nd + 7) >> 3;
    dense = k < rd;
    if (dense) {
      const int item = xcd * rd + k;
      if (item >= nd) return false;
      col = item / D.tiles;
      tile = item - col * D.tiles;
      return true;
    }
    if (ncol == 0) return false;
    k -= rd;
  }
  const int ntiles = ws.hdr[2];
  const int items = ntiles * ncol;
  const int run = (items + 7) >> 3;
  const int item = xcd * run + k;
  if (k >= run || item >= items) return false;
  tile = item / ncol;
  col = item - tile * ncol;
  return true;
}

__device__ __forceinline__ void tile_info(const MoeWs& ws, int tile, Tile& T) {
  const PfTile d = ws.tile[tile];  // one scalar load
  T.expert = d.expert;
  T.r0 = d.r0;
  T.nv = d.nv;
}

// The item's tile: the routing's record, or kM consecutive tokens.
__device__ __forceinline__ void item_tile(const MoeWs& ws, const PfDense& D, bool dense, int tile, Tile& T) {
  if (dense) {
    T.expert = 0;
    T.r0 = tile * kM;
    T.nv = D.tokens - T.r0 < kM ? D.tokens - T.r0 : kM;
  } else {
    tile_info(ws, tile, T);
  }
}

}  // namespace pf
}  // namespace q6moe
