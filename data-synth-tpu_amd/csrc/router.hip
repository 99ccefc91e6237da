// Router: FP32 softmax of the logits -> top_k -> weights divided by their sum
// -> inactive rows zeroed -> RNE to BF16 (kaggle/qwen38_tpu/math.py:277-281,
// routes_and_shared without the shared expert; numerics.py:48-51 softmax).
//
// One wave per token row, up to 1024 experts (S = 2, 4, 8 or 16 logits per
// lane for up to 128, 256, 512 and 1024 experts). The softmax
// sum and the top-k selection are wave reductions in a fixed order; top_k
// picks the largest probability, the lower expert id on ties (jax.lax.top_k),
// one selection round per k; the selected probabilities are summed in
// selection order.
#include "moe_common.h"
#include "q6moe_api.h"

namespace q6moe {

constexpr int kRouterMaxExperts = kMaxExperts;
constexpr int kRouterMaxTopK = 32;

// Wave reductions over lane exchanges that stay in the vector unit (row
// rotations and quad permutations by DPP, half-wave and row swaps by
// v_permlane32/16_swap): a few cycles a step where a shuffle through LDS takes
// some sixty, and the top-k below is a chain of K of them. The exchange at
// distance 32, 16, 8, 4, 2, 1, in this order, gives every lane the sums of a
// butterfly of xor shuffles, bit for bit: once the halves (rows, ..) agree, a
// rotation by 8 (4, 2) brings the same value as an xor by 8 (4, 2).
template <int CTRL, typename T>
__device__ __forceinline__ T dpp(T v) {
  const int w = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(w, w, CTRL, 0xf, 0xf, true));
}
template <typename T, typename F>
__device__ __forceinline__ T wave_reduce(T v, F f) {
  {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v),
                                                    false, false);
    v = f(__builtin_bit_cast(T, (uint32_t)r[0]), __builtin_bit_cast(T, (uint32_t)r[1]));
  }
  {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v),
                                                    false, false);
    v = f(__builtin_bit_cast(T, (uint32_t)r[0]), __builtin_bit_cast(T, (uint32_t)r[1]));
  }
  v = f(v, dpp<0x128>(v));  // row_ror:8
  v = f(v, dpp<0x124>(v));  // row_ror:4
  v = f(v, dpp<0x4e>(v));   // quad_perm [2,3,0,1]
  v = f(v, dpp<0xb1>(v));   // quad_perm [1,0,3,2]
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sum(float v) {
  return wave_reduce(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ int wave_min(int v) {
  return wave_reduce(v, [](int a, int b) { return a < b ? a : b; });
}

// S logits per lane. Bound by its serial chain (loads, two reductions, K
// selections of one reduction each): one token of 512 experts, top-10, 10.2 us
// with reductions through LDS and 16 slots per lane, 4.7 us so; 8 tokens of
// 128 experts, top-8, 7.4 -> 3.9 us; 4096 tokens 10.0 -> 6.2 us.
template <int S>
__global__ void __launch_bounds__(256) router_topk_kernel(const float* __restrict__ logits, int B, int E, int K,
                                                          const uint8_t* __restrict__ active,
                                                          int32_t* __restrict__ ids, uint16_t* __restrict__ wts) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= B) return;
  const float* x = logits + (int64_t)row * E;
  // expert of slot q of this lane: lane + 64q
  float v[S];
  float m = -__builtin_inff();
#pragma unroll
  for (int q = 0; q < S; ++q) {
    const int e = lane + 64 * q;
    v[q] = e < E ? x[e] : -__builtin_inff();
    m = fmaxf(m, v[q]);
  }
  m = wave_max(m);
  float part = 0.f;
#pragma unroll
  for (int q = 0; q < S; ++q) {
    v[q] = lane + 64 * q < E ? expf(v[q] - m) : 0.f;
    part += v[q];
  }
  const float total = wave_sum(part);
  float pr[S];
#pragma unroll
  for (int q = 0; q < S; ++q) pr[q] = lane + 64 * q < E ? v[q] / total : -1.f;  // probabilities are >= 0
  // top_k: one round per selection; (probability desc, id asc)
  float sel_p = 0.f, sum = 0.f;
  int sel_e = 0;
  for (int k = 0; k < K; ++k) {
    float bp = -2.f;
    int be = 1 << 30;
#pragma unroll
    for (int q = 0; q < S; ++q)
      if (pr[q] > bp) {  // slots ascend in id, so the first maximum has the lowest id
        bp = pr[q];
        be = lane + 64 * q;
      }
    // the largest probability; its lane's expert, or the lowest of the lanes' that tie
    const float top = wave_max(bp);
    const uint64_t tied = __ballot(bp == top);
    if (__popcll(tied) == 1)
      be = __builtin_amdgcn_readlane(be, __builtin_ctzll(tied));
    else
      be = wave_min(bp == top ? be : 0x7fffffff);
    // retire the selected expert on its lane
#pragma unroll
    for (int q = 0; q < S; ++q)
      if (lane + 64 * q == be) pr[q] = -1.f;
    sum += top;  // selection order, FP32
    if (lane == k) {
      sel_p = top;
      sel_e = be;
    }
  }
  if (lane < K) {
    const bool on = !active || active[row];
    const float w = on ? sel_p / sum : 0.f;
    ids[(int64_t)row * K + lane] = sel_e;
    wts[(int64_t)row * K + lane] = bf16_bits(w);
  }
}

}  // namespace q6moe

using namespace q6moe;

extern "C" int q6moe_route_topk(const float* logits, int64_t tokens, int64_t experts, int64_t top_k,
                                const uint8_t* active, int32_t* ids, uint16_t* weights, void* stream) {
  Q6MOE_REQUIRE(logits && ids && weights, "route_topk: null pointer");
  Q6MOE_REQUIRE(tokens >= 1 && tokens <= (1 << 26) && experts >= 1 && experts <= kRouterMaxExperts,
                "route_topk: 1 <= experts <= 1024");
  Q6MOE_REQUIRE(top_k >= 1 && top_k <= experts && top_k <= kRouterMaxTopK, "route_topk: 1 <= top_k <= min(experts, 32)");
  const dim3 grid((unsigned)((tokens + 3) / 4));
  const auto launch = [&](auto sc) {
    hipLaunchKernelGGL(router_topk_kernel<decltype(sc)::value>, grid, dim3(256), 0, (hipStream_t)stream, logits,
                       (int)tokens, (int)experts, (int)top_k, active, ids, weights);
  };
  if (experts <= 128)
    launch(std::integral_constant<int, 2>{});
  else if (experts <= 256)
    launch(std::integral_constant<int, 4>{});
  else if (experts <= 512)
    launch(std::integral_constant<int, 8>{});
  else
    launch(std::integral_constant<int, kRouterMaxExperts / 64>{});
  return check_launch("route_topk kernel");
}
