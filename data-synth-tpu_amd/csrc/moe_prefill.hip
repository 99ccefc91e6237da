// The tiled prefill path's host side: which calls it takes and the dispatch to
// each format's launches (moe_prefill.h, instantiated in moe_prefill_*.hip).
#include "moe_tile.h"
#include "q6moe_api.h"

namespace q6moe {

template <int FMT>
void pf_gate_up(const Proj& g, const Proj& u, const MoeWs& ws, int mtile, int max_tiles, const uint16_t* x, int B, int H,
                int I, const PfDense& D, hipStream_t s, void* gate_up_start, void* after_gate_up);
template <int FMT>
void pf_down(const Proj& d, const MoeWs& ws, int mtile, int max_tiles, int routes, int H, int I, const PfDense& D,
             hipStream_t s);
template <int FMT>
void pf_unpack(const Proj& p, int experts, uint16_t* out, hipStream_t s);

// The tiled kernels take K in halves of 128 and whole workgroup row blocks:
// gate/up 64 intermediate rows, down 128 hidden rows.
bool pf_gate_up_supported(int fmt, int64_t H, int64_t I) {
  return fmt != FMT_Q51 && H % 128 == 0 && I % (16 * pf::kWaves) == 0;
}
bool pf_down_supported(int fmt, int64_t H, int64_t I) {
  (void)fmt;
  return I % 128 == 0 && H % (32 * pf::kWaves) == 0;
}

static int pf_tiles(int tokens) { return (tokens + pf::kM - 1) / pf::kM; }

PfDense pf_dense_gate_up(const Proj& g, const Proj& u, const uint16_t* x, int tokens, uint16_t* act) {
  return PfDense{g, u, x, act, tokens, pf_tiles(tokens), g.rows / (16 * pf::kWaves), g.rows};
}
PfDense pf_dense_down(const Proj& d, const uint16_t* act, int tokens, uint16_t* y) {
  return PfDense{d, d, act, y, tokens, pf_tiles(tokens), d.rows / (32 * pf::kWaves), d.rows};
}

int launch_moe_prefill_gate_up(int fmt, const Proj& g, const Proj& u, const MoeWs& ws, int mtile, int max_tiles,
                               const uint16_t* x, int B, int H, int I, const PfDense& D, hipStream_t s,
                               void* gate_up_start, void* after_gate_up) {
  dispatch_format(fmt, [&](auto fc) {
    if constexpr (decltype(fc)::value != FMT_Q51)  // no gate/up format (pf_gate_up_supported)
      pf_gate_up<decltype(fc)::value>(g, u, ws, mtile, max_tiles, x, B, H, I, D, s, gate_up_start, after_gate_up);
  });
  return Q6MOE_OK;
}

int launch_moe_prefill_down(int fmt, const Proj& d, const MoeWs& ws, int mtile, int max_tiles, int routes, int H, int I,
                            const PfDense& D, hipStream_t s) {
  dispatch_format(fmt, [&](auto fc) {
    pf_down<decltype(fc)::value>(d, ws, mtile, max_tiles, routes, H, I, D, s);
  });
  return Q6MOE_OK;
}

int launch_pf_unpack(int fmt, const Proj& p, int experts, uint16_t* out, hipStream_t s) {
  dispatch_format(fmt, [&](auto fc) { pf_unpack<decltype(fc)::value>(p, experts, out, s); });
  return Q6MOE_OK;
}

}  // namespace q6moe
