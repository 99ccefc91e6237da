// Tiled prefill kernels of Q5_K tables.
#include "moe_prefill.h"

namespace q6moe {

template void pf_gate_up<FMT_Q5K>(const Proj&, const Proj&, const MoeWs&, int, int, const uint16_t*, int, int, int,
                              const PfDense&, hipStream_t, void*, void*);
template void pf_down<FMT_Q5K>(const Proj&, const MoeWs&, int, int, int, int, int, const PfDense&, hipStream_t);
template void pf_unpack<FMT_Q5K>(const Proj&, int, uint16_t*, hipStream_t);

}  // namespace q6moe
