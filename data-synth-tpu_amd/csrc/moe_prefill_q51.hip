// Tiled prefill kernels of Q5_1 tables.
#include "moe_prefill.h"

namespace q6moe {

template void pf_down<FMT_Q51>(const Proj&, const MoeWs&, int, int, int, int, int, const PfDense&, hipStream_t);
template void pf_unpack<FMT_Q51>(const Proj&, int, uint16_t*, hipStream_t);

}  // namespace q6moe
