// Prefill-sized fused-MoE kernels instantiated for fp16 weights.
#include "mlk_moe_wide.cuh"

namespace mlk {
template int launch_moe_wide<F16, false>(const MoeArgs &, int, float *, int, hipStream_t);
}
