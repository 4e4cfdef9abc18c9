// Prefill-sized fused-MoE kernels instantiated for soft-FP8 weights.
#include "mlk_moe_wide.cuh"

namespace mlk {
template int launch_moe_wide<BF16, true>(const MoeArgs &, int, float *, int, hipStream_t);
}
