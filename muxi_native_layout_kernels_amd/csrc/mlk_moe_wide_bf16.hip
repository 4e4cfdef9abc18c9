// Prefill-sized fused-MoE kernels instantiated for bf16 weights.
#include "mlk_moe_wide.cuh"

namespace mlk {
template int launch_moe_wide<BF16, false>(const MoeArgs &, int, float *, int, hipStream_t);
}
