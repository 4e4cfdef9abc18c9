// The eight-wave panel GeMM instantiated for soft-FP8 weights with bf16 activations.
#include "mlk_panel8_gemm.cuh"

namespace mlk {
template int launch_panel8<BF16, true>(const Panel8Args &, int, int, hipStream_t);
}
