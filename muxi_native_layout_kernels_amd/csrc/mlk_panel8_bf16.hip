// The eight-wave panel GeMM instantiated for bf16 weights and activations.
#include "mlk_panel8_gemm.cuh"

namespace mlk {
template int launch_panel8<BF16, false>(const Panel8Args &, int, int, hipStream_t);
}
