// The eight-wave panel GeMM instantiated for fp16 weights and activations.
#include "mlk_panel8_gemm.cuh"

namespace mlk {
template int launch_panel8<F16, false>(const Panel8Args &, int, int, hipStream_t);
}
