// The mid tiles of the INT8 GEMM with BF16 outputs (gemm_mid_launch.h), compiled in parallel with the other units.
#include "gemm_mid_launch.h"

namespace wq8 {
template int dispatch_mid<DT_BF16>(GemmArgs&, const Variant&, int, hipStream_t);
}  // namespace wq8
