// f16 instantiations of the four-wave GEMM (gemm4w.h): small tiles
#include "gemm4w.h"

namespace lmx {
LMX_GEMM4W_SMALL(LMX_GEMM4W_INST, f16_t)
}  // namespace lmx
