// The multi-step kernels of D2Q9 (fused_multi.hpp).
#include "fused_multi.hpp"

namespace plb {
PLB_MULTI9_INST(kF64)
PLB_MULTI9_INST(kF32)
PLB_MULTI9_INST(kF64A32)
PLB_MULTI9_INST(kF32S)
PLB_MULTI9_INST(kF16S)
}  // namespace plb
