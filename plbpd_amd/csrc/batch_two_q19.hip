// The batched two-step kernels of D3Q19 (batch_two.hpp).
#include "batch_two.hpp"

namespace plb {
PLB_BATCH2_INST_Q(19)
}  // namespace plb
