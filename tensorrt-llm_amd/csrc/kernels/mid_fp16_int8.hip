// Instantiates the barrier-free mid-M kernel for FP16 activations and int8 weights.
#include "mid_kernel.h"

namespace woq
{
int launch_mid_FP16_8(MatmulProblem const& p, MidPlan const& plan, void* stream)
{
    return launch_mid_typed<WOQ_FP16, 8>(p, plan, stream);
}
} // namespace woq
