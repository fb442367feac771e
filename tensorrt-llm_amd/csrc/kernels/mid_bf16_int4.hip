// Instantiates the barrier-free mid-M kernel for BF16 activations and int4 weights.
#include "mid_kernel.h"

namespace woq
{
int launch_mid_BF16_4(MatmulProblem const& p, MidPlan const& plan, void* stream)
{
    return launch_mid_typed<WOQ_BF16, 4>(p, plan, stream);
}
} // namespace woq
