// Direct rank-2 convolutions on the matrix cores (matrix_conv.hip).
#pragma once

#include "launch.hpp"
#include "plan.hpp"

namespace ndc {

// Runs the plan there and stores the launch's status; false when the plan is
// left to the other direct kernels.  `exact`: in the element type, whatever
// matrix form the plan asks for.
bool launch_matrix(const Plan& p, bool exact, const void* x, const void* k, void* y, LaunchContext& ctx,
                   ndc_status* status);

}  // namespace ndc
