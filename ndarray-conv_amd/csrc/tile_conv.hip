// The single-precision tile kernels (see tile_kernels.hpp).
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "tile_kernels.hpp"

namespace ndc {

template <>
ndc_status launch_tile_as<float>(const TilePlan& t, const TileArgs& a, bool cplx, int what, LaunchContext& ctx) {
    return tilek::launch_tile_r<float>(t, a, cplx, what, ctx);
}

}  // namespace ndc
