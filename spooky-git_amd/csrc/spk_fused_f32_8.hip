// spk_fused_f32_8.hip -- k_fwdx_epilogue instantiations: FP32 bulk, 8 points per thread.
#include "spk_fused_launch.hpp"

namespace spk {

SPK_FUSED_DECL(launch_fused_f32_8) {
    return launch_fwdx_epilogue_t<float, 8>(ctx, nx, ly, mode, P, probe, U, S, W, fc, tw, ts, ngroups, bt);
}

}  // namespace spk
