// spk_fused_f64_4.hip -- k_fwdx_epilogue instantiations: FP64 bulk, 4 points per thread.
#include "spk_fused_launch.hpp"

namespace spk {

SPK_FUSED_DECL(launch_fused_f64_4) {
    return launch_fwdx_epilogue_t<double, 4>(ctx, nx, ly, mode, P, probe, U, S, W, fc, tw, ts, ngroups, bt);
}

}  // namespace spk
