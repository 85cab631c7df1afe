// spk_fused.hip -- the launcher of the fused forward x pass + spectral
// epilogue + RK3 update kernel (k_fwdx_epilogue): picks the instantiation set
// (precision; points per thread) compiled in spk_fused_*.hip.
#include "spk_fused_launch.hpp"

namespace spk {

bool fused_supported_nx(int nx) { return nx >= 32 && nx <= 1024 && is_pow2(nx); }

// ef: points per thread of the x line, 4 or 8 (picked by the solver's tile autotune)
int launch_fwdx_epilogue(spk_ctx ctx, int bulk, int nx, int ly, int mode, int ef, const void *P, const void *probe,
                         void *U, void *S, void *W, const FusedConst &fc, const void *tw, TimeState *ts,
                         int ngroups) {
    Batch bt;
    SPK_TRY(make_batch(ctx, {P, U, S, W, ts, probe}, &bt));
    if (bulk == SPK_F64)
        return ef == 8 ? launch_fused_f64_8(ctx, nx, ly, mode, P, probe, U, S, W, fc, tw, ts, ngroups, bt)
                       : launch_fused_f64_4(ctx, nx, ly, mode, P, probe, U, S, W, fc, tw, ts, ngroups, bt);
    return ef == 8 ? launch_fused_f32_8(ctx, nx, ly, mode, P, probe, U, S, W, fc, tw, ts, ngroups, bt)
                   : launch_fused_f32_4(ctx, nx, ly, mode, P, probe, U, S, W, fc, tw, ts, ngroups, bt);
}

}  // namespace spk
