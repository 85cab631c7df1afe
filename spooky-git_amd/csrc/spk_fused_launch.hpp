// spk_fused_launch.hpp -- launcher templates of the fused forward x pass +
// spectral epilogue + RK3 update kernel (k_fwdx_epilogue).  The instantiations
// are spread over several translation units (precision x points per thread) so
// that they compile in parallel: spk_fused*.hip.
#pragma once

#include "spk_internal.hpp"
#include "spk_kernels.hpp"

namespace spk {

template <class T, int N, int LY, int EF, int TC, bool STRAT = false>
static void launch_ly_mode(int mode, dim3 grid, int bs, hipStream_t st, const cpx<T> *P, const cpx<T> *probe, cpx<double> *U,
                           cpx<T> *S, cpx<T> *W, const FusedConst &fc, const cpx<T> *tw, TimeState *ts,
                           const Batch &bt) {
    switch (mode) {
        case 1: k_fwdx_epilogue<T, N, LY, 1, EF, TC, STRAT><<<grid, bs, 0, st>>>(P, probe, U, S, W, fc, tw, ts, bt); break;
        case 2: k_fwdx_epilogue<T, N, LY, 2, EF, TC, STRAT><<<grid, bs, 0, st>>>(P, probe, U, S, W, fc, tw, ts, bt); break;
        default: k_fwdx_epilogue<T, N, LY, 3, EF, TC, STRAT><<<grid, bs, 0, st>>>(P, probe, U, S, W, fc, tw, ts, bt); break;
    }
}

// Boussinesq layouts: stratified runs couple the velocity and temperature
// groups in one block (k_fwdx_epilogue's STRAT instantiation)
template <class T, int N, int LY, int EF, int TC>
static int launch_bouss(int mode, dim3 grid, int bs, hipStream_t st, const cpx<T> *P, const cpx<T> *probe, cpx<double> *U, cpx<T> *S,
                        cpx<T> *W, const FusedConst &fc, const cpx<T> *tw, TimeState *ts, const Batch &bt) {
    if (!fc.e.stratification) {
        launch_ly_mode<T, N, LY, EF, TC>(mode, grid, bs, st, P, probe, U, S, W, fc, tw, ts, bt);
        return SPK_OK;
    }
    launch_ly_mode<T, N, LY, EF, TC, true>(mode, grid, bs, st, P, probe, U, S, W, fc, tw, ts, bt);
    return SPK_OK;
}

template <class T, int N, int EF, int TC>
static int launch_tc(int ly, int mode, hipStream_t st, const void *P, const void *probe, void *U, void *S, void *W,
                     const FusedConst &fc, const void *tw, TimeState *ts, int ngroups, const Batch &bt, unsigned nbz) {
    const long long ncols = (long long)fc.e.kg.ny * fc.e.kg.nzh;
    dim3 grid((unsigned)((ncols + TC - 1) / TC), ngroups, nbz);
    const int bs = TC * fx_tpl(N, EF);
    const cpx<T> *p = (const cpx<T> *)P, *pr = (const cpx<T> *)probe;
    cpx<double> *u = (cpx<double> *)U;
    cpx<T> *s = (cpx<T> *)S;  // the RK3 increment register, bulk precision
    cpx<T> *w = (cpx<T> *)W;
    const cpx<T> *t = (const cpx<T> *)tw;
    switch (ly) {
        case LY_HD: launch_ly_mode<T, N, LY_HD, EF, TC>(mode, grid, bs, st, p, pr, u, s, w, fc, t, ts, bt); break;
        case LY_HD_TH: SPK_TRY((launch_bouss<T, N, LY_HD_TH, EF, TC>(mode, grid, bs, st, p, pr, u, s, w, fc, t, ts, bt))); break;
        case LY_MHD: launch_ly_mode<T, N, LY_MHD, EF, TC>(mode, grid, bs, st, p, pr, u, s, w, fc, t, ts, bt); break;
        case LY_MHD_TH: SPK_TRY((launch_bouss<T, N, LY_MHD_TH, EF, TC>(mode, grid, bs, st, p, pr, u, s, w, fc, t, ts, bt))); break;
        default: set_error("fused epilogue: layout %d has no FFT products", ly); return SPK_ERR_STATE;
    }
    SPK_LAUNCH_CHECK();
    return SPK_OK;
}

// One column of 1024 points at 4 per thread fills a 256-thread block.  Where that makes
// more blocks than CUs, two columns to a block are faster, whose loads are twice as
// wide (FP32, us per step, one / two: 1024x128x2 HD, 256 blocks, 119 / 132; the same
// MHD, 512 blocks, 189 / 150).  The rule counts one box's blocks, so that a batch and
// its boxes launched one by one take the same tiles.
template <class T, int N, int EF>
static int launch_n(int ly, int mode, hipStream_t st, const void *P, const void *probe, void *U, void *S, void *W,
                    const FusedConst &fc, const void *tw, TimeState *ts, int ngroups, const Batch &bt, unsigned nbz) {
    constexpr int TC = fx_tcols(N, EF);
    if constexpr (TC == 1) {
        if ((long long)fc.e.kg.ny * fc.e.kg.nzh * ngroups > 256)
            return launch_tc<T, N, EF, 2>(ly, mode, st, P, probe, U, S, W, fc, tw, ts, ngroups, bt, nbz);
    }
    return launch_tc<T, N, EF, TC>(ly, mode, st, P, probe, U, S, W, fc, tw, ts, ngroups, bt, nbz);
}

template <class T, int EF>
static int launch_t(int nx, int ly, int mode, hipStream_t st, const void *P, const void *probe, void *U, void *S, void *W,
                    const FusedConst &fc, const void *tw, TimeState *ts, int ngroups, const Batch &bt,
                    unsigned nbz) {
    switch (nx) {
        case 32: return launch_n<T, 32, EF>(ly, mode, st, P, probe, U, S, W, fc, tw, ts, ngroups, bt, nbz);
        case 64: return launch_n<T, 64, EF>(ly, mode, st, P, probe, U, S, W, fc, tw, ts, ngroups, bt, nbz);
        case 128: return launch_n<T, 128, EF>(ly, mode, st, P, probe, U, S, W, fc, tw, ts, ngroups, bt, nbz);
        case 256: return launch_n<T, 256, EF>(ly, mode, st, P, probe, U, S, W, fc, tw, ts, ngroups, bt, nbz);
        case 512: return launch_n<T, 512, EF>(ly, mode, st, P, probe, U, S, W, fc, tw, ts, ngroups, bt, nbz);
        case 1024: return launch_n<T, 1024, EF>(ly, mode, st, P, probe, U, S, W, fc, tw, ts, ngroups, bt, nbz);
        default: set_error("fused epilogue: NX=%d not instantiated", nx); return SPK_ERR_ARG;
    }
}

// the instantiations of one precision and EF points per thread
template <class T, int EF>
int launch_fwdx_epilogue_t(spk_ctx ctx, int nx, int ly, int mode, const void *P, const void *probe, void *U, void *S,
                           void *W, const FusedConst &fc, const void *tw, TimeState *ts, int ngroups,
                           const Batch &bt) {
    return launch_t<T, EF>(nx, ly, mode, ctx->stream, P, probe, U, S, W, fc, tw, ts, ngroups, bt, nboxes(ctx));
}

#define SPK_FUSED_DECL(NAME)                                                                                     \
    int NAME(spk_ctx ctx, int nx, int ly, int mode, const void *P, const void *probe, void *U, void *S, void *W, \
             const FusedConst &fc, const void *tw, TimeState *ts, int ngroups, const Batch &bt)
SPK_FUSED_DECL(launch_fused_f64_4);
SPK_FUSED_DECL(launch_fused_f64_8);
SPK_FUSED_DECL(launch_fused_f32_4);
SPK_FUSED_DECL(launch_fused_f32_8);

}  // namespace spk
