// spk_planefft.hip -- the y and z passes of a 3D transform in one kernel, for
// grids whose (y, z) plane fits LDS.
//
// A plan's y and z passes each read and write every field once; both stay inside
// an x plane, NY x (NZ/2+1) complex values.  One workgroup holds one plane of one
// field in LDS: it makes the y lines and the z rows there, and the field crosses
// HBM once instead of twice (a transform: 4 sweeps instead of 6).  The plane is
// stored by rows in the z rows' own placement (PadXor), so that a row's transform
// exchanges within its row; a y line exchanges within its column.
//
// Bound by HBM, as the passes are.  A workgroup loads, transforms and stores in
// turn, so several must share a CU: planes up to 80 KB take this kernel (two to a
// CU), larger ones keep the passes.  Within that limit it was faster than the two
// passes at every shape, type and direction measured (planes of 16x32 to 256x32
// and 16x512).  Whole transforms before -> now, microseconds:
//   six FP32 fields of 512x64x128, C2R 126 -> 88, R2C 129 -> 93 (copy rate of the
//   four sweeps: 83); six FP64 fields of 256x64x64, C2R 75 -> 47, R2C 79 -> 47;
//   one FP64 field of 64^3 21.5 -> 10.8; four FP64 fields of 512x16x32 32 -> 19.
#include "spk_internal.hpp"
#include "spk_rows.hpp"

namespace spk {

constexpr size_t PF_LDS = 80 * 1024;

// a y line inside the plane: element i is PITCH elements further down the column
template <int PITCH>
struct PadColumn {
    __device__ static __forceinline__ int at(int i) { return i * PITCH; }
};

template <class T, int NY, int NZ>
struct PlaneShape {
    static constexpr int M = NZ / 2, NZH = M + 1;
    static constexpr int LL = PadXor::len(M + 1);
    // 8 points of the plane per thread within a wave and 8 waves: with twice the threads, and
    // so fewer workgroups on a CU, 512x64x64 FP64 took 76 instead of 66 us
    static constexpr int T0 = NY * M / 8, PF_T = T0 < 64 ? 64 : (T0 > 512 ? 512 : T0);
    // 8 points per thread, and 16 where 8 would leave the line a last pass of radix 2: its extra
    // twiddles cost accuracy (FP32 rel-L2 of 64x16x32 1.36e-7 against 1.33e-7, of 64x16x256 1.49e-7
    // against 1.48e-7; the separate passes 1.33e-7 and 1.48e-7), at up to 20% of the time of
    // NZ = 256 transforms (512x16x256 FP64 C2R 60 -> 69 us, the separate passes 85)
    static constexpr bool tail2(int n) { return n == 2 || (n > 8 && tail2(n / 8)); }
    static constexpr int EZ = tail2(M) ? 16 : 8, TPLZ = M / EZ, RW = PF_T / TPLZ;
    static constexpr int ey(int e) { return (NZH + PF_T / (NY / e) - 1) / (PF_T / (NY / e)); }  // rounds of columns
    // 16 also where that saves a round of columns
    static constexpr int EY = tail2(NY) || ey(16) < ey(8) ? 16 : 8;
    // FP64: two radix-8 passes with sqrt(1/2) rounded to FP64 were off by up to 2.8% more than the
    // separate passes' radix 16 and 4 (rel-L2 of 32x16x128 2.54e-16 against 2.48e-16; with it to
    // twice the precision 2.46e-16; NZ = 512 2.73e-16, 2.69e-16 and 2.64e-16), in the same time.  16 points
    // there instead took 10-40% longer (512x16x512 C2R 104 -> 150 us)
    static constexpr bool EXACT = sizeof(T) == 8;
    static constexpr int TPLY = NY / EY, TC = PF_T / TPLY;
    static constexpr int ROWS = NY + (RW > NY ? 1 : 0);  // a spare row for row groups past the plane
    static constexpr size_t bytes = (size_t)ROWS * LL * sizeof(cpx<T>);
    static constexpr bool fits = bytes <= PF_LDS && TPLZ <= 64;
};

template <class T, int NY, int NZ, int DIR>
__global__ __launch_bounds__((PlaneShape<T, NY, NZ>::PF_T)) void k_plane_yz(
    const cpx<T> *in, cpx<T> *out, long long fs_in, long long fs_out, const cpx<T> *__restrict__ twy,
    const cpx<T> *__restrict__ tw_nz, const cpx<T> *__restrict__ tw_m, Batch bt) {
    using S = PlaneShape<T, NY, NZ>;
    using Row = ZRow<T, S::M, S::EZ, false, S::EXACT>;
    constexpr int M = S::M, NZH = S::NZH, LL = S::LL;
    static_assert(Row::WAVE && Row::LL == LL, "a row's threads share one wavefront");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    cpx<T> *plane = reinterpret_cast<cpx<T> *>(smem);
    in = rebase(bt, 0, in);
    out = rebase(bt, 1, out);
    in += (long long)blockIdx.y * fs_in + (long long)blockIdx.x * NY * NZH;
    out += (long long)blockIdx.y * fs_out + (long long)blockIdx.x * NY * NZH;
    const int tid = threadIdx.x;

    auto y_pass = [&] {
        const int c = tid % S::TC, t = tid / S::TC;
#pragma unroll 1
        for (int c0 = 0; c0 < NZH; c0 += S::TC) {
            const bool live = c0 + c < NZH;
            const int col = live ? c0 + c : NZH;  // LL > NZH: a spare column, shared by the idle threads
            cpx<T> *L = plane + PadXor::at(col);
            cpx<T> v[S::EY];
#pragma unroll
            for (int i = 0; i < S::EY; i++) {
                const int n = t + i * S::TPLY;
                if constexpr (DIR > 0) v[i] = live ? in[n * NZH + col] : cpx<T>{(T)0, (T)0};
                else v[i] = L[n * LL];
            }
            if constexpr (DIR < 0) __syncthreads();  // a line's values are read before its exchanges overwrite them
            LineFFT<T, NY, S::EY, DIR, false, 0, PadColumn<LL>, S::EXACT>::run(v, L, t, twy);
#pragma unroll
            for (int i = 0; i < S::EY; i++) {
                const int n = t + i * S::TPLY;
                if constexpr (DIR > 0) L[n * LL] = v[i];
                else if (live) out[n * NZH + col] = v[i];
            }
        }
    };
    auto z_pass = [&] {
        const int rl = tid / S::TPLZ, t = tid % S::TPLZ;
#pragma unroll 1
        for (int r0 = 0; r0 < NY; r0 += S::RW) {
            const int row = r0 + rl;
            const bool live = row < NY;
            cpx<T> *L = plane + (live ? row : NY) * LL;
            cpx<T> v[S::EZ];
            if constexpr (DIR > 0) {
#pragma unroll
                for (int i = 0; i < S::EZ; i++) v[i] = L[PadXor::at(t + i * S::TPLZ)];
                const cpx<T> nyq = t == 0 ? L[PadXor::at(M)] : cpx<T>{(T)0, (T)0};
                lsync<true>();
                Row::c2r_regs(v, nyq, live, L, t, tw_nz, tw_m, (T)1);
                if (live) {
                    cpx<T> *dst = out + row * NZH;
#pragma unroll
                    for (int i = 0; i < S::EZ; i++) dst[t + i * S::TPLZ] = v[i];
                    if (t == 0) dst[M] = cpx<T>{(T)0, (T)0};
                }
            } else {
#pragma unroll
                for (int i = 0; i < S::EZ; i++)
                    v[i] = live ? in[row * NZH + t + i * S::TPLZ] : cpx<T>{(T)0, (T)0};
                Row::r2c_row(v, L, t, tw_nz, tw_m);
            }
        }
    };
    if constexpr (DIR > 0) {
        y_pass();
        __syncthreads();
        z_pass();
    } else {
        z_pass();
        __syncthreads();
        y_pass();
    }
}

template <class T, int NY, int NZ>
static int launch_nynz(spk_ctx ctx, const Grid3 &g, const Twiddles &tw, int dir, const PassArgs &a) {
    using S = PlaneShape<T, NY, NZ>;
    if constexpr (!S::fits) {
        return SPK_ERR_STATE;  // launch_plane_yz has refused the shape
    } else {
        const cpx<T> *base = reinterpret_cast<const cpx<T> *>(tw.d);
        const cpx<T> *ty = base + tw.off_y, *tz = base + tw.off_z, *tm = base + tw.off_z + g.nz;
        Batch bt;
        SPK_TRY(make_batch(ctx, {a.in, a.out}, &bt));
        const dim3 grid((unsigned)g.nx, a.nfields, nboxes(ctx));
        auto *k = dir > 0 ? k_plane_yz<T, NY, NZ, +1> : k_plane_yz<T, NY, NZ, -1>;
        if constexpr (S::bytes > 64 * 1024)
            SPK_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::bytes));
        k<<<grid, S::PF_T, S::bytes, ctx->stream>>>((const cpx<T> *)a.in, (cpx<T> *)a.out, a.fstride_in, a.fstride_out, ty,
                                                    tz, tm, bt);
        SPK_LAUNCH_CHECK();
        return SPK_OK;
    }
}

template <class T, int NY>
static bool fits_ny(int nz) {
    switch (nz) {
        case 32: return PlaneShape<T, NY, 32>::fits;
        case 64: return PlaneShape<T, NY, 64>::fits;
        case 128: return PlaneShape<T, NY, 128>::fits;
        case 256: return PlaneShape<T, NY, 256>::fits;
        case 512: return PlaneShape<T, NY, 512>::fits;
        default: return false;
    }
}
template <class T>
static bool fits_t(const Grid3 &g) {
    switch (g.ny) {
        case 16: return fits_ny<T, 16>(g.nz);
        case 32: return fits_ny<T, 32>(g.nz);
        case 64: return fits_ny<T, 64>(g.nz);
        case 128: return fits_ny<T, 128>(g.nz);
        case 256: return fits_ny<T, 256>(g.nz);
        default: return false;
    }
}

template <class T, int NY>
static int launch_ny(spk_ctx ctx, const Grid3 &g, const Twiddles &tw, int dir, const PassArgs &a) {
    switch (g.nz) {
        case 32: return launch_nynz<T, NY, 32>(ctx, g, tw, dir, a);
        case 64: return launch_nynz<T, NY, 64>(ctx, g, tw, dir, a);
        case 128: return launch_nynz<T, NY, 128>(ctx, g, tw, dir, a);
        case 256: return launch_nynz<T, NY, 256>(ctx, g, tw, dir, a);
        default: return launch_nynz<T, NY, 512>(ctx, g, tw, dir, a);
    }
}
template <class T>
static int launch_t(spk_ctx ctx, const Grid3 &g, const Twiddles &tw, int dir, const PassArgs &a) {
    switch (g.ny) {
        case 16: return launch_ny<T, 16>(ctx, g, tw, dir, a);
        case 32: return launch_ny<T, 32>(ctx, g, tw, dir, a);
        case 64: return launch_ny<T, 64>(ctx, g, tw, dir, a);
        case 128: return launch_ny<T, 128>(ctx, g, tw, dir, a);
        default: return launch_ny<T, 256>(ctx, g, tw, dir, a);
    }
}

bool plane_yz_supported(const Grid3 &g, int prec) { return prec == SPK_F64 ? fits_t<double>(g) : fits_t<float>(g); }

int launch_plane_yz(spk_ctx ctx, const Grid3 &g, const Twiddles &tw, int dir, const PassArgs &a) {
    SPK_REQUIRE(plane_yz_supported(g, tw.prec), SPK_ERR_STATE, "plane transform: %dx%d not supported", g.ny, g.nz);
    return tw.prec == SPK_F64 ? launch_t<double>(ctx, g, tw, dir, a) : launch_t<float>(ctx, g, tw, dir, a);
}

}  // namespace spk
