// spk_closure.hip -- learned subgrid-stress closure: a 4-layer 3D convolution
// network on the periodic n^3 grid of a filtered velocity field, BF16 weights
// and activations on the gfx950 matrix cores (v_mfma_f32_32x32x16_bf16) with
// FP32 accumulation; forward, backward (input and weight gradients) and Adam
// written here.
//
//   layer 1: 3 -> 32 channels, 3^3 taps, GELU
//   layers 2, 3: 32 -> 32, GELU
//   layer 4: 32 -> 6 (padded to 16), linear: the normalized stress
//            tau_xx, tau_xy, tau_xz, tau_yy, tau_yz, tau_zz
// Activations are channels-last [point][channel] BF16, point = (x n + y) n + z.
//
// Convolution as a GEMM per 4x4x32 brick of points: D[co][point] +=
// W[tap][co][ci-chunk] x X[point + tap][ci-chunk], 27 taps x (CIN / 16)
// K-chunks of 16 channels.  A block of 8 waves keeps all 27 taps' weights in LDS
// for its lifetime and stages each brick's input with a one-point halo; blocks
// loop over bricks.  16-byte LDS reads are conflict-free: the weights through an
// XOR swizzle of their 8-channel chunks by output channel, the halo at a padded
// point pitch.  The first layer's K runs over taps and its 3 (4) channels
// together, 7 K-chunks instead of 27.  The weight gradient contracts over points
// instead: dW[tap][co][ci] = sum_p dZ[p][co] X[p + tap][ci], its operands
// transposed by the LDS reads.
#include "spk_halo.hpp"
#include "spk_internal.hpp"
#include "spk_kernels.hpp"

#include <cmath>
#include <cstring>
#include <vector>

namespace spk {
namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int CH = 32;                   // hidden channels
constexpr int NTAP = 27;
constexpr int NBLK = 256;                // persistent blocks (one per CU)

__device__ __forceinline__ int swz(int q, int p) { return q ^ ((p >> 2) & (CH / 8 - 1)); }

// erfc(x) for x >= 0 by the Chebyshev fit of Press, Teukolsky, Vetterling and
// Flannery, Numerical Recipes (2nd ed., sec. 6.2, erfcc): fractional error below
// 1.2e-7 in exact arithmetic, below 1e-5 evaluated in FP32 up to x = 9; branch
// free, one reciprocal and one exponential.  The activations it feeds are
// rounded to BF16 (relative step 2^-8).
__device__ __forceinline__ float erfc_pos(float x) {
    const float t = __builtin_amdgcn_rcpf(1.0f + 0.5f * x);
    float p = 0.17087277f;
    p = fmaf(p, t, -0.82215223f);
    p = fmaf(p, t, 1.48851587f);
    p = fmaf(p, t, -1.13520398f);
    p = fmaf(p, t, 0.27886807f);
    p = fmaf(p, t, -0.18628806f);
    p = fmaf(p, t, 0.09678418f);
    p = fmaf(p, t, 0.37409196f);
    p = fmaf(p, t, 1.00002368f);
    p = fmaf(p, t, -1.26551223f);
    return t * __expf(fmaf(-x, x, p));
}
// Phi(z) = erfc(-z / sqrt 2) / 2, the normal distribution function
__device__ __forceinline__ float norm_cdf(float z) {
    const float e = 0.5f * erfc_pos(fabsf(z) * 0.70710678118654752f);
    return z > 0.0f ? 1.0f - e : e;
}
// GELU(z) = z Phi(z) = max(z, 0) - |z| exp(-z^2 / 2) Q(t), t = 1 / (1 + 0.3 |z|):
// Q is the minimax polynomial (relative error 5.7e-8 on |z| <= 13) of
// exp(z^2 / 2) erfc(|z| / sqrt 2) / 2, fitted for this.  In FP32 against 64 bits
// over |z| <= 12: largest error 2.4e-7, rms of the relative error for |z| < 4
// 1.8e-7 (z norm_cdf(z): 3.8e-7 and 2.5e-7), in two thirds of the instructions.
__device__ __forceinline__ float gelu(float z) {
    const float a = fminf(fabsf(z), 16.0f);  // past it the tail is 0 in FP32
    const float t = __builtin_amdgcn_rcpf(fmaf(a, 0.3f, 1.0f));
    float q = 0.0382711252f;
    q = fmaf(q, t, -0.168644095f);
    q = fmaf(q, t, 0.227579084f);
    q = fmaf(q, t, -0.0752666701f);
    q = fmaf(q, t, 0.141676423f);
    q = fmaf(q, t, 0.0950508391f);
    q = fmaf(q, t, 0.12182595f);
    q = fmaf(q, t, 0.119500989f);
    q = fmaf(q, t, 6.38356403e-06f);
    const float b = a * 0.84932180028801904f;  // sqrt(log2(e) / 2)
    const float r = a * (__builtin_amdgcn_exp2f(-b * b) * q);
    return z > -__builtin_inff() ? fmaxf(z, 0.0f) - r : __builtin_nanf("");  // NaN for NaN and, as z Phi(z), for -inf
}
// GELU'(z) = Phi(z) + z phi(z)
__device__ __forceinline__ float gelu_d(float z) {
    return norm_cdf(z) + z * 0.39894228040143268f * __expf(-0.5f * z * z);
}

__device__ __forceinline__ int wrap(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// Halo points of the hidden activations in LDS at a pitch of 80 bytes: the 16
// lanes of one 16-byte read cycle, on consecutive points, then fall on disjoint
// groups of 4 banks (64 banks of 4 bytes), and every tap's address is the lane's
// base address plus a constant, so the transform needs no per-tap address registers.
constexpr int XPITCH = CH + 8;
constexpr size_t CONV_LDS = (size_t)(NTAP * CH * CH + HX * HY * HZ * XPITCH) * sizeof(bf16) + CH * sizeof(float);

constexpr int CONV_T = 512;  // 8 waves, two per SIMD

// Bricks in the order that keeps halos in one XCD's L2: workgroups go to the 8
// XCDs round robin, so workgroup w is on XCD w % 8 and takes bricks of that XCD's
// eighth of the x range, x fastest, then z, then y: the bricks an XCD has at one
// time share their halos, and only the eighth's own edges are read twice.
struct Bricks {
    int n, sx, x0, k, step, count;
    __device__ Bricks(int n_) : n(n_) {
        sx = n / 32;  // bricks along x in an eighth
        x0 = (blockIdx.x & 7) * sx;
        k = blockIdx.x >> 3;
        step = gridDim.x >> 3;
        count = (n / 4) * (n / 4) * (n / 32) / 8;
    }
    __device__ bool live() const { return k < count; }
    __device__ bool more() const { return k + step < count; }
    __device__ void origin(int kk, int &x, int &y, int &z) const {
        const int r = kk / sx;
        x = (x0 + kk - r * sx) * 4;
        y = (r / sx) * 4;
        z = (r % sx) * 32;
    }
};

// One brick's input with its one-point halo (HX x HY x HZ points of CIN
// channels, channels-last, periodic wrap), held in the registers of NT threads
// between its global loads (fetch) and its LDS stores (stash), so that a block
// loads the next brick while it computes one.  The chunks' places in a brick
// (halo_place) are kept between bricks.
template <int CIN, int NT>
struct HaloPrefetch {
    static constexpr int NQ = CIN / 8;
    static constexpr int NCH = HX * HY * HZ * NQ;  // 16-byte chunks
    static constexpr int NPF = (NCH + NT - 1) / NT;
    bf16x8 v[NPF];
    int at[NPF];

    __device__ __forceinline__ HaloPrefetch(int n, int t) {
#pragma unroll
        for (int k = 0; k < NPF; k++) at[k] = halo_place(t + k * NT, n, NQ);
    }
    __device__ __forceinline__ void fetch(const bf16 *__restrict__ X, const Bricks &br, int kk, int t) {
        int x0, y0, z0;
        br.origin(kk, x0, y0, z0);
        unsigned o[NPF];
        halo_chunks(at, o, br.n, NQ, x0, y0, z0);
#pragma unroll
        for (int k = 0; k < NPF; k++)
            if (t + k * NT < NCH) v[k] = *reinterpret_cast<const bf16x8 *>(X + (size_t)o[k] * 8);
    }
    __device__ __forceinline__ void stash(bf16 *Xs, int t, int pitch) const {
#pragma unroll
        for (int k = 0; k < NPF; k++) {
            const int i = t + k * NT;
            if (i < NCH) *reinterpret_cast<bf16x8 *>(Xs + (i / NQ) * pitch + 8 * (i % NQ)) = v[k];
        }
    }
};

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
// swaps a's lanes 32..63 with b's lanes 0..31
__device__ __forceinline__ void swap_halves(unsigned &a, unsigned &b) {
    const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(a, b, false, false));
    a = r[0];
    b = r[1];
}
// A lane holds 4 channels (8 (r / 4) + 4 half + 0..3) of each of a point's four
// channel groups g; lanes li and li + 32 the two halves.  For 16-byte accesses to
// channels-last memory the pair exchanges groups: lane li then has the whole
// groups 0 and 1, lane li + 32 groups 2 and 3, 32 contiguous bytes each.
__device__ __forceinline__ void store_point(bf16 *__restrict__ P, int half, const bf16x4 (&v)[4]) {
    unsigned d[4][2];
    __builtin_memcpy(d, v, 32);
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int k = 0; k < 2; k++) swap_halves(d[g][k], d[g + 2][k]);
#pragma unroll
    for (int g = 0; g < 2; g++)
        *reinterpret_cast<u32x4 *>(P + 16 * half + 8 * g) = u32x4{d[g][0], d[g][1], d[g + 2][0], d[g + 2][1]};
}
__device__ __forceinline__ void load_point(const bf16 *__restrict__ P, int half, u32x4 (&raw)[2]) {
#pragma unroll
    for (int g = 0; g < 2; g++) raw[g] = *reinterpret_cast<const u32x4 *>(P + 16 * half + 8 * g);
}
__device__ __forceinline__ void spread_point(const u32x4 (&raw)[2], bf16x4 (&v)[4]) {
    unsigned d[4][2];
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
            unsigned a = raw[g][k], b = raw[g][k + 2];
            swap_halves(a, b);
            d[g][k] = a;
            d[g + 2][k] = b;
        }
    __builtin_memcpy(v, d, 32);
}

// Hidden layers and the input gradient, 32 -> 32 channels.
// MODE 0: Y = GELU(conv + b); 1: also Z = conv + b (training);
// 3: input gradient, Y = conv(dZ, flipped transposed W) * GELU'(Zp)
//
// What bounds it: per brick (512 points) the MFMAs, the LDS reads of their
// operands and the activation's VALU work are of one size, and a wave does them
// one after the other.  So the two waves of a SIMD take turns: waves 0-3 compute
// even bricks, waves 4-7 odd ones, and while one four has the matrix cores the
// other makes the activation and the stores of the brick it computed before.  A
// wave holds the four y columns of one x plane and takes the taps in groups of
// one (dx, dz) and one K-chunk: 6 input columns and 3 weight fragments feed 12
// MFMAs, half the LDS reads of a tap at a time.  With the brick order and 32-byte
// stores of a point, 128^3, 32 -> 32 channels: 165 -> 134 us, with the stored Z
// 180 -> 143, input gradient 190 -> 148.  Inputs in flight and out alone (no matrix
// work, no activation) take 77 us of that, the MFMAs 46.
template <int MODE>
__global__ __launch_bounds__(CONV_T) void k_conv(const bf16 *__restrict__ X, const bf16 *__restrict__ W,
                                                 const float *__restrict__ bias, bf16 *__restrict__ Y,
                                                 bf16 *__restrict__ Z, const bf16 *__restrict__ Zp, int n) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    bf16 *Ws = reinterpret_cast<bf16 *>(smem);  // [27][32][32], chunk-swizzled by co
    bf16 *Xs = Ws + NTAP * CH * CH;             // [HX*HY*HZ][XPITCH]
    float *Bs = reinterpret_cast<float *>(Xs + HX * HY * HZ * XPITCH);  // [32]
    constexpr int NQ = CH / 8, NKC = CH / 16, NG = 9 * NKC;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int xw = w & 3, four = w >> 2;
    const int li = lane & 31, half = lane >> 5;

    for (int i = tid; i < NTAP * CH * NQ; i += CONV_T) {
        const int q = i % NQ, row = i / NQ;
        const bf16x8 v = *reinterpret_cast<const bf16x8 *>(W + (size_t)row * CH + 8 * q);
        *reinterpret_cast<bf16x8 *>(Ws + row * CH + 8 * swz(q, row & 31)) = v;
    }
    Bricks br(n);
    if (MODE != 3 && tid < CH) Bs[tid] = bias[tid];

    f32x16 acc[4];
    // D[co][point]: lane holds point li of column ys, co = 8 (r / 4) + 4 half + r % 4
    auto finish = [&](int kk) {
        int x0, y0, z0;
        br.origin(kk, x0, y0, z0);
        const size_t p0 = ((size_t)(x0 + xw) * n + y0) * n + z0 + li;
        u32x4 zraw[MODE == 3 ? 4 : 1][2];
        if constexpr (MODE == 3)
#pragma unroll
            for (int ys = 0; ys < 4; ys++) load_point(Zp + (p0 + (size_t)ys * n) * CH, half, zraw[MODE == 3 ? ys : 0]);
#pragma unroll
        for (int ys = 0; ys < 4; ys++) {
            const size_t o = (p0 + (size_t)ys * n) * CH;
            bf16x4 y[4], zz[4];
            if constexpr (MODE == 3) spread_point(zraw[MODE == 3 ? ys : 0], zz);
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if constexpr (MODE == 3) {
                        y[g][j] = (bf16)(acc[ys][4 * g + j] * gelu_d((float)zz[g][j]));
                    } else {
                        const float zf = acc[ys][4 * g + j] + Bs[8 * g + 4 * half + j];
                        zz[g][j] = (bf16)zf;
                        y[g][j] = (bf16)gelu(zf);
                    }
                }
            store_point(Y + o, half, y);
            if constexpr (MODE == 1) store_point(Z + o, half, zz);
        }
    };
    auto matrix = [&]() {
#pragma unroll
        for (int ys = 0; ys < 4; ys++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[ys][r] = 0.0f;
        bf16x8 a[2][3], x[2][6];
        auto operands = [&](int g) {
            const int kc = g % NKC, dz = (g / NKC) % 3 - 1, dx = g / (3 * NKC) - 1;
            const int q = 2 * kc + half;
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
                const int t = 9 * (dx + 1) + 3 * dy + dz + 1;
                a[g & 1][dy] = *reinterpret_cast<const bf16x8 *>(Ws + (t * CH + li) * CH + 8 * swz(q, li));
            }
#pragma unroll
            for (int yy = 0; yy < 6; yy++) {
                const int hp = ((xw + 1 + dx) * HY + yy) * HZ + li + 1 + dz;
                x[g & 1][yy] = *reinterpret_cast<const bf16x8 *>(Xs + hp * XPITCH + 8 * q);
            }
        };
        operands(0);
#pragma unroll
        for (int g = 0; g < NG; g++) {
            // one group ahead and no further: more operands in flight would spill
            if (g + 1 < NG) operands(g + 1);
#pragma unroll
            for (int dy = 0; dy < 3; dy++)
#pragma unroll
                for (int ys = 0; ys < 4; ys++)
                    acc[ys] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[g & 1][dy], x[g & 1][ys + dy], acc[ys], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    HaloPrefetch<CH, CONV_T> hf(n, tid);
    if (br.live()) hf.fetch(X, br, br.k, tid);
    int turn = 0, last = -1;
    for (; br.live(); br.k += br.step, turn ^= 1) {
        __syncthreads();
        hf.stash(Xs, tid, XPITCH);
        __syncthreads();
        // the next brick's loads are in flight during this brick's matrix work (the
        // scheduling barrier keeps them ahead of it)
        if (br.more()) hf.fetch(X, br, br.k + br.step, tid);
        __builtin_amdgcn_sched_barrier(0);
        if (four == turn) {
            matrix();
        } else if (last >= 0) {
            finish(last);
        }
        last = br.k;
    }
    if (last >= 0 && four != turn) finish(last);
}

// First layer (3 channels, kept as 4): the contraction over (tap t, channel c) is
// one K index 4 t + c of 108, padded to 112, so 7 MFMAs make a column that 27
// K-chunks of 16 padded channels made before; a lane's 8 K values are two taps'
// points, two 8-byte LDS reads.  The weights stay in registers (28 of them), a
// brick's halo is 9.8 KB, and four blocks share a CU and overlap their loads,
// MFMAs, activation and stores, which bound it: 128^3, 108 -> 71 us.
constexpr int KIN = 7;  // K-chunks of 16
template <int MODE>
__global__ __launch_bounds__(256, 4) void k_conv_in(const bf16 *__restrict__ X, const bf16 *__restrict__ W,
                                                    const float *__restrict__ bias, bf16 *__restrict__ Y,
                                                    bf16 *__restrict__ Z, int n) {
    __shared__ bf16x4 Xs[HX * HY * HZ];
    __shared__ float Bs[CH];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, half = lane >> 5;
    Bricks br(n);
    int x0, y0, z0;
    br.origin(br.k, x0, y0, z0);
    for (int i = tid; i < HX * HY * HZ; i += 256) {
        const int hz = i % HZ, hy = (i / HZ) % HY, hx = i / (HZ * HY);
        const int gx = wrap(x0 + hx - 1, n), gy = wrap(y0 + hy - 1, n), gz = wrap(z0 + hz - 1, n);
        Xs[i] = *reinterpret_cast<const bf16x4 *>(X + (((size_t)gx * n + gy) * n + gz) * 4);
    }
    if (tid < CH) Bs[tid] = bias[tid];
    bf16x8 a[KIN];
    int off[KIN][2];  // halo points of the lane's two taps (the 28th, past the end, reads as 0)
#pragma unroll
    for (int kc = 0; kc < KIN; kc++) {
        a[kc] = *reinterpret_cast<const bf16x8 *>(W + (kc * CH + li) * 16 + 8 * half);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int t = 4 * kc + 2 * half + j, u = t < NTAP ? t : NTAP - 1;
            off[kc][j] = ((w + u / 9) * HY + (u / 3) % 3) * HZ + u % 3 + li;
        }
    }
    __syncthreads();
#pragma unroll 1
    for (int yp = 0; yp < 4; yp += 2) {
        f32x16 acc[2];
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[c][r] = 0.0f;
#pragma unroll
        for (int kc = 0; kc < KIN; kc++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const bf16x4 lo = Xs[off[kc][0] + (yp + c) * HZ];
                bf16x4 hi = Xs[off[kc][1] + (yp + c) * HZ];
                if (4 * kc + 3 >= NTAP && half) hi = bf16x4{};  // its weights are 0 too, but 0 inf is NaN
                const bf16x8 b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kc], b, acc[c], 0, 0, 0);
            }
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const size_t o = (((size_t)(x0 + w) * n + y0 + yp + c) * n + z0 + li) * CH;
            bf16x4 y[4], zz[4];
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float zf = acc[c][4 * g + j] + Bs[8 * g + 4 * half + j];
                    zz[g][j] = (bf16)zf;
                    y[g][j] = (bf16)gelu(zf);
                }
            store_point(Y + o, half, y);
            if constexpr (MODE == 1) store_point(Z + o, half, zz);
        }
    }
}

// its weights Wi[7][32 co][16]: K = 16 kc + kk = 4 t + c
__global__ void k_pack_in(const float *__restrict__ W, bf16 *__restrict__ Wi) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= KIN * CH * 16) return;
    const int kk = k % 16, co = (k / 16) % CH, K = 16 * (k / (16 * CH)) + kk;
    const int t = K / 4, c = K % 4;
    Wi[k] = t < NTAP && c < 3 ? (bf16)W[(t * CH + co) * 16 + c] : (bf16)0.0f;
}

// Output layer (32 -> 6 channels) on the 16-row matrix instruction
// v_mfma_f32_16x16x32_bf16: D[co < 16][16 points] += W[tap][co][32 ci] X[point + tap][32 ci],
// one instruction per tap and 16-point tile (the 6 stresses in rows 0..5), half
// the work of a 32-row tile.  out[c][p] = D + b for c < 6.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr size_t OUT_LDS = (size_t)(NTAP * 16 * CH + HX * HY * HZ * XPITCH) * sizeof(bf16);

// T = float: out[6][P], for the loss; T = double: the stresses themselves, times
// their scales, in the padded real layout [6][n][n][n + 2] (pads 0), so that no
// second pass converts them (128^3: 134 + 45 us -> 126; float 126 -> 100).
struct OutScale {
    double s[6];
};
template <class T>
__global__ __launch_bounds__(CONV_T) void k_conv_out(const bf16 *__restrict__ X, const bf16 *__restrict__ W,
                                                     const float *__restrict__ bias, T *__restrict__ out, int n,
                                                     OutScale sc) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    bf16 *Ws = reinterpret_cast<bf16 *>(smem);  // [27][16][32], chunk-swizzled by co
    bf16 *Xs = Ws + NTAP * 16 * CH;             // [HX*HY*HZ][XPITCH]
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int l16 = lane & 15, q = lane >> 4;   // 16x16x32: lane holds row/column l16, K chunk q
    const int xw = w & 3, yg = 2 * (w >> 2);

    for (int i = tid; i < NTAP * 16 * 4; i += CONV_T) {
        const int qq = i & 3, row = i >> 2;  // row = t * 16 + co
        const int t = row >> 4, co = row & 15;
        const bf16x8 v = *reinterpret_cast<const bf16x8 *>(W + ((size_t)t * CH + co) * CH + 8 * qq);
        *reinterpret_cast<bf16x8 *>(Ws + row * CH + 8 * swz(qq, co)) = v;
    }
    Bricks br(n);
    const size_t P = (size_t)n * n * n;
    HaloPrefetch<CH, CONV_T> hf(n, tid);
    if (br.live()) hf.fetch(X, br, br.k, tid);
    for (; br.live(); br.k += br.step) {
        int x0, y0, z0;
        br.origin(br.k, x0, y0, z0);
        __syncthreads();
        hf.stash(Xs, tid, XPITCH);
        __syncthreads();
        if (br.more()) hf.fetch(X, br, br.k + br.step, tid);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 acc[2][2];  // [column][16-point half]
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[c][h][r] = 0.0f;
        // taps in groups of one (dx, dz): 4 input columns and 3 weight fragments feed
        // 12 MFMAs
#pragma unroll
        for (int g = 0; g < 9; g++) {
            const int dx = g / 3 - 1, dz = g % 3 - 1;
            bf16x8 a[3], x[4][2];
#pragma unroll
            for (int dy = 0; dy < 3; dy++)
                a[dy] = *reinterpret_cast<const bf16x8 *>(
                    Ws + ((9 * (dx + 1) + 3 * dy + dz + 1) * 16 + l16) * CH + 8 * swz(q, l16));
#pragma unroll
            for (int yy = 0; yy < 4; yy++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int hp = ((xw + 1 + dx) * HY + yg + yy) * HZ + 16 * h + l16 + 1 + dz;
                    x[yy][h] = *reinterpret_cast<const bf16x8 *>(Xs + hp * XPITCH + 8 * q);
                }
#pragma unroll
            for (int dy = 0; dy < 3; dy++)
#pragma unroll
                for (int c = 0; c < 2; c++)
#pragma unroll
                    for (int h = 0; h < 2; h++)
                        acc[c][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[dy], x[c + dy][h], acc[c][h], 0, 0, 0);
        }
        // D[co][point]: lane holds point l16 of its half, co = 4 q + r
        if (q < 2) {
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    constexpr bool PAD = sizeof(T) == 8;
                    const int z = z0 + 16 * h + l16;
                    const size_t row = (size_t)(x0 + xw) * n + (y0 + yg + c);
                    const size_t p = row * (PAD ? n + 2 : n) + z, fs = PAD ? (size_t)n * n * (n + 2) : P;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int co = 4 * q + r;
                        if (co < 6) {
                            const float v = acc[c][h][r] + bias[co];
                            if constexpr (PAD) {
                                const double s = r == 0 ? (q ? sc.s[4] : sc.s[0]) : r == 1 ? (q ? sc.s[5] : sc.s[1]) : sc.s[r];
                                out[co * fs + p] = (double)v * s;
                                if (z == n - 1) out[co * fs + p + 1] = out[co * fs + p + 2] = 0.0;
                            } else {
                                out[co * fs + p] = v;
                            }
                        }
                    }
                }
        }
    }
}

// Weight gradient, per-block partial sums part[block][27][32 co][32 ci], and the
// bias gradient's bpart[block][32 co].  Both operands contract over points, so a
// lane needs 8 points of one channel, while memory and LDS are channels-last: the
// bricks are staged as they come, in 16-byte rows of 64-byte points, and the
// transposing LDS read (ds_read_b64_tr_b16: 16 lanes give 4 points x 16 channels
// and receive one channel's 4 points each) makes the fragments; a point pitch of
// 64 bytes puts the 4 points of 32 lanes on all 64 banks once.  A tap's z shift is
// an address, and the bias gradient is a 28th tap whose input is 1.  Staged
// channel-major by 2-byte stores, with the shifts made in registers, half of the
// LDS time was bank conflicts: 290 -> 156 us at 128^3, 32 channels, no conflicts
// left; the MFMAs take 48 us of that.
constexpr size_t dw_lds(int cin) { return (size_t)(512 * CH + HX * HY * HZ * cin) * sizeof(bf16); }

typedef short s16x4 __attribute__((ext_vector_type(4)));
// rows p, p + 1, p + 2, p + 3 (pitch elements apart) of the lane's 16 channels: see above
__device__ __forceinline__ bf16x8 tr_points8(const bf16 *p, int pitch) {
    typedef __attribute__((address_space(3))) s16x4 *lds_p;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_p)p);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_p)(p + 4 * pitch));
    bf16x8 v;
    __builtin_memcpy(&v, &lo, 8);
    __builtin_memcpy((char *)&v + 8, &hi, 8);
    return v;
}

template <int CIN>
__global__ __launch_bounds__(CONV_T) void k_conv_dw(const bf16 *__restrict__ X, const bf16 *__restrict__ dZ,
                                                 float *__restrict__ part, float *__restrict__ bpart, int n) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    bf16 *Ds = reinterpret_cast<bf16 *>(smem);  // [512 points][32 co]: point (bx 4 + by) 32 + z
    bf16 *Xs = Ds + 512 * CH;                   // [HX HY HZ points][CIN]
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, half = lane >> 5;
    // the lane's part of a transposing read: point 8 half + (lane / 4) % 4 of 16, and
    // 4 channels of its 16 (with 16 input channels the upper ones are 0)
    const int rp = 8 * half + ((lane >> 2) & 3), chg = (lane >> 4) & 1, c4 = 4 * (lane & 3);
    const bf16 *pa = Ds + rp * CH + 16 * chg + c4;
    const bf16 *pb = Xs + rp * CIN + (CIN == 32 ? 16 * chg : 0) + c4;
    f32x16 acc[4];  // taps w, w + 8, w + 16, w + 24 of wave w
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[k][r] = 0.0f;
    int toff[4];  // a tap's shift in the halo, elements
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int t = w + 8 * k;
        toff[k] = (((t / 9) * HY + (t / 3) % 3) * HZ + t % 3) * CIN;
    }
    bf16x8 ones;
#pragma unroll
    for (int j = 0; j < 8; j++) ones[j] = (bf16)1.0f;
    float bsum = 0.0f;  // bias gradient of co = li: the bricks' sums are added up apart from the 32 steps within one
    Bricks br(n);
    HaloPrefetch<CIN, CONV_T> hf(n, tid);
    constexpr int NPD = 512 * 4 / CONV_T;  // dZ chunks of 8 channels per thread
    bf16x8 pd[NPD];
    auto fetch_dz = [&](int kk) {
        int x0, y0, z0;
        br.origin(kk, x0, y0, z0);
#pragma unroll
        for (int k = 0; k < NPD; k++) {
            const int i = tid + k * CONV_T;
            const int q = i & 3, pt = i >> 2;
            const size_t p = ((size_t)(x0 + (pt >> 7)) * n + y0 + ((pt >> 5) & 3)) * n + z0 + (pt & 31);
            pd[k] = *reinterpret_cast<const bf16x8 *>(dZ + p * CH + 8 * q);
        }
    };
    if (br.live()) {
        fetch_dz(br.k);
        hf.fetch(X, br, br.k, tid);
    }
    for (; br.live(); br.k += br.step) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NPD; k++) *reinterpret_cast<bf16x8 *>(Ds + 8 * (tid + k * CONV_T)) = pd[k];
        hf.stash(Xs, tid, CIN);
        __syncthreads();
        // the next brick's loads are in flight during this brick's matrix work
        if (br.more()) {
            fetch_dz(br.k + br.step);
            hf.fetch(X, br, br.k + br.step, tid);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll 4
        for (int s = 0; s < 32; s++) {
            const int col = s >> 1, zr = 16 * (s & 1);
            const bf16x8 a = tr_points8(pa + (col * 32 + zr) * CH, CH);
            const bf16 *xb = pb + (((col >> 2) * HY + (col & 3)) * HZ + zr) * CIN;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int t = w + 8 * k;
                if (k < 3 || t < NTAP) {
                    bf16x8 b = tr_points8(xb + toff[k], CIN);
                    if constexpr (CIN == 16) {
                        if (chg) b = bf16x8{};
                    }
                    acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[k], 0, 0, 0);
                } else if (t == NTAP) {
                    acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, a, acc[k], 0, 0, 0);  // rows alike
                }
            }
        }
        if (w + 24 == NTAP) {
            bsum += acc[3][0];
#pragma unroll
            for (int r = 0; r < 16; r++) acc[3][r] = 0.0f;
        }
    }
    // D[co][ci]: lane holds ci = li, co = 8 (r / 4) + 4 half + r % 4
    float *pb_ = part + (size_t)blockIdx.x * NTAP * CH * CH;
    if (w + 24 == NTAP && half == 0) bpart[(size_t)blockIdx.x * CH + li] = bsum;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int t = w + 8 * k;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int co = 8 * (r / 4) + 4 * half + (r & 3);
            if (t < NTAP) pb_[((size_t)t * CH + co) * CH + li] = acc[k][r];
        }
    }
}

__global__ void k_fill0(float *__restrict__ p, int count) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < count) p[k] = 0.0f;
}

// grad[k] += sum over slice blockIdx.y of the parts: part[b][k] (grad zeroed before)
constexpr int SUM_SLICES = 16;
__global__ void k_sum_parts(const float *__restrict__ part, int nparts, int count, float *__restrict__ grad) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    const int per = (nparts + SUM_SLICES - 1) / SUM_SLICES;
    const int b0 = blockIdx.y * per, b1 = b0 + per < nparts ? b0 + per : nparts;
    float s = 0.0f;
    for (int b = b0; b < b1; b++) s += part[(size_t)b * count + k];
    atomicAdd(&grad[k], s);
}

// padded real FP64 u [3][n][n][n + 2] -> BF16 [P][4] (channel 3 zero) for the first
// layer, and [P][16] (channels 3..15 zero) for its weight gradient; times in_scale
__global__ void k_pack_input(const double *__restrict__ u, bf16 *__restrict__ xin4, bf16 *__restrict__ xin, int n,
                             float in_scale) {
    const size_t P = (size_t)n * n * n;
    const size_t fs = (size_t)n * n * (n + 2);
    for (size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x; p < P; p += (size_t)gridDim.x * blockDim.x) {
        const size_t o = p + 2 * (p / n);
        bf16x4 v;
        v[0] = (bf16)((float)u[o] * in_scale);
        v[1] = (bf16)((float)u[fs + o] * in_scale);
        v[2] = (bf16)((float)u[2 * fs + o] * in_scale);
        v[3] = (bf16)0.0f;
        *reinterpret_cast<bf16x4 *>(xin4 + p * 4) = v;
        if (xin) {
            bf16x8 v0, v1;
            for (int j = 0; j < 8; j++) v0[j] = v1[j] = (bf16)0.0f;
            for (int j = 0; j < 3; j++) v0[j] = v[j];
            *reinterpret_cast<bf16x8 *>(xin + p * 16) = v0;
            *reinterpret_cast<bf16x8 *>(xin + p * 16 + 8) = v1;
        }
    }
}

// loss = mean over 6 P of (pred - tgt)^2, tgt = tau / scale from the padded real
// layout; dZ4[p][c] = 2 (pred - tgt) / (6 P) (c < 6, else 0)
constexpr int LOSS_T = 1024;
__global__ __launch_bounds__(LOSS_T) void k_loss(const float *__restrict__ pred, const double *__restrict__ tau,
                                                 bf16 *__restrict__ dz, int n, OutScale sc, float *__restrict__ part) {
    __shared__ float sm[LOSS_T];
    float acc = 0.0f;
    const size_t P = (size_t)n * n * n, fs = (size_t)n * n * (n + 2);
    const float g = 2.0f / (6.0f * (float)P);
    for (size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x; p < P; p += (size_t)gridDim.x * blockDim.x) {
        const size_t o = p + 2 * (p / n);
        bf16x8 v0, v1;
        for (int j = 0; j < 8; j++) v0[j] = v1[j] = (bf16)0.0f;
#pragma unroll
        for (int c = 0; c < 6; c++) {
            const float d = pred[(size_t)c * P + p] - (float)(tau[(size_t)c * fs + o] / sc.s[c]);
            acc += d * d;
            v0[c] = (bf16)(g * d);
        }
        bf16 *q = dz + p * CH;
        *reinterpret_cast<bf16x8 *>(q) = v0;
        *reinterpret_cast<bf16x8 *>(q + 8) = v1;
        *reinterpret_cast<bf16x8 *>(q + 16) = v1;
        *reinterpret_cast<bf16x8 *>(q + 24) = v1;
    }
    sm[threadIdx.x] = acc;
    __syncthreads();
    for (int s = LOSS_T / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sm[threadIdx.x] += sm[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sm[0];
}

// Adam (Kingma & Ba) on the FP32 master parameters
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m, float *__restrict__ v,
                       int count, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    const float gk = g[k];
    const float mk = b1 * m[k] + (1.0f - b1) * gk;
    const float vk = b2 * v[k] + (1.0f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    w[k] -= lr * (mk / c1) / (sqrtf(vk / c2) + eps);
}

// BF16 weights of one layer from its FP32 master weights W[27][32][cin]; and the
// flipped transpose WT[26 - t][ci][co] = W[t][co][ci] (cin = 32) for the input gradient
__global__ void k_pack_weights(const float *__restrict__ W, bf16 *__restrict__ Wb, bf16 *__restrict__ WT, int cin) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= NTAP * CH * cin) return;
    const int ci = k % cin, co = (k / cin) % CH, t = k / (cin * CH);
    const bf16 v = (bf16)W[k];
    Wb[k] = v;
    if (WT) WT[((NTAP - 1 - t) * CH + ci) * CH + co] = v;
}

// ---- filtered DNS data: truncation to a coarse grid, products, SGS divergence ----

// coarse-grid index -> fine-grid index of the same wavenumber along one axis;
// -1 where the coarse mode is cut (beyond |k| <= kc, or the coarse Nyquist)
__device__ __forceinline__ long long fine_of(int i, int n, int N, int kc) {
    const int k = i < n / 2 ? i : i - n;
    if (i == n / 2 || (k < 0 ? -k : k) > kc) return -1;
    return k >= 0 ? k : k + N;
}

// lo[f][i][j][k] = scale * hi[f][fine(i)][fine(j)][k] on the modes kept, 0 elsewhere
// (complex, [NX][NY][NZ/2+1] layouts; hi at stride fs_hi, lo at stride fs_lo)
__global__ void k_truncate(const cpx<double> *__restrict__ hi, int N, long long fs_hi, cpx<double> *__restrict__ lo,
                           int n, long long fs_lo, int nf, int kc, double scale) {
    const long long ntc = (long long)n * n * (n / 2 + 1);
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < ntc * nf;
         e += (long long)gridDim.x * blockDim.x) {
        const int f = (int)(e / ntc);
        const long long idx = e - (long long)f * ntc;
        const int k = (int)(idx % (n / 2 + 1));
        const long long r = idx / (n / 2 + 1);
        const int j = (int)(r % n), i = (int)(r / n);
        const long long fi = fine_of(i, n, N, kc), fj = fine_of(j, n, N, kc);
        const bool keep = fi >= 0 && fj >= 0 && k < n / 2 && k <= kc;
        cpx<double> v = {0.0, 0.0};
        if (keep) {
            const cpx<double> h = hi[(long long)f * fs_hi + (fi * N + fj) * (N / 2 + 1) + k];
            v = cpx<double>{h.x * scale, h.y * scale};
        }
        lo[(long long)f * fs_lo + idx] = v;
    }
}

// the same cut applied on the fine grid itself (modes beyond kc set to 0)
__global__ void k_mask_fine(const cpx<double> *__restrict__ in, cpx<double> *__restrict__ out, int N, long long fs,
                            int nf, int kc) {
    const long long ntc = (long long)N * N * (N / 2 + 1);
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < ntc * nf;
         e += (long long)gridDim.x * blockDim.x) {
        const int f = (int)(e / ntc);
        const long long idx = e - (long long)f * ntc;
        const int k = (int)(idx % (N / 2 + 1));
        const long long r = idx / (N / 2 + 1);
        const int j = (int)(r % N), i = (int)(r / N);
        const int kx = i < N / 2 ? i : i - N, ky = j < N / 2 ? j : j - N;
        const bool keep = (kx < 0 ? -kx : kx) <= kc && (ky < 0 ? -ky : ky) <= kc && k <= kc;
        out[(long long)f * fs + idx] = keep ? in[(long long)f * fs + idx] : cpx<double>{0.0, 0.0};
    }
}

// padded real rows: out = a_i a_j - b_i b_j (fields i, j of a and b at stride fs)
__global__ void k_stress_prod(const double *__restrict__ a, const double *__restrict__ b, double *__restrict__ out,
                              long long fs, int i, int j) {
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < fs; e += (long long)gridDim.x * blockDim.x)
        out[e] = a[i * fs + e] * a[j * fs + e] - b[i * fs + e] * b[j * fs + e];
}

// U_i += dt P(-i mask k_j tau_ij) for the velocity of a solver (tau: 6 spectral
// fields xx xy xz yy yz zz at stride ntc); P the projection on k-perpendicular
__global__ __launch_bounds__(256) void k_sgs_update(cpx<double> *__restrict__ U, const cpx<double> *__restrict__ T,
                                                    long long ntc, KGeom kg, const TimeState *__restrict__ ts) {
    const double dt = ts->dt;
    for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < ntc;
         idx += (long long)gridDim.x * blockDim.x) {
        const long long rowi = idx / kg.nzh;
        const int k = (int)(idx - rowi * kg.nzh);
        const int j = (int)(rowi % kg.ny), i = (int)(rowi / kg.ny);
        double kx, ky, kz, m;
        kvec_at(kg, i, j, k, kx, ky, kz, m);
        const cpx<double> t0 = T[idx], t1 = T[ntc + idx], t2 = T[2 * ntc + idx], t3 = T[3 * ntc + idx],
                          t4 = T[4 * ntc + idx], t5 = T[5 * ntc + idx];
        const cpx<double> d0 = kdot3(kx, t0, ky, t1, kz, t2);
        const cpx<double> d1 = kdot3(kx, t1, ky, t3, kz, t4);
        const cpx<double> d2 = kdot3(kx, t2, ky, t4, kz, t5);
        // -i m d
        cpx<double> g[3] = {{m * d0.y, -m * d0.x}, {m * d1.y, -m * d1.x}, {m * d2.y, -m * d2.x}};
        const double k2 = kx * kx + ky * ky + kz * kz;
        if (k2 > 0.0) {
            const cpx<double> kg_ = kdot3(kx, g[0], ky, g[1], kz, g[2]);
            const double kk[3] = {kx, ky, kz};
#pragma unroll
            for (int q = 0; q < 3; q++) g[q] = cpx<double>{g[q].x - kk[q] * kg_.x / k2, g[q].y - kk[q] * kg_.y / k2};
        }
#pragma unroll
        for (int q = 0; q < 3; q++) {
            cpx<double> &u = U[q * ntc + idx];
            u = cpx<double>{u.x + dt * g[q].x, u.y + dt * g[q].y};
        }
    }
}

}  // namespace
}  // namespace spk

using namespace spk;

// parameter layout: for layer l = 1..4: W_l[27][32][cin_l] then b_l[32]; cin = 16, 32, 32, 32
static const int CIN_L[4] = {16, 32, 32, 32};
static size_t w_count(int l) { return (size_t)NTAP * CH * CIN_L[l]; }
static size_t param_offset(int l) {
    size_t o = 0;
    for (int i = 0; i < l; i++) o += w_count(i) + CH;
    return o;
}
static size_t param_total() { return param_offset(4); }

struct spk_closure_s {
    spk_ctx ctx = nullptr;
    int n = 0;
    size_t P = 0;
    double in_scale = 1.0, out_scale[6] = {1, 1, 1, 1, 1, 1};
    float *prm = nullptr, *grd = nullptr, *am = nullptr, *av = nullptr;  // FP32 master, gradient, Adam moments
    bf16 *Wb[4] = {}, *WT[4] = {};
    bf16 *xin = nullptr, *xin4 = nullptr, *Z[3] = {}, *A[3] = {}, *dzA = nullptr, *dzB = nullptr;
    float *out = nullptr, *part = nullptr, *bpart = nullptr, *lpart = nullptr;
    int adam_t = 0;
    double *tau = nullptr;          // coupling: padded real stresses [6][n][n][n + 2], transformed in place
    spk_fft_plan plan6 = nullptr;   // FP64 n^3 transforms of 6 fields
};

namespace {

int closure_alloc(spk_closure c) {
    auto al = [&](void **p, size_t bytes) -> int {
        if (hipMalloc(p, bytes) != hipSuccess) {
            *p = nullptr;
            set_error("spk_closure: hipMalloc(%zu) failed", bytes);
            return SPK_ERR_ALLOC;
        }
        return SPK_OK;
    };
    const size_t NP = param_total();
    SPK_TRY(al((void **)&c->prm, NP * 4));
    SPK_TRY(al((void **)&c->grd, NP * 4));
    SPK_TRY(al((void **)&c->am, NP * 4));
    SPK_TRY(al((void **)&c->av, NP * 4));
    for (int l = 0; l < 4; l++) {
        SPK_TRY(al((void **)&c->Wb[l], (l ? w_count(l) : (size_t)KIN * CH * 16) * 2));
        if (l > 0) SPK_TRY(al((void **)&c->WT[l], w_count(l) * 2));
    }
    SPK_TRY(al((void **)&c->xin, c->P * 16 * 2));
    SPK_TRY(al((void **)&c->xin4, c->P * 4 * 2));
    for (int l = 0; l < 3; l++) {
        SPK_TRY(al((void **)&c->Z[l], c->P * CH * 2));
        SPK_TRY(al((void **)&c->A[l], c->P * CH * 2));
    }
    SPK_TRY(al((void **)&c->dzA, c->P * CH * 2));
    SPK_TRY(al((void **)&c->dzB, c->P * CH * 2));
    SPK_TRY(al((void **)&c->out, c->P * 6 * 4));
    SPK_TRY(al((void **)&c->part, (size_t)NBLK * NTAP * CH * CH * 4));
    SPK_TRY(al((void **)&c->bpart, (size_t)NBLK * CH * 4));
    SPK_TRY(al((void **)&c->lpart, (size_t)NBLK * 4));
    SPK_HIP(hipMemsetAsync(c->prm, 0, NP * 4, c->ctx->stream));
    SPK_HIP(hipMemsetAsync(c->am, 0, NP * 4, c->ctx->stream));
    SPK_HIP(hipMemsetAsync(c->av, 0, NP * 4, c->ctx->stream));
    return SPK_OK;
}

void closure_free(spk_closure c) {
    if (c->plan6) spk_fft_plan_destroy(c->plan6);
    void *b[] = {c->prm, c->grd, c->am, c->av, c->xin, c->xin4, c->dzA, c->dzB, c->out, c->part, c->bpart, c->lpart,
                 c->tau};
    for (void *p : b)
        if (p) (void)hipFree(p);
    for (int l = 0; l < 4; l++) {
        if (c->Wb[l]) (void)hipFree(c->Wb[l]);
        if (c->WT[l]) (void)hipFree(c->WT[l]);
    }
    for (int l = 0; l < 3; l++) {
        if (c->Z[l]) (void)hipFree(c->Z[l]);
        if (c->A[l]) (void)hipFree(c->A[l]);
    }
}

int set_lds_attributes() {
    static bool done = false;
    if (done) return SPK_OK;
    SPK_HIP(hipFuncSetAttribute((const void *)k_conv<0>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)CONV_LDS));
    SPK_HIP(hipFuncSetAttribute((const void *)k_conv<1>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)CONV_LDS));
    SPK_HIP(hipFuncSetAttribute((const void *)k_conv_out<float>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)OUT_LDS));
    SPK_HIP(hipFuncSetAttribute((const void *)k_conv_out<double>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)OUT_LDS));
    SPK_HIP(hipFuncSetAttribute((const void *)k_conv<3>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)CONV_LDS));
    SPK_HIP(hipFuncSetAttribute((const void *)k_conv_dw<16>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)dw_lds(16)));
    SPK_HIP(hipFuncSetAttribute((const void *)k_conv_dw<32>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)dw_lds(32)));
    done = true;
    return SPK_OK;
}

int pack_weights(spk_closure c) {
    k_pack_in<<<(KIN * CH * 16 + 255) / 256, 256, 0, c->ctx->stream>>>(c->prm, c->Wb[0]);
    for (int l = 1; l < 4; l++) {
        const int cnt = (int)w_count(l);
        k_pack_weights<<<(cnt + 255) / 256, 256, 0, c->ctx->stream>>>(c->prm + param_offset(l), c->Wb[l], c->WT[l],
                                                                     CIN_L[l]);
    }
    SPK_LAUNCH_CHECK();
    return SPK_OK;
}

unsigned conv_grid(spk_closure c) {
    const int nb = (c->n / 4) * (c->n / 4) * (c->n / 32);
    return (unsigned)(nb < NBLK ? nb : NBLK);
}

OutScale out_scale_of(spk_closure c) {
    OutScale s;
    for (int i = 0; i < 6; i++) s.s[i] = c->out_scale[i];
    return s;
}

// tau: the stresses (inference); nullptr: training, the normalized stresses into c->out
int forward(spk_closure c, const void *u, double *tau) {
    const bool train = tau == nullptr;
    hipStream_t st = c->ctx->stream;
    const unsigned gp = (unsigned)((c->P + 255) / 256 < 4096 ? (c->P + 255) / 256 : 4096);
    k_pack_input<<<gp, 256, 0, st>>>((const double *)u, c->xin4, train ? c->xin : nullptr, c->n, (float)c->in_scale);
    const unsigned gin = (unsigned)((c->n / 4) * (c->n / 4) * (c->n / 32));
    const unsigned g = conv_grid(c);
    const float *b[4];
    for (int l = 0; l < 4; l++) b[l] = c->prm + param_offset(l) + w_count(l);
    if (train) {
        k_conv_in<1><<<gin, 256, 0, st>>>(c->xin4, c->Wb[0], b[0], c->A[0], c->Z[0], c->n);
        k_conv<1><<<g, CONV_T, CONV_LDS, st>>>(c->A[0], c->Wb[1], b[1], c->A[1], c->Z[1], nullptr, c->n);
        k_conv<1><<<g, CONV_T, CONV_LDS, st>>>(c->A[1], c->Wb[2], b[2], c->A[2], c->Z[2], nullptr, c->n);
    } else {
        k_conv_in<0><<<gin, 256, 0, st>>>(c->xin4, c->Wb[0], b[0], c->A[0], nullptr, c->n);
        k_conv<0><<<g, CONV_T, CONV_LDS, st>>>(c->A[0], c->Wb[1], b[1], c->A[1], nullptr, nullptr, c->n);
        k_conv<0><<<g, CONV_T, CONV_LDS, st>>>(c->A[1], c->Wb[2], b[2], c->A[2], nullptr, nullptr, c->n);
    }
    if (train) k_conv_out<float><<<g, CONV_T, OUT_LDS, st>>>(c->A[2], c->Wb[3], b[3], c->out, c->n, out_scale_of(c));
    else k_conv_out<double><<<g, CONV_T, OUT_LDS, st>>>(c->A[2], c->Wb[3], b[3], tau, c->n, out_scale_of(c));
    SPK_LAUNCH_CHECK();
    return SPK_OK;
}

// weight and bias gradients of layer l from its input X and its dZ, into grd
int layer_grads(spk_closure c, int l, const bf16 *X, const bf16 *dz) {
    hipStream_t st = c->ctx->stream;
    const unsigned g = conv_grid(c);
    if (CIN_L[l] == 16) k_conv_dw<16><<<g, CONV_T, dw_lds(CIN_L[l]), st>>>(X, dz, c->part, c->bpart, c->n);
    else k_conv_dw<32><<<g, CONV_T, dw_lds(CIN_L[l]), st>>>(X, dz, c->part, c->bpart, c->n);
    const int cnt = NTAP * CH * CH;
    // the [27][32][32] sums land in grd for cin = 32; for cin = 16 take ci < 16
    float *gw = c->grd + param_offset(l);
    const dim3 sg((cnt + 255) / 256, SUM_SLICES);
    float *sum_to = CIN_L[l] == 32 ? gw : c->out;  // out is free here
    k_fill0<<<(cnt + 255) / 256, 256, 0, st>>>(sum_to, cnt);
    k_sum_parts<<<sg, 256, 0, st>>>(c->part, (int)g, cnt, sum_to);
    if (CIN_L[l] != 32)
        SPK_HIP(hipMemcpy2DAsync(gw, 16 * 4, c->out, 32 * 4, 16 * 4, NTAP * CH, hipMemcpyDeviceToDevice, st));
    // the bias partials came from the same kernel (k_conv_dw), one per block
    k_fill0<<<1, CH, 0, st>>>(gw + w_count(l), CH);
    k_sum_parts<<<dim3(1, SUM_SLICES), CH, 0, st>>>(c->bpart, (int)g, CH, gw + w_count(l));
    SPK_LAUNCH_CHECK();
    return SPK_OK;
}

}  // namespace

extern "C" size_t spk_closure_num_params(void) { return param_total(); }

extern "C" int spk_closure_create(spk_ctx ctx, int n, spk_closure *out) {
    SPK_REQUIRE(ctx && out, SPK_ERR_ARG, "spk_closure_create: null argument");
    SPK_REQUIRE(n >= 32 && n % 32 == 0 && n <= 1024, SPK_ERR_ARG,
                "spk_closure_create: n = %d (a multiple of 32, 32..1024)", n);
    SPK_TRY(set_lds_attributes());
    spk_closure c = new spk_closure_s();
    c->ctx = ctx;
    c->n = n;
    c->P = (size_t)n * n * n;
    const int rc = closure_alloc(c);
    if (rc != SPK_OK) {
        closure_free(c);
        delete c;
        return rc;
    }
    ctx_retain(ctx);
    *out = c;
    return pack_weights(c);
}

extern "C" int spk_closure_destroy(spk_closure c) {
    if (!c) return SPK_OK;
    (void)hipStreamSynchronize(c->ctx->stream);
    closure_free(c);
    spk_ctx cx = c->ctx;
    delete c;
    ctx_release(cx);
    return SPK_OK;
}

extern "C" int spk_closure_set_params(spk_closure c, const float *host) {
    SPK_REQUIRE(c && host, SPK_ERR_ARG, "spk_closure_set_params: null argument");
    SPK_HIP(hipMemcpyAsync(c->prm, host, param_total() * 4, hipMemcpyHostToDevice, c->ctx->stream));
    SPK_HIP(hipMemsetAsync(c->am, 0, param_total() * 4, c->ctx->stream));
    SPK_HIP(hipMemsetAsync(c->av, 0, param_total() * 4, c->ctx->stream));
    c->adam_t = 0;
    SPK_TRY(pack_weights(c));
    SPK_HIP(hipStreamSynchronize(c->ctx->stream));
    return SPK_OK;
}

extern "C" int spk_closure_get_params(spk_closure c, float *host) {
    SPK_REQUIRE(c && host, SPK_ERR_ARG, "spk_closure_get_params: null argument");
    SPK_HIP(hipMemcpyAsync(host, c->prm, param_total() * 4, hipMemcpyDeviceToHost, c->ctx->stream));
    SPK_HIP(hipStreamSynchronize(c->ctx->stream));
    return SPK_OK;
}

extern "C" int spk_closure_get_grads(spk_closure c, float *host) {
    SPK_REQUIRE(c && host, SPK_ERR_ARG, "spk_closure_get_grads: null argument");
    SPK_HIP(hipMemcpyAsync(host, c->grd, param_total() * 4, hipMemcpyDeviceToHost, c->ctx->stream));
    SPK_HIP(hipStreamSynchronize(c->ctx->stream));
    return SPK_OK;
}

extern "C" int spk_closure_set_scales(spk_closure c, double in_scale, const double *out_scale) {
    SPK_REQUIRE(c && out_scale && in_scale > 0, SPK_ERR_ARG, "spk_closure_set_scales: bad arguments");
    c->in_scale = in_scale;
    for (int i = 0; i < 6; i++) {
        SPK_REQUIRE(out_scale[i] > 0, SPK_ERR_ARG, "spk_closure_set_scales: out_scale[%d] <= 0", i);
        c->out_scale[i] = out_scale[i];
    }
    return SPK_OK;
}

extern "C" int spk_closure_forward(spk_closure c, const void *u, void *tau) {
    SPK_REQUIRE(c && u && tau, SPK_ERR_ARG, "spk_closure_forward: null argument");
    return forward(c, u, (double *)tau);
}

extern "C" int spk_closure_grads(spk_closure c, const void *u, const void *tau_true, double *loss) {
    SPK_REQUIRE(c && u && tau_true, SPK_ERR_ARG, "spk_closure_grads: null argument");
    hipStream_t st = c->ctx->stream;
    SPK_TRY(forward(c, u, nullptr));
    k_loss<<<NBLK, LOSS_T, 0, st>>>(c->out, (const double *)tau_true, c->dzA, c->n, out_scale_of(c), c->lpart);
    SPK_LAUNCH_CHECK();
    const unsigned g = conv_grid(c);
    // layer 4, then back through layers 3, 2, 1
    SPK_TRY(layer_grads(c, 3, c->A[2], c->dzA));
    k_conv<3><<<g, CONV_T, CONV_LDS, st>>>(c->dzA, c->WT[3], nullptr, c->dzB, nullptr, c->Z[2], c->n);
    SPK_TRY(layer_grads(c, 2, c->A[1], c->dzB));
    k_conv<3><<<g, CONV_T, CONV_LDS, st>>>(c->dzB, c->WT[2], nullptr, c->dzA, nullptr, c->Z[1], c->n);
    SPK_TRY(layer_grads(c, 1, c->A[0], c->dzA));
    k_conv<3><<<g, CONV_T, CONV_LDS, st>>>(c->dzA, c->WT[1], nullptr, c->dzB, nullptr, c->Z[0], c->n);
    SPK_TRY(layer_grads(c, 0, c->xin, c->dzB));
    SPK_LAUNCH_CHECK();
    if (loss) {
        std::vector<float> h(NBLK);
        SPK_HIP(hipMemcpyAsync(h.data(), c->lpart, NBLK * 4, hipMemcpyDeviceToHost, st));
        SPK_HIP(hipStreamSynchronize(st));
        double sum = 0.0;
        for (float v : h) sum += v;
        *loss = sum / (6.0 * (double)c->P);
    }
    return SPK_OK;
}

extern "C" int spk_closure_train_step(spk_closure c, const void *u, const void *tau_true, double lr, double *loss) {
    SPK_TRY(spk_closure_grads(c, u, tau_true, loss));
    const int NP = (int)param_total();
    c->adam_t += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - powf(b1, (float)c->adam_t), c2 = 1.0f - powf(b2, (float)c->adam_t);
    k_adam<<<(NP + 255) / 256, 256, 0, c->ctx->stream>>>(c->prm, c->grd, c->am, c->av, NP, (float)lr, b1, b2, 1e-8f,
                                                         c1, c2);
    SPK_LAUNCH_CHECK();
    return pack_weights(c);
}

// SGS term of a solver's state after its step: U += dt P(-i m k_j tau_ij(u))
extern "C" int spk_closure_apply(spk_closure c, spk_solver s) {
    SPK_REQUIRE(c && s, SPK_ERR_ARG, "spk_closure_apply: null argument");
    SolverViews v;
    solver_views(s, &v);
    SPK_REQUIRE(v.incompressible && v.nx == c->n && v.ny == c->n && v.nz == c->n, SPK_ERR_ARG,
                "spk_closure_apply: needs an incompressible run on the closure's %d^3 grid", c->n);
    SPK_REQUIRE(v.ctx->stream == c->ctx->stream, SPK_ERR_ARG,
                "spk_closure_apply: the closure and the solver must share a stream");
    const int n = c->n;
    const size_t fs = (size_t)n * n * (n + 2);
    if (!c->tau) {
        if (hipMalloc((void **)&c->tau, fs * 6 * sizeof(double)) != hipSuccess) {
            c->tau = nullptr;
            set_error("spk_closure_apply: hipMalloc of the stress buffer failed");
            return SPK_ERR_ALLOC;
        }
        SPK_TRY(spk_fft_plan_create(c->ctx, n, n, n, SPK_F64, 6, &c->plan6));
    }
    SPK_TRY(spk_complex2real(s));
    SPK_TRY(forward(c, v.realbuf + (size_t)v.VX * fs, c->tau));
    SPK_TRY(spk_fft_r2c(c->plan6, c->tau, c->tau));
    k_sgs_update<<<4096, 256, 0, c->ctx->stream>>>(v.U + (long long)v.VX * v.ntc,
                                                   reinterpret_cast<const cpx<double> *>(c->tau), v.ntc, v.kg, v.ts);
    SPK_LAUNCH_CHECK();
    return SPK_OK;
}

// Filtered velocity and subgrid stress on an n^3 grid from a fine N^3 state:
// with F the sharp cut to |k_i| <= kc, kc = (2/3)(n/2 - 1) (the dealiasing
// cut of the coarse grid, wavevector.cu:70-96), ubar = F u and
// tau_ij = F(u_i u_j) - F(ubar_i ubar_j), both products formed on the fine grid.
extern "C" int spk_sgs_stress(spk_ctx ctx, const void *U_hi, int N, void *ubar_lo, void *tau_lo, int n) {
    SPK_REQUIRE(ctx && U_hi && ubar_lo && tau_lo, SPK_ERR_ARG, "spk_sgs_stress: null argument");
    SPK_REQUIRE(n >= 4 && N >= n && N % n == 0, SPK_ERR_ARG, "spk_sgs_stress: N = %d, n = %d", N, n);
    hipStream_t st = ctx->stream;
    const long long ntc_hi = (long long)N * N * (N / 2 + 1), ntc_lo = (long long)n * n * (n / 2 + 1);
    const int kc = (int)(2.0 / 3.0 * (n / 2 - 1));
    const double scale = std::pow((double)n / N, 3);
    double *ur = nullptr, *br = nullptr, *pr = nullptr;
    spk_fft_plan hi3 = nullptr, hi1 = nullptr, lo3 = nullptr, lo1 = nullptr;
    int rc = SPK_OK;
    auto run = [&]() -> int {
        SPK_HIP(hipMalloc((void **)&ur, sizeof(double) * 2 * ntc_hi * 3));
        SPK_HIP(hipMalloc((void **)&br, sizeof(double) * 2 * ntc_hi * 3));
        SPK_HIP(hipMalloc((void **)&pr, sizeof(double) * 2 * ntc_hi));
        SPK_TRY(spk_fft_plan_create(ctx, N, N, N, SPK_F64, 3, &hi3));
        SPK_TRY(spk_fft_plan_create(ctx, N, N, N, SPK_F64, 1, &hi1));
        SPK_TRY(spk_fft_plan_create(ctx, n, n, n, SPK_F64, 3, &lo3));
        SPK_TRY(spk_fft_plan_create(ctx, n, n, n, SPK_F64, 1, &lo1));
        const cpx<double> *U = reinterpret_cast<const cpx<double> *>(U_hi);
        // fine real u, and fine real F u
        SPK_TRY(spk_fft_c2r(hi3, U, ur));
        k_mask_fine<<<4096, 256, 0, st>>>(U, reinterpret_cast<cpx<double> *>(br), N, ntc_hi, 3, kc);
        SPK_LAUNCH_CHECK();
        SPK_TRY(spk_fft_c2r(hi3, br, br));
        // coarse F u
        k_truncate<<<4096, 256, 0, st>>>(U, N, ntc_hi, reinterpret_cast<cpx<double> *>(ubar_lo), n, ntc_lo, 3, kc,
                                         scale);
        SPK_LAUNCH_CHECK();
        SPK_TRY(spk_fft_c2r(lo3, ubar_lo, ubar_lo));
        const int I[6] = {0, 0, 0, 1, 1, 2}, J[6] = {0, 1, 2, 1, 2, 2};
        for (int c = 0; c < 6; c++) {
            k_stress_prod<<<4096, 256, 0, st>>>(ur, br, pr, 2 * ntc_hi, I[c], J[c]);
            SPK_LAUNCH_CHECK();
            SPK_TRY(spk_fft_r2c(hi1, pr, pr));
            double *t = (double *)tau_lo + (size_t)c * 2 * ntc_lo;
            k_truncate<<<4096, 256, 0, st>>>(reinterpret_cast<const cpx<double> *>(pr), N, ntc_hi,
                                             reinterpret_cast<cpx<double> *>(t), n, ntc_lo, 1, kc, scale);
            SPK_LAUNCH_CHECK();
            SPK_TRY(spk_fft_c2r(lo1, t, t));
        }
        SPK_HIP(hipStreamSynchronize(st));
        return SPK_OK;
    };
    rc = run();
    (void)hipStreamSynchronize(st);
    for (spk_fft_plan pl : {hi3, hi1, lo3, lo1})
        if (pl) spk_fft_plan_destroy(pl);
    for (double *b : {ur, br, pr})
        if (b) (void)hipFree(b);
    return rc;
}
