// fp32 direct convolution on NCHW tensors: the reference's fp32 conv entry
// points (aexrt_d3d12_conv2d_float32 / _silu_float32, native/aexrt.h:175-189,
// shader RT:1554-1622) and its CPU path cpu_conv2d (RT:20552-20580).
//
// Each output is acc = bias[oc], then += x * w over (input channel of the
// group, ky, kx) in that order, skipping taps outside the input, with every
// multiply and add rounded on its own (no fused multiply-add): the exact
// arithmetic of the reference's CPU loop.  SiLU is acc / (1 + e^-acc).
//
// Bound by the vector ALU: two instructions per multiply-add (a contraction
// would round once), 12 us for 64 -> 64 channels at 80 x 80 on 1024 SIMDs.  So
// the inner loop is kept to little else:
// * a wave covers 64 consecutive output positions (images joined, no lane idle
//   on small maps) and J output channels of one group; four, because an input
//   load costs about 10 clocks of the CU's address path whoever asks for it
//   (two channels to a wave are bound by that: 116 us for four images);
// * the weights, the same for every lane, come by scalar loads as the second
//   operand of the multiply, the inputs from fixed 32-bit offsets per tap, both
//   one step ahead;
// * a tap outside the input reads as zero instead of being masked (masking by
//   lane took as long again as the arithmetic).  Adding x * w = +-0 changes a sum
//   only if w is not finite, which the sum then shows, or if the sum is -0, which
//   needs a bias of -0: in both cases the wave sums again, leaving those taps out.
// 64 -> 64 at 80 x 80: 25 us for one image, 72 us for four (166 and 373 us with a
// thread per position and 4 channels, every load at its use).
// Built with -ffp-contract=off (Makefile).
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace aexrt {

namespace {

constexpr int kF32Waves = 4;

// Weights are read through the constant address space: the same for every lane,
// so by scalar loads into SGPRs.
typedef const float __attribute__((address_space(4)))* wptr_t;
__device__ __forceinline__ wptr_t wptr(const float* w) { return (wptr_t)(uintptr_t)w; }

// T taps of one or more input channels: this lane's inputs, and the weights of
// the wave's output channels.
template <int K, int U, int J>
struct Step {
    static constexpr int KK = K * K, T = U * KK;
    float x[T];
    float w[J][T];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rx, const uint32_t (&off)[KK], uint32_t at,
                                         uint32_t plane, wptr_t wp, const int (&wo)[J]) {
#pragma unroll
        for (int t = 0; t < T; ++t)
            x[t] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, off[t % KK], at + (t / KK) * plane, 0));
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int t = 0; t < T; ++t) w[j][t] = wp[wo[j] + t];
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void add(float (&acc)[J]) const {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int j = 0; j < J; ++j) acc[j] = __fadd_rn(acc[j], __fmul_rn(x[t], w[j][t]));
    }
};

// Where a wave's outputs are.
struct WavePlace {
    bool on;      // this lane's position exists
    int n, r;     // its image and position
    int iy0, ix0; // its first tap
    int gid, oc0, oc_end;
};

template <int J>
__device__ __forceinline__ WavePlace wave_place(const F32ConvParams& p, int tile, int tiles_group, int64_t pos) {
    WavePlace o;
    const int64_t ohw = (int64_t)p.OH * p.OW, all = p.N * ohw;
    o.on = pos < all;
    const int64_t m = o.on ? pos : all - 1;
    o.n = (int)(m / ohw);
    o.r = (int)(m - o.n * ohw);
    const int oh = o.r / p.OW, ow = o.r - oh * p.OW;
    o.iy0 = oh * p.SH - p.PT;
    o.ix0 = ow * p.SW - p.PL;
    const int ocpg = p.OC / p.G;
    o.gid = tile / tiles_group;
    o.oc0 = o.gid * ocpg + (tile - o.gid * tiles_group) * J;
    o.oc_end = (o.gid + 1) * ocpg;
    return o;
}

template <int J>
__device__ __forceinline__ void wave_store(const F32ConvParams& p, const WavePlace& o, const float (&acc)[J]) {
    if (!o.on) return;
    const int64_t ohw = (int64_t)p.OH * p.OW;
    float* y = p.y + ((int64_t)o.n * p.OC + o.oc0) * ohw + o.r;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        if (o.oc0 + j >= o.oc_end) break;
        float v = acc[j];
        if (p.silu) v = __fdiv_rn(v, __fadd_rn(1.0f, expf(-v)));
        y[j * ohw] = v;
    }
}

// One tap at a time, taps outside the input left out: any kernel and size.
template <int J>
__device__ __forceinline__ void sum_taps(const F32ConvParams& p, const WavePlace& o, float (&acc)[J]) {
    const int icpg = p.C / p.G, wlen = icpg * p.KH * p.KW;
    const wptr_t w = wptr(p.w + (int64_t)o.oc0 * wlen);
    int wo[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int oc = min(o.oc0 + j, o.oc_end - 1);
        acc[j] = p.bias[oc];
        wo[j] = (oc - o.oc0) * wlen;
    }
    const int64_t plane = (int64_t)p.H * p.W;
    const float* xn = p.x + ((int64_t)o.n * p.C + (int64_t)o.gid * icpg) * plane;
    int k = 0;
    for (int ic = 0; ic < icpg; ++ic, xn += plane)
        for (int ky = 0; ky < p.KH; ++ky) {
            const int64_t iy = o.iy0 + (int64_t)ky * p.DH;
            for (int kx = 0; kx < p.KW; ++kx, ++k) {
                const int64_t ix = o.ix0 + (int64_t)kx * p.DW;
                if (iy >= 0 && iy < p.H && ix >= 0 && ix < p.W) {
                    const float xv = xn[iy * p.W + ix];
#pragma unroll
                    for (int j = 0; j < J; ++j) acc[j] = __fadd_rn(acc[j], __fmul_rn(xv, w[wo[j] + k]));
                }
            }
        }
}

template <int J>
__global__ __launch_bounds__(64) void conv_f32_any_kernel(F32ConvParams p, int tiles_group, int tiles) {
    if ((int)(blockIdx.y + blockIdx.z * gridDim.y) >= tiles) return;
    const WavePlace o = wave_place<J>(p, blockIdx.y + blockIdx.z * gridDim.y, tiles_group, (int64_t)blockIdx.x * 64 + threadIdx.x);
    float acc[J];
    sum_taps(p, o, acc);
    wave_store(p, o, acc);
}

// Square kernels of K = 1 or 3 taps a side, any stride, padding and dilation,
// input below 4 GB.  wave_tiles (a power of two) of a block's waves take
// neighbouring channel tiles at the same positions, the others further ones.
template <int K, int J>
__global__ __launch_bounds__(64 * kF32Waves) void conv_f32_kernel(F32ConvParams p, int tiles_group, int tiles,
                                                                  int wave_tiles) {
    constexpr int KK = K * K;
    constexpr int U = K == 1 ? 8 : 1;  // input channels of a step
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int tile = (blockIdx.y + blockIdx.z * gridDim.y) * wave_tiles + wave % wave_tiles;
    if (tile >= tiles) return;
    const WavePlace o = wave_place<J>(
        p, tile, tiles_group, ((int64_t)blockIdx.x * (kF32Waves / wave_tiles) + wave / wave_tiles) * 64 + lane);
    const int icpg = p.C / p.G;
    const uint32_t plane = (uint32_t)p.H * (uint32_t)p.W;
    const uint32_t bytes = (uint32_t)p.N * (uint32_t)p.C * plane * 4u;
    const int wlen = icpg * KK;
    float acc[J];
    int wo[J];  // a channel past the group's last repeats it and is not stored
    bool redo = false;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int oc = min(o.oc0 + j, o.oc_end - 1);
        acc[j] = p.bias[oc];
        redo = redo || __float_as_uint(acc[j]) == 0x80000000u;
        wo[j] = (oc - o.oc0) * wlen;
    }
    wptr_t w = wptr(p.w + (int64_t)o.oc0 * wlen);
    uint32_t off[KK];
#pragma unroll
    for (int t = 0; t < KK; ++t) {
        const int iy = o.iy0 + (t / K) * p.DH, ix = o.ix0 + (t % K) * p.DW;
        const bool in = iy >= 0 && iy < p.H && ix >= 0 && ix < p.W;
        off[t] = in ? ((uint32_t)o.n * (uint32_t)p.C * plane + (uint32_t)(iy * p.W + ix)) * 4u : 0xFFFFFFFCu;
    }
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.x), 0, bytes, 0x00020000);
    const uint32_t step = plane * 4u;
    uint32_t at = (uint32_t)(o.gid * icpg) * step;
    // two steps in turn: one is loaded while the other is added
    int left = icpg / U;
    if (left > 0) {
        Step<K, U, J> a, b;
        a.load(rx, off, at, step, w, wo);
        for (; left >= 2; left -= 2) {
            at += U * step;
            w += U * KK;
            b.load(rx, off, at, step, w, wo);
            a.add(acc);
            if (left > 2) {
                at += U * step;
                w += U * KK;
            }
            a.load(rx, off, at, step, w, wo);
            b.add(acc);
        }
        if (left) a.add(acc);
        at += U * step;
        w += U * KK;
    }
    if constexpr (U > 1)
        for (int r = icpg % U; r > 0; --r, at += step, w += KK) {
            Step<K, 1, J> one;
            one.load(rx, off, at, step, w, wo);
            one.add(acc);
        }
#pragma unroll
    for (int j = 0; j < J; ++j) redo = redo || !(fabsf(acc[j]) <= 3.402823466e38f);
    if (__any(redo)) sum_taps(p, o, acc);
    wave_store(p, o, acc);
}

template <int J>
hipError_t launch_j(const F32ConvParams& p, hipStream_t stream) {
    const int tiles_group = (p.OC / p.G + J - 1) / J;
    const int64_t ohw = (int64_t)p.OH * p.OW;
    const int64_t image = (int64_t)p.C * p.H * p.W * 4;
    const int64_t tiles = (int64_t)tiles_group * p.G;
    const int wave_tiles = tiles >= 4 ? 4 : tiles >= 2 ? 2 : 1;
    // fewer than 2^32 threads to a launch's row
    const int64_t max_blocks = (((int64_t)1 << 32) - 1) / (64 * kF32Waves);
    const bool square = p.KH == p.KW && (p.KH == 1 || p.KH == 3) && image < ((int64_t)1 << 32) - 8 &&
                        ohw <= max_blocks * 64;
    const int64_t positions = square ? 64 * (kF32Waves / wave_tiles) : 64;  // of a block
    const int64_t rows = square ? (tiles + wave_tiles - 1) / wave_tiles : tiles;
    const int64_t ny = std::min<int64_t>(rows, 65535), nz = (rows + ny - 1) / ny;
    // images per launch: the grid, and 32-bit input offsets
    int64_t per = (square ? max_blocks : max_blocks * kF32Waves) * positions / ohw;
    if (square) per = std::min(per, (((int64_t)1 << 32) - 8) / image);
    if (per < 1 || nz > 65535) return hipErrorInvalidValue;
    for (int64_t n0 = 0; n0 < p.N; n0 += per) {
        F32ConvParams q = p;
        q.N = (int)std::min<int64_t>(per, p.N - n0);
        q.x += n0 * p.C * p.H * p.W;
        q.y += n0 * p.OC * ohw;
        const dim3 grid((unsigned)((q.N * ohw + positions - 1) / positions), (unsigned)ny, (unsigned)nz);
        if (!square)
            hipLaunchKernelGGL(conv_f32_any_kernel<J>, grid, dim3(64), 0, stream, q, tiles_group, (int)tiles);
        else if (p.KH == 1)
            hipLaunchKernelGGL((conv_f32_kernel<1, J>), grid, dim3(64 * kF32Waves), 0, stream, q, tiles_group, (int)tiles,
                               wave_tiles);
        else
            hipLaunchKernelGGL((conv_f32_kernel<3, J>), grid, dim3(64 * kF32Waves), 0, stream, q, tiles_group, (int)tiles,
                               wave_tiles);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

hipError_t launch_conv_f32(const F32ConvParams& p, hipStream_t stream) {
    if (p.N <= 0 || p.C <= 0 || p.OC <= 0 || p.OH <= 0 || p.OW <= 0 || p.H <= 0 || p.W <= 0 || p.KH <= 0 ||
        p.KW <= 0 || p.SH <= 0 || p.SW <= 0 || p.DH <= 0 || p.DW <= 0 || p.G <= 0 || p.C % p.G || p.OC % p.G)
        return hipErrorInvalidValue;
    // a group of one or two output channels fills no more
    const int ocpg = p.OC / p.G;
    return ocpg >= 3 ? launch_j<4>(p, stream) : ocpg == 2 ? launch_j<2>(p, stream) : launch_j<1>(p, stream);
}

}  // namespace aexrt
