// Dynamic int8 convolution: the reference's fallback int8 conv
// (native/aexrt_d3d12_runtime.cpp:2952-3115), which quantizes in the kernel
// instead of reading a prequantized tensor.  The reference dispatches it for
// int8 convs whose input tensor has fewer than 4096 elements
// (RT:21478-21479, RT:24260-24317).
//
// Per output position and 4-channel input group g:
//   1x1: amax = max|x| over the 4 channels at the position;
//   3x3: amax = max|x| over the 4 channels at the 9 taps (zero padding
//        included), one scale for the 36 values;
//   s = 127/amax (0 when amax is 0), q = round_half_even(x*s) as a byte,
//   part = sum over the taps of dot4(q, w) in int32,
//   acc += float(part) * (amax/127), in group order, fp32;
// y = acc * w_scale[oc] + bias[oc], SiLU, (+ residual), fp16 or fp32 out.
//
// These convs see at most 4095 input elements, so what counts is the chain of
// memory round trips, not the work.  A block quantizes the patches of PB
// positions once into LDS (scales and packed words); each of its four waves
// then computes 16 output channels: lane (s, o) takes channels 16 s..16 s + 15
// of a 64-channel step for output channel o, 16 bytes of weights a tap, the
// weights of the next step already in flight.  A lane's four group sums stay
// exact integers; a 4x4 exchange of the wave's 16-lane rows hands lane row s
// the sums of position s, which adds them up in group order.  Every multiply
// and add of that fp32 chain is rounded on its own (no contraction), so the
// result equals a scalar restatement of the formula bit for bit.
// 3x3 128 -> 128 at 5x5: 6.1 us (44 us with a block per position whose threads
// each read their channel's weights 4 bytes at a time, a cache line a lane).
// Built with -ffp-contract=off (Makefile).
#include "common.h"
#include "kernels.h"

namespace aexrt {

namespace {

constexpr int kDynWaves = 4;

// Rows (16 lanes) of four registers transposed: register i of row r <- register r
// of row i.
__device__ __forceinline__ void transpose_rows(uint32_t (&v)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    v[0] = c[0];
    v[1] = c[1];
    v[2] = d[0];
    v[3] = d[1];
}

// K: taps a side; PB: positions of a block, 4 or 1.
template <int K, int PB>
__global__ __launch_bounds__(64 * kDynWaves) void conv_int8_dynamic_kernel(DynConvParams p, int positions) {
    constexpr int KK = K * K;
    constexpr int U = K == 1 ? 8 : 1;  // 64-channel steps whose weights are loaded together
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    const int G = p.C / 4;
    const int Gs = (G + 15) & ~15;                         // rows of whole 64-channel steps
    uint32_t* l_q = lds;                                   // [PB][KK][Gs]
    float* l_inv = reinterpret_cast<float*>(lds + PB * KK * Gs);  // [PB][Gs]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int o = lane & 15, s = lane >> 4;
    const int pos0 = blockIdx.x * PB;
    const int ohw = p.OH * p.OW;
    constexpr int pad = K == 3 ? 1 : 0;
    const int tile = blockIdx.y * kDynWaves + wave;
    const bool computes = tile * 16 < p.OC;
    const int steps = Gs / 16;
    // this lane's weights of steps t0 .. t0 + U - 1 (lanes past the last channel: the first ones,
    // unused)
    const int8_t* wrow = p.w + (int64_t)(computes ? tile * 16 + o : o) * p.Kp;
    auto load_w = [&](int t0, v4i (&w)[U * KK]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = (t0 + u) * 64 + s * 16;
            const int8_t* wc = wrow + (c < p.C ? c : 0);
#pragma unroll
            for (int t = 0; t < KK; ++t) w[u * KK + t] = *reinterpret_cast<const v4i*>(wc + t * p.C);
        }
    };
    v4i wa[U * KK], wb[U * KK];
    load_w(0, wa);
    // ---- quantize the patches ----
    for (int e = tid; e < PB * Gs; e += 64 * kDynWaves) {
        const int pi = PB == 1 ? 0 : e / Gs, g = e - pi * Gs;
        const int pos = pos0 + pi;
        float v[KK][4];
        float am = 0.0f;
        const bool on = g < G && pos < positions;
        const int n = on ? pos / ohw : 0;
        const int r = on ? pos - n * ohw : 0;
        const int oh = r / p.OW, ow = r - oh * p.OW;
        const __half* xn = p.x + (int64_t)n * p.x_nstride + (on ? g * 4 : 0);
#pragma unroll
        for (int t = 0; t < KK; ++t) {
            const int iy = oh * p.S + t / K - pad, ix = ow * p.S + t % K - pad;
            const bool in = on && iy >= 0 && iy < p.H && ix >= 0 && ix < p.W;
            uint2 h = make_uint2(0u, 0u);
            if (in) h = *reinterpret_cast<const uint2*>(xn + (int64_t)(iy * p.W + ix) * p.x_cstride);
            const float2 lo = __half22float2(*reinterpret_cast<const __half2*>(&h.x));
            const float2 hi = __half22float2(*reinterpret_cast<const __half2*>(&h.y));
            v[t][0] = lo.x;
            v[t][1] = lo.y;
            v[t][2] = hi.x;
            v[t][3] = hi.y;
#pragma unroll
            for (int c = 0; c < 4; ++c) am = fmaxf(am, fabsf(v[t][c]));
        }
        const float sc = am > 0.0f ? __fdiv_rn(127.0f, am) : 0.0f;
        l_inv[e] = __fdiv_rn(am, 127.0f);
#pragma unroll
        for (int t = 0; t < KK; ++t)
            l_q[(pi * KK + t) * Gs + g] = pack4_q(v[t][0], v[t][1], v[t][2], v[t][3], sc);
    }
    __syncthreads();
    if (!computes) return;
    // ---- 16 output channels, the group sums in group order ----
    const int mine = PB == 1 ? 0 : s;  // the position this lane adds up
    float acc = 0.0f;
    auto add_step = [&](int t, const v4i* w) {
        uint32_t part[4][4];  // [group of this lane][position]
#pragma unroll
        for (int pi = 0; pi < 4; ++pi) {
            int d[4] = {0, 0, 0, 0};
            if (pi < PB) {
#pragma unroll
                for (int k = 0; k < KK; ++k) {
                    const v4i q = *reinterpret_cast<const v4i*>(l_q + (pi * KK + k) * Gs + t * 16 + s * 4);
#pragma unroll
                    for (int r = 0; r < 4; ++r) d[r] = __builtin_amdgcn_sdot4(q[r], w[k][r], d[r], false);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) part[r][pi] = (uint32_t)d[r];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) transpose_rows(part[r]);
        const float* inv = l_inv + mine * Gs + t * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (t * 16 + i * 4 >= G) break;
            const float4 f = *reinterpret_cast<const float4*>(inv + 4 * i);
            acc = __fadd_rn(acc, __fmul_rn((float)(int)part[0][i], f.x));
            acc = __fadd_rn(acc, __fmul_rn((float)(int)part[1][i], f.y));
            acc = __fadd_rn(acc, __fmul_rn((float)(int)part[2][i], f.z));
            acc = __fadd_rn(acc, __fmul_rn((float)(int)part[3][i], f.w));
        }
    };
    auto add_steps = [&](int t0, const v4i (&w)[U * KK]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (t0 + u < steps) add_step(t0 + u, w + u * KK);
    };
    for (int t = 0; t < steps; t += 2 * U) {
        if (t + U < steps) load_w(t + U, wb);
        add_steps(t, wa);
        if (t + 2 * U < steps) load_w(t + 2 * U, wa);
        if (t + U < steps) add_steps(t + U, wb);
    }
    // ---- scale, bias, SiLU, residual, amax ----
    const int oc = tile * 16 + o, pos = pos0 + s;
    float m = 0.0f;
    if (s < PB && pos < positions && oc < p.OC) {
        const int n = pos / ohw, r = pos - n * ohw;
        const bool do_res = (p.flags & kConvResidual) != 0;
        float v = __fadd_rn(__fmul_rn(acc, p.w_scale[oc]), p.bias[oc]);
        if (p.flags & kConvSilu) v = silu(v);
        const int64_t yo = (int64_t)n * p.y_nstride + (int64_t)r * p.y_cstride + oc;
        const float res = do_res ? __half2float(p.res[(int64_t)n * p.r_nstride + (int64_t)r * p.r_cstride + oc]) : 0.0f;
        if (p.flags & kConvOutF32) {
            if (do_res) v += res;
            static_cast<float*>(p.y)[yo] = v;
        } else {
            // fp16 conv output + fp16 residual, added in fp32 and rounded again
            if (do_res) v = __half2float(__float2half(v)) + res;
            const __half h = __float2half(v);
            static_cast<__half*>(p.y)[yo] = h;
            v = __half2float(h);
        }
        m = fabsf(v);
    }
    if (!p.y_slots.p) return;
    m = wave_max(m);
    if (lane == 0 && m > 0.0f) slot_max(slot_copy(p.y_slots, blockIdx.x) + tile, m);
}

template <int K>
hipError_t launch_k(const DynConvParams& p, int positions, hipStream_t stream) {
    const int Gs = (p.C / 4 + 15) & ~15;
    const unsigned rows = (unsigned)((p.OC + 16 * kDynWaves - 1) / (16 * kDynWaves));
    const size_t lds = (size_t)Gs * (K * K + 1) * 4;  // of a position
    // four positions to a block share its weights once that still gives every CU a block
    if (((int64_t)positions + 3) / 4 * rows >= 256 && 4 * lds <= 64 * 1024)
        hipLaunchKernelGGL((conv_int8_dynamic_kernel<K, 4>), dim3((unsigned)(positions + 3) / 4, rows),
                           dim3(64 * kDynWaves), 4 * lds, stream, p, positions);
    else
        hipLaunchKernelGGL((conv_int8_dynamic_kernel<K, 1>), dim3((unsigned)positions, rows), dim3(64 * kDynWaves), lds,
                           stream, p, positions);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_conv_int8_dynamic(const DynConvParams& p, hipStream_t stream) {
    if (p.K != 1 && p.K != 3) return hipErrorInvalidValue;
    if (p.C % 16 || p.C <= 0 || p.OC <= 0 || p.N <= 0 || p.OH <= 0 || p.OW <= 0) return hipErrorInvalidValue;
    if (p.K == 1 && (p.S != 1 || p.OH != p.H || p.OW != p.W)) return hipErrorInvalidValue;
    if (p.K == 3 && (p.S < 1 || p.S > 2 || (p.OH - 1) * p.S + 1 > p.H + 1 || (p.OW - 1) * p.S + 1 > p.W + 1))
        return hipErrorInvalidValue;
    if (p.Kp < p.K * p.K * p.C) return hipErrorInvalidValue;
    const int64_t positions = (int64_t)p.N * p.OH * p.OW;
    if (positions > (1 << 30)) return hipErrorInvalidValue;
    if (((size_t)(p.C / 4) * (1 + p.K * p.K) + (p.OC + 15) / 16) * 4 > 64 * 1024) return hipErrorInvalidValue;
    return p.K == 1 ? launch_k<1>(p, (int)positions, stream) : launch_k<3>(p, (int)positions, stream);
}

}  // namespace aexrt
