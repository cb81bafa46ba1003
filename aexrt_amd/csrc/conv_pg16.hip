// pg16 int8 convolution (per-16-input-channel activation scales) and the
// fused amax + pack of its input.
//
// The reference's pg16 conv (native/aexrt_d3d12_runtime.cpp:4770-4923) sums
// the int8 products of one 16-channel group exactly in int32, scales each
// group sum by amax[1 + g] / 127 into an fp32 accumulator, and finishes with
// the oc weight scale, the bias and SiLU.  One v_mfma_i32_16x16x64_i8 takes 64
// k, four times the 16 channels of a group, so its k holds one group at a time:
// for a 3x3 conv the group's 16 channels of four taps (lane group grp loads tap
// 4 i + grp of step i; three steps cover the nine taps, the last three k
// quarters have zero weights), for a 1x1 conv the channels of four groups with
// the weights of all but one zeroed (four products from one load of each
// operand).  Rows are 16 output channels, columns 16 positions, so a lane ends
// with channels oc0 + 4 grp + r of position col: the fragment layout of the
// per-tensor kernels, whose epilogue and 8-byte NHWC stores are reused.
//
// The int32 group sums run over all taps of the kernel before the fp32
// scaling (exact integers; the reference scales per tap for 3x3 and per 8
// channels for 1x1, which differs only in fp32 rounding).
//
// Bound by the address lookups of its loads (16 bytes of 64 places each): with
// one operand load for all lanes instead of one per lane group, 3 products per
// group instead of 9 and JN subtiles on one input, 96 -> 48 at 27x35 x5 9.1 ->
// 7.1 us, 512 -> 256 1x1 at 20x20 6.9 -> 5.8.  Two units in flight instead of one
// were slower (8.7 us; the registers cost more than the latency).
#include "conv_igemm.h"

namespace aexrt {

namespace {

using igemm::bload16;
using igemm::kOob;
using igemm::make_rsrc;
using igemm::quant8;
using igemm::rsrc_t;
using igemm::v2i;

constexpr int kPgWaves = 4;
constexpr int kPgMaxGroups = 256;  // in_channels <= 4096

// LOADER kLoaderNhwc: fp16 NHWC view quantized here with 127/amax_g (the
// reference's pack with per-group scales, RT:3330-3344); kLoaderPackedNc4: the
// reference's packed NC/4HW4 int8 ((n * C/4 + icg) * H*W + pixel words).
// A wave takes 16 positions and JN 16-channel subtiles.
template <int KK, int LOADER, int JN>
__global__ __launch_bounds__(kPgWaves * 64) void conv_int8_pg16_kernel(ConvParams p) {
    constexpr int NB = KK == 9 ? 3 : 1;  // k steps of one unit: a group (3x3), four groups (1x1)
    constexpr int R = JN * 16;
    constexpr bool kPacked = LOADER == kLoaderPackedNc4;
    __shared__ uint32_t l_max[kPgMaxGroups];
    __shared__ float l_gs[kPgMaxGroups];  // amax_g / 127
    __shared__ float l_qs[kPgMaxGroups];  // 127 / amax_g, 0 when amax_g is not > 0
    __shared__ float l_bias[R], l_scale[R];
    __shared__ uint32_t l_slots[JN];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, grp = lane >> 4;
    const int G = p.C >> 4;
    const int U = KK == 9 ? G : (p.C + 63) >> 6;
    const int oc0 = blockIdx.y * R;

    const int m = (blockIdx.x * kPgWaves + wave) * 16 + col;
    const bool mok = m < p.M;
    const int mm = mok ? m : 0;
    const int n = (int)fdiv((uint32_t)mm, p.fd_ohw);
    const int pos = mm - n * p.OH * p.OW;
    const int oh = (int)fdiv((uint32_t)pos, p.fd_ow);
    const int ow = pos - oh * p.OW;
    const uint32_t plane = (uint32_t)(p.H * p.W);
    const rsrc_t rx = make_rsrc(p.x, p.x_bytes);
    const rsrc_t rw = make_rsrc(p.w, (uint32_t)p.OCp * (uint32_t)p.Kp);
    // byte offsets of this lane's pixel (channel 0) and weights (row col of the
    // first subtile) of each k step; kOob and any channel offset on top of it
    // stay past both buffers
    uint32_t xo[NB], wo[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int tap = KK == 9 ? 4 * i + grp : 0;
        const int ky = tap / 3;
        const int iy = oh * p.S - p.P + ky, ix = ow * p.S - p.P + (tap - 3 * ky);
        const bool ok = mok && tap < KK && iy >= 0 && iy < p.H && ix >= 0 && ix < p.W;
        const uint32_t pix = (uint32_t)(iy * p.W + ix);
        if constexpr (kPacked) xo[i] = ok ? ((uint32_t)n * (uint32_t)(p.C >> 2) * plane + pix) * 4u : kOob;
        else xo[i] = ok ? ((uint32_t)((int64_t)n * p.x_nstride) + pix * (uint32_t)p.x_cstride) * 2u : kOob;
        wo[i] = tap < KK ? (uint32_t)(oc0 + col) * (uint32_t)p.Kp + (uint32_t)(tap * p.C) : kOob;
    }
    struct Unit {
        v4i x[NB][kPacked ? 1 : 2], w[NB][JN];
    };
    // operands of unit u (past the last one: unused, inside the buffers' bounds checks)
    auto load = [&](int u, Unit& q) {
        const int c0 = KK == 9 ? 16 * u : 64 * u + 16 * grp;
        const bool cok = KK == 9 || c0 < p.C;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            if constexpr (kPacked) {
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    q.x[i][0][w] = __builtin_amdgcn_raw_buffer_load_b32(
                        rx, cok ? xo[i] + (uint32_t)((c0 >> 2) + w) * plane * 4u : kOob, 0, 0);
            } else {
                q.x[i][0] = bload16(rx, cok ? xo[i] + (uint32_t)c0 * 2u : kOob);
                q.x[i][1] = bload16(rx, cok ? xo[i] + (uint32_t)c0 * 2u + 16u : kOob);
            }
#pragma unroll
            for (int j = 0; j < JN; ++j)
                q.w[i][j] = bload16(rw, cok ? wo[i] + (uint32_t)(j * 16 * p.Kp + c0) : kOob);
        }
    };
    Unit cur;
    load(0, cur);

    // group maxima: over the copies of the slot array (one thread per group and
    // run of copies, then one LDS atomic each)
    for (int g = tid; g < kPgMaxGroups; g += kPgWaves * 64) l_max[g] = 0u;
    if (tid < R) {
        const int oc = oc0 + tid;
        l_bias[tid] = oc < p.OC ? p.bias[oc] : 0.0f;
        l_scale[tid] = oc < p.OC ? p.w_scale[oc] : 0.0f;
    }
    if (tid < JN) l_slots[tid] = 0u;
    __syncthreads();
    {
        const int row = (int)fdiv((uint32_t)tid, p.fd_ns), g = tid - row * G, rows = kPgWaves * 64 / G;
        if (row < rows) {
            uint32_t v = 0u;
            for (uint32_t s = row; s < p.x_slots.stripes; s += rows) v = max(v, p.x_slots.p[s * p.x_slots.stride + g]);
            if (v) atomicMax(&l_max[g], v);
        }
    }
    __syncthreads();
    for (int g = tid; g < ((G + 3) & ~3); g += kPgWaves * 64) {
        const float a = u2f(l_max[g]);
        l_gs[g] = g < G ? a / 127.0f : 0.0f;
        l_qs[g] = a > 0.0f ? 127.0f / a : 0.0f;
    }
    __syncthreads();

    typedef float v4f_t __attribute__((ext_vector_type(4)));
    v4f_t accf[JN][1];  // channels oc0 + 16 j + 4 grp + r
#pragma unroll
    for (int j = 0; j < JN; ++j) accf[j][0] = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto quant = [&](const v4i (&x)[kPacked ? 1 : 2], float s) {
        if constexpr (kPacked) return x[0];
        const v2i q0 = quant8(x[0], s), q1 = quant8(x[kPacked ? 0 : 1], s);
        return v4i{q0[0], q0[1], q1[0], q1[1]};
    };
    auto add = [&](int j, const v4i& acc, float s) {
#pragma unroll
        for (int r = 0; r < 4; ++r) accf[j][0][r] = __builtin_fmaf((float)acc[r], s, accf[j][0][r]);
    };
    auto multiply = [&](int u, const Unit& q) {
        if constexpr (KK == 9) {
            const float s = l_qs[u], gs = l_gs[u];
            v4i acc[JN];
#pragma unroll
            for (int j = 0; j < JN; ++j) acc[j] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const v4i b = quant(q.x[i], s);
#pragma unroll
                for (int j = 0; j < JN; ++j) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(q.w[i][j], b, acc[j], 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < JN; ++j) add(j, acc[j], gs);
        } else {
            const v4i b = quant(q.x[0], l_qs[4 * u + grp]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float gs = l_gs[4 * u + r];
#pragma unroll
                for (int j = 0; j < JN; ++j) {
                    const v4i w = grp == r ? q.w[0][j] : v4i{0, 0, 0, 0};
                    add(j, __builtin_amdgcn_mfma_i32_16x16x64_i8(w, b, v4i{0, 0, 0, 0}, 0, 0, 0), gs);
                }
            }
        }
    };
    for (int u = 0; u < U; ++u) {
        Unit next;
        load(u + 1, next);
        multiply(u, cur);
        cur = next;
    }

    const bool do_silu = (p.flags & kConvSilu) != 0;
    const bool out_f32 = (p.flags & kConvOutF32) != 0;
    if (p.flags & kConvOutNchw) {
        // dense NCHW output of the reference (typed fp32 or fp16 storage)
        const rsrc_t ry = make_rsrc(p.y, p.y_bytes);
        const int ohw = p.OH * p.OW;
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int lc = 16 * j + 4 * grp + r, oc = oc0 + lc;
                float v = __builtin_fmaf(accf[j][0][r], l_scale[lc], l_bias[lc]);
                if (do_silu) v = silu(v);
                const bool ok = mok && oc < p.OC;
                const uint32_t e = (uint32_t)((n * p.OC + oc) * ohw + pos);
                if (out_f32)
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v), ry, ok ? e * 4u : kOob, 0, 0);
                else
                    __builtin_amdgcn_raw_buffer_store_b16(__half_as_short(__float2half(v)), ry, ok ? e * 2u : kOob, 0,
                                                          0);
            }
        return;
    }
    // NHWC view output: the per-tensor kernels' epilogue (scale, bias, SiLU,
    // residual, amax slots of the output)
    const rsrc_t ry = make_rsrc(p.y, p.y_bytes);
    const rsrc_t rr = make_rsrc(p.res, p.r_bytes);
    const rsrc_t racc = make_rsrc(nullptr, 0u);
    const int jmax = min(JN, (p.OCp - oc0) >> 4);
    int yo[1], ro[1], mo[1];
    yo[0] = mok ? (int)((int64_t)n * p.y_nstride + (int64_t)pos * p.y_cstride) : -1;
    ro[0] = (int)((int64_t)n * p.r_nstride + (int64_t)pos * p.r_cstride);
    mo[0] = m;
    constexpr uint32_t kAll = (1u << JN) - 1u;
    v2i rv[JN][1];
    igemm::tile_residual<JN, 1, igemm::kEpiAny>(p, rr, yo, ro, oc0, jmax, grp, kAll, rv);
    float gmax[JN];
#pragma unroll
    for (int j = 0; j < JN; ++j) gmax[j] = 0.0f;
    igemm::tile_store<true, JN, 1, igemm::kEpiAny>(p, accf, yo, mo, rv, oc0, jmax, grp, kAll, l_bias, l_scale, gmax,
                                                   ry, racc);
    igemm::flush_slots<JN>(p, gmax, oc0, jmax, kAll, out_f32, l_slots);
}

// a3: the reference's fused amax + pack (RT:4083-4149).  One block per
// (image n, 16-channel group g): the group max is taken over channels
// 16g..16g+15 of image 0's memory for every n (the reference's strip start
// carries no image offset), written to amax[1 + g] (every n writes the same
// value), and image n's four 4-channel planes of the group are packed with
// s = 127/max.  amax[0] is not written.
constexpr int kFusedThreads = 512;

template <typename T>
__device__ __forceinline__ float ld_f(const T* x, int64_t i) {
    if constexpr (sizeof(T) == 2) return __half2float(x[i]);
    else return x[i];
}

template <typename T>
__global__ __launch_bounds__(kFusedThreads) void quant_fused_pg16_kernel(const T* x, int C, int HW,
                                                                         uint32_t* packed, uint32_t* amax) {
    __shared__ float lm[kFusedThreads / 64];
    const int G = C >> 4;
    const int n = blockIdx.x / G, g = blockIdx.x - n * G;
    const int64_t b = (int64_t)g * 16 * HW;
    const int64_t span = (int64_t)16 * HW;
    float m = 0.0f;
    for (int64_t i = threadIdx.x; i < span; i += kFusedThreads) m = fmaxf(m, fabsf(ld_f(x, b + i)));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) lm[threadIdx.x >> 6] = m;
    __syncthreads();
    m = lm[0];
#pragma unroll
    for (int w = 1; w < kFusedThreads / 64; ++w) m = fmaxf(m, lm[w]);
    if (threadIdx.x == 0) amax[g + 1] = f2u(m);
    const int icg_count = C >> 2;
    const float s = 127.0f / m;
    const int64_t out0 = ((int64_t)n * icg_count + 4 * g) * HW;
    const int64_t in0 = out0 * 4;
    for (int e = threadIdx.x; e < 4 * HW; e += kFusedThreads) {
        const int il = e / HW, pp = e - il * HW;
        uint32_t v = 0u;
        if (m > 0.0f) {
            const int64_t base = in0 + (int64_t)il * 4 * HW + pp;
            v = pack4_q(ld_f(x, base), ld_f(x, base + HW), ld_f(x, base + 2 * HW), ld_f(x, base + 3 * HW), s);
        }
        packed[out0 + e] = v;
    }
}

template <int KK, int LOADER, int JN>
void launch_pg_tile(const ConvParams& p, hipStream_t stream) {
    const dim3 grid((p.M + kPgWaves * 16 - 1) / (kPgWaves * 16), (p.OCp / 16 + JN - 1) / JN);
    hipLaunchKernelGGL((conv_int8_pg16_kernel<KK, LOADER, JN>), grid, dim3(kPgWaves * 64), 0, stream, p);
}

// Blocks of 64 positions by 16 channels.
int64_t pg_blocks(const ConvParams& p) {
    return (int64_t)((p.M + kPgWaves * 16 - 1) / (kPgWaves * 16)) * (p.OCp / 16);
}

// More channel subtiles a wave read (and quantize) the input fewer times, once
// the smaller grid still gives every CU more than one block: 1x1 128 -> 128 at
// 40x40 x8 9.3 us with 1, 8.4 with 2, 7.7 with 4; 1x1 512 -> 256 at 20x20 (112
// blocks) 5.8, 8.2, 10.3.  Four only where they leave no empty subtile (64 -> 80
// at 40x40 x32: 12.4, 11.4, 12.1).
template <int KK, int LOADER>
void launch_pg(const ConvParams& p, hipStream_t stream) {
    const int64_t blocks = pg_blocks(p);
    const int ocj = p.OCp / 16;
    if (ocj % 4 == 0 && blocks / 4 >= 384) launch_pg_tile<KK, LOADER, 4>(p, stream);
    else if (ocj > 1 && blocks / 2 >= 384) launch_pg_tile<KK, LOADER, 2>(p, stream);
    else launch_pg_tile<KK, LOADER, 1>(p, stream);
}

uint64_t span_nhwc(int N, int64_t nstride, int32_t cstride, int HW, int C, int esz) {
    if (N <= 0) return 0;
    return (uint64_t)(((int64_t)(N - 1) * nstride + (int64_t)(HW - 1) * cstride + C) * esz);
}

}  // namespace

hipError_t launch_conv_int8_pg16(const ConvParams& p0, hipStream_t stream) {
    const bool packed = p0.loader == kLoaderPackedNc4;
    const bool nchw_out = (p0.flags & kConvOutNchw) != 0;
    if ((p0.loader != kLoaderNhwc && !packed) || p0.C % 16 || p0.C > 16 * kPgMaxGroups || p0.OC % 4 ||
        p0.Kp % 64 || p0.OCp % 16 || p0.acc_out || !p0.x_slots.p || !(p0.KH == p0.KW) ||
        (p0.KH != 1 && p0.KH != 3) || (nchw_out && (p0.flags & kConvResidual)))
        return hipErrorInvalidValue;
    const bool out_f32 = (p0.flags & kConvOutF32) != 0;
    const int HWi = p0.H * p0.W, HWo = p0.OH * p0.OW;
    const uint64_t x_img = packed ? (uint64_t)p0.C * HWi
                                  : std::max((uint64_t)p0.x_nstride * 2, (uint64_t)HWi * p0.x_cstride * 2);
    const uint64_t y_img = nchw_out ? (uint64_t)p0.OC * HWo * (out_f32 ? 4 : 2)
                                    : std::max((uint64_t)p0.y_nstride, (uint64_t)HWo * p0.y_cstride) *
                                          (out_f32 ? 4 : 2);
    const uint64_t per_img = std::max({x_img, y_img, p0.res ? (uint64_t)p0.r_nstride * 2 : 0});
    if ((uint64_t)p0.OCp * p0.Kp > kMaxViewBytes || per_img == 0) return hipErrorInvalidValue;
    const int per_launch = (int)std::min<uint64_t>((uint64_t)p0.N, kMaxViewBytes / per_img);
    if (per_launch < 1) return hipErrorInvalidValue;
    for (int nb = 0; nb < p0.N; nb += per_launch) {
        ConvParams p = p0;
        p.N = std::min(per_launch, p0.N - nb);
        p.M = p.N * HWo;
        if (packed) {
            p.x = static_cast<const uint8_t*>(p0.x) + (int64_t)nb * p0.C * HWi;
            p.x_bytes = (uint32_t)((uint64_t)p.N * p.C * HWi);
        } else {
            p.x = static_cast<const __half*>(p0.x) + (int64_t)nb * p0.x_nstride;
            p.x_bytes = (uint32_t)span_nhwc(p.N, p.x_nstride, p.x_cstride, HWi, p.C, 2);
        }
        const int esz = out_f32 ? 4 : 2;
        if (nchw_out) {
            p.y = static_cast<char*>(p0.y) + (int64_t)nb * p0.OC * HWo * esz;
            p.y_bytes = (uint32_t)((uint64_t)p.N * p.OC * HWo * esz);
        } else {
            p.y = static_cast<char*>(p0.y) + (int64_t)nb * p0.y_nstride * esz;
            p.y_bytes = (uint32_t)span_nhwc(p.N, p.y_nstride, p.y_cstride, HWo, p.OC, esz);
        }
        if (p0.res) {
            p.res = p0.res + (int64_t)nb * p0.r_nstride;
            p.r_bytes = (uint32_t)span_nhwc(p.N, p.r_nstride, p.r_cstride, HWo, p.OC, 2);
        }
        p.fd_ohw = make_fastdiv((uint32_t)HWo);
        p.fd_ow = make_fastdiv((uint32_t)p.OW);
        p.fd_ns = make_fastdiv((uint32_t)(p.C / 16));
        // the window kernel quantizes an input element once instead of up to nine
        // times per 16 channels, and reads weights from LDS; its longer start and
        // its barrier per group cost more on short grids of few groups.  us, this
        // kernel and the window kernel: 128 -> 128 at 40x40 x16 73.5, 29.4; 64 -> 64 at
        // 40x40 x8 (800 blocks) 16.7, 8.5; 256 -> 256 at 20x20 (112) 16.0, 13.7; 96 -> 48
        // at 27x35 x5 (222) 7.1, 9.2; 48 -> 144 at 33x17 x3 (243) 4.8, 6.4; 320 -> 96 at
        // 7x7 (6) 13.8, 19.6
        const int64_t blocks = pg_blocks(p);
        if (!packed && !nchw_out && p.KH == 3 && (blocks >= 400 || (blocks >= 64 && p.C >= 128))) {
            const hipError_t e = launch_conv_halo_pg16(p, stream);
            if (e == hipSuccess) continue;
            if (e != hipErrorNotSupported) return e;
        }
        if (p.KH == 1) {
            if (packed) launch_pg<1, kLoaderPackedNc4>(p, stream);
            else launch_pg<1, kLoaderNhwc>(p, stream);
        } else {
            if (packed) launch_pg<9, kLoaderPackedNc4>(p, stream);
            else launch_pg<9, kLoaderNhwc>(p, stream);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_quant_fused_pg16(const void* x, bool f16, int N, int C, int HW, uint32_t* packed,
                                   uint32_t* amax, hipStream_t stream) {
    if (!x || !packed || !amax || N < 1 || C < 16 || C % 16 || HW < 1) return hipErrorInvalidValue;
    const int64_t blocks = (int64_t)N * (C / 16);
    if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
    if (f16)
        hipLaunchKernelGGL(quant_fused_pg16_kernel<__half>, dim3((unsigned)blocks), dim3(kFusedThreads), 0, stream,
                           static_cast<const __half*>(x), C, HW, packed, amax);
    else
        hipLaunchKernelGGL(quant_fused_pg16_kernel<float>, dim3((unsigned)blocks), dim3(kFusedThreads), 0, stream,
                           static_cast<const float*>(x), C, HW, packed, amax);
    return hipGetLastError();
}

}  // namespace aexrt
