// Winograd F(2x2,3x3) 3x3 s1 p1 convolution + bias + SiLU on fp16 MFMA
// (reference kernels 40/46, RT:2480-2631).
//
// Per 2x2 output tile the 4x4 input patch d is transformed to V = B^T d B
// (RT:2533-2548), the 16 transform points become 16 independent GEMMs
// M_r[tile][oc] = sum_c V_r[tile][c] * U_r[c][oc] with U = G g G^T prepared
// by the compiler (packed layout 3), and the output is A^T M A + bias
// (RT:2612-2619).  A block owns 16 or 32 tiles x 32 or 64 output channels; its V
// is staged in LDS per channel chunk, U ([16][OCp][Cp] fp16, repacked at load)
// streams from L2, and the output transform runs in registers.
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace aexrt {

namespace {

constexpr int WKC = 32;        // channels per K chunk of a wave
constexpr int VROW = WKC + 8;  // padded LDS row (halves)
constexpr uint32_t kOob = 0xFFFFFFF0u;

// 4x4 input patch -> V = B^T d B for one channel (RT:2533-2548).
__device__ __forceinline__ void input_transform(const float (&d)[4][4], float (&v)[16]) {
    float t[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        t[i][0] = d[i][0] - d[i][2];
        t[i][1] = d[i][1] + d[i][2];
        t[i][2] = -d[i][1] + d[i][2];
        t[i][3] = d[i][1] - d[i][3];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[0 * 4 + j] = t[0][j] - t[2][j];
        v[1 * 4 + j] = t[1][j] + t[2][j];
        v[2 * 4 + j] = -t[1][j] + t[2][j];
        v[3 * 4 + j] = t[1][j] - t[3][j];
    }
}

// The four outputs of one tile and channel from its 16 points: A^T M A
// (RT:2612-2619).
__device__ __forceinline__ void output_transform(const float (&mr)[16], float (&o)[4]) {
    float r0[4], r1[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        r0[q] = mr[0 * 4 + q] + mr[1 * 4 + q] + mr[2 * 4 + q];
        r1[q] = mr[1 * 4 + q] - mr[2 * 4 + q] - mr[3 * 4 + q];
    }
    o[0] = r0[0] + r0[1] + r0[2];
    o[1] = r0[1] - r0[2] - r0[3];
    o[2] = r1[0] + r1[1] + r1[2];
    o[3] = r1[1] - r1[2] - r1[3];
}

// Element offsets of tile T's first output position in the output and residual
// views.
struct TilePlace {
    int64_t y, r;
};
__device__ __forceinline__ TilePlace tile_place(const ConvParams& p, int T, int tiles_w, int tiles_img) {
    const int n = T / tiles_img;
    const int rem = T - n * tiles_img;
    const int ty = rem / tiles_w, tx = rem - ty * tiles_w;
    const int64_t pos = (int64_t)ty * 2 * p.OW + tx * 2;
    return {(int64_t)n * p.y_nstride + pos * p.y_cstride, (int64_t)n * p.r_nstride + pos * p.r_cstride};
}

// Bias, activation and residual of one output value, stored at element yo of
// the output; returns |value| as stored.
__device__ __forceinline__ float output_value(const ConvParams& p, float v, float bias, int64_t yo, int64_t ro) {
    v += bias;
    if (p.flags & kConvSilu) v = silu(v);
    const bool do_res = p.flags & kConvResidual;
    if (p.flags & kConvOutF32) {
        if (do_res) v = v + __half2float(p.res[ro]);
        reinterpret_cast<float*>(p.y)[yo] = v;
        return fabsf(v);
    }
    __half h = __float2half(v);
    if (do_res)  // fp16 conv output + fp16 residual, the reference's separate add
        h = __float2half(__half2float(h) + __half2float(p.res[ro]));
    reinterpret_cast<__half*>(p.y)[yo] = h;
    return fabsf(__half2float(h));
}

// The same for four consecutive channels of one position, one access each.
__device__ __forceinline__ float output_values4(const ConvParams& p, const float (&o)[4], const float (&bias)[4],
                                                int64_t yo, int64_t ro) {
    float v[4], g = 0.0f, res[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const bool do_res = p.flags & kConvResidual;
    if (do_res) {
        const uint2 h = *reinterpret_cast<const uint2*>(p.res + ro);
        const float2 lo = __half22float2(*reinterpret_cast<const __half2*>(&h.x));
        const float2 hi = __half22float2(*reinterpret_cast<const __half2*>(&h.y));
        res[0] = lo.x, res[1] = lo.y, res[2] = hi.x, res[3] = hi.y;
    }
    const bool do_silu = p.flags & kConvSilu;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[i] = o[i] + bias[i];
        if (do_silu) v[i] = silu(v[i]);
    }
    if (p.flags & kConvOutF32) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (do_res) v[i] = v[i] + res[i];
            g = fmaxf(g, fabsf(v[i]));
        }
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.y) + yo) = make_float4(v[0], v[1], v[2], v[3]);
        return g;
    }
    __half h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[i] = __float2half(v[i]);
        if (do_res) h[i] = __float2half(__half2float(h[i]) + res[i]);
        g = fmaxf(g, fabsf(__half2float(h[i])));
    }
    uint2 w;
    __builtin_memcpy(&w, h, 8);
    *reinterpret_cast<uint2*>(reinterpret_cast<__half*>(p.y) + yo) = w;
    return g;
}

// Four channels of a 4x4 patch -> V of the tile, four halves at vs[r * rstep]
// per transform point, written NQ channels at a time (2: half the registers).
template <int NQ>
__device__ __forceinline__ void transform4(const uint2 (&d)[4][4], _Float16* vs, int rstep) {
    typedef _Float16 vh __attribute__((ext_vector_type(NQ)));
#pragma unroll
    for (int q0 = 0; q0 < 4; q0 += NQ) {
        vh out[16];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            float dq[4][4], v[16];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t w = q0 + q < 2 ? d[i][j].x : d[i][j].y;
                    const float2 f = __half22float2(*reinterpret_cast<const __half2*>(&w));
                    dq[i][j] = (q0 + q) & 1 ? f.y : f.x;
                }
            input_transform(dq, v);
#pragma unroll
            for (int r = 0; r < 16; ++r) out[r][q] = (_Float16)v[r];
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) *reinterpret_cast<vh*>(vs + r * rstep + q0) = out[r];
        if (NQ < 4) __builtin_amdgcn_sched_barrier(0);
    }
}

// A block owns 16 TS tiles x 16 OW output channels: OW of its four waves
// across the channels, the others across the tile subtiles.  Each wave computes
// its (channel, tile) subtiles for all 16 points, so after the K loop a lane
// holds every point of four consecutive channels of a tile, transforms them in
// registers and stores 8 bytes a position.  What bounds it is latency: load a
// patch, transform, LDS, barrier, U from L2.  So a thread issues its 16 patch
// loads at once (out-of-range offsets read zero, no branch), the next chunk's
// while this one is multiplied, transforms four channels and writes 8 bytes to
// LDS per point, and a block of 16 tiles takes 64 channels a chunk.
// 64 -> 64 at 40 x 40, 8 images: 9.3 us (14.8 with 32 tiles x 32 channels,
// branched loads and a 2-byte LDS write per value).
template <int TS, int OW>
__global__ __launch_bounds__(256, TS) void winograd_f2x2_kernel(ConvParams p, int vec) {
    constexpr int T_BLK = 16 * TS;        // tiles of the block
    constexpr int KC = 1024 / T_BLK;      // channels of a chunk: four a thread
    constexpr int KS = KC / 32;           // MFMA k steps of a chunk
    constexpr int MT = TS * OW / 4;       // tile subtiles of a wave
    constexpr int ROW = KC + 8;
    __shared__ __attribute__((aligned(16))) _Float16 vs[16][T_BLK][ROW];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wn = wave % OW, wt = wave / OW;
    const int lr = lane & 15, lg = lane >> 4;

    const int tiles_w = p.OW / 2, tiles_h = p.OH / 2;
    const int tiles_img = tiles_w * tiles_h;
    const int ttot = p.N * tiles_img;
    const int ntn = (p.OC + 16 * OW - 1) / (16 * OW);
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int t0 = (b / ntn) * T_BLK;
    const int n0 = (b % ntn) * 16 * OW;

    // transform unit of this thread: tile tl, channels c4..c4+3 of the chunk
    const int tl = tid / (KC / 4);
    const int c4 = (tid % (KC / 4)) * 4;
    const int T = t0 + tl;
    uint32_t base = 0, inside = 0;  // byte offset of the patch's corner; its taps inside the image
    if (T < ttot) {
        const int n = T / tiles_img;
        const int rem = T - n * tiles_img;
        const int ty = rem / tiles_w;
        const int y0 = ty * 2 - 1, x0 = (rem - ty * tiles_w) * 2 - 1;
        base = (uint32_t)((int64_t)n * p.x_nstride + ((int64_t)y0 * p.W + x0) * p.x_cstride + c4) * 2u;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if ((unsigned)(y0 + i) < (unsigned)p.H && (unsigned)(x0 + j) < (unsigned)p.W)
                    inside |= 1u << (4 * i + j);
    }
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), 0, p.x_bytes, 0x00020000);
    uint2 d[4][4];
    auto load_patch = [&](int cb) {
        const bool cok = cb + c4 < p.C;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t off = base + (uint32_t)(i * p.W + j) * (uint32_t)p.x_cstride * 2u + (uint32_t)cb * 2u;
                const auto v = __builtin_amdgcn_raw_buffer_load_b64(
                    rx, cok && (inside >> (4 * i + j) & 1u) ? off : kOob, 0, 0);
                d[i][j] = make_uint2(v[0], v[1]);
            }
    };
    const int Cp = p.Kp;
    const int oc_u = min(n0 + wn * 16 + lr, p.OCp - 1);  // (rows past the last are not stored)
    const _Float16* U = reinterpret_cast<const _Float16*>(p.w) + (int64_t)oc_u * Cp + lg * 8;
    // the points of a k step, all at once or (with 32 accumulators a lane) half
    constexpr int UR = MT == 1 ? 16 : 8;
    auto load_u = [&](int c, int r0, v8h (&u)[UR]) {
#pragma unroll
        for (int r = 0; r < UR; ++r) u[r] = *reinterpret_cast<const v8h*>(U + (int64_t)(r0 + r) * p.OCp * Cp + c);
    };

    v4f acc[MT][16];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][r] = v4f{0, 0, 0, 0};

    // with 32 accumulators a lane has no registers for a second patch; the other
    // block of its CU fills the wait instead
    constexpr bool kAhead = MT == 1;
    if (kAhead) load_patch(0);
    for (int cb = 0; cb < Cp; cb += KC) {
        if (!kAhead) load_patch(cb);
        if (cb) __syncthreads();  // the previous chunk's MFMAs are done with vs
        transform4<MT == 1 ? 4 : 2>(d, &vs[0][tl][c4], T_BLK * ROW);
        if (kAhead && cb + KC < Cp) load_patch(cb + KC);
        constexpr int NU = KS * 16 / UR;
        v8h u[NU][UR];
        load_u(cb, 0, u[0]);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < NU; ++s) {
            const int ks = s * UR / 16, r0 = s * UR % 16;
            if (cb + ks * 32 >= Cp) break;
            if (s + 1 < NU && cb + (s + 1) * UR / 16 * 32 < Cp)
                load_u(cb + (s + 1) * UR / 16 * 32, (s + 1) * UR % 16, u[s + 1]);
#pragma unroll
            for (int r = 0; r < UR; ++r)
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const v8h v =
                        *reinterpret_cast<const v8h*>(&vs[r0 + r][(wt * MT + m) * 16 + lr][ks * 32 + lg * 8]);
                    acc[m][r0 + r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(u[s][r], v, acc[m][r0 + r], 0, 0, 0);
                }
            if (MT > 1) __builtin_amdgcn_sched_barrier(0);
        }
    }

    // lane: channels oc0 .. oc0 + 3 of tile t0 + (wt MT + m) 16 + lr; point r = 4*row + col
    const int oc0 = n0 + wn * 16 + lg * 4;
    float bias[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) bias[i] = oc0 + i < p.OC ? p.bias[oc0 + i] : 0.0f;
    float gmax = 0.0f;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int Ti = t0 + (wt * MT + m) * 16 + lr;
        if (Ti >= ttot || oc0 >= p.OC) continue;
        float o[4][4];  // [position][channel]
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float mr[16], oq[4];
#pragma unroll
            for (int r = 0; r < 16; ++r) mr[r] = acc[m][r][i];
            output_transform(mr, oq);
#pragma unroll
            for (int q = 0; q < 4; ++q) o[q][i] = oq[q];
        }
        const TilePlace at = tile_place(p, Ti, tiles_w, tiles_img);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t pos = (int64_t)(q >> 1) * p.OW + (q & 1);
            const int64_t yo = at.y + pos * p.y_cstride + oc0, ro = at.r + pos * p.r_cstride + oc0;
            if (vec && oc0 + 3 < p.OC) {
                gmax = fmaxf(gmax, output_values4(p, o[q], bias, yo, ro));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (oc0 + i < p.OC) gmax = fmaxf(gmax, output_value(p, o[q][i], bias[i], yo + i, ro + i));
            }
        }
    }
    if (p.y_slots.p) {
        gmax = wave_max(gmax);
        const int g = (n0 + wn * 16) / 16;
        if (lane == 0 && n0 + wn * 16 < p.OC && gmax > 0.0f) slot_max(slot_copy(p.y_slots, blockIdx.x) + g, gmax);
    }
}

// Small maps: a block owns 16 tiles x 16 output channels and its 4 waves
// split the 32-channel chunks (wave w takes chunks w, w+4, ...), each
// transforming its own chunk into a private LDS region, so the K loop needs
// no block barrier.  The partial point sums meet in LDS; wave w then runs the
// output transform of tiles 4*lg + w.
__global__ __launch_bounds__(256) void winograd_f2x2_ksplit_kernel(ConvParams p) {
    constexpr int ST = 16;  // tiles per block
    __shared__ __attribute__((aligned(16))) uint8_t lds[4 * 16 * ST * VROW * 2 > 4 * 16 * 4 * 64 * 4
                                                             ? 4 * 16 * ST * VROW * 2
                                                             : 4 * 16 * 4 * 64 * 4];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    _Float16 (*vs)[ST][VROW] = reinterpret_cast<_Float16 (*)[ST][VROW]>(lds + wave * 16 * ST * VROW * 2);

    const int tiles_w = p.OW / 2, tiles_h = p.OH / 2;
    const int tiles_img = tiles_w * tiles_h;
    const int ttot = p.N * tiles_img;
    const int ntn = (p.OC + 15) / 16;
    const int t0 = (blockIdx.x / ntn) * ST;
    const int n0 = (blockIdx.x % ntn) * 16;

    // transform unit of this lane: tile tl, channels c4..c4+3 (+16) of the chunk
    const int tl = lane >> 2;
    const int c4 = (lane & 3) * 4;
    const int T = t0 + tl;
    int y0 = 0, x0 = 0;
    int64_t xbase = 0;
    const bool t_ok = T < ttot;
    if (t_ok) {
        const int n = T / tiles_img;
        const int rem = T - n * tiles_img;
        const int ty = rem / tiles_w;
        const int tx = rem - ty * tiles_w;
        y0 = ty * 2 - 1;
        x0 = tx * 2 - 1;
        xbase = (int64_t)n * p.x_nstride;
    }
    const __half* xh = reinterpret_cast<const __half*>(p.x);
    const _Float16* U = reinterpret_cast<const _Float16*>(p.w);
    const int oc_b = n0 + lr;
    const bool oc_b_ok = oc_b < p.OCp;

    v4f acc[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = v4f{0, 0, 0, 0};

    const int Cp = p.Kp;
    for (int cb = wave * WKC; cb < Cp; cb += 4 * WKC) {
        v8h b[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if (oc_b_ok)
                b[r] = *reinterpret_cast<const v8h*>(U + ((int64_t)r * p.OCp + oc_b) * Cp + cb + lg * 8);
            else
                b[r] = v8h{0, 0, 0, 0, 0, 0, 0, 0};
        }
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int c = cb + half * 16 + c4;
            uint2 d[4][4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int iy = y0 + i, ix = x0 + j;
                    d[i][j] = make_uint2(0u, 0u);
                    if (t_ok && c < p.C && (unsigned)iy < (unsigned)p.H && (unsigned)ix < (unsigned)p.W)
                        d[i][j] = *reinterpret_cast<const uint2*>(xh + xbase + ((int64_t)iy * p.W + ix) * p.x_cstride +
                                                                  c);
                }
            transform4<4>(d, &vs[0][tl][half * 16 + c4], ST * VROW);
        }
        // the region is private to this wave: LDS operations of one wave
        // complete in order, only the compiler must not move them
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const v8h a = *reinterpret_cast<const v8h*>(&vs[r][lr][lg * 8]);
            acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[r], acc[r], 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();
    }

    // partial sums of the 4 waves: red[wave][r][i][lane]
    float* red = reinterpret_cast<float*>(lds);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[((wave * 16 + r) * 4 + i) * 64 + lane] = acc[r][i];
    __syncthreads();

    // wave w finishes tile row i = w: tiles t0 + lg*4 + w, channel n0 + lr
    const int oc = n0 + lr;
    const int Ti = t0 + lg * 4 + wave;
    float gmax = 0.0f;
    if (oc < p.OC && Ti < ttot) {
        float mr[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float t = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; ++w) t += red[((w * 16 + r) * 4 + wave) * 64 + lane];
            mr[r] = t;
        }
        float o[4];
        output_transform(mr, o);
        const TilePlace at = tile_place(p, Ti, tiles_w, tiles_img);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t pos = (int64_t)(q >> 1) * p.OW + (q & 1);
            gmax = fmaxf(gmax, output_value(p, o[q], p.bias[oc], at.y + pos * p.y_cstride + oc,
                                            at.r + pos * p.r_cstride + oc));
        }
    }
    if (p.y_slots.p) {
        gmax = wave_max(gmax);
        if (lane == 0 && n0 < p.OC && gmax > 0.0f) slot_max(slot_copy(p.y_slots, blockIdx.x) + n0 / 16, gmax);
    }
}

}  // namespace

namespace {
template <int TS, int OW>
void launch_tile(const ConvParams& p, int64_t ttot, int vec, hipStream_t stream) {
    const int64_t blocks = ((ttot + 16 * TS - 1) / (16 * TS)) * ((p.OC + 16 * OW - 1) / (16 * OW));
    hipLaunchKernelGGL((winograd_f2x2_kernel<TS, OW>), dim3((unsigned)blocks), dim3(256), 0, stream, p, vec);
}
}  // namespace

// Tile by the blocks it leaves.  16 tiles x 64 channels need a CU to themselves
// (registers), so they are for launches of at most one block a CU (64 -> 64 at
// 40 x 40 x 8: 9.3 us against 10.2 with 32 x 32; 256 -> 256 at 40 x 40 x 2: 24.8
// against 28.8).  Beyond that 32 tiles x 64 channels, two blocks to a CU (128 ->
// 128 at 20 x 20 x 32: 17.4 us against 27.0; 64 -> 64 at 40 x 40 x 64: 30.7, 104
// before these tiles), and with up to 32 output channels 32 x 32.  Few tiles and
// many channels (10x10 / 20x20 maps at small batch): the waves split the channels.
// Inputs over 2 GB go in several launches, one image over 2 GB by 64-bit addresses.
hipError_t launch_winograd_f2x2(const ConvParams& p0, hipStream_t stream) {
    const int HW = p0.H * p0.W, tiles_img = (p0.OH / 2) * (p0.OW / 2);
    const uint64_t image = std::max<uint64_t>((uint64_t)p0.x_nstride, (uint64_t)HW * p0.x_cstride) * 2;
    const bool f32 = (p0.flags & kConvOutF32) != 0;
    auto aligned = [](const void* q, int64_t ns, int64_t cs, uintptr_t bytes) {
        return reinterpret_cast<uintptr_t>(q) % bytes == 0 && ns % 4 == 0 && cs % 4 == 0;
    };
    const int vec = aligned(p0.y, p0.y_nstride, p0.y_cstride, f32 ? 16 : 8) &&
                    (!p0.res || aligned(p0.res, p0.r_nstride, p0.r_cstride, 8));
    const int64_t all = (int64_t)p0.N * tiles_img;
    const int oc64 = (p0.OC + 63) / 64;
    if (image > kMaxViewBytes || ((all + 15) / 16 * oc64 < 128 && p0.Kp >= 4 * WKC)) {
        const int64_t small = ((all + 15) / 16) * ((p0.OC + 15) / 16);
        hipLaunchKernelGGL(winograd_f2x2_ksplit_kernel, dim3((unsigned)small), dim3(256), 0, stream, p0);
        return hipGetLastError();
    }
    const int per = (int)std::min<uint64_t>((uint64_t)p0.N, kMaxViewBytes / std::max<uint64_t>(image, 1));
    for (int n0 = 0; n0 < p0.N; n0 += per) {
        ConvParams p = p0;
        p.N = std::min(per, p0.N - n0);
        p.x = static_cast<const __half*>(p0.x) + (int64_t)n0 * p0.x_nstride;
        p.y = static_cast<char*>(p0.y) + (int64_t)n0 * p0.y_nstride * (f32 ? 4 : 2);
        if (p0.res) p.res = p0.res + (int64_t)n0 * p0.r_nstride;
        p.x_bytes = (uint32_t)(((int64_t)(p.N - 1) * p.x_nstride + (int64_t)(HW - 1) * p.x_cstride + p.C) * 2);
        const int64_t ttot = (int64_t)p.N * tiles_img;
        if (p.OC <= 32) launch_tile<2, 2>(p, ttot, vec, stream);
        else if ((ttot + 15) / 16 * oc64 <= 256) launch_tile<1, 4>(p, ttot, vec, stream);
        else launch_tile<2, 4>(p, ttot, vec, stream);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace aexrt
