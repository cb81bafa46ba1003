// YOLO output0 postprocess: decode + confidence filter, class-wise NMS and
// top-k, as the reference runs it on the GPU after the network
// (native/aexrt_d3d12_runtime.cpp:15300-15356 decode/filter, 15637-15691 NMS
// mark, 15693-15735 top-k; recorded at 27104-27219).
//
// The reference uses three dispatches and appends candidates with an atomic
// counter, so their order (and which ones survive the max_candidates cap) is
// whatever order its threads ran in.  Here candidates are in anchor order (one
// of the orders the reference can produce, and a deterministic one).  Two
// launches share a workspace: one scores every anchor (post_score_kernel),
// one compacts, marks and ranks the candidates (post_select_kernel).  Without
// a workspace (launches recorded into a graph, more anchors than it holds) one
// 1024-thread block does all of it in LDS (yolo_decode_nms_topk_kernel).
//
// Two decoders feed the same NMS and top-k:
// * decoded output0 ([4 (+1 objectness) + classes][anchors]: cx, cy, w, h,
//   scores), RT:15300-15356;
// * the raw Detect head ([64 + classes][anchors]: 4 x 16 DFL bin logits, then
//   class logits; anchors level by level), the post-conv part of the
//   reference's fused head decode (RT:15465-15636): score = sigmoid(logit),
//   per side the softmax expectation of the 16 bins, box = (anchor centre -/+
//   distance) x stride.
//
// Arithmetic follows the reference's expressions one operation at a time
// (no contraction): x1 = cx - 0.5 w, IoU = inter / max(area_a + area_b -
// inter, 1e-7) with IEEE division, strict-greater class argmax (first max
// wins), a candidate passes unless score < conf.  exp is post_exp below (the
// reference's comes from its shader compiler and driver), so that results
// are reproducible bit for bit on the host.
#include <algorithm>
#include <map>
#include <mutex>

#include "common.h"
#include "kernels.h"

extern "C" hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus*) __attribute__((weak));

namespace aexrt {

namespace {

constexpr int kPostThreads = 1024;
constexpr int kPostWaves = kPostThreads / 64;
constexpr int kDflBins = 16;

struct PostParams {
    const float* out;  // element (channel ch, anchor a) at out[ch * ch_stride + a * a_stride]
    int ch_stride, a_stride;
    int anchors, classes, has_obj;
    float conf, iou;
    int max_cand, max_det;
    float* dets;       // [max_det][6]: x1, y1, x2, y2, score, class
    uint32_t* count;   // detections written
    // raw-head decode: level l covers anchors [lev_off[l], lev_off[l+1]) of a
    // grid lev_w[l] wide, stride lev_stride[l]
    int nlev;
    int lev_off[kYoloMaxLevels + 1];
    int lev_w[kYoloMaxLevels];
    float lev_stride[kYoloMaxLevels];
};

// e^x in fp32: Cody-Waite reduction x = k ln2 + r with ln2 split into a
// 16-bit head (k * head is exact) and a tail, |r| <= ln2/2, e^r by its
// degree-7 Taylor polynomial (truncation < 6e-9 relative) in Horner form,
// scaled by 2^k.  Below -87 it returns 0 (the true value is under 2e-38),
// above 88.5 infinity.
__device__ __forceinline__ float post_exp(float x) {
#pragma clang fp contract(off)
    if (x != x) return x;
    if (x < -87.0f) return 0.0f;
    if (x > 88.5f) return __builtin_inff();
    const float k = __builtin_rintf(x * 1.44269504f);
    const float r = (x - k * 0.693145751953125f) - k * 1.42860677e-06f;
    float p = 1.0f / 5040.0f;
    p = p * r + 1.0f / 720.0f;
    p = p * r + 1.0f / 120.0f;
    p = p * r + 1.0f / 24.0f;
    p = p * r + 1.0f / 6.0f;
    p = p * r + 0.5f;
    p = p * r + 1.0f;
    p = p * r + 1.0f;
    return __builtin_ldexpf(p, (int)k);
}

__device__ __forceinline__ float post_sigmoid(float x) {
#pragma clang fp contract(off)
    return 1.0f / (1.0f + post_exp(-x));
}

__device__ __forceinline__ float box_iou(const float* a, const float* b) {
#pragma clang fp contract(off)
    const float x1 = fmaxf(a[0], b[0]);
    const float y1 = fmaxf(a[1], b[1]);
    const float x2 = fminf(a[2], b[2]);
    const float y2 = fminf(a[3], b[3]);
    const float iw = fmaxf(0.0f, x2 - x1);
    const float ih = fmaxf(0.0f, y2 - y1);
    const float inter = iw * ih;
    const float area_a = fmaxf(0.0f, a[2] - a[0]) * fmaxf(0.0f, a[3] - a[1]);
    const float area_b = fmaxf(0.0f, b[2] - b[0]) * fmaxf(0.0f, b[3] - b[1]);
    return inter / fmaxf(area_a + area_b - inter, 1e-7f);
}

// j outranks i: higher score, or equal score and earlier candidate
__device__ __forceinline__ bool outranks(float sj, int j, float si, int i) { return sj > si || (sj == si && j < i); }

template <bool DFL>
__global__ __launch_bounds__(kPostThreads) void yolo_decode_nms_topk_kernel(PostParams p) {
#pragma clang fp contract(off)
    extern __shared__ float l_cand[];  // [max_cand][6], then keep flags [max_cand]
    uint32_t* l_keep = reinterpret_cast<uint32_t*>(l_cand + 6 * p.max_cand);
    __shared__ uint32_t l_wsum[kPostWaves];
    __shared__ uint32_t l_total;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) l_total = 0;
    __syncthreads();
    const int cls_off = p.has_obj ? 5 : 4;
    // ---- decode + filter, compacted in anchor order ----
    for (int a0 = 0; a0 < p.anchors; a0 += kPostThreads) {
        const int a = a0 + tid;
        bool pass = false;
        float best = 0.0f;
        int best_cls = 0;
        if (a < p.anchors && p.classes > 0) {
            const float* col = p.out + (int64_t)a * p.a_stride;
            if constexpr (DFL) {
                const int c0 = 4 * kDflBins;
                best = post_sigmoid(col[(int64_t)c0 * p.ch_stride]);
                for (int c = 1; c < p.classes; ++c) {
                    const float s = post_sigmoid(col[(int64_t)(c0 + c) * p.ch_stride]);
                    if (s > best) {
                        best = s;
                        best_cls = c;
                    }
                }
            } else {
                const float obj = p.has_obj ? col[4 * (int64_t)p.ch_stride] : 1.0f;
                best = obj * col[(int64_t)cls_off * p.ch_stride];
                for (int c = 1; c < p.classes; ++c) {
                    const float s = obj * col[(int64_t)(cls_off + c) * p.ch_stride];
                    if (s > best) {
                        best = s;
                        best_cls = c;
                    }
                }
            }
            pass = !(best < p.conf);
        }
        const uint64_t m = __ballot(pass);
        const uint32_t below = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        if (lane == 0) l_wsum[wave] = (uint32_t)__popcll(m);
        __syncthreads();
        uint32_t off = l_total;
        for (int w = 0; w < wave; ++w) off += l_wsum[w];
        const uint32_t idx = off + below;
        if (pass && idx < (uint32_t)p.max_cand) {
            const float* col = p.out + (int64_t)a * p.a_stride;
            float* c = l_cand + 6 * idx;
            if constexpr (DFL) {
                // side d: softmax expectation of bins 16d..16d+15
                float dist[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    float m = -3.402823e38f;
                    for (int b = 0; b < kDflBins; ++b) m = fmaxf(m, col[(int64_t)(d * kDflBins + b) * p.ch_stride]);
                    float sum = 0.0f, acc = 0.0f;
                    for (int b = 0; b < kDflBins; ++b) {
                        const float e = post_exp(col[(int64_t)(d * kDflBins + b) * p.ch_stride] - m);
                        sum = sum + e;
                        acc = acc + e * (float)b;
                    }
                    dist[d] = acc / fmaxf(sum, 1e-20f);
                }
                int l = 0;
                while (l + 1 < p.nlev && a >= p.lev_off[l + 1]) ++l;
                const int pos = a - p.lev_off[l];
                const int gy = pos / p.lev_w[l];
                const float ax = (float)(pos - gy * p.lev_w[l]) + 0.5f, ay = (float)gy + 0.5f;
                const float st = p.lev_stride[l];
                c[0] = (ax - dist[0]) * st;
                c[1] = (ay - dist[1]) * st;
                c[2] = (ax + dist[2]) * st;
                c[3] = (ay + dist[3]) * st;
            } else {
                const float cx = col[0], cy = col[p.ch_stride], w = col[2 * (int64_t)p.ch_stride],
                            h = col[3 * (int64_t)p.ch_stride];
                const float hw = 0.5f * w, hh = 0.5f * h;
                c[0] = cx - hw;
                c[1] = cy - hh;
                c[2] = cx + hw;
                c[3] = cy + hh;
            }
            c[4] = best;
            c[5] = (float)best_cls;
        }
        __syncthreads();
        if (tid == 0) {
            uint32_t t = l_total;
            for (int w = 0; w < kPostWaves; ++w) t += l_wsum[w];
            l_total = t;
        }
        __syncthreads();
    }
    const int count = (int)min(l_total, (uint32_t)p.max_cand);
    // ---- NMS mark: dropped when a same-class candidate that outranks it overlaps it ----
    for (int i = tid; i < count; i += kPostThreads) {
        const float* ci = l_cand + 6 * i;
        uint32_t keep = 1u;
        for (int j = 0; j < count; ++j) {
            if (j == i) continue;
            const float* cj = l_cand + 6 * j;
            if (cj[5] != ci[5]) continue;
            if (outranks(cj[4], j, ci[4], i) && box_iou(ci, cj) > p.iou) {
                keep = 0u;
                break;
            }
        }
        l_keep[i] = keep;
    }
    __syncthreads();
    // ---- top-k: a kept candidate's rank among the kept ones is its slot ----
    uint32_t kept = 0;
    for (int i = tid; i < count; i += kPostThreads) {
        if (!l_keep[i]) continue;
        ++kept;
        const float* ci = l_cand + 6 * i;
        int rank = 0;
        for (int j = 0; j < count; ++j)
            if (j != i && l_keep[j] && outranks(l_cand[6 * j + 4], j, ci[4], i)) ++rank;
        if (rank < p.max_det)
            for (int k = 0; k < 6; ++k) p.dets[6 * rank + k] = ci[k];
    }
    // ranks of the kept candidates are 0..K-1, so the count is min(K, max_det)
    uint32_t ws = kept;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) ws += (uint32_t)__shfl_xor((int)ws, o, 64);
    if (lane == 0) l_wsum[wave] = ws;
    __syncthreads();
    if (tid == 0) {
        uint32_t k = 0;
        for (int w = 0; w < kPostWaves; ++w) k += l_wsum[w];
        p.count[0] = min(k, (uint32_t)p.max_det);
    }
}

// ---- the same over the whole GPU --------------------------------------------------
//
// One block is bound by its CU: at 8400 anchors x 80 classes it took 440 us,
// 317 us at 2100 anchors with 512 candidates (a sigmoid per class and anchor,
// then count^2 steps of NMS and of ranking).  Spread over the CUs both parts
// are a chain of a few memory round trips: 14.6 + 14.0 us, and 14.5 + 18.2 us.

// Workspace of one postprocess: per anchor the box and (score, class), a bit
// per anchor that passed, then per candidate its rank and whether it is kept.
constexpr int kWsAnchors = 36864;  // up to 1280 x 1280 pixels (33600)
struct PostWs {
    float4 box[kWsAnchors];
    float2 score[kWsAnchors];
    uint64_t passed[kWsAnchors / 64];
    uint32_t mark[kYoloMaxCandidates];
    uint32_t blocks_done;
    uint32_t unused[63];
};

constexpr int kScoreAnchors = 64;  // anchors of a score block, four threads each
constexpr int kScoreChunk = 20;    // class scores in flight per thread (a quarter of 80)

// LAST: channels last (the four threads of an anchor are neighbours and read
// its row); otherwise channels first (a wave reads 64 neighbouring anchors of
// one class).  Each thread takes a quarter of the classes, then one side of the
// box of an anchor that passes.
template <bool DFL, bool LAST>
__global__ __launch_bounds__(4 * kScoreAnchors) void post_score_kernel(PostParams p, PostWs* ws, int vec) {
#pragma clang fp contract(off)
    __shared__ float l_best[4][kScoreAnchors];
    __shared__ int l_cls[4][kScoreAnchors];
    const int tid = threadIdx.x;
    const int al = LAST ? tid >> 2 : tid & (kScoreAnchors - 1);
    const int part = LAST ? tid & 3 : tid / kScoreAnchors;
    const int a = blockIdx.x * kScoreAnchors + al;
    const bool on = a < p.anchors;
    if (blockIdx.x == 0 && tid == 0) ws->blocks_done = 0u;
    const float* col = p.out + (int64_t)(on ? a : 0) * p.a_stride;
    const int64_t cs = LAST ? 1 : p.ch_stride;
    const float* sc = col + (DFL ? 4 * kDflBins : (p.has_obj ? 5 : 4)) * cs;
    const float obj = !DFL && p.has_obj ? col[4 * cs] : 1.0f;
    const int per = (p.classes + 3) / 4;
    const int lo = min(part * per, p.classes), hi = min(lo + per, p.classes);
    // this quarter's first largest value, and the largest of its others
    float m = -__builtin_inff(), next = -__builtin_inff();
    int cls = 0;
    for (int c0 = lo; c0 < hi; c0 += kScoreChunk) {
        float t[kScoreChunk];
        if (LAST && vec) {
#pragma unroll
            for (int i = 0; i < kScoreChunk; i += 4)
                *reinterpret_cast<float4*>(t + i) = *reinterpret_cast<const float4*>(sc + min(c0 + i, hi - 4));
        } else {
#pragma unroll
            for (int i = 0; i < kScoreChunk; ++i) t[i] = sc[min(c0 + i, hi - 1) * cs];
        }
#pragma unroll
        for (int i = 0; i < kScoreChunk; ++i) {
            const float s = DFL ? t[i] : obj * t[i];
            if (c0 + i < hi) {
                next = fmaxf(next, fminf(m, s));
                if (s > m) {
                    m = s;
                    cls = c0 + i;
                }
            }
        }
    }
    float best = m;
    if constexpr (DFL) {
        // the largest logit has the largest sigmoid; one so close that rounding can bring its
        // sigmoid level (up to 8 the sigmoid still grows by over 50 ulp in 0.01; beyond -88 it is
        // 0 for all) has the sigmoids decide
        const float near = m < -80.0f ? -__builtin_inff() : fminf(m, 8.0f) - 0.01f;
        best = hi > lo ? post_sigmoid(m) : -__builtin_inff();
        if (hi > lo && next >= near) {
            best = -__builtin_inff();
            for (int c = lo; c < hi; ++c) {
                const float s = post_sigmoid(sc[c * cs]);
                if (s > best) {
                    best = s;
                    cls = c;
                }
            }
        }
    }
    if (part == 0) {
        // the comparison starts at class 0: a NaN there stays
        const float s0 = DFL ? sc[0] : obj * sc[0];
        if (s0 != s0) {
            best = s0;
            cls = 0;
        }
    }
    l_best[part][al] = best;
    l_cls[part][al] = cls;
    __syncthreads();
    best = l_best[0][al];
    cls = l_cls[0][al];
#pragma unroll
    for (int q = 1; q < 4; ++q) {
        const float b = l_best[q][al];
        if (b > best) {
            best = b;
            cls = l_cls[q][al];
        }
    }
    const bool pass = on && !(best < p.conf);
    if (pass) {
        float coord;  // x1, y1, x2, y2
        if constexpr (DFL) {
            // side `part`: softmax expectation of its 16 bins
            float v[kDflBins];
#pragma unroll
            for (int b = 0; b < kDflBins; ++b) v[b] = col[(part * kDflBins + b) * cs];
            float top = -3.402823e38f;
#pragma unroll
            for (int b = 0; b < kDflBins; ++b) top = fmaxf(top, v[b]);
            float sum = 0.0f, acc = 0.0f;
#pragma unroll
            for (int b = 0; b < kDflBins; ++b) {
                const float e = post_exp(v[b] - top);
                sum = sum + e;
                acc = acc + e * (float)b;
            }
            const float dist = acc / fmaxf(sum, 1e-20f);
            int l = 0;
            while (l + 1 < p.nlev && a >= p.lev_off[l + 1]) ++l;
            const int pos = a - p.lev_off[l];
            const int gy = pos / p.lev_w[l];
            const float ctr = (float)(part & 1 ? gy : pos - gy * p.lev_w[l]) + 0.5f;
            coord = (part < 2 ? ctr - dist : ctr + dist) * p.lev_stride[l];
        } else {
            const float ctr = col[(part & 1) * cs], half = 0.5f * col[(2 + (part & 1)) * cs];
            coord = part < 2 ? ctr - half : ctr + half;
        }
        reinterpret_cast<float*>(ws->box + a)[part] = coord;
        if (part == 0) ws->score[a] = make_float2(best, (float)cls);
    }
    // the pass bits of the 64 anchors (a wave of channels first, 16 a wave otherwise)
    if constexpr (LAST) {
        uint64_t b = __ballot(pass && part == 0);
        // every fourth bit -> 16 bits
        b = (b | (b >> 3)) & 0x0303030303030303ull;
        b = (b | (b >> 6)) & 0x000F000F000F000Full;
        b = (b | (b >> 12)) & 0x000000FF000000FFull;
        if ((tid & 63) == 0)
            reinterpret_cast<uint16_t*>(ws->passed + blockIdx.x)[tid >> 6] = (uint16_t)(b | (b >> 24));
    } else {
        const uint64_t b = __ballot(pass);
        if (tid == 0) ws->passed[blockIdx.x] = b;
    }
}

// Total order of scores as unsigned keys: larger score, larger key; -0 counts as
// 0 and a NaN comes first, so that ranks are a permutation.
__device__ __forceinline__ uint32_t score_key(float s) {
    if (s != s) return 0xFFFFFFFFu;
    const uint32_t u = __float_as_uint(s + 0.0f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr int kSelThreads = 512;
constexpr int kSelWaves = kSelThreads / 64;
constexpr uint32_t kKept = 0x80000000u;

// Sum of v over the threads before this one; total = the block's sum.  sums:
// one word per wave.
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* sums, uint32_t& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, o, 64);
        if (lane >= o) x += y;
    }
    __syncthreads();  // sums of an earlier scan are read
    if (lane == 63) sums[wave] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kSelWaves; ++w) {
        const uint32_t t = sums[w];
        before += w < wave ? t : 0u;
        all += t;
    }
    total = all;
    return before + x - v;
}

// Every block gathers all candidates into LDS, marks and ranks its share of
// them (several threads to a candidate), and the last block to finish writes
// the detections.  The count^2 steps of 512 candidates, many of one class, are
// 50 us of one CU.
__global__ __launch_bounds__(kSelThreads) void post_select_kernel(PostParams p, PostWs* ws) {
    extern __shared__ float l_cand[];  // [max_cand][6] in anchor order, then a key each
    uint32_t* l_key = reinterpret_cast<uint32_t*>(l_cand + 6 * p.max_cand);
    __shared__ uint32_t l_sums[kSelWaves];
    __shared__ uint32_t l_last;
    const int tid = threadIdx.x;
    const int words = (p.anchors + 63) / 64;
    uint32_t found = 0;
    for (int w0 = 0; w0 < words && found < (uint32_t)p.max_cand; w0 += kSelThreads) {
        uint64_t b = w0 + tid < words ? ws->passed[w0 + tid] : 0ull;
        uint32_t all;
        uint32_t k = found + block_scan((uint32_t)__popcll(b), l_sums, all);
        // candidate k's anchor, in its class word until the gather
        for (; b && k < (uint32_t)p.max_cand; b &= b - 1, ++k)
            l_cand[6 * k + 5] = __int_as_float((w0 + tid) * 64 + __builtin_ctzll(b));
        found += all;
    }
    const int count = (int)min(found, (uint32_t)p.max_cand);
    __syncthreads();
    for (int i = tid; i < count; i += kSelThreads) {
        const int a = __float_as_int(l_cand[6 * i + 5]);
        const float4 b = ws->box[a];
        const float2 s = ws->score[a];
        float* c = l_cand + 6 * i;
        c[0] = b.x;
        c[1] = b.y;
        c[2] = b.z;
        c[3] = b.w;
        c[4] = s.x;
        c[5] = s.y;
        l_key[i] = score_key(s.x);
    }
    __syncthreads();
    // ---- this block's candidates: blockIdx, blockIdx + grid, ... ----
    const int mine = count > (int)blockIdx.x ? (count - 1 - (int)blockIdx.x) / (int)gridDim.x + 1 : 0;
    int per = 1;  // threads to a candidate
    while (per < 64 && 2 * per * mine <= kSelThreads) per <<= 1;
    for (int m0 = 0; m0 < mine; m0 += kSelThreads / per) {
        const int m = m0 + tid / per, share = tid & (per - 1);
        uint32_t rank = 0;
        bool drop = false;
        const int i = blockIdx.x + m * gridDim.x;
        if (m < mine) {
            const float* ci = l_cand + 6 * i;
            const uint32_t ki = l_key[i];
            const bool ordered = ci[4] == ci[4];  // a NaN score drops nothing and is not dropped
            for (int j = share; j < count; j += per) {
                const uint32_t kj = l_key[j];
                if (!(kj > ki || (kj == ki && j < i))) continue;
                ++rank;
                const float* cj = l_cand + 6 * j;
                if (!drop && ordered && cj[5] == ci[5] && cj[4] == cj[4]) drop = box_iou(ci, cj) > p.iou;
            }
        }
        for (int o = 1; o < per; o <<= 1) {
            rank += (uint32_t)__shfl_xor((int)rank, o, 64);
            drop = __shfl_xor((int)drop, o, 64) || drop;
        }
        if (m < mine && share == 0)
            __hip_atomic_store(&ws->mark[i], rank | (drop ? 0u : kKept), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // ---- the last block: kept candidates in rank order ----
    __threadfence();
    __syncthreads();
    if (tid == 0) l_last = atomicAdd(&ws->blocks_done, 1u) == gridDim.x - 1 ? 1u : 0u;
    __syncthreads();
    if (!l_last) return;
    __threadfence();
    uint32_t* l_by = l_key;  // by rank: candidate + 1, 0 when dropped
    for (int i = tid; i < count; i += kSelThreads) {
        const uint32_t mi = __hip_atomic_load(&ws->mark[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        l_by[mi & ~kKept] = mi & kKept ? (uint32_t)i + 1u : 0u;
    }
    __syncthreads();
    uint32_t kept = 0;
    for (int r0 = 0; r0 < count; r0 += kSelThreads) {
        const uint32_t c = r0 + tid < count ? l_by[r0 + tid] : 0u;
        uint32_t all;
        const uint32_t row = kept + block_scan(c ? 1u : 0u, l_sums, all);
        if (c && row < (uint32_t)p.max_det)
            for (int k = 0; k < 6; ++k) p.dets[6 * (int64_t)row + k] = l_cand[6 * (c - 1) + k];
        kept += all;
    }
    if (tid == 0) p.count[0] = min(kept, (uint32_t)p.max_det);
}

// Workspaces: a few per device, each handed from call to call in the order of
// the streams (a call waits for the event behind the slot's last one), so that
// calls on any number of threads and streams are safe.
constexpr int kWsSlots = 4;
__device__ PostWs g_post_ws[kWsSlots];

struct WsPool {
    PostWs* ws = nullptr;
    hipEvent_t done[kWsSlots] = {};
    hipStream_t last[kWsSlots] = {};
    int next = 0;
};
std::mutex g_ws_mutex;
std::map<int, WsPool> g_ws;

// The device's pool, nullptr when it cannot be set up.
WsPool* ws_pool() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    WsPool& w = g_ws[dev];
    if (!w.ws) {
        for (hipEvent_t& e : w.done)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventDisableSystemFence) != hipSuccess) {
                e = nullptr;
                return nullptr;
            }
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_post_ws)) != hipSuccess) return nullptr;
        w.ws = static_cast<PostWs*>(p);
    }
    return &w;
}

// A launch recorded into a graph may be replayed at any time, beside any other
// call: it has no slot.
bool recording(hipStream_t stream) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    // absent from the host stand-in of the HIP runtime, which records nothing here
    if (!hipStreamIsCapturing) return false;
    return hipStreamIsCapturing(stream, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}

template <bool DFL>
void launch_post(const PostParams& p, PostWs* ws, hipStream_t stream) {
    const dim3 blocks((unsigned)((p.anchors + kScoreAnchors - 1) / kScoreAnchors));
    const int cls_off = DFL ? 4 * kDflBins : (p.has_obj ? 5 : 4);
    const int vec = p.a_stride % 4 == 0 && cls_off % 4 == 0 && p.classes % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(p.out) % 16 == 0;
    if (p.ch_stride == 1)
        hipLaunchKernelGGL((post_score_kernel<DFL, true>), blocks, dim3(4 * kScoreAnchors), 0, stream, p, ws, vec);
    else
        hipLaunchKernelGGL((post_score_kernel<DFL, false>), blocks, dim3(4 * kScoreAnchors), 0, stream, p, ws, vec);
    // 16 candidates to a block: 32 threads to each
    const int sel = std::min(64, (p.max_cand + 15) / 16);
    hipLaunchKernelGGL(post_select_kernel, dim3((unsigned)sel), dim3(kSelThreads),
                       (size_t)p.max_cand * 7 * sizeof(float), stream, p, ws);
}

}  // namespace

hipError_t launch_yolo_decode_nms_topk(const float* out, int ch_stride, int a_stride, int anchors, int classes,
                                       int has_objectness, float conf, float iou, int max_candidates,
                                       int max_detections, float* dets, uint32_t* count, hipStream_t stream,
                                       const YoloLevels* levels) {
    if ((!out && anchors > 0) || !dets || !count || anchors < 0 || classes < 0 || max_candidates < 1 ||
        max_candidates > kYoloMaxCandidates || max_detections < 1)
        return hipErrorInvalidValue;
    PostParams p{};
    p.out = out;
    p.ch_stride = ch_stride;
    p.a_stride = a_stride;
    p.anchors = anchors;
    p.classes = classes;
    p.has_obj = has_objectness ? 1 : 0;
    p.conf = conf;
    p.iou = iou;
    p.max_cand = max_candidates;
    p.max_det = max_detections;
    p.dets = dets;
    p.count = count;
    if (levels) {
        // raw Detect head: the levels must tile the anchors exactly
        if (has_objectness || levels->n < 1 || levels->n > kYoloMaxLevels) return hipErrorInvalidValue;
        int off = 0;
        for (int l = 0; l < levels->n; ++l) {
            if (levels->h[l] < 1 || levels->w[l] < 1) return hipErrorInvalidValue;
            p.lev_off[l] = off;
            p.lev_w[l] = levels->w[l];
            p.lev_stride[l] = levels->stride[l];
            off += levels->h[l] * levels->w[l];
        }
        p.lev_off[levels->n] = off;
        p.nlev = levels->n;
        if (off != anchors) return hipErrorInvalidValue;
    }
    if (anchors > 0 && anchors <= kWsAnchors && classes > 0 && !recording(stream)) {
        std::lock_guard<std::mutex> lock(g_ws_mutex);
        if (WsPool* w = ws_pool()) {
            int slot = 0;  // this stream's, else the next in turn
            while (slot < kWsSlots && w->last[slot] != stream) ++slot;
            if (slot == kWsSlots) {
                slot = w->next;
                w->next = (w->next + 1) % kWsSlots;
            }
            // an event never recorded is complete
            hipError_t e = hipStreamWaitEvent(stream, w->done[slot], 0);
            if (e != hipSuccess) return e;
            w->last[slot] = stream;
            if (levels) launch_post<true>(p, w->ws + slot, stream);
            else launch_post<false>(p, w->ws + slot, stream);
            e = hipGetLastError();
            const hipError_t r = hipEventRecord(w->done[slot], stream);
            return e != hipSuccess ? e : r;
        }
    }
    const size_t lds = (size_t)max_candidates * 7 * sizeof(float);
    if (levels)
        hipLaunchKernelGGL(yolo_decode_nms_topk_kernel<true>, dim3(1), dim3(kPostThreads), lds, stream, p);
    else
        hipLaunchKernelGGL(yolo_decode_nms_topk_kernel<false>, dim3(1), dim3(kPostThreads), lds, stream, p);
    return hipGetLastError();
}

}  // namespace aexrt
