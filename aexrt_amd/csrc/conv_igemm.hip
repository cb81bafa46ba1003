// Host side of the implicit-GEMM conv (kernel in conv_igemm.h): per-wave tile
// choice, batch splitting for 32-bit view offsets, launch parameters.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>

#include "conv_igemm.h"

namespace aexrt {

namespace igemm {
AEXRT_IGEMM_FAMILIES(AEXRT_IGEMM_EXTERN)
}  // namespace igemm

namespace {

hipError_t launch_variant(bool int8, bool mc, int epi, const ConvParams& p, const ConvTile& t, hipStream_t s) {
    using igemm::launch_family;
    if (LaunchProbe* pr = launch_probe()) {
        // the kernel template instance (as a trace names it), then the tile
        std::snprintf(pr->name, sizeof(pr->name), "conv_mfma_kernel<%s,%d,%d,%s,%s,%d>", int8 ? "true" : "false",
                      t.jn, t.pw, t.ksw ? "true" : "false", mc ? "true" : "false", epi);
        return hipSuccess;
    }
    if (int8) {
        if (mc) {
            if (epi == 1) return launch_family<true, true, 1>(p, t, s);
            if (epi == 2) return launch_family<true, true, 2>(p, t, s);
            return launch_family<true, true, 0>(p, t, s);
        }
        if (epi == 1) return launch_family<true, false, 1>(p, t, s);
        if (epi == 2) return launch_family<true, false, 2>(p, t, s);
        return launch_family<true, false, 0>(p, t, s);
    }
    if (mc) return epi == 1 ? launch_family<false, true, 1>(p, t, s) : launch_family<false, true, 0>(p, t, s);
    return epi == 1 ? launch_family<false, false, 1>(p, t, s) : launch_family<false, false, 0>(p, t, s);
}

int pow2_at_least(int v, int cap) {
    int r = 1;
    while (r < v && r < cap) r <<= 1;
    return r;
}

// Byte span of an NHWC view of N images (0 when absent).
uint64_t view_span(int N, int64_t nstride, int32_t cstride, int HW, int C, int esz) {
    if (N <= 0) return 0;
    return (uint64_t)(((int64_t)(N - 1) * nstride + (int64_t)(HW - 1) * cstride + C) * esz);
}

}  // namespace

namespace {
thread_local LaunchProbe* g_probe = nullptr;
}  // namespace

void set_launch_probe(LaunchProbe* probe) { g_probe = probe; }
LaunchProbe* launch_probe() { return g_probe; }

void conv_kernel_name(const ConvParams& p, bool int8, char* out, size_t n) {
    LaunchProbe pr{};
    std::snprintf(pr.name, sizeof(pr.name), "none");
    LaunchProbe* prev = g_probe;
    g_probe = &pr;
    const hipError_t e = launch_conv_igemm(p, int8, nullptr);
    g_probe = prev;
    std::snprintf(out, n, "%s", e == hipSuccess ? pr.name : "not launchable");
}

namespace {
// jn * 100 + pw * 10 + ksw + 1, 0 = no override
std::atomic<int> g_tile_override{0};

bool tile_instantiated(const ConvTile& t) {
    if (t.ksw) return t.pw == 1 && (t.jn == 1 || t.jn == 2 || t.jn == 4 || t.jn == 8);
    switch (t.jn * 8 + t.pw) {
        case 9: case 10: case 12: case 17: case 18: case 20: case 33: case 34: case 36: case 65: case 66:
            return true;
    }
    return false;
}
}  // namespace

namespace {
bool tile_forced() { return g_tile_override.load(std::memory_order_relaxed) != 0; }
}  // namespace

bool set_conv_tile_override(int jn, int pw, int ksw) {
    if (jn == 0 && pw == 0 && ksw == 0) {
        g_tile_override.store(0);
        return true;
    }
    const ConvTile t{jn, pw, ksw != 0};
    if (!tile_instantiated(t)) return false;
    g_tile_override.store(jn * 100 + pw * 10 + (ksw ? 1 : 0) + 1);
    return true;
}

// Tile choice.  A block is 4 waves x pw 16-position subtiles by jn
// 16-channel subtiles and walks a run of such tiles with its weights resident
// in LDS.  Cover all output channels (up to 128) so activations are read
// once, with as many positions per wave as the registers allow; maps too small
// to give every CU a tile shrink the position tile, then the channel tile, and
// finally let the 4 waves of a block split k (one position subtile per block).
ConvTile choose_conv_tile(int M, int OC, int Kp) {
    const int ov = g_tile_override.load(std::memory_order_relaxed);
    if (ov) return ConvTile{(ov - 1) / 100, ((ov - 1) / 10) % 10, ((ov - 1) % 10) != 0};
    const int ocj = (OC + 15) / 16;
    const int nks = Kp / 64;
    auto tiles = [&](int jn, int pw, bool ksw) {
        return (int64_t)((M + (ksw ? 16 : 64) * pw - 1) / ((ksw ? 16 : 64) * pw)) * ((ocj + jn - 1) / jn);
    };
    const int64_t want = 256;  // one tile per CU at least
    int jn = pow2_at_least(ocj, 8);
    int pw = jn >= 8 ? 2 : (jn >= 4 ? 4 : 4);
    while (pw > 1 && tiles(jn, pw, false) < want) pw >>= 1;
    while (jn > 1 && tiles(jn, pw, false) < want) jn >>= 1;
    if (tiles(jn, pw, false) >= want / 2 || nks < 4) return ConvTile{jn, pw, false};
    // small map: one position subtile per block, k split over the 4 waves
    jn = pow2_at_least(ocj, 8);
    while (jn > 1 && tiles(jn, 1, true) < want) jn >>= 1;
    return ConvTile{jn, 1, true};
}

namespace {

// The same for fp16 1x1 convs, whose positions cost a load and nothing else:
// two position subtiles a wave keep more loads in flight than wide channel
// tiles, so the channel tile shrinks first, to four subtiles below 384 tiles and
// two below 256, and 96 tiles are enough for the rest.  Over 220 random shapes 1.05x the time of
// the fastest tile (the rule above 1.10x): 120 -> 320 channels at 111x111 10.4 ->
// 7.9 us, 24 -> 152 at 156x160 x16 51.8 -> 39.0.
ConvTile choose_f16_1x1_tile(int M, int OC, int Kp) {
    if (tile_forced()) return choose_conv_tile(M, OC, Kp);
    const int ocj = (OC + 15) / 16;
    auto tiles = [&](int jn, int pw, bool ksw) {
        return (int64_t)((M + (ksw ? 16 : 64) * pw - 1) / ((ksw ? 16 : 64) * pw)) * ((ocj + jn - 1) / jn);
    };
    int jn = pow2_at_least(ocj, 8), pw = 2;
    if (jn > 4 && tiles(jn, pw, false) < 384) jn = 4;
    if (jn > 2 && tiles(jn, pw, false) < 256) jn = 2;
    while (pw > 1 && tiles(jn, pw, false) < 96) pw >>= 1;
    while (jn > 1 && tiles(jn, pw, false) < 96) jn >>= 1;
    if (tiles(jn, pw, false) >= 96 || Kp / 64 < 4) return ConvTile{jn, pw, false};
    jn = pow2_at_least(ocj, 8);
    while (jn > 1 && tiles(jn, 1, true) < 256) jn >>= 1;
    return ConvTile{jn, 1, true};
}

}  // namespace

int enumerate_conv_choices(const ConvParams& p, bool int8, ConvChoice* out, int cap) {
    // a fused 1x1 runs only in the 32x32-MFMA kernel's epilogue
    if (p.fuse_1x1) return p.loader == kLoaderNhwc ? enumerate_m32_choices(p, int8, out, cap) : 0;
    // an upsample copy of the output: the streaming 1x1 kernel only
    if (p.yup || p.xup) return int8 && p.KH == 1 && p.KW == 1 ? enumerate_s1x1_choices(p, int8, out, cap) : 0;
    int n = 0;
    const bool nchw = p.loader == kLoaderNchwF32;
    if (!nchw && p.Kp / 64 <= igemm::kMaxSteps) {
        static const ConvTile tiles[] = {{1, 1, false}, {1, 2, false}, {1, 4, false}, {2, 1, false}, {2, 2, false},
                                         {2, 4, false}, {4, 1, false}, {4, 2, false}, {4, 4, false}, {8, 1, false},
                                         {8, 2, false}, {1, 1, true},  {2, 1, true},  {4, 1, true},  {8, 1, true}};
        const int ocj = (p.OCp + 15) / 16;
        for (const ConvTile& t : tiles) {
            if (n >= cap) break;
            if (t.jn > 1 && t.jn / 2 >= ocj) continue;  // a channel tile past every channel
            if (t.ksw && p.Kp / 64 < 4) continue;
            ConvChoice c;
            c.kind = 1;
            c.jn = t.jn;
            c.pw = t.pw;
            c.ksw = t.ksw ? 1 : 0;
            out[n++] = c;
        }
    }
    if (n < cap && int8 && p.KH == 1 && p.KW == 1) n += enumerate_s1x1_choices(p, int8, out + n, cap - n);
    if (n < cap && nchw && !int8) n += enumerate_stem_choices(p, out + n, cap - n);
    if (n < cap && !nchw) n += enumerate_m32_choices(p, int8, out + n, cap - n);
    if (n < cap && !nchw && !int8) n += enumerate_wide_choices(p, out + n, cap - n);
    if (n < cap) n += enumerate_halo_choices(p, int8, out + n, cap - n);
    return n;
}

namespace {

// ---- 3x3 convs without a measured tile ----------------------------------------
// Every tile that the three 3x3 kernels (halo window, 32x32 MFMA, implicit
// GEMM) offer for the conv is given an estimated time, and the fastest runs.
// The estimate weighs what a launch does on its most loaded CU (weight bytes
// staged, matrix-core and LDS-read clocks, conversion work, input bytes of all
// blocks) and the serial chain of one block (iterations, their MFMA clocks and
// staging rounds, position tiles).  In the halo and the plain implicit-GEMM
// kernel several blocks share a CU and cover each other's chains, so the longer
// of the two counts; the other two run them one after the other.
//
// The rates below are microseconds per unit, fitted (non-negative least
// squares) to 38800 measured launches: 642 random shapes (batch 1-64, maps
// 4-160, 8-512 channels, strides 1 and 2) with all of their tiles.  Over those
// shapes the chosen tile takes 1.02x (int8) and 1.03x (fp16) the time of the
// best one (the same on shapes left out of the fit).  The rule before it (halo
// tiles of 4 waves by a clock count, implicit GEMM only where no halo tile fits)
// took 1.15x: 4 waves leave a CU half empty where the weights fill the LDS, and
// it never took the 32x32-MFMA kernel.  Examples, us before and after: int8
// 64 -> 128 channels at 80x80 from 160x160 x32 81.8 -> 63.8, 256 at 40x40 x2 17.9
// -> 11.4, 512 at 20x20 38.7 -> 14.4; fp16 128 at 80x80 x4 29.5 -> 22.6, 256 -> 64
// at 20x20 x8 17.1 -> 10.8.
struct TileRates {
    double base;      // launch and first loads
    double weights;   // per 10 KB of weights staged on the CU
    double mfma;      // per 10k matrix-core clocks of the CU's blocks
    double lds;       // per 10k LDS-read clocks of the CU's blocks
    double convert;   // per 1k wave-rounds of conversion (16 bytes a lane) on a SIMD
    double bytes;     // per 100 MB of input read by all blocks
    double epilogue;  // per 100 position x channel subtiles stored by the CU
    double iter;      // per 10 iterations (barrier, latency) of a block
    double chain;     // per 10k matrix-core clocks in one block's chain
    double rounds;    // per 100 staging rounds in one block's chain
    double tile;      // per 10 position tiles of a block
    bool overlap;     // the CU's work and a block's chain cover each other
};
// halo, 32x32 MFMA, implicit GEMM, implicit GEMM with k split over the waves
constexpr TileRates kRatesI8[4] = {{3.85, 0.21, 0, 3.46, 96.18, 0.33, 12.66, 0.95, 5.92, 14.76, 0.72, true},
                                   {3.66, 0.18, 7.01, 0, 40.61, 5.25, 24.7, 0, 0.04, 14.18, 6.94, false},
                                   {4.94, 0.21, 0, 0, 22.61, 0.48, 11.36, 3.5, 12.36, 7.39, 0, true},
                                   {3.81, 0, 0, 0, 16.53, 2.53, 22.57, 2.16, 44.24, 0, 14.31, false}};
constexpr TileRates kRatesF16[4] = {{3.4, 0.19, 0, 4.42, 56.91, 0.04, 12.07, 0.32, 7.99, 12.56, 0, true},
                                    {3.47, 0.19, 8.64, 0, 0, 6.21, 36.97, 0, 0, 10.27, 0, false},
                                    {4.18, 0.17, 0.13, 0.69, 13.35, 1.73, 7.84, 2.34, 9.51, 6.35, 0, true},
                                    {3.25, 0, 0, 0, 15.52, 2.63, 23.49, 1.05, 41.36, 0, 14.9, false}};

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Estimated microseconds of a 3x3 conv with tile c (as an enumerate_* function gives it).
}  // namespace

double conv_tile_time(const ConvParams& p, bool int8, const ConvChoice& c) {
    constexpr int kCus = 256, kLds = 160 * 1024;
    const int esz = int8 ? 1 : 2, wq = int8 ? 1 : 2;
    // registers of the instance, as the compiler gives them within a few
    auto waves_per_simd = [](double regs) { return 512 / (((int)(std::min(regs, 504.0) + 0.5) + 7) / 8 * 8); };
    double wbytes, mfma, lds, convert, bytes, epilogue, iters, chain, rounds, tiles;
    int family;
    if (c.kind == 1) {
        family = c.ksw ? 3 : 2;
        const int nks = p.Kp / 64, kc = igemm::chunk_steps_of(int8, c.jn, c.ksw != 0);
        const bool mc = nks > kc;
        const int chunk = kc * c.jn * 16 * 64 * esz;
        const double regs = (int8 ? 48 : 40) + (mc ? 20 : 0) + (c.ksw ? 20 : 17) * c.pw + 3.5 * c.jn * (c.pw + 1);
        const int res = std::max(1, std::min(kLds / (chunk * (mc ? 2 : 1) + 8400), waves_per_simd(regs)));
        const int64_t npt = cdiv(p.M, (c.ksw ? 16 : 64) * c.pw), ntn = cdiv(p.OCp / 16, c.jn);
        int64_t groups = npt;
        if (!c.ksw && npt * ntn > (int64_t)res * kCus) groups = std::max<int64_t>(1, (int64_t)res * kCus / ntn);
        const double per = (double)cdiv(npt, groups);
        const double blocks = (double)cdiv(npt, (int64_t)per) * ntn;
        // a k-split grid may need several rounds of resident blocks
        const double load = c.ksw && blocks > (double)kCus * res ? blocks / kCus : std::ceil(blocks / kCus);
        const double turns = per * (c.ksw ? std::ceil(blocks / ((double)kCus * res)) : 1.0);
        const double step = c.jn * c.pw * wq * 16.0, split = c.ksw ? 1.0 : 4.0;
        wbytes = load * c.jn * 16.0 * nks * 64 * esz * (mc ? per : 1.0);
        mfma = load * per * nks * step / (c.ksw ? 4.0 : 1.0);
        lds = load * per * nks * c.jn * wq * 8.0 * split;
        convert = load * per * nks * c.pw * 2.0 * split;
        bytes = blocks * per * (c.ksw ? 16 : 64) * c.pw * nks * 128.0;
        epilogue = load * per * c.jn * c.pw;
        iters = turns * (c.ksw ? cdiv(nks, 4) : nks);
        chain = iters * step;
        rounds = iters * c.pw;
        tiles = turns;
    } else {
        const bool m = c.kind == 5;
        family = m ? 1 : 0;
        const int ir = (c.tr - 1) * p.S + 3, icol = (c.tc - 1) * p.S + 3, nch = p.C / c.cc;
        const int np = ir * icol * c.cc / (m && int8 ? 16 : 8) <= 4 * 64 * c.nw ? 4 : 8;
        const int64_t ntile = (int64_t)p.N * cdiv(p.OH, c.tr) * cdiv(p.OW, c.tc);
        const int jp = c.jn * c.pw;
        double wb, tb, regs, step;
        int64_t ntn;
        if (m) {
            const int64_t steps = cdiv(9 * c.cc, int8 ? 32 : 16);
            wb = (double)nch * steps * 2 * c.jn * 32 * 16;
            tb = (double)ir * icol * c.cc * esz;
            ntn = cdiv(p.OCp, 32 * c.jn);
            step = (double)steps * jp * 32;
            lds = (double)steps * (c.jn + c.pw) * 8;
            regs = int8 ? 23 + 18 * jp + 16.3 * c.jn + 13.6 * c.pw + 11.2 * np
                        : 13 + 15.5 * jp + 19 * c.jn + 16.5 * c.pw + 7 * np;
            epilogue = c.nw / 4.0;
        } else {
            const int64_t steps = cdiv(9 * c.cc, 64);
            wb = (double)nch * steps * wq * c.jn * 1024;
            const int px = c.cc * esz;
            tb = (double)ir * icol * (px + (px / 16 % 2 ? 0 : 16));
            ntn = cdiv(p.OCp / 16, c.jn);
            step = (double)steps * jp * wq * 16;
            lds = (double)steps * (c.jn + c.pw) * wq * 8;
            regs = int8 ? 23 + 6 * jp + 11 * c.jn + 11.5 * c.pw + 8 * np
                        : 40 + 19 * jp + 6.5 * c.jn + 11.6 * c.pw + 7 * np;
            epilogue = jp * c.nw / 4.0;
        }
        const int res = std::max(1, std::min(kLds / (int)(wb + 2 * tb + 2048), waves_per_simd(regs) * 4 / c.nw));
        int64_t groups = ntile;
        if (ntile * ntn > (int64_t)res * kCus) groups = std::max<int64_t>(1, (int64_t)res * kCus / ntn);
        tiles = (double)cdiv(ntile, groups);
        const double blocks = (double)cdiv(ntile, (int64_t)tiles) * ntn;
        const double load = std::ceil(blocks / kCus);
        iters = tiles * nch;
        chain = iters * step * c.nw / 4.0;
        wbytes = load * wb;
        mfma = load * chain;
        lds *= load * iters * c.nw;
        convert = load * iters * ((double)ir * icol * c.cc / 8) / 256;
        bytes = blocks * iters * ((double)ir * icol * c.cc) * 2.0;
        epilogue *= load * tiles;
        rounds = iters * np;
    }
    const TileRates& r = (int8 ? kRatesI8 : kRatesF16)[family];
    const double cu = r.mfma * mfma * 1e-4 + r.lds * lds * 1e-4 + r.convert * convert * 1e-3 + r.bytes * bytes * 1e-8;
    const double block = r.iter * iters * 0.1 + r.chain * chain * 1e-4 + r.rounds * rounds * 1e-2 + r.tile * tiles * 0.1;
    return r.base + r.weights * wbytes * 1e-4 + r.epilogue * epilogue * 1e-2 +
           (r.overlap ? std::max(cu, block) : cu + block);
}

namespace {

// Fastest estimated tile of a 3x3 conv; false (best as it was) where none applies.  With
// a tile forced on the implicit GEMM that kernel is not among them (it runs,
// with the forced tile, where no window kernel fits).
bool choose_conv3x3(const ConvParams& p, bool int8, ConvChoice& best) {
    if (p.KH != 3 || p.KW != 3 || p.P != 1 || p.loader != kLoaderNhwc || p.fuse_1x1 || p.yup || p.xup) return false;
    // the choice is a function of the sizes below alone: the last ones of this
    // thread are kept (enumerating the tiles takes as long as a small conv)
    struct Entry {
        int key[10];
        ConvChoice best;
        bool found;
    };
    constexpr int kEntries = 64;
    static thread_local Entry memo[kEntries] = {};  // a zeroed key has N = 0: no conv's
    const int key[10] = {p.N, p.C, p.H, p.W, p.OC, p.OH, p.OW, p.S, p.Kp, (int)int8 | (tile_forced() ? 2 : 0) |
                         (p.x_cstride % 8 ? 4 : 0)};
    uint32_t h = 2166136261u;
    for (int v : key) h = (h ^ (uint32_t)v) * 16777619u;
    Entry& e = memo[(h ^ (h >> 16)) % kEntries];
    if (std::memcmp(e.key, key, sizeof(key)) != 0) {
        ConvChoice all[kMaxConvChoices];
        const int n = enumerate_conv_choices(p, int8, all, kMaxConvChoices);
        const ConvTile usual_tile = choose_conv_tile(p.M, p.OC, p.Kp);
        double best_t = 0.0;
        e.found = false;
        for (int i = 0; i < n; ++i) {
            const ConvChoice& c = all[i];
            if (c.kind != 1 && c.kind != 2 && c.kind != 5) continue;
            if (c.kind == 1) {
                // fp16: the estimate orders the plain implicit-GEMM tiles of large maps
                // wrongly (up to 1.4x), choose_conv_tile does not
                const bool usual = c.jn == usual_tile.jn && c.pw == usual_tile.pw && (c.ksw != 0) == usual_tile.ksw;
                if (tile_forced() || (int8 ? c.pw > 2 : !c.ksw && !usual)) continue;
            } else if (c.pw > 2 || (c.kind == 2 && c.jn > 4)) {
                continue;  // halo tiles of 5 channel subtiles with 2 position subtiles use scratch memory
            }
            // 32x32 MFMA: the widest tiles and the two-group blocks were the fastest at
            // a handful of shapes only, 8 waves of 4 subtiles lose up to 1.4x to others
            if (c.kind == 5 && (c.jn > 3 || c.ksw || (c.nw == 8 && c.jn * c.pw >= 4))) continue;
            const double t = conv_tile_time(p, int8, c);
            if (!e.found || t < best_t) {
                best_t = t;
                e.best = c;
                e.found = true;
            }
        }
        std::memcpy(e.key, key, sizeof(key));
    }
    if (e.found) best = e.best;
    return e.found;
}

}  // namespace

hipError_t launch_conv_igemm(const ConvParams& p0, bool int8, hipStream_t stream) {
    const bool nchw = p0.loader == kLoaderNchwF32;
    if ((p0.loader != kLoaderNhwc && !nchw) || p0.OC % 4 || p0.C % 8 || p0.Kp % 64 || p0.OCp % 16)
        return hipErrorInvalidValue;
    if (nchw && (int8 || p0.c_real < 1 || p0.c_real > 4 || p0.x_nstride != (int64_t)p0.c_real * p0.H * p0.W))
        return hipErrorInvalidValue;
    const bool out_f32 = (p0.flags & kConvOutF32) != 0;
    const int HWi = p0.H * p0.W, HWo = p0.OH * p0.OW;
    // Images per launch: every view a launch touches must stay inside
    // kMaxViewBytes so the kernel can address it with 32-bit offsets.
    const uint64_t x_img = nchw ? (uint64_t)p0.x_nstride * 4
                                : std::max((uint64_t)p0.x_nstride * 2, (uint64_t)HWi * p0.x_cstride * 2);
    const uint64_t per_img = std::max({x_img, (uint64_t)p0.y_nstride * (out_f32 ? 4 : 2),
                                       p0.res ? (uint64_t)p0.r_nstride * 2 : 0,
                                       p0.acc_out ? (uint64_t)HWo * p0.OC * 4 : 0,
                                       p0.fuse_1x1 ? (uint64_t)p0.fuse_1x1->y_nstride *
                                                         ((p0.fuse_1x1->flags & kConvOutF32) ? 4 : 2)
                                                   : 0,
                                       p0.yup ? (uint64_t)p0.yup_nstride * 2 : 0,
                                       p0.xup ? (uint64_t)p0.xup_nstride * 2 : 0});
    if ((uint64_t)p0.OCp * p0.Kp * 2 > kMaxViewBytes || per_img == 0) return hipErrorInvalidValue;
    const int per_launch = (int)std::min<uint64_t>((uint64_t)p0.N, kMaxViewBytes / per_img);
    if (per_launch < 1) return hipErrorInvalidValue;
    const int nks = p0.Kp / 64;
    if (nks > igemm::kMaxSteps) return hipErrorInvalidValue;
    if (int8 && (p0.x_slots.p == nullptr ||
                 (int64_t)p0.x_slots.stripes * p0.x_nslots > igemm::kMaxSlotReads))
        return hipErrorInvalidValue;
    // no measured tile and none forced: a 3x3 conv's by its estimated times
    ConvChoice choice = p0.choice;
    ConvChoice forced_tile;
    if (choice.kind == 0 && halo_mode_auto() && !forced_m32_choice(forced_tile) &&
        (int8 || !forced_wide_choice(forced_tile))) {
        ConvParams slice = p0;
        slice.N = std::min(per_launch, p0.N);
        slice.M = slice.N * HWo;
        choose_conv3x3(slice, int8, choice);
    }
    const ConvTile t = choice.kind == 1 ? ConvTile{choice.jn, choice.pw, choice.ksw != 0}
                       : !int8 && p0.KH == 1 && p0.KW == 1 ? choose_f16_1x1_tile(p0.M, p0.OC, p0.Kp)
                                                           : choose_conv_tile(p0.M, p0.OC, p0.Kp);
    if (choice.kind == 1 && !tile_instantiated(t)) return hipErrorInvalidValue;
    const bool mc = nks > igemm::chunk_steps_of(int8, t.jn, t.ksw);
    const int f = p0.flags & (kConvSilu | kConvResidual | kConvOutF32);
    // the int32 accumulator output (acc_out) is written by the run-time
    // flag variant only
    const int epi = p0.acc_out ? igemm::kEpiAny
                    : f == kConvSilu ? igemm::kEpiSilu
                    : (int8 && f == (kConvSilu | kConvResidual) ? igemm::kEpiSiluRes : igemm::kEpiAny);
    if (p0.fuse_1x1 && (p0.choice.kind != 5 || int8)) return hipErrorInvalidValue;
    // the upsample copy: a streaming 1x1 choice (measured, or forced)
    ConvChoice forced_up;
    if ((p0.yup || p0.xup) &&
        !(int8 && (p0.choice.kind == 6 || (p0.choice.kind == 0 && forced_s1x1_choice(forced_up)))))
        return hipErrorInvalidValue;
    for (int nb = 0; nb < p0.N; nb += per_launch) {
        ConvParams p = p0;
        p.choice = choice;
        ConvParams f2;  // the fused 1x1 on this slice of the batch
        if (p0.fuse_1x1) {
            f2 = *p0.fuse_1x1;
            f2.N = std::min(per_launch, p0.N - nb);
            f2.M = f2.N * HWo;
            const int esz2 = (f2.flags & kConvOutF32) ? 4 : 2;
            f2.y = static_cast<char*>(f2.y) + (int64_t)nb * f2.y_nstride * esz2;
            f2.y_bytes = (uint32_t)view_span(f2.N, f2.y_nstride, f2.y_cstride, HWo, f2.OC, esz2);
            if ((uint64_t)f2.OCp * f2.Kp * 2 > kMaxViewBytes || (uint64_t)f2.y_nstride * esz2 > kMaxViewBytes)
                return hipErrorInvalidValue;
            p.fuse_1x1 = &f2;
        }
        p.N = std::min(per_launch, p0.N - nb);
        p.M = p.N * HWo;
        p.x = nchw ? static_cast<const void*>(static_cast<const float*>(p0.x) + (int64_t)nb * p0.x_nstride)
                   : static_cast<const void*>(static_cast<const __half*>(p0.x) + (int64_t)nb * p0.x_nstride);
        p.y = static_cast<char*>(p0.y) + (int64_t)nb * p0.y_nstride * (out_f32 ? 4 : 2);
        if (p0.res) p.res = p0.res + (int64_t)nb * p0.r_nstride;
        if (p0.acc_out) p.acc_out = p0.acc_out + (int64_t)nb * HWo * p0.OC;
        if (p0.yup) {
            p.yup = static_cast<__half*>(p0.yup) + (int64_t)nb * p0.yup_nstride;
            p.yup_bytes = (uint32_t)view_span(p.N, p.yup_nstride, p.yup_cstride, 4 * HWo, p.OC, 2);
        }
        if (p0.xup) {
            p.xup = static_cast<const __half*>(p0.xup) + (int64_t)nb * p0.xup_nstride;
            p.xup_bytes = (uint32_t)view_span(p.N, p.xup_nstride, p.xup_cstride, HWi / 4, p.xup_cn, 2);
        }
        p.x_bytes = nchw ? (uint32_t)((uint64_t)p.N * p.x_nstride * 4)
                         : (uint32_t)view_span(p.N, p.x_nstride, p.x_cstride, HWi, p.C, 2);
        p.y_bytes = (uint32_t)view_span(p.N, p.y_nstride, p.y_cstride, HWo, p.OC, out_f32 ? 4 : 2);
        p.r_bytes = p.res ? (uint32_t)view_span(p.N, p.r_nstride, p.r_cstride, HWo, p.OC, 2) : 0u;
        p.ntn = (p.OCp / 16 + t.jn - 1) / t.jn;
        const int mtile = (t.ksw ? 16 : 64) * t.pw;
        p.npt = (p.M + mtile - 1) / mtile;
        p.fd_ntn = make_fastdiv((uint32_t)p.ntn);
        if (int8) {
            p.x_slot_bytes = ((p.x_slots.stripes - 1) * p.x_slots.stride + (uint32_t)p.x_nslots) * 4u;
            p.fd_ns = make_fastdiv((uint32_t)std::max(p.x_nslots, 1));
        }
        p.lin = 0;
        if (p.M < (1 << 24)) {
            if (!nchw && p.KH == 1 && p.KW == 1 && p.S == 1 && p.P == 0 && p.x_nstride == (int64_t)HWi * p.x_cstride &&
                p.x_cstride < (1 << 24))
                p.lin |= kLinX;
            if (p.y_nstride == (int64_t)HWo * p.y_cstride && p.y_cstride < (1 << 24) &&
                (!p.res || (p.r_nstride == (int64_t)HWo * p.r_cstride && p.r_cstride < (1 << 24))))
                p.lin |= kLinY;
        }
        p.fd_ohw = make_fastdiv((uint32_t)HWo);
        p.fd_ow = make_fastdiv((uint32_t)p.OW);
        p.fd_c = make_fastdiv((uint32_t)p.C);
        p.fd_kw = make_fastdiv((uint32_t)p.KW);
        hipError_t e = hipErrorNotSupported;
        if (p.choice.kind == 0 && int8 && p.KH == 1 && p.KW == 1) {
            ConvChoice forced;
            if (forced_s1x1_choice(forced)) {
                p.choice = forced;  // a forced tile that does not fit is an error
                e = launch_conv_s1x1(p, int8, epi, stream);
                if (e != hipSuccess) return e;
                continue;
            }
            // no tile forced on the implicit GEMM either: the streaming kernel by its rule
            if (!tile_forced() && choose_s1x1(p, int8, p.choice)) {
                e = launch_conv_s1x1(p, int8, epi, stream);
                if (e != hipSuccess) return e;
                continue;
            }
        }
        if (p.choice.kind == 6) {
            e = launch_conv_s1x1(p, int8, epi, stream);
            if (e != hipSuccess) return e;
            continue;
        }
        if (p.choice.kind == 0 && !nchw) {
            ConvChoice forced;
            if (forced_m32_choice(forced) && p.KH == 3 && p.KW == 3) {
                p.choice = forced;  // a forced tile that does not fit is an error
                e = launch_conv_m32(p, int8, epi, stream);
                if (e != hipSuccess) return e;
                continue;
            }
        }
        if (p.choice.kind == 5) {
            e = launch_conv_m32(p, int8, epi, stream);
            if (e != hipSuccess) return e;
            continue;
        }
        if (p.choice.kind == 0 && !int8 && !nchw) {
            ConvChoice forced;
            if (forced_wide_choice(forced)) {
                p.choice = forced;  // a forced wide tile that does not fit is an error
                e = launch_conv_wide(p, epi, stream);
                if (e != hipSuccess) return e;
                continue;
            }
        }
        if (p.choice.kind == 4) {
            e = launch_conv_wide(p, epi, stream);
            if (e != hipSuccess) return e;
            continue;
        }
        if (nchw && !int8 && (p.choice.kind == 0 || p.choice.kind == 3)) e = launch_conv_stem(p, stream);
        if (e == hipErrorNotSupported && p.choice.kind != 1 && p.choice.kind != 3)
            e = launch_conv_halo(p, int8, epi, stream);
        if (e == hipErrorNotSupported && !nchw && p.choice.kind != 2) e = launch_variant(int8, mc, epi, p, t, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace aexrt
