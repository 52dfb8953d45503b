// Launch geometry, weight packing and the closed-form gfx950 tile model.
//
// The reference chooses (TH, TW, TC) per layer either from a measured sweep
// (2080Ti-evaluation/TDC-LAYERS-ORACLE/gen_from_occupancy.py:51-66) or from an
// analytic score that still needs a table of measured CUDA occupancies
// (2080Ti-evaluation/TDC-LAYERS-MODELING/model.py:136-156,209-235;
// 2080Ti-evaluation/Gen-occupancy/template.cu:277-284).  This file is the
// self-contained counterpart for one MI355X: occupancy comes from the register
// and LDS footprint of the tile, latency from MFMA issue cycles per SIMD, the
// copy volume of the staged input window and weights, and wave quantisation over
// 256 compute units.  Host-only code: it runs without a GPU.
#include <algorithm>
#include <array>
#include <map>
#include <mutex>
#include <shared_mutex>
#include <unordered_map>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "tdc_internal.hpp"

namespace tdc {

const Machine &machine() {
    static const Machine m;
    return m;
}

static inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
static inline int round_up(int a, int b) { return ceil_div(a, b) * b; }

bool check_desc(const tdc_conv_desc &d, std::string *why) {
    auto fail = [&](const char *m) {
        if (why) *why = m;
        return false;
    };
    if (d.batch < 1 || d.C < 1 || d.N < 1 || d.H < 1 || d.W < 1) return fail("batch, C, N, H, W must be >= 1");
    if (d.KH < 1 || d.KW < 1) return fail("KH, KW must be >= 1");
    if (d.stride < 1) return fail("stride must be >= 1");
    if (d.pad < 0) return fail("pad must be >= 0");
    if (d.dilation < 1) return fail("dilation must be >= 1");
    const long long eh = (long long)d.H + 2LL * d.pad - (long long)d.dilation * (d.KH - 1) - 1;
    const long long ew = (long long)d.W + 2LL * d.pad - (long long)d.dilation * (d.KW - 1) - 1;
    if (eh < 0 || ew < 0) return fail("filter (with dilation) larger than padded input");
    // One image is addressed through a 32-bit buffer descriptor (byte offsets below 2^31).
    if ((long long)d.C * d.H * d.W >= (1LL << 29) || (long long)d.N * d.H * d.W >= (1LL << 29))
        return fail("per-image tensor exceeds 2^29 elements");
    if ((long long)d.N * d.C * d.KH * d.KW >= (1LL << 28)) return fail("weight tensor exceeds 2^28 elements");
    return true;
}

// LDS bank conflicts of the B-operand read.  The 64 lanes of a wave read one word each: lane l holds pixel
// l % mf of its block and input channel l / mf of the K-step, i.e. word jy*stride*RS + jx*stride + (l/mf)*CS
// (+ the same tap offset for everybody).  The LDS has 64 four-byte banks; lanes that hit one bank with
// different words are served one after the other.  Returned: that serialisation factor (1 = conflict-free),
// averaged over the pixel blocks of a workgroup tile.
static double b_read_conflict_ways(int mf, int PT, int TW, int TH, int RS, int CS, int stride) {
    double sum = 0.0;
    int blocks = 0;
    for (int j0 = 0; j0 < PT; j0 += mf, ++blocks) {
        int words[64][8], cnt[64];
        for (int b = 0; b < 64; ++b) cnt[b] = 0;
        int ways = 1;
        for (int l = 0; l < 64; ++l) {
            const int j = j0 + l % mf;
            const int jy = std::min(j / TW, TH - 1), jx = j % TW;
            const int w = jy * stride * RS + jx * stride + (l / mf) * CS;
            const int b = w & 63;
            bool seen = false;
            for (int i = 0; i < cnt[b]; ++i) seen |= (words[b][i] == w);
            if (!seen && cnt[b] < 8) words[b][cnt[b]++] = w;
            ways = std::max(ways, cnt[b]);
        }
        sum += ways;
    }
    return blocks ? sum / blocks : 1.0;
}

// LDS channel stride: the smallest stride from the raw window size upwards (inflating small windows by at
// most a quarter, larger ones by at most 64 words) that gives the B-operand read the fewest bank conflicts.
// For tiles whose pixel blocks lie in one row this is the classic rule — stride = 16 (mod 32) for the four
// channel quarters of a 16x16x4 step, 32 (mod 64) for the halves of a 32x32x2 step; narrow tiles whose
// blocks wrap over several rows cannot be made conflict-free and get the best stride there is.
static int pad_channel_stride(int raw, int mf, int vw, int PT, int TW, int TH, int RS, int stride, double *ways_out) {
    // Thousands of candidate tiles share a handful of window shapes: remember the answers (per thread).
    static thread_local std::map<std::array<int, 8>, std::pair<int, double>> memo;
    const std::array<int, 8> key{raw, mf, vw, PT, TW, TH, RS, stride};
    auto hit = memo.find(key);
    if (hit == memo.end()) {
        const int first = round_up(raw, vw);
        const int budget = std::max(raw / 4, std::min(64, raw));
        int best = first;
        double best_ways = 1e9;
        for (int cs = first; cs - raw <= budget; cs += vw) {
            const double ways = b_read_conflict_ways(mf, PT, TW, TH, RS, cs, stride);
            if (ways < best_ways - 1e-9) {
                best_ways = ways;
                best = cs;
            }
        }
        if (memo.size() > 100000) memo.clear();
        hit = memo.emplace(key, std::make_pair(best, best_ways)).first;
    }
    *ways_out = hit->second.second;
    return hit->second.first;
}

// Which logical workgroup order costs fewer L2 fills.  Bytes the eight die-private L2s fill in total, for the two orders: with
// the channel tiles of a pixel tile adjacent a die reads its share of the input and every weight; with the pixel tiles of a
// channel tile adjacent it reads every input pixel of min(channel tiles, 8) ... and its own weights.
static int channel_major_order(double in_bytes, double w_bytes, long long n_wg, int grid_y) {
    const double dies = (double)std::min<long long>(8, n_wg);
    const double pixel_major = in_bytes + dies * w_bytes;
    const double channel_major = std::min<double>(grid_y, dies) * in_bytes + std::max(1.0, dies / grid_y) * w_bytes;
    if (const char *e = std::getenv("TDC_EXPERIMENT_XCD_ORDER")) return std::atoi(e) != 0;
    return channel_major < pixel_major ? 1 : 0;
}

// tile.alg = 8: fp32 operands as three bf16 parts each (conv_split.hip, conv_core_split.hip).
static bool make_split_geometry(const tdc_conv_desc &d, const tdc_tile &t, Geometry &g, std::string *why, int tail_N) {
    auto fail = [&](const char *m) {
        if (why) *why = m;
        return false;
    };
    const bool flat = t.tw == 0, few = t.cch == 4, one = d.KH == 1 && d.KW == 1;
    const bool core = !flat && t.nb == 2;       // (conv_core_split.hip)
    if (t.mf != 16 || (t.nb != 4 && t.nb != 2) || (core && few) || (t.mb != 1 && t.mb != 2 && t.mb != 4))
        return fail("tile.alg = 8 needs mf = 16, mb = 1, 2 or 4, nb = 2 or 4 (4 with cch = 4)");
    if (t.wm < 1 || t.wn < 1 || t.wk < 1 || (long long)t.wm * t.wn * t.wk > 8) return fail("tile.alg = 8 needs 1 to 8 waves");
    if ((t.wk != 1 && !flat && !core) || t.ks != 1 || t.wl != 0)
        return fail("tile.alg = 8 has no split across workgroups and no loader waves, and splits input channels over waves only with tw = 0 or nb = 2");
    if (tail_N > 0) return fail("tile.alg = 8 cannot carry a fused tail");
    g = Geometry();
    g.Ho = (d.H + 2 * d.pad - d.dilation * (d.KH - 1) - 1) / d.stride + 1;
    g.Wo = (d.W + 2 * d.pad - d.dilation * (d.KW - 1) - 1) / d.stride + 1;
    g.P = g.Ho * g.Wo;
    g.He = d.H;
    g.We = d.W;
    g.kc = 32;
    g.taps = g.ktaps = d.KH * d.KW;
    g.max_waves_kernel = 8;
    g.waves = t.wm * t.wn * t.wk;
    g.threads = 64 * g.waves;
    g.MT = 16 * t.mb * t.wm;
    g.PT = 16 * t.nb * t.wn;
    g.cpw = t.cch / t.wk;
    g.nchunks = ceil_div(d.C, t.cch);
    g.cps = g.nchunks;
    g.c_pad = g.nchunks * t.cch;
    long long lds, units;
    int cols = 1;
    if (flat) {
        if (!one || d.stride != 1 || d.pad != 0) return fail("tile.alg = 8 with tw = 0 needs a 1x1 / stride 1 / pad 0 convolution");
        if (g.P < t.nb) return fail("tile.alg = 8 with tw = 0 needs images of at least nb pixels");
        const int kw = t.wm * t.wk;             // K-steps of a stage: every thread of the workgroup loads one octet
        if (kw != 1 && kw != 2 && kw != 4 && kw != 8) return fail("tile.alg = 8 with tw = 0 needs wm * wk = 1, 2, 4 or 8");
        if (t.mb > 2) return fail("tile.alg = 8 with tw = 0 needs mb = 1 or 2");
        if (4 * t.mb % t.wk != 0) return fail("tile.alg = 8: more channel slices than rows to finish");
        if (t.cch != 32 * kw) return fail("tile.alg = 8 with tw = 0 needs cch = 32 * wm * wk");
        g.units_image = ceil_div(g.P, t.nb);
        units = (long long)d.batch * g.units_image;
        g.units_wg = 16 * t.wn;
        g.unit_images = std::min(d.batch - 1, (g.units_wg - 2) / g.units_image + 1);
        g.TW = std::min(g.PT, g.P);
        g.TH = 1;
        while ((1 << g.oct_shift) < 4 * kw) ++g.oct_shift;
        g.ksteps = kw;
        g.RS = 1;
        g.CS = g.PT;
        g.win_L = 1;
        lds = std::max(3LL * (4 * kw) * g.CS * 16, 1024LL * g.waves * t.mb * t.nb);   // the staged octets, or the sums of all waves
    } else {
        if (few) {
            if (d.C > 4 || d.dilation != 1 || d.stride % 2 != 0)
                return fail("tile.alg = 8 with cch = 4 needs at most four input channels, an even stride and dilation 1");
        } else if (t.cch != 8 && t.cch != 16 && t.cch != 32 && !(core && (t.cch == 64 || t.cch == 128))) {
            return fail("tile.alg = 8 needs cch = 8, 16 or 32, with nb = 2 also 64 or 128 (4: at most four input channels)");
        }
        if (one) return fail("tile.alg = 8 takes 1x1 convolutions with tw = 0 only");
        if (t.tw < 1 || t.tw > g.PT || t.tw > g.Wo) return fail("tile.alg = 8: tile.tw does not fit");
        units = (long long)d.batch * g.Ho;
        g.TW = t.tw;
        g.TH = (int)std::min<long long>(g.PT / t.tw, units);
        g.units_image = g.Ho;
        g.units_wg = g.TH;
        while ((8 << g.oct_shift) < t.cch) ++g.oct_shift;
        g.row_taps = few ? ceil_div(d.KW, 2) : d.KW;
        g.ksteps = few ? ceil_div(d.KH * g.row_taps, 4) : ceil_div(g.taps << g.oct_shift, 4);
        if (g.ksteps % t.wk != 0) return fail("tile.alg = 8: wk does not divide the K-steps of a stage");
        const long long columns = (long long)(g.TW - 1) * d.stride + (few ? 2 * g.row_taps : (d.KW - 1) * d.dilation + 1);
        const long long image_rows = (long long)(g.Ho - 1) * d.stride + (long long)(d.KH - 1) * d.dilation + 1;
        // the most window rows any tile of output rows needs (the tiles repeat their place in the images after Ho of them)
        long long rows = 0;
        const long long tiles = (units + g.TH - 1) / g.TH;
        for (long long i = 0; i < std::min<long long>(tiles, g.Ho); ++i) {
            const long long a = i * g.TH, b = std::min(a + g.TH, units) - 1;
            rows = std::max(rows, (b / g.Ho - a / g.Ho) * image_rows + (b % g.Ho - a % g.Ho) * d.stride + (long long)(d.KH - 1) * d.dilation + 1);
            g.unit_images = std::max(g.unit_images, (int)(b / g.Ho - a / g.Ho));
        }
        g.unit_images = std::min(d.batch - 1, g.unit_images + 1);   // (the last rows of a window may lie in an image that no output needs)
        if (columns > 8192 || rows > 8192 || rows * columns > 65536 || image_rows + rows > 65535) return fail("tile.alg = 8: input window too large");
        g.ncols = (int)columns;
        g.nrows = (int)rows;
        g.win_L = (int)image_rows;
        g.odd_columns = (g.ncols + 1) / 2;
        g.RS = !few && d.stride == 2 ? 2 * g.odd_columns : g.ncols;
        g.CS = g.nrows * g.RS;
        // (whole rounds of the LDS banks from octet to octet, where they fit)
        if (core && ((48LL * round_up(g.CS, 16)) << g.oct_shift) + 32 <= machine().lds_bytes_per_cu) g.CS = round_up(g.CS, 16);
        lds = few ? 3LL * g.CS * 8 : std::max((48LL * g.CS) << g.oct_shift, t.wk > 1 ? 1024LL * g.waves * t.mb * t.nb : 0LL);   // (the sums of all waves)
        cols = ceil_div(g.Wo, g.TW);
    }
    if (units * std::max(g.units_image, 16) >= (1LL << 32) || units >= (1LL << 30)) return fail("batch too large for tile.alg = 8");
    if ((long long)d.H * d.W * (g.c_pad + 8) * 4 >= (1LL << 31)) return fail("image too large for tile.alg = 8");
    lds += 32;   // a word per wave in front, for what it met among the inputs
    if (lds > machine().lds_bytes_per_cu) return fail("tile needs more than 160 KiB of LDS");
    g.units = (int)units;
    g.lds_bytes = (int)lds;
    g.ntx = cols;
    g.nty = (int)((units + g.units_wg - 1) / g.units_wg);
    g.grid_y = ceil_div(d.N, g.MT);
    g.grid_z = 1;
    const long long gx = (long long)g.ntx * g.nty, n_wg = gx * g.grid_y;
    if (gx * g.ntx >= (1LL << 32) || n_wg + 8 >= (1LL << 28) || n_wg * std::max<long long>(gx, g.grid_y) >= (1LL << 32) || g.grid_y > 65535)
        return fail("grid too large");
    g.grid_x = (int)gx;
    g.wslab_floats = t.wm * t.mb * g.ksteps * 3 * 256;
    g.scale_floats = 4 + g.grid_y * g.MT;
    g.raw_floats = (size_t)d.N * d.C * g.taps;
    if ((long long)(packed_part_floats(g) + g.scale_floats) * 4 >= (1LL << 31)) return fail("packed weights exceed 2 GiB");
    g.channel_major = channel_major_order(4.0 * d.batch * d.C * d.H * d.W, 6.0 * d.N * d.C * g.taps, n_wg, g.grid_y);
    return true;
}

bool make_geometry(const tdc_conv_desc &d, const tdc_tile &t, Geometry &g, std::string *why, int tail_N) {
    auto fail = [&](const std::string &m) {
        if (why) *why = m;
        return false;
    };
    if (!check_desc(d, why)) return false;
    if (t.alg == 8) return make_split_geometry(d, t, g, why, tail_N);
    if (t.mf != 32 && t.mf != 16) return fail("tile.mf must be 16 or 32");
    if (t.mb < 1 || t.mb > 2 || t.nb < 1 ||
        (t.nb > 2 && !((t.alg == 4 || t.alg == 6 || t.alg == 7) && t.nb == 4)))
        return fail("tile.mb / tile.nb must be 1 or 2 (tile.nb may be 4 for tile.alg = 4, 6 and 7)");
    if (t.wm < 1 || t.wn < 1 || t.wk < 1) return fail("tile.wm / wn / wk must be >= 1");
    g = Geometry();
    // (256 registers per lane for the 2x2 block grid, 168 for the Winograd path)
    g.max_waves_kernel = (t.mb == 2 && t.nb == 2) ? 8 : t.alg == 1 ? 12 : 16;
    if (t.alg == 5) {
        // streamed Winograd: the launch bound follows the groups of four channels a wave keeps in registers
        const int groups = (t.wk >= 1 && t.cch % (4 * t.wk) == 0) ? t.cch / (4 * t.wk) : 0;
        g.max_waves_kernel = wino_stream_max_waves(groups);
        if (!g.max_waves_kernel) return fail("tile.alg = 5 needs cch = 4 * wk * {1, 2, 3, 4}");
    }
    if (t.alg == 7 || (t.alg == 1 && t.tw == 0)) g.max_waves_kernel = 8;
    if (t.wl < 0 || t.wl > 8) return fail("tile.wl must be in [0, 8]");
    if ((long long)t.wm * t.wn * t.wk + t.wl > g.max_waves_kernel) return fail("too many waves per workgroup for this tile");
    g.waves = t.wm * t.wn * t.wk + t.wl;
    g.threads = g.waves * 64;
    const bool flat = (d.KH == 1 && d.KW == 1 && d.stride == 1 && d.pad == 0);
    g.He = flat ? 1 : d.H;
    g.We = flat ? d.H * d.W : d.W;
    // (the copy-offset arithmetic of the kernel uses 24-bit multiplies)
    if ((long long)(d.C + 1) * g.He >= (1LL << 24) || g.We >= (1 << 24)) return fail("image too large");
    g.Ho = (g.He + 2 * d.pad - d.dilation * (d.KH - 1) - 1) / d.stride + 1;
    g.Wo = (g.We + 2 * d.pad - d.dilation * (d.KW - 1) - 1) / d.stride + 1;
    g.P = g.Ho * g.Wo;
    g.kc = (t.mf == 32) ? 2 : 4;
    g.taps = d.KH * d.KW;
    g.ktaps = g.taps;
    g.MT = t.mf * t.mb * t.wm;
    if (t.alg < 0 || t.alg > 7) return fail("tile.alg must be in [0, 8]");
    if (t.alg == 5) {
        // Winograd F(2x2,3x3) streamed from global memory: 16*wm channels of one tile row block (2 rows x 28 columns) per
        // workgroup, the input channels split over wk waves in groups of four, everything in one pass
        if (d.KH != 3 || d.KW != 3 || d.stride != 1 || d.dilation != 1 || d.pad != 1)
            return fail("tile.alg = 5 needs a 3x3 / stride 1 / pad 1 / dilation 1 convolution");
        if (d.W % 2 != 0) return fail("tile.alg = 5 needs an even image width");
        if (t.mf != 16 || t.mb != 1 || t.nb != 1 || t.wn != 1) return fail("tile.alg = 5 needs mf = 16, mb = nb = wn = 1");
        if (t.wl != 0 || t.ks != 1) return fail("tile.alg = 5 has no loader waves and no split across workgroups");
        if (tail_N > 0) return fail("tile.alg = 5 cannot carry a fused tail");
        if (t.tw != 28) return fail("tile.alg = 5 needs tw = 28");
        if (t.cch < d.C || t.cch - d.C >= t.cch / t.wk) return fail("tile.alg = 5 takes all input channels in one pass without an idle wave");
        if ((long long)t.cch * d.H * d.W * 4 >= (1LL << 31)) return fail("image too large for tile.alg = 5");
    }
    if (t.alg == 6 && (d.pad > 1 || d.stride > 2)) return fail("tile.alg = 6 needs pad <= 1 and stride <= 2");
    if (t.alg == 6 && t.nb == 4 && t.cch / std::max(t.wk, 1) > 8) return fail("tile.alg = 6 with nb = 4 takes at most two groups per wave");
    if (t.alg == 4 || t.alg == 6) {
        // 3x3 convolution streamed from global memory: 16 channels x 16 pixels per workgroup, the input channels
        // split over wk waves in groups of four, everything in one pass (alg 6: the tile's input window through LDS)
        if (d.KH != 3 || d.KW != 3 || d.dilation != 1) return fail("tile.alg = 4 needs a 3x3 / dilation 1 convolution");
        if (t.mf != 16 || t.mb != 1 || t.wn != 1) return fail("tile.alg = 4 needs mf = 16, mb = 1, wn = 1");
        if (t.nb != 1) {
            // nb pixel blocks per wave (the weights a wave holds feed nb MFMAs each): rows of 14 pixels, stride 1
            if (d.stride != 1 || t.tw != 14) return fail("tile.alg = 4 with nb > 1 needs stride 1 and tw = 14");
            if (t.nb > ceil_div(g.Wo, 14)) return fail("tile.alg = 4: more pixel blocks per wave than an image row has 14-pixel tiles");
            if (tail_N > 0 || t.ks != 1) return fail("tile.alg = 4 with nb > 1 has no fused tail and no split across workgroups");
        }
        if (t.wm * t.wk > 16) return fail("tile.alg = 4: at most 16 waves (wm channel blocks x wk channel slices)");
        if (t.wl != 0) return fail("tile.alg = 4 has no loader waves");
        const int groups = (t.cch % (4 * t.wk) == 0) ? t.cch / (4 * t.wk) : 0;
        if (groups != 1 && groups != 2 && groups != 4) return fail("tile.alg = 4 needs cch = 4 * wk * {1, 2, 4}");
        if (ceil_div(d.C, t.cch) != t.ks) return fail("tile.alg = 4 takes its input channels in one pass: ks slices of cch channels must cover them exactly");
        if ((long long)t.cch * d.H * d.W * 4 >= (1LL << 31)) return fail("image too large for tile.alg = 4");
    }
    const bool wino_batch = t.alg == 1 && t.tw == 0;
    g.wino = t.alg == 1;
    if (wino_batch) {
        // Winograd over the 2x2 tiles of the whole batch: 16*mb channels x 16*wn tiles per workgroup, wk teams of wn waves
        // split the input channels, two groups of four channels per step
        if (d.KH != 3 || d.KW != 3 || d.stride != 1 || d.dilation != 1 || d.pad > 1)
            return fail("tile.alg = 1 with tw = 0 needs a 3x3 / stride 1 / dilation 1 / pad <= 1 convolution");
        if (t.mf != 16 || t.wm != 1 || (t.wn != 2 && t.wn != 4))
            return fail("tile.alg = 1 with tw = 0 needs mf = 16, wm = 1, wn = 2 or 4");
        if (t.nb == 2 && t.mb == 2 && t.wn == 2) return fail("tile.alg = 1 with tw = 0: no sums in parts with mb = wn = 2");
        if (t.wl != 0 || t.ks != 1) return fail("tile.alg = 1 with tw = 0 has no loader waves and no split across workgroups");
        if (tail_N > 0) return fail("tile.alg = 1 cannot carry a fused tail");
        if (t.wk > 4 * t.mb) return fail("tile.alg = 1 with tw = 0: more teams than rows to finish");
        const int granule = 8 * t.wk;
        if (t.cch % granule != 0 || t.cch < d.C || t.cch - d.C >= granule)
            return fail("tile.alg = 1 with tw = 0 takes all input channels: cch = C rounded up to 8 * wk");
        g.ktaps = 16;
        g.TWt = ceil_div(g.Wo, 2);
        g.THt = ceil_div(g.Ho, 2);
        g.units_image = g.TWt * g.THt;
        const long long units = (long long)d.batch * g.units_image;
        if (units * g.units_image >= (1LL << 32) || units >= (1LL << 30)) return fail("batch too large for tile.alg = 1 with tw = 0");
        if (d.H * d.W < 8) return fail("tile.alg = 1 with tw = 0 needs images of at least 8 pixels");
        g.units = (int)units;
        g.raw_floats = (size_t)d.N * d.C * 9;
        g.unit_images = std::min(d.batch - 1, 14 / g.units_image + 1);
        g.TW = 2 * std::min(g.TWt, 16 * t.wn);
        g.TH = 2;
        g.PT = 64 * t.wn;
    }
    if (t.alg == 3) {
        // 1x1 convolution streamed from global memory: a 16x16 output block per workgroup, the input channels split
        // over wk waves in runs of 16, everything in one pass
        if (d.KH != 1 || d.KW != 1 || d.pad != 0) return fail("tile.alg = 3 needs a 1x1 / pad 0 convolution");
        if (!flat && t.ks != 1) return fail("tile.alg = 3 with stride > 1 has no split across workgroups");
        if (t.mf != 16 || t.mb != 1 || t.nb != 1 || t.wm != 1 || t.wn != 1) return fail("tile.alg = 3 needs mf = 16 and one block per workgroup");
        if (t.wl != 0) return fail("tile.alg = 3 has no loader waves");
        if (tail_N > 0) return fail("tile.alg = 3 cannot carry a fused tail");
        const int runs = (t.cch % (16 * t.wk) == 0) ? t.cch / (16 * t.wk) : 0;
        if (runs != 1 && runs != 2 && runs != 4 && runs != 8) return fail("tile.alg = 3 needs cch = 16 * wk * {1, 2, 4, 8}");
        if (runs == 8 && t.wk > 8) return fail("tile.alg = 3 with eight runs per wave is built for at most 8 waves");
        if (ceil_div(d.C, t.cch) != t.ks) return fail("tile.alg = 3 takes its input channels in one pass: ks slices of cch channels must cover them exactly");
        if (t.tw != std::min(16, g.P)) return fail("tile.alg = 3 needs tw = min(16, pixels)");
        if ((long long)t.cch * g.We * 4 >= (1LL << 31)) return fail("image too large for tile.alg = 3");
    }
    if (t.alg == 7) {
        // register-blocked 1x1 convolution: 16*mb channels x 16*nb pixels per wave, the pixels of the whole batch in one
        // row of groups of nb (or single pixels, where a group does not fit an image or the convolution has a stride)
        if (d.KH != 1 || d.KW != 1 || d.pad != 0) return fail("tile.alg = 7 needs a 1x1 / pad 0 convolution");
        if (t.mf != 16 || (t.nb != 2 && t.nb != 4)) return fail("tile.alg = 7 needs mf = 16 and nb = 2 or 4");
        if (t.wl != 0 || t.ks != 1) return fail("tile.alg = 7 has no loader waves and no split across workgroups");
        if (tail_N > 0) return fail("tile.alg = 7 cannot carry a fused tail");
        if (t.wk > 1 && t.wk > 4 * t.mb) return fail("tile.alg = 7: more channel slices than rows to finish");
        if (t.cch % (16 * t.wk) != 0 || t.cch < d.C || t.cch - d.C >= 16 * t.wk)
            return fail("tile.alg = 7 takes all input channels in one pass: cch = C rounded up to 16 * wk");
        g.gen = !flat || g.P < t.nb;
        g.units_image = g.gen ? g.P : ceil_div(g.P, t.nb);
        if (t.tw != 1 && t.tw != 8 && t.tw != 16 && t.tw != 32) return fail("tile.alg = 7 needs tw = 1, 8, 16 or 32");
        const long long units = (long long)d.batch * g.units_image;
        if (units * g.units_image >= (1LL << 32) || units >= (1LL << 30)) return fail("batch too large for tile.alg = 7");
        g.units = (int)units;
        g.unit_images = std::min(d.batch - 1, (16 * (g.gen ? t.nb : 1) - 2) / g.units_image + 1);
        if ((long long)d.H * d.W * std::max(d.C, t.cch) * 4 >= (1LL << 31)) return fail("image too large for tile.alg = 7");
    }
    if (t.alg == 2) {
        // direct 3x3 convolution with the weights read from global memory into registers, a pair of channel groups at a time
        if (d.KH != 3 || d.KW != 3 || d.dilation != 1) return fail("tile.alg = 2 needs a 3x3 / dilation 1 convolution");
        if (t.mb != 1 || t.nb != 1) return fail("tile.alg = 2 needs mb = nb = 1");
        if (tail_N > 0) return fail("tile.alg = 2 cannot carry a fused tail");
        if (t.cch % (2 * g.kc * t.wk) != 0) return fail("tile.alg = 2 needs an even number of channel groups per wave and pass");
    }
    if (t.alg == 1 && !wino_batch) {
        // Winograd F(2x2,3x3): a pixel lane holds one 2x2 output tile; the workgroup tile is THt x TWt such tiles.
        if (d.KH != 3 || d.KW != 3 || d.stride != 1 || d.dilation != 1) return fail("tile.alg needs a 3x3 / stride 1 / dilation 1 convolution");
        if (t.mf != 16 || t.mb != 1 || t.nb != 1) return fail("tile.alg needs mf = 16, mb = nb = 1");
        if (tail_N > 0) return fail("tile.alg cannot carry a fused tail");
        const int lanes = 16 * t.wn;
        const int Wt = ceil_div(g.Wo, 2), Ht = ceil_div(g.Ho, 2);
        if (t.tw < 1 || t.tw > lanes || t.tw > Wt) return fail("tile.tw must be in [1, min(ceil(Wo/2), tile lanes)]");
        g.ktaps = 16;
        g.TWt = t.tw;
        g.THt = std::min(lanes / t.tw, Ht);
        g.TW = 2 * g.TWt;
        g.TH = 2 * g.THt;
        g.PT = 4 * lanes;   // pixels the workgroup's lanes stand for
    } else if (t.alg == 5) {
        g.ktaps = 16;
        g.TW = 28;
        g.TH = 2;
        g.PT = 64;          // two rows of 32 columns in the parked tile (28 of them real)
    } else if (t.alg == 7) {
        g.PT = t.mf * t.nb * t.wn;
        g.TW = std::min(g.PT, g.P);
        g.TH = 1;
    } else if (!wino_batch) {
        g.PT = t.mf * t.nb * t.wn;
        // (the streamed 1x1 kernel walks the output in runs of 16 consecutive pixels, whatever the image's rows are)
        const bool runs = t.alg == 3 && !flat;
        if (t.tw < 1 || t.tw > g.PT || (!runs && t.tw > g.Wo)) return fail("tile.tw must be in [1, min(Wo, pixel lanes)]");
        g.TW = t.tw;
        g.TH = runs ? 1 : std::min(g.PT / t.tw, g.Ho);
        if (t.alg == 4 || t.alg == 6) g.TH = std::min(16 / t.tw, g.Ho);   // (a block is 16 pixel lanes, whatever nb is)
    }
    g.ntx = ceil_div(g.Wo, g.TW);
    if ((t.alg == 4 || t.alg == 6) && t.nb > 1) g.ntx = ceil_div(g.ntx, t.nb);   // a workgroup takes nb neighbouring tiles of a row
    g.nty = ceil_div(g.Ho, g.TH);
    if (t.alg == 3 && !flat) {
        g.ntx = ceil_div(g.P, 16);
        g.nty = 1;
    }
    if (t.alg == 7) {
        g.ntx = ceil_div(g.units, 16 * (g.gen ? t.nb : 1) * t.wn);
        g.nty = 1;
    }
    if (wino_batch) {
        g.ntx = ceil_div(g.units, 16 * t.wn);
        g.nty = 1;
    }
    const bool flat_batch = t.alg == 7 || wino_batch;   // grid_x counts the pixels (tiles) of all images
    // (the kernel divides the tile index by ntx with a 32-bit multiply-high)
    if (!flat_batch && (long long)g.ntx * g.nty > 65535 * 16) return fail("grid too large");
    if (!flat_batch && (long long)g.ntx * g.nty * g.ntx >= (1LL << 32)) return fail("grid too large");
    g.grid_x = g.ntx * g.nty;
    g.grid_y = ceil_div(d.N, g.MT);
    if (t.ks < 1 || t.ks > 64) return fail("tile.ks must be in [1, 64]");
    g.ks = t.ks;
    if ((long long)d.batch * t.ks > 65535) return fail("grid too large");
    g.grid_z = flat_batch ? 1 : d.batch * t.ks;
    if (g.grid_y > 65535) return fail("grid too large");
    const int granule = g.kc * t.wk;
    if (t.cch < granule || t.cch % granule != 0) return fail("tile.cch must be a positive multiple of kc*wk");
    if (t.alg < 3 && !wino_batch && t.cch > round_up(d.C, granule)) return fail("tile.cch exceeds the (padded) channel count");
    g.cpw = t.cch / t.wk;
    g.nchunks = ceil_div(d.C, t.cch);
    g.c_pad = g.nchunks * t.cch;
    g.cps = ceil_div(g.nchunks, t.ks);
    if ((t.ks - 1) * g.cps >= g.nchunks) return fail("tile.ks leaves a workgroup without input channels");
    g.nrows = (g.TH - 1) * d.stride + (d.KH - 1) * d.dilation + 1;
    g.ncols = (g.TW - 1) * d.stride + (d.KW - 1) * d.dilation + 1;
    // LDS rows are filled with 16-byte elements when image rows are a multiple of
    // 4 floats: the window then starts at the 4-float boundary at or left of its
    // first column, which can cost up to 3 extra columns.
    g.VW = (g.We % 4 == 0) ? 4 : 1;
    if (g.VW == 4) {
        int shift = 0;
        for (int tx = 0; tx < std::min(g.ntx, 4); ++tx) {
            const int ix0 = tx * g.TW * d.stride - d.pad;
            shift = std::max(shift, ((ix0 % 4) + 4) % 4);
        }
        g.RS = round_up(g.ncols + shift, 4);
    } else {
        g.RS = g.ncols;
    }
    // (Winograd: lane l reads the 4x4 input patch of tile l, two floats to the right and two rows down per tile)
    g.CS = t.alg == 1 ? pad_channel_stride(g.nrows * g.RS, 16, g.VW, 16 * t.wn, g.TWt, g.THt, g.RS, 2, &g.b_ways)
                  : pad_channel_stride(g.nrows * g.RS, t.mf, g.VW, g.PT, g.TW, g.TH, g.RS, d.stride, &g.b_ways);
    // Copies are issued in whole blocks of 64 elements (1 KiB with 16-byte elements): both parts of
    // a stage are rounded up to that, the slack receiving zeros.
    g.in_stage_floats = round_up(t.cch * g.CS, 256);
    g.wslab_floats = (t.wm * t.mb) * (t.cch / g.kc) * g.ktaps * 64;
    g.aff_floats = (d.KH == 1 && d.KW == 1 && d.pad == 0) ? round_up(2 * t.cch, 256) : 0;
    // (the Winograd path reads its weights straight from global memory into registers: the LDS holds input only)
    g.stage_floats = g.in_stage_floats + (t.alg ? 0 : round_up(g.wslab_floats, 256)) + g.aff_floats;   // (wino = 2 likewise)
    if (t.alg >= 3 || wino_batch) g.in_stage_floats = g.aff_floats = g.stage_floats = 0;   // nothing is staged
    g.nstage = g.cps > 1 ? 2 : 1;
    const long long stage_bytes = (long long)g.nstage * g.stage_floats * 4;
    // (the Winograd path always parks its output tiles in LDS, also without a split over waves)
    // (... and so does the streamed 3x3 kernel with several pixel blocks per wave: all its threads share the final store)
    const long long red_bytes = (t.wk > 1 || t.alg == 1 || t.alg == 5 || ((t.alg == 4 || t.alg == 6) && t.nb > 1)) ? (long long)t.wk * g.MT * g.PT * 4 : 0;
    long long lds = std::max(stage_bytes, red_bytes);
    if (wino_batch) {   // two buffers of transformed weights per team, or the outputs of all teams (nb = 2: and those of their parts)
        const long long weights = 2LL * t.wk * t.mb * 2 * 4096, outputs = (long long)t.wk * t.wn * t.mb * 4096;
        lds = t.nb == 2 ? weights + outputs : std::max(weights, t.wk > 1 ? outputs : 0);
    }
    if (tail_N > 0) {
        // A fused 1x1 tail needs every output channel of the convolution in one workgroup; its tile is parked
        // in LDS behind the split-K partials with a row stride that keeps the four channel quarters of a
        // K-step in different banks.
        if (tail_N > 4096) return fail("fused tail too wide");
        if (g.grid_y != 1) return fail("a fused tail needs all output channels in one workgroup tile");
        if (t.ks != 1) return fail("a fused tail cannot be combined with a split across workgroups");
        g.tail_N = tail_N;
        g.tail_ng = ceil_div(d.N, 4);
        g.tail_ld = (g.PT % 32 == 0) ? g.PT + 16 : g.PT;
        g.tail_f_off = t.wk > 1 ? t.wk * g.MT * g.PT : 0;
        lds = std::max(lds, ((long long)g.tail_f_off + (long long)g.MT * g.tail_ld) * 4);
    }
    if (t.alg >= 3 && t.ks > 1) lds = std::max<long long>(lds, 16);   // the drawn ticket is passed through LDS
    if (t.alg == 6) {
        // The input window of a tile: (TH-1)*stride+3 rows; columns from the multiple of four at or left of the tile's first
        // input column (up to three more than the (TW-1)*stride+3 the taps touch), in segments of four.  One slot per lane
        // of a channel quarter and request.
        g.win_rows = (g.TH - 1) * d.stride + 3;
        g.win_L = ceil_div((g.TW * t.nb - 1) * d.stride + 3 + 3, 4);   // (nb > 1: the blocks lie side by side in one window)
        g.win_nreq = ceil_div(g.win_rows * g.win_L, 16);
        if (g.win_nreq > (t.nb == 4 ? 3 : 2)) return fail("tile.alg = 6: the input window of this tile needs too many requests per group");
        if (d.W < 4) return fail("tile.alg = 6 needs an image at least four columns wide");
        g.win_ns = g.win_rows * g.win_L * 4;
        while (g.win_ns % 32 != 16) g.win_ns += 4;
        g.win_off = (int)((lds + 15) / 16 * 4);
        lds = (long long)g.win_off * 4 + (long long)g.waves * (t.cch / t.wk) * g.win_ns * 4;
    }
    if (lds > machine().lds_bytes_per_cu) return fail("tile needs more than 160 KiB of LDS");
    g.lds_bytes = (int)lds;
    if (const char *e = std::getenv("TDC_EXPERIMENT_MIN_LDS")) g.lds_bytes = std::max(g.lds_bytes, std::atoi(e));
    if ((long long)g.grid_y * g.nchunks * g.wslab_floats * 4 >= (1LL << 31)) return fail("packed weights exceed 2 GiB");
    // (the kernel decodes a one-dimensional launch index with 32-bit multiply-high divisions)
    const long long n_wg = (long long)g.grid_x * g.grid_y * g.grid_z;
    if (n_wg + 8 >= (1LL << 28) || n_wg * std::max(g.grid_x, g.grid_y) >= (1LL << 32)) return fail("grid too large");
    g.channel_major = channel_major_order(4.0 * d.C * d.H * d.W * (flat_batch ? d.batch : 1), 4.0 * d.N * d.C * g.taps, n_wg, g.grid_y);
    return true;
}

size_t packed_part_floats(const Geometry &g) { return (size_t)g.grid_y * (size_t)g.nchunks * (size_t)g.wslab_floats; }
size_t packed_weight_floats(const Geometry &g) { return packed_part_floats(g) + (size_t)g.scale_floats + g.raw_floats; }

static uint16_t to_bf16(float v) {   // nearest even; a finite value never becomes infinite
    uint32_t u;
    std::memcpy(&u, &v, 4);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    const uint32_t r = u + 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(((r & 0x7f800000u) == 0x7f800000u ? u : r) >> 16);
}
static float from_bf16(uint16_t h) {
    const uint32_t u = (uint32_t)h << 16;
    float v;
    std::memcpy(&v, &u, 4);
    return v;
}

// tile.alg = 8: per (16 channels, pass, K-step, part): [lane][8], lane (n = l % 16, k = l / 16) holding part 0, 1 or 2 of the
// weights of channel block*16 + n and K octet 4*step + k.  An octet is eight input channels of one tap, or (cch = 4) four
// channels of two neighbouring taps of a filter row.
// The last of the three parts is exact only above 2^-110, and sums below 2^-90 cost the kernel a second pass.  Trained networks
// hold whole channels that weight decay left near nothing, so a channel whose largest weight is outside 2^-40 ... 2^20 is packed
// times the power of two that brings it to 1, and its sums are multiplied by the inverse, which follows the weights.  The factor
// is negative where a weight other than zero lies below 2^-110 as packed: the kernel then mistrusts zeros and large inputs.
static float split_channel_scale(const tdc_conv_desc &d, const float *w, int n) {
    const size_t per = (size_t)d.C * d.KH * d.KW;
    float largest = 0.0f;
    for (size_t i = 0; i < per; ++i)
        if (std::isfinite(w[n * per + i])) largest = std::max(largest, std::fabs(w[n * per + i]));
    const float scale = largest == 0.0f || (largest >= 0x1p-40f && largest <= 0x1p20f) ? 1.0f : std::ldexp(1.0f, std::ilogb(largest));
    for (size_t i = 0; i < per; ++i)
        if (w[n * per + i] != 0.0f && std::fabs((double)w[n * per + i]) < 0x1p-110 * scale) return -scale;
    return scale;
}

static void pack_split_weights(const tdc_conv_desc &d, const tdc_tile &t, const Geometry &g, const float *w, float *packed) {
    float *const scales = packed + packed_part_floats(g);
    std::vector<int> shift((size_t)g.scale_floats - 4, 0);
    std::fill(scales, scales + 4, 0.0f);
    for (int n = 0; n < g.scale_floats - 4; ++n) {
        const float s = n < d.N ? split_channel_scale(d, w, n) : 1.0f;
        scales[4 + n] = s;
        shift[n] = -std::ilogb(s);
        if (s != 1.0f) scales[0] = 1.0f;
    }
    uint16_t *const dst = reinterpret_cast<uint16_t *>(packed);
    const bool few = t.tw != 0 && t.cch == 4;
    const int octets = t.cch / 8, blocks = g.grid_y * t.wm * t.mb;
    size_t base = 0;
    for (int blk = 0; blk < blocks; ++blk)
        for (int pass = 0; pass < g.nchunks; ++pass)
            for (int ks = 0; ks < g.ksteps; ++ks, base += 3 * 512)
                for (int l = 0; l < 64; ++l)
                    for (int e = 0; e < 8; ++e) {
                        const int idx = 4 * ks + l / 16, n = blk * 16 + l % 16;
                        int c, ky, kx;
                        if (few) {
                            c = e & 3;
                            ky = idx / g.row_taps;
                            kx = 2 * (idx % g.row_taps) + (e >> 2);
                        } else {
                            const int tap = idx / octets;
                            c = pass * t.cch + 8 * (idx % octets) + e;
                            ky = tap / d.KW;
                            kx = tap % d.KW;
                        }
                        float v = (n < d.N && c < d.C && ky < d.KH && kx < d.KW) ? w[(((size_t)n * d.C + c) * d.KH + ky) * d.KW + kx] : 0.0f;
                        if (shift[n]) v = std::ldexp(v, shift[n]);
                        for (int s = 0; s < 3; ++s) {
                            const uint16_t h = to_bf16(v);
                            dst[base + (size_t)s * 512 + l * 8 + e] = h;
                            v = std::isfinite(v) ? v - from_bf16(h) : 0.0f;
                        }
                    }
}

void pack_weights(const tdc_conv_desc &d, const tdc_tile &t, const Geometry &g, const float *w, float *packed) {
    const int mbw = t.wm * t.mb;
    const int ncg = t.cch / g.kc;
    const int taps = g.taps;
    float *dst = packed;
    if (g.raw_floats) std::memcpy(packed + (packed_weight_floats(g) - g.raw_floats), w, g.raw_floats * sizeof(float));
    if (t.alg == 8) {
        pack_split_weights(d, t, g, w, packed);
        return;
    }
    if (t.alg == 2 || t.alg == 4 || t.alg == 6) {
        // per (channel tile, pass, M block, channel group): [taps 0-3][lane][4] [taps 4-7][lane][4] [tap 8][lane]
        for (int by = 0; by < g.grid_y; ++by)
            for (int chunk = 0; chunk < g.nchunks; ++chunk)
                for (int mbl = 0; mbl < mbw; ++mbl)
                    for (int cg = 0; cg < ncg; ++cg, dst += 9 * 64)
                        for (int tap = 0; tap < 9; ++tap)
                            for (int l = 0; l < 64; ++l) {
                                const int n = by * g.MT + mbl * t.mf + l % t.mf;
                                const int c = chunk * t.cch + cg * g.kc + l / t.mf;
                                const float v = (n < d.N && c < d.C) ? w[((size_t)n * d.C + c) * 9 + tap] : 0.0f;
                                dst[tap < 8 ? (tap / 4) * 256 + l * 4 + tap % 4 : 512 + l] = v;
                            }
        return;
    }
    if (t.alg == 3 || t.alg == 7) {
        // per (channel block, run of 16 input channels): [lane][s], lane (n = l % 16, k = l / 16) holding
        // w[block*16 + n][16*run + 4*k + s]; the runs of all slices of a split across workgroups follow each other
        const int runs = g.nchunks * (t.cch / 16);
        for (int by = 0; by < g.grid_y * mbw; ++by)
            for (int r = 0; r < runs; ++r)
                for (int l = 0; l < 64; ++l)
                    for (int e = 0; e < 4; ++e) {
                        const int n = by * 16 + l % 16, c = 16 * r + 4 * (l / 16) + e;
                        *dst++ = (n < d.N && c < d.C) ? w[(size_t)n * d.C + c] : 0.0f;
                    }
        return;
    }
    if (g.wino || t.alg == 5) {
        // Winograd F(2x2,3x3): U = G g G^T per (output channel, input channel), G = [1 0 0; .5 .5 .5; .5 -.5 .5; 0 0 1].
        // Per (channel tile, pass, M block, channel group): [q = 0..3][64 lanes][e = 0..3] holding U[q][e] of
        // (n = l % 16, c = l / 16), so that one 128-bit LDS read fetches the A operands of four of the 16 MFMAs.
        static const double G[4][3] = {{1, 0, 0}, {0.5, 0.5, 0.5}, {0.5, -0.5, 0.5}, {0, 0, 1}};
        for (int by = 0; by < g.grid_y; ++by)
            for (int chunk = 0; chunk < g.nchunks; ++chunk)
                for (int mbl = 0; mbl < mbw; ++mbl)
                    for (int cg = 0; cg < ncg; ++cg)
                        for (int q = 0; q < 4; ++q)
                            for (int l = 0; l < 64; ++l) {
                                const int n = by * g.MT + mbl * 16 + l % 16;
                                const int c = chunk * t.cch + cg * 4 + l / 16;
                                for (int e = 0; e < 4; ++e) {
                                    double u = 0.0;
                                    if (n < d.N && c < d.C) {
                                        const float *gk = w + ((size_t)n * d.C + c) * 9;
                                        for (int r = 0; r < 3; ++r)
                                            for (int s = 0; s < 3; ++s) u += G[q][r] * (double)gk[r * 3 + s] * G[e][s];
                                    }
                                    *dst++ = (float)u;
                                }
                            }
        return;
    }
    for (int by = 0; by < g.grid_y; ++by)
        for (int chunk = 0; chunk < g.nchunks; ++chunk)
            for (int mbl = 0; mbl < mbw; ++mbl)
                for (int cg = 0; cg < ncg; ++cg)
                    for (int tap = 0; tap < taps; ++tap)
                        for (int l = 0; l < 64; ++l) {
                            const int n = by * g.MT + mbl * t.mf + l % t.mf;
                            const int c = chunk * t.cch + cg * g.kc + l / t.mf;
                            *dst++ = (n < d.N && c < d.C) ? w[((size_t)n * d.C + c) * taps + tap] : 0.0f;
                        }
}

// ---------------------------------------------------------------------------
// Analytic model
// ---------------------------------------------------------------------------
namespace {

// Calibration constants of the latency model.  The defaults were fitted to a measured sweep of every
// launchable tile of the 28 benchmark layers on one MI355X (python -m tdc_amd.fit_model); they can be
// replaced at run time through tdc_model_set_constants, e.g. for another CDNA part.  They play the role
// of num_sm / num_threads / the (a, b, c) weights / the keep-ratio in the reference's model
// (2080Ti-evaluation/TDC-LAYERS-MODELING/model.py:265-266,278).
struct ModelConst {
    double launch_us = 1.474;           // device time of an empty kernel in a back-to-back stream
    double setup_clk = 1479;          // kernel arguments and index arithmetic before the first copy is issued
    double copy_latency_clk = 798.12;   // first byte of a global->LDS copy (L2 / memory-side cache)
    double copy_bytes_per_clk = 42.0036;   // sustained global->LDS rate of one CU
    double l2_bytes_per_clk = 12019.7;   // whole-chip L2->CU rate when every CU copies at once
    double lds_bytes_per_clk = 41.148;   // LDS traffic of the split-K reduction
    double sync_clk = 275.2;            // one workgroup barrier
    double store_bytes_per_clk = 2.827;  // per CU, short runs per channel
    double kstep_issue_clk = 4.36679;      // vector-ALU / LDS-issue cycles per operand read, not hidden under MFMAs
    double pass_overhead_clk = 371.876;   // per wave and pass: copy issue, pointer set-up, pipeline fill
    double wave_setup_clk = 778.32;      // prologue cycles added per extra wave sharing a SIMD
    double ksplit_clk = 3381.18;         // split across workgroups: write-through, ticket round trip, read-back
    double copy_issue_clk = 100.5;      // a wave is held this long by every global->LDS copy instruction it issues
    double lds_read_clk = 1.44;        // LDS busy cycles per conflict-free operand read of one wave
    double wino_kstep_clk = 16.788;      // Winograd: cycles per MFMA that the input transform adds on top of the operand reads
    double gw_latency_clk = 1040.3;       // alg 2: the first weights come from L2 into registers after the input copy is under way
    double stream_setup_clk = 459;      // alg 3: index arithmetic before the requests go out (no copy tables, no stages)
    double stream_latency_clk = 774;    // alg 3: round trip of the first request, global memory -> registers
};
ModelConst MC;
std::shared_mutex MC_mutex;   // readers: every model evaluation; writer: tdc_model_set_constants
constexpr int kNumModelConst = 18;

double *mc_field(int i) {
    switch (i) {
        case 0: return &MC.launch_us;
        case 1: return &MC.setup_clk;
        case 2: return &MC.copy_latency_clk;
        case 3: return &MC.copy_bytes_per_clk;
        case 4: return &MC.l2_bytes_per_clk;
        case 5: return &MC.lds_bytes_per_clk;
        case 6: return &MC.sync_clk;
        case 7: return &MC.store_bytes_per_clk;
        case 8: return &MC.kstep_issue_clk;
        case 9: return &MC.pass_overhead_clk;
        case 10: return &MC.wave_setup_clk;
        case 11: return &MC.ksplit_clk;
        case 12: return &MC.copy_issue_clk;
        case 13: return &MC.lds_read_clk;
        case 14: return &MC.wino_kstep_clk;
        case 15: return &MC.gw_latency_clk;
        case 16: return &MC.stream_setup_clk;
        case 17: return &MC.stream_latency_clk;
        default: return nullptr;
    }
}

}  // namespace

struct CompiledKernel { const char *name; int regs, sgprs, waves; };
// hipcc's resource report for the convolution kernels of this build (written by the Makefile from the compile of
// every conv_*.hip with kernels): name, VGPRs + AGPRs per lane, scalar registers, waves per SIMD.
static const CompiledKernel compiled_kernels[] = {
#include "kernel_registers.inc"
};

static const CompiledKernel *compiled_kernel(const KernelId &k) {
    static const std::map<std::string, const CompiledKernel *> by_name = [] {
        std::map<std::string, const CompiledKernel *> m;
        for (const CompiledKernel &c : compiled_kernels) m[c.name] = &c;
        return m;
    }();
    // (a selection asks for the same hundred kernels tens of thousands of times: the name is spelt out once per thread)
    static thread_local std::unordered_map<uint64_t, const CompiledKernel *> known;
    uint64_t key = (uint64_t)k.family;
    for (int v : k.p) key = key << 8 | (uint64_t)(v & 255);
    auto hit = known.find(key);
    if (hit == known.end()) {
        const auto it = by_name.find(kernel_name(k));
        hit = known.emplace(key, it == by_name.end() ? nullptr : it->second).first;
    }
    return hit->second;
}

// Waves of this kernel that fit one SIMD, as the compiler works it out from the registers of the compiled kernel:
// 512 vector registers per lane shared by a SIMD's waves (handed out in blocks of 8), at most 8 waves, and 800 scalar
// registers in blocks of 16 — the staged kernel needs 106 (112 allocated), which leaves room for 7 waves, not 8, so
// a 1024-thread workgroup of it is alone on its compute unit however few vector registers it uses (the HIP runtime's
// occupancy query says the same).
int kernel_waves_per_simd(const KernelId &k) {
    const CompiledKernel *c = compiled_kernel(k);
    if (!c) return 0;
    const Machine &m = machine();
    const int by_vgpr = m.vgprs_per_simd_lane / ((c->regs + 7) / 8 * 8);
    const int by_sgpr = 800 / ((c->sgprs + 15) / 16 * 16);
    return std::min(std::min(m.max_waves_per_simd, by_vgpr), std::min(by_sgpr, c->waves));
}

KernelId kernel_id_with_head(const tdc_tile &t) {
    KernelId k;
    if (t.alg != 4 || t.ks != 1 || t.wk < 1 || t.cch % (4 * t.wk) != 0) return k;
    const int cg = t.cch / (4 * t.wk);
    if (cg != 1 && cg != 2 && cg != 4) return k;
    k.family = KernelId::STREAM_3x3;
    k.p[0] = cg; k.p[1] = 0; k.p[2] = 3; k.p[3] = 1;
    return k;
}

int wino_stream_max_waves(int groups) { return (groups >= 1 && groups <= 4) ? 16 : 0; }

KernelId kernel_id_for(const tdc_tile &t, int KH, int KW, int dilation, int stride, bool extras, bool single_pixels) {
    KernelId k;
    if (t.alg == 8) {
        if (t.mf != 16 || (t.nb != 2 && t.nb != 4) || (t.mb != 1 && t.mb != 2 && t.mb != 4)) return k;
        // (`extras` here can only mean the input affine of a 1x1 convolution)
        const int mode = t.tw == 0 ? 0 : t.cch == 4 ? 2 : 1;
        if (mode == 0 ? t.mb > 2 : mode == 2 && t.nb != 4) return k;
        if ((mode == 0) != (KH == 1 && KW == 1)) return k;
        if ((mode != 0 && extras) || (mode == 2 && dilation != 1)) return k;
        k.p[0] = t.mb;
        k.family = mode == 1 && t.nb == 2 ? KernelId::SPLIT_CORE : KernelId::SPLIT;
        if (k.family == KernelId::SPLIT) k.p[1] = t.nb, k.p[2] = mode, k.p[3] = extras;
        return k;
    }
    if (t.alg == 1 && t.tw == 0) {
        if (extras || KH != 3 || KW != 3 || dilation != 1 || stride != 1 || t.mf != 16 || t.wm != 1 || (t.wn != 2 && t.wn != 4) ||
            (t.mb != 1 && t.mb != 2) || (t.nb != 1 && t.nb != 2) || (t.nb == 2 && t.mb == 2 && t.wn == 2))
            return k;
        k.family = KernelId::BLOCK_WINO;
        k.p[0] = t.mb; k.p[1] = t.wn; k.p[2] = t.nb == 2;
        return k;
    }
    if (t.alg == 7) {
        // (`extras` here can only mean the input affine)
        if (KH != 1 || KW != 1 || t.mf != 16 || (t.mb != 1 && t.mb != 2) || (t.nb != 2 && t.nb != 4)) return k;
        k.family = KernelId::BLOCK_1x1;
        k.p[0] = t.mb; k.p[1] = t.nb; k.p[2] = extras; k.p[3] = single_pixels; k.p[4] = t.tw >= 8 ? t.tw : 0;
        return k;
    }
    if (t.alg == 5) {
        if (extras || KH != 3 || KW != 3 || dilation != 1 || stride != 1 || t.mf != 16 || t.mb != 1 || t.nb != 1 || t.wn != 1 ||
            t.wm < 1 || t.wk < 1 || t.ks != 1 || t.cch % (4 * t.wk) != 0)
            return k;
        const int cg = t.cch / (4 * t.wk);
        const int maxw = wino_stream_max_waves(cg);
        if (!maxw || t.wm * t.wk > maxw) return k;
        k.family = KernelId::STREAM_WINO;
        k.p[0] = cg; k.p[1] = maxw;
        return k;
    }
    if (t.alg == 4 || t.alg == 6) {
        // (`extras` can only mean a fused tail here, which the one kernel carries)
        if (KH != 3 || KW != 3 || dilation != 1 || t.mf != 16 || t.mb != 1 || t.wm < 1 || t.wn != 1 || t.wk < 1 ||
            t.wm * t.wk > 16 || t.cch % (4 * t.wk) != 0)
            return k;
        const int cg = t.cch / (4 * t.wk);
        if ((cg != 1 && cg != 2 && cg != 4) || (extras && t.ks > 1)) return k;
        const bool row = stride == 1 && t.tw == 14;   // one row of 14 pixels: the taps of a filter row are lane shifts
        if (t.nb != 1) {
            // several pixel blocks per wave: row tiles, no extras, no split across workgroups
            if ((t.nb != 2 && t.nb != 4) || !row || extras || t.ks > 1) return k;
            if (t.alg == 6 && t.nb == 4 && cg == 4) return k;
        }
        k.family = KernelId::STREAM_3x3;
        k.p[0] = cg;
        k.p[1] = t.alg == 6 ? 2 : row;
        k.p[2] = extras ? 2 : t.ks > 1 ? 1 : 0;
        k.p[3] = t.nb;
        return k;
    }
    if (t.alg == 3) {
        // (`extras` here can only mean the input affine: the host refuses a fused tail for this path)
        if (KH != 1 || KW != 1 || t.mf != 16 || t.mb != 1 || t.nb != 1 || t.wm != 1 || t.wn != 1 || t.wk < 1 ||
            t.cch % (16 * t.wk) != 0)
            return k;
        const int nq = t.cch / (16 * t.wk);
        if ((nq != 1 && nq != 2 && nq != 4 && nq != 8) || t.wk > (nq == 8 ? 8 : 16) || (stride > 1 && t.ks > 1)) return k;
        k.family = KernelId::STREAM_1x1;
        k.p[0] = nq; k.p[1] = extras; k.p[2] = stride > 1 ? 2 : t.ks > 1 ? 1 : 0;
        return k;
    }
    if (t.mf != 16 && t.mf != 32) return k;
    if (t.mb < 1 || t.mb > 2 || t.nb < 1 || t.nb > 2) return k;
    int taps;
    if (t.alg == 1) {
        if (extras || KH != 3 || KW != 3 || dilation != 1 || t.mf != 16 || t.mb != 1 || t.nb != 1) return k;
        taps = TAPS_WINO;
    } else if (t.alg == 2) {
        if (extras || KH != 3 || KW != 3 || dilation != 1 || t.mb != 1 || t.nb != 1) return k;
        taps = TAPS_3x3G;
    } else if (t.alg == 0) {
        taps = (KH == 3 && KW == 3 && dilation == 1) ? TAPS_3x3 : (KH == 1 && KW == 1) ? TAPS_1x1
             : (KH == 7 && KW == 7 && dilation == 1 && !extras) ? TAPS_7x7   // (the network stems; built without the extras)
                                                                : TAPS_GENERIC;
    } else {
        return k;
    }
    k.family = KernelId::STAGED;
    k.p[0] = t.mf; k.p[1] = t.mb; k.p[2] = t.nb; k.p[3] = taps;
    k.p[4] = taps == TAPS_WINO ? 12 : (t.mb == 2 && t.nb == 2) ? 8 : 16;   // launch bound in waves
    k.p[5] = extras;
    return k;
}

std::string kernel_name(const KernelId &k) {
    char buf[96];
    const char *tf[2] = {"false", "true"};
    switch (k.family) {
        case KernelId::STAGED:
            std::snprintf(buf, sizeof buf, "tdc_conv_mfma_kernel<%d, %d, %d, %d, %d, %s>", k.p[0], k.p[1], k.p[2], k.p[3], k.p[4], tf[k.p[5] != 0]);
            break;
        case KernelId::STREAM_1x1:
            std::snprintf(buf, sizeof buf, "tdc_conv1x1_stream_kernel<%d, %s, %d>", k.p[0], tf[k.p[1] != 0], k.p[2]);
            break;
        case KernelId::STREAM_3x3:
            if (k.p[3] > 1) std::snprintf(buf, sizeof buf, "tdc_conv3x3_stream_rownb_kernel<%d, %d, %s>", k.p[0], k.p[3], tf[k.p[1] == 2]);
            else std::snprintf(buf, sizeof buf, "tdc_conv3x3_stream_kernel<%d, %d, %d>", k.p[0], k.p[1], k.p[2]);
            break;
        case KernelId::STREAM_WINO:
            std::snprintf(buf, sizeof buf, "tdc_wino3x3_stream_kernel<%d, %d>", k.p[0], k.p[1]);
            break;
        case KernelId::BLOCK_WINO:
            std::snprintf(buf, sizeof buf, "tdc_wino3x3_block_kernel<%d, %d, %s>", k.p[0], k.p[1], tf[k.p[2] != 0]);
            break;
        case KernelId::BLOCK_1x1:
            std::snprintf(buf, sizeof buf, "tdc_conv1x1_block_kernel<%d, %d, %s, %s, %d>", k.p[0], k.p[1], tf[k.p[2] != 0], tf[k.p[3] != 0], k.p[4]);
            break;
        case KernelId::SPLIT:
            std::snprintf(buf, sizeof buf, "tdc_conv_split_kernel<%d, %d, %d, %s>", k.p[0], k.p[1], k.p[2], tf[k.p[3] != 0]);
            break;
        case KernelId::SPLIT_CORE:
            std::snprintf(buf, sizeof buf, "tdc_core_split_kernel<%d>", k.p[0]);
            break;
        default: return "";
    }
    return buf;
}

// Registers per lane of the compiled instantiation (hipcc's kernel-resource-usage report: VGPRs + AGPRs), rounded up
// to the allocation granule of 8; 0 for a kernel the library does not hold.  The reference measures occupancy per
// candidate by compiling and probing each (2080Ti-evaluation/Gen-occupancy/template.cu:277-284); here the candidates
// share about a hundred instantiations, whose report the build compiles into this file.
int kernel_vgprs(const KernelId &k) {
    const CompiledKernel *c = compiled_kernel(k);
    return c ? (c->regs + 7) / 8 * 8 : 0;
}

// Price of the split-operand tiles for filters of several taps, in us: a power mean of what a SIMD has to issue (MFMAs, K-steps,
// staging, stores), of the rounds of workgroups that each take their own chain of stages, and of the weights' way through the
// L1s, + launch + memory traffic.  `last`: share of a last, partly filled round of workgroups that counts as a whole one; `idle`: what a
// launch of fewer workgroups than compute units saves.
struct SplitPrice {
    double pipe_mfma, pipe_step, pipe_stage, pipe_block;
    double start, stage, stage_entry, step, mfma, block;
    double weights, launch_us, traffic, power, fragment;
    double last, idle;
};
static const SplitPrice split_core_price = {0.739, 191.1, 460.1, 600.3, 2930, 2593, 1098, 303.2, 0.8651, 417.2, 1.009, 3.726, 34.35, 2.024, 0.3892, 0.5, 0.0};
static double split_price(const SplitPrice &q, const tdc_conv_desc &d, const tdc_tile &t, const Geometry &g, int wg_per_cu) {
    const double wgs = (double)g.grid_x * g.grid_y / machine().cus;
    const double load = q.last * std::ceil(wgs) + (1.0 - q.last) * std::max(wgs, 1.0), simd = (double)g.waves / machine().simds_per_cu;
    const double steps = (double)g.nchunks * g.ksteps / t.wk, blocks = t.mb * t.nb, mfmas = steps * blocks * 96.0;
    const double entries = (g.lds_bytes - 32) / 48.0 / g.threads;
    const double stores = blocks * (1.0 + q.fragment * (16.0 / std::min(t.tw, 16) - 1.0));   // (short rows make short stores)
    const double shared = std::max(1.0, 0.75 * std::min(std::min((double)wg_per_cu, std::max(1.0, std::ceil(wgs))) * simd, 2.0));
    const double pipe = load * simd * (q.pipe_mfma * mfmas + q.pipe_step * steps + q.pipe_stage * g.nchunks * entries + q.pipe_block * stores);
    const double chain = std::ceil(wgs / wg_per_cu) *
                         (q.start + g.nchunks * (q.stage + q.stage_entry * entries) + q.step * steps + q.mfma * mfmas * shared + q.block * stores);
    const double l1 = q.weights * load * simd * 4.0 * steps * t.mb * 3072.0 / 56.0;
    const double clk = std::pow(std::pow(pipe, q.power) + std::pow(chain, q.power) + std::pow(l1, q.power), 1.0 / q.power);
    const double traffic = 4.0 * d.batch * ((double)d.C * d.H * d.W + (double)d.N * g.P) + 6.0 * d.C * d.N * g.ktaps;
    return std::pow(std::min(wgs, 1.0), q.idle) * (q.launch_us + clk / (machine().clock_ghz * 1e3) + traffic / (q.traffic * 1e6));
}

static bool is_core_split(const tdc_tile &t) { return t.alg == 8 && t.tw > 0 && t.nb == 2; }   // (conv_core_split.hip)

bool model_evaluate(const tdc_conv_desc &d, const tdc_tile &t, tdc_tile_info &info, std::string *why, int tail_N) {
    Geometry g;
    if (!make_geometry(d, t, g, why, tail_N)) return false;
    const Machine &m = machine();
    std::shared_lock<std::shared_mutex> constants_lock(MC_mutex);
    std::memset(&info, 0, sizeof(info));
    info.tile = t;
    info.grid_x = g.grid_x;
    info.grid_y = g.grid_y;
    info.grid_z = g.grid_z;
    info.block_threads = g.threads;
    info.lds_bytes = g.lds_bytes;
    info.nchunks = g.nchunks;
    info.th = g.TH;
    // (a fused tail needs the instantiation with the extras; an input affine, which the model does not know of, too)
    const KernelId kid = kernel_id_for(t, d.KH, d.KW, d.dilation, d.stride, tail_N > 0, g.gen);
    info.vgpr_estimate = kernel_vgprs(kid);
    if (info.vgpr_estimate <= 0) {
        if (why) *why = "no kernel instantiated for this tile";
        return false;
    }

    // --- occupancy (replaces cudaOccupancyMaxActiveBlocksPerMultiprocessor) ---
    const int waves_simd_vgpr = kernel_waves_per_simd(kid);   // registers per lane, and scalar registers per wave
    const int wg_waves_per_simd = ceil_div(g.waves, m.simds_per_cu);
    const int wg_by_vgpr = waves_simd_vgpr / wg_waves_per_simd;
    const int wg_by_lds = m.lds_bytes_per_cu / std::max(g.lds_bytes, 1);
    // (the staged kernels are never resident more than eight times per CU; the streamed one has no stage to hold)
    int wg_per_cu = std::min(std::min(wg_by_vgpr, wg_by_lds), t.alg >= 3 ? 32 : 8);
    if (wg_per_cu < 1) {
        if (why) *why = "tile does not fit one compute unit";
        return false;
    }
    info.wg_per_cu = wg_per_cu;
    info.waves_per_simd = wg_per_cu * wg_waves_per_simd;

    // --- algorithmic work and roofline ---------------------------------------
    const double P = (double)g.P;
    info.flops = 2.0 * P * d.C * d.N * g.taps * d.batch;
    info.bytes = 4.0 * ((double)d.batch * ((double)d.C * d.H * d.W + (double)d.N * P) +
                        (double)g.taps * d.C * d.N);
    if (tail_N > 0) {   // the intermediate never leaves the chip
        info.flops += 2.0 * P * d.N * tail_N * d.batch;
        info.bytes += 4.0 * ((double)d.batch * ((double)tail_N - d.N) * P + (double)d.N * tail_N);
    }
    info.roof_us = std::max(info.bytes / (m.hbm_tbps * 1e6), info.flops / (m.fp32_tflops * 1e6));

    // --- per-workgroup costs (clock cycles of one CU) ------------------------
    const long long n_wg = (long long)g.grid_x * g.grid_y * g.grid_z;
    const double mfma_clk = (t.mf == 32) ? 64.0 : 32.0;
    const double ksteps_pass = (double)(g.cpw / g.kc) * g.ktaps;
    // One wave's matrix-core time per pass; the LDS reads of a K-step (one A and
    // one B word per lane per block row/column) must fit under it.
    // (Winograd: the register transform of the input patch shares the wave's issue slots with its MFMAs)
    const double mfma_pass = ksteps_pass * t.mb * t.nb * (mfma_clk + (t.alg == 1 ? MC.wino_kstep_clk : 0.0));
    const double copy_bytes_pass = (double)g.stage_floats * 4.0;
    const double red_bytes = t.wk > 1 ? (double)t.wk * g.MT * g.PT * 4.0 * 2.0 : 0.0;
    // (the Winograd epilogue stores four pixels per instruction where tile and image width are multiples of four,
    //  two where the image width is even: cheaper per byte than single-pixel stores)
    const double store_width = t.alg != 1 ? 1.0 : ((g.TW | g.Wo) % 4 == 0) ? 0.6 : (g.Wo % 2 == 0) ? 0.85 : 1.0;
    const double out_bytes = (double)g.MT * g.PT * 4.0 * store_width;

    // Copy instructions of one pass (64 elements each) and how long issuing them holds a wave: the first
    // pass is dealt to every wave; later ones to the loader waves if there are any, else to everybody.
    const int ncomp = t.wm * t.wn * t.wk;
    const double n_instr = (double)g.in_stage_floats / (64.0 * g.VW) + (t.alg ? 0.0 : std::ceil(g.wslab_floats / 256.0));
    const double issue_first = std::ceil(n_instr / g.waves) * MC.copy_issue_clk;
    const double issue_steady = std::ceil(n_instr / (t.wl ? t.wl : g.waves)) * MC.copy_issue_clk;
    const int comp_waves_per_simd = ceil_div(ncomp, m.simds_per_cu);

    auto wg_time = [&](int r, long long concurrent_wgs) {
        if (t.alg == 5) {
            // like the streamed direct kernel: set-up, one round trip, the bytes at the achieved fill rate, the requests
            // of a wave one after the other, the MFMA chains of the waves that share a SIMD (the transform's vector work
            // mostly hides under them), output transform and drain, the reduction, the store.  Per input channel and 16
            // output channels 1 KiB of transformed weights; per input channel four rows of 128 bytes.
            // (fitted to 60 timed tiles of 13 shapes, 6 % mean error)
            const double chip_share =
                MC.l2_bytes_per_clk / std::max<double>(1.0, (double)std::min<long long>(concurrent_wgs, m.cus));
            const double rate = std::min(1.31 * MC.copy_bytes_per_clk, chip_share);
            const double bytes = (double)t.cch * (t.wm * 1024.0 + 512.0) * r;
            const double groups = (double)t.cch / (4.0 * t.wk);
            const double waves_simd = std::ceil((double)g.waves * r / m.simds_per_cu);
            double clk = MC.stream_setup_clk + MC.stream_latency_clk + 65.0 * (waves_simd - 1.0) + bytes / rate +
                         groups * 8.0 * 21.4 + waves_simd * groups * 16.0 * (mfma_clk + 10.0);
            clk += 1.6 * MC.sync_clk + 1000.0;   // MFMA drain, output transform, park, barrier
            const double rounds = std::ceil((double)g.MT * 32.0 / g.threads);
            clk += rounds * (110.0 + 8.0 * t.wk) + out_bytes * r / 200.0;
            return clk;
        }
        if (t.alg == 4 || t.alg == 6) {
            // as below; per input channel 576 bytes of weights and nine 64-byte rows of input (the rows of
            // neighbouring taps mostly hit in the L1, so they count for less than their size)
            const double chip_share =
                MC.l2_bytes_per_clk / std::max<double>(1.0, (double)std::min<long long>(concurrent_wgs, m.cus));
            // (fitted to 364 timed tiles of 35 shapes, 7 % mean error: the achieved fill rate is lower than that of the
            //  1x1 path; the nine taps of a lane are separate requests that mostly hit in the L1, three requests and lane
            //  shifts where a tile is one row of 14 pixels)
            const double rate = std::min(0.59 * MC.copy_bytes_per_clk, chip_share);
            const bool row_mode = d.stride == 1 && t.tw == 14;
            // (nb pixel blocks per wave: the input rows of every block, the weights once)
            // (alg 6: the window of the tile once, 16 bytes per slot)
            const double in_bytes_ch = t.alg == 6 ? 16.0 * g.win_rows * g.win_L * 0.7 : t.nb * (row_mode ? 0.28 : 0.66) * 576.0;
            const double bytes = (double)t.cch * t.wm * (576.0 + in_bytes_ch) * r;
            const double groups = (double)t.cch / (4.0 * t.wk);
            const double waves_simd = std::ceil((double)g.waves * r / m.simds_per_cu);
            // a wave issues its requests one after the other (about 21 cycles each): fewer groups per wave start sooner
            // (288 cycles per group: a wave's own nine MFMAs per block run one after the other)
            // (alg 6: one or two requests per group for the window, then its way through LDS: a write, nine reads)
            const double in_requests = t.alg == 6 ? (double)g.win_nreq : t.nb * (row_mode ? 3.0 : 9.0);
            double clk = MC.stream_setup_clk + MC.stream_latency_clk + 288.0 * groups + 65.0 * (waves_simd - 1.0) + bytes / rate +
                         groups * (3.0 + in_requests) * 21.4 + (t.alg == 6 ? 150.0 + 40.0 * groups * (t.nb > 1 ? 1.5 * t.nb : 1.0) : 0.0);
            // the MFMAs of the extra blocks no longer hide under the requests: the matrix pipe of a SIMD serves its waves in turn
            if (t.nb > 1) {
                clk += waves_simd * groups * 9.0 * (t.nb - 1) * mfma_clk;
                // all threads share the final sum and store; a workgroup of few waves walks its blocks in several rounds
                const double rounds = std::ceil((double)t.wm * t.nb * 256.0 / g.threads);
                clk += (rounds - 1.0) * (110.0 + 8.0 * t.wk);
            }
            if (t.wk > 1) clk += 1.6 * MC.sync_clk;
            if (tail_N > 0) {
                // park the columns, a barrier, the first touch of the tail's weights, its blocks dealt over the waves
                const double blocks = std::ceil((double)ceil_div(tail_N, 16) / g.waves);
                clk += MC.sync_clk + MC.stream_latency_clk + blocks * (g.tail_ng * 40.0 + 64.0) +
                       (double)tail_N * d.N * 4.0 * r / rate + (double)tail_N * 64.0 * r / 200.0;
                // More than eight slices cost another 0.5 to 0.6 us here (timed, 12 to 16 slices against half as many with twice the
                // channel groups each: 64 -> 16 -> 32 @14 4.73 against 4.21 us, 48 -> 16 -> 96 @20 4.74 against 4.24, 100 -> 16 -> 40
                // @21 5.46 against 5.22, 128 -> 16 -> 64 @14 5.58 against 5.35); up to eight, also times two channel blocks, nothing.
                if (t.wk > 8) clk += 1300.0;
                return clk;
            }
            if (t.ks > 1) clk += MC.ksplit_clk + 1000.0 * (t.ks - 2) + (double)t.ks * 1024.0 * r / rate;   // (timed: each slice past the second adds 0.4 us)
            clk += out_bytes * r / 200.0;
            return clk;
        }
        if (t.alg == 3) {
            // every wave requests its whole share up front and works through it as it arrives: one round trip, the
            // bytes at the CU's (or the chip's) fill rate, two chains of dependent MFMAs, the reduction over the waves
            const double chip_share =
                MC.l2_bytes_per_clk / std::max<double>(1.0, (double)std::min<long long>(concurrent_wgs, m.cus));
            const double rate = std::min(MC.copy_bytes_per_clk, chip_share);
            const double bytes = (double)t.cch * (64.0 + 64.0) * r;   // weights and input of one 16x16 block
            const double runs = (double)t.cch / (16.0 * t.wk);
            const double waves_simd = std::ceil((double)g.waves * r / m.simds_per_cu);
            // (fitted to 71 timed tiles of 23 shapes: the requests of all resident waves overlap, so only the bytes,
            //  a little per extra wave and half an MFMA time per K-step show; the stores are hidden)
            double clk = MC.stream_setup_clk + MC.stream_latency_clk + 20.0 * (waves_simd - 1.0) + bytes / (0.87 * rate) +
                         runs * 4.0 * 0.5 * mfma_clk * waves_simd;
            if (t.wk > 1) clk += 1.5 * MC.sync_clk;
            if (t.ks > 1) clk += MC.ksplit_clk + 1000.0 * (t.ks - 2) + (double)t.ks * 1024.0 * r / rate;   // (timed: each slice past the second adds 0.4 us)
            clk += out_bytes * r / 64.0;
            return clk;
        }
        // r workgroups share one CU: matrix time and the issue cycles of the operand reads add up per
        // SIMD; copies share the CU's fill rate and, chip-wide, the L2.
        const double waves_simd = (double)comp_waves_per_simd * r;
        // A wave alone on its SIMD stalls on every operand read and while it issues copies; with several
        // waves per SIMD those gaps are filled by the others until the matrix pipe itself is the limit.
        // (wino = 2: the A operands do not come from the LDS)
        const double a_reads = t.alg == 2 ? 0.25 * t.mb : (double)t.mb;
        const double stall = ksteps_pass * (a_reads + t.nb * g.b_ways) * MC.kstep_issue_clk + MC.pass_overhead_clk;
        const double alone = mfma_pass + stall;
        // ... or the LDS: every operand read keeps it busy for lds_read_clk cycles, a conflicting one longer.
        const double lds_busy = ksteps_pass * ((t.alg == 2 ? 0.0 : (double)t.mb) + t.nb * g.b_ways) * MC.lds_read_clk * ncomp * r;
        const double pipe = std::max(mfma_pass * waves_simd, lds_busy) + MC.pass_overhead_clk;
        const double compute = std::max(alone, pipe) + MC.sync_clk;
        const double compute_issuing = std::max(alone + issue_steady, pipe) + MC.sync_clk;
        const double chip_share =
            MC.l2_bytes_per_clk / std::max<double>(1.0, (double)std::min<long long>(concurrent_wgs, m.cus));
        const double rate = std::min(MC.copy_bytes_per_clk, chip_share);
        const double copy = copy_bytes_pass * r / rate;
        // First pass is exposed; afterwards the copy of pass i+1 runs under the MFMAs of pass i.
        double clk = MC.setup_clk + MC.wave_setup_clk * ((double)wg_waves_per_simd * r - 1.0) + issue_first +
                     MC.copy_latency_clk + copy + (t.alg == 2 ? MC.gw_latency_clk : 0.0);
        clk += compute;  // last pass: nothing left to hide
        if (g.cps > 1) {
            const double pass = t.wl ? std::max(compute, std::max(issue_steady, copy) + MC.copy_latency_clk)
                                     : std::max(compute_issuing, copy + MC.copy_latency_clk);
            clk += (g.cps - 1) * pass;
        }
        clk += red_bytes * r / MC.lds_bytes_per_clk + out_bytes * r / MC.store_bytes_per_clk +
               (t.wk > 1 ? 2.0 * MC.sync_clk : 0.0);
        // Split across workgroups: the partial tile goes to the workspace (the store above), and the
        // workgroup that draws the last ticket reads all ks partials back before the real store.
        if (t.ks > 1)
            clk += MC.ksplit_clk + MC.copy_latency_clk + (double)t.ks * out_bytes / rate +
                   out_bytes / MC.store_bytes_per_clk;
        // Fused tail: park the tile, one more barrier, the first touch of the tail's weights, then the 16x16
        // blocks of the small GEMM dealt over the waves, and the tail's own store.
        if (tail_N > 0) {
            const double blocks = std::ceil((double)ceil_div(tail_N, 16) * (g.PT / 16) / g.waves);
            clk += out_bytes * r / MC.lds_bytes_per_clk + MC.sync_clk + MC.copy_latency_clk +
                   blocks * (g.tail_ng * 32.0 + 64.0) * r + (double)tail_N * g.PT * 4.0 * r / MC.store_bytes_per_clk -
                   out_bytes * r / MC.store_bytes_per_clk;
        }
        return clk;
    };
    if (t.alg == 1 && t.tw == 0) {
        // Winograd over the tiles of the batch: like the register-blocked 1x1 below (the largest of matrix pipes, a wave's
        // own chain of channel groups and the L2, + launch and first operands, + the end of every workgroup, + the memory
        // traffic).  Fitted to 1160 timed tiles of 145 shapes, 7 % mean error, 1.7 % mean loss of the pick within the
        // family.  The factor in front puts the pick between families at the measured crossover, about 6 us: below it the
        // streamed kernels, whose formulas are kind to launches of this length, have the shorter start.
        const double groups = (double)t.cch / (4.0 * t.wk);
        const double wgs_cu = (double)((n_wg + m.cus - 1) / m.cus);
        const double load = std::ceil(wgs_cu * g.waves / m.simds_per_cu);
        const double pipe = groups * (16.0 * t.mb * mfma_clk + 182.0) * load;
        const double chain = groups * (16.0 * t.mb * mfma_clk + 394.0);
        const double l2 = (double)n_wg * groups * (t.wk * t.mb * 4096.0 + g.waves * 1100.0) / std::min<double>(m.cus, (double)n_wg) / 20.2;
        double clk = std::max(std::max(pipe, chain), l2) + 620.0 * t.mb * load;
        if (t.wk > 1) clk += 707.0 + 58.0 * g.waves * t.mb * std::min(wgs_cu, 3.0);
        const double traffic = 4.0 * (d.batch * ((double)d.C * d.H * d.W + (double)d.N * P) + 16.0 * d.C * d.N);
        info.pred_us = 0.85 * (3.12 + clk / (m.clock_ghz * 1e3) + traffic / 4.45e6);
        // (timed beside nb = 1 on 63 shapes of 82 to 1024 channels: 1.05 to 1.06 with four waves, at most 1.12, and 1.00 to 1.025
        //  with eight, which leave the vector instructions of a part more room)
        if (t.nb == 2) info.pred_us *= g.waves > 4 ? 1.02 : 1.06;
        info.pred_l2_bytes = 0.0;
        return true;
    }
    if (is_core_split(t)) {
        // Fitted to 15000 timed tiles of 1000 shapes (most at 3x3 / stride 2): 6 % mean error, 2.5 % mean loss of the pick within the
        // family.  The factor in front: the formula of the staged tiles is 40 % kind in the mean to those it meets.  What a pick by this
        // price gains and loses stands at core_split_takes.
        info.pred_us = 0.86 * split_price(split_core_price, d, t, g, wg_per_cu);
        info.pred_l2_bytes = 0.0;
        return true;
    }
    if (t.alg == 8) {
        // Split operands on the bf16 matrix pipe: the largest of what the matrix pipes, a workgroup's own chain of stages and
        // the L2 need, + LDS reads + the end of every workgroup + launch and memory traffic.  Fitted to 4500 timed tiles of 90
        // 1x1 shapes (6 % mean error, 2.2 % mean loss of the pick within the family) and 4100 tiles of 60 3x3 and 7x7 shapes
        // (6 %, 2.5 %).  The factor in front of the 1x1 and 3x3 forms: as measured, the formulas of the other families are 15 to
        // 25 % kind to the launches this one competes with (7 us and more; most of all those of the staged kernel at stride 2: 128 -> 128
        // @28 batch 32 23.5 us for 34.6, 256 -> 256 @14 22.8 for 41.4), those for the 7x7 stems are not.  At 0.91 no 1x1
        // shape of the 90 loses more than 2 % to its former pick and the mean gain is 9 % (0.85: 10 %, but three lose 8 to 12 %;
        // 1.0: 6 %); the lines fall at 7 to 9 us from 64 channels up, and about 25 us at 3x3 / stride 2.
        const bool flat = t.tw == 0;
        const double wgs = (double)n_wg / m.cus, load = 0.5 * (std::ceil(wgs) + std::max(wgs, 1.0)), rounds = std::ceil(wgs / wg_per_cu);
        const double simd = std::max(1.0, (double)g.waves / m.simds_per_cu), epi = load * g.waves * t.mb * t.nb;
        const double mfmas = (double)g.nchunks * g.ksteps / t.wk * t.mb * t.nb * 6.0 * 16.0;
        const double lds_reads = load * g.waves * g.nchunks * t.nb * 3.0 * 8.0;
        const double traffic = 4.0 * (d.batch * ((double)d.C * d.H * d.W + (double)d.N * P)) + 6.0 * d.C * d.N * g.taps;
        if (flat) {
            const double l2 = (double)n_wg * g.nchunks * (g.waves * t.wm * t.mb * 3072.0 + (double)t.cch * g.PT * 4.0) / std::min<double>(m.cus, (double)n_wg) / 105.9;
            double clk = std::max(std::max(0.807 * load * simd * mfmas, rounds * (1859.0 * g.nchunks + mfmas)), l2);
            clk += 1.443 * lds_reads * (t.wm + 1) + 92.1 * epi;
            if (t.wk > 1) clk += 815.0 + 5.6 * epi;
            info.pred_us = 0.91 * (2.859 + clk / (m.clock_ghz * 1e3) + traffic / 17.67e6);
        } else {
            const bool few = t.cch == 4;
            const double staged = g.nchunks * std::ceil((double)(g.CS << g.oct_shift) / g.threads) * (few ? 0.5 : 1.0);
            double clk = std::max(load * simd * (0.906 * mfmas + 757.0 * staged), rounds * (3232.0 * g.nchunks + 912.0 * staged + 1.164 * mfmas));
            clk += 1.293 * lds_reads * g.ksteps + 181.5 * epi;
            info.pred_us = (few ? 1.0 : 0.85) * (3.527 + clk / (m.clock_ghz * 1e3) + traffic / 15.3e6);
        }
        info.pred_l2_bytes = 0.0;
        return true;
    }
    if (t.alg == 7) {
        // Register-blocked 1x1: the whole launch at once, the largest of what the matrix pipes, a wave's own chain of runs,
        // the address paths and the L2 need, + launch and first operands, + a share of the memory traffic that does not
        // overlap (mostly the stores, which end together).  Fitted to 8000 timed tiles of 190 shapes, 7 % mean error, 1.5 %
        // mean loss of the pick within the family.  The factor in front: the formulas of the other 1x1 families are some
        // 8 % kind to launches of 4 us and more, and the pick between families has to fall at the measured crossover
        // (there, at about 4 us, both run equally fast; at 10 us this one needs 0.8, at 30 us and more 0.6 of the time).
        const double runs = (double)(t.cch / 16 / t.wk), run_clk = 4.0 * t.mb * t.nb * mfma_clk;
        const double wgs_cu = (double)((n_wg + m.cus - 1) / m.cus);
        const double waves_simd = std::max(1.0, (double)n_wg * g.waves / (m.cus * m.simds_per_cu));
        const double waves_simd_most = std::ceil(wgs_cu * g.waves / m.simds_per_cu);
        const double pipe = 1.366 * runs * run_clk * 0.5 * (waves_simd + waves_simd_most);
        const double chain = runs * std::max(run_clk, 396.0);
        const double requests = 18.6 * wgs_cu * g.waves * runs * (t.mb + (g.gen ? 4 * t.nb : 4));
        const double l2 = (double)n_wg * t.wk * runs * (t.wm * t.mb + t.wn * t.nb) * 1024.0 / std::min<double>(m.cus, (double)n_wg) / 29.3;
        double clk = 307.0 + std::max(std::max(pipe, chain), std::max(requests, l2));
        if (t.wk > 1) clk += 232.0 + 20.5 * g.waves * t.mb * t.nb * std::min(wgs_cu, 4.0);
        const double traffic = 4.0 * (d.batch * P * ((double)d.C + d.N) + (double)d.C * d.N);
        info.pred_us = 0.92 * (2.67 + clk / (m.clock_ghz * 1e3) + traffic / 11.95e6);
        // (timed beside tw = 1 on 66 shapes: 1.013 on average, at most 1.07; 1.036, at most 1.09; 1.044, at most 1.11)
        info.pred_us *= t.tw == 32 ? 1.013 : t.tw == 16 ? 1.036 : t.tw == 8 ? 1.044 : 1.0;
        info.pred_l2_bytes = 0.0;   // nothing is staged
        return true;
    }
    const long long slots = (long long)m.cus * wg_per_cu;
    const long long full = n_wg / slots;
    const long long rem = n_wg % slots;
    double clk = (double)full * wg_time(wg_per_cu, slots);
    if (rem) clk += wg_time((int)((rem + m.cus - 1) / m.cus), rem);
    info.pred_us = MC.launch_us + clk / (m.clock_ghz * 1e3);
    info.pred_l2_bytes = (double)n_wg * g.cps * copy_bytes_pass;
    return true;
}

std::vector<tdc_tile> model_enumerate(const tdc_conv_desc &d, int tail_N) {
    std::vector<tdc_tile> out;
    if (!check_desc(d, nullptr)) return out;
    const bool flat = (d.KH == 1 && d.KW == 1 && d.stride == 1 && d.pad == 0);
    const int He = flat ? 1 : d.H, We = flat ? d.H * d.W : d.W;
    const int Ho = (He + 2 * d.pad - d.dilation * (d.KH - 1) - 1) / d.stride + 1;
    const int Wo = (We + 2 * d.pad - d.dilation * (d.KW - 1) - 1) / d.stride + 1;
    const int P = Ho * Wo;
    static const int mfs[] = {16, 32};
    static const int wks[] = {1, 2, 4, 8, 16};
    static const int wms[] = {1, 2, 4};
    static const int wns[] = {1, 2, 4};
    // streamed 1x1 candidates: the input channels in runs of 16, 1, 2, 4 or 8 runs per wave
    if (d.KH == 1 && d.KW == 1 && d.pad == 0 && tail_N == 0 && !std::getenv("TDC_EXPERIMENT_NO_STREAMED_1X1")) {
        // (a split of the input channels over ks workgroups only where the layer leaves most of the chip idle)
        for (int ks : {1, 2, 4, 8}) {
            if (ks > 1 && !flat) break;
            const int runs = ceil_div(ceil_div(d.C, ks), 16);
            for (int per_wave : {8, 4, 2, 1}) {
                if (per_wave > runs) continue;   // (more than half of such a wave's channels would be padding)
                const int wk = ceil_div(runs, per_wave);
                if (wk > 16) continue;
                tdc_tile t{16, 1, 1, 1, 1, wk, 16 * per_wave * wk, std::min(16, P), ks, 0, 3};
                Geometry g;
                if (!make_geometry(d, t, g, nullptr, 0)) continue;
                if (ks > 1 && (long long)g.grid_x * g.grid_y * g.grid_z > 2LL * machine().cus) continue;
                out.push_back(t);
            }
        }
    }
    // split-operand candidates (bf16 matrix pipe); below 0.1 and 0.3 GFLOP (1x1, larger filters) they never came within 10 % of the
    // other families, which have the shorter start
    const bool one = d.KH == 1 && d.KW == 1;
    const double flops = 2.0 * d.batch * P * d.C * d.N * d.KH * d.KW;
    if (tail_N == 0 && flops >= (one ? 1e8 : 3e8) && !(one && (d.stride != 1 || d.pad != 0)) && !std::getenv("TDC_EXPERIMENT_NO_SPLIT")) {
        const bool few = d.C <= 4 && d.dilation == 1 && d.stride % 2 == 0;
        auto offer = [&](const tdc_tile &t) {
            Geometry g;
            if (make_geometry(d, t, g, nullptr, 0)) out.push_back(t);
        };
        std::vector<int> tws;
        for (int tw : {Wo, ceil_div(Wo, 2), ceil_div(Wo, 4), 8, 16, 32, 64})
            if (tw <= Wo && std::find(tws.begin(), tws.end(), tw) == tws.end()) tws.push_back(tw);
        for (int mb : {1, 2, 4})
            for (int wm : {1, 2, 4, 8})
                for (int wn : {1, 2, 4, 8}) {
                    if (wm * wn > 8 || 16 * mb * wm > round_up(d.N, 16 * mb)) continue;
                    if (one) {
                        for (int nb : {2, 4})
                            for (int wk : {1, 2, 4, 8})
                                if (mb <= 2 && (wm * wn * wk == 4 || wm * wn * wk == 8)) offer({16, mb, nb, wm, wn, wk, 32 * wm * wk, 0, 1, 0, 8});
                    } else if (wm * wn >= 4) {
                        for (int tw : tws)
                            for (int cch : {4, 8, 16, 32})
                                if ((cch == 4) == few && cch < 2 * d.C + 8) offer({16, mb, 4, wm, wn, 1, cch, tw, 1, 0, 8});
                    }
                }
        if (!one && d.C >= 32 && flops < 2.5e10) {
            // The form of 32 pixels per wave, for the layers its price was fitted on: up to 25 Gflop, above which it is the cheaper tile
            // for 62 of 2800 random layers (20 to 120 Gflop) and takes 0.57 to 1.10 of their time, 0.89 in the mean; five are 2 to 10 %
            // slower.  Under 32 channels its sums are no more accurate than those of 64 pixels per wave.
            for (int mb : {1, 2, 4})
                for (int wm : {1, 2, 4, 8})
                    for (int wn : {1, 2, 4})
                        for (int wk : {1, 2, 4}) {
                            if ((wm * wn * wk != 4 && wm * wn * wk != 8) || 16 * mb * wm > round_up(d.N, 16 * mb)) continue;
                            std::vector<int> widths;
                            for (int tw : {Wo, ceil_div(Wo, 2), ceil_div(Wo, 4), 8, 16}) {
                                if (tw > std::min(Wo, 32 * wn) || std::find(widths.begin(), widths.end(), tw) != widths.end()) continue;
                                const double rows = (double)d.batch * Ho, th = std::min(32.0 * wn / tw, rows);
                                if (rows * Wo >= 0.7 * 32 * wn * std::ceil(rows / std::floor(th)) * ceil_div(Wo, tw)) widths.push_back(tw);
                            }
                            for (int tw : widths)
                                for (int cch : {8, 16, 32, 64, 128})
                                    if (cch < 2 * d.C + 8 && (cch >= 32 || cch >= d.C)) offer({16, mb, 2, wm, wn, wk, cch, tw, 1, 0, 8});
                        }
        }
    }
    // register-blocked 1x1 candidates
    if (d.KH == 1 && d.KW == 1 && d.pad == 0 && tail_N == 0 && !std::getenv("TDC_EXPERIMENT_NO_BLOCKED_1X1")) {
        for (int mb : {1, 2})
            for (int nb : {2, 4})
                for (int wm : wms)
                    for (int wn : wns)
                        for (int wk : {1, 2, 4, 8}) {
                            // (the waves of a workgroup of two share a pair of SIMDs with those of the next one)
                            if (wm * wn * wk > 8 || wm * wn * wk == 2 || 16 * mb * wm > round_up(d.N, 16 * mb)) continue;
                            tdc_tile t{16, mb, nb, wm, wn, wk, round_up(d.C, 16 * wk), 1, 1, 0, 7};
                            Geometry g;
                            if (!make_geometry(d, t, g, nullptr, 0)) continue;
                            out.push_back(t);
                            // (the same with its sums in parts, where a wave has more channels than one of them; from 128 channels on
                            //  parts of 8 are too many to have the smaller error)
                            for (int part : {32, 16, 8})
                                if (t.cch / wk > part && t.cch / wk < 16 * part) {
                                    t.tw = part;
                                    out.push_back(t);
                                }
                        }
    }
    // streamed 3x3 candidates: 1, 2 or 4 groups of four channels per wave, a few shapes of the 16-pixel tile
    if (d.KH == 3 && d.KW == 3 && d.dilation == 1 && !std::getenv("TDC_EXPERIMENT_NO_STREAMED_3X3")) {
        std::vector<int> tws;
        for (int tw : {16, 14, 8, 7, 4, std::min(16, Wo)}) {
            if (tw > std::min(16, Wo) || std::find(tws.begin(), tws.end(), tw) != tws.end()) continue;
            const int th = std::min(16 / tw, Ho);
            const double util = (double)P / ((double)ceil_div(Wo, tw) * ceil_div(Ho, th) * 16);
            if (util < 0.6 && tw != std::min(16, Wo)) continue;
            tws.push_back(tw);
        }
        // (a fused tail needs every output channel in the workgroup: one wave per block of 16 and channel slice)
        const int wm = tail_N > 0 ? ceil_div(d.N, 16) : 1;
        for (int ks : {1, 2, 4, 8}) {
            if (ks > 1 && tail_N > 0) break;
            const int groups_slice = ceil_div(ceil_div(d.C, ks), 4);
            for (int per_wave : {4, 2, 1}) {
                if (per_wave > groups_slice) continue;
                const int wk = ceil_div(groups_slice, per_wave);
                if (wm * wk > 16) continue;
                for (int tw : tws) {
                    tdc_tile t{16, 1, 1, wm, 1, wk, 4 * per_wave * wk, tw, ks, 0, 4};
                    Geometry g;
                    if (!make_geometry(d, t, g, nullptr, tail_N)) continue;
                    if (ks > 1 && (long long)g.grid_x * g.grid_y * g.grid_z > 2LL * machine().cus) continue;
                    out.push_back(t);
                    // the same tile with its input window loaded in 128-bit pieces and passed through LDS
                    if (d.pad <= 1 && d.stride <= 2 && !std::getenv("TDC_EXPERIMENT_NO_STREAMED_WINDOW")) {
                        tdc_tile t6 = t;
                        t6.alg = 6;
                        if (make_geometry(d, t6, g, nullptr, tail_N)) out.push_back(t6);
                    }
                    // the same tile with 2 or 4 neighbouring 14-pixel row tiles per workgroup, sharing the weights in
                    // registers (where the image row has that many)
                    if (tw == 14 && d.stride == 1 && ks == 1 && tail_N == 0 && !std::getenv("TDC_EXPERIMENT_NO_STREAMED_NB"))
                        for (int nb : {2, 4}) {
                            if (ceil_div(Wo, 14) < nb) continue;
                            t.nb = nb;
                            if (make_geometry(d, t, g, nullptr, 0) &&
                                kernel_id_for(t, 3, 3, 1, 1, false, false).family != KernelId::NONE)
                                out.push_back(t);
                            // ... and with the rows of all blocks loaded as one window through LDS
                            if (d.pad <= 1 && !std::getenv("TDC_EXPERIMENT_NO_STREAMED_WINDOW")) {
                                tdc_tile t6 = t;
                                t6.alg = 6;
                                if (make_geometry(d, t6, g, nullptr, 0) &&
                                    kernel_id_for(t6, 3, 3, 1, 1, false, false).family != KernelId::NONE)
                                    out.push_back(t6);
                            }
                        }
                }
            }
        }
    }
    // streamed Winograd candidates: 3x3 / stride 1 / pad 1, even width, all input channels in one pass.  Offered for single
    // images only: the kernel is built for the latency of one small launch, and at batch 8 its timing alone misleads the
    // measured selection (DenseNet-121's 64 -> 16 @56x56 core at batch 8: 6.9 us alone against 8.1 us for the staged
    // Winograd tile, but the network ran 2.5 % slower with it); a forced tile still runs any batch.
    if (d.batch == 1 && d.KH == 3 && d.KW == 3 && d.stride == 1 && d.dilation == 1 && d.pad == 1 && d.W % 2 == 0 && tail_N == 0 &&
        !std::getenv("TDC_EXPERIMENT_NO_STREAMED_WINOGRAD")) {
        const int groups_total = ceil_div(d.C, 4);
        for (int wm : {1, 2}) {
            if (16 * wm > round_up(d.N, 16)) continue;
            for (int per_wave : {4, 3, 2, 1}) {
                if (per_wave > groups_total) continue;
                const int wk = ceil_div(groups_total, per_wave);
                if (wm * wk > wino_stream_max_waves(per_wave)) continue;
                if (per_wave * wk - groups_total >= per_wave) continue;   // an idle wave
                tdc_tile t{16, 1, 1, wm, 1, wk, 4 * per_wave * wk, 28, 1, 0, 5};
                Geometry g;
                if (make_geometry(d, t, g, nullptr, 0)) out.push_back(t);
            }
        }
    }
    // Winograd over the tiles of the whole batch: batches, and single images of more than 64x64 pixels (224x224 17.3 -> 15.0
    // us, 96x96 14.6 -> 12.4; at 56x56 the streamed Winograd kernel is as fast).
    const bool wino_batch = (d.batch > 1 || P > 4096) && d.KH == 3 && d.KW == 3 && d.stride == 1 && d.dilation == 1 && d.pad <= 1 &&
                            d.H * d.W >= 8 && tail_N == 0 && !std::getenv("TDC_EXPERIMENT_NO_WINOGRAD");
    if (wino_batch)
        for (int mb : {1, 2})
            for (int wn : {2, 4})
                for (int wk : {1, 2, 4}) {
                    if (wn * wk > 8 || wn * wk < 4 || 16 * mb > round_up(d.N, 16)) continue;
                    tdc_tile t{16, mb, 1, 1, wn, wk, round_up(d.C, 8 * wk), 0, 1, 0, 1};
                    Geometry g;
                    if (!make_geometry(d, t, g, nullptr, 0)) continue;
                    // (32 channels x 32 tiles, the weights shared by two waves only: deep layers of small images, whose
                    //  workgroups fit the chip at once; 256 -> 256 @7 batch 64 25.8 us against 28.2)
                    if (mb == 2 && wn == 2 && (wk < 4 || g.grid_x * g.grid_y > machine().cus)) continue;
                    out.push_back(t);
                    // (the same with its sums in parts of eight steps, where there are several)
                    t.nb = 2;
                    if (t.cch / (8 * wk) > 10 && make_geometry(d, t, g, nullptr, 0)) out.push_back(t);
                }
    // Winograd candidates for 3x3 / stride 1 convolutions with enough pixels to fill tile lanes.  Batches keep them beside the
    // tiles above: those stop where batch * tiles * tiles reaches 2^32 (224x224 from 28 images, 512x512 from one), and deep
    // layers with few output channels are cheaper with eight waves over channels.
    if (d.KH == 3 && d.KW == 3 && d.stride == 1 && d.dilation == 1 && tail_N == 0 && !std::getenv("TDC_EXPERIMENT_NO_WINOGRAD")) {
        const int Wt = ceil_div(Wo, 2), Ht = ceil_div(Ho, 2);
        for (int wm : wms)
            for (int wn : wns)
                for (int wk : wks) {
                    if (wm * wn * wk > 8) continue;
                    if (16 * wm > round_up(d.N, 16)) continue;
                    const int lanes = 16 * wn;
                    if (lanes > round_up(Wt * Ht, 16)) continue;
                    std::vector<int> tws;
                    for (int tw = 1; tw <= std::min(Wt, lanes); ++tw) {
                        const bool pow2 = (tw & (tw - 1)) == 0;
                        const bool widest = (tw == std::min(Wt, lanes));
                        if (!(widest || (pow2 && tw >= 2) || (Wt % tw == 0 && tw >= 2))) continue;
                        const int th = std::min(lanes / tw, Ht);
                        const double util = (double)(Wt * Ht) / ((double)ceil_div(Wt, tw) * ceil_div(Ht, th) * lanes);
                        if (util < 0.7 && !widest) continue;
                        tws.push_back(tw);
                    }
                    const int granule = 4 * wk;
                    std::vector<int> cchs;
                    for (int div : {1, 2, 4, 8}) {
                        const int cch = round_up(ceil_div(d.C, div), granule);
                        if (std::find(cchs.begin(), cchs.end(), cch) == cchs.end()) cchs.push_back(cch);
                    }
                    for (int fixed : {16, 32})
                        if (fixed % granule == 0 && fixed < round_up(d.C, granule) &&
                            std::find(cchs.begin(), cchs.end(), fixed) == cchs.end())
                            cchs.push_back(fixed);
                    const long long max_wgs = 4LL * machine().cus;
                    for (int tw : tws)
                        for (int cch : cchs)
                            for (int ks : {1, 2, 4})
                                for (int wl : {0, 2, 4}) {
                                    tdc_tile t{16, 1, 1, wm, wn, wk, cch, tw, ks, wl, 1};
                                    Geometry g;
                                    if (!make_geometry(d, t, g, nullptr, 0)) continue;
                                    if (ks > 1 && (long long)g.grid_x * g.grid_y * g.grid_z > max_wgs) continue;
                                    if (wl > 0 && g.cps < 2) continue;
                                    out.push_back(t);
                                }
                }
    }
    const bool global_weights = d.KH == 3 && d.KW == 3 && d.dilation == 1 && tail_N == 0 &&
                                !std::getenv("TDC_EXPERIMENT_NO_GLOBAL_WEIGHTS");
    for (int mf : mfs) {
        const int kc = (mf == 32) ? 2 : 4;
        for (int mb = 1; mb <= 2; ++mb)
            for (int nb = 1; nb <= 2; ++nb)
                for (int wm : wms)
                    for (int wn : wns)
                        for (int wk : wks) {
                            const int maxw = (mb == 2 && nb == 2) ? 8 : 16;
                            if (wm * wn * wk > maxw) continue;
                            if (mf * mb * wm > round_up(d.N, mf)) continue;  // do not tile past the problem
                            const int PT = mf * nb * wn;
                            if (PT > round_up(P, mf)) continue;
                            // Tile widths: the whole row, and power-of-two or exact-divisor widths
                            // that keep at least 70 % of the pixel lanes on real pixels.
                            std::vector<int> tws;
                            for (int tw = 1; tw <= std::min(Wo, PT); ++tw) {
                                const bool pow2 = (tw & (tw - 1)) == 0;
                                const bool widest = (tw == std::min(Wo, PT));
                                if (flat && !widest) continue;  // one row of pixels: nothing to gain from narrower runs
                                if (!(widest || (pow2 && tw >= 4) || (Wo % tw == 0 && tw >= 4))) continue;
                                const int th = std::min(PT / tw, Ho);
                                const double util = (double)P / ((double)ceil_div(Wo, tw) * ceil_div(Ho, th) * PT);
                                if (util < 0.7 && !widest) continue;
                                tws.push_back(tw);
                            }
                            const int granule = kc * wk;
                            const int c_full = round_up(d.C, granule);
                            std::vector<int> cchs;
                            for (int div : {1, 2, 4, 8}) {
                                const int cch = round_up(ceil_div(d.C, div), granule);
                                if (std::find(cchs.begin(), cchs.end(), cch) == cchs.end()) cchs.push_back(cch);
                            }
                            for (int fixed : {16, 32})
                                if (fixed % granule == 0 && fixed < c_full &&
                                    std::find(cchs.begin(), cchs.end(), fixed) == cchs.end())
                                    cchs.push_back(fixed);
                            // Splitting the passes over several workgroups only pays while the
                            // layer has fewer tiles than the chip has room for.
                            const long long max_wgs = 4LL * machine().cus;
                            for (int tw : tws)
                                for (int cch : cchs)
                                    for (int ks : {1, 2, 4, 8})
                                        for (int wl : {0, 1, 2, 4}) {
                                            tdc_tile t{mf, mb, nb, wm, wn, wk, cch, tw, ks, wl, 0};
                                            Geometry g;
                                            if (!make_geometry(d, t, g, nullptr, tail_N)) continue;
                                            if (ks > 1 && (long long)g.grid_x * g.grid_y * g.grid_z > max_wgs) continue;
                                            if (wl > 0 && g.cps < 2) continue;  // loaders only work from the second pass on
                                            out.push_back(t);
                                            // the same tile with its weights read from global memory
                                            if (global_weights && mb == 1 && nb == 1) {
                                                t.alg = 2;
                                                if (make_geometry(d, t, g, nullptr, 0)) out.push_back(t);
                                            }
                                        }
                        }
    }
    // (the other families' addressing limits hold for the library as a whole: a shape that none of them takes is refused)
    if (std::all_of(out.begin(), out.end(), [](const tdc_tile &t) { return t.alg == 8; })) out.clear();
    return out;
}

int model_constants(double *out, int cap) {
    std::shared_lock<std::shared_mutex> lock(MC_mutex);
    for (int i = 0; i < kNumModelConst && i < cap; ++i) out[i] = *mc_field(i);
    return kNumModelConst;
}

bool model_set_constants(const double *in, int n) {
    if (n != kNumModelConst) return false;
    for (int i = 0; i < n; ++i)
        if (!(in[i] > 0.0)) return false;
    std::unique_lock<std::shared_mutex> lock(MC_mutex);
    for (int i = 0; i < n; ++i) *mc_field(i) = in[i];
    return true;
}

// The price of a staged Winograd tile stands too low against the tiles over the whole batch, except where its workgroups have
// a compute unit each and eight slices of the input channels, or where four workgroups share those.  Timed against the best
// other tile, 126 shapes where its price is the lowest: outside of these two 1.21 times as long on average (up to 2.2 times),
// inside 0.85 of the time (0.65 to 1.13).
static double staged_winograd_handicap(const tdc_tile_info &info) {
    const tdc_tile &t = info.tile;
    if (t.alg != 1 || t.tw == 0) return 1.0;
    const long long n_wg = (long long)info.grid_x * info.grid_y * info.grid_z;
    return t.wl == 0 && (t.ks >= 4 ? t.wk >= 4 : t.wk >= 8 && n_wg <= machine().cus) ? 1.0 : 1.35;
}

// Expected square of an output's rounding error, in units of one rounding of the whole sum: partial sums grow along a chain of
// `chain` of the n products, which costs chain / 2, and n / chain chains are added up.  The transforms of Winograd weigh its
// products 2.84 times and add 13.4.  Measured against 64-bit sums with 534 shapes and tiles: 2.5e-8 times the
// root of this within 10 % (all but 4 % of them; extremes 0.85 and 1.17), input and weights from symmetric distributions.
static double rounding_variance(const tdc_conv_desc &d, const tdc_tile &t) {
    const bool wino = t.alg == 1 || t.alg == 5;
    const double n = wino ? d.C : (double)d.C * d.KH * d.KW;
    double chain = n / ((double)t.wk * t.ks);
    if (t.alg == 3) chain = 0.5 * std::min((double)t.cch / t.wk, n);          // (two accumulators)
    if (t.alg == 7 || (t.alg == 1 && t.tw == 0)) chain = std::min((double)t.cch / t.wk, n);
    double parts = 1.0;                                          // ... of a wave's sum
    if (t.alg == 1 && t.tw == 0 && t.nb == 2) parts += std::max(t.cch / (8 * t.wk) - 3, 0) / 8;   // (one ends every eight steps but for the last two)
    if (t.alg == 7 && t.tw > 1) parts = std::max(chain / t.tw, 1.0);
    if (parts > 1.0) {
        const double v = 0.5 * (chain / parts + parts + t.wk - 1);
        return wino ? 2.84 * v + 13.4 : v;
    }
    if ((t.alg == 4 || t.alg == 6) && t.nb == 1) chain *= 0.5;   // (likewise)
    const double v = 0.5 * (chain + n / (chain * t.ks) + (t.ks - 1));
    return wino ? 2.84 * v + 13.4 : v;
}

// The tiles a pick is made from.  Where the tiles of the other families would take a direct kernel with short chains (several
// waves share few input channels), Winograd over the tiles of the whole batch is faster, 0.6 to 0.9 of the time, but its error
// is up to 1.7 times as large (16 -> 112 @12 batch 48 0.9e-7 -> 1.5e-7), and with more input channels per chain than the staged
// Winograd tile 1.4 times (128 -> 32 @105 batch 8 2.6e-7 -> 3.5e-7).  So is that of the register-blocked 1x1 kernel, up to 2.7 times
// (304 -> 176 @53 1.1e-7 -> 3.1e-7 against five waves of 64 channels).  They are taken only where their error is no larger than
// that of the tile they take the place of.
// (Prices and places in `tiles` only: ten thousand tdc_tile_info cost a third of the time of a selection.)
struct Choice {
    int tile;
    double us, handicap;
};
static std::vector<Choice> choices_within(const tdc_conv_desc &d, int tail_N, const std::vector<tdc_tile> &tiles, double &limit) {
    auto batched = [](const tdc_tile &t) { return t.alg == 7 || (t.alg == 1 && t.tw == 0); };
    std::vector<Choice> choices;
    choices.reserve(tiles.size());
    int plain = -1;
    double plain_us = 0.0;
    for (int i = 0; i < (int)tiles.size(); ++i) {
        tdc_tile_info info;
        if (!model_evaluate(d, tiles[i], info, nullptr, tail_N)) continue;
        choices.push_back({i, info.pred_us, staged_winograd_handicap(info)});
        if (batched(tiles[i]) || tiles[i].alg >= 7 || (plain >= 0 && info.pred_us >= plain_us)) continue;
        plain = i;
        plain_us = info.pred_us;
    }
    limit = plain >= 0 ? 1.06 * rounding_variance(d, tiles[plain]) : 0.0;   // (3 % of the error: where channels are padded to whole steps)
    choices.erase(std::remove_if(choices.begin(), choices.end(), [&](const Choice &c) { return batched(tiles[c.tile]) && rounding_variance(d, tiles[c.tile]) > limit; }), choices.end());
    return choices;
}
std::vector<tdc_tile_info> model_choices(const tdc_conv_desc &d, int tail_N) {
    double limit;
    const std::vector<tdc_tile> tiles = model_enumerate(d, tail_N);
    std::vector<tdc_tile_info> infos;
    for (const Choice &c : choices_within(d, tail_N, tiles, limit)) {
        infos.emplace_back();
        if (!model_evaluate(d, tiles[c.tile], infos.back(), nullptr, tail_N)) infos.pop_back();
    }
    return infos;
}

// Whether the split-operand form of 32 pixels per wave, the cheaper one by price, takes the place of the best other tile.  Timed in turn
// with the tile it would displace, over the 3252 of 20400 random layers (2x2 to 7x7, strides 1 to 3, dilation 2; batch 1 to 64, 16 to
// 1024 channels, 0.3 to 25 Gflop) where that price is the lower one:
//   staged direct tiles (1492 layers): 0.74 of their time in the mean; 41 are more than 2 % slower, up to 16 %, most of them at 10 to 14 us,
//     and no limit on the price or the length of a launch parts those from more than three times as many that gain.
//   the form of 64 pixels per wave (1683): 0.96, but 408 are slower, up to 38 %: one stage only, or eight waves that share no K-steps, or
//     a launch that the larger tiles fill better.  The two formulas are 7 % apart in what they make of such pairs; so this choice goes by one
//     formula fitted to 3800 and 1800 timed tiles of both (5 %), and the new form has to be 2 % lower: it takes 1065 of the layers at 0.92
//     of their time, 43 of them more than 2 % slower (up to 19 %), and leaves 618, on which it would need 1.045.
//   streamed and Winograd tiles (77): 0.985, 29 slower, up to 22 %: left alone.
// The error against 64-bit sums is at most 0.97 of that of the tile displaced.
static bool core_split_takes(const tdc_conv_desc &d, const tdc_tile &core, const tdc_tile &other) {
    if (other.alg == 0 || other.alg == 2) return true;
    if (other.alg != 8) return false;
    static const SplitPrice of_core = {0.0, 197.3, 138.8, 934.7, 3074, 1993, 2116, 34.23, 0.101, 0.0, 1.432, 2.812, 37.84, 1.517, 0.2695, 0.6759, 0.1105};
    static const SplitPrice of_other = {0.0, 211.6, 763.8, 635.5, 0.0, 3036, 1168, 294.7, 0.7946, 231.1, 2.445, 3.297, 45.78, 2.322, 0.4946, 0.6586, 0.1059};
    auto price = [&](const SplitPrice &q, const tdc_tile &t) {
        Geometry g;
        tdc_tile_info info;
        make_geometry(d, t, g, nullptr, 0);
        model_evaluate(d, t, info, nullptr, 0);
        return split_price(q, d, t, g, info.wg_per_cu);
    };
    return price(of_core, core) < 0.98 * price(of_other, other);
}

bool model_select(const tdc_conv_desc &d, tdc_tile_info &best, std::string *why, int tail_N) {
    if (!check_desc(d, why)) return false;
    double limit;
    const std::vector<tdc_tile> tiles = model_enumerate(d, tail_N);
    const std::vector<Choice> cands = choices_within(d, tail_N, tiles, limit);
    const bool batched = std::any_of(cands.begin(), cands.end(), [&](const Choice &c) { return tiles[c.tile].alg == 1 && tiles[c.tile].tw == 0; });
    const Choice *pick = nullptr, *core = nullptr;
    double best_us = 0.0;
    for (const Choice &c : cands) {
        if (is_core_split(tiles[c.tile])) {
            if (!core || c.us < core->us) core = &c;
            continue;
        }
        // (the handicap takes the pick from a staged tile, but not to a kernel with a larger error)
        if (batched && tiles[c.tile].alg < 7 && rounding_variance(d, tiles[c.tile]) > limit) continue;
        const double us = c.us * (batched ? c.handicap : 1.0);
        if (!pick || us < best_us) {
            pick = &c;
            best_us = us;
        }
    }
    if (core && (!pick || (core->us < best_us && core_split_takes(d, tiles[core->tile], tiles[pick->tile])))) pick = core;
    const bool have = pick && model_evaluate(d, tiles[pick->tile], best, nullptr, tail_N);
    if (!have && why) {
        // say why the plainest tile cannot be launched: that is the limit the shape runs into
        const tdc_tile plain{16, 1, 1, 1, 1, 1, 4, 1, 1, 0, 0};
        Geometry g;
        std::string reason;
        *why = make_geometry(d, plain, g, &reason, tail_N) ? "no launchable tile for this shape"
                                                             : "no launchable tile for this shape: " + reason;
    }
    return have;
}

}  // namespace tdc
