// fp32 convolution on the bf16 matrix pipe (tile.alg = 8, tdc_conv_split_kernel).
#include "conv_device.hpp"
#include "conv_split_device.hpp"

namespace tdc {

// ---------------------------------------------------------------------------
// Every operand is split into three bf16 parts that add up to the fp32 value, and a product is the sum of the six partial
// products above 2^-24: v_mfma_f32_16x16x32_bf16 does 16 times the multiplications of v_mfma_f32_16x16x4_f32, so six of
// them still are 2.7 times as fast.  The leading products (h0*h0) have an accumulator of their own and the five small ones
// share a second one; the matrix core adds 32 products per rounding, and the error against 64-bit sums is 0.3 to 0.45 of
// that of a chain of fp32 MFMAs (K = 32 ... 2048: 3.6e-8 ... 2.5e-7 against 1.0e-7 ... 8.0e-7; with one accumulator for
// all six 3.6e-8 ... 6.9e-7).
// A workgroup is WM x WN waves over 16*MB channels x 64 pixels each.  Input channels pass through LDS in octets, split once
// per workgroup: [part][octet][pixel] x 16 bytes, which is one B operand register quad per lane; weights are split and
// packed by the host in A order and come straight from memory.
//   SPLIT_FLAT    1x1 / stride 1: the pixels of the batch in quads; a lane loads 8 channels of one quad as eight 128-bit
//                 requests, a stage (32*WM channels) ahead of the MFMAs.  Pixel e of quad q has slot e*16*WN + q, so the
//                 four blocks of a wave are the four pixels of its lanes' quads: 128-bit stores.
//   SPLIT_WINDOW  any filter: tiles of TH output rows (counted through the batch) x TW columns; the input window of 8*NO
//                 channels is staged and the K-steps run over its (tap, octet) pairs.  At stride 2 the even and the odd
//                 columns lie in separate halves of a row, so neighbouring lanes read neighbouring slots.
//   SPLIT_FEW     at most four input channels (RGB stems): 8 bytes per pixel, a K octet is a pair of neighbouring taps.
// Infinite and NaN operands (and finite ones above 3.39e38) make the split invalid: an infinity less itself is NaN.  Sums near
// 3.4e38 can overflow in the leading product alone.  Operands below 2^-110 lose their last bits, because bf16 has no subnormals
// under 2^-133.  A wave that finds an infinity or a NaN among its sums, or one under 2^-90 other than zero, computes plain fp32 sums
// of the unsplit operands for the block that holds it (direct_block) and takes those for the sums in question: 512 -> 128 @28
// batch 32 takes 28 us, with one NaN pixel 79, with nothing but NaN or sums below 2^-90 296 (out of scalar fp32 sums for every output
// of such a wave 1600 and 3200).  Channels of very small or very large weights are packed times a power of two
// (pack_split_weights) and their sums multiplied by p.w_scale.
// A sum of 2^-90 or more bears the lost bits of an operand below 2^-110 only while its partner stays under 2^20, and a zero may
// stand for parts that all vanished.  So the threads note the inputs of either kind (Extremes) and the host the channels with
// weights below 2^-110 (a negative factor): in question are also zeros where a tiny input or weight took part, sums of channels
// packed down with a tiny input, and sums of channels with tiny weights beside a large input.  The look at every
// input takes 0.5 to 2.5 % (512 -> 128 @28 batch 32 27.9 -> 28.5 us, 3x3 / stride 2 128 -> 128 @56 batch 64 98.6 -> 98.9, stem batch 32
// 78.5 -> 79.9); one tiny pixel 28.7 us, a weight of 1e-40 in every channel 31.  That some factor is not 1 is looked at behind the
// last stage: waiting for it in front of the first one, behind weights that come from memory, cost the networks 0.8 %.
// AFF: per-channel affine (+ ReLU) on the input of a 1x1 convolution.
// Bound: no single one.  512 -> 128 @28 batch 32 takes 26 us: 9 us of MFMAs at the 390 TFLOP/s of fp32 products that a bare MFMA
// loop reaches, 13 us of memory traffic, and between them LDS reads (a half of the MFMA time at mb = 2), the splitting (5
// vector operations an element) and two barriers a stage, which two to four waves per SIMD overlap only in part.
// Against the best tile of the other families (launch-to-launch, one box, us): 512 -> 128 @28 batch 32 38 -> 26, 128 -> 512 @28
// batch 32 46 -> 28, 256 -> 2048 @7 batch 64 44 -> 28, 2048 -> 256 @7 batch 64 43 -> 32, 976 -> 866 @40 batch 5 138 -> 85, 256 -> 128
// @56 batch 8 23 -> 16; 7x7 / stride 2 stem 3 -> 64 @224 batch 32 121 -> 78, batch 8 36.7 -> 26.5; 3x3 / stride 2 218 -> 124 @90 batch 27
// 338 -> 176, 128 -> 128 @56 batch 64 164 -> 101, 64 -> 64 @56 batch 32 30 -> 23.  Not faster where a launch takes under 7 us, and
// at 3x3 / stride 1, where Winograd saves more (128 -> 128 @56 batch 64 274 us against 267).
// Not kept: requesting weights four blocks ahead and pixel operands one K-step ahead (0 to 10 % slower: fewer waves fit);
// 64 channels x 32 pixels per wave in the 1x1 form (best nowhere by more than 3 %, often 10 % behind); four channel blocks with the
// weights reloaded in place a K-step ahead and the six products of a K-step from zero (218 -> 124 @90 / stride 2 batch 27 162 -> 165,
// 256 -> 256 @56 / stride 2 batch 40 177 -> 176, networks with the stem unchanged).
// ---------------------------------------------------------------------------
enum : int { SPLIT_FLAT = 0, SPLIT_WINDOW = 1, SPLIT_FEW = 2 };

template <int MB, int NB, int MODE, bool AFF>
__global__ void __launch_bounds__(512, 2) tdc_conv_split_kernel(const ConvKParams p) {
    using G = PixelGroup<NB>;
    using px_t = typename G::reg_t;
    extern __shared__ __align__(16) float lds_all[];
    float *const lds = lds_all + EXTREMES_FLOATS;
    touch_kernel_arguments();
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int logical = (int)(blockIdx.x & 7u) * p.xcd_chunk + (int)(blockIdx.x >> 3);
    if (logical >= p.n_wg) return;
    const int q1 = fdiv(logical, p.fd_g1);
    const int r1 = logical - q1 * p.fd_g1.d;
    const int bx = p.channel_major ? r1 : q1;   // pixel tile
    const int by = p.channel_major ? q1 : r1;   // channel tile
    const int t1 = MODE == SPLIT_FLAT ? fdiv(wave, p.fd_wk) : wave;
    const int slice = MODE == SPLIT_FLAT ? wave - t1 * p.WK : 0;   // of the input channels of a stage
    const int wm = fdiv(t1, p.fd_wn);
    const int wn = t1 - wm * p.WN;
    const int k = lane >> 4, n = lane & 15;
    const int threads = 64 * p.WM * p.WN;
    const unsigned HW4 = (unsigned)(p.H * p.W) * 4u;
    // (see Geometry) slots per output column, octets per stage as a power of two, K-steps per stage
    const int ss = p.slots_col, no_shift = p.oct_shift, ksteps = p.ksteps, half = p.odd_columns;

    // first unit (group of NB pixels / output row) and first image of the workgroup; column tile of a window
    const int ty = MODE == SPLIT_FLAT ? bx : fdiv(bx, p.fd_ntx);
    const int tx = MODE == SPLIT_FLAT ? 0 : bx - ty * p.ntx;
    const int u0 = MODE == SPLIT_FLAT ? bx * 16 * p.WN : ty * p.TH;
    const int b0 = fdiv(u0, p.fd_units);
    const int first = u0 - b0 * p.fd_units.d;   // ... within its image

    const __amdgpu_buffer_rsrc_t in_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(p.in + (long long)b0 * p.in_bstride), (short)0, OOB_OFFSET, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.wpk), (short)0, (int)p.wpk_bytes, 0x00020000);

    // ---- the pixels a lane finishes: block j -----------------------------------------------------------------------------
    struct Pixel {
        int img, pix;      // image and pixel offset within an output plane
        int fresh;         // FLAT: first pixel of the group that no other group stores; else 0 = stored, 1 = not
        int slot;          // LDS slot of tap 0
    };
    auto pixel = [&](int j) {
        Pixel r;
        if constexpr (MODE == SPLIT_FLAT) {
            const int u = u0 + wn * 16 + n;
            const int uc = min(u, p.units - 1);
            r.img = fdiv(uc, p.fd_units);
            const int g = uc - r.img * p.fd_units.d;
            r.pix = min(NB * g, p.P - NB);
            r.fresh = u < p.units ? NB * g - r.pix : NB;
            r.slot = j * (16 * p.WN) + wn * 16 + n;
        } else {
            const int q = (wn * NB + j) * 16 + n;
            const int row = fdiv(q, p.fd_tw);
            const int col = q - row * p.TW;
            const int ox = tx * p.TW + col;
            const bool ok = row < p.TH && u0 + row < p.units && ox < p.Wo;
            const int g = min(u0 + row, p.units - 1);
            r.img = fdiv(g, p.fd_units);
            const int oy = g - r.img * p.fd_units.d;
            r.pix = oy * p.Wo + ox;
            r.fresh = ok ? 0 : 1;
            const int wr = (r.img - b0) * p.win_L + (oy - first) * ss;
            r.slot = !ok ? 0 : MODE == SPLIT_FEW ? wr * p.RS + col * ss : wr * p.RS + (ss == 2 ? col : col * ss);   // (stride 2: even columns first)
        }
        return r;
    };
    int slot[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) slot[j] = pixel(j).slot;

    // ---- staging ---------------------------------------------------------------------------------------------------------
    bf8_t *const lds8 = reinterpret_cast<bf8_t *>(lds);
    bf4_t *const lds4 = reinterpret_cast<bf4_t *>(lds);
    const int part8 = p.CS << no_shift;         // slots per part
    Extremes extremes;
    auto affine = [&](float (&v)[8], int chunk, int c) {
        if constexpr (AFF) {
            const float *const a = p.in_aff + (size_t)chunk * 2 * p.CCH + c;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = v[e] * a[e] + a[p.CCH + e];
                if (p.in_relu) v[e] = fmaxf(v[e], 0.0f);
            }
        }
    };

    // FLAT: this thread's octet and pixel group
    px_t group[8];
    int f_oct = 0, f_unit = 0;
    unsigned f_voff = 0;
    if constexpr (MODE == SPLIT_FLAT) {
        const int t16 = tid >> 4;
        f_oct = fdiv(t16, p.fd_wn);
        f_unit = (t16 - f_oct * p.WN) * 16 + (tid & 15);
        const int uc = min(u0 + f_unit, p.units - 1);
        const int img = fdiv(uc, p.fd_units);
        const int pix = min(NB * (uc - img * p.fd_units.d), p.P - NB);
        f_voff = (unsigned)(img - b0) * (unsigned)p.in_bstride * 4u + (unsigned)pix * 4u + (unsigned)(8 * f_oct) * HW4;
    }
    auto request_flat = [&](int st) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const bool real = st * p.CCH + 8 * f_oct + e < p.C;
            group[e] = G::load(in_rsrc, real ? (int)f_voff : OOB_OFFSET, (int)((unsigned)(st * p.CCH + e) * HW4));
        }
    };
    auto park_flat = [&](int st) {
#pragma unroll
        for (int x = 0; x < NB; ++x) {
            float v[8];
            bf8_t h[3];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = group[e][x];
            affine(v, st, 8 * f_oct);
            split3(v, h);
            extremes.add(v);
#pragma unroll
            for (int s = 0; s < 3; ++s) lds8[s * part8 + f_oct * p.CS + x * (16 * p.WN) + f_unit] = h[s];
        }
    };
    auto stage_window = [&](int st) {
        constexpr int EN = MODE == SPLIT_FEW ? 8 : 4;            // entries of a thread in flight
        constexpr int CE = MODE == SPLIT_FEW ? 4 : 8;            // channels of an entry
        const int np = p.fd_npx.d;                               // pixels of the window
        const int entries = MODE == SPLIT_FEW ? np : np << no_shift;
        for (int e0 = tid; e0 < entries; e0 += EN * threads) {
            float v[EN][CE];
            int at[EN], oct[EN];
#pragma unroll
            for (int i = 0; i < EN; ++i) {
                const int e = e0 + i * threads;
                const int o = MODE == SPLIT_FEW ? 0 : fdiv(min(e, entries - 1), p.fd_npx);
                const int w = min(e, entries - 1) - o * np;
                const int wr = fdiv(w, p.fd_hww);
                const int wc = w - wr * p.fd_hww.d;
                const int a = wr + first * ss;
                const int bi = fdiv(a, p.fd_winL);
                const int y = a - bi * p.win_L - p.pad;
                const int x = tx * p.TW * ss + wc - p.pad;
                oct[i] = o;
                at[i] = e < entries ? wr * p.RS + (ss == 2 && MODE == SPLIT_WINDOW ? (wc >> 1) + (wc & 1) * half : wc) : -1;
                const bool in = (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.W && b0 + bi < p.batch && e < entries;
                const int c0 = st * p.CCH + CE * o;
                const unsigned voff = (unsigned)bi * (unsigned)p.in_bstride * 4u + (unsigned)(y * p.W + x) * 4u + (unsigned)c0 * HW4;
#pragma unroll
                for (int c = 0; c < CE; ++c)
                    v[i][c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        in_rsrc, in && c0 + c < p.C ? (int)voff : OOB_OFFSET, (int)((unsigned)c * HW4), 0));
            }
#pragma unroll
            for (int i = 0; i < EN; ++i) {
                if (at[i] < 0) continue;
                extremes.add(v[i]);
                if constexpr (MODE == SPLIT_FEW) {
                    bf4_t h[3];
                    split3(v[i], h);
#pragma unroll
                    for (int s = 0; s < 3; ++s) lds4[s * p.CS + at[i]] = h[s];
                } else {
                    bf8_t h[3];
                    split3(v[i], h);
#pragma unroll
                    for (int s = 0; s < 3; ++s) lds8[s * part8 + oct[i] * p.CS + at[i]] = h[s];
                }
            }
        }
    };

    // ---- matrix work -----------------------------------------------------------------------------------------------------
    f4_t lead[MB][NB], rest[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int j = 0; j < NB; ++j) lead[m][j] = rest[m][j] = (f4_t){0.0f, 0.0f, 0.0f, 0.0f};
    const int steps_all = p.nchunks * ksteps;
    // (requested here and looked at behind the last stage.  Read from memory and not passed: new weights may come under a captured graph)
    const float scaled_flag = *p.w_scale;
    const float *const w_scale = p.w_scale + 4;
    const int mblk0 = (by * p.WM + wm) * MB;
    struct A {
        bf8_t h[3];
    };
    auto load_a = [&](int m, int step) {
        A a;
        const int at = ((mblk0 + m) * steps_all + step) * 3072;
#pragma unroll
        for (int s = 0; s < 3; ++s)
            a.h[s] = __builtin_bit_cast(bf8_t, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, lane * 16, at + s * 1024, 0));
        return a;
    };
    // the K-steps of a stage that this wave takes: WM of them, or all
    const int ks_begin = MODE == SPLIT_FLAT ? slice * p.WM : 0, ks_count = MODE == SPLIT_FLAT ? p.WM : ksteps;
    A ahead = load_a(0, ks_begin);
    auto multiply = [&](int st) {
        for (int ki = 0; ki < ks_count; ++ki) {
            const int ks = ks_begin + ki;
            const int next = ki + 1 < ks_count ? st * ksteps + ks + 1 : (st + 1) * ksteps + ks_begin;
            bf8_t b[NB][3];
            int off;                            // this lane's octet of the K-step, as a distance from its pixel's slot
            if constexpr (MODE == SPLIT_FLAT) {
                off = (4 * ks + k) * p.CS;
            } else {
                const int idx = 4 * ks + k;     // (pairs past the last tap have zero weights: any slot will do)
                const int tap = MODE == SPLIT_FEW ? idx : min(idx >> no_shift, p.KH * p.KW - 1);
                const int kr = fdiv(tap, p.fd_wtw);
                const int kx = tap - kr * p.fd_wtw.d;
                if constexpr (MODE == SPLIT_FEW) {
                    off = min(kr, p.KH - 1) * p.RS + 2 * kx;
                } else {
                    const int cx = kx * p.dil;
                    off = (idx & ((1 << no_shift) - 1)) * p.CS + kr * p.dil * p.RS + (ss == 2 ? (cx >> 1) + (cx & 1) * half : cx);
                }
            }
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int s = 0; s < 3; ++s)
                    b[j][s] = MODE == SPLIT_FEW ? lds8[(s * p.CS + slot[j] + off) >> 1]   // (all even: the stride is)
                                                : lds8[s * part8 + slot[j] + off];
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const A a = ahead;
                // (further ahead, four blocks, costs registers and was no faster)
                ahead = m + 1 < MB ? load_a(m + 1, st * ksteps + ks) : load_a(0, min(next, steps_all - 1));
                __builtin_amdgcn_sched_barrier(0);   // (the request stays in front of the MFMAs it runs under)
#pragma unroll
                for (int j = 0; j < NB; ++j) lead[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h[0], b[j][0], lead[m][j], 0, 0, 0);
                // smallest first; NB independent chains, so that no MFMA waits for the one before it
                constexpr int ia[5] = {2, 1, 0, 1, 0}, ib[5] = {0, 1, 2, 0, 1};
#pragma unroll
                for (int t = 0; t < 5; ++t)
#pragma unroll
                    for (int j = 0; j < NB; ++j)
                        rest[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h[ia[t]], b[j][ib[t]], rest[m][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    auto barrier = [&]() {                      // orders LDS only: requests in flight stay in flight
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    if constexpr (MODE == SPLIT_FLAT) request_flat(0);
    unsigned met_word = 0;
    for (int st = 0; st < p.nchunks; ++st) {
        if (st > 0) barrier();
        if constexpr (MODE == SPLIT_FLAT) {
            park_flat(st);
            if (st + 1 < p.nchunks) request_flat(st + 1);
        } else {
            stage_window(st);
        }
        if (st + 1 == p.nchunks) {
            const unsigned met = (__builtin_amdgcn_ballot_w64(extremes.tiny()) ? 1u : 0u) | (__builtin_amdgcn_ballot_w64(extremes.large()) ? 2u : 0u);
            if (lane == 0) reinterpret_cast<unsigned *>(lds_all)[wave] = met;
        }
        barrier();
        met_word = reinterpret_cast<const unsigned *>(lds_all)[lane & 7];   // (comes in under the MFMAs; only the last one counts)
        multiply(st);
    }

    // ---- results ---------------------------------------------------------------------------------------------------------
    const int ch_base = mblk0 * 16 + 4 * k;
    const bool scaled = __builtin_amdgcn_readfirstlane(__float_as_int(scaled_flag)) == 0x3f800000;
    const unsigned met = lane < 8 && 64 * lane < threads ? met_word : 0u;
    const bool tiny_input = __builtin_amdgcn_ballot_w64((met & 1u) != 0) != 0, large_input = __builtin_amdgcn_ballot_w64((met & 2u) != 0) != 0;
    const bool has_resid = p.resid != nullptr;
    // Plain sums for pixel j of this lane's group or block (see above), lane n naming channel `ch`.
    auto plain = [&](int ch, int j) __attribute__((always_inline)) {
        const Pixel px = pixel(MODE == SPLIT_FLAT ? 0 : j);
        const int pix = MODE == SPLIT_FLAT ? px.pix + j : px.fresh ? 0 : px.pix;
        return direct_block<AFF>(ch, px.img, pix / p.Wo, pix % p.Wo);
    };
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int j = 0; j < NB; ++j) lead[m][j] += rest[m][j];

    if (MODE != SPLIT_FLAT || p.WK == 1) {
        Range range;
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) range.add(lead[m][j][i]);
        const bool bad = range.suspect();
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(bad) != 0 || tiny_input || scaled, 0)) {
#pragma unroll 1
            for (int r = 0; r < MB * NB; ++r) {
                const f4_t scale = scaled ? (f4_t)*reinterpret_cast<const f4u_t *>(w_scale + ch_base + 16 * (r / NB)) : (f4_t){1.0f, 1.0f, 1.0f, 1.0f};   // (padded to whole blocks)
                f4_t v = lead[0][0];
#pragma unroll
                for (int x = 1; x < MB * NB; ++x) v = x != r ? v : lead[x / NB][x % NB];
                bool ask[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) ask[i] = in_question(v[i], scale[i], tiny_input, large_input);
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] *= fabsf(scale[i]);
                if (__builtin_amdgcn_ballot_w64(ask[0] || ask[1] || ask[2] || ask[3]) != 0) {
                    const f4_t sums = plain((mblk0 + r / NB) * 16 + n, r % NB);
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = ask[i] ? sums[i] : v[i];
                }
#pragma unroll
                for (int x = 0; x < MB * NB; ++x) lead[x / NB][x % NB] = x != r ? lead[x / NB][x % NB] : v;
            }
        }
    }
    if constexpr (MODE == SPLIT_FLAT) {
        const Pixel px = pixel(0);
        float *__restrict__ const out = p.out + ((long long)px.img * p.out_bstride + px.pix);
        const float *__restrict__ const resid = has_resid ? p.resid + ((long long)px.img * p.resid_bstride + px.pix) : nullptr;
        auto load_resid = [&](int ch) { return (px_t)*reinterpret_cast<const typename G::mem_t *>(resid + (long long)min(ch, p.N - 1) * p.P); };
        auto finish = [&](px_t v, int ch, float bv, px_t rv) {     // one output row of this lane
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                v[j] += bv;
                if (has_resid) v[j] += rv[j];
                if (p.relu) v[j] = fmaxf(v[j], 0.0f);
            }
            if (ch >= p.N) return;
            float *const o = out + (long long)ch * p.P;
            if (px.fresh == 0) {
                *reinterpret_cast<typename G::mem_t *>(o) = v;
            } else {
#pragma unroll
                for (int j = 1; j < NB; ++j)
                    if (j >= px.fresh) o[j] = v[j];
            }
        };
        if (p.WK == 1) {
            float bv[4 * MB];
            px_t rv[4 * MB];
#pragma unroll
            for (int r = 0; r < 4 * MB; ++r) bv[r] = p.bias ? p.bias[min(ch_base + 16 * (r >> 2) + (r & 3), p.N - 1)] : 0.0f;
            if (has_resid) {
#pragma unroll
                for (int r = 0; r < 4 * MB; ++r) rv[r] = load_resid(ch_base + 16 * (r >> 2) + (r & 3));
            }
            settle(bv);
            settle(rv);
#pragma unroll
            for (int r = 0; r < 4 * MB; ++r) {
                px_t v;
#pragma unroll
                for (int j = 0; j < NB; ++j) v[j] = lead[r >> 2][j][r & 3];
                finish(v, ch_base + 16 * (r >> 2) + (r & 3), bv[r], rv[r]);
            }
            return;
        }
        // the WK waves of one (wm, wn) leave their rows in LDS, [slice][row = 4m + i][lane], and finish every WK-th row each
        barrier();
        px_t *const part = reinterpret_cast<px_t *>(lds) + (size_t)(t1 * p.WK) * (4 * MB * 64) + lane;
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                px_t v;
#pragma unroll
                for (int j = 0; j < NB; ++j) v[j] = lead[m][j][i];
                part[(slice * 4 * MB + 4 * m + i) * 64] = v;
            }
        barrier();
        const int rows = 4 * MB / p.WK;          // (WK divides 4 * MB)
        float bv[2 * MB];
        px_t rv[2 * MB];
#pragma unroll
        for (int r = 0; r < 2 * MB; ++r) {
            if (r >= rows) break;
            const int row = slice + r * p.WK, ch = ch_base + 16 * (row >> 2) + (row & 3);
            bv[r] = p.bias ? p.bias[min(ch, p.N - 1)] : 0.0f;
            if (has_resid) rv[r] = load_resid(ch);
        }
        settle(bv);
        settle(rv);
#pragma unroll
        for (int r0 = 0; r0 < 2 * MB; r0 += 2) {   // two at a time
            if (r0 >= rows) break;
            px_t v[2];
            int ch[2];
            bool bad = false;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int row = slice + min(r0 + i, rows - 1) * p.WK;
                ch[i] = ch_base + 16 * (row >> 2) + (row & 3);
                v[i] = part[row * 64];
                for (int s = 1; s < p.WK; ++s) v[i] += part[(s * 4 * MB + row) * 64];
#pragma unroll
                for (int j = 0; j < NB; ++j) bad |= suspect(v[i][j]);
            }
            float scale[2] = {1.0f, 1.0f};
            if (__builtin_expect(tiny_input || scaled, 0)) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    if (scaled) scale[i] = w_scale[ch[i]];
#pragma unroll
                    for (int j = 0; j < NB; ++j) bad |= in_question(v[i][j], scale[i], tiny_input, large_input);
                }
            }
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(bad) != 0, 0)) {
                // (rows 4k and 4k + 1 of the block of plain sums are the two of quarter k here)
                const int row = slice + min(r0 + (n & 1), rows - 1) * p.WK;
#pragma unroll 1
                for (int j = 0; j < NB; ++j) {
                    const f4_t sums = plain(mblk0 * 16 + 16 * (row >> 2) + (row & 3) + (n & 12), j);
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int x = 0; x < NB; ++x) v[i][x] = x != j ? v[i][x] : in_question(v[i][x], scale[i], tiny_input, large_input) ? sums[i] : v[i][x] * fabsf(scale[i]);
                }
            } else if (__builtin_expect(scaled, 0)) {
#pragma unroll
                for (int i = 0; i < 2; ++i) v[i] *= fabsf(scale[i]);
            }
            finish(v[0], ch[0], bv[r0], rv[r0]);
            if (r0 + 1 < rows) finish(v[1], ch[1], bv[r0 + 1], rv[r0 + 1]);
        }
    } else {
        const auto &q = *late_arguments();
        float bias[MB][4];
#pragma unroll
        for (int m = 0; m < MB; ++m) {
#pragma unroll
            for (int i = 0; i < 4; ++i) bias[m][i] = q.bias ? q.bias[min(ch_base + 16 * m + i, q.N - 1)] : 0.0f;
            settle(bias[m]);
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const Pixel px = pixel(j);
            if (px.fresh) continue;
            float resid[MB][4];
            if (q.resid) {                    // (a column of blocks at a time: all of them would not fit the registers)
                const float *__restrict__ const from = q.resid + ((long long)px.img * q.resid_bstride + px.pix);
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int i = 0; i < 4; ++i) resid[m][i] = from[(long long)min(ch_base + 16 * m + i, q.N - 1) * q.P];
#pragma unroll
                for (int m = 0; m < MB; ++m) settle(resid[m]);
            }
            float *__restrict__ const out = q.out + (long long)px.img * q.out_bstride;
#pragma unroll
            for (int m = 0; m < MB; ++m) store_four_channels(lead[m][j], ch_base + 16 * m, q.N, q.P, px.pix, bias[m], q.resid != nullptr, resid[m], q.relu, out);
        }
    }
}

using kernel_fn = void (*)(ConvKParams);

template <int MB, int NB>
static kernel_fn with_affine(bool aff) {
    return aff ? static_cast<kernel_fn>(tdc_conv_split_kernel<MB, NB, SPLIT_FLAT, true>) : tdc_conv_split_kernel<MB, NB, SPLIT_FLAT, false>;
}

const void *split_kernel_function(const KernelId &k) {
    if (k.family != KernelId::SPLIT) return nullptr;
    const int mb = k.p[0], nb = k.p[1], mode = k.p[2];
    const bool aff = k.p[3] != 0;
    kernel_fn fn = nullptr;
    if (mode == SPLIT_FLAT && nb == 4) fn = mb == 1 ? with_affine<1, 4>(aff) : mb == 2 ? with_affine<2, 4>(aff) : nullptr;
    if (mode == SPLIT_FLAT && nb == 2) fn = mb == 1 ? with_affine<1, 2>(aff) : mb == 2 ? with_affine<2, 2>(aff) : nullptr;
    if (mode == SPLIT_WINDOW && nb == 4 && !aff)
        fn = mb == 1   ? static_cast<kernel_fn>(tdc_conv_split_kernel<1, 4, SPLIT_WINDOW, false>)
             : mb == 2 ? tdc_conv_split_kernel<2, 4, SPLIT_WINDOW, false>
             : mb == 4 ? tdc_conv_split_kernel<4, 4, SPLIT_WINDOW, false> : nullptr;
    if (mode == SPLIT_FEW && nb == 4 && !aff)
        fn = mb == 1   ? static_cast<kernel_fn>(tdc_conv_split_kernel<1, 4, SPLIT_FEW, false>)
             : mb == 2 ? tdc_conv_split_kernel<2, 4, SPLIT_FEW, false>
             : mb == 4 ? tdc_conv_split_kernel<4, 4, SPLIT_FEW, false> : nullptr;
    return reinterpret_cast<const void *>(fn);
}

}  // namespace tdc
