// fp32 convolutions with larger filters on the bf16 matrix pipe (tile.alg = 8 with tw > 0 and nb = 2, tdc_core_split_kernel).
#include "conv_device.hpp"
#include "conv_split_device.hpp"

namespace tdc {

// ---------------------------------------------------------------------------
// Filters of more than one tap over more than four input channels, operands split in three bf16 parts (conv_split.hip tells how
// a product is summed, and what happens to operands that the split cannot hold; its form of 64 pixels per wave takes the largest
// launches).
// A workgroup is WM x WN x WK waves over 16*MB channels x 32 pixels each: a tile of TH output rows (counted through the
// batch) x TW columns.  The input window of CCH channels is staged in octets, split once per workgroup, and the K-steps of the
// stage, which run over its (tap, octet) pairs, are divided among the WK waves; their sums meet in LDS.  At stride 2 the even and
// the odd columns lie in separate halves of a row, so that neighbouring lanes read neighbouring slots.
// Bound: the latencies of one workgroup's chain and the issue slots of the SIMDs, not the matrix pipes: 128 -> 128 @28 / stride 2
// batch 32 has 5.0 us of MFMAs and 3.1 us of memory traffic.  Of the 19.7 us of its kernel (time stamps) a wave takes 2.5 until its
// first requests are out, 2.4 until they have landed and are split, 0.7 at the barrier, 10.3 for its 18 K-steps, 1.7 until the sums of
// the slices are added and 1.0 for the stores.  Hence
//   - the next stage is requested in front of the MFMAs of this one (four entries a thread; what a larger stage has beyond that
//     comes in rounds of its own), and the weights of a K-step are reloaded in place right behind the MFMAs that read them, a K-step
//     ahead: a ring that copies registers would make every copy wait for what was requested last;
//   - the three parts of a slot lie together, 48 bytes, one address for three reads, and octets a multiple of 16 slots, whole rounds
//     of the banks, apart, so that all four lane quarters meet the same banks.  Conflicts still take half of the cycles in which the LDS is active
//     (48 to 55 % in three layers), but waves wait for it in 1 to 2 % of their time only;
//   - all six products of a K-step start from zero and are added to the sums once: a single chain per block and half the
//     accumulators.  The error against 64-bit sums at 3x3 and 64, 128 and 512 channels is 0.9, 1.2 and 2.2e-7 of the norm
//     (with two accumulators that take the leading and the small products 1.3, 1.9 and 3.9e-7; one for all six throughout 3.7e-7
//     at 128), at 16 channels 7.0e-8 (6.6e-8).
// Two pixel blocks per wave: three to four waves per SIMD at mb = 1 and 2.  Four blocks, 24 operand registers more, are better where
// a launch has more matrix work than latency, or only one stage, behind which nothing can be requested: conv_split.hip's form keeps those
// layers (core_split_takes in tile_model.cpp).
// Measured (in one graph, in turn with the best of the other tiles, us): 3x3 / stride 2 128 -> 128 @28 batch 32 30.0 -> 20.1, 64 -> 64
// @56 batch 32 22.7 -> 21.9, 256 -> 256 @14 batch 32 36.7 -> 24.6, 5x5 64 -> 96 @40 batch 16 60.8 -> 53.1; over 2557 random layers that take
// it 0.81 of the time.  At 3x3 / stride 1 Winograd saves more.
// ---------------------------------------------------------------------------
template <int MB>
__global__ void __launch_bounds__(512, 2) tdc_core_split_kernel(const ConvKParams p) {
    constexpr int NB = 2;
    extern __shared__ __align__(16) float lds_all[];
    float *const lds = lds_all + EXTREMES_FLOATS;
    TDC_STAMP_DECL;
    TDC_STAMP(0);   // entry
    touch_kernel_arguments();
    TDC_STAMP(7);   // every line of the kernel arguments is in the scalar cache
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int logical = (int)(blockIdx.x & 7u) * p.xcd_chunk + (int)(blockIdx.x >> 3);
    if (logical >= p.n_wg) return;
    const int q1 = fdiv(logical, p.fd_g1);
    const int r1 = logical - q1 * p.fd_g1.d;
    const int bx = p.channel_major ? r1 : q1;   // pixel tile
    const int by = p.channel_major ? q1 : r1;   // channel tile
    const int t1 = fdiv(wave, p.fd_wk);
    const int slice = wave - t1 * p.WK;         // of the K-steps of a stage
    const int wm = fdiv(t1, p.fd_wn);
    const int wn = t1 - wm * p.WN;
    const int k = lane >> 4, n = lane & 15;
    const int threads = 64 * p.WM * p.WN * p.WK;
    const unsigned HW4 = (unsigned)(p.H * p.W) * 4u;
    // (see Geometry) slots per output column, octets per stage as a power of two, K-steps per stage
    const int ss = p.slots_col, oct_shift = p.oct_shift, ksteps = p.ksteps, half = p.odd_columns;

    // first unit (output row, counted through the batch) and first image of the workgroup; its column tile
    const int ty = fdiv(bx, p.fd_ntx);
    const int tx = bx - ty * p.ntx;
    const int u0 = ty * p.TH;
    const int b0 = fdiv(u0, p.fd_units);
    const int first = u0 - b0 * p.fd_units.d;   // ... within its image

    const __amdgpu_buffer_rsrc_t in_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(p.in + (long long)b0 * p.in_bstride), (short)0, OOB_OFFSET, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.wpk), (short)0, (int)p.wpk_bytes, 0x00020000);

    struct Pixel {
        int img, pix;      // image and pixel offset within an output plane
        bool live;
        int slot;          // LDS slot of tap 0
    };
    auto pixel = [&](int j) {                   // block j of this wave
        Pixel r;
        const int q = (wn * NB + j) * 16 + n;
        const int row = fdiv(q, p.fd_tw);
        const int col = q - row * p.TW;
        const int ox = tx * p.TW + col;
        r.live = row < p.TH && u0 + row < p.units && ox < p.Wo;
        const int g = min(u0 + row, p.units - 1);
        r.img = fdiv(g, p.fd_units);
        const int oy = g - r.img * p.fd_units.d;
        r.pix = oy * p.Wo + ox;
        const int wr = (r.img - b0) * p.win_L + (oy - first) * ss;
        r.slot = r.live ? wr * p.RS + (ss == 2 ? col : col * ss) : 0;   // (stride 2: even columns first)
        return r;
    };
    int slot[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) slot[j] = pixel(j).slot;

    // ---- staging: entry = (pixel of the window, octet of channels) -------------------------------------------------------------
    bf8_t *const lds8 = reinterpret_cast<bf8_t *>(lds);
    const int np = p.fd_npx.d;                  // pixels of the window
    const int entries = np << oct_shift;
    Extremes extremes;
    constexpr int EN = 4;                       // entries of a thread in flight
    float raw[EN][8];
    struct Entry {
        int at;                                 // place in LDS, < 0: none
        int c;                                  // first channel within the stage
        unsigned voff;                          // of that channel in the first stage
    };
    auto entry = [&](int e) {
        Entry r;
        const int ec = min(e, entries - 1);
        const int o = fdiv(ec, p.fd_npx);
        const int w = ec - o * np;
        const int wr = fdiv(w, p.fd_hww);
        const int wc = w - wr * p.fd_hww.d;
        const int a = wr + first * ss;
        const int bi = fdiv(a, p.fd_winL);
        const int y = a - bi * p.win_L - p.pad;
        const int x = tx * p.TW * ss + wc - p.pad;
        r.at = e < entries ? 3 * (o * p.CS + wr * p.RS + (ss == 2 ? (wc >> 1) + (wc & 1) * half : wc)) : -1;
        r.c = 8 * o;
        const bool in = (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.W && b0 + bi < p.batch && e < entries;
        r.voff = in ? (unsigned)bi * (unsigned)p.in_bstride * 4u + (unsigned)(y * p.W + x) * 4u + (unsigned)r.c * HW4 : (unsigned)OOB_OFFSET;
        return r;
    };
    auto request = [&](float (&v)[8], const Entry &r, int st) {
        const bool whole = (st + 1) * p.CCH <= p.C;
        const unsigned base = (unsigned)(st * p.CCH) * HW4;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const unsigned voff = whole || st * p.CCH + r.c + c < p.C ? r.voff : (unsigned)OOB_OFFSET;
            v[c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(in_rsrc, (int)voff, (int)(base + (unsigned)c * HW4), 0));
        }
    };
    auto park = [&](const float (&v)[8], const Entry &r) {
        if (r.at < 0) return;
        bf8_t h[3];
        extremes.add(v);
        split3(v, h);
#pragma unroll
        for (int s = 0; s < 3; ++s) lds8[r.at + s] = h[s];
    };
    Entry ent[EN];                              // the first EN * threads entries, the same in every stage
#pragma unroll
    for (int i = 0; i < EN; ++i) ent[i] = entry(tid + i * threads);
    auto request_stage = [&](int st) {
#pragma unroll
        for (int i = 0; i < EN; ++i) request(raw[i], ent[i], st);
    };
    auto park_stage = [&](int st) {
#pragma unroll
        for (int i = 0; i < EN; ++i) park(raw[i], ent[i]);
        for (int e0 = EN * threads; e0 < entries; e0 += EN * threads) {   // (what one round does not hold)
            Entry more[EN];
#pragma unroll
            for (int i = 0; i < EN; ++i) {
                more[i] = entry(e0 + tid + i * threads);
                request(raw[i], more[i], st);
            }
#pragma unroll
            for (int i = 0; i < EN; ++i) park(raw[i], more[i]);
        }
    };

    // ---- matrix work -----------------------------------------------------------------------------------------------------
    f4_t acc[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[m][j] = (f4_t){0.0f, 0.0f, 0.0f, 0.0f};
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
    const int ks_count = fdiv(ksteps, p.fd_wk);     // (WK divides ksteps)
    const int ks_begin = slice * ks_count;
    A ring[MB];                                 // the weights of a K-step, requested a K-step ahead
#pragma unroll
    for (int m = 0; m < MB; ++m) ring[m] = load_a(m, ks_begin);
    // (with at least four octets a stage lane quarter k reads every fourth of them)
    const char *own[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) own[j] = reinterpret_cast<const char *>(lds) + 48 * (k * p.CS + slot[j]);
    auto multiply = [&](int st) {
#pragma unroll 1
        for (int ki = 0; ki < ks_count; ++ki) {
            const int ks = ks_begin + ki;
            const int next = min(ki + 1 < ks_count ? st * ksteps + ks + 1 : (st + 1) * ksteps + ks_begin, steps_all - 1);
            int off;                                // distance of this K-step's slots from tap 0 of the first octet
            if (oct_shift >= 2) {                   // one tap per K-step
                const int tap = (4 * ks) >> oct_shift;
                const int kr = fdiv(tap, p.fd_wtw);
                const int cx = (tap - kr * p.fd_wtw.d) * p.dil;
                off = ((4 * ks) & ((1 << oct_shift) - 1)) * p.CS + kr * p.dil * p.RS + (ss == 2 ? (cx >> 1) + (cx & 1) * half : cx);
            } else {
                const int idx = 4 * ks + k;         // (tap, octet); pairs past the last tap have zero weights: any slot will do
                const int tap = min(idx >> oct_shift, p.KH * p.KW - 1);
                const int kr = fdiv(tap, p.fd_wtw);
                const int cx = (tap - kr * p.fd_wtw.d) * p.dil;
                off = ((idx & ((1 << oct_shift) - 1)) - k) * p.CS + kr * p.dil * p.RS + (ss == 2 ? (cx >> 1) + (cx & 1) * half : cx);
            }
            bf8_t b[NB][3];
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int s = 0; s < 3; ++s) b[j][s] = *reinterpret_cast<const bf8_t *>(own[j] + 48 * off + 16 * s);
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                // smallest first, all from zero: one addition per K-step rounds at the size of the whole sum
                constexpr int ia[6] = {2, 1, 0, 1, 0, 0}, ib[6] = {0, 1, 2, 0, 1, 0};
                f4_t t[NB];
#pragma unroll
                for (int j = 0; j < NB; ++j) t[j] = (f4_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int x = 0; x < 6; ++x)
#pragma unroll
                    for (int j = 0; j < NB; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[m].h[ia[x]], b[j][ib[x]], t[j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                ring[m] = load_a(m, next);
#pragma unroll
                for (int j = 0; j < NB; ++j) acc[m][j] += t[j];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    auto barrier = [&]() {                      // orders LDS only: requests in flight stay in flight
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    request_stage(0);
    TDC_STAMP(1);   // first stage and first weights requested
#pragma unroll 1
    for (int st = 0; st < p.nchunks; ++st) {
        if (st > 0) barrier();
        park_stage(st);
        if (st == 0) TDC_STAMP(2);   // my part of the first stage has landed and is split
        if (st + 1 == p.nchunks) {
            const unsigned met = (__builtin_amdgcn_ballot_w64(extremes.tiny()) ? 1u : 0u) | (__builtin_amdgcn_ballot_w64(extremes.large()) ? 2u : 0u);
            if (lane == 0) reinterpret_cast<unsigned *>(lds_all)[wave] = met;
        }
        barrier();
        if (st == 0) TDC_STAMP(3);   // everybody's is
        request_stage(st + 1);                  // (past the last stage: nothing but offsets out of range)
        __builtin_amdgcn_sched_barrier(0);
        multiply(st);
    }

    TDC_STAMP(4);   // all stages multiplied

    // ---- results ---------------------------------------------------------------------------------------------------------
    const unsigned met_word = reinterpret_cast<const unsigned *>(lds_all)[lane & 7];
    const bool scaled = __builtin_amdgcn_readfirstlane(__float_as_int(scaled_flag)) == 0x3f800000;
    const unsigned met = lane < 8 && 64 * lane < threads ? met_word : 0u;
    const bool tiny_input = __builtin_amdgcn_ballot_w64((met & 1u) != 0) != 0, large_input = __builtin_amdgcn_ballot_w64((met & 2u) != 0) != 0;
    if (p.WK > 1) {
        // the WK waves of one (wm, wn) leave their sums in LDS, [slice][block][lane], and finish every WK-th block each
        barrier();
        f4_t *const part = reinterpret_cast<f4_t *>(lds) + (size_t)(t1 * p.WK) * (MB * NB * 64) + lane;
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int j = 0; j < NB; ++j) part[(slice * MB * NB + m * NB + j) * 64] = acc[m][j];
        barrier();
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                if ((m * NB + j) % p.WK != slice) continue;
                f4_t v = part[(m * NB + j) * 64];
                for (int s = 1; s < p.WK; ++s) v += part[(s * MB * NB + m * NB + j) * 64];
                acc[m][j] = v;
            }
    }
    TDC_STAMP(5);   // sums of all slices added
    auto mine = [&](int r) { return p.WK == 1 || r % p.WK == slice; };
    Range range;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) range.add(acc[m][j][i]);
    const int ch_base = mblk0 * 16 + 4 * k;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(range.suspect()) != 0 || tiny_input || scaled, 0)) {
#pragma unroll 1
        for (int r = 0; r < MB * NB; ++r) {
            if (!mine(r)) continue;
            const f4_t scale = scaled ? (f4_t)*reinterpret_cast<const f4u_t *>(w_scale + ch_base + 16 * (r / NB)) : (f4_t){1.0f, 1.0f, 1.0f, 1.0f};   // (padded to whole blocks)
            f4_t v = acc[0][0];
#pragma unroll
            for (int x = 1; x < MB * NB; ++x) v = x != r ? v : acc[x / NB][x % NB];
            bool ask[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) ask[i] = in_question(v[i], scale[i], tiny_input, large_input);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] *= fabsf(scale[i]);
            if (__builtin_amdgcn_ballot_w64(ask[0] || ask[1] || ask[2] || ask[3]) != 0) {
                const Pixel px = pixel(r % NB);
                const int pix = px.live ? px.pix : 0;
                const f4_t sums = direct_block<false>((mblk0 + r / NB) * 16 + n, px.img, pix / p.Wo, pix % p.Wo);
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = ask[i] ? sums[i] : v[i];
            }
#pragma unroll
            for (int x = 0; x < MB * NB; ++x) acc[x / NB][x % NB] = x != r ? acc[x / NB][x % NB] : v;
        }
    }
    float bias[MB][4], resid[MB * NB][4];
    const bool has_resid = p.resid != nullptr;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) bias[m][i] = p.bias ? p.bias[min(ch_base + 16 * m + i, p.N - 1)] : 0.0f;
    if (has_resid) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const Pixel px = pixel(j);
            if (!px.live) continue;
            const float *__restrict__ const from = p.resid + ((long long)px.img * p.resid_bstride + px.pix);
#pragma unroll
            for (int m = 0; m < MB; ++m)
                if (mine(m * NB + j)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) resid[m * NB + j][i] = from[(long long)min(ch_base + 16 * m + i, p.N - 1) * p.P];
                }
        }
    }
#pragma unroll
    for (int m = 0; m < MB; ++m) settle(bias[m]);
#pragma unroll
    for (int r = 0; r < MB * NB; ++r) settle(resid[r]);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const Pixel px = pixel(j);
        if (!px.live) continue;
        float *__restrict__ const out = p.out + (long long)px.img * p.out_bstride;
#pragma unroll
        for (int m = 0; m < MB; ++m)
            if (mine(m * NB + j)) store_four_channels(acc[m][j], ch_base + 16 * m, p.N, p.P, px.pix, bias[m], has_resid, resid[m * NB + j], p.relu, out);
    }
    TDC_STAMP(6);   // stores issued
    TDC_STAMP_FLUSH(p, logical, wave, lane);
}

const void *core_split_kernel_function(const KernelId &k) {
    using kernel_fn = void (*)(ConvKParams);
    if (k.family != KernelId::SPLIT_CORE) return nullptr;
    const int mb = k.p[0];
    const kernel_fn fn = mb == 1   ? static_cast<kernel_fn>(tdc_core_split_kernel<1>)
                         : mb == 2 ? tdc_core_split_kernel<2>
                         : mb == 4 ? tdc_core_split_kernel<4> : nullptr;
    return reinterpret_cast<const void *>(fn);
}

}  // namespace tdc
