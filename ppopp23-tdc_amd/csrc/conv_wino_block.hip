// Winograd F(2x2,3x3) for batches (tile.alg = 1 with tile.tw = 0, tdc_wino3x3_block_kernel).
#include "conv_device.hpp"

#include <type_traits>

namespace tdc {

// ---------------------------------------------------------------------------
// 3x3 / stride 1 / dilation 1 / pad <= 1.  The 2x2-pixel output tiles of the whole batch form one row; a wave owns 16 of
// them (one per pixel lane, so neither image edges nor small images leave lanes idle) and 16*MB output channels.
//   * Input: per four channels each lane loads the 4x4 patch of its own tile as four 128-bit row pieces straight into
//     registers, two channel groups ahead, and transforms it there (V = B^T d B).  Columns outside the image are masked
//     after the row transform; rows outside it read zero through an out-of-range offset.
//   * Weights: the transformed weights U of a step (two groups of four channels) are fetched once per workgroup, a step
//     ahead, and shared through LDS, double-buffered, one barrier per step.  What a wave would otherwise pull from the L2
//     for itself, 4 KiB per four channels and 16 MFMAs, is close to all the L2s deliver: the staged Winograd kernel reads
//     3.3 GB of weights for 128 -> 128 @56 at batch 64, 11.5 TB/s.  WN waves over tiles divide it by WN.
//   * Vector instructions: an fp32 MFMA and a vector instruction of the same SIMD do not overlap, not even from different
//     waves (16 MFMAs with 0 / 32 / 64 v_add behind them take 517 / 589 / 656 cycles at four waves per SIMD; spread
//     between the MFMAs 646 / 711).  So the 40 of a transform stand in one piece per group, addresses advance through
//     scalar offsets, and MB = 2 halves their share.
// Bound: the matrix pipe, 88 % busy in the steady state at two waves per SIMD; then the start and end of a workgroup
// (first operands, 24 additions and two stores per output row) and the last, partly filled round of workgroups.
// Against the staged Winograd kernel (launch-to-launch, one box): 128 -> 128 @56 batch 64 284 -> 253 us, 256 -> 256 @7
// batch 64 35.3 -> 25.9, 128 -> 128 @14 batch 32 20.1 -> 15.3, 32 -> 32 @56 batch 32 20.1 -> 15.7; on sizes the tiles of
// that kernel do not divide 1.3 to 2 times as fast (64 -> 176 @59 batch 13 103 -> 50, 145 random shapes 1.5 on average).
// WK teams of WN waves split the input channels; their 2x2 outputs are added through LDS in team order.
// Outputs that come out infinite or NaN are computed as plain sums (direct_block); the look at them costs at most 0.1 us
// (60 -> 84 @35 batch 5 10.3 -> 10.4, 128 -> 128 @56 batch 64 within 1 %).
// ---------------------------------------------------------------------------
// PARTS: every eight steps (64 channels of the team) the outputs of the sums so far are added up in LDS and the sums start at
// zero again, 4 * MB KiB per wave.  The error of a chain grows with the root of its length: 528 -> 112 @40 batch 17 in one chain
// 7.0e-7 and 141 us, staged with four slices 3.6e-7 and 216, two teams in parts 2.7e-7 and 164.  Beside the same tile in one
// chain 1.05 to 1.06 of the time with four waves, 1.00 to 1.025 with eight (82 to 1024 channels, 63 shapes), so it is a form of
// its own, for layers whose other tiles have shorter chains than a team.
template <int MB, int WN, bool PARTS>
__global__ void __launch_bounds__(512, 2) tdc_wino3x3_block_kernel(const ConvKParams p) {
    constexpr int G = 2;                        // groups of four channels per step (four never won: fewer waves fit)
    constexpr int CHUNKS = MB * G * 4;          // KiB of transformed weights per team and step
    constexpr int NU = CHUNKS / WN;             // ... that each wave fetches
    static_assert(CHUNKS % WN == 0, "every wave of a team fetches the same number of KiB");
    extern __shared__ __align__(16) float lds[];
    touch_kernel_arguments();
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int logical = (int)(blockIdx.x & 7u) * p.xcd_chunk + (int)(blockIdx.x >> 3);
    if (logical >= p.n_wg) return;
    const int q1 = fdiv(logical, p.fd_g1);
    const int r1 = logical - q1 * p.fd_g1.d;
    const int bx = p.channel_major ? r1 : q1;   // block of tiles
    const int by = p.channel_major ? q1 : r1;   // block of channels
    const int slice = wave / WN, wn = wave % WN;
    const int k = lane >> 4, n = lane & 15;

    // this lane's tile: image (offsets are relative to the image b0 of the wave's first tile), row, column
    const int u0 = (bx * WN + wn) * 16;
    const int b0 = fdiv(min(u0, p.units - 1), p.fd_units);
    const bool live = u0 + n < p.units;
    const int uc = min(u0 + n, p.units - 1);
    const int img = fdiv(uc, p.fd_units);
    const int rest = uc - img * p.fd_units.d;
    const int ty = fdiv(rest, p.fd_wtw);
    const int tx = rest - ty * p.fd_wtw.d;
    const int x0 = 2 * tx - p.pad, y0 = 2 * ty - p.pad;
    const bool left = x0 < 0, right2 = x0 + 2 >= p.W, right3 = x0 + 3 >= p.W;   // patch columns 0, 2 and 3 outside the image
    const bool odd_width = (p.Wo & 1) != 0;     // only then can patch column 2 lie outside
    const unsigned HW4 = (unsigned)(p.H * p.W) * 4u;
    const unsigned img4 = (unsigned)(img - b0) * (unsigned)p.in_bstride * 4u;
    unsigned voff[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const bool ok = (unsigned)(y0 + r) < (unsigned)p.H;
        voff[r] = ok ? img4 + (unsigned)((y0 + r) * p.W + x0) * 4u + (unsigned)k * HW4 : (unsigned)OOB_OFFSET;
    }
    // (the range check is exact: the last row piece of the batch may reach past the end of the input)
    const long long reach = ((long long)(p.batch - 1 - b0) * p.in_bstride + (long long)p.C * (p.H * p.W)) * 4;
    const __amdgpu_buffer_rsrc_t in_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(p.in + (long long)b0 * p.in_bstride), (short)0, (int)(reach < OOB_OFFSET ? reach : OOB_OFFSET), 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.wpk), (short)0, (int)p.wpk_bytes, 0x00020000);

    const int ncg = p.CCH >> 2;                 // channel groups of the packed weights
    const int steps = p.CPW / (4 * G);          // of every team: step i of team s holds channel groups (i * WK + s) * G + 0 .. G-1,
                                                // so that what cch has more than C lies in the last steps
    const int a_base = by * MB * ncg * 4096;
    f4_t *const ubuf = reinterpret_cast<f4_t *>(lds) + slice * (CHUNKS * 64) + lane;
    const int ustage = p.WK * (CHUNKS * 64);    // f4 per buffer

    // ring of requested patches
    float d[G][4][4];
    auto request = [&](int slot, int r, unsigned off, int soff) {
        const f4_t v = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(in_rsrc, (int)off, soff, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) d[slot][r][e] = v[e];
    };
    // From group to group a scalar offset carries the patch pieces on, outside the range check (counted from 16 bytes in front
    // of the image, so that no offset is negative).  In the first and the last step the whole offset goes through the check:
    // there lie the first channel (offset -4, see below), the pieces that reach past the end of the batch and the channels
    // past C.
    auto load_patch = [&](int slot, int step, bool checked) {   // slot = channel group within the step
        const int group = (step * p.WK + slice) * G + slot;
        if (!checked) {
            const int soff = (int)((unsigned)(4 * group) * HW4) - 16;
#pragma unroll
            for (int r = 0; r < 4; ++r) request(slot, r, voff[r] + 16u, soff);
        } else {
            const int c = 4 * group + k;
            const unsigned chan = c < p.C ? (unsigned)(c - k) * HW4 : (unsigned)OOB_OFFSET + 8u;   // (past the range also from offset -4)
#pragma unroll
            for (int r = 0; r < 4; ++r) request(slot, r, voff[r] + chan, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    float v[16];                                // V = B^T d B of the group at hand
    auto transform = [&](int slot) {            // B^T = [1 0 -1 0; 0 1 1 0; 0 -1 1 0; 0 1 0 -1]
        const float(&p4)[4][4] = d[slot];
        float t[4][4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            t[0][e] = p4[0][e] - p4[2][e];
            t[1][e] = p4[1][e] + p4[2][e];
            t[2][e] = p4[2][e] - p4[1][e];
            t[3][e] = p4[1][e] - p4[3][e];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            t[q][0] = left ? 0.0f : t[q][0];
            t[q][3] = right3 ? 0.0f : t[q][3];
        }
        if (odd_width) {
#pragma unroll
            for (int q = 0; q < 4; ++q) t[q][2] = right2 ? 0.0f : t[q][2];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[4 * q + 0] = t[q][0] - t[q][2];
            v[4 * q + 1] = t[q][1] + t[q][2];
            v[4 * q + 2] = t[q][2] - t[q][1];
            v[4 * q + 3] = t[q][1] - t[q][3];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    f4_t unext[NU];
    auto load_u = [&](int step) {
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int ch = i * WN + wn;         // chunk = (channel block, group, quarter)
            const int mb = ch / (G * 4);
            unext[i] = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(
                w_rsrc, lane * 16, a_base + (mb * ncg + (step * p.WK + slice) * G) * 4096 + (ch - mb * (G * 4)) * 1024, 0));
        }
    };
    auto park_u = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NU; ++i) ubuf[buf * ustage + (i * WN + wn) * 64] = unext[i];
    };
    auto barrier = [&]() {                      // orders LDS only: the input requests in flight stay in flight
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    f4_t acc[MB][16];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int x = 0; x < 16; ++x) acc[m][x] = (f4_t){0.0f, 0.0f, 0.0f, 0.0f};

    load_u(0);
    load_patch(0, 0, true);
    // The piece left of the very first pixel of the buffer has a negative offset, which reads zero as a whole: such lanes
    // (first channel of the first image, row 0, leftmost tile) take columns 0 to 2 from a piece that starts at column 0.
    const bool before = left && img == b0 && slice + k == 0;
    if (__builtin_amdgcn_ballot_w64(before)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const f4_t w = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(
                in_rsrc, before && y0 + r == 0 ? 0 : OOB_OFFSET, 0, 0));
#pragma unroll
            for (int e = 1; e < 4; ++e)
                if (before && y0 + r == 0) d[0][r][e] = w[e - 1];
        }
    }
#pragma unroll
    for (int g = 1; g < G; ++g) load_patch(g, 0, true);
    __builtin_amdgcn_sched_barrier(0);
    park_u(0);
    load_u(min(1, steps - 1));
    barrier();
    // Weights in registers, read AHEAD quarters before their MFMAs (a quarter of MB = 1 is shorter than the way through LDS).
    constexpr int AHEAD = MB == 1 ? 2 : 1, RING = 2 * AHEAD;
    f4_t ua[RING][MB];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
#pragma unroll
        for (int m = 0; m < MB; ++m) ua[i][m] = ubuf[(m * G * 4 + i) * 64];
    // One step.  `next`: 0 = the last step, nothing to request; 1 = the step before it (the patches of the last one are
    // requested checked); 2 = any other.
    auto step = [&](int st, auto next) {
        constexpr int NEXT = decltype(next)::value;
        const f4_t *const us = ubuf + (st & 1) * ustage;
        const f4_t *const us_next = ubuf + ((st & 1) ^ 1) * ustage;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            // fp32 MFMAs and vector instructions of a SIMD do not overlap, not even between waves (see above): the transform
            // stands in one piece, and nothing but requests and LDS accesses among the MFMAs
            transform(g);
            if constexpr (NEXT > 0) load_patch(g, st + 1, NEXT == 1);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (NEXT > 0 && g == G - 1 && q == 0) {
                    park_u((st & 1) ^ 1);
                    if constexpr (NEXT == 2) load_u(st + 2);
                }
                if (NEXT > 0 && g == G - 1 && q == 4 - AHEAD) barrier();
                const int ahead = 4 * g + q + AHEAD;     // the quarter whose weights are read now
                if (NEXT > 0 || ahead < 4 * G) {
#pragma unroll
                    for (int m = 0; m < MB; ++m)
                        ua[(q + AHEAD) % RING][m] = ahead >= 4 * G ? us_next[(m * G * 4 + ahead - 4 * G) * 64] : us[(m * G * 4 + ahead) * 64];
                }
                __builtin_amdgcn_sched_barrier(0);   // (the weights of a later quarter are on their way under this one's MFMAs)
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[m][4 * q + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(ua[q % RING][m][e], v[4 * q + e], acc[m][4 * q + e], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // Y = A^T M A (A^T = [1 1 1 0; 0 1 -1 -1]): lane (k, n) holds channels 4k + i of tile n, all 16 positions
    auto output = [&](int m, int i) {
        float s[2][4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float m0 = acc[m][e][i], m1 = acc[m][4 + e][i], m2 = acc[m][8 + e][i], m3 = acc[m][12 + e][i];
            s[0][e] = m0 + m1 + m2;
            s[1][e] = m1 - m2 - m3;
        }
        return (f4_t){s[0][0] + s[0][1] + s[0][2], s[0][1] - s[0][2] - s[0][3], s[1][0] + s[1][1] + s[1][2], s[1][1] - s[1][2] - s[1][3]};
    };
    // outputs of the teams and of the parts of their sums: [wn][team][row = 4m + i][lane]
    f4_t *const part = reinterpret_cast<f4_t *>(lds) + (PARTS ? 2 * ustage : 0) + (size_t)(wn * p.WK) * (4 * MB * 64) + lane;
    f4_t *const own = part + slice * (4 * MB * 64);
    int st = 0;
    for (; st < steps - 2; ++st) {
        if (PARTS && st > 0 && st % 8 == 0) {
#pragma unroll
            for (int m = 0; m < MB; ++m) {
#pragma unroll
                for (int i = 0; i < 4; ++i) own[(4 * m + i) * 64] = st == 8 ? output(m, i) : own[(4 * m + i) * 64] + output(m, i);
#pragma unroll
                for (int x = 0; x < 16; ++x) acc[m][x] = (f4_t){0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
        step(st, std::integral_constant<int, 2>{});
    }
    if (st < steps - 1) step(st++, std::integral_constant<int, 1>{});
    step(st, std::integral_constant<int, 0>{});
    barrier();                                  // (the buffers are used again below)

    const int oy = 2 * ty, ox = 2 * tx;
    const bool two_cols = ox + 1 < p.Wo, two_rows = oy + 1 < p.Ho;
    float *__restrict__ out = p.out + ((long long)img * p.out_bstride + (oy * p.Wo + ox));
    const bool has_resid = p.resid != nullptr;
    const float *__restrict__ resid = has_resid ? p.resid + ((long long)img * p.resid_bstride + (oy * p.Wo + ox)) : nullptr;
    auto load_resid = [&](int ch) {             // (pixels outside the image repeat the tile's first: never stored)
        const float *r = resid + (long long)min(ch, p.N - 1) * p.P;
        f4_t v;
        v[0] = r[0];
        v[1] = two_cols ? r[1] : v[0];
        v[2] = two_rows ? r[p.Wo] : v[0];
        v[3] = two_cols && two_rows ? r[p.Wo + 1] : v[0];
        return v;
    };
    // The transform makes more sums infinite or NaN than those whose own window holds such a value, and sums of four inputs
    // overflow early: rows of a lane with one among their outputs are left out here and computed as plain sums at the end.
    int left_out = 0;
    auto unusual = [&](f4_t v, int row) {
        const bool bad = !((fabsf(v[0]) + fabsf(v[1])) + (fabsf(v[2]) + fabsf(v[3])) < __builtin_inff());
        left_out |= (bad ? 1 : 0) << row;
        return bad;
    };
    auto store = [&](f4_t v, int ch, bool skip) {
        if (!live || ch >= p.N || skip) return;
        float *o = out + (long long)ch * p.P;
        if (two_cols) {
            *reinterpret_cast<f2u_t *>(o) = (f2_t){v[0], v[1]};
            if (two_rows) *reinterpret_cast<f2u_t *>(o + p.Wo) = (f2_t){v[2], v[3]};
        } else {
            o[0] = v[0];
            if (two_rows) o[p.Wo] = v[2];
        }
    };
    auto finish = [&](f4_t v, float bias, f4_t r) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] += bias;
            if (has_resid) v[e] += r[e];
            if (p.relu) v[e] = fmaxf(v[e], 0.0f);
        }
        return v;
    };
    const bool parted = PARTS && steps > 10;    // (the last two steps never start a part)
    const int ch_base = by * (16 * MB) + 4 * k;
    if (p.WK == 1) {
        float bv[4 * MB];
        f4_t rv[4 * MB];
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
            f4_t v = output(r >> 2, r & 3);
            if (parted) v += own[r * 64];
            store(finish(v, bv[r], rv[r]), ch_base + 16 * (r >> 2) + (r & 3), unusual(v, r));
        }
    } else {
        // every wave of a team finishes every WK-th row
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) own[(4 * m + i) * 64] = parted ? own[(4 * m + i) * 64] + output(m, i) : output(m, i);
        // (WK need not divide the rows: 3 is taken too)
        float bv[2 * MB];
        f4_t rv[2 * MB];
#pragma unroll
        for (int r = 0; r < 2 * MB; ++r) {
            if (slice + r * p.WK >= 4 * MB) break;
            const int row = slice + r * p.WK, ch = ch_base + 16 * (row >> 2) + (row & 3);
            bv[r] = p.bias ? p.bias[min(ch, p.N - 1)] : 0.0f;
            if (has_resid) rv[r] = load_resid(ch);
        }
        __syncthreads();
        settle(bv);
        settle(rv);
#pragma unroll
        for (int r = 0; r < 2 * MB; ++r) {
            if (slice + r * p.WK >= 4 * MB) break;
            const int row = slice + r * p.WK;
            f4_t v = part[row * 64];
            for (int s = 1; s < p.WK; ++s) v += part[(s * 4 * MB + row) * 64];
            store(finish(v, bv[r], rv[r]), ch_base + 16 * (row >> 2) + (row & 3), unusual(v, row));
        }
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(left_out != 0) == 0, 1)) return;
#pragma unroll 1
    for (int m = 0; m < MB; ++m) {
        f4_t sums[4];                           // of the four pixels of the tile, rows 4m .. 4m + 3
        if (__builtin_amdgcn_ballot_w64((left_out >> (4 * m) & 15) != 0) == 0) continue;
#pragma unroll 1
        for (int e = 0; e < 4; ++e) {
            const f4_t s = direct_block<false>(ch_base - 4 * k + 16 * m + n, img, min(oy + (e >> 1), p.Ho - 1), min(ox + (e & 1), p.Wo - 1));
#pragma unroll
            for (int x = 0; x < 4; ++x) sums[x] = x == e ? s : sums[x];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ch = ch_base + 16 * m + i;
            const bool skip = (left_out >> (4 * m + i) & 1) == 0;
            f4_t rv = (f4_t){0.0f, 0.0f, 0.0f, 0.0f};
            if (has_resid) rv = load_resid(ch);
            store(finish((f4_t){sums[0][i], sums[1][i], sums[2][i], sums[3][i]}, p.bias ? p.bias[min(ch, p.N - 1)] : 0.0f, rv), ch, skip);
        }
    }
}

const void *wino_block_kernel_function(const KernelId &k) {
    using kernel_fn = void (*)(ConvKParams);
    kernel_fn fn = nullptr;
    if (k.family == KernelId::BLOCK_WINO) {
        const bool parts = k.p[2] != 0, wide = k.p[1] == 4;
        if (k.p[0] == 1 && wide) fn = parts ? static_cast<kernel_fn>(tdc_wino3x3_block_kernel<1, 4, true>) : tdc_wino3x3_block_kernel<1, 4, false>;
        if (k.p[0] == 1 && k.p[1] == 2) fn = parts ? static_cast<kernel_fn>(tdc_wino3x3_block_kernel<1, 2, true>) : tdc_wino3x3_block_kernel<1, 2, false>;
        if (k.p[0] == 2 && wide) fn = parts ? static_cast<kernel_fn>(tdc_wino3x3_block_kernel<2, 4, true>) : tdc_wino3x3_block_kernel<2, 4, false>;
        if (k.p[0] == 2 && k.p[1] == 2 && !parts) fn = tdc_wino3x3_block_kernel<2, 2, false>;
    }
    return reinterpret_cast<const void *>(fn);
}

}  // namespace tdc
