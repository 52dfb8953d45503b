// Register-blocked 1x1 convolution for batches (tile.alg = 7, tdc_conv1x1_block_kernel): where there are enough pixels to
// fill the chip, the 16x16 blocks of the streamed kernel ask the memory system for every operand far too often, and the
// staged kernel's LDS round trip leaves the matrix pipe idle most of the time.
#include "conv_device.hpp"

namespace tdc {

// ---------------------------------------------------------------------------
// One wave computes 16*MB output channels x 16*NJ pixels on v_mfma_f32_16x16x4_f32, operands straight from global memory
// into registers, one run of 16 input channels ahead of the MFMAs.  The batch is flattened: pixel groups are counted
// through all images, so small images leave no lanes idle.
//   * B operand: column n of MFMA block j is pixel NJ*n + j of the wave's stretch, so ONE 128-bit (NJ = 4) request per lane
//     feeds NJ MFMA blocks, and the NJ accumulators of a lane are NJ neighbouring pixels: 128-bit stores.  A group that
//     would run past the end of its image starts earlier and leaves the pixels of its neighbour alone.  GEN: pixels one by
//     one (strided convolutions, images of fewer than NJ pixels).
//   * A operand: the packed weights of the streamed kernel, [16 channels][run][lane][4], one 128-bit request for four K-steps.
//   * MB*NJ MFMAs per K-step from 1 + MB/4 requests: at MB = 2, NJ = 4 the address path of a compute unit is busy three eighths
//     of the time the matrix pipe is, where the 16x16 blocks of the streamed kernel need it twice as long as the pipe.
// A workgroup is WM x WN waves over channels and pixels (they share operands through the L1), times WK waves that split
// the input channels and add their partial blocks through LDS in slice order.
// AFF: per-channel affine (+ ReLU) on the input, in registers.
// Bound: the matrix pipe in the steady state (125-140 of 154 TFLOP/s measured from the slope over input channels), plus
// 6-8 us at 16 MB of output for the launch, the first operands and the stores, which end together.  Against the best tile
// of the other families (launch-to-launch, one box): 512 -> 128 @28 batch 32 51.4 -> 32.6 us, 64 -> 256 @56 batch 32
// 58.3 -> 38.8, 2048 -> 256 @7 batch 64 68.3 -> 36.5, 256 -> 128 @56 batch 8 31.6 -> 19.5, 992 -> 128 @14 batch 8
// 12.9 -> 7.8; even at about 4 us, slower below (0.2-0.3 us of index arithmetic in front of the first request).
// Blocks of 64 channels per wave (mb = 4) were slower everywhere: too few waves to cover each other's start and end.
// ---------------------------------------------------------------------------
// PART: the products of 8, 16 or 32 channels are summed apart, 0: all of a wave's in one chain, whose error grows with the root
// of its length.  They cost 1.044, 1.036 and 1.013 of the time of PART = 0 (66 shapes, on average), and are taken where the tile
// that would run otherwise has shorter chains: 304 -> 176 @53 in one chain 7.4 us and an error of 3.1e-7 against 64-bit sums, on the
// streamed kernel 9.2 us and 1.1e-7, in parts of 32 7.6 us and 1.2e-7.
template <int MB, int NJ, bool AFF, bool GEN, int PART>
__global__ void __launch_bounds__(512, 2) tdc_conv1x1_block_kernel(const ConvKParams p) {
    using G = PixelGroup<NJ>;
    using px_t = typename G::reg_t;
    extern __shared__ __align__(16) float lds[];
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
    const int t1 = fdiv(wave, p.fd_wk);
    const int slice = wave - t1 * p.WK;         // of the input channels
    const int wm = fdiv(t1, p.fd_wn);
    const int wn = t1 - wm * p.WN;
    const int k = lane >> 4, n = lane & 15;

    // this lane's pixels: of image b, relative to the wave's first image b0 (32-bit offsets from there)
    constexpr int NG = GEN ? NJ : 1;            // separately addressed pixel groups per lane
    const int u0 = (bx * p.WN + wn) * (16 * NG);
    const int b0 = fdiv(min(u0, p.units - 1), p.fd_units);
    int img[NG], pix[NG], fresh[NG];            // image, first pixel, first pixel of the group that no other group stores
    unsigned voff[NG];
    const unsigned HW4 = (unsigned)(p.H * p.W) * 4u;
#pragma unroll
    for (int j = 0; j < NG; ++j) {
        const int u = u0 + 16 * j + n;
        const int uc = min(u, p.units - 1);
        img[j] = fdiv(uc, p.fd_units);
        const int g = uc - img[j] * p.fd_units.d;
        unsigned src;
        if constexpr (GEN) {
            pix[j] = g;
            fresh[j] = u < p.units ? 0 : 1;
            const int oy = fdiv(g, p.fd_wtw);
            src = (unsigned)((oy * p.W + (g - oy * p.fd_wtw.d)) * p.stride);
        } else {
            pix[j] = min(g * NJ, p.P - NJ);
            fresh[j] = u < p.units ? g * NJ - pix[j] : NJ;
            src = (unsigned)pix[j];
        }
        voff[j] = ((unsigned)(img[j] - b0) * (unsigned)p.in_bstride + src) * 4u + (unsigned)(4 * k) * HW4;
    }
    const __amdgpu_buffer_rsrc_t in_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(p.in + (long long)b0 * p.in_bstride), (short)0, OOB_OFFSET, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.wpk), (short)0, (int)p.wpk_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t aff_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.in_aff), (short)0, p.CCH * 8, 0x00020000);

    const int runs_all = p.CCH >> 4;            // runs of the packed weights (padded to a multiple of WK)
    const int rpw = p.CPW >> 4;                 // ... per wave
    const int q_begin = slice * rpw, q_end = min(q_begin + rpw, (p.C + 15) >> 4);
    const int a_base = (by * p.WM + wm) * MB * runs_all * 1024;

    struct Run {
        f4_t a[MB];
        float b[4][NJ];
        f4_t sc, sh;
    };
    auto load = [&](Run &r, int q) {
#pragma unroll
        for (int m = 0; m < MB; ++m)
            r.a[m] = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, lane * 16, a_base + (m * runs_all + q) * 1024, 0));
        if constexpr (AFF) {
            r.sc = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(aff_rsrc, (16 * q + 4 * k) * 4, 0, 0));
            r.sh = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(aff_rsrc, (p.CCH + 16 * q + 4 * k) * 4, 0, 0));
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            // (channels past C: an out-of-range vector offset reads zero)
            const bool real = 16 * q + 4 * k + s < p.C;
            const int soff = (int)((unsigned)(16 * q + s) * HW4);
            if constexpr (GEN) {
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    r.b[s][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(in_rsrc, real ? (int)voff[j] : OOB_OFFSET, soff, 0));
            } else {
                const px_t v = G::load(in_rsrc, real ? (int)voff[0] : OOB_OFFSET, soff);
#pragma unroll
                for (int j = 0; j < NJ; ++j) r.b[s][j] = v[j];
            }
        }
        __builtin_amdgcn_sched_barrier(0);      // the requests stay in front of the MFMAs they run under
    };
    // The products of half a run, of one or of two runs are summed by themselves and then added to `acc`: those of single runs,
    // where they are few MFMAs, a run later, when their sums have long left the matrix pipe.
    constexpr bool LATE = PART == 16 && MB * NJ <= 4;
    typedef f4_t Sums[MB][NJ];
    Sums acc, s0, s1;
    auto clear = [&](Sums &x) {
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int j = 0; j < NJ; ++j) x[m][j] = (f4_t){0.0f, 0.0f, 0.0f, 0.0f};
    };
    auto add = [&](const Sums &x) {
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[m][j] += x[m][j];
        __builtin_amdgcn_sched_barrier(0);
    };
    // K-steps first ... first + count - 1 of a run; `fresh`: a part begins
    auto multiply = [&](Run &r, Sums &sum, bool fresh, int first, int count) {
#pragma unroll
        for (int s = first; s < first + count; ++s) {
            if constexpr (AFF) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    r.b[s][j] = r.b[s][j] * r.sc[s] + r.sh[s];
                    if (p.in_relu) r.b[s][j] = fmaxf(r.b[s][j], 0.0f);
                }
            }
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    sum[m][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.a[m][s], r.b[s][j], fresh && s == first ? (f4_t){0.0f, 0.0f, 0.0f, 0.0f} : sum[m][j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // the even and the odd runs of the wave; `last`: no odd run follows
    auto even = [&](Run &r, bool last) {
        if constexpr (PART == 0) {
            multiply(r, acc, false, 0, 4);
        } else if constexpr (PART == 8) {
            multiply(r, s0, true, 0, 2);
            multiply(r, s1, true, 2, 2);
            add(s0);
            add(s1);
        } else {
            multiply(r, s0, true, 0, 4);
            if constexpr (LATE) add(s1);
            else if (PART == 16 || last) add(s0);
        }
    };
    auto odd = [&](Run &r) {
        if constexpr (PART == 0 || PART == 8) {
            even(r, true);
        } else {
            multiply(r, LATE ? s1 : s0, PART == 16, 0, 4);
            add(s0);
        }
    };
    clear(acc);
    if constexpr (LATE) clear(s1);
    if (q_begin < q_end) {
        Run r0, r1;
        load(r0, q_begin);
        int q = q_begin;
        for (; q + 2 < q_end; q += 2) {
            load(r1, q + 1);
            even(r0, false);
            load(r0, q + 2);
            odd(r1);
        }
        if (q + 1 < q_end) {
            load(r1, q + 1);
            even(r0, false);
            odd(r1);
            if constexpr (LATE) add(s1);
        } else {
            even(r0, true);
            if constexpr (LATE) add(s0);
        }
    }

    // One output row of this lane: channel ch, NJ pixels.
    const bool has_resid = p.resid != nullptr;
    const float *__restrict__ resid[NG];
    float *__restrict__ out[NG];
#pragma unroll
    for (int j = 0; j < NG; ++j) {
        out[j] = p.out + ((long long)img[j] * p.out_bstride + pix[j]);
        resid[j] = has_resid ? p.resid + ((long long)img[j] * p.resid_bstride + pix[j]) : nullptr;
    }
    auto load_resid = [&](int ch) {
        px_t rv;
        const long long off = (long long)min(ch, p.N - 1) * p.P;
        if constexpr (GEN) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) rv[j] = resid[j][off];
        } else {
            rv = *reinterpret_cast<const typename G::mem_t *>(resid[0] + off);
        }
        return rv;
    };
    auto store = [&](px_t v, int ch) {
        if (ch >= p.N) return;
        const long long off = (long long)ch * p.P;
        if constexpr (GEN) {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                if (!fresh[j]) out[j][off] = v[j];
        } else if (fresh[0] == 0) {
            *reinterpret_cast<typename G::mem_t *>(out[0] + off) = v;
        } else {
#pragma unroll
            for (int j = 1; j < NJ; ++j)
                if (j >= fresh[0]) out[0][off + j] = v[j];
        }
    };
    const int ch_base = (by * p.WM + wm) * (16 * MB) + 4 * k;
    // All addends are requested and settled before the first store (see settle): the bias in one branch and first, then the residual,
    // and the whole once more without a residual, whose addends a shared copy would wait for (as one lambda for both it takes more
    // registers and up to 4 % longer).  Against loads block by block, 500 random layers: 0.95 to 0.98 of the time, by kind of tile, and
    // one of 359 layers more than 4 % slower; with a branch for every bias value and one wait for bias and residual it was 0.96 to 1.02,
    // with a residual up to 1.16 (32 -> 176 @32 batch 13 5.9 -> 6.9 us).  Where several waves share the input channels, below, a row at a
    // time behind the barrier is as fast as any: unrolled and requested in front of it 1.00 to 1.04.
    if (p.WK == 1) {
        float bv[4 * MB];
        if (has_resid) {
            px_t rv[4 * MB];
#pragma unroll
            for (int r = 0; r < 4 * MB; ++r) bv[r] = 0.0f;
            if (p.bias) {
#pragma unroll
                for (int r = 0; r < 4 * MB; ++r) bv[r] = p.bias[min(ch_base + 16 * (r >> 2) + (r & 3), p.N - 1)];
            }
            settle(bv);
#pragma unroll
            for (int r = 0; r < 4 * MB; ++r) rv[r] = load_resid(ch_base + 16 * (r >> 2) + (r & 3));
            settle(rv);
#pragma unroll
            for (int r = 0; r < 4 * MB; ++r) {
                px_t v;
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    v[j] = acc[r >> 2][j][r & 3] + bv[r];
                    v[j] += rv[r][j];
                    if (p.relu) v[j] = fmaxf(v[j], 0.0f);
                }
                store(v, ch_base + 16 * (r >> 2) + (r & 3));
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4 * MB; ++r) bv[r] = 0.0f;
            if (p.bias) {
#pragma unroll
                for (int r = 0; r < 4 * MB; ++r) bv[r] = p.bias[min(ch_base + 16 * (r >> 2) + (r & 3), p.N - 1)];
            }
            settle(bv);
#pragma unroll
            for (int r = 0; r < 4 * MB; ++r) {
                px_t v;
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    v[j] = acc[r >> 2][j][r & 3] + bv[r];
                    if (p.relu) v[j] = fmaxf(v[j], 0.0f);
                }
                store(v, ch_base + 16 * (r >> 2) + (r & 3));
            }
        }
        return;
    }
    // the WK waves of one (wm, wn) leave their rows in LDS, [slice][row = 4m + i][lane], and finish every WK-th row each
    px_t *part = reinterpret_cast<px_t *>(lds) + (size_t)(t1 * p.WK) * (4 * MB * 64) + lane;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            px_t v;
#pragma unroll
            for (int j = 0; j < NJ; ++j) v[j] = acc[m][j][i];
            part[(slice * 4 * MB + 4 * m + i) * 64] = v;
        }
    __syncthreads();
    for (int row = slice; row < 4 * MB; row += p.WK) {
        const int ch = ch_base + 16 * (row >> 2) + (row & 3);
        px_t rv;
        if (has_resid) rv = load_resid(ch);
        const float bv = p.bias ? p.bias[min(ch, p.N - 1)] : 0.0f;
        px_t v = part[row * 64];
        for (int s = 1; s < p.WK; ++s) v += part[(s * 4 * MB + row) * 64];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            v[j] += bv;
            if (has_resid) v[j] += rv[j];
            if (p.relu) v[j] = fmaxf(v[j], 0.0f);
        }
        store(v, ch);
    }
}

using kernel_fn = void (*)(ConvKParams);

template <int MB, int NJ, int PART>
static kernel_fn pick_block(bool aff, bool gen) {
    return aff ? (gen ? static_cast<kernel_fn>(tdc_conv1x1_block_kernel<MB, NJ, true, true, PART>) : tdc_conv1x1_block_kernel<MB, NJ, true, false, PART>)
               : (gen ? static_cast<kernel_fn>(tdc_conv1x1_block_kernel<MB, NJ, false, true, PART>) : tdc_conv1x1_block_kernel<MB, NJ, false, false, PART>);
}

template <int PART>
static kernel_fn pick_block(int mb, int nj, bool aff, bool gen) {
    if (nj == 4) return mb == 1 ? pick_block<1, 4, PART>(aff, gen) : mb == 2 ? pick_block<2, 4, PART>(aff, gen) : nullptr;
    if (nj == 2) return mb == 1 ? pick_block<1, 2, PART>(aff, gen) : mb == 2 ? pick_block<2, 2, PART>(aff, gen) : nullptr;
    return nullptr;
}

const void *block_kernel_function(const KernelId &k) {
    if (k.family != KernelId::BLOCK_1x1) return nullptr;
    const bool aff = k.p[2] != 0, gen = k.p[3] != 0;
    const kernel_fn fn = k.p[4] == 0    ? pick_block<0>(k.p[0], k.p[1], aff, gen)
                         : k.p[4] == 8  ? pick_block<8>(k.p[0], k.p[1], aff, gen)
                         : k.p[4] == 16 ? pick_block<16>(k.p[0], k.p[1], aff, gen)
                         : k.p[4] == 32 ? pick_block<32>(k.p[0], k.p[1], aff, gen) : nullptr;
    return reinterpret_cast<const void *>(fn);
}

}  // namespace tdc
