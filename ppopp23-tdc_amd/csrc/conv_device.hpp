// Device-side pieces shared by the convolution kernels: MFMA wrappers, the multiply-high division, the common
// epilogue of a lane that holds four channels of a pixel, the kernel-argument touch, and the time-stamp macros of
// the profiling build.  Included by every conv_*.hip with kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "tdc_internal.hpp"

#ifndef TDC_TOUCH_KERNARGS
#define TDC_TOUCH_KERNARGS 1
#endif

// Profiling build only (make STAMPS=1): every wave records s_memrealtime (the 100 MHz constant clock, comparable
// across compute units and dies) at the boundaries of its phases and leaves the eight values in a plan-owned buffer,
// [workgroup][wave][8].  The product build compiles none of it.
#ifndef TDC_STAMPS
#define TDC_STAMPS 0
#endif
#if TDC_STAMPS
#define TDC_STAMP_DECL unsigned long long tdc_stamp_[8] = {0, 0, 0, 0, 0, 0, 0, 0}
#define TDC_STAMP(i) tdc_stamp_[i] = __builtin_amdgcn_s_memrealtime()
#define TDC_STAMP_FLUSH(p, wg, wave, lane)                                                             \
    do {                                                                                               \
        if ((p).stamps && (lane) == 0) {                                                               \
            unsigned long long *dst_ = (p).stamps + ((size_t)(wg) * 16 + (wave)) * 8;                   \
            for (int i_ = 0; i_ < 8; ++i_) dst_[i_] = tdc_stamp_[i_];                                   \
        }                                                                                              \
    } while (0)
#else
#define TDC_STAMP_DECL
#define TDC_STAMP(i)
#define TDC_STAMP_FLUSH(p, wg, wave, lane)
#endif

namespace tdc {

typedef float f2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef float f16_t __attribute__((ext_vector_type(16)));
// (for places that need not be aligned: images with an odd number of pixels, channel slices)
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u_t __attribute__((ext_vector_type(2), aligned(4)));
typedef __attribute__((address_space(3))) void *lds_ptr_t;

// N neighbouring pixels of a plane, one request.
template <int N>
struct PixelGroup;
template <>
struct PixelGroup<4> {
    using mem_t = f4u_t;
    using reg_t = f4_t;
    static __device__ __forceinline__ reg_t load(__amdgpu_buffer_rsrc_t rsrc, int voff, int soff) {
        return __builtin_bit_cast(reg_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff, soff, 0));
    }
};
template <>
struct PixelGroup<2> {
    using mem_t = f2u_t;
    using reg_t = f2_t;
    static __device__ __forceinline__ reg_t load(__amdgpu_buffer_rsrc_t rsrc, int voff, int soff) {
        return __builtin_bit_cast(reg_t, __builtin_amdgcn_raw_buffer_load_b64(rsrc, voff, soff, 0));
    }
};

template <int MF>
struct Mfma;

// v_mfma_f32_32x32x2_f32: A lane l = A[l%32][l/32], B lane l = B[l/32][l%32],
// D vgpr v lane l = D[8*(v/4) + 4*(l/32) + v%4][l%32].
template <>
struct Mfma<32> {
    using acc_t = f16_t;
    static constexpr int NACC = 16;
    static constexpr int KC = 2;
    static __device__ __forceinline__ acc_t run(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int v, int lane) {
        return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
    }
    static __device__ __forceinline__ int col(int lane) { return lane & 31; }
    static __device__ __forceinline__ int ksub(int lane) { return lane >> 5; }
};

// v_mfma_f32_16x16x4_f32: A lane l = A[l%16][l/16], B lane l = B[l/16][l%16],
// D vgpr v lane l = D[4*(l/16) + v][l%16].
template <>
struct Mfma<16> {
    using acc_t = f4_t;
    static constexpr int NACC = 4;
    static constexpr int KC = 4;
    static __device__ __forceinline__ acc_t run(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int v, int lane) { return 4 * (lane >> 4) + v; }
    static __device__ __forceinline__ int col(int lane) { return lane & 15; }
    static __device__ __forceinline__ int ksub(int lane) { return lane >> 4; }
};

// TAPS_WINO: 3x3 / stride 1 as Winograd F(2x2,3x3).  A pixel lane holds one 2x2 output tile; per four input
// channels a wave reads the 4x4 input patch of its tile from the SAME zero-haloed LDS window the direct path
// uses, transforms it in registers (V = B^T d B, 32 additions), and feeds 16 MFMAs — one per position of the
// transformed domain, against weights U = G g G^T prepared on the host — where the direct path needs 36 for
// the same four pixels.  The 16 accumulators of a lane are combined at the end (Y = A^T M A, in registers:
// every lane holds all 16 positions of its tile) into the 2x2 outputs.
// TAPS_3x3G: the direct 3x3 loop with its weights read from global memory straight into registers (like the
// Winograd path) instead of being staged in LDS: the LDS then holds input only and a pass can take all input channels.
// (the TAPS_* values themselves are declared next to KernelId)

constexpr int OOB_OFFSET = 0x7ffffff0;  // beyond any buffer: the load returns zero

// Output stores (plain: the lines stay in the die's L2 until the kernel ends).
__device__ __forceinline__ void store_out(float *p, float v) { *p = v; }
__device__ __forceinline__ void store_out(float *p, f4_t v) { *reinterpret_cast<f4_t *>(p) = v; }
typedef float f2_store_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store_out(float *p, f2_store_t v) { *reinterpret_cast<f2_store_t *>(p) = v; }

__device__ __forceinline__ int fdiv(int n, const FastDiv &f) {
    return (int)(__umulhi((unsigned)n, f.m) + ((unsigned)n & f.pass));
}

// Epilogue of a lane that holds four consecutive output channels (from ch0) of one pixel: + bias, + residual, ReLU,
// store.  All eight loads are requested before the first value is needed — one memory round trip for the lane
// instead of one per load (written naively, every load sits behind the previous channel's store, which it might alias).
__device__ __forceinline__ void finish_four_channels(const f4_t &acc, int ch0, int N, long long P, long long pix,
                                                     const float *__restrict__ bias, const float *__restrict__ resid,
                                                     int relu, float *__restrict__ out) {
    float bv[4] = {0.0f, 0.0f, 0.0f, 0.0f}, rv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (bias) {
#pragma unroll
        for (int i = 0; i < 4; ++i) bv[i] = bias[min(ch0 + i, N - 1)];
    }
    if (resid) {
#pragma unroll
        for (int i = 0; i < 4; ++i) rv[i] = resid[(long long)min(ch0 + i, N - 1) * P + pix];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (ch0 + i >= N) continue;
        float val = acc[i] + bv[i];
        val += rv[i];
        if (relu) val = fmaxf(val, 0.0f);
        store_out(out + ((long long)(ch0 + i) * P + pix), val);
    }
}

// Loads and stores of a wave are counted together and in order, and bias and residual are loaded in branches: where a value of
// theirs is first used behind a store, the compiler waits for that store too, a memory round trip (about 1 us) per block of
// outputs.  So kernels whose lanes finish several blocks request all of them first and settle them here, in front of the
// first store: the one wait stands here, and nothing behind it needs another.  (Tucker block 512-128-128-512 @28 batch 32 121.6 ->
// 116.1 us, Tucker ResNet-18 batch 32 822 -> 800.)
template <int N>
__device__ __forceinline__ void settle(float (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
}
template <int N, typename V>
__device__ __forceinline__ void settle(V (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
}

// Four consecutive channels (from ch0) of one pixel with addends that are in registers (see settle).
__device__ __forceinline__ void store_four_channels(const f4_t &acc, int ch0, int N, long long P, long long pix, const float (&bias)[4],
                                                    bool has_resid, const float (&resid)[4], int relu, float *__restrict__ out) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (ch0 + i >= N) continue;
        float val = acc[i] + bias[i];
        if (has_resid) val += resid[i];
        if (relu) val = fmaxf(val, 0.0f);
        store_out(out + ((long long)(ch0 + i) * P + pix), val);
    }
}

// The kernel arguments (about 530 bytes) are read through the scalar cache.  Left alone, the compiler fetches them in
// several dependent batches, and every batch that touches a cache line for the first time costs a round trip to L2
// before the first request can go out.  Touch every line of the argument block at once: whatever order the compiler
// then loads the values in, it hits the scalar cache.
__device__ __forceinline__ void touch_kernel_arguments() {
    if constexpr (TDC_TOUCH_KERNARGS) {
        static_assert(sizeof(ConvKParams) > 8 * 64 && sizeof(ConvKParams) <= 9 * 64 + 8 * TDC_STAMPS, "touch exactly the lines of the argument block");
        const auto kargs = __builtin_amdgcn_kernarg_segment_ptr();
        unsigned t0, t1, t2, t3, t4, t5, t6, t7, t8;
        asm volatile(
            "s_load_dword %0, %9, 0x0\n\ts_load_dword %1, %9, 0x40\n\ts_load_dword %2, %9, 0x80\n\t"
            "s_load_dword %3, %9, 0xc0\n\ts_load_dword %4, %9, 0x100\n\ts_load_dword %5, %9, 0x140\n\t"
            "s_load_dword %6, %9, 0x180\n\ts_load_dword %7, %9, 0x1c0\n\ts_load_dword %8, %9, 0x200\n\ts_waitcnt lgkmcnt(0)"
            : "=&s"(t0), "=&s"(t1), "=&s"(t2), "=&s"(t3), "=&s"(t4), "=&s"(t5), "=&s"(t6), "=&s"(t7), "=&s"(t8)
            : "s"(kargs)
            : "memory");
    }
}

// Where image `img` of the batch starts in the input, the output and the residual.  A compute unit has ONE scalar
// unit for all its waves, and in the streamed kernels every wave's scalar prologue sits on the path to its first
// memory request (16 waves x ~130 scalar instructions is most of a microsecond), so the 64-bit stride products — a
// quarter of that prologue — are skipped for the first image, which is the only one in a single-image launch.
struct ImageBase {
    const float *in;
    float *out;
    const float *resid;
};
__device__ __forceinline__ ImageBase image_base(const ConvKParams &p, int img) {
    ImageBase b{p.in, p.out, p.resid};
    if (__builtin_expect(img != 0, 0)) {   // (wave-uniform: a scalar branch)
        b.in += (long long)img * p.in_bstride;
        b.out += (long long)img * p.out_bstride;
        if (b.resid) b.resid += (long long)img * p.resid_bstride;
    }
    return b;
}

// The kernel arguments, read when they are used: what only the end of a kernel needs would otherwise be loaded at its start and cost
// scalar registers all the way.  (In a kernel whose only argument is the ConvKParams.)
typedef const __attribute__((address_space(4))) ConvKParams *late_args_t;
__device__ __forceinline__ late_args_t late_arguments() {
    late_args_t args = (late_args_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    return args;
}

// A block of 16 channels x 16 pixels as plain fp32 sums over the weights as the caller gave them (w_raw, OIHW): for the rare
// outputs that a transform or a split of the operands cannot represent.  Lane (k = l / 16, n = l % 16) names channel `ch` (row n
// of the block; past N: any) and output pixel (oy, ox) of image `img` (column n); it gets rows 4k .. 4k + 3 of its pixel.  Every
// lane of the wave must call it, in a kernel whose only argument is the ConvKParams.  Padding counts (0 * inf).  AFF: the input affine of a 1x1 convolution.
// Bound: latency, sixteen channels in flight; a wave in which it runs takes several times as long.
template <bool AFF>
__device__ __forceinline__ f4_t direct_block(int ch, int img, int oy, int ox) {
    const auto &p = *late_arguments();
    const int k = (threadIdx.x >> 4) & 3;
    const int taps = p.KH * p.KW, plane = p.H * p.W;
    const float *const w = p.w_raw + (size_t)min(ch, p.N - 1) * p.C * taps;
    const float *const src = p.in + (long long)img * p.in_bstride;
    f4_t part[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) part[u] = (f4_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int tap = 0; tap < taps; ++tap) {
        const int kr = tap / p.KW;
        const int y = oy * p.stride + kr * p.dil - p.pad, x = ox * p.stride + (tap - kr * p.KW) * p.dil - p.pad;
        const bool inside = (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.W;
        const int pix = inside ? y * p.W + x : 0;
#pragma unroll 1
        for (int c0 = k; c0 < p.C + k; c0 += 16) {      // (the same number of turns for every lane)
            float a[4], b[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int c = c0 + 4 * u, cc = min(c, p.C - 1);
                a[u] = w[(size_t)cc * taps + tap];
                b[u] = src[(size_t)cc * plane + pix];
                if constexpr (AFF) {
                    const float *const aff = p.in_aff + (size_t)(cc / p.CCH) * 2 * p.CCH + cc % p.CCH;
                    b[u] = b[u] * aff[0] + aff[p.CCH];
                    if (p.in_relu) b[u] = fmaxf(b[u], 0.0f);
                }
                a[u] = c < p.C ? a[u] : 0.0f;
                b[u] = c < p.C && inside ? b[u] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) part[u] = Mfma<16>::run(a[u], b[u], part[u]);
        }
    }
    return (part[0] + part[1]) + (part[2] + part[3]);
}

}  // namespace tdc
