// i4_set_core.h -- the per-row machinery of the i4 matvec set kernel (i4_set.hip), shared with
// the data-flow decode kernel (decode_flow.hip) so that a row gives the same bits in both: the
// activations as exact integers in LDS (stage_x), the per-half-group v_dot4 arithmetic
// (half_group_int), the fixed-order workgroup sum, and the prologue arithmetic (SwiGLU,
// RMSNorm).
#pragma once

#include "i4_lane.h"

namespace tqhip {
namespace {

#ifndef TQ_SET_WAVES
#define TQ_SET_WAVES 8
#endif
constexpr int kSetWaves = TQ_SET_WAVES;     // waves per workgroup
constexpr int kSetThreads = 64 * kSetWaves;
constexpr int kSetMaxSlots = 5;   // wave-per-row slots of 64 half-groups: K <= 5 * 64 * 32

// ---- activations as exact integers -------------------------------------------------------
// Every 64 activations are scaled by a power of two 2^f of their own (their largest |x|
// lands in [2^22, 2^23)) and rounded to the nearest integer: X = x * 2^f rounded,
// |X| < 2^23, the only rounding before the epilogue. X's two's-complement bytes are its
// digits, X = b0 + 256 b1 + 65536 s2 with b0, b1 unsigned and s2 the signed third byte
// (exact while |X| < 2^23). They go to LDS as the byte operands of v_dot4: per 8-element
// block six dwords [byte p][even | odd], "even" holding elements 0, 2, 4, 6 and "odd" 1,
// 3, 5, 7 -- the order in which a code dword's low and high nibbles present the weights.
// Per half-group (32 elements) LDS also holds sum(X) (as a float) and 2^-f.
// P = 4 digits instead of 3 (weight groups of 32, whose rows an FMA kernel summed before, each product
// with all of x's bits): exponents per 32 activations, as an outlier would otherwise cost the group
// beside it bits that its own, perhaps tiny, scale does not excuse; the largest |x| lands in [2^30, 2^31), so
// that elements down to 2^-7 of it keep their 24 bits; and sum(X) and the epilogue are doubles, exact up
// to the one rounding of a half-group's value. Rel L2 against 64-bit sums, 896..9728 elements: normal
// activations P = 3 1.6e-7 to 1.8e-7, P = 4 0.6e-7 to 0.8e-7 (the FMA kernel 1.2e-7 to 1.3e-7). One activation of 64
// 3000 times the others, where it counts for little: in groups of scale 6e-8 0.9e-7 (the FMA kernel
// 1.3e-7), with weights of 0 3.1e-7 (1.2e-7). A host model of 25 bits and an fp32 epilogue gives 3.7e-5 and
// 4.6e-5 with exponents per 64, 1.0e-7 and 3.6e-5 per 32. The bits and the doubles cost 0 to 6% of a
// launch: 896x896 3.01 -> 3.08 us, 9728x2560 9.61 -> 9.81, 151936x896 25.6 -> 27.2.
constexpr int block_bytes(int P) { return 8 * P; }  // one 8-element block: P digit planes x (even, odd) dwords
constexpr int kBlockBytes = block_bytes(3);

// What LDS holds of a half-group: sum(X) and 2^-f.
template <int P>
struct alignas(8) XSum {
    float sum, unscale;
};
template <>
struct alignas(16) XSum<4> {
    double sum;
    float unscale;
};

// f for a block of activations with the largest |x| m; f <= 149 as in group_exponent (every finite x is a
// whole multiple of 2^-149). P = 3: m is raised by one bit of its mantissa, so that no X rounds up to
// 2^23, and halved, so that it stays finite (P = 4: x of 24 bits and a magnitude from 2^24 on has no
// fraction). The instruction gives 0 for the exponent of a zero, whose X are 0 with any f, and of an
// infinity or a NaN, where group_unscale gives the result.
template <int P>
__device__ inline int set_exponent(float m) {
    return P == 4 ? min(31 - __builtin_amdgcn_frexp_expf(m), 149)
                  : min(22 - __builtin_amdgcn_frexp_expf(m * 0.50000006f), 149);
}

// Round to nearest, ties to even. (Ties are common at this width, and rounding them upward in one
// instruction, v_cvt_rpi_i32_f32, adds up over a row: 2.1e-7 to 2.9e-7 at G = 64 and 2.8e-7 to 3.9e-7 at
// G = 128 instead of P = 3's figures above. The launch takes the same time: 2560x9728 7.07 us, with
// integer maxima in stage_x paying for the extra instruction.)
__device__ inline int round_int(float v) {
    int r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(rintf(v)));  // saturates: an infinity is met by group_unscale
    return r;
}

// Thread t converts 16-byte chunk c = t + kSetThreads i (elements 4c .. 4c + 3) of every chunk
// the rows read (c < C): the 16 chunks of 64 elements are one DPP row (16 lanes), the 8
// chunks of a half-group half of one.
template <int P = 3>
__device__ __forceinline__ void stage_x(float4 q, int c, int Kc, int C, unsigned char *xp, XSum<P> *hs) {
    if (c >= Kc) q = make_float4(0.f, 0.f, 0.f, 0.f);  // past K: zeros
    // magnitudes compared as integers: infinities and NaNs are above every finite value
    const auto mag = [](float v) { return static_cast<int>(__float_as_uint(v) & 0x7FFFFFFFu); };
    int mi = max(max(mag(q.x), mag(q.y)), max(mag(q.z), mag(q.w)));
    mi = max(mi, dpp_i<kDppXor1>(mi));
    mi = max(mi, dpp_i<kDppXor2>(mi));
    mi = max(mi, dpp_i<kDppHalfMirror>(mi));
    if constexpr (P == 3) mi = max(mi, dpp_i<kDppMirror>(mi));
    const float m = __int_as_float(mi);  // the largest |x| (not finite if any is not), in the block's 16 or 8 lanes
    const int f = set_exponent<P>(m);
    // the value itself is scaled (2^f is not a finite float for f >= 128; x * 2^f is exact)
    const unsigned X0 = round_int(ldexpf(q.x, f)), X1 = round_int(ldexpf(q.y, f));
    const unsigned X2 = round_int(ldexpf(q.z, f)), X3 = round_int(ldexpf(q.w, f));
    // the half-group's sum(X), in its 8 lanes (P = 4: of the upper halves, and of the lower ones)
    const auto half_sum = [](int v) {
        v += dpp_i<kDppXor1>(v);
        v += dpp_i<kDppXor2>(v);
        return v + dpp_i<kDppHalfMirror>(v);
    };
    XSum<P> h;
    if constexpr (P == 4) {
        const auto hi = [](unsigned v) { return static_cast<int>(v) >> 16; };
        const int up = half_sum(hi(X0) + hi(X1) + hi(X2) + hi(X3));
        const int low = half_sum((X0 & 0xFFFFu) + (X1 & 0xFFFFu) + (X2 & 0xFFFFu) + (X3 & 0xFFFFu));
        h.sum = 65536.0 * up + low;
    } else {
        h.sum = static_cast<float>(half_sum(static_cast<int>(X0 + X1 + X2 + X3)));
    }
    if (c >= C) return;
    // elements 4c + 0, 2 are "even" bytes 2 (c & 1) + 0, 1 of the block; 4c + 1, 3 "odd"
    unsigned char *blk = xp + (c >> 1) * block_bytes(P) + 2 * (c & 1);
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const unsigned sel = 0x0C0C0000u | ((4u + p) << 8) | p;  // byte p of the second, byte p of the first
        *reinterpret_cast<unsigned short *>(blk + 8 * p) = static_cast<unsigned short>(__builtin_amdgcn_perm(X2, X0, sel));
        *reinterpret_cast<unsigned short *>(blk + 8 * p + 4) =
            static_cast<unsigned short>(__builtin_amdgcn_perm(X3, X1, sel));
    }
    h.unscale = group_unscale(m, f);
    if ((c & 7) == 0) hs[c >> 3] = h;
}

// scale * 2^-f * (sum(q * X) - zero * sum(X)) over one half-group: the 16 code bytes cd,
// the group header hd, the half-group's 8 P operand dwords xv (4 blocks) and its
// (sum(X), 2^-f). The digit sums are exact integers (v_dot4: unsigned for the low digits,
// signed for the top one); sum(q * X) = (a0 + 256 a1) + 65536 (a2 [+ 256 a3]) is formed in fp32 (P = 4: in
// double, exactly).
template <int P>
__device__ __forceinline__ float half_group_int(const v4i &cd, unsigned hd, const unsigned (&xv)[8 * P],
                                                const XSum<P> &hs) {
    unsigned a0 = 0, a1 = 0;
    int a2 = 0, a3 = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const unsigned d = static_cast<unsigned>(cd[j]);
        const unsigned lo = d & kNibbles, hi = (d >> 4) & kNibbles;
        const unsigned *x = xv + 2 * P * j;
        a0 = __builtin_amdgcn_udot4(lo, x[0], a0, false);
        a0 = __builtin_amdgcn_udot4(hi, x[1], a0, false);
        a1 = __builtin_amdgcn_udot4(lo, x[2], a1, false);
        a1 = __builtin_amdgcn_udot4(hi, x[3], a1, false);
        if constexpr (P == 3) {
            a2 = __builtin_amdgcn_sdot4(static_cast<int>(lo), static_cast<int>(x[4]), a2, false);
            a2 = __builtin_amdgcn_sdot4(static_cast<int>(hi), static_cast<int>(x[5]), a2, false);
        } else {
            a2 = static_cast<int>(__builtin_amdgcn_udot4(lo, x[4], static_cast<unsigned>(a2), false));
            a2 = static_cast<int>(__builtin_amdgcn_udot4(hi, x[5], static_cast<unsigned>(a2), false));
            a3 = __builtin_amdgcn_sdot4(static_cast<int>(lo), static_cast<int>(x[6]), a3, false);
            a3 = __builtin_amdgcn_sdot4(static_cast<int>(hi), static_cast<int>(x[7]), a3, false);
        }
    }
    const float sc = half_bits(hd), z = half_bits(hd >> 16);
    if constexpr (P == 4) {
        const double V = fma(static_cast<double>(a2 + 256 * a3), 65536.0, static_cast<double>(a0 + a1 * 256u));
        return static_cast<float>(fma(-static_cast<double>(z), hs.sum, V) *
                                  (static_cast<double>(sc) * static_cast<double>(hs.unscale)));
    } else {
        const float V = fmaf(static_cast<float>(a2), 65536.f, static_cast<float>(a0 + a1 * 256u));
        // 2^-f times the exact integer sum first: for tiny activations (f > 126) 2^-f is subnormal and
        // sc * 2^-f could lose its digits, while 2^-f * (...) is still a normal float; for normal
        // products both orders round once and give the same bits.
        return sc * (hs.unscale * fmaf(-z, hs.sum, V));
    }
}

// Rows of at most 32 half-groups (S = 0): R rows per half-wave, 2R per wave, 8R per
// workgroup. Rows of more: R per wave over S slots, kSetWaves R per workgroup.
// Sum of v over the workgroup, in double, in a fixed order (each wave by shuffles, then the
// kSetWaves wave sums in wave order).
__device__ inline double set_block_sum(double v) {
    v = xor_sum_wave(v);
    __shared__ double red[kSetWaves];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = red[0];
#pragma unroll
    for (int w = 1; w < kSetWaves; ++w) t += red[w];
    return t;
}

__device__ inline float4 add4(float4 a, float4 b) {
    return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

// ---- activation prologues ----------------------------------------------------------------
// The arithmetic the set kernel's prologues apply to each 16-byte chunk of activations, shared
// with the data-flow decode kernel so both give the same bits.

// swiglu_ref (kernels/silu/swiglu_ref.cpp): silu(g) * u.
__device__ __forceinline__ float swiglu1(float g, float u) { return (g / (1.0f + expf(-g))) * u; }

__device__ __forceinline__ float4 swiglu4(float4 g, float4 u) {
    return make_float4(swiglu1(g.x, u.x), swiglu1(g.y, u.y), swiglu1(g.z, u.z), swiglu1(g.w, u.w));
}

// One chunk's share of rmsnorm_ref's double sum of squares (kernels/rmsnorm/rmsnorm_ref.cpp).
__device__ __forceinline__ double sq4(float4 h) {
    return static_cast<double>(h.x) * h.x + static_cast<double>(h.y) * h.y + static_cast<double>(h.z) * h.z +
           static_cast<double>(h.w) * h.w;
}

// 1 / sqrt(mean + eps) from the workgroup's double sum of squares over K elements.
__device__ __forceinline__ float rms_scale(double ss, int K, float eps) {
    const float mean_sq = static_cast<float>(ss / K);
    return 1.0f / sqrtf(mean_sq + eps);
}

// (x * scale) * w per element.
__device__ __forceinline__ float4 rms_apply(float4 x, float scale, float4 w) {
    return make_float4((x.x * scale) * w.x, (x.y * scale) * w.y, (x.z * scale) * w.z, (x.w * scale) * w.w);
}

}  // namespace
}  // namespace tqhip
