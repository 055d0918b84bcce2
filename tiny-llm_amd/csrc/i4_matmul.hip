// i4_matmul.hip -- batched-prefill i4 dequant-GEMM for gfx950.
//
// Y[M,N] = W_i4[M,K] * X[K,N] with X and Y column-major (x[n*K+k], y[n*M+m]),
// the contract of the reference's matmul_i4_ref (kernels/matvec/matmul_i4_ref.cpp:53-114):
// W row m, element k dequantizes to (q - zero) * scale of its group, in fp32.
//
// MFMA path (group size a multiple of 32):
//   1. x_to_f16: every token column n of X is scaled by an exact power of two
//      2^e_n (its largest |x| lands in [2^14, 2^15)) and rounded to fp16,
//      zero-padded to a multiple of 64 along K. The scale keeps fp16 clear of
//      overflow and gives every token the full 11-bit significand; 2^-e_n is
//      applied exactly in the epilogue.
//   2. i4_matmul_direct: workgroup tiles of 32 weight rows a wave x BN tokens, 64 K elements per
//      step. Each lane loads its row's codes and group header straight into registers, the fp16 X
//      slice comes by DMA into an LDS ring, both some steps ahead; the A operands are
//      dequantized in registers and contracted with v_mfma_f32_32x32x16_f16 (fp32
//      accumulation).
//      fp16 and bf16 MFMA run at the same rate on gfx950; fp16 keeps 8x
//      finer rounding of both operands.
// Up to 32 tokens at G = 64 (16-byte aligned X, K % 4 == 0, K <= 114240): one launch that converts X
// itself and splits K over workgroups (section 3 below).
// Other group sizes: one i4 matvec per token column.

#include "few_token_slices.h"
#include "i4_lane.h"
#include "tq_common.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace tqhip {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16x __attribute__((ext_vector_type(16)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));

constexpr int kStepK = 64;             // K elements per main-loop step

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void *base, size_t bytes) {
    const int nrec = bytes > 0xFFFFFFFFull ? -1 : static_cast<int>(static_cast<unsigned>(bytes));
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), static_cast<short>(0), nrec, kBufferFlags);
}

// q * s + nzs in fp32 is exact (q has 4 bits, s and the zero 11: q * s and nzs = -zero * s
// are exact products and their sum needs at most 24 bits), so rounding it to fp16 with
// v_cvt_pk_f16_f32 (round to nearest even) rounds once, as v_fma_mix would; measured on
// MI355X v_fma_mix issues at a third to a quarter of the rate of v_fma_f32.
// (asm: left to itself the compiler folds the fp32 FMA and the conversion back into v_fma_mix)
__device__ inline unsigned pair_f16(float a, float b) {
    unsigned r;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// ---- 1. X (fp32, column n = token) -> fp16 * 2^e_n, rows padded to Kp.
// One workgroup per token; the column is read once into registers (Kp <= 256 *
// kXRegs), its max taken, then converted and stored. Longer columns: two passes.
// PERM: within every 8 elements, element e goes to position ((e & 3) << 1) | (e >> 2), the
// k-slot order in which the packed-fp16 dequantization leaves a code dword's elements.
__device__ __forceinline__ int x_pos(int k, bool perm) {
    return perm ? (k & ~7) | ((k & 3) << 1) | ((k >> 2) & 1) : k;
}
constexpr int kXRegs = 16;
template <bool PERM>
__global__ __launch_bounds__(256) void x_to_f16(const float *__restrict__ x, int K, int Kp, _Float16 *__restrict__ xh,
                                                  float *__restrict__ xinv) {
    const int n = blockIdx.x;
    const float *xc = x + static_cast<size_t>(n) * K;
    float v[kXRegs];
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < kXRegs; ++i) {
        const int k = threadIdx.x + i * 256;
        v[i] = k < K ? xc[k] : 0.f;
        m = fmaxf(m, fabsf(v[i]));
    }
    m = xor_max_wave(m);
    __shared__ float wm[4];
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(wm[0], wm[1]), fmaxf(wm[2], wm[3]));
    int e = 0;
    if (m > 0.f && m <= 3.0e38f) {  // finite, nonzero: max * 2^e in [2^14, 2^15)
        int E;
        frexpf(m, &E);
        e = min(max(15 - E, -120), 120);
    }
    _Float16 *hc = xh + static_cast<size_t>(n) * Kp;
#pragma unroll
    for (int i = 0; i < kXRegs; ++i) {
        const int k = threadIdx.x + i * 256;
        if (k < Kp) hc[x_pos(k, PERM)] = static_cast<_Float16>(ldexpf(v[i], e));
    }
    if (threadIdx.x == 0) xinv[n] = ldexpf(1.f, -e);
}

// x_to_f16 for K % 4 == 0 and x 16-byte aligned: thread t takes 8-element chunks t + 256 i, i < CH
// (two 16-byte loads each, all in flight together) and stores each chunk's 8 fp16 values, in the
// chunk's slot order, with one 16-byte store. The same exponent and the same per-element rounding
// as x_to_f16. Bound by memory: rows of 9728 at 3001 tokens (175 MB) 32 us, where two scalar passes
// (x_to_f16_long, still used for rows past 16384 and unaligned ones) take 77.
constexpr int kXVecMax = 8;  // chunks per thread: rows of up to 2048 kXVecMax elements
template <bool PERM, int CH>
__global__ __launch_bounds__(256) void x_to_f16_vec(const float *__restrict__ x, int K, int Kp,
                                                      _Float16 *__restrict__ xh, float *__restrict__ xinv) {
    const int n = blockIdx.x;
    const float4 *xc = reinterpret_cast<const float4 *>(x + static_cast<size_t>(n) * K);
    float v[CH][8];
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = threadIdx.x + 256 * i;  // elements 8c .. 8c + 7
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool ok = 8 * c + 4 * h < K;  // K % 4 == 0: a float4 is all in or all out
            const float4 q = ok ? xc[2 * c + h] : make_float4(0.f, 0.f, 0.f, 0.f);
            v[i][4 * h] = q.x;
            v[i][4 * h + 1] = q.y;
            v[i][4 * h + 2] = q.z;
            v[i][4 * h + 3] = q.w;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(v[i][e]));
    }
    m = xor_max_wave(m);
    __shared__ float wm[4];
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(wm[0], wm[1]), fmaxf(wm[2], wm[3]));
    int e = 0;
    if (m > 0.f && m <= 3.0e38f) {  // finite, nonzero: max * 2^e in [2^14, 2^15)
        int E;
        frexpf(m, &E);
        e = min(max(15 - E, -120), 120);
    }
    uint4 *hc = reinterpret_cast<uint4 *>(xh + static_cast<size_t>(n) * Kp);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = threadIdx.x + 256 * i;
        if (8 * c >= Kp) continue;
        unsigned short o[8];
#pragma unroll
        for (int el = 0; el < 8; ++el)
            o[x_pos(el, PERM)] = __builtin_bit_cast(unsigned short, static_cast<_Float16>(ldexpf(v[i][el], e)));
        hc[c] = make_uint4(o[0] | (static_cast<unsigned>(o[1]) << 16), o[2] | (static_cast<unsigned>(o[3]) << 16),
                           o[4] | (static_cast<unsigned>(o[5]) << 16), o[6] | (static_cast<unsigned>(o[7]) << 16));
    }
    if (threadIdx.x == 0) xinv[n] = ldexpf(1.f, -e);
}

template <bool PERM>
__global__ __launch_bounds__(256) void x_to_f16_long(const float *__restrict__ x, int K, int Kp,
                                                       _Float16 *__restrict__ xh, float *__restrict__ xinv) {
    const int n = blockIdx.x;
    const float *xc = x + static_cast<size_t>(n) * K;
    float m = 0.f;
    for (int k = threadIdx.x; k < K; k += blockDim.x) m = fmaxf(m, fabsf(xc[k]));
    m = xor_max_wave(m);
    __shared__ float wm[4];
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(wm[0], wm[1]), fmaxf(wm[2], wm[3]));
    int e = 0;
    if (m > 0.f && m <= 3.0e38f) {
        int E;
        frexpf(m, &E);
        e = min(max(15 - E, -120), 120);
    }
    _Float16 *hc = xh + static_cast<size_t>(n) * Kp;
    for (int k = threadIdx.x; k < Kp; k += blockDim.x)
        hc[x_pos(k, PERM)] = static_cast<_Float16>(k < K ? ldexpf(xc[k], e) : 0.f);
    if (threadIdx.x == 0) xinv[n] = ldexpf(1.f, -e);
}

__device__ inline float half_bits_f(unsigned h) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<unsigned short>(h & 0xFFFFu)));
}

// 8 consecutive elements (one code dword, low nibble first) of one group as
// the fp16 MFMA operand: q * scale - zero * scale, rounded once (within one
// fp16 rounding of the reference's fp32 (q - zero) * scale).
// Byte b of v as a float (v_cvt_f32_ubyte{b}: no separate extract).
template <int B>
__device__ inline float ubyte_f(unsigned v) {
    float f;
    if constexpr (B == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(v));
    if constexpr (B == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(v));
    if constexpr (B == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(v));
    if constexpr (B == 3) asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(v));
    return f;
}

// The group's scale and -zero * scale as plain fp32 registers: the compiler would otherwise fold
// their fp16 -> fp32 conversion into every FMA as a v_fma_mix_f32 (the slow mixed-precision
// form).
__device__ inline void opaque_f32(float &s, float &nzs) { asm("" : "+v"(s), "+v"(nzs)); }

__device__ inline h8 dequant8(unsigned c, float s, float nzs) {
    const unsigned lo = c & 0x0F0F0F0Fu;         // elements 0, 2, 4, 6
    const unsigned hi = (c >> 4) & 0x0F0F0F0Fu;  // elements 1, 3, 5, 7
    u4v pk;
    pk[0] = pair_f16(fmaf(ubyte_f<0>(lo), s, nzs), fmaf(ubyte_f<0>(hi), s, nzs));
    pk[1] = pair_f16(fmaf(ubyte_f<1>(lo), s, nzs), fmaf(ubyte_f<1>(hi), s, nzs));
    pk[2] = pair_f16(fmaf(ubyte_f<2>(lo), s, nzs), fmaf(ubyte_f<2>(hi), s, nzs));
    pk[3] = pair_f16(fmaf(ubyte_f<3>(lo), s, nzs), fmaf(ubyte_f<3>(hi), s, nzs));
    return __builtin_bit_cast(h8, pk);
}

// ---- packed-fp16 dequantization (G = 64)
// A nibble q OR-ed into the mantissa of a fixed fp16 exponent reads as 1024 + q (bits 0..3 under
// exponent 2^10) or 64 + q (bits 4..7 under 2^6), both exact; subtracting 1024 or 64 gives q
// exactly, and fma(q, s, fp16(-z s)) rounds once. Eight elements cost 13 instructions (one shift,
// four v_and_or_b32, four v_pk_add_f16, four v_pk_fma_f16) against 23 for the fp32 form. The
// halves come out in the k-slot order (0, 4, 1, 5, 2, 6, 3, 7) of the code dword's elements, so
// X is stored in that order within every 8 elements (x_to_f16 with kPermute).
typedef _Float16 hf2 __attribute__((ext_vector_type(2)));
__device__ inline hf2 as_h2(unsigned u) { return __builtin_bit_cast(hf2, u); }
__device__ inline unsigned as_u(hf2 h) { return __builtin_bit_cast(unsigned, h); }
// (v_and_or_b32 is a VOP3 instruction: its two constants cannot both be literals, so the magic
// exponent comes in a VGPR and the mask in an SGPR)
__device__ inline unsigned and_or(unsigned c, unsigned mask, unsigned magic) {
    unsigned r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(c), "s"(mask), "v"(magic));
    return r;
}
struct PkConst {
    unsigned k64, k54;  // the two magic exponents, held in VGPRs
};
__device__ inline PkConst pk_const() {
    PkConst k{0x64006400u, 0x54005400u};
    asm volatile("" : "+v"(k.k64), "+v"(k.k54));
    return k;
}
// The group's (s, s) and (-z s, -z s) from its header dword [scale | zero].
__device__ inline void pk_header(unsigned hd, hf2 &s2, hf2 &c2) {
    s2 = as_h2(__builtin_amdgcn_perm(hd, hd, 0x01000100u));
    const hf2 z2 = as_h2(__builtin_amdgcn_perm(hd, hd, 0x03020302u));
    c2 = -(z2 * s2);
}
__device__ inline h8 dequant8_pk(unsigned c, hf2 s2, hf2 c2, PkConst k) {
    const hf2 m1024 = {static_cast<_Float16>(-1024.f), static_cast<_Float16>(-1024.f)};
    const hf2 m64 = {static_cast<_Float16>(-64.f), static_cast<_Float16>(-64.f)};
    const unsigned c8 = c >> 8;
    const hf2 q0 = as_h2(and_or(c, 0x000F000Fu, k.k64)) + m1024;   // elements 0, 4
    const hf2 q1 = as_h2(and_or(c, 0x00F000F0u, k.k54)) + m64;     // 1, 5
    const hf2 q2 = as_h2(and_or(c8, 0x000F000Fu, k.k64)) + m1024;  // 2, 6
    const hf2 q3 = as_h2(and_or(c8, 0x00F000F0u, k.k54)) + m64;    // 3, 7
    u4v pk;
    pk[0] = as_u(__builtin_elementwise_fma(q0, s2, c2));
    pk[1] = as_u(__builtin_elementwise_fma(q1, s2, c2));
    pk[2] = as_u(__builtin_elementwise_fma(q2, s2, c2));
    pk[3] = as_u(__builtin_elementwise_fma(q3, s2, c2));
    return __builtin_bit_cast(h8, pk);
}

// s_waitcnt vmcnt(n), expcnt / lgkmcnt untouched (gfx9 encoding). The count assumes the loads
// issued before it in program order: the sched_barriers keep the machine scheduler from
// moving a load across it (scheduling groups would otherwise carry a step's interleaved loads
// past the next step's wait, and vmcnt(n) would then let that step's own loads still be in
// flight).
__device__ __forceinline__ void wait_vm(int n) {
    __builtin_amdgcn_sched_barrier(0);
    switch (n) {
#define TQ_VMWAIT(N) case N: __builtin_amdgcn_s_waitcnt(((N) & 15) | (7 << 4) | (15 << 8) | (((N) >> 4) << 14)); break;
        TQ_VMWAIT(0) TQ_VMWAIT(1) TQ_VMWAIT(2) TQ_VMWAIT(3) TQ_VMWAIT(4) TQ_VMWAIT(5) TQ_VMWAIT(6) TQ_VMWAIT(7)
        TQ_VMWAIT(8) TQ_VMWAIT(9) TQ_VMWAIT(10) TQ_VMWAIT(11) TQ_VMWAIT(12) TQ_VMWAIT(13) TQ_VMWAIT(14)
        TQ_VMWAIT(15) TQ_VMWAIT(16) TQ_VMWAIT(17) TQ_VMWAIT(18) TQ_VMWAIT(19) TQ_VMWAIT(20) TQ_VMWAIT(21)
        TQ_VMWAIT(22) TQ_VMWAIT(23) TQ_VMWAIT(24) TQ_VMWAIT(25) TQ_VMWAIT(26) TQ_VMWAIT(27) TQ_VMWAIT(28)
        TQ_VMWAIT(32)
#undef TQ_VMWAIT
        default: __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8)); break;
    }
    __builtin_amdgcn_sched_barrier(0);
}

// Workgroup barrier that waits for this wave's LDS operations only (global ->
// LDS transfers of later steps stay in flight). The sched_barriers keep the machine
// scheduler from moving anything across it (a memory clobber binds only the compiler's
// IR passes: scheduling groups would otherwise hoist the step's LDS reads above it).
__device__ inline void lds_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// Byte offsets within a row of one step's two 32-element halves (each in one group, G % 32 == 0):
// group header and 16 code bytes (scalar). Past the last group: the last one's, in the row (X is
// zero there).
struct HalfOffsets {
    int hdr[2], code[2];
};
__device__ __forceinline__ HalfOffsets half_offsets(int s, int G, int gb, int groups) {
    HalfOffsets o;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int k = s * kStepK + 32 * t, g = min(k / G, groups - 1);
        o.hdr[t] = g * gb;
        o.code[t] = g * gb + 4 + min((k - g * G) / 2, G / 2 - 16);
    }
    return o;
}

// ---- K slices of a tile
//   A grid of few tiles leaves most CUs idle, so K is then cut into KS slices of whole steps, one
//   workgroup each (kSplitParts): a workgroup stores its partial product, the last of a tile to
//   arrive adds the KS partials in slice order (the same bits whatever the arrival order) and
//   stores Y. kSplitSeq gives the same bits with one workgroup per tile and no partials, for calls
//   that may not allocate them.
constexpr int kSplitNone = 0, kSplitParts = 1, kSplitSeq = 2;
constexpr int kDeviceScope = 16;  // buffer cache policy: sc1 (device-scope coherent)
constexpr int kL1Bypass = 1;      // buffer cache policy: sc0 (misses in the CU's L1, served by the XCD's L2)
typedef float f4v __attribute__((ext_vector_type(4)));

//   Partials are [tile][slice][wave][token block][float4][lane] (the MFMA's register order: every
//   store and load instruction moves 1 KB in one piece), written at device scope (sc1: through this
//   XCD's L2 to the level where all XCDs meet), so a store that has completed is visible
//   everywhere and the arrival counter (zero between launches: the last arrival resets it) needs
//   no cache write-back or invalidation, both of which act on a whole L2. The counter add carries
//   the writer's XCD (slices below kXccSlots): the last arrival reads a partial written on its own
//   XCD from that L2 (which the write went through) and any other one at device scope.
//   True for the last arrival, whose acc then holds the sum.
template <int WN, int NWV>
__device__ inline bool add_parts(f16x (&acc)[WN], float *part, unsigned long long *arrivals, int tile, int ks, int KS,
                                 int wave, int lane) {
    constexpr int kPart = 32 * NWV * 32 * WN;  // floats of one partial
    constexpr int V = 4 * WN;                  // float4s of a lane
    constexpr int B = V <= 4 ? 6 : V <= 8 ? 4 : 2;  // partials in flight at once (registers)
    __shared__ int last_s;
    __shared__ unsigned long long writers_s;
    const int xcc = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 7;  // HW_REG_XCC_ID bits 0..3
    const __amdgpu_buffer_rsrc_t pr =
        make_rsrc(part + static_cast<size_t>(tile) * KS * kPart, static_cast<size_t>(KS) * kPart * sizeof(float));
    const int lo = 16 * (64 * V * wave + lane);
    f4v own[V];
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
            own[4 * j + r4] = f4v{acc[j][4 * r4], acc[j][4 * r4 + 1], acc[j][4 * r4 + 2], acc[j][4 * r4 + 3]};
#pragma unroll
    for (int v = 0; v < V; ++v)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, own[v]), pr, lo + 4 * (ks * kPart) + 1024 * v, 0,
                                               kDeviceScope);
    wait_vm(0);       // this wave's partial stores have completed
    __syncthreads();  // and every other wave's
    if (threadIdx.x == 0) {
        // (the counter's layout: few_token_slices.h)
        const unsigned long long mine =
            (1ull << kArrivalShift) | (ks < kXccSlots ? static_cast<unsigned long long>(xcc + 1) << (4 * ks) : 0ull);
        const unsigned long long prev =
            __hip_atomic_fetch_add(arrivals + tile, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = (prev >> kArrivalShift) == static_cast<unsigned long long>(KS - 1);
        if (last) __hip_atomic_store(arrivals + tile, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last_s = last;
        writers_s = prev;
    }
    __syncthreads();
    if (!last_s) return false;
    const unsigned long long writers = writers_s;
    f4v sum[V] = {};
    for (int p0 = 0; p0 < KS; p0 += B) {
        f4v v[B][V];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int p = min(p0 + u, KS - 1);
            if (p == ks) continue;
            const bool here = p < kXccSlots && ((writers >> (4 * p)) & 15) == static_cast<unsigned>(xcc + 1);
            if (here) {
#pragma unroll
                for (int i = 0; i < V; ++i)
                    v[u][i] = __builtin_bit_cast(
                        f4v, __builtin_amdgcn_raw_buffer_load_b128(pr, lo + 4 * (p * kPart) + 1024 * i, 0, kL1Bypass));
            } else {
#pragma unroll
                for (int i = 0; i < V; ++i)
                    v[u][i] = __builtin_bit_cast(
                        f4v, __builtin_amdgcn_raw_buffer_load_b128(pr, lo + 4 * (p * kPart) + 1024 * i, 0, kDeviceScope));
            }
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
            if (p0 + u >= KS) break;
#pragma unroll
            for (int i = 0; i < V; ++i) sum[i] += p0 + u == ks ? own[i] : v[u][i];
        }
    }
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = sum[4 * j + r / 4][r % 4];
    return true;
}

// ---- 2. W straight into registers
//   Lane (row, half h) takes 32 elements of its row per step: they lie in one group (G % 32 == 0),
//   so a 4-byte load of its header and a 16-byte load of their codes, S - 1 steps ahead, bring
//   them into VGPRs and W never passes through LDS. (W staged through LDS a dword at a time, as
//   group sizes other than 64 used to be, took twice the time: 9728x2560 at G = 128 and 128 /
//   512 / 3001 tokens 45 / 80 / 358 us per call against 25 / 47 / 210; at G = 64 a step's offsets are
//   one scalar, at other sizes a select per half.)
//   X: BN rows x 128 B of fp16 a step by DMA into a ring of S stages; 16-byte chunk c of token
//   row r is stored at position c ^ ((r >> 1) & 7). A ds_read_b128 is served 16 lanes at a time,
//   one 256-byte bank sweep: the 16 rows a group reads differ in (r & 1, chunk), so they cover
//   the sweep once (no bank conflicts).
//   The loop is unrolled by S so that every register slot index is a
//   constant; its last round loads steps past the last (never consumed),
//   which keeps every wait in it one constant s_waitcnt.
//   At G = 64 (PK) the A operands are dequantized with packed fp16 arithmetic (dequant8_pk),
//   which leaves a code dword's elements in k-slot order (0, 4, 1, 5, 2, 6, 3, 7); X comes
//   from x_to_f16<true> in the same order, so both operands agree slot for slot. Other group
//   sizes keep the fp32 dequantization with its one rounding (dequant8) and X's natural order.
//   Y leaves in 16-byte stores (4 rows of a token) where M % 4 == 0 and y is 16-byte
//   aligned: four times fewer store instructions than one float each, which took
//   the 512-token call from 48 to 39 us on MI355X (the output is 20 MB there).
//   Measured on MI355X at 512 tokens with copies of this kernel that skip parts of
//   the work: without the MFMAs or without the dequantization the time hardly
//   changes; without the loads of W and X it drops by three quarters. The loop is
//   bound by the time each workgroup's loads take to arrive, not by arithmetic.
// The X DMAs d0 .. d0 + nx - 1 of a step (1 KB each, at byte 1024 d of the stage); nx <= ND.
template <int ND>
__device__ __forceinline__ void issue_x(__amdgpu_buffer_rsrc_t xr, unsigned char *st, const int *xvo, int nx, int d0,
                                        int xso) {
#pragma unroll
    for (int q = 0; q < ND; ++q)
        if (q < nx)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                xr, (__attribute__((address_space(3))) void *)(st + 1024 * (d0 + q)), 16, xvo[q], xso, 0, 0);
}

template <int GT, int WN, int S, int NWV, int SPLIT>
__global__ __launch_bounds__(64 * NWV) void i4_matmul_direct(const uint8_t *__restrict__ w,
                                                             const _Float16 *__restrict__ xh,
                                                             const float *__restrict__ xinv, float *__restrict__ y,
                                                             int M, int N, int K, int Kp, int G, int row_bytes,
                                                             int vec_y, int KS, float *__restrict__ part,
                                                             unsigned long long *__restrict__ arrivals) {
    constexpr bool PK = GT == 64;  // packed-fp16 dequantization, X in its k-slot order
    constexpr int BN = 32 * WN;
    constexpr int BM = 32 * NWV;
    constexpr int XStage = BN * 128;
    // The step's 4 WN X DMAs (1 KB each) are dealt out in order: waves below XR issue XA + 1 of
    // them, the others XA. P: this wave's loads per step (W 4 + 16 bytes, its X DMAs).
    constexpr int XA = 4 * WN / NWV, XR = 4 * WN % NWV;
    constexpr int XD = XA + (XR ? 1 : 0);
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int tile = 0, ks = 0, m0, n0;
    if constexpr (SPLIT == kSplitParts) {
        // the slices of a tile are 8 workgroups apart, so with workgroups dealt to the 8 XCDs in
        // turn they share one XCD
        tile = (blockIdx.x / (8 * KS)) * 8 + (blockIdx.x & 7);
        ks = (blockIdx.x >> 3) % KS;
        const int mtiles = (M + BM - 1) / BM, nt = tile / mtiles;
        m0 = (tile - nt * mtiles) * BM;
        n0 = nt * BN;
        if (n0 >= N) return;  // a padding tile (the tile count rounded up to 8)
    } else {
        m0 = blockIdx.x * BM;
        n0 = blockIdx.y * BN;
    }
    if constexpr (GT != 0) G = GT;
    const int gb = 4 + G / 2;
    const int groups = (K + G - 1) / G;
    const int steps = Kp / kStepK;

    const __amdgpu_buffer_rsrc_t wr = make_rsrc(w + static_cast<size_t>(m0) * row_bytes,
                                                static_cast<size_t>(M - m0) * row_bytes);
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(xh + static_cast<size_t>(n0) * Kp,
                                                static_cast<size_t>(N - n0) * Kp * 2);
    // Lane (row li, half h) takes elements 32 h .. 32 h + 31 of every step: the header of their group
    // (G % 32 == 0: they lie in one) and their 16 code bytes; MFMA k-slot 8 h + p of k-block kk
    // holds element 32 h + 8 kk + e, p = ((e & 3) << 1) | (e >> 2) (PK) or e, on the A (W) and the B (X) side.
    const int li = lane & 31, h = lane >> 5;
    const int wvo = (32 * wave + li) * row_bytes;
    const int nx = XA + (wave < XR ? 1 : 0), d0 = XA * wave + min(wave, XR);
    int xvo[XD > 0 ? XD : 1];
#pragma unroll
    for (int q = 0; q < XD; ++q) {
        const int p = 64 * min(d0 + q, 4 * WN - 1) + lane;
        const int r = p >> 3, c = (p & 7) ^ ((r >> 1) & 7);
        xvo[q] = r * Kp * 2 + 16 * c;
    }
    int xro[4][WN];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            const int r = 32 * j + li;
            xro[kk][j] = 16 * (8 * r + ((4 * h + kk) ^ ((r >> 1) & 7)));
        }

    const PkConst pkc = pk_const();
    unsigned hd[S];
    u4v cd[S];
    auto issue = [&](auto uc, int s) {  // step s into register slot and X stage u = s % S
        constexpr int u = decltype(uc)::value;
        if constexpr (GT == 64) {
            const int so = 36 * min(s, groups - 1);  // (past the last step: in-row bytes, never used)
            hd[u] = __builtin_amdgcn_raw_buffer_load_b32(wr, wvo, so, 0);
            cd[u] = __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(wr, wvo + 4 + 16 * h, so, 0));
        } else {
            const HalfOffsets o = half_offsets(s, G, gb, groups);
            hd[u] = __builtin_amdgcn_raw_buffer_load_b32(wr, wvo + (h ? o.hdr[1] : o.hdr[0]), 0, 0);
            cd[u] = __builtin_bit_cast(
                u4v, __builtin_amdgcn_raw_buffer_load_b128(wr, wvo + (h ? o.code[1] : o.code[0]), 0, 0));
        }
        issue_x<XD>(xr, smem + u * XStage, xvo, nx, d0, s * kStepK * 2);
    };
    f16x acc[WN];
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[j] = f16x{};
    // k-blocks k0 .. k1 - 1 of the step in register slot and X stage u
    auto compute = [&](auto uc, int k0, int k1) {
        constexpr int u = decltype(uc)::value;
        const unsigned char *st = smem + u * XStage;
        hf2 s2, c2;
        float fs, fz;
        if constexpr (PK) {
            pk_header(hd[u], s2, c2);
        } else {
            fs = half_bits_f(hd[u]);
            fz = -(half_bits_f(hd[u] >> 16) * fs);
            opaque_f32(fs, fz);
        }
#pragma unroll
        for (int kk = k0; kk < k1; ++kk) {
            h8 b[WN];
#pragma unroll
            for (int j = 0; j < WN; ++j) b[j] = *reinterpret_cast<const h8 *>(st + xro[kk][j]);
            h8 a;
            if constexpr (PK)
                a = dequant8_pk(cd[u][kk], s2, c2, pkc);
            else
                a = dequant8(cd[u][kk], fs, fz);
#pragma unroll
            for (int j = 0; j < WN; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b[j], acc[j], 0, 0, 0);
        }
    };
    // One step of a full round. Its loads of step s + S - 1 go in between the first and the last two
    // k-blocks' MFMAs (program order; no branch), so that a wave stalled on a full memory pipeline
    // has MFMAs in flight.
    auto round_step = [&](auto uc, int s) {
        constexpr int u = decltype(uc)::value;
        if (XR == 0 || wave < XR)  // this wave's loads of step s have landed
            wait_vm((S - 2) * (2 + XD));
        else
            wait_vm((S - 2) * (2 + XA));
        lds_barrier();  // every wave's X part has; step s - 1's stage is free
        compute(uc, 0, 2);
        issue(std::integral_constant<int, (u + S - 1) % S>{}, s + S - 1);
        compute(uc, 2, 4);
    };

    static_assert(S >= 2 && S <= 4, "register slots 0..3");
    // Steps sa .. sb - 1 into acc (slot u holds step sa + u modulo S).
    // (the sched_barriers keep each step's loads together: the waits count whole steps)
    auto run = [&](int sa, int sb) {
        issue(std::integral_constant<int, 0>{}, sa);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (S > 2) issue(std::integral_constant<int, 1>{}, sa + 1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (S > 3) issue(std::integral_constant<int, 2>{}, sa + 2);
        __builtin_amdgcn_sched_barrier(0);
        int s0 = sa;
        for (; s0 + S <= sb; s0 += S) {
            round_step(std::integral_constant<int, 0>{}, s0);
            round_step(std::integral_constant<int, 1>{}, s0 + 1);
            if constexpr (S > 2) round_step(std::integral_constant<int, 2>{}, s0 + 2);
            if constexpr (S > 3) round_step(std::integral_constant<int, 3>{}, s0 + 3);
        }
        // The last (sb - sa) % S steps: all of their loads are under way, so one wait for everything
        // and no more loads. (Issuing loads here to keep the constant waits would not do: nothing
        // reads the codes that they bring, so the compiler drops those loads and the waits then
        // count too few.)
        wait_vm(0);
        lds_barrier();
        if (s0 < sb) compute(std::integral_constant<int, 0>{}, 0, 4);
        if constexpr (S > 2) {
            if (s0 + 1 < sb) compute(std::integral_constant<int, 1>{}, 0, 4);
        }
        if constexpr (S > 3) {
            if (s0 + 2 < sb) compute(std::integral_constant<int, 2>{}, 0, 4);
        }
    };
    // each token's scale, requested before the stores below (a load behind them waits for them)
    float sc[WN];
    const auto load_scales = [&]() {
#pragma unroll
        for (int j = 0; j < WN; ++j) sc[j] = xinv[min(n0 + 32 * j + li, N - 1)];
    };
    if constexpr (SPLIT == kSplitNone) {
        run(0, steps);
    } else if constexpr (SPLIT == kSplitParts) {
        run((ks * steps) / KS, ((ks + 1) * steps) / KS);
        if (!add_parts<WN, NWV>(acc, part, arrivals, tile, ks, KS, wave, lane)) return;
    } else {
        // every slice in this workgroup, added as add_parts adds them: the same bits without partials
        f16x sum[WN];
#pragma unroll
        for (int j = 0; j < WN; ++j) sum[j] = f16x{};
        for (int p = 0; p < KS; ++p) {
            run((p * steps) / KS, ((p + 1) * steps) / KS);
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                sum[j] += acc[j];
                acc[j] = f16x{};
            }
            lds_barrier();  // (every wave is done with the stages that the next slice's loads go to)
        }
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[j] = sum[j];
    }
    load_scales();

    // epilogue: lane holds rows (r/4)*8 + (lane/32)*4 + r%4 of column lane%32
#pragma unroll
    for (int j = 0; j < WN; ++j) {
        const int n = n0 + 32 * j + li;
        if (n >= N) continue;
        float *yc = y + static_cast<size_t>(n) * M;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const int m = m0 + 32 * wave + 8 * r4 + 4 * h;
            if (vec_y && m + 3 < M) {
                *reinterpret_cast<float4 *>(yc + m) = make_float4(acc[j][4 * r4] * sc[j], acc[j][4 * r4 + 1] * sc[j],
                                                                  acc[j][4 * r4 + 2] * sc[j], acc[j][4 * r4 + 3] * sc[j]);
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (m + q < M) yc[m + q] = acc[j][4 * r4 + q] * sc[j];
            }
        }
    }
}

// ---- 3. Few tokens (N <= 32, G = 64): one launch
//   A kernel launch costs a few microseconds on this GPU whatever it does, so at a few
//   tokens a separate X conversion pass would cost as much as the GEMM. Here every
//   workgroup converts the X it needs itself. The grid is (128-row tile) x (K slice):
//   workgroup (tile, ks) forms the partial product of its 128 rows over the slice's
//   steps for all tokens; the last workgroup of a tile to finish adds the KS partials in
//   slice order (fixed, whatever the arrival order) and stores Y. One CU reads only some
//   50-90 GB/s from L2, so the fp32 X of a whole row of K per workgroup would take
//   several microseconds: the slices spread it over the CUs.
//   - X: the slice of the 32 token rows is read once (fp32, 16-byte loads), scaled per
//     token by the power of two that puts the token's largest |x| in the slice into
//     [2^13, 2^14), and stored to LDS as fp16, [step][token][64 elements] with the
//     16-byte chunks of token n at positions c ^ ((n >> 1) & 7): the 16 rows a
//     ds_read_b128 pass serves cover one 256-byte bank sweep exactly (rows n and n + 8 on
//     the same chunk, as c ^ (n & 7) had them, share banks). Within a chunk the 8 elements
//     are in the k-slot order of the packed-fp16 dequantization (dequant8_pk).
//   - W: each row's slice (9 dwords a step, contiguous) comes in with one DMA into LDS at
//     an odd dword pitch. (A load per lane and row touches a cache line per lane; the
//     DMA touches the 2-3 lines the slice spans.) Wave w then takes rows 32 w .. 32 w + 31:
//     lane (row r, half h) reads the group header and code dwords 1 + 4 h .. 4 + 4 h of each
//     step, so MFMA k-slot 8 h + p of k-block j holds element 32 h + 8 j + p of the step,
//     on the A (W) and on the B (X) side.
//   - Partials: [tile][slice][4 waves x 4 float4 x 64 lanes] fp32 (the MFMA's register
//     order: every store and load instruction moves 1 KB in one piece), written at device
//     scope. The slices of a tile are 8 workgroups apart and workgroups are dealt to the 8
//     XCDs in turn, so a tile normally stays on one XCD and the last arrival reads the
//     other partials from that XCD's L2; the arrival counter (zero between launches: the
//     last arrival resets it) carries each writer's XCD, so a partial written elsewhere is
//     read at device scope instead.
constexpr int kSkReduceBatch = 6;  // partials the last arrival has in flight at once

template <int SMAX>
__global__ __launch_bounds__(256) void i4_matmul_skinny(const uint8_t *__restrict__ w, const float *__restrict__ x,
                                                        float *__restrict__ y, int M, int K, int N, int row_bytes,
                                                        int T, int KS, float *__restrict__ part,
                                                        unsigned long long *__restrict__ arrivals, int vec_y) {
    __shared__ __align__(16) unsigned char xs[SMAX * 4096];
    __shared__ __align__(16) unsigned char ws_lds[kSkRows * (9 * SMAX + 1) * 4];
    __shared__ float inv_s[32];
    __shared__ int last_s;
    __shared__ unsigned long long writers_s;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroup b -> tile 8 (b / (8 KS)) + b % 8, slice (b / 8) % KS: the slices of a tile are
    // 8 workgroups apart, so with workgroups dealt to the 8 XCDs in turn they share one XCD
    const int tile = (blockIdx.x / (8 * KS)) * 8 + (blockIdx.x & 7), ks = (blockIdx.x >> 3) % KS;
    const int m0 = tile * kSkRows;
    if (m0 >= M) return;  // a padding tile (the tile count rounded up to 8)
    const int s0 = (ks * T) / KS, ns = ((ks + 1) * T) / KS - s0;  // steps [s0, s0 + ns), 1 <= ns <= SMAX

    // 1. X: thread t takes token n = t / 8 and float4s (t % 8) + 8 q of the token's slice
    const int n = threadIdx.x >> 3, sub = threadIdx.x & 7;
    const int k0 = 64 * s0;
    const float4 *xr = reinterpret_cast<const float4 *>(x + static_cast<size_t>(n < N ? n : 0) * K + k0);
    float4 xv[2 * SMAX];
    unsigned okm = 0;  // bit q: float4 q lies in the matrix (masked to zero after the loads land)
#pragma unroll
    for (int q = 0; q < 2 * SMAX; ++q) {
        const int f = sub + 8 * q;
        const bool ok = n < N && q < 2 * ns && k0 + 4 * f < K;  // K % 4 == 0: a float4 is all in or all out
        okm |= static_cast<unsigned>(ok) << q;
        xv[q] = xr[ok ? f : 0];
    }
    // (the X loads stay ahead of the W DMAs in the instruction stream: step 3 counts on it)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    // 2. W: the slice of each of the tile's 128 rows is 9 ns contiguous dwords; one DMA per row
    //    (wave w: rows 32 w .. 32 w + 31, lane i: dword i) lands it at LDS dword r * P, with
    //    the odd pitch P = 9 ns | 1, so the 32 rows a wave reads in step j (dword r P + 9 j + c)
    //    fall in 32 different banks
    const int P = (9 * ns) | 1;
    const int li = lane & 31, h = lane >> 5;
    if (lane < 9 * ns) {  // only the slice's lanes: a DMA lane writes LDS dword (base + lane), and
                          // lanes past 9 ns would land in the next row's dwords
        const __amdgpu_buffer_rsrc_t wr = rows_rsrc(w, M, row_bytes, m0);
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const int r = 32 * wave + i;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                wr, (__attribute__((address_space(3))) void *)(ws_lds + 4 * r * P), 4, r * row_bytes + 4 * lane,
                36 * s0, 0, 0);
        }
    }

    // 3. the slice's X to fp16 in LDS, scaled per token, while the W rows are in flight: the
    //    wave's 32 row DMAs were issued after its X loads, so vmcnt(32) is the X loads alone
    static_assert(kSkRows / 4 == 32, "32 row DMAs per wave");
    wait_vm(32);
#pragma unroll
    for (int q = 0; q < 2 * SMAX; ++q) {
        const bool ok = (okm >> q) & 1u;
        xv[q].x = ok ? xv[q].x : 0.f;
        xv[q].y = ok ? xv[q].y : 0.f;
        xv[q].z = ok ? xv[q].z : 0.f;
        xv[q].w = ok ? xv[q].w : 0.f;
    }
    float m = 0.f;
#pragma unroll
    for (int q = 0; q < 2 * SMAX; ++q)
        m = fmaxf(m, fmaxf(fmaxf(fabsf(xv[q].x), fabsf(xv[q].y)), fmaxf(fabsf(xv[q].z), fabsf(xv[q].w))));
    m = fmaxf(m, dpp_f<kDppXor1>(m));
    m = fmaxf(m, dpp_f<kDppXor2>(m));
    m = fmaxf(m, dpp_f<kDppHalfMirror>(m));  // the 8 lanes of token n
    int e = 0;  // zero or non-finite: unscaled (inf and NaN carry through)
    if (m > 0.f && m <= 3.0e38f) e = min(14 - __builtin_amdgcn_frexp_expf(m), 126);
    const float sc = ldexpf(1.f, e);
    if (sub == 0) inv_s[n] = ldexpf(1.f, -e);
    // Within each 8 elements the chunk holds them in the packed dequantization's k-slot order
    // (0, 4, 1, 5, 2, 6, 3, 7): the even thread of a pair (elements 0..3 of the 8) takes 4, 5
    // from the odd one and writes slots 0..3; the odd thread takes 2, 3 and writes slots 4..7.
    const bool odd = sub & 1;
#pragma unroll
    for (int q = 0; q < 2 * SMAX; ++q) {
        const int c = (sub >> 1) + 4 * (q & 1);  // 16-byte chunk of step q / 2
        const float a0 = xv[q].x * sc, a1 = xv[q].y * sc, a2 = xv[q].z * sc, a3 = xv[q].w * sc;  // exact scaling
        const float r0 = dpp_f<kDppXor1>(odd ? a0 : a2), r1 = dpp_f<kDppXor1>(odd ? a1 : a3);
        uint2 pk;
        pk.x = odd ? pair_f16(r0, a2) : pair_f16(a0, r0);  // one rounding each
        pk.y = odd ? pair_f16(r1, a3) : pair_f16(a1, r1);
        *reinterpret_cast<uint2 *>(xs + 4096 * (q >> 1) + 128 * n + 16 * (c ^ ((n >> 1) & 7)) + 8 * (sub & 1)) = pk;
    }
    wait_vm(0);  // this wave's W rows have landed in LDS
    lds_barrier();

    // 4. the slice's steps: lane (row 32 w + li, half h) takes the header and code dwords
    //    1 + 4 h .. 4 + 4 h of the step's group
    const PkConst pkc = pk_const();
    f16x acc = {};
    const unsigned *wl = reinterpret_cast<const unsigned *>(ws_lds) + (32 * wave + li) * P;
#pragma unroll
    for (int j = 0; j < SMAX; ++j) {
        if (j < ns) {
            const unsigned hd = wl[9 * j];
            unsigned cd[4];
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) cd[kk] = wl[9 * j + 1 + 4 * h + kk];
            hf2 s2, c2;
            pk_header(hd, s2, c2);
            h8 b[4];
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
                b[kk] = *reinterpret_cast<const h8 *>(xs + 4096 * j + 128 * li + 16 * ((4 * h + kk) ^ ((li >> 1) & 7)));
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(dequant8_pk(cd[kk], s2, c2, pkc), b[kk], acc, 0, 0, 0);
        }
    }

    // 5. the partial, stored as the MFMA leaves it: float4 r4 of lane l of wave w at index
    //    (4 w + r4) * 64 + l (rows 32 w + 8 r4 + 4 h + 0..3 of token l % 32, h = l / 32), so
    //    every store and load instruction moves 1 KB in one piece. Partials are stored at
    //    device scope (sc1: written through this XCD's L2 to the level where all XCDs meet),
    //    so a store that has completed is visible everywhere and the counter needs no cache
    //    write-back or invalidation (both act on a whole L2). The counter add carries the
    //    writer's XCD (slices < kXccSlots): the last arrival reads a partial written on its
    //    own XCD from that L2 (which the write went through) and any other one at device
    //    scope (its own L2 may hold an older copy of the line).
    const float iv = inv_s[li];
    const int xcc = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 7;  // HW_REG_XCC_ID bits 0..3
    f4v own[4];
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4)
        own[r4] = f4v{acc[4 * r4] * iv, acc[4 * r4 + 1] * iv, acc[4 * r4 + 2] * iv, acc[4 * r4 + 3] * iv};
    const __amdgpu_buffer_rsrc_t pr = make_rsrc(part + static_cast<size_t>(tile) * KS * kSkTile,
                                                static_cast<size_t>(KS) * kSkTile * sizeof(float));
    // byte offset of the lane's float4 r4 = 0 in a partial; lanes past the last token: past the
    // buffer, where stores are dropped and loads read 0 (8 tokens, a quarter of the traffic:
    // 9728x2560 13.0 -> 12.5 us, 151936x896 48.6 -> 46.6)
    const int lo = li < N ? 16 * (256 * wave + lane) : 0x40000000;
    if (KS > 1) {
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, own[r4]), pr,
                                                   lo + 4 * (ks * kSkTile) + 1024 * r4, 0, kDeviceScope);
        wait_vm(0);       // this wave's partial stores have completed
        __syncthreads();  // and every other wave's
        if (threadIdx.x == 0) {
            // (the counter's layout: few_token_slices.h)
            const unsigned long long mine =
                (1ull << kArrivalShift) | (ks < kXccSlots ? static_cast<unsigned long long>(xcc + 1) << (4 * ks) : 0ull);
            const unsigned long long prev =
                __hip_atomic_fetch_add(arrivals + tile, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool last = (prev >> kArrivalShift) == static_cast<unsigned long long>(KS - 1);
            if (last) __hip_atomic_store(arrivals + tile, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            last_s = last;
            writers_s = prev;
        }
        __syncthreads();
        if (!last_s) return;
    }
    const unsigned long long writers = writers_s;

    // 6. the last arrival: Y = the KS partials added in slice order (its own from registers,
    //    the others loaded kSkReduceBatch at a time)
    f4v sum[4] = {};
    for (int p0 = 0; p0 < KS; p0 += kSkReduceBatch) {
        f4v v[kSkReduceBatch][4];
#pragma unroll
        for (int u = 0; u < kSkReduceBatch; ++u) {
            const int p = min(p0 + u, KS - 1);
            if (p == ks) continue;
            const bool here = p < kXccSlots && ((writers >> (4 * p)) & 15) == static_cast<unsigned>(xcc + 1);
            if (here) {
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4)
                    v[u][r4] = __builtin_bit_cast(
                        f4v, __builtin_amdgcn_raw_buffer_load_b128(pr, lo + 4 * (p * kSkTile) + 1024 * r4, 0, kL1Bypass));
            } else {
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4)
                    v[u][r4] = __builtin_bit_cast(
                        f4v, __builtin_amdgcn_raw_buffer_load_b128(pr, lo + 4 * (p * kSkTile) + 1024 * r4, 0, kDeviceScope));
            }
        }
#pragma unroll
        for (int u = 0; u < kSkReduceBatch; ++u) {
            if (p0 + u >= KS) break;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const f4v t = p0 + u == ks ? own[r4] : v[u][r4];
                sum[r4][0] += t[0];
                sum[r4][1] += t[1];
                sum[r4][2] += t[2];
                sum[r4][3] += t[3];
            }
        }
    }
    if (li >= N) return;
    float *yc = y + static_cast<size_t>(li) * M;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
        const int m = m0 + 32 * wave + 8 * r4 + 4 * h;
        if (vec_y && m + 3 < M) {
            *reinterpret_cast<float4 *>(yc + m) = make_float4(sum[r4][0], sum[r4][1], sum[r4][2], sum[r4][3]);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (m + c < M) yc[m + c] = sum[r4][c];
        }
    }
}

// K slices of a call and where their partials go (part null: kSplitSeq).
struct Slices {
    int KS;
    float *part;
    unsigned long long *arrivals;
};

template <int GT, int WN, int S, int NWV, int SPLIT>
int launch_direct(const uint8_t *w, const _Float16 *xh, const float *xinv, float *y, int M, int N, int K, int Kp, int G,
                  int rb, const Slices &sl, hipStream_t stream) {
    constexpr int BN = 32 * WN, BM = 32 * NWV;
    const auto kernel = i4_matmul_direct<GT, WN, S, NWV, SPLIT>;
    constexpr size_t lds = static_cast<size_t>(S) * BN * 128;
    static_assert(lds <= 64 * 1024, "the dynamic LDS that a launch may take without raising its limit");
    if (static_cast<size_t>(BM) * rb + static_cast<size_t>(Kp) * 2 * BN >= (1ull << 31)) return kTooLarge;
    dim3 grid((M + BM - 1) / BM, (N + BN - 1) / BN);
    if (SPLIT == kSplitParts) grid = dim3((grid.x * grid.y + 7) / 8 * 8 * sl.KS);
    const int vec_y = M % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
    hipLaunchKernelGGL(kernel, grid, dim3(64 * NWV), lds, stream, w, xh, xinv, y, M, N, K, Kp, G, rb, vec_y, sl.KS,
                       sl.part, sl.arrivals);
    return hipGetLastError() == hipSuccess ? kOk : kLaunchFailed;
}

// The few-token kernel applies: G = 64, at most 32 tokens, whole 16-byte X loads (K % 4 == 0,
// X 16-byte aligned) and rows that its slices cover (whose 128 are then within 31-bit byte offsets).
bool skinny_applies(const float *x, int K, int N, int group_size) {
    return group_size == 64 && N <= 32 && K % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
           skinny_row_fits(K);
}

int launch_skinny(const uint8_t *w, const float *x, float *y, int M, int K, int N, const SkinnyGeom &g, float *part,
                  unsigned long long *arrivals, hipStream_t stream) {
    const int rb = static_cast<int>(i4_row_bytes(K, 64));
    const int vec_y = M % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;  // 16-byte Y stores
    const dim3 grid((g.tiles + 7) / 8 * 8 * g.KS), block(256);
    switch (g.smax) {
#define TQ_SKINNY(S)                                                                                             \
    case S:                                                                                                      \
        hipLaunchKernelGGL(i4_matmul_skinny<S>, grid, block, 0, stream, w, x, y, M, K, N, rb, g.T, g.KS, part, \
                           arrivals, vec_y);                                                                     \
        break;
        TQ_SKINNY(1) TQ_SKINNY(2) TQ_SKINNY(3) TQ_SKINNY(4) TQ_SKINNY(5) TQ_SKINNY(6) TQ_SKINNY(7)
#undef TQ_SKINNY
        default:
            return kBadShape;
    }
    return hipGetLastError() == hipSuccess ? kOk : kLaunchFailed;
}

// A call's tile and K slices (KS > 1: one workgroup per tile and slice).
enum TileKind { kTile32x32, kTile128x32, kTile128x64, kTile256x96 };
struct TilePlan {
    TileKind kind;
    int KS;
    size_t tiles, part_bytes;  // of a split call
};

// The plan with the least estimated time, from what a step of each tile takes on MI355X when a CU
// holds one, two or n workgroups of it (us) and what the exchange of a split adds: stores, counter
// and the last arrival's reads (16 or 32 KB a partial at 50-90 GB/s), and the partials' way through
// memory (twice, 6 TB/s). It only has to rank. Measured against the choice of one tile per token
// count without slices that it replaces (us per call, G = 64): 2560x9728 at 48 / 128 / 512 tokens
// 65 / 72 / 122 -> 21 / 24 / 50; 1024x2560 at 128 / 512 20 / 34 -> 15 / 18; 4096x2560 at 256 33 -> 19.
// The old choice where it was right: 9728x2560 at 128 (152 tiles: 21, with two to five slices 23-31)
// and at 512 (256 x 96 tiles: 41, 128 x 64 49); 896x896 at 128 whole (14 steps: 10.6, with slices 14).
// A function of the shape and the device alone: every entry point gives a call the same sums.
TilePlan tile_plan(int M, int K, int N) {
    const int steps = (K + kStepK - 1) / kStepK, cus = device_cu_count();
    struct Tile {
        TileKind kind;
        int bm, bn;
        float one, two, many;  // a step with one or two workgroups on the CU, and per workgroup with more
        float split, part;     // a split, and each partial of a tile; split 0: not split
    };
    constexpr Tile kTiles[] = {{kTile32x32, 32, 32, 0.3f, 0.3f, 0.1f, 0.f, 0.f},
                               {kTile128x32, 128, 32, 0.3f, 0.4f, 0.25f, 4.f, 0.25f},
                               {kTile128x64, 128, 64, 0.4f, 0.6f, 0.42f, 4.f, 0.45f},
                               {kTile256x96, 256, 96, 0.77f, 1.6f, 0.8f, 0.f, 0.f}};
    constexpr int kMostSlices = 32;
    static_assert(kMostSlices <= kMaxSlices, "the arrival counter's count");
    TilePlan best{};
    float cost = 0.f;
    for (const Tile &t : kTiles) {
        // one token block: the 32-token tiles; more: the others (they share W loads among tokens)
        if ((N <= 32) != (t.bn == 32)) continue;
        const size_t tiles = static_cast<size_t>((M - 1) / t.bm + 1) * ((N - 1) / t.bn + 1);
        for (int ks = 1; ks <= (t.split > 0.f ? std::min(kMostSlices, steps) : 1); ++ks) {
            const size_t n = (tiles * ks - 1) / cus + 1, bytes = ks > 1 ? tiles * ks * t.bm * t.bn * sizeof(float) : 0;
            const float step = n == 1 ? t.one : n == 2 ? t.two : t.many * static_cast<float>(n);
            const float c = static_cast<float>((steps - 1) / ks + 1) * step +
                            (ks > 1 ? t.split + t.part * static_cast<float>(ks) + static_cast<float>(bytes) / 3e6f : 0.f);
            if (best.tiles == 0 || c < cost) {
                best = TilePlan{t.kind, ks, tiles, bytes};
                cost = c;
            }
        }
    }
    return best;
}

// The MFMA path applies: a group size that is a multiple of 32 and byte offsets within 31 bits.
bool mfma_applies(int M, int K, int N, int group_size) {
    const size_t Kp = (static_cast<size_t>(K) + kStepK - 1) / kStepK * kStepK;
    return group_size % 32 == 0 && i4_row_bytes(K, group_size) * static_cast<size_t>(M) < (1ull << 31) &&
           Kp * 2 * static_cast<size_t>(N) < (1ull << 31);
}

// Other shapes: one matvec per token column.
int matmul_by_columns(const uint8_t *w, const float *x, float *y, int M, int K, int N, int group_size,
                      hipStream_t stream) {
    for (int n = 0; n < N; ++n) {
        const int st = launch_i4_matvec(w, x + static_cast<size_t>(n) * K, y + static_cast<size_t>(n) * M, M, K,
                                        group_size, stream);
        if (st != kOk) return st;
    }
    return kOk;
}

// X's fp16 copy and per-token scales; perm: in the packed dequantization's k-slot order.
template <bool PERM>
void launch_x_to_f16(const float *x, int K, int Kp, int N, _Float16 *xh, float *xinv, hipStream_t stream) {
    const bool vec = K % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;  // 16-byte loads
    const auto kernel = vec && Kp <= 2048   ? x_to_f16_vec<PERM, 1>
                        : vec && Kp <= 4096 ? x_to_f16_vec<PERM, 2>
                        : vec && Kp <= 8192 ? x_to_f16_vec<PERM, 4>
                        : vec && Kp <= 2048 * kXVecMax ? x_to_f16_vec<PERM, kXVecMax>
                        : Kp <= 256 * kXRegs           ? x_to_f16<PERM>
                                                       : x_to_f16_long<PERM>;
    hipLaunchKernelGGL(kernel, dim3(N), dim3(256), 0, stream, x, K, Kp, xh, xinv);
}
void launch_x_to_f16(bool perm, const float *x, int K, int Kp, int N, _Float16 *xh, float *xinv, hipStream_t stream) {
    if (perm)
        launch_x_to_f16<true>(x, K, Kp, N, xh, xinv, stream);
    else
        launch_x_to_f16<false>(x, K, Kp, N, xh, xinv, stream);
}

// The partials of a split call follow X's copy in the workspace.
size_t part_offset(int K, int N) { return (prefill_scratch_bytes(K, N) + 255) / 256 * 256; }

// The MFMA path with X's fp16 copy and per-token scales at ws (prefill_scratch_bytes(K, N) bytes), and
// with arrivals (tl.tiles counters, zero between launches) the partials of a split call after
// them; arrivals null: its slices one after the other.
int matmul_mfma(const uint8_t *w, const float *x, float *y, int M, int K, int N, int group_size, unsigned char *ws,
                const TilePlan &tl, unsigned long long *arrivals, hipStream_t stream) {
    const size_t rb = i4_row_bytes(K, group_size);
    const size_t Kp = (static_cast<size_t>(K) + kStepK - 1) / kStepK * kStepK;
    const size_t xh_bytes = (Kp * 2 * N + 255) / 256 * 256;
    _Float16 *xh = reinterpret_cast<_Float16 *>(ws);
    float *xinv = reinterpret_cast<float *>(ws + xh_bytes);
    const int ikp = static_cast<int>(Kp), irb = static_cast<int>(rb);
    launch_x_to_f16(group_size == 64, x, K, ikp, N, xh, xinv, stream);
    if (hipGetLastError() != hipSuccess) return kLaunchFailed;
    const Slices sl{tl.KS, arrivals ? reinterpret_cast<float *>(ws + part_offset(K, N)) : nullptr, arrivals};
    const auto go = [&](auto gc, auto wnc, auto sc, auto wvc) {
        constexpr int GT = decltype(gc)::value, WN = decltype(wnc)::value, S = decltype(sc)::value,
                      NWV = decltype(wvc)::value;
        if constexpr (WN <= 2 && NWV == 4) {
            if (tl.KS > 1 && sl.part)
                return launch_direct<GT, WN, S, NWV, kSplitParts>(w, xh, xinv, y, M, N, K, ikp, group_size, irb, sl,
                                                                  stream);
            if (tl.KS > 1)
                return launch_direct<GT, WN, S, NWV, kSplitSeq>(w, xh, xinv, y, M, N, K, ikp, group_size, irb, sl,
                                                                stream);
        }
        return launch_direct<GT, WN, S, NWV, kSplitNone>(w, xh, xinv, y, M, N, K, ikp, group_size, irb, sl, stream);
    };
    const auto tiles = [&](auto gc) {
        const std::integral_constant<int, 1> c1;
        const std::integral_constant<int, 2> c2;
        const std::integral_constant<int, 3> c3;
        const std::integral_constant<int, 4> c4;
        const std::integral_constant<int, 8> c8;
        constexpr int GT = decltype(gc)::value;
        const int st = tl.kind == kTile128x32   ? go(gc, c1, c4, c4)
                       : tl.kind == kTile128x64 ? go(gc, c2, c4, c4)
                       : tl.kind == kTile256x96 ? go(gc, c3, c3, c8)
                                                : static_cast<int>(kTooLarge);
        if (st != kTooLarge) return st;  // (rows whose tile passes the 32-bit offsets: the smallest tile)
        return launch_direct<GT, 1, 4, 1, kSplitNone>(w, xh, xinv, y, M, N, K, ikp, group_size, irb, sl, stream);
    };
    return group_size == 64 ? tiles(std::integral_constant<int, 64>{}) : tiles(std::integral_constant<int, 0>{});
}

// ---- allocation-free variant --------------------------------------------------------------
// `scratch` holds X's fp16 copy and the per-token scales for callers that cannot
// allocate (code under graph capture, serving loops). Every GPU the library runs on
// holds its own copy for the life of the process; all calls on one GPU share it, so
// calls that overlap on one GPU race. Nothing in it has to start at zero: x_to_f16
// writes every byte the GEMM reads (the padding columns included).
// The last kNoAllocArrivalBytes are the few-token kernel's arrival counters: zero when the
// code object is loaded and after every launch, and never written by anything else.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
constexpr size_t kNoAllocArrivalBytes = size_t{64} << 10;
constexpr size_t kNoAllocWorkBytes = kNoAllocScratchBytes - kNoAllocArrivalBytes;

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices];  // device address of `scratch` on each device, once looked up

// The device address of `scratch` on the current device. The host-side name is only a
// handle for the lookup; kernels get this address.
int noalloc_scratch(unsigned char **out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return kHipFailed;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return kHipFailed;
        g_scratch_ptr[dev] = p;
    }
    *out = static_cast<unsigned char *>(g_scratch_ptr[dev]);
    return kOk;
}

}  // namespace

int launch_i4_matmul_noalloc(const uint8_t *w, const float *x, float *y, int M, int K, int N, int group_size,
                             hipStream_t stream) {
    if (M < 1 || K < 1 || N < 1 || group_size < 2 || (group_size & 1)) return kBadShape;
    // (the size checks below come first, so a call's ENOSCRATCH does not depend on its pointers;
    // every launch below is preceded by the null check)
    const bool operands = w && x && y;
    if (skinny_applies(x, K, N, group_size)) {
        // launch_i4_matmul runs the few-token kernel here; another kernel would give other
        // bits, so a call whose partials do not fit is refused rather than rerouted
        // (e.g. 151936x896 at up to 32 tokens: 1187 tiles x 2 slices x 16 KiB).
        const SkinnyGeom g = skinny_geom(M, K, device_cu_count());
        if (g.room > kNoAllocWorkBytes || static_cast<size_t>(g.tiles) * 8 > kNoAllocArrivalBytes)
            return kNoScratch;
        if (!operands) return kBadShape;
        unsigned char *ws = nullptr;
        const int st = noalloc_scratch(&ws);
        if (st != kOk) return st;
        return launch_skinny(w, x, y, M, K, N, g, reinterpret_cast<float *>(ws),
                             reinterpret_cast<unsigned long long *>(ws + kNoAllocWorkBytes), stream);
    }
    const bool mfma = mfma_applies(M, K, N, group_size);
    if (mfma && prefill_scratch_bytes(K, N) > kNoAllocWorkBytes) return kNoScratch;
    if (!operands) return kBadShape;
    unsigned char *ws = nullptr;
    if (mfma) {
        const int st = noalloc_scratch(&ws);
        if (st != kOk) return st;
        return matmul_mfma(w, x, y, M, K, N, group_size, ws, tile_plan(M, K, N), nullptr, stream);
    }
    // One matvec per token column under a scratch set with no buffers: a kernel that would
    // need split-K slots is not chosen, and nothing is allocated.
    static ScratchSet *none = scratch_set_fixed(nullptr, 0);
    ScratchScope scope(none);
    return matmul_by_columns(w, x, y, M, K, N, group_size, stream);
}

int launch_i4_matmul(const uint8_t *w, const float *x, float *y, int M, int K, int N, int group_size,
                     hipStream_t stream) {
    if (M < 1 || K < 1 || N < 1 || group_size < 2 || (group_size & 1)) return kBadShape;
    if (!w || !x || !y) return kBadShape;  // nothing is launched on a null operand
    if (skinny_applies(x, K, N, group_size)) {
        const SkinnyGeom g = skinny_geom(M, K, device_cu_count());
        unsigned long long *slots = nullptr;  // zero between launches: the arrival counters
        int st = scratch_split_slots(stream, static_cast<size_t>(g.tiles), &slots);
        if (st != kOk) return st;
        void *part = nullptr;
        st = scratch_prefill(stream, g.part_bytes, &part);
        if (st != kOk) return st;
        return launch_skinny(w, x, y, M, K, N, g, static_cast<float *>(part), slots, stream);
    }
    if (!mfma_applies(M, K, N, group_size)) return matmul_by_columns(w, x, y, M, K, N, group_size, stream);
    const TilePlan tl = tile_plan(M, K, N);
    void *ws = nullptr;  // the stream's (or scope's) buffer
    unsigned long long *arrivals = nullptr;
    if (tl.KS > 1 && (scratch_prefill(stream, part_offset(K, N) + tl.part_bytes, &ws) != kOk ||
                      scratch_split_slots(stream, tl.tiles, &arrivals) != kOk)) {
        // no room for the partials (a capture, or memory is short): the slices one after the other
        ws = nullptr;
        arrivals = nullptr;
        (void)hipGetLastError();
    }
    if (!ws) {
        const int st = scratch_prefill(stream, prefill_scratch_bytes(K, N), &ws);
        if (st != kOk) return st;
    }
    const int st = matmul_mfma(w, x, y, M, K, N, group_size, static_cast<unsigned char *>(ws), tl, arrivals, stream);
    return st == kTooLarge ? matmul_by_columns(w, x, y, M, K, N, group_size, stream) : st;
}

}  // namespace tqhip
