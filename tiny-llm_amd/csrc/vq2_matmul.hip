// vq2_matmul.hip -- batched VQ2 (d=4, 256-entry fp16 codebook) product for gfx950.
//
// Y[M,N] = W_vq2[M,K] * X[K,N] with X and Y column-major (x[n*K+k], y[n*M+m]): matvec_vq2_ref
// (kernels/matvec/matvec_vq2_ref.cpp:52-81) for every token, as the reference's matmul_vq2
// decomposes it (kernels/dispatch.cpp:511-532).
//
// The weights are fp16 codebook entries and the activations fp32, so the product runs on the fp32
// matrix instruction, v_mfma_f32_32x32x2_f32: every operand exact, fp32 accumulation, as the
// matvec kernels' FMAs. A workgroup of eight waves owns 32 rows and 32 WN tokens; its waves deal
// the row's chunks of 8 indices (32 elements) among them and their sums meet in LDS in wave order
// (the same bits every time). Lane (row or token l % 32, half h = l / 32) takes indices 4 h .. 4 h
// + 3 of a chunk: one dword of indices, four codebook entries from LDS (8 bytes each), four
// 16-byte activation loads per token block straight from global memory, and the k-slot h of MFMA
// (j, i) holds element i of its index j on both operands. The next chunk's loads are in flight
// during the current one's MFMAs.
//
// A call on host arrays (matmul_vq2) was one matvec per token, each with its own upload, launch,
// download and wait: 64 tokens through a layer of 896 / 4864 wide matrices took 8.5 ms. With this
// kernel it is one of each per matrix, 590 us, of which the seven products take 114 (5-13 us each:
// launch and load latency; the matrix instructions alone need 3 us at 4864x896) and the copies
// the rest.

#include "tq_common.h"

namespace tqhip {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kMmWaves = 8;
constexpr int kMmThreads = 64 * kMmWaves;
constexpr unsigned kPastEnd = 0xFFFFFFF0u;  // a buffer offset past any record: reads 0

__device__ inline float half_f(unsigned h) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<unsigned short>(h & 0xFFFFu)));
}

// ALIGNED: index rows are dword-aligned (K % 16 == 0 and w too), one load per lane and chunk.
template <int WN, bool ALIGNED>
__global__ __launch_bounds__(kMmThreads) void vq2_matmul(const uint8_t *__restrict__ w, const float *__restrict__ x,
                                                         float *__restrict__ y, int M, int N, int K, int vec_y) {
    __shared__ uint2 cb[kVq2Entries];
    __shared__ float4 red[kMmWaves][WN][4][64];
    const int lane = threadIdx.x & 63, li = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = 32 * blockIdx.x, n0 = 32 * WN * blockIdx.y;
    const int nb = K / kVq2Dim, chunks = (nb + 7) / 8;

    const uint8_t *rows = w + kVq2CodebookBytes + static_cast<size_t>(m0) * nb;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(rows), static_cast<short>(0), min(32, M - m0) * nb, 0x00020000);
    const float4 *xp[WN];
#pragma unroll
    for (int j = 0; j < WN; ++j)  // (tokens past N repeat the last one and are not stored)
        xp[j] = reinterpret_cast<const float4 *>(x + static_cast<size_t>(min(n0 + 32 * j + li, N - 1)) * K);

    struct Chunk {
        unsigned q;
        float4 x[WN][4];
    };
    const auto load = [&](int c, Chunk &d) {
        const int p0 = 8 * c + 4 * h;
        if constexpr (ALIGNED) {
            d.q = __builtin_amdgcn_raw_buffer_load_b32(rs, p0 < nb ? li * nb + p0 : kPastEnd, 0, 0);
        } else {
            d.q = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                d.q |= static_cast<unsigned>(
                           __builtin_amdgcn_raw_buffer_load_b8(rs, p0 + i < nb ? li * nb + p0 + i : kPastEnd, 0, 0))
                       << (8 * i);
        }
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) d.x[j][i] = xp[j][min(p0 + i, nb - 1)];
    };
    f16v acc[WN];
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[j] = f16v{};
    const auto compute = [&](int c, const Chunk &d) {
        const int p0 = 8 * c + 4 * h;
        f16v t[WN];
#pragma unroll
        for (int j = 0; j < WN; ++j) t[j] = f16v{};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint2 e = cb[(d.q >> (8 * i)) & 0xFFu];
            const bool in = p0 + i < nb;  // past the row end: exactly nothing (entry 0 may be non-finite)
            const float a[4] = {in ? half_f(e.x) : 0.f, in ? half_f(e.x >> 16) : 0.f, in ? half_f(e.y) : 0.f,
                                in ? half_f(e.y >> 16) : 0.f};
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const float b[4] = {in ? d.x[j][i].x : 0.f, in ? d.x[j][i].y : 0.f, in ? d.x[j][i].z : 0.f,
                                    in ? d.x[j][i].w : 0.f};
#pragma unroll
                for (int s = 0; s < 4; ++s) t[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[s], t[j], 0, 0, 0);
            }
        }
        // a chunk's sum starts from zero and is added once: shorter chains of roundings than one
        // accumulation over the row (error against 64 bits at K 4864: 1.4e-7, with one chain per
        // wave 4.4e-7; the matvec kernels' 64 lane sums 1.7e-7)
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[j] += t[j];
    };

    Chunk even, odd;
    if (wave < chunks) load(wave, even);
    if (threadIdx.x < kVq2Entries) {
        const unsigned *e = reinterpret_cast<const unsigned *>(w) + 2 * threadIdx.x;
        cb[threadIdx.x] = make_uint2(e[0], e[1]);
    }
    __syncthreads();
    for (int c = wave; c < chunks; c += 2 * kMmWaves) {
        if (c + kMmWaves < chunks) load(c + kMmWaves, odd);
        compute(c, even);
        if (c + kMmWaves >= chunks) break;
        if (c + 2 * kMmWaves < chunks) load(c + 2 * kMmWaves, even);
        compute(c + kMmWaves, odd);
    }

    // D: lane holds rows 8 (r / 4) + 4 h + r % 4 of token l % 32
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
            red[wave][j][r4][lane] =
                make_float4(acc[j][4 * r4], acc[j][4 * r4 + 1], acc[j][4 * r4 + 2], acc[j][4 * r4 + 3]);
    __syncthreads();
    const float4 *flat = &red[0][0][0][0];
    constexpr int kOut = 256 * WN;  // float4s of the tile
    for (int t = threadIdx.x; t < kOut; t += kMmThreads) {
        float4 s = flat[t];
#pragma unroll
        for (int v = 1; v < kMmWaves; ++v) {
            const float4 p = flat[kOut * v + t];
            s.x += p.x;
            s.y += p.y;
            s.z += p.z;
            s.w += p.w;
        }
        const int n = n0 + 32 * (t >> 8) + (t & 31), m = m0 + 8 * ((t >> 6) & 3) + 4 * ((t >> 5) & 1);
        if (n >= N) continue;
        float *yc = y + static_cast<size_t>(n) * M + m;
        if (vec_y && m + 3 < M) {
            *reinterpret_cast<float4 *>(yc) = s;
        } else {
            const float v[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (m + i < M) yc[i] = v[i];
        }
    }
}

// Whether one matvec per token is faster than the matrix launch: a wave takes every eighth chunk of its row
// one after the other, 6.4 ns an element of the row whatever the number of tokens up to 32, and a matvec
// takes 2.2 us and 0.7 ns an element. A call on host arrays of 896 rows, us, matrix launch and matvecs:
// 2 tokens of 896 elements 25 and 23, of 2560 46 and 36, of 9728 87 and 47; 6 tokens of 2560 55 and 59, of 4864 69
// and 68, of 9728 99 and 90; 8 tokens of 9728 105 and 113. (Rows that are not a multiple of 16 elements: 4 us
// and more a matvec, 26 and 33 at 2 tokens of 1004.)
bool matvecs_are_faster(int K, int N) { return K % 16 == 0 && N * (2200.0 + 0.7 * K) < 6.4 * K; }

}  // namespace

int launch_vq2_matmul(const uint8_t *w, const float *x, float *y, int M, int K, int N, hipStream_t stream) {
    if (M < 1 || N < 1 || K < kVq2Dim || K % kVq2Dim || !w || !x || !y) return kBadShape;
    // 16-byte activation loads, 32-bit offsets within 32 index rows, and at most 65535 token tiles
    if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(w) & 3) || K >= (1 << 26) ||
        N > 32 * 65535 || matvecs_are_faster(K, N))
        return kNotFused;
    const bool aligned = K % 16 == 0;
    const int vec_y = M % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
    const int rows = (M - 1) / 32 + 1;
    // Two token blocks a wave share the codebook lookups and halve the index reads, where that
    // still leaves a workgroup per CU.
    const bool two = N > 32 && static_cast<long long>(rows) * ((N + 63) / 64) >= device_cu_count();
    const dim3 grid(rows, two ? (N + 63) / 64 : (N + 31) / 32), block(kMmThreads);
    const auto kernel = two ? (aligned ? vq2_matmul<2, true> : vq2_matmul<2, false>)
                            : (aligned ? vq2_matmul<1, true> : vq2_matmul<1, false>);
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, w, x, y, M, N, K, vec_y);
    return hipGetLastError() == hipSuccess ? kOk : kLaunchFailed;
}

}  // namespace tqhip
