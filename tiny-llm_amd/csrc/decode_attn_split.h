// decode_attn_split.h -- a decode step's attention with the sequence split over workgroups, for
// the engine's steps at long contexts (from split_from(head_dim) positions on).
//
// attention_step (decode_attn.h) gives a query head one workgroup, so a step costs what one CU
// takes to read the head's whole cache: 10 us at 250 positions, 24 at 1500, 46 at 3000 (14 heads
// of 64 on 2 K/V heads, MI355X), with 242 of 256 CUs idle. Here a workgroup of four waves takes a
// part of the sequence for one head, in a grid of parts x heads: 6.8, 9.1 and 10.3 us, latency
// (loads, softmax, the exchange below), not bytes: 3 MB of cache per layer at 3000 positions.
//
//   - A wave takes tiles of 64 positions, one per lane. A lane holds its position's key row and
//     forms its score from the rotated q in LDS (broadcast reads); maximum and sum of the tile are
//     wave reductions, and the value rows are read with one dimension per lane, the probabilities
//     through v_readlane. The four waves meet once, in LDS, after their tiles.
//   - Every wave finishes the head's q itself (biases, norms, RoPE: the operations of
//     attention_head); the wave that holds the step's own position also finishes k and v, uses
//     them from registers and, for the group's first head, stores them to the cache.
//   - Up to 256 positions one workgroup holds the sequence and stores the output. Beyond, the
//     parts' (maximum, sum, output) meet in HBM at device scope: each workgroup stores its partial,
//     waits for the store, and adds one to its head's arrival counter; the last one combines the
//     parts in part order (the same bits whatever the arrival order) and resets the counter. The
//     extra round trips (store, counter, read back) cost about 2 us. One wave per part, so four
//     times the parts, took 11.6 us at 2000 positions; two or four heads per wave 12.3 and 14.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "decode_attn.h"

namespace tqhip {
namespace {

constexpr int kSplitTile = 64;        // positions per tile: one per lane
constexpr int kSplitWaves = 4;        // waves of a workgroup: that many tiles side by side
constexpr int kSplitMaxParts = 128;   // parts of a sequence (longer sequences: several tiles a wave)

// Position from which a step runs the split attention, and what a step's layer takes there and nearby, us,
// attention_step against it: 14 heads of 64 19.2 and 21.0 at 64, 21.0 and 21.6 at 152, 21.7 and 21.6 at 160, 23.4 and 22.2
// at 240; 32 heads of 128 24.0 and 29.6 at 64, 31.2 and 31.4 at 216, 32.0 and 31.5 at 224; 4 heads of 256 26.4 and
// 37.7 at 64, 41.4 and 41.6 at 224, 42.1 and 41.8 at 232. What it loses is before the scores:
// attention_step's first wave has its keys requested before the position is known.
constexpr int split_from(int head_dim) { return head_dim == 64 ? 160 : kAttnPositions; }
static_assert(split_from(64) <= kAttnPositions && split_from(128) <= kAttnPositions, "attention_step's positions");

constexpr int kSplitSpan = kSplitTile * kSplitWaves;  // positions of a workgroup whose waves take one tile each

// Parts in the grid of steps up to `positions` positions: `first` times a power of two, enough for one
// tile a wave, up to kSplitMaxParts. The engine keeps a graph per grid and a step takes the smallest
// that covers its sequence: with one grid for the whole cache, 32 heads of 128 in a cache of 32768
// positions took 78 us a layer at position 180 instead of 31 (a workgroup without positions still takes a
// CU until it has read the position, and a CU holds one of these workgroups).
inline int split_parts(int positions, int first) {
    int parts = first;
    while (parts < kSplitMaxParts && parts * kSplitSpan < positions) parts *= 2;
    return parts;
}
// The smallest grid: 8 parts, so that the heads that read one part of a K/V head's cache land on one
// XCD and share its L2 (14 heads of 64 at 180 positions: a step's layer takes 21.9 us, with one part and
// the heads dealt over the XCDs 22.2), or with more heads the 4, 2 or 1 whose workgroups are resident
// at once, one per CU (64 heads of 128 at 160 to 250 positions: 34 us with 4 parts, 46 with 8).
inline int split_first_parts(int n_heads, int cus) {
    int parts = 8;
    while (parts > 1 && parts * n_heads > cus) parts /= 2;
    return parts;
}
// Grid of `parts` parts: the first 2^shift (at most 8) of every head, then the next 8, so that parts
// which the sequence does not reach go out last.
inline int split_shift(int parts) { return parts >= 8 ? 3 : parts == 4 ? 2 : parts - 1; }
inline dim3 split_grid(int n_heads, int parts) {
    return dim3(n_heads << split_shift(parts), parts >> split_shift(parts));
}
// Floats of the partials of n_heads heads: per (head, part) HD outputs, then a record
// {maximum, 0, sum as a double}.
inline size_t split_partial_floats(int n_heads, int hd, int parts) {
    return static_cast<size_t>(n_heads) * parts * (hd + 4);
}

// Relaxed device-scope accesses of the partials: a store is written through this XCD's L2, a load
// reads past it, so a store that has completed is seen by every later load.
__device__ inline void split_st(float *p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void split_st8(void *p, unsigned long long v) {
    __hip_atomic_store(static_cast<unsigned long long *>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned long long split_ld8(const void *p) {
    return __hip_atomic_load(static_cast<const unsigned long long *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline float split_lane(float v, int lane) {  // lane's value (lane uniform) as a scalar
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// One head slice of 64 * E elements held by a wave, element lane + 64 e in x[e]: RMSNorm
// (rmsnorm_ref on the head) when w is given, then RoPE with the lane's angles (c, s).
template <int HD>
__device__ inline void split_finish(float (&x)[HD / 64], const float *nw, const float (&c)[(HD + 127) / 128],
                                    const float (&s)[(HD + 127) / 128], float eps, bool norm, int lane) {
#pragma clang fp contract(off)
    constexpr int E = HD / 64;
    if (norm) {
        double ss = 0.0;
#pragma unroll
        for (int e = 0; e < E; ++e) ss += static_cast<double>(x[e]) * static_cast<double>(x[e]);
        ss = xor_sum_wave(ss);
        const float r = 1.0f / sqrtf(static_cast<float>(ss / HD) + eps);
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = (x[e] * r) * nw[e];
    }
    if constexpr (E == 1) {
        const float other = lane_xor<32>(x[0], lane);
        x[0] = lane < 32 ? x[0] * c[0] - other * s[0] : x[0] * c[0] + other * s[0];
    } else {
#pragma unroll
        for (int e = 0; e < E / 2; ++e) {
            const float x0 = x[e], x1 = x[e + E / 2];
            x[e] = x0 * c[e] - x1 * s[e];
            x[e + E / 2] = x1 * c[e] + x0 * s[e];
        }
    }
}

template <int HD>
__global__ __launch_bounds__(64 * kSplitWaves) void attention_split(
    int heads_per_kv, int n_heads, int shift, int max_seq, float theta, float eps, float scale, const int *pos_ptr,
    const float *q, const float *k, const float *v, const float *qb, const float *kb, const float *vb, const float *qn,
    const float *kn, float *kcache, float *vcache, float *partial, unsigned *arrivals, float *out) {
    constexpr int E = HD / 64, A = (HD + 127) / 128, half = HD / 2, NW = kSplitWaves;
    constexpr int VB = E == 1 ? 64 : E == 2 ? 16 : 8;  // value rows in flight (registers)
    __shared__ __attribute__((aligned(16))) float qs[NW][HD];
    __shared__ __attribute__((aligned(16))) float os[NW][HD];  // the waves' outputs
    __shared__ float ms[NW], ws[kSplitMaxParts];
    __shared__ double ls[NW];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int parts_grid = gridDim.y << shift, part = (blockIdx.y << shift) + (blockIdx.x & ((1 << shift) - 1));
    const int head = blockIdx.x >> shift, kvh = head / heads_per_kv;

    // the raw q of the head and k and v of its group, their biases and norm weights (absent ones:
    // the projection itself, unused). None of these loads depends on the position, and all are
    // unconditional: behind branches each would be waited for before the next is issued.
    float qv[E], kv[E], vv[E], bq[E], bk[E], bv[E], qn_w[E], kn_w[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int d = lane + 64 * e, qi = head * HD + d, ki = kvh * HD + d;
        qv[e] = q[qi];
        bq[e] = (qb ? qb : q)[qi];
        kv[e] = k[ki];
        bk[e] = (kb ? kb : k)[ki];
        vv[e] = v[ki];
        bv[e] = (vb ? vb : v)[ki];
        qn_w[e] = (qn ? qn : q)[d];
        kn_w[e] = (kn ? kn : q)[d];
    }
    __builtin_amdgcn_sched_barrier(0);
    const int pos = *pos_ptr, seq = pos + 1;
    const int tiles = (seq + kSplitTile - 1) / kSplitTile;
    const int per_wave = (tiles + NW * parts_grid - 1) / (NW * parts_grid);
    const int parts = (tiles + NW * per_wave - 1) / (NW * per_wave);
    if (part >= parts) return;
    const int tile0 = (part * NW + wave) * per_wave, tile_end = min(tiles, tile0 + per_wave);

    const float *kh = kcache + static_cast<size_t>(kvh) * max_seq * HD;
    const float *vh = vcache + static_cast<size_t>(kvh) * max_seq * HD;
    // Rows below pos are read: row pos is written by this launch and the rows after it are not there
    // yet (or left by a longer sequence before a reset, and not finite then). A lane past them reads
    // the key row before pos, unused; a tile's value rows go through a buffer that ends at row pos,
    // past which a load gives 0. The scalar offset of a load stays within that buffer: the range
    // check subtracts it from the buffer's size, and what a difference below zero does is not said.
    const int last_row = max(pos - 1, 0);
    constexpr int KS = HD > 128 ? 64 : HD;  // key elements held at once (the VGPRs' limit)
    float4 kreg[KS / 4];
    float vreg[VB][E];
    const auto load_keys = [&](int t0, int k0) {
        const float *kr = kh + static_cast<size_t>(min(t0 + lane, last_row)) * HD + k0;
#pragma unroll
        for (int i = 0; i < KS / 4; ++i) kreg[i] = attn_ld4(kr + 4 * i);
    };
    const auto load_values = [&](int t0, int b) {  // rows b VB .. of tile t0 / 64
        const int bytes = 4 * HD * min(max(pos - t0, 0), kSplitTile);
        const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(vh) + static_cast<size_t>(t0) * HD, static_cast<short>(0), bytes, 0x00020000);
        const int so = min(4 * HD * VB * b, bytes);
#pragma unroll
        for (int u = 0; u < VB; ++u)
#pragma unroll
            for (int e = 0; e < E; ++e)
                vreg[u][e] =
                    __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(vr, 4 * (u * HD + lane + 64 * e), so, 0));
    };
    load_keys(tile0 * kSplitTile, 0);  // (a wave past the sequence reads the last row, unused)
    load_values(tile0 * kSplitTile, 0);
    __builtin_amdgcn_sched_barrier(0);  // (the cache loads go out before the work below waits for q)

    // RoPE angles of element lane (+ 64 a) of the lower half; HD 64: lanes 32.. take that of lane - 32
    float c[A], s[A];
#pragma unroll
    for (int a = 0; a < A; ++a) {
        const int i = E == 1 ? lane % half : lane + 64 * a;
        const float inv_freq = powf(theta, -static_cast<float>(2 * i) / static_cast<float>(HD));
        const float angle = static_cast<float>(pos) * inv_freq;
        c[a] = cosf(angle);
        s[a] = sinf(angle);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        qv[e] = qb ? qv[e] + bq[e] : qv[e];
        kv[e] = kb ? kv[e] + bk[e] : kv[e];
        vv[e] = vb ? vv[e] + bv[e] : vv[e];
    }
    split_finish<HD>(qv, qn_w, c, s, eps, qn != nullptr, lane);
#pragma unroll
    for (int e = 0; e < E; ++e) qs[wave][lane + 64 * e] = qv[e];
    float own = 0.0f;  // the score of the step's own position
    if (tile0 < tile_end && tile_end == tiles) {
        split_finish<HD>(kv, kn_w, c, s, eps, qn != nullptr, lane);
#pragma unroll
        for (int e = 0; e < E; ++e) own = fmaf(qv[e], kv[e], own);
        own = xor_sum_wave(own);
        if (head % heads_per_kv == 0) {
            float *kw = kcache + (static_cast<size_t>(kvh) * max_seq + pos) * HD;
            float *vw = vcache + (static_cast<size_t>(kvh) * max_seq + pos) * HD;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                attn_st(kw + lane + 64 * e, kv[e]);
                attn_st(vw + lane + 64 * e, vv[e]);
            }
        }
    }
    __builtin_amdgcn_wave_barrier();  // (a wave's LDS accesses are served in order: its q is there for its reads)

    float m = -INFINITY, acc[E] = {};
    double l = 0.0;
    for (int tile = tile0; tile < tile_end; ++tile) {
        const int t0 = tile * kSplitTile;
        if (tile != tile0) {
            load_keys(t0, 0);
            load_values(t0, 0);
        }
        float p4[4] = {};  // (four chains: one alone waits for each FMA)
        const auto dot_keys = [&](int k0) {
#pragma unroll
            for (int i = 0; i < KS / 4; ++i) {
                const float4 b = kreg[i], a = *reinterpret_cast<const float4 *>(&qs[wave][k0 + 4 * i]);
                p4[0] = fmaf(a.x, b.x, p4[0]);
                p4[1] = fmaf(a.y, b.y, p4[1]);
                p4[2] = fmaf(a.z, b.z, p4[2]);
                p4[3] = fmaf(a.w, b.w, p4[3]);
            }
        };
        dot_keys(0);
        if constexpr (KS < HD) {
#pragma unroll 1
            for (int k0 = KS; k0 < HD; k0 += KS) {
                load_keys(t0, k0);
                dot_keys(k0);
            }
        }
        const int j = t0 + lane;
        const float dot = (p4[0] + p4[1]) + (p4[2] + p4[3]);
        const float sc = j < pos ? dot * scale : j == pos ? own * scale : -INFINITY;
        const float m_new = fmaxf(m, xor_max_wave(sc));
        const float mu = m_new == -INFINITY ? 0.0f : m_new;  // (every score -inf: probabilities 0)
        const float p = expf(sc - mu), r = expf(m - mu);
        l = l * static_cast<double>(r) + xor_sum_wave(static_cast<double>(p));
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] *= r;
        m = m_new;
#pragma unroll 1
        for (int b = 0; b < kSplitTile / VB; ++b) {
            if (b > 0) load_values(t0, b);
            float a2[2][E] = {};  // even and odd rows
#pragma unroll
            for (int u = 0; u < VB; ++u) {
                const float pj = split_lane(p, b * VB + u);
#pragma unroll
                for (int e = 0; e < E; ++e) a2[u & 1][e] = fmaf(pj, vreg[u][e], a2[u & 1][e]);
            }
#pragma unroll
            for (int e = 0; e < E; ++e) acc[e] += a2[0][e] + a2[1][e];
        }
        if (t0 + kSplitTile > pos) {  // the step's own value row (its row above was read as 0)
            const float pj = split_lane(p, pos - t0);
#pragma unroll
            for (int e = 0; e < E; ++e) acc[e] = fmaf(pj, vv[e], acc[e]);
        }
    }

    // the waves' parts, added by wave 0 in wave order
#pragma unroll
    for (int e = 0; e < E; ++e) os[wave][lane + 64 * e] = acc[e];
    if (lane == 0) {
        ms[wave] = m;
        ls[wave] = l;
    }
    __syncthreads();
    if (wave != 0) return;
    m = ms[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) m = fmaxf(m, ms[w]);
    l = 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] = 0.0f;
    const float mu = m == -INFINITY ? 0.0f : m;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const float r = expf(ms[w] - mu);
        l += static_cast<double>(r) * ls[w];
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] = fmaf(r, os[w][lane + 64 * e], acc[e]);
    }
    if (parts == 1) {
        const float inv = 1.0f / static_cast<float>(l);
#pragma unroll
        for (int e = 0; e < E; ++e) out[head * HD + lane + 64 * e] = acc[e] * inv;
        return;
    }

    // partial (head, part) is row head * parts_grid + part: HD outputs, and after all of those the
    // records {maximum, 0, sum as a double}
    float *po = partial + static_cast<size_t>(head) * parts_grid * HD;
    float *rec = partial + static_cast<size_t>(n_heads) * parts_grid * HD + 4 * static_cast<size_t>(head) * parts_grid;
#pragma unroll
    for (int e = 0; e < E; ++e) split_st(po + part * HD + lane + 64 * e, acc[e]);
    if (lane == 0) {
        split_st8(rec + 4 * part, __float_as_uint(m));
        split_st8(rec + 4 * part + 2, __builtin_bit_cast(unsigned long long, l));
    }
    // the partial is at the device's point of coherence before the arrival is counted
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    unsigned seen = 0;
    if (lane == 0) seen = __hip_atomic_fetch_add(arrivals + head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    seen = __builtin_amdgcn_readfirstlane(seen);
    if (seen != static_cast<unsigned>(parts - 1)) return;
    if (lane == 0) __hip_atomic_store(arrivals + head, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" ::: "memory");

    // The last arrival: lane i takes the records of parts i, i + 64, ...; of the outputs, lane takes
    // float4 lane % LR of the rows lane / LR + RG u. The first RB RG rows are requested together
    // with the records (one round trip).
    constexpr int LR = HD / 4, RG = 64 / LR, RB = 8, PR = kSplitMaxParts / 64;
    float pm[PR];
    double pl[PR];
    unsigned long long xy[RB], zw[RB];
    const int row_of = lane / LR;
    const auto load_rows = [&](int p0) {
#pragma unroll
        for (int u = 0; u < RB; ++u) {
            const float *r = po + min(p0 + RG * u, parts - 1) * HD + 4 * (lane % LR);
            xy[u] = split_ld8(r);
            zw[u] = split_ld8(r + 2);
        }
    };
#pragma unroll
    for (int i = 0; i < PR; ++i) {
        const int pi = min(lane + 64 * i, parts - 1);
        pm[i] = __uint_as_float(static_cast<unsigned>(split_ld8(rec + 4 * pi)));
        pl[i] = __builtin_bit_cast(double, split_ld8(rec + 4 * pi + 2));
    }
    load_rows(row_of);
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < PR; ++i) {
        pm[i] = lane + 64 * i < parts ? pm[i] : -INFINITY;
        top = fmaxf(top, pm[i]);
    }
    top = xor_max_wave(top);
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < PR; ++i) {
        const bool in = lane + 64 * i < parts;
        const float w = in ? expf(pm[i] - top) : 0.0f;
        ws[lane + 64 * i] = w;
        sum += in ? static_cast<double>(w) * pl[i] : 0.0;
    }
    const float inv = 1.0f / static_cast<float>(xor_sum_wave(sum));
    __builtin_amdgcn_wave_barrier();
    float4 t = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int p0 = row_of; p0 < parts; p0 += RB * RG) {
        if (p0 != row_of) load_rows(p0);
#pragma unroll
        for (int u = 0; u < RB; ++u) {
            const int pi = p0 + RG * u;
            const float w = ws[min(pi, parts - 1)];
            const bool in = pi < parts;
            t.x = in ? fmaf(w, __uint_as_float(static_cast<unsigned>(xy[u])), t.x) : t.x;
            t.y = in ? fmaf(w, __uint_as_float(static_cast<unsigned>(xy[u] >> 32)), t.y) : t.y;
            t.z = in ? fmaf(w, __uint_as_float(static_cast<unsigned>(zw[u])), t.z) : t.z;
            t.w = in ? fmaf(w, __uint_as_float(static_cast<unsigned>(zw[u] >> 32)), t.w) : t.w;
        }
    }
    if constexpr (RG == 4) {
        t = make_float4(sum_rows4(t.x), sum_rows4(t.y), sum_rows4(t.z), sum_rows4(t.w));
    } else if constexpr (RG == 2) {
        t.x += lane_xor<32>(t.x, lane);
        t.y += lane_xor<32>(t.y, lane);
        t.z += lane_xor<32>(t.z, lane);
        t.w += lane_xor<32>(t.w, lane);
    }
    if (lane < LR)
        *reinterpret_cast<float4 *>(out + head * HD + 4 * lane) =
            make_float4(t.x * inv, t.y * inv, t.z * inv, t.w * inv);
}

}  // namespace
}  // namespace tqhip
