// int8 quantise-and-append of K/V rows, and the reference's query preparation (RMS head norm
// with gains), one wave64 a (token, kv head, K or V) / a (token, head).
//
// Quantisation follows write_row8 (Sources/EmblaMetal/Kernels/common.metal:72-84) with kv_append /
// kv_append_b as callers (attention.metal:113-140, prefill.metal:182-212):
//   v_i = x_i (bf16-rounded when the input is bf16: the reference's bf()),
//   a = max |v_i|, q_i = rint(v_i * (127 / a)) (0 when a = 0), scale = a / 127
// stored as fp32 (reference) or fp16 (config). With norm_k the K row is first RMS-normed without
// gains (head_norm with ng = 0, common.metal:13-26): r = 1 / sqrt(Σx² / 128 + 2^-23).
// Bit-exactness: the squares are summed in a fixed butterfly (lane pairs xor 32, 16, .., 1 over
// per-lane sums of two squares) that the oracle restates; no fma contraction anywhere here.
#include "common.hpp"
#include "embla_internal.hpp"
#include "kv_row.hpp"

#pragma clang fp contract(off)

namespace embla {

/// One wave a (token, kv head, K or V): two dims a lane, quantised, then stored at their places
/// in the MFMA lane-order tiles (common.hpp; K's two bytes are adjacent, V's are not), or in plain
/// 128-byte rows for a cache that is read by gathering (row_major).
__global__ __launch_bounds__(64) void kv_quant_kernel(KVQuantArgs a) {
    const int lane = threadIdx.x;
    const int t = blockIdx.x, h = blockIdx.y;
    const bool is_v = blockIdx.z == 1;
    const int pos = a.p0 + t;
    const uint16_t* src = is_v ? a.v : a.k;
    int8_t* rows = is_v ? a.vc : a.kc;

    const uint32_t raw = *(const uint32_t*)(src + (size_t)t * a.stride + h * HD + 2 * lane);
    const float x0 = a.in_bf16 ? bf2f(raw & 0xFFFF) : h2f(raw & 0xFFFF);
    const float x1 = a.in_bf16 ? bf2f(raw >> 16) : h2f(raw >> 16);
    int q0, q1;
    const float am = quant_pair(x0, x1, !is_v && a.norm_k, a.in_bf16, q0, q1);
    store_pair8(rows, a.n_kv, a.max_s, h, pos, is_v, a.row_major, a.scale32, q0, q1, am, lane);
}

// waves a tile and rows a wave: a wave's rows are one serial chain (int8, 1024 / 2048 tokens of 4 heads:
// 5.3 / 6.4 us at 4 waves, 4.6 / 5.8 at 8, 4.35 / 5.7 at 16; ring with the pre-ops 4.6 / 5.7, 4.15 / 5.5,
// 4.1 / 5.55)
constexpr int TW = 16, TR = 32 / TW;

/// The same rows a 32-position tile at a time: a workgroup a (tile, kv head, K or V) quantises its
/// rows into LDS and writes the tile in whole 16-byte pieces. A wave a row stores V's bytes one by
/// one, 128 cache lines a row, and a 2048-token chunk of 4 heads is 16384 workgroups: 7.15 us where
/// this takes 5.7. A chunk's first and last tile may be partial: K's (and a row-major cache's) pieces
/// belong to one position each, V's are then stored byte by byte.
template <bool ROW_MAJOR>
__global__ __launch_bounds__(64 * TW) void kv_quant_tile_kernel(KVQuantArgs a) {
    constexpr int RS = HD + 16;   // bytes a row in LDS: 16-byte reads of 16 rows on distinct banks
    __shared__ __attribute__((aligned(16))) int8_t rows[32 * RS];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = blockIdx.y;
    const bool is_v = blockIdx.z == 1;
    const int tile = (a.p0 >> 5) + blockIdx.x, base = 32 * tile;
    const int k_lo = max(a.p0 - base, 0), k_hi = min(a.p0 + a.T - base, 32);   // the tile's new rows
    const uint16_t* src = (is_v ? a.v : a.k) + h * HD + 2 * lane;
    int8_t* dst = is_v ? a.vc : a.kc;
    uint32_t raw[TR];
#pragma unroll
    for (int i = 0; i < TR; i++) {   // (rows outside the chunk: a row of it, not stored)
        const int t = min(max(base + TR * w + i - a.p0, 0), a.T - 1);
        raw[i] = *(const uint32_t*)(src + (size_t)t * a.stride);
    }
    const size_t nrow = (size_t)a.n_kv * a.max_s * HD;
#pragma unroll
    for (int i = 0; i < TR; i++) {
        const int k = TR * w + i;
        const float x0 = a.in_bf16 ? bf2f(raw[i] & 0xFFFF) : h2f(raw[i] & 0xFFFF);
        const float x1 = a.in_bf16 ? bf2f(raw[i] >> 16) : h2f(raw[i] >> 16);
        int q0, q1;
        const float am = quant_pair(x0, x1, !is_v && a.norm_k, a.in_bf16, q0, q1);
        *(uint16_t*)(rows + k * RS + 2 * lane) = (uint16_t)((q0 & 0xFF) | ((q1 & 0xFF) << 8));
        if (lane == 0 && k >= k_lo && k < k_hi) {
            const size_t si = (size_t)h * a.max_s + base + k;
            if (a.scale32) ((float*)(dst + nrow))[si] = am / 127.0f;
            else ((uint16_t*)(dst + nrow))[si] = f2h(am / 127.0f);
        }
    }
    __syncthreads();
    if (threadIdx.x >= 256) return;
    const int j = w, l = lane;   // the thread's piece
    if (ROW_MAJOR) {
        const int k = threadIdx.x >> 3, d0 = 16 * (threadIdx.x & 7);
        if (k >= k_lo && k < k_hi)
            *(u4_t*)(dst + ((size_t)h * a.max_s + base + k) * HD + d0) = ld16(rows + k * RS + d0);
    } else if (!is_v) {
        const int k = 16 * (j >> 1) + (l & 15), d0 = 32 * (l >> 4) + 16 * (j & 1);
        if (k >= k_lo && k < k_hi) *(u4_t*)(dst + tile_base(h, a.max_s, base, 1) + (size_t)(64 * j + l) * 16) = ld16(rows + k * RS + d0);
    } else {
        // dims 8n + 2j and the next one, each of keys 16t + 4g + i in byte order (t, i)
        const int n = l & 15, g = l >> 4;
        u4_t v;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int8_t* p = rows + (16 * (c & 1) + 4 * g) * RS + 8 * n + 2 * j + (c >> 1);
            v[c] = (uint8_t)p[0] | ((uint32_t)(uint8_t)p[RS] << 8) | ((uint32_t)(uint8_t)p[2 * RS] << 16) |
                   ((uint32_t)(uint8_t)p[3 * RS] << 24);
        }
        int8_t* out = dst + tile_base(h, a.max_s, base, 1) + (size_t)(64 * j + l) * 16;
        if (k_lo == 0 && k_hi == 32) {
            *(u4_t*)out = v;
        } else {
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int k = 16 * ((e >> 2) & 1) + 4 * g + (e & 3);
                if (k >= k_lo && k < k_hi) out[e] = (int8_t)(v[e >> 2] >> (8 * (e & 3)));
            }
        }
    }
}

/// Rows (tokens x heads) above which an append goes a 32-position tile at a time; for few, the tile's
/// barrier and its second pass cost more than whole pieces save (us, a wave a row / a tile, at 1 to 8
/// heads alike): int8, 2048 rows 3.7 / 4.1, 3072 4.3 / 4.2, 4096 4.95 / 4.4 (fp32 scales 4.9 / 4.7), 8192
/// 7.15 / 5.7; ring 1024 2.8 / 3.2, 1536 3.1 / 3.2, 2048 3.4 / 3.2, 8192 5.9 / 4.25; ring with the
/// pre-ops 1024 3.5 / 3.8, 1536 4.1 / 3.9, 2048 4.4 / 3.9, 8192 8.7 / 5.55. Both lines lie a little above
/// where the two are equal (3000 and 1500), so that every call from there on gains.
constexpr int KV_TILE_ROWS = 4096, RING_TILE_ROWS = 2048;

int launch_kv_quant(const KVQuantArgs& a, hipStream_t st) {
    // the tile form writes 16-byte pieces: the caches' rows start on 16-byte boundaries, or a wave a row
    if (a.T * a.n_kv > KV_TILE_ROWS && !(((uintptr_t)a.kc | (uintptr_t)a.vc) & 15)) {
        const dim3 grid((a.p0 + a.T - 1) / 32 - a.p0 / 32 + 1, a.n_kv, 2);
        if (a.row_major) hipLaunchKernelGGL(kv_quant_tile_kernel<true>, grid, dim3(64 * TW), 0, st, a);
        else hipLaunchKernelGGL(kv_quant_tile_kernel<false>, grid, dim3(64 * TW), 0, st, a);
    } else {
        hipLaunchKernelGGL(kv_quant_kernel, dim3(a.T, a.n_kv, 2), dim3(64), 0, st, a);
    }
    return hipGetLastError() == hipSuccess ? EMBLA_OK : EMBLA_ERR_HIP;
}

/// Query rows normed with the gains (head_norm, common.metal:13-26), bf16-rounded as the
/// reference does before its attention (attention.metal:168-169; prefill.metal:406-426). A wave takes
/// ROWS (token, head) rows, their loads in flight together and the gains loaded once: a wave a row
/// and workgroup was 32768 workgroups for 2048 tokens, 10.4 us where this takes 8.2.
template <int ROWS>
__global__ __launch_bounds__(256) void q_prep_kernel(QPrepArgs a) {
    const int lane = threadIdx.x & 63, n = a.T * a.n_q;
    const int first = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * ROWS;   // rows token-major: t * n_q + h
    if (first >= n) return;
    uint32_t raw[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        const int row = min(first + i, n - 1), t = row / a.n_q, h = row % a.n_q;
        raw[i] = *(const uint32_t*)(a.qraw + (size_t)t * a.stride + h * HD + 2 * lane);
    }
    const f2_t ga = gain_pair(a.g1, a.ng >= 1, lane), gb = gain_pair(a.g2, a.ng >= 2, lane);
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        const int row = first + i;
        if (row >= n) return;   // uniform
        const int t = row / a.n_q, h = row % a.n_q;
        const f2_t x = q_prep_pair(raw[i], ga[0], ga[1], gb[0], gb[1]);
        uint16_t* out = a.out + (a.head_major ? (size_t)h * a.T + t : row) * HD + 2 * lane;
        const uint32_t o = a.out_bf16 ? (uint32_t)f2bf(x[0]) | ((uint32_t)f2bf(x[1]) << 16)
                                      : (uint32_t)f2h(x[0]) | ((uint32_t)f2h(x[1]) << 16);
        if (((uintptr_t)a.out & 3) == 0) {
            *(uint32_t*)out = o;
        } else {
            out[0] = (uint16_t)o;
            out[1] = (uint16_t)(o >> 16);
        }
    }
}

/// T positions p0 .. of 16-bit K and V rows into a ring (slot p % R, tile layout with ES = 2). With
/// gains (the reference's sliding layers, kv_sliding_b, prefill.metal:103-125) K is RMS-normed with
/// them, rotated (RoPE at its position) and rounded to bf16; with norm_k (a bf16 full-layer cache,
/// R = max_s: kv_append / kv_append_b without KV8, attention.metal:113-140, prefill.metal:182-212)
/// only RMS-normed and rounded; V is copied. One wave a (token, head).
__global__ __launch_bounds__(64) void ring_append_kernel(RingAppendArgs a) {
    const int lane = threadIdx.x, t = blockIdx.x, h = blockIdx.y;
    const int pos = a.p0 + t, slot = pos % a.R;
    const uint32_t kraw = *(const uint32_t*)(a.k + (size_t)t * a.stride + h * HD + 2 * lane);
    const uint32_t vraw = *(const uint32_t*)(a.v + (size_t)t * a.stride + h * HD + 2 * lane);
    uint32_t kout = kraw;
    if (a.kg) {   // bf16 rows with pre-ops
        const int d0 = (2 * lane) & 31;
        kout = norm_rope_pair(kraw, 1.0f + bf2f(a.kg[2 * lane]), 1.0f + bf2f(a.kg[2 * lane + 1]),
                              rope_pair(pos, kRopeFreq[d0], kRopeFreq[d0 + 1]), lane);
    } else if (a.norm_k) {   // bf16 rows of a full layer: RMS norm without gains (kv_append, no KV8)
        float x0 = bf2f(kraw & 0xFFFF), x1 = bf2f(kraw >> 16);
        const float r = rms_factor(x0, x1);
        kout = (uint32_t)f2bf(x0 * r) | ((uint32_t)f2bf(x1 * r) << 16);
    }
    *(uint32_t*)(a.kring + kt_off(h, a.R, slot, 2 * lane, 2) / 2) = kout;
    a.vring[vt_off(h, a.R, slot, 2 * lane, 2) / 2] = (uint16_t)(vraw & 0xFFFF);
    a.vring[vt_off(h, a.R, slot, 2 * lane + 1, 2) / 2] = (uint16_t)(vraw >> 16);
}

/// The same rows a 32-slot tile at a time (kv_quant_tile_kernel's way): a workgroup a (tile, head, K
/// or V), its rows into LDS, then whole 16-byte pieces; the tile's RoPE angles are evaluated once, into
/// LDS. 2048 tokens of 4 heads with the pre-ops: 8.7 us a wave a row, 5.55 this way.
__global__ __launch_bounds__(64 * TW) void ring_append_tile_kernel(RingAppendArgs a) {
    constexpr int RS = HD + 8;   // elements a row in LDS: 16-byte reads of 16 rows on distinct banks
    __shared__ __attribute__((aligned(16))) uint16_t rows[32 * RS];
    __shared__ f2_t rope[32 * 33];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h = blockIdx.y;
    const bool is_v = blockIdx.z == 1;
    const int tile = (a.p0 >> 5) + blockIdx.x, base = 32 * tile, slot = base % a.R;
    const int k_lo = max(a.p0 - base, 0), k_hi = min(a.p0 + a.T - base, 32);   // the tile's new rows
    const uint16_t* src = (is_v ? a.v : a.k) + h * HD + 2 * lane;
    uint32_t raw[TR];
#pragma unroll
    for (int i = 0; i < TR; i++) {   // (rows outside the chunk: a row of it, not stored)
        const int t = min(max(base + TR * w + i - a.p0, 0), a.T - 1);
        raw[i] = *(const uint32_t*)(src + (size_t)t * a.stride);
    }
    if (!is_v && a.kg) {   // bf16 rows with pre-ops
        const float g0 = 1.0f + bf2f(a.kg[2 * lane]), g1 = 1.0f + bf2f(a.kg[2 * lane + 1]);
        for (int idx = tid; idx < 32 * 32; idx += 64 * TW) {
            float c, s;
            rope_cs(base + (idx >> 5), kRopeFreq[idx & 31], c, s);
            rope[(idx >> 5) * 33 + (idx & 31)] = (f2_t){c, s};
        }
        __syncthreads();
        const int d0 = (2 * lane) & 31;
#pragma unroll
        for (int i = 0; i < TR; i++) {
            const f2_t p0 = rope[(TR * w + i) * 33 + d0], p1 = rope[(TR * w + i) * 33 + d0 + 1];
            raw[i] = norm_rope_pair(raw[i], g0, g1, RopePair{p0[0], p0[1], p1[0], p1[1]}, lane);
        }
    } else if (!is_v && a.norm_k) {   // bf16 rows of a full layer: RMS norm without gains
#pragma unroll
        for (int i = 0; i < TR; i++) {
            const float x0 = bf2f(raw[i] & 0xFFFF), x1 = bf2f(raw[i] >> 16), r = rms_factor(x0, x1);
            raw[i] = (uint32_t)f2bf(x0 * r) | ((uint32_t)f2bf(x1 * r) << 16);
        }
    }
#pragma unroll
    for (int i = 0; i < TR; i++) *(uint32_t*)&rows[(TR * w + i) * RS + 2 * lane] = raw[i];
    __syncthreads();
    uint16_t* out = (is_v ? a.vring : a.kring) + tile_base(h, a.R, slot, 2) / 2;
#pragma unroll
    for (int j = w; j < 8; j += TW) {
        const int l = lane;   // piece (j, l)
        if (!is_v) {
            const int k = 16 * (j >> 2) + (l & 15), d0 = 32 * (l >> 4) + 8 * (j & 3);
            if (k >= k_lo && k < k_hi) *(u4_t*)(out + (size_t)(64 * j + l) * 8) = ld16(&rows[k * RS + d0]);
        } else {
            // dim 8n + j of keys 16t + 4g + i, in order (t, i)
            const uint16_t* p = &rows[4 * (l >> 4) * RS + 8 * (l & 15) + j];
            uint16_t* o = out + (size_t)(64 * j + l) * 8;
            u4_t v;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint16_t* q = p + (16 * (e >> 1) + 2 * (e & 1)) * RS;
                v[e] = q[0] | ((uint32_t)q[RS] << 16);
            }
            if (k_lo == 0 && k_hi == 32) {
                *(u4_t*)o = v;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int k = 16 * (e >> 2) + 4 * (l >> 4) + (e & 3);
                    if (k >= k_lo && k < k_hi) o[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
                }
            }
        }
    }
}

int launch_ring_append(const RingAppendArgs& a, hipStream_t st) {
    if (a.T * a.n_kv > RING_TILE_ROWS && !(((uintptr_t)a.kring | (uintptr_t)a.vring) & 15)) {
        const dim3 grid((a.p0 + a.T - 1) / 32 - a.p0 / 32 + 1, a.n_kv, 2);
        hipLaunchKernelGGL(ring_append_tile_kernel, grid, dim3(64 * TW), 0, st, a);
    } else {
        hipLaunchKernelGGL(ring_append_kernel, dim3(a.T, a.n_kv), dim3(64), 0, st, a);
    }
    return hipGetLastError() == hipSuccess ? EMBLA_OK : EMBLA_ERR_HIP;
}

int launch_q_prep(const QPrepArgs& a, hipStream_t st) {
    // four rows a wave once that still gives every SIMD two waves, one for a decode step's few (2048
    // tokens of 16 heads: 9.4 us at 2 rows, 8.2 at 4, 9.0 at 8)
    const int n = a.T * a.n_q;
    if (n >= 8192) hipLaunchKernelGGL(q_prep_kernel<4>, dim3((n + 15) / 16), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(q_prep_kernel<1>, dim3((n + 3) / 4), dim3(256), 0, st, a);
    return hipGetLastError() == hipSuccess ? EMBLA_OK : EMBLA_ERR_HIP;
}

}  // namespace embla
