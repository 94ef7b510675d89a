// Batched ReLU² prefill over the reference's int8 cache (2 kv heads of 8 query heads, fp32 scales):
// p = relu(s / √128)², out = Σ p v / (√128 + Σ p), causal, optionally the last `window` positions
// (relu2_prefill_nax, Sources/EmblaMetal/Kernels/attn_nax.metal:61-364).
//
// MI355X design: a workgroup is 32 RB query rows (4 RB tokens x the kv head's 8 query heads) and its 8
// waves deal the 32-key blocks among themselves, each wave with its own O for all the rows: ReLU²
// weights need no running maximum, so the waves' sums add up at the end (through LDS) and the key
// loop has no barrier and no LDS tile. Keys are not split over workgroups (the reference's entry point
// takes no workspace; where one is given it is not used): splitting them over a workgroup's waves keeps
// every SIMD busy from few tokens on, where a workgroup of 32 tokens with all its waves on the same LDS tile left half the chip idle at
// 2048 tokens, and took a short chunk through the whole key range at one workgroup's pace.
// S^T = K·Q^T and O^T += V^T·P^T run on v_mfma_f32_32x32x16_f16 with query rows as columns; a
// wave's 16-byte loads of the int8 tiles are its operands: the k-slots of each product follow the
// tile's byte order (below), and the dims of an O^T row block follow V's.
//   K: fp16 subnormals (128 + k)·2^-24, one byte permute a pair; one more k-step adds
//      -128·2^-24·Σq (a constant of the row, as three fp16 parts), so a chain ends at 2^-24 q·k.
//   A step is KB blocks: with one row block, two blocks' independent score chains.
//   weights: with u = relu(2^-24 q·k)², a key's K scale enters as a = (2^24 scale/√128)², its V scale
//      with it as a·vscale: Σ += u a in fp32, and P = u a vscale enters the product as fp16; V itself
//      is widened exactly (biased V sums would cancel over a long context).
//   P's range: a weight is as small as its score and V's scale make it, and the sink keeps small ones
//      from being normalised away, so powers of two bring P into fp16's normal range whatever they
//      are: 2^n a query row, which puts its largest |q| in [2^12, 2^13) (then u <= 8²; the sink is
//      scaled with it), and 2^-e a wave, which keeps a·vscale <= 2^9 for the keys it has seen (raised
//      in steps when a key exceeds it, O with it; two instructions a block when none does). Without
//      them scores a tenth of unit size over V of 0.001 lost 3% of the result, over 0.0001 half.
#include "common.hpp"
#include "embla_internal.hpp"

namespace embla {

constexpr int R2_WAVES = 8;
constexpr int R2_GQ = 8;                    // query heads a kv head
constexpr int R2_TOK = 32 / R2_GQ;          // tokens a 32-row block
constexpr int R2_ROW = HD + 4;              // floats an O row in LDS

__device__ __forceinline__ f16_t mfma32h(h8_t a, h8_t b, f16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
/// 8 int8 (two dwords) as the fp16 subnormals (128 + x)·2^-24.
__device__ __forceinline__ h8_t i8x8_to_subnormal(uint32_t a, uint32_t b) {
    a ^= 0x80808080u;
    b ^= 0x80808080u;
    const u4_t r = {__builtin_amdgcn_perm(0u, a, 0x0c010c00u), __builtin_amdgcn_perm(0u, a, 0x0c030c02u),
                    __builtin_amdgcn_perm(0u, b, 0x0c010c00u), __builtin_amdgcn_perm(0u, b, 0x0c030c02u)};
    return __builtin_bit_cast(h8_t, r);
}

/// v of lane xor 32.
__device__ __forceinline__ float xchg_xor32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float((threadIdx.x & 32) ? r[0] : r[1]);
}

/// The larger of each half, unsigned.
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
    typedef uint16_t us2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2_t, a), __builtin_bit_cast(us2_t, b)));
}

template <int RB, int KB>
__global__ __launch_bounds__(64 * R2_WAVES, 1) void relu2_prefill_kernel(PrefillArgs a) {
    __shared__ __attribute__((aligned(16))) float red[R2_WAVES / 2][32][R2_ROW];
    __shared__ __attribute__((aligned(16))) h8_t qs[RB][9][64];
    __shared__ __attribute__((aligned(16))) float scl[R2_WAVES][KB][64];
    __shared__ float lred[R2_WAVES][32 * RB];
    __shared__ float sink[32 * RB];           // √128 in the row's scale
    constexpr int TOK = R2_TOK * RB;
    // consecutive workgroups: one kv head an XCD (n_kv divides the XCD count), the longest rows first
    const int kvh = blockIdx.x % a.n_kv, tb = gridDim.x / a.n_kv - 1 - blockIdx.x / a.n_kv;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int t0 = tb * TOK;
    const int last = a.p0 + min(t0 + TOK, a.T) - 1;               // the workgroup's last key
    const int lo_wg = a.window > 0 ? max(0, a.p0 + t0 - a.window + 1) : 0;   // its first key
    const int lo_all = a.window > 0 ? max(0, last - a.window + 1) : 0;       // every row sees keys from here
    const int b_first = lo_wg >> 5, nb = (last >> 5) - b_first + 1;          // its 32-key blocks

    const size_t nrow = (size_t)a.n_kv * a.max_s * HD;
    // lane l of a block's scale load: K's scale of key l % 32, then V's
    const float* sb = (const float*)((h ? a.vc : a.kc) + nrow) + (size_t)kvh * a.max_s + r;
    // K as the A operand: lane (key r, half h) loads the 16 dims 32j + 16h .. of key r for j < 4, the
    // k-slots of steps 2j and 2j + 1. V^T as the A operand, step s (keys 8s + 4h + i and 16 more):
    // lane (row r, half h) loads dims 8 (r % 16) + 4i + 2 (r / 16) and the next one, of row blocks
    // 2i and 2i + 1. Both loads cover whole 256-byte runs.
    const int8_t* kp = a.kc + tile_base(kvh, a.max_s, 0, 1) + (size_t)((2 * (r >> 4) + h) * 64 + (r & 15)) * 16;
    const int8_t* vp = a.vc + tile_base(kvh, a.max_s, 0, 1) + (size_t)((r >> 4) * 64 + (r & 15) + 16 * h) * 16;
    u4_t kr[KB][4], vr[KB][4];
    float scv[KB];
    const int nst = (nb + KB - 1) / KB;   // steps of KB blocks
    auto block_of = [&](int k, int i) { return b_first + min(KB * k + i, nb - 1); };
    auto load_k = [&](int k) {
#pragma unroll
        for (int i = 0; i < KB; i++) {
            const int b = block_of(k, i);
            scv[i] = sb[32 * b];
#pragma unroll
            for (int j = 0; j < 4; j++) kr[i][j] = ld16(kp + (size_t)b * 4096 + 256 * j);
        }
    };
    auto load_v = [&](int k) {
#pragma unroll
        for (int i = 0; i < KB; i++) {
            const int b = block_of(k, i);
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int e = 0; e < 2; e++) vr[i][2 * s + e] = ld16(vp + (size_t)b * 4096 + 2048 * e + 512 * s);
        }
    };

    // Q^T as the B operand, in K's k-slots: step 2j + e of half h holds dims 32j + 16h + 8e .. of row
    // r; in LDS in lane order (registers would leave no room for RB = 2's O), prepared by wave rb
    load_k(w);
    if (w < RB) {
        const int tok = min(t0 + R2_TOK * w + (r >> 3), a.T - 1), hq = kvh * R2_GQ + (r & 7);
        const uint16_t* qr = a.q + (size_t)tok * a.q_tok_stride + (size_t)hq * a.q_head_stride;
        u4_t raw[8];
        uint32_t mag = 0;   // the largest magnitude, as bf16 bits (past 0x7F80: a NaN)
#pragma unroll
        for (int s = 0; s < 8; s++) {
            raw[s] = ld16(qr + 32 * (s >> 1) + 16 * h + 8 * (s & 1));
#pragma unroll
            for (int i = 0; i < 4; i++) mag = pk_max_u16(mag, raw[s][i] & 0x7FFF7FFFu);
        }
        mag = max(mag & 0xFFFFu, mag >> 16);
        mag = max(mag, __float_as_uint(xchg_xor32(__uint_as_float(mag))));
        const int n = min(max(12 - ((int)(mag >> 7) - 127), -60), 60);
        const float up = __uint_as_float((uint32_t)(127 + n) << 23);   // 2^n
        // a row with an infinity (or past the range of n) has no finite output, one with a NaN no weight
        if (h == 0)
            sink[32 * w + r] = bf2f((uint16_t)mag) * up >= 65504.0f ? __uint_as_float(0x7FC00000u) : 11.313708498984761f * up * up;
        float sum = 0.0f;
        const h2_t ones = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
        for (int s = 0; s < 8; s++) {
            h2_t x[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                x[i] = (h2_t){(_Float16)(__uint_as_float(raw[s][i] << 16) * up), (_Float16)(__uint_as_float(raw[s][i] & 0xFFFF0000u) * up)};
                sum = __builtin_amdgcn_fdot2(x[i], ones, sum, false);
            }
            qs[w][s][lane] = *(const h8_t*)x;
        }
        // the bias step: -128·2^-24·Σq against A's 2^-12, as the sum of three fp16 parts
        const float v = sum_xor32(sum) * (-128.0f * 0x1p-12f);
        const _Float16 v0 = (_Float16)v, v1 = (_Float16)(v - (float)v0), v2 = (_Float16)(v - (float)v0 - (float)v1);
        h8_t bv = {};
        if (h == 0) { bv[0] = v0; bv[1] = v1; bv[2] = v2; }
        qs[w][8][lane] = bv;
    }
    const _Float16 one = (_Float16)0x1p-12f;
    const h8_t aone = {one, one, one, (_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f};
    f16_t O[RB][4];
    float lsum[RB];
    float lim = 0.0f, esc = 1.0f;   // uniform: the a·vscale that 2^-e allows for, and 2^-e
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        lsum[rb] = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) O[rb][i] = (f16_t){};
    }
    __syncthreads();

    for (int k = w; k < nst; k += R2_WAVES) {
        const int k0 = 32 * (b_first + KB * k);
        // loads complete in order: V's are issued behind K's and used a score chain later, the next
        // K's as soon as this step's are converted (the fences keep the compiler from moving them,
        // which made the wait for K one for V too)
        load_v(k);
        __builtin_amdgcn_sched_barrier(0);
        float kv[KB];
#pragma unroll
        for (int i = 0; i < KB; i++) {
            // lane l < 32: key l's a = (2^24 scale / √128)²; lane 32 + l: a times its V scale; both 0
            // outside the workgroup's keys, whose scales may never have been written
            const float sc = (uint32_t)(k0 + 32 * i - lo_wg + r) <= (uint32_t)(last - lo_wg) ? scv[i] : 0.0f;
            const float ks = sc * (0.08838834764831845f * 0x1p24f), k2 = ks * ks;
            const float o = xchg_xor32(k2);
            kv[i] = o * sc;   // (of use where h = 1)
            scl[w][i][lane] = h ? kv[i] * esc : k2;
        }
        f16_t s[KB][RB];
#pragma unroll
        for (int i = 0; i < KB; i++)
#pragma unroll
            for (int rb = 0; rb < RB; rb++) s[i][rb] = mfma32h(aone, qs[rb][8][lane], (f16_t){});
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int i = 0; i < KB; i++) {
                    const h8_t ka = i8x8_to_subnormal(kr[i][j][2 * e], kr[i][j][2 * e + 1]);
#pragma unroll
                    for (int rb = 0; rb < RB; rb++) s[i][rb] = mfma32h(ka, qs[rb][2 * j + e][lane], s[i][rb]);
                }
        __builtin_amdgcn_sched_barrier(0);
        load_k(k + R2_WAVES);
        __builtin_amdgcn_sched_barrier(0);
        float top = fabsf(kv[0]);
#pragma unroll
        for (int i = 1; i < KB; i++) top = fmaxf(top, fabsf(kv[i]));
        if (__ballot(top > lim) >> 32) {   // a key past what 2^-e allows for: e rises, O and the scales with it
            top = wave_bfly(h ? top : 0.0f, [](float x, float y) { return fmaxf(x, y); });
            const int ex = min(max((int)(__float_as_uint(top) >> 23) - 127, -100), 100) + 1;
            const float to = __uint_as_float((uint32_t)(127 + 9 - ex) << 23), f = to / esc;
            lim = __uint_as_float((uint32_t)(127 + ex) << 23);
            esc = to;
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int i = 0; i < 4; i++) O[rb][i] *= f;
            if (h)
#pragma unroll
                for (int i = 0; i < KB; i++) scl[w][i][lane] = kv[i] * esc;
        }
        wave_lds_sync();
        // item e = 4c + j of block i is key k0 + 32i + 8c + 4h + j
        if (k0 + 32 * KB - 1 > a.p0 + t0 || k0 < lo_all) {   // uniform: not every row sees every key
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                const int pos = a.p0 + min(t0 + R2_TOK * rb + (r >> 3), a.T - 1);
                const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
#pragma unroll
                for (int i = 0; i < KB; i++)
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const int key = k0 + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
                        s[i][rb][e] = key <= pos && key >= lo ? s[i][rb][e] : 0.0f;
                    }
            }
        }
        // P^T as the B operand: step st of half h holds keys 8st + 4h + j (items 4st ..) and
        // 16 + 8st + 4h + j (items 8 + 4st ..), as V's bytes have them
#pragma unroll
        for (int i = 0; i < KB; i++) {
            h8_t pb[RB][2];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const f4_t ka = *(const f4_t*)&scl[w][i][8 * c + 4 * h], kp = *(const f4_t*)&scl[w][i][32 + 8 * c + 4 * h];
#pragma unroll
                for (int rb = 0; rb < RB; rb++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float t = fmaxf(s[i][rb][4 * c + j], 0.0f), u = t * t;
                        lsum[rb] = __builtin_fmaf(u, ka[j], lsum[rb]);
                        pb[rb][c & 1][4 * (c >> 1) + j] = (_Float16)(u * kp[j]);
                    }
            }
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const h8_t va = i8x8_to_h8(vr[i][2 * st + j][2 * e], vr[i][2 * st + j][2 * e + 1]);
#pragma unroll
                        for (int rb = 0; rb < RB; rb++) O[rb][2 * j + e] = mfma32h(va, pb[rb][st], O[rb][2 * j + e]);
                    }
        }
        wave_lds_sync();   // the scales are read before the next step's replace them
    }

    // ---- the waves' sums, each times its 2^e: waves 4 .. 7 hand theirs to waves 0 .. 3, whose four are then added in the
    // output pass, a row block at a time. O^T row block i, item (b, e): row r' = 8b + 4h + e is dim
    // 8 (r' % 16) + 4 (i / 2) + 2 (r' / 16) + i % 2, so the lane holds the 8 dims of n = r' % 16 whole
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        const float l = sum_xor32(lsum[rb]);
        if (h == 0) lred[w][32 * rb + r] = l;
    }
    const float back = 1.0f / esc;
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        auto slot = [&](int b, int e, int half) -> f4_t* {
            return (f4_t*)&red[w & (R2_WAVES / 2 - 1)][r][8 * (8 * b + 4 * h + e) + 4 * half];
        };
        auto part = [&](int b, int e, int half) -> f4_t {
            const f16_t *x = &O[rb][2 * half], *y = &O[rb][2 * half + 1];
            return (f4_t){(*x)[4 * b + e], (*y)[4 * b + e], (*x)[8 + 4 * b + e], (*y)[8 + 4 * b + e]} * back;
        };
        if (rb > 0) __syncthreads();   // the previous row block's output pass has read the slots
        if (w >= R2_WAVES / 2) {
#pragma unroll
            for (int j = 0; j < 16; j++) *slot(j >> 3, (j >> 1) & 3, j & 1) = part(j >> 3, (j >> 1) & 3, j & 1);
        }
        __syncthreads();
        if (w < R2_WAVES / 2) {
#pragma unroll
            for (int j = 0; j < 16; j++) {
                f4_t* d = slot(j >> 3, (j >> 1) & 3, j & 1);
                *d = *d + part(j >> 3, (j >> 1) & 3, j & 1);
            }
        }
        __syncthreads();
        const int rr = tid >> 4, d0 = 8 * (tid & 15), ot = t0 + R2_TOK * rb + (rr >> 3);   // 8 dims a thread
        if (ot < a.T) {
            float den = sink[32 * rb + rr];
#pragma unroll
            for (int i = 0; i < R2_WAVES; i++) den += lred[i][32 * rb + rr];
            const float inv = 1.0f / den;
            u4_t out;
#pragma unroll
            for (int c = 0; c < 2; c++) {
                f4_t v = *(const f4_t*)&red[0][rr][d0 + 4 * c];
#pragma unroll
                for (int i = 1; i < R2_WAVES / 2; i++) v += *(const f4_t*)&red[i][rr][d0 + 4 * c];
                out[2 * c] = (uint32_t)f2bf(v[0] * inv) | ((uint32_t)f2bf(v[1] * inv) << 16);
                out[2 * c + 1] = (uint32_t)f2bf(v[2] * inv) | ((uint32_t)f2bf(v[3] * inv) << 16);
            }
            uint16_t* orow = a.o + (size_t)ot * a.o_tok_stride + (size_t)(kvh * R2_GQ + (rr & 7)) * a.o_head_stride + d0;
            if (((uintptr_t)orow & 15) == 0) {
                *(u4_t*)orow = out;
            } else {   // strides or a base that break 16-byte alignment
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    orow[2 * i] = (uint16_t)out[i];
                    orow[2 * i + 1] = (uint16_t)(out[i] >> 16);
                }
            }
        }
    }
}

int launch_relu2_prefill(const PrefillArgs& a, hipStream_t st) {
    if (a.n_q != R2_GQ * a.n_kv) return EMBLA_ERR_UNSUPPORTED;
    // A workgroup of two row blocks converts each K and V block once for both and takes about 1.6
    // times as long as one of one (30000 cached keys: 200 us against 126), a CU holds one workgroup,
    // so the time is rounds of 256 workgroups times that: 2048 tokens 518 us (665 with one row
    // block), 1024 262 (331), 700 210 (297), 193 (98 or 50 workgroups, one round) 126 with one row
    // block and 200 with two. The LDS-tiled kernel it replaces took 979 us at 2048 tokens and as
    // long for a few. What bounds it: issue. Two waves a SIMD each issue an instruction in 4-5
    // cycles at best, a block is ~200 VALU instructions and 17 MFMAs a row block (150 a row block
    // with two), and with the loads served by L1 the time stays the same.
    const int wg2 = (a.T + 2 * R2_TOK - 1) / (2 * R2_TOK) * a.n_kv, wg1 = (a.T + R2_TOK - 1) / R2_TOK * a.n_kv;
    constexpr int CUS = 256;
    if (3 * ((wg2 + CUS - 1) / CUS) <= 2 * ((wg1 + CUS - 1) / CUS))
        hipLaunchKernelGGL((relu2_prefill_kernel<2, 1>), dim3(wg2), dim3(64 * R2_WAVES), 0, st, a);
    else
        hipLaunchKernelGGL((relu2_prefill_kernel<1, 2>), dim3(wg1), dim3(64 * R2_WAVES), 0, st, a);
    return hipGetLastError() == hipSuccess ? EMBLA_OK : EMBLA_ERR_HIP;
}

}  // namespace embla
