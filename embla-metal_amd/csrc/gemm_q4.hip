// The 4-bit projections either side of attention at prefill: Y = X W^T for T tokens.
//
// Follows gemm.metal:1-134 (EXPERTS = 0, GATHER = 0): X [T][ldx] bf16, W in MLX's affine 4-bit
// layout (words [O][K/8], nibble q of word c the weight of column 8c + q; bf16 scales and biases
// [O][K/64], w = s * nibble + b), Y [T][ldy] through the epilogues EPI 0-4 (gemm.metal:118-131).
// The reference stages X and the dequantised W tile (one quantisation group, 64 inputs, a step)
// and multiplies 8x8 fragments into fp32 sums; MLX's own GEMM stages W as bf16, as here.
//
// MI355X design. A workgroup computes 16 MT tokens x 16 NT NW rows with 8 waves: NW row slices
// times KS shares of the inputs (NW KS = 8), each wave MT x NT tiles of v_mfma_f32_16x16x32_bf16
// (A: W rows, B: X rows, so a lane's 4 results are 4 neighbouring outputs of one token).
//  - W never passes LDS. A wave reads the words of its own rows two groups of 64 inputs at a time
//    (64 bytes a row, 16 a lane; loads of 8 or 2 bytes a lane cost the address unit as much and ran
//    a step twice as long), hands them over by v_permlane32_swap and dequantises them in registers
//    into the A operands: the nibbles exact in fp16 two at a time, s * q + b in fp32 (one
//    v_fma_mix_f32 each), rounded to bf16 by v_cvt_pk_bf16_f32. Scales and biases come from LDS
//    panels of 2048 inputs.
//  - X goes through LDS (three buffers, one barrier a step of one group a share) in 16-byte pieces
//    swizzled by the row: piece c of row r in slot c ^ (r & 15). Each wave reads its own share's.
//    Global loads go out two steps before their store (two register stages).
//  - At the end the KS shares of a tile meet in LDS, each wave adding up and storing its part of
//    the tiles.
// It replaces one 128 x 64 tile with the dequantised W in LDS, whose workgroups moved 281 bytes of
// LDS a cycle's worth of products (128 is the rate) and left most of the chip idle below 1000
// tokens. Measured (back to back in a graph), q/k/v (3072 rows, bf16 out) / o (2048 rows, += fp32) at
// K = 2048: 16 tokens 17.9 / 19.2 -> 5.9 / 5.7 us, 100 tokens 18.5 / 19.7 -> 9.9 / 9.6, 400 tokens
// 19.2 / 20.1 -> 18.3 / 13.7, 2048 tokens 44.2 / 33.3 -> 38.7 / 29.1; K = 4096, 2048 rows, 2048 tokens
// 56.0 -> 43.1 (bf16 out). At 2048 tokens the
// matrix cores are busy 29% of the time and LDS about 40%: the dequantisation's VALU work adds to the
// products (both waves of a SIMD are in the same part), and a workgroup starts and ends in 5 us.
#include <type_traits>
#include "common.hpp"
#include "embla_internal.hpp"

namespace embla {

typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));

/// Word w's 8 weights s * q + b, rounded to bf16. A nibble under the exponent of 1024 (or, 4 bits
/// up, 16 nibbles of 1024 + 16 q) is an fp16 value from which q comes exactly.
__device__ __forceinline__ b8_t dequant8(uint32_t w, float s, float b) {
    const h2_t k1024 = {(_Float16)1024.0f, (_Float16)1024.0f}, k64 = {(_Float16)64.0f, (_Float16)64.0f};
    const h2_t k16 = {(_Float16)0.0625f, (_Float16)0.0625f};
    h2_t q[4];                                   // q[j]: nibbles j and j + 4
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
        const uint32_t v = w >> (4 * j);
        q[j] = __builtin_bit_cast(h2_t, (v & 0x000F000Fu) | 0x64006400u) - k1024;
        q[j + 1] = __builtin_bit_cast(h2_t, (v & 0x00F000F0u) | 0x64006400u) * k16 - k64;
    }
    u4_t o;
#pragma unroll
    for (int e = 0; e < 4; e++) {                // weights 2 e and 2 e + 1
        const int j = 2 * (e & 1), h = e >> 1;
        const bf2_t p = {(__bf16)__builtin_fmaf((float)q[j][h], s, b), (__bf16)__builtin_fmaf((float)q[j + 1][h], s, b)};
        o[e] = __builtin_bit_cast(uint32_t, p);
    }
    return __builtin_bit_cast(b8_t, o);
}

template <int MT, int NT, int KS, bool GEN>
__global__ __launch_bounds__(512, MT * NT > 4 ? 2 : 4) void gemm_q4_kernel(GemmArgs a, int epi, int nblk, int per_xcd) {
    using Off = std::conditional_t<GEN, size_t, uint32_t>;
    constexpr int NW = 8 / KS;                   // row slices
    constexpr int QM = 16 * MT, QN = 16 * NT * NW;
    constexpr int CH = 8 * KS;                   // 16-byte pieces of X a row and step
    constexpr int NX = MT * KS / 4;              // pieces a thread stages
    constexpr int XB = QM * CH;                  // pieces a buffer
    constexpr int XCH = MT * NT * (KS - 1) * NW * 64;   // records of the final exchange
    constexpr int SP = 32 / KS, SROW = SP + 1;   // steps a panel of scales, its row (odd: 16 rows' banks differ)
    __shared__ u4_t sm[3 * XB > XCH ? 3 * XB : XCH];
    __shared__ uint32_t sc[2][KS * QN * SROW];   // [share][row][step]: bf16 scale, bias above it
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, r16 = lane & 15;
    const int ns = wv % NW, kh = wv / NW;
    // an XCD (workgroup id mod 8) takes a run of neighbouring tiles, so that its L2 serves the
    // rows of X and W that they share
    const int tile = per_xcd ? (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    const int m0 = tile / nblk * QM, nb = tile % nblk * QN, n0 = nb + ns * 16 * NT;
    const char* W = (const char*)a.W;
    const int G = a.K / 64, GS = ((G + KS - 1) / KS + 1) & ~1;   // groups; steps (a share's groups, even)

    // offsets from the tile's first row of X and the slice's first row of W (uniform addresses):
    // 32 bits, or 64 where rows are so long that a tile's pass 4 GB
    const char* X0 = (const char*)(a.X + (size_t)m0 * a.ldx);
    const int nr = min(n0, a.O - 1);
    const char* W0 = W + a.wo + (size_t)nr * G * 32;
    const int xc = tid % CH, xrow = tid / CH;    // piece i: row xrow + i 512 / CH, a multiple of 8 on
    const int xs = xrow * CH + (xc ^ (xrow & 15)), xg = xc / 8 * GS;   // its slot, its first group
    Off xo[NX], wo[NT];
#pragma unroll
    for (int i = 0; i < NX; i++)
        xo[i] = (Off)min(xrow + i * (512 / CH), a.T - 1 - m0) * (Off)a.ldx * 2 + 16 * (xc & 7);
#pragma unroll
    for (int t = 0; t < NT; t++) wo[t] = (Off)(min(n0 + 16 * t + r16, a.O - 1) - nr) * (Off)G * 32 + 16 * (g & 1);

    // Groups past the last are read as the last and enter as zeros (X, scales and biases).
    u4_t x0[NX], x1[NX], R0[NT], R1[NT];
    auto load_x = [&](int st, u4_t (&xr)[NX]) {
        const Off at = GEN ? (Off)min(xg + st, G - 1) * 128 : (Off)(xg + min(st, GS - 1)) * 128;
#pragma unroll
        for (int i = 0; i < NX; i++) xr[i] = ld16(X0 + (xo[i] + at));
    };
    auto mask_x = [&](int st, u4_t (&xr)[NX]) {
        if (GEN && xg + st >= G)
#pragma unroll
            for (int i = 0; i < NX; i++) xr[i] = (u4_t){};
    };
    auto store_x = [&](int buf, const u4_t (&xr)[NX]) {
#pragma unroll
        for (int i = 0; i < NX; i++) sm[buf * XB + (xs ^ (i * (512 / CH) & 8)) + i * 512] = xr[i];
    };
    auto load_w = [&](int st, u4_t (&R)[NT]) {   // steps st and st + 1: a row's 64 bytes over 4 lanes
        const Off at = (Off)min(kh * GS + st + (g >> 1), G - 1) * 32;
#pragma unroll
        for (int t = 0; t < NT; t++) R[t] = ld16(W0 + (wo[t] + at));
    };
    // lanes 0-31 hold step st's group and lanes 32-63 step st + 1's: afterwards words 0 and 1 are
    // every lane's of step st, 2 and 3 of step st + 1
    auto spread = [&](u4_t (&R)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const auto p = __builtin_amdgcn_permlane32_swap(R[t][j], R[t][j + 2], false, false);
                R[t][j] = p[0];
                R[t][j + 2] = p[1];
            }
    };
    // scales and biases of steps st .. st + SP - 1 for every share and row of the workgroup
    const bool svec = (((uintptr_t)W + a.so | (uintptr_t)W + a.bo) & 7) == 0 && G % 4 == 0 && GS % 4 == 0;
    auto fill = [&](int st) {
        uint32_t* d = sc[st / SP & 1];
        for (int i = tid; i < KS * QN * (SP / 4); i += 512) {
            const int c = 4 * (i % (SP / 4)), row = i / (SP / 4) % QN, sh = i / (SP / 4 * QN);
            const size_t at = (size_t)min(nb + row, a.O - 1) * G * 2;
            const int gr = sh * GS + st + c;
            uint32_t* o = d + (sh * QN + row) * SROW + c;
            if (svec) {
                u2_t s = {}, b = {};
                if (st + c < GS && gr < G) {
                    s = ld8(W + a.so + at + (size_t)gr * 2);
                    b = ld8(W + a.bo + at + (size_t)gr * 2);
                }
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    o[2 * e] = (s[e] & 0xFFFFu) | b[e] << 16;
                    o[2 * e + 1] = s[e] >> 16 | (b[e] & 0xFFFF0000u);
                }
            } else
                for (int e = 0; e < 4; e++) {
                    uint32_t v = 0;
                    if (st + c + e < GS && gr + e < G) {
                        v = *(const uint16_t*)(W + a.so + at + (size_t)(gr + e) * 2);
                        v |= (uint32_t)*(const uint16_t*)(W + a.bo + at + (size_t)(gr + e) * 2) << 16;
                    }
                    o[e] = v;
                }
        }
    };
    auto scales = [&](int st, uint32_t (&f)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; t++)
            f[t] = sc[st / SP & 1][(kh * QN + (ns * NT + t) * 16 + r16) * SROW + st % SP];
    };
    auto read_x = [&](int buf, int j, b8_t (&f)[MT]) {
        const int c = (8 * kh + 4 * (g & 1) + 2 * (g >> 1) + j) ^ r16;
#pragma unroll
        for (int i = 0; i < MT; i++) f[i] = __builtin_bit_cast(b8_t, sm[buf * XB + (r16 + 16 * i) * CH + c]);
    };
    auto dequant = [&](const u4_t (&R)[NT], int j, const uint32_t (&s)[NT], b8_t (&f)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; t++)
            f[t] = dequant8(R[t][j], __uint_as_float(s[t] << 16), __uint_as_float(s[t] & 0xFFFF0000u));
    };
    f4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[i][t] = (f4_t){};
    uint32_t s0[NT], s1[NT];
    b8_t fw0[NT], fw1[NT], fx0[MT], fx1[MT];
    auto mma = [&](const b8_t (&fw)[NT], const b8_t (&fx)[MT]) {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[i][t] = mfma16bf(fw[t], fx[i], acc[i][t]);
    };
    auto half = [&](const b8_t (&fw)[NT], const b8_t (&fx)[MT], auto reads, auto valu) {
        __builtin_amdgcn_sched_barrier(0);
        reads();
        mma(fw, fx);
#pragma unroll
        for (int i = 0; i < MT; i++) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, NT, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        valu();
        __builtin_amdgcn_sched_barrier(0);
    };
    // A step is two half steps of 32 inputs a share. While one's products run, the next one's X
    // operands are read and its weights dequantised; a step's buffer is complete a step before it
    // is read (three buffers, one barrier a step).
    auto step = [&](int st, int b0, int b1, int b2, const u4_t (&R)[NT], int j1, u4_t (&Rn)[NT], int jn,
                    uint32_t (&s)[NT], uint32_t (&sn)[NT], u4_t (&xr)[NX]) {
        scales(st + 1, sn);
        half(fw0, fx0, [&] { read_x(b0, 1, fx1); }, [&] { dequant(R, j1, s, fw1); });
        mask_x(st + 2, xr);
        store_x(b2, xr);
        load_x(st + 4, xr);
        if (jn == 0) spread(Rn);
        half(fw1, fx1, [&] { read_x(b1, 0, fx0); }, [&] { dequant(Rn, jn, sn, fw0); });
        __syncthreads();
    };
    load_w(0, R0);
    load_x(0, x0);
    load_x(1, x1);
    load_w(2, R1);
    fill(0);
    mask_x(0, x0);
    store_x(0, x0);
    load_x(2, x0);
    mask_x(1, x1);
    store_x(1, x1);
    load_x(3, x1);
    spread(R0);
    __syncthreads();
    scales(0, s0);
    dequant(R0, 0, s0, fw0);
    read_x(0, 0, fx0);
    int b0 = 0, b1 = 1, b2 = 2;
    auto pair = [&](int st, u4_t (&R)[NT], u4_t (&Rn)[NT]) {   // words of steps st, st + 1 and of the next two
        if (st % SP == 0 && st + SP < GS) fill(st + SP);
        step(st, b0, b1, b2, R, 1, R, 2, s0, s1, x0);
        step(st + 1, b1, b2, b0, R, 3, Rn, 0, s1, s0, x1);
        load_w(st + 4, R);
        const int t = b0;
        b0 = b2;
        b2 = b1;
        b1 = t;
    };
    for (int st = 0; st < GS; st += 4) {
        pair(st, R0, R1);
        if (st + 2 < GS) pair(st + 2, R1, R0);
    }
    __syncthreads();

    // tile u = i NT + t of a row slice is finished by the wave of share u % KS, which the others
    // hand theirs: record ((u (KS - 1) + r) NW + ns) 64 + lane, r the sender's distance less one
#pragma unroll
    for (int u = 0; u < MT * NT; u++) {
        const int r = (kh - u % KS + KS - 1) % KS;
        if (r < KS - 1) sm[((u * (KS - 1) + r) * NW + ns) * 64 + lane] = __builtin_bit_cast(u4_t, acc[u / NT][u % NT]);
    }
    __syncthreads();
    const bool f32 = epi >= 2;
    const bool vec = a.ldy % 4 == 0 && (uintptr_t)a.Y % (f32 ? 16 : 8) == 0;
#pragma unroll
    for (int u = 0; u < MT * NT; u++) {
        if (u % KS != kh) continue;
        f4_t v = acc[u / NT][u % NT];
#pragma unroll
        for (int r = 0; r < KS - 1; r++) v += __builtin_bit_cast(f4_t, sm[((u * (KS - 1) + r) * NW + ns) * 64 + lane]);
        const int m = m0 + 16 * (u / NT) + r16, n = n0 + 16 * (u % NT) + 4 * g;
        if (m >= a.T || n >= a.O) continue;
        const size_t at = (size_t)m * a.ldy + n;
        if (f32) {
            float* y = (float*)a.Y + at;
            const bool whole = vec && n + 4 <= a.O;
            if (epi < 4)
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = bf2f(f2bf(v[e]));
            if (whole) {
                if (epi == 2) v += *(const f4_t*)y;
                *(f4_t*)y = v;
            } else
                for (int e = 0; e < 4 && n + e < a.O; e++) y[e] = epi == 2 ? y[e] + v[e] : v[e];
        } else {
            uint16_t* y = (uint16_t*)a.Y + at;
            uint16_t o[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o[e] = f2bf(v[e]);
                if (epi == 1) {
                    const float t = fmaxf(bf2f(o[e]), 0.0f);
                    o[e] = f2bf(t * t);
                }
            }
            if (vec && n + 4 <= a.O) *(u2_t*)y = (u2_t){o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16};
            else
                for (int e = 0; e < 4 && n + e < a.O; e++) y[e] = o[e];
        }
    }
}

template <int MT, int NT, int KS, bool GEN = false>
int launch_gemm_q4_tile(const GemmArgs& a, int epi, hipStream_t st) {
    constexpr int QM = 16 * MT, QN = 16 * NT * (8 / KS);
    const int nblk = (int)(((long long)a.O + QN - 1) / QN);
    const long long tiles = nblk * (((long long)a.T + QM - 1) / QM);
    hipLaunchKernelGGL((gemm_q4_kernel<MT, NT, KS, GEN>), dim3((unsigned)tiles), dim3(512), 0, st, a, epi, nblk,
                       tiles % 8 ? 0 : (int)(tiles / 8));
    return hipGetLastError() == hipSuccess ? EMBLA_OK : EMBLA_ERR_HIP;
}

// The tile is the one of least modelled time: first + round * ceil(workgroups / 256), in tenths of a
// us at K = 2048 (other K scale all alike), fitted to a sweep of 6 .. 2048 tokens at 2048 and 3072
// rows, K = 2048 and 4096 (two of the smallest fit a CU, so that its rounds overlap). It leaves out how
// full the last round is, up to a fifth of a round of the large tiles (256 workgroups of 128 x 192:
// 37.8 us, 131 of them 31): over 1 .. 2048 tokens, 520 .. 3072 rows and K = 1024 .. 4096 the tile chosen
// takes 0.1% more than the fastest of them on average, 6% at most. The last two take what the others'
// equal shares and 32-bit offsets do not: the general instance of this kernel (3072 rows, K = 2112, 40
// tokens: 11.0 us) and the kernel with the weights in LDS (18.4), which is faster from two rounds of the
// first on (600 tokens 20.2 against 33.1).
// Below K = 1024 the starts and ends that the model scales with K decide: the kernel with the weights in
// LDS, which has the shortest, takes all but one round of the smaller tiles, from K = short_k (3072 rows,
// K = 512, 600 tokens: 128 x 64 in registers 9.7 us, in LDS 8.5; K = 192, 16 tokens: the general instance
// 6.0, in LDS 5.2; K = 512, 16 tokens: 64 x 32 6.4, in LDS 7.4): within 0.2% of the fastest on average.
struct GemmTile { int m, n, ks, first, round, short_k; int (*launch)(const GemmArgs&, int, hipStream_t); };
static const GemmTile GEMM_TILES[] = {
    {16, 16, 8, 25, 25, 1024, launch_gemm_q4_tile<1, 1, 8>},    {32, 16, 8, 0, 58, 1024, launch_gemm_q4_tile<2, 1, 8>},
    {64, 32, 4, 0, 83, 512, launch_gemm_q4_tile<4, 1, 4>},    {64, 64, 4, 0, 114, 1024, launch_gemm_q4_tile<4, 2, 4>},
    {128, 64, 2, 0, 158, 1024, launch_gemm_q4_tile<8, 1, 2>},  {128, 128, 2, 0, 205, 1024, launch_gemm_q4_tile<8, 2, 2>},
    {128, 192, 2, 0, 304, 1024, launch_gemm_q4_tile<8, 3, 2>},
    {64, 32, 0, 0, 100, 320, launch_gemm_q4_tile<4, 1, 4, true>}, {128, 64, 0, 50, 130, 0, launch_gemm_q4_lds},
};

int launch_gemm_q4(const GemmArgs& a, int epi, hipStream_t st) {
    const bool narrow = a.ldx <= 1 << 23 && a.K <= 1 << 23;
    const GemmTile* best = nullptr;
    long long least = 0;
    for (const GemmTile& t : GEMM_TILES) {
        if (t.ks && (!narrow || a.K / 64 % (2 * t.ks))) continue;
        const long long tiles = (((long long)a.T + t.m - 1) / t.m) * (((long long)a.O + t.n - 1) / t.n);
        if (a.K < t.short_k || (a.K < 1024 && t.short_k && tiles > 256)) continue;
        const long long cost = t.first + (tiles + 255) / 256 * t.round;
        if (tiles <= 0x7FFFFFFFLL && (!best || cost < least)) best = &t, least = cost;
    }
    return best ? best->launch(a, epi, st) : EMBLA_ERR_INVALID;
}

}  // namespace embla
