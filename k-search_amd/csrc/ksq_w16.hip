// ksq_w16.hip - the dequantise-then-fp32 GEMM (W4A16 / W8A16: fp32 activations, Q4_0 / Q8_0
// weights, no activation quantisation) on the gfx950 bf16 MFMA.
//
// Reference path: gemm_w4a16_naive / gemm_w4a16_tiled / gemm_w8a16_naive
// (include/gemm_cuda_naive.cuh:66-150, launchers :267-283; include/gemm_cuda_tiled.cuh:108-190,
// launcher :284-291), CPU references gemm_w4a16_reference / gemm_w8a16_reference
// (include/gemm_reference.h:73-147) and the harness oracle reference_q4_0_fp32_gemm
// (llm_kernel_test/reference/gemm_ref.py:51-97): C[m][n] = sum_k A[m][k] * d_w * q_w[n][k] in
// fp32, with q_w = q - 8 for Q4_0 and the signed quant for Q8_0.
//
// gfx950 design:
//  * Exact products on the bf16 MFMA.  Each fp32 activation is split into three bf16 terms
//    a = hi + mid + lo (hi = bf16(a), mid = bf16(a - hi), lo = bf16(a - hi - mid)): both
//    differences are exact in fp32 and the three terms carry all 24 significant bits (finite
//    |a| below the largest bf16).  The weight quants (q - 8 for Q4_0, q for Q8_0) are integers
//    of at most 8 bits, exact in bf16.  So every product of v_mfma_f32_32x32x16_bf16 is exact
//    and only the fp32 sums round, as in the reference's fp32 loop (in another order).  The
//    terms go in smallest first: lo, mid, hi.  (Above 32 rows Q4_0 is staged as (q - 8) / 16, which
//    v_cvt_off_f32_i4 gives in one operation, with the scale 16 d: powers of two, exact.)
//  * Per 32-element block, six MFMAs (three terms x two 16-element halves) give the block's partial
//    sum P = sum_k a_k q_k for a 32 x 32 patch, then acc = fma(d_w, P, acc): one VALU op per output
//    and block (the reference multiplies d_w into every weight element instead; the same value up
//    to rounding).
//  * The activations are split and the weight quants converted once per workgroup and block, into
//    LDS in fragment order: a wave's 16-byte reads are lane-linear, without bank conflicts.  Two
//    buffers: block k + 1 is converted between the MFMAs of block k, one barrier per block.
//  * Tiles of 128 x 256 (eight waves of 64 x 64), 128 x 128 (four) and 64 x 128 (four of 32 x 64),
//    chosen with the number of K splits by a cost model over the grid (w16_plan); the split partial
//    sums are added in split order by the int8 GEMM's split-K reduction (deterministic).
//  * Bound: the chip's power.  Six MFMAs take 198 cycles per patch and block, and at full rate with
//    random operands the clock falls from 2.4 to about 2 GHz; every instruction beside them costs
//    time.  M = 2048, N = K = 4096, Q4_0: 183 us (375 TFLOP/s of fp32-exact products, 1.13 PFLOP/s
//    on the bf16 pipe), of it 138 the MFMAs with their LDS reads alone, 12 the epilogue and about
//    35 the conversions (230 us on single-buffered 128 x 128 tiles with 144-byte row pitch and two
//    barriers per two blocks); Q8_0, whose weights are twice the bytes to convert, 197 (224).  M =
//    395, N = 3871, K = 1344: Q4_0 25.4 us (65.5), Q8_0 23.7 (64.2).
//  * Measured, level or slower: three buffers with the next block's first fragments read ahead of
//    the barrier, and activation loads four blocks ahead (187-195 us).
//  * Rows / columns past M or N load a clamped in-range row and are not stored.
#include "ksq_device.h"
#include "ksq_internal.h"

namespace ksq {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// BM x BN workgroup tile, waves of 32 TM x 32 TN.  Two threads per weight row stage the weights.
template <int BM_, int BN_, int TM_, int TN_>
struct W16Tile {
    static constexpr int BM = BM_, BN = BN_, TM = TM_, TN = TN_;
    static constexpr int WN = BN / (32 * TN);   // waves along N
    static constexpr int WM = BM / (32 * TM);   // waves along M
    static constexpr int NT = 64 * WN * WM;     // threads per workgroup
    static constexpr int AC = BM * 4 / NT;      // 8-float activation chunks per thread and block
    static_assert(BM * 4 % NT == 0, "every thread stages whole activation chunks");
    static_assert(NT == 2 * BN, "a thread stages half a weight block per row");
};
using W16Huge = W16Tile<128, 256, 2, 2>;
using W16Big = W16Tile<128, 128, 2, 2>;
using W16Mid = W16Tile<64, 128, 1, 2>;

typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3a4 __attribute__((ext_vector_type(3), aligned(4)));

template <int V>
struct W16Int {
    static constexpr int value = V;
};

// Two fp32 values as a bf16 pair (round to nearest even), lo in the low half: one packed
// conversion (v_cvt_pk_bf16_f32) instead of two single ones and the shift and or that merge them.
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2v{lo, hi}, bf16x2));
}
__device__ __forceinline__ float bf16_low_f32(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float bf16_high_f32(uint32_t p) { return __builtin_bit_cast(float, p & 0xFFFF0000u); }

// The four nibbles at bits 0, 8, 16, 24 of w, less 8, as two bf16 pairs.
__device__ __forceinline__ u32x2 w16_nibbles(uint32_t w) {
    float q[4];
#pragma unroll
    for (int b = 0; b < 4; b++) q[b] = __builtin_amdgcn_cvt_off_f32_i4((int)(w >> (8 * b)));
    return u32x2{bf16_pair(q[0], q[1]), bf16_pair(q[2], q[3])};
}
__device__ __forceinline__ u32x2 w16_bytes(uint32_t w) {
    float q[4];
#pragma unroll
    for (int b = 0; b < 4; b++) q[b] = (float)(int8_t)((w >> (8 * b)) & 0xFFu);
    return u32x2{bf16_pair(q[0], q[1]), bf16_pair(q[2], q[3])};
}

// WT: kWQ40 or kWQ80.  W: [N][K/32] blocks (4-byte aligned); A: fp32 [M][K] (16-byte aligned);
// C: fp32 [M][N], or split z's partial [M][N] at C + z*M*N.  nb = K/32, even.
// Workgroup x is a linear tile index whose tiles each XCD takes as one contiguous run in
// row-major tile order (xcd_tile): whole rows of tiles per XCD, so each XCD's L2 fetches its
// activation rows once (the plain grid spreads each row's column tiles over all 8 XCDs).
template <class T, int WT>
__global__ __launch_bounds__(T::NT, 2) void w16_kernel(const uint8_t* __restrict__ W, const float* __restrict__ A,
                                                       float* __restrict__ C, int M, int N, int nb) {
    constexpr int BM = T::BM, BN = T::BN, TM = T::TM, TN = T::TN, NT = T::NT, AC = T::AC;
    constexpr int BB = block_bytes(WT);                    // 18 or 34
    constexpr int WW = (WT == kWQ40) ? 6 : 10;             // weight dwords a thread loads per two blocks
    // fragment order: [32-row group][term: lo, mid, hi][16-element half][lane][8 bf16]
    constexpr int ABytes = BM * 32 * 2 * 3, WBytes = BN * 32 * 2;
    // two buffers: block k + 1 is staged while block k is multiplied
    constexpr int DBytes = 2 * BN * 4, Buf = ABytes + WBytes + DBytes;
    __shared__ __attribute__((aligned(16))) uint8_t sm[2 * Buf];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave / T::WN, wn = wave % T::WN;
    const int l32 = lane & 31, hi = lane >> 5;
    const int gn = (N + BN - 1) / BN, tiles = gn * ((M + BM - 1) / BM);
    const int L = xcd_tile((int)blockIdx.x, (int)gridDim.x);
    if (L >= tiles) return;   // padding of the grid to a multiple of 8 (whole workgroup)
    const int m0 = (L / gn) * BM, n0 = (L % gn) * BN;

    // split z covers K steps [s_lo, s_hi) of two blocks each
    const int nsteps = nb / 2, Z = (int)gridDim.z, z = (int)blockIdx.z;
    const int s_lo = (int)((long long)nsteps * z / Z), s_hi = (int)((long long)nsteps * (z + 1) / Z);
    C += (size_t)z * (size_t)M * (size_t)N;
    const size_t K = (size_t)nb * 32;

    // ---- staging assignment ----
    // activations: chunk c = t + NT i is the 8 floats at 8 (c % 4) of row c / 4 (four lanes read a
    // row's 128-byte segment); weights: row t % BN, half t / BN (wave-uniform) of its blocks
    const float* asrc[AC];
    uint32_t adst[AC];
#pragma unroll
    for (int i = 0; i < AC; i++) {
        const int c = t + NT * i, r = c >> 2, q = c & 3;
        asrc[i] = A + (size_t)min(m0 + r, M - 1) * K + 8 * q;
        // rows of a fragment are XORed with twice the chunk number: the 8 lanes of a write (2 rows
        // x 4 chunks, whose fragments lie multiples of 512 bytes apart) then hit 8 bank groups
        adst[i] = (uint32_t)((r >> 5) * 6144 + (q >> 1) * 1024 + (q & 1) * 512 + (((r & 31) ^ (2 * q)) << 4));
    }
    const int wr = t % BN, wh = t / BN;
    const uint8_t* wrow = W + (size_t)min(n0 + wr, N - 1) * nb * BB;
    f32x4 pa[2][AC][2];        // blocks k + 1 and k + 2 while block k is multiplied
    uint32_t pw[WW];           // the weights of two blocks
    auto load_a = [&](auto bv, int kb) __attribute__((always_inline)) {
        constexpr int b = decltype(bv)::value;
#pragma unroll
        for (int i = 0; i < AC; i++) {
            pa[b][i][0] = *(const f32x4*)(asrc[i] + (size_t)kb * 32);
            pa[b][i][1] = *(const f32x4*)(asrc[i] + (size_t)kb * 32 + 4);
        }
    };
    // the weight bytes of step s (two blocks) that this thread converts.  Q4_0 (36 bytes: d at 0
    // and 18, quants at 2 and 20): half h is quant bytes 8h .. 8h + 7, i.e. dwords 2h .. 2h + 2 and
    // 4 + 2h .. 6 + 2h.  Q8_0 (68 bytes: d at 0 and 34, quants at 2 and 36): half h is bytes
    // 16h .. 16h + 15, i.e. dwords 4h .. 4h + 4 and 8 + 4h .. 12 + 4h.
    auto load_w = [&](int s) __attribute__((always_inline)) {
        const uint32_t* src = (const uint32_t*)(wrow + (size_t)s * 2 * BB);
        if constexpr (WT == kWQ40) {
            const u32x3a4 x = *(const u32x3a4*)(src + 2 * wh), y = *(const u32x3a4*)(src + 4 + 2 * wh);
            pw[0] = x.x; pw[1] = x.y; pw[2] = x.z;
            pw[3] = y.x; pw[4] = y.y; pw[5] = y.z;
        } else {
            const u32x4a4 x = *(const u32x4a4*)(src + 4 * wh), y = *(const u32x4a4*)(src + 9 + 4 * wh);
            pw[0] = x.x; pw[1] = x.y; pw[2] = x.z; pw[3] = x.w; pw[4] = src[4 * wh + 4];
            pw[5] = src[8 + 4 * wh];
            pw[6] = y.x; pw[7] = y.y; pw[8] = y.z; pw[9] = y.w;
        }
    };
    // chunk i of the activation block in pa[b], as three bf16 terms, into buffer b
    auto store_a = [&](auto bv, int i, uint8_t* buf) __attribute__((always_inline)) {
        constexpr int b = decltype(bv)::value;
        uint32_t ph[4], pm[4], pl[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float a0 = pa[b][i][j >> 1][2 * (j & 1)], a1 = pa[b][i][j >> 1][2 * (j & 1) + 1];
            ph[j] = bf16_pair(a0, a1);
            const float r0 = a0 - bf16_low_f32(ph[j]), r1 = a1 - bf16_high_f32(ph[j]);
            pm[j] = bf16_pair(r0, r1);
            pl[j] = bf16_pair(r0 - bf16_low_f32(pm[j]), r1 - bf16_high_f32(pm[j]));
        }
        uint8_t* d = buf + adst[i];
        *(u32x4*)d = u32x4{pl[0], pl[1], pl[2], pl[3]};
        *(u32x4*)(d + 2048) = u32x4{pm[0], pm[1], pm[2], pm[3]};
        *(u32x4*)(d + 4096) = u32x4{ph[0], ph[1], ph[2], ph[3]};
    };
    // block b of the step in pw into weight buffer b
    auto store_w = [&](auto bv, uint8_t* buf) __attribute__((always_inline)) {
        constexpr int b = decltype(bv)::value;
        uint8_t* d = buf + ABytes + (wr >> 5) * 2048 + ((wr & 31) << 4);
        float* sd = (float*)(buf + ABytes + WBytes);   // the second BN: from the half that holds no scale, never read
        if constexpr (WT == kWQ40) {
            const uint32_t q0 = b ? pw[4] : word_at(pw, 2), q1 = b ? pw[5] : word_at(pw, 6);
            const uint32_t x0 = q0 ^ 0x88888888u, x1 = q1 ^ 0x88888888u;
            const u32x2 l0 = w16_nibbles(x0), l1 = w16_nibbles(x1);
            const u32x2 h0 = w16_nibbles(x0 >> 4), h1 = w16_nibbles(x1 >> 4);
            *(u32x4*)(d + 512 * wh) = u32x4{l0.x, l0.y, l1.x, l1.y};          // elements 8h ..
            *(u32x4*)(d + 1024 + 512 * wh) = u32x4{h0.x, h0.y, h1.x, h1.y};   // elements 16 + 8h ..
            sd[t] = 16.0f * f16_to_f32(b ? pw[3] >> 16 : pw[0] & 0xFFFFu);
        } else {
            u32x2 v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = w16_bytes(b ? pw[6 + j] : word_at(pw, 2 + 4 * j));
            *(u32x4*)(d + 1024 * wh) = u32x4{v[0].x, v[0].y, v[1].x, v[1].y};        // elements 16h ..
            *(u32x4*)(d + 1024 * wh + 512) = u32x4{v[2].x, v[2].y, v[3].x, v[3].y};  // 16h + 8 ..
            sd[t] = f16_to_f32(b ? pw[5] >> 16 : pw[0] & 0xFFFFu);
        }
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
    f32x16 zero;
#pragma unroll
    for (int r = 0; r < 16; r++) zero[r] = 0.0f;
    // byte offset of this lane's slot in half h of a fragment (chunk q = 2h + hi)
    uint32_t aoff[2];
#pragma unroll
    for (int h = 0; h < 2; h++)
        aoff[h] = (uint32_t)(wm * TM * 6144 + h * 1024 + hi * 512 + ((l32 ^ (2 * (2 * h + hi))) << 4));
    const uint32_t woff = (uint32_t)(wn * TN * 2048 + lane * 16);

    // Block b (buffer b) times its weights, with the staging of the next block (`stage`) in the same
    // straight-line code: the scheduling groups put its conversions between the MFMAs
    auto compute = [&](const uint8_t* buf, auto stage) __attribute__((always_inline)) {
        bf16x8 wf[TN][2], af[TM][3][2];
        float dw[TN];
#pragma unroll
        for (int j = 0; j < TN; j++) {
#pragma unroll
            for (int h = 0; h < 2; h++) wf[j][h] = *(const bf16x8*)(buf + ABytes + woff + j * 2048 + h * 1024);
            dw[j] = *(const float*)(buf + ABytes + WBytes + 4 * (wn * 32 * TN + 32 * j + l32));
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int e = 0; e < 3; e++)
#pragma unroll
                for (int h = 0; h < 2; h++) af[i][e][h] = *(const bf16x8*)(buf + aoff[h] + i * 6144 + e * 2048);
        stage();
        f32x16 p[2];
#pragma unroll
        for (int u = 0; u <= TM * TN; u++) {
            if (u < TM * TN) {
                const int i = u / TN, j = u % TN;
                // D[m][n]: A operand = activation fragment, B = weights, so a lane holds one column
                f32x16 c = zero;
#pragma unroll
                for (int e = 0; e < 3; e++)
#pragma unroll
                    for (int h = 0; h < 2; h++) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i][e][h], wf[j][h], c, 0, 0, 0);
                p[u & 1] = c;
            }
            if (u > 0) {
                const int i = (u - 1) / TN, j = (u - 1) % TN;
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = fmaf(dw[j], p[(u - 1) & 1][r], acc[i][j][r]);
            }
        }
        constexpr int NM = TM * TN * 6;   // MFMAs; per MFMA: a fragment read, 7 vector instructions, an LDS write
        __builtin_amdgcn_sched_group_barrier(0x100, TN * 3 + 6, 0);
#pragma unroll
        for (int k = 0; k < NM; k++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (k < 6 * (TM - 1)) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
            if (k > NM / 3) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
    };

    using B0 = W16Int<0>;
    using B1 = W16Int<1>;
    uint8_t* const buf0 = sm;
    uint8_t* const buf1 = sm + Buf;
    if (s_lo < s_hi) {
        load_w(s_lo);
        load_a(B0{}, 2 * s_lo);
        load_a(B1{}, 2 * s_lo + 1);
        store_w(B0{}, buf0);
#pragma unroll
        for (int i = 0; i < AC; i++) store_a(B0{}, i, buf0);
    }
    __syncthreads();
    for (int s = s_lo; s < s_hi; s++) {
        const int sn = min(s + 1, s_hi - 1);   // past the last step: staged again, read by nobody
        load_a(B0{}, 2 * sn);
        __builtin_amdgcn_sched_barrier(0);   // the loads go out before the block is computed
        compute(buf0, [&]() __attribute__((always_inline)) {
            store_w(B1{}, buf1);
#pragma unroll
            for (int i = 0; i < AC; i++) store_a(B1{}, i, buf1);
        });
        load_w(sn);
        __syncthreads();
        load_a(B1{}, 2 * sn + 1);
        __builtin_amdgcn_sched_barrier(0);   // the loads go out before the block is computed
        compute(buf1, [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < AC; i++) store_a(B0{}, i, buf0);
            store_w(B0{}, buf0);
        });
        __syncthreads();
    }

    // lane l holds column n = l % 32 of each 32 x 32 patch, rows m = 8 (r / 4) + 4 (l / 32) + r % 4
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int mb = m0 + (wm * TM + i) * 32 + 4 * hi;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = n0 + (wn * TN + j) * 32 + l32;
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = mb + 8 * (r >> 2) + (r & 3);
                if (m < M) C[(size_t)m * N + n] = acc[i][j][r];
            }
        }
    }
}

// ---- up to 32 activation rows ----------------------------------------------------------------
// A 32 x 128 tile, four waves side by side, one LDS buffer of two blocks and the next step's loads
// in registers.  Bound by the latency of a step, not by the matrix pipe; split along K the plain
// form is level with or ahead of the double-buffered one (N = K = 4096, M = 8: Q4_0 12.8 vs 13.2
// us, Q8_0 12.7 vs 14.0; N = 1632, K = 5440, M = 20: 12.6 vs 13.4).
constexpr int kW16SmallRows = 32;
constexpr int kW16Pitch = 72;         // bf16 per staged row: 64 values of the step + 8 padding

// 32 weight quants of one block as bf16 into dst (32 values), the block's scale into *d.  v: the
// dwords holding the block, which starts at byte O of v.
template <int WT, int O>
__device__ __forceinline__ void w16_stage_block(const uint32_t* v, uint16_t* dst, float* d) {
    *d = f16_to_f32(half_at(v, O));
    if constexpr (WT == kWQ40) {
        // element e < 16: low nibble of qs[e]; e >= 16: high nibble of qs[e - 16]; value q - 8
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t w = word_at(v, O + 2 + 4 * i);
            float lo[4], hi[4];
#pragma unroll
            for (int b = 0; b < 4; b++) {
                lo[b] = (float)((w >> (8 * b)) & 0x0Fu) - 8.0f;
                hi[b] = (float)((w >> (8 * b + 4)) & 0x0Fu) - 8.0f;
            }
            *(u32x2*)(dst + 4 * i) = u32x2{bf16_pair(lo[0], lo[1]), bf16_pair(lo[2], lo[3])};
            *(u32x2*)(dst + 16 + 4 * i) = u32x2{bf16_pair(hi[0], hi[1]), bf16_pair(hi[2], hi[3])};
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t w = word_at(v, O + 2 + 4 * i);
            float q[4];
#pragma unroll
            for (int b = 0; b < 4; b++) q[b] = (float)(int8_t)((w >> (8 * b)) & 0xFFu);
            *(u32x2*)(dst + 4 * i) = u32x2{bf16_pair(q[0], q[1]), bf16_pair(q[2], q[3])};
        }
    }
}

// W, A, C and nb as above; grid (column tiles, row tiles, splits).
template <int WT>
__global__ __launch_bounds__(256, 2) void w16_small_kernel(const uint8_t* __restrict__ W, const float* __restrict__ A,
                                                     float* __restrict__ C, int M, int N, int nb) {
    constexpr int BM = kW16SmallRows, BN = 128, P = kW16Pitch;
    constexpr int BB = block_bytes(WT);                    // 18 or 34
    constexpr int AC = BM * 16 / 256;                      // activation float4 chunks per thread
    constexpr int WW = (WT == kWQ40) ? 5 : 9;              // weight dwords a thread loads per step
    __shared__ __attribute__((aligned(16))) uint16_t sA[3][BM][P];     // lo, mid, hi planes
    __shared__ __attribute__((aligned(16))) uint16_t sW[BN][P];
    __shared__ __attribute__((aligned(16))) float sD[2][BN];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int l32 = lane & 31, hi = lane >> 5;
    const int m0 = (int)blockIdx.y * BM, n0 = (int)blockIdx.x * BN;

    // split z covers K steps [s_lo, s_hi) of two blocks each
    const int nsteps = nb / 2, Z = (int)gridDim.z, z = (int)blockIdx.z;
    const int s_lo = (int)((long long)nsteps * z / Z), s_hi = (int)((long long)nsteps * (z + 1) / Z);
    C += (size_t)z * (size_t)M * (size_t)N;
    const size_t K = (size_t)nb * 32;

    // staging assignment: activation chunk c = t + 256 i is row c / 16, float4 c % 16 of the
    // step's 64 floats (16 lanes read 256 contiguous bytes of a row); weight row t % 128,
    // block t / 128 of the step (wave-uniform)
    const int wr = t % BN, wb = t / BN;
    const uint8_t* wrow = W + (size_t)min(n0 + wr, N - 1) * nb * BB;
    f32x4 pa[AC];
    uint32_t pw[WW];
    auto load = [&](int s) {
#pragma unroll
        for (int i = 0; i < AC; i++) {
            const int c = t + 256 * i, r = c >> 4, q = c & 15;
            pa[i] = *(const f32x4*)(A + (size_t)min(m0 + r, M - 1) * K + (size_t)s * 64 + 4 * q);
        }
        // Q4_0: the step's 36 bytes are dwords 0..8 and block wb starts at byte 18 wb, so dwords
        // 4 wb .. 4 wb + 4 hold it from byte 2 wb on; Q8_0: 68 bytes, block wb at byte 34 wb,
        // dwords 8 wb .. 8 wb + 8, from byte 2 wb on
        const uint32_t* src = (const uint32_t*)(wrow + (size_t)s * 2 * BB) + (WT == kWQ40 ? 4 : 8) * wb;
#pragma unroll
        for (int i = 0; i < WW; i++) pw[i] = src[i];
    };
    auto store = [&]() {
#pragma unroll
        for (int i = 0; i < AC; i++) {
            const int c = t + 256 * i, r = c >> 4, q = c & 15;
            const float a[4] = {pa[i].x, pa[i].y, pa[i].z, pa[i].w};
            uint32_t ph[2], pm[2], pl[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                ph[j] = bf16_pair(a[2 * j], a[2 * j + 1]);
                const float r0 = a[2 * j] - bf16_low_f32(ph[j]), r1 = a[2 * j + 1] - bf16_high_f32(ph[j]);
                pm[j] = bf16_pair(r0, r1);
                pl[j] = bf16_pair(r0 - bf16_low_f32(pm[j]), r1 - bf16_high_f32(pm[j]));
            }
            *(u32x2*)&sA[0][r][4 * q] = u32x2{pl[0], pl[1]};
            *(u32x2*)&sA[1][r][4 * q] = u32x2{pm[0], pm[1]};
            *(u32x2*)&sA[2][r][4 * q] = u32x2{ph[0], ph[1]};
        }
        if (wb == 0) w16_stage_block<WT, 0>(pw, &sW[wr][0], &sD[0][wr]);
        else w16_stage_block<WT, 2>(pw, &sW[wr][32], &sD[1][wr]);
    };

    f32x16 acc, zero;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = zero[r] = 0.0f;
    const int nw = 32 * wave;   // this wave's weight rows of the tile

    if (s_lo < s_hi) load(s_lo);
    for (int s = s_lo; s < s_hi; s++) {
        store();
        __syncthreads();
        if (s + 1 < s_hi) load(s + 1);
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            bf16x8 wf[2], af[3][2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int ko = 32 * kb + 16 * h + 8 * hi;
                wf[h] = *(const bf16x8*)&sW[nw + l32][ko];
#pragma unroll
                for (int e = 0; e < 3; e++) af[e][h] = *(const bf16x8*)&sA[e][l32][ko];
            }
            f32x4 dw[4];
#pragma unroll
            for (int q = 0; q < 4; q++) dw[q] = *(const f32x4*)&sD[kb][nw + 4 * hi + 8 * q];
            // the MFMA computes D[n][m]: A operand = weight fragment, B = activations
            f32x16 p = zero;
#pragma unroll
            for (int e = 0; e < 3; e++)
#pragma unroll
                for (int h = 0; h < 2; h++) p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[h], af[e][h], p, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; r++) acc[r] = fmaf(dw[r >> 2][r & 3], p[r], acc[r]);
        }
        __syncthreads();
    }

    // lane l holds activation row m = l % 32 and weight rows n = 8 (r / 4) + 4 (l / 32) + r % 4
    const bool vec_ok = (N % 4) == 0 && (((uintptr_t)C & 15u) == 0);
    const int gm = m0 + l32;
    if (gm >= M) return;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int gn = n0 + nw + 4 * hi + 8 * q;
        if (vec_ok && gn + 3 < N) {
            *(f32x4*)(C + (size_t)gm * N + gn) = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (gn + r < N) C[(size_t)gm * N + gn + r] = acc[4 * q + r];
        }
    }
}

// ---- decode form (1-4 activation rows) ------------------------------------------------------
// A GEMV on the VALU: the bf16-MFMA tile wastes 31 of its 32 rows at M = 1 and splits K to fill
// the chip (13 us at N = K = 4096); here every lane owns pairs of adjacent weight blocks (36 or 68
// bytes, loaded straight into VGPRs), the workgroup stages the activation rows of a K tile in LDS
// with each block's fp32 sum, and a lane's block contributes
//     d_w * (sum_k a_k q_k - 8 * sum_k a_k)      (Q4_0; Q8_0: d_w * sum_k a_k q_k)
// with q_k converted once per element (v_cvt_f32_ubyte) and one fma per element and activation
// row: the reference's sum of a_k * (q_k - 8) * d_w regrouped (fp32 rounding differs).  RPW
// weight rows per 256-thread workgroup, RPW / 4 per wave, every activation value read from LDS
// serving all of them.
constexpr int kW16KTile = 4096;   // activation elements per row and K tile
// LDS layout of a staged activation row: pair p of the tile (64 floats) at p * 68 floats, so the
// 16-byte reads of 16 lanes (consecutive pairs, 272 bytes apart) hit distinct bank groups
constexpr int kW16PairPitch = 68;

// NW dwords from p (4-byte aligned) by 16-, 8- and 4-byte loads.
template <int NW>
__device__ __forceinline__ void load_dwords_a4(const uint32_t* __restrict__ p, uint32_t* w) {
#pragma unroll
    for (int i = 0; i + 4 <= NW; i += 4) {
        const u32x4a4 v = *(const u32x4a4*)(p + i);
        w[i] = v.x; w[i + 1] = v.y; w[i + 2] = v.z; w[i + 3] = v.w;
    }
    constexpr int r0 = NW & ~3;
    if constexpr (NW - r0 >= 2) {
        const u32x2a4 v = *(const u32x2a4*)(p + r0);
        w[r0] = v.x; w[r0 + 1] = v.y;
    }
    if constexpr ((NW - r0) & 1) w[NW - 1] = p[NW - 1];
}

template <int WT, int MR, int RPW>
__global__ __launch_bounds__(256) void w16_gemv_kernel(const uint8_t* __restrict__ W, const float* __restrict__ A,
                                                       float* __restrict__ C, int N, int nb) {
    constexpr int VR = RPW / 4;                                  // weight rows per wave
    constexpr int BB = block_bytes(WT), PW = BB / 2;             // pair: 36 / 68 bytes = 9 / 17 dwords
    __shared__ __attribute__((aligned(16))) float sx[MR][kW16KTile / 64 * kW16PairPitch];
    __shared__ float ssum[MR][kW16KTile / 32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row0 = (int)blockIdx.x * RPW + wave * VR;
    const size_t K = (size_t)nb * 32;
    float acc[VR][MR];
#pragma unroll
    for (int v = 0; v < VR; v++)
#pragma unroll
        for (int m = 0; m < MR; m++) acc[v][m] = 0.0f;

    for (int kb0 = 0; kb0 < nb; kb0 += kW16KTile / 32) {
        const int kbn = min(kW16KTile / 32, nb - kb0);          // blocks in this K tile (even)
        const int np = kbn / 2;
        // this lane's first pair of weight blocks for its rows, issued before the staging loads
        int p = lane;
        uint32_t w[VR][PW];
#pragma unroll
        for (int v = 0; v < VR; v++)
            if (p < np && row0 + v < N)
                load_dwords_a4<PW>((const uint32_t*)(W + ((size_t)(row0 + v) * nb + kb0 + 2 * p) * BB), w[v]);
        // stage the K tile's activations, 8 floats per thread and step, and the block sums
        for (int e = threadIdx.x; e < MR * kbn * 4; e += 256) {
            const int m = e / (kbn * 4), c = e - m * kbn * 4;        // c: 8-float chunk of row m
            const f32x4* src = (const f32x4*)(A + (size_t)m * K + (size_t)kb0 * 32 + 8 * c);
            const f32x4 x0 = src[0], x1 = src[1];
            // chunk c = elements 8c .. 8c + 7 of the tile: pair c / 8, offset 8 (c % 8) in it
            float* dst = &sx[m][(c >> 3) * kW16PairPitch + 8 * (c & 7)];
            *(f32x4*)dst = x0;
            *(f32x4*)(dst + 4) = x1;
            // the 4 chunks of a block sit in 4 consecutive lanes: their partial sums meet by DPP
            float part = ((x0.x + x0.y) + (x0.z + x0.w)) + ((x1.x + x1.y) + (x1.z + x1.w));
            part += dpp_mov<0xB1>(part);   // quad_perm [1,0,3,2]
            part += dpp_mov<0x4E>(part);   // quad_perm [2,3,0,1]
            if ((c & 3) == 0) ssum[m][c >> 2] = part;
        }
        __syncthreads();
        if (row0 < N) {
            for (bool first = true; p < np; p += 64, first = false) {
                if (!first) {
#pragma unroll
                    for (int v = 0; v < VR; v++)
                        if (row0 + v < N)
                            load_dwords_a4<PW>((const uint32_t*)(W + ((size_t)(row0 + v) * nb + kb0 + 2 * p) * BB), w[v]);
                }
#pragma unroll
                for (int h = 0; h < 2; h++) {       // block 2p + h of the tile
                    const int b = 2 * p + h;
                    float part[VR][MR];
#pragma unroll
                    for (int v = 0; v < VR; v++)
#pragma unroll
                        for (int m = 0; m < MR; m++) part[v][m] = 0.0f;
#pragma unroll
                    for (int i = 0; i < (WT == kWQ40 ? 4 : 8); i++) {
                        // 4 quants of each row: Q4_0 elements 4i..4i+3 (low nibbles) and
                        // 16+4i..16+4i+3 (high nibbles); Q8_0 elements 4i..4i+3
                        float q[VR][WT == kWQ40 ? 8 : 4];
#pragma unroll
                        for (int v = 0; v < VR; v++) {
                            const uint32_t wd = word_at(w[v], h * BB + 2 + 4 * i);
                            if constexpr (WT == kWQ40) {
                                const uint32_t lo = wd & 0x0F0F0F0Fu, hi = (wd >> 4) & 0x0F0F0F0Fu;
#pragma unroll
                                for (int j = 0; j < 4; j++) {
                                    q[v][j] = (float)((lo >> (8 * j)) & 0xFFu);
                                    q[v][4 + j] = (float)((hi >> (8 * j)) & 0xFFu);
                                }
                            } else {
#pragma unroll
                                for (int j = 0; j < 4; j++) q[v][j] = (float)(int8_t)((wd >> (8 * j)) & 0xFFu);
                            }
                        }
#pragma unroll
                        for (int m = 0; m < MR; m++) {
                            const float* xp = &sx[m][p * kW16PairPitch + 32 * h];
                            const f32x4 xl = *(const f32x4*)(xp + 4 * i);
#pragma unroll
                            for (int v = 0; v < VR; v++) {
                                part[v][m] = fmaf(xl.x, q[v][0], part[v][m]);
                                part[v][m] = fmaf(xl.y, q[v][1], part[v][m]);
                                part[v][m] = fmaf(xl.z, q[v][2], part[v][m]);
                                part[v][m] = fmaf(xl.w, q[v][3], part[v][m]);
                            }
                            if constexpr (WT == kWQ40) {
                                const f32x4 xh = *(const f32x4*)(xp + 16 + 4 * i);
#pragma unroll
                                for (int v = 0; v < VR; v++) {
                                    part[v][m] = fmaf(xh.x, q[v][4], part[v][m]);
                                    part[v][m] = fmaf(xh.y, q[v][5], part[v][m]);
                                    part[v][m] = fmaf(xh.z, q[v][6], part[v][m]);
                                    part[v][m] = fmaf(xh.w, q[v][7], part[v][m]);
                                }
                            }
                        }
                    }
#pragma unroll
                    for (int v = 0; v < VR; v++) {
                        const float d = f16_to_f32(half_at(w[v], h * BB));
#pragma unroll
                        for (int m = 0; m < MR; m++) {
                            const float t = (WT == kWQ40) ? fmaf(-8.0f, ssum[m][b], part[v][m]) : part[v][m];
                            acc[v][m] = fmaf(d, t, acc[v][m]);
                        }
                    }
                }
            }
        }
        if (kb0 + kW16KTile / 32 < nb) __syncthreads();   // the next tile overwrites the LDS
    }
#pragma unroll
    for (int v = 0; v < VR; v++)
#pragma unroll
        for (int m = 0; m < MR; m++) acc[v][m] = wave_sum(acc[v][m]);
    if (lane == 0) {
#pragma unroll
        for (int v = 0; v < VR; v++)
            if (row0 + v < N) {
#pragma unroll
                for (int m = 0; m < MR; m++) C[(size_t)m * N + row0 + v] = acc[v][m];
            }
    }
}

namespace {
constexpr int kW16MinWGs = 256, kW16TargetWGs = 512, kW16MaxSplits = 16;
constexpr int kW16GemvMaxRows = 4;
bool w16_uses_gemv(int M) { return M >= 1 && M <= kW16GemvMaxRows; }

int w16_tiles(int M, int N, int bm, int bn) { return ((N + bn - 1) / bn) * ((M + bm - 1) / bm); }

struct W16Plan {
    int tile;    // 0: 32 x 128, 1: 64 x 128, 2: 128 x 128, 3: 128 x 256
    int splits;
};

// Up to 32 rows: the 32 x 128 tile, split along K to 512 workgroups.  Above: the tile and split
// with the least predicted time.  A workgroup's step of two blocks takes, with 1, 2, 3 workgroups
// on a CU (us; measured with K = 8192 and one full round, Q4_0 / Q8_0): 64 x 128 1.07, 1.75, 2.44 /
// 1.01, 1.89, 2.77; 128 x 128 1.62, 2.88 / 1.70, 3.10; 128 x 256 2.65 / 2.90.  The constants lie between
// the two types: only the tiles' proportions matter to the pick, and those they share.  A split
// adds the reduction launch (2.5 us) and its traffic at 4 TB/s.  Splits only where the 128 x 128
// grid leaves CUs idle, at least 4 steps each.  Measured, us, best of all tiles and splits / this
// rule's pick, Q4_0 and Q8_0: 64 x 4096 x 4096 18.0 / 17.9 and 17.7 / 17.8; 128 x 14336 x 4096 52.6 /
// 53.8 and 56.7 / 57.7; 512 x 4096 x 4096 56.7 / 57.6 and 60.9 / 61.5; 700 x 3008 x 3008 52.4 / 53.3 and
// 56.4 / 56.6; 1024 x 4096 x 4096 level; 218 x 2765 x 18176 level; 2048 x 4096 x 4096 level.  Over 36
// shapes the pick is within 4% of the best for 33 (Q4_0) and 30 (Q8_0); the worst, both types: 88 x
// 1947 x 4992 17.9 / 20.0, 256 x 4096 x 4096 36.4 / 39.7.
// max_splits: what the caller's scratch holds, the tile then chosen for that.
W16Plan w16_plan(int M, int N, int K, int max_splits) {
    if (max_splits > kW16MaxSplits) max_splits = kW16MaxSplits;
    const int steps = K / 64;
    const int grid128 = w16_tiles(M, N, 128, 128);
    if (M <= kW16SmallRows) {
        const int wgs = w16_tiles(M, N, kW16SmallRows, 128);
        if (wgs >= kW16MinWGs) return {0, 1};
        int sp = (kW16TargetWGs + wgs - 1) / wgs;
        sp = sp < steps / 4 ? sp : steps / 4;
        sp = sp < max_splits ? sp : max_splits;
        return {0, sp < 1 ? 1 : sp};
    }
    constexpr int cap[4] = {0, 3, 2, 1};
    constexpr double step_us[4][4] = {{}, {0.0, 1.07, 1.86, 2.6}, {0.0, 1.7, 3.05}, {0.0, 2.85}};
    W16Plan best{1, 1};
    double best_us = 1e30;
    for (int tile = 1; tile <= 3; tile++) {
        const int tiles = w16_tiles(M, N, tile == 1 ? 64 : 128, tile == 3 ? 256 : 128);
        for (int sp = 1; sp <= max_splits; sp++) {
            if (sp > 1 && (grid128 >= kW16MinWGs || steps / sp < 4)) break;
            const int per_cu = (int)(((long long)((tiles + 7) / 8) * sp + 31) / 32);   // on the fullest XCD
            const double rounds = (double)(per_cu / cap[tile]) * step_us[tile][cap[tile]] + step_us[tile][per_cu % cap[tile]];
            double us = rounds * ((steps + sp - 1) / sp);
            if (sp > 1) us += 2.5 + (sp + 1) * (double)M * N * 4.0 / 4e6;
            if (us < best_us) {
                best_us = us;
                best = {tile, sp};
            }
        }
    }
    return best;
}
}  // namespace

int w16_splits(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || w16_uses_gemv(M)) return 1;
    return w16_plan(M, N, K, kW16MaxSplits).splits;
}

int w16_plan_code(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || w16_uses_gemv(M)) return -1;
    const W16Plan p = w16_plan(M, N, K, kW16MaxSplits);
    return p.tile + 16 * p.splits;
}

// The splits a workspace has to hold: the plan's, or the count that takes the 128 x 128 grid to 512
// workgroups where that is less.  Workspaces were sized by the latter before the plan had more than
// one tile; 57 x 10919 x 9472 then took 6 splits where the plan takes 8.
int w16_min_splits(int M, int N, int K) {
    const int sp = w16_splits(M, N, K), wgs = M > 0 && N > 0 ? w16_tiles(M, N, 128, 128) : 1;
    if (sp == 1 || M <= kW16SmallRows) return sp;
    const int most = (kW16TargetWGs + wgs - 1) / wgs;
    return sp < most ? sp : most;
}

template <class T, int WT>
static void w16_tile_launch(const float* A, const uint8_t* W, float* C, int M, int N, int nb, int splits, hipStream_t s) {
    const int tiles = w16_tiles(M, N, T::BM, T::BN);
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8), 1u, (unsigned)splits);
    hipLaunchKernelGGL((w16_kernel<T, WT>), grid, dim3(T::NT), 0, s, W, A, C, M, N, nb);
}

template <int WT>
static hipError_t w16_launch(const float* A, const uint8_t* W, float* C, int M, int N, int K, const W16Plan& p,
                             hipStream_t s) {
    const int nb = K / 32;
    if (p.tile == 0) {
        const dim3 grid((unsigned)((N + 127) / 128), (unsigned)((M + kW16SmallRows - 1) / kW16SmallRows), (unsigned)p.splits);
        hipLaunchKernelGGL((w16_small_kernel<WT>), grid, dim3(256), 0, s, W, A, C, M, N, nb);
    } else if (p.tile == 1) {
        w16_tile_launch<W16Mid, WT>(A, W, C, M, N, nb, p.splits, s);
    } else if (p.tile == 2) {
        w16_tile_launch<W16Big, WT>(A, W, C, M, N, nb, p.splits, s);
    } else {
        w16_tile_launch<W16Huge, WT>(A, W, C, M, N, nb, p.splits, s);
    }
    return hipGetLastError();
}

template <int WT, int MR>
static hipError_t w16_gemv_launch(const float* A, const uint8_t* W, float* C, int N, int K, hipStream_t s) {
    const int nb = K / 32;
    // 4 weight rows per wave while that keeps 512 workgroups, else 2 or 1 (whole call, us, with 256
    // in place of 512: N = K = 4096 M = 1 6.84 -> 5.6, M = 2 8.66 -> 6.56; N = 4096, K = 14336,
    // M = 4 33.4 -> 26.3; N = 14336 level; 1024 loses at M = 4: 35.6)
    constexpr int kGemvMinWGs = 512;
    if ((N + 15) / 16 >= kGemvMinWGs)
        hipLaunchKernelGGL((w16_gemv_kernel<WT, MR, 16>), dim3((N + 15) / 16), dim3(256), 0, s, W, A, C, N, nb);
    else if ((N + 7) / 8 >= kGemvMinWGs)
        hipLaunchKernelGGL((w16_gemv_kernel<WT, MR, 8>), dim3((N + 7) / 8), dim3(256), 0, s, W, A, C, N, nb);
    else
        hipLaunchKernelGGL((w16_gemv_kernel<WT, MR, 4>), dim3((N + 3) / 4), dim3(256), 0, s, W, A, C, N, nb);
    return hipGetLastError();
}

template <int WT>
static hipError_t w16_gemv_dispatch(const float* A, const uint8_t* W, float* C, int M, int N, int K, hipStream_t s) {
    switch (M) {
        case 1: return w16_gemv_launch<WT, 1>(A, W, C, N, K, s);
        case 2: return w16_gemv_launch<WT, 2>(A, W, C, N, K, s);
        case 3: return w16_gemv_launch<WT, 3>(A, W, C, N, K, s);
        default: return w16_gemv_launch<WT, 4>(A, W, C, N, K, s);
    }
}

hipError_t launch_w16(int wtype, const float* A, const uint8_t* W, float* C, int M, int N, int K, float* partials,
                      int max_splits, hipStream_t s) {
    if (wtype != kWQ40 && wtype != kWQ80) return hipErrorNotSupported;
    if (w16_uses_gemv(M)) {
        note_engine(KSQ_ENG_W16);
        return wtype == kWQ40 ? w16_gemv_dispatch<kWQ40>(A, W, C, M, N, K, s)
                              : w16_gemv_dispatch<kWQ80>(A, W, C, M, N, K, s);
    }
    const W16Plan plan = w16_plan(M, N, K, max_splits);
    const int splits = plan.splits;
    note_engine(KSQ_ENG_W16 | (splits > 1 ? KSQ_ENG_SPLITK : 0u));
    float* out = C;
    if (splits > 1) {
        if (!partials) return hipErrorInvalidValue;
        out = partials;
    }
    hipError_t e = wtype == kWQ40 ? w16_launch<kWQ40>(A, W, out, M, N, K, plan, s)
                                  : w16_launch<kWQ80>(A, W, out, M, N, K, plan, s);
    if (e != hipSuccess || splits == 1) return e;
    return launch_splitk_reduce(partials, C, (int64_t)M * N, splits, s);
}

}  // namespace ksq
