// Dense contractions on the matrix cores.
//
//   C[M x N] = A[M x K] . B      A fp32 row-major, fp32 accumulate
//
// fp32 B [K x N] row-major (OP_MATMUL; CpuBackend.java:168-188 in the reference): v_mfma_f32_32x32x2_f32 in k_matmul, whose
// wavefronts share a tile's K and feed the matrix cores straight from the caches, for products of few tiles;
// v_mfma_f32_32x32x16_bf16 on the exact pieces of both operands in k_matmul_split for those that the matrix rate bounds;
// k_matmul_lds (fp32 instructions, tiles through LDS) for large ones over a short K.
//
// Q8 B [N x Kp] int8 + one fp32 scale per 32-group (prefill-time Q8 GEMM; the M = 1 decode case is the HBM-bound
// kernel in kernels_q8.hip): v_mfma_f32_32x32x16_bf16 at full fp32 accuracy.  An int8 weight is exact in bf16,
// and an fp32 activation is the exact sum of three bf16 numbers (its top, middle and bottom 8 significant bits,
// taken by truncation), so x . q = hi . q + mid . q + lo . q with every product exact and fp32 accumulation: three
// bf16 MFMAs of K = 16 replace eight fp32 MFMAs of K = 2 at four times the rate.  The group scale multiplies the
// finished 32-k partial sums (one scale per accumulator column per step).  Tile shapes (64 x 64, 64 x 128,
// 128 x 128), scale groups per step and wavefront sets per workgroup are template arguments chosen per problem
// shape by launch_q8_gemm; the epilogue adds bias / GELU / residual or pairs interleaved gate/up columns (SwiGLU).
#include <cstdlib>
#include "dj_common.h"
#include "dj_device.h"
#include "gemm_epilogue.h"
#include "gemm_rows.h"

namespace dj {

typedef float floatx16 __attribute__((ext_vector_type(16)));

namespace {

constexpr int BM = 64, BN = 64;            // Q8 tiles
constexpr int BM2 = 128, BN2 = 128;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// bf16(a) | bf16(b) << 16, both by truncation
__device__ __forceinline__ uint32_t pack_bf16_hi(float a, float b) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302);
}
__device__ __forceinline__ float top_bits(float x) {      // the leading 8 significant bits of x: a bf16 value
    return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & 0xffff0000u);
}

// ── fp32 x fp32 ─────────────────────────────────────────────────────────────
// One workgroup computes a tile of 32 TM x 32 TN; its KW wavefronts each multiply the WHOLE tile over their own share of K
// (stages of 8 U consecutive k dealt in turn) and are added through LDS at the end, in a fixed order.  As no two
// wavefronts want the same operand values there is nothing to stage: every lane loads what the matrix instruction takes
// from it (row or column lane % 32, half of the stage's k by lane / 32, so A comes as 128-bit words) into registers,
// D - 1 stages ahead, and the loop has no barrier.
// Bound: the fp32 matrix rate at the large end (157 TFLOP/s: 64 cycles a 32 x 32 x 2 product), one trip to memory and the
// launch at the small one.  What limits the stages in flight is the L1: a compute unit has 256 lines, and once more than
// that are outstanding they evict one another (1 x 2752 x 1024 with twice the wavefronts: 11.4 us instead of 7.8).
// Before (64 x 64 or 128 x 128 tiles staged through LDS, two barriers per 32 k) -> now: 64 x 256 x 256 10.3 -> 3.7 us,
// 256 x 768 x 192 8.9 -> 3.9, 500 x 2752 x 1024 61 -> 32, 500 x 1024 x 2752 114 -> 33, 2048 x 1024 x 2752 125 -> 97
// (119 TFLOP/s).
__device__ __forceinline__ float at_bytes(const float *base, uint32_t bytes) {
    return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + bytes);
}

template <int TM, int TN, int KW, int U, int D, bool VEC>
__global__ void __launch_bounds__(64 * KW) k_matmul(const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C,
                                                    const int M, const int N, const int K, const int tiles_m, const int tiles_n) {
    constexpr int SK = 8 * U;
    constexpr int kStride = 36;                     // LDS row of a 32-column block (16-byte aligned, spreads the two halves)
    __shared__ __align__(16) float red[KW][32 * kStride];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = lane >> 5, l32 = lane & 31;
    // Workgroups go to the eight XCDs in turn: give each XCD a run of neighbouring tiles, along the larger operand, so
    // that its L2 holds an eighth of that one.
    const int total = tiles_m * tiles_n, xcd = blockIdx.x & 7, q = total >> 3, r = total & 7;
    const int idx = xcd * q + (xcd < r ? xcd : r) + (int)(blockIdx.x >> 3);
    const bool by_cols = N >= M;
    const int tile_n = by_cols ? idx / tiles_m : idx % tiles_n, tile_m = by_cols ? idx % tiles_m : idx / tiles_n;
    const int m0 = tile_m * 32 * TM, n0 = tile_n * 32 * TN;

    // rows and columns past the matrix repeat its last one: their products are not stored
    const float *Am = A + (int64_t)m0 * K;
    uint32_t a_off[TM], b_off[TN];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int row = 32 * i + l32 < M - m0 ? 32 * i + l32 : M - 1 - m0;
        a_off[i] = ((uint32_t)row * (uint32_t)K + 4u * U * half) * 4u;
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int col = n0 + 32 * j + l32 < N ? n0 + 32 * j + l32 : N - 1;
        b_off[j] = (4u * U * half * (uint32_t)N + (uint32_t)col) * 4u;
    }

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    struct Stage { float a[U][TM][4], b[U][TN][4]; };
    auto load = [&](Stage &st, int k0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const char *p = reinterpret_cast<const char *>(Am + k0 + 4 * u) + a_off[i];
                if constexpr (VEC) {
                    const float4 v = *reinterpret_cast<const float4 *>(p);
                    st.a[u][i][0] = v.x; st.a[u][i][1] = v.y; st.a[u][i][2] = v.z; st.a[u][i][3] = v.w;
                } else {
#pragma unroll
                    for (int x = 0; x < 4; x++) st.a[u][i][x] = reinterpret_cast<const float *>(p)[x];
                }
            }
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const float *row = B + (int64_t)(k0 + 4 * u + x) * N;
#pragma unroll
                for (int j = 0; j < TN; j++) st.b[u][j][x] = at_bytes(row, b_off[j]);
            }
        }
    };
    auto multiply = [&](const Stage &st) {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(st.a[u][i][x], st.b[u][j][x], acc[i][j], 0, 0, 0);
    };

    // No load of the loop sits under a branch (the last one is repeated instead): the number in flight is then known at
    // compile time, and a stage's products wait for that stage's loads alone.
    const int stages = K / SK, mine = (stages - wave + KW - 1) / KW;
    if (mine > 0) {
        Stage st[D];
        auto stage_k = [&](int i) { return (wave + (i < mine ? i : mine - 1) * KW) * SK; };
#pragma unroll
        for (int d = 0; d < D - 1; d++) load(st[d], stage_k(d));
        int i = 0;
        for (; i + D <= mine; i += D) {
#pragma unroll
            for (int d = 0; d < D; d++) {
                load(st[(d + D - 1) % D], stage_k(i + d + D - 1));
                __builtin_amdgcn_sched_barrier(0);      // (the scheduler would move the loads down to their use)
                multiply(st[d]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int d = 0; d < D - 1; d++)
            if (i + d < mine) multiply(st[d]);
    }
    if (stages * SK < K && wave == stages % KW) {   // what is left of K, 8 at a time: zeros past its end, in both operands
        const uint32_t back = 4u * (U - 1) * half;
#pragma unroll
        for (int i = 0; i < TM; i++) a_off[i] -= back * 4u;
#pragma unroll
        for (int j = 0; j < TN; j++) b_off[j] -= back * (uint32_t)N * 4u;
        for (int k0 = stages * SK; k0 < K; k0 += 8) {
            float a[TM][4], b[TN][4];
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const int k = k0 + 4 * half + x;
                const bool ok = k < K;
#pragma unroll
                for (int i = 0; i < TM; i++) a[i][x] = ok ? at_bytes(Am + k0 + x, a_off[i]) : 0.0f;
#pragma unroll
                for (int j = 0; j < TN; j++) b[j][x] = ok ? at_bytes(B + (int64_t)(k0 + x) * N, b_off[j]) : 0.0f;
            }
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][x], b[j][x], acc[i][j], 0, 0, 0);
        }
    }

    // acc[i][j][e] is C[32 i + 8 (e / 4) + 4 half + e % 4][32 j + l32] of the tile; 32 x 32 blocks leave one by one
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if (i + j > 0) __syncthreads();
#pragma unroll
            for (int e = 0; e < 16; e++) red[wave][(8 * (e >> 2) + 4 * half + (e & 3)) * kStride + l32] = acc[i][j][e];
            __syncthreads();
            for (int o = threadIdx.x; o < 1024; o += 64 * KW) {
                const int row = o >> 5, col = o & 31;
                float v = red[0][row * kStride + col];
#pragma unroll
                for (int w = 1; w < KW; w++) v += red[w][row * kStride + col];
                if (m0 + 32 * i + row < M && n0 + 32 * j + col < N) C[(int64_t)(m0 + 32 * i + row) * N + n0 + 32 * j + col] = v;
            }
        }
}

// Outputs of at most 512 tiles of 16 x 16, two a compute unit: tiles of 32 x 32 would leave half to all but a few of them idle, each
// tile with four times the products behind one another.  As k_matmul: 16 wavefronts share K in stages of 16 k dealt in turn, operands straight into
// registers, a stage ahead (two, three or five: 0 to 25 % slower); lane l has row or column l % 16 and the four k of a stage at 4 (l / 16), the x-th of which goes into
// the x-th product (the four groups' k add up whatever their order).
// Bound by a chain of a few trips to the caches and the launch.  k_matmul -> this, us: 256 x 192 x 768 7.4 -> 4.4, x 1003 9.3 -> 5.0;
// 16 x 2048 x 2048 15.0 -> 7.6; 4 x 2752 x 1024 8.8 -> 4.8; 128 x 384 x 1500 12.0 -> 6.1; 17 x 17 x 4000 24.7 -> 11.0; 500 x 256 x 700 7.7 ->
// 6.1; 256 x 512 x 2048 15.8 -> 13.5.  Error against float64 1.3e-7 of the result's rms at 1003 k, 1.6e-7 before.
template <bool VEC>
__global__ void __launch_bounds__(1024) k_matmul_16(const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, const int M, const int N,
                                                    const int K, const int tiles_m, const int tiles_n) {
    constexpr int kWaves = 16, kStage = 16, kPitch = 17, D = 2;
    typedef float floatx4 __attribute__((ext_vector_type(4)));
    __shared__ float red[kWaves][16 * kPitch];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, quarter = lane >> 4;
    const int total = tiles_m * tiles_n, xcd = blockIdx.x & 7, q = total >> 3, r = total & 7;      // (as k_matmul)
    const int idx = xcd * q + (xcd < r ? xcd : r) + (int)(blockIdx.x >> 3);
    const bool by_cols = N >= M;
    const int tile_n = by_cols ? idx / tiles_m : idx % tiles_n, tile_m = by_cols ? idx % tiles_m : idx / tiles_n;
    const int m0 = tile_m * 16, n0 = tile_n * 16;

    // rows and columns past the matrix repeat its last one: their products are not stored
    const float *Am = A + (int64_t)m0 * K;
    const uint32_t a_off = ((uint32_t)(l16 < M - m0 ? l16 : M - 1 - m0) * (uint32_t)K + 4u * quarter) * 4u;
    const uint32_t b_off = (4u * quarter * (uint32_t)N + (uint32_t)(n0 + l16 < N ? n0 + l16 : N - 1)) * 4u;
    floatx4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};      // (two sums of half as many products: less error)
    struct Stage { float a[4], b[4]; };
    auto load = [&](Stage &st, int k0) {
        const char *p = reinterpret_cast<const char *>(Am + k0) + a_off;
        if constexpr (VEC) {
            const float4 v = *reinterpret_cast<const float4 *>(p);
            st.a[0] = v.x; st.a[1] = v.y; st.a[2] = v.z; st.a[3] = v.w;
        } else {
#pragma unroll
            for (int x = 0; x < 4; x++) st.a[x] = reinterpret_cast<const float *>(p)[x];
        }
#pragma unroll
        for (int x = 0; x < 4; x++) st.b[x] = at_bytes(B + (int64_t)(k0 + x) * N, b_off);
    };
    auto multiply = [&](const Stage &st) {
#pragma unroll
        for (int x = 0; x < 4; x++) acc[x & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(st.a[x], st.b[x], acc[x & 1], 0, 0, 0);
    };
    const int stages = K / kStage, mine = (stages - wave + kWaves - 1) / kWaves;
    if (mine > 0) {
        Stage st[D];
        auto at = [&](int i) { return ((i < mine ? i : mine - 1) * kWaves + wave) * kStage; };
#pragma unroll
        for (int d = 0; d < D; d++) load(st[d], at(d));
        int i = 0;
        for (; i + D <= mine; i += D) {
#pragma unroll
            for (int d = 0; d < D; d++) {
                multiply(st[d]);
                load(st[d], at(i + d + D));
            }
        }
#pragma unroll
        for (int d = 0; d < D - 1; d++)
            if (i + d < mine) multiply(st[d]);
    }
    if (stages * kStage < K && wave == (stages & (kWaves - 1))) {      // the rest of K, with zeros past its end
        Stage st;
        const int k0 = stages * kStage, k = k0 + 4 * quarter;
#pragma unroll
        for (int x = 0; x < 4; x++) {
            st.a[x] = k + x < K ? at_bytes(Am + k0 + x, a_off) : 0.0f;
            st.b[x] = k + x < K ? at_bytes(B + (int64_t)(k0 + x) * N, b_off) : 0.0f;
        }
        multiply(st);
    }
    // acc[.][e] is C[4 quarter + e][l16]
#pragma unroll
    for (int e = 0; e < 4; e++) red[wave][(4 * quarter + e) * kPitch + l16] = acc[0][e] + acc[1][e];
    __syncthreads();
    if (threadIdx.x >= 256) return;
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
    float v = red[0][row * kPitch + col];
#pragma unroll
    for (int w = 1; w < kWaves; w++) v += red[w][row * kPitch + col];
    if (m0 + row < M && n0 + col < N) C[(int64_t)(m0 + row) * N + n0 + col] = v;
}

// ── fp32 x fp32 on the bf16 matrix cores ────────────────────────────────────
// An fp32 value of at least 2^-103 is the exact sum of three bf16 values (itself rounded to bf16, the remainder rounded, the
// rest), of a smaller one pieces below 2^-126 may be lost (k_matmul_split looks for results that this can be seen in); so
//   a . b = ah bh + (ah bm + am bh) + (ah bl + am bm + al bh) + ...       what is left out is about 2^-26 of |a b|
// and six bf16 products of 16 k take 0.375 of the time of eight fp32 products of 2.  The first product and the five small ones
// have accumulators of their own, so that the large sum is cut off once per 16 k and set (fp32 instructions: eight times): its
// error against float64 is 0.99e-7 to 1.3e-7 of the result's rms at 1024 k by tile, where k_matmul has 2.9e-7; 1.5e-7 to
// 2.2e-7 against 4.7e-7 at 2752; 6e-8 to 7e-8 against 1.1e-7 at 192.
// Bound: the matrix cores at the clock they run the chip down to (about 27 products of 32 x 32 x 16 a ns over the whole chip; the
// same rate at every depth of pipelining tried) once the tiles fill it, loads and splits in turn below.  k_matmul or
// k_matmul_lds -> this: 500 x 2752 x 1024 31.4 -> 24.5 us, 1000 x 2752 x 1024 69 -> 43, 1000 x 7000 x 1024 153 -> 103.
struct Pieces { bf16x8 h, m, l; };
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
// (Dot products of two with -1 and 0 would take the pieces off without unpacking them, half the instructions at more than twice the
// time: 500 x 2752 x 1024 26.5 -> 25.3 us without them, 700 x 1024 x 2752 on 64 x 96 tiles 50.0 -> 45.3, 2000 x 4000 x 1024 on them
// 153 -> 143.)
__device__ __forceinline__ floatx2 less(floatx2 x, bf16x2 piece) {
    const uint32_t p = __builtin_bit_cast(uint32_t, piece);
    return {x[0] - __builtin_bit_cast(float, p << 16), x[1] - __builtin_bit_cast(float, p & 0xffff0000u)};
}
__device__ __forceinline__ Pieces split8(const float (&v)[8], float &most) {
    union U { bf16x2 p[4]; bf16x8 b; } h, m, l;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const floatx2 x = {v[2 * j], v[2 * j + 1]};
        asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most) : "v"(v[2 * j]), "v"(v[2 * j + 1]));   // (fmaxf: three instructions)
        h.p[j] = __builtin_convertvector(x, bf16x2);
        const floatx2 r = less(x, h.p[j]);
        m.p[j] = __builtin_convertvector(r, bf16x2);
        const floatx2 t = less(r, m.p[j]);
        l.p[j] = __builtin_convertvector(t, bf16x2);
    }
    return {h.b, m.b, l.b};
}
__device__ __forceinline__ floatx16 product(bf16x8 a, bf16x8 b, floatx16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// A workgroup computes a tile of 32 TM x 32 WC in WC x KS wavefronts: a wavefront has 32 of its columns and every KS-th 16 k
// (the sets' sums meet in LDS at the end, in a fixed order).  The columns' values go from memory to the registers of the one
// wavefront that splits and multiplies them, two steps of 16 KS k ahead; the rows' are split once for the workgroup and shared
// through LDS (16-byte operands in lane order), one step ahead.
template <int TM, int WC, int KS, bool VEC>
__global__ void __launch_bounds__(64 * WC * KS) k_matmul_split(const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C,
                                                               const int M, const int N, const int K, const int tiles_m, const int tiles_n) {
    constexpr int kWaves = WC * KS, kStep = 16 * KS, kRows = 32 * TM;
    constexpr int kStages = (TM + WC - 1) / WC;     // groups of 8 values of A that a thread stages a step (some threads: one fewer)
    constexpr int kStride = 36;                     // LDS row of a 32-column block (16-byte aligned, spreads the two halves)
    constexpr int kOperands = KS * TM * 3 * 64;     // 16-byte words of a step
    __shared__ uint32_t row_most[kRows], col_most[32 * WC];
    __shared__ uint32_t again[kRows * WC], again_rows;          // the outputs to do again, a bit each; the blocks of 32 rows that hold some
    __shared__ __align__(16) uint4 lds[2 * kOperands * 16 > kWaves * 32 * kStride * 4 ? 2 * kOperands : kWaves * 32 * kStride / 4];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = lane >> 5, l32 = lane & 31, wc = wave % WC, set = wave / WC;
    // Workgroups go to the eight XCDs in turn: each XCD gets a run of neighbouring tiles, along the larger operand.
    const int total = tiles_m * tiles_n, xcd = blockIdx.x & 7, q = total >> 3, r = total & 7;
    const int idx = xcd * q + (xcd < r ? xcd : r) + (int)(blockIdx.x >> 3);
    const bool by_cols = N >= M;
    const int tile_n = by_cols ? idx / tiles_m : idx % tiles_n, tile_m = by_cols ? idx % tiles_m : idx / tiles_n;
    const int m0 = tile_m * kRows, n0 = tile_n * 32 * WC;

    // rows and columns past the matrix repeat its last one: their products are not stored
    const float *Am = A + (int64_t)m0 * K;
    uint32_t a_off[kStages];
#pragma unroll
    for (int g = 0; g < kStages; g++) {
        // wavefront w stages for set w / WC the rows 32 (w % WC) .., 32 (w % WC + WC) ..
        const int row = 32 * (wc + g * WC) + l32;
        a_off[g] = ((uint32_t)(row < M - m0 ? row : M - 1 - m0) * (uint32_t)K + 16u * set + 8u * half) * 4u;
    }
    const int col = n0 + 32 * wc + l32 < N ? n0 + 32 * wc + l32 : N - 1;
    const auto b_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), 0, (int)((uint32_t)K * (uint32_t)N * 4u), 0x00020000);
    const uint32_t b_off = ((16u * set + 8u * half) * (uint32_t)N + (uint32_t)col) * 4u;

    floatx16 acc[TM], low[TM];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][e] = low[i][e] = 0.0f;

    float most_a[kStages] = {}, most_b = 0.0f;       // the largest magnitude seen of the rows staged, of the column
    struct Eight { float v[8]; };
    auto load_a = [&](Eight (&a)[kStages], int k0) {
#pragma unroll
        for (int g = 0; g < kStages; g++) {
            if (wc + g * WC >= TM) break;           // wavefront-uniform
            const char *p = reinterpret_cast<const char *>(Am + k0) + a_off[g];
            if constexpr (VEC) {
                const float4 u = reinterpret_cast<const float4 *>(p)[0], v = reinterpret_cast<const float4 *>(p)[1];
                a[g] = {{u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w}};
            } else {
#pragma unroll
                for (int x = 0; x < 8; x++) a[g].v[x] = reinterpret_cast<const float *>(p)[x];
            }
        }
    };
    auto load_b = [&](Eight &b, int k0) {
#pragma unroll
        for (int x = 0; x < 8; x++) {
            b.v[x] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b_rsrc, (int)b_off, (int)((uint32_t)(k0 + x) * (uint32_t)N * 4u), 0));
        }
    };
    auto stage = [&](const Eight (&a)[kStages], int buffer) {
#pragma unroll
        for (int g = 0; g < kStages; g++) {
            if (wc + g * WC >= TM) break;
            const Pieces p = split8(a[g].v, most_a[g]);
            uint4 *at = lds + buffer * kOperands + (set * TM + wc + g * WC) * 192 + lane;
            at[0] = __builtin_bit_cast(uint4, p.h); at[64] = __builtin_bit_cast(uint4, p.m); at[128] = __builtin_bit_cast(uint4, p.l);
        }
    };
    auto multiply = [&](const Eight &raw, int buffer) {
        Pieces a[TM];
        const uint4 *at = lds + buffer * kOperands + set * TM * 192 + lane;
#pragma unroll
        for (int i = 0; i < TM; i++)
            a[i] = {__builtin_bit_cast(bf16x8, at[i * 192]), __builtin_bit_cast(bf16x8, at[i * 192 + 64]), __builtin_bit_cast(bf16x8, at[i * 192 + 128])};
        const Pieces b = split8(raw.v, most_b);
#define DJ_EACH(acc, x, y) _Pragma("unroll") for (int i = 0; i < TM; i++) acc[i] = product(a[i].x, b.y, acc[i])
        DJ_EACH(acc, h, h);
        DJ_EACH(low, h, m);
        DJ_EACH(low, m, h);
        DJ_EACH(low, m, m);
        DJ_EACH(low, h, l);
        DJ_EACH(low, l, h);
#undef DJ_EACH
    };

    // The loads past the last whole step repeat it: the number in flight is known at compile time.
    const int steps = K / kStep, tail = K - steps * kStep;
    if (steps > 0) {
        Eight a[2][kStages], b[2];
        auto step_k = [&](int i) { return (i < steps ? i : steps - 1) * kStep; };
        load_a(a[0], 0);
        load_b(b[0], 0);
        load_b(b[1], step_k(1));
        load_a(a[1], step_k(1));
        stage(a[0], 0);
        dev::lds_barrier();
        int i = 0;
        for (; i + 2 <= steps; i += 2) {
#pragma unroll
            for (int d = 0; d < 2; d++) {
                load_a(a[d], step_k(i + d + 2));
                multiply(b[d], d);
                load_b(b[d], step_k(i + d + 2));
                stage(a[d ^ 1], d ^ 1);
                dev::lds_barrier();
            }
        }
        if (i < steps) {
            multiply(b[0], 0);
            dev::lds_barrier();
        }
    }
    if (tail > 0) {                                 // zeros past the end of K, in both operands
        Eight a[kStages], b;
        const int k0 = steps * kStep, k = k0 + 16 * set + 8 * half;
#pragma unroll
        for (int x = 0; x < 8; x++) {
#pragma unroll
            for (int g = 0; g < kStages; g++) a[g].v[x] = wc + g * WC < TM && k + x < K ? at_bytes(Am + k0 + x, a_off[g]) : 0.0f;
            b.v[x] = k + x < K ? at_bytes(B + (int64_t)(k0 + x) * N, b_off) : 0.0f;
        }
        __syncthreads();
        stage(a, 0);
        __syncthreads();
        multiply(b, 0);
    }

    // acc[i][e] is C[32 i + 8 (e / 4) + 4 half + e % 4][l32] of the wavefront's columns
    float *red = reinterpret_cast<float *>(lds);
    for (int o = threadIdx.x; o < kRows + 32 * WC; o += 64 * kWaves) (o < kRows ? row_most[o] : col_most[o - kRows]) = 0u;
    for (int o = threadIdx.x; o < kRows * WC; o += 64 * kWaves) again[o] = 0u;
    if (threadIdx.x == 0) again_rows = 0u;
    __syncthreads();
#pragma unroll
    for (int g = 0; g < kStages; g++)
        if (wc + g * WC < TM) atomicMax(&row_most[32 * (wc + g * WC) + l32], __builtin_bit_cast(uint32_t, most_a[g]));
    atomicMax(&col_most[32 * wc + l32], __builtin_bit_cast(uint32_t, most_b));
    __syncthreads();
    // What an output may have lost with pieces below 2^-126 is at most K 2^-126 (the row's largest + the column's); limit is 2^24
    // times that (and as much for products below 2^-126), so that a larger result has lost less than one rounding.
    const float scale = (float)K * 0x1p-42f;
    auto limit = [&](uint32_t most) { return most ? (__builtin_bit_cast(float, most) + 0.5f) * 0x1p-60f * scale : -INFINITY; };    // (zeros lose nothing)
    const int c = threadIdx.x % (32 * WC);
    const float of_col = limit(col_most[c]);
    for (int o = threadIdx.x; o < kRows; o += 64 * kWaves) row_most[o] = __builtin_bit_cast(uint32_t, limit(row_most[o]));    // (read behind a barrier)
    auto store = [&](int i, auto &&of, auto &&wanted) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 16; e++) red[(wave * 32 + 8 * (e >> 2) + 4 * half + (e & 3)) * kStride + l32] = of(e);
        __syncthreads();
        for (int o = threadIdx.x; o < 1024 * WC; o += 64 * kWaves) {
            const int row = o / (32 * WC), at = ((c >> 5) * 32 + row) * kStride + (c & 31);
            float v = red[at];
#pragma unroll
            for (int w = 1; w < KS; w++) v += red[w * WC * 32 * kStride + at];
            const int out_row = m0 + 32 * i + row, out_col = n0 + c;
            if (out_row < M && out_col < N && wanted(32 * i + row, v)) C[(int64_t)out_row * N + out_col] = v;
        }
    };
#pragma unroll
    for (int i = 0; i < TM; i++)
        store(i, [&](int e) { return acc[i][e] + low[i][e]; }, [&](int row, float v) {
            if (fabsf(v) <= 3.40282347e38f && !(fabsf(v) <= __builtin_bit_cast(float, row_most[row]) + of_col)) return true;
            atomicOr(&again[row * WC + (c >> 5)], 1u << (c & 31));
            atomicOr(&again_rows, 1u << (row >> 5));
            return false;
        });
    __syncthreads();
    const uint32_t rows_again = again_rows;
    if (!rows_again) return;

    // An operand that is no finite number has no such pieces, a sum may leave the range in another order, and small values may
    // have lost theirs: those outputs come from the fp32 instructions, the 32 rows around one as in k_matmul.  1000 x 2752 x 1024:
    // 46 us, 69 with a NaN in one row, 128 with nothing else in an operand, 95 with one of values near 1e-24 (whose sums cancel
    // to below the limit here and there); a thread an output, product behind product, took 259 and 3070.
    // Lane and offsets are worked out anew, and few values are in flight: what this part keeps through the loops above, or holds
    // beyond their registers, changes how those are scheduled (500 x 2752 x 1024 23.3 -> 24.2 us with 32 k a round).
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    const int lane_of = t & 63, wave_of = __builtin_amdgcn_readfirstlane(t >> 6), half_of = lane_of >> 5, l32_of = lane_of & 31;
    const int col_of = n0 + 32 * (wave_of % WC) + l32_of;
    const uint32_t col_off = (uint32_t)(col_of < N ? col_of : N - 1) * 4u;
    const float *rows_of_tile = A + (int64_t)m0 * K;
#pragma unroll 1
    for (int i = 0; i < TM; i++) {
        if (!(rows_again >> i & 1)) continue;
        const int row = 32 * i + l32_of;
        const uint32_t row_off = (uint32_t)(row < M - m0 ? row : M - 1 - m0) * (uint32_t)K * 4u;
        floatx16 sum[2];
#pragma unroll
        for (int e = 0; e < 16; e++) sum[0][e] = sum[1][e] = 0.0f;
        auto products = [&](int k0, bool whole) __attribute__((always_inline)) {
            float av[8], bv[8];
#pragma unroll
            for (int x = 0; x < 8; x++) {
                const int k = k0 + 8 * (x >> 2) + 4 * half_of + (x & 3);
                const bool in = whole || k < K;
                av[x] = in ? at_bytes(rows_of_tile + k, row_off) : 0.0f;
                bv[x] = in ? at_bytes(B + (int64_t)k * N, col_off) : 0.0f;
            }
#pragma unroll
            for (int x = 0; x < 8; x++) sum[x & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[x], bv[x], sum[x & 1], 0, 0, 0);
        };
        int k0 = 16 * (wave_of / WC);
#pragma unroll 1
        for (; k0 + 16 <= K; k0 += 16 * KS) products(k0, true);
        if (k0 < K) products(k0, false);
        store(i, [&](int e) { return sum[0][e] + sum[1][e]; }, [&](int r, float) { return (again[r * WC + (c >> 5)] >> (c & 31) & 1) != 0; });
    }
}

// Where a tile per compute unit does not cover the product: workgroups of four wavefronts, a 64 x 64 tile (32 x 32 per
// wavefront), 32 k a step through LDS.  Both operands sit k-major there, so the 64 lanes of an operand read 32 consecutive
// floats per half (no bank conflicts).  The loads of the next step are issued before this step's products, and a compute unit
// holds four such workgroups, whose loads and barriers hide behind one another's products - the direct loads of k_matmul
// evict one another from the L1 as soon as two of its workgroups share a compute unit.
// Bound: the fp32 matrix rate.  k_matmul -> this: 1024 x 2752 x 1024 100 -> 68 us, 1000 x 7000 x 1024 266 -> 154,
// 4096 x 4096 x 256 122 -> 87.  (k_matmul_split has taken over from both over more than some 50 k.)
// A sum of K products is taken in four parts by k, as there: its error is that of k_matmul at every K (2.9e-7 of the result's
// rms at 1024 k), half of what one chain has.
__global__ void __launch_bounds__(256) k_matmul_lds(const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C,
                                                    const int M, const int N, const int K, const int tiles_n) {
    constexpr int T = 64, BK = 32, E = 8, kPad = 4, kParts = 4;  // E: values of each operand a thread stages per step
    __shared__ float As[BK][T + kPad];
    __shared__ float Bl[BK][T + kPad];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, half = lane >> 5, l32 = lane & 31;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const int m0 = ((int)blockIdx.x / tiles_n) * T, n0 = ((int)blockIdx.x % tiles_n) * T;

    const int a_row = t >> 2, a_k = (t & 3) * E;                 // E consecutive k of one row of A
    const int b_k = t >> 3, b_n = (t & 7) * E;                   // E consecutive columns of one k of B
    const bool a_vec = (K & 3) == 0, b_vec = (N & 3) == 0;
    float va[E], vb[E];
    auto fetch = [&](int k0) {
        const int row = m0 + a_row, k = k0 + b_k;
        if (row < M && a_vec && k0 + a_k + E <= K) {
            const float4 *p = reinterpret_cast<const float4 *>(A + (int64_t)row * K + k0 + a_k);
            const float4 x = p[0], y = p[1];
            va[0] = x.x; va[1] = x.y; va[2] = x.z; va[3] = x.w; va[4] = y.x; va[5] = y.y; va[6] = y.z; va[7] = y.w;
        } else {
#pragma unroll
            for (int j = 0; j < E; j++) va[j] = row < M && k0 + a_k + j < K ? A[(int64_t)row * K + k0 + a_k + j] : 0.0f;
        }
        if (k < K && b_vec && n0 + b_n + E <= N) {
            const float4 *p = reinterpret_cast<const float4 *>(B + (int64_t)k * N + n0 + b_n);
            const float4 x = p[0], y = p[1];
            vb[0] = x.x; vb[1] = x.y; vb[2] = x.z; vb[3] = x.w; vb[4] = y.x; vb[5] = y.y; vb[6] = y.z; vb[7] = y.w;
        } else {
#pragma unroll
            for (int j = 0; j < E; j++) vb[j] = k < K && n0 + b_n + j < N ? B[(int64_t)k * N + n0 + b_n + j] : 0.0f;
        }
    };

    floatx16 acc[kParts];
#pragma unroll
    for (int p = 0; p < kParts; p++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[p][e] = 0.0f;
    fetch(0);
    for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
        for (int j = 0; j < E; j++) As[a_k + j][a_row] = va[j];
#pragma unroll
        for (int j = 0; j < E; j++) Bl[b_k][b_n + j] = vb[j];
        __syncthreads();
        if (k0 + BK < K) fetch(k0 + BK);
#pragma unroll
        for (int kk = 0; kk < BK / 2; kk++)
            acc[kk % kParts] = __builtin_amdgcn_mfma_f32_32x32x2f32(As[2 * kk + half][wm + l32], Bl[2 * kk + half][wn + l32],
                                                                    acc[kk % kParts], 0, 0, 0);
        __syncthreads();
    }

    // acc[..][e] is C[8 (e / 4) + 4 half + e % 4][l32] of the wavefront's block
    const int col = n0 + wn + l32;
    if (col >= N) return;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const int row = m0 + wm + 8 * (e >> 2) + 4 * half + (e & 3);
        if (row < M) C[(int64_t)row * N + col] = (acc[0][e] + acc[1][e]) + (acc[2][e] + acc[3][e]);
    }
}

// ── Q8 weights: three-way bf16 split of the activations ────────────────────

// Workgroup tile 64 WTM x 64 WTN, WTM x WTN accumulators of 32 x 32 per wavefront (1 x 1: 64 x 64 tile; 2 x 2: 128 x 128).
// G: scale groups (of 32 k) per step.  A step costs two barriers and an LDS round trip whatever its size, and a
// 64 x 64 tile has only six products per wavefront and group to set against that, so it takes several groups a step.
// Operand element j of lane l is k = 16*step + 8*(l / 32) + j for A and B alike, so the pairing of the MFMA's
// k slots does not depend on how the hardware numbers them.
// KS: wavefront sets per workgroup (256 threads each).  Set s multiplies the groups s, s + KS, ... of every step
// into accumulators of its own and the sets are added through LDS at the end: with a grid of one small tile per
// CU this is what puts a second wavefront on every SIMD, so one set's conversions overlap the other's products.
template <int WTM, int WTN, int G, int KS>
__global__ void __launch_bounds__(256 * KS) k_gemm_q8(const float *__restrict__ A, const int8_t *__restrict__ Bq,
                                                 const float *__restrict__ Bs, float *__restrict__ C, int M,
                                                 const int N, const int K, const int kp, GemmEpilogue ep,
                                                 const int split_k, float *__restrict__ partial) {
    constexpr int TM = 64 * WTM, TN = 64 * WTN;
    constexpr int QBK = kQ8Group * G;        // k per step
    constexpr int LDK = QBK + 8;             // LDS row: the step's bf16 payload + 8 of padding (16-byte aligned, spreads banks)
    constexpr int NT = 256 * KS;
    constexpr int EL = TM * QBK / NT;        // activation floats a thread stages per step ...
    constexpr int TPR = QBK / EL;            // ... as one of TPR threads per tile row
    constexpr int ELB = TN * QBK / NT;       // weight bytes a thread stages per step ...
    constexpr int TPRB = QBK / ELB;          // ... as one of TPRB threads per tile column
    static_assert(EL >= 8 && EL <= kQ8Group && kQ8Group % EL == 0 && ELB >= 8 && ELB <= kQ8Group && kQ8Group % ELB == 0,
                  "a thread's share of a row lies inside one scale group");
    static_assert(G % KS == 0, "the step's groups divide over the sets");
    // One LDS block: the step's operands, and after the last step the sums the sets exchange.
    constexpr int kXsBytes = 3 * TM * LDK * 2, kWlBytes = TN * LDK * 2, kSsBytes = G * TN * 4;
    constexpr int kRedBytes = (KS - 1) * 4 * WTM * WTN * 16 * 64 * 4;
    constexpr int kOperandBytes = kXsBytes + kWlBytes + kSsBytes;
    __shared__ __align__(16) unsigned char lds[kOperandBytes > kRedBytes ? kOperandBytes : kRedBytes];
    uint16_t(*Xs)[TM][LDK] = reinterpret_cast<uint16_t(*)[TM][LDK]>(lds);             // hi / mid / lo pieces, k contiguous
    uint16_t(*Wl)[LDK] = reinterpret_cast<uint16_t(*)[LDK]>(lds + kXsBytes);          // weights as bf16, a row per output column
    float(*Ss)[TN] = reinterpret_cast<float(*)[TN]>(lds + kXsBytes + kWlBytes);       // the step's group scales per output column

    const int t = threadIdx.x;
    const int lane = t & 63, wave = (t >> 6) & 3, kset = t >> 8;
    const int wm = wave >> 1, wn = wave & 1;
    const int half = lane >> 5, l32 = lane & 31;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    if (ep.m_dev) {
        int live = ep.m_dev[0] + ep.m_extra;
        if (live < M) M = live;
        if (m0 >= M) return;                 // workgroup-uniform
    }
    const int groups = kp / kQ8Group;

    floatx16 acc[WTM][WTN];
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < WTN; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    const int s_row = t / TPR;               // tile row of A this thread stages, from k offset s_k
    const int s_k = (t % TPR) * EL;
    const int s_col = t / TPRB;              // tile column (row of B) this thread stages, from k offset s_kb
    const int s_kb = (t % TPRB) * ELB;
    const bool a_vec = (K & 3) == 0;

    float va[EL];
    int qraw[ELB / 4];
    float qsc = 0.0f;
    auto fetch = [&](int k0) {
        const int gr = m0 + s_row;
        if (gr < M && a_vec && k0 + s_k + EL <= K) {
            const float4 *p = reinterpret_cast<const float4 *>(A + (int64_t)gr * K + k0 + s_k);
#pragma unroll
            for (int q = 0; q < EL / 4; q++) {
                float4 x = p[q];
                va[4 * q] = x.x; va[4 * q + 1] = x.y; va[4 * q + 2] = x.z; va[4 * q + 3] = x.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < EL; j++) {
                int gk = k0 + s_k + j;
                va[j] = (gr < M && gk < K) ? A[(int64_t)gr * K + gk] : 0.0f;
            }
        }
        const int gn = n0 + s_col;
        if (gn < N && k0 + s_kb < kp) {
            const int *p = reinterpret_cast<const int *>(Bq + (int64_t)gn * kp + k0 + s_kb);  // kp is a multiple of 32: in bounds
#pragma unroll
            for (int q = 0; q < ELB / 4; q++) qraw[q] = p[q];
            qsc = Bs[(int64_t)gn * groups + (k0 + s_kb) / kQ8Group];
        } else {
#pragma unroll
            for (int q = 0; q < ELB / 4; q++) qraw[q] = 0;
            qsc = 0.0f;
        }
    };
    auto stage = [&]() {
        uint32_t ph[EL / 2], pm[EL / 2], pl[EL / 2], pw[ELB / 2];
#pragma unroll
        for (int j = 0; j < EL / 2; j++) {
            const float x0 = va[2 * j], x1 = va[2 * j + 1];
            const float h0 = top_bits(x0), h1 = top_bits(x1);
            const float r0 = x0 - h0, r1 = x1 - h1;              // exact: h is a prefix of x
            const float c0 = top_bits(r0), c1 = top_bits(r1);
            const float l0 = r0 - c0, l1 = r1 - c1;              // at most 8 significant bits left: a bf16 value
            ph[j] = pack_bf16_hi(h0, h1); pm[j] = pack_bf16_hi(c0, c1); pl[j] = pack_bf16_hi(l0, l1);
        }
#pragma unroll
        for (int q = 0; q < ELB / 4; q++) {
            const int r = qraw[q];
            pw[2 * q] = pack_bf16_hi((float)(int8_t)(r & 0xff), (float)(int8_t)((r >> 8) & 0xff));
            pw[2 * q + 1] = pack_bf16_hi((float)(int8_t)((r >> 16) & 0xff), (float)(int8_t)((r >> 24) & 0xff));
        }
#pragma unroll
        for (int q = 0; q < EL / 8; q++) {
            reinterpret_cast<uint4 *>(&Xs[0][s_row][s_k])[q] = make_uint4(ph[4 * q], ph[4 * q + 1], ph[4 * q + 2], ph[4 * q + 3]);
            reinterpret_cast<uint4 *>(&Xs[1][s_row][s_k])[q] = make_uint4(pm[4 * q], pm[4 * q + 1], pm[4 * q + 2], pm[4 * q + 3]);
            reinterpret_cast<uint4 *>(&Xs[2][s_row][s_k])[q] = make_uint4(pl[4 * q], pl[4 * q + 1], pl[4 * q + 2], pl[4 * q + 3]);
        }
#pragma unroll
        for (int q = 0; q < ELB / 8; q++)
            reinterpret_cast<uint4 *>(&Wl[s_col][s_kb])[q] = make_uint4(pw[4 * q], pw[4 * q + 1], pw[4 * q + 2], pw[4 * q + 3]);
        if (s_kb % kQ8Group == 0) Ss[s_kb / kQ8Group][s_col] = qsc;
    };

    // split_k > 0: gridDim.z workgroups share a tile's K, this one takes [k_begin, k_end) (split_k is a multiple of the
    // step) and leaves its bare sums in its own slab of `partial`; k_sum_partials_q8 adds the slabs in a fixed order
    const int k_begin = split_k > 0 ? (int)blockIdx.z * split_k : 0;
    const int k_end = split_k > 0 && k_begin + split_k < K ? k_begin + split_k : K;
    if (k_begin < k_end) fetch(k_begin);
    for (int k0 = k_begin; k0 < k_end; k0 += QBK) {
        stage();
        __syncthreads();
        if (k0 + QBK < k_end) fetch(k0 + QBK);     // next step's global loads fly while this step multiplies

        // (a run-time loop on purpose: unrolled, the products of consecutive groups get interleaved and the kernel
        // measured 4-10 % slower)
        for (int grp = kset; grp < G; grp += KS) {
        floatx16 g[WTM][WTN];                  // this group's unscaled partial sums
#pragma unroll
        for (int i = 0; i < WTM; i++)
#pragma unroll
            for (int j = 0; j < WTN; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) g[i][j][e] = 0.0f;
#pragma unroll
        for (int step = 0; step < kQ8Group / 16; step++) {
            const int kofs = grp * kQ8Group + step * 16 + half * 8;
            bf16x8 b[WTN];
#pragma unroll
            for (int tn = 0; tn < WTN; tn++) b[tn] = *reinterpret_cast<const bf16x8 *>(&Wl[wn * 32 * WTN + 32 * tn + l32][kofs]);
#pragma unroll
            for (int piece = 0; piece < 3; piece++) {
#pragma unroll
                for (int tm = 0; tm < WTM; tm++) {
                    const bf16x8 a = *reinterpret_cast<const bf16x8 *>(&Xs[piece][wm * 32 * WTM + 32 * tm + l32][kofs]);
#pragma unroll
                    for (int tn = 0; tn < WTN; tn++) g[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[tn], g[tm][tn], 0, 0, 0);
                }
            }
        }
        // every accumulator entry of a lane belongs to one output column: one scale per lane and tile column
#pragma unroll
        for (int tn = 0; tn < WTN; tn++) {
            const float sc = Ss[grp][wn * 32 * WTN + 32 * tn + l32];
#pragma unroll
            for (int tm = 0; tm < WTM; tm++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[tm][tn][e] = fmaf(g[tm][tn][e], sc, acc[tm][tn][e]);
        }
        }
        __syncthreads();
    }

    if constexpr (KS > 1) {
        // add the sets' sums: every set but the first parks its accumulators in the (no longer read) piece buffers
        float *red = reinterpret_cast<float *>(lds);                // [KS - 1][4 wavefronts][WTM*WTN*16][64 lanes]
        if (kset > 0) {
#pragma unroll
            for (int i = 0; i < WTM; i++)
#pragma unroll
                for (int j = 0; j < WTN; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        red[((((kset - 1) * 4 + wave) * WTM * WTN + i * WTN + j) * 16 + e) * 64 + lane] = acc[i][j][e];
        }
        __syncthreads();
        if (kset > 0) return;
#pragma unroll
        for (int ks = 1; ks < KS; ks++)
#pragma unroll
            for (int i = 0; i < WTM; i++)
#pragma unroll
                for (int j = 0; j < WTN; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        acc[i][j][e] += red[((((ks - 1) * 4 + wave) * WTM * WTN + i * WTN + j) * 16 + e) * 64 + lane];
    }

    // epilogue: acc[i][jn][e] is C[32*i + 8*(e/4) + 4*(lane/32) + e%4][32*jn + lane%32] of the wavefront's block
    if (split_k > 0) {
        float *slab = partial + (int64_t)blockIdx.z * M * N;
#pragma unroll
        for (int jn = 0; jn < WTN; jn++) {
            const int col = n0 + wn * 32 * WTN + 32 * jn + l32;
            if (col >= N) continue;
#pragma unroll
            for (int i = 0; i < WTM; i++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int row = m0 + wm * 32 * WTM + 32 * i + 8 * (e >> 2) + 4 * half + (e & 3);
                    if (row < M) slab[(int64_t)row * N + col] = acc[i][jn][e];
                }
        }
        return;
    }
#pragma unroll
    for (int jn = 0; jn < WTN; jn++) {
        const int col = n0 + wn * 32 * WTN + 32 * jn + l32;
        if (col >= N) continue;
        float badd = 0.0f;
        if (ep.bias) badd = ep.interleaved_bias ? ((col & 1) ? ep.bias2[col >> 1] : ep.bias[col >> 1]) : ep.bias[col];
#pragma unroll
        for (int i = 0; i < WTM; i++) {
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int row = m0 + wm * 32 * WTM + 32 * i + 8 * (e >> 2) + 4 * half + (e & 3);
                if (ep.swiglu) {
                    // gate and up of one output sit in neighbouring lanes (columns 2j, 2j + 1); N is even, so a
                    // pair is inside or outside the matrix together (SiLU.java:20-24, SwiGLULayer.java:69)
                    float v = acc[i][jn][e];
                    if (ep.bias) v = v + badd;
                    const float other = __shfl_xor(v, 1, 64);
                    if (row < M && (col & 1) == 0) {
                        const float sg = v * (1.0f / (1.0f + expf(-v)));
                        C[(int64_t)row * (N >> 1) + (col >> 1)] = sg * other;
                    }
                    continue;
                }
                if (row < M) {
                    float v = acc[i][jn][e];
                    if (ep.bias) v = v + badd;
                    if (ep.gelu) v = gemm_gelu(v);
                    if (ep.residual) v = ep.residual[(int64_t)row * N + col] + v;
                    C[(int64_t)row * N + col] = v;
                }
            }
        }
    }
}

// C = epilogue(sum over the splits of partial[z]) for the K-sharing launches of k_gemm_q8 and k_gemm_q8_rows: the same bias / GELU /
// residual / SwiGLU steps, in the same order, as the kernel's own epilogue (a fixed order of additions, so a run
// repeats bit for bit - which adding into C with atomics would not).  One thread per column pair of a row.
__global__ void __launch_bounds__(256) k_sum_partials_q8(const float *__restrict__ partial, float *__restrict__ C, int splits,
                                                        int M, int N, GemmEpilogue ep) {
    const int64_t pairs = (int64_t)M * (N >> 1), mn = (int64_t)M * N;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < pairs; i += (int64_t)gridDim.x * 256) {
        const int row = (int)(i / (N >> 1)), col = (int)(i % (N >> 1)) * 2;
        const int64_t at = (int64_t)row * N + col;
        float2 v = *reinterpret_cast<const float2 *>(partial + at);
        for (int z = 1; z < splits; z++) {
            const float2 p = *reinterpret_cast<const float2 *>(partial + (int64_t)z * mn + at);
            v.x += p.x; v.y += p.y;
        }
        if (ep.bias) {
            if (ep.interleaved_bias) { v.x = v.x + ep.bias[col >> 1]; v.y = v.y + ep.bias2[col >> 1]; }
            else { v.x = v.x + ep.bias[col]; v.y = v.y + ep.bias[col + 1]; }
        }
        if (ep.swiglu) {                        // SiLU.java:20-24, SwiGLULayer.java:69
            const float sg = v.x * (1.0f / (1.0f + expf(-v.x)));
            C[(int64_t)row * (N >> 1) + (col >> 1)] = sg * v.y;
            continue;
        }
        if (ep.gelu) { v.x = gemm_gelu(v.x); v.y = gemm_gelu(v.y); }
        if (ep.residual) {
            const float2 r = *reinterpret_cast<const float2 *>(ep.residual + at);
            v.x = r.x + v.x; v.y = r.y + v.y;
        }
        *reinterpret_cast<float2 *>(C + at) = v;
    }
}

constexpr int kFewTiles = 512, kGroupsFew = 4, kSetsFew = 4;
constexpr int kSetsBig = 1;
constexpr int kGroupsSmall = 2, kGroupsBig = 1;    // measured: 4 and 2 are slower (LDS per workgroup, registers)

// The large tile needs enough workgroups to fill the chip; small problems keep the 64 x 64 tile.
inline bool use_big_tile(int m, int n) {
    return m >= 128 && n >= 128 && (int64_t)((m + BM2 - 1) / BM2) * ((n + BN2 - 1) / BN2) >= 256;
}

}  // namespace

namespace {
template <int TM, int TN, int KW, int U, int D>
void launch_matmul(hipStream_t s, const float *a, const float *b, float *out, int m, int n, int k) {
    const int tm = (m + 32 * TM - 1) / (32 * TM), tn = (n + 32 * TN - 1) / (32 * TN);
    if ((k & 3) == 0) launch_kernel((k_matmul<TM, TN, KW, U, D, true>), dim3(tm * tn), dim3(64 * KW), 0, s, a, b, out, m, n, k, tm, tn);
    else launch_kernel((k_matmul<TM, TN, KW, U, D, false>), dim3(tm * tn), dim3(64 * KW), 0, s, a, b, out, m, n, k, tm, tn);
}
void launch_matmul_16(hipStream_t s, const float *a, const float *b, float *out, int m, int n, int k) {
    const int tm = (m + 15) / 16, tn = (n + 15) / 16;
    if ((k & 3) == 0) launch_kernel((k_matmul_16<true>), dim3(tm * tn), dim3(1024), 0, s, a, b, out, m, n, k, tm, tn);
    else launch_kernel((k_matmul_16<false>), dim3(tm * tn), dim3(1024), 0, s, a, b, out, m, n, k, tm, tn);
}
template <int TM, int WC, int KS>
void launch_matmul_split(hipStream_t s, const float *a, const float *b, float *out, int m, int n, int k) {
    const int tm = (m + 32 * TM - 1) / (32 * TM), tn = (n + 32 * WC - 1) / (32 * WC);
    if ((k & 3) == 0) launch_kernel((k_matmul_split<TM, WC, KS, true>), dim3(tm * tn), dim3(64 * WC * KS), 0, s, a, b, out, m, n, k, tm, tn);
    else launch_kernel((k_matmul_split<TM, WC, KS, false>), dim3(tm * tn), dim3(64 * WC * KS), 0, s, a, b, out, m, n, k, tm, tn);
}
}  // namespace

// The kernel and tile of least estimated time, in us: fixed + weight of its rounds x (round + k x per_k), a round being a tile
// on each of the 256 compute units.  The first of every `fit` rounds (the workgroups that a compute unit holds; k_matmul: of all)
// weighs 1 and the others `more`: about 2 for k_matmul, two of whose workgroups on a compute unit are in each other's way.
// `odd`: the factor on per_k where words are loaded one by one (k, or for k_matmul_lds k or n, no multiple of 4).  k_matmul
// and k_matmul_lds were fitted to 980 shapes of 1 to 12000 rows and columns over 4 to 6000 k, some of them odd, k_matmul_split
// to 260 of 8 to 8000 over 32 to 6000; the choice takes 1.002 times the best one's time on average over the latter, 1.09 at
// worst, where the choice without k_matmul_split takes 1.043 and 1.94.  Its 32 x 96 tile is for outputs of half a million to
// 800 thousand values, which leave half of the chip idle in tiles of 64 rows and are several rounds of k_matmul's: 700 x 1024 x
// 2752 48 -> 41 us, 600 x 1100 x 512 14.0 -> 11.5, 148 x 4712 x 1396 28.8 -> 23.7; over 260 more shapes the choice with it is never
// slower and 1.05 to 1.22 times as fast for 20.
static int matmul_kernel(int m, int n, int k) {
    struct Shape { int rows, cols; double fixed, round, per_k, more; int fit; double odd; };
    static const Shape shapes[] = {{32, 32, 2.3, 0.15, 0.0061, 1.95, 0, 1.0},     // k_matmul
                                   {32, 64, 2.9, 0.2, 0.0101, 2.1, 0, 1.0},
                                   {64, 64, 3.6, 0.6, 0.0178, 1.6, 0, 1.0},
                                   {64, 64, 3.1, 2.0, 0.0177, 0.52, 3, 1.06},     // k_matmul_split
                                   {64, 96, 0.9, 5.1, 0.0156, 0.81, 1, 1.02},
                                   {96, 128, 0.0, 7.2, 0.029, 0.8, 1, 1.03},
                                   {128, 128, 0.0, 9.6, 0.0348, 0.8, 1, 1.06},
                                   {32, 96, 2.2, 3.7, 0.0119, 1.0, 2, 1.0},
                                   {64, 64, 1.8, 1.4, 0.032, 0.5, 4, 1.6}};       // k_matmul_lds
    constexpr int kSplit = 3, kLds = 8;
    // k_matmul and k_matmul_split address a tile's rows of A in 32 bits, k_matmul a stage's rows of B, k_matmul_split all of B
    const bool in_reach = (int64_t)k * 128 * 4 <= UINT32_MAX && (int64_t)n * 17 * 4 <= UINT32_MAX;
    const bool split_reach = in_reach && (int64_t)k * n * 4 <= INT32_MAX;
    int best = kLds;
    double least = -1.0;
    for (int i = in_reach ? 0 : kLds; i <= kLds; i++) {
        if (i >= kSplit && i < kLds && !split_reach) continue;
        const Shape &h = shapes[i];
        const int64_t tiles = (int64_t)((m + h.rows - 1) / h.rows) * ((n + h.cols - 1) / h.cols), rounds = (tiles + 255) / 256;
        const int64_t firsts = h.fit ? (rounds + h.fit - 1) / h.fit : 1;
        const double weight = (double)firsts + (double)(rounds - firsts) * h.more;
        const bool odd = i == kLds ? ((k | n) & 3) != 0 : (k & 3) != 0;
        const double t = h.fixed + weight * (h.round + h.per_k * k * (odd ? h.odd : 1.0));
        if (least < 0.0 || t < least) { least = t; best = i; }
    }
    return best;
}

void launch_matmul_f32(hipStream_t s, const float *a, const float *b, float *out, int m, int n, int k) {
    if (m <= 0 || n <= 0) return;
    if (k <= 0) { launch_fill(s, reinterpret_cast<uint32_t *>(out), 0u, (int64_t)m * n); return; }
    const int64_t blocks = (int64_t)((m + 31) / 32) * ((n + 31) / 32);
    switch (matmul_kernel(m, n, k)) {
        case 0:
            // a tile per compute unit at most: more wavefronts share its K, with shorter stages so that their lines fit; up to two
            // tiles of 16 x 16, those (768 of them: 8.5 us where 32 x 32 take 8.1 at 768 k; at 256 k and less all take about 4).  They
            // have no estimate of their own: where another tile's is below that of 32 x 32, it stays with that one.
            if (k > 256 && (int64_t)((m + 15) / 16) * ((n + 15) / 16) <= 512) launch_matmul_16(s, a, b, out, m, n, k);
            else if (blocks <= 256 && k > 256) launch_matmul<1, 1, 16, 1, 2>(s, a, b, out, m, n, k);
            else if (blocks <= 256) launch_matmul<1, 1, 8, 4, 2>(s, a, b, out, m, n, k);
            else launch_matmul<1, 1, 4, 4, 2>(s, a, b, out, m, n, k);
            break;
        case 1: launch_matmul<1, 2, 4, 1, 4>(s, a, b, out, m, n, k); break;
        case 2: launch_matmul<2, 2, 4, 1, 2>(s, a, b, out, m, n, k); break;
        case 3: launch_matmul_split<2, 2, 2>(s, a, b, out, m, n, k); break;
        case 4: launch_matmul_split<2, 3, 4>(s, a, b, out, m, n, k); break;
        case 5: launch_matmul_split<3, 4, 2>(s, a, b, out, m, n, k); break;
        case 6: launch_matmul_split<4, 4, 2>(s, a, b, out, m, n, k); break;
        case 7: launch_matmul_split<1, 3, 4>(s, a, b, out, m, n, k); break;
        default: {
            const int tn = (n + 63) / 64;
            launch_kernel(k_matmul_lds, dim3((m + 63) / 64 * tn), dim3(256), 0, s, a, b, out, m, n, k, tn);
        }
    }
}

// Few tiles over a long K: how many workgroups share a tile's K (1: none).  A 64 x 64 tile's workgroup (1024 threads,
// its four wavefront sets already dividing every 128-k step) streams 64 weight rows; with fewer such workgroups than
// compute units the launch is as long as one workgroup's walk through K (64 rows x 2048 x 2048: 32 workgroups, 23 us,
// for 4.7 MB of weights; 11 us as 8 x 32).  Shares of at least two steps; one workgroup per compute unit at most (a
// second round of workgroups costs what the shorter walk saves: 64 x 5632 x 2048 16.1 us with 176 workgroups, 18.7 with 352).
int q8_gemm_k_shares(int m, int n_rows, int k) {
    if (n_rows & 1) return 1;
    if (use_big_tile(m, n_rows)) return 1;
    const int64_t tiles = (int64_t)((n_rows + BN - 1) / BN) * ((m + BM - 1) / BM);
    const int steps = (q8_padded_k(k) + kQ8Group * kGroupsFew - 1) / (kQ8Group * kGroupsFew);
    if (tiles > 128 || steps < 4) return 1;
    int shares = (int)std::min<int64_t>(std::min<int64_t>(8, 256 / tiles), steps / 2);
    if (shares < 2) return 1;
    const int per = (steps + shares - 1) / shares;
    return (steps + per - 1) / per;
}

// Two 128 x 128 workgroups fit a CU, so the tiles run in rounds of 512; when the last round would be mostly
// empty (352 or 704 tiles), 64 x 128 tiles - twice as many, three to four per CU - finish sooner
// (512 x 11264 x 2048: 101 against 113 us; 1024 rows: 194 against 229 us).
static bool last_round_empty(int m, int n_rows) {
    const int64_t tiles = (int64_t)((n_rows + BN2 - 1) / BN2) * ((m + BM2 - 1) / BM2), rounds = (tiles + 511) / 512;
    return tiles * 100 < rounds * 512 * 85;
}

// Fitted to the launches below over 2 to 700 rows, 256 to 50257 columns and 256 to 11008 k, with the weights in the memory-side
// cache and from HBM: 5 % of the time on average.  A normalisation in front is a launch of its own.
Q8GemmEstimate q8_gemm_estimate(int m, int n_rows, int k, bool norm, bool may_share) {
    static constexpr GemmCost shared{5.83, 0.38, 8.95, 0.0, 0.34, 2.08, 0.0, 0.038}, few{5.08, 0.91, 8.37, 8.6, 1.73, 0.0, 0.0, 0.016},
                              many{0.0, 2.3, 13.4, 4.7, 2.6, 0.0, 0.0, 0.0}, wide{9.0, 0.9, 8.0, 4.6, 10.7, 0.0, 0.0, 0.17}, big{0.0, 9.1, 0.0, 5.9, 16.4, 0.0, 0.0, 0.9};
    const bool large = use_big_tile(m, n_rows), by64 = large && last_round_empty(m, n_rows);
    const int tm = large && !by64 ? BM2 : BM, tn = large ? BN2 : BN;
    const int64_t m_tiles = (m + tm - 1) / tm, tiles = m_tiles * ((n_rows + tn - 1) / tn);
    const int shares = may_share ? q8_gemm_k_shares(m, n_rows, k) : 1;
    const bool four_sets = !large && tiles <= kFewTiles;
    const GemmCost &c = by64 ? wide : large ? big : !four_sets ? many : shares > 1 ? shared : few;
    const int fit = by64 ? 3 : large ? 2 : !four_sets ? 4 : shares > 1 ? 1 : 2;         // workgroups on a compute unit
    constexpr int step = kQ8Group * kGroupsFew;
    const int steps = (q8_padded_k(k) + step - 1) / step;
    const double x = (double)tiles * shares / 256.0, kk = (steps + shares - 1) / shares * step * 1e-3;
    const double us = c.us(x, x <= fit ? ceil(x) : x, kk, (double)m / (double)(m_tiles * tm), m, n_rows, k, shares);
    return {us + (norm ? 2.2 + 4e-6 * m * k : 0.0), (four_sets ? kSetsFew : 1) * shares};
}

int64_t q8_gemm_workspace_floats(int m, int n_rows, int k) {
    const int shares = q8_gemm_k_shares(m, n_rows, k);
    return shares > 1 ? (int64_t)shares * m * n_rows : 0;
}

void launch_q8_sum_partials(hipStream_t s, const float *partial, float *out, int splits, int m, int n_rows, const GemmEpilogue &ep) {
    const int64_t pairs = (int64_t)m * (n_rows / 2);
    launch_kernel(k_sum_partials_q8, dim3((unsigned)std::min<int64_t>((pairs + 255) / 256, 4096)), dim3(256), 0, s, partial, out, splits, m, n_rows, ep);
}

// Q8 GEMM used by launch_q8_linear for M > 1.  n_rows is the number of Q8 rows
// (= output columns of this launch; 2N for an interleaved gate/up weight).  workspace: room for the partial products
// of a K-sharing launch (q8_gemm_workspace_floats), or less - then no K is shared.
void launch_q8_gemm(hipStream_t s, const float *x, const int8_t *wq, const float *scales, float *out, int m,
                    int k, int n_rows, const float *bias, const float *bias2, const float *residual,
                    int interleaved_bias, const int32_t *m_dev, int m_extra, int gelu, int swiglu, float *workspace,
                    int64_t workspace_floats, GemmChain *chain) {
    if (m <= 0 || n_rows <= 0) return;
    if (swiglu && ((n_rows & 1) || residual || gelu)) fail("q8_gemm: the SwiGLU epilogue needs an even row count and takes no residual or GELU");
    GemmEpilogue ep{bias, bias2, residual, interleaved_bias, m_dev, m_extra, gelu, swiglu};
    if (!m_dev && use_big_tile(m, n_rows)) {       // a device-side row count is usually far below m: keep small tiles
        dim3 grid2((n_rows + BN2 - 1) / BN2, (m + BM2 - 1) / BM2);
        if (last_round_empty(m, n_rows)) {
            dim3 gridw(grid2.x, (m + 63) / 64);
            launch_kernel((k_gemm_q8<1, 2, 2, 1>), gridw, dim3(256), 0, s, x, wq, scales, out, m, n_rows, k, q8_padded_k(k), ep, 0, nullptr);
            return;
        }
        launch_kernel((k_gemm_q8<2, 2, kGroupsBig, kSetsBig>), grid2, dim3(256 * kSetsBig), 0, s, x, wq, scales, out, m, n_rows, k, q8_padded_k(k), ep, 0, nullptr);
        return;
    }
    dim3 grid((n_rows + BN - 1) / BN, (m + BM - 1) / BM);
    const int shares = m_dev ? 1 : q8_gemm_k_shares(m, n_rows, k);
    if (shares > 1 && workspace && workspace_floats >= (int64_t)shares * m * n_rows) {
        constexpr int step = kQ8Group * kGroupsFew;
        const int steps = (q8_padded_k(k) + step - 1) / step, per = (steps + shares - 1) / shares;
        grid.z = shares;
        launch_kernel((k_gemm_q8<1, 1, kGroupsFew, kSetsFew>), grid, dim3(256 * kSetsFew), 0, s, x, wq, scales, out, m, n_rows, k, q8_padded_k(k), ep,
                      per * step, workspace);
        if (chain && chain->next_pieces && !gelu && !swiglu && !interleaved_bias && split_operand_sum_ok(n_rows)) {
            launch_split_operand_sum(s, workspace, shares, bias, residual, out, chain->next_gamma, chain->next_beta, chain->next_pieces, m, n_rows);
            chain->left_pieces = true;
        } else {
            launch_q8_sum_partials(s, workspace, out, shares, m, n_rows, ep);
        }
        return;
    }
    // few tiles (about one per CU): a workgroup brings its own second wavefront per SIMD
    if ((int64_t)grid.x * grid.y <= kFewTiles)
        launch_kernel((k_gemm_q8<1, 1, kGroupsFew, kSetsFew>), grid, dim3(256 * kSetsFew), 0, s, x, wq, scales, out, m, n_rows, k, q8_padded_k(k), ep, 0, nullptr);
    else
        launch_kernel((k_gemm_q8<1, 1, kGroupsSmall, 1>), grid, dim3(256), 0, s, x, wq, scales, out, m, n_rows, k, q8_padded_k(k), ep, 0, nullptr);
}

}  // namespace dj
