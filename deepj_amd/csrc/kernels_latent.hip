// Decode attention over a latent KV cache (DeepSeek, MultiHeadLatentAttention.java:92-123) without expanding the cache.
//
// The cache holds cKV rows [kvRank]; a token's attention needs K = RoPE(cKV.Wuk) and V = cKV.Wuv of every cached position.
// One workgroup per (head, key split) takes tiles of 32 cached rows: their values as three bf16 pieces (exact), the head's
// 32 x hd block of K from the bf16 matrix cores as in k_gemm_q8, rotated and multiplied with the query in the accumulators -
// the rotation moved to the query's side, score = sum of ka (q0 cos + q1 sin) + kb (q1 cos - q0 sin) - and the probabilities
// then weigh the LATENT rows.  The value projection is linear, so it is applied once, to the weighted sum of all splits:
// sum_j p_j (cKV_j.Wuv) = (sum_j p_j cKV_j).Wuv, by the launch that merges the splits.  Neither K nor V reaches memory.
//
// Bound: the latency of one round of loads and of the chain behind it (16 heads of 128, kvRank 512, 300 rows: state 0.5 us,
// loads 1.5, the products of a tile 2.7, scores and soft-max 1.5, the row's sum 0.4, with a start and an end of a launch).  So
// everything is asked for at once - the rotation's words too - and in whole lines (weights, scales and rows through LDS; a row a
// lane straight into registers, 32 lines a load, took 12000 cycles where this takes 4900); a wavefront takes an eighth of K and
// all columns, so that a row's pieces are made in the registers that the products read and the row is there when its
// probability is; and the sums over lanes take no LDS.  Back to back with the merge, and before (pieces of the rows in LDS, read by the
// wavefronts of every column tile, Wuv applied by every split): 16 x 128, 512, at 300 rows 11.3 us, 16.4; at 1000
// 17.2, 22.8; 20 x 64, 512, 700 13.2, 17.6; 40 x 32, 256, 600 12.5, 16.2; 4 x 32, 32, 100 7.9, 9.0; 24 greedy tokens of a 4-layer
// model of width 2048 at 300 rows 4915 -> 4429.  Without gain: the column tiles unrolled, by two or four, and their conversions
// and scalings placed between the matrix instructions (11.5 to 11.8).
// Error against float64 (2-norm, over kvRank 32 to 512 and 40 to 700 rows): 1.1 to 1.9e-7; 1.6 to 2.1e-7 before.
#include "dj_common.h"
#include "dj_device.h"
#include "gemm_rows.h"
#include <algorithm>
#include <type_traits>

namespace dj {
namespace {

using namespace dev;

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 512, kWaves = kThreads / 64, kTile = 32;
// pitch of a column's factors: 16-byte words of 32 columns in different banks
constexpr int kFactorPitch = kTile + 4;
constexpr int kMergeThreads = 256, kMergeColumns = 16;           // of k_latent_values: its workgroup, the values it makes

__device__ __forceinline__ uint32_t pack_hi(float a, float b) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302);
}
__device__ __forceinline__ float top_bits(float x) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & 0xffff0000u); }

template <int N> using FloatV = float __attribute__((ext_vector_type(N)));

// 64 lanes x 16 bytes from each lane's address into LDS bytes [dst, dst + 1024), lane order (as load_to_lds16, gemm_rows.h)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_to_lds16_from(const float *from, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(from) : "memory", "m0");
}
#pragma clang diagnostic pop

struct Pieces { float hi, mid, lo; };        // bf16 values with hi + mid + lo == x
__device__ __forceinline__ Pieces split(float x) {
    const float h = top_bits(x), r = x - h, m = top_bits(r);
    return {h, m, r - m};
}
__device__ __forceinline__ bf16x8 weights_of(int a, int b) {      // eight int8 weights as bf16 (exact)
    const int r[2] = {a, b};
    uint32_t w[4];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        w[2 * q] = pack_hi((float)(int8_t)(r[q] & 0xff), (float)(int8_t)((r[q] >> 8) & 0xff));
        w[2 * q + 1] = pack_hi((float)(int8_t)((r[q] >> 16) & 0xff), (float)(int8_t)(r[q] >> 24));
    }
    return __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
}

// Exchanges inside the 32 lanes of a half, without LDS
template <int CTRL> __device__ __forceinline__ float from_partner(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
// the first 16 lanes' a beside their neighbours', and theirs of b: what is added to get sums of a there and of b here
__device__ __forceinline__ void swap_16(float a, float b, float &x, float &y) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
    x = __builtin_bit_cast(float, (uint32_t)r[0]); y = __builtin_bit_cast(float, (uint32_t)r[1]);      // (a bit cast of r[1] itself takes element 0)
}
template <typename Op> __device__ __forceinline__ float over_32(float v, Op op) {
    v = op(v, from_partner<0xB1>(v));                           // quad_perm [1,0,3,2]
    v = op(v, from_partner<0x4E>(v));                           // quad_perm [2,3,0,1]
    v = op(v, from_partner<0x141>(v));                          // row_half_mirror
    v = op(v, from_partner<0x140>(v));                          // row_mirror
    float x, y;
    swap_16(v, v, x, y);
    return op(x, y);
}
__device__ __forceinline__ float max_over_32(float v) { return over_32(v, [](float a, float b) { return fmaxf(a, b); }); }
__device__ __forceinline__ float sum_over_32(float v) { return over_32(v, [](float a, float b) { return a + b; }); }
// v[0..N), N 16 or 32, added up over the 32 lanes of a half: lane l32 returns the sum of v[l32 % N].  A step halves the values:
// a lane keeps the half that its bit of the lane number names and hands the other to its partner.
template <int N> __device__ __forceinline__ float scattered_sum(const FloatV<N> &v, int l32) {
    float a[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        float x, y;
        swap_16(v[i], v[i + N - 16], x, y);
        a[i] = x + y;
    }
    auto step = [&](auto ctrl, auto count, bool upper) __attribute__((always_inline)) {
        constexpr int C = decltype(ctrl)::value, n = decltype(count)::value;
#pragma unroll
        for (int i = 0; i < n; i++) {
            const float keep = upper ? a[i + n] : a[i], give = upper ? a[i] : a[i + n];
            a[i] = keep + from_partner<C>(give);
        }
    };
    step(std::integral_constant<int, 0x128>{}, std::integral_constant<int, 8>{}, (l32 & 8) != 0);      // lane ^ 8: row_ror:8
    step(std::integral_constant<int, 0x141>{}, std::integral_constant<int, 4>{}, (l32 & 4) != 0);      // lane ^ 7: row_half_mirror
    step(std::integral_constant<int, 0x4E>{}, std::integral_constant<int, 2>{}, (l32 & 2) != 0);       // lane ^ 2: quad_perm [2,3,0,1]
    step(std::integral_constant<int, 0xB1>{}, std::integral_constant<int, 1>{}, (l32 & 1) != 0);       // lane ^ 1: quad_perm [1,0,3,2]
    return a[0];
}

// NT: 32-wide column tiles of a head; NG: scale groups (32 k) a wavefront takes of every row, all columns of it.
// Weights and rows go global -> LDS in whole lines, and from there to operands: a weight's 16 bytes are one half (lane / 32)
// of a group, its first eight k meet the first product, the other eight the second, and a lane's half of its row's group is
// read in the same order.  Groups behind the last one are rows of zeros: a wavefront's products have no branch between them.
template <int NT, int NG> struct LatentLds {
    static constexpr int HD = 32 * NT, kSlices = NG * kWaves / 4;                  // slices of 128 k: a line of a weight row
    static constexpr int weights = 0, rows = weights + kSlices * HD * 128;         // [slice][column][128]; [group][row][128]
    static constexpr int scales = rows + NG * kWaves * kTile * 128;                // [column][groups]
    static constexpr int factors = scales + HD * NG * kWaves * 4;                  // [column][kFactorPitch]
    static constexpr int bytes = factors + HD * kFactorPitch * 4;
};

template <int NT, int NG>
__global__ void __launch_bounds__(kThreads) k_latent_decode(const float *__restrict__ q, const float *__restrict__ ckv, float *latent,
                                                            const int8_t *__restrict__ wq, const float *__restrict__ scales,
                                                            const int32_t *__restrict__ state, const float *__restrict__ cos_t,
                                                            const float *__restrict__ sin_t, float *__restrict__ records, int head0, int rank,
                                                            int max_seq, float scale) {
    using L = LatentLds<NT, NG>;
    constexpr int HD = L::HD, KMAX = NG * kWaves * kQ8Group, NV = 16 * NG;         // NV: values of its tile row a lane holds
    extern __shared__ __align__(16) unsigned char lds[];
    float *s_f = reinterpret_cast<float *>(lds + L::factors);   // what K's column meets in the key's score
    __shared__ __align__(16) float s_part[kWaves][kTile];       // scores: a wavefront's part

    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), half = lane >> 5, l32 = lane & 31;
    const int h = head0 + blockIdx.x, split_i = blockIdx.y, splits = gridDim.y, record = (int)blockIdx.x * splits + split_i;
    float *rec = records + (int64_t)record * KMAX;
    float *ml = records + (int64_t)gridDim.x * splits * KMAX + 2 * record;
    const int groups = (rank + kQ8Group - 1) / kQ8Group, kp = groups * kQ8Group;
    const uint32_t lds_at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds);

    const int at_state = state[0];                              // (asked for first: the rows' addresses hang on it)
    // Loads of eight columns (rows) by 128 bytes: lane l takes 16 bytes of column l / 8, and piece p goes to position p ^ (column % 8)
    // so that the lanes that read a piece of 32 columns meet different banks.  All addresses stay inside: pieces past a row's
    // end are its first again (they meet zeros).
    const int piece = (lane & 7) ^ (lane >> 3);
    const int8_t *w_head = wq + (int64_t)h * HD * kp;
#pragma unroll
    for (int i = 0; i < NG * NT; i++) {
        const int unit = wave + kWaves * i, slice = unit / (HD / 8), col = unit % (HD / 8) * 8 + (lane >> 3);
        const int at = slice * 128 + piece * 16;
        if (slice * 128 < kp) load_to_lds16(w_head, (uint32_t)(col * kp + (at < kp ? at : 0)), lds_at + L::weights + unit * 1024);
    }
    const int scale_bytes = HD * groups * 4;
#pragma unroll
    for (int i = 0; i < (HD * NG * 4 + 1023) / 1024; i++) {
        const int at = (wave + kWaves * i) * 1024;
        if (at < scale_bytes) load_to_lds16(scales + (int64_t)h * HD * groups, (uint32_t)std::min(at + lane * 16, scale_bytes - 16), lds_at + L::scales + at);
    }
    const int pos = at_state < 0 ? 0 : (at_state >= max_seq ? max_seq - 1 : at_state);     // reads stay inside; nothing is appended outside
    const int tiles = pos / kTile + 1;
    if (split_i >= tiles) {                                     // no keys for this split
        if (t == 0) { ml[0] = -INFINITY; ml[1] = 0.0f; }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // (what was asked for lands before the LDS is another workgroup's)
        return;
    }
    // a wavefront's groups of the tile's rows, for itself alone; the new token's row is not in the cache yet
    const int g0 = wave * NG;
    auto fetch_rows = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NG; i++) {
            if (g0 + i >= groups) break;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int key = tile * kTile + 8 * j + (lane >> 3), k = (g0 + i) * kQ8Group + piece * 4;
                const float *src = key >= pos ? ckv : latent + (int64_t)key * rank;
                load_to_lds16_from(src + (k < rank ? k : 0), lds_at + L::rows + (g0 + i) * (kTile * 128) + j * 1024);
            }
        }
    };
    fetch_rows(split_i);
    // the factors this thread makes: of key t / 16 of the tile, for the column pairs t % 16 + 16 i
    const int f_key = t >> 4, f_pair = t & 15;
    float cs[NT], sn[NT], q0[NT], q1[NT];
    auto load_rotation = [&](int tile) __attribute__((always_inline)) {
        const int key = tile * kTile + f_key < pos ? tile * kTile + f_key : pos;
        const uint32_t at = ((uint32_t)key * (HD / 2) + (uint32_t)f_pair) * 4u;                  // bytes: a 32-bit offset to a scalar base
#pragma unroll
        for (int i = 0; i < NT; i++) {
            cs[i] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(cos_t) + at + 64 * i);
            sn[i] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(sin_t) + at + 64 * i);
        }
    };
    load_rotation(split_i);
    {
        float2 v[NT];
        float pc[NT], ps[NT];
#pragma unroll
        for (int i = 0; i < NT; i++) {
            const int64_t at = (int64_t)pos * (HD / 2) + f_pair + 16 * i;
            v[i] = *reinterpret_cast<const float2 *>(q + h * HD + 2 * (f_pair + 16 * i));
            pc[i] = cos_t[at]; ps[i] = sin_t[at];
        }
        __builtin_amdgcn_sched_barrier(0);                      // all of them are asked for before one is waited for
#pragma unroll
        for (int i = 0; i < NT; i++) { q0[i] = v[i].x * pc[i] - v[i].y * ps[i]; q1[i] = v[i].x * ps[i] + v[i].y * pc[i]; }
    }

    float m_run = -INFINITY, l_run = 0.0f;
    FloatV<NV> sum = 0.0f;                                      // this lane's values, weighted, over the tiles
    for (int tile = split_i; tile < tiles; tile += splits) {
        const int key0 = tile * kTile;
#pragma unroll
        for (int i = 0; i < NT; i++) {
            float *f = s_f + 2 * (f_pair + 16 * i) * kFactorPitch + f_key;
            f[0] = q0[i] * cs[i] + q1[i] * sn[i];
            f[kFactorPitch] = q1[i] * cs[i] - q0[i] * sn[i];
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // this tile's rows and, for the first, the weights
        FloatV<NV> c;                                           // this lane's values of its tile row l32: of group g0 + i the 16 of its half
#pragma unroll
        for (int m = 0; m < 4 * NG; m++) {
            const int k = (g0 + (m >> 2)) * kQ8Group + half * 16 + (m & 3) * 4;
            const float4 v = *reinterpret_cast<const float4 *>(lds + L::rows + (g0 + (m >> 2)) * (kTile * 128) + l32 * 128 + (((4 * half + (m & 3)) ^ (l32 & 7)) << 4));
            c[4 * m] = k < rank ? v.x : 0.f; c[4 * m + 1] = k < rank ? v.y : 0.f; c[4 * m + 2] = k < rank ? v.z : 0.f; c[4 * m + 3] = k < rank ? v.w : 0.f;
        }
        const int k0 = g0 * kQ8Group + half * 16;
        lds_barrier();                                          // (also: these reads are done, and the previous tile's scores have been read)
        if (tile + splits < tiles) { fetch_rows(tile + splits); load_rotation(tile + splits); }
        bf16x8 rows[NG][2][3];                                  // [group][step][piece]
#pragma unroll
        for (int i = 0; i < NG; i++)
#pragma unroll
            for (int step = 0; step < 2; step++) {
                uint32_t w[3][4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const Pieces a = split(c[16 * i + 8 * step + 2 * j]), b = split(c[16 * i + 8 * step + 2 * j + 1]);
                    w[0][j] = pack_hi(a.hi, b.hi); w[1][j] = pack_hi(a.mid, b.mid); w[2][j] = pack_hi(a.lo, b.lo);
                }
#pragma unroll
                for (int piece = 0; piece < 3; piece++)
                    rows[i][step][piece] = __builtin_bit_cast(bf16x8, make_uint4(w[piece][0], w[piece][1], w[piece][2], w[piece][3]));
            }
        if (h == 0 && key0 + l32 == at_state && at_state == pos) {   // head 0 appends the new token's row (nobody reads it from the cache in this launch)
#pragma unroll
            for (int m = 0; m < 4 * NG; m++) {
                const int k = k0 + (m >> 2) * kQ8Group + (m & 3) * 4;
                if (k < rank) *reinterpret_cast<float4 *>(latent + (int64_t)pos * rank + k) = make_float4(c[4 * m], c[4 * m + 1], c[4 * m + 2], c[4 * m + 3]);
            }
        }

        // a score is a sum over columns and k: a wavefront adds up its k of all columns
        FloatV<16> s = 0.0f;
#pragma unroll 1
        for (int ct = 0; ct < NT; ct++) {
            floatx16 g[NG];
            float sk[NG];
#pragma unroll
            for (int i = 0; i < NG; i++) {
                const int group = g0 + i;
                const int4 w = *reinterpret_cast<const int4 *>(lds + L::weights + ((group >> 2) * HD + ct * 32 + l32) * 128 + (((2 * (group & 3) + half) ^ (l32 & 7)) << 4));
                const float of_group = *reinterpret_cast<const float *>(lds + L::scales + ((ct * 32 + l32) * groups + (group < groups ? group : 0)) * 4);
                sk[i] = group < groups ? of_group : 0.0f;
#pragma unroll
                for (int e = 0; e < 16; e++) g[i][e] = 0.0f;
#pragma unroll
                for (int step = 0; step < 2; step++) {
                    const bf16x8 b = step ? weights_of(w.z, w.w) : weights_of(w.x, w.y);
#pragma unroll
                    for (int piece = 0; piece < 3; piece++) g[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rows[i][step][piece], b, g[i], 0, 0, 0);
                }
            }
            // g[i][e] is K[8 (e / 4) + 4 half + e % 4][column], this group's part of it
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++) {
                const float4 f = *reinterpret_cast<const float4 *>(s_f + (ct * 32 + l32) * kFactorPitch + 8 * e4 + 4 * half);
                const float fe[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float k = g[0][4 * e4 + j] * sk[0];
                    if constexpr (NG > 1) k = fmaf(g[NG - 1][4 * e4 + j], sk[NG - 1], k);
                    s[4 * e4 + j] = fmaf(k, fe[j], s[4 * e4 + j]);
                }
            }
        }
        const float s_own = scattered_sum<16>(s, l32);
        if (l32 < 16) s_part[wave][8 * (l32 >> 2) + 4 * half + (l32 & 3)] = s_own;
        lds_barrier();

        // every wavefront for itself: lane l32 has the score of key key0 + l32, and that key's row
        float sp[4] = {0.0f, 0.0f, 0.0f, 0.0f};                 // (short chains: fewer roundings, and fewer waits)
#pragma unroll
        for (int i = 0; i < kWaves; i++) sp[i & 3] += s_part[i][l32];
        float score = ((sp[0] + sp[1]) + (sp[2] + sp[3])) * scale;
        if (key0 + l32 > pos) score = -INFINITY;
        const float m_new = fmaxf(m_run, max_over_32(score));
        const float p = __builtin_amdgcn_exp2f(score - m_new), corr = __builtin_amdgcn_exp2f(m_run - m_new);
        l_run = l_run * corr + p;                               // this lane's key's share of it
        m_run = m_new;
#pragma unroll
        for (int i = 0; i < NV; i++) sum[i] = fmaf(p, c[i], sum[i] * corr);
    }

    // the weighted row: over the tile's 32 rows, one a lane
    const float v = scattered_sum<NV>(sum, l32);
    if (NG == 2 || l32 < 16) rec[(g0 + (NG == 2 ? l32 >> 4 : 0)) * kQ8Group + half * 16 + (l32 & 15)] = v;
    if (wave == 0) {
        l_run = sum_over_32(l_run);
        if (t == 0) { ml[0] = m_run; ml[1] = l_run; }
    }
}

// out = (sum_z w_z row_z / sum_z w_z l_z) . Wuv over the splits' records, w_z = exp2(m_z - max m) (the maxima are in base-2
// units); a split without keys left m = -inf, l = 0.  A workgroup per head and 16 of its values: every one adds up the head's
// records anew (from L2), so that the values' weights are read by as many workgroups as there are.  Weights and records are
// asked for together.  (16 heads of 128 at 300 rows: 4.5 us, as merging the splits' values alone took.)
template <int NG>
__global__ void __launch_bounds__(kMergeThreads) k_latent_values(const float *__restrict__ records, int splits, const int8_t *__restrict__ wq, const float *__restrict__ scales,
                                                                 float *__restrict__ out, int head0, int hd, int rank, int d) {
    constexpr int KMAX = NG * kWaves * kQ8Group, PT = KMAX / kMergeThreads, PL = KMAX / 64, kColumns = kMergeColumns / (kMergeThreads / 64);
    __shared__ __align__(16) float s_row[KMAX];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l32 = lane & 31;
    const int groups = (rank + kQ8Group - 1) / kQ8Group, kp = groups * kQ8Group;
    const int col0 = (head0 + blockIdx.x) * hd + blockIdx.y * kMergeColumns + wave * kColumns;
    const int k_at = lane * PL < kp ? lane * PL : 0;             // (behind the last group the row is zero)
    int w[kColumns][PL / 4];
    float sc[kColumns];
#pragma unroll
    for (int i = 0; i < kColumns; i++) {
        const int64_t row = d + col0 + i;
#pragma unroll
        for (int j = 0; j < PL / 4; j++) w[i][j] = reinterpret_cast<const int *>(wq + row * kp + k_at)[j];
        sc[i] = scales[row * groups + k_at / kQ8Group];
    }
    const float *rec = records + (int64_t)blockIdx.x * splits * KMAX;
    const float *ml = records + ((int64_t)gridDim.x * KMAX + 2 * (int64_t)blockIdx.x) * splits;
    const float2 own = *reinterpret_cast<const float2 *>(ml + 2 * (l32 < splits ? l32 : 0));
    float x[PT];
#pragma unroll
    for (int j = 0; j < PT; j++) x[j] = 0.0f;
    const float m = l32 < splits ? own.x : -INFINITY;
    const float weight = __builtin_amdgcn_exp2f(m - max_over_32(m));
    const float total = sum_over_32(m != -INFINITY ? own.y * weight : 0.0f);
    for (int z0 = 0; z0 < splits; z0 += 16) {
        float v[16][PT];
#pragma unroll
        for (int z = 0; z < 16; z++)
#pragma unroll
            for (int j = 0; j < PT; j++) v[z][j] = rec[(int64_t)(z0 + z < splits ? z0 + z : z0) * KMAX + t * PT + j];
#pragma unroll
        for (int z = 0; z < 16; z++) {
            const int from = z0 + z < splits ? z0 + z : 31;
            const float wz = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, weight), from));
            const bool has = z0 + z < splits && __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), from)) != -INFINITY;
#pragma unroll
            for (int j = 0; j < PT; j++) x[j] = has ? fmaf(wz, v[z][j], x[j]) : x[j];
        }
    }
#pragma unroll
    for (int j = 0; j < PT; j++) s_row[t * PT + j] = x[j];
    lds_barrier();
    float r[PL];
#pragma unroll
    for (int j = 0; j < PL; j++) r[j] = lane * PL < kp ? s_row[lane * PL + j] : 0.0f;
#pragma unroll
    for (int i = 0; i < kColumns; i++) {
        float o = 0.0f;
#pragma unroll
        for (int j = 0; j < PL; j++) o = fmaf((float)(int8_t)(w[i][j / 4] >> (8 * (j & 3))), r[j], o);
        o = wave_sum_dpp(o * sc[i]);
        if (lane == 0) out[col0 + i] = o / total;
    }
}

constexpr int kRankMax = 512;                                   // what a thread can hold of a tile row and of the weights

constexpr int kHeadsAtOnce = 256;                               // heads of a launch: what bounds the records

template <int NT, int NG>
void launch(hipStream_t s, const LatentDecode &a, int splits) {
    for (int head0 = 0; head0 < a.heads; head0 += kHeadsAtOnce) {
        const int heads = a.heads - head0 < kHeadsAtOnce ? a.heads - head0 : kHeadsAtOnce;
        launch_kernel((k_latent_decode<NT, NG>), dim3(heads, splits), dim3(kThreads), (size_t)LatentLds<NT, NG>::bytes, s, a.q, a.ckv, a.latent, a.wq, a.scales, a.state, a.cos_t, a.sin_t,
                      a.records, head0, a.rank, a.max_seq, a.scale);
        launch_kernel(k_latent_values<NG>, dim3(heads, a.hd / kMergeColumns), dim3(kMergeThreads), 0, s, (const float *)a.records, splits, a.wq, a.scales, a.out, head0,
                      a.hd, a.rank, a.heads * a.hd);
    }
}
template <int NT>
void launch_rank(hipStream_t s, const LatentDecode &a, int splits) {
    if (q8_padded_k(a.rank) / kQ8Group <= kWaves) launch<NT, 1>(s, a, splits);
    else launch<NT, 2>(s, a, splits);
}
template <int NT, int NG>
void configure() {
    hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(k_latent_decode<NT, NG>), hipFuncAttributeMaxDynamicSharedMemorySize, LatentLds<NT, NG>::bytes),
              "hipFuncSetAttribute(k_latent_decode)");
}

}  // namespace

// more LDS than a kernel gets without asking; once per device at start-up (the first launch may sit inside a capture)
void latent_decode_configure() {
    configure<1, 1>(); configure<1, 2>(); configure<2, 1>(); configure<2, 2>(); configure<4, 1>(); configure<4, 2>();
}

// Key splits per head: workgroups for every compute unit, no more than there are tiles, and no more records than the merge
// reads in passing.  0: not a shape of this kernel (rows are read as float4s; a lane holds its share of a row).
int latent_decode_splits(int heads, int hd, int rank, int max_seq) {
    if (heads <= 0 || max_seq <= 0 || (hd != 32 && hd != 64 && hd != 128)) return 0;
    if (rank <= 0 || (rank & 3) || rank > kRankMax) return 0;
    if (max_seq > (1 << 23) || heads > (1 << 13)) return 0;     // 32-bit offsets into the rotation tables and the weight
    const int by_chip = 256 / heads, tiles = (max_seq + kTile - 1) / kTile;
    const int n = by_chip < 1 ? 1 : (by_chip > 32 ? 32 : by_chip);
    return n < tiles ? n : tiles;
}

// Scratch: of every head of a launch and split the weighted latent row, the largest score and the sum of the weights
int64_t latent_decode_scratch_floats(int heads, int hd, int rank, int max_seq) {
    const int64_t kmax = q8_padded_k(rank) > 256 ? 512 : 256;
    return (kmax + 2) * std::min(heads, kHeadsAtOnce) * latent_decode_splits(heads, hd, rank, max_seq);
}

void launch_latent_decode(hipStream_t s, LatentDecode a) {
    const int splits = latent_decode_splits(a.heads, a.hd, a.rank, a.max_seq);
    if (!splits) fail("latent_decode: shape outside this kernel's range");
    a.scale = (float)(1.4426950408889634 / sqrt((double)a.hd));        // scores in base 2
    switch (a.hd) {
        case 32: launch_rank<1>(s, a, splits); break;
        case 64: launch_rank<2>(s, a, splits); break;
        default: launch_rank<4>(s, a, splits); break;
    }
}

}  // namespace dj
