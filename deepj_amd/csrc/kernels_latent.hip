// Decode attention over a latent KV cache (DeepSeek, MultiHeadLatentAttention.java:92-123) without expanding the cache.
//
// The cache holds cKV rows [kvRank]; a token's attention needs K = RoPE(cKV.Wuk) and V = cKV.Wuv of every cached position.
// One workgroup per (head, key split) takes tiles of 32 cached rows: the rows go to LDS as three bf16 pieces (exact), the
// head's 32 x hd block of K comes out of the bf16 matrix cores as in k_gemm_q8, is rotated and multiplied with the query in
// the accumulators - the rotation moved to the query's side, score = sum of ka (q0 cos + q1 sin) + kb (q1 cos - q0 sin) -
// and the probabilities then weigh the LATENT rows, which a thread still has in registers.  The value projection is linear,
// so it is applied once, to the weighted sum: sum_j p_j (cKV_j.Wuv) = (sum_j p_j cKV_j).Wuv.  Neither K nor V reaches memory.
//
// Bound: the latency of one round of loads (the head's Q8 rows of Wuk and Wuv, 2 * hd * 1.125 * kvRank bytes, and 32 rows
// of 4 * kvRank bytes, all requested up front) and the chain behind it; a tile's 32 x hd x kvRank x 3 products are
// 0.7 us of one compute unit.  d 2048, 16 heads, kvRank 512, 300 cached rows: append, expansion, two rotations and
// attention took 38 us in five launches, this and the merge of the splits 21 (24 greedy tokens of a 4-layer model: 6.8 -> 5.04 ms).
// Error against float64 (2-norm, over kvRank 32 to 512 and 40 to 1000 rows): 1.5 to 2.2e-7, the five launches' 1.7 to 2.3e-7.
#include "dj_common.h"
#include "dj_device.h"

namespace dj {
namespace {

using namespace dev;

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 512, kWaves = kThreads / 64, kTile = 32;
// bf16 values of a piece plane's row: 8 more than it holds, so that the 32 rows a product reads start in different banks
constexpr int row_pitch(int kmax) { return kmax + 8; }

__device__ __forceinline__ uint32_t pack_hi(float a, float b) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302);
}
__device__ __forceinline__ float top_bits(float x) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & 0xffff0000u); }

// Operands a lane holds for the whole kernel, walked by loops that stay loops (a register is picked by a scalar index): with
// every loop unrolled the kernel was 14 KB of code, which a launch fetches anew, spilled registers, and took 21 us, not 16.
template <int N> using FloatV = float __attribute__((ext_vector_type(N)));
template <int N> using IntV = int __attribute__((ext_vector_type(N)));

struct Pieces { float hi, mid, lo; };        // bf16 values with hi + mid + lo == x
__device__ __forceinline__ Pieces split(float x) {
    const float h = top_bits(x), r = x - h, m = top_bits(r);
    return {h, m, r - m};
}
__device__ __forceinline__ float max_over_32(float v) {
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
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

// NT: 32-wide column tiles of a head; the eight wavefronts form 8 / NT sets that share K, of up to NG scale groups each.
// A lane's 16-byte weight load is one half (lane / 32) of a group; its first eight k meet the first product, the other eight
// the second, and the activations are read in the same order.  Groups behind the last one are zero rows in LDS and a zero
// scale: a wavefront's products have no branch between them, so the next group's reads and conversions run beside them.
// S4: the scale groups are a multiple of four, and so a lane takes its row's (a line of its own) four at a time.
template <int NT, int NG, bool S4>
__global__ void __launch_bounds__(kThreads) k_latent_decode(const float *__restrict__ q, const float *__restrict__ ckv, float *latent,
                                                            const int8_t *__restrict__ wq, const float *__restrict__ scales,
                                                            const int32_t *__restrict__ state, const float *__restrict__ cos_t,
                                                            const float *__restrict__ sin_t, float *__restrict__ records, int rank, int d,
                                                            int max_seq, float scale) {
    constexpr int HD = 32 * NT, KS = kWaves / NT;
    constexpr int KMAX = NG * KS * kQ8Group;                    // widest latent row
    constexpr int kScales = NG < 2 ? 2 : NG;
    constexpr int NM = KMAX / 64;                               // float4s of its tile row a thread holds (16 threads a row)
    constexpr int PITCH = row_pitch(KMAX), PLANE = kTile * PITCH;
    extern __shared__ __align__(16) uint16_t lds[];             // [3 pieces][kTile][PITCH]; then [kTile][KMAX] floats
    __shared__ __align__(16) float s_part[2 * kWaves][kTile];   // scores: a partial sum per 16 columns
    __shared__ __align__(16) uint16_t s_sum[3][KMAX];           // pieces of the weighted latent row
    __shared__ float s_out[kWaves][32];

    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), half = lane >> 5, l32 = lane & 31;
    const int h = blockIdx.x, split_i = blockIdx.y, splits = gridDim.y;
    float *rec = records + ((int64_t)h * splits + split_i) * (HD + 4);
    const int groups = (rank + kQ8Group - 1) / kQ8Group, kp = groups * kQ8Group;

    const int ct = wave % NT, kset = wave / NT;
    const int g0 = kset * NG;                                             // this set's first group
    const int col = ct * 32 + l32;                                        // column within the head
    IntV<4 * NG> wk, wv;
    FloatV<kScales> sk, sv;
    // 32-bit offsets to scalar bases: an address pair per load would not leave the registers for what is loaded
    auto load_weights = [&](uint32_t row, IntV<4 * NG> &w, FloatV<kScales> &sc) {
        const uint32_t at = row * (uint32_t)kp + half * 16u, at_s = row * (uint32_t)groups * 4u;
#pragma unroll
        for (int i = 0; i < NG; i++) {
            const int g = g0 + i < groups ? g0 + i : 0;
            const int4 v = *reinterpret_cast<const int4 *>(reinterpret_cast<const char *>(wq) + g * kQ8Group + at);
            w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
        }
        if constexpr (S4) {
#pragma unroll
            for (int i = 0; i < NG; i += 4) {
                const bool ok = g0 + i < groups;
                const float4 v = *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(scales) + (ok ? g0 + i : 0) * 4 + at_s);
                sc[i] = ok ? v.x : 0.f; sc[i + 1] = ok ? v.y : 0.f; sc[i + 2] = ok ? v.z : 0.f; sc[i + 3] = ok ? v.w : 0.f;
            }
        } else {
#pragma unroll
            for (int i = 0; i < NG; i++) {
                const bool ok = g0 + i < groups;
                const float v = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(scales) + (ok ? g0 + i : 0) * 4 + at_s);
                sc[i] = ok ? v : 0.f;
            }
        }
    };
    load_weights((uint32_t)(h * HD + col), wk, sk);
    // (the weights are on their way while the position is waited for)
    const int at_state = state[0];
    const int pos = at_state < 0 ? 0 : (at_state >= max_seq ? max_seq - 1 : at_state);     // reads stay inside; nothing is appended outside
    const int tiles = pos / kTile + 1;
    if (split_i >= tiles) {                                     // no keys for this split
        if (t == 0) { rec[0] = -INFINITY; rec[1] = 0.0f; }
        return;
    }
    // the tile rows this thread stages: row t / 16, float4s (t % 16) + 16 m; the new token's row is not in the cache yet
    const int s_row = t >> 4, s_at = (t & 15) * 4;
    FloatV<4 * NM> c;
    auto load_rows = [&](int tile) {
        const int key = tile * kTile + s_row;
        int at0 = s_at;
        asm volatile("" : "+v"(at0));                           // offsets are worked out anew: kept over the tiles they cost registers that are not there
        const float *src = key >= pos ? ckv : latent + (int64_t)key * rank;
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const float4 v = *reinterpret_cast<const float4 *>(src + (at0 + 64 * m < rank ? at0 + 64 * m : 0));
            c[4 * m] = v.x; c[4 * m + 1] = v.y; c[4 * m + 2] = v.z; c[4 * m + 3] = v.w;
        }
    };
    load_rows(split_i);

    // Wuv's rows are multiplied last; beside Wuk's they do not fit the registers, so for now a word of each of their lines
    // is asked for, which brings the lines to this chiplet's L2
    const int v_line = t * 128 < HD * kp ? t * 128 : 0;
    const int warm = *reinterpret_cast<const int *>(wq + (int64_t)(d + h * HD) * kp + v_line);
    // this lane's share of the rotated query: score += k (qc cos + qs sin) for its column of K before the rotation
    float qc, qs;
    {
        const int64_t at = (int64_t)pos * (HD / 2) + (col >> 1);
        const float2 v = *reinterpret_cast<const float2 *>(q + h * HD + (col & ~1));
        const float cs = cos_t[at], sn = sin_t[at];
        const float q0 = v.x * cs - v.y * sn, q1 = v.x * sn + v.y * cs;
        qc = (col & 1) ? q1 : q0;
        qs = (col & 1) ? -q0 : q1;
    }

    // acc += rows . weights over this wavefront's groups; row r of the 32 comes from base + r * pitch of each piece plane
    auto product = [&](const uint16_t *base, int pitch, int plane, const IntV<4 * NG> &w, const FloatV<kScales> &sc, floatx16 &acc) {
        constexpr int U = NG < 2 ? NG : 2;
        const uint16_t *p = base + l32 * pitch + g0 * kQ8Group + half * 16;
#pragma unroll 1
        for (int i = 0; i < NG; i += U, p += U * kQ8Group) {
            floatx16 g[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
#pragma unroll
                for (int e = 0; e < 16; e++) g[u][e] = 0.0f;
#pragma unroll
                for (int step = 0; step < 2; step++) {
                    const bf16x8 b = weights_of(w[4 * (i + u) + 2 * step], w[4 * (i + u) + 2 * step + 1]);
#pragma unroll
                    for (int piece = 0; piece < 3; piece++)
                        g[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8 *>(p + u * kQ8Group + piece * plane + step * 8), b, g[u], 0, 0, 0);
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const float v = sc[i + u];
#pragma unroll
                for (int e = 0; e < 16; e++) acc[e] = fmaf(g[u][e], v, acc[e]);
            }
        }
    };

    float m_run = -INFINITY, l_run = 0.0f;
    FloatV<4 * NM> sum = 0.0f;                                  // this thread's tile row, weighted, over the tiles

    for (int tile = split_i; tile < tiles; tile += splits) {
        const int key0 = tile * kTile;
        if (tile != split_i) load_rows(tile);
        // the rotation of this lane's 16 rows, requested before the rows are waited for
        float cs[16], sn[16];
        int pair = col >> 1;
        asm volatile("" : "+v"(pair));
#pragma unroll
        for (int e = 0; e < 16; e++) {
            int key = key0 + 8 * (e >> 2) + 4 * half + (e & 3);
            key = key < pos ? key : pos;
            const uint32_t at = ((uint32_t)key * (HD / 2) + (uint32_t)pair) * 4u;            // bytes: a 32-bit offset to a scalar base
            cs[e] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(cos_t) + at);
            sn[e] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(sin_t) + at);
        }
        float f[16];
#pragma unroll
        for (int e = 0; e < 16; e++) f[e] = qc * cs[e] + qs * sn[e];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
        for (int m = 0; m < NM; m++) {
            const bool in = s_at + 64 * m < rank;
            const Pieces a = split(in ? c[4 * m] : 0.f), b = split(in ? c[4 * m + 1] : 0.f);
            const Pieces e = split(in ? c[4 * m + 2] : 0.f), g = split(in ? c[4 * m + 3] : 0.f);
            uint16_t *dst = lds + s_row * PITCH + s_at + 64 * m;
            *reinterpret_cast<uint2 *>(dst) = make_uint2(pack_hi(a.hi, b.hi), pack_hi(e.hi, g.hi));
            *reinterpret_cast<uint2 *>(dst + PLANE) = make_uint2(pack_hi(a.mid, b.mid), pack_hi(e.mid, g.mid));
            *reinterpret_cast<uint2 *>(dst + 2 * PLANE) = make_uint2(pack_hi(a.lo, b.lo), pack_hi(e.lo, g.lo));
        }
        if (h == 0 && key0 + s_row == at_state) {                    // head 0 appends the new token's row (nobody reads it from the cache in this launch)
#pragma unroll 1
            for (int m = 0; m < NM; m++)
                if (s_at + 64 * m < rank)
                    *reinterpret_cast<float4 *>(latent + (int64_t)pos * rank + s_at + 64 * m) = make_float4(c[4 * m], c[4 * m + 1], c[4 * m + 2], c[4 * m + 3]);
        }
        lds_barrier();                                          // (and the previous tile's scores have been read)

        floatx16 acc;
#pragma unroll
        for (int e = 0; e < 16; e++) acc[e] = 0.0f;
        product(lds, PITCH, PLANE, wk, sk, acc);
        // acc[e] is K[8 (e / 4) + 4 half + e % 4][col], this set's part of it
#pragma unroll
        for (int e4 = 0; e4 < 4; e4++) {
            float s[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int e = 4 * e4 + j;
                s[j] = group_sum<16>(acc[e] * f[e]);
            }
            if ((lane & 15) == 0)
                *reinterpret_cast<float4 *>(&s_part[2 * wave + ((lane >> 4) & 1)][8 * e4 + 4 * half]) = make_float4(s[0], s[1], s[2], s[3]);
        }
        lds_barrier();

        // every wavefront for itself: lane l32 has the score of key key0 + l32
        float sp[4] = {0.0f, 0.0f, 0.0f, 0.0f};                 // (short chains: fewer roundings, and fewer waits)
#pragma unroll
        for (int i = 0; i < 2 * kWaves; i++) sp[i & 3] += s_part[i][l32];
        float s = ((sp[0] + sp[1]) + (sp[2] + sp[3])) * scale;
        if (key0 + l32 > pos) s = -INFINITY;
        const float m_new = fmaxf(m_run, max_over_32(s));
        const float p = __builtin_amdgcn_exp2f(s - m_new), corr = __builtin_amdgcn_exp2f(m_run - m_new);
        float ps = p;
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) ps += __shfl_xor(ps, o, 64);
        l_run = l_run * corr + ps;
        m_run = m_new;
        const float p_row = __shfl(p, s_row & 31, 64);
#pragma unroll
        for (int i = 0; i < 4 * NM; i++) sum[i] = fmaf(p_row, c[i], sum[i] * corr);
    }

    asm volatile("" :: "v"(warm));
    load_weights((uint32_t)(d + h * HD + col), wv, sv);
    // the weighted row: the tile rows' sums are added up through the bytes the pieces have left (every wavefront is behind
    // its last product: the barrier behind the scores)
    float *rows = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int m = 0; m < NM; m++)
        *reinterpret_cast<float4 *>(rows + s_row * KMAX + s_at + 64 * m) =
            s_at + 64 * m < rank ? make_float4(sum[4 * m], sum[4 * m + 1], sum[4 * m + 2], sum[4 * m + 3]) : make_float4(0.f, 0.f, 0.f, 0.f);
    lds_barrier();
    for (int at = t; at < KMAX; at += kThreads) {
        float part[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int r = 0; r < kTile; r += 8) {
#pragma unroll
            for (int i = 0; i < 8; i++) part[i] += rows[(r + i) * KMAX + at];
        }
        const float v = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
        const Pieces a = split(v);
        s_sum[0][at] = (uint16_t)(__builtin_bit_cast(uint32_t, a.hi) >> 16);
        s_sum[1][at] = (uint16_t)(__builtin_bit_cast(uint32_t, a.mid) >> 16);
        s_sum[2][at] = (uint16_t)(__builtin_bit_cast(uint32_t, a.lo) >> 16);
    }
    lds_barrier();
    floatx16 acc;
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = 0.0f;
    product(&s_sum[0][0], 0, KMAX, wv, sv, acc);                // one row, so all 32 of the product are the same
    if (half == 0) s_out[wave][l32] = acc[0];
    lds_barrier();
    if (t < HD) {
        float o = 0.0f;
#pragma unroll
        for (int k = 0; k < KS; k++) o += s_out[k * NT + (t >> 5)][t & 31];
        rec[4 + t] = o;
    }
    if (t == 0) { rec[0] = m_run; rec[1] = l_run; }
}

constexpr int kRankMax = 512;                                   // what a thread can hold of a tile row and of the weights

constexpr int pieces_bytes(int kmax) { return 3 * kTile * row_pitch(kmax) * 2; }

template <int NT, int NG, bool S4>
void launch_scales(hipStream_t s, const LatentDecode &a, int splits) {
    launch_kernel((k_latent_decode<NT, NG, S4>), dim3(a.heads, splits), dim3(kThreads), (size_t)pieces_bytes(NG * kWaves / NT * kQ8Group), s, a.q, a.ckv, a.latent,
                  a.wq, a.scales, a.state, a.cos_t, a.sin_t, a.records, a.rank, a.heads * a.hd, a.max_seq, a.scale);
}
template <int NT, int NG>
void launch(hipStream_t s, const LatentDecode &a, int splits) {
    if (NG % 4 == 0 && q8_padded_k(a.rank) / kQ8Group % 4 == 0) launch_scales<NT, NG, NG % 4 == 0>(s, a, splits);
    else launch_scales<NT, NG, false>(s, a, splits);
}
template <int NT>
void launch_rank(hipStream_t s, const LatentDecode &a, int splits) {
    constexpr int per256 = NT;                                  // groups per set and 256 latent values: 8 / (8 / NT)
    const int kp = q8_padded_k(a.rank);
    if (kp <= 256) launch<NT, per256>(s, a, splits);
    else launch<NT, 2 * per256>(s, a, splits);
}
template <int NT, int NG>
void configure() {
    constexpr int bytes = pieces_bytes(NG * kWaves / NT * kQ8Group);
    for (const void *kernel : {reinterpret_cast<const void *>(k_latent_decode<NT, NG, false>), reinterpret_cast<const void *>(k_latent_decode<NT, NG, NG % 4 == 0>)})
        hip_check(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes), "hipFuncSetAttribute(k_latent_decode)");
}
template <int NT>
void configure_head() { configure<NT, NT>(); configure<NT, 2 * NT>(); }

}  // namespace

// more LDS than a kernel gets without asking; once per device at start-up (the first launch may sit inside a capture)
void latent_decode_configure() { configure_head<1>(); configure_head<2>(); configure_head<4>(); }

// Key splits per head: workgroups for every compute unit, no more than there are tiles, and no more records than the merge
// reads in passing.  0: not a shape of this kernel (rows are read as float4s; the pieces of a tile have to fit the LDS).
int latent_decode_splits(int heads, int hd, int rank, int max_seq) {
    if (heads <= 0 || max_seq <= 0 || (hd != 32 && hd != 64 && hd != 128)) return 0;
    if (rank <= 0 || (rank & 3) || rank > kRankMax) return 0;
    if (max_seq > (1 << 23) || heads > (1 << 13)) return 0;     // 32-bit offsets into the rotation tables and the weight
    const int by_chip = 256 / heads, tiles = (max_seq + kTile - 1) / kTile;
    const int n = by_chip < 1 ? 1 : (by_chip > 32 ? 32 : by_chip);
    return n < tiles ? n : tiles;
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
    launch_attention_merge(s, a.records, a.out, a.heads, a.hd, splits);
}

}  // namespace dj
