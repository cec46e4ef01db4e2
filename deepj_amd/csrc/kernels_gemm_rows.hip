// Q8 GEMM for a batch of rows straight from the int8 weights: C[M x N] = X[M x K] . dequant(W)^T, W int8 [N x Kp] with one
// fp32 scale per 32 k.
//
// Arithmetic as in k_gemm_q8 (kernels_matmul.hip): an activation as three bf16 pieces that make it up exactly, the weights exact in
// bf16, three v_mfma_f32_32x32x16_bf16 per 16 k, the group scale on the finished 32-k sums.  The split happens once, in a launch
// in front that also normalises the rows (k_split_f16), where k_gemm_q8 does it anew for every column tile; the weights stay int8
// in memory and become bf16 in registers.  (Two fp16 pieces under one power of two a row, as the fp16 GEMM takes them, are a third
// less to read and multiply, 64 x 22016 over 4096 41 us, but 22 bits, and fewer for elements far below their row's largest: with one
// of 1e8 among values of about 1 that meets zero weights the error against 64 bits was 7e-5 of the result's rms, 9e-8 so.)
//
// A workgroup takes a tile of 32 TMW x 32 TNW and deals its K to four wavefronts in chunks of 128, one line of a weight row:
// no wavefront waits for another before the end, when their sums meet in LDS.  A wavefront asks for a chunk of its weights one
// chunk ahead, global -> LDS in whole lines, and for its activations NA pieces ahead, straight into registers in operand order;
// loads return in the order they were asked for, so waiting for activations that were asked for after a chunk is waiting for
// the chunk.  The matrix cores' 32 cycles a product hide the group before's scaling and the next one's conversion.
//
// Where the next product takes this one's output as it is (a feed-forward layer's hidden rows), its pieces come out of this
// epilogue (GemmRowsArgs::next), not out of a launch of their own; when that is worth it: rows_plan.
//
// What bounds it: up to 32 rows the weights' bytes (30 x 22016 over 4096: 94 MB in 34 us with the rows' normalisation and split, 42
// where they come from HBM, 87 and 90 on k_gemm_q8), then the activations, which every tile reads anew from L2 (12 KB for every
// 64 x 64 x 32: 64 x 22016 48 us, 53 from HBM, 86 and 92; 200 x 11264 over 2048 49 and 52, 66 and 67), and on small weights two
// launches' latency (30 x 2304 over 768 8.7 and 9.7 us, 13 and 12.6).
// Tried and slower, with two pieces: eight wavefronts a workgroup (two workgroups of four fill a compute unit better: 64 x 22016
// 54 us against 49), the K loop or the epilogue rolled (3 % and 10 %), a 64 x 64 tile whose wavefronts share the activations
// through LDS (latency of its reads and barriers: 400 x 768 over 3072 34 us against 22).
//
// Error against 64 bits, as a share of the result's rms: 0.77e-7 over 768 k, 0.81e-7 to 0.94e-7 over 2048, 0.94e-7 to 1.79e-7 over
// 11008, by the number of sums an output is dealt to (four wavefronts, NS sets in each, the workgroups that share K); 0.96e-7 to
// 1.88e-7 on k_gemm_q8.  No tile is taken that would do worse than k_gemm_q8 on the same product (rows_plan).  The error also
// hangs on the low pieces' products going first and on every second chunk's sign (operand_negated).
#include "dj_common.h"
#include <algorithm>
#include <cmath>
#include "gemm_epilogue.h"
#include "gemm_rows.h"

namespace dj {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kWaves = 4;
constexpr int NP = 2 * kOperandPieces, kGroupWords = NP * 64;       // products of a 32 x 32 tile and 32 k; 16-byte words of 32 rows' activations
constexpr int kChunk = kOperandChunk / kQ8Group;                   // scale groups a wavefront takes at a time: 128 k, one line of a weight row
constexpr int sum_sets(int tmw, int tnw) { return tmw * tnw > 4 ? 1 : 4 / (tmw * tnw); }       // sums a wavefront deals an output's groups to
constexpr int scale_row(int tnw) { return tnw > 2 ? 512 : 256; }
constexpr int slot_bytes(int tnw) { return 32 * tnw * 128 + kChunk * scale_row(tnw); }       // a wavefront's chunk in LDS: weights [column][128], scales [group][64 or 128]

struct GemmRowsArgs {
    const uintx4 *planes;        // activations in operand order (operand_at)
    const int8_t *wq;           // [n][kp]
    const float *scales;        // [n][groups]
    float *out;
    int m, n, groups;
    int m_tiles, n_tiles;       // tiles of the launched kernel's size
    GemmEpilogue ep;
    int share_chunks;           // > 0: gridDim.z workgroups share a tile's K, this many chunks each
    float *partial;             // [gridDim.z][m][n] when they do
    uint16_t *next;             // not null: where the next product takes this one's output as its rows, in operand order
    int next_groups;            // ... their scale groups, padded to whole chunks
};

// four int8 of a word as bf16, exactly
__device__ __forceinline__ void int8x4_to_bf16(uint32_t r, uint32_t &lo, uint32_t &hi) {
    auto pack = [](float a, float b) { return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302); };
    lo = pack((float)(int8_t)r, (float)(int8_t)(r >> 8));
    hi = pack((float)(int8_t)(r >> 16), (float)(int8_t)(r >> 24));
}

template <int TMW, int TNW>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(TNW > 2 ? 1 : 2, TNW > 2 ? 1 : 2))) k_gemm_q8_rows(const GemmRowsArgs a) {
    constexpr int TN = 32 * TNW, NL = TN / 8;          // NL: loads a wavefront makes for a chunk of its TN weight rows
    constexpr int kSlot = slot_bytes(TNW);
    extern __shared__ __align__(16) unsigned char lds[];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), half = lane >> 5, l32 = lane & 31;
    unsigned char *wl = lds + wave * 2 * kSlot;
    const uint32_t wl_at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)wl);
    // row tiles of a column tile on one XCD
    const int per_group = 8 * a.m_tiles, gi = (int)blockIdx.x / per_group, r = (int)blockIdx.x % per_group;
    const int n_tile = gi * 8 + (r & 7), m_tile = r >> 3;
    if (n_tile >= a.n_tiles) return;
    const int n0 = n_tile * TN, m0 = m_tile * 32 * TMW, kp = a.groups * kQ8Group;
    const int row_tiles = (a.m + 31) >> 5;

    const int chunks = (a.groups + kChunk - 1) / kChunk;
    const int c_begin = a.share_chunks > 0 ? (int)blockIdx.z * a.share_chunks : 0;
    const int c_end = a.share_chunks > 0 ? min(chunks, c_begin + a.share_chunks) : chunks;

    // All addresses stay inside: columns past N read the last row's weights, rows past M the zeros behind the last (or its tile
    // again), pieces past K the row's first again.
    // This lane's pieces of a chunk: 16 bytes of row 8 i + lane / 8.  Piece p of a row goes to position p ^ (row % 8).
    const int b_piece = ((lane & 7) ^ (lane >> 3)) * 16;
    const int8_t *b_base = a.wq + (int64_t)n0 * kp;
    const float *s_base = a.scales + (int64_t)n0 * a.groups;
    uint32_t b_off[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) b_off[i] = (uint32_t)min(8 * i + (lane >> 3), a.n - 1 - n0) * (uint32_t)kp + b_piece;
    // A column's scales of a chunk in one load of 16 bytes, to [column][4], where its row of them allows (groups a multiple of
    // four); else a load per group, to [group][column].  A load takes the address unit a cycle a line, and every column is a
    // line of its own: a group's scales cost it as much as 4 KB of activations (64 x 22016 over 4096 42.5 -> 41.0 us, 64 x 4096
    // over 11008 33.1 -> 31.0, 30 x 2048 over 2048 11.8 -> 11.1).
    constexpr int kScaleRow = scale_row(TNW);
    const bool scales4 = (a.groups & (kChunk - 1)) == 0;
    const int sc_col = scales4 ? 16 : 4, sc_group = scales4 ? 4 : kScaleRow, sc_at = l32 * sc_col;
    const uint32_t s_off = (uint32_t)min(min(lane, TN - 1), a.n - 1 - n0) * (uint32_t)a.groups * 4u;
    const uint32_t s_off2 = (uint32_t)min(min(64 + lane, TN - 1), a.n - 1 - n0) * (uint32_t)a.groups * 4u;
    const uint32_t q_at = l32 * 128, q_x = l32 & 7;
    const uintx4 *ap[TMW];
#pragma unroll
    for (int i = 0; i < TMW; i++) ap[i] = a.planes + (int64_t)min(m_tile * TMW + i, row_tiles - 1) * chunks * kChunk * kGroupWords;

    auto fetch_b = [&](int c, int slot) __attribute__((always_inline)) {
        const uint32_t back = c * (kChunk * kQ8Group) + b_piece < kp ? 0u : (uint32_t)b_piece;       // past the row's end: a piece that meets activations of zero
        const uint32_t dst = wl_at + slot * kSlot;
#pragma unroll
        for (int i = 0; i < NL; i++) load_to_lds16(b_base + (int64_t)c * (kChunk * kQ8Group), b_off[i] - back, dst + i * 1024);
        if (scales4) {
            load_to_lds16(s_base + c * kChunk, s_off, dst + TN * 128);
            if constexpr (TN > 64) load_to_lds16(s_base + c * kChunk, s_off2, dst + TN * 128 + 1024);
            return;
        }
#pragma unroll
        for (int g = 0; g < kChunk; g++) {
            const float *at = s_base + min(c * kChunk + g, a.groups - 1);
            load_to_lds4(at, s_off, dst + TN * 128 + g * kScaleRow);
            if constexpr (TN > 64) load_to_lds4(at, s_off2, dst + TN * 128 + g * kScaleRow + 256);
        }
    };
    // The activations come as a sequence of pieces, NP a group: low ones of the two k steps, middle ones, high ones.  NA of them
    // are in registers or on their way: as many as the registers of two wavefronts a SIMD leave room for, or of one where LDS has no
    // room for a second workgroup (96 columns).  24 instead of 12 where TMW is 1: 30 x 2304 over 768 9.2 us against 9.0; 8 instead
    // of 6 where it is 2: 128 x 50257 over 768 60 against 53, with registers spilled; 8 instead of 24 at 96 columns: 30 x 22016 over
    // 4096 37 against 33.
    constexpr int NA = TNW > 2 ? 24 : TMW == 1 ? 12 : 6;
    static_assert(kChunk * NP % NA == 0, "a piece's register is known at compile time");
    uintx4 av[TMW][NA];
    auto fetch_a = [&](int i, int q, int c) __attribute__((always_inline)) { return (ap[i] + ((int64_t)c * kChunk + q / NP) * kGroupWords)[64 * (kOperandPieces * (q & 1) + 2 - (q % NP >> 1)) + lane]; };
    constexpr int NS = sum_sets(TMW, TNW);             // a group's sum goes to set group % NS
    floatx16 acc[NS][TMW][TNW], p[2];
#pragma unroll
    for (int e = 0; e < 16; e++) {
#pragma unroll
        for (int i = 0; i < TMW; i++)
#pragma unroll
            for (int j = 0; j < TNW; j++)
#pragma unroll
                for (int z = 0; z < NS; z++) acc[z][i][j][e] = 0.0f;
        p[0][e] = p[1][e] = 0.0f;
    }
    uint32_t bw[2][8];                                 // [stage parity]: the weights of a stage (a column tile of a group) as bf16
    uintx4 qw[2];                                      // ... and as bytes, up to two stages ahead
    float sc[4] = {0.f, 0.f, 0.f, 0.f};                // their scales: of the stage before, this one and the two next
    auto read_q = [&](int slot, int g, int tn, int at, int at_sc) __attribute__((always_inline)) {
        sc[at_sc] = *reinterpret_cast<const float *>(wl + slot * kSlot + TN * 128 + sc_at + (g * sc_group + 32 * tn * sc_col));
        qw[at] = *reinterpret_cast<const uintx4 *>(wl + slot * kSlot + 4096 * tn + q_at + (((2 * g + half) ^ q_x) << 4));
    };
    int c = c_begin + wave, slot = 0;
    if (c < c_end) {
        fetch_b(c, 0);
#pragma unroll
        for (int q = 0; q < NA; q++)
#pragma unroll
            for (int i = 0; i < TMW; i++) av[i][q] = fetch_a(i, q, c);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NA * TMW) : "memory");
        read_q(0, 0, 0, 0, 1);
#pragma unroll
        for (int w = 0; w < 4; w++) int8x4_to_bf16(qw[0][w], bw[0][2 * w], bw[0][2 * w + 1]);
        read_q(0, 1 / TNW, 1 % TNW, 1, 2);
        constexpr int S = kChunk * TNW, kAhead = TNW == 1 ? 2 : 1;      // stages of a chunk; groups two stages reach ahead, whole or begun
#pragma unroll 1
        for (; c < c_end; c += kWaves, slot ^= 1) {
            const int next = min(c + kWaves, c_end - 1);
            fetch_b(next, slot ^ 1);
#pragma unroll
            for (int st = 0; st < S; st++) {
                const int g = st / TNW, tn = st % TNW;
                // two stages on is the next chunk: its weights were asked for before the activations of the groups since
                if (st == S - 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((4 - kAhead) * NP * TMW) : "memory");
                const uintx4 qn = qw[(st + 1) & 1];
                const int st2 = (st + 2) % S;
                read_q(st + 2 >= S ? slot ^ 1 : slot, st2 / TNW, st2 % TNW, st & 1, (st + 3) & 3);
#pragma unroll
                for (int tm = 0; tm < TMW; tm++) {
                    const int u = st * TMW + tm;
                    const int ptm = tm > 0 ? tm - 1 : TMW - 1, pst = tm > 0 ? st : (st + S - 1) % S, ptn = pst % TNW, pg = pst / TNW;
                    const float psc = tm > 0 ? sc[(st + 1) & 3] : sc[st & 3];
#pragma unroll
                    for (int j = 0; j < NP; j++) {
                        const int q = g * NP + j;
                        const uint32_t *w4 = bw[st & 1] + 4 * (j & 1);
                        p[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av[tm][q % NA]), __builtin_bit_cast(bf16x8, (uintx4){w4[0], w4[1], w4[2], w4[3]}),
                                                                           j == 0 ? (floatx16){} : p[u & 1], 0, 0, 0);
                        if (tn == TNW - 1) av[tm][q % NA] = q + NA < kChunk * NP ? fetch_a(tm, q + NA, c) : fetch_a(tm, q + NA - kChunk * NP, next);
                        // the sums of the tile before, and a share of the next stage's weights
#pragma unroll
                        for (int e = 0; e < 16; e++)
                            if (j == 1 + e / 4) acc[pg % NS][ptm][ptn][e] = fmaf(p[(u & 1) ^ 1][e], psc, acc[pg % NS][ptm][ptn][e]);
                        if (TMW == 1 ? j < 4 : (j & 1) == 0 && j < 4) {
                            const int w = TMW == 1 ? j : 2 * tm + j / 2;
                            int8x4_to_bf16(qn[w], bw[(st + 1) & 1][2 * w], bw[(st + 1) & 1][2 * w + 1]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 16; e++) acc[3 % NS][TMW - 1][TNW - 1][e] = fmaf(p[1][e], sc[0], acc[3 % NS][TMW - 1][TNW - 1][e]);
        if constexpr (NS > 1) {
#pragma unroll
            for (int i = 0; i < TMW; i++)
#pragma unroll
                for (int j = 0; j < TNW; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        acc[0][i][j][e] += acc[1][i][j][e];
                        if constexpr (NS == 4) acc[0][i][j][e] += acc[2][i][j][e] + acc[3][i][j][e];
                    }
        }
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the loads ahead of the last chunk have landed before LDS is used again
    // the wavefronts' sums, in a fixed order
    __syncthreads();
    float4 *red = reinterpret_cast<float4 *>(lds);
    constexpr int Q = TMW * TNW * 4;                   // runs of four rows of a lane
#pragma unroll
    for (int i = 0; i < TMW; i++)
#pragma unroll
        for (int j = 0; j < TNW; j++)
#pragma unroll
            for (int eq = 0; eq < 4; eq++)
                red[(wave * Q + (i * TNW + j) * 4 + eq) * 64 + lane] = make_float4(acc[0][i][j][4 * eq], acc[0][i][j][4 * eq + 1], acc[0][i][j][4 * eq + 2], acc[0][i][j][4 * eq + 3]);
    __syncthreads();
    const GemmEpilogue &ep = a.ep;
#pragma unroll 1
    for (int q = wave; q < Q; q += kWaves) {
        const int tile = q >> 2, eq = q & 3, tm = tile / TNW, tn = tile % TNW;
        const int row0 = m0 + 32 * tm + 8 * eq + 4 * half, col = n0 + 32 * tn + l32;
        if (m0 + 32 * tm + 8 * eq >= a.m) continue;    // wavefront-uniform
        float4 s = red[q * 64 + lane];
#pragma unroll
        for (int v = 1; v < kWaves; v++) {
            const float4 o = red[(v * Q + q) * 64 + lane];
            if ((v & 1) == 0) { s.x += o.x; s.y += o.y; s.z += o.z; s.w += o.w; }
            else { s.x -= o.x; s.y -= o.y; s.z -= o.z; s.w -= o.w; }
        }
        const float turn = c_begin & 1 ? -1.0f : 1.0f;
        s.x *= turn; s.y *= turn; s.z *= turn; s.w *= turn;
        const bool in = col < a.n;
        float badd = 0.0f;
        if (a.share_chunks == 0 && ep.bias && in) badd = ep.interleaved_bias ? ((col & 1) ? ep.bias2[col >> 1] : ep.bias[col >> 1]) : ep.bias[col];
#pragma unroll
        for (int row = row0; row < row0 + 4; row++) {  // (rolled: the steps below are most of a short launch's code)
            float v = s.x;
            s.x = s.y; s.y = s.z; s.z = s.w;
            const bool live = in && row < a.m;
            if (a.share_chunks > 0) {
                if (live) a.partial[((int64_t)blockIdx.z * a.m + row) * a.n + col] = v;
                continue;
            }
            if (ep.bias) v = v + badd;
            if (ep.swiglu) {
                // (gate, up) pairs in neighbouring lanes (SiLU.java:20-24, SwiGLULayer.java:69)
                const float other = __shfl_xor(v, 1, 64);
                v = v * (1.0f / (1.0f + expf(-v))) * other;
                if (live && (col & 1) == 0) a.out[(int64_t)row * (a.n >> 1) + (col >> 1)] = v;
            } else if (live) {
                if (ep.gelu) v = gemm_gelu(v);
                if (ep.residual) v = ep.residual[(int64_t)row * a.n + col] + v;
                a.out[(int64_t)row * a.n + col] = v;
            }
            s.w = v;                                   // (after four rows s holds the results)
        }
        if (a.next) red[q * 64 + lane] = s;            // (only this wavefront reads the place in the first wavefront's sums)
    }
    if (!a.next) return;
    // The tile's results as the next product's rows: two columns of a row a thread at a time (a loop of few instructions: a
    // launch fetches them anew).  What the tile has no result for - rows up to a multiple of 32, columns up to a whole chunk -
    // is zero.
    __syncthreads();
    constexpr int R = 32 * TMW;
    const int out_shift = ep.swiglu ? 1 : 0, n_out = a.n >> out_shift, c0 = n0 >> out_shift;
    const int columns = n_tile == a.n_tiles - 1 ? a.next_groups * kQ8Group - c0 : TN >> out_shift;
#pragma unroll 1
    for (int i = t; i < R * columns / 2; i += 64 * kWaves) {
        const int r32 = (i >> 2) % R, row = m0 + r32, at = i / (4 * R) * 8 + (i & 3) * 2, c = c0 + at;
        if (row >= row_tiles * 32) continue;
        const float *of_row = reinterpret_cast<const float *>(lds) + (((r32 >> 5) * TNW * 4 + ((r32 & 31) >> 3)) * 64 + ((r32 >> 2) & 1) * 32) * 4 + (r32 & 3);
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int local = (at + e) << out_shift;
            const float u = of_row[local < TN ? ((local >> 5) * 256 + (local & 31)) * 4 : 0];
            v[e] = row < a.m && c + e < n_out && local < TN ? (operand_negated(c) ? -u : u) : 0.0f;
        }
        uint32_t *dst = reinterpret_cast<uint32_t *>(a.next + operand_at(row, c, a.next_groups));
#pragma unroll
        for (int p = 0; p < kOperandPieces; p++) {
            const uint32_t w0 = __float_as_uint(v[0]) & 0xffff0000u, w1 = __float_as_uint(v[1]) & 0xffff0000u;
            dst[p * (kOperandPiece / 2)] = (w0 >> 16) | w1;
            v[0] -= __uint_as_float(w0); v[1] -= __uint_as_float(w1);
        }
    }
}

constexpr int lds_bytes(int tmw, int tnw) {
    const int stage = kWaves * 2 * slot_bytes(tnw), red = kWaves * tmw * tnw * 4096;
    return stage > red ? stage : red;
}

template <typename F> void each_kernel(F f) {
    f(k_gemm_q8_rows<1, 1>, 1, 1); f(k_gemm_q8_rows<1, 2>, 1, 2); f(k_gemm_q8_rows<2, 1>, 2, 1); f(k_gemm_q8_rows<2, 2>, 2, 2);
    f(k_gemm_q8_rows<1, 3>, 1, 3); f(k_gemm_q8_rows<2, 3>, 2, 3);
}

int chunks_of(int k) { return (q8_padded_k(k) / kQ8Group + kChunk - 1) / kChunk; }

// The tile and the sharing of K of least estimated time.  A column tile's row tiles lie on one XCD, so what counts is the tiles of
// the XCD that has most; two workgroups fit a compute unit, one where a tile is 96 columns wide (its lines take 112 KB of LDS).
// Fitted to the times of 2 to 700 rows, 256 to 50257 columns and 256 to 11008 k, weights from the memory-side cache and from HBM: the
// choice, k_gemm_q8 among it, takes 1.014 times the best one's time on average.  (200 x 2304 over 768: 32 x 32 12.4 us, 32 x 64
// 14.6; 64 x 22016 over 4096: 64 x 64 56 us, 64 x 96, whose 230 tiles are one round where 64 x 64 makes 344, 47; 64 x 4096 over 11008:
// 32 x 32 39, 32 x 64 with K shared by two 34.)
//
// No tile whose outputs would be worse than k_gemm_q8's: an output is `sums` sums of groups / sums terms each, and the squared error
// against 64 bits, in units of 1e-14 of the result's squared rms, was 0.55 + 0.031 a term here (768 to 11008 k, every tile) and 1.07 +
// 0.025 a term there.
//
// ready: the product in front leaves the rows' pieces, which saves a launch and its pass over the rows and costs that product's
// end up to 3 us a million values (64 x 11008 2.5, 400 x 3072 3.0).  Measured on that product and this one together, us: 64 x
// 4096 over 11008 80.9 -> 76.2, 30 x 4096 over 11008 60.7 -> 54.7, 30 x 2048 over 5632 32.3 -> 28.5, 16 x 256 over 688 15.8 ->
// 14.9; where k_gemm_q8 keeps the second one: 300 x 1024 over 2752 41.3, 43.2 with pieces, 400 x 768 over 3072 39.4, 42.7.
RowsPlan rows_plan(int m, int n_rows, int k, bool may_share, int sums_there, bool ready) {
    struct Shape { int tmw, tnw, shares; GemmCost cost; };
    static constexpr Shape shapes[] = {
        {1, 1, 1, {5.65, 0.2, 2.52, 2.03, 0.3, 0.0, 7.0, 0.075}},  {1, 2, 1, {6.46, 0.83, 3.59, 3.04, 0.0, 0.0, 6.5, 0.08}},
        {2, 1, 1, {6.24, 0.04, 3.76, 3.12, 0.85, 0.0, 8.7, 0.035}}, {2, 2, 1, {7.52, 1.04, 5.37, 4.49, 0.54, 0.0, 9.5, 0.045}},
        {1, 3, 1, {7.22, 3.37, 5.09, 5.28, 0.0, 0.0, 3.8, 0.03}},   {2, 3, 1, {9.13, 6.03, 6.36, 7.96, 0.0, 0.0, 7.9, 0.01}},
        {1, 1, 2, {7.39, 0.64, 2.86, 1.6, 0.25, 1.8, 6.7, 0.093}},  {1, 1, 4, {7.9, 0.43, 2.49, 0.34, 1.4, 1.86, 6.4, 0.12}},
        {2, 2, 2, {8.63, 0.11, 5.86, 4.19, 0.0, 3.25, 6.6, 0.1}},   {1, 2, 2, {7.96, 0.82, 3.95, 2.53, 0.0, 2.12, 5.8, 0.097}},
        {1, 2, 4, {8.46, 0.61, 4.2, 2.12, 0.0, 2.08, 6.4, 0.137}}};
    RowsPlan best{};
    const int chunks = chunks_of(k), groups = q8_padded_k(k) / kQ8Group;
    for (const Shape &h : shapes) {
        if (h.shares > 1 && (!may_share || (n_rows & 1) || chunks < 2 * h.shares)) continue;      // k_sum_partials_q8 takes columns in pairs
        const int sums = kWaves * sum_sets(h.tmw, h.tnw) * h.shares;
        if ((double)groups / sums > 16.0 + 0.75 * groups / sums_there) continue;
        const int64_t n_tiles = (n_rows + 32 * h.tnw - 1) / (32 * h.tnw), m_tiles = (m + 32 * h.tmw - 1) / (32 * h.tmw);
        const double x = (double)((n_tiles + 7) / 8 * m_tiles * h.shares) / 32.0;
        const int fit = h.tnw > 2 ? 1 : 2;
        const double rounds = x <= 2 * fit ? ceil(x) : fit * ceil(x / fit);
        const double kk = (((chunks + kWaves - 1) / kWaves + h.shares - 1) / h.shares) * kWaves * kChunk * kQ8Group * 1e-3;
        double us = h.cost.us(x, rounds, kk, 1.0, m, n_rows, k, h.shares);
        if (ready) us -= 2.5 + (h.cost.rows - 3.0) * m * k * 1e-6;
        if (!best.tmw || us < best.us) best = {h.tmw, h.tnw, h.shares, us};
    }
    return best;
}

}  // namespace

void q8_gemm_rows_configure() {
    each_kernel([](auto kernel, int tmw, int tnw) {
        hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes(tmw, tnw)), "hipFuncSetAttribute(k_gemm_q8_rows)");
    });
}

// What the fp16 GEMM does not take (fewer than 256 rows without a copy of the weights in its layout, few tiles, a short K) and
// k_gemm_q8 would take longer for, by both estimates: the split of the rows into pieces costs a launch, which takes the place of
// their normalisation where there is one (30 x 768 over 768 8.9 us against 10.8 on k_gemm_q8) and has to be made up for where there
// is none (30 x 6144 over 2048 12.1, 16.0, but 8 x 768 over 256 6.7, 6.2 and 128 x 768 over 3072 15.0, 12.1).  Up to 768 rows: long
// batches belong to k_gemm_q8's larger tiles (1500 x 50257 over 768 655 us, 504; 2048 rows 1058, 647; 1500 x 8001 over 1500 233, 158).  A
// lane's offset into a column tile's weights is 32 bits.
bool q8_gemm_rows_ok(int m, int n_rows, int k, bool norm, bool prepared, bool may_share, RowsPlan *plan, bool ready) {
    if (m > 768 || k > (1 << 24) || q8_gemm_f16_forced() == 0 || q8_gemm_f16_shape_ok(m, n_rows, k, prepared)) return false;
    const Q8GemmEstimate there = q8_gemm_estimate(m, n_rows, k, norm, may_share);
    const RowsPlan p = rows_plan(m, n_rows, k, may_share, there.sums, ready);
    if (plan) *plan = p;
    return p.tmw && (ready ? p.us < 1.01 * there.us : p.us < 0.98 * there.us - 0.2);
}

int64_t operand_floats(int m, int k) { return round_up(m, 32) * round_up(q8_padded_k(k), kOperandChunk) / 2 * kOperandPieces; }
// floats of workspace: the activations' pieces, the partial products where K is shared
int64_t q8_gemm_rows_workspace_floats(int m, int n_rows, int k, const RowsPlan &p) { return operand_floats(m, k) + (p.shares > 1 ? (int64_t)p.shares * m * n_rows : 0); }

void launch_q8_gemm_rows(hipStream_t s, const float *x, const float *gamma, const float *beta, const int8_t *wq, const float *scales, float *out, int m, int k,
                         int n_rows, const GemmEpilogue &ep, const RowsPlan &p, float *workspace, int64_t workspace_floats, GemmChain *chain) {
    if (workspace_floats < q8_gemm_rows_workspace_floats(m, n_rows, k, p)) fail("q8_gemm_rows: workspace too small");
    if (ep.swiglu && ((n_rows & 1) || ep.residual || ep.gelu)) fail("q8_gemm_rows: the SwiGLU epilogue needs an even row count and takes no residual or GELU");
    const int kp = q8_padded_k(k), ka = (int)round_up(kp, kOperandChunk), m_pad = (int)round_up(m, 32), n_out = ep.swiglu ? n_rows / 2 : n_rows;
    const int m_tiles = (m + 32 * p.tmw - 1) / (32 * p.tmw), n_tiles = (n_rows + 32 * p.tnw - 1) / (32 * p.tnw);
    uint16_t *planes = reinterpret_cast<uint16_t *>(workspace);
    float *w = workspace + operand_floats(m, k);
    if (!(chain && chain->pieces_ready)) launch_split_operand(s, x, gamma, beta, planes, m, m_pad, k, ka);      // (the product in front has left them: GemmChain)
    GemmRowsArgs a{reinterpret_cast<const uintx4 *>(planes), wq, scales, out, m, n_rows, kp / kQ8Group, m_tiles, n_tiles, ep, 0, nullptr, nullptr, 0};
    if (p.shares == 1 && chain && chain->next_pieces && !chain->next_gamma) {
        a.next = chain->next_pieces;
        a.next_groups = (int)round_up(q8_padded_k(n_out), kOperandChunk) / kQ8Group;
        chain->left_pieces = true;
    }
    dim3 grid((unsigned)((n_tiles + 7) / 8 * 8 * m_tiles));
    if (p.shares > 1) {
        a.share_chunks = (chunks_of(k) + p.shares - 1) / p.shares;
        grid.z = (chunks_of(k) + a.share_chunks - 1) / a.share_chunks;
        a.partial = w;
    }
    each_kernel([&](auto kernel, int tmw, int tnw) {
        if (tmw == p.tmw && tnw == p.tnw) launch_kernel(kernel, grid, dim3(64 * kWaves), (size_t)lds_bytes(tmw, tnw), s, a);
    });
    if (p.shares == 1) return;
    // (the next product's pieces may take the place of this one's, not of the partial products)
    const float *next = chain ? reinterpret_cast<const float *>(chain->next_pieces) : nullptr;
    if (next && chain->next_gamma && !ep.gelu && !ep.swiglu && !ep.interleaved_bias && split_operand_sum_ok(n_rows) &&
        (next + operand_floats(m, n_rows) <= w || next >= w + (int64_t)p.shares * m * n_rows)) {
        launch_split_operand_sum(s, w, (int)grid.z, ep.bias, ep.residual, out, chain->next_gamma, chain->next_beta, chain->next_pieces, m, n_rows);
        chain->left_pieces = true;
        return;
    }
    launch_q8_sum_partials(s, w, out, (int)grid.z, m, n_rows, ep);
}

}  // namespace dj
