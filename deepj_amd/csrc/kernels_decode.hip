// A decoder block for one token in two launches, for models up to 256 wide.
//
// At these widths a token is bound by what a dependent launch costs, not by its bytes: five launches a block (norm + q|k|v,
// attention, merge + output projection, norm + gate/up, down) of 2.6 to 5.6 us each, of which 1.4 us are the launch and
// about 1 us the trip that the previous launch's result makes through memory.  Here a launch carries its result one
// product further than a row can be finished by one workgroup:
//   k_decode_attn  one workgroup per head: the head's q | k | v rows, RoPE, the cache append, attention over the head's
//                  keys, and the product of the head's output with ITS columns of Wo - a partial sum of the block's row
//   k_decode_ffn   one workgroup per kFfnUnits hidden units: gate/up (or up), the activation, and their columns of the
//                  down projection - again a partial sum
// and every workgroup of the next launch adds the partial sums (H or dff / 64 rows of d floats, from L2) on its way into the
// norm.  One of them writes the finished row back: it is the residual two launches on.  The sums are taken in a fixed
// order, so runs repeat bit for bit.
//
// Inside a workgroup of 8 wavefronts the first four fetch and add the partial sums while the other four send the weights
// straight to LDS (whole rows, so that a load instruction reads consecutive memory; a matrix-core operand read straight
// from memory touches 16 rows an instruction, four times the L1 lookups).  The 16-byte chunks of a row are rotated by
// its index so that the operand reads - 16 rows at one k - use all banks.
//
// Products.  Weights stay int8 and go to v_mfma_i32_16x16x64_i8 as they are stored: a lane's 16 bytes are 16 consecutive k of
// its column.  The activations of 32 k (a scale group) are an integer times a power of two, in four signed-byte digits (29
// bits below the group's largest value - more than fp32 holds of it).  The instruction's 16 rows of A carry the digits of
// the two groups of its 64 k apart: rows 0, 1, 4, 5 the first group's (zero in the second group's k), rows 8, 9, 12, 13 the
// second's.  So a lane ends up with two digits' exact integer sums of one column and one group: 2 conversions, 3
// multiply-adds per 1024 weights and wavefront.
#include "dj_common.h"
#include "dj_device.h"
#include "gemm_epilogue.h"

namespace dj {
namespace {
using namespace dev;

typedef int intx4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512, kWaves = 8, kRowWaves = 4;
constexpr int kMaxD = 256;                 // a wavefront holds a row, float4 a lane
constexpr int kPitch = kMaxD + 16;         // of the row's digit planes
constexpr float kLog2e = 1.44269504088896340736f;

// ── activations ─────────────────────────────────────────────────────────────
// acc += the products of 16 columns (the lane's: four quarters of 16 k each) with 64 staged k
__device__ __forceinline__ float multiply_step(intx4 w, float scale, const uint8_t *planes, int pitch, const float *unit, int step, int lane, float acc) {
    const int r = lane & 15, quarter = lane >> 4;
    // this lane's row of A: digit plane (r & 1) | (r & 4) / 2 of the group r / 8; in the other group's k the row is zero
    intx4 v = *reinterpret_cast<const intx4 *>(planes + ((r & 1) | ((r >> 1) & 2)) * pitch + step * 64 + quarter * 16);
    v = (r >> 3) == (quarter >> 1) ? v : (intx4){0, 0, 0, 0};
    const intx4 c = __builtin_amdgcn_mfma_i32_16x16x64_i8(v, w, (intx4){0, 0, 0, 0}, 0, 0, 0);
    // C rows 4 quarter + e: digits 2 (quarter & 1) + e of group quarter / 2
    const float u = unit[step * 2 + (quarter >> 1)] * ((quarter & 1) ? 65536.0f : 1.0f);
    return fmaf(fmaf((float)c[1], u * 256.0f, (float)c[0] * u), scale, acc);
}

// ── weights straight to LDS ─────────────────────────────────────────────────
// M0 holds the LDS address of lane 0; the statement sets it and says so.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void to_lds16(const void *base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void to_lds4(const void *base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ uint32_t lds_address(const void *p) { return (uint32_t)(uintptr_t)p; }

// chunk c of row r of n chunks lies at chunk (c + rotation) mod n
__device__ __forceinline__ int rotation(int r, int n) { return r & (n >= 8 ? 7 : 1); }

// `rows` consecutive rows of n = d / 16 chunks to LDS rows l0 .. (l0 a multiple of 8), by kWaves - kRowWaves wavefronts
__device__ __forceinline__ void rows_to_lds(const int8_t *src, int rows, int n, uint8_t *lds, int l0, int wave, int lane) {
    const int per = 64 / n, in = lane / n, p = lane - in * n;
    const uint32_t base = lds_address(lds) + l0 * n * 16;
    for (int r0 = wave * per; r0 < rows; r0 += (kWaves - kRowWaves) * per) {
        const int r = r0 + in;
        int c = p - rotation(r, n);
        c += c < 0 ? n : 0;
        if (in < per && r < rows) to_lds16(src, (uint32_t)((r * n + c) * 16), __builtin_amdgcn_readfirstlane(base + r0 * n * 16));
    }
}
// `floats` consecutive floats, 16-byte aligned
__device__ __forceinline__ void floats_to_lds(const float *src, int floats, float *lds, int wave, int lane) {
    const uint32_t base = lds_address(lds);
    if ((floats & 3) == 0) {
        for (int i = wave * 64; i < floats / 4; i += (kWaves - kRowWaves) * 64)
            if (i + lane < floats / 4) to_lds16(src, (uint32_t)((i + lane) * 16), __builtin_amdgcn_readfirstlane(base + i * 16));
    } else {
        for (int i = wave * 64; i < floats; i += (kWaves - kRowWaves) * 64)
            if (i + lane < floats) to_lds4(src, (uint32_t)((i + lane) * 4), __builtin_amdgcn_readfirstlane(base + i * 4));
    }
}

// The products of 16 LDS rows row .. row + 15 with steps [first, end) of the staged row
template <int S>
__device__ __forceinline__ float multiply_tile(const uint8_t *lds, const float *scales, int row, int n, const uint8_t *planes, int pitch,
                                               const float *unit, int first, int end, int lane) {
    const int r = row + (lane & 15), quarter = lane >> 4, rot = rotation(r, n), groups = n >> 1;
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < S; j++) {                                  // (no branches: the reads of all steps go out together)
        const int st = first + j < end ? first + j : first;
        int c = st * 4 + quarter;
        c = c < n ? c : n - 1;                                     // a half step: the digits are zeros
        int at = c + rot;
        at -= at >= n ? n : 0;
        const intx4 w = *reinterpret_cast<const intx4 *>(lds + (r * n + at) * 16);
        const float next = multiply_step(w, scales[r * groups + (c >> 1)], planes, pitch, unit, st, lane, acc);
        acc = first + j < end ? next : acc;
    }
    return quarters_sum(acc);
}

// Columns k0 .. k0 + 63 of 16 rows of a weight, in registers (a chunk past the row's end repeats the last one: its digits
// are zeros)
struct WeightTile { intx4 q; float s; };
__device__ __forceinline__ WeightTile load_tile(const int8_t *wq, const float *scales, int row, int kp, int k0, int lane) {
    int k = k0 + (lane >> 4) * 16;
    k = k < kp ? k : kp - 16;
    return WeightTile{*reinterpret_cast<const intx4 *>(wq + (int64_t)row * kp + k), scales[(int64_t)row * (kp >> 5) + (k >> 5)]};
}
__device__ __forceinline__ float multiply_tile(const WeightTile &w, const uint8_t *planes, int pitch, const float *unit, int lane) {
    return quarters_sum(multiply_step(w.q, w.s, planes, pitch, unit, 0, lane, 0.0f));
}

// ── the row a launch starts from ────────────────────────────────────────────
// The row wavefronts' shares of the partial sums, to LDS.
__device__ __forceinline__ void add_parts(const float *part, int n_part, int d, float4 *red, int t) {
    constexpr int kBatch = 8;
    const int c = t & 63, set = t >> 6;                            // a wavefront holds the row, the four share its partial sums
    const uint32_t row = (uint32_t)d * 4, col = 4 * c < d ? c * 16 : 0, last = (uint32_t)(n_part - 1) * row + col;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p0 = set; p0 < n_part; p0 += kBatch * kRowWaves) {        // one round up to 32 parts
        float4 v[kBatch];
        uint32_t at = (uint32_t)p0 * row + col;
#pragma unroll
        for (int j = 0; j < kBatch; j++, at += kRowWaves * row)
            v[j] = *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(part) + min(at, last));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kBatch; j++) {
            const bool on = p0 + j * kRowWaves < n_part;
            s.x += on ? v[j].x : 0.0f; s.y += on ? v[j].y : 0.0f; s.z += on ? v[j].z : 0.0f; s.w += on ? v[j].w : 0.0f;
        }
    }
    red[set * 64 + c] = s;
}

// What wavefront 0 needs of the row besides the sums
struct RowOperands { float4 x, gamma, beta, bias; };
__device__ __forceinline__ RowOperands load_row(const float *x, const float *gamma, const float *beta, const float *bias, int d, int lane) {
    const int c = 4 * lane < d ? lane : 0;
    RowOperands o;
    o.x = reinterpret_cast<const float4 *>(x)[c];
    o.gamma = reinterpret_cast<const float4 *>(gamma)[c];
    o.beta = beta ? reinterpret_cast<const float4 *>(beta)[c] : make_float4(0.f, 0.f, 0.f, 0.f);
    o.bias = bias ? reinterpret_cast<const float4 *>(bias)[c] : make_float4(0.f, 0.f, 0.f, 0.f);
    return o;
}

// Wavefront 0: the finished row (to `out` from workgroup 0), normalised, as digits; *divisor what the products have to be
// divided by (RMSNorm: the root mean square - the staged row is gamma * x; LayerNorm: 1).
__device__ __forceinline__ void stage_row(const RowOperands &o, const float4 *red, bool parts, bool layernorm, int d, float *out,
                                          uint8_t *planes, float *unit, float *divisor, int lane) {
    const bool ok = 4 * lane < d;
    float4 x = o.x;
    if (parts) {
        float4 s = red[lane];
#pragma unroll
        for (int q = 1; q < kRowWaves; q++) { const float4 a = red[q * 64 + lane]; s.x += a.x; s.y += a.y; s.z += a.z; s.w += a.w; }
        x.x += s.x + o.bias.x; x.y += s.y + o.bias.y; x.z += s.z + o.bias.z; x.w += s.w + o.bias.w;
    }
    if (!ok) x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (ok && blockIdx.x == 0) reinterpret_cast<float4 *>(out)[lane] = x;
    const float inv_d = 1.0f / (float)d;
    float4 y;
    if (layernorm) {                                         // LayerNorm1D.java:34-66: mean, then the variance about it
        const float mean = wave_sum_dpp((x.x + x.y) + (x.z + x.w)) * inv_d;
        x.x -= mean; x.y -= mean; x.z -= mean; x.w -= mean;
        const float var = wave_sum_dpp(ok ? (x.x * x.x + x.y * x.y) + (x.z * x.z + x.w * x.w) : 0.0f) * inv_d, sd = sqrtf(var + kLayerNormEps);
        y = make_float4((x.x / sd) * o.gamma.x + o.beta.x, (x.y / sd) * o.gamma.y + o.beta.y, (x.z / sd) * o.gamma.z + o.beta.z,
                        (x.w / sd) * o.gamma.w + o.beta.w);
        if (lane == 0) *divisor = 1.0f;
    } else {                                                 // RMSNorm1D.java:46-57
        const float square = wave_sum_dpp((x.x * x.x + x.y * x.y) + (x.z * x.z + x.w * x.w)) * inv_d;
        if (lane == 0) *divisor = sqrtf(square + kRmsEps);
        y = make_float4(x.x * o.gamma.x, x.y * o.gamma.y, x.z * o.gamma.z, x.w * o.gamma.w);
    }
    stage_digits4(planes, kPitch, unit, lane, ok ? y : make_float4(0.f, 0.f, 0.f, 0.f));
}

// Waits for this wavefront's direct loads (and its other ones)
__device__ __forceinline__ void loads_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// ── attention half ──────────────────────────────────────────────────────────
// The head's 3 HD rows are 3 HD / 16 tiles whose K is cut into kParts: 24 units, three a wavefront.
// (Operands as separate arguments, the first-needed in front: the leading 16 words arrive in registers.)
template <int HD>
__global__ void __launch_bounds__(kThreads)
k_decode_attn(const float *x, const float *part, const int8_t *wqkv, const float *gamma, const int32_t *state, int n_part, int d,
              int max_seq, float scale, const float *s_qkv, const float *bias, const float *beta, const int8_t *wo, const float *s_wo,
              float *k_cache, float *v_cache, const float *cos_t, const float *sin_t, float *part_out, float *out) {
    constexpr int kTiles = 3 * HD / 16, kParts = 24 / kTiles, kSteps = (kMaxD / 64 + kParts - 1) / kParts;
    constexpr int LPK = HD / 4, KPW = 64 / LPK, TILE = kWaves * KPW, U = 4;
    constexpr int kPitchO = 64 + 16, kOTiles = kMaxD / 16 / kWaves;
    __shared__ __align__(16) uint8_t weights[3 * HD * kMaxD];
    __shared__ __align__(16) float scales[3 * HD * kMaxD / 32];
    __shared__ __align__(16) uint8_t planes[4 * kPitch];
    __shared__ __align__(16) float4 red[64 * kRowWaves];
    __shared__ __align__(16) float row[24 * 16];               // the units' products: [part][3 HD]
    __shared__ __align__(16) float states[kWaves * HD];
    __shared__ __align__(16) uint8_t planes_o[4 * kPitchO];
    __shared__ float unit[kMaxD / 32], unit_o[4], divisor, s_m[kWaves], s_l[kWaves];

    const int h = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int steps = (d + 63) >> 6, n = d >> 4;
    // (a vector load: it is on its way while the row's operands are requested; a scalar one would be moved to its use)
    int zero = 0;
    asm volatile("" : "+v"(zero));
    const int position = state[zero];
    RowOperands ops;
    if (wave < kRowWaves) {
        if (wave == 0) ops = load_row(x, gamma, beta, bias, d, lane);
        if (n_part < 0) add_parts(part + (int64_t)min(max(state[0], 0), max_seq - 1) * d, 1, d, red, t);
        else add_parts(part, n_part, d, red, t);
    } else {
        for (int seg = 0; seg < 3; seg++)
            rows_to_lds(wqkv + (int64_t)(seg * d + h * HD) * d, HD, n, weights, seg * HD, wave - kRowWaves, lane);
        for (int seg = 0; seg < 3; seg++)
            floats_to_lds(s_qkv + (int64_t)(seg * d + h * HD) * (d >> 5), HD * (d >> 5), scales + seg * HD * (d >> 5), wave - kRowWaves, lane);
    }
    lds_barrier();
    if (wave == 0) stage_row(ops, red, n_part != 0, beta != nullptr, d, out, planes, unit, &divisor, lane);
    else if (wave >= kRowWaves) loads_done();
    // keys and values of the first round, the rotation: behind the row (wavefront 0) or the weights
    int pos = __builtin_amdgcn_readfirstlane(position);
    if (pos > max_seq - 1) pos = max_seq - 1;                  // the host never lets this happen; stay in bounds
    if (pos < 0) pos = 0;
    const int sub = lane / LPK, dl = lane % LPK;
    float *kb = k_cache + (int64_t)h * max_seq * HD + dl * 4, *vb = v_cache + (int64_t)h * max_seq * HD + dl * 4;
    const int key0 = wave * KPW + sub;
    float4 K[U], V[U];
    auto load_round = [&](float4 (&k)[U], float4 (&v)[U], int r0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if ((r0 + u) * TILE >= pos && u > 0) break;        // workgroup-uniform: no cached key left
            const int key = key0 + (r0 + u) * TILE, at = key < pos ? key : 0;
            k[u] = *reinterpret_cast<const float4 *>(kb + (int64_t)at * HD);
            v[u] = *reinterpret_cast<const float4 *>(vb + (int64_t)at * HD);
        }
    };
    load_round(K, V, 0);
    const float2 cs = *reinterpret_cast<const float2 *>(cos_t + (int64_t)pos * (HD / 2) + dl * 2);
    const float2 sn = *reinterpret_cast<const float2 *>(sin_t + (int64_t)pos * (HD / 2) + dl * 2);
    lds_barrier();
#pragma unroll 1
    for (int i = 0; i < 3; i++) {                              // (a loop: code is fetched from memory at every launch)
        const int u = wave + kWaves * i, tile = u % kTiles, p = u / kTiles;
        const float v = multiply_tile<kSteps>(weights, scales, tile * 16, n, planes, kPitch, unit, p * steps / kParts, (p + 1) * steps / kParts, lane);
        if (lane < 16) row[u * 16 + lane] = v;
    }
    lds_barrier();
    // the head's columns of Wo, behind everybody's keys and values: requested any earlier they only delay those in the L1
    WeightTile w_out[kOTiles];
#pragma unroll
    for (int i = 0; i < kOTiles; i++) {
        const int tile = (wave + kWaves * i) * 16 < d ? wave + kWaves * i : 0;
        w_out[i] = load_tile(wo, s_wo, tile * 16 + (lane & 15), d, h * HD, lane);
    }
    float4 q = make_float4(0.f, 0.f, 0.f, 0.f), k = q, nv = q;
#pragma unroll
    for (int p = 0; p < kParts; p++) {
        const float *b = row + p * 3 * HD + dl * 4;
        const float4 a0 = *reinterpret_cast<const float4 *>(b), a1 = *reinterpret_cast<const float4 *>(b + HD), a2 = *reinterpret_cast<const float4 *>(b + 2 * HD);
        q.x += a0.x; q.y += a0.y; q.z += a0.z; q.w += a0.w;
        k.x += a1.x; k.y += a1.y; k.z += a1.z; k.w += a1.w;
        nv.x += a2.x; nv.y += a2.y; nv.z += a2.z; nv.w += a2.w;
    }
    const float inverse = 1.0f / divisor, by = residual_divisor(divisor);
    auto divide = [&](float &v) { v = quotient(v, by, inverse); };
    divide(q.x); divide(q.y); divide(q.z); divide(q.w);
    divide(k.x); divide(k.y); divide(k.z); divide(k.w);
    divide(nv.x); divide(nv.y); divide(nv.z); divide(nv.w);
    const float4 qr = make_float4(q.x * cs.x - q.y * sn.x, q.x * sn.x + q.y * cs.x, q.z * cs.y - q.w * sn.y, q.z * sn.y + q.w * cs.y);
    const float4 nk = make_float4(k.x * cs.x - k.y * sn.x, k.x * sn.x + k.y * cs.x, k.z * cs.y - k.w * sn.y, k.z * sn.y + k.w * cs.y);
    float m = -INFINITY, l = 0.0f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int r0 = 0;;) {
        const bool more = (r0 + U) * TILE <= pos;              // workgroup-uniform
        float4 K1[U], V1[U];
        if (more) load_round(K1, V1, r0 + U);
        float sc[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            sc[u] = -INFINITY;
            if ((r0 + u) * TILE > pos) { V[u] = make_float4(0.f, 0.f, 0.f, 0.f); continue; }      // workgroup-uniform
            const int key = key0 + (r0 + u) * TILE;
            if (key == pos) {                                  // the new row: used from registers, and appended
                K[u] = nk; V[u] = nv;
                *reinterpret_cast<float4 *>(kb + (int64_t)key * HD) = nk;
                *reinterpret_cast<float4 *>(vb + (int64_t)key * HD) = nv;
            }
            // (q.k) * scale as the reference computes it (HeadOps.java:96-99), then the change of base
            const float dot = group_sum<LPK>(qr.x * K[u].x + qr.y * K[u].y + qr.z * K[u].z + qr.w * K[u].w);
            sc[u] = key <= pos ? (dot * scale) * kLog2e : -INFINITY;
            if (key > pos) V[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        float mn = m;
#pragma unroll
        for (int u = 0; u < U; u++) mn = fmaxf(mn, sc[u]);
        if (mn > -INFINITY) {
            const float corr = __builtin_amdgcn_exp2f(m - mn);
            l *= corr; o.x *= corr; o.y *= corr; o.z *= corr; o.w *= corr;
#pragma unroll
            for (int u = 0; u < U; u++) {
                const float e = __builtin_amdgcn_exp2f(sc[u] - mn);
                l += e;
                o.x += e * V[u].x; o.y += e * V[u].y; o.z += e * V[u].z; o.w += e * V[u].w;
            }
            m = mn;
        }
        if (!more) break;
        r0 += U;
#pragma unroll
        for (int u = 0; u < U; u++) { K[u] = K1[u]; V[u] = V1[u]; }
    }
    // the lane groups of a wavefront, then the wavefronts (LDS)
    auto groups = [&](float v, auto op) {
        float a, b;
        if constexpr (LPK == 8) { lane_pair<8>(v, a, b); v = op(a, b); }
        if constexpr (LPK <= 16) { lane_pair<16>(v, a, b); v = op(a, b); }
        lane_pair<32>(v, a, b);
        return op(a, b);
    };
    auto add = [](float a, float b) { return a + b; };
    const float most = groups(m, [](float a, float b) { return fmaxf(a, b); }), e = most == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - most);
    m = most;
    l = groups(l * e, add);
    o = make_float4(groups(o.x * e, add), groups(o.y * e, add), groups(o.z * e, add), groups(o.w * e, add));
    if (lane == 0) { s_m[wave] = m; s_l[wave] = l; }
    if (sub == 0) *reinterpret_cast<float4 *>(&states[wave * HD + dl * 4]) = o;
    lds_barrier();
    if (t < 64 / 4) {
        float M = -INFINITY, L = 0.0f;
        o = make_float4(0.f, 0.f, 0.f, 0.f);
        if (t < LPK) {
#pragma unroll
            for (int i = 0; i < kWaves; i++) M = fmaxf(M, s_m[i]);
#pragma unroll
            for (int i = 0; i < kWaves; i++) {
                const float e = __builtin_amdgcn_exp2f(s_m[i] - M);
                const float4 a = *reinterpret_cast<const float4 *>(&states[i * HD + t * 4]);
                L += s_l[i] * e;
                o.x += a.x * e; o.y += a.y * e; o.z += a.z * e; o.w += a.w * e;
            }
            o.x /= L; o.y /= L; o.z /= L; o.w /= L;
        }
        stage_digits4(planes_o, kPitchO, unit_o, t, o);
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < kOTiles; i++) {
        const int tile = wave + kWaves * i;
        const float v = multiply_tile(w_out[i], planes_o, kPitchO, unit_o, lane);
        if (tile * 16 < d && lane < 16) part_out[(int64_t)h * d + tile * 16 + lane] = v;
    }
}

// ── feed-forward half ───────────────────────────────────────────────────────
constexpr int kFfnUnits = 64;

template <bool SWIGLU>
__global__ void __launch_bounds__(kThreads)
k_decode_ffn(const float *x, const float *part, const int8_t *wgu, const float *gamma, const int8_t *wd, int n_part, int d, int dff,
             const float *s_gu, const float *s_d, const float *bias, const float *beta, const float *bg, const float *bu,
             float *part_out, float *out) {
    constexpr int kRows = SWIGLU ? 2 * kFfnUnits : kFfnUnits, kTiles = kRows / 16, kParts = kWaves / kTiles;
    constexpr int kSteps = (kMaxD / 64 + kParts - 1) / kParts, kPitchH = kFfnUnits + 16, kOTiles = kMaxD / 16 / kWaves;
    __shared__ __align__(16) uint8_t weights[kRows * kMaxD];
    __shared__ __align__(16) float scales[kRows * kMaxD / 32];
    __shared__ __align__(16) uint8_t planes[4 * kPitch];
    __shared__ __align__(16) float4 red[64 * kRowWaves];
    __shared__ __align__(16) float prod[kParts * kRows];
    __shared__ __align__(16) float hidden[kFfnUnits];
    __shared__ __align__(16) uint8_t planes_h[4 * kPitchH];
    __shared__ float unit[kMaxD / 32], unit_h[kFfnUnits / 32], divisor;

    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int steps = (d + 63) >> 6, n = d >> 4, u0 = blockIdx.x * kFfnUnits;
    const int units = dff - u0 < kFfnUnits ? dff - u0 : kFfnUnits, rows = SWIGLU ? 2 * units : units, kp = (dff + 31) & ~31;
    RowOperands ops;
    if (wave < kRowWaves) {
        if (wave == 0) ops = load_row(x, gamma, beta, bias, d, lane);
        add_parts(part, n_part, d, red, t);
    } else {
        const int64_t first = SWIGLU ? 2 * u0 : u0;
        rows_to_lds(wgu + first * d, rows, n, weights, 0, wave - kRowWaves, lane);
        floats_to_lds(s_gu + first * (d >> 5), rows * (d >> 5), scales, wave - kRowWaves, lane);
    }
    WeightTile w_down[kOTiles];
#pragma unroll
    for (int i = 0; i < kOTiles; i++) {
        const int tile = (wave + kWaves * i) * 16 < d ? wave + kWaves * i : 0;
        w_down[i] = load_tile(wd, s_d, tile * 16 + (lane & 15), kp, u0, lane);
    }
    float b_gate = 0.0f, b_up = 0.0f;
    if (t < units) {
        if (bg) b_gate = bg[u0 + t];
        if (SWIGLU && bu) b_up = bu[u0 + t];
    }
    lds_barrier();
    if (wave == 0) stage_row(ops, red, n_part > 0, beta != nullptr, d, out, planes, unit, &divisor, lane);
    else if (wave >= kRowWaves) loads_done();
    lds_barrier();
    {
        const int tile = wave % kTiles, p = wave / kTiles;
        // (rows past the last hold whatever LDS held: their products are not used)
        const float v = multiply_tile<kSteps>(weights, scales, tile * 16, n, planes, kPitch, unit, p * steps / kParts, (p + 1) * steps / kParts, lane);
        if (lane < 16) prod[p * kRows + tile * 16 + lane] = v;
    }
    lds_barrier();
    if (t < kFfnUnits) {
        float v = 0.0f;
        if (t < units) {
            if constexpr (SWIGLU) {
                float gate = 0.0f, up = 0.0f;
#pragma unroll
                for (int q = 0; q < kParts; q++) { gate += prod[q * kRows + 2 * t]; up += prod[q * kRows + 2 * t + 1]; }
                gate = gate / divisor + b_gate;
                up = up / divisor + b_up;
                v = gate * (1.0f / (1.0f + expf(-gate))) * up;                  // SiLU.java:20-24, SwiGLULayer.java:69
            } else {
#pragma unroll
                for (int q = 0; q < kParts; q++) v += prod[q * kRows + t];
                v = gemm_gelu(v / divisor + b_gate);
            }
        }
        hidden[t] = v;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                      // (one wavefront reads what it wrote)
        if (t < kFfnUnits / 4) stage_digits4(planes_h, kPitchH, unit_h, t, *reinterpret_cast<const float4 *>(hidden + 4 * t));
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < kOTiles; i++) {
        const int tile = wave + kWaves * i;
        const float o = multiply_tile(w_down[i], planes_h, kPitchH, unit_h, lane);
        if (tile * 16 < d && lane < 16) part_out[(int64_t)blockIdx.x * d + tile * 16 + lane] = o;
    }
}

// out = x + (sum of the partial rows + bias), x where there are none: the row behind the last block
__global__ void __launch_bounds__(256) k_decode_row(const float *__restrict__ x, const float *__restrict__ part, int n_part,
                                                    const float *__restrict__ bias, float *__restrict__ out, int d) {
    __shared__ float red[16][16];
    const int c = threadIdx.x & 15, set = threadIdx.x >> 4, col = blockIdx.x * 16 + c;
    float s = 0.0f;
    if (col < d)
#pragma unroll 4
        for (int p = set; p < n_part; p += 16) s += part[(int64_t)p * d + col];
    red[set][c] = s;
    __syncthreads();
    if (threadIdx.x < 16 && col < d) {
        for (int q = 1; q < 16; q++) s += red[q][c];
        out[col] = n_part > 0 ? x[col] + (s + (bias ? bias[col] : 0.0f)) : x[col];
    }
}

template <int HD> void go_attn(hipStream_t s, const DecodeAttn &a) {
    const DecodeRow &r = a.in;
    launch_kernel(k_decode_attn<HD>, dim3(r.d / HD), dim3(kThreads), 0, s, r.x, r.part, a.wqkv, r.gamma, a.state, r.at_state ? -1 : r.n_part,
                  r.d, a.max_seq, a.scale, a.s_qkv, r.bias, r.beta, a.wo, a.s_wo, a.k_cache, a.v_cache, a.cos_t, a.sin_t, a.part, r.out);
}
template <bool SWIGLU> void go_ffn(hipStream_t s, const DecodeFfn &a) {
    const DecodeRow &r = a.in;
    launch_kernel(k_decode_ffn<SWIGLU>, dim3(decode_ffn_parts(a.dff)), dim3(kThreads), 0, s, r.x, r.part, a.wgu, r.gamma, a.wd, r.n_part, r.d,
                  a.dff, a.s_gu, a.s_d, r.bias, r.beta, a.bg, a.bu, a.part, r.out);
}

}  // namespace

bool decode_block_ok(int d, int hd, int dff) { return d > 0 && dff > 0 && (hd == 32 || hd == 64) && d % hd == 0 && d <= kMaxD; }
// One workgroup reads all of a head's keys (50 bytes a clock), where the five-launch path has four, so from some position on the
// latter is the faster one: 4-layer models, us a token here / there, at 16, 300, 700 and 1250 positions: d 64, hd 32, dff 173
// 43.8 / 56.4, 46.8 / 56.9, 51.1 / 56.8, 56.7 / 59.6; d 256, hd 32, dff 691 47.7 / 58.8, 52.4 / 58.9, 56.1 / 59.3, 62.2 / 62.4; d 64,
// hd 64, dff 173 44.4 / 55.1, 51.8 / 55.7, 60.4 / 58.4, 73.5 / 61.3; d 256, hd 64, dff 691 50.1 / 58.7, 58.7 / 59.2, 68.0 / 62.2, 81.9 /
// 65.3.  The line falls with the width; over dff from 86 to 4096, SwiGLU and GELU, it lies between 130 and 540 positions at hd 64
// and between 650 and 1650 at hd 32, and this rule is within 5 % of the better way everywhere.
int decode_block_positions(int d, int hd) { return hd == 32 ? 1536 - 11 * d / 4 : 512 - d; }
int decode_ffn_parts(int dff) { return (dff + kFfnUnits - 1) / kFfnUnits; }

void launch_decode_attn(hipStream_t s, const DecodeAttn &a) {
    if (a.hd == 32) go_attn<32>(s, a);
    else go_attn<64>(s, a);
}
void launch_decode_ffn(hipStream_t s, const DecodeFfn &a) {
    if (a.swiglu) go_ffn<true>(s, a);
    else go_ffn<false>(s, a);
}
void launch_decode_row(hipStream_t s, const DecodeRow &r) {
    launch_kernel(k_decode_row, dim3((r.d + 15) / 16), dim3(256), 0, s, r.x, r.part, r.n_part, r.bias, r.out, r.d);
}

}  // namespace dj
