// Device-side helpers shared by the decode kernels (Q8 matvec and decode attention).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace dj {
namespace dev {

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits for every outstanding global
// load (its workgroup-scope fence needs vmcnt(0)), which here would park the workgroup until the weight rows
// already requested from HBM have arrived; the staged activations only need the LDS writes to be complete.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ float dot16(const int4 &w, const float *xr) {
    float d = 0.0f;
    const int words[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        int v = words[i];
        d = fmaf(xr[4 * i + 0], (float)(int8_t)(v & 0xff), d);
        d = fmaf(xr[4 * i + 1], (float)(int8_t)((v >> 8) & 0xff), d);
        d = fmaf(xr[4 * i + 2], (float)(int8_t)((v >> 16) & 0xff), d);
        d = fmaf(xr[4 * i + 3], (float)(v >> 24), d);
    }
    return d;
}

// Sum over the 64 lanes with DPP row operations (no LDS traffic); every lane gets the total.
__device__ __forceinline__ float wave_sum_dpp(float v) {
#define DJ_DPP_ADD(ctrl, row_mask)                                                                        \
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, row_mask, 0xf, false))
    DJ_DPP_ADD(0xB1, 0xf);    // quad_perm [1,0,3,2]
    DJ_DPP_ADD(0x4E, 0xf);    // quad_perm [2,3,0,1]
    DJ_DPP_ADD(0x141, 0xf);   // row_half_mirror
    DJ_DPP_ADD(0x140, 0xf);   // row_mirror: every lane of a 16-lane row holds the row sum
    DJ_DPP_ADD(0x142, 0xa);   // row_bcast:15 into rows 1 and 3
    DJ_DPP_ADD(0x143, 0xc);   // row_bcast:31 into rows 2 and 3: lane 63 holds the total
#undef DJ_DPP_ADD
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Sum over the LPK (8, 16 or 32) consecutive lanes that share a key; every lane of the group gets the total.
// DPP row operations instead of shuffles: a shuffle is an LDS-crossbar round trip with a wait behind it, and the
// score of every key needs log2(LPK) of them in a row.
template <int LPK>
__device__ __forceinline__ float group_sum(float v) {
#define DJ_DPP_ADD(ctrl) \
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, false))
    DJ_DPP_ADD(0xB1);                             // quad_perm [1,0,3,2]
    DJ_DPP_ADD(0x4E);                             // quad_perm [2,3,0,1]: quad sums
    if constexpr (LPK >= 8) DJ_DPP_ADD(0x141);    // row_half_mirror: 8 lanes
    if constexpr (LPK >= 16) DJ_DPP_ADD(0x140);   // row_mirror: 16 lanes
#undef DJ_DPP_ADD
    if constexpr (LPK == 32) v += __shfl_xor(v, 16, 64);
    return v;
}

// Digit planes in LDS: plane p holds one byte per k (k padded with zeros to a multiple of 64), `pitch` bytes apart (16 more
// than they hold: the four planes' reads of one k fall on different banks); unit[g]
// the power of two of group g (NaN where the group holds an infinity or a NaN).
// Thread with four values of k = 4 i .. 4 i + 3 (eight consecutive lanes share a group).
__device__ __forceinline__ void stage_digits4(uint8_t *planes, int pitch, float *unit, int i, float4 v) {
    uint32_t m = max(max(__float_as_uint(v.x) & 0x7fffffffu, __float_as_uint(v.y) & 0x7fffffffu),
                     max(__float_as_uint(v.z) & 0x7fffffffu, __float_as_uint(v.w) & 0x7fffffffu));
    m = max(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1, 0xf, 0xf, false));      // quad_perm [1,0,3,2]
    m = max(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xf, 0xf, false));      // quad_perm [2,3,0,1]
    m = max(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xf, 0xf, false));     // row_half_mirror
    // m = f 2^e, f in [0.5, 1): values times 2^(29 - e) are at most 2^29.  The shift stays where 2^shift and 2^-shift are
    // normal numbers.
    const int e = __builtin_amdgcn_frexp_expf(__uint_as_float(m));
    const int shift = min(29 - e, 120);
    const float up = ldexpf(1.0f, shift);
    // t = d0 + 2^8 d1 + 2^16 d2 + 2^24 d3 with signed bytes: add 128 to each of the three low bytes, then flip their top bits
    auto digits = [&](float x) { return ((uint32_t)(int)rintf(x * up) + 0x00808080u) ^ 0x00808080u; };
    const uint32_t w0 = digits(v.x), w1 = digits(v.y), w2 = digits(v.z), w3 = digits(v.w);
    const uint32_t a = __builtin_amdgcn_perm(w1, w0, 0x05010400u), b = __builtin_amdgcn_perm(w3, w2, 0x05010400u);
    const uint32_t c = __builtin_amdgcn_perm(w1, w0, 0x07030602u), d = __builtin_amdgcn_perm(w3, w2, 0x07030602u);
    uint32_t *p = reinterpret_cast<uint32_t *>(planes) + i;
    p[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
    p[pitch / 4] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    p[2 * (pitch / 4)] = __builtin_amdgcn_perm(d, c, 0x05040100u);
    p[3 * (pitch / 4)] = __builtin_amdgcn_perm(d, c, 0x07060302u);
    if ((i & 7) == 0) unit[i >> 3] = m >= 0x7f800000u ? __uint_as_float(0x7fc00000u) : ldexpf(1.0f, -shift);
}

// The value of the lanes `OFF` apart: a of one, b of the other (the same pair for both)
template <int OFF> __device__ __forceinline__ void lane_pair(float v, float &a, float &b) {
    if constexpr (OFF == 8) {
        a = v;
        b = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf, 0xf, false));   // row_ror:8
    } else {
        const unsigned u = __builtin_bit_cast(unsigned, v);
        const auto r = OFF == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false) : __builtin_amdgcn_permlane32_swap(u, u, false, false);
        a = __builtin_bit_cast(float, (unsigned)r[0]);
        b = __builtin_bit_cast(float, (unsigned)r[1]);
    }
}
__device__ __forceinline__ float quarters_sum(float v) {
    float a, b;
    lane_pair<16>(v, a, b);
    lane_pair<32>(a + b, a, b);
    return a + b;
}

// v / by for many v: the product with 1 / by, corrected by its residual.  An infinite divisor or product has no residual: the
// first takes part as the largest float beside its reciprocal of 0, the second stands.
__device__ __forceinline__ float residual_divisor(float by) { return fminf(by, 3.402823466e38f); }
__device__ __forceinline__ float quotient(float v, float residual_by, float inverse) {
    const float y = v * inverse, q = fmaf(fmaf(-y, residual_by, v), inverse, y);
    return fabsf(y) == INFINITY ? y : q;
}

}  // namespace dev
}  // namespace dj
