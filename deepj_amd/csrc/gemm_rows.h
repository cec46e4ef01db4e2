// What the Q8 GEMM that multiplies straight from the int8 weights (kernels_gemm_rows.hip) and its helpers share.
#pragma once
#include <cstdint>
#include <hip/hip_runtime.h>
#include "gemm_epilogue.h"

namespace dj {

// Where the bf16 pieces of activation (row, c) lie for v_mfma_f32_32x32x16_bf16: blocks of 1 KB, one per 32 rows, 32 k, half of
// those k and piece; in a block 8 consecutive k for each lane.  Lane l of step s of a group holds row l % 32 and
// k = 16 (l / 32) + 8 s + j, as the weights' side does (a lane's 16 k of a weight row are 16 consecutive bytes).  The high
// piece; the middle and the low one are kOperandPiece and twice that further on.
constexpr int kOperandPiece = 512, kOperandPieces = 3;
__host__ __device__ inline int64_t operand_at(int row, int c, int groups) {
    const int g = c >> 5, h = (c >> 4) & 1, s = (c >> 3) & 1, j = c & 7;
    return ((((int64_t)(row >> 5) * groups + g) * 2 + s) * kOperandPieces * 64 + h * 32 + (row & 31)) * 8 + j;
}
// Every second 128 k are stored with their sign turned, and the sums over them are subtracted: the matrix cores cut off the
// low bits of what they add up, always downwards, and two halves of opposite sign are cut off in opposite directions (4096 x
// 11008, 4 wavefronts: 1.57e-7 of the result's rms against 64 bits without, 1.19e-7 with it).
constexpr int kOperandChunk = 128;
__host__ __device__ inline bool operand_negated(int c) { return (c / kOperandChunk) & 1; }

#if defined(__HIPCC__)
// 64 lanes x 16 (4) bytes from base + off[lane] into LDS bytes [dst, dst + 1024 (256)), lane order.  The statements write M0
// and say so in their clobber lists, so that the compiler never carries a value of its own in M0 across them (it
// initialises M0 itself for some LDS and message instructions); clang notes that M0 is a reserved register, which
// is the point of listing it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_to_lds16(const void *base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void load_to_lds4(const void *base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
#endif

// kernels_gemm_f16.hip: the rows, normalised if gamma (and beta) say so, in that order; rows [m, m_pad) as zeros
void launch_split_operand(hipStream_t s, const float *x, const float *gamma, const float *beta, uint16_t *planes, int m, int m_pad, int k, int kp);

// kernels_matmul.hip: C = epilogue(sum of the slabs of partial products)
void launch_q8_sum_partials(hipStream_t s, const float *partial, float *out, int splits, int m, int n_rows, const GemmEpilogue &ep);

// kernels_gemm_rows.hip
void q8_gemm_rows_configure();   // once per device, before the first launch
bool q8_gemm_rows_ok(int m, int n_rows, int k, bool norm, bool prepared);
int64_t q8_gemm_rows_workspace_floats(int m, int n_rows, int k, bool may_share);   // may_share: a tile's K among several workgroups
void launch_q8_gemm_rows(hipStream_t s, const float *x, const float *gamma, const float *beta, const int8_t *wq, const float *scales, float *out, int m, int k,
                         int n_rows, const GemmEpilogue &ep, float *workspace, int64_t workspace_floats, bool may_share);

}  // namespace dj
