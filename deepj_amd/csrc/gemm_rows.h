// What the Q8 GEMM that multiplies straight from the int8 weights (kernels_gemm_rows.hip) and its helpers share.
#pragma once
#include <cstdint>
#include <hip/hip_runtime.h>
#include "gemm_epilogue.h"

namespace dj {

struct GemmChain;

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
// low bits of what they add up, always downwards, and two halves of opposite sign are cut off in opposite directions (30 x
// 1023 over 11008: 1.48e-7 of the result's rms against 64 bits without, 1.10e-7 with it).
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
// .. of bytes that pass by: they take no place in the caches from what is read again
__device__ __forceinline__ void load_passing_to_lds16(const void *base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void load_to_lds4(const void *base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
#endif

// kernels_gemm_f16.hip
int q8_gemm_f16_forced();        // DEEPJ_HIP_GEMM_F16, -1 where it is not set; 0: every GEMM on k_gemm_q8
// The rows, normalised if gamma (and beta) say so, in that order; rows [m, m_pad) as zeros
void launch_split_operand(hipStream_t s, const float *x, const float *gamma, const float *beta, uint16_t *planes, int m, int m_pad, int k, int kp);
// The same for rows that are still partial products [splits][m][k] and have to be stored as well: out = residual + (their sum + bias)
bool split_operand_sum_ok(int k);
void launch_split_operand_sum(hipStream_t s, const float *partial, int splits, const float *bias, const float *residual, float *out, const float *gamma,
                              const float *beta, uint16_t *planes, int m, int k);

// An estimate of a Q8 GEMM's time in us.  With x workgroups a compute unit, in `rounds` rounds, kk thousand k a workgroup and
// `full` of its rows inside the matrix:
//   fixed + per_x x + kk (per_k + again (rounds - 1) + per_kx x full) + (slabs m n shares + rows m k + weights n k) / 10^6.
struct GemmCost {
    double fixed, per_x, per_k, again, per_kx, slabs, rows, weights;
    double us(double x, double rounds, double kk, double full, double m, double n, double k, int shares) const {
        return fixed + per_x * x + kk * (per_k + again * (rounds - 1.0) + per_kx * x * full) + ((shares > 1 ? slabs * m * n * shares : 0.0) + rows * m * k + weights * n * k) * 1e-6;
    }
};

// kernels_matmul.hip: what a product takes on k_gemm_q8, and into how many sums it deals an output's K
struct Q8GemmEstimate { double us; int sums; };
Q8GemmEstimate q8_gemm_estimate(int m, int n_rows, int k, bool norm, bool may_share);
// C = epilogue(sum of the slabs of partial products)
void launch_q8_sum_partials(hipStream_t s, const float *partial, float *out, int splits, int m, int n_rows, const GemmEpilogue &ep);

// kernels_gemm_rows.hip
void q8_gemm_rows_configure();   // once per device, before the first launch
struct RowsPlan { int tmw, tnw, shares; double us; };      // a tile's rows and columns in units of 32, the workgroups that share its K
// false: not a product for this kernel.  may_share: a tile's K among several workgroups; ready: its rows' pieces are there
bool q8_gemm_rows_ok(int m, int n_rows, int k, bool norm, bool prepared, bool may_share, RowsPlan *plan = nullptr, bool ready = false);
int64_t q8_gemm_rows_workspace_floats(int m, int n_rows, int k, const RowsPlan &plan);
void launch_q8_gemm_rows(hipStream_t s, const float *x, const float *gamma, const float *beta, const int8_t *wq, const float *scales, float *out, int m, int k,
                         int n_rows, const GemmEpilogue &ep, const RowsPlan &plan, float *workspace, int64_t workspace_floats, GemmChain *chain);

}  // namespace dj
