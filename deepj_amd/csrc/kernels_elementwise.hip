// Element-wise, broadcast and data-movement kernels of the 42 primitive opcodes
// (semantics: CpuBackend.java:56-132,190-214,300-354,466-489,542-549 in the
// reference) plus the small fused inference helpers.  All of them are HBM
// bound: one pass, 128-bit accesses where the length allows it, grid sized to
// a multiple of the 256 CUs.
//
// Transcendentals follow the CPU backend's convention - evaluate in f64, cast
// to fp32 (CpuBackend.java:24-28) - so a GPU result differs from the CPU one by
// at most the last f64 bit of the math library, not by an fp32 approximation.
#include "dj_common.h"

namespace dj {
namespace {

constexpr int kThreads = 256;

inline int grid_for(int64_t work_items, int per_thread = 1) {
    int64_t blocks = (work_items + (int64_t)kThreads * per_thread - 1) / ((int64_t)kThreads * per_thread);
    if (blocks < 1) blocks = 1;
    if (blocks > 256 * 32) blocks = 256 * 32;      // grid-stride beyond 32 blocks per CU
    return (int)blocks;
}

__device__ __forceinline__ float d_exp(float x) { return (float)exp((double)x); }
__device__ __forceinline__ float d_log(float x) { return (float)log((double)x); }
__device__ __forceinline__ float d_tanh(float x) { return (float)tanh((double)x); }
__device__ __forceinline__ float d_pow(float x, float e) { return (float)pow((double)x, (double)e); }
__device__ __forceinline__ float d_sigmoid(float x) { return 1.0f / (1.0f + d_exp(-x)); }

__device__ __forceinline__ float d_gelu(float x) {
    float c = sqrtf(2.0f / 3.14159265358979323846f);
    float x3 = x * x * x;
    float t = c * (x + 0.044715f * x3);
    return 0.5f * x * (1.0f + d_tanh(t));
}
__device__ __forceinline__ float d_gelu_deriv(float x) {
    float c = sqrtf(2.0f / 3.14159265358979323846f);
    float x2 = x * x;
    float x3 = x2 * x;
    float t = c * (x + 0.044715f * x3);
    float th = d_tanh(t);
    float sech2 = 1.0f - th * th;
    float dtdx = c * (1.0f + 3.0f * 0.044715f * x2);
    return 0.5f * (1.0f + th) + 0.5f * x * sech2 * dtdx;
}

template <int OP> __device__ __forceinline__ float binary_op(float x, float y) {
    if constexpr (OP == DJ_OP_ADD) return x + y;
    if constexpr (OP == DJ_OP_SUBTRACT) return x - y;
    if constexpr (OP == DJ_OP_MULTIPLY) return x * y;
    if constexpr (OP == DJ_OP_DIVIDE) return x / y;
    if constexpr (OP == DJ_OP_RELU_BACKWARD) return x > 0.0f ? y : 0.0f;
    if constexpr (OP == DJ_OP_GELU_BACKWARD) return y * d_gelu_deriv(x);
    return 0.0f;
}

template <int OP> __device__ __forceinline__ float unary_op(float x) {
    if constexpr (OP == DJ_OP_SQRT) return sqrtf(x);          // correctly rounded, as (float)Math.sqrt
    if constexpr (OP == DJ_OP_NEG) return -x;
    if constexpr (OP == DJ_OP_EXP) return d_exp(x);
    if constexpr (OP == DJ_OP_LOG) return d_log(x);
    if constexpr (OP == DJ_OP_TANH) return d_tanh(x);
    if constexpr (OP == DJ_OP_SIGMOID) return d_sigmoid(x);
    if constexpr (OP == DJ_OP_RELU) return x > 0.0f ? x : (x != x ? x : 0.0f);
    if constexpr (OP == DJ_OP_GELU) return d_gelu(x);
    return 0.0f;
}

template <int OP> __device__ __forceinline__ float scalar_op(float x, float s0, float s1) {
    if constexpr (OP == DJ_OP_MULTIPLY_SCALAR) return x * s0;
    if constexpr (OP == DJ_OP_ADD_SCALAR) return x + s0;
    if constexpr (OP == DJ_OP_DIVIDE_SCALAR) return x / s0;
    if constexpr (OP == DJ_OP_POW) return d_pow(x, s0);
    if constexpr (OP == DJ_OP_CLAMP) {                         // Math.min(max, Math.max(min, x))
        float mx = x > s0 ? x : s0;
        if (x != x) mx = x;
        float mn = mx < s1 ? mx : s1;
        if (mx != mx) mn = mx;
        return mn;
    }
    return 0.0f;
}

template <int OP>
__global__ void __launch_bounds__(kThreads) k_binary(const float *__restrict__ a, const float *__restrict__ b,
                                                     float *__restrict__ out, int64_t n) {
    int64_t n4 = n >> 2;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const float4 *a4 = reinterpret_cast<const float4 *>(a);
    const float4 *b4 = reinterpret_cast<const float4 *>(b);
    float4 *o4 = reinterpret_cast<float4 *>(out);
    for (int64_t i = tid; i < n4; i += stride) {
        float4 x = a4[i], y = b4[i], r;
        r.x = binary_op<OP>(x.x, y.x); r.y = binary_op<OP>(x.y, y.y);
        r.z = binary_op<OP>(x.z, y.z); r.w = binary_op<OP>(x.w, y.w);
        o4[i] = r;
    }
    for (int64_t i = (n4 << 2) + tid; i < n; i += stride) out[i] = binary_op<OP>(a[i], b[i]);
}

template <int OP>
__global__ void __launch_bounds__(kThreads) k_unary(const float *__restrict__ a, float *__restrict__ out, int64_t n) {
    int64_t n4 = n >> 2;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const float4 *a4 = reinterpret_cast<const float4 *>(a);
    float4 *o4 = reinterpret_cast<float4 *>(out);
    for (int64_t i = tid; i < n4; i += stride) {
        float4 x = a4[i], r;
        r.x = unary_op<OP>(x.x); r.y = unary_op<OP>(x.y); r.z = unary_op<OP>(x.z); r.w = unary_op<OP>(x.w);
        o4[i] = r;
    }
    for (int64_t i = (n4 << 2) + tid; i < n; i += stride) out[i] = unary_op<OP>(a[i]);
}

template <int OP>
__global__ void __launch_bounds__(kThreads) k_scalar(const float *__restrict__ a, float *__restrict__ out,
                                                     float s0, float s1, int64_t n) {
    int64_t n4 = n >> 2;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const float4 *a4 = reinterpret_cast<const float4 *>(a);
    float4 *o4 = reinterpret_cast<float4 *>(out);
    for (int64_t i = tid; i < n4; i += stride) {
        float4 x = a4[i], r;
        r.x = scalar_op<OP>(x.x, s0, s1); r.y = scalar_op<OP>(x.y, s0, s1);
        r.z = scalar_op<OP>(x.z, s0, s1); r.w = scalar_op<OP>(x.w, s0, s1);
        o4[i] = r;
    }
    for (int64_t i = (n4 << 2) + tid; i < n; i += stride) out[i] = scalar_op<OP>(a[i], s0, s1);
}

// Division of i < 2^31 by a fixed d: the high word of i * m, shifted.
struct FastDiv {
    uint32_t d, m, shift;
    explicit FastDiv(uint32_t divisor) : d(divisor), m(0), shift(0) {
        if (d == 1) return;
        while ((1ull << shift) < d) shift++;                         // ceil(log2 d)
        m = (uint32_t)(((1ull << (31 + shift)) + d - 1) / d);        // exact for i < 2^31 (31 + shift bits of 1 / d, rounded up)
        shift--;
    }
    __device__ __forceinline__ uint32_t div(uint32_t i) const { return d == 1 ? i : __umulhi(i, m) >> shift; }
};

// out[r,c] = a[r,c] (op) v[c]  (ROWVEC)  or  a[r,c] (op) v[r]  (column vector).  Bound by memory: four values a thread
// whatever the width (a group may run over the end of its row), one division by multiplication for the four - 64-bit
// divisions, one a value, made 500 x 2752 take 5.5 us; 3.3 now.
template <int OP, bool ROWVEC>
__global__ void __launch_bounds__(kThreads) k_broadcast(const float *__restrict__ a, const float *__restrict__ v,
                                                        float *__restrict__ out, int64_t n, int cols, const FastDiv by_cols) {
    const int64_t stride = (int64_t)gridDim.x * kThreads, n4 = n >> 2;
    const int64_t tid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    for (int64_t i = tid; i < n4; i += stride) {
        const float4 x = reinterpret_cast<const float4 *>(a)[i];
        uint32_t r = by_cols.div((uint32_t)(4 * i)), c = (uint32_t)(4 * i) - r * (uint32_t)cols;
        const float xs[4] = {x.x, x.y, x.z, x.w};
        float o[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            o[u] = binary_op<OP>(xs[u], ROWVEC ? v[c] : v[r]);
            if (++c == (uint32_t)cols) { c = 0; r++; }
        }
        reinterpret_cast<float4 *>(out)[i] = make_float4(o[0], o[1], o[2], o[3]);
    }
    for (int64_t i = (n4 << 2) + tid; i < n; i += stride) {
        const uint32_t r = by_cols.div((uint32_t)i), c = (uint32_t)i - r * (uint32_t)cols;
        out[i] = binary_op<OP>(a[i], ROWVEC ? v[c] : v[r]);
    }
}

// Consecutive element-wise operations over the same elements (Chain): every operand from memory once, all requested together,
// values between operations in LDS (a slot per thread: operations and slots are data, and registers cannot be indexed by
// data), every result to its buffer.  The same expressions as the kernels above: the same bits.  Bound by its instructions (16
// bytes of 500 x 2752 take 12.7 us through four operations, the four kernels' 12.4 with their operands in the L2) and by the
// launch below that; what it saves is launches and operands that come from further away (bias, bias, sigmoid and two products
// behind two matrix products: 27.6 -> 16.5 us in a trace).  The feed-forward layer of 500 rows 177 -> 169 us, six training
// steps 2270 -> 2190.
struct ChainArgs { Chain chain; FastDiv by_cols; };

__device__ __forceinline__ float chain_op(int op, float x, float y, float s0, float s1) {
    switch (op) {                                            // uniform
        case DJ_OP_ADD: return binary_op<DJ_OP_ADD>(x, y);
        case DJ_OP_SUBTRACT: return binary_op<DJ_OP_SUBTRACT>(x, y);
        case DJ_OP_MULTIPLY: return binary_op<DJ_OP_MULTIPLY>(x, y);
        case DJ_OP_DIVIDE: return binary_op<DJ_OP_DIVIDE>(x, y);
        case DJ_OP_RELU_BACKWARD: return binary_op<DJ_OP_RELU_BACKWARD>(x, y);
        case DJ_OP_GELU_BACKWARD: return binary_op<DJ_OP_GELU_BACKWARD>(x, y);
        case DJ_OP_SQRT: return unary_op<DJ_OP_SQRT>(x);
        case DJ_OP_NEG: return unary_op<DJ_OP_NEG>(x);
        case DJ_OP_EXP: return unary_op<DJ_OP_EXP>(x);
        case DJ_OP_TANH: return unary_op<DJ_OP_TANH>(x);
        case DJ_OP_SIGMOID: return unary_op<DJ_OP_SIGMOID>(x);
        case DJ_OP_RELU: return unary_op<DJ_OP_RELU>(x);
        case DJ_OP_GELU: return unary_op<DJ_OP_GELU>(x);
        case DJ_OP_MULTIPLY_SCALAR: return scalar_op<DJ_OP_MULTIPLY_SCALAR>(x, s0, s1);
        case DJ_OP_ADD_SCALAR: return scalar_op<DJ_OP_ADD_SCALAR>(x, s0, s1);
        case DJ_OP_DIVIDE_SCALAR: return scalar_op<DJ_OP_DIVIDE_SCALAR>(x, s0, s1);
        default: return scalar_op<DJ_OP_CLAMP>(x, s0, s1);
    }
}

// FULL: no vectors, and n a multiple of four.
template <bool FULL>
__global__ void __launch_bounds__(kThreads) k_chain(const ChainArgs args) {
    extern __shared__ float4 slot[];                         // [slots][kThreads]
    const Chain &p = args.chain;
    const int t = threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * kThreads, groups = (p.n + 3) >> 2;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + t; i < groups; i += stride) {
        const uint32_t first = (uint32_t)(4 * i);
        const int count = FULL || 4 * i + 4 <= p.n ? 4 : (int)(p.n - 4 * i);
        const bool whole = FULL || count == 4;
        float4 v[kChainExt];
#pragma unroll
        for (int j = 0; j < kChainExt; j++) {
            if (j >= p.n_ext) break;
            const ChainExt e = p.ext[j];
            if (FULL || (e.kind == 0 && whole)) {
                v[j] = reinterpret_cast<const float4 *>(e.p)[i];
            } else {
                uint32_t r = args.by_cols.div(first), c = first - r * (uint32_t)p.cols;
                float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    if (u < count) x[u] = e.p[e.kind == 0 ? first + u : e.kind == 1 ? c : r];
                    if (++c == (uint32_t)p.cols) { c = 0; r++; }
                }
                v[j] = make_float4(x[0], x[1], x[2], x[3]);
            }
        }
#pragma unroll
        for (int j = 0; j < kChainExt; j++)
            if (j < p.n_ext) slot[j * kThreads + t] = v[j];
        ChainOp q = p.ops[0];
#pragma unroll 1
        for (int o = 0; o < p.n_ops; o++) {
            const ChainOp next = p.ops[o + 1 < p.n_ops ? o + 1 : o];       // (requested before this one's work)
            const float4 x = slot[q.a * kThreads + t], y = slot[q.b * kThreads + t];
            const float4 r = make_float4(chain_op(q.op, x.x, y.x, q.s0, q.s1), chain_op(q.op, x.y, y.y, q.s0, q.s1),
                                         chain_op(q.op, x.z, y.z, q.s0, q.s1), chain_op(q.op, x.w, y.w, q.s0, q.s1));
            slot[q.dst * kThreads + t] = r;
            if (whole) {
                reinterpret_cast<float4 *>(q.out)[i] = r;
            } else {
                const float rs[3] = {r.x, r.y, r.z};
#pragma unroll
                for (int u = 0; u < 3; u++)
                    if (u < count) q.out[first + u] = rs[u];
            }
            q = next;
        }
    }
}

// 32x32 tile through LDS (+1 padding: no bank conflicts on the transposed read).
__device__ __forceinline__ void transpose_tile(const float *__restrict__ a, float *__restrict__ out, int rows, int cols, int c0, int r0) {
    __shared__ float tile[32][33];
    int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;     // 32 x 8
    for (int j = ty; j < 32; j += 8) {
        int r = r0 + j, c = c0 + tx;
        if (r < rows && c < cols) tile[j][tx] = a[(int64_t)r * cols + c];
    }
    __syncthreads();
    for (int j = ty; j < 32; j += 8) {
        int c = c0 + j, r = r0 + tx;                       // out is [cols x rows]
        if (r < rows && c < cols) out[(int64_t)c * rows + r] = tile[tx][j];
    }
}
__global__ void __launch_bounds__(256) k_transpose(const float *__restrict__ a, float *__restrict__ out, int rows,
                                                   int cols) {
    transpose_tile(a, out, rows, cols, blockIdx.x * 32, blockIdx.y * 32);
}
// Bound by its launch, as each of them by itself: six of a training step's (256 x 192 to 192 x 1003) and a small operation behind
// them 20.0 us, 9.2 in one; six training steps 2290 -> 2195.
__global__ void __launch_bounds__(256) k_transposes(const Transposes all) {
    Transpose t = all.t[0];
#pragma unroll
    for (int i = 1; i < kTransposes; i++)
        if (i < all.count && (int)blockIdx.x >= all.t[i].first) t = all.t[i];
    const int b = blockIdx.x - t.first, r = b / t.across;
    transpose_tile(t.a, t.out, t.rows, t.cols, (b - r * t.across) * 32, r * 32);
}

// One grid row per tensor: the parameters of a model are stepped one behind the other, and a launch for each cost more than
// the update of most (nine tensors of 0.6 M values in all: 22 us in nine launches, 6 in one).
__global__ void __launch_bounds__(kThreads) k_adamw(const AdamTensors tensors) {
    const AdamTensor p = tensors.t[blockIdx.y];
    const int64_t stride = (int64_t)gridDim.x * kThreads, tid = (int64_t)blockIdx.x * kThreads + threadIdx.x, n4 = p.n >> 2;
    auto step = [&](float w, float grad, float &m, float &v) {
        m = p.beta1 * m + (1.0f - p.beta1) * grad;
        v = p.beta2 * v + (1.0f - p.beta2) * (grad * grad);
        const float m_hat = m / p.bc1, v_hat = v / p.bc2;
        float update = (p.lr * m_hat) / (sqrtf(v_hat) + p.eps);
        if (p.wd != 0.0f) update += p.lr * p.wd * w;
        return w - update;
    };
    for (int64_t i = tid; i < n4; i += stride) {
        float4 w = reinterpret_cast<float4 *>(p.w)[i], m = reinterpret_cast<float4 *>(p.mt)[i], v = reinterpret_cast<float4 *>(p.vt)[i];
        const float4 g = reinterpret_cast<const float4 *>(p.g)[i];
        w.x = step(w.x, g.x, m.x, v.x); w.y = step(w.y, g.y, m.y, v.y);
        w.z = step(w.z, g.z, m.z, v.z); w.w = step(w.w, g.w, m.w, v.w);
        reinterpret_cast<float4 *>(p.mt)[i] = m;
        reinterpret_cast<float4 *>(p.vt)[i] = v;
        reinterpret_cast<float4 *>(p.w)[i] = w;
    }
    for (int64_t i = (n4 << 2) + tid; i < p.n; i += stride) p.w[i] = step(p.w[i], p.g[i], p.mt[i], p.vt[i]);
}

// target[idx[i], c] += grad[i, c]; indices arrive as floats (MetalBackend.java:43-54),
// rows outside the target are skipped (deepj_metal_jni.mm:606-607).
__global__ void __launch_bounds__(kThreads) k_scatter_add(float *__restrict__ target, const float *__restrict__ idx,
                                                          const float *__restrict__ grad, int target_rows, int cols,
                                                          int n_idx) {
    int64_t n = (int64_t)n_idx * cols;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride) {
        int i = (int)(t / cols);
        int c = (int)(t - (int64_t)i * cols);
        float fi = idx[i];
        if (!(fi >= 0.0f) || fi >= (float)target_rows) continue;
        int row = (int)fi;
        atomicAdd(&target[(int64_t)row * cols + c], grad[t]);
    }
}

__global__ void __launch_bounds__(kThreads) k_fill(uint32_t *__restrict__ dst, uint32_t bits, int64_t n) {
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = bits;
}

// Measurement floor of the HBM-bound decode kernels: the same bytes read with 128-bit loads, D in flight per lane,
// nothing computed but an AND over the words (so that no load can be dropped) and nothing stored unless every bit of
// the buffer is set.
template <int D>
__global__ void __launch_bounds__(kThreads) k_stream_read(const uint4 *__restrict__ src, uint32_t *__restrict__ sink,
                                                          int64_t n16, int64_t tail_from, const uint32_t *src_words,
                                                          int64_t n_words) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t acc = 0xffffffffu;
    for (; i + (D - 1) * stride < n16; i += D * stride) {
        uint4 v[D];
#pragma unroll
        for (int u = 0; u < D; u++) v[u] = src[i + u * stride];
#pragma unroll
        for (int u = 0; u < D; u++) acc &= v[u].x & v[u].y & v[u].z & v[u].w;
    }
    for (; i < n16; i += stride) { uint4 v = src[i]; acc &= v.x & v.y & v.z & v.w; }
    for (int64_t j = tail_from + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n_words; j += stride) acc &= src_words[j];
    if (acc == 0xffffffffu && n_words > 0 && src_words[0] == 0xffffffffu) sink[0] = acc;     // practically never
}

__global__ void k_nop() {}

__global__ void __launch_bounds__(kThreads) k_copy(const float *__restrict__ src, float *__restrict__ dst, int64_t n) {
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

// Uploads that were staged in pinned memory since the last launch, one grid row each.  Bound by the link (1 MiB in 22 us) and
// below that by the launch: one launch costs the host 2.4 us, so eight uploads of a flush cost 2.4 instead of the
// 8 x (sync + copy) = 75 us that a copy call per upload took.
__global__ void __launch_bounds__(kThreads) k_upload_pieces(const UploadPieces pieces) {
    const UploadPiece p = pieces.p[blockIdx.y];
    const int64_t n4 = p.n >> 2;
    const int64_t stride = (int64_t)gridDim.x * kThreads, tid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    for (int64_t i = tid; i < n4; i += stride) reinterpret_cast<float4 *>(p.dst)[i] = reinterpret_cast<const float4 *>(p.src)[i];
    if (tid < p.n - (n4 << 2)) p.dst[(n4 << 2) + tid] = p.src[(n4 << 2) + tid];
}

// dst (pinned host memory) = src, in chunks dealt to the workgroups in order; a chunk's workgroup stores `tag` in
// flags[chunk] once the chunk is there, so the host takes the chunks out while later ones are still on the link and never
// waits for a queue to drain (flag and spin 9 us after a launch, hipStreamSynchronize 11, a copy call into pageable
// memory 23 before it and 250 for 4 MiB, of which 86 are the link's).
__global__ void __launch_bounds__(kThreads) k_download(const float *__restrict__ src, float *__restrict__ dst, int64_t n,
                                                       int64_t chunk_floats, uint32_t *__restrict__ flags, uint32_t tag) {
    const int64_t chunks = (n + chunk_floats - 1) / chunk_floats;
    for (int64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        const int64_t from = c * chunk_floats, len = n - from < chunk_floats ? n - from : chunk_floats, n4 = len >> 2;
        const float4 *s4 = reinterpret_cast<const float4 *>(src + from);
        float4 *d4 = reinterpret_cast<float4 *>(dst + from);
        for (int64_t i = threadIdx.x; i < n4; i += 4 * kThreads) {
            float4 v[4];
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (i + u * kThreads < n4) v[u] = s4[i + u * kThreads];
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (i + u * kThreads < n4) d4[i + u * kThreads] = v[u];
        }
        if (threadIdx.x < len - (n4 << 2)) dst[from + (n4 << 2) + threadIdx.x] = src[from + (n4 << 2) + threadIdx.x];
        __threadfence_system();              // every thread's stores are in host memory ...
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(flags + c, tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);   // ... before the flag is
    }
}

// SiLU.java:20-24 then SwiGLULayer.java:69: (g * sigmoid(g)) * up
__global__ void __launch_bounds__(kThreads) k_silu_mul(const float *__restrict__ gate, const float *__restrict__ up,
                                                       float *__restrict__ out, int64_t n) {
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        float g = gate[i];
        float sg = g * d_sigmoid(g);
        out[i] = sg * up[i];
    }
}

// Embedding.java:28-34 (Tensor.sliceRows): out[i,:] = table[ids[i],:].  Ids were range
// checked on the host when they came from the host; ids produced on the device
// (argmax) are always < vocab.  An out-of-range id writes NaN instead of reading.
__global__ void __launch_bounds__(kThreads) k_embed_gather(const float *__restrict__ table,
                                                           const int32_t *__restrict__ ids, float *__restrict__ out,
                                                           int n_ids, int d, int vocab) {
    int i = blockIdx.x;
    if (i >= n_ids) return;
    int id = ids[i];
    bool ok = id >= 0 && id < vocab;
    const float *src = table + (int64_t)(ok ? id : 0) * d;
    float *dst = out + (int64_t)i * d;
    for (int c = threadIdx.x; c < d; c += blockDim.x) dst[c] = ok ? src[c] : __builtin_nanf("");
}

// dst[(state[0] + i), :] = src[i, :] for i < rows: append to a cache whose fill level lives on the device.
__global__ void __launch_bounds__(kThreads) k_append_rows(const float *__restrict__ src, float *__restrict__ dst,
                                                          const int32_t *__restrict__ state, int rows, int row_floats,
                                                          int max_rows) {
    const int pos0 = state[0];
    int64_t n = (int64_t)rows * row_floats;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride) {
        int i = (int)(t / row_floats);
        int j = (int)(t - (int64_t)i * row_floats);
        int r = pos0 + i;
        if (r >= 0 && r < max_rows) dst[(int64_t)r * row_floats + j] = src[t];
    }
}

// state[0] = positions held in the cache, state[1] = current token, state[2] = tokens generated.
__global__ void k_decode_advance(int32_t *state, const int32_t *token, int32_t *tokens, int capacity,
                                 int n_positions) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        int32_t t = token[0];
        int32_t g = state[2];
        if (g < capacity) tokens[g] = t;
        state[1] = t;
        state[0] = state[0] + n_positions;
        state[2] = g + 1;
    }
}

}  // namespace

#define DJ_LAUNCH(kernel, grid, block, stream, ...) \
    launch_kernel(kernel, dim3(grid), dim3(block), 0, stream, __VA_ARGS__)

void launch_binary(hipStream_t s, int op, const float *a, const float *b, float *out, int64_t n) {
    if (n <= 0) return;
    int grid = grid_for(n, 4);
    switch (op) {
        case DJ_OP_ADD: DJ_LAUNCH(k_binary<DJ_OP_ADD>, grid, kThreads, s, a, b, out, n); break;
        case DJ_OP_SUBTRACT: DJ_LAUNCH(k_binary<DJ_OP_SUBTRACT>, grid, kThreads, s, a, b, out, n); break;
        case DJ_OP_MULTIPLY: DJ_LAUNCH(k_binary<DJ_OP_MULTIPLY>, grid, kThreads, s, a, b, out, n); break;
        case DJ_OP_DIVIDE: DJ_LAUNCH(k_binary<DJ_OP_DIVIDE>, grid, kThreads, s, a, b, out, n); break;
        case DJ_OP_RELU_BACKWARD: DJ_LAUNCH(k_binary<DJ_OP_RELU_BACKWARD>, grid, kThreads, s, a, b, out, n); break;
        case DJ_OP_GELU_BACKWARD: DJ_LAUNCH(k_binary<DJ_OP_GELU_BACKWARD>, grid, kThreads, s, a, b, out, n); break;
        default: fail("launch_binary: bad op");
    }
}

void launch_unary(hipStream_t s, int op, const float *a, float *out, int64_t n) {
    if (n <= 0) return;
    int grid = grid_for(n, 4);
    switch (op) {
        case DJ_OP_SQRT: DJ_LAUNCH(k_unary<DJ_OP_SQRT>, grid, kThreads, s, a, out, n); break;
        case DJ_OP_NEG: DJ_LAUNCH(k_unary<DJ_OP_NEG>, grid, kThreads, s, a, out, n); break;
        case DJ_OP_EXP: DJ_LAUNCH(k_unary<DJ_OP_EXP>, grid, kThreads, s, a, out, n); break;
        case DJ_OP_LOG: DJ_LAUNCH(k_unary<DJ_OP_LOG>, grid, kThreads, s, a, out, n); break;
        case DJ_OP_TANH: DJ_LAUNCH(k_unary<DJ_OP_TANH>, grid, kThreads, s, a, out, n); break;
        case DJ_OP_SIGMOID: DJ_LAUNCH(k_unary<DJ_OP_SIGMOID>, grid, kThreads, s, a, out, n); break;
        case DJ_OP_RELU: DJ_LAUNCH(k_unary<DJ_OP_RELU>, grid, kThreads, s, a, out, n); break;
        case DJ_OP_GELU: DJ_LAUNCH(k_unary<DJ_OP_GELU>, grid, kThreads, s, a, out, n); break;
        default: fail("launch_unary: bad op");
    }
}

void launch_scalar(hipStream_t s, int op, const float *a, float *out, float s0, float s1, int64_t n) {
    if (n <= 0) return;
    int grid = grid_for(n, 4);
    switch (op) {
        case DJ_OP_MULTIPLY_SCALAR: DJ_LAUNCH(k_scalar<DJ_OP_MULTIPLY_SCALAR>, grid, kThreads, s, a, out, s0, s1, n); break;
        case DJ_OP_ADD_SCALAR: DJ_LAUNCH(k_scalar<DJ_OP_ADD_SCALAR>, grid, kThreads, s, a, out, s0, s1, n); break;
        case DJ_OP_DIVIDE_SCALAR: DJ_LAUNCH(k_scalar<DJ_OP_DIVIDE_SCALAR>, grid, kThreads, s, a, out, s0, s1, n); break;
        case DJ_OP_POW: DJ_LAUNCH(k_scalar<DJ_OP_POW>, grid, kThreads, s, a, out, s0, s1, n); break;
        case DJ_OP_CLAMP: DJ_LAUNCH(k_scalar<DJ_OP_CLAMP>, grid, kThreads, s, a, out, s0, s1, n); break;
        default: fail("launch_scalar: bad op");
    }
}

void launch_broadcast(hipStream_t s, int op, const float *a, const float *v, float *out, int rows, int cols) {
    int64_t n = (int64_t)rows * cols;
    if (n <= 0) return;
    if (n > 0x7fffffffLL) fail("broadcast: more than 2^31 values");
    int grid = grid_for(n, 4);
    const FastDiv by_cols((uint32_t)cols);
    switch (op) {
        case DJ_OP_ADD_ROW_VECTOR:
            DJ_LAUNCH((k_broadcast<DJ_OP_ADD, true>), grid, kThreads, s, a, v, out, n, cols, by_cols); break;
        case DJ_OP_MULTIPLY_BROADCAST_ROWS:
            DJ_LAUNCH((k_broadcast<DJ_OP_MULTIPLY, true>), grid, kThreads, s, a, v, out, n, cols, by_cols); break;
        case DJ_OP_ADD_BROADCAST_COLS:
            DJ_LAUNCH((k_broadcast<DJ_OP_ADD, false>), grid, kThreads, s, a, v, out, n, cols, by_cols); break;
        case DJ_OP_SUBTRACT_BROADCAST_COLS:
            DJ_LAUNCH((k_broadcast<DJ_OP_SUBTRACT, false>), grid, kThreads, s, a, v, out, n, cols, by_cols); break;
        case DJ_OP_DIVIDE_BROADCAST_COLS:
            DJ_LAUNCH((k_broadcast<DJ_OP_DIVIDE, false>), grid, kThreads, s, a, v, out, n, cols, by_cols); break;
        case DJ_OP_MULTIPLY_BROADCAST_COLS:
            DJ_LAUNCH((k_broadcast<DJ_OP_MULTIPLY, false>), grid, kThreads, s, a, v, out, n, cols, by_cols); break;
        default: fail("launch_broadcast: bad op");
    }
}

bool chain_takes(int op) {      // (the logarithm and the power are rare, and their code would double the kernel)
    switch (op) {
        case DJ_OP_ADD: case DJ_OP_SUBTRACT: case DJ_OP_MULTIPLY: case DJ_OP_DIVIDE: case DJ_OP_RELU_BACKWARD: case DJ_OP_GELU_BACKWARD:
        case DJ_OP_SQRT: case DJ_OP_NEG: case DJ_OP_EXP: case DJ_OP_TANH: case DJ_OP_SIGMOID: case DJ_OP_RELU: case DJ_OP_GELU:
        case DJ_OP_MULTIPLY_SCALAR: case DJ_OP_ADD_SCALAR: case DJ_OP_DIVIDE_SCALAR: case DJ_OP_CLAMP: return true;
        default: return false;
    }
}
void launch_chain(hipStream_t s, const Chain &chain) {
    if (chain.n <= 0) return;
    const ChainArgs args{chain, FastDiv((uint32_t)chain.cols)};
    bool full = (chain.n & 3) == 0;
    int slots = chain.n_ext;
    for (int j = 0; j < chain.n_ext; j++) full = full && chain.ext[j].kind == 0;
    for (int o = 0; o < chain.n_ops; o++) slots = std::max(slots, chain.ops[o].dst + 1);
    const size_t lds = (size_t)slots * kThreads * sizeof(float4);
    if (full) launch_kernel(k_chain<true>, dim3(grid_for(chain.n, 4)), dim3(kThreads), lds, s, args);
    else launch_kernel(k_chain<false>, dim3(grid_for(chain.n, 4)), dim3(kThreads), lds, s, args);
}

void launch_transpose(hipStream_t s, const float *a, float *out, int rows, int cols) {
    if (rows <= 0 || cols <= 0) return;
    dim3 grid((cols + 31) / 32, (rows + 31) / 32);
    launch_kernel(k_transpose, grid, dim3(256), 0, s, a, out, rows, cols);
}

void launch_transposes(hipStream_t s, Transposes &all) {
    int first = 0;
    for (int i = 0; i < all.count; i++) {
        Transpose &t = all.t[i];
        t.first = first;
        t.across = (t.cols + 31) / 32;
        first += t.across * ((t.rows + 31) / 32);
    }
    launch_kernel(k_transposes, dim3(first), dim3(256), 0, s, all);
}

void launch_adamw(hipStream_t s, const AdamTensors &tensors, int count) {
    int64_t most = 0;
    for (int i = 0; i < count; i++) most = tensors.t[i].n > most ? tensors.t[i].n : most;
    if (most <= 0) return;
    launch_kernel(k_adamw, dim3(grid_for(most, 4), count), dim3(kThreads), 0, s, tensors);
}

void launch_scatter_add(hipStream_t s, float *target, const float *idx, const float *grad, int target_rows, int cols,
                        int n_idx) {
    int64_t n = (int64_t)n_idx * cols;
    if (n <= 0) return;
    DJ_LAUNCH(k_scatter_add, grid_for(n), kThreads, s, target, idx, grad, target_rows, cols, n_idx);
}

void launch_fill(hipStream_t s, uint32_t *dst, uint32_t bits, int64_t n) {
    if (n <= 0) return;
    DJ_LAUNCH(k_fill, grid_for(n), kThreads, s, dst, bits, n);
}

void launch_stream_read(hipStream_t s, const float *src, float *sink, int64_t n) {
    if (n <= 0) return;
    const int64_t n16 = n / 4, per_lane = (n16 + kThreads - 1) / kThreads;    // 128-bit loads a lane would issue in a grid of one
    // as many loads in flight per lane as leave at least two workgroups per CU, at most three (the matvec's grid)
    int depth = 8;
    while (depth > 1 && per_lane / depth < 512) depth >>= 1;
    int64_t grid = (per_lane + depth - 1) / depth;
    if (grid > 768) grid = 768;
    if (grid < 1) grid = 1;
    const uint4 *p = reinterpret_cast<const uint4 *>(src);
    uint32_t *o = reinterpret_cast<uint32_t *>(sink);
    const uint32_t *w = reinterpret_cast<const uint32_t *>(src);
    switch (depth) {
        case 8: launch_kernel(k_stream_read<8>, dim3((int)grid), dim3(kThreads), 0, s, p, o, n16, n16 * 4, w, n); break;
        case 4: launch_kernel(k_stream_read<4>, dim3((int)grid), dim3(kThreads), 0, s, p, o, n16, n16 * 4, w, n); break;
        case 2: launch_kernel(k_stream_read<2>, dim3((int)grid), dim3(kThreads), 0, s, p, o, n16, n16 * 4, w, n); break;
        default: launch_kernel(k_stream_read<1>, dim3((int)grid), dim3(kThreads), 0, s, p, o, n16, n16 * 4, w, n); break;
    }
}

// One wavefront that writes (shader clock counter, 100 MHz wall clock) pairs, `samples` of them, with naps of
// sleep_reps x 127 x 64 clocks in between: run beside other work, the pairs give the shader clock over time.  Both
// loops are bounded by arguments; nothing waits for anyone.
__global__ void __launch_bounds__(64) k_clock_probe(unsigned long long *out, int samples, int sleep_reps) {
    if (threadIdx.x != 0) return;
    for (int i = 0; i < samples; i++) {
        const unsigned long long c = clock64(), w = wall_clock64();
        __hip_atomic_store(out + 2 * i, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(out + 2 * i + 1, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int j = 0; j < sleep_reps; j++) __builtin_amdgcn_s_sleep(127);
    }
}
// the wall clock at this point of a stream
__global__ void k_wall_stamp(unsigned long long *out) { if (threadIdx.x == 0) *out = wall_clock64(); }

void launch_clock_probe(hipStream_t s, unsigned long long *out, int samples, int sleep_reps) {
    hipLaunchKernelGGL(k_clock_probe, dim3(1), dim3(64), 0, s, out, samples, sleep_reps);
}
void launch_wall_stamp(hipStream_t s, unsigned long long *out) { hipLaunchKernelGGL(k_wall_stamp, dim3(1), dim3(64), 0, s, out); }

void launch_nop(hipStream_t s, int grid) {
    launch_kernel(k_nop, dim3(grid < 1 ? 1 : grid), dim3(kThreads), 0, s);
}

void launch_copy(hipStream_t s, const float *src, float *dst, int64_t n) {
    if (n <= 0) return;
    DJ_LAUNCH(k_copy, grid_for(n), kThreads, s, src, dst, n);
}

void launch_upload_pieces(hipStream_t s, const UploadPieces &pieces, int count) {
    int64_t most = 0;
    for (int i = 0; i < count; i++) most = pieces.p[i].n > most ? pieces.p[i].n : most;
    int64_t blocks = (most / 4 + kThreads - 1) / kThreads;       // one 128-bit word a thread up to 64 workgroups a piece
    blocks = blocks < 1 ? 1 : blocks > 64 ? 64 : blocks;
    launch_kernel(k_upload_pieces, dim3((int)blocks, count), dim3(kThreads), 0, s, pieces);
}

void launch_download(hipStream_t s, const float *src, float *dst, int64_t n, int64_t chunk_floats, uint32_t *flags, uint32_t tag) {
    // 64 workgroups keep the link busy; a chunk each up to there, then in turn (so that the first chunks arrive first)
    const int64_t chunks = (n + chunk_floats - 1) / chunk_floats;
    launch_kernel(k_download, dim3((int)(chunks < 64 ? chunks : 64)), dim3(kThreads), 0, s, src, dst, n, chunk_floats, flags, tag);
}

void launch_silu_mul(hipStream_t s, const float *gate, const float *up, float *out, int64_t n) {
    if (n <= 0) return;
    DJ_LAUNCH(k_silu_mul, grid_for(n), kThreads, s, gate, up, out, n);
}

void launch_append_rows(hipStream_t s, const float *src, float *dst, const int32_t *state, int rows, int row_floats,
                        int max_rows) {
    int64_t n = (int64_t)rows * row_floats;
    if (n <= 0) return;
    DJ_LAUNCH(k_append_rows, grid_for(n), kThreads, s, src, dst, state, rows, row_floats, max_rows);
}

void launch_embed_gather(hipStream_t s, const float *table, const int32_t *ids, float *out, int n_ids, int d,
                         int vocab) {
    if (n_ids <= 0) return;
    DJ_LAUNCH(k_embed_gather, n_ids, kThreads, s, table, ids, out, n_ids, d, vocab);
}

void launch_decode_advance(hipStream_t s, int32_t *state, const int32_t *token, int32_t *tokens, int capacity,
                           int n_positions) {
    DJ_LAUNCH(k_decode_advance, 1, 64, s, state, token, tokens, capacity, n_positions);
}

}  // namespace dj
