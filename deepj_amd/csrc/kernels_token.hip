// A run of tokens of a decoder model in one launch.
//
// One row of a model is a chain of dependent products, five a block.  As a launch each, a product costs 2.6 to 7 us of which
// its bytes are the smaller part: the launch 1.4, the previous one's result on its way through memory 1, and weights that
// are asked for only then.  Here all compute units stay for the whole run and hand rows to one another:
//   inside an XCD through its L2 (plain stores, loads that pass the L1 by): 0.46 us for 2048 values from 32 workgroups to all of
//   them, barrier included;
//   between XCDs through memory (stores and loads of agent scope): 1.1 us.
// So the XCDs (groups) share a block the way devices would: each takes some heads with their columns of Wo, and some hidden units
// with their columns of the down projection.  Rows cross between groups twice a block, as partial sums: member m of every
// group fetches its slice of all groups' sums, adds them in the groups' order, and gives the slice to its own group.  q | k | v, the
// attention's records and the hidden units never leave their XCD.  A model that one XCD's share of the memory feeds runs on
// one group alone, without the crossings.
//
// Exchange.  A value travels with a tag of its own in one aligned 8-byte word (float, tag), so no flag has to follow the data and
// nothing is cleared: the tag names token, block and phase, and a reader loads until it sees it.  A region is written again one
// block later; before that every reader has sent something the writer waits for - where a product is too narrow to give every
// member a tile, the members say so with a word each (`beat`).  Waits are bounded (kTokenPolls loads, seconds): if the
// device did not hold all workgroups at once, each leaves, the state stays behind the last whole token, *failed tells the host, and the
// plan's launches behind this one leave at their start.
//
// A workgroup is eight wavefronts that speak - make, send and fetch rows, attend - and eight that multiply.  The two meet at
// barriers, the same ones in the same order on both sides (named in the code).
// Weights come in the order in which a wavefront takes them (k_token_pack lays them out once): items of 16 outputs x 64 k, 1 KB in
// the lanes' order and 32 scales.  They go straight to LDS, kRing of them a wavefront, asked for ahead of the phase that is on and by a
// count of their own: the compiler, which sees branches between registers' loads and their uses, waits for all of them at each (16
// blocks of d 2048: 410 us a token with items loaded to registers, where launches take 404).  A phase's first twelve move on to
// registers before its row is there.
// Products run on v_mfma_i32_16x16x64_i8 as in kernels_decode.hip: the activations of 32 k in four signed-byte digits of one
// power of two, the two scale groups of the 64 k in rows of their own.
// The speakers' way has no load that waits for another (norm weights and biases stand at computed places, no table of pointers) and
// nothing kept in memory between phases: each such wait is one for the weights in front of it (GPT 177 us a token, 155 without).
//
// Bound by the serial chain: instructions on the way from a row's arrival to the next one's departure, one every four clocks of a
// wavefront at best (clocks, with the stamps of a DJ_TRACE build in them: a product of one item a wavefront 700 to 1200 from the staged row to
// its sums, an exchange 1300 inside a group and 4700 to 8700 between groups, from the sums to the row), and by
// memory where a block has more than some 20 MB.  Us a token, launches and this: 4 blocks of d 256, 256 words 48.0, 33.0; 8 of d 1024,
// 8192 words 126, 87.7; d 2048, 32000 words, 4 blocks 120, 92, 16 blocks 404, 310; GPT, 12 blocks of 768, 50257 words 200, 137.
// Taken back: one set of wavefronts for everything (256 registers: 51.6 us where this takes 36.5); the heads' records merged
// through LDS; all slots filled behind every phase (372 us at 16 blocks of d 2048 where this took 343); items asked for by the clock
// while the multiplying wavefronts wait (122 us at 4 blocks, where the same by counts took 114); the other groups' sums awaited by several
// wavefronts by turns (GPT 153 where one takes 152); a key tile alone without the other three's weights (registers to memory: 146).
#include <type_traits>

#include "dj_common.h"
#include "dj_device.h"
#include "gemm_rows.h"
#include "token_run.h"

namespace dj {
namespace {
using namespace dev;

typedef int intx4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef unsigned long long word;

constexpr int kWaves = kTokenWaves, kMembers = kTokenMembers;
constexpr int kSpeakers = 64 * kWaves;           // threads that make, send and receive rows; as many multiply
constexpr int kThreads = 2 * kSpeakers;
constexpr int kRing = 12;                        // items of a wavefront in LDS or on their way there (108 KB in all)
constexpr int kTogether = 3;                     // items whose products are made side by side
constexpr int kCrossSleep = 18;                  // of 64 clocks
constexpr int kRed = 12;                         // floats between two outputs' sums (the wavefronts' eight; 16-byte steps over all banks)
constexpr float kLog2e = 1.44269504088896340736f;

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// ── exchange ────────────────────────────────────────────────────────────────
// (addresses as the block's base and a word's index: one register each)
__device__ __forceinline__ void send(word *base, uint32_t at, float v, uint32_t tag, bool far) {
    const word w = (word)tag << 32 | __float_as_uint(v);
    word *const p = reinterpret_cast<word *>(reinterpret_cast<char *>(base) + at * 8u);
    if (far) __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// N times two words, loaded together past the L1 until all of them carry the tag, those of all the wavefront's lanes that are here: one
// count and one branch a try, where lanes that end by themselves cost some forty instructions of masks.  False: they did not in time.
template <int N> struct Words { uintx4 v[N]; };
#define DJ_LD(i, at, base) "global_load_dwordx4 %" #i ", %" #at ", %" #base " sc1\n\t"
__device__ __forceinline__ void fetch(Words<1> &w, const word *b, const uint32_t (&p)[1]) {
    asm volatile(DJ_LD(0, 1, 2) "s_waitcnt vmcnt(0)" : "=&v"(w.v[0]) : "v"(p[0]), "s"(b) : "memory");
}
__device__ __forceinline__ void fetch(Words<2> &w, const word *b, const uint32_t (&p)[2]) {
    asm volatile(DJ_LD(0, 2, 4) DJ_LD(1, 3, 4) "s_waitcnt vmcnt(0)" : "=&v"(w.v[0]), "=&v"(w.v[1]) : "v"(p[0]), "v"(p[1]), "s"(b) : "memory");
}
__device__ __forceinline__ void fetch(Words<3> &w, const word *b, const uint32_t (&p)[3]) {
    asm volatile(DJ_LD(0, 3, 6) DJ_LD(1, 4, 6) DJ_LD(2, 5, 6) "s_waitcnt vmcnt(0)"
                 : "=&v"(w.v[0]), "=&v"(w.v[1]), "=&v"(w.v[2]) : "v"(p[0]), "v"(p[1]), "v"(p[2]), "s"(b) : "memory");
}
__device__ __forceinline__ void fetch(Words<6> &w, const word *b, const uint32_t (&p)[6]) {
    asm volatile(DJ_LD(0, 6, 12) DJ_LD(1, 7, 12) DJ_LD(2, 8, 12) DJ_LD(3, 9, 12) DJ_LD(4, 10, 12) DJ_LD(5, 11, 12) "s_waitcnt vmcnt(0)"
                 : "=&v"(w.v[0]), "=&v"(w.v[1]), "=&v"(w.v[2]), "=&v"(w.v[3]), "=&v"(w.v[4]), "=&v"(w.v[5])
                 : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "s"(b) : "memory");
}
__device__ __forceinline__ void fetch(Words<8> &w, const word *b, const uint32_t (&p)[8]) {
    asm volatile(DJ_LD(0, 8, 16) DJ_LD(1, 9, 16) DJ_LD(2, 10, 16) DJ_LD(3, 11, 16) DJ_LD(4, 12, 16) DJ_LD(5, 13, 16) DJ_LD(6, 14, 16) DJ_LD(7, 15, 16)
                 "s_waitcnt vmcnt(0)"
                 : "=&v"(w.v[0]), "=&v"(w.v[1]), "=&v"(w.v[2]), "=&v"(w.v[3]), "=&v"(w.v[4]), "=&v"(w.v[5]), "=&v"(w.v[6]), "=&v"(w.v[7])
                 : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]), "s"(b) : "memory");
}
#undef DJ_LD
template <int N> __device__ __forceinline__ bool receive(Words<N> &w, const word *base, uint32_t (&p)[N], uint32_t tag, int polls) {
#pragma unroll
    for (int i = 0; i < N; i++) p[i] *= 8;
    bool missing;
    int n = polls;
    do {                                                                 // (once at least: w is written on every way out)
        fetch(w, base, p);
        uint32_t off = 0;
#pragma unroll
        for (int i = 0; i < N; i++) off |= (w.v[i].y ^ tag) | (w.v[i].w ^ tag);
        missing = __builtin_amdgcn_ballot_w64(off != 0) != 0;
    } while (missing && --n > 0);
    return !missing && polls > 0;
}
__device__ __forceinline__ float first(uintx4 v) { return __uint_as_float(v.x); }
__device__ __forceinline__ float second(uintx4 v) { return __uint_as_float(v.z); }
// four values of consecutive words
__device__ __forceinline__ bool receive4(float4 &v, const word *base, uint32_t p, uint32_t tag, int polls) {
    Words<2> w;
    uint32_t at[2] = {p, p + 2};
    const bool ok = receive(w, base, at, tag, polls);
    v = make_float4(first(w.v[0]), second(w.v[0]), first(w.v[1]), second(w.v[1]));
    return ok;
}

// A logit as a key that orders like DECODE_NEXT does: the larger value first, NaN above everything, the lower index on ties.
__device__ __forceinline__ uint64_t logit_key(float v, int i) {
    uint32_t b = __float_as_uint(v == 0.0f ? 0.0f : v);                  // (the two zeros are equal)
    if (v != v) b = 0x7fc00000u;
    return (uint64_t)((b & 0x80000000u) ? ~b : (b | 0x80000000u)) << 32 | (uint32_t)~i;
}
template <int CTRL> __device__ __forceinline__ uint64_t dpp_max(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, 0xf, 0xf, false),
                   hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, 0xf, 0xf, false);
    const uint64_t o = (uint64_t)hi << 32 | lo;
    return o > v ? o : v;
}
// the largest of a wavefront's, in every lane
__device__ __forceinline__ uint64_t wave_most(uint64_t v) {
    v = dpp_max<0xB1>(v);                                                // quad_perm [1,0,3,2]
    v = dpp_max<0x4E>(v);                                                // quad_perm [2,3,0,1]
    v = dpp_max<0x141>(v);                                               // row_half_mirror
    v = dpp_max<0x140>(v);                                               // row_mirror: a 16-lane row
    uint64_t m = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint64_t o = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), 16 * q) << 32 | (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 16 * q);
        m = o > m ? o : m;
    }
    return m;
}

// Timeline of the last block, for tuning builds only (-DDJ_TRACE; never in the shipped library).
#ifdef DJ_TRACE
__device__ unsigned long long g_token_trace[256 * 64];
#define DJ_STAMP(i) do { if (threadIdx.x == 0) g_token_trace[blockIdx.x * 64 + (i)] = clock64(); } while (0)
#define DJ_STAMP2(i) do { if (threadIdx.x == kSpeakers) g_token_trace[blockIdx.x * 64 + 32 + (i)] = clock64(); } while (0)
#else
#define DJ_STAMP(i) do {} while (0)
#define DJ_STAMP2(i) do {} while (0)
#endif

// kSets: of four values of the row a speaking thread (1: rows of up to 2048)
template <int HD, bool GPT, int kSets>
__global__ void __launch_bounds__(kThreads)
k_token_run(TokenRun r) {
    constexpr uint32_t kZeros = 4 * (kSets * 4 * kSpeakers + 64 + 16);   // (16 bytes of them behind the digit planes)
    constexpr bool kKeysAhead = kSets == 1 && !GPT;                              // a block's first keys and values asked for beside the down projection before it
    constexpr int LPK = HD / 4, KPW = 64 / LPK, TILE = kWaves * KPW, U = 4;
    __shared__ __align__(16) uint8_t planes[kZeros + 16];
    __shared__ __align__(16) float unit[kTokenMostD / 32 + 2];
    __shared__ __align__(16) float red[kTokenTiles * 16 * kRed];         // a pass's sums: [output][wavefront]
    __shared__ __align__(16) float row[3 * HD];                          // the head's q, k, v
    __shared__ __align__(16) float states[kWaves * HD];
    __shared__ __align__(16) float s_m[kWaves], s_l[kWaves], sums[kWaves], sums2[kWaves], means[kWaves], counts[kWaves];
    __shared__ uint64_t most[kWaves];
    __shared__ int s_fail, s_far;
    __shared__ int4 s_part[kTokenHead + 1], s_item[(kTokenHead + 1) * kWaves];

    extern __shared__ __align__(16) unsigned char ring[];               // the multiplying wavefronts' items

    const TokenShape &s = r.shape;
    const int g = blockIdx.x & 7, m = blockIdx.x >> 3, lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6) & (kWaves - 1);
    const bool speaks = uniform(threadIdx.x) < kSpeakers;
    if (g >= s.groups) return;
    const int d = s.d, X = s.groups;
    const bool crossing = X > 1;
    const int h0 = token_head0(s, g), heads = token_head0(s, g + 1) - h0, slice = heads * HD;
    const int u0 = token_unit0(s, g), units = token_unit0(s, g + 1) - u0;
    const int steps_d = (d + 63) >> 6, pitch_d = steps_d * 64 + 16, pitch_o = ((slice + 63) >> 6) * 64 + 16, pitch_h = ((units + 63) >> 6) * 64 + 16;

    // The workgroup's part of each product {first tile, tiles, steps}, and each wavefront's items of it {tile, step, items, steps}
    // (of the head: its first pass)
    if (threadIdx.x <= kTokenHead) {
        const TokenPart q = token_part(s, threadIdx.x, g, m);
        s_part[threadIdx.x] = make_int4(q.t0, q.t1 - q.t0, q.steps, 0);
    }
    if (threadIdx.x >= 64 && threadIdx.x < 64 + (kTokenHead + 1) * kWaves) {
        const int phase = (threadIdx.x - 64) / kWaves, w = (threadIdx.x - 64) % kWaves;
        const TokenPart q = token_part(s, phase, g, m);
        const TokenItems it = token_items(min(q.t1 - q.t0, kTokenTiles), q.steps, w);
        s_item[phase * kWaves + w] = make_int4(it.first / q.steps, it.first % q.steps, it.end - it.first, q.steps);
    }
    if (threadIdx.x == 0) { s_fail = 0; s_far = 0; }
    if (threadIdx.x < 4) reinterpret_cast<uint32_t *>(planes + kZeros)[threadIdx.x] = 0;
    for (int i = threadIdx.x; i < kTokenTiles * 16 * kRed; i += kThreads) red[i] = 0.0f;
    lds_barrier();

    struct Part { int t0, tiles, steps; };
    auto part_of = [&](int phase) {
        const int4 q = s_part[phase];
        return Part{uniform(q.x), uniform(q.y), uniform(q.z)};
    };
    const Part ph = part_of(kTokenHead);
    const int splits = kMembers / heads, hl = m / splits, split = m - hl * splits;       // (heads: 1 .. kMembers)
    const bool wo_tiles = part_of(kTokenWo).tiles > 0;
    // splits with keys at position p, and whether this workgroup has some
    auto active_at = [&](int p) { return min(splits, p / TILE + 1); };
    int pos = uniform(r.given ? r.pos_given : r.state[0]);
    pos = uniform(min(max(pos, 0), s.max_seq - 1));                      // (the host never lets it be another; stay in bounds)

    if (!speaks) {
        // ── the multiplying wavefronts ──
        // A wavefront's items are one stream, the same for every token.  It keeps the next kRing of them in LDS or on their way there.
        const uint32_t lane16 = lane * 16, lane_scale = 1024 + ((lane & 15) * 2 + (lane >> 5)) * 4;
        const unsigned char *const slots = ring + wave * (kRing * kTokenItemBytes);
        const uint32_t slots_at = uniform((int)(uint32_t)(uintptr_t)(const __attribute__((address_space(3))) unsigned char *)slots);
        struct Work { int tile, st, n, steps; };
        auto work_of = [&](int phase) {
            const int4 q = s_item[phase * kWaves + wave];
            return Work{uniform(q.x), uniform(q.y), uniform(q.z), uniform(q.w)};
        };
        auto head_pass = [&](int t0) {                                   // of the pass that begins with tile t0
            const TokenItems it = token_items(min(ph.t0 + ph.tiles - t0, kTokenTiles), ph.steps, wave);
            return Work{it.first / ph.steps, it.first % ph.steps, it.end - it.first, ph.steps};
        };
        const uint32_t start = uniform((int)r.offsets[(g * kMembers + m) * kWaves + wave]);
        uint32_t end = start;
        for (int p = kTokenQkv; p <= kTokenDown; p++) end += (uint32_t)(s.layers * work_of(p).n);
        end += (uint32_t)token_head_items(TokenPart{ph.t0, ph.t0 + ph.tiles, ph.steps}, wave);
        // When items are asked for.  A compute unit's loads return in order, so what is asked for in front of the words that everybody
        // waits for delays them by its way from memory; behind a row that has just been sent to the other groups, beside products and
        // beside the attention there is time for some.  A block of more items than slots needs all of these, a smaller one the few
        // that delay nothing (us a token, one and the other: 16 blocks of d 2048 314 and 330, 8 of d 1024 99 and 96).
        const bool heavy = work_of(kTokenQkv).n + work_of(kTokenWo).n + work_of(kTokenUp).n + work_of(kTokenDown).n > kRing;
        const bool passing = r.passing != 0;
        uint32_t next = start, left = (end - start) * (uint32_t)r.steps; // to be asked for: the next item, and how many in all
        int held = 0, put = 0, take = 0;                                 // asked for and not multiplied yet; the slots of the next ones
        auto ask = [&]() {
            const unsigned char *const p = r.items + (uint64_t)next * kTokenItemBytes;
            const uint32_t to = slots_at + (uint32_t)put * kTokenItemBytes;
            if (passing) {
                load_passing_to_lds16(p, lane16, to);
                if (lane < 8) load_passing_to_lds16(p + 1024, lane16, to + 1024);        // (lane i's 16 bytes go to 16 i)
            } else {
                load_to_lds16(p, lane16, to);
                if (lane < 8) load_to_lds16(p + 1024, lane16, to + 1024);
            }
            next = next + 1 == end ? start : next + 1;
            put = put + 1 == kRing ? 0 : put + 1;
            held++; left--;
        };
        // All but the last `behind` items asked for are here (two loads each; this wavefront makes no others in its loop)
        auto wait_but = [&](int behind) {
            if (behind <= 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            else if (behind == 1) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
            else if (behind == 2) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
            else if (behind == 3) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
            else if (behind == 4) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            else if (behind == 5) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
            else if (behind == 6) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
            else if (behind == 7) asm volatile("s_waitcnt vmcnt(14)" ::: "memory");
            else if (behind == 8) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(18)" ::: "memory");
        };
        // Up to n more items asked for (the slots' last reads have been answered)
        auto refill = [&](int n) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            for (; n > 0 && held < kRing && left > 0; n--) ask();
        };
        auto leave = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };         // (nothing may be on its way to LDS that is given back)
        // this lane's row of the activations: digit plane (r & 1) | (r & 4) / 2 of scale group r / 8; in the other group's k zeros
        const int quarter = lane >> 4, ar = lane & 15;
        const bool in_group = (ar >> 3) == (quarter >> 1);
        const uint32_t a_plane = (ar & 1) | ((ar >> 1) & 2), a_steps = in_group ? ~0u : 0u;
        const float high = (quarter & 1) ? 65536.0f : 1.0f;
        const uint32_t unit_at = (quarter >> 1) * 4, red_lane = (lane & 15) * (kRed * 4) + wave * 4;
        // The next c (1 to 3) items, out of their slots: whatever else of the batch is there is anything
        constexpr int Q = kTogether;
        struct Batch { intx4 w[Q]; float s[Q]; };
        auto take_batch = [&](Batch &b, int c) {
            wait_but(held - c);
#pragma unroll
            for (int q = 0, slot = take; q < Q; q++, slot = slot + 1 == kRing ? 0 : slot + 1) {
                const unsigned char *const p = slots + slot * kTokenItemBytes;
                b.w[q] = *reinterpret_cast<const intx4 *>(p + lane16);
                b.s[q] = *reinterpret_cast<const float *>(p + lane_scale);
            }
            held -= c;
            take = take + c >= kRing ? take + c - kRing : take + c;
        };
        Batch b0, b1, b2, b3;                                            // of a phase: its first items, taken before its row is there
        constexpr int kFirst = 4 * Q;
        auto take_first = [&](const Work &k) {
            if (k.n > 0) take_batch(b0, min(Q, k.n));
            if (k.n > Q) take_batch(b1, min(Q, k.n - Q));
            if (k.n > 2 * Q) take_batch(b2, min(Q, k.n - 2 * Q));
            if (k.n > 3 * Q) take_batch(b3, min(Q, k.n - 3 * Q));
        };
        // This wavefront's items with the staged row; their sums to red.
        auto products = [&](const Work &k, int pitch) {
            const uint32_t a_at = in_group ? a_plane * pitch + quarter * 16 : kZeros;
            int st = k.st;
            uint32_t to = red_lane + k.tile * (16 * kRed * 4);
            float acc = 0.0f;
            // A batch of the `rem` items that are left: operands and products together, then the sums one by one; then it takes others
            auto some = [&](Batch &b, int rem) {
                const int c = min(Q, rem);
                int sq[Q];
                intx4 v[Q], p[Q];
                float u[Q];
                sq[0] = st;
#pragma unroll
                for (int q = 1; q < Q; q++) sq[q] = sq[q - 1] + 1 == k.steps ? 0 : sq[q - 1] + 1;
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    v[q] = *reinterpret_cast<const intx4 *>(planes + (a_at + (a_steps & (uint32_t)(sq[q] * 64))));
                    u[q] = *reinterpret_cast<const float *>(reinterpret_cast<const unsigned char *>(unit) + (unit_at + (uint32_t)sq[q] * 8));
                }
                __builtin_amdgcn_sched_barrier(0);                       // (all of them on their way at once)
#pragma unroll
                for (int q = 0; q < Q; q++) p[q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v[q], b.w[q], (intx4){0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    // C rows 4 quarter + e: digits 2 (quarter & 1) + e of group quarter / 2 (up to 2^20 each: their sum is exact)
                    const float t = (float)((p[q][1] << 8) + p[q][0]) * u[q];
                    if (q < rem) {
                        acc = fmaf(t, b.s[q], acc);
                        if (sq[q] + 1 == k.steps || rem == q + 1) {
                            const float v16 = quarters_sum(acc * high);
                            if (lane < 16) *reinterpret_cast<float *>(reinterpret_cast<unsigned char *>(red) + to) = v16;
                            acc = 0.0f;
                            to += 16 * kRed * 4;
                        }
                    }
                }
                st = sq[c - 1] + 1 == k.steps ? 0 : sq[c - 1] + 1;
                const int more = rem - kFirst;
                if (more > 0) {
                    take_batch(b, min(Q, more));
                    // (what follows a product is asked for behind its sums)
                    if (more - Q > held) refill(more - Q - held);
                }
            };
            for (int rem = k.n; rem > 0; rem -= kFirst) {
                some(b0, rem);
                if (rem > Q) some(b1, rem - Q);
                if (rem > 2 * Q) some(b2, rem - 2 * Q);
                if (rem > 3 * Q) some(b3, rem - 3 * Q);
            }
        };
        refill(kRing);
        lds_barrier();                                                   // [place]
        Work k = work_of(kTokenQkv);
        take_first(k);
        for (int step = 0; step < r.steps; step++) {
            const bool attends = split < active_at(pos) && hl < heads;
            for (int i = 0; i <= 4 * s.layers; i++) {
                const int p = i == 4 * s.layers ? (int)kTokenHead : i & 3, p_next = i + 1 == 4 * s.layers ? (int)kTokenHead : (p + 1) & 3;
                const int beside = !heavy ? 0 : p == kTokenQkv ? 2 : p == kTokenWo ? 1 : p == kTokenUp ? 3 : 0;
                const int after = p == kTokenQkv ? (heavy ? 2 : 0) : p == kTokenWo ? 6 : p == kTokenUp ? (heavy ? 8 : 0) : p == kTokenDown ? 1 : kRing;
                if (GPT && (p & 1) == 0) lds_barrier();                  // [moments]
                if ((p & 1) == 0 && uniform(s_fail) != 0) return leave();
                for (int t0 = ph.t0;;) {                                 // (the head's passes; one of any other product)
                    lds_barrier();                                       // [staged]; of a pass that is not the first, [read]
                    DJ_STAMP2(2 * p);
                    __builtin_amdgcn_s_setprio(2);                       // (in front of what the speakers do beside them: 0.8 % of a token)
                    if (max(beside, k.n - kFirst - held) > 0) refill(max(beside, k.n - kFirst - held));
                    if (p != kTokenHead || ph.tiles > 0) {               // (without a tile of the head: no pass)
                        products(k, p == kTokenWo ? pitch_o : p == kTokenDown ? pitch_h : pitch_d);
                        lds_barrier();                                   // [sums]
                    }
                    DJ_STAMP2(2 * p + 1);
                    __builtin_amdgcn_s_setprio(0);
                    t0 += kTokenTiles;
                    const bool again = p == kTokenHead && t0 < ph.t0 + ph.tiles;
                    k = again ? head_pass(t0) : work_of(p == kTokenHead ? (int)kTokenQkv : p_next);
                    refill(max(after, min(k.n, kFirst) - held));
                    if (!again && p == kTokenHead && step + 1 == r.steps) break;
                    if (p != kTokenQkv) take_first(k);
                    if (!again) break;
                }
                if (p == kTokenQkv) {
                    if (attends) lds_barrier();                          // [q k v]
                    refill(heavy ? 3 : 2);
                    if (attends) lds_barrier();                          // [heads]
                    refill(max(5, k.n - held));
                    take_first(k);
                }
            }
            if (r.choose != kTokenGreedy) return leave();
            lds_barrier();                                               // [most]
            lds_barrier();                                               // [all]
            pos = uniform(min(pos + 1, s.max_seq - 1));
        }
        return leave();
    }

    // ── the speaking wavefronts ──
    // The thread's index anew in every phase: what is computed from it is not kept in registers from one to the next.
    auto me = [&]() {
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        return t;
    };
    word *const ex = r.exchange;
    word *const front = ex - kTokenFront;
    const TokenExchange e = token_exchange(s);
    const TokenVectors at_vec = token_vectors(s);
    const uint32_t mine = (uint32_t)(g * e.group);                       // the group's words
    // output i of the pass: what the wavefronts left
    auto sum_of = [&](int i) {
        const float4 a = *reinterpret_cast<const float4 *>(red + i * kRed), b = *reinterpret_cast<const float4 *>(red + i * kRed + 4);
        return ((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w));
    };
    // .. and zeros again, as they have to be for the wavefronts without items of its tile
    auto clear = [&](int i) {
        float4 *const p = reinterpret_cast<float4 *>(red + i * kRed);
        p[0] = p[1] = make_float4(0.f, 0.f, 0.f, 0.f);
    };
    // A wait that ends without its words says so; behind the next barrier the whole workgroup leaves.
    auto check = [&](bool ok) { if (!ok) s_fail = 1; };
    auto give_up = [&]() {
        if (uniform(s_fail) == 0) return false;
        if (threadIdx.x == 0) {
            __hip_atomic_store(r.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(reinterpret_cast<uint32_t *>(front), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return true;
    };
    int token = uniform(r.given ? r.token_given : r.state[1]), generated = uniform(r.given ? r.generated_given : r.state[2]);
    // A group's words stay in its L2 only if its workgroups all run on one XCD; else they go through memory.
    {
        const int t = threadIdx.x;
        const uint32_t xcc = __builtin_amdgcn_s_getreg(20 | (31 << 11));
        const uint32_t place = e.place + g * kMembers;
        if (t == 0) send(ex, place + m, __uint_as_float(xcc), r.tag, true);
        if (t < kMembers / 2) {
            Words<1> w;
            uint32_t p[1] = {place + 2 * t};
            check(receive(w, ex, p, r.tag, r.polls));
            if (w.v[0].x != xcc || w.v[0].z != xcc) s_far = 1;
        }
        // a run in front that gave up: this one would wait as long, for words that may never come
        if (t == 64) {
            const word w = __hip_atomic_load(front, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            check((uint32_t)w == 0);
            if (w >> 32) s_far = 1;
        }
    }
    lds_barrier();                                                       // [place]
    if (give_up()) return;
    const bool far = uniform(s_far) != 0;

    float4 x[kSets];
    float divisor = 1.0f, inverse = 1.0f;
    const float inv_d = 1.0f / (float)d;
    auto divide = [&](float v) {                                         // by the root mean square of the row
        if constexpr (GPT) return v;
        else return quotient(v, divisor, inverse);
    };
    auto row_operand = [&](int t, float4 (&v)[kSets], const float *p) {
#pragma unroll
        for (int q = 0; q < kSets; q++) {
            const int i = t + q * kSpeakers;
            v[q] = 4 * i < d ? *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(p) + (uint32_t)i * 16) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    auto wave_part = [&](int t, float v, float *to) {
        v = wave_sum_dpp(v);
        if ((t & 63) == 0) to[t >> 6] = v;
    };
    auto all_waves = [&](const float *from) {
        const float4 a = *reinterpret_cast<const float4 *>(from), b = *reinterpret_cast<const float4 *>(from + 4);
        return ((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w));
    };
    // Normalises x and stages it (RMSNorm1D.java:46-57: gamma * x, the products divided by the rms, which waits for nobody;
    // LayerNorm1D.java:34-66), up to the barrier [staged].
    auto stage = [&](int t, const float4 (&gamma)[kSets], const float4 (&beta)[kSets]) {
        if constexpr (GPT) {
            // the wavefronts' means and squares about them, and of those the row's: one barrier, and no large mean in the squares
            const int width = min(max(d - (t & ~63) * 4, 0), 256);       // the wavefront's values of a set of 4 * kSpeakers ...
            float sm = 0.0f, sv = 0.0f, n = (float)width;
            if constexpr (kSets > 1) n += (float)min(max(d - (t & ~63) * 4 - 4 * kSpeakers, 0), 256);
#pragma unroll
            for (int q = 0; q < kSets; q++) sm += (x[q].x + x[q].y) + (x[q].z + x[q].w);          // (zeros past the row's end)
            sm = wave_sum_dpp(sm);
            const float here = n > 0.0f ? sm * __builtin_amdgcn_rcpf(n) : 0.0f;      // (near the mean is enough: what it is off by goes in as a square)
#pragma unroll
            for (int q = 0; q < kSets; q++) {
                const bool on = 4 * (t + q * kSpeakers) < d;
                const float a = x[q].x - here, b = x[q].y - here, c = x[q].z - here, e = x[q].w - here;
                sv += on ? (a * a + b * b) + (c * c + e * e) : 0.0f;
            }
            sv = wave_sum_dpp(sv);
            if ((t & 63) == 0) { sums[t >> 6] = sm; sums2[t >> 6] = sv; means[t >> 6] = here; counts[t >> 6] = n; }
            lds_barrier();                                               // [moments]
            const float mean = all_waves(sums) * inv_d;
            float squares = 0.0f;
#pragma unroll
            for (int w = 0; w < kWaves; w += 4) {
                const float4 n_w = *reinterpret_cast<const float4 *>(counts + w), m_w = *reinterpret_cast<const float4 *>(means + w),
                             s_w = *reinterpret_cast<const float4 *>(sums2 + w);
                const float e0 = m_w.x - mean, e1 = m_w.y - mean, e2 = m_w.z - mean, e3 = m_w.w - mean;
                squares += ((s_w.x + n_w.x * e0 * e0) + (s_w.y + n_w.y * e1 * e1)) + ((s_w.z + n_w.z * e2 * e2) + (s_w.w + n_w.w * e3 * e3));
            }
            float4 c[kSets];
#pragma unroll
            for (int q = 0; q < kSets; q++) {
                const bool on = 4 * (t + q * kSpeakers) < d;
                c[q] = on ? make_float4(x[q].x - mean, x[q].y - mean, x[q].z - mean, x[q].w - mean) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
            const float deviation = sqrtf(squares * inv_d + kLayerNormEps), isd = __builtin_amdgcn_rcpf(deviation), sd = residual_divisor(deviation);
            auto over = [&](float v) { const float y = v * isd; return fmaf(fmaf(-y, sd, v), isd, y); };     // (as quotient: at most sqrt(d))
#pragma unroll
            for (int q = 0; q < kSets; q++)
                if (t + q * kSpeakers < steps_d * 16)
                    stage_digits4(planes, pitch_d, unit, t + q * kSpeakers,
                                  make_float4(over(c[q].x) * gamma[q].x + beta[q].x, over(c[q].y) * gamma[q].y + beta[q].y,
                                              over(c[q].z) * gamma[q].z + beta[q].z, over(c[q].w) * gamma[q].w + beta[q].w));
            lds_barrier();                                               // [staged]
        } else {
            float ss = 0.0f;
#pragma unroll
            for (int q = 0; q < kSets; q++) {
                ss += (x[q].x * x[q].x + x[q].y * x[q].y) + (x[q].z * x[q].z + x[q].w * x[q].w);
                if (t + q * kSpeakers < steps_d * 16)
                    stage_digits4(planes, pitch_d, unit, t + q * kSpeakers,
                                  make_float4(x[q].x * gamma[q].x, x[q].y * gamma[q].y, x[q].z * gamma[q].z, x[q].w * gamma[q].w));
            }
            wave_part(t, ss, sums);
            lds_barrier();                                               // [staged]
            divisor = sqrtf(all_waves(sums) * inv_d + kRmsEps);
            inverse = 1.0f / divisor;
            divisor = residual_divisor(divisor);
            asm volatile("" : "+v"(divisor), "+v"(inverse));             // (now, beside the products, and not where they are used)
        }
    };
    // What the workgroup's tiles p of a product leave of the row, added to x.  Between groups: the member's slice of all groups' sums
    // first.  beat: members without a tile say that they were here.
    auto exchange_row = [&](int t, int part_at, int row_at, bool beat, const Part &p, uint32_t tag) {
        const uint32_t part = part_at, to = mine + row_at;
        if (t < p.tiles * 16) {
            const float v = sum_of(t);
            if (crossing) send(ex, part + g * d + p.t0 * 16 + t, v, tag, true);
            else send(ex, to + p.t0 * 16 + t, v, tag + 1, far);
            clear(t);
        }
        DJ_STAMP(24);
        // Nothing can be here yet.  Words of the row would only be in the way, and a first try for the other groups' sums that comes too early
        // costs its whole way before the next.  Us a token at GPT 12 blocks of 768 and 16 of d 2048, by the length of the sleep: none 140.6 and
        // 302.8, 5 137.9 and 297.1, 12 136.4 and 293.4, this 135.4 and 292.6, 32 142.8 and 297.2.
        if (crossing) __builtin_amdgcn_s_sleep(kCrossSleep);
        // (by wavefronts that have, as a rule, not sent: a wait for loads waits for the stores in front of them too)
        if (crossing && t >= kSpeakers / 2 && t - kSpeakers / 2 < p.tiles * 8) {         // two outputs a thread
            const int o = p.t0 * 16 + 2 * (t - kSpeakers / 2);
            float a = 0.0f, b = 0.0f;
            Words<8> w;
            uint32_t from[8];
#pragma unroll
            for (int i = 0; i < 8; i++) from[i] = part + min(i, X - 1) * d + o;
            check(receive(w, ex, from, tag, r.polls));
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (i < X) { a += first(w.v[i]); b += second(w.v[i]); }
            send(ex, to + o, a, tag + 1, far);
            send(ex, to + o + 1, b, tag + 1, far);
        }
        DJ_STAMP(25);
        if (beat && t == kSpeakers - 1) send(ex, mine + e.beat + m, 0.0f, tag + 1, far);
        if (beat && t >= kSpeakers - kMembers / 2) {
            Words<1> w;
            uint32_t from[1] = {mine + e.beat + 2 * (t - (kSpeakers - kMembers / 2))};
            check(receive(w, ex, from, tag + 1, r.polls));
        }
#pragma unroll
        for (int q = 0; q < kSets; q++) {
            const int i = t + q * kSpeakers;
            if (4 * i < d) {
                float4 v;
                check(receive4(v, ex, to + 4 * i, tag + 1, r.polls));
                x[q].x += v.x; x[q].y += v.y; x[q].z += v.z; x[q].w += v.w;
            }
        }
    };

    const bool beats = d < 16 * kMembers, beats_up = ((GPT ? 1 : 2) * units + 15) / 16 < kMembers;
    for (int step = 0; step < r.steps; step++) {
        const uint32_t tag0 = r.tag + 1 + (uint32_t)step * token_tags(s);
        {
            const bool ok = token >= 0 && token < s.vocab;
            const float nan = __builtin_nanf("");
            const int t = me();
            row_operand(t, x, r.emb + (int64_t)(ok ? token : 0) * d);
            if (!ok)
#pragma unroll
                for (int q = 0; q < kSets; q++) x[q] = make_float4(nan, nan, nan, nan);
            if constexpr (GPT) {
                float4 p[kSets];
                row_operand(t, p, r.pos + (int64_t)pos * d);
#pragma unroll
                for (int q = 0; q < kSets; q++) { x[q].x += p[q].x; x[q].y += p[q].y; x[q].z += p[q].z; x[q].w += p[q].w; }
            }
        }
        const int active = active_at(pos);
        const bool attends = hl < heads && split < active;
        const uint32_t angle = (uint32_t)(lane % LPK) * 8;
        const float2 cs = *reinterpret_cast<const float2 *>(reinterpret_cast<const char *>(r.cos_t + (int64_t)pos * (HD / 2)) + angle);
        const float2 sn = *reinterpret_cast<const float2 *>(reinterpret_cast<const char *>(r.sin_t + (int64_t)pos * (HD / 2)) + angle);
        // (a phase's small operands are asked for while the products in front of it run)
        float4 gamma[kSets], beta[kSets];
        row_operand(me(), gamma, r.vectors + at_vec.g1);
        if constexpr (GPT) row_operand(me(), beta, r.vectors + at_vec.be1);
        // The head's keys and values; a row is HD floats, of which a lane has four.  A round of them: keys of tile
        // `split + (r0 + u) splits` of TILE (past the cached ones: the first key's, again).  At the first position row 0 holds anything,
        // and a masked value weighs nothing only where it is a number: there numbers stand in for it, the items' offsets (whole numbers) or,
        // which a GPT's tokens are the faster by, norm weights (where they are no numbers every row is none).  Us for the greedy, sampled and
        // stepped workloads of a narrow Llama, a GPT and a Llama: offsets in both families 1722, 6843 and 3825, norm weights in both
        // 1728, 6799 and 3873, as here 1707, 6801 and 3836; without a stand-in 1716, 6806 and 3838, and zeros behind the loads a GPT's 6870.
        static_assert(kMembers * kWaves >= HD, "the offsets of one group hold a row");
        floatx4 K[U], V[U];
        auto keys_at = [&](int l) { return ((int64_t)(l * s.heads + h0 + (hl < heads ? hl : 0)) * s.max_seq) * HD; };
        auto load_round = [&](int l, int r0) {
            const float *const stand_in = GPT ? r.vectors : reinterpret_cast<const float *>(r.offsets);
            const char *const kb = reinterpret_cast<const char *>(r.kc + keys_at(l)), *const vb = reinterpret_cast<const char *>(pos == 0 ? stand_in : r.vc + keys_at(l));
            const int t = me(), dl = (t & 63) % LPK, key0 = (t >> 6) * KPW + (t & 63) / LPK;
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int key = (split + (r0 + u) * splits) * TILE + key0;
                const uint32_t from = (key < pos ? key : 0) * (HD * 4) + dl * 16;
                K[u] = *reinterpret_cast<const floatx4 *>(kb + from);
                V[u] = *reinterpret_cast<const floatx4 *>(vb + from);
            }
        };
        if (kKeysAhead && attends) load_round(0, 0);
        for (int l = 0; l < s.layers; l++) {
            const float *const vec = r.vectors + (int64_t)l * at_vec.stride;
            const uint32_t tag = tag0 + (uint32_t)l * 8;
            int at_pos = pos, t = me();
            asm volatile("" : "+v"(at_pos));
            at_pos = uniform(at_pos);

            // ── q | k | v of the group's heads ──
            DJ_STAMP(0);
            stage(t, gamma, beta);
            DJ_STAMP(1);
            if (give_up()) return;
            t = me();
            const int sub = (t & 63) / LPK, dl = (t & 63) % LPK, key0 = (t >> 6) * KPW + sub;
            if (!kKeysAhead && attends) load_round(l, 0);
            const Part pa = part_of(kTokenQkv), pc = part_of(kTokenWo);
            lds_barrier();                                               // [sums]
            DJ_STAMP(3);
            if (t < pa.tiles * 16) {
                send(ex, mine + e.qkv + pa.t0 * 16 + t, divide(sum_of(t)), tag, far);
                clear(t);
            }
            DJ_STAMP(4);

            // ── attention of this workgroup's share of a head's keys ──
            // (they are here; a wait where the ways meet again would also wait for what has been sent)
#pragma unroll
            for (int u = 0; u < U; u++)
                asm volatile("" : "+v"(K[u]), "+v"(V[u]));
            if (attends) {
                if (t < 3 * HD / 2) {
                    const int part = t / (HD / 2), c = 2 * (t - part * (HD / 2));
                    Words<1> w;
                    uint32_t p[1] = {mine + e.qkv + part * slice + hl * HD + c};
                    check(receive(w, ex, p, tag, r.polls));
                    *reinterpret_cast<float2 *>(row + part * HD + c) = make_float2(first(w.v[0]), second(w.v[0]));
                }
                lds_barrier();                                           // [q k v]
                DJ_STAMP(5);
                const float4 q = *reinterpret_cast<const float4 *>(row + dl * 4), k = *reinterpret_cast<const float4 *>(row + HD + dl * 4),
                             nv = *reinterpret_cast<const float4 *>(row + 2 * HD + dl * 4);
                const float4 qr = make_float4(q.x * cs.x - q.y * sn.x, q.x * sn.x + q.y * cs.x, q.z * cs.y - q.w * sn.y, q.z * sn.y + q.w * cs.y);
                const float4 nk = make_float4(k.x * cs.x - k.y * sn.x, k.x * sn.x + k.y * cs.x, k.z * cs.y - k.w * sn.y, k.z * sn.y + k.w * cs.y);
                float mx = -INFINITY, sum = 0.0f;
                float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
                auto round = [&](int r0) {
                    float sc[U];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        sc[u] = -INFINITY;
                        const int tile = (split + (r0 + u) * splits) * TILE, key = tile + key0;
                        if (tile > at_pos) continue;                     // (uniform; like lanes past the last key it weighs nothing)
                        if (tile + TILE > at_pos && key == at_pos) {     // the new row: used from registers, and appended
                            K[u] = floatx4{nk.x, nk.y, nk.z, nk.w}; V[u] = floatx4{nv.x, nv.y, nv.z, nv.w};
                            char *const kb = reinterpret_cast<char *>(r.kc + keys_at(l)), *const vb = reinterpret_cast<char *>(r.vc + keys_at(l));
                            const uint32_t to = (uint32_t)key * (HD * 4) + dl * 16;
                            *reinterpret_cast<float4 *>(kb + to) = nk;
                            *reinterpret_cast<float4 *>(vb + to) = nv;
                        }
                        // (q.k) * scale as the reference computes it (HeadOps.java:96-99), then the change of base
                        const float dot = group_sum<LPK>(qr.x * K[u].x + qr.y * K[u].y + qr.z * K[u].z + qr.w * K[u].w);
                        sc[u] = key <= at_pos ? (dot * r.scale) * kLog2e : -INFINITY;
                    }
                    float mn = mx;
#pragma unroll
                    for (int u = 0; u < U; u++) mn = fmaxf(mn, sc[u]);
                    if (mn > -INFINITY) {
                        const float corr = __builtin_amdgcn_exp2f(mx - mn);
                        sum *= corr; o.x *= corr; o.y *= corr; o.z *= corr; o.w *= corr;
#pragma unroll
                        for (int u = 0; u < U; u++) {
                            const float w = __builtin_amdgcn_exp2f(sc[u] - mn);
                            sum += w;
                            o.x += w * V[u].x; o.y += w * V[u].y; o.z += w * V[u].z; o.w += w * V[u].w;
                        }
                        mx = mn;
                    }
                };
                round(0);
                for (int r0 = U; (split + r0 * splits) * TILE <= at_pos; r0 += U) {      // workgroup-uniform
                    load_round(l, r0);
                    round(r0);
                }
                // the lane groups of a wavefront, then the wavefronts (LDS)
                auto keys = [&](float v, auto op) {
                    float a, b;
                    if constexpr (LPK == 8) { lane_pair<8>(v, a, b); v = op(a, b); }
                    if constexpr (LPK <= 16) { lane_pair<16>(v, a, b); v = op(a, b); }
                    lane_pair<32>(v, a, b);
                    return op(a, b);
                };
                auto add = [](float a, float b) { return a + b; };
                const float top = keys(mx, [](float a, float b) { return fmaxf(a, b); }), w = top == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mx - top);
                sum = keys(sum * w, add);
                o = make_float4(keys(o.x * w, add), keys(o.y * w, add), keys(o.z * w, add), keys(o.w * w, add));
                if ((t & 63) == 0) { s_m[t >> 6] = top; s_l[t >> 6] = sum; }
                if (sub == 0) *reinterpret_cast<float4 *>(&states[(t >> 6) * HD + dl * 4]) = o;
                lds_barrier();                                           // [heads]
                if (t < HD + 2) {                                        // (record: o[HD], the maximum, the sum)
                    const float *const from = t < HD ? states + t : s_l;
                    const int pitch = t < HD ? HD : 1;
                    float wm[kWaves], part[kWaves], M = -INFINITY, v = 0.0f;
#pragma unroll
                    for (int i = 0; i < kWaves; i++) { wm[i] = s_m[i]; part[i] = from[i * pitch]; }
                    __builtin_amdgcn_sched_barrier(0);                   // (all of them on their way at once)
#pragma unroll
                    for (int i = 0; i < kWaves; i++) M = fmaxf(M, wm[i]);
#pragma unroll
                    for (int i = 0; i < kWaves; i++) v += part[i] * __builtin_amdgcn_exp2f(wm[i] - M);
                    send(ex, mine + e.rec + (hl * splits + split) * (HD + 2) + t, t == HD ? M : v, tag + 1, far);
                }
            }
            DJ_STAMP(6);

            // ── the group's heads, and its columns of Wo ──
            // A wavefront takes 32 values of the heads' output at a time: lane 8 p + q quad q of the records of splits p, p + 8, ...
            t = me();
            if (wo_tiles) {
                const int p8 = (t & 63) >> 3, q8 = t & 7;
                for (int v0 = wave * 32; v0 < pc.steps * 64; v0 += kWaves * 32) {
                    const int head = min(v0 / HD, heads - 1), c = v0 % HD + 4 * q8;      // (past the heads' values: zeros)
                    float M = -INFINITY, sum = 0.0f;
                    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
                    auto records = [&](int i, auto count) {              // of splits i + p8 and, for two, i + 8 + p8
                        constexpr int J = decltype(count)::value;
                        uint32_t p[3 * J];
#pragma unroll
                        for (int j = 0; j < J; j++) {
                            const uint32_t from = mine + e.rec + (head * splits + min(i + 8 * j + p8, active - 1)) * (HD + 2);
                            p[3 * j] = from + c; p[3 * j + 1] = from + c + 2; p[3 * j + 2] = from + HD;
                        }
                        Words<3 * J> w;
                        check(receive(w, ex, p, tag + 1, r.polls));
#pragma unroll
                        for (int j = 0; j < J; j++) {
                            const bool on = i + 8 * j + p8 < active;
                            const float m2 = on ? first(w.v[3 * j + 2]) : -INFINITY, top = fmaxf(M, m2);
                            const float a = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(M - top), b = on ? __builtin_amdgcn_exp2f(m2 - top) : 0.0f;
                            sum = sum * a + (on ? second(w.v[3 * j + 2]) : 0.0f) * b;
                            o.x = o.x * a + (on ? first(w.v[3 * j]) : 0.0f) * b; o.y = o.y * a + (on ? second(w.v[3 * j]) : 0.0f) * b;
                            o.z = o.z * a + (on ? first(w.v[3 * j + 1]) : 0.0f) * b; o.w = o.w * a + (on ? second(w.v[3 * j + 1]) : 0.0f) * b;
                            M = top;
                        }
                    };
                    if (active <= 8) records(0, std::integral_constant<int, 1>{});
                    else
                        for (int i = 0; i < active; i += 16) records(i, std::integral_constant<int, 2>{});
                    auto parts = [&](float v, auto op) {
                        float a, b;
                        lane_pair<8>(v, a, b);
                        v = op(a, b);
                        lane_pair<16>(v, a, b);
                        v = op(a, b);
                        lane_pair<32>(v, a, b);
                        return op(a, b);
                    };
                    auto add = [](float a, float b) { return a + b; };
                    const float top = parts(M, [](float a, float b) { return fmaxf(a, b); }), w = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(M - top);
                    sum = parts(sum * w, add);
                    o = make_float4(parts(o.x * w, add), parts(o.y * w, add), parts(o.z * w, add), parts(o.w * w, add));
                    const float inv = __builtin_amdgcn_rcpf(sum);
                    auto over = [&](float v) { const float y = v * inv; return fmaf(fmaf(-y, sum, v), inv, y); };
                    o = v0 < slice ? make_float4(over(o.x), over(o.y), over(o.z), over(o.w)) : make_float4(0.f, 0.f, 0.f, 0.f);
                    if (p8 == 0) stage_digits4(planes, pitch_o, unit, v0 / 4 + q8, o);
                }
            }
            DJ_STAMP(7);
            lds_barrier();                                               // [staged]
            if (give_up()) return;
            DJ_STAMP(8);
            t = me();
            row_operand(t, gamma, vec + at_vec.g2);
            if constexpr (GPT) row_operand(t, beta, vec + at_vec.be2);
            const Part pd = part_of(kTokenUp), pe = part_of(kTokenDown);
            const int unit_n = pd.t0 * (GPT ? 16 : 8) + t;               // this thread's unit of the group's
            const bool has_unit = t < pd.tiles * (GPT ? 16 : 8) && unit_n < units;
            const float bg = has_unit ? vec[at_vec.bg + u0 + unit_n] : 0.0f, bu = !GPT && has_unit ? vec[at_vec.bu + u0 + unit_n] : 0.0f;
            lds_barrier();                                               // [sums]
            DJ_STAMP(10);
            exchange_row(t, e.part, e.row, beats, pc, tag + 2);
            DJ_STAMP(13);
            t = me();

            // ── feed-forward: the group's hidden units ──
            stage(t, gamma, beta);
            DJ_STAMP(14);
            t = me();
            if (give_up()) return;
            float4 bd[kSets];
            row_operand(t, bd, vec + at_vec.bd);
            row_operand(t, gamma, vec + at_vec.stride + at_vec.g1);
            if constexpr (GPT) row_operand(t, beta, vec + at_vec.stride + at_vec.be1);
            lds_barrier();                                               // [sums]
            DJ_STAMP(16);
            t = me();
            if (has_unit) {
                float v;
                if constexpr (GPT) v = gemm_gelu(sum_of(t) + bg);
                else {
                    const float gate = divide(sum_of(2 * t)) + bg, up = divide(sum_of(2 * t + 1)) + bu;
                    v = gate * (1.0f / (1.0f + expf(-gate))) * up;               // SiLU.java:20-24, SwiGLULayer.java:69
                }
                send(ex, mine + e.hid + unit_n, v, tag + 4, far);
            }
            if (t < pd.tiles * (GPT ? 16 : 8)) {
                clear(GPT ? t : 2 * t);
                if (!GPT) clear(2 * t + 1);
            }
            if (beats_up && t == 0) send(ex, mine + e.beat2 + m, 0.0f, tag + 4, far);
            DJ_STAMP(17);
            // ── and its columns of the down projection ──
            t = me();
            {
                const int quads = ((units + 63) >> 6) * 16;
                if (beats_up && t >= kSpeakers - kMembers / 2) {
                    Words<1> w;
                    uint32_t p[1] = {mine + e.beat2 + 2 * (t - (kSpeakers - kMembers / 2))};
                    check(receive(w, ex, p, tag + 4, r.polls));
                }
                if (t < quads) {
                    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (4 * t + 3 < units) check(receive4(v, ex, mine + e.hid + 4 * t, tag + 4, r.polls));
                    else if (4 * t < units) {                            // the last hidden units of a width that is no multiple of four
                        float *const f = reinterpret_cast<float *>(&v);
                        for (int c = 0; c < 3; c++)
                            if (4 * t + c < units) {
                                bool ok = false;
                                word got = 0;
                                for (int n = 0; n < r.polls && !ok; n++) {
                                    got = __hip_atomic_load(ex + mine + e.hid + 4 * t + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                    ok = (uint32_t)(got >> 32) == tag + 4;
                                }
                                check(ok);
                                f[c] = __uint_as_float((uint32_t)got);
                            }
                    }
                    stage_digits4(planes, pitch_h, unit, t, v);
                }
                lds_barrier();                                           // [staged]
                DJ_STAMP(18);
                if (give_up()) return;
            }
            if (kKeysAhead && attends && l + 1 < s.layers) load_round(l + 1, 0);
#pragma unroll
            for (int q = 0; q < kSets; q++) { x[q].x += bd[q].x; x[q].y += bd[q].y; x[q].z += bd[q].z; x[q].w += bd[q].w; }
            lds_barrier();                                               // [sums]
            DJ_STAMP(20);
            t = me();
            exchange_row(t, e.part2, e.row2, false, pe, tag + 5);
        }
        DJ_STAMP(23);

        // ── logits ──
        stage(me(), gamma, beta);
        if (give_up()) return;
        const int t = me();
        uint64_t key = 0;
        for (int t0 = ph.t0; t0 < ph.t0 + ph.tiles; t0 += kTokenTiles) {
            const int tiles = min(ph.t0 + ph.tiles - t0, kTokenTiles), c = t0 * 16 + t;
            const bool has_logit = t < tiles * 16 && c < s.vocab;
            const float bias = has_logit ? r.blm[c] : 0.0f;
            if (t0 > ph.t0) lds_barrier();                               // [read]
            lds_barrier();                                               // [sums]
            const float sum = has_logit ? sum_of(t) : 0.0f;
            if (t < tiles * 16) clear(t);
            if (has_logit) {
                const float v = divide(sum) + bias;
                r.logits[c] = v;
                const uint64_t k = logit_key(v, c);
                key = k > key ? k : key;
            }
        }
        DJ_STAMP(26);
        if (r.choose != kTokenGreedy) {
            if (r.given && g == 0 && m == 0 && threadIdx.x == 0) { r.state[0] = pos + 1; r.state[1] = token; r.state[2] = generated; }
            return;
        }

        // ── the largest one ──
        const uint32_t tag = tag0 + (uint32_t)s.layers * 8;
        key = wave_most(key);
        if ((t & 63) == 0) most[t >> 6] = key;
        lds_barrier();                                                   // [most]
        if (t < 2) {
#pragma unroll
            for (int w = 0; w < kWaves; w++) { const uint64_t o = most[w]; key = o > key ? o : key; }
            send(ex, e.best + kTokenBestWords * (g * kMembers + m) + t, __uint_as_float(t ? (uint32_t)(key >> 32) : (uint32_t)key), tag, crossing || far);
        }
        key = 0;
        // (by wavefronts that have, as a rule, stored no logits: a wait for loads waits for the stores in front of them too)
        const int from = t - (kSpeakers - kMembers * kTokenGroupsMost);
        if (from >= 0 && from < X * kMembers) {
            Words<1> w;
            uint32_t p[1] = {(uint32_t)(e.best + kTokenBestWords * from)};
            check(receive(w, ex, p, tag, r.polls));
            key = (uint64_t)w.v[0].z << 32 | w.v[0].x;
        }
        key = wave_most(key);
        if ((t & 63) == 0) reinterpret_cast<uint64_t *>(states)[t >> 6] = key;
        lds_barrier();                                                   // [all]
        if (give_up()) return;
#pragma unroll
        for (int w = 0; w < kWaves; w++) { const uint64_t o = reinterpret_cast<const uint64_t *>(states)[w]; key = o > key ? o : key; }
        token = uniform((int)~(uint32_t)key);
        DJ_STAMP(27);
        if (g == 0 && m == 0 && threadIdx.x == 0) {
            if ((uint32_t)generated < (uint32_t)s.max_seq) r.tokens[generated] = token;
            r.state[0] = pos + 1;
            r.state[1] = token;
            r.state[2] = generated + 1;
        }
        generated++;
        pos = uniform(min(pos + 1, s.max_seq - 1));
    }
    // the next token's embedding, where the launches of a token expect it
    if (g == 0 && m == 0)
        for (int i = threadIdx.x; i < d; i += kSpeakers) r.x[i] = token >= 0 && token < s.vocab ? r.emb[(int64_t)token * d + i] : __builtin_nanf("");
}

// ── the items ───────────────────────────────────────────────────────────────
// One workgroup per wavefront of the run: its items of one phase of one block.
__global__ void __launch_bounds__(256)
k_token_pack(TokenShape s, int phase, int layer, const int8_t *wq, const float *scales, int k_total, unsigned char *items, const uint32_t *offsets) {
    const int w = blockIdx.x % kWaves, gm = blockIdx.x / kWaves, g = gm / kMembers, m = gm - g * kMembers;
    const int kp = (k_total + 31) & ~31, h0 = token_head0(s, g), slice = (token_head0(s, g + 1) - h0) * s.hd;
    const int u0 = token_unit0(s, g), units = token_unit0(s, g + 1) - u0, gates = s.gpt ? 1 : 2;
    int64_t at = offsets[blockIdx.x];
    TokenPart part = token_part(s, phase, g, m);
    int per_layer = 0, before = 0;
    for (int p = kTokenQkv; p <= kTokenDown; p++) {
        const TokenPart q = token_part(s, p, g, m);
        const TokenItems it = token_items(q.t1 - q.t0, q.steps, w);
        if (p < phase) before += it.end - it.first;
        per_layer += it.end - it.first;
    }
    at += phase == kTokenHead ? (int64_t)s.layers * per_layer : (int64_t)layer * per_layer + before;
    // the rows' first k, and how many of them the group takes
    const int k0 = phase == kTokenWo ? h0 * s.hd : phase == kTokenDown ? u0 : 0;
    const int k_end = phase == kTokenWo ? k0 + slice : phase == kTokenDown ? k0 + units : k_total;
    auto row_of = [&](int o) {                                           // the weight's row of the group's output o; -1: none
        if (phase == kTokenQkv) { const int seg = o / slice; return seg * s.d + h0 * s.hd + o - seg * slice; }
        if (phase == kTokenUp) return o < gates * units ? gates * u0 + o : -1;
        if (phase == kTokenHead) return o < s.vocab ? o : -1;
        return o;
    };
    const int lane = threadIdx.x & 63, four = threadIdx.x >> 6;
    for (int t0 = part.t0; t0 < part.t1; t0 += kTokenTiles) {            // (only the head takes more than one pass)
        const TokenItems it = token_items(part.t1 - t0 < kTokenTiles ? part.t1 - t0 : kTokenTiles, part.steps, w);
        for (int i = it.first + four; i < it.end; i += 4) {
            const int tile = i / part.steps, st = i - tile * part.steps;
            unsigned char *out = items + (at + i - it.first) * kTokenItemBytes;
            const int r0 = row_of((t0 + tile) * 16 + (lane & 15)), k = k0 + st * 64 + (lane >> 4) * 16;
            intx4 v = {0, 0, 0, 0};
            if (r0 >= 0 && k < k_end) v = *reinterpret_cast<const intx4 *>(wq + (int64_t)r0 * kp + k);
            *reinterpret_cast<intx4 *>(out + lane * 16) = v;
            if (lane < 32) {
                const int r1 = row_of((t0 + tile) * 16 + (lane >> 1)), ks = k0 + st * 64 + (lane & 1) * 32;
                *reinterpret_cast<float *>(out + 1024 + lane * 4) = r1 >= 0 && ks < k_end ? scales[(int64_t)r1 * (kp >> 5) + (ks >> 5)] : 0.0f;
            }
        }
        at += it.end - it.first;
    }
}

__global__ void __launch_bounds__(256) k_token_copy(const float *from, float *to, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) to[i] = from[i];
}

template <int HD, bool GPT> auto kernel_of(const TokenShape &s) { return s.d <= 4 * kSpeakers ? &k_token_run<HD, GPT, 1> : &k_token_run<HD, GPT, 2>; }
void (*kernel_for(const TokenShape &s))(TokenRun) {
    if (s.hd == 32) return s.gpt ? kernel_of<32, true>(s) : kernel_of<32, false>(s);
    if (s.hd == 64) return s.gpt ? kernel_of<64, true>(s) : kernel_of<64, false>(s);
    return s.gpt ? kernel_of<128, true>(s) : kernel_of<128, false>(s);
}
constexpr int kBlocks = kMembers * kTokenGroupsMost;
constexpr int kRingBytes = kWaves * kRing * kTokenItemBytes;             // (more than half of a compute unit's LDS: one workgroup each)

}  // namespace

// Shapes that the kernel's arrays hold: the row, a group's heads and hidden units, a workgroup's tiles.
bool token_run_ok(const TokenShape &s) {
    if (s.groups < 1 || s.groups > kTokenGroupsMost || (s.hd != 32 && s.hd != 64 && s.hd != 128)) return false;
    if (s.heads < 1 || s.heads > kTokenMostD / s.hd || s.d != s.heads * s.hd || s.layers < 1 || s.vocab < 1 || s.dff < 1 || s.max_seq < 1) return false;
    if (s.dff > s.groups * kTokenMostSlice) return false;
    // what the kernel counts in 32 bits: a head's rows in bytes, the head's tiles times the workgroups they are dealt to, a run's tags
    if ((int64_t)s.max_seq * s.hd * 4 > (int64_t)1 << 32) return false;
    if (s.vocab > (1 << 28) - 16 || s.layers >= 1 << 21) return false;
    for (int g = 0; g < s.groups; g++) {
        const int heads = token_head0(s, g + 1) - token_head0(s, g), units = token_unit0(s, g + 1) - token_unit0(s, g);
        if (heads < 1 || heads > kMembers || heads * s.hd > kTokenMostSlice || units < 1 || units > kTokenMostSlice) return false;
        for (int m = 0; m < kMembers; m++)
            for (int p = kTokenQkv; p <= kTokenDown; p++) {
                const TokenPart q = token_part(s, p, g, m);
                if (q.t1 - q.t0 > kTokenTiles) return false;
            }
    }
    return (int64_t)s.layers * s.heads * s.max_seq < (int64_t)1 << 31;
}

// Groups for a model.  One alone crosses nothing, and gets its weights at what one XCD's share of the memory gives; it is the better choice
// up to some 3 MB a layer (us a token on one group and on the most: 0.2 MB a layer 41.0 and 52.2, 0.8 MB 102.6 and 123.3, 1.5 MB 31.1 and
// 33.9, 2.2 MB 66.1 and 68.4, 2.6 MB 34.5 and 34.4, 3.0 MB 59.8 and 61.2, 4.5 MB 29.3 and 26.6, 5.0 MB 76.0 and 63.6, 5.4 MB 96.0 and 71.5).  Else as
// many as there are heads for (d 896: 93.2 us on eight, 97.5 on four, 119 on two).
int token_run_groups(const TokenShape &s) {
    constexpr int64_t kOneGroup = (int64_t)3 << 20;
    const int64_t bytes = ((int64_t)s.layers * (4LL * s.d * s.d + (s.gpt ? 2LL : 3LL) * s.d * s.dff) + (int64_t)s.d * s.vocab) * 9 / 8;
    TokenShape a = s;
    if (bytes <= kOneGroup * s.layers)
        for (int g : {1, 2, 4, 8}) {
            a.groups = g;
            if (token_run_ok(a)) return g;
        }
    for (int g : {8, 4, 2, 1}) {
        a.groups = g;
        if (token_run_ok(a)) return g;
    }
    return 0;
}

bool token_run_resident(const TokenShape &s) {
    int device = 0, blocks = 0, units = 0;
    DJ_HIP(hipGetDevice(&device));
    DJ_HIP(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device));
    DJ_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel_for(s)), hipFuncAttributeMaxDynamicSharedMemorySize, kRingBytes));
    DJ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, reinterpret_cast<const void *>(kernel_for(s)), kThreads, kRingBytes));
    return (int64_t)blocks * units >= kBlocks;
}

int64_t token_run_items(const TokenShape &s, uint32_t *offsets) {
    int64_t n = 0;
    for (int g = 0; g < s.groups; g++)
        for (int m = 0; m < kMembers; m++)
            for (int w = 0; w < kWaves; w++) {
                offsets[(g * kMembers + m) * kWaves + w] = (uint32_t)n;
                int64_t layer = 0;
                for (int p = kTokenQkv; p <= kTokenDown; p++) {
                    const TokenPart q = token_part(s, p, g, m);
                    const TokenItems it = token_items(q.t1 - q.t0, q.steps, w);
                    layer += it.end - it.first;
                }
                n += layer * s.layers + token_head_items(token_part(s, kTokenHead, g, m), w);
            }
    return n;
}

void launch_token_pack(hipStream_t st, const TokenShape &s, int phase, int layer, const int8_t *wq, const float *scales, int k_total, unsigned char *items, const uint32_t *offsets) {
    launch_kernel(k_token_pack, dim3(s.groups * kMembers * kWaves), dim3(256), 0, st, s, phase, layer, wq, scales, k_total, items, offsets);
}

void launch_token_vectors(hipStream_t st, const TokenShape &s, int layer, const TokenLayer &from, float *vectors) {
    const TokenVectors v = token_vectors(s);
    float *const to = vectors + (int64_t)layer * v.stride;
    auto copy = [&](const float *f, int at, int n) { if (f) launch_kernel(k_token_copy, dim3((n + 255) / 256), dim3(256), 0, st, f, to + at, n); };
    copy(from.g1, v.g1, s.d);
    copy(from.be1, v.be1, s.d);
    copy(from.g2, v.g2, s.d);
    copy(from.be2, v.be2, s.d);
    copy(from.bd, v.bd, s.d);
    copy(from.bg, v.bg, s.dff);
    copy(from.bu, v.bu, s.dff);
}

void launch_token_run(hipStream_t st, const TokenRun &r) { launch_kernel(kernel_for(r.shape), dim3(kBlocks), dim3(kThreads), kRingBytes, st, r); }

}  // namespace dj

#ifdef DJ_TRACE
extern "C" int deepj_hip_token_trace(unsigned long long *out) {
    return hipMemcpyFromSymbol(out, HIP_SYMBOL(dj::g_token_trace), sizeof(dj::g_token_trace)) == hipSuccess ? 0 : 1;
}
#endif
