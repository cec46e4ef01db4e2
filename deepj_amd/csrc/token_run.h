// Shapes and work division of the token run (kernels_token.hip): shared by its kernels, its launcher and the plan's host side.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace dj {

// A group is the kTokenMembers workgroups of one XCD, one per compute unit, of kTokenWaves wavefronts that speak and as many that multiply.
// What a group shares travels through its L2, what groups share through memory.
constexpr int kTokenMembers = 32, kTokenGroupsMost = 8, kTokenWaves = 8;
constexpr int kTokenTiles = 32;                 // tiles of 16 outputs that a workgroup takes in one pass
constexpr int kTokenItemBytes = 1024 + 128;     // 16 outputs x 64 k: the int8 weights in the lanes' order, then their 32 scales
// In front of the exchanged words, a page (so that they lie as in a block of their own), of which a run reads the first word: its low half
// is set by a run that gave up, its high half sends a group's words through memory also where its workgroups share an L2.
constexpr int kTokenFront = 512;
constexpr int kTokenBestWords = 16;             // a line each: writers of one line wait for one another
constexpr int kTokenMostD = 4096, kTokenMostSlice = 2048;
// Items of more bytes than this are loaded as passing by: the memory-side cache (256 MB) does not hold them until the next token, and
// with them on their way through the caches it does not hold the rows and keys either.  Us a token without and with: 195 MB 88.2
// and 95.1, 256 MB 121.3 and 124.4, 291 MB 102.8 and 96.6, 326 MB 152.0 and 146.4, 1 GB 344 and 331.
constexpr int64_t kTokenPassingBytes = 272LL << 20;
constexpr int kTokenPolls = 1 << 21;            // loads of a word that is waited for: 1 s inside an XCD, 2 to 4 between XCDs
enum TokenPhase { kTokenQkv = 0, kTokenWo = 1, kTokenUp = 2, kTokenDown = 3, kTokenHead = 4 };

struct TokenShape { int d, heads, hd, layers, dff, vocab, max_seq, groups, gpt; };

// Share i of n things dealt to `parts`
__host__ __device__ inline int token_share(int n, int parts, int i) { return (int)((uint32_t)n * (uint32_t)i / (uint32_t)parts); }
__host__ __device__ inline int token_head0(const TokenShape &s, int g) { return token_share(s.heads, s.groups, g); }
// A group's hidden units: whole runs of 64, the last group's cut at dff
__host__ __device__ inline int token_unit0(const TokenShape &s, int g) {
    const int u = token_share((s.dff + 63) / 64, s.groups, g) * 64;
    return u < s.dff ? u : s.dff;
}

// A workgroup's part of a product: tiles [t0, t1) of 16 outputs of the group's (the head: of everybody's), `steps` of 64 k each
struct TokenPart { int t0, t1, steps; };
__host__ __device__ inline TokenPart token_part(const TokenShape &s, int phase, int g, int m) {
    const int slice_heads = (token_head0(s, g + 1) - token_head0(s, g)) * s.hd, units = token_unit0(s, g + 1) - token_unit0(s, g);
    int tiles, k, parts = kTokenMembers, i = m;
    if (phase == kTokenQkv) { tiles = 3 * slice_heads / 16; k = s.d; }
    else if (phase == kTokenWo) { tiles = s.d / 16; k = slice_heads; }
    else if (phase == kTokenUp) { tiles = ((s.gpt ? 1 : 2) * units + 15) / 16; k = s.d; }
    else if (phase == kTokenDown) { tiles = s.d / 16; k = units; }
    else { tiles = (s.vocab + 15) / 16; k = s.d; parts = kTokenMembers * s.groups; i = g * kTokenMembers + m; }
    return TokenPart{token_share(tiles, parts, i), token_share(tiles, parts, i + 1), (k + 63) / 64};
}
// Items (tile, step), tile by tile, of `tiles` tiles that wavefront w takes: [first, end)
struct TokenItems { int first, end; };
__host__ __device__ inline TokenItems token_items(int tiles, int steps, int w) {
    return TokenItems{token_share(tiles * steps, kTokenWaves, w), token_share(tiles * steps, kTokenWaves, w + 1)};
}
// The head goes in passes of kTokenTiles tiles
__host__ __device__ inline int token_head_items(const TokenPart &p, int w) {
    int n = 0;
    for (int t = p.t0; t < p.t1; t += kTokenTiles) {
        const TokenItems it = token_items(p.t1 - t < kTokenTiles ? p.t1 - t : kTokenTiles, p.steps, w);
        n += it.end - it.first;
    }
    return n;
}

// Where the exchanged words of a group, and those that groups share, lie in the exchange block (in 8-byte words)
struct TokenExchange { int qkv, rec, row, row2, hid, beat, beat2, group; int part, part2, best, place, total; };
__host__ __device__ inline TokenExchange token_exchange(const TokenShape &s) {
    TokenExchange e;
    const int heads = (s.heads + s.groups - 1) / s.groups, units = ((s.dff + 63) / 64 + s.groups - 1) / s.groups * 64;
    int at = 0;
    auto take = [&](int n) { const int here = at; at += (n + 15) & ~15; return here; };
    e.qkv = take(3 * heads * s.hd);
    e.rec = take(kTokenMembers * (s.hd + 2));
    e.row = take(s.d);
    e.row2 = take(s.d);
    e.hid = take(units);
    e.beat = take(kTokenMembers);
    e.beat2 = take(kTokenMembers);
    e.group = at;
    at = e.group * s.groups;
    e.part = take(s.groups * s.d);
    e.part2 = take(s.groups * s.d);
    e.best = take(kTokenBestWords * kTokenMembers * s.groups);
    e.place = take(kTokenMembers * s.groups);
    e.total = at;
    return e;
}

struct TokenLayer { const float *g1, *be1, *g2, *be2, *bg, *bu, *bd; };
// A block's norm weights and biases in the plan, one behind the other in floats (the last place is the final norm's, as g1 and
// be1): addresses the kernel computes, where a table of pointers would be a load in front of every load.
struct TokenVectors { int g1, be1, g2, be2, bd, bg, bu, stride; };
__host__ __device__ inline TokenVectors token_vectors(const TokenShape &s) {
    const int d = s.d, f = (s.dff + 3) & ~3;
    return TokenVectors{0, d, 2 * d, 3 * d, 4 * d, 5 * d, 5 * d + f, 5 * d + 2 * f};
}
enum { kTokenLogits = 0, kTokenGreedy = 1 };
struct TokenRun {
    TokenShape shape;
    const unsigned char *items;           // every wavefront's items in the order it takes them
    const uint32_t *offsets;              // [groups * members * waves]: a wavefront's first item
    const float *vectors;                 // [layers + 1] of TokenVectors
    const float *emb, *pos, *blm, *cos_t, *sin_t;
    float *kc, *vc, *logits, *x;
    int32_t *state, *tokens;
    unsigned long long *exchange;         // (kTokenFront words behind the block's start)
    uint32_t *failed;                     // (pinned host memory)
    uint32_t tag;                         // of the run's first exchange
    int steps, choose;
    int given, pos_given, token_given, generated_given;       // given: the state by value, for one token without a choice; the run leaves it one position on
    int passing;                          // the items are more than kTokenPassingBytes
    int polls;                            // loads of a word until a wait is given up
    float scale;
};
constexpr int kTokenMostSteps = 256;         // tokens of a launch: a run of thousands does not hold the device in one piece
__host__ __device__ inline uint32_t token_tags(const TokenShape &s) { return (uint32_t)s.layers * 8 + 8; }   // a token's tags

bool token_run_ok(const TokenShape &s);           // (host arithmetic, like the next)
int token_run_groups(const TokenShape &s);
bool token_run_resident(const TokenShape &s);     // whether all of a run's workgroups fit on the device at once
int64_t token_run_items(const TokenShape &s, uint32_t *offsets);      // their number; offsets[groups * members * waves]
void launch_token_pack(hipStream_t st, const TokenShape &s, int phase, int layer, const int8_t *wq, const float *scales, int k_total, unsigned char *items, const uint32_t *offsets);
void launch_token_vectors(hipStream_t st, const TokenShape &s, int layer, const TokenLayer &from, float *vectors);     // (null: left as it is)
void launch_token_run(hipStream_t st, const TokenRun &r);

}  // namespace dj
