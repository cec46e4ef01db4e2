// Native decode driver: the caller on the host side of the C ABI.  It plays the part of
// the reference's LlamaModel / DeepSeekModel / GPTModel + TextGenerator
//   (src/main/java/io/github/kirstenali/deepj/models/{DecoderOnlyModel,TextGenerator}.java,
//    models/llama/LlamaModel.java, models/deepseek/DeepSeekModel.java, models/gpt/GPTModel.java)
// for inference, but instead of re-running the whole context for every token
// (TextGenerator.java:91-100) it keeps a KV cache in HBM, records ONE fused command
// stream per token and replays it as a HIP graph.  Position, current token and the
// generated ids live in device memory, so a run of N tokens needs no host round trip.
//
// Everything here goes through the public deepj_hip_* functions only: buffers are named
// by int ids, work is submitted as int32 command streams - the same boundary a Java
// HipBackend uses - so a Java facade can emit the identical streams.
//
// Weight names: "emb", "gf", "wlm", "blm" and per layer "L<i>.<w>" with w in
//   g1 g2 wq wk wv wo           (Llama;  MultiHeadSelfAttention.java:47-50)
//   g1 g2 wdq wuq wdkv wuk wuv wo (DeepSeek; MultiHeadLatentAttention.java:81-86)
//     kept as two Q8 matrices: the down-projections stacked by output row, [Wdq | pad | Wdkv], and the
//     up-projections as one block matrix that maps [cQ | pad | cKV] to [Q | K | V] (zero blocks elsewhere),
//     so MLA costs two projections and then shares the Llama attention path and its rotated K/V cache
//   wg bg wu bu wd bd           (SwiGLULayer.java:56-58)
// GPT (GPTTransformerBlock.java:52-57): g1 be1 g2 be2 (LayerNorm gamma/beta), wq wk wv wo, and the FNN's two
//   Linears as wg bg (dModel -> dFF) and wd bd (dFF -> dModel); model level adds "pos" and "bf".
// Matrices are given in the reference's orientation, fp32 [dIn x dOut] row-major.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "../../include/deepj_hip.h"

extern "C" {
void *deepj_host_random_create(int64_t seed);
void deepj_host_random_destroy(void *h);
void deepj_host_random_fill(void *h, float *out, int64_t n, double scale, int32_t threads);
float deepj_host_random_next_float(void *h);
}

namespace {

struct Config {
    int32_t kind;       // 0 Llama, 1 DeepSeek (MLA), 2 GPT; DeepSeek with the latent KV cache arrives as kind 3 and
                        // is kept here as kind 1 with `latent` set
    int32_t vocab, max_seq, d, heads, layers, dff, q_rank, kv_rank;
    bool latent = false;
};

struct Error : std::runtime_error { using std::runtime_error::runtime_error; };

// Tokens per replay of a decode graph.  A replay costs 13 us of its own, so long runs go through graphs of consecutive tokens;
// 16 of them only where a token is short enough for that to be seen (kShortStream launches, 2.6 us each: 5 % at 11 of them).
constexpr int kReplayTokens[] = {16, 4, 1};
constexpr int kShortStream = 32;

void hip(int rc) {
    if (rc != 0) throw Error(deepj_hip_last_error());
}

struct Layer {
    int32_t g1 = -1, g2 = -1, be1 = -1, be2 = -1;     // be*: LayerNorm betas (GPT)
    int32_t wqkv = -1, wo = -1;                       // Llama: fused [3d x d]
    int32_t wdown = -1, wup = -1;                     // MLA: stacked down-projections, block up-projection
    int32_t wdq = -1, wuq = -1, wdkv = -1, wukv = -1; // MLA with the latent cache: Wdq, Wuq, Wdkv, and [Wuk | Wuv] by output row
    int32_t wgu = -1, bg = -1, bu = -1, wd = -1, bd = -1;
};

struct Acts {          // activation buffers for S rows
    int32_t rows = 0;
    int32_t x = -1, x2 = -1, qkv = -1, q = -1, att = -1, ff = -1, ids = -1;
    int32_t cq = -1;                                                 // MLA: [cQ | pad | cKV] rows (latent cache: cQ rows)
    int32_t ckv = -1;                                                // MLA with the latent cache: cKV rows
    int32_t part_a = -1, part_f = -1;                                // DECODE_ATTN's / DECODE_FFN's partial sums (one row only)
};

struct Runner {
    Config cfg{};
    int32_t next_id = 0;
    std::map<std::string, bool> have;
    std::vector<Layer> layers;
    int32_t emb = -1, gf = -1, wlm = -1, blm = -1;
    int32_t pos_table = -1, bf = -1;                       // GPT: learned positions, final LayerNorm beta
    int32_t cos_t = -1, sin_t = -1, kc = -1, vc = -1;
    int32_t state = -1, tokens = -1, scratch = -1, logits = -1, last_x = -1;
    int32_t records = -1;                                  // decode attention records (merged by the Wo matvec)
    int32_t latent = -1, kv_all = -1;                      // latent cache [L][maxSeq][kvRank]; re-expanded [maxSeq][K | V] of one layer
    std::vector<int32_t> prepared;                         // the weights in the many-row GEMM's layout (first long prompt)
    bool prepared_done = false;
    int64_t prepared_budget = -1;                          // bytes such copies may take in all; -1: no limit
    int64_t prepared_bytes = 0;
    Acts dec, pre;
    int32_t sampler = -1;                                  // DECODE_SAMPLE's parameters
    // Captured per-token streams by how the token is chosen (Choose), whether the blocks are narrow, and kReplayTokens.
    int32_t graph[3][2][3] = {};
    // The model's tokens as one launch (deepj_hip_token_plan_*); 0: replayed graphs.  `pending`: the calls since the first run whose
    // outcome nobody has looked at, should they have to be done again by launches: greedy tokens, a step's token or a prompt.
    int32_t plan = 0, token_groups = 0;
    struct Pending { int32_t pos, generated, steps, token; std::vector<int32_t> prompt; bool chooses; };
    std::vector<Pending> pending;
    int32_t fed = 0, pending_fed = 0;                      // state[1] (now, in front of `pending`); -1: the token that was chosen last
    bool finalized = false;
    int32_t pos = 0;          // host mirror of state[0]
    int32_t generated = 0;    // host mirror of state[2]
    std::string error;

    int hd() const { return cfg.d / cfg.heads; }
    // up to this many positions a token's block takes two launches (DECODE_ATTN, DECODE_FFN), from there on five
    int narrow_positions() const { return cfg.kind == 1 ? 0 : deepj_hip_decode_block_positions(cfg.d, hd(), cfg.dff); }
    // MLA: width of [cQ | pad | cKV]; cKV starts at a multiple of 32 so that the Q8 groups of Wuk and Wuv
    // (32 consecutive inputs) are the ones each matrix would get on its own
    int q_rank_padded() const { return (cfg.q_rank + 31) / 32 * 32; }
    int latent_width() const { return q_rank_padded() + cfg.kv_rank; }

    int32_t alloc(int64_t floats) {
        if (floats > 0x7fffffffLL) throw Error("buffer too large for an int32 float count");
        int32_t id = next_id++;
        int32_t sz = (int32_t)floats;
        hip(deepj_hip_alloc_buffers(&id, &sz, 1));
        return id;
    }
    void release(int32_t &id) {
        if (id >= 0) { hip(deepj_hip_release(&id, 1)); id = -1; }
    }
    int32_t upload_new(const float *data, int64_t n) {
        int32_t id = alloc(n);
        hip(deepj_hip_upload(id, data, n));
        return id;
    }
    void run(const std::vector<int32_t> &s) { hip(deepj_hip_flush_ops(s.data(), (int32_t)s.size())); }
};

using Stream = std::vector<int32_t>;
// How a stream ends: with the logits, or with the next token chosen on the device.
enum Choose { kNone = 0, kGreedy = 1, kSample = 2 };
template <class... A> void emit(Stream &s, A... words) { (s.push_back((int32_t)words), ...); }

void q8_linear(Stream &s, int32_t x, int32_t w, int32_t out, int m, int k, int n, int flags, int32_t gamma = -1,
               int32_t bias = -1, int32_t bias2 = -1, int32_t residual = -1) {
    emit(s, DJ_OP_Q8_LINEAR, x, w, out, m, k, n, flags, gamma, bias, bias2, residual);
}

// ── weights ────────────────────────────────────────────────────────────────

void quantize_into(Runner &r, int32_t &dst, const float *data, int k, int n, int row_off, int row_step, int total) {
    if (dst < 0) dst = r.alloc(deepj_hip_q8_floats(k, total));
    int32_t tmp = r.upload_new(data, (int64_t)k * n);
    Stream s;
    emit(s, DJ_OP_Q8_QUANTIZE, tmp, dst, k, n, row_off, row_step, total);
    r.run(s);
    r.release(tmp);
}

void expect_shape(const std::string &name, int rows, int cols, int er, int ec) {
    if (rows != er || cols != ec)
        throw Error("weight " + name + ": expected " + std::to_string(er) + "x" + std::to_string(ec) + " but got " +
                    std::to_string(rows) + "x" + std::to_string(cols));
}

void set_weight(Runner &r, const std::string &name, const float *data, int rows, int cols) {
    const Config &c = r.cfg;
    const int d = c.d;
    if (r.finalized) throw Error("set_weight after finalize");
    if (name == "emb") { expect_shape(name, rows, cols, c.vocab, d); r.emb = r.upload_new(data, (int64_t)rows * cols); }
    else if (name == "gf") { expect_shape(name, rows, cols, 1, d); r.gf = r.upload_new(data, d); }
    else if (c.kind == 2 && name == "bf") { expect_shape(name, rows, cols, 1, d); r.bf = r.upload_new(data, d); }
    else if (c.kind == 2 && name == "pos") { expect_shape(name, rows, cols, c.max_seq, d); r.pos_table = r.upload_new(data, (int64_t)rows * cols); }
    else if (name == "blm") { expect_shape(name, rows, cols, 1, c.vocab); r.blm = r.upload_new(data, c.vocab); }
    else if (name == "wlm") { expect_shape(name, rows, cols, d, c.vocab); quantize_into(r, r.wlm, data, d, c.vocab, 0, 1, c.vocab); }
    else if (name.size() > 2 && name[0] == 'L') {
        size_t dot = name.find('.');
        if (dot == std::string::npos) throw Error("unknown weight " + name);
        int l = std::atoi(name.substr(1, dot - 1).c_str());
        if (l < 0 || l >= c.layers) throw Error("weight " + name + ": no such layer");
        Layer &L = r.layers[l];
        std::string w = name.substr(dot + 1);
        if (w == "g1") { expect_shape(name, rows, cols, 1, d); L.g1 = r.upload_new(data, d); }
        else if (w == "g2") { expect_shape(name, rows, cols, 1, d); L.g2 = r.upload_new(data, d); }
        else if (c.kind == 2 && w == "be1") { expect_shape(name, rows, cols, 1, d); L.be1 = r.upload_new(data, d); }
        else if (c.kind == 2 && w == "be2") { expect_shape(name, rows, cols, 1, d); L.be2 = r.upload_new(data, d); }
        else if (c.kind == 2 && w == "wg") { expect_shape(name, rows, cols, d, c.dff); quantize_into(r, L.wgu, data, d, c.dff, 0, 1, c.dff); }
        else if (c.kind == 2 && (w == "wu" || w == "bu")) throw Error("unknown weight " + name);
        else if (w == "bg") { expect_shape(name, rows, cols, 1, c.dff); L.bg = r.upload_new(data, c.dff); }
        else if (w == "bu") { expect_shape(name, rows, cols, 1, c.dff); L.bu = r.upload_new(data, c.dff); }
        else if (w == "bd") { expect_shape(name, rows, cols, 1, d); L.bd = r.upload_new(data, d); }
        else if (w == "wg") { expect_shape(name, rows, cols, d, c.dff); quantize_into(r, L.wgu, data, d, c.dff, 0, 2, 2 * c.dff); }
        else if (w == "wu") { expect_shape(name, rows, cols, d, c.dff); quantize_into(r, L.wgu, data, d, c.dff, 1, 2, 2 * c.dff); }
        else if (w == "wd") { expect_shape(name, rows, cols, c.dff, d); quantize_into(r, L.wd, data, c.dff, d, 0, 1, d); }
        else if (w == "wo") { expect_shape(name, rows, cols, d, d); quantize_into(r, L.wo, data, d, d, 0, 1, d); }
        else if (c.kind != 1 && (w == "wq" || w == "wk" || w == "wv")) {
            expect_shape(name, rows, cols, d, d);
            int part = w == "wq" ? 0 : (w == "wk" ? 1 : 2);
            quantize_into(r, L.wqkv, data, d, d, part * d, 1, 3 * d);
        }
        else if (c.latent && w == "wdq") { expect_shape(name, rows, cols, d, c.q_rank); quantize_into(r, L.wdq, data, d, c.q_rank, 0, 1, c.q_rank); }
        else if (c.latent && w == "wuq") { expect_shape(name, rows, cols, c.q_rank, d); quantize_into(r, L.wuq, data, c.q_rank, d, 0, 1, d); }
        else if (c.latent && w == "wdkv") { expect_shape(name, rows, cols, d, c.kv_rank); quantize_into(r, L.wdkv, data, d, c.kv_rank, 0, 1, c.kv_rank); }
        else if (c.latent && (w == "wuk" || w == "wuv")) {
            // Q8 rows [0, d) = the columns of Wuk, [d, 2d) = those of Wuv: one product re-expands a latent row to [K | V]
            expect_shape(name, rows, cols, c.kv_rank, d);
            quantize_into(r, L.wukv, data, c.kv_rank, d, w == "wuk" ? 0 : d, 1, 2 * d);
        }
        else if (c.kind == 1 && (w == "wdq" || w == "wdkv")) {
            // output rows [0, qRank) = Wdq, [qRankPadded, +kvRank) = Wdkv; the pad rows stay zero (the buffer is
            // zero-filled when it is created) and so produce zeros
            const bool q = w == "wdq";
            expect_shape(name, rows, cols, d, q ? c.q_rank : c.kv_rank);
            if (L.wdown < 0) {
                L.wdown = r.alloc(deepj_hip_q8_floats(d, r.latent_width()));
                Stream z; emit(z, DJ_OP_FILL, L.wdown, 0, deepj_hip_q8_floats(d, r.latent_width())); r.run(z);
            }
            quantize_into(r, L.wdown, data, d, cols, q ? 0 : r.q_rank_padded(), 1, r.latent_width());
        }
        else if (c.kind == 1 && (w == "wuq" || w == "wuk" || w == "wuv")) {
            // block matrix over the inputs [cQ | pad | cKV]: the matrix is widened with zero rows to the full
            // input width on the host, then its columns become Q8 rows [0,d) / [d,2d) / [2d,3d)
            const bool q = w == "wuq";
            const int in = q ? c.q_rank : c.kv_rank, k2 = r.latent_width(), off = q ? 0 : r.q_rank_padded();
            expect_shape(name, rows, cols, in, d);
            std::vector<float> wide((size_t)k2 * d, 0.0f);
            std::memcpy(wide.data() + (size_t)off * d, data, (size_t)in * d * sizeof(float));
            if (L.wup < 0) L.wup = r.alloc(deepj_hip_q8_floats(k2, 3 * d));
            quantize_into(r, L.wup, wide.data(), k2, d, (q ? 0 : (w == "wuk" ? 1 : 2)) * d, 1, 3 * d);
        }
        else throw Error("unknown weight " + name);
    } else throw Error("unknown weight " + name);
    r.have[name] = true;
}

std::vector<std::string> weight_names(const Config &c) {
    std::vector<std::string> names{"emb"};
    if (c.kind == 2) {
        names.push_back("pos");
        for (int l = 0; l < c.layers; l++) {
            std::string p = "L" + std::to_string(l) + ".";
            for (const char *w : {"g1", "be1", "g2", "be2", "wq", "wk", "wv", "wo", "wg", "bg", "wd", "bd"}) names.push_back(p + w);
        }
        names.insert(names.end(), {"gf", "bf", "wlm", "blm"});
        return names;
    }
    for (int l = 0; l < c.layers; l++) {
        std::string p = "L" + std::to_string(l) + ".";
        for (const char *w : {"g1", "g2"}) names.push_back(p + w);
        if (c.kind == 0) for (const char *w : {"wq", "wk", "wv", "wo"}) names.push_back(p + w);
        else for (const char *w : {"wdq", "wuq", "wdkv", "wuk", "wuv", "wo"}) names.push_back(p + w);
        for (const char *w : {"wg", "bg", "wu", "bu", "wd", "bd"}) names.push_back(p + w);
    }
    names.insert(names.end(), {"gf", "wlm", "blm"});
    return names;
}

// new LlamaModel(cfg, seed) / new DeepSeekModel(cfg, seed): same RNG wiring and draw order
// (LlamaModel.java:27-42, LlamaTransformerBuilder.java:45-55, DeepSeekTransformerBuilder.java:56-68).
// GPT: new GPTModel(cfg, seed) - Random(seed) for the token table, a second Random(seed) shared by the
// blocks, Random(seed + 1) for the head, Random(seed + 2) for the positions, then every parameter times
// initScale (GPTModel.java:27-46,76-81; GPTTransformerBlock.java:52-57; FNN draws its Linears in order).
void init_seeded(Runner &r, int64_t seed, int threads, float init_scale) {
    const Config &c = r.cfg;
    const int d = c.d;
    std::vector<float> buf;
    auto draw = [&](void *rng, const std::string &name, int rows, int cols) {
        buf.resize((size_t)rows * cols);
        deepj_host_random_fill(rng, buf.data(), (int64_t)rows * cols, 0.1, threads);
        if (init_scale != 1.0f) for (float &v : buf) v *= init_scale;
        set_weight(r, name, buf.data(), rows, cols);
    };
    auto constant = [&](const std::string &name, int cols, float v) {
        buf.assign((size_t)cols, init_scale != 1.0f ? v * init_scale : v);
        set_weight(r, name, buf.data(), 1, cols);
    };
    void *emb_rng = deepj_host_random_create(seed);
    void *stack_rng = deepj_host_random_create(seed);
    void *head_rng = deepj_host_random_create(seed + 1);
    void *pos_rng = deepj_host_random_create(seed + 2);
    try {
        draw(emb_rng, "emb", c.vocab, d);
        if (c.kind == 2) draw(pos_rng, "pos", c.max_seq, d);
        for (int l = 0; l < c.layers; l++) {
            std::string p = "L" + std::to_string(l) + ".";
            constant(p + "g1", d, 1.0f);
            constant(p + "g2", d, 1.0f);
            if (c.kind == 2) {
                constant(p + "be1", d, 0.0f);
                constant(p + "be2", d, 0.0f);
                for (const char *w : {"wq", "wk", "wv", "wo"}) draw(stack_rng, p + w, d, d);
                draw(stack_rng, p + "wg", d, c.dff);  constant(p + "bg", c.dff, 0.0f);
                draw(stack_rng, p + "wd", c.dff, d);  constant(p + "bd", d, 0.0f);
                continue;
            }
            if (c.kind == 0) {
                for (const char *w : {"wq", "wk", "wv", "wo"}) draw(stack_rng, p + w, d, d);
            } else {
                draw(stack_rng, p + "wdq", d, c.q_rank);
                draw(stack_rng, p + "wuq", c.q_rank, d);
                draw(stack_rng, p + "wdkv", d, c.kv_rank);
                draw(stack_rng, p + "wuk", c.kv_rank, d);
                draw(stack_rng, p + "wuv", c.kv_rank, d);
                draw(stack_rng, p + "wo", d, d);
            }
            draw(stack_rng, p + "wg", d, c.dff);  constant(p + "bg", c.dff, 0.0f);
            draw(stack_rng, p + "wu", d, c.dff);  constant(p + "bu", c.dff, 0.0f);
            draw(stack_rng, p + "wd", c.dff, d);  constant(p + "bd", d, 0.0f);
        }
        constant("gf", d, 1.0f);
        if (c.kind == 2) constant("bf", d, 0.0f);
        draw(head_rng, "wlm", d, c.vocab);
        constant("blm", c.vocab, 0.0f);
    } catch (...) {
        deepj_host_random_destroy(emb_rng); deepj_host_random_destroy(stack_rng); deepj_host_random_destroy(head_rng);
        deepj_host_random_destroy(pos_rng);
        throw;
    }
    deepj_host_random_destroy(emb_rng); deepj_host_random_destroy(stack_rng); deepj_host_random_destroy(head_rng);
    deepj_host_random_destroy(pos_rng);
}

// ── buffers ────────────────────────────────────────────────────────────────

// Buffers for `rows` rows (they only ever grow: every op takes its row count explicitly).
void alloc_acts(Runner &r, Acts &a, int rows) {
    const Config &c = r.cfg;
    if (a.rows >= rows) return;
    for (int32_t *id : {&a.x, &a.x2, &a.qkv, &a.q, &a.att, &a.ff, &a.ids, &a.cq, &a.ckv}) r.release(*id);
    int64_t S = rows, d = c.d;
    a.x = r.alloc(S * d); a.x2 = r.alloc(S * d); a.q = r.alloc(S * d); a.att = r.alloc(S * d);
    a.ff = r.alloc(S * c.dff); a.ids = r.alloc(std::max<int64_t>(S, 4));
    a.qkv = r.alloc(S * 3 * d);
    if (c.latent) { a.cq = r.alloc(S * c.q_rank); a.ckv = r.alloc(S * c.kv_rank); }
    else if (c.kind == 1) a.cq = r.alloc(S * r.latent_width());
    a.rows = rows;
}

bool warms_up();
void warm_up(Runner &r);
void decode(Runner &r, int steps, int mode, Choose how);
void reset(Runner &r);

// Tokens of a run as one launch (Llama and GPT; DeepSeek's stay launches).
void make_plan(Runner &r) {
    const Config &c = r.cfg;
    if (c.kind == 1 || r.token_groups < 0) return;
    std::vector<int32_t> w{c.kind, c.vocab, c.max_seq, c.d, c.heads, c.layers, c.dff, r.token_groups, r.emb, r.pos_table, r.gf, r.bf, r.wlm, r.blm,
                           r.cos_t, r.sin_t, r.kc, r.vc, r.state, r.tokens, r.logits, r.dec.x};
    for (const Layer &L : r.layers)
        for (int32_t id : {L.g1, L.be1, L.g2, L.be2, L.wqkv, L.wo, L.wgu, L.bg, L.bu, L.wd, L.bd}) w.push_back(id);
    hip(deepj_hip_token_plan_create(w.data(), (int32_t)w.size(), &r.plan));
}

void finalize(Runner &r) {
    const Config &c = r.cfg;
    if (r.finalized) return;
    for (const auto &n : weight_names(c))
        if (!r.have.count(n)) throw Error("weight " + n + " was never set");
    const int hd = r.hd(), half = hd / 2;
    // RotaryEmbedding.java:63-70
    std::vector<float> ct((size_t)c.max_seq * half), st((size_t)c.max_seq * half);
    for (int pos = 0; pos < c.max_seq; pos++)
        for (int i = 0; i < half; i++) {
            float expo = (2.0f * (float)i) / (float)hd;
            float theta = (float)((double)pos / std::pow((double)10000.0f, (double)expo));
            // GPT attends without rotation (MultiHeadSelfAttention.java:60-86): the identity tables turn the
            // rotation inside the attention kernels into x * 1 - y * 0 = x.
            ct[(size_t)pos * half + i] = c.kind == 2 ? 1.0f : (float)std::cos((double)theta);
            st[(size_t)pos * half + i] = c.kind == 2 ? 0.0f : (float)std::sin((double)theta);
        }
    r.cos_t = r.upload_new(ct.data(), (int64_t)ct.size());
    r.sin_t = r.upload_new(st.data(), (int64_t)st.size());
    int64_t per_layer = (int64_t)c.max_seq * c.d;
    // K (after RoPE) and V of every position, per layer [H][maxSeq][hd].  DeepSeek too: its latent rows could
    // be cached instead (kvRank floats per token rather than 2*dModel), but the reference rotates K after the
    // up-projection (MultiHeadLatentAttention.java:108-112), so the up-projection cannot be folded into the query
    // and every step would have to re-expand and re-rotate all cached positions.
    if (c.latent) {
        // The latent cache (MultiHeadLatentAttention.java:98-106 computes K and V from cKV = x.Wdkv): kvRank floats per
        // token and layer instead of 2 * dModel.  Every step re-expands the layer's cached rows to [K | V] and rotates
        // K (the reference rotates K after the up-projection, :108-112), into ONE buffer all layers take turns with.
        r.latent = r.alloc((int64_t)c.layers * c.max_seq * c.kv_rank);
        r.kv_all = r.alloc((int64_t)c.max_seq * 2 * c.d);
    } else {
        r.kc = r.alloc(per_layer * c.layers);
        r.vc = r.alloc(per_layer * c.layers);
    }
    r.state = r.alloc(4);
    r.tokens = r.alloc(c.max_seq);
    r.logits = r.alloc(c.vocab);
    r.last_x = r.alloc(c.d);
    int ns = std::max(1, std::min(16, 512 / c.heads));
    // attention scratch: the split records of one row (decode paths) or of a short prompt whose key rounds are shared
    int64_t sf = (int64_t)c.heads * ns * (hd + 4);
    for (int rows = 2; rows <= 32; rows++) sf = std::max(sf, deepj_hip_attention_scratch_floats(rows, c.heads, hd, c.max_seq));
    if (c.latent) sf = std::max(sf, (int64_t)c.heads * deepj_hip_latent_decode_splits(c.heads, hd, c.kv_rank, c.max_seq) * (hd + 4));
    r.scratch = r.alloc(sf);
    r.records = r.alloc((int64_t)c.heads * deepj_hip_attn_record_splits() * (hd + 4));
    Stream s;
    emit(s, DJ_OP_FILL, r.state, 0, 4);
    r.run(s);
    alloc_acts(r, r.dec, 1);
    if (r.narrow_positions()) {
        r.dec.part_a = r.alloc((int64_t)c.heads * c.d);
        r.dec.part_f = r.alloc((int64_t)deepj_hip_decode_ffn_parts(c.dff) * c.d);
    }
    // the prompt-sized buffers for the longest prompt the cache can take, so that no request pays for allocation
    alloc_acts(r, r.pre, c.max_seq);
    r.finalized = true;
    warm_up(r);
    make_plan(r);       // (behind the weights' fp16 copies and the workspace: a second copy for tokens takes what is left)
    if (r.plan && warms_up()) {
        decode(r, 1, 1, kGreedy);
        reset(r);
    }
}

// ── command streams ────────────────────────────────────────────────────────

// One transformer block on S rows held in a.x; result back in a.x.
void block_stream(Runner &r, Stream &s, Acts &a, int l, int S) {
    const Config &c = r.cfg;
    const Layer &L = r.layers[l];
    const int d = c.d, H = c.heads, hd = r.hd();
    bool wo_done = false, rope_fused = false;
    // a prompt's q | k | v projection takes RoPE and the cache append as its epilogue where the library has that kernel
    auto fuse_rope = [&](int k_in) { return !c.latent && !(S == 1 && &a == &r.dec) && S > 1 && deepj_hip_q8_linear_rope_ok(S, k_in, d) != 0; };
    // x2 = x + Wo . attention(RoPE(split(norm1(x) . [Wq|Wk|Wv])))      LlamaTransformerBlock.java:51
    // GPT: LayerNorm instead of RMSNorm and no rotation                  GPTTransformerBlock.java:66-68
    // DeepSeek: [Q|K|V] = ([cQ|cKV] = norm1(x).[Wdq|Wdkv]) . blockdiag(Wuq, [Wuk|Wuv])   MultiHeadLatentAttention.java:92-123
    if (c.latent) {
        // cQ = norm1(x).Wdq, Q = cQ.Wuq, cKV = norm1(x).Wdkv appended to the layer's latent rows; then, for ALL
        // cached positions, [K | V] = cKV.[Wuk | Wuv] (the row count lives on the device), RoPE on the K halves and
        // on Q, attention over the token-major rows (MultiHeadLatentAttention.java:92-123).
        const int qr = c.q_rank, kvr = c.kv_rank;
        const int64_t lat_off = (int64_t)l * c.max_seq * kvr;
        if (S == 1 && (d & 3) == 0 && d <= 4096) emit(s, DJ_OP_Q8_LINEAR_PAIR, a.x, L.g1, d, L.wdq, a.cq, qr, L.wdkv, a.ckv, kvr);
        else {
            q8_linear(s, a.x, L.wdq, a.cq, S, d, qr, DJ_LIN_RMSNORM, L.g1);
            q8_linear(s, a.x, L.wdkv, a.ckv, S, d, kvr, DJ_LIN_RMSNORM, L.g1);
        }
        q8_linear(s, a.cq, L.wuq, a.qkv, S, qr, d, 0);
        const int splits = S == 1 ? deepj_hip_latent_decode_splits(H, hd, kvr, c.max_seq) : 0;
        if (splits) {        // one row: the cache stays latent (its scratch holds the splits' records)
            emit(s, DJ_OP_LATENT_DECODE, a.qkv, a.ckv, r.latent, L.wukv, r.state, r.cos_t, r.sin_t, r.scratch, a.att, H, hd, kvr, c.max_seq, l);
        } else {
            emit(s, DJ_OP_APPEND_ROWS, a.ckv, r.latent, r.state, S, kvr, c.max_seq, lat_off);
            emit(s, DJ_OP_Q8_LINEAR_DYN, r.latent, L.wukv, r.kv_all, c.max_seq, kvr, 2 * d, r.state, S, lat_off);
            emit(s, DJ_OP_ROPE_ROWS, r.kv_all, r.kv_all, r.state, r.cos_t, r.sin_t, c.max_seq, H, hd, c.max_seq, 1, 2 * d, S);
            emit(s, DJ_OP_ROPE_ROWS, a.qkv, a.q, r.state, r.cos_t, r.sin_t, S, H, hd, c.max_seq, 0, 0, -1);
            emit(s, DJ_OP_ATTENTION_KV, a.q, r.kv_all, r.kv_all, a.att, r.state, r.scratch, S, H, hd, c.max_seq, 0, 2 * d, d);
        }
        q8_linear(s, a.att, L.wo, a.x2, S, d, d, DJ_LIN_RESIDUAL, -1, -1, -1, a.x);
        wo_done = true;
    } else if (c.kind == 1) {
        const int k2 = r.latent_width();
        q8_linear(s, a.x, L.wdown, a.cq, S, d, k2, DJ_LIN_RMSNORM, L.g1);
        if (!(rope_fused = fuse_rope(k2))) q8_linear(s, a.cq, L.wup, a.qkv, S, k2, 3 * d, 0);
        else emit(s, DJ_OP_Q8_LINEAR_ROPE, a.cq, L.wup, a.q, S, k2, d, 0, -1, -1, -1, r.kc, r.vc, r.state, r.cos_t, r.sin_t, H, hd, c.max_seq, l);
    } else if (c.kind == 2) {
        if (!(rope_fused = fuse_rope(d))) q8_linear(s, a.x, L.wqkv, a.qkv, S, d, 3 * d, DJ_LIN_LAYERNORM, L.g1, -1, L.be1);
        else emit(s, DJ_OP_Q8_LINEAR_ROPE, a.x, L.wqkv, a.q, S, d, d, DJ_LIN_LAYERNORM, L.g1, -1, L.be1, r.kc, r.vc, r.state, r.cos_t, r.sin_t, H, hd, c.max_seq, l);
    } else {
        if (!(rope_fused = fuse_rope(d))) q8_linear(s, a.x, L.wqkv, a.qkv, S, d, 3 * d, DJ_LIN_RMSNORM, L.g1);
        else emit(s, DJ_OP_Q8_LINEAR_ROPE, a.x, L.wqkv, a.q, S, d, d, DJ_LIN_RMSNORM, L.g1, -1, -1, r.kc, r.vc, r.state, r.cos_t, r.sin_t, H, hd, c.max_seq, l);
    }
    if (c.latent) {
        // attention and Wo were emitted above
    } else if (S == 1 && &a == &r.dec) {
        // the key splits' records go straight to the Wo matvec, whose prologue merges them
        emit(s, DJ_OP_ATTN_DECODE_RECORDS, a.qkv, r.kc, r.vc, r.records, r.state, r.cos_t, r.sin_t, H, hd, c.max_seq, l);
        emit(s, DJ_OP_Q8_LINEAR, r.records, L.wo, a.x2, 1, d, d, DJ_LIN_RESIDUAL | DJ_LIN_ATTN_MERGE, hd, -1, -1, a.x);
        wo_done = true;
    } else {
        if (!rope_fused) emit(s, DJ_OP_ROPE_KV_STORE, a.qkv, a.q, r.kc, r.vc, r.state, r.cos_t, r.sin_t, S, H, hd, c.max_seq, l);
        emit(s, DJ_OP_ATTENTION, a.q, r.kc, r.vc, a.att, r.state, r.scratch, S, H, hd, c.max_seq, l);
    }
    if (!wo_done) q8_linear(s, a.att, L.wo, a.x2, S, d, d, DJ_LIN_RESIDUAL, -1, -1, -1, a.x);
    if (c.kind == 2) {
        // x = x2 + W2 . GELU(W1 . ln2(x2) + b1) + b2                        GPTTransformerBlock.java:70-72, FNN.java:57-73
        q8_linear(s, a.x2, L.wgu, a.ff, S, d, c.dff, DJ_LIN_LAYERNORM | DJ_LIN_BIAS | DJ_LIN_GELU, L.g2, L.bg, L.be2);
        q8_linear(s, a.ff, L.wd, a.x, S, c.dff, d, DJ_LIN_BIAS | DJ_LIN_RESIDUAL, -1, L.bd, -1, a.x2);
        return;
    }
    // x = x2 + down(SiLU(gate(norm2(x2))) * up(norm2(x2)))                  LlamaTransformerBlock.java:52
    q8_linear(s, a.x2, L.wgu, a.ff, S, d, c.dff, DJ_LIN_RMSNORM | DJ_LIN_BIAS | DJ_LIN_SWIGLU, L.g2, L.bg, L.bu);
    q8_linear(s, a.ff, L.wd, a.x, S, c.dff, d, DJ_LIN_BIAS | DJ_LIN_RESIDUAL, -1, L.bd, -1, a.x2);
}

// The blocks of one token whose embedding row is in dec.x (without its position row), two launches each; result in dec.x.
void narrow_blocks_stream(Runner &r, Stream &s) {
    const Config &c = r.cfg;
    const Acts &a = r.dec;
    const int parts = deepj_hip_decode_ffn_parts(c.dff), hd = r.hd();
    const bool gpt = c.kind == 2;
    for (int l = 0; l < c.layers; l++) {
        const Layer &L = r.layers[l];
        if (l == 0) emit(s, DJ_OP_DECODE_ATTN, a.x, gpt ? r.pos_table : -1, gpt ? -1 : 0, -1);
        else emit(s, DJ_OP_DECODE_ATTN, a.q, a.part_f, parts, r.layers[l - 1].bd);
        emit(s, a.x2, L.g1, L.be1, c.d, L.wqkv, L.wo, r.kc, r.vc, r.state, r.cos_t, r.sin_t, a.part_a, hd, c.max_seq, l);
        emit(s, DJ_OP_DECODE_FFN, a.x2, a.part_a, c.heads, -1, a.q, L.g2, L.be2, c.d, L.wgu, L.bg, L.bu, L.wd, a.part_f, c.dff,
             gpt ? DJ_LIN_GELU : DJ_LIN_SWIGLU);
    }
    emit(s, DJ_OP_DECODE_ROW, a.q, a.part_f, parts, r.layers[c.layers - 1].bd, a.x, c.d);
}

// logits = lmHead(normF(x)) on `rows` rows                                   DecoderOnlyModel.java:62-63
void head_rows(Runner &r, Stream &s, int32_t x, int32_t out, int rows) {
    const Config &c = r.cfg;
    if (c.kind == 2) q8_linear(s, x, r.wlm, out, rows, c.d, c.vocab, DJ_LIN_LAYERNORM | DJ_LIN_BIAS, r.gf, r.blm, r.bf);
    else q8_linear(s, x, r.wlm, out, rows, c.d, c.vocab, DJ_LIN_RMSNORM | DJ_LIN_BIAS, r.gf, r.blm);
}
void head_stream(Runner &r, Stream &s, int32_t x_row) { head_rows(r, s, x_row, r.logits, 1); }

// GPT: the token rows in x (first one at position state[0]) get their learned position rows added
// (GPTModel.java:52-54).
void positions(Runner &r, Stream &s, int32_t x, int rows) {
    const Config &c = r.cfg;
    if (c.kind == 2) emit(s, DJ_OP_ADD_POSITIONS, x, r.pos_table, r.state, rows, c.d, c.max_seq);
}

// The next token, its record and its embedding row in dec.x, n positions further on.
void choose_next(Runner &r, Stream &s, Choose how, int n) {
    const Config &c = r.cfg;
    if (how == kGreedy) emit(s, DJ_OP_DECODE_NEXT, r.logits, r.state, r.tokens, c.max_seq, r.emb, r.dec.x, c.vocab, c.d, n);
    if (how == kSample) emit(s, DJ_OP_DECODE_SAMPLE, r.logits, r.state, r.tokens, c.max_seq, r.emb, r.dec.x, c.vocab, c.d, n, r.sampler);
}

// narrow: the blocks in two launches each (only where narrow_positions() says that the model takes them)
Stream decode_stream(Runner &r, Choose how, bool narrow) {
    const Config &c = r.cfg;
    Stream s;
    // A token chosen on the device: the previous step (or the prefill) already left its embedding in dec.x.  One chosen by
    // the host: gather it from state[1] first.
    if (how == kNone) emit(s, DJ_OP_EMBED_GATHER, r.emb, r.state, r.dec.x, 1, c.d, c.vocab, 1);
    if (narrow) narrow_blocks_stream(r, s);
    else {
        positions(r, s, r.dec.x, 1);
        for (int l = 0; l < c.layers; l++) block_stream(r, s, r.dec, l, 1);
    }
    head_stream(r, s, r.dec.x);
    choose_next(r, s, how, 1);
    return s;
}

// A prompt of some length runs its projections on the GEMM that loads fp16 weights straight into LDS.  The first such
// prompt writes the weights once in that layout (about 2 bytes per weight more, kept until the runner goes) instead of every
// call converting them into the workspace - layer by layer while the byte budget lasts; the layers past it convert on
// every call (same results, 40 us or so per layer and prompt slower).  (finalize()'s warm-up pass runs long prompts
// when maxSeqLen allows them, so with the warm-up on the copies exist from the start.)
void ensure_prepared(Runner &r, int n) {
    if (r.prepared_done || n < 64) return;      // (with the copies in place the GEMM takes prompts from 16 rows on, 17 to 32 aside, where its plan says so)
    r.prepared_done = true;
    const Config &c = r.cfg;
    const int d = c.d;
    Stream s;
    bool room = true;
    auto prepare = [&](int32_t w, int k, int rows) {
        int32_t tile_rows = 0;      // would the longest prompt reach the fp16 GEMM with a copy in place?
        deepj_hip_q8_gemm_tile_prepared(c.max_seq, k, rows, &tile_rows, nullptr, nullptr);
        if (!room || w < 0 || !tile_rows) return;
        const int64_t floats = deepj_hip_q8_prepared_floats(k, rows);
        if (r.prepared_budget >= 0 && r.prepared_bytes + 4 * floats > r.prepared_budget) { room = false; return; }
        int32_t p = r.alloc(floats);
        r.prepared.push_back(p);
        r.prepared_bytes += 4 * floats;
        emit(s, DJ_OP_Q8_PREPARE, w, p, k, rows);
    };
    for (const Layer &L : r.layers) {
        prepare(L.wqkv, d, 3 * d);
        prepare(L.wo, d, d);
        prepare(L.wgu, d, c.kind == 2 ? c.dff : 2 * c.dff);
        prepare(L.wd, c.dff, d);
    }
    if (!s.empty()) r.run(s);
}

void release_prepared(Runner &r) {
    for (int32_t &id : r.prepared) r.release(id);
    r.prepared.clear();
    r.prepared_bytes = 0;
    r.prepared_done = false;
}

void check_ids(const Config &c, const int32_t *ids, int n) {
    for (int i = 0; i < n; i++)
        if (ids[i] < 0 || ids[i] >= c.vocab) throw Error("Token id out of range: " + std::to_string(ids[i]));   // Embedding.java:30-32
}

// The command stream that takes the n token ids in r.pre.ids through the model at the current position.
Stream prompt_stream(Runner &r, int n, Choose how) {
    const Config &c = r.cfg;
    alloc_acts(r, r.pre, n);
    ensure_prepared(r, n);
    Stream s;
    emit(s, DJ_OP_EMBED_GATHER, r.emb, r.pre.ids, r.pre.x, n, c.d, c.vocab, 0);
    positions(r, s, r.pre.x, n);
    for (int l = 0; l < c.layers; l++) block_stream(r, s, r.pre, l, n);
    emit(s, DJ_OP_COPY, r.pre.x, r.last_x, c.d, (int64_t)(n - 1) * c.d, 0);
    head_stream(r, s, r.last_x);
    choose_next(r, s, how, n);
    return s;
}

// The device's state words as the host knows them: {positions, token, tokens generated}.
void upload_state(Runner &r, int32_t token) {
    const int32_t st[4] = {r.pos, token, r.generated, 0};
    hip(deepj_hip_upload(r.state, reinterpret_cast<const float *>(st), 4));
}

int token_launches(const Config &c, bool narrow);
void decode_steps(Runner &r, int steps, int mode, Choose how, bool narrow);
void replay(Runner &r, Choose how, bool narrow, int size, int times);

void drop_plan(Runner &r) {
    if (r.plan) hip(deepj_hip_token_plan_destroy(r.plan));
    r.plan = 0;
    r.pending.clear();
}

// A token of the caller's by launches, its logits and the state behind it
void step_by_launches(Runner &r, int32_t token, int mode) {
    upload_state(r, token);
    // Replayed like a greedy token: the launches of a token one by one cost the host 2.4 us each (43 of them: 190 us a
    // step of 8 layers, 130 as a graph).
    const bool narrow = r.pos < r.narrow_positions();
    if (mode == 1) replay(r, kNone, narrow, 2, 1);
    else r.run(decode_stream(r, kNone, narrow));
    r.pos += 1;
    r.fed = token;
    upload_state(r, token);             // the next launch takes it along, or the next step's overwrites it where it is staged
}

// DecoderOnlyModel.forward returns logits for every row; only parity tests ask for them.
void prompt_logits(Runner &r, int n, float *out) {
    const int64_t count = (int64_t)n * r.cfg.vocab;
    int32_t full = r.alloc(count);
    Stream s;
    head_rows(r, s, r.pre.x, full, n);
    r.run(s);
    hip(deepj_hip_download(full, out, count));
    r.release(full);
}

// The prompt's rows, and the state behind them
void run_prompt(Runner &r, const int32_t *ids, int n, float *all_logits, Choose how) {
    Stream s = prompt_stream(r, n, how);
    hip(deepj_hip_upload(r.pre.ids, reinterpret_cast<const float *>(ids), n));   // (prompt_stream sized r.pre for n rows)
    r.run(s);
    if (all_logits) prompt_logits(r, n, all_logits);
    r.pos += n;
    r.fed = how != kNone ? -1 : 0;
    if (how != kNone) r.generated += 1;
    else upload_state(r, 0);            // advance the position without choosing a token
}

// Whether the runs since the last look had the whole device, now that the stream has got there (`arrived`: something behind them
// has been downloaded).  Nobody waits for that before results are read, or launches follow that read them: behind a run that
// gave up none does anything, prompts work at positions that are written again, and launches do all of it once more.  True:
// results read before this call have to be read again.
bool settle(Runner &r, bool arrived = false) {
    if (r.pending.empty()) return false;
    if (!arrived) hip(deepj_hip_synchronize());
    std::vector<Runner::Pending> work;
    work.swap(r.pending);
    if (!deepj_hip_token_plan_failed(r.plan)) return false;
    drop_plan(r);
    const int32_t generated = r.generated;
    r.pos = work[0].pos;
    r.generated = work[0].generated;
    int32_t token = r.pending_fed;
    if (token < 0) {
        std::vector<int32_t> tokens((size_t)r.generated);
        hip(deepj_hip_download(r.tokens, reinterpret_cast<float *>(tokens.data()), r.generated));
        token = tokens.back();
    }
    upload_state(r, token);
    for (const Runner::Pending &w : work) {
        r.generated = w.generated;
        if (!w.prompt.empty()) run_prompt(r, w.prompt.data(), (int)w.prompt.size(), nullptr, w.chooses ? kGreedy : kNone);
        else if (!w.steps) step_by_launches(r, w.token, 0);
        else {
            Stream s;                                        // (the embedding that the launches start from)
            emit(s, DJ_OP_EMBED_GATHER, r.emb, r.state, r.dec.x, 1, r.cfg.d, r.cfg.vocab, 1);
            r.run(s);
            decode_steps(r, w.steps, 0, kGreedy, false);
            r.pos += w.steps;
        }
    }
    r.generated = generated;
    return true;
}

// Whether tokens are runs.  A plan whose memory was given back goes, once it is known what its last runs left.
bool has_plan(Runner &r) {
    if (!r.plan || deepj_hip_token_plan_groups(r.plan)) return r.plan != 0;
    settle(r);
    drop_plan(r);
    return false;
}

// Runs the prompt rows through the model, filling the cache.  Leaves the last row's
// logits in r.logits; unless `how` is kNone the next token is chosen on the device as well.
void prefill(Runner &r, const int32_t *ids, int n, float *all_logits, Choose how) {
    const Config &c = r.cfg;
    if (!r.finalized) finalize(r);
    if (n <= 0) throw Error("prefill: empty prompt");
    check_ids(c, ids, n);
    if (r.pos + n > c.max_seq)
        throw Error("context of " + std::to_string(r.pos + n) + " tokens exceeds maxSeqLen " + std::to_string(c.max_seq));
    const int32_t pos = r.pos, generated = r.generated;
    run_prompt(r, ids, n, all_logits, how);
    if (!r.pending.empty()) r.pending.push_back({pos, generated, 0, 0, {ids, ids + n}, how != kNone});
    if (all_logits && settle(r, true)) prompt_logits(r, n, all_logits);
}

void reset(Runner &r) {
    if (!r.finalized) finalize(r);
    // (what a run left is not asked for any more; one that could not finish shows in the next)
    r.pending.clear();
    r.pos = 0;
    r.generated = 0;
    r.fed = 0;
    upload_state(r, 0);
}

// A graph of kReplayTokens[size] consecutive per-token streams.
void capture(Runner &r, Choose how, bool narrow, int size) {
    Stream one = decode_stream(r, how, narrow), s;
    for (int i = 0; i < kReplayTokens[size]; i++) s.insert(s.end(), one.begin(), one.end());
    hip(deepj_hip_graph_capture(s.data(), (int32_t)s.size(), &r.graph[how][narrow][size]));
}

bool warms_up() {
    const char *env = getenv("DEEPJ_HIP_WARMUP");           // "0": skip (profiling runs that want only the request's launches)
    return !(env && env[0] == '0');
}

// The runtime builds a kernel's function object on its first launch (a few hundred microseconds each).  One pass over
// prompts of the lengths that select the different GEMM and attention variants, and a few tokens, move that from the first
// request to finalize(), and with it the capture of the graphs that greedy decoding replays first; the sequence state is
// cleared afterwards (the cache rows written here are never read: every row is rewritten before the position counter reaches
// it).  What a program may never use is left to the request that does: graphs of sampled and of caller-chosen tokens (0.5 to
// 1.3 ms once) and, for a narrow model, those of the blocks in five launches, which it takes late in a long context or never
// (1.1 ms once, where loading a 4-layer model of width 256 paid 3.3).  The 16-token graph is captured and not run: its first
// replay costs what every other does.  A model whose tokens are runs has one of a token too, behind this (finalize); the graphs
// serve what runs do not, and everything once memory or the device is shared.
void warm_up(Runner &r) {
    const Config &c = r.cfg;
    if (!warms_up()) return;
    std::vector<int32_t> ids((size_t)std::min(c.max_seq, 2048), 0);
    for (int n : {2048, 1024, 512, 256, 128, 64, 32, 16, 4}) {
        if (n > (int)ids.size()) continue;
        reset(r);
        prefill(r, ids.data(), n, nullptr, kGreedy);
    }
    const bool narrow_model = r.narrow_positions() > 0;
    if (c.max_seq >= 3 && narrow_model && r.narrow_positions() < c.max_seq) {
        reset(r);
        prefill(r, ids.data(), 1, nullptr, kGreedy);
        decode_steps(r, 1, 0, kGreedy, false);
    }
    const int steps = std::min(c.max_seq - 2, 4 + 1);
    if (steps >= 1) {
        reset(r);
        prefill(r, ids.data(), 1, nullptr, kGreedy);
        decode_steps(r, steps, 1, kGreedy, narrow_model);
    }
    if (c.max_seq > kReplayTokens[0] && token_launches(c, narrow_model) <= kShortStream) capture(r, kGreedy, narrow_model, 0);
    reset(r);
}

// `times` replays of a graph, captured on first use and again where the runtime refuses it (the workspace it used has been
// replaced by a larger one since).
void replay(Runner &r, Choose how, bool narrow, int size, int times) {
    int32_t &graph = r.graph[how][narrow][size];
    if (graph && deepj_hip_graph_launch(graph, times) == 0) return;
    if (graph) hip(deepj_hip_graph_destroy(graph));
    graph = 0;
    capture(r, how, narrow, size);
    hip(deepj_hip_graph_launch(graph, times));
}

// The launches of a token, roughly: blocks of 2 or 5 (8 over a latent cache), the row behind the narrow ones, the head and
// the choice.
int token_launches(const Config &c, bool narrow) { return narrow ? 2 * c.layers + 3 : (c.latent ? 8 : 5) * c.layers + 2; }

void decode_steps(Runner &r, int steps, int mode, Choose how, bool narrow) {
    if (mode != 1) {
        Stream s = decode_stream(r, how, narrow);
        for (int i = 0; i < steps; i++) r.run(s);
        return;
    }
    for (int size = token_launches(r.cfg, narrow) <= kShortStream ? 0 : 1; size < 3; size++) {
        if (steps >= kReplayTokens[size]) replay(r, how, narrow, size, steps / kReplayTokens[size]);
        steps %= kReplayTokens[size];
    }
}

// Steps on the device: each consumes state[1] at position state[0] and appends the token chosen as `how` says.
// mode 0: the per-token stream, eagerly; 1: the same stream as a replayed HIP graph.
void decode(Runner &r, int steps, int mode, Choose how) {
    const Config &c = r.cfg;
    if (steps <= 0) return;
    if (r.pos + steps > c.max_seq)
        throw Error("context of " + std::to_string(r.pos + steps) + " tokens exceeds maxSeqLen " + std::to_string(c.max_seq));
    if (mode == 1 && how != kNone && has_plan(r)) {
        if (how == kGreedy) {
            hip(deepj_hip_token_plan_run(r.plan, steps, 1));
            if (r.pending.empty()) r.pending_fed = r.fed;
            if (!r.pending.empty() && r.pending.back().steps) r.pending.back().steps += steps;
            else r.pending.push_back({r.pos, r.generated, steps, 0, {}, true});
        } else {                                             // (generate, which has its tokens itself, asks what became of them)
            Stream s;
            choose_next(r, s, how, 1);
            for (int i = 0; i < steps && !deepj_hip_token_plan_failed(r.plan); i++) {
                hip(deepj_hip_token_plan_run(r.plan, 1, 0));
                r.run(s);
            }
        }
        r.pos += steps;
        r.generated += steps;
        r.fed = -1;
        return;
    }
    settle(r);
    const int narrow = std::min(steps, std::max(0, r.narrow_positions() - r.pos));
    if (narrow) decode_steps(r, narrow, mode, how, true);
    if (steps > narrow) decode_steps(r, steps - narrow, mode, how, false);
    r.pos += steps;
    r.generated += steps;
    r.fed = -1;
}

// One token through the single-row path with the token chosen by the caller: logits of the
// new position end up in r.logits.  (Incremental decode with sampling done elsewhere.)
void step_token(Runner &r, int32_t token, int mode) {
    const Config &c = r.cfg;
    if (!r.finalized) finalize(r);
    check_ids(c, &token, 1);
    if (r.pos + 1 > c.max_seq)
        throw Error("context of " + std::to_string(r.pos + 1) + " tokens exceeds maxSeqLen " + std::to_string(c.max_seq));
    if (mode == 1 && has_plan(r)) {
        hip(deepj_hip_token_plan_step(r.plan, r.pos, token, r.generated));
        if (r.pending.empty()) r.pending_fed = r.fed;
        r.pending.push_back({r.pos, r.generated, 0, token, {}, false});
        r.pos += 1;
        r.fed = token;
        return;
    }
    settle(r);
    step_by_launches(r, token, mode);
}

// ── TextGenerator.sampleFromLogits on the host (temperature / top-k > 1) ────

// The stable descending order of the logits (TextGenerator.java:163-170) by a radix sort: 11 bits a pass over keys that
// order like Float.compare, least significant first, so equal logits keep their index order.
void descending_order(const std::vector<float> &logits, std::vector<int32_t> &order) {
    const size_t n = logits.size();
    struct Item { uint32_t key; int32_t index; };
    std::vector<Item> a(n), b(n);
    constexpr int kBits = 11, kBuckets = 1 << kBits;
    std::vector<uint32_t> count(3 * kBuckets, 0);
    for (size_t i = 0; i < n; i++) {
        uint32_t u;
        std::memcpy(&u, &logits[i], 4);
        if (logits[i] != logits[i]) u = 0x7fc00000u;
        u = (u & 0x80000000u) ? u : ~u & 0x7fffffffu;         // descending: positive values by falling magnitude, then negative by rising
        a[i] = {u, (int32_t)i};
        for (int pass = 0; pass < 3; pass++) count[pass * kBuckets + ((u >> (pass * kBits)) & (kBuckets - 1))]++;
    }
    for (int pass = 0; pass < 3; pass++) {
        uint32_t *c = count.data() + pass * kBuckets, at = 0;
        for (int k = 0; k < kBuckets; k++) { const uint32_t here = c[k]; c[k] = at; at += here; }
        for (const Item &it : a) b[c[(it.key >> (pass * kBits)) & (kBuckets - 1)]++] = it;
        a.swap(b);
    }
    order.resize(n);
    for (size_t i = 0; i < n; i++) order[i] = a[i].index;
}

int32_t sample_from_logits(const std::vector<float> &logits, float temperature, int top_k, void *rng) {
    int n = (int)logits.size();
    std::vector<int32_t> order;
    descending_order(logits, order);
    int k = top_k == 0 ? n : std::min(top_k, n);
    float mx = -INFINITY;
    for (int i = 0; i < k; i++) mx = std::max(mx, logits[order[i]] / temperature);
    std::vector<float> probs(k);
    float sum = 0.0f;
    for (int i = 0; i < k; i++) {
        float p = (float)std::exp((double)(logits[order[i]] / temperature - mx));
        probs[i] = p;
        sum += p;
    }
    for (float &p : probs) p /= sum;
    float u = deepj_host_random_next_float(rng), cum = 0.0f;
    for (int i = 0; i < k; i++) {
        cum += probs[i];
        if (u <= cum) return order[i];
    }
    return order[k - 1];
}

// TextGenerator.generate on token ids (TextGenerator.java:66-87).  out holds n_prompt + max_new ids.
//
// Token t is drawn from the logits of the last row of forward(last(ids, maxSeqLen)) (TextGenerator.java:91-100,
// 172-175).  While the whole sequence fits the window its rows keep their positions, so the KV cache serves them;
// once it is longer the window slides by one per token and every row's position changes, so each further token is
// a fresh forward of the maxSeqLen-row window - what the reference does for every token.
void generate_once(Runner &r, const int32_t *prompt, int n_prompt, int max_new, float temperature, int top_k,
                   int64_t seed, int32_t *out, int mode) {
    const Config &c = r.cfg;
    if (max_new < 0) throw Error("maxNewTokens must be >= 0");
    if (!(temperature > 0.0f)) throw Error("temperature must be > 0");
    if (top_k < 0) throw Error("topK must be >= 0");
    if (n_prompt <= 0 && max_new > 0) throw Error("prefill: empty prompt");
    check_ids(c, prompt, n_prompt);
    std::memcpy(out, prompt, (size_t)n_prompt * sizeof(int32_t));
    if (max_new == 0) return;
    // tokens 0 .. cached-1 see a context that fits the window (n_prompt + t <= maxSeqLen)
    const int cached = n_prompt > c.max_seq ? 0 : std::min(max_new, c.max_seq - n_prompt + 1);
    // argmax needs no random draw to pick, and greedy output is seed independent; a moderate top-k is sampled on the
    // device, so that those runs replay graphs too; the rest (whole vocabulary) is sorted and drawn from on the host
    const Choose how = top_k == 1 ? kGreedy : top_k > 0 && top_k <= DEEPJ_HIP_SAMPLE_TOP_K ? kSample : kNone;
    void *rng = how == kNone ? deepj_host_random_create(seed) : nullptr;
    try {
        std::vector<float> logits(how == kNone ? (size_t)c.vocab : 0);
        auto sample = [&](int t) {
            hip(deepj_hip_download(r.logits, logits.data(), c.vocab));
            if (settle(r, true)) hip(deepj_hip_download(r.logits, logits.data(), c.vocab));
            out[n_prompt + t] = sample_from_logits(logits, temperature, top_k, rng);
        };
        reset(r);
        if (how == kSample) {
            if (r.sampler < 0) r.sampler = r.alloc(4);
            const uint64_t start = ((uint64_t)seed ^ 0x5DEECE66DULL) & ((1ULL << 48) - 1);      // java.util.Random(seed)
            int32_t params[4] = {(int32_t)(uint32_t)start, (int32_t)(start >> 32), 0, top_k};
            std::memcpy(&params[2], &temperature, 4);
            hip(deepj_hip_upload(r.sampler, reinterpret_cast<const float *>(params), 4));
        }
        if (cached > 0 && how != kNone) {
            prefill(r, prompt, n_prompt, nullptr, how);
            decode(r, cached - 1, mode, how);
            hip(deepj_hip_download(r.tokens, reinterpret_cast<float *>(out + n_prompt), cached));
            if (r.plan && deepj_hip_token_plan_failed(r.plan)) return;          // (once more, by launches)
            r.pending.clear();
        } else if (cached > 0) {
            prefill(r, prompt, n_prompt, nullptr, kNone);
            for (int t = 0; t < cached; t++) {
                if (t > 0) step_token(r, out[n_prompt + t - 1], mode);
                sample(t);
                r.generated = t + 1;
            }
            r.fed = out[n_prompt + cached - 1];
            upload_state(r, r.fed);
        }
        for (int t = cached; t < max_new; t++) {
            reset(r);
            prefill(r, out + n_prompt + t - c.max_seq, c.max_seq, nullptr, how);
            if (how != kNone) hip(deepj_hip_download(r.tokens, reinterpret_cast<float *>(out + n_prompt + t), 1));
            else sample(t);
        }
    } catch (...) {
        if (rng) deepj_host_random_destroy(rng);
        throw;
    }
    if (rng) deepj_host_random_destroy(rng);
}

void generate(Runner &r, const int32_t *prompt, int n_prompt, int max_new, float temperature, int top_k,
              int64_t seed, int32_t *out, int mode) {
    generate_once(r, prompt, n_prompt, max_new, temperature, top_k, seed, out, mode);
    if (!r.plan || !deepj_hip_token_plan_failed(r.plan)) return;       // (its tokens have been downloaded)
    drop_plan(r);
    generate_once(r, prompt, n_prompt, max_new, temperature, top_k, seed, out, mode);
}

template <class F> int guarded(Runner *r, F &&f) {
    try {
        f();
        if (r) r->error.clear();
        return 0;
    } catch (const std::exception &ex) {
        if (r) r->error = ex.what();
        return 1;
    }
}

}  // namespace

extern "C" {

// cfg: {kind, vocab, maxSeq, dModel, nHeads, nLayers, dFF, qRank, kvRank}; id_base: first buffer id this
// runner may use (pick a range the ComputeGraph never reaches, e.g. 1 << 29).
void *deepj_runner_create(const int32_t cfg[9], int32_t id_base) {
    Config c{cfg[0], cfg[1], cfg[2], cfg[3], cfg[4], cfg[5], cfg[6], cfg[7], cfg[8]};
    if (c.kind == 3) { c.kind = 1; c.latent = true; }      // DeepSeek with the latent KV cache
    // TransformerConfig.validateCommon (models/TransformerConfig.java:19-31) + DeepSeekConfig.java:31-35
    if (c.vocab <= 0 || c.max_seq <= 0 || c.d <= 0 || c.heads <= 0 || c.layers <= 0 || c.dff <= 0) return nullptr;
    if (c.d % c.heads != 0) return nullptr;
    if (c.kind == 1 && (c.q_rank <= 0 || c.kv_rank <= 0)) return nullptr;
    if (c.kind < 0 || c.kind > 2) return nullptr;
    int hd = c.d / c.heads;
    if (hd != 32 && hd != 64 && hd != 128) return nullptr;
    auto *r = new Runner;
    r->cfg = c;
    r->next_id = id_base;
    r->layers.resize((size_t)c.layers);
    return r;
}

void deepj_runner_destroy(void *h) {
    auto *r = static_cast<Runner *>(h);
    if (!r) return;
    for (int how = 0; how < 3; how++)
        for (auto &sizes : r->graph[how])
            for (int32_t g : sizes)
                if (g) deepj_hip_graph_destroy(g);
    if (r->plan) deepj_hip_token_plan_destroy(r->plan);
    deepj_hip_synchronize();
    // every id in [id_base, next_id) that is still live belongs to this runner
    std::vector<int32_t> ids;
    auto add = [&](int32_t id) { if (id >= 0) ids.push_back(id); };
    for (auto &L : r->layers)
        for (int32_t id : {L.g1, L.g2, L.be1, L.be2, L.wqkv, L.wo, L.wdown, L.wup, L.wdq, L.wuq, L.wdkv, L.wukv, L.wgu, L.bg,
                           L.bu, L.wd, L.bd})
            add(id);
    for (int32_t id : {r->emb, r->gf, r->wlm, r->blm, r->cos_t, r->sin_t, r->kc, r->vc, r->state,
                       r->tokens, r->scratch, r->records, r->logits, r->last_x,
                       r->pos_table, r->bf, r->latent, r->kv_all, r->sampler})
        add(id);
    for (Acts *a : {&r->dec, &r->pre})
        for (int32_t id : {a->x, a->x2, a->qkv, a->q, a->att, a->ff, a->ids, a->cq, a->ckv, a->part_a, a->part_f}) add(id);
    for (int32_t id : r->prepared) add(id);
    if (!ids.empty()) deepj_hip_release(ids.data(), (int32_t)ids.size());
    delete r;
}

const char *deepj_runner_last_error(void *h) { return h ? static_cast<Runner *>(h)->error.c_str() : "null runner"; }

int deepj_runner_set_weight(void *h, const char *name, const float *data, int32_t rows, int32_t cols) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] { set_weight(*r, name, data, rows, cols); });
}

int deepj_runner_init_seeded(void *h, int64_t seed, int32_t threads) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        if (r->cfg.kind == 2) throw Error("a GPT model is seeded through deepj_runner_init_seeded_gpt (it needs initScale)");
        init_seeded(*r, seed, threads, 1.0f);
    });
}

int deepj_runner_init_seeded_gpt(void *h, int64_t seed, float init_scale, int32_t threads) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        if (r->cfg.kind != 2) throw Error("deepj_runner_init_seeded_gpt: not a GPT model");
        if (!std::isfinite(init_scale) || init_scale <= 0.0f) throw Error("initScale must be finite and > 0");   // GPTConfig.java:22-23
        init_seeded(*r, seed, threads, init_scale);
    });
}

// Bytes the runner may spend on fp16 copies of its weights for the many-row (prompt) GEMM: -1 no limit (every layer:
// + 2 bytes per weight), 0 none (every call converts into the workspace), otherwise layers in order while the budget
// lasts.  Copies held under an earlier budget are released; the next long prompt prepares anew.  Results do not
// depend on it.
int deepj_runner_set_prepared_budget(void *h, int64_t bytes) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        if (bytes < -1) throw Error("prepared-weight budget must be -1 (no limit) or a byte count");
        release_prepared(*r);
        r->prepared_budget = bytes;
    });
}

// XCDs that token runs take: 0 the library's choice, -1 none (tokens are replayed graphs).  Before finalize.
int deepj_runner_set_token_groups(void *h, int32_t groups) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        if (r->finalized) throw Error("set_token_groups after finalize");
        if (groups < -1 || groups > 8) throw Error("token groups must be -1 (no token runs), 0 (the library's choice) or 1 to 8");
        r->token_groups = groups;
    });
}

int32_t deepj_runner_token_plan(void *h) {
    const int32_t plan = h ? static_cast<Runner *>(h)->plan : 0;
    return plan && deepj_hip_token_plan_groups(plan) ? plan : 0;
}

int64_t deepj_runner_prepared_bytes(void *h) { return h ? static_cast<Runner *>(h)->prepared_bytes : 0; }

int deepj_runner_finalize(void *h) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] { finalize(*r); });
}

int deepj_runner_reset(void *h) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] { reset(*r); });
}

// all_logits: null, or room for n*vocab floats (logits of every prompt row, as DecoderOnlyModel.forward returns)
int deepj_runner_prefill(void *h, const int32_t *ids, int32_t n, float *all_logits, int32_t choose_next) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] { prefill(*r, ids, n, all_logits, choose_next != 0 ? kGreedy : kNone); });
}

int deepj_runner_decode(void *h, int32_t steps, int32_t mode) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        if (mode < 0 || mode > 1) throw Error("decode: mode must be 0 (eager) or 1 (graph)");
        decode(*r, steps, mode, kGreedy);
    });
}

int deepj_runner_step(void *h, int32_t token) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] { step_token(*r, token, 1); });
}

int deepj_runner_last_logits(void *h, float *out) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        hip(deepj_hip_download(r->logits, out, r->cfg.vocab));
        if (settle(*r, true)) hip(deepj_hip_download(r->logits, out, r->cfg.vocab));
    });
}

// tokens generated so far in this sequence (device order); returns the count through *n
int deepj_runner_tokens(void *h, int32_t *out, int32_t capacity, int32_t *n) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        int32_t count = std::min(r->generated, capacity);
        if (count > 0) hip(deepj_hip_download(r->tokens, reinterpret_cast<float *>(out), count));
        else hip(deepj_hip_synchronize());
        if (settle(*r, true) && count > 0) hip(deepj_hip_download(r->tokens, reinterpret_cast<float *>(out), count));
        if (n) *n = count;
    });
}

int deepj_runner_generate(void *h, const int32_t *prompt, int32_t n_prompt, int32_t max_new, float temperature,
                          int32_t top_k, int64_t seed, int32_t mode, int32_t *out) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        if (mode < 0 || mode > 1) throw Error("generate: mode must be 0 (eager) or 1 (graph)");
        generate(*r, prompt, n_prompt, max_new, temperature, top_k, seed, out, mode);
    });
}

// The command stream of an n-token prompt at the current position, over the ids of the last prefill of that length
// (for inspection and timing by the caller; running it advances nothing on the host side).
int deepj_runner_prefill_stream(void *h, int32_t n, int32_t *out, int32_t capacity, int32_t *len) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        if (!r->finalized) finalize(*r);
        settle(*r);
        if (n <= 0 || r->pos + n > r->cfg.max_seq) throw Error("prefill_stream: row count outside the context window");
        Stream s = prompt_stream(*r, n, kNone);
        if (len) *len = (int32_t)s.size();
        if (out && capacity >= (int32_t)s.size()) std::memcpy(out, s.data(), s.size() * sizeof(int32_t));
    });
}

// The per-token command stream (for inspection, timing and graph capture by the caller).
int deepj_runner_decode_stream(void *h, int32_t *out, int32_t capacity, int32_t *len) {
    auto *r = static_cast<Runner *>(h);
    return guarded(r, [&] {
        if (!r->finalized) finalize(*r);
        settle(*r);
        Stream s = decode_stream(*r, kGreedy, r->pos < r->narrow_positions());
        if (len) *len = (int32_t)s.size();
        if (out && capacity >= (int32_t)s.size()) std::memcpy(out, s.data(), s.size() * sizeof(int32_t));
    });
}

}  // extern "C"
