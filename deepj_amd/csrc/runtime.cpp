// Device runtime behind the C ABI: the buffer/residency manager, the command-stream
// interpreter and HIP-graph capture.  It takes the place of the reference's native
// library (native/deepj_metal_jni.mm:1350-2140: gBufferPool + the opcode switch) and
// keeps its observable contract: ids are chosen by the caller, allocating an existing
// id and releasing an unknown id are no-ops, uploads copy the caller's array length,
// and a stream is executed in program order.
//
// What is different by design:
//  * Tensors stay resident in HBM between flushes; released buffers go to a
//    size-class cache, so the "new output id + release the old id" pattern that
//    in-place ops arrive as (MetalBackend.java:400-411) costs no hipMalloc/hipFree.
//  * flush only enqueues on one in-order HIP stream; download is the single
//    synchronisation point (the reference waits for the GPU in every flush,
//    deepj_metal_jni.mm:2126-2127).
//  * The whole stream is validated on the host - opcode, stride, ids, buffer sizes,
//    shapes - before the first kernel is launched, so a malformed stream can never
//    make a kernel touch memory it does not own.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <system_error>
#include <thread>
#include <unordered_map>
#include <vector>

#include <pthread.h>
#include <sys/mman.h>

#include "dj_common.h"
#include "token_run.h"
#include "gemm_rows.h"

namespace dj {

LaunchTiming g_launch_timing;

namespace {

struct Buffer {
    void *ptr = nullptr;
    size_t capacity = 0;      // bytes actually owned (size class)
    int64_t floats = 0;       // size the caller asked for
    uint64_t made = 0;        // a number of its own
};

// Floats of device scratch that a stream needs: the workspace, and the block for the Q8 GEMM that multiplies a batch of rows
// straight from the int8 weights (the rows in pieces, its partial products).
struct Scratch { int64_t workspace = 0, row_pieces = 0; };

// A captured graph holds raw device addresses.  The buffers its stream named (id, address at capture time) and
// the workspace it used are remembered, and a replay is refused once any of them is gone or has moved.  The block of pieces
// it used is kept for it instead: products that need no workspace stay launchable whatever other streams need.
struct Graph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<std::pair<int32_t, void *>> refs;
    float *workspace = nullptr;       // set when the stream needs workspace
    float *row_pieces = nullptr;      // set when the stream needs it; freed with the last graph once a larger one has replaced it
    // (weight id, prepared id) of every Q8_LINEAR that was captured reading a prepared copy the stream had not written
    // itself: once the copy stops standing for the weights (they were written again) a replay would use stale weights
    std::vector<std::pair<int32_t, int32_t>> prepared, self_prepared;
};

// A model's tokens in one launch (kernels_token.hip).  The plan holds the weights in that kernel's order, the block its
// workgroups exchange words in, and the buffers it was made over (id, number); a run is refused once one of them is gone, also where
// another of its id lies in its place: the plan's weights are those of the first.
struct TokenPlan {
    TokenRun run{};
    std::vector<std::pair<int32_t, uint64_t>> refs;
    struct Block { void *p; size_t bytes; };
    std::vector<Block> blocks;        // device memory it owns; none: given back where other memory was short
    uint32_t next_tag = 1;            // (the exchange block starts as zeros)
    uint64_t releases_seen = 0;       // g.releases when refs were last found to be there
    int slot = -1;                    // its word of the pinned block: set by a run that could not finish
    bool launched = false;            // some run was
};
constexpr int kPlanSlots = 1024;

constexpr int kRingSegments = 4;
constexpr size_t kRingSegmentBytes = (size_t)1 << 20;
constexpr size_t kStageBytes = (size_t)4 << 20;
constexpr int64_t kMaxFlags = 16384;
constexpr size_t kStageAt = kRingSegments * kRingSegmentBytes, kFlagsAt = kStageAt + kStageBytes;
constexpr size_t kPlansAt = kFlagsAt + (size_t)kMaxFlags * sizeof(uint32_t);
constexpr size_t kPinnedBytes = kPlansAt + (size_t)kPlanSlots * sizeof(uint32_t);

// Host memory that kernels and the host read and write while either runs (the ring, the stage, flags, results whose chunks are
// announced by flags) has to be coherent; the default is so only as long as the environment (HIP_HOST_COHERENT) leaves it.
constexpr unsigned kPinnedFlags = hipHostMallocCoherent;

struct Runtime {
    bool ready = false;
    int device = 0;
    hipStream_t stream = nullptr;
    std::unordered_map<int32_t, Buffer> live;
    std::map<size_t, std::vector<void *>> cache;   // size class -> free blocks
    int64_t live_bytes = 0, cached_bytes = 0, driver_allocs = 0;
    size_t cache_limit = (size_t)16 << 30;
    int64_t memory_limit = -1;                     // bytes that may be held (device_held); -1: what the device has
    float *workspace = nullptr;
    int64_t workspace_floats = 0;
    float *row_pieces = nullptr;
    int64_t row_pieces_floats = 0;
    // Host <-> device traffic (section "transfers"): one pinned block holds the upload ring, the download stage and the
    // flags that a download's chunks set.
    unsigned char *pinned = nullptr;
    size_t ring_at = 0;                            // next free byte of the ring
    int ring_segment = 0;
    hipEvent_t ring_done[kRingSegments] = {};      // recorded behind the last launch that read the segment
    bool ring_used[kRingSegments] = {};
    UploadPieces pieces;                           // staged uploads that no launch has taken over yet
    int n_pieces = 0;
    uint32_t tag = 0;                              // of the last download
    bool capturing = false;
    std::unordered_map<int32_t, Graph> graphs;
    int32_t next_graph = 1;
    std::map<int32_t, TokenPlan> plans;
    uint64_t releases = 0, made = 0;               // buffers that have gone, and been made, so far
    int32_t next_plan = 1;
    unsigned *attn_counters = nullptr;             // kAttnCounterHeads zeroed words: decode attention's split arrivals
    unsigned char *static_scratch = nullptr;       // device address of `scratch` below on g.device
    // Set by a K-sharing fp16 GEMM that also wrote the activations of the op right behind it in that op's layout
    // (GemmChain): which op of which stream, reading which buffer through which gain.  Good for that one op only.
    struct ChainSlot { const int32_t *cmd = nullptr; int32_t pos = -1, x_id = -1, gamma_id = -1, beta_id = -1; int64_t m = 0, k = 0, pieces_at = 0; bool pieces = false, plain = false, valid = false; } chain;
    bool no_alloc = false;                         // inside deepj_hip_flush_ops_noalloc: nothing may allocate
    std::vector<std::pair<int32_t, void *>> *track = nullptr;   // graph capture: buffers the dry pass resolves
    Graph *capture_into = nullptr;                               // graph capture: the graph the run pass records for
    struct Prepared { int32_t id; int k, rows; };
    std::unordered_map<int32_t, Prepared> prepared;   // Q8 weight buffer -> its copy in the fp16 GEMM's layout (OP_Q8_PREPARE)
};

Runtime g;
thread_local std::string g_error;

// Scratch memory of deepj_hip_flush_ops_noalloc, part of the loaded code object (each GPU the library runs on
// holds its own copy until the process ends): the arrival counters of the split decode attention, then the
// workspace that Q8_LINEAR's GEMM path writes its normalised activation rows to.  Host code never uses the
// symbol itself as an address: ensure_init() asks the runtime where the array lives on the current device.
constexpr size_t kStaticCounterBytes = (size_t)kAttnCounterHeads * sizeof(unsigned);
constexpr int64_t kStaticWorkspaceFloats = DEEPJ_HIP_NOALLOC_WORKSPACE_FLOATS;   // 8 MiB: e.g. 512 rows of 4096 floats
static __device__ __align__(256) unsigned char scratch[kStaticCounterBytes + (size_t)kStaticWorkspaceFloats * 4];

void ensure_init(int device = 0) {
    if (g.ready) return;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count <= 0) fail("deepj_hip: no HIP device available");
    if (device < 0 || device >= count) fail("deepj_hip: bad device index " + std::to_string(device));
    DJ_HIP(hipSetDevice(device));
    DJ_HIP(hipStreamCreateWithFlags(&g.stream, hipStreamNonBlocking));
    DJ_HIP(hipHostMalloc((void **)&g.pinned, kPinnedBytes, kPinnedFlags));
    std::memset(g.pinned, 0, kPinnedBytes);       // the flags start at 0; and no transfer pays for a page's first use (1.4 us each)
    g.ring_at = 0; g.ring_segment = 0; g.n_pieces = 0; g.tag = 0;
    for (int i = 0; i < kRingSegments; i++) {
        DJ_HIP(hipEventCreateWithFlags(&g.ring_done[i], hipEventDisableTiming));
        g.ring_used[i] = false;
    }
    DJ_HIP(hipMalloc((void **)&g.attn_counters, kAttnCounterHeads * sizeof(unsigned)));
    DJ_HIP(hipMemset(g.attn_counters, 0, kAttnCounterHeads * sizeof(unsigned)));
    g.static_scratch = nullptr;
    DJ_HIP(hipGetSymbolAddress((void **)&g.static_scratch, HIP_SYMBOL(scratch)));
    if (!g.static_scratch) fail("deepj_hip: the static scratch array has no device address");
    DJ_HIP(hipMemset(g.static_scratch, 0, kStaticCounterBytes));
    q8_gemm_f16_configure();
    q8_gemm_rows_configure();
    latent_decode_configure();
    g.device = device;
    g.ready = true;
}

// ── transfers ───────────────────────────────────────────────────────────────
// Uploads are copied into a pinned ring and leave it in one launch per flush (k_upload_pieces), large ones piece by piece while
// the next piece is copied; downloads arrive chunk by chunk in a pinned stage, or straight in the caller's memory where that
// came from deepj_hip_host_alloc.  Nothing here waits for the stream except a full ring and a download for its own chunks.
// Measured for one tensor operation on a 64 x 32 matrix (two uploads, a product, a download): 57 us with a synchronisation
// per upload and copy calls.

// Launches what is staged.  Every path that enqueues work or hands a block to another buffer calls it first; a download
// only where it would read what is staged.
void launch_uploads() {
    if (!g.n_pieces) return;
    const int n = g.n_pieces;
    g.n_pieces = 0;
    launch_upload_pieces(g.stream, g.pieces, n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) fail(std::string("upload failed: ") + hipGetErrorString(e));
}

bool staged_for(const float *p, int64_t n) {
    for (int i = 0; i < g.n_pieces; i++)
        if (g.pieces.p[i].dst < p + n && p < g.pieces.p[i].dst + g.pieces.p[i].n) return true;
    return false;
}

// `bytes` (at most a segment) of the ring; waits for the device only where the ring comes round to a segment in use.
unsigned char *ring_take(size_t bytes) {
    bytes = (bytes + 255) & ~(size_t)255;
    if (g.ring_at + bytes > kRingSegmentBytes) {
        launch_uploads();
        DJ_HIP(hipEventRecord(g.ring_done[g.ring_segment], g.stream));
        g.ring_used[g.ring_segment] = true;
        g.ring_segment = (g.ring_segment + 1) % kRingSegments;
        g.ring_at = 0;
        if (g.ring_used[g.ring_segment]) DJ_HIP(hipEventSynchronize(g.ring_done[g.ring_segment]));
    }
    unsigned char *p = g.pinned + g.ring_segment * kRingSegmentBytes + g.ring_at;
    g.ring_at += bytes;
    return p;
}

// Copies into the ring for uploads above 4 MiB on two threads: one alone copies 26 GB/s from memory it has not touched lately,
// where the link takes 57.  The second one lives for the upload (it costs some 30 us) and copies the second half of every
// piece: 64 MiB in 1.65 ms instead of 2.5, all weights of a 1 B parameter Llama in 94 ms instead of 145.  A copy call takes 2.2
// and 117, and leaves 0.1 ms to the next synchronisation of the stream, as it pins the caller's pages.
class SecondCopier {
public:
    explicit SecondCopier(bool wanted) {
        if (!wanted || std::thread::hardware_concurrency() < 2) return;
        try {
            worker = std::thread([this] { work(); });
        } catch (const std::system_error &) {      // no thread to be had: one copies
        }
    }
    ~SecondCopier() {
        if (!worker.joinable()) return;
        to = nullptr;
        asked.store(asked.load(std::memory_order_relaxed) + 1, std::memory_order_release);
        worker.join();
    }
    void copy(unsigned char *dst, const unsigned char *src, size_t bytes) {
        const size_t first = worker.joinable() ? (bytes / 2) & ~(size_t)63 : bytes;
        if (first < bytes) {
            to = dst + first; from = src + first; size = bytes - first;
            asked.store(asked.load(std::memory_order_relaxed) + 1, std::memory_order_release);
        }
        std::memcpy(dst, src, first);
        if (first < bytes) wait(done, asked.load(std::memory_order_relaxed));
    }

private:
    static void wait(const std::atomic<uint64_t> &counter, uint64_t value) {
        for (int spins = 0; counter.load(std::memory_order_acquire) < value; spins++)
            if (spins < 1000) __builtin_ia32_pause();
            else std::this_thread::yield();
    }
    void work() {
        for (uint64_t i = 1;; i++) {
            wait(asked, i);
            if (!to) return;
            std::memcpy(to, from, size);
            done.store(i, std::memory_order_release);
        }
    }
    std::atomic<uint64_t> asked{0}, done{0};
    unsigned char *to = nullptr;
    const unsigned char *from = nullptr;
    size_t size = 0;
    std::thread worker;
};

void stage_upload(float *dst, const float *src, int64_t n) {
    // pieces of a quarter segment: the first is on the link while the next is copied; whole segments from 2 MiB on, where a
    // launch for every quarter (2.4 us) would cost a fifth of its copy
    constexpr int64_t kSegment = (int64_t)(kRingSegmentBytes / 4);
    const int64_t piece = n > 2 * kSegment ? kSegment : kSegment / 4;
    for (int i = 0; i < g.n_pieces; i++) {
        const UploadPiece &p = g.pieces.p[i];
        if (p.dst == dst && p.n == n) {                       // the same words again before anything read them: the later values stand
            std::memcpy(const_cast<float *>(p.src), src, (size_t)n * 4);
            return;
        }
    }
    if (staged_for(dst, n)) launch_uploads();                 // pieces of one launch run side by side: no two into the same words
    SecondCopier copier(n > 4 * kSegment);
    for (int64_t at = 0; at < n; at += piece) {
        const int64_t len = std::min(piece, n - at);
        unsigned char *p = ring_take((size_t)len * 4);
        copier.copy(p, reinterpret_cast<const unsigned char *>(src + at), (size_t)len * 4);
        g.pieces.p[g.n_pieces++] = UploadPiece{reinterpret_cast<const float *>(p), dst + at, len};
        if (g.n_pieces == kUploadPieces || n > piece) launch_uploads();
    }
}

// Until flags[0..n) hold `tag`, in order; done(i) runs as each arrives.  A short wait spins (the chunk is a launch away);
// a longer one lets the runtime block, and a stream that ended without setting its flags is an error, not a hang.
template <class Done> void wait_flags(volatile uint32_t *flags, int64_t n, uint32_t tag, Done &&done) {
    for (int64_t i = 0; i < n; i++) {
        for (int spins = 0; __atomic_load_n(flags + i, __ATOMIC_ACQUIRE) != tag; spins++) {
            __builtin_ia32_pause();
            if (spins < 20000) continue;                      // about 0.5 ms
            DJ_HIP(hipStreamSynchronize(g.stream));
            if (__atomic_load_n(flags + i, __ATOMIC_ACQUIRE) != tag) fail("download: the stream ended without delivering the buffer");
        }
        done(i);
    }
}

// Host memory the caller may have results put into without a copy: pinned blocks, handed out again after they come back.
// A block is dear: hipHostMalloc takes 15 us to 0.7 ms, and the host's first use of each of its pages 1.4 us (80 MB: 27 ms, ten
// times what ordinary memory takes), where a download saves 5 us at 256 KiB, 23 at 1 MiB and 5 ms at 80 MB.  So it is made -
// its pages in use, nothing of that left to whoever reads the result - for sizes (by octaves) that were asked for kHostAsked
// times without one: two of them, as a loop holds one result while the next arrives, or kHostAhead bytes where that is more (the
// arrays of a training step's tensors, which are filled again at every step), and then one more for every two times that one
// has come back and been used again.  A program that wants a few results, or keeps large ones, is given ordinary memory.
// Bounded: at most kHostLive bytes are out at a time and kHostCached kept for reuse.  Locked: finalisers of the arrays over
// them run on any thread.
// The driver keeps pinned pages out of a forked child, which may hold arrays over them (a worker that reads results): what
// the blocks in use hold is copied before the fork and moved to the blocks' addresses in the child, as ordinary memory.
struct HostPool {
    std::mutex lock;
    std::vector<std::pair<uintptr_t, void *>> saved;  // between fork's handlers: blocks in use, copies of them (null: no memory)
    bool fork_handled = false, forked = false;        // handlers registered; this process is the child of one that had blocks
    std::map<uintptr_t, size_t> out;               // blocks in use: address -> class
    std::map<size_t, std::vector<void *>> free;
    size_t live = 0, cached = 0;
    struct Octave { int asked = 0; size_t ahead = 0; } octaves[64];  // bytes of blocks made, less half of those used again
};
constexpr size_t kHostLive = (size_t)1 << 30, kHostCached = (size_t)512 << 20, kHostLeast = (size_t)64 << 10, kPage = 4096;
constexpr size_t kHostAhead = (size_t)16 << 20;
constexpr int kHostAsked = 4;
HostPool g_host;

size_t size_class(size_t bytes);

void before_fork() {
    g_host.lock.lock();
    if (g_host.forked) return;                     // (a child's arrays are its own memory)
    for (const auto &block : g_host.out) {
        void *copy = mmap(nullptr, block.second, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
        if (copy == MAP_FAILED) copy = nullptr;
        else std::memcpy(copy, reinterpret_cast<const void *>(block.first), block.second);
        g_host.saved.emplace_back(block.first, copy);
    }
}
void after_fork(bool child) {
    for (const auto &block : g_host.saved) {
        if (!block.second) continue;
        const size_t size = g_host.out[block.first];
        if (child) (void)mremap(block.second, size, size, MREMAP_MAYMOVE | MREMAP_FIXED, reinterpret_cast<void *>(block.first));
        else (void)munmap(block.second, size);
    }
    g_host.saved.clear();
    if (child && !g_host.forked) {
        g_host.forked = true;
        g_host.free.clear();
        g_host.cached = 0;
    }
    g_host.lock.unlock();
}

void *host_take(size_t bytes) {
    if (bytes < kHostLeast) return nullptr;
    const size_t cls = size_class(bytes);
    HostPool::Octave &octave = g_host.octaves[63 - __builtin_clzll(bytes)];
    {
        std::lock_guard<std::mutex> hold(g_host.lock);
        if (g_host.forked) return nullptr;
        if (!g_host.fork_handled) g_host.fork_handled = pthread_atfork(before_fork, [] { after_fork(false); }, [] { after_fork(true); }) == 0;
        if (!g_host.fork_handled) return nullptr;
        for (auto it = g_host.free.lower_bound(cls); it != g_host.free.end() && it->first <= 4 * cls; ++it) {
            if (it->second.empty() || g_host.live + it->first > kHostLive) continue;
            void *p = it->second.back();
            g_host.out.emplace((uintptr_t)p, it->first);
            it->second.pop_back();
            g_host.cached -= it->first;
            g_host.live += it->first;
            octave.ahead -= std::min(octave.ahead, cls / 2);
            return p;
        }
        if (octave.asked < kHostAsked) { octave.asked++; return nullptr; }
        if (octave.ahead + cls > std::max(2 * cls, kHostAhead) || g_host.live + cls > kHostLive) return nullptr;
        octave.ahead += cls;
        g_host.live += cls;                        // (the block itself is made outside the lock)
    }
    void *p = nullptr;
    const bool ok = hipHostMalloc(&p, cls, kPinnedFlags) == hipSuccess;
    if (ok)
        for (size_t at = 0; at < cls; at += kPage) static_cast<volatile unsigned char *>(p)[at] = 0;
    else (void)hipGetLastError();
    std::lock_guard<std::mutex> hold(g_host.lock);
    if (ok) g_host.out.emplace((uintptr_t)p, cls);
    else { octave.ahead -= std::min(octave.ahead, cls); g_host.live -= cls; }
    return ok ? p : nullptr;
}

void host_give_back(void *p) {
    std::lock_guard<std::mutex> hold(g_host.lock);
    auto it = g_host.out.find((uintptr_t)p);
    if (it == g_host.out.end()) return;
    const size_t cls = it->second;
    g_host.out.erase(it);
    g_host.live -= cls;
    if (g_host.forked) { (void)munmap(p, cls); return; }
    if (g_host.cached + cls > kHostCached) { (void)hipHostFree(p); return; }
    g_host.free[cls].push_back(p);
    g_host.cached += cls;
}

void host_trim() {
    std::lock_guard<std::mutex> hold(g_host.lock);
    for (auto &kv : g_host.free)
        for (void *p : kv.second) (void)hipHostFree(p);
    g_host.free.clear();
    g_host.cached = 0;
    for (HostPool::Octave &o : g_host.octaves) o = {};
}

bool host_owned(const void *p, size_t bytes) {
    std::lock_guard<std::mutex> hold(g_host.lock);
    auto it = g_host.out.upper_bound((uintptr_t)p);
    if (it == g_host.out.begin()) return false;
    --it;
    return (uintptr_t)p + bytes <= it->first + it->second;
}

void download(const float *src, float *dst, int64_t n) {
    uint32_t *flags = reinterpret_cast<uint32_t *>(g.pinned + kFlagsAt);
    float *stage = reinterpret_cast<float *>(g.pinned + kStageAt);
    // straight into the caller's block where the device can write there in 128-bit words
    const bool direct = ((uintptr_t)dst & 15) == 0 && host_owned(dst, (size_t)n * 4);
    for (int64_t at = 0; at < n;) {
        // chunks of 8 KiB where few of them would otherwise leave a workgroup the whole transfer, 64 KiB from 512 KiB on
        const int64_t chunk = (n - at) * 4 <= (512 << 10) ? 2048 : 16384;
        const int64_t len = std::min(n - at, direct ? kMaxFlags * chunk : (int64_t)(kStageBytes / 4));
        const int64_t chunks = (len + chunk - 1) / chunk;
        if (++g.tag == 0) g.tag = 1;
        launch_download(g.stream, src + at, direct ? dst + at : stage, len, chunk, flags, g.tag);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) fail(std::string("download failed: ") + hipGetErrorString(e));
        wait_flags(flags, chunks, g.tag, [&](int64_t c) {
            if (!direct) std::memcpy(dst + at + c * chunk, stage + c * chunk, (size_t)std::min(chunk, len - c * chunk) * 4);
        });
        at += len;
    }
}

// A prepared copy stops standing for its Q8 buffer as soon as either is released or written.
void forget_prepared(int32_t id) {
    if (g.prepared.empty()) return;
    g.prepared.erase(id);
    for (auto it = g.prepared.begin(); it != g.prepared.end();) it = it->second.id == id ? g.prepared.erase(it) : std::next(it);
}

// 256 B granularity up to 64 KiB, then four classes per power of two (<= 25 % slack).
size_t size_class(size_t bytes) {
    if (bytes < 256) return 256;
    if (bytes <= (64u << 10)) return (bytes + 255) & ~(size_t)255;
    size_t p = (size_t)1 << (63 - __builtin_clzll(bytes));      // largest power of two <= bytes
    if (p == bytes) return bytes;
    size_t step = p >> 2;
    return (bytes + step - 1) / step * step;
}

// The memory of token plans, weights that their models hold a second time: back to the driver.  Their models' tokens go on as launches.
bool give_plans_back() {
    bool some = false;
    for (auto &kv : g.plans) {
        for (const TokenPlan::Block &b : kv.second.blocks) {
            (void)hipFree(b.p);
            g.live_bytes -= (int64_t)b.bytes;
            some = true;
        }
        kv.second.blocks.clear();
    }
    return some;
}

int64_t device_held() { return g.live_bytes + g.cached_bytes + 4 * (g.workspace_floats + g.row_pieces_floats); }

// Device memory from the driver.  Where that has none left, what the pool keeps goes back to it first, then what token plans hold
// (not for the sake of another plan).
void *device_memory(size_t bytes, bool for_plan = false) {
    void *p = nullptr;
    auto ask = [&] { return g.memory_limit >= 0 && device_held() + (int64_t)bytes > g.memory_limit ? hipErrorOutOfMemory : hipMalloc(&p, bytes); };
    hipError_t e = ask();
    if (e != hipSuccess) {
        (void)hipGetLastError();
        DJ_HIP(hipStreamSynchronize(g.stream));
        for (auto &kv : g.cache) {
            for (void *q : kv.second) (void)hipFree(q);
            kv.second.clear();
        }
        g.cached_bytes = 0;
        e = ask();
        if (e != hipSuccess && !for_plan && give_plans_back()) {
            (void)hipGetLastError();
            e = ask();
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            fail("Failed to allocate HIP buffer of " + std::to_string(bytes) + " bytes: " + hipGetErrorString(e));
        }
    }
    g.driver_allocs++;
    return p;
}

void *pool_alloc(size_t cls, bool for_plan = false) {
    auto it = g.cache.find(cls);
    if (it != g.cache.end() && !it->second.empty()) {
        void *p = it->second.back();
        it->second.pop_back();
        g.cached_bytes -= (int64_t)cls;
        return p;
    }
    if (g.capturing) fail("deepj_hip: device allocation requested while a graph is being captured");
    if (g.no_alloc) fail("deepj_hip: device allocation requested inside the allocation-free entry point");
    return device_memory(cls, for_plan);
}

void pool_free(void *p, size_t cls) {
    // Work already queued on the stream may still use the block; any later user is
    // queued behind it on the same in-order stream, so recycling needs no wait.
    if ((size_t)g.cached_bytes + cls > g.cache_limit) {
        DJ_HIP(hipStreamSynchronize(g.stream));
        DJ_HIP(hipFree(p));
        return;
    }
    g.cache[cls].push_back(p);
    g.cached_bytes += (int64_t)cls;
}

void ensure_workspace(int64_t floats) {
    if (g.no_alloc) {
        if (floats > kStaticWorkspaceFloats)
            fail("flush_ops_noalloc: the stream needs " + std::to_string(floats) + " floats of workspace, the static "
                 "scratch holds " + std::to_string(kStaticWorkspaceFloats) + " (use deepj_hip_flush_ops)");
        return;
    }
    if (floats <= g.workspace_floats) return;
    if (g.capturing) fail("deepj_hip: workspace would have to grow during graph capture; run the stream once first");
    DJ_HIP(hipStreamSynchronize(g.stream));
    if (g.workspace) DJ_HIP(hipFree(g.workspace));
    g.workspace = nullptr;
    g.workspace_floats = 0;
    int64_t want = std::max<int64_t>(floats, (int64_t)1 << 20);
    g.workspace = static_cast<float *>(device_memory((size_t)want * 4));
    g.workspace_floats = want;
}

bool graph_holds_pieces(const float *block) {
    return std::any_of(g.graphs.begin(), g.graphs.end(), [&](const auto &kv) { return kv.second.row_pieces == block; });
}

void ensure_scratch(const Scratch &need) {
    ensure_workspace(need.workspace);
    if (g.no_alloc || need.row_pieces <= g.row_pieces_floats) return;      // (the fixed array: products that it does not hold take another kernel)
    DJ_HIP(hipStreamSynchronize(g.stream));
    if (g.row_pieces && !graph_holds_pieces(g.row_pieces)) DJ_HIP(hipFree(g.row_pieces));
    g.row_pieces = nullptr;
    g.row_pieces_floats = 0;
    const int64_t want = std::max<int64_t>(need.row_pieces, (int64_t)1 << 20);
    g.row_pieces = static_cast<float *>(device_memory((size_t)want * 4));
    g.row_pieces_floats = want;
}

// ── stream interpreter ──────────────────────────────────────────────────────

struct Cursor {
    const int32_t *cmd;
    int32_t len;
    int32_t pos;
    bool dry;          // validate only
    Scratch need;      // collected in the dry pass
    int32_t skip = 0;  // words behind this op whose ops its launch has taken along
    int32_t done[kTransposes] = {};     // ops further on that have run already, in order: done[next_done] is the next one to pass
    int n_done = 0, next_done = 0;
    int32_t pieces_pos = -1;            // the op that finds its rows' pieces made, and where in their block; the dry pass knows by shapes
    int64_t pieces_at = 0;
};

const char *op_name(int op);

// An op's device scratch: collected in the dry pass, in a captured graph's run pass noted as what its launches hold (weights that
// the stream itself writes or prepares may take another kernel there than the dry pass saw, in whatever scratch there is)
void need_scratch(Cursor &c, int64_t workspace, int64_t pieces) {
    if (c.dry) {
        c.need.workspace = std::max(c.need.workspace, workspace);
        c.need.row_pieces = std::max(c.need.row_pieces, pieces);
    } else if (g.capture_into) {
        if (workspace > 0 || pieces > g.row_pieces_floats) g.capture_into->workspace = g.workspace;
        if (pieces > 0) g.capture_into->row_pieces = g.row_pieces;
    }
}

int stride_of(int op) {
    switch (op) {
        case DJ_OP_SQRT: case DJ_OP_NEG: case DJ_OP_EXP: case DJ_OP_LOG: case DJ_OP_TANH: case DJ_OP_SIGMOID:
        case DJ_OP_RELU: case DJ_OP_GELU:
            return 4;
        case DJ_OP_ADD: case DJ_OP_SUBTRACT: case DJ_OP_MULTIPLY: case DJ_OP_DIVIDE: case DJ_OP_RELU_BACKWARD:
        case DJ_OP_GELU_BACKWARD: case DJ_OP_MULTIPLY_SCALAR: case DJ_OP_ADD_SCALAR: case DJ_OP_DIVIDE_SCALAR:
        case DJ_OP_TRANSPOSE: case DJ_OP_SUM_ROWS: case DJ_OP_MEAN_ALONG_ROWS: case DJ_OP_VARIANCE_ALONG_ROWS:
        case DJ_OP_SUM_ALONG_ROWS: case DJ_OP_MAX_ALONG_ROWS: case DJ_OP_SOFTMAX_ROWS: case DJ_OP_POW:
        case DJ_OP_SUM_ABS: case DJ_OP_SUM_SCALAR:
            return 5;
        case DJ_OP_CLAMP: case DJ_OP_CROSS_ENTROPY_LOSS: case DJ_OP_CROSS_ENTROPY_GRADIENT:
        case DJ_OP_SOFTMAX_BACKWARD: case DJ_OP_ADD_ROW_VECTOR: case DJ_OP_ADD_BROADCAST_COLS:
        case DJ_OP_SUBTRACT_BROADCAST_COLS: case DJ_OP_DIVIDE_BROADCAST_COLS: case DJ_OP_MULTIPLY_BROADCAST_ROWS:
        case DJ_OP_MULTIPLY_BROADCAST_COLS:
            return 6;
        case DJ_OP_MATMUL: case DJ_OP_LAYERNORM_BACKWARD: case DJ_OP_SCATTER_ADD_ROWS:
        case DJ_OP_SCATTER_ADD_ROWS_ATOMIC:
            return 7;
        case DJ_OP_ADAMW_UPDATE: return 13;
        case DJ_OP_Q8_QUANTIZE: case DJ_OP_Q8_DEQUANTIZE: return 8;
        case DJ_OP_Q8_LINEAR: return 12;
        case DJ_OP_RMSNORM: return 6;
        case DJ_OP_SILU_MUL: return 5;
        case DJ_OP_EMBED_GATHER: return 8;
        case DJ_OP_ROPE_KV_STORE: return 13;
        case DJ_OP_ATTENTION: return 12;
        case DJ_OP_ARGMAX_ROWS: return 5;
        case DJ_OP_DECODE_ADVANCE: return 6;
        case DJ_OP_COPY: return 6;
        case DJ_OP_FILL: return 4;
        case DJ_OP_ROPE_ROWS: return 13;
        case DJ_OP_ATTENTION_KV: return 14;
        case DJ_OP_DECODE_NEXT: return 10;
        case DJ_OP_ATTN_DECODE: return 13;
        case DJ_OP_APPEND_ROWS: return 8;
        case DJ_OP_Q8_LINEAR_DYN: return 10;
        case DJ_OP_LAYERNORM: return 7;
        case DJ_OP_ATTN_DECODE_RECORDS: return 12;
        case DJ_OP_ADD_POSITIONS: return 7;
        case DJ_OP_STREAM_READ: return 4;
        case DJ_OP_NOP: return 2;
        case DJ_OP_Q8_PREPARE: return 5;
        case DJ_OP_Q8_LINEAR_ROPE: return 20;
        case DJ_OP_DECODE_SAMPLE: return 11;
        case DJ_OP_DECODE_ATTN: return 20;
        case DJ_OP_DECODE_FFN: return 16;
        case DJ_OP_DECODE_ROW: return 7;
        case DJ_OP_LATENT_DECODE: return 15;
        case DJ_OP_Q8_LINEAR_PAIR: return 10;
        default: return -1;
    }
}

float *buf(int32_t id, int64_t floats, int op, const char *role);

// Words 1 .. 5 (and gamma, beta behind them) of the DECODE_* ops: the row they start from.
DecodeRow decode_row(const int32_t *w, int op, int64_t d, bool norm, const int32_t *state, int64_t table_rows) {
    DecodeRow r{};
    const int64_t parts = w[3];
    if (parts < (state ? -1 : 0)) fail(std::string(op_name(op)) + ": bad part count");
    r.d = (int)d;
    r.x = buf(w[1], d, op, "x");
    if (parts == -1) { r.part = buf(w[2], table_rows * d, op, "part"); r.n_part = 1; r.at_state = state; r.table_rows = (int)table_rows; }
    else if (parts > 0) { r.part = buf(w[2], parts * d, op, "part"); r.n_part = (int)parts; }
    if (w[4] >= 0) r.bias = buf(w[4], d, op, "bias");
    r.out = buf(w[5], d, op, "out");
    if (r.out == r.x || r.out == r.part) fail(std::string(op_name(op)) + ": out needs a buffer of its own");
    if (norm) {
        r.gamma = buf(w[6], d, op, "gamma");
        if (w[7] >= 0) r.beta = buf(w[7], d, op, "beta");
    }
    return r;
}

void q8_weight(int32_t id, int64_t k, int64_t rows, int op, const char *role, const int8_t *&wq, const float *&scales) {
    wq = reinterpret_cast<const int8_t *>(buf(id, (q8_bytes((int)k, (int)rows) + 3) / 4, op, role));
    scales = reinterpret_cast<const float *>(wq + q8_scale_offset_bytes((int)k, (int)rows));
}

float bits_to_float(int32_t b) { float f; std::memcpy(&f, &b, 4); return f; }

// Pointer to buffer `id`, after checking that it exists and holds >= floats floats.
float *buf(int32_t id, int64_t floats, int op, const char *role) {
    auto it = g.live.find(id);
    if (it == g.live.end())
        fail(std::string(op_name(op)) + ": missing GPU buffer id=" + std::to_string(id) + " (" + role + ")");
    if (floats < 0 || floats > it->second.floats)
        fail(std::string(op_name(op)) + ": buffer id=" + std::to_string(id) + " (" + role + ") holds " +
             std::to_string(it->second.floats) + " floats, op needs " + std::to_string(floats));
    if (g.track) g.track->emplace_back(id, it->second.ptr);
    return static_cast<float *>(it->second.ptr);
}
float *buf_opt(int32_t id, int64_t floats, int op, const char *role) {
    return id < 0 ? nullptr : buf(id, floats, op, role);
}

void need_positive(int op, const char *what, int64_t v) {
    if (v < 0) fail(std::string(op_name(op)) + ": negative " + what + " " + std::to_string(v));
}

// An element-wise op as a link of a chain: ids and what is done with them.  op 0: no such op.
struct Link { int op = 0, kind = 0, words = 0; int32_t a = -1, b = -1, out = -1; int64_t n = 0, rows = 0, cols = 0; float s0 = 0.0f, s1 = 0.0f; };
Link chain_link(const int32_t *w) {
    Link l;
    auto set = [&](int op, int kind, int words, int32_t a, int32_t b, int32_t out, int64_t n) { l.op = op; l.kind = kind; l.words = words; l.a = a; l.b = b; l.out = out; l.n = n; };
    auto vec = [&](int op, int kind) { set(op, kind, 6, w[1], w[2], w[3], (int64_t)w[4] * w[5]); l.rows = w[4]; l.cols = w[5]; };
    switch (w[0]) {
        case DJ_OP_ADD: case DJ_OP_SUBTRACT: case DJ_OP_MULTIPLY: case DJ_OP_DIVIDE: case DJ_OP_RELU_BACKWARD: case DJ_OP_GELU_BACKWARD:
            set(w[0], 0, 5, w[1], w[2], w[3], w[4]); break;
        case DJ_OP_MULTIPLY_SCALAR: case DJ_OP_ADD_SCALAR: case DJ_OP_DIVIDE_SCALAR:
            set(w[0], 0, 5, w[1], -1, w[2], w[4]); l.s0 = bits_to_float(w[3]); break;
        case DJ_OP_CLAMP: set(w[0], 0, 6, w[1], -1, w[2], w[5]); l.s0 = bits_to_float(w[3]); l.s1 = bits_to_float(w[4]); break;
        case DJ_OP_ADD_ROW_VECTOR: vec(DJ_OP_ADD, 1); break;
        case DJ_OP_MULTIPLY_BROADCAST_ROWS: vec(DJ_OP_MULTIPLY, 1); break;
        case DJ_OP_ADD_BROADCAST_COLS: vec(DJ_OP_ADD, 2); break;
        case DJ_OP_SUBTRACT_BROADCAST_COLS: vec(DJ_OP_SUBTRACT, 2); break;
        case DJ_OP_DIVIDE_BROADCAST_COLS: vec(DJ_OP_DIVIDE, 2); break;
        case DJ_OP_MULTIPLY_BROADCAST_COLS: vec(DJ_OP_MULTIPLY, 2); break;
        default:
            if (chain_takes(w[0]) && stride_of(w[0]) == 4) set(w[0], 0, 4, w[1], -1, w[2], w[3]);
    }
    return l;
}

// The element-wise ops from here on that work on the same elements, as one launch (k_chain): one of a few between two products
// costs little more than a launch, and each of them reads what the one before it wrote.  A product between two of them that
// has nothing to do with those in front of it goes first.  False: too few.
//
// Every thread takes its elements through all the ops, so an op may read and write what others of them read and write at the
// same elements - but a vector is read by all threads, and must be none of the results.
void exec_one(Cursor &c);
bool exec_chain(Cursor &c) {
    Chain chain{};
    int32_t ext_id[kChainExt], vectors[kChainOps], outs[kChainOps];
    Link links[kChainOps];
    int operand[kChainOps][2];                    // >= 0: an external value, < 0: the result of op -1 - operand
    int n_vec = 0, count = 0;
    int32_t at = c.pos, end = c.pos, products[2], planned[2];
    int n_products = 0, n_planned = 0;
    int64_t cols = 0;
    auto among = [](const int32_t *ids, int n, int32_t id) { return std::find(ids, ids + n, id) != ids + n; };
    while (at < c.len && count < kChainOps && at + stride_of(c.cmd[at]) <= c.len) {
        const int32_t *w = c.cmd + at;
        if (w[0] == DJ_OP_MATMUL && count > 0) {
            if (n_planned == 2 || among(outs, count, w[1]) || among(outs, count, w[2]) || among(outs, count, w[3]) ||
                among(ext_id, chain.n_ext, w[3])) break;
            planned[n_planned++] = at;
            at += 7;
            continue;
        }
        const Link l = chain_link(w);
        if (!l.op || l.n <= 0 || l.n > 0x7fffffffLL || (count && l.n != chain.n)) break;
        if (l.kind) {
            if ((cols && l.cols != cols) || l.cols <= 0 || among(outs, count, l.b) || l.out == l.b) break;
        }
        if (among(vectors, n_vec, l.out)) break;
        int n_ext = chain.n_ext;
        auto find = [&](int32_t id, int kind, int &to) {
            if (kind == 0)
                for (int k = count; k-- > 0;)
                    if (outs[k] == id) { to = -1 - k; return true; }
            for (int j = 0; j < n_ext; j++)
                if (ext_id[j] == id && chain.ext[j].kind == kind) { to = j; return true; }
            if (n_ext == kChainExt) return false;
            ext_id[n_ext] = id;
            chain.ext[n_ext].kind = kind;
            to = n_ext++;
            return true;
        };
        int a, b;
        if (!find(l.a, 0, a)) break;
        b = a;
        if (l.b >= 0 && !find(l.b, l.kind, b)) break;
        chain.n_ext = n_ext;
        if (l.kind) { cols = l.cols; vectors[n_vec++] = l.b; }
        operand[count][0] = a; operand[count][1] = b;
        outs[count] = l.out;
        links[count++] = l;
        chain.n = l.n;
        at += l.words;
        end = at;
        while (n_products < n_planned) { products[n_products] = planned[n_products]; n_products++; }
    }
    // What a launch costs against what k_chain's own code does (interpreting, LDS, half the memory rate of a kernel that does one
    // thing), us together / one by one: 500 values, 2 ops 5.8 / 5.6 behind other kernels, 4 ops 5.4 / 10.2; 500 x 1024: 2 ops
    // 4.8 .. 5.3 / 4.9 .. 5.2, behind a product 5.7 / 9.4, 4 ops 7.1 / 10.2; 500 x 2752: 2 ops 7.2 .. 9.2 / 5.4 .. 6.3, 4 ops 12.7 / 12.4,
    // 5 behind products 16.5 / 27.6; 1024 x 7000: 2 ops 20 .. 27 / 18 .. 22, 4 ops 38 / 47; 2048 x 8192: 41 .. 52 / 38 .. 41, 91 / 106.
    if (count < (chain.n < (1 << 17) ? 3 : chain.n <= (1 << 20) ? 2 : 4)) return false;

    // A result takes the slot of an operand that nothing needs any more, or a free one.  A chain that would need a ninth is not
    // taken: its first op runs by itself, and the chain from the second on is looked at anew.
    int last_use[kChainExt + kChainOps], slot_of[kChainExt + kChainOps];       // values: the external ones, then the results
    auto value = [&](int x) { return x >= 0 ? x : kChainExt + (-1 - x); };
    for (int &u : last_use) u = -1;
    for (int k = 0; k < count; k++)
        for (int x : operand[k]) last_use[value(x)] = k;
    bool used[kChainSlots] = {};
    for (int j = 0; j < chain.n_ext; j++) { slot_of[j] = j; used[j] = true; }
    for (int k = 0; k < count; k++) {
        const int va = value(operand[k][0]), vb = value(operand[k][1]);
        for (int v : {va, vb})
            if (last_use[v] == k) used[slot_of[v]] = false;
        int dst = 0;
        while (dst < kChainSlots && used[dst]) dst++;
        if (dst == kChainSlots) return false;
        slot_of[kChainExt + k] = dst;
        used[dst] = last_use[kChainExt + k] > k;
        const Link &l = links[k];
        chain.ops[k] = {l.op, slot_of[va], slot_of[vb], dst, buf(l.out, l.n, l.op, "out"), l.s0, l.s1};
    }
    for (int j = 0; j < chain.n_ext; j++) {
        const int kind = chain.ext[j].kind;
        chain.ext[j].p = buf(ext_id[j], kind == 0 ? chain.n : kind == 1 ? cols : chain.n / cols, links[0].op, "in");
    }
    chain.n_ops = count;
    chain.cols = cols ? (int)cols : (int)chain.n;
    for (int i = 0; i < n_products; i++) {
        Cursor m{c.cmd, c.len, products[i], false, {}};
        exec_one(m);
    }
    launch_chain(g.stream, chain);
    c.skip = end - c.pos - stride_of(c.cmd[c.pos]);
    return true;
}

// A transpose and those further on that could as well run now, as one launch: a backward pass transposes weights and activations
// that were there before it.  One goes first where none of the ops in front of it writes what it reads, nor reads or writes what it
// writes.  One by one and together, us, with a small operation behind them: four of 64 x 64 15.3, 9.4; six of 512 x 512 20.2, 9.9;
// two of 1024 x 1024 9.8, 9.0, four 14.7, 10.7.  Larger ones are bound by memory and stay where they are.  False: it is the only one.
bool exec_transposes(Cursor &c) {
    constexpr int kAhead = 32;
    Transposes all;
    int32_t reads[2 * kAhead], writes[kAhead], at = c.pos, found[kTransposes];
    int n_reads = 0, n_writes = 0;
    auto among = [](const int32_t *ids, int n, int32_t id) { return std::find(ids, ids + n, id) != ids + n; };
    for (int i = 0; i < kAhead && all.count < kTransposes && at + stride_of(c.cmd[at]) <= c.len; i++) {
        const int32_t *w = c.cmd + at;
        int32_t a, b = -1, out;
        int64_t n = 0;                                      // of a transpose
        switch (w[0]) {
            case DJ_OP_TRANSPOSE: n = (int64_t)w[3] * w[4]; a = w[1]; out = w[2]; break;
            case DJ_OP_SUM_ROWS: case DJ_OP_SUM_ALONG_ROWS: case DJ_OP_MEAN_ALONG_ROWS: case DJ_OP_VARIANCE_ALONG_ROWS: case DJ_OP_MAX_ALONG_ROWS:
            case DJ_OP_SOFTMAX_ROWS: a = w[1]; out = w[2]; break;
            case DJ_OP_MATMUL: a = w[1]; b = w[2]; out = w[3]; break;
            default: {
                const Link l = stride_of(w[0]) < 4 ? Link{} : chain_link(w);
                if (!l.op) i = kAhead;                      // an op that this does not look into: nothing goes past it
                a = l.a; b = l.b; out = l.out;
            }
        }
        if (i == kAhead) break;
        if (n > 0 && n <= (1 << 20) && a != out && !among(writes, n_writes, a) && !among(writes, n_writes, out) && !among(reads, n_reads, out)) {
            found[all.count] = at;
            all.t[all.count++] = Transpose{buf(a, n, w[0], "in"), buf(out, n, w[0], "out"), w[3], w[4], 0, 0};
        } else if (i == 0) {
            return false;
        }
        reads[n_reads++] = a;
        if (b >= 0) reads[n_reads++] = b;
        writes[n_writes++] = out;
        at += stride_of(w[0]);
        if (at >= c.len) break;
    }
    if (all.count < 2) return false;
    c.next_done = 0;
    c.n_done = all.count - 1;
    std::copy(found + 1, found + all.count, c.done);
    launch_transposes(g.stream, all);
    return true;
}

void exec_one(Cursor &c) {
    const int32_t *w = c.cmd + c.pos;
    const int op = w[0];
    hipStream_t s = g.stream;
    const bool run = !c.dry;
    const Runtime::ChainSlot was = g.chain;
    if (run) g.chain.valid = false;
    // this op is the one a GemmChain's first launch prepared the activations of (x, gain, shape as it saw them)
    auto chained = [&](int32_t x_id, int32_t gamma_id, int flags, int64_t m, int64_t k) {
        return run && was.valid && !was.pieces && was.cmd == c.cmd && was.pos == c.pos && was.x_id == x_id && was.gamma_id == gamma_id && was.m == m &&
               was.k == k && (flags & DJ_LIN_RMSNORM) && !(flags & DJ_LIN_LAYERNORM);
    };
    // the same for the rows' pieces that a product leaves to k_gemm_q8_rows
    auto pieces_left = [&](int64_t m, int64_t k) {
        const int flags = w[7];
        return run && was.valid && was.pieces && was.cmd == c.cmd && was.pos == c.pos && was.x_id == w[1] && was.m == m && was.k == k &&
               (was.plain ? !(flags & (DJ_LIN_RMSNORM | DJ_LIN_LAYERNORM))
                          : (flags & (DJ_LIN_RMSNORM | DJ_LIN_LAYERNORM)) && was.gamma_id == w[8] && was.beta_id == (flags & DJ_LIN_LAYERNORM ? w[10] : -1));
    };
    if (run && op < DJ_OP_Q8_QUANTIZE && exec_chain(c)) return;
    switch (op) {
        case DJ_OP_ADD: case DJ_OP_SUBTRACT: case DJ_OP_MULTIPLY: case DJ_OP_DIVIDE: case DJ_OP_RELU_BACKWARD:
        case DJ_OP_GELU_BACKWARD: {
            int64_t n = w[4]; need_positive(op, "n", n);
            const float *a = buf(w[1], n, op, "a"), *b = buf(w[2], n, op, "b");
            float *o = buf(w[3], n, op, "out");
            if (run) launch_binary(s, op, a, b, o, n);
            break;
        }
        case DJ_OP_SQRT: case DJ_OP_NEG: case DJ_OP_EXP: case DJ_OP_LOG: case DJ_OP_TANH: case DJ_OP_SIGMOID:
        case DJ_OP_RELU: case DJ_OP_GELU: {
            int64_t n = w[3]; need_positive(op, "n", n);
            const float *a = buf(w[1], n, op, "in");
            float *o = buf(w[2], n, op, "out");
            if (run) launch_unary(s, op, a, o, n);
            break;
        }
        case DJ_OP_MULTIPLY_SCALAR: case DJ_OP_ADD_SCALAR: case DJ_OP_DIVIDE_SCALAR: case DJ_OP_POW: {
            int64_t n = w[4]; need_positive(op, "n", n);
            const float *a = buf(w[1], n, op, "in");
            float *o = buf(w[2], n, op, "out");
            if (run) launch_scalar(s, op, a, o, bits_to_float(w[3]), 0.0f, n);
            break;
        }
        case DJ_OP_CLAMP: {
            int64_t n = w[5]; need_positive(op, "n", n);
            const float *a = buf(w[1], n, op, "in");
            float *o = buf(w[2], n, op, "out");
            if (run) launch_scalar(s, op, a, o, bits_to_float(w[3]), bits_to_float(w[4]), n);
            break;
        }
        case DJ_OP_MATMUL: {
            int64_t m = w[4], n = w[5], k = w[6];
            need_positive(op, "m", m); need_positive(op, "n", n); need_positive(op, "k", k);
            const float *a = buf(w[1], m * k, op, "a"), *b = buf(w[2], k * n, op, "b");
            float *o = buf(w[3], m * n, op, "out");
            if (run) launch_matmul_f32(s, a, b, o, (int)m, (int)n, (int)k);
            break;
        }
        case DJ_OP_TRANSPOSE: {
            int64_t rows = w[3], cols = w[4]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            const float *a = buf(w[1], rows * cols, op, "in");
            float *o = buf(w[2], rows * cols, op, "out");
            if (run && c.next_done == c.n_done && exec_transposes(c)) break;
            if (run) launch_transpose(s, a, o, (int)rows, (int)cols);
            break;
        }
        case DJ_OP_ADD_ROW_VECTOR: case DJ_OP_MULTIPLY_BROADCAST_ROWS: case DJ_OP_ADD_BROADCAST_COLS:
        case DJ_OP_SUBTRACT_BROADCAST_COLS: case DJ_OP_DIVIDE_BROADCAST_COLS: case DJ_OP_MULTIPLY_BROADCAST_COLS: {
            int64_t rows = w[4], cols = w[5]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            bool rowvec = (op == DJ_OP_ADD_ROW_VECTOR || op == DJ_OP_MULTIPLY_BROADCAST_ROWS);
            const float *a = buf(w[1], rows * cols, op, "a");
            const float *v = buf(w[2], rowvec ? cols : rows, op, "vector");
            float *o = buf(w[3], rows * cols, op, "out");
            if (run) launch_broadcast(s, op, a, v, o, (int)rows, (int)cols);
            break;
        }
        case DJ_OP_SUM_ROWS: {
            int64_t rows = w[3], cols = w[4]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            const float *a = buf(w[1], rows * cols, op, "in");
            float *o = buf(w[2], cols, op, "out");
            if (run) launch_sum_rows(s, a, o, (int)rows, (int)cols);
            break;
        }
        case DJ_OP_SUM_ALONG_ROWS: case DJ_OP_MEAN_ALONG_ROWS: case DJ_OP_VARIANCE_ALONG_ROWS:
        case DJ_OP_MAX_ALONG_ROWS: case DJ_OP_SUM_ABS: {
            int64_t rows = w[3], cols = w[4]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            const float *a = buf(w[1], rows * cols, op, "in");
            float *o = buf(w[2], rows, op, "out");
            if (run) launch_row_reduce(s, op, a, o, (int)rows, (int)cols);
            break;
        }
        case DJ_OP_SUM_SCALAR: {
            int64_t rows = w[3], cols = w[4]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            const float *a = buf(w[1], rows * cols, op, "in");
            float *o = buf(w[2], 1, op, "out");
            if (run) launch_sum_scalar(s, a, o, rows * cols);
            break;
        }
        case DJ_OP_SOFTMAX_ROWS: {
            int64_t rows = w[3], cols = w[4]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            const float *a = buf(w[1], rows * cols, op, "in");
            float *o = buf(w[2], rows * cols, op, "out");
            if (run) launch_softmax_rows(s, a, o, (int)rows, (int)cols);
            break;
        }
        case DJ_OP_SOFTMAX_BACKWARD: {
            int64_t rows = w[4], cols = w[5]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            const float *gr = buf(w[1], rows * cols, op, "grad"), *sm = buf(w[2], rows * cols, op, "softmax");
            float *o = buf(w[3], rows * cols, op, "out");
            if (run) launch_softmax_backward(s, gr, sm, o, (int)rows, (int)cols);
            break;
        }
        case DJ_OP_LAYERNORM_BACKWARD: {
            int64_t rows = w[5], cols = w[6]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            const float *dx = buf(w[1], rows * cols, op, "dXHat"), *xh = buf(w[2], rows * cols, op, "xHat");
            const float *sd = buf(w[3], rows, op, "std");
            float *o = buf(w[4], rows * cols, op, "out");
            if (run) launch_layernorm_backward(s, dx, xh, sd, o, (int)rows, (int)cols);
            break;
        }
        case DJ_OP_ADAMW_UPDATE: {
            // an optimiser steps its parameters one behind the other: those that share no buffer go out together
            AdamTensors batch;
            int count = 0;
            auto shares = [&](const int32_t *v) {
                for (const int32_t *u = w; u < v; u += 13)
                    for (int i = 1; i <= 4; i++)
                        for (int j = 1; j <= 4; j++)
                            if (u[i] == v[j]) return true;
                return false;
            };
            const int32_t *v = w;
            do {
                int64_t n = v[12]; need_positive(op, "n", n);
                AdamTensor &t = batch.t[count++];
                t.w = buf(v[1], n, op, "w"); t.g = buf(v[2], n, op, "g");
                t.mt = buf(v[3], n, op, "mt"); t.vt = buf(v[4], n, op, "vt");
                t.n = n;
                t.lr = bits_to_float(v[5]); t.beta1 = bits_to_float(v[6]); t.beta2 = bits_to_float(v[7]); t.eps = bits_to_float(v[8]);
                t.wd = bits_to_float(v[9]); t.bc1 = bits_to_float(v[10]); t.bc2 = bits_to_float(v[11]);
                v += 13;
            } while (run && count < kAdamTensors && v + 13 <= c.cmd + c.len && v[0] == DJ_OP_ADAMW_UPDATE && !shares(v));
            if (run) {
                launch_adamw(s, batch, count);
                c.skip = (int32_t)(v - w) - 13;
            }
            break;
        }
        case DJ_OP_SCATTER_ADD_ROWS: case DJ_OP_SCATTER_ADD_ROWS_ATOMIC: {
            // Both opcodes accumulate atomically: the non-atomic variant is racy for
            // duplicate indices by construction (deepj_metal_jni.mm:559-577).
            int64_t trows = w[4], tcols = w[5], nidx = w[6];
            need_positive(op, "rows", trows); need_positive(op, "cols", tcols); need_positive(op, "indices", nidx);
            float *t = buf(w[1], trows * tcols, op, "target");
            const float *idx = buf(w[2], nidx, op, "indices");
            const float *gr = buf(w[3], nidx * tcols, op, "grad");
            if (run) launch_scatter_add(s, t, idx, gr, (int)trows, (int)tcols, (int)nidx);
            break;
        }
        case DJ_OP_CROSS_ENTROPY_LOSS: case DJ_OP_CROSS_ENTROPY_GRADIENT: {
            int64_t rows = w[4], cols = w[5]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            bool grad = op == DJ_OP_CROSS_ENTROPY_GRADIENT;
            const float *lg = buf(w[1], rows * cols, op, "logits"), *tg = buf(w[2], rows, op, "targets");
            float *o = buf(w[3], grad ? rows * cols : rows, op, "out");
            if (run) launch_cross_entropy(s, grad, lg, tg, o, (int)rows, (int)cols);
            break;
        }

        // ── fused inference opcodes ────────────────────────────────────────
        case DJ_OP_Q8_QUANTIZE: case DJ_OP_Q8_DEQUANTIZE: {
            int64_t k = w[3], n = w[4], off = w[5], step = w[6], total = w[7];
            if (k <= 0 || n <= 0 || total <= 0 || step <= 0 || off < 0) fail(std::string(op_name(op)) + ": bad shape");
            if (off + (n - 1) * step >= total) fail(std::string(op_name(op)) + ": rows fall outside the Q8 buffer");
            int64_t qfloats = (q8_bytes((int)k, (int)total) + 3) / 4;
            bool quant = op == DJ_OP_Q8_QUANTIZE;
            float *src = buf(w[1], quant ? k * n : qfloats, op, "src");
            float *dst = buf(w[2], quant ? qfloats : k * n, op, "dst");
            if (run) {
                forget_prepared(w[2]);
                if (quant) {
                    int8_t *q = reinterpret_cast<int8_t *>(dst);
                    float *sc = reinterpret_cast<float *>(q + q8_scale_offset_bytes((int)k, (int)total));
                    launch_q8_quantize(s, src, q, sc, (int)k, (int)n, (int)off, (int)step);
                } else {
                    const int8_t *q = reinterpret_cast<const int8_t *>(src);
                    const float *sc = reinterpret_cast<const float *>(q + q8_scale_offset_bytes((int)k, (int)total));
                    launch_q8_dequantize(s, q, sc, dst, (int)k, (int)n, (int)off, (int)step);
                }
            }
            break;
        }
        case DJ_OP_Q8_LINEAR: {
            int64_t m = w[4], k = w[5], n = w[6];
            int flags = w[7];
            if (m <= 0 || k <= 0 || n <= 0) fail("OP_Q8_LINEAR: bad shape");
            if (flags & ~127) fail("OP_Q8_LINEAR: unknown flag bits");
            const bool merge = flags & DJ_LIN_ATTN_MERGE;
            int64_t rec_hd = 0;
            if (merge) {
                // x holds decode-attention records [K / hd][kAttnRecordSplits][hd + 4]; hd travels in the gamma word
                rec_hd = w[8];
                if (flags & (DJ_LIN_RMSNORM | DJ_LIN_LAYERNORM | DJ_LIN_SWIGLU | DJ_LIN_GELU))
                    fail("OP_Q8_LINEAR: ATTN_MERGE cannot be combined with a norm prologue, SWIGLU or GELU");
                if (rec_hd != 32 && rec_hd != 64 && rec_hd != 128) fail("OP_Q8_LINEAR: ATTN_MERGE head dim must be 32, 64 or 128");
                if (m != 1 || k % rec_hd != 0) fail("OP_Q8_LINEAR: ATTN_MERGE needs M = 1 and K a multiple of the head dim");
                if (q8_linear_workspace_floats(1, (int)k, (int)n, 0) != 0 || k > 11 * 1024) fail("OP_Q8_LINEAR: ATTN_MERGE: K too large");
            }
            bool sw = flags & DJ_LIN_SWIGLU;
            bool ln = flags & DJ_LIN_LAYERNORM;
            if (sw && (flags & DJ_LIN_RESIDUAL)) fail("OP_Q8_LINEAR: SWIGLU cannot be combined with RESIDUAL");
            if (sw && (flags & (DJ_LIN_LAYERNORM | DJ_LIN_GELU))) fail("OP_Q8_LINEAR: SWIGLU cannot be combined with LAYERNORM or GELU");
            if (ln && (flags & DJ_LIN_RMSNORM)) fail("OP_Q8_LINEAR: RMSNORM and LAYERNORM are exclusive");
            int64_t rows = sw ? 2 * n : n;
            Q8Linear p;
            p.x = merge ? buf(w[1], (k / rec_hd) * kAttnRecordSplits * (rec_hd + 4), op, "attention records") : buf(w[1], m * k, op, "x");
            p.rec_hd = (int)rec_hd;
            const float *wq = buf(w[2], (q8_bytes((int)k, (int)rows) + 3) / 4, op, "weight");
            p.wq = reinterpret_cast<const int8_t *>(wq);
            p.scales = reinterpret_cast<const float *>(p.wq + q8_scale_offset_bytes((int)k, (int)rows));
            p.out = buf(w[3], m * n, op, "out");
            p.m = (int)m; p.k = (int)k; p.n = (int)n; p.flags = flags;
            p.gamma = (flags & (DJ_LIN_RMSNORM | DJ_LIN_LAYERNORM)) ? buf(w[8], k, op, "gamma") : nullptr;   // (ATTN_MERGE: w[8] = hd)
            p.beta = ln ? buf(w[10], k, op, "beta") : nullptr;
            p.bias = (flags & DJ_LIN_BIAS) ? buf(w[9], n, op, "bias") : nullptr;
            p.bias2 = ((flags & DJ_LIN_BIAS) && sw) ? buf(w[10], n, op, "bias2") : nullptr;
            p.residual = (flags & DJ_LIN_RESIDUAL) ? buf(w[11], m * n, op, "residual") : nullptr;
            // a workspace that may grow is sized for the kernel's fastest path; the fixed one for the smallest
            if (m > 1) {
                auto pit = g.prepared.find(w[2]);
                if (pit != g.prepared.end() && pit->second.k == k && pit->second.rows == rows && q8_copy_pays((int)m, (int)k))
                    p.prepared = buf(pit->second.id, q8_prepared_floats((int)k, (int)rows), op, "prepared weights");
                if (p.prepared && run && g.capture_into) {
                    const std::pair<int32_t, int32_t> pr(w[2], pit->second.id);
                    auto &own = g.capture_into->self_prepared;
                    if (std::find(own.begin(), own.end(), pr) == own.end()) g.capture_into->prepared.push_back(pr);
                }
            }
            int64_t ws = g.no_alloc ? q8_linear_workspace_floats((int)m, (int)k, (int)n, flags)
                                    : q8_linear_preferred_workspace_floats((int)m, (int)k, (int)n, flags, p.prepared != nullptr);
            bool unshared = false;
            const int64_t own_pieces = g.no_alloc ? 0 : q8_linear_pieces_floats((int)m, (int)k, (int)n, flags, p.prepared != nullptr, false, &unshared);
            // The op right behind this one multiplies this output as it is: where both are products for k_gemm_q8_rows, this one's
            // epilogue leaves that one's pieces behind its own, or in front of them where there is room.  Which products do so and where
            // their pieces lie hangs on shapes alone, so that a stream has the same bits whatever size the block has grown to.
            const int32_t *behind = c.pos + stride_of(op) + 12 <= c.len ? c.cmd + c.pos + stride_of(op) : nullptr;
            const auto prepared_as = [&](int32_t weight, int64_t wk, int64_t wrows) {
                auto it = g.prepared.find(weight);
                return it != g.prepared.end() && it->second.k == wk && it->second.rows == wrows && q8_copy_pays((int)m, (int)wk);
            };
            const auto rows_of = [](const int32_t *nw) { return (nw[7] & DJ_LIN_SWIGLU) ? 2 * (int64_t)nw[6] : (int64_t)nw[6]; };
            const int64_t behind_own = (own_pieces + 63) / 64 * 64;
            int64_t plain_pieces = 0;
            if (m > 1 && own_pieces > 0 && unshared && behind && behind[0] == DJ_OP_Q8_LINEAR && behind[1] == w[3] && behind[4] == m && behind[5] == n && behind[6] > 0 &&
                behind[6] < (1 << 30) && !(behind[7] & (DJ_LIN_RMSNORM | DJ_LIN_LAYERNORM | DJ_LIN_ATTN_MERGE)))
                plain_pieces = q8_linear_pieces_floats((int)m, (int)n, behind[6], behind[7], prepared_as(behind[2], n, rows_of(behind)), true);
            const bool may_chain = run && m > 1 && !g.no_alloc && !merge;
            const bool pieces_ready = may_chain && pieces_left(m, k);
            const int64_t pieces_at = pieces_ready ? was.pieces_at : !run && c.pieces_pos == c.pos ? c.pieces_at : 0;
            const int64_t next_at = plain_pieces <= 0 || pieces_at >= plain_pieces ? 0 : pieces_at + behind_own;
            if (plain_pieces > 0) { c.pieces_pos = c.pos + stride_of(op); c.pieces_at = next_at; }
            need_scratch(c, ws, plain_pieces > 0 ? std::max(pieces_at + behind_own, next_at + plain_pieces) : own_pieces > 0 ? pieces_at + own_pieces : 0);
            // One rule for the allocation-free entry point, whatever happens to fit its fixed array: the many-row
            // fp16 GEMM (whose operands live in a workspace sized by the shape) is never taken there.
            p.small_workspace_only = g.no_alloc;
            GemmChain chain;
            int32_t next_gamma_id = -1, next_beta_id = -1;
            const int32_t next_pos = c.pos + stride_of(op);
            if (may_chain) {
                chain.planes_ready = chained(w[1], w[8], flags, m, k);
                chain.pieces_ready = pieces_ready;
                if (plain_pieces > 0 && next_at + plain_pieces <= g.row_pieces_floats)      // (less only where the dry pass saw other prepared copies)
                    chain.next_pieces = reinterpret_cast<uint16_t *>(g.row_pieces + next_at);
                // the op right behind this one normalises this output (RMSNorm) and multiplies it on the fp16 GEMM: the
                // launch may leave that op's activations ready (it does when this one shares its tiles' K)
                if (next_pos < c.len && !sw && !chain.next_pieces) {
                    const int32_t *nw = c.cmd + next_pos;
                    const bool n_rope = nw[0] == DJ_OP_Q8_LINEAR_ROPE;
                    if ((nw[0] == DJ_OP_Q8_LINEAR || n_rope) && nw[1] == w[3] && nw[4] == m && nw[5] == n && (nw[7] & DJ_LIN_RMSNORM) &&
                        !(nw[7] & (DJ_LIN_LAYERNORM | DJ_LIN_ATTN_MERGE))) {
                        const int64_t n_rows = n_rope ? 3 * (int64_t)nw[6] : ((nw[7] & DJ_LIN_SWIGLU) ? 2 * (int64_t)nw[6] : (int64_t)nw[6]);
                        if (n_rows > 0 && n_rows < (1 << 30) && (n_rope ? q8_gemm_f16_rope_ok((int)m, nw[6], (int)n) : q8_gemm_f16_shape_ok((int)m, (int)n_rows, (int)n))) {
                            next_gamma_id = nw[8];
                            chain.next_gamma = buf(next_gamma_id, n, op, "the next op's gamma");
                        }
                    }
                    // ... or on the kernel that multiplies a batch of rows from the int8 weights
                    const int norms = DJ_LIN_RMSNORM | DJ_LIN_LAYERNORM;
                    if (!chain.next_gamma && g.row_pieces && next_pos + 12 <= c.len && nw[0] == DJ_OP_Q8_LINEAR && nw[1] == w[3] && nw[4] == m && nw[5] == n &&
                        nw[6] > 0 && nw[6] < (1 << 30) && (nw[7] & norms) && !(nw[7] & DJ_LIN_ATTN_MERGE)) {
                        const int64_t pieces = q8_linear_pieces_floats((int)m, (int)n, nw[6], nw[7], prepared_as(nw[2], n, rows_of(nw)));
                        if (pieces > 0 && pieces <= g.row_pieces_floats) {
                            next_gamma_id = nw[8];
                            chain.next_gamma = buf(next_gamma_id, n, op, "the next op's gamma");
                            if (nw[7] & DJ_LIN_LAYERNORM) { next_beta_id = nw[10]; chain.next_beta = buf(next_beta_id, n, op, "the next op's beta"); }
                            chain.next_pieces = reinterpret_cast<uint16_t *>(g.row_pieces);
                        }
                    }
                }
                p.chain = &chain;
            }
            if (run) launch_q8_linear(s, p, g.workspace, g.workspace_floats, g.row_pieces + pieces_at, g.row_pieces_floats - pieces_at);
            if (chain.left_planes || chain.left_pieces) {
                g.chain.pieces_at = chain.next_gamma ? 0 : next_at; g.chain.plain = chain.left_pieces && !chain.next_gamma;
                g.chain.cmd = c.cmd; g.chain.pos = next_pos; g.chain.x_id = w[3]; g.chain.gamma_id = next_gamma_id; g.chain.beta_id = next_beta_id;
                g.chain.m = m; g.chain.k = n; g.chain.pieces = chain.left_pieces; g.chain.valid = true;
            }
            break;
        }
        case DJ_OP_Q8_LINEAR_ROPE: {
            // [op, x, weight, qOut, M, K, d, flags, gamma, bias, beta, kCache, vCache, state, cos, sin, H, hd, maxSeq, layer]
            const int64_t m = w[4], k = w[5], d = w[6], H = w[16], hd = w[17], max_seq = w[18], layer = w[19];
            const int flags = w[7];
            if (m <= 1 || k <= 0 || d <= 0 || H <= 0 || hd <= 0 || (hd & 3) || H * hd != d || max_seq <= 0 || layer < 0)
                fail("OP_Q8_LINEAR_ROPE: bad shape");
            if (flags & ~(DJ_LIN_RMSNORM | DJ_LIN_LAYERNORM | DJ_LIN_BIAS)) fail("OP_Q8_LINEAR_ROPE: only a norm prologue and a bias go with it");
            const bool ln = flags & DJ_LIN_LAYERNORM;
            if (ln && (flags & DJ_LIN_RMSNORM)) fail("OP_Q8_LINEAR_ROPE: RMSNORM and LAYERNORM are exclusive");
            if (g.no_alloc || !q8_gemm_f16_rope_ok((int)m, (int)d, (int)k))
                fail("OP_Q8_LINEAR_ROPE: this shape does not run on the fp16 GEMM (deepj_hip_q8_linear_rope_ok); use Q8_LINEAR + ROPE_KV_STORE");
            const int64_t rows = 3 * d, per_layer = H * max_seq * hd;
            Q8Linear p;
            p.x = buf(w[1], m * k, op, "x");
            const float *wq = buf(w[2], (q8_bytes((int)k, (int)rows) + 3) / 4, op, "weight");
            p.wq = reinterpret_cast<const int8_t *>(wq);
            p.scales = reinterpret_cast<const float *>(p.wq + q8_scale_offset_bytes((int)k, (int)rows));
            p.out = nullptr;
            p.m = (int)m; p.k = (int)k; p.n = (int)rows; p.flags = flags;
            p.gamma = (flags & (DJ_LIN_RMSNORM | DJ_LIN_LAYERNORM)) ? buf(w[8], k, op, "gamma") : nullptr;
            p.bias = (flags & DJ_LIN_BIAS) ? buf(w[9], rows, op, "bias") : nullptr;
            p.beta = ln ? buf(w[10], k, op, "beta") : nullptr;
            p.bias2 = nullptr; p.residual = nullptr;
            p.rope.q = buf(w[3], m * d, op, "qOut");
            p.rope.k_cache = buf(w[11], (layer + 1) * per_layer, op, "kCache") + layer * per_layer;
            p.rope.v_cache = buf(w[12], (layer + 1) * per_layer, op, "vCache") + layer * per_layer;
            p.rope.state = reinterpret_cast<const int32_t *>(buf(w[13], 4, op, "state"));
            p.rope.cos_t = buf(w[14], max_seq * (hd / 2), op, "cos");
            p.rope.sin_t = buf(w[15], max_seq * (hd / 2), op, "sin");
            p.rope.hd = (int)hd; p.rope.d = (int)d; p.rope.max_seq = (int)max_seq;
            auto pit = g.prepared.find(w[2]);
            if (pit != g.prepared.end() && pit->second.k == k && pit->second.rows == rows)
                p.prepared = buf(pit->second.id, q8_prepared_floats((int)k, (int)rows), op, "prepared weights");
            if (p.prepared && run && g.capture_into) {
                const std::pair<int32_t, int32_t> pr(w[2], pit->second.id);
                auto &own = g.capture_into->self_prepared;
                if (std::find(own.begin(), own.end(), pr) == own.end()) g.capture_into->prepared.push_back(pr);
            }
            const int64_t ws = q8_linear_preferred_workspace_floats((int)m, (int)k, (int)rows, flags, p.prepared != nullptr);
            need_scratch(c, ws, 0);
            GemmChain chain;
            chain.planes_ready = chained(w[1], w[8], flags, m, k);
            p.chain = &chain;
            if (run) launch_q8_linear(s, p, g.workspace, g.workspace_floats, g.row_pieces, g.row_pieces_floats);
            break;
        }
        case DJ_OP_RMSNORM: {
            int64_t rows = w[4], cols = w[5]; need_positive(op, "rows", rows); need_positive(op, "cols", cols);
            const float *x = buf(w[1], rows * cols, op, "x"), *gm = buf(w[2], cols, op, "gamma");
            float *o = buf(w[3], rows * cols, op, "out");
            if (run) launch_rmsnorm(s, x, gm, o, (int)rows, (int)cols);
            break;
        }
        case DJ_OP_LAYERNORM: {
            // [op, x, gamma, beta, out, rows, cols]
            int64_t rows = w[5], cols = w[6]; need_positive(op, "rows", rows);
            if (cols <= 0) fail("OP_LAYERNORM: bad shape");
            const float *x = buf(w[1], rows * cols, op, "x"), *gm = buf(w[2], cols, op, "gamma");
            const float *bt = buf(w[3], cols, op, "beta");
            float *o = buf(w[4], rows * cols, op, "out");
            if (run) launch_layernorm(s, x, gm, bt, o, (int)rows, (int)cols);
            break;
        }
        case DJ_OP_ADD_POSITIONS: {
            // [op, x, table, state, rows, d, maxSeq]
            int64_t rows = w[4], d = w[5], max_seq = w[6]; need_positive(op, "rows", rows);
            if (d <= 0 || max_seq <= 0) fail("OP_ADD_POSITIONS: bad shape");
            float *x = buf(w[1], rows * d, op, "x");
            const float *tb = buf(w[2], max_seq * d, op, "table");
            const float *st = buf(w[3], 4, op, "state");
            if (run) launch_add_positions(s, x, tb, reinterpret_cast<const int32_t *>(st), (int)rows, (int)d, (int)max_seq);
            break;
        }
        case DJ_OP_SILU_MUL: {
            int64_t n = w[4]; need_positive(op, "n", n);
            const float *a = buf(w[1], n, op, "gate"), *b = buf(w[2], n, op, "up");
            float *o = buf(w[3], n, op, "out");
            if (run) launch_silu_mul(s, a, b, o, n);
            break;
        }
        case DJ_OP_EMBED_GATHER: {
            int64_t nids = w[4], d = w[5], vocab = w[6], ids_off = w[7];
            if (nids < 0 || d <= 0 || vocab <= 0 || ids_off < 0) fail("OP_EMBED_GATHER: bad shape");
            const float *t = buf(w[1], vocab * d, op, "table");
            const float *ids = buf(w[2], ids_off + nids, op, "ids");
            float *o = buf(w[3], nids * d, op, "out");
            if (run)
                launch_embed_gather(s, t, reinterpret_cast<const int32_t *>(ids) + ids_off, o, (int)nids, (int)d,
                                    (int)vocab);
            break;
        }
        case DJ_OP_ROPE_KV_STORE: {
            int64_t S = w[8], H = w[9], hd = w[10], max_seq = w[11], layer = w[12];
            if (S <= 0 || H <= 0 || hd <= 0 || (hd & 3) || max_seq <= 0 || layer < 0) fail("OP_ROPE_KV_STORE: bad shape");
            int64_t d = H * hd, per_layer = H * max_seq * hd;
            const float *qkv = buf(w[1], S * 3 * d, op, "qkv");
            float *q_out = buf(w[2], S * d, op, "qOut");
            float *kc = buf(w[3], (layer + 1) * per_layer, op, "kCache");
            float *vc = buf(w[4], (layer + 1) * per_layer, op, "vCache");
            const float *st = buf(w[5], 4, op, "state");
            const float *ct = buf(w[6], max_seq * (hd / 2), op, "cos"), *sn = buf(w[7], max_seq * (hd / 2), op, "sin");
            if (run)
                launch_rope_kv_store(s, qkv, q_out, kc + layer * per_layer, vc + layer * per_layer,
                                     reinterpret_cast<const int32_t *>(st), ct, sn, (int)S, (int)H, (int)hd,
                                     (int)max_seq);
            break;
        }
        case DJ_OP_ROPE_ROWS: {
            // [op, x, out, state, cos, sin, rows, H, hd, maxSeq, posFromRow, rowStride, liveExtra]
            int64_t rows = w[6], H = w[7], hd = w[8], max_seq = w[9], stride = w[11], live_extra = w[12];
            if (rows <= 0 || H <= 0 || hd <= 0 || (hd & 1) || max_seq <= 0) fail("OP_ROPE_ROWS: bad shape");
            if (w[10] && rows > max_seq) fail("OP_ROPE_ROWS: more rows than RoPE table positions");
            if (stride == 0) stride = H * hd;
            if (stride < H * hd || (stride & 1) || live_extra < -1) fail("OP_ROPE_ROWS: bad row stride or live-row count");
            const float *x = buf(w[1], (rows - 1) * stride + H * hd, op, "x");
            float *o = buf(w[2], (rows - 1) * stride + H * hd, op, "out");
            const float *st = buf(w[3], 4, op, "state");
            const float *ct = buf(w[4], max_seq * (hd / 2), op, "cos"), *sn = buf(w[5], max_seq * (hd / 2), op, "sin");
            if (run)
                launch_rope_rows(s, x, o, reinterpret_cast<const int32_t *>(st), ct, sn, (int)rows, (int)H, (int)hd,
                                 (int)max_seq, w[10], (int)stride, (int)live_extra);
            break;
        }
        case DJ_OP_ATTENTION: case DJ_OP_ATTENTION_KV: {
            // ATTENTION    [op, q, kCache, vCache, out, state, scratch, S, H, hd, maxSeq, layer]  head-major cache
            // ATTENTION_KV [op, q, k, v, out, state, scratch, S, H, hd, maxSeq, 0, tokStride, vOff]  k,v token-major rows
            int64_t S = w[7], H = w[8], hd = w[9], max_seq = w[10], layer = w[11];
            if (S <= 0 || H <= 0 || max_seq <= 0 || layer < 0) fail(std::string(op_name(op)) + ": bad shape");
            if (hd != 32 && hd != 64 && hd != 128) fail(std::string(op_name(op)) + ": head dim must be 32, 64 or 128");
            int64_t d = H * hd, per_layer = H * max_seq * hd;
            AttnArgs a;
            a.q = buf(w[1], S * d, op, "q");
            bool cache = op == DJ_OP_ATTENTION;
            if (!cache && layer != 0) fail("OP_ATTENTION_KV: layer must be 0");
            int64_t tok = d, voff = 0;
            if (!cache) {
                tok = w[12] == 0 ? d : w[12];
                voff = w[13];
                if (tok < d || (tok & 3) || voff < 0 || (voff & 3)) fail("OP_ATTENTION_KV: bad token stride or value offset");
            }
            const float *kc = cache ? buf(w[2], (layer + 1) * per_layer, op, "k") : buf(w[2], (max_seq - 1) * tok + d, op, "k");
            const float *vc = cache ? buf(w[3], (layer + 1) * per_layer, op, "v")
                                    : buf(w[3], voff + (max_seq - 1) * tok + d, op, "v") + voff;
            a.k = kc + layer * per_layer; a.v = vc + layer * per_layer;
            a.k_tok_stride = cache ? hd : tok;
            a.k_head_stride = cache ? max_seq * hd : hd;
            a.out = buf(w[4], S * d, op, "out");
            a.state = reinterpret_cast<const int32_t *>(buf(w[5], 4, op, "state"));
            int64_t sf = attention_scratch_floats((int)S, (int)H, (int)hd, (int)max_seq);
            a.scratch = sf > 0 ? buf(w[6], sf, op, "scratch") : nullptr;
            a.scratch_floats = sf;
            a.counters = g.attn_counters;
            a.s = (int)S; a.h = (int)H; a.hd = (int)hd; a.max_seq = (int)max_seq;
            if (run) launch_attention(s, a);
            break;
        }
        case DJ_OP_ARGMAX_ROWS: {
            int64_t rows = w[3], cols = w[4];
            if (rows <= 0 || cols <= 0) fail("OP_ARGMAX_ROWS: bad shape");
            const float *a = buf(w[1], rows * cols, op, "logits");
            float *o = buf(w[2], rows, op, "out");
            if (run) launch_argmax_rows(s, a, reinterpret_cast<int32_t *>(o), (int)rows, (int)cols);
            break;
        }
        case DJ_OP_DECODE_ADVANCE: {
            // [op, state, token, tokens, capacity, nPositions]
            int64_t cap = w[4]; need_positive(op, "capacity", cap);
            need_positive(op, "positions", w[5]);
            float *st = buf(w[1], 4, op, "state");
            const float *tk = buf(w[2], 1, op, "token");
            float *out = buf(w[3], std::max<int64_t>(cap, 1), op, "tokens");
            if (run)
                launch_decode_advance(s, reinterpret_cast<int32_t *>(st), reinterpret_cast<const int32_t *>(tk),
                                      reinterpret_cast<int32_t *>(out), (int)cap, w[5]);
            break;
        }
        case DJ_OP_DECODE_NEXT: case DJ_OP_DECODE_SAMPLE: {
            // [op, logits, state, tokens, capacity, table, x, vocab, d, nPos(, params)]
            int64_t cap = w[4], vocab = w[7], d = w[8];
            if (cap < 0 || vocab <= 0 || d <= 0 || w[9] < 0) fail(std::string(op_name(op)) + ": bad shape");
            const float *lg = buf(w[1], vocab, op, "logits");
            float *st = buf(w[2], 4, op, "state");
            float *tk = buf(w[3], std::max<int64_t>(cap, 1), op, "tokens");
            const float *tb = buf(w[5], vocab * d, op, "table");
            float *x = buf(w[6], d, op, "x");
            float *params = op == DJ_OP_DECODE_SAMPLE ? buf(w[10], 4, op, "params") : nullptr;
            if (run && params)
                launch_decode_sample(s, lg, reinterpret_cast<int32_t *>(st), reinterpret_cast<int32_t *>(tk), (int)cap, tb, x,
                                     (int)vocab, (int)d, w[9], reinterpret_cast<uint32_t *>(params));
            else if (run)
                launch_decode_next(s, lg, reinterpret_cast<int32_t *>(st), reinterpret_cast<int32_t *>(tk), (int)cap,
                                   tb, x, (int)vocab, (int)d, w[9]);
            break;
        }
        case DJ_OP_ATTN_DECODE: {
            // [op, qkv, kCache, vCache, out, state, scratch, cos, sin, H, hd, maxSeq, layer]
            int64_t H = w[9], hd = w[10], max_seq = w[11], layer = w[12];
            if (H <= 0 || max_seq <= 0 || layer < 0) fail("OP_ATTN_DECODE: bad shape");
            if (hd != 32 && hd != 64 && hd != 128) fail("OP_ATTN_DECODE: head dim must be 32, 64 or 128");
            int64_t d = H * hd, per_layer = H * max_seq * hd;
            const float *qkv = buf(w[1], 3 * d, op, "qkv");
            float *kc = buf(w[2], (layer + 1) * per_layer, op, "kCache");
            float *vc = buf(w[3], (layer + 1) * per_layer, op, "vCache");
            float *o = buf(w[4], d, op, "out");
            const float *st = buf(w[5], 4, op, "state");
            float *sc = buf(w[6], attn_decode_scratch_floats((int)H, (int)hd), op, "scratch");
            const float *ct = buf(w[7], max_seq * (hd / 2), op, "cos"), *sn = buf(w[8], max_seq * (hd / 2), op, "sin");
            if (run)
                launch_attn_decode(s, qkv, kc + layer * per_layer, vc + layer * per_layer, o,
                                   reinterpret_cast<const int32_t *>(st), sc, ct, sn, (int)H, (int)hd, (int)max_seq,
                                   g.attn_counters);
            break;
        }
        case DJ_OP_ATTN_DECODE_RECORDS: {
            // [op, qkv, kCache, vCache, records, state, cos, sin, H, hd, maxSeq, layer]
            int64_t H = w[8], hd = w[9], max_seq = w[10], layer = w[11];
            if (H <= 0 || max_seq <= 0 || layer < 0) fail("OP_ATTN_DECODE_RECORDS: bad shape");
            if (hd != 32 && hd != 64 && hd != 128) fail("OP_ATTN_DECODE_RECORDS: head dim must be 32, 64 or 128");
            if (H > 65535) fail("OP_ATTN_DECODE_RECORDS: too many heads");
            int64_t d = H * hd, per_layer = H * max_seq * hd;
            const float *qkv = buf(w[1], 3 * d, op, "qkv");
            float *kc = buf(w[2], (layer + 1) * per_layer, op, "kCache");
            float *vc = buf(w[3], (layer + 1) * per_layer, op, "vCache");
            float *rec = buf(w[4], H * kAttnRecordSplits * (hd + 4), op, "records");
            const float *st = buf(w[5], 4, op, "state");
            const float *ct = buf(w[6], max_seq * (hd / 2), op, "cos"), *sn = buf(w[7], max_seq * (hd / 2), op, "sin");
            if (run)
                launch_attn_decode_records(s, qkv, kc + layer * per_layer, vc + layer * per_layer, rec,
                                           reinterpret_cast<const int32_t *>(st), ct, sn, (int)H, (int)hd, (int)max_seq);
            break;
        }
        case DJ_OP_DECODE_ATTN: {
            const int64_t d = w[8], hd = w[17], max_seq = w[18], layer = w[19];
            if (max_seq <= 0 || layer < 0 || !decode_block_ok((int)d, (int)hd, 1)) fail("OP_DECODE_ATTN: bad shape");
            const int64_t H = d / hd, per_layer = max_seq * d;
            DecodeAttn a;
            const int32_t *st = reinterpret_cast<const int32_t *>(buf(w[13], 4, op, "state"));
            a.in = decode_row(w, op, d, true, st, max_seq);
            q8_weight(w[9], d, 3 * d, op, "wqkv", a.wqkv, a.s_qkv);
            q8_weight(w[10], d, d, op, "wo", a.wo, a.s_wo);
            a.k_cache = buf(w[11], (layer + 1) * per_layer, op, "kCache") + layer * per_layer;
            a.v_cache = buf(w[12], (layer + 1) * per_layer, op, "vCache") + layer * per_layer;
            a.state = st;
            a.cos_t = buf(w[14], max_seq * (hd / 2), op, "cos"); a.sin_t = buf(w[15], max_seq * (hd / 2), op, "sin");
            a.part = buf(w[16], H * d, op, "partOut");
            a.hd = (int)hd; a.max_seq = (int)max_seq;
            a.scale = (float)(1.0 / std::sqrt((double)hd));
            if (a.part == a.in.part || a.part == a.in.x || a.part == a.in.out) fail("OP_DECODE_ATTN: partOut needs a buffer of its own");
            if (run) launch_decode_attn(s, a);
            break;
        }
        case DJ_OP_DECODE_FFN: {
            const int64_t d = w[8], dff = w[14];
            const int flags = w[15];
            if (dff <= 0 || !decode_block_ok((int)d, 32, (int)std::min<int64_t>(dff, 1 << 30))) fail("OP_DECODE_FFN: bad shape");
            if (flags != DJ_LIN_SWIGLU && flags != DJ_LIN_GELU) fail("OP_DECODE_FFN: flags must be SWIGLU or GELU");
            DecodeFfn a;
            a.in = decode_row(w, op, d, true, nullptr, 0);
            a.swiglu = flags == DJ_LIN_SWIGLU;
            q8_weight(w[9], d, a.swiglu ? 2 * dff : dff, op, "wgu", a.wgu, a.s_gu);
            a.bg = w[10] >= 0 ? buf(w[10], dff, op, "bg") : nullptr;
            a.bu = w[11] >= 0 && a.swiglu ? buf(w[11], dff, op, "bu") : nullptr;
            q8_weight(w[12], dff, d, op, "wd", a.wd, a.s_d);
            a.part = buf(w[13], decode_ffn_parts((int)dff) * d, op, "partOut");
            a.dff = (int)dff;
            if (a.part == a.in.part || a.part == a.in.x || a.part == a.in.out) fail("OP_DECODE_FFN: partOut needs a buffer of its own");
            if (run) launch_decode_ffn(s, a);
            break;
        }
        case DJ_OP_DECODE_ROW: {
            const int64_t d = w[6];
            if (d <= 0) fail("OP_DECODE_ROW: bad shape");
            const DecodeRow r = decode_row(w, op, d, false, nullptr, 0);
            if (run) launch_decode_row(s, r);
            break;
        }
        case DJ_OP_LATENT_DECODE: {
            // [op, q, ckv, latent, wukv, state, cos, sin, records, out, H, hd, rank, maxSeq, layer]
            const int64_t H = w[10], hd = w[11], rank = w[12], max_seq = w[13], layer = w[14];
            const int splits = latent_decode_splits((int)H, (int)hd, (int)rank, (int)max_seq);
            if (!splits || layer < 0) fail("OP_LATENT_DECODE: bad shape");
            const int64_t d = H * hd, per_layer = max_seq * rank;
            LatentDecode a{};
            a.q = buf(w[1], d, op, "q");
            a.ckv = buf(w[2], rank, op, "ckv");
            a.latent = buf(w[3], (layer + 1) * per_layer, op, "latent") + layer * per_layer;
            q8_weight(w[4], rank, 2 * d, op, "wukv", a.wq, a.scales);
            a.state = reinterpret_cast<const int32_t *>(buf(w[5], 4, op, "state"));
            a.cos_t = buf(w[6], max_seq * (hd / 2), op, "cos"); a.sin_t = buf(w[7], max_seq * (hd / 2), op, "sin");
            buf(w[8], H * splits * (hd + 4), op, "records");       // (what the launches leave each other is larger)
            a.out = buf(w[9], d, op, "out");
            a.heads = (int)H; a.hd = (int)hd; a.rank = (int)rank; a.max_seq = (int)max_seq;
            // ... and goes to the block that stays for the graphs captured over it, where a graph of the workspace ends with a larger one
            need_scratch(c, 0, latent_decode_scratch_floats((int)H, (int)hd, (int)rank, (int)max_seq));
            a.records = g.row_pieces;
            if (run) launch_latent_decode(s, a);
            break;
        }
        case DJ_OP_Q8_LINEAR_PAIR: {
            // [op, x, gamma, K, weightA, outA, nA, weightB, outB, nB]
            const int64_t k = w[3];
            if (k > (1 << 20) || !q8_linear_pair_ok((int)k) || w[6] <= 0 || w[9] <= 0) fail("OP_Q8_LINEAR_PAIR: bad shape");
            Q8LinearPair p{};
            p.x = buf(w[1], k, op, "x"); p.gamma = buf(w[2], k, op, "gamma"); p.k = (int)k;
            for (int i = 0; i < 2; i++) {
                p.n[i] = w[6 + 3 * i];
                q8_weight(w[4 + 3 * i], k, p.n[i], op, "weight", p.wq[i], p.scales[i]);
                p.out[i] = buf(w[5 + 3 * i], p.n[i], op, "out");
            }
            if (p.out[0] == p.out[1] || p.out[0] == p.x || p.out[1] == p.x) fail("OP_Q8_LINEAR_PAIR: every out needs a buffer of its own");
            if (run) launch_q8_linear_pair(s, p);
            break;
        }
        case DJ_OP_APPEND_ROWS: {
            // [op, src, dst, state, rows, rowFloats, maxRows, dstOff]: dst[dstOff + (state[0]+i)*rowFloats ..] = src row i
            int64_t rows = w[4], rf = w[5], max_rows = w[6], off = w[7];
            if (rows <= 0 || rf <= 0 || max_rows <= 0 || off < 0) fail("OP_APPEND_ROWS: bad shape");
            const float *src = buf(w[1], rows * rf, op, "src");
            float *dst = buf(w[2], off + max_rows * rf, op, "dst");
            const float *st = buf(w[3], 4, op, "state");
            if (run) launch_append_rows(s, src, dst + off, reinterpret_cast<const int32_t *>(st), (int)rows, (int)rf, (int)max_rows);
            break;
        }
        case DJ_OP_Q8_LINEAR_DYN: {
            // [op, x, w, out, Mmax, K, N, state, extraRows, xOff]: rows [0, min(Mmax, state[0]+extraRows)) of x + xOff
            int64_t m = w[4], k = w[5], n = w[6], extra = w[8], xoff = w[9];
            if (m <= 0 || k <= 0 || n <= 0 || extra < 0 || xoff < 0) fail("OP_Q8_LINEAR_DYN: bad shape");
            Q8Linear p;
            p.x = buf(w[1], xoff + m * k, op, "x") + xoff;
            const float *wq = buf(w[2], (q8_bytes((int)k, (int)n) + 3) / 4, op, "weight");
            p.wq = reinterpret_cast<const int8_t *>(wq);
            p.scales = reinterpret_cast<const float *>(p.wq + q8_scale_offset_bytes((int)k, (int)n));
            p.out = buf(w[3], m * n, op, "out");
            p.m = (int)m; p.k = (int)k; p.n = (int)n; p.flags = 0;
            p.gamma = p.bias = p.bias2 = p.residual = nullptr;
            p.m_dev = reinterpret_cast<const int32_t *>(buf(w[7], 4, op, "state"));
            p.m_extra = (int)extra;
            if (run) launch_q8_linear(s, p, g.workspace, g.workspace_floats, g.row_pieces, g.row_pieces_floats);
            break;
        }
        case DJ_OP_COPY: {
            int64_t n = w[3], so = w[4], dof = w[5];
            if (n < 0 || so < 0 || dof < 0) fail("OP_COPY: bad range");
            const float *a = buf(w[1], so + n, op, "src");
            float *o = buf(w[2], dof + n, op, "dst");
            if (run) { forget_prepared(w[2]); launch_copy(s, a + so, o + dof, n); }
            break;
        }
        case DJ_OP_Q8_PREPARE: {
            // [op, weight, prepared, K, rows]: writes the weights in the many-row GEMM's layout and lets that buffer
            // stand for them in later Q8_LINEARs with more than one row, until either buffer is released or written
            int64_t k = w[3], rows = w[4]; need_positive(op, "K", k); need_positive(op, "rows", rows);
            if (w[1] == w[2]) fail("OP_Q8_PREPARE: the prepared copy needs a buffer of its own");
            const float *wq = buf(w[1], (q8_bytes((int)k, (int)rows) + 3) / 4, op, "weight");
            float *prep = buf(w[2], q8_prepared_floats((int)k, (int)rows), op, "prepared");
            if (run) {
                const int8_t *q = reinterpret_cast<const int8_t *>(wq);
                launch_q8_prepare(s, q, reinterpret_cast<const float *>(q + q8_scale_offset_bytes((int)k, (int)rows)), prep, (int)k, (int)rows);
                forget_prepared(w[2]);
                g.prepared[w[1]] = Runtime::Prepared{w[2], (int)k, (int)rows};
                if (g.capture_into) g.capture_into->self_prepared.emplace_back(w[1], w[2]);   // every replay rewrites the copy
            }
            break;
        }
        case DJ_OP_STREAM_READ: {
            // [op, src, sink, n]: reads n floats of src and keeps nothing (sink holds >= 1 float)
            int64_t n = w[3]; need_positive(op, "n", n);
            const float *a = buf(w[1], n, op, "src");
            float *o = buf(w[2], 1, op, "sink");
            if (run) launch_stream_read(s, a, o, n);
            break;
        }
        case DJ_OP_NOP: {
            // [op, grid]: an empty kernel of `grid` workgroups of 256 threads
            if (w[1] < 1 || w[1] > 65535) fail("OP_NOP: grid must be 1..65535");
            if (run) launch_nop(s, w[1]);
            break;
        }
        case DJ_OP_FILL: {
            int64_t n = w[3]; need_positive(op, "n", n);
            float *o = buf(w[1], n, op, "dst");
            if (run) { forget_prepared(w[1]); launch_fill(s, reinterpret_cast<uint32_t *>(o), (uint32_t)w[2], n); }
            break;
        }
        default:
            fail("Unknown op code in graph: " + std::to_string(op));
    }
}

void walk(const int32_t *cmd, int32_t len, bool dry, Scratch *need) {
    Cursor c{cmd, len, 0, dry, 0};
    g.chain.valid = false;          // nothing carries over from an earlier stream (or from one that ended in an error)
    while (c.pos < len) {
        int op = cmd[c.pos];
        int stride = stride_of(op);
        if (stride < 0) fail("Unknown op code in graph: " + std::to_string(op));
        if (c.pos + stride > len)
            fail(std::string(op_name(op)) + ": command stream truncated at word " + std::to_string(c.pos));
        if (c.next_done < c.n_done && c.done[c.next_done] == c.pos) c.next_done++;
        else exec_one(c);
        c.pos += stride + c.skip;
        c.skip = 0;
    }
    if (need) *need = c.need;
}

void run_stream(const int32_t *cmd, int32_t len) {
    if (len < 0) fail("flushOps: negative stream length");
    if (len > 0 && !cmd) fail("flushOps: null command stream");
    Scratch need;
    walk(cmd, len, true, &need);      // validate everything first
    launch_uploads();
    ensure_scratch(need);
    walk(cmd, len, false, nullptr);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) fail(std::string("kernel launch failed: ") + hipGetErrorString(e));
}

const char *op_name(int op) {
    static const char *names[] = {
        "?", "OP_ADD", "OP_SUBTRACT", "OP_MULTIPLY", "OP_DIVIDE", "OP_MATMUL", "OP_MULTIPLY_SCALAR", "OP_SQRT",
        "OP_NEG", "OP_EXP", "OP_LOG", "OP_TANH", "OP_SIGMOID", "OP_RELU", "OP_RELU_BACKWARD", "OP_GELU",
        "OP_GELU_BACKWARD", "OP_SOFTMAX_ROWS", "OP_SOFTMAX_BACKWARD", "OP_LAYERNORM_BACKWARD", "OP_ADAMW_UPDATE",
        "OP_ADD_SCALAR", "OP_DIVIDE_SCALAR", "OP_TRANSPOSE", "OP_ADD_ROW_VECTOR", "OP_ADD_BROADCAST_COLS",
        "OP_SUBTRACT_BROADCAST_COLS", "OP_DIVIDE_BROADCAST_COLS", "OP_MULTIPLY_BROADCAST_ROWS", "OP_SUM_ROWS",
        "OP_MEAN_ALONG_ROWS", "OP_VARIANCE_ALONG_ROWS", "OP_MULTIPLY_BROADCAST_COLS", "OP_SUM_ALONG_ROWS",
        "OP_MAX_ALONG_ROWS", "OP_CLAMP", "OP_POW", "OP_SCATTER_ADD_ROWS", "OP_SUM_ABS", "OP_CROSS_ENTROPY_LOSS",
        "OP_CROSS_ENTROPY_GRADIENT", "OP_SUM_SCALAR", "OP_SCATTER_ADD_ROWS_ATOMIC"};
    if (op >= 1 && op <= 42) return names[op];
    switch (op) {
        case DJ_OP_Q8_QUANTIZE: return "OP_Q8_QUANTIZE";
        case DJ_OP_Q8_DEQUANTIZE: return "OP_Q8_DEQUANTIZE";
        case DJ_OP_Q8_LINEAR: return "OP_Q8_LINEAR";
        case DJ_OP_RMSNORM: return "OP_RMSNORM";
        case DJ_OP_LAYERNORM: return "OP_LAYERNORM";
        case DJ_OP_ATTN_DECODE_RECORDS: return "OP_ATTN_DECODE_RECORDS";
        case DJ_OP_ADD_POSITIONS: return "OP_ADD_POSITIONS";
        case DJ_OP_SILU_MUL: return "OP_SILU_MUL";
        case DJ_OP_EMBED_GATHER: return "OP_EMBED_GATHER";
        case DJ_OP_ROPE_KV_STORE: return "OP_ROPE_KV_STORE";
        case DJ_OP_Q8_LINEAR_ROPE: return "OP_Q8_LINEAR_ROPE";
        case DJ_OP_ATTENTION: return "OP_ATTENTION";
        case DJ_OP_ARGMAX_ROWS: return "OP_ARGMAX_ROWS";
        case DJ_OP_DECODE_ADVANCE: return "OP_DECODE_ADVANCE";
        case DJ_OP_COPY: return "OP_COPY";
        case DJ_OP_FILL: return "OP_FILL";
        case DJ_OP_ROPE_ROWS: return "OP_ROPE_ROWS";
        case DJ_OP_ATTENTION_KV: return "OP_ATTENTION_KV";
        case DJ_OP_DECODE_NEXT: return "OP_DECODE_NEXT";
        case DJ_OP_DECODE_SAMPLE: return "OP_DECODE_SAMPLE";
        case DJ_OP_DECODE_ATTN: return "OP_DECODE_ATTN";
        case DJ_OP_DECODE_FFN: return "OP_DECODE_FFN";
        case DJ_OP_DECODE_ROW: return "OP_DECODE_ROW";
        case DJ_OP_LATENT_DECODE: return "OP_LATENT_DECODE";
        case DJ_OP_Q8_LINEAR_PAIR: return "OP_Q8_LINEAR_PAIR";
        case DJ_OP_ATTN_DECODE: return "OP_ATTN_DECODE";
        case DJ_OP_APPEND_ROWS: return "OP_APPEND_ROWS";
        case DJ_OP_Q8_LINEAR_DYN: return "OP_Q8_LINEAR_DYN";
        case DJ_OP_STREAM_READ: return "OP_STREAM_READ";
        case DJ_OP_NOP: return "OP_NOP";
        case DJ_OP_Q8_PREPARE: return "OP_Q8_PREPARE";
        default: return "OP_?";
    }
}

template <class F> int guarded(F &&f) {
    try {
        f();
        g_error.clear();
        return 0;
    } catch (const std::exception &ex) {
        g_error = ex.what();
        return 1;
    } catch (...) {
        g_error = "deepj_hip: unknown native error";
        return 1;
    }
}

}  // namespace
}  // namespace dj

using namespace dj;

extern "C" {

int deepj_hip_init(int32_t device) {
    return guarded([&] { ensure_init(device); });
}

int deepj_hip_alloc_buffers(const int32_t *ids, const int32_t *sizes, int32_t count) {
    return guarded([&] {
        ensure_init();
        if (count < 0) fail("allocBuffers: negative count");
        if (count > 0 && (!ids || !sizes)) fail("allocBuffers: null array");
        for (int i = 0; i < count; i++) {
            if (g.live.count(ids[i])) continue;          // existing id: silent no-op
            if (sizes[i] < 0) fail("allocBuffers: negative size for id " + std::to_string(ids[i]));
            size_t bytes = (size_t)sizes[i] * 4;
            size_t cls = size_class(bytes);
            Buffer b;
            b.ptr = pool_alloc(cls);
            b.capacity = cls;
            b.floats = sizes[i];
            b.made = ++g.made;
            g.live.emplace(ids[i], b);
            g.live_bytes += (int64_t)cls;
        }
    });
}

int deepj_hip_upload(int32_t id, const float *src, int64_t n) {
    return guarded([&] {
        ensure_init();
        auto it = g.live.find(id);
        if (it == g.live.end()) fail("Buffer not found for upload");
        if (n < 0 || n > it->second.floats)
            fail("uploadBuffer: " + std::to_string(n) + " floats do not fit buffer id=" + std::to_string(id) + " of " +
                 std::to_string(it->second.floats));
        if (n == 0) return;
        if (!src) fail("uploadBuffer: null source");
        forget_prepared(id);
        stage_upload(static_cast<float *>(it->second.ptr), src, n);      // the caller's array is only borrowed
    });
}

int deepj_hip_download(int32_t id, float *dst, int64_t n) {
    return guarded([&] {
        ensure_init();
        auto it = g.live.find(id);
        if (it == g.live.end()) fail("Buffer not found for download");
        if (n < 0 || n > it->second.floats)
            fail("downloadBuffer: " + std::to_string(n) + " floats exceed buffer id=" + std::to_string(id) + " of " +
                 std::to_string(it->second.floats));
        if (n > 0 && !dst) fail("downloadBuffer: null destination");
        const float *src = static_cast<const float *>(it->second.ptr);
        if (n == 0 || staged_for(src, n)) launch_uploads();      // (others can wait for the next flush)
        if (n > 0) download(src, dst, n);
        else DJ_HIP(hipStreamSynchronize(g.stream));
    });
}

int deepj_hip_release(const int32_t *ids, int32_t count) {
    return guarded([&] {
        if (!g.ready) return;
        if (count > 0 && !ids) fail("releaseBuffers: null array");
        launch_uploads();                                // a released block goes to the next buffer of its size
        for (int i = 0; i < count; i++) {
            auto it = g.live.find(ids[i]);
            if (it == g.live.end()) continue;            // unknown id: silent no-op
            g.live_bytes -= (int64_t)it->second.capacity;
            pool_free(it->second.ptr, it->second.capacity);
            g.live.erase(it);
            g.releases++;
            forget_prepared(ids[i]);
        }
    });
}

int deepj_hip_flush_ops(const int32_t *cmd, int32_t len) {
    return guarded([&] {
        ensure_init();
        run_stream(cmd, len);
    });
}

// The same interpreter over the static scratch array instead of the runtime's own (growable) workspace and
// counters: no hipMalloc / hipFree on this path.  The counters are cleared by a fill kernel first (the array keeps
// whatever the last call left); calls that overlap on one GPU would share the array and race.
int deepj_hip_flush_ops_noalloc(const int32_t *cmd, int32_t len) {
    return guarded([&] {
        if (!g.ready)
            fail("flush_ops_noalloc: the runtime is not initialised (initialisation allocates: call deepj_hip_init first)");
        struct Scope {
            float *ws = g.workspace, *pieces = g.row_pieces; int64_t wsf = g.workspace_floats, pf = g.row_pieces_floats; unsigned *ctr = g.attn_counters;
            Scope() {
                g.no_alloc = true;
                g.attn_counters = reinterpret_cast<unsigned *>(g.static_scratch);
                g.workspace = g.row_pieces = reinterpret_cast<float *>(g.static_scratch + kStaticCounterBytes);      // (no op uses both)
                g.workspace_floats = g.row_pieces_floats = kStaticWorkspaceFloats;
            }
            ~Scope() { g.no_alloc = false; g.workspace = ws; g.workspace_floats = wsf; g.row_pieces = pieces; g.row_pieces_floats = pf; g.attn_counters = ctr; }
        } scope;
        if (len < 0) fail("flushOps: negative stream length");
        if (len > 0 && !cmd) fail("flushOps: null command stream");
        Scratch need;
        walk(cmd, len, true, &need);
        launch_uploads();
        ensure_scratch(need);           // only checks the need against the static size here
        launch_fill(g.stream, reinterpret_cast<uint32_t *>(g.attn_counters), 0u, kAttnCounterHeads);
        walk(cmd, len, false, nullptr);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) fail(std::string("kernel launch failed: ") + hipGetErrorString(e));
    });
}

const char *deepj_hip_last_error(void) { return g_error.c_str(); }

int deepj_hip_synchronize(void) {
    return guarded([&] {
        if (!g.ready) return;
        launch_uploads();
        DJ_HIP(hipStreamSynchronize(g.stream));
    });
}

int deepj_hip_trim(void) {
    return guarded([&] {
        if (!g.ready) return;
        launch_uploads();
        DJ_HIP(hipStreamSynchronize(g.stream));
        host_trim();
        for (auto &kv : g.cache) {
            for (void *p : kv.second) DJ_HIP(hipFree(p));
            kv.second.clear();
        }
        g.cached_bytes = 0;
    });
}

int deepj_hip_shutdown(void) {
    return guarded([&] {
        if (!g.ready) return;
        DJ_HIP(hipStreamSynchronize(g.stream));
        for (auto &kv : g.graphs) {
            if (kv.second.exec) (void)hipGraphExecDestroy(kv.second.exec);
            if (kv.second.graph) (void)hipGraphDestroy(kv.second.graph);
        }
        std::vector<float *> blocks{g.row_pieces};
        for (auto &kv : g.graphs)
            if (std::find(blocks.begin(), blocks.end(), kv.second.row_pieces) == blocks.end()) blocks.push_back(kv.second.row_pieces);
        for (float *b : blocks)
            if (b) (void)hipFree(b);
        g.row_pieces = nullptr; g.row_pieces_floats = 0;
        g.graphs.clear();
        for (auto &kv : g.plans)
            for (const TokenPlan::Block &b : kv.second.blocks) (void)hipFree(b.p);
        g.plans.clear();
        for (auto &kv : g.live) (void)hipFree(kv.second.ptr);
        g.live.clear();
        g.releases++;
        for (auto &kv : g.cache)
            for (void *p : kv.second) (void)hipFree(p);
        g.cache.clear();
        if (g.workspace) (void)hipFree(g.workspace);
        g.workspace = nullptr; g.workspace_floats = 0;
        if (g.attn_counters) (void)hipFree(g.attn_counters);
        g.attn_counters = nullptr;
        g.prepared.clear();      // the association names buffer ids; a later session may reuse them for other things
        g.n_pieces = 0;
        for (auto &ev : g.ring_done) { if (ev) (void)hipEventDestroy(ev); ev = nullptr; }
        if (g.pinned) (void)hipHostFree(g.pinned);
        g.pinned = nullptr;
        host_trim();
        (void)hipStreamDestroy(g.stream);
        g.stream = nullptr;
        g.live_bytes = g.cached_bytes = 0;
        g.ready = false;
    });
}

int deepj_hip_pool_stats(int64_t out[4]) {
    return guarded([&] {
        if (!out) fail("pool_stats: null output");
        out[0] = (int64_t)g.live.size();
        out[1] = g.live_bytes;
        out[2] = g.cached_bytes;
        out[3] = g.driver_allocs;
    });
}

int deepj_hip_limit_memory(int64_t more) {
    return guarded([&] {
        if (more < -1) fail("limit_memory: a byte count, or -1 for no limit");
        g.memory_limit = more < 0 ? -1 : device_held() + more;
    });
}

void *deepj_hip_host_alloc(int64_t bytes) {
    void *p = nullptr;
    guarded([&] {
        if (bytes <= 0) fail("host_alloc: bad size");
        ensure_init();
        p = host_take((size_t)bytes);
    });
    return p;
}

// Leaves the thread's last error alone: finalisers call it between a failed call and the reading of its message.
void deepj_hip_host_free(void *p) {
    if (!p) return;
    try {
        host_give_back(p);
    } catch (...) {            // (no memory for the list of free blocks: the block stays out of use)
    }
}

void *deepj_hip_stream(void) { return g.ready ? (void *)g.stream : nullptr; }

int32_t deepj_hip_attn_record_splits(void) { return kAttnRecordSplits; }
int32_t deepj_hip_decode_block_positions(int32_t d, int32_t hd, int32_t dff) { return decode_block_ok(d, hd, dff) ? decode_block_positions(d, hd) : 0; }
int32_t deepj_hip_latent_decode_splits(int32_t H, int32_t hd, int32_t rank, int32_t max_seq) { return latent_decode_splits(H, hd, rank, max_seq); }
int32_t deepj_hip_decode_ffn_parts(int32_t dff) { return dff > 0 ? decode_ffn_parts(dff) : 0; }

int64_t deepj_hip_attention_scratch_floats(int32_t S, int32_t H, int32_t hd, int32_t max_seq) {
    if (S <= 0 || H <= 0 || hd <= 0) return 0;
    return attention_scratch_floats(S, H, hd, max_seq);
}

int64_t deepj_hip_q8_floats(int32_t k, int32_t rows) {
    if (k <= 0 || rows <= 0) return 0;
    return (q8_bytes(k, rows) + 3) / 4;
}

int64_t deepj_hip_q8_prepared_floats(int32_t k, int32_t rows) {
    if (k <= 0 || rows <= 0) return 0;
    return q8_prepared_floats(k, rows);
}

int32_t deepj_hip_q8_gemm_path(int32_t m, int32_t k, int32_t rows) {
    if (m <= 1 || k <= 0 || rows <= 0) return 0;
    return q8_gemm_f16_tile_rows(m, rows, k);
}

void deepj_hip_q8_gemm_tile(int32_t m, int32_t k, int32_t rows, int32_t *tile_rows, int32_t *tile_cols, int32_t *k_shares) {
    int tr = 0, tc = 0, ks = 1;
    if (m > 1 && k > 0 && rows > 0) q8_gemm_f16_tile(m, rows, k, &tr, &tc, &ks);
    if (tile_rows) *tile_rows = tr;
    if (tile_cols) *tile_cols = tc;
    if (k_shares) *k_shares = ks;
}

void deepj_hip_q8_gemm_tile_prepared(int32_t m, int32_t k, int32_t rows, int32_t *tile_rows, int32_t *tile_cols, int32_t *k_shares) {
    int tr = 0, tc = 0, ks = 1;
    if (m > 1 && k > 0 && rows > 0) q8_gemm_f16_tile(m, rows, k, &tr, &tc, &ks, true);
    if (tile_rows) *tile_rows = tr;
    if (tile_cols) *tile_cols = tc;
    if (k_shares) *k_shares = ks;
}

static int32_t rows_tile(bool taken, const RowsPlan &p, int32_t *tile_rows, int32_t *tile_cols, int32_t *k_shares) {
    if (tile_rows) *tile_rows = taken ? 32 * p.tmw : 0;
    if (tile_cols) *tile_cols = taken ? 32 * p.tnw : 0;
    if (k_shares) *k_shares = taken ? p.shares : 1;
    return taken;
}
int32_t deepj_hip_q8_gemm_rows_tile(int32_t m, int32_t k, int32_t rows, int32_t norm, int32_t prepared, int32_t alloc_free, int32_t *tile_rows, int32_t *tile_cols,
                                    int32_t *k_shares) {
    RowsPlan p{};
    const bool taken = m > 0 && k > 0 && rows > 0 && q8_gemm_rows_ok(m, rows, k, norm != 0, prepared != 0 && !alloc_free, !alloc_free, &p);
    return rows_tile(taken, p, tile_rows, tile_cols, k_shares);
}
int32_t deepj_hip_q8_gemm_rows_tile_behind(int32_t m, int32_t k, int32_t rows, int32_t prepared, int32_t *tile_rows, int32_t *tile_cols, int32_t *k_shares) {
    RowsPlan p{};
    const bool taken = m > 0 && k > 0 && rows > 0 && q8_gemm_rows_ok(m, rows, k, false, prepared != 0, true, &p, true);
    return rows_tile(taken, p, tile_rows, tile_cols, k_shares);
}

int32_t deepj_hip_q8_linear_rope_ok(int32_t m, int32_t k, int32_t d) {
    if (m <= 1 || k <= 0 || d <= 0) return 0;
    return q8_gemm_f16_rope_ok(m, d, k) ? 1 : 0;
}

int32_t deepj_hip_q8_gemm_f16_extents(int32_t m, int32_t k, int32_t rows, int32_t tile_rows, int32_t tile_cols, int64_t *reach3, int64_t *size3) {
    if (m <= 1 || k <= 0 || rows <= 0 || !reach3 || !size3) return -1;
    int tr = tile_rows, tc = tile_cols;
    if (tr == 0) q8_gemm_f16_tile(m, rows, k, &tr, &tc, nullptr);
    if (!((tr == 128 || tr == 64) && (tc == 256 || tc == 192))) return -1;
    return q8_gemm_f16_extents(m, rows, k, tr, tc, reach3, size3) ? 1 : 0;
}

int deepj_hip_time_ops(const int32_t *cmd, int32_t len, int32_t iters, float *ms_total) {
    return guarded([&] {
        ensure_init();
        if (iters <= 0 || !ms_total) fail("time_ops: bad arguments");
        Scratch need;
        walk(cmd, len, true, &need);
        launch_uploads();
        ensure_scratch(need);
        hipEvent_t e0, e1;
        DJ_HIP(hipEventCreate(&e0));
        DJ_HIP(hipEventCreate(&e1));
        DJ_HIP(hipEventRecord(e0, g.stream));
        for (int i = 0; i < iters; i++) walk(cmd, len, false, nullptr);
        DJ_HIP(hipEventRecord(e1, g.stream));
        DJ_HIP(hipEventSynchronize(e1));
        DJ_HIP(hipEventElapsedTime(ms_total, e0, e1));
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) fail(std::string("kernel launch failed: ") + hipGetErrorString(e));
    });
}

// The shader clock while a stream runs: a one-wavefront kernel on a second stream (default priority) samples
// (shader clock counter, 100 MHz wall clock) pairs while `cmd` runs `iters` times on the library's stream, bracketed by
// wall-clock stamps.  pairs receives 2 * samples counters, window the wall clock before and after the runs.  The
// sampler sleeps sleep_reps x 127 x 64 clocks between samples and ends by itself after `samples` of them.
int deepj_hip_clock_probe(const int32_t *cmd, int32_t len, int32_t iters, int32_t samples, int32_t sleep_reps,
                          uint64_t *pairs, uint64_t *window) {
    return guarded([&] {
        ensure_init();
        if (iters < 0 || samples <= 0 || samples > (1 << 20) || sleep_reps < 0 || sleep_reps > 4096 || !pairs || !window)
            fail("clock_probe: bad arguments");
        Scratch need;
        if (len > 0) walk(cmd, len, true, &need);
        launch_uploads();
        ensure_scratch(need);
        hipStream_t side = nullptr;
        unsigned long long *d = nullptr;
        DJ_HIP(hipStreamCreateWithFlags(&side, hipStreamNonBlocking));
        const size_t bytes = ((size_t)2 * samples + 2) * sizeof(unsigned long long);
        hipError_t e = hipMalloc((void **)&d, bytes);
        if (e != hipSuccess) { (void)hipStreamDestroy(side); fail(std::string("clock_probe: hipMalloc: ") + hipGetErrorString(e)); }
        (void)hipMemset(d, 0, bytes);
        DJ_HIP(hipDeviceSynchronize());
        launch_clock_probe(side, d, samples, sleep_reps);
        launch_wall_stamp(g.stream, d + 2 * samples);
        for (int i = 0; i < iters && len > 0; i++) walk(cmd, len, false, nullptr);
        launch_wall_stamp(g.stream, d + 2 * samples + 1);
        e = hipStreamSynchronize(g.stream);
        if (e == hipSuccess) e = hipStreamSynchronize(side);
        if (e == hipSuccess) e = hipMemcpy(pairs, d, (size_t)2 * samples * sizeof(unsigned long long), hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(window, d + 2 * samples, 2 * sizeof(unsigned long long), hipMemcpyDeviceToHost);
        (void)hipFree(d);
        (void)hipStreamDestroy(side);
        if (e != hipSuccess) fail(std::string("clock_probe: ") + hipGetErrorString(e));
    });
}

// Per-op kernel durations: every kernel dispatch of every op of the stream carries a start and a stop event, the
// stream runs `iters` times in order with the launches of a flush, and us_per_op[i] receives the mean over the passes of the
// summed begin-to-end times of op i's dispatches in microseconds (-1 for an op that launched nothing: also one that a launch of
// an op in front of it has taken along, with all of that launch's time there).  Optional outputs of the same
// length: us_longest[i], the longest single dispatch of the op (its main kernel), and dispatches[i], how many
// dispatches the op made (at most kMaxTimedLaunches of them are timed).
int deepj_hip_profile_ops(const int32_t *cmd, int32_t len, int32_t iters, float *us_per_op, int32_t capacity,
                          int32_t *n_ops, float *us_longest, int32_t *dispatches) {
    return guarded([&] {
        ensure_init();
        if (iters <= 0 || !us_per_op || capacity < 0) fail("profile_ops: bad arguments");
        Scratch need;
        walk(cmd, len, true, &need);
        launch_uploads();
        ensure_scratch(need);
        std::vector<int32_t> starts;                 // word offset of every op
        for (int32_t pos = 0; pos < len; pos += stride_of(cmd[pos])) starts.push_back(pos);
        const int n = (int)starts.size();
        if (n_ops) *n_ops = n;
        if (n > capacity) fail("profile_ops: the stream holds " + std::to_string(n) + " ops, the output only " + std::to_string(capacity));
        constexpr int per_op = 2 * kMaxTimedLaunches;
        std::vector<hipEvent_t> ev((size_t)per_op * n, nullptr);
        std::vector<std::vector<float>> sums((size_t)n), longest((size_t)n);
        std::vector<int> launches((size_t)n, 0);
        auto cleanup = [&] {
            g_launch_timing = LaunchTiming{};
            for (hipEvent_t e : ev) if (e) (void)hipEventDestroy(e);
        };
        try {
            for (auto &e : ev) DJ_HIP(hipEventCreate(&e));
            // An op's time is the median of its passes, two more than asked for: one pass in some 400 shows a dispatch 5 to 75 us longer than
            // all others (in 1800 passes over three ops: 5), and no few passes' mean is near the kernel's time with one of them in it.
            for (int it = -2; it < iters; it++) {
                g.chain.valid = false;
                Cursor c{cmd, len, 0, false, 0};                     // (as walk)
                for (int i = 0; i < n; i++) {
                    launches[(size_t)i] = 0;
                    if (c.pos > starts[(size_t)i]) continue;         // an op in front has taken it along
                    const int32_t stride = stride_of(cmd[c.pos]);
                    if (c.next_done < c.n_done && c.done[c.next_done] == c.pos) { c.next_done++; c.pos += stride; continue; }
                    g_launch_timing.pairs = ev.data() + (size_t)per_op * i;
                    g_launch_timing.used = 0;
                    g_launch_timing.armed = true;
                    exec_one(c);
                    launches[(size_t)i] = g_launch_timing.used;
                    g_launch_timing.armed = false;
                    c.pos += stride + c.skip;
                    c.skip = 0;
                }
                DJ_HIP(hipStreamSynchronize(g.stream));
                for (int i = 0; i < n; i++) {
                    if (!launches[(size_t)i]) continue;
                    double total = 0.0, top = 0.0;
                    for (int j = 0; j < launches[(size_t)i]; j++) {
                        float ms = 0.0f;
                        DJ_HIP(hipEventElapsedTime(&ms, ev[(size_t)per_op * i + 2 * j], ev[(size_t)per_op * i + 2 * j + 1]));
                        total += (double)ms * 1e3;
                        top = std::max(top, (double)ms * 1e3);
                    }
                    sums[(size_t)i].push_back((float)total);
                    longest[(size_t)i].push_back((float)top);
                }
            }
        } catch (...) {
            cleanup();
            throw;
        }
        cleanup();
        auto median = [](std::vector<float> &v) {
            if (v.empty()) return -1.0f;
            std::sort(v.begin(), v.end());
            return 0.5f * (v[(v.size() - 1) / 2] + v[v.size() / 2]);
        };
        for (int i = 0; i < n; i++) {
            us_per_op[i] = median(sums[(size_t)i]);
            if (us_longest) us_longest[i] = median(longest[(size_t)i]);
            if (dispatches) dispatches[i] = launches[(size_t)i];
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) fail(std::string("kernel launch failed: ") + hipGetErrorString(e));
    });
}

int deepj_hip_graph_capture(const int32_t *cmd, int32_t len, int32_t *handle) {
    return guarded([&] {
        ensure_init();
        if (!handle) fail("graph_capture: null handle");
        Scratch need;
        Graph gr;
        g.track = &gr.refs;
        try {
            walk(cmd, len, true, &need);
        } catch (...) {
            g.track = nullptr;
            throw;
        }
        g.track = nullptr;
        std::sort(gr.refs.begin(), gr.refs.end());
        gr.refs.erase(std::unique(gr.refs.begin(), gr.refs.end()), gr.refs.end());
        launch_uploads();
        ensure_scratch(need);
        DJ_HIP(hipStreamSynchronize(g.stream));
        DJ_HIP(hipStreamBeginCapture(g.stream, hipStreamCaptureModeThreadLocal));
        g.capturing = true;
        g.capture_into = &gr;
        try {
            walk(cmd, len, false, nullptr);
        } catch (...) {
            g.capturing = false;
            g.capture_into = nullptr;
            hipGraph_t tmp = nullptr;
            (void)hipStreamEndCapture(g.stream, &tmp);
            if (tmp) (void)hipGraphDestroy(tmp);
            throw;
        }
        g.capturing = false;
        g.capture_into = nullptr;
        DJ_HIP(hipStreamEndCapture(g.stream, &gr.graph));
        hipError_t e = hipGraphInstantiate(&gr.exec, gr.graph, nullptr, nullptr, 0);
        if (e != hipSuccess) {
            (void)hipGraphDestroy(gr.graph);
            fail(std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
        }
        int32_t h = g.next_graph++;
        g.graphs.emplace(h, gr);
        *handle = h;
    });
}

int deepj_hip_graph_launch(int32_t handle, int32_t times) {
    return guarded([&] {
        auto it = g.graphs.find(handle);
        if (it == g.graphs.end()) fail("graph_launch: unknown graph handle " + std::to_string(handle));
        // the graph replays raw addresses: refuse when a buffer it names was released or now lives elsewhere,
        // or when the workspace it used has been replaced by a larger one
        for (const auto &ref : it->second.refs) {
            auto b = g.live.find(ref.first);
            if (b == g.live.end() || b->second.ptr != ref.second)
                fail("graph_launch: buffer id=" + std::to_string(ref.first) + " was released or reallocated after graph " +
                     std::to_string(handle) + " was captured; capture the stream again");
        }
        if (it->second.workspace && it->second.workspace != g.workspace)
            fail("graph_launch: the workspace was reallocated after graph " + std::to_string(handle) +
                 " was captured; capture the stream again");
        for (const auto &pr : it->second.prepared) {
            auto p = g.prepared.find(pr.first);
            if (p == g.prepared.end() || p->second.id != pr.second)
                fail("graph_launch: Q8 weights id=" + std::to_string(pr.first) + " were written after graph " + std::to_string(handle) +
                     " was captured with their prepared copy id=" + std::to_string(pr.second) + "; capture the stream again");
        }
        launch_uploads();
        // Bounded run-ahead: at most kRing windows of kWindow replays are queued behind the one the
        // device is executing, so a long run never piles tens of thousands of dispatches (and their
        // kernel-argument blocks) into the queue; the device is never left idle by this.
        constexpr int kWindow = 16, kRing = 4;
        static hipEvent_t ring[kRing] = {};
        for (int i = 0; i < times; i++) {
            if (i % kWindow == 0) {
                int w = i / kWindow, slot = w % kRing;
                if (!ring[slot]) DJ_HIP(hipEventCreateWithFlags(&ring[slot], hipEventDisableTiming));
                if (w >= kRing) DJ_HIP(hipEventSynchronize(ring[slot]));
                if (w > 0) DJ_HIP(hipEventRecord(ring[(w - 1) % kRing], g.stream));
            }
            DJ_HIP(hipGraphLaunch(it->second.exec, g.stream));
        }
    });
}

int deepj_hip_graph_destroy(int32_t handle) {
    return guarded([&] {
        auto it = g.graphs.find(handle);
        if (it == g.graphs.end()) return;
        DJ_HIP(hipStreamSynchronize(g.stream));
        (void)hipGraphExecDestroy(it->second.exec);
        (void)hipGraphDestroy(it->second.graph);
        float *pieces = it->second.row_pieces;
        g.graphs.erase(it);
        if (pieces && pieces != g.row_pieces && !graph_holds_pieces(pieces)) DJ_HIP(hipFree(pieces));
    });
}

// ── runs of tokens ──────────────────────────────────────────────────────────
static void plan_release(TokenPlan &p) {
    for (const TokenPlan::Block &b : p.blocks) { g.live_bytes -= (int64_t)b.bytes; pool_free(b.p, b.bytes); }
    p.blocks.clear();
}

// The groups that a plan of this shape takes; 0: it is none for one
static int shape_groups(TokenShape s) {
    if (s.groups == 0) s.groups = token_run_groups(s);
    return token_run_ok(s) ? s.groups : 0;
}

int32_t deepj_hip_token_plan_shape_groups(int32_t kind, int32_t vocab, int32_t max_seq, int32_t d, int32_t heads, int32_t layers, int32_t dff, int32_t groups) {
    if ((kind != 0 && kind != 2) || vocab <= 0 || max_seq <= 0 || d <= 0 || heads <= 0 || layers <= 0 || dff <= 0 || d % heads != 0 || groups < 0) return 0;
    return shape_groups(TokenShape{d, heads, d / heads, layers, dff, vocab, max_seq, groups, kind == 2 ? 1 : 0});
}

int deepj_hip_token_plan_create(const int32_t *w, int32_t n, int32_t *handle) {
    return guarded([&] {
        ensure_init();
        if (!handle) fail("token_plan_create: null handle");
        *handle = 0;
        if (!w || n < DEEPJ_HIP_TOKEN_PLAN_WORDS) fail("token_plan_create: truncated description");
        const int layers = w[5];
        if (layers < 1 || (int64_t)n != DEEPJ_HIP_TOKEN_PLAN_WORDS + (int64_t)layers * DEEPJ_HIP_TOKEN_PLAN_LAYER_WORDS)
            fail("token_plan_create: the description does not hold its layers");
        if (w[0] != 0 && w[0] != 2) fail("token_plan_create: kind must be 0 (Llama) or 2 (GPT)");
        for (int i : {1, 2, 3, 4, 6})
            if (w[i] <= 0) fail("token_plan_create: sizes must be positive");
        if (w[3] % w[4] != 0) fail("token_plan_create: d must be a multiple of the heads");
        if (w[7] < 0) fail("token_plan_create: bad group count");
        const bool gpt = w[0] == 2;
        TokenShape s{w[3], w[4], w[3] / w[4], layers, w[6], w[1], w[2], w[7], gpt ? 1 : 0};
        s.groups = shape_groups(s);
        if (!s.groups || (int)g.plans.size() >= kPlanSlots || !token_run_resident(s)) return;      // handle 0: not a model for it
        TokenPlan p;
        const int op = DJ_OP_Q8_LINEAR;
        std::vector<std::pair<int32_t, void *>> named;
        g.track = &named;
        std::vector<TokenLayer> table((size_t)layers + 1);                       // (the last: the final norm)
        struct Weight { const int8_t *q = nullptr; const float *s = nullptr; int k = 0; };
        std::vector<Weight> weights;
        Weight head;
        try {
            TokenRun &r = p.run;
            const int64_t d = s.d, half = s.hd / 2;
            r.shape = s;
            r.emb = buf(w[8], (int64_t)s.vocab * d, op, "emb");
            r.pos = gpt ? buf(w[9], (int64_t)s.max_seq * d, op, "pos") : nullptr;
            table.back().g1 = buf(w[10], d, op, "gf");
            if (gpt) table.back().be1 = buf(w[11], d, op, "bf");
            q8_weight(w[12], d, s.vocab, op, "wlm", head.q, head.s);
            head.k = s.d;
            r.blm = buf(w[13], s.vocab, op, "blm");
            r.cos_t = buf(w[14], s.max_seq * half, op, "cos");
            r.sin_t = buf(w[15], s.max_seq * half, op, "sin");
            r.kc = buf(w[16], (int64_t)layers * s.max_seq * d, op, "kCache");
            r.vc = buf(w[17], (int64_t)layers * s.max_seq * d, op, "vCache");
            r.state = reinterpret_cast<int32_t *>(buf(w[18], 4, op, "state"));
            r.tokens = reinterpret_cast<int32_t *>(buf(w[19], s.max_seq, op, "tokens"));
            r.logits = buf(w[20], s.vocab, op, "logits");
            r.x = buf(w[21], d, op, "x");
            r.scale = (float)(1.0 / std::sqrt((double)s.hd));
            r.polls = kTokenPolls;
            for (int l = 0; l < layers; l++) {
                const int32_t *v = w + DEEPJ_HIP_TOKEN_PLAN_WORDS + l * DEEPJ_HIP_TOKEN_PLAN_LAYER_WORDS;
                TokenLayer &L = table[(size_t)l];
                L.g1 = buf(v[0], d, op, "g1");
                if (gpt) L.be1 = buf(v[1], d, op, "be1");
                L.g2 = buf(v[2], d, op, "g2");
                if (gpt) L.be2 = buf(v[3], d, op, "be2");
                Weight qkv, wo, up, down;
                q8_weight(v[4], d, 3 * d, op, "wqkv", qkv.q, qkv.s);
                q8_weight(v[5], d, d, op, "wo", wo.q, wo.s);
                q8_weight(v[6], d, (gpt ? 1 : 2) * (int64_t)s.dff, op, "wgu", up.q, up.s);
                q8_weight(v[9], s.dff, d, op, "wd", down.q, down.s);
                qkv.k = wo.k = up.k = s.d;
                down.k = s.dff;
                L.bg = buf(v[7], s.dff, op, "bg");
                if (!gpt) L.bu = buf(v[8], s.dff, op, "bu");
                L.bd = buf(v[10], d, op, "bd");
                for (const Weight &x : {qkv, wo, up, down}) weights.push_back(x);
            }
        } catch (...) {
            g.track = nullptr;
            throw;
        }
        g.track = nullptr;
        for (const auto &ref : named) p.refs.emplace_back(ref.first, g.live.at(ref.first).made);
        std::sort(p.refs.begin(), p.refs.end());
        p.refs.erase(std::unique(p.refs.begin(), p.refs.end()), p.refs.end());
        try {
            std::vector<uint32_t> offsets((size_t)s.groups * kTokenMembers * kTokenWaves);
            const int64_t items = token_run_items(s, offsets.data());
            auto take = [&](int64_t bytes) {
                const size_t cls = size_class((size_t)bytes);
                void *m = pool_alloc(cls, true);
                p.blocks.push_back({m, cls});
                g.live_bytes += (int64_t)cls;
                return m;
            };
            const int64_t exchange_words = kTokenFront + token_exchange(s).total;
            unsigned long long *exchange;
            unsigned char *packed;
            uint32_t *at;
            float *vectors;
            try {
                packed = (unsigned char *)take(items * kTokenItemBytes);
                at = (uint32_t *)take((int64_t)offsets.size() * 4);
                vectors = (float *)take((int64_t)table.size() * token_vectors(s).stride * 4);
                exchange = (unsigned long long *)take(exchange_words * 8);
            } catch (const std::exception &) {                               // a model that fits without a plan goes on without one
                plan_release(p);
                return;
            }
            p.run.items = packed;
            p.run.exchange = exchange + kTokenFront;
            p.run.passing = items * kTokenItemBytes > kTokenPassingBytes;
            p.run.offsets = at;
            p.run.vectors = vectors;
            launch_uploads();
            stage_upload((float *)at, (const float *)offsets.data(), (int64_t)offsets.size());
            launch_uploads();
            launch_fill(g.stream, (uint32_t *)exchange, 0, exchange_words * 2);
            for (int l = 0; l <= layers; l++) launch_token_vectors(g.stream, s, l, table[(size_t)l], vectors);
            for (int l = 0; l < layers; l++)
                for (int phase = kTokenQkv; phase <= kTokenDown; phase++) {
                    const Weight &x = weights[(size_t)l * 4 + phase];
                    launch_token_pack(g.stream, s, phase, l, x.q, x.s, x.k, packed, at);
                }
            launch_token_pack(g.stream, s, kTokenHead, 0, head.q, head.s, head.k, packed, at);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) fail(std::string("kernel launch failed: ") + hipGetErrorString(e));
        } catch (...) {
            plan_release(p);
            throw;
        }
        std::vector<bool> used(kPlanSlots, false);
        for (const auto &kv : g.plans) used[(size_t)kv.second.slot] = true;
        p.slot = (int)(std::find(used.begin(), used.end(), false) - used.begin());
        p.run.failed = (uint32_t *)(g.pinned + kPlansAt) + p.slot;
        *p.run.failed = 0;
        p.releases_seen = g.releases;
        *handle = g.next_plan++;
        g.plans.emplace(*handle, std::move(p));
    });
}

// The plan, if the buffers it was made over are still there: looked up again only once some buffer has been released.
static TokenPlan &plan_of(int32_t handle, const char *call) {
    auto it = g.plans.find(handle);
    if (it == g.plans.end()) fail(std::string(call) + ": unknown plan " + std::to_string(handle));
    TokenPlan &p = it->second;
    if (p.blocks.empty()) fail(std::string(call) + ": the memory of plan " + std::to_string(handle) + " was given back");
    if (p.releases_seen == g.releases) return p;
    for (const auto &ref : p.refs) {
        auto b = g.live.find(ref.first);
        if (b == g.live.end() || b->second.made != ref.second)
            fail(std::string(call) + ": buffer id=" + std::to_string(ref.first) + " was released or reallocated after plan " + std::to_string(handle) + " was made");
    }
    p.releases_seen = g.releases;
    return p;
}

static bool plan_failed(const TokenPlan &p) { return *(volatile uint32_t *)p.run.failed != 0; }

static void plan_launch(TokenPlan &p, TokenRun r) {
    if (plan_failed(p)) return;                                  // (it would leave at once)
    const uint64_t need = 1 + (uint64_t)r.steps * token_tags(r.shape);
    if (p.next_tag + need > 0xffffffffull) {                     // tags start over: nothing of them may be left
        launch_fill(g.stream, (uint32_t *)r.exchange, 0, (int64_t)token_exchange(r.shape).total * 2);
        p.next_tag = 1;
    }
    r.tag = p.next_tag;
    p.launched = true;
    launch_token_run(g.stream, r);
    p.next_tag += (uint32_t)need;
}

int deepj_hip_token_plan_run(int32_t handle, int32_t steps, int32_t choose) {
    return guarded([&] {
        if (choose != kTokenLogits && choose != kTokenGreedy) fail("token_plan_run: choose must be 0 (logits only) or 1 (greedy)");
        if (steps < 1 || (choose == kTokenLogits && steps != 1)) fail("token_plan_run: bad step count " + std::to_string(steps));
        TokenPlan &p = plan_of(handle, "token_plan_run");
        launch_uploads();
        for (int done = 0; done < steps; done += kTokenMostSteps) {
            TokenRun r = p.run;
            r.steps = std::min(kTokenMostSteps, steps - done);
            r.choose = choose;
            plan_launch(p, r);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) fail(std::string("kernel launch failed: ") + hipGetErrorString(e));
    });
}

int deepj_hip_token_plan_step(int32_t handle, int32_t pos, int32_t token, int32_t generated) {
    return guarded([&] {
        TokenPlan &p = plan_of(handle, "token_plan_step");
        if (pos < 0 || pos >= p.run.shape.max_seq) fail("token_plan_step: position " + std::to_string(pos) + " outside the context window");
        launch_uploads();
        TokenRun r = p.run;
        r.steps = 1;
        r.choose = kTokenLogits;
        r.given = 1;
        r.pos_given = pos;
        r.token_given = token;
        r.generated_given = generated;
        plan_launch(p, r);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) fail(std::string("kernel launch failed: ") + hipGetErrorString(e));
    });
}

int32_t deepj_hip_token_plan_failed(int32_t handle) {
    auto it = g.plans.find(handle);
    return it == g.plans.end() ? 0 : (int32_t)plan_failed(it->second);
}

int32_t deepj_hip_token_plan_groups(int32_t handle) {
    auto it = g.plans.find(handle);
    return it == g.plans.end() || it->second.blocks.empty() ? 0 : it->second.run.shape.groups;
}

static TokenPlan &plan_to_set(int32_t handle, const char *call) {
    auto it = g.plans.find(handle);
    if (it == g.plans.end()) fail(std::string(call) + ": unknown plan " + std::to_string(handle));
    return it->second;
}

int deepj_hip_token_plan_set_polls(int32_t handle, int32_t polls) {
    return guarded([&] {
        TokenPlan &p = plan_to_set(handle, "token_plan_set_polls");
        if (polls < 0 || polls > kTokenPolls) fail("token_plan_set_polls: 0 to " + std::to_string(kTokenPolls));
        p.run.polls = polls;
    });
}

int deepj_hip_token_plan_set_far(int32_t handle, int32_t far) {
    return guarded([&] {
        const TokenPlan &p = plan_to_set(handle, "token_plan_set_far");
        if (p.blocks.empty()) return;
        launch_fill(g.stream, (uint32_t *)(p.run.exchange - kTokenFront) + 1, far != 0, 1);
    });
}

int deepj_hip_token_plan_set_tag(int32_t handle, uint32_t tag) {
    return guarded([&] {
        TokenPlan &p = plan_to_set(handle, "token_plan_set_tag");
        if (tag < p.next_tag) fail("token_plan_set_tag: words with tags up to " + std::to_string(p.next_tag - 1) + " may lie in the exchange block");
        p.next_tag = tag;
    });
}

int deepj_hip_token_plan_destroy(int32_t handle) {
    return guarded([&] {
        auto it = g.plans.find(handle);
        if (it == g.plans.end()) return;
        // Blocks are reused behind the stream's work; its word of the pinned block, which the host writes for the next plan, is not
        if (it->second.launched) DJ_HIP(hipStreamSynchronize(g.stream));
        plan_release(it->second);
        g.plans.erase(it);
    });
}

}  // extern "C"
