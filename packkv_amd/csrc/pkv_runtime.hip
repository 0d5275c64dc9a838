// Host-side runtime for the C-ABI library: last-error text, scratch, launch timing.
#include "pkv_block.hpp"
#include "pkv_runtime.hpp"
#include <utility>
#include <tuple>
#include <map>

#include <chrono>
#include <cstdarg>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <vector>

namespace pkv {

static thread_local char g_error[512] = "";

void set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, ap);
    va_end(ap);
}

namespace {
// One workspace per (device, stream): calls on different streams of one device never share scratch, so they may
// overlap.  A buffer that has been handed out is never freed or moved while the process lives: a request for more
// allocates a larger buffer beside it and retires the old one (a captured HIP graph may still hold its address), so
// growth costs memory (at most twice the largest request, growth is geometric) but never a synchronisation.
struct Workspace {
    int dev;
    hipStream_t stream;
    void *ptr;              // general scratch
    size_t bytes;
    uint32_t *counters;     // kAttnCounters tile counters of the attention kernel, zero between launches
    void *enc;              // the encoders' look-back state, zero between encodes
    size_t enc_bytes;
    bool enc_dirty;         // between prepare_scan_state and the launch of the kernel that clears the state
    uint64_t *last;         // pinned, host and device: outcome of the last encode on this stream (kOutcomeWords), tag 0 before it
    std::shared_ptr<std::mutex> enc_mu;
};
static_assert(2 * kOutcomeWords <= kSlotWords, "a slot (a cache line) holds the outcomes of two encodes");
constexpr int kSlotsPerChunk = 64;
std::vector<uint64_t *> g_chunks;                     // pinned slots of the encodes that are waited for (any device)
std::vector<uint64_t *> g_free_slots;                 // as many as host threads have waited at once, in chunks of 64
uint32_t g_seq = 0;                                   // tag of an outcome, 30 bits, never 0
std::vector<Workspace> g_ws;
struct Retired { int dev; hipStream_t stream; void *ptr; };
std::vector<Retired> g_retired;     // superseded buffers, kept until their stream is released (a captured graph may hold them)
std::mutex g_ws_mu;

int workspace_for(hipStream_t s, Workspace **out) {     // caller holds g_ws_mu
    int dev = 0;
    PKV_HIP_CHECK(hipGetDevice(&dev));
    for (Workspace &w : g_ws)
        if (w.dev == dev && w.stream == s) { *out = &w; return PKV_OK; }
    g_ws.push_back(Workspace{dev, s, nullptr, 0, nullptr, nullptr, 0, false, nullptr, std::make_shared<std::mutex>()});
    *out = &g_ws.back();
    return PKV_OK;
}
}  // namespace

size_t scratch_grown_size(size_t have, size_t want) {
    if (want <= have) return have;
    size_t n = have ? have : (size_t)(1 << 20);
    while (n < want) n += n / 2 + (size_t)(1 << 20);
    return n;
}

// True when `s` is recording a HIP graph: nothing may be allocated then.
static bool capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

static int refuse_in_capture(hipStream_t s) {
    PKV_REQUIRE(!capturing(s), PKV_ERR_HIP, "the result is waited for: not possible while the stream is capturing a graph");
    return PKV_OK;
}

int scratch_get(size_t bytes, hipStream_t s, void **out) {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    Workspace *w = nullptr;
    int rc = workspace_for(s, &w);
    if (rc) return rc;
    if (w->bytes < bytes) {
        if (capturing(s)) {
            set_error("stream is capturing a graph and has no scratch buffer of %zu bytes yet: make one eager call "
                      "of the same shape on this stream first", bytes);
            return PKV_ERR_CAPTURING;
        }
        const size_t want = scratch_grown_size(w->bytes, bytes);
        void *fresh = nullptr;
        PKV_HIP_CHECK(hipMalloc(&fresh, want));
        if (w->ptr) g_retired.push_back(Retired{w->dev, s, w->ptr});
        w->ptr = fresh;
        w->bytes = want;
    }
    *out = w->ptr;
    return PKV_OK;
}

// ---- the encoders' look-back state and outcome ------------------------------------------------------------------
// The outcome of the encode before it on the stream to `last` and, for a waiting caller, to `slot`; the state back to
// zero.  Of two encodes `last` keeps the second's outcome unless the first one (codes of `bits` bits) failed.  Four words
// per thread: the state of 1 GiB of input (8192 tickets) is cleared by nine workgroups.  Latency is all there is to it: 4.2 us
// there and 2.2 to 4.1 behind encoders of 8 to 32 MiB (medians of kernel traces).
__global__ void __launch_bounds__(256) finish_encode_kernel(ScanState *st, ScanState *second, uint64_t *words, uint32_t n, uint64_t *last,
                                                            uint64_t *slot, uint32_t tag, int bits) {
    constexpr uint32_t kHead = offsetof(ScanState, status) / 8;
    const uint32_t head2 = second ? (uint32_t)(reinterpret_cast<uint64_t *>(second) - words) : 0xFFFFFFFFu;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        publish_outcomes(st, second, last, slot, tag, bits);
        for (uint32_t i = 0; i < kHead; i++) {
            words[i] = 0;
            if (second) words[head2 + i] = 0;
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
        const uint32_t i = kHead + (blockIdx.x * 4u + k) * 256u + threadIdx.x;
        if (i < n && (i < head2 || i >= head2 + kHead)) words[i] = 0;
    }
}
__global__ void __launch_bounds__(256) clear_state_kernel(uint64_t *p, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

static hipError_t clear_state(const Workspace &w) {
    const size_t all = w.enc_bytes / 8;
    clear_state_kernel<<<(unsigned)((all + 255) / 256), 256, 0, w.stream>>>((uint64_t *)w.enc, all);
    return hipGetLastError();
}

// A call that failed between its launches, with the encoder perhaps under way: the state is cleared behind it, for the
// next encode and for the graphs that hold one.
ScanHandle::~ScanHandle() {
    if (!held.owns_lock() || !st) return;
    std::lock_guard<std::mutex> lock(g_ws_mu);
    Workspace *w = nullptr;
    if (workspace_for(s, &w) == PKV_OK && clear_state(*w) == hipSuccess) w->enc_dirty = false;
}

int prepare_scan_state(uint32_t nblocks, ScanHandle *out, hipStream_t s, bool waited, uint32_t nblocks2) {
    if (waited) {
        const int rc = refuse_in_capture(s);
        if (rc) return rc;
    }
    constexpr size_t head = offsetof(ScanState, status) / 8;
    const size_t n1 = head + nblocks, n = n1 + (nblocks2 ? head + nblocks2 : 0);
    Workspace *w = nullptr;
    int rc;
    {
        std::lock_guard<std::mutex> lock(g_ws_mu);
        if ((rc = workspace_for(s, &w))) return rc;
        out->mu = w->enc_mu;
    }
    out->held = std::unique_lock<std::mutex>(*out->mu);
    std::lock_guard<std::mutex> lock(g_ws_mu);
    if ((rc = workspace_for(s, &w))) return rc;            // (the list may have moved meanwhile)
    // An earlier call failed and so did the clearing behind it (~ScanHandle): the state is cleared first.  Not inside a
    // capture: that would only record it, and an eager encode before the first replay would find the state as it was left.
    if (w->enc_dirty && capturing(s)) {
        set_error("stream is capturing a graph and an encode on it has failed before: make one eager call on this stream first");
        return PKV_ERR_CAPTURING;
    }
    if (w->enc_bytes < n * 8 || !w->last) {
        if (capturing(s)) {
            set_error("stream is capturing a graph and has no scratch buffer of %zu bytes yet: make one eager call "
                      "of the same shape on this stream first", n * 8);
            return PKV_ERR_CAPTURING;
        }
        if (!w->last) {
            void *last = nullptr;
            PKV_HIP_CHECK(hipHostMalloc(&last, kOutcomeWords * 8, hipHostMallocMapped | hipHostMallocCoherent));
            std::memset(last, 0, kOutcomeWords * 8);
            w->last = (uint64_t *)last;
        }
        if (w->enc_bytes < n * 8) {
            const size_t want = scratch_grown_size(w->enc_bytes, n * 8);
            void *fresh = nullptr;
            PKV_HIP_CHECK(hipMalloc(&fresh, want));
            if (w->enc) g_retired.push_back(Retired{w->dev, s, w->enc});
            w->enc = fresh;
            w->enc_bytes = want;
            w->enc_dirty = true;
        }
    }
    if (w->enc_dirty) PKV_HIP_CHECK(clear_state(*w));
    w->enc_dirty = true;
    out->s = s;
    out->st = (ScanState *)w->enc;
    out->second = nblocks2 ? (ScanState *)((uint64_t *)w->enc + n1) : nullptr;
    out->words64 = n;
    return PKV_OK;
}

static int outcome(const volatile uint64_t *o, uint64_t *size_out, int bits) {
    const uint32_t error = (uint32_t)(o[1] & 0xFFu), max_code = (uint32_t)(o[1] >> 8) & 0xFFFFu;
    if (error == (uint32_t)PKV_ERR_CAPACITY) {
        set_error("compressed stream does not fit the output buffer");
        return PKV_ERR_CAPACITY;
    }
    if (error) {
        set_error("device-side encode failure (code %u)", error);
        return (int)error;
    }
    if (bits > 0 && max_code >= (1u << bits)) {
        set_error("not supported: code %u does not fit bits_len %d", max_code, bits);
        return PKV_ERR_UNSUPPORTED;
    }
    *size_out = o[0] & ((1ull << 34) - 1ull);
    return PKV_OK;
}

// Polls pinned memory until `n` words carry the tag: the answer is there a microsecond or two after the kernel wrote
// it, where a copy and a stream synchronisation take about 20.  After 20 ms -- a long queue ahead, or a fault -- the
// stream is waited for in the ordinary way.
static int wait_words(const volatile uint64_t *w, int n, uint32_t tag, hipStream_t s) {
    const auto t0 = std::chrono::steady_clock::now();
    for (bool synced = false;;) {
        for (int i = 0; i < 256; i++) {
            bool there = true;
            for (int k = 0; k < n; k++) there = there && (uint32_t)(w[k] >> 34) == tag;
            if (there) return PKV_OK;
            __builtin_ia32_pause();
        }
        PKV_REQUIRE(!synced, PKV_ERR_INTERNAL, "the encoder's outcome did not arrive");
        if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(20)) {
            PKV_HIP_CHECK(hipStreamSynchronize(s));
            synced = true;
        }
    }
}

static int slot_take(uint64_t **slot, uint32_t *tag) {       // caller holds g_ws_mu; slot NULL: the tag alone
    if (slot) {
        if (g_free_slots.empty()) {
            void *chunk = nullptr;
            PKV_HIP_CHECK(hipHostMalloc(&chunk, (size_t)kSlotsPerChunk * kSlotWords * 8,
                                        hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable));
            std::memset(chunk, 0, (size_t)kSlotsPerChunk * kSlotWords * 8);     // (tags are never 0)
            g_chunks.push_back((uint64_t *)chunk);
            for (int i = 0; i < kSlotsPerChunk; i++) g_free_slots.push_back((uint64_t *)chunk + (size_t)i * kSlotWords);
        }
        *slot = g_free_slots.back();
        g_free_slots.pop_back();
    }
    g_seq = (g_seq + 1) & 0x3FFFFFFFu;
    if (!g_seq) g_seq = 1;
    *tag = g_seq;
    return PKV_OK;
}

int OutcomeSlot::take(hipStream_t s) {
    const int rc = refuse_in_capture(s);
    if (rc) return rc;
    std::lock_guard<std::mutex> lock(g_ws_mu);
    return slot_take(&words, &tag);
}

int OutcomeSlot::wait(int n, hipStream_t s, uint64_t *values) {
    const int rc = wait_words(words, n, tag, s);
    for (int i = 0; i < n && !rc; i++) values[i] = ((const volatile uint64_t *)words)[i] & ((1ull << 34) - 1ull);
    return rc;
}

OutcomeSlot::~OutcomeSlot() {
    if (!words) return;
    std::lock_guard<std::mutex> lock(g_ws_mu);
    g_free_slots.push_back(words);
}

int ClosedEncode::begin(ScanHandle &h, uint32_t total, hipStream_t stream) {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    Workspace *w = nullptr;
    int rc = workspace_for(stream, &w);
    if (rc) return rc;
    uint32_t tag = 0;
    if ((rc = slot_take(nullptr, &tag))) return rc;
    s = stream;
    close.st = h.st;
    close.n = (uint32_t)h.words64;
    close.total = total;
    close.count = (uint64_t *)h.st + (h.words64 - close_words(total));
    close.last = w->last;
    close.tag = tag;
    return PKV_OK;
}

int ClosedEncode::launched(ScanHandle &h) { return scan_state_cleared(h, s); }

int scan_state_cleared(ScanHandle &h, hipStream_t s) {
    {
        std::lock_guard<std::mutex> lock(g_ws_mu);
        Workspace *w = nullptr;
        int rc = workspace_for(s, &w);
        if (rc) return rc;
        w->enc_dirty = false;
    }
    h.held.unlock();
    return PKV_OK;
}

int finish_encode(ScanHandle &h, uint64_t *size_out, int bits, hipStream_t s, uint64_t *size2_out, int bits2) {
    uint64_t *slot = nullptr;
    uint32_t tag = 0;
    {
        std::lock_guard<std::mutex> lock(g_ws_mu);
        Workspace *w = nullptr;
        int rc = workspace_for(s, &w);
        if (rc) return rc;
        if ((rc = slot_take(size_out ? &slot : nullptr, &tag))) return rc;
        const uint32_t n = (uint32_t)h.words64;
        finish_encode_kernel<<<(n + 1023u) / 1024u, 256, 0, s>>>(h.st, h.second, (uint64_t *)h.st, n, w->last, slot, tag, bits);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            if (slot) g_free_slots.push_back(slot);
            set_error("launch of the encoder's last kernel failed: %s", hipGetErrorString(e));
            return PKV_ERR_HIP;
        }
        w->enc_dirty = false;
    }
    h.held.unlock();
    if (!slot) return PKV_OK;
    int rc = wait_words(slot, h.second ? 4 : 2, tag, s);
    if (!rc) rc = outcome(slot, size_out, bits);
    if (!rc && h.second && size2_out) rc = outcome(slot + kOutcomeWords, size2_out, bits2);
    std::lock_guard<std::mutex> lock(g_ws_mu);
    g_free_slots.push_back(slot);
    return rc;
}

static int encode_status(hipStream_t s, int bits, uint64_t *size_out) {
    const uint64_t *last = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_ws_mu);
        Workspace *w = nullptr;
        int rc = workspace_for(s, &w);
        if (rc) return rc;
        last = w->last;
    }
    PKV_HIP_CHECK(hipStreamSynchronize(s));
    PKV_REQUIRE(last && (last[0] >> 34) != 0, PKV_ERR_INVALID, "no encode has run on this stream");
    return outcome(last, size_out, bits);
}

int attn_counters_get(hipStream_t s, uint32_t **out) {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    Workspace *w = nullptr;
    int rc = workspace_for(s, &w);
    if (rc) return rc;
    if (!w->counters) {
        if (capturing(s)) {
            set_error("stream is capturing a graph and has no attention counters yet: make one eager call on this "
                      "stream first");
            return PKV_ERR_CAPTURING;
        }
        void *c = nullptr;
        PKV_HIP_CHECK(hipMalloc(&c, (size_t)kAttnCounters * sizeof(uint32_t)));
        clear_state_kernel<<<kAttnCounters / 512, 256, 0, s>>>((uint64_t *)c, kAttnCounters / 2);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) (void)hipFree(c);
        PKV_HIP_CHECK(e);
        w->counters = (uint32_t *)c;
    }
    *out = w->counters;
    return PKV_OK;
}

// Gives back everything the library holds for (current device, stream `s`): waits for the stream, frees its scratch
// buffers, its tile counters and the buffers it has outgrown, and forgets the stream.
int stream_release(hipStream_t s) {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    int dev = 0;
    PKV_HIP_CHECK(hipGetDevice(&dev));
    PKV_REQUIRE(!capturing(s), PKV_ERR_INVALID, "the stream is capturing a graph");
    size_t at = g_ws.size();
    for (size_t i = 0; i < g_ws.size(); i++)
        if (g_ws[i].dev == dev && g_ws[i].stream == s) at = i;
    bool any = at < g_ws.size();
    for (const Retired &r : g_retired) any = any || (r.dev == dev && r.stream == s);
    if (!any) return PKV_OK;
    PKV_HIP_CHECK(hipStreamSynchronize(s));
    if (at < g_ws.size()) {
        Workspace &w = g_ws[at];
        if (w.ptr) PKV_HIP_CHECK(hipFree(w.ptr));
        if (w.enc) PKV_HIP_CHECK(hipFree(w.enc));
        if (w.last) PKV_HIP_CHECK(hipHostFree(w.last));
        if (w.counters) PKV_HIP_CHECK(hipFree(w.counters));
        g_ws.erase(g_ws.begin() + (long)at);
    }
    for (size_t i = 0; i < g_retired.size();) {
        if (g_retired[i].dev == dev && g_retired[i].stream == s) {
            PKV_HIP_CHECK(hipFree(g_retired[i].ptr));
            g_retired.erase(g_retired.begin() + (long)i);
        } else {
            i++;
        }
    }
    return PKV_OK;
}

int LaunchTimer::begin() {
    if (!enabled) return PKV_OK;
    PKV_HIP_CHECK(hipEventCreate(&start));
    PKV_HIP_CHECK(hipEventCreate(&stop));
    PKV_HIP_CHECK(hipEventRecord(start, stream));
    return PKV_OK;
}

int LaunchTimer::end(float *ms_out) {
    if (!enabled) return PKV_OK;
    PKV_HIP_CHECK(hipEventRecord(stop, stream));
    PKV_HIP_CHECK(hipEventSynchronize(stop));
    float ms = 0.f;
    PKV_HIP_CHECK(hipEventElapsedTime(&ms, start, stop));
    if (ms_out) *ms_out = ms;
    return PKV_OK;
}

LaunchTimer::~LaunchTimer() {
    if (start) (void)hipEventDestroy(start);
    if (stop) (void)hipEventDestroy(stop);
}

__global__ void launch_ended_kernel(const LaunchStamp st) {
    if (threadIdx.x == 0) stamp_now(st.word + 1, st.tag);
}

int StampedLaunch::end(float *ms_out) {
    if (!enabled) return PKV_OK;
    launch_ended_kernel<<<1, 64, 0, stream>>>(stamp());
    PKV_HIP_CHECK(hipGetLastError());
    uint64_t clock[2];
    int rc = slot.wait(2, stream, clock), dev = 0, khz = 0;
    if (rc) return rc;
    waited = true;
    PKV_HIP_CHECK(hipGetDevice(&dev));
    PKV_HIP_CHECK(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    PKV_REQUIRE(khz > 0, PKV_ERR_HIP, "the device reports no wall clock rate");
    *ms_out = (float)((clock[1] - clock[0]) & ((1ull << 34) - 1ull)) / (float)khz;
    return PKV_OK;
}

StampedLaunch::~StampedLaunch() {
    if (slot.words && !waited) (void)hipStreamSynchronize(stream);
}

int stagger_for(const void *kernel, int threads, uint32_t lds, uint32_t nwg, Stagger *out) {
    out->cus = out->slots = 0u;
    if (nwg < 1024u) return PKV_OK;                         // the appends of a growing cache: a handful of workgroups
    int dev = 0, cus = 0, per_cu = 0;
    PKV_HIP_CHECK(hipGetDevice(&dev));
    {   // the two figures are looked up once per (device, kernel, LDS size)
        static std::mutex mu;
        static std::map<std::tuple<int, const void *, uint32_t>, std::pair<int, int>> known;
        std::lock_guard<std::mutex> lock(mu);
        const auto key = std::make_tuple(dev, kernel, lds);
        auto it = known.find(key);
        if (it == known.end()) {
            PKV_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
            PKV_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, (size_t)lds));
            it = known.emplace(key, std::make_pair(cus, per_cu)).first;
        }
        cus = it->second.first;
        per_cu = it->second.second;
    }
    if (cus > 0 && per_cu > 1 && (uint64_t)nwg >= 4ull * (uint64_t)cus * (uint64_t)per_cu) {
        out->cus = (uint32_t)cus;
        out->slots = (uint32_t)per_cu;
    }
    return PKV_OK;
}

}  // namespace pkv

extern "C" {

int pkv_abi_version(void) { return PKV_ABI_VERSION; }

const char *pkv_last_error(void) { return pkv::g_error; }

}  // extern "C"

extern "C" int pkv_encode_status(pkv_stream_t s, int bits, uint64_t *size_out) {
    PKV_REQUIRE(size_out != nullptr, PKV_ERR_INVALID, "null pointer argument");
    return pkv::encode_status((hipStream_t)s, bits, size_out);
}

extern "C" int pkv_stream_release(pkv_stream_t s) { return pkv::stream_release((hipStream_t)s); }
