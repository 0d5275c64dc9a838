// Host-side runtime shared by the C-ABI entry points: last-error text, per-device scratch
// for the single-pass encoders, and event-based timing of a launch.
#pragma once
#include "pkv_common.hpp"

#include <memory>
#include <mutex>

namespace pkv {

// A device buffer of at least `bytes` that belongs to (current device, stream `s`): calls on different streams get
// different buffers and may overlap; calls on one stream share it and are ordered by the stream.  Buffers grow on
// demand; one that has been handed out is never freed or moved while the process lives (a larger one is allocated
// beside it), so an address captured in a HIP graph stays valid and growing never synchronises.
// While `s` is capturing a HIP graph nothing can be allocated: a request the stream's buffer cannot serve then
// returns PKV_ERR_CAPTURING (library-internal; callers fall back or report it as PKV_ERR_HIP).
constexpr int PKV_ERR_CAPTURING = 100;
int scratch_get(size_t bytes, hipStream_t s, void **out);
// Capacity after growing a buffer of `have` bytes to hold `want` (geometric, at least 1 MiB): host arithmetic only.
size_t scratch_grown_size(size_t have, size_t want);

// Tile counters of the attention kernel for (current device, stream `s`): kAttnCounters zeroed 32-bit words,
// allocated on first use; the attention kernel leaves every counter it used at zero again.
constexpr int kAttnCounters = 65536;
int attn_counters_get(hipStream_t s, uint32_t **out);
int stream_release(hipStream_t s);

// Per-call timing: records start/stop events on `stream` around fn() and returns elapsed ms
// after synchronising on the stop event (mirrors the reference launchers, which time every
// launch with events and return milliseconds: packkv_cuda_ext/src/kernels.cu:560-608).
struct LaunchTimer {
    hipEvent_t start = nullptr, stop = nullptr;
    hipStream_t stream;
    bool enabled;
    LaunchTimer(hipStream_t s, bool on) : stream(s), enabled(on) {}
    int begin();
    int end(float *ms_out);   // synchronises when enabled
    ~LaunchTimer();
};

// perm[blk * block_size + r] = index inside block blk of the token that moves to position r: descending median, equal
// medians in their original order (pkv_repack.hip).
int launch_block_order(const uint8_t *median, int ctx_len, int block_size, uint32_t *perm, hipStream_t s);

// Rows 0 .. n-1 of the windows k_out / v_out [B, H, out_rows, 128] = the dequantised codes of k / v [B, H, n, 128]
// (pkv_quant.hip).
int launch_quant_dequant(const void *k, const void *v, void *k_out, void *v_out, int dtype, int B, int H, int n, int out_rows, float k_rel,
                         float v_rel, hipStream_t s);

struct ScanState;
struct Stagger;
// The stagger of the first resident generation (stagger_first_generation, pkv_block.hpp) for `kernel` launched with
// `threads` threads and `lds` bytes of dynamic LDS over `nwg` workgroups: CU count and workgroups per CU from the
// occupancy query (looked up once per device, kernel and LDS size); zeros -- no stagger -- for launches of fewer
// than four generations.
int stagger_for(const void *kernel, int threads, uint32_t lds, uint32_t nwg, Stagger *out);

// Look-back state of the single-pass encoders, from a buffer of its own per (device, stream) that is all zero between
// encodes: a launch finds it cleared, and the kernel finish_encode launches behind the encoder takes its outcome out
// and clears it again.  One kernel per encode next to the encoder itself, and no copy: the outcome goes straight to
// pinned host memory, where a waiting host thread polls for it.  (Where no size is asked for, encoders of few workgroups do without that kernel: ClosedEncode.)
// Fused K encode of 512 tokens x 8 heads with its size:
// 35.8 us a call, against 49.7 with a clearing kernel in front and a copy and a stream synchronisation behind (V 42.4
// against 55.9); without the size both ways take 19 us.
struct ScanHandle {
    ScanState *st = nullptr;       // the state of `words` status words
    ScanState *second = nullptr;   // a second one behind it (two encodes with one wait)
    size_t words64 = 0;            // 64-bit words of the whole region
    std::shared_ptr<std::mutex> mu;        // held from prepare_scan_state until finish_encode has launched its kernel:
    std::unique_lock<std::mutex> held;     // two host threads that encode on one stream take turns
    hipStream_t s = nullptr;
    ~ScanHandle();
};
// `nblocks` status words (and `nblocks2` for a second state when it is not zero).  `waited`: the call will wait for its
// outcome or its time, which is refused while `s` is capturing, before anything is recorded.
int prepare_scan_state(uint32_t nblocks, ScanHandle *out, hipStream_t s, bool waited, uint32_t nblocks2 = 0);
// Launches the kernel that publishes the outcome and clears the state; with `size_out` waits for it and reports it
// (`size2_out`: of the second state).  `bits` > 0 additionally rejects a launch whose largest code does not fit.
// NULL: returns at once, pkv_encode_status reads the outcome later.
int finish_encode(ScanHandle &h, uint64_t *size_out, int bits, hipStream_t s, uint64_t *size2_out = nullptr, int bits2 = 0);
// An encoder whose last workgroup leaves the outcome and clears the state by itself (encode_close), in place of finish_encode's
// kernel: for calls that hand nothing back.  A size promises that the stream, block_info and the parameters are there as
// well, for any stream of the device, and inside the launch that takes a write-back of its XCD's L2 by every workgroup: K with its size,
// 8 heads, behind a kernel of its own | so released, us: 4096 tokens 40.4 | 42.5, 4 x 8192 58 | 68, 16 x 8192 116 | 176.
struct EncodeClose {
    ScanState *st = nullptr;       // the whole state, `n` words
    uint32_t n = 0, total = 0;     // total: workgroups of the launch; 0: finish_encode follows
    uint64_t *count = nullptr;     // (in the state) workgroups that are done, by groups of kCloseGroup and all together
    uint64_t *last = nullptr, tag = 0;
};
constexpr uint32_t kCloseGroup = 16, kCloseStride = 16;        // words from counter to counter: a cache line of its own each
constexpr uint32_t close_words(uint32_t total) { return kCloseStride * (1u + (total + kCloseGroup - 1u) / kCloseGroup); }
// ... for a launch of `total` workgroups whose state was prepared with close_words(total) more words behind the last status word.
struct ClosedEncode {
    EncodeClose close;
    hipStream_t s = nullptr;
    int begin(ScanHandle &h, uint32_t total, hipStream_t stream);
    int launched(ScanHandle &h);   // the launch has been made: the state will be clear behind it
};
// For a kernel whose last workgroup publishes the outcome and clears the state by itself: a pinned slot of kSlotWords words
// that are valid one by one through their tag (value, 34 bits | tag << 34), and the two ends of its life.  Refused while
// `s` is capturing (a graph's replays would write to a slot that has been given back).
constexpr int kSlotWords = 8;
struct OutcomeSlot {
    uint64_t *words = nullptr;
    uint32_t tag = 0;
    int take(hipStream_t s);
    int wait(int n, hipStream_t s, uint64_t *values);      // the first `n` words, without their tags
    ~OutcomeSlot();
};
// The time of an op that is always timed, without events: its first kernel leaves the device's wall clock as it starts
// (launch_started in workgroup 0) and a kernel of one wavefront behind the last one leaves it again, both in a pinned slot
// that the host polls.  A pair of events recorded around the launch, waited for and read costs the host 17 us, this 10, around a
// kernel of 4 us; events attached to the launch itself (hipExtLaunchKernel) 27.
struct LaunchStamp {
    uint64_t *word;                // NULL: not timed
    uint64_t tag;                  // << 34
};
struct StampedLaunch {
    OutcomeSlot slot;
    hipStream_t stream;
    bool enabled, waited = false;
    StampedLaunch(hipStream_t s, bool on) : stream(s), enabled(on) {}
    int begin() { return enabled ? slot.take(stream) : PKV_OK; }
    ~StampedLaunch();              // a call that failed in between: its stamps have arrived before the slot goes back
    LaunchStamp stamp() const { return LaunchStamp{enabled ? slot.words : nullptr, (uint64_t)slot.tag << 34}; }
    int end(float *ms_out);        // behind the last launch: marks the end and waits when enabled
};
#ifdef __HIPCC__
__device__ __forceinline__ void stamp_now(uint64_t *word, uint64_t tag) {
    __hip_atomic_store(word, ((uint64_t)wall_clock64() & ((1ull << 34) - 1ull)) | tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void launch_started(const LaunchStamp st) {
    if (st.word && (blockIdx.x | blockIdx.y | blockIdx.z | threadIdx.x) == 0) stamp_now(st.word, st.tag);
}
#endif
// ... the launch that clears `h`'s state itself has been made.
int scan_state_cleared(ScanHandle &h, hipStream_t s);
// The block codec from a code matrix through the cells kernels (pkv_quant.hip): where code_cells_serve says so, for the
// reference's block shapes and widths up to 6.  `st` holds code_cells_words status words.
bool code_cells_serve(bool is_k, int ctx_len, int hidden);
uint32_t code_cells_words(bool is_k, int ctx_len, int hidden);
uint32_t code_cells_closes(bool is_k, int ctx_len, int hidden);        // workgroups, where the launch closes by itself; 0: finish_encode follows
int launch_code_cells(bool is_k, const uint8_t *codes, int ctx_len, int hidden, int bits, uint32_t bound, uint8_t *stream,
                      uint64_t capacity, uint32_t *info, ScanState *st, const EncodeClose &close, hipStream_t s);

}  // namespace pkv
