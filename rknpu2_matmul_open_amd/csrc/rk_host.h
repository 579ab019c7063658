// Host-layer internals shared by the three operator translation units:
// context / domain objects, device buffers with per-domain accounting, the
// workspace busy flag, and small validation helpers.  Nothing here touches
// HIP types: the device is reached only through rk_hip_shim.h.
#ifndef RK_HOST_H
#define RK_HOST_H

#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "rk_hip_shim.h"
#include "rk_npu_common.h"

struct rk_npu_ctx {
    int device = 0;
    void* stream = nullptr;
    uint64_t id = 0;          // unique per open(), never reused
    int cu_count = 0;
    int clock_khz = 0;
    char arch[64] = {0};
    // This device's copy of the library's static scratch array (looked up at open; null when
    // the lookup failed): memory for the entry point that allocates nothing.
    void* scratch = nullptr;
    size_t scratch_bytes = 0;
    struct DomainMemory {
        std::atomic<uint64_t> live_bytes{0}, peak_bytes{0}, creates{0}, destroys{0};
        // Reclaim hook of the domain tag (rk_npu_iommu_domain_set_reclaim): called once when a
        // device allocation for this tag reports out-of-memory, after which the allocation is
        // tried once more.  `reclaim_epoch` counts completed calls, so that of several
        // allocations failing together only the first one runs the hook.
        std::mutex reclaim_mutex;
        rk_npu_reclaim_idle_fn reclaim = nullptr;
        void* reclaim_cookie = nullptr;
        std::atomic<uint64_t> reclaim_epoch{0};
    } memory[RK_NPU_IOMMU_DOMAIN_COUNT];
    // Device work of one context is issued on one stream; submissions from
    // different workspaces are serialised here so stream order == call order.
    std::mutex submit_mutex;
    // For panelled host calls (PanelPipe): uploads, and every second panel.  Made with the first workspace that is
    // large enough for them, under submit_mutex.
    void* up_stream = nullptr;
    void* second_stream = nullptr;
    // Per-kernel profile (rk_npu_hip_profile_begin / _end): one stream event in front of every
    // kernel launched on this context's stream while it is on.
    struct ProfileMark {
        const char* kernel;
        void* event;
    };
    std::mutex profile_mutex;
    bool profiling = false;
    std::vector<ProfileMark> profile_marks;
    // Rejected-input flags of workspaces used through the *_device entry
    // points since the last rk_npu_hip_sync().
    std::mutex pending_mutex;
    std::vector<int*> pending_flags;
    // Stream capture (rk_npu_hip_capture_begin / _end): the flags noted while capturing are kept
    // with the graph, whose every launch registers them again -- a replay runs the same kernels
    // and can reject input like the eager call did.  `graphs` lists the live graphs of this
    // context so that a workspace being freed can take its flag out of them.
    bool capturing = false;
    std::vector<int*> capture_flags;
    std::vector<struct rk_npu_hip_graph*> graphs;
};

struct rk_npu_iommu_domain {
    rk_npu_ctx* ctx = nullptr;
    uint32_t id = 0;
};

namespace rkhost {

inline int map_error(int rkh) {
    if (rkh == RKH_OK) return RK_NPU_OK;
    return rkh == RKH_ERR_NOMEM ? RK_NPU_ERR_NOMEM : RK_NPU_ERR_SUBMIT;
}

// (ctx, domain) tag remembered by every handle for the ERR_DOMAIN check.
struct Owner {
    rk_npu_ctx* ctx = nullptr;
    uint64_t ctx_id = 0;
    uint32_t domain_id = 0;
    void bind(const rk_npu_iommu_domain* d) {
        ctx = d->ctx;
        ctx_id = d->ctx->id;
        domain_id = d->id;
    }
    bool same(const Owner& o) const { return ctx_id == o.ctx_id && domain_id == o.domain_id; }
};

// Device allocation accounted against the owning domain tag.
class DeviceBuffer {
public:
    DeviceBuffer() = default;
    DeviceBuffer(const DeviceBuffer&) = delete;
    DeviceBuffer& operator=(const DeviceBuffer&) = delete;
    ~DeviceBuffer() { release(); }
    // Allocates and zero-fills.  Returns an RK_NPU_* code.
    int alloc(const Owner& owner, size_t bytes, bool zero = true);
    void release();
    template <class T = uint8_t> T* as() const { return static_cast<T*>(ptr_); }
    size_t bytes() const { return bytes_; }
    explicit operator bool() const { return ptr_ != nullptr; }

private:
    void* ptr_ = nullptr;
    size_t bytes_ = 0;
    Owner owner_;
};

// Non-reentrancy guard of a workspace: try-lock semantics, BUSY on contention.
class BusyLock {
public:
    explicit BusyLock(std::atomic_flag& flag)
        : flag_(flag), held_(!flag.test_and_set(std::memory_order_acquire)) {}
    ~BusyLock() {
        if (held_) flag_.clear(std::memory_order_release);
    }
    BusyLock(const BusyLock&) = delete;
    BusyLock& operator=(const BusyLock&) = delete;
    explicit operator bool() const { return held_; }

private:
    std::atomic_flag& flag_;
    bool held_;
};

inline bool finite_positive(const float* v, size_t n) {
    if (!v) return false;
    for (size_t i = 0; i < n; ++i)
        if (!std::isfinite(v[i]) || !(v[i] > 0.0f)) return false;
    return true;
}

using Clock = std::chrono::steady_clock;
inline double elapsed_us(Clock::time_point t0) {
    return std::chrono::duration<double, std::micro>(Clock::now() - t0).count();
}

// Stream-side stage timer: records events only when the caller asked for
// timings, so the default path adds no event traffic.
class StageTimer {
public:
    StageTimer(void* stream, bool enabled);
    ~StageTimer();
    void mark();                      // record the next event
    double span_us(int from, int to); // elapsed between marks (after sync)
    int marks() const { return count_; }

private:
    void* stream_;
    bool enabled_;
    void* events_[12] = {nullptr};
    int count_ = 0;
};

// Device int that kernels OR a 1 into when they reject input (NaN / Inf
// activations, non-finite SwiGLU middle), with a pinned host mirror so the
// read-back rides the stream before the call's single wait.
class BadFlag {
public:
    ~BadFlag();
    int init(const Owner& owner);
    int* device() const { return dev_.as<int>(); }
    int enqueue_readback(void* stream);
    bool raised() const; // as of the last read-back that has arrived
    void rearm(void* stream);
    // After the stream wait: true when input was rejected; re-arms the flag.
    bool consume(void* stream);

private:
    DeviceBuffer dev_;
    int* host_ = nullptr;
};
// Pinned, device-visible mirror of a caller's host buffer for the blocking
// host-pointer entry points.  Measured on this box: a copy between pageable
// memory and the device is staged and waited for inside the runtime (15-20 us
// per direction when small; 36 GB/s up, 17 GB/s down when large); a DMA from /
// to pinned memory costs 8-12 us when small and runs at 55 GB/s; a plain
// memcpy runs at 75-80 GB/s while its buffers fit a core's caches and at 27 beyond.
//  * Up to kLimit bytes ("direct"): no copy at all.  The quantization kernel
//    reads A from the mirror (each row once) and the GEMM writes its result
//    straight into the output's mirror, which adds ~1.5 us to a call.
//  * Up to kPipeLimit bytes: the mirror is a staging buffer.  Uploads memcpy a
//    chunk and enqueue its DMA while the next chunk is being copied; downloads
//    enqueue one DMA per chunk with an event behind it, and each chunk is copied to
//    the caller's buffer as soon as its event has passed, large results by several
//    threads: one thread reads what a DMA has just written at 27 GB/s, half the
//    rate of the DMA (16.8 MB 608 us; two threads 327, four 196, eight 140).
// Beyond that, or when the pinned allocation fails, the calls copy from / to
// the caller's buffer as the runtime sees fit.
class HostStage {
public:
    static constexpr size_t kLimit = size_t(1) << 20;
    // Results of the W8A8 and MoE calls are written in place up to 4 MiB: the reference's bench_llm_i8 at 128
    // rows (2 MiB of int32) 158 -> 143 us (4096 x 4096), 201 -> 183 us (11008 x 4096), the MoE layer of 256
    // tokens 281 -> 262 us; 8 MiB and more lose (5.6 MiB of int32: 290 -> 340 - 390 us), and the W4A8 calls
    // keep the input's limit (the FFN's 2 MiB of fp32 written in place: 510 -> 560 us).
    static constexpr size_t kOutLimit = size_t(4) << 20;
    static constexpr size_t kPipeLimit = size_t(64) << 20;
    static constexpr size_t kChunk = size_t(2) << 20;
    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    ~HostStage();
    void init(size_t bytes);        // stays off for 0 or more than kPipeLimit bytes
    explicit operator bool() const { return ptr_ != nullptr; }
    bool direct(size_t bytes) const { return ptr_ && bytes <= bytes_ && bytes <= kLimit; }
    bool direct_out(size_t bytes) const { return ptr_ && bytes <= bytes_ && bytes <= kOutLimit; }
    // direct use: the mirror filled with `bytes` from `user` (kernels read it in place) ...
    const void* fill(const void* user, size_t bytes) const;
    // ... and the mirror as a kernel's output; finish() copies it on to `user` after the wait.
    void* data() const { return ptr_; }
    void finish(void* user, size_t bytes) const;
    // staged use: enqueue the upload of `bytes` from `user` to `device` (RKH_* code)
    int upload(void* stream, void* device, const void* user, size_t bytes) const;
    // enqueue the download of `bytes` from `device`, then wait for it and deliver it to `user`
    int download(void* stream, void* user, const void* device, size_t bytes);
    int finish_download(void* stream, void* user, size_t bytes);

private:
    void* ptr_ = nullptr;
    size_t bytes_ = 0;
    std::vector<void*> events_; // one per chunk of a staged download
    bool staged_ = false;       // the enqueued download went through the mirror
};

// Large blocking calls on host buffers, in panels of rows: while one panel is multiplied or its result on its way down,
// the next ones are copied and on their way up (both directions together run at 95 GB/s, one alone at 55).  Kernels
// and downloads overlap only so far that a panel's kernels start beside the download before and end with it (below).
// Quantization is by row and sums are exact, so the panels give the bits of the whole.
//
// What it is bound by: the download of a panel, 38 us for 2 MiB, and the copies between the caller's buffers and the
// mirrors, 27 GB/s on one thread once the four buffers exceed its caches (three helpers that live as long as the call
// share them).  2048 x 4096 x 4096 on int4 weights, fp16 in and out: 1295 us as upload, kernels and download one after
// the other with one copying thread -> 930.
// Uploads go by the copy engine on a stream of their own.  Downloads are kernels of the runtime, and a kernel that
// reads or writes host memory holds up the end of every kernel beside it until it is over (GEMMs of 10 us took
// 35 - 80, whether the copy had 256 workgroups or 32).  So the panels take two streams in turn, each with
// quantization, GEMM and download in order: a panel's kernels end with the download of the panel before, and its own
// download follows at once.  Downloads behind an event on a third stream left 15 - 30 us between two of them.
class PanelPipe {
public:
    enum Check { ANY, FINITE_F16, FINITE_F32 }; // what the elements of A have to be for C to be written
    PanelPipe() = default;
    PanelPipe(const PanelPipe&) = delete;
    PanelPipe& operator=(const PanelPipe&) = delete;
    ~PanelPipe();
    // a_row / c_row: most bytes that a row has on the host.  Stays off where no call has a use for panels or
    // something could not be made.  The caller holds the context's submission lock.
    void init(const Owner& owner, int M, size_t a_row, size_t c_row);
    // Cuts one call, whose rows have this many bytes; false: it is better off, or has to go, in one piece.
    bool plan(size_t a_row, size_t c_row);
    struct Panel {
        int row, rows;    // the first, a multiple of RKH_ROW_ALIGN, and how many
        const void* a;    // its rows on the device
        void* c;
        void* stream;     // for its kernels, which another panel's may run beside: no scratch is shared
    };
    // What multiplies a panel, by reference: a std::function would allocate for it in the call, and throw where it cannot.
    class Multiply {
    public:
        template <class F>
        explicit Multiply(const F& f) : f_(&f), call_([](const void* g, const Panel& p) { return (*static_cast<const F*>(g))(p); }) {}
        int operator()(const Panel& p) const { return call_(f_, p); }

    private:
        const void* f_;
        int (*call_)(const void*, const Panel&);
    };
    // The planned call: A through a's mirror to a_dev, `multiply` -> RK_NPU_* for each panel, c_dev through c's mirror to C.
    // Gives the submission lock back when everything is enqueued.  `check` fails, or an earlier device call on the
    // workspace has raised `flag` (null where there is nothing to check): C is not written, *rejected set and the flag
    // re-armed.  Returns with nothing of the call under way.
    int run(rk_npu_ctx* ctx, std::unique_lock<std::mutex>& submit, const HostStage& a, const HostStage& c, uint8_t* a_dev,
            uint8_t* c_dev, const void* A, void* C, Check check, BadFlag* flag, bool* rejected,
            const Multiply& multiply);

private:
    static int panel_rows(int M, size_t a_row, size_t c_row);
    int M_ = 0, rows_ = 0;
    size_t a_row_ = 0, c_row_ = 0, panels_ = 0; // of the planned call
    std::vector<void*> up_, down_;              // per panel: uploaded, downloaded
    void* before_ = nullptr;                    // what was on the context's stream before the call
    std::unique_ptr<std::atomic<int>[]> left_;  // per panel: pieces that are not in the mirror yet
};

// A capture or a per-kernel profile is on, which know the context's stream only: calls keep to it.
bool keeps_to_stream(rk_npu_ctx* ctx);

// Blocking check of one raw device flag (used by rk_npu_hip_sync).
bool consume_device_flag(rk_npu_ctx* ctx, int* flag);
void note_pending_flag(rk_npu_ctx* ctx, int* flag);
// A workspace that owns `flag` is going away: no later sync or graph launch may read it.
void forget_pending_flag(rk_npu_ctx* ctx, int* flag);

// Raw upload of a host array into a fresh device buffer (used at weights_create).
int upload(const Owner& owner, DeviceBuffer& dst, const void* src, size_t bytes);

// Bytes of split-K scratch a dense GEMM of this shape may use (0 = never splits).
inline size_t splitk_scratch_bytes(int M, int N, int K, bool w_int4) {
    return rkh_gemm_scratch_bytes(M, N, K, w_int4 ? 1 : 0);
}

} // namespace rkhost

#endif // RK_HOST_H
