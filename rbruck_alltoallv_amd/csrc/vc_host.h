// vc_host.h — what the host-side translation units of librbruck_vc share: the communicator, its grow-only device buffers,
// error reporting, and the few helpers of vc_api.hip the tools in vc_tools.hip need.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/rbruck_vc.h"
#include "vc_common.h"
#include "vc_dispatch.h"
#include "vc_sched.h"
#include "vc_plan_math.h"
#include "vc_scan.h"

extern thread_local std::string g_last_error;      // text of the calling thread's last failure (vc_last_error_string)

inline int fail_hip(hipError_t e, const char *what, int line, const char *file = "vc_api.hip") {
    char buf[256];
    snprintf(buf, sizeof buf, "%s failed at %s:%d: %s", what, file, line, hipGetErrorString(e));
    g_last_error = buf;
    return VC_ERR_HIP;
}

#define HIP_TRY(expr)                                                   \
    do {                                                                \
        hipError_t e_ = (expr);                                         \
        if (e_ != hipSuccess) return fail_hip(e_, #expr, __LINE__, __FILE_NAME__);     \
    } while (0)

inline int fail_arg(const char *msg, int code = VC_ERR_ARG) {
    g_last_error = msg;
    return code;
}

// Grow-only device buffer.
struct DevBuf {
    void *p = nullptr;
    size_t cap = 0;
    hipError_t reserve(size_t bytes) {
        if (bytes <= cap) return hipSuccess;
        if (p) { hipError_t e = hipFree(p); p = nullptr; cap = 0; if (e != hipSuccess) return e; }
        size_t want = std::max(bytes, (size_t)256);
        hipError_t e = hipMalloc(&p, want);
        if (e == hipSuccess) cap = want;
        return e;
    }
    void release() { if (p) (void)hipFree(p); p = nullptr; cap = 0; }
    template <class T> T *as() const { return static_cast<T *>(p); }
};

// Device buffers a call plans into: the communicator's grow-only allocations, or slices of memory the caller of the
// planning functions carved elsewhere.
struct PlanBufs {
    int64_t *slot_off = nullptr, *row_tot = nullptr, *row_base = nullptr, *org_run_base = nullptr, *item_row_tot = nullptr,
            *item_row_base = nullptr, *row_bytes = nullptr, *chain_row_tot = nullptr, *chain_row_base = nullptr, *header = nullptr;
    VcLaunchInfo *launches = nullptr;
    int *rd_packed = nullptr;
    uint32_t *slot_lines() const { return reinterpret_cast<uint32_t *>(slot_off); }      // as a forwarded plan keeps them
    unsigned *ticket = nullptr;           // vc_launch_plan_forward's count of finished workgroups: zero between the calls
};

// What a call asked for: enough to derive its schedule again in the other execution mode.
struct CallParams {
    VcFunc f;
    int n, r, batch, esz, uniform, batch2;
};

// What a kernel needs to tell the host that it is done (VcSignal).  The words serve one kernel at a time: who launches it has them to
// itself until the wait is over.
struct VcDone {
    const unsigned *word = nullptr;       // pinned, as the host sees it ...
    unsigned *word_dev = nullptr;         // ... and the device
    unsigned *ticket = nullptr;           // VC_TICKET_BYTES, zero between the calls
    unsigned value = 0;                   // the value last enqueued for the word
};

struct vc_comm {
    int P = 0;
    int device = 0;
    std::atomic<hipStream_t> stream{nullptr};        // (the metadata steps read it beside a call that moves the communicator to the caller's)
    const int64_t *sbase = nullptr, *rbase = nullptr;
    bool timing = false;
    int forward = 1;                      // vc_comm_set_forwarding: 0 launch per digit, 1 forwarded (list or listless as the last
                                          // call suggests), 2 forwarded through a work-item list, 3 / 4 forwarded, listless with a
                                          // workgroup / a quarter of a wavefront per pair of ranks
    VcHint hint = {0, 0, 0, 0, 0};        // what the last forwarded call on this communicator looked like
    int plan_end = 2;                     // which event marks the end of the planning kernels of the call in progress
    int waits = 0;                        // times the host has waited for the stream in the call in progress
    int64_t items_before_last = 0;        // block pieces of the forwarded call before the one `hint` describes (0: there was none)
    DevBuf verdicts;                      // fixed-stride calls: two sets of VC_VERDICTS words used in turn
    bool verdict_clean = false;           // ... and the set the next call will use is known to be zero
    int verdict_turn = 0;
    DevBuf plan;                          // the plan tables of the current call, one allocation (reserve_plan_bufs)
    DevBuf desc, stage, rd_packed, scratch, counting;
    int64_t *header = nullptr;            // (in `counting`) the planner's header on the device
    VcLaunchInfo *launches = nullptr;     // (there too) the launch table of calls of more launches than travel as an argument
    double cal_copy_bytes_per_s = 0, cal_launch_s = 0, cal_sync_s = 0;   // calibrate(): the plain copy's rate, the cost of a
                                          // launch, of a launch the host waits for
    int bound_staging = 1;                // vc_comm_set_staging_bound
    bool own_allowance = false;           // ... with an allowance of the caller's
    int64_t staging_allowance = 0;        // bytes of staging a forwarded call may take whatever its payload (set with the bound)
    int live_plans = 0;                   // plans created on this communicator and not yet freed
    std::vector<void *> retired_stage;    // staging arenas that were outgrown while plans existed: a HIP graph captured from
                                          // vc_plan_execute_async holds the arena's address, so they stay until the plans go
    std::atomic_flag busy = ATOMIC_FLAG_INIT;   // a call is in progress (a communicator serves one call at a time)
    struct {                              // a call enqueued by an _async entry point that vc_comm_wait has not collected yet
        bool active = false;
        VcSched S;
        VcTables T;
        const char *sendbuf = nullptr;
        char *recvbuf = nullptr;
        int lanes = 0;                    // 0: only planned so far
        VcListlessGuard guard = {0, 0, 0, 0, 0};      // of the launch
        int n_launch_infos = 0;
        hipStream_t own_stream = nullptr; // the communicator's stream while the call runs on the caller's
        CallParams q;                     // what was asked for (the call may have to be run again another way)
    } pending;
    PlanBufs B;                           // where the current call's plan lives
    const void *last_stage = nullptr;     // staging arena of the last call
    int64_t *h_header = nullptr;          // pinned, coherent: the planner writes its header straight into it
    int64_t *h_header_dev = nullptr;      // the same memory as the device sees it
                                          // (VC_TOTALS_AT words in: the totals of a call on fixed-stride staging, slot by slot)
    int *h_flags = nullptr, *h_flags_dev = nullptr;   // pinned, coherent: the two flags of vc_displs_from_counts, as host and device see
                                          // them; behind them the words of the two signals, a cache line each
    VcDone of_call;                       // for what runs under VC_ONE_CALL, or between an _async call and its vc_comm_wait
    VcDone of_meta;                       // for the metadata steps and vc_comm_wait without a call, which do not refuse to run beside one:
    std::mutex meta_mutex;                // they take turns, each from its launch to the end of its wait
    int *max_state = nullptr;             // counting words of vc_allreduce_max_count (under meta_mutex)
    VcLaunchInfo *h_launches = nullptr;   // pinned
    std::vector<hipEvent_t> events;
    vc_stats_t stats;
    int last_nlaunch = 0;
    int64_t launch_first[VC_MAX_LAUNCHES], launch_items[VC_MAX_LAUNCHES];   // work items of the last call
    const VcDesc *last_items = nullptr;
};

// Grows the staging arena.  While plans exist the outgrown arena is kept (not freed): graphs captured from their
// launches write to its address.
inline hipError_t reserve_stage(vc_comm *c, size_t bytes) {
    if (bytes <= c->stage.cap) return hipSuccess;
    if (c->live_plans > 0 && c->stage.p) {
        c->retired_stage.push_back(c->stage.p);
        c->stage.p = nullptr;
        c->stage.cap = 0;
    }
    return c->stage.reserve(bytes);
}

inline void free_retired_stage(vc_comm *c) {
    for (void *p : c->retired_stage) (void)hipFree(p);
    c->retired_stage.clear();
}

// One call at a time per communicator: a second host thread gets VC_ERR_BUSY instead of a race on the plan buffers.
struct BusyGuard {
    vc_comm *c;
    bool mine;
    explicit BusyGuard(vc_comm *comm) : c(comm), mine(comm && !comm->busy.test_and_set(std::memory_order_acquire)) {
        if (mine) c->waits = 0;
    }
    ~BusyGuard() { if (mine) c->busy.clear(std::memory_order_release); }
    bool ok() const { return !c || mine; }
    void keep() { mine = false; }         // the call stays in progress after the entry point returns (vc_comm_wait ends it)
};
// words of h_header: the planner's header, then (in cache lines of their own) the slots of vc_totals_waves(P) wavefronts
#define VC_TOTALS_AT ((VC_HEADER_WORDS(VC_MAX_LAUNCHES) + VC_TOTALS_SLOT - 1) / VC_TOTALS_SLOT * VC_TOTALS_SLOT)
#define VC_HEADER_ROOM (VC_TOTALS_AT + VC_TOTALS_SLOT * (VC_STRIDED_MAX_PAIRS / VC_TOTALS_PER_WAVE))
// words of h_flags: the flags, the word of of_call, the word of of_meta
#define VC_CALL_DONE_AT 32
#define VC_META_DONE_AT 64
#define VC_FLAG_WORDS 96
// `counting` (device): the tickets of of_call and of_meta and max_state, zero from the start; header and launch table
#define VC_MAX_STATE_BYTES 512
#define VC_COUNTING_BYTES (2 * VC_TICKET_BYTES + VC_MAX_STATE_BYTES)
#define VC_HEADER_BYTES ((sizeof(int64_t) * VC_HEADER_WORDS(VC_MAX_LAUNCHES) + 255) / 256 * 256)
#define VC_SPIN_US 10000

// Enqueues launch(st, sig), whose last kernel tells the host by `sig` that everything before it on the stream and it itself are done, and
// waits for that.  `d` is the caller's own until the return (the call holds the communicator, or meta_mutex).  A call that takes longer than
// VC_SPIN_US is waited for by the runtime (4 us are nothing then, and it reports what went wrong), as is a call with per-launch timing on,
// whose events end behind its last kernel.
template <class Launch> inline hipError_t vc_run_and_wait(vc_comm *c, VcDone &d, Launch launch) {
    const hipStream_t st = c->stream;
    const VcSignal sig = {d.word_dev, ++d.value, d.ticket};
    const hipError_t e = launch(st, sig);
    if (e != hipSuccess) return e;
    if (c->timing) return hipStreamSynchronize(st);
    const auto t0 = std::chrono::steady_clock::now();
    for (unsigned spin = 1;; spin++) {
        if (__atomic_load_n(d.word, __ATOMIC_ACQUIRE) == sig.value) return hipSuccess;
        __builtin_ia32_pause();
        if (spin % 1024 == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(VC_SPIN_US)) return hipStreamSynchronize(st);
    }
}

// ... everything enqueued so far (see vc_done_kernel)
inline hipError_t vc_wait_stream(vc_comm *c, VcDone &d) {
    if (c->timing) return hipStreamSynchronize(c->stream);
    return vc_run_and_wait(c, d, [](hipStream_t st, VcSignal sig) { return vc_launch_done(sig.word, sig.value, st); });
}

// A metadata step: it has the words of of_meta to itself until it is over.
template <class Launch> inline hipError_t vc_run_meta(vc_comm *c, Launch launch) {
    std::lock_guard<std::mutex> lock(c->meta_mutex);
    return vc_run_and_wait(c, c->of_meta, launch);
}

// a call waits for the communicator's stream (counted: vc_stats_t.host_waits)
#define VC_WAIT(c) ((c)->waits++, vc_wait_stream((c), (c)->of_call))

#define VC_ONE_CALL(c)                                                                                              \
    BusyGuard busy_guard_(c);                                                                                       \
    if (!busy_guard_.ok()) return fail_arg("the communicator is serving another call (one call at a time)", VC_ERR_BUSY)

// ---- defined in vc_api.hip, used by vc_tools.hip ----
int ensure_events(vc_comm *c, size_t n);
bool stages_in_window(const vc_comm *c);
bool staging_out_of_bound(const vc_comm *c, int64_t stage_bytes, int64_t payload_bytes);
int staging_batches(const vc_comm *c, int64_t stage_bytes);
VcTables make_tables(vc_comm *c, const int *sc, const int *sd, const int *rc, const int *rd);
