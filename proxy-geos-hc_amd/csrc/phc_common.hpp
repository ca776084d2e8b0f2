// phc_common.hpp -- shared host-side helpers of libphc.so: thread-local error
// text, HIP call checking, device buffers and small math helpers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <string>

#include <rocprofiler-sdk-roctx/roctx.h>

#include "phc.h"

namespace phc {

// A roctx range over a host-side API call (the run, the step, the tuning):
// rocprofv3 --marker-trace shows it beside the kernels it enqueued.
struct RoctxRange {
    explicit RoctxRange(const char *name) { roctxRangePushA(name); }
    ~RoctxRange() { roctxRangePop(); }
    RoctxRange(const RoctxRange &) = delete;
    RoctxRange &operator=(const RoctxRange &) = delete;
};

void set_error(const char *fmt, ...);
phc_status fail(phc_status code, const char *fmt, ...);

// Evaluate a HIP call; on failure record "<what>: <hip error>" and return
// PHC_ERR_HIP from the enclosing function.
#define PHC_HIP(call)                                                          \
    do {                                                                       \
        hipError_t e_ = (call);                                                \
        if (e_ != hipSuccess)                                                  \
            return ::phc::fail(PHC_ERR_HIP, "%s failed: %s (%s:%d)", #call,    \
                               hipGetErrorString(e_), __FILE__, __LINE__);     \
    } while (0)

#define PHC_TRY(expr)                                                          \
    do {                                                                       \
        phc_status s_ = (expr);                                                \
        if (s_ != PHC_OK) return s_;                                           \
    } while (0)

// Owning device allocation (hipMalloc): move-only, freed by release() or
// when it goes out of scope.
struct DevBuf {
    void *ptr = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    DevBuf(DevBuf &&o) noexcept : ptr(o.ptr), bytes(o.bytes) { o.ptr = nullptr; o.bytes = 0; }
    DevBuf &operator=(DevBuf &&o) noexcept
    {
        if (this != &o) {
            release();
            ptr = o.ptr; bytes = o.bytes;
            o.ptr = nullptr; o.bytes = 0;
        }
        return *this;
    }
    ~DevBuf() { release(); }
    phc_status alloc(size_t n);
    void release();
    template <class T> T *as() const { return static_cast<T *>(ptr); }
};

// A captured chunk of a time loop.  Its nodes name no time sample (the chunk's
// samples sit in a device window that a launch before the graph fills), so
// one graph serves every chunk of the same length that starts from the same
// levels.  Captured anew, a chunk of 100 steps of the 196^2-node 2D mesh took
// 0.42 ms longer (1.19 against 0.77 ms).
struct RunGraph {
    hipGraphExec_t exec = nullptr;
    int n = -1, key = -1, nrec = -1;
    void drop()
    {
        if (exec) (void)hipGraphExecDestroy(exec);
        exec = nullptr;
        n = key = nrec = -1;
    }
};

// The last two chunk lengths that started from the same levels: a program that
// alternates between two (snapshots, a shorter last chunk per shot) captures
// each once.  With one, runs of 10 and 7 steps in turn took 500 us each for the
// capture on the 1201^2-node 2D mesh of order 4, 140 and 106 without.
struct RunGraphs {
    RunGraph slot[2];
    int used = 0;  // the slot of the last run
    hipGraphExec_t exec() const { return slot[used].exec; }
    void drop()
    {
        for (RunGraph &g : slot) g.drop();
    }
};

// Has gs.exec() be the graph of an n-step chunk, capturing `enqueue` in place
// of the one not used last where neither slot holds it (key: whatever else the
// nodes depend on).  Launches nothing: a run changes its levels only after this
// has succeeded, so that one that could not be captured can be called again.
template <class F>
phc_status prepare_captured(hipStream_t stream, RunGraphs &gs, int n, int key, int nrec, F enqueue)
{
    auto holds = [&](const RunGraph &g) { return g.exec && g.n == n && g.key == key && g.nrec == nrec; };
    if (!holds(gs.slot[gs.used])) gs.used = 1 - gs.used;
    RunGraph &g = gs.slot[gs.used];
    if (!holds(g)) {
        if (g.exec) PHC_HIP(hipStreamSynchronize(stream));  // the old graph may still run
        g.drop();
        hipGraph_t graph = nullptr;
        PHC_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
        const phc_status st = enqueue();
        const hipError_t ce = hipStreamEndCapture(stream, &graph);
        if (st != PHC_OK) {
            if (graph) (void)hipGraphDestroy(graph);
            return st;
        }
        if (ce != hipSuccess) return fail(PHC_ERR_HIP, "graph capture failed: %s", hipGetErrorString(ce));
        const hipError_t ie = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ie != hipSuccess) {
            g.exec = nullptr;
            return fail(PHC_ERR_HIP, "graph instantiate failed: %s", hipGetErrorString(ie));
        }
        g.n = n;
        g.key = key;
        g.nrec = nrec;
    }
    return PHC_OK;
}

inline int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

} // namespace phc
