// A device in host memory for host-side tests of the engine: the HIP runtime calls jfh_engine.cpp makes and the kernel
// launchers of jfh_kernels.hpp. "Device" memory is host memory with known bounds, copies and fills are checked against
// them, launches change nothing (a stage's residual rows come out as they went in; captured ones run when their graph
// does) and a clock of its own stands for
// device time: a fill takes 100 ms per MB, a launch 1 us per row.
#pragma once

#include "jfh_engine.hpp"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <stdexcept>
#include <thread>
#include <utility>
#include <vector>

namespace fake {

inline std::mutex lock;
inline std::map<uintptr_t, size_t> live;  // allocations
inline size_t live_bytes = 0;
inline size_t fail_from = ~size_t{0};     // allocations of this many bytes or more fail ...
inline size_t memory = ~size_t{0};        // ... and those that would exceed this much in all
inline double clock_ms = 0.0;
inline int faults = 0;                    // copies, fills and frees outside an allocation
inline int captures = 0;
inline hipError_t last_error = hipSuccess;  // of a refused allocation, until it is read: a launch reports it
inline std::atomic<uint32_t> step_rows{0};      // rows of the step being launched
inline std::atomic<uint32_t> longest_step{0};
inline std::atomic<int> us_per_256_rows{0};     // real time a step's synchronization takes

inline void fault(const char* what) {
    ++faults;
    std::printf("FAIL: device %s out of bounds\n", what);
}

inline bool inside(const void* p, size_t n) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    auto it = live.upper_bound(a);
    if (it == live.begin()) return false;
    --it;
    return a + n <= it->first + it->second;
}

// A launch: runs now, or with the graph being captured.
inline bool capturing = false;
using Work = std::vector<std::function<void()>>;
inline Work captured;

inline void launch(std::function<void()> work) {
    if (last_error != hipSuccess) {
        last_error = hipSuccess;
        throw std::runtime_error("a launch reports the error of an earlier call");
    }
    if (capturing) captured.push_back(std::move(work));
    else work();
}

inline void launched(double rows) {
    launch([rows] {
        std::lock_guard l(lock);
        clock_ms += rows * 1e-3;
    });
}

}  // namespace fake

struct ihipEvent_t {
    double at = 0.0;
};

extern "C" {

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t* p, int) {
    std::snprintf(p->name, sizeof p->name, "host memory");
    std::snprintf(p->gcnArchName, sizeof p->gcnArchName, "gfx950");
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "fake device error"; }
hipError_t hipGetLastError() {
    std::lock_guard l(fake::lock);
    return std::exchange(fake::last_error, hipSuccess);
}

hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard l(fake::lock);
    *p = nullptr;
    if (n >= fake::fail_from || fake::live_bytes + n > fake::memory) return fake::last_error = hipErrorOutOfMemory;
    *p = std::aligned_alloc(256, (n + 255) / 256 * 256);
    std::memset(*p, 0xA5, n);
    fake::live[reinterpret_cast<uintptr_t>(*p)] = n;
    fake::live_bytes += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard l(fake::lock);
    auto it = fake::live.find(reinterpret_cast<uintptr_t>(p));
    if (it == fake::live.end()) {
        fake::fault("free");
        return hipErrorInvalidValue;
    }
    fake::live_bytes -= it->second;
    fake::live.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }

hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
    std::lock_guard l(fake::lock);
    const bool ok = (k == hipMemcpyHostToDevice ? fake::inside(d, n) : fake::inside(s, n));
    if (!ok) {
        fake::fault("copy");
        return hipErrorInvalidValue;
    }
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void* d, int v, size_t n) {
    std::lock_guard l(fake::lock);
    if (!fake::inside(d, n)) {
        fake::fault("fill");
        return hipErrorInvalidValue;
    }
    std::memset(d, v, n);
    fake::clock_ms += 100.0 * static_cast<double>(n) / (1 << 20);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    const uint32_t rows = fake::step_rows.exchange(0);
    if (rows > fake::longest_step) fake::longest_step = rows;
    if (rows > 0) std::this_thread::sleep_for(std::chrono::microseconds(fake::us_per_256_rows * ((rows + 255) / 256)));
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    ++fake::captures;
    fake::capturing = true;
    fake::captured.clear();
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    fake::capturing = false;
    *g = reinterpret_cast<hipGraph_t>(1);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *e = reinterpret_cast<hipGraphExec_t>(new fake::Work(fake::captured));
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    for (const auto& work : *reinterpret_cast<fake::Work*>(e)) work();
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    delete reinterpret_cast<fake::Work*>(e);
    return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t* e) { *e = new ihipEvent_t; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    std::lock_guard l(fake::lock);
    e->at = fake::clock_ms;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
    *ms = static_cast<float>(b->at - a->at);
    return hipSuccess;
}

}  // extern "C"

namespace jfh::gpu {

void set_launch_events(hipEvent_t, hipEvent_t) {}
void launch_embed(const DMat&, const StepDev*, float*, int32_t n, int32_t, unsigned long long*, int32_t, hipStream_t) { fake::launched(n); }
void launch_gemv(const GemvArgs& a, hipStream_t) {
    fake::launched(a.n_tok);
    if (a.mode != kQKV) return;
    fake::launch([a] {  // reads the rows' rotations
        std::lock_guard l(fake::lock);
        for (int32_t t = 0; t < a.n_tok; ++t) {
            const size_t row = static_cast<size_t>(a.qkv.head_dim) * sizeof(float);
            if (a.qkv.rope == nullptr ||
                !fake::inside(a.qkv.rope + static_cast<size_t>(a.qkv.step->rows[a.qkv.row0 + t].pos) * a.qkv.head_dim, row)) {
                fake::fault("rope read");
                return;
            }
        }
    });
}
void launch_gemv_wide(const GemvArgs& a, hipStream_t s) { launch_gemv(a, s); }
void launch_quantize(const float*, int32_t, int32_t n, const Act8&, hipStream_t) { fake::launched(n); }
void launch_quantize_norm(const float*, int32_t, const int32_t*, const float*, float, int32_t n, const Act8&, hipStream_t) { fake::launched(n); }
size_t attention_partial_floats(int32_t rows, int32_t n_head, int32_t head_dim, int32_t splits) {
    return static_cast<size_t>(rows) * n_head * splits * (head_dim + 2);
}
void launch_attention(const float*, const StepDev* st, int32_t, int32_t, int32_t, int32_t n_head, int32_t, int32_t head_dim,
                      int32_t splits, float* partial, hipStream_t, int32_t) {
    fake::launch([=] {
        std::lock_guard l(fake::lock);
        if (partial == nullptr ||
            !fake::inside(partial, attention_partial_floats(st->n_rows, n_head, head_dim, splits) * sizeof(float))) {
            fake::fault("attention partials");
        }
        fake::step_rows = static_cast<uint32_t>(st->n_rows);
    });
}
void launch_attention_prefill(const float*, const StepDev*, int32_t n, int32_t, int32_t, int32_t, int32_t, float*, hipStream_t) {
    fake::launch([n] { fake::step_rows = static_cast<uint32_t>(n); });
}
void launch_attention_merge(const float*, const StepDev*, int32_t n, int32_t, int32_t, int32_t, float*, const Act8&, hipStream_t, int32_t) { fake::launched(n); }
void launch_finish(unsigned long long*, const StepDev*, int32_t, StepOut*, hipStream_t) {}
void launch_dequant_rows(const DMat&, int32_t, int32_t, float*, hipStream_t) {}
void launch_gather_rows(const float*, int32_t, float*, int32_t, int32_t, int32_t, int32_t, int32_t, hipStream_t) {}
int32_t wide_min_rows(uint32_t) { return 9; }
int32_t attention_splits(int32_t capacity) { return std::min(32, (capacity + 63) / 64); }
int32_t attention_slots(int32_t splits, int32_t, int32_t, int32_t) { return splits; }
int32_t attention_max_rows(int32_t) { return kMaxRows * 64; }
bool attention_prefill_supported(int32_t n_rows, int32_t, int32_t, int32_t, int32_t, int32_t) { return n_rows > kMaxRows; }
void scratch_setup(int) {}
void* scratch_address(int) { return nullptr; }
std::mutex& scratch_lock(int) {
    static std::mutex m;
    return m;
}

}  // namespace jfh::gpu
