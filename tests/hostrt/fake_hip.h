// fake_hip.h -- a stand-in for the HIP runtime and the kernels (test
// infrastructure): the host runtime (hb_seed.cpp, hb_batch.cpp, hb_serve.cpp)
// is compiled as plain C++ and linked with fake_hip.cpp, so that its handling
// of memory, errors and streams can be tested on the CPU.  Device memory is
// host memory; a failed call leaves its error until hipGetLastError reads it,
// as the runtime does, and every launcher returns that error.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <functional>

#define __align__(n) __attribute__((aligned(n)))
#define HIP_SYMBOL(x) ((const void *)&(x))

struct hb_hsp;
struct hb_scan_args;

// Controls and observations; one set for the process.
struct FakeHip {
    size_t device_total = (size_t)64 << 30;   // hipMalloc fails past this
    std::atomic<size_t> device_used{0};
    std::atomic<size_t> host_used{0};         // page-locked bytes
    std::atomic<int> mallocs{0}, host_mallocs{0}, frees{0}, host_frees{0};
    std::atomic<int> fail_host_malloc{0};     // the next n hipHostMalloc calls fail
    std::atomic<int> fail_malloc{0};          // the next n hipMalloc calls fail
    std::atomic<int> fail_stream_create{0};
    std::atomic<int> fail_order{0};           // the next n hb_launch_order calls fail
    std::atomic<int> fail_finalize{0};        // ... hb_launch_finalize(_compact) after their work
    std::atomic<int> orders{0};               // hb_launch_order calls
    std::atomic<int> host_to_device{0};       // synchronous host-to-device copies
    std::atomic<const void *> async_from{nullptr};   // source of the largest asynchronous one
    std::atomic<size_t> async_bytes{0};
    // the HSPs that a scan of one group finds (called by hb_launch_scan)
    std::function<void(const hb_scan_args &)> scan;
};
extern FakeHip g_fake;

// Work enqueued on the stream (null: the null stream) that nothing waited for.
int fake_pending(hipStream_t st);
int fake_pending_all();
// The size with which a live device buffer was allocated (0: none there).
size_t fake_device_size(const void *p);
size_t fake_host_size(const void *p);
