// fake_hip.cpp -- see fake_hip.h.
#include "fake_hip.h"

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>

#include "hb_runtime.h"

FakeHip g_fake;

namespace {
thread_local hipError_t t_last = hipSuccess;
std::mutex g_mu;
std::map<const void *, size_t> g_device, g_host;
std::map<hipStream_t, int> g_pending;
std::atomic<long> g_handles{16};

hipError_t failed(hipError_t e)
{
    t_last = e;
    return e;
}
bool take(std::atomic<int> &n)
{
    int v = n.load();
    while (v > 0)
        if (n.compare_exchange_weak(v, v - 1)) return true;
    return false;
}
template <class T>
T handle()
{
    return reinterpret_cast<T>(g_handles.fetch_add(16));
}
void enqueue(hipStream_t st)
{
    std::lock_guard<std::mutex> lk(g_mu);
    ++g_pending[st];
}
size_t size_in(const std::map<const void *, size_t> &m, const void *p)
{
    std::lock_guard<std::mutex> lk(g_mu);
    const auto it = m.find(p);
    return it == m.end() ? 0 : it->second;
}
bool inside(const std::map<const void *, size_t> &m, const void *p)
{
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = m.upper_bound(p);
    if (it == m.begin()) return false;
    --it;
    return static_cast<const char *>(p) < static_cast<const char *>(it->first) + it->second;
}
}  // namespace

int fake_pending(hipStream_t st)
{
    std::lock_guard<std::mutex> lk(g_mu);
    return g_pending[st];
}
int fake_pending_all()
{
    std::lock_guard<std::mutex> lk(g_mu);
    int n = 0;
    for (const auto &p : g_pending) n += p.second;
    return n;
}
size_t fake_device_size(const void *p) { return size_in(g_device, p); }
size_t fake_host_size(const void *p) { return size_in(g_host, p); }

extern "C" {
const char *hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetLastError(void)
{
    const hipError_t e = t_last;
    t_last = hipSuccess;
    return e;
}
hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 64 << 10;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 160 << 10;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t)
{
    *t = g_fake.device_total;
    *f = g_fake.device_total - g_fake.device_used;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes)
{
    *p = nullptr;
    if (take(g_fake.fail_malloc)) return failed(hipErrorOutOfMemory);
    if (g_fake.device_used.fetch_add(bytes) + bytes > g_fake.device_total) {
        g_fake.device_used -= bytes;
        return failed(hipErrorOutOfMemory);
    }
    *p = malloc(bytes ? bytes : 1);
    ++g_fake.mallocs;
    std::lock_guard<std::mutex> lk(g_mu);
    g_device[*p] = bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        const auto it = g_device.find(p);
        if (it == g_device.end()) return failed(hipErrorInvalidValue);
        g_fake.device_used -= it->second;
        g_device.erase(it);
        g_pending.clear();   // the runtime waits for the device
    }
    ++g_fake.frees;
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned int)
{
    *p = nullptr;
    if (take(g_fake.fail_host_malloc)) return failed(hipErrorOutOfMemory);
    *p = malloc(bytes ? bytes : 1);
    g_fake.host_used += bytes;
    ++g_fake.host_mallocs;
    std::lock_guard<std::mutex> lk(g_mu);
    g_host[*p] = bytes;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    if (!p) return hipSuccess;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        const auto it = g_host.find(p);
        if (it == g_host.end()) return failed(hipErrorInvalidValue);
        g_fake.host_used -= it->second;
        g_host.erase(it);
    }
    ++g_fake.host_frees;
    free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    memset(a, 0, sizeof(*a));
    a->type = inside(g_host, p)     ? hipMemoryTypeHost
              : inside(g_device, p) ? hipMemoryTypeDevice
                                    : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s)
{
    *p = const_cast<void *>(s);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
    if (k == hipMemcpyHostToDevice) ++g_fake.host_to_device;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    if (k == hipMemcpyHostToDevice && n > g_fake.async_bytes) {
        g_fake.async_bytes = n;
        g_fake.async_from = s;
    }
    memcpy(d, s, n);
    enqueue(st);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
    memset(d, v, n);
    enqueue(st);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void)
{
    std::lock_guard<std::mutex> lk(g_mu);
    g_pending.clear();
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int)
{
    if (take(g_fake.fail_stream_create)) return failed(hipErrorOutOfMemory);
    *s = handle<hipStream_t>();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s)
{
    std::lock_guard<std::mutex> lk(g_mu);
    g_pending[s] = 0;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = handle<hipEvent_t>();
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.f;
    return hipSuccess;
}
}  // extern "C"

// ------------------------------------------------------------------ kernels
// Each counts as work on its stream and returns the error left behind, as the
// real launchers do.
static hipError_t launched(hipStream_t st)
{
    enqueue(st);
    return hipGetLastError();
}

hipError_t hb_launch_lut(const hb_lut_job *, int, const int8_t *, int32_t, bool, hipStream_t st)
{
    return launched(st);
}
hipError_t hb_launch_scan(const hb_scan_args &a, bool, int, int, size_t, hipStream_t st)
{
    if (g_fake.scan) g_fake.scan(a);
    return launched(st);
}
hipError_t hb_scan_allow_lds(size_t) { return hipSuccess; }
hipError_t hb_scan_occupancy(bool, bool, bool, size_t lds, int, int *per_cu)
{
    *per_cu = (int)((160 << 10) / lds);
    return hipSuccess;
}
hipError_t hb_scan_short_occupancy(size_t, int *per_cu)
{
    *per_cu = 5;
    return hipSuccess;
}
hipError_t hb_launch_copy(void *d, const void *s, uint64_t n, hipStream_t st)
{
    memcpy(d, s, n);
    return launched(st);
}
hipError_t hb_launch_fill_u32(uint32_t *d, uint32_t v, uint32_t n, hipStream_t st)
{
    for (uint32_t i = 0; i < n; ++i) d[i] = v;
    return launched(st);
}
hipError_t hb_launch_finalize(const uint32_t *, uint32_t ns, const hb_hsp *recs, uint32_t n,
                              hb_subject_stats *stats, hb_hsp *out, uint32_t *, hb_fin_big *,
                              uint32_t, uint32_t *n_big, uint32_t n_zero, hipStream_t st)
{
    memset(stats, 0, ns * sizeof(*stats));
    memcpy(out, recs, n * sizeof(*out));
    memset(n_big, 0, n_zero * sizeof(*n_big));
    const hipError_t e = launched(st);
    return take(g_fake.fail_finalize) ? hipErrorUnknown : e;
}
hipError_t hb_launch_finalize_compact(const uint32_t *, uint32_t, const hb_hsp *recs, uint32_t n,
                                      hb_subject_hits *, hb_hsp *out, uint32_t *,
                                      unsigned long long *, hb_fin_big *, uint32_t,
                                      hb_fin_small *small, hipStream_t st)
{
    memset(small, 0, sizeof(*small));
    memcpy(out, recs, n * sizeof(*out));
    const hipError_t e = launched(st);
    return take(g_fake.fail_finalize) ? hipErrorUnknown : e;
}
hipError_t hb_launch_first_index(const uint32_t *, uint32_t, uint32_t *, uint32_t *, uint32_t *total,
                                 hipStream_t st)
{
    *total = 0;
    return launched(st);
}
size_t hb_sort_scratch(uint32_t n) { return (size_t)n * 24 + 1024; }
size_t hb_load_scratch(uint32_t n) { return hb_sort_scratch(n) + n / 4096 * 8 + 8; }
hipError_t hb_launch_load_records(hb_load_args a, void *, hipStream_t st)
{
    memset(a.subj, 0, a.n * sizeof(uint4));
    return launched(st);
}
hipError_t hb_launch_load_copy(const hb_load_args &, uint64_t, hipStream_t st) { return launched(st); }
hipError_t hb_launch_order(hb_order_args a, void *, hipStream_t st)
{
    ++g_fake.orders;
    for (int32_t q = 0; q <= a.n_queries; ++q) a.q_first[q] = q ? a.n : 0;
    memcpy(a.out, a.in, a.n * sizeof(*a.out));
    const hipError_t e = launched(st);
    return take(g_fake.fail_order) ? hipErrorUnknown : e;
}
hipError_t hb_launch_gap_list(const hb_gap_args &, uint32_t *, uint32_t *, uint32_t *, hipStream_t st)
{
    return launched(st);
}
hipError_t hb_launch_gapped(const hb_gap_args &, bool, int, hipStream_t st) { return launched(st); }
hipError_t hb_launch_gap_pair(const hb_gap_args &, int, hipStream_t st) { return launched(st); }
bool hb_gap_pair_ok(int32_t, int32_t, int32_t) { return true; }
hipError_t hb_launch_count_oids(const hb_hsp *, uint32_t, uint32_t *, hipStream_t st)
{
    return launched(st);
}
hipError_t hb_launch_gap_compact(const hb_gap_args &a, const uint32_t *, const uint32_t *total,
                                 hb_gapped_stats *stats, hb_gapped_hsp *, uint2 *small,
                                 hipStream_t st)
{
    memset(stats, 0, a.n_subjects * sizeof(*stats));
    *small = make_uint2(*total, 0);
    return launched(st);
}
hipError_t hb_launch_hdb_lengths(const hb_hdb_args &a, hipStream_t st)
{
    for (uint32_t i = 0; i < a.n_seqs; ++i) a.lens[i] = 16;
    return launched(st);
}
hipError_t hb_launch_hdb_copy(const hb_hdb_args &, hipStream_t st) { return launched(st); }
