// hb_seed.cpp -- host runtime behind include/hb_seed.h (plain per-query path)
// and the pieces the batched path shares (hb_runtime.h).
//
// Replaces the host half of H-BLAST (h_blast_v1.1/H-BLAST/h_blast.cu):
// device setup, the resident database (instead of an mmap + H2D copy per
// call, h_blast.cu:587-653,1094), lookup-table staging (built on the device
// here instead of copied from NCBI's BlastAaLookupTable, h_blast.cu:940-1008),
// kernel launch (h_blast.cu:1109-1145), event timing (h_blast.cu:1101,1147)
// and result fetch/compaction (H_BLAST_get_data + memory_defrag,
// h_blast.cu:1160-1252).  Errors are returned, never exit().
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <numeric>
#include <thread>
#include <vector>

#include "hb_runtime.h"

static thread_local char g_last_hip[256];

void hb_note_hip_error(hipError_t e, const char *what, int line)
{
    snprintf(g_last_hip, sizeof(g_last_hip), "%s (%s) at line %d", hipGetErrorString(e), what,
             line);
}

// BLOSUM62 in ncbistdaa order -,A,B,C,D,E,F,G,H,I,K,L,M,N,P,Q,R,S,T,V,W,X,Y,Z,U,*,O,J.
// Same values as the reference's table (h_blast_v1.1/H-BLAST/h_blast.c:42-71);
// the gap letter scores -128 so that context sentinels stop every extension.
const int8_t kHbBlosum62[HB_ALPHA][HB_ALPHA] = {
#include "hb_blosum62.inc"
};

// The contexts that there are: what one of them keeps is there for the others.
static std::mutex g_ctx_mu;
static std::vector<hb_ctx *> g_ctxs;

// Frees buffer i of the pool.
static void pool_drop(hb_ctx *c, size_t i)
{
    const hb_pool_buf b = c->pool[i];
    c->pool_bytes -= b.bytes;
    if (b.db) c->pool_db_bytes -= b.bytes;
    c->pool.erase(c->pool.begin() + (long)i);
    hipFree(b.p);
}

// hipMalloc; when it fails, again without what the contexts of the device keep.
// (A failure that is handled must not leave its error: the next launcher would
// return it.)
static void *device_alloc(int device, size_t bytes)
{
    void *p = nullptr;
    if (hipMalloc(&p, bytes) == hipSuccess) return p;
    (void)hipGetLastError();
    {
        std::lock_guard<std::mutex> lk(g_ctx_mu);
        for (hb_ctx *c : g_ctxs) {
            if (c->device != device) continue;
            std::lock_guard<std::mutex> lk2(c->pool_mu);
            while (!c->pool.empty()) pool_drop(c, c->pool.size() - 1);
        }
    }
    if (hipMalloc(&p, bytes) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
}

// A buffer of at least `bytes` and at most twice that and 4 KB.  The pool keeps
// the sizes that its buffers have, also while they are handed out: one that
// served something smaller is as large as before when it comes back.
void *hb_pool_get(hb_ctx *c, size_t bytes)
{
    {
        std::lock_guard<std::mutex> lk(c->pool_mu);
        size_t best = (size_t)-1;
        for (size_t i = 0; i < c->pool.size(); ++i)
            if (c->pool[i].bytes >= bytes && c->pool[i].bytes <= 2 * bytes + 4096 &&
                (best == (size_t)-1 || c->pool[i].bytes < c->pool[best].bytes))
                best = i;
        if (best != (size_t)-1) {
            const hb_pool_buf b = c->pool[best];
            c->pool_bytes -= b.bytes;
            if (b.db) c->pool_db_bytes -= b.bytes;
            c->pool.erase(c->pool.begin() + (long)best);
            c->lent.emplace_back(b.p, b.bytes);
            return b.p;
        }
    }
    void *p = device_alloc(c->device, bytes);
    if (!p) return nullptr;
    std::lock_guard<std::mutex> lk(c->pool_mu);
    c->lent.emplace_back(p, bytes);
    return p;
}

size_t hb_pool_held(hb_ctx *c)
{
    std::lock_guard<std::mutex> lk(c->pool_mu);
    return c->pool_bytes;
}

// A program that loads one database or volume after the other gets the last
// one's buffers again: allocating and freeing them took 1.1 ms of a load of 124
// MB.  What a database held was free for everyone before, so no more than this is
// kept of databases, oldest first out: a volume of 340 MB, its residues and
// their copy.
static constexpr size_t kDbKeep = (size_t)1 << 30;

// Returns a buffer to the pool (db: of a database).  hipFree waits for the whole
// device, so the pool frees (oldest first) only past 64 buffers or 16 GiB.
void hb_pool_put(hb_ctx *c, void *p, bool db)
{
    if (!p) return;
    std::lock_guard<std::mutex> lk(c->pool_mu);
    size_t bytes = 0;
    for (size_t i = c->lent.size(); i-- > 0 && !bytes;)   // (the last ones mostly)
        if (c->lent[i].first == p) {
            bytes = c->lent[i].second;
            c->lent[i] = c->lent.back();
            c->lent.pop_back();
        }
    if (!bytes || (db && bytes > kDbKeep)) {
        hipFree(p);
        return;
    }
    c->pool.push_back(hb_pool_buf{p, bytes, db});
    c->pool_bytes += bytes;
    if (db) c->pool_db_bytes += bytes;
    for (size_t i = 0; c->pool_db_bytes > kDbKeep;)
        if (c->pool[i].db) pool_drop(c, i);
        else ++i;
    while (c->pool.size() > 64 || c->pool_bytes > ((size_t)16 << 30)) pool_drop(c, 0);
}

template <class T>
static bool db_get(hb_ctx *c, T **p, size_t bytes)
{
    *p = static_cast<T *>(hb_pool_get(c, bytes));
    return *p != nullptr;
}
static void db_put(hb_ctx *c, void *p) { hb_pool_put(c, p, true); }

// The smallest page-locked buffer that holds the request, unless it is more than
// four times as large as one made for it: a small request must not sit on the
// buffer of the next load (a batch holds its own as long as it lives).
void *hb_pin_get(hb_ctx *c, size_t *bytes)
{
    const size_t want = (std::max<size_t>(*bytes, 1) + 0x3ffff) & ~(size_t)0x3ffff;
    {
        std::lock_guard<std::mutex> lk(c->pin_mu);
        size_t best = (size_t)-1;
        for (size_t i = 0; i < c->pins.size(); ++i)
            if (c->pins[i].second >= *bytes && c->pins[i].second <= 4 * want &&
                (best == (size_t)-1 || c->pins[i].second < c->pins[best].second))
                best = i;
        if (best != (size_t)-1) {
            void *p = c->pins[best].first;
            *bytes = c->pins[best].second;
            c->pins.erase(c->pins.begin() + (long)best);
            return p;
        }
    }
    void *p = nullptr;
    if (hipHostMalloc(&p, want, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    *bytes = want;
    return p;
}

// At most 8 buffers of up to 16 MiB are kept, the last ones put back.
void hb_pin_put(hb_ctx *c, void *p, size_t bytes)
{
    if (!p) return;
    if (bytes <= ((size_t)16 << 20)) {
        std::lock_guard<std::mutex> lk(c->pin_mu);
        c->pins.emplace_back(p, bytes);
        if (c->pins.size() <= 8) return;
        p = c->pins.front().first;
        c->pins.erase(c->pins.begin());
    }
    hipHostFree(p);
}

// Copies host memory to the device while the caller goes on (start ... finish,
// which waits for the copy).  The runtime's copy of pageable memory moves it
// through one staging buffer at 26 GB/s; here kThreads threads fill page-locked
// chunks, each kSlots of its own in turn, and a stream of their own sends them
// (the copies then go through the DMA engine at 50 GB/s while the context's
// stream makes the records).  Whole loads of 36, 108 and 216 MB: 2.16, 6.20 and
// 12.8 ms before, 1.12, 2.86 and 5.47 ms now; chunks of 2 MB 7% slower, of 1 MB
// 20%; four threads the same as two.  Below kMin, where the threads' start costs
// what they save, the caller's thread fills one buffer (the runtime page-locks
// small memory for its copy, 50 to 190 us for 360 KB: the load 310 us with that,
// 180 without).  Memory that the runtime knows (page-locked, managed, a device's)
// travels from where it is, on that stream too (36 MB and the rest of the load
// 820 us, 1,180 with a copy on the null stream behind the records).
namespace {
class Upload {
  public:
    ~Upload() { finish(); }
    void start(hb_ctx *c, void *dst, const void *src, size_t bytes)
    {
        c_ = c;
        dst_ = static_cast<char *>(dst);
        src_ = static_cast<const char *>(src);
        bytes_ = bytes;
        if (bytes && !start_own()) e_ = hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
    }
    int finish()
    {
        if (!c_) return HB_OK;
        hipError_t e = e_;
        for (auto &t : th_) t.join();
        th_.clear();
        if (own_) {
            e = hipStreamSynchronize(c_->up_stream);
            if (failed_) e = hipErrorUnknown;
        }
        hb_pin_put(c_, pin_, pin_bytes_);
        pin_ = nullptr;
        c_ = nullptr;
        if (e == hipSuccess) return HB_OK;
        hb_note_hip_error(e, "upload", __LINE__);
        return HB_ERR_DEVICE;
    }

  private:
    static constexpr size_t kThreads = 2, kSlots = 2, kChunk = (size_t)4 << 20;
    static constexpr size_t kMin = (size_t)4 << 20;
    // Starts the copy on the stream of its own; false if there is nothing to start
    // that for, or no way to.
    bool start_own()
    {
        hipPointerAttribute_t at{};
        bool known = false;
        if (hipPointerGetAttributes(&at, src_) != hipSuccess) (void)hipGetLastError();
        else known = at.type != hipMemoryTypeUnregistered;
        if (!c_->up_stream &&
            hipStreamCreateWithFlags(&c_->up_stream, hipStreamNonBlocking) != hipSuccess) {
            (void)hipGetLastError();
            c_->up_stream = nullptr;
            return false;
        }
        auto send = [&](const void *from) {
            own_ = hipMemcpyAsync(dst_, from, bytes_, hipMemcpyHostToDevice, c_->up_stream) ==
                   hipSuccess;
            if (!own_) (void)hipGetLastError();
            return own_;
        };
        if (known) return send(src_);
        pin_bytes_ = bytes_ < kMin ? bytes_ : kThreads * kSlots * kChunk;
        pin_ = static_cast<char *>(hb_pin_get(c_, &pin_bytes_));
        if (!pin_) return false;
        if (bytes_ < kMin) {
            memcpy(pin_, src_, bytes_);
            return send(pin_);
        }
        try {
            th_.reserve(kThreads);
            for (size_t t = 0; t < kThreads; ++t) th_.emplace_back([this, t] { work(t); });
        } catch (...) {   // the threads that there are do all of it
        }
        own_ = !th_.empty();
        return own_;
    }
    // Start of chunk i: two of each size from an eighth of kChunk up, so that
    // the link need not wait for a full chunk to be filled.
    static size_t chunk_at(size_t i)
    {
        constexpr size_t kEighths[7] = {0, 1, 2, 4, 6, 10, 14};   // eighths of kChunk
        return i < 7 ? kEighths[i] * (kChunk / 8) : kEighths[6] * (kChunk / 8) + (i - 6) * kChunk;
    }
    void work(size_t t)
    {
        hipEvent_t ev[kSlots] = {};
        bool ok = hipSetDevice(c_->device) == hipSuccess;
        for (hipEvent_t &e : ev)
            ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        for (size_t k = 0; ok && !failed_; ++k) {
            const size_t i = next_++, s = k % kSlots, at = chunk_at(i);
            if (at >= bytes_) break;
            const size_t len = std::min(chunk_at(i + 1), bytes_) - at;
            char *buf = pin_ + (t * kSlots + s) * kChunk;
            if (k >= kSlots) ok = hipEventSynchronize(ev[s]) == hipSuccess;
            if (!ok) break;
            memcpy(buf, src_ + at, len);
            ok = hipMemcpyAsync(dst_ + at, buf, len, hipMemcpyHostToDevice, c_->up_stream) ==
                     hipSuccess &&
                 hipEventRecord(ev[s], c_->up_stream) == hipSuccess;
        }
        if (!ok) failed_ = true;
        for (hipEvent_t e : ev)
            if (e) hipEventDestroy(e);
    }
    hb_ctx *c_ = nullptr;
    char *dst_ = nullptr, *pin_ = nullptr;
    const char *src_ = nullptr;
    size_t bytes_ = 0, pin_bytes_ = 0;
    std::vector<std::thread> th_;
    std::atomic<size_t> next_{0};
    std::atomic<bool> failed_{false};
    bool own_ = false;            // the copy is on the stream of its own
    hipError_t e_ = hipSuccess;   // ... else it is done, with this
};
}  // namespace

// Copies between host buffers, on up to four threads of 1 MiB or more, and up to
// eight of 4 MiB: a search with 4.8 MB of counters and a gapped stage with 8 MB
// took 1,159 and 1,520 us with one thread, 1,090 and 1,468 with two, 1,089 and
// 1,437 with four, and the same with eight; 48 MB of counters into new arrays took
// 2.17 ms with four and 1.85 with eight.
static void host_copy(void *dst, const void *src, size_t bytes)
{
    constexpr size_t kPart = (size_t)1 << 20;
    const size_t few = std::min<size_t>(4, std::max<size_t>(1, bytes / kPart));
    const size_t nt = std::min<size_t>(8, std::max<size_t>(few, bytes / (4 * kPart)));
    const size_t per = (bytes + nt - 1) / nt;
    auto part = [&](size_t t) {
        const size_t b = t * per, e = std::min(bytes, b + per);
        if (b < e) memcpy(static_cast<char *>(dst) + b, static_cast<const char *>(src) + b, e - b);
    };
    std::vector<std::thread> th;
    size_t t = 1;
    try {
        th.reserve(nt);
        for (; t < nt; ++t) th.emplace_back(part, t);
    } catch (...) {   // the rest is done here
    }
    part(0);
    for (; t < nt; ++t) part(t);
    for (auto &x : th) x.join();
}

// Copies of device memory to pageable host memory through page-locked memory:
// add() enqueues one, wait() waits for all, store() moves one on.  Up to kOwn
// bytes go through a buffer of their own, so that a call whose kernels are still
// running holds up no other thread's results; more through the context's (of at
// least kKeep), which is held while this lives.
namespace {
class CopyOut {
  public:
    CopyOut(hb_ctx *c, size_t bytes, hipStream_t st) : c_(c), st_(st)
    {
        bytes = std::max(room(bytes), (size_t)64);
        if (bytes <= kOwn) {
            cap_ = bytes;
            base_ = own_ = static_cast<char *>(hb_pin_get(c, &cap_));
            if (!own_) e_ = hipErrorOutOfMemory;
            return;
        }
        lk_ = std::unique_lock<std::mutex>(c->pinned_mu);
        bytes = std::max(bytes, kKeep);
        if (c->pinned_bytes < bytes) {
            if (c->pinned) hipHostFree(c->pinned);
            c->pinned = nullptr;
            c->pinned_bytes = 0;
            e_ = hipHostMalloc(&c->pinned, bytes, hipHostMallocDefault);
            if (e_ == hipSuccess) {
                c->pinned_bytes = bytes;
            } else {
                (void)hipGetLastError();
                c->pinned = nullptr;
            }
        }
        base_ = static_cast<char *>(c->pinned);
        cap_ = c->pinned_bytes;
    }
    ~CopyOut()
    {
        if (pending_) hipStreamSynchronize(st_);
        hb_pin_put(c_, own_, cap_);
    }
    CopyOut(const CopyOut &) = delete;
    CopyOut &operator=(const CopyOut &) = delete;
    static constexpr size_t kKeep = (size_t)64 << 20, kOwn = (size_t)16 << 20;
    static size_t room(size_t bytes) { return (bytes + 63) & ~(size_t)63; }
    bool fits(size_t bytes) const { return at_ + room(bytes) <= cap_; }
    size_t add(const void *src, size_t bytes)
    {
        const size_t at = at_;
        if (e_ == hipSuccess && !fits(bytes)) e_ = hipErrorInvalidValue;
        at_ += room(bytes);
        if (e_ == hipSuccess && bytes) {
            e_ = hipMemcpyAsync(ptr(at), src, bytes, hipMemcpyDeviceToHost, st_);
            pending_ = true;
        }
        return at;
    }
    void rewind() { at_ = 0; }   // after a wait: what was copied is no longer needed
    hipError_t wait()
    {
        if (e_ == hipSuccess) e_ = hipStreamSynchronize(st_);
        if (e_ == hipSuccess) pending_ = false;
        return e_;
    }
    char *ptr(size_t at) const { return base_ + at; }
    void store(void *dst, size_t at, size_t bytes) const { host_copy(dst, ptr(at), bytes); }

  private:
    hb_ctx *c_;
    hipStream_t st_;
    std::unique_lock<std::mutex> lk_;
    char *own_ = nullptr, *base_ = nullptr;
    size_t cap_ = 0, at_ = 0;
    bool pending_ = false;
    hipError_t e_ = hipSuccess;
};
}  // namespace

int hb_copy_out(hb_ctx *c, void *dst, const void *src, size_t bytes, hipStream_t st)
{
    if (bytes == 0) return HB_OK;
    CopyOut out(c, bytes, st);
    out.add(src, bytes);
    HB_CHECK(out.wait());
    out.store(dst, 0, bytes);
    return HB_OK;
}

int hb_resolve_params(const hb_params *pp, hb_resolved_params *out)
{
    hb_params p;
    hb_params_default(&p);
    if (pp) p = *pp;
    if (p.word_size != 3) return HB_ERR_UNSUPPORTED;
    // queued extensions pack the query offset in 24 bits and s - last_hit
    // (< window) in 8 bits
    if (p.window <= 3) return HB_ERR_ARG;
    if (p.window > 255) return HB_ERR_UNSUPPORTED;
    out->threshold = p.threshold;
    out->window = p.window;
    for (int i = 0; i < 32; ++i)
        for (int j = 0; j < 32; ++j)
            out->mat32[i * 32 + j] =
                (i < HB_ALPHA && j < HB_ALPHA)
                    ? (p.matrix ? p.matrix[i * HB_ALPHA + j] : kHbBlosum62[i][j])
                    : (int8_t)-128;
    return HB_OK;
}

int hb_check_query(const uint8_t *seq, int32_t len, int32_t n_ctx, const int32_t *ctx_off,
                   const int32_t *ctx_len, const int32_t *xdrop)
{
    if (!seq || len <= 0 || n_ctx <= 0 || !ctx_off || !ctx_len || !xdrop) return HB_ERR_ARG;
    if (len >= (1 << 24)) return HB_ERR_UNSUPPORTED;
    for (int32_t i = 0; i < len; ++i)
        if (seq[i] >= HB_ALPHA) return HB_ERR_RESIDUE;
    int32_t prev_end = 0;
    for (int32_t k = 0; k < n_ctx; ++k) {
        if (ctx_len[k] < 0 || ctx_off[k] < prev_end || ctx_off[k] + ctx_len[k] > len ||
            xdrop[k] <= 0)
            return HB_ERR_ARG;
        prev_end = ctx_off[k] + ctx_len[k];
    }
    return HB_OK;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

void hb_group_set_free(hb_group_set *g)
{
    if (!g || !g->ctx) return;
    hb_pool_put(g->ctx, g->d_fixed);
    hb_pool_put(g->ctx, g->d_entries);
    g->d_desc = nullptr;
    g->d_fixed = nullptr;
    g->d_entries = nullptr;
    g->d_mat = nullptr;
}

// Lookup tables of all groups are built together: one upload of the inputs,
// count pass, fill pass, one read-back of the totals.  The entries get room
// for kEntriesPerWord of each query word (BLOSUM62 at threshold 11 gives 30
// on average); tables that turn out larger are filled again with the room
// they need.
static constexpr size_t kEntriesPerWord = 64;

int hb_group_set_build(hb_ctx *c, const std::vector<hb_concat> &qs,
                       const std::vector<int32_t> &ctx_base, const hb_resolved_params &p,
                       bool multi, hipStream_t st, hb_group_set *out)
{
    const size_t n = qs.size();
    if (n == 0 || ctx_base.size() != n) return HB_ERR_ARG;
    out->ctx = c;
    out->desc.assign(n, hb_group_desc{});
    // d_fixed: the groups' tables, the uploaded inputs (score matrix, jobs,
    // descriptors, then each group's query, contexts and words), the totals
    // (a job and its tables per class of a group's diagonals)
    const size_t cells_b = HB_NCELLS * sizeof(uint2), pv_b = HB_PV_WORDS * sizeof(uint32_t);
    const size_t table_b = cells_b + pv_b + HB_NPAIRS * sizeof(uint32_t);
    std::vector<int32_t> shift(n);
    size_t nj = 0;
    for (size_t g = 0; g < n; ++g) {
        shift[g] = hb_diag_shift(c, multi, (int32_t)qs[g].seq.size(),
                                 (int32_t)qs[g].ctx_off.size(), p.window);
        nj += (size_t)1 << shift[g];
    }
    const size_t o_jobs = 1024, o_desc = o_jobs + align256(nj * sizeof(hb_lut_job));
    const size_t o_groups = o_desc + align256(n * sizeof(hb_group_desc));
    auto query_b = [&](size_t g) { return align256((qs[g].seq.size() + 15) & ~(size_t)15); };
    auto ctx_b = [&](size_t g) { return align256(3 * qs[g].ctx_off.size() * sizeof(int32_t)); };
    // words and entries of one class
    auto class_words = [&](size_t g) {
        return (qs[g].seq.size() + ((size_t)1 << shift[g]) - 1) >> shift[g];
    };
    auto n_words = [&](size_t g) { return (class_words(g) + 255) & ~(size_t)255; };
    size_t in_b = o_groups, ent_cap = 0;
    for (size_t g = 0; g < n; ++g) {
        const int32_t qlen = (int32_t)qs[g].seq.size();
        in_b += query_b(g) + ctx_b(g) + (n_words(g) * sizeof(uint16_t) << shift[g]);
        ent_cap += kEntriesPerWord * class_words(g) << shift[g];
        out->qlen_pad_max = std::max(out->qlen_pad_max, (qlen + 15) & ~15);
        out->ctx_pad_max = std::max(out->ctx_pad_max, hb_ctx_pad((int32_t)qs[g].ctx_off.size()));
        out->diag_len_max = std::max(out->diag_len_max, hb_diag_len(qlen, p.window, shift[g]));
        out->split |= shift[g] > 0;
    }
    const size_t in_o = nj * table_b, tot_o = in_o + in_b, tot_b = 2 * nj * sizeof(uint32_t);
    out->fixed_bytes = tot_o + align256(tot_b);
    out->entries_bytes = ent_cap * sizeof(uint32_t);
    size_t pin_b = in_b + tot_b;
    uint8_t *pin = static_cast<uint8_t *>(hb_pin_get(c, &pin_b));
    out->d_fixed = hb_pool_get(c, out->fixed_bytes);
    out->d_entries = static_cast<uint32_t *>(hb_pool_get(c, out->entries_bytes));
    auto done = [&](int rc) {
        if (rc) {
            hipStreamSynchronize(st);
            hb_group_set_free(out);
        }
        hb_pin_put(c, pin, pin_b);
        return rc;
    };
    if (!pin || !out->d_fixed || !out->d_entries) return done(HB_ERR_NOMEM);
    uint8_t *base = static_cast<uint8_t *>(out->d_fixed), *in = base + in_o;
    out->d_mat = reinterpret_cast<int8_t *>(in);
    out->d_desc = reinterpret_cast<hb_group_desc *>(in + o_desc);
    hb_lut_job *jobs = reinterpret_cast<hb_lut_job *>(pin + o_jobs);
    const hb_lut_job *d_jobs = reinterpret_cast<const hb_lut_job *>(in + o_jobs);
    uint32_t *totals = reinterpret_cast<uint32_t *>(pin + in_b);
    memset(pin, 0, in_b);
    memcpy(pin, p.mat32, 1024);
    size_t o = o_groups, e = 0, j = 0;
    for (size_t g = 0; g < n; ++g) {
        const hb_concat &Q = qs[g];
        const int32_t qlen = (int32_t)Q.seq.size();
        const int32_t nctx = (int32_t)Q.ctx_off.size();
        const size_t q_o = o, c_o = q_o + query_b(g), w_o = c_o + ctx_b(g);
        const uint32_t sh = (uint32_t)shift[g], nc = 1u << sh;
        const size_t nw = n_words(g);
        o = w_o + nw * nc * sizeof(uint16_t);
        memcpy(pin + q_o, Q.seq.data(), (size_t)qlen);
        int32_t *cimg = reinterpret_cast<int32_t *>(pin + c_o);
        uint16_t *words = reinterpret_cast<uint16_t *>(pin + w_o);
        for (int32_t k = 0; k < nctx; ++k) {
            cimg[k] = Q.ctx_off[k];
            cimg[nctx + k] = Q.xdrop[k];
            cimg[2 * nctx + k] = Q.cutoff[k];
            // masked residues seed no word (NCBI builds its table over the
            // unmasked segments only)
            for (int32_t w = Q.ctx_off[k]; w + 3 <= Q.ctx_off[k] + Q.ctx_len[k]; ++w)
                if (Q.mask.empty() || !(Q.mask[w] | Q.mask[w + 1] | Q.mask[w + 2]))
                    words[(w & (nc - 1)) * nw + (w >> sh)] =
                        (uint16_t)(0x8000u | Q.seq[w] | Q.seq[w + 1] << 5 | Q.seq[w + 2] << 10);
        }
        uint8_t *t = base + j * table_b;   // nc classes' cells, presence bits, pair sums
        hb_group_desc &D = out->desc[g];
        D.cells = reinterpret_cast<uint2 *>(t);
        D.pv = reinterpret_cast<uint32_t *>(t + nc * cells_b);
        D.entries = out->d_entries + e;
        D.query = in + q_o;
        D.ctx = reinterpret_cast<const int32_t *>(in + c_o);
        D.qlen = qlen;
        D.qlen_pad = (qlen + 15) & ~15;
        D.n_ctx = nctx;
        D.diag_len = hb_diag_len(qlen, p.window, shift[g]);
        D.ctx_base = ctx_base[g];
        D.shift = shift[g];
        const uint32_t cap = (uint32_t)(kEntriesPerWord * class_words(g));
        for (uint32_t k = 0; k < nc; ++k, ++j) {
            hb_lut_job &J = jobs[j];
            J.words = reinterpret_cast<const uint16_t *>(in + w_o) + k * nw;
            J.n_words = (uint32_t)nw;
            J.first = k * cap;
            J.cap = cap;
            J.shift = sh;
            J.cls = k;
            J.entries = out->d_entries + e;
            J.cells = reinterpret_cast<uint2 *>(t) + k;
            J.pv = reinterpret_cast<uint32_t *>(t + nc * cells_b + k * pv_b);
            J.pair_sum = reinterpret_cast<uint32_t *>(t + nc * (cells_b + pv_b)) + k * HB_NPAIRS;
            J.out = reinterpret_cast<uint32_t *>(base + tot_o) + 2 * j;
        }
        e += (size_t)cap * nc;
    }
    memcpy(pin + o_desc, out->desc.data(), n * sizeof(hb_group_desc));
    auto upload_fill = [&](bool count) {
        return hipMemcpyAsync(in, pin, in_b, hipMemcpyHostToDevice, st) == hipSuccess &&
               (!count || hb_launch_lut(d_jobs, (int)nj, out->d_mat, p.threshold, false, st) ==
                              hipSuccess) &&
               hb_launch_lut(d_jobs, (int)nj, out->d_mat, p.threshold, true, st) == hipSuccess &&
               hipMemcpyAsync(totals, base + tot_o, tot_b, hipMemcpyDeviceToHost, st) ==
                   hipSuccess &&
               hipStreamSynchronize(st) == hipSuccess;
    };
    if (!upload_fill(true)) return done(HB_ERR_DEVICE);
    out->n_entries.assign(n, 0);
    out->n_cells_used.resize(n);
    bool fits = true;
    size_t need = 0;
    j = 0;
    for (size_t g = 0; g < n; ++g) {
        out->n_cells_used[g] = totals[2 * j + 1];
        for (size_t k = 0; k < (size_t)1 << shift[g]; ++k, ++j) {
            out->n_entries[g] += totals[2 * j];
            fits &= totals[2 * j] <= jobs[j].cap;
        }
        need += out->n_entries[g];
    }
    if (!fits) {
        hb_pool_put(c, out->d_entries);
        out->entries_bytes = need * sizeof(uint32_t);
        out->d_entries = static_cast<uint32_t *>(hb_pool_get(c, out->entries_bytes));
        if (!out->d_entries) return done(HB_ERR_NOMEM);
        e = j = 0;
        for (size_t g = 0; g < n; ++g) {
            out->desc[g].entries = out->d_entries + e;
            uint32_t first = 0;
            for (size_t k = 0; k < (size_t)1 << shift[g]; ++k, ++j) {
                jobs[j].entries = out->d_entries + e;
                jobs[j].first = first;
                jobs[j].cap = totals[2 * j];
                first += totals[2 * j];
            }
            e += first;
        }
        memcpy(pin + o_desc, out->desc.data(), n * sizeof(hb_group_desc));
        if (!upload_fill(false)) return done(HB_ERR_DEVICE);
    }
    return done(HB_OK);
}

// Picks wavefronts per workgroup and the staging ring size: the most
// wavefronts per CU up to 16 first (measured on C1: 8 -> 12 -> 16 wavefronts
// per CU gave 27.7 -> 20.6 -> 16.8 ms; beyond 16 the kernel is bound by
// VALU issue and more wavefronts gained nothing), then the largest ring
// (subjects above it read their residues from global memory, and a larger
// ring holds the extensions of more subjects before they must run), then
// more wavefronts per workgroup (they share the query tables).  The batched
// form stages at most 2048 residues per wave: its largest class of C3
// queries lost a workgroup per CU to larger staging.
int hb_scan_config(hb_ctx *c, bool multi, bool split, int32_t qlen_pad_max, int32_t ctx_pad_max,
                   int32_t diag_len_max, uint32_t work_items, hb_launch_cfg *cfg, int place,
                   int32_t ring_cap, int32_t force_waves)
{
    const size_t fixed = hb_scan_fixed_lds(qlen_pad_max, ctx_pad_max);
    const bool gstate = place == HB_PLACE_GLOBAL;
    const int sb = hb_state_bytes(place);
    int32_t ring_top = multi ? std::min(HB_RING_MAX, 2048) : HB_RING_MAX;
    if (ring_cap > 0) ring_top = std::min(ring_top, ring_cap & ~63);
    int best_wpc = 0;
    for (int waves : {16, 8, 4, 2, 1}) {
        if (force_waves > 0 && waves != force_waves) continue;
        if (waves * HB_WAVE > hb_block_max(multi, split, gstate)) continue;
        for (int32_t ring = ring_top; ring >= 256; ring -= 64) {
            const size_t lds = fixed + waves * hb_scan_wave_lds(diag_len_max, ring, sb);
            if (lds > c->max_lds) continue;
            // no better than the best so far, as many as its LDS would let in (up
            // to 180 questions to the runtime for each scan otherwise)
            const int most = (int)std::min<size_t>(c->max_lds / lds * waves, 16);
            if (most < best_wpc || (most == best_wpc && ring <= cfg->ring)) continue;
            int per_cu = 0;
            HB_CHECK(hb_scan_occupancy(multi, gstate, split, lds, waves * HB_WAVE, &per_cu));
            const int wpc = std::min(per_cu * waves, 16);
            if (wpc > best_wpc || (wpc == best_wpc && ring > cfg->ring)) {
                best_wpc = wpc;
                cfg->waves = waves;
                cfg->lds = lds;
                cfg->ring = ring;
                cfg->blocks = per_cu;
            }
        }
    }
    if (best_wpc == 0) return HB_ERR_UNSUPPORTED;
    int blocks = c->n_cu * std::max(cfg->blocks, 1);
    if (gstate) {   // keep the global-memory state within HB_GSTATE_MAX_BYTES
        const size_t per_block = HB_GSTATE_WORD * (size_t)diag_len_max * (size_t)cfg->waves;
        blocks = std::min(blocks, (int)std::max<size_t>(1, HB_GSTATE_MAX_BYTES / per_block));
    }
    const uint32_t per_block = (uint32_t)cfg->waves;
    const int need = (int)((work_items + per_block - 1) / per_block);
    if (need < blocks) blocks = std::max(need, 1);
    cfg->blocks = blocks;
    return HB_OK;
}

// Automatic placement of the diagonal state.  LDS words beat the
// global-memory words (ordering markers in an LDS table, one load and one
// store per hit) down to about kGstateMinWaves wavefronts per CU (measured
// on 200,000 subjects, ms LDS / global: 1,000 residues 1.61 / 1.84, 8,000 at
// 4 wavefronts per CU 23.7 / 27.6, 12,000 at 3 64.7 / 39.0, 31,000 at 1
// 320 / 114).
static constexpr int kGstateMinWaves = 4;
static int lds_waves(const hb_ctx *c, int32_t D, size_t fixed, int state_bytes)
{
    const size_t per_wave = hb_scan_wave_lds(D, 256, state_bytes);
    if (fixed + per_wave > c->max_lds) return 0;
    // waves of one workgroup share the fixed part; up to 4 per workgroup
    return (int)std::min<size_t>((c->max_lds - fixed) / per_wave, 16);
}

int hb_state_choose(const hb_ctx *c, int32_t D, size_t fixed, uint64_t max_len, int32_t window)
{
    if (hb_state_lds_ok(max_len, window) && lds_waves(c, D, fixed, 4) >= kGstateMinWaves)
        return HB_PLACE_LDS;
    return HB_PLACE_GLOBAL;
}

// The fewest classes with which 16 wavefronts per CU (workgroups of 4, or one
// of 16 for a plain scan of several classes) have LDS for their diagonals and
// a ring of kSplitRing residues.  A class scans the windows of every subject
// again, so more classes than that cost: G hits/s of a plain scan with 1, 2,
// 4, .. classes, 1,500 residues 130, 122, 89; 2,000 89, 135, 104; 3,000 101,
// 145, 122; 6,000 55, 101, 138, 121; 8,001 56, 95, 76, 135, 103; 12,000 (one
// class: state in global memory) 45, ., 100, 132, 120; 24,000 41, .., 100, 89,
// 117.  Queries whose diagonals no LDS layout holds at once keep one class in
// global memory.
static constexpr int32_t kSplitRing = 512;
int32_t hb_diag_shift(const hb_ctx *c, bool multi, int32_t qlen, int32_t n_ctx, int32_t window)
{
    const size_t fixed = hb_scan_fixed_lds((qlen + 15) & ~15, hb_ctx_pad(n_ctx));
    if (fixed + hb_scan_wave_lds(hb_diag_len(qlen, window, 0), 256, 4) > c->max_lds) return 0;
    int32_t shift = 0;
    while (shift < HB_SHIFT_MAX &&
           (shift && !multi ? 1 : 4) * fixed +
                   16 * hb_scan_wave_lds(hb_diag_len(qlen, window, shift), kSplitRing, 4) >
               c->max_lds)
        ++shift;
    return shift;
}

bool hb_query_lds_ok(const hb_ctx *c, int32_t qlen, int32_t n_ctx)
{
    const size_t qpad = (size_t)((qlen + 15) & ~15);
    const size_t fixed = hb_scan_fixed_lds((int32_t)qpad, hb_ctx_pad(n_ctx));
    return fixed + hb_scan_wave_lds(0, 256, 0) <= c->max_lds;
}

size_t hb_gstate_bytes_max(const hb_ctx *c, int32_t D)
{
    const size_t full = (size_t)c->n_cu * 16 * HB_GSTATE_WORD * (size_t)D;   // 16 wavefronts per CU
    return std::min(full, std::max(HB_GSTATE_MAX_BYTES, 4 * HB_GSTATE_WORD * (size_t)D));
}

// Dynamic LDS of a workgroup of which five fit a CU: 25 steps of 1,280 bytes,
// less the kernel's own variables.
static constexpr size_t kShortLds = 25 * 1280 - 16;

struct hb_query {
    hb_ctx *ctx = nullptr;
    hb_resolved_params p;
    hb_group_set gs;
    std::vector<int32_t> ctx_off, ctx_len;   // host copies (gapped stage)
    int mode = HB_STATE_AUTO;   // requested placement of the diagonal state
    bool lds_fits = true;       // the LDS layout can hold the diagonal words
    int32_t reset_interval = 0; // hb_query_set_reset_interval (0: the placement's limit)
};

struct hb_scan {
    hb_ctx *ctx = nullptr;
    hb_db *db = nullptr;
    hb_query *q = nullptr;
    hb_hsp *d_out = nullptr;
    uint32_t cap = 0;
    uint32_t *d_misc = nullptr;   // HSP count in its own line, then the tile queues
    uint32_t *d_stats = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    bool waited = false;
    uint32_t n_out = 0;
    float gap_ms = 0.f;        // device time of the last gapped stage
    uint32_t gap_wide = 0;     // subjects it ran in the wide pass
    uint32_t *d_gstate = nullptr;   // per-wavefront diagonal words (long queries)
    int place = HB_PLACE_LDS;      // where this scan keeps the diagonal state
};

// ------------------------------------------------------------------ no-alloc scan
// Scratch of hb_scan_noalloc, one copy per GPU, held until the process ends:
// the scan's HSP cursor and tile queues (HB_NOALLOC_HEAD bytes), then the
// diagonal words of a query whose state lives in global memory.  Host code
// uses the device address hipGetSymbolAddress returns (hb_ctx::scratch_dev),
// never the array's name.
#define HB_SCAN_MISC_WORDS (HB_QUEUE_STRIDE + HB_QUEUE_WORDS)
#define HB_NOALLOC_HEAD (HB_SCAN_MISC_WORDS * 4)
static __device__ __align__(256) unsigned char scratch[HB_NOALLOC_HEAD + HB_NOALLOC_STATE_BYTES];
static std::mutex g_scratch_mu;
static unsigned char *g_scratch_dev[256];   // per device

// The device address of this GPU's scratch (the device is current).
static int scratch_address(int device, unsigned char **out)
{
    if (device < 0 || device >= 256) return HB_ERR_ARG;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[device]) {
        void *p = nullptr;
        HB_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_dev[device] = static_cast<unsigned char *>(p);
    }
    *out = g_scratch_dev[device];
    return HB_OK;
}


extern "C" {

const char *hb_strerror(int err)
{
    switch (err) {
    case HB_OK: return "ok";
    case HB_ERR_ARG: return "invalid argument";
    case HB_ERR_NOMEM: return "out of memory";
    case HB_ERR_DEVICE: return g_last_hip[0] ? g_last_hip : "HIP runtime error";
    case HB_ERR_CAPACITY: return "output array too small";
    case HB_ERR_RESIDUE: return "residue code >= 28";
    case HB_ERR_STATE: return "handle in wrong state";
    case HB_ERR_UNSUPPORTED: return "unsupported parameters";
    case HB_ERR_BUSY: return "busy";
    case HB_ERR_FORMAT: return "malformed .hDb volume or .hDbI index";
    default: return "unknown error";
    }
}

const int8_t *hb_blosum62(void) { return &kHbBlosum62[0][0]; }

void hb_params_default(hb_params *p)
{
    if (!p) return;
    p->word_size = 3;
    p->threshold = 11;
    p->window = 40;
    p->matrix = nullptr;
}

int hb_create(int device, hb_ctx **out)
{
    if (!out) return HB_ERR_ARG;
    *out = nullptr;
    int n = 0;
    HB_CHECK(hipGetDeviceCount(&n));
    if (device < 0 || device >= n) return HB_ERR_ARG;
    HB_CHECK(hipSetDevice(device));
    hb_ctx *c = new (std::nothrow) hb_ctx;
    if (!c) return HB_ERR_NOMEM;
    c->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess ||
        hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return HB_ERR_DEVICE;
    }
    c->n_cu = prop.multiProcessorCount;
    c->max_lds = prop.sharedMemPerBlock;
    int lds_optin = 0;
    if (hipDeviceGetAttribute(&lds_optin, hipDeviceAttributeSharedMemPerBlockOptin, device) ==
            hipSuccess && (size_t)lds_optin > c->max_lds)
        c->max_lds = (size_t)lds_optin;
    // one dynamic-LDS limit for every launch of the scan kernels, so that
    // launches of different sizes on different streams never disagree; the
    // no-alloc scan's scratch address of this device
    int five = 0;
    if (hb_scan_allow_lds(c->max_lds) != hipSuccess ||
        hb_scan_short_occupancy(kShortLds, &five) != hipSuccess ||
        scratch_address(device, &c->scratch_dev) != HB_OK) {
        hipStreamDestroy(c->stream);
        delete c;
        return HB_ERR_DEVICE;
    }
    c->short_scan = five >= 5;
    std::lock_guard<std::mutex> lk(g_ctx_mu);
    g_ctxs.push_back(c);
    *out = c;
    return HB_OK;
}

int hb_destroy(hb_ctx *c)
{
    if (!c) return HB_ERR_ARG;
    hipSetDevice(c->device);
    {
        std::lock_guard<std::mutex> lk(g_ctx_mu);
        g_ctxs.erase(std::remove(g_ctxs.begin(), g_ctxs.end(), c), g_ctxs.end());
    }
    if (c->stream) hipStreamSynchronize(c->stream);
    for (auto &b : c->pool) hipFree(b.p);
    if (c->pinned) hipHostFree(c->pinned);
    for (auto &b : c->pins) hipHostFree(b.first);
    if (c->stream) hipStreamDestroy(c->stream);
    if (c->up_stream) hipStreamDestroy(c->up_stream);
    delete c;
    return HB_OK;
}

int hb_mem_info(hb_ctx *c, uint64_t *free_b, uint64_t *total_b)
{
    if (!c) return HB_ERR_ARG;
    size_t f = 0, t = 0;
    HB_CHECK(hipSetDevice(c->device));
    HB_CHECK(hipMemGetInfo(&f, &t));
    if (free_b) *free_b = f + hb_pool_held(c);
    if (total_b) *total_b = t;
    return HB_OK;
}

int hb_host_alloc(hb_ctx *c, uint64_t bytes, void **out)
{
    if (!c || !out) return HB_ERR_ARG;
    *out = nullptr;
    HB_CHECK(hipSetDevice(c->device));
    if (hipHostMalloc(out, std::max<uint64_t>(bytes, 1), hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        *out = nullptr;
        return HB_ERR_NOMEM;
    }
    return HB_OK;
}

int hb_host_free(hb_ctx *c, void *p)
{
    if (!c) return HB_ERR_ARG;
    if (!p) return HB_OK;
    HB_CHECK(hipSetDevice(c->device));
    HB_CHECK(hipHostFree(p));
    return HB_OK;
}

int hb_synchronize(hb_ctx *c)
{
    if (!c) return HB_ERR_ARG;
    HB_CHECK(hipSetDevice(c->device));
    HB_CHECK(hipStreamSynchronize(c->stream));
    return HB_OK;
}

// ------------------------------------------------------------------ database
// (Also after the database's context was destroyed: its memory then goes back to
// the device.)
int hb_db_free(hb_db *db)
{
    if (!db) return HB_ERR_ARG;
    hipSetDevice(db->device);
    hipDeviceSynchronize();   // work that reads it, on any stream
    {
        std::lock_guard<std::mutex> lk(g_ctx_mu);
        const bool kept = std::find(g_ctxs.begin(), g_ctxs.end(), db->ctx) != g_ctxs.end();
        for (void *p : {db->load_scratch, (void *)db->d_res, (void *)db->d_offs, (void *)db->d_subj,
                        (void *)db->d_scan_alloc, (void *)db->d_tiles})
            if (kept) db_put(db->ctx, p);
            else hipFree(p);
        if (kept) hb_pin_put(db->ctx, db->load_pin, db->load_pin_bytes);
        else hipHostFree(db->load_pin);
    }
    delete db;
    return HB_OK;
}

// Tiles: runs of subjects in processing order that are handed out together,
// at most 64 subjects and about kTileMax residues.
// A batched launch's workgroups take tiles of one size, at least two for
// every wavefront of a full grid where the database has the subjects for it
// (four subjects or more: a workgroup's wavefronts share them).
// A plain scan's wavefronts pop tiles that shrink with what is left to do, a
// quarter of a wavefront's share of it, down to a sixteenth of its share of
// the whole database: with tiles of 16K residues throughout, 1,000 subjects
// kept 22 wavefronts of 4,096 busy (scan of a 60-residue query 334 us, 40 us
// now), 20,000 subjects 500 (350 residues: 526 us, 230 us now) and 200,000
// subjects ran 1.2 rounds of tiles (960 us, 700 us now).  Tiles of 64
// residues gained nothing over 256 on 200,000 subjects and more, and a
// single queue took 10 ns for each pop of every wavefront of the chip, which
// at one subject a tile made 200,000 subjects slower than 16K tiles did.
static constexpr uint64_t kTileMax = 16384, kQueueTileMin = 256;

// The database's lengths, longest first, as runs of equal ones.
static std::vector<std::pair<uint64_t, uint32_t>> length_runs(const hb_db *db)
{
    // (as many counters as there are lengths, so that a few short subjects do
    // not cost 65,536 of them; subjects past those are few: sorted)
    const uint64_t kCounted = std::min<uint64_t>(1 << 16, db->max_len + 1);
    std::vector<uint32_t> cnt(kCounted, 0);
    std::vector<uint64_t> longer;
    const uint64_t *offs = db->h_offs.data();
    for (uint32_t i = 0; i < db->n; ++i) {
        const uint64_t len = offs[i + 1] - offs[i];
        if (len < kCounted) ++cnt[len];
        else longer.push_back(len);
    }
    std::sort(longer.begin(), longer.end(), std::greater<uint64_t>());
    std::vector<std::pair<uint64_t, uint32_t>> runs;
    for (uint64_t len : longer) {
        if (!runs.empty() && runs.back().first == len) ++runs.back().second;
        else runs.emplace_back(len, 1u);
    }
    for (uint64_t len = kCounted; len-- > 0;)
        if (cnt[len]) runs.emplace_back(len, cnt[len]);
    return runs;
}

// Appends tile boundaries (0 first) of subjects with these lengths: a tile ends
// at 64 subjects or at `want` residues (shrink: at a quarter of a wavefront's
// share of the residues after the tile before, between want_min and kTileMax).
static uint32_t cut_tiles(const std::vector<std::pair<uint64_t, uint32_t>> &runs, uint64_t total,
                          uint64_t waves, bool shrink, uint64_t want_min,
                          std::vector<uint32_t> *tiles)
{
    const size_t t0 = tiles->size();
    tiles->push_back(0);
    auto share = [&](uint64_t left) { return std::min(kTileMax, left / (4 * waves)); };
    uint64_t acc = 0, left = total, w = share(left);
    uint32_t at = 0, cnt = 0;
    for (const auto &r : runs)
        for (uint32_t m = r.second; m > 0;) {
            uint64_t k = 64 - cnt;
            if (r.first) k = std::min(k, w > acc ? (w - acc + r.first - 1) / r.first : 1);
            else if (acc >= w) k = 1;
            const uint32_t take = (uint32_t)std::min<uint64_t>(k, m);
            m -= take;
            at += take;
            cnt += take;
            acc += take * r.first;
            left -= take * r.first;
            if (cnt >= 64 || acc >= w) {
                tiles->push_back(at);
                acc = 0;
                cnt = 0;
                if (shrink) w = std::max(want_min, share(left));
            }
        }
    if (tiles->back() != at) tiles->push_back(at);
    return (uint32_t)(tiles->size() - t0) - 1;
}

// Tiles of a database whose host offsets and longest subject are set, and the device copies of
// offsets and tiles; then, enqueued on the context's stream, the records in
// processing order (length-descending: the longest subjects start first).
// The scan reads each subject's oid, length and offset from one 16-byte
// record in processing order (sequential), not offs[oid] (one scattered
// cache line per subject); the offset points into the scan's copy of the
// residues, laid out in the same order, so consecutive subjects share no cache
// line with subjects read at other times.
static int db_meta(hb_db *db)
{
    hb_ctx *c = db->ctx;
    const uint32_t n = db->n;
    const auto runs = length_runs(db);
    db->scan_bytes = 0;   // the scan stages subjects with 16-byte loads
    for (const auto &r : runs) db->scan_bytes += ((r.first + 15) & ~15ull) * r.second;
    const uint64_t waves = c->n_cu * 16ull;
    const uint64_t want_min = std::min(kQueueTileMin, db->total / (16 * waves));
    std::vector<uint32_t> tiles;
    db->n_tiles = cut_tiles(runs, db->total, waves, false, 0, &tiles);
    db->n_qtiles = cut_tiles(runs, db->total, waves, true, want_min, &tiles);
    if (!db_get(c, &db->d_offs, ((size_t)n + 1) * sizeof(uint64_t)) ||
        !db_get(c, &db->d_subj, (size_t)std::max<uint32_t>(n, 1) * sizeof(uint4)) ||
        !db_get(c, &db->d_tiles, tiles.size() * sizeof(uint32_t)))
        return HB_ERR_NOMEM;
    db->load_scratch = hb_pool_get(c, hb_load_scratch(n));   // until the stream is waited for
    if (!db->load_scratch) return HB_ERR_NOMEM;
    hb_load_args a{};
    a.offs = db->d_offs;
    a.n = n;
    a.max_len = db->max_len;
    a.subj = db->d_subj;
    // Small ones go through a page-locked buffer and are not waited for (each copy
    // of pageable memory is, 15 us).
    constexpr size_t kStage = (size_t)1 << 20;
    const size_t b_offs = ((size_t)n + 1) * sizeof(uint64_t);
    const size_t b_tiles = tiles.size() * sizeof(uint32_t);
    db->load_pin_bytes = b_offs + b_tiles;
    if (b_offs + b_tiles <= kStage) db->load_pin = hb_pin_get(c, &db->load_pin_bytes);
    bool ok;
    if (char *pin = static_cast<char *>(db->load_pin)) {
        memcpy(pin, db->h_offs.data(), b_offs);
        memcpy(pin + b_offs, tiles.data(), b_tiles);
        ok = hipMemcpyAsync(db->d_offs, pin, b_offs, hipMemcpyHostToDevice, c->stream) ==
                 hipSuccess &&
             hipMemcpyAsync(db->d_tiles, pin + b_offs, b_tiles, hipMemcpyHostToDevice,
                            c->stream) == hipSuccess;
    } else {
        ok = hipMemcpy(db->d_offs, db->h_offs.data(), b_offs, hipMemcpyHostToDevice) ==
                 hipSuccess &&
             hipMemcpy(db->d_tiles, tiles.data(), b_tiles, hipMemcpyHostToDevice) == hipSuccess;
    }
    if (!ok || hb_launch_load_records(a, db->load_scratch, c->stream) != hipSuccess)
        return HB_ERR_DEVICE;
    return HB_OK;
}

// The scan's copy of the residues in processing order (after d_res holds
// the database); HB_ERR_RESIDUE when one is not a residue code (< 28).
static int db_scan_copy(hb_db *db)
{
    hb_ctx *c = db->ctx;
    // the flag, then the copy; padding bytes after subjects read as 0 (the
    // staged copies hold them past each subject's end)
    constexpr size_t kHead = 256;
    if (!db_get(c, &db->d_scan_alloc, kHead + db->scan_bytes + 64))
        return HB_ERR_NOMEM;
    uint8_t *d = db->d_scan_alloc;
    db->d_scan_res = d + kHead;
    hb_load_args a{};
    a.res = db->d_res;
    a.offs = db->d_offs;
    a.n = db->n;
    a.subj = db->d_subj;
    a.out = db->d_scan_res;
    a.flag = reinterpret_cast<uint32_t *>(d);
    uint32_t flag = 0;
    if (hb_launch_fill_u32(a.flag, 0u, 1, c->stream) != hipSuccess ||
        hb_launch_fill_u32(reinterpret_cast<uint32_t *>(db->d_scan_res + db->scan_bytes), 0u, 16,
                           c->stream) != hipSuccess ||
        hb_launch_load_copy(a, db->scan_bytes, c->stream) != hipSuccess ||
        hipMemcpyAsync(&flag, a.flag, sizeof(flag), hipMemcpyDeviceToHost, c->stream) !=
            hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
        return HB_ERR_DEVICE;
    db_put(c, db->load_scratch);
    db->load_scratch = nullptr;
    hb_pin_put(c, db->load_pin, db->load_pin_bytes);
    db->load_pin = nullptr;
    return flag ? HB_ERR_RESIDUE : HB_OK;
}

int hb_db_upload(hb_ctx *c, const uint8_t *residues, const uint64_t *offsets, uint32_t n,
                 hb_db **out)
{
    if (!c || !offsets || !out || (n > 0 && !residues)) return HB_ERR_ARG;
    *out = nullptr;
    // subject lengths are int32 on the device and diagonal state keeps
    // position + offset below 2^31: cap a subject at 2^28 residues
    uint64_t longest = 0;
    for (uint32_t i = 0; i < n; ++i) {
        const uint64_t len = offsets[i + 1] - offsets[i];
        if (offsets[i + 1] < offsets[i] || len > (1ull << 28)) return HB_ERR_ARG;
        longest = std::max(longest, len);
    }
    std::lock_guard<std::mutex> lk(c->mu);
    HB_CHECK(hipSetDevice(c->device));
    hb_db *db = new (std::nothrow) hb_db;
    if (!db) return HB_ERR_NOMEM;
    db->ctx = c;
    db->device = c->device;
    db->n = n;
    db->max_len = longest;
    const uint64_t first = n ? offsets[0] : 0;
    db->total = n ? offsets[n] - first : 0;
    db->h_offs.resize((size_t)n + 1);
    for (uint32_t i = 0; i <= n; ++i) db->h_offs[i] = n ? offsets[i] - first : 0;
    auto fail = [&](int r) {
        hb_db_free(db);
        return r;
    };
    if (!db_get(c, &db->d_res, db->total + 64)) return fail(HB_ERR_NOMEM);
    // the records are made while the residues travel
    Upload up;
    up.start(c, db->d_res, residues ? residues + first : nullptr, db->total);
    int rc = db_meta(db);
    if (rc == HB_OK && hipMemsetAsync(db->d_res + db->total, 0, 64, c->stream) != hipSuccess)
        rc = HB_ERR_DEVICE;
    const int rc_up = up.finish();
    if (rc == HB_OK) rc = rc_up;
    if (rc == HB_OK) rc = db_scan_copy(db);
    if (rc != HB_OK) return fail(rc);
    *out = db;
    return HB_OK;
}

int hb_db_upload_hdb(hb_ctx *c, const uint8_t *hdb, uint64_t bytes, int32_t blocksx,
                     int32_t threadsx, int32_t n_seqs, const int32_t *group_len,
                     int32_t n_groups, hb_db **out)
{
    if (!c || !out || n_seqs < 0 || n_groups < 0 || blocksx < 1 || blocksx > 65536 ||
        threadsx < 1 || threadsx > 65536 || (n_groups > 0 && !group_len) || (bytes > 0 && !hdb))
        return HB_ERR_ARG;
    *out = nullptr;
    // the layout the volume must have (ncbi_blast_files/functions.cpp:844-911)
    const uint64_t T = (uint64_t)threadsx, G = (uint64_t)blocksx * T;
    if ((uint64_t)n_groups != ((uint64_t)n_seqs + G - 1) / G) return HB_ERR_FORMAT;
    std::vector<uint64_t> gbase((size_t)n_groups + 1, 0);
    uint64_t acc = 0;
    for (int32_t g = 0; g < n_groups; ++g) {
        const int32_t L = group_len[g];
        if (L < 0 || L % 16 || L > (1 << 28)) return HB_ERR_FORMAT;
        const uint64_t members = std::min<uint64_t>(G, (uint64_t)n_seqs - (uint64_t)g * G);
        gbase[g] = acc;
        acc += (members + T - 1) / T * T * (uint64_t)L;
    }
    if (acc != bytes) return HB_ERR_FORMAT;

    std::lock_guard<std::mutex> lk(c->mu);
    HB_CHECK(hipSetDevice(c->device));
    hb_db *db = new (std::nothrow) hb_db;
    if (!db) return HB_ERR_NOMEM;
    db->ctx = c;
    db->device = c->device;
    db->n = (uint32_t)n_seqs;
    uint8_t *d_hdb = nullptr;
    uint64_t *d_gbase = nullptr;
    int32_t *d_glen = nullptr;
    uint32_t *d_lens = nullptr, *d_bad = nullptr;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    auto release = [&]() {   // after a wait for the stream
        db_put(c, d_hdb);
        db_put(c, d_gbase);
        db_put(c, d_glen);
        db_put(c, d_lens);
        db_put(c, d_bad);
        for (hipEvent_t &e : ev)
            if (e) hipEventDestroy(e);
    };
    auto fail = [&](int r) {
        hipStreamSynchronize(c->stream);
        release();
        hb_db_free(db);
        return r;
    };
    for (hipEvent_t &e : ev)
        if (hipEventCreate(&e) != hipSuccess) return fail(HB_ERR_DEVICE);
    const size_t ng1 = (size_t)std::max(n_groups, 1);
    if (!db_get(c, &d_hdb, std::max<uint64_t>(bytes, 4)) ||
        !db_get(c, &d_gbase, ng1 * sizeof(uint64_t)) || !db_get(c, &d_glen, ng1 * sizeof(int32_t)) ||
        !db_get(c, &d_lens, (size_t)std::max(n_seqs, 1) * sizeof(uint32_t)) ||
        !db_get(c, &d_bad, 64))
        return fail(HB_ERR_NOMEM);
    Upload up;
    up.start(c, d_hdb, hdb, bytes);
    if (up.finish() != HB_OK ||
        (n_groups && (hipMemcpy(d_gbase, gbase.data(), n_groups * sizeof(uint64_t),
                                hipMemcpyHostToDevice) != hipSuccess ||
                      hipMemcpy(d_glen, group_len, n_groups * sizeof(int32_t),
                                hipMemcpyHostToDevice) != hipSuccess)))
        return fail(HB_ERR_DEVICE);
    hb_hdb_args a{};
    a.hdb = d_hdb;
    a.group_base = d_gbase;
    a.group_len = d_glen;
    a.n_seqs = (uint32_t)n_seqs;
    a.blocksx = (uint32_t)blocksx;
    a.threadsx = (uint32_t)threadsx;
    a.lens = d_lens;
    std::vector<uint32_t> lens((size_t)n_seqs);
    if (hipEventRecord(ev[0], c->stream) != hipSuccess ||
        hb_launch_hdb_lengths(a, c->stream) != hipSuccess ||
        hipEventRecord(ev[1], c->stream) != hipSuccess ||
        (n_seqs && hipMemcpyAsync(lens.data(), d_lens, lens.size() * sizeof(uint32_t),
                                  hipMemcpyDeviceToHost, c->stream) != hipSuccess) ||
        hipStreamSynchronize(c->stream) != hipSuccess)
        return fail(HB_ERR_DEVICE);
    db->h_offs.resize((size_t)n_seqs + 1);
    // (sum and longest in locals: through the object each sequence's wait for the
    // stores of the one before)
    uint64_t at = 0;
    uint32_t longest = 0;
    for (int32_t i = 0; i < n_seqs; ++i) {
        db->h_offs[i] = at;
        at += lens[i];
        longest = std::max(longest, lens[i]);
    }
    db->h_offs[n_seqs] = at;
    db->max_len = longest;
    db->total = at;
    if (!db_get(c, &db->d_res, db->total + 64)) return fail(HB_ERR_NOMEM);
    int rc = db_meta(db);
    if (rc != HB_OK) return fail(rc);
    a.offs = db->d_offs;
    a.res = db->d_res;
    a.bad = d_bad;
    uint32_t bad = 0;
    if (hipMemsetAsync(db->d_res + db->total, 0, 64, c->stream) != hipSuccess ||
        hipMemsetAsync(d_bad, 0, sizeof(uint32_t), c->stream) != hipSuccess ||
        hipEventRecord(ev[2], c->stream) != hipSuccess ||
        hb_launch_hdb_copy(a, c->stream) != hipSuccess ||
        hipEventRecord(ev[3], c->stream) != hipSuccess ||
        hipMemcpyAsync(&bad, d_bad, sizeof(bad), hipMemcpyDeviceToHost, c->stream) !=
            hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
        return fail(HB_ERR_DEVICE);
    hipEventElapsedTime(&db->hdb_len_ms, ev[0], ev[1]);
    hipEventElapsedTime(&db->hdb_copy_ms, ev[2], ev[3]);
    if (bad) return fail(HB_ERR_RESIDUE);   // checked by the copy kernel
    // the volume's bytes are no longer needed: they are given back before the
    // scan's copy is allocated, so that a large volume's upload holds at most
    // the file plus the residues, then the residues twice
    release();
    d_hdb = nullptr;
    d_gbase = nullptr;
    d_glen = nullptr;
    d_lens = nullptr;
    d_bad = nullptr;
    for (hipEvent_t &e : ev) e = nullptr;
    const int rc2 = db_scan_copy(db);
    if (rc2 != HB_OK) return fail(rc2);
    *out = db;
    return HB_OK;
}

int hb_db_fetch(const hb_db *db, uint8_t *residues, uint64_t res_cap, uint64_t *offsets)
{
    if (!db || !offsets || (db->total > 0 && !residues)) return HB_ERR_ARG;
    if (res_cap < db->total) return HB_ERR_CAPACITY;
    hb_ctx *c = db->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    HB_CHECK(hipSetDevice(c->device));
    std::memcpy(offsets, db->h_offs.data(), db->h_offs.size() * sizeof(uint64_t));
    if (db->total && hipMemcpy(residues, db->d_res, db->total, hipMemcpyDeviceToHost) != hipSuccess)
        return HB_ERR_DEVICE;
    return HB_OK;
}

int hb_db_hdb_info(const hb_db *db, float *lengths_ms, float *copy_ms)
{
    if (!db || !lengths_ms || !copy_ms) return HB_ERR_ARG;
    *lengths_ms = db->hdb_len_ms;
    *copy_ms = db->hdb_copy_ms;
    return HB_OK;
}

uint32_t hb_db_subjects(const hb_db *db) { return db ? db->n : 0; }
uint64_t hb_db_residues(const hb_db *db) { return db ? db->total : 0; }

// ------------------------------------------------------------------ query
int hb_query_free(hb_query *q)
{
    if (!q) return HB_ERR_ARG;
    hipSetDevice(q->ctx->device);
    // scans of this query run on the context stream; the tables go back to
    // the pool, so they must not be reused while one still reads them
    hipStreamSynchronize(q->ctx->stream);
    hb_group_set_free(&q->gs);
    delete q;
    return HB_OK;
}

int hb_query_prepare(hb_ctx *c, const uint8_t *seq, int32_t len, int32_t n_ctx,
                     const int32_t *ctx_off, const int32_t *ctx_len, const int32_t *xdrop,
                     const int32_t *cutoff, const hb_params *params, hb_query **out)
{
    return hb_query_prepare_masked(c, seq, len, n_ctx, ctx_off, ctx_len, xdrop, cutoff, params,
                                   nullptr, out);
}

int hb_query_prepare_masked(hb_ctx *c, const uint8_t *seq, int32_t len, int32_t n_ctx,
                            const int32_t *ctx_off, const int32_t *ctx_len, const int32_t *xdrop,
                            const int32_t *cutoff, const hb_params *params,
                            const uint8_t *lut_mask, hb_query **out)
{
    if (!c || !out || !cutoff) return HB_ERR_ARG;
    *out = nullptr;
    int rc = hb_check_query(seq, len, n_ctx, ctx_off, ctx_len, xdrop);
    if (rc) return rc;
    hb_query *q = new (std::nothrow) hb_query;
    if (!q) return HB_ERR_NOMEM;
    q->ctx = c;
    rc = hb_resolve_params(params, &q->p);
    if (rc) {
        delete q;
        return rc;
    }
    q->ctx_off.assign(ctx_off, ctx_off + n_ctx);
    q->ctx_len.assign(ctx_len, ctx_len + n_ctx);
    std::vector<hb_concat> qs(1);
    qs[0].seq.assign(seq, seq + len);
    qs[0].ctx_off.assign(ctx_off, ctx_off + n_ctx);
    qs[0].ctx_len.assign(ctx_len, ctx_len + n_ctx);
    qs[0].xdrop.assign(xdrop, xdrop + n_ctx);
    qs[0].cutoff.assign(cutoff, cutoff + n_ctx);
    if (lut_mask) qs[0].mask.assign(lut_mask, lut_mask + len);
    // The diagonal state (4 bytes per diagonal) stays in LDS when it fits;
    // longer queries (the reference accepts 32,768 residues,
    // H-BLAST/h_blast.cu:1293) keep it in global memory.  The query itself,
    // its context tables and the matrix are always in LDS.
    const int32_t D = (len + q->p.window + 63) & ~63;
    if (!hb_query_lds_ok(c, len, n_ctx)) {
        delete q;
        return HB_ERR_UNSUPPORTED;
    }
    const size_t fixed = hb_scan_fixed_lds((len + 15) & ~15, hb_ctx_pad(n_ctx));
    q->lds_fits = fixed + hb_scan_wave_lds(D, 256, 4) <= c->max_lds;
    std::lock_guard<std::mutex> lk(c->mu);
    if (hipSetDevice(c->device) != hipSuccess) {
        delete q;
        return HB_ERR_DEVICE;
    }
    rc = hb_group_set_build(c, qs, std::vector<int32_t>(1, 0), q->p, false, c->stream, &q->gs);
    if (rc) {
        delete q;
        return rc;
    }
    *out = q;
    return HB_OK;
}

int hb_query_set_state_mode(hb_query *q, int mode)
{
    if (!q) return HB_ERR_ARG;
    switch (mode) {
    case HB_STATE_AUTO:
    case HB_STATE_GLOBAL: q->mode = mode; return HB_OK;
    case HB_STATE_LDS:
    case HB_STATE_LDS16:   // one LDS format now; the old 16-bit request means LDS
        if (!q->lds_fits) return HB_ERR_UNSUPPORTED;
        q->mode = HB_STATE_LDS;
        return HB_OK;
    default: return HB_ERR_ARG;
    }
}

int hb_query_set_reset_interval(hb_query *q, int32_t interval)
{
    if (!q || interval < 0) return HB_ERR_ARG;
    q->reset_interval = interval;
    return HB_OK;
}

int hb_query_state_mode(const hb_query *q)
{
    if (!q) return HB_ERR_ARG;
    return q->mode;
}

// The placement a scan of q over db uses.
static int state_place(const hb_query *q, const hb_db *db)
{
    switch (q->mode) {
    case HB_STATE_LDS:
        return hb_state_lds_ok(db->max_len, q->p.window) ? HB_PLACE_LDS : -1;
    case HB_STATE_GLOBAL: return HB_PLACE_GLOBAL;
    default:
        return hb_state_choose(q->ctx, q->gs.diag_len_max,
                               hb_scan_fixed_lds(q->gs.qlen_pad_max, q->gs.ctx_pad_max),
                               db->max_len, q->p.window);
    }
}

int hb_query_lut_info(const hb_query *q, uint32_t *n_entries, uint32_t *n_cells_used)
{
    if (!q) return HB_ERR_ARG;
    if (n_entries) *n_entries = q->gs.n_entries[0];
    if (n_cells_used) *n_cells_used = q->gs.n_cells_used[0];
    return HB_OK;
}

int hb_query_lut_fetch(const hb_query *q, uint32_t *cell_start, uint32_t *entries, uint32_t cap)
{
    if (!q || !cell_start) return HB_ERR_ARG;
    const uint32_t ne = q->gs.n_entries[0];
    if (!entries && ne) return HB_ERR_ARG;
    if (cap < ne) return HB_ERR_CAPACITY;
    HB_CHECK(hipSetDevice(q->ctx->device));
    const int32_t nc = 1 << q->gs.desc[0].shift;
    std::vector<uint2> cells((size_t)HB_NCELLS * nc);
    std::vector<uint32_t> ent(q->gs.entries_bytes / sizeof(uint32_t));
    HB_CHECK(hipMemcpy(cells.data(), q->gs.desc[0].cells, cells.size() * sizeof(uint2),
                       hipMemcpyDeviceToHost));
    if (ne)
        HB_CHECK(hipMemcpy(ent.data(), q->gs.desc[0].entries, q->gs.entries_bytes,
                           hipMemcpyDeviceToHost));
    // a cell's entries are those of its classes, ascending
    uint32_t k = 0;
    for (int i = 0; i < HB_NCELLS; ++i) {
        cell_start[i] = k;
        for (int32_t j = 0; j < nc; ++j) {
            const uint2 x = cells[(size_t)i * nc + j];
            for (uint32_t e = 0; e < x.y; ++e) entries[k++] = ent[x.x + e];
        }
        if (nc > 1) std::sort(entries + cell_start[i], entries + k);
    }
    cell_start[HB_NCELLS] = k;
    return HB_OK;
}

// ------------------------------------------------------------------ scan
// Kernel arguments of a plain scan of q over db with launch configuration
// cfg and placement place (outputs, counters and state filled by the caller).
static int plain_scan_args(const hb_db *db, const hb_query *q, int place,
                           const hb_launch_cfg &cfg, hb_scan_args *a)
{
    memset(a, 0, sizeof(*a));
    a->res = db->d_scan_res;   // subjects in processing order (a->subj's offsets)
    a->offs = db->d_offs;
    a->subj = db->d_subj;
    a->tiles = db->d_tiles + db->n_tiles + 1;   // the plain scan's tiles
    a->tile_begin = 0;
    a->tile_end = db->n_qtiles;
    a->groups = q->gs.d_desc;
    a->n_groups = 1;
    a->qlen_pad_max = q->gs.qlen_pad_max;
    a->ctx_pad_max = q->gs.ctx_pad_max;
    a->diag_len_max = q->gs.diag_len_max;
    a->split = q->gs.split;
    a->many = cfg.many;
    a->wave_lds = (uint32_t)hb_scan_wave_lds(q->gs.diag_len_max, cfg.ring, hb_state_bytes(place));
    a->ring = (uint32_t)cfg.ring;
    a->state_limit = hb_state_limit(place, db->max_len);
    if (q->reset_interval > 0) {
        // a subject and its successor must fit below the interval
        if ((uint64_t)q->reset_interval <= 2 * (db->max_len + (uint64_t)q->p.window) + 64)
            return HB_ERR_UNSUPPORTED;
        a->state_limit = std::min(a->state_limit, q->reset_interval - (int32_t)db->max_len);
    }
    a->mat32 = q->gs.d_mat;
    a->window = q->p.window;
    return HB_OK;
}

// Configuration of a plain scan.  A query of up to 152 residues leaves five
// workgroups the LDS they need with the largest ring (their share of 160 KB in
// steps of 1,280 bytes; the runtime's count knows no steps, and at 160 residues
// the fifth would start when the others are done): 20 wavefronts per CU, where
// each of them gets kShortShare residues (us with 16 and with 20: 60 residues
// against 20,000 subjects 83 and 87, 50,000 127 and 120, 200,000 414 and 370).
// (Not in a scan that must allocate nothing: that kernel has scratch.)
static constexpr uint64_t kShortShare = 4096;
static int plain_config(const hb_db *db, const hb_query *q, int place, bool noalloc,
                        hb_launch_cfg *cfg)
{
    hb_ctx *c = db->ctx;
    const uint32_t items = db->n_qtiles << q->gs.desc[0].shift;
    int rc = hb_scan_config(c, false, q->gs.split != 0, q->gs.qlen_pad_max, q->gs.ctx_pad_max,
                            q->gs.diag_len_max, items, cfg, place);
    if (rc) return rc;
    cfg->many = !noalloc && c->short_scan && place == HB_PLACE_LDS && !q->gs.split &&
                cfg->waves * HB_WAVE == HB_BLOCK && cfg->ring == HB_RING_MAX &&
                cfg->lds <= kShortLds && db->total >= c->n_cu * 16ull * kShortShare;
    if (cfg->many)
        cfg->blocks = (int)std::min<uint64_t>(5ull * c->n_cu, (items + cfg->waves - 1) / cfg->waves);
    return HB_OK;
}

static int launch_scan(hb_scan *s)
{
    hb_ctx *c = s->ctx;
    hb_db *db = s->db;
    hb_query *q = s->q;
    hb_launch_cfg cfg;
    const int place = state_place(q, db);
    if (place < 0) return HB_ERR_UNSUPPORTED;   // LDS state asked for, subjects too long
    s->place = place;
    int rc = plain_config(db, q, place, false, &cfg);
    if (rc) return rc;
    if (place == HB_PLACE_GLOBAL && !s->d_gstate) {
        s->d_gstate = static_cast<uint32_t *>(hb_pool_get(
            c, (size_t)cfg.blocks * cfg.waves * (size_t)q->gs.diag_len_max * HB_GSTATE_WORD));
        if (!s->d_gstate) return HB_ERR_NOMEM;
    }
    hb_scan_args a;
    rc = plain_scan_args(db, q, place, cfg, &a);
    if (rc) return rc;
    a.gstate = place == HB_PLACE_GLOBAL ? s->d_gstate : nullptr;   // cleared by each wavefront
    a.work_counter = s->d_misc + HB_QUEUE_STRIDE;
    a.out = s->d_out;
    a.out_cap = s->cap;
    a.out_count = s->d_misc;
    a.stats = s->d_stats;
    a.group_totals = nullptr;
    HB_CHECK(hb_launch_fill_u32(s->d_misc, 0u, HB_SCAN_MISC_WORDS, c->stream));
    if (a.split) HB_CHECK(hb_launch_fill_u32(s->d_stats, 0u, 3 * db->n, c->stream));
    HB_CHECK(hipEventRecord(s->ev0, c->stream));
    if (db->n_qtiles) HB_CHECK(hb_launch_scan(a, false, cfg.blocks, cfg.waves * HB_WAVE, cfg.lds, c->stream));
    HB_CHECK(hipEventRecord(s->ev1, c->stream));
    return HB_OK;
}

// ------------------------------------------------------------------ memory fit
// Device bytes of a plain scan of q over n subjects with `residues`
// residues (0: bounded by file_bytes), loaded from a .hDb of file_bytes
// (0: packed arrays), subjects up to max_len residues:
//   upload:   the file, the residues, lengths (4 B), offsets (8 B) and
//             processing-order records (16 B) and their sort (24 B) per
//             subject, tiles;
//   resident: the residues, their processing-order copy (spans padded to
//             16 B) and the metadata;
//   scan:     the HSP reservation (32 B records), counters (12 B per
//             subject), the diagonal state in global memory if placed there;
//   results:  per-subject stats (24 B), the ordered records, the layout's
//             scratch (4 B per subject) and the list of large subjects.
static uint64_t scan_need_bytes(const hb_ctx *c, const hb_query *q, uint64_t file_bytes,
                                uint64_t residues, uint32_t n, uint64_t max_len)
{
    const uint64_t R = residues ? residues : file_bytes;
    const uint64_t meta = 8ull * (n + 1) + 16ull * n + 4ull * (n / 16 + std::min(n, 1u << 17) + 4);
    const uint64_t upload = file_bytes + (R + 64) + 4ull * n + hb_load_scratch(n) + meta;
    const uint64_t resident = (R + 64) + (R + 16ull * n + 64) + meta;
    const uint64_t cap = std::max<uint64_t>(1u << 18, n / 4);
    uint64_t scan = 32 * cap + 12ull * n + 64;
    int place = HB_PLACE_LDS;
    switch (q->mode) {
    case HB_STATE_GLOBAL: place = HB_PLACE_GLOBAL; break;
    case HB_STATE_LDS: place = HB_PLACE_LDS; break;
    default:
        place = hb_state_choose(c, q->gs.diag_len_max,
                                hb_scan_fixed_lds(q->gs.qlen_pad_max, q->gs.ctx_pad_max), max_len,
                                q->p.window);
    }
    if (place == HB_PLACE_GLOBAL) scan += hb_gstate_bytes_max(c, q->gs.diag_len_max);
    const uint64_t results = 24ull * n + 32 * cap + 4ull * (n + n / 4096 + 1) +
                             4096 * sizeof(hb_fin_big);
    return std::max(upload, resident + scan + results);
}

int hb_check_memory(hb_ctx *c, const hb_query *q, uint64_t file_bytes, uint64_t residues,
                    uint32_t n_seqs, uint64_t max_len, int64_t budget, uint64_t *need,
                    int32_t *fits)
{
    if (!c || !q || q->ctx != c || !need || !fits) return HB_ERR_ARG;
    *need = scan_need_bytes(c, q, file_bytes, residues, n_seqs, max_len);
    uint64_t room = (uint64_t)std::max<int64_t>(budget, 0);
    if (budget < 0) {
        uint64_t total = 0;
        int rc = hb_mem_info(c, &room, &total);
        if (rc) return rc;
    }
    *fits = *need <= room ? 1 : 0;
    return HB_OK;
}

// ------------------------------------------------------------------ co-scheduled search
// The library's device steps of the co-scheduled loop (hb_cosched.cpp).
namespace {
struct CoschedDevice {
    hb_ctx *ctx = nullptr;
    hb_query *q = nullptr;
    int64_t budget = -1;
    hb_gpu_results_fn gpu = nullptr;
    void *user = nullptr;
    hb_db *db = nullptr;
    hb_scan *scan = nullptr;
    std::vector<hb_subject_stats> stats;
    std::vector<hb_hsp> hsps;

    void drop()
    {
        if (scan) hb_scan_free(scan);
        if (db) hb_db_free(db);
        scan = nullptr;
        db = nullptr;
    }
    static CoschedDevice *self(void *u) { return static_cast<CoschedDevice *>(u); }
    static int fits(void *u, int32_t, const hb_hdb_share *sh, int32_t max_len, uint64_t *need,
                    int32_t *ok)
    {
        CoschedDevice *d = self(u);
        return hb_check_memory(d->ctx, d->q, sh->bytes, 0, (uint32_t)sh->gpu_seqs,
                               (uint64_t)std::max(max_len, 0), d->budget, need, ok);
    }
    static int launch(void *u, int32_t, const uint8_t *hdb, const hb_hdb_share *sh,
                      int32_t blocksx, int32_t threadsx, const int32_t *group_len)
    {
        CoschedDevice *d = self(u);
        int rc = hb_db_upload_hdb(d->ctx, hdb, sh->bytes, blocksx, threadsx, sh->gpu_seqs,
                                  group_len, sh->n_groups, &d->db);
        if (rc) return rc;
        rc = hb_scan_start(d->ctx, d->db, d->q, &d->scan);
        if (rc) d->drop();
        return rc;
    }
    static int fetch(void *u, int32_t volume, int64_t oid_base, double *gpu_seconds,
                     uint64_t *n_hsp)
    {
        CoschedDevice *d = self(u);
        uint64_t n = 0;
        int rc = hb_scan_results(d->scan, nullptr, nullptr, 0, &n);
        const uint32_t ns = d->db ? d->db->n : 0;
        if (!rc) {
            d->stats.resize(std::max<uint32_t>(ns, 1));
            d->hsps.resize(std::max<uint64_t>(n, 1));
            rc = hb_scan_results(d->scan, d->stats.data(), d->hsps.data(), n, &n);
        }
        float ms = 0.f;
        if (!rc) rc = hb_scan_elapsed_ms(d->scan, &ms);
        d->drop();
        if (rc) return rc;
        for (uint64_t i = 0; i < n; ++i) d->hsps[i].oid += (uint32_t)oid_base;
        *gpu_seconds = ms / 1000.0;
        *n_hsp = n;
        if (d->gpu && d->gpu(d->user, volume, oid_base, d->stats.data(), ns, d->hsps.data(), n))
            return HB_ERR_STATE;
        return HB_OK;
    }
    static void abandon(void *u) { self(u)->drop(); }
};
}  // namespace

int hb_cosearch(hb_ctx *c, const char *index_path, const uint8_t *seq, int32_t len,
                int32_t n_ctx, const int32_t *ctx_off, const int32_t *ctx_len,
                const int32_t *xdrop, const int32_t *cutoff, const hb_params *params,
                const uint8_t *lut_mask, const hb_runtime_options *options,
                int32_t cpu_threads, int32_t gapped, int64_t device_budget,
                hb_cpu_search_fn cpu, hb_gpu_results_fn gpu, void *user,
                hb_volume_report *reports, int32_t report_cap, int32_t *n_volumes)
{
    if (!c || !index_path || !cpu || !n_volumes) return HB_ERR_ARG;
    hb_query *q = nullptr;
    int rc = hb_query_prepare_masked(c, seq, len, n_ctx, ctx_off, ctx_len, xdrop, cutoff, params,
                                     lut_mask, &q);
    if (rc) return rc;
    CoschedDevice dev;
    dev.ctx = c;
    dev.q = q;
    dev.budget = device_budget;
    dev.gpu = gpu;
    dev.user = user;
    hb_cosched_steps steps;
    steps.user = &dev;
    steps.fits = &CoschedDevice::fits;
    steps.launch = &CoschedDevice::launch;
    steps.fetch = &CoschedDevice::fetch;
    steps.abandon = &CoschedDevice::abandon;
    rc = hb_cosched_run(index_path, options, cpu_threads, gapped, len,
                        (uint32_t)(len / std::max(n_ctx, 1)), &steps, cpu, user, reports,
                        report_cap, n_volumes);
    dev.drop();
    hb_query_free(q);
    return rc;
}

// ------------------------------------------------------------------ no-alloc scan
int hb_scan_noalloc(hb_ctx *c, hb_db *db, hb_query *q, hb_hsp *d_hsps, uint32_t hsp_cap,
                    uint32_t *d_counts, uint32_t *d_n_hsp, void *stream)
{
    if (!c || !db || !q || db->ctx != c || q->ctx != c || !d_n_hsp || (hsp_cap && !d_hsps))
        return HB_ERR_ARG;
    if (!c->scratch_dev) return HB_ERR_STATE;
    std::lock_guard<std::mutex> lk(c->mu);
    HB_CHECK(hipSetDevice(c->device));
    hipStream_t st = stream ? static_cast<hipStream_t>(stream) : c->stream;
    const int place = state_place(q, db);
    if (place < 0) return HB_ERR_UNSUPPORTED;
    hb_launch_cfg cfg;
    int rc = plain_config(db, q, place, true, &cfg);
    if (rc) return rc;
    hb_scan_args a;
    rc = plain_scan_args(db, q, place, cfg, &a);
    if (rc) return rc;
    int blocks = cfg.blocks;
    if (place == HB_PLACE_GLOBAL) {
        // the state of every wavefront of the grid must fit the scratch:
        // fewer workgroups for long queries, none fits -> refused
        const size_t per_block = HB_GSTATE_WORD * (size_t)q->gs.diag_len_max * (size_t)cfg.waves;
        if (per_block > HB_NOALLOC_STATE_BYTES) return HB_ERR_UNSUPPORTED;
        blocks = std::min(blocks, (int)(HB_NOALLOC_STATE_BYTES / per_block));
        a.gstate = reinterpret_cast<uint32_t *>(c->scratch_dev + HB_NOALLOC_HEAD);
    }
    uint32_t *ctr = reinterpret_cast<uint32_t *>(c->scratch_dev);
    a.out_count = ctr;
    a.work_counter = ctr + HB_QUEUE_STRIDE;
    a.out = d_hsps;
    a.out_cap = hsp_cap;
    a.stats = d_counts;
    a.group_totals = nullptr;
    // the previous call's counters stay in the scratch: cleared by a kernel
    HB_CHECK(hb_launch_fill_u32(ctr, 0u, HB_SCAN_MISC_WORDS, st));
    if (a.split && d_counts) HB_CHECK(hb_launch_fill_u32(d_counts, 0u, 3 * db->n, st));
    if (db->n_qtiles)
        HB_CHECK(hb_launch_scan(a, false, blocks, cfg.waves * HB_WAVE, cfg.lds, st));
    HB_CHECK(hipMemcpyAsync(d_n_hsp, ctr, sizeof(uint32_t), hipMemcpyDeviceToDevice, st));
    return HB_OK;
}

int hb_scan_free(hb_scan *s)
{
    if (!s) return HB_ERR_ARG;
    hipSetDevice(s->ctx->device);
    if (!s->waited) hipStreamSynchronize(s->ctx->stream);
    hb_pool_put(s->ctx, s->d_out);
    hb_pool_put(s->ctx, s->d_misc);
    hb_pool_put(s->ctx, s->d_stats);
    if (s->d_gstate) hb_pool_put(s->ctx, s->d_gstate);
    if (s->ev0) hipEventDestroy(s->ev0);
    if (s->ev1) hipEventDestroy(s->ev1);
    delete s;
    return HB_OK;
}

int hb_scan_state_mode(const hb_scan *s)
{
    if (!s) return HB_ERR_ARG;
    return s->place == HB_PLACE_GLOBAL ? HB_STATE_GLOBAL : HB_STATE_LDS;
}

int hb_scan_start(hb_ctx *c, hb_db *db, hb_query *q, hb_scan **out)
{
    if (!c || !db || !q || !out || db->ctx != c || q->ctx != c) return HB_ERR_ARG;
    *out = nullptr;
    std::lock_guard<std::mutex> lk(c->mu);
    HB_CHECK(hipSetDevice(c->device));
    hb_scan *s = new (std::nothrow) hb_scan;
    if (!s) return HB_ERR_NOMEM;
    s->ctx = c;
    s->db = db;
    s->q = q;
    s->cap = std::max<uint32_t>(1u << 18, db->n / 4);
    s->d_out = (hb_hsp *)hb_pool_get(c, (size_t)s->cap * sizeof(hb_hsp));
    s->d_misc = (uint32_t *)hb_pool_get(c, HB_SCAN_MISC_WORDS * sizeof(uint32_t));
    s->d_stats = (uint32_t *)hb_pool_get(c, (size_t)std::max<uint32_t>(db->n, 1) * 3 * sizeof(uint32_t));
    if (!s->d_out || !s->d_misc || !s->d_stats) {
        hb_scan_free(s);
        return HB_ERR_NOMEM;
    }
    if (hipEventCreate(&s->ev0) != hipSuccess || hipEventCreate(&s->ev1) != hipSuccess) {
        hb_scan_free(s);
        return HB_ERR_DEVICE;
    }
    int rc = launch_scan(s);
    if (rc) {
        hb_scan_free(s);
        return rc;
    }
    *out = s;
    return HB_OK;
}

int hb_scan_wait(hb_scan *s)
{
    if (!s) return HB_ERR_ARG;
    if (s->waited) return HB_OK;
    hb_ctx *c = s->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    HB_CHECK(hipSetDevice(c->device));
    for (;;) {
        uint32_t n = 0;
        HB_CHECK(hipMemcpyAsync(&n, s->d_misc, sizeof(n), hipMemcpyDeviceToHost, c->stream));
        HB_CHECK(hipStreamSynchronize(c->stream));
        if (n <= s->cap) {
            s->n_out = n;
            break;
        }
        // The kernel counted every HSP but stored only cap: rerun with room
        // for all of them (the stage is deterministic).
        hb_pool_put(c, s->d_out);
        s->cap = n + n / 8 + 1024;
        s->d_out = (hb_hsp *)hb_pool_get(c, (size_t)s->cap * sizeof(hb_hsp));
        if (!s->d_out) {
            s->cap = 0;
            return HB_ERR_NOMEM;
        }
        int rc = launch_scan(s);
        if (rc) return rc;
    }
    s->waited = true;
    return HB_OK;
}

int hb_scan_elapsed_ms(hb_scan *s, float *ms)
{
    if (!s || !ms) return HB_ERR_ARG;
    int rc = hb_scan_wait(s);
    if (rc) return rc;
    HB_CHECK(hipEventElapsedTime(ms, s->ev0, s->ev1));
    return HB_OK;
}

int hb_scan_results(hb_scan *s, hb_subject_stats *stats, hb_hsp *hsps, uint64_t cap,
                    uint64_t *n_hsp)
{
    if (!s) return HB_ERR_ARG;
    int rc = hb_scan_wait(s);
    if (rc) return rc;
    const uint64_t n = s->n_out;
    if (n_hsp) *n_hsp = n;
    if (!hsps && !stats) return HB_OK;
    if (hsps && cap < n) return HB_ERR_CAPACITY;
    const uint32_t ns = s->db->n;
    if (ns == 0) return HB_OK;
    hb_ctx *c = s->ctx;
    HB_CHECK(hipSetDevice(c->device));
    // the layout is built on the device (counts -> first indices, records
    // grouped by subject and ordered by (s_off, q_off)), then copied out
    constexpr uint32_t kBig = 4096;
    const uint32_t nb = (ns + 4095) / 4096;
    const size_t b_st = (size_t)ns * sizeof(hb_subject_stats);
    const size_t b_rec = (size_t)std::max<uint64_t>(n, 1) * sizeof(hb_hsp);
    const size_t b_scr = ((size_t)ns + nb + 1) * sizeof(uint32_t);
    const size_t b_big = kBig * sizeof(hb_fin_big);
    auto *d_st = static_cast<hb_subject_stats *>(hb_pool_get(c, b_st));
    auto *d_rec = static_cast<hb_hsp *>(hb_pool_get(c, b_rec));
    auto *d_scr = static_cast<uint32_t *>(hb_pool_get(c, b_scr));
    auto *d_big = static_cast<hb_fin_big *>(hb_pool_get(c, b_big));
    auto release = [&]() {
        hb_pool_put(c, d_st);
        hb_pool_put(c, d_rec);
        hb_pool_put(c, d_scr);
        hb_pool_put(c, d_big);
    };
    if (!d_st || !d_rec || !d_scr || !d_big) {
        release();
        return HB_ERR_NOMEM;
    }
    uint32_t *d_nbig = d_scr + ns + nb;
    hipStream_t st = c->stream;
    uint32_t nbig = 0;
    hipError_t e = hb_launch_finalize(s->d_stats, ns, s->d_out, (uint32_t)n, d_st, d_rec, d_scr, d_big,
                                      kBig, d_nbig, 1, st);
    if (e == hipSuccess) {
        // all of it behind the kernels and one wait, unless the buffer would grow
        // for that
        const size_t w_st = stats ? b_st : 0, w_rec = hsps ? (size_t)n * sizeof(hb_hsp) : 0;
        const bool at_once = 64 + CopyOut::room(w_st) + CopyOut::room(w_rec) <= CopyOut::kKeep;
        CopyOut out(c, 64 + (at_once ? CopyOut::room(w_st) + w_rec : std::max(w_st, w_rec)), st);
        const size_t o_big = out.add(d_nbig, sizeof(nbig)), o_st = out.add(d_st, w_st);
        size_t o_rec = at_once ? out.add(d_rec, w_rec) : 0;
        e = out.wait();
        if (e == hipSuccess) {
            memcpy(&nbig, out.ptr(o_big), sizeof(nbig));
            if (w_st) out.store(stats, o_st, w_st);
            if (!at_once && w_rec) {
                out.rewind();
                o_rec = out.add(d_rec, w_rec);
                e = out.wait();
            }
            if (e == hipSuccess && w_rec) out.store(hsps, o_rec, w_rec);
        }
    }
    // subjects with many records are ordered here
    std::vector<hb_fin_big> big;
    if (e == hipSuccess && hsps && nbig) {
        if (nbig <= kBig) {
            big.resize(nbig);
            e = hipMemcpy(big.data(), d_big, nbig * sizeof(hb_fin_big), hipMemcpyDeviceToHost);
        } else {
            std::vector<hb_subject_stats> all;
            const hb_subject_stats *sp = stats;
            if (!sp) {
                all.resize(ns);
                e = hipMemcpy(all.data(), d_st, b_st, hipMemcpyDeviceToHost);
                sp = all.data();
            }
            for (uint32_t i = 0; e == hipSuccess && i < ns; ++i)
                if (sp[i].n_hsp > HB_FIN_SORT_MAX)
                    big.push_back(hb_fin_big{i, sp[i].n_hsp, (uint64_t)sp[i].first});
        }
    }
    if (e != hipSuccess) hipStreamSynchronize(st);   // the kernels that were launched
    release();
    if (e != hipSuccess) {
        hb_note_hip_error(e, "hb_scan_results", __LINE__);
        return HB_ERR_DEVICE;
    }
    for (const hb_fin_big &b : big)
        std::sort(hsps + b.first, hsps + b.first + b.n, [](const hb_hsp &x, const hb_hsp &y) {
            if (x.s_off != y.s_off) return x.s_off < y.s_off;
            return x.q_off < y.q_off;
        });
    return HB_OK;
}

int hb_scan_results_compact(hb_scan *s, hb_subject_hits *subj, uint64_t subj_cap, hb_hsp *hsps,
                            uint64_t hsp_cap, hb_scan_totals *totals)
{
    if (!s || !totals) return HB_ERR_ARG;
    int rc = hb_scan_wait(s);
    if (rc) return rc;
    std::memset(totals, 0, sizeof(*totals));
    const uint64_t n = s->n_out;
    totals->n_hsp = n;
    const uint32_t ns = s->db->n;
    if (ns == 0) return HB_OK;
    hb_ctx *c = s->ctx;
    HB_CHECK(hipSetDevice(c->device));
    // the same device layout as hb_scan_results, with the per-subject
    // entries compacted to the subjects with HSPs
    constexpr uint32_t kBig = 4096;
    const uint32_t nb = (ns + 4095) / 4096;
    const uint64_t max_subj = std::min<uint64_t>(ns, n);
    const size_t b_sub = (size_t)std::max<uint64_t>(max_subj, 1) * sizeof(hb_subject_hits);
    const size_t b_rec = (size_t)std::max<uint64_t>(n, 1) * sizeof(hb_hsp);
    const size_t b_scr = (2 * (size_t)nb + ns) * sizeof(uint32_t);
    const size_t b_big = kBig * sizeof(hb_fin_big);
    const size_t b_small = 64 + 2 * (size_t)nb * sizeof(unsigned long long);   // totals, blocks' sums
    auto *d_sub = static_cast<hb_subject_hits *>(hb_pool_get(c, b_sub));
    auto *d_rec = static_cast<hb_hsp *>(hb_pool_get(c, b_rec));
    auto *d_scr = static_cast<uint32_t *>(hb_pool_get(c, b_scr));
    auto *d_big = static_cast<hb_fin_big *>(hb_pool_get(c, b_big));
    auto *d_small = static_cast<hb_fin_small *>(hb_pool_get(c, b_small));
    auto release = [&]() {
        hb_pool_put(c, d_sub);
        hb_pool_put(c, d_rec);
        hb_pool_put(c, d_scr);
        hb_pool_put(c, d_big);
        hb_pool_put(c, d_small);
    };
    if (!d_sub || !d_rec || !d_scr || !d_big || !d_small) {
        release();
        return HB_ERR_NOMEM;
    }
    hipStream_t st = c->stream;
    hb_fin_small small{};
    hipError_t e = hb_launch_finalize_compact(
        s->d_stats, ns, s->d_out, (uint32_t)n, d_sub, d_rec, d_scr,
        reinterpret_cast<unsigned long long *>(reinterpret_cast<char *>(d_small) + 64), d_big, kBig,
        d_small, st);
    std::vector<hb_subject_hits> host_sub;
    hb_subject_hits *sp = subj;
    uint32_t nbig = 0;
    bool done = false;   // the results are copied
    if (e == hipSuccess) {
        // The records' number is known and bounds that of the entries: up to
        // kAtOnce of both are copied behind the kernels with one wait (the
        // entries too many cost less than another wait); else when the totals
        // are known.
        constexpr size_t kAtOnce = (size_t)32 << 20;
        const size_t w_sub = subj ? (size_t)max_subj * sizeof(hb_subject_hits) : 0;
        const size_t w_rec = hsps ? (size_t)n * sizeof(hb_hsp) : 0;
        const bool at_once = w_sub + w_rec <= kAtOnce;
        CopyOut out(c, 64 + (at_once ? CopyOut::room(w_sub) + w_rec : 0), st);
        const size_t o_small = out.add(d_small, sizeof(small));
        const size_t o_sub = at_once ? out.add(d_sub, w_sub) : 0;
        const size_t o_rec = at_once ? out.add(d_rec, w_rec) : 0;
        e = out.wait();
        if (e == hipSuccess) {
            memcpy(&small, out.ptr(o_small), sizeof(small));
            nbig = small.n_big;
            totals->lookup_hits = small.lookup_hits;
            totals->extensions = small.extensions;
            totals->n_subjects = small.n_subj;
            if ((subj && subj_cap < small.n_subj) || (hsps && hsp_cap < n)) {
                release();
                return HB_ERR_CAPACITY;
            }
            if (at_once) {
                if (w_sub) out.store(subj, o_sub, (size_t)small.n_subj * sizeof(hb_subject_hits));
                if (w_rec) out.store(hsps, o_rec, w_rec);
            }
        }
        if (e == hipSuccess && !sp && hsps && nbig > kBig) {   // the host needs the entries below
            host_sub.resize(small.n_subj);
            sp = host_sub.data();
        }
        done = at_once;
    }
    const uint32_t n_subj = small.n_subj;
    if (e == hipSuccess && sp && n_subj && !(done && sp == subj) &&
        hb_copy_out(c, sp, d_sub, (size_t)n_subj * sizeof(hb_subject_hits), st) != HB_OK)
        e = hipErrorUnknown;
    if (e == hipSuccess && hsps && n && !done &&
        hb_copy_out(c, hsps, d_rec, (size_t)n * sizeof(hb_hsp), st) != HB_OK)
        e = hipErrorUnknown;
    // subjects with many records are ordered here
    std::vector<hb_fin_big> big;
    if (e == hipSuccess && hsps && nbig) {
        if (nbig <= kBig) {
            big.resize(nbig);
            e = hipMemcpy(big.data(), d_big, nbig * sizeof(hb_fin_big), hipMemcpyDeviceToHost);
        } else {
            for (uint32_t i = 0; i < n_subj; ++i)
                if (sp[i].n_hsp > HB_FIN_SORT_MAX)
                    big.push_back(hb_fin_big{sp[i].oid, sp[i].n_hsp, sp[i].first});
        }
    }
    if (e != hipSuccess) hipStreamSynchronize(st);   // the kernels that were launched
    release();
    if (e != hipSuccess) {
        hb_note_hip_error(e, "hb_scan_results_compact", __LINE__);
        return HB_ERR_DEVICE;
    }
    for (const hb_fin_big &b : big)
        std::sort(hsps + b.first, hsps + b.first + b.n, [](const hb_hsp &x, const hb_hsp &y) {
            if (x.s_off != y.s_off) return x.s_off < y.s_off;
            return x.q_off < y.q_off;
        });
    return HB_OK;
}

void hb_gap_params_default(hb_gap_params *p)
{
    if (!p) return;
    p->gap_open = 11;
    p->gap_extend = 1;
    p->x_dropoff = HB_DEFAULT_GAP_XDROP;
    p->reserved = 0;
}

static bool gap_params_ok(const hb_gap_params *gp)
{
    return gp && gp->gap_open >= 0 && gp->gap_extend >= 0 && gp->x_dropoff >= 0 &&
           gp->gap_open <= 1000 && gp->gap_extend <= 1000 && gp->x_dropoff <= 100000;
}

// The gapped stage on ungapped records already on the device: st3_in holds
// 3 counters per subject (the HSP count third), rec_in the n records in any
// order.  Lays the records out by subject, runs the main and wide passes,
// compacts and copies out.  Runs on the context's stream; the caller holds
// the context lock.
static int gapped_core(hb_ctx *c, const hb_db *db, const uint8_t *d_query, const int8_t *d_mat,
                       const std::vector<int32_t> &ctx_off, const std::vector<int32_t> &ctx_len,
                       const int32_t *gap_cutoff, const hb_gap_params *gp, const uint32_t *st3_in,
                       const hb_hsp *rec_in, uint64_t n, hb_gapped_stats *stats,
                       hb_gapped_hsp *hsps, uint64_t cap, uint64_t *n_hsp, float *ms_out,
                       uint32_t *wide_out)
{
    const uint32_t ns = db->n;
    const int32_t n_ctx = (int32_t)ctx_off.size();
    // pool buffers, all returned at the end
    std::vector<void *> held;
    bool oom = false;
    auto get = [&](size_t bytes) -> void * {
        bytes = std::max<size_t>(bytes, 64);
        void *p = hb_pool_get(c, bytes);
        if (!p) oom = true;
        else held.push_back(p);
        return p;
    };
    constexpr uint32_t kBig = 4096;
    const uint32_t nb = (ns + 4095) / 4096;
    const uint64_t nr = std::max<uint64_t>(n, 1);
    auto *d_ust = static_cast<hb_subject_stats *>(get((size_t)ns * sizeof(hb_subject_stats)));
    auto *d_urec = static_cast<hb_hsp *>(get(nr * sizeof(hb_hsp)));
    // (layout's scratch; its big-subject count; the list's 128 buckets, cleared
    // with that count)
    auto *d_scr = static_cast<uint32_t *>(get(((size_t)ns + nb + 1 + 128) * sizeof(uint32_t)));
    auto *d_big = static_cast<hb_fin_big *>(get(kBig * sizeof(hb_fin_big)));
    auto *d_st3 = static_cast<uint32_t *>(get((size_t)ns * 3 * sizeof(uint32_t)));
    auto *d_gout = static_cast<hb_gapped_hsp *>(get(nr * sizeof(hb_gapped_hsp)));
    auto *d_misc = static_cast<uint32_t *>(get(((size_t)ns + 2) * sizeof(uint32_t)));
    auto *d_ctx = static_cast<int32_t *>(get((size_t)3 * n_ctx * sizeof(int32_t)));
    auto *d_first = static_cast<uint32_t *>(get(((size_t)ns + nb + 4) * sizeof(uint32_t)));
    auto *d_gst = static_cast<hb_gapped_stats *>(get((size_t)ns * sizeof(hb_gapped_stats)));
    auto *d_gdense = static_cast<hb_gapped_hsp *>(get(nr * sizeof(hb_gapped_hsp)));
    auto *d_list = static_cast<uint32_t *>(get(((size_t)ns + 1) * sizeof(uint32_t)));
    auto *d_small = static_cast<uint2 *>(get(sizeof(uint2)));
    // the pair kernel's queues and the subjects that it leaves
    const bool pair = hb_gap_pair_ok(gp->gap_open, gp->gap_extend, gp->x_dropoff);
    auto *d_mid = static_cast<uint32_t *>(
        get(pair ? (HB_QUEUE_WORDS + 1 + (size_t)ns) * sizeof(uint32_t) : 0));
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    auto release = [&]() {
        for (void *p : held) hb_pool_put(c, p);
        for (hipEvent_t e : ev)
            if (e) hipEventDestroy(e);
    };
    if (oom) {
        release();
        return HB_ERR_NOMEM;
    }
    hipStream_t st = c->stream;
    std::vector<int32_t> hctx(3 * (size_t)n_ctx);
    for (int32_t i = 0; i < n_ctx; ++i) {
        hctx[i] = ctx_off[i];
        hctx[n_ctx + i] = ctx_len[i];
        hctx[2 * n_ctx + i] = gap_cutoff[i];
    }
    hb_gap_args a{};
    a.res = db->d_res;
    a.offs = db->d_offs;
    a.query = d_query;
    a.ctx = d_ctx;
    a.n_ctx = n_ctx;
    a.mat32 = d_mat;
    a.gap_open = gp->gap_open;
    a.gap_extend = gp->gap_extend;
    a.x_dropoff = gp->x_dropoff;
    a.ust = d_ust;
    a.urec = d_urec;
    a.n_subjects = ns;
    a.counter = d_misc;
    a.out = d_gout;
    a.st3 = d_st3;
    a.wide = d_misc + 1;
    a.list = d_list + 1;
    a.n_list = d_list;
    if (pair) {
        a.queues = d_mid;
        a.mid = d_mid + HB_QUEUE_WORDS;
    }
    uint32_t n_wide = 0;
    uint32_t *d_nbig = d_scr + ns + nb;
    hipError_t e = hb_launch_finalize(st3_in, ns, rec_in, (uint32_t)n, d_ust, d_urec, d_scr, d_big,
                                      kBig, d_nbig, 1 + 128, st);
    if (e == hipSuccess)
        e = hipMemcpyAsync(d_ctx, hctx.data(), hctx.size() * sizeof(int32_t),
                           hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hb_launch_gap_list(a, d_list + 1, d_list, d_nbig + 1, st);
    for (int i = 0; ms_out && e == hipSuccess && i < 4; ++i) e = hipEventCreate(&ev[i]);
    if (e == hipSuccess && ms_out) e = hipEventRecord(ev[0], st);
    if (pair) {
        if (e == hipSuccess)
            e = hb_launch_gap_pair(a, (c->n_cu * 8 + HB_QUEUES - 1) / HB_QUEUES * HB_QUEUES, st);
        a.list = a.mid + 1;
        a.n_list = a.mid;
    }
    if (e == hipSuccess) e = hb_launch_gapped(a, false, c->n_cu * 8, st);
    if (e == hipSuccess && ms_out) e = hipEventRecord(ev[1], st);
    // The dense layout and the copies out go behind the kernels with one wait
    // for all; up to kAtOnce of records are copied before their number is known.
    constexpr size_t kAtOnce = (size_t)1 << 20;
    const size_t w_st = stats ? (size_t)ns * sizeof(hb_gapped_stats) : 0;
    const size_t w_max = hsps ? (size_t)n * sizeof(hb_gapped_hsp) : 0;
    const size_t w_all = 64 + CopyOut::room(w_st) + w_max;
    const bool at_once = w_max <= kAtOnce && w_all <= CopyOut::kKeep;
    uint32_t *d_total = d_first + ns + nb + 1;
    CopyOut out(c, w_all <= CopyOut::kKeep ? w_all : 64 + std::max(w_st, w_max), st);
    size_t o_small = 0, o_st = 0, o_rec = 0;
    uint64_t total = 0;
    auto layout = [&]() {
        if (e == hipSuccess) e = hb_launch_first_index(d_st3, ns, d_first, d_first + ns, d_total, st);
        if (e == hipSuccess)
            e = hb_launch_gap_compact(a, d_first, d_total, d_gst, d_gdense, d_small, st);
        if (e != hipSuccess) return;
        out.rewind();
        o_small = out.add(d_small, sizeof(uint2));
        o_st = out.add(d_gst, w_st);
        if (at_once) o_rec = out.add(d_gdense, w_max);
        e = out.wait();
        uint2 v = make_uint2(0, 0);
        if (e == hipSuccess) memcpy(&v, out.ptr(o_small), sizeof(v));
        total = v.x;
        n_wide = v.y;
    };
    layout();
    if (e == hipSuccess && n_wide) {
        // subjects that outgrew the LDS capacities: same code, global scratch
        std::vector<uint32_t> wl(n_wide);
        std::vector<hb_subject_stats> ust(ns);
        e = hipMemcpy(wl.data(), d_misc + 2, n_wide * sizeof(uint32_t), hipMemcpyDeviceToHost);
        if (e == hipSuccess)
            e = hipMemcpy(ust.data(), d_ust, (size_t)ns * sizeof(hb_subject_stats),
                          hipMemcpyDeviceToHost);
        uint64_t longest = 0;
        uint32_t n_max = 1;
        for (uint32_t k : wl) {
            longest = std::max<uint64_t>(longest, db->h_offs[k + 1] - db->h_offs[k]);
            n_max = std::max(n_max, ust[k].n_hsp);
        }
        uint32_t ring = 64;
        while (ring < longest + 2) ring <<= 1;
        a.ring_wide = ring;
        a.n_max = n_max;
        a.scratch_words = (uint32_t)((2 * (uint64_t)ring + 7 * (uint64_t)n_max + 63) & ~63ull);
        const uint64_t per_wave = 4ull * a.scratch_words;
        uint64_t waves = std::min<uint64_t>(n_wide, 1024);
        waves = std::max<uint64_t>(1, std::min<uint64_t>(waves, ((uint64_t)1 << 30) / per_wave));
        const int blocks = (int)((waves + 3) / 4);
        a.scratch = static_cast<int32_t *>(get((size_t)blocks * 4 * per_wave));
        a.n_wide = n_wide;
        if (oom) e = hipErrorOutOfMemory;
        if (e == hipSuccess) e = hb_launch_fill_u32(d_misc, 0u, 1, st);
        if (e == hipSuccess && ms_out) e = hipEventRecord(ev[2], st);
        if (e == hipSuccess) e = hb_launch_gapped(a, true, blocks, st);
        if (e == hipSuccess && ms_out) e = hipEventRecord(ev[3], st);
        layout();
    }
    if (wide_out) *wide_out = n_wide;
    float ms = 0.f, ms2 = 0.f;
    if (e == hipSuccess && ms_out) e = hipEventElapsedTime(&ms, ev[0], ev[1]);
    if (e == hipSuccess && ms_out && n_wide) e = hipEventElapsedTime(&ms2, ev[2], ev[3]);
    if (ms_out) *ms_out = ms + ms2;
    if (e == hipSuccess) {
        if (n_hsp) *n_hsp = total;
        if (hsps && cap < total) {
            release();
            return HB_ERR_CAPACITY;
        }
        const size_t w_rec = hsps ? (size_t)total * sizeof(hb_gapped_hsp) : 0;
        const bool room = out.fits(w_rec);
        if (!at_once && room) o_rec = out.add(d_gdense, w_rec);   // while the stats move on
        if (w_st) out.store(stats, o_st, w_st);
        if (!at_once && !room) {
            out.rewind();
            o_rec = out.add(d_gdense, w_rec);
        }
        if (!at_once) e = out.wait();
        if (e == hipSuccess && w_rec) out.store(hsps, o_rec, w_rec);
    }
    if (e != hipSuccess) hipStreamSynchronize(st);   // the kernels that were launched
    release();
    if (e != hipSuccess) {
        hb_note_hip_error(e, "gapped stage", __LINE__);
        return e == hipErrorOutOfMemory ? HB_ERR_NOMEM : HB_ERR_DEVICE;
    }
    return HB_OK;
}

int hb_scan_gapped(hb_scan *s, const hb_gap_params *gp, const int32_t *gap_cutoff,
                   hb_gapped_stats *stats, hb_gapped_hsp *hsps, uint64_t cap, uint64_t *n_hsp)
{
    if (!s || !gap_params_ok(gp) || !gap_cutoff) return HB_ERR_ARG;
    int rc = hb_scan_wait(s);
    if (rc) return rc;
    if (n_hsp) *n_hsp = 0;
    hb_ctx *c = s->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    s->gap_ms = 0.f;
    s->gap_wide = 0;
    if (s->db->n == 0) return HB_OK;
    HB_CHECK(hipSetDevice(c->device));
    return gapped_core(c, s->db, s->q->gs.desc[0].query, s->q->gs.d_mat, s->q->ctx_off,
                       s->q->ctx_len, gap_cutoff, gp, s->d_stats, s->d_out, s->n_out, stats, hsps,
                       cap, n_hsp, &s->gap_ms, &s->gap_wide);
}

int hb_gapped_search(hb_ctx *c, hb_db *db, const uint8_t *seq, int32_t len, int32_t n_ctx,
                     const int32_t *ctx_off, const int32_t *ctx_len, const int8_t *matrix,
                     const hb_hsp *in, uint64_t n_in, const hb_gap_params *gp,
                     const int32_t *gap_cutoff, hb_gapped_stats *stats, hb_gapped_hsp *hsps,
                     uint64_t cap, uint64_t *n_hsp)
{
    if (!c || !db || db->ctx != c || !gap_params_ok(gp) || !gap_cutoff || (n_in && !in))
        return HB_ERR_ARG;
    if (n_hsp) *n_hsp = 0;
    std::vector<int32_t> xd(n_ctx > 0 ? n_ctx : 1, 1);
    int rc = hb_check_query(seq, len, n_ctx, ctx_off, ctx_len, xd.data());
    if (rc) return rc;
    if (n_in >= 0xffffffffull) return HB_ERR_UNSUPPORTED;
    // every record must lie inside its context and subject, on its diagonal
    for (uint64_t i = 0; i < n_in; ++i) {
        const hb_hsp &h = in[i];
        if (h.oid >= db->n || h.context < 0 || h.context >= n_ctx || h.len < 1) return HB_ERR_ARG;
        const int64_t c0 = ctx_off[h.context], c1 = c0 + ctx_len[h.context];
        const int64_t slen = (int64_t)(db->h_offs[h.oid + 1] - db->h_offs[h.oid]);
        if (h.q_start < c0 || (int64_t)h.q_start + h.len > c1 || h.s_start < 0 ||
            (int64_t)h.s_start + h.len > slen || h.q_off - h.s_off != h.q_start - h.s_start)
            return HB_ERR_ARG;
    }
    hb_resolved_params rp;
    hb_params p;
    hb_params_default(&p);
    p.matrix = matrix;
    rc = hb_resolve_params(&p, &rp);
    if (rc) return rc;
    std::lock_guard<std::mutex> lk(c->mu);
    HB_CHECK(hipSetDevice(c->device));
    if (db->n == 0) return HB_OK;
    const uint32_t ns = db->n;
    // matrix, query (and spare bytes), records
    const size_t o_rec = align256(1024 + (size_t)len + 64);
    const size_t b_in = o_rec + std::max<size_t>(n_in, 1) * sizeof(hb_hsp);
    const size_t b_st3 = (size_t)ns * 3 * sizeof(uint32_t);
    auto *d_in = static_cast<uint8_t *>(hb_pool_get(c, b_in));
    auto *d_st3 = static_cast<uint32_t *>(hb_pool_get(c, b_st3));
    auto release = [&]() {
        hb_pool_put(c, d_in);
        hb_pool_put(c, d_st3);
    };
    if (!d_in || !d_st3) {
        release();
        return HB_ERR_NOMEM;
    }
    auto *d_mat = reinterpret_cast<int8_t *>(d_in);
    uint8_t *d_q = d_in + 1024;
    auto *d_rec = reinterpret_cast<hb_hsp *>(d_in + o_rec);
    hipStream_t st = c->stream;
    // matrix, query and (up to kStage bytes of) records in one copy
    constexpr size_t kStage = (size_t)4 << 20;
    const size_t w_rec = n_in * sizeof(hb_hsp);
    const bool staged = w_rec <= kStage;
    size_t pin_b = o_rec + (staged ? w_rec : 0);
    auto *pin = static_cast<uint8_t *>(hb_pin_get(c, &pin_b));
    hipError_t e = pin ? hipSuccess : hipErrorOutOfMemory;
    if (e == hipSuccess) {
        memcpy(pin, rp.mat32, 1024);
        memcpy(pin + 1024, seq, (size_t)len);
        if (staged && n_in) memcpy(pin + o_rec, in, w_rec);
        e = hipMemcpyAsync(d_in, pin, o_rec + (staged ? w_rec : 0), hipMemcpyHostToDevice, st);
    }
    if (e == hipSuccess && !staged)
        e = hipMemcpyAsync(d_rec, in, w_rec, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hb_launch_fill_u32(d_st3, 0u, 3 * ns, st);
    if (e == hipSuccess) e = hb_launch_count_oids(d_rec, (uint32_t)n_in, d_st3, st);
    if (e != hipSuccess) {
        hipStreamSynchronize(st);
        if (pin) hb_pin_put(c, pin, pin_b);
        release();
        hb_note_hip_error(e, "hb_gapped_search", __LINE__);
        return HB_ERR_DEVICE;
    }
    std::vector<int32_t> co(ctx_off, ctx_off + n_ctx), cl(ctx_len, ctx_len + n_ctx);
    rc = gapped_core(c, db, d_q, d_mat, co, cl, gap_cutoff, gp, d_st3, d_rec, n_in, stats, hsps,
                     cap, n_hsp, nullptr, nullptr);
    if (rc) hipStreamSynchronize(st);   // (a call that succeeds has waited)
    hb_pin_put(c, pin, pin_b);
    release();
    return rc;
}

int hb_scan_gapped_info(hb_scan *s, float *ms, uint32_t *n_wide)
{
    if (!s) return HB_ERR_ARG;
    if (ms) *ms = s->gap_ms;
    if (n_wide) *n_wide = s->gap_wide;
    return HB_OK;
}

int hb_search(hb_ctx *c, hb_db *db, const uint8_t *seq, int32_t len, int32_t n_ctx,
              const int32_t *ctx_off, const int32_t *ctx_len, const int32_t *xdrop,
              const int32_t *cutoff, const hb_params *params, hb_subject_stats *stats,
              hb_hsp *hsps, uint64_t cap, uint64_t *n_hsp)
{
    hb_query *q = nullptr;
    int rc = hb_query_prepare(c, seq, len, n_ctx, ctx_off, ctx_len, xdrop, cutoff, params, &q);
    if (rc) return rc;
    hb_scan *s = nullptr;
    rc = hb_scan_start(c, db, q, &s);
    if (!rc) rc = hb_scan_results(s, stats, hsps, cap, n_hsp);
    if (s) hb_scan_free(s);
    hb_query_free(q);
    return rc;
}

// ------------------------------------------------------------------ diagnostics
int hb_diag_copy(hb_ctx *c, uint64_t bytes, int reps, float *ms_per_copy)
{
    if (!c || bytes < 16 || reps < 1 || !ms_per_copy) return HB_ERR_ARG;
    std::lock_guard<std::mutex> lk(c->mu);
    HB_CHECK(hipSetDevice(c->device));
    bytes &= ~(uint64_t)15;
    void *a = nullptr, *b = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = HB_OK;
    if (!(a = device_alloc(c->device, bytes)) || !(b = device_alloc(c->device, bytes))) {
        rc = HB_ERR_NOMEM;
    } else if (hipMemsetAsync(a, 1, bytes, c->stream) != hipSuccess ||
               hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess ||
               hb_launch_copy(b, a, bytes, c->stream) != hipSuccess ||
               hipEventRecord(e0, c->stream) != hipSuccess) {
        rc = HB_ERR_DEVICE;
    } else {
        for (int r = 0; r < reps && rc == HB_OK; ++r)
            if (hb_launch_copy(b, a, bytes, c->stream) != hipSuccess) rc = HB_ERR_DEVICE;
        float ms = 0;
        if (rc == HB_OK &&
            (hipEventRecord(e1, c->stream) != hipSuccess ||
             hipEventSynchronize(e1) != hipSuccess ||
             hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
            rc = HB_ERR_DEVICE;
        *ms_per_copy = ms / (float)reps;
    }
    if (e0) hipEventDestroy(e0);
    if (e1) hipEventDestroy(e1);
    hipFree(a);
    hipFree(b);
    return rc;
}

}  // extern "C"
