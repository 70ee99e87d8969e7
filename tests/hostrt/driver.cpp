// driver.cpp -- the host runtime over the stand-in of fake_hip.h (test
// infrastructure): `driver NAME` runs one scenario; exit status 0 = its
// checks hold.
#include "fake_hip.h"

#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "hb_runtime.h"

static int fails = 0;
#define CHECK(c)                                                               \
    do {                                                                       \
        if (!(c)) {                                                            \
            std::fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__); \
            ++fails;                                                           \
        }                                                                      \
    } while (0)

namespace {

struct Fixture {
    hb_ctx *c = nullptr;
    Fixture() { CHECK(hb_create(0, &c) == HB_OK); }
    ~Fixture()
    {
        if (c) CHECK(hb_destroy(c) == HB_OK);
    }
    // n subjects of `len` residues
    hb_db *database(uint32_t n, uint32_t len = 16, int rc = HB_OK)
    {
        std::vector<uint8_t> res((size_t)n * len + 1, 1);
        std::vector<uint64_t> offs(n + 1);
        for (uint32_t i = 0; i <= n; ++i) offs[i] = (uint64_t)i * len;
        hb_db *db = nullptr;
        CHECK(hb_db_upload(c, res.data(), offs.data(), n, &db) == rc);
        return db;
    }
    hb_batch *batch(hb_db *db, int queries, hipStream_t st = nullptr)
    {
        hb_batch_opts o;
        hb_batch_opts_default(&o);
        o.group_residues = 768;
        o.use_graph = 0;
        hb_batch *b = nullptr;
        CHECK(hb_batch_create_on(c, db, nullptr, &o, st, &b) == HB_OK);
        const std::vector<uint8_t> seq(100, 1);
        const int32_t off = 0, len = 100, x = 16, cut = 41;
        for (int i = 0; i < queries; ++i)
            CHECK(hb_batch_add(b, seq.data(), len, 1, &off, &len, &x, &cut, nullptr) == HB_OK);
        return b;
    }
    hb_query *query(int32_t len = 100)
    {
        const std::vector<uint8_t> seq(len, 1);
        const int32_t off = 0, x = 16, cut = 41;
        hb_query *q = nullptr;
        CHECK(hb_query_prepare(c, seq.data(), len, 1, &off, &len, &x, &cut, nullptr, &q) == HB_OK);
        return q;
    }
};

// Every scan finds n HSPs of query 0.
void found(uint32_t n)
{
    g_fake.scan = [n](const hb_scan_args &a) {
        for (uint32_t i = 0; i < n && i < a.out_cap; ++i) {
            memset(&a.out[i], 0, sizeof(hb_hsp));
            a.out[i].oid = i;
        }
        *a.out_count = n;
    };
}

// A pass whose results could not be collected leaves none.
void failed_collect()
{
    Fixture f;
    hb_db *db = f.database(10);
    found(7);
    hb_batch *b = f.batch(db, 2);
    uint64_t n = 99;
    g_fake.fail_order = 1;
    CHECK(hb_batch_run(b) == HB_ERR_DEVICE);
    CHECK(hb_batch_results(b, 0, nullptr, 0, &n) == HB_ERR_STATE);
    CHECK(hb_batch_run(b) == HB_OK);
    CHECK(hb_batch_results(b, 0, nullptr, 0, &n) == HB_OK && n == 7);
    g_fake.fail_order = 1;
    CHECK(hb_batch_run(b) == HB_ERR_DEVICE);
    CHECK(hb_batch_results(b, 1, nullptr, 0, &n) == HB_ERR_STATE);
    CHECK(hb_batch_run(b) == HB_OK);
    std::vector<hb_hsp> got(7);
    CHECK(hb_batch_results(b, 0, got.data(), 7, &n) == HB_OK && n == 7 && got[6].oid == 6);
    CHECK(hb_batch_results(b, 1, nullptr, 0, &n) == HB_OK && n == 0);
    hb_batch_free(b);
    hb_db_free(db);
}

// A call that fails has waited for what it enqueued: its buffers go back to
// the pool, and the next load fills them on other streams.
void failed_calls_wait()
{
    Fixture f;
    hb_db *db = f.database(20000);
    hb_query *q = f.query();
    found(20000);
    hb_scan *s = nullptr;
    CHECK(hb_scan_start(f.c, db, q, &s) == HB_OK && hb_scan_wait(s) == HB_OK);
    std::vector<hb_subject_stats> st(20000);
    std::vector<hb_subject_hits> sub(20000);
    std::vector<hb_hsp> hsps(20000);
    std::vector<hb_gapped_stats> gst(20000);
    std::vector<hb_gapped_hsp> g(20000);
    hb_scan_totals tot;
    hb_gap_params gp;
    hb_gap_params_default(&gp);
    const int32_t cut = 30;
    uint64_t n = 0;
    for (int how = 0; how < 2; ++how) {
        // no page-locked memory, or a kernel that cannot be launched
        std::atomic<int> &fail = how ? g_fake.fail_finalize : g_fake.fail_host_malloc;
        fail = 1;
        CHECK(hb_scan_results(s, st.data(), hsps.data(), hsps.size(), &n) == HB_ERR_DEVICE);
        CHECK(fake_pending(f.c->stream) == 0);
        fail = 1;
        CHECK(hb_scan_results_compact(s, sub.data(), sub.size(), hsps.data(), hsps.size(), &tot) ==
              HB_ERR_DEVICE);
        CHECK(fake_pending(f.c->stream) == 0);
        fail = 1;
        CHECK(hb_scan_gapped(s, &gp, &cut, gst.data(), g.data(), g.size(), &n) < 0);
        CHECK(fake_pending(f.c->stream) == 0);
        CHECK(fail == 0);
    }
    found(3);
    hipStream_t own = nullptr;
    CHECK(hipStreamCreateWithFlags(&own, hipStreamNonBlocking) == hipSuccess);
    hb_batch *b = f.batch(db, 1, own);
    g_fake.fail_order = 1;
    CHECK(hb_batch_run(b) == HB_ERR_DEVICE);
    CHECK(fake_pending(own) == 0);
    hb_batch_free(b);
    hb_scan_free(s);
    hb_query_free(q);
    hb_db_free(db);
}

// An allocation that fails and is handled leaves no error for the launches
// after it: the load takes the plain copy, and the next call works.
void handled_errors()
{
    const uint32_t n = 20000, len = 300;   // 6 MB: through page-locked chunks
    for (std::atomic<int> *fail : {&g_fake.fail_host_malloc, &g_fake.fail_stream_create}) {
        Fixture g;
        *fail = 1;
        const int copies = g_fake.host_to_device;
        hb_db *db = g.database(n, len);
        CHECK(*fail == 0 && g_fake.host_to_device == copies + 1);   // the residues
        hb_db_free(db);
    }
    Fixture f;
    const uint32_t m = 60000;   // results larger than the load's page-locked buffers
    hb_db *db = f.database(m);
    hb_query *q = f.query();
    found(5);
    hb_scan *s = nullptr;
    g_fake.fail_malloc = 2;
    CHECK(hb_scan_start(f.c, db, q, &s) == HB_ERR_NOMEM);
    g_fake.fail_malloc = 0;
    CHECK(hb_scan_start(f.c, db, q, &s) == HB_OK);
    CHECK(hb_scan_wait(s) == HB_OK);
    std::vector<hb_subject_stats> st(m);
    std::vector<hb_hsp> hsps(5);
    uint64_t found_n = 0;
    g_fake.fail_host_malloc = 1;
    CHECK(hb_scan_results(s, st.data(), hsps.data(), 5, &found_n) == HB_ERR_DEVICE);
    CHECK(hb_scan_results(s, st.data(), hsps.data(), 5, &found_n) == HB_OK && found_n == 5);
    // results past 16 MiB: the context's own buffer
    hb_scan_free(s);
    hb_db_free(db);
    const uint32_t many = 1 << 20;
    db = f.database(many, 1);
    CHECK(hb_scan_start(f.c, db, q, &s) == HB_OK);
    st.resize(many);
    g_fake.fail_host_malloc = 1;
    CHECK(hb_scan_results(s, st.data(), hsps.data(), 5, &found_n) == HB_ERR_DEVICE);
    CHECK(g_fake.fail_host_malloc == 0);
    CHECK(hb_scan_results(s, st.data(), hsps.data(), 5, &found_n) == HB_OK);
    void *p = nullptr;
    g_fake.fail_host_malloc = 1;
    CHECK(hb_host_alloc(f.c, 64, &p) == HB_ERR_NOMEM);
    CHECK(hb_scan_results(s, st.data(), hsps.data(), 5, &found_n) == HB_OK);
    float ms = 0;
    g_fake.fail_malloc = 2;
    CHECK(hb_diag_copy(f.c, 4096, 1, &ms) == HB_ERR_NOMEM);
    CHECK(hb_scan_results(s, st.data(), hsps.data(), 5, &found_n) == HB_OK);
    // a batch whose order finds no memory orders on the host
    hb_batch *b = f.batch(db, 1);
    CHECK(hb_batch_run(b) == HB_OK);
    f.c->pool_mu.lock();
    for (auto &x : f.c->pool) (void)hipFree(x.p);
    f.c->pool.clear();
    f.c->pool_bytes = f.c->pool_db_bytes = 0;
    f.c->pool_mu.unlock();
    g_fake.fail_malloc = 2;
    CHECK(hb_batch_run(b) == HB_OK);
    g_fake.fail_malloc = 0;
    CHECK(hb_batch_results(b, 0, nullptr, 0, &found_n) == HB_OK && found_n == 5);
    CHECK(hb_scan_results(s, st.data(), hsps.data(), 5, &found_n) == HB_OK);
    hb_batch_free(b);
    hb_scan_free(s);
    hb_query_free(q);
    hb_db_free(db);
}

// Buffers keep their sizes in the pool whatever they served: databases of
// alternating sizes take no more memory after the first round of them, and the
// pool's bytes are the device's.
void pool_sizes()
{
    Fixture f;
    // of three buffers asked for in turn the first serves the second
    void *a = hb_pool_get(f.c, 1000000);
    hb_pool_put(f.c, a);
    void *b = hb_pool_get(f.c, 600000);
    CHECK(a == b && hb_pool_held(f.c) == 0);
    hb_pool_put(f.c, b);
    CHECK(hb_pool_held(f.c) == 1000000);
    b = hb_pool_get(f.c, 1000000);
    CHECK(a == b);
    hb_pool_put(f.c, b);
    int mallocs = 0;
    for (int round = 0; round < 4; ++round) {
        for (uint32_t n : {90000u, 50000u, 90000u, 60000u}) hb_db_free(f.database(n, 100));
        CHECK(hb_pool_held(f.c) == g_fake.device_used);
        if (round) CHECK(g_fake.mallocs == mallocs);
        mallocs = g_fake.mallocs;
    }
    // past 16 GiB the oldest go, by their own sizes
    std::vector<void *> p;
    for (int i = 0; i < 20; ++i) p.push_back(hb_pool_get(f.c, (size_t)1 << 30));
    for (void *x : p) hb_pool_put(f.c, x);
    CHECK(hb_pool_held(f.c) <= (size_t)16 << 30 && hb_pool_held(f.c) == g_fake.device_used);
    for (int i = 0; i < 16; ++i) p[i] = hb_pool_get(f.c, (size_t)6 << 27);
    for (int i = 0; i < 16; ++i) hb_pool_put(f.c, p[i]);
    CHECK(hb_pool_held(f.c) <= (size_t)16 << 30 && hb_pool_held(f.c) == g_fake.device_used);
}

// What a freed database held is free again: for the memory information, for a
// server's default budget, for another context; and little of it is kept.
void freed_memory()
{
    const size_t total = g_fake.device_total;
    Fixture f, other;
    uint64_t before = 0, after = 0;
    CHECK(hb_mem_info(f.c, &before, nullptr) == HB_OK);
    for (uint32_t n : {100000u, 400000u, 50000u}) {
        hb_db_free(f.database(n, 100));
        CHECK(hb_mem_info(f.c, &after, nullptr) == HB_OK && after == before);
        CHECK(hb_pool_held(f.c) == g_fake.device_used);
    }
    std::vector<void *> p;
    for (int i = 0; i < 5; ++i) p.push_back(hb_pool_get(f.c, 300000000));
    for (void *x : p) hb_pool_put(f.c, x, true);
    CHECK(hb_pool_held(f.c) == 900000000);   // the last three, and no older ones
    hb_pool_put(f.c, hb_pool_get(f.c, 1200000000), true);
    CHECK(hb_pool_held(f.c) == 900000000 && g_fake.device_used == 900000000);
    CHECK(hb_mem_info(f.c, &after, nullptr) == HB_OK && after == before);
    // a context that needs what another keeps
    hb_db_free(f.database(1000000, 100));
    CHECK(hb_pool_held(f.c) > 200000000);
    g_fake.device_total = 280000000;
    hb_db *db = other.database(1000000, 100);
    CHECK(db && hb_pool_held(f.c) == 0);
    hb_db_free(db);
    float ms = 0;
    CHECK(hb_diag_copy(f.c, 100000000, 1, &ms) == HB_OK);
    // half the free memory, whatever the context keeps of it
    g_fake.device_total = 120000000;
    hb_db_free(f.database(400000, 100));
    CHECK(hb_pool_held(f.c) > 80000000);
    db = f.database(1000);
    found(5);
    hb_serve_opts o;
    hb_serve_opts_default(&o);
    o.hsp_per_cell = 30e6 / 32 / (100 * 16000.0);   // about 31 MB for the request
    hb_server *s = nullptr;
    CHECK(hb_serve_start(f.c, db, nullptr, &o, &s) == HB_OK);
    const std::vector<uint8_t> seq(100, 1);
    const int32_t off = 0, len = 100, x = 16, cut = 41;
    uint64_t t = 0, n = 0;
    CHECK(hb_serve_submit(s, seq.data(), len, 1, &off, &len, &x, &cut, &t) == HB_OK);
    CHECK(hb_serve_wait(s, t, -1) == HB_OK);
    CHECK(hb_serve_results(s, t, nullptr, 0, &n) == HB_OK && n == 5);
    hb_serve_stop(s);
    hb_db_free(db);
    g_fake.device_total = total;
}

// Page-locked buffers: a small request leaves a large one alone, the smallest
// that fits is taken, and the buffers kept stay within their bounds.
void pinned_buffers()
{
    Fixture f;
    hb_db *db = f.database(20000, 300);   // leaves the upload's 16 MiB
    found(5);
    hb_batch *b = f.batch(db, 1);
    CHECK(hb_batch_run(b) == HB_OK);      // holds a small one
    const size_t before = g_fake.host_used;
    hb_db *db2 = f.database(20000, 300);
    CHECK(g_fake.host_used < before + (1 << 20));   // no new 16 MiB
    auto get = [&](size_t bytes) {
        std::pair<void *, size_t> r(nullptr, bytes);
        r.first = hb_pin_get(f.c, &r.second);
        CHECK(r.first && r.second >= bytes && fake_host_size(r.first) == r.second);
        return r;
    };
    const auto big = get(8 << 20), mid = get(1 << 20);
    hb_pin_put(f.c, big.first, big.second);
    hb_pin_put(f.c, mid.first, mid.second);
    const int n = g_fake.host_mallocs;
    const auto one = get(900 << 10);
    CHECK(one.first == mid.first && g_fake.host_mallocs == n);
    const auto two = get(5 << 20);
    CHECK(two.first == big.first && g_fake.host_mallocs == n);
    hb_pin_put(f.c, one.first, one.second);
    hb_pin_put(f.c, two.first, two.second);
    std::vector<std::pair<void *, size_t>> all;
    for (int i = 0; i < 12; ++i) all.push_back(get(16 << 20));
    for (const auto &x : all) hb_pin_put(f.c, x.first, x.second);
    CHECK(f.c->pins.size() == 8 && f.c->pins.back().first == all.back().first);
    const size_t held = g_fake.host_used;
    const auto large = get((16 << 20) + 1);
    hb_pin_put(f.c, large.first, large.second);
    CHECK(g_fake.host_used == held && f.c->pins.size() == 8);
    hb_batch_free(b);
    hb_db_free(db);
    hb_db_free(db2);
}

// Residues in memory that the runtime knows, page-locked or on the device, are
// copied by the runtime from where they are and not read by the host.
void upload_sources()
{
    Fixture f;
    const uint32_t n = 20000, len = 300;
    std::vector<uint64_t> offs(n + 1);
    for (uint32_t i = 0; i <= n; ++i) offs[i] = (uint64_t)i * len;
    void *host = nullptr, *device = nullptr;
    CHECK(hipHostMalloc(&host, n * len, 0) == hipSuccess && hipMalloc(&device, n * len) == hipSuccess);
    for (void *src : {host, device}) {
        memset(src, 1, n * len);
        g_fake.async_bytes = 0;
        hb_db *db = nullptr;
        CHECK(hb_db_upload(f.c, static_cast<const uint8_t *>(src), offs.data(), n, &db) == HB_OK);
        CHECK(g_fake.async_from == src && g_fake.async_bytes == n * len);
        hb_db_free(db);
    }
    (void)hipHostFree(host);
    (void)hipFree(device);
}

// A served batch orders its records within the budget: on the device when that
// leaves room, on the host otherwise.
void served_order()
{
    Fixture f;
    hb_db *db = f.database(20000);
    const uint32_t n = 20000;   // 1.1 MB for their order
    found(n);
    const std::vector<uint8_t> seq(100, 1);
    const int32_t off = 0, len = 100, x = 16, cut = 41;
    for (int64_t room : {1 << 14, 1 << 24}) {
        hb_serve_opts o;
        hb_serve_opts_default(&o);
        o.hsp_per_cell = 20000 / (100.0 * 320000);
        o.max_inflight = 1;
        // the request's estimate (records, tables, entries) and `room`
        o.mem_budget = (20000 + 256) * 32 + 32768 * 8 + 4096 + 4096 + 8192 + 64 * 4 * 100 + room;
        hb_server *s = nullptr;
        CHECK(hb_serve_start(f.c, db, nullptr, &o, &s) == HB_OK);
        const int orders = g_fake.orders;
        uint64_t t = 0, k = 0;
        CHECK(hb_serve_submit(s, seq.data(), len, 1, &off, &len, &x, &cut, &t) == HB_OK);
        CHECK(hb_serve_wait(s, t, -1) == HB_OK);
        std::vector<hb_hsp> got(n);
        CHECK(hb_serve_results(s, t, got.data(), n, &k) == HB_OK && k == n && got[n - 1].oid == n - 1);
        hb_serve_stats st;
        CHECK(hb_serve_stats_get(s, &st) == HB_OK);
        CHECK(st.peak_bytes <= (uint64_t)o.mem_budget);
        const bool device = room > (1 << 20);
        CHECK((g_fake.orders != orders) == device);
        CHECK((st.peak_bytes > (uint64_t)(o.mem_budget - room)) == device);
        hb_serve_stop(s);
    }
    hb_db_free(db);
}

// A database outlives its context.
void database_after_context()
{
    hb_db *db = nullptr;
    {
        Fixture f;
        db = f.database(1000);
    }
    CHECK(g_fake.device_used > 0);
    CHECK(hb_db_free(db) == HB_OK);
    CHECK(g_fake.device_used == 0);
    Fixture f;   // (a context that may stand at the same address)
    hb_db_free(f.database(1000));
    CHECK(hb_pool_held(f.c) == g_fake.device_used);
}

// The order on the host: by query, subject and offsets, with the query's own
// contexts and offsets.
void host_order()
{
    Fixture f;
    hb_db *db = f.database(20000);
    constexpr uint32_t kQueries = 48;
    for (uint32_t n : {0u, 1u, 1000u, 65535u, 65536u, 1500000u}) {
        std::vector<uint32_t> perm(n);
        for (uint32_t i = 0; i < n; ++i) perm[i] = (uint32_t)((i * 2654435761ull + 12345) % n);
        std::vector<hb_hsp> all(n);   // each value of perm may stand more than once: s_off tells
        for (uint32_t i = 0; i < n; ++i) {
            memset(&all[i], 0, sizeof(hb_hsp));
            all[i].oid = perm[i] / 64 % 20000;
            all[i].s_off = (int32_t)(perm[i] % 64);
            all[i].q_off = (int32_t)i;   // (a unique one; made relative below)
        }
        g_fake.scan = [&](const hb_scan_args &a) {
            // five queries of 100 residues and 40 between them to a group of 768
            for (uint32_t i = 0; i < n && i < a.out_cap; ++i) {
                a.out[i] = all[i];
                a.out[i].context = (int32_t)(i % kQueries);
            }
            *a.out_count = n;
        };
        hipStream_t st = nullptr;
        CHECK(hipStreamCreateWithFlags(&st, 0) == hipSuccess);
        hb_batch *b = f.batch(db, kQueries, st);
        CHECK(hb_batch_reserve(b, n + 1) == HB_OK && hb_batch_launch(b) == HB_OK);
        const int orders = g_fake.orders;
        size_t room = 0;
        CHECK(hb_batch_finish(b, &room) == HB_OK && room == 0 && g_fake.orders == orders);
        uint64_t sum = 0;
        for (uint32_t q = 0; q < kQueries; ++q) {
            uint64_t k = 0;
            std::vector<hb_hsp> got(n);
            CHECK(hb_batch_results(b, (int32_t)q, got.data(), n, &k) == HB_OK);
            sum += k;
            int32_t base = 0;   // the query's place in its group, the same for all its records
            for (uint64_t i = 0; i < k; ++i) {
                const hb_hsp &x = got[i];
                CHECK(x.context == 0);
                if (i == 0) base = -x.q_start;
                const uint32_t from = (uint32_t)(x.q_off + base);
                CHECK(x.q_start == -base && from < n && all[from].oid == x.oid &&
                      all[from].s_off == x.s_off && base % 140 == 0);
                if (i == 0) continue;
                const hb_hsp &y = got[i - 1];
                CHECK(y.oid < x.oid ||
                      (y.oid == x.oid &&
                       (y.s_off < x.s_off || (y.s_off == x.s_off && y.q_off < x.q_off))));
            }
        }
        CHECK(sum == n);
        hb_batch_free(b);
    }
    hb_db_free(db);
}

const struct {
    const char *name;
    void (*run)();
} kScenarios[] = {
    {"failed_collect", failed_collect},
    {"failed_calls_wait", failed_calls_wait},
    {"handled_errors", handled_errors},
    {"pool_sizes", pool_sizes},
    {"freed_memory", freed_memory},
    {"pinned_buffers", pinned_buffers},
    {"upload_sources", upload_sources},
    {"served_order", served_order},
    {"database_after_context", database_after_context},
    {"host_order", host_order},
};

}  // namespace

int main(int argc, char **argv)
{
    for (const auto &s : kScenarios)
        if (argc > 1 && std::string(argv[1]) == s.name) {
            s.run();
            return fails ? 1 : 0;
        }
    std::fprintf(stderr, "no such scenario\n");
    return 2;
}
