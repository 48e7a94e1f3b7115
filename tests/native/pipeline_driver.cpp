// Host-only driver for the streaming pipeline (la_pipeline_*), built with g++
// together with csrc/pipeline.hip by tests/test_native_sanitizers.py, on a
// simulated HIP runtime: streams are queues on the CPU, kernels and copies are
// functions run from them, and memory is what the driver registers.  The queues
// run as late as they may (only what a wait or a synchronisation asks for) or at
// once, so a missing wait shows as a wrong result each time, not now and then,
// and every HIP call that submits work can be made to fail.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <memory>
#include <random>
#include <vector>

#include "layer_adam.h"
#include "link_step.h"

#define CHECK(c)                                                              \
    do {                                                                      \
        if (!(c)) {                                                           \
            std::fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__); \
            std::exit(1);                                                     \
        }                                                                     \
    } while (0)

// ---------------------------------------------------------------------------
// the simulated runtime
// ---------------------------------------------------------------------------
struct Stream;
struct Event {
    Stream* stream = nullptr;
    uint64_t recorded = 0, done = 0;
};
struct Op {
    std::function<void()> run;       // reads or writes memory
    Event* wait = nullptr;           // or: waits for a record of an event, or records one
    Event* record = nullptr;
    uint64_t version = 0;
    Stream* of = nullptr;            // the stream of the record waited for
    bool callers = false;            // the caller's own work, not the pipeline's
};
struct Stream {
    std::deque<Op> q;
};
struct Region {
    char* base;
    size_t size;
    bool device;
    unsigned flags;
};

static bool g_lazy = true;
static int g_fail_at = -1, g_submitted = 0;
static int g_copies = 0, g_updates = 0, g_links = 0;
static Stream g_null;
static std::vector<Stream*> g_streams = {&g_null};
static std::vector<std::unique_ptr<Event>> g_events;   // waits in queues keep destroyed events alive
static std::vector<Region> g_regions;

static void run_one(Stream* s)
{
    Op op = s->q.front();
    s->q.pop_front();
    if (op.wait)
        while (op.wait->done < op.version) run_one(op.of);
    if (op.run) op.run();
    if (op.record && op.record->done < op.version) op.record->done = op.version;
}
static void run_all(Stream* s)
{
    while (!s->q.empty()) run_one(s);
}
static Stream* stream(hipStream_t s) { return s ? reinterpret_cast<Stream*>(s) : &g_null; }
static void push(Stream* s, Op op)
{
    s->q.push_back(std::move(op));
    if (!g_lazy) run_all(s);
}
static bool fails() { return g_submitted++ == g_fail_at; }
// queued work of the pipeline that will read or write memory
static int work_queued()
{
    int n = 0;
    for (Stream* s : g_streams)
        for (const Op& op : s->q) n += op.run && !op.callers ? 1 : 0;
    return n;
}
static const Region* region(const void* p)
{
    for (const Region& r : g_regions)
        if (p >= r.base && p < r.base + r.size) return &r;
    return nullptr;
}

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    g_streams.push_back(new Stream);
    *s = reinterpret_cast<hipStream_t>(g_streams.back());
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    CHECK(stream(s)->q.empty());
    for (size_t i = 0; i < g_streams.size(); ++i)
        if (g_streams[i] == stream(s)) g_streams.erase(g_streams.begin() + static_cast<long>(i));
    delete stream(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { run_all(stream(s)); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e)
{
    g_events.emplace_back(new Event);
    *e = reinterpret_cast<hipEvent_t>(g_events.back().get());
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.0f; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (fails()) return hipErrorUnknown;
    Event* ev = reinterpret_cast<Event*>(e);
    ev->stream = stream(s);
    Op op;
    op.record = ev;
    op.version = ++ev->recorded;
    push(stream(s), op);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    Event* ev = reinterpret_cast<Event*>(e);
    const uint64_t until = ev->recorded;
    while (ev->done < until) run_one(ev->stream);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    if (fails()) return hipErrorUnknown;
    Event* ev = reinterpret_cast<Event*>(e);
    Op op;
    op.wait = ev;
    op.version = ev->recorded;
    op.of = ev->stream;
    push(stream(s), op);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t s)
{
    if (fails()) return hipErrorUnknown;
    ++g_copies;
    Op op;
    op.run = [=] { std::memcpy(dst, src, bytes); };
    push(stream(s), op);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    const Region* r = region(p);
    if (!r) return hipErrorInvalidValue;
    a->type = r->device ? hipMemoryTypeDevice : hipMemoryTypeHost;
    a->device = 0;
    a->devicePointer = const_cast<void*>(p);
    return hipSuccess;
}
hipError_t hipHostGetFlags(unsigned* flags, void* p)
{
    const Region* r = region(p);
    if (!r || r->device) return hipErrorInvalidValue;
    *flags = r->flags;
    return hipSuccess;
}
hipError_t hipPointerGetAttribute(void* data, hipPointer_attribute what, hipDeviceptr_t p)
{
    const Region* r = region(p);
    if (!r) return hipErrorInvalidValue;
    if (what == HIP_POINTER_ATTRIBUTE_RANGE_START_ADDR) *static_cast<void**>(data) = r->base;
    else if (what == HIP_POINTER_ATTRIBUTE_RANGE_SIZE) *static_cast<size_t*>(data) = r->size;
    else return hipErrorInvalidValue;
    return hipSuccess;
}
}  // extern "C"

// ---------------------------------------------------------------------------
// the update: element by element, of any splitting the same
// ---------------------------------------------------------------------------
static void update(float* p, const float* g, float* m, float* v, uint16_t* out, uint64_t n)
{
    for (uint64_t i = 0; i < n; ++i) {
        m[i] = 0.5f * m[i] + g[i];
        v[i] = 0.25f * v[i] + g[i] * g[i];
        p[i] -= 0.125f * m[i] + 0.0625f * v[i];
        if (out) {
            uint32_t u;
            std::memcpy(&u, p + i, 4);
            out[i] = static_cast<uint16_t>(u >> 16);
        }
    }
}
static int launch(void* p, const void* g, void* m, void* v, uint64_t n, uint16_t* out, hipStream_t st, bool host_too)
{
    if (fails()) return LA_EINVAL;
    for (const void* a : {static_cast<const void*>(p), g, static_cast<const void*>(m), static_cast<const void*>(v),
                          static_cast<const void*>(out)}) {
        if (!a) continue;
        const Region* r = region(a);                 // what a kernel may touch
        CHECK(r && (r->device || (host_too && r->flags == 0)));
    }
    Op op;
    op.run = [=] {
        update(static_cast<float*>(p), static_cast<const float*>(g), static_cast<float*>(m), static_cast<float*>(v), out, n);
    };
    push(stream(st), op);
    return LA_OK;
}
extern "C" int la_adamw_step(const la_scalars_t*, int, void* p, int, const void* g, int, void* m, void* v, uint64_t n,
                             uint16_t* out, const float*, la_stream_t st)
{
    if (n == 0) return LA_OK;
    ++g_updates;
    return launch(p, g, m, v, n, out, static_cast<hipStream_t>(st), false);
}
namespace la_link {
int step(const la_scalars_t&, int, void* p, int, const void* g, int, void* m, void* v, uint64_t n, uint16_t* out,
         const float*, unsigned link_read, hipStream_t st)
{
    ++g_links;
    unsigned host = 0;   // what it reads of host memory
    for (const void* x : {static_cast<const void*>(p), g, static_cast<const void*>(m), static_cast<const void*>(v)})
        host += region(x)->device ? 0u : 4u;
    CHECK(link_read == host);
    return launch(p, g, m, v, n, out, st, true);
}
}  // namespace la_link

// ---------------------------------------------------------------------------
// the cases
// ---------------------------------------------------------------------------
// Where an array lives: device memory, page-locked memory that kernels reach,
// page-locked memory that they do not, or pageable memory.
enum Place { kDevice, kLocked, kCoarse, kPageable };

struct Buffer {
    char* at = nullptr;
    Buffer(uint64_t bytes, Place place) : at(static_cast<char*>(std::aligned_alloc(256, (bytes + 511) / 256 * 256)))
    {
        if (place != kPageable)
            g_regions.push_back({at, (bytes + 511) / 256 * 256, place == kDevice, place == kCoarse ? hipHostMallocPortable : 0u});
    }
    ~Buffer()
    {
        for (size_t i = 0; i < g_regions.size(); ++i)
            if (g_regions[i].base == at) {
                g_regions.erase(g_regions.begin() + static_cast<long>(i));
                break;
            }
        std::free(at);
    }
    Buffer(const Buffer&) = delete;
    Buffer& operator=(const Buffer&) = delete;
    float* f() { return reinterpret_cast<float*>(at); }
};

struct Layout {
    const char* name;
    Place p, mv, g, out;
    bool staging;
    bool direct;      // the path that the rule takes
};
static const Layout kLayouts[] = {
    {"all page-locked", kLocked, kLocked, kLocked, kDevice, false, true},
    {"page-locked, moments on the device", kLocked, kDevice, kDevice, kLocked, false, true},
    {"pageable, staged", kPageable, kPageable, kLocked, kDevice, true, true},
    {"pageable grads, staged", kDevice, kDevice, kPageable, kDevice, true, true},
    {"pageable, not staged", kPageable, kPageable, kPageable, kPageable, false, false},
    {"coarse", kCoarse, kCoarse, kLocked, kDevice, false, false},
    {"coarse master, pageable rest staged", kCoarse, kPageable, kPageable, kPageable, true, false},
    {"coarse copy, pageable grads staged", kDevice, kDevice, kPageable, kCoarse, true, false},
};

constexpr uint64_t kChunk = 256, kParts = 4;

struct Run {
    const Layout& l;
    uint64_t n;                       // elements of a part
    Buffer p, m, v, g, out, ws, staging;
    std::vector<float> rp, rm, rv, rg;
    std::vector<uint16_t> ro;
    la_pipeline_t* pl = nullptr;
    la_scalars_t sc{};
    std::mt19937 rng{7};
    Run(const Layout& layout, uint64_t part, int slots, int threads)
        : l(layout), n(part), p(bytes(4), l.p), m(bytes(4), l.mv), v(bytes(4), l.mv), g(bytes(4), l.g),
          out(bytes(2), l.out), ws(need(slots), kDevice), staging(need(slots), kLocked), rp(part * kParts),
          rm(rp.size()), rv(rp.size()), rg(rp.size()), ro(rp.size())
    {
        for (std::vector<float>* x : {&rp, &rm, &rv, &rg})
            for (float& e : *x) e = static_cast<float>(rng() % 2000) / 1000.0f - 1.0f;
        std::memcpy(p.f(), rp.data(), rp.size() * 4);
        std::memcpy(m.f(), rm.data(), rm.size() * 4);
        std::memcpy(v.f(), rv.data(), rv.size() * 4);
        std::memset(g.at, 0, bytes(4));
        std::memset(out.at, 0, bytes(2));
        CHECK(la_pipeline_create(kChunk, slots, &pl) == LA_OK);
        if (l.staging) CHECK(la_pipeline_set_host_staging(pl, staging.at, need(slots), threads) == LA_OK);
        ws_bytes = need(slots);
    }
    ~Run()
    {
        CHECK(la_pipeline_destroy(pl) == LA_OK);
        run_all(&g_null);
    }
    uint64_t ws_bytes = 0;
    uint64_t bytes(uint64_t elem) const { return n * kParts * elem; }
    static uint64_t need(int slots)
    {
        return la_pipeline_workspace_bytes(kChunk, slots, LA_F32, LA_F32, LA_F32, LA_ON_HOST_ALL);
    }
    unsigned mask() const
    {
        return (l.p == kDevice ? 0u : LA_ON_HOST_P) | (l.mv == kDevice ? 0u : LA_ON_HOST_M | LA_ON_HOST_V) |
               (l.g == kDevice ? 0u : LA_ON_HOST_G) | (l.out == kDevice ? 0u : LA_ON_HOST_OUT);
    }
    // one call on part k; the caller's stream holds the work that makes its grads
    int step(uint64_t k, bool wait)
    {
        const uint64_t at = k * n;
        std::vector<float> fresh(n);
        for (float& e : fresh) e = static_cast<float>(rng() % 2000) / 1000.0f - 1.0f;
        std::memcpy(rg.data() + at, fresh.data(), n * 4);
        update(rp.data() + at, rg.data() + at, rm.data() + at, rv.data() + at, ro.data() + at, n);
        float* to = g.f() + at;
        Op make;
        make.callers = true;
        make.run = [to, fresh] { std::memcpy(to, fresh.data(), fresh.size() * 4); };
        push(&g_null, make);
        la_pipeline_stats_t st;
        return la_pipeline_step(pl, &sc, LA_F32, p.f() + at, LA_F32, to, LA_F32, m.f() + at, v.f() + at, n,
                                reinterpret_cast<uint16_t*>(out.at) + at, mask(), nullptr, ws.at, ws_bytes, nullptr,
                                wait ? 1 : 0, wait ? &st : nullptr);
    }
    bool same() const
    {
        return !std::memcmp(p.at, rp.data(), bytes(4)) && !std::memcmp(m.at, rm.data(), bytes(4)) &&
               !std::memcmp(v.at, rv.data(), bytes(4)) && !std::memcmp(out.at, ro.data(), bytes(2));
    }
};

// Calls that wait and calls that return once queued, in random order on the
// parts of a layer: what a waiting call or a sync leaves is the reference's.
// `engines`: by copy engines; `turns`: asked for them now and then.
static void results(const Layout& l, uint64_t n, int slots, int threads, bool engines, bool turns)
{
    Run r(l, n, slots, threads);
    CHECK(la_pipeline_use_copy_engines(r.pl, engines ? 1 : 0) == LA_OK);
    std::mt19937 rng(static_cast<unsigned>(n) * 31u + static_cast<unsigned>(slots));
    g_copies = g_updates = g_links = 0;
    for (int call = 0; call < 24; ++call) {
        const bool wait = rng() % 4 == 0;
        if (turns && rng() % 3 == 0) CHECK(la_pipeline_use_copy_engines(r.pl, static_cast<int>(rng() % 2)) == LA_OK);
        CHECK(r.step(rng() % kParts, wait) == LA_OK);
        if (wait) {
            CHECK(work_queued() == 0);
            CHECK(r.same());
        }
    }
    CHECK(la_pipeline_sync(r.pl) == LA_OK);
    run_all(&g_null);
    CHECK(work_queued() == 0);
    CHECK(r.same());
    const bool direct = l.direct && !engines;
    CHECK(turns || (direct ? g_links > 0 && g_updates == 0 && g_copies == 0
                           : g_links == 0 && g_updates > 0 && g_copies > 0));
}

// Every submission of a call fails in turn: once the call has returned its
// error, nothing that it or an earlier call queued reads or writes memory any more.
static void failures(const Layout& l, uint64_t n, int slots, bool wait, bool behind_others, bool engines)
{
    for (int k = 0;; ++k) {
        Run r(l, n, slots, 2);
        CHECK(la_pipeline_use_copy_engines(r.pl, engines) == LA_OK);
        if (behind_others) CHECK(r.step(0, false) == LA_OK && r.step(1, false) == LA_OK);
        g_submitted = 0;
        g_fail_at = k;
        const int rc = r.step(2, wait);
        const bool reached = g_submitted > k;
        g_fail_at = -1;
        CHECK(reached == (rc != LA_OK));
        if (!reached) break;
        CHECK(work_queued() == 0);
        CHECK(la_pipeline_sync(r.pl) == LA_OK);
    }
}

// Sub-chunks of staged arrays: an eighth of the call, at least so many elements
// that a round of the host threads copies enough, unless there is little in all.
// The build's bounds are 32 and 128 elements of 24 staged bytes, kAloneBytes 1024.
static int sub_chunks(const Layout& l, uint64_t n)
{
    Run r(l, n, 2, 2);
    g_links = 0;
    CHECK(r.step(0, true) == LA_OK && r.same());
    return g_links;
}

int main()
{
    const Layout grads = {"pageable grads", kDevice, kDevice, kPageable, kDevice, true, true};
    const Layout state = {"pageable state", kPageable, kPageable, kDevice, kDevice, true, true};
    CHECK(sub_chunks(state, 1100) == 9);    // 24 bytes an element: most 128
    CHECK(sub_chunks(grads, 1000) == 8);    // 4 bytes, 4000 in all: eighths
    CHECK(sub_chunks(grads, 1100) == 6);    // 4 bytes: at least 6 x 32
    CHECK(sub_chunks(grads, 5000) == 20);   // and at most 6 x 128, here the chunk's 256
    CHECK(la_pipeline_use_copy_engines(nullptr, 1) == LA_EINVAL);
    for (const bool lazy : {true, false}) {
        g_lazy = lazy;
        for (const Layout& l : kLayouts)
            for (const uint64_t n : {1ull, 17ull, 256ull, 1000ull, 5000ull})
                for (const int slots : {1, 2, 3}) {
                    std::printf("%s, %llu elements, %d slots, %s\n", l.name, static_cast<unsigned long long>(n), slots,
                                lazy ? "late" : "at once");
                    std::fflush(stdout);
                    results(l, n, slots, 1 + slots, false, false);
                    results(l, n, slots, 1 + slots, true, false);
                    results(l, n, slots, 1 + slots, false, true);
                }
    }
    g_lazy = true;
    for (const Layout& l : kLayouts)
        for (const bool wait : {true, false}) {
            std::printf("%s, failing, %s\n", l.name, wait ? "waiting" : "queued");
            std::fflush(stdout);
            for (const bool engines : {false, true}) {
                failures(l, 3000, 2, wait, false, engines);
                failures(l, 1000, 2, wait, true, engines);
            }
        }
    std::printf("pipeline driver ok\n");
    return 0;
}
