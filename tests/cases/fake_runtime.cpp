// The library's host code on a stand-in for the HIP runtime: host memory in the place of device
// memory, kernels that do nothing, and streams that only count what was queued and what is known
// to be done.  Work stays "running" until something waits for it, so a block of memory that is
// handed out while an earlier user may still be running shows on every run, without a GPU.
// Linked with the library's sources compiled for the host alone; one scenario per run (argv[1]).
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "preprocess.h"

// ---------------------------------------------------------------------------------------------
// the stand-in
// ---------------------------------------------------------------------------------------------
struct FakeStream {
    int device = 0;
    long queued = 0, done = 0;
    std::map<FakeStream *, long> behind;          // ... and waits, on the device, for so much of others
};
struct FakeEvent {
    FakeStream *s = nullptr;
    long tick = 0;
};

static FakeStream g_null[2];                      // two devices
static int g_device = 0;
static bool g_refuse_host_waits = false, g_refuse_events = false;
static int g_host_waits = 0, g_frees = 0, g_pinned = 0;
static long g_mallocs_left = -1;                  // -1: no limit
static std::map<char *, std::pair<size_t, int>> g_memory;
static hipError_t g_last = hipSuccess;

static FakeStream *stream_of(hipStream_t s) { return s ? reinterpret_cast<FakeStream *>(s) : &g_null[g_device]; }
static hipStream_t handle_of(FakeStream &s) { return reinterpret_cast<hipStream_t>(&s); }
static hipError_t give(hipError_t e) { if (e != hipSuccess) g_last = e; return e; }
static std::set<FakeStream *> g_streams;
static void finish_device(int device)
{
    g_null[device].done = g_null[device].queued;
    for (FakeStream *s : g_streams)
        if (s->device == device) s->done = s->queued;
}
static std::map<char *, std::pair<size_t, int>>::iterator find_memory(const void *p)
{
    char *q = static_cast<char *>(const_cast<void *>(p));
    auto it = g_memory.upper_bound(q);
    if (it == g_memory.begin()) return g_memory.end();
    --it;
    return q < it->first + it->second.first ? it : g_memory.end();
}

extern "C" {
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = g_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { g_device = d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetLastError() { const hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = (size_t)288 << 30; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    if (g_mallocs_left == 0) return give(hipErrorOutOfMemory);
    if (g_mallocs_left > 0) g_mallocs_left--;
    *p = calloc(1, n);
    g_memory[static_cast<char *>(*p)] = {n, g_device};
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    if (g_refuse_host_waits) return give(hipErrorStreamCaptureUnsupported);
    g_frees++;
    auto it = g_memory.find(static_cast<char *>(p));
    finish_device(it->second.second);
    g_memory.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = calloc(1, n); g_pinned++; return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); g_pinned--; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    memset(a, 0, sizeof *a);
    a->type = find_memory(p) == g_memory.end() ? hipMemoryTypeUnregistered : hipMemoryTypeDevice;
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *n, hipDeviceptr_t p)
{
    const auto it = find_memory(p);
    if (it == g_memory.end()) return give(hipErrorNotFound);
    *base = it->first;
    *n = it->second.first;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **, const void *) { return give(hipErrorInvalidSymbol); }

hipError_t hipDeviceSynchronize()
{
    if (g_refuse_host_waits) return give(hipErrorStreamCaptureUnsupported);
    g_host_waits++;
    finish_device(g_device);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    if (g_refuse_host_waits) return give(hipErrorStreamCaptureUnsupported);
    g_host_waits++;
    stream_of(s)->done = stream_of(s)->queued;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) { *c = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    if (g_refuse_events) return give(hipErrorStreamCaptureUnsupported);
    FakeEvent *ev = reinterpret_cast<FakeEvent *>(e);
    if (ev->s) {
        long &to = stream_of(s)->behind[ev->s];
        to = std::max(to, ev->tick);
    }
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    if (g_refuse_events) return give(hipErrorOutOfMemory);
    *e = reinterpret_cast<hipEvent_t>(new FakeEvent);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<FakeEvent *>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (g_refuse_events) return give(hipErrorStreamCaptureUnsupported);
    FakeEvent *ev = reinterpret_cast<FakeEvent *>(e);
    ev->s = stream_of(s);
    ev->tick = ev->s->queued;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (g_refuse_host_waits) return give(hipErrorStreamCaptureUnsupported);
    g_host_waits++;
    FakeEvent *ev = reinterpret_cast<FakeEvent *>(e);
    if (ev->s) ev->s->done = std::max(ev->s->done, ev->tick);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e)
{
    FakeEvent *ev = reinterpret_cast<FakeEvent *>(e);
    return !ev->s || ev->s->done >= ev->tick ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) { *t = 1.0f; return hipSuccess; }
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind)
{
    memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t s)
{
    memcpy(to, from, n);
    stream_of(s)->queued++;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s)
{
    stream_of(s)->queued++;
    return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s, hipEvent_t, hipEvent_t stop, int)
{
    stream_of(s)->queued++;
    if (stop) (void)hipEventRecord(stop, s);
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 2; return hipSuccess; }

struct Launch { dim3 grid, block; size_t shared; hipStream_t s; };
static Launch g_launch;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t n, hipStream_t s) { g_launch = {g, b, n, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s)
{
    *g = g_launch.grid; *b = g_launch.block; *n = g_launch.shared; *s = g_launch.s;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *none; return &none; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}

// ---------------------------------------------------------------------------------------------
// scenarios
// ---------------------------------------------------------------------------------------------
using namespace accel;

#define CHECK(what)                                                                        \
    do {                                                                                   \
        if (!(what)) {                                                                     \
            std::printf("line %d: %s does not hold\n", __LINE__, #what);                   \
            std::exit(1);                                                                  \
        }                                                                                  \
    } while (0)

constexpr size_t kBlock = 1 << 20;

// A handle with one block of the list among its products, used on `s` by a kernel that still runs.
struct Used {
    accel_handle *h = nullptr;
    void *block = nullptr;
    FakeStream *s;
    long tick = 0;
    explicit Used(FakeStream &on) : s(&on)
    {
        const int32_t indptr[2] = {0, 1}, idx[1] = {0};
        const float val[1] = {1};
        CHECK(accel_create(indptr, idx, val, 1, 1, 1, ACCEL_PTR_HOST, &h) == ACCEL_OK);
        block = take_memory(kBlock, false);
        CHECK(block);
        h->slab = block;
        h->ready = true;
        hipEvent_t done;
        CHECK(order_run(h, handle_of(on), true, false, &done) == ACCEL_OK);
        on.queued++;
        tick = on.queued;
    }
    // p, used next by `next` (null: by the host), is another block or comes behind the kernel
    bool safe(const void *p, FakeStream *next) const
    {
        return p != block || s->done >= tick || (next && (next == s || (next->behind.count(s) && next->behind[s] >= tick)));
    }
};

static FakeStream g_side[3];

// A handle of GPU 0 closed while GPU 1 is current.
static void closed_with_another_gpu_current()
{
    Used u(g_side[0]);
    CHECK(hipSetDevice(1) == hipSuccess);
    CHECK(accel_destroy(u.h) == ACCEL_OK);
    CHECK(g_device == 1);
    CHECK(hipSetDevice(0) == hipSuccess);
    void *p = take_memory(kBlock, false);
    CHECK(u.safe(p, &g_null[0]));
    CHECK(p == u.block);                                   // waited for, so it can be handed out again
}

// A handle's buffers lie on its GPU, whichever is current.
static void reserved_with_another_gpu_current()
{
    Used u(g_side[0]);
    void *old = u.h->partial = static_cast<float *>(take_memory(kBlock, false));
    u.h->partial_floats = kBlock / 4;
    u.h->n_long_units = (int64_t)kBlock / 64;
    CHECK(hipSetDevice(1) == hipSuccess);
    CHECK(accel_run(u.h, u.h->partial, u.h->partial, 1, nullptr) == ACCEL_ERR_STATE);
    CHECK(accel_reserve(u.h, 128) == ACCEL_OK);
    CHECK(g_device == 1 && u.h->partial != old && find_memory(u.h->partial)->second.second == 0);
    CHECK(g_side[0].done == g_side[0].queued);             // the old buffer's users
}

// The wait in accel_destroy is refused (another stream of the process captures).
static void wait_refused_on_close()
{
    Used u(g_side[0]);
    g_refuse_host_waits = true;
    CHECK(accel_destroy(u.h) == ACCEL_OK);
    void *p = take_memory(kBlock, true);
    CHECK(p && u.safe(p, nullptr));                        // still refused: other memory
    g_refuse_host_waits = false;
    void *q = take_memory(kBlock, true);
    CHECK(q && u.safe(q, nullptr));
    CHECK(q == u.block);                                   // not lost
}

// Expired memory whose hipFree is refused is neither lost nor handed out unordered.
static void free_refused()
{
    Used u(g_side[0]);
    g_refuse_host_waits = true;
    CHECK(accel_destroy(u.h) == ACCEL_OK);
    CHECK(accel_release_memory() == ACCEL_OK);
    CHECK(g_frees == 0);
    g_refuse_host_waits = false;
    CHECK(accel_release_memory() == ACCEL_OK);
    CHECK(g_frees > 0 && find_memory(u.block) == g_memory.end());
}

// The waits of the next user are refused: for a block behind an event, and for one of the null stream.
static void wait_refused_on_take()
{
    void *p = take_stream_memory(kBlock, handle_of(g_side[0]));
    g_side[0].queued++;
    give_stream_memory(p, handle_of(g_side[0]));
    g_refuse_host_waits = true;
    CHECK(take_memory(kBlock, true) != p);
    g_refuse_events = true;
    CHECK(take_stream_memory(kBlock, handle_of(g_side[1])) != p);
    g_refuse_host_waits = g_refuse_events = false;
    CHECK(take_memory(kBlock, true) == p && g_side[0].done == g_side[0].queued);

    void *q;
    {
        DevBuf b;                                          // given back behind work on the null stream
        CHECK(b.alloc(4 * kBlock) == ACCEL_OK);
        q = b.p;
        g_null[0].queued++;
    }
    g_refuse_host_waits = true;
    CHECK(take_memory(4 * kBlock, true) != q);
    g_refuse_host_waits = false;
    CHECK(take_memory(4 * kBlock, true) == q && g_null[0].done == g_null[0].queued);
}

// Neither an event nor a wait can be had when memory is given back behind a stream.
static void nothing_to_be_had_on_give()
{
    void *p = take_stream_memory(kBlock, handle_of(g_side[0]));
    g_side[0].queued++;
    g_refuse_host_waits = g_refuse_events = true;
    give_stream_memory(p, handle_of(g_side[0]));
    CHECK(take_memory(kBlock, false) != p);
    g_refuse_host_waits = g_refuse_events = false;
    CHECK(take_memory(kBlock, false) == p && g_side[0].done == g_side[0].queued);
}

// accel_create that runs out of memory gives back what it took as it took it: behind the null stream.
static void create_runs_out_of_memory()
{
    void *q;
    {
        DevBuf b;
        CHECK(b.alloc(kBlock) == ACCEL_OK);
        q = b.p;
        g_null[0].queued++;
    }
    std::vector<int32_t> indptr(kBlock / 4, 0), idx(kBlock);
    std::vector<float> val(kBlock);
    indptr.back() = (int32_t)kBlock;
    g_mallocs_left = 0;
    accel_handle *h = nullptr;
    CHECK(accel_create(indptr.data(), idx.data(), val.data(), (int64_t)indptr.size() - 1, 1, (int64_t)kBlock,
                       ACCEL_PTR_HOST, &h) == ACCEL_ERR_ALLOC);
    g_mallocs_left = -1;
    void *p = take_memory(kBlock, true);
    CHECK(p != q || g_null[0].done == g_null[0].queued);
}

// A buffer that grows while the wait for its last users is refused.
static void wait_refused_on_growth()
{
    Used u(g_side[0]);
    void *old = u.h->partial = static_cast<float *>(take_memory(2 * kBlock, false));
    u.h->partial_floats = 2 * kBlock / 4;
    u.h->n_long_units = (int64_t)kBlock / 64;
    g_refuse_host_waits = true;
    (void)accel_reserve(u.h, 128);
    CHECK(take_memory(2 * kBlock, true) != old);
    g_refuse_host_waits = false;
    CHECK(take_memory(2 * kBlock, true) == old);
}

// The position map of a value update: its temporaries are in use until its wait has succeeded.
static void wait_refused_in_a_value_update()
{
    Used u(g_side[0]);
    u.h->nnz = u.h->nnz_short = (int64_t)kBlock;
    u.h->owns_sorted = true;
    void *val = nullptr;
    CHECK(hipMalloc(&val, 4 * kBlock) == hipSuccess);
    g_refuse_host_waits = true;
    CHECK(accel_update_values_async(u.h, static_cast<float *>(val), handle_of(g_side[0])) != ACCEL_OK);
    std::set<void *> before;
    for (auto &m : g_memory) before.insert(m.first);
    void *p = take_memory(4 * kBlock, false);              // the map's size
    CHECK(p && !before.count(p));
}

// Values are restored from a sorted copy that an update may still be writing: not without the wait for it.
static void wait_refused_before_values_are_restored()
{
    Used u(g_side[0]);
    u.h->owns_sorted = u.h->val_stale = true;
    u.h->src_pos = static_cast<int32_t *>(u.block);
    u.h->s_val = static_cast<float *>(u.block);
    const long queued = g_null[0].queued;
    g_refuse_host_waits = true;
    CHECK(accel_preprocess(u.h) == ACCEL_ERR_HIP);
    CHECK(g_null[0].queued == queued && u.h->val_stale);
}

// The dense product waits on the device only, and frees nothing, whichever stream used its workspace last
// and however long that is ago.
static void dense_product_never_waits()
{
    const int64_t rows = 300000;
    const int K = 300, N = 128;
    void *X, *W, *Z;
    CHECK(hipMalloc(&X, sizeof(float) * (size_t)rows * K) == hipSuccess);
    CHECK(hipMalloc(&W, sizeof(float) * (size_t)K * N) == hipSuccess);
    CHECK(hipMalloc(&Z, sizeof(float) * (size_t)rows * N) == hipSuccess);
    auto product = [&](hipStream_t s) {
        return accel_dense_xw(static_cast<float *>(X), static_cast<float *>(W), static_cast<float *>(Z), rows, K, N, 0, 0, s);
    };
    { DevBuf b; CHECK(b.alloc(kBlock) == ACCEL_OK); }      // idle memory of another size, about to expire
    CHECK(product(nullptr) == ACCEL_OK);
    const long tick = g_null[0].queued;
    std::this_thread::sleep_for(std::chrono::milliseconds(1200));
    const size_t blocks = g_memory.size();
    CHECK(product(handle_of(g_side[0])) == ACCEL_OK);
    CHECK(g_memory.size() == blocks);                      // the same workspace ...
    CHECK(g_side[0].behind[&g_null[0]] >= tick);           // ... behind the product on the null stream
    CHECK(product(handle_of(g_side[1])) == ACCEL_OK);
    CHECK(g_side[1].behind[&g_side[0]] >= g_side[0].queued);
    CHECK(product(nullptr) == ACCEL_OK);
    CHECK(g_null[0].behind[&g_side[1]] >= g_side[1].queued);
    CHECK(g_memory.size() == blocks && g_host_waits == 0 && g_frees == 0);
}

// A pinned transfer buffer whose copies could not be waited for is not used before they have been, and not lost.
static void wait_refused_in_a_transfer()
{
    std::vector<char> host(kStagePiece + 100);
    void *dev;
    CHECK(hipMalloc(&dev, host.size()) == hipSuccess);
    CHECK(upload(dev, host.data(), host.size(), nullptr) == ACCEL_OK);
    Stage *first = take_stage(host.size());                // waits for the copies out of it
    void *const pinned = first->p;
    CHECK(g_null[0].done == g_null[0].queued);
    give_stage(first);
    CHECK(upload(dev, host.data(), host.size(), nullptr) == ACCEL_OK);
    g_refuse_host_waits = true;
    Stage *other = take_stage(host.size());
    CHECK(other && other->p != pinned);
    give_stage(other);
    CHECK(download(host.data(), dev, host.size(), nullptr) != ACCEL_OK);
    Stage *third = take_stage(host.size());
    CHECK(third && third->p != pinned && third->p != other->p);
    give_stage(third);
    CHECK(g_pinned == 3);
    g_refuse_host_waits = false;
    CHECK(accel_release_memory() == ACCEL_OK);
    CHECK(g_pinned == 0 && g_null[0].done == g_null[0].queued);
}

// Preprocessing that runs out of memory half way: kernels still queued write into the pinned block that
// its results come through.
static void preprocessing_runs_out_of_memory()
{
    const int rows = 1000;
    std::vector<int32_t> indptr(rows + 1), idx(rows, 0);
    std::vector<float> val(rows, 1.0f);
    for (int i = 0; i <= rows; i++) indptr[i] = i;
    int failed = 0;
    for (int n = 0; n < 40; n++) {
        accel_handle *h = nullptr;
        CHECK(accel_create(indptr.data(), idx.data(), val.data(), rows, 1, rows, ACCEL_PTR_HOST, &h) == ACCEL_OK);
        CHECK(accel_release_memory() == ACCEL_OK);
        g_mallocs_left = n;
        const int rc = accel_preprocess(h);
        g_mallocs_left = -1;
        failed += rc == ACCEL_ERR_ALLOC;
        Mail *m = take_mail();
        CHECK(g_null[0].done == g_null[0].queued);
        give_mail(m);
        CHECK(accel_destroy(h) == ACCEL_OK);
        if (rc == ACCEL_OK) { CHECK(failed >= 4); return; }
    }
    CHECK(false);
}

int main(int argc, char **argv)
{
    g_null[1].device = 1;
    for (FakeStream &s : g_side) g_streams.insert(&s);
    const std::map<std::string, void (*)()> all = {
#define SCENARIO(name) {#name, name}
        SCENARIO(closed_with_another_gpu_current),
        SCENARIO(reserved_with_another_gpu_current),
        SCENARIO(wait_refused_on_close),
        SCENARIO(free_refused),
        SCENARIO(wait_refused_on_take),
        SCENARIO(nothing_to_be_had_on_give),
        SCENARIO(create_runs_out_of_memory),
        SCENARIO(wait_refused_on_growth),
        SCENARIO(wait_refused_in_a_value_update),
        SCENARIO(wait_refused_before_values_are_restored),
        SCENARIO(dense_product_never_waits),
        SCENARIO(wait_refused_in_a_transfer),
        SCENARIO(preprocessing_runs_out_of_memory),
    };
    if (argc != 2 || !all.count(argv[1])) {
        for (auto &s : all) std::printf("%s\n", s.first.c_str());
        return argc == 1 ? 0 : 2;
    }
    all.at(argv[1])();
    std::printf("ok\n");
    return 0;
}
