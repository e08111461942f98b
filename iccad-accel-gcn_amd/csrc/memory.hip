// Device memory of the handles, kept for the next one.
//
// A program that builds an operator per graph (sampled subgraphs, mini-batches) allocates and
// frees the same few sizes over and over, and on this GPU that is not free: hipFree of an
// allocation of 128 MB or more takes 0.24 ms and waits for the device, and the driver clears
// what was freed before it hands it out again.  Measured on create + preprocess + run + destroy
// of a 125 M-non-zero matrix (1.4 GB in nine allocations): 10 to 42 ms a cycle with hipMalloc
// and hipFree, of which the kernels are 5.3; 2.4 M non-zeros: 0.61 ms, of which 0.50.
//
// So freed memory goes to a list per process and is handed out again.  The list is bounded and
// is given back:
//   - it holds at most 1/64 of the device's memory (4.5 GB here); beyond that the memory that
//     has been idle longest is freed;
//   - what nobody has asked for within kIdleSeconds is freed by the next call that takes or
//     gives memory (not by take_stream_memory and give_stream_memory, whose callers are not to
//     wait for the device: they free only what is beyond the bound);
//   - when an allocation fails, everything idle is freed and the allocation is tried again;
//   - accel_release_memory() frees everything idle.
// Sizes are rounded up to an eighth of a power of two and a block serves requests of down to
// four fifths of it, so that subgraphs of about the same size find each other's memory.
//
// Order on the device.  hipFree waits for the device; giving memory back here does not.  A
// block may therefore still be in use by kernels queued on the null stream, or on one other
// stream, behind which it carries an event (a handle that has used several streams waits for the
// device before it gives its memory back).  The preprocessing, which takes nearly all of it,
// works on the null stream and is ordered behind the former by the stream; every other
// combination of the last use and the next waits on the device, for the event or for what the null
// stream holds now, or on the host where the next stream is not known (`any_stream`).
//
// A wait may be refused (most are while any stream of the process captures).  A block whose last
// use could not be waited for is marked so, stays on the list, and is handed out or freed only
// once a wait for its whole device has succeeded; until then requests get other memory.
#include <chrono>
#include <mutex>
#include <new>
#include <unordered_map>
#include <vector>

#include "preprocess.h"

namespace accel {

InUse wait_for_device()
{
    if (hipDeviceSynchronize() == hipSuccess) return InUse::no;
    (void)hipGetLastError();
    return InUse::unknown;
}

namespace {

using Clock = std::chrono::steady_clock;
constexpr double kIdleSeconds = 1.0;
constexpr size_t kIdleShare = 64;                 // idle memory: at most 1/64 of the device's

struct Idle {
    void *p;
    size_t bytes;
    int device;
    InUse use;                                    // what may still use it, apart from
    hipEvent_t after;                             // ... what this event stands behind (or null)
    Clock::time_point since;
};

struct Pool {
    std::mutex mu;
    std::vector<Idle> idle;                       // oldest first
    std::unordered_map<void *, std::pair<size_t, int>> live;      // bytes, device
    std::unordered_map<int, size_t> most_idle;    // bound per device
};

Pool &pool()
{
    static Pool *p = new Pool;                    // never destroyed: the runtime may be gone by then
    return *p;
}

size_t size_class(size_t bytes)
{
    if (bytes <= 4096) return 4096;
    size_t step = 512;                            // an eighth of the largest power of two <= bytes
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

// A block goes (back) on the list: one that could not be waited for, or could not be freed.
void keep_in_doubt(Idle b)
{
    b.use = InUse::unknown;
    b.since = Clock::now();
    Pool &pl = pool();
    std::lock_guard<std::mutex> lock(pl.mu);
    pl.idle.push_back(b);
}

void free_idle(std::vector<Idle> &gone)
{
    for (const Idle &b : gone) {
        OnDevice on(b.device);
        if (hipFree(b.p) != hipSuccess) {                             // waits for the device
            (void)hipGetLastError();
            keep_in_doubt(b);
        } else if (b.after) {
            (void)hipEventDestroy(b.after);
        }
    }
    gone.clear();
}

// What is queued on s from now on comes behind what the null stream holds now.
hipError_t wait_for_null_stream(hipStream_t s)
{
    hipEvent_t now = nullptr;
    hipError_t e = hipEventCreateWithFlags(&now, hipEventDisableTiming);
    if (e != hipSuccess) return e;
    e = hipEventRecord(now, nullptr);
    if (e == hipSuccess) e = hipStreamWaitEvent(s, now, 0);
    (void)hipEventDestroy(now);
    return e;
}

// Whether the next use of b, on s (with `any`: on a stream not known yet), comes behind its last one.
bool order_behind(const Idle &b, hipStream_t s, bool any)
{
    hipError_t e = hipSuccess;
    if (b.use == InUse::unknown) e = hipDeviceSynchronize();
    else if (b.after) e = any ? hipEventSynchronize(b.after) : hipStreamWaitEvent(s, b.after, 0);
    else if (b.use == InUse::null_stream && (any || s)) e = any ? hipStreamSynchronize(nullptr) : wait_for_null_stream(s);
    if (e == hipSuccess) return true;
    (void)hipGetLastError();
    return wait_for_device() == InUse::no;
}

// Takes the oldest blocks beyond the bound and (by_age) those idle for longer than kIdleSeconds off
// the list (the caller frees them, without the lock).
void expire(Pool &pl, std::vector<Idle> &gone, bool by_age)
{
    if (pl.idle.empty()) return;
    const Clock::time_point now = Clock::now();
    // nearly always nothing is old (the first is the oldest) and all of it together is below every bound (a new graph comes by
    // here some fifteen times: 0.6 us of it)
    if (!by_age || std::chrono::duration<double>(now - pl.idle.front().since).count() <= kIdleSeconds) {
        size_t all = 0, least = SIZE_MAX;
        for (const Idle &b : pl.idle) all += b.bytes;
        for (const auto &m : pl.most_idle) least = std::min(least, m.second);
        if (all <= least) return;
    }
    std::unordered_map<int, size_t> held;
    for (const Idle &b : pl.idle) held[b.device] += b.bytes;
    size_t keep = 0;
    for (size_t i = 0; i < pl.idle.size(); i++) {
        const Idle &b = pl.idle[i];
        const bool old = by_age && std::chrono::duration<double>(now - b.since).count() > kIdleSeconds;
        if (old || held[b.device] > pl.most_idle[b.device]) {
            held[b.device] -= b.bytes;
            gone.push_back(b);
        } else {
            pl.idle[keep++] = b;
        }
    }
    pl.idle.resize(keep);
}

void release_idle_device_memory()
{
    Pool &pl = pool();
    std::vector<Idle> gone;
    {
        std::lock_guard<std::mutex> lock(pl.mu);
        gone.swap(pl.idle);
    }
    free_idle(gone);
}

}  // namespace

// s: the stream the memory will be used on first; null: the null stream, or (any) one not known yet.
static void *take(size_t bytes, hipStream_t s, bool any, bool by_age)
{
    Pool &pl = pool();
    const size_t want = size_class(bytes);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
    Idle got{};
    std::vector<Idle> gone;
    {
        std::lock_guard<std::mutex> lock(pl.mu);
        size_t best = pl.idle.size();
        for (size_t i = 0; i < pl.idle.size(); i++) {             // the smallest that fits, of those the latest
            const Idle &b = pl.idle[i];
            if (b.device != dev || b.bytes < want || b.bytes > want + want / 4) continue;
            if (best == pl.idle.size() || b.bytes <= pl.idle[best].bytes) best = i;
        }
        if (best < pl.idle.size()) {
            got = pl.idle[best];
            pl.idle.erase(pl.idle.begin() + (long)best);
        }
        expire(pl, gone, by_age);
    }
    free_idle(gone);
    if (got.p && order_behind(got, s, any)) {
        if (got.after) (void)hipEventDestroy(got.after);
        std::lock_guard<std::mutex> lock(pl.mu);
        pl.live[got.p] = {got.bytes, dev};
        return got.p;
    }
    if (got.p) keep_in_doubt(got);
    void *p = nullptr;
    if (hipMalloc(&p, want) != hipSuccess) {
        (void)hipGetLastError();
        release_idle_device_memory();
        if (hipMalloc(&p, want) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
    }
    std::lock_guard<std::mutex> lock(pl.mu);
    pl.live[p] = {want, dev};
    if (!pl.most_idle.count(dev)) {
        size_t free_bytes = 0, total = 0;
        if (hipMemGetInfo(&free_bytes, &total) != hipSuccess) { (void)hipGetLastError(); total = 0; }
        pl.most_idle[dev] = total / kIdleShare;
    }
    return p;
}

static void give(void *p, InUse use, hipEvent_t after, bool by_age)
{
    if (!p) return;
    Pool &pl = pool();
    std::vector<Idle> gone;
    {
        std::lock_guard<std::mutex> lock(pl.mu);
        const auto it = pl.live.find(p);
        if (it == pl.live.end()) return;
        pl.idle.push_back({p, it->second.first, it->second.second, use, after, Clock::now()});
        pl.live.erase(it);
        expire(pl, gone, by_age);
    }
    free_idle(gone);
}

void *take_memory(size_t bytes, bool any_stream) { return take(bytes, nullptr, any_stream, true); }
void give_memory(void *p, InUse use) { give(p, use, nullptr, true); }
void *take_stream_memory(size_t bytes, hipStream_t s) { return take(bytes, s, false, false); }

void give_stream_memory(void *p, hipStream_t s)
{
    if (!s) { give(p, InUse::null_stream, nullptr, false); return; }
    hipEvent_t after = nullptr;
    if (hipEventCreateWithFlags(&after, hipEventDisableTiming) == hipSuccess && hipEventRecord(after, s) == hipSuccess) {
        give(p, InUse::no, after, false);
        return;
    }
    (void)hipGetLastError();
    if (after) (void)hipEventDestroy(after);
    const bool done = hipStreamSynchronize(s) == hipSuccess;
    if (!done) (void)hipGetLastError();
    give(p, done ? InUse::no : InUse::unknown, nullptr, false);
}

// Pinned blocks for the preprocessing's results, one per call that is under way; kept (a few KB
// each, as many as calls have run at once).
static std::mutex g_host_mu;
static std::vector<Mail *> g_mail;
// Pinned buffers for transfers: at most kIdleStages are kept (16 MiB each at most).
constexpr size_t kIdleStages = 2;
static std::vector<Stage *> g_stage;

Mail *take_mail()
{
    Mail *m = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_host_mu);
        if (!g_mail.empty()) {
            m = g_mail.back();
            g_mail.pop_back();
        }
    }
    if (!m && hipHostMalloc(reinterpret_cast<void **>(&m), sizeof(Mail), hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        set_error("allocation of pinned host memory failed");
        return nullptr;
    }
    m->bad_index = m->bad_order = 0;
    return m;
}

void give_mail(Mail *m)
{
    if (!m) return;
    std::lock_guard<std::mutex> lock(g_host_mu);
    g_mail.push_back(m);
}

// Whether nothing copies out of the buffer or into it any more.
static bool settle_stage(Stage *s)
{
    if (s->in_doubt) {
        OnDevice on(s->device);
        if (wait_for_device() != InUse::no) return false;
    } else if (s->busy && hipEventSynchronize(s->last) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    s->in_doubt = s->busy = false;
    return true;
}

// One whose copies cannot be waited for goes back on the list.
static void free_stage(Stage *s)
{
    if (!settle_stage(s)) {
        std::lock_guard<std::mutex> lock(g_host_mu);
        g_stage.insert(g_stage.begin(), s);
        return;
    }
    for (hipEvent_t e : s->event)
        if (e) (void)hipEventDestroy(e);
    if (s->last) (void)hipEventDestroy(s->last);
    if (s->p) (void)hipHostFree(s->p);
    (void)hipGetLastError();
    delete s;
}

Stage *take_stage(size_t bytes)
{
    const size_t want = std::min(std::max(bytes, (size_t)1 << 20), kStageBytes);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
    Stage *s = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_host_mu);
        for (size_t i = g_stage.size(); i-- > 0 && !s;)
            if (g_stage[i]->bytes >= want && g_stage[i]->device == dev) {
                s = g_stage[i];
                g_stage.erase(g_stage.begin() + (long)i);
            }
    }
    if (s && settle_stage(s)) return s;
    if (s) give_stage(s);         // the wait was refused: another one
    s = new (std::nothrow) Stage;
    if (!s) { set_error("host allocation failed"); return nullptr; }
    s->bytes = want;
    s->device = dev;
    bool ok = hipHostMalloc(&s->p, want, hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t &e : s->event)
        if (ok) ok = hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (ok) ok = hipEventCreateWithFlags(&s->last, hipEventDisableTiming) == hipSuccess;
    if (ok) return s;
    (void)hipGetLastError();
    free_stage(s);
    set_error("allocation of %zu bytes of pinned host memory failed", want);
    return nullptr;
}

void give_stage(Stage *s)
{
    if (!s) return;
    std::vector<Stage *> gone;
    {
        std::lock_guard<std::mutex> lock(g_host_mu);
        g_stage.push_back(s);
        while (g_stage.size() > kIdleStages) {
            gone.push_back(g_stage.front());
            g_stage.erase(g_stage.begin());
        }
    }
    for (Stage *g : gone) free_stage(g);
}

void release_idle_memory()
{
    release_idle_device_memory();
    std::vector<Stage *> stages;
    {
        std::lock_guard<std::mutex> lock(g_host_mu);
        stages.swap(g_stage);
    }
    for (Stage *s : stages) free_stage(s);
}

}  // namespace accel
