// Shared by the two halves of the preprocessing: preprocess.hip (sort, sorted CSR, partition)
// and plan.hip (the launch plan).
#pragma once
#include <algorithm>

#include "internal.h"

namespace accel {

constexpr int kThreads = 256;
constexpr int kWaves4 = kThreads / 64;

// Rows are sorted by degree through bins: bin d holds the rows of degree d = 0..384, the last
// bin all longer rows.
constexpr int kBins = kDegBound + 2;
constexpr int kLongBin = kDegBound + 1;

// Split rows of more than kWideRow non-zeros are regrouped in pieces of kWideChunk by a
// workgroup per piece, shorter ones by a wavefront each.
constexpr int kWideRow = 1024;
constexpr int kWideChunk = 4096;

constexpr int kRunParts = 1024;

// A small block of pinned host memory that kernels write their results for the host into: the
// host reads it after a synchronisation, with no copy queued in between.
struct Mail {
    int hist[kBins];          // rows per bin
    // statistics of the rows (kStat* below)
    int stat[16];
    // from the later kernels
    int bad_index;            // a column outside [0, cols)
    int bad_order;            // a saved row order is not the degree order
    int per_queue;            // units per queue of the launch plan, padding included
    int n_pieces;             // pieces of split rows
    int n_units;              // units of whole rows
    int n_blocks;             // entries of the partition (only for rows in any order)
    // the partition of rows in order: hist holds the first row of each bin then, or -1
    int part[kRunParts];      // entries of rows longer than 384, summed up per workgroup of run_bounds_kernel
};
enum {
    kStatBadIndptr, kStatUnsorted, kStatMaxDegree,        // these three: the largest value over all rows
    kStatLongBlocks, kStatWideRows, kStatWideChunks,      // the others: sums
    kStatRows16, kStatRows32, kStatRows64,                // rows stored in 16, 32, 64 column groups by row_groups' own rule
    kStatBig, kStatBigAlt,                                // rows with more than 32 times a split threshold
    kStatSampled, kStatLocal,                             // of the locality sample
    kStatLoneChunks,                                      // wide rows of one chunk
    kStatCount
};
Mail *take_mail();            // memory.hip; null when there is none
void give_mail(Mail *m);
struct MailHolder {
    Mail *m;
    bool written = false;         // every kernel that writes it has been waited for
    MailHolder() : m(take_mail()) {}
    // (on an error kernels that write it may be queued on the null stream; left alone where they cannot
    // be waited for)
    ~MailHolder()
    {
        if (written || hipStreamSynchronize(nullptr) == hipSuccess) give_mail(m);
        else (void)hipGetLastError();
    }
    MailHolder(const MailHolder &) = delete;
    MailHolder &operator=(const MailHolder &) = delete;
};

// Pinned memory that transfers go through (transfer.hip), with events for its pieces.
constexpr size_t kStageBytes = (size_t)16 << 20, kStagePiece = (size_t)2 << 20;
struct Stage {
    void *p = nullptr;
    size_t bytes = 0;
    hipEvent_t event[kStageBytes / kStagePiece] = {}, last = nullptr;
    int device = 0;
    bool busy = false;            // `last` stands behind the last copy out of it
    bool in_doubt = false;        // copies nobody has waited for, with no event behind them
};
Stage *take_stage(size_t bytes);      // memory.hip: min(bytes, kStageBytes) or more; null when there is none
void give_stage(Stage *s);
struct StageHolder {
    Stage *s;
    explicit StageHolder(size_t bytes) : s(take_stage(bytes)) {}
    ~StageHolder() { give_stage(s); }
    StageHolder(const StageHolder &) = delete;
    StageHolder &operator=(const StageHolder &) = delete;
};

// Temporaries of one preprocessing call come out of a few large pieces of device memory (there
// are some twenty of them).  The pieces are given back when the arena goes out of scope; what
// is still queued then is queued on the null stream, unless `use` says otherwise.
struct Arena {
    static constexpr int kMaxChunks = 32;
    char *chunk[kMaxChunks] = {};
    size_t cap = 0, used = 0;      // of the newest chunk
    int n_chunks = 0;
    size_t next_chunk = 0;         // size hint for the next chunk
    bool any_stream = false;       // will be used on another stream than the null stream
    InUse use = InUse::null_stream;
    Arena() = default;
    Arena(const Arena &) = delete;
    Arena &operator=(const Arena &) = delete;
    ~Arena()
    {
        for (int i = 0; i < n_chunks; i++) give_memory(chunk[i], use);
    }
    void *take(size_t bytes)
    {
        bytes = (std::max<size_t>(bytes, 4) + 255) & ~(size_t)255;
        if (n_chunks == 0 || used + bytes > cap) {
            if (n_chunks == kMaxChunks) return nullptr;
            const size_t want = std::max(bytes, next_chunk);
            void *p = take_memory(want, any_stream);
            if (!p) return nullptr;
            chunk[n_chunks++] = static_cast<char *>(p);
            cap = want;
            used = 0;
            next_chunk = std::max<size_t>(next_chunk / 4, (size_t)1 << 20);   // later chunks: leftovers only
        }
        void *p = chunk[n_chunks - 1] + used;
        used += bytes;
        return p;
    }
    template <class T> int alloc(T **out, size_t count)
    {
        *out = static_cast<T *>(take(sizeof(T) * count));
        if (*out) return ACCEL_OK;
        set_error("device allocation of %zu bytes failed", sizeof(T) * count);
        return ACCEL_ERR_ALLOC;
    }
};

struct DevBuf {  // device memory that is given back on scope exit unless it is released
    void *p = nullptr;
    InUse use = InUse::null_stream;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { give_memory(p, use); }
    int alloc(size_t bytes, bool any_stream = false)
    {
        p = take_memory(bytes, any_stream);
        if (p) return ACCEL_OK;
        set_error("device allocation of %zu bytes failed", bytes);
        return ACCEL_ERR_ALLOC;
    }
    template <class T> T *as() { return static_cast<T *>(p); }
    void *release() { void *q = p; p = nullptr; return q; }
};

inline unsigned grid_for(int64_t n) { return (unsigned)((n + kThreads - 1) / kThreads); }

// Scans over a wavefront with all lanes active, by moves between the lanes' registers: through ds_bpermute (__shfl) each
// of the six steps waits for the LDS, 0.4 us a scan on an idle chip, and the fourteen sums at the end of degree_kernel
// took 2.7 of its 8 us on 60 k non-zeros.  Lanes that a step has nothing for keep 0 (rows of 16 lanes first).
template <int kCtrl, int kRows> __device__ __forceinline__ int lanes_moved(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, kCtrl, kRows, 0xf, false);
}
template <class F> __device__ __forceinline__ int wave_scan(int v, F f)
{
    v = f(v, lanes_moved<0x111, 0xf>(v));                // from 1, 2, 4, 8 lanes below, within rows
    v = f(v, lanes_moved<0x112, 0xf>(v));
    v = f(v, lanes_moved<0x114, 0xf>(v));
    v = f(v, lanes_moved<0x118, 0xf>(v));
    v = f(v, lanes_moved<0x142, 0xa>(v));                // the last lane of rows 0 and 2 to rows 1 and 3
    return f(v, lanes_moved<0x143, 0xc>(v));             // lane 31 to rows 2 and 3
}
__device__ __forceinline__ int wave_inclusive_sum(int v)
{
    return wave_scan(v, [](int a, int b) { return a + b; });
}
__device__ __forceinline__ int wave_exclusive_sum(int v) { return wave_inclusive_sum(v) - v; }
__device__ __forceinline__ int wave_sum(int v) { return __builtin_amdgcn_readlane(wave_inclusive_sum(v), 63); }
// (of values that are not negative)
__device__ __forceinline__ int wave_max(int v)
{
    return __builtin_amdgcn_readlane(wave_scan(v, [](int a, int b) { return a > b ? a : b; }), 63);
}

// Exclusive scan of one value per thread over a workgroup of T threads; `lds` holds T / 64 ints.
template <int T>
__device__ __forceinline__ int block_exclusive_sum(int v, int *lds, int &total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int inc = wave_inclusive_sum(v);
    if (lane == 63) lds[w] = inc;
    __syncthreads();
    int prefix = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < T / 64; i++) {
        const int t = lds[i];
        if (i < w) prefix += t;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return prefix + inc - v;
}

// Lanes of this wavefront that are `valid` and hold the same value in the low kBits bits of v: four instructions a bit.
template <int kBits>
__device__ __forceinline__ unsigned long long wave_match(int v, bool valid)
{
    const unsigned long long all = __ballot(valid);
    uint32_t lo = (uint32_t)all, hi = (uint32_t)(all >> 32);
#pragma unroll
    for (int b = 0; b < kBits; b++) {
        const int bit = (v << (31 - b)) >> 31;
        const unsigned long long bal = __ballot(bit != 0);
        lo &= ~((uint32_t)bal ^ (uint32_t)bit);
        hi &= ~((uint32_t)(bal >> 32) ^ (uint32_t)bit);
    }
    return (unsigned long long)hi << 32 | lo;
}
__device__ __forceinline__ int lanes_below(unsigned long long m, int lane)
{
    return __popcll(m & ((1ull << lane) - 1ull));
}

// ---------------------------------------------------------------------------
// What one pass over the caller's rows computes about the units of whole rows (plan.hip's
// subject, formed here because the pass that sorts the rows has everything at hand).
// ---------------------------------------------------------------------------
// Rows a unit of whole rows may hold: as many as fit unit_nz non-zeros, at least one.
__device__ __forceinline__ int rows_per_unit(int d, int unit_nz) { return max(1, unit_nz / d); }

// What a unit costs, for levelling the queues: a gathered row of X per non-zero, a
// written row of Y per row, a fixed part; scaled down (shift >= 2) so that the sum over
// the matrix stays below 2^31.  (Counting units, or fixed parts of 64 or 200, measured the
// same within noise.)
__device__ __forceinline__ int unit_cost(int nz, int n_rows, int shift)
{
    return ((nz + n_rows + 8) >> shift) + 1;
}

struct UnitRule {
    int split;          // rows of more non-zeros are split, shorter ones form units of whole rows
    int unit_nz;        // most non-zeros of a unit of several whole rows
    int groups;         // column groups of split rows: 0 by row_groups' rule, else forced
    int cost_shift;
    int light_nz;       // a unit of up to this many non-zeros is a light one
};

// The unit that the row of degree d (1..split), `in_run` rows into the sorted run of its degree
// (`run_rows` rows long), starts: n rows, or 0 when it starts none.
__device__ __forceinline__ int unit_rows(int d, int in_run, int run_rows, const UnitRule &u)
{
    int w, rpb;
    slice_rule(d, w, rpb);
    const int rpu = rows_per_unit(d, u.unit_nz);
    const int off = in_run % rpb;
    if (off % rpu != 0) return 0;
    return min(min(rpu, rpb - off), run_rows - in_run);
}

// Per run of rows in the caller's order (one wavefront's share): units of whole rows that start
// there, their cost, how many of them are not light, and split rows stored in 8 column groups.
enum { kSumUnits, kSumCost, kSumHeavy, kSumRows8, kSums };

// Rows in a share and shares of a matrix: at most kMaxShares shares (enough wavefronts to fill
// the GPU; the bins of every share are scanned), of a multiple of 64 rows, 256 at least (a
// wavefront reads and writes a counter per bin whatever the length of its share).
constexpr int kMaxShares = 4096, kMinShare = 256;
struct Shares {
    int64_t rows = 0;
    int share = kMinShare, n = 0, pitch = 0;  // rows per share, shares, shares rounded up to a multiple of 4
    explicit Shares(int64_t r) : rows(r)
    {
        const int64_t want = (r + kMaxShares - 1) / kMaxShares;
        share = (int)std::max<int64_t>(kMinShare, (want + 63) / 64 * 64);
        n = (int)((r + share - 1) / share);
        pitch = (n + kWaves4 - 1) / kWaves4 * kWaves4;
    }
    unsigned groups() const { return (unsigned)(pitch / kWaves4); }
};

// Exclusive scan of the counts per share, in place, by a workgroup of T threads; the total goes
// behind the last share.
template <int T>
__device__ __forceinline__ void scan_shares(int *__restrict__ s, int n, int *lds /* T / 64 ints */)
{
    constexpr int kEach = kMaxShares / T;
    int v[kEach], acc = 0;
#pragma unroll
    for (int j = 0; j < kEach; j++) {
        const int i = (int)threadIdx.x * kEach + j;
        v[j] = i < n ? s[i] : 0;
        acc += v[j];
    }
    int total, run = block_exclusive_sum<T>(acc, lds, total);
#pragma unroll
    for (int j = 0; j < kEach; j++) {
        const int i = (int)threadIdx.x * kEach + j;
        if (i < n) s[i] = run;
        run += v[j];
    }
    if (threadIdx.x == 0) s[n] = total;
}

// ---------------------------------------------------------------------------
// Exclusive scans of up to three arrays in one launch: out[i] = add + in[0] + ... + in[i - 1],
// out[n] = the sum of all plus add (in place allowed).  A workgroup takes the next tile of its array
// by ticket, publishes the tile's sum, and adds up what the tiles before it have published: their
// sums, back to the first that already knows its prefix.  Tiles are taken in order, so every tile a
// workgroup waits for belongs to a workgroup that is running and publishes its sum before it waits
// for anything itself.  Words: value below, 1 = sum, 2 = prefix above (one 64-bit access: no
// fence).  Tickets and words are zero on entry.
// ---------------------------------------------------------------------------
constexpr int kScanItems = 8;
constexpr int kScanTile = kThreads * kScanItems;
inline int64_t scan_tiles(int64_t n) { return (n + kScanTile - 1) / kScanTile; }
struct ScanJob {
    const int *in;
    int *out;
    int64_t n;
    int add;
    int *zeroed;                              // scan_zeroed(n) ints, 8-byte aligned
};
inline int64_t scan_zeroed(int64_t n) { return 2 + 2 * scan_tiles(n); }
struct ScanJobs {
    ScanJob job[3];
    int first[3];                             // first workgroup of each job
};
static __global__ __launch_bounds__(kThreads) void scan_kernel(ScanJobs jobs)
{
    __shared__ int lds[kWaves4], my_tile, my_prefix;
    const int which = (int)blockIdx.x >= jobs.first[2] ? 2 : (int)blockIdx.x >= jobs.first[1] ? 1 : 0;
    const ScanJob jb = jobs.job[which];
    unsigned long long *word = reinterpret_cast<unsigned long long *>(jb.zeroed) + 1;
    if (threadIdx.x == 0)
        my_tile = __hip_atomic_fetch_add(jb.zeroed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int tile = my_tile;
    const int64_t base = (int64_t)tile * kScanTile + (int64_t)threadIdx.x * kScanItems;
    int v[kScanItems], acc = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; j++) {
        v[j] = base + j < jb.n ? jb.in[base + j] : 0;
        acc += v[j];
    }
    int total;
    const int exc = block_exclusive_sum<kThreads>(acc, lds, total);
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        if (lane == 0)
            __hip_atomic_store(&word[tile], ((tile ? 1ull : 2ull) << 32) | (unsigned)total, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        int prefix = 0;
        for (int look = tile - 1; look >= 0; look -= 64) {
            const int t = look - lane;
            unsigned long long s = 2ull << 32;                      // before the first tile: a prefix of 0
            if (t >= 0)
                while (((s = __hip_atomic_load(&word[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >> 32) == 0)
                    __builtin_amdgcn_s_sleep(1);
            const unsigned long long known = __ballot((s >> 32) == 2);
            const int stop = known ? __ffsll((unsigned long long)known) - 1 : 63;   // the nearest known prefix
            prefix += wave_sum(lane <= stop ? (int)(unsigned)s : 0);
            if (known) break;
        }
        if (lane == 0) {
            if (tile)
                __hip_atomic_store(&word[tile], (2ull << 32) | (unsigned)(prefix + total), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            my_prefix = prefix + jb.add;
            if ((int64_t)(tile + 1) * kScanTile >= jb.n) jb.out[jb.n] = prefix + total + jb.add;
        }
    }
    __syncthreads();
    int run = my_prefix + exc;
#pragma unroll
    for (int j = 0; j < kScanItems; j++) {
        if (base + j < jb.n) jb.out[base + j] = run;
        run += v[j];
    }
}
// The n_jobs jobs (1 to 3), each of at least one element.
inline void launch_scans(ScanJobs jobs, int n_jobs, hipStream_t s)
{
    int at = 0;
    for (int i = 0; i < 3; i++) {
        jobs.first[i] = i < n_jobs ? at : 0x7fffffff;
        if (i < n_jobs) at += (int)scan_tiles(jobs.job[i].n);
    }
    scan_kernel<<<dim3((unsigned)at), dim3(kThreads), 0, s>>>(jobs);
}

// The sorted rows as the kernels see them.
struct SortedRows {
    int64_t rows = 0;
    const int32_t *indptr = nullptr;          // the caller's
    int32_t *s_indptr = nullptr;              // sorted
    int32_t *perm = nullptr;                  // sorted row -> caller's row; null: in order already
    uint32_t *place = nullptr;                // caller's row -> sorted row
    const int *run_row = nullptr;             // [kBins + 1] first sorted row of each bin
    const int *run_nz = nullptr;              // [kBins] first non-zero of each bin
};

// The units of whole rows in the caller's order, and what the plan needs to know of them.
struct PlanUnits {
    int *sums = nullptr;                      // [kSums][pitch + kWaves4], scanned
    int4 *units = nullptr;
    int *running = nullptr;                   // [n + 1] cost of the units before each
    int *heavy_before = nullptr;              // [n + 1] units before each that are not light
    int *rank8 = nullptr;                     // split row of 8 column groups -> its rank among them in the caller's order
};

// A wavefront writes the units of whole rows that start in share c of the caller's rows, the running
// cost and the number of heavy units before each, and the rank of each split row of 8 column groups
// among those rows, all in the caller's order.
__device__ __forceinline__ void list_units(const SortedRows &sr, const UnitRule &rule, const PlanUnits &pu, int share,
                                           int n_shares, int pitch, int first_split, const int *run_row /* LDS */,
                                           const int *run_nz /* LDS */, int c)
{
    const int lane = threadIdx.x & 63;
    if (c == 0 && lane == 0) {
        const int n = pu.sums[kSumUnits * pitch + n_shares];
        pu.running[n] = pu.sums[kSumCost * pitch + n_shares];
        pu.heavy_before[n] = pu.sums[kSumHeavy * pitch + n_shares];
    }
    if (c >= n_shares) return;
    int n_units = pu.sums[kSumUnits * pitch + c], cost0 = pu.sums[kSumCost * pitch + c];
    int heavy0 = pu.sums[kSumHeavy * pitch + c], rows8 = pu.sums[kSumRows8 * pitch + c];
    const int64_t r_end = min(sr.rows, (int64_t)(c + 1) * share);
    for (int64_t r1 = (int64_t)c * share; r1 < r_end; r1 += 4 * 64) {
        int deg[4], plc[4];                              // four rounds' rows are on their way at once
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t r = r1 + j * 64 + lane;
            deg[j] = r < r_end ? sr.indptr[r + 1] - sr.indptr[r] : 0;
            plc[j] = r < r_end ? (int)sr.place[r] : 0;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int d = deg[j], p = plc[j];
            int n = 0, in_run = 0;
            if (d > 0 && d <= rule.split) {
                in_run = p - run_row[d];
                n = unit_rows(d, in_run, run_row[d + 1] - run_row[d], rule);
            }
            const int nz = d * n;
            const int cost = n > 0 ? unit_cost(nz, n, rule.cost_shift) : 0;
            const unsigned long long heads = __ballot(n > 0), heavies = __ballot(n > 0 && nz > rule.light_nz);
            const int inc = wave_inclusive_sum(cost);
            if (n > 0) {
                int w, rpb;
                slice_rule(d, w, rpb);
                const int at = n_units + lanes_below(heads, lane);
                pu.units[at] = make_int4(d, p, run_nz[d] + in_run * d, (w << 16) + n);
                pu.running[at] = cost0 + inc - cost;
                pu.heavy_before[at] = heavy0 + lanes_below(heavies, lane);
            }
            const bool is8 = d > rule.split && row_groups(d, rule.groups) == kXcds;
            const unsigned long long eights = __ballot(is8);
            if (is8) pu.rank8[p - first_split] = rows8 + lanes_below(eights, lane);
            n_units += __popcll(heads);
            cost0 += __builtin_amdgcn_readlane(inc, 63);
            heavy0 += __popcll(heavies);
            rows8 += __popcll(eights);
        }
    }
}

// ---------------------------------------------------------------------------
// Split rows in the launch plan (plan.hip's subject as well; counted next to the placing of the wide rows).
// ---------------------------------------------------------------------------
constexpr int kClasses = 4;                 // rows stored in 8, 16, 32, 64 column groups
// The split rows' unit counts per group are laid out [class][group][rank in the class].
struct ClassLayout {
    int rows[kClasses];                     // split rows of each class
    int base[kClasses];                     // where the class's counts start
    int above[kClasses];                    // rows of the classes with more groups
    int total;                              // counts in all
};

// A split row's place in its class: rows of 8 groups follow the caller's row ids, the longer
// ones come largest first (they touch all of X whatever their id; the hub workload measured
// 2 % faster that way: 2.31 against 2.36 ms at N = 256).
struct SplitRow {
    int d, groups, cls, rank;
};
__device__ __forceinline__ SplitRow split_row(const int32_t *__restrict__ s_indptr, int64_t first_split, int n_split,
                                              int lr, const int *__restrict__ rank8, const ClassLayout &cl, int forced)
{
    SplitRow s;
    s.d = s_indptr[first_split + lr + 1] - s_indptr[first_split + lr];
    s.groups = row_groups(s.d, forced);
    s.cls = 31 - __clz(s.groups / kXcds);
    s.rank = s.cls == 0 ? rank8[lr] : n_split - cl.above[s.cls] - 1 - lr;
    return s;
}

// Which split row and which of its column groups a lane of wavefront `item` looks at: rows of 8 groups eight to a
// wavefront, the others (behind them) one.  (Most have 8: of the 80,668 of a power-law matrix with 125 M non-zeros 68,512 have
// 1,024 or fewer.  With a wavefront for each, of which 56 lanes had nothing to do, the counting and the writing of the pieces
// took 43 and 33 us on 60 M non-zeros; 27 and 20 so.)
struct SplitLane {
    int lr, group;
    bool eight, valid;
};
inline __host__ __device__ int split_items(const ClassLayout &cl, int n_split) { return (cl.rows[0] + 7) / 8 + n_split - cl.rows[0]; }
__device__ __forceinline__ SplitLane split_lane(const ClassLayout &cl, int n_split, int item)
{
    const int lane = threadIdx.x & 63, n8 = cl.rows[0], items8 = (n8 + 7) / 8;
    if (item < items8) {
        const int lr = item * 8 + lane / 8;
        return {min(lr, n8 - 1), lane % 8, true, lr < n8};
    }
    return {n8 + item - items8, lane, false, true};
}
// Sum over the lanes of the row up to this one.
__device__ __forceinline__ int row_inclusive_sum(int v, bool eight)
{
    if (!eight) return wave_inclusive_sum(v);
    const int at = threadIdx.x & 7;
    int t = lanes_moved<0x111, 0xf>(v);
    v += at >= 1 ? t : 0;
    t = lanes_moved<0x112, 0xf>(v);
    v += at >= 2 ? t : 0;
    t = lanes_moved<0x114, 0xf>(v);
    return v + (at >= 4 ? t : 0);
}

// A lane per column group of a split row: pieces per group (into `bins`) and per row,
// and what they cost per queue (column group g belongs to queue g % n_queues).
struct SplitArgs {
    int *gcount;                              // [split row][64]: non-zeros per group; those of wide rows are added up here
    const int32_t *s_indptr;
    int64_t first_split;
    int n_split;
    const int *rank8;
    ClassLayout cl;
    int forced, piece, cost_shift, n_queues;
    int *bins, *row_units, *row_done;
    int n_groups;                             // workgroups that count
    int *group_cost;                          // [workgroup][8]
    int n_wide;                               // the last of them are wide rows: row i's chunks are first_chunk[i] to [i + 1]
    const int *first_chunk, *chunk_count;     // of those; [chunk][64]
};
// Threads of the workgroups that place chunks of wide rows and count split rows.  A chunk is a chain of 16 rounds by four
// wavefronts and of four by sixteen, but seven chunks are under way on a compute unit with the former and two with the
// latter: 2.45 M non-zeros (35 chunks) 10.4 us with 256 threads, 6.8 with 1,024; 30 M (4,200) 62 and 76; 125 M (5,100) 90
// and 101.  The line lies where the large workgroups stop being on the card all at once, twice over.
inline int place_threads(int64_t chunks) { return chunks > 1024 ? 256 : 1024; }
// Workgroups that count: an item (see SplitLane) per wavefront, a few items where there are very many.
constexpr int kSplitGroups = 1024;
inline int split_groups(int64_t n, int threads) { return (int)std::min<int64_t>((n + threads / 64 - 1) / (threads / 64), kSplitGroups); }
// (What the rows cost is added up by plan_head_kernel: eight atomics per workgroup, all of them to the same eight words,
// took 14 of 22 us for 29 k rows.)
template <int T>
__device__ __forceinline__ void count_split_rows(const SplitArgs &a, int workgroup, int (*part)[kXcds])
{
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int kWaves = T / 64;
    int cost = 0;
    const int n_items = split_items(a.cl, a.n_split);
    for (int item = workgroup * kWaves + w; item < n_items; item += a.n_groups * kWaves) {
        const SplitLane at = split_lane(a.cl, a.n_split, item);
        const int lr = at.lr;
        const SplitRow s = split_row(a.s_indptr, a.first_split, a.n_split, lr, a.rank8, a.cl, a.forced);
        const int wide = lr - (a.n_split - a.n_wide);
        const bool mine = at.valid && at.group < s.groups;
        int c = 0;
        if (wide >= 0) {
            const int to = a.first_chunk[wide + 1];
#pragma unroll 4
            for (int i = a.first_chunk[wide]; i < to; i++) c += a.chunk_count[(int64_t)i * kMaxGroups + at.group];
            if (mine) a.gcount[(int64_t)lr * kMaxGroups + at.group] = c;
        } else if (mine) {
            c = a.gcount[(int64_t)lr * kMaxGroups + at.group];
        }
        if (!mine) c = 0;
        const int u = (c + a.piece - 1) / a.piece;
        if (mine) a.bins[a.cl.base[s.cls] + at.group * a.cl.rows[s.cls] + s.rank] = u;
        if (c > 0) cost += ((c + 9 * u) >> a.cost_shift) + u;
        const int total = row_inclusive_sum(u, at.eight);
        if (at.valid && lane % (at.eight ? 8 : 64) == (at.eight ? 7 : 63)) {
            a.row_units[lr] = total;
            a.row_done[lr] = a.row_done[a.n_split + lr] = 0;
        }
    }
    cost += __shfl_xor(cost, 8);
    cost += __shfl_xor(cost, 16);
    cost += __shfl_xor(cost, 32);
    if (lane < kXcds) part[w][lane] = cost;
    __syncthreads();
    if ((int)threadIdx.x < kXcds) {
        for (int q = 1; q < kWaves; q++) cost += part[q][threadIdx.x];
        a.group_cost[workgroup * kXcds + threadIdx.x] = cost;
    }
}

// plan.hip
// The split rows' counters, and the kernel arguments that say where they are (gcount, first_chunk, chunk_count and n_wide left to
// the caller).  slot: what becomes the handle's long_slot, with its counters behind.
int prepare_split_rows(Arena *tmp, const accel_handle *h, const SortedRows &sr, const UnitRule &rule, const PlanUnits &pu,
                       const Mail *stats, DevBuf *slot, SplitArgs *out);
// The rest of the plan, behind the counting of the split rows.
int build_work_list(Arena *tmp, accel_handle *h, const SortedRows &sr, const UnitRule &rule, const Shares &sh,
                    const PlanUnits &pu, const SplitArgs &split, DevBuf *slot, int64_t n_short_units, int *zeroed, Mail *mail,
                    hipStream_t s);
// ints that must be zero when build_work_list is called (place_rows clears them)
int64_t plan_zeroed_ints(int64_t n_split, const Mail *stats, int groups);

}  // namespace accel
