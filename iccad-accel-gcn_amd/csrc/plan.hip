// The launch plan (work list) of a preprocessed matrix, built on the GPU.  One work unit per
// wavefront, kWavesPerGroup units per workgroup, as int4 (x, y, z, w):
//   x <= 384 : whole rows of one block4 entry (degree, first row, first non-zero,
//              (w_nz << 16) + n_rows): the entry itself, or a run of its rows when
//              the plan's unit is smaller than the entry;
//   x  > 384 : a piece of a split row: partial-sum slot x - 385, row y, first
//              non-zero z, length w <= plan_unit, all of one column group;
//   w == 0   : padding, nothing to do.
// Workgroups are dispatched to the eight dies round-robin (workgroup i runs on
// die i % 8), so the list is laid out as eight interleaved queues.  Column group
// g belongs to die g % 8.  A queue holds, in this order: the pieces of the rows
// stored in 64 groups (the longest rows), one group after the other, largest
// rows first; then the same for the rows with 32, 16 and 8 groups (the rows of
// an 8-group bin in the order of the caller's row ids); then the
// queue's share of the whole-row units.  While a die works through one group its
// L2 only has to hold that group's share of X.
// The whole-row units are put in the order of the caller's row ids (of each unit's
// first row) and that sequence is cut into eight consecutive shares, one per queue,
// sized so that all queues carry about the same load.  Graphs whose neighbouring
// row ids have neighbouring columns (most graphs with a meaningful vertex order)
// lose that locality to the degree sort; this gives it back: at any time a die
// works on a narrow band of the caller's rows.
//
// Nothing here is sorted: the pass that placed the rows (place_rows in preprocess.hip) knows of
// every row, in the caller's order, whether it starts a unit, so a scan of the counts per share
// of rows puts the units in that order (list_units in preprocess.h).  The pieces of a column group are
// ordered by a scan over (class of rows, group, row of the class).  What bounds all of it is
// the number of dependent launches (2 to 5 us each), not bytes: three launches and no
// synchronisation before the last (the units are listed and the split rows counted in launches of
// preprocess.hip), where there were 45 launches and two.
#include "preprocess.h"

namespace accel {
namespace {

static ClassLayout class_layout(int64_t n_split, const Mail *stats, int groups)
{
    ClassLayout c{};
    if (groups) {
        for (int i = 0; i < kClasses; i++) c.rows[i] = (kXcds << i) == groups ? (int)n_split : 0;
    } else {
        c.rows[1] = stats->stat[kStatRows16];
        c.rows[2] = stats->stat[kStatRows32];
        c.rows[3] = stats->stat[kStatRows64];
        c.rows[0] = (int)n_split - c.rows[1] - c.rows[2] - c.rows[3];
    }
    for (int i = 0, at = 0; i < kClasses; i++) {
        c.base[i] = at;
        at += (kXcds << i) * c.rows[i];
        c.total = at;
    }
    for (int i = kClasses - 1, n = 0; i >= 0; i--) {
        c.above[i] = n;
        n += c.rows[i];
    }
    return c;
}

__device__ __forceinline__ int64_t plan_index(int queue, int pos, int n_queues)
{
    // queue q, position p  ->  slot of wavefront (p % 4) in workgroup (p / 4) * n_queues + q
    return ((int64_t)(pos / kWavesPerGroup) * n_queues + queue) * kWavesPerGroup + pos % kWavesPerGroup;
}

// Where everything goes in the list: computed by one workgroup, read by the kernels that write it.
struct PlanHead {
    int queue_long[kXcds];       // pieces in each queue
    int cut[kXcds + 1];          // queue q takes the units whose running cost lies in [cut[q], cut[q + 1])
    int first[kXcds + 1];        // first unit of each queue
    int bin_off[kPlanBins];      // where the pieces of a (class, column group) bin start in their queue
    int per_queue;               // units per queue, a multiple of kWavesPerGroup
};

__device__ __forceinline__ int queue_of(int running_cost, const int *cut)
{
    int q = 0;
#pragma unroll
    for (int i = 1; i < kXcds; i++) q += running_cost >= cut[i];
    return q;
}

// Queue q takes max(0, level - its pieces' cost) of the whole-row units' cost, level being the
// smallest common level that takes all of it.
__global__ __launch_bounds__(512) void plan_head_kernel(const int *__restrict__ bins, ClassLayout cl, int n_split,
                                                        const int *__restrict__ group_cost, int n_groups,
                                                        const int *__restrict__ running, const int *__restrict__ sums,
                                                        int pitch, int n_shares, int n_queues,
                                                        PlanHead *__restrict__ head, Mail *__restrict__ mail)
{
    static_assert(kXcds * 64 == 512, "one wavefront per queue");
    __shared__ int at[kPlanBins + 1], off[kPlanBins], queue_long[kXcds], cut[kXcds + 1], first[kXcds + 1];
    __shared__ int part[kXcds][kXcds];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    int cost = 0;                                                  // of the split rows' pieces for die t % 8
#pragma unroll 4
    for (int i = t; i < n_groups * kXcds; i += 512) cost += group_cost[i];
    const int n = sums[kSumUnits * pitch + n_shares];
    if (t <= kPlanBins) {
        int v = 0;
        if (n_split > 0) {
            if (t == kPlanBins) {
                v = bins[cl.total];
            } else {
                int cls = 0;                                       // bins of a class: 8, 16, 32, 64 in turn
                while (t >= plan_bin(kXcds << (cls + 1), 0)) cls++;
                v = bins[cl.base[cls] + (t - plan_bin(kXcds << cls, 0)) * cl.rows[cls]];
            }
        }
        at[t] = v;
    }
    cost += __shfl_xor(cost, 8);
    cost += __shfl_xor(cost, 16);
    cost += __shfl_xor(cost, 32);
    if (lane < kXcds) part[w][lane] = cost;
    __syncthreads();
    if (t < n_queues) {
        // a die first takes the pieces of the rows with the most groups (the longest rows), one
        // group after the other, then those of the next class, ...
        int pos = 0;
        for (int ng = kMaxGroups; ng >= kXcds; ng /= 2)
            for (int g = t; g < ng; g += n_queues) {
                const int b = plan_bin(ng, g);
                off[b] = pos;
                pos += at[b + 1] - at[b];
            }
        queue_long[t] = pos;
    }
    if (w == 1) {
        // the smallest level that takes all of it, 64 candidates at a time
        const long long short_cost = sums[kSumCost * pitch + n_shares];
        int queue_cost[kXcds] = {};
#pragma unroll
        for (int q = 0; q < kXcds; q++) {
            int c = 0;
#pragma unroll
            for (int v = 0; v < kXcds; v++) c += part[v][q];
            if (n_queues == kXcds) queue_cost[q] = c; else queue_cost[0] += c;
        }
        long long lc[kXcds], lo = 0, hi = short_cost;      // the level lies in [lo, hi]
#pragma unroll
        for (int q = 0; q < kXcds; q++) {
            lc[q] = q < n_queues ? queue_cost[q] : 0x7fffffffffffffffLL;
            if (q < n_queues && lc[q] + short_cost > hi) hi = lc[q] + short_cost;
        }
        while (lo < hi) {
            const long long step = (hi - lo + 63) / 64, mid = lo + lane * step;
            long long taken = 0;
#pragma unroll
            for (int q = 0; q < kXcds; q++) taken += mid > lc[q] ? mid - lc[q] : 0;
            const int k = __popcll(__ballot(mid < hi && taken < short_cost));     // the first k are too low
            if (k == 0) break;
            const long long first_low = lo;
            lo = first_low + (k - 1) * step + 1;
            if (first_low + k * step < hi) hi = first_low + k * step;
        }
        if (lane == 0) {
            long long run = 0;
            for (int q = 0; q < n_queues; q++) {
                cut[q] = (int)(run < short_cost ? run : short_cost);
                run += lo > lc[q] ? lo - lc[q] : 0;
            }
            for (int q = n_queues; q <= kXcds; q++) cut[q] = 0x7fffffff;   // queues that do not exist take nothing
        }
    }
    __syncthreads();
    // first[q]: the first unit whose running cost reaches cut[q]; wavefront q searches, 64 units per step
    if (w < n_queues) {
        int lo = 0, hi = n;                                // the answer lies in [lo, hi]
        while (lo < hi) {
            const int step = (hi - lo + 63) / 64;
            const int i = lo + lane * step;
            const bool below = i < hi && running[i] < cut[w];
            const int k = __popcll(__ballot(below));       // the first k probes are below
            if (k == 0) { hi = lo; break; }
            const int nlo = lo + (k - 1) * step + 1, nhi = min(hi, lo + k * step);
            lo = nlo; hi = nhi;
        }
        if (lane == 0) first[w] = w == 0 ? 0 : lo;
    } else if (lane == 0) {
        first[w] = n;
    }
    if (t == 0) first[kXcds] = n;
    __syncthreads();
    if (t < kPlanBins) head->bin_off[t] = n_split > 0 ? off[t] : 0;
    if (t < kXcds) head->queue_long[t] = t < n_queues ? queue_long[t] : 0;
    if (t <= kXcds) {
        head->cut[t] = cut[t];
        head->first[t] = first[t];
    }
    if (t == 0) {
        int most = 0;
        for (int q = 0; q < n_queues; q++) most = max(most, queue_long[q] + first[q + 1] - first[q]);
        most = (most + kWavesPerGroup - 1) / kWavesPerGroup * kWavesPerGroup;
        head->per_queue = most;
        mail->per_queue = most;
        mail->n_pieces = at[kPlanBins];
        mail->n_units = n;
    }
}

// Writes the list.  The first workgroups take split rows, a lane per column group (see SplitLane),
// and write their pieces; the others the units of whole rows, one per thread.
// Inside its queue a unit goes behind the pieces, in the order of the caller's row ids,
// except that the queue's last kTailLight light units (few non-zeros: short chains of
// gathers) are held back and placed at the very end, so that a queue does not end on a
// long chain.  They are the light units with the highest ids of the queue's share, i.e.
// they lie in the band of rows the die is working on at that time anyway.
// heavy_before[s] = heavy units among the first s, [n] = all.
constexpr int kTailLight = 2048;             // two rounds of the 1,024 wavefronts a die holds
struct EmitArgs {
    const int *gcount;
    const int32_t *s_indptr;
    int64_t first_split;
    int n_split, piece_groups;               // split rows; workgroups that take them
    const int *slot, *bins, *rank8;
    ClassLayout cl;
    int forced, piece;
    const int4 *units;
    const int *running, *heavy_before;
    int n_units;
    const PlanHead *head;
    int n_queues, room;
    int4 *work;
};

__device__ __forceinline__ void emit_pieces(const EmitArgs &a, int item)
{
    const SplitLane at = split_lane(a.cl, a.n_split, item);
    const int lr = at.lr, g = at.group;
    const SplitRow s = split_row(a.s_indptr, a.first_split, a.n_split, lr, a.rank8, a.cl, a.forced);
    const int c = at.valid && g < s.groups ? a.gcount[(int64_t)lr * kMaxGroups + g] : 0;
    const int u = (c + a.piece - 1) / a.piece;
    const int c_inc = row_inclusive_sum(c, at.eight), u_inc = row_inclusive_sum(u, at.eight);
    if (c == 0) return;
    const int row = (int)(a.first_split + lr);
    const int loc = a.s_indptr[row] + c_inc - c, sl = a.slot[lr] + u_inc - u;
    const int bin0 = a.cl.base[s.cls] + g * a.cl.rows[s.cls];
    const int pos0 = a.head->bin_off[plan_bin(s.groups, g)] + a.bins[bin0 + s.rank] - a.bins[bin0];
    for (int k = 0, off = 0; off < c; k++, off += a.piece)
        a.work[plan_index(g % a.n_queues, pos0 + k, a.n_queues)] =
            make_int4(kDegBound + 1 + sl + k, row, loc + off, min(a.piece, c - off));
}

__global__ __launch_bounds__(kThreads) void emit_plan_kernel(EmitArgs a)
{
    const int per_queue = a.head->per_queue;
    if (per_queue > a.room) return;                    // the host makes room and launches again
    if ((int)blockIdx.x < a.piece_groups) {
        const int item = (int)blockIdx.x * kWaves4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (item < split_items(a.cl, a.n_split)) emit_pieces(a, item);
        return;
    }
    const int tid = ((int)blockIdx.x - a.piece_groups) * kThreads + threadIdx.x;
    if (tid < a.n_units) {
        const int q = queue_of(a.running[tid], a.head->cut);
        const int f = a.head->first[q], n_q = a.head->first[q + 1] - f;
        const int h0 = a.heavy_before[f], h_me = a.heavy_before[tid];
        const int light_all = n_q - (a.heavy_before[f + n_q] - h0);            // light units of this queue
        const int light_me = (tid - f) - (h_me - h0);                          // ... before this unit
        const bool is_light = a.heavy_before[tid + 1] == h_me;
        const int kept = max(0, light_all - kTailLight);                 // light units that stay in line
        int pos;
        if (is_light && light_me >= kept)
            pos = n_q - (light_all - light_me);                                // held back: the last ones
        else
            pos = (tid - f) - max(0, light_me - kept);                         // in line, minus those held back before it
        a.work[plan_index(q, a.head->queue_long[q] + pos, a.n_queues)] = a.units[tid];
    }
    const int all = ((int)gridDim.x - a.piece_groups) * kThreads;
    for (int q = 0; q < a.n_queues; q++) {             // the rest of the shorter queues: padding
        const int len = a.head->queue_long[q] + a.head->first[q + 1] - a.head->first[q];
        for (int pos = len + tid; pos < per_queue; pos += all)
            a.work[plan_index(q, pos, a.n_queues)] = make_int4(0, 0, 0, 0);
    }
}

}  // namespace

// Split rows are added up by the gather kernel itself (the wavefront that stores a row's last
// piece does it: one launch) when the plan holds at most this many pieces, by a second kernel
// otherwise.  In the kernel every piece ends on a wait for its stores and one atomic, some
// microseconds of latency that nothing hides on a launch-bound matrix but that is still less
// than a second launch costs; with many pieces it adds up to more.  Measured, runs queued
// back to back, in-kernel against second kernel at N = 16 / 64 / 128: 96 pieces (1.9 M
// non-zeros) 0.88 / 0.94 / 0.96; 5,160 (1.2 M) 0.88 / 0.90 / 0.96; 8,848 (1.6 M) 0.82 / 0.94 /
// 0.98; 7,760 (2.4 M) 0.99 / 0.96 / 0.98; 68,608 (14 M) 1.01 / 1.02 / 1.02; 144,561 (27 M)
// 1.24 / 1.08 / 1.09; 0.5 M pieces (115 M non-zeros, nearly every row split) 1.30 at N = 64.
constexpr int64_t kFusedReduceMaxPieces = 16384;

int64_t plan_zeroed_ints(int64_t n_split, const Mail *stats, int groups)
{
    if (n_split == 0) return 0;
    return scan_zeroed(n_split) + scan_zeroed(class_layout(n_split, stats, groups).total);
}

int prepare_split_rows(Arena *tmp, const accel_handle *h, const SortedRows &sr, const UnitRule &rule, const PlanUnits &pu,
                       const Mail *stats, DevBuf *slot, SplitArgs *out)
{
    const int n_split = (int)h->n_split_rows;
    int rc;
    SplitArgs a{};
    a.s_indptr = sr.s_indptr;
    a.first_split = h->rows - n_split;
    a.n_split = n_split;
    a.rank8 = pu.rank8;
    a.cl = class_layout(n_split, stats, rule.groups);
    a.forced = rule.groups;
    // pieces of split rows hold up to this many non-zeros, units of several whole rows up to plan_unit
    a.piece = std::max(h->plan_unit, h->plan_split);
    a.cost_shift = rule.cost_shift;
    a.n_queues = h->plan_queues;                       // 8 interleaved queues, or 1 (plain order)
    a.n_groups = split_groups(split_items(a.cl, n_split), place_threads(h->n_chunks - h->n_lone_chunks));
    // the slots of each split row, and behind them two counters per split row (zero between launches)
    if ((rc = slot->alloc(sizeof(int) * (size_t)(3 * (int64_t)n_split + 1)))) return rc;
    a.row_done = slot->as<int>() + n_split + 1;
    if (n_split > 0) {
        if ((rc = tmp->alloc(&a.row_units, (size_t)n_split))) return rc;
        if ((rc = tmp->alloc(&a.group_cost, (size_t)a.n_groups * kXcds))) return rc;
        if ((rc = tmp->alloc(&a.bins, (size_t)a.cl.total + 1))) return rc;
    }
    *out = a;
    return ACCEL_OK;
}

int build_work_list(Arena *tmp, accel_handle *h, const SortedRows &sr, const UnitRule &rule, const Shares &sh,
                    const PlanUnits &pu, const SplitArgs &split, DevBuf *dslot, int64_t n_short_units, int *zeroed, Mail *mail,
                    hipStream_t s)
{
    const int *share_sums = pu.sums, *gcount = split.gcount;
    const int piece_nz = split.piece, forced = rule.groups, nq = split.n_queues;
    const int n_split = split.n_split;
    const int64_t first_split = split.first_split;
    const ClassLayout &cl = split.cl;
    const int pitch = sh.pitch + kWaves4;
    int rc;
    const int4 *units = pu.units;
    const int *running = pu.running, *heavy = pu.heavy_before, *rank8 = pu.rank8;
    int *bins = split.bins;
    PlanHead *head;
    if ((rc = tmp->alloc(&head, 1))) return rc;
    int *slot = dslot->as<int>();
    if (n_split > 0) {
        launch_scans({{{split.row_units, slot, n_split, 0, zeroed}, {bins, bins, cl.total, 0, zeroed + scan_zeroed(n_split)}}, {}}, 2, s);
    }
    plan_head_kernel<<<dim3(1), dim3(512), 0, s>>>(bins, cl, n_split, split.group_cost, split.n_groups, running, share_sums, pitch, sh.n, nq, head,
                                                  mail);
    // Room for the list, before its length is known: the queues are level in cost, not in units,
    // so each gets half as much again as its share of the units.  Where that is not enough
    // (queues of single light rows next to queues of full units) the kernels below write nothing,
    // and a second round has the length.
    const int64_t most = n_short_units + cl.total + (h->nnz - h->nnz_short) / piece_nz;
    int64_t room = std::min(most, most / nq + most / (2 * nq) + 4096);
    DevBuf dwork;
    for (int round = 0;; round++) {
        room = (room + kWavesPerGroup - 1) / kWavesPerGroup * kWavesPerGroup;
        if (room * nq > (int64_t)0x7fffffff) {
            set_error("the launch plan would exceed 2^31 work units");
            return ACCEL_ERR_ARG;
        }
        if ((rc = dwork.alloc(sizeof(int4) * (size_t)(room * nq)))) return rc;
        const int piece_groups = (int)grid_for((int64_t)split_items(cl, n_split) * 64);
        const EmitArgs ea{gcount, sr.s_indptr, first_split, n_split, piece_groups, slot, bins, rank8, cl, forced, piece_nz,
                          units, running, heavy, (int)n_short_units, head, nq, (int)room, dwork.as<int4>()};
        emit_plan_kernel<<<dim3(piece_groups + grid_for(std::max<int64_t>(n_short_units, kThreads))), dim3(kThreads), 0,
                           s>>>(ea);
        ACCEL_HIP(hipGetLastError());
        ACCEL_HIP(hipStreamSynchronize(s));
        if (mail->per_queue <= room) break;
        if (round > 0) {
            set_error("internal: the launch plan does not fit its own length");
            return ACCEL_ERR_STATE;
        }
        room = mail->per_queue;
        give_memory(dwork.release(), InUse::no);
    }
    if (mail->n_units != (int)n_short_units) {
        set_error("internal: %d units of whole rows, %lld were expected from the degree histogram", mail->n_units,
                  (long long)n_short_units);
        return ACCEL_ERR_STATE;
    }
    h->n_units = (int64_t)mail->per_queue * nq;
    h->n_long_units = n_split > 0 ? mail->n_pieces : 0;
    h->work = static_cast<int32_t *>(dwork.release());
    h->long_slot = static_cast<int32_t *>(dslot->release());
    h->row_done = h->long_slot + n_split + 1;
    h->fused_reduce = h->plan_reduce_option == 1 ||
                      (h->plan_reduce_option == 0 && h->n_long_units <= kFusedReduceMaxPieces);
    return ACCEL_OK;
}

}  // namespace accel
