// GPU preprocessing for the SpMM operator: CSR validation, stable degree sort, sorted copy of the
// non-zeros and the block4 partition metadata (the launch plan is plan.hip's).  Integer work,
// bound by the number of dependent launches on small matrices and by streaming the non-zeros
// on large ones.
//
// The metadata rules are those of upstream's block_level_partition.py:7-21
// (tables) and :48-103 (walk); the walk is restated as a closed form per row so
// that every row can be treated by itself:
//   - a row of degree d in 1..384 that sits (r - s) rows into its maximal run of
//     equal-degree rows (run start s) opens a block iff (r - s) % rows[d] == 0;
//     the block takes up to rows[d] rows of that run;
//   - a row of degree d > 384 opens ceil(d / 384) blocks;
//   - rows of degree 0 open none.
//
// The sort is by bins: one per degree 0..384 and one for all longer rows.  With rows in
// ascending degree order each of the first 385 bins is one run of equal degree, so once the
// bins are counted everything about a row of up to 384 non-zeros is a closed form of its degree
// and its place in the bin: its sorted place, its first non-zero, the block and the unit of the
// launch plan that it opens.  One pass counts (degree_kernel), one workgroup per bin scans the
// counts over the shares of rows (bin_scan_kernel), one pass places the rows and writes all of
// that (place_rows_kernel).  The longer rows, few on most graphs, are placed by comparison (or
// by a radix sort when there are many).
// Nine launches on a graph of 2.45 M non-zeros (five more where more than 8,192 rows are longer than 384) and two
// synchronisations; a radix sort of all rows with scans for every product took 100 and four.
#include <chrono>
#include <climits>

#include "preprocess.h"

namespace accel {
namespace {

// ---------------------------------------------------------------------------
// Degrees: validation, statistics, bins
// ---------------------------------------------------------------------------
// Does the matrix have its non-zeros near the diagonal (of the rows x cols rectangle)?
// Every kLocalityStride-th row contributes up to kLocalitySample of its non-zeros, evenly spaced; one counts
// as local when its column is within `band` columns of the row's place.  Rows whose indptr
// entries point outside [0, nnz) are skipped (they are an error anyway).
constexpr int kLocalityStride = 16, kLocalitySample = 16;

struct DegreeArgs {
    const int32_t *indptr, *idx;              // idx null: no locality sample
    int64_t rows, cols, nnz;
    int share, n_shares, pitch;
    int split, alt_split;                     // the two thresholds the rows may be split at
    int band;
};

// One wavefront per share of rows: counts its rows per bin in LDS, without atomics on memory;
// a workgroup's four columns of counts go out side by side.  bins[b * pitch + share];
// stats[workgroup * 16 + kStat*].
__global__ __launch_bounds__(kThreads) void degree_kernel(DegreeArgs a, int *__restrict__ bins, int *__restrict__ stats)
{
    __shared__ int cnt[kWaves4][kBins];
    __shared__ int part[kWaves4][kStatCount];
    for (int i = threadIdx.x; i < kBins * kWaves4; i += kThreads) (&cnt[0][0])[i] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = (int)blockIdx.x * kWaves4 + w;
    int st[kStatCount];
#pragma unroll
    for (int k = 0; k < kStatCount; k++) st[k] = 0;
    const int64_t r_end = min(a.rows, (int64_t)(c + 1) * a.share);
    for (int64_t r1 = (int64_t)c * a.share; r1 < r_end; r1 += 4 * 64) {
        int los[4], his[4], befores[4];                      // four rounds' rows are on their way at once
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t r = r1 + j * 64 + lane;
            los[j] = r < r_end ? a.indptr[r] : 0;
            his[j] = r < r_end ? a.indptr[r + 1] : 0;
            befores[j] = r < r_end && r > 0 && lane == 0 ? a.indptr[r - 1] : 0;
        }
        int sample[4];                                       // position of this lane's sampled non-zero, or -1
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t r = r1 + j * 64 + lane;
            const bool ok = r < r_end;
            const int lo = los[j], hi = his[j];
            int before = __shfl_up(lo, 1);
            if (lane == 0) before = befores[j];
            int d = hi - lo;
            if (ok) {
                const bool bad = hi < lo || (r == 0 && lo != 0) || (r == a.rows - 1 && (int64_t)hi != a.nnz);
                if (hi < lo) d = 0;
                if (r > 0 && d < lo - before) st[kStatUnsorted] = 1;
                st[kStatBadIndptr] |= bad;
                st[kStatMaxDegree] = max(st[kStatMaxDegree], d);
                if (d > kDegBound) st[kStatLongBlocks] += (d + kDegBound - 1) / kDegBound;
                if (d > kWideRow) {
                    st[kStatWideRows]++;
                    st[kStatLoneChunks] += d <= kWideChunk;
                    st[kStatWideChunks] += (d + kWideChunk - 1) / kWideChunk;
                    const int ng = row_groups(d, 0);
                    st[kStatRows16] += ng == 16;
                    st[kStatRows32] += ng == 32;
                    st[kStatRows64] += ng == 64;
                }
                st[kStatBig] += d > 32 * a.split;
                st[kStatBigAlt] += d > 32 * a.alt_split;
                atomicAdd(&cnt[w][min(d, kLongBin)], 1);
            }
            // four of the 64 rows are sampled, by 16 lanes each, spread over the row whatever its order
            const int from = lane / kLocalitySample * kLocalityStride, i = lane % kLocalitySample;
            const int ra = __shfl(lo, from);
            int rd = __shfl(ok ? hi - lo : 0, from);
            if (ra < 0 || rd < 0 || (int64_t)ra + rd > a.nnz) rd = 0;
            const int n = min(rd, kLocalitySample);
            sample[j] = a.idx && i < n ? ra + (int)((int64_t)i * rd / n) : -1;
        }
        int col[4];
#pragma unroll
        for (int j = 0; j < 4; j++) col[j] = sample[j] >= 0 ? a.idx[sample[j]] : 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (sample[j] < 0) continue;
            const int64_t r = r1 + j * 64 + lane / kLocalitySample * kLocalityStride;
            const int64_t off = (int64_t)col[j] - (a.rows > 1 ? r * (a.cols - 1) / (a.rows - 1) : 0);
            st[kStatSampled]++;
            st[kStatLocal] += (off < 0 ? -off : off) <= a.band;
        }
    }
    static_assert(kLocalityStride == 16 && kLocalitySample == 16, "the lanes of a round are dealt out for these");
    static_assert(kWideRow < 2 * kXcds * kGroupMinPiece, "rows of 16 and more groups are wide ones");
#pragma unroll
    for (int k = 0; k < kStatCount; k++) {
        st[k] = k <= kStatMaxDegree ? wave_max(st[k]) : wave_sum(st[k]);
        if (lane == 0) part[w][k] = st[k];
    }
    __syncthreads();
    for (int b = threadIdx.x; b < kBins; b += kThreads)
        *reinterpret_cast<int4 *>(bins + (int64_t)b * a.pitch + (int)blockIdx.x * kWaves4) =
            make_int4(cnt[0][b], cnt[1][b], cnt[2][b], cnt[3][b]);
    if ((int)threadIdx.x < kStatCount) {
        const int k = threadIdx.x;
        int v = part[0][k];
        for (int q = 1; q < kWaves4; q++) v = k <= kStatMaxDegree ? max(v, part[q][k]) : v + part[q][k];
        stats[(int)blockIdx.x * 16 + k] = v;
    }
}

// Workgroup b < kBins: exclusive scan of bin b's counts over the shares, in place, and the bin's
// total.  The last workgroup adds up the statistics.  Totals and statistics go to the host's
// memory as well.
__global__ __launch_bounds__(kThreads) void bin_scan_kernel(int *__restrict__ bins, int pitch,
                                                            const int *__restrict__ stats, int n_groups,
                                                            int *__restrict__ total_out, Mail *__restrict__ mail)
{
    __shared__ int lds[kWaves4];
    __shared__ int part[kThreads];
    const int b = blockIdx.x;
    if (b == kBins) {
        const int k = threadIdx.x & 15;
        int v = 0;
        if (k < kStatCount)
#pragma unroll 8                                         // (not unrolled: 17 us for 958 workgroups' statistics, 6 so)
            for (int g = threadIdx.x >> 4; g < n_groups; g += kThreads / 16) {
                const int t = stats[g * 16 + k];
                v = k <= kStatMaxDegree ? max(v, t) : v + t;
            }
        part[threadIdx.x] = v;
        __syncthreads();
        if (threadIdx.x < 16) {
            for (int q = 1; q < kThreads / 16; q++) {
                const int t = part[q * 16 + k];
                v = k <= kStatMaxDegree ? max(v, t) : v + t;
            }
            mail->stat[k] = v;
        }
        return;
    }
    int *row = bins + (int64_t)b * pitch;
    constexpr int kVecs = kMaxShares / (4 * kThreads);           // 16-byte vectors per thread, all loaded at once
    int4 v[kVecs];
    int carry = 0;
#pragma unroll
    for (int j = 0; j < kVecs; j++) {
        const int c = 4 * (j * kThreads + (int)threadIdx.x);
        v[j] = c < pitch ? *reinterpret_cast<const int4 *>(row + c) : make_int4(0, 0, 0, 0);   // pitch is a multiple of 4
    }
#pragma unroll
    for (int j = 0; j < kVecs; j++) {
        const int c = 4 * (j * kThreads + (int)threadIdx.x);
        if (4 * j * kThreads >= pitch) break;
        int total, run = block_exclusive_sum<kThreads>(v[j].x + v[j].y + v[j].z + v[j].w, lds, total);
        run += carry;
        if (c < pitch)
            *reinterpret_cast<int4 *>(row + c) =
                make_int4(run, run + v[j].x, run + v[j].x + v[j].y, run + v[j].x + v[j].y + v[j].z);
        carry += total;
    }
    if (threadIdx.x == 0) {
        total_out[b] = carry;
        mail->hist[b] = carry;
    }
}

// ---------------------------------------------------------------------------
// Placing the rows
// ---------------------------------------------------------------------------
struct PlaceArgs {
    const int32_t *indptr;
    int64_t rows;
    int share, n_shares, pitch;
    const int *bins;                          // scanned counts
    const int *bin_total;
    UnitRule rule;
    // outputs
    int32_t *perm;                            // null: the rows are in order already
    uint32_t *place;                          // caller's row -> sorted row; long rows come later
    int32_t *s_indptr;
    int4 *block4;
    int *run_row, *run_nz;                    // [kBins + 1], [kBins]
    int *long_deg;                            // degrees and ids of the long rows, in the caller's order
    uint32_t *long_row;
    int *sums;                                // [kSums][pitch + kWaves4]
    int *zero;                                // n_zero ints to clear
    int64_t n_zero;
};

// One wavefront per share of rows ranks its rows inside their bins (ballots; each wavefront has
// counters of its own, so that no barrier is needed between rounds).  The sorted row pointers and
// the blocks of up to 384 non-zeros are written by position, without looking at rows.
__global__ __launch_bounds__(kThreads) void place_rows_kernel(PlaceArgs a)
{
    __shared__ int run_row[kBins + 1], run_nz[kBins], run_blk[kBins], lds[kWaves4];
    __shared__ int next[kWaves4][kBins];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    static_assert(kBins <= 2 * kThreads, "two bins per thread");
    // this wavefront's counters and its first rows are on their way while the tables are made
    const int c = (int)blockIdx.x * kWaves4 + w;
    const int64_t r_end = c < a.n_shares ? min(a.rows, (int64_t)(c + 1) * a.share) : 0;
    constexpr int kCounters = (kBins + 63) / 64;
    int before[kCounters], deg[4];
#pragma unroll
    for (int j = 0; j < kCounters; j++)
        before[j] = c < a.n_shares && j * 64 + lane < kBins ? a.bins[(int64_t)(j * 64 + lane) * a.pitch + c] : 0;
    auto load_rows = [&](int64_t r1) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t r = r1 + j * 64 + lane;
            deg[j] = r < r_end ? a.indptr[r + 1] - a.indptr[r] : 0;
        }
    };
    load_rows((int64_t)c * a.share);
    {
        int cnt[2], nz[2], blk[2], t;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int d = 2 * tid + j;
            cnt[j] = d < kBins ? a.bin_total[d] : 0;
            nz[j] = blk[j] = 0;
            if (d > 0 && d <= kDegBound) {
                int wn, rpb;
                slice_rule(d, wn, rpb);
                nz[j] = d * cnt[j];
                blk[j] = (cnt[j] + rpb - 1) / rpb;
            }
        }
        const int r0 = block_exclusive_sum<kThreads>(cnt[0] + cnt[1], lds, t);
        const int z0 = block_exclusive_sum<kThreads>(nz[0] + nz[1], lds, t);
        const int b0 = block_exclusive_sum<kThreads>(blk[0] + blk[1], lds, t);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int d = 2 * tid + j;
            if (d < kBins) {
                run_row[d] = r0 + (j ? cnt[0] : 0);
                run_nz[d] = z0 + (j ? nz[0] : 0);
                run_blk[d] = b0 + (j ? blk[0] : 0);
            }
            if (d == kBins - 1) run_row[kBins] = (int)a.rows;
        }
        __syncthreads();
    }
    if (blockIdx.x == 0) {
        for (int i = tid; i <= kBins; i += kThreads) a.run_row[i] = run_row[i];
        for (int i = tid; i < kBins; i += kThreads) a.run_nz[i] = run_nz[i];
    }
    const int64_t all = (int64_t)gridDim.x * kThreads, me = (int64_t)blockIdx.x * kThreads + tid;
    for (int64_t i = me; i < a.n_zero; i += all) a.zero[i] = 0;

    // sorted row pointers and block4 entries of the rows of up to 384 non-zeros, by sorted row
    const int n_binned = run_row[kLongBin];
    // (rows of a thread searched for together, in steps that are selections: one at a time with branches, 3.6 us here)
    constexpr int kAtOnce = 4;
    for (int64_t p0 = me; p0 < n_binned; p0 += kAtOnce * all) {
        int bin[kAtOnce];
#pragma unroll
        for (int k = 0; k < kAtOnce; k++) bin[k] = 0;
#pragma unroll
        for (int step = 256; step > 0; step >>= 1)            // the last bin that starts at or before the row
#pragma unroll
            for (int k = 0; k < kAtOnce; k++) {
                const bool on = run_row[min(bin[k] + step, kLongBin)] <= p0 + k * all;
                bin[k] += (on & (bin[k] + step < kLongBin)) ? step : 0;
            }
#pragma unroll
        for (int k = 0; k < kAtOnce; k++) {
            const int64_t p = p0 + k * all;
            if (p >= n_binned) break;
            const int d = bin[k], i = (int)p - run_row[d], loc = run_nz[d] + i * d;
            a.s_indptr[p] = loc;
            if (d > 0) {
                int wn, rpb;
                slice_rule(d, wn, rpb);
                if (i % rpb == 0)
                    a.block4[run_blk[d] + i / rpb] =
                        make_int4(d, (int)p, loc, (wn << 16) + min(rpb, run_row[d + 1] - run_row[d] - i));
            }
        }
    }
    if (me == 0) a.s_indptr[a.rows] = a.indptr[a.rows];

    // the rows of this wavefront's share
    if (c >= a.n_shares) return;
#pragma unroll
    for (int j = 0; j < kCounters; j++)
        if (j * 64 + lane < kBins) next[w][j * 64 + lane] = run_row[j * 64 + lane] + before[j];
    __builtin_amdgcn_wave_barrier();
    int n_units = 0, cost = 0, n_heavy = 0, n_rows8 = 0;
    for (int64_t r1 = (int64_t)c * a.share; r1 < r_end; r1 += 4 * 64) {
        int d4[4];
#pragma unroll
        for (int j = 0; j < 4; j++) d4[j] = deg[j];
        load_rows(r1 + 4 * 64);                                // the next four rounds' rows
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t r = r1 + j * 64 + lane;
            const bool ok = r < r_end;
            const int d = d4[j];
            const int bin = min(d, kLongBin);
            const unsigned long long peers = wave_match<9>(bin, ok);
            const int rank = lanes_below(peers, lane);
            const int p = next[w][bin] + rank;
            __builtin_amdgcn_wave_barrier();
            if (ok && rank == 0) next[w][bin] = p + __popcll(peers);
            __builtin_amdgcn_wave_barrier();
            if (ok) {
                if (d > kDegBound) {
                    a.long_deg[p - n_binned] = d;
                    a.long_row[p - n_binned] = (uint32_t)r;
                } else {
                    if (a.perm) a.perm[p] = (int32_t)r;
                    a.place[r] = (uint32_t)p;
                }
                if (d > 0 && d <= a.rule.split) {
                    const int n = unit_rows(d, p - run_row[d], run_row[d + 1] - run_row[d], a.rule);
                    if (n > 0) {
                        n_units++;
                        cost += unit_cost(d * n, n, a.rule.cost_shift);
                        n_heavy += d * n > a.rule.light_nz;
                    }
                }
                if (d > a.rule.split) n_rows8 += row_groups(d, a.rule.groups) == kXcds;
            }
        }
    }
    n_units = wave_sum(n_units);
    cost = wave_sum(cost);
    n_heavy = wave_sum(n_heavy);
    n_rows8 = wave_sum(n_rows8);
    if (lane == 0) {
        const int pitch = a.pitch + kWaves4;
        a.sums[kSumUnits * pitch + c] = n_units;
        a.sums[kSumCost * pitch + c] = cost;
        a.sums[kSumHeavy * pitch + c] = n_heavy;
        a.sums[kSumRows8 * pitch + c] = n_rows8;
    }
}

// ---------------------------------------------------------------------------
// Rows of more than 384 non-zeros, by (degree, row).  Up to kFewLong of them: each is compared with all
// (place_long_kernel), and the non-zeros, blocks and chunks of the rows before it are added up on the way, which is all
// there is to know.  More go through a stable radix sort, 8 bits a pass; their scan and their blocks are launches of their own.
// Comparing costs the square: 19 us on 4,850 rows and 25 on 6,400, where comparing for the rank alone, with the launches for
// the scans and blocks behind it, took 29 and 34 and the gaps between them; on 8,192 it would be 41, as much as the six
// launches behind the sort take on 13,000 (39).
// ---------------------------------------------------------------------------
constexpr int kFewLong = 8192;

__host__ __device__ inline int blocks_of(int d) { return (d + kDegBound - 1) / kDegBound; }
__host__ __device__ inline int chunks_of(int d) { return d > kWideRow ? (d + kWideChunk - 1) / kWideChunk : 0; }

struct LongArgs {
    const int *deg;                           // in the caller's order
    const uint32_t *row;
    int n;
    int64_t first_long;                       // sorted row of the first
    int nz0, block0;                          // non-zeros and blocks before them
    int32_t *perm;                            // null: in order already
    uint32_t *place;
    int32_t *s_indptr;
    int4 *block4;
    int *first_chunk, *chunk_row;             // of long row i (null: none is wide)
};

// Up to kFewLong long rows, completely: places, row pointers, blocks and chunks.  kRankRows rows per workgroup, few so that
// even some hundred rows are work for much of the chip, and selections instead of branches (5.5 us on 1,760 rows, where 64
// rows a workgroup and a branch per row took 17): a lane compares one of them with every 64th of all rows.  The first kSums workgroups scan the counts per share.
constexpr int kRankRows = 16, kRankTile = 2048;
__global__ __launch_bounds__(1024) void place_long_kernel(LongArgs a, int *__restrict__ sums, int sum_pitch, int n_shares)
{
    __shared__ int4 tile[kRankTile];                     // degree, blocks, chunks
    __shared__ int4 part[16][kRankRows], mine[kRankRows];
    __shared__ int deg[kRankRows];
    int b = blockIdx.x;
    if (b < kSums) { scan_shares<1024>(sums + (int64_t)b * sum_pitch, n_shares, &tile[0].x); return; }
    b -= kSums;
    const int lane = threadIdx.x & 63, seg = threadIdx.x >> 6, j = b * kRankRows + lane % kRankRows;
    const int d = j < a.n ? a.deg[j] : 0;
    const uint32_t r = j < a.n ? a.row[j] : 0;
    int below = 0, nz = 0, blk = 0, chk = 0;
    for (int t0 = 0; t0 < a.n; t0 += kRankTile) {
        constexpr int kStep = 1024 / kRankRows, kUnroll = 4;
        const int here = (min(kRankTile, a.n - t0) + kStep * kUnroll - 1) / (kStep * kUnroll) * (kStep * kUnroll);
        if (t0 > 0) __syncthreads();
        for (int i = threadIdx.x; i < here; i += 1024) {
            const int e = t0 + i < a.n ? a.deg[t0 + i] : INT_MAX;
            tile[i] = make_int4(e, blocks_of(e), chunks_of(e), 0);
        }
        __syncthreads();
        for (int i0 = 0; i0 < here; i0 += kStep * kUnroll) {
#pragma unroll
            for (int k = 0; k < kUnroll; k++) {
                const int i = i0 + k * kStep + seg * (64 / kRankRows) + lane / kRankRows;
                const int4 e = tile[i];
                // (equal degrees rank by row, which is the order they are listed in)
                const int take = -(int)(e.x < d + (t0 + i < j));
                below -= take;
                nz += e.x & take;
                blk += e.y & take;
                chk += e.z & take;
            }
        }
    }
#pragma unroll
    for (int o = kRankRows; o < 64; o *= 2) {
        below += __shfl_xor(below, o);
        nz += __shfl_xor(nz, o);
        blk += __shfl_xor(blk, o);
        chk += __shfl_xor(chk, o);
    }
    if (lane < kRankRows) part[seg][lane] = make_int4(below, nz, blk, chk);
    __syncthreads();
    if (seg == 0 && lane < kRankRows && j < a.n) {
        below = nz = blk = chk = 0;
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int4 v = part[q][lane];
            below += v.x;
            nz += v.y;
            blk += v.z;
            chk += v.w;
        }
        const int64_t p = a.first_long + below;
        if (a.perm) a.perm[p] = (int32_t)r;
        a.place[r] = (uint32_t)p;
        a.s_indptr[p] = a.nz0 + nz;
        if (a.first_chunk) {
            a.first_chunk[below] = chk;
            if (below == a.n - 1) a.first_chunk[a.n] = chk + chunks_of(d);
        }
        deg[lane] = d;
        mine[lane] = make_int4(below, a.nz0 + nz, a.block0 + blk, chk);
    }
    __syncthreads();
    static_assert(kRankRows == 16, "a row per wavefront");
    if (b * kRankRows + seg >= a.n) return;
    const int di = deg[seg];
    const int4 m = mine[seg];
    for (int k = lane; k < blocks_of(di); k += 64)
        a.block4[m.z + k] = make_int4(di, (int)a.first_long + m.x, m.y + k * kDegBound, min(kDegBound, di - k * kDegBound));
    if (a.first_chunk)
        for (int k = lane; k < chunks_of(di); k += 64) a.chunk_row[m.w + k] = m.x;
}

constexpr int kItems = 8;
constexpr int kTile = kThreads * kItems;      // elements per workgroup in the sort's passes and the scans

// Digits of the tile's keys.  hist: [tile][digit] for kSelfScan tiles and fewer, which the scatter adds up itself, else
// [digit][tile], scanned by small_scan_kernel.  The workgroups behind the tiles (first pass only) scan one kind each of the
// counts per share (sums), which has nothing to do with the rest but that both come behind place_rows.
constexpr int64_t kSelfScan = 64;
__global__ __launch_bounds__(kThreads) void radix_hist(const uint32_t *__restrict__ keys,
                                                       int64_t n, int shift,
                                                       int *__restrict__ hist, int64_t tiles,
                                                       int *__restrict__ sums, int sum_pitch, int n_shares)
{
    __shared__ int h[256];
    if ((int64_t)blockIdx.x >= tiles) {
        scan_shares<kThreads>(sums + (blockIdx.x - tiles) * sum_pitch, n_shares, h);
        return;
    }
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kTile;
#pragma unroll
    for (int j = 0; j < kItems; j++) {
        const int64_t i = base + j * kThreads + threadIdx.x;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & 255u], 1);
    }
    __syncthreads();
    hist[tiles <= kSelfScan ? (int64_t)blockIdx.x * 256 + threadIdx.x : (int64_t)threadIdx.x * tiles + blockIdx.x] =
        h[threadIdx.x];
}

// What the last pass writes instead of keys and their order: the long rows' places and sizes.
struct LongSorted {
    const uint32_t *row;                      // of the unsorted long rows (null: not the last pass)
    int64_t first_long;
    int32_t *perm;                            // null: in order already
    uint32_t *place;
    int *deg, *blocks, *chunks;               // in sorted order; chunks null: no row is wide
};

// A wavefront takes 512 keys in a row and ranks them without a barrier; then the tile's digits are placed.  With the counts
// added up here and the last pass writing what two more kernels made of its order, the sort is four launches and not nine:
// 20 M non-zeros with 13,000 long rows 397 -> 387 us from the graph to its first product, 60 M with 51,000 1028 -> 1011.
// (A workgroup reads all tiles' counts: 64 KB of them at kSelfScan tiles.)
__global__ __launch_bounds__(kThreads) void radix_scatter(
    const uint32_t *__restrict__ keys_in, const uint32_t *__restrict__ vals_in,
    uint32_t *__restrict__ keys_out, uint32_t *__restrict__ vals_out, int64_t n, int shift,
    const int *__restrict__ hist, int64_t tiles, LongSorted out)
{
    __shared__ int cnt[kWaves4][256], lds[kWaves4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, digit = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * kTile + w * (kTile / kWaves4) + lane;
    uint32_t key[kItems], val[kItems];
    int where[kItems];
#pragma unroll
    for (int j = 0; j < kItems; j++) {
        const int64_t i = first + j * 64;
        key[j] = i < n ? keys_in[i] : 0u;
        val[j] = i < n && vals_in ? vals_in[i] : (uint32_t)i;
    }
    int at = 0;                                // where this tile's keys of the thread's digit go
    if (tiles <= kSelfScan) {
        int all = 0, before = 0;
#pragma unroll 8
        for (int t = 0; t < (int)tiles; t++) {
            const int c = hist[t * 256 + digit];
            all += c;
            before += t < (int)blockIdx.x ? c : 0;
        }
        int total;
        at = block_exclusive_sum<kThreads>(all, lds, total) + before;
    } else {
        at = hist[(int64_t)digit * tiles + blockIdx.x];
    }
#pragma unroll
    for (int j = 0; j < 4; j++) cnt[w][j * 64 + lane] = 0;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < kItems; j++) {
        const bool valid = first + j * 64 < n;
        const int dg = (key[j] >> shift) & 255u;
        const unsigned long long peers = wave_match<8>(dg, valid);
        const int rank = lanes_below(peers, lane);
        where[j] = cnt[w][dg] + rank;
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) cnt[w][dg] = where[j] + __popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kWaves4; q++) {
        const int c = cnt[q][digit];
        cnt[q][digit] = at;
        at += c;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; j++) {
        if (first + j * 64 >= n) continue;
        const int pos = where[j] + cnt[w][(key[j] >> shift) & 255u];
        if (!out.row) {
            keys_out[pos] = key[j];
            vals_out[pos] = val[j];
            continue;
        }
        const uint32_t r = out.row[val[j]];
        const int d = (int)key[j];
        if (out.perm) out.perm[out.first_long + pos] = (int32_t)r;
        out.place[r] = (uint32_t)(out.first_long + pos);
        out.deg[pos] = d;
        out.blocks[pos] = blocks_of(d);
        if (out.chunks) out.chunks[pos] = chunks_of(d);
    }
}

// Exclusive scan of n ints in place by one workgroup (the radix sort's counts).
__global__ __launch_bounds__(1024) void small_scan_kernel(int *__restrict__ v, int64_t n)
{
    __shared__ int lds[16];
    int carry = 0;
    for (int64_t b = 0; b < n; b += 1024 * kItems) {
        const int64_t at = b + (int64_t)threadIdx.x * kItems;
        int x[kItems], acc = 0;
#pragma unroll
        for (int j = 0; j < kItems; j++) {
            x[j] = at + j < n ? v[at + j] : 0;
            acc += x[j];
        }
        int total, run = block_exclusive_sum<1024>(acc, lds, total);
        run += carry;
#pragma unroll
        for (int j = 0; j < kItems; j++) {
            if (at + j < n) v[at + j] = run;
            run += x[j];
        }
        carry += total;
    }
}

// Sorts many long rows (their places, and degrees, blocks and chunks in sorted order), and scans the counts per share.
int sort_long_rows(Arena *tmp, const int *deg, int n, int max_degree, const LongSorted &sorted, int *sums, int pitch,
                   int n_shares, hipStream_t s)
{
    uint32_t *keys[2], *vals[2];
    int *hist, rc;
    const int64_t tiles = ((int64_t)n + kTile - 1) / kTile;
    for (int i = 0; i < 2; i++) {
        if ((rc = tmp->alloc(&keys[i], (size_t)n))) return rc;
        if ((rc = tmp->alloc(&vals[i], (size_t)n))) return rc;
    }
    if ((rc = tmp->alloc(&hist, (size_t)(256 * tiles)))) return rc;
    const uint32_t *kin = reinterpret_cast<const uint32_t *>(deg), *vin = nullptr;
    for (int shift = 0, to = 0; shift < 32 && (max_degree >> shift) != 0; shift += 8, to ^= 1) {
        const bool last = shift == 24 || (max_degree >> (shift + 8)) == 0;
        radix_hist<<<dim3((unsigned)tiles + (shift == 0 ? kSums : 0)), dim3(kThreads), 0, s>>>(kin, n, shift, hist, tiles, sums,
                                                                                              pitch, n_shares);
        if (tiles > kSelfScan) small_scan_kernel<<<dim3(1), dim3(1024), 0, s>>>(hist, 256 * tiles);
        radix_scatter<<<dim3((unsigned)tiles), dim3(kThreads), 0, s>>>(kin, vin, keys[to], vals[to], n, shift, hist,
                                                                     tiles, last ? sorted : LongSorted{});
        kin = keys[to];
        vin = vals[to];
    }
    return ACCEL_OK;
}

// One wavefront per long row: its block4 entries, and the row of each of its chunks.
__global__ __launch_bounds__(kThreads) void long_blocks_kernel(LongArgs a, const int *__restrict__ sorted_deg,
                                                               const int32_t *__restrict__ loc_of,
                                                               const int *__restrict__ first_block)
{
    const int lane = threadIdx.x & 63, i = (int)blockIdx.x * kWaves4 + (threadIdx.x >> 6);
    if (i >= a.n) return;
    const int d = sorted_deg[i], row = (int)(a.first_long + i), loc = loc_of[row], at = first_block[i];
    for (int k = lane; k < blocks_of(d); k += 64)
        a.block4[at + k] = make_int4(d, row, loc + k * kDegBound, min(kDegBound, d - k * kDegBound));
    if (a.first_chunk && chunks_of(d) > 0) {
        const int c0 = a.first_chunk[i];
        for (int k = lane; k < chunks_of(d); k += 64) a.chunk_row[c0 + k] = i;
    }
}

// Ints that must be zero for place_long_rows (place_rows clears them).
int64_t long_zeroed_ints(int64_t n) { return n > kFewLong ? 3 * scan_zeroed(n) : 0; }

// The long rows' places, row pointers, blocks and chunks, and the scan of the counts per share of rows (sums).
int place_long_rows(Arena *tmp, const LongArgs &a, int max_degree, const int32_t *loc_of, int *zeroed,
                    int *sums, int pitch, int n_shares, hipStream_t s)
{
    int rc, *sorted_deg, *blocks, *chunks = nullptr;
    if (a.n <= kFewLong) {
        const unsigned groups = kSums + (unsigned)((a.n + kRankRows - 1) / kRankRows);
        place_long_kernel<<<dim3(groups), dim3(1024), 0, s>>>(a, sums, pitch, n_shares);
        return ACCEL_OK;
    }
    if ((rc = tmp->alloc(&sorted_deg, (size_t)a.n))) return rc;
    if ((rc = tmp->alloc(&blocks, (size_t)a.n + 1))) return rc;
    if (a.first_chunk && (rc = tmp->alloc(&chunks, (size_t)a.n))) return rc;
    const LongSorted sorted{a.row, a.first_long, a.perm, a.place, sorted_deg, blocks, chunks};
    if ((rc = sort_long_rows(tmp, a.deg, a.n, max_degree, sorted, sums, pitch, n_shares, s))) return rc;
    ScanJobs jobs{};
    int n_jobs = 0;
    auto add = [&](const int *in, int *out, int first) {
        jobs.job[n_jobs] = {in, out, a.n, first, zeroed + n_jobs * scan_zeroed(a.n)};
        n_jobs++;
    };
    add(blocks, blocks, a.block0);
    add(sorted_deg, a.s_indptr + a.first_long, a.nz0);
    if (chunks) add(chunks, a.first_chunk, 0);
    launch_scans(jobs, n_jobs, s);
    long_blocks_kernel<<<dim3(grid_for((int64_t)a.n * 64)), dim3(kThreads), 0, s>>>(a, sorted_deg, loc_of, blocks);
    return ACCEL_OK;
}

// ---------------------------------------------------------------------------
// Sorted copy of the non-zeros: the columns (idx_out, may be null) and a payload, which is the
// value of the non-zero or, when src_pos is set, its position in the caller's arrays (what a later
// value update gathers through).  Columns outside
// [0, cols) are reported to the host: every non-zero passes through here exactly once.
// ---------------------------------------------------------------------------
struct CopyArgs {
    SortedRows sr;
    const int32_t *idx;
    const float *val;
    uint32_t cols;
    int32_t *idx_out;
    int32_t *pay_out;
    int src_pos;                              // payload: positions instead of values
    Mail *mail;                               // where a bad column is reported (null: checked before)
};
__device__ __forceinline__ int payload(const CopyArgs &a, int64_t src)
{
    return a.src_pos ? (int)src : __float_as_int(a.val[src]);
}
__device__ __forceinline__ void report_bad(const CopyArgs &a, bool bad)
{
    if (a.mail && __ballot(bad) && (threadIdx.x & 63) == 0) a.mail->bad_index = 1;
}

// Rows that stay whole (up to 384 non-zeros): a workgroup copies a tile, up to kPermuteTile consecutive non-zeros of one
// run of equal degree in the sorted matrix, so that the row of a non-zero is a multiplication away; the rows'
// source offsets are put in LDS.  Bound by the lines that row segments of some hundred bytes at arbitrary addresses touch,
// twice their bytes and, for the offsets, a line per row: unless rows that are neighbours in the caller's
// matrix, which share those lines, are copied by the same die at about the same time.  So tiles go by bands of the caller's
// rows.  A run's rows are in the caller's order: tile i of its n tiles comes from about the i-th n-th of the matrix, and
// belongs to about band i B / n of B (shifted by less than a tile, each run differently, so that runs of one tile do not all
// end in the last band).  A die takes an eighth of the bands, one after the other, all runs' tiles of a band together.
// In sorted order, several runs to a tile, found by search: 16 M non-zeros 361 MB read in 80.5 us, so 183 MB in 71 (whole
// launch); 125 M 1.79 GB and 457 us, 1.28 GB and 430; 2.45 M 17.5 and 14.6 us, 60 k 8.8 and 6.0.  Tiles of 1,024
// and of 4,096: 77 and 79 us on the 16 M, 469 and 436 on the 125 M.
constexpr int kPermuteNz = 8;                        // non-zeros per thread
constexpr int kPermuteTile = kThreads * kPermuteNz;  // non-zeros per workgroup
__host__ __device__ inline int tiles_of_run(int nz) { return nz / kPermuteTile + (nz % kPermuteTile > 0); }

// Tiles of the run of degree d, n in all, that the bands before `band` hold.
__host__ __device__ inline int tiles_before(int band, int n, int d, int log2_bands)
{
    const int shift = d * 159 & ((1 << log2_bands) - 1);
    return (band * n + shift) >> log2_bands;                                    // below 2^29
}

static TileOrder order_tiles(const int *hist, int most)
{
    TileOrder t;
    int64_t all = 0;
    for (int d = 1; d <= most; d++) all += tiles_of_run(hist[d] * d);
    while ((2 << t.log2_bands) <= kMaxBands && all >> (t.log2_bands + 1) >= 64) t.log2_bands++;
    const int bands = 1 << t.log2_bands, per = bands / kXcds;
    for (int d = 1; d <= most; d++) {
        const int n = tiles_of_run(hist[d] * d);
        if (n == 0) continue;
        for (int b = 1; b <= bands; b++) t.first[b] += tiles_before(b, n, d, t.log2_bands);
    }
    for (int x = 0; x < kXcds; x++) t.per_die = std::max(t.per_die, t.first[(x + 1) * per] - t.first[x * per]);
    return t;
}

struct PermuteLds {
    int shift[kPermuteTile + 1];                     // source position minus sorted position, per row of the tile
};
// i: the number of the workgroup among those that copy tiles, i % 8 being its die's.
__device__ __forceinline__ void permute_rows(const CopyArgs &a, PermuteLds &l, const TileOrder &order, int i, int n_take)
{
    const int lane = threadIdx.x & 63;
    const int per = 1 << (order.log2_bands - 3), band0 = i % kXcds * per;
    const int t = order.first[band0] + i / kXcds;
    if (t >= order.first[band0 + per]) return;
    static_assert(kMaxBands / kXcds <= 64, "a lane per band of a die");
    const int band = band0 + __popcll(__ballot(lane < per && order.first[band0 + min(lane, per - 1)] <= t)) - 1;
    // which of the band's tiles: six degrees per lane
    constexpr int kEach = kDegBound / 64;
    int nz[kEach + 1], from[kEach], count[kEach], mine = 0;
#pragma unroll
    for (int k = 0; k <= kEach; k++) nz[k] = min(a.sr.run_nz[1 + lane * kEach + k], n_take);
#pragma unroll
    for (int k = 0; k < kEach; k++) {
        const int n = tiles_of_run(nz[k + 1] - nz[k]);
        const int degree = 1 + lane * kEach + k;
        from[k] = tiles_before(band, n, degree, order.log2_bands);
        count[k] = tiles_before(band + 1, n, degree, order.log2_bands) - from[k];
        mine += count[k];
    }
    int j = t - order.first[band] - wave_exclusive_sum(mine);
    const int owner = 63 - __clzll((long long)__ballot(j >= 0));        // (behind it the sums are larger)
    int d = 0, at = 0, end = 0, run0 = 0;
#pragma unroll
    for (int k = 0; k < kEach; k++) {
        if (j >= 0 && j < count[k]) {
            d = 1 + lane * kEach + k;
            run0 = nz[k];
            at = run0 + (from[k] + j) * kPermuteTile;
            end = nz[k + 1];
        }
        j -= count[k];
    }
    d = __builtin_amdgcn_readlane(d, owner);
    run0 = __builtin_amdgcn_readlane(run0, owner);
    const int p0 = __builtin_amdgcn_readlane(at, owner), n = min(kPermuteTile, __builtin_amdgcn_readlane(end, owner) - p0);
    const int run_row = a.sr.run_row[d];
    const int first = (p0 - run0) / d, start0 = run0 + first * d, row0 = run_row + first;
    const int n_here = (p0 + n - 1 - run0) / d - first + 1;      // at most kPermuteTile: every row holds a non-zero of the tile
    constexpr int kRows = 4;                         // rows of a thread under way at once
    for (int j0 = threadIdx.x; j0 < n_here; j0 += kRows * kThreads) {
        int src[kRows];
#pragma unroll
        for (int k = 0; k < kRows; k++) {
            const int row = row0 + min(j0 + k * kThreads, n_here - 1);
            src[k] = a.sr.perm ? a.sr.perm[row] : row;
        }
#pragma unroll
        for (int k = 0; k < kRows; k++) src[k] = a.sr.indptr[src[k]];
#pragma unroll
        for (int k = 0; k < kRows; k++)
            if (j0 + k * kThreads < n_here) l.shift[j0 + k * kThreads] = src[k] - (start0 + (j0 + k * kThreads) * d);
    }
    __syncthreads();
    const float inv = 1.0f / (float)d;
    int src[kPermuteNz], col[kPermuteNz], pay[kPermuteNz];
    bool bad = false;
#pragma unroll
    for (int q = 0; q < kPermuteNz; q++) {
        const int p = p0 + min(q * kThreads + (int)threadIdx.x, n - 1);
        src[q] = p + l.shift[(int)(((float)(p - start0) + 0.5f) * inv)];       // exact: p - start0 < 2,432
    }
#pragma unroll
    for (int q = 0; q < kPermuteNz; q++) {
        col[q] = a.idx[src[q]];
        pay[q] = payload(a, src[q]);
    }
#pragma unroll
    for (int q = 0; q < kPermuteNz; q++) {
        const int p = q * kThreads + (int)threadIdx.x;
        bad |= (uint32_t)col[q] >= a.cols;
        if (p >= n) continue;
        if (a.idx_out) a.idx_out[p0 + p] = col[q];
        a.pay_out[p0 + p] = pay[q];
    }
    report_bad(a, bad);
}

// Split rows: the row's non-zeros are written grouped by col_group(column, row_groups(degree)),
// stably inside each group, so that a work unit of such a row touches rows of X that belong to one
// column group.  counts[lr * 64 + g] receives the size of each group (counts may be null).
// Rows of up to R * 64 non-zeros: a wavefront per row.  The whole row is loaded at once, put in
// order in LDS, the columns first and then the payload, and written out in one piece per array.  Bound by memory as
// long as enough of them are under way: columns and payload together in LDS (33 KB a workgroup instead of 17) let four
// workgroups on a compute unit instead of seven, the tiles of whole rows in the same launch among them.  With that, with
// the ranks kept in registers instead of groups counted by atomics first, and with rows of one chunk placed here
// (place_chunk), the copying of 125 M non-zeros of a power-law matrix took 548 us where it had taken 683, that of 30 M with hub
// rows 155 where it had taken 202 (with wide_place_kernel; 513 and 142 since whole rows go by bands).
template <int R> struct GroupLds {
    int buf[kWaves4][R * 64];
    int cnt[kWaves4][kMaxGroups];
};
// Non-zeros e0, e0 + 64, ... of the n at src, the last one again behind the end: their columns, their payloads.
template <int R>
__device__ __forceinline__ void load_columns(const CopyArgs &a, int src, int n, int e0, int (&col)[R])
{
    const int32_t *idx = a.idx + src;
#pragma unroll
    for (int j = 0; j < R; j++) col[j] = idx[min(e0 + j * 64, n - 1)];
}
template <int R>
__device__ __forceinline__ void load_payloads(const CopyArgs &a, int src, int n, int e0, int (&pay)[R])
{
    if (a.src_pos) {
#pragma unroll
        for (int j = 0; j < R; j++) pay[j] = src + e0 + j * 64;
    } else {
        const float *val = a.val + src;
        asm("" : "+v"(e0));                              // (or the positions of the columns are kept in registers for this)
#pragma unroll
        for (int j = 0; j < R; j++) pay[j] = __float_as_int(val[min(e0 + j * 64, n - 1)]);
    }
}
// The place of this lane's non-zero among those of its group that the wavefront has met, R rounds in a row.
// cnt (64 ints of this wavefront, cleared): the sizes of the groups on return.
constexpr int kGroupBits = 6;
static_assert(kMaxGroups == 1 << kGroupBits, "a group's number");
template <int R>
__device__ __forceinline__ void rank_in_groups(const int (&col)[R], int n, int ng, int *cnt, int (&where)[R])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < R; j++) {
        if (j * 64 >= n) break;                          // uniform
        const bool valid = lane < n - j * 64;
        const int g = col_group(col[j], ng);
        const unsigned long long peers = wave_match<kGroupBits>(g, valid);
        const int rank = lanes_below(peers, lane);
        where[j] = cnt[g] + rank;
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) cnt[g] = where[j] + __popcll(peers);     // one lane per group present
        __builtin_amdgcn_wave_barrier();
    }
}
template <int R>
__device__ __forceinline__ void group_row(const CopyArgs &a, GroupLds<R> &l, int64_t r, int lr, int forced_groups,
                                          int *__restrict__ counts)
{
    static_assert(kMaxGroups == 64, "one lane per column group");
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int src0 = __builtin_amdgcn_readfirstlane(a.sr.indptr[a.sr.perm ? a.sr.perm[r] : r]);
    const int dst0 = __builtin_amdgcn_readfirstlane(a.sr.s_indptr[r]);
    const int d = __builtin_amdgcn_readfirstlane(a.sr.s_indptr[r + 1]) - dst0;
    const int ng = row_groups(d, forced_groups);
    int *my = l.cnt[w], *st = l.buf[w];
    my[lane] = 0;
    __builtin_amdgcn_wave_barrier();
    int col[R], where[R];
    bool bad = false;
    load_columns<R>(a, src0, d, lane, col);
    rank_in_groups<R>(col, d, ng, my, where);
    const int c = my[lane];                              // lane g holds the size of group g
    if (counts) counts[(int64_t)lr * kMaxGroups + lane] = c;
    const int start = wave_exclusive_sum(c);
    __builtin_amdgcn_wave_barrier();
    my[lane] = start;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < R; j++) {
        if (lane < d - j * 64) {
            bad |= (uint32_t)col[j] >= a.cols;
            where[j] += my[col_group(col[j], ng)];
            st[where[j]] = col[j];
        }
    }
    report_bad(a, bad);
    int pay[R];
    load_payloads<R>(a, src0, d, lane, pay);
    __builtin_amdgcn_wave_barrier();
    if (a.idx_out) {
#pragma unroll
        for (int j = 0; j < R; j++)
            if (lane < d - j * 64) (a.idx_out + dst0 + j * 64)[lane] = st[j * 64 + lane];
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < R; j++)
        if (lane < d - j * 64) st[where[j]] = pay[j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < R; j++)
        if (lane < d - j * 64) (a.pay_out + dst0 + j * 64)[lane] = st[j * 64 + lane];
}

// Longer rows ("wide") in chunks of kWideChunk non-zeros, a workgroup per chunk, so that a row of
// 200,000 is 49 workgroups and not a chain of 200 rounds in one.  A row of one chunk is placed at once; of the
// others the chunks' groups are counted first.  chunk_row[c] = the long row of chunk c, first_chunk[i] = the
// first chunk of long row i.
struct WideArgs {
    const int *chunk_row, *first_chunk;
    int64_t first_long;                       // sorted row of the first long row
    int n_narrow;                             // long rows before the first wide one
    int forced_groups;
    int *chunk_count;                         // [chunks][64]: non-zeros of each group
};
struct WideChunk {
    int src, row;                             // in the caller's arrays; where the row starts in the sorted ones
    int n, ng;
    bool whole;                               // the row has no other chunk
};
__device__ __forceinline__ WideChunk wide_chunk(const CopyArgs &a, const WideArgs &wa, int c)
{
    const int i = __builtin_amdgcn_readfirstlane(wa.chunk_row[c]);
    const int64_t r = wa.first_long + i;
    const int from = __builtin_amdgcn_readfirstlane(a.sr.s_indptr[r]);
    const int d = __builtin_amdgcn_readfirstlane(a.sr.s_indptr[r + 1]) - from, off = (c - wa.first_chunk[i]) * kWideChunk;
    return {__builtin_amdgcn_readfirstlane(a.sr.indptr[a.sr.perm ? a.sr.perm[r] : r]) + off, from, min(kWideChunk, d - off),
            row_groups(d, wa.forced_groups), d <= kWideChunk};
}

__device__ __forceinline__ void wide_count(const CopyArgs &a, const WideChunk &ch, int *cnt, int *__restrict__ count)
{
    if ((int)threadIdx.x < kMaxGroups) cnt[threadIdx.x] = 0;
    __syncthreads();
    int col[kWideChunk / kThreads];
    bool bad = false;
#pragma unroll
    for (int j = 0; j < kWideChunk / kThreads; j++) {
        const int e = j * kThreads + (int)threadIdx.x;
        col[j] = e < ch.n ? a.idx[ch.src + e] : 0;
    }
#pragma unroll
    for (int j = 0; j < kWideChunk / kThreads; j++) {
        if (j * kThreads + (int)threadIdx.x < ch.n) {
            bad |= (uint32_t)col[j] >= a.cols;
            atomicAdd(&cnt[col_group(col[j], ch.ng)], 1);
        }
    }
    report_bad(a, bad);
    __syncthreads();
    if ((int)threadIdx.x < kMaxGroups) count[threadIdx.x] = cnt[threadIdx.x];
}

// A chunk's non-zeros to their places, by W wavefronts.  kWhole: the chunk is the row, whose groups are counted here
// (count); else sum says how many non-zeros of each group the row has and how many the chunks before this one, to be added
// up over the wavefronts.
template <int W> struct ChunkLds {
    int buf[kWideChunk];
    int at[W][kMaxGroups], off[kMaxGroups];
};
template <int W, bool kWhole>
__device__ __forceinline__ void place_chunk(const CopyArgs &a, ChunkLds<W> &l, const WideChunk &ch, int *__restrict__ count,
                                            int (*sum)[W][kMaxGroups])
{
    constexpr int R = kWideChunk / (W * 64);             // rounds of a wavefront at most: each takes as many
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int share = (ch.n + W * 64 - 1) / (W * 64) * 64, first = w * share, n = min(share, ch.n - first);
    l.at[w][lane] = 0;
    __builtin_amdgcn_wave_barrier();
    int col[R], where[R];
    load_columns<R>(a, ch.src, ch.n, first + lane, col);
    rank_in_groups<R>(col, n, ch.ng, l.at[w], where);
    __syncthreads();
    if (w == 0) {
        int v[W], total = 0;
#pragma unroll
        for (int q = 0; q < W; q++) { v[q] = l.at[q][lane]; total += v[q]; }
        int run = wave_exclusive_sum(total);             // where the chunk's group `lane` starts in LDS
        if constexpr (kWhole) {
            count[lane] = total;
        } else {
            int all = 0, before = 0;
#pragma unroll
            for (int q = 0; q < W; q++) {
                all += sum[0][q][lane];
                before += sum[1][q][lane];
            }
            l.off[lane] = (int)ch.row + wave_exclusive_sum(all) + before - run;
        }
#pragma unroll
        for (int q = 0; q < W; q++) { l.at[q][lane] = run; run += v[q]; }
    }
    __syncthreads();
    bool bad = false;
#pragma unroll
    for (int j = 0; j < R; j++) {
        if (lane < n - j * 64) {
            bad |= (uint32_t)col[j] >= a.cols;
            where[j] += l.at[w][col_group(col[j], ch.ng)];
            l.buf[where[j]] = col[j];
        }
    }
    if (kWhole) report_bad(a, bad);                      // (else reported by wide_count)
    int pay[R];
    load_payloads<R>(a, ch.src, ch.n, first + lane, pay);
    __syncthreads();
    int to[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
        const int e = j * W * 64 + (int)threadIdx.x;
        if (e < ch.n) {
            const int c = l.buf[e];
            to[j] = (kWhole ? (int)ch.row : l.off[col_group(c, ch.ng)]) + e;
            if (a.idx_out) a.idx_out[to[j]] = c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < R; j++)
        if (lane < n - j * 64) l.buf[where[j]] = pay[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < R; j++) {
        const int e = j * W * 64 + (int)threadIdx.x;
        if (e < ch.n) a.pay_out[to[j]] = l.buf[e];
    }
}

// The units of whole rows, for which everything is known when the rows are placed.
struct UnitsArgs {
    SortedRows sr;
    UnitRule rule;
    PlanUnits pu;
    int share, n_shares, pitch, first_split;
    int groups;                               // workgroups: a share of rows per wavefront
};
struct UnitsLds {
    int run_row[kBins + 1], run_nz[kBins];
};

// All of the above in one launch (on a small matrix each would take its few microseconds after the
// other): workgroups take, in this order, shares of rows whose units are listed, chunks of wide rows to place or count, split rows
// of up to 1,024 and of up to 384 non-zeros (four each), tiles of whole rows.  The units have nothing to do with the rest
// but that both come behind the placing of the rows; a launch of their own took 8 to 10 us.
constexpr int kSmallRounds = kDegBound / 64, kMidRounds = kWideRow / 64;
struct CopyPlan {
    int n_chunks, n_mid, n_small;             // chunks; split rows
    int mid_groups, small_groups;             // workgroups for the split rows
    int64_t first_mid, first_small;           // sorted rows
    int n_take;                               // non-zeros of whole rows
    int *counts;                              // [split row][64], or null
};
__global__ __launch_bounds__(kThreads) void copy_rows_kernel(CopyArgs a, WideArgs wa, CopyPlan cp, UnitsArgs u, TileOrder order)
{
    union Lds {
        UnitsLds units;
        PermuteLds permute;
        GroupLds<kMidRounds> mid;
        GroupLds<kSmallRounds> small;
        ChunkLds<kWaves4> chunk;
    };
    __shared__ __attribute__((aligned(16))) char raw[sizeof(Lds)];
    Lds &l = *reinterpret_cast<Lds *>(raw);
    int b = blockIdx.x;
    if (b < u.groups) {
        for (int i = threadIdx.x; i <= kBins; i += kThreads) l.units.run_row[i] = u.sr.run_row[i];
        for (int i = threadIdx.x; i < kBins; i += kThreads) l.units.run_nz[i] = u.sr.run_nz[i];
        __syncthreads();
        list_units(u.sr, u.rule, u.pu, u.share, u.n_shares, u.pitch, u.first_split, l.units.run_row, l.units.run_nz,
                   b * kWaves4 + (int)(threadIdx.x >> 6));
        return;
    }
    b -= u.groups;
    if (b < cp.n_chunks) {
        const WideChunk ch = wide_chunk(a, wa, b);
        int *const count = wa.chunk_count + (int64_t)b * kMaxGroups;
        if (ch.whole) place_chunk<kWaves4, true>(a, l.chunk, ch, count, nullptr);
        else wide_count(a, ch, l.chunk.off, count);
        return;
    }
    b -= cp.n_chunks;
    if (b < cp.mid_groups) {                  // a wavefront without a row leaves; no barriers inside
        const int i = b * kWaves4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (i < cp.n_mid) group_row<kMidRounds>(a, l.mid, cp.first_mid + i, cp.n_small + i, wa.forced_groups, cp.counts);
        return;
    }
    b -= cp.mid_groups;
    if (b < cp.small_groups) {
        const int i = b * kWaves4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (i < cp.n_small) group_row<kSmallRounds>(a, l.small, cp.first_small + i, i, wa.forced_groups, cp.counts);
        return;
    }
    permute_rows(a, l.permute, order, b - cp.small_groups, cp.n_take);
}

// Counts the split rows for the plan and, in the workgroups behind, places the chunks of wide rows, one each (both
// come behind the counts of the chunks and nothing else: as launches of their own, with another that added up the
// chunks' counts, they took 12 us more on 2.45 M non-zeros).
template <int kPlaceThreads>
__global__ __launch_bounds__(kPlaceThreads) void wide_place_kernel(CopyArgs a, WideArgs wa, int first, SplitArgs split)
{
    constexpr int kWaves = kPlaceThreads / 64;
    __shared__ ChunkLds<kWaves> l;
    __shared__ int sum[2][kWaves][kMaxGroups];
    if ((int)blockIdx.x < split.n_groups) {
        count_split_rows<kPlaceThreads>(split, (int)blockIdx.x, reinterpret_cast<int (*)[kXcds]>(&sum[0][0][0]));
        return;
    }
    const int chunk = first + (int)blockIdx.x - split.n_groups;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    // the row's non-zeros of each group, and those of the chunks before this one
    const int i = wa.chunk_row[chunk], c0 = wa.first_chunk[i], c1 = wa.first_chunk[i + 1];
    int all = 0, before = 0;
#pragma unroll 4
    for (int c = c0 + w; c < c1; c += kWaves) {
        const int v = wa.chunk_count[(int64_t)c * kMaxGroups + lane];
        all += v;
        before += c < chunk ? v : 0;
    }
    sum[0][w][lane] = all;
    sum[1][w][lane] = before;
    place_chunk<kWaves, false>(a, l, wide_chunk(a, wa, chunk), nullptr, sum);
}

// Columns of a matrix whose arrays are used in place (sorted, no split row).
__global__ __launch_bounds__(kThreads) void index_check_kernel(const int32_t *__restrict__ idx,
                                                               int64_t nnz, int64_t cols,
                                                               Mail *__restrict__ mail)
{
    // 16-byte loads over the aligned middle of the array, single words at its two ends
    int bad = 0;
    auto look = [&](int c) { bad |= (c < 0) | ((int64_t)c >= cols); };
    const int64_t tid = (int64_t)blockIdx.x * kThreads + threadIdx.x, step = (int64_t)gridDim.x * kThreads;
    int64_t head = (int64_t)((16 - (reinterpret_cast<uintptr_t>(idx) & 15)) & 15) / 4;
    if (head > nnz) head = nnz;
    const int64_t n4 = (nnz - head) / 4;
    const int4 *v = reinterpret_cast<const int4 *>(idx + head);
    for (int64_t i = tid; i < n4; i += step) {
        const int4 c = v[i];
        look(c.x); look(c.y); look(c.z); look(c.w);
    }
    for (int64_t p = tid; p < head; p += step) look(idx[p]);
    for (int64_t p = head + 4 * n4 + tid; p < nnz; p += step) look(idx[p]);
    if (__ballot(bad) && (threadIdx.x & 63) == 0) mail->bad_index = 1;
}


// ---------------------------------------------------------------------------
// Partition of rows in any order (the walk is defined there too): scans over the rows.
// ---------------------------------------------------------------------------
struct SumOp {
    static constexpr int identity = 0;
    __device__ int operator()(int a, int b) const { return a + b; }
};
struct MaxOp {
    static constexpr int identity = INT_MIN;
    __device__ int operator()(int a, int b) const { return a > b ? a : b; }
};

// Exclusive scan of one value per thread over a 256-thread workgroup.
template <class Op>
__device__ int block_exclusive_scan(int v, Op op, int *wave_tot /* LDS, 4 ints */, int &total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int inc = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(inc, off);
        if (lane >= off) inc = op(t, inc);
    }
    if (lane == 63) wave_tot[w] = inc;
    __syncthreads();
    int prefix = Op::identity, tot = Op::identity;
#pragma unroll
    for (int i = 0; i < kThreads / 64; i++) {
        const int t = wave_tot[i];
        if (i < w) prefix = op(prefix, t);
        tot = op(tot, t);
    }
    __syncthreads();
    int exc = __shfl_up(inc, 1);
    if (lane == 0) exc = Op::identity;
    total = tot;
    return op(prefix, exc);
}

template <class Op>
__global__ __launch_bounds__(kThreads) void scan_reduce(const int *__restrict__ in, int64_t n,
                                                        int *__restrict__ sums)
{
    __shared__ int wave_tot[kThreads / 64];
    Op op;
    const int64_t base = (int64_t)blockIdx.x * kTile + (int64_t)threadIdx.x * kItems;
    int acc = Op::identity;
#pragma unroll
    for (int j = 0; j < kItems; j++)
        if (base + j < n) acc = op(acc, in[base + j]);
    int total;
    block_exclusive_scan(acc, op, wave_tot, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// One workgroup turns sums[0..nb) into their exclusive scan and stores the grand
// total at sums[nb].
template <class Op>
__global__ __launch_bounds__(kThreads) void scan_spine(int *__restrict__ sums, int64_t nb)
{
    __shared__ int wave_tot[kThreads / 64];
    Op op;
    int carry = Op::identity;
    for (int64_t base = 0; base < nb; base += kThreads) {
        const int64_t i = base + threadIdx.x;
        const int v = i < nb ? sums[i] : Op::identity;
        int total;
        const int exc = block_exclusive_scan(v, op, wave_tot, total);
        if (i < nb) sums[i] = op(carry, exc);
        carry = op(carry, total);
    }
    if (threadIdx.x == 0) sums[nb] = carry;
}

template <class Op, bool kInclusive>
__global__ __launch_bounds__(kThreads) void scan_apply(const int *__restrict__ in, int64_t n,
                                                       const int *__restrict__ sums,
                                                       int *__restrict__ out,
                                                       int *__restrict__ total_out, int64_t nb)
{
    __shared__ int wave_tot[kThreads / 64];
    Op op;
    const int64_t base = (int64_t)blockIdx.x * kTile + (int64_t)threadIdx.x * kItems;
    int v[kItems];
    int acc = Op::identity;
#pragma unroll
    for (int j = 0; j < kItems; j++) {
        v[j] = base + j < n ? in[base + j] : Op::identity;
        acc = op(acc, v[j]);
    }
    int total;
    int run = op(sums[blockIdx.x], block_exclusive_scan(acc, op, wave_tot, total));
#pragma unroll
    for (int j = 0; j < kItems; j++) {
        const int inc = op(run, v[j]);
        if (base + j < n) out[base + j] = kInclusive ? inc : run;
        run = inc;
    }
    if (total_out && blockIdx.x == 0 && threadIdx.x == 0) *total_out = sums[nb];
}

// out = scan(in) over n ints (in place allowed); *total_out (device, optional)
// receives the reduction of all n.  `sums` needs n/kTile + 2 ints.
template <class Op, bool kInclusive>
int device_scan(const int *in, int64_t n, int *out, int *total_out, int *sums, hipStream_t s)
{
    if (n <= 0) {
        if (total_out) return fill_u32(total_out, (uint32_t)Op::identity, 1, s);
        return ACCEL_OK;
    }
    const int64_t nb = (n + kTile - 1) / kTile;
    scan_reduce<Op><<<dim3((unsigned)nb), dim3(kThreads), 0, s>>>(in, n, sums);
    scan_spine<Op><<<dim3(1), dim3(kThreads), 0, s>>>(sums, nb);
    scan_apply<Op, kInclusive><<<dim3((unsigned)nb), dim3(kThreads), 0, s>>>(in, n, sums, out,
                                                                            total_out, nb);
    ACCEL_HIP(hipGetLastError());
    return ACCEL_OK;
}


__global__ __launch_bounds__(kThreads) void run_head_kernel(const int32_t *__restrict__ indptr, int64_t rows,
                                                            int *__restrict__ head)
{
    const int64_t r = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (r < rows)
        head[r] = (r == 0 || indptr[r + 1] - indptr[r] != indptr[r] - indptr[r - 1]) ? (int)r : 0;
}

__global__ __launch_bounds__(kThreads) void block_count_kernel(const int32_t *__restrict__ indptr,
                                                               const int *__restrict__ run_start, int64_t rows,
                                                               int *__restrict__ count)
{
    const int64_t r = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (r >= rows) return;
    const int d = indptr[r + 1] - indptr[r];
    int c = 0;
    if (d > kDegBound) {
        c = (d + kDegBound - 1) / kDegBound;
    } else if (d > 0) {
        int w, rpb;
        slice_rule(d, w, rpb);
        c = ((int)r - run_start[r]) % rpb == 0;
    }
    count[r] = c;
}

__global__ __launch_bounds__(kThreads) void emit_block4_kernel(const int32_t *__restrict__ indptr,
                                                               const int *__restrict__ run_start,
                                                               const int *__restrict__ row_block, int64_t rows,
                                                               int4 *__restrict__ block4)
{
    const int64_t r = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (r >= rows) return;
    const int loc = indptr[r], d = indptr[r + 1] - loc;
    if (d == 0) return;
    const int at = row_block[r];
    if (d > kDegBound) {
        const int nseg = (d + kDegBound - 1) / kDegBound;
        for (int k = 0; k < nseg; k++)
            block4[at + k] = make_int4(d, (int)r, loc + k * kDegBound, min(kDegBound, d - k * kDegBound));
        return;
    }
    int w, rpb;
    slice_rule(d, w, rpb);
    if (((int)r - run_start[r]) % rpb != 0) return;
    int n = 1;
    while (n < rpb && r + n < rows && indptr[r + n + 1] - indptr[r + n] == d) n++;
    block4[at] = make_int4(d, (int)r, loc, (w << 16) + n);
}

__global__ __launch_bounds__(kThreads) void compare_order_kernel(const uint32_t *__restrict__ a,
                                                                 const uint32_t *__restrict__ b, int64_t n,
                                                                 Mail *__restrict__ mail)
{
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < n && a[i] != b[i]) mail->bad_order = 1;
}

__global__ __launch_bounds__(1) void report_blocks_kernel(const int *__restrict__ total, Mail *__restrict__ mail)
{
    mail->n_blocks = *total;
}

// Rows in any order: block4 from scans over the rows.  *block4_out is the caller's to give back.
// Rows in ascending degree order: the first row of every degree up to 384 and of the longer ones, into mail->hist (-1
// where there is none), the entries of the longer ones per workgroup, and whether anything is wrong or out of order.  Four
// rows per thread.
__global__ __launch_bounds__(kThreads) void run_bounds_kernel(const int32_t *__restrict__ indptr, int64_t rows, int64_t nnz,
                                                              Mail *__restrict__ mail)
{
    __shared__ int sum[kWaves4];
    const int lane = threadIdx.x & 63;
    int long_blocks = 0;
    bool bad = false, unsorted = false;
    for (int64_t r0 = ((int64_t)blockIdx.x * kThreads + threadIdx.x - lane) * 4; r0 < rows; r0 += (int64_t)gridDim.x * kThreads * 4) {
        const int64_t r = r0 + lane * 4;                     // of this lane; the wavefront stays together
        int at[6];                                           // indptr[r - 1 .. r + 4], as far as there are
        if (r + 3 <= rows) {
            const int4 v = *reinterpret_cast<const int4 *>(indptr + r);
            at[1] = v.x; at[2] = v.y; at[3] = v.z; at[4] = v.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) at[1 + j] = r + j <= rows ? indptr[r + j] : 0;
        }
        at[0] = __shfl_up(at[4], 1);
        at[5] = __shfl_down(at[1], 1);
        if (lane == 0 && r > 0) at[0] = indptr[r - 1];
        if (lane == 63 && r + 4 <= rows) at[5] = indptr[r + 4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (r + j >= rows) break;
            const int d = at[j + 2] - at[j + 1], before = r + j > 0 ? at[j + 1] - at[j] : -1;
            bad |= d < 0 || (r + j == 0 && at[j + 1] != 0) || (r + j == rows - 1 && (int64_t)at[j + 2] != nnz);
            unsorted |= d < before;
            const int bin = min(max(d, 0), kLongBin);
            if (before < 0 || bin != min(before, kLongBin)) mail->hist[bin] = (int)(r + j);
            if (d > kDegBound) long_blocks += blocks_of(d);
        }
    }
    if (bad) mail->stat[kStatBadIndptr] = 1;
    if (unsorted) mail->stat[kStatUnsorted] = 1;
    long_blocks = wave_sum(long_blocks);
    if (lane == 0) sum[threadIdx.x >> 6] = long_blocks;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < kWaves4; q++) long_blocks += sum[q];
        if (long_blocks > 0) mail->part[blockIdx.x] = long_blocks;
    }
}

// Entries of each of the n rows from `indptr` on, and zeroed words for the scan.
__global__ __launch_bounds__(kThreads) void run_sizes_kernel(const int32_t *__restrict__ indptr, int n, int *__restrict__ blocks,
                                                             int *__restrict__ zeroed, int n_zeroed)
{
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n_zeroed) zeroed[i] = 0;                         // (fewer than the rows, but for the first few)
    if (i < n) blocks[i] = blocks_of(indptr[i + 1] - indptr[i]);
}

struct EmitRunsArgs {
    int run_row[kBins + 1], run_blk[kBins];   // first row and first entry of each degree
    const int32_t *indptr;
    const int *first_block;                   // of the rows longer than 384, scanned (null: none is wanted)
    int4 *out;
    int64_t b0;                               // entries b0 .. b0 + n - 1 go to out[0 .. n - 1]
    int n;
};
static_assert(sizeof(EmitRunsArgs) <= 4096, "kernel arguments");
__global__ __launch_bounds__(kThreads) void emit_runs_kernel(EmitRunsArgs a)
{
    __shared__ int run_row[kBins + 1], run_blk[kBins];
    for (int i = threadIdx.x; i <= kBins; i += kThreads) run_row[i] = a.run_row[i];
    for (int i = threadIdx.x; i < kBins; i += kThreads) run_blk[i] = a.run_blk[i];
    __syncthreads();
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= a.n) return;
    const int b = (int)(a.b0 + i);
    int4 e;
    if (b < run_blk[kLongBin]) {
        int lo = 1, hi = kDegBound;                          // the last degree whose entries start at or before b
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (run_blk[mid] <= b) lo = mid; else hi = mid - 1;
        }
        int w, rpb;
        slice_rule(lo, w, rpb);
        const int p = run_row[lo] + (b - run_blk[lo]) * rpb;
        e = make_int4(lo, p, a.indptr[p], (w << 16) + min(rpb, run_row[lo + 1] - p));
    } else {
        int lo = 0, hi = run_row[kBins] - run_row[kLongBin] - 1;     // the last row whose entries start at or before b
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (a.first_block[mid] <= b) lo = mid; else hi = mid - 1;
        }
        const int p = run_row[kLongBin] + lo, from = a.indptr[p], d = a.indptr[p + 1] - from, off = (b - a.first_block[lo]) * kDegBound;
        e = make_int4(d, p, from + off, min(kDegBound, d - off));
    }
    a.out[i] = e;
}

static int emit_runs_piece(const void *args, void *stage, size_t offset, size_t bytes, hipStream_t s)
{
    EmitRunsArgs a = *static_cast<const EmitRunsArgs *>(args);
    a.out = static_cast<int4 *>(stage);
    a.b0 = (int64_t)(offset / sizeof(int4));
    a.n = (int)(bytes / sizeof(int4));
    emit_runs_kernel<<<dim3(grid_for(a.n)), dim3(kThreads), 0, s>>>(a);
    ACCEL_HIP(hipGetLastError());
    return ACCEL_OK;
}

int partition_any_order(Arena *tmp, const int32_t *indptr, int64_t rows, int32_t **block4_out, int64_t *n_blocks,
                        Mail *mail, hipStream_t s)
{
    int *head, *cnt, *sums, *rb, rc;
    DevBuf b4;
    if ((rc = tmp->alloc(&head, (size_t)rows))) return rc;
    if ((rc = tmp->alloc(&cnt, (size_t)rows))) return rc;
    if ((rc = tmp->alloc(&rb, (size_t)rows + 1))) return rc;
    if ((rc = tmp->alloc(&sums, (size_t)(rows / kTile + 4)))) return rc;
    run_head_kernel<<<dim3(grid_for(rows)), dim3(kThreads), 0, s>>>(indptr, rows, head);
    if ((rc = device_scan<MaxOp, true>(head, rows, head, nullptr, sums, s))) return rc;
    block_count_kernel<<<dim3(grid_for(rows)), dim3(kThreads), 0, s>>>(indptr, head, rows, cnt);
    if ((rc = device_scan<SumOp, false>(cnt, rows, rb, rb + rows, sums, s))) return rc;
    report_blocks_kernel<<<dim3(1), dim3(1), 0, s>>>(rb + rows, mail);
    ACCEL_HIP(hipStreamSynchronize(s));
    *n_blocks = mail->n_blocks;
    if ((rc = b4.alloc(sizeof(int4) * (size_t)*n_blocks))) return rc;
    emit_block4_kernel<<<dim3(grid_for(rows)), dim3(kThreads), 0, s>>>(indptr, head, rb, rows, b4.as<int4>());
    ACCEL_HIP(hipGetLastError());
    *block4_out = static_cast<int32_t *>(b4.release());
    return ACCEL_OK;
}

}  // namespace

// Counts and statistics of the rows; on return they are in `mail` and the scanned counts in
// *bins_out, totals in *total_out.  One synchronisation.
static int count_rows(Arena *tmp, const int32_t *indptr, const int32_t *idx, int64_t rows, int64_t cols, int64_t nnz,
                      int split, int alt_split, const Shares &sh, int **bins_out, int **total_out, Mail *mail,
                      hipStream_t s)
{
    int *stats, rc;
    if ((rc = tmp->alloc(bins_out, (size_t)kBins * sh.pitch))) return rc;
    if ((rc = tmp->alloc(total_out, (size_t)kBins))) return rc;
    if ((rc = tmp->alloc(&stats, (size_t)sh.groups() * 16))) return rc;
    // Columns within 4,096 of a row's place on the diagonal count as near: 8,192 rows of X of 64
    // floats are half of one L2.
    const DegreeArgs da{indptr, nnz > 0 ? idx : nullptr, rows, cols, nnz, sh.share, sh.n, sh.pitch, split, alt_split, 4096};
    degree_kernel<<<dim3(sh.groups()), dim3(kThreads), 0, s>>>(da, *bins_out, stats);
    bin_scan_kernel<<<dim3(kBins + 1), dim3(kThreads), 0, s>>>(*bins_out, sh.pitch, stats, (int)sh.groups(), *total_out,
                                                              mail);
    ACCEL_HIP(hipGetLastError());
    ACCEL_HIP(hipStreamSynchronize(s));
    if (mail->stat[kStatBadIndptr]) {
        set_error("indptr must start at 0, be non-decreasing and end at nnz");
        return ACCEL_ERR_CSR;
    }
    return ACCEL_OK;
}

// Blocks, non-zeros and (with a unit rule) units of the rows of up to `most` non-zeros, when the
// rows are in ascending degree order: every degree is one run of hist[d] rows.
struct RunTotals {
    int64_t blocks = 0, nnz = 0, units = 0;
};
// (The GPU waits for this: 32-bit divisions, and up to `whole_most` on the way, when that is asked for.)
static RunTotals run_totals(const int *hist, int most, int unit_nz, int whole_most = 0, RunTotals *whole = nullptr)
{
    RunTotals t;
    for (int d = 1; d <= most; d++) {
        if (hist[d]) {
            int w, rpb;
            slice_rule(d, w, rpb);
            const unsigned n = (unsigned)hist[d], b = (unsigned)rpb, full = n / b, rest = n % b;
            const unsigned rpu = std::max(1u, (unsigned)unit_nz / (unsigned)d);
            t.blocks += full + (rest > 0);
            t.nnz += (int64_t)n * d;
            t.units += (int64_t)full * ((b + rpu - 1) / rpu) + (rest + rpu - 1) / rpu;
        }
        if (d == whole_most) *whole = t;
    }
    return t;
}

// Partition a row order as given (no sort): the GPU counterpart of running
// block_level_partition.py on one *.new_indptr file.  At most `cap` entries go to block4_out.
//
// Rows in ascending degree order, which is what those files hold: one pass finds where each degree's run starts, and an
// entry is a closed form of its number (of the rows longer than 384, after a scan).  The entries are written straight into the
// pinned memory they leave the device through.  2.45 M rows: the passes of the sort took 96 us and copies from device memory
// 190; so 16 and 165, bound by the link (the whole call 645 -> 566 us).
int partition_to_host(const int32_t *indptr_dev, int64_t rows, int64_t nnz, int32_t *block4_out, int64_t cap,
                      int64_t *n_blocks)
{
    hipStream_t s = nullptr;
    MailHolder mh;
    if (!mh.m) return ACCEL_ERR_ALLOC;
    Mail *mail = mh.m;
    Arena tmp;
    int rc;
    for (int &first : mail->hist) first = -1;
    for (int &v : mail->stat) v = 0;
    for (int &v : mail->part) v = 0;
    const int64_t tiles = (rows + 4 * kThreads - 1) / (4 * kThreads);
    run_bounds_kernel<<<dim3((unsigned)std::min<int64_t>(tiles, kRunParts)), dim3(kThreads), 0, s>>>(indptr_dev, rows, nnz, mail);
    ACCEL_HIP(hipGetLastError());
    ACCEL_HIP(hipStreamSynchronize(s));
    if (mail->stat[kStatBadIndptr]) {
        set_error("indptr must start at 0, be non-decreasing and end at nnz");
        return ACCEL_ERR_CSR;
    }
    if (mail->stat[kStatUnsorted]) {
        tmp.next_chunk = (size_t)rows * 13 + (1 << 16);
        int32_t *b4 = nullptr;
        rc = partition_any_order(&tmp, indptr_dev, rows, &b4, n_blocks, mail, s);
        mh.written = rc == ACCEL_OK;
        const int64_t take = std::min(*n_blocks, cap);
        if (!rc && take > 0) rc = download(block4_out, b4, sizeof(int4) * (size_t)take, s);
        give_memory(b4, InUse::null_stream);
        return rc;
    }
    mh.written = true;
    EmitRunsArgs ea{};
    ea.indptr = indptr_dev;
    ea.run_row[kBins] = (int)rows;
    int64_t n_short = 0;
    for (int d = kLongBin; d >= 0; d--) ea.run_row[d] = mail->hist[d] >= 0 ? mail->hist[d] : ea.run_row[d + 1];
    for (int d = 0; d < kLongBin; d++) {
        ea.run_blk[d] = (int)n_short;
        if (d == 0) continue;
        int w, rpb;
        slice_rule(d, w, rpb);
        n_short += (ea.run_row[d + 1] - ea.run_row[d] + rpb - 1) / rpb;
    }
    ea.run_blk[kLongBin] = (int)n_short;
    int64_t nb = n_short;
    for (const int v : mail->part) nb += v;
    const int n_long = (int)rows - ea.run_row[kLongBin];
    *n_blocks = nb;
    const int64_t take = std::min(nb, cap);
    if (n_long > 0 && take > n_short) {
        int *first_block, *zeroed;
        const int64_t n_zeroed = scan_zeroed(n_long);
        tmp.next_chunk = (size_t)n_long * 4 + (size_t)n_zeroed * 4 + (1 << 12);
        if ((rc = tmp.alloc(&first_block, (size_t)n_long + 1))) return rc;
        if ((rc = tmp.alloc(&zeroed, (size_t)n_zeroed))) return rc;
        run_sizes_kernel<<<dim3(grid_for(n_long)), dim3(kThreads), 0, s>>>(indptr_dev + ea.run_row[kLongBin], n_long, first_block,
                                                                           zeroed, (int)n_zeroed);
        launch_scans({{{first_block, first_block, n_long, (int)n_short, zeroed}}, {}}, 1, s);
        ea.first_block = first_block;
    }
    if (take == 0) return ACCEL_OK;
    return download_made(block4_out, sizeof(int4) * (size_t)take, s, emit_runs_piece, &ea);
}

// Small matrices are latency-bound: the time of a launch is the longest chain of
// dependent memory round trips in one wavefront, not the traffic.  For them a unit is
// given to a whole workgroup (four wavefronts share its rows, or its row's non-zeros),
// which shortens that chain, as long as the launch's workgroups are few: 2,048 of them are
// on the GPU at once, and from about twice as many on wavefront units are faster (four
// times fewer workgroups).  Units are about rows / 12 + nnz / 96, from the rows of a block4
// entry and the unit size.  The choice is made without N, and between some 2,400 and 4,400 units it
// depends on N which is faster: the line lies at the upper end of that, where workgroup units are still
// level at N = 64.  Measured (one matrix, runs back to back, N = 12 / 32 / 64 / 128, workgroup
// units, then wavefront units of up to 384):
//   100 k non-zeros in 10 k rows, power law (1,900):   4.8 / 5.8 / 6.8 / 11.3 us,    6.8 / 7.4 / 8.1 / 9.6
//   150 k in 10 k rows, power law (2,400):             5.1 / 6.6 / 7.3 / 9.1,        7.3 / 7.0 / 8.3 / 9.1
//   80 k in 20 k rows, near the diagonal (2,500):      4.7 / 5.4 / 5.6 / 7.6,        4.7 / 4.8 / 6.5 / 7.9
//   120 k in 20 k rows, power law (2,900):             5.2 / 6.2 / 7.8 / 9.4,        6.9 / 7.5 / 9.1 / 12.4
//   208 k in 10 k rows, power law (3,000):             5.9 / 7.6 / 8.6 / 11.0,       5.4 / 8.0 / 9.4 / 10.5
//   300 k in 3 k rows, lognormal (3,400):              5.8 / 6.8 / 7.2 / 10.1,       5.2 / 6.0 / 9.3 / 10.2
//   250 k in 10 k rows, power law (3,400):             6.5 / 8.4 / 9.3 / 14.5,       6.2 / 7.9 / 9.4 / 10.5
//   300 k in 15 k rows, power law (4,400):             7.4 / 9.4 / 11.2 / 14.2,      6.4 / 6.4 / 10.7 / 14.0
//   150 k in 38 k rows, near the diagonal (4,700):     6.5 / 6.9 / 8.4 / 13.2,       4.7 / 4.8 / 6.5 / 9.1
//   450 k in 27 k rows, hub rows (6,900):              13.1 / 14.3 / 17.0 / 22.9,    11.0 / 10.8 / 16.9 / 21.2
constexpr int64_t kTeamMaxUnits = 4096, kSmallNnz = 512 * 1024;
static bool choose_plan_team(int64_t rows, int64_t nnz)
{
    return nnz < kSmallNnz && rows / 12 + nnz / 96 < kTeamMaxUnits;
}

// Unit size of the launch plan: the most non-zeros of a unit of several whole rows (and,
// with wavefront units, of a piece of a split row).  Wavefront units keep the block4
// granularity (384: fewest descriptors and partial sums); 48 below 128 k non-zeros, where they
// are taken only when asked for.  Workgroup units want short chains: 96 non-zeros, 48 below
// 64 k non-zeros (10.0 against 11.2 us at N = 64 on a 35 k one).
static int choose_plan_unit(int64_t nnz, bool team)
{
    if (team) return nnz < (int64_t)64 * 1024 ? 48 : 96;
    return nnz < (int64_t)128 * 1024 ? 48 : kDegBound;
}

// Rows above this many non-zeros are stored by column group and cut into pieces, which
// a small matrix does not need for its balance and whose partial sums it waits for:
// 450 k non-zeros, N = 32: 4.4 us with 384, 6.3 with 192.
// Measured with 384, 256, 192, 128 and 96 (N = 64): 192 is 8 % faster than 384 on the
// dense 115 M-non-zero matrix, 2 % on the 125 M power-law one, neutral elsewhere;
// below 192 the extra partial sums start to cost at N = 16.
constexpr int kPlanSplit = 192;
static int choose_plan_split(int64_t nnz, bool team) { return team || nnz < kSmallNnz ? kDegBound : kPlanSplit; }

// Launches that fill the sorted copy (see CopyArgs).  Needs perm (or none), s_indptr, the bins' runs,
// n_split_rows and, for wide rows, the chunk tables, as the preprocessing leaves them on the handle.  The units of
// whole rows are listed (u.groups > 0) and the split rows counted for the plan (split.n_groups > 0) on the way.
static int copy_nonzeros(Arena *tmp, const accel_handle *h, const CopyArgs &a, int64_t nnz_short, const UnitsArgs &u,
                         SplitArgs split, hipStream_t s)
{
    const int64_t rows = h->rows;
    const int n_split = (int)h->n_split_rows, n_long = (int)h->n_long_rows, n_wide = (int)h->n_wide_rows;
    WideArgs wa{h->chunk_row, h->first_chunk, rows - n_long, n_long - n_wide, h->plan_groups, nullptr};
    if (n_wide > 0)
        if (int rc = tmp->alloc(&wa.chunk_count, (size_t)h->n_chunks * kMaxGroups)) return rc;
    CopyPlan cp{};
    cp.n_chunks = (int)h->n_chunks;
    cp.n_mid = n_long - n_wide;
    cp.n_small = n_split - n_long;
    cp.mid_groups = (int)grid_for((int64_t)cp.n_mid * 64);
    cp.small_groups = (int)grid_for((int64_t)cp.n_small * 64);
    cp.first_mid = rows - n_long;
    cp.first_small = rows - n_split;
    cp.n_take = (int)nnz_short;
    cp.counts = split.gcount;
    // the tiles' workgroups start at a multiple of 8, so that the i-th of them is on die i % 8
    cp.small_groups += -(u.groups + cp.n_chunks + cp.mid_groups + cp.small_groups) & (kXcds - 1);
    const int64_t groups = (int64_t)u.groups + cp.n_chunks + cp.mid_groups + cp.small_groups + (int64_t)h->tiles.per_die * kXcds;
    if (groups > 0) copy_rows_kernel<<<dim3((unsigned)groups), dim3(kThreads), 0, s>>>(a, wa, cp, u, h->tiles);
    split.n_wide = n_wide;
    split.first_chunk = wa.first_chunk ? wa.first_chunk + wa.n_narrow : nullptr;
    split.chunk_count = wa.chunk_count;
    const int lone = (int)h->n_lone_chunks, placed = cp.n_chunks - lone, threads = place_threads(placed);
    if (placed + split.n_groups > 0)
        (threads == 256 ? wide_place_kernel<256> : wide_place_kernel<1024>)<<<
            dim3((unsigned)(placed + split.n_groups)), dim3((unsigned)threads), 0, s>>>(a, wa, lone, split);
    ACCEL_HIP(hipGetLastError());
    return ACCEL_OK;
}

static SortedRows sorted_rows(const accel_handle *h)
{
    SortedRows sr;
    sr.rows = h->rows;
    sr.indptr = h->indptr;
    sr.s_indptr = h->s_indptr;
    sr.perm = h->perm;
    sr.run_row = h->runs;
    sr.run_nz = h->runs + kBins + 1;
    return sr;
}

// New values on an unchanged structure reach the sorted copy through a map from sorted
// position to the position in the caller's arrays.  The map is what the copying kernels
// of the preprocessing compute anyway (where each non-zero comes from); it is built here, by
// those kernels with only that output switched on, the first time a handle's values are
// replaced, and kept.  Allocates; synchronises s.
int build_source_positions(accel_handle *h, hipStream_t s)
{
    if (h->src_pos || !h->owns_sorted || h->nnz == 0) return ACCEL_OK;
    DevBuf map;
    Arena tmp;
    tmp.any_stream = s != nullptr;
    if (int rc = map.alloc(sizeof(int32_t) * (size_t)h->nnz, s != nullptr)) return rc;
    const CopyArgs ca{sorted_rows(h), h->idx, nullptr, (uint32_t)h->cols, nullptr, map.as<int32_t>(), 1, nullptr};
    const int rc = copy_nonzeros(&tmp, h, ca, h->nnz_short, UnitsArgs{}, SplitArgs{}, s);
    const hipError_t e = hipStreamSynchronize(s);      // the temporaries are given back on return
    tmp.use = map.use = e == hipSuccess ? InUse::no : InUse::unknown;
    if (rc) return rc;
    ACCEL_HIP(e);
    h->src_pos = static_cast<int32_t *>(map.release());
    return ACCEL_OK;
}

// s_val[p] = val[src_pos[p]]: four non-zeros per thread, the map read and the values written
// as 16-byte vectors (both arrays start 256-byte aligned).
__global__ __launch_bounds__(kThreads) void gather_values_kernel(const float *__restrict__ val,
                                                                 const int32_t *__restrict__ src_pos,
                                                                 float *__restrict__ s_val, int64_t nnz)
{
    const int64_t p = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * 4;
    if (p + 4 <= nnz) {
        const int4 q = *reinterpret_cast<const int4 *>(src_pos + p);
        const float4 v = make_float4(val[q.x], val[q.y], val[q.z], val[q.w]);
        *reinterpret_cast<float4 *>(s_val + p) = v;
    } else {
        for (int64_t i = p; i < nnz; i++) s_val[i] = val[src_pos[i]];
    }
}

// One launch on s, no allocation, no wait: the sorted copy of the values from `val` (nnz
// floats in the caller's order).  The map must exist.
int gather_values(accel_handle *h, const float *val, hipStream_t s)
{
    if (!h->owns_sorted || h->nnz == 0) return ACCEL_OK;
    if (!h->src_pos) {
        set_error("internal: the position map of the value update is missing");
        return ACCEL_ERR_STATE;
    }
    const int64_t threads = (h->nnz + 3) / 4;
    gather_values_kernel<<<dim3(grid_for(threads)), dim3(kThreads), 0, s>>>(
        val, h->src_pos, const_cast<float *>(h->s_val), h->nnz);
    ACCEL_HIP(hipGetLastError());
    return ACCEL_OK;
}

// The other direction: val[src_pos[p]] = s_val[p].  A handle that owns a copy of the caller's
// values lets that copy go stale when the values are updated from a device array (the update
// then is the one gather above); the copy is only read again by a new preprocessing of the
// same handle, which calls this first.  Synchronises s.
__global__ __launch_bounds__(kThreads) void scatter_values_kernel(const float *__restrict__ s_val,
                                                                  const int32_t *__restrict__ src_pos,
                                                                  float *__restrict__ val, int64_t nnz)
{
    const int64_t p = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * 4;
    if (p + 4 <= nnz) {
        const int4 q = *reinterpret_cast<const int4 *>(src_pos + p);
        const float4 v = *reinterpret_cast<const float4 *>(s_val + p);
        val[q.x] = v.x; val[q.y] = v.y; val[q.z] = v.z; val[q.w] = v.w;
    } else {
        for (int64_t i = p; i < nnz; i++) val[src_pos[i]] = s_val[i];
    }
}

int restore_own_values(accel_handle *h, hipStream_t s)
{
    if (!h->val_stale) return ACCEL_OK;
    if (!h->owns_input || !h->owns_sorted || !h->src_pos || !h->s_val) {
        set_error("internal: the handle's copy of the values is stale and cannot be restored");
        return ACCEL_ERR_STATE;
    }
    const int64_t threads = (h->nnz + 3) / 4;
    scatter_values_kernel<<<dim3(grid_for(threads)), dim3(kThreads), 0, s>>>(
        h->s_val, h->src_pos, const_cast<float *>(h->val), h->nnz);
    ACCEL_HIP(hipGetLastError());
    ACCEL_HIP(hipStreamSynchronize(s));
    h->val_stale = false;
    return ACCEL_OK;
}

// given: a row order from a saved state, or null.  The sort runs either way: the order it gives is
// the only one that is right for this CSR (ascending degree, ties by ascending row), so a stored
// order is checked against it and refused if it differs anywhere.
int preprocess_device(accel_handle *h, const SavedOrder *given)
{
    const auto t0 = std::chrono::steady_clock::now();
    hipStream_t s = nullptr;
    const int64_t rows = h->rows, nnz = h->nnz;
    int rc;

    h->ready = false;
    h->n_blocks = h->n_long_blocks = h->n_long_rows = h->n_zero_rows = 0;
    h->max_degree = 0;
    h->n_units = h->n_long_units = 0;
    h->n_split_rows = h->n_big_rows = h->n_wide_rows = h->n_chunks = h->n_lone_chunks = 0;
    h->plan_team = h->plan_team_option == 2 || (h->plan_team_option == 0 && choose_plan_team(rows, nnz));
    h->plan_unit = h->plan_unit_option > 0 ? h->plan_unit_option : choose_plan_unit(nnz, h->plan_team);
    h->plan_split = h->plan_split_option > 0 ? h->plan_split_option : choose_plan_split(nnz, h->plan_team);
    // a wavefront never takes more than plan_unit non-zeros; a workgroup takes a whole row of
    // up to plan_split even when units of several rows are kept smaller
    if (!h->plan_team) h->plan_split = std::min(h->plan_split, h->plan_unit);
    // Eight interleaved queues when the device is the whole MI355X (8 dies of 32 compute
    // units, workgroup i on die i % 8); any other shape (a partition of the GPU) gets the
    // plan in plain order, one queue, whose column groups are still worked on one by one.
    h->plan_queues = h->plan_queues_option > 0 ? h->plan_queues_option
                                               : (h->device_cus == kXcds * kCusPerDie ? kXcds : 1);
    if (rows == 0) {
        h->identity_perm = true;
        h->ready = true;
        return ACCEL_OK;
    }
    MailHolder mh;
    if (!mh.m) return ACCEL_ERR_ALLOC;
    Mail *mail = mh.m;

    // ---- degrees, statistics, bins: what everything else is sized by ------------
    Arena tmp;
    const Shares sh(rows);
    int *bins, *bin_total;
    tmp.next_chunk = (size_t)kBins * sh.pitch * 4 + (size_t)sh.groups() * 64 + (1 << 14);
    if ((rc = count_rows(&tmp, h->indptr, h->idx, rows, h->cols, nnz, h->plan_split, h->plan_unit, sh, &bins, &bin_total,
                         mail, s)))
        return rc;
    const int *st = mail->stat;
    // A matrix whose non-zeros lie near the diagonal keeps its locality only in rows that stay
    // whole (their neighbourhood of X is what a die has in its L2 while it works through a band
    // of rows); storing such rows by column group trades that for nothing.  Measured at N = 64
    // with columns within N(0, 2000) of the row id: threshold 384 against 192: 593 against 651 us
    // (42 M non-zeros), 31 against 35 us (1.6 M); with N(0, 50000), which no L2 holds, 192 stays
    // better (1.14 against 1.24 ms).
    h->local = st[kStatSampled] > 0 && 2 * (int64_t)st[kStatLocal] >= st[kStatSampled];
    const bool alt = h->local && h->plan_split_option == 0 && h->plan_split < h->plan_unit;
    if (alt) h->plan_split = h->plan_unit;
    h->max_degree = st[kStatMaxDegree];
    h->n_zero_rows = mail->hist[0];
    h->n_long_rows = mail->hist[kLongBin];
    h->n_long_blocks = st[kStatLongBlocks];
    h->n_wide_rows = st[kStatWideRows];
    h->n_chunks = st[kStatWideChunks];
    h->n_lone_chunks = st[kStatLoneChunks];
    h->n_big_rows = alt ? st[kStatBigAlt] : st[kStatBig];
    h->n_split_rows = h->n_long_rows;
    for (int d = h->plan_split + 1; d <= kDegBound; d++) h->n_split_rows += mail->hist[d];
    h->identity_perm = !st[kStatUnsorted];
    if (given && given->identity != h->identity_perm) {
        set_error("the saved state was made for rows in another order (it says the rows are %s sorted by "
                  "degree, this CSR's are%s)", given->identity ? "already" : "not", h->identity_perm ? "" : " not");
        return ACCEL_ERR_META;
    }
    const int64_t n_split = h->n_split_rows;
    RunTotals whole;                                                                 // the rows that stay whole
    const RunTotals binned = run_totals(mail->hist, kDegBound, h->plan_unit, h->plan_split, &whole);
    const int64_t nb = binned.blocks + h->n_long_blocks;
    if (nb + (int64_t)kMaxGroups * n_split + kXcds * kWavesPerGroup > (int64_t)INT_MAX) {
        set_error("the launch plan would exceed 2^31 work units (%lld block4 entries)", (long long)nb);
        return ACCEL_ERR_ARG;
    }

    // ---- memory: temporaries in one piece, and the products that stay in two ----------
    UnitRule rule{h->plan_split, h->plan_unit, h->plan_groups, 2, std::max(24, h->plan_unit / 4)};
    // total cost = about (nnz + 10 rows) >> shift + units < 2^31
    while (((nnz + 10 * rows) >> rule.cost_shift) + rows >= ((int64_t)1 << 30)) rule.cost_shift++;
    const int n_long = (int)h->n_long_rows, n_wide = (int)h->n_wide_rows;
    const int64_t plan_zeroed = plan_zeroed_ints(n_split, mail, h->plan_groups);
    const int64_t n_zeroed = plan_zeroed + long_zeroed_ints(n_long);
    tmp.next_chunk = (size_t)rows * 4 + (size_t)n_long * (n_long > kFewLong ? 48 : 8) + (size_t)n_zeroed * 4 +
                     (size_t)kSums * (sh.pitch + kWaves4) * 4 + (size_t)n_split * (256 + 8) +
                     (size_t)plan_zeroed * kScanTile / 2 * 4 + (size_t)h->n_chunks * 260 + (size_t)whole.units * 24 +
                     (1 << 16);
    uint32_t *place, *long_row;
    int *zeroed, *long_deg, *gcount = nullptr;
    PlanUnits pu;
    if ((rc = tmp.alloc(&place, (size_t)rows))) return rc;
    if ((rc = tmp.alloc(&pu.sums, (size_t)kSums * (sh.pitch + kWaves4)))) return rc;
    if ((rc = tmp.alloc(&pu.units, (size_t)whole.units))) return rc;
    if ((rc = tmp.alloc(&pu.running, (size_t)whole.units + 1))) return rc;
    if ((rc = tmp.alloc(&pu.heavy_before, (size_t)whole.units + 1))) return rc;
    if (n_split > 0 && (rc = tmp.alloc(&pu.rank8, (size_t)n_split))) return rc;
    if ((rc = tmp.alloc(&zeroed, (size_t)n_zeroed))) return rc;
    if ((rc = tmp.alloc(&long_deg, (size_t)n_long))) return rc;
    if ((rc = tmp.alloc(&long_row, (size_t)n_long))) return rc;
    if (n_split > 0 && (rc = tmp.alloc(&gcount, (size_t)n_split * kMaxGroups))) return rc;
    // Split rows (more than plan_split non-zeros: the last n_split rows of the sorted order) are
    // stored grouped by column group; all other rows keep their non-zero order.  The caller's
    // arrays are used in place only when the input was already sorted and has no split row.
    const bool own_copy = !h->identity_perm || n_split > 0;
    auto pad = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t b_sip = pad(sizeof(int32_t) * (size_t)(rows + 1));
    const size_t b_perm = h->identity_perm ? 0 : pad(sizeof(int32_t) * (size_t)rows);
    const size_t b_runs = pad(sizeof(int) * (2 * kBins + 1));
    const size_t b_chk = n_wide ? pad(sizeof(int) * (size_t)(n_long + 1 + h->n_chunks)) : 0;
    const size_t b_nz = own_copy ? pad(sizeof(int32_t) * (size_t)nnz) : 0;
    DevBuf slab, b4;
    if ((rc = slab.alloc(b_sip + b_perm + b_runs + b_chk + 2 * b_nz))) return rc;
    if ((rc = b4.alloc(sizeof(int4) * (size_t)nb))) return rc;
    char *at = slab.as<char>();
    h->s_indptr = reinterpret_cast<int32_t *>(at);
    at += b_sip;
    h->perm = b_perm ? reinterpret_cast<int32_t *>(at) : nullptr;
    at += b_perm;
    h->runs = reinterpret_cast<int *>(at);
    at += b_runs;
    h->first_chunk = b_chk ? reinterpret_cast<int *>(at) : nullptr;
    h->chunk_row = b_chk ? h->first_chunk + n_long + 1 : nullptr;
    at += b_chk;
    int32_t *s_idx = reinterpret_cast<int32_t *>(at);
    float *s_val = reinterpret_cast<float *>(at + b_nz);

    // ---- sort: perm, place, s_indptr, block4 ------------------------------------------
    PlaceArgs pa{};
    pa.indptr = h->indptr; pa.rows = rows; pa.share = sh.share; pa.n_shares = sh.n; pa.pitch = sh.pitch;
    pa.bins = bins; pa.bin_total = bin_total; pa.rule = rule;
    pa.perm = h->perm; pa.place = place; pa.s_indptr = h->s_indptr;
    pa.block4 = b4.as<int4>();
    pa.run_row = h->runs; pa.run_nz = h->runs + kBins + 1;
    pa.long_deg = long_deg; pa.long_row = long_row;
    pa.sums = pu.sums; pa.zero = zeroed; pa.n_zero = n_zeroed;
    place_rows_kernel<<<dim3(sh.groups()), dim3(kThreads), 0, s>>>(pa);
    LongArgs la{};
    la.deg = long_deg; la.row = long_row; la.n = n_long; la.first_long = rows - n_long;
    la.nz0 = (int)binned.nnz; la.block0 = (int)binned.blocks;
    la.perm = h->perm; la.place = place; la.s_indptr = h->s_indptr;
    la.block4 = b4.as<int4>();
    la.first_chunk = h->first_chunk; la.chunk_row = h->chunk_row;
    UnitsArgs ua{};
    ua.sr = sorted_rows(h);
    ua.sr.place = place;
    ua.rule = rule; ua.pu = pu;
    ua.share = sh.share; ua.n_shares = sh.n; ua.pitch = sh.pitch + kWaves4; ua.first_split = (int)(rows - n_split);
    ua.groups = (int)sh.groups();
    if ((rc = place_long_rows(&tmp, la, h->max_degree, h->s_indptr, zeroed + plan_zeroed, pu.sums, ua.pitch, sh.n, s)))
        return rc;
    if (given && !h->identity_perm)
        compare_order_kernel<<<dim3(grid_for(rows)), dim3(kThreads), 0, s>>>(
            reinterpret_cast<const uint32_t *>(h->perm), given->perm_dev, rows, mail);
    ACCEL_HIP(hipGetLastError());

    // ---- sorted CSR; every column is looked at once on the way -------------------------
    DevBuf slot;
    SplitArgs split;
    if ((rc = prepare_split_rows(&tmp, h, ua.sr, rule, pu, mail, &slot, &split))) return rc;
    split.gcount = gcount;
    if (own_copy) {
        h->tiles = order_tiles(mail->hist, h->plan_split);
        const CopyArgs ca{sorted_rows(h), h->idx, h->val, (uint32_t)h->cols, s_idx, reinterpret_cast<int32_t *>(s_val), 0,
                          mail};
        if ((rc = copy_nonzeros(&tmp, h, ca, whole.nnz, ua, split, s))) return rc;
    } else {
        copy_rows_kernel<<<dim3((unsigned)ua.groups), dim3(kThreads), 0, s>>>(CopyArgs{}, WideArgs{}, CopyPlan{}, ua, TileOrder{});
        if (nnz > 0) {
            const unsigned g = (unsigned)std::min<int64_t>((nnz / 4 + kThreads - 1) / kThreads + 1, 16384);
            index_check_kernel<<<dim3(g), dim3(kThreads), 0, s>>>(h->idx, nnz, h->cols, mail);
        }
    }

    // ---- work list (ends on the second synchronisation) -----------------------------------
    h->nnz_short = whole.nnz;
    if ((rc = build_work_list(&tmp, h, ua.sr, rule, sh, pu, split, &slot, whole.units, zeroed, mail, s))) return rc;
    mh.written = true;
    if (mail->bad_index) {
        set_error("a column index lies outside [0, cols)");
        return ACCEL_ERR_CSR;
    }
    if (mail->bad_order) {
        set_error("the saved row order is not the degree order of this CSR (state of another matrix, or damaged)");
        return ACCEL_ERR_META;
    }
    h->slab = slab.release();
    h->block4 = static_cast<int32_t *>(b4.release());
    h->n_blocks = nb;
    h->owns_sorted = own_copy;
    h->s_idx = own_copy ? s_idx : h->idx;
    h->s_val = own_copy ? s_val : h->val;
    h->ready = true;
    h->preprocess_ms =
        std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return ACCEL_OK;
}

}  // namespace accel
