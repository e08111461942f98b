// The SpMM gather kernels for gfx950 (wave64), the partial-sum reduction and two helpers.
//
// Work decomposition.  Upstream gives one CUDA thread block of 12 32-lane warps
// to each block4 entry (spmm_accel.cu:18-28).  Here one 64-lane wavefront takes
// one work unit and a 256-thread workgroup takes four.  A unit is either whole
// rows of one block4 entry (up to 12 rows of one degree, <= 384 non-zeros in
// total) or a piece of <= 384 non-zeros of a split row (every row with more than
// 384 non-zeros is split; the plan also splits somewhat shorter ones).  The units
// come from a launch plan built by the preprocessing step; it orders them so that
// workgroup i, which the hardware places on die i % 8, works on a share of X that
// die keeps in its own L2: a column group for the pieces of split rows, a band of
// the caller's rows for the whole-row units.  Small matrices use the same list
// with one unit per workgroup instead (spmm_team_kernel below).
//
// Inside the wavefront the lanes form G = 64 / L groups of L lanes; a group owns
// L * VEC consecutive columns of X/Y (VEC = 4 floats = one 16-byte load per lane
// when N allows), so one vector-memory instruction gathers G different rows of X.
// This replaces upstream's "combined warp" of ceil32(N) lanes that walks one
// non-zero at a time with 4-byte loads (spmm_accel.cu:37-48,56-78).  G groups are
// split over the unit's rows as gp groups per row (gp a power of two chosen per
// unit to minimise the step count); the gp partial sums of a row are combined by
// a cross-lane butterfly, so short rows need no atomics (upstream: atomicAdd for
// every row that spans more than one warp, spmm_accel.cu:82-99).
//
// The (column index, value) pairs of the unit are first staged in LDS with
// coalesced loads, one pair per lane; each group then reads its pairs back with
// broadcast LDS reads.  Pieces of split rows write their partial sums to a
// scratch buffer and a second small kernel adds them up in a fixed order, so the
// result is run-to-run deterministic.  Rows of degree 0 are zero-filled by extra
// workgroups of the same launch: Y = A X holds after every run with no memset.
#include <mutex>

#include <hip/hip_ext.h>

#include "internal.h"

// Partial sums for accel_run_static, the entry point that allocates nothing: one copy of
// this array per GPU, held from the moment the library's code is loaded on that GPU until
// the process ends.  In host code the name is only a handle for the runtime, not a device
// address: static_scratch_address() asks for the address once per GPU and everything else
// (kernel arguments included) uses that pointer.
static constexpr size_t kStaticScratchFloats = (size_t)ACCEL_STATIC_SCRATCH_BYTES / sizeof(float);
static constexpr int kMaxScratchDevices = 64;
static __device__ __align__(256) float scratch[kStaticScratchFloats];

namespace accel {
namespace {

constexpr int kWaves = kWavesPerGroup;    // wavefronts (= work units) per workgroup
constexpr int kWgThreads = 64 * kWaves;
constexpr int kZeroFloats = 8192;         // floats zero-filled per extra workgroup
constexpr int kReduceThreads = 256;       // workgroup of the partial-sum reduction

// zero-degree rows handled by one zero-fill workgroup (N is a multiple of VEC, so
// a workgroup's share is a whole number of vectors)
__host__ __device__ inline int zero_rows_per_group(int N) { return N >= kZeroFloats ? 1 : kZeroFloats / N; }

constexpr int kUnroll = 4;                // gathers in flight per lane in the main loop (2 and 8 measured within 2 %)
constexpr int kPanel = 64;                // column-panel width for wide operands on large matrices
constexpr int kPanelMinNnz = 4000000;     // smaller matrices are not worth several launches
constexpr int kPadRows = 64;              // rows that a workgroup of pad_rows_kernel copies
constexpr int kPadMaxN = 512;             // wider rows: what padding saves is less than one line in 17
constexpr size_t kPadMaxFloats = ((size_t)1 << 30) - 1;   // copies below 4 GiB, a 64th of the memory (and 32-bit offsets)
constexpr int kStreamingMinBytes = 64;    // rows of Y of at least this many bytes are stored streaming
                                          // (64-byte rows: L2-resident X -18 %, elsewhere within 1 %)

// A vector of four floats that is only 4-byte aligned: rows of X and Y start at any
// multiple of 4 bytes when N is not a multiple of 4.  The hardware takes 16-byte
// accesses at such addresses; the type keeps the compiler from assuming more.
typedef float v4f __attribute__((ext_vector_type(4)));
typedef v4f v4f_unaligned __attribute__((aligned(4)));

template <int VEC, bool kShift>
__device__ __forceinline__ void load_vec(const float *__restrict__ p, float (&v)[VEC])
{
    if constexpr (VEC == 4 && kShift) {
        const v4f t = *reinterpret_cast<const v4f_unaligned *>(p);
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    } else if constexpr (VEC == 4) {
        const float4 t = *reinterpret_cast<const float4 *>(p);
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    } else {
        static_assert(VEC == 1, "vector widths: 4 or 1");
        v[0] = *p;
    }
}

// Rows of Y are written once and not read again by this launch: a streaming
// (non-temporal) store when `streaming`.  Measured on this GPU with gathers that hit L2:
// one ordinary 256-byte store per 32 gathers lowers the gather rate from 27 to 20 TB/s, a
// non-temporal one to 26 TB/s.
template <int VEC, bool kShift>
__device__ __forceinline__ void store_vec(float *__restrict__ p, const float (&v)[VEC], bool streaming)
{
    if constexpr (VEC == 4) {
        const v4f t = {v[0], v[1], v[2], v[3]};
        if constexpr (kShift) {
            if (streaming) __builtin_nontemporal_store(t, reinterpret_cast<v4f_unaligned *>(p));
            else *reinterpret_cast<v4f_unaligned *>(p) = t;
        } else {
            if (streaming) __builtin_nontemporal_store(t, reinterpret_cast<v4f *>(p));
            else *reinterpret_cast<v4f *>(p) = t;
        }
    } else {
        if (streaming) __builtin_nontemporal_store(v[0], p);
        else *p = v[0];
    }
}

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Partial sums that another wavefront of the same launch, possibly on another die, adds up
// (the row's last piece does, see finish_split_row): stored and loaded as relaxed atomics of
// device scope.  Such a store goes through to memory instead of staying in the die's L2, and
// such a load does not take a line the die's L2 may hold from before; no cache is written
// back or invalidated as a whole, which is what a device-scope fence would do on every piece.
template <int VEC>
__device__ __forceinline__ void store_partial(float *__restrict__ p, const float (&v)[VEC])
{
#pragma unroll
    for (int i = 0; i < VEC; i++) __hip_atomic_store(p + i, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_partial(const float *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A piece of a split row has stored its partial sums (this thread's stores included).  Counts
// the piece in; returns true to all T threads of the team (one wavefront, or the workgroup)
// if it was the row's last one, after which every piece's sums are in memory: each piece
// waits for its own stores before it counts itself in, and the counter is one memory location.
// `flag` is a word of LDS of the team's own.  The counter is left at zero for the next launch.
template <int T>
__device__ __forceinline__ bool last_piece_of_row(int *__restrict__ counter, int n_pieces, int tid, int *flag)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // this thread's partial sums have arrived
    if constexpr (T > 64) __syncthreads();                    // ... and those of the other wavefronts
    if (tid == 0) {
        const int before = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int last = before == n_pieces - 1;
        if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last;
    }
    if constexpr (T > 64) __syncthreads(); else __builtin_amdgcn_wave_barrier();
    return *flag != 0;
}

// Adds the nseg partial sums of a split row in slot order and writes the row: T threads
// (a wavefront or a workgroup), `red` = T floats of LDS of their own.  The columns are
// covered cw at a time (cw = the power of two <= T that covers N, or T); the T / cw slot
// groups take every (T / cw)-th slot and their sums are added in group order, so the result
// does not depend on which piece finished last.
template <int T>
__device__ __forceinline__ void finish_split_row(const float *__restrict__ src, int nseg, float *__restrict__ y,
                                                 int N, int ld, const float *__restrict__ bias, int relu,
                                                 int tid, float *red)
{
    int cw = 1;
    while (cw < N && cw < T) cw <<= 1;
    const int sg = T / cw;
    const int c_in = tid % cw, my_sg = tid / cw;
    for (int c0 = 0; c0 < N; c0 += cw) {
        const int c = c0 + c_in;
        float acc = 0.0f;
        if (c < N) {
            int s = my_sg;
            for (; s + 7 * sg < nseg; s += 8 * sg) {          // eight loads in flight, added in order
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = load_partial(src + (int64_t)(s + u * sg) * ld + c);
#pragma unroll
                for (int u = 0; u < 8; u++) acc += v[u];
            }
            for (; s < nseg; s += sg) acc += load_partial(src + (int64_t)s * ld + c);
        }
        if (sg > 1) {
            red[tid] = acc;
            if constexpr (T > 64) __syncthreads(); else __builtin_amdgcn_wave_barrier();
            if (my_sg == 0)
                for (int q = 1; q < sg; q++) acc += red[q * cw + c_in];
            if constexpr (T > 64) __syncthreads(); else __builtin_amdgcn_wave_barrier();
        }
        if (my_sg == 0 && c < N) {
            if (bias) acc += bias[c];
            if (relu) acc = fmaxf(acc, 0.0f);
            y[c] = acc;
        }
    }
}

// Stages the n pairs at idx, val in LDS, R rounds of T threads (T * (R - 1) < n <= T * R).  All loads are
// issued before the first is waited for: nothing depends on the thread but the last round's index, which
// is clamped.  (Loads under a condition per round make the compiler wait for one round before it issues
// the next.)  st has room for what the last round writes behind the n-th pair.
template <int R, int T, bool kWide>
__device__ __forceinline__ void stage_rounds(const int32_t *__restrict__ idx, const float *__restrict__ val, int n, int tid,
                                             int ldx, int2 *st)
{
    int c[R];
    float v[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
        const uint32_t i = (uint32_t)(j < R - 1 ? tid + T * j : min(tid + T * j, n - 1));
        c[j] = idx[i];
        v[j] = val[i];
    }
#pragma unroll
    for (int j = 0; j < R; j++)
        st[tid + T * j] = make_int2(kWide ? c[j] : (int)((uint32_t)c[j] * ((uint32_t)ldx * 4u)), __float_as_int(v[j]));
}

// The vector of row `where` of X at column col.  The staged pair holds the value and, when the operand is
// smaller than 4 GiB (kWide == false), the byte offset of the row, so that the address is one 32-bit add
// to a uniform base; otherwise the column, and the address is formed with 64-bit arithmetic.
template <int VEC, bool kWide, bool kShift>
__device__ __forceinline__ void fetch_row(const float *__restrict__ X, int where, int col, int ldx, float (&x)[VEC])
{
    if constexpr (kWide)
        load_vec<VEC, kShift>(X + col + (int64_t)where * ldx, x);
    else
        load_vec<VEC, kShift>(reinterpret_cast<const float *>(reinterpret_cast<const char *>(X) +
                                                              ((uint32_t)where + (uint32_t)col * 4u)), x);
}

// S non-zeros (o, o + gp, ...) of a row, all gathers issued back to back, added in order into acc; the
// last of them may lie behind the row's end (d).
template <int S, int VEC, bool kWide, bool kShift>
__device__ __forceinline__ void gather_steps(const int2 *row_st, int o, int gp, int d, const float *__restrict__ X, int col,
                                             int ldx, float (&acc)[VEC])
{
    const int last = o + (S - 1) * gp;
    const bool on = last < d;
    int2 p[S];
    float x[S][VEC];
#pragma unroll
    for (int s = 0; s < S; s++) p[s] = row_st[s < S - 1 ? o + s * gp : min(last, d - 1)];
#pragma unroll
    for (int s = 0; s < S; s++) fetch_row<VEC, kWide, kShift>(X, p[s].x, col, ldx, x[s]);
#pragma unroll
    for (int s = 0; s < S; s++) {
        const bool use = s < S - 1 || on;
        const float a = use ? __int_as_float(p[s].y) : 0.0f;
#pragma unroll
        for (int v = 0; v < VEC; v++) acc[v] = fmaf(a, use ? x[s][v] : 0.0f, acc[v]);
    }
}

// One lane group's share of one row: non-zeros k, k + gp, ... of its d pairs, in full batches of four, and
// the rest in as many steps as there are (a gather under a condition of its own per step took as long to
// issue as four).  d and gp are the same for the whole wavefront: the branches are scalar ones.
// Together with the staging above: 114 M non-zeros, N = 64: 1748 -> 1704 us; 4 M next to the diagonal,
// N = 64: 205 -> 192; 8 M, N = 32: 104 -> 91; 208 k, N = 32, back to back: 7.9 -> 7.6.  Several row sets at a time
// (gathers of up to three rows per lane group together) need 64 and more registers: 203 and 103 us.
template <int VEC, bool kWide, bool kShift>
__device__ __forceinline__ void gather_row(const int2 *row_st, int d, int k, int lg, const float *__restrict__ X, int col,
                                           int ldx, float (&acc)[VEC])
{
    static_assert(kUnroll == 4, "the steps of a rest are dealt with one by one");
    const int gp = 1 << lg, full = d >> (lg + 2);
    int o = k;
    for (int i = 0; i < full; i++, o += kUnroll * gp) {
        int2 p[kUnroll];
        float x[kUnroll][VEC];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) p[u] = row_st[o + u * gp];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) fetch_row<VEC, kWide, kShift>(X, p[u].x, col, ldx, x[u]);
#pragma unroll
        for (int u = 0; u < kUnroll; u++)
#pragma unroll
            for (int v = 0; v < VEC; v++) acc[v] = fmaf(__int_as_float(p[u].y), x[u][v], acc[v]);
    }
    switch ((d - full * kUnroll * gp + gp - 1) >> lg) {
    case 1: gather_steps<1, VEC, kWide, kShift>(row_st, o, gp, d, X, col, ldx, acc); break;
    case 2: gather_steps<2, VEC, kWide, kShift>(row_st, o, gp, d, X, col, ldx, acc); break;
    case 3: gather_steps<3, VEC, kWide, kShift>(row_st, o, gp, d, X, col, ldx, acc); break;
    case 4: gather_steps<4, VEC, kWide, kShift>(row_st, o, gp, d, X, col, ldx, acc); break;
    }
}

// v of the lane whose number differs in bit m.
__device__ __forceinline__ float from_lane_xor(float v, int lane, int m)
{
    return __int_as_float(__builtin_amdgcn_ds_bpermute((lane ^ m) << 2, __float_as_int(v)));
}

// Zero-degree rows are the first n_zero_rows rows of the sorted order; the workgroups at
// the head of the grid write them (act(bias) with an epilogue).  They come first so that
// they do not form a tail.
template <int VEC>
__device__ __forceinline__ void zero_fill_rows(const int32_t *__restrict__ perm, float *__restrict__ Y,
                                               int N, int ld, int n_zero_rows,
                                               const float *__restrict__ bias, int relu)
{
    const int rows_here = zero_rows_per_group(N);
    const int r0 = (int)blockIdx.x * rows_here;
    const int n = min(rows_here, n_zero_rows - r0) * N;        // floats of this workgroup
    float fill[VEC];
    for (int i = (int)threadIdx.x * VEC; i < n; i += kWgThreads * VEC) {
        const int r = i / N, c = i - r * N;
        const int64_t out_row = perm ? perm[r0 + r] : r0 + r;
#pragma unroll
        for (int v = 0; v < VEC; v++) {
            float t = bias ? bias[c + v] : 0.0f;                // A X is 0 for this row
            fill[v] = relu ? fmaxf(t, 0.0f) : t;
        }
        store_vec<VEC, false>(Y + out_row * ld + c, fill, N * 4 >= kStreamingMinBytes);
    }
}

// A launch over two column halves (see spmm_launch): the even dies compute columns 0 .. half-1, the
// odd ones the others, and two neighbours go through the workgroups of both their queues in the
// same order.  wg, of n in one half: workgroup of the launch in, workgroup of the plan out.
__device__ __forceinline__ void take_half(int n, int half, int n_split, int &wg, const float *__restrict__ &X,
                                          float *__restrict__ &Y, float *__restrict__ &partial, int &N,
                                          const float *__restrict__ &bias, int *__restrict__ &row_done)
{
    const int die = wg % kXcds, i = wg / kXcds, per_queue = n / kXcds;
    const int second = i >= per_queue;
    wg = (i - (second ? per_queue : 0)) * kXcds + (die & ~1) + second;
    if (die & 1) {
        X += half;
        Y += half;
        partial += half;
        if (row_done) row_done += n_split;           // a counter per row and half
        if (bias) bias += half;
        N -= half;
    } else {
        N = half;
    }
}

// The first 14 words of arguments are in registers when a wavefront starts (see build.py); what the
// way to the first load needs comes first.
template <int L, int VEC, bool kWide, bool kShift>
__global__ __launch_bounds__(kWgThreads) void spmm_gather_kernel(
    const int4 *__restrict__ work, const int32_t *__restrict__ s_idx, const float *__restrict__ s_val,
    const int32_t *__restrict__ perm, int n_units, int n_zero_groups, int half, int N, int ldx, int ld,
    const float *__restrict__ X, float *__restrict__ Y, float *__restrict__ partial, int n_zero_rows,
    const float *__restrict__ bias, int relu, const int32_t *__restrict__ long_slot, int first_split_row,
    int *__restrict__ row_done, int n_split)
{
    // N columns are computed; rows of X are ldx floats apart, those of Y and the partial sums ld
    // (more than N when the launch covers one column panel of a wider operand)
    constexpr int G = 64 / L;        // lane groups per wavefront
    constexpr int CW = L * VEC;      // columns covered per pass
    __shared__ int2 stage[kWaves][kDegBound];

    if ((int)blockIdx.x < n_zero_groups) {
        zero_fill_rows<kShift ? 1 : VEC>(perm, Y, N, ld, n_zero_rows, bias, relu);
        return;
    }

    const int lane = threadIdx.x & 63;
    const int wv = uniform(threadIdx.x >> 6);
    int wg = (int)blockIdx.x - n_zero_groups;
    if (half > 0) take_half(n_units / kWaves, half, n_split, wg, X, Y, partial, N, bias, row_done);
    const int e = wg * kWaves + wv;
    if (e >= n_units) return;

    const int4 b = work[e];
    const int deg = uniform(b.x), row0 = uniform(b.y), loc = uniform(b.z), info = uniform(b.w);
    if (info == 0) return;                              // padding unit
    const bool is_long = deg > kDegBound;
    const int n_rows = is_long ? 1 : (info & 0xFFFF);   // spmm_accel.cu:26
    const int d = is_long ? info : deg;                 // spmm_accel.cu:28: non-zeros per row here
    const int total_nz = n_rows * d;

    // output row of each of the unit's rows, fetched up front (lane r holds row r)
    int my_out = row0 + lane;
    if (!is_long && perm) my_out = perm[row0 + min(lane, n_rows - 1)];

    int2 *st = stage[wv];
    {
        const int32_t *idx = s_idx + loc;
        const float *val = s_val + loc;
        static_assert(kDegBound == 6 * 64, "rounds of staging");
        if (total_nz <= 64) stage_rounds<1, 64, kWide>(idx, val, total_nz, lane, ldx, st);
        else if (total_nz <= 128) stage_rounds<2, 64, kWide>(idx, val, total_nz, lane, ldx, st);
        else if (total_nz <= 192) stage_rounds<3, 64, kWide>(idx, val, total_nz, lane, ldx, st);
        else if (total_nz <= 256) stage_rounds<4, 64, kWide>(idx, val, total_nz, lane, ldx, st);
        else if (total_nz <= 320) stage_rounds<5, 64, kWide>(idx, val, total_nz, lane, ldx, st);
        else stage_rounds<6, 64, kWide>(idx, val, total_nz, lane, ldx, st);
    }
    __builtin_amdgcn_wave_barrier();

    // groups per row: power of two that minimises ceil(n_rows / (G/gp)) * ceil(d / gp)
    int lg = 0;
    if constexpr (G > 1) {
        int best = 0x7fffffff;
#pragma unroll
        for (int q = 0; (1 << q) <= G; q++) {
            const int rows_at_once = G >> q;
            const int steps = ((n_rows + rows_at_once - 1) / rows_at_once) * ((d + (1 << q) - 1) >> q);
            if (steps < best) { best = steps; lg = q; }
        }
    }
    const int gp = 1 << lg;
    const int rows_at_once = G >> lg;
    const int g = lane / L, sub = lane % L;
    const int k = g & (gp - 1);          // which of the row's gp groups this is
    const int rloc = g >> lg;            // which of the rows in flight

    const bool streaming = N * 4 >= kStreamingMinBytes;
    for (int c0 = 0; c0 < N; c0 += CW) {
        int col = c0 + sub * VEC;
        const bool col_ok = col < N;
        if (kShift && col + VEC > N) col = N - VEC;   // the row's last vector ends with the row
        for (int r_it = 0; r_it < n_rows; r_it += rows_at_once) {
            const int r = r_it + rloc;
            const bool live = col_ok && r < n_rows;
            float acc[VEC];
#pragma unroll
            for (int v = 0; v < VEC; v++) acc[v] = 0.0f;
            if (live) gather_row<VEC, kWide, kShift>(st + r * d, d, k, lg, X, col, ldx, acc);
            // add the gp partial sums of each row (all lanes take part)
            for (int m = L; m < (L << lg); m <<= 1) {
#pragma unroll
                for (int v = 0; v < VEC; v++) acc[v] += from_lane_xor(acc[v], lane, m);
            }
            const int64_t out_row = __shfl(my_out, r < n_rows ? r : 0);
            if (live && k == 0) {
                if (is_long) {
                    float *p = partial + (int64_t)(deg - (kDegBound + 1)) * ld + col;
                    if (row_done) store_partial<VEC>(p, acc);
                    else store_vec<VEC, kShift>(p, acc, streaming);
                } else {
                    if (bias) {
#pragma unroll
                        for (int v = 0; v < VEC; v++) acc[v] += bias[col + v];
                    }
                    if (relu) {
#pragma unroll
                        for (int v = 0; v < VEC; v++) acc[v] = fmaxf(acc[v], 0.0f);
                    }
                    store_vec<VEC, kShift>(Y + out_row * ld + col, acc, streaming);
                }
            }
        }
    }
    // The wavefront that stores a split row's last piece adds the row up, in this launch
    // (row_done: one counter per split row; null: a second kernel does it).
    if (is_long && row_done) {
        const int lr = row0 - first_split_row;
        const int first = long_slot[lr], nseg = long_slot[lr + 1] - first;
        int *flag = reinterpret_cast<int *>(st);             // the staged pairs are no longer needed
        if (last_piece_of_row<64>(row_done + lr, nseg, lane, flag)) {
            const int64_t out_row = perm ? perm[row0] : row0;
            finish_split_row<64>(partial + (int64_t)first * ld, nseg, Y + out_row * ld, N, ld, bias, relu, lane,
                                 reinterpret_cast<float *>(st) + 64);
        }
    }
}

// The same computation with one unit per workgroup: the four wavefronts form 4 * G lane
// groups that share the unit's rows, or its row's non-zeros.  When a row's groups span
// several wavefronts their sums meet in LDS.  Used for small matrices, where the time of
// a launch is the longest chain of dependent gathers in one wavefront: the chain is four
// times shorter and rows of up to one unit need no partial sums.
template <int L, int VEC, bool kWide, bool kShift>
__global__ __launch_bounds__(kWgThreads) void spmm_team_kernel(
    const int4 *__restrict__ work, const int32_t *__restrict__ s_idx, const float *__restrict__ s_val,
    const int32_t *__restrict__ perm, int n_units, int n_zero_groups, int N, int ldx, const float *__restrict__ X,
    float *__restrict__ Y, int ld, float *__restrict__ partial, int n_zero_rows,
    const float *__restrict__ bias, int relu, const int32_t *__restrict__ long_slot, int first_split_row,
    int *__restrict__ row_done)
{
    constexpr int G = 64 / L;        // lane groups per wavefront
    constexpr int TG = G * kWaves;   // lane groups per workgroup
    constexpr int CW = L * VEC;      // columns covered per pass
    __shared__ int2 stage[2 * kWgThreads];
    __shared__ float meet[kWaves][CW];

    if ((int)blockIdx.x < n_zero_groups) {
        zero_fill_rows<kShift ? 1 : VEC>(perm, Y, N, ld, n_zero_rows, bias, relu);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int wv = uniform(threadIdx.x >> 6);
    const int e = (int)blockIdx.x - n_zero_groups;
    if (e >= n_units) return;
    const int4 b = work[e];
    const int deg = uniform(b.x), row0 = uniform(b.y), loc = uniform(b.z), info = uniform(b.w);
    if (info == 0) return;                              // padding unit (the whole workgroup leaves)
    const bool is_long = deg > kDegBound;
    const int n_rows = is_long ? 1 : (info & 0xFFFF);
    const int d = is_long ? info : deg;
    const int total_nz = n_rows * d;

    int my_out = row0 + lane;
    if (!is_long && perm && lane < n_rows) my_out = perm[row0 + lane];

    // stage the unit's (column, value) pairs: one round of the workgroup, or two
    static_assert(kDegBound <= 2 * kWgThreads, "rounds of staging");
    if (total_nz > kWgThreads)
        stage_rounds<2, kWgThreads, kWide>(s_idx + loc, s_val + loc, total_nz, (int)threadIdx.x, ldx, stage);
    else if ((int)threadIdx.x < total_nz)
        stage_rounds<1, kWgThreads, kWide>(s_idx + loc, s_val + loc, total_nz, (int)threadIdx.x, ldx, stage);
    __syncthreads();

    // groups per row: power of two that minimises ceil(n_rows / (TG/gp)) * ceil(d / gp)
    int lg = 0;
    {
        int best = 0x7fffffff;
#pragma unroll
        for (int q = 0; (1 << q) <= TG; q++) {
            const int rows_at_once = TG >> q;
            const int steps = ((n_rows + rows_at_once - 1) / rows_at_once) * ((d + (1 << q) - 1) >> q);
            if (steps < best) { best = steps; lg = q; }
        }
    }
    const int gp = 1 << lg;
    const int rows_at_once = TG >> lg;
    const int g = lane / L, sub = lane % L;
    const int vg = wv * G + g;           // this lane group among the workgroup's
    const int k = vg & (gp - 1);         // which of the row's gp groups this is
    const int rloc = vg >> lg;           // which of the rows in flight
    const int in_wave = gp < G ? gp : G;             // groups of one row inside a wavefront
    const int waves_per_row = gp > G ? gp / G : 1;   // > 1: the row's sums meet in LDS

    for (int c0 = 0; c0 < N; c0 += CW) {
        int col = c0 + sub * VEC;
        const bool col_ok = col < N;
        if (kShift && col + VEC > N) col = N - VEC;   // the row's last vector ends with the row
        for (int r_it = 0; r_it < n_rows; r_it += rows_at_once) {
            const int r = r_it + rloc;
            const bool live = col_ok && r < n_rows;
            float acc[VEC];
#pragma unroll
            for (int v = 0; v < VEC; v++) acc[v] = 0.0f;
            if (live) gather_row<VEC, kWide, kShift>(stage + r * d, d, k, lg, X, col, ldx, acc);
            // the row's groups inside this wavefront (all lanes take part)
            for (int m = L; m < L * in_wave; m <<= 1) {
#pragma unroll
                for (int v = 0; v < VEC; v++) acc[v] += from_lane_xor(acc[v], lane, m);
            }
            if (waves_per_row > 1) {                 // workgroup-uniform
                if (g == 0) {
#pragma unroll
                    for (int v = 0; v < VEC; v++) meet[wv][sub * VEC + v] = acc[v];
                }
                __syncthreads();
                if (wv % waves_per_row == 0 && g == 0) {
                    for (int q = 1; q < waves_per_row; q++) {
#pragma unroll
                        for (int v = 0; v < VEC; v++) acc[v] += meet[wv + q][sub * VEC + v];
                    }
                }
                __syncthreads();
            }
            const int64_t out_row = __shfl(my_out, r < n_rows ? r : 0);
            if (live && k == 0) {
                if (is_long) {
                    float *p = partial + (int64_t)(deg - (kDegBound + 1)) * ld + col;
                    if (row_done) store_partial<VEC>(p, acc);
                    else store_vec<VEC, kShift>(p, acc, false);
                } else {
                    if (bias) {
#pragma unroll
                        for (int v = 0; v < VEC; v++) acc[v] += bias[col + v];
                    }
                    if (relu) {
#pragma unroll
                        for (int v = 0; v < VEC; v++) acc[v] = fmaxf(acc[v], 0.0f);
                    }
                    store_vec<VEC, kShift>(Y + out_row * ld + col, acc, N * 4 >= kStreamingMinBytes);
                }
            }
        }
    }
    // the workgroup that stores a split row's last piece adds the row up (see the gather kernel)
    if (is_long && row_done) {                       // workgroup-uniform
        const int lr = row0 - first_split_row;
        const int first = long_slot[lr], nseg = long_slot[lr + 1] - first;
        __syncthreads();                             // every wavefront is done with the staged pairs
        int *flag = reinterpret_cast<int *>(stage);
        if (last_piece_of_row<kWgThreads>(row_done + lr, nseg, (int)threadIdx.x, flag)) {
            const int64_t out_row = perm ? perm[row0] : row0;
            finish_split_row<kWgThreads>(partial + (int64_t)first * ld, nseg, Y + out_row * ld, N, ld, bias, relu,
                                         (int)threadIdx.x, reinterpret_cast<float *>(stage) + 64);
        }
    }
}

// Adds the partial sums of each split row in slot order and writes the row.
// The first n_shared_groups workgroups take rpw rows each (256 / rpw threads per
// row): rows with few slots and few columns do not need a whole workgroup.  The
// remaining workgroups take one row each: the rows with very many slots.
// A thread covers VEC consecutive columns (VEC = 4: one 16-byte load per slot, when N and
// the row stride are multiples of 4 and the operands 16-byte aligned; else VEC = 1); NV = the
// row's columns counted in such vectors.
template <int VEC>
__global__ __launch_bounds__(kReduceThreads) void long_row_reduce_kernel(
    const float *__restrict__ partial, const int32_t *__restrict__ long_slot,
    const int32_t *__restrict__ perm, int64_t first_split_row, int n_shared_rows, int n_shared_groups,
    int rpw, int n_rows, float *__restrict__ Y, int NV, int ld, const float *__restrict__ bias, int relu)
{
    // rows of Y and of the partial sums are ld floats apart
    __shared__ float red[kReduceThreads][VEC];
    const bool shared_group = (int)blockIdx.x < n_shared_groups;
    const int T = shared_group ? kReduceThreads / rpw : kReduceThreads;   // threads per row
    const int sub_row = threadIdx.x / T, t = threadIdx.x % T;
    const int lr = shared_group ? (int)blockIdx.x * rpw + sub_row
                                : n_shared_rows + ((int)blockIdx.x - n_shared_groups);
    const bool row_ok = lr < (shared_group ? n_shared_rows : n_rows);
    const int first = row_ok ? long_slot[lr] : 0;
    const int nseg = row_ok ? long_slot[lr + 1] - first : 0;
    const float *src = partial + (int64_t)first * ld;
    const int64_t r = first_split_row + lr;
    const int64_t out_row = row_ok ? (perm ? perm[r] : r) : 0;
    int cw = 1;                                    // vectors per pass: power of two <= T
    while (cw < NV && cw < T) cw <<= 1;
    const int sg = T / cw;                         // slot groups
    const int c_in = t % cw, my_sg = t / cw;
    for (int c0 = 0; c0 < NV; c0 += cw) {
        const int c = (c0 + c_in) * VEC;           // first column of this thread's vector
        const bool col_ok = c0 + c_in < NV;
        float acc[VEC];
#pragma unroll
        for (int v = 0; v < VEC; v++) acc[v] = 0.0f;
        if (col_ok) {
            int sgm = my_sg;
            for (; sgm + 7 * sg < nseg; sgm += 8 * sg) {       // eight loads in flight, added in order
                float x[8][VEC];
#pragma unroll
                for (int u = 0; u < 8; u++) load_vec<VEC, false>(src + (int64_t)(sgm + u * sg) * ld + c, x[u]);
#pragma unroll
                for (int u = 0; u < 8; u++)
#pragma unroll
                    for (int v = 0; v < VEC; v++) acc[v] += x[u][v];
            }
            for (; sgm < nseg; sgm += sg) {
                float x[VEC];
                load_vec<VEC, false>(src + (int64_t)sgm * ld + c, x);
#pragma unroll
                for (int v = 0; v < VEC; v++) acc[v] += x[v];
            }
        }
        if (sg > 1) {                              // uniform over the workgroup's rows of one kind
#pragma unroll
            for (int v = 0; v < VEC; v++) red[threadIdx.x][v] = acc[v];
            __syncthreads();
            if (my_sg == 0)
                for (int q = 1; q < sg; q++)
#pragma unroll
                    for (int v = 0; v < VEC; v++) acc[v] += red[sub_row * T + q * cw + c_in][v];
            __syncthreads();
        }
        if (row_ok && my_sg == 0 && col_ok) {
            if (bias) {
#pragma unroll
                for (int v = 0; v < VEC; v++) acc[v] += bias[c + v];
            }
            if (relu) {
#pragma unroll
                for (int v = 0; v < VEC; v++) acc[v] = fmaxf(acc[v], 0.0f);
            }
            store_vec<VEC, false>(Y + out_row * ld + c, acc, false);
        }
    }
}

__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t *dst, uint32_t v, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = v;
}

__global__ __launch_bounds__(256) void copy_u32_kernel(uint32_t *__restrict__ dst,
                                                       const uint32_t *__restrict__ src, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = src[i];
}

// Copies rows of N floats, ld apart, to rows ldx apart (a multiple of 16, with zeros behind the N):
// 64 rows per workgroup, four 16-byte vectors per thread on their way.  Bound by memory: 5.8 to 6.7
// TB/s of reads and writes on 2.45 M rows of 25 to 127 floats (4.5 at 14).  The copy is written with
// ordinary stores, since the gather that follows reads it.
__global__ __launch_bounds__(kWgThreads) void pad_rows_kernel(const float *__restrict__ X, int64_t rows, int N, int64_t ld,
                                                              float *__restrict__ out, int ldx)
{
    const int64_t row0 = (int64_t)blockIdx.x * kPadRows;
    const int n_rows = (int)min((int64_t)kPadRows, rows - row0);
    const int per_row = ldx / 4, n = n_rows * per_row;
    const float *src = X + row0 * ld;
    v4f *dst = reinterpret_cast<v4f *>(out + row0 * ldx);
    const uint32_t inverse = 0xFFFFFFFFu / (uint32_t)per_row + 1;     // exact for i < 2^16, per_row <= 128
    constexpr int U = 4;
    for (int i0 = threadIdx.x; i0 < n; i0 += U * kWgThreads) {
        v4f t[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = i0 + u * kWgThreads, r = (int)__umulhi((uint32_t)i, inverse), c = (i - r * per_row) * 4;
            const bool on = i < n && c < N;
            // a row's last vector is taken from where it ends with the row, and moved down
            const int back = on ? max(c + 4 - N, 0) : 0;
            const v4f q = __builtin_nontemporal_load(
                reinterpret_cast<const v4f_unaligned *>(src + (on ? r * ld + c - back : 0)));
            t[u].x = !on ? 0.0f : back == 0 ? q.x : back == 1 ? q.y : back == 2 ? q.z : q.w;
            t[u].y = !on || back == 3 ? 0.0f : back == 0 ? q.y : back == 1 ? q.z : q.w;
            t[u].z = !on || back >= 2 ? 0.0f : back == 0 ? q.z : q.w;
            t[u].w = !on || back >= 1 ? 0.0f : q.w;
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i0 + u * kWgThreads < n) dst[i0 + u * kWgThreads] = t[u];
    }
}

struct LaunchArgs {
    bool team;
    dim3 grid;
    hipStream_t stream;
    const int4 *work;
    int n_units;
    const int32_t *s_idx;
    const float *s_val;
    const int32_t *perm;
    const float *X;
    float *Y;
    float *partial;
    int N, ldx, ld, n_zero_rows, n_zero_groups;
    const float *bias;
    int relu;
    const int32_t *long_slot;
    int first_split_row;
    int *row_done;
    int half, n_split;
    // events bound to this launch itself (its start and its end), or null: unlike an event
    // recorded behind the launch they put no packet of their own into the queue
    hipEvent_t start_ev, stop_ev;
};

template <int L, int VEC, bool kWide, bool kShift>
void launch_one(const LaunchArgs &a)
{
    // (a launch with events costs the host more than one without)
    auto launch = [&](auto kernel, auto... args) {
        if (a.start_ev || a.stop_ev)
            hipExtLaunchKernelGGL(kernel, a.grid, dim3(kWgThreads), 0, a.stream, a.start_ev, a.stop_ev, 0, args...);
        else
            kernel<<<a.grid, dim3(kWgThreads), 0, a.stream>>>(args...);
    };
    if (a.team)
        launch(spmm_team_kernel<L, VEC, kWide, kShift>, a.work, a.s_idx, a.s_val, a.perm, a.n_units, a.n_zero_groups, a.N,
               a.ldx, a.X, a.Y, a.ld, a.partial, a.n_zero_rows, a.bias, a.relu, a.long_slot, a.first_split_row,
               a.row_done);
    else
        launch(spmm_gather_kernel<L, VEC, kWide, kShift>, a.work, a.s_idx, a.s_val, a.perm, a.n_units, a.n_zero_groups,
               a.half, a.N, a.ldx, a.ld, a.X, a.Y, a.partial, a.n_zero_rows, a.bias, a.relu, a.long_slot,
               a.first_split_row, a.row_done, a.n_split);
}

// Lane-group widths: 1..64 lanes of one 16-byte vector each; scalar lanes only serve N < 4.
template <int VEC, bool kWide, bool kShift>
int launch_for_width(int L, const LaunchArgs &a)
{
    switch (L) {
    case 1: launch_one<1, VEC, kWide, kShift>(a); break;
    case 2: launch_one<2, VEC, kWide, kShift>(a); break;
    case 4: launch_one<4, VEC, kWide, kShift>(a); break;
    default:
        if constexpr (VEC == 4) {
            switch (L) {
            case 8: launch_one<8, VEC, kWide, kShift>(a); return ACCEL_OK;
            case 16: launch_one<16, VEC, kWide, kShift>(a); return ACCEL_OK;
            case 32: launch_one<32, VEC, kWide, kShift>(a); return ACCEL_OK;
            case 64: launch_one<64, VEC, kWide, kShift>(a); return ACCEL_OK;
            }
        }
        set_error("internal: unsupported group width %d", L);
        return ACCEL_ERR_ARG;
    }
    return ACCEL_OK;
}

// mode: 0 = 16-byte vectors at 16-byte aligned addresses, 1 = 16-byte vectors at any
// 4-byte aligned address with the row's last vector shifted to end with the row,
// 2 = scalar lanes
int launch_for_mode(int mode, bool wide, int L, const LaunchArgs &a)
{
    if (mode == 0) return wide ? launch_for_width<4, true, false>(L, a) : launch_for_width<4, false, false>(L, a);
    if (mode == 1) return wide ? launch_for_width<4, true, true>(L, a) : launch_for_width<4, false, true>(L, a);
    return wide ? launch_for_width<1, true, false>(L, a) : launch_for_width<1, false, false>(L, a);
}

}  // namespace

int fill_u32(void *dst, uint32_t v, size_t n, hipStream_t s)
{
    if (n == 0) return ACCEL_OK;
    const unsigned g = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
    fill_u32_kernel<<<dim3(g), dim3(256), 0, s>>>(static_cast<uint32_t *>(dst), v, n);
    ACCEL_HIP(hipGetLastError());
    return ACCEL_OK;
}

int copy_u32(void *dst, const void *src, size_t n, hipStream_t s)
{
    if (n == 0) return ACCEL_OK;
    const unsigned g = (unsigned)std::min<size_t>((n + 255) / 256, 65536);
    copy_u32_kernel<<<dim3(g), dim3(256), 0, s>>>(static_cast<uint32_t *>(dst),
                                                  static_cast<const uint32_t *>(src), n);
    ACCEL_HIP(hipGetLastError());
    return ACCEL_OK;
}

// Device address of this GPU's copy of `scratch`, looked up once per device (with that
// device current) and kept.
static int static_scratch_address(float **out)
{
    static std::mutex mu;
    static float *addr[kMaxScratchDevices] = {};
    int dev = 0;
    ACCEL_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxScratchDevices) {
        set_error("device ordinal %d is beyond the %d devices the static scratch is tracked for", dev,
                  kMaxScratchDevices);
        return ACCEL_ERR_ARG;
    }
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        float *p = nullptr;
        ACCEL_HIP(hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(scratch)));
        addr[dev] = p;
    }
    *out = addr[dev];
    return ACCEL_OK;
}

// Grows the handle's partial-sum buffer to `floats` (never shrinks).  The old buffer is
// given back: graphs captured with it must be captured again.
int reserve_partial(accel_handle *h, size_t floats, bool any_stream)
{
    if (h->partial_floats >= floats) return ACCEL_OK;
    if (h->partial) give_memory(h->partial, wait_for_device());      // nobody reads the old one
    h->partial_floats = 0;
    h->partial = static_cast<float *>(take_memory(floats * sizeof(float), any_stream));
    if (!h->partial) {
        set_error("device allocation of %zu bytes for long-row partial sums failed", floats * sizeof(float));
        return ACCEL_ERR_ALLOC;
    }
    h->partial_floats = floats;
    return ACCEL_OK;
}

// 128-byte lines that a row of N floats touches on average, rows ld floats apart from address x on.
static double lines_per_row(uintptr_t x, int N, int64_t ld)
{
    const unsigned stride = (unsigned)(ld * 4 % 128);
    unsigned step = 128;                              // the rows' places in a line are x, x + step, ...
    while (stride % step) step /= 2;
    int lines = 0, n = 0;
    for (unsigned at = (unsigned)(x % step); at < 128; at += step, n++) lines += (int)((at + 4u * (unsigned)N + 127) / 128);
    return (double)lines / n;
}

// Row stride, in floats, at which a gathered row touches as few lines as it can.
static int whole_lines(int N) { return N <= 16 ? 16 : (N + 31) / 32 * 32; }

// Seconds that a run saves when every row of X starts on a line instead of at x + i * ld.
//
// A gather is bound by the lines it pulls through the L2s, so what counts is how many of them are
// saved: Gathered * lines / 7.2 TB/s if all of them missed.  Measured share of that (rows padded by
// the caller against packed ones, power-law graphs of 8 to 125 M non-zeros): 0.4 at N = 14, 0.55 at
// 25, 0.6 at 50, 0.8 at 90, 1.0 at 127; less when X nearly fits the L2s (X of 10 MB: a third);
// 0.1 to 0.16 for a matrix whose non-zeros lie near the diagonal, where the rows share their lines.
static double saved_by_padding(const accel_handle *h, uintptr_t x, int N, int64_t ld)
{
    if (N <= 8) return 0.0;                           // a padded row would take up twice the cache and more
    double lines = lines_per_row(x, N, ld) - lines_per_row(0, N, whole_lines(N));
    const double mb = 4e-6 * (double)h->cols * N;
    // rows of whole lines can also be computed in column panels (see spmm_launch): a twelfth less
    // where X is not many times what the L2s hold
    if (N > kPanel && N % kPanel != 0 && whole_lines(N) % kPanel == 0)
        lines += whole_lines(N) / (32 * 12.0) * std::min(1.0, 100 / mb);
    const double share = h->local ? 0.1 : std::min(1.0, 0.4 + 0.005 * N) * std::min(1.0, mb / 32);
    return (double)h->nnz * lines * 128 / 7.2e12 * share;
}

// Stride at which a run with N columns wants the rows of an X that nobody has laid out yet: padded
// to whole lines if that saves more than writing and fetching the padding costs.
int row_stride(const accel_handle *h, int N)
{
    const double more = 8.0 * (double)h->cols * (whole_lines(N) - N) / 5e12;
    return saved_by_padding(h, 0, N, N) > more ? whole_lines(N) : N;
}

// Whether a run copies X to padded rows first: it has to save more than the copy (one pass over X
// at 5 TB/s, and a launch), with a fifth to spare.  That is graphs of some ten or more non-zeros per
// row and column counts that packed rows suit badly.  Measured, whole runs, 2.45 M rows and 125 M
// non-zeros: N = 25: 2.77 -> 1.92 ms (copy 0.09),
// N = 50: 4.29 -> 3.67 (0.17), N = 127: 9.40 -> 7.54 (0.43); 8 M non-zeros in 400 k rows, N = 25: 181
// -> 143 us, N = 50: 278 -> 275.
static bool pads_x(const accel_handle *h, uintptr_t x, int N, int64_t ld)
{
    if (N > kPadMaxN || (size_t)h->cols * (size_t)whole_lines(N) > kPadMaxFloats) return false;
    const double saved = saved_by_padding(h, x, N, ld);
    return saved > 5e-6 && saved > 1.2 * (4e-6 + 4.0 * (double)h->cols * (N + whole_lines(N)) / 5e12);
}

// Room for X in padded rows, kept by the handle.  Not had: no error, the run takes X as it lies.
static bool room_for_rows(accel_handle *h, size_t floats, bool any_stream)
{
    if (h->x_rows_floats >= floats) return true;
    if (h->x_rows) give_memory(h->x_rows, wait_for_device());      // nobody reads the old one
    h->x_rows_floats = 0;
    h->x_rows = static_cast<float *>(take_memory(floats * sizeof(float), any_stream));
    if (!h->x_rows) {
        (void)hipGetLastError();
        return false;
    }
    h->x_rows_floats = floats;
    return true;
}

// All that a run with up to max_N columns allocates.
int reserve_run(accel_handle *h, int max_N)
{
    if (int rc = reserve_partial(h, (size_t)h->n_long_units * (size_t)max_N, true)) return rc;
    h->reserved_N = std::max(h->reserved_N, max_N);
    size_t floats = 0;
    for (int N = std::min(max_N, kPadMaxN); N > 0 && floats == 0; N--)
        if (pads_x(h, 0, N, N)) floats = (size_t)h->cols * (size_t)whole_lines(N);
    if (floats > 0) (void)room_for_rows(h, floats, true);
    return ACCEL_OK;
}

// main_start / main_stop: events bound to the gather kernel (to the first and the last launch
// when the run is done in column panels), for timing it alone.
int spmm_launch(accel_handle *h, const float *X, float *Y, int N, hipStream_t stream,
                hipEvent_t main_start, hipEvent_t main_stop, const float *bias, int relu, bool static_partial,
                int ld, int ldx)
{
    if (h->rows == 0) return ACCEL_OK;
    (void)hipGetLastError();                         // launch errors are read back below: start from a clean slate
    if (ld <= 0) ld = N;                             // rows of Y are ld floats apart
    if (ldx <= 0) ldx = ld;                          // those of X ldx
    // partial sums of the pieces of split rows: the handle's buffer (allocated here when a
    // run needs more than it holds), or this GPU's static array, which is never allocated
    float *partial = h->partial;
    const bool uses_handle_partial = !static_partial && h->n_long_units > 0;
    // the capture status is only asked for where something depends on it: a buffer that would
    // have to grow, or a stream the handle would have to order against another
    const bool must_grow = uses_handle_partial && h->partial_floats < (size_t)h->n_long_units * (size_t)ld;
    const bool best_padded = pads_x(h, reinterpret_cast<uintptr_t>(X), N, ldx);
    bool pad = best_padded && !static_partial;
    const bool capturing = (must_grow || pad || needs_capture_status(h, stream)) && stream_is_capturing(stream);
    if (static_partial) {
        partial = nullptr;
        const size_t need = (size_t)h->n_long_units * (size_t)ld;
        if (need > kStaticScratchFloats) {
            set_error("accel_run_static: this matrix needs %zu floats of partial sums at N = %d "
                      "(%lld pieces of split rows x N), the static scratch holds %zu",
                      need, N, (long long)h->n_long_units, kStaticScratchFloats);
            return ACCEL_ERR_ARG;
        }
        if (need > 0)
            if (int rc = static_scratch_address(&partial)) return rc;
    } else if (uses_handle_partial) {
        const size_t need = (size_t)h->n_long_units * (size_t)ld;
        if (h->partial_floats < need) {
            if (capturing) {
                set_error("the partial-sum buffer has to grow for N = %d and the stream is capturing: "
                          "call accel_reserve(h, N) before the capture", N);
                return ACCEL_ERR_STATE;
            }
            if (int rc = reserve_partial(h, need, stream != nullptr)) return rc;
        }
        partial = h->partial;
    }
    // X copied to padded rows.  Not while capturing: the graph would keep the address of a buffer
    // that a later run may replace.
    if (pad) {
        const size_t need = (size_t)h->cols * (size_t)whole_lines(N);
        pad = !capturing &&
              (h->x_rows_floats >= need || (N > h->reserved_N && room_for_rows(h, need, stream != nullptr)));
    }
    // The buffer is shared by all runs of this handle, and a value update may still be
    // rewriting what this run reads: a run on another stream than the one that used them
    // last waits for that stream on the device (runs queued on one stream are ordered anyway).
    hipEvent_t run_done = nullptr;                  // to be bound to the run's last kernel
    if (int rc = order_run(h, stream, uses_handle_partial || pad, capturing, &run_done)) return rc;
    // What decides how the sums are grouped (panels and halves below, the vectors of the second kernel)
    // is the same whether X has been copied or not: a run that could not (capturing, static, no memory) gives
    // the bits of one that did.  (It pays for that where the copy would have put N = 97..127, 161..191, 225..255
    // on whole lines: two panels of packed rows both take the line they meet in.  125 M non-zeros, captured, one
    // pass and two panels: N = 127 9.19 and 10.40 ms, N = 191 12.8 and 15.2; 2.45 M, N = 127: 193 and 202 us.
    // One pass in lane groups as narrow as a panel's, which adds up in the same order, takes 10.46 and 16.1 ms.)
    const uintptr_t at_x = reinterpret_cast<uintptr_t>(X), at_y = reinterpret_cast<uintptr_t>(Y);
    const bool whole_rows = ldx % 32 == 0 || best_padded;
    const bool y_vectors = N % 4 == 0 && ld % 4 == 0 && at_y % 16 == 0;
    const bool vectors = y_vectors && ((ldx % 4 == 0 && at_x % 16 == 0) || best_padded);
    if (pad) {
        const int to = whole_lines(N);
        const dim3 grid((unsigned)((h->cols + kPadRows - 1) / kPadRows));
        pad_rows_kernel<<<grid, dim3(kWgThreads), 0, stream>>>(X, (int64_t)h->cols, N, (int64_t)ldx, h->x_rows, to);
        X = h->x_rows;
        ldx = to;
    }
    // 16-byte vectors whenever a row holds one.  When N is not a multiple of 4, or X or Y
    // is not 16-byte aligned, rows start at odd multiples of 4 bytes: the vectors are then
    // loaded and stored at 4-byte aligned addresses, and a row's last vector is moved back
    // so that it ends with the row (it overlaps the one before; both lanes hold the same
    // sums for the shared columns).  Scalar lanes are left for N < 4.
    const int mode = N < 4 ? 2 : (y_vectors && ldx % 4 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0) ? 0 : 1;
    const int vec = mode == 2 ? 1 : 4;
    // split rows are added up by the gather kernel itself (the wavefront that stores a row's
    // last piece), or, when the handle has no counters for that, by a second kernel
    int *row_done = h->fused_reduce ? h->row_done : nullptr;
    const bool has_reduce = h->n_split_rows > 0 && !row_done;
    // Wide operands are computed one column panel at a time (all units for the first
    // panel, then all units for the next): a panel's slice of X is what the L2s have
    // to hold, and a narrower slice means more rows of X fit.
    // Measured (panel 64 against one pass): N = 256 on the hub graph -12 %, N = 128 on the
    // dense and the power-law 100 M-non-zero graphs -7 % and -4 %; no gain when the
    // columns have no popularity skew or the rows are very short, and a loss when N is
    // not a multiple of the panel (N = 100: 64 + 36 leaves lanes idle).  Rows that lie on whole
    // lines count as wide as their lines: N = 127 at a stride of 128, 125 M non-zeros: -5 %.
    int panel = N;
    const int want = h->plan_panel_option > 0 ? h->plan_panel_option : kPanel;
    const bool forced = h->plan_panel_option > 0;
    const bool even = (vectors && N % want == 0) ||                         // panels of whole lines
                      (mode != 2 && whole_rows && whole_lines(N) % want == 0);
    if (N > want &&
        ((forced && vectors) || (!forced && even && h->nnz >= kPanelMinNnz && h->nnz >= 16 * h->rows)))
        panel = want;
    // With more than one panel, two neighbouring panels are computed in one launch, each by every
    // other die: a die then sees twice the units but half of every row of X, so that what it fetches
    // into its L2 serves twice the gathers.  Also where several launches would not pay.  Measured at
    // N = 128 / 256: 1.5 M non-zeros in 50 k rows 77 -> 62 / 172 -> 126 us, 2.4 M in 170 k 139 -> 126 /
    // 302 -> 258, 10 M in 1 M 724 -> 695 / 1471 -> 1400, 114 M in 233 k 3.46 -> 3.32 / 6.94 -> 6.60 ms,
    // 125 M in 2.45 M 7.00 -> 6.92 / 14.4 -> 13.8; five per row 389 -> 391 / 808.  Halves of 32 columns
    // at N = 64 lose (3.40 -> 3.57 ms on the last): as much staging for half the lines.  So do workgroup
    // units (208 k non-zeros: 12.2 -> 15.1 us), which are bound by latency.  Both dies go through the
    // same queue at the same time: through different ones is 5 to 10 % slower.
    const bool halves = even && !forced && N > want && !h->plan_team && h->plan_queues == kXcds;
    // operands below 4 GiB are addressed with 32-bit byte offsets (see gather_row)
    const bool wide = (uint64_t)h->cols * (uint64_t)ldx * 4u > 0xFFFFFFFFull;
    const int4 *wk = reinterpret_cast<const int4 *>(h->work);
    const int64_t entry_groups = h->plan_team ? h->n_units : h->n_units / kWaves;
    for (int c0 = 0, n; c0 < N; c0 += n) {
        const int half = halves && N - c0 > want ? want : 0;
        n = half ? std::min(2 * half, N - c0) : std::min(panel, N - c0);
        int L = 1;                                   // lanes per row: one per vector, a power of two
        while (L * vec < (half ? half : n) && L < 64) L <<= 1;
        // zero-fill workgroups come first; their count is rounded up to a multiple of the
        // queue count so that entry group i still lands on die i % 8 (surplus ones exit at once)
        const int zr = zero_rows_per_group(n);
        int64_t zero_groups = (h->n_zero_rows + zr - 1) / zr;
        zero_groups = (zero_groups + h->plan_queues - 1) / h->plan_queues * h->plan_queues;
        const int64_t groups = entry_groups * (half ? 2 : 1) + zero_groups;
        if (groups > 0x7fffffffLL) {
            set_error("launch of %lld workgroups exceeds the grid limit", (long long)groups);
            return ACCEL_ERR_ARG;
        }
        if (groups == 0) break;
        const dim3 grid((unsigned)groups);
        const float *Xp = X ? X + c0 : X;
        float *Yp = Y + c0, *Pp = partial ? partial + c0 : nullptr;
        const float *bp = bias ? bias + c0 : nullptr;
        const bool first = c0 == 0, last = c0 + n >= N;
        hipEvent_t stop = last ? main_stop : nullptr;
        if (last && !stop && !has_reduce) stop = run_done;      // the run ends with this launch
        const LaunchArgs la{h->plan_team, grid, stream, wk, (int)h->n_units, h->s_idx, h->s_val, h->perm,
                            Xp, Yp, Pp, n, ldx, ld, (int)h->n_zero_rows, (int)zero_groups, bp, relu,
                            h->long_slot, (int)(h->rows - h->n_split_rows), row_done, half, (int)h->n_split_rows,
                            first ? main_start : nullptr, stop};
        const int rc = launch_for_mode(mode, wide, L, la);
        if (rc) return rc;
    }
    if (!has_reduce && run_done && main_stop)       // the one launch cannot carry both events
        ACCEL_HIP(hipEventRecord(run_done, stream));
    if (has_reduce) {
        // one launch: rows with very many slots (the last n_big rows) get a workgroup each, the
        // others share one: as many rows per workgroup as leaves a row one thread per vector
        // of columns (16 at least, so that a row's loads stay coalesced)
        const int n_split = (int)h->n_split_rows, n_big = (int)h->n_big_rows, n_shared = n_split - n_big;
        const int rvec = y_vectors ? 4 : 1;          // 16-byte accesses
        const int nv = (N + rvec - 1) / rvec;
        int threads_per_row = 16;
        while (threads_per_row < nv && threads_per_row < kReduceThreads) threads_per_row <<= 1;
        const int rpw = kReduceThreads / threads_per_row;
        const int shared_groups = (n_shared + rpw - 1) / rpw;
        const dim3 rgrid((unsigned)(shared_groups + n_big));
        auto kernel = rvec == 4 ? long_row_reduce_kernel<4> : long_row_reduce_kernel<1>;
        if (run_done)
            hipExtLaunchKernelGGL(kernel, rgrid, dim3(kReduceThreads), 0, stream, nullptr, run_done,
                                  0, (const float *)partial, (const int32_t *)h->long_slot, (const int32_t *)h->perm,
                                  (int64_t)(h->rows - h->n_split_rows), n_shared, shared_groups, rpw, n_split, Y, nv,
                                  ld, bias, relu);
        else
            kernel<<<rgrid, dim3(kReduceThreads), 0, stream>>>(
                partial, h->long_slot, h->perm, h->rows - h->n_split_rows, n_shared, shared_groups, rpw,
                n_split, Y, nv, ld, bias, relu);
    }
    ACCEL_HIP(hipGetLastError());
    return ACCEL_OK;
}

}  // namespace accel
