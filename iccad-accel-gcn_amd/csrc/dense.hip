// Z = X * W in fp32 on the bf16 matrix cores: the dense half of a GCN layer, whose result is the
// dense operand of the sparse product (upstream's operator stops at A * X, spmm_accel.cu:16-102;
// a layer around it multiplies the features by a weight matrix first).
//
// The fp32 matrix instructions run at a sixteenth of the bf16 rate (157 TFLOP/s against 2.5
// PFLOP/s), so an fp32 value is taken apart into three bf16 values that add up to it exactly,
// x = x1 + x2 + x3 (each the nearest bf16 to what is left: 8 bits each of the 24), and the product
// x w is the sum of the six products x1 w1, x1 w2, x2 w1, x1 w3, x2 w2, x3 w1.  Products of bf16
// values are exact in the matrix unit and are added up in fp32.  What is left out, x2 w3 + x3 w2 + x3 w3,
// is below 2^-25 |x w|, half of what rounding one fp32 product may cost, and the accumulator is
// rounded 0.4 times per k instead of 0.5; measured against fp64 on K = 3 .. 1433 the error is
// smaller than that of v_mfma_f32_32x32x2_f32 on the same operands (2-norm of the difference over that of
// the product, K = 602: 3.7e-7 against 4.4e-7; K = 128: 1.6e-7 against 2.0e-7).  Both operands are
// multiplied by 2^24 on the way, so that the last bit of the smallest denormal is still a bf16 value, and
// the sums by 2^-48 when they are stored: small magnitudes need no other path.  Infinities, NaN, operands of
// 2^103 and more and sums of 2^79 and more leave a tile with sums that are not finite; it is computed
// again on the fp32 matrix instructions.  20,000 x 602 times 602 x 128: 40 us whatever the small
// values among the operands, 113 to 132 us with an infinity in some tiles or in all.
//
// X is rows x K with rows in the millions and K, N in the tens to hundreds, so the product
// streams X once, writes Z once and keeps W on chip.  A wavefront owns 32 rows of X and up to 128
// columns of Z (32 x 32 accumulator tiles of v_mfma_f32_32x32x16_bf16), a workgroup four of them.  K is
// walked in steps of 32.  A lane reads 64 consecutive bytes of its own row per step, two steps ahead,
// and takes them apart in registers between the matrix instructions of the step before: nobody else
// needs them, so X does not pass through LDS.  W's 32 x 128 block of the step goes through LDS, two
// blocks deep, so that one barrier per step is enough; it is taken apart by the workgroup on the
// way, or, for products large enough to pay for a launch, once beforehand (dense_prepare_kernel).
//
// Measured at 1 M x 602 times 602 x 128 (154 Gflop, 2.9 GB): 1.53 ms with the fp32 matrix instructions,
// 0.96 ms taken apart on the way, 0.93 prepared; at 2.45 M x 128 times 128 x 64: 0.44 and 0.38 ms.
// The first is bound by the matrix cores' clock and by the waits around them: of its 1.54 M cycles they are busy 58 %
// (0.53 ms at the 1.67 GHz that the clock settles at under this load; 1.06 to 1.83 over a burst, with the
// cycles the same), and the wavefronts wait for memory, LDS or the barrier 21 % of their time.
#include <atomic>

#include "preprocess.h"

namespace accel {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef v4f v4f_unaligned __attribute__((aligned(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kDenseWaves = 4;                          // wavefronts per workgroup
constexpr int kDenseThreads = kDenseWaves * 64;
constexpr int kDenseRows = 32;                          // rows per wavefront (one tile high)
constexpr int kDenseBlockRows = kDenseWaves * kDenseRows;
constexpr int kDenseStep = 32;                          // columns of X (rows of W) per step: two instructions deep
constexpr int kDenseHalf = kDenseStep / 2;              // of which a lane holds one half
constexpr int kParts = 3;                               // bf16 values per fp32 value
// Row stride of a column's 32 bf16 values in LDS, in bytes: 16-byte reads of 16 lanes whose columns
// are 80 bytes apart fall into 16 different groups of four banks.
constexpr int kWStride = 2 * kDenseStep + 16;

// Operand layout of v_mfma_f32_32x32x16_bf16: lane l holds A[l % 32][8 (l / 32) + j] and
// B[8 (l / 32) + j][l % 32], j = 0..7; accumulator register v of lane l is
// D[8 (v / 4) + 4 (l / 32) + v % 4][l % 32].  The order of the sixteen k of one instruction is free,
// only the same for A and B: lanes 0..31 carry the first half of the step's k, lanes 32..63 the second,
// 8 i .. 8 i + 7 of them in instruction i, so that a lane's 16 values are 64 consecutive bytes of its row.

// The k a half of the step starts at.  Where the row ends inside the half, the half is moved back
// to end with the row (nothing is read past it), and W is zero for the k that belong to the half or
// the step before.
__device__ __forceinline__ int half_start(int k0, int half, int K) { return min(k0 + kDenseHalf * half, K - kDenseHalf); }

// Takes two values apart, times kScale: the three parts of each, packed in pairs.
constexpr float kScale = 0x1p24f, kUnscale = 0x1p-48f;
__device__ __forceinline__ void take_apart(float a, float b, uint32_t (&part)[kParts])
{
    a *= kScale;
    b *= kScale;
#pragma unroll
    for (int p = 0; p < kParts; p++) {
        part[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
        if (p + 1 < kParts) {                           // exact: what is left has fewer bits
            a -= __uint_as_float(part[p] << 16);
            b -= __uint_as_float(part[p] & 0xFFFF0000u);
        }
    }
}

// W(k, col) of a step's half, or zero where the half does not own k (see half_start).
__device__ __forceinline__ float w_at(const float *__restrict__ W, int K, int N, int k0, int half, int j, int col)
{
    const int owned = k0 + kDenseHalf * half, k = half_start(k0, half, K) + j;
    return k >= owned && k < K && col < N ? W[(int64_t)k * N + col] : 0.f;
}

// A step of a workgroup's walk: rows [128 row_block, +128), columns [32 NT tile, +32 NT), k in [k0, k0 + 32).
struct DenseStepAt {
    int64_t row_block;
    int tile, k0;
    __device__ void advance(int K, int n_col_tiles, int64_t stride)
    {
        k0 += kDenseStep;
        if (k0 >= K) {
            k0 = 0;
            if (++tile == n_col_tiles) { tile = 0; row_block += stride; }
        }
    }
};

struct DenseArgs {
    const float *X, *W;
    float *Z;
    int64_t rows, ldx, ldz, n_row_blocks;
    int K, N, n_col_tiles, n_steps;
    const u32x4 *image;          // W taken apart (dense_prepare_kernel)
};

// One workgroup per (column tile, step): the block of W taken apart, as [part][column][32 bf16].
template <int NT>
__global__ __launch_bounds__(kDenseThreads) void dense_prepare_kernel(DenseArgs a, u32x4 *__restrict__ image)
{
    constexpr int kCols = NT * 32, kVecs = kCols * kParts * 4;
    const int tile = (int)blockIdx.x / a.n_steps, k0 = (int)blockIdx.x % a.n_steps * kDenseStep;
    u32x4 *to = image + (int64_t)blockIdx.x * kVecs;
    for (int i = threadIdx.x; i < kCols * 4; i += kDenseThreads) {
        const int c = i % kCols, v = i / kCols;             // vector v: 8 k of half v / 2
        float w[8];
#pragma unroll
        for (int j = 0; j < 8; j++) w[j] = w_at(a.W, a.K, a.N, k0, v / 2, v % 2 * 8 + j, tile * kCols + c);
        uint32_t part[4][kParts];
#pragma unroll
        for (int j = 0; j < 4; j++) take_apart(w[2 * j], w[2 * j + 1], part[j]);
#pragma unroll
        for (int p = 0; p < kParts; p++)
            to[(p * kCols + c) * 4 + v] = u32x4{part[0][p], part[1][p], part[2][p], part[3][p]};
    }
}

// How the product gets its block of W per step.
enum DenseW {
    kWPrepared,                  // from the image
    kWOnTheWay                   // taken apart by the workgroup
};

// A workgroup's block of W of a step on its way through registers into LDS.
template <int NT, DenseW kHow> struct WStage;
template <int NT> struct WStage<NT, kWPrepared> {
    static constexpr int kCols = NT * 32, kVecs = kCols * kParts * 4;
    static constexpr int kMine = (kVecs + kDenseThreads - 1) / kDenseThreads;
    u32x4 v[kMine];
    __device__ __forceinline__ void fetch(const DenseArgs &a, const DenseStepAt &at)
    {
        const u32x4 *from = a.image + ((int64_t)at.tile * a.n_steps + at.k0 / kDenseStep) * kVecs + threadIdx.x;
#pragma unroll
        for (int i = 0; i < kMine; i++)
            if (kVecs % kDenseThreads == 0 || i * kDenseThreads + (int)threadIdx.x < kVecs) v[i] = from[i * kDenseThreads];
    }
    __device__ __forceinline__ void store(const DenseArgs &, const DenseStepAt &, char *lds)
    {
#pragma unroll
        for (int i = 0; i < kMine; i++) {
            const int at = i * kDenseThreads + (int)threadIdx.x;
            if (kVecs % kDenseThreads == 0 || at < kVecs) *reinterpret_cast<u32x4 *>(lds + at / 4 * kWStride + at % 4 * 16) = v[i];
        }
    }
};
template <int NT, DenseW kHow> struct WStage {
    static constexpr int kCols = NT * 32;
    static constexpr int kRun = kDenseStep * kCols / kDenseThreads;      // consecutive k of a thread: 16, 8, 4
    float v[kRun];
    __device__ __forceinline__ void fetch(const DenseArgs &a, const DenseStepAt &at)
    {
        // the same loads on every path; what the block does not own is replaced by zero in store()
        const int c = (int)threadIdx.x % kCols, k = (int)threadIdx.x / kCols * kRun;
        const int col = min(at.tile * kCols + c, a.N - 1);
        if (at.k0 + kDenseStep <= a.K) {
            const float *wb = a.W + (int64_t)(at.k0 + k) * a.N + col;
#pragma unroll
            for (int i = 0; i < kRun; i++) v[i] = wb[(int64_t)i * a.N];
        } else {
            const int k1 = half_start(at.k0, k / kDenseHalf, a.K) + k % kDenseHalf;
#pragma unroll
            for (int i = 0; i < kRun; i++) v[i] = a.W[(int64_t)min(k1 + i, a.K - 1) * a.N + col];
        }
    }
    __device__ __forceinline__ void store(const DenseArgs &a, const DenseStepAt &at, char *lds)
    {
        const int c = (int)threadIdx.x % kCols, k = (int)threadIdx.x / kCols * kRun;
        if (at.k0 + kDenseStep > a.K || (at.tile + 1) * kCols > a.N) {
            const bool col_ok = at.tile * kCols + c < a.N;
            const int owned = at.k0 + k - k % kDenseHalf, k1 = half_start(at.k0, k / kDenseHalf, a.K) + k % kDenseHalf;
#pragma unroll
            for (int i = 0; i < kRun; i++) v[i] = col_ok && k1 + i >= owned && k1 + i < a.K ? v[i] : 0.f;
        }
        uint32_t part[kRun / 2][kParts];
#pragma unroll
        for (int i = 0; i < kRun; i += 2) take_apart(v[i], v[i + 1], part[i / 2]);
#pragma unroll
        for (int p = 0; p < kParts; p++) {
            char *to = lds + (p * kCols + c) * kWStride + 2 * k;
            if constexpr (kRun >= 8) {
#pragma unroll
                for (int i = 0; i < kRun / 2; i += 4)
                    *reinterpret_cast<u32x4 *>(to + 4 * i) = u32x4{part[i][p], part[i + 1][p], part[i + 2][p], part[i + 3][p]};
            } else {
                *reinterpret_cast<uint2 *>(to) = make_uint2(part[0][p], part[1][p]);
            }
        }
    }
};

// Adds the products of k in [0, K) to a wavefront's tile by the fp32 matrix instructions, from memory.
// v_mfma_f32_32x32x2_f32: lane l holds A[l % 32][l / 32] and B[l / 32][l % 32], the accumulators as above.  Rows and
// columns past the end repeat the last one (their sums are not stored); a k past the end is zero on both
// sides (an infinity times zero would be a NaN).
template <int NT>
__device__ __forceinline__ void add_in_fp32(const DenseArgs &a, int64_t row0, int col0, f32x16 (&acc)[NT])
{
    const int half = (threadIdx.x & 63) >> 5, l32 = threadIdx.x & 31;
    const int64_t r = row0 + l32;
    const float *xr = a.X + (r < a.rows ? r : a.rows - 1) * a.ldx;
    constexpr int U = 4;                                    // instructions whose operands are on their way together
#pragma unroll 1
    for (int k = 0; k < a.K; k += 2 * U) {
        float x[U], w[U][NT];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int at = min(k + 2 * u + half, a.K - 1);
            x[u] = xr[at];
#pragma unroll
            for (int t = 0; t < NT; t++) w[u][t] = a.W[(int64_t)at * a.N + min(col0 + 32 * t + l32, a.N - 1)];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool in = k + 2 * u + half < a.K;
#pragma unroll
            for (int t = 0; t < NT; t++)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? x[u] : 0.f, in ? w[u][t] : 0.f, acc[t], 0, 0, 0);
        }
    }
}

// The grid is sized to what the GPU holds at once and every workgroup walks blocks of 128
// rows, gridDim.x apart, as one sequence of steps: the reads of a block's first steps are
// issued while the matrix cores work on the last steps of the block before, and that block's
// rows of Z are stored behind them, so the memory latency is paid once per workgroup, not
// once per block.  The column tiles of one block of rows (N > 128) follow each other in the
// same workgroup: the rows of X they share come from L2 for all but the first.
// Loads are the same in number on every path (clamped, not branched around), which keeps the
// compiler's waits for them exact.
template <int NT, DenseW kHow>
__global__ __launch_bounds__(kDenseThreads, NT == 4 ? 2 : 3) void dense_xw_kernel(DenseArgs a)
{
    constexpr int kCols = NT * 32;
    __shared__ __attribute__((aligned(16))) char w_lds[2][kParts * kCols * kWStride];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int half = lane >> 5, l32 = lane & 31;

    // This lane's 16 values of X of a step; rows past the end of X read the last row (their results
    // are not stored), and so does a step past the end of the walk.  Narrow outputs, whose product
    // is bound by streaming X, read eight lanes to a row (whole lines per instruction) and turn the
    // values in LDS, within the wavefront (2.45 M x 100 x 32: 298 -> 275 us; with more columns the
    // detour costs as much as it gives: 128 x 64 382 -> 375 us at 2.45 M rows, 28 -> 32 at 170 k).
    constexpr bool kTurn = NT == 1;
    __shared__ v4f x_lds[kTurn ? kDenseWaves : 1][kTurn ? kDenseRows * 8 : 1];
    auto turned = [&](const v4f (&x)[4], v4f (&y)[4]) {
        if constexpr (kTurn) {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int row = 8 * q + (lane >> 3);
                x_lds[wave][row * 8 + ((lane & 7) ^ (row & 7))] = x[q];
            }
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int q = 0; q < 4; q++) y[q] = kTurn ? x_lds[wave][l32 * 8 + ((4 * half + q) ^ (l32 & 7))] : x[q];
    };
    auto fetch_x = [&](v4f (&x)[4], const DenseStepAt &at) {
        if constexpr (kTurn) {
            const int64_t r0 = at.row_block * kDenseBlockRows + wave * kDenseRows + (lane >> 3);
            const int k = half_start(at.k0, (lane >> 2) & 1, a.K) + 4 * (lane & 3);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int64_t r = r0 + 8 * q;
                x[q] = *reinterpret_cast<const v4f_unaligned *>(a.X + (r < a.rows ? r : a.rows - 1) * a.ldx + k);
            }
            return;
        }
        const int64_t r = at.row_block * kDenseBlockRows + wave * kDenseRows + l32;
        const float *xr = a.X + (r < a.rows ? r : a.rows - 1) * a.ldx;
        const int k = half_start(at.k0, half, a.K);
#pragma unroll
        for (int q = 0; q < 4; q++) x[q] = *reinterpret_cast<const v4f_unaligned *>(xr + k + 4 * q);
    };

    f32x16 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[t][v] = 0.f;

    const int64_t stride = gridDim.x;          // gridDim.x <= n_row_blocks: every workgroup has work
    DenseStepAt now{(int64_t)blockIdx.x, 0, 0}, next = now, after;
    next.advance(a.K, a.n_col_tiles, stride);
    after = next;
    after.advance(a.K, a.n_col_tiles, stride);
    v4f x0[4], x1[4];
    WStage<NT, kHow> w;
    bf16x8 apart[2][kParts];                   // this step's values of X, taken apart
    auto take_pair = [&](const v4f (&x)[4], int q, uint32_t (&pair)[kParts]) {
        take_apart(x[q / 2][2 * (q & 1)], x[q / 2][2 * (q & 1) + 1], pair);
        // (keeps the work here, between the matrix instructions, where the compiler would move it
        // to the next step)
        asm volatile("" : "+v"(pair[0]), "+v"(pair[1]), "+v"(pair[2]));
    };
    auto gather_pairs = [&](const uint32_t (&pair)[8][kParts]) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int p = 0; p < kParts; p++)
                apart[i][p] = __builtin_bit_cast(bf16x8, u32x4{pair[4 * i][p], pair[4 * i + 1][p], pair[4 * i + 2][p],
                                                               pair[4 * i + 3][p]});
    };

    w.fetch(a, now);
    fetch_x(x0, now);
    fetch_x(x1, next);
    {
        uint32_t pair[8][kParts];
        v4f y[4];
        turned(x0, y);
#pragma unroll
        for (int q = 0; q < 8; q++) take_pair(y, q, pair[q]);
        gather_pairs(pair);
    }
    w.store(a, now, w_lds[0]);
    int step = 0;
    // xf: free registers, for the step after the next; xn: the next step's X
    auto one = [&](v4f (&xf)[4], v4f (&xn)[4]) {
        const int buf = step & 1;
        __syncthreads();                       // this step's block of W is in place; the other one's readers are done
        w.fetch(a, next);
        fetch_x(xf, after);
        __builtin_amdgcn_sched_barrier(0);     // the loads go out here, ahead of the matrix work that hides them

        // The step's 12 NT matrix instructions in groups of one or two tiles' six; the reads of the
        // next group's W and a share of taking the next step's X apart go between them.
        constexpr int P = NT < 2 ? NT : 2, kGroups = 2 * NT / P;
        bf16x8 b[2][P][kParts];
        auto read_b = [&](bf16x8 (&to)[P][kParts], int g) {
#pragma unroll
            for (int u = 0; u < P; u++)
#pragma unroll
                for (int p = 0; p < kParts; p++)
                    to[u][p] = *reinterpret_cast<const bf16x8 *>(
                        &w_lds[buf][(p * kCols + 32 * (g * P % NT + u) + l32) * kWStride + 32 * half + 16 * (g * P / NT)]);
        };
        uint32_t pair[8][kParts];
        read_b(b[0], 0);
        v4f y[4];
        turned(xn, y);
#pragma unroll
        for (int g = 0; g < kGroups; g++) {
            if (g + 1 < kGroups) read_b(b[(g + 1) & 1], g + 1);
            constexpr int ap[6] = {2, 0, 1, 1, 0, 0}, bp[6] = {0, 2, 1, 0, 1, 0};     // the small products first
#pragma unroll
            for (int q = 0; q < 6; q++)
#pragma unroll
                for (int u = 0; u < P; u++)
                    acc[g * P % NT + u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(apart[g * P / NT][ap[q]], b[g & 1][u][bp[q]],
                                                                                  acc[g * P % NT + u], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (q * kGroups / 8 == g) take_pair(y, q, pair[q]);
            __builtin_amdgcn_sched_barrier(0);
        }
        gather_pairs(pair);
        w.store(a, next, w_lds[buf ^ 1]);      // its readers were done at this step's barrier

        if (next.k0 == 0) {                    // that was the last step of this tile: store it, start the next at zero
            const int64_t row0 = now.row_block * kDenseBlockRows + wave * kDenseRows;
            const int col = now.tile * kCols + l32;
            float *z = a.Z + (row0 + 4 * half) * a.ldz + col;
            bool finite = true;
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int v = 0; v < 16; v++) finite &= __builtin_isfinite(acc[t][v]);
            float unscale = kUnscale;
            if (__any(!finite)) {
                unscale = 1;
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++) acc[t][v] = 0.f;
                add_in_fp32<NT>(a, row0, now.tile * kCols, acc);
            }
            if (row0 + kDenseRows <= a.rows && now.tile * kCols + kCols <= a.N) {      // nothing to mask
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++) z[(8 * (v / 4) + v % 4) * a.ldz + t * 32] = acc[t][v] * unscale;
            } else {
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const int64_t row = row0 + 8 * (v / 4) + 4 * half + (v % 4);
                        if (col + t * 32 < a.N && row < a.rows) z[(8 * (v / 4) + v % 4) * a.ldz + t * 32] = acc[t][v] * unscale;
                    }
            }
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[t][v] = 0.f;
        }
        now = next;
        next = after;
        after.advance(a.K, a.n_col_tiles, stride);
        step++;
    };
    while (now.row_block < a.n_row_blocks) {
        one(x0, x1);
        if (now.row_block >= a.n_row_blocks) break;
        one(x1, x0);
    }
}

// K < 16: one instruction deep, so that W's columns stay in registers while a wavefront walks tiles of 32
// rows, the next tile's X ahead of the products; bound by storing Z.  kInFp32 (K = 1 and 2): by the fp32
// instructions, whose error is the smaller one there (each product is exact before it is added: one
// rounding per sum at K = 1.  2-norm of the difference over that of the product, normal operands: 2.5e-8
// against 3.5e-8 in three parts; K = 2: 3.1e-8, 3.4e-8; K = 3: 3.6e-8, 3.3e-8; K = 8: 5.3e-8, 3.1e-8).
// With several column tiles (N > 128) W is fetched again for every one of them; by workgroups of their own,
// which store the lines that two tiles meet in at different times, 10 x 300 takes 1.32 to 1.48 ms.
// 2.45 M rows, in the kernel above (W through LDS, 32 k per step) and here: 1 x 64 131 -> 117 us, 2 x 128
// 261 -> 246, 4 x 16 101 -> 53, 8 x 64 239 -> 179, 12 x 32 138 -> 93, 15 x 128 290 -> 256, 10 x 300 1093 -> 1049.
template <int NT, bool kInFp32>
__global__ __launch_bounds__(kDenseThreads, NT == 4 ? 2 : 3) void dense_short_kernel(DenseArgs a)
{
    constexpr int J = kInFp32 ? 1 : 8;         // k that a lane holds of the one instruction: J half ...
    const int lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n_row_tiles = (a.rows + kDenseRows - 1) / kDenseRows;
    const int64_t stride = (int64_t)gridDim.x * kDenseWaves;
    // those behind K read the last one and count as zero
    auto fetch_x = [&](float (&x)[J], int64_t row_tile) {
        const int64_t r = row_tile * kDenseRows + l32;
        const float *xr = a.X + (r < a.rows ? r : a.rows - 1) * a.ldx;
#pragma unroll
        for (int j = 0; j < J; j++) x[j] = xr[min(J * half + j, a.K - 1)];
    };
    auto or_zero = [&](const float (&x)[J], int j) { return J * half + j < a.K ? x[j] : 0.f; };
    struct Operand {
        bf16x8 part[kParts];
        float whole;
    };
    auto operand = [&](const float (&x)[J], Operand &to) {
        if constexpr (kInFp32) {
            to.whole = or_zero(x, 0);
        } else {
            uint32_t pair[4][kParts];
#pragma unroll
            for (int j = 0; j < 4; j++) take_apart(or_zero(x, 2 * j), or_zero(x, 2 * j + 1), pair[j]);
#pragma unroll
            for (int p = 0; p < kParts; p++)
                to.part[p] = __builtin_bit_cast(bf16x8, u32x4{pair[0][p], pair[1][p], pair[2][p], pair[3][p]});
        }
    };
    Operand w[NT];
    auto fetch_w = [&](int col0) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            float v[J];
#pragma unroll
            for (int j = 0; j < J; j++)
                v[j] = a.W[(int64_t)min(J * half + j, a.K - 1) * a.N + min(col0 + 32 * t + l32, a.N - 1)];
            operand(v, w[t]);
        }
    };
    fetch_w(0);
    float x[J], next[J];
    int64_t row_tile = (int64_t)blockIdx.x * kDenseWaves + wave;
    fetch_x(x, row_tile);
    for (; row_tile < n_row_tiles; row_tile += stride) {
        fetch_x(next, row_tile + stride);
        const int64_t row0 = row_tile * kDenseRows;
        Operand xt;
        operand(x, xt);
        for (int tile = 0; tile < (NT == 4 ? a.n_col_tiles : 1); tile++) {
            const int col0 = tile * NT * 32;
            if (NT == 4 && a.n_col_tiles > 1) fetch_w(col0);
            f32x16 acc[NT];
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[t][v] = 0.f;
            float unscale = 1;
            if constexpr (kInFp32) {
#pragma unroll
                for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(xt.whole, w[t].whole, acc[t], 0, 0, 0);
            } else {
                constexpr int ap[6] = {2, 0, 1, 1, 0, 0}, bp[6] = {0, 2, 1, 0, 1, 0};         // the small products first
#pragma unroll
                for (int q = 0; q < 6; q++)
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xt.part[ap[q]], w[t].part[bp[q]], acc[t], 0, 0, 0);
                bool finite = true;
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++) finite &= __builtin_isfinite(acc[t][v]);
                unscale = kUnscale;
                if (__any(!finite)) {
                    unscale = 1;
#pragma unroll
                    for (int t = 0; t < NT; t++)
#pragma unroll
                        for (int v = 0; v < 16; v++) acc[t][v] = 0.f;
                    add_in_fp32<NT>(a, row0, col0, acc);
                }
            }
            const int64_t rows = a.rows - row0 - 4 * half;
            const int col = col0 + l32;
            float *z = a.Z + (row0 + 4 * half) * a.ldz + col;
            asm volatile("" : "+v"(z));            // (the stores' addresses are formed here, not kept from tile to tile)
            if (row0 + kDenseRows <= a.rows && col0 + NT * 32 <= a.N) {
#pragma unroll
                for (int v = 0; v < 16; v++)
#pragma unroll
                    for (int t = 0; t < NT; t++) z[(8 * (v / 4) + v % 4) * a.ldz + t * 32] = acc[t][v] * unscale;
            } else {
#pragma unroll
                for (int v = 0; v < 16; v++)
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        if (col + t * 32 < a.N && 8 * (v / 4) + v % 4 < rows)
                            z[(8 * (v / 4) + v % 4) * a.ldz + t * 32] = acc[t][v] * unscale;
            }
        }
#pragma unroll
        for (int j = 0; j < J; j++) x[j] = next[j];
    }
}

// The grid: as many workgroups as the GPU holds at once (asked of the runtime for the kernel
// that runs, once per device and kernel), or one per block of rows when there are fewer.
constexpr int kDenseDevices = 64;
static std::atomic<int> g_resident[kDenseDevices][12];    // [device][kernel]: workgroups the device holds, 0 = not asked yet

static int dense_launch(void (*kernel)(DenseArgs), int which, const DenseArgs &a, hipStream_t s)
{
    int dev = 0;
    ACCEL_HIP(hipGetDevice(&dev));
    int resident = dev >= 0 && dev < kDenseDevices ? g_resident[dev][which].load(std::memory_order_relaxed) : 0;
    if (resident == 0) {
        int cus = 0, per_cu = 0;
        ACCEL_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        ACCEL_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kDenseThreads, 0));
        resident = (cus > 0 ? cus : 256) * (per_cu > 0 ? per_cu : 1);
        if (dev >= 0 && dev < kDenseDevices) g_resident[dev][which].store(resident, std::memory_order_relaxed);
    }
    const unsigned grid = (unsigned)(a.n_row_blocks < resident ? a.n_row_blocks : resident);
    kernel<<<grid, kDenseThreads, 0, s>>>(a);
    return ACCEL_OK;
}

// Wide products (128 columns to a workgroup) of this many multiplications and more take W apart
// beforehand: a launch more (5 us) and half the integer work inside (1 M rows: 300 x 100 548 -> 502 us,
// 602 x 128 964 -> 926, 512 x 256 1527 -> 1466).  Narrow ones are bound by memory and gain nothing
// (2.45 M x 128 x 64: 382 -> 394 us).
constexpr double kPrepareFrom = 1e10;

template <int NT>
static int dense_product(DenseArgs a, hipStream_t s, bool may_prepare)
{
    constexpr int which = NT == 1 ? 0 : NT == 2 ? 4 : 8;
    if (a.K <= 2) return dense_launch(dense_short_kernel<NT, true>, which, a, s);
    if (a.K < kDenseHalf) return dense_launch(dense_short_kernel<NT, false>, which + 1, a, s);
    if constexpr (NT == 4) {
        const size_t blocks = (size_t)a.n_col_tiles * (size_t)a.n_steps;
        const size_t image_bytes = blocks * (NT * 32 * kParts * 4) * sizeof(u32x4);
        void *mem = nullptr;
        if (may_prepare && (double)a.rows * a.K * a.N >= kPrepareFrom)
            mem = take_stream_memory(image_bytes, s);
        if (mem) {
            u32x4 *image = static_cast<u32x4 *>(mem);
            dense_prepare_kernel<NT><<<dim3((unsigned)blocks), kDenseThreads, 0, s>>>(a, image);
            a.image = image;
            const int rc = dense_launch(dense_xw_kernel<NT, kWPrepared>, which + 2, a, s);
            give_stream_memory(mem, s);
            return rc;
        }
    }
    return dense_launch(dense_xw_kernel<NT, kWOnTheWay>, which + 3, a, s);
}

// Arguments have been checked by the caller (accel_dense_xw): rows >= 1, K, N >= 1,
// ldx >= K, ldz >= N, operands readable and large enough.  may_prepare: s is not capturing (a graph's
// memory would have to live as long as the graph).
int dense_xw_launch(const float *X, const float *W, float *Z, int64_t rows, int K, int N, int64_t ldx, int64_t ldz,
                    hipStream_t s, bool may_prepare)
{
    (void)hipGetLastError();
    const int nt = N <= 32 ? 1 : N <= 64 ? 2 : 4;
    DenseArgs a{};
    a.X = X; a.W = W; a.Z = Z;
    a.rows = rows; a.ldx = ldx; a.ldz = ldz;
    a.n_row_blocks = (rows + kDenseBlockRows - 1) / kDenseBlockRows;
    a.K = K; a.N = N;
    a.n_col_tiles = (N + nt * 32 - 1) / (nt * 32);
    a.n_steps = (K + kDenseStep - 1) / kDenseStep;
    const int rc = nt == 1   ? dense_product<1>(a, s, may_prepare)
                   : nt == 2 ? dense_product<2>(a, s, may_prepare)
                             : dense_product<4>(a, s, may_prepare);
    if (rc) return rc;
    ACCEL_HIP(hipGetLastError());
    return ACCEL_OK;
}

}  // namespace accel
