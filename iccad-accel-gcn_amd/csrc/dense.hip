// Z = X * W in fp32 on the 16-bit matrix cores: the dense half of a GCN layer, whose result is the
// dense operand of the sparse product (upstream's operator stops at A * X, spmm_accel.cu:16-102;
// a layer around it multiplies the features by a weight matrix first).
//
// The fp32 matrix instructions run at a sixteenth of the 16-bit rate (157 TFLOP/s against 2.5
// PFLOP/s), so an fp32 value is taken apart into 16-bit values whose products, exact in the matrix unit, are
// added up in fp32.  In one of two ways:
//
// Three bf16 values (walk_bf16), for any K and any magnitudes: x = x1 + x2 + x3 exactly (each the nearest bf16
// to what is left: 8 bits each of the 24), and the product x w is the sum of the six products x1 w1, x1 w2,
// x2 w1, x1 w3, x2 w2, x3 w1.  What is left out, x2 w3 + x3 w2 + x3 w3,
// is below 2^-25 |x w|, half of what rounding one fp32 product may cost, and the accumulator is
// rounded 0.4 times per k instead of 0.5; measured against fp64 on K = 3 .. 1433 the error is
// smaller than that of v_mfma_f32_32x32x2_f32 on the same operands (2-norm of the difference over that of
// the product, K = 602: 3.7e-7 against 4.4e-7; K = 128: 1.6e-7 against 2.0e-7).  Both operands are
// multiplied by 2^24 on the way, so that the last bit of the smallest denormal is still a bf16 value, and
// the sums by 2^-48 when they are stored: small magnitudes need no other path.  Infinities, NaN, operands of
// 2^103 and more and sums of 2^79 and more leave a tile with sums that are not finite; it is computed
// again on the fp32 matrix instructions.
//
// Two fp16 values (walk_fp16), for products of K >= 64 that pay for two more launches: half the matrix work.  The first is
// the nearest fp16, the second 2048 times what is left, together 22 bits and more.  Three products, x1 w1 in one
// accumulator, x1 w2 and x2 w1 in another that is added at the end times 2^-11.  What is lost, a last bit of
// one value in four and x2 w2, is 7e-8 of a product, and the accumulator that counts is rounded a sixth as often
// as above: error against fp64 (uniform operands; the other way in brackets) K = 64 7.5e-8 (1.09e-7), 128 1.03e-7
// (1.62e-7), 256 1.16e-7 (2.34e-7), 602 1.73e-7 (3.70e-7), largest element error over the result's root mean square at 602
// 2.4e-6 (6.2e-6); the same order for normal, positive and half-empty operands.  Below K = 64 the two errors meet (K = 48:
// 9.1e-8 and 9.4e-8), which is where the line is.  fp16 has a short range, so both operands are scaled by powers of
// two, W per column tile, X per tile of 32 rows by its largest magnitude as far as that is known.  What the two values of a
// magnitude below 2^-29 of that lose is added by the fp32 instructions, for the steps that hold such magnitudes
// (add_lost); a tile with sums that are not finite is computed again by them; a workgroup that sees many of either goes
// on in three parts, and all do where W's magnitudes are too far apart.  1 M x 602 times 602 x 128: 0.72 ms, with a value of
// 1e-38 in 200 tiles too, 1.02 with magnitudes over 20 orders everywhere (0.93 in three parts); 50,000 rows: 45, 53 and 71 us (61).
//
// X is rows x K with rows in the millions and K, N in the tens to hundreds, so the product
// streams X once, writes Z once and keeps W on chip.  A wavefront owns 32 rows of X and up to 128
// columns of Z, a workgroup four of them.  K is
// walked in steps of 32.  A lane reads 64 consecutive bytes of its own row (walk_fp16: with three others, 64 of a row) per
// step, ahead, and takes them apart in registers between the matrix instructions of the step before: nobody else
// needs them, so X does not pass through LDS.  W's 32 x 128 block of the step goes through LDS, two
// blocks deep, so that one barrier per step is enough; it is taken apart by the workgroup on the
// way (walk_bf16) or once beforehand.
//
// Measured at 1 M x 602 times 602 x 128 (154 Gflop, 2.9 GB): 1.53 ms with the fp32 matrix instructions, 0.93 in three
// parts, 0.70 to 0.72 in two; 2.45 M x 128 times 128 x 64: 0.44, 0.36, 0.33; 100,000 x 602 times 602 x 128: 118 us in three, 78 in two.
// Reading this X and writing this Z in the same order and doing nothing else takes 0.57 ms (5.1 TB/s; rows of 2408 bytes
// do not start on lines: 0.54 with 608 columns, the product 0.65).  The product takes the same 0.70 ms at 1.7 and
// at 2.1 GHz, and 0.69 with a third of its matrix instructions: it is bound by memory.  Of 1.32 M cycles the matrix cores
// are busy 34 %.  No less with X through LDS two steps ahead, or with two tiles' W read at once.
#include <atomic>

#include "preprocess.h"

namespace accel {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef v4f v4f_unaligned __attribute__((aligned(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

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
    __device__ void advance(int K, int first_tile, int last_tile, int64_t stride)
    {
        k0 += kDenseStep;
        if (k0 >= K) {
            k0 = 0;
            if (tile == last_tile) { tile = first_tile; row_block += stride; } else { tile++; }
        }
    }
};

struct DenseArgs {
    const float *X, *W;
    float *Z;
    int64_t rows, ldx, ldz, n_row_blocks;
    int K, N, n_col_tiles, n_steps;
    int apart;                   // the column tiles of a block of rows are workgroups of their own (asked for, then decided by dense_launch)
    const u32x4 *image;          // walk_fp16: W taken apart (dense_prepare_kernel), and what is in front of that
    const int *head;
};

// Where a workgroup starts.
__device__ __forceinline__ DenseStepAt first_step(const DenseArgs &a)
{
    const int64_t b = blockIdx.x;
    // the workgroups of a block's tiles are eight apart: on one die, at about the same time
    const int64_t slot = b / kXcds;
    return a.apart ? DenseStepAt{slot / a.n_col_tiles * kXcds + b % kXcds, (int)(slot % a.n_col_tiles), 0} : DenseStepAt{b, 0, 0};
}

// A workgroup's block of W of a step on its way through registers, taken apart, into LDS.
template <int NT> struct WStage {
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
// once per block.  The column tiles of one block of rows (N > 128) belong to workgroups next to each other on
// one die, or follow each other in the same one (see dense_launch).
// Loads are the same in number on every path (clamped, not branched around), which keeps the
// compiler's waits for them exact.  Starts at `now`, at the start of a tile.
template <int NT>
__device__ __forceinline__ void walk_bf16(const DenseArgs &a, char (*w_lds)[kParts * NT * 32 * kWStride], DenseStepAt now)
{
    constexpr int kCols = NT * 32;

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

    const int64_t stride = a.apart ? gridDim.x / a.n_col_tiles : gridDim.x;
    const int first_tile = a.apart ? now.tile : 0, last_tile = a.apart ? now.tile : a.n_col_tiles - 1;
    DenseStepAt next = now, after;
    next.advance(a.K, first_tile, last_tile, stride);
    after = next;
    after.advance(a.K, first_tile, last_tile, stride);
    v4f x0[4], x1[4];
    WStage<NT> w;
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
        after.advance(a.K, first_tile, last_tile, stride);
        step++;
    };
    while (now.row_block < a.n_row_blocks) {
        one(x0, x1);
        if (now.row_block >= a.n_row_blocks) break;
        one(x1, x0);
    }
}

template <int NT>
__global__ __launch_bounds__(kDenseThreads, NT == 4 ? 2 : 3) void dense_xw_kernel(DenseArgs a)
{
    __shared__ __attribute__((aligned(16))) char w_lds[2][kParts * NT * 32 * kWStride];
    const DenseStepAt at = first_step(a);
    if (at.row_block < a.n_row_blocks) walk_bf16<NT>(a, w_lds, at);
}

// ---- two fp16 values per fp32 value -----------------------------------------------------------------------------
typedef const int __attribute__((address_space(4))) constant_int;
constexpr int kParts16 = 2;
constexpr float kLow = 2048.f;                          // what the second value is scaled up by
constexpr int kTop = 14;                                // scaled magnitudes: the largest in [2^14, 2^15) ...
constexpr int kFloor = -15;                             // ... and none but zero below 2^-15

// |v| as a sort key that leaves zero out of a minimum, and the key of 2^e.
__device__ __forceinline__ uint32_t key_of(float v) { return (__float_as_uint(v) << 1) - 1u; }
__device__ __forceinline__ uint32_t key_of_power(int e) { return ((uint32_t)max(e + 127, 0) << 24) - 1u; }
// Exponent of the power of two that takes the magnitude `largest` (its bits) to [2^14, 2^15).
__device__ __forceinline__ int scale_for(uint32_t largest)
{
    return largest == 0 ? 0 : min(max(kTop + 127 - (int)(largest >> 23), -113), 100);
}
__device__ __forceinline__ float power_of_two(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }   // e in -126..127

__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
    // within rows of 16 lanes: neighbours, pairs, halves mirrored, rows mirrored; then the four rows
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true));
    const uint32_t a = max((uint32_t)__builtin_amdgcn_readlane((int)v, 0), (uint32_t)__builtin_amdgcn_readlane((int)v, 16));
    const uint32_t b = max((uint32_t)__builtin_amdgcn_readlane((int)v, 32), (uint32_t)__builtin_amdgcn_readlane((int)v, 48));
    return max(a, b);
}

// Two values times `scale` as two fp16 values each, packed in pairs: the nearest, and 2048 times what is left.
__device__ __forceinline__ void take_apart16(float a, float b, float scale, uint32_t &top, uint32_t &rest)
{
    const float low_scale = scale * kLow;
    const f16x2 high = __builtin_convertvector(f32x2{a * scale, b * scale}, f16x2);
    const float ra = fmaf((float)high.x, -kLow, a * low_scale), rb = fmaf((float)high.y, -kLow, b * low_scale);
    top = __builtin_bit_cast(uint32_t, high);
    rest = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{ra, rb}, f16x2));
}

// What is in front of the image: [0] whether W is left to the three-part walk, [1 + tile] the exponents of the
// column tiles' scales, then for every block of W (a step of a column tile) the bits of its largest magnitude and the
// key of its smallest one that is not zero.
constexpr size_t head_words(int n_col_tiles, size_t blocks) { return (1 + n_col_tiles + 2 * blocks + 3) / 4 * 4; }

// Operand layout of v_mfma_f32_16x16x32_f16: lane l holds A[l % 16][8 (l / 16) + j] and B[8 (l / 16) + j][l % 16], j = 0..7;
// accumulator register v of lane l is D[4 (l / 16) + v][l % 16].  The order of the 32 k is free: a lane takes
// 16 (j / 4) + 4 (l / 16) + j % 4, so that four lanes read 64 consecutive bytes of a row of X per load.  So is that of the
// columns: those of four tiles interleave, and a lane stores four neighbouring ones of Z.
constexpr int kStore = 4;
__device__ __forceinline__ int column_of(int t, int c) { return t / kStore * (16 * kStore) + kStore * c + t % kStore; }

template <int NT>
__global__ __launch_bounds__(kDenseThreads) void dense_range_kernel(DenseArgs a, int *__restrict__ head)
{
    constexpr int kCols = NT * 32, kRun = kDenseStep * kCols / kDenseThreads;
    __shared__ uint32_t largest_of[kDenseWaves], least_of[kDenseWaves];
    const int tile = (int)blockIdx.x / a.n_steps, k0 = (int)blockIdx.x % a.n_steps * kDenseStep;
    const int c = (int)threadIdx.x % kCols, k = k0 + (int)threadIdx.x / kCols * kRun;
    const int col = min(tile * kCols + c, a.N - 1);
    float w[kRun];
#pragma unroll
    for (int i = 0; i < kRun; i++) w[i] = a.W[(int64_t)min(k + i, a.K - 1) * a.N + col];     // (repeats change nothing)
    uint32_t largest = 0, least = 0xFFFFFFFFu;
#pragma unroll
    for (int i = 0; i < kRun; i++) {
        largest = max(largest, __float_as_uint(w[i]) & 0x7FFFFFFFu);
        least = min(least, key_of(w[i]));
    }
    largest = wave_max(largest);
    least = ~wave_max(~least);
    if ((threadIdx.x & 63) == 0) {
        largest_of[threadIdx.x >> 6] = largest;
        least_of[threadIdx.x >> 6] = least;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kDenseWaves; i++) {
            largest = max(largest, largest_of[i]);
            least = min(least, least_of[i]);
        }
        int *to = head + 1 + a.n_col_tiles + 2 * (int)blockIdx.x;
        to[0] = (int)largest;
        to[1] = (int)least;
    }
}

// One workgroup per (column tile, step): the block of W as fp16 values, [part][column][32], unless W holds
// magnitudes further apart than these carry (or an infinity or a NaN).
template <int NT>
__global__ __launch_bounds__(kDenseThreads) void dense_prepare_kernel(DenseArgs a, int *__restrict__ head, u32x4 *__restrict__ image)
{
    constexpr int kCols = NT * 32;
    const int my_tile = (int)blockIdx.x / a.n_steps, k0 = (int)blockIdx.x % a.n_steps * kDenseStep, lane = threadIdx.x & 63;
    bool wide = false;
    int my_scale = 0;
    for (int t = 0; t < a.n_col_tiles; t++) {               // every wavefront looks at every block's range
        uint32_t largest = 0, least = 0xFFFFFFFFu;
        for (int i = lane; i < a.n_steps; i += 64) {
            const int *at = head + 1 + a.n_col_tiles + 2 * (t * a.n_steps + i);
            largest = max(largest, (uint32_t)at[0]);
            least = min(least, (uint32_t)at[1]);
        }
        largest = wave_max(largest);
        least = ~wave_max(~least);
        const int scale = scale_for(largest);
        wide |= largest >= 0x7F800000u || least < key_of_power(kFloor - scale);
        if (t == my_tile) my_scale = scale;
        if (blockIdx.x == 0 && threadIdx.x == 0) head[1 + t] = scale;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) head[0] = wide;
    if (wide) return;
    u32x4 *to = image + (int64_t)blockIdx.x * (kCols * kParts16 * 4);
    for (int i = threadIdx.x; i < kCols * 4; i += kDenseThreads) {
        const int c = i % 16, quarter = i / 16 % 4, t = i / 64;
        const int col = my_tile * kCols + column_of(t, c);
        float w[8];
#pragma unroll
        for (int j = 0; j < 8; j++) w[j] = w_at(a.W, a.K, a.N, k0, j / 4, 4 * quarter + j % 4, col);
        uint32_t part[kParts16][4];
#pragma unroll
        for (int j = 0; j < 4; j++) take_apart16(w[2 * j], w[2 * j + 1], power_of_two(my_scale), part[0][j], part[1][j]);
#pragma unroll
        for (int p = 0; p < kParts16; p++)
            to[p * kCols * 4 + i] = u32x4{part[p][0], part[p][1], part[p][2], part[p][3]};
    }
}

// Adds the products of k in [0, K) to a wavefront's tiles by the fp32 matrix instructions, from memory, as add_in_fp32 does.
// v_mfma_f32_16x16x4_f32: lane l holds A[l % 16][l / 16] and B[l / 16][l % 16], the accumulators as below.
template <int NT>
__device__ __forceinline__ void add_in_fp32_by_16(const DenseArgs &a, int64_t row0, int col0, f32x4 (&acc)[2][2 * NT])
{
    const int quarter = (threadIdx.x & 63) >> 4, c16 = threadIdx.x & 15;
    const float *xr[2];
#pragma unroll
    for (int rt = 0; rt < 2; rt++) xr[rt] = a.X + min(row0 + 16 * rt + c16, a.rows - 1) * a.ldx;
    constexpr int U = 4;                                    // instructions whose operands are on their way together
#pragma unroll 1
    for (int k = 0; k < a.K; k += 4 * U) {
        float x[U][2], w[U][2 * NT];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int at = min(k + 4 * u + quarter, a.K - 1);
#pragma unroll
            for (int rt = 0; rt < 2; rt++) x[u][rt] = xr[rt][at];
#pragma unroll
            for (int t = 0; t < 2 * NT; t++) w[u][t] = a.W[(int64_t)at * a.N + min(col0 + column_of(t, c16), a.N - 1)];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool in = k + 4 * u + quarter < a.K;
#pragma unroll
            for (int t = 0; t < 2 * NT; t++)
#pragma unroll
                for (int rt = 0; rt < 2; rt++)
                    acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? x[u][rt] : 0.f, in ? w[u][t] : 0.f, acc[rt][t], 0, 0, 0);
        }
    }
}

// What a step's small magnitudes of X lost (x 2^scale below 2^kFloor), times W, by the fp32 matrix instructions.  Piece q of
// the step and element 4 quarter + i of it is element 4 q + i of the lane, as in the walk.
template <int NT>
__device__ __forceinline__ void add_lost(const DenseArgs &a, int64_t row0, int col0, int k0, int scale, f32x4 (&acc)[2][2 * NT])
{
    const int quarter = (threadIdx.x & 63) >> 4, c16 = threadIdx.x & 15;
#pragma unroll 1
    for (int q = 0; q < 2; q++) {
        const int owned = k0 + kDenseHalf * q, k = half_start(k0, q, a.K) + 4 * quarter;
        float lost[2][4];
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {
            const v4f x = *reinterpret_cast<const v4f_unaligned *>(a.X + min(row0 + 16 * rt + c16, a.rows - 1) * a.ldx + k);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float scaled = x[i] * power_of_two(scale), low_scaled = x[i] * (power_of_two(scale) * kLow);
                const float top = (float)(_Float16)scaled, rest = (float)(_Float16)fmaf(top, -kLow, low_scaled);
                const bool take = fabsf(scaled) < power_of_two(kFloor) && k + i >= owned && k + i < a.K;
                lost[rt][i] = take ? x[i] - ldexpf(fmaf(rest, 1.f / kLow, top), -scale) : 0.f;       // (exact)
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float w[2 * NT];
#pragma unroll
            for (int t = 0; t < 2 * NT; t++) w[t] = a.W[(int64_t)min(k + i, a.K - 1) * a.N + min(col0 + column_of(t, c16), a.N - 1)];
#pragma unroll
            for (int t = 0; t < 2 * NT; t++)
#pragma unroll
                for (int rt = 0; rt < 2; rt++)
                    acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(lost[rt][i], w[t], acc[rt][t], 0, 0, 0);
        }
    }
}

// Returns where the workgroup stopped: behind its last step, or at the start of a tile from which on the other walk
// is to go on.  The words of LDS, zero at the start, count the wavefronts' tiles that took more than a few
// corrections (`bad`) and those that are seen to need them in most steps while still under way (`early`).  Each is
// written only between barriers where nobody reads it: bad behind a tile's last step and read at its first (K is more than
// one step), early in a tile's second step of four and read in the fourth.
template <int NT>
__device__ __forceinline__ DenseStepAt walk_fp16(const DenseArgs &a, char (*w_lds)[kParts16 * NT * 32 * 64], DenseStepAt now,
                                                 int *bad, int *early)
{
    constexpr int kCols = NT * 32, kVecs = kCols * kParts16 * 4, kMine = kVecs / kDenseThreads;
    static_assert(kVecs % kDenseThreads == 0, "whole rounds of W");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int quarter = lane >> 4, c16 = lane & 15;
    const int lds_at = (int)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)w_lds);
    constexpr int kTiles = 2 * NT;             // of 16 columns
    static_assert(kTiles % kStore == 0, "whole vectors of Z");

    // x[2 t + q]: piece q of the step (16 k, see half_start) of row tile t
    // (addresses: a uniform part and an offset of 32 bits; rows past the end read the last one)
    auto fetch_x = [&](v4f (&x)[4], const DenseStepAt &at) __attribute__((always_inline)) {
        const int64_t row0 = min(at.row_block * kDenseBlockRows + wave * kDenseRows, a.rows - 1);
        const int last = (int)min((int64_t)kDenseRows, a.rows - row0) - 1;
        const float *xr = a.X + row0 * a.ldx;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint32_t by = ((uint32_t)min(16 * t + c16, last) * (uint32_t)a.ldx + 4u * (uint32_t)quarter) * 4u;
#pragma unroll
            for (int q = 0; q < 2; q++)
                x[2 * t + q] = *reinterpret_cast<const v4f_unaligned *>(
                    reinterpret_cast<const char *>(xr + half_start(at.k0, q, a.K)) + by);
        }
    };
    // W's block goes from memory into LDS without passing through registers, 16 bytes a lane to consecutive places.  The
    // compiler does not know of these loads.  Its own waits can only become longer by them (loads complete in
    // order), and step_barrier() waits for them: at most the kXLoads that follow them are still on their way.
    constexpr int kXLoads = 4;
    auto fetch_w = [&](const DenseStepAt &at, int buf) __attribute__((always_inline)) {
        const u32x4 *from = a.image + ((int64_t)at.tile * a.n_steps + at.k0 / kDenseStep) * kVecs;
#pragma unroll
        for (int i = 0; i < kMine; i++)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :: "s"(lds_at + buf * (int)sizeof(*w_lds) + (i * kDenseThreads + 64 * wave) * 16), "v"(tid * 16),
                            "s"(from + i * kDenseThreads) : "memory", "m0");
    };
    auto step_barrier = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(kXLoads) : "memory");
    };

    f32x4 high[2][kTiles], low[2][kTiles];     // sums of the first values' products, and of the mixed ones, times 2048
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int t = 0; t < kTiles; t++) high[r][t] = low[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int64_t stride = a.apart ? gridDim.x / a.n_col_tiles : gridDim.x;       // (as in the other walk)
    const int first_tile = a.apart ? now.tile : 0, last_tile = a.apart ? now.tile : a.n_col_tiles - 1;
    DenseStepAt next = now, after;
    next.advance(a.K, first_tile, last_tile, stride);
    after = next;
    after.advance(a.K, first_tile, last_tile, stride);
    v4f x0[4], x1[4];
    f16x8 apart[2][kParts16];                  // this step's values of X, taken apart
    int scale = 0, scale_next = 0;             // X is multiplied by 2^scale: in this step's tile, in the next step's
    uint64_t small = 0;                        // the tile's steps with magnitudes that are not carried in full (63: from there on)

    // The scale of a tile is found from the largest magnitude of its first step and of the tile before (of some
    // values of the tile, for the first): four times that does not fit and shows as sums that are not finite.
    float largest = 0.f;                       // of the tile so far, of this lane's values (a NaN stays out of it)
    auto look_at = [&](const v4f (&x)[4], bool first) __attribute__((always_inline)) {
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) m = fmaxf(m, fabsf(x[i / 4][i % 4]));
        largest = fmaxf(largest, m);
        if (first) {
            scale_next = scale_for(wave_max(__float_as_uint(largest)));
            largest = m;
        }
    };
    auto take_pair = [&](const v4f (&x)[4], int q, float by, uint32_t (&pair)[kParts16][8]) __attribute__((always_inline)) {
        take_apart16(x[q / 2][2 * (q & 1)], x[q / 2][2 * (q & 1) + 1], by, pair[0][q], pair[1][q]);
        asm volatile("" : "+v"(pair[0][q]), "+v"(pair[1][q]));      // (as in the other walk)
    };
    auto gather_pairs = [&](const uint32_t (&pair)[kParts16][8]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int p = 0; p < kParts16; p++)
                apart[i][p] = __builtin_bit_cast(f16x8, u32x4{pair[p][4 * i], pair[p][4 * i + 1], pair[p][4 * i + 2],
                                                              pair[p][4 * i + 3]});
    };
    auto small_of = [&](const v4f (&x)[4], int k0) __attribute__((always_inline)) {
        uint32_t least = 0xFFFFFFFFu;
#pragma unroll
        for (int i = 0; i < 16; i++) least = min(least, key_of(x[i / 4][i % 4]));
        const uint64_t bit = 1ull << min(k0 / kDenseStep, 63);
        return __any(least < key_of_power(kFloor - scale_next)) ? bit : 0;
    };

    fetch_w(now, 0);
    fetch_x(x0, now);
    {
        // some values of this wavefront's first tile: 64 places of four of its rows
        const int64_t row0 = min(now.row_block * kDenseBlockRows + wave * kDenseRows, a.rows - 1);
        const int k = min((int)((int64_t)lane * a.K / 64), a.K - 4);
#pragma unroll
        for (int q = 0; q < 4; q++)
            x1[q] = *reinterpret_cast<const v4f_unaligned *>(a.X + min(row0 + 8 * q, a.rows - 1) * a.ldx + k);
        look_at(x1, false);
    }
    fetch_x(x1, next);
    look_at(x0, true);
    scale = scale_next;
    small = small_of(x0, 0);
    {
        uint32_t pair[kParts16][8];
#pragma unroll
        for (int q = 0; q < 8; q++) take_pair(x0, q, power_of_two(scale), pair);
        gather_pairs(pair);
    }
    int step = 0, tiles_done = 0;
    // xf: free registers, for the step after the next; xn: the next step's X
    auto one = [&](v4f (&xf)[4], v4f (&xn)[4]) __attribute__((always_inline)) {
        const int buf = step & 1;
        // (xn, asked for a step ago, is waited for before more is asked for)
#pragma unroll
        for (int q = 0; q < 4; q++) asm volatile("" : "+v"(xn[q]) :: "memory");
        fetch_w(next, buf ^ 1);                // its readers were done at this step's barrier
        fetch_x(xf, after);
        __builtin_amdgcn_sched_barrier(0);     // the loads go out here, ahead of the matrix work that hides them
        const bool ends = next.k0 == 0;
        look_at(xn, ends);
        const uint64_t small_next = small_of(xn, next.k0);
        const float by = power_of_two(scale_next);

        f16x8 b[2][kParts16];
        auto read_b = [&](f16x8 (&to)[kParts16], int t) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < kParts16; p++) to[p] = reinterpret_cast<const f16x8 *>(w_lds[buf])[(p * kTiles + t) * 64 + lane];
        };
        uint32_t pair[kParts16][8];
        read_b(b[0], 0);
#pragma unroll
        for (int t = 0; t < kTiles; t++) {
            if (t + 1 < kTiles) read_b(b[(t + 1) & 1], t + 1);
#pragma unroll
            for (int r = 0; r < 2; r++) low[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(apart[r][1], b[t & 1][0], low[r][t], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 2; r++) high[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(apart[r][0], b[t & 1][0], high[r][t], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 2; r++) low[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(apart[r][0], b[t & 1][1], low[r][t], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (q * kTiles / 8 == t) take_pair(xn, q, by, pair);
            __builtin_amdgcn_sched_barrier(0);
        }
        gather_pairs(pair);

        if (ends) {                            // that was the last step of this tile: store it, start the next at zero
            const int64_t row0 = now.row_block * kDenseBlockRows + wave * kDenseRows;
            // (read by the scalar unit: a vector load would be waited for behind those of X on their way)
            const int unscale = -(scale + reinterpret_cast<constant_int *>(reinterpret_cast<uintptr_t>(a.head))[1 + now.tile]);
            bool good = true;
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int t = 0; t < kTiles; t++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        high[r][t][v] = ldexpf(fmaf(low[r][t][v], 1.f / kLow, high[r][t][v]), unscale);
                        good &= __builtin_isfinite(high[r][t][v]);
                    }
            const bool again = __any(!good);
            if (again || small != 0) {
                if (again) {
#pragma unroll
                    for (int r = 0; r < 2; r++)
#pragma unroll
                        for (int t = 0; t < kTiles; t++) high[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
                    add_in_fp32_by_16<NT>(a, row0, now.tile * kCols, high);
                } else {
#pragma unroll 1
                    for (int k0 = 0; k0 < a.K; k0 += kDenseStep)
                        if (small >> min(k0 / kDenseStep, 63) & 1) add_lost<NT>(a, row0, now.tile * kCols, k0, scale, high);
                }
                if (lane == 0 && (again || 4 * (int)__popcll(small) > min(a.n_steps, 64))) atomicAdd(bad, 1);
            }
            float *z = a.Z + row0 * a.ldz + now.tile * kCols;
            uint32_t lane_at = (uint32_t)(4 * quarter) * (uint32_t)a.ldz + (uint32_t)(kStore * c16);
            asm volatile("" : "+v"(lane_at));  // (the stores' addresses are formed here, not kept from tile to tile)
            const int64_t rows = a.rows - row0 - 4 * quarter;
            const int cols = a.N - now.tile * kCols - kStore * c16;
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    float *zr = z + (16 * r + v) * a.ldz;
#pragma unroll
                    for (int g = 0; g < kTiles / kStore; g++) {
                        v4f to;
#pragma unroll
                        for (int i = 0; i < kStore; i++) to[i] = high[r][g * kStore + i][v];
                        // (streaming: 1 M x 602 times 602 x 128 0.71 -> 0.70 ms, 608 0.665 -> 0.645)
                        if (16 * r + v < rows && 16 * kStore * g + kStore <= cols) {
                            __builtin_nontemporal_store(to, reinterpret_cast<v4f_unaligned *>(zr + 16 * kStore * g + lane_at));
                        } else if (16 * r + v < rows) {
#pragma unroll
                            for (int i = 0; i < kStore; i++)
                                if (16 * kStore * g + i < cols) (zr + 16 * kStore * g + i)[lane_at] = to[i];
                        }
                    }
                }
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int t = 0; t < kTiles; t++) high[r][t] = low[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            small = 0;
            tiles_done++;
        }
        small |= small_next;
        const int in_four = now.k0 / kDenseStep % 4;
        if (in_four == 1 && !ends && lane == 0 && 2 * (int)__popcll(small) > now.k0 / kDenseStep + 2) atomicAdd(early, 1);
        scale = scale_next;
        now = next;
        next = after;
        after.advance(a.K, first_tile, last_tile, stride);
        step++;
    };
    // At a barrier: this step's block of W is in place, the other one's readers are done, and what was counted is there.
    auto go_on = [&]() __attribute__((always_inline)) {
        step_barrier();
        if (now.row_block >= a.n_row_blocks) return false;
        if (now.k0 == 0 && tiles_done > 0) {
            const int n = *bad;
            return n < 2 || n < tiles_done;
        }
        if (now.k0 / kDenseStep % 4 == 3 && *early > max(1, tiles_done)) {
            now.k0 = 0;
            return false;
        }
        return true;
    };
    for (;;) {
        if (!go_on()) break;
        one(x0, x1);
        if (!go_on()) break;
        one(x1, x0);
    }
    return now;
}

template <int NT>
__global__ __launch_bounds__(kDenseThreads, 2) void dense_xw_fp16_kernel(DenseArgs a)
{
    __shared__ __attribute__((aligned(16))) char w_lds[2 * kParts * NT * 32 * kWStride];
    __shared__ int bad, early;
    DenseStepAt at = first_step(a);
    if (at.row_block >= a.n_row_blocks) return;             // (uniform; of the last eight blocks of rows, with tiles apart)
    if (!a.head[0]) {
        if (threadIdx.x == 0) bad = early = 0;
        at = walk_fp16<NT>(a, reinterpret_cast<char (*)[kParts16 * NT * 32 * 64]>(w_lds), at, &bad, &early);
    }
    if (at.row_block < a.n_row_blocks)
        walk_bf16<NT>(a, reinterpret_cast<char (*)[kParts * NT * 32 * kWStride]>(w_lds), at);
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

static int dense_launch(void (*kernel)(DenseArgs), int which, DenseArgs a, hipStream_t s)
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
    unsigned grid = (unsigned)(a.n_row_blocks < resident ? a.n_row_blocks : resident);
    // Column tiles in workgroups of their own: where that is fewer tiles one after the other in a workgroup, and where the blocks
    // of rows are more than are under way at once: the tiles of a block are worked on together then, by
    // one die, whose L2 has the rows of X that they share; one after the other they are fetched for each tile.  Rows x K x N, in turn
    // and so: 200,000 x 602 x 256 287 and 246 us, 100,000 x 250 x 160 75 and 60, 500,000 x 512 x 256 520 and 470, 2.45 M x 512
    // x 256 2,423 and 2,340, 300,000 x 100 x 515 328 and 263, 30,000 x 100 x 300 31.4 and 27.4.  As many either way, and at
    // once: 50,000 x 602 x 256 75.0 and 76.0, 60,000 x 40 x 200 23.0 and 23.6.
    if (a.apart) {
        const int64_t set = (int64_t)kXcds * a.n_col_tiles;   // workgroups: the tiles of eight blocks of rows, one per die
        const int64_t sets = (a.n_row_blocks + kXcds - 1) / kXcds, at_once = resident / set;
        a.apart = at_once > 0 && ((sets + at_once - 1) / at_once < a.n_col_tiles * ((a.n_row_blocks + resident - 1) / resident) ||
                                  a.n_row_blocks > resident);
        if (a.apart) grid = (unsigned)(std::min(sets, at_once) * set);
    }
    kernel<<<grid, kDenseThreads, 0, s>>>(a);
    return ACCEL_OK;
}

// Two fp16 values from K = 64 on (below, they are no more exact than three bf16 values) for products of this many
// multiplications and more: two launches in front, 6 us, for a quarter of the time.  Three parts and two:
// 128 columns: 100,000 x 64 22.7 and 23.5 us, 20,000 x 602 38 and 31, 170,000 x 128 48 and 40, 50,000 x 602 61 and 44; 64
// columns: 20,000 x 256 12.6 and 17.9, 170,000 x 128 28.9 and 31.5, 2.45 M x 128 362 and 336, 1 M x 602 673 and
// 586.  32 columns are bound by reading X, which walk_bf16 does in whole lines there: 2.45 M x 100 269 and 280 us.
constexpr int kFp16FromK = 64;
template <int NT> constexpr double kFp16From = NT == 4 ? 1e9 : 4e9;
constexpr int64_t kFp16MaxStride = 1 << 24;              // (offsets inside 32 rows are 32 bits wide)

template <int NT>
static int dense_product(DenseArgs a, hipStream_t s, bool may_prepare)
{
    constexpr int which = NT == 1 ? 0 : NT == 2 ? 4 : 8;
    if (a.K <= 2) return dense_launch(dense_short_kernel<NT, true>, which, a, s);
    if (a.K < kDenseHalf) return dense_launch(dense_short_kernel<NT, false>, which + 1, a, s);
    if constexpr (NT > 1) {
        const bool pays = a.K >= kFp16FromK && (double)a.rows * a.K * a.N >= kFp16From<NT>;
        void *mem = nullptr;
        const size_t blocks = (size_t)a.n_col_tiles * (size_t)a.n_steps;
        const size_t head_bytes = head_words(a.n_col_tiles, blocks) * sizeof(int);
        if (may_prepare && pays && a.ldx <= kFp16MaxStride && a.ldz <= kFp16MaxStride)
            mem = take_stream_memory(head_bytes + blocks * (NT * 32 * kParts16 * 4) * sizeof(u32x4), s);
        if (mem) {
            int *head = static_cast<int *>(mem);
            u32x4 *image = reinterpret_cast<u32x4 *>(static_cast<char *>(mem) + head_bytes);
            a.image = image;
            a.head = head;
            dense_range_kernel<NT><<<dim3((unsigned)blocks), kDenseThreads, 0, s>>>(a, head);
            dense_prepare_kernel<NT><<<dim3((unsigned)blocks), kDenseThreads, 0, s>>>(a, head, image);
            const int rc = dense_launch(dense_xw_fp16_kernel<NT>, which + 2, a, s);
            give_stream_memory(mem, s);
            return rc;
        }
    }
    return dense_launch(dense_xw_kernel<NT>, which + 3, a, s);
}

// Few rows: a workgroup takes one column tile, and a narrower one, as long as there is a compute unit for each.  A step takes a microsecond whatever its width.  Rows x K x N, 128 columns and all tiles to a workgroup
// and so: 2,000 x 250 x 256 31.0 -> 9.4 us, 10,000 x 602 x 128 32.7 -> 21.3, 10,000 x 602 x 256 48.4 -> 29.9, 20,000 x
// 602 x 256 48.7 -> 39.3.  Beyond the line: 20,000 x 602 x 64 in halves (314 workgroups) 21.4 -> 25.6.
constexpr int64_t kFewGroups = 256;
// Arguments have been checked by the caller (accel_dense_xw): rows >= 1, K, N >= 1,
// ldx >= K, ldz >= N, operands readable and large enough.  may_prepare: s is not capturing (a graph's
// memory would have to live as long as the graph).
int dense_xw_launch(const float *X, const float *W, float *Z, int64_t rows, int K, int N, int64_t ldx, int64_t ldz,
                    hipStream_t s, bool may_prepare)
{
    (void)hipGetLastError();
    int nt = N <= 32 ? 1 : N <= 64 ? 2 : 4;
    DenseArgs a{};
    a.X = X; a.W = W; a.Z = Z;
    a.rows = rows; a.ldx = ldx; a.ldz = ldz;
    a.n_row_blocks = (rows + kDenseBlockRows - 1) / kDenseBlockRows;
    a.K = K; a.N = N;
    a.n_steps = (K + kDenseStep - 1) / kDenseStep;
    auto groups = [&](int of) { return a.n_row_blocks * ((N + of * 32 - 1) / (of * 32)); };
    if (K >= kDenseHalf) {
        while (nt > 1 && groups(nt / 2) <= kFewGroups) nt /= 2;
        a.apart = groups(nt) > a.n_row_blocks;
    }
    a.n_col_tiles = (N + nt * 32 - 1) / (nt * 32);
    const int rc = nt == 1   ? dense_product<1>(a, s, may_prepare)
                   : nt == 2 ? dense_product<2>(a, s, may_prepare)
                             : dense_product<4>(a, s, may_prepare);
    if (rc) return rc;
    ACCEL_HIP(hipGetLastError());
    return ACCEL_OK;
}

}  // namespace accel
