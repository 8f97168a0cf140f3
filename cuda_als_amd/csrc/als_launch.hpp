// Kernel argument blocks and launchers shared by the engine (host) and the
// device code. Internal to the library: the public boundary is include/als.h.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace als {

enum Prec { PREC_FP32 = 0, PREC_BF16 = 1, PREC_FP16 = 2 };
// SOLVE_CHOL_WARM: one warm-started refinement step and no other (its own
// kernel: without the classic residual code the registers fit without spills).
enum SolveKind { SOLVE_CHOL = 0, SOLVE_CG = 1, SOLVE_CHOL_REFINE = 2, SOLVE_CHOL_WARM = 3 };
constexpr int MAX_T = 9;  // augmented dimension f + 1 <= 16 * MAX_T

// The system a row solves is held in T x T blocks of 16. b = sum r y rides
// along as row f of an augmented matrix where the last block has room for it
// (f % 16 != 0); where f is a multiple of 16 that row would take a block of
// its own (T + 1 more 16x16 tiles: 15 instead of 10 at f = 64, 45 instead of
// 36 at f = 128), and b is summed beside the tiles instead. One sweep at the
// ml10M shape (69,878 x 10,677, 9.0M ratings), row in the tiles -> beside:
// f = 80 FP16 Gram and CG 0.80 -> 0.70 ms, f = 64 FP32 1.71 -> 1.50 ms, three
// warm-started BF16 models of f = 32, 64, 128 together 3.25 -> 2.79 ms.
constexpr int tiles(int f) { return (f + 15) / 16; }
constexpr bool augmented(int f) { return f % 16 != 0; }
// Row stride (floats) of every factor matrix: the augmented system's, whatever
// the solve uses.
constexpr int row_stride(int f) { return 16 * ((f + 16) / 16); }
// Row stride (halves) of the 16-bit shadows, which only the kernels see: 16T,
// rounded up to a multiple of 64 bytes above one block, so that a row touches
// as few 128-byte cache lines as its length allows. The rows are gathered in
// the order of the ratings, and what a gather costs is its lines: reading rows
// of random users (480,189 of them) took 0.724 ms at 224 bytes a row (f = 100,
// 2.5 lines) and 0.579 at 256 (2 lines), 0.486 at 160 bytes (f = 64 in an
// augmented row's stride) and 0.312 at 128, 0.855 at 288 (f = 128) and 0.580
// at 256. One sweep: the netflix shape, mixed, f = 100 6.79 -> 6.42 ms; three
// BF16 models of f = 32, 64, 128 at the ml10M shape 2.31 -> 2.26 ms.
constexpr int shadow_stride_tiles(int T) { return 16 * T + (T > 1 && T % 2 == 1 ? 16 : 0); }
constexpr int shadow_stride(int f) { return shadow_stride_tiles(tiles(f)); }
// Floats of one part of a split row or of one copy of a system: its tiles,
// and b where it is not in them.
constexpr int part_floats(int f) { return tiles(f) * (tiles(f) + 1) / 2 * 256 + (augmented(f) ? 0 : f); }
// Floats of one row's saved factor.
constexpr int factor_floats(int f) { return tiles(f) * (tiles(f) + 1) / 2 * 256; }

struct UpdateArgs {
    const int *ptr;             // CSR of the side being updated (int32, reference layout)
    const int *idx;
    const float *val;
    const float *Y;             // fixed factors, FP32, row stride row_stride(f)
    const uint16_t *Ys;         // fixed factors, 16-bit shadow, row stride shadow_stride(f) (16-bit Gram only)
    float *X;                   // updated factors, FP32, the same stride (CG: warm start in)
    uint16_t *Xs;               // 16-bit shadow of X to refresh, the shadows' stride (nullable)
    const float *lambda_rows;   // per-row lambda (nullable -> lambda)
    float lambda;
    int f;
    const int4 *units;          // {row, kb, ke, split} work units, heaviest first
    const int4 *splits;         // {slot_base, nparts, part_len, -} per split row
    int *counters;              // arrivals per split row (0 between launches)
    float *partial;             // partial Gram tiles (and b), part_floats(f) per slot
    const int *batch_begin;     // batch b = units[batch_begin[b] .. batch_begin[b+1])
    int nbatches;
    int *queue;                 // next ticket (0 between launches)
    int cg_iters;
    float cg_tol;
    int cg_fp16_a;              // CG on an FP16-rounded A
    int refine;                 // FP64-residual refinement steps (Cholesky)
    int refine_warm;            // first refinement step from the row's previous value in X
    int restage_max;            // whole rows up to this many ratings form the residual by
                                // restaging their ratings; longer ones use the tile copy
    int *fail_count;            // rows whose solve broke down (x set to 0)
    float *Lsave;               // Cholesky factor tiles per row, factor_floats(f) (nullable)
    float *scratch;             // per-wave copy of A (and b) for refinement, part_floats(f) per workgroup
    const float *zero32;        // one row of zeros (row_stride(f) floats) read by unused chunk slots
    const uint16_t *zero16;     // same, 16-bit
    int ys_bytes;               // bytes of the 16-bit Y shadow when below 2^31 (the pipelined
                                // Gram then gathers with 32-bit buffer offsets), else 0
    int y_bytes;                // bytes of Y when below 2^31 (the FP32 Gram's gathers), else 0
    int gram_dma;               // 1: the 16-bit Gram gathers straight to LDS where built
                                // (gram_dma_built), 0: through registers
};

// Augmented tile counts (als_info.T) and precisions whose update kernels carry
// the LDS-DMA Gram: a 16-bit Gram, at most 8 tiles (a chunk's gather tasks fit
// a wave) and T % 4 != 0 (the rating column of an augmented system would need
// the banks' permutation of gram_dma_loop). f = 48, 112 and 128 go by the same
// count, though their kernels of one block fewer would meet these conditions:
// they gather through registers.
constexpr bool gram_dma_built(int T, int prec) { return prec != PREC_FP32 && T <= 8 && T % 4 != 0; }

constexpr int MAX_MODELS = 4;  // engines per group (als_group_*)

struct AdjointArgs {
    const int *ptr;             // CSR of the side that was updated
    const float *X;             // forward solution, stride row_stride(f)
    const float *Lsave;         // packed factors from the forward pass
    const float *Gbar;          // dL/dX, the same stride
    float *Xbar;                // A^-1 Gbar, the same stride
    float *lambda_bar;          // -n_u Xbar_u . X_u
    int rows;
    int f;
};

// Batched CG on caller-provided dense systems (the reference's
// updateXWithCGHost boundary): A batch x f x f (symmetric, either order),
// x and b batch x f, all densely packed.
struct CgBatchArgs {
    const float *A;             // FP32 systems, or nullptr when A16 is set
    const uint16_t *A16;        // FP16 systems
    int round_a16;              // FP32 systems whose entries are rounded to FP16 on load
    int vec;                    // f % 4 == 0 and A 16-byte (A16 8-byte) aligned: a lane
                                // loads its four entries of a tile in one load
    float *x;                   // warm start in, solution out
    const float *b;
    int batch;
    int f;
    int iters;
    float tol;
};

struct YbarArgs {
    const int *cptr;            // CSC of the same matrix (columns = fixed-factor rows)
    const int *cidx;
    const float *cval;
    const float *X, *Xbar, *Y;  // stride row_stride(f)
    float *Ybar;                // the same stride (overwritten)
    int ncols;
    int f;
    // the columns' rating lists cut into parts of at most YBAR_PART ratings:
    // part p = {column, first rating, end}; column c's parts are
    // colpart[c] .. colpart[c+1]-1, in order; partial: one row per part
    const int4 *parts;
    const int *colpart;
    float *partial;             // nparts x 16 tiles(f)
    int nparts;
};
constexpr int YBAR_PART = 1024;

struct RmseArgs {
    const int *row, *col;
    const float *val;
    const float *U, *V;         // stride ld
    int64_t n;
    int f, ld;
    double *partials;           // one per block
};

// Launchers (als_kernels_*.hip). Each returns the hipError_t of the launch.
int update_lds_bytes(int f, int prec, int solve);
// variant 0: the solver's usual kernel (two waves per SIMD for the refinement
// solvers); variant 1: one wave per SIMD (warm-started refinement, f >= 96;
// null elsewhere).
hipError_t launch_update(int f, int prec, int solve, int variant, const UpdateArgs &a, int grid, int lds_bytes,
                         hipStream_t s);
const void *update_kernel_ptr(int f, int prec, int solve, int variant = 0);
// Light rows through the dual system, one launch per half-sweep after the
// update kernel (null / 0 where the variant has no dual system: f < 64, CG,
// classic refinement). dual_max_ratings: rows below it take the dual system.
const void *dual_kernel_ptr(int f, int prec, int solve);
int dual_lds_bytes(int f, int prec);
int dual_max_ratings(int f, int prec);
hipError_t launch_dual(int f, int prec, int solve, const UpdateArgs &a, int grid, int lds_bytes, hipStream_t s);
hipError_t launch_adjoint_solve(const AdjointArgs &a, hipStream_t s);
hipError_t launch_cg_batch(const CgBatchArgs &a, hipStream_t s);
hipError_t launch_ybar(const YbarArgs &a, hipStream_t s);
// RMSE partial sums of a.n ratings over `blocks` blocks into a.partials
// (blocks doubles), then out[0] = their sum (with_rmse: out[1] = sqrt(sum / n)).
constexpr int RMSE_BLOCKS = 1024;
hipError_t launch_rmse(const RmseArgs &a, int blocks, double *out, bool with_rmse, hipStream_t s);
// The 16-bit shadow of `rows` factor rows (row_stride(f) floats each).
hipError_t launch_to16(int f, int prec, const float *src, uint16_t *dst, int64_t rows, hipStream_t s);

}  // namespace als
