// Kernel parameter blocks and launchers shared between the kernel sources and
// the host engine.  Only plain C types cross this header.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pqb {

struct ddc;

// Plain permanents (R rows, NC columns, R <= NC + 1), one per grid row
// (blockIdx.y = matrix index; a single matrix is a grid of height 1).
struct PlainParams {
    const double2* M2;   // per matrix 2R x NC, packed: rows [0,R) = +2A, rows [R,2R) = -2A
                         // expanded matrices: the 2(R-1) x NC table of the scaled rows,
                         // then the product of the scales (ddc); see perm_expand.hip
    int64_t m2_stride;   // elements between consecutive matrices' M2 (2 R NC)
    int R;               // rows
    int K;               // Gray bits walked inside a chunk (rows R-K .. R-1)
    int B;               // lane bits (rows R-K-B .. R-K-1), B <= 6
    int H;               // group bits (rows 1 .. R-1-K-B), K + B + H = R - 1
                         // (expanded: R - 1 rows, K + B + H = R - 2)
    int by_flag;         // 1: only the matrices whose counter flag says this kernel
    ddc* partials;       // one dd complex per block, gridDim.x per matrix
    unsigned* counter;   // one per matrix, zero on entry (or kExpandedFlag, from the prep kernel);
                         // the last block restores it to zero
    double* out;         // 6 per matrix: [re, im, hi_re, lo_re, hi_im, lo_im]
    double scale;        // 2^-(R-1)
    unsigned* done;      // host memory, set to 1 after `out` (NULL: not wanted)
};

// Several shapes in one launch of blocks of 256 threads (plain_mixed_kernel).  The upper
// limit was measured on one list (see there), not over many.
constexpr int kMixedMinCols = 11, kMixedMaxCols = 21, kMixedShapes = 16;
struct PlainMixed {
    PlainParams p[kMixedShapes];
    int nc[kMixedShapes];
    unsigned blocks[kMixedShapes];     // per matrix
    unsigned first[kMixedShapes + 1];  // first block of each shape, then their total
    int shapes;
};
hipError_t launch_plain_mixed(const PlainMixed& m, hipStream_t st);

// The same sum with products in exact doubles (perm_exact.hip).
constexpr int kExactBlock = 1024;  // threads per block at most
struct ExactF64Params {
    const double* A2;    // R x NC, packed: 2 a_ij
    int R, K, B, H;      // walk, lane (<= 6) and group bits, K + B + H = R - 1; a wave per group
    int flush;           // steps between flushes, even
    unsigned long long* partials;  // two words per block
    unsigned* counter;
    unsigned long long* out;
    unsigned* done;      // as in PlainParams
};

// Square matrices from this size on may be swept in expanded form (perm_expand.hip);
// plain_expand_kernel decides per matrix and sets this bit of the matrix's counter.
constexpr int kExpandedMinCols = 14;
constexpr unsigned kExpandedFlag = 0x80000000u;

// Exact integer sweep (sum kept modulo 2^128).
struct ExactParams {
    const int* A;        // R x NC integers, packed
    int R, K, H;
    int group;           // column sums per 64-bit partial product (2, 6 or 13), with
                         // (max_j sum_i |a_ij|)^group < 2^63
    int64_t nlanes;      // = 2^H
    unsigned long long* partials;  // two words per block
    unsigned* counter;
    unsigned long long* out;       // [lo, hi] of sum_delta (...) mod 2^128
};

// ---- one block per matrix (perm_tiny.hip) ----
constexpr int kTinyDigits = 12;    // rows besides the anchor
constexpr int kTinySteps = 2048;   // signed terms (repeated-row tasks)
constexpr int kTinyRows = 11;      // rows of a plain permanent
constexpr int kTinySlots = 24;     // columns (column slots)
struct TinyParams {
    const double2* A;      // per matrix R x NS, packed: row 0 the anchor, row 1 + d digit d's
    int64_t stride;        // elements between consecutive matrices
    double* out;           // 6 per matrix (RepBatchParams::out)
    double scale;          // 2^-(N-1)
    unsigned* done;        // as in PlainParams; one matrix only
    int R, S, P, nlow;     // S = product of the radices, P = that of the first nlow
    unsigned lds_bytes;
    unsigned char radix[kTinyDigits];  // multiplicity + 1
};
// Fills the split of the digits whose radices are set; false: not for this kernel.
bool tiny_split(TinyParams& p, int NS, int R);
hipError_t launch_tiny(int ns, const TinyParams& p, int64_t count, hipStream_t st);
// Several shapes in one launch.
constexpr int kTinyShapes = 16;
struct TinyMixed {
    TinyParams p[kTinyShapes];
    unsigned first[kTinyShapes + 1];  // first block of each shape, then their total
    unsigned char ns[kTinyShapes];
    int shapes;
};
hipError_t launch_tiny_mixed(const TinyMixed& m, hipStream_t st);

// ---- repeated-row / batched sweep ----
// A row of multiplicity D <= kMaxDegree may be expanded (plan_task): the columns are
// divided by its entries and its digit is replaced by a term of degree D.  Tasks that are
// expanded have at least kExpandedMinSlots slots.
constexpr int kMaxDegree = 3;
constexpr int kExpandedMinSlots = 13;
constexpr int kMaxDigits = 40;
constexpr int kMaxSlots = 40;
constexpr int kMaxRepRows = kMaxDigits + 1;  // anchor and digits
constexpr int kBinomStride = 41;  // binomial table: binom[m * 41 + k], 0 <= k <= m <= 40

struct RepStep {          // one step of the low-digit Gray walk
    uint32_t row;         // row of A whose digit moves (low digit d lives in row 1 + d)
    uint32_t dir;         // 1: k += 1 (colsum -= 2a), 0: k -= 1 (colsum += 2a)
    double w;             // prod_low (-1)^k C(m, k) after the step (exact integer)
};

struct RepTask {
    const double2* A;      // R x NS: a_i (slots expanded); row 0 is the anchor, rows
                           // 1..nlow the low digits (in walk order), then the high digits
    const double2* base;   // NS: a_anchor + sum_{low i} m_i a_i  (seed of every chunk before high digits)
    const RepStep* table;  // L entries, entry t = step into Gray index t (entry 0 unused)
    int NS;                // column slots
    int L;                 // low-walk length = prod_low (m_i + 1)
    int nhigh;             // high digits
    int nlow;              // low digits (rows 1 .. nlow of A)
    uint32_t item0;        // first work item of this task (items of a task are contiguous)
    uint32_t nitems;
    uint32_t out_index;    // result slot
    uint32_t nchunks;      // prod_high (m_i + 1)
    int degree;            // 0: term prod_s c_s; D > 0: the coefficient of x^D in prod_s (c_s + x)
    int rows;              // rows of A
    const double2* xrow;   // expanded: NS, the expanded row r
    double scale[4];       // double-double complex: 2^-(N-1); expanded: D! 2^-(N-D-1), times
                           // prod_s a_rs once rep_layout_kernel has run
    uint32_t hrow[kMaxDigits];  // row (in A) of high digit h
    uint32_t hrad[kMaxDigits];  // radix m_h + 1 of high digit h (digit 0 varies fastest)
    uint32_t lrad[kMaxDigits];  // radix m_d + 1 of low digit d (row 1 + d); read by the
                                // double-double sweep, which seeds chunks from A exactly
    // double-double sweep: rows + 1 rows of the entries' parts (hi, lo) on and below a grid on
    // which no column sum rounds, the last row being the base, laid out for the lanes of a
    // chunk (fill_split in batch.hip); NULL: not in such a range
    const double2* split;
    const double2* src;    // A and base are taken from this matrix by rep_layout_kernel
                           // (row stride src_ld); NULL: they are in place
    int64_t src_ld;
    uint32_t transpose;    // rows are the matrix's columns
    uint32_t src_xrow;     // the expanded row
    uint32_t src_row[kMaxRepRows], src_slot[kMaxSlots];
};

struct RepItem {
    uint32_t task;
    uint32_t count;   // chunks in the item
    uint32_t chunk0;  // first chunk
    uint32_t pad;
};

struct RepBatchParams {
    const RepTask* tasks;
    const RepItem* items;
    const unsigned* order;  // processing order of the items (largest first)
    const double* binom;    // binomial table
    ddc* partials;          // one per item
    double* out;            // 6 doubles per task result
    unsigned* head;         // item counter, zero on entry; the reduce kernel resets it
    unsigned* done;         // as in PlainParams; one task only
    const unsigned* counts; // device: counts[0] = items, counts[1] = tasks (read by the
                            // kernels, so a captured graph serves every batch that fits)
};

constexpr int kReduceBlocks = 512;   // grid of the per-task reduction in a captured graph
constexpr int kReduceThreads = 256;  // one block of four waves per task

// Kernel instantiations cover slot ranges; rep_range_for() picks the narrowest
// one for a batch (-1: the batch needs splitting at 32 slots).
// Rows and bases of the tasks whose matrix is elsewhere; the expanded tasks' are divided by
// their expanded rows.
hipError_t launch_rep_layout(RepTask* tasks, int64_t ntasks, hipStream_t st);
int rep_range_for(int min_ns, int max_ns);
const void* rep_batch_kernel_fn(int range);
hipError_t launch_rep_batch(int range, const RepBatchParams& p, int grid_blocks, int reduce_blocks, hipStream_t st);
// per-task sum of the item partials (shared by the FP64 and double-double sweeps)
hipError_t launch_rep_reduce(const RepBatchParams& p, int blocks, hipStream_t st);

// Double-double sweep over the same tasks and items (precision PQB_PREC_INF).
// Ranges from kDDRange0 on cover up to 8, 16, 32 and 40 slots with a chunk per 1, 2, 4 and
// 4 lanes, then, rows split (RepTask::split), up to 8, 16, 24, 32 and 40 with one per 1, 2,
// 2, 4 and 4; rep_dd_walkers() = chunks per wave.
constexpr int kDDRange0 = 5;
constexpr int kRanges = kDDRange0 + 9;
int rep_dd_range_for(int max_ns, bool split);
int rep_dd_walkers(int range);
const void* rep_dd_kernel_fn(int range);
hipError_t launch_rep_dd(int range, const RepBatchParams& p, int grid_blocks, int reduce_blocks, hipStream_t st);

// ---- adjoint sweep (permanent + all first derivatives of square matrices) ----
// Adjoint mode: square n x n matrices.  Minors mode: n x (n+1) matrices, the
// n+1 permanents with one column deleted.
struct GradParams {
    const double2* A;    // count x n x cols, packed row-major
    double2* partials;   // count x (wpt / 4) x E, one per block.  Adjoint: E = n*n (G
                         // row-major); minors: E = cols
    int n;               // rows
    int cols;            // columns: n (adjoint) or n + 1 (minors)
    int L;               // delta-lane bits (<= 4)
    int H;               // high bits: K + L + H = n - 1 (K is the kernel's template argument)
    int wpt;             // waves per task, multiple of 4
};

struct GradReduceParams {
    const double2* partials;  // count x nblk x (main + (tail ? 1 : 0))
    double2* out;        // count x main
    double2* tail;       // count, or NULL
    int main, nblk, count;  // nblk: partials (blocks) per task
    double scale;        // 2^-(n-1)
};

const void* grad_kernel_fn(int M, int K, bool minors);
hipError_t launch_grad(int M, int K, bool minors, const GradParams& p, int nblocks, size_t lds_bytes,
                       hipStream_t st);
hipError_t launch_grad_reduce(const GradReduceParams& p, hipStream_t st);
// perm = sum_j a_0j G_0j per matrix (A, G packed count x n x n)
hipError_t launch_grad_perm(const double2* A, const double2* G, double2* perm, int n, int count, hipStream_t st);

// expanded: the sweep of expanded tables (square, nc >= kExpandedMinCols)
hipError_t launch_plain(int nc, bool expanded, const PlainParams& p, int nblocks, int bdim, int ntasks,
                        hipStream_t st);
// Tables and counters of `count` packed n x n matrices, M2 stride 2 n n.
hipError_t launch_plain_expand(const double2* A, double2* M2, int n, int64_t count, unsigned* counters,
                               hipStream_t st);
hipError_t launch_plain_prep(const double2* A, double2* M2, int n, int64_t count, hipStream_t st);
hipError_t launch_plain_exact_fp64(int nc, const ExactF64Params& p, int nblocks, int bdim, hipStream_t st);
hipError_t launch_plain_exact(int nc, const ExactParams& p, int nblocks, int bdim, hipStream_t st);
const void* plain_kernel_fn(int nc, bool expanded);
// The row an n x n host matrix (row stride ld) is expanded along, -1 for none: the
// choice plain_expand_kernel makes.
int plain_expand_row(const double* A, int n, int64_t ld);

constexpr int kMaxCols = 40;

}  // namespace pqb
