// Tables of the expanded sweeps: perm(A) of a square matrix by expansion
// along one row r,
//
//     perm(A) = sum_j a_rj perm(A without row r and column j)
//             = (prod_j a_rj) sum_j perm(S without column j),   S_ij = a_ij / a_rj, i != r,
//
// so that the sign-vector sum runs over the n-1 rows of S and each vector's term
// is the coefficient of x in prod_j (c_j + x), c = the column sums of S: half as
// many vectors as the sum over all n rows (BBFGPermanentCalculator.hpp:87-235),
// at 10 n instead of 2 x 6 n FP64 instructions per pair of them
// (add_expanded_term in perm_plain.hip).
//
// One block per matrix.  The row with the largest smallest entry is expanded;
// a matrix keeps the all-rows table when
//  * a row without an entry below 2^-16 of the matrix's largest and outside
//    [2^-20, 2^20] does not exist (zeros, sparse rows): the scaled column sums
//    are then below 40 x 2^16.5, their products over 40 columns and the sum over
//    2^39 vectors below 2^950, and the product of the scales is above 2^-800;
//  * an entry is not finite or beyond 2^20;
//  * every entry is a (Gaussian) whole number of up to 21 bits times a power of two that
//    they share: small ones sum without rounding, which a division would lose (rows of
//    +-1.5 among +-0.5 at n = 14: 1572.0000000000118 for 1572).
// The rule itself is in pqb_pivot.h.
// Repeated-row tasks (batch.hip plans them) are divided here too: a row of multiplicity D
// contributes the coefficient of x^D, times D!.
//
// Quotients are formed in double-double and rounded once, the product of the
// scales is kept in double-double, so the scaling adds half an ulp per entry.
//
// This unit is compiled without contraction: the exact product splits would
// otherwise be fused away.

#include <algorithm>
#include <cmath>

#include "pqb_device.h"
#include "pqb_kernels.h"
#include "pqb_pivot.h"

namespace pqb {

namespace {

struct dd {
    double h, l;
};

__device__ __forceinline__ dd dd_prod(double a, double b) {
    const double p = a * b;
    return {p, __builtin_fma(a, b, -p)};
}

__device__ __forceinline__ dd dd_sum(dd a, dd b) {
    dd_add(a.h, a.l, b.h, b.l);
    return a;
}

__device__ __forceinline__ dd dd_times(dd a, dd b) {
    const dd p = dd_prod(a.h, b.h);
    dd r;
    fast_two_sum(p.h, p.l + (a.h * b.l + a.l * b.h), r.h, r.l);
    return r;
}

__device__ __forceinline__ ddc ddc_times(const ddc& a, const ddc& b) {
    const dd rr = dd_times({a.hr, a.lr}, {b.hr, b.lr}), ii = dd_times({a.hi, a.li}, {b.hi, b.li});
    const dd ri = dd_times({a.hr, a.lr}, {b.hi, b.li}), ir = dd_times({a.hi, a.li}, {b.hr, b.lr});
    const dd re = dd_sum(rr, {-ii.h, -ii.l}), im = dd_sum(ri, ir);
    return {re.h, re.l, im.h, im.l};
}

// x / y rounded to double (x, y double-double, y.h != 0)
__device__ __forceinline__ double dd_quot(dd x, dd y) {
    const double q = x.h / y.h;
    const dd qy = dd_prod(q, y.h);
    // x - q y, leading parts cancel
    const double r = ((x.h - qy.h) - qy.l) + x.l - q * y.l;
    return q + r / y.h;
}

// a / b
__device__ __forceinline__ double2 cquot(double2 a, double2 b) {
    const dd den = dd_sum(dd_prod(b.x, b.x), dd_prod(b.y, b.y));
    return make_double2(dd_quot(dd_sum(dd_prod(a.x, b.x), dd_prod(a.y, b.y)), den),
                        dd_quot(dd_sum(dd_prod(a.y, b.x), dd_prod(-a.x, b.y)), den));
}

// The product of n <= 64 complex numbers, on every lane of a wave.
__device__ __forceinline__ ddc wave_product(const double2* v, int n, int lane) {
    ddc f = {1.0, 0.0, 0.0, 0.0};
    if (lane < n) f = ddc_from(v[lane].x, v[lane].y);
    for (int s = 1; s < kWave; s <<= 1) f = ddc_times(f, ddc_shfl_xor(f, s));
    return f;
}

}  // namespace

__global__ __launch_bounds__(256) void plain_expand_kernel(const double2* __restrict__ A, double2* __restrict__ M2,
                                                           int n, int64_t m2_stride, unsigned* counters) {
    __shared__ double row_min[kMaxCols];
    __shared__ double row_max[kMaxCols];
    __shared__ int row_low[kMaxCols];   // lowest bit of the row's entries
    __shared__ bool row_bad[kMaxCols];  // an entry not finite or too large
    __shared__ int pivot;
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    const int64_t task = blockIdx.x;
    A += task * n * n;
    M2 += task * m2_stride;

    for (int i = wid; i < n; i += 4) {  // a wave per row (n <= 40 <= 64 lanes)
        double lo = __builtin_inf(), hi = 0.0;
        int low = lowest_bit(0.0);
        bool bad = false;
        if (lane < n) {
            const double2 v = A[i * n + lane];
            const double x = fabs(v.x), y = fabs(v.y);
            bad = !pivot_admits(v.x, v.y);
            low = lowest_bit(v.x, v.y);
            lo = hi = x > y ? x : y;
        }
        for (int m = kWave / 2; m >= 1; m >>= 1) {
            lo = fmin(lo, __shfl_xor(lo, m, kWave));
            hi = fmax(hi, __shfl_xor(hi, m, kWave));
            low = min(low, __shfl_xor(low, m, kWave));
        }
        const bool any_bad = __any(bad);
        if (lane == 0) {
            row_min[i] = lo;
            row_max[i] = hi;
            row_low[i] = low;
            row_bad[i] = any_bad;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int best = 0, low = lowest_bit(0.0);
        bool bad = false;
        double hi = 0.0;
        for (int i = 0; i < n; ++i) {
            if (row_min[i] > row_min[best]) best = i;
            hi = fmax(hi, row_max[i]);
            low = min(low, row_low[i]);
            bad = bad || row_bad[i];
        }
        const bool fits = !bad && off_grid(low, hi) && row_min[best] >= pivot_least(hi);
        pivot = fits ? best : -1;
        counters[task] = fits ? kExpandedFlag : 0u;
    }
    __syncthreads();
    const int r = pivot;
    if (r < 0) {
        for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
            const double2 v = A[e];
            M2[e] = make_double2(2.0 * v.x, 2.0 * v.y);
            M2[n * n + e] = make_double2(-2.0 * v.x, -2.0 * v.y);
        }
        return;
    }
    const int m = (n - 1) * n;
    for (int e = threadIdx.x; e < m; e += blockDim.x) {
        const int k = e / n, j = e - k * n;
        double2 q = cquot(A[(k < r ? k : k + 1) * n + j], A[r * n + j]);
        q = make_double2(2.0 * q.x, 2.0 * q.y);
        M2[e] = q;
        M2[m + e] = make_double2(-q.x, -q.y);
    }
    if (wid == 0) {  // the product of the scales, after the table
        const ddc f = wave_product(A + r * n, n, lane);
        if (lane == 0) *reinterpret_cast<ddc*>(M2 + 2 * m) = f;
    }
}

// Repeated-row tasks.  Of a large batch on one matrix (thousands of transitions of one
// interferometer) only the tasks' row and slot numbers are uploaded: each task's rows, with
// a column per slot, and its base (anchor + sum of the walked rows' multiples, the seed of
// every chunk) are formed here.  4096 transitions of 8..26 photons are 18 MB of them, which
// cost the host 2.9 ms of a call to lay out, copy, upload and free.  Expanded tasks: the
// rows are divided by the expanded one, and the product of the scales, each slot's entry of
// that row, taken into the task's scale.  A block per task; bound by the host's planning,
// which it follows.
__global__ __launch_bounds__(256) void rep_layout_kernel(RepTask* tasks) {
    __shared__ double2 x[kMaxSlots];
    RepTask& T = tasks[blockIdx.x];
    const bool gather = T.src != nullptr, expand = T.degree > 0;
    if (!gather && !expand) return;
    const int NS = T.NS, lane = threadIdx.x & (kWave - 1);
    double2* const A = const_cast<double2*>(T.A);
    auto entry = [&](uint32_t row, int s) {
        return T.src[T.transpose ? (int64_t)T.src_slot[s] * T.src_ld + row : (int64_t)row * T.src_ld + T.src_slot[s]];
    };
    if (expand && threadIdx.x < NS) x[lane] = gather ? entry(T.src_xrow, lane) : T.xrow[lane];
    __syncthreads();
    if (threadIdx.x >= 3 * kWave) {  // one wave forms the scale beside the others' quotients
        if (expand) {
            const ddc f = ddc_times(wave_product(x, NS, lane), ddc_from(T.scale[0], 0.0));
            if (lane == 0) {
                T.scale[0] = f.hr;
                T.scale[1] = f.lr;
                T.scale[2] = f.hi;
                T.scale[3] = f.li;
            }
        }
    } else {
        for (int e = threadIdx.x; e < T.rows * NS; e += 3 * kWave) {
            const int r = e / NS, s = e - r * NS;
            const double2 a = gather ? entry(T.src_row[r], s) : A[e];
            A[e] = expand ? cquot(a, x[s]) : a;
        }
    }
    __syncthreads();
    if (threadIdx.x < NS) {
        double2 b = A[lane];
        for (int d = 0; d < T.nlow; ++d) {
            const double m = (double)(T.lrad[d] - 1);
            const double2 a = A[(1 + d) * NS + lane];
            b.x += m * a.x;  // two roundings, as on the host (fill_base in batch.hip)
            b.y += m * a.y;
        }
        const_cast<double2*>(T.base)[lane] = b;
    }
}

hipError_t launch_rep_layout(RepTask* tasks, int64_t ntasks, hipStream_t st) {
    hipLaunchKernelGGL(rep_layout_kernel, dim3((unsigned)ntasks), dim3(256), 0, st, tasks);
    return hipGetLastError();
}

int plain_expand_row(const double* A, int n, int64_t ld) {
    int best = -1, low = lowest_bit(0.0);
    double best_min = -1.0, hi = 0.0;
    for (int i = 0; i < n; ++i) {
        double lo = __builtin_inf();
        for (int j = 0; j < n; ++j) {
            const double re = A[2 * (i * ld + j)], im = A[2 * (i * ld + j) + 1];
            if (!pivot_admits(re, im)) return -1;
            const double x = std::fabs(re), y = std::fabs(im), v = x > y ? x : y;
            lo = v < lo ? v : lo;
            hi = v > hi ? v : hi;
            if (!off_grid(low, hi)) low = std::min(low, lowest_bit(re, im));  // off it, it stays off
        }
        if (lo > best_min) {
            best_min = lo;
            best = i;
        }
    }
    return off_grid(low, hi) && best_min >= pivot_least(hi) ? best : -1;
}

hipError_t launch_plain_expand(const double2* A, double2* M2, int n, int64_t count, unsigned* counters,
                               hipStream_t st) {
    hipLaunchKernelGGL(plain_expand_kernel, dim3((unsigned)count), dim3(256), 0, st, A, M2, n, (int64_t)2 * n * n,
                       counters);
    return hipGetLastError();
}

}  // namespace pqb
