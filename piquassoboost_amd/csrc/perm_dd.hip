// Double-double sweep of the repeated-row sum
//
//   perm = 2^-(N-1) sum_{k_i = 0..m_i} prod_i (-1)^{k_i} C(m_i, k_i)
//                    prod_s ( a_anchor,s + sum_i (m_i - 2 k_i) a_i,s )
//
// (BBFGPermanentCalculatorRepeated.hpp:116-307; the plain sum of
// BBFGPermanentCalculator.hpp:87-235 is the case where every multiplicity is
// 1) with 106-bit significands in every column sum, product and partial sum.
// It serves the reference's infinite-precision calculators
// (BBFGPermanentCalculator.cpp:100-107 and BBFGPermanentCalculatorRepeated.cpp:
// 115-122, ComplexInf / FloatInf of InfinitePrecisionComplex.h), which
// evaluate the same sum in exact MPFR arithmetic and round the result once to
// double (mpfr_get_d, round to nearest).  Here:
//
// * chunk seeds are built from the matrix rows with error-free products
//   (integer coefficient x double) and double-double sums; a Gray step adds
//   +-2 a_row (an exact double) with an error-free sum;
// * each complex product and the weighted accumulation are double-double
//   operations with relative error ~2^-104 of the operands' magnitude;
// * partial sums are combined in double-double and rounded once.
// The result is the correctly rounded sum unless the accumulated error
// (~2^-100 of the sum of |terms|) reaches half an ulp of the result, i.e.
// unless the sum cancels by more than ~2^45.
//
// Layout: the tasks, step tables, work items and persistent grid of the FP64
// batched sweep (perm_repeated.hip).  A chunk is handled by a group of G = 1,
// 2 or 4 lanes: lane q of the group holds the column sums of slots
// q*M .. q*M+M-1 (M = ceil(NS/G), four doubles per slot), multiplies them in
// two independent chains, and the group combines its partial products with
// DPP quad permutations (one for a pair, two for a quad).  A wave works on
// 64/G chunks at a time.  Each exchange repeats a product on every lane of the
// group, so smaller groups do less work, as far as their registers go.
//
// Bound by its FP64 instructions: 38 for a product of two columns.  Two forms:
//
// * Rows split on a grid (RepTask::split) for matrices whose entries lie within
//   2^40 of each other: the column sums are exact, at 5 instructions instead of
//   11 per component, and short enough that up to 32 slots a pair of lanes holds
//   them at two waves per SIMD.  The next row is loaded during the product, a
//   chunk's lanes' parts side by side: lanes 256 bytes apart (32 slots in quads)
//   took twice the time.  Calls of n = 24 / 26 / 28 / 30: 547 / 2009 / 7740 /
//   34800 us before, 400 / 1530 / 6140 / 26800 us now (quads up to 32 slots, rows
//   split: 456 / 1702 / 6594 / 29273).
// * Any other: normalised double-double sums, at most 8 slots per lane (three
//   waves per SIMD), G = 1 up to 8 slots, 2 up to 16, 4 up to 32; 33..40 slots
//   take 10 per lane at two waves per SIMD.
//
// The file also holds grad_perm_kernel (the permanent from the finished
// gradient by a double-double Laplace sum).
//
// This translation unit is compiled with -ffp-contract=off (piquassoboost_amd/
// build.py): an error-free transformation is only error-free when every
// product and sum is rounded exactly as written, and a product fused into the
// following TwoSum silently drops the low half.

#include "pqb_device.h"
#include "pqb_kernels.h"

namespace pqb {
namespace {

// Move a double across the lanes of a quad (DPP quad_perm, bound_ctrl).
template <int CTRL>
__device__ __forceinline__ double quad_move(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
constexpr int kXor1 = 0xB1;  // quad_perm [1,0,3,2]
constexpr int kXor2 = 0x4E;  // quad_perm [2,3,0,1]

template <int CTRL>
__device__ __forceinline__ ddc quad_move(const ddc& v) {
    ddc r;
    r.hr = quad_move<CTRL>(v.hr);
    r.lr = quad_move<CTRL>(v.lr);
    r.hi = quad_move<CTRL>(v.hi);
    r.li = quad_move<CTRL>(v.li);
    return r;
}

// (h, l) += v for a double v (error-free sum, renormalised).
__device__ __forceinline__ void dd_add_d(double& h, double& l, double v) {
    double s, t;
    two_sum(h, v, s, t);
    t = t + l;
    fast_two_sum(s, t, h, l);
}

// (h, l) += f * a for an integer-valued f with |f| <= 2^11: f a = p + e exactly.
__device__ __forceinline__ void dd_addmul(double& h, double& l, double f, double a) {
    const double p = f * a;
    const double e = fma(f, a, -p);
    double s, t;
    two_sum(h, p, s, t);
    t = t + (l + e);
    fast_two_sum(s, t, h, l);
}

// a *= b in double-double complex arithmetic.  Each component is the sum of
// two exact products (error-free split with FMA), the four cross terms with
// the low parts, and one renormalisation; the lo x lo terms (2^-106 of the
// result's scale) are dropped.
__device__ __forceinline__ void ddc_mul(ddc& a, const ddc& b) {
    // real: ar br - ai bi
    const double p1 = a.hr * b.hr;
    const double e1 = fma(a.hr, b.hr, -p1);
    const double p2 = a.hi * b.hi;
    const double e2 = fma(a.hi, b.hi, -p2);
    double s, t;
    two_sum(p1, -p2, s, t);
    t = t + (e1 - e2);
    t = fma(a.hr, b.lr, t);
    t = fma(a.lr, b.hr, t);
    t = fma(-a.hi, b.li, t);
    t = fma(-a.li, b.hi, t);
    // imaginary: ar bi + ai br
    const double p3 = a.hr * b.hi;
    const double e3 = fma(a.hr, b.hi, -p3);
    const double p4 = a.hi * b.hr;
    const double e4 = fma(a.hi, b.hr, -p4);
    double u, v;
    two_sum(p3, p4, u, v);
    v = v + (e3 + e4);
    v = fma(a.hr, b.li, v);
    v = fma(a.lr, b.hi, v);
    v = fma(a.hi, b.lr, v);
    v = fma(a.li, b.hr, v);
    fast_two_sum(s, t, a.hr, a.lr);
    fast_two_sum(u, v, a.hi, a.li);
}

// acc += w * x for an integer-valued weight w (|w| < 2^53, exact in a double).
__device__ __forceinline__ void ddc_acc_w(ddc& acc, double w, const ddc& x) {
    {
        const double p = w * x.hr;
        double e = fma(w, x.hr, -p);
        e = fma(w, x.lr, e);
        double s, t;
        two_sum(acc.hr, p, s, t);
        t = t + (acc.lr + e);
        fast_two_sum(s, t, acc.hr, acc.lr);
    }
    {
        const double p = w * x.hi;
        double e = fma(w, x.hi, -p);
        e = fma(w, x.li, e);
        double s, t;
        two_sum(acc.hi, p, s, t);
        t = t + (acc.li + e);
        fast_two_sum(s, t, acc.hi, acc.li);
    }
}

// Product of all column sums of the chunk, column(k) being the lane's k-th: its M slots as
// two independent chains (same number of products, twice the ILP), then across the group
// of G lanes.
template <int G, int M, class Column>
__device__ __forceinline__ ddc group_product(Column&& column) {
    constexpr int H = M / 2;  // second chain starts at slot H (M >= 2)
    ddc p = column(0);
    if constexpr (M >= 2) {
        ddc u = column(H);
#pragma unroll
        for (int k = 1; k < M; ++k) {
            if (k == H) continue;
            if (k < H)
                ddc_mul(p, column(k));
            else
                ddc_mul(u, column(k));
        }
        ddc_mul(p, u);
    }
    if constexpr (G >= 2) {
        const ddc x = quad_move<kXor1>(p);
        ddc_mul(p, x);  // product of the lane pair
    }
    if constexpr (G == 4) {
        const ddc x = quad_move<kXor2>(p);
        ddc_mul(p, x);  // product of the quad
    }
    return p;
}

// Weighted double-double sum over one chunk, column sums from the split rows (RepTask::
// split): each is h + l with h a multiple of the task's grid and l the rest, and neither
// rounds, so a row's flip is one FMA for each and the pair is normalised when it is
// multiplied: 5 instructions per component and step against 11 for an error-free sum
// that keeps it normalised.
template <int G, int M>
__device__ __forceinline__ void dd_chunk_split(cptr<RepTask> T, const double* __restrict__ binom, uint32_t chunk,
                                               int q, ddc& acc) {
    constexpr int kPitch = 2 * G * M;  // double2 per row, padding slots included
    const double2* __restrict__ S = T->split + q;  // slot k's parts at 2 k G and (2 k + 1) G
    double hr[M], lr[M], hi[M], li[M];
    const double2* base = S + (size_t)T->rows * kPitch;  // anchor and low digits at k = 0
#pragma unroll
    for (int k = 0; k < M; ++k) {
        const double2 x = base[2 * k * G], y = base[(2 * k + 1) * G];
        hr[k] = x.x;
        lr[k] = x.y;
        hi[k] = y.x;
        li[k] = y.y;
    }
    auto add = [&](int k, double f, double2 x, double2 y) __attribute__((always_inline)) {
        hr[k] = fma(f, x.x, hr[k]);
        lr[k] = fma(f, x.y, lr[k]);
        hi[k] = fma(f, y.x, hi[k]);
        li[k] = fma(f, y.y, li[k]);
    };
    // slots [k0, M) of a row, at most four (32 VGPRs) in flight
    auto add_row = [&](uint32_t r, double f, int k0) __attribute__((always_inline)) {
        const double2* row = S + (size_t)r * kPitch;
#pragma unroll
        for (int k = 0; k < M; ++k) {
            if (k < k0) continue;
            add(k, f, row[2 * k * G], row[(2 * k + 1) * G]);
            if ((k & 3) == 3) __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto product = [&]() __attribute__((always_inline)) {
        return group_product<G, M>([&](int k) __attribute__((always_inline)) {
            ddc c;
            fast_two_sum(hr[k], lr[k], c.hr, c.lr);
            fast_two_sum(hi[k], li[k], c.hi, c.li);
            return c;
        });
    };
    // high digits from the chunk index: coefficient m - 2k, chunk weight (-1)^k C(m, k)
    double wc = 1.0;
    uint32_t c = chunk;
    const int nhigh = T->nhigh;
    for (int h = 0; h < nhigh; ++h) {
        const uint32_t r = T->hrad[h];
        const uint32_t qq = c / r;
        const uint32_t kd = c - qq * r;
        c = qq;
        const int m = (int)r - 1;
        add_row(T->hrow[h], (double)(m - 2 * (int)kd), 0);
        const double b = binom[m * kBinomStride + kd];
        wc *= (kd & 1u) ? -b : b;
    }
    const cptr<RepStep> tab = to_const(T->table);
    const int L = T->L;
    // the next step's row, or the slots of it that there are registers for, is loaded while
    // this one's product is formed
    constexpr int kAhead = M < 4 ? M : M > 12 ? 4 : M > 8 ? 8 : 2;
    double2 x[kAhead], y[kAhead];
    RepStep e = tab[0];
    auto load_ahead = [&](int t) __attribute__((always_inline)) {
        e = tab[t < L ? t : 0];
        const double2* row = S + (size_t)e.row * kPitch;
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            x[k] = row[2 * k * G];
            y[k] = row[(2 * k + 1) * G];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    load_ahead(1);
    ddc_acc_w(acc, wc, product());
    for (int t = 1; t < L; ++t) {
        const double f = e.dir ? -2.0 : 2.0, w = wc * e.w;
#pragma unroll
        for (int k = 0; k < kAhead; ++k) add(k, f, x[k], y[k]);
        add_row(e.row, f, kAhead);
        load_ahead(t + 1);
        ddc_acc_w(acc, w, product());
    }
}

// Weighted double-double sum over one chunk (every lane of the group ends
// with the same value; lane q = 0's copy is used).
template <int G, int M>
__device__ __forceinline__ void dd_chunk(cptr<RepTask> T, const double* __restrict__ binom, uint32_t chunk, int q,
                                         ddc& acc) {
    const int NS = T->NS;
    const double2* __restrict__ A = T->A;
    double hr[M], lr[M], hi[M], li[M];
    bool on[M];
    // anchor row (padding slots: factor 1, never updated)
#pragma unroll
    for (int k = 0; k < M; ++k) {
        const int s = q * M + k;
        on[k] = s < NS;
        const double2 a = on[k] ? A[s] : make_double2(0.0, 0.0);
        hr[k] = on[k] ? a.x : 1.0;
        lr[k] = 0.0;
        hi[k] = a.y;
        li[k] = 0.0;
    }
    auto column = [&](int k) __attribute__((always_inline)) { return ddc{hr[k], lr[k], hi[k], li[k]}; };
    // low digits at k = 0: coefficient m
    const int nlow = T->nlow;
    for (int dg = 0; dg < nlow; ++dg) {
        const double f = (double)((int)T->lrad[dg] - 1);
        const double2* row = A + (size_t)(1 + dg) * NS;
#pragma unroll
        for (int k = 0; k < M; ++k) {
            const double2 a = on[k] ? row[q * M + k] : make_double2(0.0, 0.0);
            dd_addmul(hr[k], lr[k], f, a.x);
            dd_addmul(hi[k], li[k], f, a.y);
        }
    }
    // high digits from the chunk index: coefficient m - 2k, chunk weight (-1)^k C(m, k)
    double wc = 1.0;
    uint32_t c = chunk;
    const int nhigh = T->nhigh;
    for (int h = 0; h < nhigh; ++h) {
        const uint32_t r = T->hrad[h];
        const uint32_t qq = c / r;
        const uint32_t kd = c - qq * r;
        c = qq;
        const int m = (int)r - 1;
        const double f = (double)(m - 2 * (int)kd);
        const double2* row = A + (size_t)T->hrow[h] * NS;
#pragma unroll
        for (int k = 0; k < M; ++k) {
            const double2 a = on[k] ? row[q * M + k] : make_double2(0.0, 0.0);
            dd_addmul(hr[k], lr[k], f, a.x);
            dd_addmul(hi[k], li[k], f, a.y);
        }
        const double b = binom[m * kBinomStride + kd];
        wc *= (kd & 1u) ? -b : b;
    }
    ddc_acc_w(acc, wc, group_product<G, M>(column));
    const cptr<RepStep> tab = to_const(T->table);
    const int L = T->L;
    for (int t = 1; t < L; ++t) {
        const RepStep e = tab[t];
        const double f = e.dir ? -2.0 : 2.0;
        const double2* row = A + (size_t)e.row * NS;
#pragma unroll
        for (int k = 0; k < M; ++k) {
            const double2 a = on[k] ? row[q * M + k] : make_double2(0.0, 0.0);
            dd_add_d(hr[k], lr[k], f * a.x);
            dd_add_d(hi[k], li[k], f * a.y);
        }
        ddc_acc_w(acc, wc * e.w, group_product<G, M>(column));
    }
}

template <int G, int MLO, int MHI, bool SPLIT>
__device__ __forceinline__ void dd_dispatch(int m, cptr<RepTask> T, const double* __restrict__ binom, uint32_t chunk0,
                                            uint32_t count, int q, int walker, ddc& acc) {
    if constexpr (MLO <= MHI) {
        if (m == MLO) {
            for (uint32_t j = (uint32_t)walker; j < count; j += kWave / G) {
                if constexpr (SPLIT) dd_chunk_split<G, MLO>(T, binom, chunk0 + j, q, acc);
                else dd_chunk<G, MLO>(T, binom, chunk0 + j, q, acc);
            }
        } else {
            dd_dispatch<G, MLO + 1, MHI, SPLIT>(m, T, binom, chunk0, count, q, walker, acc);
        }
    }
}

// Persistent grid over the work items (same item protocol as rep_batch_kernel);
// a chunk per group of G lanes, slot counts up to G * MHI.
template <int G, int MHI, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MHI <= 8 ? 3 : SPLIT ? 2 : 1))) void rep_dd_kernel(
    RepBatchParams p) {
    const int lane = threadIdx.x & (kWave - 1);
    const int q = lane & (G - 1);
    const int walker = lane / G;
    const cptr<RepItem> items = to_const(p.items);
    const cptr<unsigned> order = to_const(p.order);
    const cptr<RepTask> tasks = to_const(p.tasks);
    const unsigned nitems = to_const(p.counts)[0];
    // first item = wave index, then the counter offset by the wave count (see rep_batch_kernel)
    const unsigned nwaves = gridDim.x * (blockDim.x / kWave);
    unsigned idx0 = blockIdx.x * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    while (idx0 < nitems) {
        const unsigned idx = order[idx0];
        const RepItem it = items[idx];
        const cptr<RepTask> T = tasks + it.task;
        ddc acc = {0.0, 0.0, 0.0, 0.0};
        dd_dispatch<G, 1, MHI, SPLIT>((T->NS + G - 1) / G, T, p.binom, it.chunk0, it.count, q, walker, acc);
        if (q != 0) acc = ddc{0.0, 0.0, 0.0, 0.0};
        const ddc v = wave_reduce(acc);
        if (lane == 0) p.partials[idx] = v;
        // every lane executes the atomic, only lane 0 adds (see rep_batch_kernel)
        const unsigned got = atomicAdd(p.head, lane == 0 ? 1u : 0u);
        idx0 = nwaves + __builtin_amdgcn_readlane(got, 0);
    }
}

// perm(A) = sum_j a_0j G_0j (Laplace expansion along row 0 of the finished
// gradient), products split exactly (FMA) and summed in double-double.  One
// thread per matrix.
__global__ void grad_perm_kernel(const double2* __restrict__ A, const double2* __restrict__ G,
                                 double2* __restrict__ perm, int n, int count) {
    const int task = blockIdx.x * blockDim.x + threadIdx.x;
    if (task >= count) return;
    const double2* a = A + (size_t)task * n * n;  // row 0
    const double2* g = G + (size_t)task * n * n;  // row 0
    double hr = 0.0, lr = 0.0, hi = 0.0, li = 0.0;
    for (int j = 0; j < n; ++j) {
        const double2 x = a[j], y = g[j];
        // re = x.x y.x - x.y y.y, im = x.x y.y + x.y y.x, each product as p + e exactly
        const double p1 = x.x * y.x, e1 = fma(x.x, y.x, -p1);
        const double p2 = -x.y * y.y, e2 = fma(-x.y, y.y, -p2);
        const double p3 = x.x * y.y, e3 = fma(x.x, y.y, -p3);
        const double p4 = x.y * y.x, e4 = fma(x.y, y.x, -p4);
        dd_add(hr, lr, p1, e1);
        dd_add(hr, lr, p2, e2);
        dd_add(hi, li, p3, e3);
        dd_add(hi, li, p4, e4);
    }
    perm[task] = make_double2(hr + lr, hi + li);
}

}  // namespace

hipError_t launch_grad_perm(const double2* A, const double2* G, double2* perm, int n, int count, hipStream_t st) {
    const int bd = 64;
    hipLaunchKernelGGL(grad_perm_kernel, dim3((count + bd - 1) / bd), dim3(bd), 0, st, A, G, perm, n, count);
    return hipGetLastError();
}

// Ranges: rows as they are or split, lanes per chunk G and slots per lane, by the batch's
// largest slot count.
#define PQB_DD_RANGES(X) \
    X(0, 1, 8, false) X(1, 2, 8, false) X(2, 4, 8, false) X(3, 4, 10, false) \
    X(4, 1, 8, true) X(5, 2, 8, true) X(6, 2, 12, true) X(7, 2, 16, true) X(8, 4, 10, true)

int rep_dd_range_for(int max_ns, bool split) {
#define PQB_CASE(N, G, M, S) \
    if (S == split && max_ns <= G * M) return kDDRange0 + N;
    PQB_DD_RANGES(PQB_CASE)
#undef PQB_CASE
    return -1;
}

int rep_dd_walkers(int range) {
#define PQB_CASE(N, G, M, S) \
    if (range == kDDRange0 + N) return kWave / G;
    PQB_DD_RANGES(PQB_CASE)
#undef PQB_CASE
    return kWave;
}

const void* rep_dd_kernel_fn(int range) {
#define PQB_CASE(N, G, M, S) \
    if (range == kDDRange0 + N) return reinterpret_cast<const void*>(&rep_dd_kernel<G, M, S>);
    PQB_DD_RANGES(PQB_CASE)
#undef PQB_CASE
    return nullptr;
}

hipError_t launch_rep_dd(int range, const RepBatchParams& p, int grid_blocks, int reduce_blocks, hipStream_t st) {
    switch (range - kDDRange0) {
#define PQB_CASE(N, G, M, S) \
    case N: hipLaunchKernelGGL((rep_dd_kernel<G, M, S>), dim3(grid_blocks), dim3(256), 0, st, p); break;
        PQB_DD_RANGES(PQB_CASE)
#undef PQB_CASE
        default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_rep_reduce(p, reduce_blocks, st);
}

}  // namespace pqb
