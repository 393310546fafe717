// Permanents of at most kTinySteps signed terms, one block per matrix: plain ones of up
// to 11 rows and repeated-row ones of few steps (the sums of BBFGPermanentCalculator.hpp:
// 87-235 and BBFGPermanentCalculatorRepeated.hpp:116-307).
//
// Such a call is latency: copies, launches and their gaps, not arithmetic.  Everything is
// in one launch that reads the matrix where it is -- for host calls the pinned staging
// buffer, over the bus -- and writes the result where it is read, so there is no copy in
// either direction, no table kernel, no second reduction kernel.
//
// The terms' index e = hi * P + lo is a mixed-radix number, digit d counting the negative
// copies of row 1 + d.  The column sums of the low and of the high digits (with the anchor)
// are formed once each in LDS, P + S / P rows beside the S terms, and a thread's column sum
// is the sum of two reads; the weights prod (-1)^k C(m, k) likewise.  Rows are an odd number
// of 16-byte elements apart, so that lanes reading consecutive rows hit different banks.
//
// Bound by the launch and the host's notice of the result (a call of n = 8: 14.5 us, 23.0 us
// with the copies, the general sweep and a stream synchronisation; a transition of 10
// photons to 7 modes, 192 steps: 20.1 us against 71.6 us through the batched launch).

#include <algorithm>

#include "pqb_device.h"
#include "pqb_kernels.h"
#include "pqb_terms.h"

namespace pqb {

// Matrix `index` of p, by the whole block.
template <int NS>
__device__ __forceinline__ void tiny_matrix(const TinyParams& p, int64_t index, double2* lds, ddc* red) {
    constexpr int pitch = NS | 1;
    const int R = p.R, P = p.P, T = P + p.S / P;  // T: rows of the two tables
    double2* const rows = lds;
    double2* const tab = rows + R * pitch;
    double* const wt = reinterpret_cast<double*>(tab + T * pitch);
    const double2* const A = p.A + index * p.stride;
    for (int e = threadIdx.x; e < R * NS; e += blockDim.x) rows[(e / NS) * pitch + e % NS] = A[e];
    __syncthreads();
    for (int e = threadIdx.x; e < T * NS; e += blockDim.x) {
        const int t = e / NS, j = e - t * NS;
        const bool high = t >= P;
        double2 v = high ? rows[j] : make_double2(0.0, 0.0);
        double w = 1.0;
        int c = high ? t - P : t;
        for (int d = high ? p.nlow : 0; d < (high ? R - 1 : p.nlow); ++d) {
            const int r = p.radix[d], q = c / r, k = c - q * r, m = r - 1;
            c = q;
            const double f = (double)(m - 2 * k);
            const double2 a = rows[(1 + d) * pitch + j];
            v.x = fma(f, a.x, v.x);
            v.y = fma(f, a.y, v.y);
            if (j == 0) {
                double b = 1.0;  // C(m, k), every step an integer
                for (int i = 1; i <= k; ++i) b = b * (double)(m - k + i) / (double)i;
                w *= (k & 1) ? -b : b;
            }
        }
        tab[t * pitch + j] = v;
        if (j == 0) wt[t] = w;
    }
    __syncthreads();
    double ar = 0.0, ai = 0.0;
    for (int e = threadIdx.x; e < p.S; e += blockDim.x) {
        const int hi = e / P, lo = e - hi * P;
        const double2* const x = tab + lo * pitch;
        const double2* const y = tab + (P + hi) * pitch;
        double cr[NS], ci[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const double2 u = x[j], v = y[j];
            cr[j] = u.x + v.x;
            ci[j] = u.y + v.y;
        }
        add_wterm<NS>(cr, ci, wt[lo] * wt[P + hi], ar, ai);
    }
    const ddc s = ddc_scale(block_reduce(ddc_from(ar, ai), red), p.scale);
    if (threadIdx.x == 0) {
        double* const o = p.out + 6 * index;
        o[0] = s.hr + s.lr;
        o[1] = s.hi + s.li;
        o[2] = s.hr;
        o[3] = s.lr;
        o[4] = s.hi;
        o[5] = s.li;
        announce(p.done);
    }
}

template <int NS>
__global__ __launch_bounds__(1024) void tiny_kernel(TinyParams p) {
    extern __shared__ double2 lds[];
    __shared__ ddc red[1024 / kWave];
    tiny_matrix<NS>(p, blockIdx.x, lds, red);
}

template <int NS>
__device__ __forceinline__ void tiny_dispatch(int ns, const TinyParams& p, int64_t index, double2* lds, ddc* red) {
    if constexpr (NS >= 1) {
        if (ns == NS) tiny_matrix<NS>(p, index, lds, red);
        else tiny_dispatch<NS - 1>(ns, p, index, lds, red);
    }
}

// The shapes of a list beside each other: seven launches of n = 5..11, each 5 to 10 us of
// latency, took 60 us of a list's time.  Waves without terms add zeros, so a shape's sums do
// not depend on the block's size.
__global__ __launch_bounds__(1024) void tiny_mixed_kernel(TinyMixed m) {
    extern __shared__ double2 lds[];
    __shared__ ddc red[1024 / kWave];
    int at = 0;
    while (at + 1 < m.shapes && blockIdx.x >= m.first[at + 1]) ++at;
    tiny_dispatch<kTinySlots>(m.ns[at], m.p[at], blockIdx.x - m.first[at], lds, red);
}

bool tiny_split(TinyParams& p, int NS, int R) {
    if (NS < 1 || NS > kTinySlots || R < 1 || R - 1 > kTinyDigits) return false;
    int64_t S = 1;
    for (int d = 0; d < R - 1; ++d) {
        S *= p.radix[d];
        if (S > kTinySteps) return false;
    }
    // the split of the digits with the smallest tables
    int64_t best = 0, P = 1;
    for (int d = 0; d <= R - 1; ++d) {
        const int64_t rows = P + S / P;
        if (best == 0 || rows < best) {
            best = rows;
            p.P = (int)P;
            p.nlow = d;
        }
        if (d < R - 1) P *= p.radix[d];
    }
    p.R = R;
    p.S = (int)S;
    p.lds_bytes = (unsigned)((size_t)(R + best) * (NS | 1) * sizeof(double2) + (size_t)best * sizeof(double));
    return p.lds_bytes <= 60 * 1024;
}

static int tiny_threads(const TinyParams& p) { return p.S >= 1024 ? 1024 : (p.S + kWave - 1) / kWave * kWave; }

template <int NS>
static hipError_t launch_tiny_ns(const TinyParams& p, unsigned count, hipStream_t st) {
    hipLaunchKernelGGL(tiny_kernel<NS>, dim3(count), dim3(tiny_threads(p)), p.lds_bytes, st, p);
    return hipGetLastError();
}

hipError_t launch_tiny_mixed(const TinyMixed& m, hipStream_t st) {
    if (m.shapes < 1 || m.shapes > kTinyShapes) return hipErrorInvalidValue;
    int threads = 0;
    unsigned lds = 0;
    for (int k = 0; k < m.shapes; ++k) {
        threads = std::max(threads, tiny_threads(m.p[k]));
        lds = std::max(lds, m.p[k].lds_bytes);
    }
    hipLaunchKernelGGL(tiny_mixed_kernel, dim3(m.first[m.shapes]), dim3(threads), lds, st, m);
    return hipGetLastError();
}

hipError_t launch_tiny(int ns, const TinyParams& p, int64_t count, hipStream_t st) {
    if (count < 1 || count > 0x7fffffff) return hipErrorInvalidValue;
    switch (ns) {
#define PQB_CASE(N) \
    case N: return launch_tiny_ns<N>(p, (unsigned)count, st);
        PQB_CASE(1) PQB_CASE(2) PQB_CASE(3) PQB_CASE(4) PQB_CASE(5) PQB_CASE(6) PQB_CASE(7) PQB_CASE(8)
        PQB_CASE(9) PQB_CASE(10) PQB_CASE(11) PQB_CASE(12) PQB_CASE(13) PQB_CASE(14) PQB_CASE(15) PQB_CASE(16)
        PQB_CASE(17) PQB_CASE(18) PQB_CASE(19) PQB_CASE(20) PQB_CASE(21) PQB_CASE(22) PQB_CASE(23) PQB_CASE(24)
#undef PQB_CASE
        default: return hipErrorInvalidValue;
    }
}

}  // namespace pqb
