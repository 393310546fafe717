// Exact integer permanents on the FP64 pipe.
//
// The sum of plain_exact_kernel (perm_plain.hip) -- sum_delta (prod_i delta_i)
// prod_j sum_i delta_i a_ij modulo 2^128, BBFGPermanentCalculator.hpp:87-235 in whole
// numbers -- with every product formed in doubles without rounding.  64-bit integer
// multiplies run at a quarter of the rate of FP64 ones and take several instructions
// each; this kernel needs about 24 FP64 instructions per step beside the NC column
// updates and NC - 3 products.
//
// * Column sums are doubles holding integers.  The columns are split into three groups
//   of at most g = ceil(NC / 3); the host admits matrices with cmax^g <= 2^46 (cmax: the
//   largest column abs sum, which bounds every column sum), so each group's product q is
//   an exact integer of at most 46 bits.
// * q0 q1 q2 is cut into digits X2 + X1 + X0, multiples of 2^88, 2^44 and 1, by exact
//   product splits (FMA) and by adding and subtracting 1.5 2^96 and 1.5 2^140, which
//   rounds to multiples of 2^44 and 2^88:
//       q0 q1 = H + L,  H a multiple of 2^44 (48 bits), |L| < 2^44;
//       H q2  = X2 + a, a a multiple of 2^44 below 2^88;
//       L q2  = b + X0, b a multiple of 2^44 (46 bits), |X0| < 2^44;  X1 = a + b.
// * The digits of `flush` steps are added up in doubles -- exact: with q <= 2^e the host
//   takes flush = 2^(140 - 3 e), at most 256, so that every sum stays below 2^53 units --
//   and then go into a 128-bit accumulator.
//
// Waves, lanes and seeds as in the plain sweep (perm_plain.hip): a lane per column sums
// the wave-uniform rows from LDS, the 64 lanes' own rows come from two tables of eight.
//
// A block is a whole CU's four waves per SIMD: the fewer blocks, the fewer atomics on the
// counter the grid finishes by (n = 26: 87 us in blocks of 256 threads, 84.6 us of 1024).
//
// Bound by FP64 issue.  0/1 matrices of n = 26: 264 us with 64-bit integer products
// (kernel, clock not warm), 85 us now; 283 -> 106 us a call.
//
// This unit is compiled without contraction (the digits' sums must not absorb a product).

#include "pqb_device.h"
#include "pqb_kernels.h"

namespace pqb {

namespace {

typedef unsigned __int128 u128;
typedef __int128 i128;

template <int LO, int HI, int NC>
__device__ __forceinline__ double group_product(const double (&c)[NC]) {
    if constexpr (LO >= NC) {
        return 1.0;
    } else {
        constexpr int E = HI < NC ? HI : NC;
        double q = c[LO];
#pragma unroll
        for (int j = LO + 1; j < E; ++j) q *= c[j];
        return q;
    }
}

// (s2, s1, s0) +- the digits of the product of c[0..NC)
template <int NC, bool MINUS>
__device__ __forceinline__ void add_digits(const double (&c)[NC], double& s2, double& s1, double& s0) {
    constexpr int g = (NC + 2) / 3;
    constexpr double M1 = 0x1.8p96, M2 = 0x1.8p140;
    const double q0 = group_product<0, g>(c), q1 = group_product<g, 2 * g>(c), q2 = group_product<2 * g, NC>(c);
    const double h = q0 * q1;
    const double l = __builtin_fma(q0, q1, -h);
    const double H = (h + M1) - M1;
    const double L = (h - H) + l;
    const double ah = H * q2;
    const double al = __builtin_fma(H, q2, -ah);
    const double bh = L * q2;
    const double bl = __builtin_fma(L, q2, -bh);
    const double X2 = (ah + M2) - M2;
    const double b = (bh + M1) - M1;
    const double X1 = ((ah - X2) + al) + b;
    const double X0 = (bh - b) + bl;
    if constexpr (MINUS) {
        s2 -= X2;
        s1 -= X1;
        s0 -= X0;
    } else {
        s2 += X2;
        s1 += X1;
        s0 += X0;
    }
}

}  // namespace

template <int NC>
__global__ __launch_bounds__(kExactBlock) void plain_exact_fp64_kernel(ExactF64Params p) {
    constexpr int P = NC | 1;
    __shared__ double rows[(NC + 1) * P];
    __shared__ double lanes[16 * P];
    __shared__ double bases[(kExactBlock / kWave) * P];
    __shared__ u128 red[kExactBlock / kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int R = p.R, K = p.K, B = p.B, H = p.H;
    const int64_t g = (int64_t)blockIdx.x * (blockDim.x / kWave) + wid;  // wave = group of sign vectors
    const bool wave_on = g < ((int64_t)1 << H);

    for (int e = threadIdx.x; e < R * NC; e += blockDim.x) rows[(e / NC) * P + e % NC] = 0.5 * p.A2[e];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * NC; e += blockDim.x) {
        const int k = e / NC, j = e - k * NC;
        double v = 0.0;
        for (int b = 0; b < 3; ++b) {
            const int bit = (k >= 8 ? 3 : 0) + b;
            if (bit < B) {
                const double a = rows[(R - 1 - K - bit) * P + j];
                v += ((k >> b) & 1) ? -a : a;
            }
        }
        lanes[k * P + j] = v;
    }
    double* const base = bases + wid * P;
    if (lane < NC) {
        double v = rows[lane];
        for (int b = 0; b < K; ++b) v += rows[(R - 1 - b) * P + lane];
        for (int h = 0; h < H; ++h) {
            const double a = rows[(R - 1 - K - B - h) * P + lane];
            v += ((g >> h) & 1) ? -a : a;
        }
        base[lane] = v;
    }
    __syncthreads();

    u128 acc = 0;
    if (wave_on) {
        double c[NC];
#pragma unroll
        for (int j = 0; j < NC; ++j) c[j] = base[j] + (lanes[(lane & 7) * P + j] + lanes[(8 + (lane >> 3)) * P + j]);
        const cptr<double> A2 = to_const(p.A2);
        auto flip = [&](int row, double s) __attribute__((always_inline)) {
            asm volatile("" : "+v"(s));  // in a VGPR: an instruction reads one scalar operand, the row
            const cptr<double> a = A2 + row * NC;
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                c[j] = __builtin_fma(s, a[j], c[j]);
                if ((j & 31) == 31) __builtin_amdgcn_sched_barrier(0);  // 32 columns (64 SGPRs) in flight
            }
        };
        const unsigned W = 1u << K;
        const unsigned F = (unsigned)p.flush;
        for (unsigned t0 = 0; t0 < W; t0 += F) {
            const unsigned t1 = W - t0 < F ? W : t0 + F;
            double s2 = 0.0, s1 = 0.0, s0 = 0.0;
            for (unsigned t = t0; t < t1; t += 2) {  // F is even
                if (t > 0) {
                    const unsigned b = __builtin_ctz(t);
                    const unsigned nb = ((t >> b) ^ (t >> (b + 1))) & 1u;
                    flip(R - 1 - (int)b, nb ? -1.0 : 1.0);
                }
                add_digits<NC, false>(c, s2, s1, s0);
                if (t + 1 < t1) {
                    flip(R - 1, ((t >> 1) & 1u) ? 1.0 : -1.0);
                    add_digits<NC, true>(c, s2, s1, s0);
                }
            }
            const i128 d2 = (i128)(int64_t)(s2 * 0x1p-88), d1 = (i128)(int64_t)(s1 * 0x1p-44), d0 = (int64_t)s0;
            acc += ((u128)d2 << 88) + ((u128)d1 << 44) + (u128)d0;
        }
        // sign of the lane's first term: parity of the lane's and the group's bits
        if ((__popc((unsigned)lane) + __popcll((unsigned long long)g)) & 1) acc = (u128)0 - acc;
        if (lane >= (1 << B)) acc = 0;
    }

    // block sum (wrap-around arithmetic is associative: order does not matter)
    unsigned long long lo = (unsigned long long)acc, hi = (unsigned long long)(acc >> 64);
#pragma unroll
    for (int m = kWave / 2; m >= 1; m >>= 1) {
        const unsigned long long olo = __shfl_xor(lo, m, kWave);
        const unsigned long long ohi = __shfl_xor(hi, m, kWave);
        const u128 s = (((u128)hi << 64) | lo) + (((u128)ohi << 64) | olo);
        lo = (unsigned long long)s;
        hi = (unsigned long long)(s >> 64);
    }
    if (lane == 0) red[wid] = ((u128)hi << 64) | lo;
    __syncthreads();
    __shared__ bool is_last;
    if (threadIdx.x == 0) {
        u128 s = 0;
        for (unsigned w = 0; w < blockDim.x / kWave; ++w) s += red[w];
        store_through(&p.partials[2 * blockIdx.x], (unsigned long long)s);
        store_through(&p.partials[2 * blockIdx.x + 1], (unsigned long long)(s >> 64));
        wait_stores();
        is_last = atomicAdd(p.counter, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (is_last) {  // a lane per partial, then the first wave's lanes
        if (threadIdx.x < kWave) {
            u128 s = 0;
            for (unsigned b = threadIdx.x; b < gridDim.x; b += kWave)
                s += ((u128)load_through(&p.partials[2 * b + 1]) << 64) | load_through(&p.partials[2 * b]);
            lo = (unsigned long long)s;
            hi = (unsigned long long)(s >> 64);
#pragma unroll
            for (int m = kWave / 2; m >= 1; m >>= 1) {
                const unsigned long long olo = __shfl_xor(lo, m, kWave);
                const unsigned long long ohi = __shfl_xor(hi, m, kWave);
                const u128 v = (((u128)hi << 64) | lo) + (((u128)ohi << 64) | olo);
                lo = (unsigned long long)v;
                hi = (unsigned long long)(v >> 64);
            }
            if (threadIdx.x == 0) {
                p.out[0] = lo;
                p.out[1] = hi;
                *p.counter = 0u;
                announce(p.done);
            }
        }
    }
}

#define PQB_NC_CASES(X) \
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) \
    X(17) X(18) X(19) X(20) X(21) X(22) X(23) X(24) X(25) X(26) X(27) X(28) X(29) X(30)    \
    X(31) X(32) X(33) X(34) X(35) X(36) X(37) X(38) X(39) X(40)

hipError_t launch_plain_exact_fp64(int nc, const ExactF64Params& p, int nblocks, int bdim, hipStream_t st) {
    switch (nc) {
#define PQB_CASE(N)                                                                                         \
    case N: hipLaunchKernelGGL((plain_exact_fp64_kernel<N>), dim3(nblocks), dim3(bdim), 0, st, p); break;
        PQB_NC_CASES(PQB_CASE)
#undef PQB_CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace pqb
