// Device-side helpers shared by the permanent kernels (gfx950, wave64).
//
// * complex arithmetic on split (re, im) doubles, written so that hipcc
//   contracts each component into one mul + one fma;
// * double-double ("dd") error-free sums used for every reduction of
//   partial sums across lanes, waves and blocks (the reference accumulates
//   with plain per-thread scalars, BBFGPermanentCalculator.hpp:113,169-176,
//   or with the order-bucketed ComplexM, PicComplexM.hpp:125-201);
// * wave / block reductions of dd complex values.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pqb {

constexpr int kWave = 64;

// Read-only data reached through pointers loaded from memory (task tables,
// step tables, matrices of a batch) is accessed through the constant address
// space, so wave-uniform accesses become scalar loads with SGPR results.
// (The host pass of hipcc parses device templates too; it sees plain pointers.)
#if defined(__HIP_DEVICE_COMPILE__)
template <class T>
using cptr = const __attribute__((address_space(4))) T*;
#else
template <class T>
using cptr = const T*;
#endif

template <class T>
__device__ __forceinline__ cptr<T> to_const(const T* q) {
    return (cptr<T>)q;
}

// ---------------------------------------------------------------- complex --

// (ar + i ai) *= (br + i bi); four FP64 VALU instructions after contraction.
__device__ __forceinline__ void cmul(double& ar, double& ai, double br, double bi) {
    const double t = ar * br - ai * bi;
    ai = ar * bi + ai * br;
    ar = t;
}

// ------------------------------------------------------------ double-double --

struct ddc {  // dd complex: value = (hr + lr) + i (hi + li)
    double hr, lr, hi, li;
};

// Knuth TwoSum: s + e == a + b exactly.
__device__ __forceinline__ void two_sum(double a, double b, double& s, double& e) {
    s = a + b;
    const double bb = s - a;
    e = (a - (s - bb)) + (b - bb);
}

__device__ __forceinline__ void fast_two_sum(double a, double b, double& s, double& e) {
    s = a + b;
    e = b - (s - a);
}

// dd + dd (Bailey's sloppy add with renormalisation; relative error ~2^-104
// unless the operands cancel, in which case the absolute error stays at
// 2^-104 of the larger operand, which is what a sum of partials needs).
__device__ __forceinline__ void dd_add(double& h, double& l, double h2, double l2) {
    double s, e;
    two_sum(h, h2, s, e);
    e += l + l2;
    fast_two_sum(s, e, h, l);
}

__device__ __forceinline__ void ddc_add(ddc& a, const ddc& b) {
    dd_add(a.hr, a.lr, b.hr, b.lr);
    dd_add(a.hi, a.li, b.hi, b.li);
}

__device__ __forceinline__ ddc ddc_shfl_xor(const ddc& v, int mask) {
    ddc r;
    r.hr = __shfl_xor(v.hr, mask, kWave);
    r.lr = __shfl_xor(v.lr, mask, kWave);
    r.hi = __shfl_xor(v.hi, mask, kWave);
    r.li = __shfl_xor(v.li, mask, kWave);
    return r;
}

// Butterfly reduction over the 64 lanes of a wave; every lane ends with the sum.
__device__ __forceinline__ ddc wave_reduce(ddc v) {
#pragma unroll
    for (int m = kWave / 2; m >= 1; m >>= 1) {
        ddc o = ddc_shfl_xor(v, m);
        ddc_add(v, o);
    }
    return v;
}

// Sum over the block; the result is valid in thread 0.  `sh` needs one ddc
// per wave of the block.  Summation order is fixed (deterministic).
__device__ __forceinline__ ddc block_reduce(ddc v, ddc* sh) {
    v = wave_reduce(v);
    const int lane = threadIdx.x & (kWave - 1);
    const int wid = threadIdx.x / kWave;
    const int nw = (blockDim.x + kWave - 1) / kWave;
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    ddc r = {0.0, 0.0, 0.0, 0.0};
    if (threadIdx.x == 0) {
        r = sh[0];
        for (int w = 1; w < nw; ++w) ddc_add(r, sh[w]);
    }
    return r;
}

__device__ __forceinline__ ddc ddc_from(double re, double im) {
    ddc r = {re, 0.0, im, 0.0};
    return r;
}

// A block's partial result handed to the last block of the grid to finish: written
// through to where every XCD's L2 sees it, read the same way.  With these, a wait for
// the stores is all the order the handover's counter needs; a __threadfence() on both
// sides writes back and invalidates the XCD's L2 once per block (4096 permanents of
// n = 10 in one launch: 147 us with the fences, 19.6 us with these; one of n = 20:
// 31.0 and 22.8 us).
template <class T>
__device__ __forceinline__ void store_through(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <class T>
__device__ __forceinline__ T load_through(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A synchronous host call's result is in host memory: says so there, where the host polls
// (wait_result in engine.hip), without waiting for the kernel's end to be noticed.
__device__ __forceinline__ void announce(unsigned* done) {
    if (done) __hip_atomic_store(done, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ void ddc_store_through(ddc* p, const ddc& v) {
    store_through(&p->hr, v.hr);
    store_through(&p->lr, v.lr);
    store_through(&p->hi, v.hi);
    store_through(&p->li, v.li);
}

__device__ __forceinline__ ddc ddc_load_through(const ddc* p) {
    return {load_through(&p->hr), load_through(&p->lr), load_through(&p->hi), load_through(&p->li)};
}

// (hr + lr) + i (hi + li) times the double-double complex f, the scale of an
// expanded sweep: products split exactly, the cross terms in FP64.  The empty asm
// keeps each rounded product out of contraction, so that its FMA is its error.
__device__ __forceinline__ void two_prod(double a, double b, double& p, double& e) {
    p = a * b;
    asm volatile("" : "+v"(p));
    e = fma(a, b, -p);
}

__device__ __forceinline__ void dd_mul(double ah, double al, double bh, double bl, double& h, double& l) {
    double p, e;
    two_prod(ah, bh, p, e);
    e = fma(ah, bl, fma(al, bh, e));
    fast_two_sum(p, e, h, l);
}

__device__ __forceinline__ ddc ddc_mul(const ddc& a, const ddc& f) {
    ddc r;
    double h, l;
    dd_mul(a.hr, a.lr, f.hr, f.lr, r.hr, r.lr);
    dd_mul(a.hi, a.li, f.hi, f.li, h, l);
    dd_add(r.hr, r.lr, -h, -l);
    dd_mul(a.hr, a.lr, f.hi, f.li, r.hi, r.li);
    dd_mul(a.hi, a.li, f.hr, f.lr, h, l);
    dd_add(r.hi, r.li, h, l);
    return r;
}

// Exact scaling by a power of two.
__device__ __forceinline__ ddc ddc_scale(ddc v, double s) {
    v.hr *= s; v.lr *= s; v.hi *= s; v.li *= s;
    return v;
}

}  // namespace pqb
