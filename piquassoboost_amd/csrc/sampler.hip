// The photon loop of the generalized-Clifford sampler on the GPU (fill_r_sample,
// CGeneralizedCliffordsBSimulationStrategy.cpp:281-305; compute_pmf and sample_from_pmf,
// samplingHelperFunctions.cpp:78-367), all samples of a call advanced together.
//
// With k photons in, the next output mode is drawn from
//     pmf(m) ~ | sum_j minor_j U[m, col_j] |^2,
// minor_j being the column minors of the (k-1) x k matrix U[drawn modes, entered columns].
// Which photon enters and the uniform draw of each step depend on the seed alone, so they
// are known beforehand and nothing of a step has to reach the host before the next one
// starts: the loop is a chain of launches on one stream, and the drawn modes are written to
// host memory as they fall.  (With the host in the loop -- a copy each way, a wait and the
// pmf in numpy per photon -- 8 samples of 20 photons in 60 modes took 5.28 ms, over 90% of it
// outside the kernels; now 0.32 ms, 0.24 of it kernels.)
//
// * Photons 1..kHeadPhotons: one launch, a block per sample.  The minors come from the
//   permanents of all column subsets, F[S] = perm(first |S| rows, columns S), kept in LDS:
//   a new column doubles the table, F[S + c] = a[|S|][c] F[S] + sum_{j in S} a[|S|][j]
//   F[S - j + c], and minor_j is F[all - j].  Nothing is computed twice over the steps and
//   the sums have none of the cancellation of the signed ones; a step is k - 1 levels with
//   a barrier each.
// * Later photons: two launches per step over the samples that are still filling, the
//   column-minors sweep (perm_grad.hip) and a block per sample that adds up its partials,
//   draws the mode and writes the next step's matrix.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

#include "pqb_perm.h"
#include "pqb_device.h"
#include "pqb_kernels.h"
#include "pqb_engine.h"

namespace pqb {

namespace {

// Table of 2^12 entries: 64 KB, two blocks per CU.
constexpr int kHeadPhotons = 12;
constexpr int kHeadThreads = 512;
constexpr int kStepThreads = 256;
// Columns of a mode's amplitude, and terms of a subset's permanent, that are loaded
// together: the loops are short and a block is alone on its CU, so a step is latency.
constexpr int kTogether = 4;
// pmf of up to this many modes in LDS, of more in device memory
constexpr int kLdsModes = 1024;

constexpr int choose(int n, int k) { return k > n ? 0 : k == 0 ? 1 : choose(n - 1, k - 1) + choose(n - 1, k); }
// a level's sets, and the whole, have a thread each
static_assert(choose(kHeadPhotons - 1, (kHeadPhotons - 1) / 2) < kHeadThreads);

struct SampleParams {
    const double2* Ut;    // columns x modes: the interferometer's entered columns
    const int* enter;     // count x P: column (row of Ut) of the photon entering at each step
    const double* draw;   // count x P: uniform number of each step
    const int* photons;   // count, descending
    int* drawn;           // count x P: output modes
    int* host_drawn;      // the same in host memory, of the finished samples
    double2* A;           // count x k x (k + 1): matrix of the next step, packed
    double* pmf;          // count x modes, for modes > kLdsModes
    const double2* partials;  // count x nblk x k (minors sweep)
    double scale;         // of the partials' sum
    int modes, P;
    int k, nblk;          // photon step (1-based) and partials per sample of a later step
};

// |amplitude|^2 of every mode from the step's k minors, and the mode drawn (valid in the
// first wave): the first whose running sum of the normalised weights reaches `r`, mode 0
// if none does (NaN weights among them).  col: the entered columns, in LDS.
__device__ __forceinline__ int draw_mode(const SampleParams& p, const double2* minors, const int* col, int k,
                                         double r, double* pm) {
    for (int m = threadIdx.x; m < p.modes; m += blockDim.x) {
        double ar = 0.0, ai = 0.0;
        for (int j = 0; j < k; j += kTogether) {
            double2 u[kTogether];
#pragma unroll
            for (int q = 0; q < kTogether; ++q) u[q] = p.Ut[(int64_t)col[min(j + q, k - 1)] * p.modes + m];
#pragma unroll
            for (int q = 0; q < kTogether; ++q) {
                const double2 v = j + q < k ? minors[j + q] : make_double2(0.0, 0.0);
                ar = fma(v.x, u[q].x, ar);
                ar = fma(-v.y, u[q].y, ar);
                ai = fma(v.x, u[q].y, ai);
                ai = fma(v.y, u[q].x, ai);
            }
        }
        pm[m] = ar * ar + ai * ai;
    }
    __syncthreads();
    if (threadIdx.x >= kWave) return 0;
    // a lane per run of consecutive modes; the running sums are compared with r times the
    // total, not divided by it
    const int lane = threadIdx.x, per = (p.modes + kWave - 1) / kWave;
    const int m0 = min(lane * per, p.modes), m1 = min(m0 + per, p.modes);
    double sum = 0.0;
    for (int m = m0; m < m1; ++m) sum += pm[m];
    double incl = sum;  // inclusive sums over the lanes
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const double o = __shfl_up(incl, d, kWave);
        if (lane >= d) incl += o;
    }
    double before = __shfl_up(incl, 1, kWave);
    if (lane == 0) before = 0.0;
    const double total = __shfl(incl, kWave - 1, kWave);
    if (!(total > 0.0 && total <= 1.7976931348623157e308)) return 0;  // no weight, infinite, NaN
    const double level = r * total;
    const unsigned long long hit = __ballot(m0 < m1 && incl >= level);
    if (hit == 0) return 0;
    const int who = __builtin_ctzll(hit);
    int got = -1, last = m0;
    if (lane == who) {
        double at = 0.0;
        for (int m = m0; m < m1 && got < 0; ++m) {
            at += pm[m];
            if (pm[m] > 0.0) last = m;
            if (before + at >= level) got = m;
        }
        if (got < 0) got = last;  // the lanes' sums round differently
    }
    return __shfl(got, who, kWave);
}

// The modes drawn up to step k, for the next step or, after the sample's last, for the
// host.  Written once per launch: a barrier waits for the stores before it, those over the
// bus too.
__device__ __forceinline__ void record_modes(const SampleParams& p, int s, int n, int k, const int* row) {
    int* const to = (n == k ? p.host_drawn : p.drawn) + (int64_t)s * p.P;
    if (threadIdx.x < (unsigned)k) to[threadIdx.x] = row[threadIdx.x];
}

// The k x (k + 1) matrix of step k + 1: rows the modes drawn so far, columns the entered ones.
__device__ __forceinline__ void next_matrix(const SampleParams& p, int s, int k, const int* row, const int* col) {
    double2* const A = p.A + (int64_t)s * k * (k + 1);
    for (int e = threadIdx.x; e < k * (k + 1); e += blockDim.x) {
        const int i = e / (k + 1), j = e - i * (k + 1);
        A[e] = p.Ut[(int64_t)col[j] * p.modes + row[i]];
    }
}

__global__ __launch_bounds__(kHeadThreads) void sample_head_kernel(SampleParams p) {
    __shared__ double2 F[1 << kHeadPhotons];
    __shared__ double2 a[kHeadPhotons][kHeadPhotons];
    __shared__ double2 minors[kHeadPhotons];
    __shared__ double pm_lds[kLdsModes];
    __shared__ int col[kHeadPhotons + 1], row[kHeadPhotons];
    __shared__ double draw[kHeadPhotons];
    // the subsets of the earlier columns by size, then value: those of i of the first b
    // columns are the first C(b, i) of their size's, so that a level's sets go to as many
    // consecutive threads.  (With a test of every subset's size instead, a store of each
    // mode to the host as it falls and a second scan over the normalised weights, the same
    // run took 352 us against 318.)
    __shared__ int binom[kHeadPhotons][kHeadPhotons + 1], first[kHeadPhotons + 1];
    __shared__ unsigned short by_size[1 << (kHeadPhotons - 1)];
    const int s = blockIdx.x, tid = threadIdx.x;
    const int n = p.photons[s], last = min(n, kHeadPhotons);
    double* const pm = p.modes <= kLdsModes ? pm_lds : p.pmf + (int64_t)s * p.modes;
    if (tid <= kHeadPhotons && tid < n) col[tid] = p.enter[(int64_t)s * p.P + tid];
    if (tid >= kWave && tid - kWave < last) draw[tid - kWave] = p.draw[(int64_t)s * p.P + tid - kWave];
    if (tid == 0) F[0] = make_double2(1.0, 0.0);
    if (tid < kHeadPhotons * (kHeadPhotons + 1)) {
        const int b = tid / (kHeadPhotons + 1), size = tid % (kHeadPhotons + 1);
        int c = size > b ? 0 : 1;
        for (int q = 1; q <= size; ++q) c = c * (b - size + q) / q;  // C(b, size)
        binom[b][size] = c;
    }
    __syncthreads();
    if (tid <= kHeadPhotons) {
        int at = 0;
        for (int q = 0; q < tid; ++q) at += binom[kHeadPhotons - 1][q];
        first[tid] = at;
    }
    __syncthreads();
    for (unsigned e = tid; e < (1u << (kHeadPhotons - 1)); e += blockDim.x) {
        int at = first[__builtin_popcount(e)], size = 0;
        for (unsigned left = e; left; left &= left - 1) at += binom[__builtin_ctz(left)][++size];
        by_size[at] = (unsigned short)e;
    }
    __syncthreads();
    for (int k = 1; k <= last; ++k) {
        // a[i][j], i < k - 1, j < k: the last row and the last column are new
        if (k > 1) {
            if (tid < k) a[k - 2][tid] = p.Ut[(int64_t)col[tid] * p.modes + row[k - 2]];
            else if (tid >= kWave && tid - kWave < k - 2)
                a[tid - kWave][k - 1] = p.Ut[(int64_t)col[k - 1] * p.modes + row[tid - kWave]];
            __syncthreads();
        }
        const unsigned old = 1u << (k - 1);  // the new column's bit
        for (int i = 1; i < k; ++i) {
            // sets of i columns, the new one among them; at the last level also the set of
            // all the earlier columns, whose row has just been drawn
            const int sets = binom[k - 1][i - 1];
            if (tid < sets + (i == k - 1)) {
                const unsigned T = tid < sets ? by_size[first[i - 1] + tid] | old : old - 1;
                double2 f = make_double2(0.0, 0.0);
                unsigned left = T;  // i columns
                for (int t = 0; t < i; t += kTogether) {
                    double2 c[kTogether], g[kTogether];
#pragma unroll
                    for (int q = 0; q < kTogether; ++q) {
                        const unsigned bit = left & (0u - left);
                        left ^= bit;
                        c[q] = bit ? a[i - 1][__builtin_ctz(bit | old << 1)] : make_double2(0.0, 0.0);
                        g[q] = F[bit ? T ^ bit : 0u];
                    }
#pragma unroll
                    for (int q = 0; q < kTogether; ++q) {
                        f.x = fma(c[q].x, g[q].x, f.x);
                        f.x = fma(-c[q].y, g[q].y, f.x);
                        f.y = fma(c[q].x, g[q].y, f.y);
                        f.y = fma(c[q].y, g[q].x, f.y);
                    }
                }
                F[T] = f;
            }
            __syncthreads();
        }
        if (tid < k) minors[tid] = F[(2 * old - 1) ^ (1u << tid)];
        __syncthreads();
        const int mode = draw_mode(p, minors, col, k, draw[k - 1], pm);
        if (tid == 0) row[k - 1] = mode;
        __syncthreads();
    }
    record_modes(p, s, n, last, row);
    if (n > kHeadPhotons) next_matrix(p, s, kHeadPhotons, row, col);
}

// Photon step p.k > kHeadPhotons after its minors sweep.
__global__ __launch_bounds__(kStepThreads) void sample_step_kernel(SampleParams p) {
    __shared__ ddc red[kStepThreads];
    __shared__ double2 minors[kMaxCols];
    __shared__ double pm_lds[kLdsModes];
    __shared__ int col[kMaxCols + 1], row[kMaxCols];
    const int s = blockIdx.x, tid = threadIdx.x, k = p.k;
    const int n = p.photons[s];
    double* const pm = p.modes <= kLdsModes ? pm_lds : p.pmf + (int64_t)s * p.modes;
    if (tid <= k && tid < n) col[tid] = p.enter[(int64_t)s * p.P + tid];
    if (tid >= kWave && tid - kWave < k - 1) row[tid - kWave] = p.drawn[(int64_t)s * p.P + tid - kWave];
    // the partials in double-double, `slices` threads per column
    const int slices = kStepThreads / k, j = tid % k, slice = tid / k;
    ddc v = {0.0, 0.0, 0.0, 0.0};
    if (slice < slices) {
        const double2* const src = p.partials + (int64_t)s * p.nblk * k + j;
#pragma unroll 8
        for (int b = slice; b < p.nblk; b += slices) {
            const double2 x = src[(int64_t)b * k];
            ddc_add(v, ddc_from(x.x, x.y));
        }
        red[tid] = v;
    }
    __syncthreads();
    for (int left = slices; left > 1;) {
        const int half = (left + 1) / 2;
        if (slice < left - half) ddc_add(red[tid], red[tid + half * k]);
        __syncthreads();
        left = half;
    }
    if (tid < k) {
        v = ddc_scale(red[tid], p.scale);
        minors[tid] = make_double2(v.hr + v.lr, v.hi + v.li);
    }
    __syncthreads();
    const int mode = draw_mode(p, minors, col, k, p.draw[(int64_t)s * p.P + k - 1], pm);
    if (tid == 0) row[k - 1] = mode;
    __syncthreads();
    record_modes(p, s, n, k, row);
    if (n > k) next_matrix(p, s, k, row, col);
}

}  // namespace

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// Samples `which[0 .. count)` (photons descending), on the context's stream; waits.
static int sample_group(Engine& E, const double* U, int modes, int64_t ld, const int64_t* which, int count, int P,
                        const int64_t* photons, const int64_t* entering, int64_t row_stride, const double* draws,
                        int64_t* samples) {
    const int most = (int)photons[which[0]];
    if (most == 0) return PQB_OK;
    // the entered columns, in order of their first use
    std::vector<int> column(modes, -1), order;
    for (int q = 0; q < count; ++q)
        for (int64_t t = 0; t < photons[which[q]]; ++t) {
            const int64_t c = entering[which[q] * row_stride + t];
            if (column[(size_t)c] < 0) {
                column[(size_t)c] = (int)order.size();
                order.push_back((int)c);
            }
        }
    std::vector<int> active((size_t)most + 1, 0);  // samples with at least k photons
    for (int q = 0; q < count; ++q) active[(size_t)photons[which[q]]]++;
    for (int k = most - 1; k >= 0; --k) active[(size_t)k] += active[(size_t)k + 1];

    std::vector<MinorsSweep> sweep((size_t)most + 1);
    size_t part_bytes = 0;
    for (int k = kHeadPhotons + 1; k <= most; ++k) {
        const int st = minors_sweep_plan(k - 1, active[(size_t)k], &sweep[(size_t)k]);
        if (st) return st;
        part_bytes = std::max(part_bytes, sweep[(size_t)k].partial_bytes);
    }
    const size_t np = (size_t)count * P;
    const size_t u_bytes = (size_t)modes * order.size() * sizeof(double2);
    // staged inputs: Ut, draws, entered columns, photons; then device-only areas
    const size_t draw_off = align256(u_bytes), enter_off = draw_off + align256(np * sizeof(double));
    const size_t ph_off = enter_off + align256(np * sizeof(int));
    const size_t in_bytes = ph_off + align256((size_t)count * sizeof(int));
    const size_t drawn_off = in_bytes, a_off = drawn_off + align256(np * sizeof(int));
    const size_t a_bytes = most > kHeadPhotons ? (size_t)count * (most - 1) * most * sizeof(double2) : 0;
    const size_t pmf_off = a_off + align256(a_bytes);
    const size_t pmf_bytes = modes > kLdsModes ? (size_t)count * modes * sizeof(double) : 0;
    const size_t part_off = pmf_off + align256(pmf_bytes);
    int st = E.ensure_buffers_locked(kCounterBytes + part_off + part_bytes, in_bytes + np * sizeof(int));
    if (st) return st;
    char* const d = static_cast<char*>(E.dbuf) + kCounterBytes;  // offset 0 holds the plain sweep's grid counter
    char* const h = static_cast<char*>(E.hbuf);

    double* const hu = reinterpret_cast<double*>(h);
    for (size_t c = 0; c < order.size(); ++c)
        for (int m = 0; m < modes; ++m)
            std::memcpy(hu + 2 * (c * modes + m), U + 2 * (m * ld + order[c]), 2 * sizeof(double));
    double* const hd = reinterpret_cast<double*>(h + draw_off);
    int* const he = reinterpret_cast<int*>(h + enter_off);
    int* const hp = reinterpret_cast<int*>(h + ph_off);
    for (int q = 0; q < count; ++q) {
        hp[q] = (int)photons[which[q]];
        for (int t = 0; t < P; ++t) {
            const bool in = t < hp[q];
            he[(size_t)q * P + t] = in ? column[(size_t)entering[which[q] * row_stride + t]] : 0;
            hd[(size_t)q * P + t] = in ? draws[which[q] * row_stride + t] : 0.0;
        }
    }
    hipError_t e = hipMemcpyAsync(d, h, in_bytes, hipMemcpyHostToDevice, E.stream);
    if (e != hipSuccess) return drain_fail(E, e, "hipMemcpyAsync");

    SampleParams p{};
    p.Ut = reinterpret_cast<const double2*>(d);
    p.draw = reinterpret_cast<const double*>(d + draw_off);
    p.enter = reinterpret_cast<const int*>(d + enter_off);
    p.photons = reinterpret_cast<const int*>(d + ph_off);
    p.drawn = reinterpret_cast<int*>(d + drawn_off);
    p.host_drawn = reinterpret_cast<int*>(h + in_bytes);
    p.A = reinterpret_cast<double2*>(d + a_off);
    p.pmf = reinterpret_cast<double*>(d + pmf_off);
    p.partials = reinterpret_cast<const double2*>(d + part_off);
    p.modes = modes;
    p.P = P;
    hipLaunchKernelGGL(sample_head_kernel, dim3((unsigned)active[1]), dim3(kHeadThreads), 0, E.stream, p);
    e = hipGetLastError();
    if (e != hipSuccess) return drain_fail(E, e, "sampler launch");
    for (int k = kHeadPhotons + 1; k <= most; ++k) {
        st = minors_sweep_launch(sweep[(size_t)k], p.A, d + part_off, E.stream);
        if (st) {
            (void)hipStreamSynchronize(E.stream);
            return st;
        }
        p.k = k;
        p.nblk = sweep[(size_t)k].nblk;
        p.scale = std::ldexp(1.0, -(k - 2));
        hipLaunchKernelGGL(sample_step_kernel, dim3((unsigned)active[(size_t)k]), dim3(kStepThreads), 0, E.stream, p);
        e = hipGetLastError();
        if (e != hipSuccess) return drain_fail(E, e, "sampler step launch");
    }
    e = hipStreamSynchronize(E.stream);
    if (e != hipSuccess) return hip_fail(e, "sampler");
    for (int q = 0; q < count; ++q)
        for (int t = 0; t < hp[q]; ++t) samples[which[q] * (int64_t)modes + p.host_drawn[(size_t)q * P + t]]++;
    return PQB_OK;
}

static int sample_entry(const double* U, int64_t modes, int64_t ld, int64_t count, int64_t max_photons,
                        const int64_t* photons, const int64_t* entering, const double* draws, int64_t* samples) {
    if (count < 0 || modes < 1 || modes > 0x7fffffff || max_photons < 0)
        return fail(PQB_ERR_ARG, "sample count, mode count and photon count must not be negative");
    if (max_photons > kMaxCols)
        return fail(PQB_ERR_SIZE, "more than " + std::to_string(kMaxCols) + " photons");
    if (count == 0) return PQB_OK;
    if (!U || !photons || !samples || (max_photons > 0 && (!entering || !draws)))
        return fail(PQB_ERR_ARG, "NULL pointer");
    if (ld < modes) return fail(PQB_ERR_ARG, "leading dimension smaller than the number of modes");
    for (int64_t s = 0; s < count; ++s) {
        if (photons[s] < 0 || photons[s] > max_photons) return fail(PQB_ERR_ARG, "photon count out of range");
        for (int64_t t = 0; t < photons[s]; ++t)
            if (entering[s * max_photons + t] < 0 || entering[s * max_photons + t] >= modes)
                return fail(PQB_ERR_ARG, "input mode out of range");
    }
    std::fill(samples, samples + count * modes, (int64_t)0);
    // samples of as many photons side by side, so that the ones still filling come first
    std::vector<int64_t> which((size_t)count);
    std::iota(which.begin(), which.end(), (int64_t)0);
    std::stable_sort(which.begin(), which.end(), [&](int64_t a, int64_t b) { return photons[a] > photons[b]; });

    Lease L;
    int st = L.status();
    if (st) return st;
    // groups that keep a sample's matrices and weights within a few hundred MB
    const int64_t per = 16 * max_photons * (max_photons + 1) + 8 * modes + 64;
    const int64_t group = std::min<int64_t>(4096, std::max<int64_t>(1, ((int64_t)256 << 20) / per));
    for (int64_t at = 0; at < count; at += group) {
        st = sample_group(*L, U, (int)modes, ld, which.data() + at, (int)std::min(group, count - at),
                          (int)max_photons, photons, entering, max_photons, draws, samples);
        if (st) return st;
    }
    return PQB_OK;
}

}  // namespace pqb

using namespace pqb;

extern "C" int pqb_sample_photons(const double* U, int64_t modes, int64_t ld, int64_t count, int64_t max_photons,
                                  const int64_t* photons, const int64_t* entering, const double* draws,
                                  int64_t* samples) {
    try {
        return sample_entry(U, modes, ld, count, max_photons, photons, entering, draws, samples);
    } catch (const std::exception& ex) {
        return fail(PQB_ERR_DEVICE, std::string("internal error: ") + ex.what());
    }
}
