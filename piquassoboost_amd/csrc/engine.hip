// Host engine behind the C ABI declared in include/pqb_perm.h.
//
// Responsibilities: argument checks and the reference's edge-case rules,
// choice of the sweep decomposition (chunk bits K, chunk-index bits H, lane
// count), staging host matrices into a per-process device workspace, kernel
// launches on the engine's stream, and error reporting (status code +
// thread-local message; no C++ exception crosses the ABI).
//
// The host-pointer entry points are synchronous (as the reference calculators
// are: the GIL is held and TBB blocks, GlynnPermanentCalculator_Wrapper.hpp:
// 200-377) and thread safe: each call leases one of kEngineContexts execution
// contexts (stream, device workspace, pinned staging, batch buffers and graphs)
// for its duration, so calls from different threads run on different streams
// at the same time.  The device-pointer entry points take the caller's stream
// and workspace and touch no context, only the shared device state (binding,
// occupancy of the kernels).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <atomic>
#include <mutex>
#include <string>
#include <vector>

#include "pqb_perm.h"
#include "pqb_device.h"
#include "pqb_exact_rule.h"
#include "pqb_kernels.h"
#include "pqb_engine.h"

namespace pqb {

thread_local std::string t_err;

int fail(int code, const std::string& msg) {
    t_err = msg;
    return code;
}

int hip_fail(hipError_t e, const char* what) {
    return fail(PQB_ERR_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

// A few microseconds of a small call are the runtime's: hipStreamSynchronize queues a
// marker behind the kernel and waits for its signal.  The kernel's own word in host memory
// is polled instead for about as long as a small call takes; a longer one, or one that
// failed, is waited for as usual.  The stream stays in order, so the next call needs no more.
hipError_t wait_result(Engine& E, const unsigned* done) {
    const auto began = std::chrono::steady_clock::now();
    do {
        for (int k = 0; k < 64; ++k) {
            if (__atomic_load_n(done, __ATOMIC_ACQUIRE)) return hipSuccess;
            __builtin_ia32_pause();
        }
    } while (std::chrono::steady_clock::now() - began < std::chrono::microseconds(200));
    return hipStreamSynchronize(E.stream);
}

int drain_fail(Engine& E, hipError_t e, const char* what) {
    if (E.stream) (void)hipStreamSynchronize(E.stream);
    return hip_fail(e, what);
}

DeviceState g_dev;
Engine g_ctx[kEngineContexts];

// ----------------------------------------------------------- device state --

// Binding under g_dev.mu (held): device `dev` (< 0: 0) becomes the engine's.
static int set_device_locked(int dev) {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n <= 0)
        return fail(PQB_ERR_DEVICE, "no HIP device available (the permanent engine runs on the GPU only)");
    if (dev < 0) dev = 0;
    if (dev >= n) return fail(PQB_ERR_ARG, "device index out of range");
    e = hipSetDevice(dev);
    if (e != hipSuccess) return hip_fail(e, "hipSetDevice");
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDeviceProperties");
    g_dev.cus = prop.multiProcessorCount;
    for (int i = 0; i <= PQB_MAX_COLS; ++i) g_dev.blocks_per_cu[0][i] = g_dev.blocks_per_cu[1][i] = 0;
    g_dev.device = dev;
    return PQB_OK;
}

int bind_device(int dev, int* device, int* cus) {
    {
        std::lock_guard<std::mutex> lk(g_dev.mu);
        const bool keep = g_dev.device >= 0 && (dev < 0 || dev == g_dev.device);
        // the first binding: no context has a stream or buffers yet (they are
        // created only after a binding), so nothing needs releasing
        const int st = keep ? PQB_OK : (g_dev.device < 0 ? set_device_locked(dev) : -1);
        if (st >= 0) {
            if (st == PQB_OK) {
                if (device) *device = g_dev.device;
                if (cus) *cus = g_dev.cus;
            }
            return st;
        }
    }
    // a change of device (pqb_init, never called from inside a context's lease):
    // every context is locked -- in index order, before g_dev.mu, the order every
    // caller follows -- and releases its stream and buffers first
    std::unique_lock<std::mutex> held[kEngineContexts];
    for (int k = 0; k < kEngineContexts; ++k) held[k] = std::unique_lock<std::mutex>(g_ctx[k].mu);
    std::lock_guard<std::mutex> lk(g_dev.mu);
    if (!(g_dev.device >= 0 && (dev < 0 || dev == g_dev.device))) {
        for (int k = 0; k < kEngineContexts; ++k) g_ctx[k].release_locked();
        const int st = set_device_locked(dev);
        if (st) return st;
    }
    if (device) *device = g_dev.device;
    if (cus) *cus = g_dev.cus;
    return PQB_OK;
}

int64_t resident_waves(int nc, bool expanded) {
    if (nc < 1 || nc > PQB_MAX_COLS) return 0;
    std::lock_guard<std::mutex> lk(g_dev.mu);
    int& per_cu = g_dev.blocks_per_cu[expanded][nc];
    if (per_cu == 0) {
        int nb = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, plain_kernel_fn(nc, expanded), kBlock, 0);
        if (e != hipSuccess || nb <= 0) nb = 1;
        per_cu = nb;
    }
    return (int64_t)per_cu * (kBlock / kWave) * g_dev.cus;
}

// ---------------------------------------------------------------- contexts --

void release_batch_locked(Engine& E);  // batch.hip

void Engine::release_locked() {
    if (stream) (void)hipStreamSynchronize(stream);
    release_batch_locked(*this);
    if (dbuf) (void)hipFree(dbuf);
    if (hbuf) (void)hipHostFree(hbuf);
    dbuf = nullptr;
    hbuf = nullptr;
    dbytes = hbytes = 0;
    if (stream) (void)hipStreamDestroy(stream);
    stream = nullptr;
    device = -1;
}

int Engine::ensure_init_locked() {
    int dev = -1, ncu = 0;
    int st = bind_device(-1, &dev, &ncu);
    if (st) return st;
    hipError_t e = hipSetDevice(dev);
    if (e != hipSuccess) return hip_fail(e, "hipSetDevice");
    if (device == dev && stream) return PQB_OK;
    release_locked();
    e = hipStreamCreateWithFlags(&stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        stream = nullptr;
        return hip_fail(e, "hipStreamCreate");
    }
    device = dev;
    cus = ncu;
    return PQB_OK;
}

int Engine::ensure_buffers_locked(size_t dneed, size_t hneed) {
    const size_t old_d = dbytes, old_h = hbytes;
    if (dneed > dbytes) {
        if (dbuf) {
            (void)hipStreamSynchronize(stream);
            (void)hipFree(dbuf);
            dbuf = nullptr;
            dbytes = 0;
        }
        // geometric growth: a caller whose sizes creep up (a sampler going photon by
        // photon) reallocates a few times, not at every step
        const size_t sz = std::max<size_t>(std::max<size_t>(dneed, 2 * old_d), (size_t)1 << 20);
        hipError_t e = hipMalloc(&dbuf, sz);
        if (e != hipSuccess) {
            dbuf = nullptr;
            return hip_fail(e, "hipMalloc(workspace)");
        }
        // the grid-reduction counter at offset 0 must start at zero
        e = hipMemsetAsync(dbuf, 0, kCounterBytes, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (e != hipSuccess) return hip_fail(e, "hipMemset(workspace)");
        dbytes = sz;
    }
    if (hneed > hbytes) {
        if (hbuf) {
            (void)hipStreamSynchronize(stream);
            (void)hipHostFree(hbuf);
            hbuf = nullptr;
            hbytes = 0;
        }
        const size_t sz = std::max<size_t>(std::max<size_t>(hneed, 2 * old_h), (size_t)1 << 20);
        hipError_t e = hipHostMalloc(&hbuf, sz, hipHostMallocCoherent);
        if (e != hipSuccess) {
            hbuf = nullptr;
            return hip_fail(e, "hipHostMalloc(staging)");
        }
        hbytes = sz;
    }
    return PQB_OK;
}

// A thread keeps using the context it was first given when that one is free,
// so a single-threaded caller always runs on one stream and one set of buffers.
static int preferred_context() {
    static std::atomic<unsigned> next{0};
    thread_local int pref = (int)(next.fetch_add(1u) % (unsigned)kEngineContexts);
    return pref;
}

Lease::Lease() {
    const int pref = preferred_context();
    for (int k = 0; k < kEngineContexts && !e_; ++k) {
        Engine& c = g_ctx[(pref + k) % kEngineContexts];
        std::unique_lock<std::mutex> l(c.mu, std::try_to_lock);
        if (l.owns_lock()) {
            lk_ = std::move(l);
            e_ = &c;
        }
    }
    if (!e_) {
        e_ = &g_ctx[pref];
        lk_ = std::unique_lock<std::mutex>(e_->mu);
    }
    st_ = e_->ensure_init_locked();
}

Lease::Lease(Engine& e) : e_(&e), lk_(e.mu) { st_ = e_->ensure_init_locked(); }

// --------------------------------------------------------------- planning --

static int floor_log2(int64_t v) {
    int r = -1;
    while (v > 0) {
        v >>= 1;
        ++r;
    }
    return r;
}

static int ceil_log2(int64_t v) {
    int r = 0;
    while (((int64_t)1 << r) < v) ++r;
    return r;
}

// Split of the R-1 sign bits into walk (K), lane (B) and group (H) bits and
// the number of waves.  The kernel gives every wave one contiguous run of the
// walk index (group * 2^K + t) in step pairs, so runs are equal to within one
// pair and may start and end inside a group: the launch is exactly the
// resident waves, one round at full occupancy.  (Whole groups per wave would
// need a power-of-two wave count: 4096 waves of two groups each at n=30 left a
// quarter of the work to a second round at one wave per SIMD.)  The walk is
// long enough that a run spans a few groups; small sweeps take the shortest
// walk that still amortises the seed.
PlainPlan make_plain_plan(int R, int NC, int64_t waves_resident) {
    (void)NC;
    PlainPlan pl;
    const int T = R - 1;
    const int64_t wr = std::max<int64_t>(waves_resident, 1);
    int K = T - 6 - (ceil_log2(wr) + 1);
    K = std::max(K, std::min(T, 3));
    K = std::min(K, std::min(T, 14));
    pl.K = K;
    pl.B = std::min(6, T - K);
    pl.H = T - K - pl.B;
    const int64_t units = ((int64_t)1 << (pl.H + pl.K)) / (pl.K >= 1 ? 2 : 1);  // step pairs
    // Up to a block per CU every wave gets one pair; past that runs grow to kMinRun pairs
    // before more waves are launched, since each block costs an atomic on the counter the
    // grid finishes by (n = 20: 1024 blocks of one pair per wave 22.8 us, 256 blocks 15.4 us;
    // a minimum of 16 pairs costs n = 22 25.6 against 22.2 us).
    constexpr int64_t kSpread = 1024, kMinRun = 8;
    const int64_t waves_wanted = std::max(std::min(units, kSpread), units / kMinRun);
    int64_t waves = std::min<int64_t>(waves_wanted, wr);
    if (waves >= 4) {
        waves -= waves % 4;
        pl.block = kBlock;
        pl.blocks = (int)(waves / 4);
    } else {
        pl.block = (int)(64 * waves);
        pl.blocks = 1;
    }
    pl.waves = (int64_t)pl.blocks * pl.block / kWave;
    return pl;
}

// From 12 rows on the block's LDS traffic costs more than the sweep's copy and second
// launch (device entry, tiny / sweep: n = 11 8.0 / 9.1 us, n = 12 10.4 / 9.2), and so it
// does for more matrices than CUs (8192 x 10: 69 / 31 us).
bool plain_tiny(int R, int C, int64_t count, TinyParams& p) {
    if (R > kTinyRows || count > 256) return false;
    p = TinyParams{};
    std::fill(p.radix, p.radix + (R - 1), (unsigned char)2);
    p.stride = (int64_t)R * C;
    p.scale = std::ldexp(1.0, -(R - 1));
    return tiny_split(p, C, R);
}

// The expanded sweep does 10 n instead of 12 n FP64 instructions per pair of sign
// vectors; its table costs a launch, and device matrices a second sweep launch for the
// ones that keep all rows.  From 2^24 sign vectors on that pays (all rows / expanded,
// us, device entries, one box): 1 x 24 50.3 / 53.0, 1 x 25 89 / 86, 1 x 26 169 / 153,
// 1 x 30 2929 / 2495; 16 x 20 43.2 / 45.5, 64 x 20 138 / 120, 256 x 20 502 / 422;
// 4 x 22 46.8 / 48.8, 8 x 22 82.7 / 76.6; 512 x 16 61.1 / 60.0, 2048 x 14 65.7 / 61.4.
// Below 14 columns a table of n^2 quotients per matrix costs more than the walk of
// 2^(n-2) vectors saves (8192 x 12: 64.7 / 90.3).
bool plain_expandable(int R, int C, int64_t count) {
    return R == C && C >= kExpandedMinCols && count >= ((int64_t)1 << std::max(0, 25 - C));
}

// +-2A of an R x C matrix with row stride ld.
static void fill_m2(const double* A, int R, int C, int64_t ld, double* t) {
    const size_t rc = (size_t)R * C;
    for (int i = 0; i < R; ++i)
        for (int j = 0; j < C; ++j) {
            const double re = A[2 * (i * ld + j)], im = A[2 * (i * ld + j) + 1];
            const size_t q = (size_t)i * C + j;
            t[2 * q] = 2.0 * re;
            t[2 * q + 1] = 2.0 * im;
            t[2 * (q + rc)] = -2.0 * re;
            t[2 * (q + rc) + 1] = -2.0 * im;
        }
}

PlainParams plain_params(const PlainPlan& pl, int R, const double2* m2, int64_t m2_stride, ddc* partials,
                         unsigned* counter, double* out) {
    PlainParams p;
    p.M2 = m2;
    p.m2_stride = m2_stride;
    p.R = R;
    p.K = pl.K;
    p.B = pl.B;
    p.H = pl.H;
    p.by_flag = 0;
    p.partials = partials;
    p.counter = counter;
    p.out = out;
    p.scale = std::ldexp(1.0, -(R - 1));
    p.done = nullptr;
    return p;
}

static void pack_rows(const double* A, int R, int C, int64_t ld, double* t) {
    for (int i = 0; i < R; ++i)
        std::memcpy(t + 2 * (size_t)i * C, A + 2 * i * ld, (size_t)C * sizeof(double2));
}

// Integer route eligibility.  Fills `ai` (packed R x C int32) when the matrix
// is integer valued and real, and returns log2 of an upper bound on the sweep's
// sum S = sum_delta (prod delta) prod_j (sum_i delta_i a_ij) (or -inf when S is
// provably 0).  For every shape, |S| <= 2^(R-1) prod_j c_j (c_j = column abs
// sums: each of the 2^(R-1) terms is bounded by that product; a zero column
// makes every term 0).  Only for R == C is S = 2^(R-1) perm(A), so only there
// do the row-sum bound perm(|A|) <= prod_i r_i and, for entries in {-1, 0, 1},
// Bregman's bound perm(|A|) <= prod_i (r_i!)^(1/r_i) (also applied to the
// transpose) hold; for R != C the sum is not a permanent of A (R = C + 1 gives
// 2^(R-1) perm(A without row 0), R < C counts maps with odd row multiplicities)
// and a row bound can be arbitrarily wrong.  The sweep sums modulo 2^128, so
// the result is exact when the bound is below 2^127; column sums must also fit
// in int32.
static bool integer_matrix(const double* A, int64_t R, int64_t C, int64_t ld, std::vector<int>& ai,
                           long double* log2_bound) {
    ai.assign((size_t)(R * C), 0);
    std::vector<double> rowabs((size_t)R, 0.0), colabs((size_t)C, 0.0);
    bool unit = true;
    for (int64_t i = 0; i < R; ++i) {
        for (int64_t j = 0; j < C; ++j) {
            const double re = A[2 * (i * ld + j)];
            const double im = A[2 * (i * ld + j) + 1];
            if (im != 0.0 || !(std::fabs(re) < 1073741824.0) || re != std::floor(re)) return false;
            ai[(size_t)(i * C + j)] = (int)re;
            const double a = std::fabs(re);
            if (a > 1.0) unit = false;
            rowabs[(size_t)i] += a;
            colabs[(size_t)j] += a;
        }
    }
    for (int64_t j = 0; j < C; ++j)
        if (colabs[(size_t)j] >= 1073741824.0) return false;  // int32 column sums
    auto lg_prod = [](const std::vector<double>& v, bool bregman) -> long double {
        long double s = 0.0L;
        for (double x : v) {
            if (x == 0.0) return -INFINITY;
            s += bregman ? std::lgamma((long double)x + 1.0L) / (long double)x / std::log(2.0L)
                         : std::log2((long double)x);
        }
        return s;
    };
    long double lb = lg_prod(colabs, false);
    if (R == C) {
        lb = std::min(lb, lg_prod(rowabs, false));
        if (unit) lb = std::min(lb, std::min(lg_prod(rowabs, true), lg_prod(colabs, true)));
    }
    *log2_bound = lb + (long double)(R - 1);
    return true;
}

static bool exact_fits(long double log2_bound) { return log2_bound < 126.5L; }

static size_t round256(size_t b) { return (b + 255) / 256 * 256; }

typedef __int128 i128;

static double i128_to_double(i128 v) { return (double)v; }

// Exact route: sum_delta (prod delta) prod_j c_j  (mod 2^128) on the GPU,
// then divide by 2^(R-1).  The caller holds the lease of E.
static int run_exact_locked(Engine& E, const std::vector<int>& ai, int R, int C, i128* result) {
    const int T = R - 1;
    // every running column sum is bounded by its column's abs sum
    int64_t cmax = 0;
    for (int j = 0; j < C; ++j) {
        int64_t s = 0;
        for (int i = 0; i < R; ++i) s += std::llabs((long long)ai[(size_t)i * C + j]);
        cmax = std::max(cmax, s);
    }
    const int flush = exact_fp64_flush(cmax, C);
    int K, B = 0, H, block;
    int64_t blocks;
    if (flush) {
        // four waves per SIMD, walks of at least 8 steps
        K = std::max(T - (floor_log2((int64_t)16 * E.cus) + 6), std::min(T, 3));
        B = std::min(6, T - K);
        H = T - K - B;
        const int64_t waves = (int64_t)1 << H;
        block = (int)std::min<int64_t>(kExactBlock, waves * kWave);
        blocks = waves * kWave / block;
    } else {
        const int64_t lr = E.resident_waves_locked(C) * kWave;
        H = std::min(T, std::max(0, floor_log2(std::max<int64_t>(lr, kWave))));
        K = T - H;
        const int64_t nlanes = (int64_t)1 << H;
        block = (int)std::min<int64_t>(kBlock, ((nlanes + kWave - 1) / kWave) * kWave);
        blocks = (nlanes + block - 1) / block;
    }
    if (K > 30) return fail(PQB_ERR_SIZE, "exact sweep too large");

    const size_t a_bytes = ai.size() * sizeof(double);  // doubles, or ints in half of it
    const size_t part_off = kCounterBytes;
    const size_t part_bytes = (size_t)blocks * 2 * sizeof(unsigned long long);
    const size_t a_off = part_off + round256(part_bytes);
    int st = E.ensure_buffers_locked(a_off + a_bytes, a_bytes + 256);
    if (st) return st;
    char* d = static_cast<char*>(E.dbuf);
    if (flush) {
        double* h = static_cast<double*>(E.hbuf);
        for (size_t k = 0; k < ai.size(); ++k) h[k] = 2.0 * ai[k];
    } else {
        std::memcpy(E.hbuf, ai.data(), ai.size() * sizeof(int));
    }
    hipError_t e = hipMemcpyAsync(d + a_off, E.hbuf, ai.size() * (flush ? sizeof(double) : sizeof(int)),
                                  hipMemcpyHostToDevice, E.stream);
    if (e != hipSuccess) return hip_fail(e, "hipMemcpyAsync");
    auto* partials = reinterpret_cast<unsigned long long*>(d + part_off);
    auto* counter = reinterpret_cast<unsigned*>(d);
    // the kernel writes the result to the staging buffer itself
    auto* hout = reinterpret_cast<unsigned long long*>(static_cast<char*>(E.hbuf) + a_bytes);
    auto* done = reinterpret_cast<unsigned*>(hout + 2);
    *done = 0u;
    if (flush) {
        const ExactF64Params p{reinterpret_cast<const double*>(d + a_off), R, K, B, H, flush, partials, counter, hout,
                               done};
        e = launch_plain_exact_fp64(C, p, (int)blocks, block, E.stream);
    } else {
        // 28^13, 1400^6 and (2^30)^2 are below 2^63 (integer_matrix admits column abs sums below 2^30)
        ExactParams p;
        p.A = reinterpret_cast<const int*>(d + a_off);
        p.R = R;
        p.K = K;
        p.H = H;
        p.group = cmax <= 28 ? 13 : (cmax <= 1400 ? 6 : 2);
        p.nlanes = (int64_t)1 << H;
        p.partials = partials;
        p.counter = counter;
        p.out = hout;
        e = launch_plain_exact(C, p, (int)blocks, block, E.stream);
    }
    if (e != hipSuccess) return drain_fail(E, e, "exact sweep launch");
    e = flush ? wait_result(E, done) : hipStreamSynchronize(E.stream);
    if (e != hipSuccess) return hip_fail(e, "exact sweep");
    const unsigned __int128 u = ((unsigned __int128)hout[1] << 64) | hout[0];
    const i128 sum = (i128)u;
    const i128 mask = (((i128)1) << T) - 1;
    if ((sum & mask) != 0) return fail(PQB_ERR_EXACT, "exact sweep: sum not divisible by 2^(rows-1)");
    *result = sum >> T;  // arithmetic shift: exact division
    return PQB_OK;
}

// FP64 route.  The caller holds the lease of E.
static int run_plain_locked(Engine& E, const double* A, int R, int C, int64_t ld, double* out) {
    TinyParams t;
    if (plain_tiny(R, C, 1, t)) {
        const size_t a_bytes = (size_t)R * C * sizeof(double2);
        int st = E.ensure_buffers_locked(0, a_bytes + 7 * sizeof(double));
        if (st) return st;
        double* h = static_cast<double*>(E.hbuf);
        pack_rows(A, R, C, ld, h);
        t.A = reinterpret_cast<const double2*>(h);
        t.out = h + a_bytes / sizeof(double);
        t.done = reinterpret_cast<unsigned*>(t.out + 6);
        *t.done = 0u;
        hipError_t e = launch_tiny(C, t, 1, E.stream);
        if (e == hipSuccess) e = wait_result(E, t.done);
        if (e != hipSuccess) return drain_fail(E, e, "plain sweep");
        out[0] = t.out[0];
        out[1] = t.out[1];
        return PQB_OK;
    }
    const bool expanded = plain_expandable(R, C, 1) && plain_expand_row(A, C, ld) >= 0;
    const int rows = expanded ? R - 1 : R;
    const PlainPlan pl = make_plain_plan(rows, C, E.resident_waves_locked(C, expanded));
    const size_t a_bytes = (size_t)R * C * sizeof(double2), m2_bytes = 2 * a_bytes;
    const size_t part_off = kCounterBytes;
    const size_t part_bytes = (size_t)pl.blocks * sizeof(ddc);
    const size_t m2_off = part_off + round256(part_bytes);
    const size_t a_off = m2_off + round256(m2_bytes);
    // the upload: the +-2A table, or the matrix whose expanded table a kernel builds
    const size_t up_bytes = expanded ? a_bytes : m2_bytes;
    int st = E.ensure_buffers_locked(a_off + a_bytes, up_bytes + 256);
    if (st) return st;
    double* h = static_cast<double*>(E.hbuf);
    if (expanded) pack_rows(A, R, C, ld, h);
    else fill_m2(A, R, C, ld, h);
    double* hout = h + up_bytes / sizeof(double);  // the kernel writes the result here itself
    char* d = static_cast<char*>(E.dbuf);
    unsigned* counter = reinterpret_cast<unsigned*>(d);
    double2* m2 = reinterpret_cast<double2*>(d + m2_off);
    hipError_t e = hipMemcpyAsync(d + (expanded ? a_off : m2_off), h, up_bytes, hipMemcpyHostToDevice, E.stream);
    if (e != hipSuccess) return hip_fail(e, "hipMemcpyAsync");
    if (expanded) e = launch_plain_expand(reinterpret_cast<const double2*>(d + a_off), m2, C, 1, counter, E.stream);
    PlainParams p = plain_params(pl, R, m2, 2 * R * C, reinterpret_cast<ddc*>(d + part_off), counter, hout);
    p.done = reinterpret_cast<unsigned*>(hout + 6);
    *p.done = 0u;
    if (e == hipSuccess) e = launch_plain(C, expanded, p, pl.blocks, pl.block, 1, E.stream);
    if (e == hipSuccess) e = wait_result(E, p.done);
    if (e != hipSuccess) return drain_fail(E, e, "plain sweep");
    out[0] = hout[0];
    out[1] = hout[1];
    return PQB_OK;
}

// Shape rules of the reference calculators.  Returns 1 and fills out when
// the result is decided without a sweep.
static int plain_edge(int algo, int64_t rows, int64_t cols, double* out) {
    if (algo == PQB_ALGO_SIMPLE) {
        // GlynnPermanentCalculatorSimple.hpp:65-70
        if (rows == 0 || cols == 0) { out[0] = 1.0; out[1] = 0.0; return 1; }
        if (rows != cols) {
            std::fprintf(stderr, "Matrix is not rectangular! Returning 0.\n");
            out[0] = 0.0; out[1] = 0.0; return 1;
        }
        return 0;
    }
    // BBFGPermanentCalculator.cpp:92-95, .hpp:90-95; GlynnPermanentCalculator.hpp:50-53
    if (rows == 0 || cols == 0) { out[0] = 1.0; out[1] = 0.0; return 1; }
    if (rows >= cols + 2) { out[0] = 0.0; out[1] = 0.0; return 1; }
    return 0;
}

int plain_entry(const double* A, int64_t rows, int64_t cols, int64_t ld, int algo, int precision,
                double* out, int64_t* words) {
    if (!out) return fail(PQB_ERR_ARG, "output pointer is NULL");
    if (rows < 0 || cols < 0) return fail(PQB_ERR_ARG, "negative matrix dimension");
    if (algo < PQB_ALGO_BBFG || algo > PQB_ALGO_SIMPLE) return fail(PQB_ERR_ARG, "unknown algorithm code");
    if (precision < PQB_PREC_DOUBLE || precision > PQB_PREC_INF)
        return fail(PQB_ERR_ARG, "unknown precision code");
    if (plain_edge(algo, rows, cols, out)) {
        if (words) {
            const i128 v = (i128)out[0];
            words[0] = (int64_t)(unsigned long long)v;
            words[1] = (int64_t)(v >> 64);
        }
        return PQB_OK;
    }
    if (!A) return fail(PQB_ERR_ARG, "matrix pointer is NULL");
    if (ld < cols) return fail(PQB_ERR_ARG, "leading dimension smaller than the number of columns");
    if (cols > PQB_MAX_COLS)
        return fail(PQB_ERR_SIZE, "matrix has more than " + std::to_string(PQB_MAX_COLS) + " columns");
    const int R = (int)rows, C = (int)cols;

    std::vector<int> ai;
    long double lb = 0.0L;
    const bool is_int = precision != PQB_PREC_FP64 && integer_matrix(A, rows, cols, ld, ai, &lb);
    const bool exact_ok = is_int && exact_fits(lb);
    if (precision == PQB_PREC_EXACT && !exact_ok)
        return fail(PQB_ERR_EXACT, is_int ? "exact mode: the permanent may exceed the 128-bit range"
                                          : "exact mode needs a real integer-valued matrix");

    Lease L;
    int st = L.status();
    if (st) return st;
    Engine& E = *L;
    if (exact_ok) {
        i128 v = 0;
        st = run_exact_locked(E, ai, R, C, &v);
        if (st) return st;
        out[0] = i128_to_double(v);
        out[1] = 0.0;
        if (words) {
            words[0] = (int64_t)(unsigned long long)v;
            words[1] = (int64_t)(v >> 64);
        }
        return PQB_OK;
    }
    if (precision == PQB_PREC_INF) return run_plain_dd_locked(E, A, R, C, ld, out);
    return run_plain_locked(E, A, R, C, ld, out);
}

// ------------------------------------------------------------- list entry --
//
// Plain permanents of a list of host matrices (any mix of shapes).  Each
// matrix gets the value pqb_perm gives it (double-double: the same sum, in another
// order before it is rounded); the work is regrouped:
//  * exact-route integer matrices: one exact sweep each (as per call);
//  * double-double route: every matrix planned as a single call would plan it,
//    all of them in one batched launch (in two, where many matrices whose rows
//    are split stand beside others, see kApartWork in batch.hip);
//  * FP64 route: one launch for all the shapes that are small, else one per
//    distinct shape with one grid row (blockIdx.y) per matrix, each matrix
//    with the single-call launch plan -- so every value is bit-identical to
//    its pqb_perm call -- with one upload of all +-2A tables and one
//    synchronisation.

struct ListItem {
    int64_t idx;
    int R, C;
    bool expanded;
};

// Matrices of one tiny shape, and blocks of one larger shape, up to which it shares a launch.
constexpr size_t kMixedTiny = 256, kMixedBlocks = 2048;

static int list_fp64_locked(Engine& E, const double* const* A, const int64_t* ld, std::vector<ListItem>& items,
                            double* out) {
    if (items.empty()) return PQB_OK;
    for (ListItem& it : items)
        it.expanded = plain_expandable(it.R, it.C, 1) && plain_expand_row(A[it.idx], it.C, ld[it.idx]) >= 0;
    std::stable_sort(items.begin(), items.end(), [](const ListItem& a, const ListItem& b) {
        return a.R != b.R ? a.R < b.R : (a.C != b.C ? a.C < b.C : a.expanded < b.expanded);
    });
    struct Group {
        size_t first, count;
        int R, C;
        bool expanded, tiny, mixed;
        PlainPlan pl;
        TinyParams t;
        size_t up_off;            // byte offset in the upload: +-2A tables, or (expanded) the matrices
        size_t part_off, m2_off;  // device byte offsets of the group's partials and tables
    };
    std::vector<Group> groups;
    for (size_t k = 0; k < items.size();) {
        const ListItem& f = items[k];
        size_t e = k;
        while (e < items.size() && items[e].R == f.R && items[e].C == f.C && items[e].expanded == f.expanded) ++e;
        Group g;
        g.first = k;
        g.count = e - k;
        g.R = f.R;
        g.C = f.C;
        g.expanded = f.expanded;
        g.tiny = plain_tiny(f.R, f.C, 1, g.t);
        if (!g.tiny)
            g.pl = make_plain_plan(f.expanded ? f.R - 1 : f.R, f.C, E.resident_waves_locked(f.C, f.expanded));
        // shapes of one launch: those whose matrices are few, as the others fill the chip by
        // themselves, at their own size of block and registers
        g.mixed = g.tiny ? g.count <= kMixedTiny
                         : !g.expanded && g.C >= kMixedMinCols && g.C <= kMixedMaxCols && g.pl.block == kBlock &&
                               g.count * (size_t)g.pl.blocks <= kMixedBlocks;
        groups.push_back(g);
        k = e;
    }
    const size_t n = items.size();
    size_t off = kCounterBytes;  // offset 0 stays the single-call counter
    for (Group& g : groups) {
        g.part_off = off;
        if (!g.tiny) off += round256(g.count * (size_t)g.pl.blocks * sizeof(ddc));
    }
    // the upload holds the counters, zero, the +-2A tables of the all-rows groups, used in place, and the
    // matrices of the expanded ones, whose tables a kernel builds behind it; the matrices of
    // the tiny groups stay in the staging buffer, past the upload
    const size_t up_base = off;
    const size_t cnt_off = up_base, no_tables = round256(n * sizeof(unsigned));
    size_t up_total = 0, staged = no_tables;
    for (int tiny = 0; tiny < 2; ++tiny) {
        for (Group& g : groups)
            if (g.tiny == (tiny != 0)) {
                g.up_off = staged;
                g.m2_off = up_base + staged;
                staged += round256(g.count * (size_t)g.R * g.C * sizeof(double2) * (g.expanded || g.tiny ? 1 : 2));
            }
        if (!tiny) up_total = staged;
    }
    off += up_total;
    for (Group& g : groups)
        if (g.expanded) {
            g.m2_off = off;
            off += round256(g.count * (size_t)2 * g.R * g.C * sizeof(double2));
        }
    int st = E.ensure_buffers_locked(off, staged + n * 6 * sizeof(double));
    if (st) return st;
    double* h = static_cast<double*>(E.hbuf);
    for (const Group& g : groups) {
        const size_t rc = (size_t)g.R * g.C;
        double* hg = h + g.up_off / sizeof(double);
        for (size_t k = 0; k < g.count; ++k) {
            const int64_t i = items[g.first + k].idx;
            if (g.expanded || g.tiny) pack_rows(A[i], g.R, g.C, ld[i], hg + 2 * rc * k);
            else fill_m2(A[i], g.R, g.C, ld[i], hg + 4 * rc * k);
        }
    }
    char* d = static_cast<char*>(E.dbuf);
    unsigned* counters = reinterpret_cast<unsigned*>(d + cnt_off);
    double* const hout = h + staged / sizeof(double);  // the kernels write the results here themselves
    hipError_t e = hipSuccess;
    std::memset(h, 0, n * sizeof(unsigned));
    auto params_of = [&](const Group& g, size_t o) {
        const int64_t m2n = (int64_t)2 * g.R * g.C;
        return plain_params(g.pl, g.R, reinterpret_cast<double2*>(d + g.m2_off) + o * (size_t)m2n, m2n,
                            reinterpret_cast<ddc*>(d + g.part_off) + o * (size_t)g.pl.blocks,
                            counters + g.first + o, hout + 6 * (g.first + o));
    };
    if (up_total > no_tables) e = hipMemcpyAsync(d + up_base, h, up_total, hipMemcpyHostToDevice, E.stream);
    if (e != hipSuccess) return drain_fail(E, e, "list upload");
    constexpr size_t kMaxGridY = 65535;
    TinyMixed tiny;
    PlainMixed small;
    tiny.shapes = small.shapes = 0;
    tiny.first[0] = small.first[0] = 0;
    auto flush_tiny = [&]() {
        const hipError_t le = tiny.shapes > 0 ? launch_tiny_mixed(tiny, E.stream) : hipSuccess;
        tiny.shapes = 0;
        return le;
    };
    auto flush_small = [&]() {
        const hipError_t le = small.shapes > 0 ? launch_plain_mixed(small, E.stream) : hipSuccess;
        small.shapes = 0;
        return le;
    };
    for (Group& g : groups) {
        if (g.tiny) {
            g.t.A = reinterpret_cast<const double2*>(h + g.up_off / sizeof(double));
            g.t.out = hout + 6 * g.first;
            if (g.mixed) {
                const int k = tiny.shapes++;
                tiny.p[k] = g.t;
                tiny.ns[k] = (unsigned char)g.C;
                tiny.first[k + 1] = tiny.first[k] + (unsigned)g.count;
                if (tiny.shapes == kTinyShapes) e = flush_tiny();
            } else {
                e = launch_tiny(g.C, g.t, (int64_t)g.count, E.stream);
            }
        } else if (g.mixed) {
            const int k = small.shapes++;
            small.p[k] = params_of(g, 0);
            small.nc[k] = g.C;
            small.blocks[k] = (unsigned)g.pl.blocks;
            small.first[k + 1] = small.first[k] + (unsigned)(g.count * (size_t)g.pl.blocks);
            if (small.shapes == kMixedShapes) e = flush_small();
        } else {
            if (g.expanded)
                e = launch_plain_expand(reinterpret_cast<const double2*>(d + up_base + g.up_off),
                                        reinterpret_cast<double2*>(d + g.m2_off), g.C, (int64_t)g.count,
                                        counters + g.first, E.stream);
            for (size_t o = 0; e == hipSuccess && o < g.count; o += kMaxGridY) {
                const size_t nt = std::min(kMaxGridY, g.count - o);
                e = launch_plain(g.C, g.expanded, params_of(g, o), g.pl.blocks, g.pl.block, (int)nt, E.stream);
            }
        }
        if (e != hipSuccess) return drain_fail(E, e, "list sweep launch");
    }
    e = flush_tiny();
    if (e == hipSuccess) e = flush_small();
    if (e != hipSuccess) return drain_fail(E, e, "list sweep launch");
    e = hipStreamSynchronize(E.stream);
    if (e != hipSuccess) return drain_fail(E, e, "list sweep");
    for (size_t k = 0; k < n; ++k) {
        out[2 * items[k].idx] = hout[6 * k];
        out[2 * items[k].idx + 1] = hout[6 * k + 1];
    }
    return PQB_OK;
}

int list_entry(const double* const* A, const int64_t* rows, const int64_t* cols, const int64_t* ld,
               int64_t count, int algo, int precision, double* out) {
    if (count < 0) return fail(PQB_ERR_ARG, "negative matrix count");
    if (count == 0) return PQB_OK;
    if (!A || !rows || !cols || !ld || !out) return fail(PQB_ERR_ARG, "NULL pointer");
    if (algo < PQB_ALGO_BBFG || algo > PQB_ALGO_SIMPLE) return fail(PQB_ERR_ARG, "unknown algorithm code");
    if (precision < PQB_PREC_DOUBLE || precision > PQB_PREC_INF)
        return fail(PQB_ERR_ARG, "unknown precision code");
    auto bad = [&](int64_t i, int code, const std::string& msg) {
        return fail(code, "matrix " + std::to_string(i) + ": " + msg);
    };
    std::vector<ListItem> fp64, inf;
    std::vector<std::pair<int64_t, std::vector<int>>> exact;
    for (int64_t i = 0; i < count; ++i) {
        if (rows[i] < 0 || cols[i] < 0) return bad(i, PQB_ERR_ARG, "negative matrix dimension");
        if (plain_edge(algo, rows[i], cols[i], out + 2 * i)) continue;
        if (!A[i]) return bad(i, PQB_ERR_ARG, "matrix pointer is NULL");
        if (ld[i] < cols[i]) return bad(i, PQB_ERR_ARG, "leading dimension smaller than the number of columns");
        if (cols[i] > PQB_MAX_COLS)
            return bad(i, PQB_ERR_SIZE, "matrix has more than " + std::to_string(PQB_MAX_COLS) + " columns");
        std::vector<int> ai;
        long double lb = 0.0L;
        const bool is_int = precision != PQB_PREC_FP64 && integer_matrix(A[i], rows[i], cols[i], ld[i], ai, &lb);
        const bool exact_ok = is_int && exact_fits(lb);
        if (precision == PQB_PREC_EXACT && !exact_ok)
            return bad(i, PQB_ERR_EXACT, is_int ? "exact mode: the permanent may exceed the 128-bit range"
                                                : "exact mode needs a real integer-valued matrix");
        const ListItem it{i, (int)rows[i], (int)cols[i], false};
        if (exact_ok)
            exact.emplace_back(i, std::move(ai));
        else if (precision == PQB_PREC_INF)
            inf.push_back(it);
        else
            fp64.push_back(it);
    }
    if (exact.empty() && inf.empty() && fp64.empty()) return PQB_OK;
    Lease L;
    int st = L.status();
    if (st) return st;
    Engine& E = *L;
    for (auto& ex : exact) {
        i128 v = 0;
        st = run_exact_locked(E, ex.second, (int)rows[ex.first], (int)cols[ex.first], &v);
        if (st) return bad(ex.first, st, t_err);
        out[2 * ex.first] = i128_to_double(v);
        out[2 * ex.first + 1] = 0.0;
    }
    if (!inf.empty()) {
        std::vector<const double*> pa;
        std::vector<int> pr, pc;
        std::vector<int64_t> pl;
        for (const ListItem& it : inf) {
            pa.push_back(A[it.idx]);
            pr.push_back(it.R);
            pc.push_back(it.C);
            pl.push_back(ld[it.idx]);
        }
        std::vector<double> o(2 * inf.size());
        st = run_plain_dd_list_locked(E, pa.data(), pr.data(), pc.data(), pl.data(), (int64_t)inf.size(),
                                      o.data());
        if (st) return st;
        for (size_t k = 0; k < inf.size(); ++k) {
            out[2 * inf[k].idx] = o[2 * k];
            out[2 * inf[k].idx + 1] = o[2 * k + 1];
        }
    }
    return list_fp64_locked(E, A, ld, fp64, out);
}

// ----------------------------------------------------- device-pointer API --
//
// Workspace of the device entry points: one counter per matrix (rounded up
// to 256 bytes), then `blocks_per_matrix` dd partials per matrix, then the
// +-2A tables of all matrices.  For one matrix the layout is the documented
// pqb_perm_device one (counter slot of 256 bytes, kMaxBlocks partials).

size_t plain_device_bytes(int64_t count, int64_t rows, int64_t cols, int64_t blocks_per_matrix) {
    return round256((size_t)count * sizeof(unsigned)) + (size_t)count * blocks_per_matrix * sizeof(ddc) +
           (size_t)count * 2 * rows * cols * sizeof(double2);
}

int plain_device_check(int64_t count, int64_t rows, int64_t cols) {
    if (count < 1) return fail(PQB_ERR_ARG, "batch count must be positive");
    if (rows < 1 || cols < 1 || rows >= cols + 2)
        return fail(PQB_ERR_ARG, "the device entry points need 1 <= rows <= cols + 1");
    if (cols > PQB_MAX_COLS)
        return fail(PQB_ERR_SIZE, "matrix has more than " + std::to_string(PQB_MAX_COLS) + " columns");
    return PQB_OK;
}

// Launch plans of a batch of `count` equal-size matrices: the single-matrix plan for
// the resident waves divided among the matrices, of the sweep over all rows and (where
// the matrices may be expanded) of the expanded one.  Each matrix takes one of the two
// and the partials have room for either.
static int plain_device_plan(int64_t count, int R, int C, PlainPlan* pl, PlainPlan* xp,
                             int64_t* blocks_per_matrix) {
    const int st = bind_device(-1, nullptr, nullptr);
    if (st) return st;
    *pl = make_plain_plan(R, C, std::max<int64_t>(1, resident_waves(C, false) / count));
    *blocks_per_matrix = pl->blocks;
    if (plain_expandable(R, C, count)) {
        *xp = make_plain_plan(R - 1, C, std::max<int64_t>(1, resident_waves(C, true) / count));
        *blocks_per_matrix = std::max(pl->blocks, xp->blocks);
    }
    if (*blocks_per_matrix > kMaxBlocks) return fail(PQB_ERR_SIZE, "launch plan exceeds the workspace layout");
    return PQB_OK;
}

// The launches of `count` packed R x C device matrices: tables, then the sweep over all
// rows, then (plan xp given) the expanded one; counters zero before, zero after.
int plain_device_launch(const double2* dA, int64_t count, int R, int C, const PlainPlan& pl, const PlainPlan* xp,
                        double2* m2, ddc* partials, unsigned* counters, double* d_out, hipStream_t st) {
    TinyParams t;
    if (plain_tiny(R, C, count, t)) {
        t.A = dA;
        t.out = d_out;
        const hipError_t e = launch_tiny(C, t, count, st);
        return e == hipSuccess ? PQB_OK : hip_fail(e, "plain sweep launch");
    }
    const int64_t m2n = (int64_t)2 * R * C;
    hipError_t e = xp ? launch_plain_expand(dA, m2, C, count, counters, st)
                      : launch_plain_prep(dA, m2, R * C, count, st);
    if (e != hipSuccess) return hip_fail(e, "prep launch");
    constexpr int64_t kMaxGridY = 65535;
    for (const PlainPlan* q : {&pl, xp}) {
        if (!q) continue;
        for (int64_t off = 0; off < count; off += kMaxGridY) {
            const int64_t nt = std::min(kMaxGridY, count - off);
            PlainParams p = plain_params(*q, R, m2 + off * m2n, m2n, partials + off * q->blocks, counters + off,
                                         d_out + 6 * off);
            p.by_flag = xp ? 1 : 0;
            e = launch_plain(C, q == xp, p, q->blocks, q->block, (int)nt, st);
            if (e != hipSuccess) return hip_fail(e, "plain sweep launch");
        }
    }
    return PQB_OK;
}

int plain_device_run(const double* dA, int64_t count, int64_t rows, int64_t cols, double* d_out, void* d_work,
                     size_t work_bytes, hipStream_t st, bool single) {
    if (!dA || !d_out || !d_work) return fail(PQB_ERR_ARG, "NULL device pointer");
    int s = plain_device_check(count, rows, cols);
    if (s) return s;
    const int R = (int)rows, C = (int)cols;
    PlainPlan pl, xp;
    int64_t bpm = 0;
    s = plain_device_plan(count, R, C, &pl, &xp, &bpm);
    if (s) return s;
    if (single) bpm = kMaxBlocks;  // the documented single-matrix layout
    if (work_bytes < plain_device_bytes(count, rows, cols, bpm)) return fail(PQB_ERR_ARG, "workspace too small");
    char* w = static_cast<char*>(d_work);
    unsigned* counters = reinterpret_cast<unsigned*>(w);
    ddc* partials = reinterpret_cast<ddc*>(w + round256((size_t)count * sizeof(unsigned)));
    double2* m2 = reinterpret_cast<double2*>(reinterpret_cast<char*>(partials) + (size_t)count * bpm * sizeof(ddc));
    return plain_device_launch(reinterpret_cast<const double2*>(dA), count, R, C, pl,
                               plain_expandable(R, C, count) ? &xp : nullptr, m2, partials, counters, d_out, st);
}

// Repeated-row permanent: a batch of one task (batch.hip applies the
// reference's validation and edge rules).
int repeated_entry(const double* A, int64_t rows, int64_t cols, int64_t ld, const int64_t* row_mult,
                   const int64_t* col_mult, int algo, int precision, double* out) {
    if (!out) return fail(PQB_ERR_ARG, "output pointer is NULL");
    if (precision == PQB_PREC_EXACT) return fail(PQB_ERR_ARG, "exact mode is available for the plain permanent only");
    const pqb_task t{A, rows, cols, ld, row_mult, col_mult};
    return batch_entry(&t, 1, algo, precision, out, 0);
}

}  // namespace pqb

using namespace pqb;

extern "C" {

const char* pqb_last_error(void) { return t_err.c_str(); }

int pqb_abi_version(void) { return 1; }

int pqb_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int pqb_init(int device) { return bind_device(device, nullptr, nullptr); }

int pqb_perm(const double* A, int64_t rows, int64_t cols, int64_t ld, int algo, int precision,
             double* out) {
    try {
        return plain_entry(A, rows, cols, ld, algo, precision, out, nullptr);
    } catch (const std::exception& ex) {
        return fail(PQB_ERR_DEVICE, std::string("internal error: ") + ex.what());
    }
}

int pqb_perm_list(const double* const* A, const int64_t* rows, const int64_t* cols, const int64_t* ld,
                  int64_t count, int algo, int precision, double* out) {
    try {
        return list_entry(A, rows, cols, ld, count, algo, precision, out);
    } catch (const std::exception& ex) {
        return fail(PQB_ERR_DEVICE, std::string("internal error: ") + ex.what());
    }
}

int pqb_perm_exact(const double* A, int64_t rows, int64_t cols, int64_t ld, int64_t* words,
                   double* out) {
    if (!words) return fail(PQB_ERR_ARG, "words pointer is NULL");
    try {
        return plain_entry(A, rows, cols, ld, PQB_ALGO_BBFG, PQB_PREC_EXACT, out, words);
    } catch (const std::exception& ex) {
        return fail(PQB_ERR_DEVICE, std::string("internal error: ") + ex.what());
    }
}

int pqb_perm_repeated(const double* A, int64_t rows, int64_t cols, int64_t ld, const int64_t* row_mult,
                      const int64_t* col_mult, int algo, int precision, double* out) {
    try {
        return repeated_entry(A, rows, cols, ld, row_mult, col_mult, algo, precision, out);
    } catch (const std::exception& ex) {
        return fail(PQB_ERR_DEVICE, std::string("internal error: ") + ex.what());
    }
}

int pqb_exact_bound(const double* A, int64_t rows, int64_t cols, int64_t ld, double* log2_bound) {
    if (!A || !log2_bound || rows < 1 || cols < 1 || ld < cols) return fail(PQB_ERR_ARG, "bad arguments");
    std::vector<int> ai;
    long double lb = 0.0L;
    if (!integer_matrix(A, rows, cols, ld, ai, &lb))
        return fail(PQB_ERR_EXACT, "exact mode needs a real integer-valued matrix");
    *log2_bound = (double)lb;
    return exact_fits(lb) ? PQB_OK : fail(PQB_ERR_EXACT, "exact mode: the permanent may exceed the 128-bit range");
}

size_t pqb_perm_device_workspace(int64_t rows, int64_t cols) {
    if (rows < 1 || cols < 1) return kCounterBytes;
    return plain_device_bytes(1, rows, cols, kMaxBlocks);
}

int pqb_perm_device(const double* dA, int64_t rows, int64_t cols, double* d_out, void* d_work,
                    size_t work_bytes, void* stream) {
    return plain_device_run(dA, 1, rows, cols, d_out, d_work, work_bytes, static_cast<hipStream_t>(stream), true);
}

int pqb_perm_batch_device_workspace(int64_t count, int64_t rows, int64_t cols, size_t* bytes) {
    if (!bytes) return fail(PQB_ERR_ARG, "bytes pointer is NULL");
    int st = plain_device_check(count, rows, cols);
    if (st) return st;
    int64_t bpt = 0;
    PlainPlan pl, xp;
    st = plain_device_plan(count, (int)rows, (int)cols, &pl, &xp, &bpt);
    if (st) return st;
    *bytes = plain_device_bytes(count, rows, cols, bpt);
    return PQB_OK;
}

int pqb_perm_batch_device(const double* dA, int64_t count, int64_t rows, int64_t cols, double* d_out,
                          void* d_work, size_t work_bytes, void* stream) {
    return plain_device_run(dA, count, rows, cols, d_out, d_work, work_bytes, static_cast<hipStream_t>(stream),
                            false);
}

int pqb_plain_plan(int64_t rows, int64_t cols, int64_t waves_resident, int64_t* plan) {
    if (!plan) return fail(PQB_ERR_ARG, "plan pointer is NULL");
    if (rows < 1 || cols < 1 || rows >= cols + 2 || cols > PQB_MAX_COLS)
        return fail(PQB_ERR_ARG, "no sweep for this shape");
    int64_t wr = waves_resident;
    if (wr <= 0) {
        const int st = bind_device(-1, nullptr, nullptr);
        if (st) return st;
        wr = resident_waves((int)cols, false);
    }
    const PlainPlan pl = make_plain_plan((int)rows, (int)cols, wr);
    plan[0] = pl.K;
    plan[1] = pl.B;
    plan[2] = pl.H;
    plan[3] = pl.waves;
    plan[4] = pl.block;
    plan[5] = pl.blocks;
    return PQB_OK;
}

int pqb_time_perm_device(const double* dA, int64_t rows, int64_t cols, double* d_out, int iters,
                         double* ms) {
    if (!ms || iters < 1) return fail(PQB_ERR_ARG, "bad timing arguments");
    const size_t wb = pqb_perm_device_workspace(rows, cols);
    void* w = nullptr;
    Lease L;  // the timed launches run on this context's stream, held for the call
    if (L.status()) return L.status();
    hipStream_t st = L->stream;
    hipError_t e = hipMalloc(&w, wb);
    if (e != hipSuccess) return hip_fail(e, "hipMalloc(timing workspace)");
    e = hipMemsetAsync(w, 0, kCounterBytes, st);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (e == hipSuccess) e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    int rc = PQB_OK;
    if (e == hipSuccess) e = hipEventRecord(e0, st);
    for (int i = 0; e == hipSuccess && rc == PQB_OK && i < iters; ++i)
        rc = pqb_perm_device(dA, rows, cols, d_out, w, wb, st);
    if (e == hipSuccess && rc == PQB_OK) e = hipEventRecord(e1, st);
    if (e == hipSuccess && rc == PQB_OK) e = hipEventSynchronize(e1);
    float f = 0.f;
    if (e == hipSuccess && rc == PQB_OK) e = hipEventElapsedTime(&f, e0, e1);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipStreamSynchronize(st);
    (void)hipFree(w);
    if (rc != PQB_OK) return rc;
    if (e != hipSuccess) return hip_fail(e, "timing");
    *ms = f;
    return PQB_OK;
}

}  // extern "C"
