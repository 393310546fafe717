// Host side of the repeated-row and batched sweeps: task planning, step
// tables, work items and the graph-captured persistent launch.
//
// Planning a task (one repeated-row permanent), following
// BBFGPermanentCalculatorRepeated.hpp:74-101 and :116-307:
//   * rows / columns with zero multiplicity are dropped (they contribute a
//     factor 1, BatchedPermanentCalculator.cpp:412-451 builds the same compact
//     matrix);
//   * perm(A) = perm(A^T), so the orientation with fewer Gray steps
//     S = m_min prod_{i != min} (m_i + 1) is used (the DFE host code makes the
//     same choice, GlynnPermanentCalculatorRepeatedDFE.cpp:1138);
//   * the row with the smallest multiplicity (first occurrence) becomes the
//     anchor with multiplicity 1 and the rest of its multiplicity stays a digit
//     (BBFGPermanentCalculatorRepeated.hpp:78-94);
//   * columns of multiplicity c occupy c slots;
//   * digits are split into low digits (walked in a chunk, radix product L close
//     to the requested chunk length) and high digits (chunk index).
// The low walk is a reflected mixed-radix Gray code starting at k = 0: each
// digit sweeps up then down while the faster digits complete full sweeps, so
// every step moves exactly one digit by one; tables are shared by all tasks
// whose low radices agree.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <numeric>
#include <string>
#include <system_error>
#include <thread>
#include <unordered_map>
#include <vector>

#include "pqb_perm.h"
#include "pqb_device.h"
#include "pqb_engine.h"
#include "pqb_kernels.h"
#include "pqb_pivot.h"

namespace pqb {

// ----------------------------------------------------------------- planning --

static uint64_t binom_u64(int n, int k) {
    if (k < 0 || k > n) return 0;
    uint64_t c = 1;
    for (int i = 1; i <= k; ++i) c = c * (uint64_t)(n - k + i) / (uint64_t)i;  // exact at every step
    return c;
}

// Gray steps of the repeated sweep for multiplicities v (nonzero entries; at most 2^40,
// exact in a double).
static double sweep_steps(const std::vector<int64_t>& v) {
    if (v.empty()) return 0.0;
    size_t mi = 0;
    for (size_t i = 1; i < v.size(); ++i)
        if (v[i] < v[mi]) mi = i;
    double s = (double)v[mi];
    for (size_t i = 0; i < v.size(); ++i)
        if (i != mi) s *= (double)(v[i] + 1);
    return s;
}

namespace {
struct Digit {
    int64_t src;  // oriented row
    int m;        // multiplicity walked by this digit
};
// Temporaries of plan_task, kept per thread and reused: a batch plans thousands
// of tasks on host threads, and fresh vectors per task made the allocator the
// bottleneck.
struct PlanScratch {
    std::vector<int64_t> ri, rm, ci, cm;
    std::vector<Digit> digits, low, high;
    std::vector<size_t> ord;
};
}  // namespace

// Occupied rows and columns and their multiplicities into the thread's scratch.
static void compact_occupations(int64_t rows, int64_t cols, const int64_t* rmult, const int64_t* cmult,
                                PlanScratch& sc, int64_t* N, int64_t* Nc) {
    sc.ri.clear();
    sc.rm.clear();
    sc.ci.clear();
    sc.cm.clear();
    *N = *Nc = 0;
    for (int64_t i = 0; i < rows; ++i)
        if (rmult[i] > 0) {
            sc.ri.push_back(i);
            sc.rm.push_back(rmult[i]);
            *N += rmult[i];
        }
    for (int64_t j = 0; j < cols; ++j)
        if (cmult[j] > 0) {
            sc.ci.push_back(j);
            sc.cm.push_back(cmult[j]);
            *Nc += cmult[j];
        }
}

static PlanScratch& plan_scratch() {
    thread_local PlanScratch sc;
    return sc;
}

// FP64 instructions of one Gray step (add_wterm, add_wcoeff in perm_repeated.hip).
static double step_cost(int degree, int ns) {
    if (degree == 0) return 6.0 * ns - 1.0;
    // 2 per column sum and for the weight; 4 per coefficient and column, without the
    // coefficients that are still zero or one, or can no longer reach x^D
    const int d = degree;
    return 2.0 * ns + 2.0 + 4.0 * (d + 1) * (ns - 1) - 2.0 * d * d - 2.0 * d * (d + 1);
}

// Sweeps below this many steps keep all rows: they take microseconds either way, and the
// expanded ones need the launch that divides their columns.
constexpr double kExpandMinSteps = 4096.0;

// The sweep of a repeated-row task (A: the rows x cols matrix, its occupied rows and
// columns in `sc`).  Without expansion: the orientation with fewer Gray steps.  A row of
// multiplicity D can be expanded instead of walked: with every column divided by its entry
// of that row, the row's D copies contribute the coefficient of x^D in the product of the
// (column sums + x), so its radix D + 1 leaves the walk for a term of about 4 (D + 1) + 2
// instead of 6 FP64 instructions per column -- of the D + 1 steps it replaces, 0.80, 0.72,
// 0.67 of the instructions at D = 1, 2, 3 and 26 columns, 0.78, 0.68, 0.61 at 16.  The
// cheapest orientation and multiplicity whose entries allow it is taken; the conditions
// are those of the plain sweep (pqb_pivot.h).
static SweepChoice choose_sweep(const double* A, int64_t ld, const PlanScratch& sc, bool expand) {
    SweepChoice c;
    const double sr = sweep_steps(sc.rm), st = sweep_steps(sc.cm);
    c.transpose = st < sr;
    c.steps = std::min(sr, st);
    const int NS = (int)std::accumulate(sc.rm.begin(), sc.rm.end(), (int64_t)0);
    if (!expand || c.steps < kExpandMinSteps || NS < kExpandedMinSlots) return c;

    struct Candidate {
        double cost, steps;
        bool transpose;
        int degree;
    };
    Candidate cand[2 * kMaxDegree];
    int nc = 0;
    const double kept = c.steps * step_cost(0, NS);
    for (int t = 0; t < 2; ++t) {
        const std::vector<int64_t>& m = t ? sc.cm : sc.rm;
        if (m.size() < 2) continue;
        for (int d = 1; d <= kMaxDegree; ++d) {
            const auto at = std::find(m.begin(), m.end(), (int64_t)d);
            if (at == m.end()) continue;
            // steps of the other rows: their smallest is the anchor
            int64_t lo = -1;
            double s = 1.0;
            for (auto k = m.begin(); k != m.end(); ++k)
                if (k != at) {
                    lo = lo < 0 ? *k : std::min(lo, *k);
                    s *= (double)(*k + 1);
                }
            s = s / (double)(lo + 1) * (double)lo;
            const double cost = s * step_cost(d, NS);
            if (cost < kept) cand[nc++] = Candidate{cost, s, t != 0, d};
        }
    }
    if (nc == 0) return c;
    std::sort(cand, cand + nc, [](const Candidate& a, const Candidate& b) { return a.cost < b.cost; });

    const size_t R = sc.ri.size(), C = sc.ci.size();
    double row_min[kMaxSlots], col_min[kMaxSlots], hi = 0.0;
    std::fill(row_min, row_min + R, HUGE_VAL);
    std::fill(col_min, col_min + C, HUGE_VAL);
    int low = lowest_bit(0.0);
    for (size_t r = 0; r < R; ++r)
        for (size_t k = 0; k < C; ++k) {
            const double* a = A + 2 * (sc.ri[r] * ld + sc.ci[k]);
            if (!pivot_admits(a[0], a[1])) return c;
            const double v = std::max(std::fabs(a[0]), std::fabs(a[1]));
            row_min[r] = std::min(row_min[r], v);
            col_min[k] = std::min(col_min[k], v);
            hi = std::max(hi, v);
            if (!off_grid(low, hi)) low = std::min(low, lowest_bit(a[0], a[1]));  // off it, it stays off
        }
    if (!off_grid(low, hi)) return c;
    const double least = pivot_least(hi);
    for (int q = 0; q < nc; ++q) {
        const std::vector<int64_t>& m = cand[q].transpose ? sc.cm : sc.rm;
        const double* mins = cand[q].transpose ? col_min : row_min;
        int best = -1;
        for (size_t k = 0; k < m.size(); ++k)
            if (m[k] == cand[q].degree && mins[k] >= least && (best < 0 || mins[k] > mins[best])) best = (int)k;
        if (best < 0) continue;
        c.transpose = cand[q].transpose;
        c.degree = cand[q].degree;
        c.row = (cand[q].transpose ? sc.ci : sc.ri)[(size_t)best];
        c.steps = cand[q].steps;
        return c;
    }
    return c;
}

// Whether the double-double sweep may take the rows of a task (its occupied rows and columns
// in `sc`) in two parts (RepTask::split), and E with entries below 2^E.  A column sum of at
// most 40 rows is then below 2^(E+6), so parts on the grid of 2^(E-47) add up exactly in a
// double; those below it add up to less than 2^(E-42), and are multiples of 2^(E-92) when no
// entry but zeros is below 2^(E-40), so they do too.
static bool split_exact(const double* A, int64_t ld, const PlanScratch& sc, int* E) {
    double most = 0.0, least = HUGE_VAL;
    for (int64_t r : sc.ri)
        for (int64_t k : sc.ci)
            for (int c = 0; c < 2; ++c) {
                const double v = std::fabs(A[2 * (r * ld + k) + c]);
                if (!(v <= 0x1p900)) return false;
                most = std::max(most, v);
                if (v > 0.0) least = std::min(least, v);
            }
    if (!(most >= 0x1p-900)) return false;
    *E = std::ilogb(most) + 1;
    return least >= std::ldexp(1.0, *E - 40);
}

// choice: the sweep (NULL: without expansion).
int plan_task(const double* A, int64_t rows, int64_t cols, int64_t ld, const int64_t* rmult,
              const int64_t* cmult, uint64_t target_L, TaskPlan& P, const SweepChoice* choice, bool plain) {
    P = TaskPlan();
    PlanScratch& sc = plan_scratch();
    const std::vector<int64_t>&ri = sc.ri, &rm = sc.rm, &ci = sc.ci, &cm = sc.cm;
    int64_t N = 0, Nc = 0;
    compact_occupations(rows, cols, rmult, cmult, sc, &N, &Nc);
    // plain: a rows x cols matrix with every multiplicity 1 and rows <= cols + 1
    // (the BBFG sum of BBFGPermanentCalculator.hpp:87-235, which is not
    // transpose invariant when rows != cols)
    if (!plain && N != Nc) return fail(PQB_ERR_STATE, "Number of input and output states should be equal");
    if (N == 0) {
        P.trivial = true;
        return PQB_OK;
    }
    if (Nc > kMaxSlots || (!plain && N > kMaxSlots))
        return fail(PQB_ERR_SIZE, "more than " + std::to_string(kMaxSlots) + " photons");
    SweepChoice own;
    if (!choice) {
        if (!plain) own = choose_sweep(A, ld, sc, false);
        choice = &own;
    }
    const bool transpose = choice->transpose;
    P.src = A;
    P.ld = ld;
    P.transpose = transpose;
    const std::vector<int64_t>& row_m = transpose ? cm : rm;
    const std::vector<int64_t>& col_m = transpose ? rm : cm;
    const std::vector<int64_t>& row_i = transpose ? ci : ri;
    const std::vector<int64_t>& col_i = transpose ? ri : ci;

    // column slots
    int NS = 0;
    for (size_t c = 0; c < col_m.size(); ++c)
        for (int64_t k = 0; k < col_m[c]; ++k) P.slot[NS++] = (uint32_t)col_i[c];

    // the expanded row, and the anchor: of the others the smallest multiplicity, first occurrence
    size_t expanded = row_m.size();
    if (choice->degree > 0)
        for (size_t r = 0; r < row_m.size(); ++r)
            if (row_i[r] == choice->row) expanded = r;
    size_t anchor = expanded == 0 ? 1 : 0;
    for (size_t r = anchor + 1; r < row_m.size(); ++r)
        if (r != expanded && row_m[r] < row_m[anchor]) anchor = r;
    std::vector<Digit>& digits = sc.digits;
    digits.clear();
    for (size_t r = 0; r < row_m.size(); ++r) {
        if (r == expanded) continue;
        const int64_t m = (r == anchor) ? row_m[r] - 1 : row_m[r];
        if (m > 0) digits.push_back({(int64_t)r, (int)m});
    }
    P.degree = choice->degree;
    P.scale = std::ldexp(1.0, -(int)(N - 1));
    if (P.degree > 0) {  // the columns' scales follow on the GPU (rep_layout_kernel)
        P.scale = std::ldexp(1.0, -(int)(N - P.degree - 1));
        for (int d = 2; d <= P.degree; ++d) P.scale *= d;
        P.xrow = (uint32_t)row_i[expanded];
    }
    // low / high split: largest radices first into the walk while it fits
    std::vector<size_t>& ord = sc.ord;
    ord.resize(digits.size());
    std::iota(ord.begin(), ord.end(), 0);
    // stable, largest first (insertion sort: a few dozen digits, no buffer to allocate)
    for (size_t i = 1; i < ord.size(); ++i) {
        const size_t v = ord[i];
        size_t j = i;
        for (; j > 0 && digits[ord[j - 1]].m < digits[v].m; --j) ord[j] = ord[j - 1];
        ord[j] = v;
    }
    uint64_t L = 1;
    for (;;) {
        std::vector<Digit>& low = sc.low;
        std::vector<Digit>& high = sc.high;
        low.clear();
        high.clear();
        L = 1;
        for (size_t k : ord) {
            const uint64_t rad = (uint64_t)digits[k].m + 1;
            if (L * rad <= target_L) {
                low.push_back(digits[k]);
                L *= rad;
            } else {
                high.push_back(digits[k]);
            }
        }
        double nch = 1.0;
        for (const Digit& d : high) nch *= (double)(d.m + 1);
        if (nch < 4.0e9) {
            P.nchunks = (uint64_t)nch;
            // rows: anchor, low digits in walk order, high digits
            P.R = 0;
            P.row[P.R++] = (uint32_t)row_i[anchor];
            for (const Digit& d : low) P.row[P.R++] = (uint32_t)row_i[(size_t)d.src];
            for (const Digit& d : high) P.row[P.R++] = (uint32_t)row_i[(size_t)d.src];
            P.NS = NS;
            P.N = (int)N;
            P.nlow = (int)low.size();
            P.nhigh = (int)high.size();
            P.L = L;
            for (size_t d = 0; d < low.size(); ++d) P.low_radix[d] = (unsigned char)(low[d].m + 1);
            for (size_t d = 0; d < high.size(); ++d) P.high_radix[d] = (unsigned char)(high[d].m + 1);
            return PQB_OK;
        }
        target_L *= 4;  // too many chunks for 32-bit chunk indices: walk more per chunk
    }
}

// A plan's rows (R x NS), base (NS) and expanded row (NS) from its matrix.
static void fill_rows(const TaskPlan& P, double* A) {
    for (int r = 0; r < P.R; ++r)
        for (int s = 0; s < P.NS; ++s, A += 2) {
            const double* a = P.entry(r, s);
            A[0] = a[0];
            A[1] = a[1];
        }
}

static void fill_base(const TaskPlan& P, double* base) {
    for (int s = 0; s < P.NS; ++s) {
        // anchor + sum_low m a: in the order of the reference seed
        // (BBFGPermanentCalculatorRepeated.hpp:202-226)
        double br = P.entry(0, s)[0], bi = P.entry(0, s)[1];
        for (int d = 0; d < P.nlow; ++d) {
            const double m = (double)(P.low_radix[d] - 1);
            br += P.entry(1 + d, s)[0] * m;
            bi += P.entry(1 + d, s)[1] * m;
        }
        base[2 * s] = br;
        base[2 * s + 1] = bi;
    }
}

static void fill_xrow(const TaskPlan& P, double* x) {
    for (int s = 0; s < P.NS; ++s, x += 2) {
        const double* a =
            P.src + 2 * (P.transpose ? (int64_t)P.slot[s] * P.ld + P.xrow : (int64_t)P.xrow * P.ld + P.slot[s]);
        x[0] = a[0];
        x[1] = a[1];
    }
}

// The parts of the rows and of the base.  A chunk's `group` lanes have `own` slots each, lane
// q from q * own on; a row holds the lanes' k-th slots side by side, (re_hi, re_lo) of each,
// then (im_hi, im_lo), so that a load of the wave is one line.
static void fill_split(const TaskPlan& P, int group, double* out) {
    const int own = (P.NS + group - 1) / group, slots = own * group;
    auto at = [&](int r, int s, int c) {
        return out + 2 * ((((size_t)r * own + s % own) * 2 + c) * group + s / own);
    };
    const double shift = std::ldexp(1.5, P.split_top + 5);  // ulp 2^(E-47), E as in split_exact
    std::fill(out, out + (size_t)4 * (P.R + 1) * slots, 0.0);
    for (int s = P.NS; s < slots; ++s) at(P.R, s, 0)[0] = 1.0;  // a padding slot's factor
    for (int r = 0; r < P.R; ++r) {
        const double m = r == 0 ? 1.0 : r <= P.nlow ? (double)(P.low_radix[r - 1] - 1) : 0.0;
        for (int s = 0; s < P.NS; ++s)
            for (int c = 0; c < 2; ++c) {
                const double v = P.entry(r, s)[c], hi = (v + shift) - shift, lo = v - hi;
                double *const o = at(r, s, c), *const b = at(P.R, s, c);
                o[0] = hi;
                o[1] = lo;
                b[0] += m * hi;
                b[1] += m * lo;
            }
    }
}

// Reflected mixed-radix Gray walk from k = 0 over digits with the given radices
// (digit 0 moves fastest).  Entry t describes the move into index t; the table
// has prod(radix) entries.  A step moves one digit by one, so the weight
// prod C(m, k) changes by one exact ratio of binomials (an int64: the digits of a
// walk hold at most 40 photons, prod C <= 2^40) and its sign alternates.
static void build_table(const unsigned char* radix, size_t n, RepStep* tab) {
    uint64_t L = 1;
    for (size_t k = 0; k < n; ++k) L *= radix[k];
    int g[kMaxDigits], o[kMaxDigits];
    int64_t bw[kMaxDigits][kMaxSlots + 1];
    for (size_t k = 0; k < n; ++k) {
        g[k] = 0;
        o[k] = 1;
        for (int v = 0; v < radix[k]; ++v) bw[k][v] = (int64_t)binom_u64(radix[k] - 1, v);
    }
    tab[0] = RepStep{0u, 0u, 1.0};
    int64_t w = 1;
    for (uint64_t t = 1; t < L; ++t) {
        size_t d = 0;
        int nv = 0;
        for (;;) {
            nv = g[d] + o[d];
            if (nv >= 0 && nv <= radix[d] - 1) break;
            o[d] = -o[d];
            ++d;
        }
        const bool up = nv > g[d];
        w = w / bw[d][g[d]] * bw[d][nv];
        g[d] = nv;
        tab[t].row = (uint32_t)(1 + d);
        tab[t].dir = up ? 1u : 0u;
        tab[t].w = (double)((t & 1) ? -w : w);
    }
}

// ------------------------------------------------------------ batch buffers --

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// Host worker threads kept for the life of the process (a 16-thread spawn and
// join costs ~0.5 ms, and a batch call runs four parallel phases).  One parallel
// phase at a time uses the pool; a phase that finds it busy (calls from several
// host threads) starts threads of its own.  The pool object is never destroyed,
// so no thread waits on a destroyed condition variable at process exit.
struct HostPool {
    std::mutex call_mu;  // one phase at a time
    std::mutex mu;
    std::condition_variable wake, fin;
    const std::function<void(int64_t, int64_t)>* job = nullptr;
    int64_t n = 0;
    int slices = 0, next = 0, done = 0, workers = 0;

    void worker() {
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            wake.wait(lk, [&] { return job != nullptr && next < slices; });
            run_one(lk);
        }
    }
    // claims the next slice (mu held, a slice left) and runs it with mu released
    void run_one(std::unique_lock<std::mutex>& lk) {
        const int s = next++;
        const std::function<void(int64_t, int64_t)>* f = job;
        const int64_t lo = n * s / slices, hi = n * (s + 1) / slices;
        lk.unlock();
        (*f)(lo, hi);
        lk.lock();
        if (++done == slices) fin.notify_all();
    }
    void run(int64_t count, int nslices, const std::function<void(int64_t, int64_t)>& f) {
        {
            std::lock_guard<std::mutex> g(mu);
            while (workers < nslices - 1) {  // the calling thread runs slices too
                try {
                    std::thread(&HostPool::worker, this).detach();
                } catch (const std::system_error&) {
                    break;  // fewer workers: the caller claims what is left
                }
                ++workers;
            }
            job = &f;
            n = count;
            slices = nslices;
            next = 0;
            done = 0;
        }
        wake.notify_all();
        std::unique_lock<std::mutex> lk(mu);
        while (next < slices) run_one(lk);
        fin.wait(lk, [&] { return done == slices; });
        job = nullptr;
    }
};

static HostPool& host_pool() {
    static HostPool* pool = new HostPool;  // never destroyed (see above)
    return *pool;
}

// fn(lo, hi) over [0, n) in contiguous slices on up to 16 host threads, at
// least `grain` items per slice; the caller's thread runs slices itself, and all
// of them when no thread can be started.  fn must not throw.
template <class F>
static void host_parallel(int64_t n, int64_t grain, F&& fn) {
    const int64_t hw = std::max<int64_t>(1, (int64_t)std::thread::hardware_concurrency());
    const int64_t nthreads = std::min<int64_t>(hw, std::min<int64_t>(16, (n + grain - 1) / grain));
    if (nthreads <= 1) {
        fn((int64_t)0, n);
        return;
    }
    HostPool& pool = host_pool();
    std::unique_lock<std::mutex> busy(pool.call_mu, std::try_to_lock);
    if (busy.owns_lock()) {
        const std::function<void(int64_t, int64_t)> f = [&fn](int64_t lo, int64_t hi) { fn(lo, hi); };
        pool.run(n, (int)nthreads, f);
        return;
    }
    std::vector<std::thread> spawned;
    spawned.reserve((size_t)nthreads);
    for (int64_t t = 0; t < nthreads; ++t) {
        const int64_t lo = n * t / nthreads, hi = n * (t + 1) / nthreads;
        try {
            spawned.emplace_back(fn, lo, hi);
        } catch (const std::system_error&) {
            fn(lo, hi);
        }
    }
    for (std::thread& th : spawned) th.join();
}

// Byte offsets in a batch's device buffer; the staging buffer mirrors all but the partials.
// The binomials stay, everything from the head on is uploaded for each batch.
struct BatchLayout {
    static constexpr size_t binom = 0, head = 13568;  // 41 x 41 doubles, then 256 bytes
    size_t tasks = 0, items = 0, order = 0, data = 0, part = 0, end = 0;

    void set(size_t nt, size_t ni, size_t nd) {
        tasks = head + 256;
        items = align256(tasks + nt * sizeof(RepTask));
        order = align256(items + ni * sizeof(RepItem));
        data = align256(order + ni * sizeof(unsigned));
        part = align256(data + nd);
        end = align256(part + ni * sizeof(ddc));
    }
};
static_assert(BatchLayout::head % 256 == 0 && BatchLayout::head >= sizeof(double) * kBinomStride * kBinomStride, "");

// Batches of up to this many tasks are laid out as tightly as they come and launched
// directly: the layout for the capacities, which the captured graph needs, is 120 KB longer
// to upload, and a graph's launch costs more than two kernels' (one task of
// 14 photons and 2304 steps: 64.7 -> 33.5 us a call, of 30 photons 160 -> 144 us).
constexpr size_t kDirectTasks = 64;

struct BatchBuffers {
    void* dbuf = nullptr;
    void* hbuf = nullptr;
    size_t cap_tasks = 0, cap_items = 0, cap_data = 0;
    BatchLayout at;  // for the capacities
    size_t off_out = 0, total = 0;
    hipGraphExec_t graph[kRanges] = {};  // FP64 slot ranges, then the double-double ones
    int grid[kRanges] = {};
    // last prepared batch (for replays): its graph's range, or the one-block launch
    int last_range = -1;
    int last_ntasks = 0;
    int last_tiny_ns = 0;  // > 0: last_tiny
    TinyParams last_tiny = {};
    bool last_is_direct = false;      // last_direct, of last_ntasks tasks
    RepBatchParams last_direct = {};

    // Nothing to replay: before a buffer is written over, and until the batch it is written
    // for has run (the last one's launches would read the new one's counts and tasks).
    void forget_last() {
        last_range = -1;
        last_ntasks = 0;
        last_tiny_ns = 0;
    }

    void layout(size_t nt, size_t ni, size_t nd) {
        cap_tasks = nt;
        cap_items = ni;
        cap_data = nd;
        at.set(nt, ni, nd);
        total = at.end;
        off_out = at.part;  // in the staging buffer: the kernels write there
    }
    void drop_graphs() {
        for (auto& g : graph)
            if (g) {
                (void)hipGraphExecDestroy(g);
                g = nullptr;
            }
    }
};

// The context's batch buffers, created on first use.
static BatchBuffers& batch_of(Engine& E) {
    if (!E.batch) E.batch = new BatchBuffers();
    return *E.batch;
}

// Releases a context's batch buffers and graphs (its stream is drained); the
// context lock is held.
void release_batch_locked(Engine& E) {
    if (!E.batch) return;
    BatchBuffers& B = *E.batch;
    B.drop_graphs();
    if (B.dbuf) (void)hipFree(B.dbuf);
    if (B.hbuf) (void)hipHostFree(B.hbuf);
    B.dbuf = B.hbuf = nullptr;
    B.cap_tasks = B.cap_items = B.cap_data = 0;
    for (int& g : B.grid) g = 0;
    B.forget_last();
}

// The context whose batch ran last: pqb_batch_replay replays it.
static std::atomic<Engine*> g_last_batch{nullptr};

static int ensure_batch_buffers_locked(Engine& E, size_t nt, size_t ni, size_t nd) {
    BatchBuffers& B = batch_of(E);
    if (B.dbuf && nt <= B.cap_tasks && ni <= B.cap_items && nd <= B.cap_data) return PQB_OK;
    (void)hipStreamSynchronize(E.stream);
    B.drop_graphs();
    B.forget_last();
    if (B.dbuf) (void)hipFree(B.dbuf);
    if (B.hbuf) (void)hipHostFree(B.hbuf);
    B.dbuf = B.hbuf = nullptr;
    B.layout(std::max<size_t>(nt, std::max<size_t>(2 * B.cap_tasks, 64)),
             std::max<size_t>(ni, std::max<size_t>(2 * B.cap_items, 4096)),
             std::max<size_t>(nd, std::max<size_t>(2 * B.cap_data, (size_t)1 << 20)));
    // on any failure below, leave no buffer behind: the capacity check above
    // must not accept a half-built set on the next call
    auto release = [&B]() {
        if (B.dbuf) (void)hipFree(B.dbuf);
        if (B.hbuf) (void)hipHostFree(B.hbuf);
        B.dbuf = B.hbuf = nullptr;
        B.cap_tasks = B.cap_items = B.cap_data = 0;
    };
    hipError_t e = hipMalloc(&B.dbuf, B.total);
    if (e != hipSuccess) {
        B.dbuf = nullptr;
        release();
        return hip_fail(e, "hipMalloc(batch)");
    }
    e = hipHostMalloc(&B.hbuf, B.off_out + (B.cap_tasks * 6 + 1) * sizeof(double), hipHostMallocCoherent);
    if (e != hipSuccess) {
        B.hbuf = nullptr;
        release();
        return hip_fail(e, "hipHostMalloc(batch)");
    }
    std::memset(B.hbuf, 0, B.at.data);
    double* bt = reinterpret_cast<double*>(static_cast<char*>(B.hbuf) + BatchLayout::binom);
    for (int m = 0; m < kBinomStride; ++m)
        for (int k = 0; k < kBinomStride; ++k) bt[m * kBinomStride + k] = (double)binom_u64(m, k);
    // counter + header start at zero on the device
    e = hipMemcpyAsync(B.dbuf, B.hbuf, B.at.tasks, hipMemcpyHostToDevice, E.stream);
    if (e == hipSuccess) e = hipStreamSynchronize(E.stream);
    if (e != hipSuccess) {
        release();
        return hip_fail(e, "batch init");
    }
    return PQB_OK;
}

static RepBatchParams batch_params(Engine& E, const BatchLayout& at) {
    BatchBuffers& B = batch_of(E);
    char* d = static_cast<char*>(B.dbuf);
    RepBatchParams p;
    p.tasks = reinterpret_cast<const RepTask*>(d + at.tasks);
    p.items = reinterpret_cast<const RepItem*>(d + at.items);
    p.order = reinterpret_cast<const unsigned*>(d + at.order);
    p.binom = reinterpret_cast<const double*>(d + BatchLayout::binom);
    p.partials = reinterpret_cast<ddc*>(d + at.part);
    p.out = reinterpret_cast<double*>(static_cast<char*>(B.hbuf) + B.off_out);
    p.head = reinterpret_cast<unsigned*>(d + BatchLayout::head);
    p.counts = reinterpret_cast<const unsigned*>(d + BatchLayout::head + 64);
    p.done = nullptr;
    return p;
}

static hipError_t launch_batch(int range, const RepBatchParams& p, int grid, int reduce_blocks, hipStream_t st) {
    return range >= kDDRange0 ? launch_rep_dd(range, p, grid, reduce_blocks, st)
                              : launch_rep_batch(range, p, grid, reduce_blocks, st);
}

static int batch_grid_locked(Engine& E, int range) {
    BatchBuffers& B = batch_of(E);
    if (B.grid[range] == 0) {
        int nb = 0;
        const void* fn = range >= kDDRange0 ? rep_dd_kernel_fn(range) : rep_batch_kernel_fn(range);
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, 256, 0);
        if (e != hipSuccess || nb <= 0) nb = 1;
        B.grid[range] = nb * E.cus;
    }
    return B.grid[range];
}

static int capture_batch(Engine& E, int range, const RepBatchParams& p, int reduce_blocks, hipGraphExec_t* out) {
    const int grid = batch_grid_locked(E, range);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamBeginCapture(E.stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return hip_fail(e, "hipStreamBeginCapture");
    hipError_t le = launch_batch(range, p, grid, reduce_blocks, E.stream);
    e = hipStreamEndCapture(E.stream, &g);
    if (le != hipSuccess) return hip_fail(le, "batch launch (capture)");
    if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
    hipGraphExec_t ex = nullptr;
    e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) return hip_fail(e, "hipGraphInstantiate");
    *out = ex;
    return PQB_OK;
}

static int batch_graph_locked(Engine& E, int range, hipGraphExec_t* out) {
    BatchBuffers& B = batch_of(E);
    if (!B.graph[range]) {
        const int st = capture_batch(E, range, batch_params(E, B.at), kReduceBlocks, &B.graph[range]);
        if (st) return st;
    }
    *out = B.graph[range];
    return PQB_OK;
}

// Walk lengths set by the autotuner, indexed by photon count (0 = automatic).
static std::atomic<int64_t> g_walk[PQB_MAX_COLS + 1] = {};

// Target walk length for a task of S steps when the batch holds `total`
// steps: long walks amortise the per-chunk seed, but there must be enough
// chunks to keep every resident lane busy.
static uint64_t choose_L(double S, double total, int64_t lanes, bool fp64, double step = 1.0) {
    // A lane's time is (its chunks) x (walk + per-chunk cost: the item fetch, the
    // mixed-radix decomposition of the chunk index and the seed, tens of FP64 steps
    // with many chunk digits).  With little work per lane one chunk each; in the FP64
    // sweep chunks of up to 128 steps even if up to three quarters of the lanes stay
    // idle (a single 9e6-step task on the whole grid: 0.26 ms at 4 chunks per lane,
    // 0.137 ms at one chunk of ~45 steps per lane, 0.10 ms at 128-step chunks; a
    // 4608-step task keeps its 16-step chunks).  The double-double step costs ~10x an
    // FP64 step, so there the seed is cheap and short walks stay (n = 16: 0.046 ms
    // against 0.19 ms with the floor).  Larger batches take 4 chunks per lane so that
    // uneven items balance.
    const double per_lane = std::max(total, S) / (double)std::max<int64_t>(lanes, 1);
    const double chunks_per_lane = per_lane < 1024.0 ? 1.0 : 4.0;
    double want_chunks =
        std::max<double>(chunks_per_lane * (double)lanes * S / std::max(total, S), 1.0);
    double L = S / want_chunks;
    L = std::min(L, S / 64.0);  // at least one chunk per lane of a wave
    // `step`: cost of a step in steps of the sweep over all rows; an expanded task's chunk
    // is as long in time, not in steps (30 photons, degree 3: 24-step chunks 68.4 us,
    // 36-step ones 72.3 us)
    if (fp64 && per_lane < 1024.0)
        L = std::max(L, std::min(128.0, 4.0 * S / (double)std::max<int64_t>(lanes, 1)) / step);
    L = std::min<double>(std::max<double>(L, 16.0), 2048.0);
    return (uint64_t)L;
}

// Chunks of the double-double sweep in flight on the whole grid.
static int64_t dd_chunks(Engine& E, int max_ns, bool split) {
    const int range = rep_dd_range_for(max_ns, split);
    return (int64_t)batch_grid_locked(E, range) * (kBlock / kWave) * rep_dd_walkers(range);
}

constexpr int kUnsplit = INT_MIN;  // in place of a task's split_top

// Column sums of the tasks whose rows can be split from which on they are swept apart from
// others that cannot: it saves them 5 of 11 instructions a component and costs a further
// upload, sweep and wait.  Lists of some of the first kind and one of the second, together /
// apart, us: 8 x 16 (4e6) 100 / 164, 200 and 3 x 12 (5e6) 345 / 485, 8 x 20 (8e7) 440 / 430,
// 3 x 24 (6e8) 1803 / 1648, 32 x 22 (1.5e9) 4320 / 2970.
constexpr double kApartWork = 0x1p26;

static void set_split(TaskPlan& P, int top) {
    P.split = true;
    P.split_top = top;
}

// The matrix of every task of a batch, where they share one.
struct SharedMatrix {
    const double* A = nullptr;
    int64_t rows = 0, cols = 0, ld = 0;
    size_t bytes() const { return (size_t)rows * (size_t)cols * sizeof(double2); }
};

// Run a list of planned tasks; results (6 doubles each) into out6.  dd: the
// double-double sweep (a chunk per group of lanes) instead of the FP64 one.
static int run_tasks_locked(Engine& E, std::vector<TaskPlan>& plans, std::vector<double>& out6, bool dd,
                            const SharedMatrix& shared = SharedMatrix()) {
    BatchBuffers& B = batch_of(E);
    const size_t nt = plans.size();
    out6.assign(nt * 6, 0.0);
    // sweeps to run
    std::vector<size_t> live;
    bool any_expanded = false;
    int min_ns = 1 << 30, max_ns = 0;
    for (size_t i = 0; i < nt; ++i) {
        if (plans[i].trivial) {
            out6[6 * i] = plans[i].tre;
            out6[6 * i + 1] = plans[i].tim;
            out6[6 * i + 2] = plans[i].tre;
            out6[6 * i + 4] = plans[i].tim;
            continue;
        }
        live.push_back(i);
        any_expanded = any_expanded || plans[i].degree > 0;
        min_ns = std::min(min_ns, plans[i].NS);
        max_ns = std::max(max_ns, plans[i].NS);
    }
    if (live.empty()) return PQB_OK;
    // tasks that no launch takes together run one kind after the other: up to 32 slots and more;
    // double-double, split rows and others
    auto apart = [&](auto first) {
        std::vector<TaskPlan> part[2];
        std::vector<size_t> index[2];
        for (size_t i : live) {
            const int which = first(plans[i]) ? 0 : 1;
            part[which].push_back(plans[i]);
            index[which].push_back(i);
        }
        for (int which = 0; which < 2; ++which) {
            std::vector<double> o;
            const int st = run_tasks_locked(E, part[which], o, dd, shared);
            if (st) return st;
            for (size_t k = 0; k < index[which].size(); ++k)
                std::copy(&o[6 * k], &o[6 * k] + 6, &out6[6 * index[which][k]]);
        }
        return (int)PQB_OK;
    };
    const bool split = plans[live[0]].split;
    for (size_t i : live)
        if (plans[i].split != split) return apart([](const TaskPlan& P) { return P.split; });
    const int range = dd ? rep_dd_range_for(max_ns, split) : rep_range_for(min_ns, max_ns);
    if (range < 0) return apart([](const TaskPlan& P) { return P.NS <= 32; });

    // ---- work items ----
    std::vector<RepItem> items;
    // cost class of each item: items take few distinct costs (one per task shape
    // and item size), ordered below by a counting pass instead of a sort
    std::vector<unsigned> item_class;
    std::vector<uint64_t> class_cost;
    std::unordered_map<uint64_t, unsigned> class_of;
    class_of.reserve(256);
    std::vector<std::pair<uint32_t, uint32_t>> task_items(live.size());
    // target Gray steps per lane (quad) per item: small items balance the tail of
    // an uneven batch (4096 tasks of 8..26 photons: replay 9.17 / 8.81 / 8.68 / 8.64 ms at 2048 / 1024 /
    // 512 / 256 steps), the cost being one atomic fetch per item
    const uint64_t lane_steps = 512;
    const uint64_t walkers = dd ? (uint64_t)rep_dd_walkers(range) : 64;  // chunks a wave works on at once
    auto per_item_of = [&](const TaskPlan& P) { return walkers * std::max<uint64_t>(1, lane_steps / P.L); };
    // A batch too small to give every resident wave ~4 items at that size
    // (a single mid-size task, say) gets smaller items, down to one chunk per
    // walker, so that the whole grid has work.
    uint64_t cap = ~(uint64_t)0;
    {
        const uint64_t target = 4 * (uint64_t)batch_grid_locked(E, range) * (kBlock / kWave);
        uint64_t n_default = 0, chunks = 0;
        for (size_t k : live) {
            n_default += (plans[k].nchunks + per_item_of(plans[k]) - 1) / per_item_of(plans[k]);
            chunks += plans[k].nchunks;
        }
        if (n_default < target) cap = walkers * std::max<uint64_t>(1, (chunks + target * walkers - 1) / (target * walkers));
    }
    {
        size_t nitems = 0;
        for (size_t k = 0; k < live.size(); ++k) {
            const uint64_t per_item = std::min(per_item_of(plans[live[k]]), cap);
            nitems += (size_t)((plans[live[k]].nchunks + per_item - 1) / per_item);
        }
        items.reserve(nitems);
        item_class.reserve(nitems);
    }
    uint64_t last_cost = ~(uint64_t)0;
    unsigned last_class = 0;
    for (size_t k = 0; k < live.size(); ++k) {
        const TaskPlan& P = plans[live[k]];
        const uint64_t per_item = std::min(per_item_of(P), cap);
        const uint64_t chunk_cost = P.L * (uint64_t)step_cost(P.degree, P.NS);
        task_items[k].first = (uint32_t)items.size();
        for (uint64_t c0 = 0; c0 < P.nchunks; c0 += per_item) {
            const uint64_t cnt = std::min<uint64_t>(per_item, P.nchunks - c0);
            const uint64_t cost = ((cnt + walkers - 1) / walkers) * chunk_cost;
            if (cost != last_cost) {
                const auto r = class_of.emplace(cost, (unsigned)class_cost.size());
                if (r.second) class_cost.push_back(cost);
                last_class = r.first->second;
                last_cost = cost;
            }
            item_class.push_back(last_class);
            items.push_back(RepItem{(uint32_t)k, (uint32_t)cnt, (uint32_t)c0, 0u});
        }
        task_items[k].second = (uint32_t)items.size() - task_items[k].first;
    }
    // launch order: largest cost first, ties in item order
    std::vector<unsigned> order(items.size());
    {
        std::vector<unsigned> rank(class_cost.size());
        std::iota(rank.begin(), rank.end(), 0u);
        std::sort(rank.begin(), rank.end(), [&](unsigned a, unsigned b) { return class_cost[a] > class_cost[b]; });
        std::vector<unsigned> start(class_cost.size() + 1, 0u), pos_of(class_cost.size());
        for (size_t r = 0; r < rank.size(); ++r) pos_of[rank[r]] = (unsigned)r;
        for (unsigned c : item_class) ++start[pos_of[c] + 1];
        for (size_t r = 0; r < rank.size(); ++r) start[r + 1] += start[r];
        for (size_t i = 0; i < items.size(); ++i) order[start[pos_of[item_class[i]]]++] = (unsigned)i;
    }

    // ---- data region: A, base per task, deduplicated step tables ----
    // step tables shared by the tasks whose walked radices agree, looked up by the
    // radices as a short string (radices <= 41, up to 40 digits); built below,
    // straight into the staging buffer
    std::unordered_map<std::string, size_t> table_off;
    table_off.reserve(64);
    std::string key;
    std::vector<std::pair<size_t, size_t>> tables;  // (offset, task whose radices it walks)
    std::vector<size_t> a_off(live.size()), b_off(live.size()), x_off(live.size()), t_off(live.size());
    const int group = (int)(64 / walkers);  // lanes of a chunk
    auto slots_of = [&](const TaskPlan& P) { return (P.NS + group - 1) / group * group; };
    auto area = [](size_t complexes) { return align256(complexes * sizeof(double2)); };
    size_t own = 0;  // the tasks' own rows, bases and expanded rows
    for (size_t k : live) {
        const TaskPlan& P = plans[k];
        own += area((size_t)P.R * P.NS) + area((size_t)P.NS) + (P.degree > 0 ? area((size_t)P.NS) : 0);
    }
    // a shared matrix is uploaded instead and the tasks' rows formed on the GPU (rep_layout_kernel)
    const bool direct = live.size() <= kDirectTasks;
    const bool gather = !direct && !dd && shared.A && shared.bytes() <= own;
    size_t nd = gather ? align256(shared.bytes()) : 0;
    for (size_t k = 0; k < live.size(); ++k) {
        const TaskPlan& P = plans[live[k]];
        key.assign(reinterpret_cast<const char*>(P.low_radix), (size_t)P.nlow);
        const auto it = table_off.emplace(key, nd);
        t_off[k] = it.first->second;
        if (it.second) {
            tables.emplace_back(nd, k);
            nd = align256(nd + (size_t)P.L * sizeof(RepStep));
        }
    }
    size_t uploaded = nd;
    for (size_t k = 0; k < live.size(); ++k) {
        const TaskPlan& P = plans[live[k]];
        a_off[k] = nd;
        b_off[k] = nd += area((size_t)P.R * P.NS);
        x_off[k] = nd += area((size_t)P.NS);  // expanded row, or the split rows
        if (P.degree > 0 && !gather) nd += area((size_t)P.NS);
        if (split) nd += area((size_t)2 * (P.R + 1) * slots_of(P));
    }
    if (!gather) uploaded = nd;
    int st = ensure_batch_buffers_locked(E, live.size(), items.size(), nd);
    if (st) return st;
    BatchLayout at = B.at;
    if (direct) at.set(live.size(), items.size(), nd);
    B.forget_last();
    char* h = static_cast<char*>(B.hbuf);
    char* d = static_cast<char*>(B.dbuf);
    // header: head counter (0), counts
    std::memset(h + BatchLayout::head, 0, 256);
    unsigned* counts = reinterpret_cast<unsigned*>(h + BatchLayout::head + 64);
    counts[0] = (unsigned)items.size();
    counts[1] = (unsigned)live.size();
    RepTask* T = reinterpret_cast<RepTask*>(h + at.tasks);
    if (gather)
        for (int64_t r = 0; r < shared.rows; ++r)
            std::memcpy(h + at.data + (size_t)r * shared.cols * sizeof(double2), shared.A + 2 * r * shared.ld,
                        (size_t)shared.cols * sizeof(double2));
    // descriptors and per-task data into the pinned staging buffer (disjoint
    // regions per task)
    host_parallel((int64_t)live.size(), 256, [&](int64_t lo, int64_t hi) {
    for (int64_t k = lo; k < hi; ++k) {
        const TaskPlan& P = plans[live[(size_t)k]];
        RepTask t;
        std::memset(&t, 0, sizeof(t));
        t.A = reinterpret_cast<const double2*>(d + at.data + a_off[k]);
        t.base = reinterpret_cast<const double2*>(d + at.data + b_off[k]);
        t.table = reinterpret_cast<const RepStep*>(d + at.data + t_off[k]);
        t.NS = P.NS;
        t.L = (int)P.L;
        t.nhigh = P.nhigh;
        t.nlow = P.nlow;
        for (int ld = 0; ld < P.nlow; ++ld) t.lrad[ld] = P.low_radix[ld];
        t.item0 = task_items[k].first;
        t.nitems = task_items[k].second;
        t.out_index = (uint32_t)k;
        t.nchunks = (uint32_t)P.nchunks;
        t.degree = P.degree;
        t.rows = P.R;
        t.xrow = reinterpret_cast<const double2*>(d + at.data + x_off[k]);
        t.scale[0] = P.scale;
        for (int hd = 0; hd < P.nhigh; ++hd) {
            t.hrow[hd] = (uint32_t)(1 + P.nlow + hd);
            t.hrad[hd] = P.high_radix[hd];
        }
        if (gather) {
            t.src = reinterpret_cast<const double2*>(d + at.data);
            t.src_ld = shared.cols;
            t.transpose = P.transpose;
            t.src_xrow = P.xrow;
            std::copy(P.row, P.row + P.R, t.src_row);
            std::copy(P.slot, P.slot + P.NS, t.src_slot);
        } else {
            fill_rows(P, reinterpret_cast<double*>(h + at.data + a_off[(size_t)k]));
            fill_base(P, reinterpret_cast<double*>(h + at.data + b_off[(size_t)k]));
            if (split) {
                fill_split(P, group, reinterpret_cast<double*>(h + at.data + x_off[(size_t)k]));
                t.split = reinterpret_cast<const double2*>(d + at.data + x_off[k]);
            }
            if (P.degree > 0) fill_xrow(P, reinterpret_cast<double*>(h + at.data + x_off[(size_t)k]));
        }
        T[k] = t;
    }
    });
    host_parallel((int64_t)tables.size(), 4, [&](int64_t lo, int64_t hi) {
        for (int64_t i = lo; i < hi; ++i) {
            const TaskPlan& P = plans[live[tables[(size_t)i].second]];
            build_table(P.low_radix, (size_t)P.nlow, reinterpret_cast<RepStep*>(h + at.data + tables[(size_t)i].first));
        }
    });
    RepItem* I = reinterpret_cast<RepItem*>(h + at.items);
    std::memcpy(I, items.data(), items.size() * sizeof(RepItem));
    unsigned* O = reinterpret_cast<unsigned*>(h + at.order);
    std::memcpy(O, order.data(), order.size() * sizeof(unsigned));

    hipError_t e = hipMemcpyAsync(d + BatchLayout::head, h + BatchLayout::head, at.data + uploaded - BatchLayout::head,
                                  hipMemcpyHostToDevice, E.stream);
    if (e != hipSuccess) return hip_fail(e, "batch upload");
    if (any_expanded || gather) {  // outside the graph: it divides uploaded rows in place, once
        e = launch_rep_layout(reinterpret_cast<RepTask*>(d + at.tasks), (int64_t)live.size(), E.stream);
        if (e != hipSuccess) return drain_fail(E, e, "prep launch");
    }
    if (direct) {
        RepBatchParams p = batch_params(E, at);
        if (live.size() == 1) {
            p.done = reinterpret_cast<unsigned*>(h + B.off_out + 6 * sizeof(double));
            *p.done = 0u;
        }
        e = launch_batch(range, p, batch_grid_locked(E, range), (int)live.size(), E.stream);
        if (e == hipSuccess) e = p.done ? wait_result(E, p.done) : hipStreamSynchronize(E.stream);
        if (e != hipSuccess) return drain_fail(E, e, "batch sweep");
        p.done = nullptr;
        B.last_direct = p;
    } else {
        hipGraphExec_t gx = nullptr;
        st = batch_graph_locked(E, range, &gx);
        if (st) {
            (void)hipStreamSynchronize(E.stream);  // the upload may still read the staging buffer
            return st;
        }
        e = hipGraphLaunch(gx, E.stream);
        if (e != hipSuccess) return drain_fail(E, e, "hipGraphLaunch");
        e = hipStreamSynchronize(E.stream);
        if (e != hipSuccess) return hip_fail(e, "batch sweep");
    }
    const double* res = reinterpret_cast<const double*>(h + B.off_out);
    for (size_t k = 0; k < live.size(); ++k) std::copy(&res[6 * k], &res[6 * k] + 6, &out6[6 * live[k]]);
    B.last_range = range;
    B.last_is_direct = direct;
    B.last_ntasks = (int)live.size();
    g_last_batch.store(&E);
    return PQB_OK;
}

// One task of few steps in one block (perm_tiny.hip); *done false when it does not fit.
static int run_tiny_locked(Engine& E, const pqb_task& t, const SweepChoice& choice, double* out, bool* done) {
    TaskPlan P;
    int st = plan_task(t.A, t.rows, t.cols, t.ld, t.row_mult, t.col_mult, 1, P, &choice);
    if (st || P.nhigh > kTinyDigits) return st;
    TinyParams p = {};
    for (int d = 0; d < P.nhigh; ++d) p.radix[d] = P.high_radix[d];
    if (P.nlow != 0 || P.degree != 0 || !tiny_split(p, P.NS, P.R)) return PQB_OK;
    st = ensure_batch_buffers_locked(E, 1, 1, (size_t)P.R * P.NS * sizeof(double2));
    if (st) return st;
    BatchBuffers& B = batch_of(E);
    B.forget_last();
    char* h = static_cast<char*>(B.hbuf);
    fill_rows(P, reinterpret_cast<double*>(h + B.at.data));
    p.A = reinterpret_cast<const double2*>(h + B.at.data);
    p.out = reinterpret_cast<double*>(h + B.off_out);
    p.scale = P.scale;
    p.done = reinterpret_cast<unsigned*>(p.out + 6);
    *p.done = 0u;
    hipError_t e = launch_tiny(P.NS, p, 1, E.stream);
    if (e == hipSuccess) e = wait_result(E, p.done);
    if (e != hipSuccess) return drain_fail(E, e, "batch sweep");
    out[0] = p.out[0];
    out[1] = p.out[1];
    B.last_ntasks = 1;
    B.last_tiny_ns = P.NS;
    B.last_tiny = p;
    g_last_batch.store(&E);
    *done = true;
    return PQB_OK;
}

// ------------------------------------------------------------- validation --

// Reference rules for one repeated task (BBFGPermanentCalculatorRepeated.cpp:
// 78-81, .hpp:119-128; GlynnPermanentCalculatorRepeated.hpp:55-63).  Returns
// 1 with *decided set when no sweep is needed.
static int check_task(const pqb_task& t, int algo, bool* decided, double* re) {
    *decided = false;
    if (t.rows < 0 || t.cols < 0) return fail(PQB_ERR_ARG, "negative matrix dimension");
    if ((t.rows > 0 && !t.row_mult) || (t.cols > 0 && !t.col_mult))
        return fail(PQB_ERR_ARG, "occupation pointer is NULL");
    if (algo == PQB_ALGO_BBFG && t.rows == 0) {
        *decided = true;
        *re = 1.0;
        return PQB_OK;
    }
    int64_t sr = 0, sc = 0;
    for (int64_t i = 0; i < t.rows; ++i) {
        if (t.row_mult[i] < 0) return fail(PQB_ERR_ARG, "negative occupation number");
        sr += t.row_mult[i];
    }
    for (int64_t j = 0; j < t.cols; ++j) {
        if (t.col_mult[j] < 0) return fail(PQB_ERR_ARG, "negative occupation number");
        sc += t.col_mult[j];
    }
    if (sr != sc)
        return fail(PQB_ERR_STATE,
                    algo == PQB_ALGO_BBFG
                        ? "BBFGPermanentCalculatorRepeated_Tasks::calculate:  Number of input and output states should be equal"
                        : "GlynnPermanentCalculatorRepeated::calculate:  Number of input and output states should be equal");
    if (t.rows == 0 || t.cols == 0 || sr == 0) {
        *decided = true;
        *re = 1.0;
        return PQB_OK;
    }
    if (!t.A) return fail(PQB_ERR_ARG, "matrix pointer is NULL");
    if (t.ld < t.cols) return fail(PQB_ERR_ARG, "leading dimension smaller than the number of columns");
    if (sr > PQB_MAX_COLS) return fail(PQB_ERR_SIZE, "more than " + std::to_string(PQB_MAX_COLS) + " photons");
    return PQB_OK;
}

int batch_entry(const pqb_task* tasks, int64_t ntasks, int algo, int precision, double* out, int64_t L_override) {
    if (ntasks < 0) return fail(PQB_ERR_ARG, "negative task count");
    if (ntasks > 0 && (!tasks || !out)) return fail(PQB_ERR_ARG, "NULL pointer");
    if (algo != PQB_ALGO_BBFG && algo != PQB_ALGO_GLYNN) return fail(PQB_ERR_ARG, "unknown algorithm code");
    if (precision < PQB_PREC_DOUBLE || precision > PQB_PREC_INF) return fail(PQB_ERR_ARG, "unknown precision code");
    if (precision == PQB_PREC_EXACT) return fail(PQB_ERR_ARG, "exact mode is available for the plain permanent only");
    const bool dd = precision == PQB_PREC_INF;
    std::vector<TaskPlan> plans((size_t)ntasks);
    std::vector<SweepChoice> choices((size_t)ntasks);
    std::vector<int> photons((size_t)ntasks, 0);
    std::vector<int> tops(dd ? (size_t)ntasks : 0, kUnsplit);  // TaskPlan::split_top
    // Validation and planning are per task and independent: large batches run
    // them on host threads (4096 tasks are milliseconds of host work either
    // way).  Errors come back per task; the first one by task index is
    // reported, as a serial loop would.
    std::vector<int> pst((size_t)ntasks, PQB_OK);
    std::vector<std::string> perr((size_t)ntasks);
    host_parallel(ntasks, 512, [&](int64_t lo, int64_t hi) {
        for (int64_t i = lo; i < hi; ++i) {
            try {  // nothing may escape a worker thread
                bool decided = false;
                double v = 1.0;
                const int st = check_task(tasks[i], algo, &decided, &v);
                if (st) {
                    pst[(size_t)i] = st;
                    perr[(size_t)i] = t_err;  // t_err is per thread
                    continue;
                }
                if (decided) {
                    plans[(size_t)i].trivial = true;
                    plans[(size_t)i].tre = v;
                    continue;
                }
                PlanScratch& sc = plan_scratch();
                int64_t n = 0, nc = 0;
                compact_occupations(tasks[i].rows, tasks[i].cols, tasks[i].row_mult, tasks[i].col_mult, sc, &n, &nc);
                choices[(size_t)i] = choose_sweep(tasks[i].A, tasks[i].ld, sc, !dd);
                photons[(size_t)i] = (int)n;
                int top = 0;
                if (dd && split_exact(tasks[i].A, tasks[i].ld, sc, &top)) tops[(size_t)i] = top;
            } catch (const std::exception& ex) {
                pst[(size_t)i] = PQB_ERR_DEVICE;
                perr[(size_t)i] = std::string("internal error: ") + ex.what();
            }
        }
    });
    for (int64_t i = 0; i < ntasks; ++i)
        if (pst[(size_t)i]) {
            t_err = (ntasks > 1 ? "task " + std::to_string(i) + ": " : std::string()) + perr[(size_t)i];
            return pst[(size_t)i];
        }
    // of the tasks that run together: all of them; double-double, those whose rows are split
    // [1] and those whose are not [0]
    double total[2] = {0.0, 0.0};
    int max_photons[2] = {1, 1};  // = their largest slot count
    auto kind = [&](int64_t i) { return dd && tops[(size_t)i] != kUnsplit; };
    if (dd) {
        double work = 0.0;
        bool others = false;
        for (int64_t i = 0; i < ntasks; ++i)
            if (kind(i)) work += choices[(size_t)i].steps * photons[(size_t)i];
            else others = others || !plans[(size_t)i].trivial;
        if (others && work < kApartWork) std::fill(tops.begin(), tops.end(), kUnsplit);
    }
    for (int64_t i = 0; i < ntasks; ++i) {
        total[kind(i)] += choices[(size_t)i].steps;
        max_photons[kind(i)] = std::max(max_photons[kind(i)], photons[(size_t)i]);
    }
    bool any_sweep = false;
    for (const TaskPlan& P : plans) any_sweep = any_sweep || !P.trivial;
    if (!any_sweep) {  // every result decided by the edge rules: no device needed
        for (int64_t i = 0; i < ntasks; ++i) {
            out[2 * i] = plans[(size_t)i].tre;
            out[2 * i + 1] = plans[(size_t)i].tim;
        }
        return PQB_OK;
    }
    Lease L;
    int st = L.status();
    if (st) return st;
    Engine& E = *L;
    if (ntasks == 1 && !dd && L_override <= 0 && choices[0].steps <= (double)kTinySteps && photons[0] <= kTinySlots) {
        bool done = false;
        st = run_tiny_locked(E, tasks[0], choices[0], out, &done);
        if (st || done) return st;
    }
    // chunks in flight: a lane each (FP64), a group of lanes each (double-double)
    int64_t lanes[2];
    for (int k = 0; k < 2; ++k)
        lanes[k] = dd ? dd_chunks(E, max_photons[k], k == 1) : (int64_t)batch_grid_locked(E, 2) * kBlock;
    const bool large_batch = total[0] >= 1024.0 * (double)lanes[0];  // steps per lane
    auto plan_range = [&](int64_t lo, int64_t hi) {
        for (int64_t i = lo; i < hi; ++i) {
            if (plans[(size_t)i].trivial) continue;
            int64_t photons = 0;
            for (int64_t j = 0; j < tasks[i].cols; ++j) photons += tasks[i].col_mult[j];
            // The autotuned walk lengths are measured for the FP64 sweep on a large batch
            // (thousands of steps per lane); a small batch, a single task above all, keeps
            // the automatic rule (a 6e6-step task at the tuned 1024-step walk left all but
            // ~6000 lanes idle: 0.32 ms against 0.10 ms).  They were measured on the sweep over
            // all rows and hold for expanded tasks as they are: replays of 4096 tasks of 8..26 /
            // 18..26 / 14..22 photons 6.78 / 12.78 / 1.09 ms, with walks half as long 6.76 / 12.88 /
            // 1.08, with the automatic rule (which scales by the step's cost) 6.73 / 12.93 / 1.09.
            const int64_t tuned =
                (!dd && large_batch && photons >= 0 && photons <= PQB_MAX_COLS) ? g_walk[photons].load() : 0;
            const uint64_t L = L_override > 0 ? (uint64_t)L_override
                               : tuned > 0    ? (uint64_t)tuned
                                              : choose_L(choices[(size_t)i].steps, total[kind(i)], lanes[kind(i)], !dd,
                                                         step_cost(choices[(size_t)i].degree, (int)photons) /
                                                             step_cost(0, (int)photons));
            try {  // nothing may escape a worker thread
                pst[(size_t)i] = plan_task(tasks[i].A, tasks[i].rows, tasks[i].cols, tasks[i].ld,
                                           tasks[i].row_mult, tasks[i].col_mult, L, plans[(size_t)i], &choices[(size_t)i]);
                if (pst[(size_t)i]) perr[(size_t)i] = t_err;  // t_err is per thread
                if (kind(i)) set_split(plans[(size_t)i], tops[(size_t)i]);
            } catch (const std::exception& ex) {
                pst[(size_t)i] = PQB_ERR_DEVICE;
                perr[(size_t)i] = std::string("internal error: ") + ex.what();
            }
        }
    };
    host_parallel(ntasks, 256, plan_range);
    for (int64_t i = 0; i < ntasks; ++i)
        if (pst[(size_t)i]) {
            t_err = (ntasks > 1 ? "task " + std::to_string(i) + ": " : std::string()) + perr[(size_t)i];
            return pst[(size_t)i];
        }
    SharedMatrix shared{tasks[0].A, tasks[0].rows, tasks[0].cols, tasks[0].ld};
    for (int64_t i = 1; i < ntasks && shared.A; ++i)
        if (tasks[i].A != shared.A || tasks[i].rows != shared.rows || tasks[i].cols != shared.cols ||
            tasks[i].ld != shared.ld)
            shared = SharedMatrix();
    std::vector<double> out6;
    st = run_tasks_locked(E, plans, out6, dd, shared);
    if (st) return st;
    for (int64_t i = 0; i < ntasks; ++i) {
        out[2 * i] = out6[(size_t)(6 * i)];
        out[2 * i + 1] = out6[(size_t)(6 * i + 1)];
    }
    return PQB_OK;
}

int run_plain_dd_list_locked(Engine& E, const double* const* A, const int* R, const int* C, const int64_t* ld,
                             int64_t n, double* out) {
    std::vector<TaskPlan> plans((size_t)n);
    std::vector<int> tops((size_t)n, kUnsplit);
    const std::vector<int64_t> ones(PQB_MAX_COLS + 1, 1);
    double work = 0.0;
    bool others = false;
    for (int64_t k = 0; k < n; ++k) {
        int64_t rows = 0, cols = 0;
        compact_occupations(R[k], C[k], ones.data(), ones.data(), plan_scratch(), &rows, &cols);
        if (split_exact(A[k], ld[k], plan_scratch(), &tops[(size_t)k])) {
            work += std::ldexp((double)C[k], R[k] - 1);
        } else {
            tops[(size_t)k] = kUnsplit;
            others = true;
        }
    }
    if (others && work < kApartWork) std::fill(tops.begin(), tops.end(), kUnsplit);
    for (int64_t k = 0; k < n; ++k) {
        const double S = std::ldexp(1.0, R[k] - 1);
        const bool split = tops[(size_t)k] != kUnsplit;
        const int64_t chunks = dd_chunks(E, C[k], split);  // the slots are the columns
        const int st = plan_task(A[k], R[k], C[k], ld[k], ones.data(), ones.data(), choose_L(S, S, chunks, false),
                                 plans[(size_t)k], nullptr, true);
        if (split) set_split(plans[(size_t)k], tops[(size_t)k]);
        if (st) return n > 1 ? fail(st, "matrix " + std::to_string(k) + ": " + t_err) : st;
    }
    std::vector<double> out6;
    const int st = run_tasks_locked(E, plans, out6, true);
    if (st) return st;
    for (int64_t k = 0; k < n; ++k) {
        out[2 * k] = out6[6 * k];
        out[2 * k + 1] = out6[6 * k + 1];
    }
    return PQB_OK;
}

int run_plain_dd_locked(Engine& E, const double* A, int R, int C, int64_t ld, double* out) {
    return run_plain_dd_list_locked(E, &A, &R, &C, &ld, 1, out);
}

int batch_replay(int iters, double* ms) {
    Engine* last = g_last_batch.load();
    if (!last) return fail(PQB_ERR_ARG, "no batch has been run yet");
    Lease L(*last);
    if (L.status()) return L.status();
    Engine& E = *L;
    BatchBuffers& B = batch_of(E);
    const bool tiny = B.last_tiny_ns > 0, direct = !tiny && B.last_range >= 0 && B.last_is_direct;
    if (!tiny && !direct && (B.last_range < 0 || !B.graph[B.last_range]))
        return fail(PQB_ERR_ARG, "no batch has been run yet");
    // the launches of a small batch, captured here
    hipGraphExec_t gx = tiny ? nullptr : B.graph[B.last_range];
    if (direct) {
        const int st = capture_batch(E, B.last_range, B.last_direct, B.last_ntasks, &gx);
        if (st) return st;
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    if (e == hipSuccess) e = hipEventRecord(e0, E.stream);
    for (int i = 0; e == hipSuccess && i < iters; ++i)
        e = tiny ? launch_tiny(B.last_tiny_ns, B.last_tiny, 1, E.stream)
                 : hipGraphLaunch(gx, E.stream);
    if (e == hipSuccess) e = hipEventRecord(e1, E.stream);
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    float f = 0.f;
    if (e == hipSuccess) e = hipEventElapsedTime(&f, e0, e1);
    if (direct) (void)hipGraphExecDestroy(gx);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (e != hipSuccess) return hip_fail(e, "batch replay");
    *ms = f;
    return PQB_OK;
}

}  // namespace pqb

using namespace pqb;

extern "C" {

int pqb_perm_batch(const pqb_task* tasks, int64_t ntasks, int algo, int precision, double* out) {
    try {
        return batch_entry(tasks, ntasks, algo, precision, out, 0);
    } catch (const std::exception& ex) {
        return fail(PQB_ERR_DEVICE, std::string("internal error: ") + ex.what());
    }
}

int pqb_perm_batch_tuned(const pqb_task* tasks, int64_t ntasks, int algo, int precision, int64_t walk_length,
                         double* out) {
    try {
        return batch_entry(tasks, ntasks, algo, precision, out, walk_length);
    } catch (const std::exception& ex) {
        return fail(PQB_ERR_DEVICE, std::string("internal error: ") + ex.what());
    }
}

int pqb_perm_batch_states(const double* U, int64_t rows, int64_t cols, int64_t ld, const int64_t* inputs,
                          const int64_t* outputs, int64_t count, int algo, int precision, double* out) {
    try {
        if (count < 0 || rows < 0 || cols < 0) return fail(PQB_ERR_ARG, "negative size");
        if (count == 0) return PQB_OK;
        if (!out || (rows > 0 && !outputs) || (cols > 0 && !inputs)) return fail(PQB_ERR_ARG, "NULL pointer");
        if (ld < cols) return fail(PQB_ERR_ARG, "leading dimension smaller than the number of columns");
        // one task per pair, all pointing into U and the two state arrays
        std::vector<pqb_task> t((size_t)count);
        for (int64_t i = 0; i < count; ++i)
            t[(size_t)i] = pqb_task{U, rows, cols, ld, rows > 0 ? outputs + i * rows : nullptr,
                                    cols > 0 ? inputs + i * cols : nullptr};
        return batch_entry(t.data(), count, algo, precision, out, 0);
    } catch (const std::exception& ex) {
        return fail(PQB_ERR_DEVICE, std::string("internal error: ") + ex.what());
    }
}

int pqb_set_walk_lengths(const int64_t* walk, int64_t count) {
    for (int i = 0; i <= PQB_MAX_COLS; ++i) g_walk[i].store((walk && i < count && walk[i] > 0) ? walk[i] : 0);
    return PQB_OK;
}

int pqb_batch_replay(int iters, double* ms) {
    if (!ms || iters < 1) return fail(PQB_ERR_ARG, "bad replay arguments");
    return batch_replay(iters, ms);
}

int pqb_repeated_plan(const double* A, int64_t rows, int64_t cols, int64_t ld, const int64_t* row_mult,
                      const int64_t* col_mult, int64_t walk_length, int64_t* info) {
    if (!info || walk_length < 1) return fail(PQB_ERR_ARG, "bad arguments");
    pqb_task t{A, rows, cols, ld, row_mult, col_mult};
    bool decided = false;
    double v;
    int st = check_task(t, PQB_ALGO_BBFG, &decided, &v);
    if (st) return st;
    if (decided) {
        info[0] = info[1] = info[2] = info[3] = info[4] = info[5] = 0;
        return PQB_OK;
    }
    TaskPlan P;
    st = plan_task(A, rows, cols, ld, row_mult, col_mult, (uint64_t)walk_length, P);
    if (st) return st;
    info[0] = P.NS;
    info[1] = P.R;
    info[2] = P.nlow;
    info[3] = P.nhigh;
    info[4] = (int64_t)P.L;
    info[5] = (int64_t)P.nchunks;
    return PQB_OK;
}

}  // extern "C"
