// Host-side engine state shared by the C-ABI translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <string>
#include <vector>

#include "pqb_kernels.h"
#include "pqb_perm.h"

namespace pqb {

constexpr int kBlock = 256;            // threads per block of the sweep kernels
constexpr size_t kCounterBytes = 256;  // grid-reduction counter slot at workspace offset 0
constexpr int kMaxBlocks = 4096;       // partials capacity of the device-API workspace

struct PlainPlan {
    int K = 0;            // walk bits
    int B = 0;            // lane bits
    int H = 0;            // group bits
    int64_t waves = 1;    // launched waves
    int block = 64;       // threads per block
    int blocks = 1;
};

PlainPlan make_plain_plan(int R, int NC, int64_t waves_resident);

// `count` R x C plain permanents that one block each evaluates (perm_tiny.hip): p set but
// for A and out.
bool plain_tiny(int R, int C, int64_t count, TinyParams& p);

// Whether `count` R x C matrices are worth expanding (perm_expand.hip) where their
// entries allow it.
bool plain_expandable(int R, int C, int64_t count);

struct ddc;
struct PlainParams;
PlainParams plain_params(const PlainPlan& pl, int R, const double2* m2, int64_t m2_stride, ddc* partials,
                         unsigned* counter, double* out);
// The launches of device matrices (engine.hip); xp: plan of the expanded sweep or NULL.
int plain_device_launch(const double2* dA, int64_t count, int R, int C, const PlainPlan& pl, const PlainPlan* xp,
                        double2* m2, ddc* partials, unsigned* counters, double* d_out, hipStream_t st);

// Which sweep a repeated-row task takes (batch.hip): orientation and expanded row.
struct SweepChoice {
    bool transpose = false;
    int degree = 0;          // multiplicity of the expanded row, 0: none
    int64_t row = -1;        // the expanded row: original row (column when transposed)
    double steps = 0;        // Gray steps
};

// One planned repeated-row permanent (see batch.hip).  Its rows are not copied: they are
// taken from the task's matrix where they are laid out for the sweep.  No allocations of
// its own, so that thousands of plans cost nothing to make and to drop.
struct TaskPlan {
    bool trivial = false;      // decided without a sweep: value (tre, tim)
    bool transpose = false;    // rows of the sweep are columns of the matrix
    double tre = 1.0, tim = 0.0;
    const double* src = nullptr;  // the matrix, row stride ld
    int64_t ld = 0;
    int NS = 0;                // column slots
    int R = 0;                 // rows: anchor, low digits, high digits
    int N = 0;                 // photons
    int nlow = 0, nhigh = 0;
    uint64_t L = 1;            // walk length
    uint64_t nchunks = 1;
    int degree = 0;            // RepTask::degree
    bool split = false;        // double-double sweep over split rows (RepTask::split):
    int split_top = 0;         // entries below 2^split_top
    uint32_t xrow = 0;         // expanded: the expanded row (column when transposed)
    double scale = 1.0;        // 2^-(N-1); expanded: D! 2^-(N-D-1)
    uint32_t row[kMaxRepRows];    // R rows of the matrix (columns when transposed)
    uint32_t slot[kMaxSlots];     // NS columns of it (rows when transposed)
    unsigned char low_radix[kMaxDigits], high_radix[kMaxDigits];  // multiplicity + 1

    TaskPlan() {}              // the arrays stay as they are
    const double* entry(int r, int s) const {
        return src + 2 * (transpose ? (int64_t)slot[s] * ld + row[r] : (int64_t)row[r] * ld + slot[s]);
    }
};

int plan_task(const double* A, int64_t rows, int64_t cols, int64_t ld, const int64_t* rmult,
              const int64_t* cmult, uint64_t target_L, TaskPlan& P, const SweepChoice* choice = nullptr,
              bool plain = false);
int batch_entry(const pqb_task* tasks, int64_t ntasks, int algo, int precision, double* out,
                int64_t L_override);
struct Engine;

// Plain permanent (1 <= rows <= cols + 1) by the double-double sweep; context locked.
int run_plain_dd_locked(Engine& E, const double* A, int R, int C, int64_t ld, double* out);
// `n` such permanents (matrix k: A[k], R[k] x C[k], stride ld[k]), each planned as
// run_plain_dd_locked plans it, in one or two batched launches; out: 2 doubles each.
int run_plain_dd_list_locked(Engine& E, const double* const* A, const int* R, const int* C, const int64_t* ld,
                             int64_t n, double* out);
int list_entry(const double* const* A, const int64_t* rows, const int64_t* cols, const int64_t* ld,
               int64_t count, int algo, int precision, double* out);

// Process-wide device binding: the device every context runs on, its CU count
// and the occupancy of the plain sweep per column count (read-mostly).
struct DeviceState {
    std::mutex mu;
    int device = -1;
    int cus = 0;
    int blocks_per_cu[2][PQB_MAX_COLS + 1] = {};  // [expanded]
};
extern DeviceState g_dev;

// Binds the process to `dev` (dev < 0: keep the current binding, device 0 if
// none) and reports it; a change of device releases every context's resources.
int bind_device(int dev, int* device, int* cus);
// Resident waves of the plain sweep for `nc` columns on the bound device.
int64_t resident_waves(int nc, bool expanded);

// A column-minors sweep of `count` packed rows x (rows+1) device matrices without the sum
// over its partials, nblk x (rows+1) per matrix (grad.hip).
struct MinorsSweep {
    int rows = 0, nblk = 0;
    int64_t wpt = 0, blocks = 0;
    size_t partial_bytes = 0;
};
int minors_sweep_plan(int rows, int64_t count, MinorsSweep* out);
int minors_sweep_launch(const MinorsSweep& s, const double2* dA, void* partials, hipStream_t st);

struct BatchBuffers;  // persistent-batch buffers and captured graphs (batch.hip)

// One execution context: a stream, a device workspace, a pinned staging
// buffer and the batch buffers with their captured graphs.  A host entry point
// leases a context for the whole call (class Lease): callers on different
// threads run on different contexts -- their own streams -- and overlap; a
// context is never used by two calls at once.
struct Engine {
    std::mutex mu;
    int device = -1;        // device of the stream and buffers (-1: none yet)
    hipStream_t stream = nullptr;
    int cus = 0;
    void* dbuf = nullptr;   // device workspace (counter slot at offset 0)
    size_t dbytes = 0;
    void* hbuf = nullptr;   // pinned staging
    size_t hbytes = 0;
    BatchBuffers* batch = nullptr;

    // stream and device binding (first use, or after a device change); lock held
    int ensure_init_locked();
    int ensure_buffers_locked(size_t dneed, size_t hneed);
    int64_t resident_waves_locked(int nc, bool expanded = false) { return resident_waves(nc, expanded); }
    void release_locked();  // stream, buffers and graphs (device change)
};

constexpr int kEngineContexts = 4;
extern Engine g_ctx[kEngineContexts];

// The context of a host call: a free one (the calling thread's own first),
// waiting for the thread's own when all are busy.  Bound to the device and
// with its stream created on construction; status() is the result of that.
class Lease {
  public:
    Lease();
    explicit Lease(Engine& e);  // a given context (replay of its last batch)
    Engine& operator*() const { return *e_; }
    Engine* operator->() const { return e_; }
    int status() const { return st_; }

  private:
    Engine* e_ = nullptr;
    std::unique_lock<std::mutex> lk_;
    int st_ = 0;
};

extern thread_local std::string t_err;

int fail(int code, const std::string& msg);
int hip_fail(hipError_t e, const char* what);
// Waits until the kernel queued on the context's stream last has set *done (host memory,
// zeroed before its launch).
hipError_t wait_result(Engine& E, const unsigned* done);
// hip_fail after waiting for the context's stream: for failures after an upload
// from the staging buffer was queued, so that no copy still reads it when the
// context is released.
int drain_fail(Engine& E, hipError_t e, const char* what);

}  // namespace pqb
