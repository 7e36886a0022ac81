// Conjugate gradients of matrices kept by diagonals, run by resident
// workgroups (resident.hip).
#pragma once

#include "dia.h"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <vector>

namespace dimgpu {

// One system of a solve: a right-hand side of a matrix, or a system of a batch.
struct ResidentJob {
    uint32_t row0;    // its first row in the diagonal form
    uint32_t rows;
    uint64_t vec0;    // its first entry in r, p and x
    uint32_t rb;      // rows per workgroup of its team (a multiple of 64)
    uint32_t halo;    // entries of the direction a workgroup keeps on each side of its rows
    uint32_t far;     // bit d: diagonal d reaches past the halo
    int32_t off[kDiaMax];
};

// What one workgroup does in one round: workgroup tb of the tn that work on
// `job`; the team's first workgroup has rank `base` on its XCD.
struct ResidentSeat {
    uint16_t job, tb, tn, base; // job kNoJob: idle
};
constexpr uint16_t kNoJob = 0xffff;

// Per-system state, in device memory; entry j belongs to job j.
struct ResidentState {
    const double* tol2 = nullptr;  // stop when r.r <= tol2
    const double* bnorm = nullptr; // for the history
    const double* pause = nullptr; // return when r.r < pause (may be null)
    double* rr = nullptr;          // r.r, in and out
    int* done = nullptr;           // 0 running, 1 converged, 2 breakdown; in and out
    int* iters = nullptr;          // iterations at the stop
    int* run = nullptr;            // iterations so far, in and out
    int max_iters = 0;
    double* hist = nullptr;        // job 0's relative residuals (may be null)
    int hist_cap = 0;
};

constexpr uint32_t kResidentXcds = 8;
constexpr uint32_t kResidentCus = 32; // workgroups (one per CU) of an XCD
// The largest system: 8192 rows per CU of the whole chip, and only as the one
// job of a solve. Several jobs have an XCD each at most, with the values in
// registers: 131072 rows (FP64, 5 or 7 diagonals; 3: 262144, 9: 65536; FP32:
// 262144, 9 diagonals 131072), or the launch sequence takes them all.
constexpr uint32_t kResidentRows = 1u << 21;

// How long a solve waits for the chip, first for another solve of the process
// and then for its own workgroups to be running (CUs held by other streams or
// processes), before it takes the launch sequence. Between the two a small
// system loses 3 to 14 ms (256^2 cells: 2.9 ms here, 16.7 there), so a longer
// wait costs more than it can save.
constexpr double kResidentPatience = 0.01;

// How long the workgroups of a launch wait for one another.
struct ResidentWaits {
    uint32_t need = kResidentXcds * kResidentCus; // workgroups that must be running
    double seat_seconds = kResidentPatience; // for all of them to be running
    double wait_seconds = 10.0; // for a sum of a meeting (they take microseconds)
    bool absent = false; // for tests: one workgroup of a team stays away from its meetings
};

// The tests' hold on a handle's resident launches (dim_test_resident): the
// launches from number `from` on fail as `fault` says.
struct ResidentTrial {
    enum Fault : uint32_t { kNone, kNeverSeated, kWaitsFail };
    uint32_t fault = kNone, from = 0;
    uint32_t launches = 0; // since it was set
    uint32_t ran = 0;      // of those, launches that iterated

    ResidentWaits next() {
        ResidentWaits w;
        if (launches++ >= from) {
            if (fault == kNeverSeated)
                ++w.need; // a workgroup more than there are
            if (fault == kWaitsFail) {
                w.absent = true;
                w.wait_seconds = 1e-3;
            }
        }
        return w;
    }
};

// How a set of systems is shared out.
struct ResidentPlan {
    bool ok = false;
    bool wide = false;      // one system over the whole chip
    uint32_t nd = 0;
    uint32_t rpt = 0;       // rows per thread
    uint32_t rounds = 0;
    uint32_t lds = 0;       // bytes of the largest window
    std::vector<ResidentJob> jobs;
    std::vector<ResidentSeat> seats; // rounds * 256, by XCD and rank
};

// Whether the resident solver exists for this device.
bool resident_device();

// Held (per device) from launch_resident() until the launch has ended. The
// stream must be idle when it is taken, so that nothing a holder waits for can
// depend on another thread's solve. Empty when the other solves take longer
// than kResidentPatience.
std::unique_lock<std::timed_mutex> resident_lock();

// The plan for `jobs` (row0, rows, vec0 and off filled in) with nd diagonals
// and values of vb bytes; !ok when they do not fit.
ResidentPlan plan_resident(std::vector<ResidentJob> jobs, uint32_t nd, size_t vb);

// Device memory a solve needs besides its vectors and state.
size_t resident_bytes(const ResidentPlan& p);

// Runs the iterations of every job until it stops or pauses. work:
// resident_bytes(p) bytes on a 256-byte boundary; upload: copy the plan into it
// first (a plan already there may be reused; one with an absent workgroup is
// always copied and none to be reused). *abort (in work) is set when the
// workgroups could not be seated or a wait timed out; resident_abort() reads
// it back after the launch.
hipError_t launch_resident(const ResidentPlan& p, bool f32, const void* vals, uint64_t ld, void* x, void* r, void* p_vec,
                           const ResidentState& st, const ResidentWaits& waits, void* work, bool upload,
                           hipStream_t stream);
constexpr int kResidentTimeout = 1; // a wait between workgroups passed its limit
constexpr int kResidentSeats = 2;   // not all workgroups running, or not 32 to an XCD; nothing was touched
hipError_t resident_abort(const void* work, int* code, hipStream_t stream);

} // namespace dimgpu
