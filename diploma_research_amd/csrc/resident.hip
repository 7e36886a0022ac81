// Conjugate gradients by resident workgroups, for matrices kept by diagonals.
//
// A launch per kernel costs a small system about 6 us, three times an
// iteration, whatever its size. Here one launch of a workgroup per CU runs the
// whole loop. A system is given to a team of workgroups, each
// with its share of the rows: the matrix values (where they fit), x and r stay
// in registers, the direction p in LDS, and an iteration moves through memory
// only the entries of r and p that another workgroup's rows reach.
//
// A team is normally a set of workgroups on one XCD, which meet through that
// XCD's L2, and systems of a solve (right-hand sides, or systems of a batch) run
// side by side on different teams. A system too large for one XCD takes the
// whole chip.
//
// One iteration, with two meetings of the team (reference: textbook CG,
// thesis.tex:2133-2160):
//   1. p = r + beta p for the own rows and for the halo (r of the neighbours,
//      published in step 3, and the halo's p of the iteration before); q = A p;
//      p.q
//   -- meeting: the sum of p.q, alpha
//   2. x += alpha p, r -= alpha q, r.r
//   3. r of the rows that others read goes to memory
//   -- meeting: the sum of r.r, stop test, beta
// Every workgroup computes the halo's p itself, from the same numbers in the
// same way as its owner, and keeps it, so p needs no meeting of its own and does
// not go through memory (with p published beside r: 128^3 cells to 1e-12 16.7
// ms, now 13.9; 256^2 cells 3.30 and 2.94 ms). Only where the registers are full
// (far_in_registers()) a far diagonal's p comes from its owner.
//
// The launch is an ordinary one: a cooperative launch takes a resource that
// only one process on the GPU can hold. Its workgroups first wait until all of
// them are running, and call the launch off, with nothing touched, if that does
// not come about soon; the caller then solves by launch sequence. Two resident
// solves of one process do not run side by side (each would hold CUs that the
// other waits for): one that would have to wait long for another takes the
// launch sequence too.
//
// Measured (one double per workgroup summed over the team and known to all of
// it, block reduction included): 1.1 us for 2 to 32 workgroups of an XCD, 2.4
// us for the chip in two levels.
#include "resident.h"
#include "seating.h"
#include "spmv_impl.h"

#include <algorithm>
#include <chrono>
#include <cmath>

namespace dimgpu {

namespace {

using detail::dpp_val;
using detail::lane_value;

constexpr int kThreads = 512; // 2 wavefronts per SIMD, up to 256 VGPRs each
constexpr int kWaves = kThreads / 64;
constexpr uint32_t kSeatsAll = kResidentXcds * kResidentCus;
constexpr uint32_t kWindowBytes = 150 * 1024;
// more than half a CU's LDS, so that no CU takes two workgroups
constexpr uint32_t kMinLds = 81 * 1024;
// Rows whose loads a thread has in flight together.
constexpr uint32_t chunk_rows(uint32_t rpt) {
    return rpt < 4 ? rpt : 4;
}
// The matrix values stay in registers where they take at most 112 of a
// thread's 256; otherwise every iteration reads them (from the Infinity Cache,
// for systems of this size).
constexpr bool values_resident(uint32_t nd, uint32_t rpt, size_t vb) {
    return nd * rpt * vb / 4 <= 112;
}
// x is touched once an iteration: it goes to LDS when it, r, A p, the values and
// the loads in flight would crowd the registers.
constexpr bool x_in_lds(uint32_t nd, uint32_t rpt, size_t vb) {
    return ((values_resident(nd, rpt, vb) ? rpt : chunk_rows(rpt)) * nd + chunk_rows(rpt) * 4 + 3 * rpt) * vb / 4 > 150;
}
// The direction where far diagonals reach stays in registers if there is room
// beside r, A p, x and the values (spills set in above about these counts);
// otherwise it is read from its owners' memory in every iteration.
constexpr bool far_in_registers(uint32_t nd, uint32_t rpt, size_t vb) {
    const bool res = values_resident(nd, rpt, vb);
    return ((res ? rpt : chunk_rows(rpt)) * nd + (x_in_lds(nd, rpt, vb) ? 4 : 5) * rpt) * vb / 4 <= (res ? 165 : 190);
}
constexpr long long kEmpty = -1; // a slot nobody has written: no sum has these bits

// Meeting slots, counters and the abort word, cleared before every launch.
struct Meeting {
    // [phase & 3][rank] of each XCD; a line of its own for each phase
    double local[kResidentXcds][4][kResidentCus];
    double global[4][kResidentXcds][16]; // one line per XCD sum
    unsigned seated[kResidentXcds * 2][32];
    unsigned total[32];
    int abort[32];
};

template<typename V>
struct Args {
    const V* vals;
    uint64_t ld;
    V *x, *r, *p;
    const ResidentJob* jobs;
    const ResidentSeat* seats;
    uint32_t rounds;
    ResidentState st;
    Meeting* meet;
    uint64_t limit;      // wall-clock ticks a wait may take
    uint64_t seat_limit; // and the wait for all workgroups to be running
    uint32_t need;       // how many that are
};

// What workgroups exchange: a load does not take a line that L1 kept from
// before (device scope). A store to workgroups of the same XCD ends in the L2
// that they share; one to the whole chip (device scope) is written through to
// memory, where every XCD's load finds it, and takes longer: a meeting of 32
// workgroups of an XCD over written-through slots takes 1.9 us instead of 1.1.
template<typename T>
__device__ __forceinline__ T load_shared(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template<typename T>
__device__ __forceinline__ void store_xcd(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template<typename T>
__device__ __forceinline__ void store_chip(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sum over the wavefront, the same bits in every lane
__device__ __forceinline__ double wave_total(double v) {
    v += dpp_val<detail::kDppRowShr1, 0xf>(v);
    v += dpp_val<detail::kDppRowShr2, 0xf>(v);
    v += dpp_val<detail::kDppRowShr4, 0xf>(v);
    v += dpp_val<detail::kDppRowShr8, 0xf>(v);
    v += dpp_val<detail::kDppRowBcast15, 0xa>(v);
    v += dpp_val<detail::kDppRowBcast31, 0xc>(v);
    return lane_value(v, 63);
}

struct Team {
    uint32_t xcd, rank;   // this workgroup's seat
    uint32_t tb, tn, base;
    uint32_t phase;       // meetings so far
};

// The value of a slot once it has been written; false when the wait failed.
__device__ __forceinline__ bool await_slot(const double* slot, const Meeting* m, uint64_t limit, double* out) {
    uint64_t t0 = 0;
    for (uint32_t spin = 0;; ++spin) {
        const double v = load_shared(slot);
        if (__double_as_longlong(v) != kEmpty) {
            *out = v;
            return true;
        }
        if ((spin & 63u) == 63u) {
            const uint64_t t = wall_clock64();
            if (!t0)
                t0 = t;
            if (t - t0 > limit || load_shared(&m->abort[0]))
                return false;
        }
    }
}

// Sum of `v` over the threads of the team in a fixed order, known to all of
// them; everything the team stored before is visible to it after. Four slots
// per seat are used in turn: when a workgroup has read phase n, all have
// written n and so have read n - 1, and it clears its slot of phase n + 2 (last
// used by n - 2) before it writes n + 1, which every reader of n + 2 has seen.
// Returns false (to all threads of the workgroup) when a wait failed.
template<bool WIDE>
__device__ bool meet(Meeting* m, Team& t, uint64_t limit, double v, double* sum) {
    __shared__ double part[kWaves];
    __shared__ double total;
    __shared__ int good;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double s = wave_total(v);
    if (lane == 0)
        part[w] = s;
    // the wavefront's stores have reached the memory that the team shares
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (w == 0) {
        double b = part[0];
#pragma unroll
        for (int i = 1; i < kWaves; ++i)
            b += part[i];
        if (isnan(b))
            b = __longlong_as_double(0x7ff8000000000000ll); // never the bits of an empty slot
        bool ok = true;
        if (WIDE) {
            double* local = m->local[t.xcd][t.phase & 3u];
            double(*global)[16] = m->global[t.phase & 3u];
            if (t.rank == 0) {
                // the XCD's sum
                double u = lane == 0 ? b : 0.0;
                if (lane > 0 && lane < static_cast<int>(kResidentCus))
                    ok = await_slot(local + lane, m, limit, &u);
                const double x = wave_total(u);
                // (without one of its parts there is no sum: the word that
                // ends the other workgroups' waits instead)
                if (__ballot(!ok)) {
                    if (lane == 0)
                        store_chip(&m->abort[0], kResidentTimeout);
                } else if (lane == 0) {
                    store_chip(&global[t.xcd][0], isnan(x) ? __longlong_as_double(0x7ff8000000000000ll) : x);
                }
            } else if (lane == 0) {
                store_xcd(local + t.rank, b);
            }
            double u = 0.0;
            if (lane < static_cast<int>(kResidentXcds))
                ok = ok && await_slot(&global[lane][0], m, limit, &u);
            b = wave_total(u);
            if (lane == 0) {
                const uint32_t next = (t.phase + 2u) & 3u;
                if (t.rank)
                    store_xcd(&m->local[t.xcd][next][t.rank], __longlong_as_double(kEmpty));
                else
                    store_chip(&m->global[next][t.xcd][0], __longlong_as_double(kEmpty));
            }
        } else if (t.tn > 1) {
            double* local = m->local[t.xcd][t.phase & 3u];
            if (lane == 0)
                store_xcd(local + t.rank, b);
            double u = 0.0;
            if (lane < static_cast<int>(t.tn))
                ok = await_slot(local + t.base + lane, m, limit, &u);
            b = wave_total(u);
            if (lane == 0)
                store_xcd(&m->local[t.xcd][(t.phase + 2u) & 3u][t.rank], __longlong_as_double(kEmpty));
        }
        const bool all = __ballot(!ok) == 0ull; // (of all lanes: not below lane 0's branch)
        if (lane == 0) {
            if (!all)
                store_chip(&m->abort[0], kResidentTimeout);
            total = b;
            good = all;
        }
    }
    ++t.phase;
    __syncthreads();
    *sum = total;
    return good != 0;
}

// The iterations of one job on one team; false when a wait failed. FAR: the
// lowest and the highest diagonal may reach past the halo; their entries are
// then read row by row instead of from the window.
//
// A wavefront's rows j * kThreads + 64 * wave + lane, j < nj, cover the
// workgroup's rows up to a multiple of 64. The lanes past the last row of the
// system hold zeros throughout (no values, no r), so nothing in the loop
// depends on the lane except what goes to memory.
template<typename V, int ND, int RPT, bool WIDE, bool FAR>
__device__ bool run_job(const Args<V>& a, uint32_t job, Team& team, V* win) {
    constexpr bool RES = values_resident(ND, RPT, sizeof(V));
    constexpr bool XLDS = x_in_lds(ND, RPT, sizeof(V));
    constexpr bool KEEP = FAR && far_in_registers(ND, RPT, sizeof(V));
    constexpr int CH = chunk_rows(RPT);
    // halo entries per thread in flight together (8 would spill beside the most
    // resident values: 8 FP32-refined columns of 64^3 cells 12.8 ms)
    constexpr int U = RES && RPT == 16 ? 4 : 8;
    const ResidentJob& J = a.jobs[job];
    const uint32_t n = J.rows, H = J.halo;
    const uint32_t first_row = team.tb * J.rb < n ? team.tb * J.rb : 0u;
    const uint32_t rows = team.tb * J.rb < n ? min(J.rb, n - first_row) : 0u;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nj = (static_cast<int>(rows) - 64 * wave + kThreads - 1) / kThreads; // <= 0: none
    V* R = a.r + J.vec0;
    V* P = a.p + J.vec0;
    V* X = a.x + J.vec0 + first_row;
    const V* vals = a.vals + J.row0 + first_row;
    const uint32_t far = FAR ? J.far : 0u;
    const bool far_lo = (far & 1u) != 0;
    const int d_hi = far & ~1u ? 31 - __builtin_clz(far) : ND; // the far diagonal above, or none
    int off[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
        off[d] = J.off[d];
    int o_hi = 0;
#pragma unroll
    for (int d = 1; d < ND; ++d)
        o_hi = d == d_hi ? off[d] : o_hi;

    double rr = a.st.rr[job];
    int it = a.st.run[job];
    const double tol2 = a.st.tol2[job];
    const double pause = a.st.pause ? a.st.pause[job] : -1.0;

    V* xs = win + (RPT * kThreads + 2 * H); // x, where it lives in LDS
    V x[XLDS ? 1 : RPT], r[RPT], v[RES ? RPT : 1][ND];
    V flo[KEEP ? RPT : 1], fhi[KEEP ? RPT : 1]; // p where the far diagonals reach
    for (uint32_t h = threadIdx.x; h < RPT * kThreads + 2 * H; h += kThreads)
        win[h] = V(0);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const uint32_t l = j * kThreads + threadIdx.x;
        const bool in = l < rows;
        const V xj = in ? X[l] : V(0);
        if constexpr (XLDS)
            xs[l] = xj;
        else
            x[j] = xj;
        r[j] = in ? R[first_row + l] : V(0);
        if (in)
            win[H + l] = P[first_row + l];
        if constexpr (RES) {
#pragma unroll
            for (int d = 0; d < ND; ++d)
                v[j][d] = in ? vals[d * a.ld + l] : V(0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();

    V beta = V(1);
    bool fresh = true; // p is given, not r + beta p
    int status = 0;
    bool ok = true;
    for (;;) {
        // The loop's first line of instructions is a whole one, wherever the code
        // before it ends (8 FP32-refined columns of 64^3 cells: 10.8 ms, and 11.15
        // with an end that does not suit).
        asm volatile(".p2align 6");
        // (opaque, so that the many addresses made from it are made anew in
        // every iteration instead of being kept in registers throughout)
        uint32_t tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        // ---- p of the own rows and of the halo
        if (!fresh) {
#pragma unroll
            for (int j = 0; j < RPT; ++j)
                if (j < nj) {
                    V* w = win + (H + tid);
                    w[j * kThreads] = r[j] + beta * w[j * kThreads];
                }
        }
        if (team.tn > 1 && H) {
            for (uint32_t u0 = 0; u0 < 2 * H; u0 += U * kThreads) {
                V hr[U];
                // entry h of the halo is row first_row - H + h, past the own
                // rows from h = H on
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int h = static_cast<int>(u0 + u * kThreads + tid);
                    const int row = static_cast<int>(first_row) + h + (h < static_cast<int>(H) ? -static_cast<int>(H) : static_cast<int>(rows) - static_cast<int>(H));
                    const uint32_t at = static_cast<uint32_t>(max(0, min(row, static_cast<int>(n) - 1)));
                    hr[u] = load_shared((fresh ? P : R) + at);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const uint32_t h = u0 + u * kThreads + tid;
                    const int row = static_cast<int>(first_row + h) + (h < H ? -static_cast<int>(H) : static_cast<int>(rows) - static_cast<int>(H));
                    if (h < 2 * H) {
                        V* w = win + (h < H ? h : rows + h);
                        const V pv = fresh ? hr[u] : hr[u] + beta * *w;
                        *w = row >= 0 && row < static_cast<int>(n) ? pv : V(0);
                    }
                }
            }
        }
        __syncthreads();

        // ---- q = A p, p.q
        V q[RPT];
        double acc = 0.0;
#pragma unroll
        for (int c = 0; c < RPT; c += CH) {
            __builtin_amdgcn_sched_barrier(0); // (one chunk's loads at a time)
            if (c < nj) {
                V plo[CH], phi[CH];
                if constexpr (FAR) {
                    const V* from = fresh ? P : R;
                    V qlo[KEEP ? 1 : CH], qhi[KEEP ? 1 : CH];
#pragma unroll
                    for (int j = 0; j < CH; ++j) {
                        const int row = static_cast<int>(first_row + (c + j) * kThreads + tid);
                        const int lo = max(0, min(row + off[0], static_cast<int>(n) - 1));
                        const int hi = max(0, min(row + o_hi, static_cast<int>(n) - 1));
                        plo[j] = load_shared(from + lo);
                        phi[j] = load_shared(from + hi);
                        if constexpr (!KEEP) {
                            qlo[j] = load_shared(P + lo);
                            qhi[j] = load_shared(P + hi);
                        }
                    }
#pragma unroll
                    for (int j = 0; j < CH; ++j) {
                        if constexpr (KEEP) {
                            plo[j] = fresh ? plo[j] : plo[j] + beta * flo[c + j];
                            phi[j] = fresh ? phi[j] : phi[j] + beta * fhi[c + j];
                            flo[c + j] = plo[j];
                            fhi[c + j] = phi[j];
                        } else {
                            plo[j] = fresh ? plo[j] : plo[j] + beta * qlo[j];
                            phi[j] = fresh ? phi[j] : phi[j] + beta * qhi[j];
                        }
                    }
                }
                V vc[CH][ND];
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    // (rows past the workgroup's: any row of the matrix)
                    const uint32_t l = c + j < nj ? (c + j) * kThreads + tid : tid & 63u;
#pragma unroll
                    for (int d = 0; d < ND; ++d) {
                        if constexpr (RES)
                            vc[j][d] = v[c + j][d];
                        else
                            vc[j][d] = vals[d * a.ld + l];
                    }
                }
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    V s = V(0);
#pragma unroll
                    for (int d = 0; d < ND; ++d) {
                        int o = off[d];
                        if constexpr (FAR) // (the window is not asked for what lies past it)
                            o = (d == 0 && far_lo) || d == d_hi ? 0 : o;
                        V pv = (win + (static_cast<int>(H + tid) + o))[(c + j) * kThreads];
                        if constexpr (FAR) {
                            if (d == 0)
                                pv = far_lo ? plo[j] : pv;
                            else
                                pv = d == d_hi ? phi[j] : pv;
                        }
                        s = fma(vc[j][d], pv, s);
                    }
                    q[c + j] = s;
                    if (c + j < nj)
                        acc += static_cast<double>(win[H + (c + j) * kThreads + tid]) * static_cast<double>(s);
                }
            }
        }
        double pq;
        ok = meet<WIDE>(a.meet, team, a.limit, acc, &pq);
        if (!ok)
            break;

        // ---- alpha, x, r, r.r; what other workgroups read goes to memory
        const double step = rr / pq;
        const bool broke = !(pq > 0.0) || !std::isfinite(step);
        const V alpha = broke ? V(0) : static_cast<V>(step);
        acc = 0.0;
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            if (j < nj) {
                const uint32_t l = j * kThreads + tid;
                const V pj = win[H + l];
                if constexpr (XLDS)
                    xs[l] = xs[l] + alpha * pj;
                else
                    x[j] = x[j] + alpha * pj;
                const V rj = r[j] - alpha * q[j];
                r[j] = rj;
                acc += static_cast<double>(rj) * static_cast<double>(rj);
                // (far diagonals are read from memory within a workgroup's
                // own rows too: a team may be one workgroup)
                if (l < rows && (FAR || (team.tn > 1 && (l < H || l + H >= rows)))) {
                    if constexpr (WIDE)
                        store_chip(R + first_row + l, rj);
                    else
                        store_xcd(R + first_row + l, rj);
                    if constexpr (FAR && !KEEP) {
                        if constexpr (WIDE)
                            store_chip(P + first_row + l, pj);
                        else
                            store_xcd(P + first_row + l, pj);
                    }
                }
            }
        }
        double rn;
        ok = meet<WIDE>(a.meet, team, a.limit, acc, &rn);
        if (!ok)
            break;
        ++it;
        if (a.st.hist && job == 0 && team.tb == 0 && tid == 0 && it < a.st.hist_cap) {
            const double scale = a.st.bnorm[job] > 0.0 ? a.st.bnorm[job] : 1.0;
            a.st.hist[it] = std::sqrt(rn) / scale;
        }
        beta = static_cast<V>(rn / rr);
        rr = rn;
        fresh = false;
        status = broke ? 2 : (rn <= tol2 ? 1 : 0);
        if (status || it >= a.st.max_iters || rn < pause)
            break;
    }
    if (!ok)
        return false;
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const uint32_t l = j * kThreads + threadIdx.x;
        if (l < rows) {
            if constexpr (XLDS)
                X[l] = xs[l];
            else
                X[l] = x[j];
            // a solve that goes on from here starts with the next direction
            if (!status)
                P[first_row + l] = r[j] + beta * win[H + l];
        }
    }
    if (team.tb == 0 && threadIdx.x == 0) {
        a.st.rr[job] = rr;
        a.st.run[job] = it;
        a.st.done[job] = status;
        a.st.iters[job] = status == 2 ? it - 1 : it;
    }
    return true;
}

template<typename V, int ND, int RPT, bool WIDE>
__global__ __launch_bounds__(kThreads) void k_resident(Args<V> a) {
    extern __shared__ char lds[];
    __shared__ unsigned xcd_s, rank_s;
    __shared__ int state_s;
    // take a seat: this workgroup's XCD and its rank there
    if (threadIdx.x == 0) {
        const unsigned x = __builtin_amdgcn_s_getreg(20 | (3 << 11)) & 15u; // XCC_ID
        xcd_s = x;
        rank_s = __hip_atomic_fetch_add(&a.meet->seated[x][0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __hip_atomic_fetch_add(&a.meet->total[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // All workgroups are running when the count is complete; from then on
        // every wait ends. One that has waited too long for the others (CUs
        // held by another program) calls the launch off.
        struct {
            unsigned* p;
            __device__ unsigned load() { return load_shared(p); }
            __device__ bool replace(unsigned from, unsigned to) {
                return __hip_atomic_compare_exchange_strong(p, &from, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT);
            }
        } count{&a.meet->total[0]};
        const uint64_t t0 = wall_clock64();
        Seats seats = Seats::kWaiting;
        for (;;) {
            seats = look_at_seats(count, a.need, wall_clock64() - t0 > a.seat_limit);
            if (seats != Seats::kWaiting)
                break;
            __builtin_amdgcn_s_sleep(1);
        }
        int state = seats == Seats::kComplete ? 0 : kResidentSeats;
        if (!state)
            for (uint32_t i = 0; i < kResidentXcds; ++i)
                if (load_shared(&a.meet->seated[i][0]) != kResidentCus)
                    state = kResidentSeats;
        if (state)
            store_chip(&a.meet->abort[0], state);
        state_s = state;
    }
    __syncthreads();
    if (state_s)
        return;
    const uint32_t xcd = __builtin_amdgcn_readfirstlane(xcd_s), rank = __builtin_amdgcn_readfirstlane(rank_s);
    Team team{xcd, rank, 0, 0, 0, 0};
    for (uint32_t round = 0; round < a.rounds; ++round) {
        const ResidentSeat s = a.seats[round * kSeatsAll + xcd * kResidentCus + rank];
        if (s.job == kNoJob)
            continue;
        team.tb = __builtin_amdgcn_readfirstlane(s.tb);
        team.tn = __builtin_amdgcn_readfirstlane(s.tn);
        team.base = __builtin_amdgcn_readfirstlane(s.base);
        const uint32_t job = __builtin_amdgcn_readfirstlane(s.job);
        // no team member has written this before all have read it: the
        // first meeting lies in between
        if (a.st.done[job] || a.st.run[job] >= a.st.max_iters)
            continue;
        V* win = reinterpret_cast<V*>(lds);
        const bool ok = a.jobs[job].far ? run_job<V, ND, RPT, WIDE, true>(a, job, team, win)
                                        : run_job<V, ND, RPT, WIDE, false>(a, job, team, win);
        if (!ok)
            return;
        __syncthreads(); // the window belongs to the next job
    }
}

// Empties the meeting slots and zeroes the counters.
__global__ void k_clear(Meeting* m) {
    double* slots = &m->local[0][0][0];
    constexpr size_t n = (sizeof(m->local) + sizeof(m->global)) / sizeof(double);
    for (size_t i = threadIdx.x; i < n; i += blockDim.x)
        slots[i] = __longlong_as_double(kEmpty);
    unsigned* c = &m->seated[0][0];
    constexpr size_t k = (sizeof(m->seated) + sizeof(m->total) + sizeof(m->abort)) / sizeof(unsigned);
    for (size_t i = threadIdx.x; i < k; i += blockDim.x)
        c[i] = 0u;
}

constexpr size_t up256(size_t b) {
    return (b + 255) / 256 * 256;
}

template<typename V, int ND, int RPT, bool WIDE>
hipError_t launch(const Args<V>& args, uint32_t lds, hipStream_t s) {
    Args<V> a = args;
    const void* f = reinterpret_cast<const void*>(&k_resident<V, ND, RPT, WIDE>);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess)
        return e;
    void* p[] = {&a};
    return hipLaunchKernel(f, dim3(kSeatsAll), dim3(kThreads), p, lds, s);
}

template<typename V, int ND, bool WIDE>
hipError_t launch_rpt(uint32_t rpt, const Args<V>& a, uint32_t lds, hipStream_t s) {
    switch (rpt) {
        case 2: return launch<V, ND, 2, WIDE>(a, lds, s);
        case 4: return launch<V, ND, 4, WIDE>(a, lds, s);
        case 8: return launch<V, ND, 8, WIDE>(a, lds, s);
        case 16: return launch<V, ND, 16, WIDE>(a, lds, s);
        default: return hipErrorInvalidValue;
    }
}

template<typename V>
hipError_t launch_nd(const ResidentPlan& p, const Args<V>& a, hipStream_t s) {
    const uint32_t lds = std::max(p.lds, kMinLds);
    switch (p.nd) {
#define DIM_RESIDENT_CASE(ND)                                                                                         \
    case ND:                                                                                                          \
        return p.wide ? launch_rpt<V, ND, true>(p.rpt, a, lds, s) : launch_rpt<V, ND, false>(p.rpt, a, lds, s);
        DIM_RESIDENT_CASE(3)
        DIM_RESIDENT_CASE(5)
        DIM_RESIDENT_CASE(7)
        DIM_RESIDENT_CASE(9)
#undef DIM_RESIDENT_CASE
        default: return hipErrorInvalidValue;
    }
}

template<typename V>
hipError_t run(const ResidentPlan& p, const void* vals, uint64_t ld, void* x, void* r, void* pv,
               const ResidentState& st, const ResidentWaits& waits, char* work, hipStream_t s) {
    int dev = 0, khz = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess)
        e = hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev);
    if (e != hipSuccess)
        return e;
    Args<V> a;
    a.vals = static_cast<const V*>(vals);
    a.ld = ld;
    a.x = static_cast<V*>(x);
    a.r = static_cast<V*>(r);
    a.p = static_cast<V*>(pv);
    a.meet = reinterpret_cast<Meeting*>(work);
    a.jobs = reinterpret_cast<const ResidentJob*>(work + up256(sizeof(Meeting)));
    a.seats = reinterpret_cast<const ResidentSeat*>(work + up256(sizeof(Meeting)) +
                                                    up256(p.jobs.size() * sizeof(ResidentJob)));
    a.rounds = p.rounds;
    a.st = st;
    const double second = std::max(khz, 1) * 1e3;
    a.limit = static_cast<uint64_t>(waits.wait_seconds * second);
    a.seat_limit = static_cast<uint64_t>(waits.seat_seconds * second);
    a.need = waits.need;
    hipLaunchKernelGGL(k_clear, dim3(1), dim3(1024), 0, s, a.meet);
    return launch_nd<V>(p, a, s);
}

} // namespace

std::unique_lock<std::timed_mutex> resident_lock() {
    static std::timed_mutex per_device[64];
    int dev = 0;
    (void)hipGetDevice(&dev);
    return std::unique_lock<std::timed_mutex>(per_device[dev & 63], std::chrono::duration<double>(kResidentPatience));
}

bool resident_device() {
    return detail::device_cus() == static_cast<int>(kSeatsAll);
}

namespace {

// LDS of a workgroup: p of its rows and their halo, and x where it lives there.
size_t window_bytes(uint32_t nd, uint32_t rpt, uint64_t halo, size_t vb) {
    return (size_t{rpt} * kThreads * (x_in_lds(nd, rpt, vb) ? 2 : 1) + 2 * halo) * vb;
}

// Rows per workgroup, halo and far diagonals of a job on a team of at most tn
// workgroups, each with room for rpt * kThreads rows. Returns how many of them
// have rows; 0 when the kernel does not take such a job.
uint32_t fit_job(ResidentJob& j, uint32_t nd, uint32_t tn, uint32_t rpt, size_t vb) {
    j.rb = static_cast<uint32_t>(((uint64_t{j.rows} + tn - 1) / tn + 63) / 64 * 64);
    j.halo = 0;
    j.far = 0;
    for (uint32_t d = 0; d < nd; ++d) {
        const uint64_t o = static_cast<uint64_t>(std::abs(static_cast<int64_t>(j.off[d])));
        if (o >= j.rows)
            j.off[d] = 0; // no element of the system lies there
        else if (o < j.rb && window_bytes(nd, rpt, o, vb) <= kWindowBytes)
            j.halo = std::max(j.halo, static_cast<uint32_t>(o));
        else
            j.far |= 1u << d;
    }
    // only the lowest diagonal and one above may be far
    const uint32_t above = j.far & ~1u;
    if (above & (above - 1))
        return 0;
    return (j.rows + j.rb - 1) / j.rb; // workgroups with rows
}

} // namespace

// When systems take turns, one after another on an XCD's 32 workgroups, an
// iteration of them all takes about the first sum on the XCD with the most,
// and in the launch sequence, all systems side by side, the second. The plan is
// refused where the second is smaller. Measured (5 diagonals, FP64, microseconds
// an iteration, turns and launch sequence): 272 systems of 500 rows 97 and 34;
// 192 of 4200 rows 65 and 51, 1024 of them 347 and 194; 96 of 16250 rows 36 and
// 56; 96 of 62400 rows 43 and 154. The sums are within a third of these and on
// the right side in all of 35 such pairs.
constexpr double kTurnMicros = 2.7, kTurnRowMicros = 1.5e-5;
constexpr double kSequenceMicros = 11.0, kSequenceJobMicros = 0.04, kSequenceRowMicros = 2.75e-5;

ResidentPlan plan_resident(std::vector<ResidentJob> jobs, uint32_t nd, size_t vb) {
    ResidentPlan p;
    p.nd = nd;
    if (jobs.empty() || jobs.size() >= kNoJob || !resident_device())
        return p;
    for (const ResidentJob& j : jobs)
        if (!j.rows || j.rows > (1u << 30))
            return p;
    constexpr uint32_t kMaxRpt = 16;
    const uint32_t block_rows = kMaxRpt * kThreads;
    // rows per workgroup that still keep the values in registers
    uint32_t res_rpt = 2;
    while (res_rpt < kMaxRpt && values_resident(nd, res_rpt * 2, vb))
        res_rpt *= 2;
    const uint64_t xcd_rows = uint64_t{res_rpt} * kThreads * kResidentCus;
    uint32_t widest = 0; // rows per workgroup of the fullest team
    const auto seat = [&](uint32_t round, uint32_t xcd, uint32_t rank) -> ResidentSeat& {
        return p.seats[(size_t{round} * kResidentXcds + xcd) * kResidentCus + rank];
    };
    const auto finish = [&](bool wide) {
        p.wide = wide;
        p.rpt = 2;
        while (p.rpt * kThreads < widest)
            p.rpt *= 2;
        for (const ResidentJob& j : jobs)
            p.lds = std::max(p.lds, static_cast<uint32_t>(window_bytes(nd, p.rpt, j.halo, vb)));
        p.jobs = std::move(jobs);
        p.ok = true;
    };
    const bool one_xcd = std::all_of(jobs.begin(), jobs.end(), [&](const ResidentJob& j) { return j.rows <= xcd_rows; });
    if (!one_xcd) {
        // one system over the whole chip
        if (jobs.size() != 1 || jobs[0].rows > uint64_t{block_rows} * kSeatsAll)
            return p;
        p.rounds = 1;
        p.seats.assign(kSeatsAll, ResidentSeat{0, 0, kSeatsAll, 0});
        widest = static_cast<uint32_t>(((uint64_t{jobs[0].rows} + kSeatsAll - 1) / kSeatsAll + 63) / 64 * 64);
        uint32_t rpt = 2;
        while (rpt * kThreads < widest)
            rpt *= 2;
        if (!fit_job(jobs[0], nd, kSeatsAll, rpt, vb))
            return p;
        for (uint32_t i = 0; i < kSeatsAll; ++i)
            p.seats[i].tb = static_cast<uint16_t>(i); // every workgroup meets, with rows or without
        finish(true);
        return p;
    }
    // systems to XCDs: the largest first, each to the XCD with the fewest rows
    std::vector<uint32_t> order(jobs.size());
    for (uint32_t i = 0; i < order.size(); ++i)
        order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return jobs[a].rows > jobs[b].rows; });
    std::vector<std::vector<uint32_t>> of(kResidentXcds);
    std::vector<uint64_t> load(kResidentXcds, 0);
    for (uint32_t i : order) {
        const uint32_t x = static_cast<uint32_t>(std::min_element(load.begin(), load.end()) - load.begin());
        of[x].push_back(i);
        load[x] += jobs[i].rows;
    }
    // an XCD whose systems fit side by side (every one with its values in
    // registers) shares its workgroups out by rows; otherwise they take turns,
    // each on all of them
    struct Share {
        std::vector<uint32_t> tn;
        bool turns = false;
    };
    std::vector<Share> shares(kResidentXcds);
    const uint64_t res_rows = uint64_t{res_rpt} * kThreads;
    for (uint32_t x = 0; x < kResidentXcds; ++x) {
        Share& s = shares[x];
        uint64_t need = 0;
        for (uint32_t i : of[x]) {
            s.tn.push_back(static_cast<uint32_t>((jobs[i].rows + res_rows - 1) / res_rows));
            need += s.tn.back();
        }
        if (need > kResidentCus) {
            s.turns = true;
            s.tn.assign(of[x].size(), kResidentCus);
            continue;
        }
        // the spare workgroups one by one to the team with the most rows each,
        // while that is over kTeamRows: a meeting of a few workgroups costs
        // little more than a workgroup's own reduction. 256^2 cells, 5
        // diagonals: 3.9 us an iteration at 2048 rows per workgroup, 4.9 at
        // 4096; 128^2: 3.2 at 1024 (and at 512), 3.8 at 2048.
        constexpr uint32_t kTeamRows = 1024;
        while (need < kResidentCus) {
            size_t best = s.tn.size();
            uint64_t most = kTeamRows;
            for (size_t q = 0; q < s.tn.size(); ++q) {
                const uint64_t each = jobs[of[x][q]].rows / s.tn[q];
                if (each > most) {
                    most = each;
                    best = q;
                }
            }
            if (best == s.tn.size())
                break;
            ++s.tn[best];
            ++need;
        }
    }
    p.rounds = 1;
    double turns_us = 0.0; // an iteration of everything on the XCD with the longest turns
    for (uint32_t x = 0; x < kResidentXcds; ++x)
        if (shares[x].turns) {
            p.rounds = std::max(p.rounds, static_cast<uint32_t>(of[x].size()));
            double us = 0.0;
            for (uint32_t i : of[x])
                us += kTurnMicros + kTurnRowMicros * jobs[i].rows;
            turns_us = std::max(turns_us, us);
        }
    uint64_t all_rows = 0;
    for (const ResidentJob& j : jobs)
        all_rows += j.rows;
    if (turns_us > kSequenceMicros + kSequenceJobMicros * jobs.size() + kSequenceRowMicros * all_rows)
        return p;
    p.seats.assign(size_t{p.rounds} * kSeatsAll, ResidentSeat{kNoJob, 0, 0, 0});
    // rows per thread first: the window's room for a halo depends on it
    for (uint32_t x = 0; x < kResidentXcds; ++x)
        for (size_t q = 0; q < of[x].size(); ++q) {
            const uint32_t rows = jobs[of[x][q]].rows, tn = shares[x].tn[q];
            widest = std::max(widest, static_cast<uint32_t>(((uint64_t{rows} + tn - 1) / tn + 63) / 64 * 64));
        }
    uint32_t rpt = 2;
    while (rpt * kThreads < widest)
        rpt *= 2;
    for (uint32_t x = 0; x < kResidentXcds; ++x) {
        uint32_t base = 0;
        for (size_t q = 0; q < of[x].size(); ++q) {
            const uint32_t i = of[x][q];
            const uint32_t tn = fit_job(jobs[i], nd, shares[x].tn[q], rpt, vb);
            if (!tn)
                return p;
            const uint32_t round = shares[x].turns ? static_cast<uint32_t>(q) : 0u;
            for (uint32_t b = 0; b < (shares[x].turns ? kResidentCus : tn); ++b) {
                // (teams that take turns keep all their workgroups, so that the
                // meeting slots stay in step)
                ResidentSeat& s = seat(round, x, base + b);
                s.job = static_cast<uint16_t>(i);
                s.tb = static_cast<uint16_t>(b);
                s.tn = static_cast<uint16_t>(shares[x].turns ? kResidentCus : tn);
                s.base = static_cast<uint16_t>(base);
            }
            if (!shares[x].turns)
                base += tn;
        }
    }
    finish(false);
    return p;
}

size_t resident_bytes(const ResidentPlan& p) {
    return up256(sizeof(Meeting)) + up256(p.jobs.size() * sizeof(ResidentJob)) +
           up256(p.seats.size() * sizeof(ResidentSeat));
}

hipError_t launch_resident(const ResidentPlan& p, bool f32, const void* vals, uint64_t ld, void* x, void* r, void* p_vec,
                           const ResidentState& st, const ResidentWaits& waits, void* work, bool upload,
                           hipStream_t stream) {
    if (!p.ok)
        return hipErrorInvalidValue;
    char* w = static_cast<char*>(work);
    if (upload || waits.absent) {
        const size_t at = up256(sizeof(Meeting));
        hipError_t e = hipMemcpyAsync(w + at, p.jobs.data(), p.jobs.size() * sizeof(ResidentJob),
                                      hipMemcpyHostToDevice, stream);
        std::vector<ResidentSeat> seats;
        if (waits.absent) {
            seats = p.seats;
            for (ResidentSeat& s : seats)
                if (s.job != kNoJob && s.tb && s.tb == s.tn - 1) {
                    s.job = kNoJob;
                    break;
                }
        }
        if (e == hipSuccess)
            e = hipMemcpyAsync(w + at + up256(p.jobs.size() * sizeof(ResidentJob)),
                               waits.absent ? seats.data() : p.seats.data(), p.seats.size() * sizeof(ResidentSeat),
                               hipMemcpyHostToDevice, stream);
        if (e == hipSuccess && waits.absent)
            e = hipStreamSynchronize(stream);
        if (e != hipSuccess)
            return e;
    }
    return f32 ? run<float>(p, vals, ld, x, r, p_vec, st, waits, w, stream)
               : run<double>(p, vals, ld, x, r, p_vec, st, waits, w, stream);
}

hipError_t resident_abort(const void* work, int* code, hipStream_t stream) {
    const Meeting* m = static_cast<const Meeting*>(work);
    return hipMemcpyAsync(code, &m->abort[0], sizeof(int), hipMemcpyDeviceToHost, stream);
}

} // namespace dimgpu
