// resident_dev.hpp -- what the kernels of resident.hip and resident_large.hip
// share: the waits between workgroups, the kernel arguments and the loop head.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "krylov_dev.hpp"
#include "resident.hpp"
#include "wave_dpp.hpp"

namespace mtl4g {

constexpr int kResBS = 512;                  // 8 waves per workgroup, 256 registers per lane
constexpr int kResMaxGrid = 256;             // one workgroup per CU
constexpr int kResHalo = 1024;               // diagonals this close are read from LDS, others from memory
constexpr unsigned kResMeet = 100000;        // rendezvous: 1 ms of the 100 MHz clock
constexpr unsigned kResPolls = 1u << 22;     // polls of a later wait before it gives up

// ------------------------------------------------------------------ waits between workgroups
// Sums: kSlotGens generations of slots, each slot holding a pending pattern
// until the workgroup's sum of that generation is stored.  A workgroup that has
// passed generation g knows that all have passed g - 1 and resets its slots of
// it, which are generation g + 3's.  That reset has to be seen before anyone
// polls g + 3: whoever polls it has passed g + 2, for which every workgroup has
// published, and between a workgroup's reset and its publishing of g + 2 lies a
// res_exchange (one before every even generation), whose wait_memory completes
// the reset.  With three generations a reset behind an even one met its next
// reader with no wait between.  Up to kResFlat workgroups every one publishes to
// eight copies of a slot row (one per blockIdx % 8, so 1/8 of the readers
// poll the same lines) and sums the row itself; more meet in eight groups
// first.  Measured per all-reduce: 1.9 us (32 workgroups), 2.0 (64), 2.5
// (128), 3.3 (256) flat; 2.6-2.8 in groups.
constexpr int kResFlat = 128;
constexpr uint64_t kResPending = 0x7ff5c3c3c3c3c3c3ull;   // signalling NaN: no sum ever is
constexpr int kSlotRow = 2 * kResMaxGrid;                  // two sums per workgroup
constexpr int kSlotGen = 8 * kSlotRow;                     // eight copies
constexpr int kSlotGens = 4;                               // a power of two
// words: rendezvous arrivals (or the ticket of the single steps) and state, abort
// flag, each in a 128-byte line, then one p flag per workgroup.  With the flags 128
// bytes further on a solve on a 70,001-row graph took 423 us instead of 413: their
// place among the memory channels counts.
enum { RW_ARRIVE = 0, RW_TICKET = 16, RW_STATE = 32, RW_ABORT = 64, RW_FLAG = 96 };
enum { RS_OPEN = 0, RS_MET = 1, RS_REFUSED = 2 };   // rendezvous state
constexpr int kResWords = RW_FLAG + kResMaxGrid;

__device__ __forceinline__ bool res_pending(double v) { return (uint64_t)__double_as_longlong(v) == kResPending; }

struct ResSync {
    double* slots;     // kSlotGens * kSlotGen
    unsigned* words;   // kResWords
    int grid;
    unsigned polls;    // kResPolls
};

// Two neighbouring values polled until both are there; false when the wait
// expired or another workgroup has given up.
__device__ __forceinline__ bool res_poll2(const double* p, unsigned* abort, unsigned polls, double& a, double& b) {
    a = ld_agent(p);
    b = ld_agent(p + 1);
    unsigned it = 0;
#pragma clang loop unroll(disable)
    while (res_pending(a) || res_pending(b)) {
        if ((++it & 255u) == 0 && ld_agent(abort) != 0u) return false;
        if (it > polls) {
            st_agent(abort, 1u);
            return false;
        }
        a = ld_agent(p);
        b = ld_agent(p + 1);
    }
    return true;
}

// Sums of two values over the whole grid, in a fixed order, known to every
// lane on return.  a, b: this lane's partial sums; sh: 4 * kResNW values, used
// by turns (gen % 2), so no barrier is needed behind the last read.  Returns
// false when a wait expired.
constexpr int kResNW = kResBS / kWave;
static_assert(kResNW == 8, "the waves' sums of both values fill one row of 16 lanes");
template <typename VT>
struct ResShared {
    VT part[2][2 * kResNW];
    VT tot[2][2];
    int ok[2];
};
template <typename VT, bool ONE>
__device__ __forceinline__ bool res_allsum(const ResSync& S, int gen, VT a, VT b, ResShared<VT>& sh, VT& ta, VT& tb) {
    const int l = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave, h = gen & 1;
    a = res_wave(a);
    b = res_wave(b);
    if (l == 0) {
        sh.part[h][w] = a;
        sh.part[h][kResNW + w] = b;
    }
    __syncthreads();
    if constexpr (ONE) {
        const VT v = res_row8(l < 2 * kResNW ? sh.part[h][l] : VT(0));
        ta = res_lane(v, kResNW - 1);
        tb = res_lane(v, 2 * kResNW - 1);
        return true;
    }
    if (w == 0) {
        const VT v = res_row8(l < 2 * kResNW ? sh.part[h][l] : VT(0));
        a = res_lane(v, kResNW - 1);
        b = res_lane(v, 2 * kResNW - 1);
        bool ok = true;
        const int g = blockIdx.x & 7, m = blockIdx.x >> 3;
        double* now = S.slots + (size_t)(gen & (kSlotGens - 1)) * kSlotGen;
        double* old = S.slots + (size_t)((gen - 1) & (kSlotGens - 1)) * kSlotGen;
        unsigned* ab = S.words + RW_ABORT;
        const double pend = __longlong_as_double((long long)kResPending);
        if (S.grid <= kResFlat) {
            if (l < 8) {
                st_agent(now + l * kSlotRow + 2 * blockIdx.x, (double)a);
                st_agent(now + l * kSlotRow + 2 * blockIdx.x + 1, (double)b);
            }
            a = b = VT(0);
            const double* row = now + g * kSlotRow;
#pragma clang loop unroll(disable)
            for (int i = l; i < S.grid; i += kWave) {
                double va = 0, vb = 0;
                ok = res_poll2(row + 2 * i, ab, S.polls, va, vb) && ok;
                a += (VT)va;
                b += (VT)vb;
            }
            a = res_wave(a);
            b = res_wave(b);
            if (l < 8) {
                st_agent(old + l * kSlotRow + 2 * blockIdx.x, pend);
                st_agent(old + l * kSlotRow + 2 * blockIdx.x + 1, pend);
            }
        } else {
            // groups of the workgroups with equal blockIdx % 8; the first
            // of a group sums it and publishes to one row per group
            const int gs = (S.grid - g + 7) / 8;
            double* grp = now + g * kSlotRow;             // 2 * gs slots, gs <= 32
            double* top = now + g * kSlotRow + 128;       // this group's copy of the 8 group sums
            if (l == 0) {
                st_agent(grp + 2 * m, (double)a);
                st_agent(grp + 2 * m + 1, (double)b);
            }
            if (m == 0) {
                double va = 0, vb = 0;
                if (l < gs) ok = res_poll2(grp + 2 * l, ab, S.polls, va, vb);
                a = res_wave((VT)va);
                b = res_wave((VT)vb);
                if (l < 8) {
                    st_agent(now + l * kSlotRow + 128 + 2 * g, (double)a);
                    st_agent(now + l * kSlotRow + 128 + 2 * g + 1, (double)b);
                }
            }
            double va = 0, vb = 0;
            if (l < 8) ok = res_poll2(top + 2 * l, ab, S.polls, va, vb) && ok;
            a = res_wave((VT)va);
            b = res_wave((VT)vb);
            if (l == 0) {
                st_agent(old + g * kSlotRow + 2 * m, pend);
                st_agent(old + g * kSlotRow + 2 * m + 1, pend);
            }
            if (m == 0 && l < 8) {
                st_agent(old + l * kSlotRow + 128 + 2 * g, pend);
                st_agent(old + l * kSlotRow + 128 + 2 * g + 1, pend);
            }
        }
        ok = __all(ok);
        if (l == 0) {
            sh.tot[h][0] = a;
            sh.tot[h][1] = b;
            sh.ok[h] = ok;
        }
    }
    __syncthreads();
    // the same for every lane: kept in scalar registers, the branches on them scalar
    ta = res_lane(sh.tot[h][0], 0);
    tb = res_lane(sh.tot[h][1], 0);
    return __builtin_amdgcn_readfirstlane(sh.ok[h]) != 0;
}

// All workgroups are on the chip (true), or the launch gives up (false): one
// answer for the whole grid, taken by whoever moves the state from 0.
__device__ __forceinline__ bool res_meet(const ResSync& S, int* sh) {
    if (threadIdx.x == 0) {
        unsigned* st = S.words + RW_STATE;
        const unsigned before =
            __hip_atomic_fetch_add(S.words + RW_ARRIVE, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned expect = RS_OPEN;
        if (before + 1u == (unsigned)S.grid)
            __hip_atomic_compare_exchange_strong(st, &expect, (unsigned)RS_MET, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t t0 = wall_clock64();
        unsigned v;
        while ((v = ld_agent(st)) == RS_OPEN) {
            if (wall_clock64() - t0 > kResMeet) {
                expect = RS_OPEN;
                __hip_atomic_compare_exchange_strong(st, &expect, (unsigned)RS_REFUSED, __ATOMIC_RELAXED,
                                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __builtin_amdgcn_s_sleep(1);
        }
        *sh = v == RS_MET;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*sh) != 0;
}

// p of this workgroup is stored: tell the others, then wait for the
// workgroups within `neigh` of this one (all of p they own is then readable
// with agent-scope loads).  Every lane's stores are complete before the flag.
__device__ __forceinline__ bool res_exchange(const ResSync& S, int lb, int neigh, unsigned step, int* sh) {
    wait_memory();
    __syncthreads();
    if (threadIdx.x < kWave) {
        const int l = threadIdx.x;
        if (l == 0) st_agent(S.words + RW_FLAG + lb, step);
        const int lo = max(0, lb - neigh), hi = min(S.grid - 1, lb + neigh);
        bool ok = true;
        unsigned* ab = S.words + RW_ABORT;
#pragma clang loop unroll(disable)
        for (int i = lo + l; i <= hi; i += kWave) {
            unsigned it = 0;
#pragma clang loop unroll(disable)
            while (ld_agent(S.words + RW_FLAG + i) < step) {
                if ((++it & 255u) == 0 && ld_agent(ab) != 0u) { ok = false; break; }
                if (it > S.polls) {
                    st_agent(ab, 1u);
                    ok = false;
                    break;
                }
            }
        }
        ok = __all(ok);
        if (l == 0) *sh = ok;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*sh) != 0;
}

struct ResArgs {
    int32_t n;
    // diagonal operand: offsets ascending, values slice-major; map: stored diagonal of |offset| (symmetric copy)
    const int32_t *doff, *dmap;
    const void* val;
    int ndiag, nstored, sym, fmt, halo;
    // CSR operand
    const int32_t *rowptr, *col;
    // vectors
    void *x, *r, *p;
    const void* d;
    int dfmt;   // MTL4G_F64 / MTL4G_F32; d null: identity
    int neigh;
    Ctl* c;
    double* hist;
    int32_t steps;
    ResSync S;
};

// ------------------------------------------------------------------ the loop head
// The scalars of the recurrence and of basic_iteration, held by every lane (the
// sums are the same for all of them).  Only workgroup 0 writes *c, after every
// workgroup has passed the rendezvous and so has read it.
template <typename VT>
struct ResLoop {
    VT rho, rho_1, beta, alpha, pq, rr, rz;
    double norm_r0, atol, stop, grown, fell, resid;
    int i, hist_n, max_iter, hist_cap, done, error, status, pause, want_ru, drop, limit;
    bool first, mixed;
    __device__ __forceinline__ void init(const Ctl* c) {
        first = c->first != 0;
        mixed = c->mixed != 0;
        rho = static_cast<VT>(c->rho);
        rho_1 = static_cast<VT>(c->rho_1);
        beta = static_cast<VT>(c->beta);
        alpha = static_cast<VT>(c->alpha);
        pq = static_cast<VT>(c->alpha_1);
        rr = rz = VT(0);
        norm_r0 = c->norm_r0;
        atol = c->atol;
        // conv_test: resid <= rtol*norm_r0 || resid <= atol (norm_r0 == 0: atol alone)
        stop = norm_r0 == 0 ? atol : fmax(c->rtol * norm_r0, atol);
        grown = kGrowth * c->rmax;
        fell = c->delta * c->rmax;
        i = c->i;
        hist_n = c->hist_n;
        max_iter = c->max_iter;
        hist_cap = c->hist_cap;
        done = error = status = pause = want_ru = drop = limit = 0;
        resid = 0.0;
    }
    // alpha = rho / p.q  (cg.hpp:105)
    __device__ __forceinline__ void direction() {
        alpha = rho / pq;
        rho_1 = rho;
    }
    // iter_finished / mixed_check (krylov_dev.hpp) on rr and, when the loop
    // goes on, the next rho and beta  (cg.hpp:94-101); true: leave the kernel.
    // writer: the one lane of the grid that records the residual
    __device__ __forceinline__ bool head(double* hist, bool writer) {
        resid = (double)std::sqrt(std::fabs(rr));
        const bool conv = resid <= stop, out = i >= max_iter, bad = !isfinite(resid);
        if (!mixed) {
            if (writer && hist_n < hist_cap) hist[hist_n] = resid;
            hist_n++;
            done = conv || out || bad;
            if (done && !conv) {
                if (out) error = 1;
                else status = MTL4G_ERR_NONFINITE;
            }
        } else {
            pause = bad || conv || out || resid > grown;
            want_ru = pause || resid <= fell;
            drop = bad;
            limit = !bad && !conv && out;
        }
        if (!done && !pause) {
            i++;
            first = i <= 1;
            beta = rz / rho_1;
            rho = rz;
        }
        return done || want_ru;
    }
    __device__ __forceinline__ void leave(Ctl* c, bool ok) const {
        if (!mixed) c->resid = resid;
        c->rr = (double)rr;
        c->alpha = (double)alpha;
        c->alpha_1 = (double)pq;
        c->rho_1 = (double)rho_1;
        c->rho = (double)rho;
        c->beta = (double)beta;
        c->i = i;
        c->first = first;
        c->hist_n = hist_n;
        c->done = done;
        c->error = error;
        c->status = status;
        c->pause = pause;
        c->want_ru = want_ru;
        if (drop) c->drop = 1;
        if (limit) c->limit = 1;
        if (!ok) {   // a wait expired: the solve ends with an error
            c->status = MTL4G_ERR_TIMEOUT;
            c->done = 1;
        }
    }
};

// resident_large.hip: the launch for a matrix whose values are streamed.
// `groups` groups of 16 bytes of a vector per lane; vectors of vt_bytes bytes
// per element, values of a.fmt.
int resident_large_launch(const ResArgs& a, int vt_bytes, int groups, hipStream_t s);
// The fewest groups per lane (of those that are built) with which n rows fit
// `cus` workgroups; 0: too many rows.
int resident_large_groups(int64_t n, int vt_bytes, int cus);

}  // namespace mtl4g
