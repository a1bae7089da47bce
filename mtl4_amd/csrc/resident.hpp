// resident.hpp -- itl::cg with its state on the chip (resident.hip, resident_large.hip).
#pragma once

#include <algorithm>

#include "krylov.hpp"

namespace mtl4g {

// Runs CG iterations from the state the loop head left in W (r, p, Ctl;
// cg.hpp:94-108), the identity or diagonal preconditioner, inside one kernel
// per batch of iterations.  Returns MTL4G_OK with *ran = true when the solve
// stopped (Ctl::done set), or with *ran = false, and nothing done, when this
// path does not take the matrix.  inv_diag: n values of the vector type's
// precision or of the other one (dfmt MTL4G_F64 / MTL4G_F32), null for the
// identity.  A launch runs at most `steps` iterations; after() is enqueued
// behind each (mixed precision: the FP64 refresh).
//
// A launch that does not get onto the chip (another stream's or process's
// kernel holds compute units) is followed by iterations in launches of their
// own, which need no more than one compute unit at a time and form every sum in
// the same order: the solve goes on, with the same bits.  product() enqueues
// q = A*p for those (p, q: the first two vectors of W).  The chip is tried
// again after kStepsMin of them, and after twice as many each time it refuses.
template <typename VT, typename Product, typename After>
int resident_cg(const mtl4g_matrix_s* A, int value_format, const void* inv_diag, int dfmt, Workspace<VT>& W, VT* x,
                hipStream_t s, int32_t steps, Product product, After after, bool* ran);

// The pieces the template above is made of.
struct ResidentPlan {
    int op = 0;          // 0: not taken; else the kernel variant
    int rows_log2 = 0;   // rows per lane: 1 << rows_log2
    int groups = 0;      // streamed matrix: 16-byte groups of rows per lane
    int grid = 0;        // workgroups
    int halo = 0;        // diagonal operand: neighbouring elements kept in LDS
    int neigh = 0;       // workgroups on either side whose p is read
    bool share = false;  // p goes through memory
};
// vectors of vt_bytes per element; own_diag: no inverse diagonal, or one in the vectors' type
ResidentPlan resident_plan(const mtl4g_matrix_s* A, int vt_bytes, int value_format, bool own_diag);
template <typename VT>
int resident_launch(const ResidentPlan& plan, const mtl4g_matrix_s* A, int value_format, const void* inv_diag,
                    int dfmt, Workspace<VT>& W, VT* x, int32_t steps, hipStream_t s);
// The three parts of an iteration around q = A*p and behind it, each a launch;
// RSTEP_RESID: the residual of a solve that stopped, from the rows alone.
enum { RSTEP_P = 0, RSTEP_ALPHA = 1, RSTEP_UPDATE = 2, RSTEP_RESID = 3 };
template <typename VT>
int resident_step(int part, const ResidentPlan& plan, const mtl4g_matrix_s* A, const void* inv_diag, int dfmt,
                  Workspace<VT>& W, VT* x, hipStream_t s);
// What the last solve of this thread did here (mtl4g_cg_chip).
mtl4g_cg_chip_info& resident_info();

// Compute units taken by resident grids of this process, per device: a grid
// that spans several workgroups takes its CUs before it is launched and gives
// them back after it has finished, so two such grids never wait for each
// other's CUs.  Served in the order of arrival: a solve that gives its units
// back and asks again at once stands behind those that waited.  A claim waits at
// most wait_ms per claim before it and then stands for nothing (held() false):
// whoever holds the units may itself be waiting, for earlier work on its stream.
// The caller launches all the same; two grids that meet are refused and go on in
// single steps.
struct ResidentClaim {
    int device, units;
    bool wanted;
    ResidentClaim* next = nullptr;   // behind this one in the queue
    ResidentClaim(int device, int units, int total, int wait_ms);
    ~ResidentClaim();
    bool held() const { return units > 0 || !wanted; }
    ResidentClaim(const ResidentClaim&) = delete;
    ResidentClaim& operator=(const ResidentClaim&) = delete;
};
constexpr int kClaimWait = 30;   // a holder's launches take about 20 ms at most (four of 5 ms)

// Iterations per launch, so that other streams' kernels wait no more than about
// 5 ms for the compute units: 256 of up to 20 us while the matrix is in
// registers; streamed ones take time by their rows (102^3 15.5 us, 160^3 73 us in
// FP64), so vectors of more than 8 MB get as many fewer (160^3: 65, 4.7 ms; one
// launch of 256 held all compute units for 18.8 ms).
constexpr int32_t kResidentSteps = 256;
constexpr int64_t kResidentVector = 8 << 20;
// Iterations in launches of their own after a refusal: at first about as long
// as the millisecond the refusal took; doubled, so that a GPU that stays shared
// costs a solve little more than those launches.
constexpr int kStepsMin = 32, kStepsMax = 512;
constexpr int kStepsPerRefresh = 4;   // a pause for after() skips at most three of them

template <typename VT, typename Product, typename After>
int resident_cg(const mtl4g_matrix_s* A, int value_format, const void* inv_diag, int dfmt, Workspace<VT>& W, VT* x,
                hipStream_t s, int32_t steps, Product product, After after, bool* ran) {
    *ran = false;
    mtl4g_cg_chip_info& info = resident_info();
    info = mtl4g_cg_chip_info{};
    if (W.shared_gpu) return MTL4G_OK;
    const ResidentPlan plan = resident_plan(
        A, (int)sizeof(VT), value_format, !inv_diag || dfmt == (sizeof(VT) == 8 ? MTL4G_F64 : MTL4G_F32));
    if (!plan.op) return MTL4G_OK;
    info.operand = plan.op;
    info.workgroups = plan.grid;
    info.rows_per_lane = plan.groups ? plan.groups * 16 / (int)sizeof(VT) : 1 << plan.rows_log2;
    info.halo = plan.halo;
    info.steps = steps;
    auto poll = [&]() -> int {
        M4_HIP(hipMemcpyAsync(W.h_ctl, W.ctl.p, sizeof(Ctl), hipMemcpyDeviceToHost, s));
        M4_HIP(hipStreamSynchronize(s));
        return MTL4G_OK;
    };
    int launches = 1, chunk = kStepsMin, wait = kClaimWait;
    for (;;) {
        {
            ResidentClaim claim(A->device, plan.grid > 1 ? plan.grid : 0, A->cus, wait);
            wait = claim.held() ? kClaimWait : 0;   // waited once: from then on only where units are free
            for (int k = 0; k < launches; k++) {
                M4_TRY(resident_launch<VT>(plan, A, value_format, inv_diag, dfmt, W, x, steps, s));
                M4_TRY(after());
            }
            M4_TRY(poll());
        }
        const bool refused = W.h_ctl->refused != info.refused;
        info.refused = W.h_ctl->refused;
        if (!W.h_ctl->done && refused) {
            for (int k = 0; k < chunk; k++) {
                M4_TRY(resident_step<VT>(RSTEP_P, plan, A, inv_diag, dfmt, W, x, s));
                M4_TRY(product());
                M4_TRY(resident_step<VT>(RSTEP_ALPHA, plan, A, inv_diag, dfmt, W, x, s));
                M4_TRY(resident_step<VT>(RSTEP_UPDATE, plan, A, inv_diag, dfmt, W, x, s));
                if (k % kStepsPerRefresh == kStepsPerRefresh - 1) M4_TRY(after());
            }
            info.single_steps += chunk;
            M4_TRY(poll());
        }
        if (W.h_ctl->done) {
            // An infinite alpha (p.q = 0) makes NaN of 0 - alpha*0 in the places of the
            // grid that hold no row, and of the residual with them.  Formed again here:
            // masking the places in the loop cost 3 % of a 160^3 and a 64^2 solve.
            if (W.h_ctl->status == MTL4G_ERR_NONFINITE && !W.h_ctl->mixed)
                M4_TRY(resident_step<VT>(RSTEP_RESID, plan, A, inv_diag, dfmt, W, x, s));
            *ran = true;
            return MTL4G_OK;
        }
        chunk = refused ? std::min(2 * chunk, kStepsMax) : kStepsMin;
        launches = refused ? 1 : 4;
    }
}

}  // namespace mtl4g
