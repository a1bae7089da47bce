// resident.hpp -- itl::cg with its state on the chip (resident.hip, resident_large.hip).
#pragma once

#include "krylov.hpp"

namespace mtl4g {

// Runs CG iterations from the state the loop head left in W (r, p, Ctl;
// cg.hpp:94-108), the identity or diagonal preconditioner, inside one kernel
// per batch of iterations.  Returns MTL4G_OK with *ran = true when the solve
// stopped (Ctl::done set), or with *ran = false when this path does not take
// the matrix (or the GPU stayed too busy to hold the whole grid): the caller's
// own loop goes on from the same state.  inv_diag: n values of the vector
// type's precision or of the other one (dfmt MTL4G_F64 / MTL4G_F32), null for
// the identity.  A launch runs at most `steps` iterations; after() is enqueued
// behind each (mixed precision: the FP64 refresh).
template <typename VT, typename After>
int resident_cg(const mtl4g_matrix_s* A, int value_format, const void* inv_diag, int dfmt, Workspace<VT>& W, VT* x,
                hipStream_t s, int32_t steps, After after, bool* ran);

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

// Compute units taken by resident grids of this process, per device: a grid
// that spans several workgroups takes its CUs before it is launched and gives
// them back after it has finished, so two such grids never wait for each
// other's CUs.
struct ResidentClaim {
    int device, units;
    ResidentClaim(int device, int units, int total);
    ~ResidentClaim();
    ResidentClaim(const ResidentClaim&) = delete;
    ResidentClaim& operator=(const ResidentClaim&) = delete;
};

// iterations per launch: a few milliseconds, so that other streams' kernels
// wait no longer for the compute units
constexpr int32_t kResidentSteps = 256;
constexpr int kResidentRefusals = 2000;      // refused launches before the caller's loop takes over

template <typename VT, typename After>
int resident_cg(const mtl4g_matrix_s* A, int value_format, const void* inv_diag, int dfmt, Workspace<VT>& W, VT* x,
                hipStream_t s, int32_t steps, After after, bool* ran) {
    *ran = false;
    if (W.shared_gpu) return MTL4G_OK;
    const ResidentPlan plan = resident_plan(
        A, (int)sizeof(VT), value_format, !inv_diag || dfmt == (sizeof(VT) == 8 ? MTL4G_F64 : MTL4G_F32));
    if (!plan.op) return MTL4G_OK;
    int launches = 1;
    for (;;) {
        int32_t refused = 0;
        {
            ResidentClaim claim(A->device, plan.grid > 1 ? plan.grid : 0, A->cus);
            for (int k = 0; k < launches; k++) {
                M4_TRY(resident_launch<VT>(plan, A, value_format, inv_diag, dfmt, W, x, steps, s));
                M4_TRY(after());
            }
            M4_HIP(hipMemcpyAsync(W.h_ctl, W.ctl.p, sizeof(Ctl), hipMemcpyDeviceToHost, s));
            M4_HIP(hipStreamSynchronize(s));
            refused = W.h_ctl->refused;
        }
        if (W.h_ctl->done) {
            *ran = true;
            return MTL4G_OK;
        }
        if (refused > kResidentRefusals) return MTL4G_OK;
        launches = 4;
    }
}

}  // namespace mtl4g
