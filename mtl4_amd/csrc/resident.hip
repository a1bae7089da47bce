// resident.hip -- itl::cg + pc::identity / pc::diagonal (cg.hpp:38-111) with
// the whole state of the recurrence on the chip.
//
// The three-launch iteration of krylov.hip pays a launch, a grid ramp and a
// last-workgroup reduction per kernel: 21.7 us per iteration on a 64 x 64
// Laplacian whose arithmetic takes none of it.  Here one launch runs up to
// kResidentSteps iterations: a lane keeps its rows of x, r, p, z, the inverse
// diagonal and its part of the matrix in registers, and the only traffic
// between workgroups is the direction p (written once per iteration, read
// where the matrix reaches into another workgroup's rows) and two all-reduced
// sums.  A system of up to kResBS * 8 rows is one workgroup and needs
// neither.
//
// Element-wise results are those of the epilogues in krylov.hip bit for bit
// (p, q, x, r; rows summed in column order); the sums are combined in another
// fixed order, which depends only on the system, so a solve is deterministic.
//
// Workgroups wait for each other (resident_dev.hpp), so all of them must be on the
// chip at once.  A launch first meets at a rendezvous with a bounded wait:
// when the grid does not get onto the chip (another kernel holds its CUs) the
// launch gives up before it has changed anything, and iterations in launches of
// their own (k_cg_step) go on from the same state with the same bits until the
// host tries again.  After the rendezvous every workgroup is running and every
// later wait ends; those waits are bounded too and raise an abort flag.
//
// Ordering: the inter-workgroup protocol of internal.hpp (agent-scope stores
// and loads; wait_memory before the store that announces).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>

#include "resident_dev.hpp"

namespace mtl4g {

// ------------------------------------------------------------------ the matrix of a lane's rows
// Lane t of workgroup lb holds rows lb*R*BS + k*BS + t, k < R.

template <typename VT>
__device__ __forceinline__ VT res_value(const void* v, int fmt, int64_t i) {
    if (fmt == MTL4G_F64) return static_cast<VT>(static_cast<const double*>(v)[i]);
    if (fmt == MTL4G_F32) return static_cast<VT>(static_cast<const float*>(v)[i]);
    return static_cast<VT>(bf16_to_f32(static_cast<const uint16_t*>(v)[i]));
}
__device__ __forceinline__ bool res_absent(const void* v, int fmt, int64_t i) {
    if (fmt == MTL4G_F64) return dia_absent(static_cast<const double*>(v)[i]);
    if (fmt == MTL4G_F32) return dia_absent(static_cast<const float*>(v)[i]);
    return dia_absent(static_cast<const uint16_t*>(v)[i]);
}

// Element i of a vector of at most 2^29 elements, at agent scope: a 32-bit
// offset on a uniform base (no 64-bit address per lane).
template <typename VT>
__device__ __forceinline__ VT res_ld(const VT* p, int i) {
    return ld_agent(reinterpret_cast<const VT*>(reinterpret_cast<const char*>(p) + (unsigned)i * (unsigned)sizeof(VT)));
}

// Diagonals (at most ND, |offset| <= halo but for the first and the last):
// values in registers, the workgroup's p with `halo` neighbours on both sides
// in LDS, the first and last diagonal's p from memory when they lie further
// out.  Slot ND-1 is always the last diagonal; slots without one are absent.
template <typename VT, int ND_, int R_>
struct OpDia {
    static constexpr int R = R_, ND = ND_, kRegs = R_ * ND_;
    static constexpr bool kOne = R_ <= 8;   // runs as one workgroup (up to 4096 rows) without p in memory
    static constexpr int LDS = R * kResBS + 2 * kResHalo;
    VT v[R][ND];
    unsigned mask[R];
    unsigned full;      // bit k: every entry of every lane's row k is present (wave-uniform)
    int off[ND];        // uniform
    bool flo, fhi;      // the first / last diagonal is read from memory
    int halo;
    template <typename Args>
    __device__ __forceinline__ void load(const Args& a, int row0) {
        halo = a.halo;
        full = 0;
#pragma unroll
        for (int d = 0; d < ND; d++) {
            const int di = d == ND - 1 ? a.ndiag - 1 : d;
            const bool has = d == ND - 1 || d < a.ndiag - 1;
            off[d] = has ? __builtin_amdgcn_readfirstlane(a.doff[di]) : 0;
        }
        flo = off[0] < -halo;
        fhi = off[ND - 1] > halo;
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int row = row0 + k * kResBS + (int)threadIdx.x;
            mask[k] = 0;
#pragma unroll
            for (int d = 0; d < ND; d++) {
                v[k][d] = VT(0);
                const int di = d == ND - 1 ? a.ndiag - 1 : d;
                const bool has = d == ND - 1 || d < a.ndiag - 1;
                if (has && row < a.n) {
                    const int src = a.sym && off[d] < 0 ? row + off[d] : row;
                    const int st = a.sym ? a.dmap[di] : di;
                    if (src >= 0) {
                        const int64_t i = ((int64_t)(src / kWave) * a.nstored + st) * kWave + src % kWave;
                        if (!res_absent(a.val, a.fmt, i)) {
                            v[k][d] = res_value<VT>(a.val, a.fmt, i);
                            mask[k] |= 1u << d;
                        }
                    }
                }
            }
            if (__all(mask[k] == (1u << ND) - 1u)) full |= 1u << k;
        }
        full = __builtin_amdgcn_readfirstlane(full);
    }
    // own p into LDS (a barrier follows before product())
    __device__ __forceinline__ void put(VT* lds, int k, VT p) const {
        lds[halo + k * kResBS + (int)threadIdx.x] = p;
    }
    template <bool ONE, typename Args>
    __device__ __forceinline__ void product(const Args& a, int row0, VT* lds, VT (&q)[R]) const {
        const VT* p = static_cast<const VT*>(a.p);
        VT gl[R], gh[R], h[2 * kResHalo / kResBS];
        // the lane index is made opaque, so that the addresses below are formed
        // again in every iteration instead of living in registers across it
        unsigned t = threadIdx.x;
        asm volatile("" : "+v"(t));
        const int last = a.n - 1;
#pragma unroll
        for (int k = 0; k < R; k++) gl[k] = gh[k] = VT(0);
        if constexpr (!ONE) {
            if (flo)
#pragma unroll
                for (int k = 0; k < R; k++) gl[k] = res_ld(p, min(max(row0 + k * kResBS + (int)t + off[0], 0), last));
            if (fhi)
#pragma unroll
                for (int k = 0; k < R; k++) gh[k] = res_ld(p, min(row0 + k * kResBS + (int)t + off[ND - 1], last));
#pragma unroll
            for (int i = 0; i < 2 * kResHalo / kResBS; i++) {
                const int j = (int)t + i * kResBS;   // 0..2*halo: below the rows, then above them
                const int row = j < halo ? row0 - halo + j : row0 + R * kResBS + j - halo;
                h[i] = VT(0);
                if (j < 2 * halo && row >= 0 && row <= last) h[i] = res_ld(p, row);
            }
#pragma unroll
            for (int i = 0; i < 2 * kResHalo / kResBS; i++) {
                const int j = (int)t + i * kResBS;
                if (j < 2 * halo) lds[j < halo ? j : R * kResBS + j] = h[i];
            }
            __syncthreads();
        }
#pragma unroll
        for (int k = 0; k < R; k++) {
            const VT* own = lds + (halo + k * kResBS + (int)t);
            VT g[ND];
#pragma unroll
            for (int d = 0; d < ND; d++) {
                if (!ONE && d == 0) g[d] = flo ? gl[k] : own[flo ? 0 : off[d]];
                else if (!ONE && d == ND - 1) g[d] = fhi ? gh[k] : own[fhi ? 0 : off[d]];
                else g[d] = own[off[d]];
            }
            VT acc = VT(0);
            unsigned mk = mask[k];   // opaque: no lane mask per entry kept across iterations
            asm volatile("" : "+v"(mk));
            if ((full >> k) & 1u) {
#pragma unroll
                for (int d = 0; d < ND; d++) acc += v[k][d] * g[d];
            } else {
#pragma unroll
                for (int d = 0; d < ND; d++) {
                    const VT with = acc + v[k][d] * g[d];
                    acc = (mk >> d) & 1u ? with : acc;
                }
            }
            q[k] = acc;
            // two rows' neighbours in registers at a time
            if (R > 2 && k % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
    }
};

// Any pattern: the workgroup's entries spread over its lanes (at most E each,
// values and columns in registers), products through LDS, a lane sums each of
// its rows in column order.
template <typename VT, int E_, int R_>
struct OpCsr {
    static constexpr int R = R_, E = E_, kRegs = 0;
    static constexpr bool kOne = false;
    static constexpr int LDS = E * kResBS;
    VT v[E];
    int c[E];
    int ra[R], re[R];
    int nz;
    template <typename Args>
    __device__ __forceinline__ void load(const Args& a, int row0) {
        const int t = (int)threadIdx.x;
        const int r1 = min(row0 + R * kResBS, a.n);
        const int j0 = a.rowptr[min(row0, a.n)];
        nz = a.rowptr[r1] - j0;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int j = t + e * kResBS;
            v[e] = VT(0);
            c[e] = 0;
            if (j < nz) {
                v[e] = res_value<VT>(a.val, a.fmt, j0 + j);
                c[e] = a.col[j0 + j];
            }
        }
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int row = row0 + k * kResBS + t;
            ra[k] = re[k] = 0;
            if (row < a.n) {
                ra[k] = a.rowptr[row] - j0;
                re[k] = a.rowptr[row + 1] - j0;
            }
        }
    }
    __device__ __forceinline__ void put(VT*, int, VT) const {}
    template <bool ONE, typename Args>
    __device__ __forceinline__ void product(const Args& a, int row0, VT* lds, VT (&q)[R]) const {
        const VT* p = static_cast<const VT*>(a.p);
        const int t = (int)threadIdx.x;
        VT g[E];
#pragma unroll
        for (int e = 0; e < E; e++) g[e] = t + e * kResBS < nz ? ld_agent(p + c[e]) : VT(0);
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int j = t + e * kResBS;
            if (j < nz) lds[j] = v[e] * g[e];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R; k++) {
            VT s = VT(0);
            for (int j = ra[k]; j < re[k]; j++) s += lds[j];
            q[k] = s;
        }
    }
};

// ------------------------------------------------------------------ the recurrence
// What bounds it: latency.  Per iteration a grid pays one exchange of p (store,
// flag, poll, read: about 2.5 us) and two all-reduces (2-2.8 us each); one
// workgroup pays two block reductions, three divisions and square roots and
// the LDS reads of its rows.  Measured per iteration (FP64, diagonal
// preconditioner; before: three launches): 64^2 Laplacian 21.7 -> 2.8 us,
// 61^3 diffusion 27 -> 9.3 us, 80^3 12.4 us, 100^3 18 us.
// ONE: the grid is one workgroup and the operand reads p from LDS alone.
template <typename VT, typename Op, bool ONE>
__global__ __launch_bounds__(kResBS) void k_cg_resident(ResArgs a) {
    constexpr int R = Op::R;
    // eight FP64 rows of seven diagonals fill the registers: x and the inverse
    // diagonal of those live in LDS, read and written by their own lane only
    constexpr bool XD_LDS = Op::kRegs * sizeof(VT) > 400;
    __shared__ VT xd[XD_LDS ? 2 * R * kResBS : 1];
    __shared__ VT lds[Op::LDS];
    __shared__ ResShared<VT> sh;
    __shared__ int flag;
    const int t = (int)threadIdx.x;
    // the operand's rows: consecutive workgroups of one XCD hold consecutive rows
    const int G = ONE ? 1 : a.S.grid;
    int lb = ONE ? 0 : (int)blockIdx.x;
    if (G % kXcd == 0) lb = xcd_logical_block(lb, G / kXcd);
    const int row0 = lb * R * kResBS;
    if (a.c->done || a.c->pause || a.c->want_ru) return;   // the whole grid reads the same state
    ResLoop<VT> L;
    L.init(a.c);
    VT* xg = static_cast<VT*>(a.x);
    VT* rg = static_cast<VT*>(a.r);
    VT* pg = static_cast<VT*>(a.p);
    Op op;
    op.load(a, row0);
    VT xr[XD_LDS ? 1 : R], dr[XD_LDS ? 1 : R], r[R], p[R], z[R];
    auto x = [&](int k) -> VT& { return XD_LDS ? xd[k * kResBS + t] : xr[XD_LDS ? 0 : k]; };
    auto d = [&](int k) -> VT& { return XD_LDS ? xd[(R + k) * kResBS + t] : dr[XD_LDS ? 0 : k]; };
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int row = row0 + k * kResBS + t;
        VT xk = VT(0), dk = VT(1);
        r[k] = p[k] = z[k] = VT(0);
        if (row < a.n) {
            xk = xg[row];
            r[k] = rg[row];
            p[k] = L.first ? VT(0) : pg[row];
            if (a.d) dk = res_value<VT>(a.d, a.dfmt, row);
            z[k] = dk * r[k];
        }
        x(k) = xk;
        d(k) = dk;
    }
    if (!ONE && !res_meet(a.S, &flag)) {
        if (blockIdx.x == 0 && t == 0) a.c->refused++;
        return;
    }
    bool ok = true;
    unsigned step = 0;
    int gen = 0;
    for (;;) {
        // p = z  or  p = z + beta*p  (cg.hpp:98-101)
        unsigned to = (unsigned)t;
        asm volatile("" : "+v"(to));
#pragma unroll
        for (int k = 0; k < R; k++) {
            p[k] = L.first ? z[k] : z[k] + L.beta * p[k];
            op.put(lds, k, p[k]);
            const int row = row0 + k * kResBS + (int)to;
            if (!ONE && row < a.n) st_agent(pg + row, p[k]);
        }
        step++;
        if constexpr (!ONE) {
            ok = res_exchange(a.S, lb, a.neigh, step, &flag);
            if (!ok) break;
        } else {
            __syncthreads();
        }
        // q = A*p, p.q; alpha  (cg.hpp:103-105)
        VT q[R];
        op.template product<ONE>(a, row0, lds, q);
        VT s0 = VT(0), s1 = VT(0);
#pragma unroll
        for (int k = 0; k < R; k++) s0 += p[k] * q[k];
        ok = res_allsum<VT, ONE>(a.S, gen++, s0, VT(0), sh, L.pq, s1);
        if (!ok) break;
        L.direction();
        // x += alpha*p; r -= alpha*q; r.r, r.(d.*r)  (cg.hpp:106-108)
        s0 = s1 = VT(0);
#pragma unroll
        for (int k = 0; k < R; k++) {
            x(k) = x(k) + L.alpha * p[k];
            r[k] = r[k] - L.alpha * q[k];
            z[k] = d(k) * r[k];
            s0 += r[k] * r[k];
            s1 += r[k] * z[k];
        }
        ok = res_allsum<VT, ONE>(a.S, gen++, s0, s1, sh, L.rr, L.rz);
        if (!ok) break;
        if (L.head(a.hist, blockIdx.x == 0 && t == 0) || (int)step >= a.steps) break;
    }
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int row = row0 + k * kResBS + t;
        if (row < a.n) {
            xg[row] = x(k);
            rg[row] = r[k];
            pg[row] = p[k];
        }
    }
    if (blockIdx.x == 0 && t == 0) L.leave(a.c, ok);
}

// Slots pending, words zero, before each launch; state: RS_OPEN, or RS_REFUSED
// for a launch that is to be turned away (mtl4g_set_cg_chip_limits).
__global__ void k_resident_begin(ResSync S, unsigned state) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kSlotGens * kSlotGen) S.slots[i] = __longlong_as_double((long long)kResPending);
    if (i < kResWords) S.words[i] = i == RW_STATE ? state : 0u;
}

// ------------------------------------------------------------------ iterations in launches of their own
// The same state, the same arithmetic per element and every sum in the order of
// the kernels above: a lane adds up its rows of the plan (`groups` of them, `per`
// consecutive rows each), then res_allsum's order over lanes, waves and
// workgroups.  No workgroup waits for another.  p is written first, then the
// caller's product forms q.
template <typename VT>
__global__ __launch_bounds__(kResBS) void k_cg_step_p(ResArgs a) {
    const Ctl* c = a.c;
    if (c->done || c->pause || c->want_ru) return;
    const bool first = c->first != 0;
    const VT beta = static_cast<VT>(c->beta);
    const VT* r = static_cast<const VT*>(a.r);
    VT* p = static_cast<VT*>(a.p);
    constexpr int U = 4;   // elements at once
    const int64_t stride = (int64_t)gridDim.x * kResBS;
    for (int64_t i0 = blockIdx.x * (int64_t)kResBS + threadIdx.x; i0 < a.n; i0 += U * stride) {
        VT z[U], old[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t i = min(i0 + u * stride, (int64_t)a.n - 1);
            z[u] = a.d ? res_value<VT>(a.d, a.dfmt, i) * r[i] : r[i];
            old[u] = p[i];
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i0 + u * stride < a.n) p[i0 + u * stride] = first ? z[u] : z[u] + beta * old[u];
    }
}

// PART: RSTEP_ALPHA p.q and alpha; RSTEP_UPDATE x, r, the loop head; RSTEP_RESID
// the residual that the loop head recorded last.
// Bound by memory at 160^3 (four launches, 623 MB, 145 us per iteration; one row
// at a time instead of four groups 157), by the launches at 61^3 (28 us).
template <typename VT, int PART, int PER>
__global__ __launch_bounds__(kResBS) void k_cg_step(ResArgs a, const VT* q, int groups) {
    Ctl* c = a.c;
    constexpr bool UPDATE = PART == RSTEP_UPDATE;
    if (PART != RSTEP_RESID && (c->done || c->pause || c->want_ru)) return;
    __shared__ VT part[2 * kResNW];
    const int t = (int)threadIdx.x, l = t & (kWave - 1), w = t / kWave, G = a.S.grid;
    int lb = (int)blockIdx.x;
    if (G % kXcd == 0) lb = xcd_logical_block(lb, G / kXcd);
    VT* x = static_cast<VT*>(a.x);
    VT* r = static_cast<VT*>(a.r);
    const VT* p = static_cast<const VT*>(a.p);
    const VT alpha = static_cast<VT>(c->alpha);
    VT s0 = VT(0), s1 = VT(0);
    constexpr int U = 4;   // groups at once
    for (int k0 = 0; k0 < groups; k0 += U) {
        VT pi[U * PER], qi[U * PER], ri[U * PER], xi[U * PER], di[U * PER];
        auto row = [&](int e) {
            const int64_t i = ((int64_t)(lb * groups + k0 + e / PER) * kResBS + t) * PER + e % PER;
            return k0 + e / PER < groups && i < a.n ? i : (int64_t)-1;
        };
#pragma unroll
        for (int e = 0; e < U * PER; e++) {
            const int64_t i = max(row(e), (int64_t)0);
            if (PART != RSTEP_RESID) pi[e] = p[i], qi[e] = q[i];
            if (PART != RSTEP_ALPHA) ri[e] = r[i];
            if (UPDATE) {
                xi[e] = x[i];
                di[e] = a.d ? res_value<VT>(a.d, a.dfmt, i) : VT(1);
            }
        }
#pragma unroll
        for (int e = 0; e < U * PER; e++) {
            const int64_t i = row(e);
            if (i < 0) continue;
            if (UPDATE) {
                x[i] = xi[e] + alpha * pi[e];
                const VT rn = ri[e] - alpha * qi[e];
                r[i] = rn;
                s0 += rn * rn;
                s1 += rn * (di[e] * rn);
            } else if (PART == RSTEP_RESID) {
                s0 += ri[e] * ri[e];
            } else {
                s0 += pi[e] * qi[e];
            }
        }
    }
    s0 = res_wave(s0);
    s1 = res_wave(s1);
    if (l == 0) {
        part[w] = s0;
        part[kResNW + w] = s1;
    }
    __syncthreads();
    if (w == 0) {
        const VT v = res_row8(l < 2 * kResNW ? part[l] : VT(0));
        s0 = res_lane(v, kResNW - 1);
        s1 = res_lane(v, 2 * kResNW - 1);
        if (l == 0) {
            st_agent(a.S.slots + 2 * blockIdx.x, (double)s0);
            st_agent(a.S.slots + 2 * blockIdx.x + 1, (double)s1);
        }
    }
    if (!arrive_last<kResBS>(a.S.words + RW_TICKET, (unsigned)G) || w != 0) return;
    auto sum = [&](int i, VT& ta, VT& tb) {   // workgroup i's sums
        ta += (VT)ld_agent(a.S.slots + 2 * i);
        tb += (VT)ld_agent(a.S.slots + 2 * i + 1);
    };
    s0 = s1 = VT(0);
    if (G <= kResFlat) {
        for (int i = l; i < G; i += kWave) sum(i, s0, s1);
    } else {
        for (int g = 0; g < 8; g++) {
            VT ga = VT(0), gb = VT(0);
            if (l < (G - g + 7) / 8) sum(g + 8 * l, ga, gb);
            ga = res_wave(ga);
            gb = res_wave(gb);
            if (l == g) {
                s0 = ga;
                s1 = gb;
            }
        }
    }
    s0 = res_wave(s0);
    s1 = res_wave(s1);
    if (l != 0) return;
    if (PART == RSTEP_RESID) {
        c->rr = (double)s0;
        c->resid = (double)std::sqrt(std::fabs(s0));
        if (c->hist_n > 0 && c->hist_n <= c->hist_cap) a.hist[c->hist_n - 1] = c->resid;
        return;
    }
    ResLoop<VT> L;
    L.init(c);
    if (UPDATE) {
        L.rr = s0;
        L.rz = s1;
        L.head(a.hist, true);
        L.leave(c, true);
    } else {
        L.pq = s0;
        L.direction();
        c->alpha = (double)L.alpha;
        c->alpha_1 = (double)L.pq;
        c->rho_1 = (double)L.rho_1;
    }
}

// ------------------------------------------------------------------ host
namespace {
struct Units {
    struct Device {
        int used = 0;                     // CUs held by resident grids
        ResidentClaim* first = nullptr;   // claims that wait, in the order of arrival
    };
    std::mutex mu;
    std::condition_variable cv;
    Device devices[64];
    Device& of(int device) { return devices[(unsigned)device % 64]; }
};
Units& units() {
    static Units u;
    return u;
}
}  // namespace

ResidentClaim::ResidentClaim(int dev, int n, int total, int wait_ms)
    : device(dev), units(std::min(n, total)), wanted(n > 0) {
    if (!units) return;
    Units& u = mtl4g::units();
    std::unique_lock<std::mutex> lk(u.mu);
    Units::Device& d = u.of(device);
    int ahead = 1;   // the holder
    ResidentClaim** at = &d.first;
    for (; *at; at = &(*at)->next) ahead++;
    *at = this;
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(wait_ms) * ahead;
    const bool mine = u.cv.wait_until(lk, until, [&] { return d.first == this && d.used + units <= total; });
    for (at = &d.first; *at != this; at = &(*at)->next) {}
    *at = next;
    if (mine) d.used += units;
    else units = 0;
    lk.unlock();
    u.cv.notify_all();
}

ResidentClaim::~ResidentClaim() {
    if (!units) return;
    Units& u = mtl4g::units();
    {
        std::lock_guard<std::mutex> lk(u.mu);
        u.of(device).used -= units;
    }
    u.cv.notify_all();
}

enum { ROP_NONE = 0, ROP_DIA5 = 1, ROP_DIA7 = 2, ROP_CSR8 = 3, ROP_CSR16 = 4, ROP_CSR24 = 5, ROP_LARGE = 6 };

template <typename VT, typename Op>
static int resident_go(const ResArgs& a, bool share, hipStream_t s) {
    if constexpr (Op::kOne) {
        if (!share) {
            hipLaunchKernelGGL((k_cg_resident<VT, Op, true>), dim3(1), dim3(kResBS), 0, s, a);
            M4_HIP(hipGetLastError());
            return MTL4G_OK;
        }
    }
    hipLaunchKernelGGL((k_cg_resident<VT, Op, false>), dim3(a.S.grid), dim3(kResBS), 0, s, a);
    M4_HIP(hipGetLastError());
    return MTL4G_OK;
}

ResidentPlan resident_plan(const mtl4g_matrix_s* A, int vt_bytes, int value_format, bool own_diag) {
    ResidentPlan P;
    if (A->n != A->m || A->n == 0 || reduction_order() == MTL4G_ORDER_MTL4) return P;
    const int64_t n = A->n;
    const int cus = std::min(A->cus, kResMaxGrid);
    const bool sym = A->kernel == MTL4G_SPMV_DIA_SYM;
    if (A->kernel == MTL4G_SPMV_DIA || sym) {
        const std::vector<int32_t>& off = sym ? A->h_dsym_off : A->h_dia_off;
        const int nd = (int)off.size();
        if (nd >= 2 && nd <= 7) {
            int inner = 0;
            for (int d = 1; d + 1 < nd; d++) inner = std::max(inner, std::abs(off[d]));
            int lo = std::abs(off[0]), hi = std::abs(off[nd - 1]);
            // The first diagonal is read from memory below -halo and the last one above
            // +halo, both in LDS otherwise: two diagonals far out on the same side
            // (the nearer one beyond kResHalo) fit neither.
            if (inner <= kResHalo && off[0] <= kResHalo && off[nd - 1] >= -kResHalo) {
                // the fewest rows per lane whose workgroups fit the GPU; two at
                // least (64,000 rows: 7.1 us per iteration on 63 workgroups,
                // 7.5 on 125), and one workgroup where the system fits it
                for (int rl = 1; rl <= (vt_bytes == 4 ? 4 : 3); rl++) {
                    const int64_t rows = (int64_t)kResBS << rl;
                    const int64_t g = (n + rows - 1) / rows;
                    if (g > cus || (g > 1 && n <= kResBS * 8)) continue;
                    P.op = nd <= 5 ? ROP_DIA5 : ROP_DIA7;
                    P.rows_log2 = rl;
                    P.grid = (int)g;
                    int halo = inner;
                    if (lo <= kResHalo) halo = std::max(halo, lo);
                    if (hi <= kResHalo) halo = std::max(halo, hi);
                    P.halo = halo;
                    const int64_t reach = std::max(lo, hi);
                    P.neigh = (int)std::min<int64_t>(g, (reach + rows - 1) / rows);
                    P.share = g > 1 || reach > halo;
                    return P;
                }
                // too many rows for the registers: the matrix is streamed
                // (resident_large.hip, figures there; faster than the three launches
                // at every size that fits).  Whole groups of 16 bytes, also where a
                // far diagonal reads p; other shapes keep the caller's loop.
                const int per = 16 / vt_bytes;
                const bool far = (lo <= kResHalo || lo % per == 0) && (hi <= kResHalo || hi % per == 0);
                const int groups = resident_large_groups(n, vt_bytes, cus);
                const bool types = own_diag && (value_format == MTL4G_F64) == (vt_bytes == 8);
                if (groups && types && (nd == 5 || nd == 7) && off[nd / 2] == 0 && n % per == 0 && far) {
                    const int64_t rows = (int64_t)kResBS * per * groups;
                    P.op = ROP_LARGE;
                    P.groups = groups;
                    P.grid = (int)((n + rows - 1) / rows);
                    // whole groups, so that the workgroup's own rows start on 16 bytes of the LDS
                    P.halo = std::max({inner, lo <= kResHalo ? lo : 0, hi <= kResHalo ? hi : 0});
                    P.halo = (P.halo + per - 1) / per * per;
                    P.neigh = (int)std::min<int64_t>(P.grid, (std::max(lo, hi) + rows - 1) / rows);
                    P.share = true;
                    return P;
                }
            }
        }
    }
    // one lane adds a row's products one after the other: no long rows
    if (A->max_row > 64) return P;
    for (int rl = 0; rl <= 3; rl++) {
        const int64_t rows = (int64_t)kResBS << rl;
        const int64_t g = (n + rows - 1) / rows;
        if (g > cus) continue;
        int64_t most = 0;
        for (int64_t b = 0; b < g; b++)
            most = std::max<int64_t>(most, A->h_rowptr[std::min(n, (b + 1) * rows)] - A->h_rowptr[b * rows]);
        const int64_t e = (most + kResBS - 1) / kResBS;
        if (e > 24) return P;
        P.op = e <= 8 ? ROP_CSR8 : e <= 16 ? ROP_CSR16 : ROP_CSR24;
        P.rows_log2 = rl;
        P.grid = (int)g;
        P.neigh = (int)g;
        P.share = true;
        return P;
    }
    return P;
}

mtl4g_cg_chip_info& resident_info() {
    static thread_local mtl4g_cg_chip_info info{};
    return info;
}

namespace {
// mtl4g_set_cg_chip_limits
std::atomic<int32_t> g_refuse_first{0}, g_refuse_count{0}, g_polls{0};
}  // namespace

// vectors, scalars and waits; the matrix is the launch's own
template <typename VT>
static ResArgs resident_args(const ResidentPlan& plan, const mtl4g_matrix_s* A, const void* inv_diag, int dfmt,
                             Workspace<VT>& W, VT* x) {
    ResArgs a{};
    a.n = A->n;
    a.x = x;
    a.p = W.vecs.p;
    a.r = W.vecs.p + 2 * (size_t)A->n;
    a.d = inv_diag;
    a.dfmt = dfmt;
    a.c = W.ctl.p;
    a.hist = W.hist.p;
    const int32_t polls = g_polls.load();
    a.S = ResSync{W.rslots.p, W.rwords.p, plan.grid, polls > 0 ? (unsigned)polls : kResPolls};
    return a;
}

template <typename VT>
int resident_step(int part, const ResidentPlan& plan, const mtl4g_matrix_s* A, const void* inv_diag, int dfmt,
                  Workspace<VT>& W, VT* x, hipStream_t s) {
    const ResArgs a = resident_args(plan, A, inv_diag, dfmt, W, x);
    const VT* q = W.vecs.p + (size_t)A->n;
    const int groups = plan.groups ? plan.groups : 1 << plan.rows_log2;
    auto sums = [&](auto one, auto vec) {
        if (plan.groups) hipLaunchKernelGGL(vec, dim3(plan.grid), dim3(kResBS), 0, s, a, q, groups);
        else hipLaunchKernelGGL(one, dim3(plan.grid), dim3(kResBS), 0, s, a, q, groups);
    };
    constexpr int V = 16 / (int)sizeof(VT);   // rows of a streamed layout's group
    if (part == RSTEP_P) {
        const int grid = std::min((A->n + kResBS - 1) / kResBS, 1024);
        hipLaunchKernelGGL(k_cg_step_p<VT>, dim3(grid), dim3(kResBS), 0, s, a);
    } else if (part == RSTEP_ALPHA) {
        sums(k_cg_step<VT, RSTEP_ALPHA, 1>, k_cg_step<VT, RSTEP_ALPHA, V>);
    } else if (part == RSTEP_UPDATE) {
        sums(k_cg_step<VT, RSTEP_UPDATE, 1>, k_cg_step<VT, RSTEP_UPDATE, V>);
    } else {
        // a launch of one workgroup has not set the words
        hipLaunchKernelGGL(k_resident_begin, dim3((kSlotGens * kSlotGen + 255) / 256), dim3(256), 0, s, a.S, RS_OPEN);
        sums(k_cg_step<VT, RSTEP_RESID, 1>, k_cg_step<VT, RSTEP_RESID, V>);
    }
    M4_HIP(hipGetLastError());
    return MTL4G_OK;
}

template <typename VT>
int resident_launch(const ResidentPlan& plan, const mtl4g_matrix_s* A, int fmt, const void* inv_diag, int dfmt,
                    Workspace<VT>& W, VT* x, int32_t steps, hipStream_t s) {
    if (!W.rslots.p) {
        M4_TRY(W.rslots.alloc(kSlotGens * kSlotGen));
        M4_TRY(W.rwords.alloc(kResWords));
    }
    ResArgs a = resident_args(plan, A, inv_diag, dfmt, W, x);
    const bool sym = A->kernel == MTL4G_SPMV_DIA_SYM;
    if (plan.op == ROP_DIA5 || plan.op == ROP_DIA7 || plan.op == ROP_LARGE) {
        a.doff = sym ? A->dsym_off.p : A->dia_off.p;
        a.dmap = sym ? A->dsym_map.p : nullptr;
        a.ndiag = sym ? A->ndsym : A->ndiag;
        a.nstored = sym ? A->nsym : A->ndiag;
        a.sym = sym;
        a.val = fmt == MTL4G_F64   ? (const void*)(sym ? A->dsym_val.p : A->dia_val.p)
                : fmt == MTL4G_F32 ? (const void*)(sym ? A->dsym_val32.p : A->dia_val32.p)
                                   : (const void*)(sym ? A->dsym_valbf.p : A->dia_valbf.p);
    } else {
        a.rowptr = A->rowptr.p;
        a.col = A->col.p;
        a.val = fmt == MTL4G_F64   ? (const void*)A->val.p
                : fmt == MTL4G_F32 ? (const void*)A->val32.p
                                   : (const void*)A->valbf.p;
    }
    a.fmt = fmt;
    a.halo = plan.halo;
    a.neigh = plan.neigh;
    if (plan.op == ROP_LARGE)
        steps = std::min(steps, (int32_t)std::max<int64_t>(
                                    1, kResidentSteps * kResidentVector / ((int64_t)A->n * (int64_t)sizeof(VT))));
    a.steps = resident_info().steps = steps;
    const int32_t nth = resident_info().launches++;
    if (plan.share) {
        const int32_t first = g_refuse_first.load();
        const unsigned state = nth >= first && nth - first < g_refuse_count.load() ? RS_REFUSED : RS_OPEN;
        hipLaunchKernelGGL(k_resident_begin, dim3((kSlotGens * kSlotGen + 255) / 256), dim3(256), 0, s, a.S, state);
        M4_HIP(hipGetLastError());
    }
#define M4_RES_ROWS(OP, NE)                                                                        \
    if (plan.rows_log2 == 1) return resident_go<VT, OP<VT, NE, 2>>(a, plan.share, s);              \
    if (plan.rows_log2 == 2) return resident_go<VT, OP<VT, NE, 4>>(a, plan.share, s);              \
    if constexpr (sizeof(VT) == 4 && std::is_same<OP<VT, NE, 2>, OpDia<VT, NE, 2>>::value)         \
        if (plan.rows_log2 == 4) return resident_go<VT, OpDia<VT, NE, 16>>(a, plan.share, s);      \
    return resident_go<VT, OP<VT, NE, 8>>(a, plan.share, s)
#define M4_RES_CSR(NE)                                                                             \
    if (plan.rows_log2 == 0) return resident_go<VT, OpCsr<VT, NE, 1>>(a, plan.share, s);           \
    M4_RES_ROWS(OpCsr, NE)
    switch (plan.op) {
    case ROP_DIA5: M4_RES_ROWS(OpDia, 5);
    case ROP_DIA7: M4_RES_ROWS(OpDia, 7);
    case ROP_CSR8: M4_RES_CSR(8);
    case ROP_CSR16: M4_RES_CSR(16);
    case ROP_CSR24: M4_RES_CSR(24);
    case ROP_LARGE: return resident_large_launch(a, (int)sizeof(VT), plan.groups, s);
    }
#undef M4_RES_CSR
#undef M4_RES_ROWS
    return MTL4G_ERR_INVALID;
}

template int resident_step<double>(int, const ResidentPlan&, const mtl4g_matrix_s*, const void*, int,
                                   Workspace<double>&, double*, hipStream_t);
template int resident_step<float>(int, const ResidentPlan&, const mtl4g_matrix_s*, const void*, int,
                                  Workspace<float>&, float*, hipStream_t);
template int resident_launch<double>(const ResidentPlan&, const mtl4g_matrix_s*, int, const void*, int,
                                     Workspace<double>&, double*, int32_t, hipStream_t);
template int resident_launch<float>(const ResidentPlan&, const mtl4g_matrix_s*, int, const void*, int,
                                    Workspace<float>&, float*, int32_t, hipStream_t);

}  // namespace mtl4g

using namespace mtl4g;

extern "C" {

int mtl4g_cg_chip(mtl4g_cg_chip_info* h_info) {
    if (!h_info) return MTL4G_ERR_INVALID;
    *h_info = resident_info();
    return MTL4G_OK;
}

int mtl4g_set_cg_chip_limits(int32_t refuse_first, int32_t refuse_count, int32_t polls) {
    if (refuse_first < 0 || refuse_count < 0 || polls < 0) {
        set_error("mtl4g_set_cg_chip_limits: arguments must not be negative");
        return MTL4G_ERR_INVALID;
    }
    g_refuse_first.store(refuse_first);
    g_refuse_count.store(refuse_count);
    g_polls.store(polls);
    return MTL4G_OK;
}

}  // extern "C"
