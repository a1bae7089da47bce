// resident_large.hip -- itl::cg + pc::identity / pc::diagonal (cg.hpp:38-111) on
// diagonal layouts whose values no longer fit the registers (resident.hip): the
// matrix is streamed; r and q are a lane's own (registers, and scratch where these
// run out), the workgroup's p is in LDS, and up to kLargeKeep groups per lane x and
// the inverse diagonal are kept as r is.
//
// What bounds it: memory.  Per iteration a row of the FP64 symmetric layout needs
// its 4 stored values, the far neighbours' p (2, at agent scope, past the L2), one
// write of p and, if they are streamed, the inverse diagonal and x twice: 80 bytes
// where the three-launch loop moves 136; 56 with x and the inverse diagonal kept.
// Moved past the L2 (counters): 441 MB per iteration at 160^3 where 328 are needed,
// 137 at 126^3 for 112.  The difference is scratch: with 16 groups r and q are 128
// of the 256 registers and the rest does not hold what a group in work needs, so
// the compiler stores and reloads part of r every iteration (7 diagonals: 396 bytes
// per lane at 16 groups, 256 at 14, 64 at 10, none at 9, 128 at 8 with x and the
// inverse diagonal kept).
// On top come one exchange of p and two all-reduces, about 9 us.  Measured per
// iteration, FP64, diagonal preconditioner, three launches -> here (symmetric
// layout; plain one in parentheses): 102^3 42.0 -> 15.5 us (47.8 -> 17.6), 126^3
// 59.4 -> 30.4 (71.3 -> 33.8), 140^3 76.8 -> 45.7 (92.5 -> 50.7), 160^3 105 -> 73
// (127 -> 83).  FP32 recurrence of a mixed solve, 160^3, 85 iterations and their
// refreshes: 6.5 -> 4.4 ms.
// Two groups' operands requested ahead instead of one gave nothing; non-temporal
// matrix values cost a tenth at 4.1M rows, non-temporal x and inverse diagonal
// gain a twentieth (the matrix is what the 256 MB memory-side cache can keep).
//
// A lane holds K groups of V consecutive rows (16 bytes of a vector), so the
// streams are read in 16-byte loads.  All addresses are 32-bit offsets into
// range-checked buffers, which advance by one constant per group: a row outside
// the matrix reads zeros and its stores are dropped, so no lane branches.
#include "resident_dev.hpp"

namespace mtl4g {

typedef unsigned res_u4 __attribute__((__vector_size__(4 * sizeof(unsigned int))));
typedef unsigned res_u2 __attribute__((__vector_size__(2 * sizeof(unsigned int))));
template <typename VT>
struct ResVec;
template <>
struct ResVec<double> {
    typedef double type __attribute__((ext_vector_type(2)));
};
template <>
struct ResVec<float> {
    typedef float type __attribute__((ext_vector_type(4)));
};
constexpr int kResSc1 = 16;   // buffer cache policy: agent scope, as ld_agent / st_agent
constexpr int kResNt = 2;     // non-temporal: streamed once per iteration
// Groups per lane up to which x and the inverse diagonal are kept: four arrays of 16
// bytes per group, 128 of a lane's 256 registers.  At 8 groups (126^3) 30.4 us per
// iteration against 33 with both streamed, although 128 bytes per lane go to scratch;
// more groups kept were not measured.
constexpr int kLargeKeep = 8;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t res_rsrc(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, __builtin_amdgcn_readfirstlane(bytes),
                                             0x00020000);
}
template <int B, int AUX>
struct ResRaw;   // B bytes of a buffer as stored elements
template <int AUX>
struct ResRaw<16, AUX> {
    static __device__ __forceinline__ res_u4 ld(__amdgpu_buffer_rsrc_t r, int o) {
        return __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, AUX);
    }
};
template <int AUX>
struct ResRaw<8, AUX> {
    static __device__ __forceinline__ res_u2 ld(__amdgpu_buffer_rsrc_t r, int o) {
        return __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, AUX);
    }
};
template <int AUX>
struct ResRaw<4, AUX> {
    static __device__ __forceinline__ unsigned ld(__amdgpu_buffer_rsrc_t r, int o) {
        return __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, AUX);
    }
};
template <int AUX>
struct ResRaw<2, AUX> {
    static __device__ __forceinline__ unsigned short ld(__amdgpu_buffer_rsrc_t r, int o) {
        return __builtin_amdgcn_raw_buffer_load_b16(r, o, 0, AUX);
    }
};

// SYM: the symmetric copy; diagonals below the main one are mirrored
template <typename VT, typename MT, int ND, int K, bool SYM>
__global__ __launch_bounds__(kResBS) void k_cg_large(ResArgs a) {
    constexpr int V = 16 / (int)sizeof(VT), VB = (int)sizeof(VT), MB = (int)sizeof(MT);
    constexpr int STEP = kResBS * V, OWN = K * STEP;   // rows between a lane's groups; of the workgroup
    constexpr bool KEEP = K <= kLargeKeep;
    static_assert(STEP % kWave == 0, "a lane keeps its place in the slices of 64 rows");
    using VV = typename ResVec<VT>::type;
    struct MV {
        MT v[V];
    };
    __shared__ __align__(16) VT lds[OWN + 2 * kResHalo];
    __shared__ ResShared<VT> sh;
    __shared__ int flag;
    const int t = (int)threadIdx.x;
    const int G = a.S.grid, n = a.n;
    int lb = (int)blockIdx.x;
    if (G % kXcd == 0) lb = xcd_logical_block(lb, G / kXcd);
    const int row0 = lb * OWN, first_row = row0 + t * V;
    if (a.c->done || a.c->pause || a.c->want_ru) return;   // the whole grid reads the same state
    ResLoop<VT> L;
    L.init(a.c);
    const __amdgpu_buffer_rsrc_t bx = res_rsrc(a.x, n * VB), br = res_rsrc(a.r, n * VB), bp = res_rsrc(a.p, n * VB);
    const __amdgpu_buffer_rsrc_t bd = res_rsrc(a.d, a.d ? n * VB : 0);
    const int slices = (n + kWave - 1) / kWave;
    const __amdgpu_buffer_rsrc_t bm = res_rsrc(a.val, slices * a.nstored * kWave * MB);
    const bool ident = a.d == nullptr;
    const int halo = a.halo;
    int off[ND];
    int at[ND], at2[SYM ? ND / 2 : 1];   // offsets of the lane's first group; of its last row (mirrored diagonals)
    bool whole[SYM ? ND / 2 : 1];        // a mirrored diagonal whose V values are one load
    const int adv = STEP * a.nstored * MB;   // from one group to the next
    auto place = [&](int row, int st) {      // slice-major; a row before the first is out of the buffer's range
        const int s = row >= 0 ? row / kWave : -((kWave - 1 - row) / kWave);
        return ((s * a.nstored + st) * kWave + (row - s * kWave)) * MB;
    };
#pragma unroll
    for (int d = 0; d < ND; d++) {
        off[d] = __builtin_amdgcn_readfirstlane(a.doff[d]);
        const int st = SYM ? __builtin_amdgcn_readfirstlane(a.dmap[d]) : d;
        if (SYM && d < ND / 2) {
            whole[d] = off[d] % V == 0;
            at[d] = place(first_row + off[d], st);
            at2[d] = place(first_row + off[d] + V - 1, st);
        } else {
            at[d] = place(first_row, st);
        }
    }
    const bool flo = off[0] < -halo, fhi = off[ND - 1] > halo;
    VT* mine = lds + halo + t * V;   // on 16 bytes: the halo is whole groups
    VV r[K], q[K];   // q holds z between the update and the next direction
    VV xk[KEEP ? K : 1], dk[KEEP ? K : 1];
    // The lane's places are made opaque at the head of each phase: offsets are
    // then formed where they are used (one addition) instead of living in
    // registers, K of them per stream, for the whole kernel.
    int row_at = first_row * VB;
    auto fresh = [&]() {
        asm volatile("" : "+v"(row_at));
#pragma unroll
        for (int d = 0; d < ND; d++) asm volatile("" : "+v"(at[d]));
    };
    auto ldv = [&](__amdgpu_buffer_rsrc_t b, int k) -> VV {
        return __builtin_bit_cast(VV, __builtin_amdgcn_raw_buffer_load_b128(b, row_at + k * (STEP * VB), 0, kResNt));
    };
#pragma unroll
    for (int k = 0; k < K; k++) {
        r[k] = ldv(br, k);
        VV p = ldv(bp, k);
        if (L.first) p = VV(VT(0));
        *reinterpret_cast<VV*>(mine + k * STEP) = p;
        const VV d = ident ? VV(VT(1)) : ldv(bd, k);
        q[k] = ident ? r[k] : d * r[k];
        if (KEEP) {
            xk[KEEP ? k : 0] = ldv(bx, k);
            dk[KEEP ? k : 0] = d;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if (!res_meet(a.S, &flag)) {
        if (blockIdx.x == 0 && t == 0) a.c->refused++;
        return;
    }
    struct Group {
        MV m[ND];
        VV lo, hi;     // p at the first / last diagonal when it lies beyond the halo
    };
    auto fetch = [&](int k, Group& o) {
#pragma unroll
        for (int d = 0; d < ND; d++) {
            if (!(SYM && d < ND / 2) || whole[SYM && d < ND / 2 ? d : 0]) {
                o.m[d] = __builtin_bit_cast(MV, ResRaw<V * MB, 0>::ld(bm, at[d] + k * adv));
            } else {
                // one load per row: the group may lie in two slices, whose places
                // then count up from the first row's and down from the last one's
                const bool split = at2[d] - at[d] != (V - 1) * MB;
                const int in1 = split ? kWave - (at[d] / MB & (kWave - 1)) : V;
#pragma unroll
                for (int v = 0; v < V; v++) {
                    const int o1 = v < in1 ? at[d] + v * MB : at2[d] - (V - 1 - v) * MB;
                    o.m[d].v[v] = __builtin_bit_cast(MT, ResRaw<MB, 0>::ld(bm, o1 + k * adv));
                }
            }
        }
        if (flo) o.lo = __builtin_bit_cast(VV, ResRaw<16, kResSc1>::ld(bp, row_at + (off[0] + k * STEP) * VB));
        if (fhi) o.hi = __builtin_bit_cast(VV, ResRaw<16, kResSc1>::ld(bp, row_at + (off[ND - 1] + k * STEP) * VB));
    };
    auto sum = [&](int k, const Group& o) -> VV {
        VV acc;
#pragma unroll
        for (int v = 0; v < V; v++) {
            VT s = VT(0);
#pragma unroll
            for (int d = 0; d < ND; d++) {
                const bool lo = d == 0 && flo, hi = d == ND - 1 && fhi;
                const VT g = lo ? o.lo[v] : hi ? o.hi[v] : mine[k * STEP + (lo || hi ? 0 : off[d]) + v];
                const VT with = s + dia_value<VT>(o.m[d].v[v]) * g;
                s = dia_absent(o.m[d].v[v]) ? s : with;
            }
            acc[v] = s;
        }
        return acc;
    };
    bool ok = true;
    unsigned step = 0;
    int gen = 0;
    for (;;) {
        // p = z  or  p = z + beta*p  (cg.hpp:98-101)
        fresh();
#pragma unroll
        for (int k = 0; k < K; k++) {
            VV* own = reinterpret_cast<VV*>(mine + k * STEP);
            const VV p = L.first ? q[k] : q[k] + L.beta * *own;
            *own = p;
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(res_u4, p), bp, row_at + k * (STEP * VB), 0,
                                                   kResSc1);
            __builtin_amdgcn_sched_barrier(0);
        }
        step++;
        ok = res_exchange(a.S, lb, a.neigh, step, &flag);
        if (!ok) break;
        // the neighbours' rows next to this workgroup's
        VT h[2 * kResHalo / kResBS];
#pragma unroll
        for (int i = 0; i < 2 * kResHalo / kResBS; i++) {
            const int j = t + i * kResBS;
            const int row = j < halo ? row0 - halo + j : row0 + OWN + j - halo;
            h[i] = __builtin_bit_cast(VT, ResRaw<VB, kResSc1>::ld(bp, j < 2 * halo ? row * VB : n * VB));
        }
#pragma unroll
        for (int i = 0; i < 2 * kResHalo / kResBS; i++) {
            const int j = t + i * kResBS;
            if (j < 2 * halo) lds[j < halo ? j : OWN + j] = h[i];
        }
        __syncthreads();
        // q = A*p, p.q; alpha  (cg.hpp:103-105)
        VT s0 = VT(0), s1 = VT(0);
#pragma unroll
        for (int k = 0; k < K; k++) {
            // one group's loads per wave; the eight waves of a CU keep 74 KB in
            // flight together
            fresh();
            Group g;
            fetch(k, g);
            __builtin_amdgcn_sched_barrier(0);
            q[k] = sum(k, g);
            asm volatile("" : "+v"(q[k]));   // formed here: sunk to its use, the operands of all groups would stay live
            const VV p = *reinterpret_cast<const VV*>(mine + k * STEP);
#pragma unroll
            for (int v = 0; v < V; v++) s0 += p[v] * q[k][v];
            __builtin_amdgcn_sched_barrier(0);
        }
        constexpr int C = 3;   // groups of x and d requested together, one such chunk ahead
        VV x[2][C], d[2][C];
        auto fetch_xd = [&](int k0) {
            fresh();
#pragma unroll
            for (int u = 0; u < C; u++)
                if (k0 + u < K) {
                    x[k0 / C & 1][u] = ldv(bx, k0 + u);
                    if (!ident) d[k0 / C & 1][u] = ldv(bd, k0 + u);
                }
            __builtin_amdgcn_sched_barrier(0);
        };
        if (!KEEP) fetch_xd(0);   // under way during the all-reduce
        ok = res_allsum<VT, false>(a.S, gen++, s0, VT(0), sh, L.pq, s1);
        if (!ok) break;
        L.direction();
        // x += alpha*p; r -= alpha*q; r.r, r.(d.*r)  (cg.hpp:106-108)
        s0 = s1 = VT(0);
#pragma unroll
        for (int k0 = 0; k0 < K; k0 += C) {
            if (!KEEP && k0 + C < K) fetch_xd(k0 + C);
#pragma unroll
            for (int u = 0; u < C; u++)
                if (k0 + u < K) {
                    const int k = k0 + u, in = k0 / C & 1;
                    const VV p = *reinterpret_cast<const VV*>(mine + k * STEP);
                    r[k] = r[k] - L.alpha * q[k];
                    if constexpr (KEEP) {
                        xk[k] = xk[k] + L.alpha * p;
                        q[k] = dk[k] * r[k];
                    } else {
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(res_u4, x[in][u] + L.alpha * p), bx,
                                                               row_at + k * (STEP * VB), 0, kResNt);
                        q[k] = ident ? r[k] : d[in][u] * r[k];
                    }
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        s0 += r[k][v] * r[k][v];
                        s1 += r[k][v] * q[k][v];
                    }
                    asm volatile("" : "+v"(r[k]), "+v"(q[k]), "+v"(s0), "+v"(s1));   // formed here, as in the product
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        ok = res_allsum<VT, false>(a.S, gen++, s0, s1, sh, L.rr, L.rz);
        if (!ok) break;
        if (L.head(a.hist, blockIdx.x == 0 && t == 0) || (int)step >= a.steps) break;
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        if (KEEP)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(res_u4, xk[KEEP ? k : 0]), bx,
                                                   row_at + k * (STEP * VB), 0, 0);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(res_u4, r[k]), br, row_at + k * (STEP * VB), 0, 0);
    }   // p is in memory since the last exchange
    if (blockIdx.x == 0 && t == 0) L.leave(a.c, ok);
}

// Groups per lane that are built: a size takes the fewest that fit the GPU, so
// that the workgroups left without rows are few (2.7M FP64 rows: 51 us per
// iteration with 13 groups on 206 CUs, 45 with 11 on 244).
template <typename VT>
struct LargeGroups;
template <>
struct LargeGroups<double> {
    static constexpr int v[] = {5, 6, 7, 8, 9, 10, 11, 12, 14, 16};
};
template <>
struct LargeGroups<float> {
    static constexpr int v[] = {6, 8, 10, 12, 14, 16};
};
template <typename VT>
static int large_groups(int64_t n, int cus) {
    for (int k : LargeGroups<VT>::v)
        if ((int64_t)kResBS * (16 / (int)sizeof(VT)) * k * cus >= n) return k;
    return 0;
}
int resident_large_groups(int64_t n, int vt_bytes, int cus) {
    return vt_bytes == 8 ? large_groups<double>(n, cus) : large_groups<float>(n, cus);
}

template <typename VT, typename MT, int ND, bool SYM, int I = 0>
static int large_go(const ResArgs& a, int groups, hipStream_t s) {
    if constexpr (I < (int)(sizeof(LargeGroups<VT>::v) / sizeof(int))) {
        constexpr int K = LargeGroups<VT>::v[I];
        if (groups != K) return large_go<VT, MT, ND, SYM, I + 1>(a, groups, s);
        hipLaunchKernelGGL((k_cg_large<VT, MT, ND, K, SYM>), dim3(a.S.grid), dim3(kResBS), 0, s, a);
        M4_HIP(hipGetLastError());
        return MTL4G_OK;
    }
    return MTL4G_ERR_INVALID;
}
template <typename VT, typename MT>
static int large_layout(const ResArgs& a, int groups, hipStream_t s) {
    if (a.ndiag == 5) return a.sym ? large_go<VT, MT, 5, true>(a, groups, s) : large_go<VT, MT, 5, false>(a, groups, s);
    if (a.ndiag == 7) return a.sym ? large_go<VT, MT, 7, true>(a, groups, s) : large_go<VT, MT, 7, false>(a, groups, s);
    return MTL4G_ERR_INVALID;
}
int resident_large_launch(const ResArgs& a, int vt_bytes, int groups, hipStream_t s) {
    if (vt_bytes == 8 && a.fmt == MTL4G_F64) return large_layout<double, double>(a, groups, s);
    if (vt_bytes == 4 && a.fmt == MTL4G_F32) return large_layout<float, float>(a, groups, s);
    if (vt_bytes == 4 && a.fmt == MTL4G_BF16) return large_layout<float, uint16_t>(a, groups, s);
    return MTL4G_ERR_INVALID;
}

}  // namespace mtl4g
