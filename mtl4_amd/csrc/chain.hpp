// chain.hpp -- triangular sweeps of grid-structured factors as a pipeline of
// row chains (included by precond.hip).
//
// A triangular factor whose rows depend only on the rows 1, Lc and Lc*Cx
// before them (after them, for an upper factor), with no dependency across
// the edge of a chain of Lc rows or of a plane of Cx chains -- the IC(0) /
// ILU(0) factors of 5- and 7-point stencils in natural order -- is swept
// chain by chain: chain (cx, cy) (rows (cy*Cx + cx)*Lc .. +Lc) handles its
// element e at step e + cx + cy.  A workgroup owns a tile of Tx x Ty = 64
// chains and has five waves: one computes, a lane per chain with the chain's
// last element in a register; the others move data, so that no address, load
// or store stands in the computing wave's way.  Inside a tile the chains cx-1
// and cy-1 hand over their element of the previous step lane to lane (DPP,
// ds_bpermute), between tiles through memory (the tile's last chains' rows in
// exchange slots, polled while they are empty).  The waves meet at one barrier
// per block of U steps.
//
// Memory access is coalesced although the chains' rows lie Lc apart: the
// factor's values are stored tile by tile in step-major order (slot =
// tile*stile + (step - first step of the tile)*64 + lane), so a block's values
// are contiguous and go to LDS directly, three blocks ahead; the input and
// output vectors keep their natural order and move through LDS in blocks of U
// steps (8 consecutive rows of a chain per 8 lanes).  Every row is computed by
// one lane with MTL4's subtraction order (ascending columns,
// lower_trisolve.hpp:174-209, upper_trisolve.hpp:161-176), so the results are
// the level-scheduled sweep's bit for bit.
#pragma once

#include <vector>

#include "kernels.hpp"

namespace mtl4g {

constexpr int kChainU = 8;       // steps per block (4: 0.49 ms instead of 0.43 for two 160^3 sweeps)
constexpr int kChainPad = 8;     // LDS row padding of the staging arrays (bank spread)
constexpr int kChainStages = 4;  // blocks of factor values in LDS
constexpr int kChainAhead = 4;   // blocks of v in flight or staged
constexpr int kChainTail = kChainU * kWave;   // value slots past the last tile's (its last block reads them)

struct ChainSweep {
    bool lower = true, unit = false;
    bool holes = false;             // rows inside the grid that lack one of the offsets: absent entries are marked
    int32_t n = 0, Lc = 0, Cx = 0, Cy = 0;
    int ndep = 0;                   // 1..3 offsets: 1, Lc, Lc*Cx
    int Tx = 64, Ty = 1, tiles_x = 1, tiles_y = 1;
    int64_t stile = 0, nslots = 0;  // slots per tile, slots in all
    int64_t xy = 0, xtile = 0;      // exchange slots of a tile: its last chains in x, then in y; in all
    DevBuf<int32_t> src, dsrc;      // gathered values: positions in the device factor (-1: absent / unit)
    DevBuf<double> val64, dia64;    // val: ndep arrays of nslots (entry of offset k)
    DevBuf<float> val32, dia32;
    DevBuf<uint16_t> val16, dia16;
};

template <typename MT>
struct ChainView {
    const MT* val;   // ndep * nslots, tile-local step-major
    const MT* dia;   // nslots (unused for a unit sweep)
    int32_t n, Lc, Cx, Cy, Tx, Ty, tiles_x, stile, nslots;
    int32_t holes;
    int64_t xtile, xy;
};

// Counters of a launch: ticket, abort flag, finished tiles; then the exchange
// slots (Sweep::words).
constexpr size_t chain_counter_words = 4 * kCounterStride;

// Slot of row r of the sweep's own index (rm = r for a lower sweep,
// n-1-r for an upper one) in the tile-local step-major layout.
__host__ __device__ inline int64_t chain_slot(int64_t rm, int64_t Lc, int64_t Cx, int64_t Tx, int64_t Ty,
                                              int64_t tiles_x, int64_t stile) {
    const int64_t e = rm % Lc, q = rm / Lc, cx = q % Cx, cy = q / Cx;
    const int64_t tx = cx / Tx, ty = cy / Ty;
    const int64_t l = (cy - ty * Ty) * Tx + (cx - tx * Tx);
    return (ty * tiles_x + tx) * stile + (e + cx + cy - tx * Tx - ty * Ty) * (Tx * Ty) + l;
}

// A row handed to another tile travels in an exchange slot as its bits xor
// this signalling-NaN pattern, which no row's result is: an empty slot is 0,
// the state the one tile that reads the slot leaves it in.
constexpr unsigned long long kChainEmpty = 0x7ff5c3c3c3c3c3c3ull;

// Buffer (descriptor-based) loads and stores: an offset past the buffer's
// size reads zero and drops a store, so lanes without a row this step run
// the same straight-line code as the others and every load keeps its place
// in the memory counter (vmcnt) -- the loads issued for later steps stay in
// flight across the steps in between.
typedef unsigned int chain_u2 __attribute__((__vector_size__(2 * sizeof(unsigned int))));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t chain_rsrc(const void* p, int32_t bytes) {
    // raw buffer: stride 0, 32-bit data format (the fourth descriptor word
    // of gfx9 buffers).  Every input is wave-uniform; readfirstlane keeps the
    // descriptor in scalar registers (a descriptor in vector registers makes
    // the compiler loop over the lanes' values around every access).  The
    // host admits a layout only when its largest buffer fits an int32.
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0,
                                             __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}
// off: per-lane byte offset, range-checked against the buffer's size
template <typename T>
__device__ __forceinline__ T chain_ld(__amdgpu_buffer_rsrc_t r, int32_t off);
template <>
__device__ __forceinline__ double chain_ld<double>(__amdgpu_buffer_rsrc_t r, int32_t off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
template <>
__device__ __forceinline__ float chain_ld<float>(__amdgpu_buffer_rsrc_t r, int32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// The value v of lane l-1 (lane 0: its own `edge`), for every lane: a DPP
// shift of the whole wave by one lane, no LDS.
__device__ __forceinline__ double chain_from_prev_lane(double v, double edge) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned long long e = (unsigned long long)__double_as_longlong(edge);
    const unsigned lo =
        (unsigned)__builtin_amdgcn_update_dpp((int)(unsigned)e, (int)(unsigned)b, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
    const unsigned hi =
        (unsigned)__builtin_amdgcn_update_dpp((int)(unsigned)(e >> 32), (int)(unsigned)(b >> 32), 0x138, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The value v of lane src (src4 = 4*src), for every lane: two ds_bpermute
// (the LDS crossbar, no LDS storage).
__device__ __forceinline__ double chain_from(double v, int src4) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_ds_bpermute(src4, (int)(unsigned)b);
    const unsigned hi = (unsigned)__builtin_amdgcn_ds_bpermute(src4, (int)(unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// A barrier between the waves of a tile that orders their LDS traffic only:
// global loads and stores stay in flight across it.
__device__ __forceinline__ void chain_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// wait until at most N vector memory operations of this wave are in flight
template <int N>
__device__ __forceinline__ void chain_wait_vm() {
    static_assert(N >= 0 && N < 64, "the wait counter has six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// The pipeline kernel, one workgroup of five waves per tile.  LOWER: rows
// depend on smaller rows (else on larger ones: the sweep runs in the mirrored
// index r' = n-1-r).  NDEP offsets; UNIT: no diagonal factor.  v is read as
// IT, every result is kept in w (double) and, when w32 is given, rounded to
// float there too.
//
// Lanes without a row this step compute on padding (v = 0, values 0, diagonal
// 1).  Where the grid has no holes an absent entry is one at the grid's edge:
// its value is stored as 0 and its operand is +0 (the padding before a chain's
// first element, the zeros handed to the tiles of the first chains), and
// subtracting the product +0 leaves every value's bits as they are, so the
// computing wave tests nothing.  With holes the absent entries are marked and
// their subtraction is dropped by a select.
//
// What bounds it: the dependent chain of a step in one wave (exchange, NDEP
// products and differences, the scale: 45 ns per step on a one-tile 2-D grid,
// 92 ns on a 3-D one, of which the lane exchange through the LDS crossbar is
// half) and, per tile on the longest path, the hand-over of about 4 us: a block
// of steps, the store, the poll.  One wave that also moved its data took 184 ns
// per step.  solve(P, x), two sweeps with their calls: IC(0) 160^3 0.90 -> 0.43
// ms, ILU(0) 1024^2 1.01 -> 0.34 ms.
template <typename MT, typename IT, bool LOWER, bool UNIT, int NDEP>
__global__ __launch_bounds__(5 * kWave) void k_chain(ChainView<MT> C, const IT* __restrict__ v, double* w, float* w32,
                                                     unsigned* counters, int* err, const int* skip) {
    constexpr int U = kChainU, ST = kChainStages, AH = kChainAhead;
    constexpr int RW = kWave + kChainPad;    // staging row: one step of the block, all chains
    constexpr int NARR = NDEP + (UNIT ? 0 : 1);
    if (skip && *skip) return;
    __shared__ __align__(16) MT vals[ST][NARR][U * kWave];   // factor values: [step][chain]; the diagonal last
    __shared__ double vst[2][U * RW];        // v of a block: [step][chain]
    __shared__ double wst[2][U * RW];        // results of a block
    __shared__ double exs[2][U * kWave], eys[2][U * kWave];   // other tiles' rows: [gy][step], [gx][step]
    __shared__ int s_tile;
    const int l = threadIdx.x & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    if (threadIdx.x == 0)
        s_tile = (int)__hip_atomic_fetch_add(counters, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int tile = __builtin_amdgcn_readfirstlane(s_tile);   // tiles in row-major order: producers first
    const int tx = tile % C.tiles_x, ty = tile / C.tiles_x;
    const int x0 = tx * C.Tx, y0 = ty * C.Ty;
    const int32_t Lc = C.Lc, n = C.n;
    const int xl = min(C.Cx, x0 + C.Tx) - 1, yl = min(C.Cy, y0 + C.Ty) - 1;
    const int s0 = x0 + y0, s1 = (Lc - 1) + xl + yl;
    const int nblk = (s1 - s0 + U) / U;                  // blocks of steps
    const int niter = (nblk + AH - 1) / AH * AH;         // barriers: the movers run AH blocks per turn
    constexpr int32_t kOut = 0x7ffffff0;                 // an offset past every buffer
    unsigned* abort_flag = counters + kCounterStride;
    unsigned long long* slots = reinterpret_cast<unsigned long long*>(counters + chain_counter_words);
    auto row_of = [=](int32_t rm) -> int32_t { return LOWER ? rm : n - 1 - rm; };
    // Block staging: lane l moves element jj = l % U of the chains
    // c = l/U + (64/U)*i (i < U) between the natural-order vectors and LDS.  The
    // element at block k is first + U*k (first: far below 0 where there is no
    // chain), its row at + rowdir * U*k; both parts that depend on the lane are
    // formed once.
    const int jj = l % U;
    constexpr int rowdir = LOWER ? 1 : -1;
    struct Place {
        int32_t first, row;
    };
    auto place = [=](int ccx, int ccy, int step, bool there) -> Place {
        const int e = s0 + step - ccx - ccy;
        return Place{there ? e : INT32_MIN / 2, row_of((ccy * C.Cx + ccx) * Lc + e)};
    };
    // byte offset (times B) of the element of block k, past every buffer when the chain has none
    auto offset = [=](const Place& p, int k, int B) -> int32_t {
        const bool ok = (unsigned)(p.first + k * U) < (unsigned)Lc;
        return ok ? (p.row + rowdir * k * U) * B : kOut;
    };
    // Rows handed between tiles.  Item q of a block: step j = q / T, chain
    // g = q % T of the T = Ty chains at the tile's x edge or the T = Tx chains
    // at its y edge; `back` steps behind the tile's first chains on the giving
    // side, 0 on the taking side.  Its element at block k is first + U*k, its
    // slot at + U*T*k: a block's slots are contiguous.
    struct Item {
        int32_t first, slot, j, g, T;
        bool own;
    };
    auto item = [=](bool y, int q, int back, bool there) -> Item {
        const int T = y ? C.Tx : C.Ty, j = q / T, g = q % T;
        const bool ok = there && q < T * U && (y ? x0 + g < C.Cx : y0 + g < C.Cy);
        return Item{ok ? j - back - g : INT32_MIN / 2, (j - back) * T + g, j, g, T, q < T * U};
    };
    unsigned long long* from_x = slots + (int64_t)(tile - 1) * C.xtile;                  // read when tx > 0
    unsigned long long* from_y = slots + (int64_t)(tile - C.tiles_x) * C.xtile + C.xy;   // read when ty > 0
    // every item of a block has a lane
    const bool few = C.Ty * U <= kWave && (NDEP < 3 || C.Tx * U <= kWave);
    if (wv == 1) {
        // ---- factor values to LDS.  Bare barriers: a fence would wait for the
        // blocks that are still on their way; the block the others read next
        // has arrived when the counter says so.
        constexpr int PER = 16 / (int)sizeof(MT);                    // values per lane and load
        constexpr int NL = U / PER;                                  // loads per array and block
        static_assert(U % PER == 0, "whole loads per array");
        static_assert((ST - 1) * NARR * NL < 64, "blocks in flight within the wait counter");
        auto issue = [&](int k) {
            const int kb = min(k, nblk - 1);
            const int64_t at = (int64_t)tile * C.stile + (int64_t)kb * (U * kWave) + l * PER;
#pragma unroll
            for (int q = 0; q < NARR; q++) {
                const MT* src = q < NDEP ? C.val + (int64_t)q * C.nslots + at : C.dia + at;
#pragma unroll
                for (int i = 0; i < NL; i++)
                    __builtin_amdgcn_global_load_lds(
                        (const __attribute__((address_space(1))) void*)(src + i * PER * kWave),
                        (__attribute__((address_space(3))) void*)&vals[k % ST][q][i * PER * kWave], 16, 0, 0);
            }
        };
#pragma unroll
        for (int k = 0; k < ST; k++) issue(k);
        chain_wait_vm<(ST - 2) * NARR * NL>();   // blocks 0 and 1 are there
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_barrier();            // block 0 is in the computing wave's registers
        for (int k = 0; k < niter; k++) {
            issue(k + ST);                       // the stage of block k, which is in registers
            chain_wait_vm<(ST - 2) * NARR * NL>();   // block k + 2 is there
            __builtin_amdgcn_s_barrier();
        }
        chain_wait_vm<0>();
    } else if (wv == 2) {
        // ---- v to LDS
        const __amdgpu_buffer_rsrc_t rv_ = chain_rsrc(v, n * (int32_t)sizeof(IT));
        Place at[U];
#pragma unroll
        for (int i = 0; i < U; i++) {
            const int c = l / U + i * (kWave / U), ccx = x0 + c % C.Tx, ccy = y0 + c / C.Tx;
            at[i] = place(ccx, ccy, jj, (ccx < C.Cx) & (ccy < C.Cy));
        }
        IT vin[AH][U];
        auto issue = [&](int k, IT(&to)[U]) {
#pragma unroll
            for (int i = 0; i < U; i++) to[i] = chain_ld<IT>(rv_, offset(at[i], k, (int)sizeof(IT)));
        };
        auto stage = [&](int k, const IT(&from)[U]) {
            double vi[U];
#pragma unroll
            for (int i = 0; i < U; i++) vi[i] = static_cast<double>(from[i]);
            // with holes a result can be v itself (nothing subtracted, unit
            // diagonal) and must not be the empty pattern; otherwise the
            // subtractions quiet it
            if (C.holes)
#pragma unroll
                for (int i = 0; i < U; i++)
                    if ((unsigned long long)__double_as_longlong(vi[i]) == kChainEmpty)
                        vi[i] = __longlong_as_double((long long)(kChainEmpty | 0x0008000000000000ull));
#pragma unroll
            for (int i = 0; i < U; i++) vst[k & 1][jj * RW + l / U + i * (kWave / U)] = vi[i];
        };
#pragma unroll
        for (int u = 0; u < AH; u++) issue(u, vin[u]);
        stage(0, vin[0]);
        issue(AH, vin[0]);
        stage(1, vin[1]);
        issue(AH + 1, vin[1]);
        chain_barrier();
        chain_barrier();
        for (int k = 0; k < niter; k += AH)
#pragma unroll
            for (int u = 0; u < AH; u++) {
                stage(k + u + 2, vin[(u + 2) % AH]);
                issue(k + u + 2 + AH, vin[(u + 2) % AH]);
                __builtin_amdgcn_sched_barrier(0);
                chain_barrier();
            }
    } else if (wv == 3) {
        // ---- results, one block behind: first those of the tile's last
        // chains to the exchange slots of the tiles that wait for them
        // (agent-scope stores, no announcement: a slot's value and its
        // validity are one 8-byte write), then all to w
        const __amdgpu_buffer_rsrc_t rw = chain_rsrc(w, n * 8);
        // no w32: a descriptor of size 0, every store through it is dropped
        const __amdgpu_buffer_rsrc_t rw32 = chain_rsrc(w32, w32 ? n * 4 : 0);
        Place at[U];
#pragma unroll
        for (int i = 0; i < U; i++) {
            const int c = l / U + i * (kWave / U), ccx = x0 + c % C.Tx, ccy = y0 + c / C.Tx;
            at[i] = place(ccx, ccy, jj, (ccx < C.Cx) & (ccy < C.Cy));
        }
        const bool give_x = NDEP >= 2 && tx + 1 < C.tiles_x, give_y = NDEP >= 3 && (ty + 1) * C.Ty < C.Cy;
        const Item ix = item(false, l, C.Tx - 1, give_x), iy = item(true, l, C.Ty - 1, give_y);
        unsigned long long *to_x = slots + (int64_t)tile * C.xtile, *to_y = to_x + C.xy;
        auto hand_one = [&](const Item& it, unsigned long long* to, int k, int lds) {
            const int e = it.first + k * U;
            if ((unsigned)e < (unsigned)Lc)
                st_agent(to + (it.slot + k * U * it.T),
                         (unsigned long long)__double_as_longlong(wst[k & 1][lds]) ^ kChainEmpty);
        };
        const int lx = ix.j * RW + ix.g * C.Tx + C.Tx - 1, ly = iy.j * RW + (C.Ty - 1) * C.Tx + iy.g;
        auto hand = [&](int k) {
            if (give_x) hand_one(ix, to_x, k, lx);
            if (give_y) hand_one(iy, to_y, k, ly);
            if (few) return;
            for (int q = l + kWave; q < C.Ty * U && give_x; q += kWave) {
                const Item it = item(false, q, C.Tx - 1, true);
                hand_one(it, to_x, k, it.j * RW + it.g * C.Tx + C.Tx - 1);
            }
            for (int q = l + kWave; q < C.Tx * U && give_y; q += kWave) {
                const Item it = item(true, q, C.Ty - 1, true);
                hand_one(it, to_y, k, it.j * RW + (C.Ty - 1) * C.Tx + it.g);
            }
        };
        const Item ex = item(false, l, 0, tx > 0), ey = item(true, l, 0, NDEP >= 3 && ty > 0);
        auto empty_one = [&](const Item& it, unsigned long long* from, int k) {
            if ((unsigned)(it.first + k * U) < (unsigned)Lc) st_agent(from + (it.slot + k * U * it.T), 0ull);
        };
        auto empty = [&](int k) {
            if (NDEP >= 2) empty_one(ex, from_x, k);
            if (NDEP >= 3) empty_one(ey, from_y, k);
            if (few) return;
            for (int q = l + kWave; q < C.Ty * U; q += kWave) empty_one(item(false, q, 0, tx > 0), from_x, k);
            for (int q = l + kWave; NDEP >= 3 && q < C.Tx * U; q += kWave) empty_one(item(true, q, 0, ty > 0), from_y, k);
        };
        auto store = [&](int k) {
            if (k < 0 || k >= nblk) return;
            double r[U];
#pragma unroll
            for (int i = 0; i < U; i++) r[i] = wst[k & 1][jj * RW + l / U + i * (kWave / U)];
            hand(k);
#pragma unroll
            for (int i = 0; i < U; i++)
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(chain_u2, r[i]), rw, offset(at[i], k, 8), 0, 0);
            if (w32)
#pragma unroll
                for (int i = 0; i < U; i++)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (float)r[i]), rw32,
                                                          offset(at[i], k, 4), 0, 0);
            // the slots this tile has read for block k are empty again (here and
            // not where they are read: a load would wait for these stores)
            empty(k);
        };
        chain_barrier();
        chain_barrier();
        for (int k = 0; k < niter; k++) {
            store(k - 1);
            chain_barrier();
        }
        store(niter - 1);
    } else if (wv == 4) {
        // ---- rows of the tiles before this one (chain cx-1 of gx = 0, chain
        // cy-1 of gy = 0), from their exchange slots, which are emptied again.
        // Item q as in hand(): element e of the neighbour chain for element e
        // here.  Items without a row are not read and are +0.
        const Item ix = item(false, l, 0, tx > 0), iy = item(true, l, 0, NDEP >= 3 && ty > 0);
        auto look = [&](const Item& it, const unsigned long long* from, int k) -> unsigned long long {
            return (unsigned)(it.first + k * U) < (unsigned)Lc ? ld_agent(from + (it.slot + k * U * it.T)) : 0ull;
        };
        auto finish = [&](const Item& it, const unsigned long long* from, int k, unsigned long long b, double* to) {
            double x = 0.0;
            if ((unsigned)(it.first + k * U) < (unsigned)Lc) {
                const unsigned long long* at = from + (it.slot + k * U * it.T);
                unsigned polls = 0;
#pragma clang loop unroll(disable)
                while (b == 0ull) {
                    if (++polls > (1u << 22) || ((polls & 63u) == 0 && ld_agent(abort_flag) != 0u)) {
                        st_agent(abort_flag, 1u);
                        break;
                    }
                    b = ld_agent(at);
                }
                x = __longlong_as_double((long long)(b ^ kChainEmpty));
            }
            if (it.own) to[it.g * U + it.j] = x;
        };
        // Both kinds are requested before either is waited for.  Requesting a
        // block or two ahead was slower (160^3: 0.55 ms against 0.43): the tile
        // settles that many more blocks behind the one it waits for.
        auto stage = [&](int k) {
            unsigned long long bx = 0, by = 0;
            if (NDEP >= 2) bx = look(ix, from_x, k);
            if (NDEP >= 3) by = look(iy, from_y, k);
            if (NDEP >= 2) finish(ix, from_x, k, bx, exs[k & 1]);
            if (NDEP >= 3) finish(iy, from_y, k, by, eys[k & 1]);
            if (few) return;
            for (int q = l + kWave; q < C.Ty * U; q += kWave) {
                const Item it = item(false, q, 0, tx > 0);
                finish(it, from_x, k, look(it, from_x, k), exs[k & 1]);
            }
            for (int q = l + kWave; NDEP >= 3 && q < C.Tx * U; q += kWave) {
                const Item it = item(true, q, 0, ty > 0);
                finish(it, from_y, k, look(it, from_y, k), eys[k & 1]);
            }
        };
        stage(0);
        chain_barrier();
        chain_barrier();
        for (int k = 0; k < niter; k++) {
            stage(k + 1);
            chain_barrier();
        }
    } else {
        // ---- the computing wave
        const int gx = l % C.Tx, gy = l / C.Tx;
        const int srcy = max(l - C.Tx, 0) * 4;
        double prev = 0.0;                  // the chain's element of the last step; the neighbours read it
        // the factor values and v of a block, read from LDS while the block
        // before it is computed: no step waits for LDS but through the exchange
        struct Operands {
            MT m[U][NARR];
            double v[U];
        };
        auto fetch = [&](int k, int j, Operands& o) {
            o.v[j] = vst[k & 1][j * RW + l];
#pragma unroll
            for (int q = 0; q < NARR; q++) o.m[j][q] = vals[k % ST][q][j * kWave + l];
        };
        // one block; HOLES: absent entries are marked and dropped by selects;
        // FLAT: Tx = 64, lane 0 alone has its chain cx-1 in another tile
        auto block = [&](int k, const Operands& o, Operands& next, auto holes, auto flat) {
            constexpr bool HOLES = decltype(holes)::value, FLAT = decltype(flat)::value;
            double ex[U], ey[U];
#pragma unroll
            for (int j = 0; j < U; j++) {
                if (NDEP >= 2) ex[j] = exs[k & 1][(FLAT ? 0 : gy * U) + j];
                if (NDEP >= 3) ey[j] = eys[k & 1][gx * U + j];
            }
            double* out = wst[k & 1];
#pragma unroll
            for (int j = 0; j < U; j++) {
                // operands of the previous step: the element before (prev), the
                // chains cx-1 (ox) and cy-1 (oy); the exchange comes first, it
                // is on every step's dependency chain
                double ox = 0.0, oy = 0.0;
                if (NDEP >= 3) {
                    const double ny = chain_from(prev, srcy);
                    oy = gy > 0 ? ny : ey[j];
                }
                if (NDEP >= 2) {
                    const double nx = chain_from_prev_lane(prev, ex[j]);
                    ox = FLAT || gx > 0 ? nx : ex[j];
                }
                fetch(k + 1, j, next);
                double a = o.v[j];
                // ascending columns: lower rows subtract offset Lc*Cx, Lc, 1;
                // upper rows 1, Lc, Lc*Cx
#pragma unroll
                for (int t = 0; t < NDEP; t++) {
                    const int q = LOWER ? NDEP - 1 - t : t;
                    const double op = q == 0 ? prev : q == 1 ? ox : oy;
                    const double cand = a - to_arith<double>(o.m[j][q]) * op;
                    if constexpr (HOLES) a = dia_absent(o.m[j][q]) ? a : cand;
                    else a = cand;
                }
                if (!UNIT) a = a * to_arith<double>(o.m[j][NARR - 1]);
                out[j * RW + l] = a;
                prev = a;   // on padding never read: the lanes that would read it have no row then either
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto sweep = [&](auto holes, auto flat) {
            Operands A, B;
#pragma unroll
            for (int j = 0; j < U; j++) fetch(0, j, A);
            chain_barrier();                       // its LDS may be filled again
            for (int k = 0; k < niter; k += 2) {   // niter is even
                block(k, A, B, holes, flat);
                chain_barrier();
                block(k + 1, B, A, holes, flat);
                chain_barrier();
            }
        };
        static_assert(AH % 2 == 0, "blocks are computed in pairs");
        chain_barrier();
        if (C.holes) sweep(std::true_type{}, std::false_type{});
        else if (C.Tx == kWave) sweep(std::false_type{}, std::true_type{});
        else sweep(std::false_type{}, std::false_type{});
    }
    wait_memory();
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned done =
            __hip_atomic_fetch_add(counters + 2 * kCounterStride, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
        if (done == (unsigned)gridDim.x) {   // every other tile has finished: reset for the next launch
            if (ld_agent(abort_flag) != 0u) atomicOr(err, 1);
            st_agent(counters, 0u);
            st_agent(abort_flag, 0u);
            st_agent(counters + 2 * kCounterStride, 0u);
        }
    }
}

// value of a stored entry of the chain layout, on the device
template <typename MT>
__global__ void k_fill_chain(int64_t n, int ndep, bool holes, const int32_t* __restrict__ src,
                             const int32_t* __restrict__ dsrc, const double* __restrict__ fv, MT* __restrict__ val,
                             MT* __restrict__ dia) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < ndep * n; i += stride)
        val[i] = src[i] >= 0 ? stored_as<MT>(fv[src[i]]) : holes ? dia_absent_value<MT>() : stored_as<MT>(0.0);
    if (dsrc)
        for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride)
            dia[i] = dsrc[i] < 0 ? stored_as<MT>(1.0) : stored_as<MT>(fv[dsrc[i]]);
}

}  // namespace mtl4g
