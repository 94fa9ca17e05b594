// fem_tiled.h -- the tiled fast path: one workgroup per element tile, node gather in LDS.
//
// Elements are grouped into spatially compact tiles (Morton order of their centroids, cut so
// that a tile has at most kTileElems elements and kTileNodes distinct nodes).  One workgroup
// per tile:
//   1. stages the tile's nodes (p = r + beta p for the CG apply; x and v for the RHS) in LDS,
//   2. computes every element's 12 nodal contributions (applyStiffnessCorotational /
//      accumulateForceLarge arithmetic, shared with the exact path) into LDS,
//   3. sums them per node over the node's incidence list in ascending element id.
// A node touched by one tile only ("interior") is finished in the tile: q = (1 + h rm) m p,
// then the contributions subtracted one by one in the reference's element order, projection,
// store, and its p.q enters the tile's partial.  A node touched by several tiles ("shared")
// gets one partial sum per tile, added in ascending tile order by k_fin_apply.  Every step is
// deterministic; no atomics.
//
// Scalar reductions (|b|^2, p.q, r.r) are written as per-block partials and re-reduced, in a
// fixed order, by every block of the kernel that consumes them (the first block of a scene
// persists the scalars), so no block ever waits on or fences against another block.
#pragma once

#include "fem_device.h"
#include "tiling.h"

namespace sofa_amd {

#ifndef SOFA_AMD_TILE_ELEMS
#define SOFA_AMD_TILE_ELEMS 512
#endif
constexpr int kTileElems = SOFA_AMD_TILE_ELEMS;   // max elements per tile
constexpr int kTileNodes = SOFA_AMD_TILE_ELEMS;   // max distinct nodes per tile
constexpr int kTileRow = slot_row(kTileElems);    // a row of contributions in LDS
// incidences are uint16 contribution slots (row 3 v + c of 12 rows of kTileRow)
static_assert(12 * kTileRow <= 65536, "contribution slots must fit in 16 bits");
#ifndef SOFA_AMD_NODES_PER_THREAD
#define SOFA_AMD_NODES_PER_THREAD 2
#endif
constexpr int kNodesPerThread = SOFA_AMD_NODES_PER_THREAD;   // node kernels: 256 threads x this
#ifndef SOFA_AMD_TILE_THREADS
#define SOFA_AMD_TILE_THREADS 512
#endif
constexpr int kTileThreads = SOFA_AMD_TILE_THREADS;   // threads of the MIXED inner operator kernel


struct TileDesc {
    int scene;
    int e_begin, e_count;     // permuted element range
    int ln_begin, ln_count;   // tile-local node range (into ln_* arrays)
    int flags;                // kTileFirst: first tile of its scene (persists the scene's scalars);
                              // kTileConsistent: the scene has a consistent MeshMatrixMass
    int pslot;                // slot of this tile's partial in the tile/finalize partial buffers
    int inc_begin;            // first entry of the tile's incidence lists (ln_inc)
};
constexpr int kTileFirst = 1, kTileConsistent = 2;
constexpr int kTileOneMaterial = 4;   // the scene has one E and nu: K follows from the rest volume

struct FinBlk { int scene, begin, end, pslot, bi, pad0, pad1, pad2; };  // shared-node range; bi = index in scene
struct NodeBlk { int scene, begin, end, pslot, first, pad0, pad1, pad2; };  // node range
__device__ __forceinline__ int blk_scene(const NodeBlk& b) { return b.scene; }

struct TileNodes {
    const int* __restrict__ gid;        // global node id of each tile-local node
    const int* __restrict__ inc_ptr;    // incidence range (absolute, into inc)
    const uint16_t* __restrict__ inc;   // local element slot * 4 + vertex, ascending element id
    const int* __restrict__ pslot;      // -1: interior; else shared-partial slot of (node, tile),
                                        // | kSlotOwner in the node's first tile (reference order:
                                        // the node's first per-incidence slot)
    const uint8_t* __restrict__ rank;   // reference order: per incidence of a shared node, its
                                        // slot's offset from the node's first slot (else null)
    const uint8_t* __restrict__ arank;  // reference order, CG operator: 0 for an incidence of the
                                        // node's leading run (folded into its first slot by this
                                        // tile), else its slot's offset from the node's first slot
    const uint8_t* __restrict__ lead;   // reference order, CG operator: per tile-local node, the
                                        // number of its first incidences this tile folds (else 0)
};
constexpr int kSlotOwner = 1 << 30;

struct SharedNodes {
    const int* __restrict__ gid;        // shared (and element-free) nodes
    const int* __restrict__ ptr;        // their partial slots [ptr[i], ptr[i+1]) in tile order
    const int* __restrict__ of;         // per node: its index in gid / ptr, or -1 (tile-owned)
    const uint8_t* __restrict__ acnt;   // reference order, CG operator: slots after the first
};

// per-scene slot ranges of the two partial buffers
struct Ranges {
    int t0, nt;    // tile partials
    int f0, nf;    // finalize-block partials (offset into the same buffer)
    int b0, nb;    // node-block partials (rho buffer)
};

// one DPP step of a 64-lane sum: v of the lane CTRL names in the rows ROWS enables, 0.0 where
// there is none (a double moved as its two 32-bit halves)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_from(double v) {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, CTRL, ROWS, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, lo, CTRL, ROWS, 0xf, true));
}

// sum over the 64 lanes of a wave in a fixed order: an inclusive scan within each row of 16
// lanes (row_shr 1, 2, 4, 8), then row 0's total into row 1 and row 2's into row 3
// (row_bcast 15), then the first half's total into the second half (row_bcast 31); lane 63 then
// holds the sum, and every lane reads it from there (the same bits in every lane)
__device__ __forceinline__ double wave_sum(double v) {
    v = v + dpp_from<0x111, 0xf>(v);
    v = v + dpp_from<0x112, 0xf>(v);
    v = v + dpp_from<0x114, 0xf>(v);
    v = v + dpp_from<0x118, 0xf>(v);
    v = v + dpp_from<0x142, 0xa>(v);
    v = v + dpp_from<0x143, 0xc>(v);
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                            __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// acc + buf[a0 + k] + buf[a0 + k + STRIDE] + ... below a0 + na, B terms, all loads in flight
template <int STRIDE, int B>
__device__ __forceinline__ double strided_terms(const double* __restrict__ buf, int a0, int na, int k, double acc) {
    double v[B];
#pragma unroll
    for (int j = 0; j < B; j++) v[j] = buf[a0 + min(k + j * STRIDE, na - 1)];
#pragma unroll
    for (int j = 0; j < B; j++) acc = k + j * STRIDE < na ? acc + v[j] : acc;
    return acc;
}
// buf[a0 + t] + buf[a0 + t + STRIDE] + ... below a0 + na, in that order: eight loads in flight, two
// where two are all (one after the other each waited for memory)
template <int STRIDE>
__device__ __forceinline__ double strided_sum(const double* __restrict__ buf, int a0, int na, int t) {
    if (na <= 0) return 0.0;
    if (na <= 2 * STRIDE) return strided_terms<STRIDE, 2>(buf, a0, na, t, 0.0);
    double acc = 0.0;
    for (int k = t; k < na; k += 8 * STRIDE) acc = strided_terms<STRIDE, 8>(buf, a0, na, k, acc);
    return acc;
}

// every wave of the block: the sum of buf[a0 .. a0 + na) (lane-strided partial sums, then
// wave_sum) -- no LDS and no barrier, and the same bits in every wave and every block
__device__ __forceinline__ double wave_reduce(const double* __restrict__ buf, int a0, int na) {
    return wave_sum(strided_sum<64>(buf, a0, na, (int)(threadIdx.x & 63)));
}

// fixed-order block sum of the tiled kernels (TB threads): wave_sum within each wave, then the
// wave sums added in wave order; sh holds TB / 64 doubles
template <int TB>
__device__ __forceinline__ double wave_block_sum(double v, double* sh) {
    v = wave_sum(v);
    __syncthreads();                     // a previous call's readers are done with sh
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = sh[0];
#pragma unroll
    for (int k = 1; k < TB / 64; k++) r = r + sh[k];
    return r;
}

// fixed-order sum of buf[a0 .. a0+na), all threads of the block
template <int TB = kBlock>
__device__ __forceinline__ double reduce2(const double* __restrict__ buf, int a0, int na, double* sh) {
    return wave_block_sum<TB>(strided_sum<TB>(buf, a0, na, (int)threadIdx.x), sh);
}

// a scene's sum of na partials, the same bits in every block of the scene: few partials are
// added by every wave on its own (no barrier), many are split over the block (two barriers).
// WIDE = false: the launch has no scene of more than 256 partials (the block path compiled out)
constexpr int kWavePartials = 256;
template <int TB, bool WIDE = true>
__device__ __forceinline__ double scene_sum(const double* __restrict__ buf, int a0, int na, double* sh) {
    if (!WIDE || na <= kWavePartials) return wave_reduce(buf, a0, na);
    return reduce2<TB>(buf, a0, na, sh);
}

// scene_sum in two parts: the loads at the head of a kernel, the sum where it is needed.  TB threads add
// (a larger block's others only take part in the barrier); sh holds TB / 64 doubles
constexpr int kSumBatch = 8;
struct SceneTerms {
    double v[kSumBatch];
};
template <int TB, bool WIDE>
__device__ __forceinline__ void load_terms(const double* __restrict__ buf, int na, SceneTerms& s) {
    const int lane = threadIdx.x & 63;
    static_assert(kWavePartials == 256, "four partials per lane");
#pragma unroll
    for (int k = 0; k < kSumBatch; k++) s.v[k] = 0.0;
    if (na <= 0) return;
    if (!WIDE || na <= kWavePartials) {
        s.v[0] = buf[(unsigned)min(lane, na - 1)];
        if (na > 64) {
#pragma unroll
            for (int k = 1; k < kWavePartials / 64; k++) s.v[k] = buf[(unsigned)min(lane + 64 * k, na - 1)];
        }
    } else if ((int)threadIdx.x < TB) {
        s.v[0] = buf[(unsigned)min((int)threadIdx.x, na - 1)];
        s.v[1] = buf[(unsigned)min((int)threadIdx.x + TB, na - 1)];
        if (na > 2 * TB) {
#pragma unroll
            for (int k = 2; k < kSumBatch; k++) s.v[k] = buf[(unsigned)min((int)threadIdx.x + k * TB, na - 1)];
        }
    }
}
template <int TB, bool WIDE>
__device__ __forceinline__ double sum_terms(const double* __restrict__ buf, int na, const SceneTerms& s, double* sh) {
    const int lane = threadIdx.x & 63, t = threadIdx.x;
    double acc = 0.0;
    if (!WIDE || na <= kWavePartials) {
#pragma unroll
        for (int k = 0; k < kWavePartials / 64; k++) acc = lane + 64 * k < na ? acc + s.v[k] : acc;
        return wave_sum(acc);
    }
    if (t < TB) {
#pragma unroll
        for (int k = 0; k < kSumBatch; k++) acc = t + k * TB < na ? acc + s.v[k] : acc;
        for (int k = t + kSumBatch * TB; k < na; k += 8 * TB) acc = strided_terms<TB, 8>(buf, 0, na, k, acc);
        acc = wave_sum(acc);
        if (lane == 0) sh[t >> 6] = acc;
    }
    __syncthreads();
    acc = sh[0];
#pragma unroll
    for (int k = 1; k < TB / 64; k++) acc = acc + sh[k];
    return acc;
}

template <typename VT>
__device__ __forceinline__ void ld3(const VT* __restrict__ v, int n, VT o[3]) {
    const VT* q = v + 3 * (int64_t)n;
    o[0] = q[0]; o[1] = q[1]; o[2] = q[2];
}
template <typename VT>
__device__ __forceinline__ void st3(VT* __restrict__ v, int n, const VT o[3]) {
    VT* q = v + 3 * (int64_t)n;
    q[0] = o[0]; q[1] = o[1]; q[2] = o[2];
}

// stop the scene's CG loop: every block of the kernel reaches the same decision; the first
// block records it, with the launch's mark
__device__ __forceinline__ void record_stop(InstDev* ins, bool first, int mark, int reason, int iters, double err) {
    if (first && threadIdx.x == 0) {
        ins->stopped = mark;
        ins->end_reason = reason;
        ins->last_iters = iters;
        ins->err = err;
    }
}

// the scene's tile partials are folded into its finalize-block partials (finalize block bi
// of nf adds tiles [t0 + bi*ceil(nt/nf), ...)), so consumers reduce only nf values
__device__ __forceinline__ double fold_tiles(const double* __restrict__ buf, const Ranges& rg, int bi) {
    if (rg.nf <= 0) return 0.0;
    const int chunk = (rg.nt + rg.nf - 1) / rg.nf;
    const int a0 = rg.t0 + bi * chunk;
    const int a1 = min(rg.t0 + rg.nt, a0 + chunk);
    return strided_sum<1>(buf, a0, a1 - a0, 0);
}

template <typename R, int NR>
struct TileArgs {
    const TileDesc* __restrict__ tiles;
    InstDev* __restrict__ inst;
    const Ranges* __restrict__ ranges;
    ElemView<R, NR> ev;                 // permuted element SoA (ev.tet unused)
    const uint2* __restrict__ ltet;     // 4 x uint16 tile-local node indices per element
    TileNodes tn;
    const double* __restrict__ mass;
    const int8_t* __restrict__ fixed;
    int8_t* __restrict__ contact;        // PlaneForceField contacts of the step (per node)
    const R* __restrict__ emass;        // per element rho V / 20 (consistent MeshMatrixMass), else unused
    double* __restrict__ nd;            // reference order: per-node dot terms
    // the operator's element record, SoA: rotations (written by the step's force pass), rest shape, K
    const R *rot, *rest, *kmat;
    float *rot32, *x32;                 // MIXED: the inner operator's rotations and positions, written by the force pass
};

// consistent-mass edge terms of one element, folded into its nodal contributions (which the
// node sums subtract): vertex v of the element receives emass * factor * (sum of the other
// three vertices' values), i.e. the element's share of the edge loop of MeshMatrixMass::addMDx
template <typename R>
__device__ __forceinline__ void add_edge_mass(R mf, const R u[12], R c[12]) {
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const R sum = u[i] + u[3 + i] + u[6 + i] + u[9 + i];
#pragma unroll
        for (int v = 0; v < 4; v++) c[3 * v + i] -= mf * (sum - u[3 * v + i]);
    }
}

// acc (+|-)= the node's element contributions lc[slot + c kTileRow] in incidence-list order.
// Four incidences per round: their slots are read together, then their values, so a round
// waits on LDS twice instead of eight times; the adds keep the list order (same bits).
template <bool SUB, typename R, typename VT>
__device__ __forceinline__ void sum_incidences(const uint16_t* linc, int s0, int s1, const R* lc, VT acc[3]) {
    int s = s0;
    for (; s + 4 <= s1; s += 4) {
        int sl[4];
#pragma unroll
        for (int t = 0; t < 4; t++) sl[t] = linc[s + t];
        R v[4][3];
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int i = 0; i < 3; i++) v[t][i] = lc[sl[t] + i * kTileRow];
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                if (SUB) acc[i] -= (VT)v[t][i];
                else acc[i] += (VT)v[t][i];
            }
    }
    for (; s < s1; s++) {
        const int sl = linc[s];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            if (SUB) acc[i] -= (VT)lc[sl + i * kTileRow];
            else acc[i] += (VT)lc[sl + i * kTileRow];
        }
    }
}

// one component of sum_incidences<true> (row: lc + c kTileRow)
template <typename R, typename VT>
__device__ __forceinline__ void sum_component(const uint16_t* linc, int s0, int s1, const R* row, VT& acc) {
    int s = s0;
    for (; s + 4 <= s1; s += 4) {
        R v[4];
#pragma unroll
        for (int t = 0; t < 4; t++) v[t] = row[linc[s + t]];
#pragma unroll
        for (int t = 0; t < 4; t++) acc -= (VT)v[t];
    }
    for (; s < s1; s++) acc -= (VT)row[linc[s]];
}

// reference order: each incidence's contribution lc[slot + c kTileRow] to its own global slot
// base + rank (the node's slots run in ascending element id, the order its finalize adds them);
// rank: the tile's incidence ranks, indexed like linc
template <typename R, typename VT>
__device__ __forceinline__ void store_incidences(const uint16_t* linc, const uint8_t* __restrict__ rank, int s0,
                                                 int s1, const R* lc, VT* __restrict__ sp, int base) {
    for (int s = s0; s < s1; s++) {
        const int sl = linc[s];
        VT* o = sp + 3 * (int64_t)(base + rank[s]);
#pragma unroll
        for (int i = 0; i < 3; i++) o[i] = (VT)lc[sl + i * kTileRow];
    }
}

// acc (+|-)= the partials or slots sp[s0 .. s1) in that order: the loads four at a time, then
// their adds in slot order (the same operations as one slot after the other)
template <bool SUB, typename VT>
__device__ __forceinline__ void sum_slots(const VT* __restrict__ sp, int s0, int s1, VT acc[3]) {
    int s = s0;
    for (; s + 4 <= s1; s += 4) {
        VT t[4][3];
#pragma unroll
        for (int u = 0; u < 4; u++) ld3(sp, s + u, t[u]);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                if (SUB) acc[i] -= t[u][i];
                else acc[i] += t[u][i];
            }
    }
    for (; s < s1; s++) {
        VT t[3];
        ld3(sp, s, t);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            if (SUB) acc[i] -= t[i];
            else acc[i] += t[i];
        }
    }
}

__device__ __forceinline__ void unpack_ltet(uint2 w, int l[4]) {
    l[0] = (int)(w.x & 0xffffu); l[1] = (int)(w.x >> 16); l[2] = (int)(w.y & 0xffffu); l[3] = (int)(w.y >> 16);
}

// ---------------------------------------------------------------------------------------
// RHS: rotations, element force, K v; interior nodes finished, shared nodes -> partials.
// TB threads, one element (and at most one tile-local node) per thread for TB = 512.  One LDS
// contribution buffer serves both element passes: the force pass, the node sums of f, then the
// K v pass (element record and rotation kept in registers) and the node sums of b.
// ---------------------------------------------------------------------------------------
// EXACT: the reference's summation order -- a shared node's contributions go to per-incidence
// slots (f to spf, K v to spv) instead of per-tile partials, and every node's |b|^2 term to nd
template <typename R, int NR, typename VT, int TB = 512, bool EXACT = false>
__global__ __launch_bounds__(TB) void k_tile_rhs(TileArgs<R, NR> a, const VT* __restrict__ x,
                                                  const VT* __restrict__ v, VT* __restrict__ f,
                                                  VT* __restrict__ b, VT* __restrict__ r, VT* __restrict__ xcg,
                                                  VT* __restrict__ spf, VT* __restrict__ spv,
                                                  double* __restrict__ pbb) {
    constexpr int EPT = kTileElems / TB;
    constexpr int NPT = (kTileNodes + TB - 1) / TB;
    __shared__ R lx[kTileNodes * 3];
    __shared__ R lv[kTileNodes * 3];
    __shared__ R lc[kTileRow * 12];
    __shared__ uint16_t linc[kTileElems * 4];
    __shared__ int lptr[kTileNodes + 1];
    __shared__ double sh[TB / 64];
    const TileDesc td = a.tiles[xcd_item()];
    const InstDev in = a.inst[td.scene];
    // element records of this thread's elements, in registers for both passes
    R rin[EPT][NR], kk[EPT][3], em[EPT], rot[EPT][9];
    uint2 lt[EPT];
#pragma unroll
    for (int m = 0; m < EPT; m++) {
        const int k = threadIdx.x + m * TB;
        if (k < td.e_count) {
            const int64_t e = (int64_t)td.e_begin + k;
            lt[m] = a.ltet[e];
#pragma unroll
            for (int i = 0; i < NR; i++) rin[m][i] = a.ev.rest[i * a.ev.E + e];
#pragma unroll
            for (int i = 0; i < 3; i++) kk[m][i] = a.ev.kmat[i * a.ev.E + e];
            em[m] = in.mass_kind == kMassMatrix ? a.emass[e] : (R)0;
        }
    }
    // node tables, incidence tables and node gathers at clamped indices (no branch: all in flight
    // together; values past the tile's counts unused), then staged in LDS
    int gid[NPT], psl[NPT];
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        const int li = td.ln_begin + min((int)threadIdx.x + m * TB, td.ln_count - 1);
        gid[m] = a.tn.gid[li];
        psl[m] = a.tn.pslot[li];
    }
    const int ninc = 4 * td.e_count;
    constexpr int IPT = (4 * kTileElems + TB - 1) / TB;     // incidences per thread
    constexpr int PPT = (kTileNodes + 1 + TB - 1) / TB;     // incidence pointers per thread
    int inc_r[IPT], ptr_r[PPT];
#pragma unroll
    for (int k = 0; k < IPT; k++)
        inc_r[k] = a.tn.inc[ninc > 0 ? td.inc_begin + min((int)threadIdx.x + k * TB, ninc - 1) : 0];
#pragma unroll
    for (int k = 0; k < PPT; k++)
        ptr_r[k] = a.tn.inc_ptr[td.ln_begin + min((int)threadIdx.x + k * TB, td.ln_count)] - td.inc_begin;
    VT xt[NPT][3], vt[NPT][3];
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        ld3(x, gid[m], xt[m]);
        ld3(v, gid[m], vt[m]);
    }
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        const int j = threadIdx.x + m * TB;
        if (j < td.ln_count) {
            lx[3 * j] = (R)xt[m][0]; lx[3 * j + 1] = (R)xt[m][1]; lx[3 * j + 2] = (R)xt[m][2];
            if (a.x32) {   // every tile of a shared node writes the same value
                const float xf[3] = {(float)xt[m][0], (float)xt[m][1], (float)xt[m][2]};
                st3(a.x32, gid[m], xf);
            }
            lv[3 * j] = (R)vt[m][0]; lv[3 * j + 1] = (R)vt[m][1]; lv[3 * j + 2] = (R)vt[m][2];
        }
    }
#pragma unroll
    for (int k = 0; k < IPT; k++) {
        const int j = threadIdx.x + k * TB;
        if (j < ninc) linc[j] = (uint16_t)inc_r[k];
    }
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int j = threadIdx.x + k * TB;
        if (j <= td.ln_count) lptr[j] = ptr_r[k];
    }
    __syncthreads();
    // ---- element force (accumulateForceLarge); the rotations are stored for the operator
#pragma unroll
    for (int m = 0; m < EPT; m++) {
        const int k = threadIdx.x + m * TB;
        if (k < td.e_count) {
            const int64_t e = (int64_t)td.e_begin + k;
            int l[4];
            unpack_ltet(lt[m], l);
            R p[4][3], c[12];
#pragma unroll
            for (int n = 0; n < 4; n++)
#pragma unroll
                for (int i = 0; i < 3; i++) p[n][i] = lx[3 * l[n] + i];
            elem_force_r<R, NR>(p, rin[m], kk[m], rot[m], c);
#pragma unroll
            for (int i = 0; i < 9; i++) a.ev.rot[i * a.ev.E + e] = rot[m][i];
            if (a.rot32) {   // from the positions in float, as a force pass in float has them
                float pf[3][3], rf[9];
#pragma unroll
                for (int n = 0; n < 3; n++)
#pragma unroll
                    for (int i = 0; i < 3; i++) pf[n][i] = (float)p[n][i];
                rotation_large(pf[0], pf[1], pf[2], rf);
#pragma unroll
                for (int i = 0; i < 9; i++) a.rot32[i * a.ev.E + e] = rf[i];
            }
#pragma unroll
            for (int i = 0; i < 12; i++) lc[i * kTileRow + k] = c[i];
        }
    }
    __syncthreads();
    // ---- node sums of f in ascending element id (interior nodes: with gravity)
    VT fn[NPT][3];
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        const int j = threadIdx.x + m * TB;
        if (j < td.ln_count) {
            if (psl[m] < 0) mass_gravity(in, a.mass, gid[m], fn[m]);
            else { fn[m][0] = 0; fn[m][1] = 0; fn[m][2] = 0; }
            const int s0 = lptr[j], s1 = lptr[j + 1];
            if (EXACT && psl[m] >= 0) store_incidences(linc, a.tn.rank + td.inc_begin, s0, s1, lc, spf, psl[m]);
            else sum_incidences<false>(linc, s0, s1, lc, fn[m]);
        }
    }
    __syncthreads();
    // ---- K v (+ the consistent-mass edge terms) into the same buffer
    const R krhs = (R)in.k_rhs;
    const bool edge = in.mass_kind == kMassMatrix && in.m_rhs != 0.0;
#pragma unroll
    for (int m = 0; m < EPT; m++) {
        const int k = threadIdx.x + m * TB;
        if (k < td.e_count) {
            int l[4];
            unpack_ltet(lt[m], l);
            R u[12], c[12];
#pragma unroll
            for (int n = 0; n < 4; n++)
#pragma unroll
                for (int i = 0; i < 3; i++) u[3 * n + i] = lv[3 * l[n] + i];
            if (in.k_rhs != 0.0) {
                elem_dforce_r<R, NR, std::is_same<VT, double>::value>(rot[m], rin[m], kk[m], u, krhs, c);
            } else {
#pragma unroll
                for (int i = 0; i < 12; i++) c[i] = 0;
            }
            if (edge) add_edge_mass((R)in.m_rhs * em[m], u, c);
#pragma unroll
            for (int i = 0; i < 12; i++) lc[i * kTileRow + k] = c[i];
        }
    }
    __syncthreads();
    // ---- b = h (f - rm M v - (h + rs) K v), projected; shared nodes leave partials
    double bb = 0.0;
    const VT h = (VT)in.b_scale;   // h (firstOrder: 1, b = f)
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        const int j = threadIdx.x + m * TB;
        if (j < td.ln_count) {
            const int g = gid[m];
            const int s0 = lptr[j], s1 = lptr[j + 1];
            if (psl[m] < 0) {
                const VT vn[3] = {(VT)lv[3 * j], (VT)lv[3 * j + 1], (VT)lv[3 * j + 2]};
                // PlaneForceField after the FEM (scene order); the contact is kept for addDForce
                bool touch = false;
                if (in.plane_on) {
                    const VT xn[3] = {(VT)lx[3 * j], (VT)lx[3 * j + 1], (VT)lx[3 * j + 2]};
                    touch = plane_force(in, xn, vn, fn[m]);
                    a.contact[g] = touch ? 1 : 0;
                }
                st3(f, g, fn[m]);
                VT bn[3] = {fn[m][0], fn[m][1], fn[m][2]};
                if (in.m_rhs != 0.0) mass_mdx<true>(in, NodeArrays{nullptr, nullptr, a.mass, a.fixed}, g, in.m_rhs, vn, bn);
                sum_incidences<true>(linc, s0, s1, lc, bn);
                if (touch && in.k_rhs != 0.0) plane_dforce(in, in.k_rhs, vn, bn);
                bn[0] *= h; bn[1] *= h; bn[2] *= h;
                if (a.fixed[g]) { bn[0] = 0; bn[1] = 0; bn[2] = 0; }
                st3(b, g, bn);
                st3(r, g, bn);
                const VT z[3] = {0, 0, 0};
                if (!in.warm_start) st3(xcg, g, z);   // warmStart: x stays the previous solution
                if (EXACT) a.nd[g] = dot3d(bn, bn);
                else bb += dot3d(bn, bn);
            } else if (EXACT) {
                store_incidences(linc, a.tn.rank + td.inc_begin, s0, s1, lc, spv, psl[m]);
            } else {
                const int ps = psl[m] & (kSlotOwner - 1);
                VT pv[3] = {0, 0, 0};
                sum_incidences<false>(linc, s0, s1, lc, pv);
                st3(spf, ps, fn[m]);
                st3(spv, ps, pv);
            }
        }
    }
    if (!EXACT) {
        const double tot = wave_block_sum<TB>(bb, sh);
        if (threadIdx.x == 0) pbb[td.pslot] = tot;
    }
}

template <typename VT, bool EXACT = false>
__global__ __launch_bounds__(kBlock) void k_fin_rhs(const FinBlk* __restrict__ fb_, const InstDev* __restrict__ inst,
                                                     const Ranges* __restrict__ ranges, SharedNodes sn, const double* __restrict__ mass,
                                                     const int8_t* __restrict__ fixed, const VT* __restrict__ v,
                                                     const VT* __restrict__ spf, const VT* __restrict__ spv,
                                                     VT* __restrict__ f, VT* __restrict__ b, VT* __restrict__ r,
                                                     VT* __restrict__ xcg, double* __restrict__ pbb,
                                                     const VT* __restrict__ x, int8_t* __restrict__ contact,
                                                     double* __restrict__ nd = nullptr) {
    __shared__ double sh[kBlock / 64];
    const FinBlk fb = fb_[xcd_item()];
    const InstDev in = inst[fb.scene];
    const int j = fb.begin + threadIdx.x;
    double bb = 0.0;
    if (j < fb.end) {
        const int g = sn.gid[j];
        VT fn[3], vn[3];
        ld3(v, g, vn);
        mass_gravity(in, mass, g, fn);
        const int s0 = sn.ptr[j], s1 = sn.ptr[j + 1];
        sum_slots<false>(spf, s0, s1, fn);
        // PlaneForceField after the FEM (scene order); the contact is kept for addDForce
        bool touch = false;
        if (in.plane_on) {
            VT xn[3];
            ld3(x, g, xn);
            touch = plane_force(in, xn, vn, fn);
            contact[g] = touch ? 1 : 0;
        }
        st3(f, g, fn);
        VT bn[3] = {fn[0], fn[1], fn[2]};
        if (in.m_rhs != 0.0) mass_mdx<true>(in, NodeArrays{nullptr, nullptr, mass, fixed}, g, in.m_rhs, vn, bn);
        sum_slots<true>(spv, s0, s1, bn);
        if (touch && in.k_rhs != 0.0) plane_dforce(in, in.k_rhs, vn, bn);
        const VT h = (VT)in.b_scale;   // h (firstOrder: 1, b = f)
        bn[0] *= h; bn[1] *= h; bn[2] *= h;
        if (fixed[g]) { bn[0] = 0; bn[1] = 0; bn[2] = 0; }
        st3(b, g, bn);
        st3(r, g, bn);
        const VT z[3] = {0, 0, 0};
        if (!in.warm_start) st3(xcg, g, z);   // warmStart: x stays the previous solution
        bb = dot3d(bn, bn);
        if (EXACT) nd[g] = bb;
    }
    if (EXACT) return;
    const double own = wave_block_sum<kBlock>(bb, sh);
    if (threadIdx.x == 0) pbb[fb.pslot] = fold_tiles(pbb, ranges[fb.scene], fb.bi) + own;
}

// ---------------------------------------------------------------------------------------
// CG iteration `iter` (1-based): the operator, then k_update (reference order: k_fin_exact between).
// iter = 0 is a plain operator application q = A r (no CG scalars, p untouched).
// ---------------------------------------------------------------------------------------
// The operator: one workgroup per tile, TB threads.
//   1. loads: the elements' records into registers; a thread per tile-local node reads its tables, r, p;
//   2. by the waves that have nodes: the scalars (rho, the tolerance test, beta), then p = r + beta p and
//      what the node sums need of each node, staged in LDS;
//   3. each element's contributions into LDS, 12 rows of kTileRow;
//   4. a thread per (node, component), GEO: per node: the contributions in ascending element id;
//   5. by the waves that have nodes: interior nodes finished (q), a shared node's sum left as the tile's
//      partial, p.q as one partial per tile.
// The element's rotation, rest shape and K are read back (18 floats, 21 doubles), not recomputed from the
// positions: a phase less, and 417 vector instructions per wave on 256 beams in float, 482 with GEO.  GEO: recomputed from
// the positions x, x0 all the same (same bits), for sets whose record does not stay cached from one iteration to
// the next (EngineT::recomputes has the line), the sums then by the threads that have a node's p in registers, which
// takes back the phase and its LDS traffic.  What bounds it: on a large mesh VALU issue (half of the time), LDS (a
// third) and the latency of the phases of the four tiles that a CU holds (FP64: two, by registers and LDS); on a
// small one that latency alone.  Measured, launches one after the other, with all recomputed and a thread per node for
// staging and sums, read back, and GEO: FP32 18,954 tetrahedra 8.2, 7.3, 7.5 us, 101,250 8.4, 7.6, 7.8, 1.31M 33.4, 29.2,
// 28.7; SPLIT 150k 12.1, 10.0, 10.6; FP64 360k 28.8, 22.4, 22.7; 256 beams of 8.9M FP32 169, 199, 156, SPLIT 211, 246,
// 184, FP64 379, 427, 346.  (Between the launches of a step the update passes over the vectors: the line is the step's.)
// The step of those 256 beams, ms, read back, GEO with the sums by component, and GEO: FP32 6.77, 5.95, 5.57; SPLIT 9.2,
// 7.68, 7.44; MIXED 25.3, 22.3, 20.9.
// PLANE = false: no scene of the launch has a PlaneForceField; WIDE = false: no scene has more than
// kWavePartials partials of r.r, which are then in flight with the gathers.
constexpr int kNodeMass = 1 << 12;   // the node's sum starts from the mass term
static_assert(4 * kTileElems <= kNodeMass, "a node's first incidence and the flag share 16 bits");
template <typename R, int NR, typename VT, int TB, bool WIDE, bool PLANE, bool GEO = false>
__global__ __launch_bounds__(TB) void k_tile_apply(TileArgs<R, NR> a, int iter, const VT* __restrict__ r,
                                                    VT* __restrict__ p, VT* __restrict__ q, VT* __restrict__ sp,
                                                    const double* __restrict__ pin,   // |b|^2 (iter 1) or r.r partials
                                                    double* __restrict__ pden,
                                                    int pin_nodes,     // 1: iter-1 |b|^2 partials per node block
                                                    const VT* __restrict__ x, const VT* __restrict__ x0) {   // GEO
    constexpr int EPT = kTileElems / TB;                   // elements per thread
    constexpr int NPT = (kTileNodes + TB - 1) / TB;        // tile-local nodes per thread
    __shared__ VT lu[kTileNodes * 3];        // p (in R), then the nodes' sums
    __shared__ R lc[kTileRow * 12];
    __shared__ __align__(8) uint16_t linc[kTileElems * 4];
    __shared__ VT lmass[kTileNodes];
    __shared__ uint16_t lnode[kTileNodes];   // first incidence and flags
    __shared__ double sh[TB / 64];
    __shared__ int halt;
    const TileDesc td = a.tiles[xcd_item()];
    InstDev* ins = &a.inst[td.scene];
    const InstDev in = *ins;
    const Ranges rg = a.ranges[td.scene];
    const bool consistent = (td.flags & kTileConsistent) != 0, one = (td.flags & kTileOneMaterial) != 0;
    const int ninc = 4 * td.e_count;
    // a refinement sweep that keeps the previous search direction continues CG at its iteration 1
    const bool cont = iter == 1 && in.keep_dir && in.sweep > 1;
    // p is read from iteration 2 on (or continuing a direction)
    const bool second = iter > 1 || cont;
    const int w0 = __builtin_amdgcn_readfirstlane((int)threadIdx.x & ~63);   // the wave's first thread
    // ---- 1. the nodes' tables, the partials, the element records, the incidence table
    int gid[NPT], psl[NPT], s0[NPT];
#pragma unroll
    for (int m = 0; m < NPT; m++)
        if (w0 + m * TB < td.ln_count) {
            const unsigned j = min((int)threadIdx.x + m * TB, td.ln_count - 1);
            gid[m] = (a.tn.gid + td.ln_begin)[j];
            psl[m] = (a.tn.pslot + td.ln_begin)[j];
            s0[m] = (a.tn.inc_ptr + td.ln_begin)[j] - td.inc_begin;
        }
    // the partials of |b|^2 (iteration 1) or r.r: node blocks, or finalize blocks, or the tiles of a
    // scene without shared nodes
    const bool by_node = second || pin_nodes;
    const int pa = by_node ? rg.b0 : rg.nf > 0 ? rg.f0 : rg.t0, pn = by_node ? rg.nb : rg.nf > 0 ? rg.nf : rg.nt;
    const int lane = threadIdx.x & 63;
    SceneTerms part;
    if (!WIDE && iter > 0 && w0 < td.ln_count) load_terms<TB, WIDE>(pin + pa, pn, part);
    const int mark = iter > 0 ? stop_mark(iter, 0) : 0;
    if (stopped_before(in.stopped, mark)) return;   // before the record's loads: a converged scene's launches are many
    R rot[EPT][9], rin[EPT][NR], kk[EPT][3], em[EPT];
    uint2 lt[EPT], inc[EPT];
#pragma unroll
    for (int m = 0; m < EPT; m++) {
        const unsigned k = threadIdx.x + m * TB;
        if ((int)k < td.e_count) {
            lt[m] = (a.ltet + td.e_begin)[k];
            inc[m] = reinterpret_cast<const uint2*>(a.tn.inc + td.inc_begin)[k];   // four incidences
            if (!GEO) {
#pragma unroll
                for (int i = 0; i < 9; i++) rot[m][i] = (a.rot + (i * a.ev.E + td.e_begin))[k];
#pragma unroll
                for (int i = 0; i < NR; i++) rin[m][i] = (a.rest + (i * a.ev.E + td.e_begin))[k];
            }
            if (!GEO || !one)
#pragma unroll
                for (int i = 0; i < 3; i++) kk[m][i] = (a.kmat + (i * a.ev.E + td.e_begin))[k];
            em[m] = consistent ? (a.emass + td.e_begin)[k] : (R)0;
        }
    }
    VT pv[NPT][3], po[NPT][3], ms[NPT], xt[NPT][3], x0t[NPT][3];
    int8_t fx[NPT], ct[NPT];
    const bool plane = PLANE && in.plane_on, table = in.mass_kind != kMassUniform;
#pragma unroll
    for (int m = 0; m < NPT; m++)
        if (w0 + m * TB < td.ln_count) {
            ld3(r, gid[m], pv[m]);
            if (second) ld3(p, gid[m], po[m]);
            if (GEO) { ld3(x, gid[m], xt[m]); ld3(x0, gid[m], x0t[m]); }
            ms[m] = table ? (VT)a.mass[gid[m]] : (VT)in.vertex_mass;
            fx[m] = a.fixed[gid[m]];
            ct[m] = plane ? a.contact[gid[m]] : 0;
        }
#pragma unroll
    for (int m = 0; m < EPT; m++) {
        const int k = threadIdx.x + m * TB;
        if (k < td.e_count) *reinterpret_cast<uint2*>(linc + 4 * k) = inc[m];
    }
    const bool first = (td.flags & kTileFirst) != 0;
    // ---- 2. scalars: rho, the tolerance test, beta (CGLinearSolver.inl:130-196)
    double total = 0.0, beta = 0.0;      // |b|^2 or r.r
    bool go = true;
    if (WIDE && iter > 0) total = scene_sum<TB, WIDE>(pin, pa, pn, sh);   // (early, it costs a wave per SIMD)
    if (w0 < td.ln_count) {
        if (!WIDE && iter > 0) total = sum_terms<TB, WIDE>(pin + pa, pn, part, sh);
        double err = 0.0;
        if (cont) {
            // the refinement replaced r by the true residual: beta from its r.r and the r.r that
            // built p; the tolerance is relative to the first sweep's |r|
            err = sqrt(total) / in.normb;
            if (total == 0.0 || err <= in.tol) { record_stop(ins, first, mark, 1, 1, err); go = false; }
            beta = total / in.rho_last;
            if (go && first && threadIdx.x == 0) {
                ins->rho_slot[1] = total; ins->beta = beta; ins->iter = 1; ins->err = err;
            }
        } else if (iter == 1) {
            const double normb = sqrt(total);
            err = sqrt(total) / normb;
            if (normb == 0.0) { record_stop(ins, first, mark, 4, 0, 1.0); go = false; }
            else if (err <= in.tol && !in.first_solve) { record_stop(ins, first, mark, 1, 1, err); go = false; }
            if (go && first && threadIdx.x == 0) {
                ins->normb = normb; ins->rho_slot[1] = total; ins->iter = 1; ins->err = err;
            }
        } else if (iter > 1) {
            err = sqrt(total) / in.normb;
            if (iter > in.max_iter) { record_stop(ins, first, mark, 0, in.max_iter, in.err); go = false; }
            else if (err <= in.tol) { record_stop(ins, first, mark, 1, iter, err); go = false; }
            beta = total / (iter & 1 ? in.rho_slot[0] : in.rho_slot[1]);
            if (go && first && threadIdx.x == 0) {
                ins->rho_slot[iter & 1] = total; ins->beta = beta; ins->iter = iter; ins->err = err;
            }
        }
        if (go) {   // p = r + beta p (interior nodes: this tile owns p and writes it back)
            const VT vb = (VT)beta;
#pragma unroll
            for (int m = 0; m < NPT; m++) {
                const int j = threadIdx.x + m * TB;
                if (j < td.ln_count) {
                    const bool interior = psl[m] < 0;
                    if (second) {
#pragma unroll
                        for (int i = 0; i < 3; i++) { VT t = po[m][i] * vb; t += pv[m][i]; pv[m][i] = t; }
                    }
                    if (iter > 0 && interior) st3(p, gid[m], pv[m]);
#pragma unroll
                    for (int i = 0; i < 3; i++) {
                        pv[m][i] = (VT)(R)pv[m][i];
                        lu[3 * j + i] = pv[m][i];
                        if (GEO) { lc[3 * j + i] = (R)xt[m][i]; lc[3 * kTileNodes + 3 * j + i] = (R)x0t[m][i]; }
                    }
                    if (!GEO) lmass[j] = ms[m];
                    lnode[j] = (uint16_t)(s0[m] | (in.m_cg != 0.0 && interior ? kNodeMass : 0));
                }
            }
        }
    }
    if (threadIdx.x == 0) halt = !go;
    __syncthreads();
    if (halt) return;
    if constexpr (GEO) {   // the record from the staged positions, then their buffer is free
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const int k = threadIdx.x + m * TB;
            if (k < td.e_count) {
                int l[4];
                unpack_ltet(lt[m], l);
                R xe[3][3], x0e[4][3];
#pragma unroll
                for (int v = 0; v < 4; v++)
#pragma unroll
                    for (int i = 0; i < 3; i++) {
                        if (v < 3) xe[v][i] = lc[3 * l[v] + i];
                        x0e[v][i] = lc[3 * kTileNodes + 3 * l[v] + i];
                    }
                rotation_large(xe[0], xe[1], xe[2], rot[m]);
                rest_frame<R, NR>(x0e, rin[m]);
                if (one) stiffness_from_volume(x0e, in.ks, kk[m]);
            }
        }
        __syncthreads();
    }
    // ---- 3. element K p into LDS
    const R kcg = (R)in.k_cg, mcg = (R)in.m_cg;
#pragma unroll
    for (int m = 0; m < EPT; m++) {
        const int k = threadIdx.x + m * TB;
        if (k < td.e_count) {
            int l[4];
            unpack_ltet(lt[m], l);
            R u[12], c[12];
#pragma unroll
            for (int n = 0; n < 4; n++)
#pragma unroll
                for (int i = 0; i < 3; i++) u[3 * n + i] = (R)lu[3 * l[n] + i];
            elem_dforce_r<R, NR>(rot[m], rin[m], kk[m], u, kcg, c);
            if (consistent) add_edge_mass(mcg * em[m], u, c);
#pragma unroll
            for (int i = 0; i < 12; i++) lc[i * kTileRow + k] = c[i];
        }
    }
    __syncthreads();
    // ---- 4. per-node sums in ascending element id, from LDS only
    if constexpr (!GEO) {
        const int n3 = 3 * td.ln_count;
#pragma unroll 1
        for (int j = threadIdx.x; j < n3; j += TB) {
            const int n = j / 3, c = j - 3 * n;
            const int nf = lnode[n], i0 = nf & (kNodeMass - 1);
            const int i1 = n + 1 < td.ln_count ? (int)(lnode[n + 1] & (kNodeMass - 1)) : ninc;
            VT acc = 0;
            if (nf & kNodeMass) mass_term(in, lmass[n], in.m_cg, lu[j], acc);
            sum_component(linc, i0, i1, lc + c * kTileRow, acc);
            lu[j] = acc;
        }
        __syncthreads();
    }
    // ---- 5. the nodes' results
    double pq = 0.0;
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        const int j = threadIdx.x + m * TB;
        if (w0 + m * TB < td.ln_count && j < td.ln_count) {
            VT qn[3] = {0, 0, 0};
            if constexpr (GEO) {
                const int i1 = j + 1 < td.ln_count ? (int)(lnode[j + 1] & (kNodeMass - 1)) : ninc;
                if (in.m_cg != 0.0 && psl[m] < 0) {
#pragma unroll
                    for (int i = 0; i < 3; i++) mass_term(in, ms[m], in.m_cg, pv[m][i], qn[i]);
                }
                sum_incidences<true>(linc, s0[m], i1, lc, qn);
            } else {
#pragma unroll
                for (int i = 0; i < 3; i++) qn[i] = lu[3 * j + i];
            }
            if (psl[m] < 0) {
                if (PLANE && ct[m]) plane_dforce(in, in.k_cg, pv[m], qn);
                if (fx[m]) { qn[0] = 0; qn[1] = 0; qn[2] = 0; }
                st3(q, gid[m], qn);
                pq += dot3d(pv[m], qn);
            } else {
                st3(sp, psl[m] & (kSlotOwner - 1), qn);
                // p.q is linear in q: a shared node's term is split over its tiles (p . this
                // tile's partial), its mass and plane terms added by its first tile, so that the
                // tile partials hold all of p.q and no later kernel has to add to it
                if (!fx[m]) {
                    pq += dot3d(pv[m], qn);
                    if ((psl[m] & kSlotOwner) && (in.m_cg != 0.0 || (PLANE && ct[m]))) {
                        VT mq[3] = {0, 0, 0};
                        if (in.m_cg != 0.0)
#pragma unroll
                            for (int i = 0; i < 3; i++) mass_term(in, ms[m], in.m_cg, pv[m][i], mq[i]);
                        if (PLANE && ct[m]) plane_dforce(in, in.k_cg, pv[m], mq);
                        pq += dot3d(pv[m], mq);
                    }
                }
            }
        }
    }
    if (w0 < td.ln_count) pq = wave_sum(pq);
    if (lane == 0) sh[threadIdx.x >> 6] = pq;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = sh[0];
#pragma unroll
        for (int k = 1; k < TB / 64; k++) t = t + sh[k];
        pden[td.pslot] = t;
    }
}

// The operator in the reference's summation order, the arithmetic of applyStiffnessCorotational in its
// own order.  |b|^2 and r.r come from InstDev::dots; interior nodes write their p.q term to nd; a
// shared node's leading run (its first incidences in ascending element id, when they lie in this
// tile) is summed here after the mass term into the node's first slot, every later incidence goes to
// a slot of its own (finished by k_fin_exact).
// GEO: how much element geometry is recomputed from node positions instead of read back, with
// the functions and operation order of the element set-up and no fused multiply-adds (so the
// same bits).  1: the rotation, from the current positions x (the ones the force pass used: x changes
// only after the solve) -- 9 reals less per element, 3 more per tile-local node.  2: also the rotated
// rest coordinates from the rest positions x0 (initLarge, TetrahedronFEMForceField.inl:835-868) and,
// for a scene of one material, K from the rest volume -- NR (+ 3) reals less per element, 3 more per
// local node.  Reading all of it back and summing by component, as k_tile_apply does, took 39.2 us against
// 37.4 on 16 beams of 0.56M tetrahedra in double, and 4 % more of the step: the 168 bytes per element
// push the vectors and slots out of L2, and its sums are stored incidence by incidence anyway.
// PLANE = false: no scene of the launch has a PlaneForceField (its per-node terms compiled out).
template <typename R, int NR, typename VT, int TB, int GEO, bool PLANE>
__global__ __launch_bounds__(TB) void k_tile_exact(TileArgs<R, NR> a, int iter, const VT* __restrict__ r,
                                                    VT* __restrict__ p, VT* __restrict__ q, VT* __restrict__ sp,
                                                    const VT* __restrict__ x, const VT* __restrict__ x0) {
    constexpr int EPT = kTileElems / TB;                   // elements per thread
    constexpr int NPT = (kTileNodes + TB - 1) / TB;        // tile-local nodes per thread
    static_assert(GEO == 1 || GEO == 2, "the rotation is recomputed from the positions");
    static_assert(kTileElems * 12 >= kTileNodes * 6, "positions are staged in the contribution buffer");
    __shared__ R lu[kTileNodes * 3];
    __shared__ R lc[kTileRow * 12];
    __shared__ uint16_t linc[kTileElems * 4];
    __shared__ int lptr[kTileNodes + 1];
    const TileDesc td = a.tiles[xcd_item()];
    InstDev* ins = &a.inst[td.scene];
    const InstDev in = *ins;
    const bool kvol = GEO == 2 && (td.flags & kTileOneMaterial) != 0;   // K recomputed, not loaded
    // ---- 1. issue every load that depends on the tile descriptor only: the element records of
    //         this thread (kept in registers), the tile-local node ids / slots / masks, the
    //         incidence tables, the scene record
    R rot[EPT][9], rin[EPT][NR], kk[EPT][3];
    uint2 lt[EPT];
#pragma unroll
    for (int m = 0; m < EPT; m++) {
        const int k = threadIdx.x + m * TB;
        if (k < td.e_count) {
            const int64_t e = (int64_t)td.e_begin + k;
            lt[m] = a.ltet[e];
            if (GEO < 2) {
#pragma unroll
                for (int i = 0; i < NR; i++) rin[m][i] = a.ev.rest[i * a.ev.E + e];
            }
            if (!kvol) {
#pragma unroll
                for (int i = 0; i < 3; i++) kk[m][i] = a.ev.kmat[i * a.ev.E + e];
            }
        }
    }
    // tile-local node tables: every thread loads, at its node or (past the tile's count) at the
    // tile's last node, which every tile has -- no branch, so the compiler keeps all these loads
    // and the gathers that depend on them in flight together; values past the count are unused
    int gid[NPT], psl[NPT], lead[NPT];
    int8_t fx[NPT], ct[NPT];
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        const int j = min((int)threadIdx.x + m * TB, td.ln_count - 1);
        const int li = td.ln_begin + j;
        gid[m] = a.tn.gid[li];
        psl[m] = a.tn.pslot[li];
        lead[m] = a.tn.lead[li];
    }
    // the incidence tables into registers first: their loads are in flight while the node ids
    // arrive and the node gathers below are issued; they go to LDS after those
    const int ninc = 4 * td.e_count;
    constexpr int IPT = (4 * kTileElems + TB - 1) / TB;     // incidences per thread
    constexpr int PPT = (kTileNodes + 1 + TB - 1) / TB;     // incidence pointers per thread
    // (clamped like the node tables; a tile without elements reads entry 0, which every buffer has)
    int inc_r[IPT], ptr_r[PPT];
#pragma unroll
    for (int k = 0; k < IPT; k++) {
        const int j = threadIdx.x + k * TB;
        inc_r[k] = a.tn.inc[ninc > 0 ? td.inc_begin + min(j, ninc - 1) : 0];
    }
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int j = min((int)threadIdx.x + k * TB, td.ln_count);
        ptr_r[k] = a.tn.inc_ptr[td.ln_begin + j] - td.inc_begin;
    }
    // ---- 2. the tile's nodes: r and p (dependent on the node ids), masks; issued before the
    //         scene's stop flag is tested (in-bounds loads, unused for a stopped scene)
    VT rr_[NPT][3], po_[NPT][3], xx_[NPT][3], x0_[NPT][3];
    // p is read from iteration 2 on; without a p (a plain operator application) the loads read r
    // instead, unused
    const VT* __restrict__ pl = p ? p : r;
    const bool plane = PLANE && in.plane_on;
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        ld3(r, gid[m], rr_[m]);
        ld3(pl, gid[m], po_[m]);
        ld3(x, gid[m], xx_[m]);
        if (GEO == 2) ld3(x0, gid[m], x0_[m]);
        fx[m] = a.fixed[gid[m]];
        if (PLANE) {
            const int8_t c = a.contact[gid[m]];
            ct[m] = plane ? c : 0;
        } else {
            ct[m] = 0;
        }
    }
#pragma unroll
    for (int k = 0; k < IPT; k++) {
        const int j = threadIdx.x + k * TB;
        if (j < ninc) linc[j] = (uint16_t)inc_r[k];
    }
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int j = threadIdx.x + k * TB;
        if (j <= td.ln_count) lptr[j] = ptr_r[k];
    }
    const int mark = iter > 0 ? stop_mark(iter, 0) : 0;
    if (stopped_before(in.stopped, mark)) return;
    const bool first = (td.flags & kTileFirst) != 0;
    // ---- 3. scalars: rho, the tolerance test, beta (CGLinearSolver.inl:130-196)
    double beta = 0.0;
    if (iter == 1) {
        const double bb = in.dots[kDotBB];
        const double normb = sqrt(bb);
        if (normb == 0.0) { record_stop(ins, first, mark, 4, 0, 1.0); return; }
        // rho = r.r: b.b from a cold start; warmStart: the r.r of r = b - A x
        const double rho = in.warm_start ? in.dots[kDotRR] : bb;
        const double err = sqrt(rho) / normb;
        if (err <= in.tol && !in.first_solve) { record_stop(ins, first, mark, 1, 1, err); return; }
        if (first && threadIdx.x == 0) {
            ins->normb = normb; ins->rho_slot[1] = rho; ins->iter = 1; ins->err = err;
        }
    } else if (iter > 1) {
        if (iter > in.max_iter) { record_stop(ins, first, mark, 0, in.max_iter, in.err); return; }
        const double rho = in.dots[kDotRR];
        const double err = sqrt(rho) / in.normb;
        if (err <= in.tol) { record_stop(ins, first, mark, 1, iter, err); return; }
        beta = rho / (iter & 1 ? in.rho_slot[0] : in.rho_slot[1]);
        if (first && threadIdx.x == 0) {
            ins->rho_slot[iter & 1] = rho; ins->beta = beta; ins->iter = iter; ins->err = err;
        }
    }
    // ---- 4. stage p = r + beta p (interior nodes: this tile owns p and writes it back)
    const VT vb = (VT)beta;
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        const int j = threadIdx.x + m * TB;
        if (j < td.ln_count) {
            VT pp[3] = {rr_[m][0], rr_[m][1], rr_[m][2]};
            if (iter > 1) {
#pragma unroll
                for (int i = 0; i < 3; i++) { VT t = po_[m][i] * vb; t += pp[i]; pp[i] = t; }
            }
            if (iter > 0 && psl[m] < 0) st3(p, gid[m], pp);
            lu[3 * j] = (R)pp[0]; lu[3 * j + 1] = (R)pp[1]; lu[3 * j + 2] = (R)pp[2];
#pragma unroll
            for (int i = 0; i < 3; i++) lc[3 * j + i] = (R)xx_[m][i];
            if (GEO == 2) {
#pragma unroll
                for (int i = 0; i < 3; i++) lc[3 * kTileNodes + 3 * j + i] = (R)x0_[m][i];
            }
        }
    }
    __syncthreads();
    {   // geometry from the staged positions, then the buffer is free again
        const R* lx = lc;
        const R* lx0 = lc + 3 * kTileNodes;
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const int k = threadIdx.x + m * TB;
            if (k < td.e_count) {
                int l[4];
                unpack_ltet(lt[m], l);
                R p[3][3];
#pragma unroll
                for (int v = 0; v < 3; v++)
#pragma unroll
                    for (int i = 0; i < 3; i++) p[v][i] = lx[3 * l[v] + i];
                rotation_large(p[0], p[1], p[2], rot[m]);
                if (GEO == 2) {
                    R p0[4][3];
#pragma unroll
                    for (int v = 0; v < 4; v++)
#pragma unroll
                        for (int i = 0; i < 3; i++) p0[v][i] = lx0[3 * l[v] + i];
                    rest_frame<R, NR>(p0, rin[m]);
                    if (kvol) stiffness_from_volume(p0, in.ks, kk[m]);
                }
            }
        }
        __syncthreads();
    }
    // ---- 5. element K p into LDS
    const R kcg = (R)in.k_cg;
#pragma unroll
    for (int m = 0; m < EPT; m++) {
        const int k = threadIdx.x + m * TB;
        if (k < td.e_count) {
            int l[4];
            unpack_ltet(lt[m], l);
            R u[12], c[12];
#pragma unroll
            for (int n = 0; n < 4; n++)
#pragma unroll
                for (int i = 0; i < 3; i++) u[3 * n + i] = lu[3 * l[n] + i];
            elem_dforce_r<R, NR>(rot[m], rin[m], kk[m], u, kcg, c);
#pragma unroll
            for (int i = 0; i < 12; i++) lc[i * kTileRow + k] = c[i];
        }
    }
    __syncthreads();
    // ---- 6. per-node sums in ascending element id, from LDS only
#pragma unroll
    for (int m = 0; m < NPT; m++) {
        const int j = threadIdx.x + m * TB;
        if (j < td.ln_count) {
            const int s0 = lptr[j], s1 = lptr[j + 1];
            if (psl[m] < 0) {
                const VT pp[3] = {(VT)lu[3 * j], (VT)lu[3 * j + 1], (VT)lu[3 * j + 2]};
                VT qn[3] = {0, 0, 0};
                if (in.m_cg != 0.0) mass_mdx(in, NodeArrays{nullptr, nullptr, a.mass, a.fixed}, gid[m], in.m_cg, pp, qn);
                sum_incidences<true>(linc, s0, s1, lc, qn);
                if (PLANE && ct[m]) plane_dforce(in, in.k_cg, pp, qn);
                if (fx[m]) { qn[0] = 0; qn[1] = 0; qn[2] = 0; }
                st3(q, gid[m], qn);
                a.nd[gid[m]] = dot3d(pp, qn);
            } else {
                int s = s0;
                if (lead[m] > 0) {
                    // this tile holds the node's leading run: the node's sum starts here (the mass
                    // term, then the run's contributions one by one) and goes to its first slot
                    const VT pp[3] = {(VT)lu[3 * j], (VT)lu[3 * j + 1], (VT)lu[3 * j + 2]};
                    VT acc[3] = {0, 0, 0};
                    if (in.m_cg != 0.0) mass_mdx(in, NodeArrays{nullptr, nullptr, a.mass, a.fixed}, gid[m], in.m_cg, pp, acc);
                    s = s0 + lead[m];
                    sum_incidences<true>(linc, s0, s, lc, acc);
                    st3(sp, psl[m], acc);
                }
                store_incidences(linc, a.tn.arank + td.inc_begin, s, s1, lc, sp, psl[m]);
            }
        }
    }
}

// The float record's rest shape and (a scene of one material) K from the rest positions in float, with
// the functions and operation order of the element set-up (initLarge, TetrahedronFEMForceField.inl:835-868)
// and no fused multiply-adds: an operator in float throughout, not one rounded from the host's double.
static __global__ __launch_bounds__(kBlock) void k_rest_float(const int4* __restrict__ tet, int64_t e0, int64_t e1, int64_t E,
                                                               const double* __restrict__ xd, const float* __restrict__ xf,
                                                               bool one_material, double ks0, double ks1, double ks2,
                                                               float* __restrict__ rest, float* __restrict__ kmat) {
    const int64_t e = e0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= e1) return;
    const int4 t = tet[e];
    const int v[4] = {t.x, t.y, t.z, t.w};
    float p[4][3], rin[6];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int64_t o = 3 * (int64_t)v[n] + i;
            p[n][i] = xd ? (float)xd[o] : xf[o];
        }
    rest_frame<float, 6>(p, rin);
#pragma unroll
    for (int i = 0; i < 6; i++) rest[i * E + e] = rin[i];
    if (one_material) {
        const double ks[3] = {ks0, ks1, ks2};
        float k3[3];
        stiffness_from_volume(p, ks, k3);
#pragma unroll
        for (int i = 0; i < 3; i++) kmat[i * E + e] = k3[i];
    }
}

// the rotations of the elements [e0, e1) from the engine's current positions, for a solve that does not
// follow a force pass (component-level CG)
template <typename R, typename VT>
__global__ __launch_bounds__(kBlock) void k_rotations(const int4* __restrict__ tet, int64_t e0, int64_t e1,
                                                       const VT* __restrict__ x, R* __restrict__ rot, int64_t E) {
    const int64_t e = e0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= e1) return;
    const int4 t = tet[e];
    const int v[3] = {t.x, t.y, t.z};
    R p[3][3], ro[9];
#pragma unroll
    for (int n = 0; n < 3; n++)
#pragma unroll
        for (int i = 0; i < 3; i++) p[n][i] = (R)x[3 * (int64_t)v[n] + i];
    rotation_large(p[0], p[1], p[2], ro);
#pragma unroll
    for (int i = 0; i < 9; i++) rot[i * E + e] = ro[i];
}

// reference order, after the tile apply: the shared nodes' p = r + beta p, q = (1 + h rm) M p
// minus their element contributions one by one in ascending element id (continued from the sum
// the leading run's tile left in the node's first slot), plane and projection, and their p.q
// terms for k_scandot (the work k_update does for them in tile order otherwise)
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_fin_exact(const FinBlk* __restrict__ fb_, InstDev* __restrict__ inst,
                                                       SharedNodes sn, const double* __restrict__ mass,
                                                       const int8_t* __restrict__ fixed, int iter,
                                                       const VT* __restrict__ r, VT* __restrict__ p,
                                                       VT* __restrict__ q, const VT* __restrict__ sp,
                                                       double* __restrict__ nd, const int8_t* __restrict__ contact) {
    const FinBlk fb = fb_[xcd_item()];
    const InstDev in = inst[fb.scene];
    if (in.stopped) return;
    const int j = fb.begin + threadIdx.x;
    if (j >= fb.end) return;
    const int g = sn.gid[j];
    VT pp[3];
    ld3(r, g, pp);
    if (iter > 1) {
        const VT vb = (VT)in.beta;
        VT po[3];
        ld3(p, g, po);
#pragma unroll
        for (int i = 0; i < 3; i++) { VT t = po[i] * vb; t += pp[i]; pp[i] = t; }
    }
    st3(p, g, pp);
    // the node's first slot holds its sum up to the end of its leading run (the mass term and
    // that run, added by the run's tile); the rest of its contributions follow, one per slot
    const int s0 = sn.ptr[j], s1 = s0 + 1 + (int)sn.acnt[j];
    VT qn[3];
    ld3(sp, s0, qn);
    sum_slots<true>(sp, s0 + 1, s1, qn);
    if (in.plane_on && contact[g]) plane_dforce(in, in.k_cg, pp, qn);
    if (fixed[g]) { qn[0] = 0; qn[1] = 0; qn[2] = 0; }
    st3(q, g, qn);
    nd[g] = dot3d(pp, qn);
}

// CGLinearSolver warmStart in the reference order (CGLinearSolver.inl:95-99): after the operator
// of iteration 0 on the previous solution (q = A x, shared nodes finished by k_fin_exact),
// r.eq(b, q, -1.0): r = b + q (-1) per component, and each node's r.r term for k_scandot
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_warm_begin_exact(const NodeBlk* __restrict__ nb_,
                                                              const InstDev* __restrict__ inst,
                                                              const VT* __restrict__ b, const VT* __restrict__ q,
                                                              VT* __restrict__ r, double* __restrict__ nd) {
    const NodeBlk nb = nb_[xcd_item()];
    const InstDev in = inst[nb.scene];
    if (!in.warm_start || in.stopped) return;
    const VT m1 = (VT)(-1.0);
#pragma unroll
    for (int k = 0; k < kNodesPerThread; k++) {
        const int n = nb.begin + k * kBlock + threadIdx.x;
        if (n < nb.end) {
            VT bn[3], qn[3], rn[3];
            ld3(b, n, bn);
            ld3(q, n, qn);
#pragma unroll
            for (int i = 0; i < 3; i++) rn[i] = bn[i] + qn[i] * m1;
            st3(r, n, rn);
            nd[n] = dot3d(rn, rn);
        }
    }
}

template <typename VT>
__global__ __launch_bounds__(kBlock) void k_fin_apply(const FinBlk* __restrict__ fb_, InstDev* __restrict__ inst,
                                                       const Ranges* __restrict__ ranges, SharedNodes sn,
                                                       const double* __restrict__ mass,
                                                       const int8_t* __restrict__ fixed, int iter,
                                                       const VT* __restrict__ r, VT* __restrict__ p,
                                                       VT* __restrict__ q, const VT* __restrict__ sp,
                                                       double* __restrict__ pden,
                                                       const int8_t* __restrict__ contact) {
    __shared__ double sh[kBlock / 64];
    const FinBlk fb = fb_[xcd_item()];
    const InstDev in = inst[fb.scene];
    if (in.stopped) return;
    const int j = fb.begin + threadIdx.x;
    double pq = 0.0;
    if (j < fb.end) {
        const int g = sn.gid[j];
        VT pp[3];
        ld3(r, g, pp);
        if (iter > 1) {
            const VT vb = (VT)in.beta;
            VT po[3];
            ld3(p, g, po);
#pragma unroll
            for (int i = 0; i < 3; i++) { po[i] *= vb; po[i] += pp[i]; pp[i] = po[i]; }
        }
        if (iter > 0) st3(p, g, pp);
        VT qn[3] = {0, 0, 0};
        if (in.m_cg != 0.0) mass_mdx(in, NodeArrays{nullptr, nullptr, mass, fixed}, g, in.m_cg, pp, qn);
        const int s0 = sn.ptr[j], s1 = sn.ptr[j + 1];
        sum_slots<false>(sp, s0, s1, qn);
        if (in.plane_on && contact[g]) plane_dforce(in, in.k_cg, pp, qn);
        if (fixed[g]) { qn[0] = 0; qn[1] = 0; qn[2] = 0; }
        st3(q, g, qn);
        pq = dot3d(pp, qn);
    }
    const double own = wave_block_sum<kBlock>(pq, sh);
    if (threadIdx.x == 0) pden[fb.pslot] = fold_tiles(pden, ranges[fb.scene], fb.bi) + own;
}

// z = P^-1 r of a MIXED inner CG's preconditioner (the scene's kind: 0 none, 1 the inverted
// diagonal dinv, 3 per node, 2 the inverted 3x3 block binv, 9 per node, row-major), in float
__device__ __forceinline__ void precond_load(int kind, const float* __restrict__ dinv, const float* __restrict__ binv,
                                             int n, float B[9]) {
    const float* p = kind == 2 ? binv + 9 * (int64_t)n : dinv + 3 * (int64_t)n;
#pragma unroll
    for (int i = 0; i < 9; i++) B[i] = 0.0f;
    if (kind != 0) {
#pragma unroll
        for (int i = 0; i < 3; i++) B[i] = p[i];
    }
    if (kind == 2) {
#pragma unroll
        for (int i = 3; i < 9; i++) B[i] = p[i];
    }
}
template <typename VT>
__device__ __forceinline__ void precond_mul(int kind, const float B[9], const VT r[3], VT z[3]) {
    if (kind == 1) {
#pragma unroll
        for (int i = 0; i < 3; i++) z[i] = r[i] * (VT)B[i];
    } else if (kind == 2) {
#pragma unroll
        for (int i = 0; i < 3; i++) {
            VT t = r[0] * (VT)B[3 * i];
            t += r[1] * (VT)B[3 * i + 1];
            t += r[2] * (VT)B[3 * i + 2];
            z[i] = t;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 3; i++) z[i] = r[i];
    }
}
template <typename VT>
__device__ __forceinline__ void precond_z(int kind, const float* __restrict__ dinv, const float* __restrict__ binv,
                                          int n, const VT r[3], VT z[3]) {
    float B[9];
    precond_load(kind, dinv, binv, n, B);
    precond_mul(kind, B, r, z);
}

// CG iteration `iter` after the tile apply.  Nodes shared by several tiles are finished here:
// p = r + beta p, q = (1 + h rm) M p + their tile partials in tile order, projection (the work
// CGLinearSolver's p update and GraphScatteredMatrix::apply do for them).  Then den = p.q from
// the tile partials (which already hold every node's term), the threshold test and alpha
// (CGLinearSolver.inl:207-265), x += alpha p, r -= alpha q and the r.r partials.
// EXACT: every node's p and q are final (k_fin_exact finished the shared ones), den is the
// reference-order p.q of k_scandot, and each node's r.r term goes to nd.  zbuf (MIXED inner CG
// with a preconditioner): it holds z = P^-1 r of the previous residual (shared nodes' p = z +
// beta p); each node's new z (precond_z with dinv / binv) replaces it, r.z partials in place of r.r
// One thread per node, and everything that a node may need -- a shared node's slot range and its first
// kSlotBatch partials, mass, masks, the preconditioner's block -- on its way before the sum of the tile
// partials: what bounds it is that chain of dependent loads (node block, scene and ranges, partials; node,
// its slots, their partials), not bytes.  Two nodes per thread, and the shared nodes' loads after the sum,
// took: FP32 4,000 nodes 6.3 us, now 4.8 (a launch that waits for the one before costs 4 by itself); MIXED
// with block-Jacobi 40k nodes 8.3, now 5.5; FP64 60k nodes 9.6, now 7.0; FP32 280k nodes 11.2, now 10.8.
constexpr int kUpdateThreads = kBlock * kNodesPerThread;   // a node block, as the partials of r.r are formed
static_assert(kUpdateThreads <= 1024, "one thread per node of a node block");
template <typename VT, bool EXACT = false>
__global__ __launch_bounds__(kUpdateThreads) void k_update(const NodeBlk* __restrict__ nb_, InstDev* __restrict__ inst,
                                                    const Ranges* __restrict__ ranges, int iter, SharedNodes sn,
                                                    const VT* __restrict__ sp, const double* __restrict__ mass,
                                                    const int8_t* __restrict__ fixed, VT* __restrict__ p,
                                                    const VT* __restrict__ q, VT* __restrict__ xcg, VT* __restrict__ r,
                                                    const double* __restrict__ pden, double* __restrict__ prho,
                                                    const int8_t* __restrict__ contact, double* __restrict__ nd = nullptr,
                                                    const float* __restrict__ dinv = nullptr,
                                                    const float* __restrict__ binv = nullptr, VT* __restrict__ zbuf = nullptr) {
    constexpr int kSlotBatch = 4;
    __shared__ double sh[2][kBlock / 64];
    __shared__ double upper[EXACT ? 1 : kUpdateThreads - kBlock + 1];
    const NodeBlk nb = nb_[xcd_item()];
    const int mark = stop_mark(arrived(iter, nb.scene), 1);
    InstDev* ins = &inst[nb.scene];
    const InstDev in = *ins;
    const Ranges rg = ranges[nb.scene];
    const int t = threadIdx.x, lane = t & 63;
    // node data first (registers), then the reduction: every load at a clamped node index (a node past
    // the block's end repeats its last node, unused), p and q also where the shared-node path replaces them
    const bool mine = nb.begin + t < nb.end;
    const int n = min(nb.begin + t, nb.end - 1);
    const int of = EXACT ? -1 : sn.of[n];
    SceneTerms part;
    if (!EXACT) load_terms<kBlock, true>(pden + rg.t0, rg.nt, part);
    VT pv[3], qv[3], xv[3], rv[3], zv[3];
    ld3(xcg, n, xv);
    ld3(r, n, rv);
    if (zbuf) ld3(zbuf, n, zv);
    ld3(p, n, pv);
    ld3(q, n, qv);
    if (stopped_before(in.stopped, mark)) return;
    VT m = 0;
    int8_t fx = 0, ct = 0;
    float B[9];
    int s0 = 0, s1 = 0;
    VT sv[kSlotBatch][3];
    if (!EXACT) {
        m = in.mass_kind == kMassUniform ? (VT)in.vertex_mass : (VT)mass[n];
        fx = fixed[n];
        if (in.plane_on) ct = contact[n];
        if (zbuf) precond_load(in.pcg, dinv, binv, n, B);
        if (of >= 0) {
            s0 = sn.ptr[of];
            s1 = sn.ptr[of + 1];
#pragma unroll
            for (int k = 0; k < kSlotBatch; k++) ld3(sp, min(s0 + k, s1 - 1), sv[k]);
        }
    }
    const bool cont = iter == 1 && in.keep_dir && in.sweep > 1;
    const bool first = nb.first != 0;
    double den;
    if constexpr (EXACT) den = in.dots[kDotPQ];
    else den = sum_terms<kBlock, true>(pden + rg.t0, rg.nt, part, sh[0]);
    const bool exempt = (iter == 1 && in.first_solve);
    if (den == 0.0) { record_stop(ins, first, mark, 3, iter, in.err); if (first && t == 0) ins->den = den; return; }
    if (fabs(den) <= in.thr && !exempt) {
        record_stop(ins, first, mark, 2, iter, in.err);
        if (first && t == 0) ins->den = den;
        return;
    }
    const double alpha = (iter & 1 ? in.rho_slot[1] : in.rho_slot[0]) / den;
    if (first && t == 0) { ins->den = den; ins->alpha = alpha; }
    const VT vb = (VT)in.beta;
    const VT va = (VT)alpha, vma = (VT)(-alpha);
    double rr = 0.0;
    if (mine) {
        if (of >= 0) {
            VT pp[3] = {rv[0], rv[1], rv[2]};
            if (zbuf) {
#pragma unroll
                for (int i = 0; i < 3; i++) pp[i] = zv[i];
            }
            if (iter > 1 || cont) {
#pragma unroll
                for (int i = 0; i < 3; i++) { VT w = pv[i] * vb; w += pp[i]; pp[i] = w; }
            }
            st3(p, n, pp);
            VT qn[3] = {0, 0, 0};
            if (in.m_cg != 0.0) {
#pragma unroll
                for (int i = 0; i < 3; i++) mass_term(in, m, in.m_cg, pp[i], qn[i]);
            }
#pragma unroll
            for (int k = 0; k < kSlotBatch; k++) {
#pragma unroll
                for (int i = 0; i < 3; i++) qn[i] = s0 + k < s1 ? qn[i] + sv[k][i] : qn[i];
            }
            sum_slots<false>(sp, s0 + kSlotBatch, s1, qn);
            if (ct) plane_dforce(in, in.k_cg, pp, qn);
            if (fx) { qn[0] = 0; qn[1] = 0; qn[2] = 0; }
#pragma unroll
            for (int i = 0; i < 3; i++) { pv[i] = pp[i]; qv[i] = qn[i]; }
        }
        VT xn[3], rn[3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            xn[i] = xv[i] + pv[i] * va;
            rn[i] = rv[i] + qv[i] * vma;
        }
        st3(xcg, n, xn);
        st3(r, n, rn);
        if (EXACT) {
            nd[n] = dot3d(rn, rn);
        } else if (zbuf) {   // z = P^-1 r for the next iteration, and r.z
            VT zn[3];
            precond_mul(in.pcg, B, rn, zn);
            st3(zbuf, n, zn);
            rr = dot3d(rn, zn);
        } else {
            rr = dot3d(rn, rn);
        }
    }
    if (EXACT) return;
    // the partial of r.r: nodes t, t + kBlock, ... of each of the first kBlock threads, then their tree
    if (t >= kBlock) upper[t - kBlock] = rr;
    __syncthreads();
    if (t < kBlock) {
#pragma unroll
        for (int k = 0; k + 1 < kNodesPerThread; k++) rr += upper[k * kBlock + t];
        rr = wave_sum(rr);
        if (lane == 0) sh[1][t >> 6] = rr;
    }
    __syncthreads();
    if (t == 0) {
        double v = sh[1][0];
#pragma unroll
        for (int k = 1; k < kBlock / 64; k++) v = v + sh[1][k];
        prho[nb.pslot] = v;
    }
}

// start of a component-level CG solve on the tiled kernels: r = b = the caller's right-hand side,
// x = 0, and |b|^2 as per-node-block partials (read by the tile apply of iteration 1 with
// pin_nodes = 1) or, in the reference order, as per-node terms for k_scandot
template <typename VT, bool EXACT = false>
__global__ __launch_bounds__(kBlock) void k_cg_begin_tiled(const NodeBlk* __restrict__ nb_, const VT* __restrict__ b_in,
                                                            int nb0, VT* __restrict__ b, VT* __restrict__ r,
                                                            VT* __restrict__ xcg, double* __restrict__ prho,
                                                            double* __restrict__ nd) {
    __shared__ double sh[kBlock / 64];
    const NodeBlk nb = nb_[xcd_item()];
    double bb = 0.0;
#pragma unroll
    for (int k = 0; k < kNodesPerThread; k++) {
        const int n = nb.begin + k * kBlock + threadIdx.x;
        if (n < nb.end) {
            VT bn[3];
            ld3(b_in, n - nb0, bn);
            st3(b, n, bn);
            st3(r, n, bn);
            const VT z[3] = {0, 0, 0};
            st3(xcg, n, z);
            if (EXACT) nd[n] = dot3d(bn, bn);
            else bb += dot3d(bn, bn);
        }
    }
    if (EXACT) return;
    const double tot = wave_block_sum<kBlock>(bb, sh);
    if (threadIdx.x == 0) prho[nb.pslot] = tot;
}

template <typename VT>
__global__ __launch_bounds__(kBlock) void k_integrate(const NodeBlk* __restrict__ nb_, InstDev* __restrict__ inst,
                                                       const int8_t* __restrict__ fixed,
                                                       const VT* __restrict__ xcg, VT* __restrict__ v,
                                                       VT* __restrict__ x) {
    const NodeBlk nb = nb_[xcd_item()];
    const InstDev in = inst[nb.scene];
    const VT h = (VT)in.dt;
    // v += dv (firstOrder: v = dv), x += v h, then vdamping's v *= exp(-h d)
    // (EulerImplicitSolver.cpp:246-299)
    const bool first_order = in.first_order != 0, damp = in.vdamp != 1.0;
    const VT vd = (VT)in.vdamp;
#pragma unroll
    for (int k = 0; k < kNodesPerThread; k++) {
        const int n = nb.begin + k * kBlock + threadIdx.x;
        if (n < nb.end) {
            const int64_t o = 3 * (int64_t)n;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                const VT vv = first_order ? xcg[o + i] : v[o + i] + xcg[o + i];
                x[o + i] = x[o + i] + vv * h;
                v[o + i] = damp ? vv * vd : vv;
            }
            // FixedProjectiveConstraint::projectVelocity (.inl:237-258), when activated
            if (in.project_velocity && (fixed[n] & 1)) {
#pragma unroll
                for (int i = 0; i < 3; i++) v[o + i] = 0;
            }
        }
    }
}

// scene bookkeeping after the update (one thread per scene of the launch set)
static __global__ void k_step_end_tiled(const int* __restrict__ scenes, int n, InstDev* __restrict__ inst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    InstDev* in = &inst[scenes[i]];
    if (!in->stopped) { in->stopped = 1; in->end_reason = 0; in->last_iters = in->max_iter; }
    in->first_solve = 0;
    in->step_count += 1;
    in->time += in->dt;
    in->lm_x0_set = 1;
    in->stopped = 0;   // ready for the next solve
}

}  // namespace sofa_amd
