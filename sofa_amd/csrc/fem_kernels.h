// fem_kernels.h -- the kernels of one implicit Euler step, batched over scenes.
//
// One launch per phase covers every scene of the launch set: element kernels walk a list of
// element blocks, node kernels a list of node blocks; each block belongs to exactly one scene
// (Blk.inst), so per-scene scalars (CG alpha, beta, stop flags) are block-uniform and a scene
// that has left its CG loop costs one early return per block.
//
// Step schedule (EulerImplicitSolver.cpp:83-300 + CGLinearSolver.inl:71-315):
//   k_rhs_elem    rotations from x, element force F(x), element K v          (1 element pass)
//   k_rhs_node    f = m g + sum F; b = h (f - rm M v - (h+rs) K v); project;
//                 r = b; x_cg = 0; |b| and rho = r.r                          (1 node pass)
//   per CG iteration:
//     k_cg_elem   beta; p = r + beta p at the 4 gathered nodes; element K p  (1 element pass)
//     k_cg_node   p (owned node); q = (1 + h rm) M p - h(h+rs) K p; project; p.q
//     k_cg_update alpha; x_cg += alpha p; r -= alpha q; r.r
//   k_euler_update  v += x_cg; x += h v
//   k_finalize      time += dt, timeStepCount++
// Node sums run over each node's incidence list in ascending element id: the order in which
// the reference's element loop accumulates into that node.  No float atomics anywhere.
#pragma once

#include "fem_device.h"

namespace sofa_amd {

struct NodeArrays {
    const int* __restrict__ inc_ptr;   // per node [inc_ptr[n], inc_ptr[n+1]) in inc
    const int* __restrict__ inc;       // element*4 + local vertex, ascending element id
    const double* __restrict__ mass;   // per-node mass (DiagonalMass, MeshMatrixMass vertex mass)
    const int8_t* __restrict__ fixed;  // non-zero where a projective constraint clears the response:
                                       // 1 a fixed node, 2 a node driven by an oscillator
    const int* __restrict__ em_ptr;    // MeshMatrixMass edges of each node, ascending edge id:
    const int* __restrict__ em_nbr;    //   the other end
    const double* __restrict__ em_val; //   the edge mass rho V / 20 summed over the edge's tets
    int8_t* __restrict__ contact;      // PlaneForceField: 1 where the node touched the plane at the
                                       // step's force evaluation (its addDForce contact list)
};

// mass kinds of a scene
constexpr int kMassUniform = 0, kMassDiagonal = 1, kMassMatrix = 2, kMassMatrixLumped = 3;
constexpr double kLumpTet = 2.5;   // MeshMatrixMass lumping coefficient of tetrahedra (MeshMatrixMass.inl:1476-1489)

// one component of mass_mdx, m the node's mass (uniform: the scene's).  FUSE: the product and the sum
// rounded once, in float (left to the compiler, its contraction would depend on the code around it)
template <bool FUSE, typename VT>
__device__ __forceinline__ VT mass_add(VT a, VT b, VT c) {
#pragma clang fp contract(off)
    if constexpr (std::is_same<VT, float>::value) {
        if constexpr (FUSE) return __builtin_fmaf(a, b, c);
        float t = a * b;
        asm("" : "+v"(t));
        return c + t;
    } else {
        return c + a * b;
    }
}
template <typename VT>
__device__ __forceinline__ void mass_term(const InstDev& in, VT m, double factor, VT d, VT& out) {
    const VT fct = (VT)factor;
    if (in.mass_kind == kMassUniform) {
        if (factor != 1.0) m *= fct;
        out = mass_add<true>(d, m, out);
    } else if (in.mass_kind == kMassDiagonal && factor == 1.0) {
        out = mass_add<true>(d, m, out);
    } else if (in.mass_kind == kMassMatrixLumped) {
        out = mass_add<true>((d * m) * (VT)kLumpTet, fct, out);
    } else {
        out = mass_add<true>(d * m, fct, out);
    }
}

// entries [first, first + count) of the three vectors a, b, c (n each) one after the other, to pinned host
// memory: bounded by the host link
template <typename VT>
__global__ __launch_bounds__(256) void k_read_state(const VT* __restrict__ a, const VT* __restrict__ b,
                                                    const VT* __restrict__ c, int64_t n, int64_t first, int64_t count,
                                                    VT* __restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (int64_t)gridDim.x * 256) {
        const int64_t k = first + i;
        out[i] = k < n ? a[k] : k < 2 * n ? b[k - n] : c[k - 2 * n];
    }
}

// vertex part of addMDx: UniformMass.inl:403-419, DiagonalMass.inl:536-559, MeshMatrixMass.inl:1987-2030
// SPLIT_Z: onto a sum (the right-hand side) z is rounded twice in float too
template <bool SPLIT_Z = false, typename VT>
__device__ __forceinline__ void mass_mdx(const InstDev& in, const NodeArrays& na, int n, double factor,
                                         const VT d[3], VT out[3]) {
    const auto add = [&](VT a0, VT a1, VT a2, VT f) {
        out[0] = mass_add<true>(a0, f, out[0]);
        out[1] = mass_add<true>(a1, f, out[1]);
        out[2] = mass_add<!SPLIT_Z>(a2, f, out[2]);
    };
    const VT fct = (VT)factor;
    if (in.mass_kind == kMassUniform) {
        VT m = (VT)in.vertex_mass;
        if (factor != 1.0) m *= fct;
        add(d[0], d[1], d[2], m);
    } else {
        const VT m = (VT)na.mass[n], lc = (VT)kLumpTet;
        if (in.mass_kind == kMassDiagonal && factor == 1.0) add(d[0], d[1], d[2], m);
        else if (in.mass_kind == kMassMatrixLumped) add((d[0] * m) * lc, (d[1] * m) * lc, (d[2] * m) * lc, fct);
        else add(d[0] * m, d[1] * m, d[2] * m, fct);
    }
}

// gravity of the mass's addForce: UniformMass.inl:471-496 (m g), DiagonalMass.inl:1393-1413
// (g m_i), MeshMatrixMass.inl:2073-2092 (g m_i 2.5)
template <typename VT>
__device__ __forceinline__ void mass_gravity(const InstDev& in, const double* __restrict__ mass, int n, VT f[3]) {
    if (in.mass_kind == kMassUniform) {
        f[0] = (VT)0 + (VT)in.mg[0]; f[1] = (VT)0 + (VT)in.mg[1]; f[2] = (VT)0 + (VT)in.mg[2];
    } else if (in.mass_kind == kMassDiagonal) {
        const VT m = (VT)mass[n];
#pragma unroll
        for (int i = 0; i < 3; i++) f[i] = (VT)0 + (VT)in.gravity[i] * m;
    } else {
        const VT m = (VT)mass[n], lc = (VT)kLumpTet;
#pragma unroll
        for (int i = 0; i < 3; i++) f[i] = (VT)0 + ((VT)in.gravity[i] * m) * lc;
    }
}

// edge part of the consistent MeshMatrixMass addMDx (MeshMatrixMass.inl:2014-2026): for each
// edge of node n in ascending edge id, out += d[other] * (edgeMass * factor); `dof(j, v)` gives the
// NC components of the multiplied vector at node j.  Edges are loaded several at a
// time, as Contributions does.
template <int NC, typename VT, typename F>
__device__ __forceinline__ void mass_edges(const NodeArrays& na, int n, double factor, F dof, VT out[NC]) {
    const int s0 = na.em_ptr[n], s1 = na.em_ptr[n + 1];
    const VT fct = (VT)factor;
    constexpr int B = 4;
    for (int s = s0; s < s1; s += B) {
        int nbr[B];
        VT tm[B], d[B][NC];
#pragma unroll
        for (int t = 0; t < B; t++) {
            const int i = min(s + t, s1 - 1);
            nbr[t] = na.em_nbr[i];
            tm[t] = (VT)na.em_val[i] * fct;
        }
#pragma unroll
        for (int t = 0; t < B; t++) dof(nbr[t], d[t]);
#pragma unroll
        for (int t = 0; t < B; t++)
            if (s + t < s1) {
#pragma unroll
                for (int i = 0; i < NC; i++) out[i] += d[t][i] * tm[t];
            }
    }
}

// mass_edges for one component of p = r + beta p_old, the loads of the first edges apart from their use
template <typename VT>
struct EdgeTerms {
    static constexpr int B = 8;
    int s0, s1;
    VT val[B], rv[B], pv[B];
    __device__ __forceinline__ void batch(const NodeArrays& na, int s, bool old, const VT* __restrict__ r,
                                          const VT* __restrict__ p) {
        int nbr[B];
#pragma unroll
        for (int t = 0; t < B; t++) {
            const int i = max(min(s + t, s1 - 1), 0);
            nbr[t] = na.em_nbr[i];
            val[t] = (VT)na.em_val[i];
        }
#pragma unroll
        for (int t = 0; t < B; t++) {
            const int64_t w = 3 * (int64_t)nbr[t];
            rv[t] = r[w];
            pv[t] = old ? p[w] : (VT)0;
        }
    }
    __device__ __forceinline__ void load(const NodeArrays& na, int n, bool old, const VT* __restrict__ r,
                                         const VT* __restrict__ p) {
        s0 = na.em_ptr[n];
        s1 = na.em_ptr[n + 1];
        if (s0 < s1) batch(na, s0, old, r, p);
    }
    __device__ __forceinline__ void add(const NodeArrays& na, double factor, bool old, VT beta, const VT* __restrict__ r,
                                        const VT* __restrict__ p, VT& out) {
        const VT fct = (VT)factor;
        for (int s = s0; s < s1; s += B) {
            if (s > s0) batch(na, s, old, r, p);
#pragma unroll
            for (int t = 0; t < B; t++)
                if (s + t < s1) {
                    VT d = rv[t];
                    if (old) { d = pv[t] * beta; d += rv[t]; }
                    out += d * (val[t] * fct);
                }
        }
    }
};

// A node's element contributions ef[3 slot ..] over its incidence list, in list order, eight
// incidences at a time: their slots, then their values, are loaded together (the tail at clamped
// indices), so a node of 24 tetrahedra waits for memory 6 times instead of 48.  Latency is what
// bounds the node kernels: the CG node kernel, a lane per node, went from 14.0 to 10.3 us on 525 nodes
// and from 25.7 to 21.7 on 57,000.  Contributions: one component, the loads apart from the adds, so
// that the first can be in flight while the scene's scalars are summed, and each eight while the eight
// before are added.
template <typename VT>
struct Contributions {
    static constexpr int B = 8;
    int slot[B];
    VT c[B];
    __device__ __forceinline__ void slots(const int* __restrict__ inc, int s, int s1) {
#pragma unroll
        for (int t = 0; t < B; t++) slot[t] = inc[max(min(s + t, s1 - 1), 0)];
    }
    __device__ __forceinline__ void values(const VT* __restrict__ ef) {
#pragma unroll
        for (int t = 0; t < B; t++) c[t] = ef[3 * (int64_t)slot[t]];
    }
    // the first eight values, and the next eight slots, on their way (a node of no element reads another's, or
    // entry 0, which every engine's lists and contributions have, and adds nothing)
    __device__ __forceinline__ void begin(const int* __restrict__ inc, int s0, int s1, const VT* __restrict__ ef) {
        slots(inc, s0, s1);
        values(ef);
        if (s0 + B < s1) slots(inc, s0 + B, s1);
    }
    // acc -= all of them in list order, each eight while the next are on their way
    __device__ __forceinline__ void subtract(const int* __restrict__ inc, int s0, int s1, const VT* __restrict__ ef, VT& acc) {
        for (int s = s0; s < s1; s += B) {
            VT now[B];
#pragma unroll
            for (int t = 0; t < B; t++) now[t] = c[t];
            if (s + B < s1) {
                values(ef);
                if (s + 2 * B < s1) slots(inc, s + 2 * B, s1);
            }
#pragma unroll
            for (int t = 0; t < B; t++)
                if (s + t < s1) acc -= now[t];
        }
    }
};
template <bool SUB, typename VT>
__device__ __forceinline__ void gather_contributions(const int* __restrict__ inc, int s0, int s1,
                                                     const VT* __restrict__ ef, VT acc[3]) {
    constexpr int B = 8;
    for (int s = s0; s < s1; s += B) {
        int slot[B];
        VT c[B][3];
#pragma unroll
        for (int t = 0; t < B; t++) slot[t] = inc[min(s + t, s1 - 1)];
#pragma unroll
        for (int t = 0; t < B; t++) load3(ef, slot[t], c[t][0], c[t][1], c[t][2]);
#pragma unroll
        for (int t = 0; t < B; t++)
            if (s + t < s1) {
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    if (SUB) acc[i] -= c[t][i];
                    else acc[i] += c[t][i];
                }
            }
    }
}

template <typename VT>
__device__ __forceinline__ double dot3d(const VT a[3], const VT b[3]) {
    double r = (double)a[0] * (double)b[0];
    r += (double)a[1] * (double)b[1];
    r += (double)a[2] * (double)b[2];
    return r;
}

// z = P^-1 r with P^-1 stored as 9 doubles per node (row-major): DiagonalMatrix::mult
// (z_i = d_i r_i, DiagonalMatrix.h:187-190) or BlockDiagonalMatrix::mul (z_j = sum_i B(i, j) r_i
// from 0, BlockDiagonalMatrix.h:202-221) -- the preconditioner solve of PCGLinearSolver
template <typename VT>
__device__ __forceinline__ void precond_apply(int kind, const double* __restrict__ P, const VT r[3], VT z[3]) {
    if (kind == 1) {
#pragma unroll
        for (int a = 0; a < 3; a++) z[a] = (VT)(P[4 * a] * (double)r[a]);
    } else {
#pragma unroll
        for (int j = 0; j < 3; j++) {
            double acc = 0.0;
#pragma unroll
            for (int a = 0; a < 3; a++) acc += P[3 * a + j] * (double)r[a];
            z[j] = (VT)acc;
        }
    }
}

// the end of a node kernel of three threads per node: each node's three products added in dot3d's
// order, to nd (reference order) or, by block_sum's tree over the block's 256 nodes, to one partial
__device__ __forceinline__ double tree_256(const double* sh);
__device__ __forceinline__ void node_partial(const double* pr, double* sh, double* __restrict__ nd, const Blk& bk,
                                             double* __restrict__ partial) {
    __syncthreads();
    const int t = threadIdx.x;
    if (t < kBlock) {
        double v = pr[3 * t];
        v += pr[3 * t + 1];
        v += pr[3 * t + 2];
        sh[t] = v;
        if (nd && bk.begin + t < bk.end) nd[bk.begin + t] = v;
    }
    if (nd) return;
    __syncthreads();
    if (t < 64) {
        const double v = tree_256(sh);
        if (t == 0) partial[bk.pad] = v;
    }
}

__device__ __forceinline__ int blk_scene(const Blk& b) { return b.inst; }

// CGLinearSolver.inl:86-160 for nb_iter = 1 (rho = r.r = b.b), once |b|^2 is known: the exact
// path's CG scalars of a scene at the start of a solve
__device__ __forceinline__ void cg_start(InstDev* ins, double total) {
    ins->normb = sqrt(total);
    ins->rho_slot[1] = total;
    ins->iter = 1;
    ins->stopped = 0;
    ins->end_reason = 0;
    ins->err = 1.0;
    ins->den = 0.0;
    if (ins->normb == 0.0) {
        ins->stopped = 1; ins->end_reason = 4; ins->last_iters = 0;
    } else {
        const double err = sqrt(total) / ins->normb;
        ins->err = err;
        if (err <= ins->tol && !ins->first_solve) { ins->stopped = 1; ins->end_reason = 1; ins->last_iters = 1; }
    }
}

// CGLinearSolver's first tests after a warm start: |b| from b.b, rho = r.r of r = b - A x, the
// iteration-1 tolerance test with the first step's exemption (CGLinearSolver.inl:94-105,139-170)
__device__ __forceinline__ void cg_start_warm(InstDev* ins, double bb, double rr) {
    ins->normb = sqrt(bb);
    ins->rho_slot[1] = rr;
    ins->iter = 1;
    ins->stopped = 0;
    ins->end_reason = 0;
    ins->err = 1.0;
    ins->den = 0.0;
    if (ins->normb == 0.0) {
        ins->stopped = 1; ins->end_reason = 4; ins->last_iters = 0;
    } else {
        const double err = sqrt(rr) / ins->normb;
        ins->err = err;
        if (err <= ins->tol && !ins->first_solve) { ins->stopped = 1; ins->end_reason = 1; ins->last_iters = 1; }
    }
}

// end of a component-level CG solve (no time step) on the tiled kernels: the loop's exit record,
// timeStepCount++ (CGLinearSolver.inl:300), reopened (they run with stopped == 0)
static __global__ void k_solve_end(const int* __restrict__ scenes, int n, InstDev* __restrict__ inst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    InstDev* in = &inst[scenes[i]];
    if (!in->stopped) { in->end_reason = 0; in->last_iters = in->max_iter; }
    in->first_solve = 0;
    in->step_count += 1;
    in->stopped = 0;
}

// ---------------------------------------------------------------------------------------
// RHS
// ---------------------------------------------------------------------------------------
template <typename R, int NR, typename VT>
__global__ __launch_bounds__(kBlock) void k_rhs_elem(ElemView<R, NR> ev, const Blk* __restrict__ eblk,
                                                      const InstDev* __restrict__ inst, const VT* __restrict__ x,
                                                      const VT* __restrict__ v, VT* __restrict__ ef_f,
                                                      VT* __restrict__ ef_v) {
    const Blk bk = eblk[xcd_item()];
    const InstDev in = inst[bk.inst];
    const int64_t e = (int64_t)bk.begin + threadIdx.x;
    if (e >= bk.end) return;
    const int4 t = ev.tet[e];
    R rot[9], c[12], g[12];
    elem_force<R, NR, VT>(ev, e, t, x, rot, c, g);
#pragma unroll
    for (int k = 0; k < 9; k++) ev.rot[k * ev.E + e] = rot[k];
#pragma unroll
    for (int k = 0; k < 12; k++) ef_f[12 * e + k] = (VT)c[k];
    // FEM part of addMBKv(b, v): kFactor = h + rs, skipped when 0 (BaseForceField.cpp:38-47)
    if (in.k_rhs != 0.0) {
        R u[12];
        const int nid[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
        for (int n = 0; n < 4; n++) {
            VT a, b, cc;
            load3(v, nid[n], a, b, cc);
            u[3 * n] = (R)a; u[3 * n + 1] = (R)b; u[3 * n + 2] = (R)cc;
        }
        elem_dforce<R, NR>(ev, e, rot, u, (R)in.k_rhs, c);
#pragma unroll
        for (int k = 0; k < 12; k++) ef_v[12 * e + k] = (VT)c[k];
    } else {
#pragma unroll
        for (int k = 0; k < 12; k++) ef_v[12 * e + k] = (VT)0;
    }
}

template <typename VT>
__global__ __launch_bounds__(kBlock) void k_rhs_node(const Blk* __restrict__ nblk, InstDev* __restrict__ inst,
                                                      NodeArrays na, const VT* __restrict__ ef_f,
                                                      const VT* __restrict__ ef_v, const VT* __restrict__ v,
                                                      VT* __restrict__ f, VT* __restrict__ b, VT* __restrict__ r,
                                                      VT* __restrict__ xcg, double* __restrict__ partial,
                                                      double* __restrict__ nd,     // non-null: reference dot order
                                                      const VT* __restrict__ x) {
    __shared__ double sh[kBlock];
    const Blk bk = nblk[xcd_item()];
    InstDev* ins = &inst[bk.inst];
    const int n = bk.begin + threadIdx.x;
    double bb = 0.0;
    if (n < bk.end) {
        const InstDev& in = *ins;
        VT xn[3] = {0, 0, 0}, vn[3] = {0, 0, 0};
        if (in.plane_on) {
            load3(x, n, xn[0], xn[1], xn[2]);
            load3(v, n, vn[0], vn[1], vn[2]);
        }
        // computeForce: f = 0; mass addForce (f += m g); FEM addForce (f += R F, element order)
        VT fn[3];
        mass_gravity(in, na.mass, n, fn);
        const int s0 = na.inc_ptr[n], s1 = na.inc_ptr[n + 1];
        gather_contributions<false>(na.inc, s0, s1, ef_f, fn);
        // PlaneForceField after the FEM (scene order); its contacts are kept for addDForce
        const bool touch = in.plane_on && plane_force(in, xn, vn, fn);
        if (in.plane_on) na.contact[n] = touch ? 1 : 0;
        f[3 * (int64_t)n] = fn[0]; f[3 * (int64_t)n + 1] = fn[1]; f[3 * (int64_t)n + 2] = fn[2];
        // b = f; b += (-rm) M v (mass first); b -= (h+rs) K v (FEM, element order); b *= h
        VT bn[3] = {fn[0], fn[1], fn[2]};
        if (in.m_rhs != 0.0) {
            VT vm[3];
            load3(v, n, vm[0], vm[1], vm[2]);
            mass_mdx(in, na, n, in.m_rhs, vm, bn);
            if (in.mass_kind == kMassMatrix)
                mass_edges<3>(na, n, in.m_rhs, [&](int j, VT d[3]) { load3(v, j, d[0], d[1], d[2]); }, bn);
        }
        gather_contributions<true>(na.inc, s0, s1, ef_v, bn);
        if (touch && in.k_rhs != 0.0) plane_dforce(in, in.k_rhs, vn, bn);
        const VT h = (VT)in.b_scale;   // h (firstOrder: 1, b = f)
        bn[0] *= h; bn[1] *= h; bn[2] *= h;
        if (na.fixed[n]) { bn[0] = 0; bn[1] = 0; bn[2] = 0; }
        const int64_t o = 3 * (int64_t)n;
        b[o] = bn[0]; b[o + 1] = bn[1]; b[o + 2] = bn[2];
        r[o] = bn[0]; r[o + 1] = bn[1]; r[o + 2] = bn[2];
        // PCG and a CG with warmStart start from the last solution
        if (!in.pcg && !in.warm_start) { xcg[o] = 0; xcg[o + 1] = 0; xcg[o + 2] = 0; }
        bb = dot3d(bn, bn);
        if (nd) nd[n] = bb;
    }
    double total;
    const bool last = nd ? last_block_sequential(nd, ins, total)
                         : last_block_reduce(block_sum(bb, sh), partial, ins, bk.pad, sh, total);
    if (last && threadIdx.x == 0) {
        if (ins->pcg || ins->warm_start) ins->bnorm2 = total;
        else cg_start(ins, total);
    }
}

// the exact path's start of CGLinearSolver::solve on a caller's right-hand side (component call):
// r = b, x = 0, |b|^2 and the first iteration's tests as after the RHS
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_cg_begin(const Blk* __restrict__ nblk, InstDev* __restrict__ inst,
                                                      const VT* __restrict__ b_in, int nb0, VT* __restrict__ b,
                                                      VT* __restrict__ r, VT* __restrict__ xcg,
                                                      double* __restrict__ partial, double* __restrict__ nd) {
    __shared__ double sh[kBlock];
    const Blk bk = nblk[xcd_item()];
    InstDev* ins = &inst[bk.inst];
    const int n = bk.begin + threadIdx.x;
    double bb = 0.0;
    if (n < bk.end) {
        VT bn[3];
        load3(b_in, n - nb0, bn[0], bn[1], bn[2]);
        const int64_t o = 3 * (int64_t)n;
        b[o] = bn[0]; b[o + 1] = bn[1]; b[o + 2] = bn[2];
        r[o] = bn[0]; r[o + 1] = bn[1]; r[o + 2] = bn[2];
        xcg[o] = 0; xcg[o + 1] = 0; xcg[o + 2] = 0;
        bb = dot3d(bn, bn);
        if (nd) nd[n] = bb;
    }
    double total;
    const bool last = nd ? last_block_sequential(nd, ins, total)
                         : last_block_reduce(block_sum(bb, sh), partial, ins, bk.pad, sh, total);
    if (last && threadIdx.x == 0) cg_start(ins, total);
}

// ---------------------------------------------------------------------------------------
// CG iteration.  The two node kernels run three threads per node, one per component (a lane's loads
// are then coalesced, and 57,000 nodes give 2,700 waves instead of 890), and leave their dot product
// as one partial per 256-node block; whoever needs the sum adds the partials itself, in the order the
// scalars of a solve have always been summed, so no block waits for or fences against another.  The
// scene's record is written by its first node block only: every field that the other blocks of the
// same kernel read (rho_slot of the other parity, limits) is left alone there, and a stop that it records
// is passed over by them (stopped_before): they reach it themselves.
// ---------------------------------------------------------------------------------------
constexpr int kNodeThreads = 3 * kBlock;

// the tree of block_sum over sh[0 .. 255], by the first wave (lane 0 has the sum)
__device__ __forceinline__ double tree_wave(double v) {
    v = v + __shfl_down(v, 32, 64);
    v = v + __shfl_down(v, 16, 64);
    v = v + dpp_row_from<0x108>(v);
    v = v + dpp_row_from<0x104>(v);
    v = v + dpp_row_from<0x102>(v);
    return v + dpp_row_from<0x101>(v);
}
__device__ __forceinline__ double tree_256(const double* sh) {
    const int l = threadIdx.x;
    return tree_wave((sh[l] + sh[l + 128]) + (sh[l + 64] + sh[l + 192]));
}
// the scene's sum of its node blocks' partials, in every thread: each of 256 threads a strided sum,
// then block_sum's tree (last_block_reduce's order)
template <int TB>
__device__ __forceinline__ double block_partials(const double* __restrict__ partial, const InstDev& in, double* sh) {
    const int nb = in.nblk_count, b0 = in.nblk_begin;
    for (int t = threadIdx.x; t < kBlock; t += TB) {
        double acc = 0.0;
        for (int k = t; k < nb; k += kBlock) acc = acc + partial[b0 + k];
        sh[t] = acc;
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        const double v = tree_256(sh);
        if (threadIdx.x == 0) sh[0] = v;
    }
    __syncthreads();
    return sh[0];
}
// the same from the nodes' terms (at most kSpreadBlocks node blocks, kNodeThreads threads): a wave forms a
// block's partial.  A step of 25 iterations, spread and not: 7 blocks 372 and 457 us, 26 blocks 408 and
// 484, 51 blocks 459 and 505, 64 blocks 503 and 529; beyond, adding the terms costs what the gathers gain
constexpr int kSpreadBlocks = 64, kSpread = 4;
__device__ __forceinline__ double node_partials(const double* __restrict__ nd, const InstDev& in, double* sh) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr int W = kNodeThreads / 64, B = (kSpreadBlocks + W - 1) / W;
    const double* d = nd + in.node_begin;
    double v[B][4];
#pragma unroll
    for (int k = 0; k < B; k++)
        if (wave + k * W < in.nblk_count) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int n = (wave + k * W) * kBlock + lane + 64 * i;
                v[k][i] = n < in.node_count ? d[n] : 0.0;
            }
        }
    if (threadIdx.x < kBlock) sh[threadIdx.x] = 0.0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < B; k++)
        if (wave + k * W < in.nblk_count) {
            const double t = tree_wave((v[k][0] + v[k][2]) + (v[k][1] + v[k][3]));
            if (lane == 0) sh[wave + k * W] = t;
        }
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x < 64) t = tree_256(sh);
    __syncthreads();
    if (threadIdx.x == 0) sh[0] = t;
    __syncthreads();
    return sh[0];
}
// a dot product of the scene: already in its record (`ready`: summed in the reference's order, or
// by k_cg_total), or from the partials
template <int TB>
__device__ __forceinline__ double cg_dot(const double* __restrict__ partial, const InstDev& in, int which, int ready,
                                         double* sh) {
    return ready ? in.dots[which] : block_partials<TB>(partial, in, sh);
}
// a scene of many node blocks: its partials added once, by one block per scene, instead of by every
// block of the next kernel
static __global__ __launch_bounds__(kBlock) void k_cg_total(const int* __restrict__ scenes, InstDev* __restrict__ inst,
                                                             const double* __restrict__ partial, int which) {
    __shared__ double sh[kBlock];
    InstDev* ins = &inst[scenes[blockIdx.x]];
    if (ins->stopped) return;
    const double v = block_partials<kBlock>(partial, *ins, sh);
    if (threadIdx.x == 0) ins->dots[which] = v;
}

// the tests before iteration `it` (2 or later) with rho = r.r (PCG: r.z) of the last one: false when
// the loop ends, else beta.  CGLinearSolver.inl:130-196; PCGLinearSolver.inl:241-246 (while iter <=
// maxIter && r_norm > tol).  `first` (the scene's first node block): recorded.
__device__ __forceinline__ bool cg_next(InstDev* ins, const InstDev& in, int it, double rho, bool first, double& beta) {
    const bool record = first && threadIdx.x == 0;
    const bool over = it > in.max_iter;
    double err = 0.0;
    bool stop = over;
    if (in.pcg) {
        err = in.bnorm2 != 0.0 ? rho / in.bnorm2 : 0.0;
        stop = over || !(rho > in.pcg_tol);
    } else if (!over) {
        err = sqrt(rho) / in.normb;
        stop = err <= in.tol;
    }
    beta = rho / (it & 1 ? in.rho_slot[0] : in.rho_slot[1]);
    if (record) {
        if (in.pcg || !over) ins->err = err;
        if (stop) {
            ins->stopped = stop_mark(it, 0);
            ins->end_reason = over ? 0 : 1;
            ins->last_iters = over && !in.pcg ? in.max_iter : it;
        } else {
            ins->rho_slot[it & 1] = rho;
            ins->beta = beta;
            ins->iter = it;
        }
    }
    return !stop;
}

// prr: partials of r.r (r.z) of the previous iteration
template <typename R, int NR, typename VT>
__global__ __launch_bounds__(kBlock) void k_cg_elem(ElemView<R, NR> ev, const Blk* __restrict__ eblk,
                                                     InstDev* __restrict__ inst, const VT* __restrict__ r_,
                                                     const VT* __restrict__ p_old, VT* __restrict__ ef, int it,
                                                     const double* __restrict__ prr, int ready,
                                                     const VT* __restrict__ z = nullptr) {
    __shared__ double sh[kBlock];
    const Blk bk = eblk[xcd_item()];
    InstDev* ins = &inst[bk.inst];
    const InstDev in = *ins;
    if (in.stopped) return;
    // PCG: the direction is built from the preconditioned residual z (w = z + beta w)
    const VT* __restrict__ r = (in.pcg && z) ? z : r_;
    const int64_t e = min((int64_t)bk.begin + threadIdx.x, (int64_t)bk.end - 1);
    const int4 t = ev.tet[e];
    const int nid[4] = {t.x, t.y, t.z, t.w};
    VT rn[4][3], po[4][3];
#pragma unroll
    for (int n = 0; n < 4; n++) {
        load3(r, nid[n], rn[n][0], rn[n][1], rn[n][2]);
        if (it > 1) load3(p_old, nid[n], po[n][0], po[n][1], po[n][2]);
    }
    double beta_d = 0.0;
    if (it > 1 && !cg_next(ins, in, it, cg_dot<kBlock>(prr, in, kDotRR, ready, sh), false, beta_d)) return;
    if ((int64_t)bk.begin + threadIdx.x >= bk.end) return;
    const VT beta = (VT)beta_d;
    R u[12];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int i = 0; i < 3; i++) {
            VT d = rn[n][i];
            // cgstep_beta, GraphScattered: p *= beta; p += r (CGLinearSolver.cpp:40-44)
            if (it > 1) { VT w = po[n][i] * beta; w += d; d = w; }
            u[3 * n + i] = (R)d;
        }
    R rot[9], c[12];
    load_rot(ev, e, rot);
    elem_dforce<R, NR>(ev, e, rot, u, (R)in.k_cg, c);
#pragma unroll
    for (int k = 0; k < 12; k++) ef[12 * e + k] = (VT)c[k];
}

// p (owned node), q = (1 + h rm) M p - h(h + rs) K p, projected; p.q per 256-node block into ppq, or
// per node into nd (reference order).  S > 1: S workgroups per node block, p.q per node into nd, for the
// update to form the blocks' partials (node_partials).  What bounds it: the gathers' latency, and on a
// scene of few blocks the few CUs that issue them (525 nodes: 3, 9,000: 36).  With S = 4, 525 nodes took
// 4.8 instead of 7.9 us and 9,000 nodes with edge masses 8.3 instead of 17.2, the update 4.8 and 6.3
// instead of 4.7 and 4.8.
template <typename VT, int S>
__global__ __launch_bounds__(kNodeThreads / S) void k_cg_node(const Blk* __restrict__ nblk, InstDev* __restrict__ inst,
                                                           NodeArrays na, const VT* __restrict__ ef,
                                                           const VT* __restrict__ r_, const VT* __restrict__ p_old,
                                                           VT* __restrict__ p, VT* __restrict__ q, int it,
                                                           const double* __restrict__ prr, int ready,
                                                           double* __restrict__ ppq, double* __restrict__ nd,
                                                           const VT* __restrict__ z = nullptr) {
    constexpr int N = kBlock / S;
    __shared__ double sh[kBlock], pr[3 * N];
    const int item = xcd_item();
    const Blk bk = nblk[item / S];
    const int first = bk.begin + item % S * N;
    InstDev* ins = &inst[bk.inst];
    const InstDev in = *ins;
    if (stopped_before(in.stopped, stop_mark(it, 0))) return;
    const VT* __restrict__ r = (in.pcg && z) ? z : r_;
    const int j = threadIdx.x / 3, c = threadIdx.x - 3 * j;
    const int n = min(first + j, bk.end - 1);
    const bool live = first + j < bk.end;
    const int64_t o = 3 * (int64_t)n + c;
    const VT rc = r[o], pc = p_old[o];
    const int s0 = na.inc_ptr[n], s1 = na.inc_ptr[n + 1];
    const bool fixed = na.fixed[n] != 0;
    // the node's mass, its first edges and its first contributions in flight while the scene's scalars are summed
    const VT m = in.mass_kind == kMassUniform ? (VT)in.vertex_mass : (VT)na.mass[n];
    const bool edges = in.m_cg != 0.0 && in.mass_kind == kMassMatrix;
    EdgeTerms<VT> e;
    if (edges) e.load(na, n, it > 1, r + c, p_old + c);
    Contributions<VT> g;
    g.begin(na.inc, s0, s1, ef + c);
    double beta_d = 0.0;
    if (it > 1 && !cg_next(ins, in, it, cg_dot<kNodeThreads / S>(prr, in, kDotRR, ready, sh), in.node_begin == first, beta_d)) return;
    const VT beta = (VT)beta_d;
    // p = r (first iteration) or p *= beta; p += r (cgstep_beta), from the previous p
    VT pn = rc;
    if (it > 1) { pn = pc * beta; pn += rc; }
    if (live) p[o] = pn;
    // q = 0; mass addMDx(q, p, 1 + h rm); FEM addDForce(q, p, -h(h+rs)); projectResponse(q)
    VT qn = 0;
    if (in.m_cg != 0.0) {
        mass_term(in, m, in.m_cg, pn, qn);
        if (edges) e.add(na, in.m_cg, it > 1, beta, r + c, p_old + c, qn);
    }
    g.subtract(na.inc, s0, s1, ef + c, qn);
    if (in.plane_on) {
        pr[threadIdx.x] = (double)pn;
        __syncthreads();
        if (na.contact[n]) {
            const VT dx[3] = {(VT)pr[3 * j], (VT)pr[3 * j + 1], (VT)pr[3 * j + 2]};
            VT df[3] = {qn, qn, qn};
            plane_dforce(in, in.k_cg, dx, df);
            qn = c == 0 ? df[0] : c == 1 ? df[1] : df[2];
        }
        __syncthreads();
    }
    if (fixed) qn = 0;
    if (live) q[o] = qn;
    pr[threadIdx.x] = live ? (double)pn * (double)qn : 0.0;
    if constexpr (S == 1) {
        node_partial(pr, sh, nd, bk, ppq);
    } else {
        __syncthreads();
        const int t = threadIdx.x;
        if (t < N && first + t < bk.end) {
            double v = pr[3 * t];
            v += pr[3 * t + 1];
            v += pr[3 * t + 2];
            nd[first + t] = v;
        }
    }
}

// den = p.q, the threshold test and alpha (CGLinearSolver.inl:207-265; PCG: alpha = r.z / w.s,
// PCGLinearSolver.inl:222-224), then x += p alpha; r += q (-alpha) (CGLinearSolver.cpp:46-64,
// vOp_v_inc_bf) and the partials of r.r (PCG: s = P^-1 r, r.s, PCGLinearSolver.inl:229-244)
// TERMS: p.q is formed from the nodes' terms (k_cg_node with S > 1, not ready)
template <typename VT, bool TERMS>
__global__ __launch_bounds__(kNodeThreads) void k_cg_update(const Blk* __restrict__ nblk, InstDev* __restrict__ inst,
                                                             const VT* __restrict__ p, const VT* __restrict__ q,
                                                             VT* __restrict__ xcg, VT* __restrict__ r, int it,
                                                             const double* __restrict__ ppq, int ready,
                                                             double* __restrict__ prr, double* __restrict__ nd,
                                                             const double* __restrict__ terms = nullptr,
                                                             const double* __restrict__ pinv = nullptr,
                                                             VT* __restrict__ z = nullptr) {
    __shared__ double sh[kBlock], pr[kNodeThreads];
    const Blk bk = nblk[xcd_item()];
    const int mark = stop_mark(arrived(it, bk.inst), 1);
    InstDev* ins = &inst[bk.inst];
    const InstDev in = *ins;
    if (stopped_before(in.stopped, mark)) return;
    const int j = threadIdx.x / 3, c = threadIdx.x - 3 * j;
    const int n = min(bk.begin + j, bk.end - 1);
    const bool live = bk.begin + j < bk.end;
    const int64_t o = 3 * (int64_t)n + c;
    const VT pc = p[o], qc = q[o], xc = xcg[o], rc = r[o];
    const bool pcg = in.pcg && pinv;
    const double den = TERMS ? node_partials(terms, in, sh) : cg_dot<kNodeThreads>(ppq, in, kDotPQ, ready, sh);
    const bool record = in.nblk_begin == bk.pad && threadIdx.x == 0;
    if (!in.pcg) {
        const bool exempt = it == 1 && in.first_solve;
        const int stop = den == 0.0 ? 3 : fabs(den) <= in.thr && !exempt ? 2 : 0;
        if (stop) {
            if (record) { ins->den = den; ins->stopped = mark; ins->end_reason = stop; ins->last_iters = it; }
            return;
        }
    }
    const double alpha = (it & 1 ? in.rho_slot[1] : in.rho_slot[0]) / den;
    if (record) { ins->den = den; ins->alpha = alpha; }
    const VT a = (VT)alpha, ma = (VT)(-alpha);
    const VT rn = rc + qc * ma;
    if (live) {
        xcg[o] = xc + pc * a;
        r[o] = rn;
    }
    double w = (double)rn;
    if (pcg) {
        pr[threadIdx.x] = (double)rn;
        __syncthreads();
        const VT rv[3] = {(VT)pr[3 * j], (VT)pr[3 * j + 1], (VT)pr[3 * j + 2]};
        VT zn[3];
        precond_apply(in.pcg, pinv + 9 * (int64_t)n, rv, zn);
        const VT zc = c == 0 ? zn[0] : c == 1 ? zn[1] : zn[2];
        if (live) z[o] = zc;
        w = (double)zc;
        __syncthreads();
    }
    pr[threadIdx.x] = live ? (double)rn * w : 0.0;
    node_partial(pr, sh, nd, bk, prr);
}

// ---------------------------------------------------------------------------------------
// integration and bookkeeping
// ---------------------------------------------------------------------------------------
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_euler_update(const Blk* __restrict__ nblk, const InstDev* __restrict__ inst,
                                                          const int8_t* __restrict__ fixed,
                                                          const VT* __restrict__ xcg, VT* __restrict__ v,
                                                          VT* __restrict__ x) {
    const Blk bk = nblk[xcd_item()];
    const int n = bk.begin + threadIdx.x;
    if (n >= bk.end) return;
    // MechanicalObject::vMultiOp fast path (MechanicalObject.inl:2209-2230): v += dv (firstOrder:
    // v = dv), x += v h; then vdamping's v *= exp(-h d) (EulerImplicitSolver.cpp:246-299)
    const InstDev& in = inst[bk.inst];
    const VT h = (VT)in.dt;
    const int64_t o = 3 * (int64_t)n;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const VT vv = in.first_order ? xcg[o + k] : v[o + k] + xcg[o + k];
        x[o + k] = x[o + k] + vv * h;
        v[o + k] = in.vdamp != 1.0 ? vv * (VT)in.vdamp : vv;
    }
    // FixedProjectiveConstraint::projectVelocity (.inl:237-258), when activated
    if (in.project_velocity && (fixed[n] & 1)) {
#pragma unroll
        for (int k = 0; k < 3; k++) v[o + k] = 0;
    }
}

// the end of a solve and, STEP, of its time step (one block per scene).  A loop that ran its whole
// budget is recorded here: PCG's last r.z still gives its err.
template <bool STEP>
__global__ __launch_bounds__(kBlock) void k_finalize(const int* __restrict__ scenes, InstDev* __restrict__ inst,
                                                      const double* __restrict__ prr, int ready) {
    __shared__ double sh[kBlock];
    InstDev* in = &inst[scenes[blockIdx.x]];
    const bool open = !in->stopped, pcg = in->pcg && in->max_iter > 0;
    double rho = 0.0;
    if (open && pcg) rho = cg_dot<kBlock>(prr, *in, kDotRR, ready, sh);
    if (threadIdx.x != 0) return;
    if (open) {
        in->stopped = 1;
        in->last_iters = in->max_iter;
        if (pcg) {
            in->err = in->bnorm2 != 0.0 ? rho / in->bnorm2 : 0.0;
            in->end_reason = 0;
            in->last_iters = in->max_iter + 1;
        }
    }
    in->first_solve = 0;
    in->step_count += 1;
    if (STEP) {
        in->time += in->dt;
        in->lm_x0_set = 1;     // LinearMovementProjectiveConstraint's x0 captured by this step
    }
}

// ---------------------------------------------------------------------------------------
// OscillatorProjectiveConstraint::projectPosition / projectVelocity (OscillatorProjective
// Constraint.inl:77-106) at the context time of the step start: x = mean + a sin(w t + phi),
// v = a w cos(w t + phi)
// ---------------------------------------------------------------------------------------
struct Oscillators {
    const int* __restrict__ node;        // global node id
    const double* __restrict__ mean;     // 3 per entry
    const double* __restrict__ amp;      // 3 per entry
    const double* __restrict__ w;        // pulsation
    const double* __restrict__ phase;
};

template <typename VT>
__global__ __launch_bounds__(kBlock) void k_oscillate(const Blk* __restrict__ oblk, const InstDev* __restrict__ inst,
                                                       Oscillators os, VT* __restrict__ x, VT* __restrict__ v) {
    const Blk bk = oblk[blockIdx.x];
    const int i = bk.begin + threadIdx.x;
    if (i >= bk.end) return;
    const double t = inst[bk.inst].time;
    const double w = os.w[i], ph = os.phase[i];
    const double sn = sin(w * t + ph), cs = cos(w * t + ph);
    const int64_t o = 3 * (int64_t)os.node[i];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        x[o + k] = (VT)(os.mean[3 * i + k] + os.amp[3 * i + k] * sn);
        v[o + k] = (VT)((os.amp[3 * i + k] * w) * cs);
    }
}

// ---------------------------------------------------------------------------------------
// LinearMovementProjectiveConstraint at the context time of the step start
// ---------------------------------------------------------------------------------------
// findKeyTimes (LinearMovementProjectiveConstraint.inl:296-330): true when cT lies in
// [keyTimes[k], keyTimes[k+1]) for some k (the reference's "finished && nextT != prevT"), with the
// bracketing key times and movements
__device__ inline bool lm_window(const InstDev& in, double cT, double& pT, double& nT, double pM[3], double nM[3]) {
    const int nk = in.lm_nk;
    const double* kt = in.lm_keys;
    const double* km = in.lm_keys + nk;
    if (nk == 0 || !(cT >= kt[0] && cT <= kt[nk - 1])) return false;
    nT = kt[0];
    pT = nT;
    for (int k = 0; k < nk; k++) {
        if (kt[k] <= cT) {
            pT = kt[k];
            for (int c = 0; c < 3; c++) pM[c] = km[3 * k + c];
        } else {
            nT = kt[k];
            for (int c = 0; c < 3; c++) nM[c] = km[3 * k + c];
            return nT != pT;
        }
    }
    return false;
}

// the response mask of the constrained nodes for the step starting at the scene's time: the
// movement's bit (4) while a movement is on (projectResponseT, :160-183, clears their responses)
template <bool SCENE>
__global__ __launch_bounds__(kBlock) void k_lm_mask(const Blk* __restrict__ lblk, const InstDev* __restrict__ inst,
                                                     int sid, int8_t* __restrict__ fixed) {
    int si, i;
    if (SCENE) {
        si = sid;
        i = blockIdx.x * kBlock + threadIdx.x;
        if (i >= inst[si].lm_n) return;
    } else {
        const Blk bk = lblk[blockIdx.x];
        si = bk.inst;
        i = bk.begin + threadIdx.x;
        if (i >= bk.end) return;
    }
    const InstDev& in = inst[si];
    double pT = 0, nT = 0, pM[3] = {0, 0, 0}, nM[3] = {0, 0, 0};
    const bool on = lm_window(in, in.time, pT, nT, pM, nM);
    fixed[in.lm_node[i]] = (int8_t)(in.lm_base[i] | (on ? 4 : 0));
}

// projectPosition then projectVelocity (:193-244, in the order of MechanicalProjectPosition-
// AndVelocityVisitor.cpp:35-40): x0 captured on the first projection; inside a movement window
// m = prevM + (nextM - prevM) (cT - prevT) / (nextT - prevT), x = x0 + m (relative) or m,
// v = (nextM - prevM) (1 / (nextT - prevT)).  The scene's time is the step's start; the capture
// flag is set by the step-end kernel.
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_lm_project(const Blk* __restrict__ lblk, InstDev* __restrict__ inst,
                                                        VT* __restrict__ x, VT* __restrict__ v) {
    const Blk bk = lblk[blockIdx.x];
    const int i = bk.begin + threadIdx.x;
    if (i >= bk.end) return;
    const InstDev& in = inst[bk.inst];
    const int64_t o = 3 * (int64_t)in.lm_node[i];
    double* x0 = in.lm_x0 + 3 * (int64_t)i;
    if (!in.lm_x0_set)
        for (int c = 0; c < 3; c++) x0[c] = (double)x[o + c];
    double pT = 0, nT = 0, pM[3] = {0, 0, 0}, nM[3] = {0, 0, 0};
    if (!lm_window(in, in.time, pT, nT, pM, nM)) return;
    const double dt = (in.time - pT) / (nT - pT);
    const double inv = 1.0 / (nT - pT);
    for (int c = 0; c < 3; c++) {
        const double m = pM[c] + (nM[c] - pM[c]) * dt;
        x[o + c] = (VT)(in.lm_relative ? x0[c] + m : m);
        v[o + c] = (VT)((nM[c] - pM[c]) * inv);
    }
}

// the same on one caller vector of one scene at time t (component-level projectPosition /
// projectVelocity); the caller's vector starts at the scene's first node nb0
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_lm_vec(const InstDev* __restrict__ inst, int sid, double t, int nb0,
                                                    VT* __restrict__ vec, int position) {
    const InstDev& in = inst[sid];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= in.lm_n) return;
    const int64_t o = 3 * (int64_t)(in.lm_node[i] - nb0);
    double* x0 = in.lm_x0 + 3 * (int64_t)i;
    if (position && !in.lm_x0_set)
        for (int c = 0; c < 3; c++) x0[c] = (double)vec[o + c];
    double pT = 0, nT = 0, pM[3] = {0, 0, 0}, nM[3] = {0, 0, 0};
    if (!lm_window(in, t, pT, nT, pM, nM)) return;
    const double dt = (t - pT) / (nT - pT);
    const double inv = 1.0 / (nT - pT);
    for (int c = 0; c < 3; c++) {
        const double m = pM[c] + (nM[c] - pM[c]) * dt;
        vec[o + c] = position ? (VT)(in.lm_relative ? x0[c] + m : m) : (VT)((nM[c] - pM[c]) * inv);
    }
}

static __global__ void k_lm_mark_x0(InstDev* __restrict__ inst, int sid) {
    if (threadIdx.x == 0) inst[sid].lm_x0_set = 1;
}

// ---------------------------------------------------------------------------------------
// component-level kernels (one TetrahedronFEMForceField call on caller vectors)
// ---------------------------------------------------------------------------------------
// tet holds flattened node ids; the caller's vectors start at the scene's first node `nb`
template <typename R, int NR, typename VT>
__global__ __launch_bounds__(kBlock) void k_elem_add_force(ElemView<R, NR> ev, int64_t e0, int64_t e1, int nb,
                                                            const VT* __restrict__ x, VT* __restrict__ ef) {
    const int64_t e = e0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= e1) return;
    int4 t = ev.tet[e];
    t.x -= nb; t.y -= nb; t.z -= nb; t.w -= nb;
    R rot[9], c[12], g[12];
    elem_force<R, NR, VT>(ev, e, t, x, rot, c, g);
#pragma unroll
    for (int k = 0; k < 9; k++) ev.rot[k * ev.E + e] = rot[k];
#pragma unroll
    for (int k = 0; k < 12; k++) ef[12 * e + k] = (VT)c[k];
}

template <typename R, int NR, typename VT>
__global__ __launch_bounds__(kBlock) void k_elem_add_dforce(ElemView<R, NR> ev, int64_t e0, int64_t e1, int nb,
                                                             const VT* __restrict__ dx, R fact, VT* __restrict__ ef) {
    const int64_t e = e0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= e1) return;
    const int4 t = ev.tet[e];
    const int nid[4] = {t.x - nb, t.y - nb, t.z - nb, t.w - nb};
    R u[12];
#pragma unroll
    for (int n = 0; n < 4; n++) {
        VT a, b, c;
        load3(dx, nid[n], a, b, c);
        u[3 * n] = (R)a; u[3 * n + 1] = (R)b; u[3 * n + 2] = (R)c;
    }
    R rot[9], c[12];
    load_rot(ev, e, rot);
    elem_dforce<R, NR>(ev, e, rot, u, fact, c);
#pragma unroll
    for (int k = 0; k < 12; k++) ef[12 * e + k] = (VT)c[k];
}

// out[n] (+/-)= sum of the node's contributions; node ids are global, `out` is indexed from
// the scene's first node
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_gather(const int* __restrict__ inc_ptr, const int* __restrict__ inc,
                                                    int n0, int n1, const VT* __restrict__ ef, VT* __restrict__ out,
                                                    int subtract) {
    const int n = n0 + blockIdx.x * kBlock + threadIdx.x;
    if (n >= n1) return;
    const int64_t o = 3 * (int64_t)(n - n0);
    VT a[3] = {out[o], out[o + 1], out[o + 2]};
    const int s0 = inc_ptr[n], s1 = inc_ptr[n + 1];
    if (subtract) gather_contributions<true>(inc, s0, s1, ef, a);
    else gather_contributions<false>(inc, s0, s1, ef, a);
    out[o] = a[0]; out[o + 1] = a[1]; out[o + 2] = a[2];
}

// ---------------------------------------------------------------------------------------
// component-level kernels of the masses, the projective constraints and the state (one call of
// Mass / ProjectiveConstraintSet / MechanicalState on caller vectors of one scene; the caller's
// vectors are indexed from the scene's first node nb0, engine tables by global node id)
// ---------------------------------------------------------------------------------------
// Mass::addMDx: res += factor M dx -- UniformMass.inl:403-419 (m *= factor once, then dx m),
// DiagonalMass.inl:536-559, MeshMatrixMass.inl:1987-2047 (vertex term, then the consistent mass's
// edges in ascending edge id: per node the same order as the reference's two loops)
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_mass_mdx(const InstDev* __restrict__ inst, int sid, NodeArrays na, int nb0,
                                                      int n, const VT* __restrict__ dx, VT* __restrict__ res,
                                                      double factor) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const InstDev& in = inst[sid];
    VT d[3], o[3];
    load3(dx, i, d[0], d[1], d[2]);
    load3(res, i, o[0], o[1], o[2]);
    mass_mdx(in, na, nb0 + i, factor, d, o);
    if (in.mass_kind == kMassMatrix)
        mass_edges<3>(na, nb0 + i, factor, [&](int j, VT e[3]) { load3(dx, j - nb0, e[0], e[1], e[2]); }, o);
    const int64_t q = 3 * (int64_t)i;
    res[q] = o[0]; res[q + 1] = o[1]; res[q + 2] = o[2];
}

// Mass::accFromF: a = M^-1 f -- UniformMass.inl:423-436 (f / m), DiagonalMass.inl:564-576
// (f / m_i), MeshMatrixMass.inl:2051-2069 (lumped only: f / (m_i 2.5))
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_mass_acc(const InstDev* __restrict__ inst, int sid,
                                                      const double* __restrict__ mass, int nb0, int n,
                                                      const VT* __restrict__ f, VT* __restrict__ a) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const InstDev& in = inst[sid];
    VT m;
    if (in.mass_kind == kMassUniform) m = (VT)in.vertex_mass;
    else if (in.mass_kind == kMassDiagonal) m = (VT)mass[nb0 + i];
    else m = (VT)mass[nb0 + i] * (VT)kLumpTet;
    const int64_t q = 3 * (int64_t)i;
#pragma unroll
    for (int k = 0; k < 3; k++) a[q + k] = f[q + k] / m;
}

// Mass::addForce (gravity): UniformMass.inl:471-496 (f += g m), DiagonalMass.inl:1393-1413
// (f += g m_i), MeshMatrixMass.inl:2073-2092 (f += g m_i 2.5, lumped coefficient in both modes)
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_mass_add_force(const InstDev* __restrict__ inst, int sid,
                                                            const double* __restrict__ mass, int nb0, int n,
                                                            VT* __restrict__ f) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const InstDev& in = inst[sid];
    const int64_t q = 3 * (int64_t)i;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        VT w;
        if (in.mass_kind == kMassUniform) w = (VT)in.mg[k];
        else if (in.mass_kind == kMassDiagonal) w = (VT)in.gravity[k] * (VT)mass[nb0 + i];
        else w = ((VT)in.gravity[k] * (VT)mass[nb0 + i]) * (VT)kLumpTet;
        f[q + k] += w;
    }
}

// ProjectiveConstraintSet::projectResponse of the scene's constraints: FixedProjectiveConstraint
// (FixedProjectiveConstraint.inl:184-207; fixAll clears every node) and
// OscillatorProjectiveConstraint (OscillatorProjectiveConstraint.inl:65-70) clear their nodes.
// velocity = 1: FixedProjectiveConstraint::projectVelocity (.inl:237-258): the fixed nodes only,
// and only when activate_projectVelocity is set
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_project(const InstDev* __restrict__ inst, int sid,
                                                     const int8_t* __restrict__ fixed, int nb0, int n,
                                                     VT* __restrict__ vec, int velocity) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int8_t m = fixed[nb0 + i];
    const bool clear = velocity ? (inst[sid].project_velocity && (m & 1)) : m != 0;
    if (!clear) return;
    const int64_t q = 3 * (int64_t)i;
    vec[q] = 0; vec[q + 1] = 0; vec[q + 2] = 0;
}

// OscillatorProjectiveConstraint::projectPosition / projectVelocity (.inl:72-106) at time t on a
// caller vector: x = mean + a sin(w t + phi) (position = 1) or v = a w cos(w t + phi)
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_oscillate_vec(Oscillators os, int o0, int o1, int nb0, double t,
                                                           VT* __restrict__ vec, int position) {
    const int i = o0 + blockIdx.x * kBlock + threadIdx.x;
    if (i >= o1) return;
    const double w = os.w[i], ph = os.phase[i];
    const int64_t q = 3 * (int64_t)(os.node[i] - nb0);
    if (position) {
        const double sn = sin(w * t + ph);
#pragma unroll
        for (int k = 0; k < 3; k++) vec[q + k] = (VT)(os.mean[3 * i + k] + os.amp[3 * i + k] * sn);
    } else {
        const double cs = cos(w * t + ph);
#pragma unroll
        for (int k = 0; k < 3; k++) vec[q + k] = (VT)((os.amp[3 * i + k] * w) * cs);
    }
}

// BaseMechanicalState::vDot on caller vectors (MechanicalObject::vDot, MechanicalObject.inl
// :2334-2356) in the FP64 engine's parallel blocked order: per 256-node block the
// fixed tree of block_sum, then the block partials added by one block as last_block_reduce
// does (each thread a strided sum, then block_sum) -- the oracle's dot_blocked
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_vdot_blocks(const VT* __restrict__ a, const VT* __restrict__ b, int n,
                                                         double* __restrict__ partial) {
    __shared__ double sh[kBlock];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double t = 0.0;
    if (i < n) {
        VT x[3], y[3];
        load3(a, i, x[0], x[1], x[2]);
        load3(b, i, y[0], y[1], y[2]);
        t = dot3d(x, y);
    }
    const double bs = block_sum(t, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = bs;
}
static __global__ __launch_bounds__(kBlock) void k_vdot_final(const double* __restrict__ partial, int nb,
                                                               double* __restrict__ out) {
    __shared__ double sh[kBlock];
    double acc = 0.0;
    for (int k = threadIdx.x; k < nb; k += kBlock) acc = acc + partial[k];
    const double total = block_sum(acc, sh);
    if (threadIdx.x == 0) *out = total;
}

// ---------------------------------------------------------------------------------------
// von Mises stress (TetrahedronFEMForceField::computeVonMisesStress, .inl:2197-2347)
// ---------------------------------------------------------------------------------------
// Per element, from the scene's current positions x, in double whatever the engine's precision
// (a post-process read once per step at most): the displacement gradient
// gradU(k,l) = sum_m shf(l+1,m) u_m[k] with shf the inverse of the rest matrix [1 x y z] per
// vertex and u_m either the corotational displacement of vertex m in the element frame
// (mode 1; rest minus current, as the reference's D) or x - x0 (mode 2); the strain
// (gradU + gradU^T)/2 (mode 1) or (gradU + gradU^T + gradU^T gradU)/2 (mode 2); the stress
// s = 2 mu strain + lambda tr(strain) I in Voigt order (xx, yy, zz, yz, xz, xy); von Mises
// sqrt(s0^2 + s1^2 + s2^2 - s0 s1 - s1 s2 - s2 s0 + 3 (s3^2 + s4^2 + s5^2)), values below 1e-10
// set to 0.  Mode 1 also stores the element rotation of x, as the reference does.  Every
// operation in the reference's order, no contraction where the translation unit honours the
// pragma (the FP64 engines': they match the reference bit for bit).
// shf: 12 values per element (rows 1..3 of the inverse, row-major), lm: lambda, mu per element,
// both in the engine's element order of the scene; vme in that order.  x and x0 are the scene's
// (node ids of the element record minus nb index them).
template <typename R, int NR, typename VT>
__global__ __launch_bounds__(kBlock) void k_von_mises_elem(ElemView<R, NR> ev, int64_t e0, int64_t e1, int nb,
                                                           const VT* __restrict__ x,
                                                           const double* __restrict__ x0,
                                                           const double* __restrict__ shf,
                                                           const double* __restrict__ lm, int mode,
                                                           double* __restrict__ vme) {
#pragma clang fp contract(off)
    const int64_t e = e0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= e1) return;
    const int64_t le = e - e0;
    const int4 t = ev.tet[e];
    const int nid[4] = {t.x - nb, t.y - nb, t.z - nb, t.w - nb};
    double p[4][3];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        VT a, b, c;
        load3(x, nid[m], a, b, c);
        p[m][0] = (double)a; p[m][1] = (double)b; p[m][2] = (double)c;
    }
    double D[12];
    if (mode == 2) {
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int k = 0; k < 3; k++) D[3 * m + k] = p[m][k] - x0[3 * (int64_t)nid[m] + k];
    } else {
        R gr[12], rcr[9];
        jgroups<R, NR>(ev, e, gr, rcr);
        double rc[9];
#pragma unroll
        for (int k = 0; k < 9; k++) rc[k] = (double)rcr[k];
        double rot[9];
        rotation_large<double>(p[0], p[1], p[2], rot);
#pragma unroll
        for (int k = 0; k < 9; k++) ev.rot[k * ev.E + e] = (R)rot[k];
        // deforme[k] = R_0_2 p_k, R_0_2 = transpose(rot); then relative to deforme[0]
        double df[4][3];
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                double v = rot[i] * p[k][0];
                v = v + rot[3 + i] * p[k][1];
                df[k][i] = v + rot[6 + i] * p[k][2];
            }
        df[1][0] -= df[0][0];
        df[2][0] -= df[0][0];
        df[2][1] -= df[0][1];
#pragma unroll
        for (int i = 0; i < 3; i++) df[3][i] -= df[0][i];
        D[0] = 0; D[1] = 0; D[2] = 0;
        D[3] = rc[0] - df[1][0]; D[4] = 0; D[5] = 0;
        D[6] = rc[3] - df[2][0]; D[7] = rc[4] - df[2][1]; D[8] = 0;
        D[9] = rc[6] - df[3][0]; D[10] = rc[7] - df[3][1]; D[11] = rc[8] - df[3][2];
    }
    const double* sf = shf + 12 * le;
    double gu[3][3];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int l = 0; l < 3; l++) {
            double a = 0.0;
#pragma unroll
            for (int m = 0; m < 4; m++) a += sf[4 * l + m] * D[3 * m + k];
            gu[k][l] = a;
        }
    double st[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            double a = gu[i][j] + gu[j][i];
            if (mode == 2) {
                // (gradU^T gradU)(i,j), the 3x3 product's three-term order
                double g = gu[0][i] * gu[0][j] + gu[1][i] * gu[1][j];
                g = g + gu[2][i] * gu[2][j];
                a = a + g;
            }
            st[i][j] = a * 0.5;
        }
    const double vs[6] = {st[0][0], st[1][1], st[2][2], st[1][2], st[0][2], st[0][1]};
    const double lambda = lm[2 * le], mu = lm[2 * le + 1];
    double s[6], tr = 0.0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        tr += vs[k];
        s[k] = vs[k] * 2 * mu;
    }
#pragma unroll
    for (int k = 3; k < 6; k++) s[k] = vs[k] * 2 * mu;
#pragma unroll
    for (int k = 0; k < 3; k++) s[k] += lambda * tr;
    double q = s[0] * s[0] + s[1] * s[1];
    q = q + s[2] * s[2];
    q = q - s[0] * s[1];
    q = q - s[1] * s[2];
    q = q - s[2] * s[0];
    q = q + 3 * s[3] * s[3];
    q = q + 3 * s[4] * s[4];
    q = q + 3 * s[5] * s[5];
    double v = sqrt(q);
    if (v < 1e-10) v = 0.0;
    vme[le] = v;
}

// vonMisesPerNode: the mean of the element values around each node, summed over its incidence
// list (ascending element id, getTetrahedraAroundVertex's order); 0 for a node of no element
static __global__ __launch_bounds__(kBlock) void k_von_mises_node(const int* __restrict__ inc_ptr, const int* __restrict__ inc,
                                                           int n0, int n1, int64_t e0,
                                                           const double* __restrict__ vme,
                                                           double* __restrict__ vmn) {
#pragma clang fp contract(off)
    const int n = n0 + blockIdx.x * kBlock + threadIdx.x;
    if (n >= n1) return;
    const int s0 = inc_ptr[n], s1 = inc_ptr[n + 1];
    double a = 0.0;
    for (int s = s0; s < s1; s++) a += vme[(int64_t)(inc[s] >> 2) - e0];
    if (s1 > s0) a /= (double)(s1 - s0);
    vmn[n - n0] = a;
}

// ---------------------------------------------------------------------------------------
// assembled stiffness (TetrahedronFEMForceField::addKToMatrix / buildStiffnessMatrix,
// .inl:1921-1999, with computeStiffnessMatrix, :212-232)
// ---------------------------------------------------------------------------------------
// the three strain-displacement groups of vertex v, by selects (an index known at run time would put
// the twelve in scratch memory)
template <typename R>
__device__ __forceinline__ void vertex_groups(const R g[12], int v, double& a, double& b, double& c) {
    const R g0 = g[0], g1 = g[1], g2 = g[2], g3 = g[3], g4 = g[4], g5 = g[5];
    const R g6 = g[6], g7 = g[7], g8 = g[8], g9 = g[9], g10 = g[10], g11 = g[11];
    const bool low = v < 2, odd = v & 1;
    const R la = odd ? R(g3) : R(g0), lb = odd ? R(g4) : R(g1), lc = odd ? R(g5) : R(g2);
    const R ha = odd ? R(g9) : R(g6), hb = odd ? R(g10) : R(g7), hc = odd ? R(g11) : R(g8);
    a = (double)(low ? R(la) : R(ha));
    b = (double)(low ? R(lb) : R(hb));
    c = (double)(low ? R(lc) : R(hc));
}

// block (n1, n2) of R J K J^T R^T of element e (computeStiffnessMatrix, TetrahedronFEMForceField
// .inl:212-232, with the last addForce's rotation): J's rows of n1 and n2 only, with R =
// rotations[e], JK = J(n1 rows) K, B = JK J(n2 rows)^T, S = R B, block = S R^T, every sum in the
// reference's dense-product order (zero terms of its 12x12 products leave its sums unchanged)
template <typename R, int NR>
__device__ __forceinline__ void elem_stiffness_block(const ElemView<R, NR>& ev, int64_t e, int n1, int n2, double blk[9]) {
#pragma clang fp contract(off)
    R gr[12], rcr[9];
    jgroups<R, NR>(ev, e, gr, rcr);
    double rot[9];
#pragma unroll
    for (int k = 0; k < 9; k++) rot[k] = (double)ev.rot[k * ev.E + e];
    const double k00 = (double)ev.kmat[e], k01 = (double)ev.kmat[ev.E + e], k33 = (double)ev.kmat[2 * ev.E + e];
    double Km[6][6];
#pragma unroll
    for (int l = 0; l < 6; l++)
#pragma unroll
        for (int m = 0; m < 6; m++)
            Km[l][m] = (l < 3 && m < 3) ? (l == m ? k00 : k01) : ((l == m) ? k33 : 0.0);
    // J rows of a vertex (computeStrainDisplacement's placement of its three groups)
    double J1[3][6], J2[3][6];
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
        for (int l = 0; l < 6; l++) { J1[q][l] = 0.0; J2[q][l] = 0.0; }
    {
        double a0, a1, a2, b0, b1, b2;
        vertex_groups<R>(gr, n1, a0, a1, a2);
        vertex_groups<R>(gr, n2, b0, b1, b2);
        J1[0][0] = a0; J1[0][3] = a1; J1[0][5] = a2;
        J1[1][3] = a0; J1[1][1] = a1; J1[1][4] = a2;
        J1[2][5] = a0; J1[2][4] = a1; J1[2][2] = a2;
        J2[0][0] = b0; J2[0][3] = b1; J2[0][5] = b2;
        J2[1][3] = b0; J2[1][1] = b1; J2[1][4] = b2;
        J2[2][5] = b0; J2[2][4] = b1; J2[2][2] = b2;
    }
    double JK[3][6];
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
        for (int m = 0; m < 6; m++) {
            double a = 0.0;
#pragma unroll
            for (int l = 0; l < 6; l++) a += J1[q][l] * Km[l][m];
            JK[q][m] = a;
        }
    double B[3][3];
#pragma unroll
    for (int q1 = 0; q1 < 3; q1++)
#pragma unroll
        for (int q2 = 0; q2 < 3; q2++) {
            double a = 0.0;
#pragma unroll
            for (int m = 0; m < 6; m++) a += JK[q1][m] * J2[q2][m];
            B[q1][q2] = a;
        }
    double S[3][3];
#pragma unroll
    for (int q1 = 0; q1 < 3; q1++)
#pragma unroll
        for (int p = 0; p < 3; p++) {
            double a = 0.0;
#pragma unroll
            for (int r = 0; r < 3; r++) a += rot[3 * q1 + r] * B[r][p];
            S[q1][p] = a;
        }
#pragma unroll
    for (int q1 = 0; q1 < 3; q1++)
#pragma unroll
        for (int q2 = 0; q2 < 3; q2++) {
            double a = 0.0;
#pragma unroll
            for (int p = 0; p < 3; p++) a += S[q1][p] * rot[3 * q2 + p];
            blk[3 * q1 + q2] = a;
        }
}

// The assembled matrix in two passes.  (1) One thread per element and vertex pair (n1, n2): the
// element block -(R J K J^T R^T)(n1, n2) -- J's rows of n1 and n2 only: with R = rotations[e]
// (the last addForce's), JK = J(n1 rows) K, B = JK J(n2 rows)^T, S = R B, block = S R^T, every
// sum in the reference's dense-product order (zero terms of the reference's 12x12 products leave
// its sums unchanged) -- into the scene's element-block buffer at (element - e0) * 16 + n1 * 4 +
// n2.  (2) One thread per 3x3 block (a, b): the sum, in ascending element id (the element loop's
// order), of block * k over the contributions slots[] lists for it (device element * 16 + n1 * 4
// + n2).  Each element record is read once (not once per block it touches), and both passes
// store through LDS so that a wave's stores are contiguous.  Computed in double, no contraction
// where the translation unit honours the pragma.
template <typename R, int NR>
__global__ __launch_bounds__(kBlock) void k_stiffness_elem(ElemView<R, NR> ev, int64_t e0, int64_t n16,
                                                            double* __restrict__ eblk) {
#pragma clang fp contract(off)
    __shared__ double st[9 * kBlock];
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n16) {
        double blk[9];
        const int j = (int)(i & 15);
        elem_stiffness_block<R, NR>(ev, e0 + (i >> 4), j >> 2, j & 3, blk);
#pragma unroll
        for (int k = 0; k < 9; k++) st[9 * threadIdx.x + k] = blk[k];
    }
    __syncthreads();
    const int64_t o = 9 * (int64_t)blockIdx.x * kBlock, end = 9 * n16;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        const int64_t w = o + k * kBlock + threadIdx.x;
        if (w < end) eblk[w] = st[k * kBlock + threadIdx.x];
    }
}

template <typename R, int NR>
__global__ __launch_bounds__(kBlock) void k_stiffness_blocks(const int* __restrict__ slot_ptr, const int* __restrict__ slots,
                                                             int nblk, int64_t slot0, double kf,
                                                             const double* __restrict__ eblk, double* __restrict__ out) {
#pragma clang fp contract(off)
    __shared__ double st[9 * kBlock];
    const int b = blockIdx.x * kBlock + threadIdx.x;
    if (b < nblk) {
        double acc[9];
#pragma unroll
        for (int i = 0; i < 9; i++) acc[i] = 0.0;
        for (int s = slot_ptr[b]; s < slot_ptr[b + 1]; s++) {
            const double* blk = eblk + 9 * ((int64_t)slots[s] - slot0);
#pragma unroll
            for (int i = 0; i < 9; i++) acc[i] += (-blk[i]) * kf;
        }
#pragma unroll
        for (int i = 0; i < 9; i++) st[9 * threadIdx.x + i] = acc[i];
    }
    __syncthreads();
    const int64_t o = 9 * (int64_t)blockIdx.x * kBlock, end = 9 * (int64_t)nblk;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        const int64_t w = o + k * kBlock + threadIdx.x;
        if (w < end) out[w] = st[k * kBlock + threadIdx.x];
    }
}

// ---------------------------------------------------------------------------------------
// PCGLinearSolver with a Jacobi / block-Jacobi preconditioner (PCGLinearSolver.inl:178-262,
// JacobiPreconditioner.inl:43-52, BlockJacobiPreconditioner.inl:41-52)
// ---------------------------------------------------------------------------------------
// node n's preconditioner block, inverted: mF (vertex mass) I, then kF (-R J K J^T R^T)(v, v) of
// its elements in ascending element id (MatrixLinearSystem's assembly: mass, then the FEM's
// element loop, each value scaled by its factor); the identity for a fixed node (Dirichlet row,
// MatrixLinearSystem.inl:1177-1189); then DiagonalMatrix::invert (1 / d, off-diagonal dropped) or
// Mat<3,3>::invert (invertMatrix, Mat.h:1172-1192, with the determinant of Mat.h:989-997)
// Four lanes a node (an aligned quad, all with the same n): each forms the block of every fourth
// incidence, and all of them add the quad's blocks in list order, so all have the result.  Measured with the
// groups picked by selects: 45,000 nodes 268 -> 66 us, 12,000 61 -> 16.
template <typename R, int NR>
__device__ __forceinline__ void pcg_block(const InstDev& in, const ElemView<R, NR>& ev, const int* __restrict__ inc_ptr,
                                 const int* __restrict__ inc, const double* __restrict__ mass,
                                 const int8_t* __restrict__ fixed, int n, double* __restrict__ out) {
#pragma clang fp contract(off)
    double B[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (fixed[n] & 1) {
        B[0] = B[4] = B[8] = 1.0;
    } else {
        double m = in.mass_kind == kMassUniform ? in.vertex_mass : mass[n];
        if (in.mass_kind == kMassMatrixLumped) m = m * kLumpTet;
        const double mm = m * in.m_cg;
        B[0] += mm; B[4] += mm; B[8] += mm;
        const int s0 = inc_ptr[n], s1 = inc_ptr[n + 1];
        for (int s = s0; s < s1; s += 4) {
            const int slot = inc[min(s + (int)(threadIdx.x & 3), s1 - 1)];
            double blk[9];
            elem_stiffness_block<R, NR>(ev, slot >> 2, slot & 3, slot & 3, blk);
#pragma unroll
            for (int i = 0; i < 9; i++) blk[i] = (-blk[i]) * in.k_cg;
#pragma unroll
            for (int i = 0; i < 9; i++) {
                B[i] += quad_lane<0>(blk[i]);
                if (s + 1 < s1) B[i] += quad_lane<1>(blk[i]);
                if (s + 2 < s1) B[i] += quad_lane<2>(blk[i]);
                if (s + 3 < s1) B[i] += quad_lane<3>(blk[i]);
            }
        }
    }
    if (in.pcg == 1) {
#pragma unroll
        for (int i = 0; i < 9; i++) out[i] = (i % 4 == 0) ? 1.0 / B[i] : 0.0;
        return;
    }
    auto F = [&](int r, int c) { return B[3 * r + c]; };
    const double det = F(0, 0) * F(1, 1) * F(2, 2) + F(1, 0) * F(2, 1) * F(0, 2) + F(2, 0) * F(0, 1) * F(1, 2)
                       - F(0, 0) * F(2, 1) * F(1, 2) - F(1, 0) * F(0, 1) * F(2, 2) - F(2, 0) * F(1, 1) * F(0, 2);
    out[0] = (F(1, 1) * F(2, 2) - F(2, 1) * F(1, 2)) / det;
    out[3] = (F(1, 2) * F(2, 0) - F(2, 2) * F(1, 0)) / det;
    out[6] = (F(1, 0) * F(2, 1) - F(2, 0) * F(1, 1)) / det;
    out[1] = (F(2, 1) * F(0, 2) - F(0, 1) * F(2, 2)) / det;
    out[4] = (F(2, 2) * F(0, 0) - F(0, 2) * F(2, 0)) / det;
    out[7] = (F(2, 0) * F(0, 1) - F(0, 0) * F(2, 1)) / det;
    out[2] = (F(0, 1) * F(1, 2) - F(1, 1) * F(0, 2)) / det;
    out[5] = (F(0, 2) * F(1, 0) - F(1, 2) * F(0, 0)) / det;
    out[8] = (F(0, 0) * F(1, 1) - F(1, 0) * F(0, 1)) / det;
}

// the node of this quad: blockIdx.y takes the 64-node parts of a node block
constexpr int kQuadNodes = kBlock / 4;
__device__ __forceinline__ int quad_node(int begin) {
    return begin + (int)blockIdx.y * kQuadNodes + ((int)threadIdx.x >> 2);
}

// every node of the PCG scenes of the launch set: its inverted preconditioner block (the
// rotations of this step's addForce)
template <typename R, int NR, typename BLK>
__global__ __launch_bounds__(kBlock) void k_pcg_diag(ElemView<R, NR> ev, const BLK* __restrict__ nblk,
                                                      const InstDev* __restrict__ inst, const int* __restrict__ inc_ptr,
                                                      const int* __restrict__ inc, const double* __restrict__ mass,
                                                      const int8_t* __restrict__ fixed, double* __restrict__ pinv) {
    const BLK bk = nblk[xcd_item()];
    const InstDev in = inst[blk_scene(bk)];
    if (!in.pcg) return;
    const int n = quad_node(bk.begin);
    if (n >= bk.end) return;
    double B[9];
    pcg_block<R, NR>(in, ev, inc_ptr, inc, mass, fixed, n, B);
    if ((threadIdx.x & 3) == 0) {
#pragma unroll
        for (int i = 0; i < 9; i++) pinv[9 * (int64_t)n + i] = B[i];
    }
}

// LinearMovementProjectiveConstraint's indices are Dirichlet rows of the assembled matrix
// (applyConstraint(ZeroDirichletCondition*)) whatever the time: the identity block
static __global__ __launch_bounds__(kBlock) void k_pcg_lm_identity(const Blk* __restrict__ lblk,
                                                                    const InstDev* __restrict__ inst,
                                                                    double* __restrict__ pinv) {
    const Blk bk = lblk[blockIdx.x];
    const int i = bk.begin + threadIdx.x;
    const InstDev& in = inst[bk.inst];
    if (i >= bk.end || !in.pcg) return;
    double* P = pinv + 9 * (int64_t)in.lm_node[i];
#pragma unroll
    for (int k = 0; k < 9; k++) P[k] = (k % 4 == 0) ? 1.0 : 0.0;
}

// the PCG scenes of the launch set start a solve: iteration 1, from the solution vector
static __global__ void k_pcg_open(const int* __restrict__ scenes, int n, InstDev* __restrict__ inst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    InstDev* in = &inst[scenes[i]];
    if (!in->pcg) return;
    in->stopped = 0;
    in->iter = 1;
    in->end_reason = 0;
    in->pcg_tol = in->tol * in->bnorm2;      // tol = tolerance b.b
}

// r = M x (the operator on the solution vector, element contributions from k_cg_elem at
// iteration 1 reading x), r = -r + b (cgstep_beta(r, b, -1): r *= -1; r += b), w = P^-1 r,
// r_norm = r.w, the loop's first test (PCGLinearSolver.inl:193-215); w goes to z, from which
// iteration 1's direction is taken
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_pcg_begin(const Blk* __restrict__ nblk, InstDev* __restrict__ inst,
                                                       NodeArrays na, const VT* __restrict__ ef,
                                                       const VT* __restrict__ xcg, const VT* __restrict__ b,
                                                       VT* __restrict__ r, VT* __restrict__ z,
                                                       const double* __restrict__ pinv, double* __restrict__ partial,
                                                       double* __restrict__ nd) {
    __shared__ double sh[kBlock];
    const Blk bk = nblk[xcd_item()];
    InstDev* ins = &inst[bk.inst];
    if (!ins->pcg || ins->stopped) return;
    const int n = bk.begin + threadIdx.x;
    double rz = 0.0;
    if (n < bk.end) {
        const InstDev& in = *ins;
        const int64_t o = 3 * (int64_t)n;
        VT xn[3];
        load3(xcg, n, xn[0], xn[1], xn[2]);
        VT qn[3] = {0, 0, 0};
        if (in.m_cg != 0.0) {
            mass_mdx(in, na, n, in.m_cg, xn, qn);
            if (in.mass_kind == kMassMatrix)
                mass_edges<3>(na, n, in.m_cg, [&](int j, VT d[3]) { load3(xcg, j, d[0], d[1], d[2]); }, qn);
        }
        const int s0 = na.inc_ptr[n], s1 = na.inc_ptr[n + 1];
        gather_contributions<true>(na.inc, s0, s1, ef, qn);
        if (in.plane_on && na.contact[n]) plane_dforce(in, in.k_cg, xn, qn);
        if (na.fixed[n]) { qn[0] = 0; qn[1] = 0; qn[2] = 0; }
        VT rn[3], zn[3];
#pragma unroll
        for (int k = 0; k < 3; k++) { VT t = qn[k]; t *= (VT)-1.0; t += b[o + k]; rn[k] = t; r[o + k] = t; }
        precond_apply(in.pcg, pinv + 9 * (int64_t)n, rn, zn);
        z[o] = zn[0]; z[o + 1] = zn[1]; z[o + 2] = zn[2];
        rz = dot3d(rn, zn);
        if (nd) nd[n] = rz;
    }
    double rho;
    const bool last = nd ? last_block_sequential(nd, ins, rho)
                         : last_block_reduce(block_sum(rz, sh), partial, ins, bk.pad, sh, rho);
    if (last && threadIdx.x == 0) {
        ins->rho_slot[1] = rho;
        ins->err = ins->bnorm2 != 0.0 ? rho / ins->bnorm2 : 0.0;
        if (ins->max_iter < 1 || !(rho > ins->pcg_tol)) {
            ins->stopped = 1; ins->end_reason = 1; ins->last_iters = 1;
        }
    }
}

// the warm-start scenes of the launch set open their solve: iteration 1, so that k_cg_elem
// evaluates the element part of A x from the solution vector
static __global__ void k_warm_open(const int* __restrict__ scenes, int n, InstDev* __restrict__ inst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    InstDev* in = &inst[scenes[i]];
    if (!in->warm_start || in->pcg) return;
    in->stopped = 0;
    in->iter = 1;
    in->end_reason = 0;
}

// CGLinearSolver warmStart: r = A x (mass, the element contributions of k_cg_elem on x, plane,
// projection) then r.eq(b, r, -1.0): r = b + r (-1); rho = r.r and the first tests
template <typename VT>
__global__ __launch_bounds__(kBlock) void k_cg_warm_begin(const Blk* __restrict__ nblk, InstDev* __restrict__ inst,
                                                           NodeArrays na, const VT* __restrict__ ef,
                                                           const VT* __restrict__ xcg, const VT* __restrict__ b,
                                                           VT* __restrict__ r, double* __restrict__ partial,
                                                           double* __restrict__ nd) {
    __shared__ double sh[kBlock];
    const Blk bk = nblk[xcd_item()];
    InstDev* ins = &inst[bk.inst];
    if (!ins->warm_start || ins->pcg || ins->stopped) return;
    const int n = bk.begin + threadIdx.x;
    double rr = 0.0;
    if (n < bk.end) {
        const InstDev& in = *ins;
        const int64_t o = 3 * (int64_t)n;
        VT xn[3];
        load3(xcg, n, xn[0], xn[1], xn[2]);
        VT qn[3] = {0, 0, 0};
        if (in.m_cg != 0.0) {
            mass_mdx(in, na, n, in.m_cg, xn, qn);
            if (in.mass_kind == kMassMatrix)
                mass_edges<3>(na, n, in.m_cg, [&](int j, VT d[3]) { load3(xcg, j, d[0], d[1], d[2]); }, qn);
        }
        const int s0 = na.inc_ptr[n], s1 = na.inc_ptr[n + 1];
        gather_contributions<true>(na.inc, s0, s1, ef, qn);
        if (in.plane_on && na.contact[n]) plane_dforce(in, in.k_cg, xn, qn);
        if (na.fixed[n]) { qn[0] = 0; qn[1] = 0; qn[2] = 0; }
        VT rn[3];
#pragma unroll
        for (int k = 0; k < 3; k++) { VT t = qn[k] * (VT)-1.0; rn[k] = b[o + k] + t; r[o + k] = rn[k]; }
        rr = dot3d(rn, rn);
        if (nd) nd[n] = rr;
    }
    double total;
    const bool last = nd ? last_block_sequential(nd, ins, total)
                         : last_block_reduce(block_sum(rr, sh), partial, ins, bk.pad, sh, total);
    if (last && threadIdx.x == 0) cg_start_warm(ins, ins->bnorm2, total);
}

}  // namespace sofa_amd
