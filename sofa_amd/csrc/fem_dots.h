// fem_dots.h -- node-after-node sums (MechanicalObject::vDot's order, MechanicalObject.inl
// :2334-2356) without the chain of dependent adds, bit for bit.
//
// s_{i+1} = fl(s_i + t_i) rounds to the grid of s_{i+1}'s binade.  While the running sum stays
// strictly inside one binade (2^e, 2^{e+1}) (or its mirror image below zero) that grid is the
// multiples of u = 2^{e-52}, s_i is on it, and fl(s_i + t_i) = s_i + m_i with m_i = t_i rounded to
// the nearest multiple of u -- unless t_i lies exactly half way between two multiples, where the
// choice depends on s_i.  The m_i are multiples of u and sums of them below 2^53 u are exact in any
// order, so a run of terms adds up in parallel: with M = sum m_i and A = sum |m_i| every partial
// sum lies between s + (M - A) / 2 and s + (M + A) / 2, and when those two are strictly inside the
// binade and no term is a tie, the run's last sum is s + M, the chain's bits.
//
// One workgroup per sum, a pipeline of rounds of kScanRound terms with one barrier each.  Four waves
// load and stage the terms, give every piece of 64 terms (four lanes) an approximate start by plain
// sums, so a binade to round to, and form its M and A.  A fifth wave walks the previous round's 64
// pieces from the exact sum so far, all at once by a prefix scan up to the first whose condition
// fails (another binade than guessed, a crossing, a tie, a term of the sum's own size), which it
// takes by dependent adds, with the ones right behind it that look as if they failed too (a piece that
// would keep the rule has the same sum either way).  The binades of a growing sum are crossed about log2(n)
// times, mostly within the first pieces; about 18 pieces of a sum fail (emulated on beams of 2,500 to 41,000
// nodes, both dot products of CG).  Of a sum whose terms change sign most pieces fail: it is the chain.
//
// What bounds it: one CU's latency.  A round takes 2,200 cycles (0.9 us: 470 to issue its loads, 280 to
// stage them, 970 + 490 of arithmetic at one wave per SIMD; the walk, 1,050, runs beside it), the chain
// 3.7 ns a term.  Its three rounds of 4,096 terms fill 113 KB of LDS: no tile of the operator fits beside it
// (68 KB in double), so with branches it waits for a CU that another branch's operator leaves free.
// Measured, calls of vDot in a row, n = 512, 1,000, 4,096, 8,100, 21,825, 56,889 nodes: squares 6.7, 7.1, 7.9, 11.0, 18.6, 35.5
// us (the chain alone 6.7, 7.7, 27.7, 54, 146, 371); products of either sign 6.7, 8.7, 19.9, 38, 96, 168, with the failing
// pieces one by one 8.0, 11.5, 31.9, 62, 158, 238 (the chain alone as above).  In the step of 16 beams of 500 to
// 42,000 nodes a dot product went from 45.6 us (the chain in 8 segments run at once from candidate
// starts, four launches) to 16-23 in one, the step from 5.2 to 3.6 ms.
#pragma once

#include "fem_tiled.h"

namespace sofa_amd {

constexpr int kScanWaves = 4;                    // ... that form the pieces; one more walks them
constexpr int kScanThreads = 64 * (kScanWaves + 1);
constexpr int kScanPer = 16;                     // terms per lane and round
constexpr int kScanLanes = 64 / kScanPer;        // lanes per piece
constexpr int kScanRound = 64 * kScanWaves * kScanPer;
constexpr int kScanResult = 64 * kScanWaves;     // the thread that has the sum
// a term's place in LDS: two doubles of padding behind each lane's own, so that the lanes' reads
// of their own terms spread over the banks
__device__ __forceinline__ constexpr int scan_at(int i) { return i + 2 * (i / kScanPer); }

static_assert(kScanWaves == 4 && kScanLanes == 4 && kScanRound == 64 * 64, "quads of lanes, 64 pieces a round");

// inclusive prefix sums over the lanes (wave_sum's steps)
__device__ __forceinline__ double wave_prefix(double v) {
    v = v + dpp_from<0x111, 0xf>(v);
    v = v + dpp_from<0x112, 0xf>(v);
    v = v + dpp_from<0x114, 0xf>(v);
    v = v + dpp_from<0x118, 0xf>(v);
    v = v + dpp_from<0x142, 0xa>(v);
    return v + dpp_from<0x143, 0xc>(v);
}
// over each aligned 4 lanes: their last lane holds the sum
__device__ __forceinline__ double quad_sum(double v) {
    v = v + dpp_from<0x111, 0xf>(v);
    return v + dpp_from<0x112, 0xf>(v);
}
__device__ __forceinline__ double lane_value(double v, int lane) {   // `lane` uniform
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// sign and exponent of a double whose binade the scan can use (the grid, its half and the next
// binade are normal numbers), else 0
__device__ __forceinline__ int scan_key(double s) {
    const int k = (int)((unsigned long long)__double_as_longlong(s) >> 52);
    const int eb = k & 0x7ff;
    return eb > 64 && eb < 2046 ? k : 0;
}
__device__ __forceinline__ double scan_low(int key) {   // 2^e
    return __longlong_as_double((long long)(key & 0x7ff) << 52);
}
// the lane's terms on the grid of the binade [low, 2 low): their m summed into M, |m| into A; off is
// the largest |t - m|.  The rounding holds while every |t| < low / 2 (A < low / 2 tells), and a term
// is a tie when it is half a grid step off.
__device__ __forceinline__ void scan_terms(const double t[kScanPer], double low, double& M, double& A, double& off) {
    const double c = 1.5 * low;
    double m[kScanPer], a[kScanPer], d[kScanPer];
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
        m[k] = (t[k] + c) - c;                     // nearest multiple of ulp(c) = u
        a[k] = fabs(m[k]);
        d[k] = fabs(t[k] - m[k]);
    }
#pragma unroll
    for (int h = kScanPer / 2; h > 0; h /= 2)
#pragma unroll
        for (int k = 0; k < h; k++) {
            m[k] += m[k + h];
            a[k] += a[k + h];
            d[k] = fmax(d[k], d[k + h]);
        }
    M = m[0]; A = a[0]; off = d[0];
}
// every partial sum of a run with sums M and A from s stays strictly inside the binade of `key`
__device__ __forceinline__ bool scan_inside(double s, int key, double M, double A) {
    // (mirrored for a negative sum: the partial sums' magnitudes lie between these two)
    const double low = scan_low(key), size = fabs(s), along = s > 0.0 ? M : -M;
    return (size + 0.5 * (along - A) > low) & (size + 0.5 * (along + A) < 2.0 * low);
}

// the per-node terms: stored ones, or the three-term dot products of two vectors
struct StoredTerms {
    const double* __restrict__ t;
    __device__ __forceinline__ double operator()(int i) const { return t[i]; }
    // terms i and i + 1 in one 16-byte load (t is aligned to a double only)
    __device__ __forceinline__ void pair(int i, double& a, double& b) const {
        typedef double Pair __attribute__((ext_vector_type(2), aligned(8)));
        const Pair p = *reinterpret_cast<const Pair*>(t + i);
        a = p.x; b = p.y;
    }
};
template <typename VT>
struct VectorTerms {
    const VT* __restrict__ a;
    const VT* __restrict__ b;
    __device__ __forceinline__ double operator()(int i) const {
        VT x[3], y[3];
        ld3(a, i, x);
        ld3(b, i, y);
        return dot3d(x, y);
    }
    __device__ __forceinline__ void pair(int i, double& s, double& t) const { s = (*this)(i); t = (*this)(i + 1); }
};

// the lane's terms own, own + 1, own + 128, own + 129, ... of a round, 0.0 past the end
template <typename Terms>
__device__ __forceinline__ void scan_load(Terms term, int base, int own, int n, double t[kScanPer]) {
    if (base + kScanRound <= n) {
#pragma unroll
        for (int k = 0; k < kScanPer; k += 2) term.pair(base + own + k * 64, t[k], t[k + 1]);
    } else {
#pragma unroll
        for (int k = 0; k < kScanPer; k++) {
            const int i = base + own + (k & ~1) * 64 + (k & 1);
            const double v = term(min(i, n - 1));
            t[k] = i < n ? v : 0.0;
        }
    }
}

// the h-th 32 terms of a round
__device__ __forceinline__ void scan_half(const double* buf, int h, double q[32]) {
    const double* c = buf + scan_at(32) * h;
#pragma unroll
    for (int i = 0; i < 32; i++) q[i] = c[scan_at(i)];
}

// 0.0 + term(0) + term(1) + ... + term(n - 1), n >= 1, every add rounded in that order; all
// kScanThreads threads of the workgroup call it, thread kScanResult has the result
template <typename Terms>
__device__ __forceinline__ double scan_sum(Terms term, int n) {
    constexpr int kBuf = kScanRound + kScanRound / kScanPer * 2;
    __shared__ __align__(16) double buf[3][kBuf];  // the rounds being staged, formed and walked
    __shared__ double tot[2][kScanWaves], gm[2][64], ga[2][64];
    __shared__ int gk[2][64];                      // the piece's key; 0: rule broken; -1: only zeros
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int rounds = (n + kScanRound - 1) / kScanRound;
    const int load = w * 64 * kScanPer + 2 * lane; // a lane loads terms load + 128 k and the next ...
    const int own = (int)threadIdx.x * kScanPer;   // ... and sums terms own .. own + 15
    double s = 0.0, base = 0.0, upto = 0.0;
    double next[kScanPer], t[kScanPer];
    // a wave's terms go through its own part of the buffer (no barrier), then their plain sums
    auto stage = [&](double* b) {
#pragma unroll
        for (int k = 0; k < kScanPer; k += 2)
            *reinterpret_cast<double2*>(b + scan_at(load) + k * scan_at(64)) = make_double2(next[k], next[k + 1]);
    };
    auto take = [&](const double* b, double* sums) {
#pragma unroll
        for (int k = 0; k < kScanPer; k++) t[k] = b[scan_at(own) + k];
        double p[kScanPer];
#pragma unroll
        for (int k = 0; k < kScanPer; k++) p[k] = t[k];
#pragma unroll
        for (int h = kScanPer / 2; h > 0; h /= 2)
#pragma unroll
            for (int k = 0; k < h; k++) p[k] += p[k + h];
        upto = wave_prefix(p[0]);
        if (lane == 63) sums[w] = upto;
    };
    if (w < kScanWaves) {
        scan_load(term, 0, load, n, next);
        stage(buf[0]);
        if (rounds > 1) scan_load(term, kScanRound, load, n, next);
        take(buf[0], tot[0]);
    }
    __syncthreads();
    int b0 = 0;                                    // the buffer of round `it`
    for (int it = 0; it <= rounds; it++) {
        const int b1 = b0 == 2 ? 0 : b0 + 1, slot = it & 1;
        if (w < kScanWaves) {
            if (it + 1 < rounds) {
                stage(buf[b1]);
                if (it + 2 < rounds) scan_load(term, (it + 2) * kScanRound, load, n, next);   // in flight this round
            }
            if (it < rounds) {
                // the piece's approximate start, its terms on that binade's grid
                double start = base;
#pragma unroll
                for (int j = 0; j < kScanWaves; j++) {
                    const double x = tot[slot][j];
                    base += x;
                    start += j < w ? x : 0.0;
                }
                const double before = __shfl(upto, (lane & ~(kScanLanes - 1)) - 1, 64);
                start += lane >= kScanLanes ? before : 0.0;
                int key = scan_key(start);
                const double low = scan_low(key);
                double M, A, off;
                scan_terms(t, low, M, A, off);
                // (without a binade low is 0, m is t, and A is 0 for zeros only)
                const bool broken = key == 0 ? !(A == 0.0) : !(A < 0.5 * low) | (off == low * 0x1p-53);
                if (key == 0) key = -1;
                if (__ballot(broken) >> (lane & ~(kScanLanes - 1)) & 0xf) key = 0;
                M = quad_sum(M);
                A = quad_sum(A);
                if ((lane & (kScanLanes - 1)) == kScanLanes - 1) {
                    const int g = (int)threadIdx.x / kScanLanes;
                    gm[slot][g] = M;
                    ga[slot][g] = A;
                    gk[slot][g] = key;
                }
                if (it + 1 < rounds) take(buf[b1], tot[slot ^ 1]);
            }
        } else if (it > 0) {
            const double m = gm[slot ^ 1][lane], a = ga[slot ^ 1][lane];
            const int k = gk[slot ^ 1][lane];
            const double* c0 = buf[b0 == 0 ? 2 : b0 - 1];
            for (int g = 0; g < 64;) {
                // each piece's start if every piece from g up to it keeps the rule
                const double run = wave_prefix(lane >= g ? m : 0.0);
                const double at = s + dpp_from<0x138, 0xf>(run);   // (the previous lane's)
                const bool keeps = (lane < g) | (k == -1) | ((k != 0) & (k == scan_key(at)) & scan_inside(at, k, m, a));
                const unsigned long long fails = __ballot(!keeps);
                if (fails == 0) {
                    s = lane_value(at + m, 63);
                    break;
                }
                // the failing piece and the next ones that may fail too (as far as their approximate starts tell):
                // the chain, half a piece of terms on its way while the half before is added
                const int f = __builtin_ctzll(fails);
                const unsigned long long keep = ~(fails >> f);
                const int end = keep ? f + __builtin_ctzll(keep) : 64;
                s = lane_value(at, f);
                double q0[32], q1[32];
                scan_half(c0, 2 * f, q0);
                for (int h = 2 * f; h < 2 * end; h += 2) {
                    scan_half(c0, h + 1, q1);
#pragma unroll
                    for (int i = 0; i < 32; i++) s = s + q0[i];
                    scan_half(c0, min(h + 2, 127), q0);
#pragma unroll
                    for (int i = 0; i < 32; i++) s = s + q1[i];
                }
                g = end;
            }
        }
        __syncthreads();
        b0 = b1;
    }
    return s;
}

// the scene's node terms nd summed into InstDev::dots[which], one workgroup per scene of the
// launch set; a stopped scene is skipped
static __global__ __launch_bounds__(kScanThreads) void k_scandot(const int* __restrict__ scenes, InstDev* __restrict__ inst,
                                                                 const double* __restrict__ nd, int which) {
    InstDev* ins = &inst[scenes[blockIdx.x]];
    if (ins->stopped) return;
    const double s = scan_sum(StoredTerms{nd + ins->node_begin}, ins->node_count);
    if (threadIdx.x == kScanResult) ins->dots[which] = s;
}

// BaseMechanicalState::vDot on caller vectors (MechanicalObject::vDot, MechanicalObject.inl
// :2334-2356) in the reference's order
template <typename VT>
__global__ __launch_bounds__(kScanThreads) void k_vdot_seq(const VT* __restrict__ a, const VT* __restrict__ b, int n,
                                                           double* __restrict__ out) {
    const double s = scan_sum(VectorTerms<VT>{a, b}, n);
    if (threadIdx.x == kScanResult) *out = s;
}

}  // namespace sofa_amd
