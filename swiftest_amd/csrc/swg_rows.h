// swg_rows.h -- full-row direct sums of a tile of massive bodies, their terms
// evaluated by several wavefronts and folded in partner order by one.
//
// Body b of a system sums over the partners p ascending, p /= b, taken only
// outside the pair's radii when those are tested (swiftest_kick.f90:165-371):
//  - rows: acc += (Gm_p / (r2 sqrt r2)) (r_p - r_b), over every partner for
//    the first nplm (fully interacting) bodies, over the first nplm partners
//    for the others (:219-262);
//  - triangular (more semi-interacting bodies than others, :190-216): the
//    factor is Gm_p (1 / (r2 sqrt r2)) and the partners before and after b go
//    to two sums, ahj and ahi (the one-thread order of the OpenMP reduction).
//
// A one-lane-per-body walk leaves the chip idle below about 10^5 bodies and
// puts every term's 37 issue slots on one chain.  Here a workgroup takes B
// bodies: KE wavefronts form the factors of a chunk of 64 partners, one
// partner per lane (read straight from memory into registers, a chunk ahead)
// for B / KE bodies each, into LDS, while the fold wavefronts add the chunk
// before, one lane per component of a body.  B = 16 (one fold wavefront, its
// lanes holding x, y and z of the 16 bodies) gives four times the workgroups
// of B = 64 (a fold wavefront per component, every lane of it in use): the
// first is bound by the fold, about 1 us a chunk of its chain and LDS reads, the
// second, for systems that fill the chip either way, by FP64 issue.
// Measured: 2000 bodies 32.6 us (64-body tiles with the partners staged in LDS
// and read there for every term: 69), 10000 bodies 267 us (338), 32000 bodies
// 2.0 ms (2.0); the leaf rows of 10007 bodies 267 us (one lane a body: 4466);
// half of 2000 bodies semi-interacting 60 us (one lane a body: 930).  Many
// short systems keep one body per lane (k_kick_pl_split, which says why).
#pragma once
#include "swg_math.h"

namespace swg {

constexpr int RW_C = 64;       // partners per chunk, one per lane
constexpr int RW_S = RW_C + 2; // row stride of the factors: 16-byte aligned, rows 4 banks apart

// B bodies, KE evaluation wavefronts; A: sets of eight terms the fold reads ahead
template <int B, int KE, int A = 1>
struct RowsLds {
    static constexpr int NF = (3 * B + 63) / 64;  // fold wavefronts
    static constexpr int THREADS = 64 * (KE + NF);
    // wavefronts per SIMD the registers leave room for: two workgroups of 64
    // bodies, four of 16; one of 16 that reads two sets of terms ahead
    static constexpr int WAVES = B == 64 ? 6 : A == 2 ? 2 : 5;
    __align__(16) double fac[2][B][RW_S];
    __align__(16) double pj[2][3][RW_C];  // the partners' positions
    uint64_t take[2][B];                  // bit q: the body takes its term with partner q ...
    int part[2][KE];                      // ... written where some body of the wavefront does not take one
    double out[2][3][B];
};

// Where rows_sums reads component a (x, y, z, Gm, R) of body j.  Every array is
// there, R too where radii are not tested (any array of the length).
struct RowsSrc {
    const double *x, *y, *z, *g, *R;
    int stride;  // of x, y and z
    __device__ double operator()(int a, int j) const
    {
        const double *p = a == 0 ? x : a == 1 ? y : a == 2 ? z : a == 3 ? g : R;
        return p[(int64_t)j * (a < 3 ? stride : 1)];
    }
};

// a value every lane of the wavefront holds, in scalar registers when ON
template <bool ON>
__device__ inline double rows_uniform(double v)
{
    if (!ON) return v;
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// The sums of bodies [b0, b1) (at most B, indices within the system, b0 a
// multiple of B) over their partners, by RowsLds::THREADS threads.
// init(comp, i): the fold's first value for a component of body i (rows only).
// On return (after a barrier) S.out[0] holds the rows' sums, or the triangular
// ahj with ahi in S.out[1].  fast: 0 exact, 1 Gm_p r^-3 from the reciprocal
// square root, 2 the same with the triangular factor formed as Gm_p (1 r^-3).
// FULL: the fold of a chunk fully unrolled, all of its reads ahead (2000
// bodies 35 us, 45 us without); not where two copies of the function stand in
// one kernel, which have no registers for it.
// ZERO (rows whose sums start at +0): a term not taken is folded as a zero
// factor, fma(0, d, s) = s bit for bit (a sum that starts at +0 is never -0)
// for finite d: a body at NaN, which a radius test leaves out of every sum,
// makes them NaN here.  In a step its own failed drift ends the run.  (Selection
// in the chunks with such a separation costs 3 % at every size.)  Otherwise the
// sum is kept by selection, also for a first value of -0 and for partners at
// infinity.
// SELF: the bodies are the partners themselves and leave themselves out;
// otherwise tgt holds others (test particles; nplm = npl, rows).
template <bool FULL, bool ZERO, bool SELF, int B, int KE, int A, class Init>
__device__ __attribute__((always_inline)) inline void rows_sums(RowsLds<B, KE, A> &S, const RowsSrc &load, const RowsSrc &tgt,
                                                                Init init, int b0, int b1, int nplm, int npl, bool tri,
                                                                int fast, bool use_radius)
{
    constexpr int NB = B / KE, G = 4;
    static_assert(NB * KE == B && NB % G == 0, "whole groups of bodies per wavefront");
    static_assert(B == 16 || B == 64, "a chunk holds all of a tile's bodies or none");
    const int lane = (int)(threadIdx.x & 63u), w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // partners any body of the tile needs
    const int jend = !SELF || b0 < nplm ? npl : nplm, nch = (jend + RW_C - 1) / RW_C;
    if (w < KE) {
        // ---- evaluation: this lane's partner against bodies e0 .. e0 + NB - 1
        const int e0 = w * NB;
        double xb[NB], yb[NB], zb[NB], Rb[NB];
        int jmin = npl;
#pragma unroll
        for (int k = 0; k < NB; k++) {
            const int i = min(b0 + e0 + k, b1 - 1);
            xb[k] = rows_uniform<(NB > 4)>(tgt(0, i));
            yb[k] = rows_uniform<(NB > 4)>(tgt(1, i));
            zb[k] = rows_uniform<(NB > 4)>(tgt(2, i));
            Rb[k] = rows_uniform<(NB > 4)>(tgt(4, i));
            if (SELF && i >= nplm) jmin = min(npl, nplm);
        }
        double n[5], p[5];
        auto fetch = [&](int c) __attribute__((always_inline)) {
            const int j = min(c * RW_C + lane, jend - 1);
#pragma unroll
            for (int a = 0; a < 5; a++) n[a] = load(a, j);
        };
        const bool idle = b0 + e0 >= b1;  // past the tile's bodies (never the first wavefront)
        if (idle && lane < 2) S.part[lane][w] = 0;
        if (nch > 0) fetch(0);
        for (int c = 0; c <= nch; c++) {
            if (c < nch && !idle) {
#pragma unroll
                for (int a = 0; a < 5; a++) p[a] = n[a];
                fetch(c + 1);
                const int jt = c * RW_C, j = jt + lane;
                // neither the end of any body's partners nor the tile itself
                const bool plain = jt + RW_C <= jmin && (!SELF || jt + RW_C <= b0 || jt >= b0 + B);
                const bool gok = tri || __all(pair_g_ok_int(p[3]));
                double(*f)[RW_S] = S.fac[c & 1];
                if (w == 0) {
                    S.pj[c & 1][0][lane] = p[0];
                    S.pj[c & 1][1][lane] = p[1];
                    S.pj[c & 1][2][lane] = p[2];
                }
                uint64_t m[NB], full = ~0ull;
#pragma unroll
                for (int k0 = 0; k0 < NB; k0 += G) {
                    // step by step for all of the group's bodies, so that their
                    // chains of operations run side by side
                    double r2[G], gm[G], fc[G];
#pragma unroll
                    for (int u = 0; u < G; u++) {
                        const double rx = p[0] - xb[k0 + u], ry = p[1] - yb[k0 + u], rz = p[2] - zb[k0 + u];
                        r2[u] = dot3(rx, ry, rz, rx, ry, rz);
                    }
#pragma unroll
                    for (int u = 0; u < G; u++) m[k0 + u] = ~0ull;
                    if (use_radius) {
#pragma unroll
                        for (int u = 0; u < G; u++) {
                            const double rs = Rb[k0 + u] + p[4];
                            m[k0 + u] = __ballot(r2[u] > rs * rs);
                        }
                    }
                    if (!plain) {
#pragma unroll
                        for (int u = 0; u < G; u++) {
                            const int i = b0 + e0 + k0 + u;
                            m[k0 + u] &= __ballot((j < (!SELF || i < nplm ? npl : nplm)) & (!SELF | (j != i)));
                        }
                    }
#pragma unroll
                    for (int u = 0; u < G; u++) full &= m[k0 + u];
                    uint32_t far = 0;
                    if (fast) {
                        const bool one = fast == 2 && tri;
#pragma unroll
                        for (int u = 0; u < G; u++) {
                            const double g = gm_over_r3_fast(one ? 1.0 : p[3], r2[u]);
                            fc[u] = one ? p[3] * g : g;
                        }
                    } else {
#pragma unroll
                        for (int u = 0; u < G; u++) {
                            gm[u] = tri ? 1.0 : p[3];
                            // by the high word: the exponent alone decides
                            far = max(far, (uint32_t)(__double2hiint(r2[u]) - PAIR_R2_LO_HI));
                        }
                        pair_factors(gm, r2, fc);
                        if (tri) {
#pragma unroll
                            for (int u = 0; u < G; u++) fc[u] = p[3] * fc[u];
                        }
                    }
                    // the IEEE operations where the cores' range does not hold
                    if (!fast && (!gok || __any(far > PAIR_R2_HI_HI - PAIR_R2_LO_HI))) {
#pragma unroll
                        for (int u = 0; u < G; u++)
                            fc[u] = tri ? p[3] * (1.0 / (r2[u] * sqrt(r2[u]))) : p[3] / (r2[u] * sqrt(r2[u]));
                    }
                    if (ZERO && full != ~0ull) {
#pragma unroll
                        for (int u = 0; u < G; u++) fc[u] = (m[k0 + u] >> lane) & 1 ? fc[u] : 0.0;
                    }
#pragma unroll
                    for (int u = 0; u < G; u++) f[e0 + k0 + u][lane] = fc[u];
                }
                if (!ZERO && full != ~0ull) {
#pragma unroll
                    for (int k = 0; k < NB; k++)
                        if (lane == k) S.take[c & 1][e0 + k] = m[k];
                }
                if (lane == 0) S.part[c & 1][w] = full != ~0ull;
            }
            __syncthreads();
        }
    } else {
        // ---- fold: the fold wavefronts' lanes are component by body
        // (lanes past the last repeat it)
        const int l = min((w - KE) * 64 + lane, 3 * B - 1), comp = l / B, bl = l % B, i = min(b0 + bl, b1 - 1);
        const double cb = tgt(comp, i);
        double acc = tri ? 0.0 : init(comp, i), hi = 0.0;
        // one side's sums over a chunk whose terms are all taken.  The reads of
        // factors and coordinates run AHEAD sets of eight terms before the fold:
        // two sets where the registers are there (a set's adds take less time
        // than a read comes back)
        auto fold64 = [&](double v, const double *f, const double *dc) __attribute__((always_inline)) {
            constexpr int SETS = RW_C / 8, AHEAD = FULL ? A : 1, NB2 = AHEAD + 1;
            const double2 *f2 = (const double2 *)f, *d2 = (const double2 *)dc;
            double2 fa[NB2][4], da[NB2][4];
            auto read = [&](int q) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < 4; u++) fa[q % NB2][u] = f2[4 * q + u], da[q % NB2][u] = d2[4 * q + u];
            };
#pragma unroll
            for (int q = 0; q < AHEAD; q++) read(q);
#pragma unroll (FULL ? SETS : 2)
            for (int q = 0; q < SETS; q++) {
                if (q + AHEAD < SETS) read(q + AHEAD);
                // an empty statement that no read passes
                if (AHEAD > 1) asm volatile("" ::: "memory");
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    v = fma(fa[q % NB2][u].x, da[q % NB2][u].x - cb, v);
                    v = fma(fa[q % NB2][u].y, da[q % NB2][u].y - cb, v);
                }
            }
            return v;
        };
        __syncthreads();
        for (int c = 0; c < nch; c++) {
            const double *f = S.fac[c & 1][bl], *dc = S.pj[c & 1][comp];
            const int jt = c * RW_C;
            int any = 0;
#pragma unroll
            for (int k = 0; k < KE; k++) any |= S.part[c & 1][k];
            // a chunk of taken terms holds no body of the tile (both are
            // aligned to their sizes), so it lies on one side of all of them
            if (!any) {
                if (tri && jt > i) hi = fold64(hi, f, dc);
                else acc = fold64(acc, f, dc);
            } else if (ZERO) {
                const int jn = min(RW_C, jend - jt);
                if (jn == RW_C) {
                    acc = fold64(acc, f, dc);
                } else {
#pragma unroll 8
                    for (int q = 0; q < jn; q++) acc = fma(f[q], dc[q] - cb, acc);
                }
            } else {
                const uint64_t m = S.part[c & 1][bl / NB] ? S.take[c & 1][bl] : ~0ull;
                const int jn = min(RW_C, jend - jt);
#pragma unroll 4
                for (int q = 0; q < jn; q++) {
                    const bool t = (m >> q) & 1u, up = tri & (jt + q > i);
                    const double r = fma(f[q], dc[q] - cb, up ? hi : acc);
                    acc = (t & !up) ? r : acc;
                    hi = (t & up) ? r : hi;
                }
            }
            __syncthreads();
        }
        S.out[0][comp][bl] = acc;
        S.out[1][comp][bl] = hi;
    }
    __syncthreads();
}

}  // namespace swg
