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
// first is bound by the fold's chain of about 10 cycles a term, the second,
// for systems that fill the chip either way, by FP64 issue.
// Measured: 2000 bodies 38 us (64-body tiles with the partners staged in LDS
// and read there for every term: 69), 10000 bodies 300 us (338), 32000 bodies
// 2.03 ms (2.03); the leaf rows of 10007 bodies 315 us (one lane a body: 4466);
// half of 2000 bodies semi-interacting 60 us (one lane a body: 930).
#pragma once
#include "swg_math.h"

namespace swg {

constexpr int RW_C = 64;       // partners per chunk, one per lane
constexpr int RW_S = RW_C + 2; // row stride of the factors: 16-byte aligned, rows 4 banks apart

template <int B, int KE>
struct RowsLds {
    static constexpr int NF = (3 * B + 63) / 64;  // fold wavefronts
    static constexpr int THREADS = 64 * (KE + NF);
    // wavefronts per SIMD the registers leave room for: two workgroups of 64 bodies
    static constexpr int WAVES = B == 64 ? 6 : 2;
    __align__(16) double fac[2][B][RW_S];
    __align__(16) double pj[2][3][RW_C];  // the partners' positions
    uint64_t take[2][B];                  // bit q: the body takes its term with partner q ...
    int part[2][KE];                      // ... written where some body of the wavefront does not take one
    double out[2][3][B];
};

// Where rows_sums reads component a (x, y, z, Gm, R) of body j; a missing
// array (no radii) reads as zero.
struct RowsSrc {
    const double *x, *y, *z, *g, *R;
    int stride;  // of x, y and z
    __device__ double operator()(int a, int j) const
    {
        const double *p = a == 0 ? x : a == 1 ? y : a == 2 ? z : a == 3 ? g : R;
        return p ? p[(int64_t)j * (a < 3 ? stride : 1)] : 0.0;
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
// factor, fma(0, d, s) = s bit for bit (d finite; a sum that starts at +0 is
// never -0); otherwise the sum is kept by selection, also for a first value
// of -0 and for partners at infinity.
template <bool FULL, bool ZERO, int B, int KE, class Init>
__device__ __attribute__((always_inline)) inline void rows_sums(RowsLds<B, KE> &S, const RowsSrc &load, Init init,
                                                                int b0, int b1, int nplm, int npl, bool tri, int fast,
                                                                bool use_radius)
{
    constexpr int NB = B / KE, G = NB < 4 ? NB : 4;
    static_assert(NB * KE == B && NB % G == 0, "whole groups of bodies per wavefront");
    static_assert(B == 16 || B == 64, "a chunk holds all of a tile's bodies or none");
    const int lane = (int)(threadIdx.x & 63u), w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // partners any body of the tile needs
    const int jend = b0 < nplm ? npl : nplm, nch = (jend + RW_C - 1) / RW_C;
    if (w < KE) {
        // ---- evaluation: this lane's partner against bodies e0 .. e0 + NB - 1
        const int e0 = w * NB;
        double xb[NB], yb[NB], zb[NB], Rb[NB];
        int jmin = npl;
#pragma unroll
        for (int k = 0; k < NB; k++) {
            const int i = min(b0 + e0 + k, b1 - 1);
            xb[k] = rows_uniform<(NB > 4)>(load(0, i));
            yb[k] = rows_uniform<(NB > 4)>(load(1, i));
            zb[k] = rows_uniform<(NB > 4)>(load(2, i));
            Rb[k] = rows_uniform<(NB > 4)>(load(4, i));
            if (i >= nplm) jmin = min(npl, nplm);
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
                if (c + 1 < nch) fetch(c + 1);
                const int jt = c * RW_C, j = jt + lane;
                // neither the end of any body's partners nor the tile itself
                const bool plain = jt + RW_C <= jmin && (jt + RW_C <= b0 || jt >= b0 + B);
                const bool gok = tri || __all(pair_g_ok(p[3]));
                double(*f)[RW_S] = S.fac[c & 1];
                if (w == 0) {
                    S.pj[c & 1][0][lane] = p[0];
                    S.pj[c & 1][1][lane] = p[1];
                    S.pj[c & 1][2][lane] = p[2];
                }
                uint64_t m[NB], full = ~0ull;
#pragma unroll
                for (int k0 = 0; k0 < NB; k0 += G) {
                    double r2[G], fc[G];
                    uint32_t far = 0;
#pragma unroll
                    for (int u = 0; u < G; u++) {
                        const int k = k0 + u;
                        const double rx = p[0] - xb[k], ry = p[1] - yb[k], rz = p[2] - zb[k];
                        r2[u] = dot3(rx, ry, rz, rx, ry, rz);
                        const double rs = Rb[k] + p[4];
                        m[k] = use_radius ? __ballot(r2[u] > rs * rs) : ~0ull;
                        if (!plain) {
                            const int i = b0 + e0 + k;
                            m[k] &= __ballot((j < (i < nplm ? npl : nplm)) & (j != i));
                        }
                        full &= m[k];
                        if (fast) {
                            const bool one = fast == 2 && tri;
                            const double g = gm_over_r3_fast(one ? 1.0 : p[3], r2[u]);
                            fc[u] = one ? p[3] * g : g;
                        } else {
                            const double g = div_core(tri ? 1.0 : p[3], r2[u] * sqrt_core(r2[u]));
                            fc[u] = tri ? p[3] * g : g;
                            // by the high word: the exponent alone decides
                            far = max(far, (uint32_t)(__double2hiint(r2[u]) - PAIR_R2_LO_HI));
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
        const double cb = load(comp, i);
        double acc = tri ? 0.0 : init(comp, i), hi = 0.0;
        // one side's sums over a chunk whose terms are all taken, the reads of
        // the next eight factors and coordinates issued before the current
        // eight are folded
        auto fold64 = [&](double v, const double *f, const double *dc) __attribute__((always_inline)) {
            const double2 *f2 = (const double2 *)f, *d2 = (const double2 *)dc;
            double2 fa[4], da[4];
#pragma unroll
            for (int u = 0; u < 4; u++) fa[u] = f2[u], da[u] = d2[u];
#pragma unroll (FULL ? RW_C / 8 : 2)
            for (int q = 4; q <= RW_C / 2; q += 4) {
                double2 fn[4], dn[4];
                const int qn = min(q, RW_C / 2 - 4);
#pragma unroll
                for (int u = 0; u < 4; u++) fn[u] = f2[qn + u], dn[u] = d2[qn + u];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    v = fma(fa[u].x, da[u].x - cb, v);
                    v = fma(fa[u].y, da[u].y - cb, v);
                }
#pragma unroll
                for (int u = 0; u < 4; u++) fa[u] = fn[u], da[u] = dn[u];
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
