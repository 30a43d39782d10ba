// k_step.hip -- kernels of the HELIO / SyMBA step outside the recursion:
// frame changes, linear drift, velocity kicks with the direct-sum
// accelerations, and the Danby drift.
//
// Reference behaviour: helio_step.f90:37-119, symba_step.f90:55-115,
// helio_kick.f90:91-169, helio_drift.f90:14-200, swiftest_util.f90:363-485,
// swiftest_kick.f90:69-415, symba_kick.f90:36-123, swiftest_drift.f90:60-138.
#include "swg_kernels.h"
#include "swg_math.h"
#include "swg_rows.h"


namespace swg {

static inline int cdiv(int64_t a, int b) { return (int)((a + b - 1) / b); }

// pl-pl and pl-tp terms formed together per lane before they are folded in
// order
constexpr int KPL_G = 4;
#ifndef SWG_KTP_G
#define SWG_KTP_G 4
#endif
constexpr int KTP_G = SWG_KTP_G;

__device__ inline bool pl_active(const PlDev &pl, int i) { return pl.status[i] != INACTIVE; }
__device__ inline bool tp_active(const TpDev &tp, int j) { return tp.status[j] == ACTIVE; }

// Block y copies array y.
__global__ void k_copy_list(CopyList c)
{
    const CopyItem it = c.item[blockIdx.y];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < it.n; i += (int64_t)gridDim.x * blockDim.x)
        it.dst[i] = it.src[i];
}

// symba_step_reset_system (symba_step.f90:265-331): recursion levels to -1
// and encounter radii of level 0; the systems' encounter flags and the
// recursion's counters are cleared with them
__global__ void k_reset_levels(PlDev pl, TpDev tp, SysDev sy, int32_t *sub_stats, int npl, int ntp, int nsys)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nsys) {
        sy.enc_pp[i] = 0;
        sy.enc_pt[i] = 0;
    }
    if (sub_stats && i < 4) sub_stats[i] = i == 1 ? -1 : 0;  // [1]: the deepest level, -1 = none
    if (i < npl) {
        pl.levelg[i] = -1;
        pl.levelm[i] = -1;
        pl.renc[i] = (pl.rhill[i] * RHSCALE) * 1.0;  // set_renc(0), symba_util.f90:245-267
    }
    if (i < ntp) {
        tp.levelg[i] = -1;
        tp.levelm[i] = -1;
    }
}

// Per-system sums, one workgroup per system.  Each sum is a serial chain in
// the reference's order.  The bodies go through LDS a chunk at a time as the
// terms of the sums (products and quotients formed in parallel, each exactly as
// the serial expression forms it): three wavefronts stage a chunk while the
// first one's lanes, one per sum, add the chunk before.  Bound: the chains'
// dependent adds, about 10 cycles each.  Measured at 2000 bodies: k_sums_begin
// (two walks, the second after the first) 61 -> 26 us, k_sums_end (its two walks
// side by side) 53 -> 14.5 us, against staging and adding in turn with eight
// terms read ahead.
constexpr int SUM_T = 256, SUM_CH = 384;
// largest system whose bodies the workgroup of its sums updates too: four rounds
// of its threads take about what a launch does (2.5 us for a few bodies, 4.8 us
// at 2000)
constexpr int SUM_APPLY = 1024;

struct SumStage {
    // the terms of up to six sums; two words more a row than the banks wrap at,
    // so the lanes' reads fall on different ones
    __align__(16) double t[2][6][SUM_CH + 2];
};

// The serial chain over a staged chunk: acc + t[0] + ... + t[n-1] in order.
// The reads of the next 32 terms are issued before the adds of the current 32,
// in two sets of registers that change places.  A sum that subtracts stages its
// terms negated (s - x = s + (-x) bit for bit), and a body a masked sum skips
// stages +0.0 instead: the chains start at +0.0, a sum that starts at +0 is
// never -0 (x + (-x) = +0 in round-to-nearest), and s + (+0) = s bit for bit
// for every other s, so the sums are the masked ones exactly.
__device__ inline double chain(double acc, const double *t, int n)
{
    constexpr int G = 16;  // pairs of terms per set
    const double2 *t2 = (const double2 *)t;
    const int sets = n / (2 * G);
    double2 v[G], w[G];
    auto read = [&](double2 *o, int g) {
#pragma unroll
        for (int u = 0; u < G; u++) o[u] = t2[G * g + u];
    };
    auto add = [&](const double2 *o) {
#pragma unroll
        for (int u = 0; u < G; u++) {
            acc += o[u].x;
            acc += o[u].y;
        }
    };
    if (sets > 0) {
        read(v, 0);
        for (int g = 0; g < sets; g += 2) {
            read(w, min(g + 1, sets - 1));
            add(v);
            if (g + 1 == sets) break;
            read(v, min(g + 2, sets - 1));
            add(w);
        }
    }
    for (int k = 2 * G * sets; k < n; k++) acc += t[k];
    return acc;
}

// What the sums need of a body.
struct SumBody {
    double g, x, y, z;
    bool act;
};
__device__ inline SumBody sum_body(const PlDev &pl, const Vec3p &v, int i)
{
    return SumBody{pl.Gm[i], v.x[i], v.y[i], v.z[i], pl.status[i] != INACTIVE};
}

// Chunks of bodies [p0, p1): for k = 0 ... n-1 the staging wavefronts call
// stage(b, k, body k of the chunk), and a chunk later the first one calls
// add(b, n); b is the buffer.  BOTH: stage also gets body k of the chunk as
// counted from the end of the range.  The bodies' loads are issued a chunk
// ahead of their staging, so that their latency passes behind the adds.
template <bool BOTH, class StageF, class AddF>
__device__ inline void sums_chunks(const PlDev &pl, const Vec3p &v, int p0, int p1, StageF stage, AddF add)
{
    constexpr int W = SUM_T - 64, U = SUM_CH / W;
    static_assert(U * W == SUM_CH, "whole rounds");
    const int tid = threadIdx.x, n = p1 - p0, nch = (n + SUM_CH - 1) / SUM_CH;
    if (n <= 0) return;
    if (tid >= 64) {
        SumBody f[U], r[U];
        auto load = [&](int c) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = min(c * SUM_CH + tid - 64 + u * W, n - 1);
                f[u] = sum_body(pl, v, p0 + k);
                if (BOTH) r[u] = sum_body(pl, v, p1 - 1 - k);
            }
        };
        load(0);
        for (int c = 0; c <= nch; c++) {
            SumBody a[U], b[U];
#pragma unroll
            for (int u = 0; u < U; u++) a[u] = f[u], b[u] = BOTH ? r[u] : f[u];
            if (c + 1 < nch) load(c + 1);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = tid - 64 + u * W;
                if (c * SUM_CH + k < n) stage(c & 1, k, a[u], b[u]);
            }
            __syncthreads();
        }
    } else {
        for (int c = 0; c <= nch; c++) {
            if (c > 0) add((c - 1) & 1, min(SUM_CH, n - (c - 1) * SUM_CH));
            __syncthreads();
        }
    }
}

// The sums of vh2vb (swiftest_util.f90:424-459) over bodies [p0, p1): lane 0
// returns sum(Gm), lanes 1-3 the components of -sum(Gm vh), in body order.
__device__ inline double sums_gm_vh(SumStage &S, const PlDev &pl, int p0, int p1)
{
    const int tid = threadIdx.x;
    double acc = 0.0;
    sums_chunks<false>(
        pl, pl.vh, p0, p1,
        [&](int b, int k, const SumBody &q, const SumBody &) {
            S.t[b][0][k] = q.g;
            S.t[b][1][k] = -(q.g * q.x);
            S.t[b][2][k] = -(q.g * q.y);
            S.t[b][3][k] = -(q.g * q.z);
        },
        [&](int b, int n) {
            if (tid < 4) acc = chain(acc, S.t[b][tid], n);
        });
    return acc;
}

// vb = vh + cb%vb when lfirst; then the linear drift rh += pt*dt
// (helio_drift.f90:129-163, masked)
__device__ inline void pl_begin_one(const PlDev &pl, int i, bool first, const double *cb, const double *pt, double dth)
{
    if (first) {
        pl.vb.x[i] = pl.vh.x[i] + cb[0];
        pl.vb.y[i] = pl.vh.y[i] + cb[1];
        pl.vb.z[i] = pl.vh.z[i] + cb[2];
    }
    if (pl_active(pl, i)) {
        pl.rh.x[i] = fma(pt[0], dth, pl.rh.x[i]);
        pl.rh.y[i] = fma(pt[1], dth, pl.rh.y[i]);
        pl.rh.z[i] = fma(pt[2], dth, pl.rh.z[i]);
    }
}

// Start of a step:
//   vh->vb (swiftest_util.f90:424-459) when lfirst: cb%vb = -sum(Gm vh) / (GM_cb + sum(Gm))
//   lindrift pt (helio_drift.f90:129-163): pt = sum_masked(Gm vb) / GM_cb
// Lane 0 sums Gm, lanes 1-3 the components of sum(Gm vh); then lanes 0-2 the
// components of pt.  With apply the workgroup goes on to its bodies what
// k_pl_begin_apply does.
__global__ __launch_bounds__(SUM_T) void k_sums_begin(PlDev pl, SysDev sy, int nsys, int force, double dth, int apply)
{
    __shared__ SumStage S;
    __shared__ double shr[4], scb[3], spt[3];
    const int s = blockIdx.x, tid = threadIdx.x;
    const int p0 = sy.pl_off[s], p1 = sy.pl_off[s + 1];
    if (p1 == p0 || sy.frozen[s]) return;
    const bool first = force || sy.lfirst[s];
    if (first) {
        const double acc = sums_gm_vh(S, pl, p0, p1);
        if (tid < 4) shr[tid] = acc;
        __syncthreads();
        if (tid < 3) {
            const double cb = shr[tid + 1] / (sy.GMcb[s] + shr[0]);
            scb[tid] = cb;
            sy.cbvb[3 * s + tid] = cb;
        }
        __syncthreads();
    }
    const Vec3p v = first ? pl.vh : pl.vb;
    double pt = 0.0;
    sums_chunks<false>(
        pl, v, p0, p1,
        [&](int b, int k, const SumBody &q, const SumBody &) {
            const double wx = first ? q.x + scb[0] : q.x;
            const double wy = first ? q.y + scb[1] : q.y;
            const double wz = first ? q.z + scb[2] : q.z;
            S.t[b][0][k] = q.act ? q.g * wx : 0.0;
            S.t[b][1][k] = q.act ? q.g * wy : 0.0;
            S.t[b][2][k] = q.act ? q.g * wz : 0.0;
        },
        [&](int b, int n) {
            if (tid < 3) pt = chain(pt, S.t[b][tid], n);
        });
    if (tid < 3) spt[tid] = sy.ptbeg[3 * s + tid] = pt / sy.GMcb[s];
    if (!apply) return;
    __syncthreads();
    const double cb[3] = {first ? scb[0] : 0.0, first ? scb[1] : 0.0, first ? scb[2] : 0.0};
    const double p[3] = {spt[0], spt[1], spt[2]};
    for (int i = p0 + tid; i < p1; i += SUM_T) pl_begin_one(pl, i, first, cb, p, dth);
}

__global__ void k_pl_begin_apply(PlDev pl, SysDev sy, int npl, double dth, int force)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npl) return;
    int s = pl.sys[i];
    if (sy.frozen[s]) return;
    pl_begin_one(pl, i, force || sy.lfirst[s], sy.cbvb + 3 * s, sy.ptbeg + 3 * s, dth);
}

// Massive-body half kick (helio_kick_vb_pl, helio_kick.f90:91-132):
//   ah = full-row direct sum over j ascending, j /= i, with the radius overlap
//        test (swiftest_kick.f90:219-240, symba_kick.f90:14-33);
//   ah -= (0 + ahi) + ahj over the pl-pl encounter list (symba_kick.f90:61-70,
//        swiftest_kick.f90:69-115): ahi over pairs where i is index1, ahj over
//        pairs where i is index2, each in list order;
//   rbeg/rend = rh;  vb += ah*dt.
// One lane owns body i and walks j in order, so each sum keeps the
// reference's sequence; the j bodies are staged through LDS in blocks of BLK.
template <int BLK>
__global__ __launch_bounds__(BLK) void k_kick_pl(PlDev pl, SysDev sy, ListDev pp, const Tile *tiles, double dt,
                                                 int lbeg, int use_radius, int do_pairs)
{
    static_assert(BLK % KPL_G == 0, "the grouped row walk reads LDS in whole groups");
    __shared__ double sx[BLK], syy[BLK], sz[BLK], sgm[BLK], sr[BLK];
    const Tile tl = tiles[blockIdx.x];
    const int p0 = sy.pl_off[tl.s], p1 = sy.pl_off[tl.s + 1];
    const int i = tl.b0 + (int)threadIdx.x;
    const bool valid = i < tl.b1;
    double xi = 0.0, yi = 0.0, zi = 0.0, Ri = 0.0;
    if (valid) {
        xi = pl.rh.x[i];
        yi = pl.rh.y[i];
        zi = pl.rh.z[i];
        Ri = pl.R[i];
    }
    double ax = 0.0, ay = 0.0, az = 0.0;
    for (int jt = p0; jt < p1; jt += BLK) {
        int j = jt + (int)threadIdx.x;
        bool gok = true;
        if (j < p1) {
            sx[threadIdx.x] = pl.rh.x[j];
            syy[threadIdx.x] = pl.rh.y[j];
            sz[threadIdx.x] = pl.rh.z[j];
            sgm[threadIdx.x] = pl.Gm[j];
            sr[threadIdx.x] = pl.R[j];
            gok = pair_g_ok(pl.Gm[j]);
        }
        const bool tile_gok = __syncthreads_and(gok);
        const int jn = min(BLK, p1 - jt);
        if (valid) {
            // Groups of KPL_G bodies: the factors of a group are formed
            // without branches (the exact cores, garbage where a term is
            // not taken or its r2 is outside the cores' range), the IEEE
            // operations redo the rare out-of-range terms under a
            // wave-uniform test, and the terms are folded in j order with
            // selects (a term not taken leaves the sum as it is).  BLK is a
            // multiple of KPL_G, so the LDS reads stay inside the tile.
            for (int q0 = 0; q0 < jn; q0 += KPL_G) {
                double rx[KPL_G], ry[KPL_G], rz[KPL_G], r2[KPL_G], fac[KPL_G];
                bool take[KPL_G], need[KPL_G];
                bool any_need = false;
#pragma unroll
                for (int u = 0; u < KPL_G; u++) {
                    const int q = q0 + u;
                    rx[u] = sx[q] - xi;
                    ry[u] = syy[q] - yi;
                    rz[u] = sz[q] - zi;
                    r2[u] = dot3(rx[u], ry[u], rz[u], rx[u], ry[u], rz[u]);
                    const double rs = Ri + sr[q];
                    // & and | (not && and ||): no short-circuit, no branches
                    take[u] = (q < jn) & (jt + q != i) & (!use_radius | (r2[u] > rs * rs));
                    fac[u] = div_core(sgm[q], r2[u] * sqrt_core(r2[u]));
                    need[u] = take[u] & !(tile_gok & (r2[u] >= PAIR_R2_LO) & (r2[u] <= PAIR_R2_HI));
                    any_need = any_need | need[u];
                }
                if (__ballot(any_need)) {
#pragma unroll
                    for (int u = 0; u < KPL_G; u++)
                        if (need[u]) fac[u] = sgm[q0 + u] / (r2[u] * sqrt(r2[u]));
                }
#pragma unroll
                for (int u = 0; u < KPL_G; u++) {
                    ax = take[u] ? fma(fac[u], rx[u], ax) : ax;
                    ay = take[u] ? fma(fac[u], ry[u], ay) : ay;
                    az = take[u] ? fma(fac[u], rz[u], az) : az;
                }
            }
        }
        __syncthreads();
    }
    if (!valid) return;
    if (do_pairs) {
        double hix = 0.0, hiy = 0.0, hiz = 0.0, hjx = 0.0, hjy = 0.0, hjz = 0.0;
        // Both walks gather KPL_G entries at a time (indices past the end
        // repeat the walk's current entry, whose term is then not taken) so
        // that the gathers overlap, and fold the terms in list order.
        const int64_t c0 = pp.colstart[i], c1 = c0 + pp.colcnt[i];
        for (int64_t c = c0; c < c1; c += KPL_G) {  // pairs (p, i), p < i
            double rx[KPL_G], ry[KPL_G], rz[KPL_G], fac[KPL_G];
            bool take[KPL_G];
#pragma unroll
            for (int u = 0; u < KPL_G; u++) {
                const int64_t cu = c + u < c1 ? c + u : c;
                const int p = pp.i1[pp.col[cu]];
                rx[u] = xi - pl.rh.x[p];
                ry[u] = yi - pl.rh.y[p];
                rz[u] = zi - pl.rh.z[p];
                const double rji2 = dot3(rx[u], ry[u], rz[u], rx[u], ry[u], rz[u]);
                const double rs = pl.R[p] + Ri;
                take[u] = (c + u < c1) & (rji2 > rs * rs);
                const double irij3 = 1.0 / (rji2 * sqrt(rji2));
                fac[u] = pl.Gm[p] * irij3;
            }
#pragma unroll
            for (int u = 0; u < KPL_G; u++) {
                hjx = take[u] ? fma(-fac[u], rx[u], hjx) : hjx;
                hjy = take[u] ? fma(-fac[u], ry[u], hjy) : hjy;
                hjz = take[u] ? fma(-fac[u], rz[u], hjz) : hjz;
            }
        }
        const int64_t r0 = pp.rowstart[i], r1 = r0 + pp.rowcnt[i];
        for (int64_t k = r0; k < r1; k += KPL_G) {  // pairs (i, j), j > i
            double rx[KPL_G], ry[KPL_G], rz[KPL_G], fac[KPL_G];
            bool take[KPL_G];
#pragma unroll
            for (int u = 0; u < KPL_G; u++) {
                const int64_t ku = k + u < r1 ? k + u : k;
                const int j = pp.i2[ku];
                rx[u] = pl.rh.x[j] - xi;
                ry[u] = pl.rh.y[j] - yi;
                rz[u] = pl.rh.z[j] - zi;
                const double rji2 = dot3(rx[u], ry[u], rz[u], rx[u], ry[u], rz[u]);
                const double rs = Ri + pl.R[j];
                take[u] = (k + u < r1) & (rji2 > rs * rs);
                const double irij3 = 1.0 / (rji2 * sqrt(rji2));
                fac[u] = pl.Gm[j] * irij3;
            }
#pragma unroll
            for (int u = 0; u < KPL_G; u++) {
                hix = take[u] ? fma(fac[u], rx[u], hix) : hix;
                hiy = take[u] ? fma(fac[u], ry[u], hiy) : hiy;
                hiz = take[u] ? fma(fac[u], rz[u], hiz) : hiz;
            }
        }
        ax = ax - ((0.0 + hix) + hjx);
        ay = ay - ((0.0 + hiy) + hjy);
        az = az - ((0.0 + hiz) + hjz);
    }
    Vec3p rb = lbeg ? pl.rbeg : pl.rend;
    rb.x[i] = xi;
    rb.y[i] = yi;
    rb.z[i] = zi;
    if (pl_active(pl, i)) {
        pl.vb.x[i] = fma(ax, dt, pl.vb.x[i]);
        pl.vb.y[i] = fma(ay, dt, pl.vb.y[i]);
        pl.vb.z[i] = fma(az, dt, pl.vb.z[i]);
    }
}

// ---------------------------------------------------------------------------
// The same massive-body half kick with the row's terms evaluated by KE
// wavefronts and folded in j order by others (swg_rows.h), B bodies per
// workgroup; the same bits as k_kick_pl.  With TINY the system may have
// semi-interacting bodies (GMTINY): its first nplm bodies interact with every
// body, the others only with those (symba_kick.f90:14-33).  The two
// encounter-pair walks run on evaluation wavefronts side by side, four entries
// of a body at a time on lanes 16 apart, folded in list order.
// fast: the factors from gm_over_r3_fast.
// ---------------------------------------------------------------------------


typedef const __attribute__((address_space(4))) double cdouble;
__device__ inline const cdouble *cview(const double *p) { return (const cdouble *)p; }

template <int B, int KE, int A, bool TINY, bool fast>
__global__ __launch_bounds__((RowsLds<B, KE, A>::THREADS), (RowsLds<B, KE, A>::WAVES)) void k_kick_pl_rows(PlDev pl, SysDev sy, ListDev pp,
                                                                          const Tile *tiles, double dt, int lbeg,
                                                                          int use_radius, int do_pairs)
{
    constexpr int WK = B / 16;  // wavefronts walking each side of the encounter pairs, 16 bodies each
    static_assert(KE >= 2 * WK, "the evaluation wavefronts walk the encounter pairs");
    __shared__ RowsLds<B, KE, A> S;
    __shared__ double hpart[2][3][B];
    const Tile tl = tiles[blockIdx.x];
    const int p0 = sy.pl_off[tl.s];
    // a slot's padding adds exact zeros to rows, but is not among the bodies
    // whose number chooses the branch
    const int n = TINY ? sy.nreal[tl.s] : sy.pl_off[tl.s + 1] - p0;
    const int nm = TINY ? sy.nplm[tl.s] : n;
    const bool tri = TINY && n - nm > nm;
    const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
    const RowsSrc src{pl.rh.x + p0, pl.rh.y + p0, pl.rh.z + p0, pl.Gm + p0, pl.R + p0, 1};
    const auto zero = [](int, int) { return 0.0; };
    if (tri) rows_sums<!TINY, !TINY, true>(S, src, src, zero, tl.b0 - p0, tl.b1 - p0, nm, n, true, fast ? 2 : 0, use_radius != 0);
    else rows_sums<!TINY, !TINY, true>(S, src, src, zero, tl.b0 - p0, tl.b1 - p0, nm, n, false, fast ? 2 : 0, use_radius != 0);
    if (do_pairs && w < 2 * WK) {
        // the first WK wavefronts: ahj over pairs (p, i), p < i; the next: ahi
        // over pairs (i, j)
        const int side = w / WK, l16 = lane & 15, sub = lane >> 4, bl = (w % WK) * 16 + l16, i = tl.b0 + bl;
        const bool valid = i < tl.b1;
        const int ii = valid ? i : tl.b0;
        const double xi = pl.rh.x[ii], yi = pl.rh.y[ii], zi = pl.rh.z[ii], Ri = pl.R[ii];
        const int64_t c0 = side == 0 ? pp.colstart[ii] : pp.rowstart[ii];
        const int cnt = valid ? (side == 0 ? pp.colcnt[ii] : pp.rowcnt[ii]) : 0;
        double hx = 0.0, hy = 0.0, hz = 0.0;
        for (int t = 0; __any(t < cnt); t += 4) {
            double rx = 0.0, ry = 0.0, rz = 0.0, f = 0.0;
            int take = 0;
            if (t + sub < cnt) {
                const int64_t e = c0 + t + sub;
                const int q = side == 0 ? pp.i1[pp.col[e]] : pp.i2[e];
                // from index1 to index2
                rx = side == 0 ? xi - pl.rh.x[q] : pl.rh.x[q] - xi;
                ry = side == 0 ? yi - pl.rh.y[q] : pl.rh.y[q] - yi;
                rz = side == 0 ? zi - pl.rh.z[q] : pl.rh.z[q] - zi;
                const double r2 = dot3(rx, ry, rz, rx, ry, rz), rs = pl.R[q] + Ri;
                take = r2 > rs * rs;
                f = fast ? gm_over_r3_fast(pl.Gm[q], r2) : pl.Gm[q] * (1.0 / (r2 * sqrt(r2)));
                f = side == 0 ? -f : f;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int l = 16 * u + l16;
                const double fu = __shfl(f, l, 64), x = __shfl(rx, l, 64), y = __shfl(ry, l, 64), z = __shfl(rz, l, 64);
                const bool tk = __shfl(take, l, 64) != 0;
                hx = tk ? fma(fu, x, hx) : hx;
                hy = tk ? fma(fu, y, hy) : hy;
                hz = tk ? fma(fu, z, hz) : hz;
            }
        }
        if (sub == 0) {
            hpart[side][0][bl] = hx;
            hpart[side][1][bl] = hy;
            hpart[side][2][bl] = hz;
        }
    }
    if (do_pairs) __syncthreads();
    const int bl = (int)threadIdx.x, i = tl.b0 + bl;
    if (bl >= B || i >= tl.b1) return;
    const double xi = pl.rh.x[i], yi = pl.rh.y[i], zi = pl.rh.z[i];
    double ax = S.out[0][0][bl], ay = S.out[0][1][bl], az = S.out[0][2][bl];
    if (tri) {
        ax = (0.0 + S.out[1][0][bl]) + ax;
        ay = (0.0 + S.out[1][1][bl]) + ay;
        az = (0.0 + S.out[1][2][bl]) + az;
    }
    if (do_pairs) {
        ax = ax - ((0.0 + hpart[1][0][bl]) + hpart[0][0][bl]);
        ay = ay - ((0.0 + hpart[1][1][bl]) + hpart[0][1][bl]);
        az = az - ((0.0 + hpart[1][2][bl]) + hpart[0][2][bl]);
    }
    Vec3p rb = lbeg ? pl.rbeg : pl.rend;
    rb.x[i] = xi;
    rb.y[i] = yi;
    rb.z[i] = zi;
    if (pl_active(pl, i)) {
        pl.vb.x[i] = fma(ax, dt, pl.vb.x[i]);
        pl.vb.y[i] = fma(ay, dt, pl.vb.y[i]);
        pl.vb.z[i] = fma(az, dt, pl.vb.z[i]);
    }
}

// ---------------------------------------------------------------------------
// The same with one body per lane, for ensembles of many short systems: a tile
// of 64 bodies, eight evaluating wavefronts that each form the factors of their
// eight partners of a 64-partner chunk for all 64 bodies (the exact cores,
// grouped and branch-free as in k_kick_pl) into LDS, a zero where a term is not
// taken, and three that fold the chunk before in j order, one component each.
// The partners are staged in LDS a chunk ahead.  A short system's workgroup
// spends most of its time on starting up and on the chunk that holds the tile
// itself, where a body's zero separation from itself sends whole groups of terms
// through the IEEE operations in k_kick_pl_rows and none here.
// Measured, this kernel / k_kick_pl_rows with 64 and with 16 bodies a tile, us:
// 512 systems of 128 bodies 22 / 32 / 43, 1024 of 4 to 512 89 / 102 / 116, 128
// of 512 67 / 70 / 98, 64 of 1024 128 / 123 / 171, one of 2000 67 / - / 30.
// ---------------------------------------------------------------------------
constexpr int KPLS_C = 64;  // partners per chunk
constexpr int KPLS_KE = 8;  // evaluating wavefronts

__global__ __launch_bounds__(64 * (KPLS_KE + 3)) void k_kick_pl_split(PlDev pl, SysDev sy, ListDev pp, const Tile *tiles,
                                                                     double dt, int lbeg, int use_radius, int do_pairs)
{
    constexpr int KE = KPLS_KE;
    static_assert(KPLS_C % (4 * KE) == 0, "each evaluation wavefront takes whole groups of four partners");
    static_assert(KPLS_C == 64, "one partner per lane when a chunk is staged");
    __shared__ double facb[2][KPLS_C][64];
    __shared__ double hpart[2][3][64];
    __shared__ double fsum[3][64];  // each component's fold
    // the partners of chunk c (x, y, z, Gm, R) in slot c % 3: the chunk being
    // folded, the one being evaluated and the next one
    __shared__ double pj[3][5][KPLS_C];
    const Tile tl = tiles[blockIdx.x];
    const int p0 = sy.pl_off[tl.s], p1 = sy.pl_off[tl.s + 1];
    const int lane = (int)(threadIdx.x & 63u);
    // wavefronts 0..KE-1 evaluate; KE, KE+1, KE+2 fold the x, y, z sums
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int i = tl.b0 + lane;
    const bool valid = i < tl.b1;
    double xi = 0.0, yi = 0.0, zi = 0.0, Ri = 0.0;
    if (valid) {
        xi = pl.rh.x[i];
        yi = pl.rh.y[i];
        zi = pl.rh.z[i];
        Ri = pl.R[i];
    }
    const int n = p1 - p0, nch = (n + KPLS_C - 1) / KPLS_C;
    constexpr int PER = KPLS_C / KE;
    // staging of chunk c by the first wavefront, one partner per lane
    auto stage = [&](int c) {
        const int jt = p0 + c * KPLS_C, jn = min(KPLS_C, p1 - jt);
        if (lane < jn) {
            const int j = jt + lane;
            double(*d)[KPLS_C] = pj[c % 3];
            d[0][lane] = pl.rh.x[j];
            d[1][lane] = pl.rh.y[j];
            d[2][lane] = pl.rh.z[j];
            d[3][lane] = pl.Gm[j];
            d[4][lane] = pl.R[j];
        }
    };
    // evaluation of chunk c into buffer c & 1 (wavefronts 0 .. KE-1)
    auto evaluate = [&](int c) {
        const int jt = p0 + c * KPLS_C, jn = min(KPLS_C, p1 - jt);
        const double(*d)[KPLS_C] = pj[c % 3];
        // every mass of the chunk inside the exact cores' range: one column per lane
        const bool gok_lane = lane >= jn || pair_g_ok(d[3][lane]);
        const bool tile_gok = __all(gok_lane);
        double(*fb)[64] = facb[c & 1];
        for (int q0 = w * PER; q0 < (w + 1) * PER; q0 += 4) {
            double r2[4], fac[4], rx[4], ry[4], rz[4];
            bool take[4], need[4];
            bool any_need = false;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int q = q0 + u;
                const int qq = min(q, jn - 1);  // in range; a column past the end is not taken
                rx[u] = d[0][qq] - xi;
                ry[u] = d[1][qq] - yi;
                rz[u] = d[2][qq] - zi;
                r2[u] = dot3(rx[u], ry[u], rz[u], rx[u], ry[u], rz[u]);
                const double rs = Ri + d[4][qq];
                take[u] = (q < jn) & (jt + q != i) & (!use_radius | (r2[u] > rs * rs));
                fac[u] = div_core(d[3][qq], r2[u] * sqrt_core(r2[u]));
                need[u] = take[u] & !(tile_gok & (r2[u] >= PAIR_R2_LO) & (r2[u] <= PAIR_R2_HI));
                any_need = any_need | need[u];
            }
            if (__ballot(any_need)) {
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (need[u]) fac[u] = d[3][min(q0 + u, jn - 1)] / (r2[u] * sqrt(r2[u]));
            }
#pragma unroll
            for (int u = 0; u < 4; u++) fb[q0 + u][lane] = take[u] ? fac[u] : 0.0;
        }
    };
    double acc = 0.0;  // a fold wavefront's component sum
    const int comp = w - KE;
    const double ci = comp == 0 ? xi : (comp == 1 ? yi : zi);
    if (w == 0) {
        if (nch > 0) stage(0);
        if (nch > 1) stage(1);
    }
    __syncthreads();
    if (w < KE && nch > 0) evaluate(0);
    __syncthreads();
    for (int c = 0; c < nch; c++) {
        if (w < KE) {
            if (c + 1 < nch) evaluate(c + 1);
            if (w == 0 && c + 2 < nch) stage(c + 2);
        } else {
            // fold chunk c in j order, one component per wavefront
            const int jt = p0 + c * KPLS_C, jn = min(KPLS_C, p1 - jt);
            const double(*fb)[64] = facb[c & 1];
            const double *dc = pj[c % 3][comp];
            for (int q = 0; q < jn; q++) acc = fma(fb[q][lane], dc[q] - ci, acc);
        }
        __syncthreads();
    }
    if (w >= KE) fsum[comp][lane] = acc;
    if (do_pairs && w < 2 && valid) {
        // w = 0: ahj over pairs (p, i), p < i; w = 1: ahi over pairs (i, j)
        double hx = 0.0, hy = 0.0, hz = 0.0;
        if (w == 0) {
            const int64_t c0 = pp.colstart[i], c1 = c0 + pp.colcnt[i];
            for (int64_t c = c0; c < c1; c++) {
                const int p = pp.i1[pp.col[c]];
                const double rx = xi - pl.rh.x[p], ry = yi - pl.rh.y[p], rz = zi - pl.rh.z[p];
                const double rji2 = dot3(rx, ry, rz, rx, ry, rz);
                const double rs = pl.R[p] + Ri;
                if (rji2 > rs * rs) {
                    const double fac = pl.Gm[p] * (1.0 / (rji2 * sqrt(rji2)));
                    hx = fma(-fac, rx, hx);
                    hy = fma(-fac, ry, hy);
                    hz = fma(-fac, rz, hz);
                }
            }
        } else {
            const int64_t r0 = pp.rowstart[i], r1 = r0 + pp.rowcnt[i];
            for (int64_t k = r0; k < r1; k++) {
                const int q = pp.i2[k];
                const double rx = pl.rh.x[q] - xi, ry = pl.rh.y[q] - yi, rz = pl.rh.z[q] - zi;
                const double rji2 = dot3(rx, ry, rz, rx, ry, rz);
                const double rs = Ri + pl.R[q];
                if (rji2 > rs * rs) {
                    const double fac = pl.Gm[q] * (1.0 / (rji2 * sqrt(rji2)));
                    hx = fma(fac, rx, hx);
                    hy = fma(fac, ry, hy);
                    hz = fma(fac, rz, hz);
                }
            }
        }
        hpart[w][0][lane] = hx;
        hpart[w][1][lane] = hy;
        hpart[w][2][lane] = hz;
    }
    __syncthreads();
    if (w != KE || !valid) return;
    double ax = fsum[0][lane], ay = fsum[1][lane], az = fsum[2][lane];
    if (do_pairs) {
        ax = ax - ((0.0 + hpart[1][0][lane]) + hpart[0][0][lane]);
        ay = ay - ((0.0 + hpart[1][1][lane]) + hpart[0][1][lane]);
        az = az - ((0.0 + hpart[1][2][lane]) + hpart[0][2][lane]);
    }
    Vec3p rb = lbeg ? pl.rbeg : pl.rend;
    rb.x[i] = xi;
    rb.y[i] = yi;
    rb.z[i] = zi;
    if (pl_active(pl, i)) {
        pl.vb.x[i] = fma(ax, dt, pl.vb.x[i]);
        pl.vb.y[i] = fma(ay, dt, pl.vb.y[i]);
        pl.vb.z[i] = fma(az, dt, pl.vb.z[i]);
    }
}

// ---------------------------------------------------------------------------
// Fast pair mode (SWG_PAIR_FAST): the same sums in the same j order, with the
// pair factor from the hardware reciprocal square root (gm_over_r3_fast,
// within a few ulp of the IEEE factor).  The partners' positions, masses and
// radii are read at wave-uniform indices through a constant-address view:
// the loads go through the scalar data cache into SGPRs that every lane of
// the wavefront reads, so no LDS staging, no workgroup barrier in the loop,
// and every VALU slot goes to the pair arithmetic (13 operations, one of
// them quarter-rate, and 7 of the factor).
// ---------------------------------------------------------------------------

// Massive bodies: one tile of KPL_FAST_TILE bodies of one system per
// workgroup of K wavefronts.  Wavefront w sums body i's row over its share of
// the partners, j in [p0 + w L, p0 + (w+1) L) with L a multiple of 4, and
// takes every K-th entry of the body's encounter-pair walks; the K partial
// accelerations are added in wavefront order through LDS.  K wavefronts per
// 64 bodies give a 32768-body system 4096 wavefronts (4 per SIMD at K = 8)
// where one lane per body gives 512.
template <int K>
__global__ __launch_bounds__(64 * K) void k_kick_pl_fast(PlDev pl, SysDev sy, ListDev pp, const Tile *tiles,
                                                         double dt, int lbeg, int use_radius, int do_pairs)
{
    static_assert(KPL_FAST_TILE == 64, "one lane per body in each wavefront");
    __shared__ double part[K][3][64];
    const Tile tl = tiles[blockIdx.x];
    const int p0 = sy.pl_off[tl.s], p1 = sy.pl_off[tl.s + 1];
    const int lane = (int)(threadIdx.x & 63u);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int i = tl.b0 + lane;
    const bool valid = i < tl.b1;
    double xi = 0.0, yi = 0.0, zi = 0.0, Ri = 0.0;
    if (valid) {
        xi = pl.rh.x[i];
        yi = pl.rh.y[i];
        zi = pl.rh.z[i];
        Ri = pl.R[i];
    }
    const cdouble *X = cview(pl.rh.x), *Y = cview(pl.rh.y), *Z = cview(pl.rh.z), *G = cview(pl.Gm),
                  *RR = cview(pl.R);
    const FastConst fc;
    const int n = p1 - p0;
    const int L = ((n + K - 1) / K + 3) & ~3;
    const int j0 = min(p1, p0 + w * L), j1 = min(p1, j0 + L);
    double ax = 0.0, ay = 0.0, az = 0.0;
    int j = j0;
    for (; j + 4 <= j1; j += 4) {
        // the four partners' data first, unconditionally, so that each
        // array's four values come in one scalar load
        double xs[4], ys[4], zs[4], gs[4], rr[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            xs[u] = X[j + u];
            ys[u] = Y[j + u];
            zs[u] = Z[j + u];
            gs[u] = G[j + u];
            rr[u] = RR[j + u];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const double rx = xs[u] - xi, ry = ys[u] - yi, rz = zs[u] - zi;
            const double r2 = dot3(rx, ry, rz, rx, ry, rz);
            const double rs = Ri + rr[u];
            // a self pair has r2 = 0, so the radius test leaves it out too
            const bool take = use_radius ? (r2 > rs * rs) : (j + u != i);
            const double f = take ? gm_over_r3_fast(gs[u], r2, fc.c15, fc.c1875) : 0.0;
            ax = fma(f, rx, ax);
            ay = fma(f, ry, ay);
            az = fma(f, rz, az);
        }
    }
    for (; j < j1; j++) {
        const double rx = X[j] - xi, ry = Y[j] - yi, rz = Z[j] - zi;
        const double r2 = dot3(rx, ry, rz, rx, ry, rz);
        const double rs = Ri + RR[j];
        const bool take = use_radius ? (r2 > rs * rs) : (j != i);
        const double f = take ? gm_over_r3_fast(G[j], r2, fc.c15, fc.c1875) : 0.0;
        ax = fma(f, rx, ax);
        ay = fma(f, ry, ay);
        az = fma(f, rz, az);
    }
    if (valid && do_pairs) {
        // this wavefront's share of the encounter pairs removed again
        // (symba_kick.f90:61-70)
        double hx = 0.0, hy = 0.0, hz = 0.0;
        const int64_t c0 = pp.colstart[i], c1 = c0 + pp.colcnt[i];
        for (int64_t c = c0 + w; c < c1; c += K) {  // pairs (p, i), p < i
            const int p = pp.i1[pp.col[c]];
            const double rx = xi - pl.rh.x[p], ry = yi - pl.rh.y[p], rz = zi - pl.rh.z[p];
            const double r2 = dot3(rx, ry, rz, rx, ry, rz);
            const double rs = pl.R[p] + Ri;
            if (r2 > rs * rs) {
                const double f = gm_over_r3_fast(pl.Gm[p], r2);
                hx = fma(-f, rx, hx);
                hy = fma(-f, ry, hy);
                hz = fma(-f, rz, hz);
            }
        }
        const int64_t r0 = pp.rowstart[i], r1 = r0 + pp.rowcnt[i];
        for (int64_t k = r0 + w; k < r1; k += K) {  // pairs (i, j), j > i
            const int q = pp.i2[k];
            const double rx = pl.rh.x[q] - xi, ry = pl.rh.y[q] - yi, rz = pl.rh.z[q] - zi;
            const double r2 = dot3(rx, ry, rz, rx, ry, rz);
            const double rs = Ri + pl.R[q];
            if (r2 > rs * rs) {
                const double f = gm_over_r3_fast(pl.Gm[q], r2);
                hx = fma(f, rx, hx);
                hy = fma(f, ry, hy);
                hz = fma(f, rz, hz);
            }
        }
        ax = ax - hx;
        ay = ay - hy;
        az = az - hz;
    }
    part[w][0][lane] = ax;
    part[w][1][lane] = ay;
    part[w][2][lane] = az;
    __syncthreads();
    if (w != 0 || !valid) return;
    ax = part[0][0][lane];
    ay = part[0][1][lane];
    az = part[0][2][lane];
#pragma unroll
    for (int q = 1; q < K; q++) {
        ax = ax + part[q][0][lane];
        ay = ay + part[q][1][lane];
        az = az + part[q][2][lane];
    }
    Vec3p rb = lbeg ? pl.rbeg : pl.rend;
    rb.x[i] = xi;
    rb.y[i] = yi;
    rb.z[i] = zi;
    if (pl_active(pl, i)) {
        pl.vb.x[i] = fma(ax, dt, pl.vb.x[i]);
        pl.vb.y[i] = fma(ay, dt, pl.vb.y[i]);
        pl.vb.z[i] = fma(az, dt, pl.vb.z[i]);
    }
}

// What a step does to particle j before its first half kick (phase TP_PRE) and
// after its second (TP_POST): part of the kicks, on the kick's lane, in place of
// two launches that pass over the particles again (3.7 us each for 20000; with
// the sums' updates, both drifts in one launch and no reset, a HELIO step is
// seven launches in place of fifteen: five driver steps of a small system 904 ->
// 786 us).
// Before: vb = vh - ptbeg when lfirst (swiftest_util.f90:398-421), then
// rh += ptbeg*dt (helio_drift.f90:166-200).
__device__ inline void tp_pre(const TpDev &tp, const SysDev &sy, int s, int j, double dth)
{
    const double px = sy.ptbeg[3 * s], py = sy.ptbeg[3 * s + 1], pz = sy.ptbeg[3 * s + 2];
    if (sy.lfirst[s]) {
        tp.vb.x[j] = tp.vh.x[j] + (-px);
        tp.vb.y[j] = tp.vh.y[j] + (-py);
        tp.vb.z[j] = tp.vh.z[j] + (-pz);
    }
    tp.rh.x[j] = fma(px, dth, tp.rh.x[j]);
    tp.rh.y[j] = fma(py, dth, tp.rh.y[j]);
    tp.rh.z[j] = fma(pz, dth, tp.rh.z[j]);
}
// After: rh += ptend*dt, vh = vb + ptend (vb2vh with vbcb = -ptend)
__device__ inline void tp_post(const TpDev &tp, const SysDev &sy, int s, int j, double dth)
{
    const double px = sy.ptend[3 * s], py = sy.ptend[3 * s + 1], pz = sy.ptend[3 * s + 2];
    tp.rh.x[j] = fma(px, dth, tp.rh.x[j]);
    tp.rh.y[j] = fma(py, dth, tp.rh.y[j]);
    tp.rh.z[j] = fma(pz, dth, tp.rh.z[j]);
    tp.vh.x[j] = tp.vb.x[j] - (-px);
    tp.vh.y[j] = tp.vb.y[j] - (-py);
    tp.vh.z[j] = tp.vb.z[j] - (-pz);
}

// Test particles: one lane per particle, the massive bodies at wave-uniform
// indices, four per iteration.
template <int BLK>
__global__ __launch_bounds__(BLK) void k_kick_tp_fast(TpDev tp, PlDev pl, SysDev sy, ListDev pt, const Tile *tiles,
                                                      double dt, int lbeg, int do_pairs, int phase)
{
    const Tile tl = tiles[blockIdx.x];
    const int p0 = sy.pl_off[tl.s], p1 = sy.pl_off[tl.s + 1];
    const int j = tl.b0 + (int)threadIdx.x;
    const bool valid = (j < tl.b1) && tp_active(tp, j);
    if (phase == TP_PRE && valid) tp_pre(tp, sy, tl.s, j, dt);
    const Vec3p rp = lbeg ? pl.rbeg : pl.rend;
    double xt = 0.0, yt = 0.0, zt = 0.0;
    if (valid) {
        xt = tp.rh.x[j];
        yt = tp.rh.y[j];
        zt = tp.rh.z[j];
    }
    const cdouble *X = cview(rp.x), *Y = cview(rp.y), *Z = cview(rp.z), *G = cview(pl.Gm);
    const FastConst fc;
    double px = 0.0, py = 0.0, pz = 0.0;
    int q = p0;
    if (q + 4 <= p1) {
        // the next four partners are loaded while the current four are
        // applied, so the scalar loads' latency hides behind the arithmetic;
        // the last batch reloads itself (index clamped to p1 - 4 >= q)
        double cx[4], cy[4], cz[4], cg[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            cx[u] = X[q + u];
            cy[u] = Y[q + u];
            cz[u] = Z[q + u];
            cg[u] = G[q + u];
        }
        for (; q + 4 <= p1; q += 4) {
            const int qn = min(q + 4, p1 - 4);
            double nx[4], ny[4], nz[4], ng[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                nx[u] = X[qn + u];
                ny[u] = Y[qn + u];
                nz[u] = Z[qn + u];
                ng[u] = G[qn + u];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const double rx = xt - cx[u], ry = yt - cy[u], rz = zt - cz[u];
                const double f = gm_over_r3_fast(cg[u], dot3(rx, ry, rz, rx, ry, rz), fc.c15, fc.c1875);
                px = fma(-f, rx, px);
                py = fma(-f, ry, py);
                pz = fma(-f, rz, pz);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                cx[u] = nx[u];
                cy[u] = ny[u];
                cz[u] = nz[u];
                cg[u] = ng[u];
            }
        }
    }
    for (; q < p1; q++) {
        const double rx = xt - X[q], ry = yt - Y[q], rz = zt - Z[q];
        const double f = gm_over_r3_fast(G[q], dot3(rx, ry, rz, rx, ry, rz), fc.c15, fc.c1875);
        px = fma(-f, rx, px);
        py = fma(-f, ry, py);
        pz = fma(-f, rz, pz);
    }
    if (!valid) return;
    double ax = 0.0 + px, ay = 0.0 + py, az = 0.0 + pz;
    if (do_pairs) {
        const int64_t c0 = pt.colstart[j], c1 = c0 + pt.colcnt[j];
        for (int64_t c = c0; c < c1; c++) {
            const int i = pt.i1[pt.col[c]];
            const double dx = xt - rp.x[i], dy = yt - rp.y[i], dz = zt - rp.z[i];
            const double f = gm_over_r3_fast(pl.Gm[i], dot3(dx, dy, dz, dx, dy, dz));
            ax = fma(f, dx, ax);
            ay = fma(f, dy, ay);
            az = fma(f, dz, az);
        }
    }
    tp.vb.x[j] = fma(ax, dt, tp.vb.x[j]);
    tp.vb.y[j] = fma(ay, dt, tp.vb.y[j]);
    tp.vb.z[j] = fma(az, dt, tp.vb.z[j]);
    if (phase == TP_POST) tp_post(tp, sy, tl.s, j, dt);
}

// Danby drift of the masked bodies (helio_drift_body, helio_drift.f90:14-54,
// with the SyMBA level mask of symba_drift.f90:14-61): mu = GM_cb, (rh, vb).
// The massive bodies take the first pl_blocks workgroups, the particles the
// others: one launch for both.
__global__ __launch_bounds__(256) void k_drift(DriftSet pl, DriftSet tp, int pl_blocks, SysDev sy, double dt, int irec,
                                               int use_level)
{
    const bool is_tp = (int)blockIdx.x >= pl_blocks;
    const DriftSet &d = is_tp ? tp : pl;
    const int i = ((int)blockIdx.x - (is_tp ? pl_blocks : 0)) * blockDim.x + threadIdx.x;
    if (i >= d.n) return;
    const Vec3p r = d.r, v = d.v;
    int st = d.status[i];
    bool m = is_tp ? (st == ACTIVE) : (st != INACTIVE);
    if (use_level) m = m && (d.levelg[i] == irec);
    if (!m) return;
    int s = d.sys[i];
    if (sy.frozen[s]) return;
    double rx = r.x[i], ry = r.y[i], rz = r.z[i], vx = v.x[i], vy = v.y[i], vz = v.z[i];
    int fl = drift_one(sy.GMcb[s], rx, ry, rz, vx, vy, vz, dt);
    r.x[i] = rx;
    r.y[i] = ry;
    r.z[i] = rz;
    v.x[i] = vx;
    v.y[i] = vy;
    v.z[i] = vz;
    if (fl != 0) {
        d.status[i] = DISCARDED_DRIFTERR;
        if (!is_tp) atomicOr(&sy.err[s], 2);
    }
}

// Test-particle half kick (helio_kick_vb_tp, helio_kick.f90:135-169):
//   p = sum over pl j ascending of -Gm_j (r_t - r_j)/|.|^3 at pl rbeg/rend,
//       started from zero and added to ah = 0 once (the OpenMP reduction of
//       swiftest_kick.f90:394-411);
//   ah += Gm_i dx/|dx|^3 for the particle's listed encounter pairs in list
//       order (symba_kick.f90:106-119);  vb += ah*dt.
template <int BLK>
__global__ __launch_bounds__(BLK) void k_kick_tp(TpDev tp, PlDev pl, SysDev sy, ListDev pt, const Tile *tiles,
                                                 double dt, int lbeg, int do_pairs, int phase)
{
    __shared__ double sx[BLK], syy[BLK], sz[BLK], sgm[BLK];
    const Tile tl = tiles[blockIdx.x];
    const int p0 = sy.pl_off[tl.s], p1 = sy.pl_off[tl.s + 1];
    const int j = tl.b0 + (int)threadIdx.x;
    const bool valid = (j < tl.b1) && tp_active(tp, j);
    if (phase == TP_PRE && valid) tp_pre(tp, sy, tl.s, j, dt);
    const Vec3p rp = lbeg ? pl.rbeg : pl.rend;
    double xt = 0.0, yt = 0.0, zt = 0.0;
    if (valid) {
        xt = tp.rh.x[j];
        yt = tp.rh.y[j];
        zt = tp.rh.z[j];
    }
    double px = 0.0, py = 0.0, pz = 0.0;
    for (int it = p0; it < p1; it += BLK) {
        int q0 = it + (int)threadIdx.x;
        bool gok = true;
        if (q0 < p1) {
            sx[threadIdx.x] = rp.x[q0];
            syy[threadIdx.x] = rp.y[q0];
            sz[threadIdx.x] = rp.z[q0];
            sgm[threadIdx.x] = pl.Gm[q0];
            gok = pair_g_ok(pl.Gm[q0]);
        }
        const bool tile_gok = __syncthreads_and(gok);
        const int qn = min(BLK, p1 - it);
        if (valid) {
            // Whole groups of KTP_G bodies: the factors are formed without
            // branches (exact cores; the rare out-of-range terms redone with
            // the IEEE operations under a wave-uniform test) and folded in
            // j order.  The tail of a partial tile takes the plain path.
            int q = 0;
            for (; q + KTP_G <= qn; q += KTP_G) {
                double rx[KTP_G], ry[KTP_G], rz[KTP_G], r2[KTP_G], fac[KTP_G];
                bool need[KTP_G];
                bool any_need = false;
#pragma unroll
                for (int u = 0; u < KTP_G; u++) {
                    rx[u] = xt - sx[q + u];
                    ry[u] = yt - syy[q + u];
                    rz[u] = zt - sz[q + u];
                    r2[u] = dot3(rx[u], ry[u], rz[u], rx[u], ry[u], rz[u]);
                    fac[u] = div_core(sgm[q + u], r2[u] * sqrt_core(r2[u]));
                    need[u] = !(tile_gok & (r2[u] >= PAIR_R2_LO) & (r2[u] <= PAIR_R2_HI));
                    any_need = any_need | need[u];
                }
                if (__ballot(any_need)) {
#pragma unroll
                    for (int u = 0; u < KTP_G; u++)
                        if (need[u]) fac[u] = sgm[q + u] / (r2[u] * sqrt(r2[u]));
                }
#pragma unroll
                for (int u = 0; u < KTP_G; u++) {
                    px = fma(-fac[u], rx[u], px);
                    py = fma(-fac[u], ry[u], py);
                    pz = fma(-fac[u], rz[u], pz);
                }
            }
            for (; q < qn; q++) {
                double rx = xt - sx[q], ry = yt - syy[q], rz = zt - sz[q];
                double rji2 = dot3(rx, ry, rz, rx, ry, rz);
                double fac = gm_over_r3(sgm[q], rji2, tile_gok);
                px = fma(-fac, rx, px);
                py = fma(-fac, ry, py);
                pz = fma(-fac, rz, pz);
            }
        }
        __syncthreads();
    }
    if (!valid) return;
    double ax = 0.0 + px, ay = 0.0 + py, az = 0.0 + pz;
    if (do_pairs) {
        const int64_t c0 = pt.colstart[j], c1 = c0 + pt.colcnt[j];
        for (int64_t c = c0; c < c1; c++) {
            int i = pt.i1[pt.col[c]];
            double dx = xt - rp.x[i], dy = yt - rp.y[i], dz = zt - rp.z[i];
            double rjj = dot3(dx, dy, dz, dx, dy, dz);
            double fac = pl.Gm[i] / (rjj * sqrt(rjj));
            ax = fma(fac, dx, ax);
            ay = fma(fac, dy, ay);
            az = fma(fac, dz, az);
        }
    }
    tp.vb.x[j] = fma(ax, dt, tp.vb.x[j]);
    tp.vb.y[j] = fma(ay, dt, tp.vb.y[j]);
    tp.vb.z[j] = fma(az, dt, tp.vb.z[j]);
    if (phase == TP_POST) tp_post(tp, sy, tl.s, j, dt);
}

// rh += ptend*dt (masked); vh = vb - cb%vb (all bodies)
__device__ inline void pl_end_one(const PlDev &pl, int i, const double *cb, const double *pt, double dth)
{
    if (pl_active(pl, i)) {
        pl.rh.x[i] = fma(pt[0], dth, pl.rh.x[i]);
        pl.rh.y[i] = fma(pt[1], dth, pl.rh.y[i]);
        pl.rh.z[i] = fma(pt[2], dth, pl.rh.z[i]);
    }
    pl.vh.x[i] = pl.vb.x[i] - cb[0];
    pl.vh.y[i] = pl.vb.y[i] - cb[1];
    pl.vh.z[i] = pl.vb.z[i] - cb[2];
}

// Per-system sums at the end of a step:
//   lindrift pt = sum_masked(Gm vb) / GM_cb -> ptend (forward, lanes 0-2)
//   vb->vh (swiftest_util.f90:363-395): cb%vb -= Gm vb / GM_cb over
//   i = npl..1, active only (backward, lanes 3-5): the two walk the bodies
//   from both ends side by side
// With apply the workgroup goes on to its bodies what k_pl_end_apply does.
// lfirst: the HELIO branch clears it after its vh->vb; the encounter branch
// keeps it (helio_step.f90:58-61 vs symba_step.f90:81, then symba_step.f90:47);
// nothing of a step reads it after this.
__global__ __launch_bounds__(SUM_T) void k_sums_end(PlDev pl, SysDev sy, int nsys, double dth, int apply)
{
    __shared__ SumStage S;
    __shared__ double sv[6];
    const int s = blockIdx.x, tid = threadIdx.x;
    const int p0 = sy.pl_off[s], p1 = sy.pl_off[s + 1];
    if (sy.frozen[s]) return;
    if (tid == 0 && sy.lfirst[s] && !(sy.enc_pp[s] || sy.enc_pt[s])) sy.lfirst[s] = 0;
    if (p1 == p0) return;
    const double gm = sy.GMcb[s];
    double acc = 0.0;
    sums_chunks<true>(
        pl, pl.vb, p0, p1,
        [&](int b, int k, const SumBody &q, const SumBody &r) {
            S.t[b][0][k] = q.act ? q.g * q.x : 0.0;
            S.t[b][1][k] = q.act ? q.g * q.y : 0.0;
            S.t[b][2][k] = q.act ? q.g * q.z : 0.0;
            S.t[b][3][k] = r.act ? -((r.g * r.x) / gm) : 0.0;
            S.t[b][4][k] = r.act ? -((r.g * r.y) / gm) : 0.0;
            S.t[b][5][k] = r.act ? -((r.g * r.z) / gm) : 0.0;
        },
        [&](int b, int n) {
            if (tid < 6) acc = chain(acc, S.t[b][tid], n);
        });
    if (tid < 3) sv[tid] = sy.ptend[3 * s + tid] = acc / gm;
    else if (tid < 6) sv[tid] = sy.cbvb[3 * s + tid - 3] = acc;
    if (!apply) return;
    __syncthreads();
    const double p[3] = {sv[0], sv[1], sv[2]}, cb[3] = {sv[3], sv[4], sv[5]};
    for (int i = p0 + tid; i < p1; i += SUM_T) pl_end_one(pl, i, cb, p, dth);
}

__global__ void k_pl_end_apply(PlDev pl, SysDev sy, int npl, double dth)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npl) return;
    int s = pl.sys[i];
    if (sy.frozen[s]) return;
    pl_end_one(pl, i, sy.cbvb + 3 * s, sy.ptend + 3 * s, dth);
}

// Snapshot coordinate refresh (swiftest_util.f90:2663-2682): pl vh->vb, then
// tp vb = vh - ptbeg for active particles.
__global__ void k_snapshot_tp(TpDev tp, SysDev sy, int ntp)
{
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= ntp || !tp_active(tp, j)) return;
    int s = tp.sys[j];
    if (sy.frozen[s]) return;
    tp.vb.x[j] = tp.vh.x[j] + (-sy.ptbeg[3 * s]);
    tp.vb.y[j] = tp.vh.y[j] + (-sy.ptbeg[3 * s + 1]);
    tp.vb.z[j] = tp.vh.z[j] + (-sy.ptbeg[3 * s + 2]);
}

__global__ __launch_bounds__(SUM_T) void k_vh2vb_sum(PlDev pl, SysDev sy, int nsys)
{
    __shared__ SumStage S;
    __shared__ double shr[4];
    const int s = blockIdx.x, tid = threadIdx.x;
    const int p0 = sy.pl_off[s], p1 = sy.pl_off[s + 1];
    if (p1 == p0 || sy.frozen[s]) return;
    const double acc = sums_gm_vh(S, pl, p0, p1);
    if (tid < 4) shr[tid] = acc;
    __syncthreads();
    if (tid < 3) sy.cbvb[3 * s + tid] = shr[tid + 1] / (sy.GMcb[s] + shr[0]);
}

__global__ void k_vh2vb_apply(PlDev pl, SysDev sy, int npl)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npl) return;
    int s = pl.sys[i];
    if (sy.frozen[s]) return;
    pl.vb.x[i] = pl.vh.x[i] + sy.cbvb[3 * s];
    pl.vb.y[i] = pl.vh.y[i] + sy.cbvb[3 * s + 1];
    pl.vb.z[i] = pl.vh.z[i] + sy.cbvb[3 * s + 2];
}

// The initialize sequence of one system loaded into slot s of a running
// ensemble (the per-system part of k_vh2vb_sum, k_vh2vb_apply and
// k_init_tp_vb): cb%vb from vh over the slot's bodies, vb = vh + cb%vb for its
// massive bodies and test particles.  Padding bodies have Gm = 0 and vh = 0,
// so they add exactly nothing to the sums.  One workgroup.
__global__ __launch_bounds__(SUM_T) void k_init_one(PlDev pl, TpDev tp, SysDev sy, int s)
{
    __shared__ SumStage S;
    __shared__ double shr[4];
    const int tid = threadIdx.x;
    const int p0 = sy.pl_off[s], p1 = sy.pl_off[s + 1];
    const double acc = sums_gm_vh(S, pl, p0, p1);
    if (tid < 4) shr[tid] = acc;
    __syncthreads();
    if (tid < 3) sy.cbvb[3 * s + tid] = p1 > p0 ? shr[tid + 1] / (sy.GMcb[s] + shr[0]) : 0.0;
    __syncthreads();
    const double cx = sy.cbvb[3 * s], cy = sy.cbvb[3 * s + 1], cz = sy.cbvb[3 * s + 2];
    for (int i = p0 + tid; i < p1; i += SUM_T) {
        pl.vb.x[i] = pl.vh.x[i] + cx;
        pl.vb.y[i] = pl.vh.y[i] + cy;
        pl.vb.z[i] = pl.vh.z[i] + cz;
    }
    for (int j = sy.tp_off[s] + tid; j < sy.tp_off[s + 1]; j += SUM_T) {
        tp.vb.x[j] = tp.vh.x[j] + cx;
        tp.vb.y[j] = tp.vh.y[j] + cy;
        tp.vb.z[j] = tp.vh.z[j] + cz;
    }
}

// Initialization (helio_util.f90:26-28): tp vb = vh + cb%vb
__global__ void k_init_tp_vb(TpDev tp, SysDev sy, int ntp)
{
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= ntp) return;
    int s = tp.sys[j];
    tp.vb.x[j] = tp.vh.x[j] + sy.cbvb[3 * s];
    tp.vb.y[j] = tp.vh.y[j] + sy.cbvb[3 * s + 1];
    tp.vb.z[j] = tp.vh.z[j] + sy.cbvb[3 * s + 2];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
void launch_copy_list(hipStream_t st, const CopyList &c)
{
    int64_t n = 0;
    for (int i = 0; i < c.n; i++) n = std::max(n, c.item[i].n);
    if (n) k_copy_list<<<dim3((unsigned)std::min<int64_t>((n + 255) / 256, 256), c.n), 256, 0, st>>>(c);
}
void launch_reset_levels(hipStream_t st, PlDev pl, TpDev tp, SysDev sy, int32_t *sub_stats, int npl, int ntp, int nsys)
{
    const int n = std::max(std::max(npl, ntp), std::max(nsys, 4));
    k_reset_levels<<<cdiv(n, 256), 256, 0, st>>>(pl, tp, sy, sub_stats, npl, ntp, nsys);
}
// max_npl: the largest system's bodies.  Up to SUM_APPLY the sums' workgroup
// updates its bodies itself.
void launch_sums_begin(hipStream_t st, PlDev pl, SysDev sy, int nsys, int npl, int max_npl, double dth, int force)
{
    const int apply = max_npl <= SUM_APPLY;
    k_sums_begin<<<nsys, SUM_T, 0, st>>>(pl, sy, nsys, force, dth, apply);
    if (npl && !apply) k_pl_begin_apply<<<cdiv(npl, 256), 256, 0, st>>>(pl, sy, npl, dth, force);
}
void launch_kick_pl(hipStream_t st, const Tuning &tu, PlDev pl, SysDev sy, ListDev pp, const Tile *tiles,
                    int ntiles, double dt, int lbeg, int use_radius, int do_pairs)
{
    if (!ntiles) return;
    if (tu.any_tiny) {
        // the registers of two sets of terms ahead, which this kernel needs for
        // its two copies of the sums and not to read ahead (two / one, us, with
        // 30 % of the bodies semi-interacting and with 80 %: 200 bodies 9.5 /
        // 12.4 and 13.7 / 15.1, 5000 115 / 198 and 205 / 243, 32768 2857 / 4651
        // and 1488 / 1916; 256 systems of 40 to 320 55 / 64 and 49 / 52)
        const auto kern = tu.pair_fast ? k_kick_pl_rows<RW_SMALL, 4, 2, true, true> : k_kick_pl_rows<RW_SMALL, 4, 2, true, false>;
        kern<<<ntiles, RowsLds<RW_SMALL, 4>::THREADS, 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs);
        return;
    }
    if (tu.pair_fast) {
        switch (tu.kick_pl_split) {
        case 1: k_kick_pl_fast<1><<<ntiles, 64, 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs); break;
        case 2: k_kick_pl_fast<2><<<ntiles, 128, 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs); break;
        case 4: k_kick_pl_fast<4><<<ntiles, 256, 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs); break;
        case 16: k_kick_pl_fast<16><<<ntiles, 1024, 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs); break;
        default: k_kick_pl_fast<8><<<ntiles, 512, 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs); break;
        }
        return;
    }
    if (tu.kick_pl_eval) {
        if (tu.kick_pl_eval == KPL_BODIES)
            k_kick_pl_split<<<ntiles, 64 * (KPLS_KE + 3), 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs);
        else if (tu.kick_pl_eval == KPL_ROWS_LARGE)
            k_kick_pl_rows<RW_LARGE, 8, 1, false, false><<<ntiles, RowsLds<RW_LARGE, 8>::THREADS, 0, st>>>(
                pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs);
        else if (ntiles <= RW_FEW)
            k_kick_pl_rows<RW_SMALL, 4, 2, false, false><<<ntiles, RowsLds<RW_SMALL, 4>::THREADS, 0, st>>>(
                pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs);
        else
            k_kick_pl_rows<RW_SMALL, 4, 1, false, false><<<ntiles, RowsLds<RW_SMALL, 4>::THREADS, 0, st>>>(
                pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs);
        return;
    }
    switch (tu.kick_pl_block) {
    case 64: k_kick_pl<64><<<ntiles, 64, 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs); break;
    case 128: k_kick_pl<128><<<ntiles, 128, 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs); break;
    default: k_kick_pl<256><<<ntiles, 256, 0, st>>>(pl, sy, pp, tiles, dt, lbeg, use_radius, do_pairs); break;
    }
}
void launch_drift(hipStream_t st, const DriftSet &pl, const DriftSet &tp, SysDev sy, double dt, int irec, int use_level)
{
    const int pb = cdiv(pl.n, 128), tb = cdiv(tp.n, 128);
    if (pb + tb) k_drift<<<pb + tb, 128, 0, st>>>(pl, tp, pb, sy, dt, irec, use_level);
}
void launch_kick_tp(hipStream_t st, const Tuning &tu, TpDev tp, PlDev pl, SysDev sy, ListDev pt,
                    const Tile *tiles, int ntiles, double dt, int lbeg, int do_pairs, int phase)
{
    if (!ntiles) return;
    if (tu.pair_fast) {
        switch (tu.kick_tp_block) {
        case 64: k_kick_tp_fast<64><<<ntiles, 64, 0, st>>>(tp, pl, sy, pt, tiles, dt, lbeg, do_pairs, phase); break;
        case 128: k_kick_tp_fast<128><<<ntiles, 128, 0, st>>>(tp, pl, sy, pt, tiles, dt, lbeg, do_pairs, phase); break;
        default: k_kick_tp_fast<256><<<ntiles, 256, 0, st>>>(tp, pl, sy, pt, tiles, dt, lbeg, do_pairs, phase); break;
        }
        return;
    }
    switch (tu.kick_tp_block) {
    case 64: k_kick_tp<64><<<ntiles, 64, 0, st>>>(tp, pl, sy, pt, tiles, dt, lbeg, do_pairs, phase); break;
    case 128: k_kick_tp<128><<<ntiles, 128, 0, st>>>(tp, pl, sy, pt, tiles, dt, lbeg, do_pairs, phase); break;
    default: k_kick_tp<256><<<ntiles, 256, 0, st>>>(tp, pl, sy, pt, tiles, dt, lbeg, do_pairs, phase); break;
    }
}
void launch_sums_end(hipStream_t st, PlDev pl, SysDev sy, int nsys, int npl, int max_npl, double dth)
{
    const int apply = max_npl <= SUM_APPLY;
    k_sums_end<<<nsys, SUM_T, 0, st>>>(pl, sy, nsys, dth, apply);
    if (npl && !apply) k_pl_end_apply<<<cdiv(npl, 256), 256, 0, st>>>(pl, sy, npl, dth);
}
void launch_snapshot(hipStream_t st, PlDev pl, TpDev tp, SysDev sy, int nsys, int npl, int ntp)
{
    k_vh2vb_sum<<<nsys, SUM_T, 0, st>>>(pl, sy, nsys);
    if (npl) k_vh2vb_apply<<<cdiv(npl, 256), 256, 0, st>>>(pl, sy, npl);
    if (ntp) k_snapshot_tp<<<cdiv(ntp, 256), 256, 0, st>>>(tp, sy, ntp);
}
void launch_vh2vb(hipStream_t st, PlDev pl, SysDev sy, int nsys, int npl)
{
    k_vh2vb_sum<<<nsys, SUM_T, 0, st>>>(pl, sy, nsys);
    if (npl) k_vh2vb_apply<<<cdiv(npl, 256), 256, 0, st>>>(pl, sy, npl);
}
void launch_init_one(hipStream_t st, PlDev pl, TpDev tp, SysDev sy, int s)
{
    k_init_one<<<1, SUM_T, 0, st>>>(pl, tp, sy, s);
}
void launch_init_tp_vb(hipStream_t st, TpDev tp, SysDev sy, int ntp)
{
    if (ntp) k_init_tp_vb<<<cdiv(ntp, 256), 256, 0, st>>>(tp, sy, ntp);
}

}  // namespace swg
