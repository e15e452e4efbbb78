// nxt.hip -- the routines that close a time step around the hot path:
// horizontal divergence (DYN/divhor.F90), sea-level prediction, vertical
// velocity and sea-level swap (DYN/sshwzv.F90), the tracer and momentum
// Asselin filters and swaps (TRA/tranxt.F90, DYN/dynnxt.F90), for the linear
// free surface (e3 fixed in time).
//
// All of them are HBM-bound streams of a few fields.  Arithmetic is done in
// FP64 and rounded once on store, so the FP64 form repeats the reference's
// operations and the FP32 storage form loses nothing beyond its storage
// rounding.
//
// lbc_lnk is folded into the kernels.  A read-only input (un, vn for the
// divergence) lets a ring point compute its value at its lbc source point.
// The tracers, updated in place, are written to the ring by the thread of the
// interior source point (lbc_targets); dyn_nxt's cyclic ring columns follow in a
// second launch that reads the finished source columns.  So no thread reads a
// value another thread of the same launch overwrites.
#include "common.hpp"
#include "kernels.hpp"

// the ring points whose serial lbc_lnk source ('T', 'U' or 'V' grid) is the
// interior point (i,j): the inverse of lbc_src, at most three points
template <typename F>
__device__ __forceinline__ void lbc_targets(const DevDomain &d, int i, int j, F f)
{
    if (i != 2 && i != d.jpi - 1 && j != 2 && j != d.jpj - 1) return;
    const int ci[3] = {i, 1, d.jpi}, cj[3] = {j, 1, d.jpj};
    for (int a = 0; a < 3; a++)
        for (int b = 0; b < 3; b++) {
            if (a == 0 && b == 0) continue;
            int si, sj;
            if (lbc_src(d, 'T', ci[a], cj[b], si, sj) && si == i && sj == j) f(ci[a], cj[b]);
        }
}

// levels whose loads a closure kernel issues together, ahead of their stores:
// the compiler moves no load across a store to an array that it cannot tell
// apart, so a loop that loads and stores level by level waits for each level.
// Horizontally uniform scale factors (E3U) are scalar loads (uld); as plain loads
// they would be as many vector loads as the fields.  1024x1024x75 FP32, before
// and after both: ssh_nxt 471 -> 246 us, div_hor 389 -> 244 us, with 942 MB
// each to move.  (wzv, one load per level, gains nothing from it.)
#define NXT_KB 8
// (Scale factors that vary are as many loads again, of 8 bytes each: two levels.
// Four or eight crowd the caches, 260x230x50 FP64 44, 48 and 37 us for 4, 8 and 2;
// level by level 49.)
#define NXT_E3(p, ij, k) (E3U ? uld(p, (k) - 1) : E3(p, ij, k))

// horizontal divergence at the interior point (i,j), DYN/divhor.F90:79-83.
// The column's metrics are loaded once; levels() evaluates KB levels from
// k0 (the last one repeated beyond kmax) with the reference's operation order.
template <typename T, bool E3U>
struct HdivCol {
    static constexpr int KB = E3U ? NXT_KB : 2;
    double a1, a0, b1, b0, r;
    uint32_t ij;
    const T *un, *vn;
    __device__ __forceinline__ HdivCol(const DevDomain &d, const T *un_, const T *vn_, int i, int j) : un(un_), vn(vn_)
    {
        const Metrics<double> &m = d.md;
        ij = IJ32(i, j);
        a1 = A2(m.e2u, i, j);
        a0 = A2(m.e2u, i - 1, j);
        b1 = A2(m.e1v, i, j);
        b0 = A2(m.e1v, i, j - 1);
        r = A2(m.r1_e1e2t, i, j);
    }
    __device__ __forceinline__ void levels(const DevDomain &d, int k0, int kmax, T (&h)[KB]) const
    {
        const Metrics<double> &m = d.md;
        const uint32_t js = ij - (uint32_t)d.jpi;
        T u1[KB], u0[KB], v1[KB], v0[KB];
    #pragma unroll
        for (int q = 0; q < KB; q++) {
            const int k = min(k0 + q, kmax);
            const T *u = plane_ptr(un, d.n2, k), *v = plane_ptr(vn, d.n2, k);
            u1[q] = ldp(u, ij);
            u0[q] = ldp(u, ij - 1u);
            v1[q] = ldp(v, ij);
            v0[q] = ldp(v, js);
        }
    #pragma unroll
        for (int q = 0; q < KB; q++) {
            const int k = min(k0 + q, kmax);
            h[q] = (T)((a1 * NXT_E3(m.e3u, ij, k) * (double)u1[q] - a0 * NXT_E3(m.e3u, ij - 1u, k) * (double)u0[q] +
                        b1 * NXT_E3(m.e3v, ij, k) * (double)v1[q] - b0 * NXT_E3(m.e3v, js, k) * (double)v0[q]) *
                       r / NXT_E3(m.e3t, ij, k));
        }
    }
};

// ---------------------------------------------------------------------------
// div_hor, DYN/divhor.F90:50-110: hdivn on levels 1..jpkm1 of the interior,
// then lbc_lnk('T') of all jpk levels.  One thread per NXT_KB levels.
// ---------------------------------------------------------------------------
template <typename T, bool E3U>
struct S_div_hor {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, const T *__restrict__ un, const T *__restrict__ vn, T *__restrict__ hdivn)
    {
        THREAD_IJ_V(vb_, 1, 1);
        const int k0 = (int)vb_.z * NXT_KB + 1;
        if (i > d.jpi || j > d.jpj) return;
        int si, sj;
        const bool ok = lbc_src(d, 'T', i, j, si, sj);
        const bool ring = si != i || sj != j || !ok;
        const HdivCol<T, E3U> c(d, un, vn, ok ? si : 2, ok ? sj : 2);
        const uint32_t ij = IJ32(i, j);
        constexpr int KB = HdivCol<T, E3U>::KB;
    #pragma unroll
        for (int kb = k0; kb < k0 + NXT_KB; kb += KB) {
            T hv[KB];
            c.levels(d, min(kb, d.jpk), d.jpk, hv);
    #pragma unroll
            for (int q = 0; q < KB; q++) {
                const int k = kb + q;
                if (k > d.jpk) break;
                T *h = plane_ptr(hdivn, d.n2, k);
                if (k == d.jpk) {   // level jpk is not computed: lbc_lnk only
                    if (ring) stp(h, ij, ok ? ldp((const T *)h, c.ij) : T(0));
                } else {
                    stp(h, ij, ok ? hv[q] : T(0));
                }
            }
        }
    }
};
template <typename T, bool E3U>
KERNEL void k_div_hor(DevDomain d, const T *__restrict__ un, const T *__restrict__ vn, T *__restrict__ hdivn)
{
    S_div_hor<T, E3U>::run(vb_hw(), d, un, vn, hdivn);
}

// ---------------------------------------------------------------------------
// ssh_nxt, DYN/sshwzv.F90:56-126: div_hor, then the after sea level from the
// depth-integrated divergence.  One thread per column: the column computes
// its hdivn (at its lbc source point on the ring), the integral and ssha.
// ---------------------------------------------------------------------------
template <typename T, bool E3U>
struct S_ssh_nxt {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, double z2dt, double zcoef, const T *__restrict__ un, const T *__restrict__ vn, T *__restrict__ hdivn, const double *__restrict__ sshb, const double *__restrict__ emp_b, const double *__restrict__ emp, double *__restrict__ ssha)
    {
        THREAD_IJ_V(vb_, 1, 1);
        if (i > d.jpi || j > d.jpj) return;
        int si, sj;
        const bool ok = lbc_src(d, 'T', i, j, si, sj);
        const uint32_t ij = IJ32(i, j);
        const HdivCol<T, E3U> c(d, un, vn, ok ? si : 2, ok ? sj : 2);
        constexpr int KB = HdivCol<T, E3U>::KB;
        const int nlev = d.jpk - 1;
        double zhdiv = 0.0;
        for (int k0 = 1; k0 <= nlev; k0 += KB) {
            T hv[KB];
            double e3[E3U ? 1 : KB];
            if constexpr (!E3U) {
    #pragma unroll
                for (int q = 0; q < KB; q++) e3[q] = E3(d.md.e3t, ij, min(k0 + q, nlev));
            }
            c.levels(d, k0, nlev, hv);
    #pragma unroll
            for (int q = 0; q < KB; q++) {
                const int k = k0 + q;
                if (k > nlev) break;
                const T h = ok ? hv[q] : T(0);
                stp(plane_ptr(hdivn, d.n2, k), ij, h);
                zhdiv = zhdiv + (E3U ? uld(d.md.e3t, k - 1) : e3[E3U ? 0 : q]) * (double)h;
            }
        }
        if (si != i || sj != j || !ok) A3(hdivn, i, j, d.jpk) = ok ? A3(hdivn, si, sj, d.jpk) : T(0);
        ssha[ij] = (sshb[ij] - z2dt * (zcoef * (emp_b[ij] + emp[ij]) + zhdiv)) * SSMASK(ij);
    }
};
template <typename T, bool E3U>
KERNEL void k_ssh_nxt(DevDomain d, double z2dt, double zcoef, const T *__restrict__ un, const T *__restrict__ vn,
                      T *__restrict__ hdivn, const double *__restrict__ sshb, const double *__restrict__ emp_b,
                      const double *__restrict__ emp, double *__restrict__ ssha)
{
    S_ssh_nxt<T, E3U>::run(vb_hw(), d, z2dt, zcoef, un, vn, hdivn, sshb, emp_b, emp, ssha);
}

// ---------------------------------------------------------------------------
// wzv, DYN/sshwzv.F90:129-213 (z-star / linear free surface branch): w from
// the bottom up.  e3t_a - e3t_b is formed as the reference forms it (zero
// when the scale factors are fixed).  One thread per column.
// ---------------------------------------------------------------------------
template <typename T>
struct S_wzv {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, int first, double z1_2dt, const T *__restrict__ hdivn, T *__restrict__ wn)
    {
        THREAD_IJ_V(vb_, 1, 1);
        if (i > d.jpi || j > d.jpj) return;
        const uint32_t ij = IJ32(i, j);
        if (first) A3(wn, i, j, d.jpk) = T(0);
        double w = (double)A3(wn, i, j, d.jpk);
    #pragma unroll 4
        for (int k = d.jpk - 1; k >= 1; k--) {
            const double e3 = E3(d.md.e3t, ij, k);
            w = w - (e3 * (double)A3(hdivn, i, j, k) + z1_2dt * (e3 - e3)) * TMASK(double, i, j, k);
            A3(wn, i, j, k) = (T)w;
        }
    }
};
template <typename T>
KERNEL void k_wzv(DevDomain d, int first, double z1_2dt, const T *__restrict__ hdivn, T *__restrict__ wn)
{
    S_wzv<T>::run(vb_hw(), d, first, z1_2dt, hdivn, wn);
}

// ---------------------------------------------------------------------------
// ssh_swp, DYN/sshwzv.F90:216-267 (linear free surface)
// ---------------------------------------------------------------------------
struct S_ssh_swp {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, int euler, double atfp, double *__restrict__ sshb, double *__restrict__ sshn, const double *__restrict__ ssha)
    {
        THREAD_IJ_V(vb_, 1, 1);
        if (i > d.jpi || j > d.jpj) return;
        const uint32_t ij = IJ32(i, j);
        if (!euler) sshb[ij] = sshn[ij] + atfp * (sshb[ij] - 2 * sshn[ij] + ssha[ij]);
        sshn[ij] = ssha[ij];
    }
};
KERNEL void k_ssh_swp(DevDomain d, int euler, double atfp, double *__restrict__ sshb, double *__restrict__ sshn,
                      const double *__restrict__ ssha)
{
    S_ssh_swp::run(vb_hw(), d, euler, atfp, sshb, sshn, ssha);
}

// ---------------------------------------------------------------------------
// tra_nxt, TRA/tranxt.F90:66-192 with tra_nxt_fix, lines 195-237: lbc_lnk of
// tsa; Euler: tsn = tsa on levels 1..jpkm1; leapfrog: Asselin filter on the
// interior, then lbc_lnk of tsb, tsn, tsa.  One thread per cell and tracer
// (grid.z = jpk times the tracers).
// ---------------------------------------------------------------------------
template <typename T>
struct S_tra_nxt {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, int euler, double atfp, T *__restrict__ tsb, T *__restrict__ tsn, T *__restrict__ tsa)
    {
        THREAD_IJ_V(vb_, 1, 1);
        const int k = (int)(vb_.z % (unsigned)d.jpk) + 1;
        const size_t off = (size_t)(vb_.z / (unsigned)d.jpk) * d.n3;
        if (i > d.jpi || j > d.jpj) return;
        T *pb = tsb + off, *pn = tsn + off, *pa = tsa + off;
        if (!is_interior(d, i, j)) {
            int si, sj;
            if (lbc_src(d, 'T', i, j, si, sj)) return;   // written by the thread of (si,sj)
            A3(pa, i, j, k) = T(0);
            if (euler) {
                if (k < d.jpk) A3(pn, i, j, k) = T(0);
            } else {
                A3(pb, i, j, k) = T(0);
                A3(pn, i, j, k) = T(0);
            }
            return;
        }
        const T ta = A3(pa, i, j, k);
        T tb, tn;
        if (euler) {
            tb = A3(pb, i, j, k);   // only copied to ring points by the leapfrog branch
            tn = k < d.jpk ? ta : A3(pn, i, j, k);
            if (k < d.jpk) A3(pn, i, j, k) = tn;
        } else if (k < d.jpk) {
            const double ztn = (double)A3(pn, i, j, k);
            const double ztd = (double)ta - 2.0 * ztn + (double)A3(pb, i, j, k);
            tb = (T)(ztn + atfp * ztd);
            tn = ta;
            A3(pb, i, j, k) = tb;
            A3(pn, i, j, k) = tn;
        } else {
            tb = A3(pb, i, j, k);
            tn = A3(pn, i, j, k);
        }
        lbc_targets(d, i, j, [&](int ti, int tj) {
            A3(pa, ti, tj, k) = ta;
            if (euler) {
                if (k < d.jpk) A3(pn, ti, tj, k) = tn;
            } else {
                A3(pb, ti, tj, k) = tb;
                A3(pn, ti, tj, k) = tn;
            }
        });
    }
};
template <typename T>
KERNEL void k_tra_nxt(DevDomain d, int euler, double atfp, T *__restrict__ tsb, T *__restrict__ tsn,
                      T *__restrict__ tsa)
{
    S_tra_nxt<T>::run(vb_hw(), d, euler, atfp, tsb, tsn, tsa);
}

// ---------------------------------------------------------------------------
// dyn_nxt, DYN/dynnxt.F90:66-377 (linear free surface).  One thread per column
// and component (grid.z: u, v):
//   A  lines 111-135: with dyn_spg_ts the baroclinic ua gets the barotropic
//      after velocity (ua - depth mean + ua_b); without ln_bt_fw, un the
//      advective barotropic velocity;
//   B  lines 147-176: Euler swap or Asselin filter and swap;
//   C  lines 286-297: the forward time-splitting correction of ub, with the
//      depth mean of the filtered column; then the barotropic now and before
//      velocities (299-347).
// Bound by HBM.  Each pass needs a depth sum of the pass before, and a column
// of KMAX levels or fewer keeps ua, then the filtered ub, in registers between
// them: 12 arrays move instead of 20 (1024x1024x75 FP32: 1442 us as two
// kernels that read the columns again, 856 us).  KMAX = 0 reads them
// again, for deeper columns.
// lbc_lnk('U'/'V') of line 139: ring points without a source (closed sides) are
// columns of zeros in the same launch; the ones with a source (cyclic sides)
// follow in a launch of their own (RING), which reads the finished source.  The
// ring's columns along j are jpi points apart, a cache line per lane, and few:
// one for every NXT_RING-th lane makes a wave's accesses as many times cheaper and
// spreads them over more waves.  With one per lane their launch took 51 of the 134
// us of 362x149x46 FP64, e3 varying (88 now); of the rows along i one per lane
// (300x260x40 FP32, cyclic along j: 48 us, every 8th lane 57).
// Scale factors that vary are loaded with each KB levels' other operands: loaded
// where used, after the stores of the level before, 512x512x75 FP32 took 428 us
// (385 now).
// ---------------------------------------------------------------------------
#define NXT_RING 8
// threads for the ring's rows (with a source where the domain is cyclic along j), whole waves
__host__ __device__ inline int nxt_ring_rows(const DevDomain &d) { return d.jper ? (2 * d.jpi + 63) / 64 * 64 : 0; }
template <typename T, int KMAX, bool E3U, bool RING>
struct S_dyn_nxt {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, int spg_ts, int bt_fw, int euler, double atfp, T *ub_, T *vb, T *un_, T *vn, T *ua_, T *va, const double *__restrict__ ua_b_, const double *__restrict__ va_b, const double *__restrict__ un_adv, const double *__restrict__ vn_adv, double *__restrict__ ub_b_, double *__restrict__ vb_b, double *__restrict__ un_b_, double *__restrict__ vn_b, const double *__restrict__ r1_hu_, const double *__restrict__ r1_hv)
    {
        int i, j;
        if constexpr (RING) {
            const int t = (int)(vb_.x * NH_BLOCK + threadIdx.y * blockDim.x + threadIdx.x), nr = nxt_ring_rows(d);
            if (t < nr) {
                if (t >= 2 * d.jpi) return;
                i = t < d.jpi ? t + 1 : t - d.jpi + 1;
                j = t < d.jpi ? 1 : d.jpj;
            } else {
                if ((t - nr) % NXT_RING) return;
                const int q = (t - nr) / NXT_RING;
                i = (q & 1) ? d.jpi : 1;
                j = 2 + q / 2;
                if (j > d.jpj - 1) return;
            }
        } else {
            unsigned bx, by;
            xcd_tile_v(vb_, bx, by);
            i = (int)(bx * blockDim.x + threadIdx.x) + 1;
            j = (int)(by * blockDim.y + threadIdx.y) + 1;
            if (i > d.jpi || j > d.jpj) return;
        }
        int si, sj;
        const bool ok = lbc_src(d, 'U', i, j, si, sj);
        const bool ring = !is_interior(d, i, j);
        if (RING != (ring && ok)) return;
        const bool zero = !RING && ring;
        const bool cv = vb_.z != 0;
        T *__restrict__ ub = cv ? vb : ub_;
        T *__restrict__ un = cv ? vn : un_;
        T *__restrict__ ua = cv ? va : ua_;
        const double *e3x = cv ? d.md.e3v : d.md.e3u;
        const uint32_t ij = IJ32(i, j), src = RING ? IJ32(si, sj) : ij;
        const uint32_t w = cv ? d.kvf[ij] : d.ktu[ij] >> 16;
        const int m0 = (int)(w & 255u), m1 = (int)((w >> 8) & 255u);
        const auto mask = [&](int k) { return k >= m0 && k <= m1 ? 1.0 : 0.0; };
        const double r1h = (cv ? r1_hv : r1_hu_)[ij];
        const double unb = (cv ? vn_b : un_b_)[ij];
        const int nlev = d.jpk - 1;
        constexpr int KB = NXT_KB, NB = KMAX ? KMAX / KB : 1;
        static_assert(KMAX % KB == 0, "whole batches");

        // level k0 + q (0-based, the last one repeated) of a column, KB at a time
        const auto load = [&](const T *p, uint32_t c, int k0, T *v) {
    #pragma unroll
            for (int q = 0; q < KB; q++) v[q] = ldp(plane_ptr(p, d.n2, min(k0 + q, nlev - 1) + 1), c);
        };
        // scale factors that vary: KB at a time, with the levels' other operands
        const auto load_e3 = [&](int k0, double *v) {
    #pragma unroll
            for (int q = 0; q < KB; q++) v[q] = E3U ? 1.0 : E3(e3x, ij, min(k0 + q, nlev - 1) + 1);
        };
        const auto e3_of = [&](int k, double v) { return E3U ? uld(e3x, k - 1) : v; };
        // A
        T x[NB * KB];
        double mean = 0.0;
        const bool fix = spg_ts && !RING;
        const auto sum_a = [&](int k0, const T *v) {
    #pragma unroll
            for (int q = 0; q < KB; q++) {
                const int k = k0 + q + 1;
                if (k > nlev) break;
                const double t = NXT_E3(e3x, ij, k) * (double)v[q] * mask(k);
                mean = k == 1 ? t : mean + t;
            }
        };
        if constexpr (KMAX) {
    #pragma unroll
            for (int b = 0; b < NB; b++)
                if (b * KB < nlev) load(ua, src, b * KB, x + b * KB);
            if (fix) {
    #pragma unroll
                for (int b = 0; b < NB; b++)
                    if (b * KB < nlev) sum_a(b * KB, x + b * KB);
            }
        } else if (fix) {
            for (int k0 = 0; k0 < nlev; k0 += KB) {
                load(ua, src, k0, x);
                sum_a(k0, x);
            }
        }
        mean = mean * r1h;
        const double uab = fix ? (cv ? va_b : ua_b_)[ij] : 0.0;
        const bool adv = spg_ts && !bt_fw, bt_fix = spg_ts && bt_fw && !euler;
        const double cu_adv = adv ? (cv ? vn_adv : un_adv)[ij] * r1h : 0.0;

        // B
        double sn = 0.0, sb = 0.0;   // depth sums of un and ub
        const auto filter = [&](int k0, T *v) {
            T nv[KB], bv[KB];
            double e3[KB];
            load(un, ij, k0, nv);
            load(ub, ij, k0, bv);
            load_e3(k0, e3);
    #pragma unroll
            for (int q = 0; q < KB; q++) {
                const int k = k0 + q + 1;
                if (k > nlev) break;
                const double mk = mask(k), e3k = e3_of(k, e3[q]);
                T a = v[q];
                if (fix) a = (T)(((double)a - mean + uab) * mk);
                if (zero) a = T(0);
                if (spg_ts || RING || zero) stp(plane_ptr(ua, d.n2, k), ij, a);
                T f = bv[q];
                if (!euler) {
                    const double n1 = adv ? (double)(T)(((double)nv[q] - cu_adv + unb) * mk) : (double)nv[q];
                    f = (T)(n1 + atfp * ((double)bv[q] - 2.0 * n1 + (double)a));
                    if (KMAX == 0 || !bt_fix) stp(plane_ptr(ub, d.n2, k), ij, f);
                }
                stp(plane_ptr(un, d.n2, k), ij, a);
                v[q] = f;
                const double tn = e3k * (double)a * mk, tb = e3k * (double)f * mk;
                sn = k == 1 ? tn : sn + tn;
                sb = k == 1 ? tb : sb + tb;
            }
        };
        if constexpr (KMAX) {
    #pragma unroll
            for (int b = 0; b < NB; b++)
                if (b * KB < nlev) filter(b * KB, x + b * KB);
        } else {
            for (int k0 = 0; k0 < nlev; k0 += KB) {
                load(ua, src, k0, x);
                filter(k0, x);
            }
        }
        if (zero) A3(ua, i, j, d.jpk) = T(0);
        if (RING) A3(ua, i, j, d.jpk) = A3(ua, si, sj, d.jpk);

        // C
        if (bt_fix) {
            const double cu = sb * r1h - unb;
            const auto correct = [&](int k0, const T *v) {
                double e3[KB];
                load_e3(k0, e3);
    #pragma unroll
                for (int q = 0; q < KB; q++) {
                    const int k = k0 + q + 1;
                    if (k > nlev) break;
                    const double mk = mask(k);
                    const T nb = (T)((double)v[q] - cu * mk);
                    stp(plane_ptr(ub, d.n2, k), ij, nb);
                    const double tb = e3_of(k, e3[q]) * (double)nb * mk;
                    sb = k == 1 ? tb : sb + tb;
                }
            };
            if constexpr (KMAX) {
    #pragma unroll
                for (int b = 0; b < NB; b++)
                    if (b * KB < nlev) correct(b * KB, x + b * KB);
            } else {
                for (int k0 = 0; k0 < nlev; k0 += KB) {
                    load(ub, ij, k0, x);
                    correct(k0, x);
                }
            }
        }
        (cv ? vn_b : un_b_)[ij] = sn * r1h;
        (cv ? vb_b : ub_b_)[ij] = sb * r1h;
    }
};
template <typename T, int KMAX, bool E3U, bool RING>
KERNEL void k_dyn_nxt(DevDomain d, int spg_ts, int bt_fw, int euler, double atfp, T *ub, T *vb, T *un, T *vn, T *ua, T *va,
                      const double *__restrict__ ua_b, const double *__restrict__ va_b,
                      const double *__restrict__ un_adv, const double *__restrict__ vn_adv, double *__restrict__ ub_b,
                      double *__restrict__ vb_b, double *__restrict__ un_b, double *__restrict__ vn_b,
                      const double *__restrict__ r1_hu, const double *__restrict__ r1_hv)
{
    S_dyn_nxt<T, KMAX, E3U, RING>::run(vb_hw(), d, spg_ts, bt_fw, euler, atfp, ub, vb, un, vn, ua, va, ua_b, va_b, un_adv, vn_adv, ub_b, vb_b, un_b, vn_b, r1_hu, r1_hv);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <typename T>
int launch_div_hor(const T *un, const T *vn, T *hdivn)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    g.grid.z = (unsigned)((d.jpk + NXT_KB - 1) / NXT_KB);
    if (d.e3_sij == 0) LAUNCHB("div_hor", (k_div_hor<T, true>), (S_div_hor<T, true>), g, d, un, vn, hdivn);
    else LAUNCHB("div_hor", (k_div_hor<T, false>), (S_div_hor<T, false>), g, d, un, vn, hdivn);
    return 0;
}

template <typename T>
int launch_ssh_nxt(double z2dt, double zcoef, const T *un, const T *vn, T *hdivn, const double *sshb,
                   const double *emp_b, const double *emp, double *ssha)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    if (d.e3_sij == 0) LAUNCHB("ssh_nxt", (k_ssh_nxt<T, true>), (S_ssh_nxt<T, true>), g, d, z2dt, zcoef, un, vn, hdivn, sshb, emp_b, emp, ssha);
    else LAUNCHB("ssh_nxt", (k_ssh_nxt<T, false>), (S_ssh_nxt<T, false>), g, d, z2dt, zcoef, un, vn, hdivn, sshb, emp_b, emp, ssha);
    return 0;
}

template <typename T>
int launch_wzv(int first, double z1_2dt, const T *hdivn, T *wn)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    LAUNCHB("wzv", k_wzv<T>, (S_wzv<T>), g, d, first, z1_2dt, hdivn, wn);
    return 0;
}

int launch_ssh_swp(int euler, double *sshb, double *sshn, const double *ssha)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    LAUNCHB("ssh_swp", k_ssh_swp, (S_ssh_swp), g, d, euler, d.rn_atfp, sshb, sshn, ssha);
    return 0;
}

template <typename T>
int launch_tra_nxt(int euler, T *tsb, T *tsn, T *tsa, int ntr)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    g.grid.z = (unsigned)(ntr * d.jpk);
    LAUNCHB("tra_nxt", k_tra_nxt<T>, (S_tra_nxt<T>), g, d, euler, d.rn_atfp, tsb, tsn, tsa);
    return 0;
}

template <typename T>
int launch_dyn_nxt(int euler, T *ub, T *vb, T *un, T *vn, T *ua, T *va, const double *ua_b, const double *va_b,
                   const double *un_adv, const double *vn_adv, double *ub_b, double *vb_b, double *un_b,
                   double *vn_b, const double *r1_hu, const double *r1_hv)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj), gr = grid2(1, 1);
    g.grid.z = gr.grid.z = 2;
    gr.grid.x = (unsigned)((nxt_ring_rows(d) + (d.iper ? NXT_RING * 2 * (d.jpj - 2) : 0) + NH_BLOCK - 1) / NH_BLOCK);
#define NXT_LAUNCH3(KM, U, R, gg)                                                                                    \
    LAUNCHB("dyn_nxt", (k_dyn_nxt<T, KM, U, R>), (S_dyn_nxt<T, KM, U, R>), gg, d, d.ln_dynspg_ts, d.ln_bt_fw, euler, \
            d.rn_atfp, ub, vb, un, vn, ua, va, ua_b, va_b, un_adv, vn_adv, ub_b, vb_b, un_b, vn_b, r1_hu, r1_hv)
#define NXT_LAUNCH2(KM)                                                                                   \
    do {                                                                                                  \
        if (d.e3_sij == 0) NXT_LAUNCH3(KM, true, false, g); else NXT_LAUNCH3(KM, false, false, g);         \
        if (!d.iper && !d.jper) break;                                                                    \
        if (d.e3_sij == 0) NXT_LAUNCH3(KM, true, true, gr); else NXT_LAUNCH3(KM, false, true, gr);         \
    } while (0)
    // levels kept in registers: as few as hold the column, for occupancy (in a
    // plan the largest form, so that members of different depths share a launch)
    const int nlev = d.jpk - 1;
    if (nlev > 80) NXT_LAUNCH2(0);
    else if (nlev > 48 || nh::planning()) NXT_LAUNCH2(80);
    else if (nlev > 32) NXT_LAUNCH2(48);
    else NXT_LAUNCH2(32);
#undef NXT_LAUNCH2
#undef NXT_LAUNCH3
    return 0;
}

// ---------------------------------------------------------------------------
// stp_ctl, stpctl.F90:113-121: the six maxima as a two-pass reduction
// (per-block partials, then one block), NaN-propagating; and, when a test
// fails, the first Fortran-order position of each reported extremum
// (atomic minimum of the linear index over the matching cells)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double nanmax(double a, double b) { return (a > b || a != a) ? a : b; }

template <typename T>
KERNEL void k_stp_max(DevDomain d, const double *__restrict__ sshn, const T *__restrict__ un,
                      const T *__restrict__ tsn, double *__restrict__ part)
{
    __shared__ double red[6][NH_BLOCK];
    double m[6];
#pragma unroll
    for (int c = 0; c < 6; c++) m[c] = -INFINITY;
    const size_t n2 = d.n2, n3 = d.n3;
    const size_t stride = (size_t)gridDim.x * NH_BLOCK;
    for (size_t q = (size_t)blockIdx.x * NH_BLOCK + threadIdx.x; q < n3; q += stride) {
        if (q < n2) m[0] = nanmax(m[0], fabs(sshn[q]));
        m[1] = nanmax(m[1], fabs((double)un[q]));
        const int k = (int)(q / n2) + 1;
        if (pmask<double, 0>(d.ktu, (uint32_t)(q % n2), k) == 1.0) {
            const double sv = (double)tsn[n3 + q], tv = (double)tsn[q];
            m[2] = nanmax(m[2], -sv);
            m[3] = nanmax(m[3], sv);
            m[4] = nanmax(m[4], -tv);
            m[5] = nanmax(m[5], tv);
        }
    }
#pragma unroll
    for (int c = 0; c < 6; c++) red[c][threadIdx.x] = m[c];
    __syncthreads();
    for (int h = NH_BLOCK / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
#pragma unroll
            for (int c = 0; c < 6; c++) red[c][threadIdx.x] = nanmax(red[c][threadIdx.x], red[c][threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x < 6) part[(size_t)blockIdx.x * 6 + threadIdx.x] = red[threadIdx.x][0];
}

KERNEL void k_stp_final(const double *__restrict__ part, int nb, double *__restrict__ zmax,
                        uint32_t *__restrict__ loc)
{
    __shared__ double red[NH_BLOCK];
    for (int c = 0; c < 6; c++) {
        double m = -INFINITY;
        for (int b = (int)threadIdx.x; b < nb; b += NH_BLOCK) m = nanmax(m, part[(size_t)b * 6 + c]);
        red[threadIdx.x] = m;
        __syncthreads();
        for (int h = NH_BLOCK / 2; h > 0; h >>= 1) {
            if ((int)threadIdx.x < h) red[threadIdx.x] = nanmax(red[threadIdx.x], red[threadIdx.x + h]);
            __syncthreads();
        }
        if (threadIdx.x == 0) zmax[c] = red[0];
        __syncthreads();
    }
    if (threadIdx.x < 4) loc[threadIdx.x] = 0xffffffffu;
}

// loc[0]: |ssh| max, loc[1]: |u| max, loc[2]: S min, loc[3]: S max (linear indices)
__device__ __forceinline__ bool hit(double v, double m) { return v == m || (m != m && v != v); }
template <typename T>
KERNEL void k_stp_loc(DevDomain d, const double *__restrict__ sshn, const T *__restrict__ un,
                      const T *__restrict__ tsn, const double *__restrict__ zmax, uint32_t *__restrict__ loc)
{
    const size_t n2 = d.n2, n3 = d.n3;
    const size_t stride = (size_t)gridDim.x * NH_BLOCK;
    const double m0 = zmax[0], m1 = zmax[1], m2 = zmax[2], m3 = zmax[3];
    for (size_t q = (size_t)blockIdx.x * NH_BLOCK + threadIdx.x; q < n3; q += stride) {
        if (q < n2) {
            const double s = sshn[q];
            if (hit(fabs(s), m0) || (m0 != m0 && s != s)) atomicMin(&loc[0], (uint32_t)q);
        }
        const double u = (double)un[q];
        if (hit(fabs(u), m1) || (m1 != m1 && u != u)) atomicMin(&loc[1], (uint32_t)q);
        const int k = (int)(q / n2) + 1;
        if (pmask<double, 0>(d.ktu, (uint32_t)(q % n2), k) == 1.0) {
            const double sv = (double)tsn[n3 + q];
            if (hit(-sv, m2) || (m2 != m2 && sv != sv)) atomicMin(&loc[2], (uint32_t)q);
            if (hit(sv, m3) || (m3 != m3 && sv != sv)) atomicMin(&loc[3], (uint32_t)q);
        }
    }
}

#define STP_NB 1024
template <typename T>
int launch_stp_ctl(const double *sshn, const T *un, const T *tsn, double *buf, int want_loc)
{
    const DevDomain &d = nh::dom();
    double *part = buf, *zmax = buf + (size_t)STP_NB * 6;
    uint32_t *loc = (uint32_t *)(zmax + 8);
    Grid2 g;
    g.block = dim3(NH_BLOCK, 1, 1);
    g.grid = dim3(STP_NB, 1, 1);
    if (!want_loc) {
        LAUNCH("stp_ctl", k_stp_max<T>, g, d, sshn, un, tsn, part);
        Grid2 g1;
        g1.block = dim3(NH_BLOCK, 1, 1);
        g1.grid = dim3(1, 1, 1);
        LAUNCH("stp_ctl", k_stp_final, g1, (const double *)part, STP_NB, zmax, loc);
    } else {
        LAUNCH("stp_ctl", k_stp_loc<T>, g, d, sshn, un, tsn, (const double *)zmax, loc);
    }
    return 0;
}
size_t stp_ctl_buffer_bytes() { return ((size_t)STP_NB * 6 + 8) * sizeof(double) + 4 * sizeof(uint32_t); }

// ---------------------------------------------------------------------------
// tra_sbc, TRA/trasbc.F90:97-160 (linear free surface): one
// thread per (i,j); every point swaps or resets its trends, the points of
// 2..jpim1 x 2..jpj get the new trend and update level 1 of tsa
// ---------------------------------------------------------------------------
template <typename T>
KERNEL void k_tra_sbc(DevDomain d, int first, double *__restrict__ qns, double *__restrict__ qsr,
                      const double *__restrict__ sfx, const double *__restrict__ emp, const T *__restrict__ tsn,
                      T *__restrict__ tsa, double *__restrict__ sbc, double *__restrict__ sbc_b)
{
    THREAD_IJ(1, 1);
    if (i > d.jpi || j > d.jpj) return;
    const uint32_t ij = IJ32(i, j);
    const size_t n2 = d.n2, n3 = d.n3;
    const double rcp = 3991.86795711963, r1_rau0 = 1.0 / d.rau0, r1_rau0_rcp = 1.0 / (d.rau0 * rcp);
    // lines 97-100: without penetrative solar flux the whole of qsr enters
    // the surface level through qns; with it, tra_qsr takes qsr
    double q = qns[ij];
    if (!d.ln_traqsr) {
        q = q + qsr[ij];
        qns[ij] = q;
        qsr[ij] = 0.0;
    }
    double bt, bs, ct, cs;
    if (first) {
        bt = bs = ct = cs = 0.0;
    } else {
        bt = sbc[ij];
        bs = sbc[n2 + ij];
        ct = bt;
        cs = bs;
    }
    const double zfact = first ? 1.0 : 0.5;
    if (j >= 2 && i >= 2 && i <= d.jpi - 1) {
        ct = r1_rau0_rcp * q;
        cs = r1_rau0 * sfx[ij];
        ct = ct + r1_rau0 * emp[ij] * (double)tsn[ij];
        cs = cs + r1_rau0 * emp[ij] * (double)tsn[n3 + ij];
        const double e3 = E3(d.md.e3t, ij, 1);
        tsa[ij] = (T)((double)tsa[ij] + zfact * (bt + ct) / e3);
        tsa[n3 + ij] = (T)((double)tsa[n3 + ij] + zfact * (bs + cs) / e3);
    }
    sbc_b[ij] = bt;
    sbc_b[n2 + ij] = bs;
    sbc[ij] = ct;
    sbc[n2 + ij] = cs;
}

// ---------------------------------------------------------------------------
// tra_qsr, two bands (ln_qsr_2bd), TRA/traqsr.F90:134-276: one thread per
// (i,j) column.  Every column swaps qsr_hc into qsr_hc_b (or clears it at an
// Euler start); the interior ones form qsr_hc on levels 1..nksr, add the
// trend to tsa and set fraqsr_1lev.  The attenuation of w-level k+1 for
// level k is the attenuation of w-level k for level k+1 (the same
// expression of the same depth), so one pair of exponentials per level.
// mode 0: swap, 1: Euler start (z1_2 = 1), 2: qsr_hc_b given (a restart).
// ---------------------------------------------------------------------------
template <typename T>
KERNEL void k_tra_qsr(DevDomain d, int mode, int nksr, double zz0, double zz1, double xsi0r, double xsi1r,
                      const double *__restrict__ qsr, const T *__restrict__ gdepw, double *__restrict__ hc,
                      double *__restrict__ hc_b, T *__restrict__ tsa, double *__restrict__ fraqsr)
{
    THREAD_IJ(1, 1);
    if (i > d.jpi || j > d.jpj) return;
    if (mode != 2)
        for (int k = 1; k <= d.jpk; k++) A3(hc_b, i, j, k) = mode == 0 ? A3(hc, i, j, k) : 0.0;
    if (i < 2 || i > d.jpi - 1 || j < 2 || j > d.jpj - 1) return;
    const uint32_t ij = IJ32(i, j);
    const double rcp = 3991.86795711963, r1_rau0_rcp = 1.0 / (d.rau0 * rcp);
    const double z1_2 = mode == 1 ? 1.0 : 0.5;
    const double q = qsr[ij];
    double zg = (double)A3(gdepw, i, j, 1);
    double zc0 = zz0 * exp(-zg * xsi0r) + zz1 * exp(-zg * xsi1r);
    for (int k = 1; k <= nksr; k++) {
        zg = (double)A3(gdepw, i, j, k + 1);
        const double zc1 = zz0 * exp(-zg * xsi0r) + zz1 * exp(-zg * xsi1r);
        const double h = q * (zc0 * WMASK(double, i, j, k) - zc1 * WMASK(double, i, j, k + 1));
        const uint32_t p = IJK32(i, j, k);
        at32(hc, p) = h;
        at32(tsa, p) = (T)((double)at32(tsa, p) + z1_2 * (at32(hc_b, p) + h) / E3(d.md.e3t, ij, k));
        if (k == 1) fraqsr[ij] = (q != 0.0) ? h / (r1_rau0_rcp * q) : 1.0;
        zc0 = zc1;
    }
}

template <typename T>
int launch_tra_qsr(int mode, int nksr, double rn_abs, double rn_si0, double rn_si1, const double *qsr,
                   const T *gdepw, double *qsr_hc, double *qsr_hc_b, T *tsa, double *fraqsr_1lev)
{
    const DevDomain &d = nh::dom();
    const double rcp = 3991.86795711963, r1_rau0_rcp = 1.0 / (d.rau0 * rcp);
    const double zz0 = rn_abs * r1_rau0_rcp, zz1 = (1. - rn_abs) * r1_rau0_rcp;
    Grid2 g = grid2(d.jpi, d.jpj);
    LAUNCH("tra_qsr", k_tra_qsr<T>, g, d, mode, nksr, zz0, zz1, 1.0 / rn_si0, 1.0 / rn_si1, qsr, gdepw, qsr_hc,
           qsr_hc_b, tsa, fraqsr_1lev);
    return launch_lbc<double>(fraqsr_1lev, 1, 'T', 0.0);
}

template <typename T>
int launch_tra_sbc(int first, double *qns, double *qsr, const double *sfx, const double *emp, const T *tsn, T *tsa,
                   double *sbc, double *sbc_b)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    LAUNCH("tra_sbc", k_tra_sbc<T>, g, d, first, qns, qsr, sfx, emp, tsn, tsa, sbc, sbc_b);
    return 0;
}

// ---------------------------------------------------------------------------
// the depth-mean velocities after a restart, DOM/istate.F90:159-178: every
// column, levels 1..jpkm1 summed in order from zero (linear free surface:
// the before scale factors and inverse depths are the now ones)
// ---------------------------------------------------------------------------
template <typename T>
KERNEL void k_istate_bt(DevDomain d, const T *__restrict__ un, const T *__restrict__ vn, const T *__restrict__ ub,
                        const T *__restrict__ vb, const double *__restrict__ r1_hu, const double *__restrict__ r1_hv,
                        double *__restrict__ un_b, double *__restrict__ vn_b, double *__restrict__ ub_b,
                        double *__restrict__ vb_b)
{
    THREAD_IJ(1, 1);
    if (i > d.jpi || j > d.jpj) return;
    const Metrics<double> &m = d.md;
    const uint32_t ij = IJ32(i, j);
    double a = 0., b = 0., c = 0., e = 0.;
    for (int k = 1; k <= d.jpk - 1; k++) {
        const double eu = E3(m.e3u, ij, k), ev = E3(m.e3v, ij, k);
        const double um = UMASK(double, i, j, k), vm = VMASK(double, i, j, k);
        const uint32_t p = IJK32(i, j, k);
        a = a + eu * (double)at32(un, p) * um;
        b = b + ev * (double)at32(vn, p) * vm;
        c = c + eu * (double)at32(ub, p) * um;
        e = e + ev * (double)at32(vb, p) * vm;
    }
    un_b[ij] = a * r1_hu[ij];
    vn_b[ij] = b * r1_hv[ij];
    ub_b[ij] = c * r1_hu[ij];
    vb_b[ij] = e * r1_hv[ij];
}

template <typename T>
int launch_istate_bt(const T *un, const T *vn, const T *ub, const T *vb, const double *r1_hu, const double *r1_hv,
                     double *un_b, double *vn_b, double *ub_b, double *vb_b)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    LAUNCH("rst_read", k_istate_bt<T>, g, d, un, vn, ub, vb, r1_hu, r1_hv, un_b, vn_b, ub_b, vb_b);
    return 0;
}

#define INST(T)                                                                                                  \
    template int launch_istate_bt<T>(const T *, const T *, const T *, const T *, const double *, const double *,  \
                                     double *, double *, double *, double *);                                    \
    template int launch_div_hor<T>(const T *, const T *, T *);                                                   \
    template int launch_ssh_nxt<T>(double, double, const T *, const T *, T *, const double *, const double *,    \
                                   const double *, double *);                                                    \
    template int launch_wzv<T>(int, double, const T *, T *);                                                     \
    template int launch_tra_nxt<T>(int, T *, T *, T *, int);                                                          \
    template int launch_dyn_nxt<T>(int, T *, T *, T *, T *, T *, T *, const double *, const double *,            \
                                   const double *, const double *, double *, double *, double *, double *,      \
                                   const double *, const double *);                                              \
    template int launch_stp_ctl<T>(const double *, const T *, const T *, double *, int);                        \
    template int launch_tra_qsr<T>(int, int, double, double, double, const double *, const T *, double *,      \
                                   double *, T *, double *);                                                \
    template int launch_tra_sbc<T>(int, double *, double *, const double *, const double *, const T *, T *,       \
                                   double *, double *);
INST(double)
INST(float)
#undef INST
