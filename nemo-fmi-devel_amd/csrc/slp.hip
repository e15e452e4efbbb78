// slp.hip -- the mixed-layer level (ZDF/zdfmxl.F90) and the iso-neutral
// slopes of the standard (Madec) operator (LDF/ldfslp.F90: ldf_slp and
// ldf_slp_mxl), for z-coordinates without partial steps or ice-shelf
// cavities (risfdep = 0, mikt = 1).
//
// Arithmetic is FP64 in both storage forms, rounded once on store, in the
// reference's operation order, so the FP64 form reproduces it bit for bit.
//
// The reference builds the unfiltered slopes in work arrays, applies
// lbc_lnk to them, filters and applies lbc_lnk again.  Here one kernel marches
// down a region of columns: it builds the unfiltered slopes of a level in LDS (a
// point on the ring evaluates the interior formula at its lbc source, or is
// zero on a closed boundary, which is what lbc_lnk gives), filters them and
// writes the interior; the final lbc_lnk fills the output's ring.
#include "common.hpp"
#include "kernels.hpp"

namespace {

constexpr double ZEPS = 1.e-20;

template <typename T>
struct SlpIn {
    const T *prd, *pn2;
};

// zgru / zgrv, LDF/ldfslp.F90:138-145 (defined for i <= jpim1, j <= jpjm1)
template <typename T>
__device__ __forceinline__ double gru(const DevDomain &d, const T *prd, int i, int j, int k)
{
    return UMASK(double, i, j, k) * ((double)A3(prd, i + 1, j, k) - (double)A3(prd, i, j, k));
}
template <typename T>
__device__ __forceinline__ double grv(const DevDomain &d, const T *prd, int i, int j, int k)
{
    return VMASK(double, i, j, k) * ((double)A3(prd, i, j + 1, k) - (double)A3(prd, i, j, k));
}
// zdzr at t-points, lines 162-170 (zero at level 1)
template <typename T>
__device__ __forceinline__ double dzr(const DevDomain &d, const T *prd, const T *pn2, int i, int j, int k)
{
    if (k == 1) return 0.;
    const double zm1_g = -1.0 / d.grav;
    return zm1_g * ((double)A3(prd, i, j, k) + 1.) * ((double)A3(pn2, i, j, k) + (double)A3(pn2, i, j, k + 1)) *
           (1. - 0.5 * TMASK(double, i, j, k + 1));
}
__device__ __forceinline__ double min3(double a, double b, double c) { return fmin(fmin(a, b), c); }
__device__ __forceinline__ double max2(double a, double b) { return a > b ? a : b; }

// omlmask, lines 660-668: 1 inside the mixed layer (k <= nmln - 1)
__device__ __forceinline__ double oml(const int32_t *nmln, uint32_t ij, int k) { return k <= nmln[ij] - 1 ? 1. : 0.; }

// ---------------------------------------------------------------------------
// zdf_mxl, ZDF/zdfmxl.F90:92-125: one thread per column
// ---------------------------------------------------------------------------
template <typename T, bool E3U>
KERNEL void k_zdf_mxl(DevDomain d, const T *__restrict__ rn2b, const T *__restrict__ gdept,
                      const T *__restrict__ gdepw, int nlb10, double zN2_c, int32_t *__restrict__ nmln,
                      double *__restrict__ hmlp, double *__restrict__ hmlpt)
{
    THREAD_IJ(1, 1);
    if (i > d.jpi || j > d.jpj) return;
    const uint32_t ij = IJ32(i, j);
    const int ikt = d.mbkt[ij];
    double h = 0.;
    int nm = nlb10;
    // h never falls, and nm stays at ikt + 1 from there on: the march ends where
    // every column of the wave has passed one of the two (the column read to the
    // bottom: 33 us at 512x509x75 in FP32, 11 us at 203x157x31 in FP64).  A mixed
    // layer down to the bottom of an all-wet domain has nothing to leave out:
    // 600x500x60 FP32 24 us without the test, 27 with it, 21 with the level's base
    // and a uniform e3w in scalar registers
    constexpr int KB = 8;
    for (int k0 = nlb10; k0 <= d.jpk - 1; k0 += KB) {
        T n2[KB];
#pragma unroll
        for (int q = 0; q < KB; q++) n2[q] = ldp(plane_ptr(rn2b, d.n2, min(k0 + q, d.jpk - 1)), ij);
#pragma unroll
        for (int q = 0; q < KB; q++) {
            const int k = k0 + q;
            if (k > d.jpk - 1) break;
            h = h + max2((double)n2[q], 0.) * (E3U ? uld(d.md.e3w, k - 1) : E3(d.md.e3w, ij, k));
            if (h < zN2_c) nm = (k < ikt ? k : ikt) + 1;
        }
        if (!__any(h < zN2_c && k0 + KB - 1 < ikt)) break;
    }
    const double ss = d.ssmask[ij];
    nmln[ij] = nm;
    hmlp[ij] = (double)A3(gdepw, i, j, nm) * ss;
    hmlpt[ij] = (double)A3(gdept, i, j, nm - 1) * ss;
}

// ---------------------------------------------------------------------------
// ldf_slp_mxl, LDF/ldfslp.F90:682-725, per interior column: the u/v slopes
// just below the mixed layer already divided by the depth of its last
// t-point (zslpml_hmlpu/v, lines 188-195) and the w slopes wslpiml/wslpjml
// ---------------------------------------------------------------------------
template <typename T>
KERNEL void k_slp_mxl(DevDomain d, SlpIn<T> in, const int32_t *__restrict__ nmln, const double *__restrict__ hmlpt,
                      double z1_slpmax, double *__restrict__ zsu, double *__restrict__ zsv, double *__restrict__ wiml,
                      double *__restrict__ wjml)
{
    THREAD_IJ(2, 2);
    if (i > d.jpi - 1 || j > d.jpj - 1) return;
    const Metrics<double> &m = d.md;
    const T *prd = in.prd, *pn2 = in.pn2;
    const uint32_t ij = IJ32(i, j);
    const int jpkm1 = d.jpk - 1;
    const int nm = nmln[ij], nme = nmln[ij + 1], nmn = nmln[ij + (uint32_t)d.jpi];
    const int iku = min(max(1, max(nm, nme)), jpkm1);
    const int ikv = min(max(1, max(nm, nmn)), jpkm1);
    double zbu = 0.5 * (dzr(d, prd, pn2, i, j, iku) + dzr(d, prd, pn2, i + 1, j, iku));
    double zbv = 0.5 * (dzr(d, prd, pn2, i, j, ikv) + dzr(d, prd, pn2, i, j + 1, ikv));
    const double zau = gru(d, prd, i, j, iku) * m.r1_e1u[ij];
    const double zav = grv(d, prd, i, j, ikv) * m.r1_e2v[ij];
    zbu = min3(zbu, -z1_slpmax * fabs(zau), -7.e+3 / E3(m.e3u, ij, iku) * fabs(zau));
    zbv = min3(zbv, -z1_slpmax * fabs(zav), -7.e+3 / E3(m.e3v, ij, ikv) * fabs(zav));
    const double uml = zau / (zbu - ZEPS) * UMASK(double, i, j, iku);
    const double vml = zav / (zbv - ZEPS) * VMASK(double, i, j, ikv);
    zsu[ij] = uml / max2(max2(hmlpt[ij], hmlpt[ij + 1]), 5.);
    zsv[ij] = vml / max2(max2(hmlpt[ij], hmlpt[ij + (uint32_t)d.jpi]), 5.);
    const int ik = min(nm + 1, d.jpk), ikm1 = max(1, ik - 1);
    const double zm1_2g = -0.5 / d.grav;
    const double zbw = zm1_2g * (double)A3(pn2, i, j, ik) * ((double)A3(prd, i, j, ik) + (double)A3(prd, i, j, ikm1) + 2.);
    const double zci = max2(UMASK(double, i - 1, j, ik) + UMASK(double, i, j, ik) + UMASK(double, i - 1, j, ikm1) +
                                UMASK(double, i, j, ikm1),
                            ZEPS) * m.e1t[ij];
    const double zcj = max2(VMASK(double, i, j - 1, ik) + VMASK(double, i, j, ik) + VMASK(double, i, j - 1, ikm1) +
                                VMASK(double, i, j, ikm1),
                            ZEPS) * m.e2t[ij];
    const double tm = TMASK(double, i, j, ik);
    const double zai = (gru(d, prd, i - 1, j, ik) + gru(d, prd, i, j, ik) + gru(d, prd, i - 1, j, ikm1) +
                        gru(d, prd, i, j, ikm1)) / zci * tm;
    const double zaj = (grv(d, prd, i, j - 1, ik) + grv(d, prd, i, j, ik) + grv(d, prd, i, j - 1, ikm1) +
                        grv(d, prd, i, j, ikm1)) / zcj * tm;
    const double e3w = E3(m.e3w, ij, ik);
    const double zbi = min3(zbw, -100. * fabs(zai), -7.e+3 / e3w * fabs(zai));
    const double zbj = min3(zbw, -100. * fabs(zaj), -7.e+3 / e3w * fabs(zaj));
    wiml[ij] = zai / (zbi - ZEPS) * tm;
    wjml[ij] = zaj / (zbj - ZEPS) * tm;
}

// ---------------------------------------------------------------------------
// The four slopes, marched down SLP_RX x SLP_RY columns, one per thread.  At each
// level a thread shares its prd and zdzr with its neighbours through LDS, forms
// the unfiltered slopes (zwz, zww of parts I and II) of its column from them
// and the gradients it kept from the level above, shares those, and, inside
// the tile (the region less two points on each side), applies the Shapiro
// filters and tapers of lines 232-271 and 316-356.  A region point on the
// domain's ring takes zero on a closed side, its lbc source's value on a cyclic
// one (the reference's lbc_lnk of zwz/zww, lines 231 and 315): there the region
// runs on past the domain's last column to its first, both ring columns
// included, so the source is two points away across the seam and the region
// has two more points on the side of the seam (slp_tile).  The output's ring is
// the final lbc_lnk (line 361), a separate pass.
//
// The terms of the mixed layer (a division and the depths) are formed only at
// levels where a column of the wave is in it, -7e3/e3 once per level where the
// scale factors are horizontally uniform (E3U; where they vary, they are loaded
// with the level's fields, ahead of the barrier), and levels below the region's
// deepest column are stored as the zeros the masks give.
//
// Bound by FP64 vector instructions (six divisions per point).  One level of
// a 64x4 tile per workgroup, staged in LDS with its two-point halo, ran 1020
// instructions per cell: 512x509x75 FP32 790 -> 330 us, 203x157x31 cyclic FP64
// 74 -> 39 us; all wet, and the mixed layer down to the bottom, 600x500x60 FP32
// 773 -> 695 us, 300x200x60 cyclic both ways FP64 203 -> 175 us (277 us with the
// wide halo on every side of every tile); e3 varying, 512x512x75 FP32 847 -> 407
// us (551 us with e3 loaded where used).
// ---------------------------------------------------------------------------
#define SLP_RX 32
#define SLP_RY 16
#define SLP_MAXKB 24
// The n interior points of a direction over tiles, each the middle of a region of
// R columns: a halo of two points on each side, four where the tile meets a
// seam, which the first and the last tile of a cyclic direction do.  Tile t of nt
// owns cnt points from o on (0-based), the first of them at region column h.
inline int slp_tiles(int n, int R, int per)
{
    if (!per) return (n + R - 5) / (R - 4);
    if (n <= R - 8) return 1;
    const int r = n - 2 * (R - 6);
    return r <= 0 ? 2 : 2 + (r + R - 5) / (R - 4);
}
__device__ inline void slp_tile(int t, int nt, int n, int R, int per, int &o, int &cnt, int &h)
{
    h = per && t == 0 ? 4 : 2;
    if (!per) {
        o = t * (R - 4);
        cnt = min(R - 4, n - o);
        return;
    }
    const int e = nt == 1 ? n : nt == 2 ? (n + 1) / 2 : R - 6;    // the first tile's points
    const int w = nt > 2 ? (n - 2 * e + nt - 3) / (nt - 2) : 0;   // a middle one's
    o = t == 0 ? 0 : t < nt - 1 ? e + (t - 1) * w : nt == 2 ? e : n - e;
    cnt = t == 0 ? e : t < nt - 1 ? min(w, n - e - o) : n - o;
}
template <typename T, bool E3U>
__global__ __launch_bounds__(SLP_RX * SLP_RY, 4) void k_slp(DevDomain d, SlpIn<T> in, const T *__restrict__ gdept,
                                                             const T *__restrict__ gdepw,
                                                             const int32_t *__restrict__ nmln,
                                                             const double *__restrict__ zsu,
                                                             const double *__restrict__ zsv,
                                                             const double *__restrict__ hmlp,
                                                             const double *__restrict__ wiml,
                                                             const double *__restrict__ wjml, double z1_slpmax, int kb,
                                                             T *__restrict__ uslp, T *__restrict__ vslp,
                                                             T *__restrict__ wslpi, T *__restrict__ wslpj)
{
    constexpr int N = SLP_RX * SLP_RY;
    __shared__ double sp[N], sdz[N], su[N], sv[N], swi[N], swj[N];
    __shared__ double q3u[SLP_MAXKB], q3v[SLP_MAXKB], q3w[SLP_MAXKB];   // -7e3 / e3 of the chunk's levels
    __shared__ int s_end;
    const Metrics<double> &m = d.md;
    unsigned bx, by;
    xcd_tile(bx, by);
    const int jpi = d.jpi, jpj = d.jpj, jpkm1 = d.jpk - 1;
    const int q = (int)threadIdx.x, lx = q % SLP_RX, ly = q / SLP_RX;
    int ox, cx, hx, oy, cy, hy;
    slp_tile((int)bx, (int)gridDim.x, jpi - 2, SLP_RX, d.iper, ox, cx, hx);
    slp_tile((int)by, (int)gridDim.y, jpj - 2, SLP_RY, d.jper, oy, cy, hy);
    int i = 2 + ox + lx - hx, j = 2 + oy + ly - hy;
    const bool own = lx >= hx && lx < hx + cx && ly >= hy && ly < hy + cy;
    if (d.iper) i = ((i - 1) % jpi + jpi) % jpi + 1;
    if (d.jper) j = ((j - 1) % jpj + jpj) % jpj + 1;
    const int k0 = 2 + (int)blockIdx.z * kb, k1 = min(k0 + kb - 1, jpkm1);
    const bool inner = i >= 2 && i <= jpi - 1 && j >= 2 && j <= jpj - 1;
    // columns off the domain read its nearest one and are not used
    const int ic = min(max(i, 1), jpi), jc = min(max(j, 1), jpj);
    const uint32_t c = IJ32(ic, jc);
    const uint32_t w_ = ic > 1 ? c - 1u : c, e_ = ic < jpi ? c + 1u : c;
    const uint32_t s_ = jc > 1 ? c - (uint32_t)jpi : c, n_ = jc < jpj ? c + (uint32_t)jpi : c;
    const uint32_t tc = d.ktu[c], tw = d.ktu[w_], tn = d.ktu[n_], ts = d.ktu[s_];
    const uint32_t vc = d.kvf[c], vs = d.kvf[s_], ve = d.kvf[e_], vw = d.kvf[w_];
    if (q == 0) s_end = 0;
    __syncthreads();
    atomicMax(&s_end, (int)((tc >> 8) & 255u));
    if (E3U && q < k1 - k0 + 1) {
        q3u[q] = -7.e+3 / m.e3u[k0 + q - 1];
        q3v[q] = -7.e+3 / m.e3v[k0 + q - 1];
        q3w[q] = -7.e+3 / m.e3w[k0 + q - 1];
    }
    __syncthreads();
    const int kend = min(k1, s_end);     // below: dry in every column
    // a ring point's lbc source, by its place in the region; raw: the thread
    // forms unfiltered slopes
    int si = i, sj = j;
    const bool in_dom = i >= 1 && i <= jpi && j >= 1 && j <= jpj;
    const bool ring = in_dom && !inner && lbc_src(d, 'U', i, j, si, sj);
    const int src = min(max(q + (si == i ? 0 : i == 1 ? -2 : 2) + SLP_RX * (sj == j ? 0 : j == 1 ? -2 : 2), 0), N - 1);
    const bool cyc = (d.iper || d.jper) && __syncthreads_or(ring);
    const bool edge = lx == 0 || lx == SLP_RX - 1 || ly == 0 || ly == SLP_RY - 1;
    const bool raw = inner && !edge;
    const auto um = [](uint32_t x, int k) { return k >= (int)((x >> 16) & 255u) && k <= (int)((x >> 24) & 255u); };
    const auto vm = [](uint32_t x, int k) { return k >= (int)(x & 255u) && k <= (int)((x >> 8) & 255u); };   // also tmask
    const auto msk = [](bool on, double x) { return on ? x : 0.; };
    const double zm1_g = -1.0 / d.grav, zm1_2g = -0.5 / d.grav, z1_16 = 1.0 / 16.;
    if (k0 <= kend) {
        const double r1_e1u = m.r1_e1u[c], r1_e2v = m.r1_e2v[c], e1t = m.e1t[c], e2t = m.e2t[c];
        const int ml_c = nmln[c] - 1, ml_e = nmln[e_] - 1, ml_n = nmln[n_] - 1;   // omlmask: k <= ml
        const size_t plane = d.n2;
        const auto ld = [&](const T *p, int k) { return (double)ldp(plane_ptr(p, plane, k), c); };
        double p_m = ld(in.prd, k0 - 1), p_k = ld(in.prd, k0);
        double n_k = ld(in.pn2, k0), n_p = ld(in.pn2, k0 + 1);
        // gradients of the level above, and its masks
        double gu_cm, gu_wm, gv_cm, gv_sm;
        bool um_cm = um(tc, k0 - 1), um_wm = um(tw, k0 - 1), vm_cm = vm(vc, k0 - 1), vm_sm = vm(vs, k0 - 1);
        bool um_c = um(tc, k0), vm_c = vm(vc, k0), tm_c = vm(tc, k0), tm_m = vm(tc, k0 - 1);
        sp[q] = p_m;
        __syncthreads();
        gu_cm = msk(um_cm, sp[min(q + 1, N - 1)] - p_m);
        gu_wm = msk(um_wm, p_m - sp[max(q - 1, 0)]);
        gv_cm = msk(vm_cm, sp[min(q + SLP_RX, N - 1)] - p_m);
        gv_sm = msk(vm_sm, p_m - sp[max(q - SLP_RX, 0)]);
        __syncthreads();
        for (int k = k0; k <= kend; k++) {
            const int kn = min(k + 1, d.jpk);
            const double p_n = ld(in.prd, kn), n_pn = ld(in.pn2, min(k + 2, d.jpk));   // the next level's
            double e3u = 1., e3v = 1., e3w = 1.;
            if (!E3U) {
                e3u = E3(m.e3u, c, k);
                e3v = E3(m.e3v, c, k);
                e3w = E3(m.e3w, c, k);
            }
            const bool um_w = um(tw, k), vm_s = vm(vs, k), um_cp = um(tc, k + 1), vm_cp = vm(vc, k + 1);
            const bool tm_p = vm(tc, k + 1), wm = tm_c && tm_m;
            const double dz = zm1_g * (p_k + 1.) * (n_k + n_p) * (tm_p ? 0.5 : 1.);   // zdzr, lines 162-170
            sp[q] = p_k;
            sdz[q] = dz;
            __syncthreads();
            double a = 0., b = 0., e = 0., f = 0.;
            const bool ml_uv = raw && k <= max(ml_c, max(ml_e, ml_n)), ml_w = raw && k - 1 <= ml_c;
            const bool any_uv = __any(ml_uv), any_w = __any(ml_w);
            if (raw) {
                const double gu_c = msk(um_c, sp[q + 1] - p_k), gu_w = msk(um_w, p_k - sp[q - 1]);
                const double gv_c = msk(vm_c, sp[q + SLP_RX] - p_k), gv_s = msk(vm_s, p_k - sp[q - SLP_RX]);
                const double e3u7 = E3U ? q3u[k - k0] : -7.e+3 / e3u;
                const double e3v7 = E3U ? q3v[k - k0] : -7.e+3 / e3v;
                const double e3w7 = E3U ? q3w[k - k0] : -7.e+3 / e3w;
                // I. u, v slopes, lines 197-219
                const double zau = gu_c * r1_e1u, zav = gv_c * r1_e2v;
                double zbu = 0.5 * (dz + sdz[q + 1]), zbv = 0.5 * (dz + sdz[q + SLP_RX]);
                zbu = min3(zbu, -z1_slpmax * fabs(zau), e3u7 * fabs(zau));
                zbv = min3(zbv, -z1_slpmax * fabs(zav), e3v7 * fabs(zav));
                double tu = zau / (zbu - ZEPS), tv = zav / (zbv - ZEPS);
                if (any_uv) {
                    const double oc = k <= ml_c ? 1. : 0.;
                    const double zfi = max2(oc, k <= ml_e ? 1. : 0.), zfj = max2(oc, k <= ml_n ? 1. : 0.);
                    const double gc = ld(gdept, k);
                    const double zdepu = 0.5 * ((gc + (double)ldp(plane_ptr(gdept, plane, k), e_)) - E3(m.e3u, c, d.miku[c]));
                    const double zdepv = 0.5 * ((gc + (double)ldp(plane_ptr(gdept, plane, k), n_)) - E3(m.e3v, c, d.mikv[c]));
                    tu = (1. - zfi) * zau / (zbu - ZEPS) + zfi * zdepu * zsu[c];
                    tv = (1. - zfj) * zav / (zbv - ZEPS) + zfj * zdepv * zsv[c];
                }
                a = msk(um_c, tu);
                b = msk(vm_c, tv);
                // II. w slopes, lines 277-304
                const double zbw = zm1_2g * n_k * (p_k + p_m + 2.);
                const double zci = max2((double)((int)um_w + (int)um_c + (int)um_wm + (int)um_cm), ZEPS) * e1t;
                const double zcj = max2((double)((int)vm_s + (int)vm_cm + (int)vm_sm + (int)vm_c), ZEPS) * e2t;
                const double zai = msk(wm, (gu_w + gu_cm + gu_wm + gu_c) / zci);
                const double zaj = msk(wm, (gv_s + gv_cm + gv_sm + gv_c) / zcj);
                const double zbi = min3(zbw, -100. * fabs(zai), e3w7 * fabs(zai));
                const double zbj = min3(zbw, -100. * fabs(zaj), e3w7 * fabs(zaj));
                double ti = zai / (zbi - ZEPS), tj = zaj / (zbj - ZEPS);
                if (any_w) {
                    const double zfk = max2(k <= ml_c ? 1. : 0., k - 1 <= ml_c ? 1. : 0.);
                    const double gwt = (double)A3(gdepw, ic, jc, d.mikt[c]);
                    const double zck = (ld(gdepw, k) - gwt) / max2(hmlp[c] - gwt, 10.);
                    ti = ti * (1. - zfk) + zck * wiml[c] * zfk;
                    tj = tj * (1. - zfk) + zck * wjml[c] * zfk;
                }
                e = msk(wm, ti);
                f = msk(wm, tj);
                gu_cm = gu_c; gu_wm = gu_w; gv_cm = gv_c; gv_sm = gv_s;
            }
            su[q] = a;
            sv[q] = b;
            swi[q] = e;
            swj[q] = f;
            __syncthreads();
            if (cyc) {
                if (ring) { a = su[src]; b = sv[src]; e = swi[src]; f = swj[src]; }
                __syncthreads();
                if (ring) { su[q] = a; sv[q] = b; swi[q] = e; swj[q] = f; }
                __syncthreads();
            }
            if (own) {
                const auto shapiro = [&](const double *z) {
                    const double *t = z + q;
                    return t[-SLP_RX - 1] + t[-SLP_RX + 1] + t[SLP_RX - 1] + t[SLP_RX + 1] +
                           2. * (t[-SLP_RX] + t[-1] + t[1] + t[SLP_RX]) + 4. * t[0];
                };
                double u = z1_16 * shapiro(su), v = z1_16 * shapiro(sv);
                const auto two = [](bool x, bool y) { return (double)((int)x + (int)y); };
                u = u * two(um(tn, k), um(ts, k)) * 0.5 * two(um_c, um_cp) * 0.5;
                v = v * two(vm(ve, k), vm(vw, k)) * 0.5 * two(vm_c, vm_cp) * 0.5;
                const double zcofw = wm ? z1_16 : 0.;
                const double zck = two(um_c, um_w) * two(vm_c, vm_s) * 0.25;
                stp(plane_ptr(uslp, plane, k), c, (T)u);
                stp(plane_ptr(vslp, plane, k), c, (T)v);
                stp(plane_ptr(wslpi, plane, k), c, (T)(shapiro(swi) * zcofw * zck));
                stp(plane_ptr(wslpj, plane, k), c, (T)(shapiro(swj) * zcofw * zck));
            }
            p_m = p_k; p_k = p_n;
            n_k = n_p; n_p = n_pn;
            um_cm = um_c; um_wm = um_w; vm_cm = vm_c; vm_sm = vm_s;
            um_c = um_cp; vm_c = vm_cp; tm_m = tm_c; tm_c = tm_p;
        }
    }
    if (!own) return;
    for (int k = max(k0, kend + 1); k <= k1; k++) {
        stp(plane_ptr(uslp, d.n2, k), c, T(0));
        stp(plane_ptr(vslp, d.n2, k), c, T(0));
        stp(plane_ptr(wslpi, d.n2, k), c, T(0));
        stp(plane_ptr(wslpj, d.n2, k), c, T(0));
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <typename T>
int launch_zdf_mxl(const T *rn2b, const T *gdept, const T *gdepw, int nlb10, double rho_c, int32_t *nmln,
                   double *hmlp, double *hmlpt)
{
    const DevDomain &d = nh::dom();
    const double zN2_c = d.grav * rho_c * (1.0 / d.rau0);
    Grid2 g = grid2(d.jpi, d.jpj);
    if (d.e3_sij == 0) LAUNCH("zdf_mxl", (k_zdf_mxl<T, true>), g, d, rn2b, gdept, gdepw, nlb10, zN2_c, nmln, hmlp, hmlpt);
    else LAUNCH("zdf_mxl", (k_zdf_mxl<T, false>), g, d, rn2b, gdept, gdepw, nlb10, zN2_c, nmln, hmlp, hmlpt);
    return 0;
}

template <typename T>
int launch_ldf_slp(const T *prd, const T *pn2, const T *gdept, const T *gdepw, const int32_t *nmln,
                   const double *hmlp, const double *hmlpt, double rn_slpmax, T *uslp, T *vslp, T *wslpi, T *wslpj)
{
    const DevDomain &d = nh::dom();
    if (d.jpk < 3) return 0;
    const double z1_slpmax = 1. / rn_slpmax;
    const SlpIn<T> in{prd, pn2};
    double *zsu = nh::scratch2(NH_S2_SLP), *zsv = nh::scratch2(NH_S2_SLP + 1);
    double *wiml = nh::scratch2(NH_S2_SLP + 2), *wjml = nh::scratch2(NH_S2_SLP + 3);
    Grid2 g2 = grid2(d.jpi, d.jpj);
    LAUNCH("ldf_slp", k_slp_mxl<T>, g2, d, in, nmln, hmlpt, z1_slpmax, zsu, zsv, wiml, wjml);
    Grid2 g;
    g.block = dim3(SLP_RX * SLP_RY, 1, 1);
    g.grid = dim3((unsigned)slp_tiles(d.jpi - 2, SLP_RX, d.iper), (unsigned)slp_tiles(d.jpj - 2, SLP_RY, d.jper), 1);
    // levels per workgroup: long marches repeat fewer first levels, short ones
    // fill the chip (two workgroups per CU, 512).  Where four levels each would
    // leave it unfilled, as few as fill it (FP64, four levels and one: 32x22x31
    // 27.3 and 16.6 us, 60x50x40 27.8 and 18.2 us)
    const int tiles = (int)(g.grid.x * g.grid.y), nlev = d.jpk - 2;
    int nz = (1536 + tiles - 1) / tiles;
    nz = nz < 1 ? 1 : nz > (nlev + 3) / 4 ? (nlev + 3) / 4 : nz;
    if ((nlev + nz - 1) / nz > SLP_MAXKB) nz = (nlev + SLP_MAXKB - 1) / SLP_MAXKB;
    int kb = (nlev + nz - 1) / nz;
    const int kfill = (tiles * nlev + 256) / 512;
    if (kfill < 4) kb = kfill < 1 ? 1 : kfill;
    g.grid.z = (unsigned)((nlev + kb - 1) / kb);
#define SLP_LAUNCH(U)                                                                                               \
    LAUNCH("ldf_slp", (k_slp<T, U>), g, d, in, gdept, gdepw, nmln, (const double *)zsu, (const double *)zsv, hmlp, \
           (const double *)wiml, (const double *)wjml, z1_slpmax, kb, uslp, vslp, wslpi, wslpj)
    if (d.e3_sij == 0) SLP_LAUNCH(true);
    else SLP_LAUNCH(false);
#undef SLP_LAUNCH
    return launch_lbc4<T>(uslp, vslp, wslpi, wslpj, d.jpk);
}

#define INST(T)                                                                                                 \
    template int launch_zdf_mxl<T>(const T *, const T *, const T *, int, double, int32_t *, double *, double *); \
    template int launch_ldf_slp<T>(const T *, const T *, const T *, const T *, const int32_t *, const double *,   \
                                   const double *, double, T *, T *, T *, T *);
INST(double)
INST(float)
