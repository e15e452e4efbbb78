// phys.hip -- density (the polynomial TEOS-10 / EOS-80 and the simplified
// equations of state of TRA/eosbn2.F90),
// the hydrostatic pressure gradient in z-coordinates (DYN/dynhpg.F90) and
// the iso-level laplacian viscosity (DYN/dynldf_lap_blp.F90).
//
// Arithmetic is FP64 in both storage forms, rounded once on store, in the
// reference's operation order, so the FP64 form reproduces it bit for bit.
//
// The per-cell kernels of the density multiply by the t- or w-mask.  On domains
// with enough dry waves (DRY, DevDomain::dry) a wave that is dry at its level
// stores the zeros that gives and reads nothing: 512x509x75 FP32 TEOS-10, half of
// it dry, k_rab_poly 154 -> 134 us, k_eos_poly 121 -> 113.  A wet wave then waits
// for its mask before it asks for its operands, which an all-wet domain would pay
// for nothing (600x500x60 FP32, TEOS-10: k_rab_poly 137 -> 160 us, k_eos_poly 107
// -> 122; S-EOS: k_rab 83 -> 95, k_eos 66 -> 83): there the mask is loaded last.
#include "common.hpp"
#include "eos_poly.h"
#include "kernels.hpp"

// {TEOS-10, EOS-80} coefficient tables; a kernel reads one scheme with
// compile-time offsets, so the loads are wave-uniform scalar loads
__constant__ const nemo_eos_poly_t EOS_POLY[2] = NEMO_EOS_POLY_TABLES;

// one depth coefficient (zn0..zn3) of TRA/eosbn2.F90:246-266 / 600-637:
// total degree N in (zs, zt), nested over zt; each zt-power's salinity
// polynomial c0 + zs (c1 + zs (c2 + ...)) adds its constant term last
template <int N>
__device__ __forceinline__ double poly_st(const double (&c)[7][7], double zt, double zs)
{
    double acc = c[N][0];
#pragma unroll
    for (int j = N - 1; j >= 0; j--) {
        double ts = c[j][N - j];
#pragma unroll
        for (int i = N - j - 1; i >= 1; i--) ts = ts * zs + c[j][i];
        acc = acc * zt + ts * zs + c[j][0];
    }
    return acc;
}

// zn = ((zn3 zh + zn2) zh + zn1) zh + zn0 (TRA/eosbn2.F90:268), degrees
// (D0, D1, D2, D3) of the four depth coefficients
template <int D0, int D1, int D2, int D3>
__device__ __forceinline__ double poly_z(const double (&c)[4][7][7], double zt, double zs, double zh, double &zn0)
{
    const double z3 = poly_st<D3>(c[3], zt, zs), z2 = poly_st<D2>(c[2], zt, zs);
    const double z1 = poly_st<D1>(c[1], zt, zs);
    zn0 = poly_st<D0>(c[0], zt, zs);
    return ((z3 * zh + z2) * zh + z1) * zh + zn0;
}

// ---------------------------------------------------------------------------
// eos_insitu (POT = 0), TRA/eosbn2.F90:236-274, and eos_insitu_pot (POT = 1),
// lines 399-437: polynomial TEOS-10 (SCH = 0) / EOS-80 (SCH = 1).  One
// thread per cell, levels 1..jpkm1.
// ---------------------------------------------------------------------------
template <typename T, int POT, int SCH, bool DRY>
KERNEL void k_eos_poly(DevDomain d, const T *__restrict__ pts, T *__restrict__ prd, T *__restrict__ prhop,
                       const T *__restrict__ pdep)
{
    THREAD_IJ(1, 1);
    const int k = (int)blockIdx.z + 1;
    if (i > d.jpi || j > d.jpj) return;
    const nemo_eos_poly_t &P = EOS_POLY[SCH];
    const uint32_t p = IJK32(i, j, k);
    double ztm = 0.;
    if (DRY) ztm = TMASK(double, i, j, k);
    if (DRY && !__any(ztm != 0.)) {
        if (POT) at32(prhop, p) = T(0);
        at32(prd, p) = T(0);
        return;
    }
    const double r1_rau0 = 1.0 / d.rau0;
    const double zh = (double)at32(pdep, p) * P.r1_Z0;
    const double zt = (double)at32(pts, p) * P.r1_T0;
    const double zs = sqrt(fabs((double)at32(pts + d.n3, p) + P.rdeltaS) * P.r1_S0);
    if (!DRY) ztm = TMASK(double, i, j, k);   // after the operands' loads
    double zn0;
    const double zn = poly_z<6, 4, 2, 1>(P.rho, zt, zs, zh, zn0);
    if (POT) at32(prhop, p) = (T)(zn0 * ztm);
    at32(prd, p) = (T)((zn * r1_rau0 - 1.) * ztm);
}

// rab_3d, TRA/eosbn2.F90:588-643: alpha and beta of the polynomial schemes
template <typename T, int SCH, bool DRY>
KERNEL void k_rab_poly(DevDomain d, const T *__restrict__ pts, T *__restrict__ pab, const T *__restrict__ gdept)
{
    THREAD_IJ(1, 1);
    const int k = (int)blockIdx.z + 1;
    if (i > d.jpi || j > d.jpj) return;
    const nemo_eos_poly_t &P = EOS_POLY[SCH];
    const uint32_t p = IJK32(i, j, k);
    double ztm = 0.;
    if (DRY) ztm = TMASK(double, i, j, k);
    if (DRY && !__any(ztm != 0.)) {
        at32(pab, p) = T(0);
        at32(pab + d.n3, p) = T(0);
        return;
    }
    const double r1_rau0 = 1.0 / d.rau0;
    const double zh = (double)at32(gdept, p) * P.r1_Z0;
    const double zt = (double)at32(pts, p) * P.r1_T0;
    const double zs = sqrt(fabs((double)at32(pts + d.n3, p) + P.rdeltaS) * P.r1_S0);
    if (!DRY) ztm = TMASK(double, i, j, k);   // after the operands' loads
    double z0;
    const double za = poly_z<5, 3, 1, 0>(P.alp, zt, zs, zh, z0);
    at32(pab, p) = (T)(za * r1_rau0 * ztm);
    const double zb = poly_z<5, 3, 1, 0>(P.bet, zt, zs, zh, z0);
    at32(pab + d.n3, p) = (T)(zb / zs * r1_rau0 * ztm);
}

// ---------------------------------------------------------------------------
// eos_insitu (POT = 0), TRA/eosbn2.F90:276-299, and eos_insitu_pot (POT = 1),
// lines 440-462, S-EOS.  One thread per cell, levels 1..jpkm1.
// ---------------------------------------------------------------------------
template <typename T, int POT, bool DRY>
KERNEL void k_eos(DevDomain d, SeosPar e, const T *__restrict__ pts, T *__restrict__ prd, T *__restrict__ prhop,
                  const T *__restrict__ pdep)
{
    THREAD_IJ(1, 1);
    const int k = (int)blockIdx.z + 1;
    if (i > d.jpi || j > d.jpj) return;
    const uint32_t p = IJK32(i, j, k);
    double ztm = 0.;
    if (DRY) ztm = TMASK(double, i, j, k);
    if (DRY && !__any(ztm != 0.)) {
        if (POT) at32(prhop, p) = T(0);
        at32(prd, p) = T(0);
        return;
    }
    const double r1_rau0 = 1.0 / d.rau0;
    const double zt = (double)at32(pts, p) - 10.;
    const double zs = (double)at32(pts + d.n3, p) - 35.;
    const double zh = (double)at32(pdep, p);
    if (!DRY) ztm = TMASK(double, i, j, k);
    if (POT) {
        double zn = -e.a0 * (1. + 0.5 * e.lambda1 * zt) * zt + e.b0 * (1. - 0.5 * e.lambda2 * zs) * zs -
                    e.nu * zt * zs;
        at32(prhop, p) = (T)((d.rau0 + zn) * ztm);
        zn = zn - (e.a0 * e.mu1 * zt + e.b0 * e.mu2 * zs) * zh;
        at32(prd, p) = (T)(zn * r1_rau0 * ztm);
    } else {
        const double zn = -e.a0 * (1. + 0.5 * e.lambda1 * zt + e.mu1 * zh) * zt +
                          e.b0 * (1. - 0.5 * e.lambda2 * zs - e.mu2 * zh) * zs - e.nu * zt * zs;
        at32(prd, p) = (T)(zn * r1_rau0 * ztm);
    }
}

// rab_3d, TRA/eosbn2.F90:645-662 (S-EOS): alpha and beta at t-points
template <typename T, bool DRY>
KERNEL void k_rab(DevDomain d, SeosPar e, const T *__restrict__ pts, T *__restrict__ pab,
                  const T *__restrict__ gdept)
{
    THREAD_IJ(1, 1);
    const int k = (int)blockIdx.z + 1;
    if (i > d.jpi || j > d.jpj) return;
    const uint32_t p = IJK32(i, j, k);
    double ztm = 0.;
    if (DRY) ztm = TMASK(double, i, j, k);
    if (DRY && !__any(ztm != 0.)) {
        at32(pab, p) = T(0);
        at32(pab + d.n3, p) = T(0);
        return;
    }
    const double r1_rau0 = 1.0 / d.rau0;
    const double zt = (double)at32(pts, p) - 10.;
    const double zs = (double)at32(pts + d.n3, p) - 35.;
    const double zh = (double)at32(gdept, p);
    if (!DRY) ztm = TMASK(double, i, j, k);
    double zn = e.a0 * (1. + e.lambda1 * zt + e.mu1 * zh) + e.nu * zs;
    at32(pab, p) = (T)(zn * r1_rau0 * ztm);
    zn = e.b0 * (1. - e.lambda2 * zs - e.mu2 * zh) - e.nu * zt;
    at32(pab + d.n3, p) = (T)(zn * r1_rau0 * ztm);
}

// bn2, TRA/eosbn2.F90:914-925: N^2 at w-points 2..jpkm1 (grid.z = jpk - 2)
template <typename T>
KERNEL void k_bn2(DevDomain d, const T *__restrict__ pts, const T *__restrict__ pab, T *__restrict__ pn2,
                  const T *__restrict__ gdept, const T *__restrict__ gdepw)
{
    THREAD_IJ(1, 1);
    const int k = (int)blockIdx.z + 2;
    if (i > d.jpi || j > d.jpj) return;
    const uint32_t p = IJK32(i, j, k), q = IJK32(i, j, k - 1);
    const double wm = WMASK(double, i, j, k);
    if (!__any(wm != 0.)) {
        at32(pn2, p) = T(0);
        return;
    }
    const size_t n3 = d.n3;
    const double gt = (double)at32(gdept, p);
    const double zrw = ((double)at32(gdepw, p) - gt) / ((double)at32(gdept, q) - gt);
    const double zaw = (double)at32(pab, p) * (1. - zrw) + (double)at32(pab, q) * zrw;
    const double zbw = (double)at32(pab + n3, p) * (1. - zrw) + (double)at32(pab + n3, q) * zrw;
    at32(pn2, p) = (T)(d.grav *
                       (zaw * ((double)at32(pts, q) - (double)at32(pts, p)) -
                        zbw * ((double)at32(pts + n3, q) - (double)at32(pts + n3, p))) /
                       E3(d.md.e3w, IJ32(i, j), k) * wm);
}

// ---------------------------------------------------------------------------
// hpg_zco, DYN/dynhpg.F90:286-320: per interior column, the pressure
// gradient integrated from the surface in an FP64 register
// ---------------------------------------------------------------------------
template <typename T>
KERNEL void k_hpg_zco(DevDomain d, const T *__restrict__ rhd, T *__restrict__ ua, T *__restrict__ va)
{
    THREAD_IJ(2, 2);
    if (i > d.jpi - 1 || j > d.jpj - 1) return;
    const Metrics<double> &m = d.md;
    const uint32_t ij = IJ32(i, j), ie = ij + 1u, jn = ij + (uint32_t)d.jpi;
    const size_t plane = d.n2;
    const double zcoef0 = -d.grav * 0.5;
    const double r1u = m.r1_e1u[ij], r1v = m.r1_e2v[ij];
    double zhpi, zhpj;
    {
        const double zcoef1 = zcoef0 * E3(m.e3w, ij, 1);
        const double rc = (double)ldp(rhd, ij);
        zhpi = zcoef1 * ((double)ldp(rhd, ie) - rc) * r1u;
        zhpj = zcoef1 * ((double)ldp(rhd, jn) - rc) * r1v;
        stp(ua, ij, (T)((double)ldp((const T *)ua, ij) + zhpi));
        stp(va, ij, (T)((double)ldp((const T *)va, ij) + zhpj));
    }
    double rc_m = (double)ldp(rhd, ij), re_m = (double)ldp(rhd, ie), rn_m = (double)ldp(rhd, jn);
#pragma unroll 4
    for (int k = 2; k <= d.jpk - 1; k++) {
        const T *r = plane_ptr(rhd, plane, k);
        const double rc = (double)ldp(r, ij), re = (double)ldp(r, ie), rn = (double)ldp(r, jn);
        const double zcoef1 = zcoef0 * E3(m.e3w, ij, k);
        zhpi = zhpi + zcoef1 * ((re + re_m) - (rc + rc_m)) * r1u;
        zhpj = zhpj + zcoef1 * ((rn + rn_m) - (rc + rc_m)) * r1v;
        T *uk = plane_ptr(ua, plane, k), *vk = plane_ptr(va, plane, k);
        stp(uk, ij, (T)((double)ldp((const T *)uk, ij) + zhpi));
        stp(vk, ij, (T)((double)ldp((const T *)vk, ij) + zhpj));
        rc_m = rc;
        re_m = re;
        rn_m = rn;
    }
}

// ---------------------------------------------------------------------------
// dyn_ldf_lap, DYN/dynldf_lap_blp.F90:72-100.  A workgroup marches kb levels
// of a region of LDF_RX x LDF_RY columns, one per thread, whose metrics stay in
// registers: per level a thread shares its metric-weighted velocities through
// LDS, forms the curl at its f-point and the divergence at its t-point from them
// (each as the reference evaluates zcur / zdiv), shares those, and inside the
// region's edge adds both trends.  Each level's fields are loaded one level
// ahead.  Bound by its loads: one level per workgroup read fourteen FP64
// metrics for eight field values per point: 512x509x75 FP32 409 -> 256 us.
// ---------------------------------------------------------------------------
#define LDF_RX 32
#define LDF_RY 16
template <typename T>
__global__ __launch_bounds__(LDF_RX * LDF_RY, 4) void k_dyn_ldf_lap(DevDomain d, double zsign, int kb,
                                                                     const T *__restrict__ pub,
                                                                     const T *__restrict__ pvb, T *__restrict__ pua,
                                                                     T *__restrict__ pva, const T *__restrict__ ahmt,
                                                                     const T *__restrict__ ahmf)
{
    constexpr int N = LDF_RX * LDF_RY;
    __shared__ double sa[N], sb[N], sx[N], sy[N], scur[N], sdiv[N];
    unsigned bx, by;
    xcd_tile(bx, by);
    const int q = (int)threadIdx.x, lx = q % LDF_RX, ly = q / LDF_RX;
    const int i = (int)bx * (LDF_RX - 2) + lx + 1, j = (int)by * (LDF_RY - 2) + ly + 1;   // the region starts at (1, 1)
    const int k0 = 1 + (int)blockIdx.z * kb, k1 = min(k0 + kb - 1, d.jpk - 1);
    const bool own = lx >= 1 && lx < LDF_RX - 1 && ly >= 1 && ly < LDF_RY - 1 && i <= d.jpi - 1 && j <= d.jpj - 1;
    const uint32_t c = IJ32(min(i, d.jpi), min(j, d.jpj));   // columns off the domain repeat its edge, unused
    const Metrics<double> &m = d.md;
    const double e2v = m.e2v[c], e1u = m.e1u[c], e2u = m.e2u[c], e1v = m.e1v[c];
    const double r1_e1e2f = m.r1_e1e2f[c], r1_e1e2t = m.r1_e1e2t[c];
    const double r1_e2u = m.r1_e2u[c], r1_e1u = m.r1_e1u[c], r1_e1v = m.r1_e1v[c], r1_e2v = m.r1_e2v[c];
    // neighbours in the region (the region's edge points use their own value, unused)
    const int qe = lx < LDF_RX - 1 ? q + 1 : q, qw = lx > 0 ? q - 1 : q;
    const int qn = ly < LDF_RY - 1 ? q + LDF_RX : q, qs = ly > 0 ? q - LDF_RX : q;
    struct Lv {
        T u, v, at, af, ua, va;
    };
    const auto fetch = [&](int k, Lv &l) {
        l.u = ldp(plane_ptr(pub, d.n2, k), c);
        l.v = ldp(plane_ptr(pvb, d.n2, k), c);
        l.at = ldp(plane_ptr(ahmt, d.n2, k), c);
        l.af = ldp(plane_ptr(ahmf, d.n2, k), c);
        if (own) {
            l.ua = ldp((const T *)plane_ptr(pua, d.n2, k), c);
            l.va = ldp((const T *)plane_ptr(pva, d.n2, k), c);
        }
    };
    Lv cur{}, nxt{};
    fetch(k0, cur);
    for (int k = k0; k <= k1; k++) {
        fetch(min(k + 1, k1), nxt);
        const double u = (double)cur.u, v = (double)cur.v;
        const double a = e2v * v, b = e1u * u;
        const double x = e2u * E3(m.e3u, c, k) * u, y = e1v * E3(m.e3v, c, k) * v;
        sa[q] = a;
        sb[q] = b;
        sx[q] = x;
        sy[q] = y;
        __syncthreads();
        const double zcur = (double)cur.af * E3(m.e3f, c, k) * r1_e1e2f * (sa[qe] - a - sb[qn] + b);
        const double zdiv = (double)cur.at * r1_e1e2t / E3(m.e3t, c, k) * (x - sx[qw] + y - sy[qs]);
        scur[q] = zcur;
        sdiv[q] = zdiv;
        __syncthreads();
        if (own) {
            stp(plane_ptr(pua, d.n2, k), c,
                (T)((double)cur.ua + zsign * (-((zcur - scur[qs]) * r1_e2u / E3(m.e3u, c, k)) + (sdiv[qe] - zdiv) * r1_e1u)));
            stp(plane_ptr(pva, d.n2, k), c,
                (T)((double)cur.va + zsign * ((zcur - scur[qw]) * r1_e1v / E3(m.e3v, c, k) + (sdiv[qn] - zdiv) * r1_e2v)));
        }
        cur = nxt;
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <typename T, bool DRY>
static int launch_eos_d(int neos, const SeosPar &e, int pot, const T *pts, T *prd, T *prhop, const T *pdep)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    g.grid.z = (unsigned)(d.jpk - 1);
    if (neos == NEMO_NP_TEOS10) {
        if (pot) LAUNCH("eos", (k_eos_poly<T, 1, NEMO_EOS_POLY_TEOS10, DRY>), g, d, pts, prd, prhop, pdep);
        else LAUNCH("eos", (k_eos_poly<T, 0, NEMO_EOS_POLY_TEOS10, DRY>), g, d, pts, prd, prhop, pdep);
    } else if (neos == NEMO_NP_EOS80) {
        if (pot) LAUNCH("eos", (k_eos_poly<T, 1, NEMO_EOS_POLY_EOS80, DRY>), g, d, pts, prd, prhop, pdep);
        else LAUNCH("eos", (k_eos_poly<T, 0, NEMO_EOS_POLY_EOS80, DRY>), g, d, pts, prd, prhop, pdep);
    } else {
        if (pot) LAUNCH("eos", (k_eos<T, 1, DRY>), g, d, e, pts, prd, prhop, pdep);
        else LAUNCH("eos", (k_eos<T, 0, DRY>), g, d, e, pts, prd, prhop, pdep);
    }
    return 0;
}
template <typename T>
int launch_eos(int neos, const SeosPar &e, int pot, const T *pts, T *prd, T *prhop, const T *pdep)
{
    return nh::dom().dry ? launch_eos_d<T, true>(neos, e, pot, pts, prd, prhop, pdep)
                         : launch_eos_d<T, false>(neos, e, pot, pts, prd, prhop, pdep);
}

template <typename T, bool DRY>
static int launch_rab_d(int neos, const SeosPar &e, const T *pts, T *pab, const T *gdept)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    g.grid.z = (unsigned)(d.jpk - 1);
    if (neos == NEMO_NP_TEOS10) LAUNCH("rab", (k_rab_poly<T, NEMO_EOS_POLY_TEOS10, DRY>), g, d, pts, pab, gdept);
    else if (neos == NEMO_NP_EOS80) LAUNCH("rab", (k_rab_poly<T, NEMO_EOS_POLY_EOS80, DRY>), g, d, pts, pab, gdept);
    else LAUNCH("rab", (k_rab<T, DRY>), g, d, e, pts, pab, gdept);
    return 0;
}
template <typename T>
int launch_rab(int neos, const SeosPar &e, const T *pts, T *pab, const T *gdept)
{
    return nh::dom().dry ? launch_rab_d<T, true>(neos, e, pts, pab, gdept) : launch_rab_d<T, false>(neos, e, pts, pab, gdept);
}

template <typename T>
int launch_bn2(const T *pts, const T *pab, T *pn2, const T *gdept, const T *gdepw)
{
    const DevDomain &d = nh::dom();
    if (d.jpk < 3) return 0;
    Grid2 g = grid2(d.jpi, d.jpj);
    g.grid.z = (unsigned)(d.jpk - 2);
    LAUNCH("bn2", k_bn2<T>, g, d, pts, pab, pn2, gdept, gdepw);
    return 0;
}

template <typename T>
int launch_hpg_zco(const T *rhd, T *ua, T *va)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi - 2, d.jpj - 2);
    LAUNCH("dyn_hpg", k_hpg_zco<T>, g, d, rhd, ua, va);
    return 0;
}

template <typename T>
int launch_dyn_ldf_lap(double zsign, const T *pub, const T *pvb, T *pua, T *pva, const T *ahmt, const T *ahmf)
{
    const DevDomain &d = nh::dom();
    Grid2 g;
    g.block = dim3(LDF_RX * LDF_RY, 1, 1);
    g.grid = dim3((unsigned)((d.jpi - 2 + LDF_RX - 3) / (LDF_RX - 2)), (unsigned)((d.jpj - 2 + LDF_RY - 3) / (LDF_RY - 2)), 1);
    // levels per workgroup: two rounds of the two workgroups that fit a CU (1024),
    // the metrics read once for up to 16 levels.  (At four rounds
    // 1500x40x40 FP64 took 62 us and 251x233x20 35, slower than a workgroup per
    // level of a 64x4 tile, 50 and 28; now 45 and 28)
    const int tiles = (int)(g.grid.x * g.grid.y), nlev = d.jpk - 1;
    int kb = (int)(((long)tiles * nlev + 512) / 1024);
    kb = kb < 1 ? 1 : kb > 16 ? 16 : kb;
    g.grid.z = (unsigned)((nlev + kb - 1) / kb);
    LAUNCH("dyn_ldf", k_dyn_ldf_lap<T>, g, d, zsign, kb, pub, pvb, pua, pva, ahmt, ahmf);
    return 0;
}

#define INST(T)                                                                                      \
    template int launch_eos<T>(int, const SeosPar &, int, const T *, T *, T *, const T *);            \
    template int launch_rab<T>(int, const SeosPar &, const T *, T *, const T *);                      \
    template int launch_bn2<T>(const T *, const T *, T *, const T *, const T *);                      \
    template int launch_hpg_zco<T>(const T *, T *, T *);                                              \
    template int launch_dyn_ldf_lap<T>(double, const T *, const T *, T *, T *, const T *, const T *);
INST(double)
INST(float)
#undef INST
