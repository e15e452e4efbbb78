// dyn.hip -- momentum operators of the ocean time step on gfx950.
//
//   dyn_keg       DYN/dynkeg.F90:46-192    kinetic-energy gradient (C2, Hollingsworth)
//   dyn_zad       DYN/dynzad.F90:38-121    vertical advection (vector form)
//   dyn_adv_cen2  DYN/dynadv_cen2.F90:37-144 flux-form advection
//   dyn_vor       DYN/dynvor.F90:98-828    vorticity: ENS, ENE, MIX, ENT, EET, EEN
//   dyn_zdf       DYN/dynzdf.F90:47-499    implicit vertical diffusion + drag
//
// Same conventions as tra.hip: one thread per (i,j) column, k-marched,
// coalesced along i; the lbc_lnk fills that separate reference loop nests
// are folded in through lbc_src; expression order follows the reference.
#include "common.hpp"
#include "kernels.hpp"

enum { np_COR = 1, np_RVO = 2, np_MET = 3, np_CRV = 4, np_CME = 5 };

// ---------------------------------------------------------------------------
// vector-form advection, dyn_keg then dyn_zad, fused per element
// (ua <- (ua - keg) - zad, the order of the two reference calls)
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T keg_c2(const DevDomain &d, const T *un, const T *vn, int p, int q, int k)
{
    const T u1 = A3(un, p - 1, q, k), u2 = A3(un, p, q, k), v1 = A3(vn, p, q - 1, k), v2 = A3(vn, p, q, k);
    const T zu = u1 * u1 + u2 * u2;
    const T zv = v1 * v1 + v2 * v2;
    return T(0.25) * (zv + zu);
}
template <typename T>
__device__ __forceinline__ T keg_hw(const DevDomain &d, const T *un, const T *vn, int p, int q, int k)
{
    int sp, sq;
    if (!lbc_src(d, 'T', p, q, sp, sq)) return T(0);     // lbc_lnk('dynkeg', zhke, 'T')
    p = sp;
    q = sq;
    const T r1_48 = T(1) / T(48);
    const T a = A3(un, p - 1, q - 1, k) + A3(un, p - 1, q + 1, k);
    const T b = A3(un, p, q - 1, k) + A3(un, p, q + 1, k);
    const T u1 = A3(un, p - 1, q, k), u2 = A3(un, p, q, k);
    const T zu = T(8) * (u1 * u1 + u2 * u2) + a * a + b * b;
    const T c = A3(vn, p - 1, q - 1, k) + A3(vn, p + 1, q - 1, k);
    const T e = A3(vn, p - 1, q, k) + A3(vn, p + 1, q, k);
    const T v1 = A3(vn, p, q - 1, k), v2 = A3(vn, p, q, k);
    const T zv = T(8) * (v1 * v1 + v2 * v2) + c * c + e * e;
    return r1_48 * (zv + zu);
}

// How the levels of a launch of nb workgroups per level chunk are shared out: the
// whole column per workgroup where that gives every SIMD its waves (512
// workgroups and more), else chunks of four levels or more towards 768 workgroups.
// (32x22x31 FP64, five workgroups: k_step_dyn1 34 us in one chunk, 17 us
// with its sums.)  In a plan the launch holds every member's workgroups: several
// members fill the chip without chunks, and the plan does not know their number
// when it traces one, so none are made.  A plan of one or two members is left
// short of workgroups by that (whole steps, separate calls and plan: one 32x22x31
// FP64 271 and 471 us, one 182x149x56 FP32 508 and 826; two gyres 577 and 530;
// six small members 2084 and 666).
inline int lev_chunks(unsigned nb, int nlev)
{
    if (nh::planning() || nb >= 512u || nb == 0u) return nlev;
    int n = (int)(768u / nb);
    n = n > nlev / 4 ? nlev / 4 : n;
    return n < 1 ? nlev : (nlev + n - 1) / n;
}

// One thread per column and chunk of kch levels (grid.z).
template <typename T>
struct S_dyn_keg_zad {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, int do_keg, int kscheme, int do_zad, const T * __restrict__ un, const T * __restrict__ vn, const T * __restrict__ wn, T * __restrict__ ua, T * __restrict__ va, int kch)
    {
        THREAD_IJ_V(vb_, 2, 2);
        if (i > d.jpi - 1 || j > d.jpj - 1) return;
        const Metrics<T> &m = met<T>(d);
        const size_t ij = IJ(i, j);
        const T e1u = m.e1u[ij], e2v = m.e2v[ij], r1_e1e2u = m.r1_e1e2u[ij], r1_e1e2v = m.r1_e1e2v[ij];
        const T e1e2t = m.e1e2t[ij], e1e2t_e = m.e1e2t[IJ(i + 1, j)], e1e2t_n = m.e1e2t[IJ(i, j + 1)];
        const int ka = (int)vb_.z * kch + 1, kb = min(ka + kch - 1, d.jpk - 1);
        // dynzad's fluxes at w-level kk (zero at the surface, dynzad.F90:93-94)
        const auto wflux = [&](int kk, T &cu, T &cv) {
            cu = cv = T(0);
            if (kk == 1 || kk > d.jpk - 1) return;
            const T zww = T(0.25) * e1e2t * A3(wn, i, j, kk);
            const T zww_e = T(0.25) * e1e2t_e * A3(wn, i + 1, j, kk);
            const T zww_n = T(0.25) * e1e2t_n * A3(wn, i, j + 1, kk);
            cu = (zww_e + zww) * (A3(un, i, j, kk - 1) - A3(un, i, j, kk));
            cv = (zww_n + zww) * (A3(vn, i, j, kk - 1) - A3(vn, i, j, kk));
        };
        T zwuw_k = T(0), zwvw_k = T(0);
        if (do_zad) wflux(ka, zwuw_k, zwvw_k);
        for (int k = ka; k <= kb; k++) {
            const size_t p = IJK(i, j, k);
            T a = ua[p], b = va[p];
            if (do_keg) {
                T h, he, hn;
                if (kscheme == 0) {
                    h = keg_c2(d, un, vn, i, j, k);
                    he = keg_c2(d, un, vn, i + 1, j, k);
                    hn = keg_c2(d, un, vn, i, j + 1, k);
                } else {
                    h = keg_hw(d, un, vn, i, j, k);
                    he = keg_hw(d, un, vn, i + 1, j, k);
                    hn = keg_hw(d, un, vn, i, j + 1, k);
                }
                a = a - (he - h) / e1u;
                b = b - (hn - h) / e2v;
            }
            if (do_zad) {
                T zwuw_kp1, zwvw_kp1;
                wflux(k + 1, zwuw_kp1, zwvw_kp1);
                a = a - (zwuw_k + zwuw_kp1) * r1_e1e2u / E3(m.e3u, ij, k);
                b = b - (zwvw_k + zwvw_kp1) * r1_e1e2v / E3(m.e3v, ij, k);
                zwuw_k = zwuw_kp1;
                zwvw_k = zwvw_kp1;
            }
            ua[p] = a;
            va[p] = b;
        }
    }
};
template <typename T>
KERNEL void k_dyn_keg_zad(DevDomain d, int do_keg, int kscheme, int do_zad, const T * __restrict__ un, const T * __restrict__ vn, const T * __restrict__ wn,
                              T * __restrict__ ua, T * __restrict__ va, int kch)
{
    S_dyn_keg_zad<T>::run(vb_hw(), d, do_keg, kscheme, do_zad, un, vn, wn, ua, va, kch);
}

// ---------------------------------------------------------------------------
// dyn_adv_cen2, horizontal then vertical flux divergence per element
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T cen2_zfu(const DevDomain &d, const T *un, int p, int q, int k)
{
    const Metrics<T> &m = met<T>(d);
    const size_t pq = IJ(p, q);
    return T(0.25) * m.e2u[pq] * E3(m.e3u, pq, k) * A3(un, p, q, k);
}
template <typename T>
__device__ __forceinline__ T cen2_zfv(const DevDomain &d, const T *vn, int p, int q, int k)
{
    const Metrics<T> &m = met<T>(d);
    const size_t pq = IJ(p, q);
    return T(0.25) * m.e1v[pq] * E3(m.e3v, pq, k) * A3(vn, p, q, k);
}
template <typename T>
__device__ __forceinline__ T cen2_zfw(const DevDomain &d, const T *wn, int p, int q, int k)
{
    return T(0.25) * met<T>(d).e1e2t[IJ(p, q)] * A3(wn, p, q, k);
}

template <typename T>
struct S_dyn_adv_cen2 {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, const T * __restrict__ un, const T * __restrict__ vn, const T * __restrict__ wn, T * __restrict__ ua, T * __restrict__ va)
    {
        THREAD_IJ_V(vb_, 2, 2);
        if (i > d.jpi - 1 || j > d.jpj - 1) return;
        const Metrics<T> &m = met<T>(d);
        const size_t ij = IJ(i, j);
        const T r1_e1e2u = m.r1_e1e2u[ij], r1_e1e2v = m.r1_e1e2v[ij];
        const int jpk = d.jpk;
        // surface fluxes (linear free surface), dynadv_cen2.F90:105-112
        T zfu_uw_k = T(0.5) * (m.e1e2t[ij] * A3(wn, i, j, 1) + m.e1e2t[IJ(i + 1, j)] * A3(wn, i + 1, j, 1)) * A3(un, i, j, 1);
        T zfv_vw_k = T(0.5) * (m.e1e2t[ij] * A3(wn, i, j, 1) + m.e1e2t[IJ(i, j + 1)] * A3(wn, i, j + 1, 1)) * A3(vn, i, j, 1);
        for (int k = 1; k <= jpk - 1; k++) {
            // horizontal: zfu_t(i+1), zfu_t(i), zfv_f(i,j), zfv_f(i,j-1)
            const T fu_im1 = cen2_zfu(d, un, i - 1, j, k), fu_i = cen2_zfu(d, un, i, j, k), fu_ip1 = cen2_zfu(d, un, i + 1, j, k);
            const T fu_jp1 = cen2_zfu(d, un, i, j + 1, k), fu_im1jp1 = cen2_zfu(d, un, i - 1, j + 1, k);
            const T fv_i = cen2_zfv(d, vn, i, j, k), fv_ip1 = cen2_zfv(d, vn, i + 1, j, k);
            const T fv_jm1 = cen2_zfv(d, vn, i, j - 1, k), fv_ip1jm1 = cen2_zfv(d, vn, i + 1, j - 1, k);
            const T fv_jp1 = cen2_zfv(d, vn, i, j + 1, k), fv_im1 = cen2_zfv(d, vn, i - 1, j, k);
            const T u_i = A3(un, i, j, k), u_ip1 = A3(un, i + 1, j, k), u_im1 = A3(un, i - 1, j, k);
            const T u_jp1 = A3(un, i, j + 1, k), u_jm1 = A3(un, i, j - 1, k);
            const T v_j = A3(vn, i, j, k), v_ip1 = A3(vn, i + 1, j, k), v_jp1 = A3(vn, i, j + 1, k);
            const T v_im1 = A3(vn, i - 1, j, k), v_jm1 = A3(vn, i, j - 1, k);
            const T zfu_t_ip1 = (fu_i + fu_ip1) * (u_i + u_ip1);
            const T zfu_t_i = (fu_im1 + fu_i) * (u_im1 + u_i);
            const T zfv_f_j = (fv_i + fv_ip1) * (u_i + u_jp1);
            const T zfv_f_jm1 = (fv_jm1 + fv_ip1jm1) * (u_jm1 + u_i);
            const T zfu_f_i = (fu_i + fu_jp1) * (v_j + v_ip1);
            const T zfu_f_im1 = (fu_im1 + fu_im1jp1) * (v_im1 + v_j);
            const T zfv_t_jp1 = (fv_i + fv_jp1) * (v_j + v_jp1);
            const T zfv_t_j = (fv_jm1 + fv_i) * (v_jm1 + v_j);
            const size_t p = IJK(i, j, k);
            T a = ua[p] - (zfu_t_ip1 - zfu_t_i + zfv_f_j - zfv_f_jm1) * r1_e1e2u / E3(m.e3u, ij, k);
            T b = va[p] - (zfu_f_i - zfu_f_im1 + zfv_t_jp1 - zfv_t_j) * r1_e1e2v / E3(m.e3v, ij, k);
            // vertical, dynadv_cen2.F90:113-133
            T zfu_uw_kp1 = T(0), zfv_vw_kp1 = T(0);
            if (k + 1 <= jpk - 1) {
                const int kk = k + 1;
                const T fw = cen2_zfw(d, wn, i, j, kk);
                zfu_uw_kp1 = (fw + cen2_zfw(d, wn, i + 1, j, kk)) * (A3(un, i, j, kk) + A3(un, i, j, kk - 1));
                zfv_vw_kp1 = (fw + cen2_zfw(d, wn, i, j + 1, kk)) * (A3(vn, i, j, kk) + A3(vn, i, j, kk - 1));
            }
            a = a - (zfu_uw_k - zfu_uw_kp1) * r1_e1e2u / E3(m.e3u, ij, k);
            b = b - (zfv_vw_k - zfv_vw_kp1) * r1_e1e2v / E3(m.e3v, ij, k);
            ua[p] = a;
            va[p] = b;
            zfu_uw_k = zfu_uw_kp1;
            zfv_vw_k = zfv_vw_kp1;
        }
    }
};
template <typename T>
KERNEL void k_dyn_adv_cen2(DevDomain d, const T * __restrict__ un, const T * __restrict__ vn, const T * __restrict__ wn, T * __restrict__ ua, T * __restrict__ va)
{
    S_dyn_adv_cen2<T>::run(vb_hw(), d, un, vn, wn, ua, va);
}

template <typename T>
int launch_dyn_adv(int which, int kscheme, const T *un, const T *vn, const T *wn, T *ua, T *va)
{
    // which: 1 keg only, 2 zad only, 3 keg+zad (vector form), 4 cen2
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi - 2, d.jpj - 2);
    if (which == 4) {
        LAUNCHB("dyn_adv_cen2", k_dyn_adv_cen2<T>, (S_dyn_adv_cen2<T>), g, d, un, vn, wn, ua, va);
    } else {
        const char *nm = which == 1 ? "dyn_keg" : which == 2 ? "dyn_zad" : "dyn_adv";
        const int kch = lev_chunks(g.grid.x * g.grid.y, d.jpk - 1);
        g.grid.z = (unsigned)((d.jpk - 1 + kch - 1) / kch);
        LAUNCHB(nm, k_dyn_keg_zad<T>, (S_dyn_keg_zad<T>), g, d, (which & 1), kscheme, (which & 2) ? 1 : 0, un, vn, wn, ua, va, kch);
    }
    return 0;
}
template int launch_dyn_adv<double>(int, int, const double *, const double *, const double *, double *, double *);
template int launch_dyn_adv<float>(int, int, const float *, const float *, const float *, float *, float *);

// ---------------------------------------------------------------------------
// vorticity term
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T curl_f(const DevDomain &d, const T *pu, const T *pv, int p, int q, int k)
{
    const Metrics<T> &m = met<T>(d);
    return m.e2v[IJ(p + 1, q)] * A3(pv, p + 1, q, k) - m.e2v[IJ(p, q)] * A3(pv, p, q, k) -
           m.e1u[IJ(p, q + 1)] * A3(pu, p, q + 1, k) + m.e1u[IJ(p, q)] * A3(pu, p, q, k);
}
// f-point vorticity of vor_ene / vor_ens / vor_eeT (before any lbc), p<=jpim1, q<=jpjm1
template <typename T>
__device__ __forceinline__ T fvor(const DevDomain &d, int kvor, const T *pu, const T *pv, int p, int q, int k)
{
    const Metrics<T> &m = met<T>(d);
    const size_t pq = IJ(p, q);
    switch (kvor) {
    case np_COR: return m.ff_f[pq];
    case np_RVO: return curl_f(d, pu, pv, p, q, k) * m.r1_e1e2f[pq];
    case np_MET:
        return (A3(pv, p + 1, q, k) + A3(pv, p, q, k)) * m.di_e2v_2e1e2f[pq] -
               (A3(pu, p, q + 1, k) + A3(pu, p, q, k)) * m.dj_e1u_2e1e2f[pq];
    case np_CRV: return m.ff_f[pq] + curl_f(d, pu, pv, p, q, k) * m.r1_e1e2f[pq];
    default:
        return m.ff_f[pq] + (A3(pv, p + 1, q, k) + A3(pv, p, q, k)) * m.di_e2v_2e1e2f[pq] -
               (A3(pu, p, q + 1, k) + A3(pu, p, q, k)) * m.dj_e1u_2e1e2f[pq];
    }
}
// zwz of the ENT scheme (relative vorticity) after lbc_lnk('F')
template <typename T>
__device__ __forceinline__ T zwz_ent(const DevDomain &d, const T *pu, const T *pv, int p, int q, int k)
{
    int sp, sq;
    if (!lbc_src(d, 'F', p, q, sp, sq)) return T(0);
    return curl_f(d, pu, pv, sp, sq, k) * met<T>(d).r1_e1e2f[IJ(sp, sq)];
}

// zwz of the EEN and EET schemes after lbc_lnk('F') (vorticity, for EEN times
// 1/e3f: DYN/dynvor.F90:580-643, 700-760) at the f-points around a workgroup's
// 64 x 4 cells, one level at a time, in LDS.  A cell needs eight of them, each
// with a division, four masks and eight loads: evaluated by every cell they took
// 256 registers (one wave per SIMD) and eight times the work; here 1.55 times,
// with the columns' metrics and masks in registers and the next level's
// velocities in flight.  362x149x46 FP64 in k_step_dyn1: 333 us, 97 us;
// 182x149x31 FP32 in k_dyn_vor: 226 us, 17.5 us (both with the levels shared
// out over workgroups, lev_chunks).
template <typename T, int SCHEME, int KVOR>
struct ZwzTile {
    static constexpr int TX = 64, W = TX + 2, H = NH_BLOCK / TX + 2, NR = (W * H + NH_BLOCK - 1) / NH_BLOCK;
    static constexpr bool CURL = KVOR == np_RVO || KVOR == np_CRV, FF = KVOR == np_COR || KVOR == np_CRV || KVOR == np_CME;
    static constexpr bool EEN = SCHEME == NEMO_NP_EEN;
    typedef T Lds[2][H][W];
    uint32_t pq[NR], t1[NR], t2[NR], t3[NR], t4[NR];
    T ff[NR], ve[NR], vc[NR], un[NR], uc[NR], r1f[NR];   // f; curl: e2v, e1u; else di, dj in ve, un
    T u0[NR], u1[NR], v0[NR], v1[NR];                    // the velocities of the next level
    bool ok[NR];

    __device__ __forceinline__ static int tid() { return (int)(threadIdx.y * TX + threadIdx.x); }
    // (i0, j0): the workgroup's first cell
    __device__ __forceinline__ ZwzTile(const DevDomain &d, int i0, int j0)
    {
        const Metrics<T> &m = met<T>(d);
        const uint32_t w = (uint32_t)d.jpi;
    #pragma unroll
        for (int r = 0; r < NR; r++) {
            const int n = tid() + r * NH_BLOCK, p = i0 - 1 + n % W, q = j0 - 1 + n / W;
            int sp = 2, sq = 2;
            ok[r] = n < W * H && p >= 1 && p <= d.jpi && q >= 1 && q <= d.jpj && lbc_src(d, 'F', p, q, sp, sq);
            const uint32_t c = ok[r] ? IJ32(sp, sq) : IJ32(2, 2);
            pq[r] = c;
            if (EEN) {
                t1[r] = d.ktu[c + w]; t2[r] = d.ktu[c + w + 1u]; t3[r] = d.ktu[c]; t4[r] = d.ktu[c + 1u];
            }
            if (FF) ff[r] = m.ff_f[c];
            if (CURL) {
                ve[r] = m.e2v[c + 1u]; vc[r] = m.e2v[c]; un[r] = m.e1u[c + w]; uc[r] = m.e1u[c];
                r1f[r] = m.r1_e1e2f[c];
            } else if (KVOR != np_COR) {
                ve[r] = m.di_e2v_2e1e2f[c]; un[r] = m.dj_e1u_2e1e2f[c];
            }
        }
    }
    // the deepest wet level around the workgroup's f-points (EEN: zwz is zero
    // below); s: a word of LDS.  Ends with a barrier.
    __device__ __forceinline__ int bottom(int *s) const
    {
        if (tid() == 0) *s = 0;
        __syncthreads();
        int k = 0;
    #pragma unroll
        for (int r = 0; r < NR; r++)
            if (ok[r]) k = max(k, (int)max(max((t1[r] >> 8) & 255u, (t2[r] >> 8) & 255u), max((t3[r] >> 8) & 255u, (t4[r] >> 8) & 255u)));
        atomicMax(s, k);
        __syncthreads();
        return *s;
    }
    __device__ __forceinline__ void fetch(const DevDomain &d, const T *pu, const T *pv, int k)
    {
        if (KVOR == np_COR) return;
        const T *u = plane_ptr(pu, d.n2, k), *v = plane_ptr(pv, d.n2, k);
    #pragma unroll
        for (int r = 0; r < NR; r++) {
            u0[r] = ldp(u, pq[r]); u1[r] = ldp(u, pq[r] + (uint32_t)d.jpi);
            v0[r] = ldp(v, pq[r]); v1[r] = ldp(v, pq[r] + 1u);
        }
    }
    __device__ __forceinline__ T vor(int r) const
    {
        if (KVOR == np_COR) return ff[r];
        if (CURL) {
            const T c = ve[r] * v1[r] - vc[r] * v0[r] - un[r] * u1[r] + uc[r] * u0[r];
            return KVOR == np_RVO ? c * r1f[r] : ff[r] + c * r1f[r];
        }
        if (KVOR == np_MET) return (v1[r] + v0[r]) * ve[r] - (u1[r] + u0[r]) * un[r];
        return ff[r] + (v1[r] + v0[r]) * ve[r] - (u1[r] + u0[r]) * un[r];
    }
    // level k from the fetched velocities
    __device__ __forceinline__ void put(const DevDomain &d, int k, Lds &z) const
    {
        const T *e3t = met<T>(d).e3t;
        const bool uni = d.e3_sij == 0;
        const uint32_t w = (uint32_t)d.jpi;
    #pragma unroll
        for (int r = 0; r < NR; r++) {
            T x = T(0);
            if constexpr (EEN) {
                const auto in = [&](uint32_t t) { return k >= (int)(t & 255u) && k <= (int)((t >> 8) & 255u) ? T(1) : T(0); };
                const T m1 = in(t1[r]), m2 = in(t2[r]), m3 = in(t3[r]), m4 = in(t4[r]), n = m1 + m2 + m3 + m4;
                if (ok[r] && n != T(0)) {
                    T ze3f;
                    if (uni) {
                        const T e = uld(e3t, k - 1);
                        ze3f = e * m1 + e * m2 + e * m3 + e * m4;
                    } else {
                        ze3f = E3(e3t, pq[r] + w, k) * m1 + E3(e3t, pq[r] + w + 1u, k) * m2 + E3(e3t, pq[r], k) * m3 +
                               E3(e3t, pq[r] + 1u, k) * m4;
                    }
                    T z1 = T(0);
                    if (ze3f != T(0)) z1 = (d.nn_een_e3f == 0 ? T(4) : n) / ze3f;
                    x = vor(r) * z1;
                }
            } else {
                if (ok[r]) x = vor(r);
            }
            const int q = tid() + r * NH_BLOCK;
            if (q < W * H) z[k & 1][q / W][q % W] = x;
        }
    }
};

template <typename T>
__device__ __forceinline__ void vor_ene_pt(const DevDomain &d, int kvor, const T *pu, const T *pv, int i, int j, int k,
                                           T &a, T &b)
{
    const Metrics<T> &m = met<T>(d);
    const T zy1 = m.e1v[IJ(i, j - 1)] * A3(pv, i, j - 1, k) + m.e1v[IJ(i + 1, j - 1)] * A3(pv, i + 1, j - 1, k);
    const T zy2 = m.e1v[IJ(i, j)] * A3(pv, i, j, k) + m.e1v[IJ(i + 1, j)] * A3(pv, i + 1, j, k);
    const T zx1 = m.e2u[IJ(i - 1, j)] * A3(pu, i - 1, j, k) + m.e2u[IJ(i - 1, j + 1)] * A3(pu, i - 1, j + 1, k);
    const T zx2 = m.e2u[IJ(i, j)] * A3(pu, i, j, k) + m.e2u[IJ(i, j + 1)] * A3(pu, i, j + 1, k);
    const T z_s = fvor(d, kvor, pu, pv, i, j - 1, k), z_c = fvor(d, kvor, pu, pv, i, j, k),
            z_w = fvor(d, kvor, pu, pv, i - 1, j, k);
    const T r1_4 = T(0.25);
    a = a + r1_4 * m.r1_e1u[IJ(i, j)] * (z_s * zy1 + z_c * zy2);
    b = b - r1_4 * m.r1_e2v[IJ(i, j)] * (z_w * zx1 + z_c * zx2);
}
template <typename T>
__device__ __forceinline__ void vor_ens_pt(const DevDomain &d, int kvor, const T *pu, const T *pv, int i, int j, int k,
                                           T &a, T &b)
{
    const Metrics<T> &m = met<T>(d);
    const T r1_8 = T(0.125);
    const T zuav = r1_8 * m.r1_e1u[IJ(i, j)] *
                   (m.e1v[IJ(i, j - 1)] * A3(pv, i, j - 1, k) + m.e1v[IJ(i + 1, j - 1)] * A3(pv, i + 1, j - 1, k) +
                    m.e1v[IJ(i, j)] * A3(pv, i, j, k) + m.e1v[IJ(i + 1, j)] * A3(pv, i + 1, j, k));
    const T zvau = -(r1_8 * m.r1_e2v[IJ(i, j)] *
                     (m.e2u[IJ(i - 1, j)] * A3(pu, i - 1, j, k) + m.e2u[IJ(i - 1, j + 1)] * A3(pu, i - 1, j + 1, k) +
                      m.e2u[IJ(i, j)] * A3(pu, i, j, k) + m.e2u[IJ(i, j + 1)] * A3(pu, i, j + 1, k)));
    const T z_s = fvor(d, kvor, pu, pv, i, j - 1, k), z_c = fvor(d, kvor, pu, pv, i, j, k),
            z_w = fvor(d, kvor, pu, pv, i - 1, j, k);
    a = a + zuav * (z_s + z_c);
    b = b + zvau * (z_w + z_c);
}
// EEN (use_e3f) and EET: triads of f-point vorticity around t-points.  The
// metrics of a cell's four u- and four v-points stay in registers: loaded in the
// level loop they would be loads again, since the kernel stores.
template <typename T>
struct EenCol {
    T yc, ye, ys, yse, xw, xnw, xc, xn, ru, rv;
    __device__ __forceinline__ EenCol(const DevDomain &d, uint32_t c)
    {
        const Metrics<T> &m = met<T>(d);
        const uint32_t w = (uint32_t)d.jpi;
        yc = m.e1v[c]; ye = m.e1v[c + 1u]; ys = m.e1v[c - w]; yse = m.e1v[c - w + 1u];
        xw = m.e2u[c - 1u]; xnw = m.e2u[c + w - 1u]; xc = m.e2u[c]; xn = m.e2u[c + w];
        const T r1_12 = T(1) / T(12);
        ru = r1_12 * m.r1_e1u[c];
        rv = r1_12 * m.r1_e2v[c];
    }
};
// (x, y): the cell within the workgroup; z: the level's f-points (ZwzTile)
template <typename T, int SCHEME, int W>
__device__ __forceinline__ void vor_een_pt(const DevDomain &d, const EenCol<T> &e, const T (*z)[W], int x, int y,
                                           const T *pu, const T *pv, uint32_t c, int k, T &a, T &b)
{
    const Metrics<T> &m = met<T>(d);
    const uint32_t w = (uint32_t)d.jpi;
    const T *u = plane_ptr(pu, d.n2, k), *v = plane_ptr(pv, d.n2, k);
#define ZW(di, dj) z[y + (dj) + 1][x + (di) + 1]
    // triads at t-point (i+oi, j+oj)
    auto tne = [&](int oi, int oj) { return ZW(oi - 1, oj) + ZW(oi, oj) + ZW(oi, oj - 1); };
    auto tnw = [&](int oi, int oj) { return ZW(oi - 1, oj - 1) + ZW(oi - 1, oj) + ZW(oi, oj); };
    auto tse = [&](int oi, int oj) { return ZW(oi, oj) + ZW(oi, oj - 1) + ZW(oi - 1, oj - 1); };
    auto tsw = [&](int oi, int oj) { return ZW(oi, oj - 1) + ZW(oi - 1, oj - 1) + ZW(oi - 1, oj); };
    T ne00 = tne(0, 0), nw10 = tnw(1, 0), se00 = tse(0, 0), sw10 = tsw(1, 0);
    T sw01 = tsw(0, 1), se01 = tse(0, 1), nw00 = tnw(0, 0);
    if (SCHEME == NEMO_NP_EET) {
        const T z00 = T(1) / E3(m.e3t, c, k), z10 = T(1) / E3(m.e3t, c + 1u, k), z01 = T(1) / E3(m.e3t, c + w, k);
        ne00 = ne00 * z00; nw10 = nw10 * z10; se00 = se00 * z00; sw10 = sw10 * z10;
        sw01 = sw01 * z01; se01 = se01 * z01; nw00 = nw00 * z00;
    }
#undef ZW
    const bool uni = d.e3_sij == 0;
    const auto zwx = [&](T e2u, uint32_t q) { return e2u * (uni ? uld(m.e3u, k - 1) : E3(m.e3u, q, k)) * ldp(u, q); };
    const auto zwy = [&](T e1v, uint32_t q) { return e1v * (uni ? uld(m.e3v, k - 1) : E3(m.e3v, q, k)) * ldp(v, q); };
    const T zua = e.ru * (ne00 * zwy(e.yc, c) + nw10 * zwy(e.ye, c + 1u) + se00 * zwy(e.ys, c - w) + sw10 * zwy(e.yse, c - w + 1u));
    const T zva = -(e.rv * (sw01 * zwx(e.xnw, c + w - 1u) + se01 * zwx(e.xn, c + w) + nw00 * zwx(e.xw, c - 1u) + ne00 * zwx(e.xc, c)));
    a = a + zua;
    b = b + zva;
}
// ENT: t-point vorticity times volume, DYN/dynvor.F90:225-317
template <typename T>
__device__ __forceinline__ T ent_zwt(const DevDomain &d, int kvor, const T *pu, const T *pv, int p, int q, int k)
{
    const Metrics<T> &m = met<T>(d);
    const size_t pq = IJ(p, q);
    const T e3t = E3(m.e3t, pq, k);
    const T r1_4 = T(0.25);
    switch (kvor) {
    case np_COR: return m.ff_t[pq] * m.e1e2t[pq] * e3t;
    case np_RVO: {
        const T s = zwz_ent(d, pu, pv, p - 1, q, k) + zwz_ent(d, pu, pv, p, q, k) +
                    zwz_ent(d, pu, pv, p - 1, q - 1, k) + zwz_ent(d, pu, pv, p, q - 1, k);
        return r1_4 * s * m.e1e2t[pq] * e3t;
    }
    case np_MET:
        return ((A3(pv, p, q, k) + A3(pv, p, q - 1, k)) * m.di_e2u_2[pq] -
                (A3(pu, p, q, k) + A3(pu, p - 1, q, k)) * m.dj_e1v_2[pq]) * e3t;
    case np_CRV: {
        const T s = zwz_ent(d, pu, pv, p - 1, q, k) + zwz_ent(d, pu, pv, p, q, k) +
                    zwz_ent(d, pu, pv, p - 1, q - 1, k) + zwz_ent(d, pu, pv, p, q - 1, k);
        return (m.ff_t[pq] + r1_4 * s) * m.e1e2t[pq] * e3t;
    }
    default:
        return (m.ff_t[pq] * m.e1e2t[pq] + (A3(pv, p, q, k) + A3(pv, p, q - 1, k)) * m.di_e2u_2[pq] -
                (A3(pu, p, q, k) + A3(pu, p - 1, q, k)) * m.dj_e1v_2[pq]) * e3t;
    }
}
template <typename T>
__device__ __forceinline__ void vor_ent_pt(const DevDomain &d, int kvor, const T *pu, const T *pv, int i, int j, int k,
                                           T &a, T &b)
{
    const Metrics<T> &m = met<T>(d);
    const T r1_4 = T(0.25);
    const T zc = ent_zwt(d, kvor, pu, pv, i, j, k), ze = ent_zwt(d, kvor, pu, pv, i + 1, j, k),
            zn = ent_zwt(d, kvor, pu, pv, i, j + 1, k);
    a = a + r1_4 * m.r1_e1e2u[IJ(i, j)] / E3(m.e3u, IJ(i, j), k) *
                (ze * (A3(pv, i + 1, j, k) + A3(pv, i + 1, j - 1, k)) + zc * (A3(pv, i, j, k) + A3(pv, i, j - 1, k)));
    b = b - r1_4 * m.r1_e1e2v[IJ(i, j)] / E3(m.e3v, IJ(i, j), k) *
                (zn * (A3(pu, i, j + 1, k) + A3(pu, i - 1, j + 1, k)) + zc * (A3(pu, i, j, k) + A3(pu, i - 1, j, k)));
}

// The scheme and the vorticity kinds are template parameters: each
// instantiation carries only its own stencil, which keeps register use (and so
// occupancy) at what that scheme needs.
// One thread per column and chunk of kch levels (grid.z, lev_chunks).
template <typename T, int SCHEME, int NCOR, int NRVM, int NTOT>
struct S_dyn_vor {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, const T * __restrict__ un, const T * __restrict__ vn, T * __restrict__ ua, T * __restrict__ va, int kch)
    {
        THREAD_IJ_V(vb_, 2, 2);
        const bool on = i <= d.jpi - 1 && j <= d.jpj - 1;
        const int ka = (int)vb_.z * kch + 1;
        int kb = min(ka + kch - 1, d.jpk - 1);
        if constexpr (SCHEME == NEMO_NP_EEN || SCHEME == NEMO_NP_EET) {
            typedef ZwzTile<T, SCHEME, NTOT> Z;
            __shared__ typename Z::Lds z;
            __shared__ int s_bot;
            Z f(d, (int)(bx_ * Z::TX) + 2, (int)(by_ * (Z::H - 2)) + 2);
            if (Z::EEN) kb = min(kb, f.bottom(&s_bot));   // below, the trend is zero
            if (kb < ka) return;
            const uint32_t c = on ? IJ32(i, j) : IJ32(2, 2);
            const EenCol<T> e(d, c);
            f.fetch(d, un, vn, ka);
            for (int k = ka; k <= kb; k++) {
                f.put(d, k, z);
                f.fetch(d, un, vn, min(k + 1, kb));
                __syncthreads();
                if (!on) continue;
                T *pa = plane_ptr(ua, d.n2, k), *pb = plane_ptr(va, d.n2, k);
                T a = ldp((const T *)pa, c), b = ldp((const T *)pb, c);
                vor_een_pt<T, SCHEME, Z::W>(d, e, z[k & 1], (int)threadIdx.x, (int)threadIdx.y, un, vn, c, k, a, b);
                stp(pa, c, a);
                stp(pb, c, b);
            }
        } else {
            if (!on) return;
            for (int k = ka; k <= kb; k++) {
                const size_t p = IJK(i, j, k);
                T a = ua[p], b = va[p];
                switch (SCHEME) {
                case NEMO_NP_ENE: vor_ene_pt(d, NTOT, un, vn, i, j, k, a, b); break;
                case NEMO_NP_ENS: vor_ens_pt(d, NTOT, un, vn, i, j, k, a, b); break;
                case NEMO_NP_MIX:
                    vor_ens_pt(d, NRVM, un, vn, i, j, k, a, b);
                    vor_ene_pt(d, NCOR, un, vn, i, j, k, a, b);
                    break;
                default: vor_ent_pt(d, NTOT, un, vn, i, j, k, a, b); break;
                }
                ua[p] = a;
                va[p] = b;
            }
        }
    }
};
template <typename T, int SCHEME, int NCOR, int NRVM, int NTOT>
KERNEL void k_dyn_vor(DevDomain d, const T * __restrict__ un, const T * __restrict__ vn, T * __restrict__ ua,
                      T * __restrict__ va, int kch)
{
    S_dyn_vor<T, SCHEME, NCOR, NRVM, NTOT>::run(vb_hw(), d, un, vn, ua, va, kch);
}

template <typename T, int SCHEME>
static int launch_dyn_vor_s(const DevDomain &d, const T *un, const T *vn, T *ua, T *va)
{
    Grid2 g = grid2(d.jpi - 2, d.jpj - 2);
    const int kch = lev_chunks(g.grid.x * g.grid.y, d.jpk - 1);
    g.grid.z = (unsigned)((d.jpk - 1 + kch - 1) / kch);
    // (nrvm, ntot) from the momentum advection form, DYN/dynvor.F90:903-939
    switch (d.n_dynadv) {
    case NEMO_NP_LIN_DYN:
        LAUNCHB("dyn_vor", (k_dyn_vor<T, SCHEME, np_COR, np_COR, np_COR>), (S_dyn_vor<T, SCHEME, np_COR, np_COR, np_COR>), g, d, un, vn, ua, va, kch);
        break;
    case NEMO_NP_VEC_C2:
        LAUNCHB("dyn_vor", (k_dyn_vor<T, SCHEME, np_COR, np_RVO, np_CRV>), (S_dyn_vor<T, SCHEME, np_COR, np_RVO, np_CRV>), g, d, un, vn, ua, va, kch);
        break;
    default:
        LAUNCHB("dyn_vor", (k_dyn_vor<T, SCHEME, np_COR, np_MET, np_CME>), (S_dyn_vor<T, SCHEME, np_COR, np_MET, np_CME>), g, d, un, vn, ua, va, kch);
        break;
    }
    return 0;
}

template <typename T>
int launch_dyn_vor(const T *un, const T *vn, T *ua, T *va)
{
    const DevDomain &d = nh::dom();
    switch (d.nvor_scheme) {
    case NEMO_NP_ENE: return launch_dyn_vor_s<T, NEMO_NP_ENE>(d, un, vn, ua, va);
    case NEMO_NP_ENS: return launch_dyn_vor_s<T, NEMO_NP_ENS>(d, un, vn, ua, va);
    case NEMO_NP_MIX: return launch_dyn_vor_s<T, NEMO_NP_MIX>(d, un, vn, ua, va);
    case NEMO_NP_ENT: return launch_dyn_vor_s<T, NEMO_NP_ENT>(d, un, vn, ua, va);
    case NEMO_NP_EET: return launch_dyn_vor_s<T, NEMO_NP_EET>(d, un, vn, ua, va);
    case NEMO_NP_EEN: return launch_dyn_vor_s<T, NEMO_NP_EEN>(d, un, vn, ua, va);
    default: return nh::set_error(NEMO_HIP_ERR_UNSUPPORTED, "dyn_vor: nvor_scheme = %d", d.nvor_scheme);
    }
}
template int launch_dyn_vor<double>(const double *, const double *, double *, double *);
template int launch_dyn_vor<float>(const float *, const float *, float *, float *);

// ---------------------------------------------------------------------------
// dyn_zdf, DYN/dynzdf.F90:107-485 (ln_zad_Aimp = F, iso-level momentum
// mixing, r_vvl = 0).  All columns apply the leapfrog right-hand side; the
// interior ones then solve the u and v columns (FP64 elimination).
// ---------------------------------------------------------------------------
// `pre(k, x)` maps the stored trend x at level k to the value the solve
// starts from (the identity for dyn_zdf alone; the barotropic corrections
// of dyn_spg_ts in the fused step).
struct PreIdentity {
    template <typename T>
    __device__ __forceinline__ T operator()(int, T x) const { return x; }
    template <typename T>
    __device__ __forceinline__ T wet(T x) const { return x; }   // where the level's mask is 1
};
// the levels of a wave's u (comp 0) or v (comp 1) columns, called with all 64
// lanes active (on: the lane has a column).  all: the last level above which
// every lane's masks are 1 and no bottom drag enters; end: the deepest level
// with a mask or a drag that is not zero.  Below it every row is x = 0.
struct ZdfLev {
    int all, end;
};
__device__ __forceinline__ ZdfLev zdf_levels(const DevDomain &d, int comp, int i, int j, bool on)
{
    int a = d.jpk, e = 1;
    if (on) {
        const uint32_t ij = IJ32(i, j);
        const KRange &kr = comp ? d.kV : d.kU;
        const int x0 = kr.k0[ij], x1 = kr.k1[ij];
        e = max(x1, 1);
        if (is_interior(d, i, j)) {
            const int ikb = comp ? d.mbkv[ij] : d.mbku[ij];
            e = max(e, ikb);
            a = x0 > 1 ? 0 : min(x1, ikb);
        }
    }
    const int all = wave_min(a) - 1, end = min(wave_max(e), d.jpk - 1);
    return ZdfLev{min(all, end - 1), end};
}
//
// The sweeps run from the surface to the wave's deepest masked or dragged level
// (zdf_levels), above its first bottom without mask tests; below, every row is
// x = 0 and is only stored.  A segment's operands are loaded together, and
// horizontally uniform scale factors (E3U) are scalar loads.
// k_step_dyn2, 1024x1024x75 FP32 (47 % of the cells dry): 1526 -> 1036 us (4.5
// TB/s); k_dyn_zdf, 512x512x75 FP64: 590 -> 413 us; reading the next segment
// ahead as well, 20 VGPRs more, gives 1202 and 437.
template <bool E3U, typename T, typename Pre = PreIdentity>
__device__ __forceinline__ void zdf_column(const DevDomain &d, double r2dt, int comp, int i, int j,
                                           const T *__restrict__ pb, T *__restrict__ pa, const T *__restrict__ avm,
                                           const double *__restrict__ rCdU_bot, const double *__restrict__ pa_b,
                                           const double *__restrict__ tau, const double *__restrict__ tau_b,
                                           double *__restrict__ zwd_s, const ZdfLev lv, Pre pre = Pre())
{
    const Metrics<T> &m = met<T>(d);
    const int jpk = d.jpk;
    const size_t plane = d.n2;
    const uint32_t ij = IJ32(i, j);
    const uint32_t ijn = comp ? IJ32(i, j + 1) : IJ32(i + 1, j);     // the other t-point of the u/v face
    const T *e3x = comp ? m.e3v : m.e3u;
    const T *e3xw = comp ? m.e3vw : m.e3uw;
    const KRange &kr = comp ? d.kV : d.kU;
    const int x0 = kr.k0[ij], x1 = kr.k1[ij];
    auto xmask = [&](int k) { return (k >= x0 && k <= x1) ? 1.0 : 0.0; };
    auto wxmask = [&](int k) { return (k >= x0 && k <= x1 && (k == 1 || k - 1 >= x0)) ? 1.0 : 0.0; };
    const double r_vvl = 0.0;
    const bool inner = is_interior(d, i, j);
    const bool rm_b = d.ln_drgimp && d.ln_dynspg_ts;
    const double ab = rm_b ? pa_b[ij] : 0.0;
    const auto dry = [&]() {   // the levels below the wave's deepest one
        for (int k = lv.end + 1; k <= jpk - 1; k++) stp(plane_ptr(pa, plane, k), ij, T(0));
    };
    if (!inner) {
        for (int k = 1; k <= lv.end; k++) {
            const double xm = xmask(k);
            double a = ((double)ldp(plane_ptr(pb, plane, k), ij) +
                        r2dt * (double)pre(k, ldp((const T *)plane_ptr(pa, plane, k), ij))) * xm;
            if (rm_b) a = (a - ab) * xm;
            stp(plane_ptr(pa, plane, k), ij, (T)a);
        }
        dry();
        return;
    }
    const int ikb = comp ? d.mbkv[ij] : d.mbku[ij];
    const double csum = rCdU_bot[ijn] + rCdU_bot[ij];
    const double zdt = r2dt * 0.5;
    // off-diagonal at w-level k (k >= 2), lines 208-243, from loaded operands:
    // avm at the face's two t-points, e3xw.  WET: its mask is 1
    auto zzw_v = [&](auto wet, int k, double ze3, T a_n, T a_c, T e3w) {
        const double q = zdt * ((double)a_n + (double)a_c) / (ze3 * (double)e3w);
        return decltype(wet)::value ? -q : -(q * wxmask(k));
    };
    // level k <= jpk; the scale factors by vector load with the level's other
    // operands or, horizontally uniform, by scalar load where used
    auto ld_avm = [&](int k, T &a_n, T &a_c, T &e3w) {
        const T *ak = plane_ptr(avm, plane, k);
        a_n = ldp(ak, ijn);
        a_c = ldp(ak, ij);
        if constexpr (!E3U) e3w = E3(e3xw, ij, k);
    };
    auto zz = [&](auto wet, int k, double ze3, T a_n, T a_c, T e3w) {
        return zzw_v(wet, k, ze3, a_n, a_c, E3U ? uld(e3xw, k - 1) : e3w);
    };
    auto ze3_of = [&](int k, T v) {
        const double e = (double)(E3U ? uld(e3x, k - 1) : v);
        return (1.0 - r_vvl) * e + r_vvl * e;
    };
    const std::false_type masked{};
    const std::true_type unmasked{};
    const int kend = lv.end;
    // the operands of ZDF_SEG levels from k0 (pb, pa, e3x) and of the w-levels
    // under them (avm, e3xw); levels past kend load kend's and are not used.
    // A segment's operands are loaded together (a load issued after a store to
    // pa waits for it)
    struct Seg {
        T b[ZDF_SEG], t[ZDF_SEG], e[ZDF_SEG], wn[ZDF_SEG], wc[ZDF_SEG], we[ZDF_SEG];
    };
    auto fetch = [&](int k0, Seg &g, bool with_b) {
#pragma unroll
        for (int q = 0; q < ZDF_SEG; q++) {
            const int k = min(k0 + q, kend);
            g.t[q] = ldp((const T *)plane_ptr(pa, plane, k), ij);
            if (with_b) g.b[q] = ldp(plane_ptr(pb, plane, k), ij);
            if constexpr (!E3U) g.e[q] = E3(e3x, ij, k);
            ld_avm(k + 1, g.wn[q], g.wc[q], g.we[q]);
        }
    };
    double zws_prev, zwd_prev, a_prev;
    T w1n, w1c, w1e = T(1);   // w-level k of the level to come
    Seg cur;
    ld_avm(2, w1n, w1c, w1e);
    {   // k = 1: surface row with the wind stress
        const double xm = xmask(1);
        double a = ((double)ldp(pb, ij) + r2dt * (double)pre(1, ldp((const T *)pa, ij))) * xm;
        if (rm_b) a = (a - ab) * xm;
        T e1 = T(1);
        if constexpr (!E3U) e1 = E3(e3x, ij, 1);
        const double ze3 = ze3_of(1, e1);
        if (rm_b && 1 == ikb) a = a + r2dt * 0.5 * csum * ab / ze3;
        const double zws = zz(masked, 2, ze3, w1n, w1c, w1e);
        double zwd = 1.0 - zws;
        if (d.ln_drgimp && 1 == ikb) zwd = zwd - r2dt * 0.5 * csum / ze3;
        a = a + r2dt * 0.5 * (tau_b[ij] + tau[ij]) / (ze3 * d.rau0) * xm;
        stp(pa, ij, (T)a);
        zws_prev = zws;
        zwd_prev = zwd;
        a_prev = a;
    }
    auto down = [&](auto wet, int k0) {   // ZDF_SEG levels of the forward sweep
        constexpr bool WET = decltype(wet)::value;
#pragma unroll
        for (int q = 0; q < ZDF_SEG; q++) {
            const int k = k0 + q;
            if (!WET && k > kend) break;
            double a;
            if constexpr (WET) {
                a = (double)cur.b[q] + r2dt * (double)pre.wet(cur.t[q]);
                if (rm_b) a = a - ab;
            } else {
                const double xm = xmask(k);
                a = ((double)cur.b[q] + r2dt * (double)pre(k, cur.t[q])) * xm;
                if (rm_b) a = (a - ab) * xm;
            }
            const double ze3 = ze3_of(k, cur.e[q]);
            if (!WET && rm_b && k == ikb) a = a + r2dt * 0.5 * csum * ab / ze3;
            const double zwi = zz(wet, k, ze3, w1n, w1c, w1e);
            const double zws = zz(wet, k + 1, ze3, cur.wn[q], cur.wc[q], cur.we[q]);
            double zwd = 1.0 - zwi - zws;
            if (!WET && d.ln_drgimp && k == ikb) zwd = zwd - r2dt * 0.5 * csum / ze3;
            zwd = zwd - zwi * zws_prev / zwd_prev;
            a = a - zwi / zwd_prev * a_prev;
            if (k % ZDF_SEG == 0) stp(plane_ptr(zwd_s, plane, k), ij, zwd);   // checkpoint pivots only
            stp(plane_ptr(pa, plane, k), ij, (T)a);
            zws_prev = zws;
            zwd_prev = zwd;
            a_prev = a;
            w1n = cur.wn[q]; w1c = cur.wc[q]; w1e = cur.we[q];
        }
    };
    int k0 = 2;
    for (; k0 + ZDF_SEG - 1 <= lv.all; k0 += ZDF_SEG) {
        fetch(k0, cur, true);
        down(unmasked, k0);
    }
    for (; k0 <= kend; k0 += ZDF_SEG) {
        fetch(k0, cur, true);
        down(masked, k0);
    }
    // levels kend-1 .. 1 by segments of ZDF_SEG levels, bottom segment first:
    // the forward sweep kept the pivot of every ZDF_SEG-th level only, so a
    // segment first recomputes its pivots from the one above it (the
    // operations of the forward sweep), then substitutes back
    const int kl = kend - 1;
    int s = (kl + ZDF_SEG - 1) / ZDF_SEG - 1;
    T an, ac, aw = T(1), ep = T(1);   // w-level k0 of the segment, e3x above it, and the checkpoint pivot
    double ckp = 1.0;
    auto fetch_top = [&](int kt) {
        if (kt == 1) return;
        ld_avm(kt, an, ac, aw);
        if constexpr (!E3U) ep = E3(e3x, ij, kt - 1);
        ckp = ldp((const double *)plane_ptr(zwd_s, plane, kt - 1), ij);
    };
    an = ac = T(0);
    // the last row of the whole column divides the value in hand, any other the
    // one rounded to storage, as if it had been stored and the zero below
    // substituted
    double x = (kend == jpk - 1 ? a_prev : (double)(T)a_prev) / zwd_prev;
    stp(plane_ptr(pa, plane, kend), ij, (T)x);
    dry();
    auto up = [&](auto wet) {
        constexpr bool WET = decltype(wet)::value;
        const int kt = s * ZDF_SEG + 1;
        fetch(kt, cur, false);
        fetch_top(kt);
        T pn = an, pc = ac, pw = aw;
        double zwd_p = ckp, zws_p = 0.0;
        if (s > 0) zws_p = zz(wet, kt, ze3_of(kt - 1, ep), an, ac, aw);
        double piv[ZDF_SEG], zsv[ZDF_SEG];
#pragma unroll
        for (int q = 0; q < ZDF_SEG; q++) {
            const int k = kt + q;
            const double ze3 = ze3_of(k, cur.e[q]);
            const double zws = zz(wet, k + 1, ze3, cur.wn[q], cur.wc[q], cur.we[q]);
            double zwd;
            if (k == 1) {
                zwd = 1.0 - zws;
                if (!WET && d.ln_drgimp && 1 == ikb) zwd = zwd - r2dt * 0.5 * csum / ze3;
            } else {
                const double zwi = zz(wet, k, ze3, pn, pc, pw);
                zwd = 1.0 - zwi - zws;
                if (!WET && d.ln_drgimp && k == ikb) zwd = zwd - r2dt * 0.5 * csum / ze3;
                zwd = zwd - zwi * zws_p / zwd_p;
            }
            piv[q] = zwd;
            zsv[q] = zws;
            zws_p = zws;
            zwd_p = zwd;
            pn = cur.wn[q]; pc = cur.wc[q]; pw = cur.we[q];
        }
#pragma unroll
        for (int q = ZDF_SEG - 1; q >= 0; q--) {
            const int k = kt + q;
            if (WET || k <= kl) {
                x = ((double)cur.t[q] - zsv[q] * x) / piv[q];
                stp(plane_ptr(pa, plane, k), ij, (T)x);
            }
        }
    };
    for (; s >= 0 && (s + 1) * ZDF_SEG > lv.all; s--) up(masked);
    for (; s >= 0; s--) up(unmasked);
}

// The same column solve in the FP32 storage form with jpk <= KMAX: the
// forward-substituted values (rounded to storage, as zdf_column stores
// them) stay in registers instead of passing through pa, and the FP64
// pivots are kept at every ZREG_SEG-th level, the others recomputed segment
// by segment in the back substitution from a second read of avm.  Every
// loop over levels is unrolled to KMAX so the register array is indexed by
// constants; the level count only guards.  Results equal zdf_column's bit
// for bit.
#define ZREG_SEG 8
template <int KMAX, typename Pre = PreIdentity>
__device__ __forceinline__ void zdf_column_reg(const DevDomain &d, double r2dt, int comp, int i, int j,
                                               const float *__restrict__ pb, float *__restrict__ pa,
                                               const float *__restrict__ avm, const double *__restrict__ rCdU_bot,
                                               const double *__restrict__ pa_b, const double *__restrict__ tau,
                                               const double *__restrict__ tau_b, Pre pre = Pre())
{
    const Metrics<float> &m = met<float>(d);
    const int jpk = d.jpk;
    const size_t plane = d.n2;
    const uint32_t ij = IJ32(i, j);
    const uint32_t ijn = comp ? IJ32(i, j + 1) : IJ32(i + 1, j);
    const float *e3x = comp ? m.e3v : m.e3u;
    const float *e3xw = comp ? m.e3vw : m.e3uw;
    const KRange &kr = comp ? d.kV : d.kU;
    const int x0 = kr.k0[ij], x1 = kr.k1[ij];
    auto xmask = [&](int k) { return (k >= x0 && k <= x1) ? 1.0 : 0.0; };
    auto wxmask = [&](int k) { return (k >= x0 && k <= x1 && (k == 1 || k - 1 >= x0)) ? 1.0 : 0.0; };
    const double r_vvl = 0.0;
    const bool rm_b = d.ln_drgimp && d.ln_dynspg_ts;
    const double ab = rm_b ? pa_b[ij] : 0.0;
    if (!is_interior(d, i, j)) {
        for (int k = 1; k <= jpk - 1; k++) {
            const double xm = xmask(k);
            double a = ((double)ldp(plane_ptr(pb, plane, k), ij) +
                        r2dt * (double)pre(k, ldp((const float *)plane_ptr(pa, plane, k), ij))) * xm;
            if (rm_b) a = (a - ab) * xm;
            stp(plane_ptr(pa, plane, k), ij, (float)a);
        }
        return;
    }
    const int ikb = comp ? d.mbkv[ij] : d.mbku[ij];
    const double csum = rCdU_bot[ijn] + rCdU_bot[ij];
    const double zdt = r2dt * 0.5;
    auto zzw = [&](int k, double ze3) {
        const float *ak = plane_ptr(avm, plane, k);
        return -(zdt * ((double)ldp(ak, ijn) + (double)ldp(ak, ij)) / (ze3 * (double)E3(e3xw, ij, k)) * wxmask(k));
    };
    auto ze3_of = [&](int k) { return (1.0 - r_vvl) * (double)E3(e3x, ij, k) + r_vvl * (double)E3(e3x, ij, k); };
    // the eliminated diagonal of level k >= 2 from the previous level's
    // upper diagonal and pivot (lines 208-243 and the forward elimination)
    auto pivot = [&](int k, double ze3, double zws, double zws_p, double zwd_p) {
        const double zwi = zzw(k, ze3);
        double zwd = 1.0 - zwi - zws;
        if (d.ln_drgimp && k == ikb) zwd = zwd - r2dt * 0.5 * csum / ze3;
        return zwd - zwi * zws_p / zwd_p;
    };
    constexpr int NSEG = (KMAX + ZREG_SEG - 1) / ZREG_SEG;
    float fw[KMAX];        // level k at index k - 1
    double ck[NSEG];       // the pivot of level s * ZREG_SEG at index s
    double zws_prev, zwd_prev, a_prev;
    {   // k = 1: surface row with the wind stress
        const double xm = xmask(1);
        double a = ((double)ldp(pb, ij) + r2dt * (double)pre(1, ldp((const float *)pa, ij))) * xm;
        if (rm_b) a = (a - ab) * xm;
        const double ze3 = ze3_of(1);
        if (rm_b && 1 == ikb) a = a + r2dt * 0.5 * csum * ab / ze3;
        const double zws = zzw(2, ze3);
        double zwd = 1.0 - zws;
        if (d.ln_drgimp && 1 == ikb) zwd = zwd - r2dt * 0.5 * csum / ze3;
        a = a + r2dt * 0.5 * (tau_b[ij] + tau[ij]) / (ze3 * d.rau0) * xm;
        fw[0] = (float)a;
        zws_prev = zws;
        zwd_prev = zwd;
        a_prev = a;
    }
#pragma unroll
    for (int k = 2; k < KMAX; k++) {
        if (k <= jpk - 1) {
            const double xm = xmask(k);
            double a = ((double)ldp(plane_ptr(pb, plane, k), ij) +
                        r2dt * (double)pre(k, ldp((const float *)plane_ptr(pa, plane, k), ij))) * xm;
            if (rm_b) a = (a - ab) * xm;
            const double ze3 = ze3_of(k);
            if (rm_b && k == ikb) a = a + r2dt * 0.5 * csum * ab / ze3;
            const double zwi = zzw(k, ze3);
            const double zws = zzw(k + 1, ze3);
            const double zwd = pivot(k, ze3, zws, zws_prev, zwd_prev);
            a = a - zwi / zwd_prev * a_prev;
            if (k % ZREG_SEG == 0) ck[k / ZREG_SEG] = zwd;
            fw[k - 1] = (float)a;
            zws_prev = zws;
            zwd_prev = zwd;
            a_prev = a;
        }
    }
    double x = a_prev / zwd_prev;
    stp(plane_ptr(pa, plane, jpk - 1), ij, (float)x);
    const int kl = jpk - 2;
#pragma unroll
    for (int s = NSEG - 1; s >= 0; s--) {
        const int k0 = s * ZREG_SEG + 1;
        if (k0 <= kl) {
            double piv[ZREG_SEG], zsv[ZREG_SEG];
            double zwd_p = 0.0, zws_p = 0.0;
            if (s > 0) {
                zwd_p = ck[s];
                zws_p = zzw(k0, ze3_of(k0 - 1));
            }
#pragma unroll
            for (int q = 0; q < ZREG_SEG; q++) {
                const int k = k0 + q;
                if (k < KMAX && k <= kl) {
                    const double ze3 = ze3_of(k);
                    const double zws = zzw(k + 1, ze3);
                    double zwd;
                    if (k == 1) {
                        zwd = 1.0 - zws;
                        if (d.ln_drgimp && 1 == ikb) zwd = zwd - r2dt * 0.5 * csum / ze3;
                    } else {
                        zwd = pivot(k, ze3, zws, zws_p, zwd_p);
                    }
                    piv[q] = zwd;
                    zsv[q] = zws;
                    zws_p = zws;
                    zwd_p = zwd;
                }
            }
#pragma unroll
            for (int q = ZREG_SEG - 1; q >= 0; q--) {
                const int k = k0 + q;
                if (k < KMAX && k <= kl) {
                    x = ((double)fw[k - 1] - zsv[q] * x) / piv[q];
                    stp(plane_ptr(pa, plane, k), ij, (float)x);
                }
            }
        }
    }
}
// the levels zdf_column_reg holds in registers (jpk <= ZDF_REG_KMAX): the
// 75 of the full-size configurations
#define ZDF_REG_KMAX 76

// The u and v columns of a point by one thread after the other, or, where the
// columns leave SIMDs idle (two waves each: 512 workgroups; with a remainder,
// 1024), by two workgroups (grid.z 2), with a checkpoint array each.  k_step_dyn2
// 32x22x31 FP64: 68 us in turn, 36 us; 362x149x46 FP64 113 and 81 us;
// 251x333x56 FP32 146 and 101 us.  In a plan the members' workgroups share one
// launch and the columns stay in turn (lev_chunks has what that costs a plan of
// one or two members).
inline unsigned zdf_comps(unsigned nb) { return nh::planning() || nb >= 1024u ? 1u : 2u; }
template <typename T, bool REG, bool E3U>
struct S_dyn_zdf {
    static constexpr int NTHR = NH_BLOCK, WAVES = 2;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, double r2dt, const T * __restrict__ ub, const T * __restrict__ vb, T * __restrict__ ua, T * __restrict__ va, const T * __restrict__ avm, const double * __restrict__ rCdU_bot, const double * __restrict__ ua_b, const double * __restrict__ va_b, const double * __restrict__ utau, const double * __restrict__ utau_b, const double * __restrict__ vtau, const double * __restrict__ vtau_b, double * __restrict__ zwd_s, double * __restrict__ zwd2_s)
    {
        THREAD_IJ_V(vb_, 1, 1);
        const bool on = i <= d.jpi && j <= d.jpj;
        const auto comp = [&](auto cc) {
            constexpr int c = decltype(cc)::value;
            const T *xb = c ? vb : ub;
            T *xa = c ? va : ua;
            const double *xa_b = c ? va_b : ua_b, *tau = c ? vtau : utau, *tau_b = c ? vtau_b : utau_b;
            if constexpr (REG) {
                if (!on) return;
                zdf_column_reg<ZDF_REG_KMAX>(d, r2dt, c, i, j, xb, xa, avm, rCdU_bot, xa_b, tau, tau_b);
            } else {
                const ZdfLev l = zdf_levels(d, c, i, j, on);
                if (on) zdf_column<E3U>(d, r2dt, c, i, j, xb, xa, avm, rCdU_bot, xa_b, tau, tau_b, c ? zwd2_s : zwd_s, l);
            }
        };
        if (vb_.z == 0) comp(std::integral_constant<int, 0>());
        if (vb_.z == 1 || vb_.gz == 1) comp(std::integral_constant<int, 1>());
    }
};
template <typename T, bool REG, bool E3U>
KERNEL_W(2) void k_dyn_zdf(DevDomain d, double r2dt, const T * __restrict__ ub, const T * __restrict__ vb, T * __restrict__ ua, T * __restrict__ va, const T * __restrict__ avm,
                          const double * __restrict__ rCdU_bot, const double * __restrict__ ua_b, const double * __restrict__ va_b, const double * __restrict__ utau,
                          const double * __restrict__ utau_b, const double * __restrict__ vtau, const double * __restrict__ vtau_b, double * __restrict__ zwd_s, double * __restrict__ zwd2_s)
{
    S_dyn_zdf<T, REG, E3U>::run(vb_hw(), d, r2dt, ub, vb, ua, va, avm, rCdU_bot, ua_b, va_b, utau, utau_b, vtau, vtau_b, zwd_s, zwd2_s);
}
// the register form applies: FP32 storage, jpk <= ZDF_REG_KMAX, switch zdf_reg
template <typename T>
static bool zdf_reg(const DevDomain &d)
{
    return sizeof(T) == 4 && d.jpk <= ZDF_REG_KMAX && nh::tune(nh::T_ZDF_REG);
}

template <typename T>
int launch_dyn_zdf(double r2dt, const T *ub, const T *vb, T *ua, T *va, const T *avm, const double *rCdU_bot,
                   const double *ua_b, const double *va_b, const double *utau, const double *utau_b,
                   const double *vtau, const double *vtau_b)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    g.grid.z = zdf_comps(g.grid.x * g.grid.y);
    double *zwd = (double *)nh::scratch3(nh::S_ZWT), *zwd2 = (double *)nh::scratch3(nh::S_ZWT2);
    // forward-substituted values stay in ua/va at storage precision
    if constexpr (sizeof(T) == 4) {
        if (zdf_reg<T>(d)) {
            LAUNCHB("dyn_zdf", (k_dyn_zdf<T, true, false>), (S_dyn_zdf<T, true, false>), g, d, r2dt, ub, vb, ua, va, avm, rCdU_bot, ua_b, va_b, utau,
                   utau_b, vtau, vtau_b, zwd, zwd2);
            return 0;
        }
    }
#define ZDF_LAUNCH(U) \
    LAUNCHB("dyn_zdf", (k_dyn_zdf<T, false, U>), (S_dyn_zdf<T, false, U>), g, d, r2dt, ub, vb, ua, va, avm, rCdU_bot, ua_b, va_b, utau, \
           utau_b, vtau, vtau_b, zwd, zwd2)
    if (d.e3_sij == 0) ZDF_LAUNCH(true);
    else ZDF_LAUNCH(false);
#undef ZDF_LAUNCH
    return 0;
}
template int launch_dyn_zdf<double>(double, const double *, const double *, double *, double *, const double *,
                                    const double *, const double *, const double *, const double *, const double *,
                                    const double *, const double *);
template int launch_dyn_zdf<float>(double, const float *, const float *, float *, float *, const float *,
                                   const double *, const double *, const double *, const double *, const double *,
                                   const double *, const double *);

// ---------------------------------------------------------------------------
// Fused momentum step: ua = va = 0; dyn_adv; dyn_vor; dyn_spg_ts; dyn_zdf
// (the order of step.F90:189-257) in two 3D passes around the barotropic
// sub-steps:
//   k_step_dyn1  advection + vorticity trends written once, with the vertical
//                sums of dyn_spg_ts phase 1 (DYN/dynspg_ts.F90:358-378) and the
//                bottom velocities (519-527) accumulated in the same k-march;
//   k_step_dyn2  phase 3 (lines 1214-1269) applied to un/vn and to the trend
//                on the fly, then the dyn_zdf solve of the column.
// Every stored intermediate of the separate calls is rounded to the storage
// type at the same point here, so the fused step equals the sequence of
// separate calls bit for bit in either storage form.
// ---------------------------------------------------------------------------
template <typename T, int ADV, int KEG, int SCHEME, int NCOR, int NRVM, int NTOT>
struct S_step_dyn1 {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, const T *__restrict__ un, const T *__restrict__ vn, const T *__restrict__ wn, T *__restrict__ ua, T *__restrict__ va, const double *__restrict__ r1_hu_n, const double *__restrict__ r1_hv_n, const double *__restrict__ un_b, const double *__restrict__ vn_b, double *__restrict__ zu_frc, double *__restrict__ zv_frc, double *__restrict__ su_s, double *__restrict__ sv_s, double *__restrict__ zwxb, double *__restrict__ zwyb, int kch)
    {
        THREAD_IJ_V(vb_, 1, 1);
        constexpr bool TILE = SCHEME == NEMO_NP_EEN || SCHEME == NEMO_NP_EET;
        const int jpk = d.jpk;
        // the chunk's levels; a workgroup of whole columns also sums them
        const int ka = (int)vb_.z * kch + 1, kb = min(ka + kch - 1, jpk - 1);
        const bool whole = kch >= jpk - 1;
        const bool in = i <= d.jpi && j <= d.jpj, inner = in && is_interior(d, i, j);
        const uint32_t ij = in ? IJ32(i, j) : 0u;
        if (in && !inner) {
            for (int k = ka; k <= (kb == jpk - 1 ? jpk : kb); k++) {
                A3(ua, i, j, k) = T(0);
                A3(va, i, j, k) = T(0);
            }
            if (whole) {
                double su = 0.0, sv = 0.0;
                su = su * r1_hu_n[ij];
                sv = sv * r1_hv_n[ij];
                zu_frc[ij] = su; su_s[ij] = su;
                zv_frc[ij] = sv; sv_s[ij] = sv;
            }
        }
        if (!TILE && !inner) return;
        typedef ZwzTile<T, TILE ? SCHEME : NEMO_NP_EET, NTOT> Z;
        __shared__ typename Z::Lds zf;
        __shared__ int s_bot;
        // threads without a cell of their own work on the f-points: cell (2,2)
        const uint32_t c = inner ? ij : IJ32(2, 2);
        int kvor = kb;
        [[maybe_unused]] typename std::conditional<TILE, Z, int>::type f = [&] {
            if constexpr (TILE) return Z(d, (int)(bx_ * Z::TX) + 1, (int)(by_ * (Z::H - 2)) + 1);
            else return 0;
        }();
        [[maybe_unused]] typename std::conditional<TILE, EenCol<T>, int>::type e = [&] {
            if constexpr (TILE) return EenCol<T>(d, c);
            else return 0;
        }();
        if constexpr (TILE) {
            if (Z::EEN) kvor = min(kb, f.bottom(&s_bot));   // below, the vorticity trend is zero
            if (kvor >= ka) f.fetch(d, un, vn, ka);
        }
        const Metrics<T> &m = met<T>(d);
        const T e1u = m.e1u[c], e2v = m.e2v[c], r1_e1e2u = m.r1_e1e2u[c], r1_e1e2v = m.r1_e1e2v[c];
        const T e1e2t = m.e1e2t[c], e1e2t_e = m.e1e2t[c + 1u], e1e2t_n = m.e1e2t[c + (uint32_t)d.jpi];
        // vertical fluxes at w-level kk: zad (zero at the surface, dynzad.F90:93-94)
        // or cen2 (surface flux, dynadv_cen2.F90:105-112), carried between levels
        const auto wflux = [&](int kk, T &cu, T &cv) {
            cu = cv = T(0);
            if (ADV == NEMO_NP_VEC_C2 && kk > 1 && kk <= jpk - 1) {
                const T zww = T(0.25) * e1e2t * A3(wn, i, j, kk);
                const T zww_e = T(0.25) * e1e2t_e * A3(wn, i + 1, j, kk);
                const T zww_n = T(0.25) * e1e2t_n * A3(wn, i, j + 1, kk);
                cu = (zww_e + zww) * (A3(un, i, j, kk - 1) - A3(un, i, j, kk));
                cv = (zww_n + zww) * (A3(vn, i, j, kk - 1) - A3(vn, i, j, kk));
            }
            if (ADV == NEMO_NP_FLX_C2 && kk == 1) {
                cu = T(0.5) * (e1e2t * A3(wn, i, j, 1) + e1e2t_e * A3(wn, i + 1, j, 1)) * A3(un, i, j, 1);
                cv = T(0.5) * (e1e2t * A3(wn, i, j, 1) + e1e2t_n * A3(wn, i, j + 1, 1)) * A3(vn, i, j, 1);
            }
            if (ADV == NEMO_NP_FLX_C2 && kk > 1 && kk <= jpk - 1) {
                const T fw = cen2_zfw(d, wn, i, j, kk);
                cu = (fw + cen2_zfw(d, wn, i + 1, j, kk)) * (A3(un, i, j, kk) + A3(un, i, j, kk - 1));
                cv = (fw + cen2_zfw(d, wn, i, j + 1, kk)) * (A3(vn, i, j, kk) + A3(vn, i, j, kk - 1));
            }
        };
        T cu_k = T(0), cv_k = T(0);
        if (inner) wflux(ka, cu_k, cv_k);
        double su = 0.0, sv = 0.0;
        for (int k = ka; k <= kb; k++) {
            if constexpr (TILE) {
                if (k <= kvor) {
                    f.put(d, k, zf);
                    f.fetch(d, un, vn, min(k + 1, kvor));
                    __syncthreads();
                }
                if (!inner) continue;
            }
            T a = T(0), b = T(0);
            if (ADV == NEMO_NP_VEC_C2) {
                T h, he, hn;
                if (KEG == 0) {
                    h = keg_c2(d, un, vn, i, j, k); he = keg_c2(d, un, vn, i + 1, j, k); hn = keg_c2(d, un, vn, i, j + 1, k);
                } else {
                    h = keg_hw(d, un, vn, i, j, k); he = keg_hw(d, un, vn, i + 1, j, k); hn = keg_hw(d, un, vn, i, j + 1, k);
                }
                a = a - (he - h) / e1u;
                b = b - (hn - h) / e2v;
                T cu_kp1, cv_kp1;
                wflux(k + 1, cu_kp1, cv_kp1);
                a = a - (cu_k + cu_kp1) * r1_e1e2u / E3(m.e3u, ij, k);
                b = b - (cv_k + cv_kp1) * r1_e1e2v / E3(m.e3v, ij, k);
                cu_k = cu_kp1;
                cv_k = cv_kp1;
            } else if (ADV == NEMO_NP_FLX_C2) {
                const T fu_im1 = cen2_zfu(d, un, i - 1, j, k), fu_i = cen2_zfu(d, un, i, j, k), fu_ip1 = cen2_zfu(d, un, i + 1, j, k);
                const T fu_jp1 = cen2_zfu(d, un, i, j + 1, k), fu_im1jp1 = cen2_zfu(d, un, i - 1, j + 1, k);
                const T fv_i = cen2_zfv(d, vn, i, j, k), fv_ip1 = cen2_zfv(d, vn, i + 1, j, k);
                const T fv_jm1 = cen2_zfv(d, vn, i, j - 1, k), fv_ip1jm1 = cen2_zfv(d, vn, i + 1, j - 1, k);
                const T fv_jp1 = cen2_zfv(d, vn, i, j + 1, k), fv_im1 = cen2_zfv(d, vn, i - 1, j, k);
                const T u_i = A3(un, i, j, k), u_ip1 = A3(un, i + 1, j, k), u_im1 = A3(un, i - 1, j, k);
                const T u_jp1 = A3(un, i, j + 1, k), u_jm1 = A3(un, i, j - 1, k);
                const T v_j = A3(vn, i, j, k), v_ip1 = A3(vn, i + 1, j, k), v_jp1 = A3(vn, i, j + 1, k);
                const T v_im1 = A3(vn, i - 1, j, k), v_jm1 = A3(vn, i, j - 1, k);
                const T zfu_t_ip1 = (fu_i + fu_ip1) * (u_i + u_ip1);
                const T zfu_t_i = (fu_im1 + fu_i) * (u_im1 + u_i);
                const T zfv_f_j = (fv_i + fv_ip1) * (u_i + u_jp1);
                const T zfv_f_jm1 = (fv_jm1 + fv_ip1jm1) * (u_jm1 + u_i);
                const T zfu_f_i = (fu_i + fu_jp1) * (v_j + v_ip1);
                const T zfu_f_im1 = (fu_im1 + fu_im1jp1) * (v_im1 + v_j);
                const T zfv_t_jp1 = (fv_i + fv_jp1) * (v_j + v_jp1);
                const T zfv_t_j = (fv_jm1 + fv_i) * (v_jm1 + v_j);
                a = a - (zfu_t_ip1 - zfu_t_i + zfv_f_j - zfv_f_jm1) * r1_e1e2u / E3(m.e3u, ij, k);
                b = b - (zfu_f_i - zfu_f_im1 + zfv_t_jp1 - zfv_t_j) * r1_e1e2v / E3(m.e3v, ij, k);
                T cu_kp1, cv_kp1;
                wflux(k + 1, cu_kp1, cv_kp1);
                a = a - (cu_k - cu_kp1) * r1_e1e2u / E3(m.e3u, ij, k);
                b = b - (cv_k - cv_kp1) * r1_e1e2v / E3(m.e3v, ij, k);
                cu_k = cu_kp1;
                cv_k = cv_kp1;
            }
            switch (SCHEME) {
            case NEMO_NP_ENE: vor_ene_pt(d, NTOT, un, vn, i, j, k, a, b); break;
            case NEMO_NP_ENS: vor_ens_pt(d, NTOT, un, vn, i, j, k, a, b); break;
            case NEMO_NP_MIX:
                vor_ens_pt(d, NRVM, un, vn, i, j, k, a, b);
                vor_ene_pt(d, NCOR, un, vn, i, j, k, a, b);
                break;
            case NEMO_NP_ENT: vor_ent_pt(d, NTOT, un, vn, i, j, k, a, b); break;
            default:
                if constexpr (TILE) {
                    if (k <= kvor)
                        vor_een_pt<T, SCHEME, Z::W>(d, e, zf[k & 1], (int)threadIdx.x, (int)threadIdx.y, un, vn, c, k, a, b);
                }
                break;
            }
            const size_t p = IJK(i, j, k);
            ua[p] = a;
            va[p] = b;
            su = su + (double)E3(m.e3u, ij, k) * (double)a * UMASK(double, i, j, k);
            sv = sv + (double)E3(m.e3v, ij, k) * (double)b * VMASK(double, i, j, k);
        }
        if (!inner) return;
        if (kb == jpk - 1) {
            A3(ua, i, j, jpk) = T(0);
            A3(va, i, j, jpk) = T(0);
        }
        if (!whole) return;   // k_step_sum
        su = su * r1_hu_n[ij];
        sv = sv * r1_hv_n[ij];
        zu_frc[ij] = su; su_s[ij] = su;
        zv_frc[ij] = sv; sv_s[ij] = sv;
        zwxb[ij] = (double)A3(un, i, j, d.mbku[ij]) - un_b[ij];
        zwyb[ij] = (double)A3(vn, i, j, d.mbkv[ij]) - vn_b[ij];
    }
};
template <typename T, int ADV, int KEG, int SCHEME, int NCOR, int NRVM, int NTOT>
KERNEL void k_step_dyn1(DevDomain d, const T *__restrict__ un, const T *__restrict__ vn, const T *__restrict__ wn,
                        T *__restrict__ ua, T *__restrict__ va, const double *__restrict__ r1_hu_n,
                        const double *__restrict__ r1_hv_n, const double *__restrict__ un_b,
                        const double *__restrict__ vn_b, double *__restrict__ zu_frc, double *__restrict__ zv_frc,
                        double *__restrict__ su_s, double *__restrict__ sv_s, double *__restrict__ zwxb,
                        double *__restrict__ zwyb, int kch)
{
    S_step_dyn1<T, ADV, KEG, SCHEME, NCOR, NRVM, NTOT>::run(vb_hw(), d, un, vn, wn, ua, va, r1_hu_n, r1_hv_n, un_b, vn_b, zu_frc, zv_frc, su_s, sv_s, zwxb, zwyb, kch);
}


// the sums of k_step_dyn1 where its levels are shared out: one thread per column
// and component (grid.z), eight levels' loads together
template <typename T>
struct S_step_sum {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1, KB = 8;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, const T *__restrict__ un, const T *__restrict__ vn, const T *__restrict__ ua, const T *__restrict__ va, const double *__restrict__ r1_hu_n, const double *__restrict__ r1_hv_n, const double *__restrict__ un_b, const double *__restrict__ vn_b, double *__restrict__ zu_frc, double *__restrict__ zv_frc, double *__restrict__ su_s, double *__restrict__ sv_s, double *__restrict__ zwxb, double *__restrict__ zwyb)
    {
        THREAD_IJ_V(vb_, 1, 1);
        if (i > d.jpi || j > d.jpj) return;
        const bool cv = vb_.z != 0;
        const uint32_t ij = IJ32(i, j);
        const Metrics<T> &m = met<T>(d);
        const T *a = cv ? va : ua, *e3 = cv ? m.e3v : m.e3u;
        const uint32_t w = cv ? d.kvf[ij] : d.ktu[ij] >> 16;
        const int m0 = (int)(w & 255u), m1 = (int)((w >> 8) & 255u);
        const bool inner = is_interior(d, i, j), uni = d.e3_sij == 0;
        double s = 0.0;
        if (inner) {
            for (int k0 = 1; k0 <= d.jpk - 1; k0 += KB) {
                T av[KB];
    #pragma unroll
                for (int q = 0; q < KB; q++) av[q] = ldp(plane_ptr(a, d.n2, min(k0 + q, d.jpk - 1)), ij);
    #pragma unroll
                for (int q = 0; q < KB; q++) {
                    const int k = k0 + q;
                    if (k > d.jpk - 1) break;
                    s = s + (double)(uni ? uld(e3, k - 1) : E3(e3, ij, k)) * (double)av[q] * (k >= m0 && k <= m1 ? 1.0 : 0.0);
                }
            }
        }
        s = s * (cv ? r1_hv_n : r1_hu_n)[ij];
        (cv ? zv_frc : zu_frc)[ij] = s;
        (cv ? sv_s : su_s)[ij] = s;
        if (!inner) return;
        if (cv) zwyb[ij] = (double)A3(vn, i, j, d.mbkv[ij]) - vn_b[ij];
        else zwxb[ij] = (double)A3(un, i, j, d.mbku[ij]) - un_b[ij];
    }
};
template <typename T>
KERNEL void k_step_sum(DevDomain d, const T *__restrict__ un, const T *__restrict__ vn, const T *__restrict__ ua,
                       const T *__restrict__ va, const double *__restrict__ r1_hu_n,
                       const double *__restrict__ r1_hv_n, const double *__restrict__ un_b,
                       const double *__restrict__ vn_b, double *__restrict__ zu_frc, double *__restrict__ zv_frc,
                       double *__restrict__ su_s, double *__restrict__ sv_s, double *__restrict__ zwxb,
                       double *__restrict__ zwyb)
{
    S_step_sum<T>::run(vb_hw(), d, un, vn, ua, va, r1_hu_n, r1_hv_n, un_b, vn_b, zu_frc, zv_frc, su_s, sv_s, zwxb, zwyb);
}

// ua after dyn_spg_ts: interior columns remove the vertical mean of the
// trend (phase 1, rounded to storage), every column adds the barotropic
// correction (phase 3, rounded to storage)
template <typename T>
struct PreSpg {
    double s, dd;
    int x0, x1;
    bool inner;
    __device__ __forceinline__ T operator()(int k, T x) const
    {
        const double xm = (k >= x0 && k <= x1) ? 1.0 : 0.0;
        if (inner) x = (T)((double)x - s * xm);
        return (T)((double)x + dd);
    }
    __device__ __forceinline__ T wet(T x) const { return (T)((double)(T)((double)x - s) + dd); }
};

template <typename T, bool REG, bool E3U>
struct S_step_dyn2 {
    static constexpr int NTHR = NH_BLOCK, WAVES = 2;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, double r2dt, double r1_2dt_b, const T *__restrict__ ub, const T *__restrict__ vb, T *__restrict__ ua, T *__restrict__ va, T *__restrict__ un, T *__restrict__ vn, const T *__restrict__ avm, const double *__restrict__ rCdU_bot, const double *__restrict__ ua_b, const double *__restrict__ va_b, const double *__restrict__ ub_b, const double *__restrict__ vb_b, const double *__restrict__ un_adv, const double *__restrict__ vn_adv, const double *__restrict__ r1_hu_n, const double *__restrict__ r1_hv_n, const double *__restrict__ un_b, const double *__restrict__ vn_b, const double *__restrict__ su_s, const double *__restrict__ sv_s, const double *__restrict__ utau, const double *__restrict__ utau_b, const double *__restrict__ vtau, const double *__restrict__ vtau_b, double *__restrict__ zwd_s, double *__restrict__ zwd2_s)
    {
        THREAD_IJ_V(vb_, 1, 1);
        const bool on = i <= d.jpi && j <= d.jpj;
        const size_t plane = d.n2;
        const uint32_t ij = on ? IJ32(i, j) : 0u;
        const auto comp = [&](auto cc) {
            constexpr int c = decltype(cc)::value;
            const ZdfLev l = zdf_levels(d, c, i, j, on);
            if (!on) return;
            const int *m0 = c ? d.kV.k0 : d.kU.k0, *m1 = c ? d.kV.k1 : d.kU.k1;
            const int x0 = m0[ij], x1 = m1[ij];
            // phase 3 on the now velocity, lines 1254-1259: zero where masked
            {
                T *xn = c ? vn : un;
                const double cx = (c ? vn_adv : un_adv)[ij] * (c ? r1_hv_n : r1_hu_n)[ij], xbn = (c ? vn_b : un_b)[ij];
                constexpr int KB = 8;   // levels loaded together, ahead of the stores
                for (int k0 = 1; k0 <= l.end; k0 += KB) {
                    T xo[KB];
    #pragma unroll
                    for (int q = 0; q < KB; q++) xo[q] = ldp((const T *)plane_ptr(xn, plane, min(k0 + q, l.end)), ij);
    #pragma unroll
                    for (int q = 0; q < KB; q++) {
                        const int k = k0 + q;
                        if (k > l.end) break;
                        const double xm = (k >= x0 && k <= x1) ? 1.0 : 0.0;
                        stp(plane_ptr(xn, plane, k), ij, (T)(((double)xo[q] + cx - xbn) * xm));
                    }
                }
                for (int k = l.end + 1; k <= d.jpk - 1; k++) stp(plane_ptr(xn, plane, k), ij, T(0));
            }
            const double *xa_b = c ? va_b : ua_b, *xb_b = c ? vb_b : ub_b, *tau = c ? vtau : utau, *tau_b = c ? vtau_b : utau_b;
            const T *xb = c ? vb : ub;
            T *xa = c ? va : ua;
            const PreSpg<T> px{(c ? sv_s : su_s)[ij], (xa_b[ij] - xb_b[ij]) * r1_2dt_b, x0, x1, is_interior(d, i, j)};
            if constexpr (REG) zdf_column_reg<ZDF_REG_KMAX>(d, r2dt, c, i, j, xb, xa, avm, rCdU_bot, xa_b, tau, tau_b, px);
            else zdf_column<E3U>(d, r2dt, c, i, j, xb, xa, avm, rCdU_bot, xa_b, tau, tau_b, c ? zwd2_s : zwd_s, l, px);
        };
        if (vb_.z == 0) comp(std::integral_constant<int, 0>());
        if (vb_.z == 1 || vb_.gz == 1) comp(std::integral_constant<int, 1>());
    }
};
template <typename T, bool REG, bool E3U>
KERNEL_W(2) void k_step_dyn2(DevDomain d, double r2dt, double r1_2dt_b, const T *__restrict__ ub, const T *__restrict__ vb,
                        T *__restrict__ ua, T *__restrict__ va, T *__restrict__ un, T *__restrict__ vn,
                        const T *__restrict__ avm, const double *__restrict__ rCdU_bot,
                        const double *__restrict__ ua_b, const double *__restrict__ va_b,
                        const double *__restrict__ ub_b, const double *__restrict__ vb_b,
                        const double *__restrict__ un_adv, const double *__restrict__ vn_adv,
                        const double *__restrict__ r1_hu_n, const double *__restrict__ r1_hv_n,
                        const double *__restrict__ un_b, const double *__restrict__ vn_b,
                        const double *__restrict__ su_s, const double *__restrict__ sv_s,
                        const double *__restrict__ utau, const double *__restrict__ utau_b,
                        const double *__restrict__ vtau, const double *__restrict__ vtau_b,
                        double *__restrict__ zwd_s, double *__restrict__ zwd2_s)
{
    S_step_dyn2<T, REG, E3U>::run(vb_hw(), d, r2dt, r1_2dt_b, ub, vb, ua, va, un, vn, avm, rCdU_bot, ua_b, va_b, ub_b, vb_b, un_adv, vn_adv, r1_hu_n, r1_hv_n, un_b, vn_b, su_s, sv_s, utau, utau_b, vtau, vtau_b, zwd_s, zwd2_s);
}

template <typename T, int ADV, int KEG, int SCHEME>
static int launch_step_dyn1_s(const DevDomain &d, Grid2 g, const T *un, const T *vn, const T *wn, T *ua, T *va,
                              const nemo_hip_spg_ts_t *st, double **w)
{
    const double *r1u = st->r1_hu_n, *r1v = st->r1_hv_n, *ub = st->un_b, *vb = st->vn_b;
    const int kch = lev_chunks(g.grid.x * g.grid.y, d.jpk - 1);
    g.grid.z = (unsigned)((d.jpk - 1 + kch - 1) / kch);
    switch (ADV) {
    case NEMO_NP_LIN_DYN:
        LAUNCHB("step_dyn", (k_step_dyn1<T, ADV, KEG, SCHEME, np_COR, np_COR, np_COR>), (S_step_dyn1<T, ADV, KEG, SCHEME, np_COR, np_COR, np_COR>), g, d, un, vn, wn, ua, va, r1u,
               r1v, ub, vb, w[0], w[1], w[2], w[3], w[4], w[5], kch);
        break;
    case NEMO_NP_VEC_C2:
        LAUNCHB("step_dyn", (k_step_dyn1<T, ADV, KEG, SCHEME, np_COR, np_RVO, np_CRV>), (S_step_dyn1<T, ADV, KEG, SCHEME, np_COR, np_RVO, np_CRV>), g, d, un, vn, wn, ua, va, r1u,
               r1v, ub, vb, w[0], w[1], w[2], w[3], w[4], w[5], kch);
        break;
    default:
        LAUNCHB("step_dyn", (k_step_dyn1<T, ADV, KEG, SCHEME, np_COR, np_MET, np_CME>), (S_step_dyn1<T, ADV, KEG, SCHEME, np_COR, np_MET, np_CME>), g, d, un, vn, wn, ua, va, r1u,
               r1v, ub, vb, w[0], w[1], w[2], w[3], w[4], w[5], kch);
        break;
    }
    if (g.grid.z > 1) {
        g.grid.z = 2;
        LAUNCHB("step_dyn", k_step_sum<T>, (S_step_sum<T>), g, d, un, vn, (const T *)ua, (const T *)va, r1u, r1v, ub, vb, w[0], w[1], w[2],
                w[3], w[4], w[5]);
    }
    return 0;
}
template <typename T, int SCHEME>
static int launch_step_dyn1_v(const DevDomain &d, Grid2 g, const T *un, const T *vn, const T *wn, T *ua, T *va,
                              const nemo_hip_spg_ts_t *st, double **w)
{
    switch (d.n_dynadv) {
    case NEMO_NP_LIN_DYN: return launch_step_dyn1_s<T, NEMO_NP_LIN_DYN, 0, SCHEME>(d, g, un, vn, wn, ua, va, st, w);
    case NEMO_NP_VEC_C2:
        if (d.nn_dynkeg == 0) return launch_step_dyn1_s<T, NEMO_NP_VEC_C2, 0, SCHEME>(d, g, un, vn, wn, ua, va, st, w);
        return launch_step_dyn1_s<T, NEMO_NP_VEC_C2, 1, SCHEME>(d, g, un, vn, wn, ua, va, st, w);
    case NEMO_NP_FLX_C2: return launch_step_dyn1_s<T, NEMO_NP_FLX_C2, 0, SCHEME>(d, g, un, vn, wn, ua, va, st, w);
    default: return nh::set_error(NEMO_HIP_ERR_UNSUPPORTED, "step_dyn: n_dynadv = %d", d.n_dynadv);
    }
}

template <typename T>
int launch_step_dyn(int kt, double r2dt, const T *ub, const T *vb, const T *wn, const T *avm, const double *utau_b,
                    const double *vtau_b, const nemo_hip_spg_ts_t *st)
{
    const DevDomain &d = nh::dom();
    T *ua = (T *)st->ua, *va = (T *)st->va, *un = (T *)st->un, *vn = (T *)st->vn;
    // the barotropic work arrays the phase-1 kernel of dyn_spg_ts would fill
    // (zu_frc, zv_frc, zwxb, zwyb) plus the two vertical sums phase 3 needs
    double *w[6] = {nh::scratch2(0), nh::scratch2(1), nh::scratch2(27), nh::scratch2(28), nh::scratch2(2),
                    nh::scratch2(3)};
    Grid2 g = grid2(d.jpi, d.jpj);
    int rc;
    switch (d.nvor_scheme) {
    case NEMO_NP_ENE: rc = launch_step_dyn1_v<T, NEMO_NP_ENE>(d, g, un, vn, wn, ua, va, st, w); break;
    case NEMO_NP_ENS: rc = launch_step_dyn1_v<T, NEMO_NP_ENS>(d, g, un, vn, wn, ua, va, st, w); break;
    case NEMO_NP_MIX: rc = launch_step_dyn1_v<T, NEMO_NP_MIX>(d, g, un, vn, wn, ua, va, st, w); break;
    case NEMO_NP_ENT: rc = launch_step_dyn1_v<T, NEMO_NP_ENT>(d, g, un, vn, wn, ua, va, st, w); break;
    case NEMO_NP_EET: rc = launch_step_dyn1_v<T, NEMO_NP_EET>(d, g, un, vn, wn, ua, va, st, w); break;
    default: rc = launch_step_dyn1_v<T, NEMO_NP_EEN>(d, g, un, vn, wn, ua, va, st, w); break;
    }
    if (rc) return rc;
    if ((rc = launch_dyn_spg_ts<T>(kt, st, 1))) return rc;
    const double z2dt_bf = (kt == d.nit000 && d.neuler == 0) ? d.rdt : 2.0 * d.rdt;
    g.grid.z = zdf_comps(g.grid.x * g.grid.y);
    double *zwd = (double *)nh::scratch3(nh::S_ZWT), *zwd2 = (double *)nh::scratch3(nh::S_ZWT2);
    if constexpr (sizeof(T) == 4) {
        if (zdf_reg<T>(d)) {
            LAUNCHB("step_dyn", (k_step_dyn2<T, true, false>), (S_step_dyn2<T, true, false>), g, d, r2dt, 1.0 / z2dt_bf, ub, vb, ua, va, un, vn, avm,
                   st->rCdU_bot, st->ua_b, st->va_b, st->ub_b, st->vb_b, st->un_adv, st->vn_adv, st->r1_hu_n,
                   st->r1_hv_n, st->un_b, st->vn_b, w[2], w[3], st->utau, utau_b, st->vtau, vtau_b, zwd, zwd2);
            return 0;
        }
    }
#define DYN2_LAUNCH(U) \
    LAUNCHB("step_dyn", (k_step_dyn2<T, false, U>), (S_step_dyn2<T, false, U>), g, d, r2dt, 1.0 / z2dt_bf, ub, vb, ua, va, un, vn, avm, \
           st->rCdU_bot, st->ua_b, st->va_b, st->ub_b, st->vb_b, st->un_adv, st->vn_adv, st->r1_hu_n, st->r1_hv_n, \
           st->un_b, st->vn_b, w[2], w[3], st->utau, utau_b, st->vtau, vtau_b, zwd, zwd2)
    if (d.e3_sij == 0) DYN2_LAUNCH(true);
    else DYN2_LAUNCH(false);
#undef DYN2_LAUNCH
    return 0;
}
template int launch_step_dyn<double>(int, double, const double *, const double *, const double *, const double *,
                                     const double *, const double *, const nemo_hip_spg_ts_t *);
template int launch_step_dyn<float>(int, double, const float *, const float *, const float *, const float *,
                                    const double *, const double *, const nemo_hip_spg_ts_t *);
