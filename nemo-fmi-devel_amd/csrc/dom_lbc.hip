// dom_lbc.hip -- masks / k-indices expansion (DOM/dommsk.F90, DOM/domzgr.F90)
// and the serial lateral boundary fill (LBC/lbc_lnk_generic.h90).
#include "common.hpp"
#include "kernels.hpp"

// ---------------------------------------------------------------------------
// dom_msk: expand the per-column level intervals to NEMO's REAL 0/1 masks.
// One thread per (i,j) column, k-marched, coalesced along i.
// ---------------------------------------------------------------------------
KERNEL void k_dom_msk(DevDomain d, double * __restrict__ tmask, double * __restrict__ umask, double * __restrict__ vmask, double * __restrict__ fmask, double * __restrict__ wmask,
                          double * __restrict__ wumask, double * __restrict__ wvmask, double * __restrict__ ssmask, double * __restrict__ ssumask, double * __restrict__ ssvmask)
{
    THREAD_IJ(1, 1);
    if (i > d.jpi || j > d.jpj) return;
    const size_t ij = IJ(i, j);
    for (int k = 1; k <= d.jpk; k++) {
        if (tmask) A3(tmask, i, j, k) = kmask<double>(d.kT, ij, k);
        if (umask) A3(umask, i, j, k) = kmask<double>(d.kU, ij, k);
        if (vmask) A3(vmask, i, j, k) = kmask<double>(d.kV, ij, k);
        if (fmask) A3(fmask, i, j, k) = kmask<double>(d.kF, ij, k);
        if (wmask) A3(wmask, i, j, k) = wkmask<double>(d.kT, ij, k);
        if (wumask) A3(wumask, i, j, k) = wkmask<double>(d.kU, ij, k);
        if (wvmask) A3(wvmask, i, j, k) = wkmask<double>(d.kV, ij, k);
    }
    if (ssmask) ssmask[ij] = d.ssmask[ij];
    if (ssumask) ssumask[ij] = d.ssumask[ij];
    if (ssvmask) ssvmask[ij] = d.ssvmask[ij];
}

int launch_dom_msk(double *tmask, double *umask, double *vmask, double *fmask, double *wmask, double *wumask,
                   double *wvmask, double *ssmask, double *ssumask, double *ssvmask)
{
    const DevDomain &d = nh::dom();
    Grid2 g = grid2(d.jpi, d.jpj);
    LAUNCH("dom_msk", k_dom_msk, g, d, tmask, umask, vmask, fmask, wmask, wumask, wvmask, ssmask, ssumask, ssvmask);
    return 0;
}

// ---------------------------------------------------------------------------
// lbc_lnk on (jpi,jpj,nk): one block per level; the east-west fill completes
// (barrier) before the north-south fill copies whole rows.  The nk levels may be
// those of several arrays one after the other (two tracers, both betas), so a
// level is addressed from its own 64-bit base: only one array of a domain is
// sure to stay below the 4 GiB that a 32-bit offset reaches.
// ---------------------------------------------------------------------------
template <typename T>
struct S_lbc {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, T * __restrict__ p, int nk, char nat, T pval)
    {
        const int k = (int)vb_.x + 1;
        if (k > nk) return;
        T *__restrict__ q = plane_ptr(p, d.n2, k);
        for (int j = (int)threadIdx.x + 1; j <= d.jpj; j += blockDim.x) {
            if (d.iper) {
                T a = ldp((const T *)q, IJ32(d.jpi - 1, j)), b = ldp((const T *)q, IJ32(2, j));
                stp(q, IJ32(1, j), a);
                stp(q, IJ32(d.jpi, j), b);
            } else {
                if (nat != 'F') stp(q, IJ32(1, j), pval);
                stp(q, IJ32(d.jpi, j), pval);
            }
        }
        __syncthreads();
        for (int i = (int)threadIdx.x + 1; i <= d.jpi; i += blockDim.x) {
            if (d.jper) {
                T a = ldp((const T *)q, IJ32(i, d.jpj - 1)), b = ldp((const T *)q, IJ32(i, 2));
                stp(q, IJ32(i, 1), a);
                stp(q, IJ32(i, d.jpj), b);
            } else {
                if (nat != 'F') stp(q, IJ32(i, 1), pval);
                stp(q, IJ32(i, d.jpj), pval);
            }
        }
    }
};
template <typename T>
KERNEL void k_lbc(DevDomain d, T * __restrict__ p, int nk, char nat, T pval)
{
    S_lbc<T>::run(vb_hw(), d, p, nk, nat, pval);
}

template <typename T>
int launch_lbc(T *p, int nk, char nat, T pval)
{
    const DevDomain &d = nh::dom();
    Grid2 g;
    g.grid = dim3((unsigned)nk, 1, 1);
    g.block = dim3(NH_BLOCK, 1, 1);
    LAUNCHB("lbc_lnk", k_lbc<T>, (S_lbc<T>), g, d, p, nk, nat, pval);
    return 0;
}

// the fill of four arrays of nk levels in one launch (grid.y: the array), for
// the point types whose rule is the same (T, U, V, W; zero on closed sides): a
// launch of one array is too small to fill the chip and costs about 5 us
template <typename T>
struct S_lbc4 {
    static constexpr int NTHR = NH_BLOCK, WAVES = 1;
    __device__ __forceinline__ static void run(const VB &vb_, const DevDomain &d, T *__restrict__ p0, T *__restrict__ p1, T *__restrict__ p2, T *__restrict__ p3, int nk)
    {
        T *p = vb_.y == 0 ? p0 : vb_.y == 1 ? p1 : vb_.y == 2 ? p2 : p3;
        S_lbc<T>::run(vb_, d, p, nk, 'T', T(0));
    }
};
template <typename T>
KERNEL void k_lbc4(DevDomain d, T *__restrict__ p0, T *__restrict__ p1, T *__restrict__ p2, T *__restrict__ p3, int nk)
{
    S_lbc4<T>::run(vb_hw(), d, p0, p1, p2, p3, nk);
}
template <typename T>
int launch_lbc4(T *p0, T *p1, T *p2, T *p3, int nk)
{
    const DevDomain &d = nh::dom();
    Grid2 g;
    g.grid = dim3((unsigned)nk, 4, 1);
    g.block = dim3(NH_BLOCK, 1, 1);
    LAUNCHB("lbc_lnk", k_lbc4<T>, (S_lbc4<T>), g, d, p0, p1, p2, p3, nk);
    return 0;
}
template int launch_lbc4<double>(double *, double *, double *, double *, int);
template int launch_lbc4<float>(float *, float *, float *, float *, int);
template int launch_lbc<double>(double *, int, char, double);
template int launch_lbc<float>(float *, int, char, float);
