// Device code of the exclusion pass in double, which the pair kernel's last
// workgroups run in the launch's tail: the Coulomb energy terms the pair kernel leaves out,
// the self energy -1/2 epsfac q_i^2 V(0) of every atom
// (kernel_ref_outer.h:286-326) and, for every excluded pair inside the
// cut-off, -epsfac q_i q_j V_corr(r) (Ewald) or epsfac q_i q_j (k_rf r^2 -
// c_rf) (reaction field) (kernel_ref_inner.h: excluded pairs keep the
// correction).
#pragma once

#include "nbx_internal.h"

namespace nbx
{
namespace
{

// V_corr(r) = erf(beta r)/r in double: the double build's table (the pair
// kernel's interpolation formula) or the closed form
__device__ double ewaldCorrectionD(double r, const ExclusionArgs& a)
{
    if (a.elec == kElecEwaldTable)
    {
        const double rs    = r * static_cast<double>(a.ic.tab_scale);
        const int    ri    = min(static_cast<int>(rs), a.ic.tab_n - 2);
        const double frac  = rs - static_cast<double>(ri);
        const double f0    = a.tabD[4 * ri];
        const double fexcl = f0 + frac * a.tabD[4 * ri + 1];
        return a.tabD[4 * ri + 2] - (0.5 / static_cast<double>(a.ic.tab_scale)) * frac * (f0 + fexcl);
    }
    return erf(static_cast<double>(a.ic.beta) * r) / r;
}

// The exclusion pass's terms, in double: the self term -selfCoef q^2 of a
// cluster slot (fillers carry q = 0) ...
__device__ double exclusionSelfEnergy(const ExclusionArgs& a, int slot)
{
    const double q = a.xq[slot].w;
    return -a.selfCoef * q * q;
}

// ... and the energy of an excluded pair inside the cut-off (both atoms as
// cluster slots, each pair once; box edges L).  Every load depends only on the
// index or on one list entry.
__device__ double exclusionPairEnergy(const ExclusionArgs& a, int pair, const float* L)
{
    const int2   ps   = a.pairSlots[pair];
    const float4 pi   = a.xq[ps.x];
    const float4 pj   = a.xq[ps.y];
    double       d[3] = { static_cast<double>(pi.x) - pj.x, static_cast<double>(pi.y) - pj.y,
                    static_cast<double>(pi.z) - pj.z };
    double       r2   = 0.0;
#pragma unroll
    for (int c = 0; c < 3; c++)
    {
        const double edge = L[c];
        d[c] -= edge * rint(d[c] / edge);
        r2 += d[c] * d[c];
    }
    if (r2 < a.rc2)
    {
        const double qq = a.epsfacD * static_cast<double>(pi.w) * static_cast<double>(pj.w);
        return a.elec == kElecRF ? qq * (static_cast<double>(a.ic.k_rf) * r2 - static_cast<double>(a.ic.c_rf))
                                 : -qq * ewaldCorrectionD(sqrt(r2), a);
    }
    return 0.0;
}

// The workgroup's sum of e in a fixed order (the wavefronts' sums through
// sWave, LDS) into partial[blk].
__device__ void exclusionBlockSum(const ExclusionArgs& a, int blk, int nthreads, double e, double* sWave)
{
#pragma unroll
    for (int m = 1; m < 64; m *= 2)
    {
        e += __shfl_xor(e, m, 64);
    }
    if ((threadIdx.x & 63) == 0)
    {
        sWave[threadIdx.x / 64] = e;
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        double t = 0.0;
        for (int w = 0; w < nthreads / 64; w++)
        {
            t += sWave[w];
        }
        a.partial[blk] = t;
    }
}

// One workgroup of the pass.  A single system: slots and pairs blk * nthreads +
// threadIdx.x with stride nblk * nthreads.  A batch: the slots and pairs of its
// block record, which belong to one system.  partial[blk] = the workgroup's
// sum (sWave: LDS, nthreads / 64 doubles).
__device__ void exclusionBlock(const ExclusionArgs& a, int blk, int nblk, int nthreads, double* sWave)
{
    double e = 0.0;
    if (a.blockItems)
    {
        const int4   items = a.blockItems[blk];
        const float* L     = a.boxes + 3 * a.blockSystem[blk];
        const int    n     = max(items.y - items.x, items.w - items.z);
        for (int t = threadIdx.x; t < n; t += nthreads)
        {
            e += items.x + t < items.y ? exclusionSelfEnergy(a, items.x + t) : 0.0;
            e += items.z + t < items.w ? exclusionPairEnergy(a, items.z + t, L) : 0.0;
        }
    }
    else
    {
        const int n = max(a.nslot, a.npairs);
        for (int t = blk * nthreads + static_cast<int>(threadIdx.x); t < n; t += nblk * nthreads)
        {
            e += t < a.nslot ? exclusionSelfEnergy(a, t) : 0.0;
            e += t < a.npairs ? exclusionPairEnergy(a, t, a.box) : 0.0;
        }
    }
    exclusionBlockSum(a, blk, nthreads, e, sWave);
}

} // namespace
} // namespace nbx
