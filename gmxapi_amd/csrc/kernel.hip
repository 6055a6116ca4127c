// Launching of the pair kernel (nonbonded_kernel.h): its LDS and the choice of
// the Coulomb flavour's instantiations.
#include <map>
#include <mutex>
#include <utility>

#include "nonbonded_kernel.h"

namespace nbx
{

hipError_t allowDynamicLds(const void* fn, int lds)
{
    if (lds <= 64 * 1024)
    {
        return hipSuccess;
    }
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
    {
        return e;
    }
    static std::mutex                                 lock;
    static std::map<std::pair<const void*, int>, int> allowed;
    std::lock_guard<std::mutex>                       guard(lock);
    int&                                              cur = allowed[{ fn, dev }];
    if (lds > cur)
    {
        e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e == hipSuccess)
        {
            cur = lds;
        }
    }
    return e;
}

int nonbondedLdsBytes(int ntype, int tabN, int elec, int windowSlots, bool ljPme)
{
    const LdsLayout L(ntype, elec == kElecEwaldTable ? tabN + 1 : 0, windowSlots, ljPme);
    return L.end_ * 16;
}

hipError_t launchNonbonded(hipStream_t s, const KernelArgs& a, int elec, bool energy, bool shiftForces, int numBlocks,
                           hipEvent_t start, hipEvent_t stop)
{
    if (a.ngroups == 0 || numBlocks == 0)
    {
        return hipSuccess;
    }
    const int lds = nonbondedLdsBytes(a.ntype, a.ic.tab_n, elec, a.windowSlots, a.ljPme != 0);
    if (elec == kElecRF)
    {
        return launchNonbondedRF(s, a, energy, shiftForces, numBlocks, lds, start, stop);
    }
    if (elec == kElecEwaldAna)
    {
        return launchNonbondedAnalytical(s, a, energy, shiftForces, numBlocks, lds, start, stop);
    }
    return launchNonbondedTable(s, a, energy, shiftForces, numBlocks, lds, start, stop);
}

} // namespace nbx
