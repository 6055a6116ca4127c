// The pair kernel's table Ewald correction instantiations.
#include "nonbonded_kernel.h"

namespace nbx
{

hipError_t launchNonbondedTable(hipStream_t s, const KernelArgs& a, bool energy, bool shiftForces, int numBlocks, int lds,
                               hipEvent_t start, hipEvent_t stop)
{
    return launchElec<kElecEwaldTable>(s, a, energy, shiftForces, numBlocks, lds, start, stop);
}

} // namespace nbx
