// The pair kernel's analytical Ewald correction instantiations.
#include "nonbonded_kernel.h"

namespace nbx
{

hipError_t launchNonbondedAnalytical(hipStream_t s, const KernelArgs& a, bool energy, bool shiftForces, int numBlocks, int lds,
                                    hipEvent_t start, hipEvent_t stop)
{
    return launchElec<kElecEwaldAna>(s, a, energy, shiftForces, numBlocks, lds, start, stop);
}

} // namespace nbx
