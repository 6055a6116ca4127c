// The pair kernel's reaction-field and plain cut-off Coulomb instantiations.
#include "nonbonded_kernel.h"

namespace nbx
{

hipError_t launchNonbondedRF(hipStream_t s, const KernelArgs& a, bool energy, bool shiftForces, int numBlocks, int lds,
                            hipEvent_t start, hipEvent_t stop)
{
    return launchElec<kElecRF>(s, a, energy, shiftForces, numBlocks, lds, start, stop);
}

} // namespace nbx
