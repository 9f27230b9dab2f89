// pair2_unit.hip -- the pair kernel's variants for unit weights (see pair2.hip), in a unit of their own for its flags.
#include "gs_pair_kernel.h"

namespace gs {

hipError_t launch_pair2_unit(const PairArgs& a, const PairVariant& v, size_t lds, int nblocks, int wg, hipStream_t st)
{
    return with_variant<false>(v, [&](auto k) { return k.launch(a, lds, nblocks, wg, st); });
}

int pair2_unit_occupancy(const PairVariant& v, size_t lds, int wg)
{
    return with_variant<false>(v, [&](auto k) { return k.occupancy(lds, wg); });
}

}  // namespace gs
