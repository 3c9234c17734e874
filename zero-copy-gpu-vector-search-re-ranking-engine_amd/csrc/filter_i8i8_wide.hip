// The filter scan (filter_kernel.hpp) over per-vector int8 rows of more than 512 bytes.
#include "filter_kernel.hpp"

namespace zcgvs_hip {

template int launchFilterKind<kFilterPerVector, true>(const ScanArgs&, const FilterArgs&, const PhaseArgs&,
                                                    const EmitArgs&, int, hipStream_t);

}  // namespace zcgvs_hip
