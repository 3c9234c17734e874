// The filter scan (filter_kernel.hpp) over matrix-scale int8 rows of up to 512 bytes.
#include "filter_kernel.hpp"

namespace zcgvs_hip {

template int launchFilterKind<ZCGVS_DTYPE_I8, false>(const ScanArgs&, const FilterArgs&, const PhaseArgs&, const EmitArgs&,
                                               int, hipStream_t);

}  // namespace zcgvs_hip
