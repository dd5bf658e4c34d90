// Row kernels for models with MRIPML, one CFS term (one translation unit per PML form,
// compiled in parallel).
#include "gpx_rows.h"

namespace gpx {
RowKernels row_kernel_mri1(int P, bool C, bool hu, bool big)
{
    return row_kernel_table<1, 1>(P, C, hu, big);
}
}  // namespace gpx
