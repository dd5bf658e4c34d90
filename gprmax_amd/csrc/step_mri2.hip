// Row kernels for models with MRIPML, two CFS terms (one translation unit per PML form,
// compiled in parallel).
#include "gpx_rows.h"

namespace gpx {
RowKernels row_kernel_mri2(int P, bool C, bool hu, bool big)
{
    return row_kernel_table<1, 2>(P, C, hu, big);
}
}  // namespace gpx
