// Row kernels for models with HORIPML, two CFS terms (one translation unit per PML form,
// compiled in parallel).
#include "gpx_rows.h"

namespace gpx {
RowKernels row_kernel_hori2(int P, bool C, bool hu, bool big)
{
    return row_kernel_table<0, 2>(P, C, hu, big);
}
}  // namespace gpx
