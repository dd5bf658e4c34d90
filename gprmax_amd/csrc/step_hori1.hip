// Row kernels for models with HORIPML, one CFS term (one translation unit per PML form,
// compiled in parallel).
#include "gpx_rows.h"

namespace gpx {
RowKernels row_kernel_hori1(int P, bool C, bool hu, bool big)
{
    return row_kernel_table<0, 1>(P, C, hu, big);
}
}  // namespace gpx
