// Row kernels for models without PML slabs (one translation unit per PML form,
// compiled in parallel).
#include "gpx_rows.h"

namespace gpx {
RowKernels row_kernel_plain(int P, bool C, bool hu, bool big)
{
    return row_kernel_table<0, 0>(P, C, hu, big);
}

}  // namespace gpx
