// CIC internals shared with the tiled path (pm_gravity.hip).
#pragma once

#include "pm_common.h"

namespace pm {

// mesh += sum val W with float atomics (pm_cic_scatter's kernel, one channel) over the values (a
// scalar counts as 1) of smaller magnitude than *above, or over all when it is NaN.
int cic_scatter_rest(const int16_t* pmid, const float* disp, const uint8_t* valid, const float* val, float val_scalar,
                     int64_t n, const pm_cic_geom* geom, float* mesh, const float* above, hipStream_t s);

}  // namespace pm
