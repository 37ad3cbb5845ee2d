// sk_tiles_f64.hip -- resident Sinkhorn tiles for float64 costs: at most 64
// entries (128 VGPRs) per lane.
#include "sk_resident_kernel.h"

namespace tmamd {

extern const Tile kTilesF64[] = {
    TM_TILE(double, 4, 16, 1, 4, 2), TM_TILE(double, 4, 16, 1, 4, 8),
    TM_TILE(double, 4, 16, 1, 8, 2), TM_TILE(double, 4, 16, 1, 8, 4),
    TM_TILE(double, 4, 16, 1, 16, 1), TM_TILE(double, 4, 16, 1, 16, 2),
    TM_TILE(double, 8, 16, 1, 4, 12), TM_TILE(double, 8, 16, 1, 8, 6),
    TM_TILE(double, 8, 16, 1, 16, 3), TM_TILE(double, 8, 64, 1, 8, 4),
    TM_TILE(double, 8, 64, 1, 8, 8), TM_TILE(double, 8, 64, 2, 8, 8),
};
extern const int kNumTilesF64 = sizeof(kTilesF64) / sizeof(Tile);

} // namespace tmamd
