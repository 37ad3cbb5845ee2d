// sk_tiles_wide.hip -- resident Sinkhorn tiles of up to 4096 columns (float32): 24
// to 128 entries per lane.  Four waves have 512 VGPRs a lane, eight have 256: there
// the tiles of 128 entries spill about 120 and those of 96 up to 50 (hipcc's
// report), in the building of P and around its calls; the products of a step read
// none back, the rest of it some eight addresses.
#include "sk_resident_kernel.h"

namespace tmamd {

extern const Tile kTilesWide[] = {
    TM_TILE(float, 4, 64, 1, 6, 4), TM_TILE(float, 4, 64, 1, 6, 8), TM_TILE(float, 4, 64, 1, 6, 16),
    TM_TILE(float, 4, 64, 1, 8, 4), TM_TILE(float, 4, 64, 1, 8, 8), TM_TILE(float, 4, 64, 1, 8, 12),
    TM_TILE(float, 4, 64, 1, 12, 4), TM_TILE(float, 4, 64, 1, 12, 8),
    TM_TILE(float, 4, 64, 1, 16, 4), TM_TILE(float, 4, 64, 1, 16, 8),
    TM_TILE(float, 8, 64, 1, 6, 16), TM_TILE(float, 8, 64, 1, 8, 12),
    TM_TILE(float, 8, 64, 1, 12, 8), TM_TILE(float, 8, 64, 1, 16, 8),
    TM_TILE(float, 8, 64, 2, 12, 4), TM_TILE(float, 8, 64, 2, 12, 8),
    TM_TILE(float, 8, 64, 2, 16, 4), TM_TILE(float, 8, 64, 2, 16, 8),
    TM_TILE(float, 8, 64, 4, 12, 4), TM_TILE(float, 8, 64, 4, 12, 8),
    TM_TILE(float, 8, 64, 4, 16, 4), TM_TILE(float, 8, 64, 4, 16, 8),
};
extern const int kNumTilesWide = sizeof(kTilesWide) / sizeof(Tile);

} // namespace tmamd
