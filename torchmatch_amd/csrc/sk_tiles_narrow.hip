// sk_tiles_narrow.hip -- resident Sinkhorn tiles of up to 256 columns (float32):
// TC * TR entries per lane, at most 128 (of 512 VGPRs in four waves; in eight, of
// 256, where the tiles of 128 spill: see sk_tiles_wide.hip).
#include "sk_resident_kernel.h"

namespace tmamd {

extern const Tile kTilesNarrow[] = {
    TM_TILE(float, 4, 16, 1, 4, 2), TM_TILE(float, 4, 16, 1, 4, 4), TM_TILE(float, 4, 16, 1, 4, 8),
    TM_TILE(float, 4, 16, 1, 4, 16), TM_TILE(float, 4, 16, 1, 6, 2), TM_TILE(float, 4, 16, 1, 6, 4),
    TM_TILE(float, 4, 16, 1, 6, 8), TM_TILE(float, 4, 16, 1, 6, 16), TM_TILE(float, 4, 16, 1, 8, 2),
    TM_TILE(float, 4, 16, 1, 8, 4), TM_TILE(float, 4, 16, 1, 8, 8), TM_TILE(float, 4, 16, 1, 8, 12),
    TM_TILE(float, 4, 16, 1, 12, 2), TM_TILE(float, 4, 16, 1, 12, 4),
    TM_TILE(float, 4, 16, 1, 12, 8), TM_TILE(float, 4, 16, 1, 16, 1),
    TM_TILE(float, 4, 16, 1, 16, 2), TM_TILE(float, 4, 16, 1, 16, 4),
    TM_TILE(float, 4, 16, 1, 16, 6), TM_TILE(float, 8, 16, 1, 4, 16),
    TM_TILE(float, 8, 16, 1, 8, 12), TM_TILE(float, 8, 16, 1, 12, 8),
    TM_TILE(float, 8, 16, 1, 16, 8),
};
extern const int kNumTilesNarrow = sizeof(kTilesNarrow) / sizeof(Tile);

} // namespace tmamd
