// sk_resident.h -- Sinkhorn solves whose matrix stays on the chip (internal).
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

namespace tmamd {

constexpr int kSkMaxSegments = 160;  // runs of one epsilon a schedule may hold

// How a (B, N, M) batch is laid over the chip: `G` workgroups of one tile
// configuration hold one problem (`rows` rows each), `clusters` problems are
// in flight at once.
struct SkResidentPlan {
    int cfg;       // tile configuration (narrow, then wide; float64), -1: not resident
    int G;         // workgroups per problem
    int clusters;  // problems in flight
    int rows;      // rows per workgroup
    int direct;    // every workgroup merges every column (else column owners)
    size_t xch_bytes;  // exchange buffer and the problems' marks (0 when G == 1)
};

SkResidentPlan sk_resident_plan(int64_t B, int64_t N, int64_t M, bool f64);

// Kernel arguments.
struct ResArgs {
    const void *cost;
    const uint8_t *keep;
    const double *lmu, *lnu;
    void *log_u, *log_v;
    double *lu64, *lv64;
    uint64_t *xch;
    uint32_t *given_up;      // a mark per problem
    uint32_t max_polls;      // longest wait for another workgroup
    int64_t B;
    int N, M, Mp;            // Mp: columns rounded up to 16 (exchange rows)
    int G, clusters, rows, direct, cpo;
    int n_iter, nseg, exact_only;
    double rho;
    double eps[kSkMaxSegments];
    int32_t seg_end[kSkMaxSegments];
};

// A tile configuration: NW waves, LC * WC * TC columns by (NW / WC) * RW rows per
// workgroup (RW = TR rows of a wave with LC = 64, 4 * TR with LC = 16), TC * TR
// matrix entries per lane, and its kernels.
struct Tile {
    int NW, LC, WC, TC, TR;
    const void *solo, *shared;  // one workgroup per problem, several
};
extern const Tile kTilesNarrow[], kTilesWide[], kTilesF64[];  // sk_tiles_*.hip
extern const int kNumTilesNarrow, kNumTilesWide, kNumTilesF64;

struct SkResidentIo {
    const void *cost;      // float or double (B, N, M)
    const uint8_t *keep;   // or NULL
    const double *lmu;     // natural log of the marginals, float64
    const double *lnu;
    void *log_u, *log_v;   // outputs in the cost's type
    double *lu64, *lv64;   // the same in float64 (float32 solves), or NULL
    void *xch;             // plan.xch_bytes of device memory
};

// Launches the whole iteration on `stream`.  Returns TM_OK, TM_ERR_LAUNCH, or
// TM_ERR_UNSUPPORTED_SHAPE when the schedule or the device does not allow it
// (nothing was launched then).
int sk_resident_launch(const SkResidentPlan &plan, const SkResidentIo &io, int64_t B, int64_t N,
                       int64_t M, const double *eps_sched, int32_t n_iter, double rho, bool f64,
                       hipStream_t stream);

} // namespace tmamd
