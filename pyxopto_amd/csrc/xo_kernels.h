/*
 * xo_kernels.h — launch parameters of the transport kernels (host and
 * device view; plain data, passed by value as the single kernel argument).
 */
#ifndef XO_KERNELS_H
#define XO_KERNELS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/xomc.h"

/* Threads per block: 4 wave64 wavefronts. */
#define XO_BLOCK 256
#define XO_MAX_BLOCK 1024 /* of a run with a fluence window in LDS */

/* Per-run counters accumulated by the kernels. */
enum {
    XO_STAT_STEPS = 0,     /* transport-loop iterations                  */
    XO_STAT_BOUNDARY = 1,  /* iterations that ended on a boundary        */
    XO_STAT_PACKETS = 2,   /* packets launched                           */
    XO_STAT_THREADS = 3,   /* lanes that launched at least one packet    */
    XO_STAT_CROSSINGS = 4, /* mcvox: voxel faces crossed                 */
    XO_STAT_DEPOSITS = 5,  /* non-zero fluence deposits: adds in LDS, in a
                              lane's cache or in memory                  */
    XO_STAT_TRUNCATED = 6, /* packets stopped at XO_MAX_PACKET_STEPS     */
    XO_STAT_COUNT = 7
};

/* Largest detector-bin count privatized in LDS, and largest LUT (floats)
 * staged in LDS; beyond these the kernels use global memory. */
#define XO_LDS_BINS_MAX 1024u
#define XO_LDS_LUT_MAX 4096u

namespace xo {

/* A fluence grid as the single-simulation kernels read it per deposit.
 * origin, ext, bins: the box of bins (x or r, y, z; x fastest) that a block
 * of a single-simulation kernel accumulates in LDS and adds to the
 * accumulator once; bins 0: none. */
struct alignas(16) FluenceL {
    float top_left[3];
    float k;               /* float to integer weight                     */
    float inv_step[3];
    int32_t enabled;       /* enum xo_fluence_kind                        */
    float shape[3];
    uint32_t offset;
    uint32_t origin[3];
    uint32_t nx;           /* bins of a row ...                           */
    uint32_t ext[3];
    uint32_t ny;           /* ... and rows of a slice (1 for r-z)         */
    uint32_t bins;
    int32_t rate;
};

inline FluenceL fluence_to_device(const xo_fluence &F) {
    FluenceL o = {};
    for (int k = 0; k < 3; ++k) {
        o.top_left[k] = F.top_left[k];
        o.inv_step[k] = F.inv_step[k];
        o.shape[k] = (float)F.shape[k];
    }
    o.k = (float)F.k;
    o.enabled = F.enabled;
    o.offset = F.offset;
    o.nx = F.shape[0];
    o.ny = F.enabled == XO_FLUENCE_XYZ ? F.shape[1] : 1u;
    o.rate = F.rate;
    return o;
}

/* A fluence grid in the header of a batch instance: the same fields without
 * the window, in 60 bytes (FluenceL takes 96: a batch of 16,800 instances
 * that fits XO_NOALLOC_SCRATCH_BYTES with these would not with those). */
struct FluenceGrid {
    float top_left[3];
    float k;
    float inv_step[3];
    int32_t enabled;
    float shape[3];
    uint32_t offset;
    uint32_t nx, ny;
    int32_t rate;
};

inline FluenceGrid fluence_without_window(const FluenceL &F) {
    return FluenceGrid{{F.top_left[0], F.top_left[1], F.top_left[2]}, F.k,
                       {F.inv_step[0], F.inv_step[1], F.inv_step[2]}, F.enabled,
                       {F.shape[0], F.shape[1], F.shape[2]}, F.offset, F.nx, F.ny, F.rate};
}

struct McmlParams {
    xo_mcml_cfg cfg;
    xo_trace trace;        /* max_events 0: no trace                      */
    float *trace_data;     /* [packet][max_events][XO_TRACE_ENTRY_LEN]    */
    int32_t *trace_n;      /* [packet] event counts                       */
    const uint32_t *table; /* seed-table multipliers (XO_FLAG_PACKET_KEYED) */
    const float *lut;
    uint64_t *rng_x;
    const uint32_t *rng_a;
    unsigned long long *counter;
    unsigned long long *accum;
    unsigned long long *stats;
    uint64_t npackets;
    uint32_t lanes;
    uint32_t flags;
    uint32_t lds_bins;
    uint32_t lds_lut;
    FluenceL fluence;      /* the grid of cfg.fluence, with its window    */
    uint32_t pf_rare;      /* some medium needs the general phase-function
                              sampling code (xo::pf_rare): which build runs */
};

struct McvoxParams {
    xo_mcvox_cfg cfg;
    xo_trace trace;        /* max_events 0: no trace                      */
    float *trace_data;     /* [packet][max_events][XO_TRACE_ENTRY_LEN]    */
    int32_t *trace_n;      /* [packet] event counts                       */
    const uint32_t *table; /* seed-table multipliers (XO_FLAG_PACKET_KEYED) */
    const uint8_t *voxels; /* material index per voxel, [z][y][x] */
    const float *lut;
    uint64_t *rng_x;
    const uint32_t *rng_a;
    unsigned long long *counter;
    unsigned long long *accum;
    unsigned long long *stats;
    uint64_t npackets;
    uint32_t lanes;
    uint32_t flags;
    uint32_t lds_bins;
    uint32_t lds_lut;
    FluenceL fluence;      /* the grid of cfg.fluence, with its window    */
};

/* Largest window: zeroing and adding it up costs every block about a
 * microsecond per 4096 bins. */
constexpr uint32_t kFluenceWindowMax = 10240;

size_t mcml_lds_bytes(const McmlParams &P);
size_t mcvox_lds_bytes(const McvoxParams &P);
/* Blocks of `block` threads (at most XO_MAX_BLOCK). */
hipError_t launch_mcml(const McmlParams &P, uint32_t blocks, uint32_t block, hipStream_t stream);
hipError_t launch_mcvox(const McvoxParams &P, uint32_t blocks, uint32_t block,
                        hipStream_t stream);
/* Resident blocks per CU of the build that launch_mcml / launch_mcvox would
 * run for P, at this block size and P's LDS. */
hipError_t occupancy_mcml(const McmlParams &P, uint32_t block, int *blocks_per_cu);
hipError_t occupancy_mcvox(const McvoxParams &P, uint32_t block, int *blocks_per_cu);

} // namespace xo

#endif /* XO_KERNELS_H */
