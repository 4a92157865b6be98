// hana_launch.h -- host-callable launch wrappers of the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "hana_types.h"

namespace hana {

hipError_t launch_vertex(const PassDesc* d_passes, int npasses, const Workspace& ws, int blocks, hipStream_t s);
hipError_t launch_setup(const PassDesc* d_passes, int npasses, const Workspace& ws, int blocks, bool small_tris,
                        hipStream_t s);
hipError_t launch_clip(const PassDesc* d_passes, const Workspace& ws, hipStream_t s);
// Set-up and clipping twice, to count and then to place every pair (after the
// vertices).  With `first`, the counters of a chunked binning before, all of it
// runs only where that one ran out of descriptors or bins.
struct CountedBins {
    uint32_t* pairs;         // per tile, zero
    uint32_t* next;          // per tile
    uint32_t* first;
    uint32_t region;         // the chunked binning's Workspace::seg_region
};
hipError_t launch_counted(const PassDesc* d_passes, int npasses, const Workspace& ws, const CountedBins& b, int blocks, hipStream_t s);
// vertex, set-up and clipping in one launch; `tables` (or null: they are in
// device memory already) come with it and are stored at d_passes and d_unis
hipError_t launch_front(const FrontTables* tables, PassDesc* d_passes, DevUniforms* d_unis, int npasses, const Workspace& ws,
                        int fblocks, int vblocks, hipStream_t s);
// one workgroup of `waves` (2 or 4) waves per tile of dependency group `group` (ws.tile_shift selects the tile size)
hipError_t launch_raster(const PassDesc* d_passes, int npasses, const Workspace& ws, int blocks, int group, int waves,
                         hipStream_t s);
// the persistent raster over every pass of the sequence: `workgroups` workgroups take tiles from a queue
hipError_t launch_raster_queue(const PassDesc* d_passes, int npasses, const Workspace& ws, int workgroups,
                               int waves, hipStream_t s);
hipError_t launch_fill32(uint32_t* dst, uint32_t value, size_t n, hipStream_t s);
// One plane of w x h words into host-mapped memory, as k_present does (flip) or
// as it is, in bands of `band` words; band i stored, flags[i] becomes epoch.
// done: READ_BANDS device words, zero before the first launch.
hipError_t launch_read_back(const uint32_t* src, uint32_t* dst, int w, int h, bool flip, uint32_t band, uint32_t* done,
                            uint32_t* flags, uint32_t epoch, hipStream_t s);
hipError_t launch_present(const uint32_t* src, uint32_t* dst, int w, int h, hipStream_t s);

}  // namespace hana
