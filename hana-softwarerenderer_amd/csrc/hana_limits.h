// hana_limits.h -- what a launch sequence may hold, and the flags of one that
// holds more.  Plain C++, for the kernels and the host.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define HANA_HOST_DEVICE __host__ __device__
#else
#define HANA_HOST_DEVICE
#endif

namespace hana {

enum { FLAG_BIN_OVERFLOW = 1, FLAG_POLY_OVERFLOW = 2, FLAG_POLY_TOO_LARGE = 4, FLAG_CLIPQ_OVERFLOW = 8,
       FLAG_CHUNK_OVERFLOW = 16, FLAG_PAIR_LIMIT = 32, FLAG_QUEUE_STALL = 64 };
// A workspace capacity ran out: the sequence is incomplete, its rasters write
// nothing, and the host grows the workspace and renders it again.
constexpr uint32_t FLAG_CAPACITY = FLAG_BIN_OVERFLOW | FLAG_POLY_OVERFLOW | FLAG_CLIPQ_OVERFLOW | FLAG_CHUNK_OVERFLOW;
// Flags of a sequence whose rasters do nothing.
constexpr uint32_t FLAG_NO_RASTER = FLAG_CAPACITY | FLAG_PAIR_LIMIT;
// (triangle, tile) pairs one launch sequence may hold: bin positions are
// 32-bit.  A sequence with more sets FLAG_PAIR_LIMIT and rasterises nothing.
constexpr uint32_t MAX_PAIRS = 0xFFFFFFF0u;

// The flags of a sequence for its totals: `shared` pairs binned beside the
// `region` entries that set-up workgroups have of their own, of which some are
// used; `wide` pairs of listed triangles, which take no entries.  Past the limit
// for certain, it is refused; where that depends on the entries used, it is
// binned by counting (region 0), which knows.
HANA_HOST_DEVICE inline uint32_t sequence_flags(uint64_t shared, uint64_t region, uint64_t wide, uint64_t bin_cap) {
    if (shared + wide > MAX_PAIRS) return FLAG_PAIR_LIMIT;
    return (shared + region > bin_cap ? FLAG_BIN_OVERFLOW : 0u) | (shared + region + wide > MAX_PAIRS ? FLAG_CHUNK_OVERFLOW : 0u);
}

}  // namespace hana
