// hana_types.h -- data layouts shared by the host runtime and the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hana_limits.h"

namespace hana {

enum {
    SHADER_GROUND = 0,
    SHADER_TOON = 1,
    SHADER_TEXTURE = 2,
    SHADER_TEXTURE_LIGHT = 3,
    SHADER_BLINN = 4,
    SHADER_NORMALMAP = 5,
    SHADER_SHADOW = 6
};

// Screen tiles are 2^shift pixels a side: 16x16 (shift 4) by default, 32x32
// (shift 5) where a batch's tuning picks it.  Every kernel that maps pixels
// to tiles is instantiated for both.
constexpr int TILE_SHIFT_DEFAULT = 4;
constexpr int TILE_SHIFT_MAX = 5;
__host__ __device__ constexpr int tile_edge(int shift) { return 1 << shift; }
constexpr int BLOCK = 256;                 // threads per workgroup (4 wave64)
#ifndef HANA_SMALL_PIX
#define HANA_SMALL_PIX 32
#endif
// In passes of over 4 target pixels per face, small triangles of more than
// HANA_MED_PIX candidates are shared by HANA_MED_LANES lanes each instead of
// looped over by one: a wave's trip count is then bounded by HANA_SMALL_PIX /
// HANA_MED_LANES.  Passes of smaller faces
// (micro-triangle meshes) keep one lane per triangle, which their few
// candidates suit better.
#ifndef HANA_MED_PIX
#define HANA_MED_PIX 4
#endif
#ifndef HANA_MED_LANES
#define HANA_MED_LANES 4
#endif
// A raster workgroup (one tile at a time) has 2 or 4 waves: 128 or 256 lanes,
// at most one lane per pixel of a 16x16 tile.
static_assert(HANA_SMALL_PIX >= 1 && HANA_SMALL_PIX <= 32, "small-triangle candidates: at most 32");
#ifndef HANA_VPT
#define HANA_VPT 4
#endif
#ifndef HANA_FPT
#define HANA_FPT 4
#endif
constexpr int VPT = HANA_VPT;              // vertices per thread in k_vertex
constexpr int FPT = HANA_FPT;              // faces per thread in k_setup
#ifndef HANA_FRONT_FPT
#define HANA_FRONT_FPT 1
#endif
constexpr int FRONT_FPT = HANA_FRONT_FPT;  // faces per thread in k_front
constexpr int FRONT_VPT = 1;               // vertices per thread in k_front
// Vertices the device keeps of a clipped polygon: a convex polygon gains at
// most one vertex per plane (3 + 7), rounding in the inside tests can add a
// few more; one lane of a 16-lane clip group holds each.
constexpr int POLY_MAX = 16;
constexpr int FAN_BITS = 4;                // fan index of a clipped triangle in its bin entry
constexpr uint32_t POOL_CAP_MAX = (1u << (31 - FAN_BITS)) - 1u;   // polygons a workspace may hold
constexpr int POLY_VARY = 8;               // varyings stored per clipped vertex
constexpr uint32_t NO_WINNER = 0xFFFFFFFFu;
constexpr uint32_t CLIPPED_BIT = 0x80000000u;

// Uniform block of one pass, derived on the host from ShaderData
// (SR/IShader.h:17-32) with the products the reference recomputes per vertex
// folded once: clip_m = camera_vp*model (ObjectToClipPos, SR/IShader.h:55-57),
// light_m = light_vp*model (ObjectToViewPos, SR/IShader.h:59-61).
struct DevUniforms {
    float clip_m[16];
    float light_m[16];
    float model[16];
    float model_inv[16];
    float light_vp[16];
    float view_pos[4];
    float light_dir[4];
    float light_color[4];
    float ambient[4];
    float mat_color[4];
    float mat_spec[4];
    float gloss;
    float bump_scale;
    int32_t enable_shadow;
    int32_t shadow_fp32;         // fp32 shadow-map extension (hana_uniforms)
};

// One pass = one graphics_draw_triangle call over a mesh into a target.
struct PassDesc {
    // mesh (structure of arrays)
    const float* px; const float* py; const float* pz;
    const float* nx; const float* ny; const float* nz;
    const float* tu; const float* tv;
    const int32_t* idx;          // 3 per face
    int32_t nverts, nfaces;
    int32_t kind, nvary;
    const DevUniforms* u;
    // textures: RGBA8 words in TGAColor byte order
    const uint32_t* diffuse; int32_t dw, dh;
    const uint32_t* normal;  int32_t nw, nh;
    // shadow map sampled by the fragment program (RGBA8 target words, and
    // its fp32 depth for the fp32 extension)
    const uint32_t* shadow; int32_t sw, sh;
    const float* shadow_depth;
    // target
    uint32_t* color; float* depth; uint32_t* winner;
    int32_t width, height, tiles_x, tiles_y;
    int32_t clear;               // 1: the target is cleared to clear_rgba/clear_depth first
    uint32_t clear_rgba; float clear_depth;
    int32_t share_small;         // 1: the pass averages over 4 target pixels per face (see HANA_MED_PIX)
    // workspace slices owned by this pass
    float4* vr;                  // per vertex: ndc.x, ndc.y, ndc.z, 1/w
    float* vs;                   // per vertex: nvary varyings
    uint8_t* code;               // per vertex: bit 7 is_vertex_visible, bit p outside clip plane p
    int32_t* poly_of_face;       // clipped polygon of a face (-1: none)
    uint64_t* stats;             // 5 counters (hana_pass_stats order), or null
    // first block of this pass in each kernel's grid / first global tile
    int32_t vblock0, fblock0, tile0, tblock0;
    int32_t index;               // of this pass in its sequence (its list of wide triangles)
    int32_t pad_;
};

// Buffers shared by every pass of one launch sequence.
//
// The (triangle, tile) pairs of a sequence are held as chunks: the entries of
// one set-up workgroup's triangles that touch one tile, contiguous in `bins`.
// Each tile has chunk_cap places for its chunks' descriptors, filled in the
// order the workgroups reach it.  A pair outside any workgroup's table (a
// clipped fan triangle, a table overflow) is a descriptor that holds its entry
// itself (CHUNK_INLINE).  So one pass over the triangles bins them, without
// counts, a scan or a second pass, and a raster workgroup reads its tile's
// descriptors with one coalesced load.  A triangle over more than WIDE_TILES
// tiles goes to its pass's list instead, which every tile of the pass tests.
// Where a tile has no place left the sequence is binned by counting
// (launch_counted), with the range of its pairs as each tile's one chunk.
struct Workspace {
    uint2* chunks;               // per tile, chunk_cap: first bin entry and entries, or entry and CHUNK_INLINE
    uint32_t chunk_cap;
    uint32_t* bins;              // triangle entries: face id and its FACE_* bits, or CLIPPED_BIT | polygon << 4 | fan
    uint32_t wide_cap;
    uint2* wide;                 // per pass, wide_cap: box of tiles (wide_box) and bin entry
    float4* pool_vr;             // clipped polygons: POLY_MAX vertices each
    float* pool_vs;              //   ... POLY_VARY varyings per vertex
    int32_t* pool_face;          //   face (within its pass) of each polygon
    uint64_t* clip_queue;        // faces failing the trivial accept: pass << 32 | face
    // counters of this sequence, all zero when its first triangle is set up:
    // the SEQ_* words, then a count of wide triangles per pass, then a count
    // of chunks per tile
    uint32_t* seq;
    uint32_t* wide_count;
    uint32_t* tile_chunks;
    // words the sequence's first kernel zeroes: the counters themselves where a
    // launch precedes set-up, else those of the workspace's other counter set
    uint32_t* zero;
    uint32_t zero_n;
    uint32_t* status;            // see STATUS_*
    uint32_t* status_out;        // or null: host-mapped copy of the status words, written by the raster
    uint32_t bin_cap;
    uint32_t faces;              // of all passes
    uint32_t seg_region;         // bin entries that belong to one set-up workgroup each; the rest is shared
    uint32_t poly_cap;
    uint32_t clipq_cap;
    // queue of the persistent raster (k_raster_q): its items are the tiles of
    // every pass in global tile order (shadow passes first, then main passes
    // that sample no map drawn here, then those that do)
    // (its state: seq[SEQ_QUEUE] the next item, seq[SEQ_QUEUE_DONE] the
    // group-0 tiles finished and published)
    uint32_t q_items;            // tiles of all passes
    uint32_t q_g0;               // tiles of group-0 passes
    uint32_t q_dep_from;         // first item of a pass that samples a map drawn by group 0
    int32_t tile_shift;          // tiles are 2^tile_shift pixels a side
    // per raster group, or null: for every run of 2^TILE_PASS_SHIFT
    // workgroups of k_raster, the pass (from the group's first) of the run's
    // first tile, with TILE_PASS_PURE set when the whole run lies in it, and
    // that pass's tile0 - tblock0 (workgroup b of it renders global tile
    // b + that)
    const uint2* tile_pass[2];
};
// A plane on its way to host memory in bands (k_read_back).
constexpr int READ_BANDS = 8;              // of a plane
constexpr uint32_t READ_WGS = 32;          // workgroups per band
constexpr uint32_t READ_BAND_MIN = 1u << 17;   // words of a band, at least
// The tables of a sequence of at most FRONT_PASSES passes, as launch arguments.
constexpr int FRONT_PASSES = 2;
struct FrontTables {
    PassDesc d[FRONT_PASSES];
    DevUniforms u[FRONT_PASSES];
};

constexpr int TILE_PASS_SHIFT = 6;
constexpr uint32_t TILE_PASS_PURE = 0x80000000u;

constexpr uint32_t SEG_PAIRS = 2;          // bin entries of a set-up workgroup, per face
constexpr uint32_t CHUNK_INLINE = 0x80000000u;
constexpr uint32_t CHUNK_SLACK = 16;       // places per tile beyond a reported need
// Triangles over more than WIDE_TILES tiles are listed once per pass, up to
// Workspace::wide_cap of them (WIDE_MAX, or none or all with counted binning);
// later ones take a descriptor in each of their tiles.
constexpr int WIDE_TILES = 16;
#ifndef HANA_WIDE_MAX
#define HANA_WIDE_MAX 512
#endif
constexpr uint32_t WIDE_MAX = HANA_WIDE_MAX;

// counter words of one sequence: polygons allocated, faces queued for
// clipping, the flags it raised, the most chunks of a tile with more than its
// places, the persistent raster's queue, and (64-bit
// each) the pairs outside the set-up workgroups' own entries and the pairs of
// the listed wide triangles; of counted binning, all pairs in the first of them,
// and whether they fit
enum { SEQ_POLYS = 0, SEQ_CLIPQ = 1, SEQ_FLAGS = 2, SEQ_MAX_CHUNKS = 3, SEQ_PAIRS = 4, SEQ_WIDE_PAIRS = 6,
       SEQ_QUEUE = 8, SEQ_QUEUE_DONE = 9, SEQ_COUNTED = 10, SEQ_WORDS = 16 };
// status words: set across sequences until the host reads them at a sync
// point, so that calls need not wait for one another: the flags of every
// sequence and the largest needs seen: of places for descriptors, in units of
// 1024 over all tiles of the sequence; and the complements of the faces and tiles of the smallest sequences that ran out of
// descriptors.
enum { STATUS_FLAGS = 0, STATUS_NEED_BINS = 1, STATUS_NEED_POLYS = 2, STATUS_NEED_CHUNKS = 3, STATUS_OVER_FACES = 4,
       STATUS_OVER_TILES = 5, STATUS_WORDS = 6 };
// vertex outcode bits
constexpr uint32_t CODE_VISIBLE = 0x80u;
constexpr uint32_t CODE_PLANES = 0x7Fu;
enum { ST_FACES = 0, ST_CLIPPED = 1, ST_POLYS = 2, ST_ENTRIES = 3, ST_PIXELS = 4, ST_WORDS = 5 };

}  // namespace hana
