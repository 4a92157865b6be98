// hana_runtime.cpp -- the C ABI (include/hana_gpu.h): device objects, pass
// planning, workspace management and the kernel launch sequence.
//
// A pass is one graphics_draw_triangle call (SR/graphics.cpp:378-407).  A
// frame is DrawModel::draw (SR/scene.h:53-99): an optional shadow pass into
// the shadow map, the main pass sampling it, then the shadow-map clear.  Any
// set of passes is rendered by one launch sequence over per-pass descriptor
// tables (geometry in one launch or three, then the raster of each dependency
// group), so a single frame and a batch of hundreds of frames run the same
// code; batches are captured once into a hipGraph.
#include <hip/hip_runtime.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/hana_gpu.h"
#include "hana_hostmath.h"
#include "hana_internal.h"
#include "hana_launch.h"
#include "hana_types.h"

using namespace hana;
using namespace hana::rt;

extern "C" {
static uint32_t batch_take_flags(hana_ctx* c, hana_batch* b, uint32_t* parts);
static int batch_recount(hana_ctx* c, hana_batch* b, uint32_t parts);
static int batch_launch(hana_ctx* c, hana_batch* b);
}

namespace hana {
namespace rt {

int fail(hana_ctx* c, int code, const std::string& msg) {
    if (c) c->err = msg;
    return code;
}
int hip_fail(hana_ctx* c, hipError_t e, const char* what) {
    return fail(c, HANA_E_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}
#define HIP_TRY(c, expr)                                   \
    do {                                                   \
        hipError_t e_ = (expr);                            \
        if (e_ != hipSuccess) return hip_fail(c, e_, #expr); \
    } while (0)

hipStream_t slot_stream(hana_ctx* c, int k) { return k ? c->xstream[k - 1] : c->stream; }
Arena& slot_arena(hana_ctx* c, int k) { return k ? c->xarena[k - 1] : c->arena; }
uint32_t* slot_status(hana_ctx* c, int k) { return k ? c->xstatus_host[k - 1] : c->status_host; }

int sync_all(hana_ctx* c) {
    for (int k = 0; k < c->nslots; k++)
        if (slot_stream(c, k)) HIP_TRY(c, hipStreamSynchronize(slot_stream(c, k)));
    for (auto& row : c->pend)
        for (auto& p : row) p.clear();   // every draw has completed
    return HANA_OK;
}

int join(hana_ctx* c) {
    for (int k = 1; k < c->nslots; k++)
        if (!c->pend[k][0].empty()) {
            HIP_TRY(c, hipStreamWaitEvent(c->stream, c->slot_done[k], 0));
            c->pend[k][0].clear();
        }
    return HANA_OK;
}

// The distinct targets a set of passes draws or samples.
static std::vector<hana_target*> touched_targets(const std::vector<PassSpec>& specs) {
    std::vector<hana_target*> t;
    for (const PassSpec& s : specs)
        for (hana_target* x : {s.target, s.shadow})
            if (x && std::find(t.begin(), t.end(), x) == t.end()) t.push_back(x);
    return t;
}
// Whether a call on slot a that touches targets t must wait for slot k: only
// for the calls that touched one of them last (each waited for the ones before
// it), unless slot a's stream has waited for them already.
static bool must_wait(const hana_ctx* c, int k, int a, const std::vector<hana_target*>& t) {
    const std::vector<hana_target*>& pend = c->pend[k][a];
    for (hana_target* x : t)
        if (x->slot == k && std::find(pend.begin(), pend.end(), x) != pend.end()) return true;
    return false;
}
// Notes work on slot k's stream, complete at slot_done[k], that touches
// targets t, for every other slot to wait for before it touches them.
static void note_pending(hana_ctx* c, int k, const std::vector<hana_target*>& t) {
    for (hana_target* x : t) x->slot = k;
    for (int b = 0; b < c->nslots; b++)
        if (b != k)
            for (hana_target* x : t)
                if (std::find(c->pend[k][b].begin(), c->pend[k][b].end(), x) == c->pend[k][b].end())
                    c->pend[k][b].push_back(x);
}

int ensure(hana_ctx* c, DevBuf& b, size_t bytes) {
    if (bytes <= b.cap) return HANA_OK;
    if (b.p) {
        int r = sync_all(c);
        if (r) return r;
        HIP_TRY(c, hipFree(b.p));
        b.p = nullptr;
        b.cap = 0;
    }
    size_t nb = std::max(bytes, (size_t)256);
    hipError_t e = hipMalloc(&b.p, nb);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(c, HANA_E_NOMEM, "device allocation of " + std::to_string(nb) + " bytes failed");
    }
    b.cap = nb;
    return HANA_OK;
}

uint32_t pack_bytes(const uint8_t rgba[4]) {
    return (uint32_t)rgba[0] | ((uint32_t)rgba[1] << 8) | ((uint32_t)rgba[2] << 16) | ((uint32_t)rgba[3] << 24);
}

int materialize_clear(hana_ctx* c, hana_target* t, hipStream_t s) {
    if (!t->pending_clear) return HANA_OK;
    size_t n = (size_t)t->w * t->h;
    HIP_TRY(c, launch_fill32(t->color, t->clear_rgba, n, s));
    uint32_t db;
    std::memcpy(&db, &t->clear_depth, 4);
    HIP_TRY(c, launch_fill32(reinterpret_cast<uint32_t*>(t->depth), db, n, s));
    t->pending_clear = false;
    return HANA_OK;
}

// Lays out the workspace of a set of passes.  Passes are ordered (stably) by
// raster group, and within the main group those that sample a shadow map
// drawn by the first group come last: the persistent raster's queue holds the
// tiles in pass order, so every shadow tile precedes the tiles that wait for
// them.  Every per-pass slice is aligned to the vertices of a workgroup.
int build_plan(hana_ctx* c, std::vector<PassSpec> specs, Plan& pl, const Tuning& tu, size_t front_faces, bool counted) {
    {
        std::vector<std::pair<int, size_t>> key(specs.size());
        for (size_t i = 0; i < specs.size(); i++) {
            const PassSpec& s = specs[i];
            bool dep = false;
            if (s.shadow && s.group == 1)
                for (const PassSpec& o : specs) dep = dep || (o.group == 0 && o.target == s.shadow);
            key[i] = {s.group * 2 + (dep ? 1 : 0), i};
        }
        std::stable_sort(key.begin(), key.end(),
                         [](const std::pair<int, size_t>& a, const std::pair<int, size_t>& b) { return a.first < b.first; });
        std::vector<PassSpec> sorted;
        sorted.reserve(specs.size());
        for (auto& k : key) sorted.push_back(specs[k.second]);
        pl = Plan();
        specs.swap(sorted);
        // the first pass that waits for the shadow tiles
        size_t first_dep = specs.size();
        for (size_t i = 0; i < key.size(); i++)
            if (key[i].first == 3) { first_dep = i; break; }
        pl.q_dep_from = (uint32_t)first_dep;   // a pass index until the tiles are known (below)
    }
    const int tshift = tu.tile_shift, tedge = tile_edge(tu.tile_shift);
    pl.specs = specs;
    int n = (int)specs.size();
    size_t faces = 0;
    for (const PassSpec& s : specs) faces += (size_t)s.mesh->F;
    pl.counted = counted;
    pl.front = !counted && faces <= front_faces;
    pl.args = pl.front && n <= FRONT_PASSES;
    const size_t vchunk = (size_t)BLOCK * (pl.front ? FRONT_VPT : VPT), fchunk = (size_t)BLOCK * (pl.front ? FRONT_FPT : FPT);
    pl.descs.resize(n);
    pl.unis.resize(n);
    size_t voff = 0, vsoff = 0, fo = 0;
    int vb = 0, fb = 0, tile0 = 0;
    int tb[2] = {0, 0};
    pl.small_tris = true;
    for (int i = 0; i < n; i++) {
        const PassSpec& s = specs[i];
        if (s.group < 0 || s.group > 1) return fail(c, HANA_E_INVALID, "bad pass group");
        PassDesc& d = pl.descs[i];
        std::memset(&d, 0, sizeof d);
        derive_dev_uniforms(s.u, pl.unis[i]);
        hana_mesh* m = s.mesh;
        d.nverts = m->V;
        d.nfaces = m->F;
        d.kind = s.kind;
        d.nvary = (s.kind == SHADER_GROUND || s.kind == SHADER_TOON || s.kind == SHADER_SHADOW) ? 1
                  : (s.kind == SHADER_TEXTURE ? 2 : 8);
        size_t V = (size_t)m->V;
        d.px = m->soa; d.py = m->soa + V; d.pz = m->soa + 2 * V;
        d.nx = m->soa + 3 * V; d.ny = m->soa + 4 * V; d.nz = m->soa + 5 * V;
        d.tu = m->soa + 6 * V; d.tv = m->soa + 7 * V;
        d.idx = m->idx;
        if (s.diffuse) { d.diffuse = s.diffuse->texels; d.dw = s.diffuse->w; d.dh = s.diffuse->h; }
        if (s.normal) { d.normal = s.normal->texels; d.nw = s.normal->w; d.nh = s.normal->h; }
        if (s.shadow) {
            d.shadow = s.shadow->color;
            d.shadow_depth = s.shadow->depth;
            d.sw = s.shadow->w;
            d.sh = s.shadow->h;
        }
        hana_target* t = s.target;
        d.color = t->color; d.depth = t->depth; d.winner = t->winner;
        d.width = t->w; d.height = t->h;
        d.tiles_x = (t->w + tedge - 1) / tedge;
        d.tiles_y = (t->h + tedge - 1) / tedge;
        d.share_small = (int64_t)t->w * t->h > 4 * (int64_t)m->F;
        if (d.share_small) pl.small_tris = false;
        size_t vpad = (V + vchunk - 1) / vchunk * vchunk;
        // slices: pointers are resolved by bind_plan once the arena exists
        pl.v_off.push_back(voff);
        pl.vs_off.push_back(vsoff);
        pl.f_off.push_back(fo);
        voff += vpad;
        vsoff += vpad * (size_t)d.nvary;
        fo += (size_t)m->F;
        d.vblock0 = vb;
        vb += (int)(vpad / vchunk);
        d.fblock0 = fb;
        fb += (int)(((size_t)m->F + fchunk - 1) / fchunk);
        d.tile0 = tile0;
        tile0 += d.tiles_x * d.tiles_y;
        d.tblock0 = tb[s.group];
        tb[s.group] += d.tiles_x * d.tiles_y;
        d.index = i;
    }
    pl.vblocks = vb;
    pl.fblocks = fb;
    // more faces than leave the set-up workgroups bin positions of their own
    if (!pl.front && (uint64_t)fb * SEG_PAIRS * BLOCK * FPT + 4096 > MAX_PAIRS) pl.counted = true;
    pl.total_v = voff;
    pl.total_vs = vsoff;
    pl.total_f = fo;
    pl.total_tiles = tile0;
    pl.tile_shift = tshift;
    // Waves per raster workgroup.  Until the caller sets them, a group of many
    // 16x16 tiles, so that their workgroups run in several rounds, takes two: a workgroup's life is mostly waits (for its pass, its tile's chunks,
    // entries, indices and vertices, each behind the one before), and 13 of 2
    // waves fit a CU where 8 of 4 do.  With fewer tiles, or with smaller
    // triangles, more of which keep four waves busy, four are faster.  4 and 2
    // waves, us per frame (frame-sized shadow map): 3840x2160 of 100,000 faces
    // 129 and 98, of 1,000,000 (8 pixels each) 155 and 137; 2560x1440 of
    // 300,000 (12) 80 and 73, of 1,000,000 (3.7) 98 and 109; 1920x1080 (8,160
    // tiles) of 300,000 (7) 61 and 67; 1366x768 of 100,000 35 and 44.  A batch of
    // 64 scenes of 1,000-200,000 faces, 128^2-1024^2, 421 and, in the parts that
    // this takes, 412.
    for (int g = 0; g < 2; g++) {
        int64_t px = 0, faces = 0;
        for (const PassSpec& s : specs)
            if (s.group == g) {
                px += (int64_t)s.target->w * s.target->h;
                faces += s.mesh->F;
            }
        const bool two = tu.auto_waves && tu.raster_wgs_per_cu == 0 && tshift == 4 && tb[g] >= 10000 && px >= 4 * faces;
        pl.raster_waves[g] = two ? 2 : tu.raster_waves;
    }
    pl.raster_wgs = tu.raster_wgs_per_cu > 0 ? tu.raster_wgs_per_cu * c->num_cus : 0;
    pl.q_g0 = (uint32_t)tb[0];
    pl.q_dep_from = pl.q_dep_from < (uint32_t)n ? (uint32_t)pl.descs[pl.q_dep_from].tile0 : (uint32_t)tile0;
    pl.ngroups = 0;
    for (int g = 0; g < 2; g++) {
        int first = -1, count = 0;
        for (int i = 0; i < n; i++)
            if (specs[i].group == g) {
                if (first < 0) first = i;
                count++;
            }
        pl.group_first[g] = first < 0 ? 0 : first;
        pl.group_count[g] = count;
        pl.group_blocks[g] = tb[g];
    }
    // k_raster's pass of each run of 2^TILE_PASS_SHIFT workgroups (a group's
    // passes are contiguous, in tblock0 order): one scalar load per workgroup
    // instead of a binary search over the group's descriptors
    pl.tile_pass.clear();
    for (int g = 0; g < 2 && !pl.args; g++) {
        pl.tp_first[g] = (int)pl.tile_pass.size();
        const int first = pl.group_first[g], cnt = pl.group_count[g], nb = pl.group_blocks[g];
        const int run = 1 << TILE_PASS_SHIFT;
        int p = 0;
        for (int b0 = 0; cnt > 0 && b0 < nb; b0 += run) {
            while (p + 1 < cnt && pl.descs[first + p + 1].tblock0 <= b0) p++;
            const int last = std::min(b0 + run, nb) - 1;
            const bool pure = !(p + 1 < cnt && pl.descs[first + p + 1].tblock0 <= last);
            const PassDesc& d = pl.descs[first + p];
            pl.tile_pass.push_back(make_uint2((uint32_t)p | (pure ? TILE_PASS_PURE : 0u), (uint32_t)(d.tile0 - d.tblock0)));
        }
    }
    return HANA_OK;
}

// Words of a sequence's counters: the SEQ_* words, the passes' wide triangles,
// the tiles' chunks; with counted binning, also the tiles' pairs and next places.
static size_t tile_words(const Plan& pl) { return ((size_t)pl.total_tiles + 3) & ~(size_t)3; }
static size_t counter_words(const Plan& pl) {
    return (size_t)SEQ_WORDS + ((pl.descs.size() + 3) & ~(size_t)3) + (pl.counted ? 3 : 1) * tile_words(pl);
}

// Points the plan's workspace at counter set k of the arena.
static void set_counters(Plan& pl, Arena& A, int k) {
    Workspace& ws = pl.ws;
    ws.seq = A.counters[k].as<uint32_t>();
    ws.wide_count = ws.seq + SEQ_WORDS;
    ws.tile_chunks = ws.wide_count + ((pl.descs.size() + 3) & ~(size_t)3);
}

// Per-call sequences: the arena's next counter set, which the call before left
// zeroed, with the other one to be zeroed by this call's first launch.
static int take_counters(hana_ctx* c, Plan& pl, Arena& A, hipStream_t s) {
    const int k = A.counters_next;
    if (A.counters_used[k]) {   // a call before failed to launch
        HIP_TRY(c, launch_fill32(A.counters[k].as<uint32_t>(), 0u, A.counters_used[k], s));
        A.counters_used[k] = 0;
    }
    set_counters(pl, A, k);
    pl.ws.zero = A.counters[k ^ 1].as<uint32_t>();
    pl.ws.zero_n = (uint32_t)A.counters_used[k ^ 1];
    A.counters_used[k] = counter_words(pl);
    return HANA_OK;
}
static void counters_launched(Arena& A) {
    A.counters_used[A.counters_next ^ 1] = 0;
    A.counters_next ^= 1;
}

// An arena's chunk descriptors; without memory for them it has none.
static int ensure_chunks(hana_ctx* c, Arena& A, uint64_t slots) {
    int r = ensure(c, A.chunks, sizeof(uint2) * slots);
    A.chunk_slots = r ? A.chunks.cap / sizeof(uint2) : std::max(slots, A.chunk_slots);
    return r;
}

// Allocates the arena for a plan and resolves the slice pointers.
int bind_plan(hana_ctx* c, Plan& pl, Arena& A, uint32_t min_bins, uint32_t min_polys, bool with_stats,
              hipStream_t s) {
    int n = (int)pl.descs.size();
    int r;
    pl.uni_off = (sizeof(PassDesc) * std::max(n, 1) + 255) & ~(size_t)255;
    pl.tp_off = (pl.uni_off + sizeof(DevUniforms) * std::max(n, 1) + 255) & ~(size_t)255;
    if ((r = ensure(c, A.tables, pl.tp_off + sizeof(uint2) * std::max<size_t>(pl.tile_pass.size(), 1)))) return r;
    if ((r = ensure(c, A.vr, sizeof(float4) * std::max<size_t>(pl.total_v, 1)))) return r;
    if ((r = ensure(c, A.vs, sizeof(float) * std::max<size_t>(pl.total_vs, 1)))) return r;
    if ((r = ensure(c, A.code, std::max<size_t>(pl.total_v, 4)))) return r;
    if ((r = ensure(c, A.pof, sizeof(int32_t) * std::max<size_t>(pl.total_f, 1)))) return r;
    size_t nt = (size_t)pl.total_tiles + 1;
    // (triangle, tile) entries: most triangles touch one tile and about half
    // are culled; the raster reports the exact need if this is exceeded
    const uint64_t seg_region = pl.counted ? 0 : (uint64_t)pl.fblocks * SEG_PAIRS * BLOCK * (pl.front ? FRONT_FPT : FPT);
    uint64_t want_bins = std::max<uint64_t>({(uint64_t)min_bins, (uint64_t)4 * pl.total_f + 2 * nt, 1u << 22,
                                             seg_region + (uint64_t)pl.total_f + 4096});
    if ((uint64_t)pl.fblocks * BLOCK * FPT + 4096 > MAX_PAIRS) return fail(c, HANA_E_NOMEM, "launch sequence too large (faces)");
    want_bins = std::min<uint64_t>(want_bins, MAX_PAIRS);
    if (want_bins > A.bin_cap) {
        if ((r = ensure(c, A.bins, sizeof(uint32_t) * want_bins))) return r;
        A.bin_cap = (uint32_t)want_bins;
    }
    // chunk descriptors (by counting a tile's only chunk is its range of the bins)
    const uint64_t tiles = (uint64_t)std::max(pl.total_tiles, 1);
    const uint64_t want_cap = pl.counted ? 32 : tile_places(pl.total_f, tiles);
    uint64_t want_slots = tiles * want_cap;
    if (want_slots > A.chunk_slots && (r = ensure_chunks(c, A, want_slots))) return r;
    if ((r = ensure(c, A.wide, sizeof(uint2) * WIDE_MAX * std::max(n, 1)))) return r;
    uint64_t want_polys = std::max<uint64_t>({(uint64_t)min_polys, pl.total_f / 16 + 4096});
    want_polys = std::min<uint64_t>(want_polys, POOL_CAP_MAX);
    if (want_polys > A.poly_cap) {
        if ((r = ensure(c, A.pool_vr, sizeof(float4) * POLY_MAX * want_polys))) return r;
        if ((r = ensure(c, A.pool_vs, sizeof(float) * POLY_MAX * POLY_VARY * want_polys))) return r;
        if ((r = ensure(c, A.pool_face, sizeof(int32_t) * want_polys))) return r;
        A.poly_cap = (uint32_t)want_polys;
    }
    // every face may fail the trivial accept (camera inside the mesh)
    uint64_t want_q = std::max<uint64_t>(pl.total_f, 1024);
    want_q = std::min<uint64_t>(want_q, 0xFFFFFFF0ull);
    if (want_q > A.clipq_cap) {
        if ((r = ensure(c, A.clip_queue, sizeof(uint64_t) * want_q))) return r;
        A.clipq_cap = (uint32_t)want_q;
    }
    for (int k = 0; k < 2; k++) {
        const size_t bytes = sizeof(uint32_t) * counter_words(pl);
        if (bytes <= A.counters[k].cap) continue;
        if ((r = ensure(c, A.counters[k], bytes))) return r;
        HIP_TRY(c, launch_fill32(A.counters[k].as<uint32_t>(), 0u, A.counters[k].cap / sizeof(uint32_t), s));
        A.counters_used[k] = 0;
    }
    bool fresh_status = A.status.p == nullptr;
    if ((r = ensure(c, A.status, sizeof(uint32_t) * STATUS_WORDS))) return r;
    if (fresh_status) HIP_TRY(c, launch_fill32(A.status.as<uint32_t>(), 0u, STATUS_WORDS, s));
    if ((r = ensure(c, A.stats, sizeof(uint64_t) * ST_WORDS * std::max(n, 1)))) return r;
    for (int i = 0; i < n; i++) {
        PassDesc& d = pl.descs[i];
        size_t voff = pl.v_off[i], vsoff = pl.vs_off[i], fo = pl.f_off[i];
        d.vr = A.vr.as<float4>() + voff;
        d.vs = A.vs.as<float>() + vsoff;
        d.code = A.code.as<uint8_t>() + voff;
        d.poly_of_face = A.pof.as<int32_t>() + fo;
        d.u = reinterpret_cast<const DevUniforms*>(A.tables.as<char>() + pl.uni_off) + i;
        d.stats = with_stats ? A.stats.as<uint64_t>() + (size_t)ST_WORDS * i : nullptr;
    }
    Workspace& ws = pl.ws;
    ws.bins = A.bins.as<uint32_t>();
    ws.chunks = A.chunks.as<uint2>();
    // whole 32-byte groups of descriptors (loaded four at a time), an odd
    // number of them so that the tiles' first groups spread over the caches
    uint64_t groups = std::min<uint64_t>(A.chunk_slots / tiles / 4, 1u << 28);
    ws.chunk_cap = (uint32_t)(4 * (groups - 1 + (groups & 1)));
    ws.wide = A.wide.as<uint2>();
    ws.wide_cap = pl.counted ? 0 : WIDE_MAX;
    ws.pool_vr = A.pool_vr.as<float4>();
    ws.pool_vs = A.pool_vs.as<float>();
    ws.pool_face = A.pool_face.as<int32_t>();
    ws.clip_queue = A.clip_queue.as<uint64_t>();
    ws.clipq_cap = A.clipq_cap;
    // the counters zeroed by the sequence itself; per-call sequences take
    // theirs at the launch (take_counters)
    set_counters(pl, A, 0);
    ws.zero = ws.seq;
    ws.zero_n = (uint32_t)counter_words(pl);
    ws.status = A.status.as<uint32_t>();
    ws.status_out = nullptr;
    ws.bin_cap = A.bin_cap;
    ws.faces = (uint32_t)std::min<size_t>(pl.total_f, 0xFFFFFFFFu);
    ws.seg_region = (uint32_t)seg_region;
    ws.poly_cap = A.poly_cap;
    ws.q_items = (uint32_t)pl.total_tiles;
    ws.q_g0 = pl.q_g0;
    ws.q_dep_from = pl.q_dep_from;
    ws.tile_shift = pl.tile_shift;
    for (int g = 0; g < 2; g++)
        ws.tile_pass[g] = pl.group_count[g] > 0 && !pl.args
                              ? reinterpret_cast<const uint2*>(A.tables.as<char>() + pl.tp_off) + pl.tp_first[g]
                              : nullptr;
    return HANA_OK;
}

// Resolves clear flags of the plan's targets (fused into their first pass).
void take_clears(Plan& pl) {
    for (size_t i = 0; i < pl.descs.size(); i++) {
        hana_target* t = pl.specs[i].target;
        PassDesc& d = pl.descs[i];
        d.clear = 0;
        if (t->pending_clear) {
            d.clear = 1;
            d.clear_rgba = t->clear_rgba;
            d.clear_depth = t->clear_depth;
            t->pending_clear = false;
        }
    }
}

hipEvent_t pool_event(hana_ctx* c) {
    if (!c->ev_pool.empty()) {
        hipEvent_t e = c->ev_pool.back();
        c->ev_pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
}

// Records an event pair around one launch when timing is on (never inside a
// graph capture: `timed` is false there).
struct StageTimer {
    hana_ctx* c;
    int stage;
    bool on;
    hipEvent_t a = nullptr, b = nullptr;
    StageTimer(hana_ctx* c_, int st, bool timed, hipStream_t s) : c(c_), stage(st), on(timed && c_->timing) {
        if (on) {
            a = pool_event(c);
            b = pool_event(c);
            on = a && b && hipEventRecord(a, s) == hipSuccess;
        }
    }
    void done(hipStream_t s) {
        if (on && hipEventRecord(b, s) == hipSuccess) c->ev_pending.push_back({stage, {a, b}});
    }
};

// The geometry stages: vertex, set-up with binning, clipping; or all of them
// in one launch (timed as set-up), before which a sequence that zeroes its own
// counters does so; or vertex and counted binning (also timed as set-up).
int enqueue_geometry(hana_ctx* c, const Plan& pl, const Arena& A, hipStream_t s, bool timed) {
    PassDesc* d = A.tables.as<PassDesc>();
    int n = (int)pl.descs.size();
    if (pl.front) {
        DevUniforms* u = reinterpret_cast<DevUniforms*>(A.tables.as<char>() + pl.uni_off);
        Workspace ws = pl.ws;
        FrontTables t;
        if (pl.args) {
            for (int i = 0; i < n; i++) {
                t.d[i] = pl.descs[i];
                t.u[i] = pl.unis[i];
            }
        }
        StageTimer timer(c, 1, timed, s);
        if (ws.zero == ws.seq) {
            HIP_TRY(c, launch_fill32(ws.zero, 0u, ws.zero_n, s));
            ws.zero_n = 0;
        }
        HIP_TRY(c, launch_front(pl.args ? &t : nullptr, d, u, n, ws, pl.fblocks, pl.vblocks, s));
        timer.done(s);
        return HANA_OK;
    }
    {
        StageTimer t(c, 0, timed, s);
        HIP_TRY(c, launch_vertex(d, n, pl.ws, pl.vblocks, s));
        t.done(s);
    }
    if (pl.counted) {
        StageTimer t(c, 1, timed, s);
        uint32_t* const pairs = pl.ws.tile_chunks + tile_words(pl);
        HIP_TRY(c, launch_counted(d, n, pl.ws, {pairs, pairs + tile_words(pl), nullptr, 0}, pl.fblocks, s));
        t.done(s);
        return HANA_OK;
    }
    {
        StageTimer t(c, 1, timed, s);
        HIP_TRY(c, launch_setup(d, n, pl.ws, pl.fblocks, pl.small_tris, s));
        t.done(s);
    }
    {
        StageTimer t(c, 2, timed, s);
        HIP_TRY(c, launch_clip(d, pl.ws, s));
        t.done(s);
    }
    return HANA_OK;
}

// The raster stages: one launch per dependency group, or one persistent
// launch for both (timed as the first group's stage).
int enqueue_raster(hana_ctx* c, const Plan& pl, const Arena& A, hipStream_t s, bool timed) {
    const PassDesc* d = A.tables.as<PassDesc>();
    if (pl.raster_wgs > 0) {
        StageTimer t(c, 6, timed, s);
        HIP_TRY(c, launch_raster_queue(d, (int)pl.descs.size(), pl.ws, pl.raster_wgs, pl.raster_waves[0], s));
        t.done(s);
        return HANA_OK;
    }
    for (int g = 0; g < 2; g++)
        if (pl.group_count[g]) {
            StageTimer t(c, 6 + g, timed, s);
            HIP_TRY(c, launch_raster(d + pl.group_first[g], pl.group_count[g], pl.ws, pl.group_blocks[g], g,
                                    pl.raster_waves[g], s));
            t.done(s);
        }
    return HANA_OK;
}

int enqueue_sequence(hana_ctx* c, const Plan& pl, const Arena& A, hipStream_t s, bool timed = true) {
    // every kernel reads the workspace: a plan that was never bound to an
    // arena must not reach the device
    if (pl.descs.empty() || !pl.ws.status || !A.tables.p)
        return fail(c, HANA_E_INVALID, "internal error: a sequence without a bound plan");
    int r = enqueue_geometry(c, pl, A, s, timed);
    return r ? r : enqueue_raster(c, pl, A, s, timed);
}

// Uploads descriptors and uniforms through a pinned staging slot.
// Stages the plan's descriptors and uniforms in the pinned ring and copies
// them into the arena's tables buffer (one copy).
int upload_tables(hana_ctx* c, const Plan& pl, Arena& A, hipStream_t s) {
    size_t nd = sizeof(PassDesc) * pl.descs.size(), nu = sizeof(DevUniforms) * pl.unis.size();
    size_t nt = sizeof(uint2) * pl.tile_pass.size();
    size_t need = pl.tp_off + nt;
    if (need > c->ring_bytes) {
        int r = sync_all(c);
        if (r) return r;
        for (int i = 0; i < kRing; i++) {
            if (c->ring_host[i]) HIP_TRY(c, hipHostFree(c->ring_host[i]));
            c->ring_host[i] = nullptr;
            c->ring_used[i] = false;
        }
        c->ring_bytes = 0;
        for (int i = 0; i < kRing; i++) HIP_TRY(c, hipHostMalloc(&c->ring_host[i], need * 2));
        c->ring_bytes = need * 2;
    }
    int slot = c->ring_next;
    c->ring_next = (c->ring_next + 1) % kRing;
    if (c->ring_used[slot]) HIP_TRY(c, hipEventSynchronize(c->ring_event[slot]));
    char* h = static_cast<char*>(c->ring_host[slot]);
    std::memcpy(h, pl.descs.data(), nd);
    std::memcpy(h + pl.uni_off, pl.unis.data(), nu);
    if (nt) std::memcpy(h + pl.tp_off, pl.tile_pass.data(), nt);
    HIP_TRY(c, hipMemcpyAsync(A.tables.p, h, need, hipMemcpyHostToDevice, s));
    HIP_TRY(c, hipEventRecord(c->ring_event[slot], s));
    c->ring_used[slot] = true;
    return HANA_OK;
}

// The largest needs (STATUS_NEED_*) that sequences reported, and their flags.
struct Needs {
    uint32_t w[STATUS_WORDS] = {};
    void take(const uint32_t* status) {
        w[STATUS_FLAGS] |= status[STATUS_FLAGS];
        for (int i = STATUS_FLAGS + 1; i < STATUS_WORDS; i++) w[i] = std::max(w[i], status[i]);
    }
};

// The places for chunk descriptors that an overflow asks for: those of its
// fullest tile, and a quarter more, in all tiles.
static uint64_t full_places(const Needs& need) { return (uint64_t)need.w[STATUS_NEED_CHUNKS] * 1024 / 4 * 5; }
static bool chunks_grow(const Needs& need) { return full_places(need) <= kGrownChunks; }
static int grow_chunks(hana_ctx* c, Arena& A, const Needs& need) {
    return ensure_chunks(c, A, std::max(full_places(need), A.chunk_slots));
}
// Sequences of the size of those that ran out of descriptors bin by counting from now on.
static void count_such(hana_ctx* c, const Needs& need) {
    c->counted_faces = std::min<size_t>(c->counted_faces, ~need.w[STATUS_OVER_FACES]);
    c->counted_tiles = std::min<size_t>(c->counted_tiles, ~need.w[STATUS_OVER_TILES]);
}

// Grows an arena's bins, chunk descriptors and clip pool to the needs reported
// by an overflow (capacities never shrink).
static int grow_arena(hana_ctx* c, Arena& A, const Needs& need) {
    const uint32_t flags = need.w[STATUS_FLAGS], need_bins = need.w[STATUS_NEED_BINS],
                   need_polys = need.w[STATUS_NEED_POLYS];
    if ((flags & FLAG_BIN_OVERFLOW) && (!(flags & FLAG_CHUNK_OVERFLOW) || chunks_grow(need))) {
        uint64_t want = std::max<uint64_t>((uint64_t)need_bins + need_bins / 4 + 1024, A.bin_cap);
        want = std::min<uint64_t>(want, MAX_PAIRS);
        int r = ensure(c, A.bins, sizeof(uint32_t) * want);
        if (r) return r;
        A.bin_cap = (uint32_t)want;
    }
    if (flags & FLAG_CHUNK_OVERFLOW) {
        // without memory for the places, too
        int r = chunks_grow(need) ? grow_chunks(c, A, need) : HANA_E_NOMEM;
        if (r == HANA_E_NOMEM) count_such(c, need);
        else if (r) return r;
    }
    if (flags & FLAG_POLY_OVERFLOW) {
        uint64_t want = std::max<uint64_t>((uint64_t)need_polys + need_polys / 4 + 1024, A.poly_cap);
        want = std::min<uint64_t>(want, POOL_CAP_MAX);
        int r;
        if ((r = ensure(c, A.pool_vr, sizeof(float4) * POLY_MAX * want))) return r;
        if ((r = ensure(c, A.pool_vs, sizeof(float) * POLY_MAX * POLY_VARY * want))) return r;
        if ((r = ensure(c, A.pool_face, sizeof(int32_t) * want))) return r;
        A.poly_cap = (uint32_t)want;
    }
    return HANA_OK;
}

// Whether a per-call sequence of this size bins by counting.
static bool bins_by_counting(const hana_ctx* c, size_t faces, size_t tiles) {
    return c->count_next || (faces >= c->counted_faces && tiles >= c->counted_tiles);
}

// Renders a logged call again on the context stream with slot 0's workspace
// (every stream is idle: the status check has waited for them).
static int replay_call(hana_ctx* c, LoggedCall& L, bool counted) {
    int r;
    if (counted && !L.pl.counted) {
        // laid out anew, with the clears that the call took
        Tuning t;
        t.tile_shift = L.pl.tile_shift;
        if (c->num_cus > 0) t.raster_wgs_per_cu = L.pl.raster_wgs / c->num_cus;
        Plan pl;
        if ((r = build_plan(c, L.pl.specs, pl, t, 0, true))) return r;
        for (size_t i = 0; i < pl.descs.size(); i++) {
            const PassDesc& d = L.pl.descs[i];
            pl.descs[i].clear = d.clear;
            pl.descs[i].clear_rgba = d.clear_rgba;
            pl.descs[i].clear_depth = d.clear_depth;
        }
        L.pl = std::move(pl);
    }
    Plan& pl = L.pl;
    Arena& A = slot_arena(c, 0);
    if ((r = bind_plan(c, pl, A, 0, 0, false, c->stream))) return r;
    pl.ws.status_out = c->status_dev[0];
    if ((r = take_counters(c, pl, A, c->stream))) return r;
    if (!pl.args && (r = upload_tables(c, pl, A, c->stream))) return r;
    if ((r = enqueue_geometry(c, pl, A, c->stream, false))) return r;
    counters_launched(A);
    for (const Fill& f : L.fills) {
        size_t n = (size_t)f.target->w * f.target->h;
        HIP_TRY(c, launch_fill32(f.target->color, f.rgba, n, c->stream));
        uint32_t db;
        std::memcpy(&db, &f.depth, 4);
        HIP_TRY(c, launch_fill32(reinterpret_cast<uint32_t*>(f.target->depth), db, n, c->stream));
    }
    return enqueue_raster(c, pl, A, c->stream, false);
}

// Reads the sticky status of every sequence since the last check, over all
// draw slots (waits for every stream).
// - A capacity overflow (bins, chunk descriptors, clip pool, clip queue) left its
//   sequence's targets untouched.  Every slot's workspace is grown to the
//   largest need seen and the calls since the last check are rendered again
//   in call order; a draw over the same state twice leaves it as drawn once
//   (the depth test keeps the last of the fragments at the minimum depth), so
//   the targets end as the calls in order leave them.  What the chunked binning
//   needs varies with the order in which workgroups arrive, so the second time
//   they bin by counting, whose needs are exact; so do, from then on, sequences
//   like one whose descriptors no workspace grows to.  With replay_overflow
//   off, the caller is asked to render again (HANA_E_OVERFLOW).
// - The same in a part of a batch that was run since: the part is sized again, by
//   counting, and the batches are run again in the order of their last runs, then
//   the calls, all of which came after them (hana_batch_run).
// - More (triangle, tile) pairs than 32-bit bins reach: that sequence was not
//   rasterised (HANA_E_NOMEM).
// - A clipped polygon with more than POLY_MAX vertices was dropped, the rest
//   drawn (HANA_E_UNSUPPORTED).
int check_status(hana_ctx* c) {
    if (!c->status_pending && !c->noalloc_pending && c->batches.empty()) return HANA_OK;
    int r;
    uint32_t seen = 0;
    auto forget = [&] {
        c->log.clear();
        c->batches.clear();
        c->status_pending = false;
    };
    for (int attempt = 0;; attempt++) {
        if ((r = sync_all(c))) return r;
        Needs need;
        for (int k = 0; k < c->nslots; k++) {
            const uint32_t* host = slot_status(c, k);
            if (!host) continue;
            need.take(host);
        }
        const uint32_t flags = need.w[STATUS_FLAGS];
        seen |= flags;
        if (flags) {
            for (int k = 0; k < c->nslots; k++) {
                uint32_t* host = slot_status(c, k);
                if (!host) continue;
                Arena& A = slot_arena(c, k);
                if (A.status.p) HIP_TRY(c, launch_fill32(A.status.as<uint32_t>(), 0u, STATUS_WORDS, c->stream));
                std::memset(host, 0, sizeof(uint32_t) * STATUS_WORDS);
            }
            // the next geometry stages may run on any stream
            HIP_TRY(c, hipStreamSynchronize(c->stream));
        }
        uint32_t cap = flags & FLAG_CAPACITY;
        if (cap)
            for (int k = 0; k < (c->pipelined ? c->nslots : 1); k++)
                if ((r = grow_arena(c, slot_arena(c, k), need))) {
                    forget();
                    return r;
                }
        bool rerun = false;
        for (hana_batch* b : c->batches) {
            uint32_t parts = 0;
            const uint32_t f = batch_take_flags(c, b, &parts) & ~(uint32_t)FLAG_POLY_TOO_LARGE;
            seen |= f;
            if (!(f & FLAG_CAPACITY)) continue;
            rerun = true;
            if ((r = batch_recount(c, b, parts))) {
                forget();
                return r;
            }
        }
        if (rerun && c->noalloc_pending) {
            // the frame may have drawn over the batch's targets, and cannot be drawn again
            forget();
            return fail(c, HANA_E_OVERFLOW,
                        "a batch outgrew its workspace and left targets as they were, and a no-alloc frame followed it; "
                        "the workspace was grown, render both again");
        }
        if ((rerun || (cap && c->replay_overflow)) && attempt < 4) {
            c->replays++;
            for (hana_batch* b : c->batches)
                if (rerun && (r = batch_launch(c, b))) {
                    forget();
                    return r;
                }
            for (LoggedCall& L : c->log)
                if ((r = replay_call(c, L, attempt > 0 || bins_by_counting(c, L.pl.total_f, L.pl.total_tiles)))) {
                    forget();
                    return r;
                }
            continue;   // wait for the replay and check it
        }
        forget();
        c->count_next = cap && !c->replay_overflow;
        if (cap || rerun)
            return fail(c, HANA_E_OVERFLOW,
                        c->replay_overflow ? "workspace capacity still exceeded after growing it four times"
                                           : "bin or clip-pool capacity exceeded since the last sync; buffers were "
                                             "grown, render those frames again");
        break;
    }
    // no-alloc frames: no workspace to grow, their errors are reported
    uint32_t na = 0;
    if (c->noalloc_pending) {
        na = c->noalloc_status_host[STATUS_FLAGS];
        std::memset(c->noalloc_status_host, 0, sizeof(uint32_t) * STATUS_WORDS);
        c->noalloc_pending = false;
    }
    if ((seen | na) & FLAG_QUEUE_STALL)
        return fail(c, HANA_E_DEVICE, "the persistent raster's wait for the shadow tiles timed out");
    if (na & FLAG_CAPACITY)
        return fail(c, HANA_E_OVERFLOW,
                    "a hana_render_frame_noalloc frame outgrew the bins or clip pool of the no-alloc scratch and left "
                    "its targets untouched; render it with hana_render_frame");
    seen |= na;
    if (seen & FLAG_PAIR_LIMIT)
        return fail(c, HANA_E_NOMEM,
                    "a draw, frame or batch part covered more than 4,294,967,280 (triangle, tile) pairs and was not "
                    "rasterised; split it");
    if (seen & FLAG_POLY_TOO_LARGE)
        return fail(c, HANA_E_UNSUPPORTED,
                    "a clipped polygon had more than " + std::to_string(POLY_MAX) +
                        " vertices and was dropped; the rest was drawn");
    return HANA_OK;
}

// The tuning of a per-call sequence.  Until the caller sets one, sequences of
// few large triangles take 32x32 tiles: a raster workgroup's fixed part (the
// tile's counters, its pass's wide triangles, a handful of dependent loads)
// then serves four times the pixels.  Where the targets have so many tiles
// that the workgroups run in several rounds, that is what they spend their
// time on; with fewer tiles the larger ones leave CUs idle, with smaller
// triangles their lanes.  Measured with 16x16 and 32x32 tiles, us per frame:
// 3840x2160 of 1,000 faces 77 and 47, of 20,000 81 and 48, of 100,000 (83
// pixels each) 78 and 63; 1920x1080 of 5,000 faces 27 and 21, of 20,000 (104)
// 26 and 24, with a frame-sized shadow map 48 and 56, of 100,000 32 and 43;
// 1280x720 of 1,000 faces 15 and 18.  The last condition holds where no scene
// has more pairs of a triangle (at most 8 of a face) and a 16x16 tile than bin
// positions reach, so that the rule decides nothing on what is refused.
// Statistics count 16x16 tiles.
static Tuning call_tuning(const hana_ctx* c, const std::vector<PassSpec>& specs) {
    Tuning t = c->tuning;
    if (!t.set && !c->stats_enabled) {
        int64_t px = 0, faces = 0;
        for (const PassSpec& s : specs) {
            px += (int64_t)s.target->w * s.target->h;
            faces += s.mesh->F;
        }
        if (px >= 8000 * 256 && px >= 128 * faces && px * faces < (int64_t(1) << 37)) t.tile_shift = 5;
    }
    return t;
}

// Renders a list of passes (per-call path).  Consecutive calls rotate over
// the context's slots, each a stream with its own workspace: the geometry
// stages of a call run while earlier calls rasterise, and its raster waits
// for the previous call to finish, so targets and shadow maps see the calls
// in order.  With timing or statistics on, every call uses slot 0.
int run_passes(hana_ctx* c, std::vector<PassSpec> specs) {
    int r;
    if (c->log.size() >= kMaxLoggedCalls && (r = check_status(c))) return r;
    const std::vector<hana_target*> touched = touched_targets(specs);
    std::vector<hana_target*> sampled;   // sampled as a shadow map, not drawn here
    for (auto& s : specs) {
        if (!s.shadow || !s.shadow->pending_clear) continue;
        bool drawn = false;
        for (auto& o : specs) drawn = drawn || o.target == s.shadow;
        if (!drawn && std::find(sampled.begin(), sampled.end(), s.shadow) == sampled.end()) sampled.push_back(s.shadow);
    }
    Plan pl;
    const Tuning tuning = call_tuning(c, specs);
    size_t faces = 0, tiles = 0;
    for (const PassSpec& s : specs) {
        const int edge = tile_edge(tuning.tile_shift);
        faces += (size_t)s.mesh->F;
        tiles += (size_t)((s.target->w + edge - 1) / edge) * ((s.target->h + edge - 1) / edge);
    }
    if ((r = build_plan(c, std::move(specs), pl, tuning, kFrontFaces, bins_by_counting(c, faces, tiles)))) return r;
    bool rotate = c->pipelined && !c->timing && !c->stats_enabled;
    // Large sequences into one target rotate over two slots: their rasters wait
    // for each other, and with a third in flight the 2.6 M faces of a 1.3 M-
    // triangle frame with its shadow pass ran 3 % slower (141 us, 136 with two).
    // Into three targets in turn they ran 9 % faster with four (125 us, 137).
    int nslots = pl.total_f >= kHugeSequenceFaces ? std::min(2, c->nslots) : c->nslots;
    int a = rotate ? c->next_slot % nslots : 0;
    const int last = pl.specs.back().target->slot;
    const bool stay = rotate && pl.total_f <= kStayFaces && last >= 0 && last < nslots;
    if (stay) a = last;
    else if (rotate && pl.total_f >= kLargeSequenceFaces && last == c->last_slot && last >= 0 && (last ^ 1) < nslots) a = last ^ 1;
    c->last_slot = a;
    hipStream_t S = slot_stream(c, a);
    Arena& A = slot_arena(c, a);
    // the slots' workspaces grow together, so that a sequence of calls
    // allocates (and waits for the streams) once, not once per slot
    if (rotate)
        for (int k = 0; k < nslots; k++)
            if (k != a && (r = bind_plan(c, pl, slot_arena(c, k), 0, 0, false, slot_stream(c, k)))) return r;
    if ((r = bind_plan(c, pl, A, 0, 0, c->stats_enabled, S))) return r;
    pl.ws.status_out = c->status_dev[a];   // the raster leaves the status words in host memory
    // a target sampled as a shadow map by a pass of the same plan must be drawn
    // by an earlier group; clears fuse into the first pass writing the target
    take_clears(pl);
    if ((r = take_counters(c, pl, A, S))) return r;
    if (!pl.args && (r = upload_tables(c, pl, A, S))) return r;
    int n = (int)pl.descs.size();
    if (c->stats_enabled) {
        HIP_TRY(c, launch_fill32(reinterpret_cast<uint32_t*>(A.stats.p), 0u, (size_t)ST_WORDS * 2 * n, S));
    }
    if ((r = enqueue_geometry(c, pl, A, S, true))) return r;
    counters_launched(A);
    // the raster waits for the calls in flight on other slots that touch one
    // of its targets; calls on disjoint targets run concurrently.  After a
    // no-alloc frame (context stream, targets not noted) every slot waits once.
    if (a != 0 && (c->noalloc_wait_mask & (1u << a))) {
        HIP_TRY(c, hipStreamWaitEvent(S, c->slot_done[0], 0));
        c->noalloc_wait_mask &= ~(1u << a);
    }
    for (int k = 0; k < c->nslots; k++)
        if (k != a && (c->pend[k][a].size() > kMaxPendingTargets || must_wait(c, k, a, touched))) {
            HIP_TRY(c, hipStreamWaitEvent(S, c->slot_done[k], 0));
            c->pend[k][a].clear();
        }
    std::vector<Fill> fills;
    for (hana_target* t : sampled) {
        fills.push_back({t, t->clear_rgba, t->clear_depth});
        if ((r = materialize_clear(c, t, S))) return r;
    }
    if ((r = enqueue_raster(c, pl, A, S, true))) return r;
    HIP_TRY(c, hipEventRecord(c->slot_done[a], S));
    if (c->stats_enabled) {
        if (c->stats_passes < n) {
            HIP_TRY(c, hipStreamSynchronize(S));   // the previous call may still copy into it
            if (c->stats_host) HIP_TRY(c, hipHostFree(c->stats_host));
            c->stats_host = nullptr;
            c->stats_passes = 0;
            HIP_TRY(c, hipHostMalloc((void**)&c->stats_host, sizeof(uint64_t) * ST_WORDS * n));
        }
        HIP_TRY(c, hipMemcpyAsync(c->stats_host, A.stats.p, sizeof(uint64_t) * ST_WORDS * n,
                                  hipMemcpyDeviceToHost, S));
        c->stats_passes = n;
    }
    if (c->pipelined) note_pending(c, a, touched);   // else no other slot ever draws
    if (!stay) c->next_slot = (a + 1) % nslots;
    c->status_pending = true;
    c->log.push_back({std::move(pl), std::move(fills)});
    return HANA_OK;
}

bool valid_kind(int k) { return k >= HANA_SHADER_GROUND && k <= HANA_SHADER_SHADOW; }

int tuning_from(hana_ctx* c, const hana_tuning* t, Tuning& out) {
    if (!t || !(t->tile_size == 16 || t->tile_size == 32) || t->raster_wgs_per_cu < 0 || t->raster_wgs_per_cu > 16 ||
        t->parts < 1 || t->parts > (int)kMaxBatchParts || !(t->raster_waves == 0 || t->raster_waves == 2 || t->raster_waves == 4))
        return fail(c, HANA_E_INVALID, "tuning: tile_size 16 or 32, raster_wgs_per_cu 0-16, parts 1-4, raster_waves 0, 2 or 4");
    out.tile_shift = t->tile_size == 32 ? 5 : 4;
    out.raster_wgs_per_cu = t->raster_wgs_per_cu;
    out.raster_waves = t->raster_waves ? t->raster_waves : 4;
    out.parts = t->parts;
    out.auto_waves = t->raster_waves == 0;
    out.auto_parts = false;
    out.set = true;
    return HANA_OK;
}

}  // namespace rt
}  // namespace hana

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

extern "C" {

int hana_gpu_create(int device, hana_ctx** out) { return create_context(device, kDrawSlots, out); }

}  // extern "C"

namespace hana {
namespace rt {

int create_context(int device, int nslots, hana_ctx** out) {
    if (!out || nslots < 1 || nslots > kDrawSlots) return HANA_E_INVALID;
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return HANA_E_DEVICE;
    if (device < 0 || device >= count) return HANA_E_INVALID;
    hana_ctx* c = new hana_ctx();
    c->device = device;
    c->nslots = nslots;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cus > 0)
        c->num_cus = cus;
    auto undo = [c]() {
        if (c->noalloc_status_host) (void)hipHostFree(c->noalloc_status_host);
        for (int i = 0; i < kRing; i++)
            if (c->ring_event[i]) (void)hipEventDestroy(c->ring_event[i]);
        for (int k = 0; k < c->nslots; k++) {
            if (c->slot_done[k]) (void)hipEventDestroy(c->slot_done[k]);
            if (slot_status(c, k)) (void)hipHostFree(slot_status(c, k));
            if (slot_stream(c, k)) (void)hipStreamDestroy(slot_stream(c, k));
        }
        (void)hipGetLastError();
        delete c;
        return HANA_E_DEVICE;
    };
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
        return undo();
    for (int i = 0; i < kRing; i++)
        if (hipEventCreateWithFlags(&c->ring_event[i], hipEventDisableTiming) != hipSuccess) return undo();
    for (int k = 0; k < c->nslots; k++) {
        if (k && hipStreamCreateWithFlags(&c->xstream[k - 1], hipStreamNonBlocking) != hipSuccess) return undo();
        uint32_t*& host = k ? c->xstatus_host[k - 1] : c->status_host;
        if (hipHostMalloc((void**)&host, sizeof(uint32_t) * STATUS_WORDS) != hipSuccess) return undo();
        std::memset(host, 0, sizeof(uint32_t) * STATUS_WORDS);
        if (hipHostGetDevicePointer((void**)&c->status_dev[k], host, 0) != hipSuccess) return undo();
        if (hipEventCreateWithFlags(&c->slot_done[k], hipEventDisableTiming) != hipSuccess) return undo();
    }
    if (hipHostMalloc((void**)&c->noalloc_status_host, sizeof(uint32_t) * STATUS_WORDS) != hipSuccess) return undo();
    std::memset(c->noalloc_status_host, 0, sizeof(uint32_t) * STATUS_WORDS);
    if (hipHostGetDevicePointer((void**)&c->noalloc_status_dev, c->noalloc_status_host, 0) != hipSuccess ||
        noalloc_init(c) != HANA_OK)
        return undo();
    *out = c;
    return HANA_OK;
}

}  // namespace rt
}  // namespace hana

extern "C" {

static void free_arena(Arena& a) {
    DevBuf* bufs[] = {&a.tables, &a.vr, &a.vs, &a.code, &a.pof, &a.bins, &a.chunks, &a.wide, &a.pool_vr,
                      &a.pool_vs, &a.pool_face, &a.clip_queue, &a.status, &a.stats, &a.counters[0], &a.counters[1]};
    for (DevBuf* b : bufs)
        if (b->p) {
            (void)hipFree(b->p);
            b->p = nullptr;
            b->cap = 0;
        }
    a.bin_cap = a.poly_cap = a.clipq_cap = 0;
    a.chunk_slots = 0;
    a.counters_used[0] = a.counters_used[1] = 0;
}

int hana_gpu_destroy(hana_ctx* c) {
    if (!c) return HANA_E_INVALID;
    (void)hipSetDevice(c->device);
    for (int k = 0; k < c->nslots; k++) {
        (void)hipStreamSynchronize(slot_stream(c, k));
        free_arena(slot_arena(c, k));
    }
    if (c->present.p) (void)hipFree(c->present.p);
    if (c->stage_count.p) (void)hipFree(c->stage_count.p);
    if (c->stage_host) (void)hipHostFree(c->stage_host);
    for (hipEvent_t e : c->stage_done)
        if (e) (void)hipEventDestroy(e);
    for (int i = 0; i < kRing; i++) {
        if (c->ring_host[i]) (void)hipHostFree(c->ring_host[i]);
        if (c->ring_event[i]) (void)hipEventDestroy(c->ring_event[i]);
    }
    if (c->stats_host) (void)hipHostFree(c->stats_host);
    if (c->noalloc_status_host) (void)hipHostFree(c->noalloc_status_host);
    for (int k = 0; k < c->nslots; k++) {
        if (slot_status(c, k)) (void)hipHostFree(slot_status(c, k));
        if (c->slot_done[k]) (void)hipEventDestroy(c->slot_done[k]);
    }
    for (auto& p : c->ev_pending) {
        (void)hipEventDestroy(p.second.first);
        (void)hipEventDestroy(p.second.second);
    }
    for (hipEvent_t e : c->ev_pool) (void)hipEventDestroy(e);
    for (int k = 0; k < c->nslots; k++) (void)hipStreamDestroy(slot_stream(c, k));
    delete c;
    return HANA_OK;
}

const char* hana_gpu_last_error(hana_ctx* c) { return c ? c->err.c_str() : "no context"; }

int hana_gpu_sync(hana_ctx* c) {
    if (!c) return HANA_E_INVALID;
    int r = sync_all(c);
    return r ? r : check_status(c);
}

int hana_gpu_set_timing(hana_ctx* c, int enable) {
    if (!c) return HANA_E_INVALID;
    c->timing = enable != 0;
    return sync_all(c);   // stage times never overlap a draw of the second slot
}

int hana_gpu_read_timing(hana_ctx* c, double* ms, int64_t* launches) {
    if (!c || !ms || !launches) return HANA_E_INVALID;
    int r = sync_all(c);
    if (r) return r;
    for (int i = 0; i < HANA_TIMING_STAGES; i++) {
        ms[i] = 0.0;
        launches[i] = 0;
    }
    for (auto& p : c->ev_pending) {
        float t = 0.f;
        HIP_TRY(c, hipEventElapsedTime(&t, p.second.first, p.second.second));
        ms[p.first] += t;
        launches[p.first] += 1;
        c->ev_pool.push_back(p.second.first);
        c->ev_pool.push_back(p.second.second);
    }
    c->ev_pending.clear();
    return HANA_OK;
}

int hana_gpu_replay_count(hana_ctx* c, int64_t* out) {
    if (!c || !out) return HANA_E_INVALID;
    *out = c->replays;
    return HANA_OK;
}

int hana_gpu_set_stats(hana_ctx* c, int enable) {
    if (!c) return HANA_E_INVALID;
    c->stats_enabled = enable != 0;
    return HANA_OK;
}

int hana_gpu_last_stats(hana_ctx* c, hana_pass_stats* out, int max_passes, int* n_passes) {
    if (!c || !out || !n_passes) return HANA_E_INVALID;
    int r = sync_all(c);
    if (r) return r;
    int n = std::min(max_passes, c->stats_host ? c->stats_passes : 0);
    for (int i = 0; i < n; i++) {
        const uint64_t* s = c->stats_host + (size_t)ST_WORDS * i;
        out[i].faces = (int64_t)s[ST_FACES];
        out[i].clipped_faces = (int64_t)s[ST_CLIPPED];
        out[i].polygons = (int64_t)s[ST_POLYS];
        out[i].tile_entries = (int64_t)s[ST_ENTRIES];
        out[i].pixels_written = (int64_t)s[ST_PIXELS];
    }
    *n_passes = n;
    return HANA_OK;
}

int hana_mesh_create(hana_ctx* c, int32_t nverts, const float* pos, const float* nrm, const float* uv,
                     int32_t nfaces, const int32_t* idx, hana_mesh** out) {
    if (!c || !out || nverts < 0 || nfaces < 0 || (nverts && !pos) || (nfaces && !idx))
        return fail(c, HANA_E_INVALID, "hana_mesh_create: bad arguments");
    if (nfaces > (1 << 27)) return fail(c, HANA_E_INVALID, "hana_mesh_create: at most 2^27 faces");
    for (int64_t i = 0; i < 3 * (int64_t)nfaces; i++)
        if (idx[i] < 0 || idx[i] >= nverts) return fail(c, HANA_E_INVALID, "hana_mesh_create: index out of range");
    size_t V = (size_t)nverts;
    std::vector<float> soa(8 * std::max<size_t>(V, 1), 0.0f);
    for (size_t i = 0; i < V; i++) {
        for (int k = 0; k < 3; k++) soa[k * V + i] = pos[3 * i + k];
        if (nrm)
            for (int k = 0; k < 3; k++) soa[(3 + k) * V + i] = nrm[3 * i + k];
        if (uv)
            for (int k = 0; k < 2; k++) soa[(6 + k) * V + i] = uv[2 * i + k];
    }
    hana_mesh* m = new hana_mesh();
    m->V = nverts;
    m->F = nfaces;
    if (hipMalloc((void**)&m->soa, sizeof(float) * soa.size()) != hipSuccess ||
        hipMalloc((void**)&m->idx, sizeof(int32_t) * 3 * std::max<size_t>(nfaces, 1)) != hipSuccess) {
        (void)hipGetLastError();
        if (m->soa) (void)hipFree(m->soa);
        delete m;
        return fail(c, HANA_E_NOMEM, "hana_mesh_create: device allocation failed");
    }
    hipError_t e = hipMemcpy(m->soa, soa.data(), sizeof(float) * soa.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess && nfaces) e = hipMemcpy(m->idx, idx, sizeof(int32_t) * 3 * (size_t)nfaces, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(m->soa);
        (void)hipFree(m->idx);
        delete m;
        return hip_fail(c, e, "hana_mesh_create: upload");
    }
    *out = m;
    return HANA_OK;
}

// Objects a logged call may be rendered again with are freed only after the
// status check (which may replay it); its result is returned.
int hana_mesh_destroy(hana_ctx* c, hana_mesh* m) {
    if (!c || !m) return HANA_E_INVALID;
    int st = check_status(c);
    (void)sync_all(c);
    (void)hipFree(m->soa);
    (void)hipFree(m->idx);
    delete m;
    return st;
}

int hana_texture_create(hana_ctx* c, int32_t w, int32_t h, int32_t bpp, const uint8_t* bytes, hana_texture** out) {
    if (!c || !out || w <= 0 || h <= 0 || !(bpp == 1 || bpp == 3 || bpp == 4) || !bytes)
        return fail(c, HANA_E_INVALID, "hana_texture_create: bad arguments");
    size_t n = (size_t)w * h;
    std::vector<uint32_t> words(n);
    for (size_t i = 0; i < n; i++) {
        uint32_t v = 0;
        for (int k = 0; k < bpp; k++) v |= (uint32_t)bytes[i * bpp + k] << (8 * k);   // TGAColor(p, bpp)
        words[i] = v;
    }
    hana_texture* t = new hana_texture();
    t->w = w;
    t->h = h;
    if (hipMalloc((void**)&t->texels, sizeof(uint32_t) * n) != hipSuccess) {
        (void)hipGetLastError();
        delete t;
        return fail(c, HANA_E_NOMEM, "hana_texture_create: device allocation failed");
    }
    hipError_t e = hipMemcpy(t->texels, words.data(), sizeof(uint32_t) * n, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(t->texels);
        delete t;
        return hip_fail(c, e, "hana_texture_create: upload");
    }
    *out = t;
    return HANA_OK;
}

int hana_texture_destroy(hana_ctx* c, hana_texture* t) {
    if (!c || !t) return HANA_E_INVALID;
    int st = check_status(c);
    (void)sync_all(c);
    (void)hipFree(t->texels);
    delete t;
    return st;
}

int hana_target_create(hana_ctx* c, int32_t w, int32_t h, hana_target** out) {
    // tile coordinates travel as 16-bit fields: at most 2^16 tiles a side
    if (!c || !out || w <= 0 || h <= 0 || w > (1 << 20) || h > (1 << 20) || (int64_t)w * h > (1ll << 30))
        return fail(c, HANA_E_INVALID, "hana_target_create: bad size");
    hana_target* t = new hana_target();
    t->w = w;
    t->h = h;
    size_t n = (size_t)w * h;
    if (hipMalloc((void**)&t->color, 4 * n) != hipSuccess || hipMalloc((void**)&t->depth, 4 * n) != hipSuccess) {
        (void)hipGetLastError();
        if (t->color) (void)hipFree(t->color);
        delete t;
        return fail(c, HANA_E_NOMEM, "hana_target_create: device allocation failed");
    }
    // RenderBuffer constructor state: colour {0,0,0,1} -> (0,0,0,255), depth 1
    // (SR/renderbuffer.cpp:3-18)
    t->pending_clear = true;
    t->clear_rgba = 0xFF000000u;
    t->clear_depth = 1.0f;
    *out = t;
    return HANA_OK;
}

int hana_target_destroy(hana_ctx* c, hana_target* t) {
    if (!c || !t) return HANA_E_INVALID;
    int st = check_status(c);
    (void)sync_all(c);
    (void)hipFree(t->color);
    (void)hipFree(t->depth);
    if (t->winner) (void)hipFree(t->winner);
    delete t;
    return st;
}

int hana_target_clear(hana_ctx* c, hana_target* t, const uint8_t rgba[4], float depth) {
    if (!c || !t || !rgba) return HANA_E_INVALID;
    t->pending_clear = true;
    t->clear_rgba = pack_bytes(rgba);
    t->clear_depth = depth;
    return HANA_OK;
}

int hana_target_upload(hana_ctx* c, hana_target* t, const uint8_t* rgba, const float* depth) {
    if (!c || !t) return HANA_E_INVALID;
    size_t n = (size_t)t->w * t->h;
    // draws before the upload are complete (replayed if need be) before it lands
    int r = check_status(c);
    if (r) return r;
    r = join(c);
    if (r || (r = materialize_clear(c, t, c->stream))) return r;
    if (rgba) HIP_TRY(c, hipMemcpyAsync(t->color, rgba, 4 * n, hipMemcpyHostToDevice, c->stream));
    if (depth) HIP_TRY(c, hipMemcpyAsync(t->depth, depth, 4 * n, hipMemcpyHostToDevice, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return HANA_OK;
}

// Whether every page of the range is in memory already.
static bool resident(const void* p, size_t n) {
    const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE), first = (uintptr_t)p / page,
                    end = ((uintptr_t)p + n + page - 1) / page;
    unsigned char in[1024];
    for (uintptr_t at = first; at < end; at += sizeof in) {
        const size_t k = std::min<size_t>(sizeof in, end - at);
        if (mincore(reinterpret_cast<void*>(at * page), k * page, in) != 0) return false;
        for (size_t i = 0; i < k; i++)
            if (!(in[i] & 1)) return false;
    }
    return true;
}

// The context's pinned staging, grown to hold `total` bytes or the most it
// may; null where a copy to the n bytes at dst does better without: memory the
// GPU reaches itself; pages not touched yet, which a host copy takes one fault
// at a time (0.8 us each) and the runtime's pinning in bulk; or with no pinned
// memory left.
static char* staging_for(hana_ctx* c, const void* dst, size_t n, size_t total) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, dst) != hipSuccess) (void)hipGetLastError();
    else if (a.type != hipMemoryTypeUnregistered) return nullptr;
    if (n > (64u << 10) && !resident(dst, n)) return nullptr;
    size_t want = 4096;
    while (want < total && want < 2 * kStagePiece) want *= 2;
    if (want > c->stage_cap) {
        constexpr size_t flag_bytes = sizeof(uint32_t) * 2 * READ_BANDS;
        if (c->stage_host) (void)hipHostFree(c->stage_host);
        c->stage_host = nullptr;
        c->stage_cap = 0;
        if (hipHostMalloc((void**)&c->stage_host, want + flag_bytes) != hipSuccess ||
            hipHostGetDevicePointer((void**)&c->stage_dev, c->stage_host, 0) != hipSuccess) {
            (void)hipGetLastError();
            if (c->stage_host) (void)hipHostFree(c->stage_host);
            c->stage_host = nullptr;
            return nullptr;
        }
        std::memset(c->stage_host + want, 0, flag_bytes);
        c->stage_cap = want;
    }
    for (hipEvent_t& e : c->stage_done)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            e = nullptr;
            return nullptr;
        }
    return c->stage_host;
}

// A plane of the target for the caller's memory.
struct ReadBack {
    void* dst;
    const void* src;
    bool flip;   // as hana_target_present
};

// Past the staging's size: pieces that alternate between its halves, one copied
// by the host while the next one comes.
static int read_pieces(hana_ctx* c, void* dst, const void* src, size_t n) {
    const size_t pieces = (n + kStagePiece - 1) / kStagePiece;
    for (size_t k = 0; k <= pieces; k++) {
        if (k < pieces) {
            const size_t at = k * kStagePiece;
            HIP_TRY(c, hipMemcpyAsync(c->stage_host + (k & 1) * kStagePiece, static_cast<const char*>(src) + at,
                                      std::min(kStagePiece, n - at), hipMemcpyDeviceToHost, c->stream));
            HIP_TRY(c, hipEventRecord(c->stage_done[k & 1], c->stream));
        }
        if (k) {
            const size_t at = (k - 1) * kStagePiece;
            HIP_TRY(c, hipEventSynchronize(c->stage_done[(k - 1) & 1]));
            std::memcpy(static_cast<char*>(dst) + at, c->stage_host + ((k - 1) & 1) * kStagePiece,
                        std::min(kStagePiece, n - at));
        }
    }
    return HANA_OK;
}

// Whether a sequence since the last check has raised a flag that the host sees.
static bool flags_raised(hana_ctx* c) {
    for (int k = 0; k < c->nslots; k++) {
        const uint32_t* host = slot_status(c, k);
        if (host && *static_cast<const volatile uint32_t*>(host + STATUS_FLAGS)) return true;
    }
    for (const hana_batch* b : c->batches)
        for (size_t p = 0; p < b->parts.size(); p++)
            if (*static_cast<const volatile uint32_t*>(b->status_host + STATUS_WORDS * p + STATUS_FLAGS) & FLAG_NO_RASTER) return true;
    return false;
}

// Waits until the flag says that band is stored; a finished stream says so too.
static int wait_band(hana_ctx* c, const uint32_t* flag) {
    for (uint32_t spin = 1; __atomic_load_n(flag, __ATOMIC_ACQUIRE) != c->stage_epoch; spin++) {
        if (spin % 256 == 0) {
            hipError_t e = hipStreamQuery(c->stream);
            if (e == hipSuccess) break;
            if (e != hipErrorNotReady) return hip_fail(c, e, "reading a target back");
            (void)hipGetLastError();
        }
        __builtin_ia32_pause();
    }
    return HANA_OK;
}

// Copies up to two planes of a target to the caller's memory and completes
// every draw (rendering those again that outgrew the workspace); a draw's error
// is returned after the copy.
//
// To pageable memory the runtime stages or pins by itself, which costs more than
// the transfer.  Here k_read_back stores the planes into pinned staging, enqueued
// behind the draws before they are waited for, and the host copies band after
// band on while the next ones come.  Before and after, us: 640x480 presented 93
// and 65, colour and depth read 155 and 98; 1024x768 195 and 150, 360 and 237;
// 1920x1080 475 and 370, 938 and 580, where the host's copy is the longer part.
static int read_planes(hana_ctx* c, hana_target* t, const ReadBack* b, int count) {
    const size_t n = (size_t)t->w * t->h, total = 4 * n * count;
    char* h = count ? staging_for(c, b[0].dst, 4 * n, total) : nullptr;
    if (h && count == 2 && !staging_for(c, b[1].dst, 4 * n, total)) h = nullptr;
    const bool banded = h && total <= c->stage_cap;
    int r, st = HANA_OK;
    bool checked = false;
    for (;;) {
        // a clear not yet drawn, or a no-alloc frame: first the draws before it
        if (!checked && (!banded || t->pending_clear || c->noalloc_pending)) {
            st = check_status(c);
            if (st == HANA_E_DEVICE) return st;
            checked = true;
        }
        if ((r = join(c)) || (r = materialize_clear(c, t, c->stream))) return r;
        if (!banded) break;
        if ((r = ensure(c, c->stage_count, sizeof(uint32_t) * 2 * READ_BANDS))) return r;
        if (!c->stage_epoch)
            HIP_TRY(c, launch_fill32(c->stage_count.as<uint32_t>(), 0u, 2 * READ_BANDS, c->stream));
        if (!++c->stage_epoch) c->stage_epoch = 1;
        const uint32_t band = std::max((((uint32_t)n + READ_BANDS - 1) / READ_BANDS + 3u) & ~3u, READ_BAND_MIN);
        const int bands = (int)((n + band - 1) / band);
        uint32_t* flags = reinterpret_cast<uint32_t*>(c->stage_host + c->stage_cap);
        uint32_t* flags_dev = reinterpret_cast<uint32_t*>(c->stage_dev + c->stage_cap);
        // 16-byte aligned planes: the staging is a power of two of at least 4096
        // bytes, so that where two planes fit, so do two rounded up
        const size_t pitch = (4 * n + 15) & ~(size_t)15;
        if (pitch * count > c->stage_cap) return fail(c, HANA_E_DEVICE, "internal error: planes larger than their staging");
        for (int i = 0; i < count; i++)
            HIP_TRY(c, launch_read_back(static_cast<const uint32_t*>(b[i].src), reinterpret_cast<uint32_t*>(c->stage_dev + i * pitch),
                                        t->w, t->h, b[i].flip, band, c->stage_count.as<uint32_t>() + i * READ_BANDS,
                                        flags_dev + i * READ_BANDS, c->stage_epoch, c->stream));
        bool again = false;
        for (int i = 0; i < count && !again; i++)
            for (int k = 0; k < bands; k++) {
                if (bands == 1) {
                    if (i == 0) HIP_TRY(c, hipStreamSynchronize(c->stream));
                } else if ((r = wait_band(c, flags + i * READ_BANDS + k))) {
                    return r;
                }
                // the draws have ended: an incomplete one is rendered again first
                if (!checked && i == 0 && k == 0 && flags_raised(c)) {
                    again = true;
                    break;
                }
                const size_t at = (size_t)k * band;
                std::memcpy(static_cast<char*>(b[i].dst) + 4 * at, h + i * pitch + 4 * at, 4 * std::min<size_t>(band, n - at));
            }
        if (again) {
            HIP_TRY(c, hipStreamSynchronize(c->stream));
            st = check_status(c);
            if (st == HANA_E_DEVICE) return st;
            checked = true;
            continue;
        }
        HIP_TRY(c, hipStreamSynchronize(c->stream));
        return checked ? st : check_status(c);
    }
    for (int i = 0; i < count; i++) {
        const void* src = b[i].src;
        if (b[i].flip) {
            if ((r = ensure(c, c->present, 4 * n))) return r;
            HIP_TRY(c, launch_present(t->color, c->present.as<uint32_t>(), t->w, t->h, c->stream));
            src = c->present.p;
        }
        if (h) {
            if ((r = read_pieces(c, b[i].dst, src, 4 * n))) return r;
        } else {
            HIP_TRY(c, hipMemcpyAsync(b[i].dst, src, 4 * n, hipMemcpyDeviceToHost, c->stream));
        }
    }
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return st;
}

int hana_target_read(hana_ctx* c, hana_target* t, uint8_t* rgba, float* depth) {
    if (!c || !t) return HANA_E_INVALID;
    ReadBack b[2];
    int count = 0;
    if (rgba) b[count++] = {rgba, t->color, false};
    if (depth) b[count++] = {depth, t->depth, false};
    return read_planes(c, t, b, count);
}

int hana_target_present(hana_ctx* c, hana_target* t, uint8_t* bgra) {
    if (!c || !t || !bgra) return fail(c, HANA_E_INVALID, "hana_target_present: null argument");
    const ReadBack b{bgra, t->color, true};
    return read_planes(c, t, &b, 1);
}

int hana_target_enable_winner(hana_ctx* c, hana_target* t, int enable) {
    if (!c || !t) return HANA_E_INVALID;
    if (enable && !t->winner) {
        size_t n = (size_t)t->w * t->h;
        if (hipMalloc((void**)&t->winner, 4 * n) != hipSuccess) {
            (void)hipGetLastError();
            return fail(c, HANA_E_NOMEM, "winner map allocation failed");
        }
        HIP_TRY(c, launch_fill32(t->winner, NO_WINNER, n, c->stream));
        HIP_TRY(c, hipStreamSynchronize(c->stream));   // draws of either slot may use it next
    } else if (!enable && t->winner) {
        int st = check_status(c);
        if (st) return st;
        (void)sync_all(c);
        (void)hipFree(t->winner);
        t->winner = nullptr;
    }
    return HANA_OK;
}

int hana_target_read_winner(hana_ctx* c, hana_target* t, uint32_t* winner) {
    if (!c || !t || !winner || !t->winner) return HANA_E_INVALID;
    const size_t n = (size_t)t->w * t->h;
    int st = check_status(c);
    if (st == HANA_E_DEVICE) return st;
    int r = join(c);
    if (r) return r;
    HIP_TRY(c, hipMemcpyAsync(winner, t->winner, 4 * n, hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return st;
}

int hana_draw(hana_ctx* c, const hana_draw_desc* d) {
    if (!c || !d || !d->mesh || !d->target || !d->uniforms || !valid_kind(d->shader))
        return fail(c, HANA_E_INVALID, "hana_draw: bad descriptor");
    if (d->shadow_map == d->target) return fail(c, HANA_E_INVALID, "hana_draw: shadow map is the target");
    PassSpec s{d->mesh, d->shader, *d->uniforms, d->diffuse, d->normal, d->shadow_map, d->target, 0};
    return run_passes(c, {s});
}

int hana_render_frame(hana_ctx* c, const hana_frame_desc* f) {
    if (!c || !f || !f->mesh || !f->target || !f->uniforms || !valid_kind(f->shader) ||
        (f->enable_shadow && (!f->shadow_map || f->shadow_map == f->target)))
        return fail(c, HANA_E_INVALID, "hana_render_frame: bad descriptor");
    hana_uniforms u = *f->uniforms;
    u.enable_shadow = f->enable_shadow;
    std::vector<PassSpec> specs;
    if (f->enable_shadow) specs.push_back({f->mesh, HANA_SHADER_SHADOW, u, f->diffuse, f->normal, nullptr, f->shadow_map, 0});
    specs.push_back({f->mesh, f->shader, u, f->diffuse, f->normal, f->enable_shadow ? f->shadow_map : nullptr, f->target,
                     f->enable_shadow ? 1 : 0});
    int r = run_passes(c, std::move(specs));
    if (r) return r;
    if (f->enable_shadow) {
        // shdaow_map->renderbuffer_clear_color(Black) / clear_depth(FLT_MAX)
        // after the main pass (SR/scene.h:94-98); alpha is written as 255
        f->shadow_map->pending_clear = true;
        f->shadow_map->clear_rgba = 0xFF000000u;
        f->shadow_map->clear_depth = 3.40282347e+38f;
    }
    return HANA_OK;
}

// ---- batches ----

int hana_batch_create(hana_ctx* c, hana_batch** out) {
    if (!c || !out) return HANA_E_INVALID;
    *out = new hana_batch();
    return HANA_OK;
}

int hana_batch_add_frame(hana_ctx* c, hana_batch* b, const hana_frame_desc* f) {
    if (!c || !b || !f || !f->mesh || !f->target || !f->uniforms || !valid_kind(f->shader) ||
        (f->enable_shadow && (!f->shadow_map || f->shadow_map == f->target)))
        return fail(c, HANA_E_INVALID, "hana_batch_add_frame: bad descriptor");
    if (b->finalized) return fail(c, HANA_E_INVALID, "hana_batch_add_frame: batch already finalized");
    hana_uniforms u = *f->uniforms;
    u.enable_shadow = f->enable_shadow;
    b->frame_first.push_back(b->specs.size());
    if (f->enable_shadow) b->specs.push_back({f->mesh, HANA_SHADER_SHADOW, u, f->diffuse, f->normal, nullptr, f->shadow_map, 0});
    b->specs.push_back({f->mesh, f->shader, u, f->diffuse, f->normal, f->enable_shadow ? f->shadow_map : nullptr,
                        f->target, 1});
    return HANA_OK;
}

// Every frame of a batch clears its target and shadow map first (the state
// DrawModel::draw runs in after main.cpp's per-frame clear).
static void batch_clear_flags(hana_batch_part& part) {
    for (size_t i = 0; i < part.plan.descs.size(); i++) {
        PassDesc& d = part.plan.descs[i];
        d.clear = 1;
        d.clear_rgba = 0xFF000000u;
        d.clear_depth = 3.40282347e+38f;
    }
}

// The sequence itself clears every target it draws, so a clear still pending
// from target creation or hana_target_clear is void: left pending, it would
// wipe the rendered image at the next read.
static void batch_drop_pending(hana_batch* b) {
    for (auto& s : b->specs) s.target->pending_clear = false;
}

// Each frame's first work estimate: faces plus an eighth of the pixels drawn,
// over its passes.
static std::vector<double> frame_weights(const hana_batch* b) {
    size_t nf = b->frame_first.size();
    std::vector<double> w(nf, 0.0);
    for (size_t k = 0; k < nf; k++) {
        size_t e = k + 1 < nf ? b->frame_first[k + 1] : b->specs.size();
        for (size_t i = b->frame_first[k]; i < e; i++)
            w[k] += (double)b->specs[i].mesh->F + (double)b->specs[i].target->w * b->specs[i].target->h / 8.0;
    }
    return w;
}

// The end frame of each part when the frames, in order, are split into up to
// b->tuning.parts parts of about equal estimated work w (one value per frame),
// at most one part per frame.  Not more than four: six or eight were slower on
// 256 mixed scenes, since a process gets four hardware queues, and more streams
// than that share them.
static std::vector<size_t> split_ends(const hana_batch* b, const std::vector<double>& w) {
    size_t nf = b->frame_first.size();
    size_t np = std::min(nf, std::min((size_t)b->tuning.parts, kMaxBatchParts));
    double total = 0.0;
    for (double x : w) total += x;
    // part p ends at the first frame where the running work reaches (p+1)/np
    // of the total, leaving at least one frame for each later part
    std::vector<size_t> ends(np);
    size_t k = 0;
    double run = 0.0;
    for (size_t p = 0; p < np; p++) {
        if (p + 1 == np) {
            k = nf;
        } else {
            do {
                run += w[k++];
            } while (k < nf - (np - 1 - p) && run < total * (double)(p + 1) / (double)np);
        }
        ends[p] = k;
    }
    return ends;
}

// Replaces the batch's parts by those ending at `ends` (unsized: no plan yet).
static void batch_split(hana_batch* b, const std::vector<size_t>& ends) {
    size_t nf = b->frame_first.size();
    b->parts.clear();
    b->parts.resize(ends.size());
    size_t k0 = 0;
    for (size_t p = 0; p < ends.size(); p++) {
        size_t k = ends[p];
        size_t s0 = b->frame_first[k0], s1 = k < nf ? b->frame_first[k] : b->specs.size();
        b->parts[p].specs.assign(b->specs.begin() + s0, b->specs.begin() + s1);
        b->parts[p].arena = &b->arenas[p];
        b->parts[p].f0 = k0;
        b->parts[p].f1 = k;
        k0 = k;
    }
}

// Part p of a batch runs on the stream of draw slot p (part 0 on the
// context stream), and parts beyond the slots on the batch's own streams, so
// that a context and its batches use as few streams as possible.
static hipStream_t part_stream(hana_ctx* c, hana_batch* b, size_t p) {
    return p < (size_t)c->nslots ? slot_stream(c, (int)p) : b->extra[p - c->nslots];
}

// Enqueues every part on its stream, forked from and joined back into the
// context stream (with stage timing on, all run on the context stream so
// that stage times do not overlap).
static int batch_enqueue(hana_ctx* c, hana_batch* b, bool timed) {
    int r;
    if (b->parts.size() == 1 || (timed && c->timing)) {
        for (auto& part : b->parts)
            if ((r = enqueue_sequence(c, part.plan, *part.arena, c->stream, timed))) return r;
        return HANA_OK;
    }
    HIP_TRY(c, hipEventRecord(b->fork, c->stream));
    for (size_t p = 1; p < b->parts.size(); p++) {
        HIP_TRY(c, hipStreamWaitEvent(part_stream(c, b, p), b->fork, 0));
    }
    for (size_t p = 0; p < b->parts.size(); p++) {
        hipStream_t s = part_stream(c, b, p);
        if ((r = enqueue_sequence(c, b->parts[p].plan, *b->parts[p].arena, s, timed))) return r;
    }
    for (size_t p = 1; p < b->parts.size(); p++) {
        hipStream_t s = part_stream(c, b, p);
        HIP_TRY(c, hipEventRecord(b->joined[p - 1], s));
        HIP_TRY(c, hipStreamWaitEvent(c->stream, b->joined[p - 1], 0));
    }
    return HANA_OK;
}

// Clears the parts' status words, once the batch's runs have ended; returns their
// flags, and in `parts` the parts with one of a capacity.
static uint32_t batch_take_flags(hana_ctx* c, hana_batch* b, uint32_t* parts) {
    uint32_t all = 0;
    for (size_t p = 0; p < b->parts.size(); p++) {
        uint32_t* const host = b->status_host + STATUS_WORDS * p;
        const uint32_t f = host[STATUS_FLAGS];
        if (!f) continue;
        all |= f;
        if (f & FLAG_CAPACITY) *parts |= 1u << p;
        (void)launch_fill32(b->arenas[p].status.as<uint32_t>(), 0u, STATUS_WORDS, c->stream);
        std::memset(host, 0, sizeof(uint32_t) * STATUS_WORDS);
    }
    return all;
}

// Whether the workspace of a chunked part that was just run holds what another
// run may need.  Which of the wide triangles a full list leaves out, which pairs
// a full table leaves out and which fans are clipped together follow the order
// in which workgroups and lanes arrive.  For the first there is a bound: every
// listed triangle of a pass one more descriptor in a tile, and all their pairs.
// For the others an eighth is added.  Grows what is too small (then true, and the
// part is run again) or leaves the part to counted binning.
static int batch_leave_room(hana_ctx* c, hana_batch_part& part, uint32_t* min_bins, bool* grown, bool* counted) {
    const Plan& pl = part.plan;
    Arena& A = *part.arena;
    std::vector<uint32_t> n(counter_words(pl));
    HIP_TRY(c, hipMemcpy(n.data(), pl.ws.seq, sizeof(uint32_t) * n.size(), hipMemcpyDeviceToHost));
    auto pairs = [&](int w) { return (uint64_t)n[w] | (uint64_t)n[w + 1] << 32; };
    const uint32_t *wide = n.data() + SEQ_WORDS, *chunks = n.data() + (pl.ws.tile_chunks - pl.ws.seq);
    const bool left_out = *std::max_element(wide, wide + std::max<size_t>(pl.descs.size(), 1)) > pl.ws.wide_cap;
    const uint64_t fullest = pl.total_tiles ? *std::max_element(chunks, chunks + pl.total_tiles) : 0;
    const uint64_t places = fullest + fullest / 8 + CHUNK_SLACK + (left_out ? pl.ws.wide_cap : 0);
    uint64_t shared = pairs(SEQ_PAIRS) + (left_out ? pairs(SEQ_WIDE_PAIRS) : 0);
    shared += shared / 8 + 4096;
    if (places > pl.ws.chunk_cap) {
        const uint64_t slots = (places + places / 8 + 8) * (uint64_t)std::max(pl.total_tiles, 1);
        if (slots > kGrownChunks) {
            *counted = true;
            return HANA_OK;
        }
        const int r = ensure_chunks(c, A, slots);
        if (r && r != HANA_E_NOMEM) return r;
        *(r ? counted : grown) = true;
        if (r) return HANA_OK;
    }
    if (pl.ws.seg_region + shared > pl.ws.bin_cap) {
        if (pl.ws.seg_region + shared > MAX_PAIRS) *counted = true;
        else *min_bins = (uint32_t)(pl.ws.seg_region + shared);
        *grown = true;
    }
    return HANA_OK;
}

// Sizes a part's workspace with trial runs.
static int batch_size_part(hana_ctx* c, hana_batch* b, hana_batch_part& part) {
    int r;
    uint32_t min_bins = 0, min_polys = 0;
    bool counted = part.counted, roomy = false;
    Arena& A = *part.arena;
    const size_t p = (size_t)(&part - b->parts.data());
    for (int attempt = 0; attempt < 8; attempt++) {
        if ((attempt == 0 || counted != part.plan.counted) &&
            (r = build_plan(c, part.specs, part.plan, b->tuning, kBatchFrontFaces, counted)))
            return r;
        if ((r = bind_plan(c, part.plan, A, min_bins, min_polys, false, c->stream))) return r;
        part.plan.ws.status_out = b->status_dev + STATUS_WORDS * p;
        batch_clear_flags(part);
        HIP_TRY(c, hipMemcpy(A.tables.p, part.plan.descs.data(), sizeof(PassDesc) * part.plan.descs.size(),
                             hipMemcpyHostToDevice));
        HIP_TRY(c, hipMemcpy(A.tables.as<char>() + part.plan.uni_off, part.plan.unis.data(),
                             sizeof(DevUniforms) * part.plan.unis.size(), hipMemcpyHostToDevice));
        if (!part.plan.tile_pass.empty())
            HIP_TRY(c, hipMemcpy(A.tables.as<char>() + part.plan.tp_off, part.plan.tile_pass.data(),
                                 sizeof(uint2) * part.plan.tile_pass.size(), hipMemcpyHostToDevice));
        // trial run: what it needs, exactly or (chunks) as near as another's
        if ((r = enqueue_sequence(c, part.plan, A, c->stream))) return r;
        uint32_t st[STATUS_WORDS];
        HIP_TRY(c, hipMemcpyAsync(st, A.status.p, sizeof st, hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(c, hipStreamSynchronize(c->stream));
        std::memset(b->status_host + STATUS_WORDS * p, 0, sizeof st);
        if (!(st[STATUS_FLAGS] & ~(uint32_t)FLAG_POLY_TOO_LARGE) && !counted && !roomy) {
            roomy = true;   // once: it then has room for what this run needed and more
            bool grown = false;
            if ((r = batch_leave_room(c, part, &min_bins, &grown, &counted))) return r;
            if (grown || counted) {
                HIP_TRY(c, launch_fill32(A.status.as<uint32_t>(), 0u, STATUS_WORDS, c->stream));
                continue;
            }
        }
        if (!st[STATUS_FLAGS]) return HANA_OK;
        HIP_TRY(c, launch_fill32(A.status.as<uint32_t>(), 0u, STATUS_WORDS, c->stream));
        if (st[STATUS_FLAGS] & FLAG_QUEUE_STALL)
            return fail(c, HANA_E_DEVICE, "hana_batch_finalize: the persistent raster's wait timed out");
        if (!(st[STATUS_FLAGS] & FLAG_CAPACITY)) {
            if (st[STATUS_FLAGS] & FLAG_PAIR_LIMIT)
                return fail(c, HANA_E_NOMEM, "hana_batch_finalize: a part covers more than 4,294,967,280 "
                                             "(triangle, tile) pairs; split the batch");
            return HANA_OK;   // a polygon over POLY_MAX vertices is dropped at every run, like a per-call draw
        }
        const uint64_t need_bins = (uint64_t)st[STATUS_NEED_BINS] + st[STATUS_NEED_BINS] / 8 + 1024;
        min_bins = std::max(min_bins, (uint32_t)std::min<uint64_t>(need_bins, MAX_PAIRS));
        min_polys = st[STATUS_NEED_POLYS] + st[STATUS_NEED_POLYS] / 8 + 1024;
        Needs need;
        need.take(st);
        // as in check_status: by counting where the descriptors do not grow that
        // far or have no memory to, or when growing them was not enough
        if (!counted && (attempt >= 2 || (st[STATUS_FLAGS] & FLAG_CHUNK_OVERFLOW))) {
            r = attempt < 2 && chunks_grow(need) ? grow_chunks(c, A, need) : HANA_E_NOMEM;
            if (r && r != HANA_E_NOMEM) return r;
            if (r) {
                counted = true;
                min_bins = 0;   // its own run will tell
            }
        }
    }
    return fail(c, HANA_E_OVERFLOW, "hana_batch_finalize: capacity not reached");
}

// All of them, whose trial runs draw what was to be cleared.
static int batch_size_parts(hana_ctx* c, hana_batch* b) {
    int r = HANA_OK;
    for (auto& part : b->parts)
        if ((r = batch_size_part(c, b, part))) break;
    batch_drop_pending(b);
    return r;
}

static void batch_drop_graph(hana_batch* b) {
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
}

// Captures the sized parts (with use_graph).
static int batch_capture(hana_ctx* c, hana_batch* b) {
    batch_drop_graph(b);
    if (b->use_graph) {
        HIP_TRY(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
        int er = batch_enqueue(c, b, false);
        hipGraph_t g = nullptr;
        hipError_t ec = hipStreamEndCapture(c->stream, &g);
        if (er) {
            if (g) (void)hipGraphDestroy(g);
            return er;
        }
        if (ec != hipSuccess) return hip_fail(c, ec, "hipStreamEndCapture");
        b->graph = g;
        HIP_TRY(c, hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
    }
    return HANA_OK;
}

// Sizes the given parts again, by counting.
static int batch_recount(hana_ctx* c, hana_batch* b, uint32_t parts) {
    int r;
    for (size_t p = 0; p < b->parts.size(); p++) {
        if (!(parts >> p & 1u)) continue;
        b->parts[p].counted = true;
        if ((r = batch_size_part(c, b, b->parts[p]))) return r;
    }
    return batch_capture(c, b);
}

// Splits, sizes and (with use_graph) captures the batch for b->tuning.
static int batch_prepare_parts(hana_ctx* c, hana_batch* b, bool use_graph) {
    int r;
    batch_drop_graph(b);
    std::vector<double> w = frame_weights(b);
    batch_split(b, split_ends(b, w));
    if ((r = batch_size_parts(c, b))) return r;
    if (b->parts.size() > 1) {
        // One rebalancing step.  The parts run concurrently and the batch ends
        // with its slowest one; with the first estimates the parts of 256
        // mixed scenes ended up to 0.27 ms apart.  Each part is timed alone
        // (a run to warm up, then a timed one: the sequence clears what it
        // draws, so the runs leave nothing behind), its frames' estimates are
        // scaled by its measured time per unit of estimate, and the frames
        // are split again (unless a part measured no time); if any part's frames
        // changed, every part is sized again.
        std::vector<double> cost(w.size(), 0.0);
        hipEvent_t e0 = nullptr, e1 = nullptr;
        HIP_TRY(c, hipEventCreate(&e0));
        if (hipEventCreate(&e1) != hipSuccess) {
            (void)hipEventDestroy(e0);
            return fail(c, HANA_E_DEVICE, "hipEventCreate");
        }
        r = HANA_OK;
        bool measured = true;   // every part took a positive time
        for (auto& part : b->parts) {
            float ms = 0.0f;
            for (int rep = 0; rep < 2 && !r; rep++) {
                if (hipEventRecord(e0, c->stream) != hipSuccess) r = fail(c, HANA_E_DEVICE, "hipEventRecord");
                if (!r) r = enqueue_sequence(c, part.plan, *part.arena, c->stream, false);
                if (!r && hipEventRecord(e1, c->stream) != hipSuccess) r = fail(c, HANA_E_DEVICE, "hipEventRecord");
                if (!r && hipEventSynchronize(e1) != hipSuccess) r = fail(c, HANA_E_DEVICE, "hipEventSynchronize");
                if (!r && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) r = fail(c, HANA_E_DEVICE, "hipEventElapsedTime");
            }
            double W = 0.0;
            for (size_t k = part.f0; k < part.f1; k++) W += w[k];
            measured = measured && ms > 0.0f && W > 0.0;
            for (size_t k = part.f0; k < part.f1; k++) cost[k] = W > 0.0 ? w[k] * (double)ms / W : w[k];
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        batch_drop_pending(b);
        if (r) return r;
        std::vector<size_t> ends = split_ends(b, cost), before;
        for (auto& part : b->parts) before.push_back(part.f1);
        if (measured && ends != before) {
            batch_split(b, ends);
            if ((r = batch_size_parts(c, b))) return r;
        }
    }
    if (b->parts.size() > 1 && !b->fork) HIP_TRY(c, hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
    while (b->joined.size() + 1 < b->parts.size()) {
        hipEvent_t e = nullptr;
        HIP_TRY(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
        b->joined.push_back(e);
    }
    while (b->extra.size() + c->nslots < b->parts.size()) {
        hipStream_t s = nullptr;
        HIP_TRY(c, hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        b->extra.push_back(s);
    }
    b->use_graph = use_graph;
    return batch_capture(c, b);
}

// The parts of a batch until the caller sets them, by its 16x16 tiles.  Each part
// adds its launches to the graph, and with few tiles those are what a batch
// takes; with many, more parts fill each other's tails.  1, 2 and 4 parts, us a
// batch: 1,276 tiles 64, 75 and 98; 11,396 tiles 98, 108 and 113, of larger
// meshes 113, 113 and 119; 16,973 tiles 143, 145 and 164; 22,464 tiles 166, 168
// and 163; 23,208 tiles 215, 188 and 191; 33,414 tiles 221, 210 and 218; 93,766
// tiles 430, 399 and 414; 390,000 tiles 1,282, 1,221 and 1,192.
static int parts_for(const hana_batch* b) {
    int64_t tiles = 0;
    for (const PassSpec& s : b->specs) tiles += (int64_t)((s.target->w + 15) / 16) * ((s.target->h + 15) / 16);
    return tiles <= 17000 ? 1 : (tiles <= 200000 ? 2 : 4);
}

static int batch_prepare(hana_ctx* c, hana_batch* b, bool use_graph) {
    if (!b->status_host) {
        const size_t bytes = sizeof(uint32_t) * STATUS_WORDS * kMaxBatchParts;
        if (hipHostMalloc((void**)&b->status_host, bytes) != hipSuccess ||
            hipHostGetDevicePointer((void**)&b->status_dev, b->status_host, 0) != hipSuccess) {
            (void)hipGetLastError();
            if (b->status_host) (void)hipHostFree(b->status_host);
            b->status_host = nullptr;
            return fail(c, HANA_E_NOMEM, "batch status words: pinned allocation failed");
        }
        std::memset(b->status_host, 0, bytes);
    }
    if (b->tuning.auto_parts) b->tuning.parts = parts_for(b);
    int r = batch_prepare_parts(c, b, use_graph);
    if (r == HANA_E_NOMEM && b->tuning.auto_parts && b->tuning.parts < 4) {
        // more pairs than a part of this size may hold, or a workspace too large
        b->tuning.parts = 4;
        r = batch_prepare_parts(c, b, use_graph);
    }
    return r;
}

static int batch_check_new(hana_ctx* c, hana_batch* b, const char* what) {
    if (b->specs.empty()) return fail(c, HANA_E_INVALID, std::string(what) + ": empty batch");
    if (b->finalized) return fail(c, HANA_E_INVALID, std::string(what) + ": batch already finalized");
    for (size_t i = 0; i < b->specs.size(); i++)
        for (size_t j = i + 1; j < b->specs.size(); j++)
            if (b->specs[i].target == b->specs[j].target)
                return fail(c, HANA_E_INVALID, std::string(what) + ": frames of a batch need distinct targets and shadow maps");
    return HANA_OK;
}

int hana_batch_finalize(hana_ctx* c, hana_batch* b, int use_graph) {
    if (!c || !b) return HANA_E_INVALID;
    int r;
    if ((r = batch_check_new(c, b, "hana_batch_finalize"))) return r;
    if ((r = check_status(c)) || (r = join(c))) return r;
    if ((r = batch_prepare(c, b, use_graph != 0))) return r;
    b->finalized = true;
    return HANA_OK;
}

// One run of a prepared batch on the context stream.
static int batch_launch(hana_ctx* c, hana_batch* b) {
    int r = join(c);
    if (r) return r;
    c->next_slot = 0;   // the next draw follows the sequence on the context stream
    if (b->use_graph) HIP_TRY(c, hipGraphLaunch(b->exec, c->stream));
    else if ((r = batch_enqueue(c, b, true))) return r;
    // every part has joined the context stream: draws on other slots that
    // touch the batch's targets wait for it
    HIP_TRY(c, hipEventRecord(c->slot_done[0], c->stream));
    std::vector<hana_target*> t;
    for (const PassSpec& s : b->specs)
        for (hana_target* x : {s.target, s.shadow})
            if (x) t.push_back(x);
    note_pending(c, 0, t);
    return HANA_OK;
}

// Mean time of `reps` runs after one untimed run, with events on the context
// stream (every part joins it).
static int batch_time(hana_ctx* c, hana_batch* b, int reps, double* ms) {
    int r;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    HIP_TRY(c, hipEventCreate(&e0));
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return fail(c, HANA_E_DEVICE, "hipEventCreate");
    }
    float t = 0.f;
    batch_drop_pending(b);
    r = batch_launch(c, b);
    if (!r) r = sync_all(c);
    if (!r && hipEventRecord(e0, c->stream) != hipSuccess) r = fail(c, HANA_E_DEVICE, "hipEventRecord");
    for (int i = 0; i < reps && !r; i++) r = batch_launch(c, b);
    if (!r && hipEventRecord(e1, c->stream) != hipSuccess) r = fail(c, HANA_E_DEVICE, "hipEventRecord");
    if (!r) r = sync_all(c);
    if (!r && hipEventElapsedTime(&t, e0, e1) != hipSuccess) r = fail(c, HANA_E_DEVICE, "hipEventElapsedTime");
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = (double)t / std::max(reps, 1);
    return r;
}


static void tuning_out(const Tuning& t, double ms, hana_tuning* out) {
    std::memset(out, 0, sizeof *out);
    out->tile_size = tile_edge(t.tile_shift);
    out->raster_wgs_per_cu = t.raster_wgs_per_cu;
    out->parts = t.parts;
    out->raster_waves = t.auto_waves ? 0 : t.raster_waves;
    out->ms = ms;
}

// A prepared batch's tuning as a caller can set it: the waves that were chosen
// where its rasters all have the same, else 0, which chooses them again.
static Tuning batch_tuning(const hana_batch* b) {
    Tuning t = b->tuning;
    int waves = 0;
    bool same = true;
    for (const hana_batch_part& part : b->parts)
        for (int g = 0; g < 2; g++) {
            if (part.plan.raster_wgs == 0 && !part.plan.group_count[g]) continue;
            const int w = part.plan.raster_waves[part.plan.raster_wgs > 0 ? 0 : g];
            same = same && (!waves || w == waves);
            waves = w;
        }
    if (t.auto_waves && waves && same) {
        t.raster_waves = waves;
        t.auto_waves = false;
    }
    return t;
}

int hana_gpu_set_tuning(hana_ctx* c, const hana_tuning* t) {
    if (!c) return HANA_E_INVALID;
    Tuning tu;
    int r = tuning_from(c, t, tu);
    if (r) return r;
    c->tuning = tu;
    return HANA_OK;
}

int hana_batch_set_tuning(hana_ctx* c, hana_batch* b, const hana_tuning* t) {
    if (!c || !b) return HANA_E_INVALID;
    if (b->finalized) return fail(c, HANA_E_INVALID, "hana_batch_set_tuning: batch already finalized");
    return tuning_from(c, t, b->tuning);
}

int hana_batch_get_tuning(hana_ctx* c, const hana_batch* b, hana_tuning* out) {
    if (!c || !b || !out) return HANA_E_INVALID;
    tuning_out(batch_tuning(b), b->tuned_ms, out);
    return HANA_OK;
}

// The candidates, one dimension at a time from the batch's current tuning:
// the tile size, then the raster form (per-tile workgroups or a persistent
// grid of 2, 4 or 8 workgroups per CU), then the waves per raster workgroup,
// then the number of parts; each keeps the best value found so far for the
// others.  A candidate replaces the best only if it is faster by more than
// kAutotuneMargin, so that run-to-run noise between near-equal tunings does
// not change the choice.
static constexpr double kAutotuneMargin = 0.02;

int hana_batch_autotune(hana_ctx* c, hana_batch* b, int use_graph, int reps, hana_tuning* chosen) {
    if (!c || !b || reps < 1) return HANA_E_INVALID;
    int r;
    if ((r = batch_check_new(c, b, "hana_batch_autotune"))) return r;
    if ((r = check_status(c)) || (r = join(c))) return r;
    Tuning best = b->tuning;
    double best_ms = 0.0;
    auto measure = [&](const Tuning& t, double* ms) {
        for (int tries = 0; tries < 3; tries++) {
            b->tuning = t;
            int e = batch_prepare(c, b, use_graph != 0);
            if (e || (e = batch_time(c, b, reps, ms))) return e;
            uint32_t parts = 0;
            if (!(batch_take_flags(c, b, &parts) & FLAG_NO_RASTER)) return (int)HANA_OK;
            *ms = 1e30;   // frames were left out: no time of theirs
        }
        return (int)HANA_OK;
    };
    if ((r = measure(best, &best_ms))) return r;
    best.parts = b->tuning.parts;
    const int shifts[] = {4, 5}, wgs[] = {0, 2, 4, 8}, waves[] = {4, 2}, parts[] = {1, 2, 4};
    const int* dims[4] = {shifts, wgs, waves, parts};
    const int counts[4] = {2, 4, 2, 3};
    for (int dim = 0; dim < 4; dim++) {
        const int* vals = dims[dim];
        int nv = counts[dim];
        Tuning base = best;
        for (int i = 0; i < nv; i++) {
            Tuning t = base;
            int* fields[4] = {&t.tile_shift, &t.raster_wgs_per_cu, &t.raster_waves, &t.parts};
            const int curs[4] = {base.tile_shift, base.raster_wgs_per_cu, base.raster_waves, base.parts};
            int& field = *fields[dim];
            const int cur = curs[dim];
            const bool waves_dim = dim == 2;
            if (vals[i] == cur && !(waves_dim && base.auto_waves)) continue;
            field = vals[i];
            if (waves_dim) t.auto_waves = false;
            if (dim == 3) t.auto_parts = false;
            double ms = 0.0;
            if ((r = measure(t, &ms))) return r;
            if (ms < best_ms * (1.0 - kAutotuneMargin)) {
                best = t;
                best_ms = ms;
            }
        }
    }
    b->tuning = best;
    if ((r = batch_prepare(c, b, use_graph != 0))) return r;
    b->tuned_ms = best_ms;
    b->finalized = true;
    if (chosen) tuning_out(batch_tuning(b), best_ms, chosen);
    return HANA_OK;
}

int hana_batch_run(hana_ctx* c, hana_batch* b) {
    if (!c || !b || !b->finalized) return fail(c, HANA_E_INVALID, "hana_batch_run: batch not finalized");
    // per-call draws before the batch are complete (replayed if need be)
    // before the batch draws over their targets
    int r;
    if ((c->status_pending || c->noalloc_pending) && (r = check_status(c))) return r;
    batch_drop_pending(b);
    auto& runs = c->batches;
    runs.erase(std::remove(runs.begin(), runs.end(), b), runs.end());
    runs.push_back(b);
    return batch_launch(c, b);
}

int hana_batch_destroy(hana_ctx* c, hana_batch* b) {
    if (!c || !b) return HANA_E_INVALID;
    // a run that outgrew the workspace is run again while it can be
    const bool ran = std::find(c->batches.begin(), c->batches.end(), b) != c->batches.end();
    const int st = ran ? check_status(c) : HANA_OK;
    (void)sync_all(c);
    batch_drop_graph(b);
    if (b->status_host) (void)hipHostFree(b->status_host);
    for (auto& a : b->arenas) free_arena(a);
    if (b->fork) (void)hipEventDestroy(b->fork);
    for (hipEvent_t e : b->joined) (void)hipEventDestroy(e);
    for (hipStream_t s : b->extra) (void)hipStreamDestroy(s);
    delete b;
    return st;
}

}  // extern "C"
