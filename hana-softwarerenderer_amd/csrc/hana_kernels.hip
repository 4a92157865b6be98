// hana_kernels.hip -- the gfx950 rasterisation pipeline.
//
// One launch sequence renders any number of passes (a pass is one
// graphics_draw_triangle call, SR/graphics.cpp:378-407):
//
//   k_vertex   VPT vertices per lane: vertex program, clip-space outcode
//              (is_vertex_visible and the 7 plane tests), perspective divide
//              and 1/w                                (SR/IShader.cpp, SR/graphics.cpp:29-49, 132-134, 316-337)
//   k_setup    FPT faces per lane: back-face cull, viewport, bbox, degenerate
//              test of trivially accepted faces; bins them; drops faces that
//              the first plane they cross removes whole; queues the rest for
//              clipping
//   k_clip     clips the queued faces (SR/graphics.cpp:136-161) into polygons
//              and bins their fan triangles
//   k_front    the three of them in one launch, for smaller sequences
//   k_raster   one workgroup per 16x16 tile: exact per-pixel coverage and
//              depth (SR/graphics.cpp:222-233, 349-359) resolved in LDS with
//              64-bit (depth, submission order) keys, then one fragment
//              program per covered pixel (SR/graphics.cpp:362-373)
//
// Depth test semantics.  The reference tests `z > stored` per fragment in
// submission order (LEQUAL, later primitive wins ties) and no shader
// discards, so the final pixel is the last fragment in submission order among
// those at the minimum depth.  Each fragment here forms the key
// (order-preserving bits of z, 0xFFFFFFFE - order) and the tile keeps the
// per-pixel minimum with ds_min_u64: the minimum is that same fragment
// whatever order the lanes run in.  NaN depths (which pass any test and make
// the next fragment pass) are resolved exactly by a second sweep.
#include <float.h>
#include <hip/hip_runtime.h>

#include "hana_device.h"
#include "hana_launch.h"

namespace hana {

// ---------------------------------------------------------------------------
// shared helpers
// ---------------------------------------------------------------------------

template <int WHICH>
__device__ __forceinline__ int block0_of(const PassDesc& p) {
    return WHICH == 0 ? p.vblock0 : (WHICH == 1 ? p.fblock0 : p.tblock0);
}
// largest pass index whose first block is <= block (passes sorted by it)
template <int WHICH>
__device__ __forceinline__ int find_pass(const PassDesc* P, int n, int block) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (block0_of<WHICH>(P[mid]) <= block) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}


// Triangle set-up in screen space (SR/graphics.cpp:316-347, SR/maths.cpp:20-25).
struct TriS {
    float ax, ay;        // screen A
    float s0x, s0y;      // C.x - A.x, B.x - A.x
    float s1x, s1y;      // C.y - A.y, B.y - A.y
    float uz;            // cross product z (constant over the triangle)
    float z0, z1, z2;    // screen depths
    int x0, x1, y0, y1;  // pixel loop bounds (inclusive)
    bool fast;           // cover_is_fast
};

// The screen corners, edges and depths of a triangle (SR/graphics.cpp:316-337).
struct Screen {
    float x0, y0, x1, y1, x2, y2;
};
__device__ __forceinline__ Screen tri_edges(float4 a, float4 b, float4 c, int W, int H, TriS& t) {
    float fw = (float)W, fh = (float)H;
    Screen s;
    s.x0 = (a.x + 1) * 0.5f * fw; s.y0 = (a.y + 1) * 0.5f * fh;
    s.x1 = (b.x + 1) * 0.5f * fw; s.y1 = (b.y + 1) * 0.5f * fh;
    s.x2 = (c.x + 1) * 0.5f * fw; s.y2 = (c.y + 1) * 0.5f * fh;
    t.z0 = (a.z + 1) * 0.5f;
    t.z1 = (b.z + 1) * 0.5f;
    t.z2 = (c.z + 1) * 0.5f;
    t.ax = s.x0;
    t.ay = s.y0;
    t.s0x = s.x2 - s.x0;
    t.s0y = s.x1 - s.x0;
    t.s1x = s.y2 - s.y0;
    t.s1y = s.y1 - s.y0;
    t.uz = t.s0x * t.s1y - t.s0y * t.s1x;
    return s;
}

// The reference's pixel loop bounds (SR/graphics.cpp:338-347) of a triangle
// whose u.z is not NaN, so that no corner is: its running minima and maxima,
// clamped at every step, are then the clamped minimum and maximum of the
// corners.  for (P.x = bboxmin.x; P.x <= bboxmax.x; P.x++): the start
// truncates, the bound compares the int as a float.  A start beyond the
// target (which may convert to anything over 2^30) exceeds the bound.
struct Bounds {
    float mnx, mny;
};
__device__ __forceinline__ Bounds tri_bounds(const Screen& s, int W, int H, TriS& t) {
    Bounds b;
    b.mnx = fmaxf(fminf(fminf(s.x0, s.x1), s.x2), 0.f);
    b.mny = fmaxf(fminf(fminf(s.y0, s.y1), s.y2), 0.f);
    float mxx = fminf(fmaxf(fmaxf(s.x0, s.x1), s.x2), (float)(W - 1));
    float mxy = fminf(fmaxf(fmaxf(s.y0, s.y1), s.y2), (float)(H - 1));
    t.x0 = (int)fminf(b.mnx, 0x1p30f);
    t.y0 = (int)fminf(b.mny, 0x1p30f);
    t.x1 = (int)floorf(fmaxf(mxx, -1.f));
    t.y1 = (int)floorf(fmaxf(mxy, -1.f));
    return b;
}

// What set-up found out about a triangle, for the rasters (in the bits of its
// bin entry over the face index): FACE_FAST, its coverage takes the shared
// reciprocal (cover_is_fast); FACE_SKIP_X and FACE_SKIP_Y, no pixel of the
// first column or row of its scan is covered.
constexpr uint32_t FACE_SKIP_X = 1u << 30, FACE_SKIP_Y = 1u << 29, FACE_FAST = 1u << 28;
constexpr uint32_t FACE_MASK = FACE_FAST - 1u;

// The first column (row) of the scan lies left of (above) the whole triangle
// unless a corner is exactly on it.  It is dropped where the rounding of the
// coverage test cannot reach that far: with M the largest edge component, u =
// 2^-24 and D the exact cross product of the rounded edges,
//  - P - A = b (s0y, s1y) + c (s0x, s1x) with b = Uy / D, c = Ux / D, and
//    |ux - Ux|, |uy - Uy| <= 4 u 2M (2M + 1): P is within 2M + 1 of A;
//  - |u.z - D| <= 2.1 u M^2 + u |u.z|;
//  - a covered P has uy / u.z >= 0, ux / u.z >= 0 and (ux + uy) / u.z <= 1 + u,
//    so the negative parts of its exact weights sum to at most N = u (145 M^2
//    + 64 M) / |u.z|, and P.x >= min x - u M - 2M N.
// So a column more than 2^-24 (300 M^3 + 128 M^2) / |u.z| left of the corners
// holds no covered pixel; the test below asks for 2^-15 (M^3 + M^2) / |u.z| (a
// triangle of 2 px: 2^-13 px).  Where u.z is so small that its sign is in
// doubt, that is more than a pixel.  Infinite and NaN operands keep the column.
// A triangle of e x e px then scans about e^2 pixels instead of (e + 1)^2, and
// one between two columns none: the shadow and main rasters of 20 M
// micro-triangles at 3840x2160 went from 1495 and 756 us to 948 and 555, those
// of a 1.3 M-triangle 1920x1080 frame from 60 and 46 us to 50 and 40 (reading
// bins of one range per tile; with chunks they take 1090 and 637, 59 and 48).
// (Testing the coverage of the triangles with at most 1, 2 or 3 candidates
// left in set-up and dropping the uncovered ones as well took as much time
// there as it saved here.)
__device__ __forceinline__ uint32_t tri_skips(const TriS& t, const Bounds& b) {
    float M = fmaxf(fmaxf(fabsf(t.s0x), fabsf(t.s0y)), fmaxf(fabsf(t.s1x), fabsf(t.s1y)));
    float reach = 0x1p-15f * (M * M) * (M + 1.0f), auz = fabsf(t.uz);
    return ((b.mnx - (float)t.x0) * auz > reach ? FACE_SKIP_X : 0u) |
           ((b.mny - (float)t.y0) * auz > reach ? FACE_SKIP_Y : 0u);
}

// Whether the three divisions of a triangle's candidates by u.z may share a
// refined reciprocal (tri_cover): every screen coordinate and edge within
// 2^22, and every input zero or at least 2^-8 in magnitude.  Then a nonzero
// numerator is at least 2^-62: ax and ay are multiples of 2^-31, so s0z and
// s1z are (their rounding keeps that); a product of a nonzero edge component
// and a nonzero s0z or s1z is at least 2^-39, so a multiple of 2^-62; their
// differences and the sum stay multiples of 2^-62.
// v is zero or at least 2^-8 in magnitude when (bits(v) << 1) - 1 >=
// (bits(2^-8) << 1) - 1 (zero wraps to the maximum).
__device__ __forceinline__ bool cover_is_fast(const TriS& t) {
    float ext = fmaxf(fmaxf(fmaxf(fabsf(t.ax), fabsf(t.ay)), fmaxf(fabsf(t.s0x), fabsf(t.s0y))),
                      fmaxf(fabsf(t.s1x), fabsf(t.s1y)));
    const uint32_t kMin8 = ((uint32_t)(127 - 8) << 24) - 1u;
    uint32_t mt = min(min(min((__float_as_uint(t.ax) << 1) - 1u, (__float_as_uint(t.ay) << 1) - 1u),
                          min((__float_as_uint(t.s0x) << 1) - 1u, (__float_as_uint(t.s0y) << 1) - 1u)),
                      min((__float_as_uint(t.s1x) << 1) - 1u, (__float_as_uint(t.s1y) << 1) - 1u));
    return ext <= 0x1p22f && mt >= kMin8;
}

// Set-up of a triangle for binning.  Returns false for those that can produce
// no fragment: back-facing (is_back_facing, SR/graphics.cpp:172-180),
// degenerate (|u.z| <= 1e-2, every barycentric then (-1,1,1),
// SR/graphics.cpp:230-232) or with an empty scan.  `flags` takes its FACE_*
// bits; the bounds stay the reference's scan, which binning goes by.
__device__ __forceinline__ bool tri_setup(float4 a, float4 b, float4 c, int W, int H, TriS& t, uint32_t& flags) {
    float signed_area = a.x * b.y - a.y * b.x + b.x * c.y - b.y * c.x + c.x * a.y - c.y * a.x;
    if (signed_area <= 0) return false;
    Screen s = tri_edges(a, b, c, W, H, t);
    // (double)|u.z| > 1e-2 is the same test as |u.z| > 0.01f on floats
    if (!(fabsf(t.uz) > 0.01f)) return false;
    Bounds bd = tri_bounds(s, W, H, t);
    flags = tri_skips(t, bd) | (cover_is_fast(t) ? FACE_FAST : 0u);
    return t.x1 >= t.x0 + (flags & FACE_SKIP_X ? 1 : 0) && t.y1 >= t.y0 + (flags & FACE_SKIP_Y ? 1 : 0);
}

// The same triangle in the raster, which only gets those that passed: the
// scan of the pixels that may be covered.
__device__ __forceinline__ void tri_raster(float4 a, float4 b, float4 c, int W, int H, TriS& t, uint32_t flags) {
    asm("" : "+s"(W), "+s"(H));   // uniform; as fresh(): their conversions else stay in registers, or spill
    Screen s = tri_edges(a, b, c, W, H, t);
    tri_bounds(s, W, H, t);
    if (flags & FACE_SKIP_X) t.x0++;
    if (flags & FACE_SKIP_Y) t.y0++;
    t.fast = (flags & FACE_FAST) != 0u;
}

// n / u.z as the hardware's IEEE division sequence computes it when its
// scaling steps are no-ops, from the reciprocal r = cover_recip(u.z) that
// sequence refines (the same operations in the same order, so the same bits):
// q = n r; e = fma(-u.z, q, n); q = fma(e, r, q); e = fma(-u.z, q, n);
// q = fma(e, r, q).  See tri_cover for when that holds.
__device__ __forceinline__ float cover_recip(float uz) {
    float r = __builtin_amdgcn_rcpf(uz);
    float e = fmaf(-uz, r, 1.0f);
    return fmaf(e, r, r);
}
__device__ __forceinline__ float cover_quot(float n, float uz, float r) {
    float q = n * r;
    float e = fmaf(-uz, q, n);
    q = fmaf(e, r, q);
    e = fmaf(-uz, q, n);
    return fmaf(e, r, q);
}

// barycentric + coverage + interpolate_depth at integer pixel (px, py)
// (SR/graphics.cpp:186-194, 222-233, 352-356), the three divisions by u.z
// from one refined reciprocal.  The division sequence (div_scale, rcp, four
// fma, div_fmas, div_fixup) scales its operands only when the quotient, the
// reciprocal or the numerator is near the end of the exponent range, and its
// fixup changes the result only for zero, infinite or NaN operands or a
// quotient out of range.  With the triangle's screen coordinates and edges
// within 2^22 and pixels within 2^20, |n| <= 2^47 and 2^-7 < |u.z| <= 2^45,
// so for every numerator with |n| >= 2^-80 neither happens and cover_quot
// gives the division's bits.  A zero numerator gives a zero of either sign,
// which changes neither the coverage test nor the depth (summed from +0).
// Triangles for which that is not known (cover_is_fast: rare) divide.
__device__ __forceinline__ bool tri_cover(const TriS& t, int px, int py, float& wx, float& wy, float& wz, float& z) {
    float Px = (float)px, Py = (float)py;
    float s0z = t.ax - Px;
    float s1z = t.ay - Py;
    float ux = t.s0y * s1z - s0z * t.s1y;
    float uy = s0z * t.s1x - t.s0x * s1z;
    float sum = ux + uy;
    float r = cover_recip(t.uz);
    if (t.fast) {
        wx = 1.f - cover_quot(sum, t.uz, r);
        wy = cover_quot(uy, t.uz, r);
        wz = cover_quot(ux, t.uz, r);
    } else {
        wx = 1.f - sum / t.uz;
        wy = uy / t.uz;
        wz = ux / t.uz;
    }
    if (wx < 0 || wy < 0 || wz < 0) return false;
    z = 0.0f;
    z += t.z2 * wz;
    z += t.z1 * wy;
    z += t.z0 * wx;
    return true;
}

// order-preserving 32-bit image of a depth (-0 folded onto +0)
__device__ __forceinline__ uint32_t depth_bits(float z) {
    uint32_t u = __float_as_uint(z);
    if ((u & 0x7FFFFFFFu) == 0) u = 0;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ uint64_t init_key(float d) {
    uint32_t hi = (d != d) ? 0xFFFFFFFFu : depth_bits(d);   // NaN: the first fragment passes
    return ((uint64_t)hi << 32) | 0xFFFFFFFFull;
}

__device__ __forceinline__ void stat_add(const PassDesc& P, int which, uint64_t v) {
    if (P.stats && v) atomicAdd((unsigned long long*)&P.stats[which], (unsigned long long)v);
}

// Raises a flag for this sequence and in the sticky word the host reads.
__device__ __forceinline__ void raise_flag(const Workspace& ws, uint32_t f) {
    atomicOr(&ws.seq[SEQ_FLAGS], f);
    atomicOr(&ws.status[STATUS_FLAGS], f);
}

// Lanes of the mask below this one.
__device__ __forceinline__ uint32_t mask_rank(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Inclusive prefix sum over the wave: within each row of 16 lanes, then the
// rows' last lanes into the rows after them (data-parallel primitives: no LDS
// access, and no lane masks for the compiler to keep).
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);   // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);   // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);   // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);   // row_bcast:15 into rows 1, 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);   // row_bcast:31 into rows 2, 3
    return v;
}

// Adds to a 64-bit counter of the sequence; returns its value before.
__device__ __forceinline__ uint64_t seq_add64(const Workspace& ws, int which, uint64_t v) {
    return (uint64_t)atomicAdd((unsigned long long*)(ws.seq + which), (unsigned long long)v);
}

// Zeroes the counters the launch is given to zero (Workspace::zero).
__device__ __forceinline__ void zero_counters(const Workspace& ws) {
    uint32_t gsize = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < ws.zero_n; i += gsize) gst(ws.zero + i, 0u);
}

// clip planes in clip_triangle's order (SR/graphics.cpp:136-161): w >= 1e-5,
// then x, y, z <= +w and >= -w
constexpr int CLIP_PLANES = 7;

// is_inside_plane (SR/graphics.cpp:29-49)
__device__ __forceinline__ bool inside_plane(const float* c, int plane) {
    if (plane == 0) return c[3] >= 1e-5f;
    float v = c[(plane - 1) >> 1];
    return (plane & 1) ? v <= +c[3] : v >= -c[3];
}

// ---------------------------------------------------------------------------
// k_vertex
// ---------------------------------------------------------------------------

// A vertex after its program: outcode, NDC position and 1/w.
struct PostVertex {
    uint32_t code;
    float4 r;
};
__device__ __forceinline__ PostVertex post_vertex(const float clip[4]) {
    PostVertex o;
    // is_vertex_visible (SR/graphics.cpp:132-134), then the plane tests
    o.code = (fabsf(clip[0]) <= clip[3] && fabsf(clip[1]) <= clip[3] && fabsf(clip[2]) <= clip[3]) ? CODE_VISIBLE : 0u;
#pragma unroll
    for (int pl = 0; pl < CLIP_PLANES; pl++)
        if (!inside_plane(clip, pl)) o.code |= 1u << pl;
    // clip_pos / clip_pos[3] and 1 / clip_pos[3] (SR/graphics.cpp:317, 336)
    o.r.w = 1 / clip[3];
    o.r.z = clip[2] / clip[3];
    o.r.y = clip[1] / clip[3];
    o.r.x = clip[0] / clip[3];
    return o;
}

// N vertices per lane of pass P (uniform block u), from vertex `base`: the
// loads of all N first (coalesced SoA streams), then program and stores.
template <int N>
__device__ __forceinline__ void vertex_block(const PassDesc& P, Uniforms u, int base) {
    bool need_n = P.kind != SHADER_SHADOW && P.kind != SHADER_TEXTURE;
    bool need_uv = P.kind != SHADER_SHADOW && P.kind != SHADER_GROUND && P.kind != SHADER_TOON;
    F3 pos[N], nrm[N];
    float tu[N], tv[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        int v = base + k * BLOCK + threadIdx.x;
        pos[k] = f3(0.f, 0.f, 0.f);
        nrm[k] = f3(0.f, 0.f, 0.f);
        tu[k] = tv[k] = 0.f;
        if (v < P.nverts) {
            pos[k] = f3(gld(P.px + v), gld(P.py + v), gld(P.pz + v));
            if (need_n) nrm[k] = f3(gld(P.nx + v), gld(P.ny + v), gld(P.nz + v));
            if (need_uv) {
                tu[k] = gld(P.tu + v);
                tv[k] = gld(P.tv + v);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
        int v = base + k * BLOCK + threadIdx.x;
        if (v < P.nverts) {
            float clip[4], vary[8];
            vertex_program(P.kind, u, pos[k], nrm[k], tu[k], tv[k], clip, vary);
            PostVertex o = post_vertex(clip);
            gst(P.code + v, (uint8_t)o.code);
            gst4(P.vr + v, o.r);
            if (P.nvary == 8) {
                float4* d = reinterpret_cast<float4*>(P.vs + (size_t)v * 8);
                gst4(d, make_float4(vary[0], vary[1], vary[2], vary[3]));
                gst4(d + 1, make_float4(vary[4], vary[5], vary[6], vary[7]));
            } else if (P.nvary == 2) {
                gst2(reinterpret_cast<float2*>(P.vs) + v, make_float2(vary[0], vary[1]));
            } else {
                gst(P.vs + v, vary[0]);
            }
        }
    }
}

__global__ __launch_bounds__(BLOCK) void k_vertex(const PassDesc* __restrict__ passes, int npasses, Workspace ws) {
    zero_counters(ws);
    const PassDesc& P = passes[find_pass<0>(passes, npasses, blockIdx.x)];
    vertex_block<VPT>(P, uniforms_of(P.u), (blockIdx.x - P.vblock0) * BLOCK * VPT);
}

// ---------------------------------------------------------------------------
// clipping (SR/graphics.cpp:7-161), for faces failing the trivial accept
// ---------------------------------------------------------------------------

// get_intersect_ratio (SR/graphics.cpp:51-71) of the edge p -> c
__device__ __forceinline__ float intersect_ratio(const float* p, const float* c, int plane) {
    float num, den;
    if (plane == 0) {
        num = p[3] - 1e-5f;
        den = p[3] - c[3];
    } else {
        float pv = p[(plane - 1) >> 1], cv = c[(plane - 1) >> 1];
        bool pos = plane & 1;
        num = pos ? p[3] - pv : p[3] + pv;
        den = num - (pos ? c[3] - cv : c[3] + cv);
    }
    return num / den;
}

// Orders the LDS accesses of the lanes of one wave (the wave executes them in
// order; this keeps the compiler from moving them across).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A queued face is clipped by a group of CLIP_GROUP lanes of one wave, lane i
// of the group owning vertex i of the polygon.  Its two polygon buffers
// (clip position then POLY_VARY varyings per vertex) live in LDS.
constexpr int CLIP_GROUP = 16;
constexpr int CLIP_THREADS = 512;
#ifndef HANA_CLIP_GRID
#define HANA_CLIP_GRID 2048
#endif
constexpr int CLIP_GRID = HANA_CLIP_GRID;
constexpr int COUNT_CLIP_GRID = 256;
constexpr int CLIP_FACES = CLIP_THREADS / CLIP_GROUP;   // faces per workgroup and round
constexpr int CLIP_NF = 4 + POLY_VARY;
static_assert(POLY_MAX <= CLIP_GROUP, "one lane per polygon vertex");
static_assert(POLY_MAX - 2 <= (1 << FAN_BITS), "fan index fits its bin-entry field");

// The homogeneous divide of a clip-space vertex, as the face loop applies it
// to the clipped vertices (SR/graphics.cpp:317, 336).
__device__ __forceinline__ float4 ndc_of(const float* v) {
    float w = v[3];
    float4 r;
    r.w = 1 / w;
    r.z = v[2] / w;
    r.y = v[1] / w;
    r.x = v[0] / w;
    return r;
}

// ---------------------------------------------------------------------------
// binning (Workspace): chunks of a set-up workgroup's pairs, descriptors of
// single pairs, wide triangles
// ---------------------------------------------------------------------------

// The tiles of one workgroup's (triangle, tile) pairs in an LDS hash table:
// open addressing over 2^BITS slots, a bounded probe; a tile that finds no
// slot takes a descriptor per pair instead.  512 slots when every pass has
// small triangles (a segment of 1024 faces then touches a few dozen tiles,
// and a smaller table is quicker to clear and scan), more otherwise.
constexpr int BIN_PROBES = 32;
constexpr uint32_t BIN_EMPTY = 0xFFFFFFFFu;

template <int BITS>
__device__ __forceinline__ int bin_slot(uint32_t* keys, uint32_t gt, bool insert) {
    constexpr uint32_t SLOTS = 1u << BITS;
    uint32_t h = (gt * 2654435761u) >> (32 - BITS);
    for (int p = 0; p < BIN_PROBES; p++) {
        uint32_t sl = (h + (uint32_t)p) & (SLOTS - 1);
        uint32_t k = keys[sl];
        if (k == gt) return (int)sl;
        if (k == BIN_EMPTY) {
            if (!insert) return -1;
            uint32_t old = atomicCAS(&keys[sl], BIN_EMPTY, gt);
            if (old == BIN_EMPTY || old == gt) return (int)sl;
        }
    }
    return -1;
}

// A workgroup barrier that orders LDS accesses only: unlike __syncthreads it
// does not wait for the wave's outstanding global loads first, so loads
// issued before it stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Stores descriptor idx of tile gt.  Past the tile's places it is lost, and the
// sequence rasterises nothing: the host renders it again with more of them, or
// by counting.
__device__ __forceinline__ void put_chunk(const Workspace& ws, uint32_t gt, uint32_t idx, uint2 d) {
    if (idx < ws.chunk_cap) gst2(ws.chunks + ((size_t)gt * ws.chunk_cap + idx), d);
    else atomicMax(&ws.seq[SEQ_MAX_CHUNKS], idx + 1u);
}

// The tiles of a triangle to be binned: bin entry, first and last tile.
struct TileSpan {
    uint32_t entry, t0, t1;   // x | y << 16
    __device__ __forceinline__ int x0() const { return (int)(t0 & 0xFFFFu); }
    __device__ __forceinline__ int y0() const { return (int)(t0 >> 16); }
    __device__ __forceinline__ int nx() const { return (int)(t1 & 0xFFFFu) - x0() + 1; }
    __device__ __forceinline__ int ny() const { return (int)(t1 >> 16) - y0() + 1; }
};
template <int TS>
__device__ __forceinline__ TileSpan span_of(const TriS& t, uint32_t entry) {
    TileSpan s;
    s.entry = entry;
    s.t0 = (uint32_t)(t.x0 >> TS) | ((uint32_t)(t.y0 >> TS) << 16);
    s.t1 = (uint32_t)(t.x1 >> TS) | ((uint32_t)(t.y1 >> TS) << 16);
    return s;
}

// The first and last tile of a wide triangle in one word, in units of 2^shift
// tiles that 8 bits hold; a tile's own position in those units.
__device__ __forceinline__ int wide_shift(const PassDesc& P) {
    return max(24 - __clz(max(P.tiles_x, P.tiles_y) - 1), 0);
}
__device__ __forceinline__ uint32_t wide_box(int shift, int x0, int y0, int x1, int y1) {
    return (uint32_t)(x0 >> shift) | ((uint32_t)(y0 >> shift) << 8) | ((uint32_t)(x1 >> shift) << 16) |
           ((uint32_t)(y1 >> shift) << 24);
}

// Bins the triangles over more than WIDE_TILES tiles (`wide`): into their
// pass's list while it has room, else by the whole wave into each of their
// tiles (unless the pairs pass the bins' capacity anyway).  Every active lane
// of the wave must call it together.
__device__ __forceinline__ void bin_wide(const PassDesc& P, const Workspace& ws, bool wide, const TileSpan& s) {
    if (!__ballot(wide)) return;
    uint32_t n = 0;
    bool each = false;
    if (wide) {
        n = (uint32_t)s.nx() * (uint32_t)s.ny();
        uint32_t idx = gadd(ws.wide_count + P.index, 1u);
        if (idx < ws.wide_cap) {
            gst2(ws.wide + (size_t)P.index * ws.wide_cap + idx,
                 make_uint2(wide_box(wide_shift(P), s.x0(), s.y0(), s.x0() + s.nx() - 1, s.y0() + s.ny() - 1), s.entry));
            seq_add64(ws, SEQ_WIDE_PAIRS, n);
        } else {
            each = ws.seg_region + seq_add64(ws, SEQ_PAIRS, n) + n <= ws.bin_cap;
        }
    }
    uint64_t mask = __ballot(each);
    int tile0 = P.tile0, tiles_x = P.tiles_x;
    while (mask) {
        int src = __ffsll((unsigned long long)mask) - 1;
        mask &= mask - 1;
        int wn = __shfl((int)n, src), wnx = __shfl(s.nx(), src), wx0 = __shfl(s.x0(), src), wy0 = __shfl(s.y0(), src);
        int wt0 = __shfl(tile0, src), wtx = __shfl(tiles_x, src);
        uint32_t we = __shfl(s.entry, src);
        for (int k = __lane_id(); k < wn; k += 64) {
            uint32_t gt = (uint32_t)(wt0 + (wy0 + k / wnx) * wtx + wx0 + k % wnx);
            put_chunk(ws, gt, gadd(ws.tile_chunks + gt, 1u), make_uint2(we, CHUNK_INLINE));
        }
    }
}

// k / w for 0 <= k < 1024 and 1 <= w <= 32 (a tile's pixels and row widths)
// as (k * magic) >> 16 with magic = ceil(2^16 / w): the excess
// k * (magic - 2^16/w) / 2^16 stays below 1024 / 2^16 = 1/64, less than the
// gap 1/w >= 1/32 between k/w and the next integer.
__device__ __forceinline__ uint32_t tile_div_magic(int w) { return (65536u + (uint32_t)w - 1u) / (uint32_t)w; }
__device__ __forceinline__ int tile_div(int k, uint32_t magic) { return (int)(((uint32_t)k * magic) >> 16); }

// The LDS of one workgroup's binning: the tile table, and the list of the
// triangles to bin (bin entry, first and last tile).  Set-up lists a
// workgroup's triangles, about half of its faces, before it bins them: the
// lanes of the counting and placing loops are then full, and their code is
// there once and not per face of a lane.
template <int BITS, int THREADS, int CAP>
struct SegLds {
    static constexpr int WAVES = THREADS / 64;
    uint32_t keys[1 << BITS];
    uint32_t cnt[1 << BITS];   // a slot's pairs, then its next bin position
    uint32_t entry[CAP], t0[CAP], t1[CAP];
    uint32_t n;
    uint32_t tiles[WAVES], lo[WAVES], hi[WAVES];   // the waves' SegSums
    uint32_t sum[WAVES], base, spilled;
};

// Of the narrow triangles that a lane, and then its wave, listed: their tiles,
// and the bounds of those (x | y << 16).
struct SegSums {
    uint32_t tiles = 0u, lo = 0xFFFFFFFFu, hi = 0u;
};
typedef uint16_t us2_vec __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t min_xy(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(us2_vec, a), __builtin_bit_cast(us2_vec, b)));
}
__device__ __forceinline__ uint32_t max_xy(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2_vec, a), __builtin_bit_cast(us2_vec, b)));
}

template <int BITS, int THREADS, int CAP>
__device__ __forceinline__ void seg_clear(SegLds<BITS, THREADS, CAP>& L) {
    for (int i = threadIdx.x; i < (1 << BITS); i += THREADS) {
        L.keys[i] = BIN_EMPTY;
        L.cnt[i] = 0u;
    }
    if (threadIdx.x == 0) {
        L.spilled = 0u;
        L.n = 0u;
    }
}

// A slot in an LDS counter for every lane with `want`, one LDS atomic per
// wave; wave-uniform.
__device__ __forceinline__ uint32_t wave_reserve_lds(uint32_t* counter, bool want) {
    uint64_t m = __ballot(want);
    int lane = __lane_id();
    uint32_t base = 0;
    int leader = m ? __ffsll((unsigned long long)m) - 1 : 0;
    if (m && lane == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
    base = __shfl(base, leader);
    return base + mask_rank(m);
}

// Lists the triangle of every lane with `ok`; returns its place.
template <int BITS, int THREADS, int CAP>
__device__ __forceinline__ uint32_t seg_list(SegLds<BITS, THREADS, CAP>& L, SegSums& a, bool ok, const TileSpan& s) {
    uint32_t i = wave_reserve_lds(&L.n, ok);
    if (ok) {
        L.entry[i] = s.entry;
        L.t0[i] = s.t0;
        L.t1[i] = s.t1;
        const int n = s.nx() * s.ny();
        if (n <= WIDE_TILES) {
            a.tiles += (uint32_t)n;
            a.lo = min_xy(a.lo, s.t0);
            a.hi = max_xy(a.hi, s.t1);
        }
    }
    return i;
}

// Leaves the wave's sums for bin_segment; a barrier must follow.
template <int BITS, int THREADS, int CAP>
__device__ __forceinline__ void seg_sums(SegLds<BITS, THREADS, CAP>& L, SegSums& a) {
#define HANA_DPP_STEP(ctrl, rows)                                                                            \
    a.lo = min_xy(a.lo, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)a.lo, ctrl, rows, 0xF, false));        \
    a.hi = max_xy(a.hi, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)a.hi, ctrl, rows, 0xF, false));
    HANA_DPP_STEP(0x111, 0xF)
    HANA_DPP_STEP(0x112, 0xF)
    HANA_DPP_STEP(0x114, 0xF)
    HANA_DPP_STEP(0x118, 0xF)
    HANA_DPP_STEP(0x142, 0xA)
    HANA_DPP_STEP(0x143, 0xC)
#undef HANA_DPP_STEP
    a.tiles = wave_scan(a.tiles);
    if (__lane_id() == 63) {
        const int w = threadIdx.x >> 6;
        L.tiles[w] = a.tiles;
        L.lo[w] = a.lo;
        L.hi[w] = a.hi;
    }
    a = SegSums();
}

// Bins the listed triangles, of passes pass_of(place).  Their pairs are
// counted per tile in the LDS table, the workgroup takes a descriptor per
// distinct tile with one global atomic each, all in flight together; then
// every pair takes its place with an LDS atomic.
//  - SPREAD (the one-launch geometry, all triangles of one pass, the sums made):
//    1, 2 or 4 lanes go to a triangle, by the mean number of its tiles, and the
//    table holds the rectangle of tiles that the triangles lie in, where that
//    fits -- a workgroup's faces follow one another in the mesh and mostly lie
//    close together --, else the distinct tiles by a hash, whose probes are a
//    chain of LDS accesses.  There one workgroup's chain is the launch's time
//    (128x128 with 192 faces: 15.4 -> 13.3 us a frame).  Where
//    workgroups fill the chip it is the instructions that count, and the plain
//    loop is faster (460,800 faces at 1080p: set-up 28.7 us against 32.8).
//  - The pairs go to the workgroup's own entries of the bins, [own, own_end),
//    or, where there are more, to a range of the shared rest.  (One shared
//    range for all, taken with an atomic on one counter, serialised the
//    workgroups: with 39,000 of them set-up took 818 us instead of 546.)
// Returns the own entries taken.  The table was cleared, the list and the sums
// made and a barrier passed since.
template <bool SPREAD, int BITS, int THREADS, int CAP, class PassOf>
__device__ __forceinline__ uint32_t bin_segment(SegLds<BITS, THREADS, CAP>& L, const PassOf& pass_of, const Workspace& ws,
                                                uint32_t own, uint32_t own_end) {
    constexpr int SLOTS = 1 << BITS, PER = SLOTS / THREADS, WAVES = THREADS / 64;
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t n = L.n;
    if (!n) return 0u;
    uint32_t tiles = 0u, lo = 0xFFFFFFFFu, hi = 0u;
#pragma unroll
    for (int w = 0; SPREAD && w < WAVES; w++) {
        tiles += L.tiles[w];
        lo = min_xy(lo, L.lo[w]);
        hi = max_xy(hi, L.hi[w]);
    }
    tiles = __builtin_amdgcn_readfirstlane(tiles);
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    const int bx = (int)(lo & 0xFFFFu), by = (int)(lo >> 16), bw = (int)(hi & 0xFFFFu) - bx + 1, bh = (int)(hi >> 16) - by + 1;
    const bool dense = SPREAD && tiles && bw * bh <= SLOTS;   // uniform
    const int sh = !SPREAD ? 0 : tiles > 4u * n ? 2 : (tiles > 2u * n ? 1 : 0);
    for (uint32_t i0 = 0; i0 < n; i0 += THREADS >> sh) {   // uniform
        const uint32_t i = i0 + (uint32_t)(tid >> sh);
        const bool have = i < n;
        TileSpan t{0u, 0u, 0u};
        if (have) t = TileSpan{L.entry[i], L.t0[i], L.t1[i]};
        const PassDesc& P = pass_of(have ? i : 0u);
        const int nx = t.nx(), nt = nx * t.ny(), k0 = tid & ((1 << sh) - 1);
        const bool wide = have && nt > WIDE_TILES;
        bin_wide(P, ws, wide && k0 == 0, t);
        if (have && k0 == 0 && P.stats) stat_add(P, ST_ENTRIES, (uint64_t)nt);
        if (!have || wide) continue;
        const uint32_t magic = tile_div_magic(nx);
        const int first = dense ? (t.y0() - by) * bw + t.x0() - bx : P.tile0 + t.y0() * P.tiles_x + t.x0();
        const int pitch = dense ? bw : P.tiles_x;
        for (int k = k0; k < nt; k += 1 << sh) {
            const int y = tile_div(k, magic), at = first + y * pitch + k - y * nx;
            const int sl = dense ? at : bin_slot<BITS>(L.keys, (uint32_t)at, true);
            if (sl >= 0) {
                atomicAdd(&L.cnt[sl], 1u);
            } else {
                atomicAdd(&L.spilled, 1u);
                put_chunk(ws, (uint32_t)at, gadd(ws.tile_chunks + at, 1u), make_uint2(t.entry, CHUNK_INLINE));
            }
        }
    }
    lds_barrier();
    // this lane's PER consecutive slots: their descriptors' places are fetched
    // while the workgroup's range is
    uint32_t key[PER], c[PER], idx[PER], sum = 0;
    const float inv = 1.0f / (float)bw;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int sl = tid * PER + i;
        c[i] = L.cnt[sl];
        if (dense) {
            const PassDesc& P = pass_of(0u);
            const int y = (int)(((float)sl + 0.5f) * inv);   // sl / bw: exact for such small integers
            key[i] = (uint32_t)(P.tile0 + (by + y) * P.tiles_x + bx + sl - y * bw);
        } else {
            key[i] = L.keys[sl];
        }
        idx[i] = c[i] ? gadd(ws.tile_chunks + key[i], 1u) : 0u;
        sum += c[i];
    }
    uint32_t incl = wave_scan(sum);
    if (lane == 63) L.sum[tid >> 6] = incl;
    lds_barrier();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        uint32_t v = L.sum[w];
        if (w < (tid >> 6)) before += v;
        total += v;
    }
    const uint32_t all = total + L.spilled;
    uint32_t first = own, took = total;
    bool fits = true;
    if (total > own_end - own || all != total) {   // uniform
        if (tid == 0) {
            uint64_t b = ws.seg_region + seq_add64(ws, SEQ_PAIRS, all);
            L.base = b + all <= ws.bin_cap ? (uint32_t)b : ws.bin_cap;   // past the capacity nothing is kept
        }
        lds_barrier();
        first = L.base;
        fits = first < ws.bin_cap;
        took = 0u;
    }
    uint32_t pos = first + before + incl - sum;
#pragma unroll
    for (int i = 0; i < PER; i++)
        if (c[i]) {
            put_chunk(ws, key[i], idx[i], make_uint2(pos, c[i]));
            L.cnt[tid * PER + i] = pos;
            pos += c[i];
        }
    lds_barrier();
    if (!fits) return took;
    for (uint32_t i = (uint32_t)(tid >> sh); i < n; i += THREADS >> sh) {
        TileSpan t{L.entry[i], L.t0[i], L.t1[i]};
        const int nx = t.nx(), nt = nx * t.ny();
        if (nt > WIDE_TILES) continue;
        const PassDesc& P = pass_of(i);
        const uint32_t magic = tile_div_magic(nx);
        const int at0 = dense ? (t.y0() - by) * bw + t.x0() - bx : P.tile0 + t.y0() * P.tiles_x + t.x0();
        const int pitch = dense ? bw : P.tiles_x;
        for (int k = tid & ((1 << sh) - 1); k < nt; k += 1 << sh) {
            const int y = tile_div(k, magic), at = at0 + y * pitch + k - y * nx;
            const int sl = dense ? at : bin_slot<BITS>(L.keys, (uint32_t)at, false);
            if (sl >= 0) gst(ws.bins + atomicAdd(&L.cnt[sl], 1u), t.entry);
        }
    }
    return took;
}

// Faces that fail the trivial accept, from the outcodes of their vertices:
// clip_triangle passes a polygon whose vertices are all inside a plane through
// that plane unchanged, and returns no vertex once a plane has all of them
// outside (SR/graphics.cpp:73-110, 150-152).  So a face dies whole if, at the
// first plane some vertex is outside of, every vertex is outside.
__device__ __forceinline__ bool dies_at_first_crossed_plane(uint32_t c0, uint32_t c1, uint32_t c2) {
    uint32_t some_out = (c0 | c1 | c2) & CODE_PLANES;
    if (!some_out) return false;
    uint32_t first = some_out & (0u - some_out);
    return (c0 & c1 & c2 & first) != 0u;
}

// FPT faces per lane.  Trivially accepted faces are set up from the shared
// post-transform vertices and listed, then binned by bin(pass); faces that
// clipping would remove are dropped; the others are queued for k_clip with one
// global atomic per workgroup.
template <int BITS>
struct SetupLds {
    SegLds<BITS, BLOCK, BLOCK * FPT> seg;
    uint32_t nq, qbase;
};
template <int BITS, int TS, class Bin>
__device__ __forceinline__ void setup_block(SetupLds<BITS>& S, const PassDesc* passes, int npasses, const Workspace& ws, bool stats,
                                            const Bin& bin) {
    SegLds<BITS, BLOCK, BLOCK * FPT>& L = S.seg;
    if (threadIdx.x == 0) S.nq = 0;
    int pass = find_pass<1>(passes, npasses, blockIdx.x);
    const PassDesc& P = passes[pass];
    int base = (blockIdx.x - P.fblock0) * BLOCK * FPT;
    // FPR faces per lane at a time.  Lanes past the pass's last face load that
    // face (a pass that owns a workgroup has one), so that no load waits on a
    // branch: the indices of all FPR faces are in flight together, then the
    // outcodes and post-transform vertices of all of them (gathered together,
    // so the vertices do not wait for the trivial-accept test).  The first are
    // issued before the tile table is cleared, so that the clear and its
    // barrier overlap them.
    constexpr int FPR = 4;
    static_assert(FPT % FPR == 0, "whole rounds");
    SegSums sums;
#pragma unroll 1
    for (int r = 0; r < FPT; r += FPR) {
        int ids[FPR][3];
        bool valid[FPR];
#pragma unroll
        for (int k = 0; k < FPR; k++) {
            int f = base + (r + k) * BLOCK + threadIdx.x;
            valid[k] = f < P.nfaces;
            int fl = valid[k] ? f : P.nfaces - 1;
            ids[k][0] = gld(P.idx + 3 * fl);
            ids[k][1] = gld(P.idx + 3 * fl + 1);
            ids[k][2] = gld(P.idx + 3 * fl + 2);
        }
        uint32_t codes[FPR][3];
        float4 va[FPR], vb[FPR], vc[FPR];
#pragma unroll
        for (int k = 0; k < FPR; k++) {
            for (int j = 0; j < 3; j++) codes[k][j] = gld(P.code + ids[k][j]);
            va[k] = gld4(P.vr + ids[k][0]);
            vb[k] = gld4(P.vr + ids[k][1]);
            vc[k] = gld4(P.vr + ids[k][2]);
        }
        if (r == 0) {
            seg_clear(L);
            lds_barrier();
        }
#pragma unroll
        for (int k = 0; k < FPR; k++)
            for (int j = 0; j < 3; j++) codes[k][j] = valid[k] ? codes[k][j] : 0u;
#pragma unroll
        for (int k = 0; k < FPR; k++) {
            int f = base + (r + k) * BLOCK + threadIdx.x;
            bool trivial = valid[k] && (codes[k][0] & codes[k][1] & codes[k][2] & CODE_VISIBLE);
            bool clipped = valid[k] && !trivial;
            bool clipq = clipped && !dies_at_first_crossed_plane(codes[k][0], codes[k][1], codes[k][2]);
            if (clipped && !clipq) gst(P.poly_of_face + f, -1);
            // faces to clip take the list's places from its end: a face is either
            uint32_t q = wave_reserve_lds(&S.nq, clipq);
            if (clipq) L.entry[BLOCK * FPT - 1 - q] = (uint32_t)f;
            if (stats && P.stats) {
                uint64_t nv = __popcll(__ballot(valid[k])), nc = __popcll(__ballot(clipped));
                if (__lane_id() == 0) {
                    stat_add(P, ST_FACES, nv);
                    stat_add(P, ST_CLIPPED, nc);
                }
            }
            TriS t;
            uint32_t flags = 0;
            bool ok = trivial && tri_setup(va[k], vb[k], vc[k], P.width, P.height, t, flags);
            seg_list(L, sums, ok, ok ? span_of<TS>(t, (uint32_t)f | flags) : TileSpan{0u, 0u, 0u});
        }
    }
    lds_barrier();
    if (threadIdx.x == 0) S.qbase = S.nq ? atomicAdd(&ws.seq[SEQ_CLIPQ], S.nq) : 0u;
    bin(P);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < S.nq; i += BLOCK) {
        uint32_t q = S.qbase + i;
        if (q < ws.clipq_cap) gst(ws.clip_queue + q, ((uint64_t)(uint32_t)pass << 32) | L.entry[BLOCK * FPT - 1 - i]);
        else raise_flag(ws, FLAG_CLIPQ_OVERFLOW);
    }
}

// Six waves per SIMD: the gathers of all FPT faces in flight take about 80
// VGPRs; at 64 (eight waves) the compiler serialises them and the kernel is
// slower, at 97 (five) it is slower too.
template <int BITS, int TS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(6))) void k_setup(const PassDesc* __restrict__ passes, int npasses, Workspace ws) {
    __shared__ SetupLds<BITS> S;
    setup_block<BITS, TS>(S, passes, npasses, ws, true, [&](const PassDesc& P) {
        const uint32_t own = blockIdx.x * (SEG_PAIRS * BLOCK * FPT);
        bin_segment<false>(S.seg, [&](uint32_t) -> const PassDesc& { return P; }, ws, own, own + SEG_PAIRS * BLOCK * FPT);
    });
}

// The LDS of a clipping round of FACES faces.
template <int FACES>
struct ClipLds {
    float buf[FACES][2][POLY_MAX][CLIP_NF];
    float4 ndc[FACES][POLY_MAX];
    uint32_t npoly, poly0;
};

// Clips one face per group of CLIP_GROUP lanes (`have`, uniform within the
// group) and lists its fan triangles in B (at most POLY_MAX - 2 per face) for
// bin_segment, handing their places to listed(); the whole workgroup calls it
// together.  Per
// group: the vertex program runs on the three corners in three lanes (the same
// program as k_vertex, so the same bits); then each of the seven planes of
// clip_triangle (SR/graphics.cpp:136-161) in order, one Sutherland-Hodgman
// stage (SR/graphics.cpp:73-110) computed vertex-parallel: lane i looks at the
// edge (i-1, i) and emits the intersection when the two ends differ in side
// and vertex i when it is inside, at the place the prefix sum of the lanes'
// emissions gives it -- the order and the arithmetic of the sequential loop.
// A stage with every vertex inside would copy the polygon unchanged and is
// skipped.  Pool slots (one per polygon) are reserved once per workgroup and
// round.
template <int TS, int FACES, class Seg, class Listed>
__device__ __forceinline__ void clip_round(ClipLds<FACES>& L, Seg& B, SegSums& sums, const PassDesc& P, Uniforms u, const Workspace& ws,
                                           bool have, int f, bool stats, const Listed& listed) {
    const int tid = threadIdx.x, lane = tid & 63, g = tid / CLIP_GROUP, li = tid % CLIP_GROUP;
    const uint64_t gmask = 0xFFFFull << (lane & ~(CLIP_GROUP - 1));
    if (tid == 0) L.npoly = 0;
    if (have && li < 3) {
        int v = gld(P.idx + 3 * f + li);
        bool need_n = P.kind != SHADER_SHADOW && P.kind != SHADER_TEXTURE;
        F3 p = f3(gld(P.px + v), gld(P.py + v), gld(P.pz + v));
        F3 nn = need_n ? f3(gld(P.nx + v), gld(P.ny + v), gld(P.nz + v)) : f3(0.f, 0.f, 0.f);
        float clip[4], vary[8];
        for (int c = 0; c < 8; c++) vary[c] = 0.0f;
        vertex_program(P.kind, u, p, nn, gld(P.tu + v), gld(P.tv + v), clip, vary);
        for (int c = 0; c < 4; c++) L.buf[g][0][li][c] = clip[c];
        for (int c = 0; c < POLY_VARY; c++) L.buf[g][0][li][4 + c] = vary[c];
    }
    wave_sync();
    int n = have ? 3 : 0, cur = 0;
    bool too_large = false;
    for (int plane = 0; plane < CLIP_PLANES; plane++) {
        bool act = li < n;
        bool cin = act && inside_plane(L.buf[g][cur][li], plane);
        uint64_t am = __ballot(act) & gmask, im = __ballot(cin) & gmask;
        if (n < 3 || am == im) continue;         // dead, or every vertex inside
        int prev = li == 0 ? n - 1 : li - 1;
        bool pin = act && inside_plane(L.buf[g][cur][prev], plane);
        int emit = act ? (pin != cin) + (cin ? 1 : 0) : 0;
        int incl = emit;
        for (int d = 1; d < CLIP_GROUP; d <<= 1) {
            int o = __shfl_up(incl, d, CLIP_GROUP);
            if (li >= d) incl += o;
        }
        int m = __shfl(incl, CLIP_GROUP - 1, CLIP_GROUP);
        if (m > POLY_MAX) {                      // only possible through rounding
            too_large = true;
            n = 0;
            continue;
        }
        int o = incl - emit;
        float(*in)[CLIP_NF] = L.buf[g][cur];
        float(*out)[CLIP_NF] = L.buf[g][cur ^ 1];
        if (act && pin != cin) {
            float t = intersect_ratio(in[prev], in[li], plane);
            for (int k = 0; k < CLIP_NF; k++) {
                float fv = in[prev][k];
                out[o][k] = fv + (in[li][k] - fv) * t;
            }
            o++;
        }
        if (cin)
            for (int k = 0; k < CLIP_NF; k++) out[o][k] = in[li][k];
        n = m < 3 ? 0 : m;
        cur ^= 1;
        wave_sync();
    }
    if (too_large && li == 0) raise_flag(ws, FLAG_POLY_TOO_LARGE);
    float(*poly)[CLIP_NF] = L.buf[g][cur];
    bool keep = n >= 3;                          // uniform within the group
    float4 own = make_float4(0.f, 0.f, 0.f, 0.f);
    if (keep && li < n) L.ndc[g][li] = own = ndc_of(poly[li]);
    wave_sync();
    // fan triangle (0, li+1, li+2) of the polygon in lane li
    TriS t;
    uint32_t flags = 0;   // found again by the raster
    bool ok = keep && li < n - 2 && tri_setup(L.ndc[g][0], L.ndc[g][li + 1], L.ndc[g][li + 2], P.width, P.height, t, flags);
    __syncthreads();
    uint32_t lpoly = wave_reserve_lds(&L.npoly, keep && li == 0);
    __syncthreads();
    if (tid == 0) L.poly0 = L.npoly ? atomicAdd(&ws.seq[SEQ_POLYS], L.npoly) : 0u;
    __syncthreads();
    uint32_t pid = __shfl(L.poly0 + lpoly, lane & ~(CLIP_GROUP - 1));
    if (keep && pid >= ws.poly_cap) {
        // nothing is rasterised; its triangles are still binned, for the needs
        if (li == 0) raise_flag(ws, FLAG_POLY_OVERFLOW);
        keep = false;
    }
    if (keep && li < n) {
        gst4(ws.pool_vr + ((size_t)pid * POLY_MAX + li), own);
        for (int c = 0; c < POLY_VARY; c++) gst(ws.pool_vs + (((size_t)pid * POLY_MAX + li) * POLY_VARY + c), poly[li][4 + c]);
    }
    if (have && li == 0) {
        if (keep) {
            gst(ws.pool_face + pid, f);
            if (stats) stat_add(P, ST_POLYS, 1);
        }
        gst(P.poly_of_face + f, keep ? (int)pid : -1);
    }
    uint32_t at = seg_list(B, sums, ok, ok ? span_of<TS>(t, CLIPPED_BIT | (pid << FAN_BITS) | (uint32_t)li) : TileSpan{0u, 0u, 0u});
    if (ok) listed(at);
    __syncthreads();
}

// Clips the queued faces, CLIP_FACES per workgroup and round, grid-stride over
// the queue; a round's fan triangles are then binned by bin(pass_of).
struct QueueLds {
    static constexpr int FANS = CLIP_FACES * (POLY_MAX - 2);
    ClipLds<CLIP_FACES> clip;
    SegLds<10, CLIP_THREADS, FANS> seg;
    int fan_pass[FANS];
};
template <int TS, class Bin>
__device__ __forceinline__ void clip_queue(QueueLds& Q, const PassDesc* passes, const Workspace& ws, bool stats, const Bin& bin) {
    uint32_t count = min(ws.seq[SEQ_CLIPQ], ws.clipq_cap);
    for (uint32_t base = blockIdx.x * CLIP_FACES; base < count; base += gridDim.x * CLIP_FACES) {
        seg_clear(Q.seg);
        SegSums sums;
        uint32_t q = base + threadIdx.x / CLIP_GROUP;
        bool have = q < count;
        uint64_t e = have ? gld(ws.clip_queue + q) : 0ull;
        const int pass = (int)(e >> 32);
        const PassDesc& P = passes[pass];
        clip_round<TS, CLIP_FACES>(Q.clip, Q.seg, sums, P, uniforms_of(P.u), ws, have, (int)(uint32_t)e, stats,
                                   [&](uint32_t at) { Q.fan_pass[at] = pass; });
        lds_barrier();
        bin([&](uint32_t i) -> const PassDesc& { return passes[Q.fan_pass[i]]; });
        __syncthreads();
    }
}
template <int TS>
__global__ __launch_bounds__(CLIP_THREADS) void k_clip(const PassDesc* __restrict__ passes, Workspace ws) {
    __shared__ QueueLds Q;
    clip_queue<TS>(Q, passes, ws, true, [&](const auto& pass_of) { bin_segment<false>(Q.seg, pass_of, ws, 0u, 0u); });
}

// ---------------------------------------------------------------------------
// counted binning: exact whatever the order and the sizes of the triangles
// ---------------------------------------------------------------------------

// How many descriptors the chunked binning takes depends on the order of the
// faces and on the order in which workgroups and lanes arrive.  Counted binning
// takes one bin entry per (triangle, tile) pair and nothing else: set-up and
// clipping run once to count every tile's pairs, a scan gives each tile its
// range of the bins, and they run again to place them (the pool's polygons are
// made anew, in whatever order the second run takes them).  The raster gets a
// tile's range as its one chunk.  It costs a second set-up, so it is the way
// out where the chunks do not fit.
struct Counted {
    uint32_t* pairs;         // per global tile, zero at first
    uint32_t* next;          // per global tile: where its next pair goes
    const uint32_t* first;   // or null: counters of the chunked binning before; only where that did not fit anything runs
    uint32_t region;         //   its Workspace::seg_region
    uint32_t place;          // the second run
};

// Whether the chunked binning whose counters are given ran out of descriptors
// or bins, and of nothing else.
__device__ __forceinline__ bool chunks_ran_out(const uint32_t* seq, uint32_t region, const Workspace& ws) {
    const uint64_t shared = (uint64_t)seq[SEQ_PAIRS] | ((uint64_t)seq[SEQ_PAIRS + 1] << 32);
    const uint64_t wide = (uint64_t)seq[SEQ_WIDE_PAIRS] | ((uint64_t)seq[SEQ_WIDE_PAIRS + 1] << 32);
    const uint32_t f = sequence_flags(shared, region, wide, ws.bin_cap);
    return !((seq[SEQ_FLAGS] & FLAG_NO_RASTER) || (f & FLAG_PAIR_LIMIT)) && (f || seq[SEQ_MAX_CHUNKS]);
}
__device__ __forceinline__ bool counted_runs(const Workspace& ws, const Counted& q) {
    if (q.place) return ws.seq[SEQ_COUNTED] != 0u;
    return !q.first || chunks_ran_out(q.first, q.region, ws);
}

// The counters of the chunked binning, for the raster: what it asked for is
// met.  (Its own kernels' conditions no longer read them.)
__device__ __forceinline__ void counters_met(const Workspace& ws, const Counted& q) {
    uint32_t* seq = const_cast<uint32_t*>(q.first);
    const uint64_t pairs = (uint64_t)ws.seq[SEQ_PAIRS] | ((uint64_t)ws.seq[SEQ_PAIRS + 1] << 32);
    const uint64_t past = pairs > q.region ? pairs - q.region : 0u;
    seq[SEQ_PAIRS] = (uint32_t)past;
    seq[SEQ_PAIRS + 1] = (uint32_t)(past >> 32);
    seq[SEQ_MAX_CHUNKS] = 0u;
}

// A triangle over more than WIDE_TILES tiles: listed if the pass's list holds
// them all (wide_cap > 0), else counted or placed by the whole wave in each of
// its tiles.  Past the pair limit, where nothing is rasterised, counting stops.
__device__ __forceinline__ void count_wide(const PassDesc& P, const Workspace& ws, const Counted& q, bool wide, const TileSpan& s) {
    if (!__ballot(wide)) return;
    uint32_t n = 0;
    bool each = false;
    if (wide) {
        n = (uint32_t)s.nx() * (uint32_t)s.ny();
        if (ws.wide_cap) {
            if (q.place) {
                uint32_t idx = gadd(ws.wide_count + P.index, 1u);
                if (idx < ws.wide_cap)
                    gst2(ws.wide + (size_t)P.index * ws.wide_cap + idx,
                         make_uint2(wide_box(wide_shift(P), s.x0(), s.y0(), s.x0() + s.nx() - 1, s.y0() + s.ny() - 1), s.entry));
            }
        } else {
            each = q.place || seq_add64(ws, SEQ_PAIRS, n) + n <= MAX_PAIRS;
        }
    }
    uint64_t mask = __ballot(each);
    int tile0 = P.tile0, tiles_x = P.tiles_x;
    while (mask) {
        int src = __ffsll((unsigned long long)mask) - 1;
        mask &= mask - 1;
        int wn = __shfl((int)n, src), wnx = __shfl(s.nx(), src), wx0 = __shfl(s.x0(), src), wy0 = __shfl(s.y0(), src);
        int wt0 = __shfl(tile0, src), wtx = __shfl(tiles_x, src);
        uint32_t we = __shfl(s.entry, src);
        for (int k = __lane_id(); k < wn; k += 64) {
            uint32_t gt = (uint32_t)(wt0 + (wy0 + k / wnx) * wtx + wx0 + k % wnx);
            if (q.place) {
                uint32_t pos = gadd(q.next + gt, 1u);
                if (pos < ws.bin_cap) gst(ws.bins + pos, we);
            } else {
                gadd(q.pairs + gt, 1u);
            }
        }
    }
}

// Counts or places the pairs of the listed triangles: per tile in the LDS
// table, with one global atomic per distinct tile, or where the table has no
// slot left for the tile with one per pair.
template <int BITS, int THREADS, int CAP, class PassOf>
__device__ __forceinline__ void count_segment(SegLds<BITS, THREADS, CAP>& L, const PassOf& pass_of, const Workspace& ws, const Counted& q) {
    const int tid = threadIdx.x;
    const uint32_t n = L.n;
    if (!n) return;
    uint32_t* const at_tile = q.place ? q.next : q.pairs;
    uint32_t mine = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += THREADS) {   // uniform
        const uint32_t i = i0 + (uint32_t)tid;
        const bool have = i < n;
        TileSpan t{0u, 0u, 0u};
        if (have) t = TileSpan{L.entry[i], L.t0[i], L.t1[i]};
        const PassDesc& P = pass_of(have ? i : 0u);
        const int nx = t.nx(), nt = nx * t.ny();
        const bool wide = have && nt > WIDE_TILES;
        count_wide(P, ws, q, wide, t);
        if (have && !q.place && P.stats) stat_add(P, ST_ENTRIES, (uint64_t)nt);
        if (!have || wide) continue;
        mine += (uint32_t)nt;
        for (int k = 0; k < nt; k++) {
            const uint32_t gt = (uint32_t)(P.tile0 + (t.y0() + k / nx) * P.tiles_x + t.x0() + k % nx);
            const int sl = bin_slot<BITS>(L.keys, gt, true);
            if (sl >= 0) {
                atomicAdd(&L.cnt[sl], 1u);
            } else {
                const uint32_t pos = gadd(at_tile + gt, 1u);
                if (q.place && pos < ws.bin_cap) gst(ws.bins + pos, t.entry);
            }
        }
    }
    if (!q.place) {
        const uint32_t sum = wave_scan(mine);
        if (__lane_id() == 63 && sum) seq_add64(ws, SEQ_PAIRS, sum);
    }
    lds_barrier();
    for (int sl = tid; sl < (1 << BITS); sl += THREADS)
        if (const uint32_t c = L.cnt[sl]) L.cnt[sl] = gadd(at_tile + L.keys[sl], c);
    lds_barrier();
    if (!q.place) return;
    for (uint32_t i = (uint32_t)tid; i < n; i += THREADS) {
        const TileSpan t{L.entry[i], L.t0[i], L.t1[i]};
        const int nx = t.nx(), nt = nx * t.ny();
        if (nt > WIDE_TILES) continue;
        const PassDesc& P = pass_of(i);
        for (int k = 0; k < nt; k++) {
            const uint32_t gt = (uint32_t)(P.tile0 + (t.y0() + k / nx) * P.tiles_x + t.x0() + k % nx);
            const int sl = bin_slot<BITS>(L.keys, gt, false);
            if (sl < 0) continue;   // placed above: a tile that found no slot never does
            const uint32_t pos = atomicAdd(&L.cnt[sl], 1u);
            if (pos < ws.bin_cap) gst(ws.bins + pos, t.entry);
        }
    }
}

template <int TS>
__global__ __launch_bounds__(BLOCK) void k_setup_counted(const PassDesc* __restrict__ passes, int npasses, Workspace ws, Counted q) {
    __shared__ SetupLds<10> S;
    if (!counted_runs(ws, q)) return;
    setup_block<10, TS>(S, passes, npasses, ws, !q.place, [&](const PassDesc& P) {
        count_segment(S.seg, [&](uint32_t) -> const PassDesc& { return P; }, ws, q);
    });
}
template <int TS>
__global__ __launch_bounds__(CLIP_THREADS) void k_clip_counted(const PassDesc* __restrict__ passes, Workspace ws, Counted q) {
    __shared__ QueueLds Q;
    if (!counted_runs(ws, q)) return;
    if (q.place && q.first && blockIdx.x == 0 && threadIdx.x == 0) counters_met(ws, q);
    clip_queue<TS>(Q, passes, ws, !q.place, [&](const auto& pass_of) { count_segment(Q.seg, pass_of, ws, q); });
}

// Gives every tile its range of the bins, one workgroup per SCAN_TILES tiles
// (each sums the counts before its own), and the raster that range as the
// tile's chunks; then the counters are as before the first run, for the second
// one.  Where the pairs do not fit the second run does not take place.
constexpr int SCAN_THREADS = 1024, SCAN_TILES = 4 * SCAN_THREADS;
constexpr uint32_t CHUNK_MAX = 1u << 30;   // entries of a chunk
__device__ __forceinline__ uint32_t scan_sum(uint32_t* sh, uint32_t v, uint32_t* before) {
    const int w = threadIdx.x >> 6;
    const uint32_t incl = wave_scan(v);
    if (__lane_id() == 63) sh[w] = incl;
    __syncthreads();
    uint32_t all = 0, lower = 0;
    for (int k = 0; k < SCAN_THREADS / 64; k++) {
        if (k < w) lower += sh[k];
        all += sh[k];
    }
    __syncthreads();
    if (before) *before = lower + incl - v;
    return all;
}
__global__ __launch_bounds__(SCAN_THREADS) void k_count_scan(Workspace ws, Counted q) {
    __shared__ uint32_t sh[SCAN_THREADS / 64];
    if (!counted_runs(ws, q)) return;
    const uint64_t pairs = (uint64_t)ws.seq[SEQ_PAIRS] | ((uint64_t)ws.seq[SEQ_PAIRS + 1] << 32);
    if ((ws.seq[SEQ_FLAGS] & FLAG_NO_RASTER) || pairs > ws.bin_cap) return;   // uniform
    const uint32_t n = ws.q_items, first = blockIdx.x * (uint32_t)SCAN_TILES;
    uint32_t v = 0;
    for (uint32_t t = threadIdx.x; t < first; t += SCAN_THREADS) v += gld(q.pairs + t);
    uint32_t at = scan_sum(sh, v, nullptr);
    const uint32_t t0 = first + threadIdx.x * 4u;
    uint32_t c[4];
    v = 0;
    for (uint32_t k = 0; k < 4u; k++) {
        c[k] = t0 + k < n ? gld(q.pairs + t0 + k) : 0u;
        v += c[k];
    }
    uint32_t before;
    scan_sum(sh, v, &before);
    at += before;
    for (uint32_t k = 0; k < 4u && t0 + k < n; k++) {
        const uint32_t t = t0 + k;
        gst(q.next + t, at);
        uint32_t chunks = 0;
        for (uint32_t left = c[k]; left && chunks < ws.chunk_cap; chunks++) {
            const uint32_t m = min(left, CHUNK_MAX);
            gst2(ws.chunks + ((size_t)t * ws.chunk_cap + chunks), make_uint2(at + (c[k] - left), m));
            left -= m;
        }
        gst(ws.tile_chunks + t, chunks);
        at += c[k];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ws.seq[SEQ_COUNTED] = 1u;
        ws.seq[SEQ_POLYS] = 0u;
        ws.seq[SEQ_CLIPQ] = 0u;
        for (uint32_t* w = ws.wide_count; w < ws.tile_chunks; w++) *w = 0u;
    }
}
// The geometry of a whole sequence in one launch.  Workgroups below nfb take
// FRONT_FPT faces per lane: they run the vertex program on the faces' own
// corners instead of waiting for the vertices of a launch before (each vertex
// is then transformed about six times, by the same program, so to the same
// bits), bin the trivially accepted faces and clip the others themselves, 16
// at a time.  The other workgroups run the vertex program once per vertex for
// the rasters' interpolation.  Three launches and two waits for their tails
// become one, and a workgroup of 256 faces instead of 1024 spreads small
// meshes over more CUs.  With ARGS the sequence's tables (at most two passes)
// come with the launch, and its first workgroup stores them for the rasters:
// no copy is enqueued before it.
template <int TS, bool ARGS>
__global__ __launch_bounds__(BLOCK) void k_front(FrontTables tables, PassDesc* __restrict__ d_passes,
                                                 DevUniforms* __restrict__ d_unis, int npasses, Workspace ws, int nfb) {
    constexpr int FACES = BLOCK / CLIP_GROUP, FANS = FACES * (POLY_MAX - 2);
    __shared__ SegLds<10, BLOCK, BLOCK * FRONT_FPT + FANS> L;
    __shared__ ClipLds<FACES> C;
    __shared__ uint32_t s_queue[BLOCK * FRONT_FPT];
    __shared__ uint32_t s_nq;
    zero_counters(ws);
    const PassDesc* passes = d_passes;
    const HANA_CONST_AS FrontTables* args = nullptr;
    if constexpr (ARGS) {
        // the launch's own argument memory, read through the scalar cache
        args = (const HANA_CONST_AS FrontTables*)__builtin_amdgcn_kernarg_segment_ptr();
        passes = (const PassDesc*)&args->d[0];
        if (blockIdx.x == gridDim.x - 1) {
            const HANA_CONST_AS uint32_t* sd = (const HANA_CONST_AS uint32_t*)&args->d[0];
            const HANA_CONST_AS uint32_t* su = (const HANA_CONST_AS uint32_t*)&args->u[0];
            for (int i = threadIdx.x; i < npasses * (int)(sizeof(PassDesc) / 4); i += BLOCK) gst((uint32_t*)d_passes + i, sd[i]);
            for (int i = threadIdx.x; i < npasses * (int)(sizeof(DevUniforms) / 4); i += BLOCK) gst((uint32_t*)d_unis + i, su[i]);
        }
    }
    if ((int)blockIdx.x >= nfb) {
        int vb = (int)blockIdx.x - nfb;
        int pass = find_pass<0>(passes, npasses, vb);
        const PassDesc& P = passes[pass];
        if constexpr (ARGS) vertex_block<FRONT_VPT>(P, args->u[pass], (vb - P.vblock0) * BLOCK * FRONT_VPT);
        else vertex_block<FRONT_VPT>(P, uniforms_of(P.u), (vb - P.vblock0) * BLOCK * FRONT_VPT);
        return;
    }
    if (threadIdx.x == 0) s_nq = 0;
    const int pass = find_pass<1>(passes, npasses, blockIdx.x);
    const PassDesc& P = passes[pass];
    const HANA_CONST_AS DevUniforms* up;
    if constexpr (ARGS) up = &args->u[pass];
    else up = (const HANA_CONST_AS DevUniforms*)P.u;
    const int base = ((int)blockIdx.x - P.fblock0) * BLOCK * FRONT_FPT;
    // lanes past the pass's last face take that face, so that no load waits on a branch
    F3 corner[FRONT_FPT][3];
    bool valid[FRONT_FPT];
#pragma unroll
    for (int k = 0; k < FRONT_FPT; k++) {
        int f = base + k * BLOCK + threadIdx.x;
        valid[k] = f < P.nfaces;
        int fl = valid[k] ? f : P.nfaces - 1;
        int ids[3];
        for (int j = 0; j < 3; j++) ids[j] = gld(P.idx + 3 * fl + j);
        for (int j = 0; j < 3; j++) corner[k][j] = f3(gld(P.px + ids[j]), gld(P.py + ids[j]), gld(P.pz + ids[j]));
    }
    seg_clear(L);
    lds_barrier();
    const F3 none = f3(0.f, 0.f, 0.f);
    SegSums sums;
#pragma unroll
    for (int k = 0; k < FRONT_FPT; k++) {
        int f = base + k * BLOCK + threadIdx.x;
        PostVertex va{}, vb{}, vc{};
        F3 p = corner[k][0];
#pragma unroll 1
        for (int j = 0; j < 3; j++) {   // one copy of the code: a small sequence waits for its fetch
            // the clip position alone: no normal or uv goes into it
            float clip[4], vary[8];
            vertex_program(P.kind == SHADER_SHADOW ? SHADER_SHADOW : SHADER_TEXTURE, *up, p, none, 0.f, 0.f, clip, vary);
            va = vb;
            vb = vc;
            vc = post_vertex(clip);
            p = j == 0 ? corner[k][1] : corner[k][2];
        }
        bool trivial = valid[k] && (va.code & vb.code & vc.code & CODE_VISIBLE);
        bool clipped = valid[k] && !trivial;
        bool clipq = clipped && !dies_at_first_crossed_plane(va.code, vb.code, vc.code);
        if (clipped && !clipq) gst(P.poly_of_face + f, -1);
        uint32_t q = wave_reserve_lds(&s_nq, clipq);
        if (clipq) s_queue[q] = (uint32_t)f;
        if (P.stats) {
            uint64_t nv = __popcll(__ballot(valid[k])), nc = __popcll(__ballot(clipped));
            if (__lane_id() == 0) {
                stat_add(P, ST_FACES, nv);
                stat_add(P, ST_CLIPPED, nc);
            }
        }
        TriS t;
        uint32_t flags = 0;
        bool ok = trivial && tri_setup(va.r, vb.r, vc.r, P.width, P.height, t, flags);
        seg_list(L, sums, ok, ok ? span_of<TS>(t, (uint32_t)f | flags) : TileSpan{0u, 0u, 0u});
    }
    lds_barrier();
    // clip until the list may not hold another round's fans, bin, go on
    const uint32_t nq = s_nq;
    uint32_t own = blockIdx.x * (SEG_PAIRS * BLOCK * FRONT_FPT);
    const uint32_t own_end = own + SEG_PAIRS * BLOCK * FRONT_FPT;
    for (uint32_t q0 = 0;;) {
        while (q0 < nq && L.n <= BLOCK * FRONT_FPT) {   // uniform
            uint32_t q = q0 + threadIdx.x / CLIP_GROUP;
            bool have = q < nq;
            clip_round<TS, FACES>(C, L, sums, P, *up, ws, have, have ? (int)s_queue[q] : 0, true, [](uint32_t) {});
            q0 += FACES;
        }
        seg_sums(L, sums);
        lds_barrier();
        own += bin_segment<true>(L, [&](uint32_t) -> const PassDesc& { return P; }, ws, own, own_end);
        if (q0 >= nq) break;
        __syncthreads();
        seg_clear(L);
        __syncthreads();
    }
}

// The sequence's totals, once geometry is complete: the needs the host sizes
// the next workspace by, and the flags.  Past the pair limit no workspace
// would do: that flag alone.  Returns whether the sequence is rasterised.
__device__ __forceinline__ bool sequence_fits(const Workspace& ws, bool publish) {
    typedef uint32_t u8_vec __attribute__((ext_vector_type(8)));
    u8_vec q = *(const HANA_CONST_AS u8_vec*)ws.seq;
    const uint64_t shared = (uint64_t)q[SEQ_PAIRS] | ((uint64_t)q[SEQ_PAIRS + 1] << 32);
    const uint64_t wide = (uint64_t)q[SEQ_WIDE_PAIRS] | ((uint64_t)q[SEQ_WIDE_PAIRS + 1] << 32);
    const uint32_t limits = sequence_flags(shared, ws.seg_region, wide, ws.bin_cap);
    uint32_t f = q[SEQ_FLAGS] | limits;
    if (q[SEQ_MAX_CHUNKS] && !(f & FLAG_PAIR_LIMIT)) f |= FLAG_CHUNK_OVERFLOW;
    if (publish) {
        if (!(f & FLAG_PAIR_LIMIT)) {
            const uint64_t pairs = shared + ws.seg_region;
            atomicMax(&ws.status[STATUS_NEED_BINS], pairs < MAX_PAIRS ? (uint32_t)pairs : MAX_PAIRS);
            if (f & FLAG_CHUNK_OVERFLOW) {
                // (more than any workspace grows to where no number of them would do)
                uint64_t slots = ((uint64_t)q[SEQ_MAX_CHUNKS] + CHUNK_SLACK) * ws.q_items >> 10;
                if (limits & FLAG_CHUNK_OVERFLOW) slots = 0xFFFFFFFFu;
                atomicMax(&ws.status[STATUS_NEED_CHUNKS], (uint32_t)(slots < 0xFFFFFFFFu ? slots + 1u : slots));
                atomicMax(&ws.status[STATUS_OVER_FACES], ~ws.faces);
                atomicMax(&ws.status[STATUS_OVER_TILES], ~ws.q_items);
            }
        }
        atomicMax(&ws.status[STATUS_NEED_POLYS], q[SEQ_POLYS]);
        if (f) atomicOr(&ws.status[STATUS_FLAGS], f);
        if (ws.status_out)
            for (int i = 0; i < STATUS_WORDS; i++)
                ws.status_out[i] = __hip_atomic_load(&ws.status[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return !(f & FLAG_NO_RASTER);
}

// ---------------------------------------------------------------------------
// k_raster: per-tile visibility in LDS, then one fragment program per pixel
// ---------------------------------------------------------------------------

constexpr int SMALL_PIX = HANA_SMALL_PIX;   // triangles with at most this many candidate pixels: one lane each

// A tile's entries are swept from an LDS list of this many at a time.
constexpr uint32_t TILE_LIST = 512;

// The LDS of one raster workgroup: RB lanes (2 or 4 waves) over a tile of
// 2^TS pixels a side.
template <int TS, int RB>
struct TileLds {
    static constexpr int PIX = 1 << (2 * TS);
    static constexpr int LANES = RB;
    uint64_t key[PIX];
    uint32_t nan_order[PIX];   // 1 + order of the last NaN-depth fragment
    float ax[RB], ay[RB], s0x[RB], s0y[RB], s1x[RB], s1y[RB], uz[RB];
    float z0[RB], z1[RB], z2[RB];
    uint32_t lo[RB], box[RB];
    uint8_t big[RB], med[RB];
    uint32_t list[TILE_LIST];   // the tile's entries from some position on
    uint32_t hits[2][RB / 64];  // wide triangles that touch the tile, per wave
    // staging counters of sweep round r in set r % 3 (nbig, head, nmed, mhead):
    // round r clears set (r + 2) % 3 once every wave is past round r - 1
    int cnt[3][4];
    int nan_seen;
};

// The arguments of the raster kernels, and their workspace read from there:
// like fresh(P), for the fields that only clipped triangles need.
struct RasterArgs {
    const PassDesc* passes;
    int npasses;
    Workspace ws;
};
__device__ __forceinline__ const Workspace& raster_ws() {
    const HANA_CONST_AS RasterArgs* a = (const HANA_CONST_AS RasterArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm("" : "+s"(a));
    return *(const Workspace*)&a->ws;
}

__device__ __forceinline__ void load_tri(const PassDesc& P, uint32_t e, TriS& t, uint32_t& order) {
    if (!(e & CLIPPED_BIT)) {
        int f = (int)(e & FACE_MASK);
        int i0 = gld(P.idx + 3 * f), i1 = gld(P.idx + 3 * f + 1), i2 = gld(P.idx + 3 * f + 2);
        order = (uint32_t)f << 4;
        tri_raster(gld4(P.vr + i0), gld4(P.vr + i1), gld4(P.vr + i2), P.width, P.height, t, e);
    } else {
        uint32_t pid = (e & ~CLIPPED_BIT) >> FAN_BITS, j = e & ((1u << FAN_BITS) - 1u);
        const Workspace& ws = raster_ws();
        const float4* pv = ws.pool_vr + (size_t)pid * POLY_MAX;
        order = ((uint32_t)gld(ws.pool_face + pid) << 4) + 1u + j;
        uint32_t flags = 0;
        tri_setup(gld4(pv), gld4(pv + j + 1), gld4(pv + j + 2), P.width, P.height, t, flags);
        if (flags & FACE_SKIP_X) t.x0++;
        if (flags & FACE_SKIP_Y) t.y0++;
        t.fast = (flags & FACE_FAST) != 0u;
    }
}

// One fragment of triangle t at tile-local pixel (lx, ly).
template <int TS, int RB>
__device__ __forceinline__ void frag_resolve(TileLds<TS, RB>& L, const TriS& t, uint32_t lo, int xb, int yb, int lx, int ly,
                                             bool second) {
    float wx, wy, wz, z;
    if (!tri_cover(t, xb + lx, yb + ly, wx, wy, wz, z)) return;
    int i = (ly << TS) | lx;
    if (z != z || second) {
        uint32_t order = 0xFFFFFFFEu - lo;
        if (!second) {
            atomicMax(&L.nan_order[i], order + 1u);
            L.nan_seen = 1;
            return;
        }
        uint32_t no = L.nan_order[i];
        if (no == 0u || z != z || order + 1u <= no) return;   // only fragments after the last NaN one
    }
    atomicMin((unsigned long long*)&L.key[i], ((uint64_t)depth_bits(z) << 32) | lo);
}

// A triangle staged in LDS by lane s of the sweep, with its candidate box.
template <int TS, int RB>
__device__ __forceinline__ TriS staged_tri(const TileLds<TS, RB>& L, int s, uint32_t& lo, int& x0, int& y0, int& wdt,
                                           int& npix) {
    TriS t;
    t.ax = L.ax[s]; t.ay = L.ay[s]; t.s0x = L.s0x[s]; t.s0y = L.s0y[s];
    t.s1x = L.s1x[s]; t.s1y = L.s1y[s]; t.uz = L.uz[s];
    t.z0 = L.z0[s]; t.z1 = L.z1[s]; t.z2 = L.z2[s];
    lo = L.lo[s];
    uint32_t box = L.box[s];
    x0 = box & 0xFF;
    y0 = (box >> 16) & 0xFF;
    wdt = (int)((box >> 8) & 0xFF) - x0 + 1;
    npix = wdt * ((int)((box >> 24) & 0x7F) - y0 + 1);
    t.fast = (box >> 31) != 0u;
    return t;
}

// v, but unknown to the compiler, which would otherwise compute what follows
// from it early and keep it in registers, or spill it, until then.
__device__ __forceinline__ int fresh(int v) {
    asm("" : "+v"(v));
    return v;
}

// The same for a uniform pointer: its fields are loaded where they are used, not
// together at the start, where they would not all fit in scalar registers.
__device__ __forceinline__ const PassDesc& fresh(const PassDesc& P) {
    const HANA_CONST_AS PassDesc* p = (const HANA_CONST_AS PassDesc*)&P;
    asm("" : "+s"(p));
    return *(const PassDesc*)p;
}

// A counter of the sequence (uniform; written by earlier launches of it only,
// so read through the scalar cache).
__device__ __forceinline__ uint32_t seq_count(const uint32_t* c, int i) { return *(const HANA_CONST_AS uint32_t*)(c + i); }

// What a tile has to sweep: its chunks and its pass's wide triangles.
struct TileBin {
    const uint2* chunks;
    const uint2* wide;      // boxes and entries
    int nchunks, nwide;
    uint32_t tx, ty;        // the tile in the boxes' units
};
__device__ __forceinline__ bool wide_hits(const TileBin& B, uint32_t box) {
    return B.tx >= (box & 0xFFu) && B.tx <= ((box >> 16) & 0xFFu) && B.ty >= ((box >> 8) & 0xFFu) && B.ty <= (box >> 24);
}

// How far the listing of a tile's entries has come: the next round of its pass's
// wide triangles, then the next 64 of its chunks, and the entries before those.
// The list restarts there for each TILE_LIST entries; from the first ones, whose
// descriptors were then walked again for each list, 1 M triangles on a few tiles
// took 43.3 ms instead of 30.6.
struct TileAt {
    int wide = 0, chunk = 0;
    uint32_t n = 0;
};

// Lists the wide triangles that touch the tile, of the entries from w0 on, until
// the list is full, which it returns; the whole workgroup calls it.  (On a target
// of over 256 tiles a side a box may reach a little further than its triangle,
// which the sweep then drops.)
template <int TS, int RB>
__device__ __forceinline__ bool list_wide(TileLds<TS, RB>& L, const TileBin& B, uint32_t w0, TileAt& at) {
    const int wave = threadIdx.x >> 6;
    for (; at.wide < B.nwide; at.wide += RB) {   // uniform
        const int i = fresh(at.wide + (int)threadIdx.x);
        uint2 w = make_uint2(0u, 0u);
        if (i < B.nwide) w = gld2(B.wide + i);
        const bool hit = i < B.nwide && wide_hits(B, w.x);
        const uint64_t m = __ballot(hit);
        uint32_t* hits = L.hits[(at.wide / RB) & 1];
        if (__lane_id() == 0) hits[wave] = (uint32_t)__popcll(m);
        lds_barrier();
        uint32_t p = at.n + mask_rank(m) - w0, n = at.n;
#pragma unroll
        for (int k = 0; k < RB / 64; k++) {
            uint32_t h = __builtin_amdgcn_readfirstlane(hits[k]);
            if (k < wave) p += h;
            n += h;
        }
        if (hit && p < TILE_LIST) L.list[p] = w.y;
        if (n - w0 >= TILE_LIST) return true;   // n >= w0: the round that w0 lies in, or a later one
        at.n = n;
    }
    return false;
}

// Lists the entries of the tile's chunks behind those in the same way; a barrier
// must follow.  Every wave prefix-sums the descriptors, 64 at a time, one a lane,
// and copies its share of the chunks, 4, 16 or 64 lanes to a chunk by their mean
// length, so that no barrier stands between the descriptors and the entries'
// loads.
template <int TS, int RB>
__device__ __forceinline__ bool list_chunks(TileLds<TS, RB>& L, const TileBin& B, const Workspace& ws, uint32_t w0, TileAt& at) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (; at.chunk < B.nchunks; at.chunk += 64) {   // uniform
        const int nc = min(B.nchunks - at.chunk, 64);
        uint2 d = gld2(B.chunks + at.chunk + min(lane, nc - 1));
        if (lane >= nc) d.y = 0u;
        const uint32_t n = (d.y & CHUNK_INLINE) ? 1u : d.y;
        const uint32_t incl = wave_scan(n), total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        const uint32_t first = at.n + incl - n;
        const int sh = total > 24u * nc ? 6 : (total > 6u * nc ? 4 : 2);
        for (int c0 = wave << (6 - sh); c0 < nc; c0 += (RB / 64) << (6 - sh)) {
            const int c = c0 + (lane >> sh);
            const uint32_t o = __shfl(d.x, c), y = __shfl(d.y, c), f = __shfl(first, c);
            if (c >= nc) continue;
            if (y & CHUNK_INLINE) {
                if ((lane & ((1 << sh) - 1)) == 0 && f - w0 < TILE_LIST) L.list[f - w0] = o;
            } else if (f <= w0 + (TILE_LIST - 1u)) {
                const uint32_t end = min(y, w0 + TILE_LIST - f);
                for (uint32_t i = (f < w0 ? w0 - f : 0u) + (lane & ((1 << sh) - 1)); i < end; i += 1u << sh)
                    L.list[f + i - w0] = gld(ws.bins + (o + i));
            }
        }
        if (at.n + total - w0 >= TILE_LIST) return true;
        at.n += total;
    }
    return false;
}

// One sweep over the first cnt listed entries of the tile: small triangles one per lane (in passes that
// share them, those of more than HANA_MED_PIX candidates HANA_MED_LANES lanes
// each), larger ones one per wave with the lanes spread over their candidate
// pixels.
template <int TS, int RB>
__device__ __forceinline__ int sweep(TileLds<TS, RB>& L, const PassDesc& P, uint32_t cnt, int xb, int yb,
                                     bool second, int set) {
    constexpr int EDGE = 1 << TS;
    int tid = threadIdx.x, lane = tid & 63;
    for (uint32_t base = 0; base < cnt; base += RB) {
        int* C = L.cnt[set];
        bool ok = false;
        TriS t;
        uint32_t order = 0;
        if (base + tid < cnt) {
            load_tri(P, L.list[base + tid], t, order);
            ok = true;
        }
        int bx0 = 0, bx1 = -1, by0 = 0, by1 = -1;
        if (ok) {
            bx0 = max(t.x0, xb) - xb; bx1 = min(t.x1, xb + EDGE - 1) - xb;
            by0 = max(t.y0, yb) - yb; by1 = min(t.y1, yb + EDGE - 1) - yb;
            ok = bx1 >= bx0 && by1 >= by0;
        }
        uint32_t lo = 0xFFFFFFFEu - order;
        if (ok) {
            int wdt = bx1 - bx0 + 1;
            int npix = wdt * (by1 - by0 + 1);
            if (npix <= SMALL_PIX && (!P.share_small || npix <= HANA_MED_PIX)) {
                for (int ly = by0; ly <= by1; ly++)
                    for (int lx = bx0; lx <= bx1; lx++) frag_resolve<TS, RB>(L, t, lo, xb, yb, lx, ly, second);
            } else {
                L.ax[tid] = t.ax; L.ay[tid] = t.ay; L.s0x[tid] = t.s0x; L.s0y[tid] = t.s0y;
                L.s1x[tid] = t.s1x; L.s1y[tid] = t.s1y; L.uz[tid] = t.uz;
                L.z0[tid] = t.z0; L.z1[tid] = t.z1; L.z2[tid] = t.z2;
                L.lo[tid] = lo;
                L.box[tid] = (uint32_t)bx0 | ((uint32_t)bx1 << 8) | ((uint32_t)by0 << 16) | ((uint32_t)by1 << 24) |
                             (t.fast ? 1u << 31 : 0u);
                if (npix <= SMALL_PIX) L.med[atomicAdd(&C[2], 1)] = (uint8_t)tid;
                else L.big[atomicAdd(&C[0], 1)] = (uint8_t)tid;
            }
        }
        __syncthreads();
        // every wave is past round r - 1: its set is cleared for round r + 2
        const int nmed = C[2], nbig = C[0];
        if (tid == 0) {
            int* R = L.cnt[set == 0 ? 2 : set - 1];
            R[0] = 0; R[1] = 0; R[2] = 0; R[3] = 0;
        }
        // shared small triangles: 64 / MED_LANES per wave and round
        for (;;) {
            constexpr int PER_WAVE = 64 / HANA_MED_LANES;
            if (nmed == 0) break;
            int q = 0;
            if (lane == 0) q = atomicAdd(&C[3], PER_WAVE);
            q = __shfl(q, 0);
            if (q >= nmed) break;
            int m = q + lane / HANA_MED_LANES;
            if (m < nmed) {
                uint32_t mlo;
                int x0, y0, wdt, npix;
                TriS mt = staged_tri<TS, RB>(L, L.med[m], mlo, x0, y0, wdt, npix);
                uint32_t magic = tile_div_magic(wdt);
                for (int k = lane % HANA_MED_LANES; k < npix; k += HANA_MED_LANES) {
                    int row = tile_div(k, magic);
                    frag_resolve<TS, RB>(L, mt, mlo, xb, yb, x0 + k - row * wdt, y0 + row, second);
                }
            }
        }
        for (;;) {
            if (nbig == 0) break;
            int q = 0;
            if (lane == 0) q = atomicAdd(&C[1], 1);
            q = __shfl(q, 0);
            if (q >= nbig) break;
            uint32_t blo;
            int x0, y0, wdt, npix;
            TriS bt = staged_tri<TS, RB>(L, L.big[q], blo, x0, y0, wdt, npix);
            uint32_t magic = tile_div_magic(wdt);
            for (int k = lane; k < npix; k += 64) {
                int row = tile_div(k, magic);
                frag_resolve<TS, RB>(L, bt, blo, xb, yb, x0 + k - row * wdt, y0 + row, second);
            }
        }
        // staged triangles are read until every wave is done with them (a
        // round that staged none wrote all its fragments before the barrier above)
        if (nmed | nbig) __syncthreads();
        set = set == 2 ? 0 : set + 1;
    }
    return set;
}

// Eight varyings of one corner (a 32-byte aligned row) in two 16-byte loads.
__device__ __forceinline__ void load_varyings8(const float* row, float* y) {
    float4 lo = gld4(reinterpret_cast<const float4*>(row)), hi = gld4(reinterpret_cast<const float4*>(row) + 1);
    y[0] = lo.x; y[1] = lo.y; y[2] = lo.z; y[3] = lo.w;
    y[4] = hi.x; y[5] = hi.y; y[6] = hi.z; y[7] = hi.w;
}

// Interpolates, shades and writes the winning fragment of one pixel
// (interpolate_varyings + fragment + set_depth/set_color, SR/graphics.cpp:205-220, 362-373).
__device__ __forceinline__ void shade_pixel(const PassDesc& P, uint32_t order, int px, int py) {
    uint32_t f = order >> 4, slot = order & 15u;
    float4 va, vb, vc;
    const float *sa, *sb, *sc;
    int nv;
    if (slot == 0) {
        int i0 = gld(P.idx + 3 * f), i1 = gld(P.idx + 3 * f + 1), i2 = gld(P.idx + 3 * f + 2);
        va = gld4(P.vr + i0); vb = gld4(P.vr + i1); vc = gld4(P.vr + i2);
        nv = P.nvary;
        sa = P.vs + (size_t)i0 * nv; sb = P.vs + (size_t)i1 * nv; sc = P.vs + (size_t)i2 * nv;
    } else {
        int pid = gld(P.poly_of_face + f);
        uint32_t j = slot - 1;
        const Workspace& ws = raster_ws();
        size_t base = (size_t)pid * POLY_MAX;
        va = gld4(ws.pool_vr + base); vb = gld4(ws.pool_vr + base + j + 1); vc = gld4(ws.pool_vr + base + j + 2);
        nv = POLY_VARY;
        sa = ws.pool_vs + base * POLY_VARY;
        sb = ws.pool_vs + (base + j + 1) * POLY_VARY;
        sc = ws.pool_vs + (base + j + 2) * POLY_VARY;
    }
    // the corners' live varyings, all loaded before any is awaited (8 per
    // corner as two 16-byte loads: their rows are 32-byte aligned)
    int cnt = varyings_of(P.kind);
    float ya[8], yb[8], yc[8];
    if (cnt == 8) {
        load_varyings8(sa, ya);
        load_varyings8(sb, yb);
        load_varyings8(sc, yc);
    } else {
        for (int c = 0; c < 8; c++) ya[c] = yb[c] = yc[c] = 0.0f;
        ya[0] = gld(sa); yb[0] = gld(sb); yc[0] = gld(sc);
        if (cnt == 2) { ya[1] = gld(sa + 1); yb[1] = gld(sb + 1); yc[1] = gld(sc + 1); }
    }
    TriS t;
    tri_edges(va, vb, vc, P.width, P.height, t);
    t.fast = cover_is_fast(t);
    // The weights take the same quotients as the resolve.  Where a numerator
    // is zero, tri_cover may give a zero weight of the other sign than the
    // division: wx = 1 - q is then 1 either way, and a zero wy or wz only adds
    // a signed zero beside the nonzero va.w * wx in the normaliser and in each
    // varying's sum, so no sum changes unless it is exactly zero, and then only
    // in the sign of that zero.  Depth is summed from +0 and does not change.
    float wx, wy, wz, z;
    tri_cover(t, px, py, wx, wy, wz, z);
    float k0 = va.w * wx, k1 = vb.w * wy, k2 = vc.w * wz;
    float normalizer = 1 / (k0 + k1 + k2);
    float vy[8];
    for (int c = 0; c < 8; c++) {
        if (c < cnt) {
            float sum = ya[c] * k0 + yb[c] * k1 + yc[c] * k2;
            vy[c] = sum * normalizer;
        } else {
            vy[c] = 0.0f;
        }
    }
    Tex dt{P.diffuse, P.dw, P.dh}, nt{P.normal, P.nw, P.nh};
    ShadowMap sm{P.shadow, P.shadow_depth, P.sw, P.sh};
    size_t pix = (size_t)py * P.width + px;
    // the fp32 extension's shadow pass is depth-only
    if (!(P.kind == SHADER_SHADOW && uniforms_of(P.u).shadow_fp32)) {
        C3 col = fragment_program(P.kind, uniforms_of(P.u), vy, dt, nt, sm);
        uint32_t alpha = P.clear ? P.clear_rgba : gld(P.color + pix);
        gst(P.color + pix, pack_rgb(col, alpha));
    } else if (P.clear) {
        gst(P.color + pix, P.clear_rgba);
    }
    // A NaN depth is stored as the x86 default NaN (quiet, sign set): that is
    // what the reference's own arithmetic produces for it (an invalid
    // operation such as inf/inf yields that pattern and NaN operands pass it on).
    gst(P.depth + pix, (z != z) ? __uint_as_float(0xFFC00000u) : z);
    if (P.winner) gst(P.winner + pix, order);
}

// Workgroups are dispatched to the 8 XCDs round-robin by blockIdx.  The
// logical tile of a workgroup is chosen so that each XCD receives whole runs
// of HANA_XCD_CHUNK consecutive tiles (a piece of a tile row), the runs dealt
// to the XCDs in turn: vertices, bins and texels of a run stay in one XCD's L2
// while every XCD still gets tiles from all over the target (objects cover the
// middle of a frame more than its edges).  Chunk 0 keeps blockIdx order.
#ifndef HANA_XCD_CHUNK
#define HANA_XCD_CHUNK 4
#endif
__device__ __forceinline__ int xcd_logical_block(int b, int nb) {
    const int kXcd = 8, ch = HANA_XCD_CHUNK;
    if (ch <= 0) return b;
    int full = nb / (kXcd * ch) * (kXcd * ch);
    if (b >= full) return b;
    int xcd = b % kXcd, slot = b / kXcd;
    return ((slot / ch) * kXcd + xcd) * ch + slot % ch;
}

// Renders tile lt of pass P (global tile gt, of nchunks chunks): the
// visibility of its pixels in LDS, then one fragment program per covered
// pixel; a tile no triangle reaches only takes the pass's clear.  The
// workgroup's threads all call it; it leaves L in use until they have all
// returned.
template <int TS, int RB>
__device__ void raster_tile(TileLds<TS, RB>& L, const PassDesc& P, const Workspace& ws, int lt, int gt, uint32_t nchunks,
                            uint32_t nwide) {
    constexpr int EDGE = 1 << TS, PIX = 1 << (2 * TS);
    int tx = lt % P.tiles_x, ty = lt / P.tiles_x;
    int xb = tx << TS, yb = ty << TS;
    int tid = threadIdx.x;
    int W = P.width, H = P.height;
    const int ws_shift = wide_shift(P);
    const TileBin B{ws.chunks + (size_t)gt * ws.chunk_cap, ws.wide + (size_t)P.index * ws.wide_cap,
              (int)min(nchunks, ws.chunk_cap), (int)min(nwide, ws.wide_cap), (uint32_t)(tx >> ws_shift),
              (uint32_t)(ty >> ws_shift)};

    // One copy of the code for every list of a long bin and for the second
    // sweep after NaN fragments.  Every wave reads a round's entries ahead of
    // the round's last barrier, so the next list may overwrite them.
    bool first = true, second = false;
    int set = 0;
    TileAt at;
#pragma unroll 1
    for (uint32_t w0 = 0;;) {
        bool full = list_wide<TS, RB>(L, B, w0, at);
        if (!full && at.n + (uint32_t)B.nchunks == 0u) {   // uniform: no fragment, the clear only
            const PassDesc& Q = fresh(P);
            for (int i = fresh(tid); i < PIX; i += RB) {
                int px = xb + (i & (EDGE - 1)), py = yb + (i >> TS);
                if (px >= W || py >= H) continue;
                size_t pix = (size_t)py * W + px;
                if (Q.clear) {
                    gst(Q.color + pix, Q.clear_rgba);
                    gst(Q.depth + pix, Q.clear_depth);
                }
                if (Q.winner) gst(Q.winner + pix, NO_WINNER);
            }
            return;
        }
        if (first) {
            const PassDesc& Q = fresh(P);
            for (int i = fresh(tid); i < PIX; i += RB) {
                int px = xb + (i & (EDGE - 1)), py = yb + (i >> TS);
                uint64_t k = ~0ull;
                if (px < W && py < H) k = init_key(Q.clear ? Q.clear_depth : gld(Q.depth + ((size_t)py * W + px)));
                L.key[i] = k;
                L.nan_order[i] = 0u;
            }
            if (tid < 12) (&L.cnt[0][0])[tid] = 0;
            if (tid == 0) L.nan_seen = 0;
        }
        if (!full) full = list_chunks<TS, RB>(L, B, ws, w0, at);
        first = false;
        __syncthreads();
        set = sweep<TS, RB>(L, P, full ? TILE_LIST : at.n - w0, xb, yb, second, set);
        w0 += TILE_LIST;
        if (full) continue;
        if (second || !L.nan_seen) break;
        // pixels that saw a NaN-depth fragment restart after the last one
        for (int i = fresh(tid); i < PIX; i += RB) {
            uint32_t no = L.nan_order[i];
            if (no) L.key[i] = (0xFFFFFFFFull << 32) | (uint64_t)(0xFFFFFFFEu - (no - 1u));
        }
        __syncthreads();
        second = true;
        w0 = 0;
        at = TileAt();
    }

    uint32_t written = 0;
    const PassDesc& Q = fresh(P);
    for (int i = fresh(tid); i < PIX; i += RB) {
        int px = xb + (i & (EDGE - 1)), py = yb + (i >> TS);
        if (px >= W || py >= H) continue;
        uint32_t lo = (uint32_t)L.key[i];
        size_t pix = (size_t)py * W + px;
        if (lo == 0xFFFFFFFFu) {
            if (Q.clear) {
                gst(Q.color + pix, Q.clear_rgba);
                gst(Q.depth + pix, Q.clear_depth);
            }
            if (Q.winner) gst(Q.winner + pix, NO_WINNER);
            continue;
        }
        shade_pixel(Q, 0xFFFFFFFEu - lo, px, py);
        written++;
    }
    if (Q.stats) stat_add(Q, ST_PIXELS, written);
}

// Waves per SIMD that the raster's LDS allows (160 KiB per CU, 4 SIMDs, at
// most 8 waves each).  The kernels ask the compiler for that occupancy: the
// persistent raster, whose tile loop keeps more values live, would otherwise
// take 78-84 VGPRs (6 waves per SIMD) where its LDS allows 8.
template <int TS, int RB>
constexpr int raster_occupancy() {
    constexpr int lds = (int)sizeof(TileLds<TS, RB>) + 16;
    constexpr int w = (163840 / lds) * (RB / 64) / 4;
    return w < 1 ? 1 : (w > 8 ? 8 : w);
}

// The pass of raster workgroup blk of group GROUP and its global tile: one
// scalar load of the group's lookup (Workspace::tile_pass), then, in a run of
// workgroups that spans passes, a step per pass boundary; a binary search
// without a lookup.
template <int GROUP>
__device__ __forceinline__ int raster_pass(const PassDesc* P, int n, const Workspace& ws, int blk, int& gt) {
    const uint2* tp = ws.tile_pass[GROUP];
    if (!tp) {
        int p = find_pass<2>(P, n, blk);
        gt = P[p].tile0 + blk - P[p].tblock0;
        return p;
    }
    u2_vec e = *(const HANA_CONST_AS u2_vec*)(tp + (blk >> TILE_PASS_SHIFT));
    int p = (int)(e.x & ~TILE_PASS_PURE);
    gt = blk + (int)e.y;
    if (!(e.x & TILE_PASS_PURE)) {
        while (p + 1 < n && P[p + 1].tblock0 <= blk) p++;
        gt = P[p].tile0 + blk - P[p].tblock0;
    }
    return p;
}

// One workgroup per tile of one dependency group (passes of the group, their
// tiles numbered from 0 by tblock0), XCD-banded.  GROUP only names the launch
// (the shadow passes' group 0, the main passes' group 1) in profiles.
template <int TS, int GROUP, int RB>
__global__ __launch_bounds__(RB) __attribute__((amdgpu_waves_per_eu(raster_occupancy<TS, RB>())))
void k_raster(const PassDesc* __restrict__ passes, int npasses, Workspace ws) {
    __shared__ TileLds<TS, RB> L;
    // the loads that decide the workgroup's work are issued before any of
    // them is awaited: the pass lookup, the tile's chunks, the sequence's totals
    int blk = xcd_logical_block(blockIdx.x, gridDim.x);
    int gt;
    const PassDesc& P = passes[raster_pass<GROUP>(passes, npasses, ws, blk, gt)];
    uint32_t nchunks = seq_count(ws.tile_chunks, gt), nwide = seq_count(ws.wide_count, P.index);
    // an incomplete sequence leaves its targets untouched: the host renders it again
    if (!sequence_fits(ws, blockIdx.x == 0 && threadIdx.x == 0)) return;
    raster_tile<TS, RB>(L, P, ws, blk - P.tblock0, gt, nchunks, nwide);
}

// The persistent raster: a fixed grid of workgroups takes the tiles of every
// pass of the sequence from one queue, RQ_CHUNK consecutive tiles at a time
// (they share triangles, which stay in the taking XCD's L2).  Queue items are
// global tile indices: the shadow passes' tiles first, then the main passes
// that sample no shadow map drawn here, then those that do.  A main pass of
// the last kind needs every shadow tile finished:
//  - a workgroup counts the shadow tiles it finishes and publishes the count
//    once, with one release at agent scope (its shadow-map writes become
//    visible on every XCD), when it first takes an item past them or finds
//    the queue empty;
//  - before its first item that samples a map, it waits until the published
//    total is every shadow tile, then acquires once.
// Items are taken in queue order, so every shadow tile was taken before any
// item that waits, by a workgroup that publishes before it could wait itself:
// the wait ends.  It is still bounded: past RQ_SPIN_LIMIT polls it raises
// FLAG_QUEUE_STALL (an error for the host) and goes on.
constexpr uint32_t RQ_CHUNK = 4;
constexpr uint32_t RQ_SPIN_LIMIT = 1u << 24;

// largest pass index whose first global tile is <= item (passes sorted by it)
__device__ __forceinline__ int pass_of_item(const PassDesc* P, int n, uint32_t item) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if ((uint32_t)P[mid].tile0 <= item) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

template <int TS, int RB>
__global__ __launch_bounds__(RB) __attribute__((amdgpu_waves_per_eu(raster_occupancy<TS, RB>())))
void k_raster_q(const PassDesc* __restrict__ passes, int npasses, Workspace ws) {
    __shared__ TileLds<TS, RB> L;
    __shared__ uint32_t s_first;
    if (!sequence_fits(ws, blockIdx.x == 0 && threadIdx.x == 0)) return;
    const int tid = threadIdx.x;
    uint32_t mine = 0;   // shadow tiles finished here, not yet published
    bool published = false, ready = false;
    for (;;) {
        if (tid == 0) s_first = atomicAdd(&ws.seq[SEQ_QUEUE], RQ_CHUNK);
        __syncthreads();
        // uniform: the tile's pass, bounds and tables then live in SGPRs
        uint32_t first = __builtin_amdgcn_readfirstlane(s_first);
        __syncthreads();
        uint32_t end = min(first + RQ_CHUNK, ws.q_items);
        if (!published && (first >= ws.q_g0 || first >= ws.q_items)) {
            if (tid == 0 && mine)
                __hip_atomic_fetch_add(&ws.seq[SEQ_QUEUE_DONE], mine, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            published = true;
        }
        if (first >= ws.q_items) break;
        for (uint32_t it = first; it < end; it++) {
            if (!published && it >= ws.q_g0) {
                if (tid == 0 && mine)
                    __hip_atomic_fetch_add(&ws.seq[SEQ_QUEUE_DONE], mine, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
                published = true;
            }
            if (!ready && it >= ws.q_dep_from) {
                if (tid == 0) {
                    uint32_t spins = 0;
                    while (__hip_atomic_load(&ws.seq[SEQ_QUEUE_DONE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < ws.q_g0) {
                        if (++spins > RQ_SPIN_LIMIT) {
                            raise_flag(ws, FLAG_QUEUE_STALL);
                            break;
                        }
                        __builtin_amdgcn_s_sleep(8);
                    }
                }
                __syncthreads();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                ready = true;
            }
            const PassDesc& P = passes[pass_of_item(passes, npasses, it)];
            raster_tile<TS, RB>(L, P, ws, (int)(it - (uint32_t)P.tile0), (int)it, seq_count(ws.tile_chunks, (int)it),
                                seq_count(ws.wide_count, P.index));
            __syncthreads();   // the tile's writes are issued and L is free again
            if (it < ws.q_g0) mine++;
        }
    }
}

// fills a 32-bit buffer (graph-safe clear)
__global__ void k_fill32(uint32_t* dst, uint32_t value, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) dst[i] = value;
}

// window_draw_buffer (SR/win32.cpp:348-370) without the window: row r of the
// target lands on row h-1-r, R and B bytes swap (RGBA -> BGRA), alpha is
// carried along.  One word per lane, coalesced reads and writes per row.
__global__ void k_present(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, int w, int h) {
    size_t n = (size_t)w * h;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        size_t r = i / (size_t)w, c = i - r * (size_t)w;
        uint32_t v = src[i];
        dst[((size_t)(h - 1) - r) * (size_t)w + c] = ((v & 0xFFu) << 16) | (v & 0xFF00FF00u) | ((v >> 16) & 0xFFu);
    }
}

// The word of the read-back image at i: k_present's, or the plane's own.
__device__ __forceinline__ uint32_t read_back_word(const uint32_t* src, uint32_t i, uint32_t w, uint32_t h, bool flip) {
    if (!flip) return gld(src + i);
    uint32_t r = i / w, v = gld(src + (size_t)(h - 1u - r) * w + (i - r * w));
    return ((v & 0xFFu) << 16) | (v & 0xFF00FF00u) | ((v >> 16) & 0xFFu);
}

// A plane written to host memory by the kernel itself, READ_WGS workgroups per
// band, and a flag in host memory as each band is complete: the host copies it
// on to the caller while the next ones come.  Bound by the link (2.4 MB in
// about 50 us), of which 16-byte stores keep enough in flight.
__global__ void k_read_back(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, uint32_t w, uint32_t h, int flip,
                            uint32_t band, uint32_t wgs, uint32_t* done, uint32_t* flags, uint32_t epoch) {
    const uint32_t n = w * h, b = blockIdx.x / wgs, first = b * band, end = min(n, first + band);
    for (uint32_t i = first + ((blockIdx.x - b * wgs) * BLOCK + threadIdx.x) * 4u; i < end; i += wgs * BLOCK * 4u) {
        uint32_t v[4];
        for (uint32_t k = 0; k < 4u; k++) v[k] = i + k < end ? read_back_word(src, i + k, w, h, flip != 0) : 0u;
        if (i + 4u <= end) *reinterpret_cast<uint4*>(dst + i) = make_uint4(v[0], v[1], v[2], v[3]);
        else
            for (uint32_t k = 0; i + k < end; k++) dst[i + k] = v[k];
    }
    if (gridDim.x == wgs) return;   // one band: the host waits for the launch
    __syncthreads();
    if (threadIdx.x == 0) {
        // one fence for the workgroup (one a thread took 15 us more at 360 KB);
        // a band's workgroups count up over the launches
        __threadfence_system();
        if ((gadd(done + b, 1u) + 1u) % wgs == 0u) {
            __threadfence_system();
            __hip_atomic_store(flags + b, epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------

hipError_t launch_vertex(const PassDesc* d_passes, int npasses, const Workspace& ws, int blocks, hipStream_t s) {
    if (npasses <= 0) return hipSuccess;
    // k_vertex also zeroes the sequence's counters, so it runs even when no
    // pass has a vertex
    blocks = std::max(blocks, 1);
    hipLaunchKernelGGL(k_vertex, dim3(blocks), dim3(BLOCK), 0, s, d_passes, npasses, ws);
    return hipGetLastError();
}
hipError_t launch_setup(const PassDesc* d_passes, int npasses, const Workspace& ws, int blocks, bool small_tris,
                        hipStream_t s) {
    if (blocks <= 0) return hipSuccess;
    if (ws.tile_shift == 5) {
        if (small_tris) hipLaunchKernelGGL((k_setup<9, 5>), dim3(blocks), dim3(BLOCK), 0, s, d_passes, npasses, ws);
        else hipLaunchKernelGGL((k_setup<10, 5>), dim3(blocks), dim3(BLOCK), 0, s, d_passes, npasses, ws);
    } else {
        if (small_tris) hipLaunchKernelGGL((k_setup<9, 4>), dim3(blocks), dim3(BLOCK), 0, s, d_passes, npasses, ws);
        else hipLaunchKernelGGL((k_setup<10, 4>), dim3(blocks), dim3(BLOCK), 0, s, d_passes, npasses, ws);
    }
    return hipGetLastError();
}
hipError_t launch_clip(const PassDesc* d_passes, const Workspace& ws, hipStream_t s) {
    // grid-stride: the queue length is only known on the device
    if (ws.tile_shift == 5) hipLaunchKernelGGL(k_clip<5>, dim3(CLIP_GRID), dim3(CLIP_THREADS), 0, s, d_passes, ws);
    else hipLaunchKernelGGL(k_clip<4>, dim3(CLIP_GRID), dim3(CLIP_THREADS), 0, s, d_passes, ws);
    return hipGetLastError();
}
hipError_t launch_counted(const PassDesc* d_passes, int npasses, const Workspace& ws, const CountedBins& b, int blocks, hipStream_t s) {
    Counted q{b.pairs, b.next, b.first, b.region, 0u};
    const int scan = (int)((ws.q_items + SCAN_TILES - 1) / SCAN_TILES);
    for (q.place = 0; q.place < 2u; q.place++) {
        hipError_t e;
        if (q.place) {
            hipLaunchKernelGGL(k_count_scan, dim3(std::max(scan, 1)), dim3(SCAN_THREADS), 0, s, ws, Counted{b.pairs, b.next, b.first, b.region, 0u});
            if ((e = hipGetLastError()) != hipSuccess) return e;
        }
        if (blocks > 0) {
            if (ws.tile_shift == 5) hipLaunchKernelGGL(k_setup_counted<5>, dim3(blocks), dim3(BLOCK), 0, s, d_passes, npasses, ws, q);
            else hipLaunchKernelGGL(k_setup_counted<4>, dim3(blocks), dim3(BLOCK), 0, s, d_passes, npasses, ws, q);
            if ((e = hipGetLastError()) != hipSuccess) return e;
        }
        if (ws.tile_shift == 5) hipLaunchKernelGGL(k_clip_counted<5>, dim3(COUNT_CLIP_GRID), dim3(CLIP_THREADS), 0, s, d_passes, ws, q);
        else hipLaunchKernelGGL(k_clip_counted<4>, dim3(COUNT_CLIP_GRID), dim3(CLIP_THREADS), 0, s, d_passes, ws, q);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}
hipError_t launch_front(const FrontTables* tables, PassDesc* d_passes, DevUniforms* d_unis, int npasses, const Workspace& ws,
                        int fblocks, int vblocks, hipStream_t s) {
    static const FrontTables none{};
    if (npasses <= 0) return hipSuccess;
    // the last workgroup stores the tables, so one runs even for empty meshes
    dim3 grid(std::max(fblocks + vblocks, 1)), block(BLOCK);
    const FrontTables& t = tables ? *tables : none;
    if (ws.tile_shift == 5) {
        if (tables) hipLaunchKernelGGL((k_front<5, true>), grid, block, 0, s, t, d_passes, d_unis, npasses, ws, fblocks);
        else hipLaunchKernelGGL((k_front<5, false>), grid, block, 0, s, t, d_passes, d_unis, npasses, ws, fblocks);
    } else {
        if (tables) hipLaunchKernelGGL((k_front<4, true>), grid, block, 0, s, t, d_passes, d_unis, npasses, ws, fblocks);
        else hipLaunchKernelGGL((k_front<4, false>), grid, block, 0, s, t, d_passes, d_unis, npasses, ws, fblocks);
    }
    return hipGetLastError();
}
template <int TS, int RB>
static void raster_launch(const PassDesc* d_passes, int npasses, const Workspace& ws, int blocks, int group,
                          hipStream_t s) {
    if (group) hipLaunchKernelGGL((k_raster<TS, 1, RB>), dim3(blocks), dim3(RB), 0, s, d_passes, npasses, ws);
    else hipLaunchKernelGGL((k_raster<TS, 0, RB>), dim3(blocks), dim3(RB), 0, s, d_passes, npasses, ws);
}
hipError_t launch_raster(const PassDesc* d_passes, int npasses, const Workspace& ws, int blocks, int group, int waves,
                         hipStream_t s) {
    if (blocks <= 0) return hipSuccess;
    bool two = waves == 2;
    if (ws.tile_shift == 5) {
        if (two) raster_launch<5, 128>(d_passes, npasses, ws, blocks, group, s);
        else raster_launch<5, 256>(d_passes, npasses, ws, blocks, group, s);
    } else {
        if (two) raster_launch<4, 128>(d_passes, npasses, ws, blocks, group, s);
        else raster_launch<4, 256>(d_passes, npasses, ws, blocks, group, s);
    }
    return hipGetLastError();
}
hipError_t launch_raster_queue(const PassDesc* d_passes, int npasses, const Workspace& ws, int workgroups,
                               int waves, hipStream_t s) {
    if (workgroups <= 0 || ws.q_items == 0) return hipSuccess;
    bool two = waves == 2;
    if (ws.tile_shift == 5) {
        if (two) hipLaunchKernelGGL((k_raster_q<5, 128>), dim3(workgroups), dim3(128), 0, s, d_passes, npasses, ws);
        else hipLaunchKernelGGL((k_raster_q<5, 256>), dim3(workgroups), dim3(256), 0, s, d_passes, npasses, ws);
    } else {
        if (two) hipLaunchKernelGGL((k_raster_q<4, 128>), dim3(workgroups), dim3(128), 0, s, d_passes, npasses, ws);
        else hipLaunchKernelGGL((k_raster_q<4, 256>), dim3(workgroups), dim3(256), 0, s, d_passes, npasses, ws);
    }
    return hipGetLastError();
}
hipError_t launch_read_back(const uint32_t* src, uint32_t* dst, int w, int h, bool flip, uint32_t band, uint32_t* done,
                            uint32_t* flags, uint32_t epoch, hipStream_t s) {
    const uint32_t bands = ((uint32_t)w * (uint32_t)h + band - 1u) / band;
    if (bands == 0) return hipSuccess;
    if (bands > READ_BANDS || band % 4u) return hipErrorInvalidValue;
    // a single band has as many workgroups as it fills once
    const uint32_t wgs = bands > 1 ? READ_WGS : ((uint32_t)w * (uint32_t)h + 4 * BLOCK - 1) / (4 * BLOCK);
    hipLaunchKernelGGL(k_read_back, dim3(bands * wgs), dim3(BLOCK), 0, s, src, dst, (uint32_t)w, (uint32_t)h, flip ? 1 : 0,
                       band, wgs, done, flags, epoch);
    return hipGetLastError();
}
hipError_t launch_present(const uint32_t* src, uint32_t* dst, int w, int h, hipStream_t s) {
    size_t n = (size_t)w * h;
    if (n == 0) return hipSuccess;
    int blocks = (int)std::min<size_t>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_present, dim3(blocks), dim3(256), 0, s, src, dst, w, h);
    return hipGetLastError();
}

hipError_t launch_fill32(uint32_t* dst, uint32_t value, size_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    int blocks = (int)std::min<size_t>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_fill32, dim3(blocks), dim3(256), 0, s, dst, value, n);
    return hipGetLastError();
}

}  // namespace hana
