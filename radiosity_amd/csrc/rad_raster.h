// rad_raster.h - device functions shared by the rasterizer kernels: the
// clip-space pipeline up to the snapped triangle, the drawing of a record into
// a tile's depth keys in LDS, and the run reduction of ProcessHemicube.
// Operation order is part of the item-buffer specification (compiled with
// -ffp-contract=off).
#pragma once

#include "rad_internal.h"

namespace rad {

struct CV4 {
    float c[4];
};

struct SV {
    int32_t x, y;
    float z;
};

struct FaceView {
    int32_t vpx, vpy;           // viewport origin inside the hemicube slab (Main.cpp:316-347)
    int32_t sx0, sy0, sx1, sy1; // scissor in face-local pixels, [x0,x1) x [y0,y1)
};

__device__ static inline FaceView face_view(int32_t W, int face)
{
    FaceView v;
    int32_t h2 = W / 2;
    switch (face) {
    case 0: v.vpx = 0; v.vpy = W; v.sx0 = 0; v.sy0 = 0; v.sx1 = W; v.sy1 = h2; break;
    case 1: v.vpx = W; v.vpy = h2; v.sx0 = 0; v.sy0 = h2; v.sx1 = W; v.sy1 = W; break;
    case 2: v.vpx = -h2; v.vpy = 0; v.sx0 = h2; v.sy0 = 0; v.sx1 = W; v.sy1 = W; break;
    case 3: v.vpx = W + h2; v.vpy = 0; v.sx0 = 0; v.sy0 = 0; v.sx1 = h2; v.sy1 = W; break;
    default: v.vpx = h2; v.vpy = 0; v.sx0 = 0; v.sy0 = 0; v.sx1 = W; v.sy1 = W; break;
    }
    return v;
}

__device__ static inline float clip_dist(const CV4 &v, int plane)
{
    switch (plane) {
    case 0: return v.c[2] + v.c[3];
    case 1: return kGuard * v.c[3] - v.c[0];
    case 2: return kGuard * v.c[3] + v.c[0];
    case 3: return kGuard * v.c[3] - v.c[1];
    default: return kGuard * v.c[3] + v.c[1];
    }
}

__device__ static inline SV project(const CV4 &v, float halfW)
{
    float iw = 1.0f / v.c[3];
    float xn = v.c[0] * iw, yn = v.c[1] * iw, zn = v.c[2] * iw;
    float xl = (xn + 1.0f) * halfW, yl = (yn + 1.0f) * halfW;
    SV s;
    s.x = (int32_t)rintf(xl * (float)kSub);
    s.y = (int32_t)rintf(yl * (float)kSub);
    s.z = zn * 0.5f + 0.5f;
    return s;
}

// Edge functions of a CCW triangle: E_e(p) = A_e p.x + B_e p.y + C_e, inside
// when E_e + bias_e > 0 for all three (top-left rule, y up).
struct Edges {
    int32_t A[3], B[3];
    int64_t C[3];
    int32_t bias[3];
};

__device__ static inline void make_edges(const int32_t *x, const int32_t *y, Edges &e)
{
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        int q = k == 2 ? 0 : k + 1;
        int32_t A = y[k] - y[q], B = x[q] - x[k];
        e.A[k] = A;
        e.B[k] = B;
        e.C[k] = -((int64_t)A * x[k] + (int64_t)B * y[k]);
        e.bias[k] = (A > 0 || (A == 0 && B < 0)) ? 1 : 0;
    }
}

// Depth key of face-local pixel (ix, iy) or 0 when the centre is outside
// the triangle or fails the depth range.
__device__ static inline uint64_t frag_key(const Edges &e, const RasterRec &r, int32_t ix,
                                           int32_t iy)
{
    int32_t px = ix * kSub + kSub / 2, py = iy * kSub + kSub / 2;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        int64_t E = (int64_t)e.A[k] * px + (int64_t)e.B[k] * py + e.C[k];
        if (E + e.bias[k] <= 0)
            return 0;
    }
    float z = fmaf(r.dzdx, (float)(px - r.x[0]), fmaf(r.dzdy, (float)(py - r.y[0]), r.z0));
    if (!(z > 0.0f))
        z = 0.0f;
    if (!(z < 1.0f))
        return 0;
    return ((uint64_t)__float_as_uint(z) << 32) | r.id;
}

// Clipping against the near plane and the guard band is Sutherland-Hodgman
// (clip_polygon_wave, below): planes in clip_dist order, each polygon walked from
// vertex 0, an intersection interpolated from the inside vertex towards the
// outside one.  A convex polygon gains at most one vertex per plane (3 + 5 =
// 8); more sign changes along the outline than two can only come from
// vertices within rounding of a plane, and a polygon that would outgrow
// kClipMax (fewer than two free places before a vertex) is dropped and
// flagged as an overflow.
constexpr int kClipMax = 12;

// Clip-space transform of a triangle: MVP (column-major) times (x, y, z, 1),
// each row summed left to right.
__device__ static inline void transform3(const float *mm, const float (&vx)[3][3], CV4 *poly)
{
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float x = vx[k][0], y = vx[k][1], z = vx[k][2];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            poly[k].c[r] = mm[0 * 4 + r] * x + mm[1 * 4 + r] * y + mm[2 * 4 + r] * z +
                           mm[3 * 4 + r];
    }
}

// Scissor rectangle of a face in clip space (x / w, y / w) with a one-pixel
// margin: (lo_x, hi_x, lo_y, hi_y).
__device__ static inline float4 face_scissor_clip(int32_t W, int face)
{
    FaceView fv = face_view(W, face);
    return make_float4(2.0f * (float)(fv.sx0 - 1) / (float)W - 1.0f,
                       2.0f * (float)(fv.sx1 + 1) / (float)W - 1.0f,
                       2.0f * (float)(fv.sy0 - 1) / (float)W - 1.0f,
                       2.0f * (float)(fv.sy1 + 1) / (float)W - 1.0f);
}

// Pixels of a snapped triangle inside the face-local rectangle
// [rx0, rx1) x [ry0, ry1): the bbox of the pixel centres it can cover, and
// twice its signed area.  False when it covers none (clockwise, degenerate
// or between pixel centres).
__device__ static inline bool snapped_bbox(const SV &a, const SV &b, const SV &c, int32_t rx0,
                                           int32_t ry0, int32_t rx1, int32_t ry1, int64_t &area2,
                                           int32_t &ix0, int32_t &iy0, int32_t &ix1, int32_t &iy1)
{
    area2 = (int64_t)(b.x - a.x) * (c.y - a.y) - (int64_t)(c.x - a.x) * (b.y - a.y);
    if (area2 <= 0)
        return false;
    int32_t xmin = min(a.x, min(b.x, c.x)), xmax = max(a.x, max(b.x, c.x));
    int32_t ymin = min(a.y, min(b.y, c.y)), ymax = max(a.y, max(b.y, c.y));
    ix0 = max((xmin - 128 + 255) >> 8, rx0);
    ix1 = min((xmax - 128) >> 8, rx1 - 1);
    iy0 = max((ymin - 128 + 255) >> 8, ry0);
    iy1 = min((ymax - 128) >> 8, ry1 - 1);
    return ix0 <= ix1 && iy0 <= iy1;
}

// The record of a snapped triangle: its vertices and the depth plane
// anchored at vertex 0.
__device__ static inline void make_record(const SV &a, const SV &b, const SV &c, int64_t area2,
                                          uint32_t id, RasterRec &rr)
{
    double dx1 = (double)(b.x - a.x), dy1 = (double)(b.y - a.y);
    double dx2 = (double)(c.x - a.x), dy2 = (double)(c.y - a.y);
    double dz1 = (double)b.z - (double)a.z, dz2 = (double)c.z - (double)a.z;
    double ar = (double)area2;
    rr.x[0] = a.x; rr.x[1] = b.x; rr.x[2] = c.x;
    rr.y[0] = a.y; rr.y[1] = b.y; rr.y[2] = c.y;
    rr.dzdx = (float)((dz1 * dy2 - dz2 * dy1) / ar);
    rr.dzdy = (float)((dx1 * dz2 - dx2 * dz1) / ar);
    rr.z0 = a.z;
    rr.id = id;
}

// What the exact pipeline makes of one triangle of one face.
enum TriClass { kTriOut, kTriClip, kTriIn };

// Clip-space vertices against the near plane, the guard band and the
// rectangle scis (lo_x, hi_x, lo_y, hi_y in x / w and y / w, a one-pixel
// margin included): outside, in need of clipping, or inside.
__device__ static inline TriClass classify_tri(const CV4 *poly, float4 scis)
{
    // every clip_dist >= 0 (a difference has the sign of its comparison; NaN
    // is outside) for nearly all triangles
    bool in = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float w = poly[k].c[3], gw = kGuard * w;
        in = in && poly[k].c[2] >= -w && fabsf(poly[k].c[0]) <= gw && fabsf(poly[k].c[1]) <= gw;
    }
    if (!in) {
        uint32_t all_out = 0x1f;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            uint32_t o = 0;
#pragma unroll
            for (int p = 0; p < 5; ++p)
                o |= (clip_dist(poly[k], p) >= 0.0f ? 0u : 1u) << p;
            all_out &= o;
        }
        return all_out ? kTriOut : kTriClip;
    }
    // All vertices in front of the near plane (w > 0): reject against the
    // scissor rectangle in clip space with a one-pixel margin.
    const float lo_x = scis.x, hi_x = scis.y, lo_y = scis.z, hi_y = scis.w;
    bool lx = true, hx = true, ly = true, hy = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float w = poly[k].c[3];
        lx = lx && (poly[k].c[0] < lo_x * w);
        hx = hx && (poly[k].c[0] > hi_x * w);
        ly = ly && (poly[k].c[1] < lo_y * w);
        hy = hy && (poly[k].c[1] > hi_y * w);
    }
    return lx || hx || ly || hy ? kTriOut : kTriIn;
}

// Orders the LDS accesses of a wavefront's lanes (its LDS operations are
// performed in order, so only the compiler has to keep them so).
__device__ static inline void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sutherland-Hodgman of one triangle by one wavefront: lane i holds vertex i
// of the polygon (at most kClipMax).  Per plane every lane finds its edge to
// the next vertex (the last one wraps to vertex 0), emits its vertex when
// inside and the intersection when the edge crosses, at offsets from two
// ballots, and the new polygon is gathered back through the wavefront's LDS
// buffer lp.  The arithmetic and the vertex order are those of the
// sequential walk (the oracle's clipper), vertex by vertex, and the overflow
// test is its test before the last vertex, where the count is largest.
// Returns the polygon's vertex count (0: nothing left, or dropped with
// *overflow set).
__device__ static inline int clip_polygon_wave(CV4 &v, CV4 *lp, uint32_t *overflow)
{
    const int lane = (int)(threadIdx.x & 63);
    const uint64_t lt = (1ull << lane) - 1ull;
    int n = 3;
    for (int plane = 0; plane < 5; ++plane) {
        const bool act = lane < n;
        const float d = act ? clip_dist(v, plane) : 0.0f;
        const bool in = act && d >= 0.0f;
        const int nin = __popcll(__ballot(in));
        if (nin == n)
            continue;
        if (nin == 0)
            return 0;
        const int nx = lane + 1 >= n ? 0 : lane + 1;
        CV4 q;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            q.c[c] = __shfl(v.c[c], nx, 64);
        const float dq = __shfl(d, nx, 64);
        const bool inq = dq >= 0.0f;
        const bool cross = act && in != inq;
        const uint64_t b1 = __ballot(in), b2 = __ballot(cross);
        const int off = __popcll(b1 & lt) + __popcll(b2 & lt);
        const int m = __popcll(b1) + __popcll(b2);
        const int last = (int)((b1 >> (n - 1)) & 1ull) + (int)((b2 >> (n - 1)) & 1ull);
        if (m - last + 2 > kClipMax) {
            if (lane == 0)
                atomicOr(overflow, 1u);
            return 0;
        }
        if (in)
            lp[off] = v;
        if (cross) {
            const CV4 &A = in ? v : q;
            const CV4 &B = in ? q : v;
            float da = in ? d : dq, db = in ? dq : d;
            float t = da / (da - db);
            CV4 r;
            for (int c = 0; c < 4; ++c)
                r.c[c] = A.c[c] + t * (B.c[c] - A.c[c]);
            lp[off + (in ? 1 : 0)] = r;
        }
        wave_lds_sync();
        n = m;
        if (lane < n)
            v = lp[lane];
        wave_lds_sync();
    }
    return n;
}

// The fan triangle (0, lane, lane + 1) of the clipped polygon, snapped;
// false in the lanes that hold none.  Every lane of the wavefront calls it.
__device__ static inline bool clip_fan(const CV4 &v, int n, float halfW, SV &a, SV &b, SV &c)
{
    const int lane = (int)(threadIdx.x & 63);
    b = project(v, halfW);
    a.x = __shfl(b.x, 0, 64);
    a.y = __shfl(b.y, 0, 64);
    a.z = __shfl(b.z, 0, 64);
    const int nx = lane + 1 < 64 ? lane + 1 : lane;
    c.x = __shfl(b.x, nx, 64);
    c.y = __shfl(b.y, nx, 64);
    c.z = __shfl(b.z, nx, 64);
    return lane >= 1 && lane + 1 < n;
}

// Segmented sums over the runs of equal id in a wavefront, on DPP lane
// moves (no LDS round trip).  A run starts where the id differs from the
// previous lane's; ss = the lane of the last run start at or before this
// lane, read off the wavefront's mask of run starts.  The sums are a
// Hillis-Steele scan inside each row of 16 lanes (row_shr 1, 2, 4, 8; a lane
// adds lane - d only if lane - d >= ss, so only its own run), then the
// row_bcast steps carry the sum at lane 15 / 47 into rows 1 / 3 and at lane 31
// into rows 2 and 3, again only into lanes whose run began at or before that
// lane.  Lanes a DPP move cannot read from give 0.  Returns true in the last
// lane of each run with an id (id != 0), which then holds the run's sums of f
// (and of c when with_c).  Every lane of the wavefront must call it.
template <int CTRL, int ROWS> __device__ static inline float dpp_f(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xF, true));
}
template <int CTRL, int ROWS> __device__ static inline uint32_t dpp_u(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, true);
}

template <int CTRL, int ROWS>
__device__ static inline void seg_step(float &f, uint32_t &c, bool take, bool with_c)
{
    const float fo = dpp_f<CTRL, ROWS>(f);
    f += take ? fo : 0.0f;
    if (with_c) {
        const uint32_t co = dpp_u<CTRL, ROWS>(c);
        c += take ? co : 0u;
    }
}

// The segmented scan itself, for the wavefront's mask hm of segment starts
// (lane 0 must be one): f (and c) become the sums over the lanes from the
// segment's start up to this lane.
__device__ static inline void seg_scan(uint64_t hm, float &f, uint32_t &c, bool with_c)
{
    const int lane = (int)(threadIdx.x & 63);
    const int ss = 63 - __clzll(hm & ((2ull << lane) - 1ull));
    seg_step<0x111, 0xF>(f, c, lane - 1 >= ss, with_c); // row_shr:1
    seg_step<0x112, 0xF>(f, c, lane - 2 >= ss, with_c); // row_shr:2
    seg_step<0x114, 0xF>(f, c, lane - 4 >= ss, with_c); // row_shr:4
    seg_step<0x118, 0xF>(f, c, lane - 8 >= ss, with_c); // row_shr:8
    seg_step<0x142, 0xA>(f, c, (lane & ~15) - 1 >= ss, with_c); // row_bcast:15
    seg_step<0x143, 0xC>(f, c, 31 >= ss, with_c);               // row_bcast:31
}

__device__ static inline bool wave_runs(uint32_t id, float &f, uint32_t &c, bool with_c)
{
    const int lane = (int)(threadIdx.x & 63);
    const uint32_t pid = dpp_u<0x138, 0xF>(id); // wave_shr:1
    const bool head = lane == 0 || pid != id;
    const uint64_t hm = __ballot(head);
    seg_scan(hm, f, c, with_c);
    const bool tail = lane == 63 || ((hm >> (lane + 1)) & 1ull);
    return tail && id != 0;
}

// F row entries are id - 1 - pbase for ids in [pbase + 1, pbase + rowlen]
// (pbase: first patch of the shooter's scene in a packed launch, else 0).
// Deterministic mode: a run's sum in fixed point, units of 2^-52 (exact for
// sums from 2^-29 up, well below 1e-7 relative under that; F < 4096), added
// with 64-bit integer atomics, so the total does not depend on their order.
__device__ static inline unsigned long long fixed52(float f)
{
    return __float2ull_rn(f * 4503599627370496.0f);
}

// Wave-level ProcessHemicube on 64 consecutive texels of one shooter's
// hemicube hi (any grouping of equal ids gives the same sums; consecutive
// texels make runs long): each run's sum is added by its last lane.  FQ: the
// runs go to the fixed-point rows ffq instead of ff.  Every lane of the
// wavefront must call it.
template <bool FQ>
__device__ static inline void reduce_wave(uint32_t id, float f, uint32_t hi, uint32_t pbase,
                                          uint32_t rowlen, float *__restrict__ ff,
                                          unsigned long long *__restrict__ ffq,
                                          uint32_t *__restrict__ hits,
                                          uint32_t *__restrict__ counters)
{
    uint32_t c = id ? 1u : 0u;
    if (wave_runs(id, f, c, hits != nullptr)) {
        const uint32_t p = id - 1 - pbase;
        if (p < rowlen) {
            const size_t o = (size_t)hi * rowlen + p;
            if constexpr (FQ)
                atomicAdd(&ffq[o], fixed52(f));
            else
                atomicAdd(&ff[o], f);
            if (hits)
                atomicAdd(&hits[o], c);
        } else {
            atomicAdd(&counters[kCntUnknown], 1u);
        }
    }
}

constexpr uint32_t kTileThreads = 256; // k_tile_raster's workgroup size
constexpr uint32_t kTileTable = 256;   // its LDS table of F entries (one slot per thread)
static_assert(kTileTable == kTileThreads, "the table is cleared and flushed one slot per thread");

// The tile kernel's F sums go through a per-workgroup LDS table (hk: F-row
// index + 1, 0 = free; hs, hc: the sums of f and of the texel counts), which
// is added to the global row once at the end, so that a tile adds a patch it
// sees to the row once rather than once per run: with every run straight to
// the row a pass took 10 to 19 % longer.  A run whose slot another patch holds
// does go there.  (A pass of 64 shooters over 200,000 triangles: 16 probes
// 327 us, 2 probes 324, this one 322; 1,024 slots for the tiles of more than
// 256 records took as long to clear and flush as they saved.)
__device__ static inline void table_add(uint32_t p, float f, uint32_t c, bool with_c,
                                        uint32_t *hk, float *hs, uint32_t *hc,
                                        float *__restrict__ frow, uint32_t *__restrict__ hrow,
                                        uint32_t *__restrict__ fflag, uint32_t fstride)
{
    const uint32_t key = p + 1;
    const uint32_t h = (key * 2654435761u) >> 24; // kTileTable = 2^8
    uint32_t k = hk[h];
    if (k == 0u)
        k = atomicCAS(&hk[h], 0u, key);
    if (k == 0u || k == key) {
        atomicAdd(&hs[h], f);
        if (with_c)
            atomicAdd(&hc[h], c);
        return;
    }
    atomicAdd(&frow[p], f);
    if (with_c)
        atomicAdd(&hrow[p], c);
    if (fflag)
        fflag[(p >> 6) * fstride] = 1u;
}

// One run (id, sums f and c) of a shooter's hemicube: id 0 (background) adds
// nothing; F entries are id - 1 - pbase (pbase: first patch of the shooter's
// scene in a packed launch, else 0); an id beyond the row is counted (once
// per run, Main.cpp:1259-1262) and skipped.
__device__ static inline void run_add(uint32_t id, float f, uint32_t c, uint32_t pbase,
                                      uint32_t rowlen, bool with_c, uint32_t *hk, float *hs,
                                      uint32_t *hc, float *__restrict__ frow,
                                      uint32_t *__restrict__ hrow, uint32_t *__restrict__ counters,
                                      uint32_t *__restrict__ fflag, uint32_t fstride)
{
    if (!id)
        return;
    const uint32_t p = id - 1 - pbase;
    if (p >= rowlen) {
        atomicAdd(&counters[kCntUnknown], 1u);
        return;
    }
    table_add(p, f, c, with_c, hk, hs, hc, frow, hrow, fflag, fstride);
}

// ProcessHemicube on 256 consecutive texels of one shooter's hemicube, 4
// consecutive texels per lane (ids q, ΔFF f, f = 0 where q = 0).  A run of
// equal ids inside a lane is summed in the lane; a run that reaches a lane's
// last texel (its tail run) may go on into the next lanes, so the tail runs
// are summed across lanes by the segmented scan (a segment starts at a lane
// whose tail run starts inside it, or whose first id differs from the
// previous lane's last).  Every run is added once: a lane adds its middle
// runs, its first run unless that is its tail run (plus the scanned sum the
// previous lane carries into it), and its tail run's scanned sum when the
// next lane does not go on with it.  Any grouping of equal ids gives the
// same F sums.  Every lane of the wavefront must call it.
// emit(id, f, c) adds one run.
template <typename Emit>
__device__ static inline void reduce_quad(const uint32_t (&q)[4], const float (&f)[4], bool with_c,
                                          Emit &&emit)
{
    const int lane = (int)(threadIdx.x & 63);
    const bool b1 = q[1] != q[0], b2 = q[2] != q[1], b3 = q[3] != q[2];
    const bool whole = !(b1 || b2 || b3);
    // first run [0, first boundary), tail run [last boundary, 4)
    float fs = f[0];
    uint32_t fc = 1;
    if (!b1) {
        fs += f[1];
        ++fc;
        if (!b2) {
            fs += f[2];
            ++fc;
            if (!b3) {
                fs += f[3];
                ++fc;
            }
        }
    }
    float ts = f[3];
    uint32_t tc = 1;
    if (!b3) {
        ts += f[2];
        ++tc;
        if (!b2) {
            ts += f[1];
            ++tc;
            if (!b1) {
                ts += f[0];
                ++tc;
            }
        }
    }
    // middle runs: [1, 2) or [1, 3), and [2, 3)
    if (b1 && (b2 || b3))
        emit(q[1], b2 ? f[1] : f[1] + f[2], b2 ? 1u : 2u);
    if (b2 && b3)
        emit(q[2], f[2], 1u);
    const uint32_t prev3 = dpp_u<0x138, 0xF>(q[3]); // wave_shr:1: lane - 1's last id
    const uint32_t next0 = dpp_u<0x130, 0xF>(q[0]); // wave_shl:1: lane + 1's first id
    const bool cont_prev = lane > 0 && prev3 == q[0];
    const bool cont_next = lane < 63 && next0 == q[3];
    seg_scan(__ballot(!whole || !cont_prev), ts, tc, with_c);
    const float sp = dpp_f<0x138, 0xF>(ts); // the previous lane's scanned tail sum
    const uint32_t cp = with_c ? dpp_u<0x138, 0xF>(tc) : 0u;
    if (!whole)
        emit(q[0], cont_prev ? fs + sp : fs, cont_prev ? fc + cp : fc);
    if (!cont_next)
        emit(q[3], ts, tc);
}

__device__ static inline void draw_span(const RasterRec &r, const Edges &e, int32_t vpx,
                                        int32_t vpy, int32_t ax0, int32_t ay0, uint32_t w,
                                        uint32_t area, uint32_t p0, uint32_t step, int32_t ox,
                                        int32_t oy, uint32_t tshift, uint64_t *tk)
{
    for (uint32_t p = p0; p < area; p += step) {
        int32_t tx = ax0 + (int32_t)(p % w), ty = ay0 + (int32_t)(p / w);
        uint64_t key = frag_key(e, r, tx - vpx, ty - vpy);
        uint32_t pp = (uint32_t)((ty - oy) << tshift) + (uint32_t)(tx - ox);
        if (key)
            atomicMin((unsigned long long *)&tk[pp], (unsigned long long)key);
    }
}

// The whole wavefront draws one record's pixels [ax0,ax1] x [ay0,ay1]
// (texels, at most one tile) in 8 x 8 blocks, lane = (lane & 7, lane >> 3)
// inside the block.  The edge values start from the exact 64-bit evaluation
// at the lane's first pixel and step by 8 pixels with 64-bit adds, so every
// inside test equals frag_key's; depth is frag_key's expression.
__device__ static inline void draw_wave(const RasterRec &r, const Edges &e, int32_t vpx,
                                        int32_t vpy, int32_t ax0, int32_t ax1, int32_t ay0,
                                        int32_t ay1, int32_t ox, int32_t oy, uint32_t tshift,
                                        uint64_t *tk)
{
    const int32_t lane = (int32_t)(threadIdx.x & 63), lx = lane & 7, ly = lane >> 3;
    const int32_t px0 = (ax0 - vpx + lx) * kSub + kSub / 2, py0 = (ay0 - vpy + ly) * kSub + kSub / 2;
    int64_t er[3], sx[3], sy[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        er[k] = (int64_t)e.A[k] * px0 + (int64_t)e.B[k] * py0 + e.C[k] + e.bias[k];
        sx[k] = (int64_t)e.A[k] * (8 * kSub);
        sy[k] = (int64_t)e.B[k] * (8 * kSub);
    }
    for (int32_t by = 0; ay0 + by <= ay1; by += 8) {
        const int32_t ty = ay0 + by + ly;
        const int32_t py = py0 + by * kSub;
        const float zr = fmaf(r.dzdy, (float)(py - r.y[0]), r.z0);
        int64_t e0 = er[0], e1 = er[1], e2 = er[2];
        for (int32_t bx = 0; ax0 + bx <= ax1; bx += 8) {
            const int32_t tx = ax0 + bx + lx;
            if (tx <= ax1 && ty <= ay1 && e0 > 0 && e1 > 0 && e2 > 0) {
                const int32_t px = px0 + bx * kSub;
                float z = fmaf(r.dzdx, (float)(px - r.x[0]), zr);
                if (!(z > 0.0f))
                    z = 0.0f;
                if (z < 1.0f) {
                    uint64_t key = ((uint64_t)__float_as_uint(z) << 32) | r.id;
                    uint32_t pp = (uint32_t)((ty - oy) << tshift) + (uint32_t)(tx - ox);
                    atomicMin((unsigned long long *)&tk[pp], (unsigned long long)key);
                }
            }
            e0 += sx[0];
            e1 += sx[1];
            e2 += sx[2];
        }
        er[0] += sy[0];
        er[1] += sy[1];
        er[2] += sy[2];
    }
}

// 1 for an edge that owns its pixels (A > 0, or A == 0 and B < 0), else 0:
// the sign of B - 2^16 A, for |A| and |B| below 2^15.
__device__ static inline int32_t edge_bias(int32_t A, int32_t B)
{
    return (int32_t)((uint32_t)(B - (int32_t)((uint32_t)A << 16)) >> 31);
}

// draw_wave for a record whose snapped vertices span at most 96 pixels in x
// and in y (kWave32Span subpixels): every pixel a lane visits, the 8 x 8
// blocks' overshoot past the bbox included, lies within 16 pixels of the
// vertices' box, so |A (px - x_k)| + |B (py - y_k)| < 2 * 2^15 * 2^15 = 2^31
// and the edge functions step in int32 (E + bias - 1 >= 0, exactly the
// 64-bit test).  Depth is frag_key's expression.
constexpr int32_t kWave32Span = 96 * kSub;

__device__ static inline void draw_wave32(const RasterRec &r, int32_t vpx, int32_t vpy,
                                          int32_t ax0, int32_t ax1, int32_t ay0, int32_t ay1,
                                          int32_t ox, int32_t oy, uint32_t tshift, uint64_t *tk)
{
    const int32_t lane = (int32_t)(threadIdx.x & 63), lx = lane & 7, ly = lane >> 3;
    const int32_t px0 = (ax0 - vpx + lx) * kSub + kSub / 2, py0 = (ay0 - vpy + ly) * kSub + kSub / 2;
    int32_t er[3], sx[3], sy[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int q = k == 2 ? 0 : k + 1;
        const int32_t A = r.y[k] - r.y[q], B = r.x[q] - r.x[k];
        er[k] = __mul24(A, px0 - r.x[k]) + __mul24(B, py0 - r.y[k]) + edge_bias(A, B) - 1;
        sx[k] = A * (8 * kSub);
        sy[k] = B * (8 * kSub);
    }
    for (int32_t by = 0; ay0 + by <= ay1; by += 8) {
        const int32_t ty = ay0 + by + ly;
        const int32_t py = py0 + by * kSub;
        const float zr = fmaf(r.dzdy, (float)(py - r.y[0]), r.z0);
        int32_t e0 = er[0], e1 = er[1], e2 = er[2];
        for (int32_t bx = 0; ax0 + bx <= ax1; bx += 8) {
            const int32_t tx = ax0 + bx + lx;
            if (tx <= ax1 && ty <= ay1 && (e0 | e1 | e2) >= 0) {
                const int32_t px = px0 + bx * kSub;
                float z = fmaf(r.dzdx, (float)(px - r.x[0]), zr);
                if (!(z > 0.0f))
                    z = 0.0f;
                // (no less than the cleared texel's key where z >= 1)
                const uint64_t key = ((uint64_t)__float_as_uint(z) << 32) | r.id;
                const uint32_t pp = (uint32_t)((ty - oy) << tshift) + (uint32_t)(tx - ox);
                atomicMin((unsigned long long *)&tk[pp], (unsigned long long)key);
            }
            e0 += sx[0];
            e1 += sx[1];
            e2 += sx[2];
        }
        er[0] += sy[0];
        er[1] += sy[1];
        er[2] += sy[2];
    }
}

// One lane draws a record's pixels [ax0,ax1] x [ay0,ay1] (texels).  When the
// snapped vertices span less than 64 pixels every edge value inside the bbox
// fits in int32, so the edge functions are stepped with 32-bit adds; the
// values equal the 64-bit evaluation exactly.  Depth is the same
// fmaf(dzdx, px-x0, fmaf(dzdy, py-y0, z0)) with the inner term per row;
// (float)(px - x0) is stepped by 256.0f, exact because every value is an
// integer below 2^24.  Every bbox pixel issues its ds_min_u64, which ran
// faster than branching around the atomic: outside the triangle with a key of
// all ones above, beyond the depth range (z >= 1) as it is, both no less than
// the cleared texel's (kClearKey: depth 1, id 0).  The edges' products are of
// differences below 2^15, for the full-rate 24-bit multiply.
// Rows ay0 + ph, ay0 + ph + nph, ... of the bbox (row phase ph of nph; the
// caller's other lanes draw the other phases).
constexpr int32_t kLane32Span = (64 << 8) - 1;

__device__ static inline bool span_within(const RasterRec &r, int32_t lim)
{
    const int32_t xspan = max(r.x[0], max(r.x[1], r.x[2])) - min(r.x[0], min(r.x[1], r.x[2]));
    const int32_t yspan = max(r.y[0], max(r.y[1], r.y[2])) - min(r.y[0], min(r.y[1], r.y[2]));
    return xspan <= lim && yspan <= lim;
}

__device__ static inline void draw_lane32(const RasterRec &r, int32_t vpx, int32_t vpy,
                                          int32_t ax0, int32_t ax1, int32_t ay0, int32_t ay1,
                                          int32_t ox, int32_t oy, uint32_t tshift, uint64_t *tk,
                                          uint32_t ph, uint32_t nph)
{
    ay0 += (int32_t)ph;
    if (ay0 > ay1)
        return;
    const int32_t px0 = (ax0 - vpx) * kSub + kSub / 2, py0 = (ay0 - vpy) * kSub + kSub / 2;
    int32_t v[3], dA[3], dB[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        int q = k == 2 ? 0 : k + 1;
        const int32_t A = r.y[k] - r.y[q], B = r.x[q] - r.x[k];
        // E(p) = A (p.x - x_k) + B (p.y - y_k); inside iff E + bias - 1 >= 0
        v[k] = __mul24(A, px0 - r.x[k]) + __mul24(B, py0 - r.y[k]) + edge_bias(A, B) - 1;
        dA[k] = A * kSub;
        dB[k] = B * kSub * (int32_t)nph;
    }
    int32_t py = py0;
    const uint32_t w = (uint32_t)(ax1 - ax0 + 1), rstride = nph << tshift;
    const float fx0 = (float)(px0 - r.x[0]);
    uint32_t prow = (uint32_t)((ay0 - oy) << tshift) + (uint32_t)(ax0 - ox);
    for (int32_t ty = ay0; ty <= ay1;
         ty += (int32_t)nph, py += kSub * (int32_t)nph, prow += rstride) {
        float zr = fmaf(r.dzdy, (float)(py - r.y[0]), r.z0);
        int32_t e0 = v[0], e1 = v[1], e2 = v[2];
        float fx = fx0;
        unsigned long long *p = (unsigned long long *)(tk + prow), *pend = p + w;
        for (; p != pend; ++p, fx += 256.0f) {
            float z = fmaf(r.dzdx, fx, zr);
            if (!(z > 0.0f))
                z = 0.0f;
            const uint32_t out = (uint32_t)((e0 | e1 | e2) >> 31);
            atomicMin(p, (unsigned long long)(((uint64_t)(__float_as_uint(z) | out) << 32) | r.id));
            e0 += dA[0];
            e1 += dA[1];
            e2 += dA[2];
        }
        v[0] += dB[0];
        v[1] += dB[1];
        v[2] += dB[2];
    }
}

__device__ static inline void draw_lane(const RasterRec &r, bool narrow, int32_t vpx, int32_t vpy,
                                        int32_t ax0, int32_t ax1, int32_t ay0, int32_t ay1,
                                        int32_t ox, int32_t oy, uint32_t tshift, uint64_t *tk,
                                        uint32_t ph, uint32_t nph)
{
    if (!narrow) {
        if (ph != 0)
            return; // phase 0 draws these (rare) records whole
        Edges e;
        make_edges(r.x, r.y, e);
        uint32_t w = (uint32_t)(ax1 - ax0 + 1), area = w * (uint32_t)(ay1 - ay0 + 1);
        draw_span(r, e, vpx, vpy, ax0, ay0, w, area, 0, 1, ox, oy, tshift, tk);
        return;
    }
    draw_lane32(r, vpx, vpy, ax0, ax1, ay0, ay1, ox, oy, tshift, tk, ph, nph);
}

} // namespace rad
