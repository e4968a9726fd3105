// rad_kernels.hip - CDNA4 (gfx950) kernels of the hemicube shooting path.
//
// Compiled with -ffp-contract=off: the camera, clipping, snapping and depth
// arithmetic below is written operation by operation so the item buffer is
// reproducible bit for bit on any IEEE-754 implementation of the same
// sequence (fmaf only where written).  Division and sqrt are HIP's
// correctly-rounded defaults.
//
// Kernels (one pass over K shooters):
//   k_select_* / k_topk*   shooter selection (+ FP64 residual partial sums)
//   k_prepare_clear  dB snapshot and the five face MVPs per shooter; bin
//                  counts and pass counters reset, F rows zeroed unless the
//                  previous shoot left them zero
//   k_raster_setup one lane per (triangle, shooter) over the five faces:
//                  cull, transform, snap; records into the tiles' lists
//   k_order_clip   the launch order of the tiles; the few triangle-faces that
//                  cross the near plane or the guard band
//   k_tile_raster  one workgroup per (shooter, tile): depth test in LDS, then
//                  the tile's item buffer out or ProcessHemicube fused
//   k_reduce       ProcessHemicube over a whole item buffer (wave-level
//                  run-length reduction into form factors and hit counts)
//   k_shoot        energy shooting into unshot RGB, emitter update; zeroes
//                  the F entries it reads
//
// Depth test: each texel holds a 64-bit key (float depth bits << 32 | id).
// atomicMin of keys gives the nearest fragment, ties to the smallest id,
// which is the fragment GL_LESS keeps when triangles are drawn in id order
// (Main.cpp:1104, DrawPatchLook Main.cpp:720).
#include "rad_internal.h"
#include "rad_prepare.h"
#include "rad_raster.h"
#include "rad_topk.h"

#include <hip/hip_runtime.h>

namespace rad {

// ------------------------------------------------------------------ ΔFF table
// FormFactors.cpp:23-67 (values) and 280-314 (cross layout), one thread per
// texel of one TEX_W x TEX_H copy.
__device__ static float dff_top(int n, int x, int y)
{
    float hpw = 1.0f / n;
    float pa = 2.0f / n;
    pa = pa * pa;
    float dx = ((x - n / 2) / (n / 2.0f)) + hpw;
    float dy = ((y - n / 2) / (n / 2.0f)) + hpw;
    float f = (dx * dx + dy * dy + 1);
    f = f * (f * 3.1415926535897932384626433832795028841931f);
    return pa / f;
}

__device__ static float dff_side(int n, int x, int y)
{
    float hpw = 1.0f / n;
    float pa = 2.0f / n;
    pa = pa * pa;
    float dx = (x - n / 2) / (n / 2.0f) + hpw;
    float dy = (n / 2 - 1 - y) / (n / 2.0f) + hpw;
    float f = (dx * dx + dy * dy + 1);
    f = f * (f * 3.1415926535897932384626433832795028841931f);
    return (pa * (dy + hpw)) / f;
}

__global__ void k_dff(uint32_t W, uint32_t TW, uint32_t RES, float *out)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= RES)
        return;
    uint32_t x = i % TW, y = i / TW, H = W;
    int n = (int)W;
    float v = 0.0f;
    // side[idx] with idx = xs + ys*W  ->  (xs, ys) = (idx % W, idx / W)
    if (x >= W / 2 && x < W + W / 2 && y < H) {
        v = dff_top(n, (int)(x - W / 2), (int)y);
    } else if (x < W / 2 && y < H) {
        uint32_t idx = (H / 2 - x) * W - y - 1;
        v = dff_side(n, (int)(idx % W), (int)(idx / W));
    } else if (x >= W + W / 2 && y < H) {
        uint32_t idx = (x - (W + W / 2)) * W + y;
        v = dff_side(n, (int)(idx % W), (int)(idx / W));
    } else if (x < W && y >= H) {
        uint32_t idx = (y - H) * W + x;
        v = dff_side(n, (int)(idx % W), (int)(idx / W));
    } else if (x >= W && y >= H) {
        uint32_t idx = ((H / 2 - 1) - (y - H)) * W + (x - W);
        v = dff_side(n, (int)(idx % W), (int)(idx / W));
    }
    out[i] = v;
}

void launch_dff(const Geometry &g, float *dff, hipStream_t st)
{
    k_dff<<<(g.RES + 255) / 256, 256, 0, st>>>(g.W, g.TW, g.RES, dff);
}

__global__ void k_prepare(uint32_t K, const uint32_t *__restrict__ shooters,
                          const uint32_t *__restrict__ nshoot, const float *__restrict__ frames,
                          const float *__restrict__ unshot, float *__restrict__ snap,
                          float *__restrict__ mvp)
{
    prepare_item(blockIdx.x * blockDim.x + threadIdx.x, K, shooters, nshoot, frames, unshot, snap,
                 mvp, nullptr);
}

void launch_prepare(const Geometry &g, uint32_t K, const uint32_t *shooters,
                    const uint32_t *nshoot, const float *frames, const float *unshot,
                    float *snap, float *mvp, hipStream_t st)
{
    (void)g;
    uint32_t n = K * 5;
    k_prepare<<<(n + 63) / 64, 64, 0, st>>>(K, shooters, nshoot, frames, unshot, snap, mvp);
}

// --------------------------------------------------------------------- clear
__global__ void k_clear(uint32_t *__restrict__ bin_count, size_t nbins, float *__restrict__ ff,
                        uint32_t *__restrict__ hits, size_t nff, uint32_t *__restrict__ counters)
{
    clear_range((size_t)blockIdx.x * blockDim.x + threadIdx.x, (size_t)gridDim.x * blockDim.x,
                bin_count, nbins, ff, hits, nff, counters);
}

// k_prepare and k_clear of a pass in one launch (the first np workgroups
// prepare, the others clear): both are small, so one launch saves a kernel's
// start-up and drain.
// Pass gate (the loop condition of Main.cpp:1137): once the stop test of a
// previous shoot has fired (ctl[kCtlStop]), the pass selects nobody: nshoot
// is set to 0 for the later kernels of the pass, and the prepare items of
// this launch return at once (they read the flag themselves rather than the
// nshoot this launch writes).
__global__ __launch_bounds__(256) void k_prepare_clear(
    uint32_t np, uint32_t K, const uint32_t *__restrict__ shooters,
    uint32_t *__restrict__ nshoot, const float *__restrict__ frames,
    const float *__restrict__ unshot, float *__restrict__ snap, float *__restrict__ mvp,
    uint32_t *__restrict__ bin_count, size_t nbins, float *__restrict__ ff,
    uint32_t *__restrict__ hits, size_t nff, uint32_t *__restrict__ counters,
    const uint32_t *__restrict__ ctl)
{
    if (blockIdx.x < np) {
        prepare_item(blockIdx.x * blockDim.x + threadIdx.x, K, shooters, nshoot, frames, unshot,
                     snap, mvp, ctl);
        return;
    }
    if (ctl && blockIdx.x == np && threadIdx.x == 0 && ctl[kCtlStop])
        *nshoot = 0u;
    clear_range((size_t)(blockIdx.x - np) * blockDim.x + threadIdx.x,
                (size_t)(gridDim.x - np) * blockDim.x, bin_count, nbins, ff, hits, nff, counters);
}

void launch_prepare_clear(uint32_t K, const uint32_t *shooters, uint32_t *nshoot,
                          const float *frames, const float *unshot, float *snap, float *mvp,
                          uint32_t *bin_count, uint32_t ntiles, float *ff, uint32_t *hits,
                          uint32_t ff_rows, uint32_t rowlen, uint32_t *counters,
                          const uint32_t *ctl, hipStream_t st)
{
    const uint32_t np = (K * 5 + 255) / 256;
    size_t nbins = (size_t)K * ntiles, nff = ff || hits ? (size_t)ff_rows * rowlen : 0;
    size_t n = nbins > nff ? nbins : nff;
    size_t blocks = (n + 255) / 256;
    if (blocks > 8192)
        blocks = 8192;
    if (blocks == 0)
        blocks = 1;
    k_prepare_clear<<<(unsigned)(np + blocks), 256, 0, st>>>(np, K, shooters, nshoot, frames,
                                                            unshot, snap, mvp, bin_count, nbins,
                                                            ff, hits, nff, counters, ctl);
}

void launch_clear(uint32_t K, uint32_t *bin_count, uint32_t ntiles, float *ff, uint32_t *hits,
                  uint32_t ff_rows, uint32_t rowlen, uint32_t *counters,
                  hipStream_t st)
{
    // ff null: the F rows are known to be zero (the last shoot cleared them)
    size_t nbins = (size_t)K * ntiles, nff = ff || hits ? (size_t)ff_rows * rowlen : 0;
    size_t n = nbins > nff ? nbins : nff;
    size_t blocks = (n + 255) / 256;
    if (blocks > 8192)
        blocks = 8192;
    if (blocks == 0)
        blocks = 1;
    k_clear<<<(unsigned)blocks, 256, 0, st>>>(bin_count, nbins, ff, hits, nff, counters);
}

// ---------------------------------------------------------------- rasterizer
// Sort-middle rasterizer.
//  k_raster_setup  one lane per (triangle, shooter), looping over the five
//                  faces: cull, transform, snap; every surviving triangle
//                  becomes a RasterRec and is listed in the bins of the
//                  screen tiles its bbox touches
//  k_order_clip    the bins by size, for the launch order of the tiles; the
//                  triangles to clip, as records of their own
//  k_tile_raster   one workgroup per tile: depth test in LDS with 64-bit
//                  atomicMin, then either writes the tile's ids and depths
//                  (item buffer out) or reduces it into form factors
//                  (ProcessHemicube fused)
struct BinCtx {
    RasterRec *recs;       // block regions of kRecsPerBlock, then the spill region
    uint64_t *bbox;        // texel bbox of each record slot (x0 | y0 << 16 | x1 << 32 | y1 << 48)
    uint32_t *bin_count;   // K * ntiles
    uint32_t *counters;
    uint32_t *lnrec;       // LDS: records in this block's region
    uint32_t *lcnt;        // LDS: per-tile record counts of this block
    uint32_t region;       // first record of this block's region
    uint32_t spill_base, spill_cap;
    uint2 *clipq;          // (triangle, shooter * 8 + face) jobs that need clipping
    uint32_t clip_cap;
    uint32_t ntx, ntiles, tshift; // tiles per row, per hemicube, log2(tile side)
    uint32_t *list;        // bin_cap entries (record slots) per bin
    uint32_t bin_cap;
};

// Record r into the list of a bin at place pos (bins hold bin_cap entries;
// the tile kernel draws a fuller one from the records themselves).
__device__ static inline void list_put(const BinCtx &bc, uint32_t s, uint32_t tile, uint32_t pos,
                                       uint32_t r)
{
    if (pos < bc.bin_cap)
        bc.list[((size_t)s * bc.ntiles + tile) * bc.bin_cap + pos] = r;
}

// A record of a triangle and the tiles [g0, g1] x [h0, h1] of its texel bbox.
struct Placed {
    uint32_t r, g0, g1, h0, h1;
};

// The record of a snapped triangle (face-local coordinates) into the block's
// region or, when that is full (or for a clipped triangle), into the spill
// region: 0 no record, 1 region, 2 spill.
__device__ static inline int place_tri(const SV &a, const SV &b, const SV &c, uint32_t id,
                                       const FaceView &fv, uint32_t s, int face, const BinCtx &bc,
                                       Placed &p)
{
    int64_t area2;
    int32_t ix0, iy0, ix1, iy1;
    if (!snapped_bbox(a, b, c, fv.sx0, fv.sy0, fv.sx1, fv.sy1, area2, ix0, iy0, ix1, iy1))
        return 0;
    uint32_t slot = bc.lnrec ? atomicAdd(bc.lnrec, 1u) : kRecsPerBlock;
    bool local = slot < kRecsPerBlock;
    if (local) {
        p.r = bc.region + slot;
    } else {
        if (bc.lnrec)
            atomicSub(bc.lnrec, 1u);
        uint32_t q = atomicAdd(&bc.counters[kCntSpill], 1u);
        if (q >= bc.spill_cap) {
            atomicOr(&bc.counters[kCntOverflow], 1u);
            return 0;
        }
        p.r = bc.spill_base + q;
    }
    RasterRec rr;
    make_record(a, b, c, area2, id, rr);
    rr.sf = s << 2 | (span_within(rr, kLane32Span) ? kSpanLane : 0u) |
            (span_within(rr, kWave32Span) ? kSpanWave : 0u);
    rr.vp = (uint32_t)(fv.vpx & 0xFFFF) | (uint32_t)fv.vpy << 16;
    // bbox in texel coordinates of the hemicube slab
    int32_t tx0 = fv.vpx + ix0, tx1 = fv.vpx + ix1, ty0 = fv.vpy + iy0, ty1 = fv.vpy + iy1;
    bc.recs[p.r] = rr;
    bc.bbox[p.r] = (uint64_t)(uint16_t)tx0 | ((uint64_t)(uint16_t)ty0 << 16) |
                   ((uint64_t)(uint16_t)tx1 << 32) | ((uint64_t)(uint16_t)ty1 << 48);
    p.g0 = (uint32_t)tx0 >> bc.tshift;
    p.g1 = (uint32_t)tx1 >> bc.tshift;
    p.h0 = (uint32_t)ty0 >> bc.tshift;
    p.h1 = (uint32_t)ty1 >> bc.tshift;
    return local ? 1 : 2;
}

// A spill record straight into the list of tile b of slot s.
__device__ static inline void bin_spilled(const BinCtx &bc, uint32_t s, uint32_t b, uint32_t r)
{
    const uint32_t pos = atomicAdd(&bc.bin_count[(size_t)s * bc.ntiles + b], 1u);
    if (pos & kBinSeen) // k_order_clip has summed the counts
        atomicAdd(&bc.counters[kCntEntries], 1u);
    list_put(bc, s, b, pos & ~kBinSeen, r);
}

// place_tri, and a region record counted in the LDS histogram of its tiles.
__device__ static void emit_tri(const SV &a, const SV &b, const SV &c, uint32_t id,
                                const FaceView &fv, uint32_t s, int face, const BinCtx &bc)
{
    Placed p;
    const int where = place_tri(a, b, c, id, fv, s, face, bc, p);
    if (where == 0)
        return;
    for (uint32_t gy = p.h0; gy <= p.h1; ++gy)
        for (uint32_t gx = p.g0; gx <= p.g1; ++gx) {
            const uint32_t t = gy * bc.ntx + gx;
            if (where == 1)
                atomicAdd(&bc.lcnt[t], 1u);
            else
                bin_spilled(bc, s, t, p.r);
        }
}

// Exact per-face pipeline of one triangle up to the record.  Triangles that
// need clipping (near plane or guard band) are queued for k_order_clip.
// mm: the face's MVP, scis: face_scissor_clip of the face.
__device__ static inline void setup_face(const float *mm, float4 scis, const float (&vx)[3][3],
                                         uint32_t W, uint32_t s, int face, uint32_t id,
                                         uint32_t t, const BinCtx &bc)
{
    CV4 poly[3];
    transform3(mm, vx, poly);
    FaceView fv = face_view((int32_t)W, face);
    const TriClass cl = classify_tri(poly, scis);
    if (cl == kTriOut)
        return;
    if (cl == kTriClip) {
        uint32_t q = atomicAdd(&bc.counters[kCntClip], 1u);
        if (q < bc.clip_cap)
            bc.clipq[q] = make_uint2(t, s * 8u + (uint32_t)face);
        else
            atomicOr(&bc.counters[kCntOverflow], 1u);
        return;
    }
    float halfW = 0.5f * (float)W;
    SV a = project(poly[0], halfW), b = project(poly[1], halfW), c = project(poly[2], halfW);
    emit_tri(a, b, c, id, fv, s, face, bc);
}

__device__ static uint32_t cull_faces(const float *__restrict__ sm, const float (&lv)[9][256],
                                      float4 sph, float4 back, float halfW, int f0, int f1);

// Bounding sphere of every triangle, once per scene: the centroid as stored
// and the largest vertex distance from it, inflated by 1e-5 relative so it
// bounds the vertices whatever the rounding of the distances.  And its drawn
// side: the camera mirrors (right = up x dir), so a triangle is
// counter-clockwise seen from the side of (v2 - v0) x (v1 - v0); that over the
// longest edge, which leaves the triangle's smallest height as its length,
// and the longest edge.
__global__ __launch_bounds__(256) void k_tri_sphere(const float *__restrict__ tri, uint32_t ntri,
                                                    float4 *__restrict__ sph,
                                                    float4 *__restrict__ back)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntri)
        return;
    float v[3][3];
    for (int k = 0; k < 3; ++k)
        for (int c = 0; c < 3; ++c)
            v[k][c] = tri[(size_t)(3 * k + c) * ntri + t];
    float cx = (v[0][0] + v[1][0] + v[2][0]) * (1.0f / 3.0f);
    float cy = (v[0][1] + v[1][1] + v[2][1]) * (1.0f / 3.0f);
    float cz = (v[0][2] + v[1][2] + v[2][2]) * (1.0f / 3.0f);
    float r2 = 0.0f;
    for (int k = 0; k < 3; ++k) {
        float dx = v[k][0] - cx, dy = v[k][1] - cy, dz = v[k][2] - cz;
        r2 = fmaxf(r2, dx * dx + dy * dy + dz * dz);
    }
    sph[t] = make_float4(cx, cy, cz, sqrtf(r2) * 1.00001f);
    float e1[3], e2[3], l1 = 0.0f, l2 = 0.0f, l3 = 0.0f;
    for (int c = 0; c < 3; ++c) {
        e1[c] = v[1][c] - v[0][c];
        e2[c] = v[2][c] - v[0][c];
        const float e3 = v[2][c] - v[1][c];
        l1 += e1[c] * e1[c];
        l2 += e2[c] * e2[c];
        l3 += e3 * e3;
    }
    const float edge = sqrtf(fmaxf(l1, fmaxf(l2, l3)));
    const float inv = edge > 0.0f ? 1.0f / edge : 0.0f;
    back[t] = make_float4((e2[1] * e1[2] - e2[2] * e1[1]) * inv,
                          (e2[2] * e1[0] - e2[0] * e1[2]) * inv,
                          (e2[0] * e1[1] - e2[1] * e1[0]) * inv, edge);
}

void launch_tri_sphere(const float *tri, uint32_t ntri, float4 *sph, float4 *back, hipStream_t st)
{
    if (ntri)
        k_tri_sphere<<<(ntri + 255) / 256, 256, 0, st>>>(tri, ntri, sph, back);
}

// Tile columns [g0, g1] and rows [h0, h1] of a record's texel bbox.
__device__ static inline void unpack_bbox(uint64_t v, uint32_t tshift, uint32_t &g0,
                                          uint32_t &g1, uint32_t &h0, uint32_t &h1)
{
    g0 = (uint32_t)(v & 0xFFFFu) >> tshift;
    h0 = (uint32_t)((v >> 16) & 0xFFFFu) >> tshift;
    g1 = (uint32_t)((v >> 32) & 0xFFFFu) >> tshift;
    h1 = (uint32_t)(v >> 48) >> tshift;
}

// One workgroup per (256 triangles, shooter[, face]).  Phase 1: one lane
// per triangle runs the conservative culls (cull_faces) and queues the
// surviving (triangle, face) pairs in LDS; phase 2: the lanes take the queue
// so the exact pipeline runs with every lane busy.  Records go to the block's
// own region (LDS slot counter) and are counted in an LDS tile histogram;
// phase 3 reserves their places in the tiles' lists with one returning global
// atomic per touched tile and writes them there, which took the place of a
// scan over all bins and a fill kernel that read the bboxes back: over
// 200,000 triangles at hemicube 256 a pass of one shooter takes 109 us
// instead of 125, one of 64 shooters 343 instead of 376.  Triangles are stored as 9
// planes of ntri floats (v0.x, v0.y, ..., v2.z) so consecutive lanes load
// consecutive addresses.
// In a packed launch slot s draws only its scene's triangles
// [slot_tbeg[s], slot_tbeg[s] + slot_tcnt[s]); blockIdx.x walks that range.
__global__ __launch_bounds__(256) void k_raster_setup(uint32_t W, const float *__restrict__ tri,
                                                      const float4 *__restrict__ tsph,
                                                      const float4 *__restrict__ tback,
                                                      const uint32_t *__restrict__ tri_patch,
                                                      uint32_t ntri, const float *__restrict__ mvp,
                                                      const uint32_t *__restrict__ nshoot,
                                                      BinCtx bc, uint32_t *__restrict__ blk_nrec,
                                                      const uint32_t *__restrict__ slot_tbeg,
                                                      const uint32_t *__restrict__ slot_tcnt,
                                                      const uint32_t *__restrict__ slot_w,
                                                      uint32_t group, uint32_t slot0,
                                                      uint32_t nslot)
{
    extern __shared__ uint32_t dyn_lds[];
    uint32_t *lcnt = dyn_lds; // 4 x bc.ntiles per-tile counts (dynamic LDS)
    __shared__ float lv[9][256];
    __shared__ uint32_t lid[256];
    __shared__ uint16_t lq[256 * 5 * 4];
    __shared__ uint32_t lnrec2[4], lqn;
    __shared__ float4 lscis[5];
    __shared__ float lmvp[4][80]; // the current shooters' five face MVPs
    const uint32_t ns = *nshoot < nslot ? *nshoot : nslot;
    // hemicube resolution of the slots being drawn (per slot in a pack of
    // scenes at several resolutions; slots drawn together share a scene)
    uint32_t lw = 0u;
    const uint32_t tl0 = blockIdx.x * blockDim.x;
    // gridDim.z == 5 splits the faces over blocks (small K), else one block
    // walks all five faces
    const int f0 = gridDim.z == 1 ? 0 : (int)blockIdx.z, f1 = gridDim.z == 1 ? 5 : f0 + 1;
    // record region of shooter slot sl
    auto rbof = [&](uint32_t sl) { return (sl * gridDim.z + blockIdx.z) * gridDim.x + blockIdx.x; };
    // The block's triangles stay in registers / LDS while it walks `group`
    // consecutive shooter slots (reloaded only when a packed slot changes
    // scene), so vertices are read once per group instead of once per shooter.
    // Up to four slots that draw the same triangles are taken together: their
    // culls share one queue and one exact phase, which divides the barriers
    // and the per-slot set-up by the slot count; each keeps its own record region, tile counts and
    // record count.
    uint32_t ltb = 0xFFFFFFFFu, ltc = 0;
    float4 sph = make_float4(0.0f, 0.0f, 0.0f, 0.0f), back = sph;
    for (uint32_t g = 0; g < group;) {
        const uint32_t s = (slot0 + blockIdx.y * group) + g;
        if (s >= ns)
            break;
        const uint32_t tb = slot_tbeg ? slot_tbeg[s] : 0u, tc = slot_tcnt ? slot_tcnt[s] : ntri;
        uint32_t nsh = 1;
        while (nsh < 4 && g + nsh < group && s + nsh < ns) {
            const uint32_t tb1 = slot_tbeg ? slot_tbeg[s + nsh] : 0u;
            const uint32_t tc1 = slot_tcnt ? slot_tcnt[s + nsh] : ntri;
            if (tb1 != tb || tc1 != tc)
                break;
            ++nsh;
        }
        if (tl0 >= tc) {
            // beyond the slots' scene: empty regions
            if (threadIdx.x < nsh)
                blk_nrec[rbof(s + threadIdx.x)] = 0u;
            g += nsh;
            continue;
        }
        __syncthreads(); // the previous slots' phase 2 and flush are done with LDS
        const uint32_t Ws = slot_w ? slot_w[s] : W;
        if (Ws != lw) {
            lw = Ws;
            if (threadIdx.x < 5)
                lscis[threadIdx.x] = face_scissor_clip((int32_t)Ws, (int)threadIdx.x);
        }
        if (tb != ltb || tc != ltc) {
            ltb = tb;
            ltc = tc;
            if (tl0 + threadIdx.x < tc) {
                const uint32_t t = tb + tl0 + threadIdx.x;
#pragma unroll
                for (int k = 0; k < 3; ++k)
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        lv[3 * k + c][threadIdx.x] = tri[(size_t)(3 * k + c) * ntri + t];
                lid[threadIdx.x] = tri_patch[t] + 1u;
                sph = tsph[t];
                back = tback[t];
            }
        }
        for (uint32_t i = threadIdx.x; i < nsh * bc.ntiles; i += blockDim.x)
            lcnt[i] = 0u;
        if (threadIdx.x < 4)
            lnrec2[threadIdx.x] = 0u;
        if (threadIdx.x == 0)
            lqn = 0u;
        for (uint32_t i = threadIdx.x; i < 80 * nsh; i += blockDim.x)
            lmvp[i / 80][i % 80] = mvp[(size_t)(s + i / 80) * kShooterStride + i % 80];
        __syncthreads();
        // phase 1: cheap culls; surviving (triangle, slot, face) triples go to
        // an LDS queue
        if (tl0 + threadIdx.x < tc) {
            for (uint32_t sh = 0; sh < nsh; ++sh) {
                uint32_t fm = cull_faces(mvp + (size_t)(s + sh) * kShooterStride, lv, sph, back,
                                         0.5f * (float)Ws, f0, f1);
                while (fm) {
                    int f = __ffs(fm) - 1;
                    fm &= fm - 1;
                    lq[atomicAdd(&lqn, 1u)] =
                        (uint16_t)((threadIdx.x << 5) | (sh << 3) | (uint32_t)f);
                }
            }
        }
        __syncthreads();
        // phase 2: the exact per-face pipeline over the compacted triples
        const uint32_t nq = lqn;
        for (uint32_t q = threadIdx.x; q < nq; q += blockDim.x) {
            uint32_t e = lq[q];
            uint32_t tl = e >> 5, sh = (e >> 3) & 3u;
            int face = (int)(e & 7u);
            float wv[3][3];
#pragma unroll
            for (int k = 0; k < 3; ++k)
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    wv[k][c] = lv[3 * k + c][tl];
            BinCtx b2 = bc;
            b2.region = rbof(s + sh) * kRecsPerBlock;
            b2.lnrec = &lnrec2[sh];
            b2.lcnt = lcnt + sh * bc.ntiles;
            setup_face(lmvp[sh] + face * 16, lscis[face], wv, Ws, s + sh, face, lid[tl],
                       tb + tl0 + tl, b2);
        }
        __syncthreads();
        // the records into their tiles' lists: one returning global atomic per
        // touched tile reserves the entries, whose first place takes the
        // count's place in LDS ...
        const uint32_t e1 = lnrec2[0], e2 = e1 + lnrec2[1], e3 = e2 + lnrec2[2],
                       e4 = e3 + lnrec2[3];
        auto rec_of = [&](uint32_t f, uint32_t &sh) {
            sh = (f >= e1 ? 1u : 0u) + (f >= e2 ? 1u : 0u) + (f >= e3 ? 1u : 0u);
            const uint32_t q = f - (sh == 0 ? 0u : sh == 1 ? e1 : sh == 2 ? e2 : e3);
            return rbof(s + sh) * kRecsPerBlock + q;
        };
        // (a thread's first bbox comes back during the atomics)
        uint32_t sh0 = 0, r0 = 0;
        uint64_t v0 = 0;
        if (threadIdx.x < e4) {
            r0 = rec_of(threadIdx.x, sh0);
            v0 = bc.bbox[r0];
        }
        uint32_t *const cnt = bc.bin_count + (size_t)s * bc.ntiles;
        const uint32_t nl = nsh * bc.ntiles;
        for (uint32_t i0 = threadIdx.x; i0 < nl; i0 += 4u * blockDim.x) {
            uint32_t c[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t i = i0 + j * blockDim.x;
                c[j] = i < nl ? lcnt[i] : 0u;
            }
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                if (c[j])
                    c[j] = atomicAdd(&cnt[i0 + j * blockDim.x], c[j]);
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t i = i0 + j * blockDim.x;
                if (i < nl)
                    lcnt[i] = c[j];
            }
        }
        if (threadIdx.x < nsh)
            blk_nrec[rbof(s + threadIdx.x)] = lnrec2[threadIdx.x];
        __syncthreads();
        // ... and every record counts on from it
        for (uint32_t f = threadIdx.x; f < e4; f += blockDim.x) {
            uint32_t sh = sh0, r = r0;
            if (f != threadIdx.x) {
                r = rec_of(f, sh);
                v0 = bc.bbox[r];
            }
            uint32_t g0, g1, h0, h1;
            unpack_bbox(v0, bc.tshift, g0, g1, h0, h1);
            for (uint32_t gy = h0; gy <= h1; ++gy)
                for (uint32_t gx = g0; gx <= g1; ++gx) {
                    const uint32_t b = gy * bc.ntx + gx;
                    list_put(bc, s + sh, b, atomicAdd(&lcnt[sh * bc.ntiles + b], 1u), r);
                }
        }
        g += nsh;
    }
}

// Conservative culls of one triangle for one shooter; returns the mask of
// faces in [f0, f1) the exact pipeline must look at.  The triangle's
// bounding sphere (centre, radius; k_tri_sphere) gives the centre's height
// pa over the shooter's plane and its offsets along the face axes, with a
// margin mq for float rounding:
//  - a sphere wholly below the plane (pa + rho + mq < 0) puts every vertex
//    strictly below it: in the side faces the triangle lies in the
//    scissored-away half, in the front face behind the near plane (0.01);
//  - a sphere straddling the band just above the plane falls back to the
//    per-vertex test: no vertex above the plane by more than
//    tol = min(1e-6 |v - eye|_1, 0.0099) (which also bounds the float error
//    of the height), so in the side faces the triangle lies in the
//    scissored-away half or within tol/|v - eye| * W/2 << 0.5 pixel of the
//    horizon, where the nearest kept pixel centre is half a pixel away, and
//    in the front face it is nearer than the near plane.  This removes the
//    shooter's own plane (floor under a floor patch) before any per-face work;
//  - a face whose frustum (90 degree pyramid around its axis, near 0.01)
//    misses the sphere by more than a margin;
//  - a triangle (of one face only, by the last test over all five faces, also
//    where the workgroup looks at one: on a second face it would be nearer and
//    wider than the bounds below) of area A whose plane the eye lies at least
//    D > 0 behind: with depths in [wmin, wmax] it projects to a clockwise area of at least
//    (W/2)^2 2 A D / wmax^3 square pixels.  Snapping and rounding move a
//    vertex by at most delta pixels per axis, which changes the area by at
//    most 5.7 delta L + 8 delta^2 for a longest projected edge
//    L <= sqrt2 (W/2) edge (1 + kappa) / wmin, kappa the largest |x / w|; the
//    two tests ask twice that, multiplied out, so the snapped triangle is
//    clockwise too and would be dropped.  back: k_tri_sphere's, whose product
//    with the centre's offset is 2 A D / edge.  (Two in five triangles that
//    pass the other culls in rooms with boxes; each costs the exact pipeline
//    three projections.)
__device__ static uint32_t cull_faces(const float *__restrict__ sm, const float (&lv)[9][256],
                                      float4 sph, float4 back, float halfW, int f0, int f1)
{
    if (sm[92] != 0.0f)
        return ((1u << f1) - 1u) & ~((1u << f0) - 1u);
    const float ex = sm[80], ey = sm[81], ez = sm[82];
    const float nx = sm[83], ny = sm[84], nz = sm[85];
    const float ux = sm[86], uy = sm[87], uz = sm[88];
    const float wx = sm[89], wy = sm[90], wz = sm[91];
    const float cx = sph.x - ex, cy = sph.y - ey, cz = sph.z - ez, rho = sph.w;
    const float pa = fmaf(cz, nz, fmaf(cy, ny, cx * nx));
    const float pb = fmaf(cz, uz, fmaf(cy, uy, cx * ux));
    const float pc = fmaf(cz, wz, fmaf(cy, wy, cx * wx));
    const float mq = fmaf(1e-4f, fabsf(pa) + fabsf(pb) + fabsf(pc) + rho, 1e-6f);
    if (pa + rho + mq < 0.0f)
        return 0u;
    if (pa - rho - mq <= 0.0099f) {
        bool below = true;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            float dx = lv[3 * k][threadIdx.x] - ex, dy = lv[3 * k + 1][threadIdx.x] - ey,
                  dz = lv[3 * k + 2][threadIdx.x] - ez;
            float h = dx * nx + dy * ny + dz * nz;
            float tol = fminf(1e-6f * (fabsf(dx) + fabsf(dy) + fabsf(dz)), 0.0099f);
            below = below && (h < tol);
        }
        if (below)
            return 0u;
    }
    const float m = fmaf(rho, 1.4143f, mq);
    const float far = fmaxf(fabsf(pa), fmaxf(fabsf(pb), fabsf(pc))), T = far - m;
    const uint32_t faces = ((1u << f1) - 1u) & ~((1u << f0) - 1u);
    if (!(T > 0.0f)) {
        // near the eye: face by face
        uint32_t mask = 0u;
        for (int face = f0; face < f1; ++face) {
            float q, s1, s2;
            switch (face) {
            case 0: q = pb; s1 = pa; s2 = pc; break;   // UP    (axis  u)
            case 1: q = -pb; s1 = pa; s2 = pc; break;  // DOWN  (axis -u)
            case 2: q = pc; s1 = pa; s2 = pb; break;   // LEFT  (axis n x u)
            case 3: q = -pc; s1 = pa; s2 = pb; break;  // RIGHT (axis -(n x u))
            default: q = pa; s1 = pb; s2 = pc; break;  // FRONT (axis n)
            }
            if (q + m < fabsf(s1) || q + m < fabsf(s2) || q + rho + m < 0.0099f)
                continue;
            mask |= 1u << face;
        }
        return mask;
    }
    // farther than its margin: the face of the largest coordinate and those
    // whose coordinate comes within the margin of it
    uint32_t mask = (fabsf(pb) >= T ? (pb > 0.0f ? 1u : 2u) : 0u) |
                    (fabsf(pc) >= T ? (pc > 0.0f ? 4u : 8u) : 0u) | (pa >= T ? 16u : 0u);
    const float l1 = fabsf(cx) + fabsf(cy) + fabsf(cz);
    const float db = fmaf(-4e-6f * l1, back.w, fmaf(cz, back.z, fmaf(cy, back.y, cx * back.x)));
    // (one face of all five, whichever this workgroup looks at)
    if (db > 0.0f && (mask & (mask - 1u)) == 0u) {
        const float wmin = far - rho - mq, wmax = far + rho + mq;
        const float S = __builtin_amdgcn_fmed3f(fabsf(pa), fabsf(pb), fabsf(pc)) + rho;
        const float em = 2e-6f * (fabsf(ex) + fabsf(ey) + fabsf(ez));
        const float dw = fmaf(fmaf(1.6e-5f, halfW, 0.0025f), wmin, halfW * fmaf(1e-6f, l1, em));
        const float a = 0.5f * halfW * db * wmin * wmin, w3 = 16.0f * dw * wmax * wmax * wmax;
        if (wmin > 0.02f && S <= 8.0f * wmin && a * wmin > w3 * (wmin + S) &&
            a * halfW * back.w > w3 * dw)
            mask = 0u;
    }
    return mask & faces;
}

// The launch order of the bins [bin0, bin0 + n) for the tile kernel, largest
// first, so that the heavy horizon tiles overlap the light ones instead of
// forming the tail of the launch: each bin goes to the queue of its size
// class (queue c at order + c * qstride; a class's counter of the pass
// counters reserves the places).  Class 0 holds the bins that the tile kernel
// draws as four quadrants, at most split_cap of them.  A thread's bins, and
// the bins of neighbouring threads, are far apart on the hemicube: that ran
// measurably faster in the tile kernel than neighbouring tiles launched
// together.
//
// The workgroups from norder on clip: the queued (triangle, shooter, face)
// jobs that cross the near plane or the guard band, one per wavefront: lanes
// 0 .. 2 transform their vertex as transform3 does, the wavefront clips, and
// the fan triangles (0, k, k + 1) are emitted by lanes k = 1 .. n - 2 at
// once; records go to the spill region and straight into the lists.  The
// order may miss their counts: every bin is in it whatever its count.  The
// entry total misses none: an order workgroup marks the bins it has summed
// (kBinSeen), and an entry that finds the mark adds itself.
// Latency-bound: 6 us for one shooter over 200,000 triangles, 16 us for each
// half of 64 (a scan kernel and a clip kernel took 10 and 21).
constexpr uint32_t kOrderPer = 4;

__device__ static inline uint32_t order_class(uint32_t n, uint32_t split_max)
{
    if (n >= kSplitRecs && n <= split_max)
        return 0u;
    return n >= 2048u ? 1u : n >= 1024u ? 2u : n >= 512u ? 3u : n >= 256u ? 4u : n >= 128u ? 5u
           : n >= 64u ? 6u : 7u;
}

__global__ __launch_bounds__(256) void k_order_clip(uint32_t norder, uint32_t n, uint32_t bin0,
                                                    uint32_t split_cap,
                                                    uint32_t *__restrict__ order,
                                                    uint32_t qstride, uint32_t W,
                                                    const float *__restrict__ tri,
                                                    const uint32_t *__restrict__ tri_patch,
                                                    uint32_t ntri, const float *__restrict__ mvp,
                                                    BinCtx bc,
                                                    const uint32_t *__restrict__ blk_nrec,
                                                    uint32_t nreg, uint32_t *__restrict__ pool,
                                                    uint32_t pool_cap,
                                                    const uint32_t *__restrict__ slot_w)
{
    __shared__ uint32_t lcls[kBinClasses], gcls[kBinClasses], lsum;
    __shared__ CV4 lp[4][kClipMax];
    if (blockIdx.x < norder) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            BinFacts *const f = reinterpret_cast<BinFacts *>(bc.counters + kCntFacts);
            f->blk_nrec = blk_nrec;
            f->nreg = nreg;
            f->spill_base = bc.spill_base;
            f->spill_cap = bc.spill_cap;
            f->split_cap = split_cap;
            f->pool = pool;
            f->pool_cap = pool_cap;
            f->pool_used = &bc.counters[kCntPool];
        }
        if (threadIdx.x < kBinClasses)
            lcls[threadIdx.x] = 0u;
        if (threadIdx.x == 0)
            lsum = 0u;
        __syncthreads();
        const uint32_t split_max = split_cap ? bc.bin_cap : 0u;
        uint32_t c[kOrderPer], pos[kOrderPer], sum = 0;
#pragma unroll
        for (uint32_t k = 0; k < kOrderPer; ++k) {
            const uint32_t i = (threadIdx.x * kOrderPer + k) * norder + blockIdx.x;
            const uint32_t m = i < n ? atomicOr(&bc.bin_count[bin0 + i], kBinSeen) : 0u;
            sum += m;
            c[k] = order_class(m, split_max);
        }
#pragma unroll
        for (uint32_t k = 0; k < kOrderPer; ++k) {
            const uint32_t i = (threadIdx.x * kOrderPer + k) * norder + blockIdx.x;
            if (i >= n)
                continue;
            if (c[k] == 0u) {
                const uint32_t p0 = atomicAdd(&bc.counters[kCntClass], 1u);
                if (p0 < split_cap)
                    order[p0] = bin0 + i;
                else
                    c[k] = 1u; // beyond the quadrants the launch has room for
            }
            if (c[k])
                pos[k] = atomicAdd(&lcls[c[k]], 1u);
        }
        atomicAdd(&lsum, sum);
        __syncthreads();
        if (threadIdx.x > 0 && threadIdx.x < kBinClasses && lcls[threadIdx.x])
            gcls[threadIdx.x] =
                atomicAdd(&bc.counters[kCntClass + threadIdx.x], lcls[threadIdx.x]);
        if (threadIdx.x == 0 && lsum)
            atomicAdd(&bc.counters[kCntEntries], lsum);
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < kOrderPer; ++k) {
            const uint32_t i = (threadIdx.x * kOrderPer + k) * norder + blockIdx.x;
            if (i < n && c[k])
                order[(size_t)c[k] * qstride + gcls[c[k]] + pos[k]] = bin0 + i;
        }
        return;
    }
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t nj = min(bc.counters[kCntClip], bc.clip_cap);
    for (uint32_t q = (blockIdx.x - norder) * 4u + wv; q < nj; q += (gridDim.x - norder) * 4u) {
        const uint2 job = bc.clipq[q];
        const uint32_t t = job.x, s = job.y >> 3;
        const int face = (int)(job.y & 7u);
        CV4 v;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            v.c[c] = 0.0f;
        if (lane < 3) {
            const float x = tri[(size_t)(3 * lane + 0) * ntri + t];
            const float y = tri[(size_t)(3 * lane + 1) * ntri + t];
            const float z = tri[(size_t)(3 * lane + 2) * ntri + t];
            const float *mm = mvp + (size_t)s * kShooterStride + face * 16;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                v.c[r] = mm[0 * 4 + r] * x + mm[1 * 4 + r] * y + mm[2 * 4 + r] * z + mm[3 * 4 + r];
        }
        const uint32_t Ws = slot_w ? slot_w[s] : W;
        FaceView fv = face_view((int32_t)Ws, face);
        const int np = clip_polygon_wave(v, lp[wv], &bc.counters[kCntOverflow]);
        SV a, b, cc;
        Placed p;
        bool have = false;
        if (np >= 3 && clip_fan(v, np, 0.5f * (float)Ws, a, b, cc))
            have = place_tri(a, b, cc, tri_patch[t] + 1u, fv, s, face, bc, p) != 0;
        // the records' tiles, flattened over the lanes: a list place is a
        // returning atomic, so one lane walking a large record's tiles would
        // wait for each
        const uint64_t em = __ballot(have);
        for (uint32_t base = 0, total = 64u; base < total; base += 64u) {
            total = 0;
            uint32_t r = 0, tile = ~0u;
            for (uint64_t m = em; m; m &= m - 1) {
                const int l = __ffsll((long long)m) - 1;
                auto at = [&](uint32_t x) {
                    return (uint32_t)__builtin_amdgcn_readlane((int)x, l);
                };
                const uint32_t g0 = at(p.g0), nx = at(p.g1) - g0 + 1u;
                const uint32_t h0 = at(p.h0), ny = at(p.h1) - h0 + 1u;
                const uint32_t i = base + lane - total;
                if (base + lane >= total && i < nx * ny) {
                    r = at(p.r);
                    tile = (h0 + i / nx) * bc.ntx + g0 + i % nx;
                }
                total += nx * ny;
            }
            if (tile != ~0u)
                bin_spilled(bc, s, tile, r);
        }
        wave_lds_sync(); // lp is the next job's
    }
}

// One workgroup per bin = (shooter, tile).  The bin's records are taken 256
// at a time, one per lane.  A record covering at most small_px pixels of the
// tile is drawn by its lane with incremental edge functions; larger ones go
// to an LDS queue that the wavefronts then draw one record per wavefront, one
// pixel per lane.  (Sorting the records by size first, so that a wavefront's
// lanes draw records of about the same size, cost more in loads and barriers
// than the lane divergence it saved.)  Depth is resolved in LDS with 64-bit
// atomicMin, so the drawing order does not matter; the atomic returns nothing
// and is issued without first reading the texel, so no fragment waits on an
// LDS read.  Then the tile either goes
// to the item buffer (out_ids != null; out_depth != null adds the depth
// plane) or is reduced into F rows and hit counts (ff or, in the
// deterministic mode, its fixed-point rows ffq != null).

// read by scalar loads: nothing writes it during the launch
using ConstFacts = const __attribute__((address_space(4))) BinFacts *;

// The list of a bin fuller than its list has room for: the workgroup goes
// over all records of the slot, the regions and the spill region, and writes
// those that touch the tile at (ox, oy) into the pool, where it reserves the
// bin's n entries.  *cnt (LDS): how many.
__device__ static const uint32_t *whole_list(ConstFacts f,
                                             const RasterRec *__restrict__ recs,
                                             const uint64_t *__restrict__ bbox, uint32_t s,
                                             uint32_t n, int32_t ox, int32_t oy, int32_t T,
                                             uint32_t *cnt, uint32_t *at)
{
    const uint32_t me = threadIdx.x;
    if (me == 0) {
        *cnt = 0u;
        *at = atomicAdd(f->pool_used, n);
    }
    __syncthreads();
    const uint32_t used = __builtin_amdgcn_readfirstlane(*at);
    const uint32_t cap = f->pool_cap, room = cap - min(used, cap);
    uint32_t *const out = f->pool + (cap - room);
    auto take = [&](uint32_t r) {
        const uint64_t v = bbox[r];
        if ((int32_t)(v & 0xFFFFu) < ox + T && (int32_t)((v >> 16) & 0xFFFFu) < oy + T &&
            (int32_t)((v >> 32) & 0xFFFFu) >= ox && (int32_t)(v >> 48) >= oy) {
            const uint32_t q = atomicAdd(cnt, 1u);
            if (q < room) // always, unless the pass has more entries than it may
                out[q] = r;
        }
    };
    for (uint32_t b = me >> 6; b < f->nreg; b += kTileThreads / 64u) {
        const uint32_t reg = s * f->nreg + b, k = f->blk_nrec[reg];
        for (uint32_t q = me & 63u; q < k; q += 64u)
            take(reg * kRecsPerBlock + q);
    }
    const uint32_t nsp = min((uint32_t)f->nspill, (uint32_t)f->spill_cap);
    for (uint32_t q = me; q < nsp; q += kTileThreads)
        if ((recs[f->spill_base + q].sf >> 2) == s)
            take(f->spill_base + q);
    __syncthreads();
    if (me == 0)
        *cnt = min(*cnt, room);
    __syncthreads();
    return out;
}

template <bool FQ>
__global__ __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_tile_raster(
    uint32_t W, uint32_t TW, uint32_t TH, uint32_t RES, const uint32_t *__restrict__ nshoot,
    const RasterRec *__restrict__ recs, const uint64_t *__restrict__ bbox,
    const uint32_t *__restrict__ bin_count, const uint32_t *__restrict__ list, uint32_t bin_cap,
    const BinFacts *__restrict__ facts, uint32_t ntx, uint32_t ntiles, uint32_t tshift, uint32_t small_px, uint32_t *__restrict__ out_ids,
    float *__restrict__ out_depth, const float *__restrict__ dff,
    uint32_t rowlen, const uint32_t *__restrict__ slot_pbeg, float *__restrict__ ff,
    unsigned long long *__restrict__ ffq, uint32_t *__restrict__ hits,
    uint32_t *__restrict__ counters, const uint32_t *__restrict__ order, uint32_t qstride,
    const uint32_t *__restrict__ slot_w, const uint32_t *__restrict__ slot_dffo,
    uint32_t *__restrict__ fblk, uint32_t fstride)
{
    __shared__ uint64_t tk[kMaxTile * kMaxTile];
    // the chunk queues, then (resolve) the table of F entries
    __shared__ union {
        struct {
            uint32_t perm[kTileThreads];
            uint64_t pbb[kTileThreads];
        } q;
        struct {
            uint32_t key[kTileTable];
            float sum[kTileTable];
            uint32_t cnt[kTileTable];
        } t;
    } sh;
    uint32_t *const perm = sh.q.perm;
    uint64_t *const pbb = sh.q.pbb;
    __shared__ uint32_t nbig;
    // the workgroup's bin: first the quadrants of the largest (class 0), then
    // the other classes' queues
    uint32_t bin, quad = 4u;
    {
        const auto cls = ((ConstFacts)facts)->cls;
        const uint32_t n0 = min((uint32_t)cls[0], (uint32_t)((ConstFacts)facts)->split_cap);
        uint32_t b = blockIdx.x, c = 0;
        if (b < 4u * n0) {
            quad = b & 3u;
            b >>= 2;
        } else {
            b -= 4u * n0;
            for (c = 1; c < kBinClasses && b >= cls[c]; ++c)
                b -= cls[c];
            if (c == kBinClasses)
                return;
        }
        bin = order[(size_t)c * qstride + b];
    }
    const uint32_t s = bin / ntiles;
    if (s >= *nshoot)
        return;
    const uint32_t tile = bin - s * ntiles;
    const uint32_t n = bin_count[bin] & ~kBinSeen;
    // an empty bin adds nothing to the F rows (its texels are background)
    if (n == 0 && !out_ids)
        return;
    // a slot of a pack may render at its scene's own resolution; tiles are
    // laid out for the largest, so its slab uses the first ones
    if (slot_w) {
        W = slot_w[s];
        TW = 2 * W;
        TH = W + W / 2;
        dff += slot_dffo[s];
    }
    int32_t ox = (int32_t)((tile % ntx) << tshift), oy = (int32_t)((tile / ntx) << tshift);
    if (quad < 4u && n > bin_cap) {
        // the clipped triangles overfilled it since: drawn whole
        if (quad)
            return;
        quad = 4u;
    }
    if (quad < 4u) { // a quadrant: a tile of half the side over the same list
        tshift -= 1;
        ox += (int32_t)((quad & 1u) << tshift);
        oy += (int32_t)((quad >> 1) << tshift);
    }
    const uint32_t T = 1u << tshift, TT = T * T;
    const uint32_t me = threadIdx.x;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(me >> 6);
    constexpr uint32_t kNoRec = ~0u;
    const uint32_t *lst = list + (size_t)bin * bin_cap;
    uint32_t nl = n;
    if (__builtin_expect(n > bin_cap, 0)) {
        lst = whole_list((ConstFacts)facts, recs, bbox, s, n, ox, oy, (int32_t)T, &nbig, perm);
        nl = __builtin_amdgcn_readfirstlane(nbig);
        __syncthreads();
    }
    // Lane me's record of the chunk starting at entry cb.  A chunk of m <
    // 256 records would leave waves idle: its records are dealt to
    // ceil(m / 64) wave sets (one per lane), and the nph = 4 / sets waves of a
    // set each draw row phase ph of its in-lane records (every nph-th bbox
    // row); a full chunk keeps one record per lane, nph = 1.
    auto deal = [&](uint32_t cb, uint32_t &ph, uint32_t &nph) -> uint32_t {
        const uint32_t m = min(kTileThreads, nl - cb);
        const uint32_t sets = (m + 63u) >> 6;
        nph = sets >= 3u ? 1u : 4u / sets;
        ph = wv / sets;
        const uint32_t k = (wv - ph * sets) * 64u + (me & 63u);
        return ph < nph && k < m ? lst[cb + k] : kNoRec;
    };

    // A lane's entry of the first chunk (list index and bbox) is fetched
    // while the tile clears; each later chunk's list entries are fetched
    // during the chunk before it.
    uint32_t ph = 0, nph = 1;
    uint32_t ri = nl ? deal(0u, ph, nph) : kNoRec;
    uint64_t bv = 0;
    if (ri != kNoRec)
        bv = bbox[ri];
    for (uint32_t p = threadIdx.x; p < TT; p += blockDim.x)
        tk[p] = kClearKey;
    for (uint32_t c0 = 0; c0 < nl; c0 += blockDim.x) {
        if (me == 0)
            nbig = 0u;
        uint32_t ph_n = 0, nph_n = 1;
        const uint32_t rnext = c0 + blockDim.x < nl ? deal(c0 + blockDim.x, ph_n, nph_n) : kNoRec;
        __syncthreads();
        if (ri != kNoRec) {
            const int32_t ax0 = max((int32_t)(bv & 0xFFFFu), ox);
            const int32_t ay0 = max((int32_t)((bv >> 16) & 0xFFFFu), oy);
            const int32_t ax1 = min((int32_t)((bv >> 32) & 0xFFFFu), ox + (int32_t)T - 1);
            const int32_t ay1 = min((int32_t)(bv >> 48), oy + (int32_t)T - 1);
            const uint32_t area = (uint32_t)(ax1 - ax0 + 1) * (uint32_t)(ay1 - ay0 + 1);
            if (ax1 < ax0 || ay1 < ay0) {
                // touches other quadrants only
            } else if (area <= small_px) {
                const RasterRec r = recs[ri];
                draw_lane(r, r.sf & kSpanLane, (int32_t)(int16_t)r.vp, (int32_t)(r.vp >> 16), ax0,
                          ax1, ay0, ay1, ox, oy, tshift, tk, ph, nph);
            } else if (ph == 0) {
                const uint32_t q = atomicAdd(&nbig, 1u);
                perm[q] = ri;
                pbb[q] = bv;
            }
        }
        __syncthreads();
        // large records: the whole wavefront per record in 8 x 8 pixel
        // blocks; wave w takes queue entries w, w + 4, ...
        const uint32_t nall = nbig;
        for (uint32_t q = me >> 6; q < nall; q += blockDim.x >> 6) {
            const RasterRec rb = recs[perm[q]];
            const uint64_t bb = pbb[q];
            const int32_t ax0 = max((int32_t)(bb & 0xFFFFu), ox);
            const int32_t ax1 = min((int32_t)((bb >> 32) & 0xFFFFu), ox + (int32_t)T - 1);
            const int32_t ay0 = max((int32_t)((bb >> 16) & 0xFFFFu), oy);
            const int32_t ay1 = min((int32_t)(bb >> 48), oy + (int32_t)T - 1);
            const int32_t vpx = (int32_t)(int16_t)rb.vp, vpy = (int32_t)(rb.vp >> 16);
            if (__builtin_amdgcn_readfirstlane(rb.sf) & kSpanWave) {
                draw_wave32(rb, vpx, vpy, ax0, ax1, ay0, ay1, ox, oy, tshift, tk);
            } else {
                Edges e;
                make_edges(rb.x, rb.y, e);
                draw_wave(rb, e, vpx, vpy, ax0, ax1, ay0, ay1, ox, oy, tshift, tk);
            }
        }
        ri = rnext;
        ph = ph_n;
        nph = nph_n;
        if (ri != kNoRec)
            bv = bbox[ri];
        __syncthreads();
    }
    // Resolve.  Float F rows (the shooting pass) go through the LDS table in
    // the 4-texels-per-lane layout: wavefront w takes texels [256 w, 256 w +
    // 256) of the tile in row-major order (4 waves cover a 32 x 32 tile); TW
    // and the tile side are multiples of 4, so a lane's texels lie in one row
    // and are all inside the hemicube or all outside, and their ΔFF values
    // (16-byte aligned: RES, and a pack slot's table offset, are multiples of
    // 4) are one load.  The item buffer and the fixed-point rows walk the
    // tile one texel per lane.  Every ΔFF load is issued before the last
    // barrier.
    static_assert(kMaxTile * kMaxTile == 4 * kTileThreads, "one table resolve step per tile");
    constexpr uint32_t kPer = kMaxTile * kMaxTile / kTileThreads;
    const bool table = !FQ && ff != nullptr;
    const bool reduce = ff || ffq;
    const uint32_t rp = (threadIdx.x >> 6) * 256u + (threadIdx.x & 63) * 4u;
    const int32_t rx = ox + (int32_t)(rp & (T - 1)), ry = oy + (int32_t)(rp >> tshift);
    const bool rin = rp < TT && rx < (int32_t)TW && ry < (int32_t)TH;
    float4 d4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float fd[kPer];
    if (table) {
        if (rin)
            d4 = *reinterpret_cast<const float4 *>(dff + (uint32_t)ry * TW + (uint32_t)rx);
        // the queues are done: their LDS becomes the table
        sh.t.key[threadIdx.x] = 0u;
        sh.t.sum[threadIdx.x] = 0.0f;
        sh.t.cnt[threadIdx.x] = 0u;
    } else {
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k) {
            const uint32_t p = k * kTileThreads + threadIdx.x;
            const int32_t tx = ox + (int32_t)(p & (T - 1)), ty = oy + (int32_t)(p >> tshift);
            fd[k] = reduce && p < TT && tx < (int32_t)TW && ty < (int32_t)TH
                        ? dff[(uint32_t)ty * TW + (uint32_t)tx]
                        : 0.0f;
        }
    }
    const uint32_t pbase = slot_pbeg ? slot_pbeg[s] : 0u;
    __syncthreads();
    if (table) {
        float *const frow = ff + (size_t)s * rowlen;
        uint32_t *const hrow = hits ? hits + (size_t)s * rowlen : nullptr;
        // this slot's column of the F-block flags
        uint32_t *const fflag = fblk ? fblk + s : nullptr;
        if ((threadIdx.x >> 6) * 256u < TT) { // whole wavefronts
            uint32_t q4[4] = {0u, 0u, 0u, 0u};
            float f4[4] = {0.f, 0.f, 0.f, 0.f};
            if (rin) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    q4[j] = (uint32_t)tk[rp + j];
                f4[0] = q4[0] ? d4.x : 0.f;
                f4[1] = q4[1] ? d4.y : 0.f;
                f4[2] = q4[2] ? d4.z : 0.f;
                f4[3] = q4[3] ? d4.w : 0.f;
            }
            const bool with_c = hrow != nullptr;
            reduce_quad(q4, f4, with_c, [&](uint32_t id, float f, uint32_t c) {
                run_add(id, f, c, pbase, rowlen, with_c, sh.t.key, sh.t.sum, sh.t.cnt, frow, hrow,
                        counters, fflag, fstride);
            });
        }
        __syncthreads();
        const uint32_t key = sh.t.key[threadIdx.x];
        if (key) {
            atomicAdd(&frow[key - 1], sh.t.sum[threadIdx.x]);
            if (hrow)
                atomicAdd(&hrow[key - 1], sh.t.cnt[threadIdx.x]);
            if (fflag)
                fflag[((key - 1) >> 6) * fstride] = 1u;
        }
        return;
    }
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        if (k * kTileThreads >= TT)
            break;
        const uint32_t p = k * kTileThreads + threadIdx.x;
        const int32_t tx = ox + (int32_t)(p & (T - 1)), ty = oy + (int32_t)(p >> tshift);
        const bool inside = p < TT && tx < (int32_t)TW && ty < (int32_t)TH;
        const uint64_t key = inside ? tk[p] : kClearKey;
        const uint32_t texel = (uint32_t)ty * TW + (uint32_t)tx;
        if (out_ids && inside) {
            out_ids[(size_t)s * RES + texel] = (uint32_t)key;
            if (out_depth)
                out_depth[(size_t)s * RES + texel] = __uint_as_float((uint32_t)(key >> 32));
        }
        if (reduce) {
            const uint32_t id = (uint32_t)key;
            reduce_wave<FQ>(id, id ? fd[k] : 0.0f, s, pbase, rowlen, ff, ffq, hits, counters);
        }
    }
}

// Counter block h's part of the buffers: its half's, or both halves' for a pass
// drawn whole by a context whose larger passes are split (bb.halves), so that
// what a pass may hold does not depend on whether it is.
static BinCtx bin_ctx(const BinBuffers &bb, uint32_t h, bool whole, uint32_t *counters)
{
    const uint32_t parts = whole ? bb.halves : 1u;
    BinCtx bc;
    bc.recs = bb.recs;
    bc.bbox = bb.bbox;
    bc.bin_count = bb.count;
    bc.counters = counters + h * kCntN;
    bc.lnrec = nullptr;
    bc.lcnt = nullptr;
    bc.region = 0;
    bc.spill_base = bb.spill_base + h * bb.spill_cap;
    bc.spill_cap = parts * bb.spill_cap;
    bc.clipq = bb.clipq + (size_t)h * bb.clip_cap;
    bc.clip_cap = parts * bb.clip_cap;
    bc.ntx = bb.ntx;
    bc.ntiles = bb.ntiles;
    bc.tshift = bb.tshift;
    bc.list = bb.list;
    bc.bin_cap = bb.bin_cap;
    return bc;
}

uint32_t entry_cap(const BinBuffers &bb, bool whole)
{
    const uint64_t n = (uint64_t)bb.ent_cap * (whole ? bb.halves : 1u);
    return (uint32_t)(n > kMaxEntries ? kMaxEntries : n);
}

void launch_raster_setup(const Geometry &g, uint32_t s0, uint32_t s1, uint32_t h,
                         const float *tri, const float4 *tsph, const float4 *tback,
                         const uint32_t *tri_patch, uint32_t ntri, const float *mvp, const uint32_t *nshoot,
                         const BinBuffers &bb, uint32_t *counters, const uint32_t *slot_tbeg,
                         const uint32_t *slot_tcnt, const uint32_t *slot_w, bool whole,
                         hipStream_t st)
{
    const uint32_t n = s1 - s0;
    uint32_t group = bb.setup_group ? bb.setup_group : 1u;
    if (group > n)
        group = n;
    dim3 grid(bb.nblk, (n + group - 1) / group, bb.nz);
    k_raster_setup<<<grid, 256, 4 * bb.ntiles * sizeof(uint32_t), st>>>(
        g.W, tri, tsph, tback, tri_patch, ntri, mvp, nshoot, bin_ctx(bb, h, whole, counters), bb.blk_nrec,
        slot_tbeg, slot_tcnt, slot_w, group, s0, s1);
}

// How many of a launch's nb bins may be drawn as quadrants, those of
// kSplitRecs records or more: a launch whose bins are all resident at once, or
// nearly, lasts as long as its fullest bin.  A pass of 64 shooters over 33,000
// triangles at hemicube 128 (3,072 bins) takes 85.1 us instead of 88.4.  With
// several times more bins (12,288: 64 shooters at hemicube 256) the largest,
// started first, end before the others do, and with one hemicube (192) the
// quadrants' reading of the whole list cost 1 %.  From 1,024 records on, or
// for more than 1 bin in 16, a pass of 25 shooters over 16,000 triangles lost
// up to 1 %.
// None with the fixed-point rows: which of the fullest bins become quadrants
// depends on the order of atomics (and on clipped triangles binned meanwhile),
// and a quadrant sums the runs of 16 texels in float where a whole tile sums
// those of 32, so the rows' bits would change from run to run.
static uint32_t split_cap(const BinBuffers &bb, uint32_t nb, bool fixed)
{
    return !fixed && bb.tshift == 5 && nb > 512u && nb <= 4096u ? nb / 16u : 0u;
}

void launch_bin(const Geometry &g, uint32_t s0, uint32_t s1, uint32_t h, const float *tri,
                const uint32_t *tri_patch, uint32_t ntri, const float *mvp, const BinBuffers &bb,
                uint32_t *counters, const uint32_t *slot_w, bool whole, bool fixed, hipStream_t st)
{
    const uint32_t b0 = s0 * bb.ntiles, nb = (s1 - s0) * bb.ntiles;
    const uint32_t norder = (nb + 256u * kOrderPer - 1) / (256u * kOrderPer);
    k_order_clip<<<norder + bb.clip_blocks, 256, 0, st>>>(
        norder, nb, b0, split_cap(bb, nb, fixed), bb.order + b0, bb.nbins, g.W, tri, tri_patch, ntri, mvp,
        bin_ctx(bb, h, whole, counters), bb.blk_nrec, bb.nblk * bb.nz,
        bb.pool + (size_t)h * bb.ent_cap, entry_cap(bb, whole), slot_w);
}

void launch_tile(const Geometry &g, uint32_t s0, uint32_t s1, uint32_t h, const uint32_t *nshoot,
                 const BinBuffers &bb, uint32_t small_px, uint32_t *out_ids, float *out_depth,
                 const float *dff, uint32_t rowlen, const uint32_t *slot_pbeg, float *ff,
                 unsigned long long *ffq, uint32_t *hits, uint32_t *counters,
                 const uint32_t *slot_w, const uint32_t *slot_dffo, uint32_t *fblk,
                 uint32_t fstride, hipStream_t st)
{
    const uint32_t nb = (s1 - s0) * bb.ntiles;
    const uint32_t *order = bb.order + (size_t)s0 * bb.ntiles;
    const uint32_t nwg = nb + 3u * split_cap(bb, nb, ffq != nullptr);
    uint32_t *ctr = counters + h * kCntN;
    const BinFacts *facts = reinterpret_cast<const BinFacts *>(ctr + kCntFacts);
    if (ffq)
        k_tile_raster<true><<<nwg, kTileThreads, 0, st>>>(
            g.W, g.TW, g.TH, g.RES, nshoot, bb.recs, bb.bbox, bb.count, bb.list, bb.bin_cap, facts,
            bb.ntx, bb.ntiles, bb.tshift, small_px, out_ids, out_depth, dff, rowlen, slot_pbeg, ff,
            ffq, hits, ctr, order, bb.nbins, slot_w, slot_dffo, nullptr, 0u);
    else
        k_tile_raster<false><<<nwg, kTileThreads, 0, st>>>(
            g.W, g.TW, g.TH, g.RES, nshoot, bb.recs, bb.bbox, bb.count, bb.list, bb.bin_cap, facts,
            bb.ntx, bb.ntiles, bb.tshift, small_px, out_ids, out_depth, dff, rowlen, slot_pbeg, ff,
            ffq, hits, ctr, order, bb.nbins, slot_w, slot_dffo, ff ? fblk : nullptr, fstride);
}

// Deterministic mode: n fixed-point entries (units of 2^-52) into the float
// rows, which are zero where the entries are nonzero; the fixed-point
// entries are left zero.
__global__ __launch_bounds__(256) void k_fold(unsigned long long *__restrict__ ffq,
                                              float *__restrict__ ff, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const unsigned long long q = ffq[i];
        if (q) {
            ff[i] = (float)((double)q * 0x1p-52);
            ffq[i] = 0ull;
        }
    }
}

void launch_fold(unsigned long long *ffq, float *ff, size_t n, hipStream_t st)
{
    size_t blocks = (n + 255) / 256;
    if (blocks > 8192)
        blocks = 8192;
    if (blocks)
        k_fold<<<(unsigned)blocks, 256, 0, st>>>(ffq, ff, n);
}

// ----------------------------------------------------------- ProcessHemicube
// A workgroup takes kReduceChunk consecutive texels of one hemicube's id
// plane (4 bytes per texel), 4 consecutive texels per lane per step.  Equal
// ids in a wavefront's 256 consecutive texels form runs (the span walk of
// Kernel_ProcessHemicube.h:36-49) summed in the lane and across lanes with
// a segmented scan (reduce_quad); each run's
// ΔFF sum and pixel count go into an LDS hash table keyed by id, which also
// merges the runs of the chunk's other rows; the table is then flushed with
// one global atomic per distinct id (the host accumulation of
// Main.cpp:1257-1269 fused in).  A run that finds no free slot adds to the
// global entry directly.  Acc is float, or the 2^-52 fixed point of the
// deterministic mode (LDS and global sums in 64-bit integers).
constexpr uint32_t kReduceChunk = 4096, kReduceSlotsLog2 = 11, kReduceSlots = 1u << kReduceSlotsLog2;
static_assert(kReduceChunk % 1024 == 0, "k_reduce steps of 1024 texels");
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename Acc> __device__ static inline Acc reduce_acc(float f);
template <> __device__ inline float reduce_acc<float>(float f) { return f; }
template <> __device__ inline unsigned long long reduce_acc<unsigned long long>(float f)
{
    return fixed52(f);
}

template <typename Acc>
__global__ __launch_bounds__(256) void k_reduce(uint32_t RES, const uint32_t *__restrict__ nshoot,
                                                const uint32_t *__restrict__ ids_in,
                                                const float *__restrict__ dff, uint32_t npatch,
                                                Acc *__restrict__ ff,
                                                uint32_t *__restrict__ hits,
                                                uint32_t *__restrict__ counters)
{
    __shared__ uint32_t hkey[kReduceSlots], hcnt[kReduceSlots];
    __shared__ Acc hsum[kReduceSlots];
    const uint32_t chunks = (RES + kReduceChunk - 1) / kReduceChunk;
    const uint32_t hi = blockIdx.x / chunks, c0 = (blockIdx.x - hi * chunks) * kReduceChunk;
    if (hi >= *nshoot)
        return;
    for (uint32_t q = threadIdx.x; q < kReduceSlots; q += blockDim.x) {
        hkey[q] = 0u;
        hcnt[q] = 0u;
        hsum[q] = Acc(0);
    }
    __syncthreads();
    const uint32_t *ip = ids_in + (size_t)hi * RES;
    const uint32_t c1 = min(RES, c0 + kReduceChunk);
    const bool with_c = hits != nullptr;
    // one run: into the LDS table (keyed by id), else straight to the row;
    // Main.cpp:1259-1262: an unknown patch id is counted (once per run) and
    // skipped
    auto emit = [&](uint32_t id, float f, uint32_t c) {
        if (!id)
            return;
        if (id - 1 >= npatch) {
            atomicAdd(&counters[kCntUnknown], 1u);
            return;
        }
        const Acc a = reduce_acc<Acc>(f);
        uint32_t h = (id * 2654435761u) >> (32 - kReduceSlotsLog2);
        for (int probe = 0; probe < 16; ++probe, h = (h + 1) & (kReduceSlots - 1)) {
            uint32_t k = hkey[h];
            if (k == 0u)
                k = atomicCAS(&hkey[h], 0u, id);
            if (k == 0u || k == id) {
                atomicAdd(&hsum[h], a);
                if (with_c)
                    atomicAdd(&hcnt[h], c);
                return;
            }
        }
        atomicAdd(&ff[(size_t)hi * npatch + (id - 1)], a);
        if (with_c)
            atomicAdd(&hits[(size_t)hi * npatch + (id - 1)], c);
    };
    // A step covers 1024 texels, 4 consecutive ones per lane (RES and the
    // chunk size are multiples of 4, so the 16-byte loads are aligned and a
    // lane's texels are all in the chunk or all out); the chunk's ids and
    // weights are all loaded before the first step is reduced.
    constexpr uint32_t kSteps = kReduceChunk / (4 * 256);
    u32x4 iv[kSteps];
    float4 fv[kSteps];
#pragma unroll
    for (uint32_t j = 0; j < kSteps; ++j) {
        const uint32_t t = c0 + j * 1024u + threadIdx.x * 4u;
        iv[j] = t < c1 ? __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(ip + t))
                       : u32x4{0u, 0u, 0u, 0u};
        fv[j] = t < c1 ? *reinterpret_cast<const float4 *>(dff + t) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (uint32_t j = 0; j < kSteps; ++j) {
        const uint32_t q[4] = {iv[j].x, iv[j].y, iv[j].z, iv[j].w};
        const float f[4] = {q[0] ? fv[j].x : 0.f, q[1] ? fv[j].y : 0.f, q[2] ? fv[j].z : 0.f,
                            q[3] ? fv[j].w : 0.f};
        reduce_quad(q, f, with_c, emit);
    }
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < kReduceSlots; q += blockDim.x) {
        const uint32_t id = hkey[q];
        if (id == 0u)
            continue;
        atomicAdd(&ff[(size_t)hi * npatch + (id - 1)], hsum[q]);
        if (hits)
            atomicAdd(&hits[(size_t)hi * npatch + (id - 1)], hcnt[q]);
    }
}

void launch_reduce(const Geometry &g, uint32_t K, const uint32_t *nshoot, const uint32_t *ids,
                   const float *dff, uint32_t npatch, float *ff, unsigned long long *ffq,
                   uint32_t *hits, uint32_t *counters, hipStream_t st)
{
    const uint32_t chunks = (g.RES + kReduceChunk - 1) / kReduceChunk;
    if (ffq)
        k_reduce<unsigned long long><<<K * chunks, 256, 0, st>>>(g.RES, nshoot, ids, dff, npatch,
                                                                 ffq, hits, counters);
    else
        k_reduce<float><<<K * chunks, 256, 0, st>>>(g.RES, nshoot, ids, dff, npatch, ff, hits,
                                                    counters);
}

// The ProcessHemicube kernel's own output (Kernel_ProcessHemicube.h:23-69):
// one thread per work-item of the reference (row y of the k stacked
// hemicubes, span gx of TW / nx texels, the last TW - nx * span texels of a
// row left out as there), walking its span texel by texel.  Pass 1 counts the
// slots a work-item reserves (4 per allocation block, runs of id 0 skipped);
// an exclusive scan turns them into offsets; pass 2 writes the triplets
// (hemicube, id - 1, float ΔFF sum of the run in texel order) and the zero
// padding of the last block at those offsets, so the stream comes out in
// work-item order.  Slots at or beyond cap are not written.
__global__ __launch_bounds__(256) void k_runs(uint32_t TW, uint32_t TH, uint32_t nx, uint32_t span,
                                              uint32_t nitems, const uint32_t *__restrict__ item,
                                              const float *__restrict__ dff,
                                              uint32_t *__restrict__ slots,
                                              const uint32_t *__restrict__ offs, uint32_t cap,
                                              uint32_t *__restrict__ th, uint32_t *__restrict__ tid,
                                              float *__restrict__ te)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nitems)
        return;
    const uint32_t y = t / nx, gx = t - y * nx;
    uint32_t x0 = min(gx * span, TW - 1);
    const uint32_t x1 = min(x0 + span, TW);
    const uint32_t *row = item + (size_t)y * TW;
    const float *frow = dff + (size_t)(y % TH) * TW;
    // next: the first slot of the work-item's next allocation block
    uint32_t nruns = 0, next = offs ? offs[t] : 0u, w = 0, space = 0;
    while (x0 < x1) {
        const uint32_t id = row[x0];
        float e = 0.0f;
        while (x0 < x1 && row[x0] == id) {
            if (offs)
                e += frow[x0];
            ++x0;
        }
        if (id == 0u)
            continue;
        ++nruns;
        if (!offs)
            continue;
        if (!space) {
            w = next;
            next += 4u;
            space = 3;
        } else {
            ++w;
            --space;
        }
        if (w < cap) {
            th[w] = y / TH;
            tid[w] = id - 1u;
            te[w] = e;
        }
    }
    if (!offs) {
        slots[t] = (nruns + 3u) & ~3u;
        return;
    }
    for (; space > 0; --space) {
        ++w;
        if (w < cap) {
            th[w] = 0u;
            tid[w] = 0u;
            te[w] = 0.0f;
        }
    }
}

// Exclusive scan of n counts by one workgroup of 1024 threads in chunks of
// 1024 x 8 through LDS: out[i] = sum of in[0..i), out[n] = the total.
__global__ __launch_bounds__(1024) void k_scan_excl(const uint32_t *__restrict__ in,
                                                    uint32_t *__restrict__ out, uint32_t n)
{
    __shared__ uint32_t wsum[16];
    __shared__ uint32_t carry;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (tid == 0)
        carry = 0u;
    __syncthreads();
    for (uint32_t c0 = 0; c0 < n; c0 += 1024u * 8u) {
        uint32_t x[8], sum = 0;
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            const uint32_t i = c0 + tid * 8u + k;
            x[k] = i < n ? in[i] : 0u;
            sum += x[k];
        }
        uint32_t inc = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(inc, d, 64);
            if (lane >= (uint32_t)d)
                inc += o;
        }
        if (lane == 63)
            wsum[w] = inc;
        const uint32_t base = carry;
        __syncthreads();
        if (w == 0) {
            const uint32_t y = lane < 16 ? wsum[lane] : 0u;
            uint32_t z = y;
#pragma unroll
            for (int d = 1; d < 16; d <<= 1) {
                const uint32_t o = __shfl_up(z, d, 64);
                if (lane >= (uint32_t)d)
                    z += o;
            }
            if (lane < 16)
                wsum[lane] = z - y;
            if (lane == 15)
                carry = base + z;
        }
        __syncthreads();
        uint32_t run = base + wsum[w] + inc - sum;
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            const uint32_t i = c0 + tid * 8u + k;
            if (i < n)
                out[i] = run;
            run += x[k];
        }
        __syncthreads(); // wsum and carry are reused by the next chunk
    }
    if (tid == 0)
        out[n] = carry;
}

void launch_runs_count(const Geometry &g, uint32_t k, uint32_t nx, const uint32_t *item,
                       uint32_t *slots, uint32_t *offs, hipStream_t st)
{
    const uint32_t nitems = k * g.TH * nx;
    k_runs<<<(nitems + 255) / 256, 256, 0, st>>>(g.TW, g.TH, nx, g.TW / nx, nitems, item, nullptr,
                                                 slots, nullptr, 0u, nullptr, nullptr, nullptr);
    k_scan_excl<<<1, 1024, 0, st>>>(slots, offs, nitems);
}

void launch_runs_write(const Geometry &g, uint32_t k, uint32_t nx, const uint32_t *item,
                       const float *dff, const uint32_t *offs, uint32_t cap, uint32_t *th,
                       uint32_t *tid, float *te, hipStream_t st)
{
    const uint32_t nitems = k * g.TH * nx;
    k_runs<<<(nitems + 255) / 256, 256, 0, st>>>(g.TW, g.TH, nx, g.TW / nx, nitems, item, dff,
                                                 nullptr, offs, cap, th, tid, te);
}

// ------------------------------------------------------------------ shooting
// Stop test of Main.cpp:1288-1300, run by the lane of the pass's last
// shooter j with its unshot value u before the emitter update (that is
// lastEnergy: the shooter's radiosity including what it received during the
// pass, Main.cpp:1290): u goes to ctl[kCtlLastE..+2]; when a threshold is
// set and |u| (Vector3f::f_Length in float, compared with the double
// threshold as `lastEnergy.f_Length() < 0.1` does) is below it,
// ctl[kCtlStop] makes the later passes no-ops.
__device__ static inline void stop_test(uint32_t *__restrict__ ctl, float u0, float u1, float u2)
{
    ctl[kCtlLastE + 0] = __float_as_uint(u0);
    ctl[kCtlLastE + 1] = __float_as_uint(u1);
    ctl[kCtlLastE + 2] = __float_as_uint(u2);
    const double th = *(const double *)(ctl + kCtlThresh);
    const float len = sqrtf(u0 * u0 + u1 * u1 + u2 * u2);
    if (th > 0.0 && (double)len < th)
        ctl[kCtlStop] = 1u;
}

// Passes and shooters counted by the first thread of a shoot launch.
__device__ static inline void count_pass(uint32_t *__restrict__ ctl, uint32_t n)
{
    if (n == 0)
        return;
    *(unsigned long long *)(ctl + kCtlPassLo) += 1ull;
    *(unsigned long long *)(ctl + kCtlShotLo) += n;
}

// The 64 largest keys of the sorted 64-key lists [l0, l1) by the
// workgroup's waves: each wave merges every nw-th list, loading 16 of them
// at a time (a list whose largest key is not above the 64th of the wave's
// running list cannot contribute),
// then the wave lists are merged pairwise through wl; wave 0 returns the
// result.  Every thread of the workgroup calls it.
__device__ static uint64_t merge_lists_block(const uint64_t *__restrict__ in, uint32_t l0,
                                             uint32_t l1, uint64_t (*wl)[64])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    constexpr int kLoads = 16; // lists a wave loads before merging them
    uint64_t top = 0, thr = 0;
    for (uint32_t lb = l0 + w; lb < l1; lb += (uint32_t)nw * kLoads) {
        uint64_t v[kLoads];
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            const uint32_t l = lb + (uint32_t)(q * nw);
            v[q] = l < l1 ? in[(size_t)l * 64 + lane] : 0ull;
        }
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            if (lane_read_u64(v[q], 0) <= thr)
                continue;
            top = wave_merge_desc(top, v[q]);
            thr = lane_read_u64(top, 63);
        }
    }
    return merge_wave_lists(top, wl);
}

// Wave 0 of a merge: the patches of the k largest POWER keys (a zero key
// fills no slot) and their count.
__device__ static void write_shooters(uint64_t top, uint32_t k, uint32_t *__restrict__ shooters,
                                      uint32_t *__restrict__ nshoot)
{
    const int lane = threadIdx.x & 63;
    const bool ok = (uint32_t)lane < k && (top >> 32) != 0;
    if ((uint32_t)lane < k)
        shooters[lane] = ok ? 0xFFFFFFFFu - (uint32_t)top : 0u;
    const uint64_t m = __ballot(ok);
    if (lane == 0)
        *nshoot = (uint32_t)__popcll(m);
}

__device__ static inline uint64_t wave_max_u64(uint64_t v)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        uint64_t o = __shfl_xor(v, d);
        v = o > v ? o : v;
    }
    return v;
}

// Main.cpp:1251-1295 for all receivers at once: one thread per receiver j
// accumulates the contributions of the pass's shooters, then the shooters
// move their snapshot from unshot to shot.  Every nonzero F entry it reads
// is set back to zero, so the next pass finds the F rows cleared.
// With lists != null (the last launch of a pass whose next pass selects by
// POWER), each workgroup also leaves the sorted 64 largest selection keys
// of its 1,024 receivers' new state in lists[blockIdx.x * 64 + lane], the
// per-workgroup lists k_topk64_scan would make from the stored state, so
// the next pass's selection only merges them; or, with the pool armed, it
// adds every receiver whose key is at least the pool's tau to the pool
// instead; with top1 != 0 (one shooter per pass) each workgroup leaves its
// largest key of rule top1 - 1 in lists[blockIdx.x].  NT threads per workgroup: 1,024 with lists (one merge
// level for up to 262,144 receivers); 256 without lists, and with lists
// when the pool is expected (then lists, left only when the pool is not
// armed, cover 256 receivers each).
constexpr uint32_t kShootListThreads = 1024;

template <uint32_t NT>
__global__ __launch_bounds__(NT) void k_shoot(uint32_t mode, const uint32_t *__restrict__ shooters,
                                               const uint32_t *__restrict__ nshoot,
                                               const float *__restrict__ snap,
                                               float *__restrict__ ff,
                                               uint32_t *__restrict__ fblk, uint32_t fstride,
                                               const float *__restrict__ refl,
                                               const float *__restrict__ area, uint32_t npatch,
                                               float *__restrict__ unshot,
                                               float *__restrict__ shot, uint32_t *__restrict__ ctl,
                                               uint32_t sbeg, uint32_t send, uint32_t last,
                                               uint64_t *__restrict__ lists,
                                               SelPool *__restrict__ pool, uint32_t top1)
{
    __shared__ uint32_t sid[RAD_MAX_K];
    __shared__ float sc[RAD_MAX_K * 4];
    __shared__ uint64_t wl[NT / 64][64];
    __shared__ uint32_t npool, gbase;
    const uint32_t pooled = lists && pool ? pool->armed : 0u;
    if (threadIdx.x == 0)
        npool = 0u;
    uint32_t n = *nshoot;
    for (uint32_t s = threadIdx.x; s < n; s += blockDim.x) {
        uint32_t i = shooters[s];
        sid[s] = i;
        if (mode == RAD_MODE_REFERENCE) {
            sc[4 * s + 0] = refl[3 * (size_t)i + 0];
            sc[4 * s + 1] = refl[3 * (size_t)i + 1];
            sc[4 * s + 2] = refl[3 * (size_t)i + 2];
        }
        sc[4 * s + 3] = area[i];
    }
    __syncthreads();
    if (last && blockIdx.x == 0 && threadIdx.x == 0)
        count_pass(ctl, n);
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    // the wavefront's 64 receivers are one block of the F-block flags
    const uint32_t blk = (blockIdx.x * blockDim.x + (threadIdx.x & ~63u)) >> 6;
    const bool live = j < npatch;
    float u0 = 0.f, u1 = 0.f, u2 = 0.f, r0 = 0.f, r1 = 0.f, r2 = 0.f, inv_aj = 0.f;
    if (live) {
        u0 = unshot[3 * (size_t)j + 0];
        u1 = unshot[3 * (size_t)j + 1];
        u2 = unshot[3 * (size_t)j + 2];
        if (mode != RAD_MODE_REFERENCE) {
            r0 = refl[3 * (size_t)j + 0];
            r1 = refl[3 * (size_t)j + 1];
            r2 = refl[3 * (size_t)j + 2];
            inv_aj = 1.0f / area[j];
        }
    }
    // Shooters [sbeg, send) are added here: a pass may be shot in two
    // launches, the first half's as soon as its tiles are done, the second
    // (last) one adding the rest and moving the shooters' energy; the sums
    // are the same float additions in the same order either way.
    // Shooters are taken in groups of 64 and, within a group, in shooter
    // order; only those whose F block of these receivers is flagged are
    // read (an unflagged block is zero), 8 at a time (independent loads in
    // flight).  Entries are added in shooter order, skipping zeros, so the
    // sums are those of reading every entry.  The nonzero entries of a group
    // are set back to zero after the group's last read (a load issued after
    // a store waits for it), and the group's flags are cleared, which leaves
    // the F rows zero for the next pass (its clear skips them).
    const uint32_t se = min(n, send);
    if (blk * 64u < npatch) {
        for (uint32_t g0 = sbeg; g0 < se; g0 += 64) {
            const uint32_t g1 = min(se, g0 + 64);
            uint32_t *const fl = fblk ? fblk + (size_t)blk * fstride + g0 : nullptr;
            const bool mine = g0 + lane < g1;
            uint64_t todo;
            if (fl) {
                const bool set = mine && fl[lane] != 0u;
                todo = __ballot(set);
                if (set)
                    fl[lane] = 0u;
            } else {
                todo = __ballot(mine);
            }
            uint64_t nz = 0;
            while (todo) {
                uint32_t ss[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    ss[q] = todo ? g0 + (uint32_t)__ffsll((long long)todo) - 1u : ~0u;
                    todo &= todo - 1;
                }
                float fb[8];
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    fb[q] = live && ss[q] != ~0u ? ff[(size_t)ss[q] * npatch + j] : 0.0f;
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const uint32_t s = ss[q];
                    const float f = fb[q];
                    if (s == ~0u || f == 0.0f)
                        continue;
                    nz |= 1ull << (s - g0);
                    float d0 = snap[3 * s + 0], d1 = snap[3 * s + 1], d2 = snap[3 * s + 2];
                    if (mode == RAD_MODE_REFERENCE) {
                        // Main.cpp:1274: radiosity += dB * F * 0.3 * colour_emitter
                        u0 += d0 * f * 0.3f * sc[4 * s + 0];
                        u1 += d1 * f * 0.3f * sc[4 * s + 1];
                        u2 += d2 * f * 0.3f * sc[4 * s + 2];
                    } else {
                        float g = f * (sc[4 * s + 3] * inv_aj);
                        u0 += r0 * d0 * g;
                        u1 += r1 * d1 * g;
                        u2 += r2 * d2 * g;
                    }
                }
            }
            for (uint64_t m = nz; m; m &= m - 1)
                ff[(size_t)(g0 + (uint32_t)__ffsll((long long)m) - 1) * npatch + j] = 0.0f;
        }
    }
    if (last) {
        // Main.cpp:1287-1295
        if (live && n && sid[n - 1] == j)
            stop_test(ctl, u0, u1, u2);
        // the pass's shooters among the wavefront's receivers, in order
        for (uint32_t s0 = 0; s0 < n; s0 += 64) {
            const bool here = s0 + lane < n && (sid[s0 + lane] >> 6) == blk;
            for (uint64_t m = __ballot(here); m; m &= m - 1) {
                const uint32_t s = s0 + (uint32_t)__ffsll((long long)m) - 1u;
                if (live && sid[s] == j) {
                    float d0 = snap[3 * s + 0], d1 = snap[3 * s + 1], d2 = snap[3 * s + 2];
                    shot[3 * (size_t)j + 0] += d0;
                    shot[3 * (size_t)j + 1] += d1;
                    shot[3 * (size_t)j + 2] += d2;
                    u0 -= d0;
                    u1 -= d1;
                    u2 -= d2;
                }
            }
        }
    }
    if (live) {
        unshot[3 * (size_t)j + 0] = u0;
        unshot[3 * (size_t)j + 1] = u1;
        unshot[3 * (size_t)j + 2] = u2;
    }
    if (!lists)
        return;
    // sel_key of the state just stored
    uint64_t key = 0ull;
    if (live && top1 == 1u + RAD_SELECT_REFERENCE) {
        key = ((uint64_t)__float_as_uint(u0 * u0 + u1 * u1 + u2 * u2) << 32) | j;
    } else if (live) {
        float e = area[j] * (u0 + u1 + u2);
        if (!(e > 0.0f))
            e = 0.0f;
        key = ((uint64_t)__float_as_uint(e) << 32) | (0xFFFFFFFFu - j);
    }
    if (top1) {
        key = wave_max_u64(key);
        if (lane == 0)
            wl[0][w] = key;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (uint32_t q = 1; q < NT / 64; ++q)
                key = wl[0][q] > key ? wl[0][q] : key;
            lists[blockIdx.x] = key;
        }
        return;
    }
    if (pooled) {
        // every receiver whose key is at least tau (a positive power) goes
        // to this workgroup's pool region
        const uint64_t tau = pool->tau;
        const bool c = live && key >= tau;
        const uint64_t m = __ballot(c);
        uint32_t local = 0u;
        if (m) {
            uint32_t base = 0u;
            if (lane == 0)
                base = atomicAdd(&npool, (uint32_t)__popcll(m));
            base = (uint32_t)__shfl((int)base, 0);
            local = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        }
        __syncthreads();
        if (threadIdx.x == 0)
            gbase = npool ? atomicAdd(&pool->count, npool) : 0u;
        __syncthreads();
        const uint32_t idx = gbase + local;
        if (c && idx < kPoolCap)
            pool->keys[idx] = key;
        return;
    }
    uint64_t top = wave_sort_desc(key);
    wl[w][lane] = top;
    for (uint32_t h = NT / 128; h >= 1; h >>= 1) {
        __syncthreads();
        if (w < h)
            top = wave_merge_desc(wl[w][lane], wl[w + h][lane]);
        __syncthreads();
        if (w < h)
            wl[w][lane] = top;
    }
    if (w == 0)
        lists[(size_t)blockIdx.x * 64 + lane] = top;
}

uint32_t shoot_lists(uint32_t npatch, bool pooled)
{
    const uint32_t nt = pooled ? 256u : kShootListThreads;
    return (npatch + nt - 1) / nt;
}

void launch_shoot(uint32_t mode, uint32_t K, const uint32_t *shooters, const uint32_t *nshoot,
                  const float *snap, float *ff, uint32_t *fblk, const float *refl,
                  const float *area, uint32_t npatch, float *unshot, float *shot, uint32_t *ctl,
                  uint32_t sbeg, uint32_t send, bool last, uint64_t *lists, SelPool *pool,
                  uint32_t top1, hipStream_t st)
{
    if (lists && !pool && !top1)
        k_shoot<kShootListThreads><<<shoot_lists(npatch, false), kShootListThreads, 0, st>>>(
            mode, shooters, nshoot, snap, ff, fblk, K, refl, area, npatch, unshot, shot, ctl,
            sbeg, send, last ? 1u : 0u, lists, nullptr, 0u);
    else
        k_shoot<256><<<(npatch + 255) / 256, 256, 0, st>>>(mode, shooters, nshoot, snap, ff, fblk,
                                                          K, refl, area, npatch, unshot, shot,
                                                          ctl, sbeg, send, last ? 1u : 0u, lists,
                                                          pool, top1);
}

__device__ static inline uint64_t sel_key(uint32_t rule, const float *unshot, const float *area,
                                          uint32_t j);

// The 64 largest of n unsorted keys: each wave takes every nw-th batch of
// 64, loading 8 batches at a time, and sorts and merges in those that hold
// a key above its running 64th; wave 0 returns the result.  Every thread of
// the workgroup calls it.
__device__ static uint64_t select_keys_block(const uint64_t *__restrict__ pk, uint32_t n,
                                             uint64_t (*wl)[64])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    constexpr int kLoads = 8;
    const uint32_t step = (uint32_t)nw * 64;
    uint64_t top = 0, thr = 0;
    for (uint32_t b0 = (uint32_t)w * 64; b0 < n; b0 += step * kLoads) {
        uint64_t v[kLoads];
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            const uint32_t i = b0 + (uint32_t)q * step + lane;
            v[q] = i < n ? pk[i] : 0ull;
        }
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            if (__ballot(v[q] > thr) == 0)
                continue;
            top = wave_merge_desc(top, wave_sort_desc(v[q]));
            thr = lane_read_u64(top, 63);
        }
    }
    return merge_wave_lists(top, wl);
}

// The 64 largest POWER keys of all npatch patches, by one workgroup (the
// pool's fallback): as k_topk64_scan, four batches loaded at a time.
__device__ static uint64_t select_all_block(const float *__restrict__ unshot,
                                            const float *__restrict__ area, uint32_t npatch,
                                            uint64_t (*wl)[64])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const uint32_t step = (uint32_t)nw * 64;
    uint64_t top = 0, thr = 0;
    for (uint32_t base = (uint32_t)w * 64; base < npatch; base += 4 * step) {
        uint64_t kk[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t j = base + (uint32_t)q * step + lane;
            kk[q] = j < npatch ? sel_key(RAD_SELECT_POWER, unshot, area, j) : 0ull;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (__ballot(kk[q] > thr) == 0)
                continue;
            top = wave_merge_desc(top, wave_sort_desc(kk[q]));
            thr = lane_read_u64(top, 63);
        }
    }
    return merge_wave_lists(top, wl);
}

// Arms the pool after the merge of nlists sorted lists whose 64th largest
// key is t64.  The lists hold a subset of the state's keys, so at least as
// many keys of the state as of the lists are >= any tau.  tau steps down
// from t64 by 1/8 octave of power (2^20 in the float bits of the key's
// upper word), at most 8 octaves, until the lists hold `target` keys >= tau
// (t64 itself when target <= 64).  A tau of zero power is never armed.
// hist: 64 words of LDS.  Every thread of the workgroup calls it.
__device__ static void arm_pool(const uint64_t *__restrict__ in, uint32_t nlists, uint64_t t64,
                                uint32_t target, SelPool *__restrict__ pool, uint32_t *hist)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const uint32_t th = (uint32_t)(t64 >> 32);
    if (threadIdx.x < 64)
        hist[threadIdx.x] = 0u;
    __syncthreads();
    for (uint32_t l = (uint32_t)w; l < nlists; l += (uint32_t)nw) {
        const uint64_t e = in[(size_t)l * 64 + lane];
        const uint32_t eh = (uint32_t)(e >> 32);
        // bucket (th - eh) >> 20 of the keys below t64 within 8 octaves
        // (64: none)
        uint32_t b = 64u;
        if (e < t64 && eh != 0u && th - eh < (64u << 20))
            b = (th - eh) >> 20;
        // a list is sorted, so a bucket's keys are a run of lanes: the run's
        // first lane adds its length
        const uint32_t prev = (uint32_t)__shfl_up((int)b, 1);
        const bool start = lane == 0 || prev != b;
        const uint64_t starts = __ballot(start);
        if (start && b < 64u) {
            const uint64_t after = lane == 63 ? 0ull : starts & (~0ull << (lane + 1));
            const uint32_t next = after ? (uint32_t)__ffsll((long long)after) - 1u : 64u;
            atomicAdd(&hist[b], next - (uint32_t)lane);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t armed = 0u;
        uint64_t tau = 0ull;
        if (th != 0u) {
            uint32_t c = 64u; // the merged 64 are >= t64
            if (c >= target) {
                tau = t64;
                armed = 1u;
            }
            for (uint32_t b = 0; b < 64u && !armed; ++b) {
                c += hist[b];
                if (c >= target) {
                    const uint32_t drop = (b + 1u) << 20;
                    if (th > drop) {
                        tau = (uint64_t)(th - drop + 1u) << 32;
                        armed = 1u;
                    }
                    break;
                }
            }
        }
        if (armed) {
            pool->tau = tau;
            pool->arms += 1u;
        }
        pool->armed = armed;
    }
}

// The start of the pass after one whose last shoot left per-workgroup lists
// or pooled, in one workgroup: the selection and what k_prepare_clear does
// (the stop gate, the shooters' snapshots and MVPs, bin counts and pass
// counters cleared; no F rows or hits, which the shoot leaves zero).
// The selection takes the K largest POWER keys (as k_topk64_merge):
//  - pooled: from the pool when it holds K .. pool_cap keys, which are then
//    exactly the keys >= tau, so their K largest are the state's; otherwise
//    from a scan of every patch, and the pool is disarmed (the next shoot
//    leaves lists);
//  - else: the merge of the lists, then the pool armed for `target` keys
//    (target 0: disarmed).
__global__ __launch_bounds__(1024) void k_next_pass(const uint64_t *__restrict__ lists,
                                                    uint32_t nlists, NextPass np,
                                                    const float *__restrict__ unshot,
                                                    const float *__restrict__ area,
                                                    uint32_t npatch,
                                                    const uint32_t *__restrict__ ctl,
                                                    SelPool *__restrict__ pool,
                                                    uint32_t lists_only, uint32_t target,
                                                    uint32_t pool_cap)
{
    __shared__ uint64_t wl[16][64];
    __shared__ uint32_t hist[64], ssel[64], sn;
    __shared__ uint64_t t64s;
    const int lane = threadIdx.x & 63;
    const uint32_t t = threadIdx.x;
    const uint32_t stop = ctl[kCtlStop];
    const uint32_t pooled = lists_only ? 0u : pool->armed;
    uint64_t best;
    if (pooled) {
        const uint32_t n = pool->count;
        if (n >= np.K && n <= pool_cap) {
            best = select_keys_block(pool->keys, n, wl);
            if (t == 0)
                pool->hits += 1u;
        } else {
            best = select_all_block(unshot, area, npatch, wl);
            if (t == 0) {
                pool->falls += 1u;
                pool->armed = 0u;
            }
        }
    } else {
        best = merge_lists_block(lists, 0u, nlists, wl);
        if (target) {
            if (t == 0)
                t64s = lane_read_u64(best, 63);
            __syncthreads();
            arm_pool(lists, nlists, t64s, target, pool, hist);
        } else if (t == 0) {
            pool->armed = 0u;
        }
    }
    // wave 0: the shooters (as write_shooters) into memory and LDS; the
    // stop gate of k_prepare_clear sets the count to 0
    if (t < 64) {
        const bool ok = (uint32_t)lane < np.K && (best >> 32) != 0;
        const uint32_t id = ok ? 0xFFFFFFFFu - (uint32_t)best : 0u;
        if ((uint32_t)lane < np.K) {
            np.shooters[lane] = id;
            ssel[lane] = id;
        }
        const uint32_t m = stop ? 0u : (uint32_t)__popcll(__ballot(ok));
        if (lane == 0) {
            *np.nshoot = m;
            sn = m;
        }
    }
    __syncthreads();
    // every read of the pool count is done: the next shoot pools from zero
    if (t == 0)
        pool->count = 0u;
    for (uint32_t i = t; i < np.K * 5; i += blockDim.x)
        prepare_item(i, np.K, ssel, &sn, np.frames, unshot, np.snap, np.mvp, nullptr);
    clear_range(t, blockDim.x, np.bin_count, np.nbins, nullptr, nullptr, 0, np.counters);
}

void launch_next_pass(const uint64_t *lists, uint32_t nlists, const NextPass &np,
                      const float *unshot, const float *area, uint32_t npatch,
                      const uint32_t *ctl, SelPool *pool, bool lists_only, uint32_t target,
                      uint32_t pool_cap, hipStream_t st)
{
    k_next_pass<<<1, 1024, 0, st>>>(lists, nlists, np, unshot, area, npatch, ctl, pool,
                                    lists_only ? 1u : 0u, target,
                                    pool_cap < kPoolCap ? pool_cap : kPoolCap);
}


// ----------------------------------------------------------------- selection
// Single-shooter selection, one packed 64-bit key per patch reduced with
// atomicMax into sel[0] (cleared by the previous k_sel_reset):
//  RAD_SELECT_REFERENCE: key |dB|^2 (Vector.h:356-359), ties to the larger
//    index; a zero maximum selects patch 0.  This is what the list rule of
//    ModelContainer.cpp:263-298 yields for count = 1.
//  RAD_SELECT_POWER: key A*(r+g+b), ties to the smaller index.
// The FP64 residual numerator and denominator are accumulated alongside.
__device__ static inline uint64_t sel_key(uint32_t rule, const float *unshot, const float *area,
                                          uint32_t j)
{
    float u0 = unshot[3 * (size_t)j + 0], u1 = unshot[3 * (size_t)j + 1],
          u2 = unshot[3 * (size_t)j + 2];
    if (rule == RAD_SELECT_REFERENCE) {
        float e = u0 * u0 + u1 * u1 + u2 * u2;
        return ((uint64_t)__float_as_uint(e) << 32) | j;
    }
    float e = area[j] * (u0 + u1 + u2);
    if (!(e > 0.0f))
        e = 0.0f;
    return ((uint64_t)__float_as_uint(e) << 32) | (0xFFFFFFFFu - j);
}

__device__ static inline uint32_t sel_decode(uint32_t rule, uint64_t key)
{
    if (rule == RAD_SELECT_REFERENCE)
        return (key >> 32) == 0 ? 0u : (uint32_t)key;
    return 0xFFFFFFFFu - (uint32_t)key;
}

// The start of the pass after one whose shoot left each workgroup's largest
// key: the single shooter and what k_prepare_clear does, as k_next_pass.
__global__ __launch_bounds__(1024) void k_next_top1(uint32_t rule, const uint64_t *__restrict__ keys,
                                                    uint32_t nkeys, NextPass np,
                                                    const float *__restrict__ unshot,
                                                    const uint32_t *__restrict__ ctl)
{
    __shared__ uint64_t wl[16];
    __shared__ uint32_t ssel, sn;
    const uint32_t t = threadIdx.x;
    const uint32_t stop = ctl[kCtlStop];
    uint64_t best = 0;
    for (uint32_t i = t; i < nkeys; i += blockDim.x)
        best = keys[i] > best ? keys[i] : best;
    best = wave_max_u64(best);
    if ((t & 63u) == 0)
        wl[t >> 6] = best;
    __syncthreads();
    if (t == 0) {
        for (uint32_t q = 1; q < 16; ++q)
            best = wl[q] > best ? wl[q] : best;
        ssel = sel_decode(rule, best);
        sn = stop ? 0u : 1u;
        np.shooters[0] = ssel;
        *np.nshoot = sn;
    }
    __syncthreads();
    if (t < 5)
        prepare_item(t, 1u, &ssel, &sn, np.frames, unshot, np.snap, np.mvp, nullptr);
    clear_range(t, blockDim.x, np.bin_count, np.nbins, nullptr, nullptr, 0, np.counters);
}

void launch_next_top1(uint32_t rule, const uint64_t *keys, uint32_t nkeys, const NextPass &np,
                      const float *unshot, const uint32_t *ctl, hipStream_t st)
{
    k_next_top1<<<1, 1024, 0, st>>>(rule, keys, nkeys, np, unshot, ctl);
}

template <typename T> __device__ static inline T wave_sum(T v)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1)
        v += __shfl_xor(v, d);
    return v;
}

// Block-level reduction of (max key, num, den) for 256 threads; the result
// is valid in thread 0.
__device__ static inline void block_reduce3(uint64_t &best, double &num, double &den)
{
    __shared__ uint64_t sb[4];
    __shared__ double sn[4], sd[4];
    best = wave_max_u64(best);
    num = wave_sum(num);
    den = wave_sum(den);
    int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sb[w] = best;
        sn[w] = num;
        sd[w] = den;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < (int)(blockDim.x >> 6); ++q) {
            best = sb[q] > best ? sb[q] : best;
            num += sn[q];
            den += sd[q];
        }
    }
}

// Stage 1: one partial (max key, residual numerator, denominator) per block.
__global__ __launch_bounds__(256) void k_select_top1(uint32_t rule, const float *__restrict__ unshot,
                                                     const float *__restrict__ area,
                                                     const float *__restrict__ emis,
                                                     uint32_t npatch, uint64_t *__restrict__ pkey,
                                                     double *__restrict__ pres)
{
    uint64_t best = 0;
    double num = 0.0, den = 0.0;
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < npatch;
         j += gridDim.x * blockDim.x) {
        uint64_t k = sel_key(rule, unshot, area, j);
        best = k > best ? k : best;
        double a = (double)area[j];
        num += a * ((double)unshot[3 * (size_t)j] + (double)unshot[3 * (size_t)j + 1] +
                    (double)unshot[3 * (size_t)j + 2]);
        den += a * ((double)emis[3 * (size_t)j] + (double)emis[3 * (size_t)j + 1] +
                    (double)emis[3 * (size_t)j + 2]);
    }
    block_reduce3(best, num, den);
    if (threadIdx.x == 0) {
        pkey[blockIdx.x] = best;
        pres[2 * blockIdx.x] = num;
        pres[2 * blockIdx.x + 1] = den;
    }
}

// Stage 2 (one block): reduce the partials, decode the shooter.
__global__ __launch_bounds__(256) void k_select_final(uint32_t rule, uint32_t nparts,
                                                      const uint64_t *__restrict__ pkey,
                                                      const double *__restrict__ pres,
                                                      uint32_t *__restrict__ shooters,
                                                      uint32_t *__restrict__ nshoot,
                                                      double *__restrict__ resid)
{
    uint64_t best = 0;
    double num = 0.0, den = 0.0;
    for (uint32_t b = threadIdx.x; b < nparts; b += blockDim.x) {
        best = pkey[b] > best ? pkey[b] : best;
        num += pres[2 * b];
        den += pres[2 * b + 1];
    }
    block_reduce3(best, num, den);
    if (threadIdx.x == 0) {
        if (shooters) {
            shooters[0] = sel_decode(rule, best);
            nshoot[0] = 1;
        }
        resid[0] = num;
        resid[1] = den;
    }
}

void launch_select_top1(uint32_t rule, const float *unshot, const float *area, const float *emis,
                        uint32_t npatch, uint32_t *shooters, uint32_t *nshoot, double *partials,
                        uint64_t *pkeys, uint32_t *counter, double *resid, int nblocks,
                        hipStream_t st)
{
    (void)counter;
    k_select_top1<<<nblocks, 256, 0, st>>>(rule, unshot, area, emis, npatch, pkeys, partials);
    k_select_final<<<1, 256, 0, st>>>(rule, (uint32_t)nblocks, pkeys, partials, shooters, nshoot,
                                      resid);
}

void launch_residual(const float *unshot, const float *area, const float *emis, uint32_t npatch,
                     double *partials, uint32_t *counter, double *resid, int nblocks,
                     hipStream_t st)
{
    (void)counter;
    uint64_t *pkeys = (uint64_t *)(partials + 2 * nblocks);
    k_select_top1<<<nblocks, 256, 0, st>>>(RAD_SELECT_POWER, unshot, area, emis, npatch, pkeys,
                                           partials);
    k_select_final<<<1, 256, 0, st>>>(RAD_SELECT_POWER, (uint32_t)nblocks, pkeys, partials,
                                      nullptr, nullptr, resid);
}

// ------------------------------------------------------------ top-K (POWER)
// Each block sorts a chunk of kTopkChunk packed keys descending in LDS
// (bitonic) and keeps its first k; passes repeat over the candidates until
// one block remains, which writes the shooters.  Keys are
// (A*(r+g+b) bits << 32 | ~index): larger power first, ties to the smaller
// index; only keys with positive power are selected.
constexpr int kTopkChunk = 2048;
size_t topk_cand_half(uint32_t npatch, uint32_t k);

__device__ static void bitonic_desc(uint64_t *a, int n)
{
    for (int size = 2; size <= n; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = threadIdx.x; i < n / 2; i += blockDim.x) {
                int lo = 2 * i - (i & (stride - 1));
                int hi = lo + stride;
                bool desc = ((lo & size) == 0);
                uint64_t x = a[lo], y = a[hi];
                if ((x < y) == desc) {
                    a[lo] = y;
                    a[hi] = x;
                }
            }
            __syncthreads();
        }
}

__global__ __launch_bounds__(256) void k_topk_pass(const float *__restrict__ unshot,
                                                   const float *__restrict__ area,
                                                   const uint64_t *__restrict__ in, uint32_t nin,
                                                   uint32_t k, uint64_t *__restrict__ out,
                                                   uint32_t *__restrict__ shooters,
                                                   uint32_t *__restrict__ nshoot)
{
    __shared__ uint64_t buf[kTopkChunk];
    uint32_t base = blockIdx.x * kTopkChunk;
    for (int i = threadIdx.x; i < kTopkChunk; i += blockDim.x) {
        uint32_t j = base + i;
        uint64_t key = 0;
        if (j < nin)
            key = in ? in[j] : sel_key(RAD_SELECT_POWER, unshot, area, j);
        buf[i] = key;
    }
    __syncthreads();
    bitonic_desc(buf, kTopkChunk);
    if (shooters) {
        // final pass (one block)
        __shared__ uint32_t cnt;
        if (threadIdx.x == 0)
            cnt = 0;
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < k; i += blockDim.x) {
            uint64_t key = buf[i];
            bool ok = (key >> 32) != 0;
            shooters[i] = ok ? 0xFFFFFFFFu - (uint32_t)key : 0u;
            if (ok)
                atomicAdd(&cnt, 1u);
        }
        __syncthreads();
        if (threadIdx.x == 0)
            *nshoot = cnt;
    } else {
        for (uint32_t i = threadIdx.x; i < k; i += blockDim.x)
            out[(size_t)blockIdx.x * k + i] = buf[i];
    }
}

// ---- K <= 64: one sorted list of 64 keys per wavefront, one key per lane
// (lane 0 largest).  A batch of 64 new keys is sorted with a shuffle bitonic
// network and merged into the list (max against the reversed batch gives a
// bitonic sequence holding the top 64 of both; a half-cleaner pass sorts
// it).  Waves scan the patches (a batch with no key above the wave's 64th
// is skipped), each workgroup merges its wave lists in LDS, then one
// workgroup merges the workgroup lists.  The keys are distinct (they hold
// the patch index), so the result does not depend on the merge order.
constexpr uint32_t kTopkScanWaves = 8;

__global__ __launch_bounds__(kTopkScanWaves * 64) void k_topk64_scan(const float *__restrict__ unshot,
                                                     const float *__restrict__ area,
                                                     uint32_t npatch, uint64_t *__restrict__ out)
{
    const int lane = threadIdx.x & 63;
    const uint32_t gw = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const uint32_t nw = gridDim.x * (blockDim.x >> 6);
    __shared__ uint64_t wl[kTopkScanWaves][64];
    uint64_t top = 0, thr = 0; // thr: the list's 64th key
    for (uint32_t base = gw * 64; base < npatch; base += nw * 64) {
        uint32_t j = base + lane;
        uint64_t key = j < npatch ? sel_key(RAD_SELECT_POWER, unshot, area, j) : 0ull;
        if (__ballot(key > thr) == 0)
            continue;
        top = wave_merge_desc(top, wave_sort_desc(key));
        thr = lane_read_u64(top, 63);
    }
    // the workgroup's wave lists: pairwise merge levels in LDS
    const int w = threadIdx.x >> 6;
    wl[w][lane] = top;
    for (int h = (int)kTopkScanWaves / 2; h >= 1; h >>= 1) {
        __syncthreads();
        if (w < h)
            top = wave_merge_desc(wl[w][lane], wl[w + h][lane]);
        __syncthreads();
        if (w < h)
            wl[w][lane] = top;
    }
    if (w == 0)
        out[(size_t)blockIdx.x * 64 + lane] = top;
}

// Merges nlists sorted lists of 64 (in[l * 64 + lane]) per workgroup; the
// last workgroup level (gridDim.x == 1) writes the shooters.
__global__ __launch_bounds__(1024) void k_topk64_merge(const uint64_t *__restrict__ in,
                                                       uint32_t nlists, uint32_t per_block,
                                                       uint32_t k, uint64_t *__restrict__ out,
                                                       uint32_t *__restrict__ shooters,
                                                       uint32_t *__restrict__ nshoot)
{
    __shared__ uint64_t wl[16][64];
    const uint32_t l0 = blockIdx.x * per_block;
    const uint32_t l1 = l0 + per_block < nlists ? l0 + per_block : nlists;
    const uint64_t top = merge_lists_block(in, l0, l1, wl);
    if ((threadIdx.x >> 6) != 0)
        return;
    if (shooters)
        write_shooters(top, k, shooters, nshoot);
    else
        out[(size_t)blockIdx.x * 64 + (threadIdx.x & 63)] = top;
}

void launch_select_topk(uint32_t rule, const float *unshot, const float *area, const float *emis,
                        uint32_t npatch, uint32_t k, uint32_t *shooters, uint32_t *nshoot,
                        uint64_t *cand, double *partials, uint32_t *counter, double *resid,
                        hipStream_t st)
{
    (void)rule;
    (void)emis;
    (void)partials;
    (void)counter;
    (void)resid;
    if (k <= 64) {
        // wave lists: about four batches of 64 patches per wave
        uint32_t waves = (npatch + 255) / 256;
        if (waves < kTopkScanWaves)
            waves = kTopkScanWaves;
        uint32_t blocks = (waves + kTopkScanWaves - 1) / kTopkScanWaves;
        if ((size_t)blocks * 64 > topk_cand_half(npatch, k))
            blocks = (uint32_t)(topk_cand_half(npatch, k) / 64);
        uint64_t *a = cand, *b = cand + topk_cand_half(npatch, k);
        k_topk64_scan<<<blocks, kTopkScanWaves * 64, 0, st>>>(unshot, area, npatch, a);
        uint32_t nl = blocks;
        while (nl > 256) {
            uint32_t per = 64, nb = (nl + per - 1) / per;
            k_topk64_merge<<<nb, 1024, 0, st>>>(a, nl, per, k, b, nullptr, nullptr);
            uint64_t *t = a;
            a = b;
            b = t;
            nl = nb;
        }
        k_topk64_merge<<<1, 1024, 0, st>>>(a, nl, nl, k, nullptr, shooters, nshoot);
        return;
    }
    // cand holds two ping-pong halves of topk_cand_size(npatch, k) entries
    uint32_t n = npatch;
    const uint64_t *in = nullptr;
    uint64_t *bufs[2] = {cand, cand + topk_cand_half(npatch, k)};
    int which = 0;
    while (true) {
        uint32_t nb = (n + kTopkChunk - 1) / kTopkChunk;
        if (nb <= 1) {
            k_topk_pass<<<1, 256, 0, st>>>(unshot, area, in, n, k, nullptr, shooters, nshoot);
            return;
        }
        uint64_t *out = bufs[which];
        k_topk_pass<<<nb, 256, 0, st>>>(unshot, area, in, n, k, out, nullptr, nullptr);
        in = out;
        n = nb * k;
        which ^= 1;
    }
}

size_t topk_cand_half(uint32_t npatch, uint32_t k)
{
    size_t nb = ((size_t)npatch + kTopkChunk - 1) / kTopkChunk;
    size_t bitonic = nb * k + 1;
    // the wave-list path keeps 64 keys per wave, one wave per 256 patches
    size_t waves = ((size_t)npatch + 255) / 256;
    size_t lists = (waves < 4 ? 4 : waves) + 3;
    return bitonic > lists * 64 ? bitonic : lists * 64;
}

// ----------------------------------------------- reference rule, K > 1
// ModelContainer.cpp:263-298 simulated exactly by one workgroup.  The
// list's last (smallest) key never decreases during the scan, so a chunk's
// candidates can be prefiltered in parallel against the value at the chunk
// start; the survivors are then inserted one by one in index order by the
// first wavefront with the list's push_back / stable sort / reverse /
// truncate semantics: every run of equal keys reverses its order and the new
// element goes first among its equals.
//
// Serial by its nature (an insertion decides the next test), so what counts
// is the time of one insertion: the list is held one entry per lane (R per
// lane beyond 64), every entry finds its new place from ballots of the run
// starts, the list is permuted through LDS, and the next candidate the list
// takes is found by one ballot.  772 patches, K = 10: 16 us, where one lane
// moving the entries one by one through LDS took 180.
constexpr uint32_t kRefThreads = 1024;

template <int R>
__device__ static inline void reference_insert(float (&key)[R], uint32_t (&id)[R], uint32_t &n,
                                               uint32_t k, float ek, uint32_t eid, float *lk,
                                               uint32_t *li)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint64_t head[R];
    uint32_t p = 0; // the new element's place: after every larger key
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t i = (uint32_t)r * 64u + lane;
        float prev = __shfl_up(key[r], 1, 64);
        if (r > 0 && lane == 0)
            prev = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(key[r ? r - 1 : 0]), 63));
        head[r] = __ballot(i < n && (i == 0 || key[r] != prev));
        p += (uint32_t)__popcll(__ballot(i < n && key[r] > ek));
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t i = (uint32_t)r * 64u + lane;
        const uint64_t upto = (2ull << lane) - 1ull;
        // the entry's run of equal keys [g0, g1), reversed
        uint32_t g0 = 0, g1 = n;
        bool found = false;
#pragma unroll
        for (int q = r; q >= 0; --q) {
            const uint64_t m = q == r ? head[q] & upto : head[q];
            if (!found && m) {
                g0 = (uint32_t)q * 64u + 63u - (uint32_t)__clzll(m);
                found = true;
            }
        }
        found = false;
#pragma unroll
        for (int q = r; q < R; ++q) {
            const uint64_t m = q == r ? head[q] & ~upto : head[q];
            if (!found && m) {
                g1 = (uint32_t)q * 64u + (uint32_t)__ffsll((long long)m) - 1u;
                found = true;
            }
        }
        const uint32_t to = g0 + g1 - 1u - i + (key[r] <= ek ? 1u : 0u);
        if (i < n && to < k) {
            lk[to] = key[r];
            li[to] = id[r];
        }
    }
    if (lane == 0 && p < k) {
        lk[p] = ek;
        li[p] = eid;
    }
    n = n < k ? n + 1u : k;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int r = 0; r < R; ++r) {
        key[r] = lk[r * 64 + (int)lane];
        id[r] = li[r * 64 + (int)lane];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// np.K != 0: the workgroup also does k_prepare_clear's work for the pass (no
// F rows or hits to clear), one dependent launch less.
template <int R>
__global__ __launch_bounds__(kRefThreads) void k_select_reference(
    const float *__restrict__ unshot, uint32_t npatch, uint32_t k, uint32_t *__restrict__ shooters,
    uint32_t *__restrict__ nshoot, NextPass np, const uint32_t *__restrict__ ctl)
{
    __shared__ float lk[64 * R], ck[kRefThreads];
    __shared__ uint32_t li[64 * R], ci[kRefThreads];
    __shared__ uint32_t wcnt[kRefThreads / 64];
    __shared__ float sback;
    __shared__ uint32_t sn;
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    float key[R]; // the list, in the first wavefront
    uint32_t id[R], n = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        key[r] = 0.0f;
        id[r] = 0u;
    }
    if (threadIdx.x < 64 * R) {
        lk[threadIdx.x] = 0.0f;
        li[threadIdx.x] = 0u;
    }
    if (threadIdx.x == 0) {
        sback = 0.0f;
        sn = 0u;
    }
    auto energy = [&](uint32_t j) {
        if (j >= npatch)
            return 0.0f;
        const float u0 = unshot[3 * (size_t)j], u1 = unshot[3 * (size_t)j + 1],
                    u2 = unshot[3 * (size_t)j + 2];
        return u0 * u0 + u1 * u1 + u2 * u2;
    };
    float e = energy(threadIdx.x);
    __syncthreads();
    for (uint32_t base = 0; base < npatch; base += kRefThreads) {
        const uint32_t j = base + threadIdx.x;
        const bool c = j < npatch && ((sn == 0 && j == base) || (e > 0 && sback <= e));
        // the candidates in index order
        const uint64_t m = __ballot(c);
        if (lane == 0)
            wcnt[w] = (uint32_t)__popcll(m);
        __syncthreads();
        uint32_t off = 0, total = 0;
        for (uint32_t q = 0; q < kRefThreads / 64; ++q) {
            off += q < w ? wcnt[q] : 0u;
            total += wcnt[q];
        }
        if (c) {
            const uint32_t o = off + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            ci[o] = j;
            ck[o] = e;
        }
        e = energy(base + kRefThreads + threadIdx.x); // the next chunk's
        __syncthreads();
        if (w == 0 && total) {
            // 64 candidates at a time, one per lane: the next one the list
            // takes is the first lane left whose key reaches its back
            float back = sback;
            for (uint32_t q0 = 0; q0 < total; q0 += 64u) {
                const bool in = q0 + lane < total;
                const float ek = in ? ck[q0 + lane] : 0.0f;
                const uint32_t ei = in ? ci[q0 + lane] : 0u;
                uint64_t left = __ballot(in);
                while (true) {
                    const uint64_t m = left & __ballot(n == 0 || (ek > 0 && back <= ek));
                    if (!m)
                        break;
                    const int l = __ffsll((long long)m) - 1;
                    left = m & (m - 1u);
                    reference_insert<R>(
                        key, id, n, k,
                        __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ek), l)),
                        (uint32_t)__builtin_amdgcn_readlane((int)ei, l), lk, li);
                    back = lk[n - 1u];
                }
            }
            if (lane == 0) {
                sback = back;
                sn = n;
            }
        }
        __syncthreads();
    }
    for (uint32_t i = threadIdx.x; i < k; i += kRefThreads)
        shooters[i] = i < sn ? li[i] : 0u;
    if (np.K) {
        __syncthreads(); // every thread has read sn
        if (threadIdx.x == 0 && ctl[kCtlStop])
            sn = 0u; // the stop gate of k_prepare_clear
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < np.K * 5; i += kRefThreads)
            prepare_item(i, np.K, li, &sn, np.frames, unshot, np.snap, np.mvp, nullptr);
        clear_range(threadIdx.x, kRefThreads, np.bin_count, np.nbins, nullptr, nullptr, 0,
                    np.counters);
    }
    if (threadIdx.x == 0)
        *nshoot = sn;
}

void launch_select_reference(const float *unshot, uint32_t npatch, uint32_t k, uint32_t *shooters,
                             uint32_t *nshoot, const NextPass *np, const uint32_t *ctl,
                             hipStream_t st)
{
    static_assert(RAD_MAX_K <= 256, "four list entries per lane");
    const NextPass p = np ? *np : NextPass{};
    if (k <= 64)
        k_select_reference<1><<<1, kRefThreads, 0, st>>>(unshot, npatch, k, shooters, nshoot, p,
                                                         ctl);
    else
        k_select_reference<4><<<1, kRefThreads, 0, st>>>(unshot, npatch, k, shooters, nshoot, p,
                                                         ctl);
}

} // namespace rad
