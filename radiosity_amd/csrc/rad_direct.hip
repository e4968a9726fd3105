// rad_direct.hip - the direct rasterizer: one launch from a pass's shooters
// to its F rows (or item buffers), without bins.
//
// One workgroup per (shooter, screen tile of one face).  It tests the
// bounds of the scene's triangle runs (clusters of 64, then groups of 16)
// against the tile's frustum, then the bounding spheres of the triangles
// left; those that pass go through the exact pipeline of rad_raster.h
// (transform, near-plane and guard-band clip, snap) and are drawn into the
// tile's depth keys in LDS at once.  No record, count or list goes through
// memory.
//
// It serves the passes that leave most of the chip idle, where the binned
// rasterizer (rad_kernels.hip) is a chain of five latency-bound launches
// (34 us for one shooter of the 1,534-triangle Cornell box at hemicube 128;
// this one 17).  A triangle is set up once per tile it touches and a
// workgroup holds a whole CU, so beyond two rounds of workgroups over the
// CUs, or 8,192 to 49,152 triangles by the number of workgroups, the bins win
// (direct_wins).
#include "rad_internal.h"
#include "rad_raster.h"

namespace rad {

// ------------------------------------------------------------------ clusters
// Bounds of runs of consecutive triangles, once per scene, for whole-run
// culls: groups of 16 triangles (entry 5 i + 1 + j for group j of cluster i)
// and clusters of 64 (entry 5 i).  Meshes list their faces part by part, so
// consecutive triangles are mostly neighbours on one plane and an
// axis-aligned box holds them tightly (a bounding sphere let three times as
// many (tile, cluster) pairs through in the box rooms).  Three 16-byte words:
//  0  box centre, half extent x
//  1  half extents y and z, half the thickness of the vertices along N (-1
//     when the triangles do not share N within 0.5 %), and the smallest
//     area / longest edge of a triangle
//  2  unit normal N on the side the triangles are drawn from, and the
//     smallest area of a triangle (0 when their normals are not within kTilt
//     of N)
// In a pack the clusters of scene s start at tbeg / 64 + s, which leaves
// room for a partly filled last cluster in every scene.
constexpr uint32_t kCluWords = 15; // 16-byte words per cluster
// Sine of the largest angle between N and the normals of a run taken for flat:
// well above the rounding of a plane's vertices (about 1e-7 of their
// coordinates over a triangle's height), and too small to cost the back-face
// test of a run anything (it asks for more than a milliradian).
constexpr float kTilt = 2.5e-4f;

template <int N, typename Op> __device__ static inline float lanes_red(float x, Op op)
{
    for (int o = 1; o < N; o <<= 1)
        x = op(x, __shfl_xor(x, o, 64));
    return x;
}

// The bounds over each run of N lanes' triangles, written by its first lane.
template <int N>
__device__ static inline void run_bounds(const float (&v)[3][3], const float (&n)[3], float q,
                                         float area, float4 *__restrict__ out, bool write)
{
    auto mn = [](float x, float y) { return fminf(x, y); };
    auto mx = [](float x, float y) { return fmaxf(x, y); };
    float ctr[3], half[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float lo = lanes_red<N>(fminf(v[0][c], fminf(v[1][c], v[2][c])), mn);
        const float hi = lanes_red<N>(fmaxf(v[0][c], fmaxf(v[1][c], v[2][c])), mx);
        ctr[c] = 0.5f * (lo + hi);
        half[c] = fmaxf(hi - ctr[c], ctr[c] - lo) * 1.00001f;
    }
    float nn[3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
        nn[c] = __shfl(n[c], (int)((threadIdx.x & 63u) & ~(uint32_t)(N - 1)), 64);
    const float same = lanes_red<N>(n[0] * nn[0] + n[1] * nn[1] + n[2] * nn[2], mn);
    const float kx = n[1] * nn[2] - n[2] * nn[1], ky = n[2] * nn[0] - n[0] * nn[2],
                kz = n[0] * nn[1] - n[1] * nn[0];
    const float tilt = lanes_red<N>(kx * kx + ky * ky + kz * kz, mx);
    float eps = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        eps = fmaxf(eps, fabsf((v[k][0] - ctr[0]) * nn[0] + (v[k][1] - ctr[1]) * nn[1] +
                               (v[k][2] - ctr[2]) * nn[2]));
    eps = lanes_red<N>(eps, mx) + 4e-7f * (half[0] + half[1] + half[2]);
    q = lanes_red<N>(q, mn);
    area = lanes_red<N>(area, mn);
    if (write) {
        out[0] = make_float4(ctr[0], ctr[1], ctr[2], half[0]);
        out[1] = make_float4(half[1], half[2], same >= 0.995f ? eps : -1.0f, q);
        out[2] = make_float4(nn[0], nn[1], nn[2], tilt <= kTilt * kTilt ? area : 0.0f);
    }
}

__global__ __launch_bounds__(256) void k_clusters(const float *__restrict__ tri, uint32_t ntri,
                                                  const uint32_t *__restrict__ sc_tbeg,
                                                  uint32_t nscene, uint32_t nclu,
                                                  float4 *__restrict__ clu)
{
    const uint32_t g = blockIdx.x * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (g >= nclu)
        return;
    uint32_t tb = 0, te = ntri, cb = 0;
    if (sc_tbeg) {
        // the last scene whose first cluster is at or before g
        uint32_t lo = 0, hi = nscene;
        while (lo + 1 < hi) {
            const uint32_t mid = (lo + hi) / 2;
            if (sc_tbeg[mid] / 64u + mid <= g)
                lo = mid;
            else
                hi = mid;
        }
        tb = sc_tbeg[lo];
        te = sc_tbeg[lo + 1];
        cb = tb / 64u + lo;
    }
    const uint32_t t0 = tb + (g - cb) * 64u;
    if (t0 >= te)
        return; // the spare cluster of a scene
    // lanes past the scene's last triangle repeat it
    const uint32_t t = min(t0 + lane, te - 1u);
    float v[3][3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            v[k][c] = tri[(size_t)(3 * k + c) * ntri + t];
    // the drawn side: the camera mirrors (right = up x dir), so a triangle is
    // counter-clockwise seen from the side of (v2 - v0) x (v1 - v0)
    float e1[3], e2[3], e3[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        e1[c] = v[1][c] - v[0][c];
        e2[c] = v[2][c] - v[0][c];
        e3[c] = v[2][c] - v[1][c];
    }
    float n[3] = {e2[1] * e1[2] - e2[2] * e1[1], e2[2] * e1[0] - e2[0] * e1[2],
                  e2[0] * e1[1] - e2[1] * e1[0]};
    const float len = sqrtf(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    auto sq = [](const float *e) { return e[0] * e[0] + e[1] * e[1] + e[2] * e[2]; };
    const float edge = sqrtf(fmaxf(sq(e1), fmaxf(sq(e2), sq(e3))));
    const float inv = len > 0.0f ? 1.0f / len : 0.0f;
#pragma unroll
    for (int c = 0; c < 3; ++c)
        n[c] *= inv;
    const float q = edge > 0.0f ? 0.5f * len / edge : 0.0f;
    float4 *const out = clu + kCluWords * (size_t)g;
    run_bounds<64>(v, n, q, 0.5f * len, out, lane == 0);
    run_bounds<16>(v, n, q, 0.5f * len, out + 3u * (1u + lane / 16u), (lane & 15u) == 0);
}

size_t cluster_words(uint32_t ntri, uint32_t nscene)
{
    return (size_t)kCluWords * ((ntri + 63u) / 64u + nscene);
}

void launch_clusters(const float *tri, uint32_t ntri, const uint32_t *sc_tbeg, uint32_t nscene,
                     float4 *clu, hipStream_t st)
{
    const uint32_t n = (ntri + 63u) / 64u + nscene;
    if (ntri)
        k_clusters<<<(n + 3) / 4, 256, 0, st>>>(tri, ntri, sc_tbeg, nscene, n, clu);
}

// --------------------------------------------------------------------- culls
// The tile's frustum: inward normals of its four planes through the eye (one
// pixel of margin), the shooter's normal and the depth axis, with their
// lengths, and the screen axes.
struct TileView {
    float p[6][3], len[6];
    float x[3], y[3], e[3];
    float em; // rounding of the MVP's translation: 2e-6 |eye|_1
    float mvp[16];
    uint32_t cull;
    float4 scis; // the bounds x / w, y / w of the tile with the margin
};

// Whether a box (centre offset d from the eye, half extents h) may touch the
// tile: not wholly below the shooter's plane, nor nearer than the near
// plane, nor outside one of the four planes.  m bounds the float error of
// the tests and of the exact pipeline's clip coordinates.
__device__ static inline bool box_in_tile(const TileView &v, float dx, float dy, float dz,
                                          float hx, float hy, float hz, float m)
{
    bool in = true;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const float c = fmaf(dz, v.p[k][2], fmaf(dy, v.p[k][1], dx * v.p[k][0]));
        const float h = fmaf(hz, fabsf(v.p[k][2]),
                             fmaf(hy, fabsf(v.p[k][1]), hx * fabsf(v.p[k][0])));
        in = in && !(c + h + m < (k == 5 ? 0.0099f : 0.0f));
    }
    return in;
}

// The same for a sphere.
__device__ static inline bool sphere_in_tile(const TileView &v, float4 sp)
{
    const float dx = sp.x - v.e[0], dy = sp.y - v.e[1], dz = sp.z - v.e[2];
    const float m = 3e-4f * (fabsf(dx) + fabsf(dy) + fabsf(dz) + sp.w) + 3e-6f + 4.0f * v.em;
    bool in = true;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const float c = fmaf(dz, v.p[k][2], fmaf(dy, v.p[k][1], dx * v.p[k][0]));
        in = in && !(c + fmaf(sp.w, v.len[k], m) < (k == 5 ? 0.0099f : 0.0f));
    }
    return in;
}

// The tile's view through an offset of zero that the compiler cannot see: a
// loop body that reads it this way loads it from LDS every time round, where
// hoisted out it would hold 50 registers through the drawing.
__device__ static inline const TileView &reload(const TileView &v)
{
    uint32_t z = 0;
    asm volatile("" : "+v"(z));
    return (&v)[z];
}

// v_sqrt_f32 (1 ulp) rounded up: an upper bound for the culls.
__device__ static inline float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x) * 1.000001f; }

// A run of triangles (its three bounds words) against the tile: the box
// test, then, for a run that shares one normal N (thickness eps, radius
// rho of the box):
//  - its vertices rise above the shooter's plane by at most
//    pa + |n.N| eps + |n x N| rho.  When that is under 2e-6 of their
//    distance (or under the near plane's 0.01), they project to within
//    1e-5 W / 2 << 0.5 pixel of the horizon, where the nearest kept pixel
//    centre is half a pixel away (in the front face: nearer than the near
//    plane).  This drops the shooter's own wall.
//  - the eye lies at least D > 0 behind the plane of every triangle of a flat
//    run (behind the run's plane, less what normals kTilt off N make of the
//    distance to a vertex): a triangle of area A with depths in [wmin, wmax]
//    projects to a clockwise area of at least (W/2)^2 2 A D / wmax^3 square
//    pixels.  Snapping and rounding move a vertex by at most delta pixels per
//    axis, which changes the area by at most 5.7 delta L + 8 delta^2 for a
//    longest projected edge L <= sqrt2 (W/2) edge (1 + kappa) / wmin, kappa
//    the largest |x / w|; the two tests ask twice that, so the snapped triangle
//    is clockwise too.
__device__ static inline bool run_in_tile(const TileView &v, const float4 *__restrict__ b,
                                          float halfW)
{
    float4 b0 = b[0], b1 = b[1], b2 = b[2];
    // all three loads before the first test, not the last one behind it
    asm volatile("" : "+v"(b0.x), "+v"(b1.x), "+v"(b2.x));
    const float dx = b0.x - v.e[0], dy = b0.y - v.e[1], dz = b0.z - v.e[2];
    const float hs = b0.w + b1.x + b1.y, l1 = fabsf(dx) + fabsf(dy) + fabsf(dz);
    const float m = 3e-4f * (l1 + hs) + 3e-6f + 4.0f * v.em;
    if (!box_in_tile(v, dx, dy, dz, b0.w, b1.x, b1.y, m))
        return false;
    const float eps = b1.z;
    if (eps < 0.0f)
        return true;
    const float rho = fsqrt(b0.w * b0.w + b1.x * b1.x + b1.y * b1.y);
    const float dl = fsqrt(dx * dx + dy * dy + dz * dz), dmin = dl - rho;
    const float *const n = v.p[4], *const w = v.p[5];
    const float pa = dx * n[0] + dy * n[1] + dz * n[2];
    const float cn = fabsf(n[0] * b2.x + n[1] * b2.y + n[2] * b2.z);
    const float kx = n[1] * b2.z - n[2] * b2.y, ky = n[2] * b2.x - n[0] * b2.z,
                kz = n[0] * b2.y - n[1] * b2.x;
    const float hmax = pa + cn * eps + fsqrt(kx * kx + ky * ky + kz * kz) * rho;
    if (rho < 4.0f * dmin && hmax < fminf(2e-6f * dmin, 0.0098f))
        return false;
    const float D = dx * b2.x + dy * b2.y + dz * b2.z - eps - 1e-6f * l1 - kTilt * (dl + rho);
    const float Z = dx * w[0] + dy * w[1] + dz * w[2];
    const float hw = b0.w * fabsf(w[0]) + b1.x * fabsf(w[1]) + b1.y * fabsf(w[2]);
    const float wmin = Z - hw - m, wmax = Z + hw + m;
    if (!(D > 1e-5f * dl) || !(wmin > 0.02f))
        return true;
    // the two tests multiplied out: S = kappa wmin, dw = delta wmin
    const float X = dx * v.x[0] + dy * v.x[1] + dz * v.x[2];
    const float Y = dx * v.y[0] + dy * v.y[1] + dz * v.y[2];
    const float S = fmaxf(fabsf(X), fabsf(Y)) + rho, w2 = wmin * wmin, w3 = wmax * wmax * wmax;
    const float dw = (0.0025f + 1.6e-5f * halfW) * wmin + halfW * (v.em + 1e-6f * l1);
    return !(S <= 8.0f * wmin && halfW * b1.w * D * w2 * wmin > 16.0f * dw * (wmin + S) * w3 &&
             halfW * halfW * b2.w * D * w2 > 16.0f * dw * dw * w3);
}

// -------------------------------------------------------------------- kernel
// Tiles of a hemicube for tile side T: the side faces' tiles first, the row
// next to the horizon before the others (those see the most triangles, so
// they start first), then the front face's.
__host__ __device__ static inline uint32_t direct_tiles(uint32_t W, uint32_t T)
{
    const uint32_t nf = (W + T - 1) / T, ns = (W / 2 + T - 1) / T;
    return 4u * ns * nf + nf * nf;
}

constexpr uint32_t kDirThreads = 1024;
constexpr uint32_t kDirMax = 768;     // clusters of the largest scene (direct_wins)
constexpr uint32_t kDirTri = 2048;    // triangles it queues before drawing
constexpr uint32_t kDirClip = 128;    // clip jobs a wavefront queues
constexpr uint32_t kDirTwoLevel = 48; // clusters from which they are tested before their groups

// A record's pixels of the tile by the whole wavefront, the record and its
// bbox wave-uniform.
__device__ static inline void draw_big(const RasterRec &r, int32_t x0, int32_t y0, int32_t x1,
                                       int32_t y1, int32_t ox, int32_t oy, uint32_t tshift,
                                       uint64_t *tk)
{
    if (span_within(r, kWave32Span)) {
        draw_wave32(r, 0, 0, x0, x1, y0, y1, ox, oy, tshift, tk);
    } else {
        Edges e;
        make_edges(r.x, r.y, e);
        draw_wave(r, e, 0, 0, x0, x1, y0, y1, ox, oy, tshift, tk);
    }
}

template <bool FQ>
__global__ __launch_bounds__(kDirThreads) void k_direct(DirectArgs a)
{
    constexpr uint32_t NT = kDirThreads, NW = NT / 64;
    extern __shared__ uint64_t tk[]; // T x T depth keys
    // indices within the scene: a cluster, a group (4 per cluster), a triangle
    // (64 per cluster)
    __shared__ uint16_t clist[kDirMax], glist[4 * kDirMax], tq[kDirTri];
    __shared__ uint16_t clipq[NW][kDirClip];
    __shared__ CV4 lp[NW][kClipMax];
    static_assert(64 * kDirMax <= 65536, "16-bit triangle indices");
    __shared__ uint32_t nc_, ng_, nt_;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t rank = blockIdx.x / a.nslot, s = blockIdx.x - rank * a.nslot;
    const uint32_t nshoot = *a.nshoot;
    // a slot of a pack may render at its scene's own resolution
    const uint32_t W = a.slot_w ? a.slot_w[s] : a.W, TW = 2 * W, T = 1u << a.tshift;
    if (a.slot_w && rank >= direct_tiles(W, T))
        return;
    const uint32_t tb = a.slot_tbeg ? a.slot_tbeg[s] : 0u;
    const uint32_t te = a.slot_tbeg ? tb + a.slot_tcnt[s] : a.ntri;
    const float4 *clu = a.clu + kCluWords * (size_t)(a.slot_cbeg ? a.slot_cbeg[s] : 0u);
    const uint32_t nclu = (te - tb + 63u) / 64u;
    const float *dff = a.dff + (a.slot_dffo ? a.slot_dffo[s] : 0u);
    // the tile: face, face-local origin (ox, oy) and the pixels [x0, x1) x
    // [y0, y1) of it that the face keeps
    const int32_t Ti = (int32_t)T, h2 = (int32_t)W / 2;
    const uint32_t nf = (W + T - 1) / T, ns = (W / 2 + T - 1) / T;
    int32_t ox, oy;
    int face;
    if (rank < 4u * ns * nf) {
        const uint32_t j = rank / (4u * nf), rem = rank - j * 4u * nf;
        face = (int)(rem / nf);
        const int32_t l = (int32_t)(rem % nf) * Ti;
        // the horizon is the middle row (column) of the face
        const int32_t d = face == 0 || face == 3 ? h2 - (int32_t)(j + 1) * Ti : h2 + (int32_t)j * Ti;
        ox = face < 2 ? l : d;
        oy = face < 2 ? d : l;
    } else {
        const uint32_t r = rank - 4u * ns * nf;
        face = 4;
        ox = (int32_t)(r % nf) * Ti;
        oy = (int32_t)(r / nf) * Ti;
    }
    const FaceView fv = face_view((int32_t)W, face);
    const int32_t x0 = max(ox, fv.sx0), x1 = min(ox + Ti, fv.sx1);
    const int32_t y0 = max(oy, fv.sy0), y1 = min(oy + Ti, fv.sy1);
    // the face's MVP and the culling frame, one element per lane, in flight
    // together with the shooter count
    const float *sm = a.mvp + (size_t)s * kShooterStride;
    float sv = 0.0f;
    if (wv == 0 && lane < 29)
        sv = sm[lane < 16 ? (uint32_t)face * 16u + lane : 64u + lane];
    if (s >= nshoot)
        return;
    const float halfW = 0.5f * (float)W;
    // the tile's frustum, in LDS: as wave-uniform registers it would crowd
    // out the drawing's
    __shared__ TileView v;
    if (wv == 0) {
        auto at = [&](int l) {
            return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sv), l));
        };
        const float ih = __builtin_amdgcn_rcpf(halfW); // the bounds carry a pixel of margin
        const float lox = (float)(x0 - 1) * ih - 1.0f, hix = (float)(x1 + 1) * ih - 1.0f;
        const float loy = (float)(y0 - 1) * ih - 1.0f, hiy = (float)(y1 + 1) * ih - 1.0f;
        if (lane < 16)
            v.mvp[lane] = sv;
        if (lane == 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float x = at(4 * c + 0), y = at(4 * c + 1), w = at(4 * c + 3);
                v.p[0][c] = x - lox * w;
                v.p[1][c] = hix * w - x;
                v.p[2][c] = y - loy * w;
                v.p[3][c] = hiy * w - y;
                v.p[4][c] = at(19 + c);
                v.p[5][c] = w;
                v.x[c] = x;
                v.y[c] = y;
                v.e[c] = at(16 + c);
            }
            v.len[0] = fsqrt(1.0f + lox * lox);
            v.len[1] = fsqrt(1.0f + hix * hix);
            v.len[2] = fsqrt(1.0f + loy * loy);
            v.len[3] = fsqrt(1.0f + hiy * hiy);
            v.len[4] = v.len[5] = 1.0f;
            v.em = 2e-6f * (fabsf(at(16)) + fabsf(at(17)) + fabsf(at(18)));
            v.scis = make_float4(lox, hix, loy, hiy);
            // else the frame's axes are not orthogonal
            v.cull = at(28) == 0.0f;
            nc_ = 0u;
            ng_ = 0u;
            nt_ = 0u;
        }
    }
    for (uint32_t p = threadIdx.x; p < T * T; p += NT)
        tk[p] = kClearKey;
    // appends to a list in LDS: the lanes with `take`, in lane order
    auto append = [&](bool take, uint32_t val, uint16_t *list, uint32_t *count) {
        const uint64_t m = __ballot(take);
        uint32_t base = 0;
        if (m && lane == 0)
            base = atomicAdd(count, (uint32_t)__popcll(m));
        base = __builtin_amdgcn_readfirstlane(base);
        if (take)
            list[base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)val;
    };
    __syncthreads();
    const bool cull = v.cull != 0u;
    const uint32_t ntc = te - tb;
    const bool two = cull && nclu > kDirTwoLevel;
    // the clusters, then the groups of 16, that may touch the tile
    if (two) {
        for (uint32_t c = threadIdx.x; (c & ~63u) < nclu; c += NT)
            append(c < nclu && run_in_tile(reload(v), clu + kCluWords * c, halfW), c, clist, &nc_);
        __syncthreads();
    }
    const uint32_t nq = 4u * (two ? nc_ : nclu);
    for (uint32_t i = threadIdx.x; (i & ~63u) < nq; i += NT) {
        bool vis = i < nq;
        uint32_t g = i;
        if (vis) {
            if (two)
                g = 4u * clist[i >> 2] + (i & 3u);
            vis = g * 16u < ntc;
            if (vis && cull)
                vis = run_in_tile(reload(v), clu + kCluWords * (g >> 2) + 3u * (1u + (g & 3u)), halfW);
        }
        append(vis, g, glist, &ng_);
    }
    __syncthreads();
    const uint32_t ng = ng_;
    for (uint32_t g0 = 0; g0 < ng; g0 += kDirTri / 16u) {
        const uint32_t g1 = min(ng, g0 + kDirTri / 16u);
        // the triangles whose spheres may touch the tile, so that the
        // exact pipeline runs with full wavefronts (and clips none that
        // merely reaches behind the eye)
        if (cull) {
            if (g0) {
                if (threadIdx.x == 0)
                    nt_ = 0u;
                __syncthreads();
            }
            for (uint32_t i = 16u * g0 + threadIdx.x; (i & ~63u) < 16u * g1; i += NT) {
                bool vis = i < 16u * g1;
                uint32_t t = 0;
                if (vis) {
                    t = 16u * glist[i >> 4] + (i & 15u);
                    vis = t < ntc && sphere_in_tile(reload(v), a.tsph[tb + t]);
                }
                append(vis, t, tq, &nt_);
            }
            __syncthreads();
        }
        // The exact pipeline and the drawing, every wavefront on its own:
        // up to 64 triangles per step, fewer (a power of two) when there
        // are not enough for every wavefront; then lanes share one, each
        // doing its pipeline and drawing every nph-th of its rows (1
        // shooter over 20,000 triangles at hemicube 256: 28.7 us with a
        // lane per triangle, 27.2).
        // Triangles to clip are queued by their wavefront and taken one
        // per step.
        const uint32_t nt = cull ? nt_ : 16u * (g1 - g0);
        uint32_t lb = 0; // log2 of the triangles per step
        while (lb < 6u && (NW << lb) < nt)
            ++lb;
        const uint32_t bs = 1u << lb;
        uint32_t qi = wv * bs, cn = 0;
        uint16_t *const cq = clipq[wv];
        while (true) {
            const bool batch = qi < nt && cn <= kDirClip - 64u;
            if (!batch && cn == 0)
                break;
            wave_lds_sync();
            const TileView &vw = reload(v);
            SV A, B, C;
            uint32_t id = 0;
            bool have = false;
            // row phase of the lane's triangle, log2 of the phases
            uint32_t ph = 0, lph = 0;
            if (batch) {
                bool clip = false;
                uint32_t tr = ntc;
                const uint32_t i = qi + (lane & (bs - 1u));
                ph = lane >> lb;
                lph = 6u - lb;
                if (i < nt) {
                    tr = cull ? tq[i] : 16u * glist[g0 + (i >> 4)] + (i & 15u);
                }
                if (tr < ntc) {
                    const uint32_t t = tb + tr;
                    float vx[3][3];
#pragma unroll
                    for (int k = 0; k < 3; ++k)
#pragma unroll
                        for (int c = 0; c < 3; ++c)
                            vx[k][c] = a.tri[(size_t)(3 * k + c) * a.ntri + t];
                    id = a.tri_patch[t] + 1u;
                    CV4 poly[3];
                    transform3(vw.mvp, vx, poly);
                    const TriClass cl = classify_tri(poly, vw.scis);
                    clip = cl == kTriClip && ph == 0u;
                    have = cl == kTriIn;
                    if (have) {
                        A = project(poly[0], halfW);
                        B = project(poly[1], halfW);
                        C = project(poly[2], halfW);
                    }
                }
                qi += NW * bs;
                const uint64_t m = __ballot(clip);
                if (clip)
                    cq[cn + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)tr;
                cn += (uint32_t)__popcll(m);
            } else {
                const uint32_t t = tb + cq[--cn];
                CV4 p;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    p.c[r] = 0.0f;
                if (lane < 3) {
                    const float tx = a.tri[(size_t)(3 * lane + 0) * a.ntri + t];
                    const float ty = a.tri[(size_t)(3 * lane + 1) * a.ntri + t];
                    const float tz = a.tri[(size_t)(3 * lane + 2) * a.ntri + t];
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        p.c[r] = vw.mvp[0 * 4 + r] * tx + vw.mvp[1 * 4 + r] * ty +
                                 vw.mvp[2 * 4 + r] * tz + vw.mvp[3 * 4 + r];
                }
                id = a.tri_patch[t] + 1u;
                const int n = clip_polygon_wave(p, lp[wv], &a.counters[kCntOverflow]);
                if (n >= 3)
                    have = clip_fan(p, n, halfW, A, B, C);
            }
            RasterRec r;
            int32_t bx0 = 0, by0 = 0, bx1 = -1, by1 = -1;
            if (have) {
                int64_t area2;
                have = snapped_bbox(A, B, C, x0, y0, x1, y1, area2, bx0, by0, bx1, by1);
                if (have)
                    make_record(A, B, C, area2, id, r);
            }
            // Small ones by their lanes, which takes as long as the
            // largest; the others by the whole wavefront, one after the
            // other.
            const uint32_t nph = 1u << lph;
            const uint32_t rows = ((uint32_t)(by1 - by0 + 1) + nph - 1u) >> lph;
            const bool small = have && (uint32_t)(bx1 - bx0 + 1) * rows <= a.small_px &&
                               span_within(r, kLane32Span);
            if (small)
                draw_lane32(r, 0, 0, bx0, bx1, by0, by1, ox, oy, a.tshift, tk, ph, nph);
            for (uint64_t m = __ballot(have && !small && ph == 0u); m; m &= m - 1) {
                const int l = __ffsll((long long)m) - 1;
                RasterRec u;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    u.x[k] = __builtin_amdgcn_readlane(r.x[k], l);
                    u.y[k] = __builtin_amdgcn_readlane(r.y[k], l);
                }
                u.dzdx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.dzdx), l));
                u.dzdy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.dzdy), l));
                u.z0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.z0), l));
                u.id = (uint32_t)__builtin_amdgcn_readlane((int)r.id, l);
                draw_big(u, __builtin_amdgcn_readlane(bx0, l), __builtin_amdgcn_readlane(by0, l),
                         __builtin_amdgcn_readlane(bx1, l), __builtin_amdgcn_readlane(by1, l),
                         ox, oy, a.tshift, tk);
            }
        }
        __syncthreads(); // the queues are the next groups'
    }

    __syncthreads(); // the keys are complete
    // Resolve: the tile's ids and depths out, or its runs into the F row.
    // Four consecutive texels of a tile row per lane (T >= 8).
    const uint32_t TT = T * T;
    if (a.out_ids) {
        for (uint32_t p = threadIdx.x; p < TT; p += NT) {
            const int32_t px = ox + (int32_t)(p & (T - 1)), py = oy + (int32_t)(p >> a.tshift);
            if (px >= x0 && px < x1 && py >= y0 && py < y1) {
                const uint64_t key = tk[p];
                const size_t o = (size_t)s * a.RES + (uint32_t)(fv.vpy + py) * TW +
                                 (uint32_t)(fv.vpx + px);
                a.out_ids[o] = (uint32_t)key;
                if (a.out_depth)
                    a.out_depth[o] = __uint_as_float((uint32_t)(key >> 32));
            }
        }
        return;
    }
    const uint32_t pbase = a.slot_pbeg ? a.slot_pbeg[s] : 0u;
    float *const frow = a.ff ? a.ff + (size_t)s * a.rowlen : nullptr;
    unsigned long long *const qrow = a.ffq ? a.ffq + (size_t)s * a.rowlen : nullptr;
    uint32_t *const hrow = a.hits ? a.hits + (size_t)s * a.rowlen : nullptr;
    uint32_t *const fflag = a.fblk ? a.fblk + s : nullptr;
    const bool with_c = hrow != nullptr;
    const uint32_t rp = threadIdx.x * 4u;
    uint32_t q4[4] = {0u, 0u, 0u, 0u};
    float f4[4] = {0.f, 0.f, 0.f, 0.f};
    static_assert(kMaxTile * kMaxTile <= 4 * 256, "one resolve step per tile");
    if (rp < TT) {
        const int32_t px = ox + (int32_t)(rp & (T - 1)), py = oy + (int32_t)(rp >> a.tshift);
        if (py >= y0 && py < y1) {
            const float *d = dff + (int32_t)((fv.vpy + py) * (int32_t)TW + fv.vpx + px);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (px + j >= x0 && px + j < x1) {
                    q4[j] = (uint32_t)tk[rp + (uint32_t)j];
                    f4[j] = q4[j] ? d[j] : 0.0f;
                }
        }
    }
    if ((threadIdx.x & ~63u) * 4u < TT) { // whole wavefronts
        reduce_quad(q4, f4, with_c, [&](uint32_t id, float f, uint32_t c) {
            if (!id)
                return;
            const uint32_t p = id - 1 - pbase;
            if (p >= a.rowlen) {
                atomicAdd(&a.counters[kCntUnknown], 1u);
                return;
            }
            // straight to the row: merging a tile's runs in LDS first, as the
            // binned tiles do, took as long at these sizes as it saved
            if constexpr (FQ)
                atomicAdd(&qrow[p], fixed52(f));
            else
                atomicAdd(&frow[p], f);
            if (with_c)
                atomicAdd(&hrow[p], c);
            if (fflag)
                fflag[(p >> 6) * a.fstride] = 1u;
        });
    }
}

// Whether k slots of hemicube side W over scenes of at most ntri triangles
// are drawn directly, and the tile side.  A workgroup has a CU to itself: tiles
// of 16 while those fit at once, else of 32.  It looks at every cluster of the
// scene and draws its tile's share alone, so it wins for few triangles a
// tile.  Direct against binned, us per pass (8 in a graph, box rooms): tiles of
// 16, hemicube 32 (12 tiles), 8 slots, 8,000 triangles 40.3 / 46.7, 14,000 49.7 /
// 47.6; 64 (48 tiles), 4 slots, 20,000 43.9 / 46.7, 40,000 57.4 / 52.3; 128 (192
// tiles), 1 slot, 40,000 36.7 / 38.2.  Tiles of 32, hemicube 64 (12 tiles), 16
// slots, 8,000 51.2 / 55.9, 20,000 68.5 / 59.5; 128 (48 tiles), 4 slots, 20,000
// 49.2 / 51.4, 40,000 61.1 / 53.7; 256 (192 tiles), 1 slot, 28,000 37.6 / 40.5,
// 40,000 45.5 / 43.3.  More than fit at once: 128, 8 slots, 4,000 53.4 / 54.9,
// 14,000 59.3 / 56.1; 256, 2 slots, 8,000 50.0 / 52.6; 64, 32 slots, 4,000 72.2 /
// 64.9.
bool direct_wins(uint32_t k, uint32_t W, uint32_t ntri, uint32_t *T)
{
    const uint32_t wg = k * direct_tiles(W, 32);
    *T = wg <= 64 ? 16u : 32u;
    if (ntri > 64u * kDirMax) // what k_direct's lists hold
        return false;
    if (wg > 256)
        return wg <= 384 && W >= 128 && ntri <= 8192;
    return ntri <= 600u * direct_tiles(W, *T) && (wg <= 64 || ntri <= 34816u);
}

void launch_direct(const DirectArgs &args, uint32_t T, hipStream_t st)
{
    DirectArgs a = args;
    a.tshift = T == 16 ? 4 : 5;
    const uint32_t blocks = direct_tiles(a.W, T) * a.nslot;
    const size_t lds = (size_t)T * T * sizeof(uint64_t);
    if (a.ffq)
        k_direct<true><<<blocks, kDirThreads, lds, st>>>(a);
    else
        k_direct<false><<<blocks, kDirThreads, lds, st>>>(a);
}

} // namespace rad
