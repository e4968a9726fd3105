// rad_prepare.h - what a kernel does that prepares a pass: the shooters' face
// MVPs and snapshots, bins and counters cleared.
#ifndef RAD_PREPARE_H
#define RAD_PREPARE_H

#include "rad_internal.h"

#include <hip/hip_runtime.h>

namespace rad {

// -------------------------------------------------------------------- camera
struct f3 {
    float x, y, z;
};
__device__ static inline f3 sub3(f3 a, f3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ static inline f3 add3(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ static inline f3 neg3(f3 a) { return {-a.x, -a.y, -a.z}; }
// Vector.h:534-537: a.v_Cross(b) is b x a
__device__ static inline f3 vcross(f3 a, f3 b)
{
    return {b.y * a.z - b.z * a.y, b.z * a.x - b.x * a.z, b.x * a.y - b.y * a.x};
}
// Vector.h:389-399
__device__ static inline f3 normalize3(f3 a)
{
    float t = sqrtf(a.x * a.x + a.y * a.y + a.z * a.z);
    if (t != 0) {
        t = 1 / t;
        a.x = a.x * t;
        a.y = a.y * t;
        a.z = a.z * t;
    }
    return a;
}

// Camera::lookFromPatch + GetMatrix + Perspective + P*MV (Camera.cpp:19-52,
// 97-103; Transform.cpp:26-46, 70-80, 127-156; Main.cpp:1171-1183).
__device__ static void face_mvp(const float *fr, int face, float *mvp)
{
    f3 eye = {fr[0], fr[1], fr[2]}, n = {fr[3], fr[4], fr[5]}, pu = {fr[6], fr[7], fr[8]};
    f3 target, up;
    switch (face) {
    case 0: target = pu; up = neg3(n); break;
    case 1: target = neg3(pu); up = n; break;
    case 2: target = neg3(vcross(n, pu)); up = pu; break;
    case 3: target = vcross(n, pu); up = pu; break;
    default: target = n; up = pu; break;
    }
    f3 dir = normalize3(sub3(add3(target, eye), eye));
    f3 right = normalize3(vcross(dir, up));
    f3 up2 = vcross(right, dir);
    float V[4][4];
    float rr[3] = {right.x, right.y, right.z};
    float uu[3] = {up2.x, up2.y, up2.z};
    float dd[3] = {dir.x, dir.y, dir.z};
    for (int i = 0; i < 3; ++i) {
        V[i][0] = rr[i];
        V[i][1] = uu[i];
        V[i][2] = -dd[i];
        V[i][3] = 0;
        V[3][i] = 0;
    }
    V[3][3] = 1;
    float t[4] = {-eye.x, -eye.y, -eye.z, 1.0f};
    float c3[4];
    for (int r = 0; r < 4; ++r)
        c3[r] = V[0][r] * t[0] + V[1][r] * t[1] + V[2][r] * t[2] + V[3][r] * t[3];
    for (int r = 0; r < 4; ++r)
        V[3][r] = c3[r];
    float fn = 0.01f, ff = 1000.0f;
    float fh = 1.0f * fn, fw = fh * 1.0f;
    float l = -fw, rt = fw, b = -fh, tp = fh;
    float P[4][4];
    for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 4; ++j)
            P[i][j] = 0.0f;
    P[0][0] = 2 * fn / (rt - l);
    P[2][0] = (rt + l) / (rt - l);
    P[1][1] = 2 * fn / (tp - b);
    P[2][1] = (tp + b) / (tp - b);
    P[2][2] = -(ff + fn) / (ff - fn);
    P[3][2] = -2 * ff * fn / (ff - fn);
    P[2][3] = -1;
    P[3][3] = 0;
    for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 4; ++j)
            mvp[i * 4 + j] = P[0][j] * V[i][0] + P[1][j] * V[i][1] + P[2][j] * V[i][2] +
                             P[3][j] * V[i][3];
}

// One thread per (slot, face): snapshot dB (Main.cpp:1161) and the MVP.
// Per shooter the mvp buffer holds kShooterStride floats: five column-major
// MVPs, then the culling frame used by k_raster_setup: eye, unit normal n,
// unit up u (made orthogonal to n) and n x u; then a flag (1 when the frame
// is degenerate or its up is not orthogonal to the normal within 2e-5, which
// turns the conservative culls off for that shooter).
__device__ static void prepare_item(uint32_t t, uint32_t K, const uint32_t *__restrict__ shooters,
                                    const uint32_t *__restrict__ nshoot,
                                    const float *__restrict__ frames,
                                    const float *__restrict__ unshot, float *__restrict__ snap,
                                    float *__restrict__ mvp, const uint32_t *__restrict__ ctl)
{
    if (t >= K * 5 || (ctl && ctl[kCtlStop]))
        return;
    uint32_t s = t / 5, face = t % 5;
    if (s >= *nshoot)
        return;
    uint32_t p = shooters[s];
    float fr[9];
    for (int k = 0; k < 9; ++k)
        fr[k] = frames[9 * (size_t)p + k];
    float *out = mvp + (size_t)s * kShooterStride;
    if (face == 0) {
        snap[3 * s + 0] = unshot[3 * (size_t)p + 0];
        snap[3 * s + 1] = unshot[3 * (size_t)p + 1];
        snap[3 * s + 2] = unshot[3 * (size_t)p + 2];
        f3 n = normalize3({fr[3], fr[4], fr[5]});
        f3 u = {fr[6], fr[7], fr[8]};
        float un = u.x * n.x + u.y * n.y + u.z * n.z;
        u = normalize3({u.x - un * n.x, u.y - un * n.y, u.z - un * n.z});
        f3 v = {n.y * u.z - n.z * u.y, n.z * u.x - n.x * u.z, n.x * u.y - n.y * u.x};
        float cf[12] = {fr[0], fr[1], fr[2], n.x, n.y, n.z, u.x, u.y, u.z, v.x, v.y, v.z};
        for (int k = 0; k < 12; ++k)
            out[80 + k] = cf[k];
        // the culls take the five face axes as n, +-u, +-(n x u); face_mvp
        // aims the side faces along the raw up, so they hold only while up
        // is orthogonal to n
        float ln = sqrtf(fr[3] * fr[3] + fr[4] * fr[4] + fr[5] * fr[5]);
        float lu = sqrtf(fr[6] * fr[6] + fr[7] * fr[7] + fr[8] * fr[8]);
        float cosnu = fabsf(fr[3] * fr[6] + fr[4] * fr[7] + fr[5] * fr[8]) / (ln * lu);
        bool ok = ln > 0.0f && lu > 0.0f && cosnu <= 2e-5f && isfinite(fr[0] + fr[1] + fr[2]);
        out[92] = ok ? 0.0f : 1.0f;
    }
    float m[16];
    face_mvp(fr, (int)face, m);
    for (int k = 0; k < 16; ++k)
        out[face * 16 + k] = m[k];
}

// --------------------------------------------------------------------- clear
// Per pass: bin counts and pass counters reset, F rows (ff non-null) and hit
// counts (hits non-null) to zero.  A kernel, not hipMemsetAsync, so a pass
// can be captured in a graph.
// The previous pass's overflow state is folded into the sticky counter,
// which only the host clears, so a multi-pass call reports any lost pass.
__device__ static void clear_range(size_t i, size_t stride, uint32_t *__restrict__ bin_count,
                                   size_t nbins, float *__restrict__ ff,
                                   uint32_t *__restrict__ hits, size_t nff,
                                   uint32_t *__restrict__ counters)
{
    if (i == 0) {
        // every block of pass counters (one per half-pass), the sticky flag
        // in the first
        bool bad = false;
        for (int h = 0; h < kCntBlocks; ++h) {
            const uint32_t *const cnt = counters + h * kCntN;
            const BinFacts *const f = reinterpret_cast<const BinFacts *>(cnt + kCntFacts);
            bad = bad || cnt[kCntOverflow] != 0 || cnt[kCntEntries] > f->pool_cap;
        }
        for (int h = 0; h < kCntBlocks; ++h)
            for (int k = 0; k < kCntN; ++k)
                if (h || k != kCntSticky)
                    counters[h * kCntN + k] = 0;
        if (bad)
            counters[kCntSticky] = 1;
    }
    for (size_t k = i; k < nbins; k += stride)
        bin_count[k] = 0u;
    for (size_t k = i; k < nff; k += stride) {
        if (ff)
            ff[k] = 0.0f;
        if (hits)
            hits[k] = 0u;
    }
}

} // namespace rad

#endif
