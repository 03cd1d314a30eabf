// Per-ray query bodies shared by the single-grid kernels and the persistent multi-grid kernel.
#pragma once
#include "nvq_device.h"
#include "nvq_slots.h"

namespace nvq {

// Batched ray query: Ray::worldToIndexF (math/Ray.h:258-268), isoCrossing, and the normal from
// the trilinear gradient at ray(t), Grid::indexToWorldGradF (Map::applyIJTF,
// math/Math.h:1758-1763), normalised.  v is the value at the hit voxel minus iso.
struct CrossingOut {
    uint8_t* hit;
    int32_t* ijk;
    float *t, *v, *normal;
};

// Writes ray i's outputs; C holds the corners of the cell at ray(t) where a normal is wanted.
__device__ __forceinline__ void storeCrossing(const CrossingOut& o, const GridView& g, uint64_t i, bool found,
                                              const int32_t c[3], float v, float t, const float p[3], const Cell& C)
{
    if (o.hit) o.hit[i] = found ? 1 : 0;
    if (o.ijk) {
        o.ijk[3 * i] = found ? c[0] : 0;
        o.ijk[3 * i + 1] = found ? c[1] : 0;
        o.ijk[3 * i + 2] = found ? c[2] : 0;
    }
    if (o.t) o.t[i] = found ? t : 0.0f;
    if (o.v) o.v[i] = found ? v : 0.0f;
    if (o.normal) {
        float nr[3] = {0.0f, 0.0f, 0.0f};
        if (found) {
            float gi[3], gw[3];
            trilinearGradient(C, p[0] - floorf(p[0]), p[1] - floorf(p[1]), p[2] - floorf(p[2]), gi);
#pragma unroll
            for (int a = 0; a < 3; ++a)
                gw[a] = __builtin_fmaf(gi[0], g.invMatF[a], __builtin_fmaf(gi[1], g.invMatF[3 + a], gi[2] * g.invMatF[6 + a]));
            const float len = sqrtf(gw[0] * gw[0] + gw[1] * gw[1] + gw[2] * gw[2]);
            if (len > 0.0f) {
                const float sc = 1.0f / len;
                nr[0] = sc * gw[0];
                nr[1] = sc * gw[1];
                nr[2] = sc * gw[2];
            }
        }
        o.normal[3 * i] = nr[0];
        o.normal[3 * i + 1] = nr[1];
        o.normal[3 * i + 2] = nr[2];
    }
}

template<uint32_t GT>
__device__ __forceinline__ void zeroCrossingRay(const GridView& g, const float* __restrict__ eye,
                                                const float* __restrict__ dir, uint64_t i, float iso,
                                                const CrossingOut& o)
{
    Accessor<GT> acc(g);
    const float e[3] = {eye[3 * i], eye[3 * i + 1], eye[3 * i + 2]};
    const float d[3] = {dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
    Ray ray = worldToIndexRay(g, e, d);
    int32_t c[3] = {0, 0, 0};
    float v = 0.0f, t = 0.0f, p[3] = {0.0f, 0.0f, 0.0f};
    Cell C{};
    const bool found = isoCrossingCore<GT>(acc, g, ray, iso, c, v, t);
    if (found && o.normal) {
        rayAt(ray, t, p);
        stencil8(acc, ifloor(p[0]), ifloor(p[1]), ifloor(p[2]), C);
    }
    storeCrossing(o, g, i, found, c, v, t, p, C);
}

// The same over a slot map; false, with nothing written, when the map leaves the ray open.
__device__ __forceinline__ bool zeroCrossingSlots(const SlotMap& M, const GridView& g, const float* __restrict__ eye,
                                                  const float* __restrict__ dir, uint64_t i, float iso,
                                                  const CrossingOut& o)
{
    const float e[3] = {eye[3 * i], eye[3 * i + 1], eye[3 * i + 2]};
    const float d[3] = {dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
    Ray ray = worldToIndexRay(g, e, d);
    int32_t c[3] = {0, 0, 0};
    float v = 0.0f, t = 0.0f, p[3] = {0.0f, 0.0f, 0.0f};
    Cell C{};
    bool open = false;
    const bool found = isoCrossingSlots(M, g, ray, iso, c, v, t, open);
    if (open) return false;
    if (found && o.normal) {
        rayAt(ray, t, p);
        if (!slotCorners(M, g, ifloor(p[0]), ifloor(p[1]), ifloor(p[2]), C)) return false;
    }
    storeCrossing(o, g, i, found, c, v, t, p, C);
    return true;
}

// ------------------------------------------------------------------ fog march
// Emission-absorption over the shared step structure (marchSteps): per step
// a = exp(-sigma*rho*dt), L += T*(1-a)*rho, T *= a.
template<uint32_t GT>
__device__ __forceinline__ void fogMarchRay(const GridView& g, const float* __restrict__ eye,
                                            const float* __restrict__ dir, uint64_t i, float dt, float sigma,
                                            float* __restrict__ Lout, float* __restrict__ Tout)
{
    Accessor<GT> acc(g);
    const float e[3] = {eye[3 * i], eye[3 * i + 1], eye[3 * i + 2]};
    const float d[3] = {dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
    float L = 0.0f, T = 1.0f;
    CellWindow<false> W;
    NoSink none;
    marchSteps(acc, g, e, d, dt, [&](float x0, float x1, float x2) {
        const float fx = floorf(x0), fy = floorf(x1), fz = floorf(x2);
        W.moveTo(acc, g, int32_t(fx), int32_t(fy), int32_t(fz), none);
        const float rho = trilerp(W.c, x0 - fx, x1 - fy, x2 - fz);
        const float a = stepAbsorption(sigma, rho, dt);
        L += T * (1.0f - a) * rho;
        T *= a;
    });
    if (Lout) Lout[i] = L;
    if (Tout) Tout[i] = T;
}

// The same march over a slot map (marchSteps step for step: same cells, positions and operations, so
// the same bits).  Steps of a slot are taken kMarchBatch at a time: their positions do not depend
// on the samples, so all their loads are in flight before the first is composited.  Returns false,
// with nothing written, when the ray meets a slot the map does not resolve.
//
// Bound by the L1's line rate and the VALU in turn: per step four 8-byte loads that touch the
// lines of 64 neighbouring cells, and about 60 instructions.  1024^2 rays: 1.34 ms with batches of 2,
// 1.29 ms with 4.
constexpr int kMarchBatch = 4;

template<int B>
__device__ __forceinline__ bool fogMarchSlots(const SlotMap& M, const GridView& g, const float* __restrict__ eye,
                                              const float* __restrict__ dir, uint64_t i, float dt, float sigma,
                                              float* __restrict__ Lout, float* __restrict__ Tout)
{
    const float e[3] = {eye[3 * i], eye[3 * i + 1], eye[3 * i + 2]};
    const float d[3] = {dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
    float L = 0.0f, T = 1.0f;
    Ray R = worldToIndexRay(g, e, d);
    const float Eps = 0.000001f, Delta = 0.01f;
    bool in = rayClip(R, g.bbox) && !(double(R.t1) > 1e20);
    const float t0 = R.t0 + Eps, t1 = R.t1 - Eps;
    in = in && !(t0 > t1);
    if (in) {
        float p[3];
        rayAt(R, t0, p);
        SlotCell c;
        if (!slotCell(M, ifloor(p[0]), ifloor(p[1]), ifloor(p[2]), c)) return false;
        HDDA h;
        h.init(R, t0, t1, c.dim > 8 ? c.dim : 8);
        for (;;) {
            const float ta = h.t0;
            const bool more = h.stepOnce();
            const float tb = fminf(h.t0, t1);
            const bool brick = !(c.entry & kSlotTile);
            if ((brick || (c.entry & kSlotTileOn)) && ta < tb) {
                const uint32_t base = brick ? c.entry * kBrickFloats : 0u;
                float kf = ceilf(ta / dt);
                float t = kf * dt;
                while (t < tb) {
                    float x[B][3];
                    bool ok[B], fast[B];
                    Cell cell[B];
                    ok[0] = true;
#pragma unroll
                    for (int j = 0; j < B; ++j) {
                        if (j) {
                            const float kn = kf + 1.0f;
                            t = kn * dt;
                            ok[j] = ok[j - 1] && kn != kf && t < tb; // kn == kf: beyond 2^24 steps
                            kf = kn;
                        }
                        x[j][0] = __builtin_fmaf(t, R.dir[0], R.eye[0]);
                        x[j][1] = __builtin_fmaf(t, R.dir[1], R.eye[1]);
                        x[j][2] = __builtin_fmaf(t, R.dir[2], R.eye[2]);
                        const uint32_t rx = uint32_t(ifloor(x[j][0]) - c.ox), ry = uint32_t(ifloor(x[j][1]) - c.oy),
                                       rz = uint32_t(ifloor(x[j][2]) - c.oz);
                        fast[j] = brick && (rx | ry | rz) < 8u;
                        brickCell(M, fast[j] ? base + (rx * 9u + ry) * 9u + rz : 0u, cell[j]);
                    }
#pragma unroll
                    for (int j = 0; j < B; ++j) {
                        if (!ok[j]) continue;
                        const float fx = floorf(x[j][0]), fy = floorf(x[j][1]), fz = floorf(x[j][2]);
                        float rho = trilerp(cell[j], x[j][0] - fx, x[j][1] - fy, x[j][2] - fz);
                        // a tile, or a position that rounding put just outside its slot
                        if (!fast[j] && !slotTrilinear(M, x[j][0], x[j][1], x[j][2], rho)) return false;
                        const float a = stepAbsorption(sigma, rho, dt);
                        L += T * (1.0f - a) * rho;
                        T *= a;
                    }
                    const float kn = kf + 1.0f;
                    if (!ok[B - 1] || kn == kf) break;
                    kf = kn;
                    t = kf * dt;
                }
            }
            if (!more) break;
            rayAt(R, h.t0 + Delta, p);
            if (!slotCell(M, ifloor(p[0]), ifloor(p[1]), ifloor(p[2]), c)) return false;
            h.update(R, c.dim > 8 ? c.dim : 8);
        }
    }
    if (Lout) Lout[i] = L;
    if (Tout) Tout[i] = T;
    return true;
}

// The same march by four lanes per ray: every lane of a quad walks the ray, lane q samples the q-th of
// four steps, and all four composite them in order.  For launches too small to fill the chip, where
// the time is that of one ray's chain of steps: a batch costs one sample and four compositings
// instead of four of each.  `live`: the quad has a ray.
__device__ __forceinline__ float quadLane(float x, int j)
{
    const int v = __float_as_int(x);
    switch (j) {
    case 0: return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0x00, 0xf, 0xf, false));
    case 1: return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0x55, 0xf, 0xf, false));
    case 2: return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0xaa, 0xf, 0xf, false));
    default: return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0xff, 0xf, 0xf, false));
    }
}

__device__ __forceinline__ bool fogMarchQuad(const SlotMap& M, const GridView& g, const float* __restrict__ eye,
                                             const float* __restrict__ dir, uint64_t i, float dt, float sigma,
                                             float* __restrict__ Lout, float* __restrict__ Tout)
{
    const uint32_t q = threadIdx.x & 3u;
    const float e[3] = {eye[3 * i], eye[3 * i + 1], eye[3 * i + 2]};
    const float d[3] = {dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
    float L = 0.0f, T = 1.0f;
    Ray R = worldToIndexRay(g, e, d);
    const float Eps = 0.000001f, Delta = 0.01f;
    bool in = rayClip(R, g.bbox) && !(double(R.t1) > 1e20);
    const float t0 = R.t0 + Eps, t1 = R.t1 - Eps;
    in = in && !(t0 > t1);
    if (in) {
        float p[3];
        rayAt(R, t0, p);
        SlotCell c;
        if (!slotCell(M, ifloor(p[0]), ifloor(p[1]), ifloor(p[2]), c)) return false;
        HDDA h;
        h.init(R, t0, t1, c.dim > 8 ? c.dim : 8);
        for (;;) {
            const float ta = h.t0;
            const bool more = h.stepOnce();
            const float tb = fminf(h.t0, t1);
            const bool brick = !(c.entry & kSlotTile);
            if ((brick || (c.entry & kSlotTileOn)) && ta < tb) {
                const uint32_t base = brick ? c.entry * kBrickFloats : 0u;
                float kf = ceilf(ta / dt);
                while (kf * dt < tb) {
                    // step numbers are whole floats: exact to 2^24, one at a time up there
                    const bool whole = fabsf(kf) < 16777000.0f;
                    const float t = (whole ? kf + float(q) : kf) * dt;
                    const bool ok = (q == 0 || whole) && t < tb;
                    const float x0 = __builtin_fmaf(t, R.dir[0], R.eye[0]), x1 = __builtin_fmaf(t, R.dir[1], R.eye[1]),
                                x2 = __builtin_fmaf(t, R.dir[2], R.eye[2]);
                    const float fx = floorf(x0), fy = floorf(x1), fz = floorf(x2);
                    const uint32_t rx = uint32_t(int32_t(fx) - c.ox), ry = uint32_t(int32_t(fy) - c.oy),
                                   rz = uint32_t(int32_t(fz) - c.oz);
                    const bool fast = brick && (rx | ry | rz) < 8u;
                    Cell cell;
                    brickCell(M, fast ? base + (rx * 9u + ry) * 9u + rz : 0u, cell);
                    float rho = trilerp(cell, x0 - fx, x1 - fy, x2 - fz);
                    bool open = false;
                    // a tile, or a position that rounding put just outside its slot
                    if (ok && !fast) open = !slotTrilinear(M, x0, x1, x2, rho);
                    const uint32_t quad = threadIdx.x & 60u;
                    if ((__ballot(open) >> quad) & 15u) return false; // the whole quad
                    const uint32_t valid = uint32_t(__ballot(ok) >> quad) & 15u;
                    const float a = stepAbsorption(sigma, rho, dt);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float rj = quadLane(rho, j), aj = quadLane(a, j);
                        const float Ln = L + T * (1.0f - aj) * rj, Tn = T * aj;
                        const bool use = (valid >> j) & 1u;
                        L = use ? Ln : L;
                        T = use ? Tn : T;
                    }
                    if (!whole) {
                        const float kn = kf + 1.0f;
                        if (kn == kf) break;
                        kf = kn;
                    } else {
                        if (valid != 15u) break;
                        kf += 4.0f;
                    }
                }
            }
            if (!more) break;
            rayAt(R, h.t0 + Delta, p);
            if (!slotCell(M, ifloor(p[0]), ifloor(p[1]), ifloor(p[2]), c)) return false;
            h.update(R, c.dim > 8 ? c.dim : 8);
        }
    }
    if (q == 0) {
        if (Lout) Lout[i] = L;
        if (Tout) Tout[i] = T;
    }
    return true;
}

} // namespace nvq
