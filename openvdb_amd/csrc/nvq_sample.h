// Per-query point sampling through the lane accessor: SampleFromVoxels<Acc,0> (nearest),
// <Acc,1> (trilinear) and the three gradient modes, shared by the direct kernels and the
// fallback of the binned path.
#pragma once
#include "nvq_device.h"

namespace nvq {

// Grid::worldToIndex for a Vec3f (FP64 Map, NanoVDB.h:1507-1510, math/Math.h:1718-1723)
__device__ __forceinline__ void worldToIndexF64(const GridView& g, float p[3])
{
    float t[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) t[a] = float(double(p[a]) - g.vecD[a]);
#pragma unroll
    for (int r = 0; r < 3; ++r)
        p[r] = float(__builtin_fma(double(t[0]), g.invMatD[3 * r],
                                   __builtin_fma(double(t[1]), g.invMatD[3 * r + 1], double(t[2]) * g.invMatD[3 * r + 2])));
}

struct SampleConsts {
    float fdx, fdy, fdz; // FD6 scale (BuildT).5/voxelSize, PySampleFromVoxels.cu:42
    float gsInv2dx;      // GradStencil mInv2Dx, math/Stencils.h:477
};

// One trilinear sample of the FD6 stencil at q, served from the 32-voxel plus-shaped block
// around the query's cell when its cell is the expected one, else from the accessor.
template<uint32_t GT>
__device__ __forceinline__ float fd6Sample(Accessor<GT>& acc, float qx, float qy, float qz, int32_t ei, int32_t ej,
                                           int32_t ek, const Cell& blk)
{
    const float fx = floorf(qx), fy = floorf(qy), fz = floorf(qz);
    const int32_t bi = int32_t(fx), bj = int32_t(fy), bk = int32_t(fz);
    if (bi == ei && bj == ej && bk == ek) return trilerp(blk, qx - fx, qy - fy, qz - fz);
    Cell c;
    stencil8(acc, bi, bj, bk, c);
    return trilerp(c, qx - fx, qy - fy, qz - fz);
}

// Result of one point query; fields that were not asked for hold 0.
struct SampleOut {
    float nn, val, g[3];
};

// Evaluate one query at index-space p: the nearest value when wantNN, the trilinear value when
// wantVal, and the gradient of the given mode (0 = none).
template<uint32_t GT>
__device__ __forceinline__ SampleOut sampleEval(Accessor<GT>& acc, const float p[3], bool wantNN, bool wantVal, int mode,
                                                const SampleConsts& k)
{
    SampleOut r{0.0f, 0.0f, {0.0f, 0.0f, 0.0f}};
    const float fx = floorf(p[0]), fy = floorf(p[1]), fz = floorf(p[2]);
    const int32_t i0 = int32_t(fx), j0 = int32_t(fy), k0 = int32_t(fz);
    const float u = p[0] - fx, v = p[1] - fy, w = p[2] - fz;
    Cell C;
    stencil8(acc, i0, j0, k0, C);
    if (wantNN) {
        // SampleFromVoxels<Acc,0>: getValue(Round(xyz)); Round uses rintf, which lands in this cell
        const int32_t ri = int32_t(rintf(p[0])) - i0, rj = int32_t(rintf(p[1])) - j0, rk = int32_t(rintf(p[2])) - k0;
        r.nn = ((ri | rj | rk) & ~1) ? acc.getValue(i0 + ri, j0 + rj, k0 + rk) : pick(C, ri, rj, rk);
    }
    if (wantVal) r.val = trilerp(C, u, v, w);
    float* o = r.g;
    if (mode == 1) {
        // FD6 of trilinear samples, python/cuda/PySampleFromVoxels.cu:42-47
        Cell B;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                B.v[0][b][e] = C.v[1][b][e];
                B.v[1][b][e] = acc.getValue(i0 + 2, j0 + b, k0 + e);
            }
        const float xp = fd6Sample(acc, p[0] + 1.0f, p[1] + 0.0f, p[2] + 0.0f, i0 + 1, j0, k0, B);
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                B.v[1][b][e] = C.v[0][b][e];
                B.v[0][b][e] = acc.getValue(i0 - 1, j0 + b, k0 + e);
            }
        const float xm = fd6Sample(acc, p[0] - 1.0f, p[1] - 0.0f, p[2] - 0.0f, i0 - 1, j0, k0, B);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                B.v[a][0][e] = C.v[a][1][e];
                B.v[a][1][e] = acc.getValue(i0 + a, j0 + 2, k0 + e);
            }
        const float yp = fd6Sample(acc, p[0] + 0.0f, p[1] + 1.0f, p[2] + 0.0f, i0, j0 + 1, k0, B);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                B.v[a][1][e] = C.v[a][0][e];
                B.v[a][0][e] = acc.getValue(i0 + a, j0 - 1, k0 + e);
            }
        const float ym = fd6Sample(acc, p[0] - 0.0f, p[1] - 1.0f, p[2] - 0.0f, i0, j0 - 1, k0, B);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                B.v[a][b][0] = C.v[a][b][1];
                B.v[a][b][1] = acc.getValue(i0 + a, j0 + b, k0 + 2);
            }
        const float zp = fd6Sample(acc, p[0] + 0.0f, p[1] + 0.0f, p[2] + 1.0f, i0, j0, k0 + 1, B);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                B.v[a][b][1] = C.v[a][b][0];
                B.v[a][b][0] = acc.getValue(i0 + a, j0 + b, k0 - 1);
            }
        const float zm = fd6Sample(acc, p[0] - 0.0f, p[1] - 0.0f, p[2] - 1.0f, i0, j0, k0 - 1, B);
        o[0] = (xp - xm) * k.fdx;
        o[1] = (yp - ym) * k.fdy;
        o[2] = (zp - zm) * k.fdz;
    } else if (mode == 2) {
        // GradStencil::moveTo(RoundDown(xyz)).gradient(), math/Stencils.h:148-152, 502-507
        o[0] = k.gsInv2dx * (acc.getValue(i0 + 1, j0, k0) - acc.getValue(i0 - 1, j0, k0));
        o[1] = k.gsInv2dx * (acc.getValue(i0, j0 + 1, k0) - acc.getValue(i0, j0 - 1, k0));
        o[2] = k.gsInv2dx * (acc.getValue(i0, j0, k0 + 1) - acc.getValue(i0, j0, k0 - 1));
    } else if (mode == 3) {
        trilinearGradient(C, u, v, w, o);
    }
    return r;
}

// The six FD6 sample points of the forward (sampleEval): p + (+-1 along one axis, +-0 on the others)
__host__ __device__ __forceinline__ void fd6Points(const float p[3], float q[6][3])
{
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const int ax = t >> 1;
        const bool plus = (t & 1) == 0;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const float dlt = b == ax ? 1.0f : 0.0f;
            q[t][b] = plus ? p[b] + dlt : p[b] - dlt;
        }
    }
}

// True when every voxel the query's terms reach lies in the plus-shaped block around its cell
// (cell + [-1, 2] on one axis, cell + [0, 1] on the others): always, except for FD6 sample points
// whose p +- 1 rounds into a cell other than the neighbouring one.  The cells' difference is taken, which is
// exact where it is one: floorf(p) + 1 rounds as p + 1 does, so that from 2^24 on the two agree on
// any cell.
__host__ __device__ __forceinline__ bool adjointInBlock(const float p[3], int mode)
{
    if (mode != 1) return true;
    float q[6][3];
    fd6Points(p, q);
    bool ok = true;
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const int ax = t >> 1;
        ok = ok && floorf(q[t][ax]) - floorf(p[ax]) == ((t & 1) ? -1.0f : 1.0f);
    }
    return ok;
}

// FD6 samples outside the block still start in [cell-1, cell+2], so that their corners lie in [cell-1, cell+3],
// below 2^23: p + 1 or p - 1 rounds up to the next whole number where p lies just under a power of two (or
// just under 0), never down past one.  Ordinary inputs hold such points in numbers: lattices whose
// spacing or map rounds a whole coordinate down.  False: NaN and larger coordinates, whose samples can
// land on either side.
__host__ __device__ __forceinline__ bool fd6Near(const float p[3])
{
    return fabsf(p[0]) < 8388608.0f && fabsf(p[1]) < 8388608.0f && fabsf(p[2]) < 8388608.0f;
}

// The FD6 gradient with each sample from its own cell, sampleEval's operations in their order; at(x, y, z) is
// the voxel's value.  One axis at a time: for the lanes whose samples leave the block.
template<class At>
__device__ __forceinline__ void sampleFd6Cells(At&& at, const float p[3], const SampleConsts& k, float grad[3])
{
    grad[0] = grad[1] = grad[2] = 0.0f;
#pragma unroll 1
    for (int axis = 0; axis < 3; ++axis) {
        float f[2];
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            const float d = side ? -1.0f : 1.0f;
            const float q0 = p[0] + (axis == 0 ? d : 0.0f), q1 = p[1] + (axis == 1 ? d : 0.0f), q2 = p[2] + (axis == 2 ? d : 0.0f);
            const float x = floorf(q0), y = floorf(q1), z = floorf(q2);
            Cell C;
#pragma unroll
            for (int s = 0; s < 8; ++s)
                C.v[s >> 2][(s >> 1) & 1][s & 1] = at(int32_t(x) + (s >> 2), int32_t(y) + ((s >> 1) & 1), int32_t(z) + (s & 1));
            f[side] = trilerp(C, q0 - x, q1 - y, q2 - z);
        }
        const float g = (f[0] - f[1]) * (axis == 0 ? k.fdx : (axis == 1 ? k.fdy : k.fdz));
        grad[0] = axis == 0 ? g : grad[0];
        grad[1] = axis == 1 ? g : grad[1];
        grad[2] = axis == 2 ? g : grad[2];
    }
}

// ------------------------------------------------------------------ staged queries
// The 8^3 slots that the block [cell-1, cell+2]^3 of a query overlaps (one or two per axis), resolved
// to their leaf or tile value in four stages (root, upper, lower, voxels), every load of a stage in
// flight at once.  Through the accessor each of the up to 32 voxels is its own guarded lookup and the
// lookups wait for each other: 1000 queries took 61 us, 300,007 took 163 us.
constexpr uint32_t kNoLeaf = 0xffffffffu;
struct BlockSlots {
    int32_t s0[3];    // first slot per axis
    uint32_t leaf[8]; // offset from leaf0 in units of 32 bytes, or kNoLeaf; slot (a, b, c) at 4a + 2b + c
    float tile[8];    // value of a slot without a leaf
    uint32_t index[8]; // index grids: its channel index
};

// False where the query goes through the accessor: a cell near the ends of the integer range, or leaves
// beyond the 32-bit offsets.  `keys`: fill index[].
template<uint32_t GT>
__device__ __forceinline__ bool resolveBlock(const GridView& g, int32_t i0, int32_t j0, int32_t k0, bool keys, BlockSlots& B)
{
    const int32_t cell[3] = {i0, j0, k0};
    bool two[3], ok = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        ok = ok && cell[a] > -(1 << 30) && cell[a] < (1 << 30);
        B.s0[a] = (cell[a] - 1) >> 3;
        const int32_t s1 = (cell[a] + 2) >> 3;
        two[a] = s1 != B.s0[a];
    }
    if (!ok) return false;
    auto need = [&](int s) { return (!(s & 4) || two[0]) && (!(s & 2) || two[1]) && (!(s & 1) || two[2]); };
    // root: the tile of each slot (a grid around the origin has one per octant)
    uint32_t part[3][2], tile[8], missing = 0; // tile: its number + 1, or 0
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) part[a][b] = uint32_t((B.s0[a] + b) << 3) >> 12;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        tile[s] = 0;
        missing += need(s) ? 1u : 0u;
    }
    for (uint32_t i = 0; i < g.tableSize && missing; ++i) { // uniform addresses: scalar loads
        const uint64_t key = ld_u64(g.root + rootHeaderSize(GT) + kTileSize * i);
        const uint32_t kx = uint32_t(key >> 42), ky = uint32_t(key >> 21) & 0x1fffffu, kz = uint32_t(key) & 0x1fffffu;
        const bool x[2] = {part[0][0] == kx, part[0][1] == kx}, y[2] = {part[1][0] == ky, part[1][1] == ky},
                   z[2] = {part[2][0] == kz, part[2][1] == kz};
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const bool is = x[s >> 2] && y[(s >> 1) & 1] && z[s & 1] && need(s) && tile[s] == 0; // the first match
            tile[s] = is ? i + 1u : tile[s];
            missing -= is ? 1u : 0u;
        }
    }
    const uint8_t* node[8];
    uint64_t entry[8]; // float bits or channel index of a slot that ends at the current level
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        node[s] = nullptr;
        entry[s] = 0;
        B.leaf[s] = kNoLeaf;
    }
    const uint64_t background =
        GT == GT_ONINDEX ? ld_u64(g.root + kIdxRootBackground) : uint64_t(__float_as_uint(g.background));
    {
        uint32_t mask[8];
        uint64_t e[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            mask[s] = 0;
            entry[s] = background;
            e[s] = 0;
            if (!need(s) || tile[s] == 0) continue;
            const uint8_t* t = g.root + rootHeaderSize(GT) + kTileSize * (tile[s] - 1u);
            e[s] = ld_u64(t + 8);
            entry[s] = GT == GT_ONINDEX ? ld_u64(t + kIdxTileValue) : uint64_t(ld_u32(t + 20));
        }
#pragma unroll
        for (int s = 0; s < 8; ++s)
            if (e[s]) node[s] = g.root + int64_t(e[s]);
        // upper
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if (!node[s]) continue;
            const uint32_t x = uint32_t(B.s0[0] + (s >> 2)), y = uint32_t(B.s0[1] + ((s >> 1) & 1)), z = uint32_t(B.s0[2] + (s & 1));
            const uint32_t n = (((x & 511u) >> 4) << 10) | (((y & 511u) >> 4) << 5) | ((z & 511u) >> 4);
            mask[s] = maskOn(node[s] + kUpCMask, n) ? 1u : 0u;
            e[s] = ld_u64(node[s] + kUpTable + 8 * n);
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if (!node[s]) continue;
            entry[s] = e[s];
            node[s] = mask[s] ? node[s] + int64_t(e[s]) : nullptr;
        }
        // lower
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            mask[s] = 0;
            e[s] = 0;
            if (!node[s]) continue;
            const uint32_t x = uint32_t(B.s0[0] + (s >> 2)), y = uint32_t(B.s0[1] + ((s >> 1) & 1)), z = uint32_t(B.s0[2] + (s & 1));
            const uint32_t n = ((x & 15u) << 8) | ((y & 15u) << 4) | (z & 15u);
            mask[s] = maskOn(node[s] + kLoCMask, n) ? 1u : 0u;
            e[s] = ld_u64(node[s] + kLoTable + 8 * n);
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if (!node[s]) continue;
            if (mask[s]) {
                const uint64_t off = uint64_t(node[s] + int64_t(e[s]) - g.leaf0);
                ok = ok && (off & 31u) == 0 && off < (uint64_t(kNoLeaf) << 5);
                B.leaf[s] = uint32_t(off >> 5);
            } else {
                entry[s] = e[s];
            }
        }
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        if constexpr (GT == GT_ONINDEX) {
            B.index[s] = uint32_t(entry[s]);
            B.tile[s] = 0.0f;
            if (!keys && need(s) && B.leaf[s] == kNoLeaf) B.tile[s] = g.channel[entry[s]];
        } else {
            B.tile[s] = __uint_as_float(uint32_t(entry[s]));
        }
    }
    return ok;
}

// The slot of voxel (x, y, z) of the block, its entries chosen without dynamic indexing.
template<class T>
__device__ __forceinline__ T pickSlot(const BlockSlots& B, const T (&v)[8], int32_t x, int32_t y, int32_t z)
{
    T v0 = v[0], v1 = v[1], v2 = v[2], v3 = v[3], v4 = v[4], v5 = v[5], v6 = v[6], v7 = v[7];
    asm("" : "+v"(v0), "+v"(v1), "+v"(v2), "+v"(v3), "+v"(v4), "+v"(v5), "+v"(v6), "+v"(v7));
    const bool a = (x >> 3) != B.s0[0], b = (y >> 3) != B.s0[1], c = (z >> 3) != B.s0[2];
    const T w0 = a ? v4 : v0, w1 = a ? v5 : v1, w2 = a ? v6 : v2, w3 = a ? v7 : v3;
    const T u0 = b ? w2 : w0, u1 = b ? w3 : w1;
    return c ? u1 : u0;
}

template<uint32_t GT>
__device__ __forceinline__ float blockVoxel(const GridView& g, const BlockSlots& B, int32_t x, int32_t y, int32_t z)
{
    const uint32_t leaf = pickSlot(B, B.leaf, x, y, z);
    float v = pickSlot(B, B.tile, x, y, z);
    if (leaf != kNoLeaf) v = Codec<GT>::get(g.leaf0 + (uint64_t(leaf) << 5), Accessor<GT>::leafOffset(x, y, z), g.channel);
    return v;
}

// sampleEval with its operations in its order, from the voxels of the block around the query's cell:
// at(dx, dy, dz) is the voxel at that offset from the cell's corner.  For queries whose FD6 cells are
// the neighbouring ones (adjointInBlock) and whose nearest voxel is a corner of the cell.
template<class At>
__device__ __forceinline__ SampleOut sampleFromBlock(At&& at, const float p[3], bool wantNN, bool wantVal, int mode,
                                                     const SampleConsts& k)
{
    const float fx = floorf(p[0]), fy = floorf(p[1]), fz = floorf(p[2]);
    const int32_t ri = int32_t(rintf(p[0])) - int32_t(fx), rj = int32_t(rintf(p[1])) - int32_t(fy),
                  rk = int32_t(rintf(p[2])) - int32_t(fz);
    const float u = p[0] - fx, v = p[1] - fy, w = p[2] - fz;
    Cell C;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 2; ++e) C.v[a][b][e] = at(a, b, e);
    SampleOut r{0.0f, 0.0f, {0.0f, 0.0f, 0.0f}};
    if (mode == 1) {
        // the layers next to the cell: [axis][side][the other two axes]
        float L[3][2][2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    L[0][s][a][b] = at(s ? 2 : -1, a, b);
                    L[1][s][a][b] = at(a, s ? 2 : -1, b);
                    L[2][s][a][b] = at(a, b, s ? 2 : -1);
                }
        if (wantNN) r.nn = pick(C, ri, rj, rk);
        if (wantVal) r.val = trilerp(C, u, v, w);
        float f[3][2];
#pragma unroll
        for (int axis = 0; axis < 3; ++axis)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                Cell D;
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        // near and far face of the neighbouring cell along the axis
                        const float edge = L[axis][s][a][b];
                        const float face = axis == 0 ? C.v[s][a][b] : (axis == 1 ? C.v[a][s][b] : C.v[a][b][s]);
                        const float lo = s ? face : edge, hi = s ? edge : face;
                        if (axis == 0) { D.v[0][a][b] = lo; D.v[1][a][b] = hi; }
                        if (axis == 1) { D.v[a][0][b] = lo; D.v[a][1][b] = hi; }
                        if (axis == 2) { D.v[a][b][0] = lo; D.v[a][b][1] = hi; }
                    }
                const float d = s ? 1.0f : -1.0f;
                const float qx = axis == 0 ? p[0] + d : p[0] + 0.0f, qy = axis == 1 ? p[1] + d : p[1] + 0.0f,
                            qz = axis == 2 ? p[2] + d : p[2] + 0.0f;
                f[axis][s] = trilerp(D, qx - floorf(qx), qy - floorf(qy), qz - floorf(qz));
            }
        r.g[0] = (f[0][1] - f[0][0]) * k.fdx;
        r.g[1] = (f[1][1] - f[1][0]) * k.fdy;
        r.g[2] = (f[2][1] - f[2][0]) * k.fdz;
        return r;
    }
    if (wantNN) r.nn = pick(C, ri, rj, rk);
    if (wantVal) r.val = trilerp(C, u, v, w);
    if (mode == 2) {
        const float mx = at(-1, 0, 0), my = at(0, -1, 0),
                    mz = at(0, 0, -1);
        r.g[0] = k.gsInv2dx * (C.v[1][0][0] - mx);
        r.g[1] = k.gsInv2dx * (C.v[0][1][0] - my);
        r.g[2] = k.gsInv2dx * (C.v[0][0][1] - mz);
    } else if (mode == 3) {
        trilinearGradient(C, u, v, w, r.g);
    }
    return r;
}

// Over resolved slots.  FD6 samples off the block (fd6Near) read the same slots, one axis at a time.
// False: through the accessor.
template<uint32_t GT>
__device__ __forceinline__ bool sampleStaged(const GridView& g, const float p[3], bool wantNN, bool wantVal, int mode,
                                             const SampleConsts& k, SampleOut& r)
{
    const int32_t i0 = int32_t(floorf(p[0])), j0 = int32_t(floorf(p[1])), k0 = int32_t(floorf(p[2]));
    const int32_t ri = int32_t(rintf(p[0])) - i0, rj = int32_t(rintf(p[1])) - j0, rk = int32_t(rintf(p[2])) - k0;
    const bool near = adjointInBlock(p, mode);
    BlockSlots B;
    if (((ri | rj | rk) & ~1) || !(near || fd6Near(p)) || !resolveBlock<GT>(g, i0, j0, k0, false, B)) return false;
    r = sampleFromBlock([&](int x, int y, int z) { return blockVoxel<GT>(g, B, i0 + x, j0 + y, k0 + z); }, p, wantNN,
                        wantVal, mode, k);
    if (!near)
        sampleFd6Cells([&](int32_t x, int32_t y, int32_t z) { return blockVoxel<GT>(g, B, x, y, z); }, p, k, r.g);
    return true;
}

// One query per lane.
template<uint32_t GT>
__device__ __forceinline__ SampleOut samplePoint(const GridView& g, const float p[3], bool wantNN, bool wantVal, int mode,
                                                 const SampleConsts& k)
{
    SampleOut r{0.0f, 0.0f, {0.0f, 0.0f, 0.0f}};
    if (!sampleStaged<GT>(g, p, wantNN, wantVal, mode, k, r)) {
        Accessor<GT> acc(g);
        r = sampleEval(acc, p, wantNN, wantVal, mode, k);
    }
    return r;
}

// ------------------------------------------------------------------ adjoint of the point queries
// (no counterpart in the reference, whose sampler has no backward)
//
// Every output of a query is linear in the voxel values it reads, so dLoss/dvalue of one query is
// a sum of terms, one per output: the trilinear value (math/SampleFromVoxels.h:423-476), the
// gradient (FD6 of six trilinear samples, python/cuda/PySampleFromVoxels.cu:42-47; GradStencil,
// math/Stencils.h:502-507; TrilinearSampler::gradient, math/SampleFromVoxels.h:232-271) and the
// nearest value.  A term reaches the eight corners (o + (a,b,e)) of one trilinear cell with weight
// ((s * A[a]) * B[b]) * C[e], where s is the upstream gradient times the output's constant and
// A, B, C the per-axis weights of d output / d corner: (1-u, u) for an interpolation along the
// axis, (-1, +1) for a difference along it.  A single term reaches one voxel with weight s.
//
// Contract (what makes every schedule and both launch paths bit-identical): for each distinct
// voxel, the query's contribution is the FP32 sum, in term order, of that voxel's term weights,
// starting from +0; terms whose s is zero are left out.  Term order: value, then gradient (FD6:
// +x, -x, +y, -y, +z, -z samples; GradStencil: +x, -x, +y, -y, +z, -z voxels; trilinear: d/dx,
// d/dy, d/dz), then nearest.  The contribution is converted once, to int64 fixed point
// (round to nearest even, saturating), and integer-added into the accumulator.
struct SampleGrad {
    float gn, gv, gg[3]; // dLoss / d(nearest, value, gradient xyz) of one query
};

// float -> int64 fixed point, round to nearest, saturating at +-2^62 (float->int conversion is
// undefined beyond the int64 range); a non-finite or saturated value clears `ok`.
__device__ __forceinline__ long long toFixedSat(float x, bool& ok)
{
    constexpr float kLim = 4611686018427387904.0f; // 2^62
    if (fabsf(x) < kLim) return __float2ll_rn(x);
    ok = false;
    if (x != x) return 0;
    return x > 0.0f ? (1ll << 62) : -(1ll << 62);
}

// General form of the sums, for FD6 sample cells anywhere (coordinates from 2^23 on): the whole wavefront takes one query, lane 8 t + c holding corner c of term t.
// Terms are numbered in the contract's order, so a voxel's sum is that of its lanes in lane order, and
// its first lane emits it.  (One lane looping over all pairs of corners took 330 us.)
// emit(x, y, z, contribution).  Every lane calls this with the same query.
template<class Emit>
__device__ __forceinline__ void sampleAdjointWave(const float p[3], const SampleGrad& d, int mode, const SampleConsts& k,
                                                  Emit& emit)
{
    const uint32_t lane = threadIdx.x & 63u, mine = lane >> 3, c = lane & 7u;
    uint32_t terms = 0;
    int32_t x = 0, y = 0, z = 0;
    float w = 0.0f;
    bool have = false;
    const float fx = floorf(p[0]), fy = floorf(p[1]), fz = floorf(p[2]);
    const int32_t i0 = int32_t(fx), j0 = int32_t(fy), k0 = int32_t(fz);
    const float u = p[0] - fx, v = p[1] - fy, t = p[2] - fz;
    auto cellTerm = [&](int32_t ox, int32_t oy, int32_t oz, float s, float a0, float a1, float b0, float b1, float c0,
                        float c1) {
        if (terms++ != mine) return;
        x = ox + int32_t(c >> 2);
        y = oy + int32_t((c >> 1) & 1u);
        z = oz + int32_t(c & 1u);
        w = ((s * ((c & 4u) ? a1 : a0)) * ((c & 2u) ? b1 : b0)) * ((c & 1u) ? c1 : c0);
        have = true;
    };
    if (d.gv != 0.0f) cellTerm(i0, j0, k0, d.gv, 1.0f - u, u, 1.0f - v, v, 1.0f - t, t);
    float q[6][3];
    fd6Points(p, q);
    const float fd[3] = {k.fdx, k.fdy, k.fdz};
#pragma unroll
    for (int n = 0; n < 6; ++n) {
        const float s0 = d.gg[n >> 1] * fd[n >> 1];
        const float s = (n & 1) ? -s0 : s0;
        if (s == 0.0f) continue;
        const float gx = floorf(q[n][0]), gy = floorf(q[n][1]), gz = floorf(q[n][2]);
        const float a = q[n][0] - gx, b = q[n][1] - gy, e = q[n][2] - gz;
        cellTerm(int32_t(gx), int32_t(gy), int32_t(gz), s, 1.0f - a, a, 1.0f - b, b, 1.0f - e, e);
    }
    if (d.gn != 0.0f && terms == mine && c == 0) {
        x = int32_t(rintf(p[0]));
        y = int32_t(rintf(p[1]));
        z = int32_t(rintf(p[2]));
        w = d.gn;
        have = true;
    }
    float sum = 0.0f;
    bool first = have;
#pragma unroll 4
    for (int j = 0; j < 64; ++j) {
        const bool same = __builtin_amdgcn_readlane(int(have), j) && __builtin_amdgcn_readlane(x, j) == x &&
                          __builtin_amdgcn_readlane(y, j) == y && __builtin_amdgcn_readlane(z, j) == z;
        const float wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), j));
        if (same) {
            first = first && j >= int(lane);
            sum += wj;
        }
    }
    if (first) emit(x, y, z, sum);
}

// The same sums where the FD6 cells are off the block but near it (fd6Near): the voxels they reach are the
// cell's eight and, per axis, the layers at -1, 2 and 3, which only that axis's two samples reach.  One
// voxel at a time, its terms in order.
template<class Emit>
__device__ __forceinline__ void sampleAdjointNear(const float p[3], const SampleGrad& d, const SampleConsts& k, Emit& emit)
{
    int32_t cell[3], nearest[3], o[6]; // o: cell of a sample along its axis, from `cell`
    float f[3], q[6][3], s[6], a[6];
    const float fd[3] = {k.fdx, k.fdy, k.fdz};
    fd6Points(p, q);
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const float whole = floorf(p[b]);
        cell[b] = int32_t(whole);
        f[b] = p[b] - whole;
        nearest[b] = int32_t(rintf(p[b])) - cell[b];
    }
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const float whole = floorf(q[t][t >> 1]), s0 = d.gg[t >> 1] * fd[t >> 1];
        o[t] = int32_t(whole) - cell[t >> 1];
        a[t] = q[t][t >> 1] - whole;
        s[t] = (t & 1) ? -s0 : s0;
    }
    auto weight = [](float frac, int32_t side) { return side ? frac : 1.0f - frac; };
#pragma unroll 1
    for (uint32_t v = 0; v < 44u; ++v) {
        // voxels 0..7: the cell's; 8 + 12 axis + 4 layer + side: on the layers
        const uint32_t w = v - 8u, axis = v < 8u ? 3u : w / 12u, layer = (w >> 2) % 3u;
        const int32_t far = layer == 0 ? -1 : int32_t(layer) + 1, hi = int32_t(v >> 1) & 1, lo = int32_t(v) & 1;
        const int32_t e[3] = {axis == 0 ? far : (axis == 3 ? int32_t(v >> 2) : hi), axis == 1 ? far : (axis == 2 ? lo : hi),
                              axis == 2 ? far : lo};
        const int32_t x[3] = {axis == 0 ? 0 : e[0], axis == 1 ? 0 : e[1], axis == 2 ? 0 : e[2]}; // sides of the other axes
        float sum = 0.0f;
        if (axis == 3u && d.gv != 0.0f) sum += ((d.gv * weight(f[0], x[0])) * weight(f[1], x[1])) * weight(f[2], x[2]);
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            const uint32_t ax = uint32_t(t) >> 1;
            const int32_t side = e[ax] - o[t];
            if (s[t] == 0.0f || (axis != 3u && axis != ax) || uint32_t(side) > 1u) continue;
            const float wx = ax == 0 ? weight(a[t], side) : weight(f[0], x[0]), wy = ax == 1 ? weight(a[t], side) : weight(f[1], x[1]),
                        wz = ax == 2 ? weight(a[t], side) : weight(f[2], x[2]);
            sum += ((s[t] * wx) * wy) * wz;
        }
        if (d.gn != 0.0f && e[0] == nearest[0] && e[1] == nearest[1] && e[2] == nearest[2]) sum += d.gn;
        emit(cell[0] + e[0], cell[1] + e[1], cell[2] + e[2], sum);
    }
}

// Block form of the same sums (requires adjointInBlock): 32 register accumulators at constant
// offsets; emit(x, y, z, contribution) for each of the 32 voxels of the plus-shaped block.
template<class Emit>
__host__ __device__ __forceinline__ void sampleAdjointBlock(const float p[3], const SampleGrad& d, int mode,
                                                   const SampleConsts& k, Emit& emit)
{
    const float fx = floorf(p[0]), fy = floorf(p[1]), fz = floorf(p[2]);
    const int32_t i0 = int32_t(fx), j0 = int32_t(fy), k0 = int32_t(fz);
    const float u = p[0] - fx, v = p[1] - fy, w = p[2] - fz;
    float bx[4][4][4]; // voxel (i0-1+x, j0-1+y, k0-1+z); only the plus-shaped 32 are used
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int z = 0; z < 4; ++z) bx[x][y][z] = 0.0f;
    auto cell = [&](int da, int db, int de, float s, const float A[2], const float B[2], const float C[2]) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int e = 0; e < 2; ++e) bx[da + a + 1][db + b + 1][de + e + 1] += ((s * A[a]) * B[b]) * C[e];
    };
    const float Wu[2] = {1.0f - u, u}, Wv[2] = {1.0f - v, v}, Ww[2] = {1.0f - w, w}, Dm[2] = {-1.0f, 1.0f};
    if (d.gv != 0.0f) cell(0, 0, 0, d.gv, Wu, Wv, Ww);
    if (mode == 1) {
        float q[6][3];
        fd6Points(p, q);
        const float fd[3] = {k.fdx, k.fdy, k.fdz};
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            const int ax = t >> 1;
            const float s0 = d.gg[ax] * fd[ax];
            const float s = (t & 1) ? -s0 : s0;
            if (s == 0.0f) continue;
            float A[3][2];
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                const float fr = q[t][b] - floorf(q[t][b]);
                A[b][0] = 1.0f - fr;
                A[b][1] = fr;
            }
            const int off = (t & 1) ? -1 : 1;
            cell(ax == 0 ? off : 0, ax == 1 ? off : 0, ax == 2 ? off : 0, s, A[0], A[1], A[2]);
        }
    } else if (mode == 2) {
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            const float s = k.gsInv2dx * d.gg[ax];
            if (s == 0.0f) continue;
            bx[1 + (ax == 0)][1 + (ax == 1)][1 + (ax == 2)] += s;
            bx[1 - (ax == 0)][1 - (ax == 1)][1 - (ax == 2)] += -s;
        }
    } else if (mode == 3) {
        if (d.gg[0] != 0.0f) cell(0, 0, 0, d.gg[0], Dm, Wv, Ww);
        if (d.gg[1] != 0.0f) cell(0, 0, 0, d.gg[1], Wu, Dm, Ww);
        if (d.gg[2] != 0.0f) cell(0, 0, 0, d.gg[2], Wu, Wv, Dm);
    }
    if (d.gn != 0.0f) {
        // Round lands in the cell: offsets in {0, 1}; adding +0 to the other corners leaves their
        // fixed-point value unchanged
        const int32_t ri = int32_t(rintf(p[0])) - i0, rj = int32_t(rintf(p[1])) - j0, rk = int32_t(rintf(p[2])) - k0;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int e = 0; e < 2; ++e) bx[a + 1][b + 1][e + 1] += (ri == a && rj == b && rk == e) ? d.gn : 0.0f;
    }
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int z = 0; z < 4; ++z) {
                const int out = (x == 0 || x == 3) + (y == 0 || y == 3) + (z == 0 || z == 3);
                if (out <= 1) emit(i0 - 1 + x, j0 - 1 + y, k0 - 1 + z, bx[x][y][z]);
            }
}

// Leaf-value key of a probed voxel: Float grids leaf index * 512 + voxel offset (-1 outside
// leaves), index grids the channel index.  Float leaves are 2144 B = 32 * 67.
template<uint32_t GT>
__device__ __forceinline__ int64_t adjointKey(const GridView& g, const Probe& pr)
{
    if constexpr (GT == GT_ONINDEX) return int64_t(pr.index);
    else return pr.leaf ? int64_t((uint64_t(pr.leaf - g.leaf0) >> 5) / 67u) * 512 + pr.n : -1;
}

// One query per lane, added into accum with int64 atomics; every lane of the wavefront calls this,
// `valid` or not.
template<uint32_t GT>
__device__ __forceinline__ void sampleAdjointLanes(const GridView& g, bool valid, const float p[3], const SampleGrad& d,
                                                   int mode, const SampleConsts& k, float scale,
                                                   unsigned long long* __restrict__ accum, bool& ok)
{
    auto emit = [&](int32_t x, int32_t y, int32_t z, float sum) {
        const long long q = toFixedSat(sum * scale, ok);
        if (q == 0) return;
        Accessor<GT> acc(g);
        const int64_t key = adjointKey<GT>(g, acc.probe(x, y, z));
        if (key >= 0) atomicAdd(accum + key, static_cast<unsigned long long>(q));
    };
    const bool near = adjointInBlock(p, mode), off = valid && !near && !fd6Near(p);
    if (valid && !off) {
        BlockSlots B;
        if (resolveBlock<GT>(g, int32_t(floorf(p[0])), int32_t(floorf(p[1])), int32_t(floorf(p[2])), true, B)) {
            auto staged = [&](int32_t x, int32_t y, int32_t z, float sum) {
                const long long q = toFixedSat(sum * scale, ok);
                if (q == 0) return;
                const uint32_t leaf = pickSlot(B, B.leaf, x, y, z), n = Accessor<GT>::leafOffset(x, y, z);
                int64_t key;
                if constexpr (GT == GT_ONINDEX)
                    key = leaf != kNoLeaf ? int64_t(Codec<GT_ONINDEX>::index(g.leaf0 + (uint64_t(leaf) << 5), n))
                                          : int64_t(pickSlot(B, B.index, x, y, z));
                else
                    key = leaf != kNoLeaf ? int64_t(leaf / 67u) * 512 + n : -1;
                if (key >= 0) atomicAdd(accum + key, static_cast<unsigned long long>(q));
            };
            if (near) sampleAdjointBlock(p, d, mode, k, staged);
            else sampleAdjointNear(p, d, k, staged);
        } else if (near) { // a cell whose block's slots are not resolved: beyond the range of fd6Near, or odd leaves
            sampleAdjointBlock(p, d, mode, k, emit);
        } else {
            sampleAdjointNear(p, d, k, emit);
        }
    }
    uint64_t todo = __ballot(off);
    while (todo) {
        const int src = __builtin_ctzll(todo);
        todo &= todo - 1u;
        const float P[3] = {__shfl(p[0], src, 64), __shfl(p[1], src, 64), __shfl(p[2], src, 64)};
        SampleGrad D;
        D.gn = __shfl(d.gn, src, 64);
        D.gv = __shfl(d.gv, src, 64);
#pragma unroll
        for (int a = 0; a < 3; ++a) D.gg[a] = __shfl(d.gg[a], src, 64);
        sampleAdjointWave(P, D, mode, k, emit);
    }
}

inline SampleConsts sampleConsts(const GridView& g)
{
    SampleConsts k;
    k.fdx = float(0.5 / g.voxelSize[0]);
    k.fdy = float(0.5 / g.voxelSize[1]);
    k.fdz = float(0.5 / g.voxelSize[2]);
    k.gsInv2dx = float(0.5 / g.voxelSize[0]);
    return k;
}

} // namespace nvq
