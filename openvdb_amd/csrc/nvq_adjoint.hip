// Adjoint of the emission-absorption fog march with respect to the leaf values of a Float grid,
// or the channel values of an index grid (no counterpart in the reference, which has no
// differentiable path).
//
// Forward (per ray, steps k = 0..N-1 from the shared marchSteps structure):
//   rho_k = trilinear(x_k), a_k = exp(-s*rho_k) with s = sigma*dt,
//   L = sum_k T_k (1-a_k) rho_k,  T_{k+1} = T_k a_k,  T_0 = 1.
// Adjoint:
//   dLoss/drho_k = gL * (T_k [(1-a_k) + rho_k s a_k] - s R_k) - gT * s * T_N,
//   R_k = sum_{j>k} T_j (1-a_j) rho_j = L - L_{<=k}.
// The backward kernel re-marches each ray with the identical FP32 step structure and
// arithmetic, so T_k and the running radiance L_{<=k} are recomputed bit for bit instead of
// stored per step; L and T_N come from the forward outputs.  dLoss/drho_k is spread over the
// eight trilinear corners of step k with weights (1-u|u)(1-v|v)(1-w|w).
//
// Deterministic reduction: contributions are first summed per ray and per corner voxel over
// the run of consecutive steps whose trilinear cells contain that voxel (a segmented reduction
// in the sliding corner window), then added into an int64 fixed-point accumulator per leaf
// value (key = leaf index * 512 + voxel offset) with integer atomics.  Integer addition is associative, so the result does not
// depend on thread scheduling; the accumulator is converted through FP64.
// Two kernels share this contract and give the same bits: k_fog_march_bwd_blocks over a slot map, and
// k_fog_march_bwd through the accessor for grids too large for one.
#include "nvq_device.h"
#include "nvq_internal.h"
#include "nvq_profile.h"
#include "nvq_slots.h"
#include "../../include/nvq.h"

#include <hip/hip_runtime.h>

#include <cstring>

namespace nvq {
namespace {
// The block cache of the tiled adjoint (k_fog_march_bwd_blocks).  Measured on 64 cameras of 256^2 rays
// and a 256^3 fog, forward and adjoint: 256 entries 32.7 ms (18 KB: two wavefronts per SIMD),
// 128 entries 25.7, 64 entries 25.4 of an earlier form; written back every 2 steps 16.3 ms,
// every 4 15.5, every 8 16.5; one step between looks at the wavefront's slowest ray 15.5 ms,
// four 15.7 with a lag of 4 steps, 14.0 with 8, 14.4 with 12.
constexpr uint32_t kCacheMisses = 64; // and kCacheBlocks entries
constexpr uint32_t kCacheSteps = 4, kCacheAge = 4; // write back every kCacheSteps what is kCacheAge old
constexpr float kCacheLag = 8.0f;                  // steps a ray may be ahead of the slowest
// That rule counts steps from the ray's eye and keeps rays of an image side by side.  Rays of a batch
// without an image width may have their first steps far apart (other cameras, other distances): side by side
// they would only wait for each other, one after the other.  Up to this spread of first steps such a
// wavefront keeps the rule, beyond it its rays run freely.  2^18 rays and a 256^3 fog, with the rule, without
// it, and by spread of 64, 200 and 500 steps: cameras at 16 distances shuffled 7.86, 2.49, 2.49, 2.49, 2.48 ms
// (accessor 6.38), 128^3: 3.77, 1.18, 1.18, 1.18, 1.86 (3.22); one image as rows of rays 2.82, 3.29, 2.88,
// 2.79, 2.78 (11.6); 2^20 rays of 16 images in a row 3.25, 4.02, 3.86, 3.41, 3.26 (12.0); scattered rays from one distance
// 5.01, 5.45, 5.48, 5.47, 5.04 (12.5), from four distances 11.6, 5.40, 5.40, 5.42, 5.42 (12.4).
constexpr float kCacheSpread = 200.0f;
constexpr uint32_t kMaxBlockLeaves = 1u << 20;

// float -> int64 fixed point, round to nearest, saturating at +-2^62 (float->int conversion is
// undefined beyond the int64 range); a non-finite or saturated value clears `ok`.
__device__ __forceinline__ long long toFixed(float x, bool& ok)
{
    constexpr float kLim = 4611686018427387904.0f; // 2^62
    if (fabsf(x) < kLim) return __float2ll_rn(x);
    ok = false;
    if (x != x) return 0;
    return x > 0.0f ? (1ll << 62) : -(1ll << 62);
}

__global__ void k_clear_flag(uint32_t* flag) { *flag = 0u; }

template<uint32_t GT>
__global__ __launch_bounds__(kBlock) void k_fog_march_bwd(GridView g, const float* __restrict__ eye,
                                                          const float* __restrict__ dir, Sched s,
                                                          const uint32_t* __restrict__ order, float dt, float sigma,
                                                          const float* __restrict__ Lfwd, const float* __restrict__ Tfwd,
                                                          const float* __restrict__ gLin, const float* __restrict__ gTin,
                                                          unsigned long long* __restrict__ accum, float scale,
                                                          uint32_t* __restrict__ overflow)
{
    uint64_t i;
    if (!scheduleOrdered(s, order, i)) return;
    const float gL = gLin ? gLin[i] : 0.0f, gT = gTin ? gTin[i] : 0.0f;
    if (gL == 0.0f && gT == 0.0f) return;
    Accessor<GT> acc(g);
    const float e[3] = {eye[3 * i], eye[3 * i + 1], eye[3 * i + 2]};
    const float d[3] = {dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
    const float Ltot = Lfwd[i];
    const float sdt = sigma * dt;
    const float tTerm = gTin ? gT * sdt * Tfwd[i] : 0.0f; // Tfwd may be NULL when no dL/dT is given
    float L = 0.0f, T = 1.0f;
    CellWindow<true> W;
    bool range = true; // every contribution converted without saturation
    auto sink = [&](int32_t key, float sum) {
        const long long q = toFixed(sum * scale, range);
        if (q != 0) atomicAdd(accum + key, static_cast<unsigned long long>(q));
    };
    marchSteps(acc, g, e, d, dt, [&](float x0, float x1, float x2) {
        const float fx = floorf(x0), fy = floorf(x1), fz = floorf(x2);
        W.moveTo(acc, g, int32_t(fx), int32_t(fy), int32_t(fz), sink);
        const float u = x0 - fx, v = x1 - fy, w = x2 - fz;
        const float rho = trilerp(W.c, u, v, w);
        const float a = stepAbsorption(sigma, rho, dt);
        L += T * (1.0f - a) * rho;        // same operations as the forward march
        const float R = Ltot - L;         // radiance of the later steps
        const float gk = gL * (T * ((1.0f - a) + rho * sdt * a) - sdt * R) - tTerm;
        T *= a;
        // corner (a,b,c) receives gk * wx[a] * wy[b] * wz[c], factored as (gk wx wy) wz and fused
        // into the running sum: 6 products and 8 fmas per step
        const float gx[2] = {gk * (1.0f - u), gk * u};
        const float wy[2] = {1.0f - v, v}, wz[2] = {1.0f - w, w};
#pragma unroll
        for (int aa = 0; aa < 2; ++aa)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const float gxy = gx[aa] * wy[b];
#pragma unroll
                for (int c = 0; c < 2; ++c) W.sum[aa * 4 + b * 2 + c] = fmaf(gxy, wz[c], W.sum[aa * 4 + b * 2 + c]);
            }
    });
    W.flush(sink);
    if (!range) atomicOr(overflow, 1u);
}

// Accumulator key of voxel (x, y, z): leaf * 512 + offset (Float; -1 outside leaves) or the channel
// index it reads (index grids), through the slot map where that resolves it, else the tree.
template<uint32_t GT>
__device__ __forceinline__ int32_t voxelKey(const SlotMap& M, const GridView& g, int32_t x, int32_t y, int32_t z)
{
    uint32_t i;
    const uint32_t n = Accessor<GT>::leafOffset(x, y, z);
    const uint32_t e = slotAt(M, x, y, z, i) ? M.entry[i] : kSlotOther;
    if (e == kSlotOther) {
        Accessor<GT> acc(g);
        const Probe p = acc.probe(x, y, z);
        if constexpr (GT == GT_ONINDEX) return int32_t(p.index);
        else return p.leaf ? int32_t((uint32_t(uint64_t(p.leaf - g.leaf0) >> 5) / 67u) * 512u + p.n) : -1;
    }
    if constexpr (GT == GT_ONINDEX) {
        if (e & kSlotTile) return int32_t(M.tileIndex[i]);
        return int32_t(Codec<GT_ONINDEX>::index(g.leaf0 + uint64_t(e) * g.leafSize, n));
    } else {
        return (e & kSlotTile) ? -1 : int32_t(e * 512u + n);
    }
}

// Value of voxel (x, y, z) through the tree.
template<uint32_t GT>
__device__ __forceinline__ float treeTrilinear(const GridView& g, float px, float py, float pz)
{
    const float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
    const int32_t x = int32_t(fx), y = int32_t(fy), z = int32_t(fz);
    Accessor<GT> acc(g);
    float v[2], row[2];
#pragma unroll 1
    for (int a = 0; a < 2; ++a) {
#pragma unroll 1
        for (int b = 0; b < 2; ++b) {
            const float c0 = acc.getValue(x + a, y + b, z), c1 = acc.getValue(x + a, y + b, z + 1);
            row[1] = lerpf(c0, c1, pz - fz);
            row[0] = b ? row[0] : row[1];
        }
        v[1] = lerpf(row[0], row[1], py - fy);
        v[0] = a ? v[0] : v[1];
    }
    return lerpf(v[0], v[1], px - fx);
}

// ------------------------------------------------------------------ block cache
// int64 sums of 2x2x2 voxel blocks on their way to the accumulator, one cache per wavefront in LDS.
// A block's tag is its linear position in the table's box, with strides (sx, sy, 1) whose low bits
// spread the blocks of a wavefront's slab over the entries: entry = tag mod kCacheBlocks.  10 KB:
// sixteen wavefronts to a CU's LDS.
struct BlockCache {
    unsigned long long q[kCacheBlocks * 8];
    unsigned long long missQ[kCacheMisses]; // sums whose entry was taken, and their pos * 8 + word
    uint32_t missAt[kCacheMisses];
    uint32_t tag[kCacheBlocks];             // kNoBlock: free
    uint32_t pos[kCacheBlocks];             // slot * 64 + block in the slot
    uint8_t born[kCacheBlocks];             // step that claimed the entry, mod 256
    uint8_t list[kCacheBlocks];             // entries to write back
};
static_assert(kCacheBlocks <= 256, "list holds bytes");

__device__ __forceinline__ float waveMinDpp(float x)
{
    auto step = [&](auto ctrl, auto rows) {
        const int o = __builtin_amdgcn_update_dpp(__float_as_int(x), __float_as_int(x), decltype(ctrl)::value,
                                                  decltype(rows)::value, 0xf, false);
        x = fminf(x, __int_as_float(o));
    };
    step(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{}); // row_shr 1, 2, 4, 8
    step(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{}); // row_bcast 15, 31
    step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// Where the sums of block `pos` (slot * 64 + block in the slot) go: a block of scratch (leaf * 64 +
// block), kDestTile plus a channel index (index grids: all eight voxels read it), or nowhere (Float
// tiles).
constexpr uint32_t kDestTile = 0x80000000u, kDestNone = 0xffffffffu, kDestTree = 0xfffffffeu;
template<uint32_t GT>
__device__ __forceinline__ uint32_t blockDest(const SlotMap& M, uint32_t pos)
{
    const uint32_t i = pos >> 6, e = M.entry[i];
    if (!(e & kSlotTile)) return e * 64u + (pos & 63u);
    if (e == kSlotOther) return kDestTree;
    return GT == GT_ONINDEX ? kDestTile | M.tileIndex[i] : kDestNone;
}

// Adds q to word w (the voxel's parities) of the block.
template<uint32_t GT>
__device__ __forceinline__ void blockAdd(const SlotMap& M, const GridView& g, unsigned long long* __restrict__ blocks,
                                         unsigned long long* __restrict__ accum, uint32_t pos, uint32_t dest,
                                         uint32_t w, unsigned long long q)
{
    if (!(dest & kDestTile)) {
        atomicAdd(blocks + (uint64_t(dest) * 8u + w), q);
    } else if (dest == kDestTree) {
        const uint32_t i = pos >> 6, z = i % M.n[2], r = i / M.n[2], y = r % M.n[1], x = r / M.n[1];
        const int32_t key = voxelKey<GT>(M, g, ((M.lo[0] + int32_t(x)) << 3) + int32_t(((pos >> 4) & 3u) * 2u + (w >> 2)),
                                         ((M.lo[1] + int32_t(y)) << 3) + int32_t(((pos >> 2) & 3u) * 2u + ((w >> 1) & 1u)),
                                         ((M.lo[2] + int32_t(z)) << 3) + int32_t((pos & 3u) * 2u + (w & 1u)));
        if (key >= 0) atomicAdd(accum + key, q);
    } else if (GT == GT_ONINDEX && dest != kDestNone) {
        atomicAdd(accum + (dest & ~kDestTile), q);
    }
}

// The adjoint over a slot map, one wavefront per ray tile.  Global atomics are paid per 64-byte block
// that one instruction touches, not per lane: a microbenchmark on 74 MB of int64 gave 24 G atomics/s
// to random words, 47 to pairs, 95 to quads and 188 to whole blocks.  Added one voxel at a time, the
// 827 M sums that leave the windows of 64 x 256^2 rays took 33.8 ms of which the march was 3.  So a
// wavefront gathers them in LDS by 2x2x2 block: neighbouring rays fill a block within a few steps,
// and its eight words leave together.  For that the rays of a tile march side by side (none more
// than kCacheLag steps ahead of the slowest), every step one flush of the whole wavefront.  The
// accumulator's own order splits a block over four 64-byte lines, so the blocks go to scratch and
// k_fold_blocks adds them up afterwards; integer sums, so the order does not matter.
// 10.6 ms for the 64 x 256^2 rays (36.2 ms through the accessor), bound by the VALU at 4 wavefronts per SIMD:
// 4.85 G wavefront instructions, 81 % of the issue slots of busy CUs.
template<uint32_t GT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_fog_march_bwd_blocks(SlotMap M, BlockBox X, GridView g, const float* __restrict__ eye,
                                                             const float* __restrict__ dir, Sched s,
                                                             const uint32_t* __restrict__ order, float dt, float sigma,
                                                             const float* __restrict__ Lfwd,
                                                             const float* __restrict__ Tfwd,
                                                             const float* __restrict__ gLin,
                                                             const float* __restrict__ gTin,
                                                             unsigned long long* __restrict__ blocks,
                                                             unsigned long long* __restrict__ accum, float scale,
                                                             uint32_t* __restrict__ overflow)
{
    __shared__ BlockCache C;
    const uint32_t lane = threadIdx.x;
    for (uint32_t k = lane; k < kCacheBlocks; k += 64u) {
        C.tag[k] = kNoBlock;
#pragma unroll
        for (uint32_t w = 0; w < 8; ++w) C.q[w * kCacheBlocks + k] = 0ull;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    uint64_t i = 0;
    bool alive = tileRay(s, order ? order[blockIdx.x] : blockIdx.x, lane, i);
    float gL = 0.0f, gT = 0.0f, Ltot = 0.0f, tTerm = 0.0f;
    const float sdt = sigma * dt;
    if (alive) {
        gL = gLin ? gLin[i] : 0.0f;
        gT = gTin ? gTin[i] : 0.0f;
        alive = !(gL == 0.0f && gT == 0.0f);
    }
    Ray R;
    const float Eps = 0.000001f, Delta = 0.01f;
    float t0 = 0.0f, t1 = 0.0f;
    if (alive) {
        const float e[3] = {eye[3 * i], eye[3 * i + 1], eye[3 * i + 2]};
        const float d[3] = {dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
        R = worldToIndexRay(g, e, d);
        alive = rayClip(R, g.bbox) && !(double(R.t1) > 1e20);
        t0 = R.t0 + Eps;
        t1 = R.t1 - Eps;
        alive = alive && !(t0 > t1);
        Ltot = Lfwd[i];
        tTerm = gTin ? gT * sdt * Tfwd[i] : 0.0f; // Tfwd may be NULL when no dL/dT is given
    }
    float L = 0.0f, T = 1.0f;
    bool range = true; // every contribution converted without saturation
    // The window's eight voxels by the parity of their coordinates (slot p: x, y, z odd in bits 2, 1,
    // 0): a voxel keeps its slot for as long as it stays in the window, so nothing moves between
    // registers when the cell does; p is also the voxel's word in its 2x2x2 block.
    float sum[8];
#pragma unroll
    for (int p = 0; p < 8; ++p) sum[p] = 0.0f;
    int32_t cx = 0, cy = 0, cz = 0; // the window's cell
    uint32_t step = 0, misses = 0; // the wavefront's
    // the misses, one per lane
    auto drain = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < misses) {
            const uint32_t at = C.missAt[lane], pos = at >> 3;
            blockAdd<GT>(M, g, blocks, accum, pos, blockDest<GT>(M, pos), at & 7u, C.missQ[lane]);
        }
        misses = 0;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    // Sums of the voxels `leave` (every lane of the wavefront calls this; leave = 0: none) go to their
    // blocks' entries.  A block without an entry claims it if it is free, else the sum waits in
    // the misses.
    auto flush = [&](uint32_t leave) {
        const uint32_t rx = uint32_t(cx - M.lo[0] * 8), ry = uint32_t(cy - M.lo[1] * 8), rz = uint32_t(cz - M.lo[2] * 8);
        float q[8], most = 0.0f;
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            const bool go = (leave >> p) & 1u;
            q[p] = go ? sum[p] * scale : 0.0f;
            sum[p] = go ? 0.0f : sum[p];
            most = fmaxf(most, fabsf(q[p])); // of a NaN and a number, the number: NaN is tested below
        }
        const bool in = rx + 1u < M.n[0] * 8u && ry + 1u < M.n[1] * 8u && rz + 1u < M.n[2] * 8u;
        const float nan = (q[0] + q[1]) + (q[2] + q[3]) + (q[4] + q[5]) + (q[6] + q[7]);
        // outside the table, or beyond the exact range of the rounding below
        if (!in || !(most < 1125899906842624.0f) || nan != nan) {
            // unrolled by the compiler or not, rare
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                if (q[p] != 0.0f) {
                    const int32_t key = voxelKey<GT>(M, g, (p & 4) ? cx | 1 : (cx + 1) & ~1, (p & 2) ? cy | 1 : (cy + 1) & ~1,
                                                     (p & 1) ? cz | 1 : (cz + 1) & ~1);
                    const long long v = key >= 0 ? toFixed(q[p], range) : 0;
                    if (v != 0) atomicAdd(accum + key, static_cast<unsigned long long>(v));
                }
                q[p] = 0.0f;
            }
        }
        // block coordinates of the odd voxel per axis; the even one's is the next where the cell starts
        // at an odd voxel
        const uint32_t bx = rx >> 1, by = ry >> 1, bz = rz >> 1, ox = rx & 1u, oy = ry & 1u, oz = rz & 1u;
        const uint32_t tag7 = bx * X.sx + by * X.sy + bz;
        const uint32_t ex = ox ? X.sx : 0u, ey = oy ? X.sy : 0u;
        const uint32_t bxe = bx + ox, bye = by + oy, bze = bz + oz;
        const uint32_t n2 = M.n[2] * 64u, n12 = M.n[1] * n2;
        const uint32_t px[2] = {(bxe >> 2) * n12 + (bxe & 3u) * 16u, (bx >> 2) * n12 + (bx & 3u) * 16u},
                       py[2] = {(bye >> 2) * n2 + (bye & 3u) * 4u, (by >> 2) * n2 + (by & 3u) * 4u},
                       pz[2] = {(bze >> 2) * 64u + (bze & 3u), (bz >> 2) * 64u + (bz & 3u)};
        uint32_t was[8];
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            const uint32_t tag = tag7 + (p & 4 ? 0u : ex) + (p & 2 ? 0u : ey) + (p & 1 ? 0u : oz);
            was[p] = kNoBlock - 1u;
            if (q[p] != 0.0f) was[p] = atomicCAS(&C.tag[tag & (kCacheBlocks - 1u)], kNoBlock, tag);
        }
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            const uint32_t tag = tag7 + (p & 4 ? 0u : ex) + (p & 2 ? 0u : ey) + (p & 1 ? 0u : oz);
            const uint32_t at = tag & (kCacheBlocks - 1u), pos = px[p >> 2] + py[(p >> 1) & 1] + pz[p & 1];
            // round to nearest even: the integer is the low bits of 1.5 * 2^52 + q (exact to 2^51)
            const unsigned long long v = static_cast<unsigned long long>(
                __double_as_longlong(double(q[p]) + 6755399441055744.0) - 0x4338000000000000ll);
            if (was[p] == kNoBlock) {
                C.born[at] = uint8_t(step);
                C.pos[at] = pos;
            }
            if (was[p] == kNoBlock || was[p] == tag) atomicAdd(&C.q[at * 8u + uint32_t(p)], v);
            const bool miss = q[p] != 0.0f && was[p] != kNoBlock && was[p] != tag;
            const uint64_t m = __ballot(miss);
            if (m) {
                if (misses + uint32_t(__popcll(m)) > kCacheMisses) drain();
                if (miss) {
                    const uint32_t k = misses + __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
                    C.missAt[k] = pos * 8u + uint32_t(p);
                    C.missQ[k] = v;
                }
                misses += uint32_t(__popcll(m));
            }
        }
    };
    // Blocks claimed `age` steps ago or earlier go to scratch, eight at a time: a block's eight words
    // leave in one instruction, as one request.
    auto evict = [&](uint32_t age) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint32_t n = 0;
#pragma unroll
        for (uint32_t r = 0; r < kCacheBlocks / 64u; ++r) {
            const uint32_t k = r * 64u + lane;
            const bool old = C.tag[k] != kNoBlock && ((step - C.born[k]) & 255u) >= age;
            const uint64_t m = __ballot(old);
            if (old) {
                C.list[n + __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u))] = uint8_t(k);
                C.tag[k] = blockDest<GT>(M, C.pos[k]); // until the entry is free below
            }
            n += uint32_t(__popcll(m));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (uint32_t k = lane >> 3; k < n; k += 8u) {
            const uint32_t at = C.list[k], w = lane & 7u, dest = C.tag[at];
            const unsigned long long q = C.q[at * 8u + w];
            if (!(dest & kDestTile)) {
                if (q != 0) atomicAdd(blocks + (uint64_t(dest) * 8u + w), q);
            } else if (q != 0) {
                blockAdd<GT>(M, g, blocks, accum, C.pos[at], dest, w, q);
            }
            C.q[at * 8u + w] = 0ull;
            if (w == 0) C.tag[at] = kNoBlock;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    // getDim and state of the slot at the marching position
    auto cellAt = [&](float p0, float p1, float p2, SlotCell& c) {
        const int32_t x = ifloor(p0), y = ifloor(p1), z = ifloor(p2);
        if (slotCell(M, x, y, z, c)) return;
        // a slot the map leaves open: its tree state as a tile, the steps take the tree too
        Accessor<GT> acc(g);
        const Probe pr = acc.probe(x, y, z);
        c.ox = x & ~7;
        c.oy = y & ~7;
        c.oz = z & ~7;
        c.dim = int32_t(pr.dim);
        c.entry = kSlotTile | (pr.active || pr.dim == 1u ? kSlotTileOn : 0u);
    };
    SlotCell c;
    HDDA h;
    float kf = 0.0f, t = 0.0f, tb = 0.0f, lag = -1.0f; // lag: the wavefront's
    bool pend = false, more = true, first = true;
    if (alive) {
        float p[3];
        rayAt(R, t0, p);
        cellAt(p[0], p[1], p[2], c);
        h.init(R, t0, t1, c.dim > 8 ? c.dim : 8);
    }
    for (;;) {
        // on to the next cell that holds a step
        while (alive && !pend) {
            if (!first) {
                if (!more) {
                    alive = false;
                    break;
                }
                float p[3];
                rayAt(R, h.t0 + Delta, p);
                cellAt(p[0], p[1], p[2], c);
                h.update(R, c.dim > 8 ? c.dim : 8);
            }
            first = false;
            const float ta = h.t0;
            more = h.stepOnce();
            tb = fminf(h.t0, t1);
            if ((!(c.entry & kSlotTile) || (c.entry & kSlotTileOn)) && ta < tb) {
                kf = ceilf(ta / dt);
                t = kf * dt;
                pend = t < tb;
            }
        }
        if (!__any(pend)) break;
        // rays stay within a few steps of the last one, so that the wavefront's blocks stay few
        const float kmin = waveMinDpp(pend ? kf : kFltMax);
        if (lag < 0.0f) // every ray with a step at all stands before its first
            lag = s.width || -waveMinDpp(pend ? -kf : kFltMax) - kmin <= kCacheSpread ? kCacheLag : kFltMax;
#pragma unroll 1
        for (uint32_t sub = 0; sub < kCacheSteps; ++sub) {
            const bool act = pend && (kf < kmin + lag || kf == kmin);
            const float x0 = __builtin_fmaf(t, R.dir[0], R.eye[0]), x1 = __builtin_fmaf(t, R.dir[1], R.eye[1]),
                        x2 = __builtin_fmaf(t, R.dir[2], R.eye[2]);
            const float fx = floorf(x0), fy = floorf(x1), fz = floorf(x2);
            const int32_t ni = int32_t(fx), nj = int32_t(fy), nk = int32_t(fz);
            const uint32_t rx = uint32_t(ni - c.ox), ry = uint32_t(nj - c.oy), rz = uint32_t(nk - c.oz);
            const bool fast = act && !(c.entry & kSlotTile) && (rx | ry | rz) < 8u;
            Cell cell;
            brickCell(M, fast ? c.entry * kBrickFloats + (rx * 9u + ry) * 9u + rz : 0u, cell);
            // voxels that leave the window: those of the trailing layer on each axis the cell moved along by
            // one (its parity is the old cell's, or the other when moving down)
            const int32_t dx = ni - cx, dy = nj - cy, dz = nk - cz;
            uint32_t leave = 0xffu;
            if (!(uint32_t(dx + 1) > 2u || uint32_t(dy + 1) > 2u || uint32_t(dz + 1) > 2u)) {
                const uint32_t mx = dx == 0 ? 0u : (((cx ^ (dx >> 1)) & 1) ? 0xf0u : 0x0fu);
                const uint32_t my = dy == 0 ? 0u : (((cy ^ (dy >> 1)) & 1) ? 0xccu : 0x33u);
                const uint32_t mz = dz == 0 ? 0u : (((cz ^ (dz >> 1)) & 1) ? 0xaau : 0x55u);
                leave = mx | my | mz;
            }
            if (!act) leave = 0u;
            if (__any(leave != 0u)) flush(leave);
            if (act) {
                const float u = x0 - fx, v = x1 - fy, w = x2 - fz;
                float rho = trilerp(cell, u, v, w);
                if (!fast && !slotTrilinear(M, x0, x1, x2, rho)) rho = treeTrilinear<GT>(g, x0, x1, x2);
                cx = ni;
                cy = nj;
                cz = nk;
                const float a = stepAbsorption(sigma, rho, dt);
                L += T * (1.0f - a) * rho;        // same operations as the forward march
                const float rest = Ltot - L;      // radiance of the later steps
                const float gk = gL * (T * ((1.0f - a) + rho * sdt * a) - sdt * rest) - tTerm;
                T *= a;
                // corner (a,b,c) receives gk * wx[a] * wy[b] * wz[c], factored as (gk wx wy) wz and fused
                // into the running sum; the weights go by parity as the sums do
                const bool ox = ni & 1, oy = nj & 1, oz = nk & 1;
                const float wx[2] = {ox ? u : 1.0f - u, ox ? 1.0f - u : u};
                const float wy[2] = {oy ? v : 1.0f - v, oy ? 1.0f - v : v};
                const float wz[2] = {oz ? w : 1.0f - w, oz ? 1.0f - w : w};
                const float gx[2] = {gk * wx[0], gk * wx[1]};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float gxy = gx[q >> 1] * wy[q & 1];
                    sum[2 * q] = fmaf(gxy, wz[0], sum[2 * q]);
                    sum[2 * q + 1] = fmaf(gxy, wz[1], sum[2 * q + 1]);
                }
                const float kn = kf + 1.0f;
                pend = kn != kf; // beyond 2^24 steps: the float counter cannot advance
                kf = kn;
                t = kf * dt;
                pend = pend && t < tb;
            }
            ++step;
        }
        evict(kCacheAge);
    }
    flush(0xffu);
    drain();
    evict(0u);
    if (!range) atomicOr(overflow, 1u);
}

__global__ __launch_bounds__(kBlock) void k_zero_blocks(ulonglong2* __restrict__ p, uint64_t n)
{
    const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i < n) p[i] = make_ulonglong2(0ull, 0ull);
}

// The blocks' sums into the accumulator: one wavefront per leaf, eight rows of eight voxels at a
// time (the accumulator's order), each row one request.
template<uint32_t GT>
__global__ __launch_bounds__(kBlock) void k_fold_blocks(GridView g, const unsigned long long* __restrict__ blocks,
                                                        unsigned long long* __restrict__ accum)
{
    const uint32_t lane = threadIdx.x & 63u, leaf = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    if (leaf >= g.leafCount) return;
    unsigned long long zero = 0ull; // index grids: the leaf's inactive voxels all read index 0
#pragma unroll
    for (uint32_t r = 0; r < 8; ++r) {
        const uint32_t n = r * 64u + lane, x = n >> 6, y = (n >> 3) & 7u, z = n & 7u;
        const uint32_t block = ((x >> 1) << 4) | ((y >> 1) << 2) | (z >> 1), w = ((x & 1u) << 2) | ((y & 1u) << 1) | (z & 1u);
        const unsigned long long q = blocks[(uint64_t(leaf) * 64u + block) * 8u + w];
        if (q == 0) continue;
        if constexpr (GT == GT_ONINDEX) {
            const uint64_t at = Codec<GT_ONINDEX>::index(g.leaf0 + uint64_t(leaf) * g.leafSize, n);
            if (at) atomicAdd(accum + at, q);
            else zero += q;
        } else {
            atomicAdd(accum + uint64_t(leaf) * 512u + n, q);
        }
    }
    if constexpr (GT == GT_ONINDEX) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) zero += __shfl_xor(zero, d);
        if (lane == 0 && zero) atomicAdd(accum, zero);
    }
}

__global__ __launch_bounds__(kBlock) void k_fixed_to_float(const long long* __restrict__ in, uint64_t n, double inv,
                                                           float* __restrict__ out)
{
    const uint64_t stride = uint64_t(gridDim.x) * kBlock;
    for (uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride) out[i] = float(double(in[i]) * inv);
}

} // namespace

int fogMarchBackward(const GridView& g, const float* eye, const float* dir, uint64_t n, uint32_t width, float dt,
                     float sigma, const float* L, const float* T, const float* gL, const float* gT, int64_t* accum,
                     int shift, hipStream_t s)
{
    const Sched sc = makeSched(n, width);
    const float scale = ldexpf(1.0f, shift);
    TileOrder to;
    SlotMap M;
    // The tiled adjoint wherever the grid has a slot map and its blocks (4 KB per leaf) stay within 4 GiB:
    // it was the faster one from 1024 rays on, as an image, a scattered batch or one shuffled over cameras (1024
    // rays through a 256^3 fog: accessor 7.1 ms, blocks 2.9; 1 M scattered rays from four distances 47.8 and 19.3).
    // Not for fewer than four rays, whose march does not make up for the map, the clearing and the folding of
    // 4 KB per leaf: 1, 2, 4 and 8 rays through a 512^3 fog 0.70, 1.38, 2.45 and 3.86 ms through the
    // accessor, 1.17, 1.56, 2.05 and 2.42 with blocks.
    // Decided before any of it is allocated or built.
    BlockBox X{};
    const bool tiled = n >= 4 && g.leafCount && g.leafCount <= kMaxBlockLeaves && sc.tiles < (1u << 26) && blockBoxOf(slotBoxOf(g.bbox), X);
    const uint64_t blockBytes = tiled ? uint64_t(g.leafCount) * 4096u : 0;
    if (tileOrder(g, eye, dir, sc, to, s, 256, tiled ? &M : nullptr, blockBytes) != 0) return -1;
    uint32_t* flag = reinterpret_cast<uint32_t*>(to.extra);
    hipLaunchKernelGGL(k_clear_flag, dim3(1), dim3(1), 0, s, flag);
    unsigned long long* acc = reinterpret_cast<unsigned long long*>(accum);
    const bool index = g.type == GT_ONINDEX;
    if (to.map) {
        unsigned long long* blocks = reinterpret_cast<unsigned long long*>(to.withMap);
        const uint64_t words = blockBytes / 16;
        hipLaunchKernelGGL(k_zero_blocks, dim3(uint32_t((words + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                           reinterpret_cast<ulonglong2*>(blocks), words);
        {
            ProfScope prof("k_fog_march_bwd", s);
            auto march = index ? k_fog_march_bwd_blocks<GT_ONINDEX> : k_fog_march_bwd_blocks<GT_FLOAT>;
            hipLaunchKernelGGL(march, dim3(uint32_t(sc.tiles)), dim3(64), 0, s, M, X, g, eye, dir, sc, to.order, dt,
                               sigma, L, T, gL, gT, blocks, acc, scale, flag);
        }
        auto fold = index ? k_fold_blocks<GT_ONINDEX> : k_fold_blocks<GT_FLOAT>;
        hipLaunchKernelGGL(fold, dim3((g.leafCount + kBlock / 64 - 1) / (kBlock / 64)), dim3(kBlock), 0, s, g, blocks, acc);
    } else {
        ProfScope prof("k_fog_march_bwd", s);
        auto march = index ? k_fog_march_bwd<GT_ONINDEX> : k_fog_march_bwd<GT_FLOAT>;
        hipLaunchKernelGGL(march, dim3(orderedBlocks(sc)), dim3(kBlock), 0, s, g, eye, dir, sc, to.order, dt, sigma, L, T,
                           gL, gT, acc, scale, flag);
    }
    bool ok = hipGetLastError() == hipSuccess;
    const void* st = stageCopy(flag, sizeof(uint32_t), s);
    ok = st && ok;
    ok = hipStreamSynchronize(s) == hipSuccess && ok;
    if (!ok) return -1;
    uint32_t over = 0;
    std::memcpy(&over, st, sizeof(over));
    return over ? -2 : 0;
}

int fixedToFloat(const int64_t* accum, uint64_t count, int shift, float* out, hipStream_t s)
{
    const uint64_t b = (count + kBlock - 1) / kBlock;
    const uint32_t blocks = uint32_t(b < 1 ? 1 : (b > (1u << 20) ? (1u << 20) : b));
    hipLaunchKernelGGL(k_fixed_to_float, dim3(blocks), dim3(kBlock), 0, s, reinterpret_cast<const long long*>(accum),
                       count, ldexp(1.0, -shift), out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

} // namespace nvq
