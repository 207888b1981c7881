// Second pass of the volume gradients (the first, in the reverse walks, stores
// every sample's density adjoint and the rays): the eight corner gradients of
// every sample (renderer/renderer_interpolation.cuh:299-389) are added into a
// bricked scratch, which k_debrick adds into the caller's gradient.
//
// A device-memory float atomic costs one 64-byte request whether one lane or
// sixteen lanes of an instruction address that chunk, so corner gradients are
// first summed per 64-byte brick (2x2x4 voxels) in an LDS table.  The walks of
// the first pass keep one ray a lane and have few registers and little LDS to
// spare: a table of 64 or 128 slots a wave, too small for the >100 bricks that 64
// rays two voxels apart touch with one sample.  Here nothing else lives beside the
// table: eight waves share 512 slots, a tile of 64 rays and a slab of samples, so
// the neighbouring samples of a brick meet in the table while it is there, and it
// is emptied with whole 16-lane groups.
// Bound by the LDS pipe (64 % busy on 8 x 256 x 256 rays through 256^3) and the
// issue of the table look-ups beside it.  The slab is 8 to 32 samples: rays 3.5 voxels
// apart overran the table at 32 (14.7 ms, 5.3 ms with 8 to 16).  The sums are
// doubles: ds_add_f32 is served one lane after another.  256^3, 8 x 256 x 256 rays
// (66 M samples): 3430 us with float sums, 1310 us with doubles; 256 threads and
// slots 2130 us, 1024 threads and slots 1650 us.
#include "dvr_tiled_impl.hpp"

namespace dvr {

constexpr int kScatterBlock = 512;
constexpr int kWaves = kScatterBlock / 64;
constexpr int kSlots = 512;          // 66 KiB: two workgroups (sixteen waves) a CU
constexpr int kBuckets = kSlots / 4;
constexpr int kSlab = 32;            // most samples between two looks at the table's load
constexpr unsigned kFree = 0xFFFFFFFFu;

struct ScatterTable {
    unsigned tags[kSlots];           // brick number, kFree = none; four slots are a bucket
    double vals[kSlots * 16];
    unsigned taken[4];
};

struct ScatterVolume {
    int X, Y, Z;
    unsigned BY, BZ;
    float* brick;
};

// Buckets run along z and step by odd numbers in y and x, so that a compact group of bricks spreads
// evenly over them.
__device__ __forceinline__ unsigned scatter_bucket(unsigned bx, unsigned by, unsigned bz)
{
    return (bz + by * 11u + bx * 45u) & unsigned(kBuckets - 1);
}

// Slot of brick q in bucket b, claimed if need be; kFree when its four slots hold other bricks.
__device__ __forceinline__ unsigned scatter_match(const uint4& t, unsigned q, unsigned b)
{
    unsigned s = kFree;
    s = t.x == q ? 4u * b : s;
    s = t.y == q ? 4u * b + 1u : s;
    s = t.z == q ? 4u * b + 2u : s;
    s = t.w == q ? 4u * b + 3u : s;
    return s;
}
template <int TRY>
__device__ __forceinline__ void scatter_claim(ScatterTable& L, uint4& t, unsigned q, unsigned b, unsigned& s)
{
    if constexpr (TRY < 4) {
        if (s == kFree) {
            const unsigned w = t.x == kFree ? 0u : (t.y == kFree ? 1u : (t.z == kFree ? 2u : (t.w == kFree ? 3u : 4u)));
            if (w < 4u) {
                const unsigned old = atomicCAS(&L.tags[4u * b + w], kFree, q);
                if (old == kFree || old == q) s = 4u * b + w;
                t.x = w == 0u ? old : t.x;
                t.y = w == 1u ? old : t.y;
                t.z = w == 2u ? old : t.z;
                t.w = w == 3u ? old : t.w;
                scatter_claim<TRY + 1>(L, t, q, b, s);
            }
        }
    }
}
// slot of brick q: in its bucket, else in the bucket half the table away, else kFree
__device__ __forceinline__ unsigned scatter_slot(ScatterTable& L, unsigned q, unsigned b)
{
    uint4 t = *reinterpret_cast<const uint4*>(&L.tags[4u * b]);
    unsigned s = scatter_match(t, q, b);
    scatter_claim<0>(L, t, q, b, s);
    if (s == kFree) {
        const unsigned b2 = b ^ unsigned(kBuckets / 2);
        t = *reinterpret_cast<const uint4*>(&L.tags[4u * b2]);
        s = scatter_match(t, q, b2);
        scatter_claim<0>(L, t, q, b2, s);
    }
    return s;
}

// adds v at position pos of brick q, which has slot s (kFree: straight to device memory)
__device__ __forceinline__ void scatter_add(ScatterTable& L, const ScatterVolume& V, unsigned s, unsigned q, unsigned pos,
                                            float v)
{
    if (s != kFree) atomicAdd(&L.vals[s * 16u + pos], double(v));
    else gatomic_add(V.brick, q * 16u + pos, v);
}

// corner pair (x, y, z0), (x, y, z1)
__device__ __forceinline__ void scatter_pair(ScatterTable& L, const ScatterVolume& V, int x, int y, int z0, int z1,
                                             float v0, float v1)
{
    const unsigned bx = unsigned(x) >> 1, by = unsigned(y) >> 1, bz0 = unsigned(z0) >> 2, bz1 = unsigned(z1) >> 2;
    const unsigned row = (bx * V.BY + by) * V.BZ, pos = (unsigned(x & 1) << 3) | (unsigned(y & 1) << 2);
    const unsigned q0 = row + bz0;
    const unsigned s0 = scatter_slot(L, q0, scatter_bucket(bx, by, bz0));
    scatter_add(L, V, s0, q0, pos | unsigned(z0 & 3), v0);
    if (bz1 == bz0) {
        scatter_add(L, V, s0, q0, pos | unsigned(z1 & 3), v1);
    } else {
        const unsigned q1 = row + bz1;
        const unsigned s1 = scatter_slot(L, q1, scatter_bucket(bx, by, bz1));
        scatter_add(L, V, s1, q1, pos | unsigned(z1 & 3), v1);
    }
}

// adds the table into the scratch, a 16-lane group a slot; every thread of the workgroup, between barriers
__device__ __forceinline__ void scatter_flush(ScatterTable& L, const ScatterVolume& V)
{
    const unsigned j = threadIdx.x & 15u;
    for (unsigned s = threadIdx.x >> 4; s < unsigned(kSlots); s += kScatterBlock / 16) {
        const unsigned q = L.tags[s];
        if (q == kFree) continue;
        const double v = L.vals[s * 16u + j];
        if (v != 0.0) {
            gatomic_add(V.brick, q * 16u + j, float(v));
            L.vals[s * 16u + j] = 0.0;
        }
    }
}

template <int FILTER>
__global__ __launch_bounds__(kScatterBlock) void k_scatter_volume(ScatterParams P)
{
    __shared__ __attribute__((aligned(16))) ScatterTable L;
    const int blk = xcd_remap(blockIdx.x, P.nTiles * P.parts);
    const int tile = blk / P.parts, part = blk - tile * P.parts;
    ScatterVolume V;
    if (P.views) {
        int lo = 0, hi = P.nViews - 1;
        while (lo < hi) {  // the last view whose first tile is <= tile
            const int mid = (lo + hi + 1) >> 1;
            if (P.views[mid].tileBegin <= P.tile0 + tile) lo = mid;
            else hi = mid - 1;
        }
        const BVol vol = P.vols[P.views[lo].vol];
        if (vol.adj == nullptr) return;  // uniform: no gradient of this volume
        V.X = vol.X; V.Y = vol.Y; V.Z = vol.Z;
        V.brick = vol.brick;
    } else {
        V.X = P.X; V.Y = P.Y; V.Z = P.Z;
        V.brick = P.brick + size_t((P.tile0 + tile) / P.tilesPerVolume + int(blockIdx.y)) * P.brickFloats;
    }
    V.BY = unsigned(V.Y + 1) >> 1;
    V.BZ = unsigned(V.Z + 3) >> 2;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // eight rays of the tile a wave, each in the eight lanes of every eighth of the slab
    const int ray = wave * 8 + (lane & 7), eighth = lane >> 3;
    const float* rec = P.S.rays + size_t(tile) * (kRayRecord * kBlock);
    const int nMax = wave_max(min(__float_as_int(rec[8 * kBlock + lane]), P.S.cap));
    rec += ray;
    const int n = min(__float_as_int(rec[8 * kBlock]), P.S.cap);
    // this workgroup's samples, a multiple of the slab length
    const int len = ((nMax + P.parts - 1) / P.parts + kSlab - 1) & ~(kSlab - 1);
    const int begin = part * len, end = min(nMax, begin + len);
    if (begin >= end) return;  // uniform
    const int last = min(n, end);
    const f3 p0 = mk3(rec[0], rec[kBlock], rec[2 * kBlock]);
    const f3 dp = mk3(rec[3 * kBlock], rec[4 * kBlock], rec[5 * kBlock]);
    const float t0 = rec[6 * kBlock], step = rec[7 * kBlock];
    const float* adj = P.S.adj + blockIdx.y * P.adjPlane + size_t(tile) * (size_t(P.S.cap + kAdjSpill) * kBlock) + ray;

    for (int e = threadIdx.x; e < kSlots; e += kScatterBlock) L.tags[e] = kFree;
    for (int e = threadIdx.x; e < kSlots * 16; e += kScatterBlock) L.vals[e] = 0.0;
    if (threadIdx.x < 4) L.taken[threadIdx.x] = 0u;
    __syncthreads();

    unsigned round = 0;
    int slab = 16;
    for (int i0 = begin; i0 < end;) {
        const int per = slab / 8, first = i0 + eighth * per;
        float a[kSlab / kWaves];
#pragma unroll
        for (int m = 0; m < kSlab / kWaves; ++m) {
            const int i = first + m;
            a[m] = m < per && i < last ? *(const gfloat*)(adj + size_t(i) * kBlock) : 0.0f;
        }
#pragma unroll
        for (int m = 0; m < kSlab / kWaves; ++m) {
            const float v = a[m];
            if (v == 0.0f) continue;
            const float t = t0 + float(first + m) * step;
            const f3 p = mk3(fmaf(t, dp.x, p0.x), fmaf(t, dp.y, p0.y), fmaf(t, dp.z, p0.z));
            if constexpr (FILTER == 0) {
                int x, y, z;
                nearest_index(p, V.X, V.Y, V.Z, x, y, z);
                const unsigned bx = unsigned(x) >> 1, by = unsigned(y) >> 1, bz = unsigned(z) >> 2;
                const unsigned q = (bx * V.BY + by) * V.BZ + bz;
                scatter_add(L, V, scatter_slot(L, q, scatter_bucket(bx, by, bz)), q,
                            (unsigned(x & 1) << 3) | (unsigned(y & 1) << 2) | unsigned(z & 3), v);
            } else {
                const int ix = int(p.x), iy = int(p.y), iz = int(p.z);
                float w[8];
                const float none[8] = {};
                f3 unused;
                tri_adjoint<false>(none, p.x - float(ix), p.y - float(iy), p.z - float(iz), v, w, unused);
                int x0, x1, y0, y1, z0, z1;
                cell_axis(ix, V.X, x0, x1);
                cell_axis(iy, V.Y, y0, y1);
                cell_axis(iz, V.Z, z0, z1);
                scatter_pair(L, V, x0, y0, z0, z1, w[0], w[1]);
                scatter_pair(L, V, x0, y1, z0, z1, w[2], w[3]);
                scatter_pair(L, V, x1, y0, z0, z1, w[4], w[5]);
                scatter_pair(L, V, x1, y1, z0, z1, w[6], w[7]);
            }
        }
        i0 += slab;
        // empty the table when another slab might not fit
        __syncthreads();
        unsigned used = 0;
#pragma unroll
        for (int k = 0; k < kSlots / kScatterBlock; ++k)
            used += unsigned(__popcll(__ballot(L.tags[threadIdx.x + k * kScatterBlock] != kFree)));
        if (lane == 0 && used != 0u) atomicAdd(&L.taken[round & 3u], used);
        __syncthreads();
        const unsigned taken = L.taken[round & 3u];
        const bool flush = taken > unsigned(kSlots) * 7 / 16 || i0 >= end;
        // rays far apart fill the table with fewer samples, rays close together with more
        if (taken > unsigned(kSlots) * 3 / 4) slab = max(slab / 2, kWaves);
        else if (taken < unsigned(kSlots) / 2) slab = min(slab * 2, kSlab);
        if (threadIdx.x == 0) L.taken[(round + 2u) & 3u] = 0u;
        ++round;
        if (flush) {
            scatter_flush(L, V);
            __syncthreads();
            for (int e = threadIdx.x; e < kSlots; e += kScatterBlock) L.tags[e] = kFree;
            __syncthreads();
        }
    }
}

hipError_t launch_scatter_volume(const ScatterParams& P, int filter, hipStream_t s, int channels)
{
    if (P.nTiles <= 0) return hipSuccess;
    ScatterParams Q = P;
    // few tiles: several workgroups share a tile's samples
    Q.parts = 1;
    while (Q.parts < 16 && Q.nTiles * Q.parts < 2048) Q.parts *= 2;
    const dim3 grid(unsigned(Q.nTiles) * unsigned(Q.parts), unsigned(channels));
    if (filter == 0) hipLaunchKernelGGL(k_scatter_volume<0>, grid, dim3(kScatterBlock), 0, s, Q);
    else hipLaunchKernelGGL(k_scatter_volume<1>, grid, dim3(kScatterBlock), 0, s, Q);
    return hipGetLastError();
}

}  // namespace dvr
