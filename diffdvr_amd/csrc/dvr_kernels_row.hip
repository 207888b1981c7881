// Row kernels (16 lanes a ray, dvr_row_impl.hpp): launchers.
#include "dvr_row_impl.hpp"

namespace dvr {

// At most 2^20 tiles of 1024 threads: a launch holds less than 2^32 threads.
constexpr int kMaxRowTiles = 1 << 20;

// voxel edges per step and voxel edges per pixel, both averaged over the axes;
// a per-ray step or a box in device memory counts as the usual half voxel / unit box
float step_voxels(const RenderParams& P)
{
    if (P.st || P.bsize) return 0.5f;
    const float n[3] = {float(P.X - 1), float(P.Y - 1), float(P.Z - 1)};
    float v = 0.0f;
    for (int a = 0; a < 3; ++a) v += P.stU * n[a] / (3.0f * P.bsizeU[a]);
    return v;
}
float pixel_voxels(const RenderParams& P)
{
    return float(P.X + P.Y + P.Z) / (3.0f * float(P.W < P.H ? P.W : P.H));
}

// Few rays leave the tiled kernel's chain of samples exposed: up to 768 tiles the row kernel wins at
// every size measured, up to 1024 and 2048 but for small volumes seen closely (row against tiled, us:
// 1024 tiles 43 / 67 through 64^3, 122 / 275 through 256^3; 2048 tiles 114 / 191 through 128^3, 54 /
// 46 through 32^3).  Beyond, it pays by what the gathers touch: 64 neighbouring rays reach further
// apart than 16 consecutive samples where g = (voxels per pixel) x (voxels per step) is large, and
// more so where the volume exceeds the 4 MiB L2s.  Below 0.3 voxels per pixel the tiled kernel's
// twenty workgroups a CU win: 4096 tiles 200 / 189, 8192 tiles 598 / 538.  Others: g = 0.5, 256^3, 8192
// tiles 507 / 1387, 16384 tiles 988 / 2149; g = 0.375, 192^3, 362 / 665, 96^3, 16384 tiles 451 / 430;
// g = 0.25, 256^3, 8192 tiles 728 / 878, 16384 tiles 890 / 920, 32768 tiles 1742 / 1617, 128^3, 4096
// tiles 151 / 186, 16384 tiles 514 / 480; quarter-voxel steps, 0.5 voxels per pixel, 128^3, 8192 tiles
// 388 / 451, 16384 tiles 774 / 691, 256^3, 16384 tiles 1450 / 1494.  A nearest-neighbour sample gathers
// one voxel, not eight, and gains up to 768 tiles.
bool use_row_forward(const RenderParams& P, int filter)
{
    const int tiles = tiled_num_tiles(P);
    if (tiles <= 768) return true;
    if (filter != 1 || tiles > kMaxRowTiles) return false;
    const float step = step_voxels(P), pixel = pixel_voxels(P), g = step * pixel;
    const size_t voxels = size_t(P.X) * P.Y * P.Z;
    if (g >= 0.3f) return tiles <= 8192 || voxels >= (size_t(2) << 20);
    if (pixel <= 0.3f) return tiles <= (pixel <= 0.15f ? 1024 : 2048);
    const bool large = voxels >= 4000000;
    if (step < 0.4f) return tiles <= (large ? 16384 : 8192);
    return tiles <= (large && g >= 0.24f ? 16384 : 4096);
}

// Position gradients alone (row_reverse): the row kernel gains with the samples of a ray, which the tiled
// kernel walks one after the other, with their distance (its gathers then meet in fewer lines than 64 rays')
// and with the cost of a sample's shading, which it does once; it loses with the tiles, which fill the chip
// without it.  Up to 1024 tiles always, then up to c x (samples per axis) x sqrt(voxels per pixel): over 570
// launches of 1024 to 32768 tiles this is 0.3 % off the better kernel on average, 19 % at most.  Row / tiled,
// us: identity TF, 128^3, 4096 tiles 210 / 243 at 0.5 voxels a pixel, 296 / 251 at 0.25, 64^3, 16384 tiles 534 / 257;
// linear 418 / 494 and 652 / 748 at 128^3, 8192 tiles, 578 / 435 at 64^3, 16384; Gaussian of four rows 968 / 1358
// at 128^3, 16384, 513 / 371 at 32^3.
// Volume gradients (split_reverse) in two passes: 185 / 262 and 273 / 277 us at 1024 tiles, 415 / 350 at
// 2048; in one pass 634 / 1038 at 2048, 2707 / 2684 at 4096.  TF gradients: 137 / 160 us at 1024
// tiles, 238 / 184 at 2048; the identity TF's walk is short, 53 / 65 at 576 and 83 / 67 at 1024, but beside the
// forward march of a fused launch the row kernel pays up to 1024 (90 / 91 at 64^3, 224 / 346 at 256^3).
// The loss and TF gradients are summed in doubles: the row kernel adds four times a tile, and 4096 or more
// floats added to one scalar in any order are off by 1e-6 of it and more.  Without memory for these sums the
// tiled kernel runs.
bool use_row_adjoint(const RenderParams& P, const AdjointParams& A, const CkptParams& CK, const LossParams& L, int tfm)
{
    const int tiles = tiled_num_tiles(P);
    if (tiles > kMaxRowTiles || (L.lossOut && !L.lossSum) || (A.atf && !A.atfSum)) return false;
    if (A.avol) return tiles <= (CK.as.adj ? 1024 : 2048);
    if (A.atf) return tiles <= (tfm == 0 && !A.ars && !A.ast && !L.target ? 768 : 1024);
    const float samples = float(P.X + P.Y + P.Z) / (3.0f * step_voxels(P));
    const float c = tfm == 3 ? 266.0f : (tfm == 2 ? 94.0f : 33.0f);
    return tiles <= 1024 || float(tiles) <= c * samples * sqrtf(pixel_voxels(P));
}

template <int FILTER, int TFM, int BLEND>
static hipError_t fwd_row_t(const RenderParams& P, const CkptParams& CK, hipStream_t s)
{
    const int tilesX = (P.W + kTileW - 1) / kTileW, tilesY = (P.H + kTileH - 1) / kTileH;
    const int nTiles = tilesX * tilesY * P.B;
    if (nTiles == 0) return hipSuccess;
    const size_t lds = sizeof(float) * size_t(P.R) * tf_lds_stride<TFM>();
    hipLaunchKernelGGL((k_forward_row<FILTER, TFM, BLEND>), dim3(nTiles * row_blocks_per_tile(kRowBlock)),
                       dim3(kRowBlock), lds, s, P, CK, tilesX, tilesX * tilesY, nTiles);
    return hipGetLastError();
}

hipError_t launch_forward_row(const RenderParams& P, const CkptParams& CK, int filter, int tfm, int blend, hipStream_t s)
{
    DVR_DISPATCH3(filter, tfm, blend, return fwd_row_t, (P, CK, s));
    return hipErrorInvalidValue;
}

template <int FILTER, int TFM, int BLEND, int GM>
static hipError_t adj_row_g(const RenderParams& P, const AdjointParams& A, const CkptParams& CK, const LossParams& L,
                            bool fused, bool ckFromFwd, hipStream_t s)
{
    const int tilesX = (P.W + kTileW - 1) / kTileW, tilesY = (P.H + kTileH - 1) / kTileH;
    const int nTiles = tilesX * tilesY * P.B;
    if (nTiles == 0) return hipSuccess;
    const int RC = P.R * P.C;
    constexpr int kThreads = kRowAdjBlock;
    const bool usePriv = TFM == 3 && A.atf && RC <= 48;  // private slices <= 48 KiB of LDS
    const int copyStride = tf_grad_copy_stride(RC);
    const int ng = A.atf ? tf_grad_floats(RC, usePriv, kThreads, copyStride) : 0;
    int aggLog2 = kAggLog2;
    const int tfFloats = tf_grad_offset(P.R * tf_lds_stride<TFM>());
    size_t lds = sizeof(float) * size_t(tfFloats + ng);
    if ((GM & 2) && A.avol) {
        // the largest chunk table per wave beside the TF tables that leaves room for sixteen waves per CU
        const size_t base = sizeof(float) * size_t(agg_offset(tfFloats, ng));
        constexpr size_t kWaves = kThreads / 64;
        while (aggLog2 > kAggMinLog2 && base + kWaves * agg_bytes(aggLog2, sizeof(float)) > size_t(kLdsPerCu) * kWaves / kTiledVolWgPerCu)
            --aggLog2;
        lds = base + kWaves * agg_bytes(aggLog2, sizeof(float));
    }
    hipLaunchKernelGGL((k_adjoint_row<FILTER, TFM, BLEND, GM>), dim3(nTiles * row_blocks_per_tile(kThreads)),
                       dim3(kThreads), lds, s, P, A, CK, L, fused ? 1 : 0, ckFromFwd ? 1 : 0, usePriv ? 1 : 0, copyStride,
                       tilesX, tilesX * tilesY, nTiles, aggLog2);
    return hipGetLastError();
}

template <int FILTER, int TFM, int BLEND>
static hipError_t adj_row_t(const RenderParams& P, const AdjointParams& A, const CkptParams& CK, const LossParams& L,
                            bool fused, bool ckFromFwd, hipStream_t s)
{
    const bool pos = A.ars || A.ast;
    if (A.avol && CK.as.adj) {  // volume gradients in two passes
        if (pos) return adj_row_g<FILTER, TFM, BLEND, 13>(P, A, CK, L, fused, ckFromFwd, s);
        return adj_row_g<FILTER, TFM, BLEND, 9>(P, A, CK, L, fused, ckFromFwd, s);
    }
    if (pos && A.avol) return adj_row_g<FILTER, TFM, BLEND, 7>(P, A, CK, L, fused, ckFromFwd, s);
    if (pos && A.atf) return adj_row_g<FILTER, TFM, BLEND, 5>(P, A, CK, L, fused, ckFromFwd, s);
    if (pos) return adj_row_g<FILTER, TFM, BLEND, 4>(P, A, CK, L, fused, ckFromFwd, s);
    if (A.avol) return adj_row_g<FILTER, TFM, BLEND, 3>(P, A, CK, L, fused, ckFromFwd, s);
    return adj_row_g<FILTER, TFM, BLEND, 1>(P, A, CK, L, fused, ckFromFwd, s);
}

hipError_t launch_adjoint_row(const RenderParams& P, const AdjointParams& A, const CkptParams& CK, const LossParams& L,
                              bool fused, bool ckFromFwd, int filter, int tfm, int blend, hipStream_t s)
{
    DVR_DISPATCH3(filter, tfm, blend, return adj_row_t, (P, A, CK, L, fused, ckFromFwd, s));
    return hipErrorInvalidValue;
}

}  // namespace dvr
