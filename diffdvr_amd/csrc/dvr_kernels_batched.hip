// Dispatcher over the batched persistent kernel instance slices (kernels in
// dvr_batched_impl.hpp).
#include "dvr_launch.hpp"

namespace dvr {

#define DVR_DECL_INST(F, B, K)                                                                                  \
    hipError_t batched_inst_##F##_##B##_##K(const BatchParams&, int, int, int, size_t, hipStream_t, int*);
#define DVR_DECL_K(F, B) DVR_DECL_INST(F, B, 4) DVR_DECL_INST(F, B, 8) DVR_DECL_INST(F, B, 16) DVR_DECL_INST(F, B, 32)
DVR_DECL_K(0, 0)
DVR_DECL_K(0, 1)
DVR_DECL_K(1, 0)
DVR_DECL_K(1, 1)
#undef DVR_DECL_K
#undef DVR_DECL_INST

hipError_t launch_batched(const BatchParams& P, int filter, int tfm, int blend, int K, int gm, int grid, size_t lds,
                          hipStream_t s, int* occ)
{
    if (filter < 0 || filter > 1 || blend < 0 || blend > 1) return hipErrorInvalidValue;
    if (gm == 0) K = 16;  // the forward-only instances live in the K = 16 slices
#define DVR_CALL(F, B, KK) return batched_inst_##F##_##B##_##KK(P, tfm, gm, grid, lds, s, occ)
#define DVR_SEL_K(F, B)                      \
    switch (K) {                             \
    case 4: DVR_CALL(F, B, 4);               \
    case 8: DVR_CALL(F, B, 8);               \
    case 16: DVR_CALL(F, B, 16);             \
    case 32: DVR_CALL(F, B, 32);             \
    default: return hipErrorInvalidValue;    \
    }
    if (filter == 0 && blend == 0) { DVR_SEL_K(0, 0) }
    if (filter == 0 && blend == 1) { DVR_SEL_K(0, 1) }
    if (filter == 1 && blend == 0) { DVR_SEL_K(1, 0) }
    { DVR_SEL_K(1, 1) }
#undef DVR_SEL_K
#undef DVR_CALL
}

// Adds a volume's bricked gradient scratch (2 x 2 x 4 voxels per 64-byte chunk,
// bricks z-fastest) into the caller's X x Y x Z gradient: a thread per 2 x 2
// column of voxels, consecutive threads on consecutive z, so that a wave reads
// whole chunks and, with z innermost, adds to four contiguous rows.  Other
// streams may add to the same gradient at the same time (calls with their own
// scratch and plans are not ordered with each other): device atomics, of the
// voxels that have a gradient (256^3, every voxel touched: 8 us more than a read-modify-write in a
// call of 2.4 ms).
__device__ __forceinline__ void debrick(const DebrickSeg& S)
{
    // a volume of at most 2^30 voxels has fewer than 2^31 columns
    const unsigned Z = unsigned(S.Z), BY = unsigned(S.Y + 1) >> 1, BZ = (Z + 3) >> 2;
    const unsigned n = (unsigned(S.X + 1) >> 1) * BY * Z;
    for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
        const unsigned r = i / Z, z = i - r * Z, xb = r / BY, yb = r - xb * BY;
        const float* src = S.brick + size_t(r * BZ + (z >> 2)) * 16 + (z & 3);
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = src[4 * q];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int x = int(2 * xb) + (q >> 1), y = int(2 * yb) + (q & 1);
            if (v[q] != 0.0f && x < S.X && y < S.Y) atomicAdd(S.adj + x * S.sx + y * S.sy + int(z) * S.sz, v[q]);
        }
    }
}
// blockIdx.y = volume of a plan
__global__ __launch_bounds__(256) void k_debrick(const DebrickSeg* segs)
{
    const DebrickSeg S = segs[blockIdx.y];
    debrick(S);
}
// blockIdx.y = batch of one call's gradient
__global__ __launch_bounds__(256) void k_debrick_call(DebrickSeg S, long long brickFloats, long long sb)
{
    S.brick += blockIdx.y * brickFloats;
    S.adj += blockIdx.y * sb;
    debrick(S);
}

__global__ __launch_bounds__(256) void k_clear(float4* p, long long n)
{
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
        p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

hipError_t launch_clear(float* p, size_t n, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    const long long v = (long long)(n / 4);
    const long long bx = (v + 255) / 256;
    hipLaunchKernelGGL(k_clear, dim3(unsigned(bx < 4096 ? bx : 4096)), dim3(256), 0, s, reinterpret_cast<float4*>(p), v);
    return hipGetLastError();
}

hipError_t launch_debrick_call(const DebrickSeg& S, int batches, long long sb, hipStream_t s)
{
    const long long bf = (long long)brick_floats(S.X, S.Y, S.Z);
    const long long bx = (bf / 4 + 255) / 256;
    hipLaunchKernelGGL(k_debrick_call, dim3(unsigned(bx < 8192 ? bx : 8192), unsigned(batches)), dim3(256), 0, s, S, bf, sb);
    return hipGetLastError();
}

// blockIdx.y = segment
__global__ __launch_bounds__(256) void k_add_sums(const SumSeg* segs)
{
    const SumSeg S = segs[blockIdx.y];
    for (int i = blockIdx.x * 256 + threadIdx.x; i < S.n; i += gridDim.x * 256)
        atomicAdd(S.dst + i, float(S.sum[i]));  // tables may share a gradient
}
// the loss and the TF gradients of one call: batch, row and column strides of its tensor
__global__ __launch_bounds__(256) void k_add_call_sums(const double* lossSum, float* lossOut, const double* sum, float* dst,
                                                       int n, int RC, int C, int sb, int sr, int sc)
{
    if (lossSum && blockIdx.x == 0 && threadIdx.x < 64) {
        double v = threadIdx.x < kLossSlots ? lossSum[threadIdx.x * kLossStride] : 0.0;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
        if (threadIdx.x == 0) atomicAdd(lossOut, float(v));
    }
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int b = i / RC, e = i - b * RC, r = e / C, c = e - r * C;
    atomicAdd(dst + b * sb + r * sr + c * sc, float(sum[i]));  // an expanded gradient shares elements
}

hipError_t launch_add_sums(const SumSeg* dSegs, int nSegs, int maxN, hipStream_t s)
{
    if (nSegs == 0) return hipSuccess;
    hipLaunchKernelGGL(k_add_sums, dim3(unsigned((maxN + 255) / 256), unsigned(nSegs)), dim3(256), 0, s, dSegs);
    return hipGetLastError();
}

hipError_t launch_add_call_sums(const LossParams* L, const AdjointParams& A, int B, int R, int C, hipStream_t s)
{
    const double* lossSum = L ? L->lossSum : nullptr;
    const int n = A.atfSum ? (A.atfSb != 0 ? B : 1) * R * C : 0;
    if (n == 0 && !lossSum) return hipSuccess;
    hipLaunchKernelGGL(k_add_call_sums, dim3(unsigned(n > 0 ? (n + 255) / 256 : 1)), dim3(256), 0, s, lossSum,
                       L ? L->lossOut : nullptr, A.atfSum, A.atf, n, R * C, C, A.atfSb, A.atfSr, A.atfSc);
    return hipGetLastError();
}

hipError_t launch_debrick(const DebrickSeg* dSegs, int nSegs, long long maxBricks, hipStream_t s)
{
    if (nSegs <= 0) return hipSuccess;
    long long bx = (4 * maxBricks + 255) / 256;
    if (bx > 8192) bx = 8192;
    if (bx < 1) bx = 1;
    hipLaunchKernelGGL(k_debrick, dim3(unsigned(bx), unsigned(nSegs)), dim3(256), 0, s, dSegs);
    return hipGetLastError();
}

}  // namespace dvr
