// Pre-shaded volumes (renderer/renderer_interpolation.cuh:390-579,
// renderer/renderer_tf.cuh:818-854): the volume carries red, green, blue and
// absorption in its four batch slices; a sample's colour is the trilinear
// interpolation of each slice and the TF passes it on unchanged.  The render
// batch is a single image set (B taken from the camera, TF and step tensors).
//
// The adjoint method is the reference's: the accumulator is reconstructed by
// inverting the blend step.  The position adjoint of a channel is the gradient
// of its trilinear form; the reference writes the z term into the y component
// (renderer_interpolation.cuh:557-562), which these kernels do not reproduce.
//
// Two forms.  With call scratch the four slices are first packed into one RGBA
// volume, so a new cell is eight 16-byte loads instead of 32 floats from four
// planes, a workgroup takes an 8x8 tile of rays instead of pixels of an image row,
// and the adjoint leaves the corner gradients to k_scatter_volume, a pass per
// channel.  4 x 128^3, 4 x 256 x 256 rays: forward 1506 -> 245 us with the packing,
// adjoint 14379 -> 1705 us (walk 553, scatter 1113, packing and k_debrick 38).  Without scratch (C callers, memory short, few rays for the volume)
// one thread per pixel gathers from the planes and adds the corner gradients
// with device atomics.
#include "dvr_tiled_impl.hpp"
#include "dvr_launch.hpp"

namespace dvr {

constexpr int kInvalidCell4 = -0x40000000;

// the 8 corners of a cell in each of the 4 channels
__device__ __forceinline__ void cell4_load(const RenderParams& P, int ix, int iy, int iz, float d[4][8])
{
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) cell_load(make_vol(P, ch), ix, iy, iz, d[ch]);
}

__device__ __forceinline__ f4 cell4_value(const float d[4][8], float fx, float fy, float fz)
{
    return mk4(tri_lerp(d[0], fx, fy, fz), tri_lerp(d[1], fx, fy, fz), tri_lerp(d[2], fx, fy, fz),
               tri_lerp(d[3], fx, fy, fz));
}

template <int BLEND>
__global__ __launch_bounds__(256) void k_forward_preshaded(RenderParams P, int total)
{
    const int stride = blockDim.x * gridDim.x;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int b = i / (P.W * P.H);
        const int y = (i - b * P.W * P.H) / P.W;
        const int x = i - P.W * (y + P.H * b);
        const Ray r = setup_ray(P, x, y, b);
        float d[4][8];
        int cx = kInvalidCell4, cy = 0, cz = 0;
        f4 acc = mk4(0.f, 0.f, 0.f, 0.f);
        int n;
        for (n = 0; n < kMaxSamples; ++n) {
            const float t = r.t0 + float(n) * r.step;
            if (t > r.t1) break;
            if (acc.w > P.earlyOut) break;
            const f3 p = sample_pos(r, t);
            const int ix = int(p.x), iy = int(p.y), iz = int(p.z);
            if (ix != cx || iy != cy || iz != cz) {
                cell4_load(P, ix, iy, iz, d);
                cx = ix; cy = iy; cz = iz;
            }
            blend<BLEND>(acc, cell4_value(d, p.x - float(ix), p.y - float(iy), p.z - float(iz)), r.step);
        }
        float* o = P.color + b * P.colSb + y * P.colSy + x * P.colSx;
        o[0] = acc.x; o[P.colSc] = acc.y; o[2 * P.colSc] = acc.z; o[3 * P.colSc] = acc.w;
        P.term[b * P.termSb + y * P.termSy + x * P.termSx] = n;
    }
}

// corner gradients of the current cell, 4 channels, added to adj_volume with atomics
__device__ __forceinline__ void flush_cell4(const RenderParams& P, const AdjointParams& A, int cx, int cy, int cz,
                                            float w[4][8])
{
    const int lx = iclamp(cx, 0, P.X - 1), hx = iclamp(cx + 1, 0, P.X - 1);
    const int ly = iclamp(cy, 0, P.Y - 1), hy = iclamp(cy + 1, 0, P.Y - 1);
    const int lz = iclamp(cz, 0, P.Z - 1), hz = iclamp(cz + 1, 0, P.Z - 1);
    const int xs[2] = {lx * A.avSx, hx * A.avSx}, ys[2] = {ly * A.avSy, hy * A.avSy}, zs[2] = {lz * A.avSz, hz * A.avSz};
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {
        float* base = A.avol + ch * A.avSb;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (w[ch][k] != 0.0f) atomicAdd(base + xs[(k >> 2) & 1] + ys[(k >> 1) & 1] + zs[k & 1], w[ch][k]);
            w[ch][k] = 0.0f;
        }
    }
}

__device__ __forceinline__ void write_pos_adjoint(const AdjointParams& A, int b, int x, int y, float adj_step,
                                                  const f3& adj_start, const f3& adj_dir)
{
    if (A.ast) {
        float* o = A.ast + b * A.astSb + y * A.astSy + x * A.astSx;
        if (A.stepBroadcast) atomicAdd(o, adj_step);
        else *o = adj_step;
    }
    if (A.ars) {
        float* os = A.ars + b * A.arsSb + y * A.arsSy + x * A.arsSx;
        float* od = A.ard + b * A.ardSb + y * A.ardSy + x * A.ardSx;
        if (A.camBroadcast) {
            atomicAdd(os, adj_start.x); atomicAdd(os + A.arsSc, adj_start.y); atomicAdd(os + 2 * A.arsSc, adj_start.z);
            atomicAdd(od, adj_dir.x); atomicAdd(od + A.ardSc, adj_dir.y); atomicAdd(od + 2 * A.ardSc, adj_dir.z);
        } else {
            os[0] = adj_start.x; os[A.arsSc] = adj_start.y; os[2 * A.arsSc] = adj_start.z;
            od[0] = adj_dir.x; od[A.ardSc] = adj_dir.y; od[2 * A.ardSc] = adj_dir.z;
        }
    }
}

template <int BLEND>
__global__ __launch_bounds__(256) void k_adjoint_preshaded(RenderParams P, AdjointParams A, int total)
{
    const int stride = blockDim.x * gridDim.x;
    const bool wantVol = A.avol != nullptr;
    const bool wantPos = (A.ars != nullptr) || (A.ast != nullptr);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int b = i / (P.W * P.H);
        const int y = (i - b * P.W * P.H) / P.W;
        const int x = i - P.W * (y + P.H * b);
        const Ray r = setup_ray(P, x, y, b);
        const float* fc = A.fcol + b * A.fcSb + y * A.fcSy + x * A.fcSx;
        f4 acc = mk4(fc[0], fc[A.fcSc], fc[2 * A.fcSc], fc[3 * A.fcSc]);
        const int n = min(A.fterm[b * A.ftSb + y * A.ftSy + x * A.ftSx], kMaxSamples);
        const float* ac = A.acol + b * A.acSb + y * A.acSy + x * A.acSx;
        f4 adj_acc = mk4(ac[0], ac[A.acSc], ac[2 * A.acSc], ac[3 * A.acSc]);
        float adj_step = 0.0f;
        f3 adj_start = mk3(0.f, 0.f, 0.f), adj_dir = mk3(0.f, 0.f, 0.f);
        float d[4][8], w[4][8];
#pragma unroll
        for (int ch = 0; ch < 4; ++ch)
#pragma unroll
            for (int k = 0; k < 8; ++k) w[ch][k] = 0.0f;
        int cx = kInvalidCell4, cy = 0, cz = 0;
        for (int s_i = n - 1; s_i >= 0; --s_i) {
            const float t = r.t0 + float(s_i) * r.step;
            const f3 p = sample_pos(r, t);
            const int ix = int(p.x), iy = int(p.y), iz = int(p.z);
            if (ix != cx || iy != cy || iz != cz) {
                if (wantVol && cx != kInvalidCell4) flush_cell4(P, A, cx, cy, cz, w);
                cell4_load(P, ix, iy, iz, d);
                cx = ix; cy = iy; cz = iz;
            }
            const float fx = p.x - float(ix), fy = p.y - float(iy), fz = p.z - float(iz);
            const f4 s = cell4_value(d, fx, fy, fz);
            const f4 accIn = blend_invert<BLEND>(acc, s, r.step);
            f4 adj_s;
            float adj_st;
            blend_adjoint<BLEND>(accIn.w, s, r.step, adj_acc, adj_s, adj_st);
            acc = accIn;
            // the TF is the identity on the colour: adj_colour of the fetch = adj_s
            const float as[4] = {adj_s.x, adj_s.y, adj_s.z, adj_s.w};
            f3 adj_p = mk3(0.f, 0.f, 0.f);
#pragma unroll
            for (int ch = 0; ch < 4; ++ch) {
                float wc[8];
                f3 ap;
                if (wantPos) tri_adjoint<true>(d[ch], fx, fy, fz, as[ch], wc, ap);
                else tri_adjoint<false>(d[ch], fx, fy, fz, as[ch], wc, ap);
                if (wantPos) adj_p = add3(adj_p, ap);
#pragma unroll
                for (int k = 0; k < 8; ++k) w[ch][k] += wc[k];
            }
            if (wantPos) {
                const f3 adj_w = mul3(adj_p, r.invVoxel);
                adj_start = add3(adj_start, adj_w);
                adj_dir = add3(adj_dir, scl3(adj_w, t));
                adj_step += dot3(adj_w, r.dir) * float(s_i);
            }
            adj_step += adj_st;
        }
        if (wantVol && cx != kInvalidCell4) flush_cell4(P, A, cx, cy, cz, w);
        write_pos_adjoint(A, b, x, y, adj_step, adj_start, adj_dir);
    }
}

// ---------------------------------------------------------------------------
// packed form
// ---------------------------------------------------------------------------
typedef float vfloat4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) vfloat4 gfloat4;

// voxel (x, y, z) of the four slices -> packed[(x * Y + y) * Z + z]
__global__ __launch_bounds__(256) void k_pack_preshaded(RenderParams P, float* packed)
{
    const unsigned n = unsigned(P.X) * unsigned(P.Y) * unsigned(P.Z);
    for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
        const unsigned r = i / unsigned(P.Z);
        const int z = int(i - r * unsigned(P.Z)), x = int(r / unsigned(P.Y)), y = int(r - unsigned(x) * unsigned(P.Y));
        float c[4];
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
            const Vol V = make_vol(P, ch);
            c[ch] = gld(V.p, unsigned(x) * unsigned(V.sx) + unsigned(y) * unsigned(V.sy) + unsigned(z) * unsigned(V.sz));
        }
        *(gfloat4*)((gchar*)packed + i * 16u) = vfloat4{c[0], c[1], c[2], c[3]};
    }
}

__device__ __forceinline__ void cell4_load_packed(const RenderParams& P, const float* packed, int ix, int iy, int iz,
                                                  float d[4][8])
{
    const CellOffsets o = cell_offsets(ix, iy, iz, P.X, P.Y, P.Z, P.Y * P.Z, P.Z, 1);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const unsigned e = o.base + ((k & 4) ? o.dx : 0u) + ((k & 2) ? o.dy : 0u) + ((k & 1) ? o.dz : 0u);
        const vfloat4 v = *(const gfloat4*)((const gchar*)packed + e * 16u);
        d[0][k] = v.x; d[1][k] = v.y; d[2][k] = v.z; d[3][k] = v.w;
    }
}

// The cell of the next sample is requested as soon as the current sample is interpolated, so that its
// loads overlap the blend step.
struct PackedPipe {
    float d[4][8];
    int cx, cy, cz;
    __device__ __forceinline__ void start(const RenderParams& P, const float* packed, const f3& p)
    {
        cx = int(p.x); cy = int(p.y); cz = int(p.z);
        cell4_load_packed(P, packed, cx, cy, cz, d);
    }
    __device__ __forceinline__ f4 value(const f3& p) const
    {
        return cell4_value(d, p.x - float(cx), p.y - float(cy), p.z - float(cz));
    }
    __device__ __forceinline__ void request(const RenderParams& P, const float* packed, const f3& p)
    {
        const int ix = int(p.x), iy = int(p.y), iz = int(p.z);
        if (ix != cx || iy != cy || iz != cz) {
            cell4_load_packed(P, packed, ix, iy, iz, d);
            cx = ix; cy = iy; cz = iz;
        }
    }
};

// Four lanes a ray: lane q of a quad interpolates every fourth sample, and all four lanes blend the samples in
// order, each taking them from the lane that holds it.  The march is a chain of cell loads (0.8 us a sample
// with one lane a ray, the CUs a third busy); a quad has four in flight and four times the waves
// (forward 360 -> 232 us, adjoint walk 1115 -> 553 us on the scene above).
// A wave takes two rows of eight pixels, a workgroup the tile.
constexpr int kQuadBlock = 4 * kBlock;

struct QuadXY {
    int tile, b, x, y;
    int q;     // lane of the quad
    int slot;  // lane of the ray in its 8x8 tile (store layout)
};
__device__ __forceinline__ QuadXY quad_xy(int tilesX, int tilesPerView, int nTiles, int tile0)
{
    QuadXY t;
    t.tile = tile0 + xcd_remap(blockIdx.x, nTiles);
    t.b = t.tile / tilesPerView;
    const int tl = t.tile - t.b * tilesPerView;
    const int ty = tl / tilesX, tx = tl - ty * tilesX;
    t.q = threadIdx.x & 3;
    t.slot = threadIdx.x >> 2;
    t.x = tx * kTileW + (t.slot & 7);
    t.y = ty * kTileH + (t.slot >> 3);
    return t;
}
template <int Q>
__device__ __forceinline__ f4 quad_sample(const f4& s)
{
    auto get = [](float v) {
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), Q * 0x55, 0xf, 0xf, true));
    };
    return mk4(get(s.x), get(s.y), get(s.z), get(s.w));
}
__device__ __forceinline__ float quad_sum(float v)
{
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));  // lanes 1 0 3 2
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xf, 0xf, true));  // lanes 2 3 0 1
    return v;
}

// sample n of the quad's ray, in lane n & 3: false when the march ends in front of it
template <int BLEND, int Q>
__device__ __forceinline__ void quad_blend(const RenderParams& P, const Ray& r, const f4& s, f4& acc, int& n, bool& go)
{
    const f4 v = quad_sample<Q>(s);
    go = go && !(r.t0 + float(n) * r.step > r.t1) && !(acc.w > P.earlyOut);
    if (go) {
        blend<BLEND>(acc, v, r.step);
        ++n;
    }
}

template <int BLEND>
__global__ __launch_bounds__(kQuadBlock) void k_forward_preshaded_packed(RenderParams P, const float* packed, int tilesX,
                                                                         int tilesPerView, int nTiles)
{
    const QuadXY tc = quad_xy(tilesX, tilesPerView, nTiles, 0);
    if (tc.x >= P.W || tc.y >= P.H) return;
    const int b = tc.b, x = tc.x, y = tc.y;
    const Ray r = setup_ray(P, x, y, b);
    f4 acc = mk4(0.f, 0.f, 0.f, 0.f);
    int n = 0;
    bool go = true;
    PackedPipe pipe;
    f3 p = sample_pos(r, r.t0 + float(tc.q) * r.step);
    pipe.start(P, packed, p);
    while (go && n < kMaxSamples) {
        const f4 s = pipe.value(p);
        const float t = r.t0 + float(n + 4 + tc.q) * r.step;
        p = sample_pos(r, t);
        if (!(t > r.t1)) pipe.request(P, packed, p);
        quad_blend<BLEND, 0>(P, r, s, acc, n, go);
        quad_blend<BLEND, 1>(P, r, s, acc, n, go);
        quad_blend<BLEND, 2>(P, r, s, acc, n, go);
        quad_blend<BLEND, 3>(P, r, s, acc, n, go);
    }
    if (tc.q == 0) {
        float* o = P.color + b * P.colSb + y * P.colSy + x * P.colSx;
        o[0] = acc.x; o[P.colSc] = acc.y; o[2 * P.colSc] = acc.z; o[3 * P.colSc] = acc.w;
        P.term[b * P.termSb + y * P.termSy + x * P.termSx] = n;
    }
}

// steps over the sample that lane Q holds, the ray's i-th (i < 0: none); its adjoint goes to that lane's mine
template <int BLEND, int Q>
__device__ __forceinline__ void quad_adjoint(const Ray& r, const f4& s, int q, int i, f4& acc, f4& adj_acc, f4& mine,
                                             float& adj_step)
{
    const f4 v = quad_sample<Q>(s);
    if (i < 0) return;
    const f4 accIn = blend_invert<BLEND>(acc, v, r.step);
    f4 adj_s;
    float adj_st;
    blend_adjoint<BLEND>(accIn.w, v, r.step, adj_acc, adj_s, adj_st);
    acc = accIn;
    adj_step += q == 0 ? adj_st : 0.0f;
    if (q == Q) mine = adj_s;
}

// The density adjoints of k_scatter_volume are here the four colour adjoints of a sample, channel ch
// at S.adj + ch * plane (S.adj NULL: no volume gradient).
template <int BLEND, bool POS>
__global__ __launch_bounds__(kQuadBlock) void k_adjoint_preshaded_packed(RenderParams P, AdjointParams A,
                                                                         const float* packed, AdjStore S, size_t plane,
                                                                         int tilesX, int tilesPerView, int nTiles,
                                                                         int tile0)
{
    const QuadXY tc = quad_xy(tilesX, tilesPerView, nTiles, tile0);
    if (tc.x >= P.W || tc.y >= P.H) {
        if (S.adj && tc.q == 0) store_ray(S, tc.tile - tile0, tc.slot, Ray{}, 0);
        return;
    }
    const int b = tc.b, x = tc.x, y = tc.y, q = tc.q;
    const Ray r = setup_ray(P, x, y, b);
    const float* fc = A.fcol + b * A.fcSb + y * A.fcSy + x * A.fcSx;
    f4 acc = mk4(fc[0], fc[A.fcSc], fc[2 * A.fcSc], fc[3 * A.fcSc]);
    const int n = min(A.fterm[b * A.ftSb + y * A.ftSy + x * A.ftSx], kMaxSamples);
    const float* ac = A.acol + b * A.acSb + y * A.acSy + x * A.acSx;
    f4 adj_acc = mk4(ac[0], ac[A.acSc], ac[2 * A.acSc], ac[3 * A.acSc]);
    float adj_step = 0.0f;
    f3 adj_start = mk3(0.f, 0.f, 0.f), adj_dir = mk3(0.f, 0.f, 0.f);
    float* store = nullptr;
    if (S.adj) {
        if (q == 0) store_ray(S, tc.tile - tile0, tc.slot, r, n);
        store = adj_store<false>(S, tc.tile - tile0, tc.slot).p;
    }
    PackedPipe pipe;
    if (n > 0) pipe.start(P, packed, sample_pos(r, r.t0 + float(max(n - 1 - q, 0)) * r.step));
    for (int last = n - 1; last >= 0; last -= 4) {
        const int i = last - q;  // this lane's sample (negative: none; its cell is the first sample's)
        const float t = r.t0 + float(max(i, 0)) * r.step;
        const f3 p = sample_pos(r, t);
        // the position adjoint needs the corners after the blend steps
        if constexpr (POS) pipe.request(P, packed, p);
        const f4 s = pipe.value(p);
        if constexpr (!POS) pipe.request(P, packed, sample_pos(r, r.t0 + float(max(i - 4, 0)) * r.step));
        f4 mine = mk4(0.f, 0.f, 0.f, 0.f);
        quad_adjoint<BLEND, 0>(r, s, q, last, acc, adj_acc, mine, adj_step);
        quad_adjoint<BLEND, 1>(r, s, q, last - 1, acc, adj_acc, mine, adj_step);
        quad_adjoint<BLEND, 2>(r, s, q, last - 2, acc, adj_acc, mine, adj_step);
        quad_adjoint<BLEND, 3>(r, s, q, last - 3, acc, adj_acc, mine, adj_step);
        if (i < 0) continue;
        if (store) {
            if (i < S.cap) {
                gfloat* o = (gfloat*)(store + i * kBlock);
                o[0] = mine.x; o[plane] = mine.y; o[2 * plane] = mine.z; o[3 * plane] = mine.w;
            } else {  // past the capacity: straight to the gradient
                VolDirect vs;
                vs.L = LinearLayout{P.X, P.Y, P.Z, A.avSx, A.avSy, A.avSz};
                const Vol V = make_vol(P, 0);
#pragma unroll 1
                for (int ch = 0; ch < 4; ++ch) {
                    vs.p = A.avol + ch * A.avSb;
                    add_sample<1>(vs, V, p, ch == 0 ? mine.x : (ch == 1 ? mine.y : (ch == 2 ? mine.z : mine.w)));
                }
            }
        }
        if constexpr (POS) {
            const float as[4] = {mine.x, mine.y, mine.z, mine.w};
            const float fx = p.x - float(pipe.cx), fy = p.y - float(pipe.cy), fz = p.z - float(pipe.cz);
            f3 adj_p = mk3(0.f, 0.f, 0.f);
#pragma unroll
            for (int ch = 0; ch < 4; ++ch) {
                float unused[8];
                f3 ap;
                tri_adjoint<true>(pipe.d[ch], fx, fy, fz, as[ch], unused, ap);
                adj_p = add3(adj_p, ap);
            }
            const f3 adj_w = mul3(adj_p, r.invVoxel);
            adj_start = add3(adj_start, adj_w);
            adj_dir = add3(adj_dir, scl3(adj_w, t));
            adj_step += dot3(adj_w, r.dir) * float(i);
        }
    }
    if (A.ast || A.ars) {
        adj_step = quad_sum(adj_step);
        adj_start = mk3(quad_sum(adj_start.x), quad_sum(adj_start.y), quad_sum(adj_start.z));
        adj_dir = mk3(quad_sum(adj_dir.x), quad_sum(adj_dir.y), quad_sum(adj_dir.z));
        if (q == 0) write_pos_adjoint(A, b, x, y, adj_step, adj_start, adj_dir);
    }
}

// The forward march gathers 32 floats per new cell: at most two 256-thread
// workgroups per CU keep the rays in flight within what L1 holds (C2 scene
// pre-shaded, 4 x 128^3: 3.04 -> 2.72 ms).  The adjoint is bound by its
// volume-gradient atomics and keeps the register-limited occupancy.
constexpr int kPreshadedFwdWgPerCu = 2;

static int preshaded_grid(int total)
{
    const int want = (total + 255) / 256;
    return want < 4096 ? want : 4096;
}

hipError_t launch_pack_preshaded(const RenderParams& P, float* packed, hipStream_t s)
{
    const size_t n = size_t(P.X) * P.Y * P.Z;
    const size_t bx = (n + 255) / 256;
    hipLaunchKernelGGL(k_pack_preshaded, dim3(unsigned(bx < 8192 ? bx : 8192)), dim3(256), 0, s, P, packed);
    return hipGetLastError();
}

hipError_t launch_forward_preshaded(const RenderParams& P, int blend, const float* packed, hipStream_t s)
{
    const int total = P.W * P.H * P.B;
    if (total == 0) return hipSuccess;
    if (packed) {
        const int tilesX = (P.W + kTileW - 1) / kTileW, tilesPerView = tilesX * ((P.H + kTileH - 1) / kTileH);
        const int nTiles = tilesPerView * P.B;
        if (blend == 0)
            hipLaunchKernelGGL(k_forward_preshaded_packed<0>, dim3(nTiles), dim3(kQuadBlock), 0, s, P, packed, tilesX,
                               tilesPerView, nTiles);
        else
            hipLaunchKernelGGL(k_forward_preshaded_packed<1>, dim3(nTiles), dim3(kQuadBlock), 0, s, P, packed, tilesX,
                               tilesPerView, nTiles);
        return hipGetLastError();
    }
    const size_t lds = occupancy_lds(0, kPreshadedFwdWgPerCu);
    if (blend == 0) hipLaunchKernelGGL(k_forward_preshaded<0>, dim3(preshaded_grid(total)), dim3(256), lds, s, P, total);
    else hipLaunchKernelGGL(k_forward_preshaded<1>, dim3(preshaded_grid(total)), dim3(256), lds, s, P, total);
    return hipGetLastError();
}

hipError_t launch_adjoint_preshaded_packed(const RenderParams& P, const AdjointParams& A, const CkptParams& CK,
                                           size_t plane, const float* packed, int blend, hipStream_t s)
{
    const int tilesX = (P.W + kTileW - 1) / kTileW, tilesPerView = tilesX * ((P.H + kTileH - 1) / kTileH);
    const bool pos = A.ars || A.ast;
#define DVR_PACKED(BL, PS)                                                                                            \
    hipLaunchKernelGGL((k_adjoint_preshaded_packed<BL, PS>), dim3(CK.tileN), dim3(kQuadBlock), 0, s, P, A, packed, CK.as, \
                       plane, tilesX, tilesPerView, CK.tileN, CK.tile0)
    if (blend == 0) {
        if (pos) DVR_PACKED(0, true);
        else DVR_PACKED(0, false);
    } else {
        if (pos) DVR_PACKED(1, true);
        else DVR_PACKED(1, false);
    }
#undef DVR_PACKED
    return hipGetLastError();
}

hipError_t launch_adjoint_preshaded(const RenderParams& P, const AdjointParams& A, int blend, hipStream_t s)
{
    const int total = P.W * P.H * P.B;
    if (total == 0) return hipSuccess;
    if (blend == 0) hipLaunchKernelGGL(k_adjoint_preshaded<0>, dim3(preshaded_grid(total)), dim3(256), 0, s, P, A, total);
    else hipLaunchKernelGGL(k_adjoint_preshaded<1>, dim3(preshaded_grid(total)), dim3(256), 0, s, P, A, total);
    return hipGetLastError();
}

}  // namespace dvr
