// Row kernels for small launches: the 16 lanes of a DPP row march 16 consecutive
// samples of ONE ray, so a wave64 holds 4 rays (2x2 pixels) instead of 64.
//
// What bounds a small launch is the serial chain of a ray (one sample after the
// other, each with its gathers, LDS reads and ~130 dependent instructions) with
// too few waves to hide it.  Everything a sample needs except the transmittance
// in front of it depends on its index alone, so the 16 lanes fetch, shade and
// (in reverse) differentiate 16 samples at once; only the transmittance, and in
// reverse the adjoint of the accumulated alpha, run through the samples in
// order, as a chain of 16 multiplies whose operands are broadcast inside the row
// (v_mul_f32 with row_newbcast).  The chain multiplies in the order of the
// one-ray-per-lane march, so transmittances, checkpoints, densities and sample
// counts are bitwise those of k_forward_tiled.  So are the colours: the row's 16
// shaded samples pass through LDS, and each lane adds the samples of one
// channel in order (30 instructions for 16 samples, against 112 with operands
// broadcast inside the row).  Gradients are summed per lane and then across the
// row.
//
// Two reverse marches:
//   row_reverse     position (camera / step) gradients alone: 16 samples at once,
//                   as the forward.  It keeps no per-segment register arrays
//                   (105-116 VGPRs against 160-232) and shades each sample once, so
//                   it serves large launches as well.
//   split_reverse   TF and volume gradients: their sinks merge consecutive
//                   samples of a ray in registers, so the 16 lanes take 16
//                   consecutive parts of the ray instead of 16 consecutive
//                   samples, each walked back by march_reverse.  A part starts
//                   from the checkpoint in front of it; the adjoint of the
//                   accumulated alpha behind it is the composition of the later
//                   parts' affine maps, formed in a first pass.
//
// Measured (MI355X, kernel time against the tiled kernels): forward of 128^2 rays
// through 64^3, linear TF, 83 -> 20 us; 256^2 rays x 8 views through 256^3, 1313 -> 785 us
// (a wave of 64 neighbouring rays touches more cache lines than 4 rays x 16 samples
// where pixels lie further apart than samples); adjoint of 128^2 rays: TF gradient
// 250 -> 65 us (128^3, quarter-voxel steps), volume gradient of 256^3 3002 -> 321 us,
// camera gradient with a 4-row Gaussian TF 593 -> 57 us.  Where each kernel is the
// better one: use_row_forward, use_row_adjoint (dvr_kernels_row.hip).
//
// Checkpoints and densities keep the layout of the tiled kernels ([tile][c][64],
// [tile][i][64]): either kind of forward may precede either kind of adjoint.
#pragma once
#include "dvr_tiled_impl.hpp"

namespace dvr {

constexpr int kRowBlock = 256;   // threads of a forward workgroup: 16 rays, 4x4 pixels (a wave: 2x2)
// Threads of an adjoint workgroup.  The rays of a workgroup share one LDS TF-gradient table: one-wave
// workgroups add four times as often to the caller's few entries and meet there (identity TF, 2048
// tiles: 175 us and 4e-6 rounding of the many partial sums against 159 us and 1e-6; 512 threads
// were slower from 1024 tiles on, 187 against 141 us with a 5-point linear TF).
constexpr int kRowAdjBlock = 256;
constexpr int row_blocks_per_tile(int threads) { return kBlock * kRow / threads; }

// value of lane S of the caller's row; every lane of the row must be active
template <int S>
__device__ __forceinline__ float row_bcast(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + S, 0xf, 0xf, true));  // row_newbcast
}

__device__ __forceinline__ float row_sum(float v)
{
#pragma unroll
    for (int o = kRow / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// T: transmittance before the row's first sample, after its last one on return;
// before: the one in front of this lane's sample.
template <int S = 0>
__device__ __forceinline__ void row_transmittance(int s, float keep, float& T, float& before)
{
    if constexpr (S < kRow) {
        before = s == S ? T : before;
        T *= row_bcast<S>(keep);
        row_transmittance<S + 1>(s, keep, T, before);
    }
}

// Adjoint of the accumulated alpha, from the row's last sample to its first:
// a' = a * keep - drop per sample; at: the one behind this lane's sample.
template <int S = kRow - 1>
__device__ __forceinline__ void row_adjoint_alpha(int s, float keep, float drop, float& a, float& at)
{
    if constexpr (S >= 0) {
        at = s == S ? a : at;
        a = fmaf(a, row_bcast<S>(keep), -row_bcast<S>(drop));
        row_adjoint_alpha<S - 1>(s, keep, drop, a, at);
    }
}

struct RowXY {
    int tile, b, x, y;
    int s;      // sample of the row
    int slot;   // lane of the ray in its 8x8 tile (checkpoint and density layout)
};

template <int THREADS>
__device__ __forceinline__ RowXY row_xy(int tilesX, int tilesPerView, int nTiles)
{
    constexpr int kPer = row_blocks_per_tile(THREADS);
    const int blk = xcd_remap(blockIdx.x, nTiles * kPer);
    const int tile = blk / kPer;
    const int wave = (blk - tile * kPer) * (THREADS / 64) + int(threadIdx.x >> 6);  // 0..15 in the tile
    const int row = (threadIdx.x & 63) >> 4;
    RowXY t;
    t.tile = tile;
    t.b = tile / tilesPerView;
    const int tl = tile - t.b * tilesPerView;
    const int ty = tl / tilesX, tx = tl - ty * tilesX;
    // 2x2 pixels a wave, 4x4 four consecutive waves
    const int lx = ((wave >> 2) & 1) * 4 + (wave & 1) * 2 + (row & 1);
    const int ly = (wave >> 3) * 4 + ((wave >> 1) & 1) * 2 + (row >> 1);
    t.x = tx * kTileW + lx;
    t.y = ty * kTileH + ly;
    t.s = threadIdx.x & (kRow - 1);
    t.slot = ly * kTileW + lx;
    return t;
}

// LDS exchange of a row: 16 floats each of r, g, b, alpha, the weight T * alpha of
// the colours and T; the stride puts the 16-byte reads of the four rows on
// different banks.  The accumulated alpha is summed as fma(T, alpha, A), which is
// what the compiler makes of march_forward's A += T * alpha.
constexpr int kRowXchg = 6 * kRow + 4;
constexpr int kRowXchgFloats = (kRowBlock / kRow) * kRowXchg;

// Forward march of a row's ray (see march_forward for frozen, ck, cap, dsw and
// dsCap; a checkpoint every 2^ckShift samples).  Every lane of the wave calls it; xc
// is the row's exchange.  On return the lane holds channel s & 3 of the ray's RGBA
// in `channel`, and the ray's sample count in n.
template <int FILTER, int TFM, int BLEND>
__device__ __forceinline__ void row_forward(const Vol& V, const Tf& T, const Ray& r, bool valid, int s, float earlyOut,
                                            int frozen, float* xc, float& channel, int& n, float* ck, int ckShift,
                                            int cap, float* dsw, int dsCap)
{
    float Tr = 1.0f;
    const float4* xv = reinterpret_cast<const float4*>(xc + (s & 3) * kRow);
    const float4* xwt = reinterpret_cast<const float4*>(xc + ((s & 3) == 3 ? 5 : 4) * kRow);
    channel = 0.0f;
    n = 0;
    const float tEarly = 1.0f - earlyOut;
    const int rowShift = int(threadIdx.x & 63u) - s;
    bool alive = valid;  // the row's ray may have more samples (uniform over the row)
    for (int i0 = 0; i0 < kMaxSamples && __any(alive); i0 += kRow) {
        const int i = i0 + s;
        const float t = r.t0 + float(i) * r.step;
        const bool in = alive && (frozen >= 0 ? i < frozen : !(t > r.t1));
        float d = 0.0f, alpha = 0.0f, keep = 1.0f;
        f4 c = mk4(0.f, 0.f, 0.f, 0.f);
        if (in) {
            Cell cell;
            cell_invalidate(cell);
            d = fetch<FILTER>(V, sample_pos(r, t), cell);
            c = tf_eval<TFM, true>(T, d);
            alpha_keep<BLEND>(c.w, r.step, alpha, keep);
        }
        float before = 0.0f;
        row_transmittance(s, keep, Tr, before);
        // samples of this round that the march takes: up to the first one past the ray's end or
        // behind the early-out threshold
        const bool go = in && (frozen >= 0 || !(before < tEarly));
        const unsigned bits = unsigned(__ballot(go) >> rowShift) & ((1u << kRow) - 1u);
        const int cnt = __builtin_ctz(~bits);
        const bool taken = s < cnt;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        xc[s] = taken ? c.x : 0.0f;
        xc[kRow + s] = taken ? c.y : 0.0f;
        xc[2 * kRow + s] = taken ? c.z : 0.0f;
        xc[3 * kRow + s] = taken ? alpha : 0.0f;
        xc[4 * kRow + s] = taken ? before * alpha : 0.0f;
        xc[5 * kRow + s] = taken ? before : 0.0f;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
        for (int k = 0; k < kRow / 4; ++k) {
            const float4 v = xv[k], w = xwt[k];
            channel = fmaf(w.x, v.x, channel);
            channel = fmaf(w.y, v.y, channel);
            channel = fmaf(w.z, v.z, channel);
            channel = fmaf(w.w, v.w, channel);
        }
        if (taken) {
            if (dsw) *(gfloat*)(dsw + min(i, dsCap - 1) * kBlock) = d;
            if (ck && ((i + 1) & ((1 << ckShift) - 1)) == 0) {
                const int k = ((i + 1) >> ckShift) - 1;
                if (k < cap) ck[k * kBlock] = before * keep;
            }
        }
        if (alive) {
            n = i0 + cnt;
            alive = cnt == kRow;
        }
    }
}

// channel C of a row's colour in every lane (quad_perm broadcast)
template <int C>
__device__ __forceinline__ float row_channel(float channel)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(channel), C * 0x55, 0xf, 0xf, true));
}

// Reverse march of a row's ray (see march_reverse): position gradients.  Every
// lane of the wave calls it; adj_start, adj_dir and adj_step are per-lane sums.
template <int FILTER, int TFM, int BLEND>
__device__ __forceinline__ void row_reverse(const Vol& V, const Tf& T, const Ray& r, int s, int n, f4 adj_acc,
                                            const float* ck, int cap, int ckShift, bool wantPos, f3& adj_start,
                                            f3& adj_dir, float& adj_step, const float* dsr)
{
    // the trilinear position adjoint needs the corner densities: it gathers them and interpolates again
    const bool gather = dsr == nullptr || (FILTER == 1 && wantPos);
    int seg = (n + kRow - 1) / kRow - 1;
    while (__any(seg >= 0)) {
        const bool on = seg >= 0;
        const int i0 = max(seg, 0) * kRow;
        // transmittance before sample i0: from the last checkpoint at or in front of it
        float Tr = 1.0f;
        int j = 0;
        if (on) {
            const int c = min(i0 >> ckShift, cap);
            if (c > 0) Tr = ck[(c - 1) * kBlock];
            j = c << ckShift;
        }
        while (__any(on && j < i0)) {  // checkpoints further apart than a row, or a ray past their capacity
            const int i = j + s;
            float alpha, keep = 1.0f;
            if (on && i < i0) {
                Cell cell;
                cell_invalidate(cell);
                const float d = dsr ? *(const gfloat*)(dsr + i * kBlock)
                                    : fetch<FILTER>(V, sample_pos(r, r.t0 + float(i) * r.step), cell);
                alpha_keep<BLEND>(tf_absorption<TFM, true>(T, d), r.step, alpha, keep);
            }
            float unused = 0.0f;
            row_transmittance(s, keep, Tr, unused);
            j += kRow;
        }
        const int i = i0 + s;
        const float t = r.t0 + float(i) * r.step;
        const bool in = on && i < n;
        Cell cell;
        cell_invalidate(cell);
#pragma unroll
        for (int k = 0; k < 8; ++k) cell.d[k] = 0.0f;
        f3 p = mk3(0.f, 0.f, 0.f);
        float d = 0.0f, alpha = 0.0f, keep = 1.0f, keepA = 1.0f, dotc = 0.0f;
        f4 c = mk4(0.f, 0.f, 0.f, 0.f);
        TfPre pre;
        if (in) {
            p = sample_pos(r, t);
            if (gather) d = fetch<FILTER>(V, p, cell);
            else d = *(const gfloat*)(dsr + i * kBlock);
            tf_prepare<TFM, true>(T, d, pre);
            c = tf_eval<TFM, true>(T, d, &pre);
            alpha_keep<BLEND>(c.w, r.step, alpha, keep);
            adjoint_alpha_keep<BLEND>(c.w, r.step, alpha, keep, keepA);
            dotc = adj_acc.x * c.x + adj_acc.y * c.y + adj_acc.z * c.z;
        }
        float before = 0.0f, at = 0.0f;
        row_transmittance(s, keep, Tr, before);
        row_adjoint_alpha(s, keepA, alpha * dotc, adj_acc.w, at);
        if (in) {
            f4 a = adj_acc, adj_s;
            a.w = at;
            float adj_st;
            blend_adjoint_ak<BLEND>(before, c, r.step, alpha, keepA, a, adj_s, adj_st);
            if (FILTER == 1 && wantPos) {
                SinkNone none;
                const float adj_d = tf_adjoint<TFM, false, SinkNone, true>(T, d, adj_s, none, &pre);
                float w[8];
                f3 adj_p;
                tri_adjoint<true>(cell.d, p.x - float(int(p.x)), p.y - float(int(p.y)), p.z - float(int(p.z)), adj_d, w,
                                  adj_p);
                const f3 adj_w = mul3(adj_p, r.invVoxel);
                adj_start = add3(adj_start, adj_w);
                adj_dir = add3(adj_dir, scl3(adj_w, t));
                adj_step += dot3(adj_w, r.dir) * float(i);
            }
            adj_step += adj_st;
        }
        --seg;
    }
}

// a at lane s: the maps a -> a * A + B of the lanes behind it, last lane first
template <int S = kRow - 1>
__device__ __forceinline__ float row_compose_behind(int s, float A, float B, float a)
{
    if constexpr (S > 0) {
        const float b = fmaf(a, row_bcast<S>(A), row_bcast<S>(B));
        return row_compose_behind<S - 1>(s, A, B, s < S ? b : a);
    } else {
        return a;
    }
}

// Reverse march of a row's ray, its 16 lanes on 16 parts of whole K-sample
// segments (see march_reverse).  Every lane of the wave calls it.
template <int FILTER, int TFM, int BLEND, int K, int GM, class Sink, class VS>
__device__ __forceinline__ void split_reverse(const Vol& V, const Tf& T, const Ray& r, int s, int n, f4 adj_acc,
                                              const float* ck, int cap, int ckShift, Sink& sink, bool wantTf,
                                              bool wantVol, bool wantPos, VS& vs, f3& adj_start, f3& adj_dir,
                                              float& adj_step, const float* dsr, AdjLane<true> as)
{
    const int nseg = (n + K - 1) / K;
    const int per = (nseg + kRow - 1) / kRow;
    const int lo = min(s * per, nseg);
    const int end = min(n, (lo + per) * K);  // first sample behind the part
    // the part's map of the adjoint of the accumulated alpha: a -> a * A + B
    float A = 1.0f, B = 0.0f;
    {
        Cell cell;
        cell_invalidate(cell);
#pragma unroll 4
        for (int i = lo * K; i < end; ++i) {
            const float d = dsr ? *(const gfloat*)(dsr + i * kBlock)
                                : fetch<FILTER>(V, sample_pos(r, r.t0 + float(i) * r.step), cell);
            const f4 c = tf_eval<TFM, true>(T, d);
            float alpha, keep, keepA;
            alpha_keep<BLEND>(c.w, r.step, alpha, keep);
            adjoint_alpha_keep<BLEND>(c.w, r.step, alpha, keep, keepA);
            B = fmaf(-A, alpha * (adj_acc.x * c.x + adj_acc.y * c.y + adj_acc.z * c.z), B);
            A *= keepA;
        }
    }
    adj_acc.w = row_compose_behind(s, A, B, adj_acc.w);
    march_reverse<FILTER, TFM, BLEND, K, GM, Sink, false, VS>(V, T, r, end, adj_acc, ck, kBlock, cap, ckShift, sink,
                                                              wantTf, wantVol, wantPos, vs, adj_start, adj_dir,
                                                              adj_step, dsr, kBlock, lo, as);
}

template <int FILTER, int TFM, int BLEND>
__global__ __launch_bounds__(kRowBlock) void k_forward_row(RenderParams P, CkptParams CK, int tilesX, int tilesPerView,
                                                           int nTiles)
{
    extern __shared__ float lds[];
    __shared__ __attribute__((aligned(16))) float s_x[kRowXchgFloats];
    const RowXY tc = row_xy<kRowBlock>(tilesX, tilesPerView, nTiles);
    stage_tf<TFM>(P, tc.b, lds);
    __syncthreads();
    const bool valid = tc.x < P.W && tc.y < P.H;
    const Ray r = setup_ray(P, min(tc.x, P.W - 1), min(tc.y, P.H - 1), tc.b);
    const Vol V = make_vol(P, tc.b);
    constexpr int kC = tf_cols<TFM>();
    const Tf T{lds, P.R, kC, tf_lds_stride<TFM>(), 1};
    float* ck = CK.buf ? CK.buf + (size_t(tc.tile) * CK.cap) * kBlock + tc.slot : nullptr;
    float* ds = CK.ds ? CK.ds + (size_t(tc.tile) * CK.dsCap) * kBlock + tc.slot : nullptr;
    float channel;
    int n;
    row_forward<FILTER, TFM, BLEND>(V, T, r, valid, tc.s, P.earlyOut, -1, s_x + (threadIdx.x / kRow) * kRowXchg, channel,
                                    n, ck, __builtin_ctz(CK.K * CK.every), CK.cap, ds, CK.dsCap);
    if (valid && tc.s < 4) {
        P.color[tc.b * P.colSb + tc.y * P.colSy + tc.x * P.colSx + tc.s * P.colSc] = channel;
        if (tc.s == 0) P.term[tc.b * P.termSb + tc.y * P.termSy + tc.x * P.termSx] = n;
    }
}

// GM: bit0 TF, bit1 volume, bit2 position; GM 4 (position alone) is row_reverse,
// the others split_reverse in 16-sample segments.  A wave keeps its own chunk
// table of volume gradients; the TF-gradient table is the workgroup's.
template <int FILTER, int TFM, int BLEND, int GM>
__global__ __launch_bounds__(kRowAdjBlock) __attribute__((amdgpu_waves_per_eu(GM == 3 ? 4 : 1))) void k_adjoint_row(
    RenderParams P, AdjointParams A, CkptParams CK, LossParams LP, int fused, int ckFromFwd, int usePriv,
    int copyStride, int tilesX, int tilesPerView, int nTiles, int aggLog2)
{
    constexpr int kThreads = kRowAdjBlock;
    extern __shared__ float lds[];
    __shared__ __attribute__((aligned(16))) float s_x[kRowXchgFloats];
    float* xc = s_x + (threadIdx.x / kRow) * kRowXchg;
    const int RC = P.R * P.C;
    float* s_tf = lds;
    const int tfFloats = tf_grad_offset(P.R * tf_lds_stride<TFM>());
    float* s_g = lds + tfFloats;
    const RowXY tc = row_xy<kThreads>(tilesX, tilesPerView, nTiles);
    const bool wantTf = (GM & 1) && A.atf != nullptr;
    const int ng = wantTf ? tf_grad_floats(RC, usePriv != 0, kThreads, copyStride) : 0;
    stage_tf<TFM>(P, tc.b, s_tf);
    for (int e = threadIdx.x; e < ng; e += kThreads) s_g[e] = 0.0f;
    constexpr bool kVolInst = (GM & 2) != 0;
    using VS = std::conditional_t<kVolInst, VolAgg<LinearLayout, float>, VolDirect>;
    VS vs;
    vs.L = LinearLayout{P.X, P.Y, P.Z, A.avSx, A.avSy, A.avSz};
    const bool aggOn = kVolInst && A.avol != nullptr;
    if constexpr (kVolInst) {
        if (aggOn) {
            char* table = reinterpret_cast<char*>(lds + agg_offset(tfFloats, ng));
            vs.init(table + (threadIdx.x >> 6) * agg_bytes(aggLog2, sizeof(float)), aggLog2);
            vs.bind(A.avol + tc.b * A.avSb);
        }
    } else {
        vs.p = nullptr;
    }
    __syncthreads();

    const bool valid = tc.x < P.W && tc.y < P.H;
    const int b = tc.b, x = min(tc.x, P.W - 1), y = min(tc.y, P.H - 1);
    const Ray r = setup_ray(P, x, y, b);
    const Vol V = make_vol(P, b);
    constexpr int kC = tf_cols<TFM>();
    const Tf T{s_tf, P.R, kC, tf_lds_stride<TFM>(), 1};
    const int ckShift = __builtin_ctz(CK.K * CK.every);
    float* ck = CK.buf + (size_t(tc.tile) * CK.cap) * kBlock + tc.slot;
    float* ds = CK.ds ? CK.ds + (size_t(tc.tile) * CK.dsCap) * kBlock + tc.slot : nullptr;
    float lossLocal = 0.0f;
    int n = 0;
    f4 adj_acc;
    if (fused) {
        float channel;
        row_forward<FILTER, TFM, BLEND>(V, T, r, valid, tc.s, P.earlyOut, -1, xc, channel, n, ck, ckShift, CK.cap, ds,
                                        CK.dsCap);
        const f4 acc = mk4(row_channel<0>(channel), row_channel<1>(channel), row_channel<2>(channel),
                           row_channel<3>(channel));
        const float* tg = LP.target + b * LP.tgSb + y * LP.tgSy + x * LP.tgSx;
        const float d0 = acc.x - tg[0], d1 = acc.y - tg[LP.tgSc], d2 = acc.z - tg[2 * LP.tgSc],
                    d3 = acc.w - tg[3 * LP.tgSc];
        const bool writer = valid && tc.s == 0;
        if (writer) {
            float* o = P.color + b * P.colSb + y * P.colSy + x * P.colSx;
            o[0] = acc.x; o[P.colSc] = acc.y; o[2 * P.colSc] = acc.z; o[3 * P.colSc] = acc.w;
            P.term[b * P.termSb + y * P.termSy + x * P.termSx] = n;
        }
        if (LP.kind == DVR_LOSS_L1) {
            auto sgn = [](float v) { return v > 0.f ? 1.f : (v < 0.f ? -1.f : 0.f); };
            adj_acc = mk4(sgn(d0) * LP.scale, sgn(d1) * LP.scale, sgn(d2) * LP.scale, sgn(d3) * LP.scale);
            if (writer) lossLocal = (fabsf(d0) + fabsf(d1) + fabsf(d2) + fabsf(d3)) * LP.scale;
        } else {
            adj_acc = mk4(2.f * d0 * LP.scale, 2.f * d1 * LP.scale, 2.f * d2 * LP.scale, 2.f * d3 * LP.scale);
            if (writer) lossLocal = (d0 * d0 + d1 * d1 + d2 * d2 + d3 * d3) * LP.scale;
        }
    } else {
        n = valid ? min(A.fterm[b * A.ftSb + y * A.ftSy + x * A.ftSx], kMaxSamples) : 0;
        const float* ac = A.acol + b * A.acSb + y * A.acSy + x * A.acSx;
        adj_acc = mk4(ac[0], ac[A.acSc], ac[2 * A.acSc], ac[3 * A.acSc]);
        if (!ckFromFwd) {
            float channel;
            int n2;
            row_forward<FILTER, TFM, BLEND>(V, T, r, valid, tc.s, P.earlyOut, n, xc, channel, n2, ck, ckShift, CK.cap, ds,
                                            CK.dsCap);
        }
    }
    if (fused || !ckFromFwd) {
        // a ray's checkpoints and densities were written by other lanes of its row
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
    f3 adj_start = mk3(0.f, 0.f, 0.f), adj_dir = mk3(0.f, 0.f, 0.f);
    float adj_step = 0.0f;
    const bool wantPos = (GM & 4) && (A.ars != nullptr || A.ast != nullptr);
    const float* dsr = ds != nullptr && __all(n <= CK.dsCap) ? ds : nullptr;
    if constexpr (GM == 4) {
        row_reverse<FILTER, TFM, BLEND>(V, T, r, tc.s, n, adj_acc, ck, CK.cap, ckShift, wantPos, adj_start, adj_dir,
                                        adj_step, dsr);
    } else {
        AdjLane<true> as;
        if constexpr ((GM & 8) != 0) {
            vs.p = A.avol + b * A.avSb;
            as = adj_store<true>(CK.as, tc.tile, tc.slot);
            if (tc.s == 0) store_ray(CK.as, tc.tile, tc.slot, r, n);
        }
        SinkTiled<TFM> sink;
        sink.init(s_g, kC, usePriv != 0, kThreads, usePriv ? 0 : copyStride);
        split_reverse<FILTER, TFM, BLEND, kRow, GM>(V, T, r, tc.s, n, adj_acc, ck, CK.cap, ckShift, sink, wantTf, aggOn,
                                                    wantPos, vs, adj_start, adj_dir, adj_step, dsr, as);
        if constexpr (kVolInst) {
            if (aggOn) vs.flush();
        }
        if (wantTf) sink.template finish<TFM == 2 ? 5 : 4>();
    }
    if constexpr ((GM & 4) != 0) {
        if (A.ast) {
            const float v = row_sum(adj_step);
            if (valid && tc.s == 0) {
                float* o = A.ast + b * A.astSb + y * A.astSy + x * A.astSx;
                if (A.stepBroadcast) atomicAdd(o, v);
                else *o = v;
            }
        }
        if (A.ars) {
            const f3 st = mk3(row_sum(adj_start.x), row_sum(adj_start.y), row_sum(adj_start.z));
            const f3 di = mk3(row_sum(adj_dir.x), row_sum(adj_dir.y), row_sum(adj_dir.z));
            if (valid && tc.s == 0) {
                float* os = A.ars + b * A.arsSb + y * A.arsSy + x * A.arsSx;
                float* od = A.ard + b * A.ardSb + y * A.ardSy + x * A.ardSx;
                if (A.camBroadcast) {
                    atomicAdd(os, st.x); atomicAdd(os + A.arsSc, st.y); atomicAdd(os + 2 * A.arsSc, st.z);
                    atomicAdd(od, di.x); atomicAdd(od + A.ardSc, di.y); atomicAdd(od + 2 * A.ardSc, di.z);
                } else {
                    os[0] = st.x; os[A.arsSc] = st.y; os[2 * A.arsSc] = st.z;
                    od[0] = di.x; od[A.ardSc] = di.y; od[2 * A.ardSc] = di.z;
                }
            }
        }
    }
    if (fused && LP.lossOut) {
        __shared__ double s_loss[kThreads / 64];
        const float v = wave_sum(lossLocal);
        if ((threadIdx.x & 63) == 0) s_loss[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x == 0) {
            double sum = 0.0;
#pragma unroll
            for (int k = 0; k < kThreads / 64; ++k) sum += s_loss[k];
            loss_add(LP, sum);
        }
    }
    if (wantTf) {
        __syncthreads();
        if (usePriv) {  // a wave sums the threads' slices of an entry
            const int lane = threadIdx.x & 63;
            for (int e = threadIdx.x >> 6; e < RC; e += kThreads / 64) {
                float v = 0.0f;
#pragma unroll
                for (int k = 0; k < kThreads / 64; ++k) v += s_g[e * kThreads + k * 64 + lane];
                v = wave_sum(v);
                if (lane == 0) tf_grad_add(P, A, b, e, v);
            }
        } else {
            for (int e = threadIdx.x; e < RC; e += kThreads) {
                tf_grad_add(P, A, b, e, tf_grad_sum(s_g, e, copyStride));
            }
        }
    }
}

}  // namespace dvr
