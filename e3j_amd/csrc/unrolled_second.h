// Kernel templates of the second-order backward (gfx950, float32, trailing-channels layout): the
// VJP of the convolution's VJP, which a loss on forces needs.
//
// With L(x, y, s) = <dm, convolution(x, y, s)>, linear in each argument, and the cotangents x', y',
// s' of (dx, dy, ds), the gradients of L(x', y, s) + L(x, y', s) + L(x, y, s') are
//
//   with respect to dm : convolution(x', y, s) + convolution(x, y', s) + convolution(x, y, s')
//   and to x, y, s     : two terms each, e.g. for s : sum_i dm_i (w_ij(y) x'_j + w_ij(y') x_j)
//
// As calls of the first-order operators that is three forward and three backward passes and the
// sums of their results: the stream of radial weights (E, S, K) crosses the memory twelve times.
// The two kernels here compute all terms of an edge while its operands are in registers: one owns
// the receiver's row (gradient with respect to dm), the other walks tiles of receivers like
// `unrolled_bwd_tile_kernel` (gradients with respect to x, y, s); five crossings in all (s and s' by
// both, the gradient written once).  Merged into one kernel the accumulated rows and the dm rows
// would have to be resident together, which leaves one wave per SIMD.
//
// 120k edges, K = 128, l <= 3: 0.71 ms (rows; the two streams alone 0.60 ms at the rate of a copy) and
// 1.22 ms (tiles; three streams, 0.90 ms) against 4.1 ms for the composed form (3 x 0.35 forward,
// 3 x 0.73 backward, 0.9 of sums); forward, backward and second-order backward together 5.37 -> 3.11 ms.
// (Every table with tiles takes them: at 64 to 256 channels, 30 to 6 000 nodes, even or hub rows, the built-in
// tables take 0.51 to 0.72 of the composed form's time.)
// Both are bound by their vector instructions (4 370 and 6 210 per edge and 128 channels) at two to three
// waves per SIMD, the tile kernel next by the latency of its first loads per tile.
#ifndef E3J_AMD_CSRC_UNROLLED_SECOND_H_
#define E3J_AMD_CSRC_UNROLLED_SECOND_H_

#include "unrolled.h"

namespace e3j_amd {

// ---------------------------------------------------------------------------
// gradient with respect to dm: rows of receivers, as the forward pass
// ---------------------------------------------------------------------------
template <typename Part, int K, int CPL>
__device__ __forceinline__ void second_dm_part(const float *__restrict__ x, const float *__restrict__ y,
                                               const float *__restrict__ s, const float *__restrict__ x2,
                                               const float *__restrict__ y2, const float *__restrict__ s2,
                                               const int32_t *__restrict__ sender,
                                               const int32_t *__restrict__ perm, float *__restrict__ row_out,
                                               int num_nodes, float scale, unsigned y_flip, int slice, int lane,
                                               int e, int e1) {
    constexpr int NX = Part::NX, NS = Part::NS, NZ = Part::NZ, Y = Part::Y;
    constexpr int X = Part::X, S = Part::S;
    using V = Vec<CPL>;
    using SL = Slice<K, CPL>;
    static_assert(SL::SUB == 1 && SL::FULL, "whole waves of channels");
    const int c0 = slice * SL::WIDTH + lane * CPL;

    V acc[NZ];
#pragma unroll
    for (int i = 0; i < NZ; i++) acc[i] = vzero<CPL>();

    V xn[NX], xn2[NX], sn[NS], sn2[NS];
    YRow<Y> yn, yn2;
    unsigned flips[YRow<Y>::N];
    YRow<Y>::signs(y_flip, lane, flips);
    EdgeBatch batch;
    auto fetch = [&](int at) {
        const int64_t ee = batch.edge_at(at);
        const int64_t xo = (int64_t)batch.sender_at(at) * (X * K) + c0, so = ee * (int64_t)(S * K) + c0;
        yn.load(y + ee * Y, lane);
        yn2.load(y2 + ee * Y, lane);
#pragma unroll
        for (int j = 0; j < NX; j++) {
            xn[j] = load_vec<CPL>(x + xo + Part::kX[j] * K);
            xn2[j] = load_vec<CPL>(x2 + xo + Part::kX[j] * K);
        }
#pragma unroll
        for (int l = 0; l < NS; l++) {
            sn[l] = load_stream<CPL>(s + so + Part::kS[l] * K);
            sn2[l] = load_stream<CPL>(s2 + so + Part::kS[l] * K);
        }
    };
    for (; e < e1; e += kWave) {
        batch.load(sender, perm, e, e1, num_nodes, lane);
        bool more = batch.live != 0;
        if (more) fetch(batch.take());
        while (more) {
            V xc[NX], xc2[NX], sc[NS], sc2[NS];
            float yc[Y], yc2[Y];
#pragma unroll
            for (int j = 0; j < NX; j++) {
                xc[j] = xn[j];
                xc2[j] = xn2[j];
            }
#pragma unroll
            for (int l = 0; l < NS; l++) {
                sc[l] = sn[l];
                sc2[l] = sn2[l];
            }
            yn.template spread<0>(yc, flips);
            yn2.template spread<0>(yc2, flips);
            more = batch.live != 0;
            if (more) fetch(batch.take());
            Part::template edge_second_dm<CPL>(xc, yc, sc, xc2, yc2, sc2, acc);
        }
    }
#pragma unroll
    for (int i = 0; i < NZ; i++) store_stream<CPL>(row_out + Part::kZ[i] * K + c0, vmul(acc[i], scale));
}

template <int K, int CPL, int I, typename Part, typename... Rest>
__device__ __forceinline__ void dispatch_second_dm(int part, const float *x, const float *y, const float *s,
                                                   const float *x2, const float *y2, const float *s2,
                                                   const int32_t *sender, const int32_t *perm, float *row_out,
                                                   int num_nodes, float scale, unsigned y_flip, int slice,
                                                   int lane, int e, int e1) {
    if (part == I)
        second_dm_part<Part, K, CPL>(x, y, s, x2, y2, s2, sender, perm, row_out, num_nodes, scale, y_flip, slice,
                                     lane, e, e1);
    else if constexpr (sizeof...(Rest) > 0)
        dispatch_second_dm<K, CPL, I + 1, Rest...>(part, x, y, s, x2, y2, s2, sender, perm, row_out, num_nodes,
                                                   scale, y_flip, slice, lane, e, e1);
}

// One wave per (receiver, channel slice, part); a listed piece of a long row is an item of its own,
// whose sums go to a row of `partials` (see `row_or_piece`).
template <int K, int CPL, int WPB, int MINW, typename... Parts>
__global__ __launch_bounds__(kWave *WPB, MINW) void second_dm_kernel(
    const float *__restrict__ x, const float *__restrict__ y, const float *__restrict__ s,
    const float *__restrict__ x2, const float *__restrict__ y2, const float *__restrict__ s2,
    const int32_t *__restrict__ sender, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ perm,
    const int32_t *__restrict__ row_order, float *__restrict__ out, int num_nodes, float scale, unsigned y_flip,
    int row_cap, int row_piece, const int32_t *__restrict__ segments, int max_segments,
    float *__restrict__ partials) {
    using P0 = typename FirstOfParts<Parts...>::type;
    constexpr int NP = sizeof...(Parts), CW = Slice<K, CPL>::COUNT;
    int64_t item;
    bool piece;
    if (!row_or_piece<WPB, CW * NP>(num_nodes, segments, max_segments, item, piece)) return;
    const int part = uniform((int)(item % NP));
    const int slice = uniform((int)((item / NP) % CW));
    const int q = uniform((int)(item / (NP * CW)));
    int e, e1;
    float *row_out;
    if (piece) {
        e = segments[5 + 3 * q];
        e1 = segments[6 + 3 * q];
        row_out = partials + (int64_t)q * (P0::Z * K);
    } else {
        const int r = row_order ? row_order[q] : q;
        e = row_ptr[r];
        e1 = row_ptr[r + 1];
        if (row_cap > 0 && e1 - e > row_cap) e1 = e + row_piece;
        row_out = out + (int64_t)r * (P0::Z * K);
    }
    dispatch_second_dm<K, CPL, 0, Parts...>(part, x, y, s, x2, y2, s2, sender, perm, row_out, num_nodes, scale,
                                            y_flip, slice, threadIdx.x, uniform(e), uniform(e1));
}

// ---------------------------------------------------------------------------
// gradients with respect to x, y and s: tiles of receivers, as `unrolled_bwd_tile_kernel`
// (schedule, staging of dm in LDS, sums over runs of one sender and straight edge loop are described there)
// ---------------------------------------------------------------------------
template <typename Part, int K, int CPL, bool kAtomicDy>
__device__ __forceinline__ void second_tile_part(
    const float *__restrict__ x, const float *__restrict__ y, const float *__restrict__ s,
    const float *__restrict__ x2, const float *__restrict__ y2, const float *__restrict__ s2,
    const float *__restrict__ dm, const int32_t *__restrict__ t_sender, const int32_t *__restrict__ t_edge,
    const int32_t *__restrict__ t_local, const int32_t *__restrict__ row_order, float *__restrict__ dx,
    float *__restrict__ dy, float *__restrict__ ds, int num_nodes, float scale, unsigned y_flip, int tile,
    int tile_rows, int begin, int end, int slice, float *tile_lds) {
    constexpr int NX = Part::NX, NS = Part::NS, NZ = Part::NZ, Y = Part::Y;
    constexpr int X = Part::X, S = Part::S, Z = Part::Z;
    using V = Vec<CPL>;
    using SL = Slice<K, CPL>;
    using Red = WaveReduceBlocks<Y, kWave>;
    constexpr int WIDTH = SL::WIDTH;
    static_assert(SL::SUB == 1 && SL::FULL, "whole waves of channels");

    const int lane = threadIdx.x;
    const int wave = uniform(threadIdx.y), nw = blockDim.y;
    const int c0 = slice * WIDTH + lane;  // further channels of the lane: + 64, + 128, ...

    // this wave's share of the list, cut at sender boundaries
    const int n = end - begin;
    const int lo = run_start(t_sender, begin, begin + (int)((int64_t)n * wave / nw), end, lane);
    const int hi = run_start(t_sender, begin, begin + (int)((int64_t)n * (wave + 1) / nw), end, lane);

    // Indices of up to 64 positions, one per lane; read by lane in the loop.  Padding edges (their
    // dy/ds rows are zero-filled separately) are the tail of a tile's list.
    int base = lo, count = 0, snd_v = 0, ee_v = 0, loc_v = 0;
    auto read_batch = [&]() {
        const int left = hi - base, p = min(base + lane, max(hi - 1, 0));
        if (left <= 0) { count = 0; return; }
        snd_v = t_sender[p];
        ee_v = t_edge[p];
        loc_v = t_local[p];
        count = __builtin_popcountll(__ballot(lane < left && (unsigned)snd_v < (unsigned)num_nodes));
    };

    V xc[NX], xc2[NX], xn[NX], xn2[NX], sn[NS], sn2[NS], acc[NX];
    YRow<Y> yn, yn2;
    unsigned flips[YRow<Y>::N];
    YRow<Y>::signs(y_flip, lane, flips);
    bool newx_n = false;
    int snd_n = 0, loc_n = 0;
    int64_t ee_n = 0;
    auto fetch = [&](int at, int held) {  // position base + at
        snd_n = __builtin_amdgcn_readlane(snd_v, at);
        ee_n = __builtin_amdgcn_readlane(ee_v, at);
        loc_n = __builtin_amdgcn_readlane(loc_v, at);
        newx_n = snd_n != held;
        if (newx_n) {
            const int64_t xo = (int64_t)snd_n * (X * K) + c0;
#pragma unroll
            for (int j = 0; j < NX; j++) {
                xn[j] = load_apart<CPL>(x + xo + Part::kX[j] * K);
                xn2[j] = load_apart<CPL>(x2 + xo + Part::kX[j] * K);
            }
        }
        yn.load(y + ee_n * Y, lane);
        yn2.load(y2 + ee_n * Y, lane);
        const int64_t so = ee_n * (int64_t)(S * K) + c0;
#pragma unroll
        for (int l = 0; l < NS; l++) {
            sn[l] = load_apart_stream<CPL>(s + so + Part::kS[l] * K);
            sn2[l] = load_apart_stream<CPL>(s2 + so + Part::kS[l] * K);
        }
    };
    auto flush = [&](int snd) {
        float *dxr = dx + (int64_t)snd * (X * K) + c0;
#pragma unroll
        for (int j = 0; j < NX; j++) {
#pragma unroll
            for (int t = 0; t < CPL; t++) unsafeAtomicAdd(dxr + Part::kX[j] * K + t * kWave, acc[j].v[t]);
        }
    };

    int held = -1, run = -1;
    read_batch();
    if (count > 0) fetch(0, held);
    {  // stage the dm rows of the tile's receivers (scaled): row (t, i) at (t * NZ + i) * WIDTH
        const int first = tile * tile_rows;
        const int rows = num_nodes - first < tile_rows ? num_nodes - first : tile_rows;
        for (int t = wave; t < rows; t += nw) {
            const int r = row_order ? row_order[first + t] : first + t;
            const float *zr = dm + (int64_t)r * (Z * K) + c0;
            float *dst = tile_lds + t * (NZ * WIDTH) + lane * CPL;
            V v[NZ];
#pragma unroll
            for (int i = 0; i < NZ; i++) v[i] = load_apart_stream<CPL>(zr + Part::kZ[i] * K);
#pragma unroll
            for (int i = 0; i < NZ; i++) store_vec<CPL>(dst + i * WIDTH, vmul(v[i], scale));
        }
    }
    __syncthreads();

    while (count > 0) {
        // entered with nothing in flight: the waits inside the loop are exact counts of one turn
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
        for (int at = 0; at < count; at++) {
            V sc[NS], sc2[NS];
            float yc[Y], yc2[Y];
            if (newx_n) {
#pragma unroll
                for (int j = 0; j < NX; j++) {
                    xc[j] = xn[j];
                    xc2[j] = xn2[j];
                }
                held = snd_n;
            }
#pragma unroll
            for (int l = 0; l < NS; l++) {
                sc[l] = sn[l];
                sc2[l] = sn2[l];
            }
            yn.template spread<0>(yc, flips);
            yn2.template spread<0>(yc2, flips);
            const int snd = snd_n, loc = loc_n;
            const int64_t ee = ee_n;
            if (at + 1 < count) fetch(at + 1, held);
            if (snd != run) {
                if (run >= 0) flush(run);
                run = snd;
#pragma unroll
                for (int j = 0; j < NX; j++) acc[j] = vzero<CPL>();
            }
            float dye[Red::P];
#pragma unroll
            for (int k = 0; k < Red::P; k++) dye[k] = 0.f;
            const DsRows<CPL, K> ds_rows{ds + ee * (int64_t)(S * K) + c0, true};
            const DmTile<CPL> dm_rows{tile_lds + loc * (NZ * WIDTH) + lane * CPL};
            Part::template edge_second<CPL>(xc, yc, sc, xc2, yc2, sc2, dm_rows, acc, dye, ds_rows);
            Red::run(dye, lane, [&](int k, float sum) {
                const float total = flip_sign(sum, y_flip, k);
                if (!kAtomicDy) dy[ee * Y + k] = total;
                else unsafeAtomicAdd(dy + ee * Y + k, total);  // dy zero-filled by the launcher
            });
        }
        if (count < kWave) break;
        base += kWave;
        read_batch();
        if (count > 0) fetch(0, held);
    }
    if (run >= 0) flush(run);
}

template <int K, int CPL, bool A, int I, typename Part, typename... Rest>
__device__ __forceinline__ void dispatch_second_tile(
    int part, const float *x, const float *y, const float *s, const float *x2, const float *y2, const float *s2,
    const float *dm, const int32_t *t_sender, const int32_t *t_edge, const int32_t *t_local,
    const int32_t *row_order, float *dx, float *dy, float *ds, int num_nodes, float scale, unsigned y_flip,
    int tile, int tile_rows, int begin, int end, int slice, float *tile_lds) {
    if (part == I)
        second_tile_part<Part, K, CPL, A>(x, y, s, x2, y2, s2, dm, t_sender, t_edge, t_local, row_order, dx, dy, ds,
                                          num_nodes, scale, y_flip, tile, tile_rows, begin, end, slice, tile_lds);
    else if constexpr (sizeof...(Rest) > 0)
        dispatch_second_tile<K, CPL, A, I + 1, Rest...>(part, x, y, s, x2, y2, s2, dm, t_sender, t_edge, t_local,
                                                        row_order, dx, dy, ds, num_nodes, scale, y_flip, tile,
                                                        tile_rows, begin, end, slice, tile_lds);
}

template <int K, int CPL, int WPB, int MINW, typename... Parts>
__global__ __launch_bounds__(kWave *WPB, MINW) void second_tile_kernel(
    const float *__restrict__ x, const float *__restrict__ y, const float *__restrict__ s,
    const float *__restrict__ x2, const float *__restrict__ y2, const float *__restrict__ s2,
    const float *__restrict__ dm, const int32_t *__restrict__ work, const int32_t *__restrict__ t_sender,
    const int32_t *__restrict__ t_edge, const int32_t *__restrict__ t_local,
    const int32_t *__restrict__ row_order, float *__restrict__ dx, float *__restrict__ dy,
    float *__restrict__ ds, int num_nodes, int tile_rows, int num_work, float scale, unsigned y_flip) {
    extern __shared__ __attribute__((aligned(16))) float second_lds[];
    constexpr int NP = sizeof...(Parts);
    constexpr int CW = Slice<K, CPL>::COUNT;
    constexpr bool kAtomicDy = NP * CW > 1;  // several waves add into one dy row
    const int used = min(work[3], num_work);
    const int64_t items = (int64_t)used * (CW * NP);
    const int64_t per_xcd = (items + kXcds - 1) / kXcds;
    if ((int64_t)(blockIdx.x / kXcds) >= per_xcd) return;  // whole block: no barrier is left waiting
    const int64_t item = (int64_t)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (item >= items) return;
    const int part = (int)(item % NP);
    const int slice = (int)((item / NP) % CW);
    const int64_t w = item / (NP * CW);
    const int tile = work[4 * w], begin = work[4 * w + 1], end = work[4 * w + 2];
    if (begin >= end) return;  // unused descriptor or a tile without edges (uniform over the block)
    dispatch_second_tile<K, CPL, kAtomicDy, 0, Parts...>(part, x, y, s, x2, y2, s2, dm, t_sender, t_edge, t_local,
                                                         row_order, dx, dy, ds, num_nodes, scale, y_flip, tile,
                                                         tile_rows, begin, end, slice, second_lds);
}

template <int K, int CPL, int WPB, int MINW, typename... Parts>
int launch_second_dm(const e3j_amd_conv_params &p, const SecondOperands &a, const int32_t *sender,
                     const int32_t *row_ptr, const int32_t *perm, float *out, hipStream_t stream) {
    constexpr int PER_NODE = Slice<K, CPL>::COUNT * (int)sizeof...(Parts);
    const int64_t blocks = row_or_piece_grid<WPB, PER_NODE>(p.num_nodes, p.segments ? p.max_segments : 0);
    if (blocks > 0x7fffffffLL) return set_error(E3J_AMD_INVALID_ARGUMENT, "convolution_bwd_bwd: grid too large");
    if (blocks == 0) return E3J_AMD_OK;
    hipLaunchKernelGGL((second_dm_kernel<K, CPL, WPB, MINW, Parts...>), dim3((unsigned)blocks), dim3(kWave, WPB), 0,
                       stream, a.x, a.y, a.s, a.x2, a.y2, a.s2, sender, row_ptr, perm, p.row_order, out, p.num_nodes,
                       p.coef_scale, p.y_flip, p.segments ? p.row_cap : 0,
                       p.row_piece > 0 ? p.row_piece : p.row_cap, p.segments, p.max_segments, p.partials);
    return check_hip(hipGetLastError(), "convolution second-order backward (dm) launch");
}

template <int K, int CPL, int WPB, int MINW, int Y, int X, typename... Parts>
int launch_second_tile(const e3j_amd_conv_params &p, const SecondOperands &a, const int32_t *sender,
                       const int32_t *row_ptr, const int32_t *perm, const e3j_amd_tile_schedule &sch, float *dx,
                       float *dy, float *ds, hipStream_t stream) {
    constexpr int64_t PER_WORK = (int64_t)Slice<K, CPL>::COUNT * sizeof...(Parts);
    const size_t lds = (size_t)tile_row_bytes<CPL, Parts...>() * (size_t)sch.tile_rows;
    int rc = launch_bwd_targets(p, sender, row_ptr, perm, dx, dy, ds, PER_WORK > 1, stream);
    if (rc) return rc;
    const int64_t blocks = padded_grid((int64_t)sch.num_work * PER_WORK);
    if (blocks > 0x7fffffffLL) return set_error(E3J_AMD_INVALID_ARGUMENT, "convolution_bwd_bwd: grid too large");
    if (blocks == 0) return E3J_AMD_OK;
    auto kernel = second_tile_kernel<K, CPL, WPB, MINW, Parts...>;
    rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxTileLds),
                   "hipFuncSetAttribute(second_tile)");
    if (rc) return rc;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kWave, WPB), lds, stream, a.x, a.y, a.s, a.x2, a.y2,
                       a.s2, a.dm, sch.work, sch.sender, sch.edge, sch.local, p.row_order, dx, dy, ds, p.num_nodes,
                       sch.tile_rows, sch.num_work, p.coef_scale, p.y_flip);
    return check_hip(hipGetLastError(), "convolution second-order backward (tiles) launch");
}

}  // namespace e3j_amd
#endif
