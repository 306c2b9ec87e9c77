// Row regrouping around the per-degree channel mixing that follows a convolution.
//
// A convolution writes node rows (N, Z, K): for every output degree l its `mul` copies of 2l + 1
// components, rows base_l + u * dim_l + m.  The linear layer after it mixes copies and channels
// per degree, x'[n, m, c] = sum_{u, k} out[n, base_l + u * dim_l + m, k] W_l[u, k, c]: one plain
// matrix product per degree once the rows are regrouped as A_l[(n, m), (u, k)].  The kernel below
// moves every row of K values between the two arrangements in one launch, in whole 16-byte
// pieces, driven by two numbers per row: regrouped address of (n, i, k) = row_base[i] +
// n * row_stride[i] + k.  The products themselves are library matrix products (the one dense
// contraction of this step; src/e3j/core/linear.py of the reference does the same with an einsum).
// The backward pass uses the same kernel in the other direction, so the cotangent rows are
// written once (no zero fill, no additions of per-degree slices).
#include "common.h"
#include "split_bf16.h"

namespace e3j_amd {
namespace {

// VEC: elements per 16-byte piece
template <typename T, int VEC, bool kGather>
__global__ void rows_regroup_kernel(const T *__restrict__ src, T *__restrict__ dst, int64_t num_nodes,
                                    int32_t rows, int32_t channels, const int64_t *__restrict__ row_base,
                                    const int64_t *__restrict__ row_stride) {
    struct alignas(16) Piece { T v[VEC]; };
    const int32_t pieces = channels / VEC;
    const int64_t total = num_nodes * rows * pieces;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += stride) {
        const int32_t q = (int32_t)(t % pieces);
        const int64_t row = t / pieces;  // n * rows + i
        const int32_t i = (int32_t)(row % rows);
        const int64_t n = row / rows;
        const int64_t plain = row * channels + (int64_t)q * VEC;
        const int64_t grouped = row_base[i] + n * row_stride[i] + (int64_t)q * VEC;
        if (kGather)   // plain (N, rows, K) -> regrouped
            *reinterpret_cast<Piece *>(dst + grouped) = *reinterpret_cast<const Piece *>(src + plain);
        else           // regrouped -> plain
            *reinterpret_cast<Piece *>(dst + plain) = *reinterpret_cast<const Piece *>(src + grouped);
    }
}

template <typename T>
int launch(const void *src, void *dst, int64_t num_nodes, int32_t rows, int32_t channels,
           const int64_t *row_base, const int64_t *row_stride, bool gather, hipStream_t stream) {
    constexpr int VEC = 16 / sizeof(T);
    const int64_t total = num_nodes * rows * (channels / VEC);
    const unsigned blocks = (unsigned)std::min<int64_t>((total + 255) / 256, 1 << 20);
    if (gather)
        hipLaunchKernelGGL((rows_regroup_kernel<T, VEC, true>), dim3(blocks), dim3(256), 0, stream,
                           static_cast<const T *>(src), static_cast<T *>(dst), num_nodes, rows, channels, row_base,
                           row_stride);
    else
        hipLaunchKernelGGL((rows_regroup_kernel<T, VEC, false>), dim3(blocks), dim3(256), 0, stream,
                           static_cast<const T *>(src), static_cast<T *>(dst), num_nodes, rows, channels, row_base,
                           row_stride);
    return check_hip(hipGetLastError(), "rows_regroup launch");
}

// ---------------------------------------------------------------------------
// The mixing itself in one launch (float32, 64 or 128 channels): no regrouped copies, no library
// calls.  A wave takes 32 nodes and one output row (degree l, component m) and runs
// v_mfma_f32_32x32x16_bf16 with the nodes as rows on operands split three ways (see split_bf16.h): lane t holds, for
// node t % 32, the 32 consecutive channels 32 (t / 32) .. + 31 of a source row (the row of a node is read by
// sixteen lanes side by side and turned through LDS; with a lane reading its own 128 bytes every access touched 64
// lines, which the first-level cache does not hold until the next one), and step s of the product takes
// channels 32 (t / 32) + 8 s .. + 7 from every lane; the second operand is the matching piece of a weight column.
// The waves of a block work on one output row and share its weights through LDS, 64 summed channels (a chunk) at a
// time, each wave splitting a fourth of the columns.  A tile with a value that does not split (an infinity, a NaN, bits
// below the smallest bfloat16) is summed again on v_mfma_f32_32x32x2_f32 from memory, behind everything else: as a
// branch in each chunk it took the registers that the loads on their way need (200 bytes of scratch at 128 channels).
// For the same reason the loads past the last chunk read it again instead of being left out.
// Forward: the products of the mul copies of the degree accumulate into one output row.  Backward (weights
// transposed by the caller): the cotangent row is read once and gives one product per copy.
// At 128 channels a block of the backward makes 64 output channels: the operand of both chunks of a row stays in
// registers, and the cotangent rows that are read twice are few.  A forward block makes all.
// A chunk is summed by itself (see split_bf16.h): error against float64 over normal values, rms, 64 channels 3.0e-7 -> 0.7e-7
// forward and 1.1e-7 -> 0.5e-7 backward, 128 channels 4.3e-7 -> 0.8e-7 and 1.6e-7 -> 0.5e-7, for 2 to 5 % of the time.
// Bound by the stream and, in a block's chain of chunks, by latency: 99 rows to 16, 6 000 nodes, 64 channels: 55 -> 44 us
// forward and 63 -> 37 backward where float32 products took 32 and the stream takes 35; 128 channels 225 -> 156 and
// 231 -> 127 (stream 70), 20 000 nodes 569 -> 459 and 578 -> 427, 200 nodes 66 -> 63 and 68 -> 29 (64 channels
// there: 21 -> 21 and 22 -> 16).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kMixDegrees = 8;
constexpr int kMixWaves = 4;  // waves per block, 32 nodes each, on one output row
struct MixShape {
    int32_t degrees;
    int32_t mul[kMixDegrees], dim[kMixDegrees];
};

template <int K, bool kTranspose>
__global__ __launch_bounds__(256, K == 64 ? 3 : 2) void channel_mix_kernel(
    const float *__restrict__ src, float *__restrict__ dst, const float *__restrict__ w, int64_t num_nodes,
    MixShape shape, uint32_t plain_stride, uint32_t mixed_stride) {
    // chunks of 64 summed channels, output channels of a block, tiles of 32 of them
    constexpr int KC = K / 64, KO = kTranspose ? 64 : K, KT = KO / 32;
    const int lane = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.y), r = lane & 31, h = lane >> 5;
    constexpr int ROWS = KO / 16;              // weights: a thread stages ROWS rows of four columns,
    constexpr int GROUPS = KO / kMixWaves / 4;  //   GROUPS lanes side by side the columns of their wave
    constexpr int WEIGHT_PITCH = 64 + 8;       // bfloat16 values a column (16-byte reads of 32 columns spread over the banks)
    constexpr int PITCH = 32 + 4;              // (16-byte reads of 64 rows side by side spread over the banks)
    __shared__ __attribute__((aligned(16))) uint16_t weights[3][KO * WEIGHT_PITCH];
    __shared__ __attribute__((aligned(16))) float rows[kMixWaves][32 * PITCH];
    __shared__ int odd_weights;                // set for good by a chunk whose weights do not split
    // (the waves of a block take neighbouring tiles of one output row; tiles past the last one run along)
    const int64_t row_blocks = (num_nodes + 32 * kMixWaves - 1) / (32 * kMixWaves);
    const int64_t block = blockIdx.x / (K / KO);
    const int64_t tile = block % row_blocks * kMixWaves + wave;
    const int xr = (int)(block / row_blocks), out0 = blockIdx.x % (K / KO) * KO;
    // first node of the tile and how many it has (none or fewer: tiles past the last one)
    const int64_t node0 = tile * 32;
    const int nodes = (int)(num_nodes - node0 < 0 ? 0 : num_nodes - node0 < 32 ? num_nodes - node0 : 32);
    // `count` values of a row of each of the tile's nodes, as a buffer: loads past the last node are zeros, stores
    // past it are dropped, an address is one register
    auto tile_rows = [&](const float *first, uint32_t node_stride, int count) {
        const uint32_t bytes = nodes > 0 ? ((uint32_t)(nodes - 1) * node_stride + count) * 4u : 0u;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(first) + node0 * node_stride, 0, bytes, 0x00020000);
    };
    // the degree and component of mixed row xr, the first plain row and the first weight of the degree
    int l = 0, zbase = 0, xbase = 0;
    int64_t wbase = 0;
    while (l < shape.degrees - 1 && xr >= xbase + shape.dim[l]) {
        zbase += shape.mul[l] * shape.dim[l];
        xbase += shape.dim[l];
        wbase += (int64_t)shape.mul[l] * K * K;
        l++;
    }
    const int m = xr - xbase, mul = shape.mul[l], dim = shape.dim[l];
    // 64 channels of a row of the wave's 32 nodes, from `first` (row of node 0) on: read in whole lines,
    // sixteen lanes a node, and turned through LDS into the operand a lane supplies
    auto fetch_rows = [&](const float *first, uint32_t node_stride, f32x4 (&piece)[8]) {
        const auto buffer = tile_rows(first, node_stride, 64);
        uint32_t at = (lane / 16 * node_stride + lane % 16 * 4) * 4u;
        asm volatile("" : "+v"(at));  // (the eight addresses are made where they are used, not kept)
#pragma unroll
        for (int i = 0; i < 8; i++)
            piece[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                buffer, at + 16 * i * node_stride, 0, 0));
    };
    // returns whether there is a value that does not split
    auto turn_rows = [&](const f32x4 (&piece)[8], Split3 (&a)[4]) {
        float *mine = rows[wave];
        uint32_t lost = 0;
#pragma unroll
        for (int half = 0; half < 2; half++) {  // sixteen channels of each lane half at a time: 18 KB a block, not 35
            if (lane / 4 % 2 == half) {
#pragma unroll
                for (int i = 0; i < 8; i++)
                    *reinterpret_cast<f32x4 *>(mine + (4 * i + lane / 16) * PITCH + lane / 8 % 2 * 16 + lane % 4 * 4) = piece[i];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 2; q++) {
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; j += 4) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(mine + r * PITCH + 16 * h + 8 * q + j);
                    x[j] = v.x; x[j + 1] = v.y; x[j + 2] = v.z; x[j + 3] = v.w;
                }
                a[2 * half + q] = split3_nearest(x, lost);
                asm volatile("" : "+v"(lost));  // (one value is kept, not those that it was made of)
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        return __any(lost != 0) != 0;
    };
    auto store_tile = [&](const f32x16 (&acc)[KT], float *row0, uint32_t node_stride) {
        const auto buffer = tile_rows(row0 + out0, node_stride, KO);
        // register v of lane t: node 8 (v / 4) + 4 (t / 32) + v % 4 of the tile, output channel t % 32 of tile ct
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const uint32_t at = ((8 * (v / 4) + 4 * h + v % 4) * node_stride + r) * 4u;
#pragma unroll
            for (int ct = 0; ct < KT; ct++)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[ct][v]), buffer, at + ct * 128, 0, 0);
        }
    };
    f32x16 acc[KT];
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto clear = [&]() {
#pragma unroll
        for (int ct = 0; ct < KT; ct++) acc[ct] = zero;
    };
    // One chunk of 64 summed channels: its weight rows lie in LDS for the waves of the block, those of
    // the next chunk are on their way while the products of this one run.
    const float *wl = w + wbase + out0;
    const int chunks = mul * KC;
    const int col0 = wave * (KO / kMixWaves) + lane % GROUPS * 4, k0 = lane / GROUPS * ROWS;
    f32x4 staged[ROWS];
    auto fetch = [&](int q) {
        const auto buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(wl) + (int64_t)q * (64 * K), 0,
                                                              (63 * K + KO) * 4, 0x00020000);
#pragma unroll
        for (int i = 0; i < ROWS; i++)
            staged[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                buffer, ((k0 + i) * K + col0) * 4, 0, 0));
    };
    typedef uint32_t Pairs __attribute__((ext_vector_type(ROWS / 2)));  // ROWS bfloat16 values
    struct Weights {
        Pairs term[3][4];
        uint32_t lost;
    };
    auto split_weights = [&]() {
        Weights out;
        out.lost = 0;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            float rest[ROWS];
#pragma unroll
            for (int i = 0; i < ROWS; i++) rest[i] = staged[i][c];
#pragma unroll
            for (int u = 0; u < 3; u++)
#pragma unroll
                for (int i = 0; i < ROWS; i += 2) out.term[u][c][i / 2] = take_nearest(rest[i], rest[i + 1]);  // see split3_nearest
#pragma unroll
            for (int i = 0; i < ROWS; i++) out.lost |= __float_as_uint(rest[i]);
            asm volatile("" : "+v"(out.lost));
            __builtin_amdgcn_sched_barrier(0);
        }
        return out;
    };
    auto commit = [&](const Weights &split) {
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int u = 0; u < 3; u++)
                *reinterpret_cast<Pairs *>(&weights[u][(col0 + c) * WEIGHT_PITCH + k0]) = split.term[u][c];
        if (split.lost != 0) odd_weights = 1;
    };
    auto products = [&](const Split3 (&a)[4]) {
        constexpr int TILES = 2;
#pragma unroll
        for (int c0 = 0; c0 < KT; c0 += TILES) {
            f32x16 chunk[TILES];  // (summed by itself, the small products first: see split_bf16.h)
#pragma unroll
            for (int i = 0; i < TILES; i++) chunk[i] = zero;
            auto piece_of = [&](int i, int u, int s) {
                return *reinterpret_cast<const bf16x8 *>(&weights[u][((c0 + i) * 32 + r) * WEIGHT_PITCH + 32 * h + 8 * s]);
            };
#pragma unroll
            for (int s = 0; s < 4; s++) {
                bf16x8 b[TILES][3];
#pragma unroll
                for (int i = 0; i < TILES; i++)
#pragma unroll
                    for (int u = 0; u < 3; u++) b[i][u] = piece_of(i, u, s);
#pragma unroll
                for (int u = 0; u < 5; u++)
#pragma unroll
                    for (int i = 0; i < TILES; i++)
                        chunk[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s].term[kPairs[u][0]], b[i][kPairs[u][1]],
                                                                           chunk[i], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);  // (the operands of one step at a time in registers)
            }
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int i = 0; i < TILES; i++)
                    chunk[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s].term[0], piece_of(i, 0, s), chunk[i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < TILES; i++) acc[c0 + i] += chunk[i];
        }
    };
    // chunk `q` of the weights in float32; `first`, node_stride: its source rows
    auto plain_products = [&](const float *first, uint32_t node_stride, int q) {
        const auto buffer = tile_rows(first, node_stride, 64);
        const float *wk = wl + ((int64_t)q * 64 + 32 * h) * K + r;
#pragma unroll 1
        for (int s = 0; s < 32; s++) {
            const float x = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                buffer, (r * node_stride + 32 * h + s) * 4u, 0, 0));
#pragma unroll
            for (int ct = 0; ct < KT; ct++)
                acc[ct] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, wk[s * K + ct * 32], acc[ct], 0, 0, 0);
        }
    };
    // after the products of a chunk: its weights make room for those of the next
    auto next_chunk = [&](int q) {
        if (q < chunks) {
            const Weights split = split_weights();
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            commit(split);
        }
        __syncthreads();
    };
    if (lane + wave == 0) odd_weights = 0;
    fetch(0);
    __syncthreads();
    commit(split_weights());
    f32x4 piece[8];
    if (!kTranspose) {
        clear();
        // the source row of the next chunk is read while the products of the one at hand run
        auto row_of = [&](int q) { return src + (int64_t)(zbase + q / KC * dim + m) * K + q % KC * 64; };
        fetch_rows(row_of(0), plain_stride, piece);
        __syncthreads();
        bool odd = false;
        for (int q = 0; q < chunks; q++) {
            Split3 a[4];
            odd |= turn_rows(piece, a);
            __builtin_amdgcn_sched_barrier(0);
            const int next = min(q + 1, chunks - 1);  // (past the last chunk: it again)
            fetch(next);
            fetch_rows(row_of(next), plain_stride, piece);
            products(a);
            next_chunk(q + 1);
        }
        if (odd || odd_weights != 0) {
            clear();
            for (int q = 0; q < chunks; q++) plain_products(row_of(q), plain_stride, q);
        }
        store_tile(acc, dst + (int64_t)xr * K, mixed_stride);
    } else {
        Split3 a[KC][4];
        bool odd = false;
#pragma unroll
        for (int kc = 0; kc < KC; kc++) {
            fetch_rows(src + (int64_t)xr * K + kc * 64, mixed_stride, piece);
            odd |= turn_rows(piece, a[kc]);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        for (int u = 0; u < mul; u++) {
            clear();
#pragma unroll
            for (int kc = 0; kc < KC; kc++) {
                const int q = u * KC + kc;
                fetch(min(q + 1, chunks - 1));
                products(a[kc]);
                next_chunk(q + 1);
            }
            store_tile(acc, dst + (int64_t)(zbase + u * dim + m) * K, plain_stride);
        }
        if (odd || odd_weights != 0) {
            __threadfence();  // (these stores come after those)
            for (int u = 0; u < mul; u++) {
                clear();
#pragma unroll 1
                for (int kc = 0; kc < KC; kc++) plain_products(src + (int64_t)xr * K + kc * 64, mixed_stride, u * KC + kc);
                store_tile(acc, dst + (int64_t)(zbase + u * dim + m) * K, plain_stride);
            }
        }
    }
}

template <int K>
int launch_mix(const float *src, float *dst, const float *w, int64_t num_nodes, const MixShape &shape,
               int rows_plain, int rows_mixed, bool transpose, hipStream_t stream) {
    const int64_t blocks = (num_nodes + 32 * kMixWaves - 1) / (32 * kMixWaves) * rows_mixed * (transpose ? K / 64 : 1);
    if (blocks > 0x7fffffffLL) return set_error(E3J_AMD_INVALID_ARGUMENT, "channel_mix: too many nodes for one launch");
    const int64_t plain = (int64_t)rows_plain * K, mixed = (int64_t)rows_mixed * K;
    if (num_nodes > 1 && std::max(plain, mixed) > (int64_t)1 << 25) {  // (the nodes of a tile are 32 bits of bytes apart)
        for (int64_t n = 0; n < num_nodes; n++) {
            int rc = launch_mix<K>(src + n * (transpose ? mixed : plain), dst + n * (transpose ? plain : mixed), w, 1, shape,
                                   rows_plain, rows_mixed, transpose, stream);
            if (rc) return rc;
        }
        return E3J_AMD_OK;
    }
    // (of one node no stride is used but to tell the nodes that are not there: one row apart will do)
    const uint32_t plain_stride = num_nodes > 1 ? (uint32_t)plain : K, mixed_stride = num_nodes > 1 ? (uint32_t)mixed : K;
    if (transpose)
        hipLaunchKernelGGL((channel_mix_kernel<K, true>), dim3((unsigned)blocks), dim3(kWave, kMixWaves), 0, stream,
                           src, dst, w, num_nodes, shape, plain_stride, mixed_stride);
    else
        hipLaunchKernelGGL((channel_mix_kernel<K, false>), dim3((unsigned)blocks), dim3(kWave, kMixWaves), 0, stream,
                           src, dst, w, num_nodes, shape, plain_stride, mixed_stride);
    return check_hip(hipGetLastError(), "channel_mix launch");
}

}  // namespace
}  // namespace e3j_amd

extern "C" int e3j_amd_channel_mix(const void *src, void *dst, const void *weights, int64_t num_nodes,
                                   int32_t channels, int32_t num_degrees, const int32_t *mul, const int32_t *dim,
                                   int32_t transpose, void *stream) {
    using namespace e3j_amd;
    if (num_nodes < 0 || num_degrees < 1 || num_degrees > kMixDegrees || mul == nullptr || dim == nullptr)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "channel_mix: 1 to 8 degrees, their multiplicities and dimensions");
    if (channels != 64 && channels != 128)
        return set_error(E3J_AMD_UNIMPLEMENTED, "channel_mix: 64 or 128 channels (other counts: e3j_amd_rows_regroup "
                                                "around matrix products)");
    MixShape shape;
    shape.degrees = num_degrees;
    int rows_plain = 0, rows_mixed = 0;
    for (int l = 0; l < kMixDegrees; l++) {
        shape.mul[l] = l < num_degrees ? mul[l] : 0;
        shape.dim[l] = l < num_degrees ? dim[l] : 0;
        if (l < num_degrees && (mul[l] < 1 || dim[l] < 1))
            return set_error(E3J_AMD_INVALID_ARGUMENT, "channel_mix: multiplicities and dimensions must be >= 1");
        rows_plain += shape.mul[l] * shape.dim[l];
        rows_mixed += shape.dim[l];
    }
    if (num_nodes == 0) return E3J_AMD_OK;
    if (src == nullptr || dst == nullptr || weights == nullptr)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "channel_mix: null operand");
    if (reinterpret_cast<uintptr_t>(src) % 16 != 0 || reinterpret_cast<uintptr_t>(dst) % 16 != 0 ||
        reinterpret_cast<uintptr_t>(weights) % 16 != 0)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "channel_mix: operands must be 16-byte aligned");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const float *a = static_cast<const float *>(src), *wt = static_cast<const float *>(weights);
    float *out = static_cast<float *>(dst);
    if (channels == 64) return launch_mix<64>(a, out, wt, num_nodes, shape, rows_plain, rows_mixed, transpose != 0, s);
    return launch_mix<128>(a, out, wt, num_nodes, shape, rows_plain, rows_mixed, transpose != 0, s);
}

extern "C" int e3j_amd_rows_regroup(const void *src, void *dst, int64_t num_nodes, int32_t rows, int32_t channels,
                                    const int64_t *row_base, const int64_t *row_stride, int32_t to_plain,
                                    int32_t val_dtype, void *stream) {
    using namespace e3j_amd;
    if (num_nodes < 0 || rows < 0 || channels < 0)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "rows_regroup: negative size");
    if (num_nodes == 0 || rows == 0 || channels == 0) return E3J_AMD_OK;
    if (src == nullptr || dst == nullptr || row_base == nullptr || row_stride == nullptr)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "rows_regroup: null operand");
    const int vec = val_dtype == E3J_AMD_F64 ? 2 : 4;
    if (val_dtype != E3J_AMD_F32 && val_dtype != E3J_AMD_F64)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "rows_regroup: unsupported value dtype");
    if (channels % vec != 0 || reinterpret_cast<uintptr_t>(src) % 16 != 0 || reinterpret_cast<uintptr_t>(dst) % 16 != 0)
        return set_error(E3J_AMD_INVALID_ARGUMENT,
                         "rows_regroup: rows are moved in 16-byte pieces (channels a multiple of 4 floats / 2 "
                         "doubles, 16-byte aligned operands, row_base and row_stride multiples of that)");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (val_dtype == E3J_AMD_F32)
        return launch<float>(src, dst, num_nodes, rows, channels, row_base, row_stride, to_plain == 0, s);
    return launch<double>(src, dst, num_nodes, rows, channels, row_base, row_stride, to_plain == 0, s);
}
