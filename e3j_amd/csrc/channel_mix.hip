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
// v_mfma_f32_32x32x2_f32 with the nodes as rows: lane t holds, for node t % 32, the 32 consecutive
// channels 32 (t / 32) .. + 31 of a source row (the row of a node is read by sixteen lanes side by
// side and turned through LDS; with a lane reading its own 128 bytes every access touched 64 lines,
// which the first-level cache does not hold until the next one), and step s of the product takes
// channel 32 (t / 32) + s from every lane, which is the layout of the instruction's first operand when
// its two summed indices are read as "channel s of the lower / of the upper half"; the second operand is
// the matching row of the weight, 32 consecutive output channels per half wave.  The waves of a block
// work on one output row and share its weights through LDS, 64 summed channels at a time (with every
// wave reading them from the caches a chunk's 64 loads and its products took turns).
// 6 000 nodes, 64 channels, 99 rows to 16: 85 -> 60 us each way; the products alone take 32 us at the
// float32 rate of the matrix cores, the stream 35 us.  At 128 channels a block takes 68 KB of LDS (two blocks a
// compute unit) and up to 240 registers: 6 000 nodes 287 -> 227 us forward and 282 -> 237 backward, 20 000 nodes
// 846 -> 568 and 935 -> 587, 200 nodes 122 -> 72 and 120 -> 71; the products alone take 128 us at 6 000.  Forward: the products of the mul copies of the
// degree accumulate into one output row.  Backward (weights transposed by the caller): the cotangent row
// is read once and gives one product per copy.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kMixDegrees = 8;
constexpr int kMixWaves = 4;  // waves per block, 32 nodes each, on one output row
struct MixShape {
    int32_t degrees;
    int32_t mul[kMixDegrees], dim[kMixDegrees];
};

template <int K, bool kTranspose>
__global__ __launch_bounds__(256) void channel_mix_kernel(const float *__restrict__ src, float *__restrict__ dst,
                                                          const float *__restrict__ w, int64_t num_nodes,
                                                          MixShape shape, int32_t rows_plain, int32_t rows_mixed) {
    constexpr int KC = K / 64, KT = K / 32;   // chunks of 64 summed channels, tiles of 32 output channels
    const int lane = threadIdx.x, r = lane & 31, h = lane >> 5;
    constexpr int THREADS = kWave * kMixWaves, PIECES = 64 * K / 4 / THREADS;
    constexpr int HALF = 32 * K + 32;  // (the halves of a wave read rows 32 apart: the pad puts them on other banks)
    constexpr int PITCH = 64 + 4;              // (16-byte reads of 64 rows side by side spread over the banks)
    __shared__ __attribute__((aligned(16))) float weights[2 * HALF];
    __shared__ __attribute__((aligned(16))) float rows[kMixWaves][32 * PITCH];
    const int tid = threadIdx.y * kWave + lane;
    // (the waves of a block take neighbouring tiles of one output row; tiles past the last one run along)
    const int64_t row_blocks = (num_nodes + 32 * kMixWaves - 1) / (32 * kMixWaves);
    const int64_t tile = (int64_t)blockIdx.x % row_blocks * kMixWaves + threadIdx.y;
    const int xr = (int)(blockIdx.x / row_blocks);
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
    auto fetch_rows = [&](const float *first, int64_t node_stride, f32x4 (&piece)[8]) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int64_t n = tile * 32 + 4 * i + lane / 16;  // (past the end: the last node)
            piece[i] = *reinterpret_cast<const f32x4 *>(first + (n < num_nodes ? n : num_nodes - 1) * node_stride +
                                                        lane % 16 * 4);
        }
    };
    auto turn_rows = [&](const f32x4 (&piece)[8], float (&a)[32]) {
        float *mine = rows[threadIdx.y];
#pragma unroll
        for (int i = 0; i < 8; i++)
            *reinterpret_cast<f32x4 *>(mine + (4 * i + lane / 16) * PITCH + lane % 16 * 4) = piece[i];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const f32x4 v = *reinterpret_cast<const f32x4 *>(mine + r * PITCH + 32 * h + 4 * q);
            a[4 * q] = v.x; a[4 * q + 1] = v.y; a[4 * q + 2] = v.z; a[4 * q + 3] = v.w;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto store_tile = [&](const f32x16 (&acc)[KT], float *row0, int64_t node_stride) {
        // register v of lane t: node 8 (v / 4) + 4 (t / 32) + v % 4 of the tile, output channel t % 32 of tile ct
#pragma unroll
        for (int ct = 0; ct < KT; ct++) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int64_t n = tile * 32 + 8 * (v / 4) + 4 * h + v % 4;
                if (n < num_nodes) row0[n * node_stride + ct * 32 + r] = acc[ct][v];
            }
        }
    };
    f32x16 acc[KT];
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // One chunk of 64 summed channels: its weight rows lie in LDS for the waves of the block, those of
    // the next chunk are on their way while the products of this one run.
    const float *wl = w + wbase;
    const int chunks = mul * KC;
    f32x4 staged[PIECES];
    auto fetch = [&](int q) {
#pragma unroll
        for (int i = 0; i < PIECES; i++)
            staged[i] = *reinterpret_cast<const f32x4 *>(wl + (int64_t)q * (64 * K) + (i * THREADS + tid) * 4);
    };
    auto commit = [&]() {
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
            const int at = (i * THREADS + tid) * 4;
            *reinterpret_cast<f32x4 *>(&weights[at + (at >= 32 * K ? 32 : 0)]) = staged[i];
        }
    };
    auto products = [&](const float (&a)[32]) {
        const float *wk = &weights[h * HALF + r];
#pragma unroll
        for (int s = 0; s < 32; s++) {
#pragma unroll
            for (int ct = 0; ct < KT; ct++)
                acc[ct] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], wk[s * K + ct * 32], acc[ct], 0, 0, 0);
        }
    };
    // after the products of a chunk: its weights make room for those of the next
    auto next_chunk = [&](int q) {
        __syncthreads();
        if (q < chunks) commit();
        __syncthreads();
    };
    fetch(0);
    commit();
    const int64_t plain_stride = (int64_t)rows_plain * K, mixed_stride = (int64_t)rows_mixed * K;
    f32x4 piece[8];
    if (!kTranspose) {
#pragma unroll
        for (int ct = 0; ct < KT; ct++) acc[ct] = zero;
        // the source row of the next chunk is read while the products of the one at hand run
        auto row_of = [&](int q) { return src + (int64_t)(zbase + q / KC * dim + m) * K + q % KC * 64; };
        fetch_rows(row_of(0), plain_stride, piece);
        __syncthreads();
        for (int q = 0; q < chunks; q++) {
            float a[32];
            turn_rows(piece, a);
            if (q + 1 < chunks) {
                fetch(q + 1);
                fetch_rows(row_of(q + 1), plain_stride, piece);
            }
            products(a);
            next_chunk(q + 1);
        }
        store_tile(acc, dst + (int64_t)xr * K, mixed_stride);
    } else {
        float a[KC][32];
#pragma unroll
        for (int kc = 0; kc < KC; kc++) {
            fetch_rows(src + (int64_t)xr * K + kc * 64, mixed_stride, piece);
            turn_rows(piece, a[kc]);
        }
        __syncthreads();
        for (int u = 0; u < mul; u++) {
#pragma unroll
            for (int ct = 0; ct < KT; ct++) acc[ct] = zero;
#pragma unroll
            for (int kc = 0; kc < KC; kc++) {
                const int q = u * KC + kc;
                if (q + 1 < chunks) fetch(q + 1);
                products(a[kc]);
                next_chunk(q + 1);
            }
            store_tile(acc, dst + (int64_t)(zbase + u * dim + m) * K, plain_stride);
        }
    }
}

template <int K>
int launch_mix(const float *src, float *dst, const float *w, int64_t num_nodes, const MixShape &shape,
               int rows_plain, int rows_mixed, bool transpose, hipStream_t stream) {
    const int64_t blocks = (num_nodes + 32 * kMixWaves - 1) / (32 * kMixWaves) * rows_mixed;
    if (blocks > 0x7fffffffLL) return set_error(E3J_AMD_INVALID_ARGUMENT, "channel_mix: too many nodes for one launch");
    if (transpose)
        hipLaunchKernelGGL((channel_mix_kernel<K, true>), dim3((unsigned)blocks), dim3(kWave, kMixWaves), 0, stream,
                           src, dst, w, num_nodes, shape, rows_plain, rows_mixed);
    else
        hipLaunchKernelGGL((channel_mix_kernel<K, false>), dim3((unsigned)blocks), dim3(kWave, kMixWaves), 0, stream,
                           src, dst, w, num_nodes, shape, rows_plain, rows_mixed);
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
