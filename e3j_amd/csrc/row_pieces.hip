// Long rows of the forward pass, summed in a fixed order.  The pieces of a row longer than
// row_cap are summed by waves of their own, in the launch that sums the rows.  Instead of adding them
// to the output row with float atomics, whose order changes from run to run, every piece stores its
// sum in a row of a scratch array, and a second kernel adds the rows of a receiver's pieces to its
// output row in the order of their positions.  No counterpart
// in the reference, whose forward kernel walks the edges of a receiver one after another in one
// block (lib/e3j_ops/cuda/convolution/fwd.cuh:346-363) and is run-to-run reproducible for that
// reason (tests/test_ops/test_convolution_op.py:322-342); this keeps that property while sharing the row.

#include "row_pieces.h"

#include <algorithm>

#include "common.h"

namespace e3j_amd {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Block (g, chunk) walks the pieces g, g + gridDim.x, ...: where a piece is the first listed piece of
// its row, the rows of all pieces of that row are added to 256 floats of the output row.  A row of few
// pieces is summed by a thread per float, piece after piece (most hub rows have one or two pieces: 500 of
// them cost 15 us, with a wave per quarter of the pieces and 64 floats at a time 23 us).  Of a
// longer one the four waves of the block each sum a quarter of the pieces (contiguous ranges, sixteen
// loads in flight), one after another in list order; the four sums are then added in order.  The grouping
// is fixed by the list, so are the bits.  (The grid does not grow with the bound on the number of pieces:
// most graphs have none, and a launch of a block per possible piece and chunk would cost more than the
// sums.)
constexpr int kCombineWaves = 4;
constexpr int kCombineThreads = kWave * kCombineWaves;
constexpr int kCombineStride = 256;
constexpr int kFewPieces = 8;
__global__ __launch_bounds__(kCombineThreads) void combine_pieces_kernel(
    const int32_t *__restrict__ segments, const int32_t *__restrict__ row_ptr, int max_segments, int row_piece,
    int64_t row_floats, const float *__restrict__ partials, float *__restrict__ out) {
    __shared__ float sums[kCombineWaves][kWave];
    __shared__ int found[kCombineThreads][3], num_found;
    const int count = min(segments[0], max_segments);
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int64_t chunk = (int64_t)blockIdx.y * kCombineThreads;
    // the pieces g, g + gridDim.x, ... of this block, a thread each: which of them begin a row's run
    for (int base = blockIdx.x; base < count; base += gridDim.x * blockDim.x) {
        if (threadIdx.x == 0) num_found = 0;
        __syncthreads();
        const int q = base + (int)threadIdx.x * (int)gridDim.x;
        if (q < count) {
            const int r = segments[4 + 3 * q], b = segments[5 + 3 * q];
            const int begin = row_ptr[r], end = row_ptr[r + 1];
            if (b == begin + row_piece) {  // the first listed piece of row r
                const int at = atomicAdd(&num_found, 1);
                found[at][0] = q;
                found[at][1] = min((end - begin - 1) / row_piece, count - q);
                found[at][2] = r;
            }
        }
        __syncthreads();
        const int n = num_found;
        for (int f = 0; f < n; f++) {
            const int first_piece = found[f][0], pieces = found[f][1];
            float *row = out + (int64_t)found[f][2] * row_floats;
            if (pieces <= kFewPieces) {
                const int64_t t = chunk + threadIdx.x;
                if (t < row_floats) {
                    float sum = 0.f;
                    for (int k = first_piece; k < first_piece + pieces; k++) sum += partials[(int64_t)k * row_floats + t];
                    row[t] += sum;
                }
                continue;
            }
            const int first = first_piece + (int)((int64_t)pieces * wave / kCombineWaves);
            const int end = first_piece + (int)((int64_t)pieces * (wave + 1) / kCombineWaves);
            for (int64_t t0 = chunk; t0 < chunk + kCombineThreads && t0 < row_floats; t0 += kWave) {
                const int64_t t = t0 + lane;
                const bool inside = t < row_floats;
                const int64_t tt = inside ? t : 0;
                float sum = 0.f;
                int k = first;
                for (; k + 16 <= end; k += 16) {
                    float v[16];
#pragma unroll
                    for (int u = 0; u < 16; u++) v[u] = partials[(int64_t)(k + u) * row_floats + tt];
#pragma unroll
                    for (int u = 0; u < 16; u++) sum += v[u];
                }
                for (; k < end; k++) sum += partials[(int64_t)k * row_floats + tt];
                sums[wave][lane] = sum;
                __syncthreads();
                if (wave == 0 && inside) {
                    float total = row[t];
#pragma unroll
                    for (int w = 0; w < kCombineWaves; w++) total += sums[w][lane];
                    row[t] = total;
                }
                __syncthreads();  // `sums` is free for the next floats
            }
        }
        __syncthreads();  // `found` is free for the next pieces
    }
}

}  // namespace

size_t row_partials_bytes(int64_t max_segments, int64_t row_floats) {
    if (max_segments <= 0 || row_floats <= 0) return 0;
    return sizeof(float) * (size_t)max_segments * (size_t)row_floats;
}

int launch_combine_pieces(const int32_t *segments, const int32_t *row_ptr, int32_t max_segments, int32_t row_piece,
                          int64_t row_floats, const float *partials, float *out, hipStream_t stream) {
    if (max_segments <= 0) return E3J_AMD_OK;
    const int64_t chunks = (row_floats + kCombineThreads - 1) / kCombineThreads;
    if (chunks > 65535) return set_error(E3J_AMD_INVALID_ARGUMENT, "row pieces: output row too long");
    hipLaunchKernelGGL(combine_pieces_kernel, dim3((unsigned)std::min(max_segments, kCombineStride), (unsigned)chunks),
                       dim3(kCombineThreads), 0, stream, segments, row_ptr, max_segments, row_piece, row_floats,
                       partials, out);
    return check_hip(hipGetLastError(), "row pieces: combine");
}

}  // namespace e3j_amd
