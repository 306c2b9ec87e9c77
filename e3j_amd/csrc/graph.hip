// Graph preparation on the device: CSR row pointers and the stable edge sort
// behind the unsorted (GraphOrdering NONE) path and the transposed adjacency.
//
// Restates GraphCSR (src/e3j/data/graph.py:49-73): row_ptr = [0] +
// cumsum(bincount(key, length = N)) with out-of-range keys dropped, and
// sort = stable argsort by key.  The sort is rocPRIM's radix sort (via hipCUB)
// on unsigned keys, so sentinel and negative keys land after every live row.

#include <hipcub/hipcub.hpp>

#include <mutex>

#include "common.h"

namespace e3j_amd {
namespace {

// Histogram of the in-range keys into counts[key + 1].  A thread walks a short run of
// consecutive positions and issues one atomic per run of equal keys: sorted keys (the
// common case) then cost one atomic per thread instead of one per edge on a hot address.
constexpr int kCountChunk = 16;
__global__ void count_keys_kernel(const int32_t *__restrict__ key, int64_t num_edges, int num_nodes,
                                  int32_t *__restrict__ counts) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x * kCountChunk;
    for (int64_t base = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * kCountChunk;
         base < num_edges; base += stride) {
        const int64_t end = base + kCountChunk < num_edges ? base + kCountChunk : num_edges;
        int run_key = key[base], run = 1;
        for (int64_t e = base + 1; e < end; e++) {
            const int k = key[e];
            if (k == run_key) { run++; continue; }
            if ((unsigned)run_key < (unsigned)num_nodes) atomicAdd(&counts[run_key + 1], run);
            run_key = k; run = 1;
        }
        if ((unsigned)run_key < (unsigned)num_nodes) atomicAdd(&counts[run_key + 1], run);
    }
}

__global__ void iota_kernel(int32_t *__restrict__ out, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = (int32_t)i;
}

__global__ void gather_kernel(const int32_t *__restrict__ src, const int32_t *__restrict__ perm,
                              int32_t *__restrict__ dst, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        dst[i] = src[perm[i]];
}

// One sweep of minimum-label propagation over a CSR adjacency:
// next[n] = min(cur[n], cur[m] for every m in row n), no atomics.
// A row is read up to kLabelRowCap positions: the labels only steer which rows run together,
// and a thread that walked a hub's whole row would outlast the rest of the sweep many times.
constexpr int kLabelRowCap = 128;
constexpr int64_t kLabelBlocks = 1 << 20;  // (a launch has fewer than 2^32 threads: past 2^26 rows a thread takes several)
// kLanes: lanes that share a row (its gathers then run that many at a time), see sweep_labels
template <int kLanes>
__global__ void min_label_kernel(const int32_t *__restrict__ other,
                                 const int32_t *__restrict__ row_ptr, int num_nodes,
                                 const int32_t *__restrict__ cur, int32_t *__restrict__ next,
                                 uint32_t *__restrict__ keys, int32_t *__restrict__ vals, int bits) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x, lanes = (int64_t)num_nodes * kLanes;
    // (the lanes of a row go round together: they exchange below)
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < lanes; t += stride) {
        const int n = (int)(t / kLanes), part = (int)(t % kLanes);
        // cur == nullptr: every node still carries its own id (the first sweep)
        int best = cur ? cur[n] : n;
        const int begin = row_ptr[n];
        const int end = min(row_ptr[n + 1], begin + kLabelRowCap);
        for (int e = begin + part; e < end; e += kLanes) {
            const int m = other[e];
            if ((unsigned)m < (unsigned)num_nodes) best = min(best, cur ? cur[m] : m);
        }
#pragma unroll
        for (int off = 1; off < kLanes; off *= 2) best = min(best, __shfl_xor(best, off, kWave));
        if (part != 0) continue;
        if (keys == nullptr) {
            next[n] = best;
        } else {
            // the last of two sweeps: key = (label after it, label before it); one sort lists the coarse
            // clusters and, inside them, the fine ones
            keys[n] = ((uint32_t)best << bits) | (uint32_t)cur[n];
            if (vals != nullptr) vals[n] = n;
        }
    }
}

// Sixteen lanes a row up to 2^14 rows, where a hub's row is what a sweep waits for (5 000 rows of 30 with hubs among
// them: two sweeps 17 -> 10 us); four from there on, where the rows fill the chip and lanes without a position cost
// (the row order of 1M rows of 4 positions 324 us and 395 with sixteen, of 30 positions 394 and 421, of 100 000 rows of
// 16 131 and 136; of 300 000 rows of 120 positions 377 and 346).
void sweep_labels(const int32_t *other, const int32_t *row_ptr, int num_nodes, const int32_t *cur, int32_t *next,
                  uint32_t *keys, int32_t *vals, int bits, hipStream_t stream) {
    const bool few = num_nodes <= 1 << 14;
    const int64_t blocks = std::min<int64_t>(((int64_t)num_nodes * (few ? 16 : 4) + 255) / 256, kLabelBlocks);
    hipLaunchKernelGGL(few ? min_label_kernel<16> : min_label_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, stream, other,
                       row_ptr, num_nodes, cur, next, keys, vals, bits);
}

__global__ void copy_i32_kernel(const int32_t *__restrict__ src, int32_t *__restrict__ dst, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

// Pieces of the rows longer than `cap`, past their first `piece` positions: a row reserves its
// pieces with one atomic on the count (the order of the rows in the list is free).
__device__ __forceinline__ void list_row_pieces(int r, int begin, int end, int cap, int piece, int max_segments,
                                                int32_t *__restrict__ segments) {
    if (end - begin <= cap) return;
    const int extra = (end - begin - 1) / piece;  // pieces after the first
    const int at = atomicAdd(segments, extra);
    for (int k = 0; k < extra && at + k < max_segments; k++) {
        const int b = begin + (k + 1) * piece;
        int32_t *seg = segments + 4 + 3 * (at + k);
        seg[0] = r;
        seg[1] = b;
        seg[2] = b + piece < end ? b + piece : end;
    }
}

__global__ void row_segments_kernel(const int32_t *__restrict__ row_ptr, int num_nodes, int cap, int piece,
                                    int max_segments, int32_t *__restrict__ segments) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= num_nodes) return;
    list_row_pieces(r, row_ptr[r], row_ptr[r + 1], cap, piece, max_segments, segments);
}

// Rows with more than twice the mean number of edges ("long rows"): flag per list position.
__global__ void long_row_flags_kernel(const int32_t *__restrict__ order, const int32_t *__restrict__ row_ptr,
                                      int num_nodes, int32_t *__restrict__ flags, int row_cap, int row_piece,
                                      int max_segments, int32_t *__restrict__ segments) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_nodes) return;
    const int r = order[i], begin = row_ptr[r], end = row_ptr[r + 1];
    flags[i] = (int64_t)(end - begin) * num_nodes > 2 * (int64_t)row_ptr[num_nodes] ? 1 : 0;
    if (segments != nullptr) list_row_pieces(r, begin, end, row_cap, row_piece, max_segments, segments);
}

// The kernels hand one contiguous eighth of the row list to each XCD and every XCD walks its
// eighth front to back.  Long rows started late leave the machine waiting for a few waves at
// the end, so they are dealt to the fronts of the eighths: eighth p takes the p-th eighth of the
// long rows, then the p-th eighth of the others, both in list order.  `rank` is the
// inclusive prefix sum of `flags`.  Without long rows the list is unchanged.
constexpr int64_t kDealParts = 8;
// `rank`: inclusive number of long rows up to list position i
__device__ __forceinline__ int64_t dealt_position(int i, bool is_long, int64_t rank, int64_t num_long, int num_nodes) {
    const int64_t num_short = num_nodes - num_long;
    const int64_t mine = is_long ? rank - 1 : i - rank;  // position among the rows of its kind
    const int64_t kind = is_long ? num_long : num_short;
    int64_t part = 0;
    while (part < kDealParts - 1 && (part + 1) * kind / kDealParts <= mine) part++;
    const int64_t start = part * num_long / kDealParts + part * num_short / kDealParts;
    const int64_t longs_here = (part + 1) * num_long / kDealParts - part * num_long / kDealParts;
    return is_long ? start + (mine - part * num_long / kDealParts)
                   : start + longs_here + (mine - part * num_short / kDealParts);
}
__global__ void deal_long_rows_kernel(const int32_t *__restrict__ order, const int32_t *__restrict__ flags,
                                      const int32_t *__restrict__ rank, int num_nodes,
                                      int32_t *__restrict__ dealt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_nodes) return;
    dealt[dealt_position(i, flags[i] != 0, rank[i], rank[num_nodes - 1], num_nodes)] = order[i];
}

constexpr int kBlockThreads = 1024;

// Stable sort of up to kBlockThreads * ITEMS (key, value) pairs by one workgroup, at most eight bits a
// pass, from and to `pairs` in LDS.  A wave takes 64 * ITEMS consecutive pairs, 64 at a time; the lanes of
// equal digits find each other with eight ballots, so a digit's count per wave needs no atomics and the
// ranks keep the order.
template <int ITEMS>
struct BlockSort {
    static constexpr int WAVES = kBlockThreads / kWave, DIGITS = 256;
    uint2 pairs[kBlockThreads * ITEMS];
    uint16_t counts[DIGITS][WAVES];  // pairs of a digit in a wave, then the place of the first of them
    int sums[WAVES];

    __device__ __forceinline__ void sort(int bits) {
        const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
        const int passes = (bits + 7) / 8, step = (bits + passes - 1) / passes;
        const unsigned mask = (1u << step) - 1;
        for (int shift = 0; shift < bits; shift += step) {
            uint2 pair[ITEMS];
            int rank[ITEMS];
            for (int i = lane; i < DIGITS; i += kWave) counts[i][wave] = 0;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int k = 0; k < ITEMS; k++) {
                pair[k] = pairs[(wave * ITEMS + k) * kWave + lane];
                const unsigned digit = (pair[k].x >> shift) & mask;
                unsigned long long same = ~0ull;
#pragma unroll
                for (int bit = 0; bit < 8; bit++) {
                    if (bit == step) break;
                    const unsigned long long set = __ballot((digit >> bit) & 1u);
                    same &= (digit >> bit) & 1u ? set : ~set;
                }
                const int before = counts[digit][wave];
                rank[k] = before + __popcll(same & ((1ull << lane) - 1ull));
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if ((same >> lane) == 1ull) counts[digit][wave] = (uint16_t)(rank[k] + 1);  // the last of its digit
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            __syncthreads();
            // exclusive prefix sums over (digit, wave): four consecutive counts a thread
            uint16_t *flat = &counts[0][0] + 4 * threadIdx.x;
            int local[4], sum = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) { local[i] = sum; sum += flat[i]; }
            int after = sum;
#pragma unroll
            for (int off = 1; off < kWave; off *= 2) {
                const int add = __shfl_up(after, off, kWave);
                if (lane >= off) after += add;
            }
            if (lane == kWave - 1) sums[wave] = after;
            __syncthreads();
            int base = after - sum;
            for (int w = 0; w < wave; w++) base += sums[w];
#pragma unroll
            for (int i = 0; i < 4; i++) flat[i] = (uint16_t)(base + local[i]);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < ITEMS; k++)
                pairs[counts[(pair[k].x >> shift) & mask][wave] + rank[k]] = pair[k];
            __syncthreads();
        }
    }
};

// The end of the row order for up to kBlockThreads * ITEMS rows, by one workgroup: the sort of the
// keys, the deal of the long rows and, with `segments`, the list of their pieces.  Nine launches of
// the general path (sort 4-6, flags, scan 2, deal) in one: each of those takes 3-5 us here whatever
// it moves.  5 000 rows: 25 us (32 us with the library's sort of a block, about 45 us in nine launches);
// what is left is the issue rate of one compute unit.
template <int ITEMS>
__global__ __launch_bounds__(kBlockThreads) void order_block_kernel(const uint32_t *__restrict__ keys,
                                                                    const int32_t *__restrict__ row_ptr,
                                                                    int num_nodes, int key_bits,
                                                                    int32_t *__restrict__ order, int row_cap,
                                                                    int row_piece, int max_segments,
                                                                    int32_t *__restrict__ segments) {
    extern __shared__ __attribute__((aligned(16))) unsigned char order_lds[];
    BlockSort<ITEMS> &sorter = *reinterpret_cast<BlockSort<ITEMS> *>(order_lds);
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
        // (the sort is stable: the entries past the last row stay behind every row of the same key)
        const int i = k * kBlockThreads + threadIdx.x;
        sorter.pairs[i] = make_uint2(i < num_nodes ? keys[i] : ~0u, i < num_nodes ? i : 0);
    }
    __syncthreads();
    sorter.sort(key_bits);
    const int64_t live = row_ptr[num_nodes];
    // a wave's entries: 64 consecutive ones per k; long rows are counted with ballots
    int row[ITEMS], begin[ITEMS], end[ITEMS], rank[ITEMS], longs = 0;
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
        row[k] = (int)sorter.pairs[(wave * ITEMS + k) * kWave + lane].y;
        begin[k] = row_ptr[row[k]];
        end[k] = row_ptr[row[k] + 1];
    }
    bool flag[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
        const int i = (wave * ITEMS + k) * kWave + lane;
        flag[k] = i < num_nodes && (int64_t)(end[k] - begin[k]) * num_nodes > 2 * live;
        const unsigned long long mask = __ballot(flag[k]);
        rank[k] = longs + __popcll(mask & ((2ull << lane) - 1ull));
        longs += __popcll(mask);
    }
    if (lane == 0) sorter.sums[wave] = longs;
    __syncthreads();
    int before = 0, num_long = 0;
    for (int w = 0; w < BlockSort<ITEMS>::WAVES; w++) {
        if (w < wave) before += sorter.sums[w];
        num_long += sorter.sums[w];
    }
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
        const int i = (wave * ITEMS + k) * kWave + lane;
        if (i >= num_nodes) continue;
        const int64_t at = num_long == 0 ? i : dealt_position(i, flag[k], before + rank[k], num_long, num_nodes);
        order[at] = row[k];
        if (segments != nullptr)
            list_row_pieces(row[k], begin[k], end[k], row_cap, row_piece, max_segments, segments);
    }
}
template <int ITEMS>
int launch_order_block(const uint32_t *keys, const int32_t *row_ptr, int num_nodes, int key_bits, int32_t *order,
                       int row_cap, int row_piece, int max_segments, int32_t *segments, hipStream_t stream) {
    constexpr size_t lds = sizeof(BlockSort<ITEMS>);
    static_assert(lds <= 160 * 1024, "LDS of a workgroup");
    auto kernel = order_block_kernel<ITEMS>;
    if (lds > 64 * 1024) {
        const int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                                 "hipFuncSetAttribute(order_block)");
        if (rc) return rc;
    }
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kBlockThreads), lds, stream, keys, row_ptr, num_nodes, key_bits, order,
                       row_cap, row_piece, max_segments, segments);
    return check_hip(hipGetLastError(), "locality_order (one workgroup)");
}

size_t align_up(size_t v, size_t a = 256) { return (v + a - 1) / a * a; }

unsigned grid_for(int64_t n) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 4096)); }

size_t scan_temp_bytes(int32_t num_nodes) {
    size_t bytes = 0;
    hipcub::DeviceScan::InclusiveSum(nullptr, bytes, (int32_t *)nullptr, (int32_t *)nullptr,
                                     num_nodes + 1);
    return bytes;
}

size_t sort_temp_bytes(int64_t num_edges) {
    size_t bytes = 0;
    hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                       (const int32_t *)nullptr, (int32_t *)nullptr, (int)num_edges);
    return bytes;
}

int row_ptr_impl(const int32_t *key, int64_t num_edges, int32_t num_nodes, int32_t *row_ptr,
                 void *temp, size_t temp_bytes, hipStream_t stream) {
    int rc = launch_fill_zero(row_ptr, sizeof(int32_t) * ((size_t)num_nodes + 1), stream);
    if (rc) return rc;
    if (num_edges > 0) {
        hipLaunchKernelGGL(count_keys_kernel, dim3(grid_for((num_edges + kCountChunk - 1) / kCountChunk)),
                           dim3(256), 0, stream, key, num_edges, num_nodes, row_ptr);
        rc = check_hip(hipGetLastError(), "csr count launch");
        if (rc) return rc;
    }
    return check_hip(hipcub::DeviceScan::InclusiveSum(temp, temp_bytes, row_ptr, row_ptr,
                                                      num_nodes + 1, stream),
                     "csr scan");
}

// Global node ids of a sharded graph reduced to shard-local ids; the sentinel stays.
__device__ __forceinline__ int32_t wrap_node(int32_t v, int32_t num_nodes) {
    if ((uint32_t)v < (uint32_t)num_nodes || v == INT32_MAX) return v;
    const int32_t r = v % num_nodes;  // Python semantics: the result takes the divisor's sign
    return r < 0 ? r + num_nodes : r;
}
__global__ void wrap_index_kernel(const int32_t *__restrict__ index, int64_t n, int32_t num_nodes,
                                  int32_t *__restrict__ out) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = wrap_node(index[i], num_nodes);
}

// ---- rows of an adjacency from its endpoints, in few launches -----------------------------------
// With the keys in order, row_ptr[r] is the position of the first key >= r: every thread compares a key
// with the one before it and writes the rows that begin there.  No counters to clear, no atomics, no
// scan: one launch in the place of six (two index reductions, clear, count, two of the scan).  Keys
// out of order are noticed on the way; the counts are then made by one workgroup (as the
// count / scan path makes them), a launch that otherwise returns at once.

// rows first .. last of row_ptr = value for every lane of the wave (none where last < first); the
// lanes with a single row write it themselves, longer runs (rows without edges) are written by the wave
__device__ __forceinline__ void fill_rows(int32_t *row_ptr, int first, int last, int value, int lane) {
    if (first == last) row_ptr[first] = value;
    unsigned long long runs = __ballot(last > first);
    while (runs) {
        const int src = __ffsll(runs) - 1;
        runs &= runs - 1;
        const int f = __shfl(first, src, kWave), l = __shfl(last, src, kWave), v = __shfl(value, src, kWave);
        for (int r = f + lane; r <= l; r += kWave) row_ptr[r] = v;
    }
}

// positions wave * 64 .. of every waves * 64; `perm`: other[perm[pos]] belongs to pos, and the keys are
// those of `sort_input_kernel` (padding: num_nodes).
// Returns whether a key of this thread was smaller than the one before it.
__device__ __forceinline__ bool rows_from_keys(const int32_t *key, const int32_t *other, const int32_t *perm,
                                               int64_t num_edges, int num_nodes, int32_t *other_out,
                                               int32_t *row_ptr, int64_t wave, int64_t waves, int lane) {
    bool unsorted = false;
    for (int64_t base = wave * kWave; base < num_edges; base += waves * kWave) {
        const int64_t e = base + lane;
        int first = 1, last = 0, past_first = 1, past_last = 0;
        if (e < num_edges) {
            other_out[e] = wrap_node(other[perm ? perm[e] : e], num_nodes);
            int k = key[e], before = e > 0 ? key[e - 1] : -1;
            if (perm == nullptr) {  // (sorted keys were reduced before the sort)
                k = wrap_node(k, num_nodes);
                if (e > 0) before = wrap_node(before, num_nodes);
            }
            unsorted |= k < before;
            first = min(before, num_nodes) + 1;
            last = min(k, num_nodes);
            if (e == num_edges - 1 && k < num_nodes) {
                past_first = k + 1;
                past_last = num_nodes;
            }
        }
        fill_rows(row_ptr, first, last, (int)e, lane);
        fill_rows(row_ptr, past_first, past_last, (int)num_edges, lane);
    }
    return unsorted;
}

// row_ptr = [0] + cumsum(bincount(key)) of keys in any order, by one workgroup of kBlockThreads
__device__ __forceinline__ void rows_by_count(const int32_t *key, int64_t num_edges, int num_nodes,
                                              int32_t *row_ptr) {
    __shared__ int sums[kBlockThreads];
    const int tid = threadIdx.x;
    auto read = [&](int64_t i) { return __hip_atomic_load(row_ptr + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    auto write = [&](int64_t i, int v) {
        __hip_atomic_store(row_ptr + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    for (int64_t i = tid; i <= num_nodes; i += kBlockThreads) write(i, 0);
    __threadfence();
    __syncthreads();
    for (int64_t e = tid; e < num_edges; e += kBlockThreads) {
        const int k = wrap_node(key[e], num_nodes);
        if ((unsigned)k < (unsigned)num_nodes) atomicAdd(row_ptr + k + 1, 1);
    }
    __threadfence();
    __syncthreads();
    const int64_t each = ((int64_t)num_nodes + kBlockThreads) / kBlockThreads;  // of num_nodes + 1 entries
    const int64_t from = min((int64_t)tid * each, (int64_t)num_nodes + 1);
    const int64_t to = min(from + each, (int64_t)num_nodes + 1);
    int sum = 0;
    for (int64_t i = from; i < to; i++) sum += read(i);
    sums[tid] = sum;
    __syncthreads();
    for (int off = 1; off < kBlockThreads; off *= 2) {
        const int add = tid >= off ? sums[tid - off] : 0;
        __syncthreads();
        sums[tid] += add;
        __syncthreads();
    }
    int running = sums[tid] - sum;
    for (int64_t i = from; i < to; i++) {
        running += read(i);
        write(i, running);
    }
}

constexpr int kMaxRowsBlocks = 1024;
// `unsorted` (one word per block; null: the keys are known to be in order)
__global__ __launch_bounds__(256) void rows_kernel(const int32_t *__restrict__ key, const int32_t *__restrict__ other,
                                                   const int32_t *__restrict__ perm, int64_t num_edges, int num_nodes,
                                                   int32_t *__restrict__ other_out, int32_t *__restrict__ row_ptr,
                                                   int32_t *__restrict__ unsorted, int32_t *__restrict__ segments) {
    if (segments != nullptr && blockIdx.x == 0 && threadIdx.x < 4) segments[threadIdx.x] = 0;
    const int64_t thread = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool mine = rows_from_keys(key, other, perm, num_edges, num_nodes, other_out, row_ptr, thread / kWave,
                                     (int64_t)gridDim.x * blockDim.x / kWave, threadIdx.x % kWave);
    if (unsorted == nullptr) return;
    const int any = __syncthreads_or(mine ? 1 : 0);
    if (threadIdx.x == 0) unsorted[blockIdx.x] = any;
}
__global__ __launch_bounds__(kBlockThreads) void recount_rows_kernel(const int32_t *__restrict__ key,
                                                                     int64_t num_edges, int num_nodes,
                                                                     const int32_t *__restrict__ unsorted, int blocks,
                                                                     int32_t *__restrict__ row_ptr) {
    if (!__syncthreads_or((int)threadIdx.x < blocks && unsorted[threadIdx.x] != 0)) return;
    rows_by_count(key, num_edges, num_nodes, row_ptr);
}
// both, and the pieces of long rows, for graphs whose edges one workgroup reads in a few microseconds
constexpr int64_t kRowsBlockEdges = 16384;
__global__ __launch_bounds__(kBlockThreads) void rows_block_kernel(const int32_t *__restrict__ key,
                                                                   const int32_t *__restrict__ other,
                                                                   int64_t num_edges, int num_nodes,
                                                                   int32_t *__restrict__ other_out, int32_t *row_ptr,
                                                                   bool list_pieces, int row_cap, int row_piece,
                                                                   int max_segments, int32_t *segments) {
    if (segments != nullptr && threadIdx.x < 4) segments[threadIdx.x] = 0;
    const bool mine = rows_from_keys(key, other, nullptr, num_edges, num_nodes, other_out, row_ptr,
                                     threadIdx.x / kWave, kBlockThreads / kWave, threadIdx.x % kWave);
    // the rows above are ordered before another wave of the workgroup clears them for the counts
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (__syncthreads_or(mine ? 1 : 0)) rows_by_count(key, num_edges, num_nodes, row_ptr);
    if (!list_pieces || segments == nullptr) return;
    __threadfence();
    __syncthreads();
    for (int r = threadIdx.x; r < num_nodes; r += kBlockThreads) {
        const int begin = __hip_atomic_load(row_ptr + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int end = __hip_atomic_load(row_ptr + r + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        list_row_pieces(r, begin, end, row_cap, row_piece, max_segments, segments);
    }
}
// keys to sort by (padding: num_nodes, behind every row) and the positions they come from
__global__ void sort_input_kernel(const int32_t *__restrict__ key, int64_t num_edges, int num_nodes,
                                  int32_t *__restrict__ keys, int32_t *__restrict__ positions) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < num_edges; i += stride) {
        keys[i] = min(wrap_node(key[i], num_nodes), num_nodes);
        positions[i] = (int32_t)i;
    }
}

// Stable sort of edge positions by key for 1 025 to kSortChunk * kSortChunks edges of fewer than 2^16 nodes (`own_sort`), in
// two passes of at most eight bits, a count and a scatter each: four launches, where the library's sort takes
// eight and the launch that writes its keys a ninth (150k edges, 5 000 nodes: 58 us -> 20; 3-5 us a launch whatever
// it moves).  A workgroup takes kSortChunk consecutive edges; the scatter of each adds up for itself how
// many edges of a smaller digit, or of the same one in an earlier chunk, there are.
constexpr int kSortItems = 4, kSortChunk = kBlockThreads * kSortItems, kSortChunks = 64, kSortDigits = 256;

// `key` from the endpoints (`reduce`: as sort_input_kernel makes it) or from the pass before
__device__ __forceinline__ unsigned sort_key(const int32_t *key, int64_t i, int num_nodes, bool reduce) {
    return (unsigned)(reduce ? min(wrap_node(key[i], num_nodes), num_nodes) : key[i]);
}
__global__ __launch_bounds__(kBlockThreads) void edge_digits_kernel(const int32_t *__restrict__ key, int64_t num_edges,
                                                                    int num_nodes, bool reduce, int shift, unsigned mask,
                                                                    int32_t *__restrict__ digits) {
    __shared__ int count[kSortDigits];
    if (threadIdx.x < kSortDigits) count[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSortItems; k++) {
        const int64_t i = (int64_t)blockIdx.x * kSortChunk + k * kBlockThreads + threadIdx.x;
        if (i < num_edges) atomicAdd(&count[sort_key(key, i, num_nodes, reduce) >> shift & mask], 1);
    }
    __syncthreads();
    if (threadIdx.x < kSortDigits) digits[blockIdx.x * kSortDigits + threadIdx.x] = count[threadIdx.x];
}
// `from`: position a key came from (null: its own)
__global__ __launch_bounds__(kBlockThreads) void edge_scatter_kernel(
    const int32_t *__restrict__ key, const int32_t *__restrict__ from, int64_t num_edges, int num_nodes, bool reduce,
    int shift, int step, const int32_t *__restrict__ digits, int32_t *__restrict__ key_out, int32_t *__restrict__ from_out) {
    constexpr int WAVES = kBlockThreads / kWave, PARTS = kBlockThreads / kSortDigits;
    __shared__ uint16_t counts[kSortDigits][WAVES];  // edges of a digit in a wave, then in the waves before it
    __shared__ int before[PARTS][kSortDigits], all[PARTS][kSortDigits], sums[kSortDigits / kWave];
    const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
    const unsigned mask = (1u << step) - 1;
    {   // a quarter of the chunks each: edges of a digit in all of them and in those before this one
        const int digit = tid % kSortDigits, part = tid / kSortDigits, chunks = gridDim.x;
        int mine = 0, total = 0;
        for (int c = part; c < chunks; c += PARTS) {
            const int v = digits[c * kSortDigits + digit];
            total += v;
            if (c < (int)blockIdx.x) mine += v;
        }
        before[part][digit] = mine;
        all[part][digit] = total;
    }
    for (int i = lane; i < kSortDigits; i += kWave) counts[i][wave] = 0;
    unsigned item[kSortItems];
    int rank[kSortItems], source[kSortItems];
    const int64_t first = (int64_t)blockIdx.x * kSortChunk + wave * (kSortItems * kWave);
#pragma unroll
    for (int k = 0; k < kSortItems; k++) {
        const int64_t i = first + k * kWave + lane;
        item[k] = i < num_edges ? sort_key(key, i, num_nodes, reduce) : 0u;
        source[k] = i < num_edges ? (from != nullptr ? from[i] : (int)i) : 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int k = 0; k < kSortItems; k++) {  // (as in BlockSort: lanes of equal digits find each other with ballots)
        const bool inside = first + k * kWave + lane < num_edges;
        const unsigned digit = item[k] >> shift & mask;
        unsigned long long same = __ballot(inside);
#pragma unroll
        for (int bit = 0; bit < 8; bit++) {
            if (bit == step) break;
            const unsigned long long set = __ballot((digit >> bit) & 1u);
            same &= (digit >> bit) & 1u ? set : ~set;
        }
        const int earlier = counts[digit][wave];
        rank[k] = earlier + __popcll(same & ((1ull << lane) - 1ull));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (inside && (same >> lane) == 1ull) counts[digit][wave] = (uint16_t)(rank[k] + 1);  // the last of its digit
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    int start = 0, total = 0;
    if (tid < kSortDigits) {
#pragma unroll
        for (int p = 0; p < PARTS; p++) {
            start += before[p][tid];
            total += all[p][tid];
        }
        int sum = 0;
        for (int w = 0; w < WAVES; w++) {
            const int c = counts[tid][w];
            counts[tid][w] = (uint16_t)sum;
            sum += c;
        }
        int after = total;  // edges of this digit and of smaller ones
#pragma unroll
        for (int off = 1; off < kWave; off *= 2) {
            const int add = __shfl_up(after, off, kWave);
            if (lane >= off) after += add;
        }
        if (lane == kWave - 1) sums[wave] = after;
        start += after - total;
    }
    __syncthreads();
    if (tid < kSortDigits) {
        for (int w = 0; w < wave; w++) start += sums[w];
        before[0][tid] = start;  // where the chunk's edges of the digit begin
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSortItems; k++) {
        if (first + k * kWave + lane >= num_edges) continue;
        const unsigned digit = item[k] >> shift & mask;
        const int to = before[0][digit] + counts[digit][wave] + rank[k];
        key_out[to] = (int32_t)item[k];
        from_out[to] = source[k];
    }
}

__global__ void live_keys_kernel(const int32_t *__restrict__ other, const int32_t *__restrict__ row_ptr,
                                 int32_t num_nodes, int64_t num_edges, int32_t *__restrict__ keys) {
    const int64_t live_end = row_ptr[num_nodes];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < num_edges; i += stride) {
        const int32_t v = other[i];
        keys[i] = (i < live_end && (unsigned)v < (unsigned)num_nodes) ? v : INT32_MAX;
    }
}


// ---- schedule of the backward over tiles of receivers ---------------------------------------
// Tiles are `tile_rows` consecutive entries of the row order.  A scan of the tiles' position
// counts places each tile's list; one wave per tile, or a workgroup where the tiles are longer than a
// wave, then writes the list, sorted by sender.

__global__ void tile_rank_kernel(const int32_t *__restrict__ row_order, int num_nodes,
                                 int32_t *__restrict__ rank) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= num_nodes) return;
    rank[row_order ? row_order[q] : q] = q;
}

// Per tile, two numbers that one prefix sum carries side by side in a 64-bit word: the positions
// of the tile (high half) and the work descriptors it is cut into (low half); both totals stay
// below 2^31, so the low half never carries into the high one.
__device__ inline int tile_start(uint64_t packed) { return (int)(packed >> 32); }
__device__ inline int tile_first_piece(uint64_t packed) { return (int)(uint32_t)packed; }

// (positions of tile t, descriptors of tile t)
__device__ __forceinline__ uint64_t tile_count(const int32_t *row_order, const int32_t *row_ptr, int num_nodes,
                                               int tile_rows, int max_work_edges, int t) {
    int total = 0;
    for (int q = t * tile_rows; q < (t + 1) * tile_rows && q < num_nodes; q++) {
        const int r = row_order ? row_order[q] : q;
        total += row_ptr[r + 1] - row_ptr[r];
    }
    const int pieces = total == 0 ? 1 : (total + max_work_edges - 1) / max_work_edges;
    return ((uint64_t)total << 32) | (uint64_t)pieces;
}

// packed[t + 1] = the counts of tile t; packed[0] = 0
__global__ void tile_count_kernel(const int32_t *__restrict__ row_order, const int32_t *__restrict__ row_ptr,
                                  int num_nodes, int tile_rows, int num_tiles, int max_work_edges,
                                  uint64_t *__restrict__ packed) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0) packed[0] = 0;
    if (t >= num_tiles) return;
    packed[t + 1] = tile_count(row_order, row_ptr, num_nodes, tile_rows, max_work_edges, t);
}

// The three lists of one tile, by WPT waves: the tile's positions (its rows in tile order, each
// row's positions ascending) are keyed by (sender, position), padding senders after the live
// ones.  A tile of at most kTileSortLimit positions is listed in the order of the keys: they are all
// different, so a position's place is the number of smaller keys, which every lane counts for its
// positions over the keys in LDS (all lanes read the same one).  Sorted with a bitonic network
// by one wave instead, the 28 dependent steps of a tile of 120 positions were the kernel's time (150k
// edges in tiles of four rows: 18 -> 14 us).
// Longer tiles (hub rows) are not sorted by sender, only split into live positions first
// and padding positions last, which is all the kernel needs for correctness (it sums runs of
// equal senders wherever they occur); a hub's senders are mostly distinct anyway.
// The entries past the last row (padding positions that belong to no tile) are filled by all
// threads of the grid before they turn to their tiles.
constexpr int kTileSortLimit = 512;
template <int WPT>
__global__ __launch_bounds__(256) void tile_lists_kernel(
    const int32_t *__restrict__ other, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ perm,
    const int32_t *__restrict__ row_order, const uint64_t *__restrict__ packed, int num_nodes, int64_t num_edges,
    int tile_rows, int num_tiles, int32_t *__restrict__ t_sender, int32_t *__restrict__ t_edge,
    int32_t *__restrict__ t_local) {
    static_assert(WPT == 1 || WPT == 4, "a wave or the workgroup per tile");
    constexpr int TILES = 4 / WPT, LANES = kWave * WPT;
    __shared__ __attribute__((aligned(16))) uint64_t keys_all[TILES][kTileSortLimit];
    __shared__ uint16_t local_all[TILES][kTileSortLimit];
    {
        const int64_t stride = (int64_t)gridDim.x * blockDim.x;
        for (int64_t i = (int64_t)row_ptr[num_nodes] + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
             i < num_edges; i += stride) {
            t_sender[i] = -1; t_edge[i] = 0; t_local[i] = 0;
        }
    }
    const int tile = threadIdx.x / LANES, lane = threadIdx.x % kWave, at_lane = threadIdx.x % LANES;
    const int t = blockIdx.x * TILES + tile;
    if (t >= num_tiles) return;  // (with WPT 4: the whole workgroup, also below)
    uint64_t *keys = keys_all[tile];
    uint16_t *locals = local_all[tile];
    const int begin = tile_start(packed[t]), m = tile_start(packed[t + 1]) - begin;
    if (m == 0) return;
    const int first = t * tile_rows;
    const int rows = num_nodes - first < tile_rows ? num_nodes - first : tile_rows;
    if (m <= kTileSortLimit) {
        auto put = [&](int q, int pos, int row) {
            const int snd = other[pos];
            const uint64_t sk = (unsigned)snd < (unsigned)num_nodes ? (uint64_t)snd : (uint64_t)num_nodes;
            // (sender, position) orders the list; the row the position came from travels beside it
            keys[q] = (sk << 32) | (uint64_t)(uint32_t)pos;
            locals[q] = (uint16_t)row;
        };
        if (rows <= kWave) {
            // a lane per row reads where it lies, then the positions are taken across the rows
            int b = 0, d = 0;
            if (lane < rows) {
                const int r = row_order ? row_order[first + lane] : first + lane;
                b = row_ptr[r];
                d = row_ptr[r + 1] - b;
            }
            int after = d;  // inclusive prefix sum over the rows
#pragma unroll
            for (int off = 1; off < kWave; off *= 2) {
                const int add = __shfl_up(after, off, kWave);
                if (lane >= off) after += add;
            }
            for (int q0 = 0; q0 < m; q0 += LANES) {
                const int q = q0 + at_lane;
                int row = 0, pos = 0;
                for (int i = 0; i < rows; i++) {
                    const int stop = __builtin_amdgcn_readlane(after, i), len = __builtin_amdgcn_readlane(d, i);
                    const int start = __builtin_amdgcn_readlane(b, i);
                    if (q < stop && q >= stop - len) { row = i; pos = start + q - (stop - len); }
                }
                if (q < m) put(q, pos, row);
            }
        } else {
            for (int i = 0, filled = 0; i < rows; i++) {
                const int r = row_order ? row_order[first + i] : first + i;
                const int b = row_ptr[r], d = row_ptr[r + 1] - b;
                for (int q = at_lane; q < d; q += LANES) put(filled + q, b + q, i);
                filled += d;
            }
        }
        constexpr int PER = kTileSortLimit / LANES;  // positions of a lane
        for (int q = m + at_lane; q < (m + LANES - 1) / LANES * LANES; q += LANES) keys[q] = ~0ull;  // above every key
        if (WPT == 1) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
        uint64_t mine[PER];
        int place[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            place[k] = 0;
            mine[k] = k * LANES < m ? keys[k * LANES + at_lane] : ~0ull;
        }
        for (int j = 0; j < m; j += 2) {  // (an odd m: entry m was written, LANES is even)
            const ulonglong2 pair = *reinterpret_cast<const ulonglong2 *>(keys + j);
#pragma unroll
            for (int k = 0; k < PER; k++) {
                if (k * LANES >= m) continue;
                place[k] += (pair.x < mine[k] ? 1 : 0) + (pair.y < mine[k] ? 1 : 0);
            }
        }
#pragma unroll
        for (int k = 0; k < PER; k++) {
            if (k * LANES + at_lane >= m) continue;
            const int slot = begin + place[k], pos = (int)(uint32_t)mine[k];
            const uint64_t sk = mine[k] >> 32;
            t_sender[slot] = sk == (uint64_t)num_nodes ? -1 : (int32_t)sk;
            t_edge[slot] = perm ? perm[pos] : pos;
            t_local[slot] = locals[k * LANES + at_lane];
        }
        return;
    }
    if (at_lane >= kWave) return;  // the rest is one wave's
    // a long tile: live positions in tile order, then the padding positions
    int at = begin;
    for (int pass = 0; pass < 2; pass++) {
        for (int i = 0; i < rows; i++) {
            const int r = row_order ? row_order[first + i] : first + i;
            const int b = row_ptr[r], d = row_ptr[r + 1] - b;
            for (int q0 = 0; q0 < d; q0 += 64) {
                const int q = q0 + lane;
                const int snd = q < d ? other[b + q] : -1;
                const bool live = (unsigned)snd < (unsigned)num_nodes;
                const bool mine = q < d && (live == (pass == 0));
                const unsigned long long mask = __ballot(mine);
                if (mine) {
                    const int slot = at + __popcll(mask & ((1ull << lane) - 1ull));
                    t_sender[slot] = live ? snd : -1;
                    t_edge[slot] = perm ? perm[b + q] : b + q;
                    t_local[slot] = i;
                }
                at += __popcll(mask);
            }
        }
    }
}

// descriptors (tile, begin, end, 0), the first num_used of the num_work entries (a tile without
// positions takes one, with begin == end; the entries behind the used ones are not written),
// num_used in the fourth field of descriptor 0; `packed`: inclusive prefix sums, entry 0 = 0
__device__ __forceinline__ void write_tile_work(int t, uint64_t before, uint64_t after, int num_used,
                                                int max_work_edges, int32_t *work) {
    const int begin = tile_start(before), end = tile_start(after);
    int w = tile_first_piece(before);
    if (begin == end) {
        work[4 * w] = t; work[4 * w + 1] = begin; work[4 * w + 2] = begin; work[4 * w + 3] = 0;
    }
    for (int b = begin; b < end; b += max_work_edges, w++) {
        work[4 * w] = t;
        work[4 * w + 1] = b;
        work[4 * w + 2] = b + max_work_edges < end ? b + max_work_edges : end;
        work[4 * w + 3] = 0;
    }
    // the number of descriptors in use, for the kernel to deal them evenly to the XCDs (the
    // thread of tile 0 wrote descriptor 0 just above)
    if (t == 0) work[3] = num_used;
}
__global__ void tile_work_kernel(const uint64_t *__restrict__ packed, int num_tiles, int max_work_edges,
                                 int32_t *__restrict__ work) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= num_tiles) return;
    write_tile_work(t, packed[t], packed[t + 1], tile_first_piece(packed[num_tiles]), max_work_edges, work);
}

// Counts, prefix sums and work descriptors of up to kBlockThreads * kTileItems tiles by one workgroup
// (the four launches of the general path take 3-5 us each on a schedule of this size).
constexpr int kTileItems = 4;
__global__ __launch_bounds__(kBlockThreads) void tile_plan_block_kernel(
    const int32_t *__restrict__ row_order, const int32_t *__restrict__ row_ptr, int num_nodes, int tile_rows,
    int num_tiles, int max_work_edges, uint64_t *__restrict__ packed, int32_t *__restrict__ work) {
    using Scan = hipcub::BlockScan<uint64_t, kBlockThreads>;
    __shared__ typename Scan::TempStorage temp;
    uint64_t count[kTileItems], before[kTileItems], all;
    const int first = (int)threadIdx.x * kTileItems;
#pragma unroll
    for (int k = 0; k < kTileItems; k++) {
        const int t = first + k;
        count[k] = t < num_tiles ? tile_count(row_order, row_ptr, num_nodes, tile_rows, max_work_edges, t) : 0;
    }
    Scan(temp).ExclusiveSum(count, before, all);
    if (threadIdx.x == 0) packed[0] = 0;
#pragma unroll
    for (int k = 0; k < kTileItems; k++) {
        const int t = first + k;
        if (t >= num_tiles) continue;
        packed[t + 1] = before[k] + count[k];
        write_tile_work(t, before[k], before[k] + count[k], tile_first_piece(all), max_work_edges, work);
    }
}

size_t scan64_temp_bytes(int32_t n) {
    size_t bytes = 0;
    hipcub::DeviceScan::InclusiveSum(nullptr, bytes, (uint64_t *)nullptr, (uint64_t *)nullptr, (int)std::max(n, 1));
    return bytes;
}

struct TileWorkspace {
    size_t temp, temp_bytes, packed, total;
    TileWorkspace(int32_t num_nodes, int32_t tile_rows) {
        const size_t n = (size_t)num_nodes;
        const size_t tiles = (n + (size_t)tile_rows - 1) / (size_t)tile_rows;
        size_t at = 0;
        auto take = [&](size_t bytes) { const size_t here = at; at += align_up(bytes); return here; };
        temp_bytes = scan64_temp_bytes((int32_t)tiles + 1);
        temp = take(temp_bytes);
        packed = take(8 * (tiles + 1));
        total = at;
    }
};


// rows[pos] = the CSR row that holds position pos; INT32_MAX past the last row
__global__ void expand_rows_kernel(const int32_t *__restrict__ row_ptr, int num_nodes, int64_t num_edges,
                                   int32_t *__restrict__ rows) {
    const int64_t live_end = row_ptr[num_nodes];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t pos = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; pos < num_edges; pos += stride) {
        if (pos >= live_end) { rows[pos] = INT32_MAX; continue; }
        int lo = 0, hi = num_nodes;  // row_ptr[lo] <= pos < row_ptr[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (row_ptr[mid] <= pos) lo = mid; else hi = mid;
        }
        rows[pos] = lo;
    }
}

__global__ void compose_perm_kernel(const int32_t *__restrict__ outer, const int32_t *__restrict__ inner,
                                    int64_t n, int32_t *__restrict__ out) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = inner ? inner[outer[i]] : outer[i];
}

// ---- pairing of rows for the backward over tiles of two receivers ------------------------------
// Two rows that share most of their senders should sit in one tile: the tile then issues one set
// of dx atomics for every shared sender.  Every row picks, among the rows it has an edge from,
// the one with which it has the most senders in common; rows that pick each other are paired, the
// rest pick again among the rows still free (a few rounds of this greedy matching pair most rows
// of a radius graph).  Pairs are then listed first, in the order their earlier member had, each
// pair on an even and the following odd position; the unpaired rows follow in their old order.
constexpr int kPairMaxDegree = 128;  // rows with more edges (or none) stay unpaired
constexpr int kPairSlots = 256;      // hash slots per wave for the senders of its row
constexpr int kPairRounds = 4;

__device__ __forceinline__ unsigned pair_hash(int v) { return ((unsigned)v * 2654435761u) >> 24; }

// common[pos] = number of senders that the row of position pos and the row other[pos] share
// (-1: no candidate).  One wave per row; its senders go into a hash set in LDS, then every lane
// walks the row of one neighbour and counts hits.
__global__ __launch_bounds__(256) void pair_common_kernel(const int32_t *__restrict__ other,
                                                          const int32_t *__restrict__ row_ptr, int num_nodes,
                                                          int32_t *__restrict__ common) {
    __shared__ int32_t slots_all[4][kPairSlots];
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int i = blockIdx.x * 4 + wave;
    if (i >= num_nodes) return;
    int32_t *slots = slots_all[wave];
    const int begin = row_ptr[i], deg = row_ptr[i + 1] - begin;
    if (deg < 1) return;
    if (deg > kPairMaxDegree) {
        for (int q = lane; q < deg; q += 64) common[begin + q] = -1;
        return;
    }
    for (int t = lane; t < kPairSlots; t += 64) slots[t] = -1;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int q = lane; q < deg; q += 64) {
        const int v = other[begin + q];
        if ((unsigned)v >= (unsigned)num_nodes) continue;
        unsigned h = pair_hash(v);
        for (int probe = 0; probe < kPairSlots; probe++) {
            const int old = atomicCAS(&slots[h], -1, v);
            if (old == -1 || old == v) break;
            h = (h + 1) % kPairSlots;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int q = lane; q < deg; q += 64) {
        const int p = other[begin + q];
        int count = -1;
        if ((unsigned)p < (unsigned)num_nodes && p != i) {
            const int pb = row_ptr[p], pd = row_ptr[p + 1] - pb;
            if (pd >= 1 && pd <= kPairMaxDegree) {
                count = 0;
                for (int t = 0; t < pd; t++) {
                    const int v = other[pb + t];
                    if ((unsigned)v >= (unsigned)num_nodes) continue;
                    unsigned h = pair_hash(v);
                    for (int probe = 0; probe < kPairSlots; probe++) {
                        const int held = slots[h];
                        if (held == v) { count++; break; }
                        if (held == -1) break;
                        h = (h + 1) % kPairSlots;
                    }
                }
            }
        }
        common[begin + q] = count;
    }
}

// best[i] = the free row with the most senders in common with free row i (smaller id on ties), -1 if none
__global__ void pair_best_kernel(const int32_t *__restrict__ other, const int32_t *__restrict__ row_ptr,
                                 const int32_t *__restrict__ common, const int32_t *__restrict__ partner,
                                 int num_nodes, int32_t *__restrict__ best) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_nodes) return;
    int pick = -1, most = -1;
    const int begin = row_ptr[i], deg = row_ptr[i + 1] - begin;
    if (partner[i] < 0 && deg >= 1 && deg <= kPairMaxDegree) {
        for (int q = 0; q < deg; q++) {
            const int c = common[begin + q];
            if (c < 0) continue;
            const int p = other[begin + q];
            if (partner[p] >= 0) continue;
            if (c > most || (c == most && p < pick)) { most = c; pick = p; }
        }
    }
    best[i] = pick;
}

__global__ void pair_match_kernel(const int32_t *__restrict__ best, int num_nodes, int32_t *__restrict__ partner) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_nodes) return;
    const int p = best[i];
    if (p >= 0 && best[p] == i) partner[i] = p;  // (the thread of row p writes partner[p] = i)
}

__global__ void pair_keys_kernel(const int32_t *__restrict__ partner, const int32_t *__restrict__ rank,
                                 int num_nodes, uint32_t *__restrict__ keys, int32_t *__restrict__ vals) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_nodes) return;
    const int p = partner[i];
    const unsigned mine = rank ? rank[i] : i;
    vals[i] = i;
    if (p < 0) {
        keys[i] = 2u * (unsigned)num_nodes + mine;
    } else {
        const unsigned theirs = rank ? rank[p] : p;
        keys[i] = 2u * (mine < theirs ? mine : theirs) + (mine > theirs ? 1u : 0u);
    }
}

__global__ void fill_i32_kernel(int32_t *__restrict__ out, int64_t n, int32_t value) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = value;
}

}  // namespace

int launch_live_keys(const int32_t *other, const int32_t *row_ptr, int32_t num_nodes,
                     int64_t num_edges, int32_t *keys, hipStream_t stream) {
    if (num_edges == 0) return E3J_AMD_OK;
    hipLaunchKernelGGL(live_keys_kernel, dim3(grid_for(num_edges)), dim3(256), 0, stream, other, row_ptr,
                       num_nodes, num_edges, keys);
    return check_hip(hipGetLastError(), "live keys launch");
}

int launch_expand_rows(const int32_t *row_ptr, int32_t num_nodes, int64_t num_edges, int32_t *rows,
                       hipStream_t stream) {
    if (num_edges == 0) return E3J_AMD_OK;
    hipLaunchKernelGGL(expand_rows_kernel, dim3(grid_for(num_edges)), dim3(256), 0, stream, row_ptr, num_nodes,
                       num_edges, rows);
    return check_hip(hipGetLastError(), "expand rows launch");
}

int launch_compose_perm(const int32_t *outer, const int32_t *inner, int64_t n, int32_t *out, hipStream_t stream) {
    if (n == 0) return E3J_AMD_OK;
    hipLaunchKernelGGL(compose_perm_kernel, dim3(grid_for(n)), dim3(256), 0, stream, outer, inner, n, out);
    return check_hip(hipGetLastError(), "compose permutation launch");
}

}  // namespace e3j_amd

using namespace e3j_amd;

extern "C" {

size_t e3j_amd_csr_workspace_bytes(int32_t num_nodes, int64_t num_edges) {
    if (num_nodes < 0 || num_edges < 0) return 0;
    // [scan temp | sort temp | keys_out (E) | iota (E)]
    return align_up(scan_temp_bytes(num_nodes)) + align_up(sort_temp_bytes(num_edges)) +
           2 * align_up(sizeof(int32_t) * (size_t)num_edges) + 256;
}

int e3j_amd_csr_row_ptr(const int32_t *key, int64_t num_edges, int32_t num_nodes, int32_t *row_ptr,
                        void *workspace, void *stream_) {
    if (num_nodes < 0 || num_nodes >= INT32_MAX || num_edges < 0 || num_edges > 0x7fffffffLL)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "csr_row_ptr: bad sizes");
    if (row_ptr == nullptr || workspace == nullptr || (num_edges > 0 && key == nullptr))
        return set_error(E3J_AMD_INVALID_ARGUMENT, "csr_row_ptr: null operand");
    return row_ptr_impl(key, num_edges, num_nodes, row_ptr, workspace, scan_temp_bytes(num_nodes),
                        static_cast<hipStream_t>(stream_));
}

// ---- row pointers without a workspace argument ------------------------------------------------
// The scan of e3j_amd_csr_row_ptr needs a few KB of temporary storage.  Callers that cannot
// allocate (code under graph capture, serving loops) get it from this array instead: device
// memory of the library's code object, one copy per GPU, held until the process ends.
constexpr size_t kStaticScratchBytes = 256 * 1024;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices];  // address of `scratch` on each device, looked up once
// The device address of the array on the current device (the array's name is only a host-side
// handle of the symbol).
int static_scratch(void **ptr) {
    int device = 0;
    int rc = check_hip(hipGetDevice(&device), "csr_row_ptr_static: hipGetDevice");
    if (rc) return rc;
    if (device < 0 || device >= kMaxDevices)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "csr_row_ptr_static: device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[device] == nullptr) {
        void *address = nullptr;
        rc = check_hip(hipGetSymbolAddress(&address, HIP_SYMBOL(scratch)), "csr_row_ptr_static: hipGetSymbolAddress");
        if (rc) return rc;
        g_scratch_ptr[device] = address;
    }
    *ptr = g_scratch_ptr[device];
    return E3J_AMD_OK;
}
}  // namespace

int32_t e3j_amd_csr_row_ptr_static_max_nodes(void) {
    // the scan's temporary storage grows with the number of entries; largest count that fits
    int32_t lo = 0, hi = INT32_MAX - 1;
    while (lo < hi) {
        const int32_t mid = lo + (hi - lo + 1) / 2;
        if (scan_temp_bytes(mid) <= kStaticScratchBytes) lo = mid; else hi = mid - 1;
    }
    return lo;
}

int e3j_amd_csr_row_ptr_static(const int32_t *key, int64_t num_edges, int32_t num_nodes, int32_t *row_ptr,
                               void *stream_) {
    // (num_nodes + 1 entries are scanned: INT32_MAX nodes would overflow the count)
    if (num_nodes < 0 || num_nodes >= INT32_MAX || num_edges < 0 || num_edges > 0x7fffffffLL)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "csr_row_ptr_static: bad sizes");
    if (row_ptr == nullptr || (num_edges > 0 && key == nullptr))
        return set_error(E3J_AMD_INVALID_ARGUMENT, "csr_row_ptr_static: null operand");
    const size_t need = scan_temp_bytes(num_nodes);
    if (need > kStaticScratchBytes)
        return set_error(E3J_AMD_INVALID_ARGUMENT,
                         "csr_row_ptr_static: " + std::to_string(num_nodes) + " nodes need " + std::to_string(need) +
                             " bytes of scan storage, the built-in scratch holds " +
                             std::to_string(kStaticScratchBytes) + " (use e3j_amd_csr_row_ptr with a workspace)");
    void *temp = nullptr;
    int rc = static_scratch(&temp);
    if (rc) return rc;
    return row_ptr_impl(key, num_edges, num_nodes, row_ptr, temp, need, static_cast<hipStream_t>(stream_));
}

int64_t e3j_amd_row_segments_max(int64_t num_edges, int32_t row_piece) {
    if (num_edges <= 0 || row_piece <= 0) return 0;
    return num_edges / row_piece;  // a piece after the first follows row_piece positions of its row
}

int e3j_amd_row_segments_build(const int32_t *receiver_ptr, int32_t num_nodes, int32_t row_cap,
                               int32_t row_piece, int32_t max_segments, int32_t *segments, void *stream_) {
    if (num_nodes < 0 || row_piece <= 0 || row_cap < row_piece || max_segments < 0)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "row_segments_build: bad sizes");
    if (segments == nullptr || (num_nodes > 0 && receiver_ptr == nullptr))
        return set_error(E3J_AMD_INVALID_ARGUMENT, "row_segments_build: null operand");
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    int rc = launch_fill_zero(segments, sizeof(int32_t) * 4, stream);
    if (rc || num_nodes == 0) return rc;
    hipLaunchKernelGGL(row_segments_kernel, dim3((unsigned)(((int64_t)num_nodes + 255) / 256)), dim3(256), 0, stream,
                       receiver_ptr, num_nodes, row_cap, row_piece, max_segments, segments);
    return check_hip(hipGetLastError(), "row_segments_build");
}

int e3j_amd_wrap_index(const int32_t *index, int64_t n, int32_t num_nodes, int32_t *out,
                       void *stream_) {
    if (n < 0 || num_nodes <= 0)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "wrap_index: bad sizes");
    if (n == 0) return E3J_AMD_OK;
    if (index == nullptr || out == nullptr)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "wrap_index: null operand");
    hipLaunchKernelGGL(wrap_index_kernel, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream_,
                       index, n, num_nodes, out);
    return check_hip(hipGetLastError(), "wrap_index");
}

namespace {
struct PairWorkspace {
    size_t temp, temp_bytes, common, best, partner, rank, keys_in, keys_out, vals_in, total;
    PairWorkspace(int32_t num_nodes, int64_t num_edges) {
        const size_t n = (size_t)num_nodes, e = (size_t)num_edges;
        size_t at = 0;
        auto take = [&](size_t bytes) { const size_t here = at; at += align_up(bytes); return here; };
        temp_bytes = sort_temp_bytes(num_nodes);
        temp = take(temp_bytes);
        common = take(4 * e);
        best = take(4 * n); partner = take(4 * n); rank = take(4 * n);
        keys_in = take(4 * n); keys_out = take(4 * n); vals_in = take(4 * n);
        total = at + 256;
    }
};
}  // namespace

size_t e3j_amd_pair_rows_workspace_bytes(int32_t num_nodes, int64_t num_edges) {
    if (num_nodes < 0 || num_edges < 0) return 0;
    return PairWorkspace(num_nodes, num_edges).total;
}

int e3j_amd_pair_rows(const int32_t *other, const int32_t *row_ptr, int32_t num_nodes, int64_t num_edges,
                      const int32_t *order_in, int32_t *order_out, void *workspace, void *stream_) {
    if (num_nodes < 0 || num_edges < 0 || num_edges > 0x7fffffffLL || num_nodes > 0x3fffffff)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "pair_rows: bad sizes");
    if (num_nodes == 0) return E3J_AMD_OK;
    if (order_out == nullptr || workspace == nullptr || row_ptr == nullptr || (num_edges > 0 && other == nullptr))
        return set_error(E3J_AMD_INVALID_ARGUMENT, "pair_rows: null operand");
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    unsigned char *ws = static_cast<unsigned char *>(workspace);
    const PairWorkspace w(num_nodes, num_edges);
    int32_t *common = reinterpret_cast<int32_t *>(ws + w.common);
    int32_t *best = reinterpret_cast<int32_t *>(ws + w.best);
    int32_t *partner = reinterpret_cast<int32_t *>(ws + w.partner);
    int32_t *rank = reinterpret_cast<int32_t *>(ws + w.rank);
    uint32_t *keys_in = reinterpret_cast<uint32_t *>(ws + w.keys_in);
    uint32_t *keys_out = reinterpret_cast<uint32_t *>(ws + w.keys_out);
    int32_t *vals_in = reinterpret_cast<int32_t *>(ws + w.vals_in);
    const unsigned rows_grid = (unsigned)((num_nodes + 255) / 256);

    hipLaunchKernelGGL(fill_i32_kernel, dim3(grid_for(num_nodes)), dim3(256), 0, stream, partner,
                       (int64_t)num_nodes, -1);
    hipLaunchKernelGGL(pair_common_kernel, dim3((unsigned)((num_nodes + 3) / 4)), dim3(256), 0, stream, other,
                       row_ptr, num_nodes, common);
    int rc = check_hip(hipGetLastError(), "pair_rows common");
    if (rc) return rc;
    for (int round = 0; round < kPairRounds; round++) {
        hipLaunchKernelGGL(pair_best_kernel, dim3(rows_grid), dim3(256), 0, stream, other, row_ptr, common, partner,
                           num_nodes, best);
        hipLaunchKernelGGL(pair_match_kernel, dim3(rows_grid), dim3(256), 0, stream, best, num_nodes, partner);
    }
    if (order_in != nullptr)
        hipLaunchKernelGGL(tile_rank_kernel, dim3(rows_grid), dim3(256), 0, stream, order_in, num_nodes, rank);
    hipLaunchKernelGGL(pair_keys_kernel, dim3(rows_grid), dim3(256), 0, stream, partner,
                       order_in != nullptr ? rank : nullptr, num_nodes, keys_in, vals_in);
    rc = check_hip(hipGetLastError(), "pair_rows keys");
    if (rc) return rc;
    int key_bits = 2;  // keys are below 3 * num_nodes
    while (key_bits < 32 && ((uint64_t)1 << key_bits) < 3ull * (uint64_t)num_nodes) key_bits++;
    size_t temp_bytes = w.temp_bytes;
    return check_hip(hipcub::DeviceRadixSort::SortPairs(ws + w.temp, temp_bytes, keys_in, keys_out, vals_in,
                                                        order_out, (int)num_nodes, 0, key_bits, stream),
                     "pair_rows sort");
}

size_t e3j_amd_order_workspace_bytes(int32_t num_nodes) {
    if (num_nodes < 0) return 0;
    // [sort / scan temp | label a | label b | keys in | keys out | order tmp]
    return align_up(std::max(sort_temp_bytes(num_nodes), scan_temp_bytes(num_nodes))) +
           5 * align_up(sizeof(int32_t) * (size_t)num_nodes) + 256;
}

namespace {
// Where the caller wants the pieces of the rows longer than `cap` listed (segments[0] is zero when the
// order is made); segments null: nowhere.
struct PieceList {
    int32_t cap, piece, max_segments;
    int32_t *segments;
};
int locality_order(const int32_t *other, const int32_t *row_ptr, int32_t num_nodes, int32_t rounds, int32_t *order,
                   const PieceList &pieces, void *workspace, hipStream_t stream) {
    if (num_nodes < 0 || rounds < 0 || rounds > 64)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "locality_order: bad sizes");
    if (num_nodes == 0) return E3J_AMD_OK;
    if (order == nullptr || workspace == nullptr || row_ptr == nullptr)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "locality_order: null operand");
    unsigned char *ws = static_cast<unsigned char *>(workspace);
    const size_t sort_bytes = std::max(sort_temp_bytes(num_nodes), scan_temp_bytes(num_nodes));
    const size_t vec = align_up(sizeof(int32_t) * (size_t)num_nodes);
    void *sort_temp = ws;
    int32_t *lab_a = reinterpret_cast<int32_t *>(ws + align_up(sort_bytes));
    int32_t *lab_b = reinterpret_cast<int32_t *>(ws + align_up(sort_bytes) + vec);
    uint32_t *keys_in = reinterpret_cast<uint32_t *>(ws + align_up(sort_bytes) + 2 * vec);
    uint32_t *keys_out = reinterpret_cast<uint32_t *>(ws + align_up(sort_bytes) + 3 * vec);
    int32_t *order_tmp = reinterpret_cast<int32_t *>(ws + align_up(sort_bytes) + 4 * vec);
    const unsigned ngrid = grid_for(num_nodes);
    const unsigned rows_grid = (unsigned)((num_nodes + 255) / 256);

    int rc = E3J_AMD_OK;
    const int32_t *listed = order;  // where the order stands before the long rows are dealt
    // Levels: after 1, 2, 4, 8, ... sweeps the labels name ever larger clusters.  The order is
    // refined from the finest level to the coarsest with stable sorts, so the coarsest clusters
    // are contiguous and, inside them, the finer ones.
    int done = 0;
    int label_bits = 1;  // labels are node ids: the sort passes stop at their highest bit
    while (label_bits < 32 && ((int64_t)1 << label_bits) < (int64_t)num_nodes) label_bits++;
    const bool two_levels = rounds == 2 && 2 * label_bits <= 32;
    if (two_levels) {
        sweep_labels(other, row_ptr, num_nodes, nullptr, lab_b, nullptr, nullptr, 0, stream);
        const bool one_block = num_nodes <= 8 * kBlockThreads;
        sweep_labels(other, row_ptr, num_nodes, lab_b, lab_a, keys_in, one_block ? nullptr : order, label_bits, stream);
        if (one_block) {
            // (the kernel's time is the instructions of one compute unit, for padded entries too)
            using Launch = int (*)(const uint32_t *, const int32_t *, int, int, int32_t *, int, int, int, int32_t *,
                                   hipStream_t);
            static const Launch launches[8] = {launch_order_block<1>, launch_order_block<2>, launch_order_block<3>,
                                               launch_order_block<4>, launch_order_block<5>, launch_order_block<6>,
                                               launch_order_block<7>, launch_order_block<8>};
            const Launch launch = launches[(num_nodes - 1) / kBlockThreads];
            return launch(keys_in, row_ptr, num_nodes, 2 * label_bits, order, pieces.cap, pieces.piece,
                          pieces.max_segments, pieces.segments, stream);
        }
        rc = check_hip(hipGetLastError(), "locality_order sweeps");
        if (rc) return rc;
        // the two levels in one sort: same order as the two stable sorts below, half the passes
        size_t temp_bytes = sort_bytes;
        rc = check_hip(hipcub::DeviceRadixSort::SortPairs(sort_temp, temp_bytes, keys_in, keys_out, order, order_tmp,
                                                          (int)num_nodes, 0, 2 * label_bits, stream),
                       "locality_order sort");
        if (rc) return rc;
        listed = order_tmp;
        rounds = 0;  // done: skip the level loop
    } else {
        hipLaunchKernelGGL(iota_kernel, dim3(ngrid), dim3(256), 0, stream, lab_a, (int64_t)num_nodes);
        hipLaunchKernelGGL(iota_kernel, dim3(ngrid), dim3(256), 0, stream, order, (int64_t)num_nodes);
        rc = check_hip(hipGetLastError(), "locality_order init");
        if (rc) return rc;
    }
    for (int level = 1; level <= rounds; level *= 2) {
        for (; done < level; done++) {
            sweep_labels(other, row_ptr, num_nodes, lab_a, lab_b, nullptr, nullptr, 0, stream);
            int32_t *t = lab_a; lab_a = lab_b; lab_b = t;
        }
        hipLaunchKernelGGL(gather_kernel, dim3(ngrid), dim3(256), 0, stream, lab_a, order,
                           reinterpret_cast<int32_t *>(keys_in), (int64_t)num_nodes);
        rc = check_hip(hipGetLastError(), "locality_order sweep");
        if (rc) return rc;
        size_t temp_bytes = sort_bytes;
        rc = check_hip(hipcub::DeviceRadixSort::SortPairs(sort_temp, temp_bytes, keys_in, keys_out, order,
                                                          order_tmp, (int)num_nodes, 0, label_bits, stream),
                       "locality_order sort");
        if (rc) return rc;
        hipLaunchKernelGGL(copy_i32_kernel, dim3(ngrid), dim3(256), 0, stream, order_tmp, order,
                           (int64_t)num_nodes);
    }
    // long rows to the fronts of the eighths of the list
    int32_t *flags = reinterpret_cast<int32_t *>(keys_in), *rank = reinterpret_cast<int32_t *>(keys_out);
    hipLaunchKernelGGL(long_row_flags_kernel, dim3(rows_grid), dim3(256), 0, stream, listed, row_ptr, num_nodes,
                       flags, pieces.cap, pieces.piece, pieces.max_segments, pieces.segments);
    rc = check_hip(hipGetLastError(), "locality_order flags");
    if (rc) return rc;
    size_t scan_bytes = sort_bytes;
    rc = check_hip(hipcub::DeviceScan::InclusiveSum(sort_temp, scan_bytes, flags, rank, num_nodes, stream),
                   "locality_order scan");
    if (rc) return rc;
    if (listed == order_tmp) {  // dealt straight into the result
        hipLaunchKernelGGL(deal_long_rows_kernel, dim3(rows_grid), dim3(256), 0, stream, listed, flags, rank,
                           num_nodes, order);
    } else {
        hipLaunchKernelGGL(deal_long_rows_kernel, dim3(rows_grid), dim3(256), 0, stream, listed, flags, rank,
                           num_nodes, order_tmp);
        hipLaunchKernelGGL(copy_i32_kernel, dim3(ngrid), dim3(256), 0, stream, order_tmp, order,
                           (int64_t)num_nodes);
    }
    return check_hip(hipGetLastError(), "locality_order");
}
}  // namespace

int e3j_amd_locality_order(const int32_t *other, const int32_t *row_ptr, int32_t num_nodes,
                           int32_t rounds, int32_t *order, void *workspace, void *stream) {
    return locality_order(other, row_ptr, num_nodes, rounds, order, PieceList{0, 0, 0, nullptr}, workspace,
                          static_cast<hipStream_t>(stream));
}

namespace {
struct PrepareWorkspace {
    size_t order, sort_temp, sort_bytes, keys_in, keys_out, positions, unsorted, total;
    // The sort of this file: keys of two eight-bit digits, and no more chunks than the counts of which a workgroup reads
    // by itself.  It is the faster one up to there (CSR and sort: 60 000 rows, 262 144 edges 42 us for the library's
    // 103; 5 000 rows, 150 000 edges 34 for 63; 4 500 edges 26 for 33; 2 000 edges 26 for 28); up to 1 024 edges
    // the library sorts in one launch (500 edges: 20 us for 25).
    static bool own_sort(int32_t num_nodes, int64_t num_edges) {
        return num_nodes < (1 << 16) && num_edges > 1024 && num_edges <= (int64_t)kSortChunk * kSortChunks;
    }
    PrepareWorkspace(int32_t num_nodes, int64_t num_edges, bool sorted) {
        size_t at = 0;
        auto take = [&](size_t bytes) { const size_t here = at; at += align_up(bytes); return here; };
        order = take(e3j_amd_order_workspace_bytes(num_nodes));
        unsorted = take(sizeof(int32_t) * kMaxRowsBlocks);
        sort_bytes = sorted ? 0 : own_sort(num_nodes, num_edges) ? sizeof(int32_t) * kSortChunks * kSortDigits
                                                                 : sort_temp_bytes(num_edges);
        sort_temp = take(sort_bytes);
        const size_t list = sorted ? 0 : sizeof(int32_t) * (size_t)num_edges;
        keys_in = take(list);
        keys_out = take(list);
        positions = take(list);
        total = at;
    }
};
}  // namespace

size_t e3j_amd_prepare_rows_workspace_bytes(int32_t num_nodes, int64_t num_edges, int32_t sorted) {
    if (num_nodes < 1 || num_edges < 1 || num_edges > 0x7fffffffLL) return 0;
    return PrepareWorkspace(num_nodes, num_edges, sorted != 0).total + 256;
}

int e3j_amd_prepare_rows(const int32_t *key, const int32_t *other, int64_t num_edges, int32_t num_nodes,
                         int32_t sorted, int32_t rounds, int32_t *perm, int32_t *other_out, int32_t *row_ptr,
                         int32_t *order, int32_t row_cap, int32_t row_piece, int32_t max_segments,
                         int32_t *segments, void *workspace, void *stream_) {
    if (num_nodes < 1 || num_nodes >= INT32_MAX || num_edges < 1 || num_edges > 0x7fffffffLL || rounds < 0 ||
        rounds > 64 || (segments != nullptr && (row_piece < 1 || row_cap < row_piece || max_segments < 0)))
        return set_error(E3J_AMD_INVALID_ARGUMENT, "prepare_rows: bad sizes");
    if (key == nullptr || other == nullptr || other_out == nullptr || row_ptr == nullptr || workspace == nullptr ||
        (!sorted && perm == nullptr))
        return set_error(E3J_AMD_INVALID_ARGUMENT, "prepare_rows: null operand");
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    unsigned char *ws = static_cast<unsigned char *>(workspace);
    ws += (256 - reinterpret_cast<uintptr_t>(ws) % 256) % 256;
    const PrepareWorkspace w(num_nodes, num_edges, sorted != 0);
    int32_t *unsorted = reinterpret_cast<int32_t *>(ws + w.unsorted);
    const int blocks = (int)std::min<int64_t>((num_edges + 255) / 256, kMaxRowsBlocks);
    bool listed = false;  // pieces listed by the launches below
    int rc = E3J_AMD_OK;
    if (!sorted) {
        int32_t *keys_in = reinterpret_cast<int32_t *>(ws + w.keys_in);
        int32_t *keys_out = reinterpret_cast<int32_t *>(ws + w.keys_out);
        int32_t *positions = reinterpret_cast<int32_t *>(ws + w.positions);
        int bits = 1;  // the keys reach num_nodes
        while (bits < 32 && ((int64_t)1 << bits) <= (int64_t)num_nodes) bits++;
        if (PrepareWorkspace::own_sort(num_nodes, num_edges)) {
            int32_t *digits = reinterpret_cast<int32_t *>(ws + w.sort_temp);
            const dim3 chunks((unsigned)((num_edges + kSortChunk - 1) / kSortChunk)), threads(kBlockThreads);
            const int low = (bits + 1) / 2, high = bits - low > 0 ? bits - low : 1;
            const int32_t *here = nullptr;
            hipLaunchKernelGGL(edge_digits_kernel, chunks, threads, 0, stream, key, num_edges, num_nodes, true, 0,
                               (1u << low) - 1, digits);
            hipLaunchKernelGGL(edge_scatter_kernel, chunks, threads, 0, stream, key, here, num_edges, num_nodes, true, 0,
                               low, digits, keys_in, positions);
            hipLaunchKernelGGL(edge_digits_kernel, chunks, threads, 0, stream, keys_in, num_edges, num_nodes, false, low,
                               (1u << high) - 1, digits);
            hipLaunchKernelGGL(edge_scatter_kernel, chunks, threads, 0, stream, keys_in, positions, num_edges, num_nodes,
                               false, low, high, digits, keys_out, perm);
            rc = check_hip(hipGetLastError(), "prepare_rows sort");
        } else {
            hipLaunchKernelGGL(sort_input_kernel, dim3(grid_for(num_edges)), dim3(256), 0, stream, key, num_edges,
                               num_nodes, keys_in, positions);
            rc = check_hip(hipGetLastError(), "prepare_rows keys");
            if (rc) return rc;
            size_t temp_bytes = w.sort_bytes;
            rc = check_hip(hipcub::DeviceRadixSort::SortPairs(
                               ws + w.sort_temp, temp_bytes, reinterpret_cast<const uint32_t *>(keys_in),
                               reinterpret_cast<uint32_t *>(keys_out), positions, perm, (int)num_edges, 0, bits, stream),
                           "prepare_rows sort");
        }
        if (rc) return rc;
        hipLaunchKernelGGL(rows_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, keys_out, other, perm, num_edges,
                           num_nodes, other_out, row_ptr, static_cast<int32_t *>(nullptr), segments);
    } else if (num_edges <= kRowsBlockEdges) {
        listed = order == nullptr;
        hipLaunchKernelGGL(rows_block_kernel, dim3(1), dim3(kBlockThreads), 0, stream, key, other, num_edges,
                           num_nodes, other_out, row_ptr, listed, row_cap, row_piece, max_segments, segments);
    } else {
        hipLaunchKernelGGL(rows_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, key, other,
                           static_cast<const int32_t *>(nullptr), num_edges, num_nodes, other_out, row_ptr, unsorted,
                           segments);
        hipLaunchKernelGGL(recount_rows_kernel, dim3(1), dim3(kBlockThreads), 0, stream, key, num_edges, num_nodes,
                           unsorted, blocks, row_ptr);
    }
    rc = check_hip(hipGetLastError(), "prepare_rows");
    if (rc) return rc;
    if (order != nullptr)
        return locality_order(other_out, row_ptr, num_nodes, rounds, order,
                              PieceList{row_cap, row_piece, max_segments, segments}, ws + w.order, stream);
    if (segments != nullptr && !listed) {
        hipLaunchKernelGGL(row_segments_kernel, dim3((unsigned)(((int64_t)num_nodes + 255) / 256)), dim3(256), 0,
                           stream, row_ptr, num_nodes, row_cap, row_piece, max_segments, segments);
        rc = check_hip(hipGetLastError(), "prepare_rows pieces");
    }
    return rc;
}

int64_t e3j_amd_tile_schedule_num_work(int32_t num_nodes, int64_t num_edges, int32_t tile_rows,
                                       int32_t max_work_edges) {
    if (num_nodes < 0 || num_edges < 0 || tile_rows < 1 || max_work_edges < 1) return 0;
    const int64_t tiles = ((int64_t)num_nodes + tile_rows - 1) / tile_rows;
    return tiles + num_edges / max_work_edges;  // sum over tiles of max(1, ceil(count / max)) at most
}

size_t e3j_amd_tile_schedule_workspace_bytes(int32_t num_nodes, int64_t num_edges, int32_t tile_rows) {
    if (num_nodes < 0 || num_edges < 0 || tile_rows < 1) return 0;
    (void)num_edges;
    return TileWorkspace(num_nodes, tile_rows).total + 256;
}

int e3j_amd_tile_schedule_build(const int32_t *other, const int32_t *row_ptr, const int32_t *edge_perm,
                                const int32_t *row_order, int32_t num_nodes, int64_t num_edges,
                                int32_t tile_rows, int32_t max_work_edges, int32_t *work,
                                int32_t *t_sender, int32_t *t_edge, int32_t *t_local, void *workspace,
                                void *stream_) {
    if (num_nodes < 0 || num_edges < 0 || num_edges > 0x7fffffffLL || tile_rows < 1 || tile_rows > 65535 ||
        max_work_edges < 1)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "tile_schedule_build: bad sizes");
    if (num_nodes == 0) return E3J_AMD_OK;
    if (row_ptr == nullptr || work == nullptr || workspace == nullptr ||
        (num_edges > 0 && (other == nullptr || t_sender == nullptr || t_edge == nullptr || t_local == nullptr)))
        return set_error(E3J_AMD_INVALID_ARGUMENT, "tile_schedule_build: null operand");
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    unsigned char *ws = static_cast<unsigned char *>(workspace);
    ws += (256 - reinterpret_cast<uintptr_t>(ws) % 256) % 256;
    const TileWorkspace w(num_nodes, tile_rows);
    uint64_t *packed = reinterpret_cast<uint64_t *>(ws + w.packed);
    const int num_tiles = (num_nodes + tile_rows - 1) / tile_rows;
    const unsigned tiles_grid = (unsigned)((num_tiles + 255) / 256);

    int rc = E3J_AMD_OK;
    if (num_tiles <= kBlockThreads * kTileItems) {
        hipLaunchKernelGGL(tile_plan_block_kernel, dim3(1), dim3(kBlockThreads), 0, stream, row_order, row_ptr,
                           num_nodes, tile_rows, num_tiles, max_work_edges, packed, work);
    } else {
        hipLaunchKernelGGL(tile_count_kernel, dim3(tiles_grid), dim3(256), 0, stream, row_order, row_ptr, num_nodes,
                           tile_rows, num_tiles, max_work_edges, packed);
        rc = check_hip(hipGetLastError(), "tile schedule counts");
        if (rc) return rc;
        size_t temp_bytes = w.temp_bytes;
        rc = check_hip(hipcub::DeviceScan::InclusiveSum(ws + w.temp, temp_bytes, packed, packed, num_tiles + 1,
                                                        stream),
                       "tile schedule scan");
        if (rc) return rc;
        hipLaunchKernelGGL(tile_work_kernel, dim3(tiles_grid), dim3(256), 0, stream, packed, num_tiles,
                           max_work_edges, work);
    }
    rc = check_hip(hipGetLastError(), "tile schedule work");
    if (rc || num_edges == 0) return rc;
    // the lists: a workgroup per tile where a tile is longer than a wave (each of its threads then counts the
    // keys below one or two), a wave per tile where it is not
    const bool wide = num_edges > 64ll * num_tiles;
    hipLaunchKernelGGL(wide ? tile_lists_kernel<4> : tile_lists_kernel<1>,
                       dim3((unsigned)(wide ? num_tiles : (num_tiles + 3) / 4)), dim3(256), 0, stream, other, row_ptr,
                       edge_perm, row_order, packed, num_nodes, num_edges, tile_rows, num_tiles, t_sender, t_edge,
                       t_local);
    return check_hip(hipGetLastError(), "tile schedule lists");
}

int e3j_amd_sort_edges(const int32_t *key, const int32_t *other, int64_t num_edges,
                       int32_t num_nodes, int32_t *perm, int32_t *other_sorted, int32_t *row_ptr,
                       void *workspace, void *stream_) {
    if (num_nodes < 0 || num_edges < 0 || num_edges > 0x7fffffffLL)
        return set_error(E3J_AMD_INVALID_ARGUMENT, "sort_edges: bad sizes");
    if (row_ptr == nullptr || workspace == nullptr ||
        (num_edges > 0 && (key == nullptr || other == nullptr || perm == nullptr || other_sorted == nullptr)))
        return set_error(E3J_AMD_INVALID_ARGUMENT, "sort_edges: null operand");
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    unsigned char *ws = static_cast<unsigned char *>(workspace);
    const size_t scan_bytes = scan_temp_bytes(num_nodes);
    const size_t sort_bytes = sort_temp_bytes(num_edges);
    void *scan_temp = ws;
    void *sort_temp = ws + align_up(scan_bytes);
    uint32_t *keys_out = reinterpret_cast<uint32_t *>(ws + align_up(scan_bytes) + align_up(sort_bytes));
    int32_t *iota = reinterpret_cast<int32_t *>(reinterpret_cast<unsigned char *>(keys_out) +
                                                align_up(sizeof(int32_t) * (size_t)num_edges));
    int rc = row_ptr_impl(key, num_edges, num_nodes, row_ptr, scan_temp, scan_bytes, stream);
    if (rc || num_edges == 0) return rc;
    hipLaunchKernelGGL(iota_kernel, dim3(grid_for(num_edges)), dim3(256), 0, stream, iota, num_edges);
    rc = check_hip(hipGetLastError(), "sort iota launch");
    if (rc) return rc;
    size_t temp_bytes = sort_bytes;
    rc = check_hip(hipcub::DeviceRadixSort::SortPairs(sort_temp, temp_bytes,
                                                      reinterpret_cast<const uint32_t *>(key), keys_out,
                                                      iota, perm, (int)num_edges, 0, 32, stream),
                   "edge sort");
    if (rc) return rc;
    hipLaunchKernelGGL(gather_kernel, dim3(grid_for(num_edges)), dim3(256), 0, stream, other, perm,
                       other_sorted, num_edges);
    return check_hip(hipGetLastError(), "sort gather launch");
}

}  // extern "C"
