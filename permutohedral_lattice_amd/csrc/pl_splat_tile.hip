// The splat of rows of many channels for a lattice whose build merged its tiles: the rows of sums of
// a workgroup's points meet in LDS before they go to the vertex table.
// (reference: src/PermutohedralLatticeCPU.h:306-331, one row per point and corner)
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pl_device.h"
#include "pl_kernels.h"

namespace plk {

namespace {

using namespace device;

// A workgroup's 256 points have 256 * d1 (corner, vertex) pairs but only about a hundred distinct
// vertices, which they name by a place in the workgroup's table.  The pairs are sorted by place with a
// counting sort in LDS -- each pair's rank comes back from the count of its place -- and 32 groups of sixteen lanes, a lane on channels c, c + 16, ..., then run over their share of
// the sorted pairs each: weight times the point's row (in LDS, loaded once) into registers until the
// vertex changes, and one request per line of the vertex's row then.
// What bounds it is the instructions of that last loop and the requests to the L2 atomic unit, about
// 130 rows a workgroup.  k_splat_channels, which takes a wavefront's pairs vertex by vertex, loads the
// rows once per two corners and sends a row per wavefront and vertex (about 165): 2 x 321x481 points, pd = 5,
// vd = 22: 37.0 us a launch, this 25.5 (26.5 when it looked its vertices up in a table of hashes first).
// After a merging build only (TileVertices).
// Two threads to a point, which share its corners (one thread to a point, 16 groups of lanes: 27.6 us).
constexpr unsigned kSides = 2, kThreads = kSides * kBlock;
constexpr unsigned kMaxCorners = (kMaxPd + 1 + kSides - 1) / kSides;   // of a thread

template <int K>
__device__ __forceinline__ void splat_tile_of(uint2 *sorted, int d1, int vd, const PointMap &map,
                                              const float *__restrict__ input, int in_channels,
                                              const ReplayEntry *__restrict__ replay, float *values, int xcd_aware,
                                              unsigned block, unsigned blocks) {
    // sorted: [kBlock * d1]: weight, point | slot << 8; then the points' rows
    __shared__ int slot_index[kTileSlots];
    __shared__ unsigned slot_count[kTileSlots];
    __shared__ unsigned wave_pairs[kThreads / 64];
    unsigned vblock;
    if (!block_of_points(map, xcd_aware, block, blocks, vblock)) return;
    float *rows = reinterpret_cast<float *>(sorted + (size_t)kBlock * d1);   // [kBlock][in_channels]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int point = tid % kBlock, side = tid / kBlock;   // (its corners: side, side + 2, ...)
    const int n = point_of_thread(map, vblock, point);
    static_assert(kTileSlots == kThreads, "a slot per thread");
    const uint32_t *words = words_of_tile(replay, vblock, d1);
    const int used = map.tile_vertices.used[vblock];
    const int own_vertex = map.tile_vertices.of(vblock)[tid];
    slot_count[tid] = 0u;

    int index[kMaxCorners];
    float weight[kMaxCorners];
#pragma unroll
    for (int i = 0; i < (int)kMaxCorners; ++i) {
        const int r = (int)kSides * i + side;
        const uint32_t place = place_of_corner(words[(r < d1 ? r / kPlacesPerWord : 0) * kBlock + point], r);
        index[i] = r < d1 && n >= 0 && place < (uint32_t)kTileSlots ? (int)place : -1;
        weight[i] = weights_behind(words, d1)[(r < d1 ? r : 0) * kBlock + point];
    }
    // element i of the wavefront's 64 rows belongs to point i / in_channels, channel i % in_channels
    // (eight loads asked for before the first is stored; a point without data reads point 0; the two
    // wavefronts of the same points take every other 64 elements)
    {
        float *wave_rows = rows + (size_t)(wave % (kBlock / 64)) * 64 * in_channels;
        const int e0 = lane + 64 * side;
        int p = e0 / in_channels, c = e0 - p * in_channels;
        const int step_p = (64 * (int)kSides) / in_channels, step_c = 64 * (int)kSides - step_p * in_channels;
        constexpr int kBatch = 8, kStep = 64 * (int)kSides;
        for (int i0 = e0; i0 < 64 * in_channels; i0 += kStep * kBatch) {
            float x[kBatch];
            bool has[kBatch];
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const bool inside = i0 + kStep * k < 64 * in_channels;
                const int np = __shfl(n, inside ? p : 0);
                has[k] = inside && np >= 0;
                x[k] = input[(size_t)(has[k] ? np : 0) * in_channels + (has[k] ? c : 0)];
                p += step_p;
                c += step_c;
                if (c >= in_channels) {
                    c -= in_channels;
                    p += 1;
                }
            }
#pragma unroll
            for (int k = 0; k < kBatch; ++k) asm volatile("" : "+v"(x[k]));
#pragma unroll
            for (int k = 0; k < kBatch; ++k)
                if (i0 + kStep * k < 64 * in_channels) wave_rows[i0 + kStep * k] = has[k] ? x[k] : 0.0f;
        }
    }
    __syncthreads();   // the slots are empty (and the rows there)

    // place[r]: the slot of corner r's vertex (its place in the table) and, above it, the pair's rank among
    // the slot's.  The first lane of a run of lanes with one vertex counts for the run (8x8
    // pixels: 29 runs; LDS atomics on one address take turns).
    unsigned place[kMaxCorners];
    constexpr unsigned kNoPair = 0xffffffffu;
#pragma unroll
    for (int r = 0; r < (int)kMaxCorners; ++r) {
        const int before = __shfl_up(index[r], 1);
        const bool opens = lane == 0 || before != index[r];
        const uint64_t opening = wave_ballot(opens);
        const uint64_t behind = lane == 63 ? 0ull : opening >> (lane + 1);
        const unsigned length = behind ? (unsigned)__builtin_ctzll(behind) + 1u : 64u - (unsigned)lane;
        unsigned found = kNoPair;
        if (opens && index[r] >= 0) found = (unsigned)index[r] | atomicAdd(&slot_count[index[r]], length) << 16;
        const int opener = 63 - __builtin_clzll(opening & (~0ull >> (63 - lane)));
        found = (unsigned)__shfl((int)found, opener);
        place[r] = index[r] >= 0 && found != kNoPair ? found + ((unsigned)(lane - opener) << 16) : kNoPair;
    }
    __syncthreads();   // the slots are counted

    // the count of a slot becomes the place of its first pair (a thread takes one slot)
    const unsigned own_count = slot_count[tid];
    unsigned inclusive = own_count;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned other = __shfl_up(inclusive, d);
        if (lane >= d) inclusive += other;
    }
    if (lane == 63) wave_pairs[wave] = inclusive;
    __syncthreads();
    unsigned before = inclusive - own_count, pairs = 0;
#pragma unroll
    for (int w = 0; w < (int)kThreads / 64; ++w) {
        if (w < wave) before += wave_pairs[w];
        pairs += wave_pairs[w];
    }
    slot_count[tid] = before;
    slot_index[tid] = tid < used ? own_vertex : -1;
    __syncthreads();

#pragma unroll
    for (int r = 0; r < (int)kMaxCorners; ++r) {
        if (place[r] == kNoPair) continue;
        const unsigned slot = place[r] & 0xffffu;
        sorted[slot_count[slot] + (place[r] >> 16)] =
            make_uint2(__float_as_uint(weight[r]), (unsigned)point | slot << 8);
    }
    __syncthreads();   // the pairs are in the order of their slots

    constexpr unsigned kGroups = kThreads / 16;
    const unsigned per = (pairs + kGroups - 1u) / kGroups;
    const unsigned from = (unsigned)(tid >> 4) * per;
    const unsigned to = from + per < pairs ? from + per : pairs;
    if (from >= to) return;
    const int c0 = tid & 15;
    float acc[K];
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = 0.0f;
    auto add_row = [&](unsigned slot) {
        const int vertex = slot_index[slot];
        float *row = values + (unsigned)vertex * (unsigned)vd;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (vertex >= 0 && c0 + 16 * k < vd) atomicAdd(row + c0 + 16 * k, acc[k]);
            acc[k] = 0.0f;
        }
    };
    unsigned current = sorted[from].y >> 8;
    constexpr unsigned kAhead = 8;   // pairs whose rows are asked for together
    for (unsigned i0 = from; i0 < to; i0 += kAhead) {
        uint2 pair[kAhead];
        float x[kAhead][K];
#pragma unroll
        for (unsigned j = 0; j < kAhead; ++j) pair[j] = sorted[i0 + j < to ? i0 + j : to - 1u];
#pragma unroll
        for (unsigned j = 0; j < kAhead; ++j) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int c = c0 + 16 * k;
                const float value = rows[(int)(pair[j].y & 255u) * in_channels + (c < in_channels ? c : 0)];
                x[j][k] = c < in_channels ? value : 1.0f;
            }
        }
#pragma unroll
        for (unsigned j = 0; j < kAhead; ++j) {
            const unsigned slot = pair[j].y >> 8;
            if (slot != current) {
                add_row(current);
                current = slot;
            }
            // (past the end: the last pair again, not counted)
            const float w = __uint_as_float(pair[j].x);
#pragma unroll
            for (int k = 0; k < K; ++k) acc[k] = i0 + j < to ? acc[k] + w * x[j][k] : acc[k];
        }
    }
    add_row(current);
}
template <int K>
__global__ __launch_bounds__(kThreads) void k_splat_tile(int d1, int vd, PointMap map, const float *__restrict__ input,
                                                        int in_channels, const ReplayEntry *__restrict__ replay,
                                                        float *values, int xcd_aware) {
    extern __shared__ uint2 sorted[];
    splat_tile_of<K>(sorted, d1, vd, map, input, in_channels, replay, values, xcd_aware, blockIdx.x, gridDim.x);
}
// The same for several lattices.
template <int K>
__global__ __launch_bounds__(kThreads) void k_splat_tiles(Items<PointsWork, kJointItems> items, int d1, int vd,
                                                         int in_channels, int xcd_aware) {
    extern __shared__ uint2 sorted[];
    unsigned block, blocks;
    const PointsWork &work = item_of(items, block, blocks);
    if (block >= work.map.n_blocks) return;
    splat_tile_of<K>(sorted, d1, vd, work.map, work.input, in_channels, work.replay, work.values, xcd_aware, block,
                     work.map.n_blocks);
}

}  // namespace

hipError_t splat_tile(int pd, int vd, const PointMap &map, const float *input, int in_channels, const ReplayEntry *replay,
                      float *values, int xcd_aware, hipStream_t s) {
    if (map.n_blocks == 0) return hipSuccess;
    if (!map.tile_vertices.table || !splat_tile_takes(vd) || pd < 1 || pd > kMaxPd || in_channels < 1 || in_channels > vd)
        return hipErrorInvalidValue;
    const int d1 = pd + 1;
    const size_t lds = kBlock * ((size_t)d1 * sizeof(uint2) + (size_t)in_channels * sizeof(float));
    const auto kernel = vd <= 16 ? k_splat_tile<1> : k_splat_tile<2>;
    hipLaunchKernelGGL(kernel, dim3(map.n_blocks), dim3(kThreads), lds, s, d1, vd, map, input, in_channels, replay,
                       values, xcd_aware);
    return hipGetLastError();
}

hipError_t splat_tile_joint(int pd, int vd, int n, const PointsWork *work, int in_channels, int xcd_aware, hipStream_t s) {
    if (!splat_tile_takes(vd) || pd < 1 || pd > kMaxPd || in_channels < 1 || in_channels > vd || n < 1 || n > kJointItems)
        return hipErrorInvalidValue;
    const Items<PointsWork, kJointItems> items = items_of_points<kJointItems>(n, work);
    const int d1 = pd + 1;
    const size_t lds = kBlock * ((size_t)d1 * sizeof(uint2) + (size_t)in_channels * sizeof(float));
    const auto kernel = vd <= 16 ? k_splat_tiles<1> : k_splat_tiles<2>;
    hipLaunchKernelGGL(kernel, dim3(all_blocks(items)), dim3(kThreads), lds, s, items, d1, vd, in_channels, xcd_aware);
    return hipGetLastError();
}

}  // namespace plk
