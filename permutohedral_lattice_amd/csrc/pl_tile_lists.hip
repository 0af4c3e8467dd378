// The splat of a lattice whose build merged its tiles and that is applied many times.
//
// pl_gather.hip lists, per vertex, all (point, corner) rows that name it, and an apply gathers every
// point's values once a corner.  After a merging build the points of a workgroup share their vertices, so
// here an apply sums in two steps: a workgroup brings its 256 points' values to LDS, each read once, and sums
// them per vertex of its table (its corners sorted by vertex when the lattice is built); then every vertex
// adds up the rows of the workgroups that touch it.  No atomics, no zero fill, and sums in one order on every
// call.  (reference: src/PermutohedralLatticeCPU.h:306-331)
//
// us, lists of corners (pl_gather.hip) and this: an apply's splat of 1024x1024 points, pd 5, vd 4, 27.8 and 24.0
// (19.1 and 4.9 for the two steps); of two pairs of lattices of 512x512 points, pd 5 and 2, 21 classes, 63 and
// 52 (40.5 and 11.6); the lists themselves, 1024x1024 points, 67 and 45.
#include "pl_device.h"
#include "pl_kernels.h"

namespace plk {

namespace {

using namespace device;


// ------------------------------------------------------------------------------------------------
// When the lattice is built: every workgroup's corners sorted by their places in its table, 64 * 4 * D1 of
// them, and every row of sums' rank among its vertex's.  An entry: the weight; the point (8 bits), the
// place (10, kNoPlace: no corner) and the entry's rank in its run of entries of one place, counted within
// its 64 (6 bits from bit 18).
// ------------------------------------------------------------------------------------------------
constexpr unsigned kEntryPlace = 8, kEntryRank = kEntryPlace + kPlaceBits;
__device__ __forceinline__ unsigned entry_point(unsigned y) { return y & 0xffu; }
__device__ __forceinline__ unsigned entry_place(unsigned y) { return (y >> kEntryPlace) & kNoPlace; }
__device__ __forceinline__ unsigned entry_rank(unsigned y) { return y >> kEntryRank; }

template <int D1>
__global__ __launch_bounds__(kBlock) void k_sort_tile(PointMap map, const ReplayEntry *__restrict__ replay,
                                                       uint2 *entries, unsigned *count, unsigned *row_rank,
                                                       int max_vertices) {
    __shared__ uint2 sorted[kBlock * D1];
    __shared__ unsigned place_count[kTileSlots];
    __shared__ unsigned wave_sum[kBlock / 64];
    unsigned vblock;
    if (!block_of_points(map, 1, vblock)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = point_of_thread(map, vblock, tid);
    const uint32_t *words = words_of_tile(replay, vblock, D1);
    uint32_t word[replay_words(D1)];
    float weight[D1];
#pragma unroll
    for (int w = 0; w < replay_words(D1); ++w) word[w] = words[w * kBlock + tid];
#pragma unroll
    for (int r = 0; r < D1; ++r) weight[r] = weights_behind(words, D1)[r * kBlock + tid];
    const int used = map.tile_vertices.used[vblock];
    const int *table = map.tile_vertices.of(vblock);
    static_assert(kTileSlots == 2 * kBlock, "two places a thread");
    const int vertex[2] = {table[2 * tid], table[2 * tid + 1]};
    place_count[2 * tid] = place_count[2 * tid + 1] = 0u;
    for (int i = tid; i < kBlock * D1; i += kBlock) sorted[i] = make_uint2(0u, kNoPlace << kEntryPlace);
    __syncthreads();
    // (the first lane of a run of lanes with one place counts for the run, as in k_splat_tile)
    unsigned at[D1];
#pragma unroll
    for (int r = 0; r < D1; ++r) {
        const unsigned p = place_of_corner(word[r / kPlacesPerWord], r);
        const int place = n >= 0 && p < (unsigned)kTileSlots ? (int)p : -1;
        const int before = __shfl_up(place, 1);
        const uint64_t opening = wave_ballot(lane == 0 || before != place);
        const uint64_t behind = lane == 63 ? 0ull : opening >> (lane + 1);
        const unsigned length = behind ? (unsigned)__builtin_ctzll(behind) + 1u : 64u - (unsigned)lane;
        const int opener = 63 - __builtin_clzll(opening & (~0ull >> (63 - lane)));
        unsigned base = 0u;
        if (opener == lane && place >= 0) base = atomicAdd(&place_count[place], length);
        base = (unsigned)__shfl((int)base, opener);
        at[r] = place >= 0 ? (unsigned)place << 16 | (base + (unsigned)(lane - opener)) : ~0u;
    }
    __syncthreads();
    const unsigned own[2] = {place_count[2 * tid], place_count[2 * tid + 1]};
    unsigned inclusive = own[0] + own[1];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned other = __shfl_up(inclusive, d);
        if (lane >= d) inclusive += other;
    }
    if (lane == 63) wave_sum[wave] = inclusive;
    __syncthreads();
    unsigned first = inclusive - own[0] - own[1];
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w)
        if (w < wave) first += wave_sum[w];
    place_count[2 * tid] = first;
    place_count[2 * tid + 1] = first + own[0];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < D1; ++r) {
        if (at[r] == ~0u) continue;
        const unsigned place = at[r] >> 16, from = place_count[place], i = from + (at[r] & 0xffffu);
        const unsigned chunk = i & ~63u, rank = i - (from > chunk ? from : chunk);
        sorted[i] = make_uint2(__float_as_uint(weight[r]), (unsigned)tid | place << kEntryPlace | rank << kEntryRank);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < D1; ++i) entries[(size_t)vblock * kBlock * D1 + i * kBlock + tid] = sorted[i * kBlock + tid];
    // (a vertex number beyond the table cannot come out of a build that fitted)
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (2 * tid + i < used && (unsigned)vertex[i] < (unsigned)max_vertices)
            row_rank[(size_t)vblock * kTileSlots + 2 * tid + i] = atomicAdd(&count[vertex[i]], 1u);
}

// (behind the scan of the counts: start[v] is the first of v's rows)
__global__ __launch_bounds__(kBlock) void k_place_rows(PointMap map, const unsigned *__restrict__ start, unsigned *row_of) {
    unsigned vblock;
    if (!block_of_points(map, 1, vblock)) return;
    const int used = map.tile_vertices.used[vblock];
    const int *table = map.tile_vertices.of(vblock);
    for (int i = threadIdx.x; i < used; i += kBlock) {
        const int v = table[i];
        if (v >= 0) row_of[(size_t)vblock * kTileSlots + i] += start[v];
    }
}

// ------------------------------------------------------------------------------------------------
// An apply, step 1: the rows of sums of a workgroup's points, whose values lie in LDS.
//
// Up to four channels: the entries, in the order of their places, are dealt out 64 at a time, consecutive
// ones to a wavefront, a lane an entry: weight times the point's values, summed along the runs of one place by
// sum_groups_in_order, and the last lane of a run stores the row.  A run that continues in the wavefront's
// next 64 hands its sum on; one that continues in the next wavefront's is completed by the wavefront it
// began in, which adds what the others have left in LDS (`head`) after a barrier.
// ------------------------------------------------------------------------------------------------
template <int VD>
constexpr int kFewStride = VD == 2 ? 2 : 4;   // floats of a point's values in LDS

// (lane l's sums over its run up to it, without the products by 0 and 1)
template <int VD>
__device__ __forceinline__ void sum_runs_plainly(float (&x)[VD], int rank) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
#pragma unroll
        for (int j = 0; j < VD; ++j) {
            const float other = __shfl_up(x[j], off);
            x[j] += rank >= off ? other : 0.0f;
        }
    }
}
template <int VD>
__device__ __forceinline__ void store_few(float *row, const float (&x)[VD]) {
    if constexpr (VD == 4) {
        *reinterpret_cast<float4 *>(row) = make_float4(x[0], x[1], x[2], x[3]);
    } else if constexpr (VD == 2) {
        *reinterpret_cast<float2 *>(row) = make_float2(x[0], x[1]);
    } else {
#pragma unroll
        for (int j = 0; j < VD; ++j) row[j] = x[j];
    }
}
// IN: channels of an input row, VD - 1 (the last channel is the bare weight) or VD
template <int VD, int IN, int D1>
__global__ __launch_bounds__(kBlock) void k_splat_rows(PointMap map, const uint2 *__restrict__ entries,
                                                        const unsigned *__restrict__ row_of_place,
                                                        const float *__restrict__ input, float *rows) {
    struct alignas(IN == 3 ? 4 : 4 * IN) InputRow {
        float c[IN];
    };
    constexpr int kWaves = kBlock / 64;
    __shared__ float values[kBlock * kFewStride<VD>];
    __shared__ unsigned row_of[kTileSlots];
    __shared__ float head[kWaves][VD];
    __shared__ bool head_goes_on[kWaves];
    unsigned vblock;
    if (!block_of_points(map, 1, vblock)) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the wavefront's D1 times 64 entries, and the places of the entries beside them
    const uint2 *mine = entries + ((size_t)vblock * kWaves + (unsigned)wave) * (64 * D1);
    uint2 e[D1];
#pragma unroll
    for (int c = 0; c < D1; ++c) e[c] = mine[c * 64 + lane];
    const unsigned beside_before = mine[wave > 0 ? -1 : 0].y, beside_behind = mine[wave + 1 < kWaves ? 64 * D1 : 0].y;
    // (of places that are not used: anything; there is memory for kTileSlots)
    static_assert(kTileSlots == 2 * kBlock, "two places a thread");
    const uint2 two = reinterpret_cast<const uint2 *>(row_of_place + (size_t)vblock * kTileSlots)[tid];
    const int n = point_of_thread(map, vblock, tid);
    const InputRow in = reinterpret_cast<const InputRow *>(input)[n >= 0 ? n : 0];
    float x[kFewStride<VD>];
    bool finite = true;
#pragma unroll
    for (int j = 0; j < kFewStride<VD>; ++j) {
        x[j] = j < IN ? (n >= 0 ? in.c[j < IN ? j : 0] : 0.0f) : j < VD ? 1.0f : 0.0f;
        finite = finite && __builtin_fabsf(x[j]) < 1e29f;
    }
    reinterpret_cast<uint2 *>(row_of)[tid] = two;
    if constexpr (VD == 2)
        reinterpret_cast<float2 *>(values)[tid] = make_float2(x[0], x[1]);
    else
        reinterpret_cast<float4 *>(values)[tid] = make_float4(x[0], x[1], x[2], x[3]);
    if (lane == 0) head_goes_on[wave] = false;
    // (sums of up to 256 values below 1e29 times weights of at most one are far from overflowing)
    const bool tame = __syncthreads_or(!finite) == 0;

    const unsigned before = wave > 0 ? entry_place(beside_before) : kNoPlace;
    const unsigned behind = wave + 1 < kWaves ? entry_place(beside_behind) : kNoPlace;
    // (the run of the first entry began in an earlier wavefront's, and none has ended here yet)
    bool in_head = before != kNoPlace && before == entry_place((unsigned)lane_value((int)e[0].y, 0));
    bool open = false;             // the last entry's run goes on in the next wavefront's, and began here
    unsigned open_place = 0;
    float carry[VD];               // of the run that goes on
    const float is_first = lane == 0 ? 1.0f : 0.0f;
#pragma unroll
    for (int j = 0; j < VD; ++j) carry[j] = 0.0f;
#pragma unroll
    for (int c = 0; c < D1; ++c) {
        const unsigned y = e[c].y, place = entry_place(y), rank = entry_rank(y);
        const unsigned last = entry_place((unsigned)lane_value((int)y, 63));
        const unsigned next = c + 1 < D1 ? entry_place((unsigned)lane_value((int)e[c + 1 < D1 ? c + 1 : c].y, 0)) : behind;
        const bool goes_on = last != kNoPlace && next == last;
        const float w = __uint_as_float(e[c].x);
        const float *value = values + entry_point(y) * kFewStride<VD>;
        float sum[VD];
        if constexpr (VD == 2) {
            const float2 v = *reinterpret_cast<const float2 *>(value);
            sum[0] = v.x * w, sum[1] = v.y * w;
        } else {
            const float4 v = *reinterpret_cast<const float4 *>(value);
            const float four[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < VD; ++j) sum[j] = four[j] * w;
        }
        if (tame) {
            if (c > 0) {
#pragma unroll
                for (int j = 0; j < VD; ++j) sum[j] = __builtin_fmaf(carry[j], is_first, sum[j]);
            }
            sum_groups_in_order(sum, steps_that_count(lane, rank));
        } else {
#pragma unroll
            for (int j = 0; j < VD; ++j) sum[j] += lane == 0 ? carry[j] : 0.0f;
            sum_runs_plainly<VD>(sum, (int)rank);
        }
#pragma unroll
        for (int j = 0; j < VD; ++j) carry[j] = goes_on ? __int_as_float(lane_value(__float_as_int(sum[j]), 63)) : 0.0f;
        // (wave_shl:1, a zero above lane 63)
        const unsigned above = (unsigned)__builtin_amdgcn_update_dpp(0, (int)rank, 0x130, 0xf, 0xf, true);
        const bool ends = above == 0u && place != kNoPlace && !(lane == 63 && goes_on);
        if (ends) {
            if (in_head && rank == (unsigned)lane) {
#pragma unroll
                for (int j = 0; j < VD; ++j) head[wave][j] = sum[j];
            } else {
                store_few<VD>(rows + (size_t)row_of[place] * VD, sum);
            }
        }
        if (wave_ballot(ends) != 0) in_head = false;
        if (c + 1 == D1 && goes_on) {
            // the rest of an earlier wavefront's run, all of it, or the start of one that is completed here
            open = !in_head;
            open_place = last;
            if (in_head && lane == 0) {
                head_goes_on[wave] = true;
#pragma unroll
                for (int j = 0; j < VD; ++j) head[wave][j] = carry[j];
            }
        }
    }
    __syncthreads();
    if (!open || lane != 0) return;
    for (int w = wave + 1; w < kWaves; ++w) {
#pragma unroll
        for (int j = 0; j < VD; ++j) carry[j] += head[w][j];
        if (!head_goes_on[w]) break;
    }
    store_few<VD>(rows + (size_t)row_of[open_place] * VD, carry);
}

// More channels: 128 groups of four lanes, which share a row's C channels, run over 2 * D1 consecutive
// entries each: weight times the point's values until the place changes, and the row is stored then.  Runs
// across groups as above.  Bound by what a workgroup waits for (24 wavefronts a CU) and its vector
// instructions, half of the time.  (Two pairs of 512x512 points, 21 classes: 40.5 us; sums across lanes as
// above 85; entries read behind the values' barrier 48.8; rows of 22 floats, not 24, and three 8-byte
// accesses a lane 51.5.)
constexpr int kManyThreads = 2 * kBlock, kQuads = kManyThreads / 4;
template <int C>
constexpr int kManyStride = C + 4;   // floats of a point's values in LDS
// A quad's lane I's x
template <int I>
__device__ __forceinline__ unsigned of_quad(unsigned x) {
    return (unsigned)__builtin_amdgcn_mov_dpp((int)x, I * 0x55, 0xf, 0xf, true);
}
__device__ __forceinline__ uint2 of_quad(uint2 e, int i) {
    return i == 0   ? make_uint2(of_quad<0>(e.x), of_quad<0>(e.y))
           : i == 1 ? make_uint2(of_quad<1>(e.x), of_quad<1>(e.y))
           : i == 2 ? make_uint2(of_quad<2>(e.x), of_quad<2>(e.y)) : make_uint2(of_quad<3>(e.x), of_quad<3>(e.y));
}
// The channels of a quad's lane of the C of a row: 4 sub .. (2 sub .. of eight), and behind the quad's first
// sixteen the rest alike, so that a quad's accesses are one stretch.
template <int C>
__device__ __forceinline__ void copy_floats(const float *row, int sub, float (&x)[C / 4]) {
    if constexpr (C == 8) {
        const float2 v = *reinterpret_cast<const float2 *>(row + 2 * sub);
        x[0] = v.x, x[1] = v.y;
    } else {
        const float4 v = *reinterpret_cast<const float4 *>(row + 4 * sub);
        x[0] = v.x, x[1] = v.y, x[2] = v.z, x[3] = v.w;
        if constexpr (C == 24) {
            const float2 u = *reinterpret_cast<const float2 *>(row + 16 + 2 * sub);
            x[4] = u.x, x[5] = u.y;
        } else if constexpr (C == 32) {
            const float4 u = *reinterpret_cast<const float4 *>(row + 16 + 4 * sub);
            x[4] = u.x, x[5] = u.y, x[6] = u.z, x[7] = u.w;
        }
    }
}
// (left: floats of the row from here on, a multiple of eight)
template <int C>
__device__ __forceinline__ void store_floats(float *row, int sub, int left, const float (&x)[C / 4]) {
    if constexpr (C == 8) {
        *reinterpret_cast<float2 *>(row + 2 * sub) = make_float2(x[0], x[1]);
    } else {
        if (4 * sub < left) *reinterpret_cast<float4 *>(row + 4 * sub) = make_float4(x[0], x[1], x[2], x[3]);
        if constexpr (C == 24) {
            *reinterpret_cast<float2 *>(row + 16 + 2 * sub) = make_float2(x[4], x[5]);
        } else if constexpr (C == 32) {
            if (16 + 4 * sub < left)
                *reinterpret_cast<float4 *>(row + 16 + 4 * sub) = make_float4(x[4], x[5], x[6], x[7]);
        }
    }
}
// A quad's entries of a workgroup's, a lane every fourth, and the places of the entries beside them
template <int D1>
struct QuadEntries {
    static constexpr int kPer = kBlock * D1 / kQuads, kLoads = (kPer + 3) / 4;
    uint2 e[kLoads];
    unsigned before, behind;
    __device__ __forceinline__ void load(const uint2 *__restrict__ entries) {
        const int sub = threadIdx.x & 3, quad = threadIdx.x >> 2;
        const uint2 *mine = entries + quad * kPer;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) e[i] = mine[4 * i + sub < kPer ? 4 * i + sub : 0];
        before = mine[quad > 0 ? -1 : 0].y;
        behind = mine[quad + 1 < kQuads ? kPer : 0].y;
    }
};
// (every thread of the workgroup, head and head_goes_on free: a barrier between two.  The workgroup's channels are from `from` on in the rows, which end before C where they have no multiple of it.)
template <int D1, int C>
__device__ __forceinline__ void sum_many_runs(const QuadEntries<D1> &entries, const float *values,
                                              const unsigned *row_of, float *rows, int from, int stride,
                                              float (*head)[C], unsigned char *head_goes_on) {
    constexpr int F = C / 4, kPer = QuadEntries<D1>::kPer;
    const int sub = threadIdx.x & 3, quad = threadIdx.x >> 2;
    const unsigned before = quad > 0 ? entry_place(entries.before) : kNoPlace;
    const unsigned behind = quad + 1 < kQuads ? entry_place(entries.behind) : kNoPlace;
    unsigned current = entry_place(of_quad<0>(entries.e[0].y));
    bool in_head = before != kNoPlace && before == current;
    bool changed = false;
    float acc[F];
#pragma unroll
    for (int j = 0; j < F; ++j) acc[j] = 0.0f;
    auto end_run = [&]() {
        if (in_head)
            store_floats<C>(head[quad], sub, C, acc);
        else if (current != kNoPlace)
            store_floats<C>(rows + (size_t)row_of[current] * stride + from, sub, stride - from, acc);
    };
    // (the values of four entries are asked for before the first is looked at)
#pragma unroll
    for (int i0 = 0; i0 < kPer; i0 += 4) {
        uint2 entry[4];
        float x[4][F];
#pragma unroll
        for (int i = 0; i < 4 && i0 + i < kPer; ++i) {
            entry[i] = of_quad(entries.e[i0 / 4], i);
            copy_floats<C>(values + entry_point(entry[i].y) * kManyStride<C>, sub, x[i]);
        }
#pragma unroll
        for (int i = 0; i < 4 && i0 + i < kPer; ++i) {
            const unsigned place = entry_place(entry[i].y);
            if (place != current) {
                end_run();
                in_head = false;
                changed = true;
                current = place;
#pragma unroll
                for (int j = 0; j < F; ++j) acc[j] = 0.0f;
            }
            const float w = __uint_as_float(entry[i].x);
#pragma unroll
            for (int j = 0; j < F; ++j) acc[j] = __builtin_fmaf(w, x[i][j], acc[j]);
        }
    }
    const bool goes_on = current != kNoPlace && behind == current, open = goes_on && !in_head;
    if (!open) end_run();
    // (all of a quad's entries are of the run that goes on)
    if (sub == 0) head_goes_on[quad] = goes_on && !changed;
    __syncthreads();
    if (open) {
        for (int q = quad + 1; q < kQuads; ++q) {
            float x[F];
            copy_floats<C>(head[q], sub, x);
#pragma unroll
            for (int j = 0; j < F; ++j) acc[j] += x[j];
            if (!head_goes_on[q]) break;
        }
        in_head = false;
        end_run();
    }
}

struct TileSplat {
    PointMap map;              // (its tile_vertices: a's)
    const uint2 *entries_a, *entries_b;
    const unsigned *row_of_a, *row_of_b;
    const float *input;
    float *rows_a, *rows_b;
};
// D1B: corners of a second lattice over the same points, 0: none.  workgroup (x, y): channels C y .. .  Rows of
// sums are `stride` floats apart.
template <int D1A, int D1B, int C, int N>
__global__ __launch_bounds__(kManyThreads) void k_splat_rows_channels(Items<TileSplat, N> items, int vd, int in_channels,
                                                                      int stride) {
    __shared__ float4 lds[kBlock * kManyStride<C> / 4];
    __shared__ float4 heads[kQuads * C / 4];
    __shared__ unsigned row_of_a[kTileSlots], row_of_b[D1B > 0 ? kTileSlots : 1];
    __shared__ unsigned char head_goes_on[kQuads];
    float *const values = reinterpret_cast<float *>(lds);
    float(*const head)[C] = reinterpret_cast<float(*)[C]>(heads);
    unsigned block, blocks, vblock;
    const TileSplat &work = item_of(items, block, blocks);
    if constexpr (N == 1) {
        if (!block_of_points(work.map, 1, vblock)) return;
    } else {
        if (block >= work.map.n_blocks) return;
        vblock = xcd_contiguous_block(block, work.map.n_blocks, 1);
    }
    const int tid = threadIdx.x, from = C * (int)blockIdx.y;
    static_assert(kTileSlots == kManyThreads, "a place a thread");
    const unsigned own_row_a = work.row_of_a[(size_t)vblock * kTileSlots + tid];
    unsigned own_row_b = 0;
    if constexpr (D1B > 0) own_row_b = work.row_of_b[(size_t)vblock * kTileSlots + tid];
    QuadEntries<D1A> entries_a;
    entries_a.load(work.entries_a + (size_t)vblock * kBlock * D1A);
    QuadEntries<(D1B > 0 ? D1B : 1)> entries_b;
    if constexpr (D1B > 0) entries_b.load(work.entries_b + (size_t)vblock * kBlock * D1B);
    // two lanes a point, every other piece of four channels each
    constexpr int kPieces = C / 4, kOwn = (kPieces + 1) / 2;
    const int n = point_of_thread(work.map, vblock, tid / 2);
    const float *row = work.input + (size_t)(n >= 0 ? n : 0) * in_channels;
    FourFloats x[kOwn];
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
        // (the piece, or where it does not lie in the row whole the row's last four)
        const int c = from + 4 * (2 * k + (tid & 1)), at = c < in_channels - 4 ? c : in_channels - 4;
        x[k] = *reinterpret_cast<const FourFloats *>(row + at);
    }
    row_of_a[tid] = own_row_a;
    if constexpr (D1B > 0) row_of_b[tid] = own_row_b;
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
        const int q = 2 * k + (tid & 1), c = from + 4 * q, at = c < in_channels - 4 ? c : in_channels - 4, shift = c - at;
        float y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = shift + j;
            const float in = one_of(i, x[k].c[0], x[k].c[1], x[k].c[2], x[k].c[3]);
            y[j] = c + j < in_channels ? (n >= 0 ? in : 0.0f) : c + j < vd ? 1.0f : 0.0f;
        }
        if (q < kPieces)
            *reinterpret_cast<float4 *>(values + tid / 2 * kManyStride<C> + 4 * q) = make_float4(y[0], y[1], y[2], y[3]);
    }
    __syncthreads();
    sum_many_runs<D1A, C>(entries_a, values, row_of_a, work.rows_a, from, stride, head,
                          head_goes_on);
    if constexpr (D1B > 0) {
        __syncthreads();
        sum_many_runs<D1B, C>(entries_b, values, row_of_b, work.rows_b, from, stride,
                              head, head_goes_on);
    }
}

// ------------------------------------------------------------------------------------------------
// Step 2: every vertex's row is the sum of its workgroups' rows, which lie one behind the other: L lanes a
// vertex, G rows side by side, four channels a lane (C <= 4: a lane takes whole rows).
// ------------------------------------------------------------------------------------------------
struct RowSums {
    const ListChunk *vertices;   // {first row, end, vertex, 1}
    unsigned n;
    const float *rows;
    float *values;
};
template <int VD, int N>
__global__ __launch_bounds__(kBlock) void k_add_rows(Items<RowSums, N> items, int, int) {
    constexpr int L = 4, kAhead = 2;
    unsigned block, blocks;
    const RowSums &work = item_of(items, block, blocks);
    const unsigned i = xcd_contiguous_block(block, blocks, 1) * (kBlock / L) + threadIdx.x / L, sub = threadIdx.x % L;
    const uint4 d = reinterpret_cast<const uint4 *>(work.vertices)[i < work.n ? i : 0];
    const unsigned to = i < work.n ? d.y : d.x;
    float acc[VD];
#pragma unroll
    for (int j = 0; j < VD; ++j) acc[j] = 0.0f;
    for (unsigned k = d.x + sub; k < to; k += kAhead * L) {
        float x[kAhead][VD];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const float *row = work.rows + (size_t)(k + u * L < to ? k + u * L : k) * VD;
#pragma unroll
            for (int j = 0; j < VD; ++j) x[u][j] = row[j];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
#pragma unroll
            for (int j = 0; j < VD; ++j) acc[j] += k + u * L < to ? x[u][j] : 0.0f;
        }
    }
#pragma unroll
    for (int off = 1; off < L; off <<= 1) {
#pragma unroll
        for (int j = 0; j < VD; ++j) acc[j] += __shfl_xor(acc[j], off);
    }
    if (i < work.n && sub == 0) {
#pragma unroll
        for (int j = 0; j < VD; ++j) work.values[(size_t)d.z * VD + j] = acc[j];
    }
}
template <int L, int N>
__global__ __launch_bounds__(kBlock) void k_add_rows_channels(Items<RowSums, N> items, int vd, int stride) {
    constexpr int kAhead = 8;
    unsigned block, blocks;
    const RowSums &work = item_of(items, block, blocks);
    const unsigned i = xcd_contiguous_block(block, blocks, 1) * (kBlock / L) + threadIdx.x / L;
    if (i >= work.n) return;
    const uint4 d = reinterpret_cast<const uint4 *>(work.vertices)[i];
    for (int c = 4 * (threadIdx.x % L); c < vd; c += 4 * L) {
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (unsigned k = d.x; k < d.y; k += kAhead) {
            float4 x[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
                x[u] = *reinterpret_cast<const float4 *>(work.rows + (size_t)(k + u < d.y ? k + u : k) * stride + c);
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const bool counts = k + u < d.y;
                acc[0] += counts ? x[u].x : 0.0f;
                acc[1] += counts ? x[u].y : 0.0f;
                acc[2] += counts ? x[u].z : 0.0f;
                acc[3] += counts ? x[u].w : 0.0f;
            }
        }
        float *to = work.values + (size_t)d.z * vd + c;
        if (c + 4 <= vd) {
            *reinterpret_cast<FourFloats *>(to) = FourFloats{{acc[0], acc[1], acc[2], acc[3]}};
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (c + j < vd) to[j] = acc[j];
        }
    }
}

template <int N>
hipError_t add_rows(int vd, int n, const RowSums *work, hipStream_t s) {
    const int lanes = vd <= 4 ? 4 : vd <= 16 ? 4 : vd <= 32 ? 8 : 16;
    Items<RowSums, N> items{};
    for (int i = 0; i < n; ++i) {
        if (!work[i].n) continue;
        items.item[items.n] = work[i];
        items.blocks[items.n++] = multiple_of_xcds(blocks_for(work[i].n, kBlock / lanes));
    }
    if (!items.n) return hipSuccess;
    const auto kernel = vd == 2   ? k_add_rows<2, N>
                        : vd == 3 ? k_add_rows<3, N>
                        : vd == 4 ? k_add_rows<4, N>
                        : lanes == 4 ? k_add_rows_channels<4, N>
                        : lanes == 8 ? k_add_rows_channels<8, N> : k_add_rows_channels<16, N>;
    hipLaunchKernelGGL(kernel, dim3(all_blocks(items)), dim3(kBlock), 0, s, items, vd, tile_row_floats(vd));
    return hipGetLastError();
}

TileSplat one_lattice(const VertexLists &lists, const float *input) {
    return TileSplat{lists.map, reinterpret_cast<const uint2 *>(lists.entries), nullptr, lists.places, nullptr, input,
                     lists.chunks.partial_rows, nullptr};
}
// (channels of a workgroup's rows)
int splat_channels(int vd) { return vd <= 8 ? 8 : vd <= 16 ? 16 : vd <= 24 ? 24 : 32; }

}  // namespace

hipError_t sort_tiles(int pd, const PointMap &map, const ReplayEntry *replay, int max_vertices, const VertexLists &lists,
                      hipStream_t s) {
    PLK_DISPATCH_PD(pd, hipLaunchKernelGGL((k_sort_tile<PD + 1>), dim3(map.n_blocks), dim3(kBlock), 0, s, map, replay,
                                           reinterpret_cast<uint2 *>(lists.entries), lists.count, lists.places, max_vertices));
    return hipGetLastError();
}
hipError_t place_rows(const PointMap &map, const VertexLists &lists, hipStream_t s) {
    hipLaunchKernelGGL(k_place_rows, dim3(map.n_blocks), dim3(kBlock), 0, s, map, lists.start, lists.places);
    return hipGetLastError();
}

hipError_t splat_tile_lists(int vd, const VertexLists &lists, unsigned n_vertices, const float *input, int in_channels,
                            float *values, hipStream_t s) {
    if (!lists.map.tile_vertices.table || in_channels < (vd <= 4 ? vd - 1 : 4) || in_channels > vd) return hipErrorInvalidValue;
    if (n_vertices == 0) return hipSuccess;
    const TileSplat work = one_lattice(lists, input);
    if (vd <= 4) {
#define PLK_SPLAT_ROWS_OF(VD, IN)                                                                                   \
    PLK_DISPATCH_PD(lists.pd, hipLaunchKernelGGL((k_splat_rows<VD, IN, PD + 1>), dim3(lists.map.n_blocks), dim3(kBlock), 0, \
                                                 s, lists.map, work.entries_a, work.row_of_a, input, work.rows_a))
#define PLK_SPLAT_ROWS(VD)                                                                                          \
    case VD:                                                                                                        \
        if (in_channels == VD)                                                                                      \
            PLK_SPLAT_ROWS_OF(VD, VD)                                                                               \
        else                                                                                                        \
            PLK_SPLAT_ROWS_OF(VD, VD - 1)                                                                           \
        break;
        switch (vd) { PLK_SPLAT_ROWS(2) PLK_SPLAT_ROWS(3) PLK_SPLAT_ROWS(4) }
#undef PLK_SPLAT_ROWS_OF
#undef PLK_SPLAT_ROWS
    } else {
        Items<TileSplat, 1> items{};
        items.item[0] = work;
        items.blocks[0] = lists.map.n_blocks;
        items.n = 1;
        const int C = splat_channels(vd);
        const dim3 grid(lists.map.n_blocks, (unsigned)((vd + C - 1) / C)), block(kManyThreads);
#define PLK_SPLAT_ROWS(C)                                                                                            \
    case C:                                                                                                          \
        PLK_DISPATCH_PD(lists.pd, hipLaunchKernelGGL((k_splat_rows_channels<PD + 1, 0, C, 1>), grid, block, 0, s, items, \
                                                     vd, in_channels, (int)tile_row_floats(vd)))                     \
        break;
        switch (C) { PLK_SPLAT_ROWS(8) PLK_SPLAT_ROWS(16) PLK_SPLAT_ROWS(24) PLK_SPLAT_ROWS(32) }
#undef PLK_SPLAT_ROWS
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const RowSums sums{lists.chunks.chunk, n_vertices, lists.chunks.partial_rows, values};
    return add_rows<1>(vd, 1, &sums, s);
}

bool splat_tile_pairs_take(int pd_a, int pd_b, int vd) {
    return vd >= kManyChannels && vd <= 32 &&
           ((pd_b == 2 && (pd_a == 3 || pd_a == 5)) || (pd_b == 3 && (pd_a == 4 || pd_a == 6)));
}
hipError_t splat_tile_pairs(int vd, int in_channels, int n, const GatherWork *work, hipStream_t s) {
    const int pairs = n / 2;
    if (n < 2 || n > kManyItems || n % 2 || in_channels < 4 || in_channels > vd) return hipErrorInvalidValue;
    const VertexLists &first_a = *work[0].lists, &first_b = *work[pairs].lists;
    if (!splat_tile_pairs_take(first_a.pd, first_b.pd, vd)) return hipErrorInvalidValue;
    Items<TileSplat> items{};
    RowSums sums[kManyItems];
    for (int i = 0; i < pairs; ++i) {
        const VertexLists &a = *work[i].lists, &b = *work[pairs + i].lists;
        items.item[i] = one_lattice(a, work[i].input);
        items.item[i].entries_b = reinterpret_cast<const uint2 *>(b.entries);
        items.item[i].row_of_b = b.places;
        items.item[i].rows_b = b.chunks.partial_rows;
        items.blocks[i] = multiple_of_xcds(a.map.n_blocks);
    }
    items.n = pairs;
    for (int i = 0; i < n; ++i)
        sums[i] = RowSums{work[i].chunks.chunk, work[i].n_chunks, work[i].chunks.partial_rows, work[i].values};
    const int C = splat_channels(vd);
    const dim3 grid(all_blocks(items)), block(kManyThreads);
#define PLK_SPLAT_PAIR(A, B, C_)                                                                              \
    if (first_a.pd == A && first_b.pd == B && C == C_)                                                        \
        hipLaunchKernelGGL((k_splat_rows_channels<A + 1, B + 1, C_, kManyItems>), grid, block, 0, s, items, vd,     \
                           in_channels, (int)tile_row_floats(vd));
#define PLK_SPLAT_PAIRS(A, B) PLK_SPLAT_PAIR(A, B, 8) PLK_SPLAT_PAIR(A, B, 16) PLK_SPLAT_PAIR(A, B, 24) PLK_SPLAT_PAIR(A, B, 32)
    PLK_SPLAT_PAIRS(3, 2) PLK_SPLAT_PAIRS(5, 2) PLK_SPLAT_PAIRS(4, 3) PLK_SPLAT_PAIRS(6, 3)
#undef PLK_SPLAT_PAIRS
#undef PLK_SPLAT_PAIR
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : add_rows<kManyItems>(vd, n, sums, s);
}

}  // namespace plk
