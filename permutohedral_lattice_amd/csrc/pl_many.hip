// The applies of several lattices, pass by pass in one launch each, and the message passing of a dense
// CRF on them: both messages of a point are sliced by the same lanes, added up, and the mean field's
// softmax taken where they are.  No counterpart in the reference (one lattice at a time,
// src/LatticeFilterKernel.cpp:152-179, and no CRF).
//
// At 512x512 points of 21 classes every pass of one lattice is a kernel of 5 to 25 us that fills a third
// of the GPU, and an iteration on two images and their four lattices was 22 launches on four streams (and 13
// events): the host needed as long for them as the GPU.  Here it is six or seven launches on one stream.
// Two images, five iterations: 1154 us as launches of their own, 720 this way.
#include <type_traits>

#include "pl_device.h"
#include "pl_kernels.h"

namespace plk {

namespace {

using namespace device;


// ------------------------------------------------------------------------------------------------
// Blur of rows of five and more channels: a thread per vertex and run of four of its channels (the
// last run is the row's last four, so that no load leaves the row; what two runs share is written
// twice, the same), one axis or two as k_blur_element and k_blur2_element of pl_kernels.hip apply them: same
// arithmetic, same results, a quarter of the load instructions.  Bound by three round trips to memory, in
// one launch for all lattices (two images, 97 000 vertices of 22 channels: 8.8 us a pass of two axes; a
// launch a lattice, a thread per channel, 5.4 us each).  A lattice alone takes it too (an op and its
// gradient on 2 x 321x481 points of 21 channels, twelve passes of two axes: 306.7 and 292.8 us).
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ FourFloats blur_taps(const FourFloats &a, const FourFloats &self, const FourFloats &b) {
    FourFloats out;
#pragma unroll
    for (int j = 0; j < 4; ++j) out.c[j] = blur_tap(a.c[j], self.c[j], b.c[j]);
    return out;
}
template <int N>
__device__ __forceinline__ void gather_runs(const float *__restrict__ src, int vd, int from, const int (&u)[N],
                                            FourFloats (&x)[N]) {
    // (every load is issued, from a row that exists, and replaced by zeros afterwards)
#pragma unroll
    for (int k = 0; k < N; ++k)
        x[k] = *reinterpret_cast<const FourFloats *>(src + (size_t)(u[k] >= 0 ? u[k] : 0) * vd + from);
#pragma unroll
    for (int k = 0; k < N; ++k) {
#pragma unroll
        for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(x[k].c[j]));
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[k].c[j] = u[k] >= 0 ? x[k].c[j] : 0.0f;
    }
}
template <int N>   // lattices a launch may be given
__global__ __launch_bounds__(kBlock) void k_blur_runs(Items<BlurWork, N> items, int vd) {
    unsigned block, blocks;
    const BlurWork &work = item_of(items, block, blocks);
    const unsigned runs = (unsigned)(vd + 3) / 4u;
    SegmentWalk walk(work.counters, work.max_vertices, block, blocks);
    unsigned rb;
    while (walk.next(runs, 1u, rb)) {
        const unsigned i = rb * kBlock + threadIdx.x;
        if (i >= walk.count * runs) continue;
        const unsigned in_run = i / runs, run = i - in_run * runs;
        const int v = (int)(walk.first + in_run);
        const int from = 4 * (int)run < vd - 4 ? 4 * (int)run : vd - 4;
        FourFloats out;
        if (work.nbr_second) {
            int u[9];
            two_axis_sources(work.nbr_first, work.nbr_second, v, u);
            FourFloats x[9];
            gather_runs<9>(work.src, vd, from, u, x);
            out = blur_taps(blur_taps(x[0], x[1], x[2]), blur_taps(x[3], x[4], x[5]), blur_taps(x[6], x[7], x[8]));
        } else {
            const int2 nb = work.nbr_first[v];
            const int u[3] = {nb.x, v, nb.y};
            FourFloats x[3];
            gather_runs<3>(work.src, vd, from, u, x);
            out = blur_taps(x[0], x[1], x[2]);
        }
        *reinterpret_cast<FourFloats *>(work.dst + (size_t)v * vd + from) = out;
        if (work.reset_cell_keys && run == 0) work.reset_cell_keys[work.vertex_cell[v]] = kEmptyCell;
    }
}

// ------------------------------------------------------------------------------------------------
// The slice of two lattices over the same points, added up: L lanes per point (4 or 8), lane i on the
// channels 4i .. 4i+3, two points per group of lanes, loads and sums as in k_slice_quads of pl_kernels.hip.
// The sum of both messages is the output, or, with logits, the softmax of logits + sum (terms and order as
// in k_mean_field_update): the messages, 22 MB each for 512x512 points of 21 classes, are neither
// written nor read again.  Bound by the nine rows of 88 bytes it gathers a point (2 x 512x512 points: 40 us,
// 56 with the softmax; as two slices an image and the softmax as a pass 65 and 98).  One point per group
// instead of two: the same.
// ------------------------------------------------------------------------------------------------
constexpr int kPairPoints = 2;

template <int D1, int L>
__device__ __forceinline__ void sliced_channels(int vd, const ReplayEntry *__restrict__ replay,
                                                const TileVertices &tiles,
                                                const float *__restrict__ values, unsigned vblock,
                                                const unsigned (&slot)[kPairPoints], const int (&n)[kPairPoints],
                                                int sub, float (&message)[kPairPoints][4]) {
    constexpr int E = (D1 + L - 1) / L;     // replay rows a lane reads per point
    ReplayEntry mine[kPairPoints][E];
#pragma unroll
    for (int q = 0; q < kPairPoints; ++q) {
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const int r = u * L + sub;
            mine[q][u] = replay_corner(replay, tiles, vblock, D1, r < D1 ? r : 0, slot[q]);
        }
    }
    const int c = 4 * sub;
    const int start = c < vd - 4 ? c : vd - 4;
    FourFloats x[kPairPoints][D1];
    float w[kPairPoints][D1];
#pragma unroll
    for (int q = 0; q < kPairPoints; ++q) {
#pragma unroll
        for (int r = 0; r < D1; ++r) {
            const int index = __shfl(mine[q][r / L].index, r % L, L);
            w[q][r] = __shfl(mine[q][r / L].weight, r % L, L);
            const bool present = index >= 0 && n[q] >= 0;
            x[q][r] = *reinterpret_cast<const FourFloats *>(values + (size_t)(present ? index : 0) * vd + start);
            if (!present) w[q][r] = 0.0f, x[q][r] = FourFloats{{0.0f, 0.0f, 0.0f, 0.0f}};
        }
    }
    // the homogeneous channel vd-1 is with the lane (vd-1)/4; a lane past the row's start has its last four
    const int with = (vd - 1) / 4;
    const int with_start = 4 * with < vd - 4 ? 4 * with : vd - 4;
    const int at = vd - 1 - with_start, shift = c - start;
#pragma unroll
    for (int q = 0; q < kPairPoints; ++q) {
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int r = 0; r < D1; ++r) {
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] += w[q][r] * x[q][r].c[j];
        }
        const float own = at == 0 ? acc[0] : at == 1 ? acc[1] : at == 2 ? acc[2] : acc[3];
        const float scale = (float)(1.0 / (double)__shfl(own, with, L));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = shift + j;
            const float v = i == 0 ? acc[0] : i == 1 ? acc[1] : i == 2 ? acc[2] : acc[3];
            message[q][j] = v * scale;
        }
    }
}

template <int D1A, int D1B, int L>
__global__ __launch_bounds__(kBlock) void k_slice_pairs(Items<SlicePair> items, int vd) {
    constexpr int kGroups = kBlock / L;
    unsigned block, blocks;
    const SlicePair &work = item_of(items, block, blocks);
    if (block >= work.map.n_blocks) return;
    const unsigned vblock = xcd_contiguous_block(block, work.map.n_blocks, 1);
    const int sub = threadIdx.x % L;
    unsigned slot[kPairPoints];
    int n[kPairPoints];
#pragma unroll
    for (int q = 0; q < kPairPoints; ++q) {
        slot[q] = (blockIdx.y * kPairPoints + q) * kGroups + threadIdx.x / L;
        n[q] = point_of_thread(work.map, vblock, slot[q]);   // (the same for all L lanes)
    }
    float a[kPairPoints][4], b[kPairPoints][4];
    sliced_channels<D1A, L>(vd, work.replay_a, work.map.tile_vertices, work.values_a, vblock, slot, n, sub, a);
    sliced_channels<D1B, L>(vd, work.replay_b, work.tiles_b, work.values_b, vblock, slot, n, sub, b);
    const int classes = vd - 1, c = 4 * sub;
#pragma unroll
    for (int q = 0; q < kPairPoints; ++q) {
        float y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = a[q][j] + b[q][j];
        const size_t row = (size_t)(n[q] >= 0 ? n[q] : 0) * classes;
        if (work.logits) {
            const int start = c < classes - 4 ? c : classes - 4, shift = c - start;
            const FourFloats l = *reinterpret_cast<const FourFloats *>(work.logits + row + start);
            float highest = -INFINITY;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = shift + j;
                const float logit = i == 0 ? l.c[0] : i == 1 ? l.c[1] : i == 2 ? l.c[2] : l.c[3];
                y[j] = logit + y[j];
                if (c + j < classes) highest = fmaxf(highest, y[j]);
            }
#pragma unroll
            for (int off = 1; off < L; off <<= 1) highest = fmaxf(highest, __shfl_xor(highest, off));
            double wide_sum = 0.0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                y[j] = expf(y[j] - highest);
                if (c + j < classes) wide_sum += (double)y[j];
            }
#pragma unroll
            for (int off = 1; off < L; off <<= 1) wide_sum += __shfl_xor(wide_sum, off);
            const float sum = (float)wide_sum;
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = y[j] / sum;
        }
        if (n[q] < 0) continue;
        float *out = work.output + row + c;
        if (c + 4 <= classes) {
            *reinterpret_cast<FourFloats *>(out) = FourFloats{{y[0], y[1], y[2], y[3]}};
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (c + j < classes) out[j] = y[j];
        }
    }
}

// ------------------------------------------------------------------------------------------------
// The slices of many channels after a merging build.  A workgroup's points touch a hundred or two of
// vertices between them, where its corners are 256 * D1: the vertices' rows go to LDS, each read once, and
// two lanes a point sum the rows from there, every other piece of four channels each.  What they make of a
// point goes out by way of LDS as well, so that a wavefront's stores are runs of memory.  Workgroups of more
// vertices than there are rows in LDS gather from memory, corner by corner.  Sums in the order of k_slice_quads
// and sliced_channels, each product and sum rounded once instead of twice.
// Bound by what a workgroup waits for (table, rows, LDS, its stores), 32 wavefronts a CU for a lattice alone, 24
// for two; vector instructions half of the time.  321x481 points, pd 5, vd 22: 9.2 us a launch (k_slice_quads on
// replay rows 12.6, on places 14.0; a lane a point with its stores 84 bytes apart 14.8; eight lanes a point
// 13.2).  Pairs of 2 x 512x512 points with the softmax, 21 classes: 43.7 us (k_slice_pairs on rows 56.5; a lane
// a point 55.1; eight lanes 62.0; with five wavefronts a SIMD, not six, 49.3).
// (A row in LDS is an odd number of 16-byte pieces: the same piece of sixteen rows lies in different banks.)
// ------------------------------------------------------------------------------------------------
constexpr int kTileLanes = 2, kTileThreads = kTileLanes * kBlock;
constexpr int kTileChannels = 32;   // channels a workgroup takes at most
// Channels from `from` on of the rows of one lattice of a workgroup's points
struct Tile {
    const int *table;
    const float *values;
    int used, vd, from;
    float *rows, *last;   // in LDS: Q pieces of four channels, row_stride(Q) floats apart; the homogeneous channels
};
__host__ __device__ constexpr int row_stride(int Q) { return 4 * (Q | 1); }
// Rows in LDS.  A CU holds four workgroups of these kernels, three of pairs (`per_cu`), whatever LDS each takes up to
// its share of the CU's, and a launch of fewer workgroups leaves more to each: at 21 channels 335 rows (453 of
// pairs) and up to all 512, where 28 KB a workgroup were 247.  us an apply, 28 KB and this, crowded tiles (pd 5,
// 8 corners a vertex): vd 22 64x64 22.1 and 20.8, 321x481 71.4 and 67.6; vd 32 64x64 23.2 and 20.2, 1024x1024 473 and 440;
// pairs of 2 x 512x512 points, 21 classes, a slice 47.2 and 42.6.  (64 KB at most: what a launch may ask for anywhere.)
inline unsigned tile_rows(int Q, unsigned workgroups, unsigned per_cu) {
    const unsigned a_cu = (workgroups + 255u) / 256u, at_once = a_cu < per_cu ? a_cu : per_cu;
    const unsigned share = (160u << 10) / (at_once ? at_once : 1u), lds = (share < 64u << 10 ? share : 64u << 10) - 2048u;
    const unsigned rows = lds / (sizeof(float) * (unsigned)(row_stride(Q) + 1));
    return rows < (unsigned)kTileSlots ? rows : (unsigned)kTileSlots;
}
// (what the rows leave takes the 256 points' channels later)
inline size_t tile_lds(int Q, unsigned rows) {
    const size_t in = (size_t)rows * (row_stride(Q) + 1), out = (size_t)kBlock * 4 * Q;
    return sizeof(float) * (in > out ? in : out);
}
// The four channels from c on of a row in memory (what is past vd: anything)
__device__ __forceinline__ FourFloats piece_of_row(const float *row, int vd, int c) {
    const int start = c < vd - 4 ? c : vd - 4, shift = c - start;
    const FourFloats x = *reinterpret_cast<const FourFloats *>(row + start);
    if (shift == 0) return x;
    return FourFloats{{one_of(shift, x.c[0], x.c[1], x.c[2], x.c[3]), one_of(shift + 1, x.c[0], x.c[1], x.c[2], x.c[3]),
                       x.c[3], x.c[3]}};
}
// (as many lanes a row as it has pieces, or some more; two rows a group of lanes in flight)
template <int Q>
__device__ __forceinline__ void rows_to_lds(const Tile &tile) {
    constexpr int L = Q <= 2 ? 2 : Q <= 4 ? 4 : 8, kGroups = kTileThreads / L, kAhead = 2;
    const int sub = threadIdx.x % L;
    for (int i0 = threadIdx.x / L; i0 < tile.used; i0 += kAhead * kGroups) {
        int v[kAhead];
        FourFloats x[kAhead];
        float last[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = tile.table[i0 + u * kGroups < tile.used ? i0 + u * kGroups : i0];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const float *row = tile.values + (size_t)(v[u] >= 0 ? v[u] : 0) * tile.vd;
            x[u] = piece_of_row(row, tile.vd, tile.from + 4 * sub);
            last[u] = row[tile.vd - 1];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int i = i0 + u * kGroups;
            if (i >= tile.used) continue;
            if (sub < Q)
                *reinterpret_cast<float4 *>(tile.rows + i * row_stride(Q) + 4 * sub) =
                    make_float4(x[u].c[0], x[u].c[1], x[u].c[2], x[u].c[3]);
            if (sub == 0) tile.last[i] = last[u];
        }
    }
}
// A point's corners: places (of points that are none, or that the build could not place: 0) and weights
template <int D1>
struct Corners {
    int place[D1];
    float weight[D1];
};
template <int D1>
__device__ __forceinline__ Corners<D1> corners_of(const ReplayEntry *__restrict__ replay, unsigned vblock, int point,
                                                  int used) {
    const uint32_t *words = words_of_tile(replay, vblock, D1);
    uint32_t word[replay_words(D1)];
#pragma unroll
    for (int w = 0; w < replay_words(D1); ++w) word[w] = words[w * kBlock + point];
    Corners<D1> corners;
#pragma unroll
    for (int r = 0; r < D1; ++r) {
        corners.weight[r] = weights_behind(words, D1)[r * kBlock + point];
        const int place = (int)place_of_corner(word[r / kPlacesPerWord], r);
        corners.place[r] = place < used ? place : 0;
    }
    return corners;
}
// (a piece of all corners in flight, not all pieces: the next one's addresses come after this one's sums)
template <int D1>
__device__ __forceinline__ void next_piece(Corners<D1> &corners, float (&sums)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(sums[j]));
#pragma unroll
    for (int r = 0; r < D1; ++r) asm volatile("" : "+v"(corners.place[r]), "+v"(sums[0]));
}
// acc := piece q of the point's channels
template <int D1, int Q, bool IN_LDS>
__device__ __forceinline__ void sum_corners(const Tile &tile, int q, const Corners<D1> &corners, float (&acc)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = 0.0f;
#pragma unroll
    for (int r = 0; r < D1; ++r) {
        FourFloats y;
        if constexpr (IN_LDS) {
            const float4 x = *reinterpret_cast<const float4 *>(tile.rows + corners.place[r] * row_stride(Q) + 4 * q);
            y = FourFloats{{x.x, x.y, x.z, x.w}};
        } else {
            const int v = tile.table[corners.place[r]];
            y = piece_of_row(tile.values + (size_t)(v >= 0 ? v : 0) * tile.vd, tile.vd, tile.from + 4 * q);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = __builtin_fmaf(corners.weight[r], y.c[j], acc[j]);
    }
}
// The sum of the homogeneous channel
template <int D1, bool IN_LDS>
__device__ __forceinline__ float sum_of_last(const Tile &tile, const Corners<D1> &corners) {
    float sum = 0.0f;
#pragma unroll
    for (int r = 0; r < D1; ++r) {
        if constexpr (IN_LDS) {
            sum = __builtin_fmaf(corners.weight[r], tile.last[corners.place[r]], sum);
        } else {
            const int v = tile.table[corners.place[r]];
            sum = __builtin_fmaf(corners.weight[r], tile.values[(size_t)(v >= 0 ? v : 0) * tile.vd + tile.vd - 1], sum);
        }
    }
    return sum;
}

// x of lane I of this lane's two (quad_perm [0,0,2,2] or [1,1,3,3])
template <int I>
__device__ __forceinline__ float lane_of_two(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), I == 0 ? 0xA0 : 0xF5, 0xf, 0xf, true));
}

// The workgroup's 256 points' rows of `channels` channels (at least four) in memory, `stride` floats apart and
// offset by `from`, piece by piece: floats 4 i .. 4 i + 3 of the rows one behind the other, which lie one
// behind the other in memory as well where neighbours in the workgroup are neighbours there.  per_channel:
// 2^20 / channels, rounded up (i / channels for i < 2^14 as a product, channels < 64).
struct PointRows {
    int channels, stride, from;
    unsigned per_channel;
};
struct Piece {
    int p, c;      // its first float: point and channel
    bool whole;    // four floats of memory
};
__device__ __forceinline__ Piece piece_at(int i, const PointRows &rows, const int *n_of) {
    Piece piece;
    piece.p = (int)(((unsigned)(4 * i) * rows.per_channel) >> 20);
    piece.c = 4 * i - piece.p * rows.channels;
    const int left = rows.channels - piece.c;   // of this point's
    piece.whole = n_of[piece.p] >= 0 &&
                  (left >= 4 || (rows.channels == rows.stride && n_of[piece.p + 1] == n_of[piece.p] + 1));
    return piece;
}
__device__ __forceinline__ void store_points(const float *from_lds, float *output, const PointRows &rows, const int *n_of) {
    for (int i = threadIdx.x; i < kBlock / 4 * rows.channels; i += kTileThreads) {
        const Piece piece = piece_at(i, rows, n_of);
        const float4 x = reinterpret_cast<const float4 *>(from_lds)[i];
        const float y[4] = {x.x, x.y, x.z, x.w};
        if (piece.whole) {
            *reinterpret_cast<FourFloats *>(output + (size_t)n_of[piece.p] * rows.stride + rows.from + piece.c) =
                FourFloats{{y[0], y[1], y[2], y[3]}};
        } else {
            int p = piece.p, c = piece.c;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int n = n_of[p];
                if (n >= 0) output[(size_t)n * rows.stride + rows.from + c] = y[j];
                if (++c == rows.channels) c = 0, ++p;
            }
        }
    }
}
// (the pieces this thread brings to LDS: read before the LDS is free for them, left there afterwards)
template <int Q>
__device__ __forceinline__ void load_points(const float *input, const PointRows &rows, const int *n_of,
                                            FourFloats (&x)[(4 * Q * kBlock / 4 + kTileThreads - 1) / kTileThreads]) {
#pragma unroll
    for (int k = 0; k < (4 * Q * kBlock / 4 + kTileThreads - 1) / kTileThreads; ++k) {
        const int i = (int)threadIdx.x + k * kTileThreads;
        if (i >= kBlock / 4 * rows.channels) continue;
        const Piece piece = piece_at(i, rows, n_of);
        if (piece.whole) {
            x[k] = *reinterpret_cast<const FourFloats *>(input + (size_t)n_of[piece.p] * rows.stride + rows.from + piece.c);
        } else {
            int p = piece.p, c = piece.c;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int n = n_of[p];
                x[k].c[j] = n >= 0 ? input[(size_t)n * rows.stride + rows.from + c] : 0.0f;
                if (++c == rows.channels) c = 0, ++p;
            }
        }
    }
}
template <int Q>
__device__ __forceinline__ void points_to_lds(float *lds, const PointRows &rows,
                                              const FourFloats (&x)[(4 * Q * kBlock / 4 + kTileThreads - 1) / kTileThreads]) {
#pragma unroll
    for (int k = 0; k < (4 * Q * kBlock / 4 + kTileThreads - 1) / kTileThreads; ++k) {
        const int i = (int)threadIdx.x + k * kTileThreads;
        if (i < kBlock / 4 * rows.channels)
            reinterpret_cast<float4 *>(lds)[i] = make_float4(x[k].c[0], x[k].c[1], x[k].c[2], x[k].c[3]);
    }
}

// workgroup (x, y): channels 32 y .. of the points of block x.  Q: pieces of four channels of a workgroup's.
template <int D1, int Q>
__device__ __forceinline__ void slice_channels_of_tile(float *lds, int vd, const PointMap &map,
                                                       const ReplayEntry *__restrict__ replay,
                                                       const float *__restrict__ values, float *__restrict__ output,
                                                       int normalize, int n_rows, PointRows rows, unsigned block,
                                                       unsigned blocks) {
    __shared__ int n_of[kBlock + 1];
    unsigned vblock;
    if (!block_of_points(map, 1, block, blocks, vblock)) return;
    const int tid = threadIdx.x, sub = tid % kTileLanes, point = tid / kTileLanes;
    rows.from = rows.channels * (int)blockIdx.y;
    if (rows.stride - rows.from < rows.channels) {   // (the last of several workgroups of a tile)
        rows.channels = rows.stride - rows.from;
        rows.per_channel = ((1u << 20) + (unsigned)rows.channels - 1u) / (unsigned)rows.channels;
    }
    const Tile tile{map.tile_vertices.of(vblock), values, map.tile_vertices.used[vblock],
                    vd, rows.from, lds, lds + n_rows * row_stride(Q)};
    Corners<D1> corners = corners_of<D1>(replay, vblock, point, tile.used);
    const bool in_lds = tile.used <= n_rows;
    if (in_lds) rows_to_lds<Q>(tile);
    if (tid <= kBlock) n_of[tid] = tid < kBlock ? point_of_thread(map, vblock, tid) : -1;
    __syncthreads();
    constexpr int kOwn = (Q + kTileLanes - 1) / kTileLanes;   // pieces of a lane
    float y[kOwn][4];
    auto slice_point = [&](auto rows_in_lds) {
        constexpr bool kInLds = decltype(rows_in_lds)::value;
        const float scale = normalize ? (float)(1.0 / (double)sum_of_last<D1, kInLds>(tile, corners)) : 1.0f;
#pragma unroll
        for (int k = 0; k < kOwn; ++k) {
            const int q = kTileLanes * k + sub;
            sum_corners<D1, Q, kInLds>(tile, q < Q ? q : 0, corners, y[k]);
#pragma unroll
            for (int j = 0; j < 4; ++j) y[k][j] = normalize ? y[k][j] * scale : y[k][j];
            next_piece(corners, y[k]);
        }
    };
    if (in_lds)
        slice_point(std::true_type{});
    else
        slice_point(std::false_type{});
    __syncthreads();        // the rows are done with
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
        const int c = 4 * (kTileLanes * k + sub);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (c + j < rows.channels) lds[point * rows.channels + c + j] = y[k][j];
    }
    __syncthreads();
    store_points(lds, output, rows, n_of);
}
template <int D1, int Q>
__global__ __launch_bounds__(kTileThreads) void k_slice_tile_channels(int vd, PointMap map,
                                                                      const ReplayEntry *__restrict__ replay,
                                                                      const float *__restrict__ values,
                                                                      float *__restrict__ output, int normalize,
                                                                      int n_rows, PointRows rows) {
    extern __shared__ float4 lds[];
    slice_channels_of_tile<D1, Q>(reinterpret_cast<float *>(lds), vd, map, replay, values, output, normalize, n_rows, rows,
                                  blockIdx.x, gridDim.x);
}
// The same for several lattices.
template <int D1, int Q>
__global__ __launch_bounds__(kTileThreads) void k_slice_tile_channels_of(Items<PointsWork, kJointItems> items, int vd,
                                                                         int normalize, int n_rows, PointRows rows) {
    extern __shared__ float4 lds[];
    unsigned block, blocks;
    const PointsWork &work = item_of(items, block, blocks);
    if (block >= work.map.n_blocks) return;
    slice_channels_of_tile<D1, Q>(reinterpret_cast<float *>(lds), vd, work.map, work.replay, work.values, work.output,
                                  normalize, n_rows, rows, block, work.map.n_blocks);
}

// Q: pieces of four classes
template <int D1A, int D1B, int Q>
__global__ __launch_bounds__(kTileThreads, D1A <= 6 ? 6 : 4) void k_slice_tile_pairs(Items<SlicePair> items, int vd, int n_rows,
                                                                   PointRows rows) {
    extern __shared__ float4 lds4[];
    __shared__ int n_of[kBlock + 1];
    float *lds = reinterpret_cast<float *>(lds4);
    unsigned block, blocks;
    const SlicePair &work = item_of(items, block, blocks);
    if (block >= work.map.n_blocks) return;
    const unsigned vblock = xcd_contiguous_block(block, work.map.n_blocks, 1);
    const int tid = threadIdx.x, sub = tid % kTileLanes, point = tid / kTileLanes;
    if (tid <= kBlock) n_of[tid] = tid < kBlock ? point_of_thread(work.map, vblock, tid) : -1;
    const int used_a = work.map.tile_vertices.used[vblock], used_b = work.tiles_b.used[vblock];
    const Tile a{work.map.tile_vertices.of(vblock), work.values_a, used_a, vd, 0, lds,
                 lds + n_rows * row_stride(Q)};
    const Tile b{work.tiles_b.of(vblock), work.values_b, used_b, vd, 0,
                 a.rows + used_a * row_stride(Q), a.last + used_a};
    Corners<D1A> corners_a = corners_of<D1A>(work.replay_a, vblock, point, used_a);
    Corners<D1B> corners_b = corners_of<D1B>(work.replay_b, vblock, point, used_b);
    const bool in_lds = used_a + used_b <= n_rows;
    if (in_lds) {
        rows_to_lds<Q>(a);
        rows_to_lds<Q>(b);
    }
    __syncthreads();
    FourFloats logits[(4 * Q * kBlock / 4 + kTileThreads - 1) / kTileThreads];
    if (work.logits) load_points<Q>(work.logits, rows, n_of, logits);
    constexpr int kOwn = (Q + kTileLanes - 1) / kTileLanes;   // pieces of a lane
    float y[kOwn][4];
    auto slice_point = [&](auto rows_in_lds) {
        constexpr bool kInLds = decltype(rows_in_lds)::value;
        // (a division a lane, one lattice's each)
        const float last_a = sum_of_last<D1A, kInLds>(a, corners_a), last_b = sum_of_last<D1B, kInLds>(b, corners_b);
        const float one_over = (float)(1.0 / (double)(sub == 0 ? last_a : last_b));
        const float scale_a = lane_of_two<0>(one_over), scale_b = lane_of_two<1>(one_over);
#pragma unroll
        for (int k = 0; k < kOwn; ++k) {
            const int q = kTileLanes * k + sub < Q ? kTileLanes * k + sub : 0;
            float z[4];
            sum_corners<D1A, Q, kInLds>(a, q, corners_a, y[k]);
            sum_corners<D1B, Q, kInLds>(b, q, corners_b, z);
#pragma unroll
            for (int j = 0; j < 4; ++j) y[k][j] = y[k][j] * scale_a + z[j] * scale_b;
            next_piece(corners_a, y[k]);
            next_piece(corners_b, y[k]);
        }
    };
    if (in_lds)
        slice_point(std::true_type{});
    else
        slice_point(std::false_type{});
    __syncthreads();        // the rows are done with
    float *const own = lds + point * rows.channels;
    if (work.logits) {
        points_to_lds<Q>(lds, rows, logits);
        __syncthreads();
        float highest = -INFINITY;
#pragma unroll
        for (int k = 0; k < kOwn; ++k) {
            const int c = 4 * (kTileLanes * k + sub);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (c + j < rows.channels) {
                    y[k][j] = own[c + j] + y[k][j];
                    highest = fmaxf(highest, y[k][j]);
                }
            }
        }
        highest = fmaxf(lane_of_two<0>(highest), lane_of_two<1>(highest));
        double wide_sum = 0.0;
#pragma unroll
        for (int k = 0; k < kOwn; ++k) {
            const int c = 4 * (kTileLanes * k + sub);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                y[k][j] = expf(y[k][j] - highest);
                if (c + j < rows.channels) wide_sum += (double)y[k][j];
            }
        }
        wide_sum += __shfl_xor(wide_sum, 1);
        // (a product of doubles rounded once: within 2^-29 of an ulp of the quotient's rounding)
        const double one_over = 1.0 / (double)(float)wide_sum;
#pragma unroll
        for (int k = 0; k < kOwn; ++k) {
#pragma unroll
            for (int j = 0; j < 4; ++j) y[k][j] = (float)((double)y[k][j] * one_over);
        }
    }
    // (a point's channels are its own two lanes' in LDS)
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
        const int c = 4 * (kTileLanes * k + sub);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (c + j < rows.channels) own[c + j] = y[k][j];
    }
    __syncthreads();
    store_points(lds, work.output, rows, n_of);
}

}  // namespace

static PointRows point_rows(int channels, int stride) {
    return PointRows{channels, stride, 0, ((1u << 20) + (unsigned)channels - 1u) / (unsigned)channels};
}

hipError_t slice_tile_channels(int pd, int vd, const PointMap &map, const ReplayEntry *replay, const float *values,
                               float *output, int normalize, hipStream_t s) {
    if (map.n_blocks == 0) return hipSuccess;
    if (!map.tile_vertices.table || vd < kManyChannels) return hipErrorInvalidValue;
    const int out_ch = normalize ? vd - 1 : vd, groups = (out_ch + kTileChannels - 1) / kTileChannels;
    const int channels = groups == 1 ? out_ch : ((out_ch + groups - 1) / groups + 3) / 4 * 4;
    const int Q = (channels + 3) / 4;
    const dim3 grid(map.n_blocks, (unsigned)groups), block(kTileThreads);
    const unsigned n_rows = tile_rows(Q, grid.x * grid.y, 4);
#define PLK_SLICE_TILE(Q)                                                                                     \
    case Q:                                                                                                   \
        PLK_DISPATCH_PD(pd, hipLaunchKernelGGL((k_slice_tile_channels<PD + 1, Q>), grid, block,               \
                                               tile_lds(Q, n_rows), s, vd, map, replay, values, output,       \
                                               normalize, (int)n_rows, point_rows(channels, out_ch)));        \
        break;
    switch (Q) {
        PLK_SLICE_TILE(1) PLK_SLICE_TILE(2) PLK_SLICE_TILE(3) PLK_SLICE_TILE(4) PLK_SLICE_TILE(5)
        PLK_SLICE_TILE(6) PLK_SLICE_TILE(7) PLK_SLICE_TILE(8)
        default: return hipErrorInvalidValue;
    }
#undef PLK_SLICE_TILE
    return hipGetLastError();
}

hipError_t slice_tile_channels_joint(int pd, int vd, int n, const PointsWork *work, int normalize, hipStream_t s) {
    const int out_ch = normalize ? vd - 1 : vd;
    if (n < 1 || n > kJointItems || vd < kManyChannels || out_ch > kTileChannels) return hipErrorInvalidValue;
    const Items<PointsWork, kJointItems> items = items_of_points<kJointItems>(n, work);
    const int Q = (out_ch + 3) / 4;
    const dim3 grid(all_blocks(items)), block(kTileThreads);
    const unsigned n_rows = tile_rows(Q, grid.x, 4);
#define PLK_SLICE_TILE_OF(PD, Q)                                                                                     \
    case Q:                                                                                                          \
        hipLaunchKernelGGL((k_slice_tile_channels_of<PD + 1, Q>), grid, block, tile_lds(Q, n_rows), s, items, vd,    \
                           normalize, (int)n_rows, point_rows(out_ch, out_ch));                                      \
        break;
#define PLK_SLICE_TILES(PD)                                                                                          \
    case PD:                                                                                                         \
        switch (Q) {                                                                                                 \
            PLK_SLICE_TILE_OF(PD, 1) PLK_SLICE_TILE_OF(PD, 2) PLK_SLICE_TILE_OF(PD, 3) PLK_SLICE_TILE_OF(PD, 4)      \
            PLK_SLICE_TILE_OF(PD, 5) PLK_SLICE_TILE_OF(PD, 6) PLK_SLICE_TILE_OF(PD, 7) PLK_SLICE_TILE_OF(PD, 8)      \
        }                                                                                                            \
        break;
    switch (pd) {
        PLK_SLICE_TILES(2) PLK_SLICE_TILES(3) PLK_SLICE_TILES(4) PLK_SLICE_TILES(5)
        default: return hipErrorInvalidValue;
    }
#undef PLK_SLICE_TILES
#undef PLK_SLICE_TILE_OF
    return hipGetLastError();
}

template <int N>
static hipError_t blur_runs(int vd, int n, const BlurWork *work, hipStream_t s) {
    Items<BlurWork, N> items{};
    items.n = n;
    const unsigned runs = (unsigned)(vd + 3) / 4u;
    for (int i = 0; i < n; ++i) {
        items.item[i] = work[i];
        items.blocks[i] = vertex_blocks((size_t)work[i].launch_vertices * runs);
    }
    hipLaunchKernelGGL((k_blur_runs<N>), dim3(all_blocks(items)), dim3(kBlock), 0, s, items, vd);
    return hipGetLastError();
}
hipError_t blur_many(int vd, int n, const BlurWork *work, hipStream_t s) {
    if (n < 1 || n > kManyItems || vd < kManyChannels) return hipErrorInvalidValue;
    return n == 1 ? blur_runs<1>(vd, n, work, s) : blur_runs<kManyItems>(vd, n, work, s);
}

// The pairs of dimensions and the widths k_slice_pairs is compiled for (two or three extents, a grey or an RGB
// guide, up to 8 lanes of four channels a point), not a line of speed: lattices of other shapes are applied one
// by one because there is no kernel for them.  Five iterations on two images, one by one and together, us:
// 512x512, RGB guide, 4 classes 987 and 658, 15 1140 and 810, 31 1921 and 1423; grey guide, 21 classes 970 and
// 606; 32x96x96 voxels, grey, 21 classes 1125 and 833, RGB, 31 1797 and 1317; 128x128, RGB, 21 classes 919 and
// 239.  Without a kernel: 512x512, 33 classes 2317, guides of two and four channels, 21 classes 1135 and 2522.
bool slice_pairs_take(int pd_a, int pd_b, int vd) {
    return vd >= kManyChannels && vd <= 32 &&
           ((pd_b == 2 && (pd_a == 3 || pd_a == 5)) || (pd_b == 3 && (pd_a == 4 || pd_a == 6)));
}

hipError_t slice_pairs(int pd_a, int pd_b, int vd, int n, const SlicePair *work, hipStream_t s) {
    if (n < 1 || n > kManyItems || !slice_pairs_take(pd_a, pd_b, vd)) return hipErrorInvalidValue;
    const Items<SlicePair> items = items_of_points<kManyItems>(n, work);
    const unsigned blocks = all_blocks(items);
    if (!blocks) return hipSuccess;
    const int lanes = vd <= 16 ? 4 : 8;
    bool tiles = true;
    for (int i = 0; i < n; ++i) tiles = tiles && work[i].map.tile_vertices.table && work[i].tiles_b.table;
    const int Q = (vd - 1 + 3) / 4;
    const unsigned n_rows = tile_rows(Q, blocks, 3);
    const dim3 grid(blocks, tiles ? 1u : (unsigned)(lanes / kPairPoints)), block(tiles ? kTileThreads : kBlock);
#define PLK_PAIR_TILES(A, B, Q)                                                                            \
    case Q:                                                                                                \
        hipLaunchKernelGGL((k_slice_tile_pairs<A + 1, B + 1, Q>), grid, block, tile_lds(Q, n_rows), s, items, \
                           vd, (int)n_rows, point_rows(vd - 1, vd - 1));                                   \
        break;
#define PLK_PAIR(A, B)                                                                                     \
    if (pd_a == A && pd_b == B) {                                                                          \
        if (tiles)                                                                                         \
            switch (Q) {                                                                                   \
                PLK_PAIR_TILES(A, B, 1) PLK_PAIR_TILES(A, B, 2) PLK_PAIR_TILES(A, B, 3) PLK_PAIR_TILES(A, B, 4)                    \
                PLK_PAIR_TILES(A, B, 5) PLK_PAIR_TILES(A, B, 6) PLK_PAIR_TILES(A, B, 7)                    \
                PLK_PAIR_TILES(A, B, 8)                                                                    \
            }                                                                                              \
        else if (lanes == 4)                                                                               \
            hipLaunchKernelGGL((k_slice_pairs<A + 1, B + 1, 4>), grid, block, 0, s, items, vd);            \
        else                                                                                               \
            hipLaunchKernelGGL((k_slice_pairs<A + 1, B + 1, 8>), grid, block, 0, s, items, vd);            \
    }
    PLK_PAIR(3, 2) PLK_PAIR(5, 2) PLK_PAIR(4, 3) PLK_PAIR(6, 3)
#undef PLK_PAIR
#undef PLK_PAIR_TILES
    return hipGetLastError();
}

}  // namespace plk
