// The applies of several lattices, pass by pass in one launch each, and the message passing of a dense
// CRF on them: both messages of a point are sliced by the same lanes, added up, and the mean field's
// softmax taken where they are.  No counterpart in the reference (one lattice at a time,
// src/LatticeFilterKernel.cpp:152-179, and no CRF).
//
// At 512x512 points of 21 classes every pass of one lattice is a kernel of 5 to 25 us that fills a third
// of the GPU, and an iteration on two images and their four lattices was 22 launches on four streams (and 13
// events): the host needed as long for them as the GPU.  Here it is six or seven launches on one stream.
// Two images, five iterations: 1154 us as launches of their own, 720 this way.
#include "pl_device.h"
#include "pl_kernels.h"

namespace plk {

namespace {

using namespace device;

struct alignas(4) FourFloats {
    float c[4];
};

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
                                                const float *__restrict__ values, unsigned vblock,
                                                const unsigned (&slot)[kPairPoints], const int (&n)[kPairPoints],
                                                int sub, float (&message)[kPairPoints][4]) {
    constexpr int E = (D1 + L - 1) / L;     // replay rows a lane reads per point
    ReplayEntry mine[kPairPoints][E];
#pragma unroll
    for (int q = 0; q < kPairPoints; ++q) {
        const size_t t = (size_t)vblock * kBlock * D1 + slot[q];
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const int r = u * L + sub;
            mine[q][u] = replay[(size_t)(r < D1 ? r : 0) * kBlock + t];
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
    sliced_channels<D1A, L>(vd, work.replay_a, work.values_a, vblock, slot, n, sub, a);
    sliced_channels<D1B, L>(vd, work.replay_b, work.values_b, vblock, slot, n, sub, b);
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

}  // namespace

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
    Items<SlicePair> items{};
    items.n = n;
    for (int i = 0; i < n; ++i) {
        items.item[i] = work[i];
        items.blocks[i] = multiple_of_xcds(work[i].map.n_blocks);
    }
    const unsigned blocks = all_blocks(items);
    if (!blocks) return hipSuccess;
    const int lanes = vd <= 16 ? 4 : 8;
    const dim3 grid(blocks, (unsigned)(lanes / kPairPoints)), block(kBlock);
#define PLK_PAIR(A, B)                                                                                     \
    if (pd_a == A && pd_b == B) {                                                                          \
        if (lanes == 4)                                                                                    \
            hipLaunchKernelGGL((k_slice_pairs<A + 1, B + 1, 4>), grid, block, 0, s, items, vd);            \
        else                                                                                               \
            hipLaunchKernelGGL((k_slice_pairs<A + 1, B + 1, 8>), grid, block, 0, s, items, vd);            \
    }
    PLK_PAIR(3, 2) PLK_PAIR(5, 2) PLK_PAIR(4, 3) PLK_PAIR(6, 3)
#undef PLK_PAIR
    return hipGetLastError();
}

}  // namespace plk
