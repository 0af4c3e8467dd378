// The pointwise step of a dense CRF's mean field: q = softmax(logits + (message_a + message_b)) over
// the classes of every point.  No counterpart in the reference, which holds no CRF code; the loop
// around it is crf.py's.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pl_kernels.h"

namespace plk {

namespace {

// A workgroup takes `kRows` points: their sums go to LDS as they lie in memory (16-byte loads of
// consecutive lanes), every thread then has one point's row there to itself (rows an odd number of
// words apart: no bank conflicts), and the results leave as the logits came.  What bounds it is the
// four arrays' way through memory, each once (q may be one of the others: no __restrict__, everything is
// read before the first barrier and written behind the second): two sums and a softmax as separate passes moved
// eight (2 x 512x512 points of 21 classes: 73.5 us, now 32.3, 5.4 TB/s).
template <int kRows>
__global__ __launch_bounds__(kRows) void k_mean_field_update(float *q, const float *logits, const float *message_a,
                                                              const float *message_b, size_t n_points, int classes) {
    extern __shared__ float rows[];   // [kRows][classes | 1]
    const int pitch = classes | 1;
    const size_t first = (size_t)blockIdx.x * kRows;
    const int n_rows = n_points - first < (size_t)kRows ? (int)(n_points - first) : kRows;
    const size_t base = first * (size_t)classes;
    const int n = n_rows * classes;
    // (kRows * classes floats are a multiple of 16 bytes: a block starts as aligned as its array,
    // and only the last block has a remainder)
    const int n4 = n / 4;
    const float4 *l4 = reinterpret_cast<const float4 *>(logits + base);
    const float4 *a4 = reinterpret_cast<const float4 *>(message_a + base);
    const float4 *b4 = reinterpret_cast<const float4 *>(message_b + base);
    float4 *q4 = reinterpret_cast<float4 *>(q + base);
    // element e of the block is class e % classes of row e / classes; a thread's next four
    // elements are 4 * kRows further on
    const int step_row = 4 * kRows / classes, step_class = 4 * kRows - step_row * classes;
    int row = 4 * (int)threadIdx.x / classes, cls = 4 * (int)threadIdx.x - row * classes;
    const int row0 = row, cls0 = cls;
    for (int i = threadIdx.x; i < n4; i += kRows) {
        const float4 l = l4[i];
        const float4 a = message_a ? a4[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const float4 b = message_a ? b4[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const float x[4] = {l.x + (a.x + b.x), l.y + (a.y + b.y), l.z + (a.z + b.z), l.w + (a.w + b.w)};
        int r = row, c = cls;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            rows[r * pitch + c] = x[k];
            if (++c == classes) {
                c = 0;
                r += 1;
            }
        }
        row += step_row;
        cls += step_class;
        if (cls >= classes) {
            cls -= classes;
            row += 1;
        }
    }
    for (int e = 4 * n4 + (int)threadIdx.x; e < n; e += kRows)
        rows[(e / classes) * pitch + e % classes] =
            logits[base + e] + (message_a ? message_a[base + e] + message_b[base + e] : 0.0f);
    __syncthreads();
    if ((int)threadIdx.x < n_rows) {
        float *own = rows + (int)threadIdx.x * pitch;
        float highest = own[0];
        for (int c = 1; c < classes; ++c) highest = fmaxf(highest, own[c]);
        // (a sum of doubles: one after the other in single precision the exponentials of 128 classes
        // cost the result three times the error of a tree's sum, 1.7e-7 against 5.6e-8 of its norm)
        double wide_sum = 0.0;
        for (int c = 0; c < classes; ++c) {
            const float e = expf(own[c] - highest);
            own[c] = e;
            wide_sum += (double)e;
        }
        const float sum = (float)wide_sum;
        for (int c = 0; c < classes; ++c) own[c] = own[c] / sum;
    }
    __syncthreads();
    row = row0;
    cls = cls0;
    for (int i = threadIdx.x; i < n4; i += kRows) {
        float x[4];
        int r = row, c = cls;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k] = rows[r * pitch + c];
            if (++c == classes) {
                c = 0;
                r += 1;
            }
        }
        q4[i] = make_float4(x[0], x[1], x[2], x[3]);
        row += step_row;
        cls += step_class;
        if (cls >= classes) {
            cls -= classes;
            row += 1;
        }
    }
    for (int e = 4 * n4 + (int)threadIdx.x; e < n; e += kRows)
        q[base + e] = rows[(e / classes) * pitch + e % classes];
}

}  // namespace

hipError_t mean_field_update(float *q, const float *logits, const float *message_a, const float *message_b,
                             size_t n_points, int classes, hipStream_t s) {
    if (n_points == 0) return hipSuccess;
    const uintptr_t all = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(logits) |
                          reinterpret_cast<uintptr_t>(message_a) | reinterpret_cast<uintptr_t>(message_b);
    if (!q || !logits || !message_a != !message_b || all % 16u != 0u || classes < 1 ||
        classes > kMeanFieldMaxClasses)
        return hipErrorInvalidValue;
    // (256 rows of up to 40 classes are 42 KB of LDS, three workgroups a CU; 64 rows of up to 128, 33 KB)
    const bool wide = classes > 40;
    const unsigned rows = wide ? 64 : 256;
    const size_t blocks = (n_points + rows - 1) / rows;
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    const size_t lds = sizeof(float) * rows * (size_t)(classes | 1);
    if (wide)
        hipLaunchKernelGGL((k_mean_field_update<64>), dim3((unsigned)blocks), dim3(64), lds, s, q, logits, message_a,
                           message_b, n_points, classes);
    else
        hipLaunchKernelGGL((k_mean_field_update<256>), dim3((unsigned)blocks), dim3(256), lds, s, q, logits,
                           message_a, message_b, n_points, classes);
    return hipGetLastError();
}

}  // namespace plk
