// What the wide model's and the width-16 network's optimizer kernels share (cuda/optim.cuh:67-106).  Every fused
// multiply-add is written out, so that the two compile to the same arithmetic.
#pragma once
#include "common.h"
#include <math.h>

struct AdamArgs {
    float lr, beta1, beta2, eps, weight_decay, bc1, sqrt_bc2, clip;
};
// bias correction with the current beta1 (cuda/optim.cuh:90-91), evaluated on the host in fp32
inline AdamArgs adam_args(float lr, float beta1, float beta2, float eps, float weight_decay, float clip, uint64_t step) {
    return AdamArgs{lr, beta1, beta2, eps, weight_decay, 1.f - powf(beta1, float(step + 1)),
                    sqrtf(1.f - powf(beta2, float(step + 1))), clip};
}
// one parameter: returns the new weight, updates m and v
TG_DEVICE float adamw_element(const AdamArgs &a, float decay, float scale, float w, float &m, float &v, float g) {
    const float gs = g * scale;
    m = fmaf(1.f - a.beta1, fmaf(g, scale, -m), m);
    v = fmaf(a.beta2, v, gs * ((1.f - a.beta2) * gs));
    return fmaf(w, fmaf(-a.lr, decay, 1.f), -((a.lr / a.bc1) * m / (sqrtf(v) / a.sqrt_bc2 + a.eps)));
}
// Sum of squares of four elements, in the order every norm pass adds them.
TG_DEVICE float quad_squares(const f32x4 &v) {
    return fmaf(v[3], v[3], fmaf(v[2], v[2], fmaf(v[0], v[0], v[1] * v[1])));
}
// A block of 256 threads adds one value each, in a fixed tree; every thread gets the sum.  `waves`: shared, 4 floats.
TG_DEVICE float block_sum_256(float x, float *waves) {
    x = wave_sum(x);
    if ((threadIdx.x & 63) == 0)
        waves[threadIdx.x >> 6] = x;
    __syncthreads();
    return (waves[0] + waves[1]) + (waves[2] + waves[3]);
}
// Sums of squares of a list of ranges of g, one block of 256 threads per range.  Starts and lengths multiples of 4.
struct SumsqSegment {
    int64_t start, length;
};
struct SumsqSegments {
    const float *g;
    const SumsqSegment *segments;
    int count;
    float *partials;
};
inline void check_sumsq_segments(const SumsqSegments &s) {
    require(s.g && !(reinterpret_cast<uintptr_t>(s.g) & 15), "sumsq_segments: g must be non-null and 16-byte aligned");
    require(s.segments && !(reinterpret_cast<uintptr_t>(s.segments) & 7) && s.partials && s.count > 0 && s.count <= 4096,
            "sumsq_segments: 1..4096 ranges in a device array, and their partials");
}
TG_DEVICE void sumsq_segment(const SumsqSegments &s, int at, float *waves) { // `waves`: shared, 4 floats; the block's first 256 threads
    const SumsqSegment segment = s.segments[at];
    const f32x4 *p = reinterpret_cast<const f32x4 *>(s.g + segment.start);
    const int quads = threadIdx.x < 256 ? int(segment.length >> 2) : 0;
    float sum = 0.f;
#pragma unroll 8
    for (int i = threadIdx.x; i < quads; i += 256) {
        const f32x4 v = p[i];
        sum += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    }
    sum = wave_sum(sum);
    if ((threadIdx.x & 63) == 0 && threadIdx.x < 256)
        waves[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0)
        s.partials[at] = (waves[0] + waves[1]) + (waves[2] + waves[3]);
}
// Clip factor from the norm partials: every block folds the same partials in the same order (cuda/optim.cuh:67-80).
TG_DEVICE float clip_factor(float clip, const float *__restrict__ norm_partials, int norm_count, float *waves) {
    if (!(clip > 0.f))
        return 1.f;
    float sum = 0.f;
    for (int i = threadIdx.x; i < norm_count; i += 256)
        sum += norm_partials[i];
    return fminf(1.f, clip / (sqrtf(block_sum_256(sum, waves)) + 1e-6f));
}
