// Whole training-step halves of the width-16 network, for the engine: the same kernels as tgk_w16_*, with the batch
// sampled, the losses averaged and the gradient squared on the way.
#pragma once
#include "optimizer.h"

struct W16Weights {
    uint16_t *hi, *lo;
};
// the bytes a batch is drawn from (cuda/dataset.cuh:13-27)
struct W16Data {
    const uint8_t *bytes;
    int64_t size;
    uint64_t seed, step;
};
int w16_norm_count(int depth);
int w16_norm_parts();
// Samples batch `data.step` into `tokens`, forward, backward: gradient, per-position mean losses and w16_norm_count(depth)
// sums of the gradient's squares in w16_norm_parts() parts each.  A context of 4 or 8.
void w16_gradient(hipStream_t stream, int depth, int batch, int context, const W16Weights &weights, const W16Data &data,
                  uint8_t *tokens, void *workspace, float *token_losses, float *means, float *gradient, float *norms);
// AdamW on embedding, scales and head, Muon on the hidden matrices (cuda/optim.cuh:66-119): reads the weights at `from`,
// writes them to `to` (which may be the same).  norms: norm_count sums of squares, in norm_parts parts each (1 or
// w16_norm_parts()).
struct MuonArgs {
    float lr, momentum, weight_decay;
    int ns_steps;
};
void w16_update(hipStream_t stream, int depth, const W16Weights &from, const W16Weights &to, float *momentum, float *variance,
                const float *gradient, const float *norms, int norm_count, int norm_parts, const AdamArgs &adam,
                const MuonArgs &muon);
