// Whole training-step halves of the width-16 network, for the engine: the same kernels as tgk_w16_*, with the batch
// sampled, the losses averaged and the gradient squared on the way.  Batches in flight may share their launches: a few
// sequences fill a few compute units, and a launch costs the host more than it costs them.
#pragma once
#include "optimizer.h"

constexpr int W16_BATCHES = 16; // most batches (or optimizer steps) a launch takes
struct W16Weights {
    uint16_t *hi, *lo;
};
// the bytes a batch is drawn from (cuda/dataset.cuh:13-27)
struct W16Data {
    const uint8_t *bytes;
    int64_t size;
    uint64_t seed;
};
// One batch: the weights that it reads, the step that it is drawn for, and what it leaves: its tokens, losses and their
// per-position means, the gradient, and w16_norm_count(depth) sums of the gradient's squares in w16_norm_parts() parts each.
struct W16Batch {
    W16Weights weights;
    uint64_t step;
    uint8_t *tokens;
    void *workspace;
    float *token_losses, *means, *gradient, *norms;
};
int w16_blocks(int batch, int context); // of a batch's forward and backward pass
int w16_norm_count(int depth);
int w16_norm_parts();
// Samples the batches, forward, backward.  A context of 4 or 8.  flying: how many such calls run side by side, on streams of their own.
void w16_gradients(hipStream_t stream, int depth, int batch, int context, const W16Data &data, int count, int flying, const W16Batch *batches);
// AdamW on embedding, scales and head, Muon on the hidden matrices (cuda/optim.cuh:66-119): each step reads the weights at
// `from`, which are those that the step before it wrote, and writes them to `to` (which may be the same).  norms:
// norm_count sums of squares, in norm_parts parts each (1 or w16_norm_parts()).
struct MuonArgs {
    float lr, momentum, weight_decay;
    int ns_steps;
};
struct W16Step {
    W16Weights from, to;
    const float *gradient, *norms;
    AdamArgs adam;
    MuonArgs muon;
};
void w16_updates(hipStream_t stream, int depth, float *momentum, float *variance, int norm_count, int norm_parts, int count,
                 const W16Step *steps);
