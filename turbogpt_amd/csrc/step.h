// Launches of elementwise.hip that the engine makes beside the tgk_* entries: parts of a step that do not wait for one
// another, in one launch.  0 or -1, as there.
#pragma once
#include "common.h"

// tgk_sample_batch and tgk_embed_fwd of what it drew
int sample_embed(hipStream_t stream, const uint8_t *data, int64_t size, uint64_t seed, uint64_t step, int batch, int context,
                 int D, uint8_t *x, uint8_t *y, const uint16_t *table, const uint16_t *positions, uint16_t *out);

// tgk_layernorm_bwd_fold, tgk_embed_bwd_onehot and, where `means` is given, tgk_position_means; nothing accumulates
struct BackwardRest {
    int B, T, D;
    const uint8_t *tokens;
    const uint16_t *dh;
    uint16_t *onehot;
    float *dpositions;
    const float *partials; // the LayerNorms' partial rows, `partials_stride` floats a LayerNorm
    size_t partials_stride;
    int layernorms, partial_rows; // partial_rows is filled in
    const void *targets;
    const float *token_losses;
    float *means;
};
int backward_rest(hipStream_t stream, BackwardRest rest);
