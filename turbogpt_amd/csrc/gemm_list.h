// tgk_gemm_wgrad_list for widths that are multiples of `unit` (the public entries' 256, or 128); see tgk_kernels.h.
#pragma once
#include "common.h"
#include "optimizer.h"
#include "../../include/tgk_kernels.h"

size_t wgrad_list_table_bytes(int M, int count, const TgkWgradJob *jobs, int unit);
size_t wgrad_list_workspace(int M, int count, const TgkWgradJob *jobs, int unit);
int wgrad_list_sumsq_count(int M, int count, const TgkWgradJob *jobs, int unit);
void wgrad_list_prepare(int M, int count, const TgkWgradJob *jobs, int unit, void *table, size_t table_bytes);
// `ranges`: tgk_sumsq_segments of gradients that are there already, in the same launch where the tiles are small.  Returns whether
// it did that; where not, they are the caller's.
bool wgrad_list(hipStream_t stream, int M, int count, const TgkWgradJob *jobs, int unit, const void *table, void *workspace,
                size_t workspace_bytes, float *sumsq, const SumsqSegments &ranges = {});

// tgk_gemm_fwd with gelu_out where no backward pass follows: the pre-activation is not written.  0 or -1, as there.
int gemm_fwd_gelu_only(hipStream_t stream, int M, int N, int K, const bf16_t *X, int ldx, const bf16_t *W, int ldw,
                       bf16_t *activation, int lda);
