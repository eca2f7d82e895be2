/*
 * sisa_hip_ce.h -- the scalars of the linear cross-entropy's mean (libsisa_hip.so; conventions of sisa_hip.h).
 */
#ifndef SISA_HIP_CE_H
#define SISA_HIP_CE_H

#include "sisa_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* n_valid = the number of labels other than ignore_index, as fp32, and inv_n = 1 / n_valid (device scalars). */
int sisa_ce_count(const int64_t* labels, int64_t N, int64_t ignore_index, float* n_valid, float* inv_n, void* stream);

/* mean = (sum of the N rows) / n_valid, the sum in fp64 in a fixed order. */
int sisa_ce_mean(const float* rows, int64_t N, const float* n_valid, float* mean, void* stream);

/* The same over several workgroups, whose partial sums (sisa_ce_workspace_bytes(N) bytes, 8-byte aligned, one call's
 * contents of no use to the next) a second launch adds in order. N >= 1. */
int64_t sisa_ce_workspace_bytes(int64_t N);
int sisa_ce_count_wide(const int64_t* labels, int64_t N, int64_t ignore_index, float* n_valid, float* inv_n,
                       void* workspace, void* stream);
int sisa_ce_mean_wide(const float* rows, int64_t N, const float* n_valid, float* mean, void* workspace, void* stream);

#ifdef __cplusplus
}
#endif

#endif
