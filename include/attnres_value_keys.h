/*
 * Value-derived LR keys with their projection: keys[s] = rms_norm(values[s]) @ W^T
 * and its backward, on the matrix cores, for the shapes attnres_value_keys_fits
 * accepts.  Additions to attnres_hip.h (its attnres_value_norm_* around a library
 * GEMM are the general form); its conventions hold.
 */
#ifndef ATTNRES_VALUE_KEYS_H
#define ATTNRES_VALUE_KEYS_H

#include "attnres_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* 1 when the calls below take this description with this rank: bf16 rows of a
 * multiple of 64 elements up to 4096, aligned to 16 bytes, rank 32, 64 or 128; else 0.
 * Host computation. */
int attnres_value_keys_fits(const attnres_value_key_desc* desc, int32_t rank);

/* weight [rank, dim] dense (dtype, aligned to 16 bytes) -> keys [n_src, n_tok,
 * rank] dense (dtype); inv_rms [n_src, n_tok] fp32 (for the backward; may be NULL). */
int attnres_value_keys_forward(const attnres_value_key_desc* desc, const void* weight, int32_t rank, void* keys,
                               float* inv_rms, void* stream);

/* Workspace bytes of attnres_value_keys_backward (host computation). */
size_t attnres_value_keys_backward_workspace_size(const attnres_value_key_desc* desc, int32_t rank);

/* grad_keys [n_src] device pointers, each [n_tok, rank] dense and aligned to 16
 * bytes, or NULL (zero); keys and inv_rms: the forward's.  grad_values [n_src]
 * pointers, each [n_tok, dim] dense (the pointer array NULL: not computed);
 * grad_weight [rank, dim] (dtype; NULL: not computed). */
int attnres_value_keys_backward(const attnres_value_key_desc* desc, const void* weight, int32_t rank,
                                const void* const* grad_keys, const void* keys, const float* inv_rms,
                                void* const* grad_values, void* grad_weight, void* workspace, size_t workspace_bytes,
                                void* stream);

#ifdef __cplusplus
}
#endif

#endif /* ATTNRES_VALUE_KEYS_H */
