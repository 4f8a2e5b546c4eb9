/*
 * Phase 1 from a query bank in one call each way: attnres_keyed_logits_forward
 * followed by attnres_phase1_forward on its logits, and their backward with the
 * two value gradients already added.  Additions to attnres_hip.h for the shapes
 * that attnres_phase1_bank_fits accepts; its conventions (device pointers,
 * asynchronous on the caller's stream, no allocation, attnres_last_error) hold.
 */
#ifndef ATTNRES_PHASE1_BANK_H
#define ATTNRES_PHASE1_BANK_H

#include "attnres_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* 1 when the calls below take this description (up to 12 sources and 12 sites,
 * rows of a multiple of 4 up to 2048 elements, rows and queries aligned to four
 * elements), else 0: then the composition applies.  Host computation. */
int attnres_phase1_bank_fits(const attnres_keyed_logits_desc* desc);

/* out [Q, n_tok, dim] (dtype), lse [Q, n_tok] fp32.  For a backward: logits
 * [Q, S, n_tok] (dtype) and, with key_norm, inv_rms [S, n_tok] fp32 (NULL when
 * none follows). */
int attnres_phase1_bank_forward(const attnres_keyed_logits_desc* desc, void* out, float* lse, void* logits,
                                float* inv_rms, void* stream);

/* Workspace bytes of attnres_phase1_bank_backward with dqueries (host computation). */
size_t attnres_phase1_bank_backward_workspace_size(const attnres_keyed_logits_desc* desc);

/* grad_out [Q, n_tok, dim] (dtype, aligned to four elements), grad_lse [Q, n_tok]
 * fp32 or NULL (zero) -> dvalues[s] [n_tok, dim] dense, dqueries [Q, dim] (dtype;
 * NULL: not computed, no workspace needed). */
int attnres_phase1_bank_backward(const attnres_keyed_logits_desc* desc, const void* grad_out, const float* grad_lse,
                                 const void* logits, const float* inv_rms, void* const* dvalues, void* dqueries,
                                 void* workspace, size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* ATTNRES_PHASE1_BANK_H */
