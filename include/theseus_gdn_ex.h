/*
 * libtheseus_wkv7 -- more of the gated delta rule's C ABI (theseus_gdn.h): sizes for the
 * fastest forms, and the training pair with the layers' q/k normalisation inside.
 */
#ifndef THESEUS_GDN_EX_H
#define THESEUS_GDN_EX_H

#include "theseus_gdn.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The workspace with which theseus_gdn_forward (saved_states = 0) or
 * theseus_gdn_forward_train (1) runs fastest: theseus_gdn_forward_workspace_size, or more
 * where the buffers of more time segments help (few heads). */
size_t theseus_gdn_forward_best_workspace_size(int B, int T, int H, int N, int saved_states);

/* theseus_gdn_forward_train and theseus_gdn_backward with qk_l2norm (as
 * theseus_gdn_forward's): q and k are L2-normalised in the kernels,
 * x / sqrt(sum x^2 + 1e-6) (use_qk_l2norm_in_kernel), and dq, dk are the gradients of q
 * and k as given.  Both calls of a pair take the same flag. */
int theseus_gdn_forward_train_ex(int B, int T, int H, int N, int dtype, int qk_l2norm, const void* q, const void* k,
                                 const void* v, const float* g, const float* beta, const float* s0, void* o,
                                 float* sT, float* ckpt, void* workspace, size_t workspace_bytes,
                                 hipStream_t stream);
int theseus_gdn_backward_ex(int B, int T, int H, int N, int dtype, int qk_l2norm, const void* q, const void* k,
                            const void* v, const float* g, const float* beta, const float* ckpt, const void* dout,
                            const float* dsT, void* dq, void* dk, void* dv, float* dg, float* dbeta, float* ds0,
                            void* workspace, size_t workspace_bytes, hipStream_t stream);

#ifdef __cplusplus
}
#endif
#endif
