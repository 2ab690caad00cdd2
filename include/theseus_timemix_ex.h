/*
 * libtheseus_wkv7 -- more of the fused TimeMix C ABI (theseus_timemix.h): fewer launches for
 * calls without gradients.
 */
#ifndef THESEUS_TIMEMIX_EX_H
#define THESEUS_TIMEMIX_EX_H

#include "theseus_timemix.h"

#ifdef __cplusplus
extern "C" {
#endif

/* theseus_tm_kk_fwd and theseus_tm_add_param_fwd in one launch: also w = (w0 + zw) in bf16. */
int theseus_tm_kk_w_fwd(int B, int T, int C, const void* k, const void* za, const float* a0, const float* k_k,
                        const float* k_a, void* kw, void* aw, void* bw, const void* zw, const float* w0, void* w,
                        hipStream_t stream);
/* n <= 16 parameter vectors of C elements (dtypes: theseus_wkv7_dtype each) as the float32
 * rows [n][C] that the kernels here read; src and dtypes are read during the call only. */
int theseus_tm_pack_params(int n, int C, const void* const* src, const int* dtypes, float* out,
                           hipStream_t stream);

#ifdef __cplusplus
}
#endif
#endif
