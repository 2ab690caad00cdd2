/*
 * libtheseus_wkv7 -- more of the gated delta rule's C ABI (theseus_gdn.h): sizes for the
 * fastest forms.
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

#ifdef __cplusplus
}
#endif
#endif
