// Entry points of libmaxsim_amd.so for the torch binding of this package: not
// part of the C ABI of include/maxsim_amd.h.
#pragma once

#include "../../include/maxsim_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Bytes of device workspace (16-byte aligned) that
 * maxsim_internal_contrastive_forward makes use of for these inputs; 0 when
 * it needs none.  `queries` and `documents` are looked at for their alignment
 * only. */
size_t maxsim_internal_contrastive_forward_workspace(maxsim_dtype dtype, const void* queries,
                                                     int64_t num_queries, int64_t Lq,
                                                     const void* documents, int64_t total_d_tokens,
                                                     int64_t num_documents, int64_t dim);

/* maxsim_amd_contrastive_forward_with_argmax (argmax may be NULL) with a
 * workspace; a NULL, misaligned or smaller one gives that entry point's
 * result without it.  Same results, bit for bit, either way. */
int maxsim_internal_contrastive_forward(maxsim_dtype dtype, const void* queries,
                                        int64_t num_queries, int64_t Lq, const void* documents,
                                        int64_t total_d_tokens, const int32_t* document_offsets,
                                        int64_t num_documents, int64_t dim, float* scores,
                                        int32_t* argmax, void* workspace, size_t workspace_bytes,
                                        void* stream);

#ifdef __cplusplus
}
#endif
