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

/* The kernel of that forward: 0 a pair kernel, 1 the tiled one, 2 the K-loop
 * kernel on the rows in place, 3 the K-loop kernel with the workspace. */
int maxsim_internal_contrastive_route(maxsim_dtype dtype, const void* queries, int64_t num_queries,
                                      int64_t Lq, const void* documents, int64_t total_d_tokens,
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

/* 1 where the contrastive gradients' documents allow both in one launch (vec:
 * aligned rows; dd_bucket: the bucketing dd kernel takes the batch). */
int maxsim_internal_contrastive_grads_one_launch(maxsim_dtype dtype, int vec, int dd_bucket,
                                                 int64_t rows, int64_t num_documents,
                                                 int64_t dim);

/* 1 where both padded gradients are one launch: by the gradients' type, whether
 * dd writes whole rows per lane group, and dd's bytes. */
int maxsim_internal_padded_grads_one_launch(int out16, int whole_rows, int64_t dd_bytes);

/* One index array of a layout check: CSR offsets (strictly increasing from 0
 * to `limit`), ids in [0, limit) or lengths in [1, limit]; int32 or int64. */
enum maxsim_check_kind { MAXSIM_CHECK_CSR = 0, MAXSIM_CHECK_IDS = 1, MAXSIM_CHECK_LENGTHS = 2 };
#define MAXSIM_CHECK_ARRAYS 4
typedef struct {
  const void* values; /* device memory */
  int64_t n;
  int64_t limit;
  int kind;
  int is64;
} maxsim_check_array;

/* Checks the arrays on `stream` and writes maxsim_internal_check_words() words
 * of pinned host memory at `status`, which the caller has zeroed: bit 0 done,
 * bit 1 a value is bad, bits 32 and up the longest segment of the first array
 * if it holds CSR offsets. */
int maxsim_internal_check_words(const maxsim_check_array* arrays, int count);
int maxsim_internal_check_layout(const maxsim_check_array* arrays, int count, uint64_t* status,
                                 void* stream);

#ifdef __cplusplus
}
#endif
