/*
 * How the last launch of a synchronous operation can end it without a launch of its own behind it (host sources and
 * kernels; nothing here leaves the library).
 */
#ifndef YVEX_ROCM_PUBLICATION_H
#define YVEX_ROCM_PUBLICATION_H

#include <stdint.h>

#include "../../../include/yvex_rocm_kernels.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The arguments of yvex_hip_publish, and where the workgroups of a launch count each other: YVEX_HIP_ARRIVAL_BYTES of
 * device memory that belong to one stream, zero before the launch and zero again behind it. The status word that goes with
 * them starts on eight bytes, and the word behind it counts too. */
typedef struct {
    uint32_t *arrivals;
    uint32_t *host;
    uint32_t sequence;
    int clear;
} yvex_hip_publication;

enum { YVEX_HIP_ARRIVAL_BYTES = 16 * 128 };

/* yvex_hip_matvec, yvex_hip_matvec_quantizing and yvex_hip_argmax_f32 whose last launch publishes by itself where its kernel
 * can: *published says whether it did, yvex_hip_publish is the caller's to make if not. */
int yvex_hip_matvec_publishing(const uint8_t *encoded, unsigned int qtype, uint64_t row_count, uint64_t row_width,
                               uint64_t row_bytes, const void *input, int input_q8, uint64_t input_rows,
                               uint64_t input_stride, const float *additive, float *out, uint64_t out_stride,
                               int output_bf16, int *status, const yvex_hip_publication *publication, int *published,
                               yvex_hip_stream stream);
int yvex_hip_matvec_quantizing_publishing(const uint8_t *encoded, unsigned int qtype, uint64_t row_count,
                                          uint64_t row_width, uint64_t row_bytes, const float *input,
                                          uint64_t input_rows, uint64_t input_stride, const float *additive, float *out,
                                          uint64_t out_stride, int output_bf16, int *status,
                                          const yvex_hip_publication *publication, int *published, yvex_hip_stream stream);
/* (The results are published behind the head: ties, tokens and values end to end, as they lie in device memory.) */
int yvex_hip_argmax_f32_publishing(const float *values, uint64_t row_count, uint64_t row_width, uint32_t *selected_tokens,
                                   float *selected_values, uint64_t *tie_counts, void *scratch, uint64_t scratch_bytes,
                                   int *status, const yvex_hip_publication *publication, int *published,
                                   yvex_hip_stream stream);

#ifdef __cplusplus
}
#endif

#endif
