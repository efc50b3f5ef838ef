// What the host path takes from the kernels' library beyond the public interface.
#pragma once
#include <stdint.h>

// i8f_quant_rowwise without a rotation and, in the same launch, t = x A^T: x [M,K] and lora_a [rank,K] of one 16-bit dtype, t
// [M,rank] of it (binary32 sums, one rounding).  K % 64 == 0, rank 16 or 32 with K <= 6144, 48 or 64 with K <= 4096, 16-byte aligned operands and
// ldx % 8 == 0, else I8F_ERR_UNSUPPORTED with nothing launched.
extern "C" int i8f_internal_quant_lora(const void *x, int dtype, int64_t M, int64_t K, int64_t ldx, const void *lora_a, int64_t rank, int8_t *q,
                                       float *scale, void *t, void *stream);
