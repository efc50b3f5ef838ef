// What the host path takes from the kernels' library beyond the public interface.
#pragma once
#include <stdint.h>

// i8f_linear_w8a16_small_m on the rotated x in one launch: the bits of i8f_rotate128 and that call.  I8F_ERR_UNSUPPORTED, with
// nothing launched, where the two launches are the better way or x, w or ldx are not 16-byte aligned.
extern "C" int i8f_internal_w8a16_rotated(const void *x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const int8_t *w, const float *w_scale,
                                          float w_scale_host, int scale_mode, const void *bias, int bias_dtype, void *out, int64_t N, void *stream);
