// Shared declarations of libmortar_hip.so (host side).
#ifndef MORTAR_INTERNAL_H
#define MORTAR_INTERNAL_H

#include "../../include/mortar_hip.h"

// Records the calling thread's error message and returns `code`.
int mortar_fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));

int mortar_check_bcsr_host(const int32_t *row_ptr, const int16_t *col, int32_t Rb, int32_t Cb);

// The kernels address the octet stream with 32-bit byte offsets (1 KiB of 4-bit codes per octet): refuses larger matrices.
// Cb and seg_cb are positive.
__attribute__((visibility("hidden"))) int mortar_check_octets(const mortar_bcsr_t *W);

// Plain product on the +-1 / 0 codes alone, unrounded: y32[m, :] = sum over the kept blocks of codes . x[m, :] in fp32
// (the one-scale kernels with the scale left out).  Returns MORTAR_NO_KERNEL when the pack has no such kernel for M rows.
__attribute__((visibility("hidden"))) int mortar_spmm_codes_f32(const mortar_bcsr_t *W, const int32_t *sched, const uint16_t *x,
                                                                 int64_t M, int64_t ldx, float *y32, int64_t ldy, void *stream);

// qv[m, :] = x[m, :] W^T + bias for few tokens (bias may be null): K shared by the waves of a workgroup.  The caller has checked
// the shapes: d_in % 8 == 0, d_in <= 2048, d_out % 4 == 0, all pointers and rows 16-byte aligned.  xn [M, d_in], M <= 16: the rows of x
// are RMS-normalised first (norm_w may be null) and written there as well.
__attribute__((visibility("hidden"))) int mortar_router_project_skinny(const uint16_t *x, int64_t M, int32_t d_in, int64_t ldx, const float *wq,
                                                                       int32_t d_out, const float *bias, float *qv, int64_t ldq, void *stream,
                                                                       const uint16_t *norm_w = nullptr, float eps = 0.f, uint16_t *xn = nullptr);

#endif
