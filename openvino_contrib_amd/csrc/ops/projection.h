// Projections of few rows with what follows them: what the plugin asks of libhipops beside the public operators of hipops.h, for the
// groups of operators that it finds in a model.
#pragma once

#include "hipops.h"

extern "C" {

/* The products of one input x [rows, k], rows <= 64, with one to three weights [n[i], k], and the
 * operator behind them in the same two launches (HIPOPS_PROJECTION_GLU: in one):
 *   _ROPE  out[i] = x * weights[i]^T, those named by a bit of rotated_outputs with the rotary embedding
 *          of hipops_rope over whole heads (rotate-half; row t of cos and sin is positions[t], or t)
 *   _ADD   out[0] = x * weights[0]^T + residual and, with gamma, normalised = hipops_rms_norm of out[0]
 *   _GLU   out[0] [rows, n[0] / 2] = hipops_glu of x * weights[0]^T
 * Everything is `dtype` (HIPATTN_F16 / BF16) but the tables and gamma; sums and what is done to them are
 * fp32, rounded once (the products are not rounded before).  n[i] is a multiple of 8, k of 64, pointers are
 * 16-byte aligned, what _GLU writes is no part of x, and normalised none of residual
 * (but may be all of it) nor out[0] of gamma; HIPATTN_UNSUPPORTED, with nothing launched, for what the kernels do not take: the
 * operators one by one do.  The workspace holds rows * sum(n) floats or more (not needed for _GLU);
 * hipops_matmul_workspace_size's is enough for every split of k. */
#define HIPOPS_PROJECTION_ROPE 0
#define HIPOPS_PROJECTION_ADD 1
#define HIPOPS_PROJECTION_GLU 2
typedef struct hipops_projection_desc {
    int kind;
    int dtype;
    int num_weights;
    int rotated_outputs, head_size, table_dtype; /* _ROPE */
    int gamma_dtype;                             /* _ADD with gamma */
    float eps;
    int glu_activation, glu_gate_first;          /* _GLU */
    int64_t rows, k;
    int64_t n[3];
    int64_t table_row_stride;
} hipops_projection_desc;
typedef struct hipops_projection_args {
    const void* x;
    const void* weights[3];
    void* outs[3];
    const void* cos;
    const void* sin;
    const int32_t* positions;
    const void* residual;
    const void* gamma;
    void* normalised;
} hipops_projection_args;
hipattn_status hipops_projection(const hipops_projection_desc* desc, const hipops_projection_args* device_tensors,
                                 void* device_workspace, size_t workspace_bytes, hipattn_stream stream);

/* The second half of _ADD with gamma for any number of rows, behind a product that is there: out = product + residual, rounded, and
 * normalised = hipops_rms_norm of it, all [rows, n] of `dtype` (HIPATTN_F16 / BF16); n a multiple of 8 up to 16,384, pointers 16-byte
 * aligned, normalised no part of residual (but it may be all of it) nor out of gamma (HIPATTN_UNSUPPORTED otherwise). */
hipattn_status hipops_residual_norm(const void* device_product, const void* device_residual, const void* device_gamma, void* device_out,
                                    void* device_normalised, int64_t rows, int64_t n, float eps, int dtype, int gamma_dtype,
                                    hipattn_stream stream);

}  // extern "C"
