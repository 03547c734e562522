// norm_params.hpp -- the kernel parameter list shared by the RMSNorm engines
// (norm_kernels.hip, norm_row_kernels.hip).
#pragma once

// Kernel parameters of the NormArgs engines.  A by-value struct is not
// preloaded into SGPRs, so the fields are passed one by one, in this order:
// the counts and the pointers the first loads need (and epsilon) fill the
// first 56 bytes, which arrive in user SGPRs at wave launch (kernarg
// preload), so a wavefront's first row load waits on no scalar load; the
// outputs written only at the end follow.  wpb (wavefronts per workgroup)
// and pair_stride (the row distance of a wavefront's second row) come from
// the host instead of blockDim / gridDim, which are kernarg loads too.
#define ATLAS_NORM_KPARAMS                                                                               \
    uint32_t p_rows, uint32_t p_hidden, uint32_t wpb, uint32_t pair_stride, const float* p_x,              \
        const float* p_residual, const float* p_weight, float* p_out, float p_epsilon, float* p_normalized, \
        float* p_residual_out, const float* p_scale
#define ATLAS_NORM_UNPACK                                                                                  \
    const NormArgs a {                                                                                     \
        p_x, p_weight, p_residual, p_normalized, p_residual_out, p_out, p_scale, p_rows, p_hidden, p_epsilon \
    }
#define ATLAS_NORM_KARGS(a, wpb, pair_stride)                                                                   \
    (a).rows, (a).hidden, (wpb), (pair_stride), (a).x, (a).residual, (a).weight, (a).out, (a).epsilon,          \
        (a).normalized, (a).residual_out, (a).scale
