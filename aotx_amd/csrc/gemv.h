/* What the Q8_0 products (rgemv.hip) do with their results: fp32 store, fp16 store, residual
 * add, gated unit (SwiGLU), or the rotary turn with the key/value page write. Replaces the
 * kernels that follow aotx_gemv_pass / aotx_gemm_tile in the reference's captured graph
 * (cuda/model/norm.cu:79-105, cuda/model/rope.cu:200-234). */
#ifndef AOTX_GEMV_H
#define AOTX_GEMV_H

#include "aotx_internal.h"

enum {
    AOTX_EPI_F32 = 0,     /* y fp32 [m][ldy] */
    AOTX_EPI_F16 = 1,     /* y fp16 [m][ldy] */
    AOTX_EPI_RESID = 2,   /* y fp32 [m][ldy] += result */
    AOTX_EPI_SWIGLU = 3,  /* segments 0/1 = gate/up; y fp16 act [m][ldy] */
    AOTX_EPI_QKV = 4      /* segments q/k/v; adjacent rotary pairs; qh + pages */
};

/* Rotary + page-write parameters of AOTX_EPI_QKV. */
struct aotx_qkv_epi {
    unsigned short *qh;          /* fp16 [tokens][heads*d] */
    const unsigned int *pos;     /* cache position of each token */
    const unsigned int *agent;   /* slot of each token */
    aotx_state *state;           /* page table + fault count */
    aotx_kvl_shape shape;
    unsigned int layer;
    unsigned int heads;
    unsigned int kv_heads;
    unsigned int head_dim;
    float theta;
    const float *factor;         /* optional rope frequency factors [d/2] */
};

#endif
