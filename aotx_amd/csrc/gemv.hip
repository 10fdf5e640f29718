/* Q8_0 rows of a tensor as fp16 (the products over Q8_0 are in rgemv.hip). */
#include "aotx_internal.h"

#include <algorithm>

/* Dequantize rows to fp16 (cuda/model/dequant.cu:9-70): half(q * scale). */
__global__ void aotx_q8_dequant_kernel(const unsigned char *w, unsigned int k,
                                       unsigned int first, unsigned int rows,
                                       unsigned short *out)
{
    unsigned long long total = (unsigned long long)rows * k;
    unsigned long long row_bytes = (unsigned long long)(k / 32u) * 34ull;
    for (unsigned long long i = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x;
         i < total; i += (unsigned long long)gridDim.x * blockDim.x) {
        unsigned long long r = i / k;
        unsigned int c = (unsigned int)(i - r * k);
        const unsigned char *blk = w + (first + r) * row_bytes + (c / 32u) * 34ull;
        unsigned short sb = (unsigned short)(blk[0] | (blk[1] << 8));
        float scale = aotx_h2f(sb);
        int q = (int)(signed char)blk[2u + c % 32u];
        out[i] = aotx_f2h((float)q * scale);
    }
}

extern "C" int aotx_q8_dequant(const void *w, unsigned int k, unsigned int first_row,
                               unsigned int rows, void *out, void *stream)
{
    if (w == nullptr || out == nullptr || k % 32u != 0u || rows == 0u) return 1;
    unsigned long long total = (unsigned long long)rows * k;
    unsigned int blocks = (unsigned int)std::min<unsigned long long>((total + 255u) / 256u, 65535ull);
    hipLaunchKernelGGL(aotx_q8_dequant_kernel, dim3(blocks), dim3(256), 0, aotx_stream(stream),
                       (const unsigned char *)w, k, first_row, rows, (unsigned short *)out);
    AOTX_LAUNCH_CHECK();
    return 0;
}
