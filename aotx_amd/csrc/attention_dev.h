/* Device code of paged decode attention (attention.hip): the per-workgroup body.
 */
#ifndef AOTX_ATTENTION_DEV_H
#define AOTX_ATTENTION_DEV_H

#include "aotx_internal.h"
#include "coherent.h"

typedef unsigned int aotx_u4a __attribute__((ext_vector_type(4)));
typedef _Float16 aotx_h4a __attribute__((ext_vector_type(4)));
typedef short aotx_s4a __attribute__((ext_vector_type(4)));
typedef _Float16 aotx_h8a __attribute__((ext_vector_type(8)));
typedef float aotx_f4a __attribute__((ext_vector_type(4)));

struct aotx_attn_args {
    const unsigned short *q;      /* fp16 [tokens][heads][d] */
    unsigned short *out;          /* fp16 [tokens][heads][d] */
    const unsigned int *pos;      /* [tokens] */
    const unsigned int *agent;    /* [tokens] */
    const unsigned int *m_dev;    /* device token count, or null */
    unsigned int tokens;
    unsigned int heads;
    unsigned int kv_heads;
    unsigned int layer;
    unsigned int splits;          /* chunks per (token, KV head) at most */
    unsigned int chunk_max;       /* the largest context planned for */
    aotx_kvl_shape shape;
    aotx_state *state;
    float *partial;               /* [tokens*kv_heads][splits][G*(d+2)] */
    unsigned int *count;          /* [tokens*kv_heads] chunk arrivals, zero between launches */
    unsigned int out_frag;        /* out in the fragment layout (aotx_xfrag_at) */
};

/* Half index of out for query row t, head h, dimension e. */
static __device__ __forceinline__ unsigned long long aotx_attn_out_at(const aotx_attn_args &a,
                                                                    unsigned int t, unsigned int h,
                                                                    unsigned int e, unsigned int d)
{
    return a.out_frag ? aotx_xfrag_at(t, h * d + e) : ((unsigned long long)t * a.heads + h) * d + e;
}

#define ATTN_CHUNK_ALIGN 64u   /* a chunk is a whole number of 16-position blocks per wave */
#define ATTN_MAX_SPLITS 32u
#define ATTN_TARGET_GROUPS 192u
/* Cache policy bits of the decode key/value block loads: 2 is the non-temporal (nt) bit.
 * Each block is read once per step, so it is streamed past the caches instead of being
 * kept there (batch 32 at context 2048: 50.2 -> 46.0 us per launch; sc1, 16, no change).
 * Prompt pieces keep the default policy: their runs re-read a sequence's prefix. */
#ifndef AOTX_ATTN_CPOL
#define AOTX_ATTN_CPOL 2
#endif
#ifndef AOTX_ATTN_NT_BLOCKS
#define AOTX_ATTN_NT_BLOCKS 32u
#endif

/* A kernel-constant word (the device token count) read through the scalar cache. */
static __device__ __forceinline__ unsigned int aotx_attn_scalar(const unsigned int *p)
{
    return *(const __attribute__((address_space(4))) unsigned int *)p;
}

/* 2^x with the hardware v_exp_f32: exp2(-inf) = 0, results below 2^-126 flush to 0 (weights
 * that small do not change an fp32 sum of weights of order one). */
static __device__ __forceinline__ float aotx_exp2(float x)
{
    return __builtin_amdgcn_exp2f(x);
}

/* Chunk partials cross workgroups on different XCDs: device-scope stores and loads. */
static __device__ __forceinline__ void aotx_attn_put(float *p, float v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
static __device__ __forceinline__ float aotx_attn_get(const float *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* Chunk length of a token with n positions under S splits (whole 64-position units). */
static __device__ __forceinline__ unsigned int aotx_attn_chunk(unsigned int n, unsigned int S)
{
    unsigned int chunk = (n + S - 1u) / S;
    return (chunk + ATTN_CHUNK_ALIGN - 1u) / ATTN_CHUNK_ALIGN * ATTN_CHUNK_ALIGN;
}

/* The block loop shared by the attention bodies. They expect, in scope: a, kv, agent, b1,
 * lane, r, g, kbyte, vbyte, wbase, pages, kr, vr, absent, CPOL, KK, VP, NS, VS, D, qb, o,
 * mrun, lrun, missing, scale, p0, plim, vw (this wave's LDS value slot) and vtr.
 * MMA_WINDOW(B0): the page addresses of blocks B0 .. B0 + 63 (one per lane).
 * MMA_LOAD(BUF, B): block B's keys and values into register buffer BUF.
 * MMA_COMPUTE(BUF, B): block B's scores, online softmax and P . V. */
#define MMA_WINDOW(B0)                                                                      \
    do {                                                                                    \
        wbase = (B0);                                                                       \
        unsigned int bl = wbase + lane;                                                     \
        pages = bl < b1 ? (unsigned long long)aotx_kvl_block(a.shape, kv, agent, a.layer, bl * 16u) \
                        : 0ull;                                                             \
    } while (0)
#define MMA_LOAD(BUF, B)                                                                    \
    do {                                                                                    \
        if ((B) - wbase >= 64u) MMA_WINDOW(B);                                              \
        unsigned long long pb = __shfl(pages, (int)((B) - wbase), 64);                     \
        pb = ((unsigned long long)(unsigned int)__builtin_amdgcn_readfirstlane((unsigned int)(pb >> 32)) << 32) \
           | (unsigned long long)(unsigned int)__builtin_amdgcn_readfirstlane((unsigned int)pb); \
        absent[BUF] = pb == 0ull;                                                           \
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(                      \
            (void *)pb, (short)0, absent[BUF] ? 0 : (int)a.shape.block_bytes, 0x00020000);  \
        _Pragma("unroll") for (int kk = 0; kk < KK; ++kk)                                   \
            kr[BUF][kk] = __builtin_amdgcn_raw_buffer_load_b128(rs, kbyte + kk * 64, 0, CPOL); \
        _Pragma("unroll") for (int u = 0; u < VP; ++u)                                      \
            vr[BUF][u] = __builtin_amdgcn_raw_buffer_load_b128(rs, vbyte + u * 1024, 0, CPOL); \
    } while (0)

#define MMA_COMPUTE(BUF, B)                                                                 \
    do {                                                                                    \
        if (absent[BUF]) missing = 1;                                                       \
        aotx_f4a sc = {0.0f, 0.0f, 0.0f, 0.0f};                                             \
        _Pragma("unroll") for (int kk = 0; kk < KK; ++kk)                                   \
            sc = __builtin_amdgcn_mfma_f32_16x16x32_f16(                                    \
                __builtin_bit_cast(aotx_h8a, kr[BUF][kk]), qb[kk], sc, 0, 0, 0);             \
        /* the block's values into this wave's LDS slot (row-major, padded rows) */         \
        _Pragma("unroll") for (int u = 0; u < VP; ++u) {                                    \
            const unsigned int piece = (unsigned int)u * 64u + lane;                        \
            *(aotx_u4a *)(vw + (piece / (D / 8)) * VS + (piece % (D / 8)) * 8u) = vr[BUF][u]; \
        }                                                                                   \
        float pr[4];                                                                        \
        float mb = -INFINITY;                                                               \
        _Pragma("unroll") for (int i = 0; i < 4; ++i) {                                     \
            const unsigned int p = (B) * 16u + 4u * g + (unsigned int)i;                    \
            const bool ok = p >= p0 && p < plim && !absent[BUF];                            \
            pr[i] = ok ? sc[i] * scale : -INFINITY;                                         \
            mb = fmaxf(mb, pr[i]);                                                          \
        }                                                                                   \
        mb = fmaxf(mb, __shfl_xor(mb, 16, 64));                                             \
        mb = fmaxf(mb, __shfl_xor(mb, 32, 64));                                             \
        const float mnew = fmaxf(mrun, mb);                                                 \
        /* 0 from -inf; a column with no position yet keeps its (empty) sums */           \
        const float shift = mnew == -INFINITY ? 1.0f : aotx_exp2(mrun - mnew);              \
        mrun = mnew;                                                                        \
        aotx_h4a pa;                                                                        \
        float mass = 0.0f;                                                                  \
        _Pragma("unroll") for (int i = 0; i < 4; ++i) {                                     \
            const _Float16 ph = mnew == -INFINITY ? (_Float16)0.0f                          \
                              : (_Float16)aotx_exp2(pr[i] - mnew);   /* 0 when masked */    \
            pa[i] = ph;                                                                     \
            mass += (float)ph;                                                              \
        }                                                                                   \
        lrun = lrun * shift + mass;                                                         \
        /* the accumulators of heads 4g + i take those heads' shifts */                     \
        if (__any(shift != 1.0f)) {                                                         \
            float sh[4];                                                                    \
            _Pragma("unroll") for (int i = 0; i < 4; ++i) sh[i] = __shfl(shift, (int)(4u * g) + i, 64); \
            _Pragma("unroll") for (int cc = 0; cc < NS; ++cc)                               \
                _Pragma("unroll") for (int i = 0; i < 4; ++i) o[cc][i] *= sh[i];            \
        }                                                                                   \
        _Pragma("unroll") for (int cc = 0; cc < NS; ++cc) {                                 \
            /* B[k = 4g + i][n = r] = V[row 4g + i][16 cc + r]: one transposing read, each \
             * lane addressing 4 halves of a row (aotx_vtr) */                               \
            const aotx_s4a t4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(                    \
                (__attribute__((address_space(3))) aotx_s4a *)(vw + vtr + 16u * (unsigned int)cc)); \
            o[cc] = __builtin_amdgcn_mfma_f32_16x16x16f16(pa, __builtin_bit_cast(aotx_h4a, t4), \
                                                          o[cc], 0, 0, 0);                  \
        }                                                                                   \
    } while (0)

/* One workgroup = W waves = one (token, KV head, context chunk); each wave takes a
 * contiguous run of 16-position layout blocks. Per wave and block, on the matrix cores:
 *   - scores S[pos][head] = K . q^T: one v_mfma_f32_16x16x32_f16 per 32 of d, keys as the A
 *     operand straight from memory (lane (r, g) holds row r, d 32kk + 8g..+7), the query
 *     heads of the KV head as the B columns (heads past G are zero);
 *   - the score layout (lane (r, g): head r, positions 4g..4g+3) is the A-operand layout of
 *     v_mfma_f32_16x16x16_f16, so the probabilities feed P . V as fp16 (the mass adds the
 *     same rounded probabilities, so numerator and denominator agree);
 *   - the values need positions along k: the wave writes its block (row-major, rows padded
 *     against bank conflicts) to a private LDS slot and reads 16-bit columns back;
 *   - online softmax in base 2 per head with a max over the 4 lane groups of the head.
 * The output accumulators hold heads 4g..4g+3 x 16 d columns per lane and PV step. */
template <int D, int G, int W, int QT>
static __device__ __forceinline__ void aotx_attend_body(const aotx_attn_args &a, unsigned int bx)
{
    static_assert(QT == 1, "one query per workgroup: prompt pieces take aotx_attend_runs");
    constexpr int C = G * QT;           /* score columns: G heads */
    static_assert(C <= 16, "one MFMA tile of query columns");
    constexpr int KK = D / 32;          /* score MFMA steps */
    constexpr int VP = D / 32;          /* 16-byte value pieces per lane per block */
    constexpr int NS = D / 16;          /* P.V MFMAs (16 d columns each) */
    constexpr int VS = D + 8;           /* LDS row stride of a value block (halves) */
    __shared__ float wm[W][C], wl[W][C];
    __shared__ float wo[W][C][D];
    __shared__ __attribute__((aligned(16))) unsigned short vl[W][16 * VS];

    const unsigned int lane = threadIdx.x & 63u;
    const unsigned int wave = threadIdx.x >> 6;
    const unsigned int r = lane & 15u, g = lane >> 4;
    /* one unconditional scalar load (of the device count, or of a word of the positions
     * when there is none, then not used): a load under a condition would be waited for
     * where the paths join. (Not the address of an argument: that would point at a private
     * copy of the arguments, which a scalar load cannot read.) */
    const unsigned int counted = aotx_attn_scalar(a.m_dev != nullptr ? a.m_dev : a.pos);
    unsigned int tokens = a.m_dev != nullptr ? counted : a.tokens;
    unsigned int S, c, kh, t, n, st, p0, p1, nq = 1u, plim;
    unsigned int agent;
    S = a.splits;
    /* chunk-major: the workgroups of one chunk index are consecutive, so they spread
     * over every XCD whichever chunks are empty (dispatch goes round the XCDs) */
    const unsigned int units = a.tokens * a.kv_heads;
    c = bx / units;
    const unsigned int rest = bx - c * units;
    kh = rest % a.kv_heads;
    t = rest / a.kv_heads;
    /* the token's position and slot are read before its row count is known (t is below
     * the launch's token capacity, so both words exist): one memory round trip for all
     * three, where a load after the count's test would wait for the count first */
    const unsigned int pos_t = a.pos[t];
    agent = a.agent[t];
    __builtin_amdgcn_sched_barrier(0);
    if (tokens > a.tokens) tokens = a.tokens;
    /* the test reads both words, so neither load is sunk past it (a position of all
     * ones, which no sequence reaches, would end the workgroup as a token past the
     * count does) */
    if (t >= tokens || (pos_t & agent) == 0xFFFFFFFFu) return;
    n = pos_t + 1u;
    const unsigned int chunk = aotx_attn_chunk(n, S);
    st = (n + chunk - 1u) / chunk;
    if (c >= st) return;
    p0 = c * chunk;
    p1 = (p0 + chunk < n) ? p0 + chunk : n;
    plim = p1;
    const unsigned int nblk = (p1 - p0 + 15u) / 16u;
    const unsigned int per = (nblk + W - 1u) / W;
    const unsigned int b0 = p0 / 16u + wave * per;
    unsigned int b1 = b0 + per;
    if (b1 > (p1 + 15u) / 16u) b1 = (p1 + 15u) / 16u;
    const aotx_kv_table *kv = &a.state->kv;
    const float scale = 1.4426950408889634f / sqrtf((float)D);

    aotx_h8a qb[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        aotx_u4a w = {0u, 0u, 0u, 0u};
        const unsigned int qi = r / (unsigned int)G, hh = r % (unsigned int)G;
        if (r < (unsigned int)C && qi < nq)
            w = co_load4(a.q + ((unsigned long long)(t + qi) * a.heads + kh * G + hh) * D
                             + 32 * kk + 8 * g);
        qb[kk] = __builtin_bit_cast(aotx_h8a, w);
    }
    float mrun = -INFINITY, lrun = 0.0f;     /* head r of this lane */
    aotx_f4a o[NS];
#pragma unroll
    for (int cc = 0; cc < NS; ++cc) o[cc] = (aotx_f4a){0.0f, 0.0f, 0.0f, 0.0f};
    int missing = 0;
    const unsigned int kbyte = ((kh * AOTX_KVL_BLOCK + r) * D + 8u * g) * 2u;
    const unsigned int vbyte = ((a.kv_heads + kh) * AOTX_KVL_BLOCK * D + lane * 8u) * 2u;
    unsigned short *vw = vl[wave];
    /* ds_read_tr16_b64: lane j of a 16-lane group gets halves j % 4 of the chunks that
     * lanes 4e + j / 4 address, e = 0..3; lane (r, g) = 16 g + 4 i + q addresses row 4g + i,
     * halves 4q..4q+3 of a 16-column slice, so that it gets column r of rows 4g..4g+3 */
    const unsigned int vtr = (4u * g + (lane & 15u) / 4u) * VS + 4u * (lane & 3u);

    aotx_u4a kr[2][KK], vr[2][VP];
    bool absent[2];
    unsigned long long pages = 0ull;
    unsigned int wbase = b0;
    /* The next block's loads are issued on every step: past the wave's last block the page
     * address is zero and the loads go through a zero-size resource (they return zeros
     * and touch no memory; that buffer is never computed). With a load on one path only,
     * the compiler's wait before a block's MFMAs would also cover part of the next block's
     * loads. */
#define MMA_RUN()                                                                           \
    do {                                                                                    \
        if (b0 < b1) {                                                                      \
            unsigned int b = b0;                                                            \
            MMA_WINDOW(b0);                                                                 \
            MMA_LOAD(0, b);                                                                 \
            for (;;) {                                                                      \
                MMA_LOAD(1, b + 1u);                                                        \
                MMA_COMPUTE(0, b);                                                          \
                b += 1u;                                                                    \
                if (b >= b1) break;                                                         \
                MMA_LOAD(0, b + 1u);                                                        \
                MMA_COMPUTE(1, b);                                                          \
                b += 1u;                                                                    \
                if (b >= b1) break;                                                         \
            }                                                                               \
        }                                                                                   \
    } while (0)
    /* runs of up to AOTX_ATTN_NT_BLOCKS blocks per wave stream with the policy above; longer
     * runs (one wave's run sets a long sequence's time) keep the default policy */
    if (QT == 1 && b1 - b0 <= AOTX_ATTN_NT_BLOCKS) {
        constexpr int CPOL = AOTX_ATTN_CPOL;
        MMA_RUN();
    } else {
        constexpr int CPOL = 0;
        MMA_RUN();
    }
#undef MMA_RUN
    /* a head's mass over its 4 lane groups */
    lrun += __shfl_xor(lrun, 16, 64);
    lrun += __shfl_xor(lrun, 32, 64);
    missing = __any(missing);
    if (missing && lane == 0u) atomicAdd(&a.state->faults, 1u);
    if (g == 0u && r < (unsigned int)C) {
        wm[wave][r] = missing ? -INFINITY : mrun;
        wl[wave][r] = missing ? 0.0f : lrun;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const unsigned int head = 4u * g + (unsigned int)i;
        if (head < (unsigned int)C) {
#pragma unroll
            for (int cc = 0; cc < NS; ++cc) wo[wave][head][16 * cc + r] = missing ? 0.0f : o[cc][i];
        }
    }
    __syncthreads();
    /* merge the W waves in wave order */
    const unsigned int unit = t * a.kv_heads + kh;
    const unsigned int stride = G * (D + 2);
    float *mine = a.partial + ((unsigned long long)unit * S + c) * stride;
    for (unsigned int idx = threadIdx.x; idx < (unsigned int)(C * D / 2); idx += 64u * W) {
        const unsigned int j = idx / (D / 2), e = 2u * (idx - j * (D / 2));
        /* column j: query j / G (of the prompt piece; 0 in decode), head j % G */
        const unsigned int qj = j / (unsigned int)G, hj = j % (unsigned int)G;
        if (qj >= nq) continue;
        float top = wm[0][j];
#pragma unroll
        for (int w = 1; w < W; ++w) top = fmaxf(top, wm[w][j]);
        float msum = 0.0f, osum[2] = {0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < W; ++w) {
            float f = (wm[w][j] == -INFINITY) ? 0.0f : exp2f(wm[w][j] - top);
            msum += wl[w][j] * f;
            osum[0] += wo[w][j][e] * f;
            osum[1] += wo[w][j][e + 1u] * f;
        }
        if (st == 1u) {
            float back = msum > 0.0f ? 1.0f / msum : 0.0f;
            co_store2h(a.out + aotx_attn_out_at(a, t + qj, kh * G + hj, e, D),
                           aotx_f2h(osum[0] * back), aotx_f2h(osum[1] * back));
        } else {
            aotx_attn_put(mine + j * (D + 2) + 2 + e, osum[0]);
            aotx_attn_put(mine + j * (D + 2) + 3 + e, osum[1]);
            if (e == 0u) {
                aotx_attn_put(mine + j * (D + 2), top);
                aotx_attn_put(mine + j * (D + 2) + 1, msum);
            }
        }
    }
    if (st == 1u) return;
    /* The last chunk of the (token, KV head) to finish merges all of them, in chunk order:
     * M = max m_c, out = half(sum_c o_c 2^(m_c - M) / sum_c l_c 2^(m_c - M)). Partials
     * are written and read as device-scope accesses (through to the point where all XCDs
     * meet, past the per-XCD L2), and every one of this workgroup's writes has completed
     * before its arrival is counted, so no cache write-back or invalidation is needed. The
     * last arrival puts the counter back to zero for the next launch. */
    __shared__ unsigned int last;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0u) {
        last = atomicAdd(a.count + unit, 1u) == st - 1u ? 1u : 0u;
        if (last != 0u) atomicExch(a.count + unit, 0u);
    }
    __syncthreads();
    if (last == 0u) return;
    const float *all = a.partial + (unsigned long long)unit * S * stride;
    /* One output value per lane: a wave's 64 lanes lie in one head (D is 64 or 128). Lane
     * c < st reads chunk c's max and mass and the wave shares them (uniform-index
     * shuffles), so a lane issues st + 2 loads, all in flight together, and the sums run
     * in chunk order as before. */
    for (unsigned int idx = threadIdx.x; idx < (unsigned int)(G * D); idx += 64u * W) {
        const unsigned int j = idx / D, e = idx % D;
        const float *col = all + j * (D + 2);
        const unsigned int cl = lane < st ? lane : 0u;
        const float m_l = aotx_attn_get(col + cl * stride);
        const float l_l = aotx_attn_get(col + cl * stride + 1u);
        float oc[ATTN_MAX_SPLITS];
#pragma unroll
        for (unsigned int cc = 0; cc < ATTN_MAX_SPLITS; ++cc)
            oc[cc] = cc < st ? aotx_attn_get(col + cc * stride + 2u + e) : 0.0f;
        float top = lane < st ? m_l : -INFINITY;
#pragma unroll
        for (int sh = 1; sh < 64; sh <<= 1) top = fmaxf(top, __shfl_xor(top, sh, 64));
        const float f_l = lane < st && m_l != -INFINITY ? aotx_exp2(m_l - top) : 0.0f;
        float msum = 0.0f, osum = 0.0f;
#pragma unroll
        for (unsigned int cc = 0; cc < ATTN_MAX_SPLITS; ++cc) {
            if (cc < st) {
                const float f = __shfl(f_l, (int)cc, 64);
                msum += __shfl(l_l, (int)cc, 64) * f;
                osum += oc[cc] * f;
            }
        }
        const float back = msum > 0.0f ? 1.0f / msum : 0.0f;
        const float v = osum * back;
        const float v1 = __shfl_down(v, 1, 64);
        if ((e & 1u) == 0u)
            co_store2h(a.out + aotx_attn_out_at(a, t, kh * G + j, e, D), aotx_f2h(v), aotx_f2h(v1));
    }
}

/* The largest of a value over the four lanes r, r + 16, r + 32 and r + 48. */
static __device__ __forceinline__ float aotx_attn_max4(float v)
{
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    const unsigned int w = __builtin_bit_cast(unsigned int, v);
    const u2 a = __builtin_bit_cast(u2, __builtin_amdgcn_permlane32_swap(w, w, false, false));
    const unsigned int a0 = a.x, a1 = a.y;
    const float m = fmaxf(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1));
    const unsigned int x = __builtin_bit_cast(unsigned int, m);
    const u2 b = __builtin_bit_cast(u2, __builtin_amdgcn_permlane16_swap(x, x, false, false));
    const unsigned int b0 = b.x, b1 = b.y;
    return fmaxf(__builtin_bit_cast(float, b0), __builtin_bit_cast(float, b1));
}

/* One query row by one wave, the values of the positions it attends and no others: the rows
 * that the products left NaN. There a position that a row does not attend has weight 0, and 0
 * times a value of Inf or NaN (another sequence's, a later token's, or one past the sequence's
 * last position) is NaN. Writes the dimensions [d0, d1), those that the wave wrote. Rare and not
 * fast: lanes over 64 positions for the scores, then over the dimensions for the values, 32-bit
 * weights. */
template <int D>
static __device__ void aotx_attend_row(const aotx_attn_args &a, unsigned int t, unsigned int kh, unsigned int h,
                                       unsigned int d0, unsigned int d1)
{
    constexpr int E = D / 64;                        /* dimensions per lane */
    const unsigned int lane = threadIdx.x & 63u;
    const unsigned int agent = a.agent[t], n = a.pos[t] + 1u;
    const aotx_kv_table *kv = &a.state->kv;
    const float scale = 1.4426950408889634f / sqrtf((float)D);
    const unsigned short *q = a.q + ((unsigned long long)t * a.heads + h) * D;
    float m = -INFINITY, l = 0.0f, o[E];
    bool missing = false;
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] = 0.0f;
    for (unsigned int p0 = 0u; p0 < n; p0 += 64u) {
        const unsigned int p = p0 + lane;
        const unsigned char *blk = p < n
            ? (const unsigned char *)aotx_kvl_block(a.shape, kv, agent, a.layer, p / 16u * 16u) : nullptr;
        missing = missing || __any(p < n && blk == nullptr);
        float s = -INFINITY;
        if (blk != nullptr) {
            const unsigned char *k = blk + (unsigned long long)(kh * AOTX_KVL_BLOCK + p % 16u) * D * 2u;
            s = 0.0f;
            for (int e = 0; e < D; e += 8) {
                const aotx_h8a kk = *(const aotx_h8a *)(k + 2 * e), qq = __builtin_bit_cast(aotx_h8a, co_load4(q + e));
#pragma unroll
                for (int i = 0; i < 8; ++i) s += (float)kk[i] * (float)qq[i];
            }
            s *= scale;
        }
        float mb = s;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) mb = fmaxf(mb, __shfl_xor(mb, d, 64));
        const float mnew = fmaxf(m, mb), msafe = mnew == -INFINITY ? 0.0f : mnew;
        const float shift = aotx_exp2(m - msafe), w = blk != nullptr ? aotx_exp2(s - msafe) : 0.0f;
        m = mnew;
        float mass = w;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) mass += __shfl_xor(mass, d, 64);
        l = l * shift + mass;
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] *= shift;
        const unsigned int here = n - p0 < 64u ? n - p0 : 64u;
        for (unsigned int j = 0; j < here; ++j) {
            const unsigned long long at = __shfl((unsigned long long)blk, (int)j, 64);
            const float wj = __shfl(w, (int)j, 64);
            if (at == 0ull) continue;
            const unsigned short *v = (const unsigned short *)at
                                    + (unsigned long long)((a.kv_heads + kh) * AOTX_KVL_BLOCK + (p0 + j) % 16u) * D;
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] += wj * aotx_h2f(v[(unsigned int)e * 64u + lane]);
        }
    }
    const float back = 1.0f / (l > 0.0f ? l : 1.0f);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const unsigned int at = (unsigned int)e * 64u + lane;
        if (at >= d0 && at < d1) a.out[aotx_attn_out_at(a, t, h, at, D)] = aotx_f2h(missing ? 0.0f : o[e] * back);
    }
}

/* The addresses of a sequence's blocks, 64 at a time, one per lane. */
struct aotx_attn_pages {
    unsigned long long pages;
    unsigned int base, agent, nblk;
    bool held;
};
static __device__ __forceinline__ void aotx_attn_look(const aotx_attn_args &a, aotx_attn_pages &w, unsigned int pair)
{
    const unsigned int b0 = 2u * pair;
    if (w.held && b0 + 1u - w.base < 64u) return;
    w.held = true;
    w.base = (unsigned int)__builtin_amdgcn_readfirstlane((int)b0);
    /* (the first pair's divisions would be taken out of the loop over the sequences and kept) */
    asm volatile("" : "+s"(w.base));
    const unsigned int bl = w.base + (threadIdx.x & 63u);
    w.pages = bl < w.nblk
        ? (unsigned long long)aotx_kvl_block(a.shape, &a.state->kv, w.agent, a.layer, bl * 16u) : 0ull;
}
/* The scalar resource of block b (zero-size: loads return zeros) and whether it is missing. */
static __device__ __forceinline__ __amdgpu_buffer_rsrc_t aotx_attn_block(const aotx_attn_args &a, const aotx_attn_pages &w,
                                                                         unsigned int b, bool &gone)
{
    const unsigned int at = (b - w.base) & 63u;
    const unsigned int hi = (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)(w.pages >> 32), (int)at);
    const unsigned int lo = (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)w.pages, (int)at);
    const unsigned long long pb = ((unsigned long long)hi << 32) | lo;
    gone = pb == 0ull && b < w.nblk;
    return __builtin_amdgcn_make_buffer_rsrc((void *)pb, (short)0, pb == 0ull ? 0 : (int)a.shape.block_bytes, 0x00020000);
}

/* A wave's NC tiles of 16 score columns and what it has added up for them. */
template <int D, int NC>
struct aotx_attn_cols {
    aotx_h8a qb[NC][D / 32];
    float mrun[NC];                                  /* column 16c + r */
    aotx_f4a o[NC][D / 16], mass[NC];                /* columns 16c + 4g .. + 3 */
    unsigned int plim[NC];                           /* column 16c + r: the positions it attends */
    unsigned int *miss;                              /* [NC] in LDS: bit r, column 16c + r met a missing page */
};
template <int D, int NC>
static __device__ __forceinline__ void aotx_attn_begin(aotx_attn_cols<D, NC> &s, unsigned int *miss)
{
    s.miss = miss;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        s.mrun[c] = -INFINITY;
        miss[c] = 0u;                                /* the wave's own */
        s.mass[c] = (aotx_f4a){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int cc = 0; cc < D / 16; ++cc) s.o[c][cc] = (aotx_f4a){0.0f, 0.0f, 0.0f, 0.0f};
    }
}

/* Scores of pair p's blocks to weights, mass and the shifted accumulators; then the values at
 * vw. EARLY: slices of the values read before the softmax, the others before the first products
 * (with a wave's own loads in flight they cost registers that spill). masked: some column does
 * not attend all of the pair's positions, or a block is missing. */
template <int D, int NC, int EARLY>
static __device__ __forceinline__ void aotx_attn_weigh(aotx_attn_cols<D, NC> &s, aotx_f4a (&scs)[NC][2], unsigned int p,
                                                       bool gone0, bool gone1, bool masked, const unsigned short *vw,
                                                       unsigned int lane)
{
    constexpr int NS = D / 16, VS = D + 8;
    const unsigned int g = lane >> 4;
    const float scale = 1.4426950408889634f / sqrtf((float)D);
    /* the transposing read of a block's slice (see aotx_attend_body) */
    const unsigned int vtr = (4u * g + (lane & 15u) / 4u) * VS + 4u * (lane & 3u);
    const _Float16 one = (_Float16)1.0f;
    const aotx_h8a ones = {one, one, one, one, one, one, one, one};
    aotx_h8a vv[NS];
    const auto values = [&](int cc) {
        const aotx_s4a v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) aotx_s4a *)(vw + vtr + 16u * (unsigned int)cc));
        const aotx_s4a v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) aotx_s4a *)(vw + 16u * VS + vtr + 16u * (unsigned int)cc));
        vv[cc] = __builtin_bit_cast(aotx_h8a, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
    };
#pragma unroll
    for (int cc = 0; cc < EARLY; ++cc) values(cc);
    if (EARLY != 0) __builtin_amdgcn_sched_barrier(0);
    aotx_h8a pa[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        aotx_f4a *const sc = scs[c];
        if (masked) {
            if (gone0 || gone1)
                s.miss[c] |= (unsigned int)__ballot((gone0 && 32u * p < s.plim[c]) || (gone1 && 32u * p + 16u < s.plim[c])) & 0xffffu;
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const unsigned int at = 32u * p + 16u * (unsigned int)e + 4u * g + (unsigned int)i;
                    if (at >= s.plim[c] || (e == 0 ? gone0 : gone1)) sc[e][i] = -INFINITY;
                }
        }
        float mb = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])),
                         fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
        mb = aotx_attn_max4(mb) * scale;
        const float mnew = fmaxf(s.mrun[c], mb);
        /* a column with no position yet: weights and shift of 0 from -inf */
        const float msafe = mnew == -INFINITY ? 0.0f : mnew;
        const bool moved = mnew != s.mrun[c];
        const float shift = moved ? aotx_exp2(s.mrun[c] - msafe) : 1.0f;
        s.mrun[c] = mnew;
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                pa[c][4 * e + i] = (_Float16)aotx_exp2(__builtin_fmaf(sc[e][i], scale, -msafe));
        if (__any(moved)) {
            float sh[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) sh[i] = __shfl(shift, (int)(4u * g) + i, 64);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s.mass[c][i] *= sh[i];
#pragma unroll
                for (int cc = 0; cc < NS; ++cc) s.o[c][cc][i] *= sh[i];
            }
        }
        s.mass[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[c], ones, s.mass[c], 0, 0, 0);
    }
#pragma unroll
    for (int cc = EARLY; cc < NS; ++cc) values(cc);
    if (EARLY != 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int cc = 0; cc < NS; ++cc)
#pragma unroll
        for (int c = 0; c < NC; ++c)
            s.o[c][cc] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[c], vv[cc], s.o[c][cc], 0, 0, 0);
}

/* One sequence's blocks, the pairs part, part + PARTS, ... of them, by a wave that waits for no
 * other: keys into registers and values through its own LDS slot vw. nmin: the positions that
 * every column attends. */
template <int D, int NC, int PARTS>
static __device__ __forceinline__ void aotx_attn_walk(const aotx_attn_args &a, aotx_attn_cols<D, NC> &s, unsigned int agent,
                                                      unsigned int n, unsigned int nmin, unsigned int kh,
                                                      unsigned int part, unsigned short *vw, unsigned int lane)
{
    constexpr int KK = D / 32, VP = D / 32, VS = D + 8;
    const unsigned int r = lane & 15u, g = lane >> 4;
    const unsigned int kbyte = ((kh * AOTX_KVL_BLOCK + r) * D + 8u * g) * 2u;          /* A operand */
    const unsigned int vbyte = ((a.kv_heads + kh) * AOTX_KVL_BLOCK * D + lane * 8u) * 2u;
    aotx_attn_pages w = {0ull, 0u, agent, (n + 15u) / 16u, false};
    const unsigned int pairs = (w.nblk + 1u) / 2u;
    aotx_u4a kr[2][KK], vr[2][VP];
    bool gone[2] = {false, false};
    const auto load = [&](unsigned int p) {
        aotx_attn_look(a, w, p);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const __amdgpu_buffer_rsrc_t rs = aotx_attn_block(a, w, 2u * p + (unsigned int)e, gone[e]);
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) kr[e][kk] = __builtin_amdgcn_raw_buffer_load_b128(rs, kbyte + kk * 64, 0, 0);
#pragma unroll
            for (int u = 0; u < VP; ++u) vr[e][u] = __builtin_amdgcn_raw_buffer_load_b128(rs, vbyte + u * 1024, 0, 0);
        }
    };
    if (part < pairs) load(part);
    for (unsigned int p = part; p < pairs; p += PARTS) {
        aotx_f4a scs[NC][2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int u = 0; u < VP; ++u) {
                const unsigned int piece = (unsigned int)u * 64u + lane;
                *(aotx_u4a *)(vw + ((unsigned int)e * 16u + piece / (D / 8)) * VS + (piece % (D / 8)) * 8u) = vr[e][u];
            }
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                scs[c][e] = (aotx_f4a){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int kk = 0; kk < KK; ++kk)
                    scs[c][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(aotx_h8a, kr[e][kk]),
                                                                       s.qb[c][kk], scs[c][e], 0, 0, 0);
            }
        const bool gone0 = gone[0], gone1 = gone[1];
        /* the registers are used: the next pair's loads run under the rest of this step
         * (unconditional: no copies where paths join) */
        __builtin_amdgcn_sched_barrier(0);
        load(p + PARTS);
        __builtin_amdgcn_sched_barrier(0);
        aotx_attn_weigh<D, NC, 0>(s, scs, p, gone0, gone1, 32u * p + 32u > nmin || gone0 || gone1, vw, lane);
    }
}

/* The PARTS waves of one group of columns add their parts, in part order, and write the rows:
 * column col is head kh G + col % G of token at(col), if that is below `tokens`. acc, pm, pl and
 * pmiss are the group's LDS: [PARTS][16 NC][D] floats, [PARTS][16 NC] maxima and masses,
 * [PARTS][NC] columns that met a missing page (acc may hold what the walks used: a barrier comes
 * before its first write). Two barriers, which every wave of the workgroup meets. */
template <int D, int G, int NC, int PARTS, class AT>
static __device__ __forceinline__ void aotx_attn_finish(const aotx_attn_args &a, aotx_attn_cols<D, NC> &s, float *acc,
                                                        float *pm, float *pl, unsigned int *pmiss, unsigned int part,
                                                        unsigned int kh, unsigned int tokens, unsigned int lane, AT at)
{
    constexpr int NS = D / 16;
    constexpr unsigned int COLS = 16u * NC, ACC = COLS * D;
    constexpr int NP = NS >= PARTS ? NS / PARTS : 1;       /* d slices that a part adds up */
    const unsigned int r = lane & 15u, g = lane >> 4;
    /* maxima by column, masses by accumulator row (each lane group of a column saw all of its
     * blocks) */
    unsigned int missed = 0u;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        missed |= s.miss[c];
        if (g == 0u) pm[part * COLS + 16u * (unsigned int)c + r] = s.mrun[c];
        if (r == 0u)
#pragma unroll
            for (int i = 0; i < 4; ++i) pl[part * COLS + 16u * (unsigned int)c + 4u * g + (unsigned int)i] = s.mass[c][i];
    }
    if (missed != 0u && lane == 0u) atomicAdd(&a.state->faults, 1u);
    __syncthreads();
    /* without branches: a part with no position has m = -inf, mass 0 and weight 2^-inf = 0 */
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const unsigned int col = 16u * (unsigned int)c + 4u * g + (unsigned int)i;
            float m[PARTS], top = -INFINITY, sum = 0.0f;
            unsigned int absent = 0u;
#pragma unroll
            for (unsigned int k = 0; k < (unsigned int)PARTS; ++k) {
                m[k] = pm[k * COLS + col];
                top = fmaxf(top, m[k]);
                absent |= pmiss[k * NC + (unsigned int)c] >> (col & 15u);
            }
            top = top == -INFINITY ? 0.0f : top;
#pragma unroll
            for (unsigned int k = 0; k < (unsigned int)PARTS; ++k) sum += pl[k * COLS + col] * aotx_exp2(m[k] - top);
            const float whole = 1.0f / (sum > 0.0f ? sum : 1.0f);
            const float f = (absent & 1u) != 0u ? 0.0f : aotx_exp2(pm[part * COLS + col] - top) * whole;
#pragma unroll
            for (int cc = 0; cc < NS; ++cc)
                acc[part * ACC + ((c * NS + cc) * 4 + i) * 64 + lane] = s.o[c][cc][i] * f;
        }
    __syncthreads();
    /* part k adds the slices [k NP, (k + 1) NP) of all parts in part order */
    if (part * (unsigned int)NP >= (unsigned int)NS) return;
    unsigned int odd = 0u;                           /* bit 4c + i: NaN in this lane's column */
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const unsigned int col = 16u * (unsigned int)c + 4u * g + (unsigned int)i;
            const unsigned int t = at(col);
            float v[NP];
            bool bad = false;
#pragma unroll
            for (int x = 0; x < NP; ++x) {
                const unsigned int cc = part * (unsigned int)NP + (unsigned int)x;
                v[x] = 0.0f;
#pragma unroll
                for (unsigned int k = 0; k < (unsigned int)PARTS; ++k)
                    v[x] += acc[k * ACC + (((unsigned int)c * NS + cc) * 4u + (unsigned int)i) * 64u + lane];
                bad = bad || v[x] != v[x];
            }
            if (t < tokens) {
#pragma unroll
                for (int x = 0; x < NP; ++x) {
                    const unsigned int cc = part * (unsigned int)NP + (unsigned int)x;
                    a.out[aotx_attn_out_at(a, t, kh * G + col % (unsigned int)G, 16u * cc + r, D)] = aotx_f2h(v[x]);
                }
                odd |= bad ? 1u << (4 * c + i) : 0u;
            }
        }
    if (!__any(odd != 0u)) return;
    const unsigned int d0 = part * (unsigned int)NP * 16u;
#pragma unroll 1
    for (unsigned int col = 0; col < COLS; ++col) {
        /* column 16c + 4g + i: bit 4c + i of the 16 lanes of group g */
        const bool mine = (odd >> (4u * (col / 16u) + col % 4u)) & 1u && g == col / 4u % 4u;
        if (__any(mine)) {
            const unsigned int t = (unsigned int)__builtin_amdgcn_readfirstlane((int)at(col));
            aotx_attend_row<D>(a, t, kh, kh * G + col % (unsigned int)G, d0, d0 + (unsigned int)NP * 16u);
        }
    }
}

/* Batches with prompt pieces: a workgroup takes 16 NC H score columns of a KV head, the G
 * query heads of 16 NC H / G consecutive tokens. Its 4 H waves are H halves of the columns (NC
 * tiles of 16 each) times 4 parts of the positions: part k takes every fourth pair of
 * 16-position blocks, the parts are added at the end, in part order. Per pair of blocks and
 * tile:
 *   - scores: keys as the A operand, 16 positions by 16 columns per MFMA as in the decode body;
 *   - the largest score over the 32 positions by four lane groups (row swaps, no LDS); the
 *     weights 2^(score - max) round to fp16 in the A layout of v_mfma_f32_16x16x32_f16, block
 *     0's positions 4g .. 4g + 3 and then block 1's, and the values come from LDS in that order
 *     (two transposing reads, shared by the tiles);
 *   - the mass is the product of the same fp16 weights with ones, on the matrix core, where it
 *     has the rows of the accumulators.
 * With one half (H = 1) a wave loads its pairs by itself (aotx_attn_walk). With two (H = 2) and
 * one sequence the halves of a part load a block of the pair each into LDS for both,
 * double-buffered, one barrier per pair: half the reads from the L2s, which bound many columns
 * otherwise. The next pair is on its way while one is computed. Columns of several sequences:
 * each half goes over the blocks of one sequence after the other by itself, and a column that
 * does not take part keeps its state (but for values that are not finite: aotx_attend_row).
 * Bound by the softmax's vector work and the matrix work of a step, about 1600 cycles a wave.
 * Against a wave per 16 / G queries with one block per pass of softmax, at 32 / 8 heads x 128:
 * 512 tokens after 2000 cached ones 74.3 -> 42.8 us (H = 2; 55 with H = 1), a 512-token prompt
 * 21.7 -> 15.6, 256 tokens 14.6 -> 9.6, 128 tokens 10.8 -> 6.9, 200 tokens after 7800
 * 210 -> 78. Four tiles per wave at one wave per SIMD took 64 us in the first case.
 *
 * Tokens that are the only one of their run of a slot (decode rows beside a prompt piece, among
 * the batch's first AOTX_RUN_SINGLES) are not columns of their place: walked there, their
 * sequences would follow one another in the few workgroups of that range (63 rows at 2048
 * positions beside a 449-token prompt 479 us, 366 by a wave per piece). Every workgroup takes its
 * share of them at the end, a (token, KV head) at a time with the positions in 4 H parts: 108 us,
 * where the keys and values alone (530 MB) take 88 at 6 TB/s. A launch without such tokens pays
 * for the search 0.3 to 0.6 us (a 256-token prompt 10.0 -> 10.5, 512 tokens 16.5 -> 17.0). */
#define AOTX_RUN_SINGLES 512u
template <int D, int G, int NC, int H>
static __device__ __forceinline__ void aotx_attend_runs(const aotx_attn_args &a, unsigned int bx)
{
    constexpr int KK = D / 32;                      /* score MFMA steps */
    constexpr int VP = D / 32;                      /* 16-byte pieces per lane and block */
    constexpr int VS = D + 8;                       /* LDS row stride (halves) */
    constexpr unsigned int TW = 16u * NC * H / G;   /* tokens */
    constexpr unsigned int PARTS = 4u, WAVES = PARTS * H;
    constexpr unsigned int COLS = 16u * NC;         /* columns of a half */
    static_assert(TW >= 1u && TW <= 64u && (TW & (TW - 1u)) == 0u && COLS % G == 0u,
                  "a lane per token, whole tokens per half");
    /* the waves' value slots; H = 2 with one sequence: [buffer][part][keys, values] of a pair;
     * after the loop the waves' accumulators */
    constexpr unsigned int ROWS = 32u * VS * 2u, ACC = COLS * D * 4u;
    constexpr unsigned int STAGE = H == 1 ? PARTS * ROWS : 2u * PARTS * 2u * ROWS;
    __shared__ __attribute__((aligned(16))) unsigned char lds[STAGE > H * PARTS * ACC ? STAGE : H * PARTS * ACC];
    __shared__ float pm[H * PARTS * COLS], pl[H * PARTS * COLS];
    __shared__ unsigned int pmiss[H * PARTS * NC];
    constexpr unsigned int WORDS = AOTX_RUN_SINGLES / 64u;
    __shared__ unsigned long long same[WORDS];       /* bit t: token t + 1 is of the same slot */
    __shared__ unsigned int lag[64], lps[64];        /* the tokens' slots and positions: the walks leave no
                                                        registers for them (every wave writes the same) */

    const unsigned int lane = threadIdx.x & 63u;
    /* a scalar, so that the wave's blocks, loads and tests are scalar too */
    const unsigned int wave = (unsigned int)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned int part = wave % PARTS, half = H == 1 ? 0u : wave / PARTS;
    const unsigned int r = lane & 15u, g = lane >> 4;
    const unsigned int counted = aotx_attn_scalar(a.m_dev != nullptr ? a.m_dev : a.pos);
    const unsigned int kh = bx % a.kv_heads;
    const unsigned int t0 = (bx / a.kv_heads) * TW;             /* the workgroup's first token */
    /* lane i holds the slot and position of token t0 + i and its neighbours' slots; all words are
     * read before the row count is known (below the launch's capacity every one exists), in one
     * round trip with those of the batch's first tokens */
    const auto slot_of = [&](unsigned int t) { return a.agent[t < a.tokens ? t : a.tokens - 1u]; };
    const unsigned int tl = t0 + (lane < TW ? lane : 0u);
    const unsigned int ag = slot_of(tl), ag0 = slot_of(tl != 0u ? tl - 1u : 0u), ag1 = slot_of(tl + 1u);
    const unsigned int ps = a.pos[tl < a.tokens ? tl : a.tokens - 1u];
    constexpr unsigned int ROUNDS = WORDS / WAVES;
    unsigned int b0[ROUNDS], b1[ROUNDS];
#pragma unroll
    for (unsigned int i = 0u; i < ROUNDS; ++i) {
        b0[i] = slot_of(i * 64u * WAVES + threadIdx.x);
        b1[i] = slot_of(i * 64u * WAVES + threadIdx.x + 1u);
    }
    __builtin_amdgcn_sched_barrier(0);
    unsigned int tokens = a.m_dev != nullptr ? counted : a.tokens;
    if (tokens > a.tokens) tokens = a.tokens;
    if (t0 >= tokens) return;
    const bool live = lane < TW && tl < tokens;
    const bool apart = tl < AOTX_RUN_SINGLES && (tl == 0u || ag0 != ag) && (tl + 1u == tokens || ag1 != ag);
    const unsigned long long batch = __ballot(live), all = __ballot(live && !apart);
#pragma unroll
    for (unsigned int i = 0u; i < ROUNDS; ++i) {
        const unsigned long long e = __ballot(i * 64u * WAVES + threadIdx.x + 1u < tokens && b0[i] == b1[i]);
        if (lane == 0u) same[i * WAVES + wave] = e;
    }
    lag[lane] = ag;
    lps[lane] = ps;

    if (all != 0ull) {
        const unsigned int c0 = half * COLS;                    /* this half's first column */
        aotx_attn_cols<D, NC> s;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const unsigned int col = c0 + 16u * (unsigned int)c + r;
            const unsigned int tc = col / (unsigned int)G, hh = col % (unsigned int)G;
            /* a column past the batch reads its last token's query (its results are not written) */
            const unsigned int tq = t0 + tc < tokens ? t0 + tc : tokens - 1u;
            const unsigned short *q = a.q + ((unsigned long long)tq * a.heads + kh * G + hh) * D + 8u * g;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) s.qb[c][kk] = __builtin_bit_cast(aotx_h8a, co_load4(q + 32 * kk));
        }
        aotx_attn_begin(s, pmiss + (half * PARTS + part) * NC);
        /* the tokens `group` of slot `agent`, in any order of positions: the positions attended by
         * any of them (n) and by every column (nmin, 0 if a column is another's) */
        unsigned int agent = 0u, n = 0u, nmin = 0u;
        const auto sequence = [&](unsigned long long group, unsigned long long columns, unsigned int ps) {
            const bool in = (group >> lane) & 1ull;
            n = in ? ps + 1u : 0u;
            nmin = in ? ps + 1u : 0xFFFFFFFFu;
#pragma unroll
            for (int d = (int)TW / 2; d >= 1; d >>= 1) {              /* over the tokens' lanes */
                const unsigned int on = (unsigned int)__shfl_xor((int)n, d, 64), om = (unsigned int)__shfl_xor((int)nmin, d, 64);
                n = on > n ? on : n;
                nmin = om < nmin ? om : nmin;
            }
            n = (unsigned int)__builtin_amdgcn_readfirstlane((int)n);
            nmin = group == columns ? (unsigned int)__builtin_amdgcn_readfirstlane((int)nmin) : 0u;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const unsigned int tc = (c0 + 16u * (unsigned int)c + r) / (unsigned int)G;
                const unsigned int pt = (unsigned int)__shfl((int)ps, (int)tc, 64) + 1u;
                s.plim[c] = (group >> tc) & 1ull ? pt : 0u;
            }
        };
        agent = (unsigned int)__builtin_amdgcn_readlane((int)ag, __builtin_ctzll(all));
        const unsigned long long first = __ballot(ag == agent) & all;
        if (H == 1 || first != all) {
            /* the tokens of this half's columns */
            const unsigned long long here = COLS / G >= 64u ? ~0ull : ((1ull << (COLS / G)) - 1ull) << (c0 / G);
            unsigned long long left = all & here;
            while (left != 0ull) {
                unsigned int li = lane;
                asm volatile("" : "+v"(li));         /* read from LDS, not kept from where it was stored */
                const unsigned int al = lag[li];
                agent = (unsigned int)__builtin_amdgcn_readlane((int)al, __builtin_ctzll(left));
                const unsigned long long group = __ballot(al == agent) & left;
                left &= ~group;
                sequence(group, batch & here, lps[li]);
                aotx_attn_walk<D, NC, (int)PARTS>(a, s, agent, n, nmin, kh, part, (unsigned short *)(lds + wave * ROWS), lane);
            }
        } else if constexpr (H == 2) {
            /* a wave brings block `half` of its part's pair; every wave meets every barrier */
            sequence(first, batch, ps);
            aotx_attn_pages w = {0ull, 0u, agent, (n + 15u) / 16u, false};
            const unsigned int pairs = (w.nblk + 1u) / 2u;
            const unsigned int kbase = (kh * AOTX_KVL_BLOCK * D + lane * 8u) * 2u;             /* whole rows */
            const unsigned int vbase = ((a.kv_heads + kh) * AOTX_KVL_BLOCK * D + lane * 8u) * 2u;
            const auto slot = [&](unsigned int buf, unsigned int what) {
                return (unsigned short *)(lds + ((buf * PARTS + part) * 2u + what) * ROWS);
            };
            aotx_u4a kl[VP], vr[VP];
            bool gone[2] = {false, false};
            const auto load = [&](unsigned int p) {
                aotx_attn_look(a, w, p);
                bool g0, g1;
                const __amdgpu_buffer_rsrc_t r0 = aotx_attn_block(a, w, 2u * p, g0), r1 = aotx_attn_block(a, w, 2u * p + 1u, g1);
                gone[0] = g0;
                gone[1] = g1;
                const __amdgpu_buffer_rsrc_t rs = half == 0u ? r0 : r1;
#pragma unroll
                for (int u = 0; u < VP; ++u) kl[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, kbase + u * 1024, 0, 0);
#pragma unroll
                for (int u = 0; u < VP; ++u) vr[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, vbase + u * 1024, 0, 0);
            };
            const auto store = [&](unsigned int buf) {
#pragma unroll
                for (int u = 0; u < VP; ++u) {
                    const unsigned int piece = (unsigned int)u * 64u + lane;
                    const unsigned int at = (half * 16u + piece / (D / 8)) * VS + (piece % (D / 8)) * 8u;
                    *(aotx_u4a *)(slot(buf, 0u) + at) = kl[u];
                    *(aotx_u4a *)(slot(buf, 1u) + at) = vr[u];
                }
            };
            const bool mine = first >> (c0 / G) << (64u - (COLS + G - 1u) / G) != 0ull;   /* any column here */
            load(part);
            store(0u);
            __syncthreads();
            const unsigned int steps = (pairs + PARTS - 1u) / PARTS;
            for (unsigned int st = 0; st < steps; ++st) {
                const unsigned int p = part + st * PARTS;
                const bool gone0 = gone[0], gone1 = gone[1];
                load(p + PARTS);
                __builtin_amdgcn_sched_barrier(0);
                if (p < pairs && mine) {
                    const unsigned short *kw = slot(st & 1u, 0u);
                    aotx_f4a scs[NC][2];
                    aotx_h8a k8[2][KK];
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int kk = 0; kk < KK; ++kk)
                            k8[e][kk] = *(const aotx_h8a *)(kw + ((unsigned int)e * 16u + r) * VS + 32u * (unsigned int)kk + 8u * g);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int c = 0; c < NC; ++c) scs[c][e] = (aotx_f4a){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
                        for (int e = 0; e < 2; ++e)
#pragma unroll
                            for (int c = 0; c < NC; ++c)
                                scs[c][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k8[e][kk], s.qb[c][kk], scs[c][e], 0, 0, 0);
                    aotx_attn_weigh<D, NC, D / 32>(s, scs, p, gone0, gone1, 32u * p + 32u > nmin || gone0 || gone1, slot(st & 1u, 1u), lane);
                }
                store((st + 1u) & 1u);
                __syncthreads();
            }
        }
        const auto token = [&](unsigned int col) {
            const unsigned int tc = (c0 + col) / (unsigned int)G;
            return (all >> tc) & 1ull ? t0 + tc : 0xFFFFFFFFu;
        };
        aotx_attn_finish<D, G, NC, (int)PARTS>(a, s, (float *)lds + half * PARTS * (ACC / 4u), pm + half * PARTS * COLS,
                                               pl + half * PARTS * COLS, pmiss + half * PARTS * NC, part, kh, tokens, lane, token);
    } else {
        __syncthreads();                             /* `same` is there */
    }

    /* a lane number of its own, so that no address made from it is kept in registers over the
     * walks above, which have none to spare */
    unsigned int ln = threadIdx.x & 63u;
    asm volatile("" : "+v"(ln));
    /* the tokens apart, lane i those of 64i .. 64i + 63 */
    const unsigned int wi = ln < WORDS ? lane : 0u, past = 64u * wi < tokens ? tokens - 64u * wi : 0u;
    const unsigned long long e = same[wi], e0 = wi != 0u ? same[wi - 1u] >> 63 : 0ull;
    const unsigned long long alone = ln < WORDS ? ~e & ~(e << 1 | e0) & (past >= 64u ? ~0ull : (1ull << past) - 1ull) : 0ull;
    if (!__any(alone != 0ull)) return;
    /* (token, KV head) number u to workgroup u mod the workgroups with tokens */
    const unsigned int groups = (tokens + TW - 1u) / TW * a.kv_heads;
    const unsigned int mine = (unsigned int)__builtin_popcountll(alone);
    unsigned int upto = mine;                        /* those of this lane's word and the ones before */
#pragma unroll
    for (unsigned int d = 1u; d < WORDS; d <<= 1) {
        const unsigned int o = (unsigned int)__shfl_up((int)upto, d, 64);
        if (ln >= d) upto += o;
    }
    const unsigned int units = (unsigned int)__builtin_amdgcn_readlane((int)upto, (int)WORDS - 1) * a.kv_heads;
    for (unsigned int u = bx; u < units; u += groups) {
        /* the k-th of them: in the first word that reaches past k */
        unsigned int k = u / a.kv_heads;
        const unsigned int word = (unsigned int)__builtin_ctzll(__ballot(ln < WORDS && upto > k));
        k -= (unsigned int)__builtin_amdgcn_readlane((int)(upto - mine), (int)word);
        unsigned long long bits = (unsigned long long)(unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)(alone >> 32), (int)word) << 32
                                | (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)alone, (int)word);
        for (; k != 0u; --k) bits &= bits - 1ull;
        const unsigned int t = word * 64u + (unsigned int)__builtin_ctzll(bits);
        const unsigned int uh = u % a.kv_heads;
        const unsigned int agent = (unsigned int)__builtin_amdgcn_readfirstlane((int)a.agent[t]);
        const unsigned int n = (unsigned int)__builtin_amdgcn_readfirstlane((int)a.pos[t]) + 1u;
        /* G columns; the others repeat them and are not written */
        aotx_attn_cols<D, 1> s;
        const unsigned short *q = a.q + ((unsigned long long)t * a.heads + uh * G + (ln & 15u) % (unsigned int)G) * D + 8u * (ln >> 4);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) s.qb[0][kk] = __builtin_bit_cast(aotx_h8a, co_load4(q + 32 * kk));
        s.plim[0] = n;
        __syncthreads();                             /* the accumulators before are read */
        aotx_attn_begin(s, pmiss + wave);
        aotx_attn_walk<D, 1, (int)WAVES>(a, s, agent, n, n, uh, wave, (unsigned short *)(lds + wave * ROWS), ln);
        aotx_attn_finish<D, G, 1, (int)WAVES>(a, s, (float *)lds, pm, pl, pmiss, wave, uh, tokens, ln,
                                              [&](unsigned int col) { return col < (unsigned int)G ? t : 0xFFFFFFFFu; });
    }
}

#undef MMA_WINDOW
#undef MMA_LOAD
#undef MMA_COMPUTE

#endif
