/* Sampler and Philox stream.
 *
 * Reference: aotx_model_pick (cuda/model/sample.cu:456-765) and the Philox4x32-10 stream
 * (cuda/rng/rng.cuh:29-94). Several workgroups of 256 threads take one row of logits. The steps,
 * their order and every float expression follow the reference so that the same logits
 * give the same token: the largest logit (ties to the lowest thread = token mod 256, then
 * the lowest token), a temperature of zero returns it; otherwise the row sum of
 * exp(v - top), a two-pass 256-bucket search over the 42 below the top for a cut that
 * keeps at most 256 candidates, the candidates sorted largest first, then top-k, min-p,
 * top-p on the T = 1 probabilities, the temperature, and the inverse CDF at the Philox
 * uniform of (seed, slot, lane 0, draw position). Every sum runs in the reference's
 * order: thread t adds tokens t, t + 256, ..., then thread 0 adds the 256 partials in
 * thread order. One deliberate difference: where the reference leaves a choice to timing
 * (which candidates fill the 256 places when more pass the cut; the order of equal values
 * after its bitonic network), this kernel takes the lowest token ids, so the result is a
 * function of the logits alone.
 *
 * The penalties, voice bias and thinking masks of aotx_pick_value (sample.cu:277-319)
 * read the decode runtime's sequence table, which is outside this path; with a null
 * per-row `how` (the aotx_model_sample case) the reference leaves the logit unchanged
 * and so does this kernel.
 */
#include "aotx_internal.h"

#include <hip/hip_runtime.h>

#define PICK_THREADS 256u
#define PICK_BUCKETS 256u
#define PICK_CHUNKS 64u   /* workgroups per row of the largest-logit search */
#define PICK_SUMS 16u     /* of the 256 partial sums of a row, those of one workgroup */
#define PICK_STEPS 64u    /* tokens of each between two barriers */
#define PICK_AHEAD 8u     /* such blocks loaded together */
#define PICK_SLICES 16u   /* workgroups per row of the candidates */

#pragma clang fp contract(off)

struct aotx_u32x4 {
    unsigned int x, y, z, w;
};

static __device__ __forceinline__ aotx_u32x4 aotx_philox_dev(unsigned int c0, unsigned int c1,
                                                             unsigned int c2, unsigned int c3,
                                                             unsigned int k0, unsigned int k1)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r != 0) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        unsigned int lo0 = 0xD2511F53u * c0;
        unsigned int hi0 = __umulhi(0xD2511F53u, c0);
        unsigned int lo1 = 0xCD9E8D57u * c2;
        unsigned int hi1 = __umulhi(0xCD9E8D57u, c2);
        unsigned int n0 = hi1 ^ c1 ^ k0;
        unsigned int n2 = hi0 ^ c3 ^ k1;
        c0 = n0;
        c1 = lo1;
        c2 = n2;
        c3 = lo0;
    }
    aotx_u32x4 out = {c0, c1, c2, c3};
    return out;
}

__global__ void aotx_philox_kernel(const unsigned int *ctr, const unsigned int *key,
                                   unsigned int n, unsigned int *out)
{
    unsigned int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    aotx_u32x4 w = aotx_philox_dev(ctr[4 * i], ctr[4 * i + 1], ctr[4 * i + 2], ctr[4 * i + 3],
                                   key[2 * i], key[2 * i + 1]);
    out[4 * i] = w.x;
    out[4 * i + 1] = w.y;
    out[4 * i + 2] = w.z;
    out[4 * i + 3] = w.w;
}

struct aotx_pick_args {
    const float *logits;          /* [rows][ld] */
    unsigned int ld;
    unsigned int vocab;
    const unsigned int *rows_dev; /* device row count, or null */
    unsigned int rows;
    const unsigned int *agent;    /* [rows] */
    const aotx_model_how *how;    /* per-row settings, or null */
    unsigned int top_k;
    float top_p;
    float temperature;
    unsigned long long seed;
    int *token;
    unsigned int *draw;
    aotx_state *state;
    const aotx_model_run *run;    /* when set, every per-call value comes from here */
    unsigned int *best;           /* [rows][PICK_CHUNKS][2]: each chunk's (value bits, token) */
    unsigned int *hist;           /* [rows][PICK_BUCKETS] first-pass counts */
    float *sums;                  /* [rows][PICK_THREADS] partial sums of exp(v - top) */
    float *total;                 /* [rows] their sum */
    unsigned int *cand;           /* [rows][PICK_SLICES][AOTX_MODEL_PICK_MAX][2] (value bits, token) */
    unsigned int *found;          /* [rows][PICK_SLICES] candidates of each slice */
    unsigned int *seen;           /* [rows] slices done */
};

/* (v, i) ranks ahead of (bv, bi) in the reference's largest-logit search: a larger value;
 * among equal values the lower token mod 256 (the reference's lower thread), then the
 * lower token (that thread's earlier stride). NaN ranks nowhere. */
static __device__ __forceinline__ bool aotx_pick_ahead(float v, unsigned int i, float bv,
                                                       unsigned int bi)
{
    return v > bv || (v == bv && ((i & 255u) < (bi & 255u) || ((i & 255u) == (bi & 255u) && i < bi)));
}

/* The row's largest logit from the slices of aotx_argmax_kernel (reference order): one
 * slice per lane, merged across the wave; every lane of a full wave gets the winner. */
static_assert(PICK_CHUNKS <= 64u, "one slice per lane");
static __device__ __forceinline__ void aotx_pick_top(const aotx_pick_args &a, unsigned int r,
                                                     float &best, unsigned int &at)
{
    const unsigned int *cand = a.best + (unsigned long long)r * PICK_CHUNKS * 2u;
    const unsigned int lane = threadIdx.x & 63u;
    best = -INFINITY;
    at = 0u;
    if (lane < PICK_CHUNKS) {
        best = __uint_as_float(cand[2u * lane]);
        at = cand[2u * lane + 1u];
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(best, off, 64);
        const unsigned int oi = __shfl_xor(at, off, 64);
        if (aotx_pick_ahead(ov, oi, best, at)) {
            best = ov;
            at = oi;
        }
    }
}

/* The row's sampling settings (a per-row `how` overrides the call's). */
static __device__ __forceinline__ float aotx_pick_warmth(const aotx_pick_args &a, unsigned int r)
{
    const aotx_model_how *how = a.run ? a.run->how : a.how;
    if (how != nullptr) return how[r].temperature;
    return a.run ? a.run->temperature : a.temperature;
}

/* The largest logit of each of PICK_CHUNKS slices of a row (grid: chunks x rows). The
 * winner over the slices under aotx_pick_ahead is the reference's (thread-strided scan,
 * then the thread-order merge), so the slices can be searched in parallel. A slice whose
 * values are all -inf (or NaN) leaves (-inf, 0), as a reference thread does. */
__global__ __launch_bounds__(PICK_THREADS) void aotx_argmax_kernel(aotx_pick_args a)
{
    __shared__ float wv[PICK_THREADS / 64];
    __shared__ unsigned int wi[PICK_THREADS / 64];
    const unsigned int tid = threadIdx.x;
    const unsigned int r = blockIdx.y;
    const unsigned int c = blockIdx.x;
    const aotx_model_run *run = a.run;
    unsigned int rows = run ? run->rows : (a.rows_dev ? *a.rows_dev : a.rows);
    int *token_out = run ? run->token : a.token;
    if (r >= rows || token_out == nullptr) return;
    if (run && run->select != AOTX_MODEL_ROWS_LAST) return;
    /* the row's histogram and counts start at zero for the launches that follow (their place
     * in the sampler's buffer depends on the call's row count, so an earlier call with
     * another count may have left other words there) */
    if (c == 0u) {
        for (unsigned int i = tid; i < PICK_BUCKETS; i += PICK_THREADS)
            a.hist[(unsigned long long)r * PICK_BUCKETS + i] = 0u;
        if (tid == 0u) a.seen[r] = 0u;
    }
    const float *row = a.logits + (unsigned long long)r * a.ld;
    const unsigned int span = (a.vocab + PICK_CHUNKS - 1u) / PICK_CHUNKS;
    const unsigned int lo = c * span;
    const unsigned int hi = lo + span < a.vocab ? lo + span : a.vocab;
    float best = -INFINITY;
    unsigned int at = 0u;
#pragma unroll 8
    for (unsigned int i = lo + tid; i < hi; i += PICK_THREADS) {
        float one = row[i];
        if (aotx_pick_ahead(one, i, best, at)) {
            best = one;
            at = i;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        float ov = __shfl_xor(best, off, 64);
        unsigned int oi = __shfl_xor(at, off, 64);
        if (aotx_pick_ahead(ov, oi, best, at)) {
            best = ov;
            at = oi;
        }
    }
    if ((tid & 63u) == 0u) {
        wv[tid >> 6] = best;
        wi[tid >> 6] = at;
    }
    __syncthreads();
    if (tid == 0u) {
        for (unsigned int w = 1u; w < PICK_THREADS / 64u; ++w) {
            if (aotx_pick_ahead(wv[w], wi[w], best, at)) {
                best = wv[w];
                at = wi[w];
            }
        }
        unsigned int *out = a.best + ((unsigned long long)r * PICK_CHUNKS + c) * 2u;
        out[0] = __float_as_uint(best);
        out[1] = at;
    }
}

/* The ordered sums of exp(v - top) of a sampled row and the first pass of the cut search.
 * The reference's thread t adds tokens t, t + 256, ... one after another, so a workgroup
 * takes PICK_SUMS of the 256 sums over the whole row (grid: 256 / PICK_SUMS x rows): its
 * threads make the exponentials of PICK_STEPS tokens of each sum in LDS, and one lane per sum
 * adds them in order while the others make the next block's. Every thread also counts its
 * values in the 256-bucket histogram over [top - 42, top] (counts: any order; a copy per lane
 * quarter spreads the bulk of the logits, which falls into few buckets). Rows at temperature
 * 0 do nothing. Bound by the exponentials and the LDS counts of a workgroup. A launch that
 * stored every exponential (12.4 us at 32 rows of 128256) and one workgroup per row that added
 * them and walked the row twice more (86.7 us) became this one (15.7) and the next (24). */
__global__ __launch_bounds__(PICK_THREADS) void aotx_pick_exp_kernel(aotx_pick_args a)
{
    __shared__ unsigned int bucket[4][PICK_BUCKETS + 1u];
    __shared__ float block[2][PICK_STEPS][PICK_SUMS + 1u];
    const unsigned int tid = threadIdx.x;
    const unsigned int r = blockIdx.y;
    const aotx_model_run *run = a.run;
    unsigned int rows = run ? run->rows : (a.rows_dev ? *a.rows_dev : a.rows);
    int *token_out = run ? run->token : a.token;
    if (r >= rows || token_out == nullptr) return;
    if (run && run->select != AOTX_MODEL_ROWS_LAST) return;
    if (aotx_pick_warmth(a, r) <= 0.0f) return;
    for (unsigned int i = tid; i < 4u * (PICK_BUCKETS + 1u); i += PICK_THREADS) (&bucket[0][0])[i] = 0u;
    constexpr unsigned int PER = PICK_STEPS * PICK_SUMS / PICK_THREADS;    /* values per thread and block */
    constexpr unsigned int ROWS = PICK_THREADS / PICK_SUMS;                /* steps of one load */
    const float *row = a.logits + (unsigned long long)r * a.ld;
    const unsigned int c = tid % PICK_SUMS, s0 = tid / PICK_SUMS;
    const unsigned int col = blockIdx.x * PICK_SUMS + c;
    const unsigned int steps = (a.vocab + PICK_THREADS - 1u) / PICK_THREADS;
    const float lo = -AOTX_MODEL_PICK_SPAN, hi = 0.0f, band = hi - lo;
    unsigned int *mine = bucket[(tid >> 4) & 3u];
    float sum = 0.0f, top = 0.0f;
    for (unsigned int first = 0u; first < steps; first += PICK_AHEAD * PICK_STEPS) {
        float v[PICK_AHEAD][PER];
#pragma unroll
        for (unsigned int k = 0u; k < PICK_AHEAD; ++k)
#pragma unroll
            for (unsigned int e = 0u; e < PER; ++e) {
                const unsigned int i = (first + k * PICK_STEPS + e * ROWS + s0) * PICK_THREADS + col;
                v[k][e] = row[i < a.vocab ? i : 0u];
            }
        if (first == 0u) {           /* the largest logit while the first values are on their way */
            unsigned int at;
            aotx_pick_top(a, r, top, at);
            __syncthreads();
        }
#pragma unroll
        for (unsigned int k = 0u; k < PICK_AHEAD; ++k) {
            const unsigned int base = first + k * PICK_STEPS;
            if (base < steps) {
    #pragma unroll
                for (unsigned int e = 0u; e < PER; ++e) {
                    const unsigned int step = e * ROWS + s0;
                    const bool in = (base + step) * PICK_THREADS + col < a.vocab;
                    const float scaled = v[k][e] - top;
                    if (in) block[k & 1u][step][c] = expf(scaled);
                    if (in && scaled >= lo && scaled <= hi) {
                        unsigned int b = (unsigned int)((scaled - lo) * (float)PICK_BUCKETS / band);
                        if (b >= PICK_BUCKETS) b = PICK_BUCKETS - 1u;
                        atomicAdd(&mine[b], 1u);
                    }
                }
                __syncthreads();
                /* the block's values of a sum in token order; the block before it was read before
                 * this barrier, so the next one may overwrite that */
                if (tid < PICK_SUMS) {
                    const unsigned int left = a.vocab > base * PICK_THREADS + col
                                            ? (a.vocab - base * PICK_THREADS - col + PICK_THREADS - 1u) / PICK_THREADS : 0u;
                    if (left >= PICK_STEPS) {
                        float x[PICK_STEPS];
    #pragma unroll
                        for (unsigned int i = 0u; i < PICK_STEPS; ++i) x[i] = block[k & 1u][i][c];
    #pragma unroll
                        for (unsigned int i = 0u; i < PICK_STEPS; ++i) sum += x[i];
                    } else {
                        for (unsigned int i = 0u; i < left; ++i) sum += block[k & 1u][i][c];
                    }
                }
            }
        }
        __syncthreads();
    }
    if (tid < PICK_SUMS) a.sums[(unsigned long long)r * PICK_THREADS + col] = sum;
    __syncthreads();
    unsigned int *h = a.hist + (unsigned long long)r * PICK_BUCKETS;
    for (unsigned int i = tid; i < PICK_BUCKETS; i += PICK_THREADS) {
        const unsigned int n = bucket[0][i] + bucket[1][i] + bucket[2][i] + bucket[3][i];
        if (n != 0u) atomicAdd(h + i, n);
    }
}

/* The cut over a band's counts, by the first 64 threads of a workgroup: the reference goes
 * down from the highest bucket and stops at the one with which more than AOTX_MODEL_PICK_MAX
 * values would be held; the cut is that bucket's upper end, and when nothing is held yet the
 * band narrows to the bucket. Lane l holds buckets 4l .. 4l + 3. */
static __device__ __forceinline__ void aotx_pick_cut(const unsigned int *bucket, float lo, float band, float &cut,
                                                     unsigned int &more, float &lo2)
{
    static_assert(PICK_BUCKETS == 256u, "four buckets per lane");
    const unsigned int lane = threadIdx.x;
    unsigned int n[4], above = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        n[i] = bucket[4u * lane + (unsigned int)i];
        above += n[i];
    }
    /* the counts of this lane's buckets and all higher ones */
#pragma unroll
    for (unsigned int d = 1u; d < 64u; d <<= 1) {
        const unsigned int o = __shfl_down(above, d, 64);
        if (lane + d < 64u) above += o;
    }
    /* this lane's highest bucket with which more than the most are held, if any */
    unsigned int held = above - n[0] - n[1] - n[2] - n[3], b = 0u, before = 0u;
#pragma unroll
    for (int i = 3; i >= 0; --i) {
        if (b == 0u && held + n[i] > AOTX_MODEL_PICK_MAX) {
            b = 4u * lane + (unsigned int)i + 1u;
            before = held;
        }
        held += n[i];
    }
    const unsigned long long any = __ballot(b != 0u);
    if (any == 0ull) {
        cut = lo;
        more = 0u;
        return;
    }
    const int from = 63 - __builtin_clzll(any);
    b = (unsigned int)__shfl((int)b, from, 64);
    before = (unsigned int)__shfl((int)before, from, 64);
    cut = lo + band * (float)b / (float)PICK_BUCKETS;
    more = before == 0u ? 1u : 0u;
    lo2 = lo + band * (float)(b - 1u) / (float)PICK_BUCKETS;
}

/* A word another workgroup (on another XCD, past its L2) wrote or will read. */
static __device__ __forceinline__ void aotx_pick_put(unsigned int *p, unsigned int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
static __device__ __forceinline__ unsigned int aotx_pick_get(const unsigned int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* PICK_SLICES workgroups per row: each finds the cut from the first pass's counts and puts
 * the candidates of its slice in the row's list; the last one done picks. (The sort orders
 * candidates by (value, id), a total order, so their places in the list do not matter.) When
 * one bucket holds too many (logits equal to within 0.16, the reference's second pass) or the
 * candidates exceed their places, the last one goes through the whole row instead (32 rows of
 * 128256 logits of N(0, 0.01) 148 us in all against 50 of N(0, 2), equal ones 380). Bound by
 * its chain of memory round trips (counts, candidates, arrivals, lists) and the ordered sums. */
__global__ __launch_bounds__(PICK_THREADS) void aotx_pick_kernel(aotx_pick_args a)
{
    __shared__ unsigned int mark[PICK_THREADS];
    __shared__ unsigned int bucket[PICK_BUCKETS];
    __shared__ __attribute__((aligned(16))) float value[AOTX_MODEL_PICK_MAX];
    __shared__ __attribute__((aligned(16))) unsigned int index[AOTX_MODEL_PICK_MAX];
    __shared__ __attribute__((aligned(16))) float t_min[AOTX_MODEL_PICK_MAX], t_mass[AOTX_MODEL_PICK_MAX], t_heat[AOTX_MODEL_PICK_MAX];
    __shared__ float s_top, s_sum, s_cut, s_lo, s_hi;
    __shared__ unsigned int s_more, s_position, s_slot, s_last;

    const unsigned int tid = threadIdx.x;
    const unsigned int r = blockIdx.y;
    /* The slice with the sum is mostly the last one done and takes the row's tail. Workgroups go
     * round the 8 XCDs and then their 32 CUs: it has another place in each row, so that the tails
     * of up to 256 rows lie on CUs of their own. */
    const unsigned int slice = (blockIdx.x + r + r / PICK_SLICES) % PICK_SLICES;
    const aotx_model_run *run = a.run;
    unsigned int rows = run ? run->rows : (a.rows_dev ? *a.rows_dev : a.rows);
    int *token_out = run ? run->token : a.token;
    unsigned int *draw_out = run ? run->draw : a.draw;
    if (r >= rows || token_out == nullptr) return;
    if (run && run->select != AOTX_MODEL_ROWS_LAST) return;
    const float *row = a.logits + (unsigned long long)r * a.ld;
    const unsigned int vocab = a.vocab;
    unsigned int agent = run ? run->agent[r] : a.agent[r];
    if (agent >= AOTX_SLOTS) agent = 0u;

    const aotx_model_how *how = run ? run->how : a.how;
    unsigned int want_k = run ? run->top_k : a.top_k;
    float want_p = run ? run->top_p : a.top_p;
    float warmth = run ? run->temperature : a.temperature;
    unsigned long long stream = run ? run->seed : a.seed;
    float min_p = 0.0f;
    if (how != nullptr) {
        want_k = how[r].top_k;
        want_p = how[r].top_p;
        warmth = how[r].temperature;
        stream = how[r].seed;
        min_p = how[r].min_p;
    }

    if (warmth <= 0.0f) {
        /* the largest logit's place, from the slices of aotx_argmax_kernel */
        if (slice != 0u || tid >= 64u) return;
        float best;
        unsigned int at;
        aotx_pick_top(a, r, best, at);
        if (tid == 0u) {
            const unsigned int drawn = atomicAdd(&a.state->draw[agent], 1u);
            if (draw_out != nullptr) draw_out[r] = drawn;
            token_out[r] = (int)at;
        }
        return;
    }
    /* the largest logit, and the cut; the row's sum in thread order by a lane of the last
     * slice, published like the candidates */
    bucket[tid] = a.hist[(unsigned long long)r * PICK_BUCKETS + tid];
    if (slice == PICK_SLICES - 1u) t_mass[tid] = a.sums[(unsigned long long)r * PICK_THREADS + tid];
    if (tid == 0u) s_slot = 0u;
    __syncthreads();
    if (tid < 64u) {
        float best;
        unsigned int at;
        aotx_pick_top(a, r, best, at);
        float cut = 0.0f, lo2 = 0.0f;
        unsigned int more = 0u;
        aotx_pick_cut(bucket, -AOTX_MODEL_PICK_SPAN, AOTX_MODEL_PICK_SPAN, cut, more, lo2);
        if (tid == 0u) {
            s_top = best;
            s_cut = cut;
            s_more = more;
            s_lo = lo2;
            s_hi = cut;
        }
    }
    __syncthreads();
    const float top = s_top;
    if (slice == PICK_SLICES - 1u && tid == PICK_THREADS - 1u) {
        float sum = 0.0f;
#pragma unroll 1
        for (unsigned int h = 0u; h < PICK_THREADS; h += 64u) {
            float x[64];
#pragma unroll
            for (int i = 0; i < 64; ++i) x[i] = t_mass[h + (unsigned int)i];
#pragma unroll
            for (int i = 0; i < 64; ++i) sum += x[i];
        }
        aotx_pick_put((unsigned int *)a.total + r, __float_as_uint(sum));
    }
    unsigned int *cand = a.cand + (unsigned long long)r * PICK_SLICES * AOTX_MODEL_PICK_MAX * 2u;
    unsigned int *founds = a.found + r * PICK_SLICES;
    const bool aligned = ((unsigned long long)row & 15ull) == 0ull;
    if (s_more == 0u) {
        /* this slice's candidates, into LDS and then into its list */
        const float cut = s_cut;
        const unsigned int span = ((vocab + PICK_SLICES - 1u) / PICK_SLICES + 3u) & ~3u;
        const unsigned int b0 = slice * span < vocab ? slice * span : vocab;
        const unsigned int b1 = b0 + span < vocab ? b0 + span : vocab;
        const unsigned int body = aligned ? b0 + (b1 - b0) / 4u * 4u : b0;
        const auto take = [&](float v, unsigned int i) {
            const float scaled = v - top;
            if (scaled >= cut) {
                const unsigned int slot = atomicAdd(&s_slot, 1u);
                if (slot < AOTX_MODEL_PICK_MAX) {
                    value[slot] = scaled;
                    index[slot] = i;
                }
            }
        };
#pragma unroll 8
        for (unsigned int i = b0 + 4u * tid; i < body; i += 4u * PICK_THREADS) {
            const float4 f = *(const float4 *)(row + i);
            take(f.x, i);
            take(f.y, i + 1u);
            take(f.z, i + 2u);
            take(f.w, i + 3u);
        }
#pragma unroll 8
        for (unsigned int i = body + tid; i < b1; i += PICK_THREADS) take(row[i], i);
        __syncthreads();
        const unsigned int n = s_slot < AOTX_MODEL_PICK_MAX ? s_slot : AOTX_MODEL_PICK_MAX;
        unsigned int *list = cand + slice * AOTX_MODEL_PICK_MAX * 2u;
        for (unsigned int i = tid; i < n; i += PICK_THREADS) {
            aotx_pick_put(list + 2u * i, __float_as_uint(value[i]));
            aotx_pick_put(list + 2u * i + 1u, index[i]);
        }
        if (tid == 0u) aotx_pick_put(founds + slice, s_slot);
    }
    /* what the slice published is out before it counts as done */
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0u) s_last = atomicAdd(a.seen + r, 1u) == PICK_SLICES - 1u ? 1u : 0u;
    __syncthreads();
    if (s_last == 0u) return;
    /* the slices' counts; the row's draw and sum with them */
    if (tid < PICK_SLICES) mark[tid] = s_more == 0u ? aotx_pick_get(founds + tid) : 0u;
    if (tid == 64u) {
        s_position = atomicAdd(&a.state->draw[agent], 1u);
        if (draw_out != nullptr) draw_out[r] = s_position;
    }
    if (tid == 128u) {
        s_sum = __uint_as_float(aotx_pick_get((const unsigned int *)a.total + r));
        s_slot = 0u;
    }
    __syncthreads();
    unsigned int found = 0u, in = 0u, mine_at = 0u;      /* thread t holds candidate t of the slices' in order */
#pragma unroll
    for (unsigned int i = 0u; i < PICK_SLICES; ++i) {
        const unsigned int n = mark[i];
        if (tid >= found) {
            in = i;
            mine_at = tid - found;
        }
        found += n;
    }
    /* every value of the row, by this workgroup alone: 16-byte loads where the row allows, 16 of
     * them on their way (with single words a pass over 128256 took 64 us instead of 16) */
    const auto each = [&](auto f) {
        const unsigned int body = aligned ? vocab / 4u * 4u : 0u;
#pragma unroll 16
        for (unsigned int i = 4u * tid; i < body; i += 4u * PICK_THREADS) {
            const float4 v = *(const float4 *)(row + i);
            f(v.x, i);
            f(v.y, i + 1u);
            f(v.z, i + 2u);
            f(v.w, i + 3u);
        }
#pragma unroll 16
        for (unsigned int i = body + tid; i < vocab; i += PICK_THREADS) f(row[i], i);
    };
    if (s_more != 0u) {
        /* the second pass of the cut search, over the band of one bucket */
        const float lo = s_lo, hi = s_hi, band = hi - lo;
        for (unsigned int i = tid; i < PICK_BUCKETS; i += PICK_THREADS) bucket[i] = 0u;
        __syncthreads();
        each([&](float v, unsigned int) {
            const float scaled = v - top;
            if (scaled >= lo && scaled <= hi) {
                unsigned int b = (unsigned int)((scaled - lo) * (float)PICK_BUCKETS / band);
                if (b >= PICK_BUCKETS) b = PICK_BUCKETS - 1u;
                atomicAdd(&bucket[b], 1u);
            }
        });
        __syncthreads();
        if (tid < 64u) {
            float cut = 0.0f, lo2 = 0.0f;
            unsigned int more = 0u;
            aotx_pick_cut(bucket, lo, band, cut, more, lo2);
            if (tid == 0u) s_cut = cut;
        }
    }
    __syncthreads();
    const float cut = s_cut;
    if (s_more == 0u && found <= AOTX_MODEL_PICK_MAX) {
        if (tid < found) {
            const unsigned int *one = cand + (in * AOTX_MODEL_PICK_MAX + mine_at) * 2u;
            value[tid] = __uint_as_float(aotx_pick_get(one));
            index[tid] = aotx_pick_get(one + 1u);
        }
        if (tid == 0u) s_slot = found;
    } else {
        /* the whole row: every candidate takes the next place while places remain */
        each([&](float v, unsigned int i) {
            const float scaled = v - top;
            if (scaled >= cut) {
                const unsigned int slot = atomicAdd(&s_slot, 1u);
                if (slot < AOTX_MODEL_PICK_MAX) {
                    value[slot] = scaled;
                    index[slot] = i;
                }
            }
        });
    }
    __syncthreads();
    unsigned int count = s_slot;
    if (count > AOTX_MODEL_PICK_MAX) {
        /* more than the places (logits equal to within the finest band, where the reference
         * keeps whichever arrive first): the lowest token ids are kept. Each thread takes a
         * contiguous run of tokens and a prefix over the threads places them in order. */
        const unsigned int per = (vocab + PICK_THREADS - 1u) / PICK_THREADS;
        const unsigned int first = tid * per;
        const unsigned int after = first + per < vocab ? first + per : vocab;
        unsigned int run_mine = 0u;
#pragma unroll 16
        for (unsigned int i = first; i < after; ++i) {
            if (row[i] - top >= cut) run_mine += 1u;
        }
        unsigned int slot = run_mine;                /* those of this thread and the ones before */
#pragma unroll
        for (unsigned int d = 1u; d < 64u; d <<= 1) {
            const unsigned int o = __shfl_up(slot, d, 64);
            if ((tid & 63u) >= d) slot += o;
        }
        __syncthreads();
        if ((tid & 63u) == 63u) mark[tid >> 6] = slot;
        __syncthreads();
#pragma unroll
        for (unsigned int w = 0u; w + 1u < PICK_THREADS / 64u; ++w) slot += w < tid >> 6 ? mark[w] : 0u;
        slot -= run_mine;
        /* (a run past the last place has nothing to put there) */
#pragma unroll 16
        for (unsigned int i = slot < AOTX_MODEL_PICK_MAX ? first : after; i < after; ++i) {
            float scaled = row[i] - top;
            if (scaled >= cut) {
                if (slot < AOTX_MODEL_PICK_MAX) {
                    value[slot] = scaled;
                    index[slot] = i;
                }
                slot += 1u;
            }
        }
        count = AOTX_MODEL_PICK_MAX;
    }
    /* largest first, ties to the lower id: a thread per candidate counts those ahead of it (a
     * total order, so the counts are the places). The terms of each candidate are the
     * expressions of the reference's serial loops; the places past the count hold nothing. */
    static_assert(PICK_THREADS == AOTX_MODEL_PICK_MAX, "a thread per candidate");
    if (tid >= count) {
        value[tid] = -INFINITY;
        index[tid] = 0xFFFFFFFFu;
    }
    __syncthreads();
    const float mine = value[tid];
    const unsigned int my_id = index[tid];
    unsigned int place = tid;
    if (tid < count) {
        place = 0u;
#pragma unroll 4
        for (unsigned int j = 0u; j < count; j += 4u) {
            const float4 v = *(const float4 *)(value + j);
            const uint4 o = *(const uint4 *)(index + j);
            place += v.x > mine || (v.x == mine && o.x < my_id) ? 1u : 0u;
            place += v.y > mine || (v.y == mine && o.y < my_id) ? 1u : 0u;
            place += v.z > mine || (v.z == mine && o.z < my_id) ? 1u : 0u;
            place += v.w > mine || (v.w == mine && o.w < my_id) ? 1u : 0u;
        }
        if (place == 0u) s_lo = mine;
    }
    __syncthreads();
    const float v0 = s_lo;
    const float heat = warmth;
    index[place] = my_id;
    t_min[place] = expf(mine - v0);
    t_mass[place] = expf(mine) / s_sum;
    t_heat[place] = expf((mine - v0) / heat);
    __syncthreads();
    /* the running sums of the masses and of the tempered terms in candidate order, by a lane
     * of two waves each: what the serial walks hold after each candidate */
    if (tid == 0u || tid == 64u) {
        float *t = tid == 0u ? t_mass : t_heat;
        float sum = 0.0f;
#pragma unroll 1
        for (unsigned int h = 0u; h < count; h += 64u) {
            float x[64];
#pragma unroll
            for (int i = 0; i < 64; ++i) x[i] = t[h + (unsigned int)i];
#pragma unroll
            for (int i = 0; i < 64; ++i) {
                sum += x[i];
                x[i] = sum;
            }
#pragma unroll
            for (int i = 0; i < 64; ++i) t[h + (unsigned int)i] = x[i];
        }
    }
    __syncthreads();
    /* the walks: the first candidate at which each stops, over lane-parallel tests (thread i
     * tests candidate i) */
    const auto first = [&](bool stop, unsigned int none) {
        const unsigned long long at = __ballot(stop);
        if ((tid & 63u) == 0u) mark[tid >> 6] = at != 0ull ? tid + (unsigned int)__builtin_ctzll(at) : 0xFFFFFFFFu;
        __syncthreads();
        unsigned int f = mark[0];
#pragma unroll
        for (unsigned int w = 1u; w < PICK_THREADS / 64u; ++w) f = mark[w] < f ? mark[w] : f;
        __syncthreads();
        return f < none ? f : none;
    };
    unsigned int keep = (want_k == 0u || want_k > count) ? count : want_k;
    if (min_p > 0.0f && min_p <= 1.0f)         /* up to the first below it, the largest always */
        keep = first(tid >= 1u && tid < keep && t_min[tid] < min_p, keep > 1u ? keep : 1u);
    const float limit = (want_p <= 0.0f || want_p > 1.0f) ? 1.0f : want_p;
    /* up to and with the first at which the mass reaches the limit */
    const unsigned int reached = first(tid < keep && t_mass[tid] >= limit, keep);
    const unsigned int taken = reached < keep ? reached + 1u : keep;
    const float heat_total = taken != 0u ? t_heat[taken - 1u] : 0.0f;
    const aotx_u32x4 word = aotx_philox_dev(s_position, 0u, 0u, agent, (unsigned int)stream,
                                            (unsigned int)(stream >> 32));
    const float pick = (float)(word.x >> 8) * (1.0f / 16777216.0f) * heat_total;
    const unsigned int chosen = first(tid < taken && t_heat[tid] >= pick, taken != 0u ? taken - 1u : 0u);
    if (tid == 0u) token_out[r] = (int)index[chosen];
}

size_t aotx_pick_scratch(unsigned int rows, unsigned int vocab)
{
    (void)vocab;
    return (size_t)rows * (PICK_CHUNKS * 2u + PICK_BUCKETS + PICK_THREADS + PICK_SLICES * (AOTX_MODEL_PICK_MAX * 2u + 1u)
                           + 2u) * sizeof(unsigned int);
}

void aotx_launch_pick(const float *logits, unsigned int ld, unsigned int vocab,
                      const unsigned int *rows_dev, unsigned int rows,
                      const unsigned int *agent, const aotx_model_how *how,
                      unsigned int top_k, float top_p, float temperature,
                      unsigned long long seed, int *token, unsigned int *draw,
                      const aotx_model_run *run, unsigned int *best, hipStream_t s)
{
    aotx_pick_args a;
    a.logits = logits;
    a.ld = ld;
    a.vocab = vocab;
    a.rows_dev = rows_dev;
    a.rows = rows;
    a.agent = agent;
    a.how = how;
    a.top_k = top_k;
    a.top_p = top_p;
    a.temperature = temperature;
    a.seed = seed;
    a.token = token;
    a.draw = draw;
    a.state = aotx_state_device();
    a.run = run;
    a.best = best;
    a.hist = best + (size_t)rows * PICK_CHUNKS * 2u;
    a.sums = (float *)(a.hist + (size_t)rows * PICK_BUCKETS);
    a.cand = (unsigned int *)(a.sums + (size_t)rows * PICK_THREADS);
    a.found = a.cand + (size_t)rows * PICK_SLICES * AOTX_MODEL_PICK_MAX * 2u;
    a.seen = a.found + (size_t)rows * PICK_SLICES;
    a.total = (float *)(a.seen + rows);
    hipLaunchKernelGGL(aotx_argmax_kernel, dim3(PICK_CHUNKS, rows), dim3(PICK_THREADS), 0, s, a);
    AOTX_LAUNCH_CHECK();
    hipLaunchKernelGGL(aotx_pick_exp_kernel, dim3(PICK_THREADS / PICK_SUMS, rows), dim3(PICK_THREADS), 0, s, a);
    AOTX_LAUNCH_CHECK();
    hipLaunchKernelGGL(aotx_pick_kernel, dim3(PICK_SLICES, rows), dim3(PICK_THREADS), 0, s, a);
    AOTX_LAUNCH_CHECK();
}

extern "C" int aotx_pick(const float *logits, unsigned int rows, unsigned int vocab,
                         const unsigned int *agent, const aotx_model_how *how,
                         unsigned int top_k, float top_p, float temperature,
                         unsigned long long seed, int *token, unsigned int *draw, void *stream)
{
    if (logits == nullptr || agent == nullptr || token == nullptr || rows == 0u || vocab == 0u)
        return 1;
    unsigned int *best = (unsigned int *)aotx_scratch(AOTX_SCRATCH_PICK, aotx_pick_scratch(rows, vocab));
    aotx_launch_pick(logits, vocab, vocab, nullptr, rows, agent, how, top_k, top_p,
                     temperature, seed, token, draw, nullptr, best, aotx_stream(stream));
    return 0;
}

extern "C" int aotx_philox(const unsigned int *ctr, const unsigned int *key, unsigned int n,
                           unsigned int *out, void *stream)
{
    if (ctr == nullptr || key == nullptr || out == nullptr) return 1;
    if (n == 0u) return 0;
    hipLaunchKernelGGL(aotx_philox_kernel, dim3((n + 255u) / 256u), dim3(256), 0,
                       aotx_stream(stream), ctr, key, n, out);
    AOTX_LAUNCH_CHECK();
    return 0;
}
