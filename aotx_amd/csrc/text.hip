/* Byte-level BPE tokenizer and detokenizer (the reference's cuda/text/).
 *
 * The vocabulary is built on the host from the model file's arrays and copied to the
 * device once: a token table by string (FNV-1a, open addressing), a pair table by (left,
 * right) that holds the merge rank and the merged token (so the merge step never joins
 * strings), the token of each single byte, and the control bits.
 *
 * Encoding is five launches, six with special tokens; each works on many places of a text
 * at a time:
 *   - clean: a workgroup per text, four bytes per thread, replaces what is not UTF-8;
 *   - special tokens (when the vocabulary has any): a wave per text lists their places;
 *   - pre-tokens: one thread per byte. The family's split pattern is a state machine that
 *     takes the first alternative matching at a position (cuda/text/pretok.cu:1-45); a
 *     thread at a place where every match must begin anew (is_sync) runs it up to the next
 *     such place, so a text is cut in parallel;
 *   - merge: a wave per 64 bytes, one lane per pre-token that starts there: its symbols and
 *     the rank of each symbol's pair in LDS, each round the pair of the lowest rank (the
 *     leftmost of equal ranks), and only the two pairs next to it looked up again;
 *   - pre-tokens of more than TX_SHORT bytes: a workgroup of 64 lanes each, the same rounds
 *     with a wave minimum;
 *   - gather: a workgroup per text, a prefix sum over the tokens of each place.
 * Detokenizing is one wave per text: token lengths, a wave prefix sum, then the bytes.
 */
#include "aotx_internal.h"
#include "unicode_classes.h"
#include "../../include/aotx_text.h"
#include "../../include/aotx_modelfile.h"

#include <stdlib.h>
#include <string.h>

#include <string>
#include <unordered_map>
#include <vector>

/* ---- character classes and UTF-8 -------------------------------------------------------- */

static __device__ int uc_in(const unsigned int *r, unsigned int n, unsigned int cp)
{
    unsigned int lo = 0u, hi = n;            /* ranges [2i, 2i + 1], sorted */
    while (lo < hi) {
        const unsigned int mid = (lo + hi) >> 1;
        if (cp < r[2u * mid]) hi = mid;
        else if (cp > r[2u * mid + 1u]) lo = mid + 1u;
        else return 1;
    }
    return 0;
}
static __device__ __forceinline__ int is_letter(unsigned int p)
{
    if (p < 0x80u) return (p >= 'A' && p <= 'Z') || (p >= 'a' && p <= 'z');
    return uc_in(aotx_uc_letter, AOTX_UC_LETTER_RANGES, p);
}
static __device__ __forceinline__ int is_number(unsigned int p)
{
    if (p < 0x80u) return p >= '0' && p <= '9';
    return uc_in(aotx_uc_number, AOTX_UC_NUMBER_RANGES, p);
}
static __device__ __forceinline__ int is_space(unsigned int p)
{
    if (p < 0x80u) return p == 0x20u || (p >= 0x09u && p <= 0x0Du);
    return uc_in(aotx_uc_space, AOTX_UC_SPACE_RANGES, p);
}
static __device__ __forceinline__ int is_mark(unsigned int p)
{
    return p >= 0x80u && uc_in(aotx_uc_mark, AOTX_UC_MARK_RANGES, p);
}

/* The code point at `at` and its byte count; a byte run that is not UTF-8 reads as
 * U+FFFD of one byte. */
static __device__ unsigned int utf8_at(const unsigned char *b, unsigned int end, unsigned int at,
                                       unsigned int *point)
{
    const unsigned int c = b[at];
    unsigned int need, cp, min;
    if (c < 0x80u) { *point = c; return 1u; }
    if ((c & 0xE0u) == 0xC0u) { need = 1u; cp = c & 0x1Fu; min = 0x80u; }
    else if ((c & 0xF0u) == 0xE0u) { need = 2u; cp = c & 0x0Fu; min = 0x800u; }
    else if ((c & 0xF8u) == 0xF0u) { need = 3u; cp = c & 0x07u; min = 0x10000u; }
    else { *point = 0xFFFDu; return 1u; }
    if (at + need >= end) { *point = 0xFFFDu; return 1u; }     /* cut off by the end */
    for (unsigned int i = 1u; i <= need; ++i) {
        const unsigned int d = b[at + i];
        if ((d & 0xC0u) != 0x80u) { *point = 0xFFFDu; return 1u; }
        cp = (cp << 6) | (d & 0x3Fu);
    }
    if (cp < min || cp > 0x10FFFFu || (cp >= 0xD800u && cp <= 0xDFFFu)) { *point = 0xFFFDu; return 1u; }
    *point = cp;
    return need + 1u;
}

/* The byte-level alphabet: each byte stands as one code point that is printable UTF-8
 * (the GPT-2 byte map; cuda/text/text.cuh:256-290). */
static __host__ __device__ __forceinline__ unsigned int byte_point(unsigned int b)
{
    if ((b >= 0x21u && b <= 0x7Eu) || (b >= 0xA1u && b <= 0xACu) || (b >= 0xAEu && b <= 0xFFu)) return b;
    if (b <= 0x20u) return 0x100u + b;
    if (b <= 0xA0u) return 0x100u + 33u + (b - 0x7Fu);
    return 0x100u + 67u;                                   /* 0xAD */
}
static __device__ __forceinline__ unsigned int point_byte(unsigned int p)
{
    if ((p >= 0x21u && p <= 0x7Eu) || (p >= 0xA1u && p <= 0xACu) || (p >= 0xAEu && p <= 0xFFu)) return p;
    if (p < 0x100u || p > 0x143u) return 0x100u;
    const unsigned int a = p - 0x100u;
    if (a <= 0x20u) return a;
    if (a <= 66u) return 0x7Fu + (a - 33u);
    return 0xADu;
}
static __host__ __device__ __forceinline__ unsigned int utf8_put(unsigned int p, unsigned char *o)
{
    if (p < 0x80u) { o[0] = (unsigned char)p; return 1u; }
    if (p < 0x800u) { o[0] = (unsigned char)(0xC0u | (p >> 6)); o[1] = (unsigned char)(0x80u | (p & 0x3Fu)); return 2u; }
    if (p < 0x10000u) {
        o[0] = (unsigned char)(0xE0u | (p >> 12)); o[1] = (unsigned char)(0x80u | ((p >> 6) & 0x3Fu));
        o[2] = (unsigned char)(0x80u | (p & 0x3Fu)); return 3u;
    }
    o[0] = (unsigned char)(0xF0u | (p >> 18)); o[1] = (unsigned char)(0x80u | ((p >> 12) & 0x3Fu));
    o[2] = (unsigned char)(0x80u | ((p >> 6) & 0x3Fu)); o[3] = (unsigned char)(0x80u | (p & 0x3Fu));
    return 4u;
}

static __host__ __device__ __forceinline__ unsigned long long fnv_step(unsigned long long h, unsigned int byte)
{
    return (h ^ (unsigned long long)byte) * 1099511628211ull;
}
#define FNV_BASIS 14695981039346656037ull
static __host__ __device__ __forceinline__ unsigned long long pair_mix(unsigned long long k)
{
    k ^= k >> 33; k *= 0xFF51AFD7ED558CCDull; k ^= k >> 33; k *= 0xC4CEB9FE1A85EC53ull; k ^= k >> 33;
    return k;
}

/* ---- the vocabulary ------------------------------------------------------------------- */

struct aotx_text_vocab {
    const unsigned char *token_bytes;
    const unsigned long long *token_at;
    unsigned int tokens;
    unsigned int slots;                 /* power of two */
    const unsigned int *slot;           /* token of each slot, or AOTX_TEXT_NONE */
    unsigned int pairs;                 /* power of two */
    const uint4 *pair;                  /* right, left (all ones: empty), rank, merged token */
    const unsigned int *control;        /* one bit per token */
    const unsigned int *special;        /* tokens of the control and user types */
    unsigned int specials;
    unsigned long long first[4];        /* bits of the first bytes of the specials */
    unsigned int pattern;
    unsigned int whole;
    unsigned int byte_token[256];
};

static aotx_text_vocab g_vocab;
static int g_ready = 0;
static unsigned int g_report[4];

/* The merge rank (and merged token) of two symbol pairs, AOTX_TEXT_NONE for no merge. Both
 * probes are in flight together: a lookup is one 16-byte load unless its place was taken. */
static __device__ __forceinline__ void find_pairs(const aotx_text_vocab &v, unsigned int l0, unsigned int r0,
                                                  unsigned int l1, unsigned int r1, unsigned int rank[2],
                                                  unsigned int res[2])
{
    const unsigned int mask = v.pairs - 1u;
    unsigned int at0 = (unsigned int)pair_mix(((unsigned long long)l0 << 32) | r0) & mask;
    unsigned int at1 = (unsigned int)pair_mix(((unsigned long long)l1 << 32) | r1) & mask;
    bool on0 = l0 != AOTX_TEXT_NONE && r0 != AOTX_TEXT_NONE, on1 = l1 != AOTX_TEXT_NONE && r1 != AOTX_TEXT_NONE;
    rank[0] = rank[1] = AOTX_TEXT_NONE;
    res[0] = res[1] = 0u;
    for (unsigned int i = 0u; i <= mask && (on0 || on1); ++i) {
        const uint4 e0 = v.pair[at0], e1 = v.pair[at1];
        if (on0 && e0.x == r0 && e0.y == l0) { rank[0] = e0.z; res[0] = e0.w; on0 = false; }
        if (on1 && e1.x == r1 && e1.y == l1) { rank[1] = e1.z; res[1] = e1.w; on1 = false; }
        on0 = on0 && !(e0.x == AOTX_TEXT_NONE && e0.y == AOTX_TEXT_NONE);
        on1 = on1 && !(e1.x == AOTX_TEXT_NONE && e1.y == AOTX_TEXT_NONE);
        at0 = (at0 + 1u) & mask;
        at1 = (at1 + 1u) & mask;
    }
}
static __device__ __forceinline__ unsigned int find_pair(const aotx_text_vocab &v, unsigned int l,
                                                         unsigned int r, unsigned int *result)
{
    if (l == AOTX_TEXT_NONE || r == AOTX_TEXT_NONE) return AOTX_TEXT_NONE;
    const unsigned int mask = v.pairs - 1u;
    unsigned int at = (unsigned int)pair_mix(((unsigned long long)l << 32) | r) & mask;
    for (unsigned int i = 0; i <= mask; ++i) {
        const uint4 e = v.pair[at];
        if (e.x == r && e.y == l) { *result = e.w; return e.z; }
        if (e.x == AOTX_TEXT_NONE && e.y == AOTX_TEXT_NONE) return AOTX_TEXT_NONE;
        at = (at + 1u) & mask;
    }
    return AOTX_TEXT_NONE;
}

/* The token whose string is the byte-level form of bytes [0, n), or AOTX_TEXT_NONE. */
static __device__ unsigned int find_bytes(const aotx_text_vocab &v, const unsigned char *b, unsigned int n)
{
    unsigned long long h = FNV_BASIS;
    unsigned int len = 0u;
    for (unsigned int i = 0; i < n; ++i) {
        unsigned char u[4];
        const unsigned int k = utf8_put(byte_point(b[i]), u);
        for (unsigned int j = 0; j < k; ++j) h = fnv_step(h, u[j]);
        len += k;
    }
    const unsigned int mask = v.slots - 1u;
    unsigned int at = (unsigned int)h & mask;
    for (unsigned int step = 0; step <= mask; ++step) {
        const unsigned int t = v.slot[at];
        if (t == AOTX_TEXT_NONE) return AOTX_TEXT_NONE;
        const unsigned long long f = v.token_at[t];
        if (v.token_at[t + 1u] - f == len) {
            const unsigned char *s = v.token_bytes + f;
            unsigned int pos = 0u;
            bool same = true;
            for (unsigned int i = 0; i < n && same; ++i) {
                unsigned char u[4];
                const unsigned int k = utf8_put(byte_point(b[i]), u);
                for (unsigned int j = 0; j < k; ++j) same = same && s[pos + j] == u[j];
                pos += k;
            }
            if (same) return t;
        }
        at = (at + 1u) & mask;
    }
    return AOTX_TEXT_NONE;
}

/* ---- pre-tokens (cuda/text/pretok.cu:1-45 states the alternatives) -------------------- */

/* 's 't 're 've 'm 'll 'd at `at`, small letters (or any case); bytes of the match or 0 */
static __device__ unsigned int contraction(const unsigned char *b, unsigned int at, unsigned int end,
                                           int any_case)
{
    if (b[at] != '\'' || at + 1u >= end) return 0u;
    unsigned int c1 = b[at + 1u], c2 = at + 2u < end ? b[at + 2u] : 0u;
    if (any_case) {
        if (c1 >= 'A' && c1 <= 'Z') c1 += 32u;
        if (c2 >= 'A' && c2 <= 'Z') c2 += 32u;
    }
    if (c1 == 's' || c1 == 't' || c1 == 'm' || c1 == 'd') return 2u;
    if ((c1 == 'r' && c2 == 'e') || (c1 == 'v' && c2 == 'e') || (c1 == 'l' && c2 == 'l')) return 3u;
    return 0u;
}
static __device__ unsigned int letter_run(const unsigned char *b, unsigned int end, unsigned int at, int marks)
{
    while (at < end) {
        unsigned int p;
        const unsigned int k = utf8_at(b, end, at, &p);
        if (!(is_letter(p) || (marks && is_mark(p)))) break;
        at += k;
    }
    return at;
}
static __device__ unsigned int number_run(const unsigned char *b, unsigned int end, unsigned int at,
                                          unsigned int most)
{
    for (unsigned int n = 0u; at < end && (most == 0u || n < most); ++n) {
        unsigned int p;
        const unsigned int k = utf8_at(b, end, at, &p);
        if (!is_number(p)) break;
        at += k;
    }
    return at;
}
/* characters that are not space, letter or number (nor marks, when marks are letters) */
static __device__ unsigned int other_run(const unsigned char *b, unsigned int end, unsigned int at, int marks)
{
    while (at < end) {
        unsigned int p;
        const unsigned int k = utf8_at(b, end, at, &p);
        if (is_space(p) || is_letter(p) || is_number(p) || (marks && is_mark(p))) break;
        at += k;
    }
    return at;
}
/* the space alternatives at a space character: with the newline rule, \s*[\r\n]+ first;
 * then \s+(?!\S) (the run gives back its last character when a non-space follows); \s+ */
static __device__ unsigned int spaces(const unsigned char *b, unsigned int end, unsigned int at,
                                      unsigned int span, int newline_rule)
{
    unsigned int stop = at, last = at, newline = 0u;
    bool found = false;
    while (stop < end) {
        unsigned int p;
        const unsigned int k = utf8_at(b, end, stop, &p);
        if (!is_space(p)) break;
        if (p == '\r' || p == '\n') { newline = stop; found = true; }
        last = stop;
        stop += k;
    }
    if (stop == at) return span;
    if (newline_rule && found) return newline + 1u - at;
    if (stop == end) return stop - at;
    if (last > at) return last - at;
    return stop - at;
}
static __device__ unsigned int match(unsigned int pattern, const unsigned char *b, unsigned int at,
                                     unsigned int end)
{
    unsigned int first;
    const unsigned int span = utf8_at(b, end, at, &first);
    if (pattern == AOTX_TEXT_PATTERN_GPT2) {
        const unsigned int c = contraction(b, at, end, 0);
        if (c != 0u) return c;
        const unsigned int from = first == ' ' ? at + 1u : at;
        unsigned int walk = letter_run(b, end, from, 0);
        if (walk == from) walk = number_run(b, end, from, 0u);
        if (walk == from) walk = other_run(b, end, from, 0);
        if (walk > from) return walk - at;
        return spaces(b, end, at, span, 0);
    }
    const int marks = pattern == AOTX_TEXT_PATTERN_QWEN35;
    const unsigned int most = pattern == AOTX_TEXT_PATTERN_LLAMA3 ? 3u : 1u;
    const unsigned int c = contraction(b, at, end, 1);
    if (c != 0u) return c;
    {
        unsigned int from = at;
        if (first != '\r' && first != '\n' && !is_letter(first) && !is_number(first)
            && !(marks && is_mark(first)))
            from = at + span;
        const unsigned int walk = letter_run(b, end, from, marks);
        if (walk > from) return walk - at;
    }
    if (is_number(first)) return number_run(b, end, at, most) - at;
    {
        const unsigned int from = first == ' ' ? at + 1u : at;
        unsigned int walk = other_run(b, end, from, marks);
        if (walk > from) {
            while (walk < end && (b[walk] == '\r' || b[walk] == '\n')) walk += 1u;
            return walk - at;
        }
    }
    return spaces(b, end, at, span, 1);
}

/* The sum of `mine` over the threads before this one of a workgroup of 1024, and over all of
 * them in *total. `part` is 16 words of LDS; ends with every thread past its reads. */
static __device__ __forceinline__ unsigned int block_before(unsigned int mine, unsigned int *part,
                                                            unsigned int *total)
{
    const unsigned int lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    unsigned int incl = mine;
#pragma unroll
    for (unsigned int d = 1u; d < 64u; d <<= 1) {
        const unsigned int o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
    }
    if (lane == 63u) part[wave] = incl;
    __syncthreads();
    unsigned int before = 0u, all = 0u;
#pragma unroll
    for (unsigned int w = 0u; w < 16u; ++w) {
        const unsigned int n = part[w];
        before += w < wave ? n : 0u;
        all += n;
    }
    __syncthreads();
    *total = all;
    return before + incl - mine;
}

/* Whether a character starts at `at`, reading forward from `from`: every byte but those that
 * a whole character before it holds. A lead byte is never inside another character, so the
 * bytes up to the nearest lead decide it. */
static __device__ bool char_starts(const unsigned char *b, unsigned int from, unsigned int end, unsigned int at)
{
    if ((b[at] & 0xC0u) != 0x80u) return true;
    for (unsigned int j = 1u; j <= 3u && at >= from + j; ++j) {
        if ((b[at - j] & 0xC0u) == 0x80u) continue;
        unsigned int p;
        return utf8_at(b, end, at - j, &p) <= j;
    }
    return true;
}

/* A workgroup per text, four bytes per thread: the text with every byte that does not start a
 * UTF-8 character (and the bytes of a cut or malformed one) written as U+FFFD, EF BF BD
 * (cuda/text/text.cuh:367-374); text t goes to out + 3 at[t], its length to clean_len[t], and
 * the marks of its places (mark, the pre-token pass's) are cleared. Each byte decides by
 * itself whether it is kept (one byte) or replaced (three), and a prefix sum places it. Bound
 * by the latency of its byte loads; 64 texts of 4000 bytes 2765 -> 14.5 us against one thread
 * per text. */
__global__ __launch_bounds__(1024) void aotx_text_clean_kernel(const unsigned char *bytes,
                                                               const unsigned long long *at,
                                                               unsigned int texts, unsigned char *out,
                                                               unsigned char *mark, unsigned int *clean_len,
                                                               unsigned int *longs)
{
    __shared__ unsigned int part[16];
    for (unsigned int t = blockIdx.x; t < texts; t += gridDim.x) {
        const unsigned char *b = bytes + at[t];
        const unsigned int end = (unsigned int)(at[t + 1u] - at[t]);
        unsigned char *o = out + 3ull * at[t], *m = mark + 3ull * at[t];
        if (t == 0u && threadIdx.x == 0u) *longs = 0u;
        unsigned int done = 0u;
        for (unsigned int tile = 0u; tile < end; tile += 4096u) {
            const unsigned int i0 = tile + 4u * threadIdx.x;
            unsigned int bad = 0u, n = 0u;
#pragma unroll
            for (unsigned int j = 0u; j < 4u; ++j) {
                const unsigned int i = i0 + j;
                if (i >= end) continue;
                bool replace = false;
                if (b[i] >= 0x80u && char_starts(b, 0u, end, i)) {
                    unsigned int p;
                    replace = utf8_at(b, end, i, &p) == 1u;
                }
                bad |= replace ? 1u << j : 0u;
                n += replace ? 3u : 1u;
            }
            unsigned int total;
            unsigned int w = done + block_before(n, part, &total);
#pragma unroll
            for (unsigned int j = 0u; j < 4u; ++j) {
                const unsigned int i = i0 + j;
                if (i >= end) continue;
                if ((bad >> j) & 1u) {
                    o[w] = 0xEFu; o[w + 1u] = 0xBFu; o[w + 2u] = 0xBDu;
                    m[w] = 0u; m[w + 1u] = 0u; m[w + 2u] = 0u;
                    w += 3u;
                } else {
                    o[w] = b[i];
                    m[w] = 0u;
                    w += 1u;
                }
            }
            done += total;
        }
        if (threadIdx.x == 0u) clean_len[t] = done;
    }
}

/* The longest special token whose bytes start at `at` (cuda/text/pretok.cu:339-372): its
 * length, 0 for none. */
static __device__ unsigned int special_at(const aotx_text_vocab &v, const unsigned char *b,
                                          unsigned int at, unsigned int end, unsigned int *token)
{
    const unsigned int c = b[at];
    if (((v.first[c >> 6] >> (c & 63u)) & 1ull) == 0ull) return 0u;
    unsigned int best = 0u;
    for (unsigned int i = 0u; i < v.specials; ++i) {
        const unsigned int id = v.special[i];
        const unsigned long long f = v.token_at[id];
        const unsigned int n = (unsigned int)(v.token_at[id + 1u] - f);
        if (n <= best || at + n > end) continue;
        unsigned int k = 0u;
        while (k < n && v.token_bytes[f + k] == b[at + k]) k += 1u;
        if (k == n) { best = n; *token = id; }
    }
    return best;
}

#define TX_MARK_START   1u     /* a pre-token starts here */
#define TX_MARK_SPECIAL 2u     /* a special token starts here */

/* One wave per text: the places of its special tokens, in order: the leftmost first, the
 * longest there, then from its end on. The i-th of text t starts at sat[3 at[t] + i] and ends
 * at send[3 at[t] + i]; scount[t] counts them. */
__global__ __launch_bounds__(64) void aotx_text_special_kernel(aotx_text_vocab v, const unsigned char *bytes,
                                                               const unsigned long long *at,
                                                               const unsigned int *clean_len, unsigned int texts,
                                                               unsigned char *mark, unsigned int *sat,
                                                               unsigned int *send, unsigned int *scount)
{
    const unsigned int lane = threadIdx.x;
    for (unsigned int t = blockIdx.x; t < texts; t += gridDim.x) {
        const unsigned long long base = 3ull * at[t];
        const unsigned char *b = bytes + base;
        const unsigned int end = clean_len[t];
        unsigned int pos = 0u, n = 0u;
        for (unsigned int tile = 0u; tile < end; tile += 512u) {
            unsigned int c[8];
#pragma unroll
            for (unsigned int j = 0u; j < 8u; ++j) {
                const unsigned int i = tile + 64u * j + lane;
                c[j] = b[i < end ? i : tile];
            }
#pragma unroll
            for (unsigned int j = 0u; j < 8u; ++j) {
                const unsigned int i = tile + 64u * j + lane;
                const bool maybe = i < end && ((v.first[c[j] >> 6] >> (c[j] & 63u)) & 1ull) != 0ull;
                if (!__any(maybe)) continue;
                unsigned int id = 0u;
                const unsigned int span = maybe ? special_at(v, b, i, end, &id) : 0u;
                unsigned long long found = __ballot(span != 0u);
                while (found != 0ull) {
                    const unsigned int l = (unsigned int)__builtin_ctzll(found);
                    found &= found - 1ull;
                    const unsigned int p = tile + 64u * j + l, k = (unsigned int)__shfl((int)span, (int)l, 64);
                    if (p < pos) continue;                   /* inside the one before */
                    if (lane == 0u) {
                        mark[base + p] = TX_MARK_SPECIAL;
                        sat[base + n] = p;
                        send[base + n] = p + k;
                    }
                    n += 1u;
                    pos = p + k;
                }
            }
        }
        if (lane == 0u) scount[t] = n;
    }
}

/* Whether every way of cutting the text up to `at` has a cut at `at`, a place where a
 * character starts in the run [from, end): its start; or a letter (or, with the family's
 * marks, a mark) or a number before it and no such character at it. A pre-token that holds a
 * letter is a run of letters or a contraction, and one that holds a number is a run of
 * numbers; both end where the run ends (one that is cut at AOTX_TEXT_CHUNK_BYTES ends
 * earlier, and the rest is matched again). */
static __device__ bool is_sync(unsigned int pattern, const unsigned char *b, unsigned int from,
                               unsigned int end, unsigned int at)
{
    if (at == from) return true;
    unsigned int before = 0xFFFDu, here, k = at - 1u;
    while (k > from && at - k < 4u && (b[k] & 0xC0u) == 0x80u) k -= 1u;
    unsigned int p;
    if (utf8_at(b, end, k, &p) == at - k) before = p;
    const int marks = pattern == AOTX_TEXT_PATTERN_QWEN35;
    const bool letter = is_letter(before) || (marks && is_mark(before));
    if (!letter && !is_number(before)) return false;
    utf8_at(b, end, at, &here);
    return letter ? !(is_letter(here) || (marks && is_mark(here))) : !is_number(here);
}

/* One thread per byte of the cleaned texts (chunks workgroups of 256 per text, each taking
 * every chunks-th tile): a thread at a place of is_sync runs the pattern from there to the
 * next such place, mostly one or two pre-tokens, and marks each start. A text without letters
 * or numbers is one thread's, as every text was before. Bound by the chain of byte loads of a
 * word: 64 texts of 4000 bytes 6812 -> 45 us. */
__global__ __launch_bounds__(256) void aotx_text_pretok_kernel(aotx_text_vocab v, const unsigned char *bytes,
                                                               const unsigned long long *at,
                                                               const unsigned int *clean_len, unsigned int texts,
                                                               unsigned int chunks, const unsigned int *sat,
                                                               const unsigned int *send, const unsigned int *scount,
                                                               unsigned char *mark)
{
    for (unsigned int t = blockIdx.x / chunks; t < texts; t += gridDim.x / chunks) {
        const unsigned long long base = 3ull * at[t];
        const unsigned char *b = bytes + base;
        const unsigned int text_end = clean_len[t];
        for (unsigned int tile = (blockIdx.x % chunks) * 256u; tile < text_end; tile += chunks * 256u) {
            unsigned int pos = tile + threadIdx.x;
            if (pos >= text_end) break;
            unsigned int from = 0u, end = text_end;
            if (v.specials != 0u) {
                /* the run between special tokens that holds pos: after the last one at or before it */
                unsigned int lo = 0u, hi = scount[t];
                while (lo < hi) {
                    const unsigned int mid = (lo + hi) >> 1;
                    if (sat[base + mid] <= pos) lo = mid + 1u; else hi = mid;
                }
                if (lo > 0u) from = send[base + lo - 1u];
                if (lo < scount[t]) end = sat[base + lo];
                if (pos < from) continue;                    /* inside a special token */
            }
            if (!char_starts(b, from, end, pos) || !is_sync(v.pattern, b, from, end, pos)) continue;
            do {
                unsigned int m = match(v.pattern, b, pos, end);
                if (m == 0u) m = 1u;
                if (m > AOTX_TEXT_CHUNK_BYTES) {          /* cut at a character boundary */
                    unsigned int cut = 0u;
                    while (cut < end - pos) {
                        unsigned int p;
                        const unsigned int k = utf8_at(b, end, pos + cut, &p);
                        if (cut + k > AOTX_TEXT_CHUNK_BYTES) break;
                        cut += k;
                    }
                    m = cut;
                }
                mark[base + pos] = TX_MARK_START;
                pos += m;
            } while (pos < end && !is_sync(v.pattern, b, from, end, pos));
        }
    }
}

/* ---- merge -------------------------------------------------------------------------------- */

#define TX_N AOTX_TEXT_CHUNK_BYTES
#define TX_SHORT 32u           /* bytes of the pre-tokens that one lane merges */
#define TX_WAVES 4u

/* A wave per 64 places of a cleaned text. The lane at a pre-token's first byte owns it; the
 * tokens go where its bytes are (never more than those), their number to count[place], which
 * is 0 at every other place. The pairs of neighbouring bytes are looked up by all lanes at
 * once; then every lane merges its own pre-token in its bytes' places of LDS. Most pre-tokens
 * hold a few bytes, so a wave of lanes with one each is busier than a wave for each, and needs
 * 6 KB of LDS instead of 64 (64 texts of 4000 bytes 370 -> 37 us, bound by the chain of table
 * lookups). Longer ones are left to aotx_text_long_kernel, in a list of (text, place,
 * bytes). */
__global__ __launch_bounds__(64 * TX_WAVES) void aotx_text_merge_kernel(aotx_text_vocab v, const unsigned char *bytes,
                                                                        const unsigned long long *at,
                                                                        const unsigned int *clean_len,
                                                                        const unsigned char *mark, unsigned int texts,
                                                                        unsigned int chunks, unsigned int *out,
                                                                        unsigned short *count,
                                                                        unsigned int *long_list, unsigned int *longs)
{
    __shared__ unsigned int tokl[TX_WAVES][64 + TX_SHORT], rankl[TX_WAVES][64 + TX_SHORT], resl[TX_WAVES][64 + TX_SHORT];
    __shared__ unsigned char nxtl[TX_WAVES][64 + TX_SHORT], prvl[TX_WAVES][64 + TX_SHORT];
    const unsigned int lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    unsigned int *tok = tokl[wave], *rank = rankl[wave], *res = resl[wave];
    unsigned char *nxt = nxtl[wave], *prv = prvl[wave];
    for (unsigned int t = blockIdx.x / chunks; t < texts; t += gridDim.x / chunks) {
        const unsigned long long base = 3ull * at[t];
        const unsigned char *b = bytes + base;
        const unsigned int end = clean_len[t];
        for (unsigned int w = ((blockIdx.x % chunks) * TX_WAVES + wave) * 64u; w < end; w += chunks * TX_WAVES * 64u) {
            const unsigned int p = w + lane;
            const unsigned int kind = p < end ? mark[base + p] : 0u;
            const unsigned long long starts = __ballot(kind != 0u);
            if (p < end) count[base + p] = 0u;
            if (starts == 0ull) continue;                    /* inside a longer one */
            /* the end of the last pre-token that starts here */
            unsigned int after = w + 64u;
            for (; after < end; after += 64u) {
                const unsigned int q = after + lane;
                const unsigned long long more = __ballot(q < end && mark[base + (q < end ? q : after)] != 0u);
                if (more != 0ull) {
                    after += (unsigned int)__builtin_ctzll(more);
                    break;
                }
            }
            if (after > end) after = end;
            const unsigned long long later = lane == 63u ? 0ull : starts >> (lane + 1u);
            const unsigned int n = later != 0ull ? 1u + (unsigned int)__builtin_ctzll(later) : after - p;
            unsigned int *dst = out + base + p;
            bool open = kind != 0u;
            if (kind == TX_MARK_SPECIAL) {
                unsigned int id = AOTX_TEXT_NONE;
                special_at(v, b, p, end, &id);
                dst[0] = id;
                count[base + p] = 1u;
                open = false;
            } else if (open && v.whole) {
                const unsigned int whole = find_bytes(v, b + p, n);
                if (whole != AOTX_TEXT_NONE) {
                    dst[0] = whole;
                    count[base + p] = 1u;
                    open = false;
                }
            }
            if (open && n > TX_SHORT) {
                unsigned int *item = long_list + 3ull * atomicAdd(longs, 1u);
                item[0] = t;
                item[1] = p;
                item[2] = n;
                open = false;
            }
            const unsigned long long mine = __ballot(open);
            if (mine == 0ull) continue;
            /* every byte's token and its pair with the next, the last pre-token's bytes past the
             * window in a second round */
#pragma unroll
            for (unsigned int round = 0u; round < 2u; ++round) {
                const unsigned int i = round * 64u + lane;
                const unsigned long long upto = round != 0u ? starts : starts & (~0ull >> (63u - lane));
                const unsigned int own = upto != 0ull ? 63u - (unsigned int)__builtin_clzll(upto) : 64u;
                const unsigned int size = (unsigned int)__shfl((int)n, (int)(own & 63u), 64);
                if (i < 64u + TX_SHORT && own < 64u && ((mine >> own) & 1ull) != 0ull && i < own + size) {
                    const unsigned int x = v.byte_token[b[w + i]];
                    unsigned int r = 0u, k = AOTX_TEXT_NONE;
                    if (i + 1u < own + size) k = find_pair(v, x, v.byte_token[b[w + i + 1u]], &r);
                    tok[i] = x;
                    rank[i] = k;
                    res[i] = r;
                    nxt[i] = (unsigned char)(i + 1u);
                    prv[i] = i == own ? 0xFFu : (unsigned char)(i - 1u);
                }
            }
            /* the wave's writes before its lanes' reads of one another's places */
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (open) {
                const unsigned int last = lane + n;
                for (;;) {
                    unsigned int best = AOTX_TEXT_NONE, i = lane;
                    for (unsigned int q = lane; q < last; ++q) {
                        const unsigned int k = rank[q];
                        if (k < best) { best = k; i = q; }
                    }
                    if (best == AOTX_TEXT_NONE) break;
                    const unsigned int j = nxt[i], k = nxt[j], f = prv[i], x = res[i];
                    unsigned int ranks[2], made[2];
                    find_pairs(v, x, k < last ? tok[k] : AOTX_TEXT_NONE, f != 0xFFu ? tok[f] : AOTX_TEXT_NONE, x, ranks,
                               made);
                    tok[i] = x;
                    nxt[i] = (unsigned char)k;
                    if (k < last) prv[k] = (unsigned char)i;
                    rank[j] = AOTX_TEXT_NONE;
                    rank[i] = ranks[0];
                    res[i] = made[0];
                    if (f != 0xFFu) {
                        rank[f] = ranks[1];
                        res[f] = made[1];
                    }
                }
                unsigned int c = 0u;
                for (unsigned int i = lane; i < last; i = nxt[i]) dst[c++] = tok[i];
                count[base + p] = (unsigned short)c;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
}

/* The pre-tokens of more than TX_SHORT bytes, a workgroup each (a fixed grid goes through the
 * list that the merge left). */
__global__ __launch_bounds__(64) void aotx_text_long_kernel(aotx_text_vocab v, const unsigned char *bytes,
                                                            const unsigned long long *at,
                                                            const unsigned int *long_list, const unsigned int *longs,
                                                            unsigned int *out, unsigned short *count)
{
    __shared__ unsigned int tok[TX_N], rank[TX_N], res[TX_N];
    __shared__ unsigned short nxt[TX_N], prv[TX_N];
    const unsigned int lane = threadIdx.x;
    const unsigned int items = *longs;
    for (unsigned int item = blockIdx.x; item < items; item += gridDim.x) {
        const unsigned long long place = 3ull * at[long_list[3ull * item]] + long_list[3ull * item + 1u];
        const unsigned int n = long_list[3ull * item + 2u];
        const unsigned char *b = bytes + place;
        unsigned int *dst = out + place;
        __syncthreads();                      /* the item before is read */
        for (unsigned int i = lane; i < n; i += 64u) {
            tok[i] = v.byte_token[b[i]];
            nxt[i] = (unsigned short)(i + 1u);
            prv[i] = (unsigned short)(i == 0u ? 0xFFFFu : i - 1u);
        }
        __syncthreads();
        for (unsigned int i = lane; i < n; i += 64u) {
            unsigned int r = 0u;
            rank[i] = i + 1u < n ? find_pair(v, tok[i], tok[i + 1u], &r) : AOTX_TEXT_NONE;
            res[i] = r;
        }
        __syncthreads();
        for (;;) {
            unsigned long long best = ~0ull;
            for (unsigned int i = lane; i < n; i += 64u) {
                const unsigned long long k = ((unsigned long long)rank[i] << 32) | i;
                best = k < best ? k : best;
            }
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
                const unsigned long long o = __shfl_xor(best, d, 64);
                best = o < best ? o : best;
            }
            if ((unsigned int)(best >> 32) == AOTX_TEXT_NONE) break;
            __syncthreads();
            if (lane == 0u) {
                const unsigned int i = (unsigned int)best, j = nxt[i], k = nxt[j], f = prv[i], x = res[i];
                unsigned int ranks[2], made[2];
                find_pairs(v, x, k < n ? tok[k] : AOTX_TEXT_NONE, f != 0xFFFFu ? tok[f] : AOTX_TEXT_NONE, x, ranks, made);
                tok[i] = x;
                nxt[i] = (unsigned short)k;
                if (k < n) prv[k] = (unsigned short)i;
                rank[j] = AOTX_TEXT_NONE;
                rank[i] = ranks[0];
                res[i] = made[0];
                if (f != 0xFFFFu) {
                    rank[f] = ranks[1];
                    res[f] = made[1];
                }
            }
            __syncthreads();
        }
        if (lane == 0u) {
            unsigned int c = 0u;
            for (unsigned int i = 0u; i < n; i = nxt[i]) dst[c++] = tok[i];
            count[place] = (unsigned short)c;
        }
    }
}

/* A workgroup per text, four places per thread: the tokens of every place, in order, to
 * ids + 3 at[t] (64 texts of 4000 bytes 277 -> 6.4 us against a wave that went from pre-token
 * to pre-token). */
__global__ __launch_bounds__(1024) void aotx_text_gather_kernel(const unsigned long long *at,
                                                                const unsigned int *clean_len, unsigned int texts,
                                                                const unsigned int *tokens,
                                                                const unsigned short *place_count,
                                                                unsigned int *ids, unsigned int *count)
{
    __shared__ unsigned int part[16];
    for (unsigned int t = blockIdx.x; t < texts; t += gridDim.x) {
        const unsigned long long base = 3ull * at[t];
        const unsigned int end = clean_len[t];
        unsigned int done = 0u;
        for (unsigned int tile = 0u; tile < end; tile += 4096u) {
            unsigned int c[4], mine = 0u;
#pragma unroll
            for (unsigned int j = 0u; j < 4u; ++j) {
                const unsigned int i = tile + 4u * threadIdx.x + j;
                c[j] = i < end ? place_count[base + i] : 0u;
                mine += c[j];
            }
            unsigned int total;
            unsigned int w = done + block_before(mine, part, &total);
#pragma unroll
            for (unsigned int j = 0u; j < 4u; ++j) {
                const unsigned long long src = base + tile + 4u * threadIdx.x + j;
                for (unsigned int i = 0u; i < c[j]; ++i) ids[base + w + i] = tokens[src + i];
                w += c[j];
            }
            done += total;
        }
        if (threadIdx.x == 0u) count[t] = done;
    }
}

/* ---- detokenize ------------------------------------------------------------------------ */

static __device__ unsigned int detok_token(const aotx_text_vocab &v, unsigned int id, unsigned char *o,
                                           unsigned int room)
{
    if (id >= v.tokens || ((v.control[id >> 5] >> (id & 31u)) & 1u)) return 0u;
    const unsigned char *s = v.token_bytes + v.token_at[id];
    const unsigned int n = (unsigned int)(v.token_at[id + 1u] - v.token_at[id]);
    unsigned int w = 0u;
    for (unsigned int i = 0u; i < n;) {
        unsigned int p;
        const unsigned int k = utf8_at(s, n, i, &p);
        const unsigned int byte = point_byte(p);
        if (byte < 0x100u) {
            if (o != nullptr && w < room) o[w] = (unsigned char)byte;
            w += 1u;
        } else {
            for (unsigned int j = 0u; j < k; ++j) {
                if (o != nullptr && w < room) o[w] = s[i + j];
                w += 1u;
            }
        }
        i += k;
    }
    return w;
}

__global__ __launch_bounds__(64) void aotx_text_detok_kernel(aotx_text_vocab v, const unsigned int *ids,
                                                             const unsigned long long *at, unsigned char *bytes,
                                                             unsigned int limit, unsigned int *length)
{
    const unsigned int t = blockIdx.x, lane = threadIdx.x;
    const unsigned long long a0 = at[t], a1 = at[t + 1u];
    unsigned char *dst = bytes + (unsigned long long)t * limit;
    unsigned int w = 0u;
    for (unsigned long long c = a0; c < a1; c += 64u) {
        const unsigned long long i = c + lane;
        const unsigned int mine = i < a1 ? detok_token(v, ids[i], nullptr, 0u) : 0u;
        unsigned int incl = mine;
#pragma unroll
        for (unsigned int d = 1u; d < 64u; d <<= 1) {
            const unsigned int o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        const unsigned int from = w + incl - mine;
        if (i < a1 && from < limit) detok_token(v, ids[i], dst + from, limit - from);
        w += __shfl(incl, 63, 64);
    }
    if (lane == 0u) length[t] = w < limit ? w : limit;
}

/* ---- host -------------------------------------------------------------------------------- */

struct aotx_text_family { const char *name; unsigned int pattern, whole; };
/* cuda/text/families.h:24-43: tokenizer.ggml.pre value, split pattern, whole rule */
static const aotx_text_family kFamilies[] = {
    {"qwen2", AOTX_TEXT_PATTERN_QWEN2, 0u}, {"deepseek-r1-qwen", AOTX_TEXT_PATTERN_QWEN2, 0u},
    {"kormo", AOTX_TEXT_PATTERN_QWEN2, 0u}, {"f2llmv2", AOTX_TEXT_PATTERN_QWEN2, 0u},
    {"llama3", AOTX_TEXT_PATTERN_LLAMA3, 1u}, {"llama-v3", AOTX_TEXT_PATTERN_LLAMA3, 1u},
    {"llama-bpe", AOTX_TEXT_PATTERN_LLAMA3, 1u}, {"falcon3", AOTX_TEXT_PATTERN_LLAMA3, 1u},
    {"falcon-h1", AOTX_TEXT_PATTERN_LLAMA3, 1u}, {"pixtral", AOTX_TEXT_PATTERN_LLAMA3, 1u},
    {"midm-2.0", AOTX_TEXT_PATTERN_LLAMA3, 1u}, {"lfm2", AOTX_TEXT_PATTERN_LLAMA3, 1u},
    {"jina-v5-nano", AOTX_TEXT_PATTERN_LLAMA3, 1u}, {"gpt-2", AOTX_TEXT_PATTERN_GPT2, 0u},
    {"mpt", AOTX_TEXT_PATTERN_GPT2, 0u}, {"olmo", AOTX_TEXT_PATTERN_GPT2, 0u},
    {"jais", AOTX_TEXT_PATTERN_GPT2, 0u}, {"trillion", AOTX_TEXT_PATTERN_GPT2, 0u},
    {"granite-docling", AOTX_TEXT_PATTERN_GPT2, 0u}, {"qwen35", AOTX_TEXT_PATTERN_QWEN35, 0u},
};
static const unsigned int kFamilyCount = sizeof kFamilies / sizeof kFamilies[0];

extern "C" int aotx_text_family_find(const char *name, unsigned long long length, unsigned int *row)
{
    if (name == nullptr || row == nullptr) return 1;
    for (unsigned int i = 0; i < kFamilyCount; ++i) {
        if (strlen(kFamilies[i].name) == length && memcmp(kFamilies[i].name, name, length) == 0) {
            *row = i;
            return 0;
        }
    }
    return 1;
}

static unsigned int pow2_at_least(unsigned long long n)
{
    unsigned int p = 16u;
    while (p < n) p <<= 1;
    return p;
}

template <class T>
static T *store_put(aotx_text_store *st, const T *src, size_t count)
{
    void *d = nullptr;
    const size_t bytes = count * sizeof(T) > 0 ? count * sizeof(T) : sizeof(T);
    AOTX_CHECK(hipMalloc(&d, bytes));
    if (count) AOTX_CHECK(hipMemcpy(d, src, count * sizeof(T), hipMemcpyHostToDevice));
    st->block[st->blocks++] = d;
    st->bytes += bytes;
    return (T *)d;
}

extern "C" void aotx_text_vocab_release(aotx_text_store *store)
{
    if (store == nullptr) return;
    for (unsigned int i = 0; i < store->blocks; ++i) AOTX_CHECK(hipFree(store->block[i]));
    store->blocks = 0u;
    store->bytes = 0ull;
    g_ready = 0;
}

extern "C" int aotx_text_vocab_build(const aotx_text_source *src, aotx_text_store *store)
{
    if (src == nullptr || store == nullptr || src->tokens == 0ull || src->tokens >= 0xFFFFFFFFull
        || src->token_bytes == nullptr || src->token_at == nullptr || src->family >= kFamilyCount
        || (src->merges != 0ull && (src->merge_bytes == nullptr || src->merge_at == nullptr)))
        return 1;
    const unsigned int n = (unsigned int)src->tokens;
    std::unordered_map<std::string, unsigned int> id;
    id.reserve(n * 2u);
    for (unsigned int t = 0; t < n; ++t) {
        std::string s((const char *)src->token_bytes + src->token_at[t], src->token_at[t + 1u] - src->token_at[t]);
        id.emplace(s, t);                                /* the lowest id of a repeated string */
    }
    /* the token table by string */
    const unsigned int slots = pow2_at_least(2ull * n);
    std::vector<unsigned int> slot(slots, AOTX_TEXT_NONE);
    for (unsigned int t = 0; t < n; ++t) {
        const unsigned long long f = src->token_at[t], e = src->token_at[t + 1u];
        std::string s((const char *)src->token_bytes + f, e - f);
        if (id[s] != t) continue;
        unsigned long long h = FNV_BASIS;
        for (unsigned long long i = f; i < e; ++i) h = fnv_step(h, src->token_bytes[i]);
        unsigned int at = (unsigned int)h & (slots - 1u);
        while (slot[at] != AOTX_TEXT_NONE) at = (at + 1u) & (slots - 1u);
        slot[at] = t;
    }
    /* the pair table: rank = merge index, result = the token of the joined string */
    const unsigned int pairs = pow2_at_least(2ull * (src->merges + 1ull));
    std::vector<uint4> pair(pairs, make_uint4(AOTX_TEXT_NONE, AOTX_TEXT_NONE, AOTX_TEXT_NONE, AOTX_TEXT_NONE));
    unsigned int taken = 0u, refused = 0u;
    for (unsigned long long m = 0; m < src->merges; ++m) {
        std::string line((const char *)src->merge_bytes + src->merge_at[m], src->merge_at[m + 1u] - src->merge_at[m]);
        const size_t sp = line.find(' ', 1);
        if (sp == std::string::npos) { refused += 1u; continue; }
        const std::string l = line.substr(0, sp), r = line.substr(sp + 1);
        auto il = id.find(l), ir = id.find(r), ij = id.find(l + r);
        if (il == id.end() || ir == id.end() || ij == id.end()) { refused += 1u; continue; }
        const unsigned long long k = ((unsigned long long)il->second << 32) | ir->second;
        unsigned int at = (unsigned int)pair_mix(k) & (pairs - 1u);
        bool seen = false;
        while (pair[at].x != AOTX_TEXT_NONE || pair[at].y != AOTX_TEXT_NONE) {
            if (pair[at].x == ir->second && pair[at].y == il->second) { seen = true; break; }
            at = (at + 1u) & (pairs - 1u);
        }
        if (seen) { refused += 1u; continue; }              /* a repeated pair keeps its first rank */
        pair[at] = make_uint4(ir->second, il->second, (unsigned int)m, ij->second);
        taken += 1u;
    }
    /* control bits and the single bytes */
    std::vector<unsigned int> control((n + 31u) / 32u, 0u);
    unsigned int controls = 0u;
    if (src->token_type != nullptr)
        for (unsigned int t = 0; t < n; ++t)
            if (src->token_type[t] == AOTX_TEXT_TYPE_CONTROL) { control[t >> 5] |= 1u << (t & 31u); controls += 1u; }
    aotx_text_vocab v;
    memset(&v, 0, sizeof v);
    std::vector<unsigned int> special;
    if (src->token_type != nullptr)
        for (unsigned int t = 0; t < n; ++t)
            if ((src->token_type[t] == AOTX_TEXT_TYPE_CONTROL || src->token_type[t] == AOTX_TEXT_TYPE_USER)
                && src->token_at[t + 1u] > src->token_at[t]) {
                special.push_back(t);
                const unsigned int c = src->token_bytes[src->token_at[t]];
                v.first[c >> 6] |= 1ull << (c & 63u);
            }
    for (unsigned int b = 0; b < 256u; ++b) {
        unsigned char u[4];
        const unsigned int k = utf8_put(byte_point(b), u);
        auto it = id.find(std::string((const char *)u, k));
        if (it == id.end()) return 1;
        v.byte_token[b] = it->second;
    }
    aotx_text_vocab_release(store);
    v.token_bytes = store_put(store, src->token_bytes, src->token_at[n]);
    v.token_at = store_put(store, src->token_at, (size_t)n + 1u);
    v.tokens = n;
    v.slots = slots;
    v.slot = store_put(store, slot.data(), slots);
    v.pairs = pairs;
    v.pair = store_put(store, pair.data(), pairs);
    v.control = store_put(store, control.data(), control.size());
    v.special = store_put(store, special.data(), special.size());
    v.specials = (unsigned int)special.size();
    v.pattern = kFamilies[src->family].pattern;
    v.whole = kFamilies[src->family].whole;
    g_vocab = v;
    g_ready = 1;
    g_report[0] = n;
    g_report[1] = taken;
    g_report[2] = refused;
    g_report[3] = controls;
    return 0;
}

extern "C" int aotx_text_vocab_file(const aotx_modelfile *file, aotx_text_store *store)
{
    if (file == nullptr || store == nullptr) return 1;
    aotx_string_array tokens, merges;
    memset(&merges, 0, sizeof merges);
    if (aotx_modelfile_strings(file, "tokenizer.ggml.tokens", &tokens) != 0) return 1;
    if (aotx_modelfile_strings(file, "tokenizer.ggml.merges", &merges) != 0) merges.count = 0u;
    const int32_t *types = nullptr;
    uint64_t type_count = 0u;
    if (aotx_modelfile_i32s(file, "tokenizer.ggml.token_type", &types, &type_count) != 0
        || type_count != tokens.count)
        types = nullptr;
    const char *pre = nullptr;
    size_t pre_len = 0u;
    unsigned int family = 0u;                       /* row 0 when the file names none */
    if (aotx_modelfile_string(file, "tokenizer.ggml.pre", &pre, &pre_len) == 0
        && aotx_text_family_find(pre, pre_len, &family) != 0)
        return 1;
    aotx_text_source src;
    src.token_bytes = tokens.bytes;
    src.token_at = (const unsigned long long *)tokens.offsets;
    src.tokens = tokens.count;
    src.merge_bytes = merges.count ? merges.bytes : nullptr;
    src.merge_at = merges.count ? (const unsigned long long *)merges.offsets : nullptr;
    src.merges = merges.count;
    src.token_type = types;
    src.family = family;
    return aotx_text_vocab_build(&src, store);
}

extern "C" int aotx_text_vocab_report(unsigned int report[4])
{
    if (report == nullptr || !g_ready) return 1;
    memcpy(report, g_report, sizeof g_report);
    return 0;
}

extern "C" int aotx_text_encode(const unsigned char *bytes, const unsigned long long *at, unsigned int texts,
                                unsigned int *ids, unsigned int *count, void *stream)
{
    if (!g_ready || bytes == nullptr || at == nullptr || ids == nullptr || count == nullptr || texts == 0u)
        return 1;
    hipStream_t s = aotx_stream(stream);
    unsigned long long total = 0ull;
    AOTX_CHECK(hipMemcpyAsync(&total, at + texts, sizeof total, hipMemcpyDeviceToHost, s));
    AOTX_CHECK(hipStreamSynchronize(s));
    if (total == 0ull) {
        AOTX_CHECK(hipMemsetAsync(count, 0, texts * sizeof(unsigned int), s));
        AOTX_CHECK(hipStreamSynchronize(s));
        return 0;
    }
    /* one allocation: the cleaned bytes (every byte may become U+FFFD), the marks, and per
     * place the tokens, their number and the special tokens' places; the list of longer
     * pre-tokens holds one per TX_SHORT + 1 bytes at most */
    const size_t room = 3ull * total;
    size_t at_byte = 0u;
    const auto put = [&at_byte](size_t bytes) {
        const size_t here = at_byte;
        at_byte += (bytes + 255u) & ~(size_t)255u;
        return here;
    };
    const size_t o_clean = put(room), o_mark = put(room), o_tok = put(room * 4u), o_count = put(room * 2u),
                 o_len = put((size_t)texts * 4u), o_long = put((room / TX_SHORT + 1u) * 12u), o_longs = put(4u),
                 o_sat = put(g_vocab.specials ? room * 4u : 4u), o_send = put(g_vocab.specials ? room * 4u : 4u),
                 o_scount = put((size_t)texts * 4u);
    unsigned char *buf = nullptr;
    AOTX_CHECK(hipMallocAsync((void **)&buf, at_byte, s));
    unsigned char *clean = buf + o_clean, *mark = buf + o_mark;
    unsigned int *tok = (unsigned int *)(buf + o_tok), *clean_len = (unsigned int *)(buf + o_len);
    unsigned short *pcount = (unsigned short *)(buf + o_count);
    unsigned int *long_list = (unsigned int *)(buf + o_long), *longs = (unsigned int *)(buf + o_longs);
    unsigned int *sat = (unsigned int *)(buf + o_sat), *send = (unsigned int *)(buf + o_send),
                 *scount = (unsigned int *)(buf + o_scount);
    /* 256-byte tiles of the mean text, each a workgroup (a longer text's take several) */
    const unsigned long long tiles = (total / texts + 255ull) / 256ull;
    const unsigned long long most = 65536ull / texts > 0ull ? 65536ull / texts : 1ull;
    const unsigned int chunks = (unsigned int)(tiles < 1ull ? 1ull : (tiles < most ? tiles : most));
    /* workgroups for so many texts, each going on with later ones: a launch holds 2^32 threads, and
     * a text takes up to 1024 */
    const unsigned int most_texts = 1u << 20, here = texts < most_texts ? texts : most_texts;
    hipLaunchKernelGGL(aotx_text_clean_kernel, dim3(here), dim3(1024), 0, s, bytes, at, texts, clean, mark, clean_len,
                       longs);
    AOTX_LAUNCH_CHECK();
    if (g_vocab.specials != 0u) {
        hipLaunchKernelGGL(aotx_text_special_kernel, dim3(here), dim3(64), 0, s, g_vocab, clean, at, clean_len, texts,
                           mark, sat, send, scount);
        AOTX_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(aotx_text_pretok_kernel, dim3(here * chunks), dim3(256), 0, s, g_vocab, clean, at, clean_len,
                       texts, chunks, sat, send, scount, mark);
    AOTX_LAUNCH_CHECK();
    hipLaunchKernelGGL(aotx_text_merge_kernel, dim3(here * chunks), dim3(64 * TX_WAVES), 0, s, g_vocab, clean, at,
                       clean_len, mark, texts, chunks, tok, pcount, long_list, longs);
    AOTX_LAUNCH_CHECK();
    hipLaunchKernelGGL(aotx_text_long_kernel, dim3(512), dim3(64), 0, s, g_vocab, clean, at, long_list, longs, tok,
                       pcount);
    AOTX_LAUNCH_CHECK();
    hipLaunchKernelGGL(aotx_text_gather_kernel, dim3(here), dim3(1024), 0, s, at, clean_len, texts, tok, pcount, ids,
                       count);
    AOTX_LAUNCH_CHECK();
    AOTX_CHECK(hipFreeAsync(buf, s));
    AOTX_CHECK(hipStreamSynchronize(s));
    return 0;
}

extern "C" int aotx_text_detok(const unsigned int *ids, const unsigned long long *at, unsigned int texts,
                               unsigned char *bytes, unsigned int limit, unsigned int *length, void *stream)
{
    if (!g_ready || ids == nullptr || at == nullptr || bytes == nullptr || length == nullptr || texts == 0u)
        return 1;
    hipLaunchKernelGGL(aotx_text_detok_kernel, dim3(texts), dim3(64), 0, aotx_stream(stream), g_vocab, ids, at,
                       bytes, limit, length);
    AOTX_LAUNCH_CHECK();
    return 0;
}
