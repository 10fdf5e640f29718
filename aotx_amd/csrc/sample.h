/* Sampler (sample.hip): launch interface for the model runtime. */
#ifndef AOTX_SAMPLE_H
#define AOTX_SAMPLE_H

#include "aotx_internal.h"

void aotx_launch_pick(const float *logits, unsigned int ld, unsigned int vocab,
                      const unsigned int *rows_dev, unsigned int rows,
                      const unsigned int *agent, const aotx_model_how *how,
                      unsigned int top_k, float top_p, float temperature,
                      unsigned long long seed, int *token, unsigned int *draw,
                      const aotx_model_run *run, unsigned int *best, hipStream_t s);
/* Bytes of the sampler's buffer (`best`) for `rows` rows of `vocab` logits: each row's largest
 * logits by slice, first-pass bucket counts, partial sums and their total, and the slices'
 * candidates with their counts (35 KB a row, whatever the vocabulary). Every call sets what it
 * counts in to zero. */
size_t aotx_pick_scratch(unsigned int rows, unsigned int vocab);

#endif
