/*
 * The score of one lane of a row of 16 in the Gomoku PUCT loop's decisions (puct_gomoku.hip, row_decisions): a lane holds an
 * edge or nothing, and the largest score of the row is looked for among all its lanes.  Plain C99 / C++ / HIP, so that the
 * host can check the terms over every word that a lane may have loaded.
 */
#ifndef MCTSNC_PUCT_ROW_H
#define MCTSNC_PUCT_ROW_H
#include <float.h>
#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#define PROW_FN __host__ __device__ inline
#else
#define PROW_FN static inline
#endif

typedef struct { float q, cp; int den; } prow_terms;   /* mean value, cpuct * prior, visits + claims in flight + 1 */

/* Terms of a lane.  A lane without an edge has loaded a slot that nobody may have written yet: none of its words counts, and
 * its score is finite and below that of every edge (whose terms are below 1e30 and whose den is positive). */
PROW_FN prow_terms prow_terms_of(int has_edge, float q, float cp, int den) {
    prow_terms t;
    t.q = has_edge ? q : -FLT_MAX;
    t.cp = has_edge ? cp : 0.0f;
    t.den = has_edge ? den : 1;
    return t;
}

PROW_FN float prow_score(prow_terms t, float sqrt_parent) { return t.q + t.cp * sqrt_parent / (float)t.den; }

/* Order-preserving integer image of a finite score; -0.0f counts as +0.0f. */
PROW_FN uint32_t prow_image(float score) {
    const float s = score + 0.0f;
    uint32_t b;
    memcpy(&b, &s, sizeof b);
    return b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
}
#endif
