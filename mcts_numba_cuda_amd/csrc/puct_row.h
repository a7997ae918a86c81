/*
 * The score of one lane of a row of 16 in the Gomoku PUCT loop's decisions (puct_gomoku.hip, row_decisions): a lane holds an
 * edge or nothing, and the largest score of the row is looked for among all its lanes.  Plain C99 / C++ / HIP, so that the
 * host can check the terms over every word that a lane may have loaded.
 */
#ifndef MCTSNC_PUCT_ROW_H
#define MCTSNC_PUCT_ROW_H
#include <float.h>
#include <math.h>

#if defined(__HIPCC__)
#define PROW_FN __host__ __device__ inline
#else
#define PROW_FN static inline
#endif

/* The terms of a lane's score: mean value, cpuct * prior, and visits + claims in flight + 1.  A lane without an edge has loaded a
 * slot that nobody may have written yet: none of its words counts, and its score is finite and below that of every edge (whose
 * terms are below 1e30 and whose denominator is positive). */
PROW_FN float prow_q(int has_edge, float q) { return has_edge ? q : -FLT_MAX; }
PROW_FN float prow_cp(int has_edge, float cp) { return has_edge ? cp : 0.0f; }
PROW_FN int prow_den(int has_edge, int den) { return has_edge ? den : 1; }
PROW_FN float prow_score(float q, float cp, float sqrt_parent, int den) { return q + cp * sqrt_parent / (float)den; }

/* num / den, correctly rounded, from a reciprocal of den that is right to an ulp: the steps of the division that the compiler makes,
 * without those that see to operands near the ends of a float's range (8 instructions instead of 11).  For den from 1 to 2^31 and num
 * 0 or from 1e-20 to 1e20, where nothing on the way overflows or becomes subnormal. */
PROW_FN float prow_quotient(float num, float den, float reciprocal) {
    const float r = fmaf(fmaf(-den, reciprocal, 1.0f), reciprocal, reciprocal);
    float u = num * r;
    u = fmaf(fmaf(-den, u, num), r, u);
    return fmaf(fmaf(-den, u, num), r, u);
}
/* A cpuct * prior that stays in that range whatever the root of the parent's count, which is from 1 to 2^16. */
PROW_FN int prow_cp_fits(float cp) { return cp == 0.0f || (cp >= 1e-20f && cp <= 1e15f); }
#endif
