/*
 * The scores of one lane of a row of 16 in the Gomoku PUCT loop's decisions (puct_gomoku.hip: row_decisions, quick_row_decisions): a
 * lane holds an edge or nothing, and the largest score of the row is looked for among all its lanes.  Plain C99 / C++ / HIP, so that the
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

/* num / den, correctly rounded, from a reciprocal of den that is right to an ulp: a Newton step on the reciprocal, then two corrections of the
 * quotient by its residual (Markstein's), without what a division does for operands near the ends of a float's range
 * (8 instructions instead of 11).  For den from 1 to 2^31 and num
 * 0 or from 1e-20 to 1e20, where nothing on the way overflows or becomes subnormal. */
PROW_FN float prow_quotient(float num, float den, float reciprocal) {
    const float r = fmaf(fmaf(-den, reciprocal, 1.0f), reciprocal, reciprocal);
    float u = num * r;
    u = fmaf(fmaf(-den, u, num), r, u);
    return fmaf(fmaf(-den, u, num), r, u);
}
/* A cpuct * prior that stays in that range whatever the root of the parent's count, which is from 1 to 2^16. */
PROW_FN int prow_cp_fits(float cp) { return cp == 0.0f || (cp >= 1e-20f && cp <= 1e15f); }
/* prow_score where prow_cp_fits: what row_decisions compares. */
PROW_FN float prow_row_score(float q, float cp, float root, int den, float reciprocal) { return q + prow_quotient(cp * root, (float)den, reciprocal); }

/* The quick score, from cp times the reciprocal of den (cp_by) in one fused operation, and by how much an edge may be below the largest quick
 * score and still be the one with the largest score: a share of `largest`, the largest |q| + u that any of the row's decisions may see
 * (prow_quick_size, by the last root).  In units of 2^-24 of that, an edge's quick score is off by 4 for u, 2 and 2 for the sums (q has been
 * lifted so that no score is negative, and a score is at most twice that then), its score by 2 and 1, the sum with what this
 * returns by 2: 24 for two edges, and 32 are allowed for. */
PROW_FN float prow_quick_score(float q, float cp_by, float root) { return fmaf(cp_by, root, q); }
PROW_FN float prow_quick_size(float q, float cp_by, float root) { return fabsf(q) + cp_by * root; }
PROW_FN float prow_quick_apart(float largest) { return largest * 1.9073486328125e-06f /* 2^-19 */; }
#endif
