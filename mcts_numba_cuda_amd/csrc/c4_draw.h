/*
 * The uniform of a Connect 4 playout's draw from the generator's 64-bit output.  Plain C99 / C++ / HIP, so that the host can
 * compare it with the reference's arithmetic (tests/test_c4_draw.py).
 */
#ifndef MCTSNC_C4_DRAW_H
#define MCTSNC_C4_DRAW_H
#include <stdint.h>

#if defined(__HIPCC__)
#define C4DRAW_FN __host__ __device__ __forceinline__
#else
#define C4DRAW_FN static inline
#endif

/* The uniform times 2^32.  The reference's is the float32 of the upper 53 bits, a single rounding; here it takes four
 * instructions without float64 (which took six, four of them conversions): the upper word's conversion rounds as the whole
 * would if its last bit says whether anything follows, as long as at least two bits are dropped, that is from 2^25 on.
 * Below that the ordinal is 0 anyway: with at most 8 columns it is as long as the uniform is below 1/8. */
C4DRAW_FN float c4_draw(uint64_t output) {
    const uint32_t rest = (uint32_t)output >> 11;
    return (float)((uint32_t)(output >> 32) | (rest < 1u ? rest : 1u));
}
#endif
