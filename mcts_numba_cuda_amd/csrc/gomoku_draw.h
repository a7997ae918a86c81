/*
 * Where in a playout's list of cells a draw falls.  Plain C99 / C++ / HIP, so that the host can compare it with the reference's
 * arithmetic (tests/test_gomoku_draw.py).
 *
 * The reference's ordinal is int(u * float(count)), u the float32 of the output's upper 53 bits (src/mctsnc.py:1882): two roundings.
 * With h, the output's upper word, u * count is not far from z = h * count / 2^32, which is one integer product: the bits below h
 * add less than count / 2^32, u's rounding moves it by at most count * 128 / 2^32 (half a unit of a float32 below 1) and the
 * product's by at most count * 256 / 2^32 (half a unit of a float32 up to count).  So the ordinal is z's whole part wherever
 * z's fraction keeps count * 384 / 2^32 from 0 and count * 385 / 2^32 from 1.
 */
#ifndef MCTSNC_GOMOKU_DRAW_H
#define MCTSNC_GOMOKU_DRAW_H
#include <stdint.h>

#if defined(__HIPCC__)
#define GDRAW_FN __host__ __device__ __forceinline__
#else
#define GDRAW_FN static inline
#endif

/* z + most * 385 / 2^32, times 2^32, for a list of count cells, at most `most` <= 4096: the ordinal is the upper word, unless the lower
 * one is below gomoku_unsure(most). */
GDRAW_FN uint64_t gomoku_place(uint64_t output, uint32_t count, uint32_t most) {
    return (uint64_t)(uint32_t)(output >> 32) * count + (uint64_t)(most * 385u);
}
GDRAW_FN uint32_t gomoku_unsure(uint32_t most) { return most * (384u + 385u); }
#endif
