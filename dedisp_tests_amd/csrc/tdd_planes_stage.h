// Staging of one window of the bit-plane channel sum: which row words make its
// positions and where they go in LDS. Plain arithmetic on 32-bit unsigned
// values, so that a host program can enumerate it.
#pragma once

#include <stdint.h>

#include "kernels.h"

#ifdef __HIPCC__
#define DD_STAGE_FN __device__ __forceinline__
#else
#define DD_STAGE_FN static inline
#endif

// Position (in 32-bit wrap) in the window of word u of a lane that holds
// position p < T of the rows, for a window that starts at sample a: u*T + p is
// a's run r0 = a/T % 32 plus u. Negative, as a large unsigned, for a first word
// before the window.
DD_STAGE_FN uint32_t planes_window_pos(uint32_t a, uint32_t p, uint32_t u)
{
    return p - a % DD_TDD_PLANES_T + u * DD_TDD_PLANES_T;
}

// LDS word of a lane's first word in the window of slot, windows of stride
// positions of nbits words, and of its word u from that. The whole sum stays a
// 32-bit unsigned (a first word before the window wraps, and is not written),
// so no address outside LDS is ever formed.
DD_STAGE_FN uint32_t planes_lds_first(uint32_t slot, uint32_t stride, uint32_t a, uint32_t p, uint32_t nbits)
{
    return (slot * stride + planes_window_pos(a, p, 0)) * nbits;
}
DD_STAGE_FN uint32_t planes_lds_word(uint32_t first, uint32_t u, uint32_t nbits)
{
    return first + u * (DD_TDD_PLANES_T * nbits);
}

// Words a lane has for a window of P positions from sample a on.
DD_STAGE_FN uint32_t planes_words(uint32_t a, uint32_t P)
{
    const uint32_t nu = (a % DD_TDD_PLANES_T + P + DD_TDD_PLANES_T - 1) / DD_TDD_PLANES_T;
    return nu > 1 ? nu : 1;
}

// Whether the window's runs pass the start of the next tile, so that the third
// row word is read.
DD_STAGE_FN bool planes_needs_third(uint32_t a, uint32_t P)
{
    return a / DD_TDD_PLANES_T % 32 + (a % DD_TDD_PLANES_T + P + DD_TDD_PLANES_T - 1) / DD_TDD_PLANES_T > 32;
}

// put(k, shift, u, in) for every word u of a lane at position p of the rows:
// the funnel shift by shift (mod 32) of row words k and k + 1 of the window's
// start tile, written at planes_window_pos(a, p, u) where in. Only the first
// and the last word of a lane may lie outside; from u = 32 - r0 on the runs
// start in the next tile.
template <typename Put>
DD_STAGE_FN void planes_stage(uint32_t a, uint32_t P, uint32_t p, Put put)
{
    const uint32_t r0 = a / DD_TDD_PLANES_T % 32;
    const uint32_t last = planes_words(a, P) - 1;
    const uint32_t u1 = last < 32 - r0 ? last : 32 - r0;
    put(0, r0, 0u, planes_window_pos(a, p, 0) < P);
    for (uint32_t u = 1; u < u1; ++u) put(0, r0 + u, u, true);
    for (uint32_t u = u1 > 1 ? u1 : 1; u < last; ++u) put(1, r0 + u, u, true);
    if (last > 0) {
        const bool in = planes_window_pos(a, p, last) < P;
        if (r0 + last < 32) put(0, r0 + last, last, in);
        else put(1, r0 + last, last, in);
    }
}
