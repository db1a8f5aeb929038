/*
 * wg_span.h -- steps through a range [p, e) of edge positions.
 *
 * A graph may have up to 2^32 - 2 edges, so p + lane or p + width of a step near
 * the end of the last range can wrap around: the position then passes a test
 * against e, and a loop that adds its width starts again at the front of the edge
 * list.  What is left of the range, e - p, cannot.
 */
#ifndef WG_SPAN_H
#define WG_SPAN_H

#include <stdint.h>

#ifdef __HIPCC__
#define WG_SPAN_HD __host__ __device__
#else
#define WG_SPAN_HD
#endif

/* Positions that a step of `width` from p takes: p + i for i < the result, which is
 * 0 at the end.  The next step starts at p + the result. */
static inline WG_SPAN_HD uint32_t wg_step(uint32_t p, uint32_t e, uint32_t width)
{
    const uint32_t left = e - p;
    return left < width ? left : width;
}

#endif
