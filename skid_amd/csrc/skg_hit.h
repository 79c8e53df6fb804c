// skg_hit.h -- the term that one marked entry of a tile's list adds to a mover's
// sums.  Plain C++ without device functions, so that a test can compile it for
// the host.
#pragma once
#include <math.h>
#ifndef SKG_HIT_FN
#define SKG_HIT_FN __device__ __forceinline__
#endif

// d f for a hit, else zero.  The list steps have no branch around their sums: a
// lane adds a term for each of its marks, and for none when it has no mark left.
// The zero is selected, not multiplied in: an entry at a position that is not
// finite, or so far off that d overflows, is marked for every lane (its test
// value is unordered) and dropped by the exact test, and 0 d would be NaN.
SKG_HIT_FN float hit_term(bool hit, float d, float f) { return hit ? d * f : 0.f; }

// Whether a separation from this position, with a period's shift, can fail to be
// finite.  Where no mover of the tile and no entry of the window lies so, a step
// multiplies by zero instead: one select a mark, not three (the selects in every
// window cost 0.9% of a pass of 2,097,152 particles of gas and dark matter, 1.3%
// of one of 48 uneven boxes).
SKG_HIT_FN bool far_off(float x, float y, float z) { return !(fabsf(x) + fabsf(y) + fabsf(z) < 1e37f); }
