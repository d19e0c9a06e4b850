// ee_tile_div.h -- the quotient of a tile index by a tile count that is only known on the
// device.  Plain C++ (host or device), so that a host program can check it.
#pragma once
#include <cstdint>

#ifndef EE_TILE_DIV_FN
#define EE_TILE_DIV_FN inline
#endif

// i / t for 0 <= i < 2^30 and 0 < t < 2^30 (a launch has fewer than 2^26 wavefronts); rt: 1 / float(t) to within 1 ulp (v_rcp_f32).
// A first quotient from f32 (off by up to i / t * 2^-21 + 1), a second from its remainder (off
// by at most one), and one compare: exact for every list of tiles that a grid can hold.  The remainder is taken
// modulo 2^32; its own size stays below 2^31.  (An integer division by a count from memory, ~40 dependent
// instructions on the kernel's critical path, cost 0.4 us per launch.)
EE_TILE_DIV_FN int tile_div_rcp(int i, int t, float rt) {
    uint32_t q = (uint32_t)(int)((float)i * rt);
    const int r0 = (int)((uint32_t)i - q * (uint32_t)t);
    q += (uint32_t)(int)((float)r0 * rt);
    const int r = (int)((uint32_t)i - q * (uint32_t)t);
    return (int)q + (r >= t ? 1 : r < 0 ? -1 : 0);
}
