// Cells around a particle (on the device; the same code compiles for the host).
#ifndef SPHERE_AMD_DEM_CELLS_HPP_
#define SPHERE_AMD_DEM_CELLS_HPP_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sphx {

// The cell coordinate floor(v) along an axis of n cells, src/contactsearch.cuh:
// 352-354.  A coordinate so far outside that every cell next to it is skipped
// (find_dist_mod shifts by one period at most) is moved to the nearest such
// one: the coordinates beside it then exist as integers.  They would not beside
// the largest one, which the conversion of a far particle gives; the compiler
// takes that for granted and accepted the cells above it, 2^31 layers away.
__host__ __device__ inline __attribute__((always_inline)) int cell_coord(double v, int n) {
    const double lo = -(double)n - 2.0, hi = 2.0 * n + 1.0;
    const double c = v == v ? floor(v) : 0.0;
    return (int)(c < lo ? lo : c > hi ? hi : c);
}

// findDistMod, src/contactsearch.cuh:12-83.  Returns the image code (see
// CW_SHIFT_*) or -1 when the target cell lies outside the grid.
template <class Params>
__host__ __device__ inline __attribute__((always_inline)) int find_dist_mod(Params& p, int& tx,
                                                                          int& ty, int tz) {
    const int nx = (int)p.num[0], ny = (int)p.num[1], nz = (int)p.num[2];
    int code = 0;
    if (p.periodic == 1) {
        if (tx < 0) { tx += nx; code |= 1; }
        if (tx >= nx) { tx -= nx; code |= 2; }
        if (ty < 0) { ty += ny; code |= 4; }
        if (ty >= ny) { ty -= ny; code |= 8; }
    }
    if (p.periodic == 2) {
        if (tx < 0) { tx += nx; code |= 1; }
        if (tx >= nx) { tx -= nx; code |= 2; }
        if (ty < 0 || ty >= ny) return -1;
    }
    if (p.periodic > 2 || p.periodic < 1) {
        if (tx < 0 || tx >= nx) return -1;
        if (ty < 0 || ty >= ny) return -1;
    }
    if (tz < 0 || tz >= nz) return -1;
    // A particle far outside the grid can leave tx/ty out of range after one
    // periodic shift; the reference then reads outside cellStart.  Such a
    // cell is skipped here.
    if (tx < 0 || tx >= nx || ty < 0 || ty >= ny) return -1;
    return code;
}

}  // namespace sphx

#endif
