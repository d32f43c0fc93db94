// The grid of the overlap search, chosen from the extremes of the positions
// and radii (on the device; the same code compiles for the host).
#ifndef SPHERE_AMD_OVERLAP_GRID_HPP_
#define SPHERE_AMD_OVERLAP_GRID_HPP_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sphx {

// Uniform grid of the overlap search: cells of side 1/inv_h >= the largest
// contact distance, n[d] cells per axis from lo[d]; key = (z n1 + y) n0 + x.
struct OverlapGrid {
    double lo[3];
    double inv_h;
    int n[3];
    int use;                   // 0: positions or extents not finite, no grid
    unsigned long long total;  // overlaps found
};

// A uniform grid whose cells are at least the largest contact distance
// (2 r_max, with a margin for the rounding of the cell coordinates) holds
// every overlapping pair within adjacent cells.  The grid is coarsened until
// it has at most ncap cells.  v: lowest x, y, z, highest x, y, z, largest
// radius, 1 if all positions are finite.  Positions that are not finite, or
// so far apart that their distance along an axis is not, have no grid (the
// ratio of such an extent to a cell would never fall below the limit).  With
// finite extents an infinite cell has one cell per axis, and a cell side
// grows from the smallest double to that in fewer than 4,096 rounds.
__host__ __device__ inline void choose_overlap_grid(const double (&v)[8], uint32_t ncap,
                                                    OverlapGrid& g) {
    double maxabs = 0.0, emax = 0.0, ext[3];
    bool finite = v[7] == 1.0;
    for (int d = 0; d < 3; ++d) {
        maxabs = fmax(maxabs, fmax(fabs(v[d]), fabs(v[3 + d])));
        ext[d] = v[3 + d] - v[d];
        emax = fmax(emax, ext[d]);
        finite = finite && __builtin_isfinite(ext[d]);
        g.lo[d] = v[d];
        g.n[d] = 1;
    }
    double h = 2.0 * v[6] * (1.0 + 1e-6) + 1e-12 * maxabs;
    if (!(h > 0.0)) h = emax > 0.0 ? emax : 1.0;
    g.use = 0;
    for (int round = 0; finite && !g.use && round < 4096; ++round) {
        uint64_t total = 1;
        for (int d = 0; d < 3; ++d) {
            g.n[d] = (int)fmin(ext[d] / h, (double)(1 << 20)) + 1;
            total *= (uint64_t)g.n[d];
        }
        if (total <= (uint64_t)ncap) g.use = 1;
        else h *= 1.5;
    }
    g.inv_h = 1.0 / h;
}

}  // namespace sphx

#endif
