// Output-side readers (overlap list, porosity profile) on the GPU.
#ifndef SPHERE_AMD_ANALYSIS_HPP_
#define SPHERE_AMD_ANALYSIS_HPP_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "overlap_grid.hpp"

namespace sphx {

// DEM::findOverlaps over one simulation's np particles (original order):
// with pairs == nullptr, counts[i] = overlapping j > i; else the pairs and
// overlaps written from offs[i] (exclusive prefix of counts).
hipError_t launch_overlaps(const double4* x, const double4* vel, uint32_t np, uint32_t* counts,
                           const uint64_t* offs, uint32_t* pairs, double* delta, hipStream_t s);

constexpr uint32_t OV_SLAB = 8;      // overlaps kept per particle
constexpr uint32_t OV_PPB = 64;      // particles per search workgroup
constexpr uint32_t OV_BOUNDS = 256;  // workgroups of the extremes

// Device arrays of the grid search for up to np particles.
struct OverlapWork {
    OverlapGrid* grid;
    double* bounds;       // OV_BOUNDS x 8 extremes
    uint32_t* key;        // cell per particle
    uint32_t* cj;         // index | fixed flag, in cell order
    double4* cx;          // position and radius, in cell order
    uint32_t* counts;     // overlaps with j > i
    uint32_t* slab_j;     // OV_SLAB partners per particle, ascending
    double* slab_d;
    uint32_t* cell_start; // ncap + 1
    uint32_t* cursor;
    uint32_t* cell_sum;
    unsigned long long* block_off;
    uint32_t ncap;        // most cells of the grid
};

// The arrays placed from `base` on; returns the bytes they take.
size_t overlap_work_layout(uint32_t np, char* base, OverlapWork* w);
// The search: afterwards w.grid holds whether the grid served and the total.
hipError_t launch_overlap_search(const double4* x, const double4* vel, uint32_t np,
                                 const OverlapWork& w, hipStream_t s);
// The list of a search, launch_overlaps' list; nothing if it exceeds cap.
hipError_t launch_overlap_emit(const double4* x, uint32_t np, const OverlapWork& w,
                               uint32_t* pairs, double* delta, uint64_t cap, hipStream_t s);

// DEM::porosity of z_slices slices of height h_slice (volume V_slice).
hipError_t launch_porosity(const double4* x, uint32_t np, int z_slices, double h_slice,
                           double V_slice, double* z_pos, double* porosity, hipStream_t s);

}  // namespace sphx

#endif
