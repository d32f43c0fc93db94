// Output-side readers of the step's state on the GPU: the pairwise overlap
// list of DEM::findOverlaps (src/sphere.cpp:674-724, behind `sphere
// --contacts`) and the porosity profile of DEM::porosity
// (src/sphere.cpp:486-592).  Both give the reference's results exactly: the
// same expressions in the same order, FP64 throughout.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "analysis.hpp"

namespace sphx {

namespace {

constexpr uint32_t TILE = 256;
constexpr double PI_D = 3.14159265358979323846;  // M_PI

// Pass 1 (pairs == nullptr): count, per i, the overlapping j > i.  Pass 2:
// write them from offs[i] on, in ascending j.  Workgroup b takes
// i in [256 b, 256 b + 256) and walks the j tiles from its own onwards
// through LDS.
__global__ __launch_bounds__(TILE) void k_overlaps(const double4* __restrict__ x,
                                                   const double4* __restrict__ vel, uint32_t np,
                                                   uint32_t* __restrict__ counts,
                                                   const uint64_t* __restrict__ offs,
                                                   uint32_t* __restrict__ pairs,
                                                   double* __restrict__ delta) {
    __shared__ double4 tx[TILE];
    __shared__ double tfix[TILE];
    const uint32_t i = blockIdx.x * TILE + threadIdx.x;
    const bool in = i < np;
    const double4 xi = in ? x[i] : make_double4(0.0, 0.0, 0.0, 0.0);
    const double fi = in ? vel[i].w : 1.0;
    uint32_t n = 0;
    uint64_t w = (in && pairs) ? offs[i] : 0;
    for (uint32_t t0 = blockIdx.x * TILE; t0 < np; t0 += TILE) {
        const uint32_t j = t0 + threadIdx.x;
        if (j < np) {
            tx[threadIdx.x] = x[j];
            tfix[threadIdx.x] = vel[j].w;
        }
        __syncthreads();
        const uint32_t m = np - t0 < TILE ? np - t0 : TILE;
        if (in && fi == 0) {
            for (uint32_t k = 0; k < m; ++k) {
                const uint32_t jj = t0 + k;
                if (jj <= i) continue;
                const double4 xj = tx[k];
                const double dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
                const double len = __builtin_sqrt(dx * dx + dy * dy + dz * dz);
                const double dn = len - (xi.w + xj.w);
                if (dn < 0.0 && tfix[k] == 0) {
                    if (pairs) {
                        pairs[2 * w] = i;
                        pairs[2 * w + 1] = jj;
                        delta[w] = dn;
                        ++w;
                    } else {
                        ++n;
                    }
                }
            }
        }
        __syncthreads();
    }
    if (in && !pairs) counts[i] = n;
}

// ---------------------------------------------------------------------------
// The overlap list through a uniform grid, without a host round trip before
// the list's length is known: extremes (many workgroups), the grid from them
// (one work-item), cell counts, their exclusive scan, the particles copied in
// cell order, the search (16 work-items per particle, up to OV_SLAB overlaps
// kept, ordered by j), the exclusive scan of the counts, and the list.  Bound
// by the launches on small simulations (ten of 3-5 us), by the search on
// large ones: 100,003 particles 0.10 ms in all, 47 us of it the search; one
// work-item per particle walking 27 cells through an index took 89 us for
// each of two passes and 55 on 5,000 (11 here), with the scans on the host
// between them.

constexpr uint32_t OV_WG = 256;
constexpr uint32_t OV_CELLS = 8;        // cells per work-item of the scans
constexpr uint32_t OV_LANES = 16;       // work-items per particle of the search
constexpr uint32_t OV_SEARCH_WG = 1024;
constexpr uint32_t OV_FIXED = 0x80000000u;
static_assert(OV_SEARCH_WG / OV_LANES == OV_PPB, "particles per search workgroup");

__global__ __launch_bounds__(OV_WG) void k_ov_bounds(const double4* __restrict__ x, uint32_t np,
                                                     OverlapWork w) {
    __shared__ double red[8][OV_WG / 64];
    const uint32_t stride = gridDim.x * OV_WG;
    for (uint32_t c = blockIdx.x * OV_WG + threadIdx.x; c <= w.ncap; c += stride) w.cell_start[c] = 0u;
    double v[8] = {__builtin_inf(), __builtin_inf(), __builtin_inf(), -__builtin_inf(),
                   -__builtin_inf(), -__builtin_inf(), 0.0, 1.0};
    for (uint32_t i = blockIdx.x * OV_WG + threadIdx.x; i < np; i += stride) {
        const double4 p = x[i];
        v[0] = fmin(v[0], p.x);
        v[1] = fmin(v[1], p.y);
        v[2] = fmin(v[2], p.z);
        v[3] = fmax(v[3], p.x);
        v[4] = fmax(v[4], p.y);
        v[5] = fmax(v[5], p.z);
        v[6] = fmax(v[6], p.w);
        if (!(__builtin_isfinite(p.x) && __builtin_isfinite(p.y) && __builtin_isfinite(p.z) &&
              __builtin_isfinite(p.w) && p.w >= 0.0))
            v[7] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        for (int h = 32; h > 0; h >>= 1) {
            const double o = __shfl_xor(v[k], h, 64);
            v[k] = (k < 3 || k == 7) ? fmin(v[k], o) : fmax(v[k], o);
        }
        if ((threadIdx.x & 63u) == 0) red[k][threadIdx.x / 64u] = v[k];
    }
    __syncthreads();
    if (threadIdx.x < 8) {
        const int k = (int)threadIdx.x;
        double r = red[k][0];
        for (uint32_t q = 1; q < OV_WG / 64; ++q)
            r = (k < 3 || k == 7) ? fmin(r, red[k][q]) : fmax(r, red[k][q]);
        w.bounds[blockIdx.x * 8 + k] = r;
    }
}

// The extremes of all blocks, and the grid chosen from them.
__global__ __launch_bounds__(64) void k_ov_grid(uint32_t nblocks, OverlapWork w) {
    const uint32_t lane = threadIdx.x;
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const bool lower = k < 3 || k == 7;
        v[k] = w.bounds[k];
        for (uint32_t b = lane; b < nblocks; b += 64)
            v[k] = lower ? fmin(v[k], w.bounds[b * 8 + k]) : fmax(v[k], w.bounds[b * 8 + k]);
        for (int h = 32; h > 0; h >>= 1) {
            const double o = __shfl_xor(v[k], h, 64);
            v[k] = lower ? fmin(v[k], o) : fmax(v[k], o);
        }
    }
    if (lane != 0) return;
    OverlapGrid g;
    g.total = 0;
    choose_overlap_grid(v, w.ncap, g);
    *w.grid = g;
}

__device__ __forceinline__ int grid_coord(double v, double lo, double inv_h, int n) {
    const double a = (v - lo) * inv_h;
    int c = a >= 0.0 ? (int)fmin(a, (double)(n - 1)) : 0;
    return c;
}

__device__ __forceinline__ uint32_t grid_key(const double4& p, const OverlapGrid& g) {
    const int ix = grid_coord(p.x, g.lo[0], g.inv_h, g.n[0]);
    const int iy = grid_coord(p.y, g.lo[1], g.inv_h, g.n[1]);
    const int iz = grid_coord(p.z, g.lo[2], g.inv_h, g.n[2]);
    return ((uint32_t)iz * (uint32_t)g.n[1] + (uint32_t)iy) * (uint32_t)g.n[0] + (uint32_t)ix;
}

// cell_start[c] holds cell c's count until the scan.
__global__ __launch_bounds__(OV_WG) void k_ov_bin(const double4* __restrict__ x, uint32_t np,
                                                  OverlapWork w) {
    const uint32_t i = blockIdx.x * OV_WG + threadIdx.x;
    if (!w.grid->use || i >= np) return;
    const uint32_t k = grid_key(x[i], *w.grid);
    w.key[i] = k;
    atomicAdd(&w.cell_start[k], 1u);
}

// Exclusive prefix of a value per work-item over the workgroup of T, and the
// workgroup's total.
template <typename V, uint32_t T>
__device__ __forceinline__ V block_exclusive(V v, V& total) {
    __shared__ V wave_sum[T / 64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x / 64u;
    V inc = v;
    for (uint32_t h = 1; h < 64; h <<= 1) {
        const V o = __shfl_up(inc, h, 64);
        if (lane >= h) inc += o;
    }
    if (lane == 63) wave_sum[wave] = inc;
    __syncthreads();
    V before = 0;
    total = 0;
#pragma unroll
    for (uint32_t k = 0; k < T / 64; ++k) {
        const V s = wave_sum[k];
        before += k < wave ? s : (V)0;
        total += s;
    }
    __syncthreads();
    return before + inc - v;
}

__global__ __launch_bounds__(OV_WG) void k_ov_cell_sums(OverlapWork w) {
    const uint32_t c0 = (blockIdx.x * OV_WG + threadIdx.x) * OV_CELLS;
    uint32_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < OV_CELLS; ++k)
        if (c0 + k <= w.ncap) s += w.cell_start[c0 + k];
    uint32_t total;
    (void)block_exclusive<uint32_t, OV_WG>(s, total);
    if (threadIdx.x == 0) w.cell_sum[blockIdx.x] = total;
}

// Exclusive scan in place of n block sums by one workgroup; returns the total.
template <typename V>
__device__ __forceinline__ V scan_sums(V* v, uint32_t n) {
    V run = 0;
    for (uint32_t b = 0; b < n; b += 1024) {
        const uint32_t k = b + threadIdx.x;
        const V s = k < n ? v[k] : (V)0;
        V total;
        const V pre = block_exclusive<V, 1024>(s, total);
        if (k < n) v[k] = run + pre;
        run += total;
    }
    return run;
}

__global__ __launch_bounds__(1024) void k_ov_scan_cells(OverlapWork w, uint32_t n) {
    (void)scan_sums(w.cell_sum, n);
}

__global__ __launch_bounds__(1024) void k_ov_scan_counts(OverlapWork w, uint32_t n) {
    const unsigned long long total = scan_sums(w.block_off, n);
    if (threadIdx.x == 0) w.grid->total = total;
}

__global__ __launch_bounds__(OV_WG) void k_ov_cells(OverlapWork w) {
    const uint32_t c0 = (blockIdx.x * OV_WG + threadIdx.x) * OV_CELLS;
    uint32_t n[OV_CELLS], s = 0;
#pragma unroll
    for (uint32_t k = 0; k < OV_CELLS; ++k) {
        n[k] = c0 + k <= w.ncap ? w.cell_start[c0 + k] : 0u;
        s += n[k];
    }
    uint32_t total;
    uint32_t run = block_exclusive<uint32_t, OV_WG>(s, total) + w.cell_sum[blockIdx.x];
#pragma unroll
    for (uint32_t k = 0; k < OV_CELLS; ++k) {
        if (c0 + k > w.ncap) continue;
        w.cell_start[c0 + k] = run;
        if (c0 + k < w.ncap) w.cursor[c0 + k] = run;
        run += n[k];
    }
}

// The particles in cell order (any order within a cell), with their index and
// whether they are fixed (fixvel other than 0 takes part in no overlap).
__global__ __launch_bounds__(OV_WG) void k_ov_scatter(const double4* __restrict__ x,
                                                      const double4* __restrict__ vel, uint32_t np,
                                                      OverlapWork w) {
    const uint32_t i = blockIdx.x * OV_WG + threadIdx.x;
    if (!w.grid->use || i >= np) return;
    const double4 xi = x[i];
    const bool fixed = !(vel[i].w == 0);
    const uint32_t pos = atomicAdd(&w.cursor[w.key[i]], 1u);
    w.cx[pos] = xi;
    w.cj[pos] = i | (fixed ? OV_FIXED : 0u);
}

// The cells of row r (0..8: z major, then y) around a particle: their range of
// particles in cell order.
__device__ __forceinline__ void cell_row(const OverlapWork& w, const OverlapGrid& g, int cx, int cy,
                                         int cz, int r, uint32_t& lo, uint32_t& hi) {
    const int y = cy + r % 3 - 1, z = cz + r / 3 - 1;
    lo = hi = 0;
    if (y < 0 || y >= g.n[1] || z < 0 || z >= g.n[2]) return;
    const int x0 = cx > 0 ? cx - 1 : 0, x1 = cx + 1 < g.n[0] ? cx + 1 : g.n[0] - 1;
    const uint32_t base = ((uint32_t)z * (uint32_t)g.n[1] + (uint32_t)y) * (uint32_t)g.n[0];
    lo = w.cell_start[base + (uint32_t)x0];
    hi = w.cell_start[base + (uint32_t)x1 + 1u];
}

// The overlap test of DEM::findOverlaps (src/sphere.cpp:694-716) for the
// j > i in the 27 cells around i's, a row of three cells (one range in cell
// order) per work-item.  The first OV_SLAB overlaps of a particle are kept in
// ascending j; a particle with more is searched again when the list is
// written.
__global__ __launch_bounds__(OV_SEARCH_WG) void k_ov_search(const double4* __restrict__ x,
                                                            const double4* __restrict__ vel,
                                                            uint32_t np, OverlapWork w) {
    __shared__ uint32_t s_n[OV_PPB];
    __shared__ uint32_t s_j[OV_PPB][OV_SLAB];
    __shared__ double s_d[OV_PPB][OV_SLAB];
    const OverlapGrid g = *w.grid;
    if (!g.use) return;
    const uint32_t t = threadIdx.x / OV_LANES, lane = threadIdx.x % OV_LANES;
    const uint32_t i = blockIdx.x * OV_PPB + t;
    if (lane == 0) s_n[t] = 0;
    __syncthreads();
    const bool in = i < np;
    if (in && lane < 9 && vel[i].w == 0) {
        const double4 xi = x[i];
        const int cx = grid_coord(xi.x, g.lo[0], g.inv_h, g.n[0]);
        const int cy = grid_coord(xi.y, g.lo[1], g.inv_h, g.n[1]);
        const int cz = grid_coord(xi.z, g.lo[2], g.inv_h, g.n[2]);
        uint32_t lo, hi;
        cell_row(w, g, cx, cy, cz, (int)lane, lo, hi);
        for (uint32_t k = lo; k < hi; k += 4) {
            uint32_t jj[4];
            double4 xj[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const uint32_t at = k + u < hi ? k + u : k;
                jj[u] = w.cj[at];
                xj[u] = w.cx[at];
            }
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                if (k + u >= hi || (jj[u] & OV_FIXED) || jj[u] <= i) continue;
                const double dx = xj[u].x - xi.x, dy = xj[u].y - xi.y, dz = xj[u].z - xi.z;
                const double len = __builtin_sqrt(dx * dx + dy * dy + dz * dz);
                const double dn = len - (xi.w + xj[u].w);
                if (dn < 0.0) {
                    const uint32_t at = atomicAdd(&s_n[t], 1u);
                    if (at < OV_SLAB) {
                        s_j[t][at] = jj[u];
                        s_d[t][at] = dn;
                    }
                }
            }
        }
    }
    __syncthreads();
    const uint32_t n = s_n[t];
    if (in && n <= OV_SLAB && lane < n) {
        const uint32_t j = s_j[t][lane];
        uint32_t rank = 0;
        for (uint32_t k = 0; k < n; ++k) rank += s_j[t][k] < j ? 1u : 0u;
        w.slab_j[(size_t)i * OV_SLAB + rank] = j;
        w.slab_d[(size_t)i * OV_SLAB + rank] = s_d[t][lane];
    }
    if (in && lane == 0) w.counts[i] = n;
    if (threadIdx.x < 64) {
        unsigned long long s = s_n[threadIdx.x];
        for (int h = 32; h > 0; h >>= 1) s += __shfl_xor(s, h, 64);
        if (threadIdx.x == 0) w.block_off[blockIdx.x] = s;
    }
}

// Orders the wavefront's memory accesses around it.
__device__ __forceinline__ void ov_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

// The n entries (partner in pairs[2 k + 1], overlap in delta[k]) sorted in
// place by partner, by one wavefront: a bitonic network whose first stage of
// each round compares mirrored places, so that every comparison puts the
// smaller entry first and places from n on need not exist.
__device__ void sort_entries(uint32_t* pairs, double* delta, uint32_t n, uint32_t lane) {
    auto exchange = [&](uint32_t a, uint32_t b) {
        if (b >= n) return;
        const uint32_t ja = pairs[2 * a + 1], jb = pairs[2 * b + 1];
        if (ja <= jb) return;
        const double da = delta[a], db = delta[b];
        pairs[2 * a + 1] = jb;
        pairs[2 * b + 1] = ja;
        delta[a] = db;
        delta[b] = da;
    };
    uint32_t half = 1;
    while (2 * half < n) half <<= 1;
    for (uint32_t k = 2; k <= 2 * half; k <<= 1) {
        for (uint32_t t = lane; t < half; t += 64) {
            const uint32_t base = t / (k / 2) * k, off = t % (k / 2);
            exchange(base + off, base + k - 1u - off);
        }
        ov_wave_sync();
        for (uint32_t d = k / 4; d > 0; d >>= 1) {
            for (uint32_t t = lane; t < half; t += 64) {
                const uint32_t a = t / d * (2 * d) + t % d;
                exchange(a, a + d);
            }
            ov_wave_sync();
        }
    }
}

// The list, one workgroup per search workgroup's particles.  Nothing is
// written when it is longer than `cap`.  The first wavefront copies the
// particles of up to OV_SLAB overlaps; the wavefronts then take the others in
// turn and search their 27 cells again, 64 candidates at a time, the overlaps
// found ordered in LDS by counting (up to OV_STAGE) or in place.  Calls on
// 20,000 particles, against one work-item inserting a particle's overlaps one
// by one: 4.7 overlaps a particle 0.48 / 0.64 ms, 18 1.1 / 3.6, 69 3.1 / 37, 253
// 18 / 482.  Bound by the candidates' loads and, on long lists, the download.
constexpr uint32_t OV_EMIT_WAVES = 4;
constexpr uint32_t OV_STAGE = 512;
__global__ __launch_bounds__(64 * OV_EMIT_WAVES) void k_ov_emit(
    const double4* __restrict__ x, uint32_t np, OverlapWork w, uint32_t* __restrict__ pairs,
    double* __restrict__ delta, unsigned long long cap) {
    static_assert(OV_PPB == 64, "a wavefront per block");
    __shared__ unsigned long long s_at[OV_PPB];
    __shared__ uint32_t s_n[OV_PPB];
    __shared__ unsigned long long s_many;
    __shared__ double s_d[OV_EMIT_WAVES][OV_STAGE];
    __shared__ uint32_t s_j[OV_EMIT_WAVES][OV_STAGE];
    const OverlapGrid g = *w.grid;
    if (!g.use || g.total > cap) return;
    const uint32_t lane = threadIdx.x % 64u, wave = threadIdx.x / 64u;
    if (wave == 0) {
        const uint32_t i = blockIdx.x * OV_PPB + lane;
        const uint32_t n = i < np ? w.counts[i] : 0u;
        uint32_t inc = n;
        for (uint32_t h = 1; h < 64; h <<= 1) {
            const uint32_t o = __shfl_up(inc, h, 64);
            if (lane >= h) inc += o;
        }
        const unsigned long long w0 = w.block_off[blockIdx.x] + (inc - n);
        const unsigned long long many = __ballot(n > OV_SLAB);
        s_at[lane] = w0;
        s_n[lane] = n;
        if (lane == 0) s_many = many;
        if (n <= OV_SLAB) {
            for (uint32_t k = 0; k < n; ++k) {
                pairs[2 * (w0 + k)] = i;
                pairs[2 * (w0 + k) + 1] = w.slab_j[(size_t)i * OV_SLAB + k];
                delta[w0 + k] = w.slab_d[(size_t)i * OV_SLAB + k];
            }
        }
    }
    __syncthreads();
    uint32_t turn = 0;
    for (unsigned long long many = s_many; many != 0; many &= many - 1ull, ++turn) {
        if (turn % OV_EMIT_WAVES != wave) continue;
        const uint32_t t = (uint32_t)__ffsll((long long)many) - 1u;
        const uint32_t i = blockIdx.x * OV_PPB + t, n = s_n[t];
        uint32_t* const out = pairs + 2 * s_at[t];
        double* const dout = delta + s_at[t];
        const double4 xi = x[i];
        const int cx = grid_coord(xi.x, g.lo[0], g.inv_h, g.n[0]);
        const int cy = grid_coord(xi.y, g.lo[1], g.inv_h, g.n[1]);
        const int cz = grid_coord(xi.z, g.lo[2], g.inv_h, g.n[2]);
        // The nine rows' ranges, numbered through.
        uint32_t lo = 0, hi = 0;
        if (lane < 9) cell_row(w, g, cx, cy, cz, (int)lane, lo, hi);
        uint32_t first[9], end[9], total = 0;
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            first[r] = (uint32_t)__builtin_amdgcn_readlane((int)lo, r) - total;
            total += (uint32_t)__builtin_amdgcn_readlane((int)(hi - lo), r);
            end[r] = total;
        }
        const bool staged = n <= OV_STAGE;
        uint32_t m = 0;
        for (uint32_t c0 = 0; c0 < total; c0 += 64) {
            const uint32_t c = c0 + lane;
            uint32_t at = first[0] + c;
#pragma unroll
            for (int r = 1; r < 9; ++r) at = c >= end[r - 1] ? first[r] + c : at;
            uint32_t j = OV_FIXED;
            double dn = 0.0;
            if (c < total) {
                j = w.cj[at];
                const double4 xj = w.cx[at];
                const double dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
                const double len = __builtin_sqrt(dx * dx + dy * dy + dz * dz);
                dn = len - (xi.w + xj.w);
            }
            const bool hit = !(j & OV_FIXED) && j > i && dn < 0.0;
            const unsigned long long hits = __ballot(hit);
            const uint32_t k = m + (uint32_t)__popcll(hits & ((1ull << lane) - 1ull));
            m += (uint32_t)__popcll(hits);
            if (hit && k < n) {
                if (staged) {
                    s_j[wave][k] = j;
                    s_d[wave][k] = dn;
                } else {
                    out[2 * k + 1] = j;
                    dout[k] = dn;
                }
            }
        }
        ov_wave_sync();
        if (staged) {
            for (uint32_t e = lane; e < n; e += 64) {
                const uint32_t j = s_j[wave][e];
                uint32_t rank = 0;
                for (uint32_t k = 0; k < n; ++k) rank += s_j[wave][k] < j ? 1u : 0u;
                out[2 * rank] = i;
                out[2 * rank + 1] = j;
                dout[rank] = s_d[wave][e];
            }
            ov_wave_sync();
        } else {
            sort_entries(out, dout, n, lane);
            for (uint32_t e = lane; e < n; e += 64) out[2 * e] = i;
        }
    }
}

__device__ __forceinline__ double spherical_cap(double h, double r) {
    return PI_D * h * h / 3.0 * (3.0 * r - h);
}

// The terms particle xi takes from the void of the slice [lo, hi), in the
// reference's order: at most two (the lower and the upper boundary).
// Returns how many.
__device__ __forceinline__ int slice_terms(const double4 xi, double lo, double hi, double& t0,
                                           double& t1) {
    const double zc = xi.z, r = xi.w;
    const double zl = zc - r, zh = zc + r;
    // Entirely above or below the slice: no condition holds (at zl == hi the
    // cap is zero).
    if (r >= 0.0 && (zl >= hi || zh < lo)) return 0;
    const double V_sphere = 4.0 / 3.0 * PI_D * r * r * r;
    if (lo <= zl && zh <= hi) {
        t0 = V_sphere;
        return 1;
    }
    double t[2] = {0.0, 0.0};
    bool low = true, up = true;
    if (lo >= zc && lo <= zh)
        t[0] = spherical_cap(zh - lo, r);
    else if (lo < zc && lo > zl)
        t[0] = V_sphere + spherical_cap(lo - zl, r);
    else
        low = false;
    if (hi <= zc && hi >= zl)
        t[1] = spherical_cap(hi - zl, r);
    else if (hi > zc && hi < zh)
        t[1] = V_sphere + spherical_cap(zh - hi, r);
    else
        up = false;
    t0 = low ? t[0] : t[1];
    t1 = t[1];
    return (low ? 1 : 0) + (up ? 1 : 0);
}

// One work-item per slice, the particles in index order (the reference's
// serial subtraction per slice).
__global__ __launch_bounds__(64) void k_porosity(const double4* __restrict__ x, uint32_t np,
                                                 int z_slices, double h_slice, double V_slice,
                                                 double* __restrict__ z_pos,
                                                 double* __restrict__ porosity) {
    const int iz = (int)(blockIdx.x * 64 + threadIdx.x);
    if (iz >= z_slices) return;
    double V_void = V_slice;
    const double lo = iz * h_slice;
    const double hi = lo + h_slice;
    for (uint32_t i = 0; i < np; ++i) {
        double t0, t1;
        const int n = slice_terms(x[i], lo, hi, t0, t1);
        if (n > 0) V_void -= t0;
        if (n > 1) V_void -= t1;
    }
    z_pos[iz] = lo + 0.5 * h_slice;
    porosity[iz] = V_void / V_slice;
}

// One workgroup per slice.  The subtraction is a serial chain in particle
// order (each slice's result is rounded term by term), so the terms are
// formed apart from it: the wavefronts after the first evaluate a tile of
// particles each round and leave the terms in LDS, compacted in particle
// order, while the first work-item subtracts the tiles before, sixteen terms
// read ahead of the adds.  Bound by the rounds (about 3.6 us for 1,920
// particles) and, where a slice holds many particles, by the chain of adds.
// One work-item per slice took 0.23-0.29 us a particle for any number of
// slices: 100,003 particles in 12 slices 29.4 ms there, 0.19 ms here; 5,000 in
// 10 slices 1.26 ms and 0.014 ms.
constexpr uint32_t PW = 16;                // wavefronts
constexpr uint32_t PTILE = 64 * (PW - 1);  // particles per tile
constexpr uint32_t PU = 2;                 // tiles per round
__global__ __launch_bounds__(64 * PW) void k_porosity_slice(const double4* __restrict__ x,
                                                            uint32_t np, double h_slice,
                                                            double V_slice,
                                                            double* __restrict__ z_pos,
                                                            double* __restrict__ porosity) {
    __shared__ __align__(16) double term[2 * PU * PTILE + 32];
    __shared__ uint32_t cnt[2][PU * PW];
    const int iz = (int)blockIdx.x;
    const double lo = iz * h_slice;
    const double hi = lo + h_slice;
    const uint32_t wave = threadIdx.x / 64u, lane = threadIdx.x % 64u;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t rounds = (np + PU * PTILE - 1) / (PU * PTILE);
    double V_void = V_slice;
    // This round's particles, i and i + PTILE (wave > 0).
    uint32_t i = threadIdx.x - 64u;
    double4 xi[PU];
#pragma unroll
    for (uint32_t u = 0; u < PU; ++u) {
        xi[u] = make_double4(0.0, 0.0, 0.0, 0.0);
        if (wave > 0 && i + u * PTILE < np) xi[u] = x[i + u * PTILE];
    }
    if (threadIdx.x < 2 * PU * PW) cnt[threadIdx.x / (PU * PW)][threadIdx.x % (PU * PW)] = 0;
    __syncthreads();
    // Round r evaluates its tiles and subtracts those of round r - 1.
    for (uint32_t r = 0; r <= rounds; ++r) {
        const uint32_t h = r & 1u;
        double t0[PU], t1[PU];
        int n[PU];
        uint32_t at[PU];
#pragma unroll
        for (uint32_t u = 0; u < PU; ++u) n[u] = 0;
        if (wave > 0) {
#pragma unroll
            for (uint32_t u = 0; u < PU; ++u) {
                if (i + u * PTILE < np) n[u] = slice_terms(xi[u], lo, hi, t0[u], t1[u]);
                const uint64_t b0 = __ballot(n[u] > 0), b1 = __ballot(n[u] > 1);
                at[u] = (uint32_t)(__popcll(b0 & below) + __popcll(b1 & below));
                if (lane == 0)
                    cnt[h][u * PW + wave] = (uint32_t)(__popcll(b0) + __popcll(b1));
            }
            i += PU * PTILE;
#pragma unroll
            for (uint32_t u = 0; u < PU; ++u)
                if (i + u * PTILE < np) xi[u] = x[i + u * PTILE];
        } else if (threadIdx.x == 0 && r > 0) {
            uint32_t m = 0;
            for (uint32_t w = 0; w < PU * PW; ++w) m += cnt[h ^ 1u][w];
            double a[16], b[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) a[k] = term[k];
            uint32_t j = 0;
            for (; j + 32 <= m; j += 32) {
#pragma unroll
                for (int k = 0; k < 16; ++k) b[k] = term[j + 16 + k];
#pragma unroll
                for (int k = 0; k < 16; ++k) V_void -= a[k];
#pragma unroll
                for (int k = 0; k < 16; ++k) a[k] = term[j + 32 + k];
#pragma unroll
                for (int k = 0; k < 16; ++k) V_void -= b[k];
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) b[k] = term[j + 16 + k];
#pragma unroll
            for (int k = 0; k < 16; ++k)
                if (j + k < m) V_void -= a[k];
#pragma unroll
            for (int k = 0; k < 16; ++k)
                if (j + 16 + k < m) V_void -= b[k];
        }
        __syncthreads();
#pragma unroll
        for (uint32_t u = 0; u < PU; ++u) {
            if (n[u] > 0) {
                uint32_t off = at[u];
                for (uint32_t w = 0; w < u * PW + wave; ++w) off += cnt[h][w];
                term[off] = t0[u];
                if (n[u] > 1) term[off + 1] = t1[u];
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        z_pos[iz] = lo + 0.5 * h_slice;
        porosity[iz] = V_void / V_slice;
    }
}

}  // namespace

hipError_t launch_overlaps(const double4* x, const double4* vel, uint32_t np, uint32_t* counts,
                           const uint64_t* offs, uint32_t* pairs, double* delta, hipStream_t s) {
    if (np == 0) return hipSuccess;
    hipLaunchKernelGGL(k_overlaps, dim3((np + TILE - 1) / TILE), dim3(TILE), 0, s, x, vel, np,
                       counts, offs, pairs, delta);
    return hipGetLastError();
}

size_t overlap_work_layout(uint32_t np, char* base, OverlapWork* w) {
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char* p = base + off;
        off += up(bytes);
        return p;
    };
    w->ncap = np < 2048u ? 4096u : 2u * np;
    const size_t cells = w->ncap + 1u;
    w->grid = (OverlapGrid*)take(sizeof(OverlapGrid));
    w->bounds = (double*)take(OV_BOUNDS * 64);
    w->key = (uint32_t*)take((size_t)np * 4);
    w->cj = (uint32_t*)take((size_t)np * 4);
    w->cx = (double4*)take((size_t)np * 32);
    w->counts = (uint32_t*)take((size_t)np * 4);
    w->slab_j = (uint32_t*)take((size_t)np * OV_SLAB * 4);
    w->slab_d = (double*)take((size_t)np * OV_SLAB * 8);
    w->cell_start = (uint32_t*)take(cells * 4);
    w->cursor = (uint32_t*)take(cells * 4);
    w->cell_sum = (uint32_t*)take((cells / (OV_WG * OV_CELLS) + 1) * 4);
    w->block_off = (unsigned long long*)take((np / OV_PPB + 1) * 8);
    return off;
}

hipError_t launch_overlap_search(const double4* x, const double4* vel, uint32_t np,
                                 const OverlapWork& w, hipStream_t s) {
    const uint32_t nb = (np + OV_WG - 1) / OV_WG;
    const uint32_t bounds = nb < OV_BOUNDS ? nb : OV_BOUNDS;
    const uint32_t cb = (w.ncap + 1u + OV_WG * OV_CELLS - 1) / (OV_WG * OV_CELLS);
    const uint32_t sb = (np + OV_PPB - 1) / OV_PPB;
    hipLaunchKernelGGL(k_ov_bounds, dim3(bounds), dim3(OV_WG), 0, s, x, np, w);
    hipLaunchKernelGGL(k_ov_grid, dim3(1), dim3(64), 0, s, bounds, w);
    hipLaunchKernelGGL(k_ov_bin, dim3(nb), dim3(OV_WG), 0, s, x, np, w);
    hipLaunchKernelGGL(k_ov_cell_sums, dim3(cb), dim3(OV_WG), 0, s, w);
    hipLaunchKernelGGL(k_ov_scan_cells, dim3(1), dim3(1024), 0, s, w, cb);
    hipLaunchKernelGGL(k_ov_cells, dim3(cb), dim3(OV_WG), 0, s, w);
    hipLaunchKernelGGL(k_ov_scatter, dim3(nb), dim3(OV_WG), 0, s, x, vel, np, w);
    hipLaunchKernelGGL(k_ov_search, dim3(sb), dim3(OV_SEARCH_WG), 0, s, x, vel, np, w);
    hipLaunchKernelGGL(k_ov_scan_counts, dim3(1), dim3(1024), 0, s, w, sb);
    return hipGetLastError();
}

hipError_t launch_overlap_emit(const double4* x, uint32_t np, const OverlapWork& w,
                               uint32_t* pairs, double* delta, uint64_t cap, hipStream_t s) {
    hipLaunchKernelGGL(k_ov_emit, dim3((np + OV_PPB - 1) / OV_PPB), dim3(64 * OV_EMIT_WAVES), 0, s, x,
                       np, w, pairs, delta, (unsigned long long)cap);
    return hipGetLastError();
}

hipError_t launch_porosity(const double4* x, uint32_t np, int z_slices, double h_slice,
                           double V_slice, double* z_pos, double* porosity, hipStream_t s) {
    // A workgroup per slice pays while the chip holds them in few rounds (512
    // at a time).  5,000 particles: 0.36 ms against 1.11 at 8,192 slices, the
    // same at 32,768; 500 particles: 0.14 against 0.16 at 8,192; 50 particles:
    // equal at 1,000, 0.09 against 0.06 at 8,192.
    if (z_slices <= 1024 || (z_slices <= 8192 && (uint32_t)z_slices / 16u <= np))
        hipLaunchKernelGGL(k_porosity_slice, dim3(z_slices), dim3(64 * PW), 0, s, x, np, h_slice,
                           V_slice, z_pos, porosity);
    else
        hipLaunchKernelGGL(k_porosity, dim3((z_slices + 63) / 64), dim3(64), 0, s, x, np,
                           z_slices, h_slice, V_slice, z_pos, porosity);
    return hipGetLastError();
}

}  // namespace sphx
