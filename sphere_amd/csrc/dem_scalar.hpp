// Scalar reads of what is uniform over a launch.
#ifndef SPHERE_AMD_DEM_SCALAR_HPP_
#define SPHERE_AMD_DEM_SCALAR_HPP_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sphx {

// Scalar loads of one word of each 64-byte line of [ptr, ptr + BYTES), all in
// flight together.  The compiler reads kernel arguments, parameters and loop
// state where they are used, each read waiting for a line the scalar cache
// has not seen in this launch; after one such pass they all hit.  Measured
// with the contact pass's first loads ungated (no chunk map for one
// simulation, list entries and position requested with the original index):
// contact 13.3 -> 11.4 us on 601 particles, 26.2 -> 23.9 on 1e5 (beds tiled from
// settled cells); integration
// 6.2 -> 5.8 and walls 3.3 -> 3.0 on 601.
typedef const __attribute__((address_space(4))) void cvoid;
template <uint32_t BYTES, uint32_t BYTES2 = 0>
__device__ __forceinline__ void touch_lines(cvoid* ptr, cvoid* ptr2 = nullptr) {
    // A structure need not start on a line: its last word is read as well.
    constexpr uint32_t n = (BYTES + 63) / 64 + 1, n2 = BYTES2 ? (BYTES2 + 63) / 64 + 1 : 0;
    static_assert(n + n2 <= 12, "at most 12 lines");
    const auto* w = (const __attribute__((address_space(4))) uint32_t*)ptr;
    const auto* w2 = (const __attribute__((address_space(4))) uint32_t*)ptr2;
    uint32_t v[12];
#pragma unroll
    for (uint32_t k = 0; k < 12; ++k) {
        const uint32_t at = 16 * k < (BYTES - 4) / 4 ? 16 * k : (BYTES - 4) / 4;
        v[k] = w[at];
        if constexpr (BYTES2 > 0) {
            const uint32_t k2 = k < n ? 0 : k - n;
            const uint32_t at2 = 16 * k2 < (BYTES2 - 4) / 4 ? 16 * k2 : (BYTES2 - 4) / 4;
            if (k >= n) v[k] = w2[at2];
        }
    }
    asm volatile("" ::"s"(v[0]), "s"(v[1]), "s"(v[2]), "s"(v[3]), "s"(v[4]), "s"(v[5]), "s"(v[6]),
                 "s"(v[7]), "s"(v[8]), "s"(v[9]), "s"(v[10]), "s"(v[11]));
}

}  // namespace sphx

#endif
