// Bands per launch of the density pass (host code).
#pragma once

#include <algorithm>
#include <cstddef>

namespace apw {

constexpr std::size_t RHO_BYTES = (std::size_t)3 << 30;   // S and X of one launch
constexpr int RHO_BANDS = 4096;                           // and its band index, a grid dimension

// Bands that a launch takes in a workspace for held bytes now, which may grow into half of the free
// memory: the other half stays for what the call and the caller allocate next, and no allocation
// is tried that would fail.  At most chunk bands: the Hamiltonian's own buffers serve (chunk of them).
inline int rho_bands(int nbands, int chunk, std::size_t band_bytes, std::size_t held, std::size_t free_bytes) {
    const std::size_t bytes = std::min(RHO_BYTES, std::max(held, free_bytes / 2));
    const std::size_t n = std::min({bytes / band_bytes, (std::size_t)RHO_BANDS, (std::size_t)nbands});
    return (int)n > chunk ? (int)n : std::min(nbands, chunk);
}

}  // namespace apw
