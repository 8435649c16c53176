// Bands per launch of the density pass, by what is held and free.
#include <cstdio>

#include "rho_bands.hpp"

#define EXPECT(c)                                       \
    do {                                                \
        if (!(c)) {                                     \
            std::printf("line %d: %s\n", __LINE__, #c); \
            return 1;                                   \
        }                                               \
    } while (0)

int main() {
    using apw::rho_bands;
    const std::size_t MIB = 1u << 20, GIB = 1u << 30, lots = 200 * GIB;
    EXPECT(rho_bands(432, 4, 42 * MIB, 0, lots) == 73);          // 3 GiB of 160^3 bands
    EXPECT(rho_bands(40, 4, 42 * MIB, 0, lots) == 40);           // no more than there are
    EXPECT(rho_bands(432, 4, 42 * MIB, 0, 2 * GIB) == 24);       // half of what is free
    EXPECT(rho_bands(432, 4, 42 * MIB, 73 * 42 * MIB, 0) == 73); // what is held needs no more
    EXPECT(rho_bands(432, 4, 42 * MIB, 30 * 42 * MIB, 2 * GIB) == 30);
    EXPECT(rho_bands(432, 4, 42 * MIB, 0, 300 * MIB) == 4);      // H|psi>'s chunk, its own buffers
    EXPECT(rho_bands(3, 4, 42 * MIB, 0, 300 * MIB) == 3);
    EXPECT(rho_bands(432, 1, 4 * GIB, 0, lots) == 1);            // a band past the bound
    EXPECT(rho_bands(432, 1, 400 * MIB, 0, lots) == 7);          // 320^3: not sixteen
    EXPECT(rho_bands(100000, 256, 100000, 0, lots) == 4096);     // a grid dimension
    std::printf("ok\n");
    return 0;
}
