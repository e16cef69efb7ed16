// Prints, for populations of 2, 4 and 8 bytes and rows of 1 to 80 segments: bytes, flagged blocks, segments,
// tile width, and for a cap of 3, 4 and 5 waves a SIMD the LDS of a block.
#include "launch_rules.hpp"

#include <cstdio>

int main() {
    for (size_t elem = 2; elem <= 8; elem *= 2)
        for (int flagged = 0; flagged <= 1; ++flagged)
            for (uint32_t s = 1; s <= 80; ++s) {
                const uint32_t w = cfd_hip::step_tile_width(s, elem, flagged != 0);
                const long threads = w < 256 ? 256 : w;  // narrow tiles take several rows
                std::printf("%zu %d %u %u", elem, flagged, s, w);
                for (long waves = 3; waves <= 5; ++waves) std::printf(" %u", cfd_hip::occupancy_lds(waves, threads));
                std::printf("\n");
            }
}
