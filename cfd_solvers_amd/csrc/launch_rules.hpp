// launch_rules.hpp -- tile width and occupancy cap of the step kernels (host arithmetic only).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace cfd_hip {

// Width of a step tile on rows of `segments` 64-cell segments, with populations of `elem` bytes;
// `flagged_blocks`: a lattice with flags in row blocks.  Neighbouring tiles of a row share cache lines at
// their common edge (populations are read and written at x - 1, x and x + 1), so a tile spans the row where
// a block can (256^3 cavity: 454 us a step with 256-wide tiles, 484 with 128, 563 with 64), and it launches
// no whole wavefronts beyond the row's end: five to seven segments are one tile of just that width (320 x
// 150 x 141 FP32 cavity: 185 us a step against 216 with 256-wide tiles, 384 wide 225 against 256, 440 wide
// 260 against 275; in plain planes 320 x 640 x 400 2.29 ms against 2.90, 440 x 512 x 300 2.04 against
// 2.17).  Up to four segments take the 256-thread tile (192 wide, 192^3 FP32: 191 us with a 192-thread
// tile, 187 with 256).
//
// Eight segments are two 256-wide tiles or one of 512.  In FP32 a 512-thread block leaves the occupancy cap
// only steps of two waves a SIMD: two tiles (512 x 200 x 160 cavity 438 us against 453, D3Q27 512 x 160 x
// 100 300 against 319, D3Q27 512^2 x 200 in plain planes 1.90 ms against 2.21; elsewhere equal to 3 %).
// FP16S is not capped that low: one tile is ahead on periodic lattices (512 x 256^2 459 us against 500,
// 512^3 1.88 ms against 2.13) and in plain planes (512^3 cavity 1.95 against 1.98), two tiles with flags in
// row blocks (512 x 256^2 cavity 468 us against 490, out of place for the adjoint 587 against 636).
//
// Longer rows take the width that launches least, 256 unless that adds more than 1/8 to the row (2-D, 1100
// wide: 25.4 us with 256, 26.1-27.4 with 320-512).  FP64 needs the registers of a 256-thread block, so its
// rows of more than four segments take 128 where that launches fewer (260 wide: 309 us against 405).
inline uint32_t step_tile_width(uint32_t segments, size_t elem, bool flagged_blocks) {
    const auto launched = [segments](uint32_t w) { return (segments + w - 1U) / w * w; };
    if (segments <= 4U) return segments <= 1U ? 64U : segments == 2U ? 128U : 256U;
    if (elem == 8) return launched(2U) < launched(4U) ? 128U : 256U;
    if (segments == 8U) return elem == 2 && !flagged_blocks ? 512U : 256U;
    if (segments <= 7U) return 64U * segments;
    if (launched(4U) * 8U <= segments * 9U) return 256U;
    uint32_t best = 4U;
    for (uint32_t w = 5U; w <= 7U; ++w)
        if (launched(w) < launched(best)) best = w;
    return 64U * best;
}

// LDS per block (160 KiB a CU) that caps the resident wavefronts of a SIMD at about `waves` (3 to 7; other
// values: no cap), as near as whole blocks come: a block of `threads` threads is threads / 256 wavefronts
// on each SIMD.  In 320- to 448-thread blocks the nearest cap was within 3 % of the best of all caps (FP32
// D3Q19 and D3Q27, row blocks and plain planes, bounded and periodic).
inline uint32_t occupancy_lds(long waves, long threads) {
    if (waves < 3 || waves >= 8) return 0U;
    const long blocks = std::max(1L, (waves * 256 + threads / 2) / threads);
    return static_cast<uint32_t>(std::min(163840 / blocks - 1024, 65536L));
}

}  // namespace cfd_hip
