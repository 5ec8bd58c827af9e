// Rules by which a call takes one kernel or another.  Host code without the
// device runtime, so that they can be run on the CPU.
#pragma once

namespace arc {

// The clustered antiradiance's list entries filed into LDS per pass.  The
// setting 1536 is the default and leaves it to the kernel: staged (the cone model
// over Lambertian materials) wants 110 registers, and with 3072 entries, 34 KB,
// four waves per SIMD are what the LDS allows and it gets them; with fewer it is
// held to 96 and spills 17 (1920x1080 pixels, 1M AVPLs: 0.9 GB of traffic and 26.2
// ms a frame against 2.0 GB and 28.0 with 1536).  The other models cost alike.
constexpr int kAntiBlock = 1536, kAntiBlockStaged = 3072;
constexpr int anti_block(int setting, bool staged) {
    return setting == kAntiBlock && staged ? kAntiBlockStaged : setting;
}

// Whether a moment cut's tiles are all cut serially, a node at a time, with the
// sums in the same wave, the heaviest first by the last cut's costs.  A tile that
// meets its budget is decided twice by the kernel that takes 64 nodes at a time,
// so the line lies where most tiles would: at budgets below 8192, and, where the
// last cut of this setting says so (`bad`: tiles that met their budget, or found
// a pool full that does not grow), from a quarter of the tiles on.  Below 2048
// tiles a serial wave's latency is what counts, and the other kernel's is shorter.
// Milliseconds a frame, serial and decided, over 20000, 60000 and 250001 AVPLs:
//                 200x120        640x360        1283x719
//   budget  4096  0.91   1.12    1.63   2.02     4.49    6.41
//           8192  1.63   1.30    2.22   2.83     6.82    8.65
//          12000  1.94   0.66    2.82   3.88     8.5    10.0   (a quarter and 30 % of the tiles, none of 200x120)
//          16384  1.94   0.66    3.30   2.83     9.2     9.2   (1.5 % and 13 %)
constexpr int kSerialBudget = 8192, kSerialMinTiles = 2048;
constexpr bool serial_cut(int budget, int tiles, int bad) {
    return budget < kSerialBudget || (tiles >= kSerialMinTiles && 4LL * bad >= tiles);
}

}  // namespace arc
