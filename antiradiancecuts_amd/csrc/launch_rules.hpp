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
// so the line lies where many tiles would: at budgets below 8192, and, where the
// last cut of this setting says so (`bad`: tiles that met their budget, or found
// a pool full that does not grow), from a third of the tiles on, or from a fifth
// where there are fewer than 16384, four rounds of the chip's waves: such tiles
// are then the end of the launch, and with the expansion criterion, whose few
// large tiles stand out more, from a 30th.  Below 2048 tiles a serial wave's latency is what
// counts, and the other kernel's is shorter.  Milliseconds a frame, serial and
// decided, and the share of such tiles, over 20000, 60000, 250001 and 1000000 AVPLs:
//                 200x120       640x360             1283x719            1920x1080
//   budget  4096  0.86  1.12    1.53  2.02          4.50  6.41
//           8192  1.53  1.27    2.08  2.83  0.65    6.84  8.67  0.44    22.3  23.6  0.37
//          12000  1.94  0.65    2.50  3.73  0.24    8.25  9.95  0.30    25.4  24.5  0.33
//          14000                2.65  3.03  0.10    8.64  9.83  0.21    26.4  24.1  0.25
//          16384                2.93  2.76  0.01    9.10  9.49  0.13    27.3  25.0  0.21
// expansion  8192               (30 tiles: 2.49)    6.24  6.95  0.068   19.9  17.9  0.14
//           10000                                   6.32  7.07  0.038   20.3  17.0  0.11
//           14000                                   6.39  6.11  0.010
// and at 65536 with nodes of up to 128 exact (bound 0.0045, floor 4)
//                                                  15.7  15.2   0.16
constexpr int kSerialBudget = 8192, kSerialMinTiles = 2048, kSerialFewTiles = 16384;
constexpr bool serial_cut(int budget, int tiles, int bad, bool expansion = false) {
    const long long line = tiles >= kSerialFewTiles ? 3 : expansion ? 30 : 5;
    return budget < kSerialBudget || (tiles >= kSerialMinTiles && line * bad >= tiles);
}

// Whether a wave's 64 rays go through the triangle tree together, one ray a lane,
// or eight by eight, each ray in eight lanes of its own.  Together a node costs
// the wave 14 instructions a child however few of the rays enter it, so that pays
// where a tree has few nodes for the rays, and with fewer rays the chip is not
// full.  A camera's rays enter much the same nodes; a path's go everywhere, but
// those that leave one light start alike and a long shoot takes many; rays from
// the caller may be in any order.  Microseconds, together and in groups of eight:
//   nodes                  5          31           100           413          1058
//   pixels  640x360     10   13    18    26     22    29     43     55     62     86
//         3840x2160     74  325   231   710    266   783    554   1510    854   2427
//   paths      1e5     388  693   570   733   1046   813   2691    992   4311   1074
//              5e5     995 2589  1123  2778   1640  3121   4012   3663   6918   3924
//              2e6    2786 9825  2922 10538   4039 11554  10999  13792  19540  14744
//   rays, at random
//              1e5      12   11    54    22    124    34    356     54    705     75
//              1e6      36   79   181   156    413   253   1162    386   2271    514
// A picture of more nodes than that would gain too as long as its neighbouring
// pixels see the same triangles; where they do not, it is the rays at random.
enum class Rays { kCamera, kPaths, kAny };
constexpr int kTogetherRays = 200000, kTogetherPaths = 100000, kPathsPerNode = 1600;
constexpr bool rays_together(Rays kind, long long rays, int nodes) {
    if (kind == Rays::kPaths) return rays >= kTogetherPaths && rays >= (long long)kPathsPerNode * nodes && nodes <= 512;
    return rays >= kTogetherRays && nodes <= (kind == Rays::kCamera ? 512 : 16);
}

}  // namespace arc
