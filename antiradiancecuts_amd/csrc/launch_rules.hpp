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

}  // namespace arc
