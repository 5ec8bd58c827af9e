// The rules of csrc/launch_rules.hpp.  Prints the first that does not hold and
// ends with 1.
#include <cstdio>
#include <initializer_list>

#include "launch_rules.hpp"

namespace {
int failures = 0;
void check(bool ok, const char* what) {
    if (!ok && failures++ == 0) std::printf("does not hold: %s\n", what);
}
}  // namespace

int main() {
    // a caller that sets the launch shape's defaults gets what one that sets nothing gets
    check(arc::anti_block(1536, true) == 3072, "the default block of the staged walk");
    check(arc::anti_block(1536, false) == 1536, "the default block of the others");
    for (int staged = 0; staged < 2; ++staged)
        for (int set : {768, 3072}) check(arc::anti_block(set, staged) == set, "a block that was set");
    check(arc::serial_cut(8191, 100, 0) && !arc::serial_cut(8192, 100, 0), "the budget's line");
    check(!arc::serial_cut(65536, 2047, 2047), "few tiles are not cut serially");
    check(arc::serial_cut(65536, 2048, 410) && !arc::serial_cut(65536, 2048, 409) && arc::serial_cut(65536, 16383, 3277) &&
              !arc::serial_cut(65536, 16384, 5461) && arc::serial_cut(65536, 16384, 5462) &&
              arc::serial_cut(65536, 16383, 547, true) && !arc::serial_cut(65536, 16383, 546, true) &&
              !arc::serial_cut(65536, 16384, 5461, true) && !arc::serial_cut(65536, 2047, 2047, true),
          "the tiles' line");
    check(arc::serial_cut(65536, 2000000000, 2000000000), "many tiles");
    using arc::Rays;
    check(arc::rays_together(Rays::kCamera, 200000, 512) && !arc::rays_together(Rays::kCamera, 199999, 512) &&
              !arc::rays_together(Rays::kCamera, 33177600, 513),
          "the lines of a camera's rays");
    check(arc::rays_together(Rays::kAny, 200000, 16) && !arc::rays_together(Rays::kAny, 199999, 16) &&
              !arc::rays_together(Rays::kAny, 2147483647, 17),
          "the lines of the caller's rays");
    check(arc::rays_together(Rays::kPaths, 100000, 62) && !arc::rays_together(Rays::kPaths, 100000, 63) &&
              !arc::rays_together(Rays::kPaths, 99999, 1) && !arc::rays_together(Rays::kPaths, 2147483647, 513) &&
              arc::rays_together(Rays::kPaths, 819200, 512) && !arc::rays_together(Rays::kPaths, 2147483647, 2147483647),
          "the lines of a shoot's paths");
    if (!failures) std::printf("launch rules hold\n");
    return failures ? 1 : 0;
}
