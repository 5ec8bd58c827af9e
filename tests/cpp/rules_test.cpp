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
    check(arc::serial_cut(65536, 2048, 512) && !arc::serial_cut(65536, 2048, 511), "the tiles' line");
    check(arc::serial_cut(65536, 2000000000, 2000000000), "many tiles");
    if (!failures) std::printf("launch rules hold\n");
    return failures ? 1 : 0;
}
