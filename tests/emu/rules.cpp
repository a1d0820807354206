// rules.cpp -- TEST ONLY.  Prints what the library's dispatch rules say:
//   rules xdrop <items> <X> <gap> <xd_coop> <xd_wave>
// -> "small16 split sorted all_band".
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../pastis_amd/csrc/pa_internal.h"

int main(int argc, char **argv)
{
    if (argc == 7 && std::strcmp(argv[1], "xdrop") == 0) {
        const pa::XdRoute r =
            pa::xd_route(std::strtoull(argv[2], nullptr, 10), std::atoi(argv[3]),
                         std::atoi(argv[4]), std::atoi(argv[5]),
                         std::atoi(argv[6]));
        std::printf("%d %d %d %d\n", r.small16, r.split, r.sorted, r.all_band);
        return 0;
    }
    return 2;
}
