// Prints which of a run of uses go without resident launches; argv[1]: for
// each use that is tried, in turn, '-' it gave up, '+' it ended well
#include <cstdio>
#include <cstring>

#include "backoff.hpp"

int main(int, char** argv)
{
    ins::Backoff b;
    int tried = 0, skipped = 0;
    const char* what = argv[1];
    while (what[tried]) {
        if (b.skip()) {
            skipped++;
            continue;
        }
        std::printf("%d ", skipped);
        skipped = 0;
        if (what[tried++] == '-') b.gave_up();
        else b.ended_well();
    }
    std::printf("\n");
    return 0;
}
