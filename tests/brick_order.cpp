// Prints the brick order of a grid (csrc/brick.h): L1 L2 L3, then a first rank,
// a stride and a count; one line per rank with the cell.
#include <cstdio>
#include <cstdlib>

#include "brick.h"

int main(int argc, char** argv)
{
    if (argc != 7) return 2;
    long long a[6];
    for (int i = 0; i < 6; ++i) a[i] = std::atoll(argv[i + 1]);
    for (long long k = 0; k < a[5]; ++k) {
        const long long r = a[3] + k * a[4];
        std::printf("%lld %d\n", r, sph::brick_cell((int)a[0], (int)a[1], (int)a[2], (int)r));
    }
    return 0;
}
