// Host check of launch limits (dumses-hybrid_amd/csrc/dmx_tiling.h): over the
// thin and long domains that dmx_create accepts, a face/edge stage launched as
// one block per Riemann problem stays within 65535 blocks along z, whatever its
// line in blocks.  Prints "bad 0" on success.
#include <cstdio>
#include <initializer_list>

#include "dmx_tiling.h"

using namespace dmx;

int main()
{
    long bad = 0, split = 0, whole = 0;
    for (int nx : {3, 4, 31, 60, 61, 124, 200, 700})
        for (int ny : {3, 4, 7, 8, 40})
            for (int nz = 3; nz <= 20000; nz += nz < 40 ? 1 : 37)
                for (long long most : {6000LL, 16384LL, 1000000LL}) {
                    const long long x = (nx + 4 + 63) / 64, y = (ny + 1 + 3) / 4, z = nz + 1;
                    const bool s = split_fits(x, y, z, most);
                    if (s && (6 * z > 65535 || x * y * z > most)) {
                        if (bad++ < 5) printf("bad launch: n %d %d %d, %lld blocks along z\n", nx, ny, nz, 6 * z);
                    }
                    if (!s && 6 * z <= 65535 && x * y * z <= most) bad++;
                    s ? split++ : whole++;
                }
    printf("split %ld whole %ld bad %ld\n", split, whole, bad);
    return bad != 0 || !split || !whole;
}
