/* Checks the explicit kernels' planes per thread (march_planes in
 * pllc_grid.h): prints the number of cases in which the launch has more than
 * 65535 blocks along z, takes more planes a thread than it must for that, or
 * departs from the rule on waves where the blocks are few.  Then the number of
 * z-line lengths for which the autotuner does not time each block shape of the
 * z-sweep (1, 2 and 4 waves) exactly once. */
#include <cstdio>
#include <initializer_list>

#include "pllc_grid.h"

int main()
{
    long bad = 0;
    const int nxs[] = {1, 2, 24, 64, 512, 4096, 16383, 16384, 16385, 16500, 32767, 32768, 40000, 65533};
    for (int nx : nxs)
        for (int fields = 1; fields <= 4; fields++)
            for (int members : {1, 2, 64, 1000})
                for (double cells : {1.0, 4.0, 9.0, 100.0, 65536.0}) {
                    const int groups = fields * members;
                    if (groups > 65535) continue;
                    const double waves = cells * nx * groups / 64 / 1024;
                    const int np = pllc::march_planes(waves, nx, groups);
                    auto blocks = [&](int n) { return (long)((nx + n - 1) / n) * groups; };
                    int rule = 1;
                    while (rule < 8 && waves >= 5.0 * rule) rule *= 2;
                    if (blocks(np) > 65535 || np < rule || (np > rule && blocks(np / 2) <= 65535)) bad++;
                }
    long untuned = 0;
    for (int n = 1; n <= 1024; n++) {
        int c[4], seen[5] = {0, 0, 0, 0, 0};
        const int m = pllc::tune_lines(2, n, c);
        for (int q = 0; q < m; q++) seen[pllc::z_block_waves(c[q], n, 4)]++;
        if (seen[1] != 1 || seen[2] != 1 || seen[3] || seen[4] != 1 || pllc::z_block_waves(0, n, 4) != 4) untuned++;
    }
    printf("%ld %ld\n", bad, untuned);
    return 0;
}
