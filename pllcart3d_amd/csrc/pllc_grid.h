// pllc_grid.h -- launch shapes that follow from sizes alone (plain C++).
#pragma once

namespace pllc {

// Consecutive planes in x that a thread of the explicit kernels takes, for
// `planes` planes of `groups` fields (of every member) with `waves` waves per
// vector unit at one plane a thread.  More planes reuse more of the x neighbours
// in registers (24 loads a point instead of 37) and share a thread's set-up, but
// leave fewer waves: the largest power of two up to 8 that leaves 2.5 waves per
// vector unit.  us a step at 1, 2, 4, 8: 64x32x32 mixed 221, 220, 224, -;
// 97x45x39 FP64 428, 423, 426, -; 150x70x51 mixed 513, 490, 483, 492;
// 256x128x128 FP64 -, -, 2457, 2416; 512x256x256 mixed 11785, 10640, 10424, 10177
// (16: 10119, but 150x70x51 508).  More where the launch would have over 65535
// blocks along z, the API's limit (grids of few points per plane and more than
// 16384 planes of four fields).
inline int march_planes(double waves, int planes, int groups)
{
    int np = 1;
    while (np < 8 && waves >= 2 * np * 2.5) np *= 2;
    while (np < planes && (long)((planes + np - 1) / np) * groups > 65535) np *= 2;
    return np;
}

// z-lines of n rows that a wave takes (k_sweep_wave_z): 64 / G, G the power of
// two of at least the line's chunks of 16 rows
inline int z_lines_per_wave(int n)
{
    int G = 1;
    while (16 * G < n) G *= 2;
    return G > 64 ? 1 : 64 / G;
}
// waves in a block of the z-sweep, `most` of them unless tuned to `lines` per block
inline int z_block_waves(int lines, int n, int most)
{
    if (lines <= 0) return most;
    const int w = lines / z_lines_per_wave(n);
    return w < 1 ? 1 : w > most ? most : w;
}

// the lines per block that the autotuner times for lines of n rows along
// direction dir (0 x, 1 y, 2 z): for z those of 1, 2 and 4 waves (8 to 64 lines
// are one and the same launch for n <= 16, and for n <= 32 none of them the
// default's 4 waves)
inline int tune_lines(int dir, int n, int (&c)[4])
{
    if (dir == 2) {
        for (int q = 0; q < 3; q++) c[q] = z_lines_per_wave(n) << q;
        return 3;
    }
    const int all[4] = {8, 16, 32, 64};
    for (int q = 0; q < 4; q++) c[q] = all[q];
    return 4;
}

}  // namespace pllc
