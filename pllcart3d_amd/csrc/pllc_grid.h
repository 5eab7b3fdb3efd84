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

}  // namespace pllc
