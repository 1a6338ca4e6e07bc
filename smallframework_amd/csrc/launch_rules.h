// Rules by which a launcher chooses a kernel or a grid (host-only C++, no HIP types, so that they can be tested on a machine
// without a GPU).
#pragma once

#include <algorithm>

namespace shp
{

constexpr int NUM_XCD = 8;                // MI355X: 8 XCDs x 32 CUs, one L2 per XCD
constexpr int NUM_CU = 256;

// conv3x3_c16_f32_kernel: the persistent workgroups of a channel group, for n_tiles tiles of 16 x 16 pixels and n_cg groups; 0 where
// another kernel is ahead.  The workgroups of all groups are resident at once, two per compute unit, in whole rounds over the XCDs: one more
// starts when the first ends and runs as long again (96 channels @104x104 batch 64, 528 workgroups 147 us, 504 119; 192 channels
// 305, 215; 80 channels + pooling batch 16 44.7, 30.1).  Taken where the runs keep those places at least 65% busy, counted by the
// longest run: 32 channels @208x208 + pooling batch 2 (66%) 12.0 -> 9.6 us, @104x104 batch 8 (77%) 11.5 -> 10.1, 160 @61x47 batch 17
// (66%) 21.9 -> 20.2, 224 @104x104 batch 3 (67%) 19.6 -> 18.4; below, 80 @104x104 batch 2 (57%) 7.7 -> 8.9, 128 batch 3 (57%) 12.3 ->
// 14.8, 192 @61x47 batch 8 (56%) 13.0 -> 13.5, 96 batch 17 (60%) level.
inline int c16_runs(long n_tiles, int n_cg, bool always = false)
{
    const int most = 2 * NUM_CU / n_cg / NUM_XCD * NUM_XCD;
    if (most == 0) return 0;
    const long longest = (n_tiles + most - 1) / most;
    if (!always && 20 * n_tiles * n_cg < 13 * longest * 2 * NUM_CU) return 0;
    return (int)std::min<long>(most, (n_tiles + NUM_XCD - 1) / NUM_XCD * NUM_XCD);
}

} // namespace shp
