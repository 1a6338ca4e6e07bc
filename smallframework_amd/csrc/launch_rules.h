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

// Equal shares of the reduction (conv_mfma_f32_streamk_kernel): the wave tile's pixel tiles (2x1 or 2x2), 0 where whole tiles are ahead.
// n_cg groups of 64 output channels, P pixels, nsteps K-steps.  Between half a round and three rounds of 64 x 128 workgroup tiles that are no
// whole rounds, and a long reduction (min_steps: 128 unless a measurement asks for another).  Float32 MFMAs, without -> with, batch 16 on 13x13 maps:
// 512 -> 1024 3x3 287 -> 264 us, 1024 -> 1024 519 -> 467, 256 -> 512 (144 steps) 81 -> 69; with 72 steps or fewer the fix-up pass
// costs more than the balance gains.  With split products 512 -> 1024 162.9 -> 158.2, 1024 -> 1024 319.6 -> 301.3, 256 -> 512 52.8 -> 50.2,
// with 72 steps 40.9 -> 50.2.
// 2x1, or 2x2 (a sixth fewer operands to split for a product) where there are more than 256 of the 2x1 workgroup tiles and 256 steps: 2x1 -> 2x2,
// 1024 -> 1024 304.7 -> 285.2, batch 20 371.5 -> 360.8, 28 494.7 -> 475.4; 512 -> 1024 160.9 -> 154.8, batch 32 300.8 -> 285.6; 512 -> 512
// @28x28 batch 12 260.7 -> 247.7; fewer tiles, 512 -> 1024 batch 10 (224) 106.7 -> 110.3, 512 -> 512 @28x28 batch 4 (200) 96.6 -> 104.2.  Its
// workgroup tiles are 64 x 256, and the half of one that lies past the last pixel is multiplied all the same: at most a sixteenth of the work.
// 2x1 -> 2x2, 1x1 4096 -> 4096 with 625 pixels (five blocks of 128 or three of 256) 128.3 -> 137.5, 8192 with 320 (three, two) 140.2 -> 173.3,
// 20480 with 121 (one, one) 134.3 -> 213.2, 2048 with 1089 (nine, five) 112.3 -> 118.7, 1984 with 1290 (eleven, six) 132.0 -> 136.3.
// More than 256 tiles and fewer steps are whole rounds and a rest in the other launch (256 -> 512 batch 26, 280 tiles, 73.7 -> 67.7,
// 32 86.9 -> 81.1, 49 123.2 -> 110.2; 2304 -> 512 1x1 117.2 -> 103.8; 256 -> 256 @30x30 batch 11 80.1 -> 76.4; with 288 steps 512 -> 1024
// batch 13 131.0, 133.8 without equal shares, 25 224.2, 222.1, with 576 1024 -> 1024 batch 13 238.7, 264.3).
inline int equal_share_pixel_tiles(int n_cg, long P, int nsteps, int min_steps = 128)
{
    const long px = (P + 127) / 128, tiles = n_cg * px;
    if (tiles <= NUM_CU / 2 || tiles >= 3 * NUM_CU || tiles % NUM_CU == 0 || nsteps < min_steps) return 0;
    if (tiles <= NUM_CU) return 1;
    if (nsteps < 256) return 0;
    return 32 * ((P + 255) / 256) <= 17 * px ? 2 : 1;
}

// conv_pw_dw3x3_f32_kernel: 32-channel tiles of a workgroup, 1 (four waves of two pixel tiles each, four workgroups per compute unit) or 2 (eight
// waves of one pixel tile, two workgroups: the pixels are read and split for twice the channels).  cib blocks of input channels, n_tiles
// spatial tiles over all images.  Two where the K loop is the larger part: 32 -> 64 channels, 128 -> 256 @28x28 batch 64 36.0 -> 33.7 us, 96 -> 192
// 24.3 -> 22.8, 128 -> 128 @56x56 stride 2 58.3 -> 56.6; 64 -> 128 @56x56 batch 64 45.0 -> 45.6.  And where its workgroups come in rounds of one
// per compute unit that are more than half full, or are six such rounds at least: a nearly empty round lasts as long as a full one.  128 -> 256
// @28x28, rounds 2.0: 21.3 -> 19.7, 2.1: 24.6 -> 25.9, 2.5 level, 2.8: 28.4 -> 26.7, 3.2: 32.8 -> 33.1, 3.8: 37.1 -> 34.5, 4.1 level, 4.6: 44.9 ->
// 42.0; 128 -> 320 @15x12 stride 2, 2.3: 9% behind.  Of 64 output channels 1 is ahead everywhere (128 -> 64 @42x41, rounds 2.0: 10%, 6.2: 2%; 96
// -> 64 @28x14 2 to 7%).
inline int pw_dw_channel_tiles(int cib, int Co, long n_tiles)
{
    const long n = n_tiles * (Co / 64), part = n % NUM_CU;
    if (cib < 6 || Co % 64 != 0 || Co < 128 || n < 2 * NUM_CU) return 1;
    return part == 0 || part > NUM_CU / 2 || n >= 6 * NUM_CU ? 2 : 1;
}

// Whole-model launch of a depthwise-separable chain: do bands of rows on several compute units pay for storing the last pair's rows and
// for the workgroup that gathers them?  `saved`: what the longest band does less than a whole image, in depthwise outputs (four channels of a
// pixel) over the 1024 lanes plus a quarter of the 16 x 16 x 16 products over the 16 waves; about a microsecond each.  The exchange is
// one of them, and a second one when every compute unit stores at the same time.  47 chains of one to five pairs at batches 1 to 120, us of whole
// images -> bands: DS-CNN (saved 12.8) 25.7 -> 15.6, 64 channels @13x9 and one pair to 16 (2.1) 9.1 -> 7.9, 32 @8x13 (1.5) level, batch 60 (1.2) 9.7 ->
// 11.0; few rows, whose bands compute each other's halo: 48-64-80 @3x1 9.4 -> 10.7, 64-80-64-128 @3x7 level; tiny ones, 16 @13x6 6.5 -> 6.9, batch 60
// 6.8 -> 7.7.  Against the faster form each time this rule loses 0.13 us at most where it cuts and 0.6 where it does not.
inline bool bands_pay(float saved, int batch, int bands) { return saved > 1.f + (float)batch * (float)bands / NUM_CU; }

} // namespace shp
