// CPU unit test of the launch rules (smallframework_amd/csrc/launch_rules.h).
#include <cstdio>

#include "../../smallframework_amd/csrc/launch_rules.h"

using namespace shp;

static int g_failures = 0;
#define CHECK(c)                                                                  \
    do                                                                            \
    {                                                                             \
        if (!(c))                                                                 \
        {                                                                         \
            std::printf("FAILED %s:%d: %s\n", __FILE__, __LINE__, #c);            \
            ++g_failures;                                                         \
        }                                                                         \
    } while (0)

// 3x3 convolutions of sixteen input channels: the workgroups of all channel groups are resident at once (two per compute unit), every
// XCD has as many, and none of the tiles is left out
static void test_c16_workgroups_are_resident_at_once()
{
    for (int always = 0; always < 2; ++always)
        for (int n_cg = 1; n_cg <= 80; ++n_cg)
            for (long n_tiles = 1; n_tiles <= 20000; n_tiles += n_tiles < 700 ? 1 : 37)
            {
                const int n = c16_runs(n_tiles, n_cg, always != 0);
                CHECK(n * n_cg <= 2 * NUM_CU && n % NUM_XCD == 0 && n >= 0);
                if (g_failures) return;
            }
    CHECK(c16_runs(3136, 1) == 512 && c16_runs(3136, 2) == 256 && c16_runs(3136, 3) == 168 && c16_runs(3136, 5) == 96);
    CHECK(c16_runs(3136, 64) == 8 && c16_runs(3136, 65) == 0);
}

// few tiles, or runs of unequal length: the places are not busy enough
static void test_c16_leaves_ragged_launches_to_the_others()
{
    CHECK(c16_runs(338, 1) == 344 && c16_runs(392, 1) == 392);                          // 66%, 77%
    CHECK(c16_runs(98, 3) == 0 && c16_runs(147, 4) == 0 && c16_runs(204, 3) == 0);      // 57%, 57% (two tiles for 1.1), 60%
    CHECK(c16_runs(98, 3, true) == 104);
}

// equal shares of the reduction: 64 x 256 tiles only where the blocks of 256 pixels cover at most a sixteenth more than those of 128
static void test_equal_shares_with_large_tiles_waste_no_work()
{
    for (int n_cg = 1; n_cg <= 768; ++n_cg)
        for (long P = 1; P <= 98304 / n_cg + 300; P += P < 3000 ? 1 : 61)
        {
            const long b128 = (P + 127) / 128, b256 = (P + 255) / 256, tiles = n_cg * b128;
            const int t = equal_share_pixel_tiles(n_cg, P, 256);
            CHECK((t != 0) == (tiles > 128 && tiles < 768 && tiles % 256 != 0));
            CHECK(t != 2 || (tiles > 256 && 16 * (2 * b256 - b128) <= b128));
            CHECK(t != 1 || tiles <= 256 || 16 * (2 * b256 - b128) > b128);
            CHECK(equal_share_pixel_tiles(n_cg, P, 255) == (tiles > 256 ? 0 : t) && equal_share_pixel_tiles(n_cg, P, 127) == 0);
            if (g_failures) return;
        }
    CHECK(equal_share_pixel_tiles(64, 625, 256) == 1 && equal_share_pixel_tiles(320, 121, 256) == 1 && equal_share_pixel_tiles(128, 320, 256) == 1);
    CHECK(equal_share_pixel_tiles(16, 2704, 288) == 2 && equal_share_pixel_tiles(64, 754, 256) == 2);
}

// pointwise + depthwise launch: workgroups of 64 channels where they fill their rounds
static void test_workgroups_of_sixty_four_channels_fill_their_rounds()
{
    for (int cib = 1; cib <= 8; ++cib)
        for (int Co = 32; Co <= 1024; Co += 32)
            for (long nt = 1; nt <= 3000; ++nt)
            {
                const long n = nt * (Co / 64);
                const int c = pw_dw_channel_tiles(cib, Co, nt);
                CHECK(c == 1 || (c == 2 && cib >= 6 && Co % 64 == 0 && Co > 64 && n >= 512));
                CHECK(c == 1 || n >= 1536 || (n + 255) / 256 * 256 - n < 128);
                if (g_failures) return;
            }
    CHECK(pw_dw_channel_tiles(8, 256, 256) == 2 && pw_dw_channel_tiles(8, 128, 256) == 2);      // 1024 and 512 workgroups
    CHECK(pw_dw_channel_tiles(8, 256, 136) == 1 && pw_dw_channel_tiles(8, 448, 76) == 1);       // 544 and 532: a third round of 32 and 20
    CHECK(pw_dw_channel_tiles(8, 64, 576) == 1 && pw_dw_channel_tiles(4, 256, 256) == 1);
}

// bands of rows: not for a model whose bands save less than the exchange costs, and more is asked when every compute unit stores
static void test_bands_pay()
{
    CHECK(bands_pay(12.8f, 1, 25) && bands_pay(6.28f, 128, 2));
    CHECK(!bands_pay(0.9f, 1, 25) && !bands_pay(1.5f, 128, 2) && bands_pay(1.5f, 1, 8));
}

int main()
{
    test_bands_pay();
    test_workgroups_of_sixty_four_channels_fill_their_rounds();
    test_equal_shares_with_large_tiles_waste_no_work();
    test_c16_workgroups_are_resident_at_once();
    test_c16_leaves_ragged_launches_to_the_others();
    std::printf(g_failures ? "%d CHECKS FAILED\n" : "ALL PASSED\n", g_failures);
    return g_failures ? 1 : 0;
}
