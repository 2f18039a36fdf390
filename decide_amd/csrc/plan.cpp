// See plan.h. Two parts:
//   * a table measured on an MI355X: for decide's engine shapes (K, N) at 42
//     row counts from 1 to 2307, at most 27 % apart above 16, the fastest
//     (tile variant, split-K) and its time with weights streaming from HBM —
//     the MI355X counterpart of decide's M1 Pro RECOMMENDED table
//     (crates/decide-metal/src/gemm_configs.rs:247-283). `python -m
//     decide_amd.tune_gemm` times the menu at these rows, as the calls the
//     table's times are of; in a later run of it over all 378 points the
//     table's choices were 1.2 % from that run's fastest. Four rows more
//     (800, 1400 and 1800 rows of the N = 2560 and 2048 shapes) cover ranges
//     of 30 to 60 row counts where the choice between two of the 42 was 5-8 %
//     behind; at 108 points between the rows it is 0.7 % behind on average;
//   * a cost model for every other shape, fitted to the table's points (over
//     the seven fastest choices of each in that later run: rms error 10 %, its
//     pick 3.5 % from the fastest). Off the fit, 77 points of seven other
//     shapes from 3 to 2,200 rows: its pick 9 % from the fastest, mostly below
//     100 rows; engine shapes at 3,000, 4,096 and 8,192 rows: the fastest, or
//     within 2 %. A 64-wide K stage takes the
//     longer of its MFMAs and of its operands at the 57 GB/s a CU takes in, a
//     workgroup a fixed part that grows with its tile (prologue and epilogue),
//     blocks run in rounds of 256 (one per CU), the weights stream at most at
//     5 TB/s, and split-K adds a reduction over its partials.
// A measured M takes its row. Between two, the choices of the rows around M are compared at M
// itself: each one's measured time, scaled by what the model says that choice
// gains or loses between its M and this one (a tile may need one more row of
// tiles or one more round of 256). Where the table had rows only 2 x apart and
// the model took over between them, the choice was 20-70 % slower than the
// fastest over most of that range (M = 40: gate|up 32.5 against 22.7 us, down
// 22.2 against 16.4; M = 1900 down 118 against 97). Apart from both,
// plan_order picks the tiles' work order for the XCDs' L2s.
#include "plan.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <limits>

#include "dh_kernels.h"

namespace dh {

namespace {
constexpr double kCUs = 256.0;
constexpr double kHbmBytesPerUs = 5.08e6;     // weights streaming from HBM
constexpr double kMfmaUs = 0.0252;            // 64-wide stage, per 16 x 16 fragment of a wave
constexpr double kMfma8 = 0.844;              // the same with two waves per SIMD
constexpr double kFeedUs = 0.57;              // 64-wide stage, per 256 operand rows (32 KB)
constexpr double kMinStageUs = 0.279;         // a stage is never cheaper than its barrier and waits
constexpr double kTileUs = 2.22, kTileAreaUs = 3.60;  // per workgroup, and per 160 x 160 of its tile
constexpr double kLaunchUs = 2.09;
constexpr double kReduceUs = 2.18, kReduceBytesPerUs = 4.78e6;
constexpr uint32_t kSplitMenu[] = {1, 2, 3, 4, 6, 8};

uint32_t ceil_div(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

struct Measured {
  uint16_t k, n, m;
  uint8_t variant, splits;
  float us;
};

// {k, n, m, variant, splits, us}: fastest on an MI355X (gfx950, 256 CUs),
// weights rotated over > 256 MB; the variant indexes the compiled menu
// (kVariants, gemm_tile.hip). K = 4096 is timed with the norm that follows it
// (dh_gemm_add_rmsnorm) and K = 9216 with and without, so the sum over the
// partials costs what it does there. Choices within 2 % of the fastest count
// as ties and go to the one that covers the least padded area: sustained, the
// chip is power-limited, and MFMA work on padding rows costs energy that a
// burst of launches does not show. N = 2048 has no rows up to 16: there the
// streaming kernel, which comes after the table, takes as long (plan.h).
const Measured kMeasured[] = {
    {2560, 12352, 1, 22, 1, 16.5f}, {2560, 12352, 3, 22, 1, 16.8f}, {2560, 12352, 8, 0, 4, 17.5f},
    {2560, 12352, 12, 22, 1, 17.3f}, {2560, 12352, 16, 0, 4, 18.4f}, {2560, 12352, 20, 22, 1, 18.3f},
    {2560, 12352, 24, 22, 1, 18.6f}, {2560, 12352, 28, 22, 1, 19.0f}, {2560, 12352, 32, 22, 1, 19.2f},
    {2560, 12352, 40, 19, 3, 19.5f}, {2560, 12352, 48, 19, 3, 20.1f}, {2560, 12352, 56, 19, 3, 20.6f},
    {2560, 12352, 64, 19, 3, 21.3f}, {2560, 12352, 80, 10, 3, 22.8f}, {2560, 12352, 96, 10, 3, 24.1f},
    {2560, 12352, 112, 14, 3, 26.4f}, {2560, 12352, 128, 14, 3, 27.6f}, {2560, 12352, 144, 14, 3, 27.4f},
    {2560, 12352, 163, 19, 1, 28.8f}, {2560, 12352, 176, 19, 1, 29.1f}, {2560, 12352, 200, 10, 1, 29.7f},
    {2560, 12352, 230, 10, 1, 31.8f}, {2560, 12352, 256, 10, 1, 33.3f}, {2560, 12352, 276, 10, 1, 33.9f},
    {2560, 12352, 320, 14, 1, 38.6f}, {2560, 12352, 370, 14, 1, 37.0f}, {2560, 12352, 430, 14, 1, 39.2f},
    {2560, 12352, 490, 8, 1, 45.6f}, {2560, 12352, 550, 8, 1, 47.8f}, {2560, 12352, 603, 4, 1, 49.5f},
    {2560, 12352, 680, 5, 1, 54.3f}, {2560, 12352, 760, 5, 1, 55.8f}, {2560, 12352, 850, 9, 1, 61.1f},
    {2560, 12352, 950, 17, 1, 65.0f}, {2560, 12352, 1024, 17, 1, 66.3f}, {2560, 12352, 1150, 16, 1, 74.5f},
    {2560, 12352, 1300, 5, 1, 101.4f}, {2560, 12352, 1500, 5, 1, 106.8f}, {2560, 12352, 1700, 11, 1, 120.0f},
    {2560, 12352, 1900, 17, 1, 127.1f}, {2560, 12352, 2100, 17, 1, 133.4f}, {2560, 12352, 2307, 16, 1, 144.7f},
    {2560, 10240, 1, 22, 2, 14.1f}, {2560, 10240, 3, 0, 4, 15.9f}, {2560, 10240, 8, 22, 2, 14.1f},
    {2560, 10240, 12, 22, 2, 14.2f}, {2560, 10240, 16, 22, 2, 14.5f}, {2560, 10240, 20, 22, 2, 14.8f},
    {2560, 10240, 24, 22, 2, 14.8f}, {2560, 10240, 28, 22, 2, 15.7f}, {2560, 10240, 32, 22, 2, 15.4f},
    {2560, 10240, 40, 18, 2, 16.5f}, {2560, 10240, 48, 19, 4, 17.6f}, {2560, 10240, 56, 19, 4, 17.9f},
    {2560, 10240, 64, 19, 4, 18.6f}, {2560, 10240, 80, 18, 1, 18.8f}, {2560, 10240, 96, 18, 1, 20.2f},
    {2560, 10240, 112, 20, 1, 20.9f}, {2560, 10240, 128, 18, 1, 22.0f}, {2560, 10240, 144, 20, 1, 23.1f},
    {2560, 10240, 163, 15, 1, 24.1f}, {2560, 10240, 176, 15, 1, 24.5f}, {2560, 10240, 200, 21, 1, 25.3f},
    {2560, 10240, 230, 21, 1, 27.7f}, {2560, 10240, 256, 19, 1, 29.6f}, {2560, 10240, 276, 21, 1, 30.8f},
    {2560, 10240, 320, 10, 1, 31.4f}, {2560, 10240, 370, 10, 1, 33.8f}, {2560, 10240, 430, 14, 1, 37.9f},
    {2560, 10240, 490, 14, 1, 38.6f}, {2560, 10240, 550, 14, 1, 38.4f}, {2560, 10240, 603, 14, 1, 39.6f},
    {2560, 10240, 680, 4, 1, 46.9f}, {2560, 10240, 760, 4, 1, 50.4f}, {2560, 10240, 850, 5, 1, 55.8f},
    {2560, 10240, 950, 5, 1, 55.4f}, {2560, 10240, 1024, 9, 1, 60.5f}, {2560, 10240, 1150, 17, 1, 64.9f},
    {2560, 10240, 1300, 16, 1, 72.0f}, {2560, 10240, 1500, 16, 1, 74.7f}, {2560, 10240, 1700, 14, 1, 105.2f},
    {2560, 10240, 1900, 14, 1, 106.8f}, {2560, 10240, 2100, 9, 1, 119.4f}, {2560, 10240, 2307, 17, 1, 125.1f},
    {2560, 18432, 1, 22, 1, 19.4f}, {2560, 18432, 3, 22, 1, 19.4f}, {2560, 18432, 8, 22, 1, 19.5f},
    {2560, 18432, 12, 22, 1, 19.9f}, {2560, 18432, 16, 22, 1, 20.1f}, {2560, 18432, 20, 22, 1, 20.6f},
    {2560, 18432, 24, 22, 1, 20.9f}, {2560, 18432, 28, 22, 1, 21.2f}, {2560, 18432, 32, 22, 1, 21.4f},
    {2560, 18432, 40, 18, 1, 22.8f}, {2560, 18432, 48, 18, 1, 23.6f}, {2560, 18432, 56, 18, 1, 24.5f},
    {2560, 18432, 64, 18, 1, 25.1f}, {2560, 18432, 80, 20, 1, 26.9f}, {2560, 18432, 96, 20, 1, 28.8f},
    {2560, 18432, 112, 15, 1, 30.9f}, {2560, 18432, 128, 15, 1, 31.7f}, {2560, 18432, 144, 21, 1, 32.8f},
    {2560, 18432, 163, 10, 1, 34.1f}, {2560, 18432, 176, 10, 1, 34.3f}, {2560, 18432, 200, 14, 1, 35.8f},
    {2560, 18432, 230, 14, 1, 36.9f}, {2560, 18432, 256, 14, 1, 38.1f}, {2560, 18432, 276, 14, 1, 38.5f},
    {2560, 18432, 320, 14, 1, 39.2f}, {2560, 18432, 370, 4, 1, 45.8f}, {2560, 18432, 430, 5, 1, 48.5f},
    {2560, 18432, 490, 9, 1, 54.3f}, {2560, 18432, 550, 11, 1, 55.5f}, {2560, 18432, 603, 11, 1, 56.6f},
    {2560, 18432, 680, 17, 1, 62.7f}, {2560, 18432, 760, 17, 1, 64.4f}, {2560, 18432, 850, 12, 1, 76.4f},
    {2560, 18432, 950, 5, 1, 92.4f}, {2560, 18432, 1024, 5, 1, 94.6f}, {2560, 18432, 1150, 9, 1, 104.9f},
    {2560, 18432, 1300, 13, 1, 116.4f}, {2560, 18432, 1500, 17, 1, 125.5f}, {2560, 18432, 1700, 16, 1, 135.5f},
    {2560, 18432, 1900, 11, 1, 164.0f}, {2560, 18432, 2100, 17, 1, 180.4f}, {2560, 18432, 2307, 16, 1, 193.6f},
    {4096, 2560, 1, 22, 6, 11.2f}, {4096, 2560, 3, 22, 6, 11.2f}, {4096, 2560, 8, 22, 6, 11.5f},
    {4096, 2560, 12, 22, 6, 11.6f}, {4096, 2560, 16, 22, 8, 11.7f}, {4096, 2560, 20, 22, 6, 11.9f},
    {4096, 2560, 24, 22, 6, 11.9f}, {4096, 2560, 28, 22, 6, 12.1f}, {4096, 2560, 32, 22, 6, 12.1f},
    {4096, 2560, 40, 22, 4, 12.5f}, {4096, 2560, 48, 22, 4, 12.6f}, {4096, 2560, 56, 22, 4, 12.9f},
    {4096, 2560, 64, 22, 4, 13.2f}, {4096, 2560, 80, 22, 3, 13.9f}, {4096, 2560, 96, 22, 3, 14.4f},
    {4096, 2560, 112, 18, 4, 15.6f}, {4096, 2560, 128, 18, 4, 16.0f}, {4096, 2560, 144, 18, 3, 16.0f},
    {4096, 2560, 163, 18, 3, 16.5f}, {4096, 2560, 176, 18, 3, 17.1f}, {4096, 2560, 200, 18, 2, 18.5f},
    {4096, 2560, 230, 20, 3, 18.6f}, {4096, 2560, 256, 20, 3, 19.2f}, {4096, 2560, 276, 20, 3, 19.9f},
    {4096, 2560, 320, 21, 4, 21.9f}, {4096, 2560, 370, 15, 3, 22.7f}, {4096, 2560, 430, 21, 3, 23.8f},
    {4096, 2560, 490, 21, 2, 26.2f}, {4096, 2560, 550, 21, 2, 27.2f}, {4096, 2560, 603, 14, 4, 28.4f},
    {4096, 2560, 680, 10, 2, 30.9f}, {4096, 2560, 760, 10, 2, 32.3f}, {4096, 2560, 800, 14, 3, 32.5f},
    {4096, 2560, 850, 8, 3, 36.2f}, {4096, 2560, 950, 4, 3, 38.1f}, {4096, 2560, 1024, 14, 2, 38.3f},
    {4096, 2560, 1150, 14, 2, 40.0f}, {4096, 2560, 1300, 21, 1, 45.9f}, {4096, 2560, 1500, 10, 1, 50.8f},
    {4096, 2560, 1700, 5, 2, 56.7f}, {4096, 2560, 1900, 5, 2, 59.0f}, {4096, 2560, 2100, 14, 1, 64.3f},
    {4096, 2560, 2307, 14, 1, 65.5f},
    {9216, 2560, 1, 22, 8, 15.5f}, {9216, 2560, 3, 22, 8, 15.6f}, {9216, 2560, 8, 22, 8, 15.8f},
    {9216, 2560, 12, 22, 8, 15.9f}, {9216, 2560, 16, 22, 8, 15.9f}, {9216, 2560, 20, 22, 8, 15.9f},
    {9216, 2560, 24, 22, 8, 16.1f}, {9216, 2560, 28, 22, 8, 16.3f}, {9216, 2560, 32, 22, 8, 16.3f},
    {9216, 2560, 40, 18, 8, 16.9f}, {9216, 2560, 48, 18, 8, 17.3f}, {9216, 2560, 56, 18, 8, 17.7f},
    {9216, 2560, 64, 18, 8, 17.9f}, {9216, 2560, 80, 20, 8, 19.2f}, {9216, 2560, 96, 20, 8, 20.0f},
    {9216, 2560, 112, 19, 8, 21.4f}, {9216, 2560, 128, 19, 8, 21.9f}, {9216, 2560, 144, 21, 8, 23.1f},
    {9216, 2560, 163, 10, 8, 24.7f}, {9216, 2560, 176, 10, 8, 25.3f}, {9216, 2560, 200, 19, 4, 26.9f},
    {9216, 2560, 230, 20, 3, 28.2f}, {9216, 2560, 256, 19, 4, 29.6f}, {9216, 2560, 276, 3, 8, 31.2f},
    {9216, 2560, 320, 10, 4, 31.9f}, {9216, 2560, 370, 21, 3, 33.7f}, {9216, 2560, 430, 21, 3, 36.9f},
    {9216, 2560, 490, 4, 6, 40.0f}, {9216, 2560, 550, 14, 4, 41.1f}, {9216, 2560, 603, 14, 4, 42.2f},
    {9216, 2560, 680, 10, 2, 48.3f}, {9216, 2560, 760, 4, 4, 49.5f}, {9216, 2560, 800, 14, 3, 50.8f},
    {9216, 2560, 850, 8, 3, 56.9f}, {9216, 2560, 950, 5, 4, 60.5f}, {9216, 2560, 1024, 4, 3, 61.3f},
    {9216, 2560, 1150, 14, 2, 65.0f}, {9216, 2560, 1300, 8, 2, 77.5f}, {9216, 2560, 1400, 9, 3, 79.5f},
    {9216, 2560, 1500, 4, 2, 82.7f}, {9216, 2560, 1700, 5, 2, 91.7f}, {9216, 2560, 1900, 5, 2, 97.4f},
    {9216, 2560, 2100, 9, 2, 107.7f}, {9216, 2560, 2307, 14, 1, 115.3f},
    {2560, 2048, 20, 22, 4, 8.4f}, {2560, 2048, 24, 22, 4, 8.5f}, {2560, 2048, 28, 22, 4, 8.6f},
    {2560, 2048, 32, 22, 3, 8.9f}, {2560, 2048, 40, 22, 4, 8.7f}, {2560, 2048, 48, 22, 4, 8.8f},
    {2560, 2048, 56, 18, 4, 9.9f}, {2560, 2048, 64, 22, 2, 9.8f}, {2560, 2048, 80, 22, 3, 9.4f},
    {2560, 2048, 96, 22, 3, 9.6f}, {2560, 2048, 112, 22, 2, 10.3f}, {2560, 2048, 128, 18, 4, 11.0f},
    {2560, 2048, 144, 22, 2, 10.8f}, {2560, 2048, 163, 22, 1, 11.5f}, {2560, 2048, 176, 22, 1, 11.8f},
    {2560, 2048, 200, 22, 1, 11.7f}, {2560, 2048, 230, 18, 2, 13.0f}, {2560, 2048, 256, 18, 1, 14.0f},
    {2560, 2048, 276, 18, 1, 13.4f}, {2560, 2048, 320, 18, 2, 14.3f}, {2560, 2048, 370, 18, 1, 15.8f},
    {2560, 2048, 430, 18, 1, 15.7f}, {2560, 2048, 490, 18, 1, 16.0f}, {2560, 2048, 550, 18, 1, 16.2f},
    {2560, 2048, 603, 20, 1, 17.8f}, {2560, 2048, 680, 20, 1, 18.0f}, {2560, 2048, 760, 20, 1, 19.8f},
    {2560, 2048, 850, 20, 1, 20.0f}, {2560, 2048, 950, 20, 1, 20.4f}, {2560, 2048, 1024, 15, 1, 21.0f},
    {2560, 2048, 1150, 21, 1, 23.1f}, {2560, 2048, 1300, 15, 1, 22.8f}, {2560, 2048, 1500, 21, 1, 24.8f},
    {2560, 2048, 1700, 21, 1, 27.2f}, {2560, 2048, 1800, 10, 1, 31.3f}, {2560, 2048, 1900, 4, 2, 35.2f},
    {2560, 2048, 2100, 14, 1, 33.5f}, {2560, 2048, 2307, 14, 1, 34.9f},
    {2560, 8192, 1, 22, 2, 12.5f}, {2560, 8192, 3, 22, 2, 12.6f}, {2560, 8192, 8, 22, 2, 12.8f},
    {2560, 8192, 12, 22, 2, 13.2f}, {2560, 8192, 16, 22, 2, 13.3f}, {2560, 8192, 20, 22, 2, 13.9f},
    {2560, 8192, 24, 22, 2, 13.8f}, {2560, 8192, 28, 22, 2, 14.2f}, {2560, 8192, 32, 22, 2, 14.4f},
    {2560, 8192, 40, 18, 2, 15.4f}, {2560, 8192, 48, 19, 4, 15.9f}, {2560, 8192, 56, 19, 4, 16.7f},
    {2560, 8192, 64, 19, 4, 17.1f}, {2560, 8192, 80, 18, 1, 18.2f}, {2560, 8192, 96, 10, 4, 19.7f},
    {2560, 8192, 112, 20, 1, 20.1f}, {2560, 8192, 128, 2, 4, 21.5f}, {2560, 8192, 144, 20, 1, 22.4f},
    {2560, 8192, 163, 15, 1, 22.9f}, {2560, 8192, 176, 15, 1, 23.7f}, {2560, 8192, 200, 21, 1, 24.6f},
    {2560, 8192, 230, 21, 1, 26.6f}, {2560, 8192, 256, 2, 2, 28.8f}, {2560, 8192, 276, 7, 2, 30.0f},
    {2560, 8192, 320, 10, 1, 30.1f}, {2560, 8192, 370, 10, 1, 32.4f}, {2560, 8192, 430, 8, 2, 36.4f},
    {2560, 8192, 490, 14, 1, 35.4f}, {2560, 8192, 550, 14, 1, 36.5f}, {2560, 8192, 603, 14, 1, 38.0f},
    {2560, 8192, 680, 3, 1, 42.2f}, {2560, 8192, 760, 3, 1, 43.7f}, {2560, 8192, 850, 8, 1, 46.5f},
    {2560, 8192, 950, 4, 1, 47.8f}, {2560, 8192, 1024, 4, 1, 49.6f}, {2560, 8192, 1150, 5, 1, 55.4f},
    {2560, 8192, 1300, 9, 1, 61.2f}, {2560, 8192, 1500, 17, 1, 65.5f}, {2560, 8192, 1700, 16, 1, 72.8f},
    {2560, 8192, 1900, 16, 1, 77.2f}, {2560, 8192, 2100, 5, 1, 102.6f}, {2560, 8192, 2307, 5, 1, 105.6f},
    {2560, 6144, 1, 22, 4, 10.9f}, {2560, 6144, 3, 22, 3, 11.1f}, {2560, 6144, 8, 22, 4, 11.0f},
    {2560, 6144, 12, 22, 4, 11.1f}, {2560, 6144, 16, 22, 4, 11.2f}, {2560, 6144, 20, 22, 4, 11.5f},
    {2560, 6144, 24, 22, 4, 11.5f}, {2560, 6144, 28, 22, 3, 12.3f}, {2560, 6144, 32, 22, 4, 12.1f},
    {2560, 6144, 40, 18, 4, 12.8f}, {2560, 6144, 48, 18, 4, 13.2f}, {2560, 6144, 56, 18, 4, 13.8f},
    {2560, 6144, 64, 18, 4, 14.0f}, {2560, 6144, 80, 20, 4, 15.3f}, {2560, 6144, 96, 20, 4, 16.1f},
    {2560, 6144, 112, 22, 1, 16.4f}, {2560, 6144, 128, 18, 2, 17.0f}, {2560, 6144, 144, 18, 1, 18.0f},
    {2560, 6144, 163, 20, 2, 19.1f}, {2560, 6144, 176, 20, 2, 19.5f}, {2560, 6144, 200, 18, 1, 18.1f},
    {2560, 6144, 230, 18, 1, 19.9f}, {2560, 6144, 256, 18, 1, 20.9f}, {2560, 6144, 276, 15, 1, 22.3f},
    {2560, 6144, 320, 20, 1, 21.8f}, {2560, 6144, 370, 20, 1, 24.2f}, {2560, 6144, 430, 15, 1, 24.9f},
    {2560, 6144, 490, 21, 1, 25.9f}, {2560, 6144, 550, 21, 1, 27.6f}, {2560, 6144, 603, 21, 1, 30.7f},
    {2560, 6144, 680, 14, 1, 35.4f}, {2560, 6144, 760, 14, 1, 37.6f}, {2560, 6144, 850, 14, 1, 36.6f},
    {2560, 6144, 950, 14, 1, 38.7f}, {2560, 6144, 1024, 8, 1, 44.3f}, {2560, 6144, 1150, 4, 1, 48.2f},
    {2560, 6144, 1300, 5, 1, 52.3f}, {2560, 6144, 1500, 5, 1, 54.2f}, {2560, 6144, 1700, 9, 1, 60.0f},
    {2560, 6144, 1900, 17, 1, 64.0f}, {2560, 6144, 2100, 16, 1, 68.8f}, {2560, 6144, 2307, 16, 1, 72.9f},
    {2560, 9216, 1, 22, 2, 13.1f}, {2560, 9216, 3, 22, 2, 13.2f}, {2560, 9216, 8, 22, 2, 14.1f},
    {2560, 9216, 12, 22, 2, 13.4f}, {2560, 9216, 16, 22, 2, 13.8f}, {2560, 9216, 20, 22, 2, 15.4f},
    {2560, 9216, 24, 22, 2, 14.2f}, {2560, 9216, 28, 22, 2, 14.5f}, {2560, 9216, 32, 22, 2, 14.8f},
    {2560, 9216, 40, 22, 1, 15.6f}, {2560, 9216, 48, 22, 1, 16.5f}, {2560, 9216, 56, 22, 1, 16.9f},
    {2560, 9216, 64, 22, 1, 17.4f}, {2560, 9216, 80, 18, 1, 18.6f}, {2560, 9216, 96, 18, 1, 19.2f},
    {2560, 9216, 112, 20, 1, 20.0f}, {2560, 9216, 128, 20, 1, 21.1f}, {2560, 9216, 144, 20, 1, 21.9f},
    {2560, 9216, 163, 15, 1, 23.8f}, {2560, 9216, 176, 21, 1, 23.8f}, {2560, 9216, 200, 21, 1, 24.9f},
    {2560, 9216, 230, 21, 1, 27.1f}, {2560, 9216, 256, 15, 1, 29.1f}, {2560, 9216, 276, 21, 1, 30.3f},
    {2560, 9216, 320, 10, 1, 30.9f}, {2560, 9216, 370, 10, 1, 32.1f}, {2560, 9216, 430, 14, 1, 36.5f},
    {2560, 9216, 490, 14, 1, 35.7f}, {2560, 9216, 550, 14, 1, 37.1f}, {2560, 9216, 603, 14, 1, 38.3f},
    {2560, 9216, 680, 8, 1, 44.5f}, {2560, 9216, 760, 8, 1, 47.7f}, {2560, 9216, 850, 4, 1, 49.3f},
    {2560, 9216, 950, 5, 1, 54.3f}, {2560, 9216, 1024, 5, 1, 55.3f}, {2560, 9216, 1150, 9, 1, 61.6f},
    {2560, 9216, 1300, 13, 1, 67.2f}, {2560, 9216, 1500, 17, 1, 69.7f}, {2560, 9216, 1700, 16, 1, 77.0f},
    {2560, 9216, 1900, 5, 1, 106.1f}, {2560, 9216, 2100, 5, 1, 107.0f}, {2560, 9216, 2307, 11, 1, 118.3f},
};
}  // namespace

Plan plan_make(int variant, uint32_t splits, uint32_t m, uint32_t n, uint32_t k) {
  const VariantInfo v = variant_info(variant);
  Plan p{};
  p.variant = variant;
  const uint32_t stages = ceil_div(k, kBK);
  splits = std::max(1u, std::min(splits, std::max(stages, 1u)));
  p.kps = ceil_div(stages, splits) * kBK;
  p.splits = p.kps ? ceil_div(k, p.kps) : 1;  // splits that would be empty are dropped; K = 0: one, empty
  p.mtiles = ceil_div(m, (uint32_t)v.bm());
  p.stripes = ceil_div(n, (uint32_t)v.bn());
  p.grid = p.mtiles * p.stripes * p.splits;
  p.ws_bytes = p.splits > 1 ? (uint64_t)p.splits * m * n * sizeof(float) : 0;
  p.est_us = plan_estimate_us(variant, p.splits, m, n, k);
  return p;
}

double plan_estimate_us(int variant, uint32_t splits, uint32_t m, uint32_t n, uint32_t k) {
  const VariantInfo v = variant_info(variant);
  const uint32_t stages = ceil_div(k, kBK);
  if (splits < 1 || splits > stages) return std::numeric_limits<double>::infinity();
  const uint32_t st_per_split = ceil_div(stages, splits);
  splits = ceil_div(stages, st_per_split);
  const double mtiles = ceil_div(m, (uint32_t)v.bm()), stripes = ceil_div(n, (uint32_t)v.bn());
  const double blocks = mtiles * stripes * splits;
  const double rounds = std::ceil(blocks / kCUs);
  const double stage_us = std::max({kMfmaUs * v.fm * v.fn * (v.spw == 2 ? kMfma8 : 1.0),
                                    kFeedUs * (v.bm() + v.bn()) / 256.0, kMinStageUs});
  const double tile_us = kTileUs + kTileAreaUs * v.bm() * v.bn() / 25600.0;
  double t = kLaunchUs + std::max(rounds * (st_per_split * stage_us + tile_us),
                                  kTileUs + 2.0 * n * k / kHbmBytesPerUs);
  if (splits > 1) t += kReduceUs + (splits + 1.0) * m * n * 4.0 / kReduceBytesPerUs;
  return t;
}

namespace {
Plan plan_model(uint32_t m, uint32_t n, uint32_t k, uint64_t max_ws) {
  Plan best{};
  best.est_us = std::numeric_limits<double>::infinity();
  best.variant = -1;
  for (int v = 0; v < variant_count(); ++v) {
    for (uint32_t s : kSplitMenu) {
      const double t = plan_estimate_us(v, s, m, n, k);
      if (!(t < best.est_us)) continue;
      const Plan p = plan_make(v, s, m, n, k);
      if (p.ws_bytes > max_ws) continue;
      best = p;
    }
  }
  return best;
}
}  // namespace

// The weight-streaming kernel for M <= 16: one workgroup per 32 columns and
// K split, splits chosen so that about two workgroups per CU stream at once
// (each split a whole number of 128-wide k blocks; no split when the
// workspace is capped, as for grouped launches).
Plan plan_stream(uint32_t m, uint32_t n, uint32_t k, uint64_t max_ws) {
  Plan p{};
  p.variant = kStreamVariant;
  const uint32_t blocks = n / 32, kb = k / 128;
  uint32_t s = std::min(std::max(1u, ceil_div(512, blocks)), kb);
  const uint32_t kpb = ceil_div(kb, s);
  s = ceil_div(kb, kpb);
  p.splits = s;
  p.kps = kpb * 128;
  p.ws_bytes = s > 1 ? (uint64_t)s * m * n * 4 : 0;
  if (p.ws_bytes > max_ws) {
    p.splits = 1;
    p.kps = k;
    p.ws_bytes = 0;
  }
  p.mtiles = 1;
  p.stripes = blocks;
  p.grid = blocks * p.splits;
  p.est_us = kLaunchUs + kTileUs + 2.0 * n * k / kHbmBytesPerUs;
  return p;
}

Plan plan_gemm(uint32_t m, uint32_t n, uint32_t k, uint64_t max_ws) {
  // decide's contract admits N = 0 (nothing to launch: an empty grid) and K = 0 (the tiles run no
  // stage and store the empty sum).
  if (n == 0 || k == 0) return plan_make(0, 1, m, n, k);
  const Measured* best = nullptr;
  double best_us = std::numeric_limits<double>::infinity();
  for (const Measured& e : kMeasured) {
    if (e.k != k || e.n != n) continue;
    const bool fits = e.splits == 1 || (uint64_t)e.splits * m * n * sizeof(float) <= max_ws;
    if (e.m == m && fits) {
      best = &e;
      break;
    }
    const uint32_t lo = std::min<uint32_t>(m, e.m), hi = std::max<uint32_t>(m, e.m);
    if (hi - lo > 4 && hi > lo * 1.3) continue;
    const double us = e.us * plan_estimate_us(e.variant, e.splits, m, n, k) /
                      plan_estimate_us(e.variant, e.splits, e.m, n, k);
    if (us < best_us && fits) {
      best_us = us;
      best = &e;
    }
  }
  if (best) return plan_make(best->variant, best->splits, m, n, k);
  if (m <= kStreamMaxM && n <= kStreamMaxN && k % 128 == 0 && n % 32 == 0) return plan_stream(m, n, k, max_ws);
  return plan_model(m, n, k, max_ws);
}

uint64_t plan_ws_need(uint32_t max_m, uint32_t n, uint32_t k, uint64_t max_ws) {
  uint64_t need = 0;
  for (uint32_t m = 1; m <= max_m; ++m) need = std::max(need, plan_gemm(m, n, k, max_ws).ws_bytes);
  return need;
}

Plan plan_grouped(uint32_t m, uint32_t k, const uint32_t* ns, uint32_t count) {
  // Members share X and launch together: plan as one GEMM of the summed width
  // (the table's row for that width is measured on the grouped launch where
  // the engine has one), unless the members' own stripe rounding would add a
  // round of 256 tiles to that plan; then the model picks, counting the
  // stripes member by member.
  uint32_t n_total = 0;
  for (uint32_t i = 0; i < count; ++i) n_total += ns[i];
  const Plan p = plan_gemm(m, n_total, k, 0);
  if (p.variant == kStreamVariant) return p;
  // the width whose single-GEMM stripe count equals the grouped one for variant v
  auto grouped_n = [&](int v) {
    const uint32_t bn = (uint32_t)variant_info(v).bn();
    uint32_t s = 0;
    for (uint32_t i = 0; i < count; ++i) s += ceil_div(ns[i], bn);
    return s * bn;
  };
  const uint32_t cus = (uint32_t)kCUs;
  const uint32_t bn = (uint32_t)variant_info(p.variant).bn();
  if (ceil_div(p.mtiles * (grouped_n(p.variant) / bn), cus) <= ceil_div(p.grid, cus)) return p;
  Plan best = p;
  double best_us = std::numeric_limits<double>::infinity();
  for (int v = 0; v < variant_count(); ++v) {
    const double t = plan_estimate_us(v, 1, m, grouped_n(v), k);
    if (t < best_us) {
      best_us = t;
      best = plan_make(v, 1, m, n_total, k);
    }
  }
  return best;
}

namespace {
// Bytes-per-K of the distinct X tiles (bm rows each) and W stripes (bn columns
// each) that work ids [a, b) of one split touch in the order of group width g.
double span_cost(uint32_t a, uint32_t b, uint32_t mtiles, uint32_t nstripes, uint32_t g, double bm, double bn) {
  if (a >= b) return 0.0;
  if (g == 0) {
    const uint32_t dm = std::min(b - a, mtiles), ds = (b - 1) / mtiles - a / mtiles + 1;
    return dm * bm + ds * bn;
  }
  const uint32_t gw = mtiles * g;
  double cost = 0.0;
  for (uint32_t grp = a / gw; grp * gw < b; ++grp) {
    const uint32_t gsz = std::min(g, nstripes - grp * g);
    const uint32_t base = grp * gw, lo = std::max(a, base) - base, hi = std::min(b, base + mtiles * gsz) - base;
    if (lo >= hi) continue;
    const uint32_t ds = std::min(hi - lo, gsz), dm = (hi - 1) / gsz - lo / gsz + 1;
    cost += dm * bm + ds * bn;
  }
  return cost;
}

double order_cost(const Plan& p, uint32_t g, double bm, double bn) {
  constexpr uint32_t kXcds = 8, kSlots = 32;  // workgroups per XCD per round (one per CU)
  constexpr uint32_t kRounds = 4;  // rounds counted per XCD: later ones repeat the pattern, and this bounds host time
  const uint32_t per_split = p.mtiles * p.stripes, per = p.grid / kXcds, extra = p.grid % kXcds;
  double cost = 0.0;
  for (uint32_t x = 0; x < kXcds; ++x) {
    const uint32_t start = x * per + std::min(x, extra), count = per + (x < extra ? 1u : 0u);
    for (uint32_t j = 0; j < count && j < kRounds * kSlots; j += kSlots) {
      uint32_t a = start + j;
      const uint32_t b = start + std::min(count, j + kSlots);
      while (a < b) {  // split boundaries: each split reads its own K range
        const uint32_t s = a / per_split, e = std::min(b, (s + 1) * per_split);
        cost += span_cost(a - s * per_split, e - s * per_split, p.mtiles, p.stripes, g, bm, bn);
        a = e;
      }
    }
  }
  return cost;
}

// DH_GEMM_TILE_GROUP=<g>: -1 (unset, or not a number in 0..64) lets the planner choose; 0..64 fixes the order
// (widths past a launch's stripe count act as one group; the cap keeps mtiles · g far from wrapping in the kernel).
int env_tile_group() {
  static const int v = [] {
    const char* e = std::getenv("DH_GEMM_TILE_GROUP");
    if (!e || !*e) return -1;
    char* end = nullptr;
    const long g = std::strtol(e, &end, 10);
    return *end == '\0' && g >= 0 && g <= 64 ? (int)g : -1;
  }();
  return v;
}
}  // namespace

uint32_t plan_order(const Plan& p) {
  if (p.variant == kStreamVariant || p.grid == 0) return 0;
  if (env_tile_group() >= 0) return (uint32_t)env_tile_group();
  if (p.mtiles < 2 || p.stripes < 2) return 0;
  // a forward plans the same few shapes in every layer: the last answers per thread, keyed by what they depend on
  struct Memo {
    int variant = -1;
    uint32_t mtiles = 0, stripes = 0, splits = 0, order = 0;
  };
  thread_local Memo memo[8];
  Memo& mo = memo[(p.mtiles * 31u + p.stripes * 7u + p.splits * 3u + (uint32_t)p.variant) & 7u];
  if (mo.variant == p.variant && mo.mtiles == p.mtiles && mo.stripes == p.stripes && mo.splits == p.splits)
    return mo.order;
  const VariantInfo v = variant_info(p.variant);
  const double bm = v.bm(), bn = v.bn();
  uint32_t best = 0;
  double best_cost = order_cost(p, 0, bm, bn);
  for (uint32_t g : {1u, 2u, 3u, 4u, 6u, 8u}) {
    if (g >= p.stripes) break;
    const double c = order_cost(p, g, bm, bn);
    if (c < best_cost * 0.98) {  // a clear gain only: otherwise keep the M-fastest order
      best_cost = c;
      best = g;
    }
  }
  mo = Memo{p.variant, p.mtiles, p.stripes, p.splits, best};
  return best;
}

}  // namespace dh
