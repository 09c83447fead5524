// Which sizes may run on MFMA tiles as far as the results are concerned.
//
// Strips, column blocks and the batch kernel multiply sums by the scale in fp32; the MFMA tiles multiply the weights, which
// rounds each of them to fp16 as the reference does, and with up to 256 sums per lane have no registers for the other form.
// The first is the more accurate, so a size that has been computed that way stays with it, whatever the two cost: a default
// choice never moves an existing size to rounded weights.  Two sets of sizes are kept out of the tiles:
//
// * Every size that the streaming kernels were given when the tiles were priced against them alone, before the batch kernel
//   (first_choice_streams).  The prices of that comparison are what defines the set; the kernels they describe are gone or
//   have changed, and they are not costs of anything today (those are in api.cpp).
// * Sizes that moved from tiles to the batch kernel since (moved_to_fp32).  Bounds on size, inside which it was given
//   everything; with 16 groups of K and more it is also the faster one there (us, batch kernel against the best tile, cold
//   weights: 8192 x 16384 at 80 tokens 31.8 against 43.2, 4096 x 4096 at 244 13.2 against 17.6, 8192 x 1024 at 976 27.2
//   against 27.4, 14336 x 2048 at 488 37.5 against 42.8).  With fewer groups, and where N is an odd multiple of 64, the
//   precision costs time: 1536 x 16384 at 160 20.2 against 16.6, 512 x 8192 at 600 26.1 against 9.7, 4096 x 11200 at 384 57.0
//   against 43.4, 4096 x 22080 at 2048 574 against 308.  So it does in the first set (4096 x 10944 at 3329 509 against 295,
//   1664 x 9920 at 641 58 against 28).  No matrix of the 7B and 70B layers is that wide.
#include "w4a16_internal.h"

#include <cmath>

namespace w4a16 {

namespace {

constexpr int kTileRowsK = 128;

// The tiles of the first comparison: microseconds per K step for the whole grid at 1, 2, 3, 4 and 8 workgroups per CU; `alone`
// for those that filled a CU by themselves and went in whole rounds; K steps in multiples of `depth`.
struct FirstTile {
    int   tile_t, tile_n, depth;
    bool  alone;
    float step_us[5];
};
constexpr FirstTile kFirstTiles[] = {
    {128, 256, 2, true, {1.810f, 3.630f, 5.240f, 6.740f, 12.980f}},
    {256, 128, 2, true, {2.071f, 4.498f, 6.126f, 8.397f, 15.010f}},
    {128, 128, 2, false, {1.016f, 1.860f, 3.067f, 4.002f, 7.185f}},
    {64, 128, 4, false, {0.672f, 1.111f, 1.664f, 2.271f, 4.773f}},
    {64, 64, 4, false, {0.425f, 0.673f, 1.000f, 1.340f, 2.833f}},
    {64, 128, 4, true, {0.553f, 1.209f, 1.906f, 2.609f, 5.351f}},
    {64, 256, 4, true, {1.034f, 2.290f, 3.605f, 4.644f, 8.583f}},
};

bool first_tile_fits(const FirstTile& t, int splits, int N, int T, int K, const Scratch& lim)
{
    if (N % t.tile_n != 0 || (int64_t)T * K * 2 >= (1ll << 32) || (int64_t)N * 64 >= (1ll << 32)) return false;
    const int64_t grid = (int64_t)(N / t.tile_n) * ((T + t.tile_t - 1) / t.tile_t);
    if (splits > 1) {
        if (t.tile_t > 128 || K / kTileRowsK < 2 * splits) return false;
        if (grid * splits * t.tile_n * t.tile_t * 4 > (int64_t)lim.ws_bytes || grid > lim.cnt_len) return false;
    }
    return grid * splits < (1ll << 31);
}

double first_tile_us(const FirstTile& t, int splits, int N, int T, int K)
{
    const double load = (double)(N / t.tile_n) * ((T + t.tile_t - 1) / t.tile_t) * splits / 256.0;
    const double le   = t.alone ? std::ceil(load) : load;
    double       step;
    if (le <= 4.0) step = t.step_us[le <= 1.0 ? 0 : le <= 2.0 ? 1 : le <= 3.0 ? 2 : 3];
    else if (le <= 8.0) step = t.step_us[3] + (t.step_us[4] - t.step_us[3]) * (le - 4.0) / 4.0;
    else step = t.step_us[4] * le / 8.0;
    if (t.alone && load < 1.0) step *= 0.7 + 0.3 * load;
    if (!t.alone && t.tile_t == 64 && load > 2.0) step *= 1.25;
    const int each = (K / kTileRowsK + splits - 1) / splits;
    double    us   = 3.0 + (each + t.depth - 1) / t.depth * t.depth * step;
    if (splits > 1) us += 2.0 + 0.6 * splits + splits * ((double)((T + t.tile_t - 1) / t.tile_t) * t.tile_t) * N * 8.0 / 4.0e6;
    return us;
}

bool first_choice_streams(int N, int T, int K, const Scratch& lim)
{
    // the weights once per 16 tokens, later passes partly from the caches
    const double stream_us = 3.0 + std::pow((T + 15) / 16, 0.85) * ((double)K * N / 2) / 4.2e6 * (N / 16 < 512 ? 1.4 : 1.0);
    for (const FirstTile& t : kFirstTiles)
        for (int splits : {1, 2, 4, 8})
            if (first_tile_fits(t, splits, N, T, K, lim) && first_tile_us(t, splits, N, T, K) < stream_us) return false;
    return true;
}

bool moved_to_fp32(int N, int T, int K)
{
    const int     groups  = K / kTileRowsK;
    const int64_t outputs = (int64_t)N * T;
    if (N % 128 != 0 && (T <= 384 || N > 22016 || groups <= 10 || outputs <= 1300000)) return true;
    return (groups < 16 ? T <= 160 : T <= 80 && outputs <= 1400000) || outputs <= (groups < 8 ? 5000000 : 1000000);
}

}  // namespace

bool scales_in_fp32(int nq, int N, int T, int K, const Scratch& lim)
{
    const int groups = K / kTileRowsK;
    if (N % 64 != 0 || T <= 32 || groups < 2 || (nq > 1 && N % 128 != 0)) return true;
    if (nq > 1) {
        // (as long as the weights, streamed once per 16 tokens, took less than the K steps of 256 x 128 tiles)
        const double tiles_us = 3.0 + std::ceil((T + 255) / 256 * (N / 128) / 256.0) * groups * 2.4;
        return (T + 15) / 16 * (3.0 + (double)K * N / 6.0e6) <= tiles_us;
    }
    return moved_to_fp32(N, T, K) || first_choice_streams(N, T, K, lim);
}

}  // namespace w4a16
