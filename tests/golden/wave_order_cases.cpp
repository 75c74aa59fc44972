// The map from a launch's waves to the tiles of an image (cvcuda/WaveOrder.hpp): every tile once, surplus waves below the image, launches
// within 2^32 threads along each dimension. Prints "ok".
#include <WaveOrder.hpp>

#include <cstdio>
#include <vector>

using namespace cvamd;

static int s_bad = 0;

static void Check(bool good, const char *what, int w, int h, int tileW, int tileH, int waves)
{
    if (!good && ++s_bad < 20)
    {
        std::printf("%s: %d x %d in tiles of %d x %d, %d waves to a block\n", what, w, h, tileW, tileH, waves);
    }
}

static void EveryTileOnce(int w, int h, int tileW, int tileH, int waves, const WaveOrder &order)
{
    const WaveBlocks blocks = BlocksOfWaves(w, h, tileW, tileH, order, waves);
    const int        across = (w + tileW - 1) / tileW, down = (h + tileH - 1) / tileH;
    Check(order.across == 0 || waves == 1 || blocks.x % 16 != 0, "blocks", w, h, tileW, tileH, waves);
    Check(waves > 1 || (int64_t)blocks.x * blocks.y == (int64_t)across * down, "single waves", w, h, tileW, tileH, waves);
    std::vector<int> seen((size_t)across * down);
    for (uint32_t y = 0; y < blocks.y; ++y)
    {
        for (uint32_t x = 0; x < blocks.x; ++x)
        {
            for (int k = 0; k < waves; ++k)
            {
                const WaveTile t = TileOfWave(order, x, y, (uint32_t)k, (uint32_t)waves);
                if (t.y < down)
                {
                    Check(t.x >= 0 && t.x < across && t.y >= 0, "place", w, h, tileW, tileH, waves);
                    ++seen[(size_t)t.y * across + t.x];
                }
            }
        }
    }
    for (int n : seen)
    {
        Check(n == 1, "times", w, h, tileW, tileH, waves);
    }
}

// The first, the last and some waves of a launch too large to go through, against the exact division.
static void Ends(int w, int h, int tileW, int tileH, int waves, bool counted)
{
    const WaveOrder  order  = AlongRows(w, h, tileW, tileH);
    const WaveBlocks blocks = BlocksOfWaves(w, h, tileW, tileH, order, waves);
    Check((order.across != 0) == counted, "order", w, h, tileW, tileH, waves);
    Check(order.across == 0 || waves == 1 || blocks.x % 16 != 0, "blocks", w, h, tileW, tileH, waves);
    Check((uint64_t)blocks.x * 64 * (uint64_t)waves < (uint64_t)1 << 32, "threads", w, h, tileW, tileH, waves);
    if (order.across == 0)
    {
        return;
    }
    const uint64_t total = (uint64_t)blocks.x * (uint64_t)waves, tiles = TilesIn(w, tileW) * (uint64_t)TilesIn(h, tileH);
    for (uint64_t i = 0; i < total; i += i < 4096 || i + 4096 >= total ? 1 : 4095)
    {
        const WaveTile t = TileOfWave(order, (uint32_t)(i / waves), 0, (uint32_t)(i % waves), (uint32_t)waves);
        if (i < tiles)
        {
            Check(t.x == (int)(i % order.across) && t.y == (int)(i / order.across), "place", w, h, tileW, tileH, waves);
        }
        else
        {
            Check(t.y >= TilesIn(h, tileH), "surplus", w, h, tileW, tileH, waves);
        }
    }
}

int main()
{
    for (int waves : {1, 4})
    {
        for (int tileW : {64, 256})
        {
            for (int tileH : {1, 4, 16})
            {
                for (int w : {1, 63, 64, 65, 129, 257, 1025, 1917, 4097})
                {
                    for (int h : {1, 3, 4, 5, 16, 17, 64, 255})
                    {
                        const WaveOrder order = AlongRows(w, h, tileW, tileH);
                        Check(order.across != 0, "order", w, h, tileW, tileH, waves);
                        EveryTileOnce(w, h, tileW, tileH, waves, order);
                        EveryTileOnce(w, h, tileW, tileH, waves, WaveOrder{0, 0});
                    }
                }
            }
        }
        // at the limits and one tile past them: 2^26 waves with a block to spare, and products of 2^32 beyond which the division is not exact
        const int most = (1 << 26) - 8;
        Ends(1, most, 64, 1, waves, true);
        Ends(1, most + 1, 64, 1, waves, false);
        Ends(64, 4 * most, 64, 4, waves, true);
        Ends(64, 4 * most + 1, 64, 4, waves, false);
        Ends(3 * 64, most / 3, 64, 1, waves, true);
        Ends(3 * 64, most / 3 + 1, 64, 1, waves, false);
        Ends(97 * 64, (int)((((int64_t)1 << 32) - 1) / (97 * 97)), 64, 1, waves, true);
        Ends(97 * 64, (int)((((int64_t)1 << 32) - 1) / (97 * 97)) + 1, 64, 1, waves, false);
        Ends(128 * 64, (1 << 18) - 1, 64, 1, waves, true);
        Ends(128 * 64, 1 << 18, 64, 1, waves, false);
        Ends(65535 * 64, 1, 64, 1, waves, true);
        Ends(65536 * 64, 1, 64, 1, waves, false);
    }
    // without an order of their own: 4 waves to a block
    for (int tiles : {1, 3, 64})
    {
        const int most = ((1 << 26) - 8) / tiles;
        Check(TilesAlongRows(tiles * 64 - 63, most, 64) == tiles, "fits", tiles * 64 - 63, most, 64, 1, 4);
        Check(TilesIn(tiles * (int64_t)most, 4) * 256 < (int64_t)1 << 32, "threads", tiles * 64 - 63, most, 64, 1, 4);
        Check(TilesAlongRows(tiles * 64, most + 1, 64) == 0, "too many", tiles * 64, most + 1, 64, 1, 4);
    }
    std::puts(s_bad == 0 ? "ok" : "bad");
    return s_bad != 0;
}
