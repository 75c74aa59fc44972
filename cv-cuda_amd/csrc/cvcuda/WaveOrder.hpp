// Which tile of a tensor each wave of a launch works on. Plain arithmetic, the same on the host and the device.
#ifndef CVCUDA_AMD_WAVEORDER_HPP
#define CVCUDA_AMD_WAVEORDER_HPP

#include <cstdint>

namespace cvamd {

struct WaveTile // in units of a wave's tile
{
    int x, y;
};

// How the waves of a launch are counted: along the rows of tiles, `across` of them in a row, wherever a block ends; across = 0:
// a block's waves stand below one another.
struct WaveOrder
{
    uint32_t across, magic; // magic: 2^32 / across and a little more (0: across is 1), exact up to 2^32 / across waves
};

constexpr int64_t TilesIn(int64_t size, int64_t tile)
{
    return (size + tile - 1) / tile;
}

// Whether `waves` waves, in blocks of up to four, fit the one dimension of a launch, which has less than 2^32 threads, with a block to
// spare. (Of rows of one or a few tiles there may be more: one column of 67.2 million 12-byte pixels.)
constexpr bool WavesFitARow(int64_t waves)
{
    return ((waves + 3) / 4 + 1) * 256 < (int64_t)1 << 32;
}

constexpr WaveOrder AlongRows(int dstW, int dstH, int waveW, int waveH)
{
    const int64_t across = TilesIn(dstW, waveW), down = TilesIn(dstH, waveH);
    if (across * across * down >= (int64_t)1 << 32 || !WavesFitARow(across * down))
    {
        return WaveOrder{0, 0};
    }
    return WaveOrder{(uint32_t)across, across == 1 ? 0u : (uint32_t)(((uint64_t)1 << 32) / (uint64_t)across + 1)};
}

// The tiles of a row where a launch's waves, of one row each, are counted along the rows and divided by them; 0: more waves than fit.
constexpr int TilesAlongRows(int dstW, int dstH, int waveW)
{
    const int64_t across = TilesIn(dstW, waveW);
    return WavesFitARow(across * dstH) ? (int)across : 0;
}

// The tile of wave `wave` of the `waves` in block (blockX, blockY).
constexpr WaveTile TileOfWave(const WaveOrder &order, uint32_t blockX, uint32_t blockY, uint32_t wave, uint32_t waves)
{
    // (arithmetic, not a branch: behind a branch the compiler loads the kernel's other arguments only after
    // that test, one more round trip to memory before a wave's first pixel load, 0.3 us on the 4 - 6 us launches of small
    // batches)
    const uint32_t along = blockX * waves + wave, row = order.magic == 0 ? along : (uint32_t)(((uint64_t)along * order.magic) >> 32);
    const bool     stacked = order.across == 0;
    return WaveTile{(int)(stacked ? blockX : along - row * order.across), (int)(stacked ? blockY * waves + wave : row)};
}

// The blocks of a launch whose waves own tiles of waveW x waveH, `waves` of them to a block.
struct WaveBlocks
{
    uint32_t x, y;
};

// Blocks go to the 8 XCDs in turn and on each of them to its 4 shader engines. Where an image has a multiple of 16 or of 32 blocks, the same
// part of every image therefore lands on the same CUs, and the blocks of its last rows, whose waves take the guarded forms, several times longer, all on
// an eighth or a thirty-second of them. One block more, below the image, moves each image on by one. us without / with it: nearest neighbour
// u8x3 168 x 708 x 29 -> 1533 x 82 33.0 / 22.0, 67 x 259 x 52 -> 931 x 128 13.9 / 9.4; means over images of a multiple of 16 and of 32, nearest
// neighbour u8x3 0.93 and 0.87 of the time, u8x1 0.96 and 0.93, bilinear strips 0.80 and 0.75, bicubic u8x3 0.97, others 1.00. Of 8 blocks it
// gains less than the block costs (u8x3 1.02), and so it is with blocks of one wave, whose launches are short: 1.00 to 1.02 in the means of 30 classes, 8 x
// 1080p u8x3 -> 224 x 224 4.11 / 4.16 us, u8x1 bilinear 3.87 / 4.14.
constexpr WaveBlocks BlocksOfWaves(int dstW, int dstH, int waveW, int waveH, const WaveOrder &order, int waves)
{
    if (order.across == 0)
    {
        return WaveBlocks{(uint32_t)TilesIn(dstW, waveW), (uint32_t)TilesIn(dstH, (int64_t)waves * waveH)};
    }
    const uint32_t blocks = (uint32_t)TilesIn(order.across * TilesIn(dstH, waveH), waves);
    return WaveBlocks{waves > 1 && blocks % 16 == 0 ? blocks + 1 : blocks, 1};
}

} // namespace cvamd

#endif // CVCUDA_AMD_WAVEORDER_HPP
