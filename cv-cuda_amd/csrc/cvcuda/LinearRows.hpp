// Where the whole rows of ResizeLinearRowsKernel stand in LDS, and how many of its blocks a CU has room for.
#ifndef CVCUDA_AMD_LINEARROWS_HPP
#define CVCUDA_AMD_LINEARROWS_HPP

namespace cvamd {

constexpr int kLdsBytes = 163840, kLdsPiece = 1280; // of a CU, and what a block's share of it is a multiple of

// Floats from one staged row to the next: dense rows follow one another as they do in memory, others each start behind as much as a row's
// distance from a 128-byte boundary may be.
constexpr int LinearRowsPitch(int dstW, bool dense)
{
    return dense ? dstW : ((dstW + 3) & ~3) + 32;
}

// LDS bytes of a block of `rows` rows (dense ones: behind the block's own distance from such a boundary).
constexpr int LinearRowsLds(int dstW, bool dense, int rows)
{
    return (rows * LinearRowsPitch(dstW, dense) + (dense ? 32 : 0)) * 4;
}

constexpr int BlocksPerCu(int lds)
{
    return kLdsBytes / ((lds + kLdsPiece - 1) / kLdsPiece * kLdsPiece);
}

} // namespace cvamd

#endif // CVCUDA_AMD_LINEARROWS_HPP
