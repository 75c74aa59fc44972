// The staged rows of ResizeLinearRowsKernel (cvcuda/LinearRows.hpp): what is written and read of them lies in the block's LDS, and each width has the
// number of blocks per CU that its rows leave room for. Prints "ok".
#include <LinearRows.hpp>

#include <cstdio>
#include <initializer_list>

using namespace cvamd;

int main()
{
    int bad = 0;
    for (int w = 96; w < 10000; ++w)
    {
        for (int rows : {4, 8, 16})
        {
            for (int used : {1, 3, rows - 1, rows})
            {
                for (int lead = 0; lead < 32; ++lead)
                {
                    // floats are read by fours from the boundary on, up to behind the last one
                    const int dense = (lead + used * w + 3) / 4 * 4, last = (used - 1) * LinearRowsPitch(w, false) + (lead + w + 3) / 4 * 4;
                    bad += dense * 4 > LinearRowsLds(w, true, rows) || last * 4 > LinearRowsLds(w, false, rows);
                    bad += lead + w > LinearRowsPitch(w, false) || LinearRowsPitch(w, false) % 4 != 0;
                }
            }
        }
    }
    struct
    {
        int  w;
        bool dense;
        int  blocks;
    } const widths[] = {{1917, true, 5}, {2500, true, 4}, {2552, true, 4}, {2553, true, 3}, {3352, true, 3}, {3353, true, 2}, {3840, true, 2},
                        {2497, false, 4}, {2528, false, 4}, {2529, false, 3}, {3328, false, 3}, {3329, false, 2}};
    for (const auto &c : widths)
    {
        if (BlocksPerCu(LinearRowsLds(c.w, c.dense, 4)) != c.blocks)
        {
            std::printf("%d floats%s: %d blocks\n", c.w, c.dense ? ", dense" : "", BlocksPerCu(LinearRowsLds(c.w, c.dense, 4)));
            ++bad;
        }
    }
    std::puts(bad == 0 ? "ok" : "bad");
    return bad != 0;
}
