// The 4096-word rows on the matrix cores.
//
// Bound by VALU issue: 234 VALU instructions per word (376 with register DFTs), the 24 matrix
// instructions of a wave per word of its lanes among them; without its loads and stores the kernel takes 34 of its 43 us at
// n = 2^22, without the matrix instructions as well 28.  128 registers keep four waves per
// SIMD (48 hold the DFT matrix; three waves, or the next group's words fetched ahead at that
// cost, measured 45 us).
//
// Groups per wave: a row of 16 waves with one group each ends soonest while every row has a
// compute unit to itself; more rows than that run as rows of four waves with four groups each,
// four such workgroups on a unit.  Row pass, one group against four: R = 16 10.4 / 14.5 us,
// R = 256 12.8 / 16.4, R = 512 25.3 / 24.9, R = 1024 48.1 / 43.1, R = 2048 88.6 / 75.8.
#include "lnt_launch.hpp"

template <int GW>
static void go_row16(const lnt::Plan &pl, const LntParams &P, hipStream_t s, int mode) {
    dim3 grid(pl.R), block(1024 / GW);
    if (mode == LNT_FORWARD)
        hipLaunchKernelGGL((lnt_k_row16<GW, LNT_FORWARD>), grid, block, 0, s, P);
    else if (mode == LNT_MULTIPLY)
        hipLaunchKernelGGL((lnt_k_row16<GW, LNT_MULTIPLY>), grid, block, 0, s, P);
    else
        hipLaunchKernelGGL((lnt_k_row16<GW, LNT_SQUARE>), grid, block, 0, s, P);
}

// Compute units of an MI355X: rows up to this many run one per unit.
static constexpr u32 ROW16_WIDE = 256;

bool lnt_launch_row16(const lnt::Plan &pl, const LntParams &P, hipStream_t s, int mode) {
    if (pl.row3 != 16 || pl.C != 4096) return false;
    // the product modes share the transform-domain slots, so the choice is by R alone
    if (pl.R <= ROW16_WIDE)
        go_row16<1>(pl, P, s, mode);
    else
        go_row16<4>(pl, P, s, mode);
    return true;
}

bool lnt_launch_batch_row16(const lnt::Plan &pl, const LntParams *Ps, u32 count, hipStream_t s) {
    if (pl.row3 != 16 || pl.C != 4096) return false;
    // by all slots, of which a group has eight at least: the wide form is for up to 32 rows, whose
    // launch is one row's latency whatever the slots hold
    if (pl.R * count <= ROW16_WIDE)
        hipLaunchKernelGGL(lnt_kb_row16<1>, dim3(pl.R * count), dim3(1024), 0, s, Ps, pl.R);
    else
        hipLaunchKernelGGL(lnt_kb_row16<4>, dim3(pl.R * count), dim3(256), 0, s, Ps, pl.R);
    return true;
}
