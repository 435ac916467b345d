// Rows of 256 .. 2048 words on the matrix cores, one row per workgroup of a wave per 256 words
// with four words per thread: as long as the rows do not fill the chip a row pass is the latency
// of one row, 3.7 us at 256 words, 4.7 at 512, 5.3 at 1024, 7.0 at 2048 (the 2-phase kernels
// with 16 .. 64 words per thread take 12 us for 128 and 13.8 for 256 words).
#include "lnt_launch.hpp"

// Batches that fill the chip: the 2048-word kernel's 166 registers leave a unit one workgroup of
// eight waves, which waits for its own loads and exchanges.  Four rows per workgroup at 128
// registers (lnt_rowm_rows_body; 4 spilled) let two workgroups share a unit: 11 tests of 2^19 178 -> 152 us
// per squaring of all.  With the rows of 14 tests of 2^17 (64 each) it gains nothing (62 / 60 us),
// and the shorter rows already run several workgroups per unit (13 tests of 2^18 94 / 98 us).
static constexpr u32 ROWM_ROWS = 4, ROWM_FULL = 1024;

template <int S>
static void go_rowm(const lnt::Plan &pl, const LntParams &P, hipStream_t s, int mode) {
    dim3 grid(pl.R), block(64 * S);
    if (mode == LNT_FORWARD)
        hipLaunchKernelGGL((lnt_k_rowm<S, LNT_FORWARD>), grid, block, 0, s, P);
    else if (mode == LNT_MULTIPLY)
        hipLaunchKernelGGL((lnt_k_rowm<S, LNT_MULTIPLY>), grid, block, 0, s, P);
    else
        hipLaunchKernelGGL((lnt_k_rowm<S, LNT_SQUARE>), grid, block, 0, s, P);
}

bool lnt_launch_rowm(const lnt::Plan &pl, const LntParams &P, hipStream_t s, int mode) {
    if (pl.C != 256 * pl.rowm) return false;
    switch (pl.rowm) {
        case 1: go_rowm<1>(pl, P, s, mode); return true;
        case 2: go_rowm<2>(pl, P, s, mode); return true;
        case 4: go_rowm<4>(pl, P, s, mode); return true;
        case 8: go_rowm<8>(pl, P, s, mode); return true;
    }
    return false;
}

bool lnt_launch_batch_rowm(const lnt::Plan &pl, const LntParams *Ps, u32 count, hipStream_t s) {
    if (pl.C != 256 * pl.rowm) return false;
    const dim3 block(64 * pl.rowm);
    // a quarter of the slots, as for the columns (lnt_k_colm.hip)
    if (pl.rowm == 8 && pl.R % ROWM_ROWS == 0 && pl.R * (count / 4) >= ROWM_FULL) {
        const u32 wgs = pl.R / ROWM_ROWS;
        hipLaunchKernelGGL((lnt_kb_rowm_rows<8, ROWM_ROWS>), dim3(wgs * count), block, 0, s, Ps, wgs);
        return true;
    }
    const dim3 grid(pl.R * count);
    switch (pl.rowm) {
        case 1: hipLaunchKernelGGL(lnt_kb_rowm<1>, grid, block, 0, s, Ps, pl.R); return true;
        case 2: hipLaunchKernelGGL(lnt_kb_rowm<2>, grid, block, 0, s, Ps, pl.R); return true;
        case 4: hipLaunchKernelGGL(lnt_kb_rowm<4>, grid, block, 0, s, Ps, pl.R); return true;
        case 8: hipLaunchKernelGGL(lnt_kb_rowm<8>, grid, block, 0, s, Ps, pl.R); return true;
    }
    return false;
}
