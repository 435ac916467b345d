// Columns of 256 and 1024 words on the matrix cores (the 1024-word ones take about as long as the
// 3-phase kernels: with one tile per compute unit the load, the carry, the transform and the
// store follow each other there, and only the transform got shorter).
//
// Of 128 registers 48 hold the DFT matrix.  The 1024-word forward kernel spills 6 (28 bytes per
// lane, which is the 39.8 MB written per launch at n = 2^22 where the tile is 33.6; 27 with a halo
// of eight digits), the four-wave form of the 256-word one 2 (24); the others spill none.
//
// Batches with more tiles than compute units run the 256-word tiles
// with 4 waves of four groups each, four tiles on a unit that work past each other's loads and
// barriers, where one test takes 16 waves a tile: per squaring of all, 16 tests of 2^20 402 -> 334 us,
// 13 of 2^18 94 -> 79, one test of 2^20 in eight slots 81 -> 62; with fewer tiles the 16 waves stay
// ahead (6 tests of 2^18 53 against 63).  A quarter of the slots is counted: a group is formed with
// two to four slots for each member, from five members on, and its graph stays the same while
// members come and go, so a group that most members left keeps the form of its slots.
#include "lnt_launch.hpp"

// Compute units of an MI355X.
static constexpr u32 COLM_UNITS = 256;

bool lnt_launch_colm_fwd(const lnt::Plan &pl, const LntParams &P, bool sub2, hipStream_t s) {
    if (pl.R != 256 * pl.colm || pl.K != 16) return false;
    const dim3 grid(pl.C / 16), block(1024);
#define CM(S)                                                                                              \
    if (pl.colm == S) {                                                                                    \
        if (pl.M == 4) hipLaunchKernelGGL((lnt_k_colm_fwd<S, 4>), grid, block, 0, s, P, (int)sub2);        \
        else hipLaunchKernelGGL((lnt_k_colm_fwd<S, 8>), grid, block, 0, s, P, (int)sub2);                  \
        return true;                                                                                       \
    }
    CM(1) CM(4)
#undef CM
    return false;
}

bool lnt_launch_colm_inv(const lnt::Plan &pl, const LntParams &P, hipStream_t s) {
    if (pl.R != 256 * pl.colm || pl.K != 16) return false;
    const dim3 grid(pl.C / 16), block(1024);
#define CM(S)                                                              \
    if (pl.colm == S) {                                                    \
        hipLaunchKernelGGL(lnt_k_colm_inv<S>, grid, block, 0, s, P);       \
        return true;                                                       \
    }
    CM(1) CM(4)
#undef CM
    return false;
}

bool lnt_launch_batch_colm_fwd(const lnt::Plan &pl, const LntParams *Ps, u32 count, hipStream_t s) {
    if (pl.R != 256 * pl.colm || pl.K != 16) return false;
    const u32 wgs = pl.C / 16;
    const dim3 grid(wgs * count);
#define CM(S, W)                                                                                         \
    {                                                                                                    \
        if (pl.M == 4) hipLaunchKernelGGL((lnt_kb_colm_fwd<S, 4, W>), grid, dim3(64 * W), 0, s, Ps, wgs); \
        else hipLaunchKernelGGL((lnt_kb_colm_fwd<S, 8, W>), grid, dim3(64 * W), 0, s, Ps, wgs);          \
        return true;                                                                                     \
    }
    if (pl.colm == 4) CM(4, 16)
    if (pl.colm == 1 && wgs * (count / 4) > COLM_UNITS) CM(1, 4)
    if (pl.colm == 1) CM(1, 16)
#undef CM
    return false;
}

bool lnt_launch_batch_colm_inv(const lnt::Plan &pl, const LntParams *Ps, u32 count, hipStream_t s) {
    if (pl.R != 256 * pl.colm || pl.K != 16) return false;
    const u32 wgs = pl.C / 16;
    const dim3 grid(wgs * count);
#define CM(S, W)                                                                           \
    {                                                                                      \
        hipLaunchKernelGGL((lnt_kb_colm_inv<S, W>), grid, dim3(64 * W), 0, s, Ps, wgs);    \
        return true;                                                                       \
    }
    if (pl.colm == 4) CM(4, 16)
    if (pl.colm == 1 && wgs * (count / 4) > COLM_UNITS) CM(1, 4)
    if (pl.colm == 1) CM(1, 16)
#undef CM
    return false;
}
