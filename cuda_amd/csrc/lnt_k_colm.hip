// Columns of 256 and 1024 words on the matrix cores (the 1024-word ones take about as long as the
// 3-phase kernels: with one tile per compute unit the load, the carry, the transform and the
// store follow each other there, and only the transform got shorter).
#include "lnt_launch.hpp"

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
    const dim3 grid(wgs * count), block(1024);
#define CM(S)                                                                                \
    if (pl.colm == S) {                                                                      \
        if (pl.M == 4) hipLaunchKernelGGL((lnt_kb_colm_fwd<S, 4>), grid, block, 0, s, Ps, wgs); \
        else hipLaunchKernelGGL((lnt_kb_colm_fwd<S, 8>), grid, block, 0, s, Ps, wgs);        \
        return true;                                                                         \
    }
    CM(1) CM(4)
#undef CM
    return false;
}

bool lnt_launch_batch_colm_inv(const lnt::Plan &pl, const LntParams *Ps, u32 count, hipStream_t s) {
    if (pl.R != 256 * pl.colm || pl.K != 16) return false;
    const u32 wgs = pl.C / 16;
    const dim3 grid(wgs * count), block(1024);
#define CM(S)                                                              \
    if (pl.colm == S) {                                                    \
        hipLaunchKernelGGL(lnt_kb_colm_inv<S>, grid, block, 0, s, Ps, wgs); \
        return true;                                                       \
    }
    CM(1) CM(4)
#undef CM
    return false;
}
