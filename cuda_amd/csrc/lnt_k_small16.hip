// The single-workgroup kernels on the matrix cores, n = 64 .. 4096.
//
// One test on one compute unit is bound by the latency of its dependent steps.  Microseconds
// per squaring against the register-DFT kernels before (8, 16 or 64 words per thread; n = 2048
// as three launches): n = 64 1.3 / 7.7, 128 2.0 / 16.4, 256 2.6 / 17.1, 512 3.3 / 7.2, 1024 3.5 / 40.8, 2048 4.7 / 21.9,
// 4096 9.4 / 24.6.  Built with the max-ilp machine scheduler (-amdgpu-sched-strategy=max-ilp,
// set for this file in the Makefile): with at most four waves per SIMD nothing else hides the
// wait states of the carry chains (n = 256 .. 2048 2.8, 3.6, 4.1, 4.8 us without, 4096 equal).
// At n = 4096 the addresses are formed again in every iteration: kept across it they spilled
// (14.4 us).  Registers still spilled per lane: n = 2048 4 of 256 (12 with a halo of eight
// digits), n = 4096 none of 128 (12), the others none.
#include "lnt_launch.hpp"

template <int S, int M>
static void go_small16_m(const LntParams &P, u32 iters, bool sub2_first, bool ll, hipStream_t s, int mode) {
    dim3 grid(1), block(64 * S);
    if (mode == LNT_FORWARD)
        hipLaunchKernelGGL((lnt_k_small16<S, M, LNT_FORWARD>), grid, block, 0, s, P, 1u, (int)sub2_first, (int)ll);
    else if (mode == LNT_MULTIPLY)
        hipLaunchKernelGGL((lnt_k_small16<S, M, LNT_MULTIPLY>), grid, block, 0, s, P, 1u, (int)sub2_first, (int)ll);
    else
        hipLaunchKernelGGL((lnt_k_small16<S, M, LNT_SQUARE>), grid, block, 0, s, P, iters, (int)sub2_first, (int)ll);
}

template <int N1, int M>
static void go_tiny_m(const LntParams &P, u32 iters, bool sub2_first, bool ll, hipStream_t s, int mode) {
    if (mode == LNT_FORWARD)
        hipLaunchKernelGGL((lnt_k_tiny<N1, M, LNT_FORWARD>), dim3(1), dim3(64), 0, s, P, 1u, (int)sub2_first, (int)ll);
    else if (mode == LNT_MULTIPLY)
        hipLaunchKernelGGL((lnt_k_tiny<N1, M, LNT_MULTIPLY>), dim3(1), dim3(64), 0, s, P, 1u, (int)sub2_first, (int)ll);
    else
        hipLaunchKernelGGL((lnt_k_tiny<N1, M, LNT_SQUARE>), dim3(1), dim3(64), 0, s, P, iters, (int)sub2_first,
                           (int)ll);
}

template <int N1>
static bool go_tiny(const lnt::Plan &pl, const LntParams &P, u32 iters, bool sub2_first, bool ll, hipStream_t s,
                    int mode) {
    if (pl.M == 4) go_tiny_m<N1, 4>(P, iters, sub2_first, ll, s, mode);
    else go_tiny_m<N1, 8>(P, iters, sub2_first, ll, s, mode);
    return true;
}

template <int N1>
static bool go_batch_tiny(const lnt::Plan &pl, const LntParams *Ps, u32 count, u32 iters, bool ll, hipStream_t s) {
    if (pl.M == 4) hipLaunchKernelGGL((lnt_kb_tiny<N1, 4>), dim3(count), dim3(64), 0, s, Ps, iters, (int)ll);
    else hipLaunchKernelGGL((lnt_kb_tiny<N1, 8>), dim3(count), dim3(64), 0, s, Ps, iters, (int)ll);
    return true;
}

bool lnt_launch_small16(const lnt::Plan &pl, const LntParams &P, u32 iters, bool sub2_first, bool ll, hipStream_t s,
                        int mode) {
    if (pl.tiny && pl.n == 64) return go_tiny<8>(pl, P, iters, sub2_first, ll, s, mode);
    if (pl.tiny && pl.n == 128) return go_tiny<16>(pl, P, iters, sub2_first, ll, s, mode);
    if (pl.n != 256 * pl.small16) return false;
#define SM(S)                                                                 \
    if (pl.small16 == S) {                                                    \
        if (pl.M == 4) go_small16_m<S, 4>(P, iters, sub2_first, ll, s, mode); \
        else go_small16_m<S, 8>(P, iters, sub2_first, ll, s, mode);           \
        return true;                                                          \
    }
    SM(1) SM(2) SM(4) SM(8) SM(16)
#undef SM
    return false;
}

bool lnt_launch_batch_small16(const lnt::Plan &pl, const LntParams *Ps, u32 count, u32 iters, bool ll, hipStream_t s) {
    if (pl.tiny && pl.n == 64) return go_batch_tiny<8>(pl, Ps, count, iters, ll, s);
    if (pl.tiny && pl.n == 128) return go_batch_tiny<16>(pl, Ps, count, iters, ll, s);
    if (pl.n != 256 * pl.small16) return false;
#define SM(S)                                                                                                     \
    if (pl.small16 == S) {                                                                                        \
        if (pl.M == 4) hipLaunchKernelGGL((lnt_kb_small16<S, 4>), dim3(count), dim3(64 * S), 0, s, Ps, iters, (int)ll); \
        else hipLaunchKernelGGL((lnt_kb_small16<S, 8>), dim3(count), dim3(64 * S), 0, s, Ps, iters, (int)ll);     \
        return true;                                                                                              \
    }
    SM(1) SM(2) SM(4) SM(8) SM(16)
#undef SM
    return false;
}
