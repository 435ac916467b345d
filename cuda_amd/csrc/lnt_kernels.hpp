// Kernel bodies for one LL/PRP iteration, x <- x^2 (- 2) mod 2^p - 1, as an
// irrational-base weighted NTT over GF(2^64 - 2^32 + 1).
//
// Residue layout (n = R * C words, digit i = c + C * r): natural digit order, each word a
// field element that encodes a signed integer |v| < P/2.  Between iterations the words
// hold the *pre-carry* convolution outputs of the last squaring; the carry (and the LL
// "-2") of iteration k is applied at the start of iteration k+1, fused into the first
// kernel.  Readout normalises on the host.
//
// Transform decomposition (a "line" of L = B1 * B2 words, B1 >= B2, both <= 64):
//   phase 1: thread t < B2 holds words t + B2*j (j < B1), a B1-point register DFT,
//            then the inter-block twiddle omega_L^(t * k2);
//   phase 2: after an LDS transpose, B2-point register DFTs over t.
//   Output X[B1*k1 + k2].  Lines of 256, 512, 1024, 2048 and 4096 words take 16-point DFTs on the
//   matrix cores instead (mdft.hpp; bodies below).  All roots of order <= 64 are powers of two, so the only
//   general twiddle inside a line is the one between the phases.  3-phase lines
//   (rows of 16^3 words, columns of BA * BB * BC words) add one more phase and twiddle.
// Large residues (n >= 2^13) are a 2-D split: C-word rows (contiguous) and R-word
// columns (stride C), with the 4-step twiddle omega_n^(c * kcol) between the column and
// the row transforms.
//
// Per iteration (large path), state x and work buffer y (the carry of one column tile
// reads halo digits of the neighbouring tile, so col_fwd must not write x):
//   col_fwd : x -> y  carry(+ -2) of the previous pre-carry values, weight, column NTT
//   row_sq  : y -> y  4-step twiddle, row NTT, pointwise square, inverse row NTT,
//                     inverse 4-step twiddle
//   col_inv : y -> x  inverse column NTT, unweight (includes 1/n)
// These play the roles of the reference's r2b + m2 + w_fftc_tw (kernels/r2b.cu:25-50,
// kernels/m2.cu:23-41, kernels/w_fftc_tw__r2_8to4k.cu:20-46), fftr_sqr_ifftr
// (kernels/fftr_sqr_ifftr__r2_8to4k.cu:20-56) and tw_ifftc_uw
// (kernels/tw_ifftc_uw__r2_8to4k.cu:20-46).  Small residues (n <= 4096) run the whole
// iteration loop inside one workgroup (the role of w_fft_sqr_ifft_uw__*,
// kernels/w_fft_sqr_ifft_uw__r2_8to4k.cu:20-55, plus r2b and m2).
//
// Carry: "m-level" carry-save normalisation.  Each level splits every value into a
// balanced remainder |lo| <= 2^(w-1) and a carry hi, and adds the carry of the previous
// digit.  After m levels digit j depends only on the pre-carry values j-m..j, so a
// workgroup that owns a run of digits needs just m "halo" values before the run, read
// from memory - no inter-workgroup ordering.  The value sum v_j 2^e_j mod 2^p - 1 is
// preserved exactly (the carry out of digit n-1 enters digit 0 with weight 2^p = 1).
#pragma once
#include "dft.hpp"
#include "mdft.hpp"
#include "simt.hpp"

struct LntParams {
    GView<u64> x;            // n words: residue state (pre-carry values between iterations)
    GView<u64> y;            // n words: transform-domain work buffer
    GView<const u64> w, uw;  // IBDWT weights, unweights * n^-1: n words in digit order (one-workgroup
                             // path: the weights as pairs (w, -2^31 w) at 2i, the unweights at i);
                             // large path: row factors indexed by lnt_wslot, the weights as
                             // pairs at 2 * slot, the unweights at slot
    GView<const u64> tw4, itw4;  // 4-step twiddles (large path), natural slots, times the column
                                 // weight factor (unweight factor * n^-1)
                                 // (all twiddle tables and the large path's unweights are in
                                 // the Montgomery form that gl_mmul takes)
    GView<const u64> twr, itwr;  // row-line twiddles (C words)
    GView<const u64> twr2, itwr2;  // second-level row twiddles (3-phase rows: B^2 words)
    GView<const u64> twc, itwc;  // column-line twiddles (R words)
    GView<const u64> twc2, itwc2;  // second-level column twiddles (3-phase columns: R / BA words)
    GView<const u64> f;      // n words: the other operand of a product, transform domain
    u32 p, n, log_n, C, R;
    u32 levels;              // carry levels m
    u32 sub2;                // batched launches: this test's LL "-2" is due at the next carry
    u32 bias;                // large path: carried digits go to the weight multiply as d + 2^31
};

// Weight exponents on the large path.  Digit i = c + C r has weight B^e_i, e_i = (-p i) mod n
// (B^n = 2), and e_i = e_c + f_r - n [e_c + f_r >= n] with e_c = (-p c) mod n and
// f_r = (-p C r) mod n.  So w_i = B^e_c * B^f_r * 2^-[wrap]: the column factor B^e_c is
// constant down a column and commutes with the column transform, so the 4-step twiddles
// carry it; the row factor B^f_r, or B^f_r / 2 on a wrap, sits in a table of 2R words at
// slot 2r + wrap (unweights likewise: B^-f_r and 2 B^-f_r, with B^-e_c n^-1 in itw4).
GL_HD u32 lnt_wexp(u32 p, u32 n, u64 i) { return (0u - (u32)((u64)p * i)) & (n - 1); }
// mC = -p C mod 2^32 (so f_r = (mC r) mod n, n being a power of two), ec = e_c.
GL_HD u32 lnt_wslot(u32 ec, u32 mC, u32 n, u32 r) {
    const u32 fr = (mC * r) & (n - 1);
    return 2 * r + (ec + fr >= n ? 1u : 0u);
}

// Balanced split of v by width w: v = lo + hi * 2^w, -2^(w-1) <= lo < 2^(w-1).
GL_HD int64_t lnt_split(int64_t v, int w, int64_t &lo) {
    int64_t hi = (v + (int64_t(1) << (w - 1))) >> w;
    lo = (int64_t)((u64)v - ((u64)hi << w));
    return hi;
}

// m-level carry over a run: v[0..M) are the M digits before the run (halo), v[M..M+K)
// the run itself, starting at digit g0.  On return v[M..M+K) hold final digits.
template <int M, int K>
GL_HD void lnt_carry_run(int64_t (&v)[M + K], u32 p, u32 log_n, u64 g0, u32 levels,
                         bool sub2) {
    const u64 n = 1ull << log_n;
    // widths: with R_g = (p g + n - 1) mod n, the width of digit g is
    // floor((R_g + p) / n) = p / n + [R_g + (p mod n) >= n] and R_(g+1) = (R_g + p) mod n;
    // R_n = R_0, so the recurrence runs across the wrap from digit n-1 to digit 0
    const u32 nm = (u32)n - 1, pm = p & nm, wmin = p >> log_n;
    u32 R = ((u32)p * (u32)((g0 + n - M) & (n - 1)) + nm) & nm;
    int w[M + K];
#pragma unroll
    for (int j = 0; j < M + K; j++) {
        const u32 s = R + pm;
        w[j] = (int)(wmin + (s >> log_n));
        R = s & nm;
    }
    // LL "-2" on digit 0, at window position M - g0 when g0 <= M: in the run itself
    // (g0 = 0) or in the halo of a run just after it (every window that holds digit 0 must
    // see the same value); a select per position, no indexing by a run-time value
    if (sub2 && g0 <= (u64)M) {
#pragma unroll
        for (int j = 0; j <= M; j++) v[j] -= (g0 + (u64)j == (u64)M) ? 2 : 0;
    }
    for (u32 l = 0; l < levels; l++) {
        int64_t hprev = 0;
#pragma unroll
        for (int j = 0; j < M + K; j++) {
            int64_t lo;
            int64_t h = lnt_split(v[j], w[j], lo);
            v[j] = lo + hprev;
            hprev = h;
        }
    }
}

// Carry of one piece of a 16-digit run staged in LDS: PR neighbouring threads of one wave share
// the run, thread s takes its digits [s PK, s PK + PK).  row0 is the LDS word of the run's first
// digit, digit g0 of the residue; h holds the M words before the run (for s = 0).  The digits
// go back to LDS as d + 2^31 for the biased weight multiply, else field-encoded.
template <int M, int PK, int PR>
LNT_KFN void lnt_carry_piece(LView lds, u32 row0, int s, const u64 (&h)[M], const LntParams &P, u64 g0, bool sub2) {
    int64_t v[M + PK];
#pragma unroll
    for (int j = 0; j < M; j++) {
        const int at = PK * s - M + j;  // negative: before the run
        u64 x = h[j];
        if (PR > 1 && s) x = (PK < M && at < 0) ? P.x[(g0 + P.n + at) & (P.n - 1)] : lds[row0 + (u32)at];
        v[j] = gl_to_i64(x);
    }
#pragma unroll
    for (int j = 0; j < PK; j++) v[M + j] = gl_to_i64(lds[row0 + (u32)(PK * s + j)]);
    LNT_WAVE_SYNC();  // every word read before any is overwritten
    lnt_carry_run<M, PK>(v, P.p, P.log_n, g0 + PK * s, P.levels, sub2);
#pragma unroll
    for (int j = 0; j < PK; j++)
        lds[row0 + (u32)(PK * s + j)] =
            P.bias ? (u64)(u32)(v[M + j] + (int64_t(1) << 31)) : gl_from_i64(v[M + j]);
}

constexpr int LNT_PAD = 1;

// ------------------------------------------------------------------ column forward
// grid: C / K workgroups (column tile c0 = bid * K), block: K * B2 threads.
// LDS words: lnt_col_fwd_lds<B1, B2, K>().
// Row stride of the carry staging layout: one word of padding keeps the per-row carry
// accesses (one thread per row) on distinct LDS banks while the stage fits in 144 KiB.
template <int B1, int B2, int K>
constexpr int lnt_col_ks() { return B1 * B2 * (K + 1) <= 18432 ? K + 1 : K; }
template <int B1, int B2, int K>
constexpr u32 lnt_col_fwd_lds() {
    return (u32)(B1 * B2 * lnt_col_ks<B1, B2, K>() > B1 * (B2 + LNT_PAD) * K ? B1 * B2 * lnt_col_ks<B1, B2, K>()
                                                                           : B1 * (B2 + LNT_PAD) * K);
}

template <int B1, int B2, int K, int M>
LNT_KFN void lnt_col_fwd_body(int tid, int bid, LView lds, const LntParams &P, bool sub2) {
    constexpr int T = K * B2;
    constexpr int RR = B1 * B2;
    constexpr int RP = B1 / B2;
    constexpr int S = B2 + LNT_PAD;
    constexpr int KS = lnt_col_ks<B1, B2, K>();
    constexpr int RT = (RR + T - 1) / T;  // carry rows per thread
    constexpr int PR = RR < T ? T / RR : 1;  // carry: threads per row where rows are fewer than threads
    const u64 C = P.C;
    const u64 n = P.n;
    const u64 c0 = (u64)bid * K;
    const int cl = tid % K, t = tid / K;
    const u64 c = c0 + cl;
    const u32 ec = lnt_wexp(P.p, P.n, c), mC = 0u - P.p * P.C;  // weight slot parameters

    // 0. loads: the tile (K adjacent lanes read one row run: 8K contiguous bytes), the M
    //    digits before each of this thread's carry rows, and the weights of phase 1.
    // Tables are prefetched into registers when a thread's line fits (B1 <= 32).
    // The halo digits are prefetched too when there are few of them per thread.
    constexpr bool PF = B1 <= 32, HP = RT * M <= 16;
    // short lines (latency-bound passes; registers to spare) fetch the weights' second halves and
    // the twiddles too, here and in the inverse: squaring 2^15 13.85 -> 13.3 us, 2^17 18.1 -> 17.2
    constexpr bool PT = B1 <= 8;
    u64 a[B1], wv[PF ? B1 : 1], wb[PT ? B1 : 1], tw[PT ? B1 : 1], h[HP ? RT : 1][M];
#pragma unroll
    for (int j = 0; j < B1; j++) a[j] = P.x[c + C * (u64)(t + B2 * j)];
    if (HP) {
#pragma unroll
        for (int q = 0; q < RT; q++) {
            const u64 g0 = C * (u64)(tid / PR + T * q) + c0;
#pragma unroll
            for (int j = 0; j < M; j++)
                h[HP ? q : 0][j] =
                    (tid / PR + T * q < RR && tid % PR == 0) ? P.x[(g0 + n - M + j) & (n - 1)] : 0;
        }
    }
    if (PF) {
#pragma unroll
        for (int j = 0; j < B1; j++) {
            const u32 sl = lnt_wslot(ec, mC, P.n, (u32)(t + B2 * j));
            wv[PF ? j : 0] = P.w[2 * sl];
            if (PT) wb[PT ? j : 0] = P.w[2 * sl + 1];
            if (PT) tw[PT ? j : 0] = P.twc[(u64)j * B2 + t];
        }
    }
#pragma unroll
    for (int j = 0; j < B1; j++) lds[(u32)((t + B2 * j) * KS + cl)] = a[j];
    LNT_SYNC();

    // 1. carry + (-2): one thread per row run of K digits (plus the M halo digits), or PR
    //    threads per run where there are more threads than rows (16 to 64 rows: the carry is
    //    a quarter to a half of the chain that these short kernels are)
    if constexpr (PR > 1) {
        static_assert(HP && K == 16, "the halo words are prefetched");
        lnt_carry_piece<M, K / PR, PR>(lds, (u32)(tid / PR * KS), tid % PR, h[0], P, C * (u64)(tid / PR) + c0, sub2);
    }
#pragma unroll
    for (int q = 0; q < (PR > 1 ? 0 : RT); q++) {
        const int r = tid + T * q;
        if (r >= RR) break;
        int64_t v[M + K];
        const u64 g0 = C * (u64)r + c0;
#pragma unroll
        for (int j = 0; j < M; j++) v[j] = gl_to_i64(HP ? h[HP ? q : 0][j] : P.x[(g0 + n - M + j) & (n - 1)]);
#pragma unroll
        for (int j = 0; j < K; j++) v[M + j] = gl_to_i64(lds[(u32)(r * KS + j)]);
        lnt_carry_run<M, K>(v, P.p, P.log_n, g0, P.levels, sub2);
        // the digit as d + 2^31 for the biased weight multiply, else field-encoded
#pragma unroll
        for (int j = 0; j < K; j++)
            lds[(u32)(r * KS + j)] = P.bias ? (u64)(u32)(v[M + j] + (int64_t(1) << 31)) : gl_from_i64(v[M + j]);
    }
    LNT_SYNC();

    // 2. phase 1: weight, B1-point DFT down the column, inter-block twiddle
    if (P.bias) {
#pragma unroll
        for (int j = 0; j < B1; j++) {
            const u32 sl = lnt_wslot(ec, mC, P.n, (u32)(t + B2 * j));
            a[j] = gl_mul_biased((u32)lds[(u32)((t + B2 * j) * KS + cl)], PF ? wv[PF ? j : 0] : P.w[2 * sl],
                                 PT ? wb[PT ? j : 0] : P.w[2 * sl + 1]);
        }
    } else {
#pragma unroll
        for (int j = 0; j < B1; j++)
            a[j] = gl_mul(lds[(u32)((t + B2 * j) * KS + cl)],
                          PF ? wv[PF ? j : 0] : P.w[2 * lnt_wslot(ec, mC, P.n, (u32)(t + B2 * j))]);
    }
    dft_fwd<B1>(a);
    if (B2 > 1) {
#pragma unroll
        for (int rho = 1; rho < B1; rho++)
            a[rho] = gl_mmul(a[rho], PT ? tw[PT ? rho : 0] : P.twc[(u64)rho * B2 + t]);
    }
    LNT_SYNC();
#pragma unroll
    for (int rho = 0; rho < B1; rho++)
        lds[(u32)((brev_c<B1>(rho) * S + t) * K + cl)] = a[rho];
    LNT_SYNC();

    // 3. phase 2: B2-point DFTs, store (row r' = t*B1 + q*B2 + rho'); the 4-step twiddle
    //    is applied by the row pass as it loads the row
#pragma unroll
    for (int q = 0; q < RP; q++) {
        const int k2 = t * RP + q;
#pragma unroll
        for (int i1 = 0; i1 < B2; i1++) a[q * B2 + i1] = lds[(u32)((k2 * S + i1) * K + cl)];
        dft_fwd<B2>(a + q * B2);
    }
#pragma unroll
    for (int i = 0; i < B1; i++) P.y[c + C * ((u64)t * B1 + i)] = a[i];
}

// ------------------------------------------------------------------ column inverse
template <int B1, int B2, int K>
LNT_KFN void lnt_col_inv_body(int tid, int bid, LView lds, const LntParams &P) {
    constexpr int RP = B1 / B2;
    constexpr int S = B2 + LNT_PAD;
    const u64 C = P.C;
    const int cl = tid % K, t = tid / K;
    const u64 c = (u64)bid * K + cl;
    const u32 ec = lnt_wexp(P.p, P.n, c), mC = 0u - P.p * P.C;  // weight slot parameters
    constexpr bool PF = B1 <= 32;  // prefetch the unweighting factors (fits when B1 <= 32)
    constexpr bool PT = B1 <= 8;   // and the twiddles of short lines
    u64 a[B1], uv[PF ? B1 : 1], tw[PT ? B1 : 1];
    // (the inverse 4-step twiddle was applied by the row pass as it stored the row)
#pragma unroll
    for (int i = 0; i < B1; i++) a[i] = P.y[c + C * ((u64)t * B1 + i)];
    if (PF) {
#pragma unroll
        for (int j = 0; j < B1; j++) {
            uv[PF ? j : 0] = P.uw[lnt_wslot(ec, mC, P.n, (u32)(t + B2 * j))];
            if (PT) tw[PT ? j : 0] = P.itwc[(u64)j * B2 + t];
        }
    }
#pragma unroll
    for (int q = 0; q < RP; q++) {
        dft_inv<B2>(a + q * B2);
        const int k2 = t * RP + q;
#pragma unroll
        for (int i1 = 0; i1 < B2; i1++) lds[(u32)((k2 * S + i1) * K + cl)] = a[q * B2 + i1];
    }
    LNT_SYNC();
#pragma unroll
    for (int rho = 0; rho < B1; rho++) {
        u64 v = lds[(u32)((brev_c<B1>(rho) * S + t) * K + cl)];
        a[rho] = (B2 > 1 && rho > 0) ? gl_mmul(v, PT ? tw[PT ? rho : 0] : P.itwc[(u64)rho * B2 + t]) : v;
    }
    dft_inv<B1>(a);
#pragma unroll
    for (int j = 0; j < B1; j++) {
        const u64 idx = c + C * ((u64)t + (u64)B2 * j);
        P.x[idx] = gl_mmul(a[j], PF ? uv[PF ? j : 0] : P.uw[lnt_wslot(ec, mC, P.n, (u32)(t + B2 * j))]);
    }
}

// ------------------------------------------------------------------ 3-phase columns
// Column line R = BA * BB * BC handled by A = BB * BC threads per column (K columns per
// workgroup, block K * A threads, BA words per thread).  Row r = a + A j (a < A, j < BA):
//  phase 1: thread a, BA-point DFT over j -> k1, twiddle w_R^(a k1)
//  phase 2: items (k1, u), u < BC (BA / BB per thread): BB-point DFT over v of the words
//           a = u + BC v -> k2, twiddle w_A^(u k2)
//  phase 3: items (k1, k2) (BA / BC per thread): BC-point DFT over u -> k3
// Frequency k1 + BA (k2 + BB k3) ends in slot t*BA + q*BC + rho (k3 = brev(rho)).
// LDS word (row, column) at row * KP + column, rows k1 * (A + 1) + a.
template <int BA, int BB, int BC, int K>
struct LntCol3 {
    static constexpr int A = BB * BC, R = BA * A;
    static constexpr int QB = BA / BB, QC = BA / BC;
    static constexpr int RS = A + 1;
    static constexpr int KP = BA * RS * (K + 1) <= 18432 ? K + 1 : K;  // padded when it fits 144 KiB
    static constexpr int KS = R * (K + 1) <= 18432 ? K + 1 : K;        // carry staging row width
    static constexpr u32 LDS = (u32)(BA * RS * KP > R * KS ? BA * RS * KP : R * KS);
    static_assert(BA % BB == 0 && BA % BC == 0 && BB >= BC, "3-phase column radices");
};

template <int BA, int BB, int BC, int K, int M>
LNT_KFN void lnt_col3_fwd_body(int tid, int bid, LView lds, const LntParams &P, bool sub2) {
    using S = LntCol3<BA, BB, BC, K>;
    constexpr int A = S::A, RR = S::R, RS = S::RS, KP = S::KP, KS = S::KS;
    constexpr int NT = K * A;
    constexpr int RT = (RR + NT - 1) / NT;  // carry rows per thread
    constexpr bool HP = RT * M <= 16;
    const u64 C = P.C;
    const u64 n = P.n;
    const u64 c0 = (u64)bid * K;
    const int cl = tid % K, t = tid / K;
    const u64 c = c0 + cl;
    const u32 ec = lnt_wexp(P.p, P.n, c), mC = 0u - P.p * P.C;  // weight slot parameters

    // 0. loads: rows t + A j of column c (K adjacent lanes read one row run), the halo
    //    digits of this thread's carry rows, the weights (prefetched into registers only
    //    in blocks of <= 512 threads, whose register budget allows it)
    constexpr bool PW = NT <= 512;
    u64 a[BA], wv[PW ? BA : 1], wb[PW ? BA : 1], h[HP ? RT : 1][M];
#pragma unroll
    for (int j = 0; j < BA; j++) a[j] = P.x[c + C * (u64)(t + A * j)];
    if (HP) {
#pragma unroll
        for (int q = 0; q < RT; q++) {
            const u64 g0 = C * (u64)(tid + NT * q) + c0;
#pragma unroll
            for (int j = 0; j < M; j++)
                h[HP ? q : 0][j] = (tid + NT * q < RR) ? P.x[(g0 + n - M + j) & (n - 1)] : 0;
        }
    }
    if (PW) {
#pragma unroll
        for (int j = 0; j < BA; j++) {
            const u32 sl = lnt_wslot(ec, mC, P.n, (u32)(t + A * j));
            wv[PW ? j : 0] = P.w[2 * sl];
            wb[PW ? j : 0] = P.w[2 * sl + 1];
        }
    }
#pragma unroll
    for (int j = 0; j < BA; j++) lds[(u32)((t + A * j) * KS + cl)] = a[j];
    LNT_SYNC();

    // 1. carry + (-2): one thread per row run of K digits (plus the M halo digits)
#pragma unroll
    for (int q = 0; q < RT; q++) {
        const int r = tid + NT * q;
        if (r >= RR) break;
        // streamed in pieces of PK digits, each piece's halo being the M pre-carry values
        // before it: the whole 16-digit run in one piece where it fits the 128 registers of
        // a 1024-thread block (BA = 16, M = 4), pieces of 8 where one piece would spill
        constexpr int PK = (NT >= 1024 && K > 8 && (M > 4 || BA < 16)) ? 8 : K;
        const u64 g0 = C * (u64)r + c0;
        int64_t halo[M];
#pragma unroll
        for (int j = 0; j < M; j++) halo[j] = gl_to_i64(HP ? h[HP ? q : 0][j] : P.x[(g0 + n - M + j) & (n - 1)]);
#pragma unroll
        for (int s = 0; s < K / PK; s++) {
            int64_t v[M + PK];
#pragma unroll
            for (int j = 0; j < M; j++) v[j] = halo[j];
#pragma unroll
            for (int j = 0; j < PK; j++) v[M + j] = gl_to_i64(lds[(u32)(r * KS + s * PK + j)]);
#pragma unroll
            for (int j = 0; j < M; j++) halo[j] = v[PK + j];
            lnt_carry_run<M, PK>(v, P.p, P.log_n, g0 + s * PK, P.levels, sub2);
            // the digit as d + 2^31 for the biased weight multiply, else field-encoded
#pragma unroll
            for (int j = 0; j < PK; j++)
                lds[(u32)(r * KS + s * PK + j)] =
                    P.bias ? (u64)(u32)(v[M + j] + (int64_t(1) << 31)) : gl_from_i64(v[M + j]);
        }
    }
    LNT_SYNC();

    // 2. phase 1: weight, BA-point DFT, twiddle
    if (P.bias) {
#pragma unroll
        for (int j = 0; j < BA; j++) {
            const u32 sl = PW ? 0 : lnt_wslot(ec, mC, P.n, (u32)(t + A * j));
            a[j] = gl_mul_biased((u32)lds[(u32)((t + A * j) * KS + cl)], PW ? wv[PW ? j : 0] : P.w[2 * sl],
                                 PW ? wb[PW ? j : 0] : P.w[2 * sl + 1]);
        }
    } else {
#pragma unroll
        for (int j = 0; j < BA; j++)
            a[j] = gl_mul(lds[(u32)((t + A * j) * KS + cl)],
                          PW ? wv[PW ? j : 0] : P.w[2 * lnt_wslot(ec, mC, P.n, (u32)(t + A * j))]);
    }
    dft_fwd<BA>(a);
#pragma unroll
    for (int rho = 1; rho < BA; rho++) a[rho] = gl_mmul(a[rho], P.twc[(u64)rho * A + t]);
    LNT_SYNC();
#pragma unroll
    for (int rho = 0; rho < BA; rho++) lds[(u32)((brev_c<BA>(rho) * RS + t) * KP + cl)] = a[rho];
    LNT_SYNC();

    // 3. phase 2 (each item rewrites exactly the LDS rows it read: no barrier inside)
#pragma unroll
    for (int q = 0; q < S::QB; q++) {
        const int I = q * A + t, k1 = I / BC, u = I % BC;
        u64 b[BB];
#pragma unroll
        for (int v = 0; v < BB; v++) b[v] = lds[(u32)((k1 * RS + u + BC * v) * KP + cl)];
        dft_fwd<BB>(b);
#pragma unroll
        for (int rho = 0; rho < BB; rho++) lds[(u32)((k1 * RS + BC * brev_c<BB>(rho) + u) * KP + cl)] = b[rho];
    }
    LNT_SYNC();

    // 4. phase 3 with the phase-2 twiddle w_A^(u k2) at the read, store slot
    //    t*BA + q*BC + rho (the row pass applies the 4-step twiddle)
#pragma unroll
    for (int q = 0; q < S::QC; q++) {
        const int I = q * A + t, k1 = I / BB, k2 = I % BB;
        const u64 tb = (u64)brev_c<BB>(k2) * BC;
#pragma unroll
        for (int u = 0; u < BC; u++)
            a[q * BC + u] = gl_mmul(lds[(u32)((k1 * RS + BC * k2 + u) * KP + cl)], P.twc2[tb + u]);
        dft_fwd<BC>(a + q * BC);
    }
#pragma unroll
    for (int i = 0; i < BA; i++) P.y[c + C * ((u64)t * BA + i)] = a[i];
}

template <int BA, int BB, int BC, int K>
LNT_KFN void lnt_col3_inv_body(int tid, int bid, LView lds, const LntParams &P) {
    using S = LntCol3<BA, BB, BC, K>;
    constexpr int A = S::A, RS = S::RS, KP = S::KP;
    const u64 C = P.C;
    const int cl = tid % K, t = tid / K;
    const u64 c = (u64)bid * K + cl;
    const u32 ec = lnt_wexp(P.p, P.n, c), mC = 0u - P.p * P.C;  // weight slot parameters
    u64 a[BA], uv[BA];
#pragma unroll
    for (int i = 0; i < BA; i++) a[i] = P.y[c + C * ((u64)t * BA + i)];
#pragma unroll
    for (int j = 0; j < BA; j++) uv[j] = P.uw[lnt_wslot(ec, mC, P.n, (u32)(t + A * j))];
    // phase 3 inverse, then the inverse phase-2 twiddle
#pragma unroll
    for (int q = 0; q < S::QC; q++) {
        const int I = q * A + t, k1 = I / BB, k2 = I % BB;
        const u64 tb = (u64)brev_c<BB>(k2) * BC;
        dft_inv<BC>(a + q * BC);
#pragma unroll
        for (int u = 0; u < BC; u++)
            lds[(u32)((k1 * RS + BC * k2 + u) * KP + cl)] = gl_mmul(a[q * BC + u], P.itwc2[tb + u]);
    }
    LNT_SYNC();
    // phase 2 inverse
#pragma unroll
    for (int q = 0; q < S::QB; q++) {
        const int I = q * A + t, k1 = I / BC, u = I % BC;
        u64 b[BB];
#pragma unroll
        for (int rho = 0; rho < BB; rho++) b[rho] = lds[(u32)((k1 * RS + BC * brev_c<BB>(rho) + u) * KP + cl)];
        dft_inv<BB>(b);
#pragma unroll
        for (int v = 0; v < BB; v++) lds[(u32)((k1 * RS + u + BC * v) * KP + cl)] = b[v];
    }
    LNT_SYNC();
    // phase 1 inverse, unweight, store
#pragma unroll
    for (int rho = 0; rho < BA; rho++) {
        u64 v = lds[(u32)((brev_c<BA>(rho) * RS + t) * KP + cl)];
        a[rho] = rho ? gl_mmul(v, P.itwc[(u64)rho * A + t]) : v;
    }
    dft_inv<BA>(a);
#pragma unroll
    for (int j = 0; j < BA; j++) {
        const u64 idx = c + C * ((u64)t + (u64)A * j);
        P.x[idx] = gl_mmul(a[j], uv[j]);
    }
}

// ------------------------------------------------------------------ columns on the matrix cores
// Columns of R = 256 S words (S = 1, 4), 16 adjacent columns per workgroup of 16 waves,
// 4 S words per thread: the 16 columns of a tile are the 16 DFTs of a matrix instruction, so
// lane (q, n) works on column c0 + n throughout.  With row r = a1 + 16 S j, a1 = a + S b:
//   phase 1: group a1 = S w + g of wave w: DFT over j -> k2, twiddle omega_R^(a1 k2)         (twc)
//   phase 2: group (k2 = w, a = g): DFT over b -> kb, twiddle omega_16S^(a kb)               (twc2)
//   phase 3: S-point DFTs over a = g, in registers -> k3 (bit-reversed)
// Frequency k2 + 16 (kb + 16 k3) goes to slot (16 k2 + kb) S + k3, where lnt_tw4_m puts its 4-step
// twiddle.  Every DFT writes the LDS words that it read, so only the exchange between phases 1
// and 2 and the hand-over of the carried digits wait for other waves.  LDS word (row r, column
// n) at RS r + n; RS keeps the words of neighbouring lane groups (2 S rows apart in phase 2) on
// the two halves of the banks.
// W = 16 waves take S groups each (four times as many with W = 4, S = 1).
template <int S, int W = 16>
struct LntColM {
    static constexpr int R = 256 * S, L = 16 * S;
    static constexpr int RS = S == 1 && W == 16 ? 24 : 18;
    static constexpr u32 LDS = (u32)(R * RS);
};

template <int S, int M, int W = 16>
LNT_KFN void lnt_colm_fwd_body(int tid, int bid, LView lds, const LntParams &P, bool sub2) {
    static_assert(S == 1 || W == 16, "phase 3 takes the words of one k2 from the wave's own places");
    using Z = LntColM<S, W>;
    constexpr int RS = Z::RS, L = Z::L, G = 16 * S / W;
    constexpr int PR = W / (4 * S), PK = 16 / PR;  // carry: threads per row, digits per thread
    const LntLane16 T = lnt_lane16(tid);
    const int q = T.q, n = T.n, w = T.w;
    const u64 C = P.C, c0 = (u64)bid * 16;
    // the tile, 16 columns of a row by 16 lanes; row r's M digits before it by the thread of
    // its first piece
    {
        u64 a[PK], h[M];
#pragma unroll
        for (int i = 0; i < PK; i++) a[i] = P.x[c0 + n + C * (u64)(tid / 16 + 4 * W * i)];
        const u64 g0 = C * (u64)(tid / PR) + c0;
#pragma unroll
        for (int j = 0; j < M; j++) h[j] = tid % PR == 0 ? P.x[(g0 + P.n - M + j) & (P.n - 1)] : 0;
#pragma unroll
        for (int i = 0; i < PK; i++) lds[(u32)(RS * (tid / 16 + 4 * W * i) + n)] = a[i];
        LNT_SYNC();
        // carry + (-2): PR neighbouring threads per row run of 16 digits
        lnt_carry_piece<M, PK, PR>(lds, (u32)(RS * (tid / PR)), tid % PR, h, P, g0, sub2);
    }
    LntM16 Mx;
    lnt_m16_load(Mx, tid);
    const u32 ec = lnt_wexp(P.p, P.n, c0 + n), mC = 0u - P.p * P.C;  // weight slot parameters
    // phase 1 with the weights, those of a group fetched before the barrier or the DFT ahead of it
    // (S = 1 at 2^18: 8.4 -> 7.7 us; S = 4: no change)
    u64 wv[4], wb[4];
    auto fetch_w = [&](int a1) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const u32 sl = lnt_wslot(ec, mC, P.n, (u32)(a1 + L * lnt_m16_word(q, e)));
            wv[e] = P.w[2 * sl];
            wb[e] = P.w[2 * sl + 1];
        }
    };
    fetch_w(G * w);
    LNT_SYNC();
#pragma unroll 1
    for (int a1 = G * w; a1 < G * w + G; a1++) {
        u64 z[4], tw[4];
        const u32 at = (u32)(RS * a1 + n);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const u64 d = lds[at + (u32)(RS * L * lnt_m16_word(q, e))];
            z[e] = P.bias ? gl_mul_biased((u32)d, wv[e], wb[e]) : gl_mul(d, wv[e]);
            tw[e] = P.twc[L * brev_v16(lnt_m16_word(q, e)) + a1];
        }
        if (G > 1 && a1 + 1 < G * w + G) fetch_w(a1 + 1);
        lnt_m16_dft(Mx, z);
#pragma unroll
        for (int v = 0; v < 4; v++) lds[at + (u32)(RS * L * lnt_m16_word(q, v))] = gl_mmul(z[v], tw[v]);
    }
    LNT_SYNC();
    // phase 2 (S = 1: the last); with S > 1 its words go through this lane's own LDS places to phase 3
#pragma unroll 1
    for (int i = 0; i < G; i++) {
        const int k2 = S == 1 ? G * w + i : w, g = S == 1 ? 0 : i;
        u64 z[4];
        const u32 at = (u32)(RS * (L * k2 + g) + n);
#pragma unroll
        for (int e = 0; e < 4; e++) z[e] = lds[at + (u32)(RS * S * lnt_m16_word(q, e))];
        lnt_m16_dft(Mx, z);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int kb = lnt_m16_word(q, v);
            if (S == 1) P.y[c0 + n + C * (u64)(16 * k2 + kb)] = z[v];
            else lds[at + (u32)(RS * S * kb)] = gl_mmul(z[v], P.twc2[S * brev_v16(kb) + g]);
        }
    }
    if (S == 1) return;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int kb = lnt_m16_word(q, v);
        u64 t[S];
#pragma unroll
        for (int g = 0; g < S; g++) t[g] = lds[(u32)(RS * (L * w + g + S * kb) + n)];
        dft_fwd<S>(t);
#pragma unroll
        for (int g = 0; g < S; g++) P.y[c0 + n + C * (u64)((16 * w + kb) * S + brev_c<S>(g))] = t[g];
    }
}

template <int S, int W = 16>
LNT_KFN void lnt_colm_inv_body(int tid, int bid, LView lds, const LntParams &P) {
    static_assert(S == 1 || W == 16, "phase 3 leaves the words of one k2 in the wave's own places");
    using Z = LntColM<S, W>;
    constexpr int RS = Z::RS, L = Z::L, G = 16 * S / W;
    const LntLane16 T = lnt_lane16(tid);
    const int q = T.q, n = T.n, w = T.w;
    const u64 C = P.C, c = (u64)bid * 16 + n;
    // phase 3 inverse over k3 and the inverse phase-2 twiddle, into this lane's own LDS places
    if (S > 1) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int kb = lnt_m16_word(q, v);
            u64 t[S];
#pragma unroll
            for (int g = 0; g < S; g++) t[g] = P.y[c + C * (u64)((16 * w + kb) * S + brev_c<S>(g))];
            dft_inv<S>(t);
#pragma unroll
            for (int g = 0; g < S; g++)
                lds[(u32)(RS * (L * w + g + S * kb) + n)] = gl_mmul(t[g], P.itwc2[S * brev_v16(kb) + g]);
        }
    }
    LntM16 Mx;
    lnt_m16_load(Mx, tid);
    // phase 2 inverse: output place v is b = -lnt_m16_word(q, v)
#pragma unroll 1
    for (int i = 0; i < G; i++) {
        const int k2 = S == 1 ? G * w + i : w, g = S == 1 ? 0 : i;
        u64 z[4], tw[4];
        const u32 at = (u32)(RS * (L * k2 + g) + n);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int kb = lnt_m16_word(q, e);
            z[e] = S == 1 ? P.y[c + C * (u64)(16 * k2 + kb)] : lds[at + (u32)(RS * S * kb)];
            tw[e] = P.itwc[L * brev_v16(k2) + g + S * lnt_m16_neg(q, e)];
        }
        LNT_WAVE_SYNC();
        lnt_m16_dft(Mx, z);
#pragma unroll
        for (int v = 0; v < 4; v++) lds[at + (u32)(RS * S * lnt_m16_neg(q, v))] = gl_mmul(z[v], tw[v]);
    }
    const u32 ec = lnt_wexp(P.p, P.n, c), mC = 0u - P.p * P.C;  // weight slot parameters
    LNT_SYNC();
    // phase 1 inverse, unweight, store
#pragma unroll 1
    for (int a1 = G * w; a1 < G * w + G; a1++) {
        u64 y[4], uv[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            y[e] = lds[(u32)(RS * (L * lnt_m16_word(q, e) + a1) + n)];
            uv[e] = P.uw[lnt_wslot(ec, mC, P.n, (u32)(a1 + L * lnt_m16_neg(q, e)))];
        }
        lnt_m16_dft(Mx, y);
#pragma unroll
        for (int v = 0; v < 4; v++) P.x[c + C * (u64)(a1 + L * lnt_m16_neg(q, v))] = gl_mmul(y[v], uv[v]);
    }
}

// ------------------------------------------------------------------ row pass
// grid: R / G workgroups, block: G * B2 threads (G rows per workgroup).
// LDS words: G * B1 * (B2 + PAD).
// MODE 0: square (one iteration).  MODE 1: forward only; the transform-domain words go
// to slot base + t*B1 + i of y.  MODE 2: forward, multiply by the other operand's words f
// (same slots, written by a MODE 1 pass), inverse.
constexpr int LNT_SQUARE = 0, LNT_FORWARD = 1, LNT_MULTIPLY = 2;
template <int B1, int B2, int G, int MODE = LNT_SQUARE>
LNT_KFN void lnt_row_body(int tid, int bid, LView lds, const LntParams &P) {
    constexpr int RP = B1 / B2;
    constexpr int S = B2 + LNT_PAD;
    constexpr int LINE = B1 * S;
    const int t = tid % B2, g = tid / B2;
    const u64 base = (u64)P.C * ((u64)bid * G + g);
    const u32 lb = (u32)(g * LINE);
    u64 a[B1];
#pragma unroll
    for (int j = 0; j < B1; j++) {
        const u64 idx = base + t + (u64)B2 * j;
        a[j] = gl_mmul(P.y[idx], P.tw4[idx]);  // 4-step twiddle of the column pass
    }
    dft_fwd<B1>(a);
    if (B2 > 1) {
#pragma unroll
        for (int rho = 1; rho < B1; rho++) a[rho] = gl_mmul(a[rho], P.twr[(u64)rho * B2 + t]);
    }
#pragma unroll
    for (int rho = 0; rho < B1; rho++) lds[lb + (u32)(brev_c<B1>(rho) * S + t)] = a[rho];
    LNT_SYNC();
#pragma unroll
    for (int q = 0; q < RP; q++) {
        const int k2 = t * RP + q;
#pragma unroll
        for (int i1 = 0; i1 < B2; i1++) a[q * B2 + i1] = lds[lb + (u32)(k2 * S + i1)];
        dft_fwd<B2>(a + q * B2);
        if (MODE == LNT_FORWARD) {
#pragma unroll
            for (int i1 = 0; i1 < B2; i1++) P.y[base + (u64)t * B1 + q * B2 + i1] = a[q * B2 + i1];
            continue;
        }
        if (MODE == LNT_MULTIPLY) {
#pragma unroll
            for (int i1 = 0; i1 < B2; i1++)
                a[q * B2 + i1] = gl_mmul(a[q * B2 + i1], P.f[base + (u64)t * B1 + q * B2 + i1]);
        } else {
#pragma unroll
            for (int i1 = 0; i1 < B2; i1++) a[q * B2 + i1] = gl_mmul(a[q * B2 + i1], a[q * B2 + i1]);
        }
        dft_inv<B2>(a + q * B2);
#pragma unroll
        for (int i1 = 0; i1 < B2; i1++) lds[lb + (u32)(k2 * S + i1)] = a[q * B2 + i1];
    }
    if (MODE == LNT_FORWARD) return;
    LNT_SYNC();
#pragma unroll
    for (int rho = 0; rho < B1; rho++) {
        u64 v = lds[lb + (u32)(brev_c<B1>(rho) * S + t)];
        a[rho] = (B2 > 1 && rho > 0) ? gl_mmul(v, P.itwr[(u64)rho * B2 + t]) : v;
    }
    dft_inv<B1>(a);
#pragma unroll
    for (int j = 0; j < B1; j++) {
        const u64 idx = base + t + (u64)B2 * j;
        P.y[idx] = gl_mmul(a[j], P.itw4[idx]);  // inverse 4-step twiddle
    }
}

// ------------------------------------------------------------------ 3-phase row pass
// Rows of C = B^3 words, B^2 threads per row each holding B words (more waves per SIMD
// than the 2-phase row: B registers instead of B1 = 64).  With i = i1 + B^2 i2
// (i1 < B^2) and i1 = a + B b:
//   phase 1: thread i1: B-point DFT over i2 -> k2, twiddle omega_C^(i1 k2)      (twr)
//   phase 2: thread (k2, a): B-point DFT over b -> kb, twiddle omega_B^2^(a kb) (twr2)
//   phase 3: thread (k2, kb): B-point DFT over a -> ka; X[B (B ka + kb) + k2]
// then the pointwise square (or the product modes of lnt_row_body) and the inverse in
// reverse.  Within the LDS row of k2 a word (r, a) sits at r * (B + 1) + a, so every
// phase reads and writes conflict-free strides.  Transform-domain slot for MODE 1/2:
// base + k2 * B^2 + kb * B + i (thread-contiguous).
// Reached for B = 8 (rows of 512 words) when a plan or the tuner asks for 3-phase rows.
// LDS layout: word (k2, a) of a row at k2 * RS + a with runs of B words, unpadded by default:
// the phase-3 runs are then 16-byte aligned and pair into 128-bit LDS accesses.
template <int B, int G, int MODE = LNT_SQUARE, int PAD = 0>
LNT_KFN void lnt_row3_body(int tid, int bid, LView lds, const LntParams &P) {
    constexpr int T = B * B;        // threads per row
    constexpr int RS = B * (B + PAD); // LDS words per k2 row
    constexpr int LINE = B * RS;    // LDS words per row
    const int t = tid % T, g = tid / T;
    const u64 base = (u64)P.C * ((u64)bid * G + g);
    const u32 lb = (u32)(g * LINE);
    const int hi = t / B, lo = t % B;  // phases 2/3: (k2, a) or (k2, kb)
    u64 a[B];
    // phase 1
#pragma unroll
    for (int j = 0; j < B; j++) {
        const u64 idx = base + t + (u64)T * j;
        a[j] = gl_mmul(P.y[idx], P.tw4[idx]);  // 4-step twiddle of the column pass
    }
    // the inverse 4-step twiddles of the final store, fetched now so their latency hides
    // behind the transforms
    u64 iv[MODE == LNT_FORWARD ? 1 : B];
    if (MODE != LNT_FORWARD) {
#pragma unroll
        for (int j = 0; j < B; j++) iv[MODE == LNT_FORWARD ? 0 : j] = P.itw4[base + t + (u64)T * j];
    }
    dft_fwd<B>(a);
#pragma unroll
    for (int rho = 1; rho < B; rho++) a[rho] = gl_mmul(a[rho], P.twr[(u64)rho * T + t]);
#pragma unroll
    for (int rho = 0; rho < B; rho++) lds[lb + (u32)(brev_c<B>(rho) * RS + (t / B) * (B + PAD) + t % B)] = a[rho];
    LNT_SYNC();
    // phase 2: thread (k2 = hi, a = lo) over b
#pragma unroll
    for (int b = 0; b < B; b++) a[b] = lds[lb + (u32)(hi * RS + b * (B + PAD) + lo)];
    // (this thread rewrites exactly the slots it just read: no barrier needed)
    dft_fwd<B>(a);
#pragma unroll
    for (int rho = 1; rho < B; rho++) a[rho] = gl_mmul(a[rho], P.twr2[(u64)rho * B + lo]);
#pragma unroll
    for (int rho = 0; rho < B; rho++) lds[lb + (u32)(hi * RS + brev_c<B>(rho) * (B + PAD) + lo)] = a[rho];
    LNT_SYNC();
    // phase 3: thread (k2 = hi, kb = lo) over a
#pragma unroll
    for (int i = 0; i < B; i++) a[i] = lds[lb + (u32)(hi * RS + lo * (B + PAD) + i)];
    dft_fwd<B>(a);
    if (MODE == LNT_FORWARD) {
#pragma unroll
        for (int i = 0; i < B; i++) P.y[base + (u64)t * B + i] = a[i];
        return;
    }
    if (MODE == LNT_MULTIPLY) {
#pragma unroll
        for (int i = 0; i < B; i++) a[i] = gl_mmul(a[i], P.f[base + (u64)t * B + i]);
    } else {
#pragma unroll
        for (int i = 0; i < B; i++) a[i] = gl_mmul(a[i], a[i]);
    }
    dft_inv<B>(a);
#pragma unroll
    for (int i = 0; i < B; i++) lds[lb + (u32)(hi * RS + lo * (B + PAD) + i)] = a[i];
    LNT_SYNC();
    // phase 2 inverse: thread (k2, a): registers rho hold kb = brev(rho)
#pragma unroll
    for (int rho = 0; rho < B; rho++) {
        u64 v = lds[lb + (u32)(hi * RS + brev_c<B>(rho) * (B + PAD) + lo)];
        a[rho] = rho ? gl_mmul(v, P.itwr2[(u64)rho * B + lo]) : v;
    }
    dft_inv<B>(a);
#pragma unroll
    for (int b = 0; b < B; b++) lds[lb + (u32)(hi * RS + b * (B + PAD) + lo)] = a[b];
    LNT_SYNC();
    // phase 1 inverse: thread i1 = t, registers rho hold k2 = brev(rho)
#pragma unroll
    for (int rho = 0; rho < B; rho++) {
        u64 v = lds[lb + (u32)(brev_c<B>(rho) * RS + (t / B) * (B + PAD) + t % B)];
        a[rho] = rho ? gl_mmul(v, P.itwr[(u64)rho * T + t]) : v;
    }
    dft_inv<B>(a);
#pragma unroll
    for (int j = 0; j < B; j++) P.y[base + t + (u64)T * j] = gl_mmul(a[j], iv[MODE == LNT_FORWARD ? 0 : j]);
}

// ------------------------------------------------------------------ lines of 256 S words on the matrix cores
// The transform of a line of L = 256 S words (S = 1, 2, 4, 8, 16) by S waves, four words per
// thread: L = 16 * 16 * S with the 16-point DFTs of mdft.hpp in phases 1 and 2 and an S-point
// one in phase 3 (S = 2, 4 in registers, 8 and 16 on the matrix cores).  With i = i1 + 16 S j,
// i1 = a + S b; wave w, lane (q, n), id = 16 w + n:
//   phase 1: DFT i1 = id over j -> k2, twiddle omega_L^(i1 k2)                       (twr)
//   phase 2: DFT (k2, a) = (id / S, id mod S) over b -> kb, twiddle omega_16S^(a kb) (twr2)
//   phase 3: DFTs (k2, kb) over a, all k2 of one wave; square (or the product modes)
// and the inverse in reverse.  A wave keeps its k2 between phase 1 and the inverse phase 2: only
// the exchanges around these wait for the other waves.  LDS words A + ... of the region: runs of 16
// words 18 apart, so that they start 16-byte aligned, 16 neighbouring runs cover all banks and
// the reads of adjacent word pairs are 128-bit.
// lnt_line16 takes phase 1's inputs z (place e: i1 = id, j = lnt_m16_word(q, e)) and leaves the
// inverse's outputs (place v: j = -lnt_m16_word(q, v) mod 16).  T holds the thread's twiddles
// tw1, tw2, itw2, itw1 (loaded by line16_load_*; the before_* hooks may load them late).
// Transform-domain words for MODE 1/2 at slot + v.
template <int S>
constexpr u32 lnt_line16_lds() { return 288 * S; }

// a of this thread's phase-3 place v: S = 16 (w, n, -word(q, v)), S = 8 (2w + v / 2, n, -(2q + v % 2)),
// S = 4 (4w + q, n, v), S = 2 (8w + 2q + v / 2, n, v % 2)
template <int S>
GL_HD constexpr int lnt_line16_a(int q, int v) {
    return S == 16 ? lnt_m16_neg(q, v) : S == 8 ? (8 - 2 * q - (v & 1)) & 7 : S == 4 ? v : v & 1;
}

struct LntTw16 {
    u64 tw1[4], tw2[4], itw2[4], itw1[4];
};
template <int S>
LNT_KFN void line16_load_tw1(LntTw16 &T, const LntLane16 &L, const LntParams &P) {
#pragma unroll
    for (int e = 0; e < 4; e++) T.tw1[e] = P.twr[16 * S * brev_v16(lnt_m16_word(L.q, e)) + L.id];
}
template <int S>
LNT_KFN void line16_load_tw2(LntTw16 &T, const LntLane16 &L, const LntParams &P) {
    if (S == 1) return;
#pragma unroll
    for (int e = 0; e < 4; e++) T.tw2[e] = P.twr2[S * brev_v16(lnt_m16_word(L.q, e)) + L.id % S];
}
template <int S>
LNT_KFN void line16_load_itw2(LntTw16 &T, const LntLane16 &L, const LntParams &P) {
    if (S == 1) return;
#pragma unroll
    for (int v = 0; v < 4; v++) T.itw2[v] = P.itwr2[S * brev_v16(L.n) + lnt_line16_a<S>(L.q, v)];
}
template <int S>
LNT_KFN void line16_load_itw1(LntTw16 &T, const LntLane16 &L, const LntParams &P) {
#pragma unroll
    for (int v = 0; v < 4; v++)
        T.itw1[v] = P.itwr[16 * S * brev_v16(L.id / S) + L.id % S + S * lnt_m16_neg(L.q, v)];
}

// Returns with z transformed, or (MODE_FORWARD) with the transform in y.  The region at A must be
// free when phase 1 writes it (after z was read) and is free again after the next barrier.
template <int S, int MODE, class H2, class HI2, class HI1>
LNT_KFN void lnt_line16(u64 (&z)[4], const LntM16 &Mx, const LntM8 &M8, LView lds, u32 A, const LntLane16 &L, LntTw16 &T,
                        const LntParams &P, u64 slot, H2 before_tw2, HI2 before_itw2, HI1 before_itw1) {
    const int q = L.q, n = L.n, id = L.id;
    const u32 t1 = A + (u32)(18 * (id % S) + id / S);  // place of i1 = id within a k2
    const u32 own = A + (u32)(18 * id + 2 * q);        // this lane's words of run id
    const u32 area = A + (u32)(288 * L.w);             // this wave's runs
    // phase-3 layout of the wave's area: word (k2, kb, a)
    auto p3 = [&](int k2l, int kb, int a) {
        return area + (u32)(S == 16 ? 18 * kb + a : (16 * S + 2) * k2l + S * kb + a);
    };
    lnt_m16_dft(Mx, z);
#pragma unroll
    for (int v = 0; v < 4; v++) lds[(u32)(18 * S * lnt_m16_word(q, v)) + t1] = gl_mmul(z[v], T.tw1[v]);
    before_tw2();
    LNT_SYNC();
    // phase 2
#pragma unroll
    for (int e = 0; e < 4; e++) z[e] = lds[own + lnt_m16_word(0, e)];
    LNT_WAVE_SYNC();
    lnt_m16_dft(Mx, z);
    if (S > 1) {
#pragma unroll
        for (int v = 0; v < 4; v++) lds[p3(n / S, lnt_m16_word(q, v), n % S)] = gl_mmul(z[v], T.tw2[v]);
        if (MODE != LNT_FORWARD) before_itw2();
        LNT_WAVE_SYNC();
        // phase 3
#pragma unroll
        for (int v = 0; v < 4; v++)
            z[v] = lds[S == 16  ? p3(0, n, 2 * q) + lnt_m16_word(0, v)
                       : S == 8 ? p3(v / 2, n, 2 * q + v % 2)
                       : S == 4 ? p3(q, n, v)
                                : p3(2 * q + v / 2, n, v % 2)];
        LNT_WAVE_SYNC();
    }
    auto phase3 = [&](bool inverse) {
        if (S == 16) lnt_m16_dft(Mx, z);
        if (S == 8) {
            u64 h[2] = {z[0], z[1]}, g[2] = {z[2], z[3]};
            lnt_m8_dft(M8, Mx, h);
            lnt_m8_dft(M8, Mx, g);
            z[0] = h[0], z[1] = h[1], z[2] = g[0], z[3] = g[1];
        }
        if (S == 4) inverse ? dft_inv<4>(z) : dft_fwd<4>(z);
        if (S == 2) {
            inverse ? dft_inv<2>(z) : dft_fwd<2>(z);
            inverse ? dft_inv<2>(z + 2) : dft_fwd<2>(z + 2);
        }
    };
    phase3(false);
    // pointwise
#pragma unroll
    for (int v = 0; v < 4; v++) {
        if (MODE == LNT_FORWARD) P.y[slot + v] = z[v];
        else z[v] = gl_mmul(z[v], MODE == LNT_MULTIPLY ? P.f[slot + v] : z[v]);
    }
    if (MODE == LNT_FORWARD) return;
    if (S > 1) {
        phase3(true);
        before_itw1();
        // inverse phase-2 twiddle; runs (k2, a) of words kb again
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int k2l = S == 16 ? 0 : S == 8 ? v / 2 : S == 4 ? q : 2 * q + v / 2;
            lds[area + (u32)(18 * (S * k2l + lnt_line16_a<S>(q, v)) + n)] = gl_mmul(z[v], T.itw2[v]);
        }
        LNT_WAVE_SYNC();
#pragma unroll
        for (int e = 0; e < 4; e++) z[e] = lds[own + lnt_m16_word(0, e)];
        LNT_WAVE_SYNC();
    }
    // inverse phase 2: output place v is b = -k
    lnt_m16_dft(Mx, z);
#pragma unroll
    for (int v = 0; v < 4; v++) lds[A + (u32)(18 * id + lnt_m16_neg(q, v))] = gl_mmul(z[v], T.itw1[v]);
    LNT_SYNC();
    // inverse phase 1
#pragma unroll
    for (int e = 0; e < 4; e++) z[e] = lds[(u32)(18 * S * lnt_m16_word(q, e)) + t1];
    lnt_m16_dft(Mx, z);
}

// ROWS rows per workgroup, one after the other, for launches that fill the chip: the DFT matrix is
// loaded once, the factors are read where they are used, which keeps to the 128 registers of
// four waves per SIMD, and consecutive rows take turns on two LDS regions, so that a row's first
// exchange need not wait for the last reads of the row before.
template <int S, int ROWS>
LNT_KFN void lnt_rowm_rows_body(int tid, int bid, LView lds, const LntParams &P) {
    LntM16 Mx;
    LntM8 M8;
    lnt_m16_load(Mx, tid);
    if (S == 8) lnt_m8_load(M8, Mx, tid);
#pragma unroll 1
    for (int r = 0; r < ROWS; r++) {
        LNT_OPAQUE_LANE(tid);
        const LntLane16 L = lnt_lane16(tid);
        const u64 base = (u64)(256 * S) * ((u64)bid * ROWS + r);
        u64 z[4], t4[4];
        LntTw16 T;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const u64 idx = base + L.id + 16 * S * lnt_m16_word(L.q, e);
            z[e] = gl_mmul(P.y[idx], P.tw4[idx]);
        }
        line16_load_tw1<S>(T, L, P);
        auto last = [&]() {
            line16_load_itw1<S>(T, L, P);
#pragma unroll
            for (int v = 0; v < 4; v++) t4[v] = P.itw4[base + L.id + 16 * S * lnt_m16_neg(L.q, v)];
        };
        lnt_line16<S, LNT_SQUARE>(
            z, Mx, M8, lds, (u32)((r & 1) * lnt_line16_lds<S>()), L, T, P, 0,
            [&]() { S > 1 ? line16_load_tw2<S>(T, L, P) : last(); },
            [&]() { line16_load_itw2<S>(T, L, P); }, last);
#pragma unroll
        for (int v = 0; v < 4; v++) P.y[base + L.id + 16 * S * lnt_m16_neg(L.q, v)] = gl_mmul(z[v], t4[v]);
    }
}

// The row pass for rows of 256 S words (S <= 8), one row per workgroup of S waves: 4-step
// twiddles around the line, all factors fetched at the start.  MODEs as in lnt_row_body; slots
// base + 4 t + v.
template <int S, int MODE = LNT_SQUARE>
LNT_KFN void lnt_rowm_body(int tid, int bid, LView lds, const LntParams &P) {
    static_assert(S <= 8, "16 waves have no registers for the factors: lnt_row16_body");
    const u64 base = (u64)(256 * S) * (u64)bid;
    const LntLane16 L = lnt_lane16(tid);
    u64 z[4], t4[4];
    LntTw16 T;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const u64 idx = base + L.id + 16 * S * lnt_m16_word(L.q, e);
        z[e] = gl_mmul(P.y[idx], P.tw4[idx]);
    }
    line16_load_tw1<S>(T, L, P);
    line16_load_tw2<S>(T, L, P);
    if (MODE != LNT_FORWARD) {
        line16_load_itw2<S>(T, L, P);
        line16_load_itw1<S>(T, L, P);
#pragma unroll
        for (int v = 0; v < 4; v++) t4[v] = P.itw4[base + L.id + 16 * S * lnt_m16_neg(L.q, v)];
    }
    LntM16 Mx;
    LntM8 M8;
    lnt_m16_load(Mx, tid);
    if (S == 8) lnt_m8_load(M8, Mx, tid);
    auto loaded = [] {};
    lnt_line16<S, MODE>(z, Mx, M8, lds, 0, L, T, P, base + 4 * (u64)tid, loaded, loaded, loaded);
    if (MODE == LNT_FORWARD) return;
#pragma unroll
    for (int v = 0; v < 4; v++) P.y[base + L.id + 16 * S * lnt_m16_neg(L.q, v)] = gl_mmul(z[v], t4[v]);
}

// ------------------------------------------------------------------ 4096-word rows on the matrix cores
// The row pass for C = 4096 = 16^3 with the 16-point DFTs of mdft.hpp: one row per workgroup
// of W = 16 / GW waves, GW groups of 16 DFTs per wave and phase (4 GW words per thread).  With
// i = i1 + 256 j, i1 = a + 16 b; group h = GW w + g of wave w, lane (q, n):
//   phase 1: DFTs i1 = 16 h + n over j -> k2, twiddle omega_C^(i1 k2)     (twr)
//   phase 2: DFTs (k2 = h, a = n) over b -> kb, twiddle omega_256^(a kb)  (twr2)
//   phase 3: DFTs (k2 = h, kb = n) over a; square (or the product modes); the inverse takes
//            the result as it lies.
// A wave keeps its k2 between phase 1 and the inverse phase 2, so only the exchanges around
// these wait for the other waves.  LDS word (row r of 16 words, x) at 18 r + x: runs of 16 words
// start 16-byte aligned and 16 neighbouring runs cover all 64 banks, so the reads of adjacent
// word pairs are 128-bit and free of conflicts.  Transform-domain slot for MODE 1/2: base + 4 GW t + 4 g + place.
constexpr u32 LNT_ROW16_LDS = 256 * 18;
template <int GW, int MODE = LNT_SQUARE>
LNT_KFN void lnt_row16_body(int tid, int bid, LView lds, const LntParams &P) {
    const int w = LNT_UNIFORM(tid / 64), q = (tid % 64) / 16, n = tid % 16;
    const u64 base = (u64)4096 * (u64)bid;
    LntM16 M;
    u64 z[4], tw[4];
    if (GW > 1) lnt_m16_load(M, tid);  // ahead of the loads of phase 1 (94.4 -> 92.6 us per squaring at 2^22)
    // phase 1
#pragma unroll 1
    for (int h = GW * w; h < GW * w + GW; h++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = lnt_m16_word(q, e);
            const u64 idx = base + 16 * h + n + 256 * k;
            z[e] = gl_mmul(P.y[idx], P.tw4[idx]);  // 4-step twiddle of the column pass
            tw[e] = P.twr[256 * brev_v16(k) + 16 * h + n];
        }
        if (GW == 1) lnt_m16_load(M, tid);
        lnt_m16_dft(M, z);
#pragma unroll
        for (int v = 0; v < 4; v++)
            lds[(u32)(288 * lnt_m16_word(q, v) + 18 * n + h)] = gl_mmul(z[v], tw[v]);
    }
    LNT_SYNC();
    // phases 2 and 3, the pointwise step and their inverses
#pragma unroll 1
    for (int h = GW * w; h < GW * w + GW; h++) {
        const u32 row = (u32)(288 * h), own = row + (u32)(18 * n + 2 * q);  // this lane's words of run n
#pragma unroll
        for (int e = 0; e < 4; e++) {
            z[e] = lds[own + lnt_m16_word(0, e)];
            tw[e] = P.twr2[16 * brev_v16(lnt_m16_word(q, e)) + n];
        }
        lnt_m16_dft(M, z);
        LNT_WAVE_SYNC();
#pragma unroll
        for (int v = 0; v < 4; v++) lds[(u32)(row + 18 * lnt_m16_word(q, v) + n)] = gl_mmul(z[v], tw[v]);
        LNT_WAVE_SYNC();
#pragma unroll
        for (int e = 0; e < 4; e++) z[e] = lds[own + lnt_m16_word(0, e)];
        if (MODE != LNT_FORWARD) {
#pragma unroll
            for (int v = 0; v < 4; v++) tw[v] = P.itwr2[16 * brev_v16(n) + ((16 - lnt_m16_word(q, v)) & 15)];
        }
        lnt_m16_dft(M, z);
        LNT_WAVE_SYNC();
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const u64 slot = base + 4 * GW * (u64)tid + 4 * (h - GW * w) + v;
            if (MODE == LNT_FORWARD) P.y[slot] = z[v];
            else z[v] = gl_mmul(z[v], MODE == LNT_MULTIPLY ? P.f[slot] : z[v]);
        }
        if (MODE == LNT_FORWARD) continue;
        lnt_m16_dft(M, z);  // inverse phase 3: output place v is the word -k
#pragma unroll
        for (int v = 0; v < 4; v++)
            lds[(u32)(row + 18 * ((16 - lnt_m16_word(q, v)) & 15) + n)] = gl_mmul(z[v], tw[v]);
        LNT_WAVE_SYNC();
#pragma unroll
        for (int e = 0; e < 4; e++) {
            z[e] = lds[own + lnt_m16_word(0, e)];
            tw[e] = P.itwr[256 * brev_v16(h) + n + 16 * ((16 - lnt_m16_word(q, e)) & 15)];
        }
        lnt_m16_dft(M, z);  // inverse phase 2
        LNT_WAVE_SYNC();
#pragma unroll
        for (int v = 0; v < 4; v++)
            lds[(u32)(row + 18 * n + ((16 - lnt_m16_word(q, v)) & 15))] = gl_mmul(z[v], tw[v]);
    }
    if (MODE == LNT_FORWARD) return;
    LNT_SYNC();
    // inverse phase 1, inverse 4-step twiddle, store
#pragma unroll 1
    for (int h = GW * w; h < GW * w + GW; h++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            z[e] = lds[(u32)(288 * lnt_m16_word(q, e) + 18 * n + h)];
            tw[e] = P.itw4[base + 16 * h + n + 256 * ((16 - lnt_m16_word(q, e)) & 15)];
        }
        lnt_m16_dft(M, z);
#pragma unroll
        for (int v = 0; v < 4; v++)
            P.y[base + 16 * h + n + 256 * ((16 - lnt_m16_word(q, v)) & 15)] = gl_mmul(z[v], tw[v]);
    }
}

// ------------------------------------------------------------------ mixed-radix 3-phase rows
// Rows of C = BA * BB * BC words (8192 = 32*16*16 or 16*32*16, 16384 = 32*32*16 or
// 16*32*32), one row per workgroup of A = BB * BC threads holding BA words each.  The
// phases are those of the 3-phase columns (phase 1 over j of words t + A j; phase 2 items
// (k1, u), BA * BC of them; phase 3 items (k1, k2), BA * BB of them), with the 4-step
// twiddles at load and store and the square (or product) in the middle.  The phase-2
// twiddle is applied where phase 3 reads (and its inverse where inverse phase 3 writes).
// With BA = 16 a phase may have fewer items than threads (the rest wait at the barrier):
// 16 words per thread keep the register count low enough for twice the waves of BA = 32.
// LDS word of (k1, a = u + BC v): k1 * RS + v * (BC + 1) + u (padded runs).
template <int BA, int BB, int BC>
struct LntRow3m {
    static constexpr int A = BB * BC, C = BA * A;
    static constexpr int N2 = BA * BC, N3 = BA * BB;  // phase 2 / phase 3 items
    static constexpr int Q2 = (N2 + A - 1) / A, Q3 = (N3 + A - 1) / A;  // items per thread
    static constexpr int RS = BB * (BC + 1) + 1;
    static constexpr u32 LDS = (u32)(BA * RS);
    static_assert(N2 % A == 0 || A % N2 == 0, "phase 2 items");
    static_assert(N3 % A == 0 || A % N3 == 0, "phase 3 items");
};

template <int BA, int BB, int BC, int MODE = LNT_SQUARE>
LNT_KFN void lnt_row3m_body(int tid, int bid, LView lds, const LntParams &P) {
    using S = LntRow3m<BA, BB, BC>;
    constexpr int A = S::A, RS = S::RS, N2 = S::N2, N3 = S::N3, Q2 = S::Q2, Q3 = S::Q3;
    const int t = tid;
    const u64 base = (u64)P.C * (u64)bid;
    auto pos = [](int k1, int a) { return (u32)(k1 * RS + (a / BC) * (BC + 1) + a % BC); };
    u64 a[BA];
#pragma unroll
    for (int j = 0; j < BA; j++) {
        const u64 idx = base + t + (u64)A * j;
        a[j] = gl_mmul(P.y[idx], P.tw4[idx]);  // 4-step twiddle of the column pass
    }
    // phase 1
    dft_fwd<BA>(a);
#pragma unroll
    for (int rho = 1; rho < BA; rho++) a[rho] = gl_mmul(a[rho], P.twr[(u64)rho * A + t]);
#pragma unroll
    for (int rho = 0; rho < BA; rho++) lds[pos(brev_c<BA>(rho), t)] = a[rho];
    LNT_SYNC();
    // phase 2 (each item rewrites exactly the LDS words it read)
#pragma unroll
    for (int q = 0; q < Q2; q++) {
        const int I = q * A + t, k1 = I / BC, u = I % BC;
        if (N2 >= A || I < N2) {
            u64 b[BB];
#pragma unroll
            for (int v = 0; v < BB; v++) b[v] = lds[pos(k1, u + BC * v)];
            dft_fwd<BB>(b);
#pragma unroll
            for (int rho = 0; rho < BB; rho++) lds[pos(k1, u + BC * brev_c<BB>(rho))] = b[rho];
        }
    }
    LNT_SYNC();
    // phase 3 (with the phase-2 twiddle w_A^(u k2) at the read, where every thread has an
    // item: phase 2 keeps only its DFT registers live), the pointwise step, inverse phase 3
    // and the inverse phase-2 twiddle.  Item q of thread t: slots (q * A + t) * BC + rho.
#pragma unroll
    for (int q = 0; q < Q3; q++) {
        const int I = q * A + t, k1 = I / BB, k2 = I % BB;
        if (N3 >= A || I < N3) {
            const u64 tb = (u64)brev_c<BB>(k2) * BC;  // twr2 row of k2
            u64 e[BC];
#pragma unroll
            for (int u = 0; u < BC; u++) e[u] = gl_mmul(lds[pos(k1, u + BC * k2)], P.twr2[tb + u]);
            dft_fwd<BC>(e);
            const u64 so = base + (u64)I * BC;
            if (MODE == LNT_FORWARD) {
#pragma unroll
                for (int i = 0; i < BC; i++) P.y[so + i] = e[i];
                continue;
            }
            if (MODE == LNT_MULTIPLY) {
#pragma unroll
                for (int i = 0; i < BC; i++) e[i] = gl_mmul(e[i], P.f[so + i]);
            } else {
#pragma unroll
                for (int i = 0; i < BC; i++) e[i] = gl_mmul(e[i], e[i]);
            }
            dft_inv<BC>(e);
#pragma unroll
            for (int u = 0; u < BC; u++) lds[pos(k1, u + BC * k2)] = gl_mmul(e[u], P.itwr2[tb + u]);
        }
    }
    if (MODE == LNT_FORWARD) return;
    LNT_SYNC();
    // inverse phase 2 (its twiddle was applied by inverse phase 3)
#pragma unroll
    for (int q = 0; q < Q2; q++) {
        const int I = q * A + t, k1 = I / BC, u = I % BC;
        if (N2 >= A || I < N2) {
            u64 b[BB];
#pragma unroll
            for (int rho = 0; rho < BB; rho++) b[rho] = lds[pos(k1, u + BC * brev_c<BB>(rho))];
            dft_inv<BB>(b);
#pragma unroll
            for (int v = 0; v < BB; v++) lds[pos(k1, u + BC * v)] = b[v];
        }
    }
    LNT_SYNC();
    // inverse phase 1, inverse 4-step twiddle, store
#pragma unroll
    for (int rho = 0; rho < BA; rho++) {
        u64 v = lds[pos(brev_c<BA>(rho), t)];
        a[rho] = rho ? gl_mmul(v, P.itwr[(u64)rho * A + t]) : v;
    }
    dft_inv<BA>(a);
#pragma unroll
    for (int j = 0; j < BA; j++) {
        const u64 idx = base + t + (u64)A * j;
        P.y[idx] = gl_mmul(a[j], P.itw4[idx]);
    }
}

// ------------------------------------------------------------------ small residues
// One workgroup of B2 threads runs `iters` whole iterations on n = B1 * B2 words kept
// in LDS (natural order, field elements).  LDS words: max(n, B1 * (B2 + PAD)).
// MODE 0: `iters` squarings.  MODE 1 (iters = 1): forward transform of x into y (slot
// t*B1 + i), x unchanged.  MODE 2 (iters = 1): x <- x * (the operand whose transform is f).
template <int B1, int B2, int M, int MODE = LNT_SQUARE>
LNT_KFN void lnt_small_body(int tid, LView lds, const LntParams &P, u32 iters, bool sub2_first,
                            bool ll) {
    constexpr int RP = B1 / B2;
    constexpr int S = B2 + LNT_PAD;
    constexpr u32 N = B1 * B2;
    const int t = tid;
#pragma unroll
    for (int j = 0; j < B1; j++) lds[(u32)(t + B2 * j)] = P.x[(u64)t + B2 * j];
    LNT_SYNC();
    for (u32 it = 0; it < iters; it++) {
        // tables re-read each iteration (from cache) instead of living in registers
        const u64 *pw = P.w.p, *puw = P.uw.p, *ptw = P.twr.p, *pitw = P.itwr.p;
        LNT_OPAQUE(pw);
        LNT_OPAQUE(puw);
        LNT_OPAQUE(ptw);
        LNT_OPAQUE(pitw);
        const GView<const u64> Tw{pw, P.w.n}, Tuw{puw, P.uw.n}, Ttw{ptw, P.twr.n}, Titw{pitw, P.itwr.n};
        // carry over this thread's chunk [t*B1, (t+1)*B1), streamed in pieces of PK
        // digits; each piece's halo is the M pre-carry values just before it.
        {
            constexpr int PK = B1 < 16 ? B1 : 16;
            const u32 g0 = (u32)t * B1;
            int64_t halo[M];
#pragma unroll
            for (int j = 0; j < M; j++) halo[j] = gl_to_i64(lds[(g0 + N - M + j) & (N - 1)]);
            LNT_SYNC();  // every halo read before any chunk is overwritten
            const bool sub2 = it == 0 ? sub2_first : ll;
            for (int s = 0; s < B1 / PK; s++) {
                int64_t v[M + PK];
#pragma unroll
                for (int j = 0; j < M; j++) v[j] = halo[j];
#pragma unroll
                for (int j = 0; j < PK; j++) v[M + j] = gl_to_i64(lds[g0 + s * PK + j]);
#pragma unroll
                for (int j = 0; j < M; j++) halo[j] = v[PK + j];
                lnt_carry_run<M, PK>(v, P.p, P.log_n, g0 + s * PK, P.levels, sub2);
#pragma unroll
                for (int j = 0; j < PK; j++)
                    lds[g0 + s * PK + j] =
                        P.bias ? (u64)(u32)(v[M + j] + (int64_t(1) << 31)) : gl_from_i64(v[M + j]);
            }
            LNT_SYNC();
        }
        u64 a[B1];
#pragma unroll
        for (int j = 0; j < B1; j++) {
            const u32 i = t + B2 * j;
            a[j] = P.bias ? gl_mul_biased((u32)lds[i], Tw[2 * i], Tw[2 * i + 1]) : gl_mul(lds[i], Tw[2 * i]);
        }
        dft_fwd<B1>(a);
        if (B2 > 1) {
#pragma unroll
            for (int rho = 1; rho < B1; rho++) a[rho] = gl_mmul(a[rho], Ttw[(u64)rho * B2 + t]);
        }
        LNT_SYNC();
#pragma unroll
        for (int rho = 0; rho < B1; rho++) lds[(u32)(brev_c<B1>(rho) * S + t)] = a[rho];
        LNT_SYNC();
#pragma unroll
        for (int q = 0; q < RP; q++) {
            const int k2 = t * RP + q;
#pragma unroll
            for (int i1 = 0; i1 < B2; i1++) a[q * B2 + i1] = lds[(u32)(k2 * S + i1)];
            dft_fwd<B2>(a + q * B2);
            if (MODE == LNT_FORWARD) {
#pragma unroll
                for (int i1 = 0; i1 < B2; i1++) P.y[(u64)t * B1 + q * B2 + i1] = a[q * B2 + i1];
                continue;
            }
            if (MODE == LNT_MULTIPLY) {
#pragma unroll
                for (int i1 = 0; i1 < B2; i1++)
                    a[q * B2 + i1] = gl_mul(a[q * B2 + i1], P.f[(u64)t * B1 + q * B2 + i1]);
            } else {
#pragma unroll
                for (int i1 = 0; i1 < B2; i1++) a[q * B2 + i1] = gl_sqr(a[q * B2 + i1]);
            }
            dft_inv<B2>(a + q * B2);
#pragma unroll
            for (int i1 = 0; i1 < B2; i1++) lds[(u32)(k2 * S + i1)] = a[q * B2 + i1];
        }
        if (MODE == LNT_FORWARD) return;
        LNT_SYNC();
#pragma unroll
        for (int rho = 0; rho < B1; rho++) {
            u64 v = lds[(u32)(brev_c<B1>(rho) * S + t)];
            a[rho] = (B2 > 1 && rho > 0) ? gl_mmul(v, Titw[(u64)rho * B2 + t]) : v;
        }
        dft_inv<B1>(a);
        LNT_SYNC();
#pragma unroll
        for (int j = 0; j < B1; j++) {
            const u32 i = t + B2 * j;
            lds[i] = gl_mul(a[j], Tuw[i]);
        }
        LNT_SYNC();
    }
#pragma unroll
    for (int j = 0; j < B1; j++) P.x[(u64)t + B2 * j] = lds[(u32)(t + B2 * j)];
}

// ------------------------------------------------------------------ n = 64 and 128 in one wave
// n = N1 * 8 words (N1 = 8, 16) in one wave with N1-point DFTs over j (i = i1 + 8 j) and 8-point
// DFTs over i1, both on the matrix cores.  Phase 1 has eight DFTs, so the lanes n >= 8 repeat
// those of n - 8 and write nothing.  One wave needs no barrier, and all factors stay in registers.
// Tables as for the 2-phase kernel (line N1 x 8).  LDS: n words in natural order, then the
// transform, word (k2, i1) at 10 k2 + i1.  MODEs as above.
template <int N1>
constexpr u32 lnt_tiny_lds() { return 8 * N1 + 10 * N1; }

template <int N1, int M, int MODE = LNT_SQUARE>
LNT_KFN void lnt_tiny_body(int tid, LView lds, const LntParams &P, u32 iters, bool sub2_first, bool ll) {
    constexpr u32 N = 8 * N1, Z = N;
    constexpr int W1 = N1 / 4;  // phase-1 words per lane
    constexpr int PK = N / 64;  // digits per thread in the carry
    const int q = tid / 16, n = tid % 16, c = n & 7, k2 = N1 == 16 ? n : c;
    const bool act = n < 8, act2 = N1 == 16 || act;
    // phase-1 input j / output k2 at place e, and the inverse's output j at place v
    auto word = [&](int e) { return N1 == 16 ? lnt_m16_word(q, e) : 2 * q + e; };
    auto neg = [&](int e) { return (N1 - word(e)) & (N1 - 1); };
    LntM16 Mx;
    LntM8 M8;
    lnt_m16_load(Mx, tid);
    lnt_m8_load(M8, Mx, tid);
    u64 wv[W1], wb[W1], tw[W1], uv[W1], itw[2];
    const u64 r2 = gl_mul(GL_R, GL_R);
#pragma unroll
    for (int e = 0; e < W1; e++) {
        const u32 i = (u32)(c + 8 * word(e));
        wv[e] = P.w[2 * i];
        wb[e] = P.w[2 * i + 1];
        tw[e] = P.twr[8 * (N1 == 16 ? brev_v16(word(e)) : brev_v16(word(e)) >> 1) + c];
        uv[e] = gl_mul(P.uw[c + 8 * neg(e)], r2);  // (the 2^128 as in lnt_small16_body)
    }
#pragma unroll
    for (int v = 0; v < 2; v++)
        itw[v] = P.itwr[8 * (N1 == 16 ? brev_v16(k2) : brev_v16(k2) >> 1) + ((8 - 2 * q - v) & 7)];
    auto dft1 = [&](u64 (&z)[4]) {
        if (N1 == 16) lnt_m16_dft(Mx, z);
        else {
            u64 h[2] = {z[0], z[1]};
            lnt_m8_dft(M8, Mx, h);
            z[0] = h[0], z[1] = h[1];
        }
    };
#pragma unroll
    for (int j = 0; j < PK; j++) lds[(u32)(tid + 64 * j)] = P.x[(u64)tid + 64 * j];
    LNT_WAVE_SYNC();
    for (u32 it = 0; it < iters; it++) {
        {
            const u32 g0 = PK * (u32)tid;
            int64_t v[M + PK];
#pragma unroll
            for (int j = 0; j < M + PK; j++) v[j] = gl_to_i64(lds[(g0 + N - M + j) & (N - 1)]);
            LNT_WAVE_SYNC();  // every word read before any is overwritten
            lnt_carry_run<M, PK>(v, P.p, P.log_n, g0, P.levels, it == 0 ? sub2_first : ll);
#pragma unroll
            for (int j = 0; j < PK; j++)
                lds[g0 + j] = P.bias ? (u64)(u32)(v[M + j] + (int64_t(1) << 31)) : gl_from_i64(v[M + j]);
        }
        LNT_WAVE_SYNC();
        u64 z[4] = {}, g[2];
#pragma unroll
        for (int e = 0; e < W1; e++) {
            const u64 d = lds[(u32)(c + 8 * word(e))];
            z[e] = P.bias ? gl_mul_biased((u32)d, wv[e], wb[e]) : gl_mul(d, wv[e]);
        }
        dft1(z);
#pragma unroll
        for (int v = 0; v < W1; v++) {
            const u64 t = gl_mmul(z[v], tw[v]);
            if (act) lds[Z + (u32)(10 * word(v) + c)] = t;
        }
        LNT_WAVE_SYNC();
#pragma unroll
        for (int v = 0; v < 2; v++) g[v] = lds[Z + (u32)(10 * k2 + 2 * q + v)];
        lnt_m8_dft(M8, Mx, g);
        const u64 slot = 2 * (u64)(q * N1 + k2);
#pragma unroll
        for (int v = 0; v < 2; v++) {
            if (MODE == LNT_FORWARD) {
                if (act2) P.y[slot + v] = g[v];
            } else {
                g[v] = gl_mmul(g[v], MODE == LNT_MULTIPLY ? P.f[slot + v] : g[v]);
            }
        }
        if (MODE == LNT_FORWARD) return;
        lnt_m8_dft(M8, Mx, g);
        LNT_WAVE_SYNC();
#pragma unroll
        for (int v = 0; v < 2; v++) {
            const u64 t = gl_mmul(g[v], itw[v]);
            if (act2) lds[Z + (u32)(10 * k2 + ((8 - 2 * q - v) & 7))] = t;
        }
        LNT_WAVE_SYNC();
#pragma unroll
        for (int e = 0; e < W1; e++) z[e] = lds[Z + (u32)(10 * word(e) + c)];
        dft1(z);
#pragma unroll
        for (int v = 0; v < W1; v++) {
            const u64 t = gl_mmul(z[v], uv[v]);
            if (act) lds[(u32)(c + 8 * neg(v))] = t;
        }
        LNT_WAVE_SYNC();
    }
#pragma unroll
    for (int j = 0; j < PK; j++) P.x[(u64)tid + 64 * j] = lds[(u32)(tid + 64 * j)];
}

// ------------------------------------------------------------------ small residues on the matrix cores
// One workgroup of S waves runs `iters` iterations on n = 256 S words, a line of lnt_line16
// between the carry and weights and the unweights.  One test is a chain of dependent steps on
// one compute unit, so what counts is its latency: four words per thread put four times the
// waves of the former 16-word kernels to work on it, an iteration has four barriers, and up to
// S = 8 the factors of a thread's words stay in registers (at S = 8, where eight waves have 256
// registers each, all but 4 of them, and all but 12 with a halo of eight digits).  For n = 4096 that would take more
// than the 128 registers of 16 waves: weights and twiddles are re-read (from the L2, ahead of
// their use) and the unweights lie in LDS.
// LDS: two regions, the residue (or its digits) in natural order in one while the other holds
// the transform.  MODEs as above.
template <int S>
constexpr u32 lnt_small16_lds() { return 2 * lnt_line16_lds<S>() + (S == 16 ? 256 * S : 0); }

template <int S, int M, int MODE = LNT_SQUARE>
LNT_KFN void lnt_small16_body(int tid, LView lds, const LntParams &P, u32 iters, bool sub2_first, bool ll) {
    constexpr u32 N = 256 * S;
    constexpr bool RES = S <= 8;                    // factors live in registers
    constexpr u32 U = 2 * lnt_line16_lds<S>();      // unweights (S = 16)
    LntLane16 L = lnt_lane16(tid);
    LntM16 Mx;
    LntM8 M8;
    lnt_m16_load(Mx, tid);
    if (S == 8) lnt_m8_load(M8, Mx, tid);
    u64 wv[4], wb[4], uv[4];
    LntTw16 T;
    auto load_w = [&]() {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const u32 i = (u32)(L.id + 16 * S * lnt_m16_word(L.q, e));
            wv[e] = P.w[2 * i];
            wb[e] = P.w[2 * i + 1];
        }
    };
    if (RES) {
        load_w();
        line16_load_tw1<S>(T, L, P);
        line16_load_tw2<S>(T, L, P);
        line16_load_itw2<S>(T, L, P);
        line16_load_itw1<S>(T, L, P);
    }
    const u64 r2 = gl_mul(GL_R, GL_R);
#pragma unroll
    for (int v = 0; v < 4; v++) {
        // unweight of output place v, times 2^128: one 2^64 for its Montgomery multiply and one
        // for the factor 2^-64 that the pointwise product leaves
        const u32 i = (u32)(L.id + 16 * S * lnt_m16_neg(L.q, v));
        const u64 u = gl_mul(P.uw[i], r2);
        if (RES) uv[v] = u;
        else lds[U + i] = u;
    }
    u32 A = 0, B = lnt_line16_lds<S>();
#pragma unroll
    for (int j = 0; j < 4; j++) lds[A + (u32)(tid + 64 * S * j)] = P.x[(u64)tid + 64 * S * j];
    LNT_SYNC();
    for (u32 it = 0; it < iters; it++) {
        if (!RES) {
            LNT_OPAQUE_LANE(tid);
            L = lnt_lane16(tid);
        }
        // carry of digits 4 tid .. 4 tid + 3 from the M pre-carry words before them on: A -> B
        {
            const u32 g0 = 4 * (u32)tid;
            int64_t v[M + 4];
#pragma unroll
            for (int j = 0; j < M; j++) v[j] = gl_to_i64(lds[A + ((g0 + N - M + j) & (N - 1))]);
#pragma unroll
            for (int j = 0; j < 4; j++) v[M + j] = gl_to_i64(lds[A + g0 + j]);
            lnt_carry_run<M, 4>(v, P.p, P.log_n, g0, P.levels, it == 0 ? sub2_first : ll);
#pragma unroll
            for (int j = 0; j < 4; j++)
                lds[B + g0 + j] = P.bias ? (u64)(u32)(v[M + j] + (int64_t(1) << 31)) : gl_from_i64(v[M + j]);
        }
        if (!RES) {
            load_w();
            line16_load_tw1<S>(T, L, P);
        }
        LNT_SYNC();
        // weights from B, the line in A, unweights into B: the residue of the next iteration
        u64 z[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const u64 d = lds[B + (u32)(L.id + 16 * S * lnt_m16_word(L.q, e))];
            z[e] = P.bias ? gl_mul_biased((u32)d, wv[e], wb[e]) : gl_mul(d, wv[e]);
        }
        lnt_line16<S, MODE>(
            z, Mx, M8, lds, A, L, T, P, 4 * (u64)tid, [&]() { if (!RES) line16_load_tw2<S>(T, L, P); },
            [&]() { if (!RES) line16_load_itw2<S>(T, L, P); }, [&]() { if (!RES) line16_load_itw1<S>(T, L, P); });
        if (MODE == LNT_FORWARD) return;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const u32 i = (u32)(L.id + 16 * S * lnt_m16_neg(L.q, v));
            lds[B + i] = gl_mmul(z[v], RES ? uv[v] : lds[U + i]);
        }
        LNT_SYNC();
        const u32 c = A;
        A = B;
        B = c;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) P.x[(u64)tid + 64 * S * j] = lds[A + (u32)(tid + 64 * S * j)];
}

// ------------------------------------------------------------------ tables
// Twiddle tables are in Montgomery form (times GL_R) for gl_mmul.
// Twiddles of a line of L = B1 * B2 words: tw[rho * B2 + t] = omega_L^(t * brev_B1(rho)).
GL_HD u64 lnt_line_tw(u64 omega_L, u32 B1, u32 B2, u32 idx) {
    u32 rho = idx / B2, t = idx % B2;
    u32 br = 0;
    for (u32 b = 1, v = rho; b < B1; b <<= 1, v >>= 1) br = (br << 1) | (v & 1);
    return gl_mul(gl_pow(omega_L, (u64)t * br), GL_R);
}

// 4-step twiddle for slot idx = c + C * r', r' = t*B1 + q*B2 + rho' (column line B1 x B2):
// omega_n^(c * kcol), kcol = B1 * brev_B2(rho') + t*(B1/B2) + q.
GL_HD u64 lnt_tw4(u64 omega_n, u32 C, u32 B1, u32 B2, u64 idx) {
    u32 c = (u32)(idx % C);
    u32 rr = (u32)(idx / C);
    u32 t = rr / B1, q = (rr % B1) / B2, rp = rr % B2;
    u32 br = 0;
    for (u32 b = 1, v = rp; b < B2; b <<= 1, v >>= 1) br = (br << 1) | (v & 1);
    u64 kcol = (u64)B1 * br + (u64)t * (B1 / B2) + q;
    return gl_mul(gl_pow(omega_n, (u64)c * kcol), GL_R);
}

// 4-step twiddle of a 3-phase column (radices BA, BB, BC): slot s = t*BA + q*BC + rho
// holds frequency k1 + BA (k2 + BB brev_BC(rho)), (k1, k2) = (I / BB, I % BB), I = q*A + t.
GL_HD u64 lnt_tw4_3(u64 omega_n, u32 C, u32 BA, u32 BB, u32 BC, u64 idx) {
    const u32 c = (u32)(idx % C), s = (u32)(idx / C), A = BB * BC;
    const u32 t = s / BA, q = (s % BA) / BC, rho = s % BC;
    const u32 I = q * A + t, k1 = I / BB, k2 = I % BB;
    u32 br = 0;
    for (u32 b = 1, v = rho; b < BC; b <<= 1, v >>= 1) br = (br << 1) | (v & 1);
    const u64 kcol = k1 + (u64)BA * (k2 + (u64)BB * br);
    return gl_mul(gl_pow(omega_n, (u64)c * kcol), GL_R);
}

// 4-step twiddle of a matrix-core column (256 S words): slot (16 k2 + kb) S + k3 holds frequency
// k2 + 16 (kb + 16 k3).
GL_HD u64 lnt_tw4_m(u64 omega_n, u32 C, u32 S, u64 idx) {
    const u32 c = (u32)(idx % C), s = (u32)(idx / C);
    const u32 k2 = s / (16 * S), kb = s / S % 16, k3 = s % S;
    return gl_mul(gl_pow(omega_n, (u64)c * (k2 + 16 * (kb + 16 * k3))), GL_R);
}

// Large-path weight tables (the factorisation at lnt_wexp), row slots 2r + h.
// Unweights: B^f_r (B the inverse weight base), times m = 2 when h = 1, times GL_R^2: one
// GL_R for the Montgomery multiply that applies it, one for the 2^-64 the square left.
GL_HD u64 lnt_row_factor(u64 B, u64 m, u32 p, u32 n, u32 C, u32 slot) {
    const u64 v = gl_mul(gl_pow(B, lnt_wexp(p, n, (u64)C * (slot >> 1))), gl_mul(GL_R, GL_R));
    return (slot & 1) ? gl_mul(v, m) : v;
}
// Weights: word i is half of the pair (w, -2^31 w) of slot i / 2 (gl_mul_biased takes both),
// w = B^f_r, halved when h = 1.
GL_HD u64 lnt_weight_pair(u64 Bw, u32 p, u32 n, u32 C, u32 i) {
    const u32 slot = i >> 1;
    u64 w = gl_pow(Bw, lnt_wexp(p, n, (u64)C * (slot >> 1)));
    if (slot & 1) w = gl_mul(w, (GL_P + 1) / 2);
    return (i & 1) ? gl_mul(w, GL_P - (1ull << 31)) : w;
}
// Column factor B^e_c times s (s = 1 for weights, n^-1 for unweights), c = idx mod C.
GL_HD u64 lnt_col_factor(u64 B, u64 s, u32 p, u32 n, u32 C, u64 idx) {
    return gl_mul(gl_pow(B, lnt_wexp(p, n, idx % C)), s);
}

// IBDWT weight of digit i (common/pre_calculation.cu:23-36): B^(n - (p i mod n)) for
// i > 0 and 1 for i = 0, with B = 7^((P-1)/192/n*5) (so B^n = 2).
GL_HD u64 lnt_weight(u64 Bw, u32 p, u32 n, u32 i) {
    if (i == 0) return 1;
    u32 r = (u32)((u64)p * i) & (n - 1);
    return gl_pow(Bw, (u64)(n - r));
}
