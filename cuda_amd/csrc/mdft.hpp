// 16-point DFTs over GF(2^64 - 2^32 + 1) on the matrix cores.
//
// omega_16 = 2^12, so a 16-point DFT only shifts and adds its inputs: as an integer matrix it
// maps the 16 * 8 bytes of the inputs to 16 * 8 byte-weighted limbs of the outputs.  Byte p of
// input j adds byte * 2^(8p + 12jk) to output k; with 2^96 = -1 and 2^64 = 2^32 - 1 that lands
// on one limb (or on limbs i and i + 4 with opposite signs), times 1 or 16.  Every entry fits
// a signed byte, every sum 17 bits, so v_mfma_i32_16x16x64_i8 computes it exactly.
//
// One matrix instruction takes 16 DFTs (its columns).  In a wave, lane (q, n) (n = lane % 16,
// q = lane / 16) holds the words j = 2q, 2q+1, 8+2q, 9+2q of DFT n, two 128-bit operands, and
// receives the words k = 2q, 2q+1, 8+2q, 9+2q of its transform, so a transform's output can be
// the next one's input without an exchange.  The inverse uses the same matrix: output slot k
// is then the word -k mod 16.
//
// Per word the vector units only flip the bytes' signs (2 instructions) and put eight limbs
// together (11), where the register DFT (dft.hpp) takes 41; the 16 matrix instructions of
// 16 DFTs take 16 cycles each (64 cycles per 64 words), beside the vector work of other waves.
//
// Bytes are signed for the matrix unit: with b - 128 for every byte each word loses 128 R,
// R = 2^0 + 2^8 + ... + 2^56, which the DFT turns into -2048 R on output 0 alone.
#pragma once
#include "gl64.hpp"
#include "simt.hpp"

// Word held by lane group q at place e (inputs j and outputs k alike).
GL_HD constexpr int lnt_m16_word(int q, int e) { return 8 * (e >> 1) + 2 * q + (e & 1); }

// Entry of limb `limb` of output k for byte p of input j.
GL_HD constexpr int lnt_m16_entry(int limb, int k, int j, int p) {
    const int s = (12 * j * k) % 192 + 8 * p;  // byte * 2^s, 0 <= s < 256
    const int e = s % 192, pos = (e % 96) / 8, val = (e >= 96 ? -1 : 1) << (e % 8);
    // limbs 8 .. 11: 2^(64 + 8m) = 2^(32 + 8m) - 2^(8m)
    return pos < 8 ? (pos == limb ? val : 0) : (limb == pos - 4 ? val : limb == pos - 8 ? -val : 0);
}

// Operand tiles: tile (v, h) holds the rows (q, i) = limb 4h + i of output word (q, v) and the
// columns of inputs j < 8 (16 bytes per lane: row lane % 16, inputs 2q', 2q'+1 of q' = lane / 16).
// For inputs j >= 8 the tile is the same times (-1)^k, k = v mod 2: tiles 8 .. 11 are the
// negated tiles of odd v.
constexpr int LNT_M16_TILES = 12;
struct LntM16Table {
    signed char b[LNT_M16_TILES * 64 * 16];
};
// The same for 8-point DFTs (omega_8 = 2^24, every entry 0 or +-1): lane (q, n) holds the words
// 2q, 2q+1 of DFT n, one matrix instruction per tile (v, h).
constexpr int LNT_M8_TILES = 4;
struct LntM8Table {
    signed char b[LNT_M8_TILES * 64 * 16];
};
constexpr LntM8Table lnt_m8_make() {
    LntM8Table t{};
    for (int tile = 0; tile < LNT_M8_TILES; tile++)
        for (int lane = 0; lane < 64; lane++)
            for (int byte = 0; byte < 16; byte++) {
                const int row = lane % 16, k = 2 * (row / 4) + tile / 2, limb = 4 * (tile % 2) + row % 4;
                const int j = 2 * (lane / 16) + byte / 8;
                t.b[(tile * 64 + lane) * 16 + byte] = (signed char)lnt_m16_entry(limb, 2 * k, j, byte % 8);
            }
    return t;
}
constexpr LntM16Table lnt_m16_make() {
    LntM16Table t{};
    for (int tile = 0; tile < LNT_M16_TILES; tile++) {
        const bool neg = tile >= 8;
        const int v = neg ? 1 + 2 * ((tile - 8) / 2) : tile / 2, h = tile % 2;
        for (int lane = 0; lane < 64; lane++)
            for (int byte = 0; byte < 16; byte++) {
                const int row = lane % 16, k = lnt_m16_word(row / 4, v), limb = 4 * h + row % 4;
                const int j = 2 * (lane / 16) + byte / 8;
                const int val = lnt_m16_entry(limb, k, j, byte % 8);
                t.b[(tile * 64 + lane) * 16 + byte] = (signed char)(neg ? -val : val);
            }
    }
    return t;
}

// Every limb starts at its offset o_i, which keeps it positive (no limb of the sums exceeds
// 202 * 128 = 25856 in magnitude) and weighs 2^9 P = 0 in all.
GL_HD constexpr int lnt_m16_offset(int i) {
    return i == 0 ? 0x7000 : i == 1 ? 0x7092 : i == 2 ? 0x708f : i == 3 ? 0x808f
         : i == 4 ? 0x707f : i == 5 ? 0x708d : i == 6 ? 0x708f : 0x1ff8f;
}
static_assert((lnt_m16_offset(0) + ((u64)lnt_m16_offset(1) << 8) + ((u64)lnt_m16_offset(2) << 16) +
               ((u64)lnt_m16_offset(3) << 24)) == (u64(0x81) << 32) + 0x200 &&
              (lnt_m16_offset(4) + ((u64)lnt_m16_offset(5) << 8) + ((u64)lnt_m16_offset(6) << 16) +
               ((u64)lnt_m16_offset(7) << 24)) == (u64(0x200) << 32) - 0x200 - 0x81,
              "the offsets add up to 2^9 P");

// Eight limbs 0 < l < 2^18 (limb i weighs 2^8i), and dc (1 + 2^32) when the output is place 0,
// to hi:lo plus carry 2^64, any representative.  With a0 .. a3 of 16 bits' weight each,
// u = a0 + 2^16 a1 and v = a2 + 2^16 a3 = v0 + 2^32 v1:  u + 2^32 v = u - v1 + 2^32 (v0 + v1),
// and the high word's sum may carry (about once in 2^23 words).
template <bool DC>
GL_HD u32 lnt_limbs(const int (&l)[8], u64 dc, u32 k16, int km1, u32 &lo, u32 &t) {
    const u32 a0 = (u32)(l[0] + (l[1] << 8)), a1 = (u32)(l[2] + (l[3] << 8));
    const u32 a2 = (u32)(l[4] + (l[5] << 8)), a3 = (u32)(l[6] + (l[7] << 8));  // < 2^26
    const u64 v = (u64)a3 * k16 + (DC ? a2 + dc : a2);
    const int v1 = (int)(v >> 32);
    const u64 u = (u64)((int64_t)v1 * km1 + (int64_t)((u64)a1 * k16 + (DC ? a0 + dc : a0)));
    lo = (u32)u;
    t = (u32)v1 + (u32)(u >> 32);  // < 2^12
    return (u32)v;                 // the high word is this plus t
}

constexpr u64 LNT_M16_DC = 2048ull * 0x01010101ull;  // 2048 R = DC + 2^32 DC
constexpr u64 LNT_M8_DC = 1024ull * 0x01010101ull;   // 8 points: 1024 R

#if defined(LNT_EMU)
// Emulation: the words of a wave meet in an array between two barriers, and the sums run over
// the same operand bytes as on the device.
static u64 lnt_emu_wave[1024][4];
static const LntM16Table lnt_m16_tab = lnt_m16_make();
struct LntM16 {
    int tid;
};
LNT_KFN void lnt_m16_load(LntM16 &M, int tid) { M.tid = tid; }
LNT_KFN void lnt_m16_dft(const LntM16 &M, u64 (&x)[4]) {
    const int tid = M.tid, q = (tid % 64) / 16, wb = tid & ~63, n = tid % 16;
    for (int e = 0; e < 4; e++) lnt_emu_wave[tid][e] = x[e] ^ 0x8080808080808080ull;
    LNT_SYNC();
    for (int v = 0; v < 4; v++) {
        int l[8];
        for (int limb = 0; limb < 8; limb++) {
            const int h = limb / 4, row = 4 * q + limb % 4;
            int sum = 0;
            for (int s = 0; s < 2; s++) {
                const int tile = (s == 1 && v % 2) ? 8 + (v / 2) * 2 + h : 2 * v + h;
                for (int qq = 0; qq < 4; qq++)
                    for (int byte = 0; byte < 16; byte++) {
                        const u64 w = lnt_emu_wave[wb + 16 * qq + n][2 * s + byte / 8];
                        sum += lnt_m16_tab.b[(tile * 64 + 16 * qq + row) * 16 + byte] *
                               (int)(signed char)(w >> (8 * (byte % 8)));
                    }
            }
            l[limb] = sum + lnt_m16_offset(limb);
            LNT_CHECK(l[limb] > 0 && l[limb] < 1 << 18, "limb range");
        }
        u32 lo, t;
        const u32 v0 = v == 0 ? lnt_limbs<true>(l, q == 0 ? LNT_M16_DC : 0, 65536, -1, lo, t)
                              : lnt_limbs<false>(l, 0, 65536, -1, lo, t);
        const u64 hi = (u64)v0 + t;
        x[v] = ((hi << 32) | lo) + (hi >> 32 ? GL_EPS : 0);
    }
    LNT_SYNC();
}
static const LntM8Table lnt_m8_tab = lnt_m8_make();
struct LntM8 {
    int tid;
};
LNT_KFN void lnt_m8_load(LntM8 &M, const LntM16 &, int tid) { M.tid = tid; }
LNT_KFN void lnt_m8_dft(const LntM8 &M, const LntM16 &, u64 (&x)[2]) {
    const int tid = M.tid, q = (tid % 64) / 16, wb = tid & ~63, n = tid % 16;
    for (int e = 0; e < 2; e++) lnt_emu_wave[tid][e] = x[e] ^ 0x8080808080808080ull;
    LNT_SYNC();
    for (int v = 0; v < 2; v++) {
        int l[8];
        for (int limb = 0; limb < 8; limb++) {
            int sum = 0;
            for (int qq = 0; qq < 4; qq++)
                for (int byte = 0; byte < 16; byte++)
                    sum += lnt_m8_tab.b[((2 * v + limb / 4) * 64 + 16 * qq + 4 * q + limb % 4) * 16 + byte] *
                           (int)(signed char)(lnt_emu_wave[wb + 16 * qq + n][byte / 8] >> (8 * (byte % 8)));
            l[limb] = sum + lnt_m16_offset(limb);
            LNT_CHECK(l[limb] > 0 && l[limb] < 1 << 18, "limb range");
        }
        u32 lo, t;
        const u32 v0 = v == 0 ? lnt_limbs<true>(l, q == 0 ? LNT_M8_DC : 0, 65536, -1, lo, t)
                              : lnt_limbs<false>(l, 0, 65536, -1, lo, t);
        const u64 hi = (u64)v0 + t;
        x[v] = ((hi << 32) | lo) + (hi >> 32 ? GL_EPS : 0);
    }
    LNT_SYNC();
}
#else
typedef int lnt_v4i __attribute__((ext_vector_type(4)));
static __device__ const LntM16Table lnt_m16_tab = lnt_m16_make();
struct LntM16 {
    lnt_v4i t[LNT_M16_TILES], o[2];
    u64 dc;  // constant of output place 0 (lane group 0 holds output 0)
    u32 k16;
    int km1;
};
LNT_KFN void lnt_m16_load(LntM16 &M, int tid) {
    const int lane = tid & 63;
#pragma unroll
    for (int i = 0; i < LNT_M16_TILES; i++)
        M.t[i] = *reinterpret_cast<const lnt_v4i *>(&lnt_m16_tab.b[(i * 64 + lane) * 16]);
#pragma unroll
    for (int i = 0; i < 8; i++) M.o[i / 4][i % 4] = lnt_m16_offset(i);
    M.dc = lane < 16 ? LNT_M16_DC : 0;
    // opaque, so that a product by them stays one v_mad (with its sum)
    M.k16 = 65536;
    M.km1 = -1;
    asm volatile("" : "+s"(M.k16), "+s"(M.km1));
    asm volatile("" : "+v"(M.o[0]), "+v"(M.o[1]));
}
// The four words of this lane's DFT, in place (every lane of the wave takes part).
LNT_KFN void lnt_m16_dft(const LntM16 &M, u64 (&x)[4]) {
    lnt_v4i b[2];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            b[s][2 * i] = (int)((u32)x[2 * s + i] ^ 0x80808080u);
            b[s][2 * i + 1] = (int)((u32)(x[2 * s + i] >> 32) ^ 0x80808080u);
        }
    bool c[4];  // the word carried out of 64 bits
#pragma unroll
    for (int v = 0; v < 4; v++) {
        lnt_v4i d[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            d[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(M.t[2 * v + h], b[0], M.o[h], 0, 0, 0);
            d[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(M.t[v % 2 ? 8 + (v / 2) * 2 + h : 2 * v + h], b[1], d[h], 0, 0,
                                                         0);
        }
        const int l[8] = {d[0][0], d[0][1], d[0][2], d[0][3], d[1][0], d[1][1], d[1][2], d[1][3]};
        u32 lo, t, hi;
        const u32 v0 = v == 0 ? lnt_limbs<true>(l, M.dc, M.k16, M.km1, lo, t)
                              : lnt_limbs<false>(l, 0, M.k16, M.km1, lo, t);
        c[v] = __builtin_add_overflow(v0, t, &hi);
        x[v] = ((u64)hi << 32) | lo;
    }
    // 2^64 = EPS for the words that carried: one rarely taken branch for the four
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(c[0] | c[1] | c[2] | c[3]) != 0, 0)) {
#pragma unroll
        for (int v = 0; v < 4; v++) x[v] += c[v] ? GL_EPS : 0;
    }
}

static __device__ const LntM8Table lnt_m8_tab = lnt_m8_make();
struct LntM8 {
    lnt_v4i t[LNT_M8_TILES];
    u64 dc;
};
LNT_KFN void lnt_m8_load(LntM8 &M, const LntM16 &, int tid) {
    const int lane = tid & 63;
#pragma unroll
    for (int i = 0; i < LNT_M8_TILES; i++)
        M.t[i] = *reinterpret_cast<const lnt_v4i *>(&lnt_m8_tab.b[(i * 64 + lane) * 16]);
    M.dc = lane < 16 ? LNT_M8_DC : 0;
}
// The two words of this lane's 8-point DFT, in place; the offsets and constants are M16's.
LNT_KFN void lnt_m8_dft(const LntM8 &M, const LntM16 &M16, u64 (&x)[2]) {
    lnt_v4i b;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        b[2 * i] = (int)((u32)x[i] ^ 0x80808080u);
        b[2 * i + 1] = (int)((u32)(x[i] >> 32) ^ 0x80808080u);
    }
    bool c[2];
#pragma unroll
    for (int v = 0; v < 2; v++) {
        lnt_v4i d[2];
#pragma unroll
        for (int h = 0; h < 2; h++) d[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(M.t[2 * v + h], b, M16.o[h], 0, 0, 0);
        const int l[8] = {d[0][0], d[0][1], d[0][2], d[0][3], d[1][0], d[1][1], d[1][2], d[1][3]};
        u32 lo, t, hi;
        const u32 v0 = v == 0 ? lnt_limbs<true>(l, M.dc, M16.k16, M16.km1, lo, t)
                              : lnt_limbs<false>(l, 0, M16.k16, M16.km1, lo, t);
        c[v] = __builtin_add_overflow(v0, t, &hi);
        x[v] = ((u64)hi << 32) | lo;
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(c[0] | c[1]) != 0, 0)) {
#pragma unroll
        for (int v = 0; v < 2; v++) x[v] += c[v] ? GL_EPS : 0;
    }
}
#endif

// The lane's part in its workgroup's DFTs: wave w, lane (q, n), id = 16 w + n.
struct LntLane16 {
    int w, q, n, id;
};
LNT_KFN LntLane16 lnt_lane16(int tid) {
    const int w = LNT_UNIFORM(tid / 64);
    return LntLane16{w, (tid % 64) / 16, tid % 16, 16 * w + tid % 16};
}
// word of output place v of an inverse DFT
GL_HD constexpr int lnt_m16_neg(int q, int v) { return (16 - lnt_m16_word(q, v)) & 15; }
