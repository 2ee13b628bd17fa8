// How the passes are cut into blocks: host arithmetic on sizes and on what a
// compute unit holds, free of the GPU runtime.
#pragma once

#include <algorithm>
#include <cstddef>

namespace blgpu {

// ---- x transform of N = N1 N2 points (k_dct_fwd_m, k_dct_inv_m) ----

// row stride of the complex intermediate: odd, so that 16 lanes reading one
// entry of 16 rows use different banks
constexpr int dct_ld(int N2) { return N2 | 1; }
// LDS elements of the line area (even: the complex area behind it is aligned)
constexpr int dct_lines(int LB, int N) { return (LB * N + 1) / 2 * 2; }
// LDS bytes of one line and its spectrum, elements of es bytes
constexpr size_t dct_line_bytes(int N, int N1, size_t es) {
    return es * (N + 1 + 2 * (size_t)(N1 / 2 + 1) * dct_ld(N / N1));
}
// What the kernels hold of N = N1 N2 points: an entry of a line's spectrum and a row
// k1 <= N1/2 in the range of small_div, one line of either direction in 160 KB.
constexpr bool dct_holds(int N, int N1, size_t es) {
    return N1 / 2 + 1 <= 128 && (N1 / 2 + 1) * (N / N1) < 16384 && 2 * dct_line_bytes(N, N1, es) <= 163840;
}
// FP64 lengths that bl_create takes: both factors up to 32, or 16-byte values of two
// lines, their spectra and both factors' roots in 64 KB (primes up to 811).  That is
// narrower than dct_holds, and kept: which lengths are refused is part of the interface.
constexpr bool dct_takes_fp64(int N, int N1) {
    const int K1 = N1 / 2 + 1, N2 = N / N1;
    return (N1 <= 31 && N2 <= 32) || 16 * (2 * (size_t)N + 2 * (size_t)K1 * N2 + N1 + N2) <= 65536;
}
// FP32 lengths that go through these kernels, the others through the dense
// split-BF16 product.  A long factor is a matrix product of its own here: at 1 x 251
// points, 25542 lines, both directions take 131 us against 101 for the dense product
// with its divergence pass, but in FP32 factors, not in 2^-18; longer ones would be
// further behind.
constexpr bool dct_takes_mixed(int N, int N1) { return N / N1 <= 256 && dct_holds(N, N1, 4); }
// both factors within one row tile and two column tiles: two lines in two waves
constexpr bool dct_small(int N, int N1) { return N1 <= 31 && N / N1 <= 31; }

struct DctPlan {
    int lines, waves;  // per block
};

// Products of step C in lb lines: 16 columns of (line, k1) by 16 rows.
constexpr int dct_products(int N, int N1, int lb) { return (lb * (N1 / 2 + 1) + 15) / 16 * ((N / N1 / 2 + 16) / 16); }

// Past the small shapes a block has four waves, or eight for more than four
// products, which would otherwise go through the same waves in two or more
// rounds of dependent loads (2 x 251 points: four waves 288 us, eight 228), and
// its lines fill 16 columns: rounded down or up, whichever takes fewer waves'
// time per line (K1 = 3: five lines in one column tile, not six in two, the second
// with two columns; 4 x 181 points FP32 322 -> 266 us for both directions, but with two
// row tiles the second column tile costs no further round, and six lines stay:
// 4 x 53 FP64 40 us against 49).  80 KB of LDS (two blocks per CU) bound the lines.
// With many lines and step A on the matrix cores, as many more as four products
// hold while four blocks fit a CU: one column tile is two products of two row
// tiles, and two of the four waves idled (both directions, 25542 lines: 16 x 32 points
// FP64 322 -> 275 us, FP32 191 -> 161; 14 x 41 358 -> 287 and 222 -> 170).
// Fewer lines where the blocks would not reach every compute unit (127 points,
// 1536 lines: 16 lines 14.9 and 11.8 us, 8 lines 12.6 and 10.5), and eight waves
// while all of them reside at once, 16 per CU in FP64 and 24 in FP32 by their
// registers (129 points, 3774 lines: 19 and 17 us; but 16 x 32 FP64, 1170 lines, 585
// blocks: 31 us with four waves, 42 with eight in two rounds).
constexpr int kDctShort = 4;  // most rows k1 <= N1/2 of a step A on the vector units
inline DctPlan dct_plan(int N, int N1, size_t es, int nlines, int n_cu) {
    if (dct_small(N, N1)) return {2, 2};
    const int K1 = N1 / 2 + 1;
    const size_t line = dct_line_bytes(N, N1, es);
    auto waves = [&](int lb) { return dct_products(N, N1, lb) > 4 ? 8 : 4; };
    auto slots = [&](int lb) { return (dct_products(N, N1, lb) + waves(lb) - 1) / waves(lb) * waves(lb); };
    const int up = std::max(2, (15 + K1) / K1), down = std::max(2, 16 / K1);
    int lb = slots(down) * up < slots(up) * down ? down : up;
    lb = std::max(1, std::min(lb, (int)(81920 / line)));
    if (K1 > kDctShort)
        while (dct_products(N, N1, lb + 1) <= 4 && (lb + 1) * line <= 40960 && nlines / (lb + 1) >= 8 * n_cu) ++lb;
    if ((nlines + lb - 1) / lb < n_cu) lb = (lb + 1) / 2;
    return {lb, (nlines + lb - 1) / lb <= (es == 4 ? 3 : 2) * n_cu ? 8 : waves(lb)};
}

// ---- marches in z ----

// The chunk of nk planes with the fewest plane steps in sequence, rounds of the
// resident blocks (`slots`) times (chunk + 2), since a block also loads the planes
// before and behind its chunk; blocks: of the launch, `tiles` columns of chunks.
// Of chunks with equally many, the longest, or the shortest while the launch has
// no more than `most` blocks.
struct ZChunk {
    int planes;
    long long blocks;
};
inline ZChunk fewest_plane_steps(int nk, int tiles, int slots, long long most = 0) {
    ZChunk best{nk, 0};
    long long cost = -1;
    for (int chunk = nk; chunk >= 1; --chunk) {
        const long long blocks = (long long)tiles * ((nk + chunk - 1) / chunk);
        const long long c = (blocks + slots - 1) / slots * (chunk + 2);
        if (cost < 0 || c < cost || (c == cost && blocks <= most)) {
            cost = c;
            best = {chunk, blocks};
        }
    }
    return best;
}

// Tiles of the RK march (k_rk_march): 64 x 8 cells in FP64, 64 x 12 in FP32.
template <class T>
struct MarchTile {
    static constexpr int TX = 64;                          // tile width (x)
    static constexpr int RPT = sizeof(T) == 4 ? 3 : 2;    // rows per thread
    static constexpr int TY = (256 / TX) * RPT, HX = TX + 2, HY = TY + 2, Plane = HX * HY;
};
template <class T>
constexpr int march_tiles(int nxg, int nyg) {
    return (nxg - 1 + MarchTile<T>::TX - 1) / MarchTile<T>::TX * ((nyg - 2 + MarchTile<T>::TY - 1) / MarchTile<T>::TY);
}
// LDS bytes of a block: two planes of U and V, three of W, with an eddy
// viscosity three of nu_t, and the tile's metrics
template <class T>
constexpr size_t march_lds(bool les) {
    return sizeof(T) * ((les ? 10 : 7) * MarchTile<T>::Plane + 4 * MarchTile<T>::TX + 8 * MarchTile<T>::TY);
}
// blocks that reside on a compute unit: three by the registers of the stages
// (128 to 168 of them), two with an eddy viscosity in FP64 by its 54 KB of LDS
template <class T>
constexpr int march_resident(bool les) {
    return std::min<int>(3, 163840 / march_lds<T>(les));
}

// z-chunk length of the RK march over nz planes.
// While the launch is of up to six blocks per compute unit, the chip is not
// filled by bytes but by plane steps in sequence, and the chunk is the one with
// the fewest of them.  RK stage, chunks of 16 or 24 planes -> this rule:
// 192x32x8 21 -> 9 us, 129x49x34 LES FP32 54 -> 12, 257x97x64 LES FP32 76 -> 34,
// 131x75x53 36 -> 20, 262x66x230 FP32 103 -> 52, 513x97x130 139 -> 109.  FP64 LES,
// of which two blocks reside, with three counted -> with two: 278x266x34 74 -> 58
// us, 257x97x64 54 -> 42, 622x259x49 193 -> 158; short chunks of equal cost fill
// the last round (390x244x57 FP64 LES: 28 planes 123 us, 8 planes 112).
// Larger launches are bound by HBM.  The tiles run in XCD-contiguous order
// with the z chunk slowest, so with a multiple of 8 chunks each XCD holds
// whole chunk layers and a tile's x and y neighbours (whose halos it shares)
// sit in the same L2; the count is the multiple of 8 that gives chunks of
// about 24 planes.  At 814x257x193 (8 chunks of 24 planes) this measured 1 %
// (FP64) and 2.4 % (FP32) faster than 12 chunks of 16, and 3 % and 9 % faster
// than the 28 planes that the first rule would take.  Below 128 planes, chunks
// of up to 16 planes (the two re-read halo planes stay a small share).
inline int march_chunk(int nz, int tiles, int n_cu, int resident) {
    const long long few = 6LL * n_cu;
    const ZChunk c = fewest_plane_steps(nz, tiles, resident * n_cu, few);
    if (c.blocks <= few) return c.planes;
    const int nch = nz >= 8 * 16 ? 8 * std::max(1, (nz + 8 * 12) / (8 * 24))  // multiple of 8 nearest nz / 24
                                 : (nz + 15) / 16;
    return std::max(1, (nz + nch - 1) / nch);
}

// Blocks of the dynamic model's marching passes that reside on a compute unit:
// k_dsm_vfilter has four waves of 122 registers in FP32 fields and of 170 in FP64
// (two blocks; with four counted 130x100x32 took 23 us, now 19, 400x128x96 115 and
// 121; 42 sizes 4 % less on average, the chunk among equal ones the shortest up to
// six blocks); k_dsm_stress seven waves of up to 128 and 72 to 76 KB of LDS: at
// 257x97x64 (144 tiles, 512 slots) it takes 9 planes, two full rounds, against 8
// planes in 2.25 rounds.
template <class T>
constexpr int vfilter_resident() {
    return sizeof(T) == 4 ? 4 : 2;
}
constexpr int kStressResident = 2;

// ---- partitioned Thomas solve (k_thomas_seg) ----

// rows per segment (held in registers) and segments per system, so systems up to
// NM = 256 rows take that kernel
constexpr int kThSeg = 32, kThMaxP = 8;
// LDS bytes of a block, whatever its segments: the interface values of up to eight,
// the coefficients, and the rows of the (0,0) system for the block that solves it
constexpr size_t kThomasLds = sizeof(double) * (6 * kThMaxP * 64 + (3 + 5) * kThSeg * kThMaxP);
// Blocks of P waves that reside on a compute unit: eight waves by their registers
// (more than 128), four blocks by their LDS.  A launch of more leaves blocks that
// start with few tiles left: one segment, eight -> four blocks, 600x16x120 FP64 20.2
// -> 17.8 us, 300x25x290 FP32 19.3 -> 17.5.
constexpr int thomas_resident(int P) { return std::min<int>(kThMaxP / P, 163840 / kThomasLds); }

}  // namespace blgpu
