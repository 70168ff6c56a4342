// Column tiles of the FFT passes, by pencil length and element bytes: the one table that the kernels' instances,
// the tile options and the handle's choice between them go by. Plain C++.
#pragma once

#include <cstdint>

namespace xtr {

enum {
    FFT_TILE_DEFAULT = 0,
    FFT_TILE_NARROW = 1,
    FFT_TILE_WIDE = 2,
    FFT_TILE_NARROW_T512 = 3,
    FFT_TILE_REG = 4,        // register-resident stages (lengths 64..512), the default column count
    FFT_TILE_REG_ALT = 5,    // the same with twice the columns (half where that exceeds 64 KB of LDS)
};

// Columns of a tile of pencils of p elements of e bytes. The default tile has 16 while p x 16 stays within 32 KB,
// else 8. For lengths from 64 the narrow tiles have half as many (more workgroups per CU), and the wide one (within
// 128 KB) and the alternative register tile (within 64 KB, else half) twice as many.
constexpr int fft_tile_cols(int p, int e, int tile)
{
    const int d = p * 16 * e <= 32768 ? 16 : 8;
    if (p < 64) return d;
    if (tile == FFT_TILE_WIDE) return p * 2 * d * e <= 131072 ? 2 * d : d;
    if (tile == FFT_TILE_NARROW || tile == FFT_TILE_NARROW_T512) return d / 2;
    if (tile == FFT_TILE_REG_ALT) return p * 2 * d * e <= 65536 ? 2 * d : d / 2;
    return d;
}

// What a tile's measured time is multiplied by before tiles are compared. Rows shorter than a cache line of 128
// bytes cost more on a first pass over large spectra, which are not in the Infinity Cache then as they are in a
// repeated one: at 128 x 128 x 32 (two right-hand sides, 201 MB) the 4-column tile of the forward x pass takes
// 50 us repeated and 80 on new buffers, the 16-column one 52 both times. There they have to gain a tenth; at
// 64 x 64 x 32 in complex64 (25 MB) an apply takes 95 us with them and 98 without, and a first pass 175 us either
// way. The line is drawn by one right-hand side's spectrum, half of the usual two: a choice is kept for every number
// of them, so it must not hang on how many the first apply had.
constexpr double fft_tile_weight(int64_t spectrum_bytes, int p, int e, int tile)
{
    return fft_tile_cols(p, e, tile) * e < 128 && spectrum_bytes > (int64_t)32 << 20 ? 1.1 : 1.0;
}

}  // namespace xtr
