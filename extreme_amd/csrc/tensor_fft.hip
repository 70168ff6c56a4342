// 2-D FFTs of assembled tensors (FP64).
#include "xtr_pencil.h"

namespace xtr {

// the pencils of an assembled tensor: kernels of this unit's own
struct IoTensor : IoPlain<double> {
};

// the register-resident pencils where the length has them (at 512 points 0.5 ms against 0.63-0.95 ms for the LDS
// kernel's tiles, per 1.6 GB pass)
static int tile_of(int p) { return reg_length(p) ? FFT_TILE_REG : FFT_TILE_DEFAULT; }

void launch_fft2_plain(double2 *data, int n1, int n2, int64_t ncols, const double2 *tw1, const double2 *tw2, hipStream_t s)
{
    // along n2: columns (i1, c), pencil stride ncols
    IoTensor y{{data, 0, (int64_t)n1 * ncols, ncols, (int64_t)n2 * ncols, ncols, n2, n2}};
    // along n1: columns (i2, c) flattened, pencil stride n2*ncols
    IoTensor x{{data, 0, (int64_t)n2 * ncols, (int64_t)n2 * ncols, 0, (int64_t)n2 * ncols, n1, n1}};
    launch_pencil<double, -1, IoTensor, TILES_TWO>(n2, y, (int64_t)n1 * ncols, 1, tw2, s, tile_of(n2));
    launch_pencil<double, -1, IoTensor, TILES_TWO>(n1, x, (int64_t)n2 * ncols, 1, tw1, s, tile_of(n1));
}

// Pencils of a folded Green tensor in its own buffer [Nx+1][Ny+1][gblk]: points p < half hold the values at
// non-negative offsets, and the rest of the 2 half points that the transform sees follow from the mirror
// parities (zero at the offset `half`, +- the value at 2 half - p beyond it), so they are formed on load and
// never stored; of the spectrum only k <= half is kept. A pencil is read whole before it is written, and no
// other workgroup touches its columns, so the transform runs in place.
// The two passes are bound by HBM: they read and write the folded tensor, a quarter of the padded one (at
// 128 x 128 x 32 2.2 GB a pass instead of 8.7 GB), and need neither its 4.4 GB buffer, nor the clear before
// nor the fold after. With the scratch kept on the handle calculate_green_tensor and one chi0 apply there
// take 8.5 ms instead of 15 ms when hipMalloc was quick and 160-190 ms when it was not.
// Parity gives the sign of column position o of a block on the far side of axis 0 (x) or 1 (y).
template <class Parity>
struct IoMirror : IoPlain<double> {
    Parity par;
    int gblk, half, axis;
    // columns and blocks fit 32 bits (a division of 64 takes several times the instructions)
    __device__ int64_t at(int64_t c, int p) const
    {
        const unsigned col = (unsigned)c, per = (unsigned)cpr, row = col / per;
        return row * row_stride + (col - row * per) + p * pstride;
    }
    __device__ double2 load(int, int64_t c, int p) const
    {
        if (c >= ncols || p == half) return make_double2(0, 0);
        const double2 v = buf[at(c, p < half ? p : 2 * half - p)];
        const double s = p < half ? 1.0 : par.sign((int)((unsigned)c % (unsigned)gblk), axis);
        return make_double2(s * v.x, s * v.y);
    }
    __device__ void store(int, int64_t c, int p, double2 v) const
    {
        if (c < ncols && p <= half) buf[at(c, p)] = v;
    }
};

// [xx S | xy S | yy S | zz S | xz A | yz A]: xy is odd in x and y, xz in x, yz in y
struct AtoaParity {
    int S, A;
    __device__ double sign(int o, int axis) const
    {
        const int xy = (int)(o >= S) & (int)(o < 2 * S), xz = (int)(o >= 4 * S) & (int)(o < 4 * S + A),
                  yz = (int)(o >= 4 * S + A);
        return (xy | (axis == 0 ? xz : yz)) ? -1.0 : 1.0;
    }
};

// components of nz values, bit c of odd[axis] set where component c is odd
struct LevelParity {
    int nz;
    unsigned odd[2];
    __device__ double sign(int o, int axis) const { return (axis == 0 ? odd[0] : odd[1]) >> (o / nz) & 1 ? -1.0 : 1.0; }
};

// Half the columns of the default tile, so more workgroups a CU, or register pencils, a pass at nz = 32 (16, 16 and
// 8 from 192 points): 96 points 74 us (default tile 77), 128 135 (165; registers 148), 192 74 (80), 256 153 (174;
// registers 174), 512 196 (283; registers 147); at 64 points 34, 32 and 32.
static int mirror_tile(int p) { return p == 64 || p == 512 ? FFT_TILE_REG : p > 64 ? FFT_TILE_NARROW : FFT_TILE_DEFAULT; }

template <class Parity>
static void fft2_mirror(double2 *folded, int nx, int ny, int64_t gb, const Parity &par, const double2 *tw_x,
                        const double2 *tw_y, hipStream_t s)
{
    using Io = IoMirror<Parity>;
    const int64_t row = (ny + 1) * gb;
    const Io y{{folded, 0, nx * gb, gb, row, gb, 0, 0}, par, (int)gb, ny, 1};
    const Io x{{folded, 0, row, row, 0, row, 0, 0}, par, (int)gb, nx, 0};
    launch_pencil<double, -1, Io, TILES_NARROW>(2 * ny, y, nx * gb, 1, tw_y, s, mirror_tile(2 * ny));
    launch_pencil<double, -1, Io, TILES_NARROW>(2 * nx, x, row, 1, tw_x, s, mirror_tile(2 * nx));
}

void launch_fft2_mirror(double2 *folded, const Geom &g, const double2 *tw_x, const double2 *tw_y, hipStream_t s)
{
    fft2_mirror(folded, g.nx, g.ny, g.gblk(), AtoaParity{(int)g.S(), g.nz * g.nz}, tw_x, tw_y, s);
}

void launch_fft2_mirror_level(double2 *folded, const Geom &g, int ncomp, const unsigned *odd, const double2 *tw_x,
                              const double2 *tw_y, hipStream_t s)
{
    fft2_mirror(folded, g.nx, g.ny, (int64_t)ncomp * g.nz, LevelParity{g.nz, {odd[0], odd[1]}}, tw_x, tw_y, s);
}

// Forward transform of a source [Nx][Ny][C], zero-padded as it is read and only where it is not zero throughout
// (ToOCalculator.PrepareForForwardFft :143-157): along y the rows i < Nx, then along x.
struct IoPadY {
    const double2 *src;
    double2 *dst;
    int nx, ny, C;
    __device__ double2 load(int, int64_t c, int p) const
    {
        if (c >= (int64_t)nx * C || p >= ny) return make_double2(0, 0);
        const unsigned i = (unsigned)c / (unsigned)C, col = (unsigned)c - i * C;
        return src[((int64_t)i * ny + p) * C + col];
    }
    __device__ void store(int, int64_t c, int p, double2 v) const
    {
        if (c >= (int64_t)nx * C) return;
        const unsigned i = (unsigned)c / (unsigned)C, col = (unsigned)c - i * C;
        dst[((int64_t)i * 2 * ny + p) * C + col] = v;
    }
};

void launch_fft2_padded(const double2 *src, double2 *spec, const Geom &g, int C, const double2 *tw_x, const double2 *tw_y,
                        hipStream_t s)
{
    const int64_t nc = 2LL * g.ny * C;
    const IoPadY y{src, spec, g.nx, g.ny, C};
    const IoTensor x{{spec, 0, nc, nc, 0, nc, g.nx, 2 * g.nx}};
    launch_pencil<double, -1, IoPadY, TILES_TWO>(2 * g.ny, y, (int64_t)g.nx * C, 1, tw_y, s, tile_of(2 * g.ny));
    launch_pencil<double, -1, IoTensor, TILES_TWO>(2 * g.nx, x, nc, 1, tw_x, s, tile_of(2 * g.nx));
}

// Backward transform of spec [2Nx][2Ny][C], cropped to [Nx][Ny][C] and scaled (ToOCalculator.cs:38-42, 159-172):
// along x, keeping the rows i < Nx, then those along y.
struct IoCropY {
    const double2 *src;
    double2 *dst;
    int nx, ny, C;
    double scale;
    __device__ double2 load(int, int64_t c, int p) const
    {
        if (c >= (int64_t)nx * C) return make_double2(0, 0);
        const unsigned i = (unsigned)c / (unsigned)C, col = (unsigned)c - i * C;
        return src[((int64_t)i * 2 * ny + p) * C + col];
    }
    __device__ void store(int, int64_t c, int p, double2 v) const
    {
        if (c >= (int64_t)nx * C || p >= ny) return;
        const unsigned i = (unsigned)c / (unsigned)C, col = (unsigned)c - i * C;
        dst[((int64_t)i * ny + p) * C + col] = cscale<double>(v, scale);
    }
};

void launch_fft2_cropped(double2 *spec, double2 *dst, const Geom &g, int C, double scale, const double2 *tw_x,
                         const double2 *tw_y, hipStream_t s)
{
    const int64_t nc = 2LL * g.ny * C;
    const IoTensor x{{spec, 0, nc, nc, 0, nc, 2 * g.nx, g.nx}};
    const IoCropY y{spec, dst, g.nx, g.ny, C, scale};
    launch_pencil<double, +1, IoTensor, TILES_TWO>(2 * g.nx, x, nc, 1, tw_x, s, tile_of(2 * g.nx));
    launch_pencil<double, +1, IoCropY, TILES_TWO>(2 * g.ny, y, (int64_t)g.nx * C, 1, tw_y, s, tile_of(2 * g.ny));
}

}  // namespace xtr
