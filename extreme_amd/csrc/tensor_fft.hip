// 2-D FFTs of assembled tensors (FP64).
#include "xtr_pencil.h"

namespace xtr {

// the pencils of an assembled tensor: kernels of this unit's own
struct IoTensor : IoPlain<double> {
};

void launch_fft2_plain(double2 *data, int n1, int n2, int64_t ncols, const double2 *tw1, const double2 *tw2,
                       int sign, hipStream_t s)
{
    // along n2: columns (i1, c), pencil stride ncols
    IoTensor y{{data, 0, (int64_t)n1 * ncols, ncols, (int64_t)n2 * ncols, ncols, n2, n2}};
    // along n1: columns (i2, c) flattened, pencil stride n2*ncols
    IoTensor x{{data, 0, (int64_t)n2 * ncols, (int64_t)n2 * ncols, 0, (int64_t)n2 * ncols, n1, n1}};
    // the register-resident pencils where the length has them (at 512 points 0.5 ms against
    // 0.63-0.95 ms for the LDS kernel's tiles, per 1.6 GB pass)
    const int t2 = reg_length(n2) ? FFT_TILE_REG : FFT_TILE_DEFAULT, t1 = reg_length(n1) ? FFT_TILE_REG : FFT_TILE_DEFAULT;
    if (sign < 0) {
        launch_pencil<double, -1, IoTensor, false>(n2, y, (int64_t)n1 * ncols, 1, tw2, s, t2);
        launch_pencil<double, -1, IoTensor, false>(n1, x, (int64_t)n2 * ncols, 1, tw1, s, t1);
    } else {
        launch_pencil<double, +1, IoTensor, false>(n2, y, (int64_t)n1 * ncols, 1, tw2, s, t2);
        launch_pencil<double, +1, IoTensor, false>(n1, x, (int64_t)n2 * ncols, 1, tw1, s, t1);
    }
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
struct IoMirror : IoPlain<double> {
    int gblk, S, A;
    int half, axis;           // axis 0: x, 1: y
    // columns and blocks fit 32 bits (a division of 64 takes several times the instructions)
    __device__ int64_t at(int64_t c, int p) const
    {
        const unsigned col = (unsigned)c, per = (unsigned)cpr, row = col / per;
        return row * row_stride + (col - row * per) + p * pstride;
    }
    // xy is odd in x and y, xz in x, yz in y
    __device__ double sign(int64_t c) const
    {
        const int o = (int)((unsigned)c % (unsigned)gblk);
        const int xy = (int)(o >= S) & (int)(o < 2 * S), xz = (int)(o >= 4 * S) & (int)(o < 4 * S + A),
                  yz = (int)(o >= 4 * S + A);
        return (xy | (axis == 0 ? xz : yz)) ? -1.0 : 1.0;
    }
    __device__ double2 load(int, int64_t c, int p) const
    {
        if (c >= ncols || p == half) return make_double2(0, 0);
        const double2 v = buf[at(c, p < half ? p : 2 * half - p)];
        const double s = p < half ? 1.0 : sign(c);
        return make_double2(s * v.x, s * v.y);
    }
    __device__ void store(int, int64_t c, int p, double2 v) const
    {
        if (c < ncols && p <= half) buf[at(c, p)] = v;
    }
};

void launch_fft2_mirror(double2 *folded, const Geom &g, const double2 *tw_x, const double2 *tw_y, hipStream_t s)
{
    const int64_t gb = g.gblk(), row = (g.ny + 1) * gb;
    const int S = (int)g.S(), A = g.nz * g.nz;
    const IoMirror y{{folded, 0, g.nx * gb, gb, row, gb, 0, 0}, (int)gb, S, A, g.ny, 1};
    const IoMirror x{{folded, 0, row, row, 0, row, 0, 0}, (int)gb, S, A, g.nx, 0};
    const int ty = reg_length(2 * g.ny) ? FFT_TILE_REG : FFT_TILE_DEFAULT;
    const int tx = reg_length(2 * g.nx) ? FFT_TILE_REG : FFT_TILE_DEFAULT;
    launch_pencil<double, -1, IoMirror, false>(2 * g.ny, y, g.nx * gb, 1, tw_y, s, ty);
    launch_pencil<double, -1, IoMirror, false>(2 * g.nx, x, row, 1, tw_x, s, tx);
}

}  // namespace xtr
