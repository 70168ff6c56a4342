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

}  // namespace xtr
