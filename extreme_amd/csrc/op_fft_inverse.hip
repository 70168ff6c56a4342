// Inverse FFT passes of the operator apply: along x, then along y with the crop, the b scaling and the
// last step fused into the stores.
//
// Spectrum layout (the reference's FFT buffer, Extreme.Cartesian/Fft/FftBuffer.cs:78-96,
// ConvolutionOperator.cs:250-272): buf[(i*2Ny + j)*3Nz + c*Nz + k], one buffer per
// right-hand side; the 1/(4 Nx Ny) of the unnormalised transforms lives in the backward factors b.
#include "xtr_pencil.h"

namespace xtr {

// right-hand sides without a model R of their own use the handle's R
static RhsPtrs with_r(const ApplyArgs &a)
{
    RhsPtrs v = a.v;
    for (int i = 0; i < a.nrhs; ++i)
        if (!v.R[i]) v.R[i] = a.R;
    return v;
}

// complex64 vectors go with the FP32 apply only
static void check_vec32(const ApplyArgs &a)
{
    if (a.vec32 && !a.precision) throw hip_error("complex64 vectors need the FP32 apply");
}

__device__ __forceinline__ double2 widen(double2 v) { return v; }
__device__ __forceinline__ double2 widen(float2 v) { return to_d(v); }

// (ConvolutionOperator.cs:187-231): keeps j < Ny of rows i < Nx, scales by b, and writes
// y = x - b*conv - R*x (A) or y = b*conv + R*x (Chi0), formed in FP64 and stored as complex128 (or
// complex64 when V = float).
template <typename T, typename V>
struct IoInvY {
    RhsPtrs v;                // x, y, and R per right-hand side
    const double *b;
    cplx<T> *buf;
    int64_t M;
    int nx, ny, nz, type;
    __device__ cplx<T> load(int rhs, int64_t c, int p) const
    {
        const unsigned C = 3u * nz;
        if (c >= (int64_t)nx * C) return mk<T>(0, 0);
        const unsigned i = (unsigned)c / C, col = (unsigned)c - i * C;
        return buf[rhs * M + ((int64_t)i * 2 * ny + p) * C + col];
    }
    __device__ void store(int rhs, int64_t c, int p, cplx<T> val) const
    {
        const unsigned C = 3u * nz;
        if (c >= (int64_t)nx * C || p >= ny) return;
        const unsigned i = (unsigned)c / C, col = (unsigned)c - i * C, k = col % (unsigned)nz;
        const int64_t ij = (int64_t)i * ny + p, t = ij * C + col;
        double2 conv;
        if constexpr (sizeof(T) == 8) conv = cscale<double>(val, b[k]);
        else conv = cscale<double>(to_d(val), b[k]);
        const double2 xv = widen(reinterpret_cast<const cplx<V> *>(v.x[rhs])[t]);
        const double2 rx = cmul<double>(v.R[rhs][ij * nz + k], xv);
        double2 out;
        if (type == 0) out = csub<double>(csub<double>(xv, conv), rx);
        else out = cadd<double>(conv, rx);
        reinterpret_cast<cplx<V> *>(v.y[rhs])[t] = from_d<V>(out);
    }
};

template <typename T>
static void inv_x(const ApplyArgs &a, hipStream_t s)
{
    const int64_t ncols = 2LL * a.g.ny * a.g.C();
    IoPlain<T> io{(cplx<T> *)a.buf, a.g.M(), ncols, ncols, 0, ncols, 2 * a.g.nx, a.g.nx};
    launch_pencil<T, +1>(2 * a.g.nx, io, ncols, a.nrhs, a.tw_x, s, a.fft_tile[2]);
}

template <typename T, typename V>
static void inv_y(const ApplyArgs &a, hipStream_t s)
{
    IoInvY<T, V> io{with_r(a), a.b, (cplx<T> *)a.buf, a.g.M(), a.g.nx, a.g.ny, a.g.nz, a.type};
    launch_pencil<T, +1>(2 * a.g.ny, io, (int64_t)a.g.nx * a.g.C(), a.nrhs, a.tw_y, s, a.fft_tile[3]);
}

void launch_inv_x(const ApplyArgs &a, hipStream_t s) { a.precision ? inv_x<float>(a, s) : inv_x<double>(a, s); }
void launch_inv_y(const ApplyArgs &a, hipStream_t s)
{
    check_vec32(a);
    if (a.vec32) inv_y<float, float>(a, s);
    else if (a.precision) inv_y<float, double>(a, s);
    else inv_y<double, double>(a, s);
}

}  // namespace xtr
