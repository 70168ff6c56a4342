// Forward FFT passes of the operator apply: along y with the R and f scaling fused into the loads, then
// along x; and the tile options the operator handle measures.
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

// First forward pass along y, fused with ApplyOperatorR and PrepareForForwardFft
// (ConvolutionOperator.cs:233-272): reads x (complex128, or complex64 when V = float) and R, writes
// f * R * x into rows i < Nx of the padded buffer; columns c = i*3Nz + col; points j < Ny are data,
// j >= Ny are the padding. R * x is formed in FP64.
template <typename T, typename V>
struct IoFwdY {
    RhsPtrs v;                // x, and R per right-hand side
    const double *f;
    cplx<T> *buf;
    int64_t M;
    int nx, ny, nz;
    __device__ cplx<T> load(int rhs, int64_t c, int p) const
    {
        const unsigned C = 3u * nz;
        if (c >= (int64_t)nx * C || p >= ny) return mk<T>(0, 0);
        const unsigned i = (unsigned)c / C, col = (unsigned)c - i * C, k = col % (unsigned)nz;
        const int64_t ij = (int64_t)i * ny + p;
        const cplx<V> *x = reinterpret_cast<const cplx<V> *>(v.x[rhs]);
        double2 rx = cmul<double>(v.R[rhs][ij * nz + k], widen(x[ij * C + col]));
        return from_d<T>(cscale<double>(rx, f[k]));
    }
    __device__ void store(int rhs, int64_t c, int p, cplx<T> val) const
    {
        const unsigned C = 3u * nz;
        if (c >= (int64_t)nx * C) return;
        const unsigned i = (unsigned)c / C, col = (unsigned)c - i * C;
        buf[rhs * M + ((int64_t)i * 2 * ny + p) * C + col] = val;
    }
};

int fft_tile_options(int p, int precision, int *tiles)
{
    int n = 0;
    tiles[n++] = FFT_TILE_DEFAULT;
    if (p < 64) return n;
    const int e = precision ? 8 : 16;
    tiles[n++] = FFT_TILE_NARROW;
    if (fft_tile_cols(p, e, FFT_TILE_WIDE) > fft_tile_cols(p, e, FFT_TILE_DEFAULT)) tiles[n++] = FFT_TILE_WIDE;
    if (p >= 128) tiles[n++] = FFT_TILE_NARROW_T512;
    if (p == 64 || p == 128 || p == 256 || p == 512) {
        tiles[n++] = FFT_TILE_REG;
        tiles[n++] = FFT_TILE_REG_ALT;
    }
    return n;
}

// even lengths 2^a m, m in {1, 3, 5, 15, 25, 75}, up to 512 (Nx, Ny <= 256)
bool fft_length_supported(int p)
{
    switch (p) {
    case 4:
    case 6:
    case 8:
    case 10:
    case 12:
    case 16:
    case 20:
    case 24:
    case 30:
    case 32:
    case 40:
    case 48:
    case 50:
    case 60:
    case 64:
    case 80:
    case 96:
    case 100:
    case 120:
    case 128:
    case 150:
    case 160:
    case 192:
    case 200:
    case 240:
    case 256:
    case 300:
    case 320:
    case 384:
    case 400:
    case 480:
    case 512:
        return true;
    default:
        return false;
    }
}

template <typename T, typename V>
static void fwd_y(const ApplyArgs &a, hipStream_t s)
{
    IoFwdY<T, V> io{with_r(a), a.f, (cplx<T> *)a.buf, a.g.M(), a.g.nx, a.g.ny, a.g.nz};
    launch_pencil<T, -1>(2 * a.g.ny, io, (int64_t)a.g.nx * a.g.C(), a.nrhs, a.tw_y, s, a.fft_tile[0]);
}

template <typename T>
static void fwd_x(const ApplyArgs &a, hipStream_t s)
{
    const int64_t ncols = 2LL * a.g.ny * a.g.C();
    IoPlain<T> io{(cplx<T> *)a.buf, a.g.M(), ncols, ncols, 0, ncols, a.g.nx, 2 * a.g.nx};
    launch_pencil<T, -1>(2 * a.g.nx, io, ncols, a.nrhs, a.tw_x, s, a.fft_tile[1]);
}

void launch_fwd_y(const ApplyArgs &a, hipStream_t s)
{
    check_vec32(a);
    if (a.vec32) fwd_y<float, float>(a, s);
    else if (a.precision) fwd_y<float, double>(a, s);
    else fwd_y<double, double>(a, s);
}
void launch_fwd_x(const ApplyArgs &a, hipStream_t s) { a.precision ? fwd_x<float>(a, s) : fwd_x<double>(a, s); }

}  // namespace xtr
