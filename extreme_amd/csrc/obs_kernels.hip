// Observation-level kernels (FP64): the anomalous current jQ from the solved chi, and the
// anomaly-to-observation convolution of ToOCalculator.CalculateAnomalyField
// (Extreme.Cartesian/Forward/ToObs/ToOCalculator.cs:21-125) on the device.
#include "xtr_common.h"
#include "xtr_kernels.h"

namespace xtr {

namespace {

// jQ = E_s (zeta - zeta0) + j_s with E_s = (2 sqrt(Re zeta0) chi - j_s) / (zeta + conj zeta0)
// (ForwardSolver.CalculateEScatteredFrom / CalculateJqFrom, ForwardSolver.cs:319-436), written as
// jQ = R (2 f chi - j_s) + j_s with the A-type R = (zeta - zeta0)/(zeta + conj zeta0), f = sqrt(Re zeta0).
__global__ void jq_kernel(const double2 *chi, const double2 *js, const double2 *R, const double *f, int nz,
                          int64_t n, double2 *jq)
{
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        const int k = (int)(e % nz);
        const int64_t cell = e / (3LL * nz);
        const double2 c = chi[e], s = js[e], r = R[cell * nz + k];
        const double2 t = make_double2(2 * f[k] * c.x - s.x, 2 * f[k] * c.y - s.y);
        jq[e] = cadd<double>(cmul<double>(r, t), s);
    }
}

// One 64-lane wave per tensor block, in 64 / WIDTH groups of lanes that share the block's images between them;
// lane of a group = transmitter layer: the nine (electric) or eight (magnetic) Zgemv of
// ApplyGreenTensorAlongZForE/H (:47-125) for each wavenumber the block serves, reduced over the layers.
// G: [blocks][ncomp][nz] (electric xx yy zz xy xz yz zx zy; magnetic xx xy yx xz yz zx zy), all L wavenumbers or
// folded, kx <= Nx, ky <= Ny: then a block is read once for its up to 4 images, with the signs of the odd
// components. u: [L][3nz]. Bound by HBM: 128 x 128 x 32, folded, 32 (electric) and 29 us for 168 MB (57 with one
// group of 64 lanes, half of them idle and 4 images in each lane's registers; 61 from the full tensor).
template <int ELECTRIC, int WIDTH>
__global__ __launch_bounds__(256) void atoo_contract_kernel(const double2 *__restrict__ G, const double2 *__restrict__ u,
                                                            int64_t blocks, int nx, int ny, int nz, int folded,
                                                            double2 *out)
{
    constexpr int NC = ELECTRIC ? 8 : 7;
    constexpr int GROUPS = 64 / WIDTH, PER = 4 / GROUPS;
    const int lane = threadIdx.x & (WIDTH - 1), grp = (threadIdx.x & 63) / WIDTH;
    const int64_t b = (int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
    if (b >= blocks) return;
    const FoldImages im = fold_images(folded ? b : 0, nx, ny);
    const int images = folded ? im.n : 1;
    double2 o[PER][3];
#pragma unroll
    for (int m = 0; m < PER; ++m) o[m][0] = o[m][1] = o[m][2] = make_double2(0, 0);
    for (int k = lane; k < nz; k += WIDTH) {
        double2 g[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) g[c] = G[(b * NC + c) * nz + k];
#pragma unroll
        for (int m = 0; m < PER; ++m) {
            const int q = m * GROUPS + grp;
            if (q >= images) break;
            const int64_t l = folded ? im.l(q) : b;
            // signs of the components odd in x, in y, and in both, in this image
            const double fx = folded && im.mx(q) ? -1.0 : 1.0, fy = folded && im.my(q) ? -1.0 : 1.0, fxy = fx * fy;
            const double2 sx = u[l * 3 * nz + k], sy = u[l * 3 * nz + nz + k], sz = u[l * 3 * nz + 2 * nz + k];
            if constexpr (ELECTRIC) {
                const double2 xx = g[0], yy = g[1], zz = g[2], xy = cscale<double>(g[3], fxy), xz = cscale<double>(g[4], fx),
                              yz = cscale<double>(g[5], fy), zx = cscale<double>(g[6], fx), zy = cscale<double>(g[7], fy);
                o[m][0] = cfma<double>(cfma<double>(cfma<double>(o[m][0], xx, sx), xy, sy), xz, sz);
                o[m][1] = cfma<double>(cfma<double>(cfma<double>(o[m][1], xy, sx), yy, sy), yz, sz);
                o[m][2] = cfma<double>(cfma<double>(cfma<double>(o[m][2], zx, sx), zy, sy), zz, sz);
            } else {
                const double2 xx = cscale<double>(g[0], fxy), xy = g[1], yx = g[2], xz = cscale<double>(g[3], fy),
                              yz = cscale<double>(g[4], fx), zx = cscale<double>(g[5], fy), zy = cscale<double>(g[6], fx);
                o[m][0] = cfms<double>(cfms<double>(cfms<double>(o[m][0], xx, sx), xy, sy), xz, sz);   // -(xx sx + xy sy + xz sz)
                o[m][1] = cfma<double>(cfma<double>(cfma<double>(o[m][1], yx, sx), xx, sy), yz, sz);
                o[m][2] = cfma<double>(cfms<double>(o[m][2], zx, sx), zy, sy);                       // -zx sx + zy sy
            }
        }
    }
#pragma unroll
    for (int m = 0; m < PER; ++m) {
        const int q = m * GROUPS + grp;
#pragma unroll
        for (int c = 0; c < 3; ++c)
            for (int off = WIDTH / 2; off > 0; off >>= 1) {
                o[m][c].x += __shfl_xor(o[m][c].x, off, 64);
                o[m][c].y += __shfl_xor(o[m][c].y, off, 64);
            }
        if (lane == 0 && q < images) {
            const int64_t l = folded ? im.l(q) : b;
            out[l * 3 + 0] = o[m][0];
            out[l * 3 + 1] = o[m][1];
            out[l * 3 + 2] = o[m][2];
        }
    }
}

}  // namespace

void launch_jq(const double2 *chi, const double2 *js, const double2 *R, const double *f, const Geom &g, double2 *jq,
               hipStream_t s)
{
    hipLaunchKernelGGL(jq_kernel, dim3(2048), dim3(256), 0, s, chi, js, R, f, g.nz, g.n(), jq);
    XTR_LAUNCH_CHECK("jq_kernel");
}

void launch_level_field(const double2 *G, int electric, int folded, const double2 *jq, const Geom &g, double2 *spec,
                        double2 *small, const double2 *tw_x, const double2 *tw_y, double2 *field, hipStream_t s)
{
    launch_fft2_padded(jq, spec, g, 3 * g.nz, tw_x, tw_y, s);
    const int64_t blocks = folded ? g.Lq() : g.L();
    const dim3 grid((unsigned)ceil_div(blocks, 4));
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, G, spec, blocks, g.nx, g.ny, g.nz, folded, small);
    };
    // lanes past nz idle: groups of 16 or 32 lanes where the layers fit them
    if (!folded || g.nz > 32) electric ? run(atoo_contract_kernel<1, 64>) : run(atoo_contract_kernel<0, 64>);
    else if (g.nz > 16) electric ? run(atoo_contract_kernel<1, 32>) : run(atoo_contract_kernel<0, 32>);
    else electric ? run(atoo_contract_kernel<1, 16>) : run(atoo_contract_kernel<0, 16>);
    XTR_LAUNCH_CHECK("atoo_contract_kernel");
    launch_fft2_cropped(small, field, g, 3, 1.0 / ((double)g.nx * (double)g.ny * 4), tw_x, tw_y, s);
}

}  // namespace xtr
