// Contraction of the operator apply for a folded Green tensor of few layers: a wave per block, no LDS.
#include "xtr_common.h"
#include "xtr_kernels.h"
#include "xtr_mfma.h"

namespace xtr {
namespace {

template <typename T>
struct DirectArgs {
    const cplx<T> *G;
    cplx<T> *buf;
    int64_t M;
    int Lq, nrhs, nx, ny;
};

__device__ __forceinline__ int xor8(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true); }
__device__ __forceinline__ float xor8(float v) { return __int_as_float(xor8(__float_as_int(v))); }
__device__ __forceinline__ double xor8(double v)
{
    return __hiloint2double(xor8(__double2hiint(v)), xor8(__double2loint(v)));
}

// ApplyGreenTensorAlongZ (ConvolutionOperator.cs:274-327) over a folded tensor, as the block kernel
// (contract_block.h) does it: Y = G U of the block's 4 images x the right-hand sides, B = [Re U | Im U] 8 complex
// columns a tile, D1 = Re G . B, D2 = Im G . B, on 16x16x4 MFMAs. Here a wave takes a whole block: the rows x, y, z
// follow each other in its 16-row tiles (the block kernel pads each to 16), and its A and B values come straight
// from memory into the lanes that need them, all loads of the block in flight at once.
//
// Bound by HBM on large grids (75 x 75 x 4, 8 right-hand sides: 76 MB in 22 us where the block kernel takes 35, and
// 120 x 120 x 3 in 37 instead of 80; 64 x 64 x 10, 2: 1.24 times as fast), by the latency of one block on small ones.
template <typename T, int NZ, int CT>
__global__ __launch_bounds__(256) void contract_direct_kernel(DirectArgs<T> p)
{
    using acc_t = typename MfmaAcc<T>::type;
    constexpr int C = 3 * NZ, S = NZ * (NZ + 1) / 2, A = NZ * NZ, GB = 4 * S + 2 * A;
    constexpr int TILES = (C + 15) / 16, KS = (C + 3) / 4;
    constexpr int MASK = NZ % 16 == 0 ? 15 : (NZ % 8 == 0 ? 7 : 0);      // asym_swizzle_mask
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int b = blockIdx.x * 4 + wave;
    if (b >= p.Lq) return;                                               // waves meet at no barrier
    const int qx = b / (p.ny + 1), qy = b - qx * (p.ny + 1);
    const int kl = lane >> 4, part = (lane >> 3) & 1, q = lane & 7;
    // G[row][k] of this lane's row and k = 4 s + kl; rows and k past the end repeat the last ones
    const cplx<T> *g = p.G + (int64_t)b * GB;
    cplx<T> av[TILES][KS];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const int row = min(16 * t + (lane & 15), C - 1), ar = row / NZ, i = row - ar * NZ;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int k = min(4 * s + kl, C - 1), ac = k / NZ, c = k - ac * NZ;
            const int hi = max(i, c), lo = min(i, c), sym = lo + hi * (hi + 1) / 2;
            const bool zr = ar == 2, zc = ac == 2;
            // xx xy / xy yy / zz packed symmetric; xz, yz rows over receivers; -xz^T, -yz^T
            const int o = zr == zc ? (zr ? 3 : ar + ac) * S + sym
                                   : 4 * S + (zr ? ac * A + c * NZ + (i ^ (c & MASK)) : ar * A + i * NZ + (c ^ (i & MASK)));
            cplx<T> v = g[o];
            if (zr && !zc) v = mk<T>(-v.x, -v.y);
            av[t][s] = v;
        }
    }
    // images: bit 0 mirrors x, bit 1 mirrors y, where a mirror image exists; else the image stands for the other
    const int img = q & 3;
    const bool mx = (img & 1) && qx > 0 && qx < p.nx, my = (img >> 1) && qy > 0 && qy < p.ny;
    const int64_t l = (int64_t)(mx ? 2 * p.nx - qx : qx) * (2 * p.ny) + (my ? 2 * p.ny - qy : qy);
    T *col[CT];
    T bv[CT][KS];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        col[ct] = reinterpret_cast<T *>(p.buf + min(2 * ct + (q >> 2), p.nrhs - 1) * p.M + l * C) + part;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int k = 4 * s + kl;
            T v = col[ct][2 * min(k, C - 1)];
            if ((mx && k < NZ) || (my && k >= NZ && k < 2 * NZ)) v = -v;
            bv[ct][s] = 4 * s + 3 < C || k < C ? v : T(0);
        }
    }
    const T sp = part ? T(1) : T(-1);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        acc_t d1[TILES], d2[TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            d1[t] = d2[t] = acc_t{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                d1[t] = mfma16(av[t][s].x, bv[ct][s], d1[t]);
                d2[t] = mfma16(av[t][s].y, bv[ct][s], d2[t]);
            }
        }
        const bool there = 2 * ct + (q >> 2) < p.nrhs;
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * t + mfma_row<T>(lane, r);
                T v = fma(sp, xor8(d2[t][r]), d1[t][r]);
                if ((mx && row < NZ) || (my && row >= NZ && row < 2 * NZ)) v = -v;
                if (there && row < C) col[ct][2 * row] = v;
            }
    }
}

template <typename T, int NZ>
void launch_direct(const ApplyArgs &a, hipStream_t s)
{
    const DirectArgs<T> p{(const cplx<T> *)a.G, (cplx<T> *)a.buf, a.g.M(), (int)a.g.Lq(), a.nrhs, a.g.nx, a.g.ny};
    const dim3 grid((unsigned)ceil_div(a.g.Lq(), 4)), nt(256);
    if (a.nrhs <= 2) hipLaunchKernelGGL((contract_direct_kernel<T, NZ, 1>), grid, nt, 0, s, p);
    else if (a.nrhs <= 4) hipLaunchKernelGGL((contract_direct_kernel<T, NZ, 2>), grid, nt, 0, s, p);
    else hipLaunchKernelGGL((contract_direct_kernel<T, NZ, 4>), grid, nt, 0, s, p);
    XTR_LAUNCH_CHECK("contract_direct_kernel");
}

template <typename T, int NZ = 1>
bool direct_depth(const ApplyArgs &a, hipStream_t s)
{
    if constexpr (NZ > kDirectMostLayers) {
        return false;
    } else {
        if (a.g.nz != NZ) return direct_depth<T, NZ + 1>(a, s);
        launch_direct<T, NZ>(a, s);
        return true;
    }
}

}  // namespace

bool contract_direct(const ApplyArgs &a, hipStream_t s)
{
    return a.precision ? direct_depth<float>(a, s) : direct_depth<double>(a, s);
}

}  // namespace xtr
