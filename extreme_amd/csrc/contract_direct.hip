// Contractions of the operator apply for a folded Green tensor whose operands go straight from memory into the
// lanes of the MFMAs that need them: few layers, a wave per block; and blocks too large for LDS, a wave per 16 rows.
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

// v with its sign bit flipped where s has bit 31 set: every sign below is a mask, not a branch
__device__ __forceinline__ float flip(float v, unsigned s) { return __uint_as_float(__float_as_uint(v) ^ s); }
__device__ __forceinline__ double flip(double v, unsigned s)
{
    return __hiloint2double(__double2hiint(v) ^ (int)s, __double2loint(v));
}
__device__ __forceinline__ unsigned sign_if(bool b) { return (unsigned)b << 31; }
// sign of the mirrored element k of a column: x components by fx, y components by fy, of nz each
__device__ __forceinline__ unsigned sign_of(int k, int nz, unsigned fx, unsigned fy)
{
    return (k < nz ? fx : 0u) | (k >= nz && k < 2 * nz ? fy : 0u);
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
            const unsigned neg = sign_if(zr && !zc);
            const cplx<T> v = g[o];
            av[t][s] = mk<T>(flip(v.x, neg), flip(v.y, neg));
        }
    }
    // images: bit 0 mirrors x, bit 1 mirrors y, where a mirror image exists; else the image stands for the other
    const int img = q & 3;
    const bool mx = (img & 1) && qx > 0 && qx < p.nx, my = (img >> 1) && qy > 0 && qy < p.ny;
    const int64_t l = (int64_t)(mx ? 2 * p.nx - qx : qx) * (2 * p.ny) + (my ? 2 * p.ny - qy : qy);
    const unsigned fx = sign_if(mx), fy = sign_if(my);
    T *col[CT];
    T bv[CT][KS];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        col[ct] = reinterpret_cast<T *>(p.buf + min(2 * ct + (q >> 2), p.nrhs - 1) * p.M + l * C) + part;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int k = 4 * s + kl;
            const T v = flip(col[ct][2 * min(k, C - 1)], sign_of(k, NZ, fx, fy));
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
                const T v = flip(fma(sp, xor8(d2[t][r]), d1[t][r]), sign_of(row, NZ, fx, fy));
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
    note_contract(a, "contract_direct_kernel", NZ, a.nrhs <= 2 ? 1 : a.nrhs <= 4 ? 2 : 4);
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

// The same for a block that does not fit in LDS: a workgroup per block and group of right-hand sides, a wave per 16
// rows. The spectrum columns (8 CT of 3nz values) are copied into LDS, zero past the last; A values come straight
// from memory, 8 k-steps ahead. Every element of the packed components is read by up to two waves and lies in a row
// of its own for most lanes, so the wave-loads, 64 cache lines each, bound it:
// 40 x 40 x 57, 1 right-hand side 150 us for 353 MB (the kernel for one wavenumber at a time, which expands a block
// through registers: 773), 2: 153 (594), 5: 419 (973); 40 x 40 x 63, 1: 163 (1072); 24 x 24 x 80, 1: 112 (682).
constexpr int kRowsAhead = 8;

template <typename T, int CT>
__global__ __launch_bounds__(1024) void contract_rows_kernel(DirectArgs<T> p, int nz, int mask)
{
    using acc_t = typename MfmaAcc<T>::type;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    cplx<T> *cols = reinterpret_cast<cplx<T> *>(smem);                   // [8 CT][ld]
    const int C = 3 * nz, S = nz * (nz + 1) / 2, A = nz * nz, KS = (C + 3) / 4;
    const int steps = (KS + kRowsAhead - 1) / kRowsAhead * kRowsAhead;
    const int ld = 4 * steps + 2;                                        // 2 mod 4: the columns on different banks
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int b = blockIdx.x, h0 = 2 * CT * blockIdx.y;
    const int qx = b / (p.ny + 1), qy = b - qx * (p.ny + 1);
    // image img of the block: bit 0 mirrors x, bit 1 y, where a mirror image exists
    const bool two_x = qx > 0 && qx < p.nx, two_y = qy > 0 && qy < p.ny;
    auto column = [&](int q, int ct) {                                   // of right-hand side h0 + 2 ct + (q >> 2)
        const bool mx = (q & 1) && two_x, my = (q & 2) && two_y;
        const int64_t l = (int64_t)(mx ? 2 * p.nx - qx : qx) * (2 * p.ny) + (my ? 2 * p.ny - qy : qy);
        return p.buf + min(h0 + 2 * ct + (q >> 2), p.nrhs - 1) * p.M + l * C;
    };
    const cplx<T> *g = p.G + (int64_t)b * (4 * S + 2 * A);
    const int kl = lane >> 4, part = (lane >> 3) & 1, q = lane & 7;
    const int row = min(16 * wave + (lane & 15), C - 1), ar = row / nz, i = row - ar * nz;
    const bool zr = ar == 2;
    auto get = [&](int s) __attribute__((always_inline)) {               // G[row][k], k = 4 s + kl
        const int k = min(4 * s + kl, C - 1), ac = (int)(k >= nz) + (int)(k >= 2 * nz), c = k - ac * nz;
        const int hi = max(i, c), lo = min(i, c);
        const bool zc = ac == 2;
        const int sym = (zr ? 3 : ar + ac) * S + lo + hi * (hi + 1) / 2;
        const int asym = 4 * S + (zr ? ac * A + c * nz + (i ^ (c & mask)) : ar * A + i * nz + (c ^ (i & mask)));
        return g[zr == zc ? sym : asym];
    };
    const unsigned neg = sign_if(zr);                                    // of a z row's values with k < 2nz
    cplx<T> av[kRowsAhead];
#pragma unroll
    for (int s = 0; s < kRowsAhead; ++s) av[s] = get(s);
    for (int e = threadIdx.x; e < 8 * CT * 4 * steps; e += blockDim.x) {
        const int col = e / (4 * steps), k = e - col * (4 * steps), qc = col & 7;
        const unsigned f = sign_of(k, nz, sign_if((qc & 1) && two_x), sign_if((qc & 2) && two_y));
        const cplx<T> v = column(qc, col >> 3)[min(k, C - 1)];
        cols[col * ld + k] = k < C ? mk<T>(flip(v.x, f), flip(v.y, f)) : mk<T>(0, 0);
    }
    __syncthreads();
    const T *u = reinterpret_cast<const T *>(cols + q * ld + kl) + part;
    acc_t d1[CT], d2[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) d1[ct] = d2[ct] = acc_t{0, 0, 0, 0};
    for (int s0 = 0; s0 < steps; s0 += kRowsAhead) {
        cplx<T> now[kRowsAhead];
#pragma unroll
        for (int s = 0; s < kRowsAhead; ++s) {
            const unsigned f = 4 * (s0 + s) + kl < 2 * nz ? neg : 0u;
            now[s] = mk<T>(flip(av[s].x, f), flip(av[s].y, f));
            av[s] = get(s0 + kRowsAhead + s);                            // past the end: the last one again, unused
        }
#pragma unroll
        for (int s = 0; s < kRowsAhead; ++s)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const T bv = u[2 * (8 * ct * ld + 4 * (s0 + s))];
                d1[ct] = mfma16(now[s].x, bv, d1[ct]);
                d2[ct] = mfma16(now[s].y, bv, d2[ct]);
            }
    }
    const unsigned fx = sign_if((q & 1) && two_x), fy = sign_if((q & 2) && two_y);
    const T sp = part ? T(1) : T(-1);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        T *dst = reinterpret_cast<T *>(column(q, ct)) + part;
        const bool there = h0 + 2 * ct + (q >> 2) < p.nrhs;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = 16 * wave + mfma_row<T>(lane, r);
            const T v = flip(fma(sp, xor8(d2[ct][r]), d1[ct][r]), sign_of(o, nz, fx, fy));
            if (there && o < C) dst[2 * o] = v;
        }
    }
}

template <typename T, int CT>
void launch_rows(const ApplyArgs &a, hipStream_t s)
{
    const DirectArgs<T> p{(const cplx<T> *)a.G, (cplx<T> *)a.buf, a.g.M(), (int)a.g.Lq(), a.nrhs, a.g.nx, a.g.ny};
    const int C = 3 * a.g.nz, steps = (int)ceil_div(ceil_div(C, 4), kRowsAhead) * kRowsAhead;
    const dim3 grid((unsigned)a.g.Lq(), (unsigned)ceil_div(a.nrhs, 2 * CT)), nt((unsigned)(ceil_div(C, 16) * 64));
    const size_t lds = (size_t)8 * CT * (4 * steps + 2) * sizeof(cplx<T>);
    hipLaunchKernelGGL((contract_rows_kernel<T, CT>), grid, nt, lds, s, p, a.g.nz, asym_swizzle_mask(a.g.nz));
    XTR_LAUNCH_CHECK("contract_rows_kernel");
    note_contract(a, "contract_rows_kernel", 0, CT);
}

}  // namespace

bool contract_direct(const ApplyArgs &a, hipStream_t s)
{
    return a.precision ? direct_depth<float>(a, s) : direct_depth<double>(a, s);
}

bool contract_rows(const ApplyArgs &a, hipStream_t s)
{
    if (3 * a.g.nz > kRowsMost) return false;
    if (a.nrhs <= 2) a.precision ? launch_rows<float, 1>(a, s) : launch_rows<double, 1>(a, s);
    else a.precision ? launch_rows<float, 2>(a, s) : launch_rows<double, 2>(a, s);
    return true;
}

}  // namespace xtr
