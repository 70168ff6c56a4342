// LDS-staged and register-resident pencil FFTs (templates), shared by the apply's four passes
// (op_fft_forward.hip, op_fft_inverse.hip) and the 2-D transforms of assembled tensors (tensor_fft.hip).
//
// 2-D transforms are unnormalised, sign -1 forward, +1 backward (Fft/FftW/FftWTransform.cs:20-27).
//
// A pencil kernel owns TC adjacent columns and all P points of each: it stages the
// TC x P tile in LDS (column index fastest, so global loads of a row of TC columns are
// contiguous), runs a Stockham radix-4/2/3/5 transform with every stage reading its
// butterfly inputs into registers before a barrier and writing after it, and writes
// the tile back. The zero padding of the forward passes and the cropping of the inverse
// passes are applied at load/store time, so padded rows are never read or written twice.
#pragma once

#include <string>
#include <type_traits>

#include "xtr_common.h"
#include "xtr_kernels.h"

namespace xtr {

constexpr int kFftThreads = 256;

// ---- compile-time radix plan: 4s first, then 2, then 3, then 5 ---------------------------------
constexpr int radix_of(int len)
{
    return (len % 4 == 0) ? 4 : (len % 2 == 0) ? 2 : (len % 3 == 0) ? 3 : 5;
}

template <typename T, int R, int DIR>
__host__ __device__ inline void dft_small(cplx<T> *a)
{
    if constexpr (R == 2) {
        cplx<T> t = a[0];
        a[0] = cadd<T>(t, a[1]);
        a[1] = csub<T>(t, a[1]);
    } else if constexpr (R == 4) {
        cplx<T> t0 = cadd<T>(a[0], a[2]), t1 = csub<T>(a[0], a[2]);
        cplx<T> t2 = cadd<T>(a[1], a[3]), d = csub<T>(a[1], a[3]);
        // t3 = d * (DIR i)
        cplx<T> t3 = DIR < 0 ? mk<T>(d.y, -d.x) : mk<T>(-d.y, d.x);
        a[0] = cadd<T>(t0, t2);
        a[1] = cadd<T>(t1, t3);
        a[2] = csub<T>(t0, t2);
        a[3] = csub<T>(t1, t3);
    } else if constexpr (R == 5) {
        // w = exp(DIR 2 pi i / 5): with s1 = a1 + a4, d1 = a1 - a4, s2 = a2 + a3, d2 = a2 - a3,
        // y1,4 = a0 + c1 s1 + c2 s2 +- DIR i (n1 d1 + n2 d2), y2,3 = a0 + c2 s1 + c1 s2 +- DIR i (n2 d1 - n1 d2),
        // c1 = cos(2 pi/5) = (sqrt5 - 1)/4, c2 = cos(4 pi/5) = -(sqrt5 + 1)/4, n1 = sin(2 pi/5), n2 = sin(4 pi/5)
        const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
        const T n1 = (T)0.95105651629515357212, n2 = (T)0.58778525229247312917;
        const cplx<T> s1 = cadd<T>(a[1], a[4]), d1 = csub<T>(a[1], a[4]);
        const cplx<T> s2 = cadd<T>(a[2], a[3]), d2 = csub<T>(a[2], a[3]);
        const cplx<T> m1 = mk<T>(a[0].x + c1 * s1.x + c2 * s2.x, a[0].y + c1 * s1.y + c2 * s2.y);
        const cplx<T> m2 = mk<T>(a[0].x + c2 * s1.x + c1 * s2.x, a[0].y + c2 * s1.y + c1 * s2.y);
        const cplx<T> e1 = mk<T>(n1 * d1.x + n2 * d2.x, n1 * d1.y + n2 * d2.y);
        const cplx<T> e2 = mk<T>(n2 * d1.x - n1 * d2.x, n2 * d1.y - n1 * d2.y);
        // DIR i e
        const cplx<T> j1 = DIR < 0 ? mk<T>(e1.y, -e1.x) : mk<T>(-e1.y, e1.x);
        const cplx<T> j2 = DIR < 0 ? mk<T>(e2.y, -e2.x) : mk<T>(-e2.y, e2.x);
        a[0] = mk<T>(a[0].x + s1.x + s2.x, a[0].y + s1.y + s2.y);
        a[1] = cadd<T>(m1, j1);
        a[4] = csub<T>(m1, j1);
        a[2] = cadd<T>(m2, j2);
        a[3] = csub<T>(m2, j2);
    } else {  // R == 3, w = exp(DIR 2 pi i / 3)
        const T h = (T)0.86602540378443864676;  // sqrt(3)/2
        cplx<T> s = cadd<T>(a[1], a[2]), d = csub<T>(a[1], a[2]);
        cplx<T> m = mk<T>(a[0].x - (T)0.5 * s.x, a[0].y - (T)0.5 * s.y);
        // (DIR h) i d
        cplx<T> id = DIR < 0 ? mk<T>(h * d.y, -h * d.x) : mk<T>(-h * d.y, h * d.x);
        a[0] = cadd<T>(a[0], s);
        a[1] = cadd<T>(m, id);
        a[2] = csub<T>(m, id);
    }
}

// exp(DIR 2 pi i j / 16) applied to x, j in 0..15 known at compile time after unrolling. The
// cosines of multiples of pi/8 are 1, cos(pi/8), sqrt(1/2), sin(pi/8), 0 and their mirrors.
template <typename T, int DIR>
__host__ __device__ inline cplx<T> rot16(cplx<T> x, int j)
{
    constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173, h = 0.70710678118654752440;
    const double cs[16] = {1, c1, h, s1, 0, -s1, -h, -c1, -1, -c1, -h, -s1, 0, s1, h, c1};
    j &= 15;
    if (j == 0) return x;
    if (j == 4) return DIR < 0 ? mk<T>(x.y, -x.x) : mk<T>(-x.y, x.x);       // DIR i
    if (j == 8) return mk<T>(-x.x, -x.y);
    if (j == 12) return DIR < 0 ? mk<T>(-x.y, x.x) : mk<T>(x.y, -x.x);      // -DIR i
    const T c = (T)cs[j], sn = (T)(DIR < 0 ? -cs[(j + 12) & 15] : cs[(j + 12) & 15]);   // sin = cos(. - pi/2)
    return mk<T>(x.x * c - x.y * sn, x.x * sn + x.y * c);
}

// In-register DFT of length R = 8 or 16 (sign DIR): n = (R/4) n1 + n2, k = k1 + 4 k2, a length-4
// DFT over n1 for each n2, the twiddles exp(DIR 2 pi i n2 k1 / R), then a length-R/4 DFT over n2.
template <typename T, int R, int DIR>
__host__ __device__ inline void dft_pow2(cplx<T> *a)
{
    static_assert(R == 8 || R == 16, "dft_pow2 covers 8 and 16");
    constexpr int R2 = R / 4;
    cplx<T> b[R];
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
        cplx<T> t[4] = {a[n2], a[R2 + n2], a[2 * R2 + n2], a[3 * R2 + n2]};
        dft_small<T, 4, DIR>(t);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) b[n2 * 4 + k1] = rot16<T, DIR>(t[k1], n2 * k1 * (16 / R));
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        cplx<T> t[R2];
#pragma unroll
        for (int n2 = 0; n2 < R2; ++n2) t[n2] = b[n2 * 4 + k1];
        dft_small<T, R2, DIR>(t);
#pragma unroll
        for (int k2 = 0; k2 < R2; ++k2) a[k1 + 4 * k2] = t[k2];
    }
}

// One Stockham stage over the LDS tile s[p*TC + c] (NT threads) and the recursion to the next stage.
template <typename T, int P, int TC, int DIR, int LEN, int ST, int NT>
__device__ inline void fft_stage(cplx<T> *s, const cplx<T> *tw, int tid)
{
    constexpr int R = radix_of(LEN);
    constexpr int M = LEN / R;
    constexpr int NB = (P / R) * TC;
    constexpr int NPT = (NB + NT - 1) / NT;
    cplx<T> y[NPT][R];
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
        const int b = tid + k * NT;
        if (NB % NT == 0 || b < NB) {
            const int cl = b % TC, bb = b / TC;
            const int p = bb / ST, q = bb % ST;
            cplx<T> a[R];
#pragma unroll
            for (int t = 0; t < R; ++t) a[t] = s[(q + ST * (p + t * M)) * TC + cl];
            dft_small<T, R, DIR>(a);
#pragma unroll
            for (int u = 1; u < R; ++u) a[u] = cmul<T>(a[u], tw[p * u * (P / LEN)]);
#pragma unroll
            for (int u = 0; u < R; ++u) y[k][u] = a[u];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
        const int b = tid + k * NT;
        if (NB % NT == 0 || b < NB) {
            const int cl = b % TC, bb = b / TC;
            const int p = bb / ST, q = bb % ST;
#pragma unroll
            for (int u = 0; u < R; ++u) s[(q + ST * (R * p + u)) * TC + cl] = y[k][u];
        }
    }
    __syncthreads();
    if constexpr (M > 1) fft_stage<T, P, TC, DIR, M, ST * R, NT>(s, tw, tid);
}

// ---- load/store policies -------------------------------------------------------------------

// Generic strided pencils of one array per right-hand side. Column c lives at
// (c / cpr) * row_stride + (c % cpr); point p at + p * pstride. Columns fit 32 bits (a division of 64 takes
// several times the instructions).
template <typename T>
struct IoPlain {
    cplx<T> *buf;
    int64_t rhs_stride;
    int64_t ncols, cpr, row_stride, pstride;
    int n_in, n_out;
    __device__ int64_t addr(int rhs, int64_t c, int p) const
    {
        const unsigned col = (unsigned)c, per = (unsigned)cpr, row = col / per;
        return rhs * rhs_stride + row * row_stride + (col - row * per) + (int64_t)p * pstride;
    }
    __device__ cplx<T> load(int rhs, int64_t c, int p) const
    {
        if (c >= ncols || p >= n_in) return mk<T>(0, 0);
        return buf[addr(rhs, c, p)];
    }
    __device__ void store(int rhs, int64_t c, int p, cplx<T> v) const
    {
        if (c < ncols && p < n_out) buf[addr(rhs, c, p)] = v;
    }
};

// Column tile of workgroup b among nb. Workgroups go to the 8 XCDs round-robin (b mod 8), and
// each XCD has its own L2. Giving XCD x a contiguous run of tiles puts neighbouring tiles, which
// share cache lines of narrow rows (and the R values of the three components of one cell), on one
// L2; in launch order they would sit on eight different ones. A bijection on [0, nb).
__device__ __forceinline__ int64_t xcd_tile(int64_t b, int64_t nb)
{
    const int64_t per = nb / 8, rem = nb % 8, x = b % 8, i = b / 8;
    return x * per + (x < rem ? x : rem) + i;
}

template <typename T, int P, int TC, int DIR, class IO, int NT>
__global__ __launch_bounds__(NT) void pencil_fft_kernel(IO io, const cplx<T> *__restrict__ twg)
{
    __shared__ cplx<T> s[P * TC];
    __shared__ cplx<T> tw[P];
    const int tid = threadIdx.x;
    for (int k = tid; k < P; k += NT) {
        cplx<T> w = twg[k];
        tw[k] = DIR < 0 ? w : cconj<T>(w);
    }
    const int64_t c0 = xcd_tile(blockIdx.x, gridDim.x) * TC;
    const int rhs = blockIdx.y;
    constexpr int NE = (P * TC + NT - 1) / NT;
#pragma unroll
    for (int k = 0; k < NE; ++k) {
        const int e = tid + k * NT;
        if ((P * TC) % NT == 0 || e < P * TC) {
            const int p = e / TC, cl = e % TC;
            s[p * TC + cl] = io.load(rhs, c0 + cl, p);
        }
    }
    __syncthreads();
    fft_stage<T, P, TC, DIR, P, 1, NT>(s, tw, tid);
#pragma unroll
    for (int k = 0; k < NE; ++k) {
        const int e = tid + k * NT;
        if ((P * TC) % NT == 0 || e < P * TC) {
            const int p = e / TC, cl = e % TC;
            io.store(rhs, c0 + cl, p, s[p * TC + cl]);
        }
    }
}

// ---- register-resident pencils for lengths 64, 128, 256, 512 -------------------------------
// The same Stockham stages with radix 16 or 8, so a length takes two or three stages: the first
// reads its butterfly inputs straight from global memory (through the load policy), the last
// writes its outputs straight to global memory, and only the exchanges between stages go through
// the LDS tile (one exchange for 64, 128 and 256; two for 512 = 8 x 8 x 8).
constexpr int reg_radix(int len)
{
    return (len == 512 || len == 64 || len % 16 != 0) ? 8 : 16;
}
constexpr bool reg_length(int p) { return p == 64 || p == 128 || p == 256 || p == 512; }
template <int P, int TC>
constexpr int reg_threads()
{
    const int n = TC * (P / reg_radix(P));
    return n < 64 ? 64 : n > 512 ? 512 : n;
}

// An exchange is made in two halves, the real parts and then the imaginary ones, so that the LDS tile takes half
// the bytes and more workgroups share a CU: what bounds a pass is the bytes in flight, since a workgroup does
// not load while it transforms. Against exchanging whole complex values (more LDS, two barriers fewer), the same
// arithmetic: 512 points, 256 x 256 x 64 cells, 304 -> 264, 506 -> 495, 544 -> 523, 359 -> 350 us for the four
// passes of an apply; the folded Green tensor's passes at 256 points 0.90 -> 0.74 ms.
template <typename T, int P, int TC, int DIR, int LEN, int ST, int NT, class IO>
__device__ __forceinline__ void reg_stage(const IO &io, int rhs, int64_t c0, T *s, const cplx<T> *tw, int tid,
                                            cplx<T> (&a)[(P / reg_radix(LEN) * TC + NT - 1) / NT][reg_radix(LEN)])
{
    constexpr int R = reg_radix(LEN), M = LEN / R, NB = (P / R) * TC, NPT = (NB + NT - 1) / NT;
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
        const int b = tid + k * NT;
        if (NB % NT == 0 || b < NB) {
            dft_pow2<T, R, DIR>(a[k]);
            const int cl = b % TC, bb = b / TC;
            if constexpr (M == 1) {
#pragma unroll
                for (int u = 0; u < R; ++u) io.store(rhs, c0 + cl, bb % ST + ST * u, a[k][u]);
            } else {
#pragma unroll
                for (int u = 1; u < R; ++u) a[k][u] = cmul<T>(a[k][u], tw[bb / ST * u * (P / LEN)]);
            }
        }
    }
    if constexpr (M > 1) {
        constexpr int R2 = reg_radix(M), M2 = M / R2, NB2 = (P / R2) * TC, NPT2 = (NB2 + NT - 1) / NT;
        cplx<T> n[NPT2][R2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (LEN < P || h) __syncthreads();         // the last half's reads are done
#pragma unroll
            for (int k = 0; k < NPT; ++k) {
                const int b = tid + k * NT;
                if (NB % NT == 0 || b < NB) {
                    const int cl = b % TC, bb = b / TC, p = bb / ST, q = bb % ST;
#pragma unroll
                    for (int u = 0; u < R; ++u) s[(q + ST * (R * p + u)) * TC + cl] = h ? a[k][u].y : a[k][u].x;
                }
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < NPT2; ++k) {
                const int b = tid + k * NT;
                if (NB2 % NT == 0 || b < NB2) {
                    const int cl = b % TC, bb = b / TC, p = bb / (ST * R), q = bb % (ST * R);
#pragma unroll
                    for (int t = 0; t < R2; ++t) {
                        const T v = s[(q + ST * R * (p + t * M2)) * TC + cl];
                        if (h) n[k][t].y = v;
                        else n[k][t].x = v;
                    }
                }
            }
        }
        reg_stage<T, P, TC, DIR, M, ST * R, NT>(io, rhs, c0, s, tw, tid, n);
    }
}

template <typename T, int P, int TC, int DIR, class IO, int NT>
__global__ __launch_bounds__(NT) void pencil_fft_reg_kernel(IO io, const cplx<T> *__restrict__ twg)
{
    static_assert(reg_length(P), "register pencils cover 64, 128, 256 and 512");
    constexpr int R = reg_radix(P), M = P / R, NB = (P / R) * TC, NPT = (NB + NT - 1) / NT;
    __shared__ T s[P * TC];
    __shared__ cplx<T> tw[P];
    const int tid = threadIdx.x, rhs = blockIdx.y;
    const int64_t c0 = xcd_tile(blockIdx.x, gridDim.x) * TC;
    cplx<T> a[NPT][R];
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
        const int b = tid + k * NT;
        if (NB % NT == 0 || b < NB) {
#pragma unroll
            for (int t = 0; t < R; ++t) a[k][t] = io.load(rhs, c0 + b % TC, b / TC + t * M);
        }
    }
    for (int k = tid; k < P; k += NT) {
        cplx<T> w = twg[k];
        tw[k] = DIR < 0 ? w : cconj<T>(w);
    }
    __syncthreads();
    reg_stage<T, P, TC, DIR, P, 1, NT>(io, rhs, c0, s, tw, tid, a);
}

// Column tiles per pencil length (fft_tile_cols): the default, for lengths from 64 a narrow and a wide one, and
// from 128 the narrow tile also with 512 threads (twice the waves per CU for the same LDS). Which
// one a pass uses is measured on the device (the operator's tile tuning); the choice does not change
// the arithmetic, only how the columns are grouped and how many threads share a tile.
template <typename T, int P>
constexpr int tile_cols_of(int tile)
{
    return fft_tile_cols(P, (int)sizeof(cplx<T>), tile);
}
template <int P>
constexpr int tile_threads_of(int tile)
{
    return tile == FFT_TILE_NARROW_T512 && P >= 128 ? 512 : kFftThreads;
}

// TILES_ALL: every tile (the apply's passes, which measure them); otherwise the default, the register pencil of the
// default column count and, with TILES_NARROW, the narrow tile.
enum { TILES_TWO, TILES_NARROW, TILES_ALL };
template <typename T, int DIR, class IO, int TILES = TILES_ALL>
void launch_pencil(int P, const IO &io, int64_t ncols, int nrhs, const void *tw, hipStream_t s, int tile)
{
    auto go = [&](auto pc) {
        constexpr int PP = decltype(pc)::value;
        constexpr int TD = tile_cols_of<T, PP>(FFT_TILE_DEFAULT), TW = tile_cols_of<T, PP>(FFT_TILE_WIDE),
                      TN = tile_cols_of<T, PP>(FFT_TILE_NARROW);
        constexpr int NW = tile_threads_of<PP>(FFT_TILE_NARROW_T512);
        auto run = [&](auto tc, auto nt) {
            constexpr int TC = decltype(tc)::value, NT = decltype(nt)::value;
            dim3 grid((unsigned)ceil_div(ncols, TC), nrhs);
            hipLaunchKernelGGL((pencil_fft_kernel<T, PP, TC, DIR, IO, NT>), grid, dim3(NT), 0, s, io,
                               (const cplx<T> *)tw);
        };
        using T256 = std::integral_constant<int, kFftThreads>;
        if constexpr (reg_length(PP)) {
            if (tile == FFT_TILE_REG || tile == FFT_TILE_REG_ALT) {
                auto reg = [&](auto tc) {
                    constexpr int TC = decltype(tc)::value, NT = reg_threads<PP, TC>();
                    dim3 grid((unsigned)ceil_div(ncols, TC), nrhs);
                    hipLaunchKernelGGL((pencil_fft_reg_kernel<T, PP, TC, DIR, IO, NT>), grid, dim3(NT), 0, s, io,
                                       (const cplx<T> *)tw);
                };
                if constexpr (TILES == TILES_ALL) {
                    if (tile == FFT_TILE_REG_ALT) {
                        reg(std::integral_constant<int, tile_cols_of<T, PP>(FFT_TILE_REG_ALT)>{});
                        return;
                    }
                }
                reg(std::integral_constant<int, tile_cols_of<T, PP>(FFT_TILE_REG)>{});
                return;
            }
        }
        if constexpr (TILES >= TILES_NARROW) {
            if (tile == FFT_TILE_NARROW && TN != TD) return run(std::integral_constant<int, TN>{}, T256{});
        }
        if constexpr (TILES == TILES_ALL) {
            if (tile == FFT_TILE_WIDE && TW != TD) return run(std::integral_constant<int, TW>{}, T256{});
            if (tile == FFT_TILE_NARROW_T512 && TN != TD && NW != kFftThreads)
                return run(std::integral_constant<int, TN>{}, std::integral_constant<int, NW>{});
        }
        run(std::integral_constant<int, TD>{}, T256{});
    };
    switch (P) {
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 8: go(std::integral_constant<int, 8>{}); break;
    case 10: go(std::integral_constant<int, 10>{}); break;
    case 12: go(std::integral_constant<int, 12>{}); break;
    case 16: go(std::integral_constant<int, 16>{}); break;
    case 20: go(std::integral_constant<int, 20>{}); break;
    case 24: go(std::integral_constant<int, 24>{}); break;
    case 30: go(std::integral_constant<int, 30>{}); break;
    case 32: go(std::integral_constant<int, 32>{}); break;
    case 40: go(std::integral_constant<int, 40>{}); break;
    case 48: go(std::integral_constant<int, 48>{}); break;
    case 50: go(std::integral_constant<int, 50>{}); break;
    case 60: go(std::integral_constant<int, 60>{}); break;
    case 64: go(std::integral_constant<int, 64>{}); break;
    case 80: go(std::integral_constant<int, 80>{}); break;
    case 96: go(std::integral_constant<int, 96>{}); break;
    case 100: go(std::integral_constant<int, 100>{}); break;
    case 120: go(std::integral_constant<int, 120>{}); break;
    case 128: go(std::integral_constant<int, 128>{}); break;
    case 150: go(std::integral_constant<int, 150>{}); break;
    case 160: go(std::integral_constant<int, 160>{}); break;
    case 192: go(std::integral_constant<int, 192>{}); break;
    case 200: go(std::integral_constant<int, 200>{}); break;
    case 240: go(std::integral_constant<int, 240>{}); break;
    case 256: go(std::integral_constant<int, 256>{}); break;
    case 300: go(std::integral_constant<int, 300>{}); break;
    case 320: go(std::integral_constant<int, 320>{}); break;
    case 384: go(std::integral_constant<int, 384>{}); break;
    case 400: go(std::integral_constant<int, 400>{}); break;
    case 480: go(std::integral_constant<int, 480>{}); break;
    case 512: go(std::integral_constant<int, 512>{}); break;
    default: throw hip_error("unsupported FFT length " + std::to_string(P));
    }
    XTR_LAUNCH_CHECK("pencil_fft_kernel");
}

}  // namespace xtr
