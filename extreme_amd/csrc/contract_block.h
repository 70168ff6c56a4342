// Contraction of the operator apply for a folded Green tensor whose block fits in LDS, one kernel per depth.
// Included by the units that instantiate it (contract_block_*.hip), which split the depths for the build.
#pragma once

#include <algorithm>
#include <utility>

#include "xtr_common.h"
#include "xtr_kernels.h"
#include "xtr_mfma.h"

namespace xtr {

// ApplyGreenTensorAlongZ (ConvolutionOperator.cs:274-327) over a folded tensor, for every depth whose block
// fits (complex128: nz <= 47, complex64: nz <= 63) except those with kernels of their own. A folded block
// serves 4 wavenumbers (its images) x the right-hand sides: Y = G U is a small GEMM,
// (3nz x 3nz) x (3nz x columns), on 16x16x4 MFMAs with B = [Re U | Im U] (8 complex columns per tile),
// D1 = Re G . B, D2 = Im G . B, Re Y = D1[:, :8] - D2[:, 8:], Im Y = D1[:, 8:] + D2[:, :8].
//
// Bound by HBM (the block is read once) if the copies stay ahead of the arithmetic and the arithmetic is not
// drowned in address computations. A persistent workgroup holds one block image in LDS, in two regions that
// are copied and contracted in turn (global_load_lds, no registers): region 1 the packed xx, xy, yy, zz and
// the spectrum columns, region 2 xz and yz. While one region is contracted the other is in flight, so half an
// image is always on its way even where only one workgroup fits a CU (nz = 40: 118 KB); at smaller depths
// several workgroups share a CU. The spectrum columns are read into registers (B fragments with the mirror
// signs) before region 1 is contracted, which frees them with region 1. Waves: ceil(2nz/16) own 16-row tiles
// of the x and y rows, ceil(nz/16) own tiles of the z rows, so the sign of -xz^T, -yz^T is the same for a
// whole wave; each component's k range is padded to 4 KC with zero B values.
// The depth is a template parameter: with it every LDS offset is an immediate or a register computed once, and
// a block costs a wave little more than its MFMAs (with the depth as an argument, 1000 instructions a block
// around the 36 MFMAs of nz = 24, and 77 us instead of 60 at 48 x 96 x 24).
//
// Measured, time of the contraction per apply, against the kernels it replaced (vector FMAs or MFMA on a block
// expanded through registers up to nz = 31, one workgroup per wavenumber from 33, a one-region MFMA kernel for
// 32): 32 x 32 x 8, 1 right-hand side 11.3 -> 8.3 us; 48 x 96 x 24, 2: 150 -> 60 us (264 MB, 4.4 TB/s; the
// copies without arithmetic 47); 40 x 40 x 40, 2: 209 -> 58 us (copies 43); 64 x 64 x 16, 8: 220 -> 77 us
// (copies 56, arithmetic 65 to 80); nz = 32: 64 x 64, 1: 85 -> 79 us, 4: 167 -> 141 us, 128 x 128, 2: 301 us both.
// What is left above the copies is the last, partly filled round of blocks, and MFMA work for padding
// (nz = 24: 80 of 72 rows).
//
// Edge blocks (kx or ky at 0 or N) have fewer than 4 images. They run as the others, with the missing images
// standing for existing ones, and so do right-hand sides past the last, and rows past the last of a tile:
// duplicates compute and store the same values as what they stand for, and no lane is ever masked. The number
// of stores is therefore known, and the waits can count them.
template <typename T, int NZ, int NR>
struct BlockCfg {
    static constexpr int S = NZ * (NZ + 1) / 2, A = NZ * NZ, C = 3 * NZ;
    static constexpr int GB = 4 * S + 2 * A;
    static constexpr int KC = (NZ + 3) / 4;                      // k-steps of one component
    static constexpr int CT = (4 * NR + 7) / 8;                  // column tiles
    static constexpr int TXY = (2 * NZ + 15) / 16, TZ = (NZ + 15) / 16, W = TXY + TZ;
    static constexpr int E = (int)sizeof(cplx<T>);
    static constexpr int MASK = NZ % 16 == 0 ? 15 : (NZ % 8 == 0 ? 7 : 0);   // asym_swizzle_mask
    // column stride: 3nz rounded up to 2 mod 4, so that the 8 columns of a tile fall on different LDS banks
    static constexpr int LDU = (C + 1) / 4 * 4 + 2;
    // complex64 columns of odd length start at odd multiples of 8 bytes: copied 4 bytes a lane
    static constexpr bool U4 = E == 8 && C % 2 == 1;
    static constexpr int UB = U4 ? 256 : 1024;                   // bytes of one spectrum wave-load
    // wave-loads: region 1, spectrum columns, region 2
    static constexpr int N1 = (4 * S * E + 1023) / 1024, NU = (4 * NR * LDU * E + UB - 1) / UB,
                         N2 = (2 * A * E + 1023) / 1024;
    static constexpr int OFFU = N1 * 1024, OFF2 = OFFU + (NU * UB + 1023) / 1024 * 1024, LDS = OFF2 + N2 * 1024;
    __host__ __device__ static constexpr int most(int n) { return (n + W - 1) / W; }   // of one wave
    static constexpr int STORES = 4 * CT;
    // B fragments and accumulators have to leave the waves of a workgroup in the register file
    static constexpr bool ok = LDS <= 160 * 1024 && 3 * KC * CT * (int)sizeof(T) / 4 <= 100 && C >= NR;
    // B fragments, accumulators, LDS offsets and copy sources, in registers; what the waves of a workgroup leave of
    // the register file holds 16 more at the most without spills (complex64 in groups of 4: 152 at 47 layers fit in
    // 168, 154 at 58 and 60 spill 2 and 3 values, 188 at 63 spill 37).
    static constexpr int REGS = (3 * KC + 8) * CT * (int)sizeof(T) / 4 + 2 * KC + most(N1) + most(N2) + 4 * most(NU);
    static constexpr bool spills = REGS + 16 > 512 / ((W + 3) / 4) / 8 * 8;
};

template <typename T>
struct BlockArgs {
    const cplx<T> *G;
    cplx<T> *buf;
    int64_t M;
    int Lq, nrhs, nx, ny;
};

// f(integral_constant<int, t>) for t = 0 .. N-1: array indices known at compile time, so that per-lane arrays
// stay in registers
template <typename F, int... Ts>
__device__ __forceinline__ void static_for(std::integer_sequence<int, Ts...>, F &&f)
{
    (f(std::integral_constant<int, Ts>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for(std::make_integer_sequence<int, N>{}, f);
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void copy16_lds(const void *base, unsigned off, unsigned dst)
{
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(__builtin_amdgcn_readfirstlane(dst)), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void copy16_lds(const void *src, unsigned dst)
{
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(__builtin_amdgcn_readfirstlane(dst)), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ void copy4_lds(const void *src, unsigned dst)
{
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off" ::"s"(__builtin_amdgcn_readfirstlane(dst)), "v"(src) : "memory", "m0");
}
#pragma clang diagnostic pop
// A store that is issued exactly here and by every lane: the waits count it.
__device__ __forceinline__ void store_counted(double *p, double v)
{
    asm volatile("global_store_dwordx2 %0, %1, off" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void store_counted(float *p, float v)
{
    asm volatile("global_store_dword %0, %1, off" ::"v"(p), "v"(v) : "memory");
}

// the value of the lane 8 further in its row of 16 (lane ^ 8)
__device__ __forceinline__ int lane_xor8(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true); }
__device__ __forceinline__ float lane_xor8(float v) { return __int_as_float(lane_xor8(__float_as_int(v))); }
__device__ __forceinline__ double lane_xor8(double v)
{
    return __hiloint2double(lane_xor8(__double2hiint(v)), lane_xor8(__double2loint(v)));
}
// v with its sign bit flipped where s has bit 31 set
__device__ __forceinline__ float flip_sign(float v, unsigned s) { return __uint_as_float(__float_as_uint(v) ^ s); }
__device__ __forceinline__ double flip_sign(double v, unsigned s)
{
    return __hiloint2double(__double2hiint(v) ^ (int)s, __double2loint(v));
}

// Byte offsets, from the spectrum of a right-hand side, of a block's images: the unmirrored one, and what the x
// and the y mirror add (0 where there is no mirror image); the sign bit of a mirrored image's x, y components.
struct BlockPos {
    unsigned at, dx, dy, fx, fy;
    // mx, my: all bits set for a mirrored image (no selects: of struct members they go through scratch)
    __device__ unsigned of(unsigned mx, unsigned my) const { return at + (mx & dx) + (my & dy); }
};

// The block loop of one wave; ZROW: it owns z rows, else x and y rows. Every wave passes the same barriers.
template <typename T, int NZ, int NR, bool ZROW>
__device__ __forceinline__ void block_run(const BlockArgs<T> &p, unsigned char *smem, int wave, int lane)
{
    using K = BlockCfg<T, NZ, NR>;
    using acc_t = typename MfmaAcc<T>::type;
    constexpr int KC = K::KC, CT = K::CT, W = K::W, E = K::E;
    constexpr int M1 = K::most(K::N1), MU = K::most(K::NU), M2 = K::most(K::N2);
    const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem;
    const cplx<T> *img0 = reinterpret_cast<const cplx<T> *>(smem);

    // this lane's operator row (rows past the end repeat the last one)
    const int kl = lane >> 4, part = (lane >> 3) & 1;
    const int t0 = 16 * (ZROW ? wave - K::TXY : wave);
    constexpr int rows = ZROW ? NZ : 2 * NZ;
    const int row = min(t0 + (lane & 15), rows - 1);
    const int a = ZROW ? 2 : (row >= NZ ? 1 : 0), i = ZROW ? row : row - a * NZ;
    // LDS offsets of the A values of k = 4 s + kl: packed symmetric (o1: xx or xy, or zz; xy or yy follow S
    // further on) and xz, yz (o2)
    unsigned o1[KC], o2[KC];
#pragma unroll
    for (int s = 0; s < KC; ++s) {
        const int c = min(4 * s + kl, NZ - 1), hi = max(i, c), lo = min(i, c);
        o1[s] = E * (unsigned)((ZROW ? 3 : a) * K::S + lo + hi * (hi + 1) / 2);
        o2[s] = K::OFF2 + E * (unsigned)(ZROW ? c * NZ + (i ^ (c & K::MASK)) : a * K::A + i * NZ + (c ^ (i & K::MASK)));
    }
    // sources of this wave's copies: offsets within a block, and the lane's place in the spectrum columns
    unsigned s1[M1], s2[M2];
    static_for<M1>([&](auto t) { s1[t] = min((unsigned)((wave + W * t) * 64 + lane) * 16u, 4u * K::S * E - 16u); });
    static_for<M2>([&](auto t) {
        s2[t] = 4u * K::S * E + min((unsigned)((wave + W * t) * 64 + lane) * 16u, 2u * K::A * E - 16u);
    });
    const char *su[MU];
    unsigned ux[MU], uy[MU];
    static_for<MU>([&](auto t) {
        constexpr int EPL = 16 / E;
        const int d = (wave + W * t) * 64 + lane;
        const int e = K::U4 ? d >> 1 : d * EPL;                       // U4: d counts the reals of the columns
        const int col = min(e / K::LDU, 4 * NR - 1);
        const int kk = min(e - col * K::LDU, K::U4 ? K::C - 1 : K::C - EPL);
        ux[t] = 0u - (unsigned)(col & 1);
        uy[t] = 0u - (unsigned)(col >> 1 & 1);
        su[t] = reinterpret_cast<const char *>(p.buf + min(col >> 2, p.nrhs - 1) * p.M + kk) + (K::U4 ? 4 * (d & 1) : 0);
    });
    // this lane's columns: LDS address, destination and image
    const int img = lane & 3;
    const unsigned mx = 0u - (unsigned)(img & 1), my = 0u - (unsigned)(img >> 1);
    unsigned ul[CT];
    char *yd[CT];
    unsigned ro[4];                                                   // byte offsets of the lane's four rows
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int q = 8 * ct + (lane & 7), h = min(q >> 2, p.nrhs - 1);
        ul[ct] = K::OFFU + E * (unsigned)((NR == 1 ? img : q) * K::LDU + kl) + (unsigned)(part * sizeof(T));
        yd[ct] = reinterpret_cast<char *>(p.buf + h * p.M + (ZROW ? 2 * NZ : 0)) + part * sizeof(T);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) ro[r] = E * (unsigned)min(t0 + mfma_row<T>(lane, r), rows - 1);

    const int g = gridDim.x, ny1 = p.ny + 1;
    const int dqx = g / ny1, dqy = g - dqx * ny1;
    int b = blockIdx.x;                                               // the launch keeps gridDim.x <= Lq
    int qx = b / ny1, qy = b - qx * ny1;
    const unsigned rowb = 2u * p.ny * K::C * E;
    auto pos = [&](int px, int py) __attribute__((always_inline)) {
        const bool tx = px > 0 && px < p.nx, ty = py > 0 && py < p.ny;
        return BlockPos{px * rowb + (unsigned)py * (K::C * E), tx ? 2u * (p.nx - px) * rowb : 0u,
                        ty ? 2u * (p.ny - py) * (K::C * E) : 0u, tx ? 0x80000000u : 0u, ty ? 0x80000000u : 0u};
    };
    auto issue1 = [&](int blk, const BlockPos &ps) __attribute__((always_inline)) {
        const char *gp = reinterpret_cast<const char *>(p.G + (int64_t)blk * K::GB);
        static_for<M1>([&](auto t) {
            if ((t + 1) * W <= K::N1 || wave + W * t < K::N1) copy16_lds(gp, s1[t], base + (wave + W * t) * 1024u);
        });
        static_for<MU>([&](auto t) {
            if ((t + 1) * W <= K::NU || wave + W * t < K::NU) {
                const char *src = su[t] + ps.of(ux[t], uy[t]);
                const unsigned dst = base + K::OFFU + (wave + W * t) * (unsigned)K::UB;
                if constexpr (K::U4) copy4_lds(src, dst);
                else copy16_lds(src, dst);
            }
        });
    };
    auto issue2 = [&](int blk) __attribute__((always_inline)) {
        const char *gp = reinterpret_cast<const char *>(p.G + (int64_t)blk * K::GB);
        static_for<M2>([&](auto t) {
            if ((t + 1) * W <= K::N2 || wave + W * t < K::N2)
                copy16_lds(gp, s2[t], base + K::OFF2 + (wave + W * t) * 1024u);
        });
    };
    // copies of this wave beyond the count every wave issues
    const int x2 = wave < K::N2 % W ? 1 : 0;
    const int x1 = (wave < K::N1 % W ? 1 : 0) + (wave < K::NU % W ? 1 : 0);
    constexpr int B1 = K::N1 / W + K::NU / W, B2 = K::N2 / W;

    BlockPos ps = pos(qx, qy);
    issue1(b, ps);
    issue2(b);
    bool first = true;                                                // no stores are out yet
    for (;;) {
        const int bn = b + g;
        const bool more = bn < p.Lq;
        // region 1 and the columns: all but the copies of region 2 and the last block's stores, issued later
        if (first) {
            if (x2) wait_vm<B2 + 1>();
            else wait_vm<B2>();
        } else {
            if (x2) wait_vm<B2 + 1 + K::STORES>();
            else wait_vm<B2 + K::STORES>();
        }
        XTR_BARRIER();
        T bf[CT][3][KC];                                              // B[k][n], the mirror signs applied
        const unsigned fx = mx & ps.fx, fy = my & ps.fy;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int s = 0; s < KC; ++s) {
                T v[3];
#pragma unroll
                for (int ci = 0; ci < 3; ++ci) v[ci] = lds_part<T>(img0, ul[ct] + E * (ci * NZ + 4 * s));
                if (4 * s + 3 >= NZ) {                                // the k past this component
                    const bool in = 4 * s + kl < NZ;
#pragma unroll
                    for (int ci = 0; ci < 3; ++ci) v[ci] = in ? v[ci] : T(0);
                }
                bf[ct][0][s] = flip_sign(v[0], fx);
                bf[ct][1][s] = flip_sign(v[1], fy);
                bf[ct][2][s] = v[2];
            }
        acc_t d1[CT], d2[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) d1[ct] = d2[ct] = acc_t{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < KC; ++s) {
            const cplx<T> g0 = lds_cplx<T>(img0, o1[s]);
            if constexpr (ZROW) {
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    d1[ct] = mfma16(g0.x, bf[ct][2][s], d1[ct]);
                    d2[ct] = mfma16(g0.y, bf[ct][2][s], d2[ct]);
                }
            } else {
                const cplx<T> g1 = lds_cplx<T>(img0, o1[s] + E * K::S);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    d1[ct] = mfma16(g0.x, bf[ct][0][s], d1[ct]);
                    d2[ct] = mfma16(g0.y, bf[ct][0][s], d2[ct]);
                    d1[ct] = mfma16(g1.x, bf[ct][1][s], d1[ct]);
                    d2[ct] = mfma16(g1.y, bf[ct][1][s], d2[ct]);
                }
            }
        }
        XTR_BARRIER();                                                // region 1 and the columns are read
        BlockPos pn = ps;
        if (more) {
            qx += dqx;
            qy += dqy;
            if (qy >= ny1) {
                qy -= ny1;
                ++qx;
            }
            pn = pos(qx, qy);
            issue1(bn, pn);
            // region 2: all but the last block's stores and the copies just issued
            if (first) {
                if (x1 == 0) wait_vm<B1>();
                else if (x1 == 1) wait_vm<B1 + 1>();
                else wait_vm<B1 + 2>();
            } else {
                if (x1 == 0) wait_vm<B1 + K::STORES>();
                else if (x1 == 1) wait_vm<B1 + 1 + K::STORES>();
                else wait_vm<B1 + 2 + K::STORES>();
            }
        } else {
            wait_vm<0>();
        }
        XTR_BARRIER();
#pragma unroll
        for (int s = 0; s < KC; ++s) {
            const cplx<T> g0 = lds_cplx<T>(img0, o2[s]);
            if constexpr (ZROW) {                                     // -xz^T u_x - yz^T u_y
                const cplx<T> g1 = lds_cplx<T>(img0, o2[s] + E * K::A);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    d1[ct] = mfma16s<true>(g0.x, bf[ct][0][s], d1[ct]);
                    d2[ct] = mfma16s<true>(g0.y, bf[ct][0][s], d2[ct]);
                    d1[ct] = mfma16s<true>(g1.x, bf[ct][1][s], d1[ct]);
                    d2[ct] = mfma16s<true>(g1.y, bf[ct][1][s], d2[ct]);
                }
            } else {
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    d1[ct] = mfma16(g0.x, bf[ct][2][s], d1[ct]);
                    d2[ct] = mfma16(g0.y, bf[ct][2][s], d2[ct]);
                }
            }
        }
        XTR_BARRIER();                                                // region 2 is read
        if (more) issue2(bn);
        const unsigned at = ps.of(mx, my);
        const T sp = part ? T(1) : T(-1);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            char *dst = yd[ct] + at;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                T v = fma(sp, lane_xor8(d2[ct][r]), d1[ct][r]);
                if constexpr (!ZROW) v = flip_sign(v, ro[r] < (unsigned)(NZ * E) ? fx : fy);
                store_counted(reinterpret_cast<T *>(dst + ro[r]), v);
            }
        }
        if (!more) break;
        first = false;
        b = bn;
        ps = pn;
    }
    wait_vm<0>();                                                     // no copy may land after exit
}

template <typename T, int NZ, int NR>
__global__ __launch_bounds__((64 * BlockCfg<T, NZ, NR>::W)) void contract_block_kernel(BlockArgs<T> p)
{
    using K = BlockCfg<T, NZ, NR>;
    static_assert(K::N1 / K::W + K::NU / K::W + 2 + K::STORES < 64 && K::N2 / K::W + 1 + K::STORES < 64, "vmcnt range");
    __shared__ __attribute__((aligned(16))) unsigned char smem[K::LDS];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    p.buf += (int64_t)(blockIdx.y * NR) * p.M;                         // this workgroup's right-hand sides
    p.nrhs -= blockIdx.y * NR;
    if (wave < K::TXY) block_run<T, NZ, NR, false>(p, smem, wave, lane);
    else block_run<T, NZ, NR, true>(p, smem, wave, lane);
}

// The right-hand sides in groups of NR, a row of workgroups (blockIdx.y) each: one launch, so that a group fills
// the CUs that the last blocks of another leave. In launches of up to 8, one after the other, 8 right-hand sides
// took 64 instead of 54 us at 64 x 64 x 12, 84 instead of 77 us at nz = 16, 200 instead of 166 us at nz = 24, and
// at 48 x 40 x 40 (launches of 2) 250 instead of 211 us.
template <typename T, int NZ, int NR>
void launch_block(const ApplyArgs &a, hipStream_t s)
{
    using K = BlockCfg<T, NZ, NR>;
    // as many workgroups as are resident at once (registers and LDS): more would run in rounds
    static const int resident = [] {
        int nb = 0;
        XTR_CHECK((hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &nb, (const void *)contract_block_kernel<T, NZ, NR>, 64 * K::W, 0)));
        return std::max(1, nb);
    }();
    BlockArgs<T> p{(const cplx<T> *)a.G, (cplx<T> *)a.buf, a.g.M(), (int)a.g.Lq(), a.nrhs, a.g.nx, a.g.ny};
    const unsigned groups = (unsigned)ceil_div(a.nrhs, NR);
    const unsigned grid = (unsigned)std::min<int64_t>(p.Lq, ceil_div((int64_t)resident * device_cus(), groups));
    hipLaunchKernelGGL((contract_block_kernel<T, NZ, NR>), dim3(grid, groups), dim3(64 * K::W), 0, s, p);
    XTR_LAUNCH_CHECK("contract_block_kernel");
    note_contract(a, "contract_block_kernel", NZ, NR);
}

// Depths LO..HI; false for another depth or one whose block does not fit. One right-hand side or two by
// themselves; more in groups of 4 or 2 (a group reads the tensor once).
template <typename T, int LO, int HI>
bool contract_block_range(const ApplyArgs &a, hipStream_t s)
{
    if constexpr (LO > HI) {
        return false;
    } else {
        if (a.g.nz != LO) return contract_block_range<T, LO + 1, HI>(a, s);
        if constexpr (!BlockCfg<T, LO, 1>::ok) {
            return false;
        } else {
            // Groups of 2 where they leave room for more workgroups on a CU than groups of 4 (3 or 4 instead of 2
            // to 3, by registers and LDS): 8 right-hand sides at 64 x 64, groups of 2 and of 4: nz = 16 77 and
            // 82 us, 20: 130 and 155, 24: 166 and 188; outside these depths 12: 60 and 54, 32: 287 and 266.
            constexpr int most = BlockCfg<T, LO, 4>::ok && (LO < 16 || LO > 25) ? 4 : BlockCfg<T, LO, 2>::ok ? 2 : 1;
            // Where a group of 4 spills, 3 and 4 go in two groups of 2: complex64, 40 x 40 x 63 114 and 118 us instead
            // of 139 and 144, x 57 103 and 107 instead of 124 and 129, x 60 108 and 111 instead of 109 and 110; 16 x 20
            // x 63 32 instead of 43. More than 4 stay in two groups of 4: a third group reads the tensor once more
            // (5 at 40 x 40 x 63: 263 us, in groups of 2 300).
            constexpr int two = BlockCfg<T, LO, 2>::ok ? 2 : 1;
            if (a.nrhs == 1) launch_block<T, LO, 1>(a, s);
            else if (a.nrhs == 2 || (a.nrhs <= 4 && most == 4 && BlockCfg<T, LO, 4>::spills)) launch_block<T, LO, two>(a, s);
            else launch_block<T, LO, most>(a, s);
            return true;
        }
    }
}

}  // namespace xtr
