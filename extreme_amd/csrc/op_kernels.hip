// Per-wavenumber 3x3-block Green-tensor contraction of the operator apply for gfx950, and the Green
// tensor's layout conversions. Spectrum layout: buf[(i*2Ny + j)*3Nz + c*Nz + k], one buffer per
// right-hand side.
//
// The contraction kernels copy the Green tensor (read once per apply: 1.1 GB at 128 x 128 x 32,
// 17 GB at 256 x 256 x 64) HBM -> LDS with the non-temporal hint (nt) on global_load_lds_dwordx4,
// so the stream does not allocate in L2 and the Infinity Cache over the lines the kernel writes
// (the folded contraction at 128 x 128 x 32: 0.337 -> 0.300 ms).
#include <algorithm>
#include <map>
#include <mutex>
#include <utility>
#include <cstdlib>
#include <cstring>

#include "xtr_common.h"
#include "xtr_kernels.h"
#include "xtr_mfma.h"

namespace xtr {

// ---- contraction -----------------------------------------------------------------------------
// ApplyGreenTensorAlongZ (ConvolutionOperator.cs:274-327): for every wavenumber l
//   y_x = XX u_x + XY u_y + XZ u_z
//   y_y = XY u_x + YY u_y + YZ u_z
//   y_z = -XZ^T u_x - YZ^T u_y + ZZ u_z
// XX, XY, YY, ZZ complex-symmetric (stored packed), XZ, YZ full row-major [rc][tr].
// A workgroup owns W wavenumbers and all right-hand sides; thread = (w, rhs, component, row).
// Each of the six blocks is staged in LDS as a padded full nz x (nz+1) matrix (the packed
// blocks are expanded on the way in), so both row and column reads are conflict-light.
// The spectrum is updated in place: every workgroup reads its u into LDS before writing y.
template <typename T>
__global__ __launch_bounds__(1024) void contract_kernel(const cplx<T> *__restrict__ G, cplx<T> *buf, int64_t L,
                                                         int nz, int nrhs, int W, int64_t M,
                                                         const uint16_t *__restrict__ packed_rc, int fold_nx,
                                                         int fold_ny)
{
    // fold_nx > 0: G is folded (block b(l), mirrored components negated on u and y)
    extern __shared__ unsigned char smem_raw[];
    cplx<T> *blk = reinterpret_cast<cplx<T> *>(smem_raw);   // [W][nz][nz+1]
    const int ld = nz + 1;
    cplx<T> *u = blk + (int64_t)W * nz * ld;                  // [W][nrhs][3nz]
    const int C = 3 * nz;
    const int S = nz * (nz + 1) / 2;
    const int64_t gblk = 4LL * S + 2LL * nz * nz;
    const int tid = threadIdx.x, nth = blockDim.x;
    const int64_t l0 = (int64_t)blockIdx.x * W;
    const int per_w = nrhs * C;
    const int swz = asym_swizzle_mask(nz);

    for (int e = tid; e < W * per_w; e += nth) {
        const int w = e / per_w, rest = e % per_w;
        const int rhs = rest / C, q = rest % C;
        const int64_t l = l0 + w;
        cplx<T> v = (l < L) ? buf[rhs * M + l * C + q] : mk<T>(0, 0);
        if (fold_nx > 0 && l < L && q < 2 * nz) {
            const FoldPos p = fold_pos(l, fold_nx, fold_ny);
            if (q < nz ? p.mx : p.my) v = mk<T>(-v.x, -v.y);
        }
        u[e] = v;
    }

    const bool active = tid < W * per_w;
    const int w = active ? tid / per_w : 0;
    const int rest = active ? tid % per_w : 0;
    const int rhs = rest / C, q = rest % C;
    const int a = q / nz, r = q % nz;
    const cplx<T> *uw = u + (w * nrhs + rhs) * C;
    const cplx<T> *bw = blk + (int64_t)w * nz * ld;
    cplx<T> acc = mk<T>(0, 0);

    // block order in memory: xx, xy, yy, zz (packed S), xz, yz (nz*nz)
    for (int bi = 0; bi < 6; ++bi) {
        const bool sym = bi < 4;
        const int64_t off = sym ? (int64_t)bi * S : 4LL * S + (int64_t)(bi - 4) * nz * nz;
        const int sz = sym ? S : nz * nz;
        __syncthreads();
        for (int e = tid; e < W * sz; e += nth) {
            const int ww = e / sz, o = e % sz;
            const int64_t l = l0 + ww;
            const int64_t gb = fold_nx > 0 ? fold_pos(l, fold_nx, fold_ny).b : l;
            const cplx<T> g = (l < L) ? G[gb * gblk + off + o] : mk<T>(0, 0);
            cplx<T> *bb = blk + (int64_t)ww * nz * ld;
            if (sym) {
                const int rc = packed_rc[2 * o], tr = packed_rc[2 * o + 1];
                bb[rc * ld + tr] = g;
                bb[tr * ld + rc] = g;
            } else {
                const int rc = o / nz;
                bb[rc * ld + ((o % nz) ^ (rc & swz))] = g;
            }
        }
        __syncthreads();
        if (!active) continue;
        // row product acc += B[r][:] . u_col  (col component cc) ; or transposed
        int cc = -1;       // component of u for the row product
        int ct = -1;       // component of u for the transposed product (subtracted)
        switch (bi) {
        case 0: cc = (a == 0) ? 0 : -1; break;                           // XX
        case 1: cc = (a == 0) ? 1 : (a == 1) ? 0 : -1; break;            // XY
        case 2: cc = (a == 1) ? 1 : -1; break;                           // YY
        case 3: cc = (a == 2) ? 2 : -1; break;                           // ZZ
        case 4: cc = (a == 0) ? 2 : -1; ct = (a == 2) ? 0 : -1; break;   // XZ
        case 5: cc = (a == 1) ? 2 : -1; ct = (a == 2) ? 1 : -1; break;   // YZ
        }
        if (cc >= 0) {
            const cplx<T> *uc = uw + cc * nz;
            const cplx<T> *row = bw + r * ld;
            cplx<T> s0 = mk<T>(0, 0);
            for (int c = 0; c < nz; ++c) s0 = cfma<T>(s0, row[c], uc[c]);
            acc = cadd<T>(acc, s0);
        }
        if (ct >= 0) {
            const cplx<T> *uc = uw + ct * nz;
            cplx<T> s0 = mk<T>(0, 0);
            for (int m = 0; m < nz; ++m) s0 = cfma<T>(s0, bw[m * ld + r], uc[m]);
            acc = csub<T>(acc, s0);
        }
    }
    if (active) {
        const int64_t l = l0 + w;
        if (l < L) {
            if (fold_nx > 0 && q < 2 * nz) {
                const FoldPos p = fold_pos(l, fold_nx, fold_ny);
                if (q < nz ? p.mx : p.my) acc = mk<T>(-acc.x, -acc.y);
            }
            buf[rhs * M + l * C + q] = acc;
        }
    }
}

// ---- streaming contraction (nz = 32) ---------------------------------------------------------------
// Persistent: one 256-thread workgroup per CU walks wavenumbers l = blockIdx.x, += gridDim.x.
// Each wavenumber's whole Green block (4 packed + 2 swizzled asymmetric blocks, 4160 elements) and
// its spectrum columns are copied straight from HBM into LDS by global_load_lds_dwordx4 (64 lanes x
// 16 B = 1 KB per wave-load), into a ring of NBUF buffers: the copies of the next NBUF-1 wavenumbers
// are in flight while one is contracted, so the HBM stream does not wait for the arithmetic
// (complex128: 68 KB per wavenumber, 2 buffers; complex64: 34 KB, 4 buffers). The copies are issued
// from inline asm so that the only waits on them are the explicit vmcnt waits below: vector-memory
// operations of one wave complete in order, so with k wave-loads issued after those of wavenumber l,
// vmcnt(k) means l has landed.
// Contraction: wave w owns columns [8w, 8w+8); lane (s, r) takes row r and columns 8w + 4s + j
// (j < 4) of all six blocks, for all three components and both right-hand sides, with its u slice
// in registers (36 FMAs per 8 LDS reads). Partial rows are summed across s by a lane shuffle and
// across the four waves through LDS.
namespace stream {
constexpr int NZ = 32, C = 3 * NZ, S = NZ * (NZ + 1) / 2, A = NZ * NZ, GB = 4 * S + 2 * A;
constexpr int MASK = 15;                    // asym_swizzle_mask(32)
template <typename T> struct Cfg {
    static constexpr int E = (int)sizeof(cplx<T>);            // bytes per element
    static constexpr int EPL = 16 / E;                        // elements per lane per wave-load
    static constexpr int EPC = 64 * EPL;                      // elements per wave-load
    static constexpr int RAW = (GB + 4 * C + EPC - 1) / EPC;  // wave-loads for Green + 4 rhs columns
    static constexpr int NCHUNK = (RAW + 3) / 4 * 4;          // padded to the 4 waves
    static constexpr int PER_WAVE = NCHUNK / 4;
    static constexpr int BUF = NCHUNK * EPC;                  // elements per LDS buffer
    static constexpr int NBUF = E == 16 ? 2 : 4;
};
static_assert(GB % 2 == 0 && C % 2 == 0, "element pairs never straddle the Green/spectrum boundary");
static_assert(Cfg<double>::PER_WAVE * (Cfg<double>::NBUF - 1) <= 63, "vmcnt range");
static_assert(Cfg<float>::PER_WAVE * (Cfg<float>::NBUF - 1) <= 63, "vmcnt range");
static_assert(Cfg<double>::NBUF * Cfg<double>::BUF * 16 + 4 * 2 * C * 16 <= 160 * 1024, "LDS");
static_assert(Cfg<float>::NBUF * Cfg<float>::BUF * 8 + 4 * 2 * C * 8 <= 160 * 1024, "LDS");
constexpr int kMaxStreamRhs = 4;
}  // namespace stream

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// This wave's PER_WAVE wave-loads of wavenumber l (Green block and nrhs spectrum columns) into the
// LDS buffer at byte address dst.
template <typename T>
__device__ __forceinline__ void stream_issue(const cplx<T> *__restrict__ G, const cplx<T> *buf, int64_t M, int64_t l,
                                             int nrhs, unsigned dst, int wave, int lane)
{
    using namespace stream;
    using K = Cfg<T>;
#pragma unroll
    for (int t = 0; t < K::PER_WAVE; ++t) {
        const int k = wave + 4 * t;
        const int e = k * K::EPC + lane * K::EPL;                  // first element this lane copies
        const cplx<T> *src;
        if (e < GB) {
            src = G + l * GB + e;
        } else {
            int q = e - GB;                                         // spectrum column of this wavenumber
            if (q > nrhs * C - K::EPL) q = nrhs * C - K::EPL;       // padding lanes re-read valid data
            const int rhs = q / C;
            src = buf + rhs * M + l * C + (q - rhs * C);
        }
        const unsigned m0 = __builtin_amdgcn_readfirstlane(dst + (unsigned)k * 1024u);
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(m0), "v"(src) : "memory", "m0");
    }
}
#pragma clang diagnostic pop

// Right-hand sides h0 .. h0 + NRHS - 1 of the wavenumber in blk; partial rows into part [4][NRHS][C].
template <typename T, int NRHS>
__device__ __forceinline__ void stream_compute(const cplx<T> *__restrict__ blk, cplx<T> *__restrict__ part, int wave,
                                               int lane, int h0)
{
    using namespace stream;
    const cplx<T> *u = blk + GB + h0 * C;                        // [NRHS][C] of this pass
    const int s = lane >> 5, r = lane & 31, r15 = r & MASK;
    const int cb = wave * 8 + s * 4;
    const int trir = r * (r + 1) / 2;
    cplx<T> ux[NRHS][4], uy[NRHS][4], uz[NRHS][4];
#pragma unroll
    for (int h = 0; h < NRHS; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            ux[h][j] = u[h * C + cb + j];
            uy[h][j] = u[h * C + NZ + cb + j];
            uz[h][j] = u[h * C + 2 * NZ + cb + j];
        }
    cplx<T> yx[NRHS], yy[NRHS], yz[NRHS];
#pragma unroll
    for (int h = 0; h < NRHS; ++h) {
        yx[h] = mk<T>(0, 0);
        yy[h] = yx[h];
        yz[h] = yx[h];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int c = cb + j;
        const int pidx = c >= r ? r + c * (c + 1) / 2 : c + trir;    // packed (min, max)
        const cplx<T> gxx = blk[pidx], gxy = blk[S + pidx], gyy = blk[2 * S + pidx], gzz = blk[3 * S + pidx];
        const int ro = r * NZ + (c ^ r15), co = c * NZ + (r ^ (c & MASK));   // (r, c) and (c, r), swizzled
        const cplx<T> gxz = blk[4 * S + ro], gyz = blk[4 * S + A + ro];
        const cplx<T> gzx = blk[4 * S + co], gzy = blk[4 * S + A + co];
#pragma unroll
        for (int h = 0; h < NRHS; ++h) {
            yx[h] = cfma<T>(yx[h], gxx, ux[h][j]);
            yx[h] = cfma<T>(yx[h], gxy, uy[h][j]);
            yx[h] = cfma<T>(yx[h], gxz, uz[h][j]);
            yy[h] = cfma<T>(yy[h], gxy, ux[h][j]);
            yy[h] = cfma<T>(yy[h], gyy, uy[h][j]);
            yy[h] = cfma<T>(yy[h], gyz, uz[h][j]);
            yz[h] = cfms<T>(yz[h], gzx, ux[h][j]);             // -XZ^T u_x
            yz[h] = cfms<T>(yz[h], gzy, uy[h][j]);             // -YZ^T u_y
            yz[h] = cfma<T>(yz[h], gzz, uz[h][j]);
        }
    }
#pragma unroll
    for (int h = 0; h < NRHS; ++h) {
        yx[h].x += __shfl_xor(yx[h].x, 32, 64);
        yx[h].y += __shfl_xor(yx[h].y, 32, 64);
        yy[h].x += __shfl_xor(yy[h].x, 32, 64);
        yy[h].y += __shfl_xor(yy[h].y, 32, 64);
        yz[h].x += __shfl_xor(yz[h].x, 32, 64);
        yz[h].y += __shfl_xor(yz[h].y, 32, 64);
    }
    // both halves now hold the wave's row sums; half s stores right-hand side s
    if (NRHS == 1 && s) return;
    const int h = NRHS == 1 ? 0 : s;
    cplx<T> *pw = part + (wave * NRHS + h) * C;
    // component-wise selects (a select of whole vector values would go through scratch)
    const T vxx = h ? yx[NRHS - 1].x : yx[0].x, vxy = h ? yx[NRHS - 1].y : yx[0].y;
    const T vyx = h ? yy[NRHS - 1].x : yy[0].x, vyy = h ? yy[NRHS - 1].y : yy[0].y;
    const T vzx = h ? yz[NRHS - 1].x : yz[0].x, vzy = h ? yz[NRHS - 1].y : yz[0].y;
    pw[r] = mk<T>(vxx, vxy);
    pw[NZ + r] = mk<T>(vyx, vyy);
    pw[2 * NZ + r] = mk<T>(vzx, vzy);
}

// waits until at most `after` groups of PER_WAVE wave-loads are outstanding
template <int PW>
__device__ __forceinline__ void wait_groups(int after)
{
    switch (after) {
    case 0: wait_vm<0>(); break;
    case 1: wait_vm<PW>(); break;
    case 2: wait_vm<2 * PW>(); break;
    default: wait_vm<3 * PW>(); break;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void contract_stream_kernel(const cplx<T> *__restrict__ G, cplx<T> *buf, int64_t L,
                                                              int64_t M, int nrhs)
{
    using namespace stream;
    using K = Cfg<T>;
    static_assert(K::NBUF <= 4, "wait_groups covers up to three groups in flight after the current one");
    __shared__ cplx<T> ring[K::NBUF * K::BUF];
    __shared__ cplx<T> part[4 * 2 * C];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, t = threadIdx.x;
    const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) cplx<T> *)ring;
    const int64_t g = gridDim.x;                                 // the launch keeps gridDim.x <= L
    const int64_t l0 = blockIdx.x;
    const int64_t cnt = (L - 1 - l0) / g + 1;                    // wavenumbers of this workgroup
#pragma unroll
    for (int p = 0; p < K::NBUF - 1; ++p)
        if (p < cnt)
            stream_issue<T>(G, buf, M, l0 + p * g, nrhs, base + (unsigned)(p * K::BUF * K::E), wave, lane);
    for (int64_t i = 0; i < cnt; ++i) {
        const int64_t l = l0 + i * g;
        const int64_t ahead = i + K::NBUF - 1;                   // the wavenumber index to prefetch now
        if (ahead < cnt)
            stream_issue<T>(G, buf, M, l0 + ahead * g, nrhs, base + (unsigned)((ahead % K::NBUF) * K::BUF * K::E),
                            wave, lane);
        // groups issued after wavenumber i's: i+1 .. min(cnt-1, i+NBUF-1)
        const int64_t after = (cnt - 1 - i) < (K::NBUF - 1) ? (cnt - 1 - i) : (K::NBUF - 1);
        wait_groups<K::PER_WAVE>((int)after);
        const cplx<T> *blk = ring + (i % K::NBUF) * K::BUF;
        // right-hand sides in passes of two over the same LDS-resident Green block
        for (int h0 = 0; h0 < nrhs; h0 += 2) {
            const int nh = nrhs - h0 >= 2 ? 2 : 1;
            XTR_BARRIER();                                       // block in LDS / previous pass read
            if (nh == 2) stream_compute<T, 2>(blk, part, wave, lane, h0);
            else stream_compute<T, 1>(blk, part, wave, lane, h0);
            XTR_BARRIER();                                       // partials complete
            if (t < nh * C) {
                cplx<T> acc = part[t];
#pragma unroll
                for (int w = 1; w < 4; ++w) acc = cadd<T>(acc, part[w * nh * C + t]);
                const int h = h0 + t / C;
                buf[h * M + l * C + (t % C)] = acc;
            }
        }
    }
    wait_vm<0>();                                                // no copy may land after exit
}

// ---- streaming contraction, nz = 64 --------------------------------------------------------------------
// A wavenumber's Green block (264 KB in FP64, 132 KB in FP32) is streamed as four units through a
// ring of 72-wave-load slots: U0 = xx|xy (+ the right-hand sides' spectrum columns), U1 = yy|zz,
// U2 = xz, U3 = yz. The units of all the workgroup's wavenumbers form one stream: step s contracts
// unit s while units s+1 .. s+NSLOT-1 are in flight (FP64: 2 slots of 72 KB; FP32: 4 slots of 36 KB).
// Wave w owns columns [16w, 16w+16); lane (hc, r) owns rows r and r + 32 and columns 16w + 8hc + j
// (j < 8); accumulators persist across a wavenumber's four units. The spectrum columns are copied
// from U0's slot into a small LDS area that outlives the slot; partial rows are reduced in U3's slot.
namespace stream64 {
constexpr int NZ = 64, C = 3 * NZ, S = NZ * (NZ + 1) / 2, A = NZ * NZ, GB = 4 * S + 2 * A;
constexpr int MASK = 15;                  // asym_swizzle_mask(64)
constexpr int SLOT = 72 * 64;             // elements per slot: 72 wave-loads of 1 KB (FP64), 36 (FP32)
constexpr int MAXRHS = 2;
__host__ __device__ constexpr int ubegin(int u) { return u == 0 ? 0 : u == 1 ? 2 * S : u == 2 ? 4 * S : 4 * S + A; }
__host__ __device__ constexpr int ulen(int u) { return u < 2 ? 2 * S : A; }
__host__ __device__ constexpr int uimage(int u) { return u == 0 ? 2 * S + MAXRHS * C : ulen(u); }
template <typename T>
struct Cfg {
    static constexpr int E = (int)sizeof(cplx<T>);   // bytes per element
    static constexpr int EPL = 16 / E;               // elements per lane and wave-load
    static constexpr int EPC = 64 * EPL;             // elements per wave-load
    static constexpr int NSLOT = E == 16 ? 2 : 4;
    __host__ __device__ static constexpr int upw(int u) { return ((uimage(u) + EPC - 1) / EPC + 3) / 4; }
    // wave-loads a wave has issued after unit u's when step u waits (`last`: no next wavenumber)
    __host__ __device__ static constexpr int ahead(int u, bool last)
    {
        int n = 0;
        for (int k = 1; k < NSLOT; ++k) {
            if (last && u + k > 3) break;
            n += upw((u + k) % 4);
        }
        return n;
    }
};
static_assert(4 * Cfg<double>::upw(0) * Cfg<double>::EPC <= SLOT && 4 * Cfg<float>::upw(0) * Cfg<float>::EPC <= SLOT,
              "slot size");
static_assert(2 * SLOT * 16 + MAXRHS * C * 16 <= 160 * 1024 && 4 * SLOT * 8 + MAXRHS * C * 8 <= 160 * 1024, "LDS");
static_assert(Cfg<double>::ahead(0, false) < 64 && Cfg<float>::ahead(0, false) < 64, "vmcnt range");
}  // namespace stream64

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <typename T, int U>
__device__ __forceinline__ void s64_issue(const cplx<T> *__restrict__ G, const cplx<T> *buf, int64_t M, int64_t l,
                                          int nrhs, unsigned dst, int wave, int lane)
{
    using namespace stream64;
    using K = Cfg<T>;
#pragma unroll
    for (int t = 0; t < K::upw(U); ++t) {
        const int k = wave + 4 * t;
        const int e = k * K::EPC + lane * K::EPL;        // first element of this unit's LDS image this lane copies
        const cplx<T> *src;
        if (e < ulen(U)) {
            src = G + l * GB + ubegin(U) + e;
        } else if (U == 0) {
            int q = e - ulen(0);                         // spectrum column q of this wavenumber
            if (q > nrhs * C - K::EPL) q = nrhs * C - K::EPL;   // padding lanes re-read valid data
            const int rhs = q / C;
            src = buf + rhs * M + l * C + (q - rhs * C);
        } else {
            src = G + l * GB + ubegin(U) + ulen(U) - K::EPL;     // padding lanes re-read valid data
        }
        const unsigned m0 = __builtin_amdgcn_readfirstlane(dst + (unsigned)k * 1024u);
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(m0), "v"(src) : "memory", "m0");
    }
}
#pragma clang diagnostic pop

template <typename T, int U, int NRHS>
__device__ __forceinline__ void s64_compute(const cplx<T> *__restrict__ blk, const cplx<T> *__restrict__ ua, int wave,
                                            int lane, cplx<T> (&yx)[2][NRHS], cplx<T> (&yy)[2][NRHS],
                                            cplx<T> (&yz)[2][NRHS])
{
    using namespace stream64;
    const int hc = lane >> 5, r0 = lane & 31;
    const int cb = wave * 16 + hc * 8;
#pragma unroll 2
    for (int j = 0; j < 8; ++j) {
        const int c = cb + j;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = r0 + 32 * q;
            cplx<T> g0, g1;
            if (U < 2) {
                const int p = c >= r ? r + c * (c + 1) / 2 : c + r * (r + 1) / 2;   // packed (min, max)
                g0 = blk[p];
                g1 = blk[S + p];
            } else {
                g0 = blk[r * NZ + (c ^ (r & MASK))];       // B(r, c)
                g1 = blk[c * NZ + (r ^ (c & MASK))];       // B(c, r)
            }
#pragma unroll
            for (int h = 0; h < NRHS; ++h) {
                const cplx<T> *u = ua + h * C;
                if (U == 0) {          // xx, xy
                    const cplx<T> ux = u[c], uy = u[NZ + c];
                    yx[q][h] = cfma<T>(cfma<T>(yx[q][h], g0, ux), g1, uy);
                    yy[q][h] = cfma<T>(yy[q][h], g1, ux);
                } else if (U == 1) {   // yy, zz
                    yy[q][h] = cfma<T>(yy[q][h], g0, u[NZ + c]);
                    yz[q][h] = cfma<T>(yz[q][h], g1, u[2 * NZ + c]);
                } else if (U == 2) {   // xz: row product, then -xz^T
                    yx[q][h] = cfma<T>(yx[q][h], g0, u[2 * NZ + c]);
                    yz[q][h] = cfms<T>(yz[q][h], g1, u[c]);
                } else {               // yz: row product, then -yz^T
                    yy[q][h] = cfma<T>(yy[q][h], g0, u[2 * NZ + c]);
                    yz[q][h] = cfms<T>(yz[q][h], g1, u[NZ + c]);
                }
            }
        }
    }
}

// One step of the unit stream: contract unit U of wavenumber l (slot U % NSLOT) after issuing unit
// U + NSLOT - 1 into the slot the previous step freed.
template <typename T, int NRHS, int U>
__device__ __forceinline__ void s64_step(const cplx<T> *__restrict__ G, cplx<T> *buf, int64_t M, int64_t l,
                                         int64_t lnext, bool has_next, cplx<T> *ring, cplx<T> *ua, unsigned base,
                                         int wave, int lane, int t, cplx<T> (&yx)[2][NRHS], cplx<T> (&yy)[2][NRHS],
                                         cplx<T> (&yz)[2][NRHS])
{
    using namespace stream64;
    using K = Cfg<T>;
    constexpr int V = U + K::NSLOT - 1;                 // unit issued now
    constexpr unsigned vdst = (unsigned)((V % K::NSLOT) * SLOT * K::E);
    if (V <= 3) s64_issue<T, V % 4>(G, buf, M, l, NRHS, base + vdst, wave, lane);
    else if (has_next) s64_issue<T, V % 4>(G, buf, M, lnext, NRHS, base + vdst, wave, lane);
    if (has_next) wait_vm<K::ahead(U, false)>();
    else wait_vm<K::ahead(U, true)>();
    XTR_BARRIER();                                      // unit U in LDS for every wave
    cplx<T> *blk = ring + (U % K::NSLOT) * SLOT;
    if (U == 0) {
        for (int o = t; o < NRHS * C; o += 256) ua[o] = blk[ulen(0) + o];   // spectrum columns -> u area
        XTR_BARRIER();
    }
    s64_compute<T, U, NRHS>(blk, ua, wave, lane, yx, yy, yz);
    if (U == 3) {
        // rows r0 and r0 + 32 summed over the lane halves, then over the waves in this slot
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int h = 0; h < NRHS; ++h) {
                yx[q][h].x += __shfl_xor(yx[q][h].x, 32, 64);
                yx[q][h].y += __shfl_xor(yx[q][h].y, 32, 64);
                yy[q][h].x += __shfl_xor(yy[q][h].x, 32, 64);
                yy[q][h].y += __shfl_xor(yy[q][h].y, 32, 64);
                yz[q][h].x += __shfl_xor(yz[q][h].x, 32, 64);
                yz[q][h].y += __shfl_xor(yz[q][h].y, 32, 64);
            }
        XTR_BARRIER();                                  // slot read by every wave
        cplx<T> *part = blk;                            // [4][NRHS][C]
        const int hc = lane >> 5, r = (lane & 31) + 32 * hc;   // half hc stores row r0 + 32 hc
#pragma unroll
        for (int h = 0; h < NRHS; ++h) {
            cplx<T> *pw = part + (wave * NRHS + h) * C;
            // component-wise selects (a select of whole vector values would go through scratch)
            pw[r] = mk<T>(hc ? yx[1][h].x : yx[0][h].x, hc ? yx[1][h].y : yx[0][h].y);
            pw[NZ + r] = mk<T>(hc ? yy[1][h].x : yy[0][h].x, hc ? yy[1][h].y : yy[0][h].y);
            pw[2 * NZ + r] = mk<T>(hc ? yz[1][h].x : yz[0][h].x, hc ? yz[1][h].y : yz[0][h].y);
        }
        XTR_BARRIER();
        for (int o = t; o < NRHS * C; o += 256) {
            const int h = o / C, qq = o % C;
            cplx<T> acc = part[h * C + qq];
#pragma unroll
            for (int w = 1; w < 4; ++w) acc = cadd<T>(acc, part[(w * NRHS + h) * C + qq]);
            buf[h * M + l * C + qq] = acc;
        }
    }
    XTR_BARRIER();                                      // slot free for the next step's copy
}

template <typename T, int NRHS>
__global__ __launch_bounds__(256) void contract_stream64_kernel(const cplx<T> *__restrict__ G, cplx<T> *buf,
                                                                int64_t L, int64_t M)
{
    using namespace stream64;
    using K = Cfg<T>;
    __shared__ cplx<T> ring[K::NSLOT * SLOT];
    __shared__ cplx<T> ua[MAXRHS * C];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, t = threadIdx.x;
    const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) cplx<T> *)ring;
    const int64_t g = gridDim.x;                                 // the launch keeps gridDim.x <= L
    const int64_t l0 = blockIdx.x;
    const int64_t cnt = (L - 1 - l0) / g + 1;
    // units 0 .. NSLOT-2 of the first wavenumber (NSLOT - 1 <= 3)
    s64_issue<T, 0>(G, buf, M, l0, NRHS, base, wave, lane);
    if (K::NSLOT > 2) {
        s64_issue<T, 1>(G, buf, M, l0, NRHS, base + (unsigned)(SLOT * K::E), wave, lane);
        s64_issue<T, 2>(G, buf, M, l0, NRHS, base + (unsigned)(2 * SLOT * K::E), wave, lane);
    }
    for (int64_t i = 0; i < cnt; ++i) {
        const int64_t l = l0 + i * g, ln = l + g;
        const bool nx = i + 1 < cnt;
        cplx<T> yx[2][NRHS], yy[2][NRHS], yz[2][NRHS];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int h = 0; h < NRHS; ++h) {
                yx[q][h] = mk<T>(0, 0);
                yy[q][h] = yx[q][h];
                yz[q][h] = yx[q][h];
            }
        s64_step<T, NRHS, 0>(G, buf, M, l, ln, nx, ring, ua, base, wave, lane, t, yx, yy, yz);
        s64_step<T, NRHS, 1>(G, buf, M, l, ln, nx, ring, ua, base, wave, lane, t, yx, yy, yz);
        s64_step<T, NRHS, 2>(G, buf, M, l, ln, nx, ring, ua, base, wave, lane, t, yx, yy, yz);
        s64_step<T, NRHS, 3>(G, buf, M, l, ln, nx, ring, ua, base, wave, lane, t, yx, yy, yz);
    }
    wait_vm<0>();                                                // no copy may land after exit
}

static bool contract_stream64(const ApplyArgs &a, hipStream_t s);

// XTR_CONTRACT_KERNEL=generic selects contract_kernel for every shape (to compare the two kernels).
static bool contract_force_generic()
{
    const char *e = std::getenv("XTR_CONTRACT_KERNEL");
    return e && std::strcmp(e, "generic") == 0;
}

int device_cus()
{
    static int cus[64] = {0};
    int dev = 0;
    XTR_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) throw hip_error("device index out of range");
    if (!cus[dev]) XTR_CHECK(hipDeviceGetAttribute(&cus[dev], hipDeviceAttributeMultiprocessorCount, dev));
    return cus[dev];
}

// nz = 64, one or two right-hand sides, FP64 or FP32
template <typename T>
static void launch_stream64(const ApplyArgs &a, unsigned grid, hipStream_t s)
{
    const int64_t L = a.g.L();
    if (a.nrhs == 2)
        hipLaunchKernelGGL((contract_stream64_kernel<T, 2>), dim3(grid), dim3(256), 0, s, (const cplx<T> *)a.G,
                           (cplx<T> *)a.buf, L, a.g.M());
    else
        hipLaunchKernelGGL((contract_stream64_kernel<T, 1>), dim3(grid), dim3(256), 0, s, (const cplx<T> *)a.G,
                           (cplx<T> *)a.buf, L, a.g.M());
}

static bool contract_stream64(const ApplyArgs &a, hipStream_t s)
{
    if (a.g.nz != stream64::NZ || (a.nrhs != 1 && a.nrhs != 2) || contract_force_generic()) return false;
    const unsigned grid = (unsigned)std::min<int64_t>(a.g.L(), device_cus());
    if (a.precision == 0) launch_stream64<double>(a, grid, s);
    else launch_stream64<float>(a, grid, s);
    XTR_LAUNCH_CHECK("contract_stream64_kernel");
    note_contract(a, "contract_stream64_kernel", 0, a.nrhs);
    return true;
}

// The streaming kernel covers nz = 32 with one to four right-hand sides; other shapes use contract_kernel.
template <typename T>
static bool contract_stream(const ApplyArgs &a, hipStream_t s)
{
    if (a.g.nz != stream::NZ || a.nrhs < 1 || a.nrhs > stream::kMaxStreamRhs || contract_force_generic()) return false;
    const int64_t L = a.g.L();
    const unsigned grid = (unsigned)std::min<int64_t>(L, device_cus());
    hipLaunchKernelGGL((contract_stream_kernel<T>), dim3(grid), dim3(256), 0, s, (const cplx<T> *)a.G,
                       (cplx<T> *)a.buf, L, a.g.M(), a.nrhs);
    XTR_LAUNCH_CHECK("contract_stream_kernel");
    note_contract(a, "contract_stream_kernel");
    return true;
}

// ---- folded contraction on MFMA, nz = 64 -------------------------------------------------------------
// A folded block (264 KB in FP64, 132 KB in FP32) is streamed through LDS in units, through a ring of
// four slots of 33 wave-loads (33 KB) with three units in flight. FP64: nine units (the spectrum
// columns of the block's images, xx, xy, yy, zz, and the xz and yz blocks each as a diagonal and an
// off-diagonal pair of 32 x 32 quadrants); FP32: five (the spectrum, xx + xy, yy + zz, xz, yz: each
// a contiguous run of the block). Wave w = 4 g + t owns rows 16t..16t+15 of x, y and z and the k-half
// g (k in 32g..32g+31 of every input component); waves t and 4 + t add their partial sums at the end
// of the block. The spectrum unit is read once per block into registers: lane (kl, n) keeps B[k][n]
// of its 24 k-steps, B = [Re U | Im U] with the image's mirror signs applied. Two accumulators per
// tile, D1 = Re G . B and D2 = Im G . B, give Re Y = D1[:, :8] - D2[:, 8:] and Im Y = D1[:, 8:] +
// D2[:, :8] through one lane exchange at the end; xy's A values serve both of its products. The
// -xz^T, -yz^T blocks enter through the FP64 MFMA's negate modifier (FP32: negated values). In FP64 a
// quadrant pair holds the quadrants (row half h, column half h) (diagonal unit) or (h, 1 - h); the
// direct and the transposed product of wave (t, g) both need the quadrant (t / 2, g) or (g, t / 2),
// so each quadrant unit is contracted by the four waves with g == t / 2 (diagonal) or g != t / 2, one
// per SIMD. In FP32 every wave works on every unit.
namespace fold64 {
constexpr int NZ = 64, C = 3 * NZ, S = NZ * (NZ + 1) / 2, A = NZ * NZ, GB = 4 * S + 2 * A;
constexpr int MASK = 15;                  // asym_swizzle_mask(64)
constexpr int NCOL = 8, UCOLS = NCOL * C;
constexpr int NWAVE = 8, NTHR = 64 * NWAVE;
constexpr int KS = 8;                     // k-steps of one component's k-half (32 values, 4 per step)
constexpr int NSLOT = 4;
template <typename T>
struct Cfg {
    static constexpr bool WIDE = sizeof(T) == 4;            // FP32: whole xz, yz blocks in one slot
    static constexpr int NUNIT = WIDE ? 5 : 9;
    static constexpr int E = (int)sizeof(cplx<T>);
    static constexpr int EPL = 16 / E;
    static constexpr int EPC = 64 * EPL;
    __host__ __device__ static constexpr int uelems(int u)
    {
        return u == 0 ? UCOLS : WIDE ? (u <= 2 ? 2 * S : A) : (u <= 4 ? S : A / 2);
    }
    __host__ __device__ static constexpr int nw(int u) { return (uelems(u) + EPC - 1) / EPC; }
    static constexpr int SLOTW = 33;                        // the largest unit, in wave-loads
    static constexpr int SLOT = SLOTW * EPC;
    static constexpr int EXCH = 4 * 3 * 64;                 // exchange: [t][tile][lane] of 4 T
    // wave-loads of unit u issued by wave w
    __host__ __device__ static constexpr int cnt(int u, int w) { return (nw(u) - w + NWAVE - 1) / NWAVE; }
    // wave-loads a wave has issued after unit u's when step u waits (units u+1 .. u+NSLOT-2: unit
    // u+NSLOT-1 goes out after that step's barrier)
    __host__ __device__ static constexpr int ahead(int u, bool has_next, int w)
    {
        int n = 0;
        for (int k = 1; k < NSLOT - 1; ++k)
            if (u + k < NUNIT || has_next) n += cnt((u + k) % NUNIT, w);
        return n;
    }
    __host__ __device__ static constexpr bool fits()
    {
        for (int u = 0; u < NUNIT; ++u)
            if (nw(u) > SLOTW) return false;
        return true;
    }
};
static_assert(Cfg<double>::fits() && Cfg<float>::fits(), "every unit fits a slot");
static_assert(NSLOT * Cfg<double>::SLOT * 16 + Cfg<double>::EXCH * 4 * 8 <= 160 * 1024, "LDS (FP64)");
static_assert(NSLOT * Cfg<float>::SLOT * 8 + Cfg<float>::EXCH * 4 * 4 <= 160 * 1024, "LDS (FP32)");
static_assert(Cfg<double>::ahead(0, true, 0) < 64 && Cfg<float>::ahead(0, true, 0) < 64, "vmcnt range");
static_assert(NSLOT - 1 < Cfg<double>::NUNIT && NSLOT - 1 < Cfg<float>::NUNIT, "look-ahead within one block");
static_assert(S % 2 == 0 && C % 2 == 0, "two-element lanes stay inside one run");
static_assert(Cfg<double>::nw(0) * Cfg<double>::EPC == UCOLS && Cfg<float>::nw(0) * Cfg<float>::EPC == UCOLS,
              "the spectrum unit has no padding lanes");
}  // namespace fold64

// Step U's wait: wave w lets through the wave-loads it issued after unit U's (counts differ by wave;
// `wave` is uniform, so the dispatch is scalar).
template <typename T, int U, bool HN, int W = 0>
__device__ __forceinline__ void fold64_wait_wave(int wave)
{
    if constexpr (W < fold64::NWAVE) {
        if (wave == W) wait_vm<fold64::Cfg<T>::ahead(U, HN, W)>();
        else fold64_wait_wave<T, U, HN, W + 1>(wave);
    }
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// Copy of unit UT of block b into the slot at LDS address dst. In the spectrum unit, column q's
// element kk sits at position (kk + 2q) mod C, which spreads the columns over the LDS banks for the
// B reads.
template <typename T, int UT>
__device__ __forceinline__ void fold64_issue(const cplx<T> *__restrict__ G, const cplx<T> *buf, int64_t M, int64_t b,
                                             const FoldImages &im, int nrhs, unsigned dst, int wave, int lane)
{
    using namespace fold64;
    using K = Cfg<T>;
    constexpr int NWU = K::nw(UT);
#pragma unroll
    for (int t = 0; t < (NWU + NWAVE - 1) / NWAVE; ++t) {
        const int k = __builtin_amdgcn_readfirstlane(wave + NWAVE * t);
        if (k >= NWU) break;
        const int e = k * K::EPC + lane * K::EPL;
        const cplx<T> *src;
        if constexpr (UT == 0) {
            int q = e / C, j = e - q * C;
            if (q >= im.n * nrhs) q = j = 0;                 // unused column: valid data
            int kk = j - 2 * q;                              // even, so a lane's two FP32 elements
            if (kk < 0) kk += C;                             // stay contiguous
            const int img = q / nrhs, h = q - img * nrhs;
            src = buf + h * M + im.l(img) * C + kk;
        } else if constexpr (K::WIDE) {
            // contiguous runs: xx + xy, yy + zz (2S elements), xz, yz (A)
            constexpr int base = UT == 1 ? 0 : UT == 2 ? 2 * S : UT == 3 ? 4 * S : 4 * S + A;
            constexpr int len = K::uelems(UT);
            src = G + b * GB + base + (e < len ? e : len - K::EPL);   // padding lanes re-read
        } else if constexpr (UT <= 4) {
            src = G + b * GB + (UT - 1) * S + (e < S ? e : S - K::EPL);   // padding lanes re-read
        } else {
            // quadrant pair: rows 0-31 with column half H0, rows 32-63 with half 1 - H0 (diag: H0 = 0,
            // rows 32-63 with half 1; off: the other halves); 32 elements per quadrant row
            constexpr int base = UT <= 6 ? 4 * S : 4 * S + A;
            constexpr bool diag = UT == 5 || UT == 7;
            const int qd = e >> 10, w = e & 1023;
            const int rc = qd * 32 + (w >> 5), half = diag ? qd : 1 - qd;
            src = G + b * GB + base + rc * NZ + 32 * half + (w & 31);
        }
        const unsigned m0 = __builtin_amdgcn_readfirstlane(dst + (unsigned)k * 1024u);
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(m0), "v"(src) : "memory", "m0");
    }
}
#pragma clang diagnostic pop

// Per-lane byte offsets of the A values of k-step s (k = 32 g + 4 s + kl, local to the component)
// for row r = 16 t + i, within a slot: the packed symmetric layout (po), and the direct (row r,
// column k: qo) and the transposed (row k, column r: to) element of an xz or yz block, as a
// quadrant pair (FP64) or the whole swizzled block (FP32). They depend only on the lane and the
// wave, so each wave computes them once.
template <typename T>
__device__ __forceinline__ void fold64_offsets(int t, int g, int lane, unsigned (&po)[fold64::KS],
                                               unsigned (&qo)[fold64::KS], unsigned (&to)[fold64::KS])
{
    using namespace fold64;
    constexpr unsigned E = sizeof(cplx<T>);
    const int r = 16 * t + (lane & 15), kl = lane >> 4;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int c = 32 * g + 4 * s + kl, cq = 4 * s + kl;  // cq = c & 31
        po[s] = E * (unsigned)(c >= r ? r + c * (c + 1) / 2 : c + r * (r + 1) / 2);
        if constexpr (Cfg<T>::WIDE) {
            qo[s] = E * (unsigned)(r * NZ + (c ^ (r & MASK)));
            to[s] = E * (unsigned)(c * NZ + (r ^ (c & MASK)));
        } else {
            qo[s] = E * (unsigned)((r >> 5) * 1024 + (r & 31) * 32 + (cq ^ (r & MASK)));
            to[s] = E * (unsigned)(g * 1024 + cq * 32 + ((r & 31) ^ (cq & MASK)));
        }
    }
}

// D1 += (NEG ? -Re a : Re a) b, D2 += (NEG ? -Im a : Im a) b over the 8 k-steps of one A tile at byte
// offset OFF + off[s] of the slot.
template <typename T, bool NEG, unsigned OFF = 0>
__device__ __forceinline__ void fold64_job(const cplx<T> *__restrict__ blk, const unsigned (&off)[fold64::KS],
                                           const T (&b)[fold64::KS], typename MfmaAcc<T>::type &d1,
                                           typename MfmaAcc<T>::type &d2)
{
    cplx<T> a[fold64::KS];
#pragma unroll
    for (int s = 0; s < fold64::KS; ++s) a[s] = lds_cplx<T>(blk, OFF + off[s]);
#pragma unroll
    for (int s = 0; s < fold64::KS; ++s) {
        d1 = mfma16s<NEG>(a[s].x, b[s], d1);
        d2 = mfma16s<NEG>(a[s].y, b[s], d2);
    }
}

// xy . u_y -> y_x and xy . u_x -> y_y from the same A values (xy at byte offset OFF of the slot).
template <typename T, unsigned OFF>
__device__ __forceinline__ void fold64_xy(const cplx<T> *__restrict__ blk, const unsigned (&po)[fold64::KS],
                                          const T (&bf)[3][fold64::KS], typename MfmaAcc<T>::type (&d1)[3],
                                          typename MfmaAcc<T>::type (&d2)[3])
{
    cplx<T> a[fold64::KS];
#pragma unroll
    for (int s = 0; s < fold64::KS; ++s) a[s] = lds_cplx<T>(blk, OFF + po[s]);
#pragma unroll
    for (int s = 0; s < fold64::KS; ++s) {
        d1[0] = mfma16s<false>(a[s].x, bf[1][s], d1[0]);
        d2[0] = mfma16s<false>(a[s].y, bf[1][s], d2[0]);
        d1[1] = mfma16s<false>(a[s].x, bf[0][s], d1[1]);
        d2[1] = mfma16s<false>(a[s].y, bf[0][s], d2[1]);
    }
}

// The MFMAs of unit UT for wave (t, g).
template <typename T, int UT>
__device__ __forceinline__ void fold64_compute(const cplx<T> *__restrict__ blk, const T (&bf)[3][fold64::KS],
                                               const unsigned (&po)[fold64::KS], const unsigned (&qo)[fold64::KS],
                                               const unsigned (&to)[fold64::KS], int t, int g,
                                               typename MfmaAcc<T>::type (&d1)[3], typename MfmaAcc<T>::type (&d2)[3])
{
    using namespace fold64;
    constexpr unsigned SB = (unsigned)S * sizeof(cplx<T>);     // bytes of one packed block
    if constexpr (Cfg<T>::WIDE) {
        if constexpr (UT == 1) {
            fold64_job<T, false>(blk, po, bf[0], d1[0], d2[0]);      // xx . u_x -> y_x
            fold64_xy<T, SB>(blk, po, bf, d1, d2);
        } else if constexpr (UT == 2) {
            fold64_job<T, false>(blk, po, bf[1], d1[1], d2[1]);      // yy . u_y -> y_y
            fold64_job<T, false, SB>(blk, po, bf[2], d1[2], d2[2]);  // zz . u_z -> y_z
        } else {
            constexpr int o = UT == 3 ? 0 : 1;                       // xz (x) or yz (y)
            fold64_job<T, false>(blk, qo, bf[2], d1[o], d2[o]);      // xz . u_z -> y_x
            fold64_job<T, true>(blk, to, bf[o], d1[2], d2[2]);       // -xz^T . u_x -> y_z
        }
    } else if constexpr (UT == 1) {
        fold64_job<T, false>(blk, po, bf[0], d1[0], d2[0]);
    } else if constexpr (UT == 2) {
        fold64_xy<T, 0>(blk, po, bf, d1, d2);
    } else if constexpr (UT == 3) {
        fold64_job<T, false>(blk, po, bf[1], d1[1], d2[1]);
    } else if constexpr (UT == 4) {
        fold64_job<T, false>(blk, po, bf[2], d1[2], d2[2]);
    } else {
        constexpr int o = UT <= 6 ? 0 : 1;
        constexpr bool diag = UT == 5 || UT == 7;
        if ((g == (t >> 1)) == diag) {
            fold64_job<T, false>(blk, qo, bf[2], d1[o], d2[o]);
            fold64_job<T, true>(blk, to, bf[o], d1[2], d2[2]);
        }
    }
}

// One step of the unit stream: wait for unit U of block b (slot s % NSLOT); after the barrier every
// wave is done with the previous step's slot, so unit U + NSLOT - 1 is copied into it; then contract
// (unit 0: read this wave's B values).
template <typename T, int U>
__device__ __forceinline__ void fold64_step(const cplx<T> *__restrict__ G, cplx<T> *buf, int64_t M, int64_t b,
                                            int64_t bn, bool has_next, const FoldImages &im, const FoldImages &imn,
                                            int nrhs, int64_t s, cplx<T> *ring, unsigned base, int wave, int lane,
                                            T (&bf)[3][fold64::KS], const unsigned (&po)[fold64::KS],
                                            const unsigned (&qo)[fold64::KS], const unsigned (&to)[fold64::KS],
                                            typename MfmaAcc<T>::type (&d1)[3], typename MfmaAcc<T>::type (&d2)[3])
{
    using namespace fold64;
    using K = Cfg<T>;
    if (has_next) fold64_wait_wave<T, U, true>(wave);
    else fold64_wait_wave<T, U, false>(wave);
    XTR_BARRIER();                                         // unit U in LDS; previous slot's reads done
    constexpr int V = U + NSLOT - 1;                       // unit copied now, into the previous step's slot
    const unsigned vdst = base + (unsigned)(((s + NSLOT - 1) % NSLOT) * K::SLOT * K::E);
    if constexpr (V < K::NUNIT) fold64_issue<T, V>(G, buf, M, b, im, nrhs, vdst, wave, lane);
    else if (has_next) fold64_issue<T, V - K::NUNIT>(G, buf, M, bn, imn, nrhs, vdst, wave, lane);
    const cplx<T> *blk = ring + (s % NSLOT) * K::SLOT;
    const int t = wave & 3, g = wave >> 2;
    if constexpr (U == 0) {
        // lane (kl, n): B[k][n] for k = 64 ci + 32 g + 4 s + kl, column q = n % 8, Re (n < 8) or Im
        const int n = lane & 15, q = n & 7, part = n >> 3, kl = lane >> 4;
        const int img = (q / nrhs) & 3;
        const bool fx = im.mx(img) != 0, fy = im.my(img) != 0;
        const T *ucol = reinterpret_cast<const T *>(blk + q * C) + part;
#pragma unroll
        for (int ci = 0; ci < 3; ++ci)
#pragma unroll
            for (int st = 0; st < KS; ++st) {
                int j = 64 * ci + 32 * g + 4 * st + kl + 2 * q;
                if (j >= C) j -= C;
                const T v = ucol[2 * j];
                const bool flip = (ci == 0 && fx) || (ci == 1 && fy);
                bf[ci][st] = flip ? -v : v;
            }
    } else {
        fold64_compute<T, U>(blk, bf, po, qo, to, t, g, d1, d2);
    }
}

// Tile of rows 16t.. from D1 and D2 (the Re/Im exchange between lanes n and n ^ 8).
template <typename T>
__device__ __forceinline__ typename MfmaAcc<T>::type fold64_combine(typename MfmaAcc<T>::type d1,
                                                                   typename MfmaAcc<T>::type d2, int lane)
{
    const int part = (lane >> 3) & 1;
    typename MfmaAcc<T>::type y;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const T other = __shfl_xor(d2[r], 8, 64);
        y[r] = part ? d1[r] + other : d1[r] - other;
    }
    return y;
}

template <typename T, int O>
__device__ __forceinline__ void fold64_store(typename MfmaAcc<T>::type y, cplx<T> *buf, int64_t M,
                                             const FoldImages &im, int nrhs, int t, int lane)
{
    using namespace fold64;
    const int n = lane & 15, q = n & 7, part = n >> 3;
    const int img = (q / nrhs) & 3, h = q % nrhs;
    const bool live = q < im.n * nrhs;
    const bool flip = (O == 0 && im.mx(img)) || (O == 1 && im.my(img));
    T *dst = reinterpret_cast<T *>(buf + h * M + im.l(img) * C + O * NZ) + part;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int rr = 16 * t + mfma_row<T>(lane, r);
        const T v = flip ? -y[r] : y[r];
        if (live) dst[2 * rr] = v;
    }
}

// All the block's steps, 0 .. NUNIT - 1.
template <typename T, int... Us>
__device__ __forceinline__ void fold64_block(std::integer_sequence<int, Us...>, const cplx<T> *__restrict__ G,
                                             cplx<T> *buf, int64_t M, int64_t b, int64_t bn, bool hn,
                                             const FoldImages &im, const FoldImages &imn, int nrhs, int64_t s,
                                             cplx<T> *ring, unsigned base, int wave, int lane,
                                             T (&bf)[3][fold64::KS], const unsigned (&po)[fold64::KS],
                                             const unsigned (&qo)[fold64::KS], const unsigned (&to)[fold64::KS],
                                             typename MfmaAcc<T>::type (&d1)[3], typename MfmaAcc<T>::type (&d2)[3])
{
    (fold64_step<T, Us>(G, buf, M, b, bn, hn, im, imn, nrhs, s + Us, ring, base, wave, lane, bf, po, qo, to, d1, d2),
     ...);
}

template <typename T>
__global__ __launch_bounds__(fold64::NTHR) void contract_fold64_kernel(const cplx<T> *__restrict__ G, cplx<T> *buf, int64_t Lq,
                                                              int64_t M, int nrhs, int nx, int ny)
{
    using namespace fold64;
    using K = Cfg<T>;
    using acc_t = typename MfmaAcc<T>::type;
    __shared__ cplx<T> ring[NSLOT * K::SLOT];
    __shared__ acc_t exch[K::EXCH];                              // [t][tile][lane]: waves 4..7 -> 0..3
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int t = wave & 3, g = wave >> 2;
    const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) cplx<T> *)ring;
    const int64_t gs = gridDim.x;                                // the launch keeps gridDim.x <= Lq
    const int64_t b0 = blockIdx.x;
    const int64_t cnt = (Lq - 1 - b0) / gs + 1;
    unsigned po[KS], qo[KS], to[KS];
    fold64_offsets<T>(t, g, lane, po, qo, to);
    {
        // units 0 .. NSLOT-2 of the first block into slots 0 .. NSLOT-2
        const FoldImages im0 = fold_images(b0, nx, ny);
        fold64_issue<T, 0>(G, buf, M, b0, im0, nrhs, base, wave, lane);
        fold64_issue<T, 1>(G, buf, M, b0, im0, nrhs, base + 1u * K::SLOT * K::E, wave, lane);
        fold64_issue<T, 2>(G, buf, M, b0, im0, nrhs, base + 2u * K::SLOT * K::E, wave, lane);
    }
    static_assert(NSLOT == 4, "the prologue issues units 0 .. 2");
    T bf[3][KS];
    for (int64_t i = 0; i < cnt; ++i) {
        const int64_t b = b0 + i * gs, bn = b + gs;
        const bool hn = i + 1 < cnt;
        const FoldImages im = fold_images(b, nx, ny);
        const FoldImages imn = fold_images(hn ? bn : b, nx, ny);
        acc_t d1[3], d2[3];
#pragma unroll
        for (int o = 0; o < 3; ++o) d1[o] = d2[o] = acc_t{0, 0, 0, 0};
        fold64_block<T>(std::make_integer_sequence<int, K::NUNIT>{}, G, buf, M, b, bn, hn, im, imn, nrhs,
                        i * K::NUNIT, ring, base, wave, lane, bf, po, qo, to, d1, d2);
        acc_t y[3];
#pragma unroll
        for (int o = 0; o < 3; ++o) y[o] = fold64_combine<T>(d1[o], d2[o], lane);
        // waves 4..7 hand their partial sums to waves 0..3; the exchange area was last read before
        // this block's first barrier
        if (g == 1)
#pragma unroll
            for (int o = 0; o < 3; ++o) exch[(t * 3 + o) * 64 + lane] = y[o];
        XTR_BARRIER();
        if (g == 0) {
#pragma unroll
            for (int o = 0; o < 3; ++o) y[o] += exch[(t * 3 + o) * 64 + lane];
            fold64_store<T, 0>(y[0], buf, M, im, nrhs, t, lane);
            fold64_store<T, 1>(y[1], buf, M, im, nrhs, t, lane);
            fold64_store<T, 2>(y[2], buf, M, im, nrhs, t, lane);
        }
    }
    wait_vm<0>();                                                // no copy may land after exit
}

// Folded tensor, nz = 64: right-hand sides in launches of up to two.
static bool contract_fold64(const ApplyArgs &a, hipStream_t s)
{
    if (!a.folded || a.g.nz != fold64::NZ || contract_force_generic()) return false;
    const int64_t Lq = a.g.Lq();
    const unsigned grid = (unsigned)std::min<int64_t>(Lq, device_cus());
    for (int h0 = 0; h0 < a.nrhs; h0 += 2) {
        const int nh = std::min(2, a.nrhs - h0);
        if (a.precision == 0)
            hipLaunchKernelGGL((contract_fold64_kernel<double>), dim3(grid), dim3(fold64::NTHR), 0, s,
                               (const double2 *)a.G, (double2 *)a.buf + h0 * a.g.M(), Lq, a.g.M(), nh, a.g.nx, a.g.ny);
        else
            hipLaunchKernelGGL((contract_fold64_kernel<float>), dim3(grid), dim3(fold64::NTHR), 0, s, (const float2 *)a.G,
                               (float2 *)a.buf + h0 * a.g.M(), Lq, a.g.M(), nh, a.g.nx, a.g.ny);
        XTR_LAUNCH_CHECK("contract_fold64_kernel");
    }
    note_contract(a, "contract_fold64_kernel");
    return true;
}

// Folded tensor, a block that fits in LDS (contract_block.h), or a wave per block (contract_direct.hip) where the
// blocks are small and enough of them fill the chip; 1-8 right-hand sides.
static bool contract_block(const ApplyArgs &a, hipStream_t s)
{
    // byte offsets within one right-hand side's spectrum are 32-bit
    if (!a.folded || a.nrhs < 1 || a.nrhs > kMaxRhs || contract_force_generic() || a.g.M() * 16 > 0xffffffffLL) return false;
    // Up to 10 layers; a wave per block needs 6 blocks a CU (2 up to 5 layers, one row tile). Times of the block
    // kernel over those of the wave's, 1 to 8 right-hand sides, complex128: nz = 8 at 120 x 100 1.04-1.14, 64 x 64
    // 0.99-1.19, 32 x 32 0.92-1.05, 16 x 16 0.79-1.10; nz = 5 1.44-1.78, 1.36-1.47, 1.12-1.32, 0.98-1.16. Past 10
    // layers 48 x 40 x 12 0.95-1.17, 64 x 64 x 16 0.70-0.97.
    if (a.g.nz <= kDirectMostLayers && a.g.Lq() >= (a.g.nz <= 5 ? 2 : 6) * device_cus() && contract_direct(a, s)) return true;
    using Range = bool (*)(const ApplyArgs &, hipStream_t);
    static const Range c128[] = {contract_block_c128_a, contract_block_c128_b, contract_block_c128_c, contract_block_c128_d};
    static const Range c64[] = {contract_block_c64_a, contract_block_c64_b, contract_block_c64_c, contract_block_c64_d};
    for (Range r : a.precision ? c64 : c128)
        if (r(a, s)) return true;
    return false;
}

template <typename T>
static void contract(const ApplyArgs &a, hipStream_t s)
{
    if (!a.folded && contract_stream<T>(a, s)) return;
    if (!a.folded && contract_stream64(a, s)) return;
    if (contract_fold64(a, s)) return;
    if (contract_block(a, s)) return;
    const int nz = a.g.nz, C = 3 * nz;
    const int per_w = a.nrhs * C;
    int W = per_w >= 256 ? 1 : 256 / per_w;
    if (W < 1) W = 1;
    int threads = (int)ceil_div((int64_t)W * per_w, 64) * 64;
    if (threads > 1024) throw hip_error("contraction: 3*nz*nrhs exceeds 1024 threads");
    // folded, a block past LDS: 1.3 to 6 times as fast from 48 layers on, 1 to 5 right-hand sides, as what follows
    if (a.folded && !contract_force_generic() && contract_rows(a, s)) return;
    const size_t lds = sizeof(cplx<T>) * ((size_t)W * nz * (nz + 1) + (size_t)W * per_w);
    const int64_t L = a.g.L();
    dim3 grid((unsigned)ceil_div(L, W));
    hipLaunchKernelGGL(contract_kernel<T>, grid, dim3(threads), lds, s, (const cplx<T> *)a.G, (cplx<T> *)a.buf, L,
                       nz, a.nrhs, W, a.g.M(), a.packed_rc, a.folded ? a.g.nx : 0, a.g.ny);
    XTR_LAUNCH_CHECK("contract_kernel");
    note_contract(a, "contract_kernel");
}

void launch_contract(const ApplyArgs &a, hipStream_t s) { a.precision ? contract<float>(a, s) : contract<double>(a, s); }

// ---- Green tensor layout conversion -----------------------------------------------------------
__global__ void green_interleave_kernel(const double2 *xx, const double2 *xy, const double2 *xz, const double2 *yy,
                                        const double2 *yz, const double2 *zz, double2 *dev, int64_t L, int nz,
                                        int dir)
{
    const int S = nz * (nz + 1) / 2, A = nz * nz;
    const int64_t gblk = 4LL * S + 2LL * A;
    const int64_t total = L * gblk;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t l = e / gblk;
        const int64_t o = e % gblk;
        const double2 *src;
        int64_t si;
        if (o < 4LL * S) {
            const int b = (int)(o / S);
            const double2 *comps[4] = {xx, xy, yy, zz};
            src = comps[b];
            si = l * S + (o % S);
        } else {
            const int b = (int)((o - 4LL * S) / A);
            const int pos = (int)((o - 4LL * S) % A);          // device (swizzled) position
            const int rc = pos / nz, tr = (pos % nz) ^ (rc & asym_swizzle_mask(nz));
            src = b == 0 ? xz : yz;
            si = l * A + (int64_t)rc * nz + tr;
        }
        if (dir == 0) dev[e] = src[si];
        else const_cast<double2 *>(src)[si] = dev[e];
    }
}

void launch_green_interleave(const double2 *comp[6], double2 *dev, const Geom &g, hipStream_t s)
{
    hipLaunchKernelGGL(green_interleave_kernel, dim3(2048), dim3(256), 0, s, comp[0], comp[1], comp[2], comp[3],
                       comp[4], comp[5], dev, g.L(), g.nz, 0);
    XTR_LAUNCH_CHECK("green_interleave_kernel");
}

void launch_green_deinterleave(const double2 *dev, double2 *comp[6], const Geom &g, hipStream_t s)
{
    hipLaunchKernelGGL(green_interleave_kernel, dim3(2048), dim3(256), 0, s, comp[0], comp[1], comp[2], comp[3],
                       comp[4], comp[5], const_cast<double2 *>(dev), g.L(), g.nz, 1);
    XTR_LAUNCH_CHECK("green_deinterleave_kernel");
}

// ---- folded Green tensor -------------------------------------------------------------------------
// Sign of element o of a device block (xx, xy, yy, zz, xz, yz) in the image (mx, my) of its block.
__device__ __forceinline__ double fold_sign(int64_t o, int64_t S, int64_t A, int mx, int my)
{
    if (o < S) return 1.0;
    if (o < 2 * S) return (mx ^ my) ? -1.0 : 1.0;
    if (o < 4 * S) return 1.0;
    if (o < 4 * S + A) return mx ? -1.0 : 1.0;
    return my ? -1.0 : 1.0;
}

// dir 0: folded[b] = full[source wavenumber of b]; dir 1: full[l] = sign * folded[b(l)]
__global__ void green_fold_kernel(double2 *full, double2 *folded, int nx, int ny, int nz, int dir)
{
    const int64_t S = (int64_t)nz * (nz + 1) / 2, A = (int64_t)nz * nz, gblk = 4 * S + 2 * A;
    const int64_t total = (dir == 0 ? (int64_t)(nx + 1) * (ny + 1) : 4LL * nx * ny) * gblk;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t k = e / gblk, o = e % gblk;
        if (dir == 0) {
            const int64_t qx = k / (ny + 1), qy = k % (ny + 1);
            folded[e] = full[(qx * 2 * ny + qy) * gblk + o];
        } else {
            const FoldPos p = fold_pos(k, nx, ny);
            const double sg = fold_sign(o, S, A, p.mx, p.my);
            const double2 v = folded[p.b * gblk + o];
            full[e] = make_double2(sg * v.x, sg * v.y);
        }
    }
}

void launch_green_fold(const double2 *full, double2 *folded, const Geom &g, hipStream_t s)
{
    hipLaunchKernelGGL(green_fold_kernel, dim3(2048), dim3(256), 0, s, const_cast<double2 *>(full), folded, g.nx, g.ny,
                       g.nz, 0);
    XTR_LAUNCH_CHECK("green_fold_kernel");
}

void launch_green_unfold(const double2 *folded, double2 *full, const Geom &g, hipStream_t s)
{
    hipLaunchKernelGGL(green_fold_kernel, dim3(2048), dim3(256), 0, s, full, const_cast<double2 *>(folded), g.nx, g.ny,
                       g.nz, 1);
    XTR_LAUNCH_CHECK("green_unfold_kernel");
}

// Non-negative doubles order like their bit patterns, so an unsigned 64-bit atomic max is a max.
__global__ __launch_bounds__(256) void green_mirror_check_kernel(const double2 *full, int nx, int ny, int nz,
                                                                 unsigned long long *stat)
{
    const int64_t S = (int64_t)nz * (nz + 1) / 2, A = (int64_t)nz * nz, gblk = 4 * S + 2 * A;
    const int64_t total = 4LL * nx * ny * gblk;
    double m[12];
#pragma unroll
    for (int c = 0; c < 12; ++c) m[c] = 0.0;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t l = e / gblk, o = e % gblk;
        const int c = o < 4 * S ? (int)(o / S) : 4 + (int)((o - 4 * S) / A);
        const double2 v = full[e];
        const double mag = fmax(fabs(v.x), fabs(v.y));
        const FoldPos p = fold_pos(l, nx, ny);
        double d = 0.0;
        if (p.mx || p.my) {
            const int64_t qx = p.b / (ny + 1), qy = p.b % (ny + 1);
            const double sg = fold_sign(o, S, A, p.mx, p.my);
            const double2 w = full[(qx * 2 * ny + qy) * gblk + o];
            d = fmax(fabs(v.x - sg * w.x), fabs(v.y - sg * w.y));
        }
#pragma unroll
        for (int k = 0; k < 6; ++k)
            if (k == c) {
                m[2 * k] = fmax(m[2 * k], d);
                m[2 * k + 1] = fmax(m[2 * k + 1], mag);
            }
    }
    __shared__ double red[12][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int c = 0; c < 12; ++c) {
        double v = m[c];
        for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
        if (lane == 0) red[c][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x < 12) {
        const double v = fmax(fmax(red[threadIdx.x][0], red[threadIdx.x][1]), fmax(red[threadIdx.x][2], red[threadIdx.x][3]));
        atomicMax(stat + threadIdx.x, (unsigned long long)__double_as_longlong(v));
    }
}

void launch_green_mirror_check(const double2 *full, const Geom &g, double *stat, hipStream_t s)
{
    XTR_CHECK(hipMemsetAsync(stat, 0, 12 * sizeof(double), s));
    hipLaunchKernelGGL(green_mirror_check_kernel, dim3(1024), dim3(256), 0, s, full, g.nx, g.ny, g.nz,
                       reinterpret_cast<unsigned long long *>(stat));
    XTR_LAUNCH_CHECK("green_mirror_check_kernel");
}

__global__ void to_f32_kernel(const double2 *src, float2 *dst, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = to_f(src[i]);
}

void launch_to_f32(const double2 *src, float2 *dst, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL(to_f32_kernel, dim3(4096), dim3(256), 0, s, src, dst, n);
    XTR_LAUNCH_CHECK("to_f32_kernel");
}

}  // namespace xtr
