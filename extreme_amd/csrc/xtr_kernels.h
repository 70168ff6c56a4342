// Host-side launchers of the gfx950 kernels. Every launcher enqueues on the given stream and
// checks the launch; none synchronises.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "xtr_tiles.h"

namespace xtr {

constexpr int kMaxRhs = 8;

// Geometry of one operator (Nx, Ny, Nz) and derived sizes.
struct Geom {
    int nx, ny, nz;
    int64_t n() const { return 3LL * nx * ny * nz; }          // unknowns
    int64_t L() const { return 4LL * nx * ny; }               // padded lateral plane
    int64_t C() const { return 3LL * nz; }                    // spectrum columns per wavenumber
    int64_t M() const { return L() * C(); }                   // spectrum elements
    int64_t S() const { return (int64_t)nz * (nz + 1) / 2; }  // packed symmetric block
    int64_t gblk() const { return 4 * S() + 2LL * nz * nz; }  // Green elements per wavenumber
    int64_t Lq() const { return (int64_t)(nx + 1) * (ny + 1); } // blocks of a folded Green tensor
};

// Folded Green tensor. The mirrored lateral tensor is even or odd in x and in y per component
// (xx, yy, zz even/even; xy odd/odd; xz odd/even; yz even/odd), so its 2-D spectrum satisfies
// G(2Nx-kx, ky) = D_x G(kx, ky) D_x and G(kx, 2Ny-ky) = D_y G(kx, ky) D_y with D_x = diag(-I, I, I),
// D_y = diag(I, -I, I) on the (x, y, z) components. A folded tensor stores only kx <= Nx, ky <= Ny,
// block b = qx (Ny+1) + qy; wavenumber l = kx 2Ny + ky uses block b with u_x, y_x negated when
// kx > Nx (mx) and u_y, y_y negated when ky > Ny (my).
struct FoldPos {
    int64_t b;
    int mx, my;
};
__host__ __device__ inline FoldPos fold_pos(int64_t l, int nx, int ny)
{
    const int kx = (int)(l / (2 * ny)), ky = (int)(l % (2 * ny));
    FoldPos p;
    p.mx = kx > nx;
    p.my = ky > ny;
    const int qx = p.mx ? 2 * nx - kx : kx, qy = p.my ? 2 * ny - ky : ky;
    p.b = (int64_t)qx * (ny + 1) + qy;
    return p;
}
// Wavenumbers that use folded block b (its images): n = 1, 2 or 4. Image i < n has kx mirrored
// (mx) and/or ky mirrored (my); image 0 is the unmirrored wavenumber. Computed from i rather than
// stored in arrays: a lane-dependent index into a private array would put it in scratch.
struct FoldImages {
    int n;
    int qx, qy, nx, ny;
    bool two_x, two_y;
    __host__ __device__ int mx(int i) const { return two_x ? (i & 1) : 0; }
    __host__ __device__ int my(int i) const { return two_y ? (two_x ? (i >> 1) & 1 : i & 1) : 0; }
    __host__ __device__ int64_t l(int i) const
    {
        const int kx = mx(i) ? 2 * nx - qx : qx, ky = my(i) ? 2 * ny - qy : qy;
        return (int64_t)kx * 2 * ny + ky;
    }
};
__host__ __device__ inline FoldImages fold_images(int64_t b, int nx, int ny)
{
    FoldImages im;
    im.qx = (int)(b / (ny + 1));
    im.qy = (int)(b % (ny + 1));
    im.nx = nx;
    im.ny = ny;
    im.two_x = im.qx > 0 && im.qx < nx;
    im.two_y = im.qy > 0 && im.qy < ny;
    im.n = (im.two_x ? 2 : 1) * (im.two_y ? 2 : 1);
    return im;
}

// Device position of the asymmetric-block element (rc, tr) (xz and yz, nz*nz each): rows are
// XOR-swizzled, tr ^ (rc & mask), so that a block copied linearly into LDS can be read along rows
// and along columns without bank conflicts. mask = 15 when 16 | nz, 7 when 8 | nz, else 0
// (plain row-major). The reference layout at the set/get boundary is plain row-major [rc][tr].
__host__ __device__ inline int asym_swizzle_mask(int nz) { return nz % 16 == 0 ? 15 : (nz % 8 == 0 ? 7 : 0); }
__host__ __device__ inline int asym_pos(int rc, int tr, int nz, int mask) { return rc * nz + (tr ^ (rc & mask)); }

// Per-call vector pointers (device; complex128, or complex64 when the apply's vec32 is set) for up
// to kMaxRhs right-hand sides.
// R[i] is the R function of right-hand side i's model ([nx*ny*nz]); models that share the grid,
// background and frequency share the Green tensor, so one apply can serve several of them.
struct RhsPtrs {
    const double2 *x[kMaxRhs];
    double2 *y[kMaxRhs];
    const double2 *R[kMaxRhs];
};

// The kernel that a contraction launched: its name and, after the element type, its template arguments (0: none).
struct ContractKernel {
    const char *name = nullptr;
    int precision = 0, depth = 0, group = 0;
};

// ---- operator apply (op_kernels.hip) -------------------------------------------------------
// Twiddle tables exp(-2 pi i k / P), k < P, in the apply precision.
// precision: 0 = FP64 (double2 buffers / Green), 1 = FP32 (float2).
struct ApplyArgs {
    Geom g;
    int precision;
    int nrhs;
    int type;                 // 0 = A, 1 = Chi0
    const double2 *R;         // [nx*ny*nz] FP64, used for right-hand sides whose v.R[i] is null
    const double *f;          // [nz] forward factors (real)
    const double *b;          // [nz] backward factors (real)
    const void *G;            // [nblk][gblk] in apply precision
    int folded;               // G holds the folded tensor (nblk = Lq) rather than all L wavenumbers
    const uint16_t *packed_rc;// [S][2] (rc, tr) of each packed element
    void *buf;                // nrhs * M spectrum in apply precision
    const void *tw_x;         // twiddles for P = 2 nx
    const void *tw_y;         // twiddles for P = 2 ny
    int fft_tile[4];          // column tile of fwd_y, fwd_x, inv_x, inv_y (FFT_TILE_*)
    int vec32;                // v.x and v.y point to complex64 vectors (float2; precision FP32 only)
    RhsPtrs v;
    ContractKernel *ran;      // where launch_contract notes its kernel, or null
};

// the column tiles a pencil length offers in this precision (FFT_TILE_*), into tiles[8]; returns how many
int fft_tile_options(int p, int precision, int *tiles);

inline void note_contract(const ApplyArgs &a, const char *name, int depth = 0, int group = 0)
{
    if (a.ran) *a.ran = ContractKernel{name, a.precision, depth, group};
}

// Stage launchers (used separately for per-stage timing).
void launch_fwd_y(const ApplyArgs &a, hipStream_t s);
void launch_fwd_x(const ApplyArgs &a, hipStream_t s);
void launch_contract(const ApplyArgs &a, hipStream_t s);
// the contraction of a folded tensor whose block fits in LDS (contract_block.h), by ranges of depths; false:
// not a depth of the range, or one that does not fit
bool contract_block_c128_a(const ApplyArgs &a, hipStream_t s);
bool contract_block_c128_b(const ApplyArgs &a, hipStream_t s);
bool contract_block_c128_c(const ApplyArgs &a, hipStream_t s);
bool contract_block_c128_d(const ApplyArgs &a, hipStream_t s);
bool contract_block_c64_a(const ApplyArgs &a, hipStream_t s);
bool contract_block_c64_b(const ApplyArgs &a, hipStream_t s);
bool contract_block_c64_c(const ApplyArgs &a, hipStream_t s);
bool contract_block_c64_d(const ApplyArgs &a, hipStream_t s);
// the same for up to kDirectMostLayers layers, a wave per block (contract_direct.hip)
constexpr int kDirectMostLayers = 10;
bool contract_direct(const ApplyArgs &a, hipStream_t s);
// and for up to kRowsMost rows (3nz), a wave per 16 rows (contract_direct.hip)
constexpr int kRowsMost = 256;
bool contract_rows(const ApplyArgs &a, hipStream_t s);
int device_cus();            // compute units of the current device
void launch_inv_x(const ApplyArgs &a, hipStream_t s);
void launch_inv_y(const ApplyArgs &a, hipStream_t s);

// In-place forward 2-D FFT of an [n1][n2][ncols] array (an assembled tensor), FP64.
void launch_fft2_plain(double2 *data, int n1, int n2, int64_t ncols, const double2 *tw1, const double2 *tw2, hipStream_t s);
// The same for a Green tensor held folded, [Nx+1][Ny+1][gblk], in place: points (i, j), i < Nx and j < Ny,
// hold the tensor at those lateral offsets on entry, and every block the spectrum on return; the negative
// offsets follow from the mirror parities.
void launch_fft2_mirror(double2 *folded, const Geom &g, const double2 *tw_x, const double2 *tw_y, hipStream_t s);
// The same for a level tensor [Nx+1][Ny+1][ncomp][nz]; bit c of odd[0] (odd[1]): component c is odd in x (y).
void launch_fft2_mirror_level(double2 *folded, const Geom &g, int ncomp, const unsigned *odd, const double2 *tw_x,
                              const double2 *tw_y, hipStream_t s);
// Forward FFT of src [Nx][Ny][C], zero-padded, into spec [2Nx][2Ny][C]; backward FFT of spec (which it works in),
// cropped and scaled, into dst [Nx][Ny][C].
void launch_fft2_padded(const double2 *src, double2 *spec, const Geom &g, int C, const double2 *tw_x, const double2 *tw_y,
                        hipStream_t s);
void launch_fft2_cropped(double2 *spec, double2 *dst, const Geom &g, int C, double scale, const double2 *tw_x,
                         const double2 *tw_y, hipStream_t s);
bool fft_length_supported(int p);

// Reorders the Green tensor between the reference layout (six component arrays) and the
// device layout [L][xx S | xy S | yy S | zz S | xz nz^2 | yz nz^2].
void launch_green_interleave(const double2 *comp[6], double2 *dev, const Geom &g, hipStream_t s);
void launch_green_deinterleave(const double2 *dev, double2 *comp[6], const Geom &g, hipStream_t s);
// full [L][gblk] -> folded [Lq][gblk] (blocks kx <= Nx, ky <= Ny), and back with the mirror signs
void launch_green_fold(const double2 *full, double2 *folded, const Geom &g, hipStream_t s);
void launch_green_unfold(const double2 *folded, double2 *full, const Geom &g, hipStream_t s);
// stat[2c] = max |G_c(l) - s_c G_c(mirror source of l)|, stat[2c+1] = max |G_c| over a full
// tensor, c in device block order (xx, xy, yy, zz, xz, yz); stat (12 doubles) cleared here
void launch_green_mirror_check(const double2 *full, const Geom &g, double *stat, hipStream_t s);
void launch_to_f32(const double2 *src, float2 *dst, int64_t n, hipStream_t s);
void launch_probe_stream(const void *src, void *dst, int64_t blocks, int read_kb, int write_kb, hipStream_t s);

// Observation level (obs_kernels.hip): jQ from chi (operator prepared as A: R and f of that type),
// and the anomalous field at a level from jQ with the AtoO tensor G ([L][ncomp][nz], or folded the
// (Nx+1)(Ny+1) blocks kx <= Nx, ky <= Ny); spec holds L * 3nz and small L * 3 complex128 of scratch; field
// is [Nx][Ny][3].
void launch_jq(const double2 *chi, const double2 *js, const double2 *R, const double *f, const Geom &g, double2 *jq,
               hipStream_t s);
void launch_level_field(const double2 *G, int electric, int folded, const double2 *jq, const Geom &g, double2 *spec,
                        double2 *small, const double2 *tw_x, const double2 *tw_y, double2 *field, hipStream_t s);
// Components of a level tensor that are odd in x (odd[0]) and in y (odd[1]), as bit masks in their order
inline void level_parity(int electric, unsigned *odd)
{
    // electric xx yy zz xy xz yz zx zy; magnetic xx xy yx xz yz zx zy
    odd[0] = electric ? 1u << 3 | 1u << 4 | 1u << 6 : 1u << 0 | 1u << 4 | 1u << 6;
    odd[1] = electric ? 1u << 3 | 1u << 5 | 1u << 7 : 1u << 0 | 1u << 3 | 1u << 5;
}

// ---- Krylov (krylov_kernels.hip) -----------------------------------------------------------
// Vectors are complex128 (double2) or complex64 (float2, the mixed-precision correction solves);
// every kernel accumulates in FP64.
constexpr int kRedBlocks = 512;   // most partial sums of a reduction
int reduction_blocks(int64_t n);  // partial sums of a Gram-Schmidt step's reductions over n elements

// their sum, in the order the kernels use
double sum_partials(const double *p, int n);

// A right-hand side's vectors in the batched kernels of a Gram-Schmidt step.
template <typename VT>
struct StepRhs {
    const VT *V;        // basis columns (contiguous, stride n); b of a residual
    const VT *u;        // A x of a residual, else null
    VT *w;              // the vector worked on
    VT *next;           // where w / |w| (mul: (1 / |w|) w) goes, or null
    double2 *partial;   // [cnt][reduction_blocks(n)] scratch
    double *norm_dev;   // [reduction_blocks(n)] scratch
    double2 *h;         // [cnt] the projections (host memory, device address)
    double *norm;       // [reduction_blocks(n)] partial sums of |w|^2 (host memory, device address)
    int cnt, mul;
};
template <typename VT>
struct StepArgs {
    StepRhs<VT> rhs[kMaxRhs];
};
// h = V^H w, w -= V h, |w|^2, next
void launch_cgs_step(const StepArgs<double2> &a, int nrhs, int64_t n, hipStream_t s);
void launch_cgs_step(const StepArgs<float2> &a, int nrhs, int64_t n, hipStream_t s);
// |w|^2, with w = V - u first where u is given, and next
void launch_step_norm(const StepArgs<double2> &a, int nrhs, int64_t n, hipStream_t s);
void launch_step_norm(const StepArgs<float2> &a, int nrhs, int64_t n, hipStream_t s);

// partial sums of |w|^2 (kRedBlocks) ; out = sum of partials
void launch_norm2(const double2 *w, int64_t n, double *partial, hipStream_t s);
void launch_reduce_r(const double *partial, double *out, hipStream_t s);
// dst = a * src (the complex64 copy of a scaled residual)
void launch_mul(const double2 *src, double a, float2 *dst, int64_t n, hipStream_t s);
// dst = a - b
void launch_sub(const double2 *a, const double2 *b, double2 *dst, int64_t n, hipStream_t s);
// x += sum_k B_k y_k  (ConstructCurrentSolution, y passed by value)
struct Coef32 { double2 c[32]; };
void launch_update_solution(const double2 *B, int cnt, const Coef32 &y, double2 *x, int64_t n, hipStream_t s);
void launch_update_solution(const float2 *B, int cnt, const Coef32 &y, float2 *x, int64_t n, hipStream_t s);
void launch_update_solution(const float2 *B, int cnt, const Coef32 &y, double2 *x, int64_t n, hipStream_t s);

}  // namespace xtr
