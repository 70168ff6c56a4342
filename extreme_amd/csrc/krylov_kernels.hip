// Krylov-basis kernels for the FGMRES driver: block dot V^H w, the classical Gram-Schmidt update
// with the new norm, norms, scaling and the solution update.
//
// Vectors are complex128 (the reference's arithmetic) or complex64 (the correction solves of the
// mixed-precision refinement): every kernel is a template on the stored element type and widens each
// element to FP64 on load, so products, dot sums and norms accumulate in FP64 either way; complex64
// results are rounded once, on store.
//
// The kernels of a Gram-Schmidt step serve several right-hand sides at once (grid z), those whose solves run in
// step, each on its own vectors: small grids leave one right-hand side far too few workgroups to fill the chip.
//
// Reductions are two-stage and deterministic: a number of workgroups that depends only on n write partial sums
// (grid-stride loops, wavefront shuffles, then LDS), which are summed in a fixed order: the projections by every
// workgroup of the update that uses them (the partials sit in L2; a kernel for it would cost a launch), the
// norms by the kernel that scales by them and, in the same order, by the host, into whose memory they are written
// too. So repeated solves give identical iterates, and a right-hand side's do not depend on which others run
// beside it. The host polls those values themselves (a NaN of its own marks one that is not there yet): it goes
// on as soon as the last workgroup has stored, not when the kernel's end has reached an event.
#include <algorithm>

#include "xtr_common.h"
#include "xtr_kernels.h"

namespace xtr {

constexpr int kThreads = 256;
constexpr int kDotChunk = 8;   // basis columns per pass of block_dots

__device__ __forceinline__ double2 ld(const double2 &v) { return v; }
__device__ __forceinline__ double2 ld(const float2 &v) { return to_d(v); }
__device__ __forceinline__ void st(double2 &d, double2 v) { d = v; }
__device__ __forceinline__ void st(float2 &d, double2 v) { d = to_f(v); }

__device__ inline double warp_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// sum over the workgroup of v; valid in thread 0
__device__ inline double block_sum(double v, double *sh)
{
    v = warp_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r += sh[i];
    __syncthreads();
    return r;
}

// Sums over the wavefront of 16 values a lane; lane l ends with the sum of value (l >> 2) & 15. Each step trades
// half of what is left with the lane that keeps the other half: 17 shuffles instead of 16 x 6.
__device__ __forceinline__ double wave_sum16(double (&v)[16], int lane)
{
#pragma unroll
    for (int half = 8, o = 32; half >= 1; half >>= 1, o >>= 1) {
        const bool up = lane & o;
#pragma unroll
        for (int k = 0; k < half; ++k) {
            const double keep = up ? v[half + k] : v[k], give = up ? v[k] : v[half + k];
            v[k] = keep + __shfl_xor(give, o, 64);
        }
    }
    double r = v[0];
    r += __shfl_xor(r, 2, 64);
    r += __shfl_xor(r, 1, 64);
    return r;
}

int reduction_blocks(int64_t n)
{
    return (int)std::max<int64_t>(1, std::min<int64_t>(kRedBlocks, ceil_div(n, 2 * kThreads)));
}

// A value for the host, which may be polling it.
__device__ __forceinline__ void to_host(double *p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// partial[k][blk] = sum_i conj(V[k][i]) w[i] over this block's i, 8 columns per grid y
template <typename VT>
__global__ __launch_bounds__(kThreads) void block_dots_kernel(StepArgs<VT> a, int64_t n)
{
    __shared__ double sh[kThreads / 64][16];
    const StepRhs<VT> &r = a.rhs[blockIdx.z];
    const VT *__restrict__ V = r.V, *__restrict__ w = r.w;
    const int k0 = blockIdx.y * kDotChunk;
    const int kc = min(kDotChunk, r.cnt - k0);
    if (kc <= 0) return;
    double2 acc[kDotChunk];
#pragma unroll
    for (int k = 0; k < kDotChunk; ++k) acc[k] = make_double2(0, 0);
    // two elements per iteration, i and i + stride, all loads issued before the products (the
    // accumulation order per thread is the plain grid-stride order)
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x;
    for (; i + stride < n; i += 2 * stride) {
        const VT w0 = w[i], w1 = w[i + stride];
        VT v0[kDotChunk], v1[kDotChunk];
#pragma unroll
        for (int k = 0; k < kDotChunk; ++k)
            if (k < kc) {
                v0[k] = V[(int64_t)(k0 + k) * n + i];
                v1[k] = V[(int64_t)(k0 + k) * n + i + stride];
            }
#pragma unroll
        for (int k = 0; k < kDotChunk; ++k)
            if (k < kc) {
                acc[k] = cfma_conj<double>(acc[k], ld(v0[k]), ld(w0));
                acc[k] = cfma_conj<double>(acc[k], ld(v1[k]), ld(w1));
            }
    }
    if (i < n) {
        const double2 wv = ld(w[i]);
#pragma unroll
        for (int k = 0; k < kDotChunk; ++k)
            if (k < kc) acc[k] = cfma_conj<double>(acc[k], ld(V[(int64_t)(k0 + k) * n + i]), wv);
    }
    double v[16];
#pragma unroll
    for (int k = 0; k < kDotChunk; ++k) {
        v[2 * k] = acc[k].x;
        v[2 * k + 1] = acc[k].y;
    }
    const int lane = threadIdx.x & 63;
    const double t = wave_sum16(v, lane);
    if ((lane & 3) == 0) sh[threadIdx.x >> 6][lane >> 2] = t;
    __syncthreads();
    if (threadIdx.x < 2 * kc) {
        double q = 0;
        for (int wv = 0; wv < kThreads / 64; ++wv) q += sh[wv][threadIdx.x];
        reinterpret_cast<double *>(r.partial)[((int64_t)(k0 + threadIdx.x / 2) * gridDim.x + blockIdx.x) * 2 +
                                              (threadIdx.x & 1)] = q;
    }
}

// h = the projections from their partials; w[i] -= sum_k V[k][i] h[k]; norm[blk] = sum |w_new|^2 (of the stored,
// rounded w), and h itself, into host memory
template <typename VT>
__global__ __launch_bounds__(kThreads) void cgs_update_kernel(StepArgs<VT> a, int64_t n)
{
    __shared__ double sh[kThreads / 64];
    __shared__ double2 hs[32];
    const StepRhs<VT> &r = a.rhs[blockIdx.z];
    const VT *__restrict__ V = r.V;
    VT *w = r.w;
    const int cnt = r.cnt, nblk = gridDim.x, lane = threadIdx.x & 63;
    for (int k = threadIdx.x >> 6; k < cnt; k += kThreads / 64) {
        double re = 0, im = 0;
        for (int b = lane; b < nblk; b += 64) {
            const double2 p = r.partial[(int64_t)k * nblk + b];
            re += p.x;
            im += p.y;
        }
        re = warp_sum(re);
        im = warp_sum(im);
        if (lane == 0) {
            hs[k] = make_double2(re, im);
            if (blockIdx.x == 0) {
                to_host(&r.h[k].x, re);
                to_host(&r.h[k].y, im);
            }
        }
    }
    __syncthreads();
    double nn = 0;
    // two elements per iteration, i and i + stride, so that twice the loads are in flight; each
    // element's sum over k and the norm's sum over elements keep the plain grid-stride order
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x;
    for (; i + stride < n; i += 2 * stride) {
        double2 a0 = make_double2(0, 0), a1 = a0;
        int k = 0;
        for (; k + kDotChunk <= cnt; k += kDotChunk) {          // 2 x 8 loads issued together
            VT v0[kDotChunk], v1[kDotChunk];
#pragma unroll
            for (int j = 0; j < kDotChunk; ++j) {
                v0[j] = V[(int64_t)(k + j) * n + i];
                v1[j] = V[(int64_t)(k + j) * n + i + stride];
            }
#pragma unroll
            for (int j = 0; j < kDotChunk; ++j) {
                a0 = cfma<double>(a0, ld(v0[j]), hs[k + j]);
                a1 = cfma<double>(a1, ld(v1[j]), hs[k + j]);
            }
        }
        for (; k < cnt; ++k) {
            const VT v0 = V[(int64_t)k * n + i], v1 = V[(int64_t)k * n + i + stride];
            a0 = cfma<double>(a0, ld(v0), hs[k]);
            a1 = cfma<double>(a1, ld(v1), hs[k]);
        }
        VT t0, t1;
        st(t0, csub<double>(ld(w[i]), a0));
        st(t1, csub<double>(ld(w[i + stride]), a1));
        w[i] = t0;
        w[i + stride] = t1;
        const double2 n0 = ld(t0), n1 = ld(t1);
        nn = fma(n0.x, n0.x, nn);
        nn = fma(n0.y, n0.y, nn);
        nn = fma(n1.x, n1.x, nn);
        nn = fma(n1.y, n1.y, nn);
    }
    if (i < n) {
        double2 t = make_double2(0, 0);
        for (int k = 0; k < cnt; ++k) t = cfma<double>(t, ld(V[(int64_t)k * n + i]), hs[k]);
        VT u;
        st(u, csub<double>(ld(w[i]), t));
        w[i] = u;
        const double2 nw = ld(u);
        nn = fma(nw.x, nw.x, nn);
        nn = fma(nw.y, nw.y, nn);
    }
    nn = block_sum(nn, sh);
    if (threadIdx.x == 0) {
        r.norm_dev[blockIdx.x] = nn;
        to_host(r.norm + blockIdx.x, nn);
    }
}

// norm[blk] = sum |v|^2, v = w, or v = w = V - u rounded as stored where u is given (the residual b - A x)
template <typename VT>
__global__ __launch_bounds__(kThreads) void step_norm_kernel(StepArgs<VT> a, int64_t n)
{
    __shared__ double sh[kThreads / 64];
    const StepRhs<VT> &r = a.rhs[blockIdx.z];
    double nn = 0;
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        VT t;
        if (r.u) {
            st(t, csub<double>(ld(r.V[i]), ld(r.u[i])));
            r.w[i] = t;
        } else {
            t = r.w[i];
        }
        const double2 v = ld(t);
        nn = fma(v.x, v.x, nn);
        nn = fma(v.y, v.y, nn);
    }
    nn = block_sum(nn, sh);
    if (threadIdx.x == 0) {
        if (r.next) r.norm_dev[blockIdx.x] = nn;
        to_host(r.norm + blockIdx.x, nn);
    }
}

// next = w / |w| (v_{j+1}, Gmres.cs:267-268) or, where mul, (1 / |w|) w (V_0, Gmres.cs:117), |w| from its nblk
// partial sums in the order of sum_partials
template <typename VT>
__global__ __launch_bounds__(kThreads) void step_next_kernel(StepArgs<VT> a, int nblk, int64_t n)
{
    __shared__ double sh;
    const StepRhs<VT> &r = a.rhs[blockIdx.z];
    if (!r.next) return;
    if (threadIdx.x < 64) {
        double v = 0;
        for (int b = threadIdx.x; b < nblk; b += 64) v += r.norm_dev[b];
        v = warp_sum(v);
        if (threadIdx.x == 0) sh = r.mul ? 1 / sqrt(v) : sqrt(v);
    }
    __syncthreads();
    const double d = sh;
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        const double2 v = ld(r.w[i]);
        st(r.next[i], r.mul ? make_double2(d * v.x, d * v.y) : make_double2(v.x / d, v.y / d));
    }
}

double sum_partials(const double *p, int n)
{
    double v[64];
    for (int l = 0; l < 64; ++l) {
        v[l] = 0;
        for (int b = l; b < n; b += 64) v[l] += p[b];
    }
    for (int o = 32; o > 0; o >>= 1)       // warp_sum's order: lane 0 adds the lane o further on
        for (int l = 0; l < o; ++l) v[l] += v[l + o];
    return v[0];
}

template <typename VT>
static void launch_next(const StepArgs<VT> &a, int nrhs, int64_t n, hipStream_t s)
{
    bool any = false;
    for (int r = 0; r < nrhs; ++r) any = any || a.rhs[r].next;
    if (!any) return;
    const unsigned nb = (unsigned)std::min<int64_t>(2048, ceil_div(n, kThreads));
    hipLaunchKernelGGL(step_next_kernel<VT>, dim3(nb, 1, nrhs), dim3(kThreads), 0, s, a, reduction_blocks(n), n);
    XTR_LAUNCH_CHECK("step_next_kernel");
}

// One classical Gram-Schmidt pass of each right-hand side. The scaled vector follows at once, before the host has
// seen the norm: where the host then asks for a second pass, or ends the cycle, it is not used.
template <typename VT>
static void cgs_step(const StepArgs<VT> &a, int nrhs, int64_t n, hipStream_t s)
{
    int most = 0;
    for (int r = 0; r < nrhs; ++r) most = std::max(most, a.rhs[r].cnt);
    if (nrhs < 1 || nrhs > kMaxRhs || most < 1 || most > 32) throw hip_error("Gram-Schmidt step: 1 to 8 right-hand sides, 1 to 32 vectors");
    const unsigned nb = (unsigned)reduction_blocks(n);
    hipLaunchKernelGGL(block_dots_kernel<VT>, dim3(nb, (unsigned)ceil_div(most, kDotChunk), nrhs), dim3(kThreads), 0, s, a, n);
    XTR_LAUNCH_CHECK("block_dots_kernel");
    hipLaunchKernelGGL(cgs_update_kernel<VT>, dim3(nb, 1, nrhs), dim3(kThreads), 0, s, a, n);
    XTR_LAUNCH_CHECK("cgs_update_kernel");
    launch_next(a, nrhs, n, s);
}
void launch_cgs_step(const StepArgs<double2> &a, int nrhs, int64_t n, hipStream_t s) { cgs_step(a, nrhs, n, s); }
void launch_cgs_step(const StepArgs<float2> &a, int nrhs, int64_t n, hipStream_t s) { cgs_step(a, nrhs, n, s); }

template <typename VT>
static void step_norm(const StepArgs<VT> &a, int nrhs, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL(step_norm_kernel<VT>, dim3((unsigned)reduction_blocks(n), 1, nrhs), dim3(kThreads), 0, s, a, n);
    XTR_LAUNCH_CHECK("step_norm_kernel");
    launch_next(a, nrhs, n, s);
}
void launch_step_norm(const StepArgs<double2> &a, int nrhs, int64_t n, hipStream_t s) { step_norm(a, nrhs, n, s); }
void launch_step_norm(const StepArgs<float2> &a, int nrhs, int64_t n, hipStream_t s) { step_norm(a, nrhs, n, s); }

// partial sums of |w|^2, and their sum on the device (the learned preconditioner's scale)
__global__ __launch_bounds__(kThreads) void norm2_kernel(const double2 *__restrict__ w, int64_t n, double *partial)
{
    __shared__ double sh[kThreads / 64];
    double nn = 0;
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        nn = fma(w[i].x, w[i].x, nn);
        nn = fma(w[i].y, w[i].y, nn);
    }
    nn = block_sum(nn, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = nn;
}

void launch_norm2(const double2 *w, int64_t n, double *partial, hipStream_t s)
{
    hipLaunchKernelGGL(norm2_kernel, dim3(kRedBlocks), dim3(kThreads), 0, s, w, n, partial);
    XTR_LAUNCH_CHECK("norm2_kernel");
}

__global__ __launch_bounds__(kThreads) void reduce_r_kernel(const double *partial, double *out)
{
    __shared__ double sh[kThreads / 64];
    double v = 0;
    for (int b = threadIdx.x; b < kRedBlocks; b += kThreads) v += partial[b];
    v = block_sum(v, sh);
    if (threadIdx.x == 0) *out = v;
}

void launch_reduce_r(const double *partial, double *out, hipStream_t s)
{
    hipLaunchKernelGGL(reduce_r_kernel, dim3(1), dim3(kThreads), 0, s, partial, out);
    XTR_LAUNCH_CHECK("reduce_r_kernel");
}

template <typename VS, typename VD>
__global__ void mul_kernel(const VS *src, double a, VD *dst, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const double2 v = ld(src[i]);
        st(dst[i], make_double2(a * v.x, a * v.y));
    }
}

void launch_mul(const double2 *src, double a, float2 *dst, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL((mul_kernel<double2, float2>), dim3(2048), dim3(256), 0, s, src, a, dst, n);
    XTR_LAUNCH_CHECK("mul_kernel");
}

template <typename VT>
__global__ void sub_kernel(const VT *a, const VT *b, VT *dst, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        st(dst[i], csub<double>(ld(a[i]), ld(b[i])));
}

void launch_sub(const double2 *a, const double2 *b, double2 *dst, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL(sub_kernel<double2>, dim3(2048), dim3(256), 0, s, a, b, dst, n);
    XTR_LAUNCH_CHECK("sub_kernel");
}
// x[i] += sum_k B[k][i] y[k]  (ConstructCurrentSolution: r0 = Z y; x = x + r0)
template <typename VB, typename VX>
__global__ __launch_bounds__(kThreads) void update_solution_kernel(const VB *__restrict__ B, int cnt, Coef32 y,
                                                                   VX *x, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        double2 a = make_double2(0, 0);
        for (int k = 0; k < cnt; ++k) a = cfma<double>(a, ld(B[(int64_t)k * n + i]), y.c[k]);
        st(x[i], cadd<double>(ld(x[i]), a));
    }
}

void launch_update_solution(const double2 *B, int cnt, const Coef32 &y, double2 *x, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL((update_solution_kernel<double2, double2>), dim3(2048), dim3(kThreads), 0, s, B, cnt, y, x, n);
    XTR_LAUNCH_CHECK("update_solution_kernel");
}
void launch_update_solution(const float2 *B, int cnt, const Coef32 &y, float2 *x, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL((update_solution_kernel<float2, float2>), dim3(2048), dim3(kThreads), 0, s, B, cnt, y, x, n);
    XTR_LAUNCH_CHECK("update_solution_kernel");
}
void launch_update_solution(const float2 *B, int cnt, const Coef32 &y, double2 *x, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL((update_solution_kernel<float2, double2>), dim3(2048), dim3(kThreads), 0, s, B, cnt, y, x, n);
    XTR_LAUNCH_CHECK("update_solution_kernel");
}

}  // namespace xtr
