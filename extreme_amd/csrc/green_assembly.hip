// Device assembly of the anomaly-to-anomaly (AtoA) electric Green tensor in FP64.
//
// Stages (reference files in brackets):
//   host  scalar plans: NumberOfHankels interleaved log-rho grids and their lambda grids
//         [Green/Scalar/ScalarPlansCreater.cs:102-176, ScalarPlan.cs:76-97, HankelCoefficients.cs:67-76]
//   K1    per (plan item, lambda): eta, exp(-2 eta h), the P/Q reflection recursions for the
//         "1" and "Sigma" coefficient sets  [PlanCalculatorFast.cs:203-318, AlphaBeta.cs:24-42]
//   K2    per (transceiver pair, item, lambda): the vertical integrals T, R, C, D, the transfer
//         coefficient A[rc][tr] and U1..U5, normalised for the Hankel transform
//         [VolumeToVolumeCalculatorUFast.cs:34-337, green_scalar.c:86-386, ScalarMathUtils.cs:243-263]
//   K3    431-tap Hankel filter onto the merged rho grid, normalised by 1/(2 pi rho)
//         [HankelCoefficients.cs:103-118, ScalarMathUtils.cs:189-241, InnerResultsCombiner.cs:19-62]
//   K4    piecewise-linear segments I(rho) = A rho + B  [ScalarSegments.cs:86-128]
//   K5    lateral integration of every cell of the positive quadrant by line integrals along
//         its four edges (the knots of all cells' edges first, knots_kernel; then per cell the segments'
//         weights, in LDS, and their sums with the pairs' coefficients), written straight into the
//         device layout (a full tensor with its mirror images; a folded one gets them from the parities
//         in the FFT's loads)
//         [GreenTensorCalculator.cs:166-552, IntegralFactors.cs:17-30, QSign.cs:64-67,
//          GreenTensorFftPopulator.cs:37-148]
//   FFT   forward 2-D pencil FFT of every column  [AtoAGreenTensorCalculatorComponent.cs:197-279]
//
// A workgroup of K5 takes one cell: its threads form the weights of 32 segments at a time together, and each then
// sums them for a transceiver pair of its own, whose segment coefficients are read coalesced. Where pairs are few,
// groups of threads share a pair's segments.
#include "xtr_common.h"
#include "xtr_green.h"
#include "xtr_kernels.h"
#include "xtr_mfma.h"

#include <algorithm>
#include <complex>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

namespace xtr {

namespace {

constexpr int kTaps = 431;
constexpr int kL2 = 130;          // HankelCoefficients._l2: lambda index of 1/rho[0]
constexpr int kMaxLayers = 16;
constexpr double kPi = 3.14159265358979323846;
constexpr double kMu0 = 4.0 * kPi * 1.0E-07;

// ---- complex helpers (FP64) ---------------------------------------------------------------
__device__ inline double2 cexp_d(double2 z)
{
    double s, c;
    sincos(z.y, &s, &c);
    const double e = exp(z.x);
    return make_double2(e * c, e * s);
}

// principal square root
__device__ inline double2 csqrt_d(double2 z)
{
    const double a = z.x, b = z.y;
    if (a == 0 && b == 0) return make_double2(0, b);
    const double r = hypot(a, b);
    if (a >= 0) {
        const double t = sqrt(0.5 * (r + a));
        return make_double2(t, b / (2 * t));
    }
    const double t = sqrt(0.5 * (r - a));
    return make_double2(fabs(b) / (2 * t), copysign(t, b));
}

// a / b (Smith)
__device__ inline double2 cdiv_d(double2 a, double2 b)
{
    if (fabs(b.x) >= fabs(b.y)) {
        const double r = b.y / b.x, den = b.x + b.y * r;
        return make_double2((a.x + a.y * r) / den, (a.y - a.x * r) / den);
    }
    const double r = b.x / b.y, den = b.x * r + b.y;
    return make_double2((a.x * r + a.y) / den, (a.y * r - a.x) / den);
}

__device__ inline double2 c_(double re, double im = 0) { return make_double2(re, im); }
__device__ inline double2 operator+(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 operator-(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ inline double2 operator-(double2 a) { return make_double2(-a.x, -a.y); }
__device__ inline double2 operator*(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ inline double2 operator*(double s, double2 a) { return make_double2(s * a.x, s * a.y); }
__device__ inline double2 operator/(double2 a, double2 b) { return cdiv_d(a, b); }

// ---- K1: per (item, lambda) layer recursions ----------------------------------------------
struct LayerModel {
    int nl;
    double2 zeta[kMaxLayers];
    double thick[kMaxLayers];
    double depth[kMaxLayers + 1];   // depth[k] = top of layer k
    double omega;
};

// Bound by the chain of complex divisions, roots and exponentials through the layers: a quarter of the grid
// (blockIdx.z) runs each of the four recursions, with its layers' roots and exponentials in registers:
// 9 us for 5 layers where one thread with all four in scratch arrays took 18.
__global__ __launch_bounds__(64) void layer_aux_kernel(const LayerModel *lmp, int nitems, int nlam_max, const int *nlam, const double *lam,
                                 double2 *eta, double2 *ex, double2 *p1, double2 *q1, double2 *ps, double2 *qs)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    const int it = blockIdx.y;
    if (it >= nitems || m >= nlam[it]) return;
    const LayerModel &lm = *lmp;
    const int nl = lm.nl, n = nl - 1;
    const double l = lam[(int64_t)it * nlam_max + m];
    const int64_t base = ((int64_t)it * nlam_max + m) * nl;
    // value = i omega * zeta * Mu0; eta = sqrt(lambda^2 - value)  (CalcEta, green_scalar.c:30-34)
    auto root = [&](int k) { return csqrt_d(c_(l * l) - (c_(0, lm.omega) * lm.zeta[k]) * c_(kMu0)); };
    auto expo = [&](int k, double2 E) { return cexp_d((-2 * lm.thick[k]) * E); };    // CalcExp (green_scalar.c:36-41)
    // the sigma recursions carry the layers' zeta, the others 1
    const bool sig = blockIdx.z & 1;
    auto ratio = [&](int k, int j) { return sig ? lm.zeta[k] / lm.zeta[j] : c_(1); };
    if (blockIdx.z < 2) {
        // P: p[1] from the top interface, then downwards (CalculatePBelow1, PlanCalculatorFast.cs:266-280)
        double2 *out = (sig ? ps : p1) + base;
        double2 e0 = root(0), e1 = root(1);
        double2 v = sig ? (lm.zeta[0] * e1 - lm.zeta[1] * e0) / (lm.zeta[0] * e1 + lm.zeta[1] * e0) : (e1 - e0) / (e1 + e0);
        out[0] = c_(0);
        out[1] = v;
        if (!sig) {
            eta[base] = e0;
            eta[base + 1] = e1;
        }
        for (int k = 1; k < nl - 1; ++k) {
            e0 = e1;
            e1 = root(k + 1);
            const double2 pe = v * expo(k, e0);
            const double2 part = (ratio(k + 1, k) * (e0 / e1)) * ((pe - c_(1)) / (pe + c_(1)));
            v = (c_(1) + part) / (c_(1) - part);
            out[k + 1] = v;
            if (!sig) eta[base + k + 1] = e1;
        }
    } else {
        // Q: q[n] = 0 at the bottom, then upwards (CalculateQ, PlanCalculatorFast.cs:292-318)
        double2 *out = (sig ? qs : q1) + base;
        double2 e1 = root(n), e0 = root(n - 1);                      // of layers k, k - 1
        const double2 first = ratio(n - 1, n) * (e1 / e0);
        double2 v = (c_(1) - first) / (c_(1) + first);
        out[n] = c_(0);
        if (!sig) ex[base + n] = expo(n, e1);
        if (n > 1) out[0] = c_(0);
        out[n - 1] = v;
        for (int k = n - 1; k >= 0; --k) {
            e1 = e0;
            const double2 X = expo(k, e1);
            if (!sig) ex[base + k] = X;
            if (k > 0) e0 = root(k - 1);
            if (k <= 1) continue;
            const double2 qe = v * X;
            const double2 part = (ratio(k - 1, k) * (e1 / e0)) * ((qe - c_(1)) / (qe + c_(1)));
            v = (c_(1) + part) / (c_(1) - part);
            out[k - 1] = v;
        }
    }
}

// ---- K2: U1..U5 per (pair, item, lambda) ----------------------------------------------------
struct PairInfo {
    int r, s, t, b, kase;     // background layers of rc/tr, min/max; 0 match, 1 rc below, 2 rc above
    double r1, r2, s1, s2, dt, db1;
    double2 iz;               // 1 / (2 zeta_rc), times zeta_rc / zeta_tr where rc is the lower layer
};

// A[rc][tr] (CalculateA :160-200; CalculateASigma :138-158 for sigma = 1), A of the lower triangle with the ratio
// zeta_rc / zeta_tr for sigma = 1; ann_over: without that ratio and over den
__device__ inline double2 ann_over(const LayerModel &lm, const double2 *E, const double2 *X, const double2 *P,
                                   const double2 *Q, int rc, int tr, double2 den)
{
    const int smax = rc > tr ? rc : tr, rmin = rc < tr ? rc : tr;
    double2 prev = c_(1) / (E[smax] * (c_(1) - P[smax] * Q[smax] * X[smax]) * den);
    for (int k = smax - 1; k >= rmin; --k) {
        const double2 q = ((c_(1) + P[k + 1]) / (c_(1) + P[k] * X[k])) * cexp_d(lm.depth[k + 1] * (E[k + 1] - E[k]));
        prev = q * prev;
    }
    return prev;
}
__device__ inline double2 ann_at(const LayerModel &lm, const double2 *E, const double2 *X, const double2 *P,
                                 const double2 *Q, int rc, int tr, int sigma)
{
    const double2 a = ann_over(lm, E, X, P, Q, rc, tr, c_(1));
    return sigma && rc > tr ? (lm.zeta[rc] / lm.zeta[tr]) * a : a;
}

// The layer model lies in memory: indexed by a pair's layer, an argument would go through scratch.
__global__ __launch_bounds__(64) void pair_u_kernel(const LayerModel *lmp, int npairs, const PairInfo *pairs, int asym, int nitems,
                              int nlam_max, const int *nlam, const double *lam, const double2 *eta,
                              const double2 *ex, const double2 *p1, const double2 *q1, const double2 *ps,
                              const double2 *qs, double2 *U)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    const int it = blockIdx.y;
    const int p = blockIdx.z;
    if (it >= nitems || m >= nlam[it] || p >= npairs) return;
    const PairInfo pi = pairs[p];
    const LayerModel &lm = *lmp;
    const int nl = lm.nl;
    const int64_t base = ((int64_t)it * nlam_max + m) * nl;
    const double2 *E = eta + base, *X = ex + base;
    const double l = lam[(int64_t)it * nlam_max + m];
    const double2 er = E[pi.r], es = E[pi.s], et = E[pi.t], eb = E[pi.b];
    // PreCalculate (VolumeToVolumeCalculatorUFast.cs:34-46): T, R, C and D are each four exponentials, +- at the
    // two faces of either layer, that is the term at the faces that make it largest times (1 - e^(-tau_r eta_r))
    // (1 - e^(-tau_s eta_s)), tau the thicknesses. Six complex exponentials a thread instead of sixteen (they are
    // nearly all of its work: 1.25 -> 0.65 ms a build at 128 x 128 x 32, 0.42 ms with the registers a block of 64
    // threads may have instead of spills), and the differences of nearly equal
    // exponentials at small lambda lose one factor of eps / (tau eta) instead of the product of both: against 40
    // digits over 0 to 6 km, 1e-3 to 10 Hz and lambda 1e-9 to 3, the mean error falls from 2e-11..2e-14 to
    // 3e-14..4e-15. No intermediate exceeds the largest of the four terms.
    const double2 xr = cexp_d(-(pi.r2 - pi.r1) * er), xs = cexp_d(-(pi.s2 - pi.s1) * es);
    const double2 faces = (c_(1) - xr) * (c_(1) - xs);
    const double2 T = cexp_d(-pi.r1 * er - pi.s1 * es + 2 * pi.dt * et) * faces;
    const double2 Rv = cexp_d(-2 * pi.db1 * eb + pi.s2 * es + pi.r2 * er) * faces;
    double2 C = c_(0), D = c_(0);
    const double2 F = -2 * pi.db1 * eb + 2 * pi.dt * et;
    if (pi.kase == 2) {   // rc above tr: Ctop, Dtop
        C = cexp_d(-pi.s1 * es + pi.r2 * er) * faces;
        D = cexp_d(F + pi.s2 * es - pi.r1 * er) * faces;
    } else if (pi.kase == 1) {   // rc below tr: Cbot, Dbot
        C = cexp_d(-pi.r1 * er + pi.s2 * es) * faces;
        D = cexp_d(F - pi.s1 * es + pi.r2 * er) * faces;
    }
    const int ncomp = asym ? 1 : 3;
    double2 *out = U + (((int64_t)p * nitems + it) * ncomp) * nlam_max + m;
    // A complex division is some 60 instructions, and there were five or six a thread: the ones by zeta are per pair
    // (iz, with ann's ratio of zetas), those by eta go into ann's: 0.42 -> 0.35 ms.
    const double2 ee = asym ? es : er * es;
    for (int set = asym ? 1 : 0; set < 2; ++set) {
        const double2 *P = (set ? ps : p1) + base;
        const double2 *Q = (set ? qs : q1) + base;
        const double2 Pt = P[pi.t], Qb = Q[pi.b];
        const double2 annfac = ann_over(lm, E, X, P, Q, pi.r, pi.s, ee);
        double2 psi1, psi3;
        if (pi.kase == 0) {
            const int n = pi.r;
            const double tau = pi.r2 - pi.r1;
            const double dn1 = lm.depth[n + 1] - lm.depth[n];
            const double2 en = E[n];
            const double2 PQ = P[n] * Q[n];
            // CalcPsi1RcAndTrMatch (:313-332)
            const double2 part1 = tau * en - (c_(1) - xr);
            const double2 part2 = PQ * ((tau * en + c_(1)) * cexp_d(-2 * dn1 * en) - cexp_d(-2 * dn1 * en + tau * en));
            psi1 = 2.0 * (part1 - part2);
            psi3 = c_(0);
        } else if (pi.kase == 1) {
            psi1 = C + Pt * Qb * D;
            psi3 = -C + Pt * Qb * D;
        } else {
            psi1 = C + Pt * Qb * D;
            psi3 = C - Pt * Qb * D;
        }
        if (set == 0) {
            // U1 (:144-159), normalised by i omega Mu0 / 2
            const double2 u1 = annfac * (Pt * T + Qb * Rv + psi1);
            out[0] = u1 * (c_(0, lm.omega * kMu0) * c_(0.5));
            continue;
        }
        if (asym) {
            // U3 (:195-210), normalised by lambda / (2 zeta_rc)
            const double2 u3 = annfac * (-1.0 * (Pt * T) + Qb * Rv + psi3);
            out[0] = u3 * (l * pi.iz);
            return;
        }
        // U2 (:183-193), normalised by 1 / (2 zeta_rc)
        const double2 u2 = annfac * ee * (Pt * T + Qb * Rv - psi1);
        out[(int64_t)1 * nlam_max] = u2 * pi.iz;
        // U5 (:161-181, 290-311), normalised by lambda^2 / (2 zeta_rc)
        double2 u5;
        if (pi.kase == 0) {
            const int n = pi.r;
            const double tau = pi.r2 - pi.r1;
            const double ln = lm.thick[n];
            const double2 kk = (c_(0, lm.omega) * lm.zeta[n]) * c_(kMu0);
            const double2 en = E[n];
            const double2 PQ = P[n] * Q[n];
            const double2 part1 = -(c_(1) - xr);
            const double2 part2 = PQ * (cexp_d(-(2 * ln - tau) * en) - cexp_d(-2 * ln * en));
            const double2 part3 = ((1 / (l * l)) * kk) * (c_(1) - PQ * cexp_d(-2 * ln * en)) * (tau * en);
            const double2 psi5 = 2.0 * (part1 + part2 + part3);
            u5 = annfac * (Pt * T + Qb * Rv + psi5);
        } else {
            u5 = annfac * (Pt * T + Qb * Rv + psi1);
        }
        out[(int64_t)2 * nlam_max] = u5 * (l * l * pi.iz);
    }
}

// ---- K3: Hankel filter onto the merged rho grid -------------------------------------------
// For every (row p, item, component): I[k][c][p] = sgn_c (sum_j hank[430 - j] U[p][item][c][ix + j]) / (den rho_k),
// k the place of the item's radius ix among the merged radii; component c uses J0 where bit c of j0 is set.
// The filter is the same for every row, so the sums are a product of the banded Toeplitz matrix
// H[ix][lambda] = hank[430 - (lambda - ix)] with the rows' U: 16 radii x 4 lambdas x 8 rows (Re, Im) per
// 16x16x4 MFMA, one wave per 8 rows with up to 8 radius tiles at once, tiles outside the band skipped. H comes
// from a zero-padded filter in LDS, U straight from memory, read once. At 128 x 128 x 32 the 5 GFLOP take
// 136 us where one thread per radius, whose neighbours read other items' rows, took 1460.
struct HankelArgs {
    int np, nitems, ncomp, nlam_max, nrho_max;
    const double2 *U;
    const int *nlam, *mpos;       // mpos[item][ix]: the radius's place
    const double *radii, *h0, *h1;
    int j0;
    double sgn[5], den;
    double2 *I;
};
// TILES radius tiles a wave. Few rows leave most of the chip idle and a wave with 8 tiles is a chain of 2000 MFMAs:
// then a wave takes 2 tiles, and `groups` workgroups share the radii (the rows are read again, from L2):
// the 32 rows of a level at 128 x 128 x 32 take 21 us instead of 47, the 36 and 64 of 32 x 32 x 8 20 instead of 37.
template <int TILES>
__global__ __launch_bounds__(256) void hankel_kernel(HankelArgs a, int groups)
{
    constexpr int PAD = 16 * TILES - 1, STEPS = (kTaps - 1 + 16 * TILES + 15) / 16 * 4;   // k-steps of a full group
    constexpr int TABLE = PAD + 4 * STEPS;
    __shared__ double h[TABLE];
    const int it = blockIdx.y, c = blockIdx.z;
    const double *hank = (a.j0 >> c) & 1 ? a.h0 : a.h1;
    for (int x = threadIdx.x; x < TABLE; x += blockDim.x) {
        const int j = x - PAD;
        h[x] = j >= 0 && j < kTaps ? hank[kTaps - 1 - j] : 0.0;
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int grp = blockIdx.x % groups, p0 = ((int)blockIdx.x / groups * 4 + wave) * 8;
    if (p0 >= a.np) return;
    const int n = lane & 15, kl = lane >> 4, p = p0 + (n >> 1), part = n & 1;
    const int nlam = a.nlam[it], nrho = nlam - kTaps;
    const double *u = reinterpret_cast<const double *>(
                          a.U + (((int64_t)min(p, a.np - 1) * a.nitems + it) * a.ncomp + c) * a.nlam_max) + part;
    const double *hl = h + PAD + kl - n;                             // H[i = n][k = kl], plus 4 step - 16 tile
    for (int ix0 = 16 * TILES * grp; ix0 < nrho; ix0 += 16 * TILES * groups) {
        const int tiles = min(TILES, (nrho - ix0 + 15) / 16);
        const int chunks = (kTaps - 1 + 16 * tiles + 15) / 16;         // of 4 k-steps
        auto get = [&](int step) __attribute__((always_inline)) {      // past the row's end: no radius uses it
            const int k = ix0 + 4 * step + kl;
            const double v = u[2 * min(k, nlam - 1)];
            return k < nlam ? v : 0.0;
        };
        mfma_d4 acc[TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t) acc[t] = mfma_d4{0, 0, 0, 0};
        double bn[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) bn[q] = get(q);
        for (int ch = 0; ch < chunks; ++ch) {
            double b[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) b[q] = bn[q];
#pragma unroll
            for (int q = 0; q < 4; ++q) bn[q] = get(4 * (ch + 1) + q);
            const double *hc = hl + 16 * ch;
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                // radii 16 t .. 16 t + 15 use lambdas 16 t .. 16 t + 15 + 430 of this group
                if (t < tiles && t <= ch && 16 * ch <= 16 * t + 15 + kTaps - 1) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[t] = mfma16(hc[4 * q - 16 * t], b[q], acc[t]);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ix = ix0 + 16 * t + mfma_row<double>(lane, r);
                if (ix < nrho && p < a.np) {
                    const int k = a.mpos[it * a.nrho_max + ix];
                    reinterpret_cast<double *>(a.I)[(((int64_t)k * a.ncomp + c) * a.np + p) * 2 + part] =
                        a.sgn[c] * acc[t][r] / (a.den * a.radii[k]);
                }
            }
    }
}

void launch_hankel(const HankelArgs &a, hipStream_t s)
{
    const int64_t rows = ceil_div(a.np, 32);
    // fewer waves than SIMDs
    if (4 * rows * a.nitems * a.ncomp < 4 * device_cus()) {
        const int groups = (int)ceil_div(a.nrho_max, 32);
        hipLaunchKernelGGL(hankel_kernel<2>, dim3((unsigned)(rows * groups), a.nitems, a.ncomp), dim3(256), 0, s, a, groups);
    } else {
        hipLaunchKernelGGL(hankel_kernel<8>, dim3((unsigned)rows, a.nitems, a.ncomp), dim3(256), 0, s, a, 1);
    }
    XTR_LAUNCH_CHECK("hankel_kernel");
}

// ---- K4: segments --------------------------------------------------------------------------
// segA, segB and I are [k][comp][row]; `stride` values per radius
__global__ __launch_bounds__(256) void segments_kernel(int64_t stride, int64_t total, const double *radii, const double2 *I,
                                                       double2 *segA, double2 *segB)
{
    for (int64_t o = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; o < total; o += (int64_t)gridDim.x * blockDim.x) {
        const int64_t k = o / stride;
        const double s = radii[k], u = radii[k + 1], div = u - s;
        const double2 i0 = I[o], i1 = I[o + stride];
        const double2 a = make_double2((i1.x - i0.x) / div, (i1.y - i0.y) / div);
        segA[o] = a;
        segB[o] = make_double2(i0.x - a.x * s, i0.y - a.y * s);
    }
}

void launch_segments(int ncomp, int np, int nmerged, const double *radii, const double2 *I, double2 *segA, double2 *segB,
                     hipStream_t s)
{
    const int64_t stride = (int64_t)ncomp * np, total = (nmerged - 1) * stride;
    hipLaunchKernelGGL(segments_kernel, dim3((unsigned)std::min<int64_t>(ceil_div(total, 256), 4096)), dim3(256), 0, s,
                       stride, total, radii, I, segA, segB);
    XTR_LAUNCH_CHECK("segments_kernel");
}

// ---- K5: lateral integration, mirroring, device layout ---------------------------------------
struct Knot { int index; double radius; };

__device__ inline Knot make_knot(const double *radii, int nr, double x, double y)
{
    const double r = sqrt(x * x + y * y);
    int lo = 0, hi = nr - 1, idx = -1;
    while (lo <= hi) {
        const int mid = lo + (hi - lo) / 2;
        const double v = radii[mid];
        if (v == r) { idx = mid; break; }
        if (v < r) lo = mid + 1; else hi = mid - 1;
    }
    if (idx < 0) idx = lo - 1;
    if (idx == nr - 1) idx--;
    if (idx < 0) idx = 0;
    return Knot{idx, r};
}

struct Factors { double d1a, d1b, d2a, d2b, d3a, d3b; };

__device__ inline Factors factors(double s, double u, double rs, double ru, double v)
{
    Factors f;
    const double lg = log((u + ru) / (s + rs));
    f.d1a = v == 0 ? (u * ru - s * rs) / 2 : (u * ru - s * rs + v * v * lg) / 2;
    f.d1b = u - s;
    f.d2a = v == 0 ? 0 : -(u - s) * v;
    f.d2b = v == 0 ? 0 : -(v * lg);
    f.d3a = -(u * u - s * s) / 2;
    f.d3b = -(ru - rs);
    return f;
}

struct LatArgs {
    int nx, ny, nz, npairs;
    int p0;                       // first pair of this chunk
    int width;                    // threads, and pairs, of a group
    int cols, skip;               // cells of blockIdx.x: rows of cols, those with i, j < skip left out
    int folded;                   // G holds blocks [Nx+1][Ny+1], else [2Nx][2Ny]
    double dx, dy;
    const double2 *segA, *segB;   // [seg][comp][pair]
    const double *radii;
    const Knot *knots;            // of cell i ny + j
    double2 *G;
    int64_t gblk;
    int64_t off[4];               // component offsets in the per-wavenumber block, q-order
    int xs[4], ys[4];             // mirror parities, q-order
};

// One stretch of an edge with its ends on one side of the axis: at distance v from the other axis, from s to u
// along it, through the segments left.index .. right.index (Integrate, GreenTensorCalculator.cs:367-411).
struct Stretch {
    Knot left, right;
    double s, u, v;
    int sign, mirrored;           // sign of the edge; the stretch lies on the axis's negative side
    __device__ Factors at(const double *radii, int e) const
    {
        const int i = left.index + e;
        const bool first = e == 0, last = i == right.index;
        const double r1 = first ? left.radius : radii[i], r2 = last ? right.radius : radii[i + 1];
        return factors(first ? s : sqrt(r1 * r1 - v * v), last ? u : sqrt(r2 * r2 - v * v), r1, r2, v);
    }
};

// Stretch e = 0..7 of the four edges of a cell (x1, x2) x (y1, y2): edges along x at y1 (sign -1) and y2 (+1), then
// along y at x1, x2 (RunAlongX :254-298, RunAlongY :318-361), each in one stretch, or in two from the axis outwards
// where it crosses it; false: this one does not exist.
struct StretchEnds {
    double s, u, v;               // along the edge, and its distance from the axis parallel to it
    double l, r;                  // the coordinates along the edge whose radii bound it
    int sign, mirrored;
};
__device__ inline bool stretch_ends(int e, double x1, double x2, double y1, double y2, StretchEnds &t)
{
    const int along_y = e >> 2, far = (e >> 1) & 1, half = e & 1;
    const double a1 = along_y ? y1 : x1, a2 = along_y ? y2 : x2;
    t.v = along_y ? (far ? x2 : x1) : (far ? y2 : y1);
    t.sign = far ? 1 : -1;
    t.mirrored = 0;
    const int pos = (int)(a1 > 0) & (int)(a2 > 0), neg = (int)(a1 < 0) & (int)(a2 < 0);
    if (pos) { t.s = t.l = a1; t.u = t.r = a2; return half == 0; }
    if (neg) { t.l = a2; t.r = a1; t.s = -a2; t.u = -a1; t.mirrored = 1; return half == 0; }
    t.s = t.l = 0;
    if (half == 0) { t.u = -a1; t.r = a1; t.mirrored = 1; }
    else { t.u = t.r = a2; }
    return true;
}

// The two ends of a cell's eight stretches among the radii: thread (cell, stretch, side), cells (i, j), i from i0,
// j from j0, ncy a row. A binary search is a chain of a dozen loads, which every workgroup of a cell went through
// before it could start: at 128 x 128 x 32 9 us here, lateral_kernel 0.73 -> 0.60 ms and atoo_lateral_kernel 60
// and 50 -> 44 and 36 us.
__global__ __launch_bounds__(256) void knots_kernel(const double *radii, int nr, double dx, double dy, double xs, double ys,
                                                    int i0, int j0, int ncy, int cells, Knot *knots)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x, cell = t >> 4, e = (t >> 1) & 7;
    if (cell >= cells) return;
    const int i = i0 + cell / ncy, j = j0 + cell % ncy;
    StretchEnds st;
    stretch_ends(e, dx * (i - 0.5) - xs, dx * (i + 0.5) - xs, dy * (j - 0.5) - ys, dy * (j + 0.5) - ys, st);
    const double c = t & 1 ? st.r : st.l;
    knots[t] = e < 4 ? make_knot(radii, nr, c, st.v) : make_knot(radii, nr, st.v, c);
}

// The four edge integrals of one cell (x1, x2) x (y1, y2) as weights on the segments I_c(rho) = A_c rho + B_c they
// cross. A component's value is sum over segments of w . (A, B); w holds, for the edges along x and along y, the
// signed factors d1, d2, d3 (each for A and B) summed over the edge pair: sign -1 for the nearer edge, +1 for the
// farther. What FillResultAlongX/Y (:413-437) multiply by the QSigns tables (QSign.cs:31-38, 64-67) is a sign of
// the component and, for d3 only, the opposite sign on a stretch mirrored about the axis (rows AlongXSymm,
// AlongYSymm); the latter is in the weights here, the former with the components' sums.
// The weights are the same for every pair of layers, so a team of threads forms them once in LDS, from the knots
// that knots_kernel found: a logarithm and two square roots for each (segment, stretch), then the sums. Each
// coefficient is then read once per cell and segment instead of once per edge and segment.
enum { W1A, W1B, W2A, W2B, W3A, W3B, WN };
template <int SEGS>
struct CellWeights {
    Stretch st[8];
    int is[8];
    double f[SEGS][8][WN];
    double w[SEGS][2][WN];        // [edges along x, along y]
    // the cell's stretches, their ends from knots_kernel; range returns the segments they cross (after the team's
    // next sync)
    __device__ void ends(int tid, const Knot *knots, double x1, double x2, double y1, double y2)
    {
        if (tid >= 16) return;
        const int e = tid >> 1, side = tid & 1;
        const Knot k = knots[tid];
        StretchEnds t;
        const bool there = stretch_ends(e, x1, x2, y1, y2, t);
        if (side) {
            st[e].right = k;
        } else {
            st[e].left = k;
            st[e].s = t.s;
            st[e].u = t.u;
            st[e].v = t.v;
            st[e].sign = t.sign;
            st[e].mirrored = t.mirrored;
            is[e] = there;
        }
    }
    __device__ void range(int &lo, int &hi) const
    {
        lo = 1 << 30;
        hi = -1;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (is[e]) {
                lo = min(lo, st[e].left.index);
                hi = max(hi, st[e].right.index);
            }
    }
    __device__ void factors_of(int tid, int nt, const double *radii, int seg0, int n)
    {
        for (int t = tid; t < 8 * n; t += nt) {
            const int k = t >> 3, e = t & 7, i = seg0 + k - st[e].left.index;
            double d[WN] = {0, 0, 0, 0, 0, 0};
            if (is[e] && i >= 0 && seg0 + k <= st[e].right.index) {
                const Factors q = st[e].at(radii, i);
                const double sg = st[e].sign, s3 = st[e].mirrored ? sg : -sg;
                d[W1A] = sg * q.d1a; d[W1B] = sg * q.d1b;
                d[W2A] = sg * q.d2a; d[W2B] = sg * q.d2b;
                d[W3A] = s3 * q.d3a; d[W3B] = s3 * q.d3b;
            }
#pragma unroll
            for (int c = 0; c < WN; ++c) f[k][e][c] = d[c];
        }
    }
    __device__ void sum(int tid, int nt, int n)
    {
        for (int t = tid; t < 2 * WN * n; t += nt) {
            const int k = t / (2 * WN), r = t % (2 * WN), ax = r / WN, c = r % WN;
            w[k][ax][c] = (f[k][4 * ax][c] + f[k][4 * ax + 1][c]) + (f[k][4 * ax + 2][c] + f[k][4 * ax + 3][c]);
        }
    }
};

__device__ __forceinline__ double2 wab(const double (&w)[WN], int c, double2 q, double2 A, double2 B)
{
    return make_double2(fma(w[c], A.x, fma(w[c + 1], B.x, q.x)), fma(w[c], A.y, fma(w[c + 1], B.y, q.y)));
}

// One workgroup per cell and a share of the pairs; groups of `width` threads share the segments between them, and
// their sums meet in LDS. Bound by the L2 reads of the segments' coefficients (96 bytes a pair and segment) on a
// large grid, and on a small one by the chain of the cells next to the source, which cross up to 200 segments. At
// 128 x 128 x 32, 256 pairs a group: 0.60 ms for both sets; 3.6 ms with every thread working out the edges'
// geometry for its own pair, 1.16 ms with the geometry shared but one pass over the segments per edge.
// 32 x 32 x 8 (64 and 36 pairs), 4 groups of 64 against one: 38 and 101 us a set, each with its searches.
constexpr int kCellSegs = 32, kNearCells = 8;

template <int ASYM, bool GROUPS>
__global__ __launch_bounds__(256) void lateral_kernel(LatArgs a)
{
    __shared__ CellWeights<kCellSegs> cw;
    const int64_t cell = blockIdx.x;
    const int i = (int)(cell / a.cols), j = (int)(cell % a.cols);
    if (i < a.skip && j < a.skip) return;
    const int grp = GROUPS ? threadIdx.x / a.width : 0, tp = threadIdx.x - grp * a.width;
    const int groups = GROUPS ? blockDim.x / a.width : 1;
    const int p = blockIdx.y * a.width + tp, np = a.npairs;
    cw.ends(threadIdx.x, a.knots + (i * a.ny + j) * 16, a.dx * (i - 0.5), a.dx * (i + 0.5), a.dy * (j - 0.5),
            a.dy * (j + 0.5));
    __syncthreads();
    int lo, hi;
    cw.range(lo, hi);
    // asym {xz, yz}; symm {xx, yy, zz, xy}
    constexpr int nq = ASYM ? 2 : 4;
    double2 G[nq];
#pragma unroll
    for (int t = 0; t < nq; ++t) G[t] = c_(0);
    for (int seg0 = lo; seg0 <= hi; seg0 += kCellSegs) {
        const int n = min(kCellSegs, hi - seg0 + 1);
        cw.factors_of(threadIdx.x, blockDim.x, a.radii, seg0, n);
        __syncthreads();
        cw.sum(threadIdx.x, blockDim.x, n);
        __syncthreads();
        if (p < np)
#pragma unroll 2
            for (int k = grp; k < n; k += groups) {
                const double (&wx)[WN] = cw.w[k][0], (&wy)[WN] = cw.w[k][1];
                const int64_t o = (int64_t)(seg0 + k) * (ASYM ? 1 : 3) * np + p;
                if constexpr (ASYM) {      // edges along y give xz, along x yz (AddToQBuff..., D1)
                    const double2 A3 = a.segA[o], B3 = a.segB[o];
                    G[0] = wab(wy, W1A, G[0], A3, B3);
                    G[1] = wab(wx, W1A, G[1], A3, B3);
                } else {                   // AddToQBuffAlongXElectric (:505-516), AlongY (:517-528)
                    const double2 A1 = a.segA[o], B1 = a.segB[o], A2 = a.segA[o + np], B2 = a.segB[o + np];
                    const double2 A5 = a.segA[o + 2 * np], B5 = a.segB[o + 2 * np];
                    const double nyw[WN] = {0, 0, -wy[W2A], -wy[W2B], 0, 0}, nxw[WN] = {0, 0, -wx[W2A], -wx[W2B], 0, 0};
                    G[0] = wab(nyw, W2A, wab(wx, W2A, G[0], A1, B1), A2, B2);
                    G[1] = wab(nxw, W2A, wab(wy, W2A, G[1], A1, B1), A2, B2);
                    G[2] = wab(nyw, W2A, wab(nxw, W2A, G[2], A5, B5), A5, B5);
                    G[3] = wab(wy, W3A, wab(wx, W3A, G[3], A2, B2), A1, B1);
                }
            }
        __syncthreads();                                       // the weights are read
    }
    if constexpr (GROUPS) {
        static_assert(sizeof(cw.f) >= 2 * 256 * sizeof(double2), "two components of 256 threads");
        double2 *red = reinterpret_cast<double2 *>(cw.f);
#pragma unroll
        for (int t = 0; t < nq; t += 2) {
            if (t) __syncthreads();
            red[threadIdx.x] = G[t];
            red[256 + threadIdx.x] = G[t + 1];
            __syncthreads();
            if (grp == 0)
                for (int o = a.width; o < (int)blockDim.x; o += a.width) {
                    G[t] = cadd<double>(G[t], red[o + tp]);
                    G[t + 1] = cadd<double>(G[t + 1], red[256 + o + tp]);
                }
        }
    }
    if (p >= np || grp > 0) return;
    // write G(i,j) and, into a full tensor, its mirror images (GreenTensorFftPopulator.cs:88-148); of a folded
    // one the FFT forms the images from the parities as it reads
    const int64_t nx2 = 2LL * a.nx, ny2 = a.folded ? a.ny + 1 : 2LL * a.ny;
    // asym pairs are rc-major (p = rc*nz + tr); the device block stores them swizzled
    const int pa = a.p0 + p;
    const int pd = ASYM ? asym_pos(pa / a.nz, pa % a.nz, a.nz, asym_swizzle_mask(a.nz)) : pa;
#pragma unroll
    for (int t = 0; t < nq; ++t) {
        const int64_t o = a.off[t] + pd;
        const double2 g = G[t];
        a.G[((int64_t)i * ny2 + j) * a.gblk + o] = g;
        if (a.folded) continue;
        if (i >= 1) a.G[((nx2 - i) * ny2 + j) * a.gblk + o] = (double)a.xs[t] * g;
        if (j >= 1) a.G[((int64_t)i * ny2 + (ny2 - j)) * a.gblk + o] = (double)a.ys[t] * g;
        if (i >= 1 && j >= 1) a.G[((nx2 - i) * ny2 + (ny2 - j)) * a.gblk + o] = (double)(a.xs[t] * a.ys[t]) * g;
    }
}

void launch_knots(const double *radii, int nr, double dx, double dy, double xs, double ys, int i0, int j0, int ncy,
                  int64_t cells, Knot *knots, hipStream_t s)
{
    hipLaunchKernelGGL(knots_kernel, dim3((unsigned)ceil_div(16 * cells, 256)), dim3(256), 0, s, radii, nr, dx, dy, xs, ys, i0,
                       j0, ncy, (int)cells, knots);
    XTR_LAUNCH_CHECK("knots_kernel");
}

// ---- host: plans ------------------------------------------------------------------------------
// HankelCoefficients.GetLog10RhoStep (:67): (float)Math.Pow(10, 1/_ndec) with _ndec a float 40
double log10_rho_step()
{
    const float inv = 1.0f / 40.0f;
    return (double)(float)std::pow(10.0, (double)inv);
}

struct HostPlan {
    std::vector<std::vector<double>> rho, lam;
    std::vector<double> merged;           // with a zero-rho plan, merged[0] = 0 and m_item[0] = -1
    std::vector<int> m_item, m_idx;
    bool zero_rho = false;
};

// ScalarPlansCreater.CreateFor (:102-110) over [rmin, rmax]; zero_rho puts rho = 0 in front of the
// merged radii (ScalarPlan.GetSortedRho :56-65, GreenScalarCalculator.CalculateZeroRho :147-157)
HostPlan make_plan(int number_of_hankels, double rmin, double rmax, bool zero_rho)
{
    HostPlan hp;
    hp.zero_rho = zero_rho;
    const int nh = std::abs(number_of_hankels);
    if (nh < 1 || !(rmin > 0)) throw hip_error("scalar plan needs NumberOfHankels >= 1 and rho_min > 0");
    const double step = log10_rho_step();
    std::vector<double> r1;                                                 // CreateRhoFromMin :142-157
    for (double nr = rmin; nr <= rmax; nr *= step) r1.push_back(nr);
    r1.push_back(r1.back() * step);
    const double rr2 = r1[r1.size() - 1], rr1 = r1[r1.size() - 2];
    const double st = (rr2 - rr1) / nh;
    hp.rho.push_back(r1);
    for (int i = 1; i < nh; ++i) {                                          // CreateRhoFromMax :159-176
        std::vector<double> rn;
        double nr = rr2 - i * st;
        while (nr >= rmin) {
            rn.push_back(nr);
            nr /= step;
        }
        rn.push_back(nr);
        std::reverse(rn.begin(), rn.end());
        hp.rho.push_back(rn);
    }
    for (auto &rho : hp.rho) {                                              // ScalarPlan.cs:76-97
        const int nlam = kTaps + (int)rho.size();
        std::vector<double> k(nlam);
        k[kL2] = 1 / rho[0];
        for (int i = kL2 + 1; i <= nlam - 1; ++i) k[i] = k[i - 1] / step;
        for (int i = kL2 - 1; i >= 0; --i) k[i] = k[i + 1] * step;
        hp.lam.push_back(k);
    }
    struct E { double r; int it, ix; };                                     // InnerResultsCombiner.cs:19-33
    std::vector<E> all;
    for (int it = 0; it < nh; ++it)
        for (int ix = 0; ix < (int)hp.rho[it].size(); ++ix) all.push_back({hp.rho[it][ix], it, ix});
    std::stable_sort(all.begin(), all.end(), [](const E &a, const E &b) { return a.r < b.r; });
    if (zero_rho) {
        hp.merged.push_back(0.0);
        hp.m_item.push_back(-1);
        hp.m_idx.push_back(0);
    }
    for (auto &e : all) {
        if ((int)hp.merged.size() > (int)zero_rho && hp.merged.back() == e.r) continue;
        hp.merged.push_back(e.r);
        hp.m_item.push_back(e.it);
        hp.m_idx.push_back(e.ix);
    }
    if (hp.merged.size() != all.size() + (zero_rho ? 1 : 0))
        throw hip_error("scalar plan has duplicate rho values; the reference's radii and scalars would misalign");
    return hp;
}

// the anomaly's own range, CreateForAnomalyToAnomaly (ScalarPlansCreater.cs:95-100, 360-380)
HostPlan make_plan(const GreenInput &in)
{
    const double h1 = in.dx / 2, h2 = in.dy / 2;
    const double mx = in.g.nx * in.dx - h1, my = in.g.ny * in.dy - h2;
    return make_plan(in.number_of_hankels, std::min(h1, h2), std::sqrt(mx * mx + my * my), false);
}

// FindRhoMin along one axis (ScalarPlansCreater.cs:245-266) for a level shifted by `shift` against
// the cell centres 0, h, ..., (n - 1) h. The reference's System.Decimal arithmetic and these doubles
// agree whenever h and the shift are whole multiples of a power-of-two fraction of a metre.
double level_rho_min_axis(int n, double h, double shift)
{
    const double a0 = -h / 2, a1 = n * h - h / 2;
    const double y0 = shift - h / 2, y1 = y0 + h * n;
    if ((y0 >= a0 && y0 <= a1) || (y1 >= a0 && y1 <= a1)) {
        const double rem = std::fmod(std::fabs(a0 - y0), h);
        return rem == 0 ? h / 2 : std::fabs(h / 2 - rem);
    }
    const double c1 = h * (n - 1);
    return std::min(std::min(std::fabs(y0), std::fabs(y0 - c1)), std::min(std::fabs(y1), std::fabs(y1 - c1)));
}

// CreateForAnomalyToObservationLevels (:51-66) for one level shifted by (sx, sy): FindRhoMax over
// the anomaly's corner cells and the level footprint's corners (:200-236), FindRhoMin (:238-243),
// and a zero-rho plan from 0.001 min(dx, dy) when the minimum is 0.
HostPlan make_level_plan(const GreenInput &in, double sx, double sy)
{
    const double ex = in.dx * (in.g.nx - 1), ey = in.dy * (in.g.ny - 1);
    const double x1 = sx - in.dx / 2, y1 = sy - in.dy / 2;
    const double x2 = x1 + in.dx * in.g.nx, y2 = y1 + in.dy * in.g.ny;
    const double ax[4] = {0, 0, ex, ex}, ay[4] = {0, ey, ey, 0};
    const double cx[4] = {x1, x2, x2, x1}, cy[4] = {y1, y1, y2, y2};
    double rmax = 0;
    for (int a = 0; a < 4; ++a)
        for (int c = 0; c < 4; ++c)
            rmax = std::max(rmax, std::sqrt((cx[c] - ax[a]) * (cx[c] - ax[a]) + (cy[c] - ay[a]) * (cy[c] - ay[a])));
    double rmin = std::min(level_rho_min_axis(in.g.nx, in.dx, sx), level_rho_min_axis(in.g.ny, in.dy, sy));
    const bool zero = rmin <= 0;
    if (zero) rmin = std::min(in.dx, in.dy) * 0.001;
    return make_plan(in.number_of_hankels, rmin, rmax, zero);
}

// Host arrays that one copy takes to the device: add() returns where an array lies in it.
struct Pack {
    std::vector<unsigned char> bytes;
    template <typename T> size_t add(const std::vector<T> &v)
    {
        const size_t at = bytes.size();
        bytes.resize(at + GreenScratch::padded(v.size() * sizeof(T)));
        std::memcpy(bytes.data() + at, v.data(), v.size() * sizeof(T));
        return at;
    }
};

// The scalar plan and the filter on the device, and the layer recursions of every (item, lambda).
struct PlanDev {
    const int *nlam, *mpos;
    const double *lam, *radii, *h0, *h1;
    const LayerModel *lm;
    double2 *eta, *ex, *p1, *q1, *ps, *qs;
};
struct PlanHost {
    int nitems = 0, nlam_max = 0, nmerged = 0, nrho_max = 0;
    std::vector<int> nlam;
    Pack pack;
    size_t at[7];
    size_t auxn = 0;
    PlanHost(const HostPlan &hp, const GreenInput &in, const LayerModel &lm)
    {
        nitems = (int)hp.rho.size();
        nmerged = (int)hp.merged.size();
        for (auto &l : hp.lam) {
            nlam.push_back((int)l.size());
            nlam_max = std::max(nlam_max, nlam.back());
        }
        std::vector<double> flat((size_t)nitems * nlam_max, 0.0);
        for (int it = 0; it < nitems; ++it) std::copy(hp.lam[it].begin(), hp.lam[it].end(), flat.begin() + (size_t)it * nlam_max);
        at[0] = pack.add(nlam);
        nrho_max = nlam_max - kTaps;
        std::vector<int> mpos((size_t)nitems * nrho_max, 0);
        for (int k = 0; k < nmerged; ++k)
            if (hp.m_item[k] >= 0) mpos[(size_t)hp.m_item[k] * nrho_max + hp.m_idx[k]] = k;
        at[1] = pack.add(mpos);
        at[2] = pack.add(flat);
        at[3] = pack.add(hp.merged);
        at[4] = pack.add(in.hank0);
        at[5] = pack.add(in.hank1);
        at[6] = pack.add(std::vector<LayerModel>{lm});
        auxn = (size_t)nitems * nlam_max * lm.nl;
    }
    size_t device_bytes() const
    {
        return GreenScratch::padded(pack.bytes.size()) + 6 * GreenScratch::padded(auxn * sizeof(double2));
    }
    // uploads the pack (its device address into base) and runs the recursions; the pack must outlive them
    PlanDev upload(GreenScratch &work, unsigned char *&base, hipStream_t s) const
    {
        base = work.take<unsigned char>(pack.bytes.size());
        XTR_CHECK(hipMemcpyAsync(base, pack.bytes.data(), pack.bytes.size(), hipMemcpyHostToDevice, s));
        PlanDev d;
        d.nlam = (const int *)(base + at[0]);
        d.mpos = (const int *)(base + at[1]);
        d.lam = (const double *)(base + at[2]);
        d.radii = (const double *)(base + at[3]);
        d.h0 = (const double *)(base + at[4]);
        d.h1 = (const double *)(base + at[5]);
        d.lm = (const LayerModel *)(base + at[6]);
        double2 **aux[6] = {&d.eta, &d.ex, &d.p1, &d.q1, &d.ps, &d.qs};
        for (auto *a : aux) *a = work.take<double2>(auxn);
        dim3 grid((unsigned)ceil_div(nlam_max, 64), nitems, 4);
        hipLaunchKernelGGL(layer_aux_kernel, grid, dim3(64), 0, s, d.lm, nitems, nlam_max, d.nlam, d.lam, d.eta, d.ex,
                           d.p1, d.q1, d.ps, d.qs);
        XTR_LAUNCH_CHECK("layer_aux_kernel");
        return d;
    }
};

LayerModel layer_model(const GreenInput &in)
{
    const int nl = (int)in.section.thickness.size();
    if (nl > kMaxLayers) throw hip_error("too many background layers for the device recursion");
    LayerModel lm{};
    lm.nl = nl;
    lm.omega = in.omega;
    const double eps0 = 1.0 / (kMu0 * 299792458.0 * 299792458.0);
    double d = in.section.zero_level;
    for (int k = 0; k < nl; ++k) {
        lm.zeta[k] = make_double2(in.section.sigma[k], -in.omega * eps0);
        lm.thick[k] = in.section.thickness[k];
        lm.depth[k] = d;
        d += in.section.thickness[k];
    }
    lm.depth[nl] = d;
    return lm;
}

int layer_at_depth(const Section &s, double depth)   // ScalarMathUtils.cs:15-31
{
    const int k = layer_index_at_depth(s, depth);
    if (k < 0) throw hip_error("anomaly is not within 1D section");
    return k;
}

}  // namespace

// The pairs of one set pass through the stages in equal chunks whose U stays in the 256 MB Infinity Cache
// between pair_u and hankel, which also bounds the scratch (about 250 MB) whatever nz.
constexpr size_t kChunkBytes = (size_t)160 << 20;

void build_green_atoa(const GreenInput &in, GreenScratch &work, double2 *G, bool folded, const double2 *tw_x,
                      const double2 *tw_y, hipStream_t s)
{
    const Geom &g = in.g;
    const int nz = g.nz;
    const LayerModel lm = layer_model(in);
    const HostPlan hp = make_plan(in);
    PlanHost ph(hp, in, lm);

    // transceiver pairs: Combine (rc-major) for asym, CombineSymm (tr-major, rc <= tr) for symm
    std::vector<PairInfo> pairs[2];
    auto add = [&](int asym, int rc, int tr) {
        PairInfo pi{};
        pi.r1 = in.depth[rc];
        pi.r2 = in.depth[rc] + in.thick[rc];
        pi.s1 = in.depth[tr];
        pi.s2 = in.depth[tr] + in.thick[tr];
        pi.r = layer_at_depth(in.section, pi.r1 + (pi.r2 - pi.r1) / 2);
        pi.s = layer_at_depth(in.section, pi.s1 + (pi.s2 - pi.s1) / 2);
        pi.t = std::min(pi.r, pi.s);
        pi.b = std::max(pi.r, pi.s);
        pi.dt = lm.depth[pi.t];
        pi.db1 = lm.depth[pi.b + 1];
        const std::complex<double> zr(lm.zeta[pi.r].x, lm.zeta[pi.r].y), zs(lm.zeta[pi.s].x, lm.zeta[pi.s].y);
        const std::complex<double> iz = 0.5 / (pi.r > pi.s ? zs : zr);
        pi.iz = make_double2(iz.real(), iz.imag());
        const double zw = pi.r1 + (pi.r2 - pi.r1) / 2;
        pi.kase = (zw > pi.s1 && zw < pi.s2) ? 0 : (zw >= pi.s2 ? 1 : 2);
        pairs[asym].push_back(pi);
    };
    for (int rc = 0; rc < nz; ++rc)
        for (int tr = 0; tr < nz; ++tr) add(1, rc, tr);
    for (int tr = 0; tr < nz; ++tr)
        for (int rc = 0; rc <= tr; ++rc) add(0, rc, tr);
    size_t pairs_at[2];
    int chunk[2];
    size_t need[4] = {0, 0, 0, 0};
    for (int asym = 0; asym < 2; ++asym) {
        pairs_at[asym] = ph.pack.add(pairs[asym]);
        const int np = (int)pairs[asym].size(), ncomp = asym ? 1 : 3;
        const size_t u1 = (size_t)ph.nitems * ncomp * ph.nlam_max;     // U of one pair
        const int64_t chunks = ceil_div((int64_t)(np * u1 * sizeof(double2)), (int64_t)kChunkBytes);
        chunk[asym] = (int)std::min<int64_t>(np, ceil_div(ceil_div(np, chunks), 8) * 8);   // 8 rows a wave of hankel
        need[0] = std::max(need[0], chunk[asym] * u1);
        need[1] = std::max(need[1], (size_t)chunk[asym] * ncomp * ph.nmerged);
        need[2] = need[3] = need[1];
    }
    const int64_t cells = (int64_t)g.nx * g.ny;
    size_t bytes = ph.device_bytes() + GreenScratch::padded(16 * cells * sizeof(Knot));
    for (size_t n : need) bytes += GreenScratch::padded(n * sizeof(double2));
    work.reserve(bytes);
    unsigned char *base;
    const PlanDev d = ph.upload(work, base, s);
    double2 *U = work.take<double2>(need[0]), *I = work.take<double2>(need[1]), *segA = work.take<double2>(need[2]),
            *segB = work.take<double2>(need[3]);
    Knot *knots = work.take<Knot>(16 * cells);
    launch_knots(d.radii, ph.nmerged, in.dx, in.dy, 0.0, 0.0, 0, 0, g.ny, cells, knots, s);
    if (!folded) XTR_CHECK(hipMemsetAsync(G, 0, (size_t)g.L() * g.gblk() * sizeof(double2), s));

    const int nitems = ph.nitems, nlam_max = ph.nlam_max, nmerged = ph.nmerged;
    for (int asym = 1; asym >= 0; --asym) {
        const int ncomp = asym ? 1 : 3, all = (int)pairs[asym].size();
        for (int p0 = 0; p0 < all; p0 += chunk[asym]) {
            const int np = std::min(chunk[asym], all - p0);
            const PairInfo *dp = (const PairInfo *)(base + pairs_at[asym]) + p0;
            hipLaunchKernelGGL(pair_u_kernel, dim3((unsigned)ceil_div(nlam_max, 64), nitems, np), dim3(64), 0, s, d.lm, np,
                               dp, asym, nitems, nlam_max, d.nlam, d.lam, d.eta, d.ex, d.p1, d.q1, d.ps, d.qs, U);
            XTR_LAUNCH_CHECK("pair_u_kernel");
            // I3 with J0; I1, I2, I5 with J1, I1 negated (HankelCoefficients.cs:103-118, ScalarMathUtils.cs:189-241)
            launch_hankel(HankelArgs{np, nitems, ncomp, nlam_max, ph.nrho_max, U, d.nlam, d.mpos, d.radii, d.h0, d.h1,
                                     asym, {asym ? 1.0 : -1.0, 1, 1, 1, 1}, 2 * kPi, I}, s);
            launch_segments(ncomp, np, nmerged, d.radii, I, segA, segB, s);
            LatArgs la{};
            la.nx = g.nx;
            la.ny = g.ny;
            la.nz = nz;
            la.npairs = np;
            la.p0 = p0;
            la.folded = folded ? 1 : 0;
            la.dx = in.dx;
            la.dy = in.dy;
            la.segA = segA;
            la.segB = segB;
            la.radii = d.radii;
            la.knots = knots;
            la.G = G;
            la.gblk = g.gblk();
            const int64_t S = g.S(), A = (int64_t)nz * nz;
            if (asym) {   // q-order {xz, yz}; device block [xx|xy|yy|zz|xz|yz]; parities XZ (-,+), YZ (+,-)
                la.off[0] = 4 * S; la.off[1] = 4 * S + A;
                la.xs[0] = -1; la.ys[0] = 1;
                la.xs[1] = 1; la.ys[1] = -1;
            } else {      // q-order {xx, yy, zz, xy}; parities (+,+) x3, XY (-,-)
                la.off[0] = 0; la.off[1] = 2 * S; la.off[2] = 3 * S; la.off[3] = S;
                for (int t = 0; t < 3; ++t) { la.xs[t] = 1; la.ys[t] = 1; }
                la.xs[3] = -1; la.ys[3] = -1;
            }
            int wgs = (int)ceil_div(np, 256);                        // of a cell, with equal shares of the pairs
            la.width = (int)(ceil_div(ceil_div(np, wgs), 64) * 64);
            int threads = la.width;
            // Few pairs, or too few cells for 4 workgroups a CU: 256 threads in groups of as many as the pairs take,
            // and fewer until the cells fill the chip.
            if (la.width <= 128 || cells * wgs < 4 * device_cus()) {
                threads = la.width = 256;
                while (la.width > 16 && (la.width / 2 >= np || cells * ceil_div(np, la.width) < 4 * device_cus())) la.width /= 2;
                wgs = (int)ceil_div(np, la.width);
            }
            auto run = [&](int64_t n, int y, int nt) {
                const dim3 grid((unsigned)n, (unsigned)y), block((unsigned)nt);
                auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, s, la); };
                if (nt > la.width) asym ? go(lateral_kernel<1, true>) : go(lateral_kernel<0, true>);
                else asym ? go(lateral_kernel<1, false>) : go(lateral_kernel<0, false>);
            };
            la.cols = g.ny;
            la.skip = 0;
            // The cells next to the source, with up to 200 segments, by groups in a launch of their own, unless the
            // others take longer than their chain (140 us) anyway (16384 workgroups, about 0.1 ms) or all go by
            // groups. 48 x 48 x 32: 39 + 58 and 58 + 73 us a set where one launch took 165 and 190 (all with their
            // searches), the whole call 1157 -> 1117 us; 96 x 48 x 17 605 -> 577 us.
            if (threads == la.width && cells * wgs < 64 * device_cus()) {
                const int wide = la.width;
                la.width = 64;
                la.cols = std::min(kNearCells, g.ny);
                run((int64_t)std::min(kNearCells, g.nx) * la.cols, (int)ceil_div(np, 64), 256);
                la.width = wide;
                la.cols = g.ny;
                la.skip = kNearCells;
            }
            run(cells, wgs, threads);
            XTR_LAUNCH_CHECK("lateral_kernel");
        }
    }
    if (folded) launch_fft2_mirror(G, g, tw_x, tw_y, s);
    else launch_fft2_plain(G, 2 * g.nx, 2 * g.ny, g.gblk(), tw_x, tw_y, s);
    XTR_CHECK(hipStreamSynchronize(s));   // the host pack is freed on return
}


// =============================================================================================
// AtoO: anomaly layers (volume transmitters) to one observation level (point receivers)
// =============================================================================================
namespace {

// slots of the AtoO components (AtoOLevelGreenTensorCalculator.cs:21-75)
enum { AO_XX, AO_YY, AO_ZZ, AO_XY, AO_YX, AO_XZ, AO_YZ, AO_ZX, AO_ZY, AO_N };

struct PointInfo {            // one transmitter layer seen from the level
    int r, s, t, b, kase;     // background layers of receiver / transmitter, min / max; 0 match 1 below 2 above
    double zw, z1, z2, dt, db1;
};

// CalculateCTop/CBot/DTop/DBot (VolumeToPointCalculatorU.cs:166-208) for layers (r, s)
__device__ inline double2 ctop_(const double2 *E, int r, int s, double zw, double z1, double z2)
{
    return cexp_d(-z1 * E[s] + zw * E[r]) - cexp_d(-z2 * E[s] + zw * E[r]);
}
__device__ inline double2 cbot_(const double2 *E, int r, int s, double zw, double z1, double z2)
{
    return cexp_d(-zw * E[r] + z2 * E[s]) - cexp_d(-zw * E[r] + z1 * E[s]);
}
__device__ inline double2 dtop_(const LayerModel &lm, const double2 *E, int r, int s, double zw, double z1, double z2)
{
    const int t = r < s ? r : s, b = r > s ? r : s;
    const double2 base = -2.0 * (lm.depth[b + 1] * E[b] - lm.depth[t] * E[t]);
    return cexp_d(base + z2 * E[s] - zw * E[r]) - cexp_d(base + z1 * E[s] - zw * E[r]);
}
__device__ inline double2 dbot_(const LayerModel &lm, const double2 *E, int r, int s, double zw, double z1, double z2)
{
    const int t = r < s ? r : s, b = r > s ? r : s;
    const double2 base = -2.0 * (lm.depth[b + 1] * E[b] - lm.depth[t] * E[t]);
    return cexp_d(base - z1 * E[s] + zw * E[r]) - cexp_d(base - z2 * E[s] + zw * E[r]);
}

// U[tr][item][comp][lambda], normalised before the Hankel filter (PlanCalculator.CalculateForE/H
// :58-108, VolumeToPointCalculatorU.cs:34-337, ScalarMathUtils.NormalizeBeforeHankelForE/H).
// electric: comps I1..I5 <- U1 (A1 set) * i w mu0 / 2, U2 / 2z, U3 l / 2z, U4 (-l) / 2z, U5 l^2 / 2z
// magnetic: comps I1..I4 <- U31, U4Sigma, U1Sigma * l, U11 * l
__global__ __launch_bounds__(64) void point_u_kernel(const LayerModel *lmp, int nz, const PointInfo *pts, int electric, int nitems, int nlam_max,
                               const int *nlam, const double *lam, const double2 *eta, const double2 *ex,
                               const double2 *p1, const double2 *q1, const double2 *ps, const double2 *qs,
                               double2 *U)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    const int it = blockIdx.y;
    const int tr = blockIdx.z;
    if (it >= nitems || m >= nlam[it] || tr >= nz) return;
    const PointInfo pi = pts[tr];
    const LayerModel &lm = *lmp;
    const int nl = lm.nl;
    const int64_t base = ((int64_t)it * nlam_max + m) * nl;
    const double2 *E = eta + base, *X = ex + base;
    const double l = lam[(int64_t)it * nlam_max + m];
    const int r = pi.r, s = pi.s, t = pi.t, b = pi.b;
    const double zw = pi.zw, z1 = pi.z1, z2 = pi.z2;
    const double2 er = E[r], es = E[s], et = E[t], eb = E[b];
    // CalculateT / CalculateR (:150-165)
    const double2 T = cexp_d(-zw * er - z1 * es + 2 * pi.dt * et) - cexp_d(-zw * er - z2 * es + 2 * pi.dt * et);
    const double2 R = cexp_d(-2 * pi.db1 * eb + z2 * es + zw * er) - cexp_d(-2 * pi.db1 * eb + z1 * es + zw * er);
    const double2 zrc2 = 2.0 * lm.zeta[r];
    const int ncomp = electric ? 5 : 4;
    double2 *out = U + (((int64_t)tr * nitems + it) * ncomp) * nlam_max + m;
    for (int set = 0; set < 2; ++set) {
        const double2 *P = (set ? ps : p1) + base;
        const double2 *Q = (set ? qs : q1) + base;
        const double2 pt = P[t], qb = Q[b];
        const double2 ann = ann_at(lm, E, X, P, Q, r, s, set);
        double2 psi1, psi3;
        if (pi.kase == 0) {          // receiver inside the transmitter layer (:210-240)
            const int n = r;
            const double2 pq = P[n] * Q[n];
            psi1 = ctop_(E, n, n, zw, zw, z2) + cbot_(E, n, n, zw, z1, zw) +
                   pq * (dtop_(lm, E, n, n, zw, zw, z2) + dbot_(lm, E, n, n, zw, z1, zw));
            psi3 = ctop_(E, n, n, zw, zw, z2) - cbot_(E, n, n, zw, z1, zw) +
                   pq * (dtop_(lm, E, n, n, zw, z1, zw) - dtop_(lm, E, n, n, zw, zw, z2));
        } else if (pi.kase == 1) {   // receiver below (:227-233, 249-256)
            psi1 = cbot_(E, r, s, zw, z1, z2) + pt * qb * dbot_(lm, E, r, s, zw, z1, z2);
            psi3 = -1.0 * cbot_(E, r, s, zw, z1, z2) + pt * qb * dbot_(lm, E, r, s, zw, z1, z2);
        } else {                     // receiver above (:219-226, 241-248)
            psi1 = ctop_(E, r, s, zw, z1, z2) + pt * qb * dtop_(lm, E, r, s, zw, z1, z2);
            psi3 = ctop_(E, r, s, zw, z1, z2) - pt * qb * dtop_(lm, E, r, s, zw, z1, z2);
        }
        const double2 u1 = (ann / es) * (pt * T + qb * R + psi1);
        const double2 u3 = (ann * (er / es)) * (-1.0 * (pt * T) + qb * R + psi3);
        const double2 u4 = ann * (-1.0 * (pt * T) + qb * R - psi3);
        if (electric) {
            if (set == 0) {
                out[0] = u1 * (c_(0, lm.omega * kMu0) * c_(0.5));
                continue;
            }
            const double2 u2 = (ann * er) * (pt * T + qb * R - psi1);
            double2 u5;
            if (pi.kase == 0) {      // CalcPsi5RcAndTrMatch (:258-272)
                const int n = r;
                const double ln = lm.thick[n];
                const double2 kk = (c_(0, lm.omega) * lm.zeta[n]) * c_(kMu0);
                const double2 en = E[n], pq = P[n] * Q[n];
                const double2 psi5 = pq * (cexp_d(-(2 * ln - (z2 - zw)) * en) + cexp_d(-(2 * ln - (zw - z1)) * en)) -
                                     (cexp_d(-(z2 - zw) * en) + cexp_d(-(zw - z1) * en)) +
                                     2.0 * (kk * ((c_(1) - pq * cexp_d(-2 * ln * en)) / c_(l * l)));
                u5 = (ann / es) * (pt * T + qb * R + psi5);
            } else {
                u5 = u1;
            }
            out[(int64_t)1 * nlam_max] = u2 / zrc2;
            out[(int64_t)2 * nlam_max] = u3 * (c_(l) / zrc2);
            out[(int64_t)3 * nlam_max] = u4 * (c_(-l) / zrc2);
            out[(int64_t)4 * nlam_max] = u5 * (c_(l * l) / zrc2);
        } else {
            if (set == 0) {
                out[0] = u3;                                 // I1 <- U31
                out[(int64_t)3 * nlam_max] = u1 * c_(l);     // I4 <- U11 * lambda
            } else {
                out[(int64_t)1 * nlam_max] = u4;             // I2 <- U4Sigma
                out[(int64_t)2 * nlam_max] = u1 * c_(l);     // I3 <- U1Sigma * lambda
            }
        }
    }
}

// The zero-rho point (CalculateZeroRhoForE/H, ScalarMathUtils.cs:33-81), radius 0 of the merged ones: I1, I2
// (and I5) are 0 there, I3 and I4 are (f[1] a^2 - f[2]) / (a^2 - 1) from the first item's 2nd and 3rd radii (at
// k1, k2), a the rho step.
__global__ void zero_rho_kernel(int nz, int ncomp, int k1, int k2, double alpha2, double2 *I)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ncomp * nz) return;
    const int c = e / nz;
    double2 v = make_double2(0, 0);
    if (c == 2 || c == 3) {
        const double2 f1 = I[(int64_t)k1 * ncomp * nz + e], f2 = I[(int64_t)k2 * ncomp * nz + e];
        v = make_double2((f1.x * alpha2 - f2.x) / (alpha2 - 1), (f1.y * alpha2 - f2.y) / (alpha2 - 1));
    }
    I[e] = v;
}

struct AoArgs {
    int nx, ny, nz;
    double dx, dy;
    double xs, ys;                // minus the level's shift (AtoOLevelGreenTensorCalculator.cs:119-125)
    const double2 *segA, *segB;   // [seg][comp][tr]
    const double *radii;
    const Knot *knots;            // of the offsets in order
    double2 *G;                   // [2Nx][2Ny][components][nz], components as in atoo_components
    int folded;                   // [Nx+1][Ny+1][components][nz], offsets i, j >= 0 only
    int width;                    // lanes of a group: a power of 2, the layers or 64
    int i0, i1, j0, j1;           // the offsets near the receiver, [i0, i1) x [j0, j1)
};

// The four edge integrals of RunAlongX / RunAlongY (GreenTensorCalculator.cs:192-281) for each lateral offset (i, j)
// in (-Nx, Nx) x (-Ny, Ny), or its non-negative quadrant where the tensor is folded (a level that is not shifted),
// written at TransformI/J (AtoOLevelGreenTensorCalculator.cs:106-117). A team of waves owns an offset: it forms its
// weights (CellWeights), 8 segments a wave at a time, a thread for each (segment, stretch), and sums over the
// segments in groups of `width` lanes, lane = transmitter layer, each group its own segments.
// Bound by the chain over the segments of the offsets next to the receiver, up to 200 of some 1500 where one 8 cells
// away crosses 22: those within kAoNear cells are shared by the 4 waves of a workgroup, which come first; the others
// take a wave each. 128 x 128 x 32, folded: 44 (electric) and 36 us; 60 and 50 with the searches for the knots in it,
// 120 and 114 with a wave for every offset as well; over all offsets 0.26 and 0.22 ms then, and 0.64 ms each with
// every thread working out the geometry.
constexpr int kAoWaves = 4, kAoSegs = 8, kAoNear = 8;

// Sums of one offset for the layers tr0 .. tr0 + width - 1, complete in the first `width` lanes of the team's first wave
template <int ELECTRIC, int TEAM, typename Sync>
__device__ __forceinline__ void ao_sums(const AoArgs &a, CellWeights<kAoSegs * TEAM> &cw, int tid, int lo, int hi, int tr0,
                                        double2 *G, const Sync &sync)
{
    constexpr int nc = ELECTRIC ? 5 : 4, no = ELECTRIC ? 8 : 7, SEGS = kAoSegs * TEAM;
    const int lane = tid & 63, tr = tr0 + (lane & (a.width - 1)), grp = tid / a.width, groups = 64 * TEAM / a.width;
#pragma unroll
    for (int t = 0; t < no; ++t) G[t] = c_(0);
    for (int seg0 = lo; seg0 <= hi; seg0 += SEGS) {
        const int n = min(SEGS, hi - seg0 + 1);
        cw.factors_of(tid, 64 * TEAM, a.radii, seg0, n);
        sync();
        cw.sum(tid, 64 * TEAM, n);
        sync();
        if (tr < a.nz)
            for (int k = grp; k < n; k += groups) {
                const double (&wx)[WN] = cw.w[k][0], (&wy)[WN] = cw.w[k][1];
                const double2 *A = a.segA + (int64_t)(seg0 + k) * nc * a.nz + tr;
                const double2 *B = a.segB + (int64_t)(seg0 + k) * nc * a.nz + tr;
                double2 sa[nc], sb[nc];                         // I1 .. I5 (I4)
#pragma unroll
                for (int c = 0; c < nc; ++c) {
                    sa[c] = A[(int64_t)c * a.nz];
                    sb[c] = B[(int64_t)c * a.nz];
                }
                // AddToQBuffAlong{X,Y}{Electric,Magnetic} (GreenTensorCalculator.cs:505-560) with the signs of the
                // QSigns tables (QSign.cs:31-38)
                const double nxw[WN] = {0, 0, -wx[W2A], -wx[W2B], 0, 0}, nyw[WN] = {0, 0, -wy[W2A], -wy[W2B], 0, 0};
                if constexpr (ELECTRIC) {                       // xx yy zz xy xz yz zx zy
                    G[0] = wab(nyw, W2A, wab(wx, W2A, G[0], sa[0], sb[0]), sa[1], sb[1]);
                    G[1] = wab(nxw, W2A, wab(wy, W2A, G[1], sa[0], sb[0]), sa[1], sb[1]);
                    G[2] = wab(nyw, W2A, wab(nxw, W2A, G[2], sa[4], sb[4]), sa[4], sb[4]);
                    G[3] = wab(wy, W3A, wab(wx, W3A, G[3], sa[1], sb[1]), sa[0], sb[0]);
                    G[4] = wab(wy, W1A, G[4], sa[2], sb[2]);
                    G[5] = wab(wx, W1A, G[5], sa[2], sb[2]);
                    G[6] = wab(wy, W1A, G[6], sa[3], sb[3]);
                    G[7] = wab(wx, W1A, G[7], sa[3], sb[3]);
                } else {                                        // xx xy yx xz yz zx zy
                    G[0] = wab(wy, W3A, wab(wx, W3A, G[0], sa[1], sb[1]), sa[0], sb[0]);
                    G[1] = wab(wy, W2A, wab(nxw, W2A, G[1], sa[1], sb[1]), sa[0], sb[0]);
                    G[2] = wab(nyw, W2A, wab(wx, W2A, G[2], sa[0], sb[0]), sa[1], sb[1]);
                    G[3] = wab(wx, W1A, G[3], sa[2], sb[2]);
                    G[4] = wab(wy, W1A, G[4], sa[2], sb[2]);
                    G[5] = wab(wx, W1A, G[5], sa[3], sb[3]);
                    G[6] = wab(wy, W1A, G[6], sa[3], sb[3]);
                }
            }
        sync();                                                 // the weights are read
    }
#pragma unroll
    for (int t = 0; t < no; ++t)
        for (int off = a.width; off < 64; off <<= 1) {
            G[t].x += __shfl_xor(G[t].x, off, 64);
            G[t].y += __shfl_xor(G[t].y, off, 64);
        }
    if constexpr (TEAM > 1) {
        static_assert(sizeof(cw.f) >= (TEAM - 1) * 4 * 64 * sizeof(double2), "four components of the other waves");
        double2 *red = reinterpret_cast<double2 *>(cw.f);
#pragma unroll
        for (int t0 = 0; t0 < no; t0 += 4) {
            const int wave = tid >> 6;
            if (wave > 0)
#pragma unroll
                for (int t = t0; t < t0 + 4 && t < no; ++t) red[((wave - 1) * 4 + t - t0) * 64 + lane] = G[t];
            sync();
            if (wave == 0)
#pragma unroll
                for (int t = t0; t < t0 + 4 && t < no; ++t)
#pragma unroll
                    for (int w = 0; w < TEAM - 1; ++w) G[t] = cadd<double>(G[t], red[(w * 4 + t - t0) * 64 + lane]);
            sync();
        }
    }
}

template <int ELECTRIC, int TEAM, typename Sync>
__device__ __forceinline__ void ao_offset(const AoArgs &a, CellWeights<kAoSegs * TEAM> &cw, int tid, int i, int j,
                                          const Sync &sync)
{
    constexpr int no = ELECTRIC ? 8 : 7;
    const int first_i = a.folded ? 0 : 1 - a.nx, first_j = a.folded ? 0 : 1 - a.ny, ncy = a.folded ? a.ny : 2 * a.ny - 1;
    cw.ends(tid, a.knots + ((i - first_i) * ncy + j - first_j) * 16, a.dx * (i - 0.5) - a.xs, a.dx * (i + 0.5) - a.xs,
            a.dy * (j - 0.5) - a.ys, a.dy * (j + 0.5) - a.ys);
    sync();
    int lo, hi;
    cw.range(lo, hi);
    const int64_t ti = i < 0 ? 2 * a.nx + i : i, tj = j < 0 ? 2 * a.ny + j : j;
    for (int tr0 = 0; tr0 < a.nz; tr0 += a.width) {
        double2 G[no];
        ao_sums<ELECTRIC, TEAM>(a, cw, tid, lo, hi, tr0, G, sync);
        if (tid < a.width && tr0 + tid < a.nz) {
            double2 *dst = a.G + (ti * (a.folded ? a.ny + 1 : 2 * a.ny) + tj) * (int64_t)(no * a.nz) + tr0 + tid;
#pragma unroll
            for (int t = 0; t < no; ++t) dst[(int64_t)t * a.nz] = G[t];
        }
    }
}

template <int ELECTRIC>
__global__ __launch_bounds__(64 * kAoWaves) void atoo_lateral_kernel(AoArgs a)
{
    __shared__ union Weights {
        CellWeights<kAoSegs> one[kAoWaves];
        CellWeights<kAoSegs * kAoWaves> team;
    } cw;
    const int nny = a.j1 - a.j0, near = (a.i1 - a.i0) * nny;     // offsets [i0, i1) x [j0, j1)
    if ((int)blockIdx.x < near) {
        ao_offset<ELECTRIC, kAoWaves>(a, cw.team, threadIdx.x, a.i0 + blockIdx.x / nny, a.j0 + blockIdx.x % nny,
                                      [] { __syncthreads(); });
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int ncy = a.folded ? a.ny : 2 * a.ny - 1, cells = (a.folded ? a.nx : 2 * a.nx - 1) * ncy;
    const int cell = ((int)blockIdx.x - near) * kAoWaves + wave;
    if (cell >= cells) return;                                  // waves do not meet at a barrier
    const int i = cell / ncy - (a.folded ? 0 : a.nx - 1), j = cell % ncy - (a.folded ? 0 : a.ny - 1);
    if (i >= a.i0 && i < a.i1 && j >= a.j0 && j < a.j1) return;
    // LDS writes of this wave become visible to it in order; the fence only keeps the compiler from moving them
    ao_offset<ELECTRIC, 1>(a, cw.one[wave], lane, i, j, [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    });
}

}  // namespace

int atoo_components(int electric, int *slot)
{
    // compact order: electric xx yy zz xy xz yz zx zy; magnetic xx xy yx xz yz zx zy
    static const int e[AO_N] = {0, 1, 2, 3, -1, 4, 5, 6, 7};
    static const int h[AO_N] = {0, -1, -1, 1, 2, 3, 4, 5, 6};
    for (int t = 0; t < AO_N; ++t) slot[t] = electric ? e[t] : h[t];
    return electric ? 8 : 7;
}

void build_green_atoo_level(const GreenInput &in, GreenScratch &work, double level_z, double shift_x, double shift_y,
                            int electric, bool folded, double2 *G, const double2 *tw_x, const double2 *tw_y, hipStream_t s)
{
    const Geom &g = in.g;
    const int nz = g.nz;
    const LayerModel lm = layer_model(in);
    // the level's own scalar plan (AtoOCalculator.cs:129, 151)
    const HostPlan hp = make_level_plan(in, shift_x, shift_y);
    if (hp.zero_rho && hp.rho[0].size() < 3) throw hip_error("zero-rho plan needs three radii in its first item");
    PlanHost ph(hp, in, lm);
    const int nitems = ph.nitems, nlam_max = ph.nlam_max, nmerged = ph.nmerged;
    // transmitters: the anomaly layers; receiver: the level point (AuxContainer.CreateContainer)
    const int r = layer_at_depth(in.section, level_z);
    std::vector<PointInfo> pts(nz);
    for (int tr = 0; tr < nz; ++tr) {
        PointInfo pi{};
        pi.zw = level_z;
        pi.z1 = in.depth[tr];
        pi.z2 = in.depth[tr] + in.thick[tr];
        pi.r = r;
        pi.s = layer_at_depth(in.section, pi.z1 + (pi.z2 - pi.z1) / 2);
        pi.t = std::min(pi.r, pi.s);
        pi.b = std::max(pi.r, pi.s);
        pi.dt = lm.depth[pi.t];
        pi.db1 = lm.depth[pi.b + 1];
        pi.kase = (pi.zw > pi.z1 && pi.zw < pi.z2) ? 0 : (pi.zw >= pi.z2 ? 1 : 2);   // CalcUGeneral (:54-62)
        pts[tr] = pi;
    }
    const int ncomp = electric ? 5 : 4;
    const int nseg = nmerged - 1;
    const size_t pts_at = ph.pack.add(pts);
    const size_t need[4] = {(size_t)nz * nitems * ncomp * nlam_max, (size_t)ncomp * nz * nmerged,
                            (size_t)nseg * ncomp * nz, (size_t)nseg * ncomp * nz};
    const int ncx = folded ? g.nx : 2 * g.nx - 1, ncy = folded ? g.ny : 2 * g.ny - 1, cells = ncx * ncy;
    size_t bytes = ph.device_bytes() + GreenScratch::padded(16 * cells * sizeof(Knot));
    for (size_t n : need) bytes += GreenScratch::padded(n * sizeof(double2));
    work.reserve(bytes);
    unsigned char *base;
    const PlanDev d = ph.upload(work, base, s);
    double2 *U = work.take<double2>(need[0]), *I = work.take<double2>(need[1]), *segA = work.take<double2>(need[2]),
            *segB = work.take<double2>(need[3]);
    Knot *knots = work.take<Knot>((size_t)16 * cells);
    launch_knots(d.radii, nmerged, in.dx, in.dy, -shift_x, -shift_y, folded ? 0 : 1 - g.nx, folded ? 0 : 1 - g.ny, ncy, cells,
                 knots, s);
    hipLaunchKernelGGL(point_u_kernel, dim3((unsigned)ceil_div(nlam_max, 64), nitems, nz), dim3(64), 0, s, d.lm, nz,
                       (const PointInfo *)(base + pts_at), electric, nitems, nlam_max, d.nlam, d.lam, d.eta, d.ex, d.p1,
                       d.q1, d.ps, d.qs, U);
    XTR_LAUNCH_CHECK("point_u_kernel");
    // HankelCoefficients.ConvoluteWith (:86-99), NormalizeAfterHankelForE/H (ScalarMathUtils.cs:131-155): electric
    // J1 -, J1 +, J0 +, J0 +, J1 + over 2 pi rho; magnetic J1 -, J1 -, J0 -, J0 + over 4 pi rho
    HankelArgs ha{nz, nitems, ncomp, nlam_max, ph.nrho_max, U, d.nlam, d.mpos, d.radii, d.h0, d.h1, 0xc,
                  {-1, 1, 1, 1, 1}, 2 * kPi, I};
    if (!electric) {
        ha.sgn[1] = ha.sgn[2] = -1;
        ha.den = 4 * kPi;
    }
    launch_hankel(ha, s);
    if (hp.zero_rho) {
        const auto place = [&](int ix) {
            for (int k = 0; k < nmerged; ++k)
                if (hp.m_item[k] == 0 && hp.m_idx[k] == ix) return k;
            throw hip_error("zero-rho plan: radius not found");
        };
        hipLaunchKernelGGL(zero_rho_kernel, dim3((unsigned)ceil_div(ncomp * nz, 256)), dim3(256), 0, s, nz, ncomp, place(1),
                           place(2), log10_rho_step() * log10_rho_step(), I);
        XTR_LAUNCH_CHECK("zero_rho_kernel");
    }
    launch_segments(ncomp, nz, nmerged, d.radii, I, segA, segB, s);
    int slot[9];
    const int ntc = atoo_components(electric, slot);
    AoArgs a{};
    a.nx = g.nx;
    a.ny = g.ny;
    a.nz = nz;
    a.dx = in.dx;
    a.dy = in.dy;
    a.xs = -shift_x;
    a.ys = -shift_y;
    a.segA = segA;
    a.segB = segB;
    a.radii = d.radii;
    a.knots = knots;
    a.G = G;
    a.folded = folded ? 1 : 0;
    if (!folded) XTR_CHECK(hipMemsetAsync(G, 0, (size_t)g.L() * ntc * nz * sizeof(double2), s));
    for (a.width = 8; a.width < nz && a.width < 64;) a.width *= 2;
    // within kAoNear cells of the receiver, as far as the offsets go (i1 = i0 where none is)
    auto window = [&](double shift, double d, int n, int &from, int &to) {
        const double c = std::fmin(std::fmax(std::nearbyint(shift / d), -2.0 * n), 2.0 * n);
        const int first = folded ? 0 : 1 - n;
        from = std::min(std::max((int)c - kAoNear + 1, first), n);
        to = std::max(std::min((int)c + kAoNear, n), from);
    };
    window(a.xs, a.dx, g.nx, a.i0, a.i1);
    window(a.ys, a.dy, g.ny, a.j0, a.j1);
    const dim3 grid((unsigned)((a.i1 - a.i0) * (a.j1 - a.j0) + ceil_div(cells, kAoWaves))), nt(64 * kAoWaves);
    if (electric) hipLaunchKernelGGL(atoo_lateral_kernel<1>, grid, nt, 0, s, a);
    else hipLaunchKernelGGL(atoo_lateral_kernel<0>, grid, nt, 0, s, a);
    XTR_LAUNCH_CHECK("atoo_lateral_kernel");
    if (folded) {
        unsigned odd[2];
        level_parity(electric, odd);
        launch_fft2_mirror_level(G, g, ntc, odd, tw_x, tw_y, s);
    } else {
        launch_fft2_plain(G, 2 * g.nx, 2 * g.ny, (int64_t)ntc * nz, tw_x, tw_y, s);
    }
    XTR_CHECK(hipStreamSynchronize(s));   // the host pack is freed on return
}

}  // namespace xtr
