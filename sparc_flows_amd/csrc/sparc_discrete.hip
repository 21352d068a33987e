// sparc_discrete.hip -- exact discrete adjoint of the 2D option-17 step.
//
// The reference's adjoint (driver.f90:144-147, kernels.f90:286-355) is the
// continuous recipe: a time-reversed forward run with -v0 whose snapshots are
// correlated with the forward ones.  This file is its exact counterpart for
// gradients: the transpose of the discrete step of step.f90:43-119 (five
// low-storage RK stages of MP_QUIET_PML_2D_DISPL, physics2d.f90:943-1094, the
// z filter FILTER_VARS_2D, physics2d.f90:509-556, and the PML auxiliaries),
// run backwards over a recomputed forward trajectory, with the gradient of a
// functional of the vz traces with respect to c^2 rho0, v0x and v0z
// accumulated stage by stage, then mapped to the stream function and the
// sound speed.
//
// Building blocks (all batched over the S sources, fields [S][nz][nx]):
//   * x-derivatives: the library's FFT row kernel; its transpose is -Dx (the
//     multiplier i k is odd and the Nyquist bin is dropped);
//   * z-derivatives and their transposes: the segmented compact-FD solve
//     (sparc_zseg.hip); for an nz that it does not take, the dbyd2 map of each
//     ibc as a dense nz x nz matrix (built by the library's own compact-FD
//     solve of an identity block), applied by an LDS-tiled kernel (k_dz_dense);
//   * pointwise kernels for the PML, pressure, density and flow terms of the
//     forward stage (k_fwd_b, k_fwd_c) and of its transpose (k_adj_a,
//     k_adj_b, k_adj_c), the z filter and its transpose.
// The forward stages here are unfused and recomputed from the trajectory; they
// agree with the fused solver to rounding.  Bound: HBM and the launches (6 to 29 us
// each).  A forward stage is six launches and a transposed one seven: the pointwise
// kernels write the next stage's input or the accumulated adjoint themselves, and
// derivatives of different fields share a launch.  With a pass of its own for every
// update and accumulation a step of 8 sources at 256 x 300 took 415 us forward and
// 620 transposed; here 317 and 455.
#include <algorithm>
#include <utility>

#include "sparc_device.h"
#include "sparc_launch.h"

namespace sparc {

namespace {

constexpr int kTX = 64, kTJ = 32, kTI = 64;

// out[b][j][x] = sum_i M[j][i] in[b][i][x] + vN[j] * preScale * pre[b * preStride + x]
// (the last term only when vN is not null).  Block: 64 columns x 32 output
// rows, the input tile and the matrix tile staged in LDS.
__global__ __launch_bounds__(256) void k_dz_dense(const double *__restrict__ in, double *__restrict__ out, int nz,
                                                  int nx, const double *__restrict__ M,
                                                  const double *__restrict__ vN, const double *__restrict__ pre,
                                                  size_t preStride, double preScale)
{
    __shared__ double Ms[kTJ][kTI + 1];
    __shared__ double Is[kTI][kTX];
    const int tx = threadIdx.x & (kTX - 1), rg = threadIdx.x >> 6;
    const int x = blockIdx.x * kTX + tx, j0 = blockIdx.y * kTJ, b = blockIdx.z;
    const double *inb = in + (size_t)b * nz * nx;
    double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int i0 = 0; i0 < nz; i0 += kTI) {
        for (int r = rg; r < kTI; r += 4) {
            const int i = i0 + r;
            Is[r][tx] = (i < nz && x < nx) ? inb[(size_t)i * nx + x] : 0.0;
        }
        for (int u = 0; u < kTJ * kTI / 256; u++) {
            const int e = threadIdx.x + 256 * u, jj = e / kTI, ii = e % kTI;
            const int j = j0 + jj, i = i0 + ii;
            Ms[jj][ii] = (j < nz && i < nz) ? M[(size_t)j * nz + i] : 0.0;
        }
        __syncthreads();
#pragma unroll 4
        for (int ii = 0; ii < kTI; ii++) {
            const double v = Is[ii][tx];
#pragma unroll
            for (int r = 0; r < 8; r++) acc[r] += Ms[rg * 8 + r][ii] * v;
        }
        __syncthreads();
    }
    if (x >= nx) return;
    const double pv = vN ? preScale * pre[(size_t)b * preStride + x] : 0.0;
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const int j = j0 + rg * 8 + r;
        if (j < nz) out[((size_t)b * nz + j) * nx + x] = acc[r] + (vN ? vN[j] * pv : 0.0);
    }
}

// out[b][x] = sum_k w[k] in[b][k][x]
__global__ void k_colsum_w(const double *__restrict__ in, const double *__restrict__ w, double *__restrict__ out,
                           int nz, int nx, int nb)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nb * nx) return;
    const int b = q / nx, x = q - b * nx;
    double s = 0.0;
    for (int k = 0; k < nz; k++) s += w[k] * in[((size_t)b * nz + k) * nx + x];
    out[q] = s;
}

// Geometry of point r of one source's [nz][nx] field: row, column, its z-PML
// row (-1 outside the layers) and x-PML column (-1 outside).
struct Pt {
    int b, k, i, pj, ci;
};
__device__ __forceinline__ Pt point(int b, unsigned r, const Dims &d)
{
    Pt p;
    p.b = b;
    p.k = (int)(r / (unsigned)d.nx);
    p.i = (int)r - p.k * d.nx;
    p.pj = p.k < d.npmlbot ? p.k : (p.k >= d.nz - d.npmltop ? d.npmlbot + (p.k - (d.nz - d.npmltop)) : -1);
    p.ci = p.i < d.nh ? p.i : (p.i >= d.nx - d.nh ? d.nh + (p.i - (d.nx - d.nh)) : -1);
    return p;
}
// The pointwise kernels' grid: blocks of 256 points of a source in x, sources in y
// (each point costs one 32-bit division; with flat 64-bit indices over all sources the
// divisions bound the filters, 45 us a launch at 8 x 256 x 300).
inline dim3 grid2(const Dims &d)
{
    return dim3((unsigned)((d.nz * d.nx + 255) / 256), (unsigned)(d.S < 65535 ? d.S : 65535));
}
#define FOR_POINTS(d, r, b)                                                                        \
    const unsigned r = blockIdx.x * 256u + threadIdx.x, n2_ = (unsigned)d.nz * (unsigned)d.nx;     \
    if (r >= n2_) return;                                                                          \
    for (int b = blockIdx.y; b < d.S; b += gridDim.y)

// Full-state views: a [4][S][nz][nx], pz [2][S][nzpml][nx], px [2][S][nz][nph].
struct Views {
    size_t SN, PZ1, PX1;   // one field of a, pz, px
};
__device__ __forceinline__ size_t pzi(const Dims &d, const Pt &p) { return ((size_t)p.b * d.nzpml + p.pj) * d.nx + p.i; }
__device__ __forceinline__ size_t pxi(const Dims &d, const Pt &p) { return ((size_t)p.b * d.nz + p.k) * d.nph + p.ci; }

// Forward stage, first pointwise part (physics2d.f90:957-998, :1043): z-PML of
// dxi_z/dz, x-PML of dxi_x/dx, div, p, rho'.  dzxi includes the kept last
// row (:954).  Writes DIV, P, RHO and psivz, psivx of the next stage's
// input Yn = U + beta * RHS (step.f90:60-62), where every element is read only at
// its own point before: Yn may be Y.
__global__ __launch_bounds__(256) void k_fwd_b(Dims d, Bg bg, Views v, const double *Y,
                                               const double *__restrict__ dxxi, const double *__restrict__ dzxi,
                                               double *__restrict__ DIV, double *__restrict__ P,
                                               double *__restrict__ RHO, const double *U, double beta, double *Yn)
{
    FOR_POINTS(d, r2, b)
    {
        const Pt p = point(b, r2, d);
        const size_t q = (size_t)b * n2_ + r2, pz = 4 * v.SN, px = pz + 2 * v.PZ1;
        double dz = dzxi[q], dx = dxxi[q];
        if (p.pj >= 0) {
            const size_t e = pz + pzi(d, p), c = (size_t)p.pj * d.nx + p.i;
            const double psi = Y[e];
            Yn[e] = U[e] + beta * (bg.az[c] * dz + bg.bz[c] * psi);
            dz = dz + psi;
        }
        if (p.ci >= 0) {
            const size_t e = px + pxi(d, p), c = (size_t)p.k * d.nph + p.ci;
            const double psi = Y[e];
            dx = dx + psi;
            Yn[e] = U[e] + beta * (bg.ax[c] * dx + bg.bx[c] * psi);
        }
        const double div = dx + dz, xiz = Y[v.SN + q];
        DIV[q] = div;
        P[q] = -(bg.c2rho0[r2] * div) - bg.gp0[r2] * xiz;
        RHO[q] = -(bg.rho0[r2] * div) - bg.gr0[r2] * xiz;
    }
}

// Forward stage, second pointwise part (physics2d.f90:1003-1092): PMLs of the
// pressure gradient, RHS v_x, v_z, xi, the source of time t, the flow terms,
// the zeroed rows and columns, and the next stage's input Yn = U + beta * RHS.
// DV = [dvx/dx, dvz/dx, dvx/dz, dvz/dz].  Yn may be Y, as in k_fwd_b.
__global__ __launch_bounds__(256) void k_fwd_c(Dims d, Bg bg, Views v, Src src, int t, const double *Y,
                                               const double *__restrict__ gpx_in, const double *__restrict__ gpz_in,
                                               const double *__restrict__ RHO, const double *__restrict__ DV,
                                               const double *U, double beta, double *Yn)
{
    FOR_POINTS(d, r2, b)
    {
        const Pt p = point(b, r2, d);
        const size_t q = (size_t)b * n2_ + r2, pz = 4 * v.SN + v.PZ1, px = 4 * v.SN + 2 * v.PZ1 + v.PX1;
        double gpx = gpx_in[q], gpz = gpz_in[q];
        if (p.ci >= 0) {
            const size_t e = px + pxi(d, p), c = (size_t)p.k * d.nph + p.ci;
            const double psi = Y[e];
            gpx = gpx + psi;
            Yn[e] = U[e] + beta * (bg.ax[c] * gpx + bg.bx[c] * psi);
        }
        if (p.pj >= 0) {
            const size_t e = pz + pzi(d, p), c = (size_t)p.pj * d.nx + p.i;
            const double psi = Y[e];
            Yn[e] = U[e] + beta * (bg.az[c] * gpz + bg.bz[c] * psi);
            gpz = gpz + psi;
        }
        double rvx = -bg.rhoinv[r2] * gpx;
        double rvz = -bg.rhoinv[r2] * (gpz + RHO[q] * bg.g[p.k]);
        const double rxx = Y[2 * v.SN + q], rxz = Y[3 * v.SN + q];
        if (t <= src.limit) {                                   // :1051-1061
            const double fs = (t >= 0 && t < src.nfwd) ? src.fwd[t] : 0.0;
            if (src.mode == 1 && p.k == src.row)
                rvz += src.vr[(size_t)b * d.nx + p.i] * fs * src.delta_width / bg.rho0_src[p.i];
            else if (src.mode == 3)
                rvz += src.vr[(size_t)b * d.nx + p.i] * fs * src.zprof[p.k];
        }
        rvx = rvx - 2.0 * bg.v0x[r2] * DV[q];                   // :1065-1079
        rvx = rvx - 2.0 * bg.v0z[r2] * DV[2 * v.SN + q];
        rvz = rvz - 2.0 * bg.v0x[r2] * DV[v.SN + q];
        rvz = rvz - 2.0 * bg.v0z[r2] * DV[3 * v.SN + q];
        const bool zero = p.k == 0 || p.i == 0 || p.i == d.nx - 1;  // :1083-1092
        Yn[q] = U[q] + beta * (zero ? 0.0 : rxx);
        Yn[v.SN + q] = U[v.SN + q] + beta * (zero ? 0.0 : rxz);
        Yn[2 * v.SN + q] = U[2 * v.SN + q] + beta * (zero ? 0.0 : rvx);
        Yn[3 * v.SN + q] = U[3 * v.SN + q] + beta * (zero ? 0.0 : rvz);
    }
}

// FILTER_VARS_2D (physics2d.f90:509-556): rows 5..nz-6 (0-based) take the
// 11-point filter, rows nz-5..nz-2 the two-point mean, for columns nh-1 .. nx-nh.
// One lane filters kFR rows of a column of one field, from a window of kFR + 10 rows:
// 2.25 loads a row in place of 11.  us per launch at 8 x 256 x 300, one lane a
// point with 64-bit index arithmetic -> here: 45 -> 11, transposed 44 -> 15.
constexpr int kFR = 8;
__device__ __forceinline__ double kfc(int m)
{
    constexpr double c[6] = {0.75390625, 0.41015625, -0.234375, 0.087890625, -0.01953125, 0.001953125};
    return c[m];
}
inline dim3 grid_filter(const Dims &d)
{
    return dim3((unsigned)(((d.nz + kFR - 1) / kFR * d.nx + 255) / 256), (unsigned)std::min(4 * (long)d.S, 65535L));
}
// The window of the lane's rows in each of the 4 S columns of fields, and the PML
// variables behind them element by element: body(field base, first row, column,
// window), tail(element).
template <class Body, class Tail>
__device__ __forceinline__ void filter_walk(const Dims &d, const Views &v, const double *__restrict__ in, Body &&body,
                                            Tail &&tail)
{
    const size_t n4 = 4 * v.SN, nall = n4 + 2 * v.PZ1 + 2 * v.PX1, total = (size_t)gridDim.x * gridDim.y * 256;
    for (size_t q = n4 + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x; q < nall; q += total) tail(q);
    const unsigned id = blockIdx.x * 256u + threadIdx.x;
    const int g = (int)(id / (unsigned)d.nx), x = (int)id - g * d.nx, j0 = g * kFR;
    if (j0 >= d.nz) return;
    for (int fb = blockIdx.y; fb < 4 * d.S; fb += gridDim.y) {
        const size_t base = (size_t)fb * d.nz * d.nx + x;
        double w[kFR + 10];
#pragma unroll
        for (int u = 0; u < kFR + 10; u++) w[u] = in[base + (size_t)min(max(j0 - 5 + u, 0), d.nz - 1) * d.nx];
        body(base, j0, x, w);
    }
}

// A = filter(Y) on the 4 fields of the last stage's update (step.f90:107-112),
// the PML variables copied.
__global__ __launch_bounds__(256) void k_filter(Dims d, Views v, const double *__restrict__ Y, double *__restrict__ A)
{
    filter_walk(d, v, Y,
        [&](size_t base, int j0, int x, const double (&w)[kFR + 10]) {
            const bool xin = x >= d.nh - 1 && x <= d.nx - d.nh;
#pragma unroll
            for (int i = 0; i < kFR; i++) {
                const int k = j0 + i;
                if (k >= d.nz) break;
                double val = w[i + 5];
                if (xin && k >= 5 && k <= d.nz - 2) {
                    if (k <= d.nz - 6) {
                        val = kfc(0) * val;
#pragma unroll
                        for (int m = 1; m <= 5; m++) val += 0.5 * kfc(m) * (w[i + 5 - m] + w[i + 5 + m]);
                    } else {
                        val = 0.5 * (w[i + 6] + w[i + 4]);
                    }
                }
                A[base + (size_t)k * d.nx] = val;
            }
        },
        [&](size_t q) { A[q] = Y[q]; });
}

// Transpose of the filter on the 4 fields (pz, px copied): acc = F^T lam, and
// the last stage's RHS adjoint Rb = dt acc.
__global__ __launch_bounds__(256) void k_filter_T(Dims d, Views v, const double *__restrict__ lam, double dt,
                                                  double *__restrict__ acc, double *__restrict__ Rb)
{
    filter_walk(d, v, lam,
        [&](size_t base, int j0, int x, const double (&w)[kFR + 10]) {
            const int nz = d.nz;
            const bool xin = x >= d.nh - 1 && x <= d.nx - d.nh;
#pragma unroll
            for (int i = 0; i < kFR; i++) {
                const int j = j0 + i;
                if (j >= nz) break;
                double val = w[i + 5];
                if (xin) {
                    if (j >= 5 && j <= nz - 2) val = 0.0;          // rows the filter replaces
#pragma unroll
                    for (int m = -5; m <= 5; m++) {
                        const int k = j + m;
                        if (k >= 5 && k <= nz - 6) val += (m == 0 ? kfc(0) : 0.5 * kfc(m < 0 ? -m : m)) * w[i + 5 + m];
                    }
                    if (j - 1 >= nz - 5 && j - 1 <= nz - 2) val += 0.5 * w[i + 4];
                    if (j + 1 >= nz - 5 && j + 1 <= nz - 2) val += 0.5 * w[i + 6];
                }
                acc[base + (size_t)j * d.nx] = val;
                Rb[base + (size_t)j * d.nx] = dt * val;
            }
        },
        [&](size_t q) {
            const double val = lam[q];
            acc[q] = val;
            Rb[q] = dt * val;
        });
}

// The adjoint y of one element of a stage's input: into the adjoint of the step's
// start, and times beta the RHS adjoint of the stage before.
__device__ __forceinline__ void accumulate(double *acc, double *Rb, size_t e, double y, double beta)
{
    acc[e] += y;
    Rb[e] = beta * y;
}

// Transpose of k_fwd_c's RHS (and of the flow terms' inputs):
// FX = [-2 v0x Rvx, -2 v0x Rvz, adjoint of dp/dx], FZ = [-2 v0z Rvx,
// -2 v0z Rvz], GZ = adjoint of the raw dp/dz; accumulates the adjoints of
// psi_gradp_x and psip.  The three adjoint kernels read and then replace Rb at
// their own points only, each its own elements.
__global__ __launch_bounds__(256) void k_adj_a(Dims d, Bg bg, Views v, double *__restrict__ Rb,
                                               double *__restrict__ acc, double beta, double *__restrict__ FX,
                                               double *__restrict__ FZ, double *__restrict__ GZ)
{
    FOR_POINTS(d, r2, b)
    {
        const Pt p = point(b, r2, d);
        const size_t q = (size_t)b * n2_ + r2;
        const bool zero = p.k == 0 || p.i == 0 || p.i == d.nx - 1;
        const double rvx = zero ? 0.0 : Rb[2 * v.SN + q], rvz = zero ? 0.0 : Rb[3 * v.SN + q];
        FX[q] = -2.0 * bg.v0x[r2] * rvx;
        FX[v.SN + q] = -2.0 * bg.v0x[r2] * rvz;
        FZ[q] = -2.0 * bg.v0z[r2] * rvx;
        FZ[v.SN + q] = -2.0 * bg.v0z[r2] * rvz;
        double gpx = -bg.rhoinv[r2] * rvx;
        if (p.ci >= 0) {
            const size_t e = 4 * v.SN + 2 * v.PZ1 + v.PX1 + pxi(d, p), c = (size_t)p.k * d.nph + p.ci;
            const double r = Rb[e], tot = gpx + bg.ax[c] * r;
            accumulate(acc, Rb, e, tot + bg.bx[c] * r, beta);
            gpx = tot;
        }
        FX[2 * v.SN + q] = gpx;
        double gpz = -bg.rhoinv[r2] * rvz;
        if (p.pj >= 0) {
            const size_t e = 4 * v.SN + v.PZ1 + pzi(d, p), c = (size_t)p.pj * d.nx + p.i;
            const double r = Rb[e];
            accumulate(acc, Rb, e, gpz + bg.bz[c] * r, beta);
            gpz = gpz + bg.az[c] * r;
        }
        GZ[q] = gpz;
    }
}

// Second transposed part: v adjoints, p adjoint, div adjoint through both
// PMLs of the displacement derivatives, the gradient contributions of this
// stage: G = [d/d(c^2 rho0), d/dv0x, d/dv0z] += pairs with the stage's
// forward quantities D = [div, dvx/dx, dvz/dx, dvx/dz, dvz/dz].
__global__ __launch_bounds__(256) void k_adj_b(Dims d, Bg bg, Views v, double *__restrict__ Rb,
                                               double *__restrict__ acc, double beta, const double *__restrict__ DFX,
                                               const double *__restrict__ DFZ, const double *__restrict__ DGZ,
                                               const double *__restrict__ D, double *__restrict__ XZP,
                                               double *__restrict__ DXB, double *__restrict__ DZB,
                                               double *__restrict__ G)
{
    FOR_POINTS(d, r2, b)
    {
        const Pt p = point(b, r2, d);
        const size_t q = (size_t)b * n2_ + r2;
        const bool zero = p.k == 0 || p.i == 0 || p.i == d.nx - 1;
        const double rxx = zero ? 0.0 : Rb[q], rxz = zero ? 0.0 : Rb[v.SN + q];
        const double rvx = zero ? 0.0 : Rb[2 * v.SN + q], rvz = zero ? 0.0 : Rb[3 * v.SN + q];
        accumulate(acc, Rb, 2 * v.SN + q, -DFX[q] + DFZ[q] + rxx, beta);           // dx^T = -dx
        accumulate(acc, Rb, 3 * v.SN + q, -DFX[v.SN + q] + DFZ[v.SN + q] + rxz, beta);
        const double pb = -DFX[2 * v.SN + q] + DGZ[q];
        const double rb = -bg.rhoinv[r2] * bg.g[p.k] * rvz;                        // adjoint of rho'
        const double divb = -bg.rho0[r2] * rb - bg.c2rho0[r2] * pb;
        XZP[q] = -bg.gr0[r2] * rb - bg.gp0[r2] * pb;
        double dxb = divb, dzb = divb;
        if (p.ci >= 0) {
            const size_t e = 4 * v.SN + 2 * v.PZ1 + pxi(d, p), c = (size_t)p.k * d.nph + p.ci;
            const double r = Rb[e], tot = divb + bg.ax[c] * r;
            accumulate(acc, Rb, e, tot + bg.bx[c] * r, beta);
            dxb = tot;
        }
        if (p.pj >= 0) {
            const size_t e = 4 * v.SN + pzi(d, p), c = (size_t)p.pj * d.nx + p.i;
            const double r = Rb[e];
            accumulate(acc, Rb, e, divb + bg.bz[c] * r, beta);
            dzb = divb + bg.az[c] * r;
        }
        DXB[q] = dxb;
        DZB[q] = dzb;
        G[q] += -pb * D[q];
        G[v.SN + q] += -2.0 * (rvx * D[v.SN + q] + rvz * D[2 * v.SN + q]);
        G[2 * v.SN + q] += -2.0 * (rvx * D[3 * v.SN + q] + rvz * D[4 * v.SN + q]);
    }
}

// The kept last row of dxi_z/dz is -dxi_x/dx unstretch (:954): its adjoint
// goes back into the last row of the dxi_x/dx adjoint.
__global__ void k_adj_preset(const double *__restrict__ pb, double *__restrict__ DXB, int nz, int nx, int nb,
                             double unstretch_last)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nb * nx) return;
    const int b = q / nx, x = q - b * nx;
    DXB[((size_t)b * nz + nz - 1) * nx + x] += -unstretch_last * pb[q];
}

// The displacement's adjoints: xi_x = -dx(DXB), xi_z = XZP + Dz3^T DZB
__global__ __launch_bounds__(256) void k_adj_c(Views v, const double *__restrict__ DDXB,
                                               const double *__restrict__ XZP, const double *__restrict__ DZ3B,
                                               double *__restrict__ Rb, double *__restrict__ acc, double beta)
{
    const size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (q >= v.SN) return;
    accumulate(acc, Rb, q, -DDXB[q], beta);
    accumulate(acc, Rb, v.SN + q, XZP[q] + DZ3B[q], beta);
}

// lam[vz][b][o_rad][x] += gvz[b][k][x]
__global__ void k_inject(double *__restrict__ lam, const double *__restrict__ gvz, int k, int nt, int orow,
                         int nz, int nx, int nb, size_t SN)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nb * nx) return;
    const int b = q / nx, x = q - b * nx;
    lam[3 * SN + ((size_t)b * nz + orow) * nx + x] += gvz[((size_t)b * nt + k) * nx + x];
}

// gradient of the flow map (driver.f90:94-126): inputs Gx, Gz (d/dv0x,
// d/dv0z) -> WX = Gx / rho0, WZ = Gz / rho0 (for Dz1^T and dx^T)
__global__ void k_flow_in(Views v, int n2, const double *__restrict__ rho0, const double *__restrict__ G,
                          double *__restrict__ WX, double *__restrict__ WZ)
{
    const size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (q >= v.SN) return;
    const double r = rho0[q % n2];
    WX[q] = G[v.SN + q] / r;
    WZ[q] = G[2 * v.SN + q] / r;
}

// d pv = -Dz1^T WX - dx WZ; gpsi = d pv rho0 c / (Rsun/1e8); gc = 2 c rho0 G2
// / dimc + d pv rho0 psi / (Rsun/1e8) / dimc, with c = sqrt(c2) in code units
__global__ void k_flow_out(Views v, int n2, const double *__restrict__ rho0, const double *__restrict__ c2,
                           const double *__restrict__ psi, double scale, double dimc,
                           const double *__restrict__ G, const double *__restrict__ DZWX,
                           const double *__restrict__ DXWZ, double *__restrict__ gpsi, double *__restrict__ gc)
{
    const size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (q >= v.SN) return;
    const size_t r2 = q % n2;
    const double gpv = -DZWX[q] - DXWZ[q];
    const double c = sqrt(c2[r2]);
    if (gpsi) gpsi[q] = gpv * rho0[r2] * c / scale;
    if (gc) gc[q] = 2.0 * c * rho0[r2] * G[q] / dimc + (psi ? gpv * rho0[r2] * psi[r2] / scale / dimc : 0.0);
}

inline dim3 grid1(size_t n, int bs = 256) { return dim3((unsigned)((n + bs - 1) / bs)); }

}  // namespace

#define DCHK(expr)                                   \
    do {                                             \
        hipError_t e_ = (expr);                      \
        if (e_ != hipSuccess) return e_;             \
    } while (0)

static ZDer zder_args(const DiscreteCtx &c, const double *in, double *out, int nbatch, int ibc, bool transposed)
{
    ZDer a{};
    a.in = in;
    a.out = out;
    a.ncols = c.d.nx;
    a.nz = c.d.nz;
    a.nbatch = nbatch;
    a.ibc = ibc;
    a.stretch = c.bg.stretch;
    a.transposed = transposed;
    if (transposed) dbyd2_edge_rows(c.d.nz, ibc, a.eb);
    return a;
}

// A second group of fields in the launch of a.
static void zder_second(ZDer &a, const double *in, double *out, int nbatch, int ibc)
{
    a.in2 = in;
    a.out2 = out;
    a.nbatch2 = nbatch;
    a.ibc2 = ibc;
    if (a.transposed) dbyd2_edge_rows(a.nz, ibc, a.eb2);
}

bool discrete_segmented(const DiscreteCtx &c, int nbatch)
{
    return zder_fits(zder_args(c, nullptr, nullptr, nbatch, 1, true), c.zseg);
}

// One group of fields of a z-derivative: out = Dz_ibc in (or its transpose) of
// nbatch fields, ibc 1..3.
struct ZGroup {
    const double *in;
    double *out;
    int nbatch, ibc;
};

// out = Dz_ibc in, the kept last row of ibc 3 preScale * pre[b * preStride + x]
// (0 when pre is null; for the first group), kept first row of ibc 2 0; g2 (may
// be null) a second group in the same launch.
static hipError_t dz(const DiscreteCtx &c, const ZGroup &g, const ZGroup *g2, const double *pre, size_t preStride,
                     double preScale)
{
    ZDer a = zder_args(c, g.in, g.out, g.nbatch, g.ibc, false);
    if (discrete_segmented(c, g.nbatch + (g2 ? g2->nbatch : 0))) {
        a.pre = pre;
        a.pre_stride = preStride;
        a.pre_scale = preScale;
        a.zero_kept = 1;
        if (g2) zder_second(a, g2->in, g2->out, g2->nbatch, g2->ibc);
        return launch_zder(a, c.zseg, c.stream);
    }
    for (const ZGroup *k : {&g, g2}) {
        if (!k) continue;
        dim3 grid((c.d.nx + kTX - 1) / kTX, (c.d.nz + kTJ - 1) / kTJ, k->nbatch);
        const double *const kp = k == &g ? pre : nullptr;
        hipLaunchKernelGGL(k_dz_dense, grid, dim3(256), 0, c.stream, k->in, k->out, c.d.nz, c.d.nx, c.M[k->ibc - 1],
                           kp ? c.vN3 : nullptr, kp, preStride, preScale);
        DCHK(hipGetLastError());
    }
    return hipSuccess;
}

// out = Dz_ibc^T in (ibc 1..3, kept rows 0); prebar (may be null) gets the
// adjoint of ibc 3's kept last row [nbatch][nx]; g2 as in dz.
static hipError_t dz_T(const DiscreteCtx &c, const ZGroup &g, const ZGroup *g2, double *prebar)
{
    ZDer a = zder_args(c, g.in, g.out, g.nbatch, g.ibc, true);
    if (discrete_segmented(c, g.nbatch + (g2 ? g2->nbatch : 0))) {
        a.prebar = prebar;
        a.prebar_stride = (size_t)c.d.nx;
        if (g2) zder_second(a, g2->in, g2->out, g2->nbatch, g2->ibc);
        return launch_zder(a, c.zseg, c.stream);
    }
    if (prebar) {
        hipLaunchKernelGGL(k_colsum_w, grid1((size_t)g.nbatch * c.d.nx), dim3(256), 0, c.stream, g.in, c.vN3, prebar,
                           c.d.nz, c.d.nx, g.nbatch);
        DCHK(hipGetLastError());
    }
    for (const ZGroup *k : {&g, g2}) {
        if (!k) continue;
        dim3 grid((c.d.nx + kTX - 1) / kTX, (c.d.nz + kTJ - 1) / kTJ, k->nbatch);
        hipLaunchKernelGGL(k_dz_dense, grid, dim3(256), 0, c.stream, k->in, k->out, c.d.nz, c.d.nx, c.MT[k->ibc - 1],
                           nullptr, nullptr, 0, 0.0);
        DCHK(hipGetLastError());
    }
    return hipSuccess;
}

// Dz3^T of the dxi_z/dz adjoint DZB, and the adjoint of its kept last row
// (-dxi_x/dx unstretch, physics2d.f90:954) into the last row of DXB: by the
// segmented solve itself, or by a column sum.
static hipError_t dz3_T(const DiscreteCtx &c, const DiscreteWork &w)
{
    const Dims &d = c.d;
    if (discrete_segmented(c, d.S)) {
        ZDer a = zder_args(c, w.DZB, w.DZ3B, d.S, 3, true);
        a.prebar = w.DXB + (size_t)(d.nz - 1) * d.nx;
        a.prebar_stride = (size_t)d.nz * d.nx;
        a.prebar_add = -c.unstretch_last;
        return launch_zder(a, c.zseg, c.stream);
    }
    DCHK(dz_T(c, {w.DZB, w.DZ3B, d.S, 3}, nullptr, w.PB));
    hipLaunchKernelGGL(k_adj_preset, grid1((size_t)d.S * d.nx), dim3(256), 0, c.stream, w.PB, w.DXB, d.nz, d.nx, d.S,
                       c.unstretch_last);
    return hipGetLastError();
}

static hipError_t ddx(const DiscreteCtx &c, const double *in, double *out, int nrows, const double *in2 = nullptr,
                      double *out2 = nullptr, int nrows2 = 0)
{
    return launch_ddx_rows2(in, out, nrows, in2, out2, nrows2, c.d.nx, c.bg.tw, c.bg.dmul, c.bg.cdx, c.bg.stretchx,
                            c.stream);
}

// One forward stage: the next stage's input Yn = U + beta * RHS(Y, t) (Yn may be Y,
// not U) and the stage quantities D = [div, dvx/dx, dvz/dx, dvx/dz, dvz/dz].
static hipError_t fwd_stage(const DiscreteCtx &c, const DiscreteWork &w, const double *Y, int t, const double *U,
                            double beta, double *Yn, double *D)
{
    const Dims &d = c.d;
    const Views v{w.SN, w.PZ1, w.PX1};
    const int S = d.S;
    // dxi_x/dx; dv_x/dx, dv_z/dx
    DCHK(ddx(c, Y, w.T0, S * d.nz, Y + 2 * w.SN, D + w.SN, 2 * S * d.nz));
    // dxi_z/dz (ibc 3, kept last row -dxi_x/dx unstretch); dv_x/dz, dv_z/dz (ibc 1)
    const ZGroup vel{Y + 2 * w.SN, D + 3 * w.SN, 2 * S, 1};
    DCHK(dz(c, {Y + w.SN, w.T1, S, 3}, &vel, w.T0 + (size_t)(d.nz - 1) * d.nx, (size_t)d.nz * d.nx,
            -c.unstretch_last));
    hipLaunchKernelGGL(k_fwd_b, grid2(d), dim3(256), 0, c.stream, d, c.bg, v, Y, w.T0, w.T1, D, w.T2, w.T3, U, beta,
                       Yn);
    DCHK(hipGetLastError());
    // dp/dx, dp/dz (ibc 2, its first row 0)
    DCHK(ddx(c, w.T2, w.T0, S * d.nz));
    DCHK(dz(c, {w.T2, w.T1, S, 2}, nullptr, nullptr, 0, 0.0));
    hipLaunchKernelGGL(k_fwd_c, grid2(d), dim3(256), 0, c.stream, d, c.bg, v, c.src, t, Y, w.T0, w.T1, w.T3,
                       D + w.SN, U, beta, Yn);
    return hipGetLastError();
}

// One forward step U -> Unew (Unew != U), keeping the stage quantities in
// Dst[5] when not null.
static hipError_t fwd_step(const DiscreteCtx &c, const DiscreteWork &w, const double *U, int t, double *Unew,
                           double *Dst)
{
    for (int s = 0; s < 5; s++)
        DCHK(fwd_stage(c, w, s == 0 ? U : w.Y, t, U, s < 4 ? c.betas[s + 1] : c.deltat, w.Y,
                       Dst ? Dst + (size_t)s * 5 * w.SN : w.Dscr));
    hipLaunchKernelGGL(k_filter, grid_filter(c.d), dim3(256), 0, c.stream, c.d, Views{w.SN, w.PZ1, w.PX1}, w.Y, Unew);
    return hipGetLastError();
}

// Transpose of one step at time t: lam (adjoint of the state after the step)
// -> acc, the adjoint of U_t, accumulating the gradient into G.  Dkept: the
// step's stage quantities [5][5][SN] kept by the segment recompute, or null to
// recompute them from U here.
static hipError_t bwd_step(const DiscreteCtx &c, const DiscreteWork &w, const double *U, int t, const double *lam,
                           double *acc, double *G, const double *Dkept)
{
    const Dims &d = c.d;
    const Views v{w.SN, w.PZ1, w.PX1};
    const int S = d.S;
    const double *Dst = Dkept;
    if (!Dst) {
        DCHK(fwd_step(c, w, U, t, w.Unext, w.Dst));          // the stage quantities of this step
        Dst = w.Dst;
    }
    hipLaunchKernelGGL(k_filter_T, grid_filter(d), dim3(256), 0, c.stream, d, v, lam, c.deltat, acc, w.Rb);
    DCHK(hipGetLastError());
    for (int s = 4; s >= 0; s--) {
        const double beta = s > 0 ? c.betas[s] : 0.0;
        hipLaunchKernelGGL(k_adj_a, grid2(d), dim3(256), 0, c.stream, d, c.bg, v, w.Rb, acc, beta, w.FX, w.FZ, w.GZ);
        DCHK(hipGetLastError());
        DCHK(ddx(c, w.FX, w.DFX, 3 * S * d.nz));
        const ZGroup gradp{w.GZ, w.DGZ, S, 2};
        DCHK(dz_T(c, {w.FZ, w.DFZ, 2 * S, 1}, &gradp, nullptr));
        hipLaunchKernelGGL(k_adj_b, grid2(d), dim3(256), 0, c.stream, d, c.bg, v, w.Rb, acc, beta, w.DFX, w.DFZ, w.DGZ,
                           Dst + (size_t)s * 5 * w.SN, w.XZP, w.DXB, w.DZB, G);
        DCHK(hipGetLastError());
        DCHK(dz3_T(c, w));
        DCHK(ddx(c, w.DXB, w.DDXB, S * d.nz));
        hipLaunchKernelGGL(k_adj_c, grid1(w.SN), dim3(256), 0, c.stream, v, w.DDXB, w.XZP, w.DZ3B, w.Rb, acc, beta);
        DCHK(hipGetLastError());
    }
    return hipSuccess;
}

hipError_t discrete_gradient(const DiscreteCtx &c, const DiscreteWork &w, int maxtime, int interval,
                             const double *gvz, int nt, double *G)
{
    const Dims &d = c.d;
    const int S = d.S;
    const int C = interval;
    const int nseg = (maxtime + C) / C;                       // segments start at 0, C, 2C, ...
    // forward pass from the zero state, keeping the state at every segment
    // start; the last segment's own steps are left to its recompute
    double *U = w.U, *Un = w.Unext;
    DCHK(launch_fill(U, w.NST, 0.0, c.stream));
    for (int t = 0; t <= (nseg - 1) * C; t++) {
        if (t % C == 0)
            DCHK(hipMemcpyAsync(w.ck + (size_t)(t / C) * w.NST, U, w.NST * sizeof(double), hipMemcpyDeviceToDevice,
                                c.stream));
        if (t == (nseg - 1) * C) break;
        DCHK(fwd_step(c, w, U, t, Un, nullptr));
        std::swap(U, Un);
    }
    double *lam = w.lam, *acc = w.acc;
    DCHK(launch_fill(lam, w.NST, 0.0, c.stream));
    DCHK(launch_fill(G, 3 * w.SN, 0.0, c.stream));
    for (int j = nseg - 1; j >= 0; j--) {
        const int t0 = j * C, t1 = std::min(maxtime, t0 + C - 1);
        // states U_t of the segment
        DCHK(hipMemcpyAsync(w.seg, w.ck + (size_t)j * w.NST, w.NST * sizeof(double), hipMemcpyDeviceToDevice,
                            c.stream));
        // states U_t0..U_t1 and, when w.Dseg holds a segment, the stage
        // quantities of steps t0..t1 (the state after step t1 is not needed)
        const size_t D1 = (size_t)25 * w.SN;
        for (int t = t0; t < t1 + (w.Dseg ? 1 : 0); t++)
            DCHK(fwd_step(c, w, w.seg + (size_t)(t - t0) * w.NST, t,
                          t < t1 ? w.seg + (size_t)(t - t0 + 1) * w.NST : w.Unext,
                          w.Dseg ? w.Dseg + (size_t)(t - t0) * D1 : nullptr));
        for (int t = t1; t >= t0; t--) {
            if (t % c.steps == 0) {                            // output k after step t
                hipLaunchKernelGGL(k_inject, grid1((size_t)S * d.nx), dim3(256), 0, c.stream, lam, gvz, t / c.steps, nt,
                                   c.orow, d.nz, d.nx, S, w.SN);
                DCHK(hipGetLastError());
            }
            DCHK(bwd_step(c, w, w.seg + (size_t)(t - t0) * w.NST, t, lam, acc, G,
                          w.Dseg ? w.Dseg + (size_t)(t - t0) * D1 : nullptr));
            std::swap(lam, acc);
        }
    }
    return hipSuccess;
}

hipError_t discrete_flow_chain(const DiscreteCtx &c, const DiscreteWork &w, const double *G, const double *rho0,
                               const double *c2, const double *psi, double scale, double dimc, double *gpsi,
                               double *gc)
{
    const Dims &d = c.d;
    const Views v{w.SN, w.PZ1, w.PX1};
    const int n2 = d.nz * d.nx;
    hipLaunchKernelGGL(k_flow_in, grid1(w.SN), dim3(256), 0, c.stream, v, n2, rho0, G, w.FX, w.FZ);
    DCHK(hipGetLastError());
    DCHK(dz_T(c, {w.FX, w.DFX, d.S, 1}, nullptr, nullptr));                  // Dz1^T (Gx / rho0)
    DCHK(ddx(c, w.FZ, w.DFZ, d.S * d.nz));                                   // dx (Gz / rho0)
    hipLaunchKernelGGL(k_flow_out, grid1(w.SN), dim3(256), 0, c.stream, v, n2, rho0, c2, psi, scale, dimc, G,
                       w.DFX, w.DFZ, gpsi, gc);
    return hipGetLastError();
}

hipError_t discrete_apply(const DiscreteCtx &c, const double *in, double *out, int nbatch, int which,
                          double *presetN_bar)
{
    // which: 0..2 Dz of ibc 1..3, 3..5 their transposes
    if (which < 0 || which > 5) return hipErrorInvalidValue;
    return which < 3 ? dz(c, {in, out, nbatch, which + 1}, nullptr, nullptr, 0, 0.0)
                     : dz_T(c, {in, out, nbatch, which - 2}, nullptr, which == 5 ? presetN_bar : nullptr);
}

}  // namespace sparc
