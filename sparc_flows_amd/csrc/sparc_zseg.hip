// sparc_zseg.hip -- segmented z kernels: the z passes of a 3D stage
// (displacement.f90:400-473) with the compact-FD derivatives of dbyd2 /
// mtridag (dbyd2.f:8-200) solved by segments.
//
// A block holds NC neighbouring columns for all nz rows: every column is cut
// into P <= kZSegP segments of MS rows, one lane per (column, segment), columns
// fastest, so that a wave instruction touches 64 / NC rows of 8 NC consecutive
// bytes.  A z-derivative is the segment's right-hand side from a window of MS + 6
// rows, a Thomas solve of the segment in registers, the exchange of the
// segment end values through LDS and the exact correction with the interface
// values (sparc_seg.h, the arithmetic of the 2D column pass).  Each input row
// is read once from memory (the windows' six halo rows hit the caches) and
// nothing is written but the results: the one-lane sweeps this replaces write
// and read back their forward-sweep values and re-read the field.
#include <algorithm>

#include "sparc_launch.h"
#include "sparc_zseg.h"

namespace sparc {
namespace {

// Loads and stores at a 32-bit byte offset from a wave-uniform base address
// (SGPR base + VGPR offset); arrays indexed this way span less than 2^32 bytes.
#define SPARC_GLOBAL __attribute__((address_space(1)))
__device__ __forceinline__ double ldg(const double *base, unsigned ob)
{
    return *(const SPARC_GLOBAL double *)((const SPARC_GLOBAL char *)base + ob);
}
__device__ __forceinline__ void stg(double *base, unsigned ob, double v)
{
    *(SPARC_GLOBAL double *)((SPARC_GLOBAL char *)base + ob) = v;
}

// One lane's part of a column: segment s, rows a .. a + MS - 1 of column c.
struct Lane {
    int c, s, a;
    bool act, first, last;      // a segment of the column; its first; it holds rows nz-2, nz-1
    unsigned col, rowb;         // byte offset of row 0; bytes per row
    int nz;
    // byte offset of row r, clamped to the column
    __device__ __forceinline__ unsigned row(int r) const { return col + (unsigned)min(max(r, 0), nz - 1) * rowb; }
    __device__ __forceinline__ bool valid(int i) const { return act && a + i < nz; }
};

// The window and end rows of one field's segment.
template <int MS>
__device__ __forceinline__ void load_window(const double *F, const Lane &ln, double (&win)[MS + 6], double (&e)[5])
{
#pragma unroll
    for (int k = 0; k < MS + 6; k++) win[k] = ldg(F, ln.row(ln.a - 3 + k));
#pragma unroll
    for (int k = 0; k < 5; k++) e[k] = 0.0;
    if (ln.last) {
#pragma unroll
        for (int k = 0; k < 5; k++) e[k] = ldg(F, ln.row(ln.nz - 5 + k));
    }
}

// n doubles (even) from global memory to LDS by the whole block, 16 bytes per
// load, four loads in flight.
__device__ __forceinline__ void stage_lds(double *dst, const double *src, int n, int tid, int nthr)
{
    const double2 *s2 = (const double2 *)src;
    double2 *d2 = (double2 *)dst;
    const int n2 = n >> 1;
    for (int q = tid; q < n2; q += 4 * nthr) {
        double2 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = s2[min(q + u * nthr, n2 - 1)];
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (q + u * nthr < n2) d2[q + u * nthr] = v[u];
    }
}

__device__ __forceinline__ void zero_lds(double *dst, int n, int tid, int nthr)
{
    for (int q = tid; q < n; q += nthr) dst[q] = 0.0;
}

}  // namespace

// The z-derivative of a batch of fields, or its transpose: D = S A^-1 B with B
// dbyd2's right-hand side, A its tridiagonal matrix and S the stretch, so D^T =
// B^T A^-T S: the solve by the transposed tables first, then B^T, a stencil on
// the solved column (its four edge rows apart), through an LDS tile.  Bound:
// HBM for a large batch (16 B per point), latency for a small one.  us per
// launch, one-lane Thomas sweep (or, in the discrete adjoint, the product with
// the dense nz x nz matrix) -> here: one 128x150 field 52 -> 6, 16 fields of
// 256x300 58 -> 7.5 (transposed 9.3).
constexpr int kZdCols = 16;
template <int MS, bool TR>
__global__ __launch_bounds__(512) void k_zder(ZDer z, ZSeg sg)
{
    constexpr int NC = kZdCols;
    extern __shared__ __align__(16) double lds[];
    const int P = sg.P, hw = sg.hw, nzp = P * MS, LY = 2 * P + 4 * hw + 2, nset = zseg_set_len(P, hw, MS);
    double *const band = lds, *const yb = lds + nset;       // [NC][LY]
    double *const tile = yb + NC * LY + 2 * NC;             // filter, transpose: [nzp] rows of NC, two more before and after
    const int tid = threadIdx.x, nthr = blockDim.x, nz = z.nz;
    const int c0 = (int)blockIdx.x * NC + tid % NC;
    const bool two = (int)blockIdx.y >= z.nbatch;           // the second set of fields
    const int ibc = two ? z.ibc2 : z.ibc, fb = (int)blockIdx.y - (two ? z.nbatch : 0);
    const size_t fo = (size_t)fb * nz * z.ncols;
    const double *const in = (two ? z.in2 : z.in) + fo;
    double *const oc = (two ? z.out2 : z.out) + fo;
    const double *const pre = two ? nullptr : z.pre;
    Lane ln;
    ln.c = tid % NC;
    ln.s = min(tid / NC, P - 1);
    ln.act = tid / NC < P && c0 < z.ncols;
    ln.a = ln.s * MS;
    ln.first = ln.s == 0;
    ln.last = ln.a + MS > nz - 2;
    ln.rowb = (unsigned)z.ncols * 8u;
    ln.col = (unsigned)min(c0, z.ncols - 1) * 8u;
    ln.nz = nz;
    const bool seg = tid / NC < P;
    double Y[MS], st[MS];
#pragma unroll
    for (int i = 0; i < MS; i++) st[i] = z.stretch ? z.stretch[min(ln.a + i, nz - 1)] : 1.0;
    double win[MS + 6], e[5], p0 = 0.0, pN = 0.0;
    if (TR) {
#pragma unroll
        for (int i = 0; i < MS; i++) Y[i] = ldg(in, ln.row(ln.a + i));
    } else {
        load_window<MS>(in, ln, win, e);
        if (ibc == 2 && !z.zero_kept) p0 = ldg(oc, ln.row(0));
        if (ibc == 3 && (pre || !z.zero_kept))
            pN = pre ? z.pre_scale * pre[(size_t)fb * z.pre_stride + (ln.col >> 3)]
                       : ldg(oc, ln.row(nz - 1));
    }
    zero_lds(yb, NC * LY, tid, nthr);
    stage_lds(lds, sg.img + (size_t)(TR ? 3 + ibc : ibc) * nset, nset, tid, nthr);
    if (TR && tid < 2 * NC) {                               // zero rows around the tile
        tile[tid - 2 * NC] = 0.0;
        tile[nzp * NC + tid] = 0.0;
    }
    __syncthreads();
    const double *const zt = band + 2 * P * (4 * hw + 4) + seg_kind(ln.s, P) * MS;
    auto tab = [&](int t, int i) { return zt[t * 3 * MS + i]; };
    if (TR) {
#pragma unroll
        for (int i = 0; i < MS; i++) Y[i] = ln.a + i < nz ? Y[i] * st[i] : 0.0;
    } else {
        seg_rhs<MS>([&](int k) { return win[k]; }, e, Y, ln.a, nz, ln.first, ln.last, ibc, p0, pN, sg.c1, sg.c2,
                    sg.cb);
    }
    seg_solve<MS>(Y, tab);
    double *const yc = yb + ln.c * LY;
    if (seg) {
        yc[2 * hw + 2 * ln.s] = Y[0];
        yc[2 * hw + 2 * ln.s + 1] = Y[MS - 1];
    }
    __syncthreads();
    seg_correct<MS>(Y, ln.s, P, hw, yc, band, tab);
    if (!TR) {
#pragma unroll
        for (int i = 0; i < MS; i++) Y[i] = Y[i] * st[i];
        if (!z.filt) {
#pragma unroll
            for (int i = 0; i < MS; i++)
                if (ln.valid(i)) stg(oc, ln.col + (unsigned)(ln.a + i) * ln.rowb, Y[i]);
            return;
        }
    }
    // rows 0, 1, nz-2, nz-1 of the solved column enter B^T by their own
    // coefficients: kept apart, and zero in the tile
    double *const ed = yb;                                  // [4][NC], once every lane has left yb
    __syncthreads();
    if (seg) {
#pragma unroll
        for (int i = 0; i < MS; i++) {
            const int j = ln.a + i, er = j < 2 ? j : j - nz + 4;
            const bool edge = TR && (j < 2 || (j >= nz - 2 && j < nz));
            tile[j * NC + ln.c] = edge || j >= nz ? 0.0 : Y[i];
            if (edge) ed[er * NC + ln.c] = Y[i];
            if (TR && z.prebar && !two && ibc == 3 && j == nz - 1 && ln.act) {
                double *const pb = z.prebar + (size_t)fb * z.prebar_stride + c0;
                *pb = z.prebar_add != 0.0 ? *pb + z.prebar_add * Y[i] : Y[i];
            }
        }
    }
    __syncthreads();
    if (!ln.act) return;
    const double *const t = tile + ln.c, *const eb = two ? z.eb2 : z.eb;
#pragma unroll
    for (int i = 0; i < MS; i++) {
        const int j = ln.a + i;
        if (j >= nz) break;
        double v;
        if (TR) {
            v = sg.c1 * (t[(j - 1) * NC] - t[(j + 1) * NC]) + sg.c2 * (t[(j - 2) * NC] - t[(j + 2) * NC]);
            const int k = j < 5 ? j : j - nz + 5;
            if (j < 5) v += eb[k] * ed[ln.c] + eb[5 + k] * ed[NC + ln.c];
            if (j >= nz - 5) v += eb[10 + j - nz + 5] * ed[2 * NC + ln.c] + eb[15 + j - nz + 5] * ed[3 * NC + ln.c];
        } else if (j == 0 || j == nz - 1) {
            v = Y[i];
        } else if (j <= 4 || j >= nz - 5) {                // FILTER_VAR_Z (kernels.f90:891-928)
            v = 0.5 * (t[(j + 1) * NC] + t[(j - 1) * NC]);
        } else {
            v = filt11(t, (size_t)j * NC, NC);
        }
        stg(oc, ln.col + (unsigned)j * ln.rowb, v);
    }
}

namespace {

size_t zder_lds(const ZDer &a, const ZSeg &sg)
{
    return sizeof(double) * ((size_t)zseg_set_len(sg.P, sg.hw, sg.m) + (size_t)kZdCols * yb_len(sg.P, sg.hw) +
                             (a.filt || a.transposed ? (size_t)kZdCols * (sg.P * sg.m + 4) : 0));
}
// Raises a kernel's dynamic-LDS limit when a launch needs more than the default.
hipError_t allow_lds(const void *k, size_t n)
{
    return n > 64 * 1024 ? hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)n) : hipSuccess;
}
int lanes(int cols, int P) { return (cols * P + 63) / 64 * 64; }

}  // namespace

bool zder_fits(const ZDer &a, const ZSeg &sg)
{
    return sg.img && sg.P <= kZSegP && (size_t)a.nz * a.ncols < ((size_t)1 << 28) && a.nbatch + a.nbatch2 <= 65535 &&
           zder_lds(a, sg) <= 160 * 1024;
}

hipError_t launch_zder(const ZDer &a, const ZSeg &sg, hipStream_t st)
{
    const size_t shm = zder_lds(a, sg);
    const dim3 grid((unsigned)((a.ncols + kZdCols - 1) / kZdCols), (unsigned)(a.nbatch + a.nbatch2)), block(lanes(kZdCols, sg.P));
#define L(M)                                                                                     \
    if (sg.m == M) {                                                                             \
        const void *k = a.transposed ? (const void *)k_zder<M, true> : (const void *)k_zder<M, false>; \
        const hipError_t e = allow_lds(k, shm);                                                  \
        if (e != hipSuccess) return e;                                                           \
        if (a.transposed) hipLaunchKernelGGL((k_zder<M, true>), grid, block, shm, st, a, sg);    \
        else hipLaunchKernelGGL((k_zder<M, false>), grid, block, shm, st, a, sg);                \
        return hipGetLastError();                                                                \
    }
    SPARC_ZDER_SIZES(L)
#undef L
    return hipErrorInvalidValue;
}

namespace d3 {

// Zp: d xi_z/dz (ibc 1) with the z-PML (displacement.f90:400-409), div, p and
// rho' (:411-415), and rho' g / rho0 for RHS v_z (:458).  Bound: HBM, 48 B per
// point (xi_z, two x/y-derivatives and c^2 rho0 read, two fields written).
// 16 columns are one 128-byte line of every row.  us per launch, one-lane
// sweep -> here: 256x256x300 395 -> 290 (3.3 TB/s of a 4.9 TB/s copy),
// 128x128x150 182 -> 40, 96x90x100 104 -> 20.
constexpr int kZpCols = 16;
template <int MS>
__global__ __launch_bounds__(512) void k3_zp_seg(Z3 z, ZSeg sg)
{
    constexpr int NC = kZpCols, U = MS <= 8 ? MS : 4;
    extern __shared__ __align__(16) double lds[];
    const int P = sg.P, hw = sg.hw, nzp = P * MS, LY = 2 * P + 4 * hw + 2, nset = zseg_set_len(P, hw, MS);
    double *const band = lds, *const tabs = band + 2 * P * (4 * hw + 4);
    double *const yb = lds + nset;                      // [NC][LY]
    double *const pf = yb + NC * LY;                    // [6][nzp] stretch, d p0/dz, d rho0/dz, rho0, 1/rho0, g
    const int tid = threadIdx.x, nthr = blockDim.x, nz = z.nz;
    const unsigned bl = xcd_block(blockIdx.x, gridDim.x);
    const int c0 = (int)bl * NC + tid % NC;
    const bool real = c0 < z.nxy;
    Lane ln;
    ln.c = tid % NC;
    ln.s = min(tid / NC, P - 1);
    ln.act = tid / NC < P && real;
    ln.a = ln.s * MS;
    ln.first = ln.s == 0;
    ln.last = ln.a + MS > nz - 2;
    ln.rowb = (unsigned)z.nxy * 8u;
    ln.col = (unsigned)min(c0, z.nxy - 1) * 8u;
    ln.nz = nz;
    double win[MS + 6], e[5];
    load_window<MS>(z.B, ln, win, e);
    zero_lds(yb, NC * LY, tid, nthr);
    stage_lds(lds, sg.img + nset, nset, tid, nthr);         // ibc 1
    for (int q = tid; q < nzp; q += nthr) {
        const int j = min(q, nz - 1);
        const double v0 = z.stretch[j], v1 = z.gp0z[j], v2 = z.gr0z[j], v3 = z.rho0[j], v4 = z.rhoinv[j], v5 = z.g[j];
        pf[q] = v0;
        pf[nzp + q] = v1;
        pf[2 * nzp + q] = v2;
        pf[3 * nzp + q] = v3;
        pf[4 * nzp + q] = v4;
        pf[5 * nzp + q] = v5;
    }
    __syncthreads();
    const double *const zt = tabs + seg_kind(ln.s, P) * MS;
    auto tab = [&](int t, int i) { return zt[t * 3 * MS + i]; };
    double Y[MS], own[MS];
    seg_rhs<MS>([&](int k) { return win[k]; }, e, Y, ln.a, nz, ln.first, ln.last, 1, 0.0, 0.0, sg.c1, sg.c2, sg.cb);
#pragma unroll
    for (int i = 0; i < MS; i++) own[i] = win[3 + i];
    seg_solve<MS>(Y, tab);
    double *const yc = yb + ln.c * LY;
    if (tid / NC < P) {
        yc[2 * hw + 2 * ln.s] = Y[0];
        yc[2 * hw + 2 * ln.s + 1] = Y[MS - 1];
    }
    __syncthreads();
    seg_correct<MS>(Y, ln.s, P, hw, yc, band, tab);
#pragma unroll
    for (int i0 = 0; i0 < MS; i0 += U) {
        double dxi[U], dyi[U], c2r[U], fz[U], az[U], bz[U], ps[U], pb[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const unsigned q = ln.row(ln.a + min(i0 + u, MS - 1));
            dxi[u] = ldg(z.dxi, q);
            dyi[u] = ldg(z.dyi, q);
            c2r[u] = ldg(z.c2rho0, q);
            fz[u] = 1.0;
            az[u] = bz[u] = ps[u] = pb[u] = 0.0;
        }
        if (ln.a + i0 < z.nb || ln.a + min(i0 + U, MS) > nz - z.nt) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int pj = pml_index(min(ln.a + i0 + u, nz - 1), nz, z.nb, z.nt);
                if (pj >= 0) {
                    const unsigned qp = ln.col + (unsigned)pj * ln.rowb;
                    fz[u] = ldg(z.fz, qp);
                    az[u] = ldg(z.az, qp);
                    bz[u] = ldg(z.bz, qp);
                    ps[u] = ldg(z.psi, qp);
                    pb[u] = ldg(z.pml, qp);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = i0 + u;
            if (i >= MS) break;
            const int j = ln.a + i;
            const double *const f = pf + j;
            double dz = Y[i] * f[0];
            const double gp = f[nzp] * fz[u], gr = f[2 * nzp] * fz[u];
            const int pj = pml_index(j, nz, z.nb, z.nt);
            const bool v = ln.valid(i);
            if (pj >= 0 && v) stg(z.pnext, ln.col + (unsigned)pj * ln.rowb, pb[u] + z.beta * (az[u] * dz + bz[u] * ps[u]));
            dz = dz + ps[u];
            const double div = (dxi[u] + dyi[u]) + dz;
            const double p = -(c2r[u] * div) - own[i] * gp;
            const double rho = -(f[3 * nzp] * div) - own[i] * gr;
            if (v) {
                const unsigned q = ln.col + (unsigned)j * ln.rowb;
                stg(z.P, q, p);
                stg(z.RG, q, f[4 * nzp] * rho * f[5 * nzp]);
            }
        }
    }
}

// Zv: the z-derivatives of v_x, v_y, v_z (ibc 1) and of p (ibc 0, with the
// z-PML, :422-431) of the lane's segment, all four kept in registers, then RHS
// v_i = -2 v0 . grad v_i - d_i p / rho0 (:436-452), RHS v_z - rho' g / rho0
// (:458) + forcing * source_dep (:460-462), RHS xi_i = v_i (:466-468), rows 1
// and nz zeroed (:470-473).  The xi updates need only v: they are written as
// each v window passes.  Bound: HBM, 224 B per point (22 fields read, 6
// written).  us per launch, one-lane sweep -> here: 256x256x300 1350 -> 1105
// (4.0 TB/s), 128x128x300 968 -> 360, 128x128x150 497 -> 143, 96x90x100 264 ->
// 68, 32x32x40 91 -> 19.  Segments of at most 10 rows keep the four derivatives
// and a row's loads in 256 registers; 19-row segments spilled (1440 us at
// 256x256x300).  12, 14 and 16 rows (nz above 320, and 22 depths below whose last
// segment would hold fewer than three rows otherwise: nz = 121, 122, 131, 132, 141, 142,
// 151, 152, 241, 242, 261, 262 and so on by tens from 271 to 312) keep 160 to 536 bytes a lane in
// scratch and still win: 128x128x121 405 -> 145, 96x90x301 920 -> 294, 256x256x301
// 1326 -> 1296, 256x256x448 2011 -> 1762.  One lane group per field, which reads v0 once
// per group, took 1500 us there, and blocks of 8 columns 1750: below 128 bytes
// a row's piece is half a line.
template <int MS, int NC>
__global__ __launch_bounds__(512, 2) void k3_zv_seg(Z3 z, ZSeg sg)
{
    constexpr int U = 1;
    extern __shared__ __align__(16) double lds[];
    const int P = sg.P, hw = sg.hw, nzp = P * MS, LY = 2 * P + 4 * hw + 2, nset = zseg_set_len(P, hw, MS);
    double *const yb = lds + 2 * nset;                  // [4][NC][LY]
    double *const pf = yb + 4 * NC * LY;                // [3][nzp] stretch, 1/rho0, source_dep
    const int tid = threadIdx.x, nthr = blockDim.x, nz = z.nz;
    const unsigned bl = xcd_block(blockIdx.x, gridDim.x);
    const int c0 = (int)bl * NC + tid % NC;
    Lane ln;
    ln.c = tid % NC;
    ln.s = min(tid / NC, P - 1);
    ln.act = tid / NC < P && c0 < z.nxy;
    ln.a = ln.s * MS;
    ln.first = ln.s == 0;
    ln.last = ln.a + MS > nz - 2;
    ln.rowb = (unsigned)z.nxy * 8u;
    ln.col = (unsigned)min(c0, z.nxy - 1) * 8u;
    ln.nz = nz;
    zero_lds(yb, 4 * NC * LY, tid, nthr);
    stage_lds(lds, sg.img, 2 * nset, tid, nthr);            // ibc 0, ibc 1
    for (int q = tid; q < nzp; q += nthr) {
        const int j = min(q, nz - 1);
        const double v0 = z.stretch[j], v1 = z.rhoinv[j], v2 = z.srcdep[j];
        pf[q] = v0;
        pf[nzp + q] = v1;
        pf[2 * nzp + q] = v2;
    }
    // forcing of this column (physics.f90:678-737 for the adjoint)
    double forcing = 0.0;
    if (ln.a <= z.e_rad + 4 && ln.a + MS > z.e_rad - 4 && z.time <= z.src.limit) {
        const int c = (int)(ln.col >> 3);
        if (z.src.mode == 1)
            forcing = (z.time >= 0 && z.time < z.src.nfwd) ? z.src.vr[c] * z.src.fwd[z.time] : 0.0;
        else if (z.src.mode == 2)
            forcing = lagrange_forcing(z.src, 0, c, z.nxy, z.time);
    }
    __syncthreads();
    const int kofs = 2 * P * (4 * hw + 4) + seg_kind(ln.s, P) * MS;
    double Y[4][MS];
#pragma unroll
    for (int f = 0; f < 4; f++) {
        const double *const band = lds + (f < 3 ? nset : 0), *const zt = band + kofs;
        double win[MS + 6], e[5];
        load_window<MS>(f < 3 ? z.B + (size_t)f * z.N : z.P, ln, win, e);
        if (f < 3) {
            const double *const ax = z.a + (size_t)f * z.N;
            double *const tx = z.tnext + (size_t)f * z.N, *const rx = z.rhs + (size_t)f * z.N;
            double bx[MS];
#pragma unroll
            for (int i = 0; i < MS; i++) bx[i] = ldg(ax, ln.row(ln.a + i));
#pragma unroll
            for (int i = 0; i < MS; i++) {
                const int j = ln.a + i;
                const double r = j == 0 || j == nz - 1 ? 0.0 : win[3 + i];
                if (ln.valid(i)) {
                    const unsigned q = ln.col + (unsigned)j * ln.rowb;
                    stg(tx, q, bx[i] + z.beta * r);
                    if (z.last) stg(rx, q, r);
                }
            }
        }
        seg_rhs<MS>([&](int k) { return win[k]; }, e, Y[f], ln.a, nz, ln.first, ln.last, f < 3 ? 1 : 0, 0.0, 0.0, sg.c1,
                    sg.c2, sg.cb);
        seg_solve<MS>(Y[f], [&](int t, int i) { return zt[t * 3 * MS + i]; });
        if (tid / NC < P) {
            double *const yc = yb + (f * NC + ln.c) * LY + 2 * hw + 2 * ln.s;
            yc[0] = Y[f][0];
            yc[1] = Y[f][MS - 1];
        }
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < 4; f++) {
        const double *const band = lds + (f < 3 ? nset : 0), *const zt = band + kofs;
        seg_correct<MS>(Y[f], ln.s, P, hw, yb + (f * NC + ln.c) * LY, band,
                        [&](int t, int i) { return zt[t * 3 * MS + i]; });
    }
    const size_t N = z.N, np = (size_t)(z.nb + z.nt) * z.nxy;
#pragma unroll
    for (int i0 = 0; i0 < MS; i0 += U) {
        double dx[3][U], dy[3][U], u0[3][U], gp[2][U], rg[U], bv[3][U], az[U], bz[U], ps[U], pb[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const unsigned q = ln.row(ln.a + min(i0 + u, MS - 1));
#pragma unroll
            for (int f = 0; f < 3; f++) {
                dx[f][u] = ldg(z.dxv + f * N, q);
                dy[f][u] = ldg(z.dyv + f * N, q);
                bv[f][u] = ldg(z.a + (3 + f) * N, q);
            }
            u0[0][u] = ldg(z.v0x, q);
            u0[1][u] = ldg(z.v0y, q);
            u0[2][u] = ldg(z.v0z, q);
            gp[0][u] = ldg(z.dxp, q);
            gp[1][u] = ldg(z.dyp, q);
            rg[u] = ldg(z.RG, q);
            az[u] = bz[u] = ps[u] = pb[u] = 0.0;
        }
        if (ln.a + i0 < z.nb || ln.a + min(i0 + U, MS) > nz - z.nt) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int pj = pml_index(min(ln.a + i0 + u, nz - 1), nz, z.nb, z.nt);
                if (pj >= 0) {
                    const unsigned qp = ln.col + (unsigned)pj * ln.rowb;
                    az[u] = ldg(z.az, qp);
                    bz[u] = ldg(z.bz, qp);
                    ps[u] = ldg(z.psi + np, qp);
                    pb[u] = ldg(z.pml + np, qp);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = i0 + u;
            if (i >= MS) break;
            const int j = ln.a + i;
            const bool edge = j == 0 || j == nz - 1, v = ln.valid(i);
            const unsigned q = ln.col + (unsigned)j * ln.rowb;
            const double st = pf[j], ri = pf[nzp + j];
            double adv[3], gpz = Y[3][i] * st;
#pragma unroll
            for (int f = 0; f < 3; f++)
                adv[f] = -2.0 * ((u0[0][u] * dx[f][u] + u0[1][u] * dy[f][u]) + u0[2][u] * (Y[f][i] * st));
            const int pj = pml_index(j, nz, z.nb, z.nt);
            if (pj >= 0 && v)
                stg(z.pnext + np, ln.col + (unsigned)pj * ln.rowb, pb[u] + z.beta * (az[u] * gpz + bz[u] * ps[u]));
            gpz = gpz + ps[u];
            double rhs[3];
            rhs[0] = edge ? 0.0 : adv[0] - ri * gp[0][u];
            rhs[1] = edge ? 0.0 : adv[1] - ri * gp[1][u];
            double rz = adv[2] - ri * gpz;
            rz = rz - rg[u];
            const int dk = j - z.e_rad;
            if (dk >= -4 && dk <= 4) rz = rz + forcing * pf[2 * nzp + j];
            rhs[2] = edge ? 0.0 : rz;
            if (v) {
#pragma unroll
                for (int f = 0; f < 3; f++) {
                    stg(z.tnext + (3 + f) * N, q, bv[f][u] + z.beta * rhs[f]);
                    if (z.last) stg(z.rhs + (3 + f) * N, q, rhs[f]);
                }
            }
        }
    }
}

namespace {

size_t zp_lds(const ZSeg &sg)
{
    return sizeof(double) * ((size_t)zseg_set_len(sg.P, sg.hw, sg.m) + (size_t)kZpCols * yb_len(sg.P, sg.hw) +
                             (size_t)6 * sg.P * sg.m);
}
size_t zv_lds(const ZSeg &sg, int nc)
{
    return sizeof(double) * ((size_t)2 * zseg_set_len(sg.P, sg.hw, sg.m) + (size_t)4 * nc * yb_len(sg.P, sg.hw) +
                             (size_t)3 * sg.P * sg.m);
}

}  // namespace

bool zseg3_fits(const Z3 &z, const ZSeg &sg)
{
    return sg.img && sg.m <= kZSegMax3 && sg.P <= kZSegP && z.N < ((size_t)1 << 28) && zp_lds(sg) <= 160 * 1024 &&
           zv_lds(sg, sg.P <= kZSegP / 2 ? 32 : 16) <= 160 * 1024;
}

hipError_t launch_zp_seg(const Z3 &z, const ZSeg &sg, hipStream_t st)
{
    const size_t shm = zp_lds(sg);
    const dim3 grid((unsigned)((z.nxy + kZpCols - 1) / kZpCols)), block(lanes(kZpCols, sg.P));
#define L(M)                                                                            \
    if (sg.m == M) {                                                                    \
        const hipError_t e = allow_lds((const void *)k3_zp_seg<M>, shm);                \
        if (e != hipSuccess) return e;                                                  \
        hipLaunchKernelGGL(k3_zp_seg<M>, grid, block, shm, st, z, sg);                  \
        return hipGetLastError();                                                       \
    }
    SPARC_ZSEG_SIZES(L)
#undef L
    return hipErrorInvalidValue;
}

hipError_t launch_zv_seg(const Z3 &z, const ZSeg &sg, hipStream_t st)
{
    // 32 columns (256 bytes of each row) where they fill the 256 compute units and
    // 512 threads, but not at four rows a segment, whose registers let a unit hold
    // three blocks of 16 columns and one of 32.  us on 16 / 32 columns: 128x128x150
    // 164 / 141, x100 149 / 106; 100x100x150 118 / 112, x100 77 / 74; 90x91x100 46 / 43;
    // four rows (nz = 60): 64x64 25 / 34, 96x90 52 / 65, 128x112 64 / 68, 160x160 143 / 154,
    // 192x192 205 / 204.  32 lose elsewhere where their last round of blocks is nearly
    // empty or the grid is large: 96x90x100 (270 blocks) 64 / 68, 160x160x150 226 / 251,
    // 256x256x150 527 / 542 (x100 427 / 389).
    const int nc = sg.P <= kZSegP / 2 && sg.m > 4 && z.nxy >= 32 * 256 ? 32 : 16;
    const size_t shm = zv_lds(sg, nc);
    const dim3 grid((unsigned)((z.nxy + nc - 1) / nc)), block(lanes(nc, sg.P));
#define L(M)                                                                                 \
    if (sg.m == M) {                                                                         \
        constexpr int W = M > 4 ? 32 : 16;                                                   \
        auto *const k = nc == 32 ? &k3_zv_seg<M, W> : &k3_zv_seg<M, 16>;                     \
        const hipError_t e = allow_lds((const void *)k, shm);                                \
        if (e != hipSuccess) return e;                                                       \
        hipLaunchKernelGGL(k, grid, block, shm, st, z, sg);                                  \
        return hipGetLastError();                                                            \
    }
    SPARC_ZSEG_SIZES(L)
#undef L
    return hipErrorInvalidValue;
}

}  // namespace d3
}  // namespace sparc
