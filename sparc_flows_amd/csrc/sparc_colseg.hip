// sparc_colseg.hip -- segmented column pass of the 2D option-17 solver.
//
// Same work as the column half of one RK stage of step.f90:48-106 /
// physics2d.f90:943-1094: the z-derivatives of xi_z, v_z, v_x and p by dbyd2
// (dbyd2.f:8-200, mtridag.f:95-112), the z-PML, divergence, pressure and
// density perturbation, RHS v_z with the source and flow terms, the zeroed
// rows and columns, the RK stage update and, after the last stage,
// FILTER_VARS_2D (physics2d.f90:509-556).
//
// Every column is split into P <= kSegMax segments of exactly MS rows; one
// lane holds one segment of one field of one column (k_colsplit), or of all three
// (k_colone, batches), and a block covers TC columns.  Each z-derivative is: dbyd2 right-hand side
// from a 7-row window, local Thomas solve of the segment, exchange of the
// segment's end values through LDS, and the exact correction
// y - L_{s-1} V - F_{s+1} W.  Loads use clamped row indices and 32-bit byte
// offsets from wave-uniform bases; stores of padding rows are masked off.
#include <algorithm>
#include <type_traits>

#include "sparc_device.h"
#include "sparc_launch.h"
#include "sparc_seg.h"

namespace sparc {

// The epilogue profiles of the LDS image, [kZF][nzp], in this order.
enum PfRow { F_STR = 0, F_G, F_RHO, F_GRHO, F_GP, F_RINV };
static_assert(F_RINV + 1 == kZF, "staged z profiles");
// The block's z-PML data staged in LDS, [kPL][nzpml][TC]: az, bz, fz and the
// two auxiliary fields (psivz, psip), stage value and base.
enum PRow { P_AZ = 0, P_BZ, P_FZ, P_T0, P_B0, P_T1, P_B1, kPL };

// Dynamic LDS of one block, in this order: the staged region (the three
// sets' interface rows [3][nk][2][4hw+4], the segment tables [kZS][3][ms],
// the z profiles [kZF][nzp], dbyd2's kCB boundary-row coefficients, the z-PML data [kPL][nzpml][TC], the mode-3 source z profile [nzp] (zero on
// padding rows; only staged in that mode); filled in one pass at the start), the four
// end-value exchange buffers [4][TC][2P + 4hw + 2] (each column's 2P end
// values between 2hw and 2hw+2 zeros), and three [TC][nzp] row buffers: the
// group-1 and group-0 parts of RHS v_z and p.
// A set's interface rows repeat away from the column's ends, so keeping one
// interior pair holds a block's LDS at 76 KB (TC = 4, MS = 10, nz = 300, 24 PML
// rows) where all 2P rows took 104 KB, and the image that it stages at 3 846 doubles
// for 7 302.
inline size_t colsplit_staged(int tc, const SegTab &sg, int nzpml)
{
    // rounded up to an even count, so that the end-value buffers after it
    // start on 16 bytes (the interface correction reads them in pairs)
    const size_t n = (size_t)3 * sg.nk * 2 * (4 * sg.hw + 4) + (size_t)kZS * 3 * sg.m + (size_t)kZF * sg.nzp +
                     (size_t)kCB + (size_t)kPL * nzpml * tc + (size_t)sg.nzp;
    return (n + 1) & ~(size_t)1;
}
inline size_t colsplit_lds_bytes(int tc, const SegTab &sg, int nzpml)
{
    return sizeof(double) * (colsplit_staged(tc, sg, nzpml) + (size_t)4 * tc * yb_len(sg.P, sg.hw) +
                             (size_t)3 * tc * sg.nzp);
}

// ---------------------------------------------------------------------------
// The column pass, one lane per (column, segment, field): the three
// independent first derivatives (xi_z, v_z, v_x) run in three lane groups of
// G = roundup(TC*P, 64) <= 128 threads each (blockDim = 3G, so every wave
// holds one field), which splits the window loads, solves, corrections and epilogue
// work of the first half three ways.  Group 0 (xi_z) then does d p/dz and
// the v_z update; group 1 writes the xi_z update and passes its part of RHS
// v_z through LDS; group 2 writes RHS v_x and the xi_x update.  After the
// last stage each group filters one field.  Store/load order across groups:
// xi_z (TN[1]) is written only after the first barrier, when every lane's
// window reads of T[1] are complete (T and TN are one buffer after the first
// stage); v_z (TN[3]) after the third.
// Every table the pass reads comes from LDS, so no lane waits on global
// memory for them once the staging barrier has passed.

// The fields are row-pair arrays, so that every access of a lane moves two rows
// (16 bytes).  With plain rows the pass was bound by the L1's one access per
// clock: at TC = 2 a wave instruction touched 32 lines for 16 bytes each, 21 000
// accesses per block, 9 of its 14 us (one source at 256x300; 21.1 us a launch
// between events, then 17.2, and 16.9 with the source off the first solve's path and
// shared windows of end values; 128x150 17.3 -> 15.8 -> 15.1).
//
// Loads and stores at a 32-bit byte offset from a wave-uniform base address:
// the compiler then uses the SGPR-base + VGPR-offset addressing form, with no
// 64-bit address arithmetic per access.  The host checks that every array
// indexed this way spans less than 2^31 bytes.
#define SPARC_GLOBAL __attribute__((address_space(1)))
__device__ __forceinline__ double ldb(const double *base, unsigned ob)
{
    return *(const SPARC_GLOBAL double *)((const SPARC_GLOBAL char *)base + ob);
}
__device__ __forceinline__ void stb(double *base, unsigned ob, double v)
{
    *(SPARC_GLOBAL double *)((SPARC_GLOBAL char *)base + ob) = v;
}
// Two rows of a column (a row pair, sparc_device.h) at once, 16 bytes.
typedef double dpair __attribute__((ext_vector_type(2)));
__device__ __forceinline__ dpair ldp(const double *base, unsigned ob)
{
    return *(const SPARC_GLOBAL dpair *)((const SPARC_GLOBAL char *)base + ob);
}
__device__ __forceinline__ void stp(double *base, unsigned ob, double v0, double v1)
{
    *(SPARC_GLOBAL dpair *)((SPARC_GLOBAL char *)base + ob) = dpair{v0, v1};
}
// A value every lane of the wave holds, moved to a scalar register.
template <typename T>
__device__ __forceinline__ T *wave_ptr(T *p)
{
    const unsigned long long u = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    return (T *)(((unsigned long long)hi << 32) | lo);
}

template <int MS, int LAST>
__global__ __launch_bounds__(384) void k_colsplit(Dims d, Bg bg, DbyCoef cf, SegTab sg, State st,
                                                  ColArgs ca, Src src, Clock clk, Sink sink, int TC)
{
    static_assert(MS % 2 == 0, "segments are whole row pairs");
    extern __shared__ double lds_dyn[];
    const int P = sg.P, n2P = 2 * P, nzp = sg.nzp;
    const int nrow = 2 * (4 * sg.hw + 4), nband = sg.nk * nrow;
    const int nzpml = d.nzpml;
    double *const mv = lds_dyn;                        // [3][nk][nrow] interface rows
    double *const zl = mv + 3 * nband;                 // [kZS][3][MS] segment tables
    double *const zf = zl + kZS * 3 * MS;              // [kZF][nzp] z profiles
    double *const cbl = zf + kZF * nzp;                // [kCB] dbyd2 boundary-row coefficients
    double *const pl = cbl + kCB;                      // [kPL][nzpml][TC] z-PML data
    double *const zpl = pl + kPL * nzpml * TC;         // [nzp] mode-3 source z profile
    const int nstaged = (3 * nband + kZS * 3 * MS + kZF * nzp + kCB + kPL * nzpml * TC + nzp + 1) & ~1;
    const int LY = n2P + 4 * sg.hw + 2, hw2 = 2 * sg.hw;
    double *const yb0 = lds_dyn + nstaged;             // [4][TC][LY] end values: field groups 0-2, d p/dz
    double *const wl = yb0 + 4 * TC * LY;              // [TC][nzp] group 1's part of RHS v_z,
                                                       // then [TC][nzp] group 0's part, [TC][nzp] p
    const int tid = threadIdx.x, G = blockDim.x / 3;
    const int f = __builtin_amdgcn_readfirstlane(tid / G);   // the field group: one per wave
    // end-value buffers by offset from the LDS base (an array of pointers
    // indexed by f would turn these accesses into flat ones)
    double *const ybf = yb0 + f * TC * LY, *const yb3 = yb0 + 3 * TC * LY;
    const int l = tid - f * G;
    const int c = l % TC, s = l / TC;
    const bool act = s < P;
    const int sc = act ? s : 0;
    const int a = sc * MS;
    const bool first = act && s == 0;
    const bool lastseg = a + MS > d.nz - 2;            // holds rows nz-2 and nz-1
    int bx = blockIdx.x, by = blockIdx.y;
    {
        const int lg = (int)xcd_block(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
        bx = lg % gridDim.x;
        by = lg / gridDim.x;
    }
    const int x = bx * TC + c, b = by;
    const int nx = d.nx, nz = d.nz;
    const int nxb = nx * 8;                            // bytes per row of a plain array
    // byte offset of (b, row pair 0, x) in a row-pair array of S sources, and of
    // one source; bytes per row pair; the last pair
    const int colb = (b * d.nzq * nx + 2 * x) * 8, gcolb = 16 * x, pairb = 16 * nx, lastp = d.nzq / 2 - 1;
    const int time = clock_t_(clk);
    const int nb = d.npmlbot, ntop = d.npmltop;
    const int pz0b = (b * nzpml * nx + x) * 8;
    const int pz1b = ((d.S + b) * nzpml * nx + x) * 8;
    const double *zs = zf + a;                         // row a of the staged z profiles
    // this segment's tables: those of the first, an interior or the last
    // segment (every interior segment's are the same), row r at zt[r * 3 MS + i]
    const double *zt = zl + seg_kind(sc, P) * MS;
    auto plv = [&](int k, int pj) -> double { return pl[(k * nzpml + pj) * TC + c]; };

    // byte offset of row pair h of this column, h clamped to the column
    auto pairo = [&](int h) -> unsigned { return (unsigned)(min(max(h, 0), lastp) * pairb); };
    const int h0 = a >> 1;                             // the segment's first pair (a is even)
    // rows i, i + 1 of this segment (i even) to a row-pair array; past the
    // column's end nothing, and 0 in the pad row of an odd nz
    auto put2 = [&](double *base, int i, double v0, double v1) {
        if (act && a + i < nz) stp(base, colb + (unsigned)((h0 + (i >> 1)) * pairb), v0, a + i + 1 < nz ? v1 : 0.0);
    };
    auto valid = [&](int i) -> bool { return act && a + i < nz; };
    auto pmlrow = [&](int j) -> int {
        const int jc = min(j, nz - 1);
        return jc < nb ? jc : min(nzpml - 1, nb + max(jc - (nz - ntop), 0));
    };
    auto is_pml = [&](int j) -> bool { return j < nb || (j >= nz - ntop && j < nz); };
    // The epilogues take their z-PML form for the whole wave when any lane's
    // segment meets a PML layer: that form leaves rows outside the layers as
    // the plain form does (the PML terms are selected off and the auxiliary
    // stores masked), and a per-lane choice would run both forms one after
    // the other in every wave that holds a layer.
    const bool segpml = __ballot(a < nb || a + MS > nz - ntop) != 0;

    // --- first derivatives: group 0 d xi_z/dz (ibc 3, top row preset),
    //     group 1 d v_z/dz (ibc 1), group 2 d v_x/dz (ibc 1)
    const double *F = wave_ptr(f == 0 ? ca.T[1] : (f == 1 ? ca.T[3] : ca.T[2]));
    double win[MS + 8];                                // rows a - 4 .. a + MS + 3
#pragma unroll
    for (int k = 0; k < MS + 8; k += 2) {
        const dpair v = ldp(F, colb + pairo(h0 - 2 + (k >> 1)));
        win[k] = v.x;
        win[k + 1] = v.y;
    }
    const double topv = f == 0 ? ldb(st.topbc, (b * nx + x) * 8) : 0.0;
    double e[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (lastseg) {
#pragma unroll
        for (int k = 0; k < 5; k++) {
            const int r = nz - 5 + k;
            e[k] = ldb(F, colb + (unsigned)((r >> 1) * pairb + (r & 1) * 8));
        }
    }
    // the first epilogue's inputs, which no lane of this kernel writes before
    // the barrier after the first solve: group 0 d xi_x/dx, c^2 rho0 and the v_z
    // base; groups 1, 2 the x-derivative, the base of their update and the flow
    double pa[MS], pb[MS], pc[MS], pd[MS];
    {
        const double *const A = wave_ptr(f == 0 ? (const double *)st.dxixdx : (f == 1 ? st.dxvz : st.dxvx));
        const double *const Cf = wave_ptr(f == 0 ? bg.c2rho0_p : bg.v0x_p);
        const double *const B0 = wave_ptr((const double *)st.a[f == 0 ? 3 : (f == 1 ? 1 : 0)]);
#pragma unroll
        for (int i = 0; i < MS; i += 2) {
            const unsigned r = pairo(h0 + (i >> 1));
            const dpair va = ldp(A, colb + r), vb = ldp(Cf, gcolb + r), vc = ldp(B0, colb + r);
            dpair vd = {0.0, 0.0};
            if (f != 0) vd = ldp(bg.v0z_p, gcolb + r);
            pa[i] = va.x; pa[i + 1] = va.y;
            pb[i] = vb.x; pb[i + 1] = vb.y;
            pc[i] = vc.x; pc[i + 1] = vc.y;
            pd[i] = vd.x; pd[i + 1] = vd.y;
        }
    }
    {
        // zero the pads of the end-value buffers
        const int npad = 4 * TC, padw = LY - n2P;
        for (int q = tid; q < npad * padw; q += blockDim.x) {
            const int r = q / padw, u = q - r * padw;
            yb0[r * LY + (u < hw2 ? u : n2P + u)] = 0.0;
        }
    }
    {
        // the staged region in one pass for the usual shapes: the interface rows
        // and z tables are one contiguous copy of sg.stage (kStage loads per
        // thread), the z-PML data come from their own arrays (two elements per
        // thread and kind); every load of a round is issued before its stores
        constexpr int kStage = 12;
        const int nA = 3 * nband + kZS * 3 * MS + kZF * nzp + kCB, npl = nzpml * TC, stride = blockDim.x;
        const int x0 = bx * TC;
        const int rounds = max((nA + kStage * stride - 1) / (kStage * stride),
                               (max(npl, nzp) + 2 * stride - 1) / (2 * stride));
        const bool zsrc = src.mode == 3;
        const double *const stg = wave_ptr(sg.stage);
        for (int r0 = 0; r0 < rounds; r0++) {
            double va[kStage], vb[kPL][2], vz[2] = {0.0, 0.0};
            const int qa0 = r0 * kStage * stride + tid, qb0 = r0 * 2 * stride + tid;
#pragma unroll
            for (int u = 0; u < kStage; u++) va[u] = ldb(stg, (unsigned)min(qa0 + u * stride, nA - 1) * 8u);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int q = min(qb0 + h * stride, npl - 1);
                const int pj = q / TC, xc = x0 + (q - pj * TC);
                const unsigned gq = (unsigned)(pj * nx + xc) * 8u;
                const unsigned s0 = (unsigned)((b * nzpml + pj) * nx + xc) * 8u;
                const unsigned s1 = (unsigned)(((d.S + b) * nzpml + pj) * nx + xc) * 8u;
                vb[P_AZ][h] = ldb(bg.az, gq);
                vb[P_BZ][h] = ldb(bg.bz, gq);
                vb[P_FZ][h] = ldb(bg.fz, gq);
                vb[P_T0][h] = ldb(st.pz_tmp, s0);
                vb[P_B0][h] = ldb(st.pz_base, s0);
                vb[P_T1][h] = ldb(st.pz_tmp, s1);
                vb[P_B1][h] = ldb(st.pz_base, s1);
            }
            if (zsrc) {
#pragma unroll
                for (int h = 0; h < 2; h++) vz[h] = ldb(src.zprof, (unsigned)min(qb0 + h * stride, nz - 1) * 8u);
            }
#pragma unroll
            for (int u = 0; u < kStage; u++)
                if (qa0 + u * stride < nA) lds_dyn[qa0 + u * stride] = va[u];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int q = qb0 + h * stride;
                if (q < npl) {
#pragma unroll
                    for (int k = 0; k < kPL; k++) pl[k * npl + q] = vb[k][h];
                }
                if (zsrc && q < nzp) zpl[q] = q < nz ? vz[h] : 0.0;
            }
        }
    }
    __syncthreads();
    const int slot_f = f == 0 ? 2 : 0;                 // dbyd2 table set: ibc 3 or ibc 1
    double Y[MS], own[MS];
    const double *const cbt = cbl;                      // LDS: read only by the end segments' lanes
    seg_rhs<MS>([&](int k) { return win[k + 1]; }, e, Y, a, nz, first, lastseg, f == 0 ? 3 : 1, 0.0, topv, cf.c1,
                cf.c2, cbt);
#pragma unroll
    for (int i = 0; i < MS; i++) own[i] = win[4 + i];
    const double *const zt_f = zt + 5 * slot_f * 3 * MS;   // this group's table set
    auto gtab = [&](int t, int i) { return zt_f[t * 3 * MS + i]; };
    seg_solve<MS>(Y, gtab);
    if (act) { ybf[c * LY + hw2 + 2 * s] = Y[0]; ybf[c * LY + hw2 + 2 * s + 1] = Y[MS - 1]; }
    __syncthreads();
    const double *const mvs = mv + seg_band_kind(sc, P, sg.E) * nrow;   // this segment's rows of set 0
    if (act)
        seg_correct_rows<MS>(Y, s, P, sg.hw, ybf + c * LY, mvs + (f == 0 ? 2 * nband : 0), gtab);

    double *const w0 = wl + (TC + c) * nzp + a;       // group 0: -rho'/rho0 g
    double *const pcol = wl + (2 * TC + c) * nzp;     // p of this column (group 0)
    if (f == 0) {
        // z-PML (:957-967), divergence, p and rho' (:990-998, :1043)
        // (its LDS writes after all its LDS reads: the compiler cannot tell
        // them apart, and in source order every row would wait for the last)
        double pv[MS], bv[MS];
        auto epi = [&](auto pml_c) {
            constexpr bool PML = decltype(pml_c)::value;
#pragma unroll
            for (int i = 0; i < MS; i++) {
                double lpsi = 0.0, laz = 0.0, lbz = 0.0, lpb = 0.0, lfz = 0.0;
                if (PML) {
                    const int pj = pmlrow(a + i);
                    lpsi = plv(P_T0, pj);
                    lpb = plv(P_B0, pj);
                    laz = plv(P_AZ, pj);
                    lbz = plv(P_BZ, pj);
                    lfz = plv(P_FZ, pj);
                }
                const int j = a + i;
                const double str = zs[F_STR * nzp + i], r0 = zs[F_RHO * nzp + i];
                const double rinv = zs[F_RINV * nzp + i], gz = zs[F_G * nzp + i];
                double dz = Y[i] * str;
                double fdec = 1.0;
                if (PML) {
                    const bool pm = is_pml(j);
                    fdec = pm ? lfz : 1.0;
                    const double prhs = laz * dz + lbz * lpsi;
                    dz = pm ? dz + lpsi : dz;
                    const double pnew = lpb + ca.bnext * prhs;
                    if (pm && act) {
                        const unsigned qp = pz0b + pmlrow(j) * nxb;
                        stb(st.pz_tmp, qp, pnew);
                        if (LAST) stb(st.pz_base, qp, pnew);
                    }
                }
                const double gp0 = zs[F_GP * nzp + i] * fdec, gr0 = zs[F_GRHO * nzp + i] * fdec;
                const double xiz = own[i];
                const double div = pa[i] + dz;
                pv[i] = -(pb[i] * div) - gp0 * xiz;
                const double rho = -(r0 * div) - gr0 * xiz;
                bv[i] = -rinv * (rho * gz);
                // one row after the other: with all rows' table reads in flight the 10-row
                // form spilled
                asm volatile("" : "+v"(bv[i]), "+v"(pv[i]) :: "memory");
            }
        };
        if (segpml) epi(std::true_type{});
        else epi(std::false_type{});
#pragma unroll
        for (int i = 0; i < MS; i += 2) put2(st.p, i, pv[i], pv[i + 1]);
        if (act) {
#pragma unroll
            for (int i = 0; i < MS; i++) {
                if (a + i < nz) pcol[a + i] = pv[i];
                w0[i] = bv[i];
            }
        }
    } else {
        // group 1: source and flow part of RHS v_z (:1051-1061, :1073-1077) to LDS,
        // xi_z update; group 2: RHS v_x flow part (:1067-1071), xi_x update.  The
        // source's loads and the adjoint's interpolation (seven divisions) stand here
        // because group 0's epilogue takes 1.2 us longer than this one (before the
        // first solve every wave of the block waited for them), and after the updates
        // because their operands then need no registers any more.
        double r1[MS], r2[MS];                         // the xi update; group 1 its part of RHS v_z, group 2 RHS v_x
#pragma unroll
        for (int i = 0; i < MS; i++) {
            const int j = a + i;
            const bool zero = j == 0 || x == 0 || x == nx - 1;
            const double rv = -(2.0 * pb[i] * pa[i]) - 2.0 * pd[i] * (Y[i] * zs[F_STR * nzp + i]);
            r2[i] = f == 2 && zero ? 0.0 : rv;
            r1[i] = pc[i] + ca.bnext * (zero ? 0.0 : own[i]);
        }
        double *const X = wave_ptr(ca.TN[f == 1 ? 1 : 0]);
#pragma unroll
        for (int i = 0; i < MS; i += 2) {
            put2(X, i, r1[i], r1[i + 1]);
            if (f == 2) put2(st.rvx, i, r2[i], r2[i + 1]);
        }
        double srcv = 0.0, pamp = 0.0;
        const int isrc = src.row - a;
        if (f == 1 && act && time <= src.limit) {
            if (src.mode == 3) {
                pamp = profile_amp(src, b, x, nx, a, MS, time);
            } else if (isrc >= 0 && isrc < MS) {
                if (src.mode == 1) {
                    // the loads issued before any is used (clamped time index)
                    double fsr = src.fwd[min(max(time, 0), max(src.nfwd - 1, 0))];
                    double vrx = src.vr[b * nx + x], r0 = ldb(bg.rho0_src, x * 8);
                    asm volatile("" : "+v"(fsr), "+v"(vrx), "+v"(r0));
                    const double fs = (time >= 0 && time < src.nfwd) ? fsr : 0.0;
                    srcv = vrx * fs * src.delta_width / r0;
                } else if (src.mode == 2) {
                    srcv = lagrange_forcing(src, b, x, nx, time) * src.delta_width / ldb(bg.rho0_src, x * 8);
                }
            }
        }
        if (f == 1 && act) {
#pragma unroll
            for (int i = 0; i < MS; i++) {
                if (src.mode == 3) r2[i] = r2[i] + pamp * zpl[a + i];
                wl[c * nzp + a + i] = (i == isrc) ? r2[i] + srcv : r2[i];
            }
        }
    }

    // --- d p/dz (ibc 2, :1023) with the z-PML (:1025-1035), RHS v_z, the
    //     zeroed rows/columns (:1083-1093) and the v_z update: group 0
    __syncthreads();
    if (f == 0) {
        double wp[MS + 6];
#pragma unroll
        for (int k = 0; k < MS + 6; k++) wp[k] = pcol[min(max(a - 3 + k, 0), nz - 1)];
        double ep[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (lastseg) {
#pragma unroll
            for (int k = 0; k < 5; k++) ep[k] = pcol[nz - 5 + k];
        }
        seg_rhs<MS>([&](int k) { return wp[k]; }, ep, Y, a, nz, first, lastseg, 2, 0.0, 0.0, cf.c1, cf.c2, cbt);
        auto ltab = [&](int t, int i) { return zt[(5 + t) * 3 * MS + i]; };   // ibc 2 set
        seg_solve<MS>(Y, ltab);
        if (act) { yb3[c * LY + hw2 + 2 * s] = Y[0]; yb3[c * LY + hw2 + 2 * s + 1] = Y[MS - 1]; }
    }
    __syncthreads();
    if (f == 0) {
        auto ltab = [&](int t, int i) { return zt[(5 + t) * 3 * MS + i]; };   // ibc 2 set
        if (act) seg_correct_rows<MS>(Y, s, P, sg.hw, yb3 + c * LY, mvs + nband, ltab);
        const int sslot = (LAST && sink.snap) ? out_slot(time, clk.steps, sink.k0, sink.nsnap) : -1;
        const bool snap = sslot >= 0;
        const size_t slot = snap ? ((size_t)b * sink.nsnap + sslot) * sink.nfield : 0;
        auto epi = [&](auto pml_c) {
            constexpr bool PML = decltype(pml_c)::value;
#pragma unroll
            for (int i = 0; i < MS; i++) {
                double lpsi = 0.0, laz = 0.0, lbz = 0.0, lpb = 0.0;
                if (PML) {
                    const int pj = pmlrow(a + i);
                    lpsi = plv(P_T1, pj);
                    lpb = plv(P_B1, pj);
                    laz = plv(P_AZ, pj);
                    lbz = plv(P_BZ, pj);
                }
                const int j = a + i;
                double gpz = Y[i] * zs[F_STR * nzp + i];
                if (PML) {
                    const bool pm = is_pml(j);
                    const double prhs = laz * gpz + lbz * lpsi;
                    gpz = pm ? gpz + lpsi : gpz;
                    const double pnew = lpb + ca.bnext * prhs;
                    if (pm && act) {
                        const unsigned qp = pz1b + pmlrow(j) * nxb;
                        stb(st.pz_tmp, qp, pnew);
                        if (LAST) stb(st.pz_base, qp, pnew);
                    }
                }
                double rvz = -zs[F_RINV * nzp + i] * gpz + (w0[i] + wl[c * nzp + a + i]);
                rvz = (j == 0 || x == 0 || x == nx - 1) ? 0.0 : rvz;
                pa[i] = pc[i] + ca.bnext * rvz;
                if (snap && valid(i)) sink.snap[((slot + (sink.adjoint ? 3 : 5)) * nz + j) * nx + x] = rvz;
            }
#pragma unroll
            for (int i = 0; i < MS; i += 2) put2(ca.TN[3], i, pa[i], pa[i + 1]);
        };
        if (segpml) epi(std::true_type{});
        else epi(std::false_type{});
    }
    if (LAST) {
        // FILTER_VARS_2D (physics2d.f90:509-556): group 0 filters v_z, group 1
        // xi_z, group 2 xi_x, each from a window of rows a-5 .. a+MS+4
        __syncthreads();
        const int fi = f == 0 ? 3 : (f == 1 ? 1 : 0);
        const int sslot = sink.snap ? out_slot(time, clk.steps, sink.k0, sink.nsnap) : -1;
        const bool snap = sslot >= 0;
        const size_t slot = snap ? ((size_t)b * sink.nsnap + sslot) * sink.nfield : 0;
        const int oslot = sink.vz_out ? out_slot(time, clk.steps, sink.k0, sink.nout) : -1;
        const bool out = oslot >= 0;
        const int nh = d.nh;
        const bool xin = x >= nh - 1 && x <= nx - nh;
        const double *Fw = wave_ptr((const double *)ca.TN[fi]);
        double *const Aw = wave_ptr(st.a[fi]);
        double w[MS + 12];                             // rows a - 6 .. a + MS + 5
#pragma unroll
        for (int q = 0; q < MS + 12; q += 2) {
            const dpair v = ldp(Fw, colb + pairo(h0 - 3 + (q >> 1)));
            w[q] = v.x;
            w[q + 1] = v.y;
        }
        double fv[MS];
        // snapshot field: forward xi_x 0, xi_z 1, v_z 3; adjoint v_z 1
        const int fs = sink.adjoint ? (fi == 3 ? 1 : -1) : fi;
#pragma unroll
        for (int i = 0; i < MS; i++) {
            const int j = a + i;
            const int q = i + 6;
            const double f11 = 0.75390625 * w[q] + 0.5 * 0.41015625 * (w[q - 1] + w[q + 1]) +
                               0.5 * -0.234375 * (w[q - 2] + w[q + 2]) +
                               0.5 * 0.087890625 * (w[q - 3] + w[q + 3]) +
                               0.5 * -0.01953125 * (w[q - 4] + w[q + 4]) +
                               0.5 * 0.001953125 * (w[q - 5] + w[q + 5]);
            const double f2 = 0.5 * (w[q + 1] + w[q - 1]);
            double v = w[q];
            if (xin && j >= 5 && j <= nz - 2) v = (j <= nz - 6) ? f11 : f2;
            fv[i] = v;
            if (valid(i)) {
                if (fi == 3 && out && j == sink.orow)
                    sink.vz_out[((size_t)b * sink.nout + oslot) * nx + x] = v;
                if (snap && fs >= 0) sink.snap[(slot + fs) * nz * nx + (size_t)j * nx + x] = v;
            }
        }
#pragma unroll
        for (int i = 0; i < MS; i += 2) put2(Aw, i, fv[i], fv[i + 1]);
    }
}

// ---------------------------------------------------------------------------
// The column pass of a batch, one lane per (column, segment) for all fields: the
// three first derivatives one after the other, then the epilogue of a row pair
// at a time (the next pair's nine inputs in flight meanwhile), d p/dz and the v_z
// update.  Against the lane groups above it reads the flow once, stages the
// tables for twice the columns per block or more and holds seven or eight waves per
// compute unit where those hold six; but a lane's chain is twice as long, so it wants
// enough columns to fill the chip twice.  Bound: registers (244 at MS = 6, two
// waves per SIMD; MS = 8 spills a little, longer segments more than they gain)
// and HBM, 128 B per point.  us per launch, lane groups -> here: 16 sources at
// 256x300 67 -> 51, 8 sources 37 -> 29, 6 sources 36 -> 27; 4 sources (307 000
// points) 21 -> 24, 16 at 128x150 (307 000) 20 -> 23: the line between the forms
// lies at 450 000 points.  With shared windows of end values 16 sources take 47
// (3.3 TB/s) and 8 take 27, the lane groups' 16 at 128x150 19.
//
// It also wants many blocks on a compute unit: a lane group's wave does about a third of
// a one-lane wave's work, so where the tables' LDS, and not the registers, bounds the
// blocks of a unit, the lane groups have three times the waves.  The form runs where a
// unit holds at least three of its blocks for one of the lane groups', and above 128
// lanes, where the lane groups do not fit.  us per launch at the best shape of each form,
// lane groups / one lane: 64 sources of 100x100 47 / 63, 16 of 250x150 52 / 67, 8 of
// 255x300 64 / 89, 100 of 256x60 74 / 78, 400 of 300x60 551 / 604; 8 of 1000x100 52 / 45,
// 60 of 150x60 86 / 68, 1000 of 17x40 214 / 160, 16 of 256x300 70 / 50.  Over 48 grids the
// best shape under this rule is 0.1 % (at most 1.9 %) behind the best of both forms; lines
// at 2 or 4 in place of 3 cost up to 10 % and 26 %.
constexpr size_t kOneLanePoints = 450000;
constexpr int kOneLaneBlocks = 3;
constexpr int kWavesPerUnit = 8;   // both forms: two waves per SIMD by registers
constexpr int kCA = 9;      // epilogue inputs of a row pair
struct PairIn {
    dpair v[kCA];           // d xi_x/dx, c^2 rho0, d v_z/dx, d v_x/dx, v0x, v0z, xi_z base, xi_z, v_z
};

template <int MS, int LAST>
__global__ __launch_bounds__(512) void k_colone(Dims d, Bg bg, DbyCoef cf, SegTab sg, State st, ColArgs ca, Src src,
                                                Clock clk, Sink sink, int TC)
{
    static_assert(MS % 2 == 0, "segments are whole row pairs");
    extern __shared__ __align__(16) double lds1[];
    const int P = sg.P, nzp = sg.nzp, hw2 = 2 * sg.hw, LY = 2 * P + 4 * sg.hw + 2;
    const int nrow = 2 * (4 * sg.hw + 4), nband = sg.nk * nrow;
    const int nimg = (3 * nband + kZS * 3 * MS + kZF * nzp + kCB + 1) & ~1;
    double *const zl = lds1 + 3 * nband, *const zf = zl + kZS * 3 * MS, *const cbl = zf + kZF * nzp;
    double *const yb = lds1 + nimg;                    // [4][TC][LY] end values: xi_z, v_z, v_x, p
    double *const pl = yb + 4 * TC * LY;               // [TC][nzp] p
    const int tid = threadIdx.x, nthr = blockDim.x, nx = d.nx, nz = d.nz;
    const int lg = (int)xcd_block(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int b = lg / gridDim.x, x = (lg - b * gridDim.x) * TC + tid % TC;
    const int c = tid % TC, s0 = tid / TC, s = min(s0, P - 1), a = s * MS, h0 = a >> 1;
    const bool act = s0 < P, first = s == 0, lastseg = a + MS > nz - 2;
    const int nb = d.npmlbot, ntop = d.npmltop, nzpml = d.nzpml, lastp = d.nzq / 2 - 1, pairb = 16 * nx;
    const unsigned colb = (unsigned)(b * d.nzq * nx + 2 * x) * 8u, gcolb = 16u * x;
    auto pairo = [&](int h) -> unsigned { return (unsigned)(min(max(h, 0), lastp) * pairb); };
    auto put2 = [&](double *base, int i, double v0, double v1) {
        if (act && a + i < nz) stp(base, colb + (unsigned)((h0 + (i >> 1)) * pairb), v0, a + i + 1 < nz ? v1 : 0.0);
    };
    auto pmlrow = [&](int j) -> int {                  // PML row of grid row j, -1 outside the layers
        return j < nb ? j : (j >= nz - ntop && j < nz ? nb + j - (nz - ntop) : -1);
    };
    const int time = clock_t_(clk);

    // source value of this column at its injection row (physics2d.f90:1051-1061)
    double srcv = 0.0;
    const int isrc = src.row - a;
    if (act && isrc >= 0 && isrc < MS && time <= src.limit) {
        if (src.mode == 1) {
            double fsr = src.fwd[min(max(time, 0), max(src.nfwd - 1, 0))];
            double vrx = src.vr[b * nx + x];
            asm volatile("" : "+v"(fsr), "+v"(vrx));
            const double fs = (time >= 0 && time < src.nfwd) ? fsr : 0.0;
            srcv = vrx * fs * src.delta_width / ldb(bg.rho0_src, x * 8u);
        } else if (src.mode == 2) {
            srcv = lagrange_forcing(src, b, x, nx, time) * src.delta_width / ldb(bg.rho0_src, x * 8u);
        }
    }
    const double pamp = act ? profile_amp(src, b, x, nx, a, MS, time) : 0.0;
    // --- the first derivatives: d xi_z/dz (ibc 3, top row preset), d v_z/dz,
    //     d v_x/dz (ibc 1)
    double W0[MS + 8], e0[5];
    auto window = [&](const double *F, double (&w)[MS + 8], double (&ee)[5]) {
#pragma unroll
        for (int k = 0; k < MS + 8; k += 2) {
            const dpair v = ldp(F, colb + pairo(h0 - 2 + (k >> 1)));
            w[k] = v.x;
            w[k + 1] = v.y;
        }
#pragma unroll
        for (int k = 0; k < 5; k++) ee[k] = 0.0;
        if (lastseg) {
#pragma unroll
            for (int k = 0; k < 5; k++) {
                const int r = nz - 5 + k;
                ee[k] = ldb(F, colb + (unsigned)((r >> 1) * pairb + (r & 1) * 8));
            }
        }
    };
    window(ca.T[1], W0, e0);
    const double topv = ldb(st.topbc, (unsigned)(b * nx + x) * 8u);
    for (int q = tid; q < 4 * TC * LY; q += nthr) yb[q] = 0.0;
    {
        const double2 *const im = (const double2 *)sg.stage;
        double2 *const dst = (double2 *)lds1;
        const int n2 = nimg >> 1;
        for (int q = tid; q < n2; q += 8 * nthr) {
            double2 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = im[min(q + u * nthr, n2 - 1)];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (q + u * nthr < n2) dst[q + u * nthr] = v[u];
        }
    }
    __syncthreads();
    const double *const zt = zl + seg_kind(s, P) * MS;
    auto tab = [&](int set) { return [zt, set](int t, int i) { return zt[(5 * set + t) * 3 * MS + i]; }; };
    const double *const mvs = lds1 + seg_band_kind(s, P, sg.E) * nrow;
    double *const yc = yb + c * LY;
    double Y0[MS], Y1[MS], Y2[MS];
    auto ends = [&](int f, const double (&Y)[MS]) {
        if (act) {
            yc[f * TC * LY + hw2 + 2 * s] = Y[0];
            yc[f * TC * LY + hw2 + 2 * s + 1] = Y[MS - 1];
        }
    };
    seg_rhs<MS>([&](int k) { return W0[k + 1]; }, e0, Y0, a, nz, first, lastseg, 3, 0.0, topv, cf.c1, cf.c2, cbl);
    window(ca.T[3], W0, e0);
    seg_solve<MS>(Y0, tab(2));
    ends(0, Y0);
    seg_rhs<MS>([&](int k) { return W0[k + 1]; }, e0, Y1, a, nz, first, lastseg, 1, 0.0, 0.0, cf.c1, cf.c2, cbl);
    window(ca.T[2], W0, e0);
    seg_solve<MS>(Y1, tab(0));
    ends(1, Y1);
    seg_rhs<MS>([&](int k) { return W0[k + 1]; }, e0, Y2, a, nz, first, lastseg, 1, 0.0, 0.0, cf.c1, cf.c2, cbl);
    // xi_x update: its T is read by no lane, so it need not wait
#pragma unroll
    for (int i = 0; i < MS; i += 2) {
        const dpair bx = ldp(st.a[0], colb + pairo(h0 + (i >> 1)));
        const bool zx = x == 0 || x == nx - 1;
        put2(ca.TN[0], i, bx.x + ca.bnext * (zx || a + i == 0 ? 0.0 : W0[4 + i]),
             bx.y + ca.bnext * (zx ? 0.0 : W0[5 + i]));
    }
    seg_solve<MS>(Y2, tab(0));
    ends(2, Y2);
    auto load_pair = [&](int i, PairIn &q) {
        const unsigned r = pairo(h0 + (i >> 1));
        q.v[0] = ldp(st.dxixdx, colb + r);
        q.v[1] = ldp(bg.c2rho0_p, gcolb + r);
        q.v[2] = ldp(st.dxvz, colb + r);
        q.v[3] = ldp(st.dxvx, colb + r);
        q.v[4] = ldp(bg.v0x_p, gcolb + r);
        q.v[5] = ldp(bg.v0z_p, gcolb + r);
        q.v[6] = ldp(st.a[1], colb + r);
        q.v[7] = ldp(ca.T[1], colb + r);
        q.v[8] = ldp(ca.T[3], colb + r);
    };
    PairIn in[2];
    load_pair(0, in[0]);
    __syncthreads();
    seg_correct_rows<MS, 1>(Y0, s, P, sg.hw, yc, mvs + 2 * nband, tab(2));
    seg_correct_rows<MS, 1>(Y1, s, P, sg.hw, yc + TC * LY, mvs, tab(0));
    seg_correct_rows<MS, 1>(Y2, s, P, sg.hw, yc + 2 * TC * LY, mvs, tab(0));
    // --- z-PML (:957-967), divergence, p and rho' (:990-998, :1043), the flow
    //     terms (:1067-1077), xi_z; w: RHS v_z but the pressure gradient
    const double *const zs = zf + a;
    double w[MS];
#pragma unroll
    for (int i = 0; i < MS; i += 2) {
        const PairIn &q = in[(i >> 1) & 1];
        if (i + 2 < MS) load_pair(i + 2, in[((i >> 1) + 1) & 1]);
        double pv[2], xz[2], rx[2];
        // z-PML data of d xi_z/dz; a row outside the layers takes its neighbour's
        // and drops it
        dpair az = {0.0, 0.0}, bz = {0.0, 0.0}, fz = {1.0, 1.0}, ps = {0.0, 0.0}, pb = {0.0, 0.0};
        const int p0 = pmlrow(a + i), p1 = pmlrow(a + i + 1);
        if (p0 >= 0 || p1 >= 0) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int pj = u ? (p1 >= 0 ? p1 : p0) : (p0 >= 0 ? p0 : p1);
                const unsigned g = (pj * nx + x) * 8u, f = ((b * nzpml + pj) * nx + x) * 8u;
                az[u] = ldb(bg.az, g);
                bz[u] = ldb(bg.bz, g);
                fz[u] = ldb(bg.fz, g);
                ps[u] = ldb(st.pz_tmp, f);
                pb[u] = ldb(st.pz_base, f);
            }
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int j = a + i + u, pj = pmlrow(j);
            const double str = zs[F_STR * nzp + i + u], rinv = zs[F_RINV * nzp + i + u];
            const bool zero = j == 0 || x == 0 || x == nx - 1;
            double dz = Y0[i + u] * str;
            double fdec = 1.0;
            if (pj >= 0) {
                fdec = fz[u];
                const double prhs = az[u] * dz + bz[u] * ps[u];
                dz = dz + ps[u];
                if (act) {
                    const unsigned qp = ((b * nzpml + pj) * nx + x) * 8u;
                    const double pnew = pb[u] + ca.bnext * prhs;
                    stb(st.pz_tmp, qp, pnew);
                    if (LAST) stb(st.pz_base, qp, pnew);
                }
            }
            const double gp0 = zs[F_GP * nzp + i + u] * fdec, gr0 = zs[F_GRHO * nzp + i + u] * fdec;
            const double div = q.v[0][u] + dz;
            pv[u] = -(q.v[1][u] * div) - gp0 * q.v[7][u];
            const double rho = -(zs[F_RHO * nzp + i + u] * div) - gr0 * q.v[7][u];
            double bzv = -rinv * (rho * zs[F_G * nzp + i + u]);
            if (src.mode == 3 && j < nz) bzv = bzv + pamp * src.zprof[j];
            bzv = i + u == isrc ? bzv + srcv : bzv;
            const double flow = -(2.0 * q.v[4][u] * q.v[2][u]) - 2.0 * q.v[5][u] * (Y1[i + u] * str);
            w[i + u] = bzv + flow;
            rx[u] = zero ? 0.0 : -(2.0 * q.v[4][u] * q.v[3][u]) - 2.0 * q.v[5][u] * (Y2[i + u] * str);
            xz[u] = q.v[6][u] + ca.bnext * (zero ? 0.0 : q.v[8][u]);
            if (act && j < nz) pl[c * nzp + j] = pv[u];
        }
        put2(st.p, i, pv[0], pv[1]);
        put2(st.rvx, i, rx[0], rx[1]);
        put2(ca.TN[1], i, xz[0], xz[1]);
    }
    __syncthreads();
    // --- d p/dz (ibc 2, :1023) with the z-PML (:1025-1035), RHS v_z, the zeroed
    //     rows/columns (:1083-1093) and the v_z update
    dpair bv[MS / 2];
#pragma unroll
    for (int i = 0; i < MS; i += 2) bv[i >> 1] = ldp(st.a[3], colb + pairo(h0 + (i >> 1)));
    {
        const double *const pcol = pl + c * nzp;
#pragma unroll
        for (int k = 0; k < MS + 6; k++) W0[k] = pcol[min(max(a - 3 + k, 0), nz - 1)];
#pragma unroll
        for (int k = 0; k < 5; k++) e0[k] = lastseg ? pcol[nz - 5 + k] : 0.0;
        seg_rhs<MS>([&](int k) { return W0[k]; }, e0, Y0, a, nz, first, lastseg, 2, 0.0, 0.0, cf.c1, cf.c2, cbl);
    }
    seg_solve<MS>(Y0, tab(1));
    ends(3, Y0);
    __syncthreads();
    seg_correct_rows<MS, 1>(Y0, s, P, sg.hw, yc + 3 * TC * LY, mvs + nband, tab(1));
    const int sslot = (LAST && sink.snap) ? out_slot(time, clk.steps, sink.k0, sink.nsnap) : -1;
    const bool snap = sslot >= 0;
    const size_t slot = snap ? ((size_t)b * sink.nsnap + sslot) * sink.nfield : 0;
#pragma unroll
    for (int i = 0; i < MS; i += 2) {
        double vn[2];
        const int p0 = pmlrow(a + i), p1 = pmlrow(a + i + 1);
        double az[2] = {0.0, 0.0}, bz[2] = {0.0, 0.0}, ps[2] = {0.0, 0.0}, pb[2] = {0.0, 0.0};
        if (p0 >= 0 || p1 >= 0) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int pj = u ? (p1 >= 0 ? p1 : p0) : (p0 >= 0 ? p0 : p1);
                const unsigned g = (pj * nx + x) * 8u, f = (((d.S + b) * nzpml + pj) * nx + x) * 8u;
                az[u] = ldb(bg.az, g);
                bz[u] = ldb(bg.bz, g);
                ps[u] = ldb(st.pz_tmp, f);
                pb[u] = ldb(st.pz_base, f);
            }
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int j = a + i + u, pj = u ? p1 : p0;
            double gpz = Y0[i + u] * zs[F_STR * nzp + i + u];
            if (pj >= 0) {
                const double prhs = az[u] * gpz + bz[u] * ps[u];
                gpz = gpz + ps[u];
                if (act) {
                    const unsigned qp = (((d.S + b) * nzpml + pj) * nx + x) * 8u;
                    const double pnew = pb[u] + ca.bnext * prhs;
                    stb(st.pz_tmp, qp, pnew);
                    if (LAST) stb(st.pz_base, qp, pnew);
                }
            }
            double rvz = -zs[F_RINV * nzp + i + u] * gpz + w[i + u];
            rvz = (j == 0 || x == 0 || x == nx - 1) ? 0.0 : rvz;
            vn[u] = bv[i >> 1][u] + ca.bnext * rvz;
            if (snap && act && j < nz) sink.snap[((slot + (sink.adjoint ? 3 : 5)) * nz + j) * nx + x] = rvz;
        }
        put2(ca.TN[3], i, vn[0], vn[1]);
    }
    if (LAST) {
        // FILTER_VARS_2D (physics2d.f90:509-556) of v_z, xi_z, xi_x, each from a
        // window of rows a-6 .. a+MS+5
        __syncthreads();
        const int oslot = sink.vz_out ? out_slot(time, clk.steps, sink.k0, sink.nout) : -1;
        const bool xin = x >= d.nh - 1 && x <= nx - d.nh;
#pragma unroll
        for (int g = 0; g < 3; g++) {
            const int fi = g == 0 ? 3 : (g == 1 ? 1 : 0);
            double v[MS + 12];
#pragma unroll
            for (int q = 0; q < MS + 12; q += 2) {
                const dpair t = ldp(ca.TN[fi], colb + pairo(h0 - 3 + (q >> 1)));
                v[q] = t.x;
                v[q + 1] = t.y;
            }
            // snapshot field: forward xi_x 0, xi_z 1, v_z 3; adjoint v_z 1
            const int fs = sink.adjoint ? (fi == 3 ? 1 : -1) : fi;
            double fv[MS];
#pragma unroll
            for (int i = 0; i < MS; i++) {
                const int j = a + i, q = i + 6;
                const double f11 = 0.75390625 * v[q] + 0.5 * 0.41015625 * (v[q - 1] + v[q + 1]) +
                                   0.5 * -0.234375 * (v[q - 2] + v[q + 2]) +
                                   0.5 * 0.087890625 * (v[q - 3] + v[q + 3]) +
                                   0.5 * -0.01953125 * (v[q - 4] + v[q + 4]) +
                                   0.5 * 0.001953125 * (v[q - 5] + v[q + 5]);
                const double f2 = 0.5 * (v[q + 1] + v[q - 1]);
                fv[i] = xin && j >= 5 && j <= nz - 2 ? (j <= nz - 6 ? f11 : f2) : v[q];
                if (act && j < nz) {
                    if (fi == 3 && oslot >= 0 && j == sink.orow)
                        sink.vz_out[((size_t)b * sink.nout + oslot) * nx + x] = fv[i];
                    if (snap && fs >= 0) sink.snap[(slot + fs) * nz * nx + (size_t)j * nx + x] = fv[i];
                }
            }
#pragma unroll
            for (int i = 0; i < MS; i += 2) put2(st.a[fi], i, fv[i], fv[i + 1]);
        }
    }
}

// Segment lengths of the one-lane form: longer ones do not fit its registers.  Eight
// rows keep 29 to 38 of them in scratch (120 to 188 bytes a lane) and 47 to 60 scalar
// registers in spill lanes; every shape is compared with the oracle.
#define SPARC_COLONE_SIZES(X) X(4) X(6) X(8)

inline size_t colone_lds_bytes(int tc, const SegTab &sg)
{
    const size_t img = ((size_t)3 * sg.nk * 2 * (4 * sg.hw + 4) + (size_t)kZS * 3 * sg.m + (size_t)kZF * sg.nzp + kCB + 1) &
                       ~(size_t)1;
    return sizeof(double) * (img + (size_t)4 * tc * yb_len(sg.P, sg.hw) + (size_t)tc * sg.nzp);
}

namespace {
int g_lds_max = 64 * 1024;   // dynamic LDS a block may use on this device
// Blocks of so many waves and bytes of LDS that a compute unit holds.
int resident(int waves, size_t lds)
{
    return std::min((int)((size_t)g_lds_max / lds), kWavesPerUnit / waves);
}
}  // namespace

// The form that a batch takes with blocks of tc columns.
bool col_one_lane(const Dims &d, const SegTab &sg, int tc)
{
    if (sg.m > 8 || (size_t)d.S * d.nx * d.nz < kOneLanePoints) return false;
    const int waves = (tc * sg.P + 63) / 64;
    if (waves > 2) return true;                      // more than the lane groups' 128 lanes
    return resident(waves, colone_lds_bytes(tc, sg)) >=
           kOneLaneBlocks * resident(3 * waves, colsplit_lds_bytes(tc, sg, d.nzpml));
}

// Raises every instantiation's dynamic-LDS limit to the device's maximum per
// block (gfx950: 160 KB).
hipError_t colseg_init()
{
    int dev = 0, v = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && v > 0)
        g_lds_max = v;
#define A(MSV)                                                                                          \
    if (hipFuncSetAttribute((const void *)k_colsplit<MSV, 0>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                            g_lds_max) != hipSuccess ||                                                 \
        hipFuncSetAttribute((const void *)k_colsplit<MSV, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                            g_lds_max) != hipSuccess) {                                                 \
        (void)hipGetLastError();                                                                        \
        g_lds_max = 64 * 1024;                                                                          \
    }
    SPARC_COLSEG_SIZES(A)
#undef A
#define A(MSV)                                                                                          \
    if (hipFuncSetAttribute((const void *)k_colone<MSV, 0>, hipFuncAttributeMaxDynamicSharedMemorySize,  \
                            g_lds_max) != hipSuccess ||                                                 \
        hipFuncSetAttribute((const void *)k_colone<MSV, 1>, hipFuncAttributeMaxDynamicSharedMemorySize,  \
                            g_lds_max) != hipSuccess) {                                                 \
        (void)hipGetLastError();                                                                        \
        g_lds_max = 64 * 1024;                                                                          \
    }
    SPARC_COLONE_SIZES(A)
#undef A
    return hipSuccess;
}

}  // namespace sparc

namespace sparc {

bool colsplit_fits(int tc, const Dims &d, const SegTab &sg)
{
    if (col_one_lane(d, sg, tc))
        return d.nx % tc == 0 && tc * sg.P <= 512 && colone_lds_bytes(tc, sg) <= (size_t)g_lds_max;
    return d.nx % tc == 0 && (tc * sg.P + 63) / 64 <= 2 &&
           colsplit_lds_bytes(tc, sg, d.nzpml) <= (size_t)g_lds_max;
}

hipError_t launch_colsplit(int tc, int ms, const Dims &d, const Bg &bg, const DbyCoef &cf, const SegTab &sg,
                           const State &s, const ColArgs &ca, const Src &src, const Clock &c, const Sink &sk,
                           hipStream_t st)
{
    if ((tc != 1 && tc != 2 && tc != 4 && tc != 8 && tc != 16) || d.nx % tc || sg.m != ms || sg.P > kSegMax)
        return hipErrorInvalidValue;
    if (col_one_lane(d, sg, tc)) {
        const size_t shm = colone_lds_bytes(tc, sg);
        if (tc * sg.P > 512 || shm > (size_t)g_lds_max) return hipErrorInvalidValue;
        const dim3 grid(d.nx / tc, d.S), block((tc * sg.P + 63) / 64 * 64);
#define L(MSV)                                                                                          \
    if (ms == MSV) {                                                                                    \
        if (ca.last) hipLaunchKernelGGL((k_colone<MSV, 1>), grid, block, shm, st, d, bg, cf, sg, s, ca, src, c, sk, tc); \
        else hipLaunchKernelGGL((k_colone<MSV, 0>), grid, block, shm, st, d, bg, cf, sg, s, ca, src, c, sk, tc);         \
        return hipGetLastError();                                                                       \
    }
        SPARC_COLONE_SIZES(L)
#undef L
        return hipErrorInvalidValue;
    }
    const int G = (tc * sg.P + 63) / 64 * 64;
    if (3 * G > 384) return hipErrorInvalidValue;
    dim3 grid(d.nx / tc, d.S), block(3 * G);
    const size_t shm = colsplit_lds_bytes(tc, sg, d.nzpml);
    if (shm > (size_t)g_lds_max) return hipErrorInvalidValue;
#define L(MSV)                                                                                          \
    if (ms == MSV) {                                                                                    \
        if (ca.last) hipLaunchKernelGGL((k_colsplit<MSV, 1>), grid, block, shm, st, d, bg, cf, sg, s, ca, src, c, sk, tc); \
        else hipLaunchKernelGGL((k_colsplit<MSV, 0>), grid, block, shm, st, d, bg, cf, sg, s, ca, src, c, sk, tc);         \
        return hipGetLastError();                                                                       \
    }
    SPARC_COLSEG_SIZES(L)
#undef L
    return hipErrorInvalidValue;
}

}  // namespace sparc
