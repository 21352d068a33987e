// sparc_zseg.h -- the segmented z kernels (sparc_zseg.hip): the two z passes of
// the 3D stage and the z-derivative (and its transpose) of a batch of fields.
#pragma once
#include "sparc_device.h"
#include "sparc_seg.h"

namespace sparc {

// Tables of one nz on the device (build_zseg): the sets of ibc 0, 1, 2, 3, then
// (2D handles) of the transposed matrices of ibc 1, 2, 3; the right-hand side's
// coefficients by value.
struct ZSeg {
    int P, m, hw;
    const double *img;
    double c1, c2, cb[kCB];
};
constexpr int kZSegSets = 4, kZSegSetsT = 7;

// The z-derivative (ddz, derivatives.f90:10-24; with filt, ddzkern,
// kernels.f90:648-661) of nbatch fields [nz][ncols], or its transpose.
struct ZDer {
    const double *in;
    double *out;                // may be in
    int ncols, nz, nbatch, ibc;
    const double *stretch;      // [nz], or null: plain dbyd2
    int filt;                   // pass the result through FILTER_VAR_Z
    // the kept first / last row of ibc 2 / 3: the row of out, or 0 with
    // zero_kept, or for ibc 3 pre_scale * pre[b * pre_stride + column] when
    // pre is given
    int zero_kept;
    const double *pre;
    size_t pre_stride;
    double pre_scale;
    // transposed (ibc 1..3, kept rows 0): eb from dbyd2_edge_rows; prebar[b *
    // prebar_stride + column] gets the adjoint of ibc 3's kept last row (may be null), or
    // prebar_add times it added where that is not 0
    int transposed;
    double eb[20];
    double *prebar;
    size_t prebar_stride;
    double prebar_add;
    // a second set of nbatch2 fields (0: none) of another ibc, without pre and prebar
    const double *in2;
    double *out2;
    int nbatch2, ibc2;
    double eb2[20];
};
// Whether the segmented form takes it: tables, and 32-bit offsets in a field.
bool zder_fits(const ZDer &a, const ZSeg &sg);
hipError_t launch_zder(const ZDer &a, const ZSeg &sg, hipStream_t st);

namespace d3 {

// Arguments of the two z passes of a 3D stage.
struct Z3 {
    const double *B;            // Zp: xi_z; Zv: v_x (v_y, v_z follow at +N, +2N)
    double *W;                  // one-lane sweeps only: forward-sweep values, one [nz][nxy] block per chain
    size_t N;                   // points per field
    int nxy, nz, nb, nt;
    const double *stretch;      // [nz]
    DbyCoef cf;
    Tri tr1, tr0;               // dbyd2 factors for ibc 1 and ibc 0
    const double *rhoinv;       // [nz] 1/rho0
    const double *az, *bz;      // [npml][nxy]
    const double *psi;          // z-PML variables of this stage [2][npml][nxy]: d xi_z/dz, d p/dz
    // the next stage's input (step.f90:60-62) or, after the fifth stage, the
    // updated state (:107-108): out = base + beta * RHS, for the fields and
    // the z-PML variables; the fifth stage also keeps the RHS in rhs
    const double *a, *pml;      // base: state a [6][nz][nxy], pmlvars [2][npml][nxy]
    double *tnext, *pnext;      // T of the next stage (or a), its PML variables (or pmlvars)
    double beta;
    int last;
    // Zp
    const double *dxi, *dyi;    // d xi_x/dx, d xi_y/dy
    const double *c2rho0;       // [nz][nxy]
    const double *gp0z, *gr0z;  // [nz] d p0/dz, d rho0/dz before the PML factor
    const double *fz;           // [npml][nxy] PML factor of the two
    const double *rho0, *g;     // [nz]
    double *P, *RG;             // p; rho' g / rho0
    // Zv
    const double *dxv, *dyv;    // d v_i/dx, d v_i/dy, [3][nz][nxy]
    const double *v0x, *v0y, *v0z;
    const double *dxp, *dyp;    // d p/dx, d p/dy
    double *rhs;                // scr [6][nz][nxy]
    const double *srcdep;       // [nz]
    Src src;
    int time, e_rad;
};

// Row of a PML array that holds grid row j, -1 outside the layers.
__device__ __forceinline__ int pml_index(int j, int nz, int nb, int nt)
{
    return j < nb ? j : (j >= nz - nt ? nb + (j - (nz - nt)) : -1);
}

// Whether the segmented passes take this grid: segments of at most kZSegMax3
// rows (every nz up to 512 but the ten that zseg_length names) and a field of less
// than 2^31 bytes (32-bit byte offsets).
bool zseg3_fits(const Z3 &z, const ZSeg &sg);
hipError_t launch_zp_seg(const Z3 &z, const ZSeg &sg, hipStream_t st);
hipError_t launch_zv_seg(const Z3 &z, const ZSeg &sg, hipStream_t st);

}  // namespace d3
}  // namespace sparc
