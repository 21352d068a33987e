// sparc_zseg.h -- the segmented z kernels (sparc_zseg.hip): the two z passes of
// the 3D stage and the z-derivative (and its transpose) of a batch of fields.
#pragma once
#include "sparc_device.h"
#include "sparc_seg.h"

namespace sparc {

// Tables of one nz on the device (build_zseg): sets of one ibc each, one
// after the other in img; the right-hand side's coefficients by value.
struct ZSeg {
    int P, m, hw;
    const double *img;
    double c1, c2, cb[kCB];
};

namespace d3 {

// Arguments of the two z passes of a 3D stage.
struct Z3 {
    const double *B;            // Zp: xi_z; Zv: v_x (v_y, v_z follow at +N, +2N)
    double *W;                  // one-lane sweeps: forward-sweep values, one [nz][nxy] block per chain
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

// Whether the segmented passes take this grid: the tables exist (nz <= 512)
// and a field spans less than 2^31 bytes (32-bit byte offsets).
bool zseg3_fits(const Z3 &z, const ZSeg &sg);
// sg: sets ibc 1, ibc 0.
hipError_t launch_zp_seg(const Z3 &z, const ZSeg &sg, hipStream_t st);
hipError_t launch_zv_seg(const Z3 &z, const ZSeg &sg, hipStream_t st);

}  // namespace d3
}  // namespace sparc
