// Whole cross-plane solves with the plane in LDS (plane.hip).
#pragma once
#include "common.h"
#include "proj.h"

namespace duct {

constexpr int kPlaneMaxN = 128;   // interior points per direction: 8 tiles of 16

enum PlaneKind : int {
    PLANE_FWD = 0,   // helm3d: boundary mode bmode for Dirichlet fields, gauge and edges for Neumann ones
    PLANE_ADJ = 1,   // the transposed solve (duct_helm3d_adjoint_batch_dev_)
    PLANE_WALL = 2,  // helm3d_temp: separate y and z bases, wall data, edges per wall type
};

struct PlaneBasis {
    const double* A[4];       // bases of the four passes (build_frag, padded to NP)
    const double* lamy;       // eigenvalues of the y and z bases, padded to NP
    const double* lamz;
    const double* prow;       // FWD, ADJ Neumann: P(a, :), a the null mode
    const double* pcol;       // ADJ Neumann: P(:, a)
    const double* DC;         // Neumann: m x m
    const double* AM1;        // Neumann: 4 x 4
    double pdiag, wanted;
    int gauge;                // a, 0-based; -1 for Dirichlet and WALL
    int NP;
};

struct PlaneArgs {
    const d2v* in[kMaxFields];
    d2v* out[kMaxFields];
    double alambda[kMaxFields];
    int bnd[kMaxFields];      // 0 Dirichlet, 1 Neumann: the field's basis b[bnd] (WALL: 0)
    PlaneBasis b[2];
    int nf, nmodes, mode0, my, mz;
    int bmode;                // BoundaryMode of the Dirichlet fields (FWD)
    double alp;
    // WALL (as TempArgs)
    const double* bcy;
    const double* bcz;
    const double* vec;
    int by1, by2, bz1, bz2;
};
// whether planes of these sizes fit LDS
bool plane_supported(int my, int mz);
hipError_t launch_plane(int kind, const PlaneArgs& a, hipStream_t st);

}  // namespace duct
